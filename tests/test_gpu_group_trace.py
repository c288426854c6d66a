"""Short ray launches walk each ray with several lanes; their hit records equal the per-lane walk's.

A launch with traversal statistics always takes the per-lane walk (checked against the oracle elsewhere), so it
is the reference here, at the ray counts where the lanes per ray change and on the rays a group walk hands back:
exact ties (every triangle twice), hits at t < 0, and rays that are empty, infinite or not numbers.
"""

import numpy as np
import pytest
import torch

from bajo_amd import scenes
from bajo_amd.bvh import TRACE, Camera, build_triangle_blas_set, build_triangle_bvh
from conftest import announce

pytestmark = pytest.mark.gpu

F32_MAX = float(np.finfo(np.float32).max)


def _rays(n, seed):
    rng = np.random.default_rng(seed)
    r = np.empty((8, n), np.float32)
    r[0:3] = rng.uniform(-0.1, 1.1, (3, n))
    r[3] = np.where(rng.random(n) < 0.1, -0.2, 0.0)  # some hits behind the origin count
    d = rng.normal(size=(3, n))
    r[4:7] = d / np.linalg.norm(d, axis=0) * rng.uniform(0.5, 2.0, n)
    r[7] = np.where(rng.random(n) < 0.5, F32_MAX, rng.uniform(0.0, 1.0, n))
    for k, (row, value) in enumerate([(7, -1.0), (7, np.inf), (7, np.nan), (0, np.nan), (4, np.nan), (4, np.inf),
                                      (7, 0.0), (5, 0.0), (0, 1e6), (0, 1e30)]):
        r[row, k * 7 % n] = value
    return torch.from_numpy(r.reshape(-1)).to("cuda:0")


def _bits(t):
    return t.view(torch.int32).cpu().numpy().reshape(-1, 8)


@pytest.mark.parametrize("width", [2, 4, 8])
@pytest.mark.parametrize("mesh", ["soup", "twice", "one"])
def test_group_walks_equal_per_lane(gpu_ctx, width, mesh):
    v = scenes.soup(1 if mesh == "one" else 6000, initstate=3, edge_min=0.01, edge_max=0.2)
    if mesh == "twice":
        v = np.concatenate([v, v])
    bvh = build_triangle_bvh(torch.from_numpy(v).to("cuda:0"), node_width=width)
    for n in (1, 65, 8192, 8193, 24577, 32769, 98305, 196609, 294913):
        announce(f"group trace {mesh} width {width} rays {n}")
        rays = _rays(n, n)
        hits = torch.full((8 * n,), 7.0, device="cuda:0")
        want = torch.full((8 * n,), 7.0, device="cuda:0")
        stats = torch.empty(5 * n, dtype=torch.int32, device="cuda:0")
        bvh.launch_rays(rays, want, stats=stats)
        bvh.launch_rays(rays, hits)
        torch.cuda.synchronize()
        assert np.array_equal(_bits(hits), _bits(want))
        bvh.launch_rays(rays, hits, mode=TRACE.ANY_HIT)
        torch.cuda.synchronize()
        got, ref = _bits(hits), _bits(want)
        found = ref[:, 2] != -1
        occluded = (got[:, 7] == 0) & (np.asarray(rays.cpu())[7 * n:] != 0)
        assert np.array_equal(occluded[rays.cpu().numpy()[7 * n:] != 0], found[rays.cpu().numpy()[7 * n:] != 0])
        assert np.all(got[:, 2:4] == -1)


@pytest.mark.parametrize("width", [2, 8])
def test_group_walks_of_set_cameras(gpu_ctx, width):
    sets = [torch.from_numpy(scenes.soup(n, initstate=5, initseq=n, edge_min=0.05, edge_max=0.3)).to("cuda:0")
            for n in (1, 2, 300, 1, 4097)]
    bset = build_triangle_blas_set(sets, node_width=width)
    cams = np.concatenate([Camera((0.5, 0.5, -1.5 - 0.1 * k), (0.5, 0.5, 0.5), (0.0, 1.0, 0.0), 0.41421356).flatten()
                           for k in range(len(sets))])
    cams = torch.from_numpy(cams).to("cuda:0")
    for w, h in ((13, 7), (61, 47), (150, 120)):
        n = len(sets) * w * h
        announce(f"set cameras width {width} {w}x{h}")
        hits = torch.full((8 * n,), 7.0, device="cuda:0")
        want = torch.full((8 * n,), 7.0, device="cuda:0")
        stats = torch.empty(5 * n, dtype=torch.int32, device="cuda:0")
        bset.launch_camera(cams, want, w, h, stats=stats)
        bset.launch_camera(cams, hits, w, h)
        torch.cuda.synchronize()
        assert np.array_equal(_bits(hits), _bits(want))
