"""Short ray launches walk each ray with several lanes; their hit records equal the per-lane walk's.

A launch with traversal statistics always takes the per-lane walk (checked against the oracle elsewhere), so it
is the reference here, at the ray counts where the lanes per ray change and on the rays a group walk hands back:
exact ties (every triangle twice), hits at t < 0, and rays that are empty, infinite or not numbers.
"""

import json
from pathlib import Path

import numpy as np
import pytest
import torch

import oracle
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


@pytest.mark.parametrize("width,n", [(2, 65536), (2, 65537), (8, 12288), (8, 12289)])
@pytest.mark.parametrize("triangles", [16384, 16385])
def test_lanes_by_the_number_of_triangles(gpu_ctx, width, n, triangles):
    """Hierarchies of few triangles change the lanes per ray at fewer rays."""
    announce(f"group trace of {triangles} triangles, width {width}, rays {n}")
    v = scenes.soup(triangles, initstate=6, edge_min=0.01, edge_max=0.1)
    bvh = build_triangle_bvh(torch.from_numpy(v).to("cuda:0"), node_width=width)
    rays = _rays(n, n + triangles)
    hits = torch.full((8 * n,), 7.0, device="cuda:0")
    want = torch.full((8 * n,), 7.0, device="cuda:0")
    bvh.launch_rays(rays, want, stats=torch.empty(5 * n, dtype=torch.int32, device="cuda:0"))
    bvh.launch_rays(rays, hits)
    torch.cuda.synchronize()
    assert np.array_equal(_bits(hits), _bits(want))
    bvh.free()


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


def _facing(p, d, s):
    u = np.cross(d, [0.3, 0.5, -0.8])
    u /= np.linalg.norm(u)
    w = np.cross(d, u)
    return [p + s * u, p + s * (-0.5 * u + 0.8 * w), p + s * (-0.5 * u - 0.8 * w)]


def _edge_on(case, seed):
    """A triangle seen edge on whose computed hit lies before its own box, and a triangle facing the ray between the
    two: whether a walk that takes nodes in order meets the first depends on when it finds the second.  Others that
    the ray misses put the two into different nodes."""
    o, d = np.array(case["origin"]), np.array(case["direction"])
    tri = np.array(case["triangle"]).reshape(3, 3)
    rng = np.random.default_rng(seed)
    with np.errstate(divide="ignore"):
        a, b = (tri.min(0) - o) / d, (tri.max(0) - o) / d
    enter, leave = np.minimum(a, b).max(), np.maximum(a, b).min()
    u = np.cross(d, [0, 1, 0])
    u /= np.linalg.norm(u)
    w = np.cross(d, u)
    out = [tri, _facing(o + enter * (1 - 6e-6) * d, d, 0.002)]
    for k in range(6):
        if seed == 0:
            out.append(_facing(o + (enter - 0.05 - 0.03 * k) * d + (0.02 + 0.01 * k) * u, d, 0.004))
            out.append(_facing(o + (leave + 0.1 + 0.05 * k) * d + (0.02 + 0.01 * k) * u, d, 0.004))
        else:
            out.append(_facing(o + (enter - 0.3 - 0.05 * k) * d + rng.normal(size=3) * 0.05, d, 0.01))
            out.append(_facing(o + (leave + 0.02 + 0.05 * k) * d + rng.normal(size=3) * 0.05, d, 0.004))
    out += [_facing(o + (enter + 2) * d + 0.5 * w, d, 0.3), _facing(o + (enter - 2) * d - 0.5 * w + 0.5 * u, d, 0.3)]
    rays = np.zeros(8, np.float32)
    rays[0:3], rays[4:7], rays[7] = o, d, F32_MAX
    return np.array(out, np.float32).reshape(-1), rays


@pytest.mark.parametrize("width,leaf", [(2, 0), (8, 1), (8, 4)])
def test_hits_before_their_box(gpu_ctx, width, leaf):
    """Triangles seen edge on next to others: the lane groups' hits are the ordered walk's (the oracle's), whatever
    the number of rays and so of lanes."""
    cases = json.loads((Path(__file__).parent / "golden" / "grazing_hits.json").read_text())["cases"]
    decided = 0
    for k, case in enumerate(cases):
        for seed in range(4):
            v, ray = _edge_on(case, seed)
            lb = oracle.build_lbvh(v)
            if width == 2:
                want = oracle.trace_bvh2(v, lb, ray)
            else:
                want = oracle.trace_wide(v, lb["leaf_ids"], oracle.collapse_wide(lb, leaf), ray)[0]
            decided += not np.array_equal(want[2:3].view(np.uint32), oracle.trace_brute(v, ray)[2:3].view(np.uint32))
            bvh = build_triangle_bvh(torch.from_numpy(v).to("cuda:0"), node_width=width, leaf_size=leaf)
            for n in (32, 20_000, 90_000, 200_000):
                if k == 0:
                    announce(f"edge-on triangles width {width} leaf {leaf} rays {n}")
                rays = torch.from_numpy(np.repeat(ray[:, None], n, 1).reshape(-1)).to("cuda:0")
                hits = torch.full((8 * n,), 7.0, device="cuda:0")
                bvh.launch_rays(rays, hits)
                torch.cuda.synchronize()
                got = _bits(hits)
                assert (got == got[0]).all()
                assert np.array_equal(got[0], want.reshape(-1).view(np.int32)), (k, seed, n)
            bvh.free()
    assert decided >= 5  # the order of the walk decided some of them
