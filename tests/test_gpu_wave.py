"""The wave traversal (mt_traverse.h) where it can go wrong: runs that end in
the middle of a wave, more pending subtrees than a lane's LDS rows, rays and
boxes that need intersectBoundT's NaN rules, a scene that is a single leaf.
Bar: prim, t and occlusion bit-exact against the oracle, in every mode that
uses it (direct, staged and sorted)."""
import numpy as np
import pytest
import torch

from mambatracer_amd import _lib, api
from oracle import orc_py as orc

pytestmark = pytest.mark.gpu

MODES = [_lib.MT_TRACE_PACKED, _lib.MT_TRACE_PACKED_POOL, _lib.MT_TRACE_PACKED_BINNED]


def _check(ctx, arrs, o, d, mode, count=None):
    points, faces, nodes, bounds, depth = arrs
    sc = api.Scene(ctx, points, faces, nodes, bounds, depth)
    n = o.shape[0]
    m = n if count is None else count
    dc = ctx.scalar_i32(m)
    do, dd = ctx.to_device(o), ctx.to_device(d)
    prim, t, _ = api.intersect_primitives(ctx, sc, do, dd, count=dc, mode=mode)
    occ, _ = api.intersect_occlusion(ctx, sc, do, dd, count=dc, mode=mode)
    rays = ctx.to_device(api.ray_records(o, d))
    hits = torch.full((n,), 7, dtype=torch.int32, device="cuda")
    api.intersect_occlusion_records(ctx, sc, rays, hits, count=dc, mode=mode)
    isects = torch.full((n, api.INTERSECTION_RECORD_WORDS), 3, dtype=torch.int32, device="cuda")
    api.intersect_records(ctx, sc, rays, isects, count=dc, mode=mode)
    torch.cuda.synchronize()
    oprim, ot, _, _ = orc.trace_closest(points, faces, nodes, bounds, o[:m], d[:m])
    oocc, _, _ = orc.trace_any(points, faces, nodes, bounds, o[:m], d[:m])
    np.testing.assert_array_equal(prim.cpu().numpy()[:m], oprim)
    np.testing.assert_array_equal(t.cpu().numpy()[:m].view(np.int32), ot.view(np.int32))
    np.testing.assert_array_equal(occ.cpu().numpy()[:m], oocc)
    np.testing.assert_array_equal(hits.cpu().numpy(), np.concatenate([oocc, np.full(n - m, 7, np.int32)]))
    rec = isects.cpu().numpy()
    np.testing.assert_array_equal(rec[:m, 20], (oprim >= 0).astype(np.int32))
    np.testing.assert_array_equal(rec[:m][oprim >= 0, 19], oprim[oprim >= 0])
    np.testing.assert_array_equal(rec[m:, 20], 0)
    return oprim


def _build(points, faces):
    return (points, faces, *api.CNormalBVH.build(points, faces))


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n,count", [(1, None), (15, None), (17, 16), (64, 63), (65, None), (1000, 513), (70001, 69990)])
def test_runs_of_every_length(ctx, c0, mode, n, count):
    print(f"[case] wave runs mode={mode} n={n} count={count}", flush=True)
    o, d = api.gen_random_rays(n, 0, n, [-0.9] * 3, [0.9] * 3)
    assert (_check(ctx, c0, o, d, mode, count) >= 0).all()  # inside the room box


def _nested(n):
    """n wide triangles at z = 2.1^i: the midpoint split peels the farthest one
    off at every level, and a ray along +z through them all hits both children
    at every level, so n - 1 subtrees are pending when it reaches its first
    leaf."""
    points = np.zeros((3 * n, 4), np.float32)
    faces = np.zeros((n, 10), np.int32)
    faces[:, 3:9] = -1
    for i in range(n):
        z = np.float32(2.1) ** i
        points[3 * i:3 * i + 3, :3] = [[-9, -9, z], [9, -9, z], [0, 9, z]]
        faces[i, :3] = [3 * i, 3 * i + 1, 3 * i + 2]
    return _build(points, faces)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", [9, 10, 11, 13, 14, 15, 16, 90])
def test_stack_past_the_lds_rows(ctx, mode, n):
    print(f"[case] wave stack mode={mode} n={n}", flush=True)
    arrs = _nested(n)
    rng = np.random.default_rng(n)
    r = 300
    o = np.zeros((r, 4), np.float32)
    d = np.zeros((r, 4), np.float32)
    o[:, :2] = rng.uniform(-3, 3, (r, 2))
    o[:, 2] = np.where(rng.random(r) < 0.7, 0.0, 9e29)
    d[:, :2] = rng.normal(0, 1e-3, (r, 2))
    d[:, 2] = np.where(o[:, 2] > 0, -1.0, 1.0)
    d[:, 3] = np.inf
    o[:, 3] = np.where(rng.random(r) < 0.5, 0.0, 2.1 ** (n // 2))  # a tMin that rejects the first half
    _check(ctx, arrs, o, d, mode)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("n", [64, 4097])
def test_rays_that_need_the_nan_rules(ctx, c0, mode, n):
    """Axis-parallel rays that start on box planes (0 * inf), directions with
    infinite, zero and denormal components, origins that are not finite; mixed
    with ordinary rays in the same waves."""
    print(f"[case] wave nan mode={mode} n={n}", flush=True)
    points, faces, nodes, bounds, _ = c0
    rng = np.random.default_rng(n)
    o, d = api.gen_random_rays(7, 0, n, [-0.9] * 3, [0.9] * 3)
    pick = rng.integers(0, bounds.shape[0], n)
    ax = rng.integers(0, 3, n)
    k = np.arange(n)
    special = rng.random(n) < (1.0 if n == 64 else 0.02)
    o[k[special], ax[special]] = bounds[pick, ax][special]
    d[k[special], ax[special]] = rng.choice(np.float32([0.0, -0.0, 1e-40, -1e-40, np.inf, np.nan]), n)[special]
    far = rng.random(n) < 0.01
    o[far, 0] = rng.choice(np.float32([np.inf, -np.inf, np.nan, 1e35]), n)[far]
    _check(ctx, c0, o, d, mode)


@pytest.mark.parametrize("mode", MODES)
def test_boxes_that_are_not_plain(ctx, c0, mode):
    """Inverted and infinite boxes turn the whole scene to the exact slab test."""
    print(f"[case] wave boxes mode={mode}", flush=True)
    points, faces, nodes, bounds, depth = c0
    bounds = bounds.copy()
    rng = np.random.default_rng(3)
    b = rng.integers(1, bounds.shape[0], 500)
    bounds[b[:250], 0], bounds[b[:250], 4] = bounds[b[:250], 4], bounds[b[:250], 0].copy()
    bounds[b[250:], 5] = np.inf
    o, d = api.gen_random_rays(9, 0, 5000, [-0.9] * 3, [0.9] * 3)
    _check(ctx, (points, faces, nodes, bounds, depth), o, d, mode)


@pytest.mark.parametrize("mode", MODES)
def test_scene_of_one_leaf(ctx, mode):
    print(f"[case] wave one leaf mode={mode}", flush=True)
    points = np.zeros((3, 4), np.float32)
    points[:, :3] = [[-1, -1, 2], [1, -1, 2], [0, 1, 2]]
    faces = np.full((1, 10), -1, np.int32)
    faces[0, :3] = [0, 1, 2]
    faces[0, 9] = 0
    o, d = api.gen_camera_rays([0, 0, 0], [0, 0, 1], [0, 1, 0], 80.0, 20, 20)
    prim = _check(ctx, _build(points, faces), o, d, mode)
    assert 0 < (prim == 0).sum() < prim.size
