"""Scenes of more than 2^26 interior nodes, whose records lie beyond a 32-bit
byte offset: the traversal kernels then address nodes with 64 bits (WIDE).  A
height field of 67.3M triangles, made and built on the device, seen where the
tree's last-numbered nodes are.  Bar: the bits of the reference-layout kernels,
which read the flat arrays with their own indices (and are held to the oracle
in test_gpu_trace.py), for every batch mode, the record forms and the renders."""
import ctypes

import numpy as np
import pytest
import torch

from mambatracer_amd import _lib, api
from mambatracer_amd import workloads as W

pytestmark = pytest.mark.gpu

NX, NY = 8208, 4100  # quads


class _DeviceScene:
    """mt_scene_create over arrays that are on the device already."""

    def __init__(self, ctx, points, faces, nodes, bounds, depth):
        self.keep = (points, faces, nodes, bounds)
        desc = _lib.SceneDesc(points.data_ptr(), None, None, faces.data_ptr(), nodes.data_ptr(), bounds.data_ptr(),
                              int(faces.shape[0]), int(points.shape[0]), depth)
        self.handle = ctypes.c_void_p()
        torch.cuda.synchronize()
        api.call("mt_scene_create", ctx.handle, ctypes.byref(desc), ctypes.byref(self.handle))


@pytest.fixture(scope="module")
def wide(ctx):
    if torch.cuda.mem_get_info(0)[0] < 64 << 30:
        pytest.skip("needs 64 GiB of device memory")
    g = torch.Generator(device="cuda")
    g.manual_seed(3)
    points = torch.zeros(((NX + 1) * (NY + 1), 4), device="cuda")
    v = torch.arange(points.shape[0], device="cuda")
    points[:, 0] = (v % (NX + 1)) * 0.01
    points[:, 2] = (v // (NX + 1)) * 0.01
    points[:, 1] = torch.rand((points.shape[0],), generator=g, device="cuda") * 0.02
    n = 2 * NX * NY
    faces = torch.full((n, 10), -1, dtype=torch.int32, device="cuda")
    q = torch.arange(NX * NY, device="cuda")
    a = ((q // NX) * (NX + 1) + q % NX).to(torch.int32)
    faces[0::2, 0], faces[0::2, 1], faces[0::2, 2] = a, a + 1, a + NX + 1
    faces[1::2, 0], faces[1::2, 1], faces[1::2, 2] = a + 1, a + NX + 2, a + NX + 1
    faces[:, 9] = torch.randint(0, 257, (n,), generator=g, device="cuda", dtype=torch.int32)
    del v, q, a
    torch.cuda.synchronize()
    nodes, bounds, depth = api.CNormalBVH.build_device(ctx, points, faces)
    assert n - 1 > 1 << 26
    sc = _DeviceScene(ctx, points, faces, nodes, bounds, depth)
    # centroids of the triangles whose parents have the largest packed indices
    leaf = nodes[:, 5] != 0
    last = leaf.nonzero().reshape(-1)[-200_000:]
    parent = nodes[last, 4].long()
    packed = parent - leaf.to(torch.int32).cumsum(0, dtype=torch.int32)[parent]
    tri = nodes[last, 6].long()[packed >= 1 << 26]
    assert tri.numel() > 100_000
    centre = points[faces[tri, :3].long(), :3].mean(1)
    yield sc, centre
    _lib.load().mt_scene_destroy(sc.handle)
    del sc, nodes, bounds, faces, points, leaf, last, parent, packed, tri, centre
    torch.cuda.empty_cache()


def _rays(centre):
    """Rays at points of those triangles, from above and from the sides."""
    g = torch.Generator(device="cuda")
    g.manual_seed(4)
    k = centre.shape[0]
    o = torch.zeros((k, 4), device="cuda")
    o[:, :3] = centre + torch.rand((k, 3), generator=g, device="cuda") * torch.tensor([0.6, 0.5, 0.6], device="cuda")
    d = torch.zeros((k, 4), device="cuda")
    d[:, :3] = centre - o[:, :3]
    d[:, :3] /= d[:, :3].norm(dim=1, keepdim=True)
    d[:, 3] = float("inf")
    return o, d


def test_rays(ctx, wide):
    print("[case] wide rays", flush=True)
    sc, centre = wide
    o, d = _rays(centre)
    rprim, rt, _ = api.intersect_primitives(ctx, sc, o, d, mode=_lib.MT_TRACE_REFERENCE)
    rocc, _ = api.intersect_occlusion(ctx, sc, o, d, mode=_lib.MT_TRACE_REFERENCE)
    assert int((rprim >= 0).sum()) > centre.shape[0] * 9 // 10
    recs = ctx.to_device(api.ray_records(o.cpu().numpy(), d.cpu().numpy()))
    for mode in (_lib.MT_TRACE_PACKED, _lib.MT_TRACE_PACKED_POOL, _lib.MT_TRACE_PACKED_BINNED):
        print(f"mode {mode}", flush=True)
        prim, t, _ = api.intersect_primitives(ctx, sc, o, d, mode=mode)
        occ, _ = api.intersect_occlusion(ctx, sc, o, d, mode=mode)
        hits = torch.full_like(rocc, -7)
        api.intersect_occlusion_records(ctx, sc, recs, hits, mode=mode)
        isects = torch.zeros((o.shape[0], api.INTERSECTION_RECORD_WORDS), dtype=torch.int32, device="cuda")
        api.intersect_records(ctx, sc, recs.clone(), isects, mode=mode)
        torch.cuda.synchronize()
        assert torch.equal(prim, rprim) and torch.equal(t.view(torch.int32), rt.view(torch.int32))
        assert torch.equal(occ, rocc) and torch.equal(hits, rocc)
        assert torch.equal(isects[:, 20], (rprim >= 0).to(torch.int32))
        assert torch.equal(isects[rprim >= 0, 19], rprim[rprim >= 0])


@pytest.mark.parametrize("w,h,spp", [(64, 48, 3), (601, 450, 1)])  # one launch; launches per bounce
def test_renders(ctx, wide, w, h, spp):
    print(f"[case] wide renders {w}x{h}x{spp}", flush=True)
    sc, centre = wide
    env = api.CEnvironment(ctx)
    env.setEnvironmentMap(W.env_map())
    dm = ctx.to_device(W.c1_materials())
    c = centre.double().median(0).values.tolist()
    job = W.RenderJob(width=w, height=h, spp=spp, seed=7, pos=(c[0] + 0.1, c[1] + 0.4, c[2] + 0.1), look=tuple(c))
    out = []
    for mode, flags in ((_lib.MT_TRACE_REFERENCE, 0), (_lib.MT_TRACE_PACKED, 0), (_lib.MT_TRACE_PACKED_POOL, 0),
                        (_lib.MT_TRACE_PACKED, _lib.MT_RENDER_PROFILE),
                        (_lib.MT_TRACE_PACKED, _lib.MT_RENDER_TAIL_FROM(1))):
        print(f"mode {mode} flags {flags}", flush=True)
        job.mode, job.flags = mode, flags
        img, st = api.render(ctx, sc, dm, env, job)
        out.append((img.cpu().numpy().view(np.int32), [int(st.extension_rays), int(st.shadow_rays),
                                                       *st.bounce_counts]))
    assert out[0][1][3] > w * h * spp // 2  # most paths hit the ground
    for img, st in out[1:]:
        np.testing.assert_array_equal(img, out[0][0])
        assert st == out[0][1]
