"""Renders in MT_TRACE_PACKED_BINNED mode: the sort's workspace is the one a
render keeps its state in, so a render takes the mode as MT_TRACE_PACKED_POOL.
Bar: the default mode's image bits and ray counts, on a context without a
workspace and on one whose workspace already has room for a sort; profiled,
counted, captured and replayed too."""
import numpy as np
import pytest
import torch

from mambatracer_amd import _lib, api
from mambatracer_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("room", [False, True])
@pytest.mark.parametrize("w,h,spp", [(1, 1, 1), (96, 54, 4), (600, 450, 1)])
def test_binned_renders_as_the_default(w, h, spp, room):
    print(f"[case] binned render {w}x{h}x{spp} room={room}", flush=True)
    ctx = api.Context(0)
    points, faces, nodes, bounds, depth = W.soup_scene(5000, 61)
    sc = api.Scene(ctx, points, faces, nodes, bounds, depth)
    dm = ctx.to_device(W.c1_materials())
    env = api.CEnvironment(ctx)
    env.setEnvironmentMap(W.env_map())
    job = W.soup_job(W.JobSpec(0, 0, 8, spp, 31))
    job.width, job.height = w, h
    if room:  # a workspace larger than the render's state and the sort's together
        o, d = (ctx.to_device(x) for x in api.gen_random_rays(3, 0, 4_000_000, [-0.9] * 3, [0.9] * 3))
        api.intersect_occlusion(ctx, sc, o, d, mode=_lib.MT_TRACE_PACKED_BINNED)
        ctx.sync()

    def eager(mode, flags=0):
        job.mode, job.flags = mode, flags
        img, st = api.render(ctx, sc, dm, env, job)
        return img.cpu().numpy().view(np.int32), [int(st.extension_rays), int(st.shadow_rays), *st.bounce_counts]

    for flags in (0, _lib.MT_RENDER_PROFILE, _lib.MT_RENDER_TRAVERSAL_STATS, _lib.MT_RENDER_TAIL_FROM(2)):
        img, st = eager(_lib.MT_TRACE_PACKED_BINNED, flags)
        ref, ref_st = eager(_lib.MT_TRACE_PACKED)
        np.testing.assert_array_equal(img, ref)
        assert st == ref_st
    job.mode, job.flags = _lib.MT_TRACE_PACKED_BINNED, 0
    g = api.RenderGraph(ctx, sc, dm, env, job)
    for _ in range(3):
        g.launch(job.seed)
        st = g.stats()
        np.testing.assert_array_equal(g.image.cpu().numpy().view(np.int32), ref)
        assert [int(st.extension_rays), int(st.shadow_rays), *st.bounce_counts] == ref_st
        eager(_lib.MT_TRACE_PACKED)  # eager work between replays
        torch.cuda.synchronize()
    g.close()
    sc.close()
    ctx.close()
