"""The multi-job engine where its launches change shape: queues far from full
(the closest hits are spread by the queue's length, not its capacity), queues
of a few entries, and more iterations per step than the any hit on the side
stream has events.  Bar: the image bits of plain renders that keep their
launches per bounce."""
import numpy as np
import pytest
import torch

from mambatracer_amd import _lib, api
from mambatracer_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("capacity,iters", [(64, 70), (4097, 2), (1 << 17, 70), (1 << 21, 9)])
def test_engine_and_renders_agree(ctx, capacity, iters, graphs):
    print(f"[case] engine capacity={capacity} iters={iters} graphs={graphs}", flush=True)
    scenes = [api.Scene(ctx, *W.soup_scene(n, seed)) for n, seed in ((900, 51), (30_000, 52))]
    dm = ctx.to_device(W.c1_materials())
    env = api.CEnvironment(ctx)
    env.setEnvironmentMap(W.env_map())
    sides = [(0, 5, 1), (1, 11, 2), (0, 1, 1)] if capacity == 64 else [(0, 130, 3), (1, 61, 9), (1, 200, 1), (0, 1, 1)]
    b = api.Batch(ctx, queue_capacity=capacity, arena_bytes=64 << 20, max_jobs=8)
    b.set_graphs(graphs)
    b.set_iterations(iters)
    got = []
    for tag, (k, side, spp) in enumerate(sides):
        job = W.soup_job(W.JobSpec(tag, k, side, spp, 700 + tag))
        got.append((k, job, ctx.empty((side * side, 4), torch.float32)))
        b.submit(tag, scenes[k], dm, env, job, got[-1][2])
    assert sorted(b.run()) == list(range(len(sides)))
    b.close()
    for k, job, img in got:
        job.flags = _lib.MT_RENDER_PROFILE
        ref, _ = api.render(ctx, scenes[k], dm, env, job)
        np.testing.assert_array_equal(img.cpu().numpy().view(np.int32), ref.cpu().numpy().view(np.int32))
