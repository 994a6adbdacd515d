"""mt_batch_set_trace_mode picks a kernel: each mode's own form of the walk runs
(kernel names from torch's profiler), also after the engine's iterations were
recorded in another mode, and gives the images of plain renders."""
import numpy as np
import pytest
import torch

from mambatracer_amd import _lib, api
from mambatracer_amd import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graphs", [True, False])
def test_modes_run_their_own_kernels(ctx, graphs):
    print(f"[case] engine modes graphs={graphs}", flush=True)
    sc = api.Scene(ctx, *W.soup_scene(3000, 71))
    dm = ctx.to_device(W.c1_materials())
    env = api.CEnvironment(ctx)
    env.setEnvironmentMap(W.env_map())
    job = W.soup_job(W.JobSpec(0, 0, 90, 3, 5))
    ref, _ = api.render(ctx, sc, dm, env, job)
    img = ctx.empty((90 * 90, 4), torch.float32)
    b = api.Batch(ctx, queue_capacity=1 << 14, arena_bytes=64 << 20, max_jobs=4)
    b.set_graphs(graphs)
    names = {}
    for mode in (_lib.MT_BATCH_TRACE_SPLIT, _lib.MT_TRACE_PACKED_STACK, _lib.MT_TRACE_PACKED_POOL,
                 _lib.MT_TRACE_PACKED):
        b.set_trace_mode(mode)
        for _ in range(2):  # recorded, then replayed
            img.fill_(-1)
            torch.cuda.synchronize()
            with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA]) as prof:
                b.submit(0, sc, dm, env, job, img)
                b.run()
                torch.cuda.synchronize()
            np.testing.assert_array_equal(img.cpu().numpy().view(np.int32), ref.cpu().numpy().view(np.int32))
            names[mode] = {e.key for e in prof.key_averages() if "k_trace_jobs" in e.key}
    b.close()
    print(names, flush=True)
    assert all(len(v) == 1 for v in names.values())
    assert names[_lib.MT_TRACE_PACKED] == names[_lib.MT_BATCH_TRACE_SPLIT]
    assert len(set().union(*names.values())) == 3
