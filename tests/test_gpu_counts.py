"""Launches whose device count the wrapper makes itself, with the context on
torch's current stream and on another one.  Bar: every entry traced, equal to
the oracle."""
import numpy as np
import pytest
import torch

from mambatracer_amd import _lib, api
from oracle import orc_py as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("current", [True, False])
@pytest.mark.parametrize("n", [1, 4097, 100_003])
def test_counts_on_either_stream(c0, n, current):
    print(f"[case] counts n={n} current={current}", flush=True)
    points, faces, nodes, bounds, depth = c0
    o, d = api.gen_random_rays(n, 0, n, [-0.9] * 3, [0.9] * 3)
    oprim, ot, _, _ = orc.trace_closest(points, faces, nodes, bounds, o, d)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side if current else torch.cuda.current_stream()):
        ctx = api.Context(0, stream=side)
        sc = api.Scene(ctx, points, faces, nodes, bounds, depth)
        do, dd = ctx.to_device(o), ctx.to_device(d)
        flags = (torch.arange(n, device="cuda") % 3 == 0).to(torch.int32)
        torch.cuda.synchronize()
        for _ in range(3):  # the word's memory is handed out again
            prim, t, _ = api.intersect_primitives(ctx, sc, do, dd)
            idx, count, _ = api.compact(ctx, flags)
            ctx.sync()
            np.testing.assert_array_equal(prim.cpu().numpy(), oprim)
            np.testing.assert_array_equal(t.cpu().numpy().view(np.int32), ot.view(np.int32))
            assert int(count.item()) == (n + 2) // 3
            np.testing.assert_array_equal(idx.cpu().numpy()[:(n + 2) // 3], np.arange(0, n, 3))
        sc.close()
        ctx.close()
