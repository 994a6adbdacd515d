"""Queues whose device count lies far below their capacity, as after each
compaction of a wavefront: waves are sized by the count (plain_run), the grid
by the capacity.  Bars: every live entry equals the oracle and nothing past
the count is written, but for the misses of the record form; and such a queue
takes no longer than 1.4 times a queue of its own size (20K live of 2M: 1.0,
with runs sized by the capacity 1.8 to 2.2)."""
import time

import numpy as np
import pytest
import torch

from mambatracer_amd import _lib, api
from oracle import orc_py as orc

pytestmark = pytest.mark.gpu

CAPACITY = 300_001
MODES = [_lib.MT_TRACE_PACKED, _lib.MT_TRACE_PACKED_REFILL, _lib.MT_TRACE_PACKED_POOL, _lib.MT_TRACE_PACKED_BINNED]


@pytest.fixture(scope="module")
def rays(c0):
    points, faces, nodes, bounds, _ = c0
    o, d = api.gen_random_rays(11, 0, CAPACITY, [-0.9] * 3, [0.9] * 3)
    return o, d, orc.trace_closest(points, faces, nodes, bounds, o, d), orc.trace_any(points, faces, nodes, bounds, o, d)


@pytest.mark.parametrize("mode", MODES)
@pytest.mark.parametrize("count", [-1, 0, 1, 16, 17, 2047, 2049, 32769, 131_073, 300_000, 300_001, 400_000])
def test_counts_below_the_capacity(ctx, c0, rays, mode, count):
    print(f"[case] count {count} of {CAPACITY} mode={mode}", flush=True)
    o, d, (oprim, ot, _, _), (oocc, _, _) = rays
    points, faces, nodes, bounds, depth = c0
    sc = api.Scene(ctx, points, faces, nodes, bounds, depth)
    do, dd, dc = ctx.to_device(o), ctx.to_device(d), ctx.scalar_i32(count)
    m = min(max(count, 0), CAPACITY)
    prim = torch.full((CAPACITY,), -7, dtype=torch.int32, device="cuda")
    t = torch.full((CAPACITY,), -7.0, device="cuda")
    occ = torch.full((CAPACITY,), -7, dtype=torch.int32, device="cuda")
    hits = torch.full((CAPACITY,), -7, dtype=torch.int32, device="cuda")
    isects = torch.full((CAPACITY, api.INTERSECTION_RECORD_WORDS), -7, dtype=torch.int32, device="cuda")
    recs = ctx.to_device(api.ray_records(o, d))
    api.call("mt_trace_closest", ctx.handle, sc.handle, do.data_ptr(), dd.data_ptr(), dc.data_ptr(), CAPACITY,
             prim.data_ptr(), t.data_ptr(), None, mode)
    api.call("mt_trace_any", ctx.handle, sc.handle, do.data_ptr(), dd.data_ptr(), dc.data_ptr(), CAPACITY,
             occ.data_ptr(), None, mode)
    api.intersect_occlusion_records(ctx, sc, recs, hits, count=dc, mode=mode)
    api.intersect_records(ctx, sc, recs, isects, count=dc, mode=mode)
    torch.cuda.synchronize()
    for got, want in ((prim, oprim), (occ, oocc), (hits, oocc)):
        got = got.cpu().numpy()
        np.testing.assert_array_equal(got[:m], want[:m])
        assert (got[m:] == -7).all()
    t = t.cpu().numpy()
    np.testing.assert_array_equal(t[:m].view(np.int32), ot[:m].view(np.int32))
    assert (t[m:] == -7).all()
    rec = isects.cpu().numpy()
    np.testing.assert_array_equal(rec[:m, 20], (oprim[:m] >= 0).astype(np.int32))
    np.testing.assert_array_equal(rec[:m, 19][oprim[:m] >= 0], oprim[:m][oprim[:m] >= 0])
    assert (rec[m:, 20] == 0).all() and (rec[m:, 18] == -1).all()
    rest = np.delete(rec[m:], [18, 20], axis=1)
    assert (rest == -7).all()


@pytest.mark.parametrize("mode", [_lib.MT_TRACE_PACKED, _lib.MT_TRACE_PACKED_POOL])
def test_a_shrunken_queue_costs_what_it_holds(ctx, c0, mode):
    live, capacity = 20_000, 2_000_000
    print(f"[case] {live} of {capacity} mode={mode}", flush=True)
    points, faces, nodes, bounds, depth = c0
    sc = api.Scene(ctx, points, faces, nodes, bounds, depth)
    o, d = (ctx.to_device(x) for x in api.gen_random_rays(12, 0, capacity, [-0.9] * 3, [0.9] * 3))
    recs = torch.zeros((capacity, api.RAY_RECORD_WORDS), device="cuda")
    recs[:live] = ctx.to_device(api.ray_records(o[:live].cpu().numpy(), d[:live].cpu().numpy()))
    hits = torch.zeros((capacity,), dtype=torch.int32, device="cuda")
    count = ctx.scalar_i32(live)

    def best(n, call):
        times = []
        for rep in range(9):
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for _ in range(10):
                call(n)
            torch.cuda.synchronize()
            times.append(time.perf_counter() - t0)
        return min(times)

    for name, call in (("closest", lambda n: api.intersect_primitives(ctx, sc, o[:n], d[:n], count=count, mode=mode)),
                       ("any", lambda n: api.intersect_occlusion(ctx, sc, o[:n], d[:n], count=count, mode=mode)),
                       ("records", lambda n: api.intersect_occlusion_records(ctx, sc, recs[:n], hits[:n], count=count,
                                                                             mode=mode))):
        whole, own = best(capacity, call), best(live, call)
        print(f"{name}: {whole * 1e5:.0f} us of {capacity}, {own * 1e5:.0f} us of {live}", flush=True)
        assert whole < 1.4 * own
