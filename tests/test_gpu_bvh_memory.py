"""What the device BVH builder keeps of the GPU's memory: its state stays with
the context up to 512 MiB and is given back by the call beyond.  Bar: device
memory outside torch's allocator grows by no more than that (allocation pieces of
2 MiB allowed for), a second build takes nothing
more, and the tree is the host builder's."""
import numpy as np
import pytest
import torch

from mambatracer_amd import api

pytestmark = pytest.mark.gpu


def _held():
    torch.cuda.synchronize()
    free, total = torch.cuda.mem_get_info(0)
    return total - free - torch.cuda.memory_reserved(0)


@pytest.mark.parametrize("n,most", [(1_000_000, 160 << 20), (4_000_000, 512 << 20), (5_000_000, 8 << 20)])
def test_build_state_is_bounded(n, most):
    print(f"[case] bvh memory n={n}", flush=True)
    ctx = api.Context(0)
    p, f = api.gen_soup(n, n, -1, 1, 0.001, 0.01)
    dp, df = ctx.to_device(p), ctx.to_device(f)
    api.CNormalBVH.build_device(ctx, dp[:300], df[:100])  # code object, scan workspace
    before = _held()
    dn, db, dd = api.CNormalBVH.build_device(ctx, dp, df)
    grown = _held() - before
    api.CNormalBVH.build_device(ctx, dp, df)
    again = _held() - before
    print(f"grown by {grown >> 20} MiB, then {again >> 20} MiB", flush=True)
    assert grown <= most and again <= grown
    hn, hb, hd = api.CNormalBVH.build(p, f)
    np.testing.assert_array_equal(dn.cpu().numpy(), hn)
    np.testing.assert_array_equal(db.cpu().numpy(), hb)
    assert dd == hd
    ctx.close()
