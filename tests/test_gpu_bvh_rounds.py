"""The device BVH builder's two regimes (mt_bvh.hip: rounds over the whole
order while a node has more than 256 primitives, then a work-group per
subtree) where they meet and where their windows of 512 and tiles of 2048
positions end.  Bar: node records and bounds equal to the host builder's, same depth."""
import numpy as np
import pytest
import torch

from mambatracer_amd import api

pytestmark = pytest.mark.gpu


def _mesh(kind, n):
    if kind == "soup":
        return api.gen_soup(n, n, -1, 1, 0.01, 0.3)
    p, f = api.gen_soup(n, n, -1, 1, 0.01, 0.3)
    if kind == "coincident":      # every split falls back to halving the range
        return p, np.repeat(f[:1], n, axis=0)
    # peeled: centroids at 1.9^i in runs of four, so that a split takes a few
    # primitives off one side and the tree is deep
    k = np.repeat(np.arange(n) // 4 % 120, 3)
    p[:, :3] *= 0.01
    p[:, 0] += (np.float32(1.9) ** k.astype(np.float32))
    return p, f


@pytest.mark.parametrize("kind", ["soup", "coincident", "peeled"])
@pytest.mark.parametrize("n", [255, 256, 257, 258, 511, 512, 513, 514, 515, 769, 1025, 2048, 2049, 4097, 30011])
def test_rounds_and_subtrees(ctx, kind, n):
    print(f"[case] bvh rounds {kind} n={n}", flush=True)
    p, f = _mesh(kind, n)
    hn, hb, hd = api.CNormalBVH.build(p, f)
    dn, db, dd = api.CNormalBVH.build_device(ctx, ctx.to_device(p), ctx.to_device(f))
    torch.cuda.synchronize()
    np.testing.assert_array_equal(dn.cpu().numpy(), hn)
    np.testing.assert_array_equal(db.cpu().numpy(), hb)
    assert dd == hd
