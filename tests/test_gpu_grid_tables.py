"""Light-grid sampling from the per-cell tables against sampling from the SAT
itself (the oracle comparisons of both are in test_gpu_sat.py): cells of all
kinds, among them empty ones and ones whose sums are not in order or not
finite, and samples at and past the ends.  Bar: the same tile, position and
pdf bits (a NaN equals a NaN)."""
import ctypes as C

import numpy as np
import pytest
import torch

from mambatracer_amd import _lib, api

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["random", "sparse", "huge", "special"])
def test_tables_and_sat_agree(ctx, kind):
    print(f"[case] grid tables {kind}", flush=True)
    rng = np.random.default_rng(5)
    accum = rng.random((1600, 1600), dtype=np.float32)
    if kind == "sparse":  # most tiles and whole cells empty
        accum *= rng.random((1600, 1600)) < 0.01
        accum[:800] *= rng.random((800, 1600)) < 0.05
    elif kind == "huge":  # the SAT's differences round: rows out of order
        accum = np.exp(accum * 60 - 30).astype(np.float32)
    elif kind == "special":
        at = rng.random((1600, 1600)) < 0.0005
        accum[at] = rng.choice(np.float32([np.inf, np.nan, -1.0, 3e38, -0.0]), int(at.sum()))
    grid = api.CAdaptiveEnvironment(ctx)
    grid.write_accum(accum)
    grid.update()
    n = 200_003
    cell = torch.from_numpy(rng.integers(0, 5000, n).astype(np.int32)).cuda()
    u = rng.random((n, 2), dtype=np.float32)
    end = rng.random((n, 2)) < 0.02
    u[end] = rng.choice(np.float32([0.0, 1.0, 0.99999994, -0.5, 1.5, 0.5, np.nan]), int(end.sum()))
    u = torch.from_numpy(u).cuda()
    from_tables = [x.cpu().numpy() for x in grid.sample(cell, u)]
    a, f, s = C.c_void_p(), C.c_void_p(), C.c_void_p()
    _lib.call("mt_lightgrid_arrays", grid.handle, C.byref(a), C.byref(f), C.byref(s))  # the tables are not used any more
    from_sat = [x.cpu().numpy() for x in grid.sample(cell, u)]
    np.testing.assert_array_equal(from_tables[0], from_sat[0])
    for x, y in zip(from_tables[1:], from_sat[1:]):
        assert ((x.view(np.int32) == y.view(np.int32)) | (np.isnan(x) & np.isnan(y))).all()
    assert np.unique(from_sat[0][:, 1]).size == 32 and np.unique(from_sat[0][:, 0]).size == 16
