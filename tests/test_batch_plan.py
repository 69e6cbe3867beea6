"""Which kernel a batched matvec takes (frq_gemv_batch_plan), on the CPU."""

from __future__ import annotations

import pytest

from flatrun_amd import FrqError, device


@pytest.mark.parametrize("q,n,k,rows,route,tile", [
    ("Q4_K", 3584, 18944, 2, "small", 0), ("Q4_K", 4096, 4096, 33, "gemm", 0), ("Q4_K", 4096, 14336, 16, "few", 32),
    ("Q4_K", 18944, 3584, 333, "pair", 128), ("Q5_K", 14336, 4096, 2, "rows", 0), ("Q5_K", 14336, 4096, 97, "pair", 64),
    ("Q6_K", 4096, 14336, 16, "pair", 32), ("Q8_0", 4096, 4096, 512, "gemm", 0), ("Q1_0", 8192, 4096, 16, "few", 32),
    ("Q1_0", 2048, 2048, 4, "rows", 0), ("Q1_0", 4096, 4096, 4, "rows", 0), ("Q1_0", 2048, 2048, 5, "few", 32),
    ("Q1_0", 1024, 1024, 4, "few", 32), ("Q1_0", 4097, 4096, 4, "few", 32), ("Q1_0", 896, 4864, 4, "few", 32),
    ("Q1_0", 2048, 2176, 4, "few", 32),
])
def test_routes(q, n, k, rows, route, tile):
    got = device.batch_plan(q, n, k, rows)
    assert got[:2] == (route, tile)
    assert (got[3] > 0) == (route in ("pair", "few"))


@pytest.mark.parametrize("args", [("Q4_K", 0, 256, 2), ("Q4_K", 4, 250, 2), ("Q4_K", 4, 256, 1), ("Q1_0", 4, 64, 2)])
def test_refused_shapes(args):
    with pytest.raises(FrqError):
        device.batch_plan(*args)
