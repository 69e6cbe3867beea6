"""The 256 x 256 tile of the prefill GEMM (Q4_K products whose 256 x 128 tiles
take two rounds or more), at ragged rows and columns, the smallest k and odd
numbers of blocks: against the oracle, and bit for bit against the same rows
of W in products that the 256 x 128 tiles run (the order of sums is the same).
These are pieces of 8448 rows of W or more, which are not split over k at 257 or
more rows of x, and of 16384 at most, which one round of the smaller tiles covers
up to 512 rows of x."""

from __future__ import annotations

import numpy as np
import pytest

from conftest import bits_equal
from flatrun_amd import synth
from test_gpu_gemm import check, make_case
from test_gpu_gemm_group import run_group, single

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,ns,k", [(257, (16385, 12161), 256), (511, (28546,), 512), (512, (14336, 14336), 768),
                                    (300, (9000, 8449, 8500), 1280)])
def test_big_tile(frq, m, ns, k):
    xb = make_case(m, 1, k, seed=m)[1]
    row = k // 256 * 144
    raws = [synth.make_blocks("Q4_K", n, k, seed=n) for n in ns]
    stride = sum(ns) + 3 if len(ns) > 1 else 0
    ys = run_group([("Q4_K", raw, n) for raw, n in zip(raws, ns)], xb, m, k, y_stride=stride)
    for raw, n, y in zip(raws, ns, ys):
        # (16385 rows have no such pair of pieces: the larger overlaps the smaller)
        cuts = [(0, n)] if n <= 16384 else [(0, max(n // 2, 8448)), (n - max(n // 2, 8448), n)]
        for a, b in cuts:
            assert 8448 <= b - a <= 16384
            assert bits_equal(np.ascontiguousarray(y[:, a:b]), single("Q4_K", raw[a * row:b * row], xb, b - a, k))
        tail = n - 300
        check(np.ascontiguousarray(y[:, tail:]), raw[tail * row:], xb, 300, k)
