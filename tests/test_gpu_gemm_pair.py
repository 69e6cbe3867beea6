"""The batched matvec on pairs of fp16 values (frq_gemm_pair.hip) against the
oracle, at the sizes where its tiles, units and splits end.

Rows around the 32-, 64- and 128-row tiles, columns around the 256-column tile
(one wave, one lane short of it), rows of W from one block to several units
with a remainder in every split, each format, and what the pairs do not carry
and is computed weight by weight: rows of x with non-finite values, outputs that
hang on x far below their row's largest, weights with non-finite scales. The bound is the matvec's: 1e-5 of sum |w_j x_j| per output
and of max |y| per row (conftest.assert_matvec_close).
"""

from __future__ import annotations

import numpy as np
import pytest

from conftest import assert_matvec_close, bits_equal
from flatrun_amd import device, synth
from oracle import gguf_np as G

pytestmark = pytest.mark.gpu


def run(q, raw, xs, n, k):
    b = xs.shape[0]
    w, xd = device.DeviceBuffer.from_host(raw), device.DeviceBuffer.from_host(xs)
    yd = device.DeviceBuffer.from_host(np.full(b * n, np.nan, np.float32))
    try:
        device.gemv(q, w, xd, yd, n, k, batch=b)
        device.synchronize()
        return yd.to_host(np.float32).reshape(b, n)
    finally:
        for d in (w, xd, yd):
            d.free()


def check(q, raw, xs, n, k, y, what):
    y64, a64 = G.matmul_f64(q, xs, raw, n, k), G.abs_matmul_f64(q, xs, raw, n, k)
    for r in range(xs.shape[0]):
        assert_matvec_close(y[r], y64[r], a64[r], what=f"{what} row {r}")


@pytest.mark.parametrize("q,n,k,rows", [
    ("Q5_K", 1, 256, 4), ("Q5_K", 255, 512, 31), ("Q5_K", 257, 1280, 32), ("Q5_K", 289, 768, 33),
    ("Q5_K", 300, 4352, 64), ("Q5_K", 513, 256, 65), ("Q5_K", 256, 2304, 97), ("Q5_K", 33, 20992, 7),
    ("Q5_K", 257, 1280, 16), ("Q5_K", 70, 768, 17), ("Q5_K", 2100, 2304, 15), ("Q1_0", 511, 896, 16),
    ("Q4_K", 1500, 16384, 16), ("Q4_K", 18000, 1536, 17), ("Q4_K", 9000, 2816, 9),
    ("Q1_0", 1, 128, 4), ("Q1_0", 31, 384, 5), ("Q1_0", 257, 640, 32), ("Q1_0", 300, 4224, 63),
    ("Q1_0", 256, 2048, 130), ("Q1_0", 65, 18944, 33),
    ("Q4_K", 255, 256, 65), ("Q4_K", 257, 1280, 129), ("Q4_K", 300, 2816, 100), ("Q4_K", 64, 1024, 1030),
    ("Q4_K", 1500, 16384, 7), ("Q4_K", 1500, 16384, 40), ("Q6_K", 1500, 16384, 11), ("Q6_K", 1501, 16640, 33),
    ("Q6_K", 1500, 16384, 70), ("Q6_K", 6001, 4096, 129),
])
def test_edges(frq, q, n, k, rows):
    raw = synth.make_blocks(q, n, k, seed=n + k)
    xs = synth.make_x(k, seed=rows, batch=rows)
    y = run(q, raw, xs, n, k)
    some = sorted({0, 1, 30, 31, 32, 63, 64, 95, 96, 127, 128, rows // 2, rows - 2, rows - 1} & set(range(rows)))
    check(q, raw, xs[some], n, k, y[some], f"{q} {n}x{k} rows {rows}")


@pytest.mark.parametrize("q,n,k,rows,plan", [
    # the few-row kernel: one and two row tiles, ragged rows of W, an odd number
    # of Q1_0 blocks, k unsplit (results stored directly), all of its LDS (eight
    # units of Q4_K and Q5_K), more units than it has loads in flight
    ("Q1_0", 8192, 4096, 16, ("few", 32, 8)), ("Q1_0", 8190, 4224, 16, ("few", 32, 6)),
    ("Q1_0", 8200, 4224, 30, ("few", 32, 6)), ("Q1_0", 65551, 384, 4, ("few", 32, 1)),
    ("Q5_K", 14301, 4096, 17, ("few", 32, 4)), ("Q5_K", 14336, 4096, 32, ("few", 32, 4)),
    ("Q5_K", 65537, 512, 16, ("few", 32, 1)), ("Q5_K", 65601, 2048, 16, ("few", 32, 1)),
    ("Q4_K", 66000, 1024, 20, ("few", 32, 1)), ("Q4_K", 65600, 2048, 16, ("few", 32, 1)),
    ("Q4_K", 65601, 1280, 11, ("few", 32, 1)), ("Q5_K", 8192, 12544, 8, ("few", 32, 7)),
    # the 128-row tile, one row or column past its end, k unsplit and split
    ("Q4_K", 33000, 1024, 65, ("pair", 128, 1)), ("Q4_K", 20001, 768, 300, ("pair", 128, 1)),
    ("Q4_K", 18945, 1280, 257, ("pair", 128, 1)), ("Q4_K", 18945, 3584, 200, ("pair", 128, 3)),
    ("Q4_K", 33001, 1792, 66, ("pair", 128, 1)), ("Q6_K", 62765, 1024, 383, ("pair", 64, 1)),
    # rows of x in two and three registers' worth of pieces, and too long for them
    ("Q6_K", 3001, 8192, 33, ("pair", 64, 16)), ("Q6_K", 1500, 20480, 40, ("pair", 64, 40)),
    ("Q5_K", 100, 24832, 33, ("pair", 64, 49)), ("Q5_K", 100, 20736, 70, ("pair", 64, 41)),
    ("Q1_0", 300, 24704, 70, ("pair", 64, 49)),
])
def test_planned_edges(frq, q, n, k, rows, plan):
    assert device.batch_plan(q, n, k, rows)[:3] == plan
    raw = synth.make_blocks(q, n, k, seed=n + k)
    xs = synth.make_x(k, seed=rows, batch=rows)
    y = run(q, raw, xs, n, k)
    assert np.isfinite(y).all()
    some = np.unique(np.r_[:min(n, 260), max(0, n - 300):n, np.random.default_rng(n).choice(n, min(n, 400), replace=False)])
    part = np.ascontiguousarray(raw.reshape(n, -1)[some]).reshape(-1)
    check(q, part, xs, some.size, k, y[:, some], f"{q} {n}x{k} rows {rows}")


@pytest.mark.parametrize("q,n,k,rows", [("Q5_K", 70, 4096, 9), ("Q1_0", 70, 4096, 40), ("Q4_K", 70, 2048, 66)])
def test_rows_beyond_the_pairs(frq, q, n, k, rows):
    """Outliers from 2^14 to 2^40 above the rest, all rows tiny or huge, one inf
    and one NaN: every finite row meets the bound, the others are not finite,
    and ordinary rows keep their bits."""
    raw = synth.make_blocks(q, n, k, seed=5)
    xs = synth.make_x(k, seed=6, batch=rows)
    calm = xs.copy()
    for r, e in ((0, 14), (1, 18), (2, 24), (3, 40)):
        xs[r, 7 * r + 3] = 2.0**e
    xs[4] *= np.float32(2.0**-120)
    xs[5] *= np.float32(2.0**105)
    xs[6, 11] = np.inf
    xs[7, 12] = np.nan
    y = run(q, raw, xs, n, k)
    check(q, raw, xs[:4], n, k, y[:4], q)
    W = G.DEQUANT[q](raw, (n, k), np.float32).astype(np.float64)
    for r in (4, 5):
        x64 = xs[r].astype(np.float64)
        with np.errstate(over="ignore"):
            ok = np.abs(W @ x64) < float(np.finfo(np.float32).max) / 2
        err, bound = np.abs(y[r] - W @ x64), 1e-5 * (np.abs(W) @ np.abs(x64)) + k * 2.0**-150
        assert np.all(err[ok] <= bound[ok]), r
    assert not np.any(np.isfinite(y[6][W[:, 11] != 0])) and np.all(np.isnan(y[7]))
    assert bits_equal(y[8:], run(q, raw, calm, n, k)[8:])


def zero_weights(q, raw, n, k, keep):
    """raw with every weight zero but, in the rows `keep[i]` true, those of one
    sub-block (Q1_0: block) near the middle of the row; where that is in the row."""
    nb, b0 = k // G.BLOCK[q][1], k // G.BLOCK[q][1] // 2
    r = raw.reshape(n, nb, -1).copy()
    if q == "Q1_0":
        r[:, :b0, :2] = r[:, b0 + 1:, :2] = 0
        r[~keep, b0, :2] = 0
        return r.reshape(-1), slice(b0 * 128, b0 * 128 + 128)
    sc = slice(4, 16) if q in ("Q4_K", "Q5_K") else slice(192, 208)
    one = r[:, b0, sc].copy()
    r[:, :, sc] = 0
    if q == "Q6_K":
        r[:, b0, 197] = np.where(one[:, 5] == 0, 9, one[:, 5])     # elements 80 .. 95
        r[~keep, b0, 197] = 0
        return r.reshape(-1), slice(b0 * 256 + 80, b0 * 256 + 96)
    r[:, b0, 6] = (one[:, 2] & 63) | 1                             # sub-block 2's scale and minimum
    r[:, b0, 10] = one[:, 6] & 63
    r[~keep, b0, sc] = 0
    return r.reshape(-1), slice(b0 * 256 + 64, b0 * 256 + 96)


@pytest.mark.parametrize("q,n,k,rows,plan", [
    ("Q4_K", 8192, 4096, 16, ("few", 32, 8)), ("Q5_K", 14336, 4096, 20, ("few", 32, 4)),
    ("Q1_0", 8192, 4096, 9, ("few", 32, 8)), ("Q5_K", 65537, 512, 9, ("few", 32, 1)),
    ("Q5_K", 70, 4096, 9, ("pair", 32, 16)), ("Q6_K", 66000, 512, 11, ("pair", 32, 1)),
    ("Q4_K", 70, 2048, 66, ("pair", 64, 8)), ("Q6_K", 1500, 16384, 40, ("pair", 64, 32)),
    ("Q1_0", 65600, 512, 40, ("pair", 64, 1)), ("Q4_K", 33000, 1024, 66, ("pair", 128, 1)),
    ("Q6_K", 33000, 1024, 66, ("pair", 64, 2)),
])
def test_small_x_beside_large_on_zero_weights(frq, q, n, k, rows, plan):
    """x of a row 2^-15 to 2^-80 below its largest decide outputs whose other
    weights are all zero: the bound is componentwise, so what the row's scale
    costs them counts; dense rows of W and rows that are zero stay as they are."""
    assert device.batch_plan(q, n, k, rows)[:3] == plan
    dense = synth.make_blocks(q, n, k, seed=n + k)
    rng = np.random.default_rng(n)
    pick = np.sort(rng.choice(n, min(n, 40), replace=False))
    thin, at = zero_weights(q, dense, n, k, np.arange(n) % 3 != 0)
    raw = dense.reshape(n, -1)
    raw[pick] = thin.reshape(n, -1)[pick]
    raw = raw.reshape(-1)
    xs = synth.make_x(k, seed=rows, batch=rows)
    for r in range(rows):
        xs[r, at] *= np.float32(2.0 ** -(15 + 5 * (r % 14)))
    y = run(q, raw, xs, n, k)
    some = np.unique(np.r_[pick, rng.choice(n, min(n, 60), replace=False)])
    part = np.ascontiguousarray(raw.reshape(n, -1)[some]).reshape(-1)
    y64, a64 = G.matmul_f64(q, xs, part, some.size, k), G.abs_matmul_f64(q, xs, part, some.size, k)
    for r in range(rows):
        assert_matvec_close(y[r, some], y64[r], a64[r], what=f"{q} {n}x{k} row {r}")


@pytest.mark.parametrize("q,n,k,rows,plan", [
    ("Q4_K", 8192, 4096, 16, ("few", 32, 8)), ("Q5_K", 65537, 512, 9, ("few", 32, 1)),
    ("Q1_0", 8200, 4224, 30, ("few", 32, 6)), ("Q5_K", 300, 2048, 9, ("pair", 32, 8)),
    ("Q6_K", 66000, 512, 11, ("pair", 32, 1)), ("Q4_K", 70, 2048, 66, ("pair", 64, 8)),
    ("Q1_0", 65600, 512, 40, ("pair", 64, 1)), ("Q4_K", 33000, 1024, 66, ("pair", 128, 1)),
])
def test_scales_that_are_not_finite(frq, q, n, k, rows, plan):
    """Blocks whose scale (Q4_K, Q5_K: or minimum) is an infinity or a NaN: each
    output is the infinity or the NaN that the dequantized weights give, whether
    x has one sign, both or zeros, and the other rows of W are as without them."""
    assert device.batch_plan(q, n, k, rows)[:3] == plan
    bad = synth.make_blocks(q, n, k, seed=n).reshape(n, k // G.BLOCK[q][1], -1)
    xs = synth.make_x(k, seed=rows, batch=rows)
    xs[0::3] = np.abs(xs[0::3])
    xs[1::3] = -np.abs(xs[1::3])
    xs[2, ::2] = 0.0
    clean = run(q, bad.reshape(-1), xs, n, k)
    at = {"Q6_K": (208,), "Q1_0": (0,)}.get(q, (0, 2))
    hit = []
    for i, (off, bits) in enumerate((o, b) for o in at for b in (0x7C00, 0xFC00, 0x7E00)):
        row, blk = (7 + 41 * i) % n, (3 * i) % bad.shape[1]
        if q == "Q6_K":
            bad[row, blk, :192], bad[row, blk, 192:208] = 0, 5      # codes -32
        if q == "Q1_0":
            bad[row, blk, 2:] = 255
        bad[row, blk, off:off + 2] = (bits & 255, bits >> 8)
        hit.append(row)
    y = run(q, bad.reshape(-1), xs, n, k)
    with np.errstate(invalid="ignore"):
        want = G.matmul_f64(q, xs, np.ascontiguousarray(bad[hit]).reshape(-1), len(hit), k)
    assert np.isinf(want).any() and np.isnan(want).any() and not np.isfinite(want).all(axis=0).any()
    assert np.array_equal(y[:, hit], want.astype(np.float32), equal_nan=True)
    rest = np.setdiff1d(np.arange(n), hit)
    assert bits_equal(y[:, rest], clean[:, rest])


@pytest.mark.parametrize("q,n,k,rows,bad", [("Q5_K", 1030, 2048, 9, 9), ("Q1_0", 300, 4224, 70, 67),
                                            ("Q4_K", 70, 2048, 66, 5), ("Q6_K", 1500, 16384, 40, 6)])
def test_many_rows_weight_by_weight(frq, q, n, k, rows, bad):
    """Rows of x below the pairs' range, which are computed several at a time,
    their number one to three past a multiple of that and beyond 64."""
    raw = synth.make_blocks(q, n, k, seed=n)
    xs = synth.make_x(k, seed=rows, batch=rows)
    xs[np.random.default_rng(1).choice(rows, bad, replace=False)] *= np.float32(2.0 ** -110)
    check(q, raw, xs, n, k, run(q, raw, xs, n, k), q)


@pytest.mark.parametrize("q,n,k,rows,plan", [
    ("Q5_K", 8192, 4096, 12, ("few", 32, 8)), ("Q5_K", 11008, 3584, 24, ("few", 32, 5)), ("Q5_K", 4096, 11008, 40, ("pair", 64, 15)),
    ("Q5_K", 8192, 4096, 97, ("pair", 64, 4)), ("Q1_0", 8192, 4096, 97, ("pair", 64, 4)),
])
def test_error_no_larger_than_one_gemv_per_row(frq, q, n, k, rows, plan):
    """The formats whose rows otherwise run one GEMV each: the batch is no
    further from 64 bits (2-norms over all outputs; 4 % for the samples')."""
    assert device.batch_plan(q, n, k, rows)[:3] == plan
    raw = synth.make_blocks(q, n, k, seed=n + k)
    xs = synth.make_x(k, seed=rows, batch=rows)
    xs *= np.where(np.random.default_rng(1).random(xs.shape) < 1 / 300, 20, 1).astype(np.float32)
    y64 = G.matmul_f64(q, xs, raw, n, k)
    alone = np.stack([run(q, raw, xs[r:r + 1], n, k)[0] for r in range(rows)])
    err, err_alone = (np.linalg.norm(y - y64) for y in (run(q, raw, xs, n, k), alone))
    assert err <= 1.04 * err_alone, (err / np.linalg.norm(y64), err_alone / np.linalg.norm(y64))


def test_group_shares_the_pairs(frq):
    """A group whose matrices take both element orders (Q5_K and Q6_K / Q1_0):
    each has the bits it has alone."""
    k, rows = 1024, 70
    qs, ns = ("Q5_K", "Q1_0", "Q4_K", "Q5_K"), (300, 70, 256, 33)
    raws = [synth.make_blocks(q, n, k, seed=n) for q, n in zip(qs, ns)]
    xs = synth.make_x(k, seed=3, batch=rows)
    ws = [device.DeviceBuffer.from_host(r) for r in raws]
    xd, yd = device.DeviceBuffer.from_host(xs), device.DeviceBuffer(4 * rows * sum(ns))
    try:
        off, parts = 0, []
        for q, n, w, r in zip(qs, ns, ws, raws):
            parts.append((q, w, n, yd.ptr + 4 * off, r.nbytes))
            off += n
        device.gemv_group(parts, xd, k, batch=rows, y_stride=sum(ns))
        device.synchronize()
        y = yd.to_host(np.float32).reshape(rows, sum(ns))
    finally:
        for b in ws + [xd, yd]:
            b.free()
    off = 0
    for q, n, r in zip(qs, ns, raws):
        assert bits_equal(y[:, off:off + n], run(q, r, xs, n, k)), q
        off += n


def test_small_x_in_groups_and_graphs(frq):
    """Matrices that share the pairs of a SwiGLU-made x, with outputs that hang on
    its smallest values (k split and not): each has the bits it has alone, in a
    group and in replays of a graph, and the bound holds."""
    k, rows = 1024, 40
    specs = [("Q5_K", 300), ("Q4_K", 33000), ("Q5_K", 65600)]
    assert [device.batch_plan(q, n, k, rows)[:3] for q, n in specs] == [("pair", 64, 4), ("pair", 64, 1), ("pair", 64, 1)]
    raws, at = [], None
    for q, n in specs:
        dense = synth.make_blocks(q, n, k, seed=n)
        thin, at = zero_weights(q, dense, n, k, np.arange(n) % 2 == 0)
        raw = dense.reshape(n, -1)
        raw[::97] = thin.reshape(n, -1)[::97]
        raws.append(raw.reshape(-1))
    g, up = synth.make_x(k, seed=1, batch=rows) * 20, synth.make_x(k, seed=2, batch=rows)
    xs = (g / (1 + np.exp(-g)) * up).astype(np.float32)
    xs[:, at] *= np.float32(2.0 ** -45)
    ws = [device.DeviceBuffer.from_host(r) for r in raws]
    total = sum(n for _, n in specs)
    xd, yd = device.DeviceBuffer.from_host(xs), device.DeviceBuffer(4 * rows * total)
    s = device.Stream()
    parts, off = [], 0
    for (q, n), w, r in zip(specs, ws, raws):
        parts.append((q, w, n, yd.ptr + 4 * off, r.nbytes))
        off += n
    try:
        device.gemv_group(parts, xd, k, batch=rows, y_stride=total, stream=s)
        s.synchronize()
        y = yd.to_host(np.float32).reshape(rows, total)
        with device.Graph.capture(s) as cap:
            device.gemv_group(parts, xd, k, batch=rows, y_stride=total, stream=s)
        try:
            for _ in range(3):
                device.gemv("Q4_K", ws[1], xd, yd, 33000, k, batch=7, stream=s, w_bytes=raws[1].nbytes)
                cap.launch(s)
                s.synchronize()
                assert bits_equal(yd.to_host(np.float32).reshape(rows, total), y)
        finally:
            cap.destroy()
    finally:
        for b in ws + [xd, yd]:
            b.free()
        s.destroy()
    off = 0
    for (q, n), r in zip(specs, raws):
        mine = np.ascontiguousarray(y[:, off:off + n])
        assert bits_equal(mine, run(q, r, xs, n, k)), q
        some = np.unique(np.r_[0:n:97, n - 40:n])
        check(q, np.ascontiguousarray(r.reshape(n, -1)[some]).reshape(-1), xs, some.size, k, mine[:, some], q)
        off += n
