"""Layers whose rows or columns are no multiple of 64, on the matrix cores.

Such 16-bit layers run their products on zero-padded copies when the
workspace has room for them.  Each is compared with the float64 oracle (the
operands rounded as the kernels' contract says) and, for the backward, with
the general kernels: the C entry given a workspace without room for the
copies.  Float outputs of the two paths differ by fp32 summation order only:
sums of n products in any two orders are within 2 n 2^-24 of each other
relative to the sum of magnitudes, about sqrt(n) below that in the 2-norm on
random data: under 1e-5 for the K <= 50304 here (evidence, fp32), and a bf16
output moves by an ulp in a few elements (1e-3 in the 2-norm).

Sizes: one past and one before multiples of 64 and 256, rows and columns that
start off 16-byte and off 4-byte boundaries, one ragged dimension at a time
and both, the vocabulary table of GPT-2, samples of no particular number, and
a plan that splits K (columns no multiple of 4 included)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"
DT = {"bf16": torch.bfloat16, "f16": torch.float16}
CODE = {"bf16": 2, "f16": 1}


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def t(a, dtype=None):
    x = torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    return x if dtype is None else x.to(dtype)


def rel(got, want):
    got, want = np.asarray(got, dtype=np.float64), np.asarray(want, dtype=np.float64)
    return float(np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-300))


def rnd(a, dt):
    return torch.from_numpy(np.asarray(a, dtype=np.float32)).to(DT[dt]).float().numpy()


def problem(rows, cols, m, dt, seed):
    rng = np.random.default_rng(seed)
    packed = oracle.pack_coordinate(rng.integers(-127, 128, size=(rows, cols)).astype(np.int8))
    x = rnd(rng.standard_normal((m, cols)), dt)
    dy = rnd(rng.standard_normal((m, rows)), dt)
    scale = (np.abs(rng.standard_normal(rows)) * 0.02 + 0.01).astype(np.float32)
    return packed, x, dy, scale, (rng.standard_normal(rows) * 0.1).astype(np.float32)


BACKWARD = [(65, 1000, 300), (1000, 65, 517), (255, 257, 129), (321, 130, 999), (130, 320, 2046), (777, 768, 64),
            (257, 254, 4100), (1025, 1023, 100), (50257, 768, 70)]


@pytest.mark.parametrize("rows,cols,m", BACKWARD)
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("need_input,with_bias", [(True, True), (True, False), (False, True)])
def test_backward(rows, cols, m, dt, need_input, with_bias):
    from qste_amd import kernels

    if rows > 50000 and (dt == "f16" or not need_input):
        pytest.skip("the largest table once, with its input gradient")
    print(f"ragged backward {rows}x{cols} m={m} {dt} {need_input} {with_bias}", flush=True)
    lib = kernels._lib.load()
    packed, x, dy, scale, _ = problem(rows, cols, m, dt, rows + cols + m)
    xbits, off, xs = oracle.pack_affine_rows(x)
    tdy, txb, to, txs, tp, ts = t(dy, DT[dt]), t(xbits), t(off), t(xs), t(packed), t(scale)
    dx, ev, gs, db = kernels.linear_backward(tdy, txb, to, txs, tp, ts, cols, need_bias=with_bias,
                                             need_input=need_input)
    rx, rev, rgs, rdb = (None if a is None else torch.empty_like(a) for a in (dx, ev, gs, db))
    # the general kernels: 16-byte rounding of what they need is far below the copies' size
    need = lib.qste_linear_backward_workspace_bytes_dtype(m, rows, cols, CODE[dt])
    copies = (m * (-(-rows // 64) * 64) * 2 if rows % 64 else 0) + (rows * (-(-cols // 128) * 16) if cols % 64 else 0)
    small = need - copies // 2
    work = torch.empty(small, dtype=torch.uint8, device=DEV)
    ptr = lambda a: None if a is None else a.data_ptr()  # noqa: E731
    rc = lib.qste_linear_backward(
        ptr(tdy), CODE[dt], ptr(txb), ptr(to), ptr(txs), ptr(tp), ptr(ts), ptr(rx), ptr(rev), ptr(rgs), ptr(rdb), m,
        rows, cols, work.data_ptr(), small, torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    torch.cuda.synchronize()
    got = [None if a is None else a.float().cpu().numpy() for a in (dx, ev, gs, db)]
    general = [None if a is None else a.float().cpu().numpy() for a in (rx, rev, rgs, rdb)]
    for a, b, bar in zip(got, general, (1e-3, 1e-5, 1e-4, 1e-5)):
        if a is not None:
            assert rel(a, b) <= bar
    idx = np.arange(rows)
    if rows * cols * m > 1 << 30:
        idx = np.sort(np.random.default_rng(0).choice(rows, 300, replace=False))
    dys = np.ascontiguousarray(dy[:, idx])
    e0 = oracle.evidence(dys, xbits, cols, rnd(xs, dt)) + oracle.offset_correction(dys, off)[:, None]
    assert rel(got[1][idx], e0 * scale[idx, None]) <= 1e-5
    assert rel(got[2][idx], oracle.row_inner(e0.astype(np.float32), np.ascontiguousarray(packed[idx]), cols)) <= 1e-4
    if with_bias:
        assert rel(got[3], dy.astype(np.float64).sum(0)) <= 1e-5
    if need_input:
        tok = np.arange(min(m, 64))
        assert rel(got[0][tok], rnd(oracle.linear_dgrad(np.ascontiguousarray(dy[tok]), packed, cols, rnd(scale, dt)),
                                    dt)) <= 1e-3


@pytest.mark.parametrize("rows,cols,m", [(1112, 3264, 128), (777, 768, 64), (1910, 320, 48)])
def test_few_samples_without_an_input_gradient_stay_on_the_general_kernels(rows, cols, m):
    """The evidence alone is a short chain there: it has the bits of the call
    without room for the copies, which the call with an input gradient has not."""

    from qste_amd import kernels

    lib = kernels._lib.load()
    packed, x, dy, scale, _ = problem(rows, cols, m, "bf16", rows + cols + m)
    xbits, off, xs = oracle.pack_affine_rows(x)
    tdy, txb, to, txs, tp, ts = t(dy, torch.bfloat16), t(xbits), t(off), t(xs), t(packed), t(scale)
    alone, both = (kernels.linear_backward(tdy, txb, to, txs, tp, ts, cols, need_bias=False, need_input=n)[1]
                   for n in (False, True))
    copies = (m * (-(-rows // 64) * 64) * 2 if rows % 64 else 0) + (rows * (-(-cols // 128) * 16) if cols % 64 else 0)
    small = lib.qste_linear_backward_workspace_bytes_dtype(m, rows, cols, 2) - copies // 2
    work, general, gs = torch.empty(small, dtype=torch.uint8, device=DEV), torch.empty_like(alone), torch.empty_like(ts)
    assert lib.qste_linear_backward(
        tdy.data_ptr(), 2, txb.data_ptr(), to.data_ptr(), txs.data_ptr(), tp.data_ptr(), ts.data_ptr(), None,
        general.data_ptr(), gs.data_ptr(), None, m, rows, cols, work.data_ptr(), small,
        torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(alone, general)
    assert not torch.equal(both, general)


@pytest.mark.parametrize("rows,cols,m", [(300, 65, 5), (300, 100, 64), (1000, 777, 65), (129, 4161, 1), (65, 130, 300),
                                         (4097, 1000, 33), (256, 192, 16), (1000, 8001, 70), (50257, 767, 20)])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_forward(rows, cols, m, dt):
    from qste_amd import kernels

    packed, x, _, scale, bias = problem(rows, cols, m, dt, rows + cols + m)
    got = kernels.packed_linear_affine(t(x, DT[dt]), t(packed), t(scale), t(bias), cols).float().cpu().numpy()
    plain = torch.empty(m, rows, dtype=DT[dt], device=DEV)
    tx, tp, ts, tb = t(x, DT[dt]), t(packed), t(scale), t(bias)
    assert kernels._lib.load().qste_packed_linear_affine(
        tx.data_ptr(), CODE[dt], tp.data_ptr(), ts.data_ptr(), tb.data_ptr(), plain.data_ptr(), m, rows, cols,
        torch.cuda.current_stream().cuda_stream) == 0
    want = rnd(oracle.linear_fwd(x, packed, scale, bias, cols), dt)
    assert rel(got, want) <= 1e-3 and np.mean(got != want) < 0.01
    assert rel(got, plain.float().cpu().numpy()) <= 1e-3


def test_offset_dot_is_taken():
    """A caller's offset sums are used with the padded copy, too."""

    from qste_amd import kernels

    rows, cols, m = 321, 500, 600
    packed, x, dy, scale, _ = problem(rows, cols, m, "bf16", 5)
    xbits, off, xs = oracle.pack_affine_rows(x)
    args = (t(dy, DT["bf16"]), t(xbits), t(off), t(xs), t(packed), t(scale), cols)
    _, ev, gs, _ = kernels.linear_backward(*args, need_bias=False)
    dot = t(oracle.offset_correction(dy, off).astype(np.float32))
    _, ev2, gs2, _ = kernels.linear_backward(*args, need_bias=False, offset_dot=dot)
    assert rel(ev2.cpu().numpy(), ev.cpu().numpy()) <= 1e-6 and rel(gs2.cpu().numpy(), gs.cpu().numpy()) <= 1e-4
    _, ev3, _, _ = kernels.linear_backward(*args, need_bias=False, offset_dot=dot + 1)
    assert rel(ev3.cpu().numpy(), ev.cpu().numpy()) > 1e-3


F32 = [(300, 300, 24), (2048, 2048, 24), (65, 1000, 700), (1000, 1001, 600), (1001, 1000, 64), (4100, 130, 130),
       (256, 256, 256), (300, 300, 1300)]


@pytest.mark.parametrize("rows,cols,m", F32)
@pytest.mark.parametrize("need_input", [True, False])
def test_fp32_layer(rows, cols, m, need_input):
    """fp32 layers of few rows, odd sizes and few output tiles (K in ranges):
    exact limb products, so only fp32 sums of up to 3 * 4100 terms and the
    scale's rounding separate them from the oracle (1e-6 in the 2-norm)."""

    from qste_amd import kernels

    print(f"fp32 {rows}x{cols} m={m}", flush=True)
    rng = np.random.default_rng(rows + cols + m)
    packed = oracle.pack_coordinate(rng.integers(-127, 128, size=(rows, cols)).astype(np.int8))
    x = rng.standard_normal((m, cols)).astype(np.float32)
    dy = rng.standard_normal((m, rows)).astype(np.float32)
    scale = (np.abs(rng.standard_normal(rows)) * 0.02 + 0.01).astype(np.float32)
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    y = kernels.packed_linear_affine(t(x), t(packed), t(scale), t(bias), cols).cpu().numpy()
    assert rel(y, oracle.linear_fwd(x, packed, scale, bias, cols)) <= 1e-6
    xbits, off, xs = oracle.pack_affine_rows(x)
    dx, ev, gs, db = kernels.linear_backward(t(dy), t(xbits), t(off), t(xs), t(packed), t(scale), cols,
                                             need_bias=True, need_input=need_input)
    e0 = oracle.evidence(dy, xbits, cols, xs) + oracle.offset_correction(dy, off)[:, None]
    assert rel(ev.cpu().numpy(), e0 * scale[:, None]) <= 1e-6
    assert rel(gs.cpu().numpy(), oracle.row_inner(e0.astype(np.float32), packed, cols)) <= 1e-4
    assert rel(db.cpu().numpy(), dy.astype(np.float64).sum(0)) <= 1e-6
    if need_input:
        assert rel(dx.cpu().numpy(), oracle.linear_dgrad(dy, packed, cols, scale)) <= 1e-6


@pytest.mark.parametrize("rows,cols,m", [(6400, 256, 257), (4097, 130, 300), (16384, 512, 64)])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
def test_input_gradient_in_ranges(rows, cols, m, dt):
    """Few dX tiles over many rows: K in ranges, combined (one rounding)."""

    from qste_amd import kernels

    packed, x, dy, scale, _ = problem(rows, cols, m, dt, rows + m)
    xbits, off, xs = oracle.pack_affine_rows(x)
    dx, _, _, _ = kernels.linear_backward(t(dy, DT[dt]), t(xbits), t(off), t(xs), t(packed), t(scale), cols,
                                          need_bias=False)
    want = rnd(oracle.linear_dgrad(dy, packed, cols, rnd(scale, dt)), dt)
    got = dx.float().cpu().numpy()
    assert rel(got, want) <= 1e-3 and np.mean(got != want) < 0.02
