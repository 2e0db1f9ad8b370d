"""Forward and input-gradient products at the edges of 128-row tiles.

Token counts one below, at and one past 128 and 256 (more than the skinny
kernel takes), outputs one past and one before multiples of 256, odd and
off 16-byte boundaries, one K step and many, few tiles and a little more
than whole rounds of 512 half tiles.  The 16-bit input gradient runs on half
tiles inside a layer's backward only (from transposed signs), so that is
tested through ``linear_backward`` at sizes whose route says so; the product
called alone (``packed_transpose``) runs on 256-row tiles, on the general
kernel where its columns are no multiple of 64, and in fp32 as the forward
does.  Against the float64 oracle with the
operands rounded as the kernels take them: fp32 accumulation of K <= 4096
products is within K 2^-24 of it relative to the magnitudes, so an output in
the operand dtype differs by an ulp in a few elements (1e-3 in the 2-norm),
an fp32 one by 1e-5."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

DT = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BAR = {"bf16": 1e-3, "f16": 1e-3, "f32": 1e-5}


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def t(a, dtype=None):
    x = torch.from_numpy(np.ascontiguousarray(a)).to("cuda")
    return x if dtype is None else x.to(dtype)


def rnd(a, dt):
    return torch.from_numpy(np.asarray(a, dtype=np.float32)).to(DT[dt]).float().numpy()


def rel(got, want):
    got, want = np.asarray(got, dtype=np.float64), np.asarray(want, dtype=np.float64)
    return float(np.linalg.norm(got - want) / max(np.linalg.norm(want), 1e-300))


@pytest.mark.parametrize("m,rows,cols", [(127, 256, 64), (128, 255, 128), (129, 257, 64), (255, 511, 192),
                                         (257, 513, 64), (383, 1000, 256), (1531, 1023, 512), (65, 300, 4096),
                                         (130, 4097, 64), (8191, 2049, 64), (513, 30011, 64)])
@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
def test_products(m, rows, cols, dt):
    from qste_amd import kernels

    print(f"half tiles {m} x {rows} over {cols} {dt}", flush=True)
    rng = np.random.default_rng(m + rows + cols)
    packed = oracle.pack_coordinate(rng.integers(-127, 128, size=(rows, cols)).astype(np.int8))
    x = rnd(rng.standard_normal((m, cols)), dt)
    scale = (np.abs(rng.standard_normal(rows)) * 0.02 + 0.01).astype(np.float32)
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    got = kernels.packed_linear_affine(t(x, DT[dt]), t(packed), t(scale), t(bias), cols)
    # the last row and column of every tile among the rows checked
    tok = np.unique(np.concatenate([np.arange(min(m, 3)), np.arange(127, m, 128), np.arange(128, m, 128), [m - 1]]))
    want = oracle.linear_fwd(np.ascontiguousarray(x[tok]), packed, scale, bias, cols)
    assert rel(got.float().cpu().numpy()[tok], rnd(want, dt) if dt != "f32" else want) <= BAR[dt]
    assert torch.isfinite(got).all()

    # the transposed product: tokens x rows -> tokens x cols, its outputs the
    # ragged dimension above
    wt = oracle.pack_coordinate(rng.integers(-127, 128, size=(cols, rows)).astype(np.int8))
    ts = (np.abs(rng.standard_normal(cols)) * 0.02 + 0.01).astype(np.float32)
    dx = kernels.packed_transpose(t(x, DT[dt]), t(wt), rows, t(ts))
    sc = rnd(ts, dt) if dt != "f32" else ts
    want = oracle.linear_dgrad(np.ascontiguousarray(x[tok]), wt, rows, sc)
    assert rel(dx.float().cpu().numpy()[tok], rnd(want, dt) if dt != "f32" else want) <= BAR[dt]
    assert torch.isfinite(dx).all()


HALF_TILES = 4  # QSTE_ROUTE_HALF_TILES


@pytest.mark.parametrize("rows,cols,m", [(1372, 2155, 4384), (1516, 1545, 7117), (710, 1320, 7910), (1078, 1600, 4504),
                                         (1088, 1542, 4501), (768, 3072, 8184)])
@pytest.mark.parametrize("dt,with_bias", [("bf16", True), ("f16", False)])
def test_input_gradient_of_a_layer(rows, cols, m, dt, with_bias):
    """dX on half tiles: padded and unpadded rows of dy, widths odd, even, a
    multiple of 8 and of 64 (scalar, unaligned and whole stores), a partial last
    tile either way.  Tokens checked: the first and last rows of tiles; all
    columns; the evidence beside it on sampled rows."""

    from qste_amd import kernels

    lib = kernels._lib.load()
    assert lib.qste_linear_backward_route(m, rows, cols, {"bf16": 2, "f16": 1}[dt], 1) == HALF_TILES
    print(f"half tiles dX {m} x {rows} -> {cols} {dt}", flush=True)
    rng = np.random.default_rng(rows)
    packed = oracle.pack_coordinate(rng.integers(-127, 128, size=(rows, cols)).astype(np.int8))
    xbits = rng.integers(0, 256, size=(m, (cols + 7) // 8), dtype=np.uint8)
    if cols % 8:
        xbits[:, -1] &= (1 << (cols % 8)) - 1
    off, xs = (rng.standard_normal(m) * 0.1).astype(np.float32), (rng.random(m) + 0.5).astype(np.float32)
    dy = rnd(rng.standard_normal((m, rows), dtype=np.float32), dt)
    scale = (np.abs(rng.standard_normal(rows)) * 0.02 + 0.01).astype(np.float32)
    dx, ev, _, _ = kernels.linear_backward(t(dy, DT[dt]), t(xbits), t(off), t(xs), t(packed), t(scale), cols,
                                           need_bias=with_bias)
    assert torch.isfinite(dx).all()
    tok = np.unique(np.concatenate([[0, 1, 127, 128, 255, 256], np.arange(127, m, 1280), np.arange(128, m, 1280),
                                    np.arange(m // 128 * 128, m), [m - 1]]))
    tok = tok[tok < m]
    want = rnd(oracle.linear_dgrad(np.ascontiguousarray(dy[tok]), packed, cols, rnd(scale, dt)), dt)
    got = dx.float().cpu().numpy()[tok]
    assert rel(got, want) <= BAR[dt]
    for c in (0, 255, 256, cols // 256 * 256 - 1, cols // 256 * 256 - (cols % 256 == 0), cols - 1):
        assert rel(got[:, c], want[:, c]) <= 4 * BAR[dt], c
    idx = np.unique(np.concatenate([[0, 255, 256, rows - 1], rng.choice(rows, 24, replace=False)]))
    dys = np.ascontiguousarray(dy[:, idx])
    e0 = oracle.evidence(dys, xbits, cols, rnd(xs, dt)) + oracle.offset_correction(dys, off)[:, None]
    assert rel(ev.cpu().numpy()[idx], e0 * scale[idx, None]) <= 1e-5
