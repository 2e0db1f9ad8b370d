"""The one-launch preparation of a 16-bit backward's operands.

Its roles (column sums, transposed signs of x and W, 16-bit scales) share a
grid, so each is checked with the others present and absent: with and
without the input gradient and the bias gradient, and with the caller's
offset sums (no column sums at all).  Sizes at the edges of each role's
ranges: samples around the sums' 256-sample chunks and the transpose's
128-row tiles, rows around their 512-column workgroups, and 256 scales.
Against the float64 oracle: fp32 sums of n <= 1025 products are within n 2^-24
of it relative to the magnitudes (1e-5 in the 2-norm on random data; the
scale gradient sums the evidence over its row again, 1e-4), a 16-bit input
gradient an ulp in a few elements (1e-3)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle
from test_gpu_half_tiles import DT, rel, rnd, t

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("m,rows,cols", [(1, 64, 64), (63, 512, 128), (128, 576, 192), (129, 448, 576), (256, 64, 1024),
                                         (257, 1088, 320), (1025, 256, 512)])
@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("need_input,with_bias,given", [(True, True, False), (True, False, False),
                                                        (False, True, False), (False, False, False),
                                                        (True, False, True), (False, False, True)])
def test_roles(m, rows, cols, dt, need_input, with_bias, given):
    from qste_amd import kernels

    print(f"operands {m} {rows}x{cols} {dt} {need_input} {with_bias} {given}", flush=True)
    rng = np.random.default_rng(m + rows + cols)
    packed = oracle.pack_coordinate(rng.integers(-127, 128, size=(rows, cols)).astype(np.int8))
    dy = rnd(rng.standard_normal((m, rows)), dt)
    scale = (np.abs(rng.standard_normal(rows)) * 0.02 + 0.01).astype(np.float32)
    xbits, off, xs = oracle.pack_affine_rows(rnd(rng.standard_normal((m, cols)), dt))
    v = oracle.offset_correction(dy, off)
    if given:  # other sums than dy's own show whose are used
        v = v + 1.0
    dx, ev, gs, db = kernels.linear_backward(
        t(dy, DT[dt]), t(xbits), t(off), t(xs), t(packed), t(scale), cols, need_bias=with_bias,
        need_input=need_input, offset_dot=t(v.astype(np.float32)) if given else None)
    e0 = oracle.evidence(dy, xbits, cols, rnd(xs, dt)) + v[:, None]
    assert rel(ev.cpu().numpy(), e0 * scale[:, None]) <= 1e-5
    assert rel(gs.cpu().numpy(), oracle.row_inner(e0.astype(np.float32), packed, cols)) <= 1e-4
    assert (dx is not None) == need_input and (db is not None) == with_bias
    if with_bias:
        assert rel(db.cpu().numpy(), dy.astype(np.float64).sum(0)) <= 1e-5
    if need_input:
        want = oracle.linear_dgrad(dy, packed, cols, rnd(scale, dt))
        assert rel(dx.float().cpu().numpy(), rnd(want, dt)) <= 1e-3
