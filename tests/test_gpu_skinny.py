"""The skinny forward past 16 rows, in fp32, and over split ranges of K.

Against the float64 oracle: every product is exact (x or -x), so the only
errors are fp32 sums and one output rounding.  A sum of n terms in any order
is within (n - 1) * 2^-24 * sum |x| of the exact one; the longest chain here
is the MFMAs of a wave's chunks, the 8 waves, the ranges and the limbs, under
K / 8 + 64 additions (an MFMA adds 32 columns, internally rounded at most
that often).  fp32 outputs take scale and bias with two more roundings; 16-bit
outputs one rounding to the dtype.

Sizes sit where the kernel's layout can go wrong: row counts at the edges of
its 4-, 16-, 32-, 48- and 64-row instances, K inside a 512-column chunk and
over several chunks of a wave, N inside a block of 16 and of a workgroup,
output rows whose start is not 16-byte aligned, every number of blocks that an
instance has (one to eight up to 32 rows, to six up to 48, to four up to 64: the
largest images of the sums in LDS; K is long enough there that the call stays
off the tiles), and plans that split K (the C entry without a workspace runs the
same call unsplit)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"
CODE = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}
HALF_ULP = {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12, torch.float32: 2.0 ** -24}


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def _problem(rows, cols, m, dtype, seed):
    rng = np.random.default_rng(seed)
    packed = rng.integers(0, 256, size=(rows, cols // 8), dtype=np.uint8)
    x = torch.from_numpy(rng.standard_normal((m, cols)).astype(np.float32)).to(dtype).float().numpy()
    scale = (np.abs(rng.standard_normal(rows)) * 0.02 + 0.01).astype(np.float32)
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    return packed, x, scale, bias


def _check(got, x, packed, scale, bias, cols):
    want = oracle.linear_fwd(x, packed, scale, bias, cols)
    err = np.abs(got.double().cpu().numpy() - want)
    mag = np.abs(x).astype(np.float64).sum(axis=1)[:, None] * scale.astype(np.float64)[None, :]
    bound = (cols / 8 + 64) * 2.0 ** -24 * mag + 2.0 ** -23 * (np.abs(want) + np.abs(bias)[None, :])
    if got.dtype != torch.float32:
        bound = bound + 2 * HALF_ULP[got.dtype] * np.abs(want) + 1e-7
    assert np.all(err <= bound), np.max(err / bound)


SHAPES = [(300, 1024, 17), (4097, 896, 33), (129, 4224, 48), (1000, 8192, 49), (16, 128, 64), (9001, 640, 32),
          (4096, 14336, 24), (1026, 5120, 40), (8200, 1152, 64)]


# (blocks, rows of x): ceil(rows / 4096) blocks of 16 weight rows a workgroup
BLOCKS = [(rows, cols, m) for cols, m, most in ((2048, 1, 8), (2176, 16, 8), (4096, 32, 8), (6144, 40, 6), (8192, 64, 4))
          for rows in (4096 * n - 77 for n in range(1, most + 1))]


@pytest.mark.parametrize("rows,cols,m", BLOCKS)
def test_every_number_of_blocks(rows, cols, m):
    """bf16 and, where three limbs a row make that instance, fp32: outputs of
    weight rows at the edges of blocks and workgroups, all rows of x."""

    from qste_amd import kernels

    rng = np.random.default_rng(rows + m)
    packed = rng.integers(0, 256, size=(rows, cols // 8), dtype=np.uint8)
    scale = (rng.random(rows) * 0.02 + 0.01).astype(np.float32)
    bias = (rng.standard_normal(rows) * 0.1).astype(np.float32)
    pick = np.unique(np.concatenate([np.arange(0, rows, 997), np.arange(15, rows, 1009), np.arange(max(0, rows - 140), rows)]))
    for dtype, n in ((torch.bfloat16, m), (torch.float32, m // 3)):
        if n == 0:
            continue
        print(f"skinny {rows}x{cols} m={n} {dtype}", flush=True)
        x = torch.from_numpy(rng.standard_normal((n, cols), dtype=np.float32)).to(dtype)
        y = kernels.packed_linear_affine(x.to(DEV), torch.from_numpy(packed).to(DEV), torch.from_numpy(scale).to(DEV),
                                         torch.from_numpy(bias).to(DEV), cols)
        assert torch.isfinite(y).all()
        _check(y[:, torch.from_numpy(pick).to(DEV)], x.float().numpy(), np.ascontiguousarray(packed[pick]), scale[pick],
               bias[pick], cols)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,cols,m", SHAPES)
def test_rows_past_sixteen(rows, cols, m, dtype):
    from qste_amd import kernels

    print(f"skinny {rows}x{cols} m={m} {dtype}", flush=True)
    packed, x, scale, bias = _problem(rows, cols, m, dtype, rows + cols + m)
    tx, tp = torch.from_numpy(x).to(DEV, dtype), torch.from_numpy(packed).to(DEV)
    ts, tb = torch.from_numpy(scale).to(DEV), torch.from_numpy(bias).to(DEV)
    _check(kernels.packed_linear_affine(tx, tp, ts, tb, cols), x, packed, scale, bias, cols)
    plain = torch.empty(m, rows, dtype=dtype, device=DEV)
    rc = kernels._lib.load().qste_packed_linear_affine(
        tx.data_ptr(), CODE[dtype], tp.data_ptr(), ts.data_ptr(), tb.data_ptr(), plain.data_ptr(), m, rows, cols,
        torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    _check(plain, x, packed, scale, bias, cols)


@pytest.mark.parametrize("rows,cols,m", [(300, 1024, 1), (17, 384, 2), (2048, 2048, 5), (129, 4224, 6), (1, 640, 16),
                                         (4097, 896, 21), (1000, 8192, 11), (8192, 16384, 4)])
def test_fp32_rows(rows, cols, m):
    """fp32 x as three limbs; one row holds an infinity, whose outputs are
    infinities after the weights' signs."""

    from qste_amd import kernels

    packed, x, scale, bias = _problem(rows, cols, m, torch.float32, rows + cols + m)
    tp, ts, tb = torch.from_numpy(packed).to(DEV), torch.from_numpy(scale).to(DEV), torch.from_numpy(bias).to(DEV)
    got = kernels.packed_linear_affine(torch.from_numpy(x).to(DEV), tp, ts, tb, cols)
    _check(got, x, packed, scale, bias, cols)
    x[m - 1, cols - 3] = np.inf
    got = kernels.packed_linear_affine(torch.from_numpy(x).to(DEV), tp, ts, tb, cols).cpu().numpy()
    bit = (packed[:, (cols - 3) // 8] >> ((cols - 3) % 8)) & 1
    assert np.array_equal(got[m - 1], np.where(bit == 1, np.inf, -np.inf).astype(np.float32))
    if m > 1:
        _check(torch.from_numpy(got[:m - 1]), x[:m - 1], packed, scale, bias, cols)


# few rows with two chunks of x in LDS at a time: a wave's third chunk (past
# 8192 columns) reuses a buffer, the last chunk is cut short, and the sums of
# one and two blocks land where x rows were staged
@pytest.mark.parametrize("rows,cols,m,dtype", [(4097, 14464, 1, torch.bfloat16), (8192, 16512, 4, torch.float16),
                                               (1000, 9088, 2, torch.bfloat16), (40, 28672, 3, torch.float16),
                                               (5000, 12416, 1, torch.float32)])
def test_few_rows_over_many_chunks(rows, cols, m, dtype):
    from qste_amd import kernels

    print(f"skinny {rows}x{cols} m={m} {dtype}", flush=True)
    packed, x, scale, bias = _problem(rows, cols, m, dtype, rows + cols + m)
    pick = np.unique(np.concatenate([np.arange(0, rows, max(1, rows // 97)), np.arange(max(0, rows - 40), rows)]))
    got = kernels.packed_linear_affine(torch.from_numpy(x).to(DEV, dtype), torch.from_numpy(packed).to(DEV),
                                       torch.from_numpy(scale).to(DEV), torch.from_numpy(bias).to(DEV), cols)
    assert torch.isfinite(got).all()
    _check(got[:, torch.from_numpy(pick).to(DEV)], x, np.ascontiguousarray(packed[pick]), scale[pick], bias[pick], cols)


@pytest.mark.parametrize("rows,cols,dtype,steps", [
    (8192, 28672, torch.bfloat16, (1, 4, 5, 16)), (300, 8192, torch.float16, (1, 2, 16)),
    (14336, 4096, torch.bfloat16, (1, 3, 11, 16)), (4096, 14336, torch.float16, (17, 24, 32)),
    (1000, 8192, torch.bfloat16, (33, 40, 48)), (8192, 16384, torch.bfloat16, (49, 64)),
    (2048, 2048, torch.float32, (1, 5, 6, 11, 21)), (1000, 8192, torch.float32, (1, 2, 16, 17, 21))])
def test_a_rows_bits_do_not_depend_on_the_batch(rows, cols, dtype, steps):
    """The first row of a call is bit for bit the same however many rows come
    with it (up to 16, and inside each of the larger instances; in fp32 up to
    21): K is cut, and its chunks are added, by the layer's sizes alone."""

    from qste_amd import kernels

    g = torch.Generator(device=DEV).manual_seed(rows)
    tp = torch.randint(0, 256, (rows, cols // 8), generator=g, device=DEV, dtype=torch.uint8)
    ts = torch.rand(rows, generator=g, device=DEV) * 0.02 + 0.01
    tx = torch.randn(steps[-1], cols, generator=g, device=DEV).to(dtype)
    ys = [kernels.packed_linear_affine(tx[:m].contiguous(), tp, ts, None, cols) for m in steps]
    for m, y in zip(steps, ys):
        assert torch.equal(y, ys[-1][:m]), m


@pytest.mark.parametrize("rows,cols,m,dtype", [(50257, 768, 64, torch.float16), (32000, 256, 48, torch.float16),
                                               (16384, 320, 33, torch.bfloat16), (50257, 832, 64, torch.float16)])
def test_wide_layers_of_short_k_run_on_the_tiles(rows, cols, m, dtype):
    """An output head at up to 64 rows over few columns is faster on the tiles:
    it has the bits of the call with more rows than the skinny kernel takes."""

    from qste_amd import kernels

    g = torch.Generator(device=DEV).manual_seed(rows)
    tp = torch.randint(0, 256, (rows, cols // 8), generator=g, device=DEV, dtype=torch.uint8)
    ts = torch.rand(rows, generator=g, device=DEV) * 0.02 + 0.01
    tx = torch.randn(65, cols, generator=g, device=DEV).to(dtype)
    y = kernels.packed_linear_affine(tx[:m].contiguous(), tp, ts, None, cols)
    assert torch.equal(y, kernels.packed_linear_affine(tx, tp, ts, None, cols)[:m])


@pytest.mark.parametrize("rows,cols,m,scalar", [(50257, 128, 21, True), (50257, 65, 2, True), (50257, 768, 21, False),
                                                (2048, 256, 1, False)])
def test_fp32_rows_of_short_k_stay_scalar(rows, cols, m, scalar):
    """fp32 rows over few columns of a wide layer have the scalar kernel's bits
    (those of the call without a workspace), longer K the skinny kernel's."""

    from qste_amd import kernels

    g = torch.Generator(device=DEV).manual_seed(rows)
    tp = torch.randint(0, 256, (rows, (cols + 7) // 8), generator=g, device=DEV, dtype=torch.uint8)
    ts = torch.rand(rows, generator=g, device=DEV) * 0.02 + 0.01
    tx = torch.randn(m, cols, generator=g, device=DEV)
    y, plain = kernels.packed_linear_affine(tx, tp, ts, None, cols), torch.empty(m, rows, device=DEV)
    assert kernels._lib.load().qste_packed_linear_affine(
        tx.data_ptr(), 0, tp.data_ptr(), ts.data_ptr(), None, plain.data_ptr(), m, rows, cols,
        torch.cuda.current_stream().cuda_stream) == 0
    assert torch.equal(y, plain) == scalar
    assert torch.allclose(y, plain, rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("rows,cols,m", [(8192, 28672, 16), (1000, 8192, 64), (4096, 14336, 24)])
def test_split_plans_are_deterministic(rows, cols, m):
    """Shapes whose plan splits K: two calls agree bit for bit, and with the
    unsplit call up to fp32 summation order (at most one ulp, on few)."""

    from qste_amd import kernels

    g = torch.Generator(device=DEV).manual_seed(m)
    tp = torch.randint(0, 256, (rows, cols // 8), generator=g, device=DEV, dtype=torch.uint8)
    ts = torch.rand(rows, generator=g, device=DEV) * 0.02 + 0.01
    tx = torch.randn(m, cols, generator=g, device=DEV).to(torch.bfloat16)
    a = kernels.packed_linear_affine(tx, tp, ts, None, cols)
    assert torch.equal(a, kernels.packed_linear_affine(tx, tp, ts, None, cols))
    plain = torch.empty_like(a)
    assert kernels._lib.load().qste_packed_linear_affine(
        tx.data_ptr(), 2, tp.data_ptr(), ts.data_ptr(), None, plain.data_ptr(), m, rows, cols,
        torch.cuda.current_stream().cuda_stream) == 0
    a, plain = a.float(), plain.float()
    assert (a != plain).float().mean() < 0.01
    assert torch.all((a - plain).abs() <= plain.abs() * 2.0 ** -7 + 1e-6)
