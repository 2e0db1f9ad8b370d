"""tanh-GELU's value from the kernel, and the tabulated bf16 kernels' edges.

The value is torch's bit for bit (every bf16 and fp16 input, normal fp32 ones),
in torch's layout.  Rows are independent, so a call large enough for the table
(4M elements) is compared, bit for bit, with the same rows in calls too small
for it: at the threshold and one row under it, for each of the three row
shapes (a wave, 256 and 1024 threads per row), with inputs inside the table's
range, outside it, infinite and NaN."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


def same(a, b):
    return torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(a[~torch.isnan(a)], b[~torch.isnan(b)])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_tanh_gelu_value(dtype):
    from qste_amd import kernels

    if dtype is torch.float32:
        x = torch.randn(1024, 4096, device="cuda", generator=torch.Generator("cuda").manual_seed(1)) * 3
    else:
        x = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(dtype).reshape(256, 256)
    want = F.gelu(x, approximate="tanh")
    out, payload, scale = kernels.smooth_activation(x, "gelu_tanh")
    assert same(out, want)
    _, given_payload, given_scale = kernels.smooth_activation(x, "gelu_tanh", output=want)
    assert torch.equal(payload, given_payload) and same(scale, given_scale)


@pytest.mark.parametrize("make", [lambda x: x.transpose(0, 1), lambda x: x.permute(2, 0, 1), lambda x: x[:, ::2],
                                  lambda x: x[..., 1:], lambda x: x[:0], lambda x: x[0, 0, 0]])
def test_tanh_gelu_layout(make):
    from qste_amd import nn as qnn

    base = torch.randn(6, 8, 40, device="cuda", dtype=torch.bfloat16)
    x, y = (make(base).detach().requires_grad_(True) for _ in range(2))
    got, want = qnn.gelu(x, "tanh"), F.gelu(y, approximate="tanh")
    assert same(got, want) and got.stride() == want.stride() and got.shape == want.shape
    g = torch.randn_like(want)
    got.backward(g)
    want.backward(g)
    assert x.numel() == 0 or float((x.grad - y.grad).abs().max()) <= 0.02 * float(y.grad.abs().max()) + 1e-6


@pytest.mark.parametrize("kind", ["gelu", "gelu_tanh", "silu"])
@pytest.mark.parametrize("rows,cols", [(4096, 1024), (4095, 1024), (1366, 3072), (1365, 3072), (5000, 840), (1022, 4104),
                                       (293, 14336), (256, 16384), (4200, 1001)])
def test_table_rows_equal_small_calls(kind, rows, cols):
    from qste_amd import kernels

    g = torch.Generator("cuda").manual_seed(rows + cols)
    x = (torch.randn(rows, cols, device="cuda", generator=g) * torch.exp(2 * torch.randn(rows, 1, device="cuda", generator=g)))
    x[3, 5], x[4, cols - 1], x[5, 0], x[6, 7], x[rows - 1, 1] = float("inf"), float("-inf"), float("nan"), 1e-30, 300.0
    x = x.bfloat16()
    out, payload, scale = kernels.smooth_activation(x, kind)
    for r0 in range(0, rows, 251):
        o, p, s = kernels.smooth_activation(x[r0:r0 + 251], kind)
        assert same(out[r0:r0 + 251], o) and torch.equal(payload[r0:r0 + 251], p) and same(scale[r0:r0 + 251], s)
