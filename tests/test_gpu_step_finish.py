"""The one-launch end of an optimizer step: log-scales clamped, flips added.

One surface and more than one launch's 64, rows at the edges of a workgroup's
256, longer than a launch's 64 workgroups, none; NaN, infinities and the
bounds themselves; every counter, some, none.  Equal to torch's operators."""

from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("sizes,counted", [([1], 1), ([255, 256, 257], 3), ([64 * 256 + 1, 0, 5], 1), ([7] * 64, 64),
                                           ([100] * 65, 65), ([3] * 130, 66), ([40], 0)])
def test_equals_torch(sizes, counted):
    from qste_amd import kernels

    lo, hi = math.log(1e-5), math.log(10.0)
    g = torch.Generator("cuda").manual_seed(len(sizes))
    scales = [8 * torch.randn(n, device="cuda", generator=g) for n in sizes]
    special = torch.tensor([float("nan"), float("inf"), float("-inf"), lo, hi], device="cuda")
    for t in scales:
        t[:5] = special[:t.numel()]
    want = [t.clone().clamp_(lo, hi) for t in scales]
    flips = [torch.tensor(3 ** i % (1 << 40), device="cuda") for i in range(counted)]
    total = kernels.step_finish(scales, lo, hi, flips)
    for a, b in zip(scales, want):
        assert torch.equal(a.view(torch.int32), b.view(torch.int32)) or (
            torch.equal(a.isnan(), b.isnan()) and torch.equal(a[~a.isnan()], b[~b.isnan()]))
    if counted:
        assert int(total) == sum(int(f) for f in flips)


def test_others_are_left_to_torch():
    from qste_amd import kernels

    x = torch.full((4,), 9.0, device="cuda")
    for bad in (x.half(), x.cpu(), torch.nn.Parameter(x), torch.full((4, 2), 9.0, device="cuda")[:, 0]):
        assert kernels.step_finish([x, bad], 0.0, 1.0, []) is None
    assert kernels.step_finish([x], 0.0, 1.0, [torch.zeros((), device="cuda")]) is None
    assert bool((x == 9.0).all())
