"""The coordinate step in several launches, where its grids change.

The passes take four rows a wave, a workgroup per CU at least and 1024 at most
(row path), strips of 4 to 64 rows and as many workgroups as there are rows or
momentum blocks (other shapes).  Rows here sit on both sides of those lines,
with blocks of 8 to 256 columns, the last chunk of a row partly empty, a step
that writes nothing, and the clip idle and engaged from step 64 on.  Bit for bit
against the oracle, flips included."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu

DEV = "cuda"
KEYS = ("coordinate", "packed", "moment_q", "moment_scale", "row_v", "col_v")


@pytest.fixture(autouse=True)
def _gpu():
    if not torch.cuda.is_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("rows,cols,block", [(3072, 768, 256), (1023, 256, 8), (1025, 768, 64), (4100, 512, 128),
                                             (16500, 256, 256), (5, 1280, 32), (300, 1000, 256), (255, 1001, 128),
                                             (1030, 72, 8), (4099, 40, 256)])
def test_matches_oracle(rows, cols, block):
    from qste_amd import kernels

    print(f"step {rows}x{cols} block {block}", flush=True)
    assert kernels._lib.load().qste_coordinate_update_one_launch(rows, cols, block) == 0
    rng = np.random.default_rng(rows + cols + block)
    state = oracle.fresh_state(rng.integers(-127, 128, size=(rows, cols)).astype(np.int8), block)
    gpu = {k: torch.from_numpy(v.copy()).to(DEV) for k, v in state.items()}
    off = torch.zeros((), dtype=torch.uint8, device=DEV)
    for step, clip, enabled in ((0, 2.0, None), (1, 2.0, off), (64, 1e6, None), (65, 0.05, None)):
        ev = (rng.standard_normal((rows, cols)) * 0.1).astype(np.float32)
        kw = dict(beta1=0.9, beta2=0.99, update_clip=clip, coordinate_lr=0.7, block_size=block, seed=3, step=step)
        flips = kernels.coordinate_update(torch.from_numpy(ev).to(DEV), *(gpu[k] for k in KEYS), update_enabled=enabled,
                                          **kw)
        want = 0 if enabled is not None else oracle.coordinate_update(ev, state, **kw)
        for k in KEYS:
            assert np.array_equal(gpu[k].cpu().numpy().view(np.uint8), state[k].view(np.uint8)), (step, k)
        assert flips == want
