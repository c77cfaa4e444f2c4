"""The wave-per-eight-blocks q8_0 encoder at the edges of its rounds, bit for bit
against the oracle: fewer blocks than one wave takes at a time, a count that is
not a multiple of it, more than one round of the launch's fixed grid, and rows
that are no multiple of 256 columns."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import matvec as om
from tests.helpers import awq_scales

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,k,scaled", [(1, 32, False), (3, 96, True), (37, 1120, True), (8195, 4128, True)])
def test_q8_0_blocks_bit_exact(cuda, rows, k, scaled):
    import torch

    from qwowl35_amd import runtime as rt

    rng = np.random.default_rng(rows)
    w = (rng.standard_normal((rows, k)) * 0.02 * np.exp2(rng.uniform(-12, 6, (rows, 1)))).astype(np.float32)
    w[0, :32] = 0.0 if rows > 1 else w[0, :32]
    w[-1, -32:] = np.arange(32) - 15.5
    w[-1, -1] = 127.0  # d = 1 without a scale: quotients on halves
    s = awq_scales(rng, k) if scaled else None
    got = rt.quantize(torch.from_numpy(w).to(cuda), om.TYPE_Q8_0,
                      col_scale=torch.from_numpy(s).to(cuda) if scaled else None).cpu().numpy()
    v = (w * s[None, :]).astype(np.float32) if scaled else w
    want = np.asarray(om.quantize(om.TYPE_Q8_0, v)).view(np.uint8)
    assert np.array_equal(got.reshape(rows, -1), want.reshape(rows, -1))
