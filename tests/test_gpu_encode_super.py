"""The wave-per-super-block encoders (GF2, Q4_K, Q5_K, Q6_K) at the edges of
their grid, bit for bit against the oracle: fewer super-blocks than one wave
takes at a time, a count that is not a multiple of it, and more than one round
of the launch's fixed grid (2048 blocks of 4 waves of 4 super-blocks)."""
from __future__ import annotations

import numpy as np
import pytest

from oracle import matvec as om
from oracle import q6_k as oq6
from tests.helpers import awq_scales

pytestmark = pytest.mark.gpu

CODECS = {"gf2": om.TYPE_GF2, "q4_k": om.TYPE_Q4_K, "q5_k": om.TYPE_Q5_K, "q6_k": om.TYPE_Q6_K}


@pytest.mark.parametrize("name", list(CODECS))
@pytest.mark.parametrize("rows,k,scaled", [(3, 256, False), (7, 768, True), (2051, 4096, True)])
def test_super_block_encoders_bit_exact(cuda, name, rows, k, scaled):
    import torch

    from qwowl35_amd import runtime as rt

    rng = np.random.default_rng(rows)
    w = (rng.standard_normal((rows, k)) * 0.02 * np.exp2(rng.uniform(-12, 6, (rows, 1)))).astype(np.float32)
    w[0, 16:80] = 0.0
    w[1, :256] = np.abs(w[1, :256])  # no negative minimum
    w[2, :256] = -np.abs(w[2, :256])
    w[-2, -256:] = (np.arange(256) % 31 - 8) * 0.5  # quotients on and beside ties
    w[-1, -256:] = 0.0
    s = awq_scales(rng, k) if scaled else None
    got = rt.quantize(torch.from_numpy(w).to(cuda), CODECS[name],
                      col_scale=torch.from_numpy(s).to(cuda) if scaled else None)
    v = (w * s[None, :]).astype(np.float32) if scaled else w
    want = oq6.q6_k_quantize(v) if name == "q6_k" else om.quantize(CODECS[name], v)
    assert np.array_equal(got.cpu().numpy().reshape(rows, -1), np.asarray(want).reshape(rows, -1).view(np.uint8))


@pytest.mark.parametrize("name", ["q4_k", "q5_k", "q6_k"])
def test_sub_blocks_far_below_the_largest(cuda, name):
    """Sub-blocks whose range is just under 1.5 steps of the super-block's scale,
    so that scale code 1 leaves quotients far past the last code, beside ranges
    that round to scale code 0 and one that is zero throughout."""
    import torch

    from qwowl35_amd import runtime as rt

    rng = np.random.default_rng(7)
    rows, k = 8, 512
    steps = 127.0 if name == "q6_k" else 63.0
    w = rng.uniform(-1.0, 1.0, (rows, k)).astype(np.float32)
    w[:, ::16] = 1.0
    w[:, 1::16] = -1.0  # every 16- and 32-column range the same
    ratio = np.ones((rows, k), dtype=np.float32)
    ratio[:, 32:96] = 1.48 / steps
    ratio[:, 96:128] = 0.4 / steps
    ratio[:, 128:160] = 0.0
    ratio[:, 288:512] = 1.47 / steps
    v = w * ratio * np.float32(0.7)
    got = rt.quantize(torch.from_numpy(v).to(cuda), CODECS[name]).cpu().numpy().reshape(rows, -1)
    want = oq6.q6_k_quantize(v) if name == "q6_k" else om.quantize(CODECS[name], v)
    assert np.array_equal(got, np.asarray(want).reshape(rows, -1).view(np.uint8))


@pytest.mark.parametrize("name", [*CODECS, "q8_0"])
def test_groups_of_nan(cuda, name):
    """A scale group with no number in it (outside the contract, src must be
    finite): its largest magnitude is that of no elements, zero, as the NaN of a
    group beside numbers is passed over, so one such group neither spreads to
    the super-block's scale nor becomes a NaN scale itself."""
    import torch

    from qwowl35_amd import runtime as rt

    rng = np.random.default_rng(3)
    w = rng.standard_normal((4, 512)).astype(np.float32)
    w[0, 32:64] = np.nan    # whole groups of every codec (16 or 32 columns)
    w[1, 7] = np.nan        # one element
    w[2, :256] = np.nan     # a whole super-block
    zeros = w.copy()
    zeros[0, 32:64] = 0.0
    zeros[2, :256] = 0.0
    type_id = {**CODECS, "q8_0": om.TYPE_Q8_0}[name]
    got, want = (rt.quantize(torch.from_numpy(v).to(cuda), type_id).cpu().numpy().reshape(4, -1).copy()
                 for v in (w, zeros))
    if name == "q8_0":  # a scale of zero, codes of -127 (NaN * 0, clamped) where zeros have 0
        for v in (got, want):
            blocks = v.reshape(4, 16, 34)
            blocks[0, 1, 2:] = blocks[2, :8, 2:] = 0
    if name in ("q4_k", "q5_k"):  # the range of no elements is -inf, its minimum -0
        block = got[2, :got.shape[1] // 2]
        assert block[:4].tobytes() == b"\x00\xfc\x00\x80" and not block[4:].any()
        got[2], want[2] = 0, 0
    assert np.array_equal(got, want)
