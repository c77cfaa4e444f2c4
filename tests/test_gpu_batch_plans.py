"""The batch 3..8 GEMV plans at the edges where the row-tile count per workgroup
or the wave count changes: 256 / 512 / 768 / 1024 row tiles of 16, 8 / 12 / 16 /
24 chunks of 256 columns, and the K split of longer rows.  Each output against
an fp64 product of the library's dequantised weights (bit-exact against the
oracle in the other tests) within 1e-6 relative L2 plus, for GF2's thirds and
the fp16 hi/lo activations, their 2^-22: 2e-6."""
from __future__ import annotations

import pytest

pytestmark = pytest.mark.gpu

TYPES = {"gf4": 100, "gf2": 101, "q8_0": 8, "q4_k": 12, "q5_k": 13, "q6_k": 14}
# rows, k, the plan's (row tiles, waves) for a plain GEMV at batch 3..8
SHAPES = [(4096, 1536, (1, 8)), (4096, 2560, (1, 16)), (4088, 3584, (1, 16)), (1000, 5120, (1, 12)),
          (4104, 1536, (2, 8)), (4104, 2560, (2, 8)), (8192, 3584, (2, 16)), (4104, 5120, (2, 12)),
          (8200, 2560, (3, 8)), (12288, 5120, (3, 8)), (12296, 1536, (4, 8)), (12296, 5120, (4, 8))]
# q8_0, whose tiles take longer, where its plan differs
Q8_PLANS = {(4104, 1536, 3): (1, 8), (12296, 1536, 3): (1, 8), (12296, 1536, 8): (2, 8), (12288, 5120, 3): (1, 8),
            (12296, 5120, 3): (2, 12)}


def _weight(name, rows, k, seed):
    import torch

    from qwowl35_amd import runtime as rt

    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return rt.quantize_weight(torch.randn((rows, k), generator=g, device="cuda") * 0.02, TYPES[name])


def _close(y, want):
    err = float((y.double() - want).norm() / want.norm())
    assert err <= 2e-6, err


@pytest.mark.parametrize("nb", [3, 8])
@pytest.mark.parametrize("name", list(TYPES))
@pytest.mark.parametrize("rows,k,plan", SHAPES)
def test_batch_plans(cuda, name, rows, k, plan, nb):
    import torch

    from qwowl35_amd import runtime as rt

    w = _weight(name, rows, k, rows + nb)
    kernel, args = rt.gemv_kernel(w, nb)["name"].split("<")
    if kernel != "gf4_mfma_gemv":  # (GF4 whose staged batch fits LDS runs its own kernel)
        if name == "q8_0":
            plan = Q8_PLANS.get((rows, k, nb), plan)
        assert tuple(int(v) for v in args.split(",")[2:4]) == plan, args
    x = torch.randn((nb, k), device=cuda)
    awq = torch.rand(k, device=cuda) + 0.5
    d = rt.dequantize(w).double()
    _close(rt.decode_matvec(w, x), x.double() @ d.t())
    base = torch.randn((nb, rows), device=cuda)
    y = rt.decode_matvec(w, x, dst=base.clone(), residual=True, awq=awq)
    _close(y, base.double() + (x * awq).double() @ d.t())


@pytest.mark.parametrize("nb", [4, 7])
@pytest.mark.parametrize("name", [t for t in TYPES if t != "q6_k"])
@pytest.mark.parametrize("rows,k", [(4096, 3584), (4104, 3584), (8200, 3584), (8200, 5120), (12304, 2560)])
def test_fused_batch_plans(cuda, name, rows, k, nb):
    import torch

    from qwowl35_amd import runtime as rt

    gate, up = _weight(name, rows, k, 1), _weight(name, rows, k, 2)
    x = torch.randn((nb, k), device=cuda)
    g, u = (x.double() @ rt.dequantize(w).double().t() for w in (gate, up))
    _close(rt.ffn_gate_up_swiglu(gate, up, x), g / (1 + torch.exp(-g)) * u)


@pytest.mark.parametrize("name", [t for t in TYPES if t != "q8_0"])
@pytest.mark.parametrize("rows", [4104, 6144])
def test_long_rows_split(cuda, name, rows):
    """Three tiles and two K splits in rounds (k = 13312 = 52 chunks), every replay the same bits."""
    import torch

    from qwowl35_amd import runtime as rt

    k, nb = 13312, 5
    w = _weight(name, rows, k, rows)
    plan = rt.gemv_kernel(w, nb, workspace=True)
    assert plan["workspace_bytes"] > 0
    assert plan["name"].startswith("kq_mfma_gemv_long<") and plan["name"].split(",")[2:4] == [" 3", " 12"], plan
    assert plan["grid"] == 2 * -(-rows // 48)  # two workgroups per group of three row tiles
    ws = rt.decode_matvec_workspace(w, nb, device=cuda)
    x = torch.randn((nb, k), device=cuda)
    y = rt.decode_matvec(w, x, workspace=ws)
    _close(y, x.double() @ rt.dequantize(w).double().t())
    for _ in range(3):
        assert torch.equal(rt.decode_matvec(w, x, workspace=ws), y)


@pytest.mark.parametrize("name", [t for t in TYPES if t != "q6_k"])
@pytest.mark.parametrize("rows,k", [(4104, 13312), (1000, 12288)])
def test_recorded_fused_long_rows(cuda, name, rows, k):
    """A recorded gate/up op of a shape whose plain GEMV splits K (recorded ops have a workspace)."""
    import torch

    from qwowl35_amd import runtime as rt

    nb = 5
    gate, up = _weight(name, rows, k, 1), _weight(name, rows, k, 2)
    x, y = torch.randn((nb, k), device=cuda), torch.empty((nb, rows), device=cuda)
    plan = rt.DecodePlan()
    plan.swiglu(gate, up, x, y)
    plan.record()
    plan.launch()
    rt.sync()
    assert torch.equal(y, rt.ffn_gate_up_swiglu(gate, up, x))


@pytest.mark.parametrize("nb", [3, 8])
@pytest.mark.parametrize("name", list(TYPES))
@pytest.mark.parametrize("rows,k", [(4096, 2048), (4104, 1536), (8200, 2048), (12304, 1536)])
def test_short_rows(cuda, name, rows, k, nb):
    """Rows of at most eight chunks (one per wave): the fused form, and the greedy
    head with a workspace that was sized for batch 8."""
    import torch

    from qwowl35_amd import runtime as rt

    w = _weight(name, rows, k, 1)
    x = torch.randn((nb, k), device=cuda)
    want = x.double() @ rt.dequantize(w).double().t()
    if name != "q6_k":
        up = _weight(name, rows, k, 2)
        u = x.double() @ rt.dequantize(up).double().t()
        _close(rt.ffn_gate_up_swiglu(w, up, x), want / (1 + torch.exp(-want)) * u)
    token, logit = rt.output_argmax(w, x, workspace=rt.output_argmax_workspace(w, 8))
    best = want.max(dim=1)
    assert torch.equal(token.long(), best.indices)  # (random rows: no ties within 2e-6)
    assert float((logit.double() - best.values).abs().max()) <= 2e-6 * float(want.norm(dim=1).max())


@pytest.mark.parametrize("nb", [3, 8])
@pytest.mark.parametrize("name", ["q8_0", "q4_k", "q5_k"])
@pytest.mark.parametrize("rows,k", [(4104, 6400), (8200, 6400), (12304, 7168)])
def test_fused_rounds(cuda, name, rows, k, nb):
    """Fused rows of more than 24 chunks: eight waves in rounds, the last one partly idle."""
    import torch

    from qwowl35_amd import runtime as rt

    gate, up = _weight(name, rows, k, 1), _weight(name, rows, k, 2)
    x = torch.randn((nb, k), device=cuda)
    g, u = (x.double() @ rt.dequantize(w).double().t() for w in (gate, up))
    _close(rt.ffn_gate_up_swiglu(gate, up, x), g / (1 + torch.exp(-g)) * u)


@pytest.mark.parametrize("nb", [3, 8])
@pytest.mark.parametrize("name,rows,k,plan", [
    ("gf4", 1000, 7168, (1, 8, 4)),                                      # 28 chunks in one round of eight waves
    ("gf4", 16392, 6400, (3, 8, 2)), ("q8_0", 4104, 6400, (2, 8, 2)),    # 1025 and 257 row tiles, 25 chunks
    ("q4_k", 16392, 2560, None), ("q6_k", 16408, 6656, None), ("gf2", 16392, 5120, None)])
def test_row_tile_rounds(cuda, name, rows, k, plan, nb):
    """Row counts one past a round of workgroups, rows of one and of several passes."""
    import torch

    from qwowl35_amd import runtime as rt

    w = _weight(name, rows, k, rows + nb)
    kernel, args = rt.gemv_kernel(w, nb)["name"].split("<")
    if plan and kernel != "gf4_mfma_gemv":
        assert tuple(int(v) for v in args.split(",")[2:5]) == plan, args
    x = torch.randn((nb, k), device=cuda)
    _close(rt.decode_matvec(w, x), x.double() @ rt.dequantize(w).double().t())


@pytest.mark.parametrize("nb", [1, 2, 3, 8])
@pytest.mark.parametrize("rows", [1000, 4104, 8200, 12304, 16392, 65552])
def test_gf4_head_plans(cuda, rows, nb):
    """The GF4 greedy head runs the chunked kernel at every batch and length, the GF4 GEMV its own."""
    import torch

    from qwowl35_amd import runtime as rt

    for k in (1024, 1536, 2560, 3584, 6400) if rows < 65536 else (2560,):
        w = _weight("gf4", rows, k, k)
        x = torch.randn((nb, k), device=cuda)
        want = x.double() @ rt.dequantize(w).double().t()
        token, logit = rt.output_argmax(w, x)
        best = want.max(dim=1)
        assert torch.equal(token.long(), best.indices), k
        assert float((logit.double() - best.values).abs().max()) <= 2e-6 * float(want.norm(dim=1).max())
