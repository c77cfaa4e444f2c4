"""The work that a user of this library has it do, as cases that can be timed and compared.

A Qwen3.5 engine built on the library spends its time in the calls below: the
decode GEMVs (alone, as a layer's FFN, and as the recorded 9B step), the greedy
head, the multi-token matmul of a prefill (alone and as a recorded chunk of
layers), and, around them, the weight producer, the fp16 prefill image and the
embedding gather.  ``listed()`` names one case for each, ``draw()`` gives others
of the same ranges: any codec, odd row counts, every batch, chunks from 9
tokens.  Weights are tensor bytes written here in plain torch from the seed
(not by the library's encoders), with the value spread of N(0, 0.02) weights;
``exact()`` decodes the same bytes in float64.
"""
from __future__ import annotations

import math

import torch

from qwowl35_amd import qwen35 as q35
from qwowl35_amd import runtime as rt

TYPES = {"gf4": rt.TYPE_GF4, "gf2": rt.TYPE_GF2, "q8_0": rt.TYPE_Q8_0, "q4_k": rt.TYPE_Q4_K, "q5_k": rt.TYPE_Q5_K,
         "q6_k": rt.TYPE_Q6_K, "f16": rt.TYPE_F16}
DEV = "cuda"


# ---- the cases ---------------------------------------------------------------------------------------------------

def listed() -> list[dict]:
    return [
        # the smallest call: an attention layer's k / v projection for one token, called by itself
        {"name": "matvec_q8_0_kv_b1", "kind": "matvec", "type": "q8_0", "rows": 1024, "k": 4096, "batch": 1,
         "awq": False, "residual": False},
        # the FFN of eight layers for one token: gate/up/SwiGLU and the down projection into the residual stream
        {"name": "ffn_gf4_b1", "kind": "ffn", "type": "gf4", "emb": 4096, "ffn": 12288, "layers": 8, "batch": 1,
         "awq": True},
        # the same of a wider model in a k-quant, for five sequences; k = 17408 is longer than one round of the GEMV
        {"name": "ffn_q5_k_wide_b5", "kind": "ffn", "type": "q5_k", "emb": 5120, "ffn": 17408, "layers": 2,
         "batch": 5, "awq": False},
        # greedy decoding's head: token and logit of one row against the whole vocabulary
        {"name": "head_q6_k_b1", "kind": "head", "type": "q6_k", "vocab": 248320, "k": 4096, "batch": 1},
        # one decode step's projections of the 9B model with full logits, one sequence and eight
        {"name": "step_9b_b1", "kind": "step", "layers": 32, "vocab": 248320, "batch": 1},
        {"name": "step_9b_b8", "kind": "step", "layers": 32, "vocab": 248320, "batch": 8},
        # a prefill chunk through one period of the hybrid stack (three DeltaNet layers, one attention layer): the
        # default chunk of 128 tokens, and a prompt's short odd remainder
        {"name": "chunk_m128", "kind": "chunk", "layers": 4, "tokens": 128},
        {"name": "chunk_m37", "kind": "chunk", "layers": 4, "tokens": 37},
        # a long prompt's up projection on bf16 activations with AWQ scales, bf16 out
        {"name": "matmul_gf4_m2048", "kind": "matmul", "type": "gf4", "rows": 12288, "k": 4096, "tokens": 2048,
         "f32": False, "awq": True, "out_f32": False},
        # an output projection over a 509-token chunk, fp32 in and out
        {"name": "matmul_q8_0_m509", "kind": "matmul", "type": "q8_0", "rows": 4096, "k": 4096, "tokens": 509,
         "f32": True, "awq": False, "out_f32": True},
        # the cook: an up projection's fp32 rows into Q4_K blocks, with the AWQ column scale
        {"name": "quantize_q4_k", "kind": "quantize", "type": "q4_k", "rows": 12288, "k": 4096, "scale": True},
        # loading a Q6_K value projection for prefill: its fp16 image
        {"name": "image_q6_k", "kind": "image", "type": "q6_k", "rows": 4096, "k": 4096},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _rows_k(rng, kind: str, rows: int, lo: int, hi: int) -> tuple[int, int]:
    """Rows and a k (multiple of 256) within [lo, hi]; Q6_K rows need k % 512 == 0 and whole 16-byte segments."""
    k = 256 * _log_int(rng, lo // 256, hi // 256)
    if kind == "q6_k":
        k = max(512, k // 512 * 512)
        rows = max(8, rows // 8 * 8)
    return rows, k


def draw(rng) -> dict:
    kind = rng.choice(["matvec", "ffn", "head", "step", "chunk", "chunk", "matmul", "matmul", "matmul", "quantize",
                       "image", "gather"])
    any_type = ["gf4", "gf2", "q8_0", "q4_k", "q5_k", "q6_k"]
    flip = lambda: rng.random() < 0.5  # noqa: E731
    if kind == "matvec":
        t = rng.choice(any_type)
        rows, k = _rows_k(rng, t, _log_int(rng, 256, 16384), 1024, 17408)
        if t == "q8_0" and rng.random() < 0.2:
            k += 32 * rng.randint(1, 7)
        return {"kind": kind, "type": t, "rows": rows, "k": k, "batch": rng.randint(1, 8), "awq": flip(),
                "residual": flip()}
    if kind == "ffn":
        t = rng.choice(["gf4", "gf4", "gf2", "q8_0", "q4_k", "q5_k"])
        return {"kind": kind, "type": t, "emb": 256 * rng.randint(8, 20), "ffn": 256 * rng.randint(16, 68),
                "layers": rng.randint(1, 4), "batch": rng.randint(1, 8), "awq": flip()}
    if kind == "head":
        t = rng.choice(["q6_k", "q4_k", "gf4", "q8_0"])
        rows, k = _rows_k(rng, t, _log_int(rng, 16000, 248320), 2048, 4096)
        return {"kind": kind, "type": t, "vocab": rows, "k": k, "batch": rng.randint(1, 8)}
    if kind == "step":
        return {"kind": kind, "layers": 4 * rng.randint(1, 7), "vocab": _log_int(rng, 16000, 248320),
                "batch": rng.randint(1, 8)}
    if kind == "chunk":
        return {"kind": kind, "layers": 4, "tokens": _log_int(rng, 9, 512)}
    if kind == "matmul":
        t = rng.choice(["gf4", "gf4", "q8_0", "q8_0", "q4_k", "q5_k", "q6_k", "gf2"])
        rows, k = _rows_k(rng, t, _log_int(rng, 512, 12288), 1024, 12288)
        return {"kind": kind, "type": t, "rows": rows, "k": k, "tokens": _log_int(rng, 9, 2048), "f32": flip(),
                "awq": flip(), "out_f32": flip()}
    if kind == "quantize":
        rows, k = _rows_k(rng, rng.choice(any_type), _log_int(rng, 512, 12288), 1024, 12288)
        return {"kind": kind, "type": rng.choice([t for t in any_type if t != "q6_k" or (k % 512 == 0 and rows % 8 == 0)]),
                "rows": rows, "k": k, "scale": flip()}
    t = rng.choice(any_type)
    if kind == "image":
        rows, k = _rows_k(rng, t, _log_int(rng, 512, 12288), 1024, 12288)
        return {"kind": kind, "type": t, "rows": rows, "k": k}
    rows, k = _rows_k(rng, t, _log_int(rng, 16000, 100000), 2048, 4096)  # embedding rows of a prompt's tokens
    return {"kind": kind, "type": t, "rows": rows, "k": k, "ids": _log_int(rng, 1, 2048)}


# ---- weights: tensor bytes from the seed, and their float64 values -------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _codes(g, n: int, mean: float, std: float, lo: int, hi: int) -> torch.Tensor:
    v = torch.randn(n, generator=g, device=DEV, dtype=torch.float32)
    return v.mul_(std).add_(mean).round_().clamp_(lo, hi).to(torch.int16)


def _uniform(g, n: int, lo: float, hi: float) -> torch.Tensor:
    return torch.rand(n, generator=g, device=DEV, dtype=torch.float32).mul_(hi - lo).add_(lo)


def _e5m2_byte(v: torch.Tensor) -> torch.Tensor:
    bits = v.to(torch.float16).view(torch.int16).to(torch.int32) & 0xFFFF
    return ((bits + 0x80) >> 8) & 0xFF


def _e5m2_value(b: torch.Tensor) -> torch.Tensor:
    return (b.to(torch.int32) << 8).to(torch.int16).view(torch.float16).to(torch.float64)


def _half_bytes(v: torch.Tensor) -> torch.Tensor:
    return v.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _f16(b: torch.Tensor) -> torch.Tensor:
    """[n, 2] bytes -> [n, 1] float64 of the little-endian binary16."""
    return b.contiguous().view(torch.float16).to(torch.float64)


def _pack_scales(sc: torch.Tensor, mn: torch.Tensor) -> torch.Tensor:
    """Eight 6-bit scales and mins per super-block -> 12 bytes (get_scale_min_k4)."""
    lo = (sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6)
    mid = (mn[:, :4] & 63) | ((mn[:, 4:] >> 4) << 6)
    hi = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    return torch.cat([lo, mid, hi], dim=1).to(torch.uint8)


def _block_bytes(g, kind: str, n: int) -> torch.Tensor:
    """n weights' tensor bytes (n a multiple of the block) as flat uint8."""
    if kind == "f16":
        return torch.randn(n, generator=g, device=DEV).mul_(0.02).to(torch.float16).view(torch.uint8)
    if kind == "gf4":  # word: e5m2 scale byte, eight 3-bit codes; the group's largest weight has code -4
        m = n // 8
        c = _codes(g, n, 0.0, 1.8, -4, 3).reshape(m, 8)
        c.scatter_(1, torch.randint(0, 8, (m, 1), generator=g, device=DEV), -4)
        sign = torch.randint(0, 2, (m,), generator=g, device=DEV) * 2 - 1
        w = _e5m2_byte(_uniform(g, m, 0.02, 0.06) * sign).to(torch.int64)
        for i in range(8):
            w |= (c[:, i].to(torch.int64) & 7) << (8 + 3 * i)
        w = torch.where(w >= 1 << 31, w - (1 << 32), w)
        return w.to(torch.int32).view(torch.uint8)
    if kind == "gf2":  # 16 words of 2-bit codes, their 16 scale bytes
        m = n // 16
        c = torch.randint(0, 4, (m, 16), generator=g, device=DEV, dtype=torch.int32)
        w = torch.zeros(m, dtype=torch.int32, device=DEV)
        for i in range(16):
            w |= c[:, i] << (2 * i)
        s = _e5m2_byte(_uniform(g, m, 0.02, 0.06)).to(torch.uint8).reshape(-1, 16)
        return torch.cat([w.view(torch.uint8).reshape(-1, 64), s], dim=1).reshape(-1)
    if kind == "q8_0":
        m = n // 32
        q = _codes(g, n, 0.0, 45.0, -127, 127).to(torch.int8).view(torch.uint8).reshape(m, 32)
        return torch.cat([_half_bytes(_uniform(g, m, 0.0003, 0.0006)), q], dim=1).reshape(-1)
    m = n // 256
    if kind == "q6_k":
        q = _codes(g, n, 32.0, 11.0, 0, 63).reshape(m, 2, 4, 32)  # [super-block][h][g][l]
        ql = torch.stack([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)],
                         dim=2)
        qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
        sc = torch.randint(60, 128, (m, 16), generator=g, device=DEV, dtype=torch.int16)
        sc *= torch.randint(0, 2, (m, 16), generator=g, device=DEV, dtype=torch.int16) * 2 - 1
        d = _half_bytes(_uniform(g, m, 1.5e-5, 2.5e-5))
        return torch.cat([ql.reshape(m, 128).to(torch.uint8), qh.reshape(m, 64).to(torch.uint8),
                          sc.to(torch.int8).view(torch.uint8), d], dim=1).reshape(-1)
    top = 31 if kind == "q5_k" else 15  # q4_k and q5_k: w = d sc q - dmin m
    q = _codes(g, n, top / 2, top / 5, 0, top).reshape(m, 8, 32)
    sc = torch.randint(30, 64, (m, 8), generator=g, device=DEV, dtype=torch.int16)
    mn = (sc + torch.randint(-4, 5, (m, 8), generator=g, device=DEV, dtype=torch.int16)).clamp_(0, 63)
    d = _uniform(g, m, 0.8, 1.2) * (0.02 / (top / 5 * 48))
    head = torch.cat([_half_bytes(d), _half_bytes(d * (top / 2)), _pack_scales(sc, mn)], dim=1)
    nib = ((q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)).reshape(m, 128).to(torch.uint8)
    if kind == "q4_k":
        return torch.cat([head, nib], dim=1).reshape(-1)
    qh = torch.zeros((m, 32), dtype=torch.int16, device=DEV)
    for j in range(8):
        qh |= (q[:, j] >> 4) << j
    return torch.cat([head, qh.to(torch.uint8), nib], dim=1).reshape(-1)


ROWS_AT_ONCE = 16384


def _raw(g, kind: str, rows: int, k: int) -> torch.Tensor:
    rb = rt.row_bytes(TYPES[kind], k)
    raw = torch.empty(rows * rb, dtype=torch.uint8, device=DEV)
    for r0 in range(0, rows, ROWS_AT_ONCE):
        n = min(ROWS_AT_ONCE, rows - r0)
        raw[r0 * rb:(r0 + n) * rb] = _block_bytes(g, kind, n * k)
    return raw


def _weight(g, kind: str, rows: int, k: int) -> rt.HipWeight:
    return rt.HipWeight.from_device(_raw(g, kind, rows, k), TYPES[kind], rows, k)


def _values(kind: str, raw: torch.Tensor) -> torch.Tensor:
    """Tensor bytes -> their weights, flat float64."""
    if kind == "f16":
        return raw.contiguous().view(torch.float16).to(torch.float64)
    if kind == "gf4":
        w = raw.contiguous().view(torch.int32).to(torch.int64) & 0xFFFFFFFF
        s = _e5m2_value(w & 0xFF) * -0.25
        c = torch.stack([(((w >> (8 + 3 * i)) & 7) ^ 4) - 4 for i in range(8)], dim=1)
        return (c.to(torch.float64) * s[:, None]).reshape(-1)
    if kind == "gf2":
        b = raw.reshape(-1, 80)
        w = b[:, :64].contiguous().view(torch.int32).reshape(-1)
        s = _e5m2_value(b[:, 64:].reshape(-1).to(torch.int32))
        c = torch.stack([(w >> (2 * i)) & 3 for i in range(16)], dim=1)
        return ((2.0 * c.to(torch.float64) - 3.0) / 3.0 * s[:, None]).reshape(-1)
    if kind == "q8_0":
        b = raw.reshape(-1, 34)
        return (_f16(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)).reshape(-1)
    if kind == "q6_k":
        b = raw.reshape(-1, 210).to(torch.int16)
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | (((qh >> 6) & 3) << 4)],
                        dim=2)
        sc = raw.reshape(-1, 210)[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
        d = _f16(raw.reshape(-1, 210)[:, 208:])
        return ((q.reshape(-1, 16, 16).to(torch.float64) - 32.0) * (sc * d)[:, :, None]).reshape(-1)
    b = raw.reshape(-1, 176 if kind == "q5_k" else 144)
    d, dmin = _f16(b[:, 0:2]), _f16(b[:, 2:4])
    s = b[:, 4:16].to(torch.int32)
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], dim=1).to(torch.float64)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], dim=1).to(torch.float64)
    nib = b[:, -128:].reshape(-1, 4, 32)
    q = torch.stack([nib & 15, nib >> 4], dim=2).reshape(-1, 8, 32)
    if kind == "q5_k":
        q = q + torch.stack([((b[:, 16:48] >> j) & 1) << 4 for j in range(8)], dim=1)
    return (q.to(torch.float64) * (d * sc)[:, :, None] - (dmin * mn)[:, :, None]).reshape(-1)


def _times(kind: str, raw: torch.Tensor, rows: int, k: int, x: torch.Tensor) -> torch.Tensor:
    """x [n, k] @ W^T in float64, some rows at a time."""
    rb = rt.row_bytes(TYPES[kind], k)
    out = torch.empty((x.shape[0], rows), dtype=torch.float64, device=DEV)
    for r0 in range(0, rows, ROWS_AT_ONCE):
        n = min(ROWS_AT_ONCE, rows - r0)
        out[:, r0:r0 + n] = x @ _values(kind, raw[r0 * rb:(r0 + n) * rb]).reshape(n, k).t()
    return out


def _normal(g, *shape, dtype=torch.float32) -> torch.Tensor:
    return torch.randn(shape, generator=g, device=DEV, dtype=torch.float32).to(dtype)


def _awq(g, k: int) -> torch.Tensor:
    return _uniform(g, k, 0.5, 2.0)


def _silu(v: torch.Tensor) -> torch.Tensor:
    return v / (1.0 + torch.exp(-v))


# ---- one set of functions per kind ---------------------------------------------------------------------------------

def _hparams(c) -> q35.Hparams:
    return q35.Hparams(transformer_layers=c["layers"], vocab=c.get("vocab", 1024))


STACK = {"mixer": "q8_0", "ffn": "gf4", "head": "q4_k"}


def _stack(c, g) -> q35.ProjectionStack:
    """Weights of every projection, each layer its own."""
    hp = _hparams(c)
    layers = []
    for il in range(hp.transformer_layers):
        ws = {p.name: _weight(g, STACK["mixer"], p.rows, p.k) for p in q35.mixer_projections(hp, il)}
        ws.update({p.name: _weight(g, STACK["ffn"], p.rows, p.k) for p in q35.ffn_projections(hp)})
        layers.append(ws)
    head = _weight(g, STACK["head"], hp.vocab, hp.embedding_length)
    return q35.ProjectionStack(hp, q35.StackTypes(), layers, head)


def _rows_of(c) -> int:
    return c["batch"] if c["kind"] == "step" else c["tokens"]


def _stack_inputs(c, seed):
    g = _gen(seed)
    stack = _stack(c, g)
    bufs = q35.StepBuffers.make(stack.hp, _rows_of(c), g, awq=False, shared_outputs=True)
    return stack, bufs


def _stack_outputs(c, bufs) -> dict:
    """The residual stream, the last layers' projections (their buffers are shared by the layers) and the logits."""
    out = {"act": bufs.act, "ffn_act": bufs.ffn_act[-1], "mixer": {}}
    for d in bufs.mixer_out:
        out["mixer"].update(d)
    if c["kind"] == "step":
        out["logits"] = bufs.logits
    return out


def _stack_exact(c, seed) -> dict:
    stack, bufs = _stack_inputs(c, seed)
    act, mixer, hid = bufs.act.double(), {}, None

    def times(w, kind, x):
        return _times(kind, w.storage, w.rows, w.k, x)

    norm, ffn_norm = bufs.norm.double(), bufs.ffn_norm.double()
    for il, ws in enumerate(stack.layers):
        mix = q35.mixer_projections(stack.hp, il)
        last = il + 4 >= len(stack.layers)  # later layers write the same buffers
        if last:
            for p in mix[:-1]:
                mixer[p.name] = times(ws[p.name], STACK["mixer"], norm)
        act += times(ws[mix[-1].name], STACK["mixer"], bufs.core[mix[-1].k].double())
        hid = _silu(times(ws["ffn_gate"], STACK["ffn"], ffn_norm)) * times(ws["ffn_up"], STACK["ffn"], ffn_norm)
        act += times(ws["ffn_down"], STACK["ffn"], hid)
    out = {"act": act, "ffn_act": hid, "mixer": mixer}
    if c["kind"] == "step":
        out["logits"] = times(stack.head, STACK["head"], norm)
    return out


def _ffn_inputs(c, seed):
    g = _gen(seed)
    e, f, t = c["emb"], c["ffn"], c["type"]
    layers = [(_weight(g, t, f, e), _weight(g, t, f, e), _weight(g, t, e, f)) for _ in range(c["layers"])]
    x, act0 = _normal(g, c["batch"], e), _normal(g, c["batch"], e)
    return layers, x, act0, _awq(g, e) if c["awq"] else None


def _matmul_inputs(c, seed):
    g = _gen(seed)
    w = _weight(g, c["type"], c["rows"], c["k"])
    a = _normal(g, c["tokens"], c["k"], dtype=torch.float32 if c["f32"] else torch.bfloat16)
    return w, a, _awq(g, c["k"]) if c["awq"] else None


def _matvec_inputs(c, seed):
    g = _gen(seed)
    w = _weight(g, c["type"], c["rows"], c["k"])
    x, base = _normal(g, c["batch"], c["k"]), _normal(g, c["batch"], c["rows"])
    return w, x, base, _awq(g, c["k"]) if c["awq"] else None


def _head_inputs(c, seed):
    g = _gen(seed)
    return _weight(g, c["type"], c["vocab"], c["k"]), _normal(g, c["batch"], c["k"])


def prepare(case: dict, seed: int) -> dict:
    c = case
    s = {"case": c}
    if c["kind"] == "matvec":
        w, x, base, awq = _matvec_inputs(c, seed)
        s.update(w=w, x=x, base=base, awq=awq, dst=torch.empty_like(base),
                 ws=rt.decode_matvec_workspace(w, c["batch"], device=DEV))
    elif c["kind"] == "ffn":
        layers, x, act0, awq = _ffn_inputs(c, seed)
        hid, act = torch.empty((c["batch"], c["ffn"]), device=DEV), torch.empty_like(act0)
        plan = rt.DecodePlan()
        for gate, up, down in layers:
            plan.swiglu(gate, up, x, hid, awq=awq)
            plan.matvec(down, hid, act, residual=True)
        s.update(plan=plan.record(), act0=act0, act=act, hid=hid)
    elif c["kind"] == "head":
        w, x = _head_inputs(c, seed)
        s.update(w=w, x=x, ws=rt.output_argmax_workspace(w, c["batch"], device=DEV))
    elif c["kind"] in ("step", "chunk"):
        stack, bufs = _stack_inputs(c, seed)
        s.update(bufs=bufs, act0=bufs.act.clone())
        if c["kind"] == "step":
            s["plan"] = q35.build_plan(stack, bufs)
        else:
            s["plan"] = q35.build_chunk_plan(stack, bufs, q35.chunk_workspace(stack, c["tokens"]), head=False)
    elif c["kind"] == "matmul":
        w, a, awq = _matmul_inputs(c, seed)
        w = w.prefill
        dt = torch.float32 if c["out_f32"] else torch.bfloat16
        s.update(w=w, a=a, awq=awq, dt=dt, ws=rt.prefill_workspace(w, c["tokens"], device=DEV),
                 dst=torch.empty((c["tokens"], c["rows"]), dtype=dt, device=DEV))
    elif c["kind"] == "quantize":
        g = _gen(seed)
        s.update(src=_normal(g, c["rows"], c["k"]).mul_(0.02), scale=_awq(g, c["k"]) if c["scale"] else None)
    else:  # image, gather
        g = _gen(seed)
        s["w"] = _weight(g, c["type"], c["rows"], c["k"])
        if c["kind"] == "gather":
            s["ids"] = torch.randint(0, c["rows"], (c["ids"],), generator=g, device=DEV, dtype=torch.int32)
    return s


def run(s: dict):
    c = s["case"]
    kind = c["kind"]
    if kind == "matvec":
        if c["residual"]:
            s["dst"].copy_(s["base"])
        return rt.decode_matvec(s["w"], s["x"], s["dst"], residual=c["residual"], awq=s["awq"], workspace=s["ws"])
    if kind == "ffn":
        s["act"].copy_(s["act0"])
        s["plan"].launch()
        return {"act": s["act"], "hid": s["hid"]}
    if kind == "head":
        token, logit = rt.output_argmax(s["w"], s["x"], workspace=s["ws"])
        return {"token": token, "logit": logit}
    if kind in ("step", "chunk"):
        s["bufs"].act.copy_(s["act0"])  # the embedding rows enter the residual stream
        s["plan"].launch()
        return _stack_outputs(c, s["bufs"])
    if kind == "matmul":
        return rt.matmul_prefill(s["w"], s["a"], awq=s["awq"], out_dtype=s["dt"], dst=s["dst"], workspace=s["ws"])
    if kind == "quantize":
        return rt.quantize(s["src"], TYPES[c["type"]], s["scale"])
    if kind == "image":
        return rt.prefill_image(s["w"]).storage
    return rt.dequantize(s["w"], s["ids"])


def exact(case: dict, seed: int):
    c = case
    if c["kind"] == "matvec":
        w, x, base, awq = _matvec_inputs(c, seed)
        y = _times(c["type"], w.storage, w.rows, w.k, x.double() * (1.0 if awq is None else awq.double()))
        return y + base.double() if c["residual"] else y
    if c["kind"] == "ffn":
        layers, x, act, awq = _ffn_inputs(c, seed)
        x, act, hid = x.double() * (1.0 if awq is None else awq.double()), act.double(), None

        def times(w, v):
            return _times(c["type"], w.storage, w.rows, w.k, v)

        for gate, up, down in layers:
            hid = _silu(times(gate, x)) * times(up, x)
            act = act + times(down, hid)
        return {"act": act, "hid": hid}
    if c["kind"] == "head":
        w, x = _head_inputs(c, seed)
        y = _times(c["type"], w.storage, w.rows, w.k, x.double())
        return {"token": y.argmax(dim=1).to(torch.int32), "logit": y.amax(dim=1)}
    if c["kind"] in ("step", "chunk"):
        return _stack_exact(c, seed)
    if c["kind"] == "matmul":
        w, a, awq = _matmul_inputs(c, seed)
        v = a.double() * (1.0 if awq is None else awq.double())
        return _times(c["type"], w.storage, w.rows, w.k, v)
    if c["kind"] == "gather":
        s = prepare(c, seed)
        rb = rt.row_bytes(TYPES[c["type"]], c["k"])
        rows = s["w"].storage.reshape(c["rows"], rb)[s["ids"].long()]
        return _values(c["type"], rows.reshape(-1)).reshape(c["ids"], c["k"])
    return None  # quantize, image: bytes


# ---- what a pass cannot do without, and how far two right answers may be apart -------------------------------------

def _weight_bytes(kind: str, rows: int, k: int) -> int:
    return rows * rt.row_bytes(TYPES[kind], k)


def work(case: dict) -> dict:
    c = case
    if c["kind"] in ("matvec", "head"):
        rows, b = c.get("rows", c.get("vocab")), c["batch"]
        out = 8 * b if c["kind"] == "head" else 4 * b * rows * (2 if c["residual"] else 1)
        extra = 4 * c["k"] if c.get("awq") else 0
        return {"bytes": _weight_bytes(c["type"], rows, c["k"]) + 4 * b * c["k"] + out + extra,
                "flops": 2 * b * rows * c["k"]}
    if c["kind"] == "ffn":
        e, f, b, n = c["emb"], c["ffn"], c["batch"], c["layers"]
        w = 2 * _weight_bytes(c["type"], f, e) + _weight_bytes(c["type"], e, f)
        return {"bytes": n * w + 4 * b * (3 * e + f) + (4 * e if c["awq"] else 0), "flops": n * 6 * b * e * f}
    if c["kind"] in ("step", "chunk"):
        hp, n = _hparams(c), _rows_of(c)
        total, flops = 0, 0
        for il in range(hp.transformer_layers):
            for p in q35.mixer_projections(hp, il):
                total += _weight_bytes(STACK["mixer"], p.rows, p.k)
                flops += 2 * n * p.rows * p.k
            for p in q35.ffn_projections(hp):
                total += _weight_bytes(STACK["ffn"], p.rows, p.k)
                flops += 2 * n * p.rows * p.k
        mix = sum(p.rows for il in (0, 3) for p in q35.mixer_projections(hp, il)[:-1])
        total += 4 * n * (5 * hp.embedding_length + hp.feed_forward_length + mix)
        if c["kind"] == "step":
            total += _weight_bytes(STACK["head"], hp.vocab, hp.embedding_length) + 4 * n * hp.vocab
            flops += 2 * n * hp.vocab * hp.embedding_length
        return {"bytes": total, "flops": flops}
    if c["kind"] == "matmul":
        n, rows, k = c["tokens"], c["rows"], c["k"]
        kind = c["type"] if c["type"] in ("gf4", "q8_0", "q4_k") else "f16"  # the others run on their fp16 image
        return {"bytes": _weight_bytes(kind, rows, k) + n * k * (4 if c["f32"] else 2) + n * rows * (4 if c["out_f32"] else 2),
                "flops": 2 * n * rows * k}
    if c["kind"] == "quantize":
        return {"bytes": 4 * c["rows"] * c["k"] + _weight_bytes(c["type"], c["rows"], c["k"]), "flops": 0}
    if c["kind"] == "image":
        return {"bytes": _weight_bytes(c["type"], c["rows"], c["k"]) + 2 * c["rows"] * c["k"], "flops": 0}
    return {"bytes": _weight_bytes(c["type"], c["ids"], c["k"]) + 4 * c["ids"] * c["k"], "flops": 0}


def tolerance(case: dict):
    c = case
    if c["kind"] in ("quantize", "image", "gather"):
        return "exact"
    if c["kind"] == "matmul":
        if not c["out_f32"]:
            return {"rel": 7e-3, "max": 3e-2}  # one rounding to bf16
        # fp32 sums of fp16 hi/lo pairs; bf16 activations with AWQ are rounded once to fp16, as is a k-quant's image
        rough = (not c["f32"] and c["awq"]) or c["type"] in ("q8_0", "q4_k", "q5_k", "q6_k", "gf2")
        return {"rel": 9e-4, "max": 1e-2} if rough else {"rel": 4e-6, "max": 1e-4}
    if c["kind"] == "chunk":
        return {"rel": 9e-4, "max": 1e-2}  # q8_0 weights as fp16(d q)
    # decode: GF4's biased codes at batch 1 and 2 cost seven bits of the fp32 sums; the others are plain fp32 sums
    gf4 = c["kind"] == "step" or c["type"] == "gf4"
    return {"rel": 1e-4, "max": 3e-3} if gf4 else {"rel": 4e-6, "max": 1e-4}
