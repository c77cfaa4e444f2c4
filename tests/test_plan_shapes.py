"""Every shape that the GEMV entry points accept names a launch.

The launch planner picks a kernel by codec, batch, row tiles and 256-column
chunks; a plan without an instantiation is an error of the call (and of
recording a decode plan, whose ops are described with a K-split workspace).
qw35_hip_gemv_kernel describes the launch without a GPU, so this walks both
sides of every bound of the planner: plain and fused, with and without a
workspace."""
from __future__ import annotations

import ctypes as C

import pytest

from qwowl35_amd import _ffi
from tests.test_plan_coverage import GF2, GF4, Q4K, Q5K, Q6K, Q8, ROW_BYTES, kernel

# row tiles of 16 on both sides of 256, 384, 512, 768, 1280 and 4096, ragged last tiles among them
ROWS = [16, 1000, 4096, 4104, 6144, 6152, 8192, 8200, 12288, 12296, 17408, 20488, 65536, 65552]
CHUNKS = [1, 2, 4, 6, 8, 10, 12, 14, 16, 18, 24, 26, 32, 34, 48, 50, 52, 64, 68, 96, 98, 256]


@pytest.fixture(scope="module")
def lib():
    return _ffi.load()


@pytest.mark.parametrize("type_id", [GF4, GF2, Q8, Q4K, Q5K, Q6K])
@pytest.mark.parametrize("ws", [False, True])
@pytest.mark.parametrize("swiglu", [False, True])
def test_every_shape_has_a_launch(lib, type_id, swiglu, ws):
    if swiglu and type_id == Q6K:
        pytest.skip("no fused q6_k")
    for rows in ROWS:
        for chunks in CHUNKS:  # (even counts: q6_k takes k % 512 == 0)
            if type_id == Q6K and chunks % 2:
                continue
            for nb in range(1, 9):
                assert kernel(type_id, rows, 256 * chunks, nb, swiglu=swiglu, ws=ws), (rows, chunks, nb)


@pytest.mark.parametrize("type_id", [GF4, GF2, Q8, Q4K, Q5K, Q6K])
@pytest.mark.parametrize("rows,k", [(151936, 1024), (151936, 2048), (32000, 2048), (32000, 4096), (65552, 2048),
                                    (20488, 2560), (151936, 5120), (100000, 6144)])
def test_head_workspace_serves_smaller_batches(lib, type_id, rows, k):
    """A workspace sized for some batch is accepted by calls of every smaller
    one (the size is what the call asks for or more, and never falls)."""
    w = _ffi.Weight()
    w.data, w.k, w.rows, w.type_id, w.bytes = 256, k, rows, type_id, ROW_BYTES[type_id](k) * rows
    sizes = [lib.qw35_hip_output_argmax_workspace_size(C.byref(w), nb) for nb in range(1, 9)]
    assert sizes[0] > 0 and sizes == sorted(sizes), sizes
    # what a call of each batch needs: its token and logit partials, one per workgroup and batch row
    g = C.c_uint32()
    for nb in range(1, 9):
        if type_id == GF4:  # (the GF4 GEMV is another kernel than its head; covered by the sizes)
            break
        _ffi.call("qw35_hip_gemv_kernel", C.byref(w), None, nb, 0, 0, None, 0, C.byref(g), None, None, None)
        need = 2 * ((4 * nb * g.value + 255) // 256 * 256)
        assert all(size >= need for size in sizes[nb - 1:]), (nb, need, sizes)


@pytest.mark.parametrize("type_id", [GF4, GF2, Q8, Q4K, Q5K, Q6K])
@pytest.mark.parametrize("swiglu", [False, True])
def test_no_dead_chunk(lib, type_id, swiglu):
    """Batch 3..8, rows of up to 4096 columns: no chunk that every wave loads lies past the row."""
    if swiglu and type_id == Q6K:
        pytest.skip("no fused q6_k")
    for rows in ROWS:
        if rows >= 65536:  # (vocabulary-sized heads of 9..12 chunks have plans for 16)
            continue
        for chunks in (2, 4, 6, 8, 10, 12, 14, 16):
            for nb in range(3, 9):
                name = kernel(type_id, rows, 256 * chunks, nb, swiglu=swiglu)
                if name.startswith("kq_"):  # <codec, batch, row tiles, waves, chunks per wave, ...>
                    waves, per_wave = (int(v) for v in name.split("<")[1].split(",")[3:5])
                    assert (per_wave - 1) * waves < chunks, (rows, chunks, nb, name)


@pytest.mark.parametrize("type_id", [GF4, GF2, Q8, Q4K, Q5K, Q6K])
@pytest.mark.parametrize("swiglu", [False, True])
def test_no_nearly_empty_round(lib, type_id, swiglu):
    """Batch 3..8: the rounds of 256 workgroups that the row tiles of a launch
    make run at most a third more tiles one after the other than the best count
    of tiles per workgroup would (1088 row tiles: two rounds of four are eight,
    five of one are five)."""
    if swiglu and type_id == Q6K:
        pytest.skip("no fused q6_k")
    for rows in [r for r in ROWS if r < 65536] + [9728, 13824, 24576, 32000]:
        tiles = -(-rows // 16)
        serial = {rt: rt * -(-tiles // (256 * rt)) for rt in range(1, 5)}
        for chunks in (6, 12, 16, 20, 32, 68):
            for nb in range(3, 9):
                name = kernel(type_id, rows, 256 * chunks, nb, swiglu=swiglu)
                if name.startswith("kq_"):
                    rt = int(name.split("<")[1].split(",")[2])
                    assert serial[rt] <= 4 / 3 * min(serial.values()), (rows, chunks, nb, name)


@pytest.mark.parametrize("type_id", [GF4, GF2, Q8, Q4K, Q5K, Q6K])
@pytest.mark.parametrize("rows,k", [(65552, 4096), (248320, 4096), (151936, 2560), (32000, 2048)])
def test_head_workspace_tensor_serves_smaller_batches(lib, type_id, rows, k):
    """The runtime's workspace tensor also where the C ABI's size is that of one batch (vocabulary-sized heads)."""
    from qwowl35_amd import runtime as rt

    w = _ffi.Weight()
    w.data, w.k, w.rows, w.type_id, w.bytes = 256, k, rows, type_id, ROW_BYTES[type_id](k) * rows
    head = rt.HipWeight(None, w)
    for n in range(1, 9):
        numel = rt.output_argmax_workspace(head, n, device="cpu").numel()
        for nb in range(1, n + 1):
            assert numel - 256 >= lib.qw35_hip_output_argmax_workspace_size(C.byref(w), nb), (n, nb)
    for bad in (0, 9):
        with pytest.raises(_ffi.Qw35Error, match="invalid weight or batch"):
            rt.output_argmax_workspace(head, bad, device="cpu")
