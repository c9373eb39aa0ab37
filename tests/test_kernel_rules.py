"""What the kernels' entry points decide and check on the host, without a GPU: how the list of single-token attention is
divided, and operands that are refused before anything is launched."""
import ctypes
import random

import pytest


@pytest.fixture(scope="module")
def lib():
    from rustinfer_amd.kernels import build
    return build.load()


def _divide(lib, rows, max_kv_len, heads):
    """The list of ``rows`` = [(first, end)] as the kernel walks it: {row: {slot: [spans]}} and {row: slots counted}.  ``end`` is cut
    at max_kv_len, as the kernel cuts it."""
    rows = [(a, min(b, max_kv_len)) for a, b in rows]
    n = [lib.ri_attention_list_spans(a, b) for a, b in rows]
    total = sum(n)
    if not total:
        return {}, {}
    planned = len(rows) * ((max_kv_len + 31) // 32 + 1)                       # the entry point's bound of the list
    assert planned >= total and planned * 512 < 1 << 32
    waves = lib.ri_attention_list_waves(total, max(1, min(512 // heads, planned)), max_kv_len)
    begins = [sum(n[:i]) for i in range(len(n))]
    slots, counts = {}, {}
    assert lib.ri_attention_list_from(0, total, waves) == 0 and lib.ri_attention_list_from(waves, total, waves) == total
    for w in range(waves):
        f0, f1 = lib.ri_attention_list_from(w, total, waves), lib.ri_attention_list_from(w + 1, total, waves)
        assert f1 > f0
        for i, (b, m) in enumerate(zip(begins, n)):
            mine = range(max(f0, b), min(f1, b + m))
            if len(mine):
                w0 = lib.ri_attention_list_wave_of(b, total, waves)
                slots.setdefault(i, {}).setdefault(w - w0, []).extend(rows[i][0] // 32 + f - b for f in mine)
                if w == w0:
                    counts[i] = lib.ri_attention_list_wave_of(b + m - 1, total, waves) - w0 + 1
    return slots, counts


@pytest.mark.parametrize("seed", range(40))
def test_list_of_spans_holds_every_span_once_in_slots_that_are_there(lib, seed):
    rng = random.Random(seed)
    for _ in range(10):
        T, heads, window = rng.randint(1, 64), rng.choice([1, 2, 3, 8, 32, 512]), rng.choice([0, 0, 1, 33, 700])
        longest = rng.choice([1, 31, 32, 33, 64, 700, 2048, 2049, 3000, 9000])
        ends = [rng.choice([0, 1, longest, rng.randint(0, longest)]) for _ in range(T)]
        # kv_lens may say more than the step was planned for
        max_kv_len = rng.choice([longest, -(-longest // 1024) * 1024, max(1, longest // 2)])
        rows = [(max(0, e - window) if window else 0, e) for e in ends]
        slots, counts = _divide(lib, rows, max_kv_len, heads)
        assert counts.keys() == slots.keys()
        for i, (a, b) in enumerate(rows):
            b = min(b, max_kv_len)
            if b <= a:
                assert i not in slots
                continue
            got = slots[i]
            assert sorted(s for spans in got.values() for s in spans) == list(range(a // 32, (b + 31) // 32))
            assert sorted(got) == list(range(counts[i])) and counts[i] <= lib.ri_attention_list_slots(max_kv_len)


@pytest.mark.parametrize("shifted", ["k", "v", "q", "workspace"])
def test_exact_attention_refuses_operands_that_its_loads_cannot_take(lib, shifted):
    """Single tokens: values and partial results go 16 bytes at a time; portions take values from any address.  (Addresses that are never used: the check
    comes before the launch.)"""
    at = {name: ctypes.c_void_p((1 << 20) + 4 * (name == shifted)) for name in ("q", "out", "k", "v", "table", "i32", "workspace")}
    i = at["i32"]
    f, zero = ctypes.c_float(0.125), ctypes.c_void_p(0)
    H, Hkv, hd, page, T, longest = 4, 2, 64, 16, 3, 300
    lib.ri_attention_exact_decode_workspace.restype = ctypes.c_size_t
    need = lib.ri_attention_exact_decode_workspace(T, H, hd, longest)
    rc = lib.ri_attention_exact_decode_f32(at["q"], H * hd, at["out"], H * hd, at["k"], at["v"], 64, page, H, Hkv, hd, at["table"], 32, i, i, i, T, longest, f, 0,
                                           at["workspace"], ctypes.c_size_t(need), zero)
    assert rc != 0 and b"unaligned" in lib.ri_last_error()
    if shifted == "k":
        rc = lib.ri_attention_exact_f32(at["q"], H * hd, at["out"], H * hd, at["k"], at["v"], 64, page, H, Hkv, hd, at["table"], 32, i, i, i, 1, T, f, 0, zero)
        assert rc != 0 and b"unaligned" in lib.ri_last_error()


def test_exact_attention_of_single_tokens_divides_long_rows(lib):
    """A row of any length is taken by blocks of at most 64 blocks of keys in turn (a chain of some 110 us), whatever the number of rows; every slot
    has a block, and no half of the chip is left the empty ones."""
    blocks, rng = ctypes.c_int(), ctypes.c_int()
    for T in (1, 3, 16, 63, 64, 100, 128, 1000, 60000):
        for heads in (1, 2, 8, 32):
            for longest in (1, 128, 129, 500, 1024, 1025, 2048, 4096, 16000, 131072):
                lib.ri_attention_exact_split(T, heads, longest, ctypes.byref(blocks), ctypes.byref(rng))
                slots = (longest + 63) // 64 + 1
                if longest <= 128:
                    assert (blocks.value, rng.value) == (1, 0)
                    continue
                assert 1 <= rng.value <= 64 and blocks.value * rng.value >= slots and blocks.value % 2 == 1
                assert (blocks.value - 2) * rng.value < slots
                assert rng.value == 1 or T * heads * slots > 30000


@pytest.mark.parametrize("M,N,out_f32,parts", [
    (2385, 16384, 0, [(0, 2048, 0, 16384), (2048, 337, 0, 16384)]),           # rows that make whole rounds, and the rest
    (2048, 18448, 0, [(0, 2048, 0, 16384), (0, 2048, 16384, 2064)]),          # columns
    (600, 5000, 1, [(0, 600, 0, 5000)])])
def test_a_library_product_in_parts_is_asked_for_whole_where_a_part_is_refused(lib, M, N, out_f32, parts):
    """Only the whole product's refusal is the caller's: it bars the weight's size from the library for every number of rows."""
    whole = (0, M, 0, N)

    def calls(refused):
        got, count = (ctypes.c_int * 16)(), ctypes.c_int(0)
        rc = lib.ri_gemm_library_calls(M, N, out_f32, refused[1], refused[3], got, ctypes.byref(count))
        return rc, [tuple(got[4 * i:4 * i + 4]) for i in range(count.value)]

    assert calls((0, 0, 0, 0)) == (0, parts)
    if len(parts) == 2:
        assert calls(parts[1]) == (0, parts + [whole])
        assert calls(parts[0]) == (0, [parts[0], whole])
    assert calls(whole) == ((0, parts) if len(parts) == 2 else (2, [whole]))


@pytest.mark.parametrize("change,takes", [
    ({}, 1), (dict(M=1), 1), (dict(M=0), 0), (dict(M=9), 0), (dict(hd=32), 0), (dict(hd=96), 0), (dict(hd=64), 1), (dict(page=32), 0), (dict(d=2048 + 256), 0),
    (dict(d=0), 0), (dict(d=8192), 1), (dict(d=8704), 0), (dict(H=34), 0), (dict(H=24), 1), (dict(H=64), 0), (dict(H=64, Hkv=16), 1), (dict(H=68, Hkv=17), 0),
    (dict(H=32, hd=64, Hkv=2), 0), (dict(H=32, hd=64, Hkv=4), 1), (dict(ff=14336), 1), (dict(ff=14848), 0), (dict(ff=1184), 0), (dict(ff=0), 0),
    (dict(V=1000), 0), (dict(V=0), 0), (dict(Hkv=0), 0), (dict(M=8, H=64, Hkv=64, hd=64), 0)])
def test_steps_that_go_in_one_launch(lib, change, takes):
    """What the kernel holds: eight rows, whole steps of K for its eight waves, 512 outputs of a group of heads, pages of 16."""
    sizes = dict(M=8, d=2048, ff=8192, H=32, Hkv=8, hd=128, page=16, V=128256)
    sizes.update(change)
    assert lib.ri_decode_stack_takes(*sizes.values()) == takes
    assert lib.ri_decode_stack_give_control(ctypes.c_void_p(4096)) != 0           # (never taken)


@pytest.mark.parametrize("H,Hkv,hd", [(24, 8, 128), (32, 8, 64), (32, 8, 128), (40, 8, 64), (72, 9, 64), (8, 1, 64), (8, 8, 128), (36, 9, 128)])
def test_divided_rows_share_no_line_in_the_one_launch_step(lib, H, Hkv, hd):
    """A row is merged while others still write their parts, and its lines may then stay in an L2: no two slots of parts have a line in common, nor
    do outputs and sums, and all lie within the stretch."""
    from_, to, line = (ctypes.c_size_t * 2)(), (ctypes.c_size_t * 2)(), ctypes.c_size_t(0)
    for M in range(1, 9):
        for blocks in (8, 256):
            owner = {}
            for slot in range(blocks):
                lib.ri_decode_stack_slot(M, 512, 512, H, Hkv, hd, blocks, slot, from_, to, ctypes.byref(line))
                assert line.value >= 128 and to[0] - from_[0] == H // Hkv * hd * 4 and to[1] - from_[1] == H // Hkv * 8
                for kind in range(2):
                    for n in range(from_[kind] // line.value, (to[kind] - 1) // line.value + 1):
                        assert owner.setdefault(n, (slot, kind)) == (slot, kind), (M, blocks, slot, kind)


@pytest.mark.parametrize("rows,hd,keys,pays", [(1, 128, 1 << 20, True), (2, 128, 131072, True), (8, 128, 8192, True), (8, 128, 10240, True), (8, 128, 11264, False),
                                               (4, 128, 20480, True), (4, 128, 32768, False), (3, 128, 131072, False), (8, 64, 131072, True)])
def test_long_rows_leave_the_one_launch_step(rows, hd, keys, pays):
    from rustinfer_amd.kernels import ops
    assert ops.decode_stack_pays(rows, hd, keys) is pays


def test_no_control_block_is_no_error(lib):
    """Where the memory of the one-launch step's control blocks is not to be had, here as there is no device, there is no block: steps go part by part."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("there is a device")
    block, word = ctypes.c_void_p(1), ctypes.c_void_p(1)
    assert lib.ri_decode_stack_take_control(ctypes.byref(block), ctypes.byref(word)) == 0
    assert block.value is None and word.value is None
    from rustinfer_amd.engine.context import Workspace
    from rustinfer_amd.kernels import ops
    real, ops.torch.cuda.is_current_stream_capturing = ops.torch.cuda.is_current_stream_capturing, lambda: False
    try:
        ws = Workspace(torch.device("cpu"))
        assert ops.decode_stack_control(ws) is None and not ops.decode_stack_gave_up(ws)
    finally:
        ops.torch.cuda.is_current_stream_capturing = real


def test_the_library_switch_leaves_no_norm_between_products_out(monkeypatch):
    """FORCE_LIBRARY_GEMM: no fused form, of 32-bit products as of bfloat16 ones (the rotation's obeys it too)."""
    import torch
    from rustinfer_amd.kernels import ops
    w, norm = torch.zeros(256, 128), torch.ones(256)
    assert ops.linear_residual_ok(4, w, None, norm) and ops.linear_residual_ok(4, w.bfloat16(), w, norm)
    monkeypatch.setattr(ops, "FORCE_LIBRARY_GEMM", True)
    assert not ops.linear_residual_ok(4, w, None, norm) and not ops.linear_residual_ok(4, w.bfloat16(), w, norm)


@pytest.mark.parametrize("N,K,pays", [
    (2048, 2048, (1, 1, 1, 1)), (4096, 14336, (1, 1, 1, 1)), (5120, 5120, (1, 1, 1, 0)), (6144, 6144, (1, 1, 1, 0)), (5120, 13824, (0, 0, 0, 0)), (6144, 16384, (0, 0, 0, 0)),
    (6656, 6656, (0, 0, 1, 1)), (7168, 18944, (0, 0, 1, 1)), (8192, 8192, (1, 1, 1, 1)), (9216, 9216, (1, 1, 1, 0))])
def test_norms_between_32_bit_products(N, K, pays):
    """At 1, 2, 4 and 8 rows: not where the product by itself is a faster kernel by more than the norm's own takes."""
    import torch
    from rustinfer_amd.kernels import ops
    w = torch.empty(N, K, device="meta")
    assert tuple(int(ops.linear_residual_f32_pays(M, w)) for M in (1, 2, 4, 8)) == pays


@pytest.mark.parametrize("N,K", [(5120, 13824), (5120, 5120), (6144, 6144), (4608, 4608), (4096, 4096), (8192, 8192), (2048, 8192), (4224, 128)])
def test_residual_form_of_32_bit_rows_takes_the_fewer_rounds(lib, N, K):
    """Of 8 and 16 columns a block, in rounds of 256 blocks (16 columns take twice as long): never the one with the more, where they differ by a quarter."""
    for M in range(1, 9):
        parts = lib.ri_gemm_f32_residual_parts(M, N, K)
        assert parts in (N // 8, N // 16) and parts % 4 == 0
        eight, sixteen = -(-N // 8 // 256), 2 * -(-N // 16 // 256)
        if N > 4096 and 4 * eight <= 3 * sixteen:
            assert parts == N // 8


@pytest.mark.parametrize("N,K,forms", [
    # columns, values, the kernel at 1, 2, 3, 4 and 8 rows (-1: the one of FMAs): whole tiles and chunks, rows no power of two apart
    (4096, 14336, (0, 0, 0, 0, 1)), (2560, 11008, (0, 0, 0, 0, 1)), (5120, 5120, (-1, -1, 3, 3, 3)), (7168, 3584, (-1, 2, 2, 2, 2)), (8192, 3072, (0, 2, 2, 2, 2)),
    (10240, 2560, (0, 0, 0, 0, 3)), (12288, 6912, (3, 3, 3, 3, 3)), (16384, 2304, (0, 2, 2, 2, 2)), (20480, 9216, (0, 2, 2, 2, 2)), (24576, 2304, (3, 3, 3, 3, 3)),
    (24576, 2560, (-1, -1, -1, -1, 3)), (128256, 1536, (3, 3, 3, 3, 3)), (128256, 3072, (-1, -1, -1, -1, 3)),
    # remainders, and rows a power of two apart: as they were
    (5001, 2304, (-1, -1, -1, -1, 3)), (10240, 2564, (-1, -1, -1, -1, 4)), (16384, 2048, (0, 2, 2, 2, 2)), (128256, 2048, (-1, -1, -1, -1, 3)),
    # five rows and more: sixteen columns a block from 2,560 on, also where rows are 8,192 values or more apart
    (2056, 8192, (0, 0, 0, 0, 0)), (2560, 8192, (0, 0, 0, 0, 1)), (3072, 8192, (0, 0, 0, 0, 1)), (2048, 8192, (0, 0, 0, 0, 0))])
def test_kernel_of_32_bit_products_of_few_rows(lib, N, K, forms):
    assert tuple(lib.ri_gemm_f32_form(M, N, K, K) for M in (1, 2, 3, 4, 8)) == forms


@pytest.mark.parametrize("I,K,pays", [(9728, 2560, 1), (13824, 5120, 1), (18944, 3584, 1), (9216, 3072, 1), (6912, 2560, 0), (7168, 3584, 0), (2560, 3588, 0), (24576, 6144, 0),
                                      (14336, 4096, 1), (8192, 2048, 1)])
def test_swiglu_in_the_32_bit_product_of_few_rows(lib, I, K, pays):
    assert [lib.ri_gemm_f32_swiglu_pays(M, I, K, K) for M in (1, 4, 8, 9)] == [pays, pays, 1, 0]
