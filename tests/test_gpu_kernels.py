"""Each kernel alone against a plain PyTorch 32-bit/64-bit reference of the same op, at sizes
other than the engine tests use (widths and vocabularies that are no power of two, head sizes
in steps of 16, odd head counts and groups)."""
import ctypes
import math
from types import SimpleNamespace

import numpy as np
import pytest
import torch

import plain_llama
from rustinfer_amd.engine.context import Workspace

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


@pytest.fixture(scope="module")
def ops():
    from rustinfer_amd.kernels import build, ops
    build.load()
    return ops


def rnd(*shape, dtype=torch.float32, seed=0, scale=1.0):
    g = torch.Generator().manual_seed(seed + sum(shape))
    return (torch.randn(*shape, generator=g) * scale).to(dtype).to(DEV)


def tol(dtype):
    return dict(rtol=2e-5, atol=2e-5) if dtype == torch.float32 else dict(rtol=1.6e-2, atol=1.6e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,d,V", [(1, 64, 50), (7, 200, 333), (33, 2056, 1001)])
def test_embed(ops, dtype, T, d, V):
    table = rnd(V, d, dtype=dtype)
    ids = torch.randint(0, V, (T,), dtype=torch.int32, device=DEV)
    out = torch.empty(T, d, device=DEV)
    ops.embed(ids, table, out)
    assert torch.equal(out, table[ids.long()].float())


@pytest.mark.parametrize("dtype,wdtype", [(torch.float32, torch.float32), (torch.bfloat16, torch.bfloat16),
                                          (torch.bfloat16, torch.float32)])
@pytest.mark.parametrize("T,d,eps", [(1, 64, 1e-5), (5, 200, 1e-6), (3, 4096, 1e-5), (2, 5000, 1e-3)])
def test_add_rmsnorm(ops, dtype, wdtype, T, d, eps):
    x = rnd(T, d, seed=1)
    delta = rnd(T, d, dtype=dtype, seed=2)
    w = (1 + 0.1 * rnd(d, seed=3)).to(wdtype)
    out = torch.empty(T, d, dtype=dtype, device=DEV)
    x0 = x.clone()
    ops.add_rmsnorm(x, delta, w, eps, out)
    s = x0.double() + delta.double()
    assert torch.allclose(x.double(), s, rtol=1e-6, atol=1e-6)          # residual written back in 32-bit
    ref = s * torch.rsqrt((s * s).mean(-1, keepdim=True) + eps) * w.double()
    assert torch.allclose(out.double(), ref, **tol(dtype))
    # without a delta the residual is untouched
    x1 = x.clone()
    ops.add_rmsnorm(x, None, w, eps, out)
    assert torch.equal(x, x1)
    ref = x1.double() * torch.rsqrt((x1.double() ** 2).mean(-1, keepdim=True) + eps) * w.double()
    assert torch.allclose(out.double(), ref, **tol(dtype))
    # unit weight: mean square of the output is 1 (crates/infer-backend-cpu/src/lib.rs:1317-1328)
    if dtype == torch.float32:
        ops.add_rmsnorm(x, None, torch.ones(d, device=DEV), eps, out)
        assert torch.allclose((out.double() ** 2).mean(-1), torch.ones(T, dtype=torch.float64, device=DEV), atol=1e-2)


def test_add_rmsnorm_adds_up_partial_sums(ops):
    T, d, eps = 6, 2048, 1e-5
    x = rnd(T, d, seed=40)
    parts = rnd(4, T, d, seed=41)
    w = (1 + 0.1 * rnd(d, seed=42)).to(torch.bfloat16)
    out = torch.empty(T, d, dtype=torch.bfloat16, device=DEV)
    x0 = x.clone()
    ops.add_rmsnorm(x, parts, w, eps, out)
    s = x0.double() + parts.double().sum(0)
    assert torch.allclose(x.double(), s, rtol=1e-6, atol=1e-6)
    ref = s * torch.rsqrt((s * s).mean(-1, keepdim=True) + eps) * w.double()
    assert torch.allclose(out.double(), ref, **tol(torch.bfloat16))


@pytest.mark.parametrize("M,N,K", [(1, 2048, 8192), (8, 2048, 2048), (20, 4096, 14336), (64, 160, 416), (3, 100, 72)])
def test_linear_delta_feeds_the_norm(ops, M, N, K):
    """A product with few rows and columns is split over K; the norm adds the slices up."""
    ws = Workspace(DEV)
    x = rnd(M, K, dtype=torch.bfloat16, seed=43)
    w = rnd(N, K, dtype=torch.bfloat16, seed=44, scale=0.02)
    delta = ops.linear_delta(x, w, ws, "t")
    wt = ops.tile_weight(w)
    ref = x.double() @ w.double().t()
    if wt is not None:
        tiled = ops.linear_delta(x, w, Workspace(DEV), "t", wt)
        if M <= 16:
            assert torch.equal(tiled, delta)          # the same kernel on a copy in another order
        else:                                         # 17..64 rows: another kernel, other slices of K
            assert tiled.dim() == 3 and tiled.dtype == torch.float32
            assert torch.allclose(tiled.double().sum(0), ref, rtol=0, atol=2e-6 * max(1.0, ref.abs().max().item()))
    got = delta.double().sum(0) if delta.dim() == 3 else delta.double()
    # split where columns are few and K is long; but a weight without its second copy goes to the
    # GEMM library from 17 rows on (or if it is large), which leaves whole sums in bfloat16
    to_library = M >= ops.UNTILED_LIBRARY_MIN_ROWS or N * K >= ops.UNTILED_LIBRARY_LARGE
    assert (delta.dim() == 3) == (N * 2 <= 8192 and K >= 2048 and not to_library)
    assert delta.dim() == 2 or delta.dtype == torch.float32
    assert torch.allclose(got, ref, rtol=0, atol=(2e-6 if delta.dim() == 3 else 1.6e-2) * max(1.0, ref.abs().max().item()))
    res = rnd(M, N, seed=45)
    res0 = res.clone()
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.add_rmsnorm(res, delta, torch.ones(N, device=DEV), 1e-5, out)
    s = res0.double() + got
    assert torch.allclose(out.double(), s * torch.rsqrt((s * s).mean(-1, keepdim=True) + 1e-5), **tol(torch.bfloat16))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_add_rmsnorm_selected_rows(ops, dtype):
    T, d, eps = 9, 328, 1e-5
    x = rnd(T, d, seed=4)
    delta = rnd(T, d, dtype=dtype, seed=5)
    w = (1 + 0.1 * rnd(d, seed=6)).to(dtype)
    rows = torch.tensor([8, 0, 3, 3], dtype=torch.int32, device=DEV)
    out = torch.empty(4, d, dtype=dtype, device=DEV)
    x0 = x.clone()
    ops.add_rmsnorm(x, delta, w, eps, out, rows)
    assert torch.equal(x, x0)                       # a gather leaves the residual alone
    s = (x0.double() + delta.double())[rows.long()]
    ref = s * torch.rsqrt((s * s).mean(-1, keepdim=True) + eps) * w.double()
    assert torch.allclose(out.double(), ref, **tol(dtype))
    # the sums of the gathered rows can be had as well: the residual stream cut down to those rows
    x_rows = torch.full((4, d), 7.0, device=DEV)
    out2 = torch.empty_like(out)
    ops.add_rmsnorm(x, delta, w, eps, out2, rows, x_rows)
    assert torch.equal(x, x0) and torch.equal(out2, out)
    assert torch.allclose(x_rows.double(), s, rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("T,I", [(1, 176), (6, 1000), (3, 8192)])
def test_swiglu(ops, dtype, T, I):
    gu = rnd(T, 2 * I, dtype=dtype, seed=7, scale=2.0)
    out = torch.empty(T, I, dtype=dtype, device=DEV)
    ops.swiglu(gu, out)
    g, u = gu[:, :I].double(), gu[:, I:].double()
    assert torch.allclose(out.double(), g / (1 + torch.exp(-g)) * u, **tol(dtype))


def test_silu_values(ops):
    # silu(0) = 0, silu(1) = 0.7311 (crates/infer-backend-cpu/src/lib.rs:1387-1394)
    gu = torch.tensor([[0.0, 1.0, 1.0, 1.0]], device=DEV)
    out = torch.empty(1, 2, device=DEV)
    ops.swiglu(gu, out)
    assert abs(out[0, 0].item()) == 0.0 and abs(out[0, 1].item() - 0.731058) < 1e-5


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(1, 50, 64), (3, 333, 200), (8, 1000, 416), (9, 130, 72),
                                   (16, 2048, 2048), (17, 48, 8192), (33, 100, 1024), (64, 4100, 520),
                                   (70, 257, 136), (200, 96, 1000), (4, 31, 44), (70, 96, 44), (200, 31, 100), (130, 77, 36)])
def test_linear(ops, dtype, M, N, K):
    x = rnd(M, K, dtype=dtype, seed=8)
    w = rnd(N, K, dtype=dtype, seed=9, scale=0.1)
    out = torch.empty(M, N, dtype=dtype, device=DEV)
    ops.linear(x, w, out)
    ref = x.double() @ w.double().t()
    # a 32-bit sum of K terms: rounding grows like sqrt(K) * 2^-24 * the size of the sums
    f32 = dict(rtol=0, atol=1.2e-7 * math.sqrt(K) * ref.abs().max().item())
    assert torch.allclose(out.double(), ref, **(f32 if dtype == torch.float32 else tol(dtype)))
    if dtype == torch.bfloat16:                      # 32-bit output of bfloat16 operands (logits)
        out32 = torch.empty(M, N, device=DEV)
        ops.linear(x, w, out32)
        assert torch.allclose(out32.double(), ref, **f32)
        wt = ops.tile_weight(w)                      # the tile-ordered copy gives the same bits
        assert (wt is not None) == (N % 16 == 0 and K % 32 == 0)
        if wt is not None:
            out_t = torch.empty(M, N, device=DEV)
            ops.linear(x, w, out_t, wt)
            if M < ops.UNTILED_LIBRARY_MIN_ROWS and N * K < ops.UNTILED_LIBRARY_LARGE:
                assert torch.equal(out_t, out32)     # the few-row kernel either way
            else:                                    # without the copy the GEMM library took the product
                assert torch.allclose(out_t.double(), ref, **f32)
        if M > ops.SKINNY_MAX_ROWS:
            # where the GEMM library has no kernel for a problem, the engine's own tiled kernel runs
            # it; here the library is taken to have refused, whatever it would have said
            shape = (N, K, x.stride(0), w.stride(0), N, torch.bfloat16)
            refused = shape in ops._LIBRARY_REFUSED
            ops._LIBRARY_REFUSED.add(shape)
            try:
                own = torch.full((M, N), float("nan"), dtype=dtype, device=DEV)
                ops.linear(x, w, own)
            finally:
                if not refused:
                    ops._LIBRARY_REFUSED.discard(shape)
            assert torch.allclose(own.double(), ref, **tol(dtype))
            print(f"library GEMM for M={M} N={N} K={K}: {'refused' if refused else 'took it'}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,I,K", [(1, 176, 64), (5, 416, 160), (17, 100, 72), (64, 1000, 520), (70, 96, 136), (9, 2048, 512)])
def test_linear_swiglu(ops, dtype, M, I, K):
    x = rnd(M, K, dtype=dtype, seed=20)
    w = rnd(2 * I, K, dtype=dtype, seed=21, scale=0.05)
    out = torch.empty(M, I, dtype=dtype, device=DEV)
    scratch = torch.empty(M, 2 * I, dtype=dtype, device=DEV)
    ops.linear_swiglu(x, w, out, scratch)
    wt = ops.tile_weight(w) if dtype == torch.bfloat16 else None
    g, u = x.double() @ w[:I].double().t(), x.double() @ w[I:].double().t()
    ref = g / (1 + torch.exp(-g)) * u
    if wt is not None:
        out_t = torch.empty_like(out)
        ops.linear_swiglu(x, w, out_t, scratch, wt)
        if M < ops.UNTILED_LIBRARY_MIN_ROWS:
            assert torch.equal(out_t, out)              # the few-row kernel, whichever order it reads the weight in
        else:                                            # without the second copy: the library's product, then the activation
            assert torch.allclose(out_t.double(), ref, **tol(dtype))
    f32 = dict(rtol=0, atol=5e-7 * math.sqrt(K) * max(1.0, ref.abs().max().item()))   # two 32-bit sums of K terms, multiplied
    assert torch.allclose(out.double(), ref, **(f32 if dtype == torch.float32 else tol(dtype)))


@pytest.mark.parametrize("M,N,K", [(17, 16, 32), (64, 4096, 4096), (33, 80, 96), (48, 2048, 8192), (49, 1008, 160), (20, 4096, 14336),
                                   (64, 48, 544), (40, 8192, 160), (50, 24576, 64), (40, 32896, 64)])
def test_rows_kernel_with_activations_in_lds(ops, M, N, K):
    """17..64 rows: the kernel whose blocks share their activations through LDS, as partial sums over
    slices of K, as a whole product in either output type and with the fused SwiGLU."""
    import ctypes
    lib = ops._lib()
    x = rnd(M, K, dtype=torch.bfloat16, seed=90)
    w = rnd(N, K, dtype=torch.bfloat16, seed=91, scale=0.05)
    wt = ops.tile_weight(w)
    ref = x.double() @ w.double().t()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    for nt, groups in ((1, 1), (2, 1), (1, 2), (2, 2), (1, 4), (2, 4)):
        for parts in (1, 2, 3, 16):
            stack = torch.full((parts, M, N), float("nan"), device=DEV)
            assert lib.ri_gemm_rows_bf16(P(x), K, P(wt), P(stack), N, M, N, K, 0, 0, parts, ctypes.c_longlong(M * N), nt, groups, stream) == 0, lib.ri_last_error()
            assert torch.allclose(stack.double().sum(0), ref, rtol=0, atol=2e-6 * max(1.0, ref.abs().max().item()) * math.sqrt(K / 32))
        out = torch.full((M, N + 16), float("nan"), dtype=torch.bfloat16, device=DEV)       # rows with a stride
        assert lib.ri_gemm_rows_bf16(P(x), K, P(wt), P(out), N + 16, M, N, K, 1, 0, 1, ctypes.c_longlong(0), nt, groups, stream) == 0
        assert torch.allclose(out[:, :N].double(), ref, **tol(torch.bfloat16)) and torch.isnan(out[:, N:]).all()
    # through the operations: partial sums for the norm, and SwiGLU where the columns are many
    ws = Workspace(DEV)
    delta = ops.linear_delta(x, w, ws, "t", wt)
    got = delta.double().sum(0) if delta.dim() == 3 else delta.double()
    assert torch.allclose(got, ref, **(dict(rtol=0, atol=2e-6 * max(1.0, ref.abs().max().item()) * math.sqrt(K / 32))
                                       if delta.dim() == 3 else tol(torch.bfloat16)))
    if N % 32 == 0:
        I = N // 2
        act = torch.empty(M, I, dtype=torch.bfloat16, device=DEV)
        g, u = ref[:, :I], ref[:, I:]
        want = g / (1 + torch.exp(-g)) * u
        for groups in (1, 2, 4):
            act = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV)
            assert lib.ri_gemm_rows_bf16(P(x), K, P(wt), P(act), I, M, I, K, 1, 1, 1, ctypes.c_longlong(0), 1, groups, stream) == 0
            assert torch.allclose(act.double(), want, **tol(torch.bfloat16))
        act = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV)
        # four groups at I = 4096, two at 12288, one at 16448, else the few-row kernel
        ops.linear_swiglu(x, w, act, None, wt)
        assert torch.allclose(act.double(), want, **tol(torch.bfloat16))
    bad = lib.ri_gemm_rows_bf16(P(x), K, P(wt), P(out), N, M, N, K, 1, 1, 1, ctypes.c_longlong(0), 2, 1, stream)
    assert bad != 0 and b"one gate and one up tile" in lib.ri_last_error()


def test_slices_and_groups_of_the_rows_kernel(ops):
    """The plan for products whose partial sums a norm adds up: no more blocks than run at once."""
    import ctypes
    lib = ops._lib()

    def plan(M, N, K):
        parts, groups = ctypes.c_int(), ctypes.c_int()
        assert lib.ri_gemm_rows_plan(M, N, K, 1, ctypes.byref(parts), ctypes.byref(groups)) == 0
        return parts.value, groups.value

    assert plan(64, 4096, 4096) == (4, 2) and plan(64, 4096, 14336) == (8, 1)
    assert plan(64, 8192, 8192) == (4, 1) and plan(64, 8192, 28672) == (4, 1)
    assert plan(64, 5120, 5120) == (4, 1) and plan(32, 5120, 5120) == (8, 1)     # 80 blocks of columns: 640 at 64 rows would not
    assert plan(64, 2048, 8192) == (8, 2) and plan(20, 64, 64) == (1, 1)
    assert ops._swiglu_groups(8192) == 4 and ops._swiglu_groups(14336) == 2 and ops._swiglu_groups(11008) == 2
    assert ops._swiglu_groups(28672) == 1 and ops._swiglu_groups(9000) == 0 and ops._swiglu_groups(2048) == 0
    # the product that adds to the residual stream itself: not beyond eight rows against a large
    # weight, nor where its blocks of 16 columns fill the chip badly
    shape = lambda N, K: torch.empty(N, K, device="meta")
    pays = ops.linear_residual_pays
    assert pays(8, shape(4096, 14336)) and not pays(9, shape(4096, 14336)) and pays(16, shape(4096, 4096))
    assert not pays(1, shape(5120, 13824)) and pays(16, shape(5120, 5120)) and pays(16, shape(3072, 8192))
    assert pays(8, shape(8192, 8192)) and not pays(16, shape(8192, 8192)) and pays(16, shape(2048, 8192))


@pytest.mark.parametrize("M,N,f32,first", [(1153, 32768, 0, 1024), (1433, 32768, 1, 1024), (1434, 32768, 0, 0), (1024, 32768, 0, 0), (767, 32768, 0, 0), (2049, 16384, 0, 2048),
                                           (2100, 16640, 0, 0), (4500, 8192, 1, 4096)])
def test_library_gemm_of_whole_rounds_and_the_rest(ops, M, N, f32, first):
    """Rows that make whole rounds of tiles go in a call of their own: every row once, rows inside wider buffers, nothing beside them."""
    K = 128
    assert ops._lib().ri_gemm_library_first_rows(M, N) == first
    xb = rnd(M, K + 8, dtype=torch.bfloat16, seed=1)
    x, w = xb[:, :K], rnd(N, K, dtype=torch.bfloat16, seed=2, scale=0.1)
    out = torch.full((M, N + 8), float("nan"), dtype=torch.float32 if f32 else torch.bfloat16, device=DEV)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=DEV)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    assert ops._lib().ri_gemm_library_bf16(p(x), K + 8, p(w), K, p(out), N + 8, M, N, K, f32, p(ws), ctypes.c_size_t(ws.numel()),
                                           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    ref = x.float() @ w.float().t()
    # one rounding to bfloat16, or a sum of 128 products in 32 bits
    assert torch.all((out[:, :N].float() - ref).abs() <= (2.0 ** -8 * ref.abs() if not f32 else 0) + 2.0 ** -16 * ref.abs().max())
    assert torch.isnan(out[:, N:]).all()


@pytest.mark.parametrize("M,N,f32,first", [(2048, 8208, 0, 8192), (1793, 11456, 0, 8192), (1792, 11456, 0, 0), (2000, 18448, 1, 16384), (2048, 11600, 0, 0), (2048, 8208, 1, 0),
                                           (512, 33000, 0, 32768), (448, 33000, 0, 32768), (447, 33000, 0, 0), (1024, 44096, 0, 32768), (1024, 42000, 0, 0), (8192, 2300, 0, 2048)])
def test_library_gemm_of_whole_rounds_of_columns(ops, M, N, f32, first):
    """Columns that make whole rounds of tiles likewise."""
    K = 128
    assert ops._lib().ri_gemm_library_first_rows(M, N) == 0 and ops._lib().ri_gemm_library_first_columns(M, N, f32) == first
    xb = rnd(M, K + 8, dtype=torch.bfloat16, seed=1)
    x, w = xb[:, :K], rnd(N, K, dtype=torch.bfloat16, seed=2, scale=0.1)
    out = torch.full((M, N + 8), float("nan"), dtype=torch.float32 if f32 else torch.bfloat16, device=DEV)
    ws = torch.empty(64 << 20, dtype=torch.uint8, device=DEV)
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    assert ops._lib().ri_gemm_library_bf16(p(x), K + 8, p(w), K, p(out), N + 8, M, N, K, f32, p(ws), ctypes.c_size_t(ws.numel()),
                                           ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    ref = x.float() @ w.float().t()
    # one rounding to bfloat16, or a sum of 128 products in 32 bits
    assert torch.all((out[:, :N].float() - ref).abs() <= (2.0 ** -8 * ref.abs() if not f32 else 0) + 2.0 ** -16 * ref.abs().max())
    assert torch.isnan(out[:, N:]).all()


def test_library_gemm_with_a_tuned_kernel(ops, tmp_path):
    """With tuning on, a product of more than 64 rows times the library's kernels once for its row
    bucket, keeps the choice in a file, and gives the same result (to bfloat16 rounding) as before."""
    M, N, K = 96, 320, 256
    x = rnd(M, K, dtype=torch.bfloat16, seed=80)
    w = rnd(N, K, dtype=torch.bfloat16, seed=81, scale=0.05)
    ref = x.double() @ w.double().t()
    plain = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    ops.linear(x, w, plain)
    file = tmp_path / "tuned.txt"
    before = ops.gemm_tuned_shapes()
    try:
        ops.set_gemm_tuning(True, str(file))
        out = torch.empty(M + 3, N, dtype=torch.bfloat16, device=DEV)          # other row counts of the bucket (81..96)
        for rows in (M - 3, M, 85):
            ops.linear(torch.cat([x, x[:3]])[:rows], w, out[:rows])
            assert torch.allclose(out[:min(rows, M)].double(), ref[:min(rows, M)], **tol(torch.bfloat16))
        assert ops.gemm_tuned_shapes() == before + 1                             # one bucket, tuned once
        lines = file.read_text().split("\n")
        assert len([l for l in lines if l.strip()]) == 1 and lines[0].split()[:4] == ["96", str(N), str(K), "0"]
    finally:
        ops.set_gemm_tuning(False)
    assert torch.allclose(plain.double(), ref, **tol(torch.bfloat16))


def test_library_gemm_asks_for_a_kernel_once_a_row_bucket(ops):
    """Prompt portions of changing length: the library is asked to choose a kernel once for a
    (row bucket, N, K), not once for every row count, and every row count gives the right product."""
    N, K = 448, 352
    w = rnd(N, K, dtype=torch.bfloat16, seed=83, scale=0.05)
    x = rnd(1100, K, dtype=torch.bfloat16, seed=82)
    ref = x.double() @ w.double().t()
    _, asked0 = ops.gemm_library_stats()
    rows = [129, 200, 131, 255, 256, 300, 511, 257, 600, 1000, 1024, 513, 130, 1100]      # buckets 144, 208, 256, 320, 512, 288, 640, 1024, 1152
    for M in rows:
        out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
        ops.linear(x[:M], w, out)
        assert torch.allclose(out.double(), ref[:M], **tol(torch.bfloat16)), M
    plans, asked = ops.gemm_library_stats()
    assert asked - asked0 <= 9 + 2, (asked0, asked)      # one question a bucket (one more where a bucket's kernel refuses a row count)
    assert plans >= len(set(rows))


def test_library_gemm_does_not_depend_on_what_was_served_before(ops):
    """Which of the library's kernels a row count gets depends on its bucket and on itself, not on
    the row counts that came earlier: the same product has the same bits whether a shorter or a
    longer portion of its bucket was served first."""
    N, K = 704, 480
    w = rnd(N, K, dtype=torch.bfloat16, seed=85, scale=0.05)
    x = rnd(512, K, dtype=torch.bfloat16, seed=84)
    got = {}
    for order in ((130, 250, 400, 512), (512, 400, 250, 130), (250, 512, 130, 400)):
        ops.gemm_library_reset()
        for M in order:
            out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
            ops.linear(x[:M], w, out)
            got.setdefault(M, []).append(out)
    ref = x.double() @ w.double().t()
    for M, outs in got.items():
        assert torch.allclose(outs[0].double(), ref[:M], **tol(torch.bfloat16))
        assert all(torch.equal(outs[0], o) for o in outs[1:]), M


def test_linear_identity_and_strided_output(ops):
    # identity weight returns the input; a strided output view leaves its padding untouched
    # (crates/infer-backend-cpu/src/lib.rs:1330-1352)
    x = rnd(5, 48, seed=10)
    eye = torch.eye(48, device=DEV)
    buf = torch.full((5, 64), 7.0, device=DEV)
    ops.linear(x, eye, buf[:, :48])
    assert torch.equal(buf[:, :48], x) and torch.all(buf[:, 48:] == 7.0)


def test_linear_rows_do_not_depend_on_the_batch(ops):
    # the exact path: a row's result is the same bits whatever else is in the batch
    x = rnd(70, 136, seed=11)
    w = rnd(257, 136, seed=12)
    full = torch.empty(70, 257, device=DEV)
    ops.linear(x, w, full)
    one = torch.empty(1, 257, device=DEV)
    for r in (0, 33, 69):
        ops.linear(x[r:r + 1], w, one)
        # one row and 70 take tiles of other sizes: the sums are made in one order
        assert torch.equal(one[0], full[r])
    # 1, 5, 8, 13 and 16 rows: the few-row kernel and one row of tiles of 16 x 16
    x2, w2 = rnd(16, 1352, seed=13), rnd(1001, 1352, seed=14)
    all16 = torch.empty(16, 1001, device=DEV)
    ops.linear(x2, w2, all16)
    ref = x2.double() @ w2.double().t()
    assert torch.allclose(all16.double(), ref, rtol=0, atol=6e-8 * ref.abs().max().item())    # half a unit of the last place
    for rows in ([3], [0, 1, 2, 3, 4], list(range(4, 12)), list(range(13)), list(range(15, -1, -1))):
        sub = torch.empty(len(rows), 1001, device=DEV)
        ops.linear(x2[rows].contiguous(), w2, sub)
        assert torch.equal(sub, all16[rows])
    # 17..64 rows: more rows of such tiles
    x3 = rnd(64, 1352, seed=15)
    x3[20] = x2[3]
    for M in (17, 37, 64):
        out = torch.full((M, 1001), float("nan"), device=DEV)
        ops.linear(x3[:M].contiguous(), w2, out)
        ref = x3[:M].double() @ w2.double().t()
        assert torch.allclose(out.double(), ref, rtol=0, atol=6e-8 * ref.abs().max().item())
        if M > 20:
            assert torch.equal(out[20], all16[3])


@pytest.mark.parametrize("M,N,K", [(5, 16, 4), (16, 17, 60), (17, 33, 132), (31, 2064, 36), (33, 4100, 64), (49, 300, 260),
                                   (65, 47, 1352), (160, 2050, 72), (300, 515, 516), (1030, 100, 20)])
def test_linear_f32_on_the_matrix_instruction(ops, M, N, K):
    # edges of the tiles of 16 x 16, 32 x 16 and 16 x 32 (the larger ones: the test below), a last chunk of K that is not whole, fewer chunks than waves, rows inside a wider buffer
    xb, wb = rnd(M, K + 8, seed=M), rnd(N, K + 4, seed=N)
    x, w = xb[:, 4:K + 4], wb[:, :K]
    out = torch.full((M, N + 3), float("nan"), device=DEV)
    ops.linear(x, w, out[:, :N])
    ref = x.double() @ w.double().t()
    # a 64-bit sum rounded once: half a unit of the last place of each result
    assert torch.all((out[:, :N].double() - ref).abs() <= ref.abs() * 2.0 ** -24 + 1e-12 * ref.abs().max())
    assert torch.all(torch.isnan(out[:, N:]))


def test_linear_f32_gives_a_row_the_same_bits_on_every_tile(ops):
    """Rows of terms that cancel to some 2^-23 of the largest, so that the order of the 64-bit sums shows in the 32-bit
    results: the first rows alone and among more rows, on each of the tiles, edges and a last part of K that is no
    whole turn of a wave included."""
    M, N, K = 600, 3075, 532
    g = torch.Generator().manual_seed(3)
    x = torch.randn(M, K, generator=g) * 2.0 ** torch.randint(-20, 21, (M, K), generator=g)
    x[:, K // 2:] = -x[:, :K // 2]
    w = torch.randn(N, K, generator=g)
    w[:, K // 2:] = w[:, :K // 2] * (1 + torch.randint(0, 2, (N, K // 2), generator=g) * 2.0 ** -23)
    x, w = x.to(DEV), w.to(DEV)
    tiles, first = set(), None
    for rows in (5, 17, 65, 300, 600):
        a, b = ctypes.c_int(0), ctypes.c_int(0)
        ops._lib().ri_gemm_f32_tile(rows, N, ctypes.byref(a), ctypes.byref(b))
        tiles.add((a.value, b.value))
        out = torch.full((rows, N), float("nan"), device=DEV)
        ops.linear(x[:rows], w, out)
        first = out[:5].clone() if first is None else first
        assert torch.equal(out[:5], first), rows
        ref = x[:rows].double() @ w.double().t()                   # K products in 64 bits, added in another order
        assert torch.all((out.double() - ref).abs() <= ref.abs() * 2.0 ** -24 + K * 2.0 ** -52 * (x[:rows].double().abs() @ w.double().abs().t()))
    assert tiles == {(16, 16), (32, 16), (16, 32), (32, 32), (48, 32)}


@pytest.mark.parametrize("M,N,K", [(1, 1, 4), (8, 7, 28), (3, 9, 32), (7, 17, 124), (5, 8, 128), (2, 33, 132), (8, 4097, 160), (6, 4096, 164), (4, 24577, 256),
                                   (7, 24599, 292), (8, 40, 1020), (1, 25, 1024), (6, 4111, 1056), (5, 4100, 1284), (8, 24600, 548), (3, 300, 2316)])
def test_linear_f32_of_up_to_eight_rows(ops, M, N, K):
    # 8, 16 and 24 columns a block and their edges; K below, at and past a half's and a turn's chunks, with fewer turns than
    # are under way, as many, and more; the last row of x not finite, which only its own results may show
    xb, wb = rnd(M + 1, K + 8, seed=M), rnd(N, K + 4, seed=N)
    x, w = xb[:M, 4:K + 4], wb[:, :K]
    out = torch.full((M, N + 3), float("nan"), device=DEV)
    ops.linear(x, w, out[:, :N])
    ref = x.double() @ w.double().t()
    # a 64-bit sum rounded once: half a unit of the last place of each result
    assert torch.all((out[:, :N].double() - ref).abs() <= ref.abs() * 2.0 ** -24 + 1e-12 * ref.abs().max())
    assert torch.all(torch.isnan(out[:, N:]))
    more = torch.empty(9, N, device=DEV)               # nine rows: tiles of sixteen, the same sums in the same order
    ops.linear(torch.cat([x, rnd(9 - M, K, seed=5)]), w, more)
    assert torch.equal(more[:M], out[:, :N])
    if M > 1:
        y = x.clone()
        y[M - 1, K // 2] = float("inf")
        y[M - 1, K - 1] = float("nan")
        bad = torch.empty(M, N, device=DEV)
        ops.linear(y, w, bad)
        assert torch.equal(bad[:M - 1], out[:M - 1, :N]) and torch.all(torch.isnan(bad[M - 1]))


@pytest.mark.parametrize("M,N,K,form", [(1, 4097, 2052, -1), (4, 5001, 2304, -1), (3, 2049, 5124, -1), (2, 3077, 7172, -1), (4, 32771, 1028, -1), (3, 4111, 772, -1),
                                        (2, 5120, 4096, -1), (8, 3000, 1540, 1), (5, 4096, 4096, 1), (6, 8190, 1024, 2), (2, 16384, 2048, 2), (8, 6144, 896, 3),
                                        (7, 12287, 1536, 3), (1, 8192, 1664, 0), (8, 4100, 900, 4), (8, 2056, 8192, 0)])
def test_linear_f32_of_up_to_eight_rows_on_every_form(ops, M, N, K, form):
    """The kernel of FMAs (long rows, but for rows a power of two apart whose tiles fill their rounds) and the forms of the tiles: 64-bit sums
    rounded once, and a row that is not finite alone with its results."""
    assert ops._lib().ri_gemm_f32_form(M, N, K, K) == form
    x, w = rnd(M, K + 4, seed=M)[:, :K], rnd(N, K, seed=N)
    out = torch.full((M, N + 3), float("nan"), device=DEV)
    ops.linear(x, w, out[:, :N])
    ref = x.double() @ w.double().t()
    # a 64-bit sum rounded once: half a unit of the last place of each result
    assert torch.all((out[:, :N].double() - ref).abs() <= ref.abs() * 2.0 ** -24 + 1e-12 * ref.abs().max())
    assert torch.all(torch.isnan(out[:, N:]))
    if M > 1:
        y = x.clone()
        y[M - 1, K // 2] = float("inf")
        y[M - 1, K - 1] = float("nan")
        bad = torch.empty(M, N, device=DEV)
        ops.linear(y, w, bad)
        assert torch.equal(bad[:M - 1], out[:M - 1, :N]) and torch.all(torch.isnan(bad[M - 1]))


@pytest.mark.parametrize("M,I,K,fused", [(1, 6912, 2560, 0), (4, 2560, 3588, 0), (2, 8192, 2560, 1), (4, 4096, 4096, 1), (8, 6912, 2560, 1)])
def test_swiglu_f32_of_up_to_eight_rows_by_the_length_of_rows(ops, M, I, K, fused):
    assert ops._lib().ri_gemm_f32_swiglu_pays(M, I, K, K) == fused
    x, w = rnd(M, K, seed=M), rnd(2 * I, K, seed=I) * (8.0 / K) ** 0.5
    ref = x.double() @ w.double().t()
    ref = torch.nn.functional.silu(ref[:, :I]) * ref[:, I:]
    for out in (torch.empty(M, I, device=DEV), torch.full((M, I + 5), float("nan"), device=DEV)[:, :I]):       # whole, and columns of a wider buffer
        ops.linear_swiglu(x, w, out, torch.empty(M, 2 * I, device=DEV))
        # a rounding of the gate's sum x moves silu by up to 1 + |x| times as much, |x| < 16; the up sum, exp to 2 units of the last
        # place and three 32-bit operations: 32 half units in all
        assert torch.all((out.double() - ref).abs() <= 2.0 ** -19 * ref.abs() + 1e-7)


@pytest.mark.parametrize("M,I,K", [(1, 1, 4), (8, 7, 132), (3, 8, 288), (6, 4099, 1028), (5, 24, 2304), (2, 9001, 160)])
def test_swiglu_f32_of_up_to_eight_rows_is_the_product_and_the_activation(ops, M, I, K):
    x, w = rnd(M, K + 4, seed=M)[:, :K], rnd(2 * I, K, seed=I) * 0.3
    scratch, want = torch.empty(M, 2 * I, device=DEV), torch.empty(M, I, device=DEV)
    ops.linear(x, w, scratch)
    ops.swiglu(scratch, want)
    out = torch.full((M, I + 5), float("nan"), device=DEV)
    ops.linear_swiglu(x, w, out[:, :I], torch.empty(M, 2 * I, device=DEV))
    assert torch.equal(out[:, :I], want) and torch.isnan(out[:, I:]).all()


# Digits (gemm_digits): whatever the rows hold, a result is rounded once (half a unit of the last place, of the least of them for results below the
# normal numbers) and is within 2^-27 of itself, or is a 64-bit sum, as the reference here: K 2^-52 of the sum of magnitudes for both.
def _digits_bound(x, w, ref):
    mag = x.double().abs() @ w.double().abs().t()
    return ref.abs() * (2.0 ** -24 + 2.0 ** -27) + 2.0 ** -150 + x.shape[1] * 2.0 ** -52 * mag


@pytest.mark.parametrize("M,N,K", [(24, 1024, 1024), (33, 3072, 2048), (64, 2080, 4096), (65, 4128, 1056), (129, 544, 9120), (100, 992, 14336), (300, 2048, 25984), (193, 8192, 288)])
def test_linear_f32_from_digits(ops, M, N, K):
    """Edges of tiles and of the slices of K, a last block of fewer than four tiles of columns, rows inside a wider buffer; exponents from the
    least to the largest, rows of zeros; a row's bits are the same alone with others, whatever the slices."""
    from rustinfer_amd.engine.context import Workspace
    xb = rnd(M, K + 8, seed=M)
    x, w = xb[:, 4:K + 4], rnd(N, K, seed=N) * 0.02
    x[3] = 0
    x[5] *= 1e-38                                        # some of them below the normal numbers
    x[7] *= 1e34
    w[9] *= 2.0 ** -100
    x[11] = x[11].abs().clamp(min=0.5)                   # first digits near their ends
    x[11, 1] = -(2.0 - 2.0 ** -23)
    wt = ops.tile_weight(w)
    assert wt is not None and wt.whole
    ws = Workspace(torch.device(DEV))
    parts = ops._digits_parts(x, w, wt, M, N, K) or 1
    ref = x.double() @ w.double().t()
    outs = []
    for p in {1, 2, parts}:
        out = torch.full((M, N + 3), float("nan"), device=DEV)
        ops._linear_digits(x, w, out[:, :N], wt, ws, p)
        assert torch.isnan(out[:, N:]).all()
        outs.append(out[:, :N])
        assert torch.equal(outs[-1], outs[0])
    few = torch.empty(M - 20, N, device=DEV)
    ops._linear_digits(x[20:].contiguous(), w, few, wt, ws, 1)
    assert torch.equal(few, outs[0][20:])
    assert torch.all((outs[0].double() - ref).abs() <= _digits_bound(x, w, ref))
    rows = [i for i in range(M) if i not in (3, 5)]
    plain = torch.empty(M, N, device=DEV)
    ops.linear(x, w, plain)
    e = lambda y: ((y[rows].double() - ref[rows]) / ref[rows].norm(dim=1, keepdim=True)).norm().item()
    assert e(outs[0]) <= 1.0005 * e(plain)               # no further from 64 bits than 64-bit sums are


def test_linear_f32_rows_without_digits(ops):
    """Rows that hold an infinity or a NaN, and rows whose values spread over more than the digits hold, go by 64-bit sums, in whole products
    and in slices; the other rows keep their bits."""
    from rustinfer_amd.engine.context import Workspace
    M, N, K = 100, 2080, 2048
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    wt, ws = ops.tile_weight(w), Workspace(torch.device(DEV))
    clean = torch.empty(M, N, device=DEV)
    ops._linear_digits(x, w, clean, wt, ws, 1)
    y = x.clone()
    y[2, 7], y[40, 0], y[40, 1], y[99, K - 1] = float("inf"), float("nan"), 1.0, -float("inf")
    spread = [0, 33, 64]
    g = torch.Generator().manual_seed(3)
    y[spread] = (torch.randn(3, K, generator=g) * 2.0 ** torch.randint(-60, 61, (3, K), generator=g)).to(DEV)
    ref = y.double() @ w.double().t()
    for parts in (1, 4):
        out = torch.full((M, N), float("nan"), device=DEV)
        ops._linear_digits(y, w, out, wt, ws, parts)
        special = [2, 40, 99] + spread
        rest = [i for i in range(M) if i not in special]
        assert torch.equal(out[rest], clean[rest])
        assert torch.isnan(out[40]).all() and torch.equal(out[[2, 99]], ref[[2, 99]].float())
        mag = y[spread].double().abs() @ w.double().abs().t()
        assert torch.all((out[spread].double() - ref[spread]).abs() <= ref[spread].abs() * 2.0 ** -24 + K * 2.0 ** -52 * mag)
    w2 = w.clone()
    w2[70, 3] = float("inf")
    assert ops.tile_weight(w2) is None and ops.tile_weight(w[:, :2046]) is None and ops.tile_weight(w[:2047]) is None


@pytest.mark.parametrize("M,N,K,bad", [(600, 4128, 256, 600), (100, 8224, 288, 37), (24, 2048, 1056, 1)])
def test_linear_f32_rows_without_digits_are_those_of_64_bit_sums(ops, M, N, K, bad):
    """More tiles of listed rows than blocks, a last tile of them that is not full, a single one: to the bit what the kernel of 64-bit sums gives."""
    from rustinfer_amd.engine.context import Workspace
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    g = torch.Generator().manual_seed(3)
    rows = torch.randperm(M, generator=g)[:bad]
    x[rows.to(DEV)] *= (2.0 ** torch.randint(-60, 61, (bad, K), generator=g).float()).to(DEV)
    wt, ws = ops.DigitWeight(w), Workspace(torch.device(DEV))
    want, out = torch.empty(M, N, device=DEV), torch.full((M, N + 4), float("nan"), device=DEV)
    ops.linear(x, w, want)
    for parts in (1, 3):
        ops._linear_digits(x, w, out[:, :N], wt, ws, parts)
        again = ws.get("digits.again", M + 1, N // 16 + 2, torch.int32).flatten()
        assert again[0] == bad and sorted(again[1:1 + bad].tolist()) == sorted(rows.tolist())
        assert torch.equal(out[rows.to(DEV), :N], want[rows.to(DEV)]) and torch.isnan(out[:, N:]).all()


def _digits_operands(form, M, N, K):
    """Finite rows whose results lie far below the products of the rows' largest values, or do in some columns."""
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2) * 0.02
    at = torch.arange(K, device=DEV)
    if form.startswith("outliers"):                      # one large value in each row of both, in other columns, where the other's are zero in the last form
        p = int(form.split()[1])
        x[:, 5] *= 2.0 ** p
        w[:, 9] *= 2.0 ** p
        if form.endswith("apart"):
            x[:, 9] = 0
            w[:, 5] = 0
    elif form.startswith("halves"):                      # a little more than half of x large, where w is zero
        small = at % 100 >= 54
        x[:, small] *= 2.0 ** -int(form.split()[1])
        w[:, ~small] = 0
    elif form == "cancelling":                           # sums of large products that cancel but for the values' last bits
        x[:, 1::2] = x[:, ::2]
        w[:, 1::2] = -w[:, ::2] * (1 + 2.0 ** -22)
    elif form == "some rows":                            # rows of all kinds, in one tile and apart
        x[::7, 11] *= 2.0 ** 20
        x[3] = x[3] * 2.0 ** (-(at % 40).float())
        w[::5, 13] *= 2.0 ** 14
        w[4] = w[4] * 2.0 ** (-(at % 40).float())
    return x.contiguous(), w.contiguous()


@pytest.mark.parametrize("form", ["outliers 10", "outliers 12", "outliers 12 apart", "halves 20", "halves 30", "halves 42", "cancelling", "some rows"])
@pytest.mark.parametrize("M,N,K", [(70, 544, 8192), (33, 1056, 2048)])
def test_linear_f32_from_digits_whatever_the_rows_hold(ops, form, M, N, K):
    """Each result to its own bound, not to that of the rows' largest values; in whole products and in slices."""
    from rustinfer_amd.engine.context import Workspace
    x, w = _digits_operands(form, M, N, K)
    wt, ws = ops.DigitWeight(w), Workspace(torch.device(DEV))
    ref = x.double() @ w.double().t()
    plain = torch.empty(M, N, device=DEV)
    ops.linear(x, w, plain)
    for parts in (1, 3):
        out = torch.full((M, N), float("nan"), device=DEV)
        ops._linear_digits(x, w, out, wt, ws, parts)
        assert torch.all((out.double() - ref).abs() <= _digits_bound(x, w, ref)), (form, parts)
        assert (out.double() - ref).norm() <= 1.0005 * (plain.double() - ref).norm() + 2.0 ** -40 * ref.norm()


@pytest.mark.parametrize("M,I,K", [(40, 1024, 2048), (130, 8192, 1024), (64, 2720, 1056), (33, 14336, 512)])
def test_swiglu_mlp_f32_from_digits(ops, M, I, K):
    """Both products of a 32-bit MLP through digits, in whole products and slices, the activation rounded between them: the second no further from 64 bits than 64-bit sums
    of the same activation; a row that is not finite, one whose activation passes the 32-bit range, and one of widely spread values."""
    from rustinfer_amd.engine.context import Workspace
    D = 1024
    x, wgu, wd = rnd(M, K, seed=1), rnd(2 * I, K, seed=2) * 0.05, rnd(D, I, seed=3) * 0.02
    tgu, td, ws = ops.tile_weight(wgu), ops.tile_weight(wd), Workspace(torch.device(DEV))
    scratch, act = torch.empty(M, 2 * I, device=DEV), torch.empty(M, I, device=DEV)
    ops._linear_digits(x, wgu, scratch, tgu, ws, 1)
    assert torch.all((scratch.double() - x.double() @ wgu.double().t()).abs() <= _digits_bound(x, wgu, x.double() @ wgu.double().t()))
    scratch[1, 5] = float("nan")
    scratch[2, 7], scratch[2, I + 7] = 1e20, 1e20
    g = torch.Generator().manual_seed(3)
    scratch[3, I:] = (torch.randn(I, generator=g) * 2.0 ** torch.randint(-60, 61, (I,), generator=g)).to(DEV)
    ops.swiglu(scratch, act)
    ref, want = act.double() @ wd.double().t(), torch.empty(M, D, device=DEV)
    ops.linear(act, wd, want)
    rows = [i for i in range(M) if i not in (1, 2)]
    for parts in (1, 3):
        got = torch.full((M, D), float("nan"), device=DEV)
        ops._linear_digits(act, wd, got, td, ws, parts)
        assert torch.isnan(got[1]).all() and torch.isinf(got[2]).all() and torch.equal(got[2], want[2])
        assert torch.all((got[rows].double() - ref[rows]).abs() <= _digits_bound(act[rows], wd, ref[rows]))
        assert torch.all((got[rows].double() - ref[rows]).norm(dim=1) <= (want[rows].double() - ref[rows]).norm(dim=1) * 1.05)


@pytest.mark.parametrize("M", [3, 20])
def test_linear_f32_of_rows_further_apart_than_32_bit_distances_reach(ops, M):
    far, K = (1 << 24) + 4, 12                          # 48 rows of such a distance: over 3 GiB
    buf = torch.empty(M * far, device=DEV)
    x = buf.as_strided((M, K), (far, 1))
    x.copy_(rnd(M, K, seed=1))
    w = rnd(19, K, seed=2)
    out = torch.empty(M, 19, device=DEV)
    ops.linear(x, w, out)
    ref = x.double() @ w.double().t()
    assert torch.all((out.double() - ref).abs() <= ref.abs() * 2.0 ** -24 + 1e-12 * ref.abs().max())


def test_linear_f32_of_more_tiles_than_a_launch_holds(ops):
    """66,016 rows of 131,072 columns, as the logits of a whole large batch are: 34.6 GB in two launches; rows around the
    seam, the first and the last."""
    M, N, K = 66016, 131072, 4
    x, w = rnd(M, K, seed=1), rnd(N, K, seed=2)
    out = torch.full((M, N), float("nan"), device=DEV)
    a, b = ctypes.c_int(0), ctypes.c_int(0)
    ops._lib().ri_gemm_f32_tile(M, N, ctypes.byref(a), ctypes.byref(b))
    seam = ((1 << 23) - 1) // (N // b.value) * a.value
    assert 0 < seam < M - 64
    ops.linear(x, w, out)
    assert not out.sum().isnan()
    for r in (0, 31, 32, seam - 1, seam, seam + 40, M - 1):
        ref = x[r].double() @ w.double().t()
        assert torch.all((out[r].double() - ref).abs() <= ref.abs() * 2.0 ** -24 + 1e-15), r
    del out
    torch.cuda.empty_cache()


@pytest.mark.parametrize("M,N,K,acts", [(1, 64, 32, [(0, 64, "relu2")]), (8, 2064, 64, [(16, 2048, "relu2")]), (5, 96, 96, [(16, 16, "tanh"), (48, 32, "relu2")]),
                                        (16, 32800, 64, [(32784, 16, "tanh"), (0, 32768, "relu2")]), (17, 4112, 128, [(2048, 2064, "relu2")]), (40, 160, 2048, [(0, 32, "tanh"), (144, 16, "relu2")]),
                                        (64, 16400, 32, [(0, 16400, "relu2")]), (9, 80, 32, [(8, 24, "tanh")]), (70, 64, 64, [(16, 32, "relu2")])])
def test_linear_with_activated_columns(ops, M, N, K, acts):
    """In the product's epilogue (edges of tiles and of the stretches, one and several tiles a wave) and behind it (more rows, columns that
    begin inside a tile): against 64-bit arithmetic on the unrounded sums, and nothing else is touched."""
    x = rnd(M, K, seed=M).to(torch.bfloat16)
    w = (rnd(N, K, seed=N) * 0.2).to(torch.bfloat16)
    out = torch.full((M, N + 8), float("nan"), dtype=torch.bfloat16, device=DEV)
    bufs = [torch.full((M, n + 24), float("nan"), dtype=torch.bfloat16, device=DEV) for _, n, _ in acts]
    given = [(c0, n, f, out[:, c0:c0 + n] if f == "tanh" else b[:, 8:8 + n]) for (c0, n, f), b in zip(acts, bufs)]
    ops.linear_activated(x, w, out[:, :N], ops.tile_weight(w) if N % 16 == 0 and K % 32 == 0 else None, given)
    ref = x.double() @ w.double().t()
    plain = torch.ones(N, dtype=torch.bool)
    for (c0, n, f), b in zip(acts, bufs):
        z = ref[:, c0:c0 + n]
        want = torch.relu(z).square() if f == "relu2" else torch.tanh(z)
        got = out[:, c0:c0 + n] if f == "tanh" else b[:, 8:8 + n]
        # bfloat16 rounds to 2^-8: the result, and behind the product the sum too, which the square doubles; 2^-6 covers the three
        assert torch.all((got.double() - want).abs() <= 2.0 ** -6 * want.abs() + 2.0 ** -8 * z.abs().clamp(max=1.0) * (f == "tanh") + 1e-4)
        if f == "relu2":
            assert torch.isnan(b[:, :8]).all() and torch.isnan(b[:, 8 + n:]).all()
        plain[c0:c0 + n] = False
    assert torch.all((out[:, :N][:, plain].double() - ref[:, plain]).abs() <= 2.0 ** -8 * ref[:, plain].abs() + 1e-4)
    assert torch.isnan(out[:, N:]).all()


@pytest.mark.parametrize("M,N,K,acts", [(1, 64, 32, [(0, 64, "relu2")]), (8, 2064, 64, [(16, 2048, "relu2"), (0, 16, "tanh")]), (16, 32800, 64, [(0, 32768, "relu2")]),
                                        (33, 4112, 2048, [(2048, 2064, "relu2")]), (64, 160, 2048, [(0, 32, "tanh"), (144, 16, "relu2")])])
def test_activated_columns_are_made_of_unrounded_sums(ops, monkeypatch, M, N, K, acts):
    """In the product's epilogue, no kernel behind it: one bfloat16 rounding (2^-8 of the value) and 32-bit sums, where rounded sums would be squared with twice
    that of their own."""
    def refuse(*a):
        raise AssertionError("the activation's kernel ran")
    monkeypatch.setattr(ops, "unary", refuse)
    x = rnd(M, K, seed=M).to(torch.bfloat16)
    w = (rnd(N, K, seed=N) * 0.2).to(torch.bfloat16)
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    bufs = [torch.empty(M, n, dtype=torch.bfloat16, device=DEV) for _, n, _ in acts]
    ops.linear_activated(x, w, out, ops.tile_weight(w), [(c0, n, f, b) for (c0, n, f), b in zip(acts, bufs)])
    ref = x.double() @ w.double().t()
    size = x.double().abs() @ w.double().abs().t()                 # of the sums' terms: 32-bit rounding of a sum is under 2^-18 of it
    for (c0, n, f), b in zip(acts, bufs):
        z, e = ref[:, c0:c0 + n], size[:, c0:c0 + n] * 2.0 ** -18
        want, slope = (torch.relu(z).square(), 2 * torch.relu(z) + e) if f == "relu2" else (torch.tanh(z), torch.ones_like(z))
        assert torch.all((b.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1.01 * slope * e + 1e-30)


@pytest.mark.parametrize("T,n,group,pad", [(1, 8, 8, 0), (3, 2048, 2048, 0), (5, 2304, 256, 8), (2, 3072, 1024, 16), (7, 1024, 512, 0), (4, 4096, 2048, 8), (3, 192, 64, 4),
                                           (2, 72, 24, 0), (2, 4096, 4096, 0), (300, 128, 16, 8),
                                           (2, 1024, 1024, 0), (3, 1536, 512, 8), (2, 512, 512, 0), (5, 1536, 256, 0), (128, 2048, 64, 0), (127, 2048, 64, 8),
                                           (1030, 256, 32, 0), (9, 256, 128, 0), (9, 128, 128, 0), (1100, 64, 16, 0), (2, 4, 4, 0), (3, 6, 2, 2)])
@pytest.mark.parametrize("dtype,w_dtype", [(torch.bfloat16, torch.float32), (torch.bfloat16, torch.bfloat16), (torch.float32, torch.float32)])
def test_gated_group_norm_of_eight_values_a_thread(ops, T, n, group, pad, dtype, w_dtype):
    # groups in a few lanes, a wave, two and four waves; rows that end inside a block; and what the other kernel keeps (strides, sizes)
    o = (rnd(T, n + pad, seed=n) * 3)[:, :n]
    gate = rnd(T, n + pad, seed=1).to(dtype)[:, :n]
    w = (rnd(n, seed=2) + 1).to(w_dtype)
    for kw in (dict(), dict(gate_activation="silu"), dict(gate_activation="silu", gate_first=True)):
        for weight, z in ((w, gate), (None, gate), (w, None)):
            out = torch.full((T, n + 8), float("nan"), dtype=dtype, device=DEV)
            ops.gated_group_norm(o, weight, z, out[:, :n], group, 1e-5, **kw)
            a = o.double()
            g = torch.ones_like(a) if z is None else torch.sigmoid(z.double()) if not kw else torch.nn.functional.silu(z.double())
            if kw.get("gate_first"):
                a, g = a * g, torch.ones_like(g)
            y = a.view(T, -1, group)
            y = (y / torch.sqrt(y.square().mean(-1, keepdim=True) + 1e-5)).reshape(T, n) * g * (1.0 if weight is None else weight.double())
            tol = 2e-6 if dtype == torch.float32 else 2.0 ** -8 + 2e-6          # rounding, and 32-bit arithmetic
            assert torch.all((out[:, :n].double() - y).abs() <= tol * y.abs() + 1e-6)
            assert torch.isnan(out[:, n:]).all()


def _paged_setup(dtype, B, H, Hkv, hd, page, q_lens, starts, seed=0, num_pages=128, shuffle=True):
    """A cache with random pages for each request, the step's q/k/v, and contiguous copies."""
    g = torch.Generator().manual_seed(seed)
    max_blocks = max(80, max(s + q for s, q in zip(starts, q_lens)) // page + 2)
    perm = torch.randperm(num_pages, generator=g).tolist() if shuffle else list(range(num_pages))
    table = torch.full((B, max_blocks), -1, dtype=torch.int32)
    kv_lens = [s + q for s, q in zip(starts, q_lens)]
    used = 0
    for b in range(B):
        n = (kv_lens[b] + page - 1) // page
        table[b, :n] = torch.tensor(perm[used:used + n], dtype=torch.int32)
        used += n
    T = sum(q_lens)
    positions, rows = [], []
    for b in range(B):
        positions += list(range(starts[b], kv_lens[b]))
        rows += [b] * q_lens[b]
    qkv_dim = (H + 2 * Hkv) * hd
    qkv = (torch.randn(T, qkv_dim, generator=g)).to(dtype).to(DEV)
    # pages are never cleared in the engine: what was not written may hold anything
    kc = torch.full((num_pages, Hkv, page, hd), float("nan"), dtype=dtype, device=DEV)
    vc = torch.full((num_pages, Hkv, hd, page), float("nan"), dtype=dtype, device=DEV)
    # history: random keys/values at positions [0, start)
    hist_k = [torch.randn(kv_lens[b], Hkv, hd, generator=g).to(dtype) for b in range(B)]
    hist_v = [torch.randn(kv_lens[b], Hkv, hd, generator=g).to(dtype) for b in range(B)]
    for b in range(B):
        for lo in range(0, starts[b], page):
            hi = min(starts[b], lo + page)
            blk = int(table[b, lo // page])
            kc[blk, :, :hi - lo] = hist_k[b][lo:hi].permute(1, 0, 2).to(DEV)
            vc[blk, :, :, :hi - lo] = hist_v[b][lo:hi].permute(1, 2, 0).to(DEV)
    ctx = SimpleNamespace(
        num_tokens=T, num_rows=B,
        positions=torch.tensor(positions, dtype=torch.int32, device=DEV),
        row_of_token=torch.tensor(rows, dtype=torch.int32, device=DEV),
        kv_lens=torch.tensor(kv_lens, dtype=torch.int32, device=DEV),
        q_start=torch.tensor(starts, dtype=torch.int32, device=DEV),
        cu_q=torch.tensor(np.concatenate([[0], np.cumsum(q_lens)]), dtype=torch.int32, device=DEV),
        max_q_len=max(q_lens), max_kv_len=max(kv_lens), decode_only=max(q_lens) == 1,
        host_q_lens=q_lens, host_q_start=starts, host_kv_lens=kv_lens, workspace=Workspace(DEV))
    # as the engine's steps do: the tokens of the rows of one token, then -1
    singles = [int(t) for t, q in zip(np.concatenate([[0], np.cumsum(q_lens)])[:-1], q_lens) if q == 1]
    ctx.num_single = len(singles)
    ctx.single_tokens = torch.tensor(singles + [-1] * (B - len(singles)), dtype=torch.int32, device=DEV)
    longer = [b for b, q in enumerate(q_lens) if q > 1]
    ctx.num_portion = len(longer)
    ctx.portion_rows = torch.tensor(longer + [-1] * (B - len(longer)), dtype=torch.int32, device=DEV)
    return qkv, kc, vc, table.to(DEV), ctx, hist_k, hist_v


ATT_CASES = [
    # B, H, Hkv, hd, page, q_lens, starts
    (1, 4, 2, 16, 16, [33], [0]),
    (3, 5, 1, 32, 8, [1, 7, 20], [40, 0, 13]),
    (2, 6, 3, 48, 16, [1, 1], [15, 16]),
    (2, 8, 2, 64, 16, [17, 1], [3, 99]),
    (1, 3, 3, 80, 4, [9], [22]),
    (2, 4, 1, 128, 16, [40, 2], [0, 130]),
    (1, 2, 2, 256, 16, [5], [11]),
    # single tokens at sizes the split-key matrix-core kernel takes (head 64 / 128, page 16 / 32)
    (3, 8, 2, 64, 16, [1, 1, 1], [0, 127, 300]),
    (2, 12, 4, 128, 16, [1, 1], [128, 515]),
    (2, 16, 1, 64, 32, [1, 1], [255, 256]),
    (4, 4, 4, 128, 16, [1, 1, 1, 1], [15, 16, 17, 1000]),
    # portions of prompts at sizes the tiled matrix-core kernel takes, alone and beside single tokens
    (2, 8, 2, 64, 16, [70, 33], [0, 50]),
    (3, 12, 4, 128, 16, [17, 1, 40], [100, 200, 0]),
    (1, 16, 1, 64, 32, [100], [29]),
    (2, 6, 2, 128, 16, [5, 64], [250, 3]),
    (3, 3, 3, 64, 16, [2, 16, 31], [0, 16, 1]),
    # portions whose blocks share keys and values through LDS and take the steps below the diagonal
    # two at a time (64 queries with 64 keys or more before them): one, three and no such double steps
    (2, 8, 2, 64, 16, [200, 130], [70, 0]),
    (2, 4, 2, 128, 16, [150, 64], [300, 5]),
    # head size 128 with so many tiles and heads that the tiled kernel runs two waves per SIMD
    (2, 128, 16, 128, 16, [1100, 100], [0, 37]),
    # single tokens over contexts so long that a wave of the split-key kernel takes several chunks
    (8, 8, 4, 64, 16, [1] * 8, [4500, 4099, 64, 1, 3000, 4351, 2047, 4496]),
    (8, 8, 4, 128, 32, [1] * 8, [4200, 63, 4159, 0, 1024, 4223, 17, 4100]),
    # single tokens of so many requests and kv heads that one block takes all chunks of a (token, kv head)
    (16, 16, 8, 64, 16, [1] * 16, [700, 0, 63, 64, 1023, 1024, 2500, 15, 16, 17, 300, 1, 2, 999, 48, 47]),
    (16, 24, 8, 128, 16, [1] * 16, [2047, 5, 1300, 128, 127, 64, 1000, 0, 1, 15, 16, 31, 32, 500, 63, 65]),
    (32, 20, 4, 64, 32, [1] * 32, [100, 1, 0, 500, 31, 32, 33, 2000, 64, 65, 1500, 7] + [(53 * i) % 400 for i in range(20)]),
    # ... and so many pairs that it does so whatever the number of chunks (here 9 and more a wave)
    (32, 16, 16, 64, 16, [1] * 32, [8300] + [(37 * i) % 200 for i in range(1, 32)]),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("case", ATT_CASES)
@pytest.mark.parametrize("window", [0, 11])
def test_rope_write_and_attention(ops, dtype, case, window):
    """rope_kv_write then paged_attention equal rotation + causal attention computed plainly
    over each request's whole sequence."""
    _check_rope_write_and_attention(ops, dtype, case, window)


def test_attention_of_a_long_portion_at_head_size_64(ops):
    """So many tiles and heads (128 over 32 kv heads, 2,100 tokens) that the tiled kernel takes
    four heads per wave with the keys and values shared through LDS and two waves per SIMD;
    three kv heads' groups are compared with the plain computation."""
    _check_rope_write_and_attention(ops, torch.bfloat16, (1, 128, 32, 64, 16, [2100], [0]), 0, kv_heads=(0, 13, 31))


@pytest.mark.parametrize("H,hd,q_lens,starts", [
    # 32 kv heads, pages of 16: what a wave and a block take, by waves and by the keys before the step
    (128, 64, [70, 1, 33], [30, 40, 0]),                         # one head, one tile a block; odd numbers of tiles
    (128, 64, [570], [0]), (128, 64, [400, 65, 129], [300, 0, 7]),    # two heads, one tile a block
    (128, 64, [1040, 3], [0, 50]),                               # two heads, pairs of tiles
    (128, 64, [1030], [600]),                                    # four heads, one tile a block
    (96, 64, [800, 2], [0, 9]),                                  # three heads a kv head: one head, pairs of tiles
    (128, 64, [200], [2100]), (128, 128, [200], [2100]),         # two ranges of keys, two heads a wave
    (128, 128, [520, 70], [0, 129]), (128, 128, [1100], [0]),    # two heads, single tiles and pairs
    (96, 128, [500], [0]), (96, 128, [1000], [64]),              # three heads a kv head: one head, and two with one idle
])
def test_attention_of_portions_however_they_are_divided(ops, H, hd, q_lens, starts):
    """Tiles of queries, heads and ranges of keys dealt to waves and blocks in each way the sizes can ask for; three kv
    heads' groups are compared with the plain computation."""
    _check_rope_write_and_attention(ops, torch.bfloat16, (len(q_lens), H, 32, hd, 16, q_lens, starts), 0, kv_heads=(0, 13, 31))


@pytest.mark.parametrize("interleaved", [False, True])
@pytest.mark.parametrize("H,Hkv,hd,q_lens,starts,window", [
    (8, 2, 64, [70, 1, 33], [30, 200, 0], 50), (3, 3, 24, [40, 7], [0, 90], 0), (6, 2, 128, [33], [64], 33), (2, 1, 256, [9, 1], [20, 40], 17),
    (8, 2, 64, [1] * 4, [0, 31, 64, 300], 100), (12, 2, 40, [1, 1], [5, 130], 0), (2, 2, 128, [1], [4500], 0), (2, 1, 256, [1, 1], [63, 65], 1)])
def test_turned_values_with_weights_in_three_parts(ops, monkeypatch, H, Hkv, hd, q_lens, starts, window, interleaved):
    """Values cached turned by their positions: the bfloat16 matrix instructions with the weights in three parts give what
    the 32-bit kernel gives, to the outputs' rounding (two roundings of one number: a unit in the last place, 2^-7 at
    most), in portions, mixed steps and single tokens, over the edges of tiles and partial results."""
    B = len(q_lens)
    need = sum((s + q + 15) // 16 for s, q in zip(starts, q_lens))
    qkv, kc, vc, table, ctx, hist_k, hist_v = _paged_setup(torch.bfloat16, B, H, Hkv, hd, 16, q_lens, starts, seed=hd + H,
                                                           num_pages=max(128, need + 16))
    for b in range(B):
        for j in range(starts[b], starts[b] + q_lens[b]):
            kc[int(table[b, j // 16]), :, j % 16] = hist_k[b][j].to(DEV)
            vc[int(table[b, j // 16]), :, :, j % 16] = hist_v[b][j].to(DEV)
    ang = torch.arange(5000, dtype=torch.float64)[:, None] * 300.0 ** (-torch.arange(hd // 2, dtype=torch.float64) / (hd // 2))
    tables = (ang.cos().float().to(DEV), ang.sin().float().to(DEV))
    q, got = qkv[:, :H * hd].contiguous(), []
    for parts in (True, False):
        monkeypatch.setattr(ops, "WINDOW_ATTENTION_PARTS", parts)
        monkeypatch.setattr(ops, "WINDOW_ATTENTION_MFMA", False)
        out = torch.empty_like(q)
        ops.window_attention(q, out, H, Hkv, hd, hd, kc, vc, table, 16, ctx, hd ** -0.5, window, value_rotary=tables,
                             interleaved_values=interleaved)
        got.append(out.float())
    assert got[1].isfinite().all() and got[1].abs().max() > 0.02      # (a mean of n unit normals is about n^-0.5: 0.015 for the longest row)
    assert ((got[0] - got[1]).abs() <= 2.0 ** -7 * got[1].abs() + 2e-5).all()


def test_attention_of_more_tiles_than_a_grid_has_places_for(ops):
    """One row of 8.4 M tokens with a window: some pairs of tiles beyond 65,535, the middle of the row."""
    hd, window, T = 64, 32, 2 * 65535 * 64 + 1000
    pages = -(-T // 16)
    q, k, v = (torch.randn(pages * 16, hd, device=DEV, dtype=torch.bfloat16, generator=torch.Generator(DEV).manual_seed(i)) for i in range(3))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    pos = torch.arange(T, dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(num_tokens=T, num_rows=1, cu_q=i32([0, T]), q_start=i32([0]), kv_lens=i32([T]), positions=pos,
                          row_of_token=torch.zeros_like(pos), max_q_len=T, max_kv_len=T, host_q_lens=[T], workspace=Workspace(torch.device(DEV)))
    out = torch.full((T, hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.paged_attention(q[:T], out, 1, 1, hd, k.view(pages, 1, 16, hd), v.view(pages, 16, hd).transpose(1, 2).contiguous().view(pages, 1, hd, 16),
                        torch.arange(pages, dtype=torch.int32, device=DEV).view(1, pages), 16, ctx, hd ** -0.5, window)
    assert out.isfinite().all()
    for p in (0, 40, 65535 * 64 - 1, 65535 * 64, 65535 * 64 + 500, 65535 * 64 + 999, 65535 * 64 + 1000, T - 1):
        lo = max(0, p + 1 - window)
        w = torch.softmax((k[lo:p + 1].double() @ q[p].double()) * hd ** -0.5, 0)
        assert ((w @ v[lo:p + 1].double()) - out[p].double()).abs().max() < 2e-2, p


RANGE_CASES = [
    # B, H, Hkv, hd, page, q_lens, starts; ranges of keys asked for (0: the kernel's own choice)
    ((1, 8, 2, 128, 16, [16], [2040]), 0),                       # a short portion behind many keys: six ranges of 384
    ((1, 8, 2, 128, 16, [16], [2040]), 16),                      # ranges of 129 -> 256 keys
    ((3, 8, 2, 64, 16, [200, 1, 70], [700, 300, 0]), 0),         # beside a single token; the third row ends inside the first range
    ((3, 8, 2, 64, 16, [200, 1, 70], [700, 300, 0]), 3),
    ((2, 4, 1, 128, 16, [130, 64], [1000, 129]), 5),             # a tile of queries that begins in one range and ends in the next
    ((2, 4, 1, 128, 16, [130, 64], [1000, 129]), 2),
    ((1, 8, 8, 64, 16, [1000], [0]), 4),                         # from the first token: ranges that the early tiles never reach
    ((3, 24, 8, 128, 16, [300, 300, 200], [2100, 0, 17]), 0),    # waves enough but for the one row behind many keys: three ranges
    ((2, 6, 2, 128, 16, [3, 259], [381, 250]), 2),               # a range's edge (256) inside a portion, odd lengths
]


@pytest.mark.parametrize("case,ranges", RANGE_CASES)
def test_attention_of_a_portion_with_the_keys_divided_between_blocks(ops, monkeypatch, case, ranges):
    """Short portions behind many cached keys: blocks take ranges of keys and a second kernel
    puts a query's ranges together; the result is the plain attention whatever the ranges."""
    import ctypes
    B, H, Hkv, hd, page, q_lens, starts = case
    lib = ops._lib()
    lib.ri_attention_prefill_workspace.restype = ctypes.c_size_t
    # the case does divide the keys (else it would test nothing new)
    portions = [(s, q) for s, q in zip(starts, q_lens) if q > 1]
    assert lib.ri_attention_prefill_workspace(H, Hkv, hd, page, 0, sum(q_lens), max(s for s, _ in portions),
                                              max(s + q for s, q in portions), ranges) > 0
    monkeypatch.setattr(ops, "PREFILL_KEY_RANGES", ranges)
    _check_rope_write_and_attention(ops, torch.bfloat16, case, 0)


@pytest.mark.parametrize("blocks", [2, 3, 8])
@pytest.mark.parametrize("window", [0, 700])
@pytest.mark.parametrize("case", [
    (8, 8, 4, 64, 16, [1] * 8, [4500, 4099, 64, 1, 3000, 4351, 2047, 4496]),
    (8, 8, 4, 128, 32, [1] * 8, [4200, 63, 4159, 0, 1024, 4223, 17, 4100]),
    (16, 24, 8, 128, 16, [1] * 16, [2047, 5, 1300, 128, 127, 64, 1000, 0, 1, 15, 16, 31, 32, 500, 63, 65]),
    (3, 12, 4, 128, 16, [17, 1, 40], [100, 1200, 0]),            # beside prompt portions
])
def test_single_token_attention_with_several_blocks_a_pair(ops, monkeypatch, case, window, blocks):
    """Single tokens whose (kv head, token) pairs are too few to fill the chip with a block each:
    several blocks of several waves a pair, each leaving one partial result.  Rows shorter than a
    block's first chunk leave that block's slot unwritten, and with a window a block may find every
    chunk of its own passed; the result is the plain attention all the same."""
    monkeypatch.setattr(ops, "DECODE_PAIR_BLOCKS", blocks)
    _check_rope_write_and_attention(ops, torch.bfloat16, case, window)


@pytest.mark.parametrize("case,window", [
    ((3, 8, 4, 128, 16, [1] * 3, [0, 0, 0]), 0),                                             # one span a row, fewer than waves
    ((5, 12, 4, 128, 16, [1] * 5, [30, 31, 32, 63, 64]), 0),                                 # ends around a span's
    ((9, 16, 1, 128, 64, [1] * 9, [2500, 0, 700, 15, 16, 17, 1300, 95, 3]), 0),              # 512 waves a head; rows of one span among long ones
    ((7, 8, 8, 128, 32, [1] * 7, [4200, 63, 4159, 10, 1024, 4223, 17]), 700),
    ((4, 6, 2, 128, 16, [1] * 4, [999, 1000, 1001, 1040]), 33),                              # a window that begins inside a span
    ((64, 8, 2, 128, 16, [1] * 64, [(i * 37) % 211 for i in range(64)]), 0),                 # a row a lane
    ((65, 8, 2, 128, 16, [1] * 65, [(i * 37) % 211 for i in range(65)]), 0),                 # one more: not as a list
])
def test_single_token_attention_of_rows_of_any_lengths(ops, case, window):
    """Rows' keys as one list whose stretches end anywhere in a row; slots never written and pages given back are NaN."""
    _check_rope_write_and_attention(ops, torch.bfloat16, case, window)


@pytest.mark.parametrize("case,window,as_list", [
    ((5, 16, 8, 128, 16, [1] * 5, [30, 31, 32, 63, 64]), 0, 1),                                  # ends around a span's
    ((3, 3, 3, 128, 16, [1] * 3, [0, 63, 300]), 0, 0),                                           # fewer than 12 pairs
    ((3, 8, 4, 128, 16, [1] * 3, [0, 64, 1]), 0, 1),
    ((64, 4, 1, 128, 16, [1] * 64, [2047, 0] * 32), 0, 1),                                       # 64 spans: a slot a span
    ((64, 4, 1, 128, 16, [1] * 64, [2048, 0] * 32), 0, 1),                                       # one more: stretches of two
    ((32, 4, 1, 128, 64, [1] * 32, [2500, 0, 700, 15, 16, 17, 1300, 95] * 4), 0, 1),             # 512 waves a head; rows of one span among long ones
    ((16, 6, 2, 128, 16, [1] * 16, [999, 1000, 1001, 1040] * 4), 33, 1),                         # a window that begins inside a span
    ((17, 8, 8, 128, 16, [1] * 17, [1023] * 9 + [5] * 8), 0, 0),                                 # one block a pair nearly fills the chip ...
    ((17, 8, 8, 128, 16, [1] * 17, [1024] * 9 + [5] * 8), 0, 1),                                 # ... from so many keys on not
    ((32, 8, 8, 128, 64, [1] * 32, [700] + [40] * 31), 0, 0),
    ((16, 8, 8, 128, 64, [1] * 16, [700] + [40] * 15), 0, 1),
    ((33, 8, 8, 128, 32, [1] * 33, [(i * 29) % 300 for i in range(33)]), 0, 1),                  # 264 pairs
])
def test_single_token_attention_as_a_list_where_it_pays(ops, case, window, as_list):
    B, H, Hkv, hd, page, q_lens, starts = case
    assert ops._lib().ri_attention_decode_as_list(B, Hkv, hd, page, max(starts) + 1) == as_list
    _check_rope_write_and_attention(ops, torch.bfloat16, case, window)


@pytest.mark.parametrize("heads", [2, 8])
def test_single_token_attention_as_a_list_with_padding_and_rows_out_of_order(ops, heads):
    B, H, Hkv, hd, page = 6, 8, heads, 128, 16
    lens = [300, 7, 1200, 64, 65, 500]
    qkv, kc, vc, table, ctx, _, _ = _paged_setup(torch.bfloat16, B, H, Hkv, hd, page, [1] * B, [n - 1 for n in lens], seed=3, num_pages=160)
    ops.rope_kv_write(qkv, H, Hkv, hd, None, ctx.positions, ctx.row_of_token, kc, vc, table, page)
    want = torch.empty(B, H * hd, dtype=torch.bfloat16, device=DEV)
    ops.paged_attention(qkv, want, H, Hkv, hd, kc, vc, table, page, ctx, 0.1, 0)
    order = [4, -1, 2, 0, -1, 5, 3, 1]                                     # token -> row
    at = torch.tensor([max(b, 0) for b in order], device=DEV)
    ctx.num_tokens, ctx.num_rows = len(order), B
    ctx.row_of_token, ctx.positions = torch.tensor(order, dtype=torch.int32, device=DEV), ctx.positions[at].contiguous()
    got = torch.full((len(order), H * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.paged_attention(qkv[at].contiguous(), got, H, Hkv, hd, kc, vc, table, page, ctx, 0.1, 0)
    for t, b in enumerate(order):
        if b < 0:
            assert torch.all(got[t] == 0)
        else:                                                              # stretches of the list end elsewhere: rounding of the output
            assert torch.allclose(got[t].float(), want[b].float(), rtol=2.0 ** -7, atol=1e-3), t


def test_single_token_attention_as_a_list_with_scores_of_minus_infinity(ops):
    """Keys whose scores are -inf have no weight, also where a whole span of 32 has no other (its first, in the middle, its last) or a wave's whole stretch."""
    B, H, Hkv, hd, page = 12, 8, 8, 128, 16
    lens = [300, 64, 90, 33, 300, 200, 40, 70, 100, 300, 65, 96]
    qkv, kc, vc, table, ctx, _, _ = _paged_setup(torch.bfloat16, B, H, Hkv, hd, page, [1] * B, [n - 1 for n in lens], seed=6, num_pages=200)
    qkv[:, :H * hd] = qkv[:, :H * hd].abs()             # so that a key of -inf scores -inf
    ops.rope_kv_write(qkv, H, Hkv, hd, None, ctx.positions, ctx.row_of_token, kc, vc, table, page)
    dead = [range(0, 32), range(32, 63), range(0, 64), range(0, 32), range(0, 288), range(64, 192), range(0, 39), range(10, 69), range(0, 96), range(5, 299), (), range(32, 64)]
    for b, keys in enumerate(dead):
        for j in keys:
            kc[int(table[b, j // page]), :, j % page] = float("-inf")
    assert ops._lib().ri_attention_decode_as_list(B, Hkv, hd, page, max(lens)) == 1
    got = torch.full((B, H * hd), float("nan"), dtype=torch.bfloat16, device=DEV)
    ops.paged_attention(qkv, got, H, Hkv, hd, kc, vc, table, page, ctx, 0.01, 0)
    for b, n in enumerate(lens):
        pages = table[b, :(n + page - 1) // page].long()
        k = kc[pages].permute(1, 0, 2, 3).reshape(Hkv, -1, hd)[:, :n].double()
        v = vc[pages].permute(1, 0, 3, 2).reshape(Hkv, -1, hd)[:, :n].double()
        p = torch.softmax((qkv[b, :H * hd].view(H, 1, hd).double() * k).sum(-1) * 0.01, -1)
        ref = (p[..., None] * v).sum(1).reshape(-1)
        # one bfloat16 rounding of the output, on weights of two bfloat16 (2^-16)
        assert torch.all((got[b].double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 1e-4), b


@pytest.mark.parametrize("window", [0, 500])
def test_single_token_attention_as_a_list_ends_at_the_steps_longest_length(ops, window):
    """A row that kv_lens says is longer than the step was planned for: its keys beyond that are not looked at, and the others' results
    are theirs."""
    B, H, Hkv, hd, page, longest = 12, 8, 8, 128, 16, 320
    lens = [300, 7, 900, 64, 320, 321, 5, 17, 310, 32, 33, 1]
    qkv, kc, vc, table, ctx, _, _ = _paged_setup(torch.bfloat16, B, H, Hkv, hd, page, [1] * B, [n - 1 for n in lens], seed=4, num_pages=200)
    ops.rope_kv_write(qkv, H, Hkv, hd, None, ctx.positions, ctx.row_of_token, kc, vc, table, page)
    ctx.max_kv_len = longest
    got, want = (torch.full((B, H * hd), float("nan"), dtype=torch.bfloat16, device=DEV) for _ in range(2))
    ops.paged_attention(qkv, got, H, Hkv, hd, kc, vc, table, page, ctx, 0.1, window)
    ctx.kv_lens = ctx.kv_lens.clamp(max=longest)
    ops.paged_attention(qkv, want, H, Hkv, hd, kc, vc, table, page, ctx, 0.1, window)
    assert torch.equal(got, want) and torch.isfinite(got).all()
    if window:                                         # the row of 900: its window of keys 400 .. 899 begins behind the last key
        assert torch.all(got[2] == 0)


def _check_rope_write_and_attention(ops, dtype, case, window, kv_heads=None):
    B, H, Hkv, hd, page, q_lens, starts = case
    need = sum((s + q + page - 1) // page for s, q in zip(starts, q_lens))
    qkv, kc, vc, table, ctx, hist_k, hist_v = _paged_setup(dtype, B, H, Hkv, hd, page, q_lens, starts, seed=hd + B,
                                                           num_pages=max(128, need + 16))
    freqs = plain_llama.rope_frequencies(hd, 10000.0, None)
    maxpos = max(1100, max(starts) + max(q_lens) + 1)
    ang = np.arange(maxpos)[:, None] * freqs[None, :]
    cos = torch.tensor(np.cos(ang), dtype=torch.float32, device=DEV)
    sin = torch.tensor(np.sin(ang), dtype=torch.float32, device=DEV)
    qkv0 = qkv.clone()
    ops.rope_kv_write(qkv, H, Hkv, hd, (cos, sin, hd), ctx.positions, ctx.row_of_token, kc, vc, table, page)
    out = torch.empty(ctx.num_tokens, H * hd, dtype=dtype, device=DEV)
    scale = 1.0 / math.sqrt(hd)
    ops.paged_attention(qkv, out, H, Hkv, hd, kc, vc, table, page, ctx, scale, window)
    if 1 in q_lens and max(q_lens) > 1:
        # single tokens beside portions: the same without the lists of them (a context that brings none)
        ctx.single_tokens = ctx.portion_rows = None
        again = torch.empty_like(out)
        ops.paged_attention(qkv, again, H, Hkv, hd, kc, vc, table, page, ctx, scale, window)
        assert torch.equal(out, again)
    t0 = 0
    for b in range(B):
        q_len, s = q_lens[b], starts[b]
        rows = qkv0[t0:t0 + q_len].double().cpu().numpy()
        q = rows[:, :H * hd].reshape(q_len, H, hd)
        k_new = rows[:, H * hd:(H + Hkv) * hd].reshape(q_len, Hkv, hd)
        v_new = rows[:, (H + Hkv) * hd:].reshape(q_len, Hkv, hd)
        pos = np.arange(s, s + q_len)
        q_rot = plain_llama.rope(q, pos, freqs)
        k_rot = plain_llama.rope(k_new, pos, freqs)
        if dtype == torch.bfloat16:                  # the cache holds rounded keys; q is rounded in place
            k_rot = torch.tensor(k_rot).to(torch.bfloat16).double().numpy()
            q_rot = torch.tensor(q_rot).to(torch.bfloat16).double().numpy()
        k_all = np.concatenate([hist_k[b][:s].double().numpy(), k_rot])
        v_all = np.concatenate([hist_v[b][:s].double().numpy(), v_new])
        # whole-sequence attention with dummy queries for the cached part
        q_all = np.concatenate([np.zeros((s, H, hd)), q_rot])
        got = out[t0:t0 + q_len].double().cpu().numpy().reshape(q_len, H, hd)
        lim = 1e-5 if dtype == torch.float32 else 2e-2
        if kv_heads is None:
            ref = plain_llama.attention(q_all, k_all, v_all, scale, window or None)[s:]
            assert np.max(np.abs(got - ref)) < lim, (case, window, np.max(np.abs(got - ref)))
        else:
            G = H // Hkv
            for g in kv_heads:                       # a kv head with its group of query heads
                ref = plain_llama.attention(q_all[:, g * G:(g + 1) * G], k_all[:, g:g + 1], v_all[:, g:g + 1], scale, window or None)[s:]
                err = np.max(np.abs(got[:, g * G:(g + 1) * G] - ref))
                assert err < lim, (case, window, g, err)
        # q was rotated in place
        got_q = qkv[t0:t0 + q_len, :H * hd].double().cpu().numpy().reshape(q_len, H, hd)
        assert np.max(np.abs(got_q - q_rot)) < (1e-5 if dtype == torch.float32 else 1e-6 + 2e-2)
        t0 += q_len


@pytest.mark.parametrize("B,H,Hkv,hd,page,K", [(1, 4, 2, 16, 16, 64), (5, 5, 1, 32, 8, 160), (8, 32, 8, 64, 16, 2048),
                                                (33, 6, 2, 128, 16, 96), (64, 3, 3, 48, 16, 224),
                                                # 33..64 tokens: the kernel that shares the activations through LDS
                                                (40, 32, 8, 128, 16, 4096), (64, 32, 8, 64, 16, 2048), (49, 12, 4, 128, 32, 544),
                                                (32, 8, 2, 64, 16, 512)])
def test_fused_projection_rotation_and_cache_write(ops, monkeypatch, B, H, Hkv, hd, page, K):
    """The one-kernel form for single tokens equals projection, then rope_kv_write.  (33 tokens and
    more: the kernel with the activations in LDS, here whatever the number of columns.)"""
    monkeypatch.setattr(ops, "QKV_ROPE_LDS_MIN_COLUMNS", 0)
    _check_fused_projection(ops, B, H, Hkv, hd, page, K)


@pytest.mark.parametrize("B,H,Hkv,hd,page,K", [
    (17, 8, 2, 64, 16, 512), (20, 5, 5, 48, 8, 224), (32, 32, 8, 128, 16, 1024),     # blocks of 32 columns
    (24, 96, 24, 128, 16, 128),                                                      # 18432 columns: blocks of 64
    (64, 48, 12, 128, 16, 256), (40, 40, 40, 80, 16, 96)])                           # more than 32 rows: 64 from 8208 columns on
def test_fused_projection_through_lds_from_17_tokens_and_in_wider_blocks(ops, monkeypatch, B, H, Hkv, hd, page, K):
    """The kernel with the activations in LDS, as it is taken for large weights from 17 tokens on,
    and with blocks of 64 columns where those of 32 would not all run at once."""
    monkeypatch.setattr(ops, "QKV_ROPE_LDS_MIN_COLUMNS", 0)
    monkeypatch.setattr(ops, "QKV_ROPE_LDS_LARGE", 0)
    lib, taken = ops._lib(), []
    entry = lib.ri_gemm_rows_qkv_rope
    monkeypatch.setattr(lib, "ri_gemm_rows_qkv_rope", lambda *a: taken.append(1) or entry(*a))
    _check_fused_projection(ops, B, H, Hkv, hd, page, K)
    assert taken


@pytest.mark.parametrize("q_lens,starts,H,Hkv,hd,page,K,parts", [
    ([65], [0], 4, 2, 16, 16, 64, 1), ([40, 1, 60, 33], [5, 30, 16, 0], 8, 2, 64, 16, 1024, 4), ([129], [15], 6, 6, 48, 32, 576, 2),
    ([1] * 70, [3] * 70, 4, 4, 32, 16, 4096, 8), ([64, 200], [0, 48], 12, 4, 128, 16, 1344, 2)])
def test_projection_in_slices_rotation_and_cache_write(ops, q_lens, starts, H, Hkv, hd, page, K, parts):
    """More than 64 tokens: the product over slices of K and the kernel that adds, rotates and writes, against
    projection and rope_kv_write; whole groups of 16 values and single ones, a padding token."""
    B, T = len(q_lens), sum(q_lens)
    qkv, kc, vc, table, ctx, _, _ = _paged_setup(torch.bfloat16, B, H, Hkv, hd, page, q_lens, starts, seed=K, num_pages=640)
    ctx.row_of_token[T // 2] = -1
    x, w = rnd(T, K, dtype=torch.bfloat16, seed=50), rnd((H + 2 * Hkv) * hd, K, dtype=torch.bfloat16, seed=51, scale=0.05)
    ang = np.arange(512)[:, None] * plain_llama.rope_frequencies(hd, 10000.0, None)[None, :]
    rotary = tuple(torch.tensor(f(ang), dtype=torch.float32, device=DEV) for f in (np.cos, np.sin)) + (hd,)
    wf = ops.qkv_rope_weight(w, hd)
    assert ops._mid_plan(T, (H + 2 * Hkv) * hd, K, False, True)[0] == parts
    kc1, vc1, kc2, vc2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    ref, got = torch.zeros_like(qkv), torch.zeros_like(qkv)
    ops.linear(x, w, ref)
    ops.rope_kv_write(ref, H, Hkv, hd, rotary, ctx.positions, ctx.row_of_token, kc1, vc1, table, page)
    assert ops.qkv_rope_split(x, wf, got, H, Hkv, hd, rotary, ctx.positions, ctx.row_of_token, kc2, vc2, table, page, Workspace(torch.device(DEV)))
    live = (ctx.row_of_token >= 0).cpu()
    big = max(1.0, ref[live].float().abs().max().item() / 2)       # two roundings of the largest sum against one
    assert torch.allclose(got[live, :H * hd].float(), ref[live, :H * hd].float(), atol=2e-2 * big, rtol=2e-2)
    assert torch.equal(torch.isnan(kc2), torch.isnan(kc1)) and torch.equal(torch.isnan(vc2), torch.isnan(vc1))
    for a, b in ((kc2, kc1), (vc2, vc1)):
        assert torch.allclose(torch.nan_to_num(a.float()), torch.nan_to_num(b.float()), atol=2e-2 * big, rtol=2e-2)
    assert torch.all(got[~live] == 0)                              # the padding token


@pytest.mark.parametrize("M,N,K", [(65, 16, 64), (127, 112, 320), (128, 4096, 64), (129, 2064, 1088), (300, 528, 4096), (513, 240, 704)])
def test_products_of_some_hundred_rows(ops, M, N, K):
    """Slices of K and the gate/up product with its activation, at the edges of blocks, tiles and slices."""
    xb = rnd(M, K + 16, dtype=torch.bfloat16, seed=M)
    x, w = xb[:, 8:K + 8], rnd(N, K, dtype=torch.bfloat16, seed=N)
    ref = x.double() @ w.double().t()
    got = ops.linear_delta(x, w, Workspace(torch.device(DEV)), "t", ops.tile_weight(w))
    parts = ops._mid_plan(M, N, K, False)[0]
    assert parts >= 1 and (got.dim() == 3) == (parts > 1)
    if parts > 1:                                                  # 32-bit sums of K products of numbers around one
        assert got.shape == (parts, M, N)
        assert torch.allclose(got.double().sum(0), ref, rtol=0, atol=2e-6 * K ** 0.5 * 4)
    I = N // 32 * 16
    if I:
        w, ref = w[:2 * I], ref[:, :2 * I]
        out = torch.full((M, I), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert ops._mid_plan(M, I, K, True)[0] == 1
        ops.linear_swiglu(x, w, out, None, ops.tile_weight(w))
        want = torch.nn.functional.silu(ref[:, :I]) * ref[:, I:]
        assert torch.allclose(out.double(), want, rtol=2.0 ** -8, atol=2.0 ** -8 + 1e-5 * K ** 0.5)


@pytest.mark.parametrize("parts,wide", [(p, w) for p in (2, 3, 5, 8) for w in (0, 1)])
def test_slices_of_any_number_in_blocks_of_either_width(ops, monkeypatch, parts, wide):
    """What the plan may choose for products of some hundred rows: blocks that are no whole number of rounds, a last
    block of columns that is not whole, slices of unequal length and one without any."""
    monkeypatch.setattr(ops, "_mid_plan", lambda *a: (parts, wide))
    monkeypatch.setattr(ops, "_slices_pay", lambda *a: True)
    for M, N, K in ((129, 2064, 1088), (300, 720, 832), (200, 272, 576)):
        x, w = rnd(M, K, dtype=torch.bfloat16, seed=M), rnd(N, K, dtype=torch.bfloat16, seed=N)
        got = ops.linear_delta(x, w, Workspace(torch.device(DEV)), "t", ops.tile_weight(w))
        assert got.shape == (parts, M, N)                          # 32-bit sums of K products of numbers around one
        assert torch.allclose(got.double().sum(0), x.double() @ w.double().t(), rtol=0, atol=2e-6 * K ** 0.5 * 4)


@pytest.mark.parametrize("M,N,K,rotated,plan", [
    (256, 4096, 14336, False, (4, 1)), (384, 2560, 2560, False, (2, 0)), (100, 2048, 2048, False, (8, 0)), (256, 2048, 2048, False, (4, 0)),
    (224, 6144, 4096, True, (2, 1)), (65, 5120, 3072, True, (3, 0)), (65, 128, 64, True, (1, 0)), (2048, 4096, 4096, False, (0, 1))])
def test_plan_of_products_of_some_hundred_rows(ops, M, N, K, rotated, plan):
    """The slices and widths that were fastest, or next to it, of all that were measured."""
    assert ops._mid_plan(M, N, K, False, rotated) == plan


def test_where_slices_pay(ops):
    """Sizes on both sides of each line."""
    assert all(ops._slices_pay(*a) for a in ((512, 1024, 1024), (113, 4608, 640), (700, 2048, 2048), (2048, 896, 4864)))
    assert not any(ops._slices_pay(*a) for a in ((768, 1024, 1024), (160, 4608, 640), (640, 1536, 1536), (1025, 2048, 2048)))
    assert all(ops.qkv_split_pays(*a) for a in ((256, 6144, 4096), (307, 5120, 3072), (256, 3072, 2048), (195, 1536, 1024)))
    assert not any(ops.qkv_split_pays(*a) for a in ((384, 5120, 3072), (257, 3072, 2048), (100, 2048, 2304), (300, 1536, 1024), (128, 6144, 2048), (100, 12288, 4096)))


@pytest.mark.parametrize("M,I,K,plan", [(128, 8192, 2048, (1, 0)), (128, 8704, 4096, (1, 1)), (128, 11008, 4096, (1, 1)), (256, 5632, 4096, (1, 1)),
                                        (384, 5376, 2048, (0, 1)), (320, 8192, 2048, (0, 1))])
def test_plan_of_gate_up_products(ops, M, I, K, plan):
    """Narrow blocks where they fit the units once, wide ones where those do, each XCD taking whole columns of blocks."""
    assert ops._mid_plan(M, I, K, True) == plan


def _check_fused_projection(ops, B, H, Hkv, hd, page, K):
    q_lens, starts = [1] * B, [(7 * i + 3) % 60 for i in range(B)]
    qkv, kc, vc, table, ctx, _, _ = _paged_setup(torch.bfloat16, B, H, Hkv, hd, page, q_lens, starts, seed=K, num_pages=640)
    ctx.row_of_token[B // 2] = -1 if B > 2 else ctx.row_of_token[B // 2]      # a padding row touches nothing
    x = rnd(B, K, dtype=torch.bfloat16, seed=50)
    w = rnd((H + 2 * Hkv) * hd, K, dtype=torch.bfloat16, seed=51, scale=0.05)
    freqs = plain_llama.rope_frequencies(hd, 10000.0, None)
    ang = np.arange(128)[:, None] * freqs[None, :]
    rotary = (torch.tensor(np.cos(ang), dtype=torch.float32, device=DEV), torch.tensor(np.sin(ang), dtype=torch.float32, device=DEV), hd)
    wf = ops.qkv_rope_weight(w, hd)
    assert wf is not None
    kc1, vc1, kc2, vc2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    ref = torch.zeros_like(qkv)
    ops.linear(x, w, ref)
    ops.rope_kv_write(ref, H, Hkv, hd, rotary, ctx.positions, ctx.row_of_token, kc1, vc1, table, page)
    got = torch.zeros_like(qkv)
    assert ops.qkv_rope_fused(x, wf, got, H, Hkv, hd, rotary, ctx.positions, ctx.row_of_token, kc2, vc2, table, page)
    live = (ctx.row_of_token >= 0).cpu()
    nn = torch.nan_to_num
    # the separate kernels round the projection to bfloat16 before rotating; the fused one does not:
    # two roundings of values up to the largest sum against one
    big = max(1.0, ref[live].float().abs().max().item() / 2)
    assert torch.allclose(got[live, :H * hd].float(), ref[live, :H * hd].float(), atol=2e-2 * big, rtol=2e-2)
    assert torch.allclose(nn(kc2).float(), nn(kc1).float(), atol=2e-2 * big, rtol=2e-2)
    assert torch.allclose(nn(vc2).float(), nn(vc1).float(), atol=1e-2, rtol=1e-2)
    # and against the product in 64-bit, rotated: one rounding to bfloat16
    full = x.double() @ w.double().t()
    q = full[:, :H * hd].view(B, H, hd)
    c, sn = rotary[0][ctx.positions.long()].double()[:, None, :], rotary[1][ctx.positions.long()].double()[:, None, :]
    a, b = q[..., :hd // 2], q[..., hd // 2:]
    want = torch.cat([a * c - b * sn, a * sn + b * c], -1).reshape(B, H * hd)
    assert torch.allclose(got[live, :H * hd].double(), want[live], atol=1e-3, rtol=2.0 ** -8)
    assert torch.equal(torch.isnan(kc2), torch.isnan(kc1)) and torch.equal(torch.isnan(vc2), torch.isnan(vc1))
    # against 64-bit arithmetic the fused form is the closer one
    x64, w64 = x.double().cpu().numpy(), w.double().cpu().numpy()
    qf = (x64 @ w64.T)[:, :H * hd].reshape(B, H, hd)
    for b in np.nonzero(live.numpy())[0][:4]:
        want = plain_llama.rope(qf[b:b + 1], np.array([starts[b]]), freqs)[0].reshape(-1)
        # one bfloat16 rounding: half a unit in the 8th bit of each value
        assert np.all(np.abs(got[b, :H * hd].double().cpu().numpy() - want) <= 2.0 ** -8 * np.maximum(1.0, np.abs(want)))


@pytest.mark.parametrize("M,K", [(17, 32), (32, 96), (33, 64), (48, 160), (49, 1056), (64, 2080), (20, 4128), (37, 8160), (4, 32), (9, 96), (15, 1056), (16, 8160)])
def test_products_of_some_rows_through_the_ring(ops, M, K):
    """Fewer stretches of 64 than groups and stages, an odd last step, 16 columns and edges of blocks; rows beside and beyond which all is NaN; every number of groups
    and slices: partial sums, gate/up, whole products of one and two tiles a wave."""
    lib = ops._lib()
    buf = torch.full((M + 2, K + 64), float("nan"), dtype=torch.bfloat16, device=DEV)
    x = buf[1:M + 1, 32:K + 32]
    x.copy_(rnd(M, K, dtype=torch.bfloat16, seed=1))
    N = 272
    w = rnd(2 * N, K, dtype=torch.bfloat16, seed=2, scale=0.2)
    wt, wt1 = ops.tile_weight(w), ops.tile_weight(w[:N].contiguous())
    ref = x.double() @ w.double().t()
    # K additions in 32 bits, each off by at most 2^-23 of a partial sum; of random signs those are of the size of the root of the sum of squares (eight
    # times that never), and the errors' signs are random as well but for the bias of a truncation, half of them.  One product missing or twice shows: it is
    # 1 / sqrt(K) of that root, far above.
    tol = K * 2.0 ** -23 * ((x.double() ** 2) @ (w.double() ** 2).t()).sqrt()
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    st = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for groups in (1, 2, 4):
        for parts, nt in ((1, 1), (1, 2), (2, 1), (3, 1), (8, 1)):
            out = torch.full((parts, M + 1, N), float("nan"), device=DEV)
            assert lib.ri_gemm_rows_bf16(p(x), x.stride(0), p(wt1), p(out), N, M, N, K, ops.F32, 0, parts,
                                         ctypes.c_longlong((M + 1) * N if parts > 1 else 0), nt, groups, st) == 0
            assert torch.all((out[:, :M].double().sum(0) - ref[:, :N]).abs() <= tol[:, :N]), (groups, parts, nt)
            assert torch.isnan(out[:, M]).all()
        out = torch.full((M + 1, N), float("nan"), dtype=torch.bfloat16, device=DEV)
        assert lib.ri_gemm_rows_bf16(p(x), x.stride(0), p(wt), p(out), N, M, N, K, ops.BF16, 1, 1, ctypes.c_longlong(0), 1, groups, st) == 0
        want = torch.nn.functional.silu(ref[:, :N]) * ref[:, N:]
        assert torch.all((out[:M].double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * want.abs().max()), groups
        assert torch.isnan(out[M]).all()
    x[3, K - 1] = float("inf")
    bad = torch.empty(M, N, device=DEV)
    assert lib.ri_gemm_rows_bf16(p(x), x.stride(0), p(wt1), p(bad), N, M, N, K, ops.F32, 0, 1, ctypes.c_longlong(0), 1, 2, st) == 0
    rest = [i for i in range(M) if i != 3]
    assert torch.all((bad[rest].double() - ref[rest, :N]).abs() <= tol[rest, :N]) and not torch.isfinite(bad[3]).any()


@pytest.mark.parametrize("M,N,K,delta,whole", [(9, 2048, 8192, (8, 4), None), (12, 1024, 544, (8, 1), None), (16, 3072, 1056, (8, 1), None), (8, 2048, 2048, None, None),
                                               (9, 4096, 2080, (8, 2), None), (16, 5136, 2048, None, (1, 4)), (7, 5120, 512, None, None), (8, 5120, 512, None, (1, 4)),
                                               (10, 5120, 512, (8, 1), (1, 4)), (10, 960, 1024, None, None),
                                               (11, 8208, 256, None, None), (12, 8208, 256, None, (1, 4)), (9, 16400, 4128, None, (2, 1)), (17, 272, 96, None, (1, 4)),
                                               (64, 8208, 160, None, (1, 2))])
def test_where_products_take_the_ring(ops, monkeypatch, M, N, K, delta, whole):
    """Slices for a norm, whole products and gate/up on both sides of the lines between the kernels, against 64-bit sums."""
    lib, taken, entry = ops._lib(), [], ops._lib().ri_gemm_rows_bf16
    monkeypatch.setattr(lib, "ri_gemm_rows_bf16", lambda *a: taken.append((a[10], a[12], a[13])) or entry(*a))
    x = rnd(M, K, dtype=torch.bfloat16, seed=1)
    w = rnd(N, K, dtype=torch.bfloat16, seed=2, scale=0.1)
    wt, ws = ops.tile_weight(w), Workspace(torch.device(DEV))
    ref = x.double() @ w.double().t()
    tol = K * 2.0 ** -23 * ((x.double() ** 2) @ (w.double() ** 2).t()).sqrt()      # as for the ring itself
    out = torch.full((M, N), float("nan"), device=DEV)
    ops.linear(x, w, out, wt)
    assert taken == ([(1,) + whole] if whole else [])
    assert torch.all((out.double() - ref).abs() <= tol)
    if M <= 16:
        taken.clear()
        got = ops.linear_delta(x, w, ws, "t", wt, torch.float32)
        assert taken == ([(delta[0], 1, delta[1])] if delta else [(1,) + whole] if whole and got.dim() == 2 else [])
        assert torch.all(((got.double().sum(0) if got.dim() == 3 else got.double()) - ref).abs() <= tol)
    half = N // 2 // 16 * 16
    gu, act = w[:2 * half].contiguous(), torch.full((M, half), float("nan"), dtype=torch.bfloat16, device=DEV)
    taken.clear()
    ops.linear_swiglu(x, gu, act, None, ops.tile_weight(gu))
    assert len(taken) == (M >= 9 and half >= 4096)
    want = torch.nn.functional.silu(ref[:, :half]) * ref[:, half:2 * half]
    assert torch.all((act.double() - want).abs() <= 2.0 ** -8 * want.abs() + 1e-4 * want.abs().max())


@pytest.mark.parametrize("B,H,Hkv,hd,K", [(9, 32, 8, 128, 2400), (16, 24, 8, 128, 3072), (12, 70, 10, 128, 1536)])
def test_fused_projection_of_up_to_sixteen_tokens_through_the_ring(ops, monkeypatch, B, H, Hkv, hd, K):
    lib, taken = ops._lib(), []
    entry = lib.ri_gemm_rows_qkv_rope
    monkeypatch.setattr(lib, "ri_gemm_rows_qkv_rope", lambda *a: taken.append(1) or entry(*a))
    _check_fused_projection(ops, B, H, Hkv, hd, 64, K)
    assert taken == [1]


@pytest.mark.parametrize("M,N,K", [(1, 16, 32), (8, 48, 96), (3, 2048, 2048), (8, 2048, 2080), (7, 1024, 4128), (4, 3072, 3104), (2, 4096, 1056),
                                   (8, 5120, 2048), (1, 6144, 8192), (8, 2048, 8224)])
def test_the_product_before_a_norm_in_pairs_of_steps(ops, M, N, K):
    """Eight columns a block, two steps of K a load: an odd number of steps, fewer than the waves, whole batches and parts of one; what lies beside the
    rows in a wider buffer, and a row that is not finite, touch nothing else."""
    lib = ops._lib()
    assert lib.ri_gemm_skinny_residual_parts(M, N) == N // 8
    buf = torch.full((M + 1, K + 64), float("nan"), dtype=torch.bfloat16, device=DEV)
    act = buf[:M, 32:K + 32]
    act.copy_(rnd(M, K, dtype=torch.bfloat16, seed=1))
    w = rnd(N, K, dtype=torch.bfloat16, seed=2, scale=0.05)
    wt, wn, x0, ws = ops.tile_weight(w), 1.0 + rnd(N, seed=3, scale=0.1), rnd(M, N, seed=4), Workspace(DEV)
    x = x0.clone()
    a, ssq = ops.linear_residual(act, w, wt, x, wn, ws, "t")
    a, ssq = a.clone(), ssq.clone()
    prod = act.double() @ w.double().t()
    # K additions in 32 bits, each off by at most 2^-23 of a partial sum, which of random signs is of the size of the root of the sum of squares;
    # and the addition to x
    mag = ((act.double() ** 2) @ (w.double() ** 2).t()).sqrt()
    assert torch.all((x.double() - x0.double() - prod).abs() <= K * 2.0 ** -23 * mag + 2.0 ** -23 * x.double().abs())
    assert torch.equal(a, (x * wn).to(torch.bfloat16)) and tuple(ssq.shape) == (M, N // 8)
    assert torch.allclose(ssq.double(), (x.double() ** 2).view(M, N // 8, 8).sum(2), rtol=1e-6)
    if M > 1:
        act[1, K - 1] = float("inf")
        y = x0.clone()
        ops.linear_residual(act, w, wt, y, wn, ws, "u")
        rest = [i for i in range(M) if i != 1]
        assert torch.equal(y[rest], x[rest]) and not torch.isfinite(y[1]).any()


@pytest.mark.parametrize("M,N", [(1, 3072), (3, 3072), (2, 64)])
def test_the_product_before_a_norm_of_rows_further_apart_than_32_bit_distances_reach(ops, M, N):
    far, K = (1 << 27) + 8, 1056
    buf = torch.empty((M - 1) * far + K, dtype=torch.bfloat16, device=DEV)
    act = buf.as_strided((M, K), (far, 1))
    act.copy_(rnd(M, K, dtype=torch.bfloat16, seed=1))
    w = rnd(N, K, dtype=torch.bfloat16, seed=2, scale=0.05)
    wt, wn, ws = ops.tile_weight(w), 1.0 + rnd(N, seed=3, scale=0.1), Workspace(DEV)
    x = torch.zeros(M, N, device=DEV)
    a, ssq = ops.linear_residual(act, w, wt, x, wn, ws, "t")
    mag = ((act.double() ** 2) @ (w.double() ** 2).t()).sqrt()                  # the bound of the test above
    assert torch.all((x.double() - act.double() @ w.double().t()).abs() <= K * 2.0 ** -23 * mag)
    assert torch.equal(a, (x * wn).to(torch.bfloat16))
    assert torch.allclose(ssq.double().sum(1), (x.double() ** 2).sum(1), rtol=1e-5)


@pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("M,N,K,I,eps", [(1, 64, 64, 176, 1e-5), (5, 384, 1056, 416, 1e-6), (8, 2048, 8192, 1024, 1e-5),
                                         (16, 4096, 14336, 512, 1e-5), (13, 160, 416, 48, 1e-5), (2, 2304, 2304, 1184, 1e-6)])
def test_a_norm_done_by_the_products_around_it(ops, wdtype, M, N, K, I, eps):
    """Few rows: the product before a norm adds its sums to the residual stream and leaves
    x * w and partial sums of x^2; the products after it (plain, SwiGLU) multiply their sums by
    rsqrt(mean(x^2) + eps).  Against 64-bit arithmetic, and against the norm's own kernel."""
    act = rnd(M, K, dtype=torch.bfloat16, seed=60)
    w = rnd(N, K, dtype=torch.bfloat16, seed=61, scale=0.05)
    wt = ops.tile_weight(w)
    x = rnd(M, N, seed=62, scale=2.0)
    wn = (1.0 + rnd(N, seed=63, scale=0.1)).to(wdtype)
    assert ops.linear_residual_ok(M, w, wt, wn) and not ops.linear_residual_ok(ops.DEFERRED_NORM_MAX_ROWS + 1, w, wt, wn)
    ws = Workspace(DEV)
    x0 = x.clone()
    a, ssq = ops.linear_residual(act, w, wt, x, wn, ws, "t")
    want_x = x0.double() + act.double() @ w.double().t()
    assert a.dtype == torch.bfloat16 and tuple(a.shape) == (M, N) and ssq.shape[0] == M
    assert torch.allclose(x.double(), want_x, rtol=0, atol=2e-5 * max(1.0, want_x.abs().max().item()))
    assert torch.equal(a, (x * wn.float()).to(torch.bfloat16))                    # rounded once, from the 32-bit sum
    assert torch.allclose(ssq.double().sum(1), (x.double() ** 2).sum(1), rtol=1e-5)
    # the products behind the norm
    n64 = want_x * torch.rsqrt((want_x ** 2).mean(-1, keepdim=True) + eps) * wn.double()
    w2 = rnd(2 * I, N, dtype=torch.bfloat16, seed=64, scale=0.05)
    w2t = ops.tile_weight(w2)
    out = torch.empty(M, I, dtype=torch.bfloat16, device=DEV)
    ops.linear_swiglu(a, w2, out, None, w2t, scale=(ssq, eps))
    g, u = n64 @ w2[:I].double().t(), n64 @ w2[I:].double().t()
    ref = g / (1 + torch.exp(-g)) * u
    assert torch.allclose(out.double(), ref, rtol=1.6e-2, atol=1.6e-2 * max(1.0, ref.abs().max().item()) / 4)
    for odt, tiled in ((torch.float32, w2t), (torch.bfloat16, None)):
        lin = torch.empty(M, 2 * I, dtype=odt, device=DEV)
        ops.linear(a, w2, lin, tiled, scale=(ssq, eps))
        ref = n64 @ w2.double().t()
        assert torch.allclose(lin.double(), ref, rtol=1.6e-2, atol=1.6e-2 * max(1.0, ref.abs().max().item()) / 4)
    # the same through the norm's own kernel: rows rounded after the factor instead of before it
    normed = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    xr = x0.clone()
    delta = torch.empty(M, N, dtype=torch.float32, device=DEV)
    ops.linear(act, w, delta, wt)
    ops.add_rmsnorm(xr, delta, wn, eps, normed)
    assert torch.allclose(xr, x, rtol=0, atol=1e-5 * max(1.0, x.abs().max().item()))
    lin2 = torch.empty(M, 2 * I, dtype=torch.float32, device=DEV)
    ops.linear(normed, w2, lin2, w2t)
    lin = torch.empty(M, 2 * I, dtype=torch.float32, device=DEV)
    ops.linear(a, w2, lin, w2t, scale=(ssq, eps))
    assert torch.allclose(lin, lin2, rtol=2e-2, atol=2e-2 * max(1.0, lin2.abs().max().item()) / 4)
    # more rows than the few-row kernel takes: the factors have no product to go with
    big = rnd(80, N, dtype=torch.bfloat16, seed=65)
    with pytest.raises(ops.KernelError, match="deferred norm"):
        ops.linear(big, w2, torch.empty(80, 2 * I, dtype=torch.float32, device=DEV), w2t,
                   scale=(torch.ones(80, 4, device=DEV), eps))


@pytest.mark.parametrize("B,H,Hkv,hd,K", [(1, 4, 2, 64, 256), (2, 6, 2, 128, 384), (8, 32, 8, 64, 2048), (16, 3, 3, 48, 96),
                                          (13, 5, 1, 32, 160)])
def test_fused_projection_finishes_a_deferred_norm(ops, B, H, Hkv, hd, K):
    """Single tokens: the fused projection, rotation and cache write on rows x * w with the factor
    rsqrt(mean(x^2) + eps) applied to its sums equals the same kernel on rows normalised before."""
    page, eps = 16, 1e-5
    q_lens, starts = [1] * B, [(11 * i + 5) % 60 for i in range(B)]
    qkv, kc, vc, table, ctx, _, _ = _paged_setup(torch.bfloat16, B, H, Hkv, hd, page, q_lens, starts, seed=K, num_pages=64)
    x = rnd(B, K, seed=70, scale=2.0)
    wn = (1.0 + rnd(K, seed=72, scale=0.1)).to(torch.bfloat16)
    w = rnd((H + 2 * Hkv) * hd, K, dtype=torch.bfloat16, seed=73, scale=0.05)
    freqs = plain_llama.rope_frequencies(hd, 10000.0, None)
    ang = np.arange(128)[:, None] * freqs[None, :]
    rotary = (torch.tensor(np.cos(ang), dtype=torch.float32, device=DEV), torch.tensor(np.sin(ang), dtype=torch.float32, device=DEV), hd)
    wf = ops.qkv_rope_weight(w, hd)
    kc1, vc1, kc2, vc2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
    normed = torch.empty(B, K, dtype=torch.bfloat16, device=DEV)
    ops.add_rmsnorm(x.clone(), None, wn, eps, normed)
    ref = torch.zeros_like(qkv)
    assert ops.qkv_rope_fused(normed, wf, ref, H, Hkv, hd, rotary, ctx.positions, ctx.row_of_token, kc1, vc1, table, page)
    # the deferred form: rows x * w, sums of squares in 7 uneven parts
    a = (x * wn.float()).to(torch.bfloat16)
    sq = x * x
    cuts = [0, 1, K // 7, K // 3, K // 2, K - 9, K - 1, K]
    ssq = torch.stack([sq[:, lo:hi].sum(1) for lo, hi in zip(cuts[:-1], cuts[1:])], dim=1).contiguous()
    got = torch.zeros_like(qkv)
    assert ops.qkv_rope_fused(a, wf, got, H, Hkv, hd, rotary, ctx.positions, ctx.row_of_token, kc2, vc2, table, page,
                              scale=(ssq, eps))
    nn = torch.nan_to_num
    assert torch.allclose(got[:, :H * hd].float(), ref[:, :H * hd].float(), atol=3e-2, rtol=3e-2)
    assert torch.allclose(nn(kc2).float(), nn(kc1).float(), atol=3e-2, rtol=3e-2)
    assert torch.allclose(nn(vc2).float(), nn(vc1).float(), atol=3e-2, rtol=3e-2)
    assert torch.equal(torch.isnan(kc2), torch.isnan(kc1)) and torch.equal(torch.isnan(vc2), torch.isnan(vc1))
    # against 64-bit arithmetic
    x64 = x.double()
    n = x64 * torch.rsqrt((x64 * x64).mean(-1, keepdim=True) + eps) * wn.double()
    qf = (n.cpu().numpy() @ w.double().cpu().numpy().T)[:, :H * hd].reshape(B, H, hd)
    for b in range(B):
        want = plain_llama.rope(qf[b:b + 1], np.array([starts[b]]), freqs)[0].reshape(-1)
        assert np.all(np.abs(got[b, :H * hd].double().cpu().numpy() - want) <= 1.6e-2 * np.maximum(1.0, np.abs(want)))


@pytest.mark.parametrize("q_len", [1, 5, 40])
def test_attention_finds_a_far_key(ops, q_len):
    """One key among hundreds is made to stand out for the last query: the output must be that
    key's value (a fault at a page edge, in the split of long histories or in a tile's key order
    would miss it).  q_len 1 takes the split-key kernel, longer portions the tiled one."""
    B, H, Hkv, hd, page = 1, 4, 2, 64, 16
    start = 512 - (q_len - 1)
    for far in (0, 3, 4, 7, 8, 15, 16, 31, 32, 127, 128, 255, 256, 300, 383, 384, 511):
        qkv, kc, vc, table, ctx, hk, hv = _paged_setup(torch.bfloat16, B, H, Hkv, hd, page, [q_len], [start], seed=far)
        ops.rope_kv_write(qkv, H, Hkv, hd, None, ctx.positions, ctx.row_of_token, kc, vc, table, page)
        blk = int(table[0, far // page])
        q = qkv[q_len - 1, :H * hd].view(H, hd)
        for g in range(Hkv):
            kc[blk, g, far % page] = (q[g * (H // Hkv)] * 4.0)
        out = torch.empty(q_len, H * hd, dtype=torch.bfloat16, device=DEV)
        ops.paged_attention(qkv, out, H, Hkv, hd, kc, vc, table, page, ctx, 1.0, 0)
        for g in range(Hkv):
            h = g * (H // Hkv)
            assert torch.allclose(out[q_len - 1, h * hd:(h + 1) * hd].float(), vc[blk, g, :, far % page].float(), atol=2e-2), far


@pytest.mark.parametrize("H,Hkv,hd,page,window", [(8, 2, 64, 16, 0), (6, 1, 128, 16, 0), (5, 5, 48, 8, 70), (16, 2, 80, 16, 0)])
def test_exact_attention_of_a_portion_does_not_depend_on_the_cut(ops, H, Hkv, hd, page, window):
    """The tiled kernel of the 32-bit path: a token's output is the same bits whether its portion
    is the whole prompt's tail or cut in two (key blocks are aligned to absolute positions, a
    row's sums go in a fixed order), it agrees with the generic kernel to rounding, and it finds
    one far key that is made to stand out."""
    from types import SimpleNamespace
    start, n = 200, 37
    qkv, kc, vc, table, ctx, hk, hv = _paged_setup(torch.float32, 1, H, Hkv, hd, page, [n], [start], seed=hd)
    ops.rope_kv_write(qkv, H, Hkv, hd, None, ctx.positions, ctx.row_of_token, kc, vc, table, page)
    scale = 1.0 / math.sqrt(hd)

    def portion(lo, hi):
        c = SimpleNamespace(num_tokens=hi - lo, num_rows=1, positions=ctx.positions[lo:hi].contiguous(),
                            row_of_token=ctx.row_of_token[lo:hi].contiguous(),
                            kv_lens=torch.tensor([start + hi], dtype=torch.int32, device=DEV),
                            q_start=torch.tensor([start + lo], dtype=torch.int32, device=DEV),
                            cu_q=torch.tensor([0, hi - lo], dtype=torch.int32, device=DEV),
                            max_q_len=hi - lo, max_kv_len=start + hi, decode_only=False,
                            host_q_lens=[hi - lo], host_q_start=[start + lo], host_kv_lens=[start + hi], workspace=ctx.workspace)
        o = torch.full((hi - lo, H * hd), float("nan"), device=DEV)
        ops.paged_attention(qkv[lo:hi], o, H, Hkv, hd, kc, vc, table, page, c, scale, window)
        return o

    if window:
        # pages that lie below the window of the portion's first token have been given back
        table[0, :(start + 1 - window) // page] = -1
    whole = portion(0, n)
    assert torch.equal(torch.cat([portion(0, 20), portion(20, n)]), whole)
    assert torch.equal(torch.cat([portion(0, 2), portion(2, 35), portion(35, n)]), whole)
    # single tokens take the split-key kernel: the same bits again, alone or several in a step
    for i in (0, 1, 19, n - 1):
        assert torch.equal(portion(i, i + 1), whole[i:i + 1]), i
    rows = [3, 30, 11]
    c = SimpleNamespace(num_tokens=3, num_rows=3, positions=ctx.positions[rows].contiguous(),
                        row_of_token=torch.tensor([0, 1, 2], dtype=torch.int32, device=DEV),
                        kv_lens=torch.tensor([start + r + 1 for r in rows], dtype=torch.int32, device=DEV),
                        max_q_len=1, max_kv_len=start + n, decode_only=True, workspace=ctx.workspace)
    o = torch.full((3, H * hd), float("nan"), device=DEV)
    ops.paged_attention(qkv[rows].contiguous(), o, H, Hkv, hd, kc, vc, table[[0, 0, 0]].contiguous(), page, c, scale, window)
    assert torch.equal(o, whole[rows])
    generic = torch.empty_like(whole)
    lib = ops._lib()
    import ctypes
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    assert lib.ri_attention_generic(P(qkv), qkv.stride(0), P(generic), generic.stride(0), 0, P(kc), P(vc), kc.shape[0], page,
                                    H, Hkv, hd, P(table), table.shape[1], P(ctx.row_of_token), P(ctx.positions), P(ctx.kv_lens),
                                    n, ctypes.c_float(scale), window, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
    assert torch.allclose(whole, generic, rtol=0, atol=2e-6)
    # a far key for the last query (inside the window where there is one)
    G = H // Hkv
    for far in (0, 63, 64, 127, 199, 200, 235):
        if window and far < start + n - window:
            continue
        blk = int(table[0, far // page])
        saved = kc[blk, :, far % page].clone()
        q = qkv[n - 1, :H * hd].view(H, hd)
        for g in range(Hkv):
            kc[blk, g, far % page] = q[g * G] * (40.0 / float(q[g * G].norm()) ** 2) / scale
        o = portion(0, n)
        for g in range(Hkv):
            assert torch.allclose(o[n - 1, g * G * hd:(g * G + 1) * hd], vc[blk, g, :, far % page], atol=1e-4), far
        kc[blk, :, far % page] = saved


@pytest.mark.parametrize("hd", [20, 64, 128])
@pytest.mark.parametrize("size,scale", [(1.0, 2.0 ** 40), (2.0 ** -67, 2.0 ** 126)])
@pytest.mark.parametrize("single", [True, False])
def test_exact_attention_sums_are_a_chain_of_fused_multiply_adds(ops, hd, size, scale, single):
    """Bit for bit, products and sums below the smallest normal number kept.  Scores: of two keys one is random and the other scores what libm's fmaf gives
    for the first; at this scale half a unit between them moves the weights from one half each.  Weighted values: 50 keys of one score, whose weights are
    one, so the sum is the values' in ascending order, rounded at each."""
    fmaf = ctypes.CDLL("libm.so.6").fmaf
    fmaf.restype, fmaf.argtypes = ctypes.c_float, [ctypes.c_float] * 3
    H, page, n = 6, 16, 50
    g = torch.Generator().manual_seed(hd)
    q, k, v = torch.randn(H, hd, generator=g) * size, torch.randn(H, hd, generator=g) * size, torch.randn(H, n, hd, generator=g) * (1.0 if size == 1.0 else 2.0 ** -130)
    q[:, 0] = size
    want = torch.zeros(H)
    for h in range(H):
        s = 0.0
        for a, b in zip(q[h].tolist(), k[h].tolist()):
            s = fmaf(a, b, s)
        want[h] = s
    assert size == 1.0 or (want.abs() < 2.0 ** -126).any()
    total = torch.zeros(H, hd)
    for j in range(n):
        total = total + v[:, j]                      # 32-bit additions on the host
    kc, vc = torch.full((8, H, page, hd), float("nan"), device=DEV), torch.full((8, H, hd, page), float("nan"), device=DEV)
    kc[0, :, 0], kc[0, :, 1] = k.to(DEV), torch.cat([(want / size)[:, None], torch.zeros(H, hd - 1)], 1).to(DEV)     # (size is a power of two: exact)
    vc[0, :, :, 0], vc[0, :, :, 1] = 1.0, 0.0
    pages = torch.tensor([1, 2, 3, 4])
    for j in range(n):
        kc[int(pages[j // page]), :, j % page] = 0.0
        vc[int(pages[j // page]), :, :, j % page] = v[:, j].to(DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    # two rows: the two keys, and the 50; as single tokens, or each behind a token of a portion whose output nobody looks at
    rows, positions, first = ([0, 1], [1, n - 1], [1, n - 1]) if single else ([0, 0, 1, 1], [0, 1, n - 2, n - 1], [0, n - 2])
    ctx = SimpleNamespace(num_tokens=len(rows), num_rows=2, positions=i32(positions), row_of_token=i32(rows), kv_lens=i32([2, n]), q_start=i32(first),
                          cu_q=i32([0, 1, 2] if single else [0, 2, 4]), max_q_len=1 if single else 2, max_kv_len=n, decode_only=single, workspace=Workspace(DEV))
    table = i32([[0] * 4, [1, 2, 3, 4]])
    qkv = torch.zeros(len(rows), H * hd, device=DEV)
    at = [0, 1] if single else [1, 3]
    qkv[at[0]] = q.view(-1).to(DEV)
    out = torch.empty(len(rows), H * hd, device=DEV)
    ops.paged_attention(qkv, out, H, H, hd, kc, vc, table, page, ctx, scale, 0)
    assert torch.all(out[at[0]] == 0.5)
    assert torch.equal(out[at[1]].cpu().view(H, hd), total / n)


@pytest.mark.parametrize("H,Hkv,hd,page,window", [(8, 2, 64, 16, 0), (4, 4, 128, 4, 40)])
def test_exact_attention_of_portions_takes_values_from_any_address(ops, H, Hkv, hd, page, window):
    qkv, kc, vc, table, ctx, _, _ = _paged_setup(torch.float32, 2, H, Hkv, hd, page, [40, 70], [90, 0], seed=hd)
    ops.rope_kv_write(qkv, H, Hkv, hd, None, ctx.positions, ctx.row_of_token, kc, vc, table, page)
    want, got = (torch.full((110, H * hd), float("nan"), device=DEV) for _ in range(2))
    ops.paged_attention(qkv, want, H, Hkv, hd, kc, vc, table, page, ctx, 0.1, window)
    off = torch.empty(vc.numel() + 1, device=DEV)[1:].view(vc.shape)
    off.copy_(vc)
    assert off.data_ptr() % 16 == 4
    ops.paged_attention(qkv, got, H, Hkv, hd, kc, off, table, page, ctx, 0.1, window)
    assert torch.equal(got, want) and torch.isfinite(got).all()


@pytest.mark.parametrize("H,Hkv,hd,page,window", [(8, 2, 64, 16, 0), (40, 2, 80, 16, 0), (40, 2, 64, 4, 90), (3, 3, 4, 1, 0), (6, 2, 100, 5, 33), (32, 1, 128, 64, 0),
                                                  (12, 4, 128, 2, 0), (7, 1, 20, 128, 130), (34, 2, 128, 6, 0)])
def test_exact_attention_of_single_tokens_on_every_route(ops, H, Hkv, hd, page, window):
    """Tokens as part of portions, a block of keys a block, and all keys a block (many tokens, or few keys): the same bits, and
    64-bit arithmetic to 32-bit rounding.  Keys end in a block of 64, at its edge, and one past it; slots never written are NaN."""
    from types import SimpleNamespace
    ends = [1, 2, 63, 64, 65, 127, 128, 129, 192, 200, 260]
    starts = [max(0, e - 20) for e in ends]
    q_lens = [e - s for e, s in zip(ends, starts)]
    qkv, kc, vc, table, ctx, hk, hv = _paged_setup(torch.float32, len(ends), H, Hkv, hd, page, q_lens, starts, seed=hd, num_pages=max(64, 1400 // page + 16))
    ops.rope_kv_write(qkv, H, Hkv, hd, None, ctx.positions, ctx.row_of_token, kc, vc, table, page)
    scale = 1.0 / math.sqrt(hd)
    whole = torch.full((sum(q_lens), H * hd), float("nan"), device=DEV)
    ops.paged_attention(qkv, whole, H, Hkv, hd, kc, vc, table, page, ctx, scale, window)
    assert torch.isfinite(whole).all()
    # 64-bit arithmetic over what the cache holds
    at = torch.tensor([sum(q_lens[:b + 1]) - 1 for b in range(len(ends))], device=DEV)      # the last token of each request
    G = H // Hkv
    ref = torch.empty(len(ends), H, hd, dtype=torch.float64, device=DEV)
    for b, n in enumerate(ends):
        pages = table[b, :(n + page - 1) // page].long()
        k = kc[pages].permute(1, 0, 2, 3).reshape(Hkv, -1, hd)[:, :n].double()
        v = vc[pages].permute(1, 0, 3, 2).reshape(Hkv, -1, hd)[:, :n].double()
        lo = max(0, n - window) if window else 0
        q = qkv[at[b], :H * hd].view(Hkv, G, 1, hd).double()
        p = torch.softmax((q * k[:, None, lo:]).sum(-1) * scale, -1)
        ref[b] = (p[..., None] * v[:, None, lo:]).sum(2).reshape(H, hd)
    # scores of a few units: a 32-bit sum of hd terms, exp, and a sum of up to 260 weights
    assert torch.allclose(whole[at].double(), ref.view(len(ends), -1), rtol=0, atol=4e-6)

    def single(rows, longest):
        toks = at[rows]
        c = SimpleNamespace(num_tokens=len(rows), num_rows=len(rows), positions=ctx.positions[toks].contiguous(),
                            row_of_token=torch.arange(len(rows), dtype=torch.int32, device=DEV), kv_lens=ctx.kv_lens[rows].contiguous(),
                            max_q_len=1, max_kv_len=longest, decode_only=True, workspace=ctx.workspace)
        o = torch.full((len(rows), H * hd), float("nan"), device=DEV)
        ops.paged_attention(qkv[toks].contiguous(), o, H, Hkv, hd, kc, vc, table[rows].contiguous(), page, c, scale, window)
        assert torch.equal(o, whole[toks])

    single(list(range(len(ends))), 260)                       # a block of keys a block (or all keys, from 512 pairs on)
    single(list(range(len(ends))) * 3, 1024)                  # as a captured step passes it: a longest length that none has
    single([0, 3, 6], 128)                                    # few keys
    single((list(range(len(ends))) * 50)[:512 // Hkv + 1], 260)
    single((list(range(len(ends))) * 50)[:512 // Hkv + 1], 2000)        # ranges of four blocks of keys, two to a row
    single(list(range(len(ends))), 60000 * 8 // Hkv)          # ranges of several blocks of keys, most of them behind the rows' ends


def test_attention_padding_rows_touch_nothing(ops):
    qkv, kc, vc, table, ctx, _, _ = _paged_setup(torch.float32, 2, 4, 2, 16, 16, [1, 1], [5, 9])
    kc0, vc0 = kc.clone(), vc.clone()
    ctx.row_of_token = torch.tensor([0, -1], dtype=torch.int32, device=DEV)
    ops.rope_kv_write(qkv, 4, 2, 16, None, ctx.positions, ctx.row_of_token, kc, vc, table, 16)
    blk = int(table[0, 0])
    nn = torch.nan_to_num
    assert not torch.equal(nn(kc[blk]), nn(kc0[blk]))
    kc0[blk], vc0[blk] = kc[blk], vc[blk]
    assert torch.equal(nn(kc), nn(kc0)) and torch.equal(nn(vc), nn(vc0))
    out = torch.full((2, 64), 3.0, device=DEV)
    ops.paged_attention(qkv, out, 4, 2, 16, kc, vc, table, 16, ctx, 0.25, 0)
    assert torch.all(out[1] == 0)


@pytest.mark.parametrize("R,V", [(1, 50), (3, 333), (5, 128256)])
def test_argmax_lowest_index_on_ties(ops, R, V):
    logits = rnd(R, V, seed=13)
    ref = logits.argmax(-1)
    out = torch.empty(R, dtype=torch.int32, device=DEV)
    ops.argmax(logits, out)
    assert torch.equal(out.long(), ref)
    logits[:, V // 2] = 100.0
    logits[:, V // 3] = 100.0
    ops.argmax(logits, out)
    assert torch.all(out == V // 3)


def _plain_sample(logits, temperature, top_k, top_p, min_p, u):
    order, w = plain_llama.filtered_distribution(logits, temperature, top_k, top_p, min_p)
    return plain_llama.sample_from(order, w, u), set(order.tolist())


@pytest.mark.parametrize("V", [7, 50, 1000, 32003, 140001])
def test_sample_matches_plain(ops, V):
    """Same token as the plain sorted walk for the same uniform number, under every filter.
    (32,003 tokens: four slices of the vocabulary, each with a list of its tokens ordered by bin;
    140,001: slices longer than such a list can be, the kernel reads the row instead.)"""
    rng = np.random.default_rng(V)
    cases = []
    for temperature in (0.7, 1.0, 1.5):
        for top_k, top_p, min_p in ((0, 1.0, 0.0), (5, 1.0, 0.0), (0, 0.9, 0.0), (0, 1.0, 0.05),
                                    (20, 0.8, 0.01), (1000000, 0.5, 0.0), (3, 0.3, 0.2)):
            for _ in range(6):
                cases.append((temperature, top_k, top_p, min_p, float(rng.random())))
    R = len(cases)
    logits = torch.tensor(rng.normal(0, 2.0, (R, V)), dtype=torch.float32)
    logits[::3, : min(V, 4)] = 3.0                   # ties among the largest
    dl = logits.to(DEV)
    f = lambda i, dt: torch.tensor([c[i] for c in cases], dtype=dt, device=DEV)
    out = torch.empty(R, dtype=torch.int32, device=DEV)
    ops.sample(dl, f(0, torch.float32), f(1, torch.int32).clamp(max=2**31 - 1), f(2, torch.float32),
               f(3, torch.float32), f(4, torch.float64), out)
    got = out.tolist()
    bad = 0
    for r, (temperature, top_k, top_p, min_p, u) in enumerate(cases):
        want, kept = _plain_sample(logits[r].numpy(), temperature, top_k, top_p, min_p, u)
        assert got[r] in kept, (r, cases[r], got[r])          # never outside the kept set
        bad += got[r] != want
    assert bad <= max(1, R // 100), f"{bad} of {R} draws differ from the plain walk"


def test_sample_rows_with_many_equal_or_far_logits(ops):
    """Rows the bins of the kernel do not separate: thousands of equal logits (more than it sorts
    in one go, so the descent over key digits answers) and a peaked row whose tokens nearly all
    lie far below the largest (weight 0 in fixed point)."""
    V = 9000
    rng = np.random.default_rng(5)
    flat = np.full(V, 1.0, dtype=np.float32)
    flat[[17, 4000, 8999]] = [2.5, 2.5, 0.5]
    peaked = np.full(V, -60.0, dtype=np.float32) + rng.normal(0, 3.0, V).astype(np.float32)
    peaked[[3, 77, 5000, 8000]] = [4.0, 3.5, 3.5, 1.0]
    cases = []
    for row in (flat, peaked):
        for top_k, top_p, min_p in ((0, 1.0, 0.0), (5000, 1.0, 0.0), (0, 0.7, 0.0), (6000, 0.9, 0.0), (0, 1.0, 0.3)):
            for u in (0.0, 0.013, 0.35, 0.5, 0.77, 0.999999):
                cases.append((row, 1.0, top_k, top_p, min_p, u))
    R = len(cases)
    dl = torch.tensor(np.stack([c[0] for c in cases]), device=DEV)
    f = lambda i, dt: torch.tensor([c[i] for c in cases], dtype=dt, device=DEV)
    out = torch.empty(R, dtype=torch.int32, device=DEV)
    ops.sample(dl, f(1, torch.float32), f(2, torch.int32), f(3, torch.float32), f(4, torch.float32),
               f(5, torch.float64), out)
    got = out.tolist()
    bad = 0
    for r, (row, temperature, top_k, top_p, min_p, u) in enumerate(cases):
        want, kept = _plain_sample(row, temperature, top_k, top_p, min_p, u)
        assert got[r] in kept, (r, cases[r][1:], got[r])
        bad += got[r] != want
    assert bad <= 1, f"{bad} of {R} draws differ from the plain walk"


def test_sample_reference_vectors(ops):
    """The reference's own sampler cases (crates/infer-worker/src/application/sampler_stack.rs:421-446):
    logits [3, 2, 1] with top_p 0.5 and draw 0.99 give token 0; top-k never leaves its set."""
    logits = torch.tensor([[3.0, 2.0, 1.0]], device=DEV)
    out = torch.empty(1, dtype=torch.int32, device=DEV)
    one = lambda v, dt: torch.tensor([v], dtype=dt, device=DEV)
    ops.sample(logits, one(1.0, torch.float32), one(0, torch.int32), one(0.5, torch.float32),
               one(0.0, torch.float32), one(0.99, torch.float64), out)
    assert out.item() == 0
    logits = torch.tensor([[0.1, 5.0, 4.9, -1.0, 4.8]], device=DEV)
    for u in np.linspace(0, 0.999999, 50):
        ops.sample(logits, one(1.0, torch.float32), one(2, torch.int32), one(1.0, torch.float32),
                   one(0.0, torch.float32), one(float(u), torch.float64), out)
        assert out.item() in (1, 2)


def test_sample_frequencies_and_greedy_rows(ops):
    """Over many draws the frequencies follow softmax(logits / T); temperature 0 rows are greedy."""
    V, R, T = 11, 20000, 0.8
    rng = np.random.default_rng(5)
    row = rng.normal(0, 1.5, V).astype(np.float32)
    logits = torch.tensor(row, device=DEV).repeat(R, 1)
    temp = torch.full((R,), T, device=DEV)
    temp[:10] = 0.0
    out = torch.empty(R, dtype=torch.int32, device=DEV)
    u = torch.tensor(rng.random(R), dtype=torch.float64, device=DEV)
    ops.sample(logits, temp, torch.zeros(R, dtype=torch.int32, device=DEV), torch.ones(R, device=DEV),
               torch.zeros(R, device=DEV), u, out)
    got = out.cpu().numpy()
    assert np.all(got[:10] == int(np.argmax(row)))
    p = plain_llama.softmax(row.astype(np.float64) / T)
    freq = np.bincount(got[10:], minlength=V) / (R - 10)
    assert np.max(np.abs(freq - p)) < 0.015


def test_sample_log_probabilities(ops):
    """ln p of the chosen token and of the five most probable kept tokens equal the plain
    computation, for greedy rows, plain temperature, and every filter; the tokens are the same
    with and without asking for them."""
    V, rng = 3001, np.random.default_rng(5)
    cases = [(0.0, 0, 1.0, 0.0), (1.0, 0, 1.0, 0.0), (0.7, 40, 1.0, 0.0), (1.3, 0, 0.8, 0.0),
             (0.9, 0, 1.0, 0.05), (0.5, 3, 0.9, 0.01), (1.0, 1, 1.0, 0.0), (2.0, 0, 0.3, 0.0)]
    R = len(cases)
    logits = torch.tensor(rng.normal(0, 3, (R, V)), dtype=torch.float32)
    logits[2, 5] = logits[2, 9] = logits[2].max() + 1                       # a tie at the top
    u = rng.random(R)
    dev = lambda a, dt: torch.tensor(a, dtype=dt, device=DEV)
    temp = dev([c[0] for c in cases], torch.float32)
    tk = dev([c[1] for c in cases], torch.int32)
    tp = dev([c[2] for c in cases], torch.float32)
    mp = dev([c[3] for c in cases], torch.float32)
    draws = dev(u, torch.float64)
    out0 = torch.empty(R, dtype=torch.int32, device=DEV)
    ops.sample(logits.to(DEV), temp, tk, tp, mp, draws, out0)
    out = torch.empty(R, dtype=torch.int32, device=DEV)
    lp = torch.empty(R, dtype=torch.float32, device=DEV)
    ids = torch.empty(R, 5, dtype=torch.int32, device=DEV)
    tlp = torch.empty(R, 5, dtype=torch.float32, device=DEV)
    want = dev([1] * (R - 1) + [0], torch.int32)
    ops.sample(logits.to(DEV), temp, tk, tp, mp, draws, out, lp, ids, tlp, want)
    assert torch.equal(out, out0)
    for r, (t, k, p, m) in enumerate(cases):
        greedy_row = t <= 0 or k == 1 or p <= 0
        tok, chosen, top = plain_llama.sample_with_logprobs(logits[r].numpy(), t if t > 0 else 1.0, k, p, m, u[r], greedy_row)
        assert out[r].item() == tok
        assert abs(lp[r].item() - chosen) < 1e-3, (r, lp[r].item(), chosen)
        got = [(i, x) for i, x in zip(ids[r].tolist(), tlp[r].tolist()) if i >= 0]
        if greedy_row or r == R - 1:                 # no list for greedy rows and for rows that did not ask
            assert got == []
        else:
            assert [i for i, _ in got] == [i for i, _ in top], (r, got, top)
            assert all(abs(a - b) < 1e-3 for (_, a), (_, b) in zip(got, top)), (r, got, top)


def _walk64(r, k, v, S, w, b, u):
    """S <- diag(w) S - b (u^T S) + k v^T, o = S^T r in 64 bits; r, k, w, b, u [T, H, dk], v [T, H, dv], S [H, dk, dv]"""
    out = []
    for t in range(r.shape[0]):
        S = w[t][:, :, None] * S - b[t][:, :, None] * (u[t][:, :, None] * S).sum(1, keepdim=True) + k[t][:, :, None] * v[t][:, None]
        out.append((r[t][:, :, None] * S).sum(1))
    return torch.stack(out), S


@pytest.mark.parametrize("form,d,keys", [("delta", 64, "random"), ("delta", 128, "random"), ("delta", 64, "repeated"), ("delta", 128, "repeated"), ("delta", 64, "fast decay"),
                                         ("delta", 64, "shared"), ("delta", 128, "shared"), ("decay", 64, "random"), ("decay", 128, "random"),
                                         ("decay", 64, "shared"), ("decay", 128, "shared"), ("rotated", 64, "random"), ("rotated", 128, "random")])
def test_state_walk_in_chunks(ops, monkeypatch, form, d, keys):
    """Rows of many tokens go through chunks of 32, the others through the walk; new and continued states, last chunks
    that are not whole, more chunks than a pass takes.  Both against 64 bits: neither the outputs nor the states of the chunks
    are further from it than the walk's, whatever the keys have in common."""
    H, q_lens, starts = 3, [32, 5, 33, 1, 300, 64], [0, 3, 40, 7, 31, 0]
    T, B = sum(q_lens), len(q_lens)
    bf = lambda *shape, seed, scale=1.0: rnd(*shape, dtype=torch.bfloat16, seed=seed, scale=scale)  # noqa: E731
    r, k, v = bf(T, H * d, seed=1), bf(T, H * d, seed=2), bf(T, H * d, seed=3)
    wl, al, w0, ab = bf(T, H * d, seed=4), bf(T, H * d, seed=5), rnd(H * d, seed=6), rnd(H * d, seed=7)
    if keys == "repeated":                        # one key all along, given up and written whole, hardly any decay: L is all ones
        k, w0, ab = k[:1].repeat(T, 1), torch.full_like(w0, -12.0), torch.full_like(ab, 12.0)
    elif keys == "shared":                        # keys around one direction, as a trained model's are, given up slowly
        r, k, w0, ab = r + k[:1] if form == "decay" else r, k[:1] + 0.3 * k, w0 - 3.0, ab + 2.0
    elif keys == "fast decay":                    # decays at their bound and next to one side by side
        w0 = torch.where(torch.arange(H * d, device=DEV) % 2 == 0, 12.0, -12.0)
    decay = torch.tensor([0.999, 0.7, 0.02], device=DEV)
    state0 = rnd(B + 1, H, d, d, seed=8)
    cu = torch.tensor([0] + list(np.cumsum(q_lens)), dtype=torch.int32, device=DEV)
    slots = torch.tensor([3, 0, 6, 1, 5, 2], dtype=torch.int32, device=DEV)
    ctx = SimpleNamespace(cu_q=cu, q_start=torch.tensor(starts, dtype=torch.int32, device=DEV), state_slots=slots, num_rows=B,
                          max_q_len=max(q_lens), max_kv_len=max(s + n for s, n in zip(starts, q_lens)), host_q_lens=q_lens,
                          workspace=Workspace(torch.device(DEV)))
    ang = np.arange(512)[:, None] * plain_llama.rope_frequencies(d, 10000.0, None)[None, :]
    rotary = tuple(torch.tensor(f(ang), dtype=torch.float32, device=DEV) for f in (np.cos, np.sin)) + (d,)
    kw = dict(wl=wl, al=al, w0=w0, ab=ab, unit_eps=1e-6, decay_c=math.exp(-0.5)) if form == "delta" else dict(decay=decay, silu_in=True) \
        if form == "decay" else dict(decay=decay, rotary=rotary, k_scale=0.3)
    heads = lambda t: t.double().view(-1, H, d)  # noqa: E731
    r64, k64, v64 = heads(r), heads(k), heads(v)
    if form == "delta":
        u64 = k64 / torch.sqrt(k64.square().sum(-1, keepdim=True) + 1e-6)
        w64, b64 = torch.exp(-math.exp(-0.5) * torch.sigmoid(heads(wl) + heads(w0))), torch.sigmoid(heads(al) + heads(ab)) * u64
    else:
        w64, u64 = decay.double()[None, :, None].expand(T, H, d), torch.zeros_like(k64)
        b64 = u64
        if form == "decay":
            r64, k64, v64 = (torch.nn.functional.silu(t) for t in (r64, k64, v64))
        else:
            pos = torch.cat([torch.arange(s, s + n, device=DEV) for s, n in zip(starts, q_lens)])
            c, sn = (t[pos].double()[:, None] for t in rotary[:2])
            turn = lambda t: torch.cat([t[..., :d // 2] * c - t[..., d // 2:] * sn, t[..., d // 2:] * c + t[..., :d // 2] * sn], -1)  # noqa: E731
            r64, k64 = turn(r64), 0.3 * turn(k64)
    errors = {}
    for chunks in (False, True):
        monkeypatch.setattr(ops, "_scan_in_chunks", lambda *a: chunks)
        state, out = state0.clone(), torch.full((T, H * d), float("nan"), device=DEV)
        ops.linear_scan(r, k, v, state, out, ctx, H, d, d, **kw)
        worst, lo = [0.0, 0.0], 0                                  # outputs and states, added over the rows of many tokens
        for b, n in enumerate(q_lens):
            S = state0[slots[b]].double() if starts[b] else torch.zeros(H, d, d, dtype=torch.float64, device=DEV)
            part = slice(lo, lo + n)
            o64, S64 = _walk64(r64[part], k64[part], v64[part], S, w64[part], b64[part], u64[part])
            for i, (got, want) in enumerate(((out[part].double().view(n, H, d), o64), (state[slots[b]].double(), S64))):
                error = ((got - want).norm() / want.norm()).item()
                assert error < 2e-6, (b, i, error)
                worst[i] += error if n >= 32 else 0.0
            lo += n
        assert torch.equal(state[4], state0[4])                    # no request's slot
        errors[chunks] = worst
    assert all(c <= 1.02 * w for c, w in zip(errors[True], errors[False])), errors       # (0.02: what rounds otherwise by chance)


def _scan_step(form, d, H, q_lens, starts, seed=20, unit_eps=1e-6):
    """(r, k, v, state, ctx, keywords) of ``linear_scan`` for a step of these rows."""
    T, B = sum(q_lens), len(q_lens)
    bf = lambda i: rnd(T, H * d, dtype=torch.bfloat16, seed=seed + i)  # noqa: E731
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)  # noqa: E731
    several = [b for b, n in enumerate(q_lens) if n > 1]
    ctx = SimpleNamespace(cu_q=i32([0] + list(np.cumsum(q_lens))), q_start=i32(starts), state_slots=i32(list(range(B))), num_rows=B,
                          max_q_len=max(q_lens), max_kv_len=max(s + n for s, n in zip(starts, q_lens)), host_q_lens=list(q_lens),
                          portion_rows=i32(several + [-1] * (B - len(several))), num_portion=len(several), workspace=Workspace(torch.device(DEV)))
    kw = dict(wl=bf(4), al=bf(5), w0=rnd(H * d, seed=seed + 6), ab=rnd(H * d, seed=seed + 7), unit_eps=unit_eps, decay_c=math.exp(-0.5)) \
        if form == "delta" else dict(decay=torch.linspace(0.9, 0.999, H, device=DEV), silu_in=True)
    return bf(1), bf(2), bf(3), rnd(B, H, d, d, seed=seed + 8), ctx, kw


def _scan_both_ways(ops, monkeypatch, H, d, r, k, v, state0, ctx, kw):
    """[(outputs, states)] of the walk and of the chunks."""
    got = []
    for chunks in (False, True):
        monkeypatch.setattr(ops, "_scan_in_chunks", lambda *a: chunks)
        state, out = state0.clone(), torch.full((r.shape[0], H * d), 7.0, device=DEV)
        ops.linear_scan(r, k, v, state, out, ctx, H, d, d, **kw)
        got.append((out, state))
    return got


@pytest.mark.parametrize("d", [64, 128])
def test_state_walk_in_chunks_of_keys_without_an_epsilon(ops, monkeypatch, d):
    """unit_eps = 0: the places past the end of a last chunk hold no key that could be divided by its length of zero."""
    r, k, v, state, ctx, kw = _scan_step("delta", d, 2, [33, 64, 95], [0, 5, 70], unit_eps=0.0)
    (out0, state0), (out1, state1) = _scan_both_ways(ops, monkeypatch, 2, d, r, k, v, state, ctx, kw)
    for a, b in ((out1, out0), (state1, state0)):
        assert a.isfinite().all() and (a - b).norm() <= 5e-7 * b.norm()


@pytest.mark.parametrize("n", [32, 64, 65, 96, 128, 150, 192, 1000])
def test_state_walk_in_chunks_of_a_single_row(ops, monkeypatch, n):
    """Heads of 128 with fixed decays: three chunks are under way for a single row, two beside another: the same bits, and the walk's to 32-bit rounding."""
    H, d = 2, 128
    r, k, v, state, ctx, kw = _scan_step("decay", d, H, [n], [40])
    (out0, state0), (out1, state1) = _scan_both_ways(ops, monkeypatch, H, d, r, k, v, state, ctx, kw)
    for a, b in ((out1, out0), (state1, state0)):
        assert a.isfinite().all() and (a - b).norm() <= 5e-7 * b.norm()
    _, _, _, _, ctx2, _ = _scan_step("decay", d, H, [n, 33], [40, 0])
    more = [torch.cat([t, t[:33] if n >= 33 else t.repeat(2, 1)[:33]]) for t in (r, k, v)]
    both, out2 = torch.cat([state, state]), torch.empty(n + 33, H * d, device=DEV)
    ops.linear_scan(*more, both, out2, ctx2, H, d, d, **kw)
    assert torch.equal(out2[:n], out1) and torch.equal(both[:1], state1)


@pytest.mark.parametrize("form,d,what,value,at", [
    ("delta", 64, "v", "inf", 705), ("delta", 64, "k", "nan", 40), ("delta", 128, "k", 1e37, 40), ("delta", 64, "r", "-inf", 50), ("delta", 64, "wl", "nan", 45),
    ("delta", 128, "al", "nan", 690), ("delta", 64, "v", "nan", 0), ("decay", 64, "v", "-inf", 44), ("decay", 64, "k", "inf", 700), ("decay", 128, "r", "nan", 63)])
def test_state_walk_in_chunks_of_tokens_that_are_not_finite(ops, monkeypatch, form, d, what, value, at):
    """One number of one token of the first of three rows (of 22 chunks a pass its first or second): the tokens before it, the
    other head and the other rows stay what they are, the rest is what the walk makes of it; a key so large that its
    quotient by a chunk's decays has no 32-bit value stays one that the walk can take."""
    H, q_lens = 2, [720, 33, 64]
    r, k, v, state, ctx, kw = _scan_step(form, d, H, q_lens, [0, 5, 70], seed=40)
    if value == 1e37:
        v = v * 1e-3
        kw["w0"] = torch.full_like(kw["w0"], 12.0)                 # decays at their bound: 1e37 / w^32 is beyond 32 bits
    {"r": r, "k": k, "v": v, "wl": kw.get("wl"), "al": kw.get("al")}[what][at, d + 3] = float(value)     # head 1
    (out0, state0), (out1, state1) = _scan_both_ways(ops, monkeypatch, H, d, r, k, v, state, ctx, kw)
    assert torch.equal(out0.isfinite(), out1.isfinite()) and torch.equal(state0.isfinite(), state1.isfinite())
    assert out0[:at].isfinite().all() and (value == 1e37 or not out0[at, d:].isfinite().all())
    lo = 0
    for b, n in enumerate(q_lens):
        for h in range(H):
            for x, y in ((out1[lo:lo + n, h * d:(h + 1) * d], out0[lo:lo + n, h * d:(h + 1) * d]), (state1[b, h], state0[b, h])):
                x, y = (torch.where(y.isfinite(), t, 0.0).double() for t in (x, y))
                assert (x - y).norm() <= 5e-7 * y.norm(), (b, h)
        lo += n


@pytest.mark.parametrize("form,d", [("delta", 64), ("decay", 64), ("delta", 128), ("decay", 128)])
def test_state_walk_in_chunks_beside_decoding_rows(ops, monkeypatch, form, d):
    """Two portions among more rows of single tokens than a pass has chunks: what the chunks need is the portions', not the
    rows', and the other rows' tokens and states are the walk's to the bit."""
    H, q_lens = 2, [1] * 33 + [130] + [1] * 20 + [2, 75] + [1] * 17
    starts = [(7 * i) % 50 for i in range(len(q_lens))]
    r, k, v, state, ctx, kw = _scan_step(form, d, H, q_lens, starts, seed=60)
    (out0, state0), (out1, state1) = _scan_both_ways(ops, monkeypatch, H, d, r, k, v, state, ctx, kw)
    unit = 32 * d + d * d + (d * d + d if form == "delta" else 0) + 4
    assert 0 < ctx.workspace.nbytes() <= 4 * (64 * H * unit + len(q_lens) * H * d // 16)
    lo = 0
    for b, n in enumerate(q_lens):
        for x, y in ((out1[lo:lo + n], out0[lo:lo + n]), (state1[b], state0[b])):
            assert torch.equal(x, y) if n < 32 else (x - y).norm() <= 5e-7 * y.norm(), b
        lo += n


@pytest.mark.parametrize("form", ["delta", "decay"])
def test_state_walk_takes_its_workspace_with_the_first_portion(ops, form):
    """A step whose portions the walk takes (so may the one that the cache pool's size is measured with) leaves nothing for later
    steps to allocate, whatever they hold."""
    H, d, ws = 2, 64, Workspace(torch.device(DEV))
    sizes = []
    for q_lens in ([40] * 24, [100], [3000], [400, 300], [1] * 24, [200] * 4 + [1] * 20):
        r, k, v, _, ctx, kw = _scan_step(form, d, H, q_lens, [0] * len(q_lens))
        ctx.workspace = ws
        ops.linear_scan(r, k, v, torch.zeros(25, H, d, d, device=DEV), torch.empty(r.shape[0], H * d, device=DEV), ctx, H, d, d, **kw)
        sizes.append(ws.nbytes())
    assert not ops._scan_in_chunks(form == "delta", d, 24, 40) and ops._scan_in_chunks(form == "delta", d, 1, 3000)
    assert sizes[0] > 0 and len(set(sizes)) == 1, sizes


@pytest.mark.parametrize("T,n,pad,shift", [(300, 2056, 8, 0), (257, 2048, 0, 8), (600, 1000, 4, 0), (256, 2048, 8, 3), (65, 8200, 8, 16), (4, 7, 1, 0), (3, 64, 0, 0)])
@pytest.mark.parametrize("name", ["relu2", "tanh"])
def test_unary_in_wide_and_single_elements(ops, name, T, n, pad, shift):
    """Rows that allow 16 bytes a thread and rows that do not (odd widths, strides and offsets): the same bits as the
    function in 32-bit, rounded once (the square of relu), and as a contiguous copy of the rows gives (both); in place
    too, infinities and what is no number included."""
    fn = [k for k in ops.UNARY if ("tanh" in k) == (name == "tanh")][0]
    wide = torch.randn(T, n + pad + shift, generator=torch.Generator().manual_seed(n)).to(torch.bfloat16).to(DEV)
    wide[0, shift:shift + 3] = torch.tensor([float("inf"), float("-inf"), float("nan")], device=DEV)
    x = wide[:, shift:shift + n]
    out = torch.empty_like(wide)[:, shift:shift + n]
    ops.unary(fn, x, out)
    single = torch.empty(T, n + 1, dtype=torch.bfloat16, device=DEV)[:, 1:]      # never 16-byte rows
    ops.unary(fn, x, single)
    assert torch.equal(out.contiguous().view(torch.int16), single.contiguous().view(torch.int16))
    if name != "tanh":
        z = x.float()
        assert torch.equal(out[:, 3:], (z.clamp(min=0) ** 2).to(torch.bfloat16)[:, 3:])
    ops.unary(fn, x, x)
    assert torch.equal(x.contiguous().view(torch.int16), single.contiguous().view(torch.int16))


@pytest.mark.parametrize("M,N,K", [(1, 128, 128), (8, 384, 256), (3, 2176, 128), (6, 3072, 2048), (5, 4224, 640), (7, 2048, 384), (2, 8192, 128)])
def test_a_norm_between_32bit_products_of_few_rows(ops, M, N, K):
    """The product before the norm and each kind of product behind it, against 64 bits: 8 and 16 columns a block, fewer and more partial
    sums of squares than lanes ask for at once, rows of the stream that are not finite with their own results only."""
    from rustinfer_amd.engine.context import Workspace
    ws = Workspace(torch.device(DEV))
    act, w, x0, wn = rnd(M, K, seed=M), rnd(N, K, seed=N) * 0.1, rnd(M, N, seed=3), 1 + 0.2 * rnd(N, seed=4)
    assert ops.linear_residual_ok(M, w, None, wn) and not ops.linear_residual_ok(9, w, None, wn)
    x = x0.clone()
    a, ssq = ops.linear_residual(act, w, None, x, wn, ws, "t")
    want = x0.double() + act.double() @ w.double().t()
    # the sum rounded to 32 bits, the addition, and one product with the norm's weight
    scale = x0.double().abs() + (act.double() @ w.double().t()).abs()
    assert torch.all((x.double() - want).abs() <= 2.0 ** -23 * scale)
    assert torch.all((a.double() - want * wn.double()).abs() <= 2.0 ** -22 * scale * wn.double().abs())
    squares = want.square().sum(1)
    assert torch.all((ssq.double().sum(1) - squares).abs() <= 2.0 ** -18 * squares)
    eps = 1e-5
    n = want * torch.rsqrt(squares[:, None] / N + eps) * wn.double()
    I = 72
    wo = rnd(2 * I, N, seed=5) * (4.0 / N) ** 0.5
    ref = n @ wo.double().t()
    # each row's operand is off by 2^-22 of the largest terms at most, in any direction
    slack = 2.0 ** -20 * ((scale * torch.rsqrt(squares[:, None] / N + eps) * wn.double().abs()) @ wo.double().abs().t()) + 2.0 ** -18 * ref.abs()
    out = torch.full((M, 2 * I + 3), float("nan"), device=DEV)
    ops.linear(a, wo, out[:, :2 * I], scale=(ssq, eps))
    assert torch.all((out[:, :2 * I].double() - ref).abs() <= slack) and out[:, 2 * I:].isnan().all()
    gated = torch.full((M, I + 1), float("nan"), device=DEV)
    ops.linear_swiglu(a, wo, gated[:, :I], None, scale=(ssq, eps))
    both = torch.nn.functional.silu(ref[:, :I]) * ref[:, I:]
    # silu moves by at most 1.1 times what its argument does, and is at most the argument
    assert torch.all((gated[:, :I].double() - both).abs() <= 1.1 * slack[:, :I] * ref[:, I:].abs() + slack[:, I:] * (ref[:, :I].abs() + slack[:, :I]) + 2.0 ** -20 * both.abs() + 1e-7)
    if M > 1:
        bad = x0.clone()
        bad[M - 1, N - 1] = float("nan")
        b, bq = ops.linear_residual(act, w, None, bad, wn, ws, "u")
        other = torch.empty(M, 2 * I, device=DEV)
        ops.linear(b, wo, other, scale=(bq, eps))
        assert torch.equal(other[:M - 1], out[:M - 1, :2 * I]) and other[M - 1].isnan().all()


@pytest.mark.parametrize("M,H,Hkv,hd,K", [(1, 1, 1, 16, 128), (8, 4, 2, 64, 256), (5, 6, 3, 48, 640), (7, 8, 2, 128, 2048)])
def test_qkv_f32_of_few_rows_with_rotation_and_pages(ops, M, H, Hkv, hd, K):
    """q in place, k and v in the pages, against the product and the kernel that rotates; a token of no request and one without a page leave nothing."""
    page, rows, blocks = 16, 3, 8
    x, w = rnd(M, K, seed=1), rnd((H + 2 * Hkv) * hd, K, seed=2) * 0.1
    ang = torch.arange(128, device=DEV)[:, None] * (10000.0 ** (-torch.arange(hd // 2, device=DEV) / (hd / 2)))
    rotary = (ang.cos().float().contiguous(), ang.sin().float().contiguous(), hd)
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)  # noqa: E731
    positions = i32([(19 * i + 5) % 100 for i in range(M)])
    row_of_token = i32([(i % rows) if i != 3 else -1 for i in range(M)])
    table = torch.randperm(24, device=DEV).to(torch.int32)[:rows * blocks].view(rows, blocks).contiguous()
    if M > 4:
        table[4 % rows, int(positions[4]) // page] = -1
    got, want = [[torch.full((M, (H + 2 * Hkv) * hd), 7.0, device=DEV), torch.full((24, Hkv, page, hd), 9.0, device=DEV), torch.full((24, Hkv, hd, page), 9.0, device=DEV)] for _ in range(2)]
    ssq = (x.double().square().view(M, 4, -1).sum(2)).float().contiguous()
    factor = torch.rsqrt(x.double().square().mean(1, keepdim=True) + 1e-5)
    for scale in (None, (ssq, 1e-5)):
        assert ops.qkv_rope_f32(x, w, got[0], H, Hkv, hd, rotary, positions, row_of_token, got[1], got[2], table, page, scale=scale)
        full = x.double() @ w.double().t()
        want[0].copy_(full if scale is None else full * factor)
        ops.rope_kv_write(want[0], H, Hkv, hd, rotary, positions, row_of_token, want[1], want[2], table, page)
        live = row_of_token >= 0
        # both round the same sums (the factor's own error aside) and turn them: three 32-bit operations on either side
        size = (x.double().abs() @ w.double().abs().t()).max() * (1 if scale is None else factor.max())
        for a, b in ((got[0][live, :H * hd], want[0][live, :H * hd]), (got[1], want[1]), (got[2], want[2])):
            assert (a - b).abs().max() <= 2.0 ** -20 * size
    assert not ops.qkv_rope_f32(rnd(9, K, seed=1), w, rnd(9, (H + 2 * Hkv) * hd, seed=1), H, Hkv, hd, rotary, positions, row_of_token, got[1], got[2], table, page)


@pytest.mark.parametrize("M,N,K,acts", [(1, 64, 32, [(0, 64, "relu2")]), (8, 2064, 2048, [(16, 2048, "relu2"), (0, 16, "tanh")]), (5, 12304, 512, [(0, 8192, "relu2")]), (3, 80, 32, [(8, 24, "tanh")])])
def test_activated_columns_behind_a_deferred_norm(ops, M, N, K, acts):
    """The norm's factor comes before the activation, in the epilogue and behind the product (columns that begin inside a tile)."""
    x = rnd(M, K, seed=M).to(torch.bfloat16)
    w = (rnd(N, K, seed=N) * 0.2).to(torch.bfloat16)
    ssq = (x.double().square().view(M, 4, -1).sum(2) * 3).float().contiguous()
    out = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    bufs = [torch.empty(M, n, dtype=torch.bfloat16, device=DEV) for _, n, _ in acts]
    ops.linear_activated(x, w, out, ops.tile_weight(w), [(c0, n, f, b) for (c0, n, f), b in zip(acts, bufs)], scale=(ssq, 1e-5))
    ref = (x.double() @ w.double().t()) * torch.rsqrt(ssq.double().sum(1, keepdim=True) / K + 1e-5)
    plain = torch.ones(N, dtype=torch.bool)
    for (c0, n, f), b in zip(acts, bufs):
        z = ref[:, c0:c0 + n]
        want = torch.relu(z).square() if f == "relu2" else torch.tanh(z)
        # bfloat16 rounds to 2^-8: the result, and behind the product the sum too, which the square doubles; 2^-6 covers the three
        assert torch.all((b.double() - want).abs() <= 2.0 ** -6 * want.abs() + 2.0 ** -8 * z.abs().clamp(max=1.0) * (f == "tanh") + 1e-4)
        plain[c0:c0 + n] = False
    assert torch.all((out[:, plain].double() - ref[:, plain]).abs() <= 2.0 ** -7 * ref[:, plain].abs() + 1e-4)
