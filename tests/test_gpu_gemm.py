"""The matrix product of the layer's projections against float32 products, at the edges of its tiles, k steps and k slices."""

import ctypes

import pytest
import torch

from bi_mamba2_amd import _lib

pytestmark = pytest.mark.gpu


def rows_of(rows, cols, pad, dtype, gen):
    """rows x cols in a wider buffer whose spare columns are NaN where the kernel must not care"""
    t = torch.full((rows, (cols + 7) // 8 * 8 + pad), float("nan"), device="cuda", dtype=dtype)
    t[:, :cols] = torch.randn(rows, cols, device="cuda", generator=gen).to(dtype)
    return t[:, :cols]


def plan(m, n, k, a_kc):
    """the tile (0: 256 x 256, 1: 256 x 192, 2: 128 x 128, 3: 64 x 64) and the slices of the sum"""
    p, slices = _lib.GemmParams(), ctypes.c_int()
    p.m, p.n, p.k, p.a_kcontig = m, n, k, a_kc
    return _lib.load().bimamba2_gemm_plan(ctypes.byref(p), ctypes.byref(slices)), slices.value


# one element; a whole 64 tile and one more than it; ragged k below, at and above one and four steps; many k slices with a
# ragged last one; 128 and 256 tiles with remainders; few columns (the rest of a library product)
@pytest.mark.parametrize("m,n,k", [(1, 1, 8), (64, 64, 32), (65, 70, 40), (197, 1688, 384), (300, 100, 33), (257, 259, 1000),
                                   (130, 6, 2047), (768, 300, 16381), (1000, 500, 96), (4099, 3224, 136)])
@pytest.mark.parametrize("a_kc,b_kc", [(1, 1), (1, 0), (0, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_product(m, n, k, a_kc, b_kc, dtype):
    if b_kc:
        k = (k + 7) // 8 * 8
    gen = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = rows_of(m, k, 8, dtype, gen) if a_kc else rows_of(k, m, 16, dtype, gen)
    b = rows_of(n, k, 0, dtype, gen) if b_kc else rows_of(k, n, 8, dtype, gen)
    bias = torch.randn(n, device="cuda", generator=gen).to(dtype) if m % 2 else None
    c = torch.full((m, n + 8 + (-n) % 8), 3.0, device="cuda", dtype=dtype)
    lib, p = _lib.load(), _lib.GemmParams()
    p.m, p.n, p.k, p.a_kcontig, p.b_kcontig = m, n, k, a_kc, b_kc
    p.dtype = {torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}[dtype]
    p.lda, p.ldb, p.ldc = a.stride(0), b.stride(0), c.stride(0)
    p.a, p.b, p.c = a.data_ptr(), b.data_ptr(), c.data_ptr()
    p.bias = bias.data_ptr() if bias is not None else None
    need = lib.bimamba2_gemm_workspace_bytes(ctypes.byref(p))
    ws = torch.empty(max(need, 1), dtype=torch.uint8, device="cuda")
    p.partial, p.partial_bytes, p.stream = ws.data_ptr(), need, torch.cuda.current_stream().cuda_stream
    assert lib.bimamba2_gemm(ctypes.byref(p)) == 0
    want = (a.float() if a_kc else a.float().t()) @ (b.float().t() if b_kc else b.float())
    if bias is not None:
        want = want + bias.float()
    got = c[:, :n].float()
    assert bool((c[:, n:] == 3.0).all())
    assert (got - want).norm() <= (4e-3 if dtype == torch.bfloat16 else 6e-4) * want.norm()
    assert (got - want).abs().max() <= (8e-3 if dtype == torch.bfloat16 else 1e-3) * want.abs().max()


# Shapes that take the 256 x 192 (first two lines) and 256 x 256 tiles uncut, with edges in both directions and sums that end in every place of the ring of five
# steps, a whole last step among them; sums cut in slices, the last one ragged
@pytest.mark.parametrize("m,n,k", [(11016, 649, 40), (13379, 514, 72), (13816, 543, 104), (13374, 522, 128), (7406, 1064, 168), (13854, 513, 200),
                                   (12357, 643, 232), (11150, 641, 264),
                                   (6402, 1775, 24), (5960, 1935, 72), (4621, 2537, 104), (6675, 1750, 136), (8281, 1347, 168), (5897, 1937, 192),
                                   (7246, 1555, 232), (4865, 2324, 264), (700, 1500, 16381), (1700, 2100, 9001), (3224, 768, 16373)])
@pytest.mark.parametrize("a_kc,b_kc", [(1, 1), (1, 0), (0, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_product_large_tiles(m, n, k, a_kc, b_kc, dtype):
    tile, slices = plan(m, n, (k + 7) // 8 * 8 if b_kc else k, a_kc)
    assert tile in (0, 1) if k > 9000 else tile == (n < 1100), tile
    assert (slices > 1) == (k > 9000)
    test_product(m, n, k, a_kc, b_kc, dtype)


# a last step of 256 x 256 tiles that is not whole: infinities behind its end
@pytest.mark.parametrize("a_kc,b_kc", [(1, 1), (1, 0), (0, 0)])
def test_large_tiles_infinities_behind_the_end(a_kc, b_kc):
    m, n, k = 4865, 2324, 200
    gen = torch.Generator(device="cuda").manual_seed(5)
    # the operand's last 8 (or the last rows) hold infinities where k ends; k = 200 of 224 elements
    a = torch.randint(-3, 4, (m, 224) if a_kc else (224, 4872), device="cuda", generator=gen).bfloat16()
    b = torch.randint(-3, 4, (n, 224) if b_kc else (224, 2328), device="cuda", generator=gen).bfloat16()
    for t, kc in ((a, a_kc), (b, b_kc)):
        (t[:, k:] if kc else t[k:]).fill_(float("inf"))
    c = torch.empty(m, 2328, device="cuda", dtype=torch.bfloat16)
    lib, p = _lib.load(), _lib.GemmParams()
    p.m, p.n, p.k, p.a_kcontig, p.b_kcontig, p.dtype = m, n, k, a_kc, b_kc, _lib.BF16
    p.lda, p.ldb, p.ldc = a.stride(0), b.stride(0), c.stride(0)
    p.a, p.b, p.c, p.stream = a.data_ptr(), b.data_ptr(), c.data_ptr(), torch.cuda.current_stream().cuda_stream
    assert plan(m, n, k, a_kc) == (0, 1)
    assert lib.bimamba2_gemm_workspace_bytes(ctypes.byref(p)) == 0 and lib.bimamba2_gemm(ctypes.byref(p)) == 0
    af, bf = (a[:, :k].float() if a_kc else a[:k, :m].float().t()), (b[:, :k].float().t() if b_kc else b[:k, :n].float())
    assert torch.equal(c[:, :n], (af @ bf).bfloat16())


@pytest.mark.parametrize("b_kc", [1, 0])
def test_infinities_in_the_last_step(b_kc):
    """what the loads find behind a k that is no multiple of a step takes no part, infinities included"""
    m, n, k = 70, 66, 40
    a = torch.ones(m, k, device="cuda", dtype=torch.bfloat16)
    b = torch.ones(n, k, device="cuda", dtype=torch.bfloat16)
    b[3, 36], b[5, k - 1] = float("inf"), float("-inf")
    rows = b if b_kc else torch.cat([b.t(), b.new_zeros(k, 6)], 1)
    c = torch.empty(m, 72, device="cuda", dtype=torch.bfloat16)
    lib, p = _lib.load(), _lib.GemmParams()
    p.m, p.n, p.k, p.a_kcontig, p.b_kcontig, p.dtype = m, n, k, 1, b_kc, _lib.BF16
    p.lda, p.ldb, p.ldc = k, rows.stride(0), 72
    p.a, p.b, p.c, p.stream = a.data_ptr(), rows.data_ptr(), c.data_ptr(), torch.cuda.current_stream().cuda_stream
    assert lib.bimamba2_gemm_workspace_bytes(ctypes.byref(p)) == 0 and lib.bimamba2_gemm(ctypes.byref(p)) == 0
    assert torch.equal(c[:, :n], (a.float() @ b.float().t()).bfloat16())


def test_rejects():
    lib, p = _lib.load(), _lib.GemmParams()
    x = torch.zeros(64, 64, device="cuda", dtype=torch.bfloat16)
    p.m = p.n = p.k = 64
    p.dtype, p.a_kcontig, p.b_kcontig = _lib.BF16, 1, 1
    p.lda = p.ldb = p.ldc = 64
    p.a = p.b = p.c = x.data_ptr()
    for field, value in (("dtype", _lib.F32), ("lda", 63), ("a", x.data_ptr() + 2), ("a_kcontig", 0), ("k", 60)):
        old = getattr(p, field)
        setattr(p, field, value)
        assert lib.bimamba2_gemm(ctypes.byref(p)) < 0
        setattr(p, field, old)
