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
