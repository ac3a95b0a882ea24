"""The forward pass of short sequences in one launch, against the quadratic form in float64 and against the chunked launches (which run where
initial states go in: zeros here), at the edges of its row tiles, steps and operands."""

import ctypes

import pytest
import torch

from bi_mamba2_amd import _lib
from bi_mamba2_amd.ops import bimamba_chunk_scan_combined
from oracle import bimamba2_oracle as O

pytestmark = pytest.mark.gpu

# Relative 2-norm.  float32: sums of up to 256 products in any order, about sqrt(256) 2^-24 = 1e-6 at worst.  16 bits: the decayed products and the
# result are rounded once each, 2^-9 (2^-12) uniform: at most sqrt(2) 2^-9 = 2.8e-3 (3.5e-4).
BOUND = {torch.float32: 1e-6, torch.bfloat16: 2.8e-3, torch.float16: 3.5e-4}
# the chunked launches round C.B^T or the states to 16 bits besides
CHUNKED = {torch.float32: 2e-6, torch.bfloat16: 5e-3, torch.float16: 1e-3}


def one_launch(t, chunk):
    """what bimamba2_fwd does with these operands: 0 the chunked launches, 1 scan_once_kernel, 2 the walk"""
    p, (b, L, H, P), (G, N) = _lib.Params(), t["x"].shape, t["B"].shape[2:]
    p.batch, p.seqlen, p.nheads, p.headdim, p.ngroups, p.dstate, p.chunk_size = b, L, H, P, G, N, chunk
    p.dtype = {torch.float32: _lib.F32, torch.bfloat16: _lib.BF16, torch.float16: _lib.F16}[t["x"].dtype]
    for name, field, strides in (("x", "x", "x_sb x_sl x_sh"), ("B", "Bm", "B_sb B_sl B_sg"), ("C", "Cm", "C_sb C_sl C_sg"), ("z", "z", "z_sb z_sl z_sh")):
        if name in t:
            setattr(p, field, t[name].data_ptr())
            for s, v in zip(strides.split(), t[name].stride()):
                setattr(p, s, v)
    p.has_z = "z" in t
    return _lib.load().bimamba2_fwd_one_launch(ctypes.byref(p))


def call(t, chunk, initial=False, final=False):
    (b, _, H, P), N = t["x"].shape, t["B"].shape[-1]
    zeros = torch.zeros(b, H, P, N, device="cuda") if initial else None
    with torch.no_grad():
        return bimamba_chunk_scan_combined(t["x"], t["dt"], t["A"], t["B"], t["C"], chunk, D=t.get("D"), z=t.get("z"), dt_bias=t["dt_bias"],
                                           dt_softplus=True, initial_states_f=zeros, initial_states_b=zeros, return_final_states=final)


def check(t, dtype, chunk, D=True, z=True):
    t = dict(t)
    if not D:
        t.pop("D")
    if not z:
        t.pop("z")
    dev = {k: v.cuda() if not v.is_cuda else v for k, v in t.items()}
    r = {k: v.double().cpu() for k, v in t.items()}
    want, _ = O.bimamba2_quadratic(r["x"], r["dt"], r["A"], r["B"], r["C"], D=r.get("D"), z=r.get("z"), dt_bias=r["dt_bias"], dt_softplus=True)
    assert one_launch(dev, chunk)
    got, general = call(dev, chunk), call(dev, chunk, initial=True)
    assert bool(torch.isfinite(got).all())
    for a, b, bound in ((got.double().cpu(), want, BOUND[dtype]), (got.double(), general.double(), CHUNKED[dtype])):
        assert (a - b).norm() <= bound * b.norm(), ((a - b).norm() / b.norm()).item()


SHAPES = [  # heads, headdim, groups, dstate
    (torch.float32, 4, 32, 1, 16), (torch.float32, 2, 16, 2, 32), (torch.float32, 1, 64, 1, 64), (torch.float32, 2, 48, 1, 16),
    (torch.bfloat16, 4, 64, 1, 64), (torch.bfloat16, 2, 128, 2, 128), (torch.float16, 3, 64, 3, 32), (torch.float16, 2, 64, 1, 64)]


@pytest.mark.parametrize("L", [1, 15, 16, 17, 32, 33, 64, 65, 100, 127, 129, 197, 224, 255, 256])
@pytest.mark.parametrize("dtype,H,P,G,N", SHAPES)
def test_lengths(L, dtype, H, P, G, N):
    check(O.make_inputs(2, L, H, P, G, N, seed=L, dtype=dtype, with_z=True), dtype, 64 if dtype == torch.float32 else 256)


@pytest.mark.parametrize("dtype,H,P,G,N", SHAPES)
@pytest.mark.parametrize("D,z", [("none", True), ("hp", False), ("h", False), ("hp", True)])
def test_operands(dtype, H, P, G, N, D, z):
    t = O.make_inputs(1, 130, H, P, G, N, seed=3, dtype=dtype, with_z=True)
    if D == "hp":
        t["D"] = torch.randn(H, P, generator=torch.Generator().manual_seed(4))
    check(t, dtype, 128, D=D != "none", z=z)


@pytest.mark.parametrize("dt_dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("dtype,H,P,G,N", [SHAPES[0], SHAPES[4], SHAPES[7]])
def test_views_and_what_lies_behind_the_end(dt_dtype, dtype, H, P, G, N):
    """operands as slices of wider buffers, heads and positions at other strides, NaN in every element that is not theirs"""
    b, L = 3, 77
    t = O.make_inputs(b, L, H, P, G, N, seed=5, dtype=dtype, with_z=True)
    t["dt"] = t["dt"].to(dt_dtype)

    def inside(v, spare):
        wide = torch.full((b, L + 60) + v.shape[2:-1] + (v.shape[-1] + spare,), float("nan"), dtype=v.dtype, device="cuda")
        wide[:, :L, ..., :v.shape[-1]] = v.cuda()
        return wide[:, :L, ..., :v.shape[-1]]

    for k, spare in (("x", 16), ("z", 8), ("B", 8), ("C", 24), ("dt", 3)):
        t[k] = inside(t[k], spare)
    check(t, dtype, 64)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_strong_decay(dtype):
    """sums of up to -4000 over the sequence: neither side's factor may overflow, and neighbours keep their weight"""
    t = O.make_inputs(1, 256, 2, 64, 1, 64, seed=6, dtype=dtype, with_z=False)
    t["A"] = torch.tensor([-16.0, -1.0])
    t["dt_bias"] = torch.tensor([1.0, 1.0])
    check(t, dtype, 256, z=False)


@pytest.mark.parametrize("dtype,H,P,G,N", SHAPES)
def test_a_row_does_not_depend_on_the_batch(dtype, H, P, G, N):
    t = {k: v.cuda() for k, v in O.make_inputs(7, 200, H, P, G, N, seed=8, dtype=dtype, with_z=True).items()}
    row = {k: v[4:5] if k in ("x", "dt", "B", "C", "z") else v for k, v in t.items()}
    assert torch.equal(call(t, 256)[4:5], call(row, 256))


@pytest.mark.parametrize("L", [40, 256])
@pytest.mark.parametrize("dtype,H,P,G,N", SHAPES)
def test_final_states_besides(dtype, H, P, G, N, L):
    """the same result in bits, and the final states of the chunked launches"""
    t = {k: v.cuda() for k, v in O.make_inputs(2, L, H, P, G, N, seed=9, dtype=dtype, with_z=True).items()}
    out, *final = call(t, 64, final=True)
    assert torch.equal(out, call(t, 64))
    for a, b in zip(final, call(t, 64, initial=True, final=True)[1:]):
        assert torch.equal(a, b)


def test_final_states_take_no_launch_more_than_the_chunked_pass():
    """float32, chunks of 64: sums, states and their passing are two launches, as where the scan is the chunked one"""
    t = {k: v.cuda() for k, v in O.make_inputs(2, 256, 4, 32, 1, 16, seed=9, with_z=True).items()}
    call(t, 64, final=True)
    torch.cuda.synchronize()
    with torch.profiler.profile(activities=[torch.profiler.ProfilerActivity.CUDA, torch.profiler.ProfilerActivity.CPU]) as prof:
        call(t, 64, final=True)
        torch.cuda.synchronize()
    names = [e.name for e in prof.events() if e.device_type == torch.autograd.DeviceType.CUDA and "bm2::" in e.name]
    if not names:
        pytest.skip("no kernels in the profiler's record")
    assert len(names) == 3 and sum("scan_once" in n for n in names) == 1, names


# rows from which on the workgroups own whole sequences and walk through several heads (up to 64, 128, 256 positions)
ROWS = {64: 700, 128: 300, 256: 110}
WALK_SHAPES = [(torch.float32, 5, 32, 1, 16), (torch.float32, 4, 48, 2, 32), (torch.float32, 3, 64, 1, 64),
               (torch.bfloat16, 5, 64, 1, 64), (torch.bfloat16, 2, 128, 1, 128), (torch.float16, 6, 64, 2, 32), (torch.float16, 5, 64, 1, 64)]


def many(b, L, dtype, H, P, G, N, D, z):
    g = torch.Generator(device="cuda").manual_seed(L)
    r = lambda *s, t=dtype: torch.randn(*s, device="cuda", generator=g).to(t)
    t = dict(x=r(b, L, H, P), dt=0.5 * r(b, L, H, t=torch.float32), A=-1 - 15 * torch.rand(H, device="cuda", generator=g), B=r(b, L, G, N), C=r(b, L, G, N),
             dt_bias=r(H, t=torch.float32) - 3)
    if D != "none":
        t["D"] = r(*((H, P) if D == "hp" else (H,)), t=torch.float32)
    if z:
        t["z"] = r(b, L, H, P)
    return t


def rows_of(t, at):
    return {k: v[at] if k in ("x", "dt", "B", "C", "z") else v for k, v in t.items()}


@pytest.mark.parametrize("L", [1, 17, 64, 65, 100, 128, 129, 160, 192, 193, 197, 224, 225, 255, 256])
@pytest.mark.parametrize("dtype,H,P,G,N", WALK_SHAPES)
def test_many_rows_same_bits_as_one(L, dtype, H, P, G, N):
    """whole sequences a workgroup, several heads each: the bits that one row alone gives (over more than 128 positions by the other kernel)"""
    b = ROWS[64 if L <= 64 else 128 if L <= 128 else 256]
    t = many(b, L, dtype, H, P, G, N, *[("h", True), ("hp", False), ("none", True), ("hp", True), ("none", False)][(L + H) % 5])
    out = call(t, 64)
    assert bool(torch.isfinite(out).all())
    for k in (0, 1, b // 2, b - 1):
        row = rows_of(t, slice(k, k + 1))
        assert (one_launch(t, 64), one_launch(row, 64)) == (2, 2 if L <= 128 else 1)
        assert torch.equal(out[k:k + 1], call(row, 64))


def test_more_workgroups_than_one_launch_takes():
    """2.2 million sequences of one position: in pieces of the batch"""
    b = 2200000
    t = many(b, 1, torch.bfloat16, 4, 64, 1, 32, "h", False)
    out = call(t, 64)
    for at in (0, 2097152 - 500, b - 1000):
        assert torch.equal(out[at:at + 1000], call(rows_of(t, slice(at, at + 1000)), 64))
