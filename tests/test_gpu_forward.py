"""GPU parity of the forward path: every stage kernel and the whole operator against the float64 oracle,
through the C ABI (bi_mamba2_amd.ops calls libbimamba2_hip.so via ctypes)."""
import pytest
import torch

from oracle import bimamba2_oracle as O
from tests.helpers import assert_close, make_case, to64, to_dev

pytestmark = pytest.mark.gpu

INF = float("inf")

# batch, seqlen, H, P, G, N, chunk
STAGE_SHAPES = [
    (2, 200, 4, 32, 2, 16, 64),     # partial last chunk, grouped heads
    (1, 512, 2, 64, 1, 64, 256),    # the benchmark's tile sizes
    (2, 96, 4, 16, 4, 4, 32),       # small dims (padding inside the MFMA tiles)
    (1, 100, 2, 128, 1, 128, 48),   # two headdim / dstate tiles, chunk not a multiple of 64
]


@pytest.fixture(scope="module")
def ops():
    from bi_mamba2_amd import ops
    return ops


@pytest.mark.parametrize("shape", STAGE_SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_forward_stages(ops, shape, dtype):
    b, L, H, P, G, N, Q = shape
    inp = make_case(b, L, H, P, G, N, dtype, with_z=True, D_has_hdim=(P == 32))
    r = to64(inp)
    d = to_dev(inp)
    # stage 1: cumsum
    dt_ref, csf_ref, csb_ref = O.stage_chunk_cumsum(r["dt"], r["A"], Q, r["dt_bias"], True)
    csf, csb, dt_out = ops._chunk_cumsum_fwd(d["dt"], d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    assert_close(dt_out, dt_ref, torch.float32, "dt_out")
    assert_close(csf, csf_ref, torch.float32, "cs_f")
    assert_close(csb, csb_ref, torch.float32, "cs_b")
    # later stages take the device cumsums as input; the oracle takes the same values in float64
    csf64, csb64, dt64 = csf.double().cpu(), csb.double().cpu(), dt_out.double().cpu()
    # stage 2: CB
    CB = ops._bmm_chunk_fwd(d["C"], d["B"], Q)
    CB_ref = O.stage_bmm_chunk(r["C"], r["B"], Q)
    assert_close(CB, CB_ref, dtype, "CB")
    # stage 3: chunk states
    sf, sb = ops._chunk_state_fwd(d["B"], d["x"], dt_out, csf, csb)
    sf_ref, sb_ref = O.stage_chunk_state(r["B"], r["x"], dt64, csf64, csb64)
    assert_close(sf, sf_ref, dtype, "states_f")
    assert_close(sb, sb_ref, dtype, "states_b")
    # stage 4: inter-chunk scan (float32 arithmetic on float32 inputs)
    pf, pb, ff, fb = ops._state_passing_fwd(sf, sb, csf, csb)
    pf_ref, pb_ref, ff_ref, fb_ref = O.stage_state_passing(sf.double().cpu(), sb.double().cpu(), csf64, csb64)
    for got, ref, name in ((pf, pf_ref, "prev_f"), (pb, pb_ref, "prev_b"), (ff, ff_ref, "final_f"), (fb, fb_ref, "final_b")):
        assert_close(got, ref, torch.float32, name)
    # stage 5: chunk scan
    out, out_x = ops._chunk_scan_fwd(CB, d["x"], dt_out, csf, csb, d["C"], pf, pb, D=d["D"], z=d["z"])
    out_ref, outx_ref = O.stage_chunk_scan(CB.double().cpu(), r["x"], dt64, csf64, csb64, r["C"], pf.double().cpu(),
                                           pb.double().cpu(), r["D"], r["z"])
    big = N > 64      # dot products over 128 state columns of 16-bit operands: outputs of RMS ~ 10
    assert_close(out_x, outx_ref, dtype, "out_x", scaled=big)
    assert_close(out, out_ref, dtype, "out", scaled=big)


# the reference's own end-to-end forward grid (tests/test_fwd_scan.py:8-16 there): z = None, D = None
REF_FWD_GRID = [(b, L, 4, P, 4, N, 32) for b in (1, 2) for L in (32, 64, 128) for P in (4, 16) for N in (4, 16)]


@pytest.mark.parametrize("shape", REF_FWD_GRID)
def test_forward_reference_grid(ops, shape):
    b, L, H, P, G, N, Q = shape
    inp = make_case(b, L, H, P, G, N, torch.float32, with_D=False, ref_style=True)
    r, d = to64(inp), to_dev(inp)
    out = ops.bimamba_chunk_scan_combined(d["x"], d["dt"], d["A"], d["B"], d["C"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    ref = O.bimamba2_quadratic(r["x"], r["dt"], r["A"], r["B"], r["C"], dt_bias=r["dt_bias"], dt_softplus=True)[0]
    assert_close(out, ref, torch.float32, "out")


E2E = [
    # batch, seqlen, H, P, G, N, chunk, dtype, z, D ('none'|'h'|'hp'), bias, softplus, limit
    (2, 256, 4, 32, 1, 16, 64, torch.float32, False, "h", True, True, (0.0, INF)),       # the reference’s own CPU-runnable benchmark shape
    (2, 250, 4, 32, 2, 16, 64, torch.float32, True, "hp", True, True, (0.0, INF)),
    (1, 130, 2, 64, 1, 64, 128, torch.float32, True, "h", False, False, (0.0, INF)),
    (2, 200, 4, 16, 4, 8, 32, torch.float32, False, "none", True, True, (0.01, 0.2)),
    (2, 512, 8, 64, 1, 64, 256, torch.bfloat16, True, "h", True, True, (0.0, INF)),
    (1, 700, 4, 64, 2, 128, 256, torch.bfloat16, False, "h", True, True, (0.0, INF)),
    (1, 300, 2, 128, 1, 32, 64, torch.bfloat16, True, "hp", True, True, (0.0, INF)),
    (2, 256, 4, 64, 4, 64, 128, torch.float16, True, "h", True, True, (0.0, INF)),
]


@pytest.mark.parametrize("case", E2E)
def test_forward_end_to_end(ops, case):
    b, L, H, P, G, N, Q, dtype, z, Dk, bias, sp, lim = case
    inp = make_case(b, L, H, P, G, N, dtype, with_z=z, with_D=(Dk != "none"), D_has_hdim=(Dk == "hp"), with_bias=bias)
    r, d = to64(inp), to_dev(inp)
    out, ff, fb = ops.bimamba_chunk_scan_combined(d["x"], d["dt"], d["A"], d["B"], d["C"], Q, D=d["D"], z=d["z"],
                                                  dt_bias=d["dt_bias"], dt_softplus=sp, dt_limit=lim,
                                                  return_final_states=True)
    ref = O.bimamba2_sequential(r["x"], r["dt"], r["A"], r["B"], r["C"], D=r["D"], z=r["z"], dt_bias=r["dt_bias"],
                                dt_softplus=sp, dt_limit=lim)
    assert out.dtype == dtype and ff.dtype == torch.float32
    assert_close(out, ref[0], dtype, "out", scaled=not sp)      # raw dt without softplus: outputs far from unit scale
    assert_close(ff, ref[2], dtype, "final_f")
    assert_close(fb, ref[3], dtype, "final_b")


def test_forward_strided_inputs(ops):
    """x, B, C carved out of one projection output (as the BiMamba2 layer does): strided views, no copies."""
    b, L, H, P, G, N, Q = 2, 192, 4, 32, 1, 16, 64
    inp = make_case(b, L, H, P, G, N, torch.float32)
    r, d = to64(inp), to_dev(inp)
    packed = torch.cat([d["x"].flatten(2), d["B"].flatten(2), d["C"].flatten(2)], -1)
    x, B, C = torch.split(packed, [H * P, G * N, G * N], -1)
    out = ops.bimamba_chunk_scan_combined(x.unflatten(-1, (H, P)), d["dt"], d["A"], B.unflatten(-1, (G, N)),
                                          C.unflatten(-1, (G, N)), Q, D=d["D"], dt_bias=d["dt_bias"], dt_softplus=True)
    ref = O.bimamba2_quadratic(r["x"], r["dt"], r["A"], r["B"], r["C"], D=r["D"], dt_bias=r["dt_bias"], dt_softplus=True)[0]
    assert_close(out, ref, torch.float32, "out")


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_stages_rebuild_cb_when_it_is_not_given(ops, dtype):
    """The scan, dx and dCB stages called without CB (the way the composites call them at such shapes) agree with the
    same stages reading the CB of the bmm stage.  Ragged last chunk (44 rows), two head groups."""
    b, L, H, P, G, N, Q = 2, 300, 4, 64, 2, 64, 256
    inp = make_case(b, L, H, P, G, N, dtype, with_z=True)
    d = to_dev(inp)
    csf, csb, dt_out = ops._chunk_cumsum_fwd(d["dt"], d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    CB = ops._bmm_chunk_fwd(d["C"], d["B"], Q)
    sf, sb = ops._chunk_state_fwd(d["B"], d["x"], dt_out, csf, csb)
    pf, pb, _, _ = ops._state_passing_fwd(sf, sb, csf, csb)
    out1, outx1 = ops._chunk_scan_fwd(CB, d["x"], dt_out, csf, csb, d["C"], pf, pb, D=d["D"], z=d["z"])
    out2, outx2 = ops._chunk_scan_fwd(None, d["x"], dt_out, csf, csb, d["C"], pf, pb, D=d["D"], z=d["z"], B=d["B"])
    assert_close(outx2, outx1.double().cpu(), dtype, "out_x without CB")
    assert_close(out2, out1.double().cpu(), dtype, "out without CB")
    g = torch.Generator().manual_seed(11)
    dout = torch.randn(d["x"].shape, generator=g).to(dtype).cuda()
    dsf = torch.randn(pf.shape, generator=g).cuda() * 0.1
    dsb = torch.randn(pf.shape, generator=g).cuda() * 0.1
    dx1, ddt1, dD1 = ops._chunk_scan_chunk_state_bwd_dx(d["x"], dt_out, csf, csb, d["B"], CB, dout, dsf, dsb, D=d["D"])
    dx2, ddt2, dD2 = ops._chunk_scan_chunk_state_bwd_dx(d["x"], dt_out, csf, csb, d["B"], None, dout, dsf, dsb, D=d["D"], C=d["C"])
    assert_close(dx2, dx1.double().cpu(), dtype, "dx without CB")
    # positions past the end of the sequence are not written by either path
    valid = (torch.arange(ddt1.shape[2])[:, None] * Q + torch.arange(Q)[None, :] < L).to(ddt1.device)
    assert_close(torch.where(valid, ddt2, 0.0), torch.where(valid, ddt1, 0.0).double().cpu(), dtype, "ddt_direct without CB", scaled=True)
    assert_close(dD2, dD1.double().cpu(), dtype, "dD without CB", scaled=True)
    dCB1, da1 = ops._chunk_scan_bwd_dcb(d["x"], dt_out, csf, csb, dout, CB, ngroups=G)
    dCB2, da2 = ops._chunk_scan_bwd_dcb(d["x"], dt_out, csf, csb, dout, None, ngroups=G, B=d["B"], C=d["C"])
    assert_close(dCB2, dCB1.double().cpu(), dtype, "dCB without CB", scaled=True)
    assert_close(da2, da1.double().cpu(), dtype, "da_intra without CB", scaled=True)
    # shapes whose kernels cannot rebuild CB refuse a missing CB instead of reading a null pointer
    with pytest.raises(ValueError):
        ops._chunk_scan_fwd(None, d["x"].float(), dt_out, csf, csb, d["C"].float(), pf, pb, B=d["B"].float())


@pytest.mark.parametrize("b,L,H,P,G,N,Q,dtype,dt_dtype", [
    (2, 130, 3, 16, 3, 16, 64, torch.float32, torch.float32),        # several tiles of C.B^T, one of states
    (1, 257, 2, 72, 1, 80, 256, torch.float32, torch.float16),       # four tiles of states: the first one's workgroup writes the sums
    (1, 64, 2, 64, 1, 64, 64, torch.float32, torch.bfloat16),
    (2, 75, 4, 24, 2, 24, 50, torch.bfloat16, torch.bfloat16),       # chunk no multiple of 4 positions a lane
    (1, 300, 2, 8, 1, 136, 100, torch.float16, torch.float32),
])
def test_first_kernels_in_one_launch(b, L, H, P, G, N, Q, dtype, dt_dtype):
    """bimamba2_fwd's launch of cumulative sums, chunk states and C.B^T against the stages one by one"""
    from bi_mamba2_amd import ops
    d = to_dev(make_case(b, L, H, P, G, N, dtype))
    dt = d["dt"].to(dt_dtype)
    res = ops._mamba_chunk_scan_combined_fwd(d["x"], dt, d["A"], d["B"], d["C"], Q, D=d["D"], dt_bias=d["dt_bias"], dt_softplus=True)
    csf, csb, dt_out = ops._chunk_cumsum_fwd(dt, d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    for got, want in zip(res[2:5], (dt_out, csf, csb)):
        if dtype == torch.float32:
            assert torch.equal(got, want)
        else:                                # (that stage alone always sums in 64 bits: up to 256 additions rounded to 24 bits here)
            torch.testing.assert_close(got, want, rtol=256 * 2.0 ** -24, atol=0)
    dt_out, csf, csb = res[2:5]
    sf, sb = ops._chunk_state_fwd(d["B"], d["x"], dt_out, csf, csb)
    sf, sb = ops._state_passing_fwd(sf, sb, csf, csb)[:2]
    CB = ops._bmm_chunk_fwd(d["C"], d["B"], Q)
    out = ops._chunk_scan_fwd(CB, d["x"], dt_out, csf, csb, d["C"], sf, sb, D=d["D"])[0]
    # the weights of the states come from the sums in registers instead of memory: the same values, the same order of products
    for got, want in zip((res[5], res[6], res[0]), (sf, sb, out)):
        assert torch.equal(got, want)


@pytest.mark.parametrize("case", [
    (1, 257, 4, 64, 2, 128, 256, torch.bfloat16, torch.float32),     # two tiles of states, sixteen of C.B^T, one of them past the end
    (2, 33, 9, 128, 1, 128, 32, torch.float16, torch.float16),       # more than eight heads a group: the other order of tiles
    (1, 200, 2, 64, 1, 192, 96, torch.bfloat16, torch.bfloat16),     # a chunk that is no whole tile of C.B^T
])
def test_first_kernels_of_wide_heads_in_one_launch(case):
    """the same for the states by direct loads"""
    test_first_kernels_in_one_launch(*case)


@pytest.mark.parametrize("P,N", [(8, 8), (16, 72), (24, 16), (64, 40), (72, 64), (128, 136)])
@pytest.mark.parametrize("L,Q,dtype", [(1, 32, torch.bfloat16), (95, 64, torch.float16), (129, 128, torch.bfloat16), (100, 50, torch.bfloat16)])
def test_chunk_states_of_narrow_tiles(P, N, L, Q, dtype):
    """the kernel with direct loads of whole tiles (16 bits, up to 128 positions, sizes that are multiples of 8) for states and for
    their gradients, rows and columns that are no whole tile included, against float64"""
    from bi_mamba2_amd import ops
    b, H, G = 2, 4, 2
    d = to_dev(make_case(b, L, H, P, G, N, dtype))
    csf, csb, dt = ops._chunk_cumsum_fwd(d["dt"], d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    nc = csf.shape[2]
    pad = lambda t: torch.nn.functional.pad(t.double(), (0, 0, 0, 0, 0, nc * Q - L)).view(b, nc, Q, *t.shape[2:])
    rows = lambda e: e.double().permute(0, 2, 3, 1)                                        # (b, nc, Q, H)
    ends = dict(x=(csf[..., -1:] - csf, csb[..., :1] - csb, dt), d=(csf, csb, torch.ones_like(dt)))      # exponents of the weights and their factor
    for got, mate, (ef, eb, d0) in ((ops._chunk_state_fwd(d["B"], d["x"], dt, csf, csb), d["B"], ends["x"]), (ops._chunk_scan_bwd_dstates(d["C"], csf, csb, d["x"]), d["C"], ends["d"])):
        for g, e in zip(got, (ef, eb)):
            xs, ms = pad(d["x"]) * rows(d0.double() * e.double().exp())[..., None], pad(mate).repeat_interleave(H // G, 3)
            want = torch.einsum("bcqhp,bcqhn->bchpn", xs, ms)
            # One operand carries the weight and enters as two numbers of the inputs' type: each rounds by at most half a unit in its
            # last place, 2^-8 (8 bits of significand) or 2^-11 (11 bits), the second of what the first left: 2^-16 or 2^-22 of
            # each product, or 2^-25, half of float16's smallest number, where that is subnormal.  The weight is off by the
            # rounding of its exponent's multiple (2^-23 of it) and a few roundings of its own, 256 sums in float32 by 2^-16.
            u, tiny = {torch.bfloat16: (2.0 ** -16, 0.0), torch.float16: (2.0 ** -22, 2.0 ** -25)}[dtype]
            off = u + 2.0 ** -16 + (rows(e).abs()[..., None] + 4) * 2.0 ** -23
            bound = torch.einsum("bcqhp,bcqhn->bchpn", xs.abs() * off, ms.abs()) + tiny * ms.abs().sum(2)[..., None, :] + 1e-30
            assert float(((g - want).abs() / bound).max()) <= 1.0


@pytest.mark.parametrize("L,Q,N,dtype,one_row", [(300, 256, 64, torch.bfloat16, False), (100, 64, 64, torch.float16, False),
                                                 (257, 128, 128, torch.bfloat16, True)])
def test_sums_beside_the_chunk_states_take_the_products_unrounded(ops, L, Q, N, dtype, one_row):
    """Pairs of dt that cancel: 1 and -(1 - k / 65536).  1 * A is exact, so a sum that takes the second product unrounded is off by
    its additions alone, at the size of the small sums; a rounded product is off by 2^-25 |A|.  one_row: seq_idx without a boundary."""
    H, nc = 4, -(-L // Q)
    d = to_dev(make_case(2, L, H, 64, 2, N, dtype))
    k = torch.randint(1, 9, (2, nc * Q // 4, H), generator=torch.Generator().manual_seed(4)).float()
    dt = torch.zeros(2, nc * Q // 4, 4, H)
    dt[:, :, 0, 0::2], dt[:, :, 1, 0::2] = 1.0, k[..., 0::2] / 65536 - 1.0        # even heads: the exact product comes first
    dt[:, :, 2, 1::2], dt[:, :, 3, 1::2] = k[..., 1::2] / 65536 - 1.0, 1.0        # odd heads: ... first in the reverse sums
    dt = dt.flatten(1, 2)[:, :L // 4 * 4]
    dt = torch.nn.functional.pad(dt, (0, 0, 0, L - dt.shape[1])).cuda()
    A = -torch.rand(H, generator=torch.Generator().manual_seed(5)).cuda() - 1.0
    si = torch.zeros(2, L, dtype=torch.int32, device="cuda") if one_row else None
    res = ops._mamba_chunk_scan_combined_fwd(d["x"], dt, A, d["B"], d["C"], Q, dt_limit=(-INF, INF), seq_idx=si)
    a = torch.nn.functional.pad(dt, (0, 0, 0, nc * Q - L)).double().view(2, nc, Q, H).permute(0, 3, 1, 2) * A.double()[:, None, None]
    for got, want, heads, big in ((res[3], a.cumsum(-1), slice(0, None, 2), 0), (res[4], a.flip(-1).cumsum(-1).flip(-1), slice(1, None, 2), 3)):
        got, want = (t[:, heads].unflatten(-1, (Q // 4, 4)) for t in (got.double(), want))
        small = [e for e in range(4) if e != big]                                # (the sum behind the first of a pair is about A)
        # (four positions of a lane, six steps over the wave, what is in front of the lane by a difference, and their sum)
        err, bound = float((got - want)[..., small].abs().max()), 12 * 2.0 ** -24 * float(want[..., small].abs().max())
        assert err <= bound
