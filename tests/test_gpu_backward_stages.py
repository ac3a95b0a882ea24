"""GPU parity of every backward stage on its own (the reference tests its backward kernels one by one as well:
tests/test_bwd_chunk_scan.py, tests/test_bwd_chunk_state.py, tests/test_bwd_state_passing.py there), through the stage
wrappers of bi_mamba2_amd.ops and the C ABI.

The expected value of a backward stage is torch.autograd through the oracle's restatement of the matching FORWARD stage
(oracle.bimamba2_oracle.stage_*, pinned on the CPU by "the stages composed equal the closed form"), in float64, fed with
the device's own inputs to that stage - so an error is attributed to the stage that made it, and no backward formula is
written down a second time."""
import pytest
import torch
import torch.nn.functional as F

from oracle import bimamba2_oracle as O
from tests.helpers import assert_close, make_case, to64, to_dev

pytestmark = pytest.mark.gpu

# batch, seqlen, H, P, G, N, chunk
SHAPES = [
    (2, 200, 4, 32, 2, 16, 64),     # partial last chunk, grouped heads
    (1, 512, 2, 64, 1, 64, 256),    # the benchmark's tile sizes
    (2, 96, 4, 16, 4, 4, 32),       # small dims (padding inside the MFMA tiles)
    (1, 100, 2, 128, 1, 128, 48),   # two headdim / dstate tiles, chunk not a multiple of 64
    (1, 300, 32, 64, 1, 64, 256),   # 32 heads in one group: four head slices of partial dB / dC sums
    (1, 128, 32, 16, 2, 16, 64),    # 16 heads per group: two slices
]


@pytest.fixture(scope="module")
def ops():
    from bi_mamba2_amd import ops
    return ops


def _leaf(t):
    return t.detach().double().cpu().requires_grad_(True)


def _c(t):
    return t.detach().double().cpu()


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_backward_stages(ops, shape, dtype):
    b, L, H, P, G, N, Q = shape
    inp = make_case(b, L, H, P, G, N, dtype, with_z=True, D_has_hdim=(P == 32))
    r, d = to64(inp), to_dev(inp)
    big = dtype != torch.float32      # 16-bit: summed gradients in units of their RMS (see tests/helpers.py)
    dout = torch.randn(inp["x"].shape, generator=torch.Generator().manual_seed(9)).to(dtype)
    nc = (L + Q - 1) // Q
    valid = (torch.arange(nc)[:, None] * Q + torch.arange(Q)[None, :] < L)      # (nc, Q): positions inside the sequence

    # ---- forward intermediates on the device (each checked on its own in test_gpu_forward.py)
    csf, csb, dt_out = ops._chunk_cumsum_fwd(d["dt"], d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    CB = ops._bmm_chunk_fwd(d["C"], d["B"], Q)
    sf, sb = ops._chunk_state_fwd(d["B"], d["x"], dt_out, csf, csb)
    pf, pb, _, _ = ops._state_passing_fwd(sf, sb, csf, csb)
    out, out_x = ops._chunk_scan_fwd(CB, d["x"], dt_out, csf, csb, d["C"], pf, pb, D=d["D"], z=d["z"])
    csf64, csb64, dt64, CB64 = _c(csf), _c(csb), _c(dt_out), _c(CB)

    # ---- dz, dout * silu(z)   (a8)
    dz, dout_x = ops._chunk_scan_bwd_dz(d["x"], d["z"], out_x, dout.cuda(), Q)
    z64 = _leaf(inp["z"])
    (_c(out_x) * F.silu(z64)).backward(dout.double())
    assert_close(dz, z64.grad, dtype, "dz")
    assert_close(dout_x, dout.double() * F.silu(r["z"]), dtype, "dout_x")
    dy64 = _c(dout_x)

    def scan(CBv, x, dtv, cf, cb_, C, prf, prb, D):
        return O.stage_chunk_scan(CBv, x, dtv, cf, cb_, C, prf, prb, D, None)[0]

    # ---- gradient with respect to the states entering the chunks   (a9)
    dpf, dpb = ops._chunk_scan_bwd_dstates(d["C"], csf, csb, dout_x)
    prf, prb = _leaf(pf), _leaf(pb)
    scan(CB64, r["x"], dt64, csf64, csb64, r["C"], prf, prb, r["D"]).backward(dy64)
    assert_close(dpf, prf.grad, dtype, "dprev_f", scaled=big)
    assert_close(dpb, prb.grad, dtype, "dprev_b", scaled=big)

    # ---- the two stages above as one launch, where that kernel exists: the same bits
    if dtype != torch.float32 and N == 64 and P % 64 == 0 and Q % 32 == 0:
        dz1, dox1, dpf1, dpb1 = ops._chunk_scan_bwd_dz_dstates(d["z"], out_x, dout.cuda(), d["C"], csf, csb)
        assert torch.equal(dz1, dz) and torch.equal(dox1, dout_x), "dz / dout_x of the merged launch"
        assert torch.equal(dpf1, dpf) and torch.equal(dpb1, dpb), "dstates of the merged launch"

    # ---- adjoint of the two inter-chunk recurrences + gradient of the chunk totals   (a10)
    dSf, dSb, ddAcf, ddAcb = ops._state_passing_bwd(pf, pb, csf, csb, dpf, dpb)
    Sf, Sb, cf, cb_ = _leaf(sf), _leaf(sb), _leaf(csf), _leaf(csb)
    opf, opb, _, _ = O.stage_state_passing(Sf, Sb, cf, cb_)
    torch.autograd.backward([opf, opb], [_c(dpf), _c(dpb)])
    assert_close(dSf, Sf.grad, torch.float32, "dstates_f")          # float32 arithmetic on float32 inputs
    assert_close(dSb, Sb.grad, torch.float32, "dstates_b")
    assert_close(ddAcf, cf.grad[..., -1], torch.float32, "ddA_chunk_f", scaled=True)
    assert_close(ddAcb, cb_.grad[..., 0], torch.float32, "ddA_chunk_b", scaled=True)

    # ---- dx, ddt_direct, dD   (a11): the scan's x path and the chunk states' x path
    dx, ddt_direct, dD = ops._chunk_scan_chunk_state_bwd_dx(d["x"], dt_out, csf, csb, d["B"], CB, dout_x, dSf, dSb, D=d["D"])
    x64, dtl, D64 = _leaf(inp["x"]), _leaf(dt_out), _leaf(inp["D"])
    y = scan(CB64, x64, dtl, csf64, csb64, r["C"], _c(pf), _c(pb), D64)
    S2f, S2b = O.stage_chunk_state(r["B"], x64, dtl, csf64, csb64)
    torch.autograd.backward([y, S2f, S2b], [dy64, _c(dSf), _c(dSb)])
    assert_close(dx, x64.grad, dtype, "dx")
    m = valid.to(ddt_direct.device)
    # sums over headdim of products of size 100 and more (RMS 176, maximum 1546 at the 32-head shape): in units of the RMS
    assert_close(torch.where(m, ddt_direct, 0.0), dtl.grad, dtype, "ddt_direct", scaled=True)
    assert_close(dD, D64.grad, dtype, "dD", scaled=big)

    # ---- dB through the chunk states + its decay terms   (a12)
    dBs, vf, vb = ops._chunk_state_bwd_db(d["x"], dt_out, csf, csb, dSf, dSb, B=d["B"], ngroups=G)
    assert dBs.shape[0] == (H // G + 7) // 8
    B64, cf, cb_ = _leaf(inp["B"]), _leaf(csf), _leaf(csb)
    S3f, S3b = O.stage_chunk_state(B64, r["x"], dt64, cf, cb_)
    torch.autograd.backward([S3f, S3b], [_c(dSf), _c(dSb)])
    assert_close(dBs.sum(0), B64.grad, dtype, "dB (state part)", scaled=big)
    # S_f = sum_k e^{cs_f[Q-1] - cs_f[k]} (...): v_f[k] = -dL/dcs_f[k] for k < Q-1; S_b likewise with cs_b[0], k > 0
    assert_close(torch.where(m, vf, 0.0)[..., :-1], -cf.grad[..., :-1], dtype, "v_f", scaled=big)
    assert_close(torch.where(m, vb, 0.0)[..., 1:], -cb_.grad[..., 1:], dtype, "v_b", scaled=big)

    # ---- dC through the entering states + its decay terms   (a13): the scan without its within-chunk part
    dCs, uf, ub = ops._chunk_scan_bwd_dC(pf, pb, csf, csb, dout_x, C=d["C"], ngroups=G)
    C64, cf, cb_ = _leaf(inp["C"]), _leaf(csf), _leaf(csb)
    scan(torch.zeros_like(CB64), r["x"], dt64, cf, cb_, C64, _c(pf), _c(pb), None).backward(dy64)
    assert_close(dCs.sum(0), C64.grad, dtype, "dC (state part)", scaled=big)
    assert_close(torch.where(m, uf, 0.0), cf.grad, dtype, "u_f", scaled=big)
    assert_close(torch.where(m, ub, 0.0), cb_.grad, dtype, "u_b", scaled=big)

    # ---- dCB   (a14)
    dCB, da = ops._chunk_scan_bwd_dcb(d["x"], dt_out, csf, csb, dout_x, CB, ngroups=G)
    CBl = _leaf(CB)
    scan(CBl, r["x"], dt64, csf64, csb64, r["C"], _c(pf), _c(pb), None).backward(dy64)
    lim = min(Q, L - (nc - 1) * Q)     # the last chunk's rows and columns past the sequence end are not part of the contract
    got, ref = _c(dCB).clone(), CBl.grad.clone()
    got[:, -1, :, lim:, :] = 0; got[:, -1, :, :, lim:] = 0
    ref[:, -1, :, lim:, :] = 0; ref[:, -1, :, :, lim:] = 0
    assert_close(got, ref, dtype, "dCB", scaled=big)

    # ---- dB, dC: partial sums + the two products with dCB   (a15)
    dB, dC = ops._bmm_chunk_bwd(d["B"], d["C"], dCB, dBs, dCs)
    B64, C64 = _leaf(inp["B"]), _leaf(inp["C"])
    O.stage_bmm_chunk(C64, B64, Q).backward(ref)
    assert_close(dB, B64.grad + _c(dBs).sum(0), dtype, "dB", scaled=big)
    assert_close(dC, C64.grad + _c(dCs).sum(0), dtype, "dC", scaled=big)

    # ---- ddt, dA, ddt_bias   (a16 + a17): everything that reaches dt * A, against autograd of the whole staged forward
    ddt, dA, ddt_bias = ops._chunk_cumsum_bwd(da, uf, ub, vf, vb, ddAcf, ddAcb, ddt_direct, d["dt"], d["A"],
                                              dt_bias=d["dt_bias"], dt_softplus=True)
    dt_l, A_l, bias_l = _leaf(inp["dt"]), _leaf(inp["A"]), _leaf(inp["dt_bias"])
    O.bimamba2_staged(r["x"], dt_l, A_l, r["B"], r["C"], Q, D=r["D"], dt_bias=bias_l, dt_softplus=True)[0].backward(dy64)
    assert_close(ddt, dt_l.grad, dtype, "ddt", scaled=big)
    assert_close(dA, A_l.grad, dtype, "dA", scaled=big)
    assert_close(ddt_bias, bias_l.grad, dtype, "ddt_bias", scaled=big)


# batch, seqlen, H, P, G, N, chunk, dtype: one K step, a last chunk of one position, two channel tiles, grouped heads, fp16
MERGED = [
    (2, 64, 2, 64, 1, 64, 32, torch.bfloat16),
    (1, 257, 4, 64, 2, 64, 256, torch.bfloat16),
    (1, 200, 2, 128, 2, 64, 96, torch.bfloat16),
    (2, 300, 4, 64, 4, 64, 128, torch.float16),
]


@pytest.mark.parametrize("case", MERGED)
def test_dz_and_dstates_in_one_launch(ops, case):
    """bimamba2_chunk_scan_bwd_dz_dstates against the two separate entry points (themselves held to the oracle above), on
    strided z / dout views as the layer passes them, and its refusal of what it does not cover."""
    b, L, H, P, G, N, Q, dtype = case
    gen = torch.Generator().manual_seed(5)
    wide = torch.randn(b, L, 2 * H * P + 8, generator=gen).to(dtype).cuda()
    z = wide[..., :H * P].view(b, L, H, P)                      # row stride 2 H P + 8: a slice of a wider projection
    dout = wide[..., H * P + 8:].view(b, L, H, P)
    out_x = torch.randn(b, L, H, P, generator=gen).to(dtype).cuda()
    C = torch.randn(b, L, G, N, generator=gen).to(dtype).cuda()
    dt = torch.rand(b, L, H, generator=gen).cuda() * 0.1
    A = -torch.rand(H, generator=gen).cuda() - 0.5
    csf, csb, _ = ops._chunk_cumsum_fwd(dt, A, Q)
    dz, dox = ops._chunk_scan_bwd_dz(out_x, z, out_x, dout, Q)
    dz1, dox1, dpf1, dpb1 = ops._chunk_scan_bwd_dz_dstates(z, out_x, dout, C, csf, csb)
    if dtype == torch.bfloat16:
        assert torch.equal(dz1, dz) and torch.equal(dox1, dox)
    else:
        # float16: the compiler rounds the products to 16 bits in one step in one kernel and in two in the other, which
        # moves one value in 10 000 by one unit in the last place
        for got, want in ((dz1, dz), (dox1, dox)):
            torch.testing.assert_close(got.float(), want.float(), rtol=2.0 ** -10, atol=2.0 ** -24)
            assert int((got != want).sum()) <= got.numel() // 2000
    dpf, dpb = ops._chunk_scan_bwd_dstates(C, csf, csb, dox1)    # from the merged launch's own dout_x: the same bits
    assert torch.equal(dpf1, dpf) and torch.equal(dpb1, dpb)
    with pytest.raises(ValueError):                             # float32: the two separate kernels only (unsupported)
        ops._chunk_scan_bwd_dz_dstates(z.float(), out_x.float(), dout.float(), C.float(), csf, csb)


@pytest.mark.parametrize("N,dtype,z", [(64, torch.bfloat16, True), (128, torch.bfloat16, False), (128, torch.float16, True)])
def test_dcb_between_the_merged_launches_in_sixteen_bits(ops, monkeypatch, N, dtype, z):
    """Inside bimamba2_bwd dCB travels in the operands' type, at state dimension 128 too: its reader rounded the float32 values to
    that type before its product anyway, so a caller who brings float32 dCB and dCBT gets the same bits."""
    b, L, H, P, G, Q = 2, 600, 8, 64, 2, 256
    d = to_dev(make_case(b, L, H, P, G, N, dtype, with_z=z))
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(7)).to(dtype).cuda()
    args = (d["x"], d["dt"], d["A"], d["B"], d["C"])
    kw = dict(D=d["D"], z=d["z"], dt_bias=d["dt_bias"], dt_softplus=True)
    res = ops._mamba_chunk_scan_combined_fwd(*args, Q, return_intermediates=False, keep_for_bwd=True, **kw)

    def bwd():
        return ops._mamba_chunk_scan_combined_bwd(dout, *args, res[1], Q, saved=res[9], **kw)

    own, ws = bwd(), ops._Call.workspace

    def with_dcb(call, is_bwd):
        for field in ("dCB", "dCBT"):
            call.new(field, (b, -(-L // Q), G, Q, Q))
        return ws(call, is_bwd)

    monkeypatch.setattr(ops._Call, "workspace", with_dcb)
    for a, c in zip(own, bwd()):
        assert (a is None and c is None) or torch.equal(a, c)


@pytest.mark.parametrize("P", [8, 16, 24, 32, 40, 64, 72, 128])
@pytest.mark.parametrize("L,Q,dtype", [(64, 64, torch.bfloat16), (130, 128, torch.bfloat16), (449, 256, torch.float16)])
def test_dcb_of_heads_that_are_no_whole_steps(ops, P, L, Q, dtype):
    """The ring kernel brings rows in steps of 32 or 64 columns; what a narrower head leaves of them counts as zero.  Against the
    float32 kernel on the same values: products of 16-bit values are exact in float32, so both differ by the order of sums over
    P terms and by a unit in the last place of the exponentials (1e-6 of a value each)."""
    b, H, G = 2, 6, 2
    d = to_dev(make_case(b, L, H, P, G, 16, dtype))
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(5)).to(dtype).cuda()
    csf, csb, dt = ops._chunk_cumsum_fwd(d["dt"], d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    CB = torch.randn(b, -(-L // Q), G, Q, Q, generator=torch.Generator().manual_seed(6)).cuda()
    want = ops._chunk_scan_bwd_dcb(d["x"].float(), dt, csf, csb, dout.float(), CB, ngroups=G)
    got = ops._chunk_scan_bwd_dcb(d["x"], dt, csf, csb, dout, CB, ngroups=G)
    for g, w in zip(got, want):
        assert float((g - w).norm() / w.norm()) < 4e-6


@pytest.mark.parametrize("b,H,G,P,L,Q,dtype", [
    (1, 5, 1, 64, 65, 64, torch.bfloat16),        # few tiles: four waves share one, one of them with two heads; one row in the last chunk
    (1, 3, 1, 64, 449, 256, torch.float16),       # fewer heads than waves, a ragged tile on the diagonal
    (16, 6, 2, 64, 1030, 128, torch.bfloat16),    # 1152 tiles of 3 heads: two waves a tile
    (16, 16, 8, 64, 1030, 64, torch.float16),     # 2176 tiles of 2 heads: one wave a tile
    (4, 9, 9, 64, 1030, 256, torch.bfloat16),     # 2880 tiles of 1 head
])
def test_dcb_by_waves_that_share_a_tile(ops, b, H, G, P, L, Q, dtype):
    """4, 2 or 1 waves take the heads of a tile in turn (bounds as in the test above); rows behind the end of the sequence count nothing"""
    d = to_dev(make_case(b, L, H, P, G, 16, dtype))
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(5)).to(dtype).cuda()
    csf, csb, dt = ops._chunk_cumsum_fwd(d["dt"], d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    CB = torch.randn(b, -(-L // Q), G, Q, Q, generator=torch.Generator().manual_seed(6)).cuda()
    want = ops._chunk_scan_bwd_dcb(d["x"].float(), dt, csf, csb, dout.float(), CB, ngroups=G)
    got = ops._chunk_scan_bwd_dcb(d["x"], dt, csf, csb, dout, CB, ngroups=G)
    for g, w in zip(got, want):
        assert float((g - w).norm() / w.norm()) < 4e-6


@pytest.mark.parametrize("b,H,G,L,Q", [(1, 5, 1, 449, 256), (16, 6, 2, 1030, 128), (16, 16, 8, 1030, 64)])      # four waves, two, one to a tile
@pytest.mark.parametrize("N", [32, 64, 96, 160])
def test_dcb_that_rebuilds_cb(ops, N, b, H, G, L, Q):
    """C.B^T from the rows of C and B, 64 columns at a time, the last 32 of a dstate that is no multiple of 64 by themselves: against the tiles as
    they are computed in float64 from the same values.  The kernel's own are sums of N exact products in float32 (relative to their
    norm within 2^-24 sqrt(N), 1e-6), which adds to the bound of the test above only in the vectors they enter."""
    dtype = torch.bfloat16 if N % 64 else torch.float16
    d = to_dev(make_case(b, L, H, 64, G, N, dtype))
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(5)).to(dtype).cuda()
    csf, csb, dt = ops._chunk_cumsum_fwd(d["dt"], d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    nc = -(-L // Q)
    rows = lambda t: F.pad(t.double(), (0, 0, 0, 0, 0, nc * Q - L)).view(b, nc, Q, G, N).transpose(2, 3)
    CB = torch.matmul(rows(d["C"]), rows(d["B"]).transpose(-1, -2).contiguous()).float()
    want = ops._chunk_scan_bwd_dcb(d["x"].float(), dt, csf, csb, dout.float(), CB, ngroups=G)
    got = ops._chunk_scan_bwd_dcb(d["x"], dt, csf, csb, dout, None, ngroups=G, B=d["B"], C=d["C"])
    for g, w in zip(got, want):
        assert float((g - w).norm() / w.norm()) < 5e-6


@pytest.mark.parametrize("N", [8, 16, 20, 32, 36, 64])
@pytest.mark.parametrize("H,G,P,L,Q,dtype", [(6, 2, 16, 130, 128, torch.bfloat16), (8, 1, 72, 75, 64, torch.float32), (3, 3, 32, 257, 256, torch.float16)])
def test_state_parts_of_db_and_dc_with_narrow_states(ops, N, H, G, P, L, Q, dtype):
    """one, two or four column tiles of the state: dB's and dC's state parts and the decays' gradients against float64"""
    b, hpg = 2, H // G
    d = to_dev(make_case(b, L, H, P, G, N, dtype))
    gen = torch.Generator().manual_seed(9)
    csf, csb, dt = ops._chunk_cumsum_fwd(d["dt"], d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    nc = csf.shape[2]
    sf, sb = (torch.randn(b, nc, H, P, N, generator=gen).cuda() for _ in range(2))
    dout = torch.randn(b, L, H, P, generator=gen).to(dtype).cuda()
    pad = lambda t: F.pad(t.double(), (0, 0, 0, 0, 0, nc * Q - L)).view(b, nc, Q, *t.shape[2:])
    # the kernels' operands: states rounded to the inputs' type; products in float32, rows scaled afterwards
    r = lambda s: s.to(dtype).double()
    scale = lambda e: e.double().exp().permute(0, 2, 3, 1)                                 # (b, nc, Q, H)
    grp = lambda t: t.view(b, nc, Q, G, hpg, N).sum(4)
    wide = lambda t: pad(t).repeat_interleave(hpg, 3)
    for got, rows, mate, wf, wb in (
            (ops._chunk_state_bwd_db(d["x"], dt, csf, csb, sf, sb, B=d["B"], ngroups=G), d["x"], d["B"], dt.double().permute(0, 2, 3, 1) * scale(csf[..., -1:] - csf), dt.double().permute(0, 2, 3, 1) * scale(csb[..., :1] - csb)),
            (ops._chunk_scan_bwd_dC(sf, sb, csf, csb, dout, C=d["C"], ngroups=G), dout, d["C"], scale(csf), scale(csb))):
        tf, tb = (torch.einsum("bcqhp,bchpn->bcqhn", pad(rows), r(s)) for s in (sf, sb))
        want = grp(wf[..., None] * tf + wb[..., None] * tb).reshape(b, nc * Q, G, N)[:, :L]
        assert float((got[0].sum(0) if got[0].dim() == 5 else got[0]).sub(want).norm() / want.norm()) < 1e-5
        for g, w, t in ((got[1], wf, tf), (got[2], wb, tb)):
            want = (w * (t * wide(mate)).sum(-1)).permute(0, 3, 1, 2).reshape(b, H, -1)[:, :, :L]
            assert float((g.reshape(b, H, -1)[:, :, :L] - want).norm() / want.norm()) < 1e-5


@pytest.mark.parametrize("b,H,G,L,Q,hps,dtype,P", [
    (1, 5, 1, 129, 64, 5, torch.bfloat16, 64),        # four waves share a tile, one of them with two heads; one row in the last chunk
    (1, 3, 1, 449, 256, 2, torch.float16, 64),        # fewer heads than waves, the second slice with one; a ragged tile and one with no rows
    (2, 26, 1, 300, 128, 8, torch.bfloat16, 64),      # four slices, the last with two heads
    (16, 4, 2, 1030, 128, 2, torch.bfloat16, 64),     # 576 tiles of two heads and role: two waves a tile
    (16, 16, 8, 1030, 64, 2, torch.float16, 64),      # 2176 tiles of two heads: one wave a tile
    (4, 18, 9, 1030, 256, 1, torch.bfloat16, 64),     # 900 tiles, two slices of one head each
    (1, 7, 1, 200, 128, 7, torch.float16, 128),       # heads in two pieces
    (8, 4, 2, 1030, 64, 2, torch.bfloat16, 128),
])
def test_state_parts_of_db_and_dc_by_waves_that_take_heads(ops, monkeypatch, b, H, G, L, Q, hps, dtype, P):
    """dstate 64, headdim 64 and 128 with the states and their gradients in 16-bit copies, both in one launch: against float64 on the
    copies as they are.  Exact products, float32 sums over P terms and the heads: 1e-5 as above.  (Behind the sequence's end the rows'
    sums are whatever they are: nothing reads them.)"""
    N = 64
    d = to_dev(make_case(b, L, H, P, G, N, dtype))
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(5)).to(dtype).cuda()
    nc, hpg, kept = -(-L // Q), H // G, {}
    own = ops._Call.workspace

    def workspace(c, is_bwd):
        if is_bwd:
            c.p.dbdc_heads = hps
            for name in ("dBs", "dCs"):
                kept[name] = c.new(name, (-(-hpg // hps), b, L, G, N)).fill_(float("nan"))
            for name in ("u_f", "u_b", "v_f", "v_b", "dt_out", "cs_f", "cs_b"):
                kept[name] = c.new(name, (b, H, nc, Q))
            for name in ("states16_f", "states16_b", "dstates16_f", "dstates16_b"):
                kept[name] = c.new(name, (b, nc, H, P, N), dtype)
        return own(c, is_bwd)

    monkeypatch.setattr(ops._Call, "workspace", workspace)
    ops._mamba_chunk_scan_combined_bwd(dout, d["x"], d["dt"], d["A"], d["B"], d["C"], None, Q, dt_bias=d["dt_bias"], dt_softplus=True)
    k = {n: t.double() for n, t in kept.items()}
    pad = lambda t: F.pad(t.double(), (0, 0, 0, 0, 0, nc * Q - L)).view(b, nc, Q, *t.shape[2:])
    rows_of = lambda t: t.permute(0, 2, 3, 1)                                               # (b, nc, Q, H)
    csf, csb, dt = (k[n] for n in ("cs_f", "cs_b", "dt_out"))
    for out, name, rows, mate, w, states in (
            ("dCs", "u", dout, d["C"], (csf.exp(), csb.exp()), "states16"),
            ("dBs", "v", d["x"], d["B"], (dt * (csf[..., -1:] - csf).exp(), dt * (csb[..., :1] - csb).exp()), "dstates16")):
        total = 0
        for way, weight in zip("fb", w):
            t = torch.matmul(pad(rows).transpose(2, 3), k[f"{states}_{way}"]).transpose(2, 3)              # (b, nc, Q, H, N)
            total = total + rows_of(weight)[..., None] * t
            want = (rows_of(weight) * (t * pad(mate).repeat_interleave(hpg, 3)).sum(-1)).permute(0, 3, 1, 2).reshape(b, H, -1)[:, :, :L]
            got = k[f"{name}_{way}"].reshape(b, H, -1)
            assert float((got[:, :, :L] - want).norm() / want.norm()) < 1e-5
        total = total.view(b, nc, Q, G, hpg, N).sum(4).reshape(b, nc * Q, G, N)[:, :L]
        assert float((k[out].sum(0) - total).norm() / total.norm()) < 1e-5


@pytest.mark.parametrize("nc", [1, 7, 8, 9, 16, 17, 63, 64, 65, 129])
@pytest.mark.parametrize("PN", [(8, 4), (40, 30)])
def test_state_passing_over_many_chunks(ops, nc, PN):
    """both recurrences and their gradients at the edges of what is loaded ahead (8 chunks) and handed out together (64), with one
    partly filled workgroup and with two"""
    b, H, Q, (P, N) = 2, 3, 32, PN
    gen = torch.Generator().manual_seed(nc)
    r = lambda *s: torch.randn(*s, generator=gen).cuda()
    cs = [-0.1 * torch.rand(b, H, nc, Q, generator=gen).cuda().cumsum(-1) for _ in range(2)]
    csf, csb = cs[0], cs[1].flip(-1).contiguous()                  # the reverse sums' total stands at the first position
    st, dprev = [r(b, nc, H, P, N) for _ in range(2)], [r(b, nc, H, P, N) for _ in range(2)]
    ef, eb = csf[..., -1].double().exp(), csb[..., 0].double().exp()
    got = ops._state_passing_fwd(*st, csf, csb)
    back = ops._state_passing_bwd(got[0], got[1], csf, csb, *dprev)
    for k, (e, order) in enumerate(((ef, range(nc)), (eb, reversed(range(nc))))):
        order, s, enter = list(order), torch.zeros(b, H, P, N, dtype=torch.float64).cuda(), {}
        for c in order:
            enter[c] = s
            s = e[:, :, c, None, None] * s + st[k][:, c].double()
        g, ds, dda = torch.zeros_like(s), {}, {}
        for c in reversed(order):
            ds[c] = g
            dda[c] = e[:, :, c] * (g * got[k][:, c].double()).sum((-1, -2))
            g = dprev[k][:, c].double() + e[:, :, c, None, None] * g
        stack = lambda d, dim: torch.stack([d[c] for c in range(nc)], dim)
        # float32 recurrences whose terms shrink by e^-1.6 a chunk; inner products of P N terms
        for have, want in ((got[k], stack(enter, 1)), (got[2 + k], s), (back[k], stack(ds, 1)), (back[2 + k], stack(dda, 2))):
            assert float((have - want).norm()) <= 1e-5 * float(want.norm())


@pytest.mark.parametrize("PN", [(64, 16), (64, 64), (72, 68)])
@pytest.mark.parametrize("nc", [1, 2, 3, 4, 5])
def test_state_passing_over_few_chunks(ops, nc, PN):
    """several groups of 1024 elements a workgroup: one group of the state, four, and five (a workgroup with a group behind the end)"""
    test_state_passing_over_many_chunks(ops, nc, PN)


@pytest.mark.parametrize("L", [100, 333, 1000])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_state_passing_beside_dcb_does_not_depend_on_the_batch(L, dtype):
    """many rows: several groups of 1024 elements a workgroup in the launch of dCB; one row: one group where the sequence is long.  The
    gradients of the states, and what is made of them alone, are the same bits"""
    from bi_mamba2_amd.ops import bimamba_chunk_scan_combined
    b, H, P, N = 32, 4, 64, 64
    gen = torch.Generator().manual_seed(L)
    inp = to_dev(make_case(b, L, H, P, 1, N, dtype))
    init = [torch.randn(b, H, P, N, generator=gen).cuda() for _ in range(2)]
    dout = torch.randn(b, L, H, P, generator=gen).to(dtype).cuda()
    dfin = [torch.randn(b, H, P, N, generator=gen).cuda() for _ in range(2)]

    def grads(rows):
        x = inp["x"][:rows].clone().requires_grad_(True)
        st = [t[:rows].clone().requires_grad_(True) for t in init]
        out = bimamba_chunk_scan_combined(x, inp["dt"][:rows], inp["A"], inp["B"][:rows], inp["C"][:rows], 128, dt_bias=inp["dt_bias"], dt_softplus=True,
                                          initial_states_f=st[0], initial_states_b=st[1], return_final_states=True)
        return torch.autograd.grad(out, [x] + st, [dout[:rows]] + [t[:rows] for t in dfin])

    for many, one in zip(grads(b), grads(1)):
        assert torch.equal(many[:1], one)


@pytest.mark.parametrize("H,L,dtype", [(24, 1500, torch.bfloat16), (24, 2700, torch.float16), (20, 4343, torch.bfloat16)])      # 6, 11 and 17 chunks
def test_state_passing_of_float32_states_beside_dcb_does_not_depend_on_the_batch(ops, monkeypatch, H, L, dtype):
    """the same at dstate 128, whose states and their gradients are float32: two rows have 512 workgroups or more of one group, so that a workgroup takes
    two; one row has fewer and keeps one.  The inner products that it leaves for d(dt A) are compared as well"""
    b, P, N, Q, nsplit = 2, 64, 128, 256, 8
    gen = torch.Generator().manual_seed(L)
    inp = to_dev(make_case(b, L, H, P, 1, N, dtype))
    states = lambda: [torch.randn(b, H, P, N, generator=gen).cuda() for _ in range(2)]
    init, dfin, dout = states(), states(), torch.randn(b, L, H, P, generator=gen).to(dtype).cuda()
    own, kept = ops._Call.workspace, {}

    def workspace(c, is_bwd):
        for name in ("ddA_chunk_f", "ddA_chunk_b"):
            kept[name] = c.new(name, (c.p.batch, H, -(-L // Q), nsplit)).fill_(float("nan"))
        return own(c, is_bwd)

    monkeypatch.setattr(ops._Call, "workspace", workspace)

    def results(rows):
        res = ops._mamba_chunk_scan_combined_bwd(dout[:rows], inp["x"][:rows], inp["dt"][:rows], inp["A"], inp["B"][:rows], inp["C"][:rows], None, Q,
                                                 dt_bias=inp["dt_bias"], dt_softplus=True, initial_states=[t[:rows] for t in init], dfinal_states=[t[:rows] for t in dfin])
        return [res[0], *res[8], *kept.values()]

    for many, one in zip(results(b), results(1)):
        assert torch.isfinite(many).all() and torch.equal(many[:1], one)


@pytest.mark.parametrize("H,L,N,dtype", [(17, 1536, 192, torch.bfloat16), (24, 1700, 160, torch.float16), (64, 1600, 192, torch.bfloat16)])      # 6 and 7 chunks: 96 and 112 tiles
def test_heads_of_64_in_one_slice_of_dcb_where_no_launch_adds_slices_up(ops, monkeypatch, H, L, N, dtype):
    """more than 16 heads, dCB in the launch of the state passing; against two slices in buffers of the caller's, a launch that adds them up and a state passing of
    its own.  dB and dC enter the sums of a tile's heads in another order: a float32 sum off by its last bits rounds to another unit of the type now and then"""
    b, G, P, Q = 1, 1, 64, 256
    nc = -(-L // Q)
    inp = to_dev(make_case(b, L, H, P, G, N, dtype))
    dout = torch.randn(b, L, H, P, generator=torch.Generator().manual_seed(L)).to(dtype).cuda()
    grads = lambda: ops._mamba_chunk_scan_combined_bwd(dout, inp["x"], inp["dt"], inp["A"], inp["B"], inp["C"], None, Q, dt_bias=inp["dt_bias"], dt_softplus=True)
    got, own, kept = grads(), ops._Call.workspace, {}

    def workspace(c, is_bwd):
        c.p.dcb_slices = 2
        for name in ("dCB", "dCBT"):
            kept[name] = c.new(name, (2, b, nc, G, Q, Q))
        return own(c, is_bwd)

    monkeypatch.setattr(ops._Call, "workspace", workspace)
    want = grads()
    assert len(kept) == 2
    for i, (g, w) in enumerate(zip(got, want)):
        if not torch.is_tensor(g):
            continue
        assert torch.isfinite(g.float()).all()
        if g.shape == inp["B"].shape:
            assert float((g.double() - w.double()).norm()) <= (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12) * float(w.double().norm())
        else:
            assert torch.equal(g, w), i
