"""GPU parity of the backward path against torch.autograd on the float64 oracle, through the C ABI."""
import pytest
import torch

from oracle import bimamba2_oracle as O
from tests.helpers import assert_close, is_reduced, make_case, to64, to_dev

pytestmark = pytest.mark.gpu
INF = float("inf")


@pytest.fixture(scope="module")
def ops():
    from bi_mamba2_amd import ops
    return ops


def _run_bwd(ops, inp, Q, sp, lim, seed=5):
    d = to_dev(inp)
    leaves = {k: (v.clone().requires_grad_(True) if v is not None else None) for k, v in d.items()}
    out = ops.bimamba_chunk_scan_combined(leaves["x"], leaves["dt"], leaves["A"], leaves["B"], leaves["C"], Q, D=leaves["D"],
                                          z=leaves["z"], dt_bias=leaves["dt_bias"], dt_softplus=sp, dt_limit=lim)
    g = torch.Generator().manual_seed(seed)
    dout = torch.randn(out.shape, generator=g).to(out.dtype)
    out.backward(dout.to(out.device))
    grads = {"d" + k: (v.grad if v is not None else None) for k, v in leaves.items()}
    r = to64(inp)
    ref = O.bimamba2_grads(dout.double(), r["x"], r["dt"], r["A"], r["B"], r["C"], D=r["D"], z=r["z"], dt_bias=r["dt_bias"],
                           dt_softplus=sp, dt_limit=lim)
    return out, grads, ref


def _check(out, grads, ref, dtype, big=False):
    """big: the case's outputs are far from unit scale (raw dt without softplus: steps of size 1), so the absolute
    tolerance of every tensor is taken in units of its RMS; otherwise only the summed gradients (helpers.REDUCED) are."""
    assert_close(out, ref["out"], dtype, "out", scaled=big)
    for k in ("dx", "dB", "dC", "dz"):
        if ref[k] is not None:
            assert grads[k].dtype == dtype
            assert_close(grads[k], ref[k], dtype, k, scaled=big or is_reduced(k, dtype))
    for k in ("ddt", "dA", "dD", "ddt_bias"):
        if ref[k] is not None:
            assert_close(grads[k], ref[k], dtype, k, scaled=big or is_reduced(k, dtype))


# the reference's own end-to-end backward grid (tests/test_bwd_scan.py:8-16 there)
REF_BWD_GRID = [(b, L, 1, P, 1, N, 32) for b in (1, 2) for L in (32, 64, 128) for P in (1, 4) for N in (1, 4)]


@pytest.mark.parametrize("shape", REF_BWD_GRID)
def test_backward_reference_grid(ops, shape):
    b, L, H, P, G, N, Q = shape
    inp = make_case(b, L, H, P, G, N, torch.float32, with_D=False, ref_style=True)
    out, grads, ref = _run_bwd(ops, inp, Q, True, (0.0, INF))
    _check(out, grads, ref, torch.float32)


E2E = [
    # batch, seqlen, H, P, G, N, chunk, dtype, z, D, bias, softplus, limit
    (2, 256, 4, 32, 1, 16, 64, torch.float32, False, "h", True, True, (0.0, INF)),
    (2, 250, 4, 32, 2, 16, 64, torch.float32, True, "hp", True, True, (0.0, INF)),
    (1, 130, 2, 64, 1, 64, 128, torch.float32, True, "h", False, False, (0.0, INF)),
    (2, 200, 4, 16, 4, 8, 32, torch.float32, False, "none", True, True, (0.01, 0.2)),
    (1, 100, 2, 128, 1, 128, 48, torch.float32, True, "hp", True, True, (0.0, INF)),
    (2, 512, 8, 64, 1, 64, 256, torch.bfloat16, True, "h", True, True, (0.0, INF)),
    (1, 700, 4, 64, 2, 128, 256, torch.bfloat16, False, "h", True, True, (0.0, INF)),
    (2, 256, 4, 64, 4, 64, 128, torch.float16, True, "h", True, True, (0.0, INF)),
    # shapes whose scan kernels rebuild CB themselves, with a ragged last chunk (44 valid rows), grouped heads,
    # resp. two headdim tiles
    (2, 300, 4, 64, 2, 64, 256, torch.bfloat16, False, "hp", True, True, (0.0, INF)),
    (1, 200, 2, 128, 1, 64, 128, torch.float16, True, "h", True, True, (0.0, INF)),
]


@pytest.mark.parametrize("case", E2E)
def test_backward_end_to_end(ops, case):
    b, L, H, P, G, N, Q, dtype, z, Dk, bias, sp, lim = case
    inp = make_case(b, L, H, P, G, N, dtype, with_z=z, with_D=(Dk != "none"), D_has_hdim=(Dk == "hp"), with_bias=bias)
    out, grads, ref = _run_bwd(ops, inp, Q, sp, lim)
    _check(out, grads, ref, dtype, big=not sp)


@pytest.mark.parametrize("case", [E2E[1], E2E[5]])
def test_backward_with_recomputation(ops, case, monkeypatch):
    """The backward pass recomputes the forward intermediates (as the reference does) instead of reading the
    ones the forward kept."""
    monkeypatch.setattr(ops, "KEEP_FORWARD_INTERMEDIATES", False)
    b, L, H, P, G, N, Q, dtype, z, Dk, bias, sp, lim = case
    inp = make_case(b, L, H, P, G, N, dtype, with_z=z, with_D=(Dk != "none"), D_has_hdim=(Dk == "hp"), with_bias=bias)
    out, grads, ref = _run_bwd(ops, inp, Q, sp, lim)
    _check(out, grads, ref, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_sixteen_bit_state_copies_against_float32_states(ops, dtype):
    """Where the kernels can, the composites keep the states entering the chunks (and their gradients) in copies of the
    input's 16-bit type instead of float32, and the scan kernels that know the copies run.  Every kernel that reads the
    entering states rounds them to that type for its MFMA anyway, so both ways must agree within the tolerance of the type
    (different kernels with different rounding points: not bit for bit).  The float32 side: forward with the states returned as tensors, which switches
    the copies off."""
    import ctypes
    from bi_mamba2_amd import _lib
    Q = 256
    inp = make_case(2, 700, 4, 64, 2, 64, dtype, with_z=True)
    d = to_dev(inp)
    args = (d["x"], d["dt"], d["A"], d["B"], d["C"], Q)
    kw = dict(D=d["D"], z=d["z"], dt_bias=d["dt_bias"], dt_softplus=True)
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(7)).to(dtype).cuda()

    c = ops._problem(*args, d["D"], d["z"], d["dt_bias"], True, (0.0, INF))
    assert _lib.load().bimamba2_state_copies(ctypes.byref(c.p)) == 1
    c32 = ops._problem(d["x"].float(), d["dt"], d["A"], d["B"].float(), d["C"].float(), Q, d["D"], d["z"].float(), d["dt_bias"], True, (0.0, INF))
    assert _lib.load().bimamba2_state_copies(ctypes.byref(c32.p)) == 0

    res_c = ops._mamba_chunk_scan_combined_fwd(*args, **kw, return_intermediates=False, keep_for_bwd=True)
    assert res_c[9][2][3] == ops._BLOB_FIELDS_COPIES
    res_f = ops._mamba_chunk_scan_combined_fwd(*args, **kw, return_intermediates=True, keep_for_bwd=True)
    # (two 16-bit results against each other, each with its own rounding: absolute tolerance in units of the RMS)
    assert_close(res_c[0], res_f[0].double(), dtype, "out", scaled=True)
    assert_close(res_c[1], res_f[1].double(), dtype, "out_x", scaled=True)
    g_c = ops._mamba_chunk_scan_combined_bwd(dout, *args[:5], res_c[1], Q, **kw, saved=res_c[9])
    g_f = ops._mamba_chunk_scan_combined_bwd(dout, *args[:5], res_f[1], Q, **kw, saved=res_f[9])
    names = ("dx", "ddt", "dA", "dB", "dC", "dD", "dz", "ddt_bias")
    for name, a, b in zip(names, g_c, g_f):
        assert_close(a, b.double(), dtype, name, scaled=True)


def test_backward_takes_a_misaligned_gradient_view(ops):
    """The gradient arrives as a view that is neither 16-byte aligned nor has strides that are multiples of 8 elements
    (a slice of a wider tensor at an odd column), at a shape where the forward kept only the 16-bit copies of the entering
    states: the backward pass must give what it gives for the contiguous copy of the same values."""
    b, L, H, P, G, N, Q, dtype = 2, 512, 4, 64, 1, 64, 256, torch.bfloat16
    d = to_dev(make_case(b, L, H, P, G, N, dtype, with_z=False))
    wide = torch.randn(b, L, H, P + 3, generator=torch.Generator().manual_seed(3)).to(dtype).cuda()
    view = wide[..., 1:P + 1]
    assert view.data_ptr() % 16 and view.stride(2) % 8
    res = []
    for g in (view, view.contiguous()):
        leaves = {k: d[k].clone().requires_grad_(True) for k in ("x", "dt", "A", "B", "C", "D", "dt_bias")}
        out = ops.bimamba_chunk_scan_combined(leaves["x"], leaves["dt"], leaves["A"], leaves["B"], leaves["C"], Q, D=leaves["D"],
                                              dt_bias=leaves["dt_bias"], dt_softplus=True)
        out.backward(g)
        res.append({k: v.grad for k, v in leaves.items()})
    for k in res[0]:
        assert torch.equal(res[0][k], res[1][k]), k


@pytest.mark.parametrize("b,L,H,P,G,N,Q,dtype,dt_dtype,z", [
    (1, 130, 4, 16, 2, 16, 64, torch.float32, torch.float32, True),        # two row tiles, nothing to add up
    (2, 75, 8, 16, 1, 24, 50, torch.float32, torch.float32, False),        # head slices of dCB, chunk no whole tile
    (1, 257, 12, 24, 1, 72, 128, torch.bfloat16, torch.bfloat16, True),    # slices, two tiles of the state
    (1, 100, 16, 32, 1, 64, 64, torch.float16, torch.float32, False),      # slices with unconditional loads
    (1, 100, 6, 16, 1, 16, 64, torch.bfloat16, torch.float16, True),       # dt of a third type: the two launches
])
def test_last_launch_adds_up_head_slices(ops, b, L, H, P, G, N, Q, dtype, dt_dtype, z):
    """bimamba2_bwd against a caller that brings its own dCB and dCBT, which are added up by a launch of their own, in four slices"""
    d = to_dev(make_case(b, L, H, P, G, N, dtype, with_z=z))
    dt = d["dt"].to(dt_dtype)
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(7)).to(dtype).cuda()
    args, kw = (d["x"], dt, d["A"], d["B"], d["C"]), dict(D=d["D"], z=d["z"], dt_bias=d["dt_bias"], dt_softplus=True)
    res = ops._mamba_chunk_scan_combined_fwd(*args, Q, return_intermediates=False, keep_for_bwd=True, **kw)
    bwd = lambda: ops._mamba_chunk_scan_combined_bwd(dout, *args, res[1] if z else res[0], Q, saved=res[9], **kw)
    own, ws = bwd(), ops._Call.workspace

    def with_dcb(call, is_bwd):
        call.p.dcb_slices = min(4, H // G)
        for field in ("dCB", "dCBT"):
            call.new(field, (call.p.dcb_slices, b, -(-L // Q), G, Q, Q))
        return ws(call, is_bwd)

    ops._Call.workspace = with_dcb
    try:
        brought = bwd()
    finally:
        ops._Call.workspace = ws
    tol = {torch.float32: 1e-5, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]      # (four slices: another order of the same sum, rounded once)
    for a, c in zip(own, brought):
        if a is not None:
            assert float((a.double() - c.double()).norm()) <= tol * float(c.double().norm())


@pytest.mark.parametrize("case", [
    (1, 300, 13, 64, 1, 64, 256, torch.bfloat16, torch.float32, True),     # three slices, the last with fewer heads; a ragged chunk
    (1, 257, 16, 128, 2, 128, 256, torch.float16, torch.float16, False),   # two slices a group; float32 states and gradients
    (1, 130, 24, 64, 1, 64, 128, torch.bfloat16, torch.bfloat16, True),    # the last launch for chunks of up to 128
    (2, 65, 8, 64, 1, 64, 64, torch.bfloat16, torch.float16, False),       # a dt type without it: the slices' own launch
])
def test_head_slices_of_wide_heads(ops, case):
    """the same for the launch that rebuilds C.B^T and passes the states beside it, on grids small enough for slices"""
    test_last_launch_adds_up_head_slices(ops, *case)


@pytest.mark.parametrize("b,L,H,P,G,N,Q,dtype,z", [
    (1, 130, 4, 16, 2, 16, 64, torch.float32, True),          # one column tile of the state, two chunks and a rest
    (1, 128, 3, 64, 1, 32, 128, torch.float32, False),        # two; two headdim tiles a dx workgroup owns one of
    (1, 100, 2, 128, 1, 64, 64, torch.float32, True),         # four, unconditional loads
    (1, 70, 2, 64, 1, 128, 64, torch.float32, False),         # two tiles of 64
    (1, 200, 4, 32, 2, 128, 128, torch.bfloat16, True),
    (1, 65, 5, 128, 5, 16, 64, torch.float16, False),
    (2, 96, 6, 16, 1, 40, 96, torch.bfloat16, True),          # chunk no whole tile: dCB and the states' gradients on their own
])
def test_launches_of_several_roles(ops, b, L, H, P, G, N, Q, dtype, z):
    """bimamba2_bwd with dCB and the states' gradients in one launch and dx, dB and dC in another against the stages one by one: the
    same work in other workgroups, so the same bits where a stage's result is the call's"""
    d = to_dev(make_case(b, L, H, P, G, N, dtype, with_z=z))
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(7)).to(dtype).cuda()
    args, kw = (d["x"], d["dt"], d["A"], d["B"], d["C"]), dict(D=d["D"], z=d["z"], dt_bias=d["dt_bias"], dt_softplus=True)
    res = ops._mamba_chunk_scan_combined_fwd(*args, Q, keep_for_bwd=True, **kw)
    dt_out, csf, csb, sf, sb = res[2:7]
    got = ops._mamba_chunk_scan_combined_bwd(dout, *args, res[1] if z else res[0], Q, saved=res[9], **kw)
    dox = ops._chunk_scan_bwd_dz(res[1], d["z"], res[1], dout, Q)[1] if z else dout
    dpf, dpb = ops._chunk_scan_bwd_dstates(d["C"], csf, csb, dox)
    dsf, dsb = ops._state_passing_bwd(sf, sb, csf, csb, dpf, dpb)[:2]
    CB = ops._bmm_chunk_fwd(d["C"], d["B"], Q)
    dx, _, dD = ops._chunk_scan_chunk_state_bwd_dx(d["x"], dt_out, csf, csb, d["B"], CB, dox, dsf, dsb, D=d["D"])
    assert torch.equal(got[0], dx) and torch.equal(got[5], dD)
    # dB and dC: the slices of heads differ between the two (their sum is rounded in another order)
    dBs = ops._chunk_state_bwd_db(d["x"], dt_out, csf, csb, dsf, dsb, B=d["B"], ngroups=G)[0]
    dCs = ops._chunk_scan_bwd_dC(sf, sb, csf, csb, dox, C=d["C"], ngroups=G)[0]
    dCB = ops._chunk_scan_bwd_dcb(d["x"], dt_out, csf, csb, dox, CB, ngroups=G)[0]
    dB, dC = ops._bmm_chunk_bwd(d["B"], d["C"], dCB, dBs, dCs)
    tol = {torch.float32: 1e-6, torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12}[dtype]      # (now and then one unit of the result's type)
    for g, w in ((got[3], dB), (got[4], dC)):
        assert float((g.double() - w.double()).norm()) <= tol * float(w.double().norm())


@pytest.mark.parametrize("case", [
    (3, 700, 16, 64, 2, 64, 128, torch.float32, True),        # 576 dx workgroups: dB and dC share a launch, dx has its own
    (2, 260, 12, 128, 1, 128, 128, torch.float32, False),     # 288 of dstate 128
    (3, 333, 30, 24, 3, 40, 64, torch.float32, True),         # no whole tiles
    (8, 500, 20, 32, 1, 64, 128, torch.bfloat16, False),      # 640 heads' tiles of 16 bits: one launch
    (9, 500, 32, 32, 1, 64, 128, torch.float16, True),        # 1152: two
    (4, 1030, 32, 64, 16, 96, 128, torch.bfloat16, True),     # two; the state passing is the longer part of dCB's launch
])
def test_db_and_dc_in_one_launch(ops, case):
    """the same where dx does not ride along"""
    test_launches_of_several_roles(ops, *case)
