"""GPU tests of the native host path (csrc/host.cpp): the layer as one autograd function against the same layer composed of
its pieces, with frozen parameters and projection biases; the count of packed sequences' boundaries that decides the chunk
size, and gradients that arrive as views the kernels cannot read in place."""
import pytest
import torch

from tests.helpers import assert_close, make_case, to_dev

pytestmark = pytest.mark.gpu

LAYERS = [
    # batch, seqlen, kwargs, dtype, bias of the projections, frozen parameters
    (2, 70, dict(d_model=64, d_state=16, headdim=16, chunk_size=64), torch.float32, True, ()),
    (1, 1, dict(d_model=64, d_state=16, headdim=32, ngroups=2), torch.float32, False, ("A_log", "conv1d.weight")),
    (2, 300, dict(d_model=128, d_state=64, headdim=64), torch.bfloat16, True, ("in_proj.weight", "norm.weight", "D")),
    (1, 257, dict(d_model=128, d_state=128, headdim=64, conv_bias=False), torch.float16, False, ("out_proj.weight",)),
    # in_proj as one library product (2192 columns, 3.4 GFLOP), with its last 144 columns by the own kernel (from 4096 rows on), and
    # an out_proj of 320 columns that stays whole
    (1, 1500, dict(d_model=512), torch.bfloat16, False, ()),
    (2, 2048, dict(d_model=512), torch.bfloat16, False, ()),
    (1, 12000, dict(d_model=320), torch.bfloat16, False, ()),
]


@pytest.mark.parametrize("case", LAYERS)
def test_layer_equals_its_composition(case, monkeypatch):
    from bi_mamba2_amd.modules import BiMamba2, _GradPieces
    batch, seqlen, kw, dtype, bias, frozen = case
    torch.manual_seed(0)
    m = BiMamba2(bias=bias, **kw).cuda().to(dtype)
    for name, p in m.named_parameters():
        p.requires_grad_(name not in frozen)
    u = torch.randn(batch, seqlen, kw["d_model"], device="cuda").to(dtype).requires_grad_(True)
    dy = torch.randn_like(u)
    live = {"u": u, **{n: p for n, p in m.named_parameters() if p.requires_grad and n != "fc_D.weight"}}

    def step():
        out = m(u)
        with torch.no_grad():
            assert_close(m(u), out.detach().double(), dtype, "output without autograd", scaled=True)
        return (out.detach(),) + torch.autograd.grad(out, list(live.values()), dy)

    assert m._native_tensors(u) is not None
    native = step()
    monkeypatch.setattr(_GradPieces, "on_copied", staticmethod(lambda copied: None))      # (its observer gets the composition)
    assert m._native_tensors(u) is None
    for name, a, b in zip(["out"] + list(live), native, step()):
        assert a.shape == b.shape and a.dtype == b.dtype, name
        assert_close(a, b.double(), dtype, name, scaled=True)


@pytest.mark.parametrize("batch,seqlen,kw,dtype,frozen", [
    (1, 1, dict(d_model=64, d_state=16, headdim=32), torch.float32, ()),                             # one row of partial sums; only A_log converted
    (2, 70, dict(d_model=64, d_state=16, headdim=16, conv_bias=False), torch.bfloat16, ()),
    (3, 301, dict(d_model=192, d_state=64, headdim=64), torch.float16, ("D", "conv1d.bias", "norm.weight")),
    (2, 1030, dict(d_model=128, d_state=64, headdim=64, d_conv=3), torch.bfloat16, ("A_log",)),      # more partial sums than one round of loads
])
def test_layer_sums_in_one_launch(batch, seqlen, kw, dtype, frozen, monkeypatch):
    """the sums that end the stages of a layer's backward pass and their conversions in one launch against a launch each: the same
    order of additions, one rounding to the parameter's type, the same bits.  A_log and the norm's weight stay float32."""
    from bi_mamba2_amd.modules import BiMamba2, _GradPieces
    torch.manual_seed(0)
    m = BiMamba2(**kw).cuda().to(dtype)
    m.A_log.data = m.A_log.data.float()
    m.norm.weight.data = m.norm.weight.data.float()
    small = {n: p for n, p in m.named_parameters() if n.split(".")[0] in ("A_log", "D", "dt_bias", "conv1d", "norm")}
    for n, p in small.items():
        p.requires_grad_(n not in frozen)
    live = [p for p in small.values() if p.requires_grad]
    u = torch.randn(batch, seqlen, kw["d_model"], device="cuda").to(dtype).requires_grad_(True)
    dy = torch.randn_like(u)
    step = lambda: torch.autograd.grad(m(u), live, dy)
    assert m._native_tensors(u) is not None
    native = step()
    monkeypatch.setattr(_GradPieces, "on_copied", staticmethod(lambda copied: None))
    for a, b in zip(native, step()):
        assert a.dtype == b.dtype and torch.equal(a, b)


def test_layer_with_hooks_or_autocast_is_composed():
    from bi_mamba2_amd.modules import BiMamba2
    m = BiMamba2(d_model=64, d_state=16, headdim=16, chunk_size=64).cuda()
    u = torch.randn(1, 40, 64, device="cuda")
    seen = []
    handle = m.in_proj.register_forward_hook(lambda mod, args, out: seen.append(out.shape))
    with torch.no_grad():
        hooked = m(u)
        handle.remove()
        assert len(seen) == 1 and torch.allclose(hooked, m(u), rtol=1e-4, atol=1e-5)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            assert m(u).dtype == torch.bfloat16


@pytest.mark.parametrize("chunk", [32, 48, 256])
def test_boundary_count(chunk):
    from bi_mamba2_amd import _lib, ops
    g = torch.Generator().manual_seed(1)
    seq = (torch.rand(3, 521, generator=g) < 0.3).cumsum(1).to(torch.int32)
    seq[1] = 0
    seq[2, 256:] += 1
    p = _lib.Params()
    for k, v in dict(batch=3, seqlen=521, nheads=1, headdim=1, ngroups=1, dstate=1, chunk_size=chunk).items():
        setattr(p, k, v)
    dev, counts = seq.cuda(), torch.empty(3 * -(-521 // chunk), dtype=torch.int32, pin_memory=True)
    p.seq_idx, p.stream = dev.data_ptr(), torch.cuda.current_stream().cuda_stream
    assert _lib.load().bimamba2_seq_boundaries(p, counts.data_ptr()) == 0
    torch.cuda.synchronize()
    want = [ops.seq_boundaries_per_chunk(seq[b:b + 1], chunk) for b in range(3)]
    assert counts.view(3, -1).amax(1).tolist() == want


def test_gradient_views_that_break_the_alignment_are_copied():
    from bi_mamba2_amd import ops
    d = to_dev(make_case(1, 300, 2, 64, 1, 64, torch.bfloat16, with_z=False))
    leaves = [d[k].clone().requires_grad_(True) for k in ("x", "dt", "A", "B", "C")]
    out = ops.bimamba_chunk_scan_combined(*leaves, 256, D=d["D"], dt_bias=d["dt_bias"], dt_softplus=True)
    wide = torch.randn(1, 300, 131, device="cuda", dtype=torch.bfloat16)
    odd = wide[..., 3:].unflatten(-1, (2, 64))
    for view in (odd, odd.transpose(2, 3).contiguous().transpose(2, 3)):
        got = torch.autograd.grad(out, leaves, view, retain_graph=True)
        for a, b in zip(got, torch.autograd.grad(out, leaves, view.contiguous(), retain_graph=True)):
            assert torch.equal(a, b)


def small_layer(**kw):
    """a layer whose projection has 296 columns: no multiple of the 64 its rows are padded to"""
    from bi_mamba2_amd.modules import BiMamba2
    torch.manual_seed(0)
    m = BiMamba2(d_model=64, d_state=16, headdim=16, chunk_size=64, **kw).cuda().to(torch.bfloat16)
    u = torch.randn(2, 100, 64, device="cuda").to(torch.bfloat16).requires_grad_(True)
    return m, u, [u] + [p for n, p in m.named_parameters() if n != "fc_D.weight"]


def scan_of(d, leaves):
    from bi_mamba2_amd import ops
    return ops.bimamba_chunk_scan_combined(*leaves, 64, D=d["D"], z=d["z"], dt_bias=d["dt_bias"], dt_softplus=True)


@pytest.mark.parametrize("how", ["layer", "scan"])
def test_saved_tensor_hooks_and_checkpointing(how):
    from torch.utils.checkpoint import checkpoint
    if how == "layer":
        m, u, leaves = small_layer()
        fn = lambda: m(u)
    else:
        d = to_dev(make_case(2, 100, 4, 16, 2, 16, torch.bfloat16, with_z=True))
        leaves = [d[k].clone().requires_grad_(True) for k in ("x", "dt", "A", "B", "C")]
        fn = lambda: scan_of(d, leaves)
    out = fn()
    dy = torch.randn_like(out)
    want = torch.autograd.grad(out, leaves, dy)
    with torch.autograd.graph.save_on_cpu():
        out = fn()
    kept = torch.autograd.grad(out, leaves, dy)
    for a, b, c in zip(want, kept, torch.autograd.grad(checkpoint(fn, use_reentrant=False), leaves, dy)):
        assert torch.equal(a, b) and torch.equal(a, c)


@pytest.mark.parametrize("how", ["layer", "composed layer", "scan", "scan without kept intermediates"])
def test_second_derivatives_are_refused(how, monkeypatch):
    """the gradients of a recorded backward pass are the same values, and no constants in a loss"""
    from bi_mamba2_amd import ops
    from bi_mamba2_amd.modules import _GradPieces
    if "layer" in how:
        m, u, leaves = small_layer()
        fn = lambda: m(u)
        if how.startswith("composed"):
            monkeypatch.setattr(_GradPieces, "on_copied", staticmethod(lambda copied: None))
    else:
        if "without" in how:
            monkeypatch.setattr(ops, "KEEP_FORWARD_INTERMEDIATES", False)
        d = to_dev(make_case(2, 100, 4, 16, 2, 16, torch.bfloat16, with_z=True))
        leaves = [d[k].clone().requires_grad_(True) for k in ("x", "dt", "A", "B", "C")]
        fn = lambda: scan_of(d, leaves)
    out = fn()
    dy = torch.randn_like(out).requires_grad_("kept" in how)         # (Python functions see it by what comes from upstream)
    recorded = torch.autograd.grad(out, leaves, dy, create_graph=True)
    for a, b in zip(torch.autograd.grad(fn(), leaves, dy.detach()), recorded):
        assert torch.equal(a, b)
    penalty = recorded[0].float().pow(2).sum()
    for loss in (penalty, fn().float().sum() + penalty):
        with pytest.raises(RuntimeError, match="no second derivative|differentiate twice"):
            loss.backward(retain_graph=True)
        if "kept" not in how and "composed" not in how:
            with pytest.raises(RuntimeError, match="no second derivative"):
                torch.autograd.grad(loss, leaves[0], retain_graph=True)


def test_forward_mode_is_refused():
    import torch.autograd.forward_ad as fwAD
    m, u, _ = small_layer()
    d = to_dev(make_case(1, 64, 2, 16, 1, 16, torch.bfloat16, with_z=True))
    with fwAD.dual_level(), torch.no_grad():
        for call in (lambda: m(fwAD.make_dual(u.detach(), torch.ones_like(u))),
                     lambda: scan_of(d, [fwAD.make_dual(d["x"], d["x"])] + [d[k] for k in ("dt", "A", "B", "C")])):
            with pytest.raises((RuntimeError, NotImplementedError)):
                call()


def test_layer_parameters_of_other_shapes():
    m, u, _ = small_layer()
    with torch.no_grad():
        want = m(u)
        m.D = torch.nn.Parameter(m.D[:, None].expand(-1, 16).contiguous())          # one value a channel: the composition takes it
        assert_close(m(u), want.double(), torch.bfloat16, "D per channel", scaled=True)
        with pytest.raises(RuntimeError):
            m(torch.zeros(2, 100, 72, device="cuda", dtype=torch.bfloat16))


def held_for_backward(fn):
    """bytes that the result of fn() keeps besides the tensors it returns"""
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = fn()
    return torch.cuda.memory_allocated() - before - out.untyped_storage().nbytes(), out


def test_cb_kept_or_formed_again():
    """C.B^T is kept for the backward pass with eight heads in a group of 64-position chunks (8 KB for each group and position
    beside 9.5) and formed again there with two (beside 2.4): what belongs to one head is the same, bit for bit"""
    b, L, P, G, N, Q = 2, 200, 16, 2, 16, 64
    d = to_dev(make_case(b, L, 16, P, G, N, torch.bfloat16, with_z=True))
    from bi_mamba2_amd import ops
    dy = torch.randn_like(d["x"])
    nc, cb = -(-L // Q), 2 * 4 * b * -(-L // Q) * G * Q * Q

    def grads(heads):
        x, dt, z = (d[k][:, :, heads].clone().requires_grad_(True) for k in ("x", "dt", "z"))
        A, D, bias = (d[k][heads].clone() for k in ("A", "D", "dt_bias"))
        held, out = held_for_backward(lambda: ops.bimamba_chunk_scan_combined(x, dt, A, d["B"], d["C"], Q, D=D, z=z, dt_bias=bias, dt_softplus=True))
        H = len(heads)
        own = 4 * (3 * b * H * nc * Q + 2 * b * nc * H * P * N) + 2 * x.numel()            # decays, states, the result in front of the gate
        return held, own, (out.detach(),) + torch.autograd.grad(out, (x, dt, z), dy[:, :, heads])

    held, own, all_heads = grads(list(range(16)))
    assert own + cb <= held <= own + cb + 4096
    few = [0, 1, 8, 9]
    held, own, some = grads(few)
    assert own <= held <= own + 4096
    for a, s in zip(all_heads, some):
        assert torch.equal(a[:, :, few], s)


def test_memory_held_for_the_backward_pass():
    """what a call keeps follows its operands, however large C.B^T is beside them (17 MB beside an x of 1 MB)"""
    d = to_dev(make_case(2, 2048, 4, 16, 4, 16, torch.float32, with_z=True))
    from bi_mamba2_amd import ops
    x = d["x"].clone().requires_grad_(True)
    held, out = held_for_backward(lambda: ops.bimamba_chunk_scan_combined(x, d["dt"], d["A"], d["B"], d["C"], 128, D=d["D"], z=d["z"],
                                                                          dt_bias=d["dt_bias"], dt_softplus=True))
    assert held <= 4 * x.numel() * 4
