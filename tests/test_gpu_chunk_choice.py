"""The chunk size that the kernels run with instead of the caller's (bimamba2_chunk_for): out and every gradient against float64
autograd of the oracle's recurrence, at sizes where the rule takes another one, through the native route and the Python one."""
import pytest
import torch

from oracle import bimamba2_oracle as O
from tests.helpers import make_case

pytestmark = pytest.mark.gpu

# as elsewhere: float32 differs by the order of sums; 16-bit operands enter every product rounded (2^-9 resp. 2^-12) and the results
# are rounded once more, a few roundings one after the other
REL = {torch.float32: 2e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}


@pytest.mark.parametrize("b,L,H,P,G,N,Q,runs,dtype,z,pack", [
    (1, 385, 4, 16, 2, 16, 256, 64, torch.float32, True, False),         # down to 64, one position in the last chunk
    (2, 260, 64, 32, 1, 16, 256, 128, torch.float32, False, False),      # down to 128
    (1, 300, 6, 32, 2, 32, 256, 128, torch.bfloat16, True, False),       # another 16-bit shape: down
    (2, 257, 64, 16, 8, 80, 64, 128, torch.float16, True, False),        # and up, dstate no multiple of 32
    (2, 520, 64, 64, 8, 64, 64, 128, torch.bfloat16, True, False),       # kernels that rebuild C.B^T: up
    (2, 300, 64, 64, 64, 128, 64, 128, torch.bfloat16, False, False),    # state dimension 128 with one head a group
    (2, 300, 64, 16, 8, 16, 64, 128, torch.bfloat16, False, True),       # packed sequences
])
def test_results_do_not_depend_on_the_choice(monkeypatch, b, L, H, P, G, N, Q, runs, dtype, z, pack):
    from bi_mamba2_amd import ops
    inp = make_case(b, L, H, P, G, N, dtype, with_z=z)
    d = {k: None if v is None else v.cuda().requires_grad_(True) for k, v in inp.items()}
    si = (torch.arange(L) // 45).expand(b, L).contiguous() if pack else None
    si_gpu = si.to(torch.int32).cuda() if pack else None
    assert ops._chunk_for(d["x"], d["dt"], d["A"], d["B"], d["C"], Q, d["D"], d["z"], d["dt_bias"], si_gpu) == runs
    dout = torch.randn(inp["x"].shape, generator=torch.Generator().manual_seed(3)).to(dtype)
    # (the recurrence step by step in float64, on the GPU: many heads, where the rule chooses by the size of the launch)
    r = {k: None if v is None else v.detach().double().cuda().requires_grad_(True) for k, v in inp.items()}
    want = O.bimamba2_sequential(r["x"], r["dt"], r["A"], r["B"], r["C"], D=r["D"], z=r["z"], dt_bias=r["dt_bias"], dt_softplus=True,
                                 **({"seq_idx": si.cuda()} if pack else {}))[0]
    names = [k for k, v in r.items() if v is not None]
    want = (want.detach(),) + torch.autograd.grad(want, [r[k] for k in names], dout.double().cuda())
    for keep in (True, False):                                           # native route, Python route
        monkeypatch.setattr(ops, "KEEP_FORWARD_INTERMEDIATES", keep)
        out = ops.bimamba_chunk_scan_combined(d["x"], d["dt"], d["A"], d["B"], d["C"], Q, D=d["D"], z=d["z"], dt_bias=d["dt_bias"],
                                              dt_softplus=True, seq_idx=si_gpu)
        got = (out.detach(),) + torch.autograd.grad(out, [d[k] for k in names], dout.cuda())
        for name, g, w in zip(["out"] + names, got, want):
            err = (g.double() - w).norm() / w.norm()
            assert err < REL[dtype], (name, float(err))


@pytest.mark.parametrize("L,H,P,G,N,Q,dtype,z", [
    (520, 128, 64, 8, 64, 64, torch.bfloat16, True), (300, 128, 64, 1, 128, 64, torch.bfloat16, True), (300, 128, 64, 2, 64, 64, torch.float16, True),
    (520, 128, 64, 8, 64, 160, torch.float16, True), (300, 128, 64, 1, 64, 96, torch.float16, True), (300, 128, 32, 2, 32, 256, torch.bfloat16, True),
    (300, 128, 16, 8, 16, 256, torch.float16, True), (300, 128, 16, 2, 16, 256, torch.float32, True),
    (200, 128, 32, 2, 32, 256, torch.bfloat16, False), (128, 128, 32, 1, 16, 256, torch.float16, False)])
def test_no_result_is_further_off_than_in_the_chunks_asked_for(monkeypatch, L, H, P, G, N, Q, dtype, z):
    """errors against float64 in the chunks that the rule takes over those in the caller's, of a pass with and one without gradients.
    Tensors of tens of thousands of elements and more agree to a percent, with float16's 0.4 % for chunks twice as long; dA and ddt_bias
    have 256 values here, and two root mean squares of 256 independent errors differ by 1 / sqrt(256) = 6 %: 2.5 times that.  (dD takes
    the same sums over a chunk's positions whatever the chunks are.)"""
    from bi_mamba2_amd import ops
    chosen, errors = ops._chunk_for, {}
    monkeypatch.setattr(ops, "KEEP_FORWARD_INTERMEDIATES", False)
    for seed in (0, 1):
        d = {k: None if v is None else v.cuda().requires_grad_(True) for k, v in make_case(1, L, H, P, G, N, dtype, with_z=z, seed=seed).items()}
        dout = torch.randn(1, L, H, P, generator=torch.Generator().manual_seed(seed)).to(dtype).cuda()
        d = {k: v for k, v in d.items() if v is not None}
        r = {k: v.detach().double().requires_grad_(True) for k, v in d.items()}
        want = O.bimamba2_sequential(r["x"], r["dt"], r["A"], r["B"], r["C"], D=r["D"], z=r.get("z"), dt_bias=r["dt_bias"], dt_softplus=True)[0]
        want = (want.detach(),) * 2 + torch.autograd.grad(want, list(r.values()), dout.double())
        for side, rule in ((0, chosen), (1, lambda x, dt, A, B, C, chunk_size, *a: chunk_size)):
            monkeypatch.setattr(ops, "_chunk_for", rule)
            call = lambda: ops.bimamba_chunk_scan_combined(d["x"], d["dt"], d["A"], d["B"], d["C"], Q, D=d["D"], z=d.get("z"), dt_bias=d["dt_bias"], dt_softplus=True)
            with torch.no_grad():
                alone = call()
            out = call()
            got = (alone, out.detach()) + torch.autograd.grad(out, list(d.values()), dout)
            for name, g, w in zip(["out without gradients", "out"] + list(d), got, want):
                errors.setdefault(name, [0.0, 0.0])[side] += float((g.double() - w).norm() ** 2 / w.norm() ** 2)
    for name, (ours, asked) in errors.items():
        if name != "D":
            assert ours ** 0.5 <= (1.15 if name in ("A", "dt_bias") else 1.01) * asked ** 0.5, (name, ours ** 0.5, asked ** 0.5)


@pytest.mark.parametrize("odd", [(), ("x",), ("B",), ("dout",)])
def test_both_routes_choose_the_same(monkeypatch, odd):
    """operands at an odd element, which another kernel of the chunk states takes: the route through Python runs in the chunks that
    the native one runs in, with the same kernels, so that the results are equal in bits"""
    from bi_mamba2_amd import ops
    b, L, H, P, N, dtype = 2, 900, 8, 16, 16, torch.bfloat16

    def place(name, t):
        if t is None or name not in odd:
            return t
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)
    d = {k: None if v is None else place(k, v.cuda()).requires_grad_(True) for k, v in make_case(b, L, H, P, 1, N, dtype).items()}
    dout = place("dout", torch.randn(b, L, H, P, generator=torch.Generator().manual_seed(3)).to(dtype).cuda())
    leaves = [v for v in d.values() if v is not None]

    def run(**kw):
        out = ops.bimamba_chunk_scan_combined(d["x"], d["dt"], d["A"], d["B"], d["C"], 256, D=d["D"], dt_bias=d["dt_bias"], dt_softplus=True, **kw)
        return (out.detach(),) + torch.autograd.grad(out, leaves, dout)
    native, places = run(), run(grad_places={})
    monkeypatch.setattr(ops, "KEEP_FORWARD_INTERMEDIATES", False)
    for route in (places, run()):
        for k, a, w in zip(["out"] + [k for k, v in d.items() if v is not None], route, native):
            assert torch.equal(a, w), k


@pytest.mark.parametrize("keep", [True, False])
@pytest.mark.parametrize("L,H,P,N", [(900, 8, 16, 16), (300, 4, 64, 64)])        # two-part chunk states; 16-bit states kept for the backward pass
def test_a_contiguous_gradient_at_an_odd_address_is_copied(monkeypatch, keep, L, H, P, N):
    from bi_mamba2_amd import ops
    monkeypatch.setattr(ops, "KEEP_FORWARD_INTERMEDIATES", keep)
    d = {k: None if v is None else v.cuda().requires_grad_(True) for k, v in make_case(2, L, H, P, 1, N, torch.bfloat16).items()}
    dout = torch.randn(2, L, H, P, generator=torch.Generator().manual_seed(3)).bfloat16().cuda()
    odd = torch.cat([dout.new_zeros(1), dout.flatten()])[1:].view(dout.shape)
    leaves = [v for v in d.values() if v is not None]
    out = ops.bimamba_chunk_scan_combined(d["x"], d["dt"], d["A"], d["B"], d["C"], 256, D=d["D"], dt_bias=d["dt_bias"], dt_softplus=True)
    want, got = (torch.autograd.grad(out, leaves, g, retain_graph=True) for g in (dout, odd))
    for name, a, w in zip([k for k, v in d.items() if v is not None], got, want):
        assert torch.equal(a, w), name


@pytest.mark.parametrize("L,H,P,N,Q,dtype", [
    (1024, 8, 64, 64, 256, torch.float32), (1024, 16, 32, 16, 128, torch.float32), (1024, 8, 64, 64, 64, torch.bfloat16), (520, 8, 64, 128, 64, torch.bfloat16),
    (1024, 8, 32, 16, 64, torch.float16), (300, 12, 20, 16, 64, torch.bfloat16)])
@pytest.mark.parametrize("training", [False, True])
def test_a_row_does_not_depend_on_the_batch(L, H, P, N, Q, dtype, training):
    """forward results of a row alone, in two rows and in eight: equal in bits, at sizes on both sides of the lines of the chunk choice"""
    from bi_mamba2_amd import ops
    d = {k: None if v is None else v.cuda() for k, v in make_case(8, L, H, P, 1, N, dtype, with_z=True).items()}

    def run(rows):
        x, dt, B, C, z = (d[k][rows].requires_grad_(training) for k in ("x", "dt", "B", "C", "z"))
        return ops.bimamba_chunk_scan_combined(x, dt, d["A"], B, C, Q, D=d["D"], z=z, dt_bias=d["dt_bias"], dt_softplus=True, return_final_states=True)
    alone = run(slice(7, 8))
    for rows in (slice(6, 8), slice(0, 8)):
        for name, got, want in zip(("out", "final_f", "final_b"), run(rows), alone):
            assert torch.equal(got[-1:], want), (name, rows)

