"""A sequence that one chunk holds, without states going in or out: neither the chunk states and their passing nor the state parts of
the backward pass are formed.  A caller that takes the final states has all of them formed; the result is the same in bits, as what is
left out are terms of zero."""
import pytest
import torch

from bi_mamba2_amd import ops
from bi_mamba2_amd.ops import bimamba_chunk_scan_combined
from tests.helpers import make_case, to_dev

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16, torch.float16]
# H, P, G, N, chunk: the kernels that rebuild C.B^T at both state dimensions, headdim 128, the generic ones with their narrow tiles, a
# chunk that is no multiple of 64, one that is no multiple of 32
SHAPES = [(4, 64, 1, 64, 256), (8, 64, 2, 128, 256), (3, 128, 1, 64, 128), (6, 32, 2, 16, 128), (4, 16, 1, 128, 64), (2, 64, 1, 64, 96), (2, 40, 1, 20, 72),
          (36, 64, 1, 64, 256)]


def passes(inp, Q, dout, final, training, seq_idx=None):
    leaves = {k: v.clone().requires_grad_(training) for k, v in inp.items()}
    out = bimamba_chunk_scan_combined(leaves["x"], leaves["dt"], leaves["A"], leaves["B"], leaves["C"], Q, D=leaves["D"], z=leaves.get("z"),
                                      dt_bias=leaves["dt_bias"], dt_softplus=True, return_final_states=final, seq_idx=seq_idx)
    out = out[0] if final else out
    return [out] + (list(torch.autograd.grad(out, list(leaves.values()), dout)) if training else [])


@pytest.mark.parametrize("L", [1, 63, 64, 96, 200, 256])
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", DTYPES)
def test_same_bits_as_with_states(dtype, shape, L):
    H, P, G, N, Q = shape
    L = min(L, Q)
    for with_z in (False, True):
        inp = to_dev(make_case(2, L, H, P, G, N, dtype, with_z=with_z, D_has_hdim=with_z))
        inp = {k: v for k, v in inp.items() if v is not None}
        dout = torch.randn(inp["x"].shape, generator=torch.Generator().manual_seed(L)).to(dtype).cuda()
        for training in (False, True):
            for a, b in zip(passes(inp, Q, dout, False, training), passes(inp, Q, dout, True, training)):
                assert torch.equal(a, b)


@pytest.mark.parametrize("bounds", [((), ()), ((1,), (56,)), ((5, 6, 7), (22,)), ((4, 32), (3, 31, 55))])      # inside a lane's four positions, between them, at both ends
@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("dtype", DTYPES)
def test_same_bits_as_with_states_where_sequences_are_packed(dtype, shape, bounds):
    H, P, G, N, Q = shape
    L = 57
    seq_idx = torch.stack([sum((torch.arange(L) >= at).int() for at in (0,) + row) for row in bounds]).int().cuda()
    assert ops.chunk_size_for_seq_idx(seq_idx, Q) >= L
    inp = {k: v for k, v in to_dev(make_case(2, L, H, P, G, N, dtype, with_z=True)).items() if v is not None}
    dout = torch.randn(inp["x"].shape, generator=torch.Generator().manual_seed(L)).to(dtype).cuda()
    for training in (False, True):
        for a, b in zip(passes(inp, Q, dout, False, training, seq_idx), passes(inp, Q, dout, True, training, seq_idx)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", DTYPES)
def test_rows_at_odd_addresses(dtype):
    """x, B and C as views that the kernels for aligned rows do not take"""
    inp = to_dev(make_case(2, 100, 4, 64, 1, 64, dtype, with_z=True))
    odd = lambda t: torch.cat([t[..., :1], t], -1)[..., 1:]
    dout = torch.randn(inp["x"].shape, generator=torch.Generator().manual_seed(1)).to(dtype).cuda()

    def grads(final):
        leaves = {k: v.detach().requires_grad_(True) for k, v in inp.items()}
        out = bimamba_chunk_scan_combined(odd(leaves["x"]), leaves["dt"], leaves["A"], odd(leaves["B"]), odd(leaves["C"]), 128, D=leaves["D"], z=leaves["z"],
                                          dt_bias=leaves["dt_bias"], dt_softplus=True, return_final_states=final)
        out = out[0] if final else out
        return [out] + list(torch.autograd.grad(out, list(leaves.values()), dout))

    for a, b in zip(grads(False), grads(True)):
        assert torch.equal(a, b)


def test_the_same_call_with_and_without_states_in_turn():
    """through the Python functions, whose workspace sizes are remembered: a size asked for without states is not used with them"""
    inp = to_dev(make_case(1, 100, 4, 64, 1, 64, torch.bfloat16))
    args = (inp["x"], inp["dt"], inp["A"], inp["B"], inp["C"], 128)
    kw = dict(D=inp["D"], dt_bias=inp["dt_bias"], dt_softplus=True, return_intermediates=False)
    outs = [ops._mamba_chunk_scan_combined_fwd(*args, **kw, want_final=f)[0] for f in (False, True, False)]
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("H,P,G,N,Q,heads_per_slice", [(4, 64, 1, 64, 256, 0), (6, 32, 2, 16, 128, 2), (26, 64, 1, 128, 64, 8)])
@pytest.mark.parametrize("dtype", DTYPES)
def test_state_parts_that_the_caller_has_places_for_are_zero(monkeypatch, dtype, H, P, G, N, Q, heads_per_slice):
    """through bimamba2_bwd with buffers of the caller's; the gradients are those without them"""
    b, L = 2, 57
    inp = to_dev(make_case(b, L, H, P, G, N, dtype))
    dout = torch.randn(inp["x"].shape, generator=torch.Generator().manual_seed(2)).to(dtype).cuda()
    rows, sums = (b, H, 1, Q), (-(-(H // G) // (heads_per_slice or 8)), b, L, G, N)
    shapes = {**dict.fromkeys(("u_f", "u_b", "v_f", "v_b"), rows), **dict.fromkeys(("ddA_chunk_f", "ddA_chunk_b"), (b, H, 1, -(-P * N // 1024))), "dBs": sums, "dCs": sums}
    own, kept = ops._Call.workspace, {}

    def workspace(c, is_bwd):
        c.p.dbdc_heads = heads_per_slice
        for name, shape in shapes.items():
            kept[name] = c.new(name, shape).fill_(float("nan"))
        return own(c, is_bwd)

    grads = lambda: ops._mamba_chunk_scan_combined_bwd(dout, inp["x"], inp["dt"], inp["A"], inp["B"], inp["C"], None, Q, dt_bias=inp["dt_bias"], dt_softplus=True)
    want = grads()
    monkeypatch.setattr(ops._Call, "workspace", workspace)
    got = grads()
    assert len(kept) == 8 and all(bool((t == 0).all()) for t in kept.values())
    assert all(a is b or torch.equal(a, b) for a, b in zip(got, want))
