"""GPU parity of the single-direction (causal) comparator, forward and backward, against the oracle's causal operator
in float64, through the C ABI; and its refusal of shapes it has no kernels for."""
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


CASES = [
    # batch, seqlen, H, P, G, N, chunk, dtype, z, D
    (2, 512, 8, 64, 1, 64, 256, torch.bfloat16, True, "h"),
    (1, 700, 4, 64, 2, 64, 256, torch.bfloat16, False, "hp"),     # ragged last chunk (188 valid rows), grouped heads
    (2, 256, 4, 128, 4, 64, 128, torch.float16, True, "h"),       # two headdim tiles, one 16-row tile per wave
    (1, 192, 2, 64, 1, 64, 64, torch.bfloat16, True, "none"),
]


@pytest.mark.parametrize("case", CASES)
def test_causal_forward_and_backward(ops, case):
    b, L, H, P, G, N, Q, dtype, z, Dk = case
    inp = make_case(b, L, H, P, G, N, dtype, with_z=z, with_D=(Dk != "none"), D_has_hdim=(Dk == "hp"))
    d = to_dev(inp)
    leaves = {k: (v.clone().requires_grad_(True) if v is not None else None) for k, v in d.items()}
    out = ops.causal_chunk_scan_combined(leaves["x"], leaves["dt"], leaves["A"], leaves["B"], leaves["C"], Q, D=leaves["D"],
                                         z=leaves["z"], dt_bias=leaves["dt_bias"], dt_softplus=True)
    dout = torch.randn(out.shape, generator=torch.Generator().manual_seed(5)).to(out.dtype)
    out.backward(dout.to(out.device))
    r = to64(inp)
    ref = O.bimamba2_grads(dout.double(), r["x"], r["dt"], r["A"], r["B"], r["C"], D=r["D"], z=r["z"], dt_bias=r["dt_bias"],
                           dt_softplus=True, form="causal", chunk_size=Q)
    assert_close(out, ref["out"], dtype, "out")
    for k in ("x", "B", "C", "z", "dt", "A", "D", "dt_bias"):
        if ref["d" + k] is not None:
            assert_close(leaves[k].grad, ref["d" + k], dtype, "d" + k, scaled=is_reduced("d" + k, dtype))


@pytest.mark.parametrize("H,G,Q,dtype", [(6, 2, 128, torch.bfloat16), (16, 8, 64, torch.float16)])      # two waves a 64 x 64 tile, one
def test_causal_gradients_do_not_depend_on_the_batch(ops, H, G, Q, dtype):
    """16 rows have tiles enough for two waves or one to a tile in the dCB kernel; a row by itself, as in the cases above, has four.  What a wave leaves
    by heads is the same in bits; the heads of a group are added up in another order, so dB and dC may be off by a unit of their type
    now and then"""
    b, L = 16, 1030
    d = to_dev(make_case(b, L, H, 64, G, 64, dtype, with_z=True))
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(5)).to(dtype).cuda()

    def grads(rows):
        leaves = [d[k][rows].clone().requires_grad_(True) for k in ("x", "dt", "z", "B", "C")]
        x, dt, z, B, C = leaves
        out = ops.causal_chunk_scan_combined(x, dt, d["A"], B, C, Q, D=d["D"], z=z, dt_bias=d["dt_bias"], dt_softplus=True)
        return torch.autograd.grad(out, leaves, dout[rows])

    many = grads(slice(0, b))
    for row in (0, b - 1):
        one = grads(slice(row, row + 1))
        assert all(torch.equal(m[row:row + 1], o) for m, o in zip(many[:3], one))
        for m, o in zip(many[3:], one[3:]):
            assert float((m[row].double() - o[0].double()).norm()) <= (2.0 ** -9 if dtype == torch.bfloat16 else 2.0 ** -12) * float(o.double().norm())


def test_causal_refuses_shapes_without_kernels(ops):
    inp = to_dev(make_case(1, 128, 2, 32, 1, 16, torch.float32))
    with pytest.raises(ValueError):
        ops.causal_chunk_scan_combined(inp["x"], inp["dt"], inp["A"], inp["B"], inp["C"], 64, D=inp["D"],
                                       dt_bias=inp["dt_bias"], dt_softplus=True)
