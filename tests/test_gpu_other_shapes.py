"""GPU parity, forward and backward, on the shapes between the kernels' tiles: heads and states narrower than a tile (whole
16-byte vectors of them, and odd widths that are read element by element), the state of 128 columns, and numbers of heads
per group that the dB / dC kernels cut into slices of one to eight."""
import pytest
import torch

from oracle import bimamba2_oracle as O
from tests.helpers import assert_close, is_reduced, make_case, to64, to_dev

pytestmark = pytest.mark.gpu

CASES = [
    # batch, seqlen, H, P, G, N, chunk, dtype, z, D
    (2, 130, 6, 16, 2, 16, 64, torch.bfloat16, True, "h"),        # one 16-column tile of each
    (1, 300, 4, 32, 1, 32, 128, torch.float16, False, "hp"),
    (1, 150, 3, 48, 1, 40, 96, torch.bfloat16, True, "h"),        # whole vectors, no whole tiles
    (1, 150, 3, 20, 1, 12, 96, torch.float32, True, "hp"),        # the same in float32
    (1, 90, 2, 18, 1, 10, 64, torch.float32, False, "none"),      # odd widths
    (1, 90, 2, 18, 2, 10, 64, torch.bfloat16, True, "h"),
    (1, 520, 4, 64, 1, 64, 256, torch.float32, True, "h"),        # float32: whole tiles, three chunks
    (1, 200, 2, 32, 1, 128, 64, torch.float32, False, "h"),       # ... and the wide state
    (2, 300, 5, 64, 1, 128, 256, torch.bfloat16, False, "h"),     # wide state, 16-bit: two n tiles a head, 44 rows in the last chunk
    (1, 257, 4, 128, 2, 128, 128, torch.float16, True, "hp"),     # ... two headdim chunks as well
    (1, 64, 24, 16, 1, 16, 64, torch.bfloat16, False, "h"),       # one chunk, 24 heads in a group
    (1, 300, 11, 64, 1, 64, 256, torch.bfloat16, True, "h"),      # 11 heads: slices of unequal length
]


@pytest.mark.parametrize("case", CASES)
def test_shapes_between_the_tiles(case):
    from bi_mamba2_amd import ops
    b, L, H, P, G, N, Q, dtype, z, Dk = case
    inp = make_case(b, L, H, P, G, N, dtype, with_z=z, with_D=Dk != "none", D_has_hdim=Dk == "hp")
    names = [k for k in ("x", "dt", "A", "B", "C", "D", "z", "dt_bias") if inp[k] is not None]
    d = to_dev(inp)
    leaves = {k: d[k].clone().requires_grad_(True) for k in names}
    out = ops.bimamba_chunk_scan_combined(leaves["x"], leaves["dt"], leaves["A"], leaves["B"], leaves["C"], Q, D=leaves.get("D"),
                                          z=leaves.get("z"), dt_bias=leaves["dt_bias"], dt_softplus=True)
    dout = torch.randn(out.shape, generator=torch.Generator().manual_seed(5)).to(dtype)
    grads = torch.autograd.grad(out, list(leaves.values()), dout.cuda())
    r = to64(inp)
    ref = O.bimamba2_grads(dout.double(), r["x"], r["dt"], r["A"], r["B"], r["C"], D=r["D"], z=r["z"], dt_bias=r["dt_bias"],
                           dt_softplus=True)
    big = dtype != torch.float32                                  # 16-bit operands: the absolute part in units of the RMS
    assert_close(out, ref["out"], dtype, "out", scaled=big)
    for k, g in zip(names, grads):
        assert_close(g, ref["d" + k], dtype, "d" + k, scaled=big or is_reduced("d" + k, dtype))


# dCB in head slices where the grid is small: 11 heads in slices of three (the last of two), 5 in slices of two and three, a 16-bit
# shape, a chunk whose square is no multiple of four (no slices), and the ring of direct loads with a narrow state (9 heads of 64)
@pytest.mark.parametrize("case", [(1, 200, 11, 64, 1, 64, 64, torch.float32, True, "h"), (1, 300, 5, 32, 1, 16, 256, torch.float32, False, "none"),
                                  (2, 130, 10, 32, 2, 16, 64, torch.float16, True, "hp"), (1, 130, 8, 16, 1, 16, 65, torch.float32, False, "h"),
                                  (2, 130, 9, 64, 1, 16, 64, torch.bfloat16, False, "h")])
def test_dcb_head_slices(case):
    test_shapes_between_the_tiles(case)


@pytest.mark.parametrize("headdim,dtype", [(64, torch.bfloat16), (128, torch.float16), (64, torch.float32), (32, torch.bfloat16)])
def test_dcb_slices_of_the_callers_choice(headdim, dtype):
    """9 heads in 4 slices start at 0, 3, 6 and 9: the last one is empty and adds nothing, with the ring of direct loads (16 bits,
    whole 64-column tiles) and through registers"""
    from bi_mamba2_amd import ops
    b, L, H, Q = 2, 100, 9, 64
    d = to_dev(make_case(b, L, H, headdim, 1, 16, dtype))
    csf, csb, dt = ops._chunk_cumsum_fwd(d["dt"], d["A"], Q, dt_bias=d["dt_bias"], dt_softplus=True)
    CB = ops._bmm_chunk_fwd(d["C"], d["B"], Q)
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(3)).to(dtype).cuda()

    def dcb(slices):
        c = ops._Call(b, L, H, headdim, 1, 1, Q, dtype, dout.device)
        c.set_x(d["x"]); c.set_dout(dout)
        for name, t in (("CB", CB), ("dt_out", dt), ("cs_f", csf), ("cs_b", csb)):
            c.put(name, t, torch.float32)
        c.p.dcb_slices = slices
        dCB, dCBT = (c.new(name, (slices, b, 2, 1, Q, Q))[0] for name in ("dCB", "dCBT"))
        da = c.new("da_intra", (b, H, 2, 1, 2, 64))
        c.run("bimamba2_chunk_scan_bwd_dcb")
        return dCB, dCBT, da

    (one, oneT, da1), (four, fourT, da4) = dcb(1), dcb(4)
    assert torch.equal(da1, da4)
    # the same nine float32 terms an element, added in another order
    assert (four - one).norm() <= 1e-6 * one.norm() and torch.equal(fourT, four.transpose(-1, -2))
    assert torch.equal(oneT, one.transpose(-1, -2))
