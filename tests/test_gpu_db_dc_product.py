"""dB and dC complete from the launch that sums their state parts (one slice of heads, chunks of 256, 16 bits), against the two launches that
run where the caller brings dCB in float32: the same products in the same order, so the same bits."""

import ctypes

import pytest
import torch

from bi_mamba2_amd import _lib
from tests.helpers import make_case, to_dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from bi_mamba2_amd import ops
    return ops


# batch, heads, groups, headdim: four, two and one wave to a tile of 64 rows (at eight chunks), heads in two pieces
SHAPES = [(2, 8, 2, 64), (2, 32, 8, 64), (4, 32, 8, 64), (2, 3, 1, 64), (4, 16, 8, 128), (1, 4, 2, 128)]


def grads(ops, d, dout, Q=256):
    args = (d["x"], d["dt"], d["A"], d["B"], d["C"])
    kw = dict(D=d.get("D"), z=d.get("z"), dt_bias=d["dt_bias"], dt_softplus=True)
    res = ops._mamba_chunk_scan_combined_fwd(*args, Q, return_intermediates=False, keep_for_bwd=True, **kw)
    return ops._mamba_chunk_scan_combined_bwd(dout, *args, res[1], Q, saved=res[9], **kw)


def compare(ops, monkeypatch, d, dout):
    b, L = d["x"].shape[:2]
    G, N = d["B"].shape[2:]
    ws, complete = ops._Call.workspace, []

    def asked(call, is_bwd):
        ws(call, is_bwd)
        if is_bwd:
            complete.append(_lib.load().bimamba2_bwd_db_dc_complete(ctypes.byref(call.p)))

    monkeypatch.setattr(ops._Call, "workspace", asked)
    got = grads(ops, d, dout)

    def with_dcb(call, is_bwd):
        if is_bwd:
            for field in ("dCB", "dCBT"):
                call.new(field, (b, -(-L // 256), G, 256, 256))
        return asked(call, is_bwd)

    monkeypatch.setattr(ops._Call, "workspace", with_dcb)
    want = grads(ops, d, dout)
    assert complete == [1, 0]
    seen = 0
    for a, c in zip(got, want):
        assert (a is None) == (c is None)
        if a is not None:
            assert bool(torch.isfinite(a.float()).all()) and torch.equal(a, c)
            seen += a.shape == (b, L, G, N)
    assert seen == 2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("b,H,G,P", SHAPES)
@pytest.mark.parametrize("L", [2048, 1793, 1855, 1856, 1921, 1952, 2047])      # rows of the last chunk: 256, 1, 63, 64, 129, 160, 255
def test_rows(ops, monkeypatch, b, H, G, P, L, dtype):
    d = to_dev(make_case(b, L, H, P, G, 64, dtype, with_z=L % 2 == 0))
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(L)).to(dtype).cuda()
    compare(ops, monkeypatch, d, dout)


@pytest.mark.parametrize("b,H,G,P", SHAPES[:3])
def test_views_and_what_lies_behind_the_end(ops, monkeypatch, b, H, G, P):
    """B and C as slices of a wider buffer, NaN in every element that is not theirs"""
    L = 900
    d = to_dev(make_case(b, L, H, P, G, 64, torch.bfloat16))
    for k, spare in (("B", 8), ("C", 24)):
        wide = torch.full((b, L + 70, G, 64 + spare), float("nan"), dtype=torch.bfloat16, device="cuda")
        wide[:, :L, :, :64] = d[k]
        d[k] = wide[:, :L, :, :64]
    dout = torch.randn(d["x"].shape, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    compare(ops, monkeypatch, d, dout)
