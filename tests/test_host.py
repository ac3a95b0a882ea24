"""CPU-only tests of the host side: the C-ABI library loads and exports what include/bimamba2.h declares, argument
checks answer with error codes before anything is launched, and the Python mirror of the reference interface
refuses what the reference refuses.  No kernel runs here."""
import ctypes
import os
import re
import subprocess
import sys

import pytest
import torch

from bi_mamba2_amd import _lib, ops
from bi_mamba2_amd.modules import BiMamba2

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    lib = _lib.load()
    header = open(os.path.join(ROOT, "include", "bimamba2.h")).read()
    declared = set(re.findall(r"\b(bimamba2_[a-z_0-9]+)\s*\(", header))
    assert declared == set(_lib.ALL_SYMBOLS), declared ^ set(_lib.ALL_SYMBOLS)
    for name in declared:
        assert getattr(lib, name) is not None
    assert lib.bimamba2_version() >= 100
    assert lib.bimamba2_params_size() == ctypes.sizeof(_lib.Params)


def _params(**kw):
    p = _lib.Params()
    base = dict(batch=2, seqlen=100, nheads=4, headdim=32, ngroups=2, dstate=16, chunk_size=64, dtype=_lib.BF16,
                dt_dtype=_lib.F32, dt_max=float("inf"))
    base.update(kw)
    for k, v in base.items():
        setattr(p, k, v)
    return p


def test_argument_checks_return_error_codes():
    lib = _lib.load()
    assert lib.bimamba2_fwd(None) == -1
    assert lib.bimamba2_fwd(ctypes.byref(_params())) == -3                      # no workspace
    assert lib.bimamba2_chunk_cumsum_fwd(ctypes.byref(_params())) == -1         # null pointers
    assert lib.bimamba2_fwd(ctypes.byref(_params(chunk_size=512))) == -2        # chunk too large
    assert lib.bimamba2_fwd(ctypes.byref(_params(chunk_size=16))) == -2         # chunk too small (reference: >= 32)
    assert lib.bimamba2_fwd(ctypes.byref(_params(headdim=256))) == -2
    assert lib.bimamba2_fwd(ctypes.byref(_params(nheads=3))) == -1              # heads not divisible by groups
    assert lib.bimamba2_fwd(ctypes.byref(_params(dtype=7))) == -2
    assert lib.bimamba2_bwd(ctypes.byref(_params(fwd_saved=1, workspace=1, workspace_bytes=1 << 40))) == -1
    # the forward without a workspace refuses what its built-in buffer cannot hold, before any GPU call
    big = _params(batch=16, seqlen=65536, nheads=64, headdim=64, ngroups=1, dstate=64, chunk_size=256)
    assert lib.bimamba2_fwd_static(ctypes.byref(big)) == -5
    assert lib.bimamba2_fwd_static(None) == -1
    for code in (0, -1, -2, -3, -4, -5, -99):
        assert lib.bimamba2_strerror(code)
    with pytest.raises(ValueError):
        _lib.call("bimamba2_chunk_cumsum_fwd", _params())


def test_workspace_sizes():
    lib = _lib.load()
    p = _params()
    fwd, bwd = lib.bimamba2_workspace_bytes(ctypes.byref(p), 0), lib.bimamba2_workspace_bytes(ctypes.byref(p), 1)
    nc = 2
    states = 2 * 2 * nc * 4 * 32 * 16 * 4
    assert fwd >= states and bwd > 2 * fwd - 4096
    assert lib.bimamba2_workspace_bytes(ctypes.byref(_params(chunk_size=8)), 0) == 0


def _cpu_inputs(b=1, L=64, H=2, P=4, G=1, N=4):
    return (torch.randn(b, L, H, P), torch.randn(b, L, H), -torch.rand(H), torch.randn(b, L, G, N), torch.randn(b, L, G, N))


def test_no_cpu_fallback():
    x, dt, A, B, C = _cpu_inputs()
    with pytest.raises(RuntimeError, match="no CPU fallback"):
        ops.bimamba_chunk_scan_combined(x, dt, A, B, C, 32)


def test_shape_checks_match_the_reference():
    x, dt, A, B, C = _cpu_inputs()
    with pytest.raises(AssertionError):
        ops.bimamba_chunk_scan_combined(x, dt, A, B, C, 16)                       # chunk_size >= 32
    with pytest.raises(AssertionError):
        ops.bimamba_chunk_scan_combined(x, dt[:, :-1], A, B, C, 32)
    with pytest.raises(AssertionError):
        ops.bimamba_chunk_scan_combined(x, dt, A, B, C[..., :-1], 32)
    with pytest.raises(AssertionError):
        ops.bimamba_chunk_scan_combined(x, dt, A, B, C, 32, D=torch.randn(3))
    with pytest.raises(AssertionError):
        ops.bimamba_chunk_scan_combined(x, dt, A, B, C, 32, z=torch.randn(1, 64, 2, 5))


def test_missing_library_fails_loudly(tmp_path):
    code = ("import os; os.environ['BIMAMBA2_LIB'] = %r\n"
            "from bi_mamba2_amd import _lib\n"
            "try:\n    _lib.load()\nexcept RuntimeError as e:\n    print('RAISED', 'no CPU or PyTorch fallback' in str(e))\n") % str(tmp_path / "absent.so")
    out = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert "RAISED True" in out.stdout, out.stdout + out.stderr


def test_bench_refuses_more_than_one_gpu():
    out = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), "--gpus", "2"], capture_output=True, text=True)
    assert out.returncode != 0 and "ONE GPU" in out.stderr


def test_bimamba2_layer_parameters():
    """Same parameter names and shapes as the reference layer (src/ssd/modules.py:65-116 there)."""
    m = BiMamba2(d_model=64, d_state=16, headdim=16, ngroups=2, learnable_init_states=True)
    shapes = {k: tuple(v.shape) for k, v in m.state_dict().items()}
    d_inner, nheads, bc = 128, 8, 2 * 2 * 16
    assert shapes == {
        "in_proj.weight": (2 * d_inner + bc + nheads, 64), "conv1d.weight": (d_inner + bc, 1, 7), "conv1d.bias": (d_inner + bc,),
        "init_states": (nheads, 16, 16), "dt_bias": (nheads,), "A_log": (nheads,), "D": (nheads,),
        "fc_D.weight": (nheads, d_inner), "norm.weight": (d_inner,), "out_proj.weight": (64, d_inner)}
    assert torch.all(m.A_log == 0) and torch.all(m.D == 1)
    dt0 = torch.nn.functional.softplus(m.dt_bias)
    assert dt0.min() >= 1e-4 and dt0.max() <= 0.1 + 1e-6


def test_import_aliases():
    from ssd.bi.ssd_combined import bimamba_chunk_scan_combined, MambaChunkScanCombinedFn
    from ssd.modules import BiMamba2 as Alias
    assert bimamba_chunk_scan_combined is ops.bimamba_chunk_scan_combined
    assert MambaChunkScanCombinedFn is ops.MambaChunkScanCombinedFn and Alias is BiMamba2


def test_norm_and_conv_argument_checks():
    """The layer's two extra entry-point families check their arguments before anything is launched."""
    lib = _lib.load()
    assert lib.bimamba2_rmsnorm_gated_fwd(None) == -1 and lib.bimamba2_conv1d_silu_fwd(None) == -1
    n = _lib.NormParams()
    n.rows, n.cols, n.group_size, n.dtype = 4, 64, 48, _lib.F32
    assert lib.bimamba2_rmsnorm_gated_fwd(ctypes.byref(n)) == -1                # groups do not divide the row
    n.group_size = 64
    assert lib.bimamba2_rmsnorm_gated_fwd(ctypes.byref(n)) == -1                # null pointers
    assert lib.bimamba2_rmsnorm_gated_workspace_bytes(ctypes.byref(n)) == 0     # (0 for a problem that fails the checks)
    c = _lib.ConvParams()
    c.batch, c.seqlen, c.channels, c.width, c.dtype = 2, 16, 8, 4, _lib.BF16
    c.x = c.weight = c.out = 256                                               # never dereferenced: the width check comes first
    assert lib.bimamba2_conv1d_silu_fwd(ctypes.byref(c)) == -2                  # even filter width
    c.width = 11
    assert lib.bimamba2_conv1d_silu_fwd(ctypes.byref(c)) == -2                  # wider than the kernels are built for
    c.width, c.x = 7, None
    assert lib.bimamba2_conv1d_silu_fwd(ctypes.byref(c)) == -1                  # null input
    c.x = 256
    c.dout = c.dx = c.dweight = 256
    assert lib.bimamba2_conv1d_silu_bwd(ctypes.byref(c)) == -3                  # backward without workspace
    assert lib.bimamba2_conv1d_silu_workspace_bytes(ctypes.byref(c)) >= 2 * 16 // 56 * 8 * 8 * 4


def test_causal_flag_and_second_direction_buffers():
    """The single-direction comparator refuses a reverse final state."""
    lib = _lib.load()
    p = _params(causal=1, final_b=256, workspace=256, workspace_bytes=1 << 40)
    assert lib.bimamba2_fwd(ctypes.byref(p)) == -1


def test_state_copies_are_for_the_fast_path_only():
    """bimamba2_state_copies() says where the kernels can keep the entering states in 16-bit copies; the workspace of the
    composites holds them there, and a stage that does not know them refuses them (before any launch)."""
    lib = _lib.load()
    fast = dict(batch=2, seqlen=512, nheads=8, headdim=64, ngroups=1, dstate=64, chunk_size=256,
                x_sb=512 * 8 * 64, x_sl=8 * 64, x_sh=64, B_sb=512 * 64, B_sl=64, B_sg=64, C_sb=512 * 64, C_sl=64, C_sg=64,
                x=256, Bm=256, Cm=256)
    assert lib.bimamba2_state_copies(ctypes.byref(_params(**fast))) == 1
    assert lib.bimamba2_state_copies(ctypes.byref(_params(**dict(fast, dtype=_lib.F32)))) == 0
    assert lib.bimamba2_state_copies(ctypes.byref(_params(**dict(fast, dstate=128, B_sl=128, C_sl=128)))) == 0
    assert lib.bimamba2_state_copies(ctypes.byref(_params())) == 0
    # the copies are part of the forward workspace where they are used, and a caller who brings them saves that much
    stn = 2 * 2 * 8 * 64 * 64
    own = lib.bimamba2_workspace_bytes(ctypes.byref(_params(**fast)), 0)
    brought = lib.bimamba2_workspace_bytes(ctypes.byref(_params(**dict(fast, states16_f=256, states16_b=512))), 0)
    assert own - brought == 2 * stn * 2
    # the generic state passing (float32 problem) does not know the copies
    p = _params(cs_f=256, cs_b=256, states_f=256, states_b=256, states16_f=256, states16_b=256, dtype=_lib.F32)
    assert lib.bimamba2_state_passing_fwd(ctypes.byref(p)) == -2


def test_chunk_size_follows_the_number_of_sequence_boundaries():
    """Packed sequences: the host lowers the chunk size until no chunk holds more boundaries than the float32 cumulative sums
    resolve (runs on CPU tensors: only the count is taken here)."""
    import torch
    from bi_mamba2_amd import ops
    lim = ops.MAX_SEQ_BOUNDARIES_PER_CHUNK
    one = torch.zeros(2, 300, dtype=torch.int32)
    assert ops.seq_boundaries_per_chunk(one, 256) == 0 and ops.chunk_size_for_seq_idx(one, 256) == 256
    # a boundary in front of position l counts for the chunk of l (forward sums) and for the chunk of l - 1 (reverse sums)
    edge = torch.zeros(1, 512, dtype=torch.int32)
    edge[0, 256:] = 1
    assert ops.seq_boundaries_per_chunk(edge, 256) == 1
    four = torch.arange(512)[None].div(4, rounding_mode="floor")            # 64 boundaries per 256 positions
    assert ops.seq_boundaries_per_chunk(four, 256) == 64 and ops.seq_boundaries_per_chunk(four, 128) == 32
    assert ops.chunk_size_for_seq_idx(four, 256) == 128
    single = torch.arange(256)[None]                                        # every token its own sequence
    assert ops.chunk_size_for_seq_idx(single, 256) == 32
    assert ops.seq_boundaries_per_chunk(single, 32) <= lim
    mixed = torch.cat([torch.zeros(1, 256, dtype=torch.int64), 1 + torch.arange(256)[None].div(5, rounding_mode="floor")], dim=1)
    assert ops.chunk_size_for_seq_idx(mixed, 256) == 128                    # the densest chunk decides
    assert ops.chunk_size_for_seq_idx(four, 64) == 64                       # never above what the caller asked for


def test_a_callers_slices_of_db_and_dc_hold_eight_heads():
    """bimamba2_bwd's own slices may be longer; a caller's are refused, before any launch, also where the kernel would take them"""
    lib = _lib.load()
    for more in (dict(dBs=256, dCs=256), dict(dBs=256), dict(dCs=256)):
        p = _params(batch=2, seqlen=512, nheads=26, headdim=64, ngroups=1, dstate=64, chunk_size=256, dbdc_heads=13, workspace=256, workspace_bytes=1 << 40, **more,
                    **dict.fromkeys("x dt A Bm Cm dout dx ddt dA dB dC".split(), 256))
        assert lib.bimamba2_bwd(ctypes.byref(p)) == -1


@pytest.mark.parametrize("seqlen,chunk,saved", [(100, 128, 0), (100, 256, 0), (100, 256, 5), (100, 72, 0), (64, 64, 5), (600, 256, 0), (600, 256, 1), (600, 128, 1)])
@pytest.mark.parametrize("dtype,headdim,dstate", [(_lib.BF16, 64, 64), (_lib.F16, 128, 128), (_lib.BF16, 16, 16), (_lib.F32, 64, 64)])
def test_a_backward_pass_asks_for_every_operand_before_any_launch(dtype, headdim, dstate, seqlen, chunk, saved):
    """rows as the fast kernels take them, over one chunk and over several, with the forward pass's intermediates and without"""
    p = dict(_contiguous(2, seqlen, 4, headdim, 1, dstate, chunk, dtype), has_z=1, has_D=1, has_dt_bias=1, fwd_saved=saved, workspace=256, workspace_bytes=1 << 40)
    p.update({"z" + k[1:]: v for k, v in p.items() if k.startswith("x_")}, **{"dout" + k[1:]: v for k, v in p.items() if k.startswith("x_")})
    if saved:
        p.update(dt_out=256, cs_f=256, cs_b=256)
    if saved & 4 == 0 and saved:
        p.update(states_f=256, states_b=256)
    named = "x dt A Bm Cm dout dx ddt dA dB dC dt_bias D dD z out_x dz".split()
    for missing in named:
        got = _lib.load().bimamba2_bwd(ctypes.byref(_params(**p, **dict.fromkeys(set(named) - {missing}, 256))))
        assert got == -1, (missing, got)


@pytest.mark.parametrize("dtype,headdim,dstate", [(_lib.BF16, 64, 64), (_lib.F16, 128, 64), (_lib.BF16, 64, 128), (_lib.BF16, 16, 16), (_lib.F32, 64, 64)])
@pytest.mark.parametrize("batch,seqlen,chunk", [(2, 100, 128), (2, 100, 256), (2, 100, 72), (4, 2048, 256), (1, 1000, 128)])
@pytest.mark.parametrize("is_bwd", [0, 1])
def test_a_workspace_asked_for_before_the_states_are_named_is_enough(is_bwd, batch, seqlen, chunk, dtype, headdim, dstate):
    """no operand is named either, so that a workspace that is taken leads to the refusal of these, before any launch"""
    lib = _lib.load()
    pairs = ["initial", "final", "states", "states16"] + (["dstates", "dstates16", "dinitial", "dfinal"] if is_bwd else [])
    for heads, groups in ((4, 1), (32, 1), (24, 8)):
        p = dict(_contiguous(batch, seqlen, heads, headdim, groups, dstate, chunk, dtype), workspace=256)
        asked = lib.bimamba2_workspace_bytes(ctypes.byref(_params(**p)), is_bwd)
        for subset in range(1 << len(pairs)):
            named = {f"{n}_{way}": 256 for i, n in enumerate(pairs) if subset >> i & 1 for way in "fb"}
            got = (lib.bimamba2_bwd if is_bwd else lib.bimamba2_fwd)(ctypes.byref(_params(**p, **named, workspace_bytes=asked)))
            assert got == -1, (heads, groups, sorted(named))


def _dcb_slices(**kw):
    """head slices of dCB that bimamba2_bwd works with: what its workspace holds beside a caller's dCB and dCBT"""
    lib = _lib.load()
    own, brought = (lib.bimamba2_workspace_bytes(ctypes.byref(_params(**kw, **extra)), 1) for extra in ({}, dict(dCB=256, dCBT=256)))
    nc = -(-kw["seqlen"] // kw["chunk_size"])
    slices, rest = divmod(own - brought, 2 * 4 * kw["batch"] * nc * kw["ngroups"] * kw["chunk_size"] ** 2)
    assert rest < 512                      # (each piece begins at a multiple of 256)
    return slices


def _contiguous(batch, seqlen, nheads, headdim, ngroups, dstate, chunk_size, dtype):
    return dict(batch=batch, seqlen=seqlen, nheads=nheads, headdim=headdim, ngroups=ngroups, dstate=dstate, chunk_size=chunk_size,
                dtype=dtype, x_sb=seqlen * nheads * headdim, x_sl=nheads * headdim, x_sh=headdim, B_sb=seqlen * ngroups * dstate,
                B_sl=ngroups * dstate, B_sg=dstate, C_sb=seqlen * ngroups * dstate, C_sl=ngroups * dstate, C_sg=dstate)


def test_no_head_slice_of_dcb_is_empty():
    """a slice starts at its number times ceil(heads / slices): 9 heads in 4 slices, 11 in 5 and 17 in 8 would leave the last one
    behind the end of the group"""
    cut = set()
    for dtype, headdim, dstate in ((_lib.F32, 64, 64), (_lib.BF16, 64, 16), (_lib.F16, 32, 16)):
        for rows in (1, 3, 30, 192, 400, 800):                     # (batch, chunk) pairs
            for hpg in range(1, 257):
                n = _dcb_slices(**_contiguous(rows, 64, 2 * hpg, headdim, 2, dstate, 64, dtype))
                assert 1 <= n <= max(8, hpg // 32) and (n - 1) * -(-hpg // n) < hpg, (dtype, rows, hpg, n)
                cut.add(n)
    assert {1, 2, 3, 4, 8} <= cut


# heads in one group, (batch, chunk) pairs, chunk, headdim, dstate, dtype -> slices.  Cut only where the kernel reads C.B^T (dstate
# 64 and 16 bits rebuilds it), where the grid is small, and in 16 bits (in float32 below six heads) only with heads enough for it.
@pytest.mark.parametrize("heads,rows,chunk,headdim,dstate,dtype,slices", [
    (24, 16, 256, 64, 16, _lib.BF16, 3), (24, 16, 256, 64, 64, _lib.BF16, 1), (128, 16, 256, 64, 64, _lib.BF16, 4),
    (24, 32, 256, 64, 16, _lib.BF16, 1), (8, 20, 256, 64, 16, _lib.BF16, 1), (8, 20, 256, 32, 16, _lib.F16, 1),
    (24, 4, 256, 32, 64, _lib.BF16, 8), (8, 20, 256, 64, 64, _lib.F32, 2), (4, 12, 256, 64, 64, _lib.F32, 1),
    (4, 4, 256, 64, 64, _lib.F32, 2), (64, 64, 256, 64, 64, _lib.F32, 2), (24, 64, 65, 64, 64, _lib.F32, 3), (25, 63, 65, 64, 64, _lib.F32, 1)])
def test_head_slices_of_dcb(heads, rows, chunk, headdim, dstate, dtype, slices):
    assert _dcb_slices(**_contiguous(rows, chunk, heads, headdim, 1, dstate, chunk, dtype)) == slices


# wide 16-bit heads over 4 (batch, chunk) pairs: up to 16 heads are cut only where the last launch adds the slices up
@pytest.mark.parametrize("chunk,dstate,more,added", [
    (256, 64, {}, True), (256, 64, dict(dt_dtype=_lib.F16), True), (128, 64, dict(dt_dtype=_lib.BF16), True), (64, 64, {}, True), (128, 96, {}, True),
    (128, 64, dict(dt_dtype=_lib.F16), False), (64, 128, dict(dt_dtype=_lib.F16), False),       # chunks of up to 128: dt in float32 or the type of x
    (192, 64, {}, False), (256, 96, {}, False), (256, 64, dict(dB=258), False), (256, 64, dict(dC_sl=1028), False)])
def test_head_slices_of_dcb_where_nothing_adds_them_up(chunk, dstate, more, added):
    for heads, slices in ((8, 2 if added else 1), (16, 4 if added else 1), (17, 4), (48, 4)):
        assert _dcb_slices(**_contiguous(4, chunk, heads, 64, 1, dstate, chunk, _lib.BF16), **more) == slices, heads


# heads of 64 at the line between 64 and 96 tiles: fewer slices behind it, one where no launch adds them up
@pytest.mark.parametrize("heads,rows,chunk,dstate,slices", [(24, 4, 256, 64, 4), (24, 6, 256, 64, 2), (48, 6, 256, 128, 2), (24, 15, 256, 64, 2), (24, 16, 256, 64, 1), (32, 16, 256, 64, 2),
                                                            (32, 17, 256, 64, 1), (48, 4, 256, 192, 4),
                                                            (24, 6, 256, 192, 1), (64, 6, 256, 192, 1), (65, 6, 256, 192, 2), (24, 32, 256, 192, 1), (24, 7, 192, 64, 4), (24, 11, 192, 64, 1)])
def test_head_slices_of_dcb_of_heads_of_64(heads, rows, chunk, dstate, slices):
    assert _dcb_slices(**_contiguous(rows, chunk, heads, 64, 1, dstate, chunk, _lib.BF16)) == slices


def test_workspace_sizes_are_kept_apart_by_what_the_slices_depend_on():
    """16 heads of 64 in chunks of 128: four slices of dCB with dt in float32, one with dt of a type of its own, or dB at an odd address in chunks of 256"""
    def size(chunk, dt_dtype, dB):
        c = ops._Call(1, 512, 16, 64, 1, 64, chunk, torch.bfloat16, torch.device("cpu"), dt_dtype)
        for name, n in _contiguous(1, 512, 16, 64, 1, 64, chunk, _lib.BF16).items():
            setattr(c.p, name, n)
        c.p.dB = dB
        c.workspace(True)
        return c.p.workspace_bytes
    assert size(128, torch.float16, 256) < size(128, torch.float32, 256)
    assert size(256, torch.float32, 258) < size(256, torch.float32, 256)


# what a caller asks for -> what the kernels run with, at the lines of the rule: workgroups of one row in a launch against the chip's 256
@pytest.mark.parametrize("batch,seqlen,heads,headdim,groups,dstate,dtype,training,chunk,runs", [
    # float32: down to 128 where that fills the chip, else to 64; never up
    (2, 1111, 16, 64, 2, 64, "F32", 1, 256, 128), (1, 4096, 4, 32, 1, 16, "F32", 1, 256, 128), (1, 4064, 4, 32, 1, 16, "F32", 0, 256, 64),
    (1, 100, 1, 16, 1, 16, "F32", 0, 128, 64), (4, 2048, 16, 64, 1, 64, "F32", 1, 64, 64), (4, 2048, 16, 64, 1, 64, "F32", 1, 32, 32),
    # wide heads: up to 256 (without gradients) or 128 where that leaves enough workgroups; never down
    (4, 2048, 16, 64, 1, 64, "BF16", 0, 64, 256), (4, 2048, 16, 64, 1, 64, "BF16", 1, 64, 128), (4, 2048, 15, 64, 1, 64, "BF16", 0, 64, 128), (1, 512, 8, 64, 1, 64, "BF16", 1, 64, 128),
    (1, 508, 8, 64, 1, 64, "BF16", 1, 64, 64), (1, 300, 4, 64, 1, 64, "F16", 0, 64, 64),
    (1, 300, 4, 64, 1, 64, "F16", 0, 256, 256), (4, 2048, 8, 128, 1, 64, "F16", 0, 128, 256), (4, 2048, 8, 128, 1, 64, "F16", 1, 128, 128), (4, 2048, 8, 128, 1, 64, "F16", 1, 192, 192), (4, 136, 8, 128, 2, 128, "BF16", 0, 64, 64),
    (4, 2048, 16, 64, 8, 128, "BF16", 0, 64, 256), (4, 2048, 16, 64, 8, 128, "BF16", 1, 256, 256), (4, 2048, 16, 64, 2, 128, "BF16", 1, 64, 128),
    (4, 2048, 16, 128, 8, 128, "BF16", 1, 64, 128), (1, 1024, 4, 64, 1, 128, "BF16", 1, 64, 128), (1, 1023, 4, 64, 1, 64, "BF16", 1, 64, 64),
    # ... and in training from multiples of 64 only at state dimension 64 (other sizes keep its states in float32)
    (4, 2048, 16, 64, 1, 64, "F16", 1, 96, 96), (4, 2048, 16, 64, 1, 64, "F16", 1, 160, 160), (4, 2048, 16, 64, 1, 64, "F16", 0, 160, 256), (4, 2048, 16, 64, 1, 128, "F16", 1, 96, 128),
    # the other 16-bit shapes: 128, from below only where that fills the chip
    (1, 320, 4, 16, 1, 16, "BF16", 1, 256, 128), (1, 300, 4, 16, 1, 16, "BF16", 1, 64, 64), (4, 1024, 8, 32, 1, 16, "BF16", 0, 64, 128), (4, 1016, 8, 32, 1, 16, "BF16", 0, 64, 64),
    (4, 1024, 8, 96, 1, 64, "BF16", 0, 224, 128), (4, 1024, 8, 64, 1, 80, "F16", 1, 32, 128),
    # ... and from above only where the chunk states take their weighted operand in two parts
    (1, 300, 4, 20, 1, 16, "BF16", 1, 256, 256), (1, 300, 4, 16, 1, 20, "BF16", 0, 256, 256), (1, 300, 4, 64, 1, 192, "F16", 0, 256, 256),
    # ... nor in training without a gate where the sequence is hardly longer than one chunk and does not fit into 128
    (1, 319, 4, 16, 1, 16, "BF16", 1, 256, 256), (1, 129, 4, 16, 1, 16, "BF16", 1, 256, 256), (1, 128, 4, 16, 1, 16, "BF16", 1, 256, 128), (1, 129, 4, 16, 1, 16, "BF16", 0, 256, 128),
    (1, 199, 4, 16, 1, 16, "F16", 1, 160, 160), (1, 200, 4, 16, 1, 16, "F16", 1, 160, 128),
    # sizes that are no whole steps of the kernels stay
    (4, 2048, 16, 64, 1, 64, "F32", 1, 200, 200), (4, 2048, 16, 16, 1, 64, "BF16", 1, 33, 33),
])
def test_chunk_size_that_the_kernels_run_with(batch, seqlen, heads, headdim, groups, dstate, dtype, training, chunk, runs):
    lib = _lib.load()
    p = _params(batch=batch, seqlen=seqlen, nheads=heads, headdim=headdim, ngroups=groups, dstate=dstate, dtype=getattr(_lib, dtype), chunk_size=chunk)
    assert lib.bimamba2_chunk_for(ctypes.byref(p), training) == runs
    for p.batch in (1, 2, 64, batch):                                          # (a row runs as it would alone)
        assert lib.bimamba2_chunk_for(ctypes.byref(p), training) == runs
    if training and dtype != "F32" and 128 < seqlen < 1.25 * chunk and runs == chunk and headdim == dstate == 16:
        p.has_z = 1
        assert lib.bimamba2_chunk_for(ctypes.byref(p), training) == 128
        p.has_z = 0
    p.causal = 1                                                               # (the comparator runs as it is asked to)
    assert lib.bimamba2_chunk_for(ctypes.byref(p), training) == chunk
    p.causal, p.seq_idx = 0, 4096
    assert lib.bimamba2_chunk_for(ctypes.byref(p), training) == (chunk if chunk <= 32 else runs)   # 32: needs no count of boundaries
    assert lib.bimamba2_chunk_for(ctypes.byref(_params(chunk_size=16)), training) == 16            # (refused by the entry points)


@pytest.mark.parametrize("training", [False, True])
def test_python_route_chooses_the_chunk_by_the_operands_themselves(training):
    """bfloat16, 900 positions, 8 heads of 16: chunks of 256 become 128 only where the kernel with two-part operands runs, which takes
    aligned rows; the native route hands the strides and addresses over, and so does the Python one"""
    def at(shape, offset=0, width=None, dtype=torch.bfloat16):         # offset: elements behind an aligned address; width: of a wider row
        rows, n = shape[0] * shape[1], shape[2] * shape[3]
        width = width or n
        return torch.zeros(rows * width + offset, dtype=dtype)[offset:].view(*shape[:2], width)[..., :n].unflatten(-1, shape[2:])
    X, N = (2, 900, 8, 16), (2, 900, 1, 16)
    dt, A = torch.zeros(2, 900, 8), torch.zeros(8)

    def chosen(x, B, C, z=None, **kw):
        leaf = A.clone().requires_grad_(training)
        return ops._chunk_for(x, dt, leaf, B, C, 256, None, z, None, None, **kw)
    assert chosen(at(X), at(N), at(N)) == 128
    assert chosen(at(X), at(N), at(N), at(X)) == 128
    for odd in (dict(offset=1), dict(width=132)):
        assert chosen(at(X, **odd), at(N), at(N)) == 256
    assert chosen(at(X), at(N, offset=1), at(N)) == 256 and chosen(at(X), at(N), at(N, offset=4)) == 256
    # what is converted or copied on its way to the kernels arrives aligned
    assert chosen(at(X), at(N, offset=1, dtype=torch.float32), at(N)) == 128
    assert chosen(at(X), at(N), torch.zeros(2, 16, 1, 901, dtype=torch.bfloat16)[..., 1:].permute(0, 3, 2, 1)) == 128


def test_initial_states_count_as_training():
    """heads of 64 at dstate 128, few of them a group: chunks grow to 256 in a pass without gradients only"""
    x, bc = torch.zeros(4, 2048, 16, 64, dtype=torch.bfloat16), torch.zeros(4, 2048, 8, 128, dtype=torch.bfloat16)
    dt, A, state = torch.zeros(4, 2048, 16), torch.zeros(16), torch.zeros(4, 16, 64, 128)
    assert ops._chunk_for(x, dt, A, bc, bc, 64, None, None, None, None, (state, None)) == 256
    assert ops._chunk_for(x, dt, A, bc, bc, 64, None, None, None, None, (None, state.requires_grad_(True))) == 128


@pytest.mark.parametrize("heads,headdim,groups,dstate", [(16, 64, 1, 64), (16, 64, 1, 128), (8, 128, 1, 64)])
@pytest.mark.parametrize("training", [0, 1])
def test_chunks_of_wide_heads_grow_only_where_their_kernels_run(heads, headdim, groups, dstate, training):
    """4 x 2048 in bfloat16, chunks of 128 asked for, without gradients: 256 with the kernel for aligned rows, as asked with those for any rows"""
    lib, named = _lib.load(), dict(x=256, Bm=256, Cm=256, z=256, has_z=1)

    def chosen(**kw):
        p = _contiguous(4, 2048, heads, headdim, groups, dstate, 128, _lib.BF16)
        z = {"z" + k[1:]: v for k, v in p.items() if k.startswith("x_")}
        return lib.bimamba2_chunk_for(ctypes.byref(_params(**{**p, **z, **named, **kw})), training)
    grown = 128 if training else 256
    assert chosen() == grown and chosen(x_sl=heads * headdim + 8, B_sl=2 * groups * dstate) == grown
    assert lib.bimamba2_chunk_for(ctypes.byref(_params(**_contiguous(4, 2048, heads, headdim, groups, dstate, 128, _lib.BF16))), training) == grown
    for odd in (dict(x=258), dict(Bm=264), dict(Cm=258), dict(x_sl=heads * headdim + 4), dict(B_sl=groups * dstate + 1), dict(C_sb=4097)):
        assert chosen(**odd) == 128, odd
    assert chosen(z=258) == 128 and chosen(z_sl=heads * headdim + 2) == 128 and chosen(B_sl=1 << 22) == 128



def gemm_plan(m, n, k, a_kcontig):
    p, slices = _lib.GemmParams(), ctypes.c_int()
    p.m, p.n, p.k, p.a_kcontig = m, n, k, a_kcontig
    return _lib.load().bimamba2_gemm_plan(ctypes.byref(p), ctypes.byref(slices)), slices.value


# 64 x 64 tiles that share a CU cost each other: the first two took 34 and 30 us in them, 29 and 28 in 128 x 128, the third 4.9 in 128 x 128
@pytest.mark.parametrize("m,n,k,tile", [(1546, 320, 9110, 2), (1546, 320, 7808, 2), (1288, 256, 84, 3), (320, 640, 1300, 3), (3224, 768, 16384, 0), (768, 1536, 16384, 1)])
def test_tiles_of_weight_gradients(m, n, k, tile):
    assert gemm_plan(m, n, k, 0)[0] == tile


# us by the library and by the own kernel: 207 and 258, 285 and 366, 776 and 879, 42 and 53, 129 and 150; 128 and 47, 82 and 71; then the edges of the rule
@pytest.mark.parametrize("rows,columns,terms,own", [(14629, 1280, 5288, False), (9152, 1984, 8126, False), (21882, 2176, 8900, False), (30528, 256, 1544, False), (5760, 1600, 6706, False),
                                                    (128, 3328, 13672, True), (16384, 768, 3224, True),
                                                    (2559, 1536, 6320, True), (2560, 1536, 6320, False), (1000, 4160, 20600, False), (512, 768, 1536, True), (65536, 384, 300, False)])
def test_input_gradients_that_go_to_the_own_kernel(rows, columns, terms, own):
    assert _lib.host().own_input_gradient(rows, columns, terms) == own


# us before and by the own kernel: 19 and 29, 32 and 41, 16 and 25, 28 and 38, 12 and 13; 21 and 16, 14 and 10; then the edges of the rule
@pytest.mark.parametrize("rows,columns,inputs,own", [(116, 8900, 2176, False), (128, 13672, 3328, False), (15617, 1030, 192, False), (600, 7738, 1856, False), (1032, 2708, 640, False),
                                                     (3712, 2062, 448, True), (1344, 2320, 512, True),
                                                     (1000, 2578, 576, True), (1023, 4384, 576, False), (4095, 2318, 448, True), (4096, 2318, 448, False), (3000, 2304, 512, False),
                                                     (3000, 2708, 640, False), (3000, 3000, 576, False)])
def test_forward_products_that_go_to_the_own_kernel(rows, columns, inputs, own):
    """in training; without gradients the line for small ones is at 1.5 GFLOP"""
    assert _lib.host().own_forward_product(rows, columns, inputs, True) == own
    assert _lib.host().own_forward_product(rows, columns, inputs, False) == (own and (rows >= 1024 or 2 * rows * columns * inputs <= 1.5e9))


# one row's workgroups of 64 (float32: 32) positions at the line up to which short sequences go in one launch
ONE_LAUNCH = [(_lib.BF16, 256, 12, 64, 64), (_lib.BF16, 197, 12, 64, 64), (_lib.F16, 256, 8, 64, 128), (_lib.BF16, 256, 12, 64, 32), (_lib.BF16, 64, 48, 64, 64),
              (_lib.BF16, 128, 24, 64, 64), (_lib.F32, 256, 16, 32, 16), (_lib.F32, 256, 10, 32, 32), (_lib.F32, 192, 4, 64, 64), (_lib.F32, 64, 24, 32, 16),
              (_lib.F32, 64, 6, 64, 64)]


@pytest.mark.parametrize("dtype,seqlen,heads,headdim,dstate", ONE_LAUNCH)
def test_short_sequences_in_any_batch(dtype, seqlen, heads, headdim, dstate):
    """few rows are cut into workgroups of some positions, many are not: there each would fetch the whole sequence and form C.B^T again (64 x 256
    positions, 8 heads, dstate 128: 59 us where the chunked launches take 30).  Whether it is one launch does not follow the rows."""
    lib = _lib.load()
    form = lambda batch, heads=heads, **kw: lib.bimamba2_fwd_one_launch(ctypes.byref(
        _params(batch=batch, seqlen=seqlen, nheads=heads, headdim=headdim, ngroups=1, dstate=dstate, chunk_size=64, dtype=dtype, **kw)))
    assert [form(b) for b in (1, 2, 64, 256, 2200000)] == [1, 1, 2, 2, 2] if seqlen > 128 else [2] * 5
    assert form(1, heads + 1) == form(64, heads + 1) == 0
    assert form(64, causal=1) == form(64, initial_f=256) == form(64, states_f=256) == 0


def test_gradients_of_b_and_c_complete_from_one_launch():
    """one slice of heads, chunks of 256, at least 16 (batch, chunk, group), and nobody asked for what the launch would leave out"""
    lib = _lib.load()
    form = lambda **kw: lib.bimamba2_bwd_db_dc_complete(ctypes.byref(_params(**{**dict(
        batch=2, seqlen=2048, nheads=8, headdim=64, ngroups=2, dstate=64, chunk_size=256, x_sb=2048 * 512, x_sl=512, x_sh=64, dout_sb=2048 * 512, dout_sl=512, dout_sh=64,
        B_sb=2048 * 128, B_sl=128, B_sg=64, C_sb=2048 * 128, C_sl=128, C_sg=64), **kw})))
    assert form() == form(dtype=_lib.F16) == form(seqlen=1793) == 1
    assert form(batch=1, seqlen=1792) == form(chunk_size=128) == form(dtype=_lib.F32) == form(dBs=256) == form(dCB=256) == form(dstates_f=256) == form(B_sl=129) == 0


@pytest.mark.parametrize("name,function", [("kernels_gemm.hip", "store_tile"), ("kernels_scan_once.hip", "scan_once_kernel"), ("kernels_scan_once.hip", "scan_once_walk_kernel")])
def test_no_bare_barrier_in_front_of_ordinary_lds_accesses(name, function):
    """these write LDS by stores that the compiler knows of, where other waves read before: s_barrier alone does not keep it from moving them up"""
    text = open(os.path.join(ROOT, "bi_mamba2_amd", "csrc", name)).read()
    body = text[text.index(f" {function}("):]
    body = body[:body.index("\n}\n")]
    assert "ordered_lds_barrier()" in body or "__syncthreads()" in body
    assert not re.search(r"raw_lds_barrier|amdgcn_s_barrier", body)
