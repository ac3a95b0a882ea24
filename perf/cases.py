"""The work that users of this package have it do, as cases that can be prepared, run and priced.

A case is a dict of plain values.  ``kind`` says which public entry point it goes through and in which direction:

  scan_fwd    bimamba_chunk_scan_combined under torch.no_grad()                 (inference, feature extraction)
  scan_step   the same function, forward and backward through autograd          (training of a model built on the operator)
  layer_fwd   the BiMamba2 module under torch.no_grad()
  layer_step  the BiMamba2 module, forward and backward, every parameter's gradient included

The remaining keys are the arguments of these: sizes, data type, which of the optional operands (z gate, D, initial states,
packed sequences) are given.  Value distributions are those of the package's own benchmark and tests: x, B, C, z and the
upstream gradient are standard normal, A = -exp(U(log 1, log 16)), dt ~ N(0, 0.5) in front of softplus with a dt_bias that is
the inverse softplus of a log-uniform step in [1e-3, 1e-1].
"""
import math

import torch

from bi_mamba2_amd.modules import BiMamba2
from bi_mamba2_amd.ops import bimamba_chunk_scan_combined

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_BYTES = {"f32": 4, "bf16": 2, "f16": 2}


def _scan(name, kind, batch, seqlen, heads, headdim, groups, dstate, chunk, dtype, z, D, states=False, pack=0):
    """D: "none", "h" (one value a head) or "hp" (one a channel).  states: both initial states go in and both final states come
    out.  pack: 0, or several sequences lie one behind the other in each row, their lengths log-uniform in [pack, 16 * pack]."""
    return dict(name=name, kind=kind, batch=batch, seqlen=seqlen, heads=heads, headdim=headdim, groups=groups, dstate=dstate,
                chunk=chunk, dtype=dtype, z=z, D=D, states=states, pack=pack)


def _layer(name, kind, batch, seqlen, d_model, dstate, groups, dtype):
    return dict(name=name, kind=kind, batch=batch, seqlen=seqlen, d_model=d_model, dstate=dstate, groups=groups, dtype=dtype)


def listed():
    return [
        # The smallest call in use: the baseline's plumbing configuration (a model being brought up in float32, or one short
        # request); what counts is what a call costs before any data is moved.
        _scan("scan_fwd_small_f32", "scan_fwd", 2, 256, 4, 32, 1, 16, 64, "f32", z=False, D="h"),
        # A small float32 model in training: the shape on which the original project plots its times.
        _scan("scan_step_small_f32", "scan_step", 2, 2048, 4, 16, 4, 16, 128, "f32", z=True, D="h"),
        # The baseline's forward configuration: ordinary inference in bf16.
        _scan("scan_fwd_bf16", "scan_fwd", 4, 2048, 32, 64, 1, 64, 256, "bf16", z=True, D="h"),
        # The same shape in training: the headline of the package's benchmark.
        _scan("scan_step_bf16", "scan_step", 4, 2048, 32, 64, 1, 64, 256, "bf16", z=True, D="h"),
        # The baseline's training configuration with eight groups of B and C.
        _scan("scan_step_groups_bf16", "scan_step", 4, 4096, 32, 64, 8, 64, 256, "bf16", z=True, D="h"),
        # The baseline's long sequences (documents, audio, DNA) with the wider state.
        _scan("scan_fwd_long_bf16", "scan_fwd", 2, 16384, 48, 64, 1, 128, 256, "bf16", z=False, D="h"),
        # Training with the wider state, at a length that is no multiple of anything.
        _scan("scan_step_n128_bf16", "scan_step", 2, 3001, 24, 64, 1, 128, 256, "bf16", z=False, D="h"),
        # Training in float32 throughout (fine-tuning, numerics work), ragged as well.
        _scan("scan_step_f32", "scan_step", 2, 1111, 16, 64, 2, 64, 256, "f32", z=True, D="h"),
        # Sequences of different lengths packed into one row, the usual way to train on them without padding.
        _scan("scan_step_packed_bf16", "scan_step", 1, 8192, 24, 64, 1, 64, 256, "bf16", z=True, D="h", pack=64),
        # A long sequence worked through in pieces: states come in and go out, and their gradients with them; float16, wide
        # heads, one D per channel.
        _scan("scan_step_states_f16", "scan_step", 2, 1500, 8, 128, 1, 64, 256, "f16", z=False, D="hp", states=True),
        # One request through one layer of a small vision or text encoder (14 x 14 patches and a class token).
        _layer("layer_fwd_small_bf16", "layer_fwd", 1, 197, 384, 64, 1, "bf16"),
        # The baseline's layer configuration in training.
        _layer("layer_step_bf16", "layer_step", 16, 1024, 768, 64, 1, "bf16"),
    ]


def _cost(case):
    """What draw() holds against the largest listed case: bytes or operations, float32 operations (whose matrix rate is a
    sixteenth) counted at their price."""
    w = work(case)
    return max(w["bytes"], w["flops"] / 50 * (16 if case["dtype"] == "f32" else 1))


def draw(rng):
    most = max(_cost(c) for c in listed())
    log_int = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    while True:
        kind = rng.choice(["scan_fwd", "scan_step", "scan_step", "layer_fwd", "layer_step"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        batch, seqlen = log_int(1, 16), log_int(64, 4096 if kind.startswith("layer") else 16384)
        if kind.startswith("layer"):
            groups = rng.choice([1, 1, 1, 2])
            case = _layer(None, kind, batch, seqlen, 64 * rng.randint(2, 16), rng.choice([64, 64, 128]), groups, dtype)
        else:
            groups = rng.choice([1, 1, 1, 2, 4, 8])
            heads = groups * max(1, log_int(4, 48) // groups)
            case = _scan(None, kind, batch, seqlen, heads, rng.choice([16, 32, 64, 64, 64, 128]), groups,
                         rng.choice([16, 32, 64, 64, 128, 128]), rng.choice([64, 128, 256, 256]), dtype,
                         z=rng.random() < 0.5, D=rng.choice(["none", "h", "h", "hp"]), states=rng.random() < 0.15,
                         pack=log_int(16, 256) if rng.random() < 0.15 else 0)
        del case["name"]
        if _cost(case) <= most:
            return case


def _packed(case, gen):
    """seq_idx of rows that hold several sequences: lengths log-uniform in [pack, 16 * pack]."""
    batch, seqlen, lo = case["batch"], case["seqlen"], case["pack"]
    n = seqlen // lo + 1
    u = torch.rand(batch, n, device="cuda", generator=gen)
    ends = torch.exp(math.log(lo) + u * math.log(16.0)).floor().to(torch.int64).clamp_(min=1).cumsum(1)
    at = torch.arange(seqlen, device="cuda").expand(batch, seqlen).contiguous()
    return torch.searchsorted(ends, at, right=True).to(torch.int32)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    normal = lambda *shape, dtype=dtype: torch.randn(*shape, device="cuda", generator=gen).to(dtype)
    step = case["kind"].endswith("_step")
    batch, seqlen = case["batch"], case["seqlen"]
    if case["kind"].startswith("layer"):
        with torch.random.fork_rng(devices=[torch.cuda.current_device()]):
            torch.manual_seed(seed)
            layer = BiMamba2(d_model=case["d_model"], d_state=case["dstate"], ngroups=case["groups"], device="cuda").to(dtype)
        u = normal(batch, seqlen, case["d_model"]).requires_grad_(step)
        # (fc_D belongs to the module's state but takes no part in its forward pass)
        leaves = [u] + [p for name, p in layer.named_parameters() if not name.startswith("fc_D")]
        return {"layer": layer, "u": u, "leaves": leaves if step else None, "dout": normal(*u.shape) if step else None}
    heads, headdim, groups, dstate = case["heads"], case["headdim"], case["groups"], case["dstate"]
    uniform = lambda *shape: torch.rand(*shape, device="cuda", generator=gen)
    dt0 = torch.exp(uniform(heads) * (math.log(0.1) - math.log(0.001)) + math.log(0.001))
    ops = {
        "x": normal(batch, seqlen, heads, headdim),
        "dt": 0.5 * normal(batch, seqlen, heads, dtype=torch.float32),
        "A": -torch.exp(uniform(heads) * math.log(16.0)),
        "B": normal(batch, seqlen, groups, dstate),
        "C": normal(batch, seqlen, groups, dstate),
        "D": None if case["D"] == "none" else normal(*((heads,) if case["D"] == "h" else (heads, headdim)), dtype=torch.float32),
        "z": normal(batch, seqlen, heads, headdim) if case["z"] else None,
        "dt_bias": dt0 + torch.log(-torch.expm1(-dt0)),
    }
    douts = [normal(batch, seqlen, heads, headdim)]
    if case["states"]:
        ops["initial_states_f"] = normal(batch, heads, headdim, dstate, dtype=torch.float32)
        ops["initial_states_b"] = normal(batch, heads, headdim, dstate, dtype=torch.float32)
        douts += [normal(batch, heads, headdim, dstate, dtype=torch.float32) for _ in range(2)]
    leaves = [t.requires_grad_(step) for t in ops.values() if t is not None]
    opts = {"dt_softplus": True, "return_final_states": case["states"]}
    if case["pack"]:
        opts["seq_idx"] = _packed(case, gen)
    return {"ops": ops, "opts": opts, "chunk": case["chunk"], "leaves": leaves if step else None, "douts": douts if step else None}


def run(state):
    if "layer" in state:
        if state["leaves"] is None:
            with torch.no_grad():
                return state["layer"](state["u"])
        out = state["layer"](state["u"])
        return (out,) + torch.autograd.grad(out, state["leaves"], state["dout"])
    if state["leaves"] is None:
        with torch.no_grad():
            return bimamba_chunk_scan_combined(chunk_size=state["chunk"], **state["ops"], **state["opts"])
    out = bimamba_chunk_scan_combined(chunk_size=state["chunk"], **state["ops"], **state["opts"])
    outs = out if isinstance(out, tuple) else (out,)
    return outs + torch.autograd.grad(outs, state["leaves"], state["douts"])


def _scan_flops(batch, seqlen, heads, headdim, groups, dstate, chunk, step):
    """The chunked algorithm at the caller's chunk size: chunk states and their use in both directions, C.B^T, the product
    over pairs of positions; backward the gradients of each, nothing computed twice."""
    q = min(chunk, seqlen)
    per_head = 2 * q * headdim + 8 * headdim * dstate
    per_group = 2 * q * dstate
    if step:
        per_head += 4 * q * headdim + 16 * headdim * dstate
        per_group += 4 * q * dstate
    return batch * seqlen * (heads * per_head + groups * per_group)


def work(case):
    e, step = _BYTES[case["dtype"]], case["kind"].endswith("_step")
    rows = case["batch"] * case["seqlen"]
    if case["kind"].startswith("layer"):
        dm = case["d_model"]
        inner, bc = 2 * dm, case["groups"] * case["dstate"]
        heads, conv = inner // 64, inner + 2 * bc
        proj = inner + conv + heads
        params = dm * proj + inner * dm + conv * 8 + inner + 3 * heads
        flops = rows * (2 * dm * proj + 2 * inner * dm + 2 * 7 * conv) * (3 if step else 1)
        flops += _scan_flops(case["batch"], case["seqlen"], heads, 64, case["groups"], case["dstate"], 256, step)
        # u and the parameters in, the result out; in training also the gradients: of the result in, of u and the parameters out
        return {"bytes": e * (2 * rows * dm + params) * (2 if step else 1), "flops": flops}
    heads, headdim, groups, dstate = case["heads"], case["headdim"], case["groups"], case["dstate"]
    wide, narrow = e * rows * heads * headdim, e * rows * groups * dstate
    state = 4 * case["batch"] * heads * headdim * dstate
    once = wide * (3 if case["z"] else 2) + 2 * narrow + 4 * rows * heads        # x, out (z), B, C, dt
    if case["states"]:
        once += 4 * state
    # in training every operand has a gradient that is written, every result one that is read
    return {"bytes": once * (2 if step else 1) + (4 * rows if case["pack"] else 0),
            "flops": _scan_flops(case["batch"], case["seqlen"], heads, headdim, groups, dstate, case["chunk"], step)}


def tolerance(case):
    # 16-bit operands carry 8 (bf16) or 11 (f16) bits and enter every product rounded; float32 results differ by the order of
    # their sums and by the resolution of the cumulative decays (exponents of up to a few hundred).  The layer rounds its
    # activations to 16 bits between five operators in each direction.
    rel = {"f32": 5e-5, "bf16": 1e-2, "f16": 2e-3}[case["dtype"]]
    return {"rel": 2 * rel if case["kind"].startswith("layer") and case["dtype"] != "f32" else rel}
