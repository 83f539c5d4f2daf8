"""The calls that a program built on this framework makes, at the sizes it makes them.

`listed()` names the workloads, `draw()` gives others of the same ranges, `prepare()` makes what a
program holds before the call, `run()` is one pass through the public entry points, `work()` the bytes
and operations of a pass that no implementation can leave out, `tolerance()` how far two correct
implementations of the same precision may lie apart.

Shapes are those of the repository's benchmark configurations and of its tests' families of sizes:
b batch, nh heads, L sequence length, d features per head, Q chunk size (EMA scan); in the Mamba-2 SSD
cases P is the head size, N the state size and g the number of B / C groups.
"""
import math
import os
import sys

import torch

# the package that is measured is the one of the tree this runs in (its root is the working folder)
sys.path.insert(0, os.path.join(os.getcwd(), "triton-kernels_amd"))

from kernels.ema_kernels.ema_combined_fwd import ema_matmul_scan_combined
from kernels.ema_kernels.ema_cumsum import ema_chunk_cumsum_fwd
from kernels.ema_kernels.ema_scan_fwd import _ema_scan_fwd
from kernels.ema_kernels.ema_state_fwd import _ema_chunk_state_fwd
from kernels.ema_kernels.ema_state_pass import _ema_state_passing_fwd
from kernels.ema_kernels_bwd.ema_chunk_scan_bwd_dc import _ema_chunk_scan_bwd_dC
from kernels.ema_kernels_bwd.ema_chunk_scan_chunk_state_bwd_dx import _chunk_scan_chunk_state_bwd_dx as _ema_bwd_dx
from kernels.ema_kernels_bwd.ema_chunk_state_bwd_db import _ema_chunk_state_bwd_db
from kernels.ema_kernels_bwd.ema_scan_bwd import _ema_chunk_scan_bwd_dstates
from kernels.ema_kernels_bwd.ema_scan_da import _ema_chunk_scan_bwd_ddAcs_stable
from kernels.ema_kernels_bwd.ema_state_passing_bwd_dstates import _ema_state_passing_bwd
from kernels.ema_seq import ema_seq_scan
from kernels.mamba_kernels.mamba_bmm import _bmm_chunk_fwd
from kernels.mamba_kernels.mamba_combined_fwd import _mamba_chunk_scan_combined_fwd, mamba_chunk_scan_combined_fwd
from kernels.mamba_kernels_bwd.mamba_chunk_scan_bwd_da import _chunk_scan_bwd_ddAcs_stable
from kernels.mamba_kernels_bwd.mamba_chunk_scan_bwd_dc import _chunk_scan_bwd_dC
from kernels.mamba_kernels_bwd.mamba_chunk_scan_chunk_state_bwd_dx import _chunk_scan_chunk_state_bwd_dx
from kernels.mamba_kernels_bwd.mamba_chunk_state_bwd_db import _chunk_state_bwd_db
from kernels.mamba_kernels_bwd.mamba_scan_state_passing_bwd import _chunk_scan_state_passing_bwd

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16}
_MAX_EMA = 4 * 2 * 32768 * 1024   # elements of x in the largest EMA case
_MAX_SSD = 8 * 8192 * 32 * 64     # elements of x in the largest SSD case


def listed():
    return [
        # EMA scan, a training step at the smallest configuration: launches and host work
        dict(name="ema_step_small", op="ema_step", dtype="f32", b=1, nh=2, L=512, d=64, Q=128, u=2.0),
        # one position per call with the state carried by the caller: autoregressive decoding
        dict(name="ema_decode", op="ema_decode", dtype="bf16", b=64, nh=2, L=1, d=1024),
        # packed sequences of ragged length, raw probabilities, states in and out, both directions
        dict(name="ema_packed", op="ema_packed", dtype="bf16", b=6, nh=2, L=1777, d=264, nseq=5),
        # flat layout, ragged length, a chunk size below the 128 rows the kernels tile by
        dict(name="ema_step_chunk64", op="ema_step", dtype="bf16", b=8, nh=0, L=3000, d=520, Q=64, u=2.0),
        # forward only in float32 on the reference benchmark's own shape: inference over long inputs
        dict(name="ema_forward_f32", op="ema_forward", dtype="f32", b=16, nh=0, L=8192, d=1024, Q=128, u=2.0),
        # the headline training step
        dict(name="ema_step", op="ema_step", dtype="bf16", b=16, nh=2, L=4096, d=1024, Q=128, u=2.0),
        # the longest sequences, with long memory
        dict(name="ema_step_long", op="ema_step", dtype="bf16", b=4, nh=2, L=32768, d=1024, Q=256, u=4.0),
        # the per-stage launchers of both directions, called one after the other
        dict(name="ema_stages", op="ema_stages", dtype="bf16", b=4, nh=2, L=4096, d=1024, Q=256, u=2.0),
        # Mamba-2 SSD forward at a small size in float32
        dict(name="ssd_forward_small", op="ssd_forward", dtype="f32", b=1, L=512, nh=4, P=64, g=1, N=64, Q=64,
             skip=True, gate=False, bias=False, init=True, nseq=0),
        # a packed batch with everything a mixer layer uses, states per sequence returned
        dict(name="ssd_forward_packed", op="ssd_forward", dtype="bf16", b=1, L=5000, nh=24, P=64, g=2, N=128, Q=128,
             skip=True, gate=True, bias=True, init=False, nseq=6),
        # the prefill of one prompt
        dict(name="ssd_prefill", op="ssd_forward", dtype="bf16", b=1, L=4096, nh=32, P=64, g=1, N=128, Q=256,
             skip=True, gate=True, bias=True, init=True, nseq=0),
        # a training step: the forward, then the backward launchers fed by what it leaves
        dict(name="ssd_step", op="ssd_step", dtype="bf16", b=8, L=8192, nh=32, P=64, g=1, N=128, Q=256, skip=False),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["ema_step", "ema_step", "ema_forward", "ema_decode", "ema_packed", "ema_stages", "ssd_forward",
                     "ssd_forward", "ssd_step", "ssd_step"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
    if op.startswith("ema"):
        room = _MAX_EMA * 7 // 8 // (1 if dtype == "bf16" else 2) // (2 if op == "ema_stages" else 1)
        d = 8 * _log(rng, 4, 256)
        nh = rng.choice([0, 1, 2, 3, 4])
        if op == "ema_decode":
            return dict(op=op, dtype=dtype, b=_log(rng, 1, 256), nh=nh, L=_log(rng, 1, 8), d=d)
        b = _log(rng, 1, 32)
        L = _log(rng, 100, max(100, min(32768, room // (b * max(nh, 1) * d))))
        if op == "ema_packed":
            return dict(op=op, dtype=dtype, b=b, nh=nh, L=min(L, 8192), d=d, nseq=rng.randint(2, 12))
        return dict(op=op, dtype=dtype, b=b, nh=nh, L=L, d=d, Q=rng.choice([64, 128, 128, 256, 512]),
                    u=rng.choice([2.0, 4.0]))
    P, N, g = rng.choice([64, 64, 64, 128]), rng.choice([64, 128, 128]), rng.choice([1, 1, 1, 2])
    nh, Q = g * rng.randint(2, 32 // g), rng.choice([64, 128, 256, 256])
    room = _MAX_SSD // (1 if dtype == "bf16" else 8) // (P // 64)
    packed = op == "ssd_forward" and rng.random() < 0.25
    b = 1 if packed else _log(rng, 1, 8)
    L = _log(rng, 200, max(200, min(8192, room // (b * nh * P))))
    if op == "ssd_step":
        return dict(op=op, dtype=dtype, b=b, L=L, nh=nh, P=P, g=g, N=N, Q=Q, skip=rng.random() < 0.5)
    return dict(op=op, dtype=dtype, b=b, L=L, nh=nh, P=P, g=g, N=N, Q=Q, skip=rng.random() < 0.5,
                gate=rng.random() < 0.5, bias=rng.random() < 0.5, init=not packed and rng.random() < 0.5,
                nseq=rng.randint(2, 12) if packed else 0)


# ------------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------------

def _starts(b, L, nseq, gen):
    """(b, nseq - 1) sorted first positions of the second and later sequences of a packed batch."""
    order = torch.rand(b, L - 1, generator=gen, device=gen.device).argsort(dim=1)
    return (order[:, : min(nseq, L) - 1] + 1).sort(dim=1).values


def _ids(starts, L):
    ids = torch.zeros(starts.shape[0], L, dtype=torch.int32, device=starts.device)
    ids.scatter_(1, starts, 1)
    return ids.cumsum(1, dtype=torch.int32)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]

    def normal(*shape, to=torch.float32):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32).to(to)

    op, b, L = case["op"], case["b"], case["L"]
    s = {"case": case}
    if op.startswith("ema"):
        nh, d = case["nh"], case["d"]
        heads = (nh,) if nh else ()  # nh = 0: the flat (B, L, T) layout
        s["x"] = normal(b, L, *heads, d, to=dtype)
        decay = torch.nn.functional.logsigmoid(normal(b, L, *heads) + case.get("u", 2.0))
        if op in ("ema_decode", "ema_packed"):
            s["p"] = -torch.expm1(decay)
            s["init"] = normal(b, *heads, d)
        else:
            s["A"] = decay
        if op in ("ema_step", "ema_packed", "ema_stages"):
            s["dy"] = normal(b, L, *heads, d, to=dtype)
        if op == "ema_packed":
            s["dfinal"] = normal(b, *heads, d)
            s["seq_idx"] = _ids(_starts(b, L, case["nseq"], gen), L)
        for k in {"ema_step": ("x", "A"), "ema_packed": ("x", "p", "init")}.get(op, ()):
            s[k].requires_grad_()
        return s
    nh, P, g, N = case["nh"], case["P"], case["g"], case["N"]
    s["x"] = normal(b, L, nh, P, to=dtype)
    s["B"] = normal(b, L, g, N, to=dtype)
    s["C"] = normal(b, L, g, N, to=dtype)
    s["A"] = -torch.exp(torch.rand(nh, generator=gen, device="cuda") * math.log(16.0))
    s["D"] = normal(nh) if case["skip"] else None
    if op == "ssd_step":
        s["dt"] = torch.nn.functional.softplus(normal(b, L, nh) * 0.5 - 2.0)
        s["dout"] = normal(b, L, nh, P, to=dtype)
        return s
    s["z"] = normal(b, L, nh, P, to=dtype) if case["gate"] else None
    s["bias"] = normal(nh) * 0.25 - 2.0 if case["bias"] else None
    raw = normal(b, L, nh) * 0.5
    s["dt"] = raw if case["bias"] else torch.nn.functional.softplus(raw - 2.0)
    s["init"] = normal(b, nh, P, N) if case["init"] else None
    s["seq_idx"] = s["cu_seqlens"] = None
    if case["nseq"]:
        starts = _starts(b, L, case["nseq"], gen)
        s["seq_idx"] = _ids(starts, L)
        ends = torch.tensor([0, L], dtype=torch.int32, device="cuda")
        s["cu_seqlens"] = torch.cat([ends[:1], starts[0].to(torch.int32), ends[1:]])
    return s


# ------------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------------

def _ema_step(s):
    x, A = s["x"], s["A"]
    x.grad = A.grad = None
    y = ema_matmul_scan_combined(A, x, s["case"]["Q"])
    y.backward(s["dy"])
    return {"y": y.detach(), "dx": x.grad, "dA": A.grad}


def _ema_forward(s):
    with torch.no_grad():
        return {"y": ema_matmul_scan_combined(s["A"], s["x"], s["case"]["Q"])}


def _ema_decode(s):
    with torch.no_grad():
        y, state = ema_seq_scan(s["p"], s["x"], form="probability", initial_states=s["init"], return_final_states=True)
    return {"y": y, "state": state}


def _ema_packed(s):
    x, p, init = s["x"], s["p"], s["init"]
    x.grad = p.grad = init.grad = None
    y, final = ema_seq_scan(p, x, form="probability", initial_states=init, return_final_states=True,
                            seq_idx=s["seq_idx"])
    torch.autograd.backward((y, final), (s["dy"], s["dfinal"]))
    return {"y": y.detach(), "final": final.detach(), "dx": x.grad, "dp": p.grad, "dinit": init.grad}


def _ema_stages(s):
    x, dy = s["x"], s["dy"]
    cs = ema_chunk_cumsum_fwd(s["A"], s["case"]["Q"])
    states = _ema_chunk_state_fwd(x, cs)
    prev, final = _ema_state_passing_fwd(states, cs[..., -1], out_dtype=torch.float32)
    y = _ema_scan_fwd(x, cs, prev)
    ds = _ema_chunk_scan_bwd_dstates(cs, dy)
    g, ddA_chunk, _ = _ema_state_passing_bwd(prev, cs[..., -1], ds)
    dx = _ema_bwd_dx(x, cs, dy, g)
    ddA_next = _ema_chunk_state_bwd_db(x, cs, g)
    ddA_prev = _ema_chunk_scan_bwd_dC(prev, cs, dy)
    ddA = _ema_chunk_scan_bwd_ddAcs_stable(x, cs, dy)
    return {"y": y, "final": final, "dx": dx, "ddA_chunk": ddA_chunk, "ddA_next": ddA_next, "ddA_prev": ddA_prev,
            "ddA": ddA}


def _ssd_forward(s):
    c = s["case"]
    out = mamba_chunk_scan_combined_fwd(
        s["x"], s["dt"], s["A"], s["B"], s["C"], c["Q"], D=s["D"], z=s["z"], dt_bias=s["bias"],
        initial_states=s["init"], seq_idx=s["seq_idx"], cu_seqlens=s["cu_seqlens"], dt_softplus=c["bias"],
        return_final_states=True, return_varlen_states=c["nseq"] > 0)
    return dict(zip(("y", "final", "varlen"), out))


def _ssd_step(s):
    c, x, B, C, D, dout = s["case"], s["x"], s["B"], s["C"], s["D"], s["dout"]
    out, _, dt, dA, states, final = _mamba_chunk_scan_combined_fwd(x, s["dt"], s["A"], B, C, c["Q"], D=D)
    cb = _bmm_chunk_fwd(C, B, c["Q"], output_dtype=torch.float32)
    dstates, ddA_chunk, _ = _chunk_scan_state_passing_bwd(C, dA, dout, states)
    dx, ddt, dD = _chunk_scan_chunk_state_bwd_dx(x, dt, dA, B, cb, dout, dstates, D=D)
    dB, ddA_next = _chunk_state_bwd_db(x, dt, dA, dstates, B=B, ngroups=c["g"])
    dC, ddA_prev = _chunk_scan_bwd_dC(states, dA, dout, C=C, ngroups=c["g"])
    ddA = _chunk_scan_bwd_ddAcs_stable(x, dt, dA, dout, cb)
    res = {"out": out, "final": final, "dx": dx, "ddt": ddt, "dB": dB, "dC": dC, "ddA_chunk": ddA_chunk,
           "ddA_next": ddA_next, "ddA_prev": ddA_prev, "ddA": ddA}
    if dD is not None:
        res["dD"] = dD
    return res


_RUN = {"ema_step": _ema_step, "ema_forward": _ema_forward, "ema_decode": _ema_decode, "ema_packed": _ema_packed,
        "ema_stages": _ema_stages, "ssd_forward": _ssd_forward, "ssd_step": _ssd_step}


def run(state):
    return _RUN[state["case"]["op"]](state)


# ------------------------------------------------------------------------------------------------
# what a pass cannot do without, and what it may differ by
# ------------------------------------------------------------------------------------------------

def work(case):
    """Every input of a call read once, every output written once.  A training step is two calls with
    the caller's loss between them, so its backward reads the inputs again; the stage launchers are a
    call each."""
    es = 2 if case["dtype"] == "bf16" else 4
    op, b, L = case["op"], case["b"], case["L"]
    if op.startswith("ema"):
        n = b * max(case["nh"], 1)
        x, a, st = n * L * case["d"] * es, n * L * 4, n * case["d"] * 4
        el = n * L * case["d"]
        if op == "ema_forward":
            return {"bytes": 2 * x + a, "flops": 2 * el}
        if op == "ema_decode":
            return {"bytes": 2 * x + a + 2 * st, "flops": 3 * el}
        if op == "ema_step":
            return {"bytes": 5 * x + 3 * a, "flops": 8 * el}
        if op == "ema_packed":
            return {"bytes": 5 * x + 3 * a + 4 * st + 4 * b * L, "flops": 11 * el}
        chunks = -(-L // case["Q"]) * st  # one state per chunk
        return {"bytes": 10 * x + 13 * a + 12 * chunks + st, "flops": 20 * el}
    nh, P, g, N, Q = case["nh"], case["P"], case["g"], case["N"], case["Q"]
    C = -(-L // Q)
    x, bc, dt = b * L * nh * P * es, b * L * g * N * es, b * L * nh * 4
    state = b * nh * P * N
    causal, states = b * L * nh * Q * P, 2 * b * L * nh * P * N  # multiply-adds of a lower triangle, a state product
    scores = b * L * g * Q * N
    fwd = {"bytes": 2 * x + 2 * bc + dt + 4 * state, "flops": scores + causal + 2 * states}
    if op == "ssd_forward":
        fwd["bytes"] += (x if case["gate"] else 0) + (4 * state if case["init"] else 0) + 4 * state * case["nseq"]
        return fwd
    kept = 2 * dt + C * state * es  # processed dt, its cumsum and the carried states, from forward to backward
    bwd_bytes = 3 * x + 2 * bc + 2 * b * L * g * N * 4 + kept + 4 * dt
    return {"bytes": fwd["bytes"] + kept + bwd_bytes, "flops": fwd["flops"] + scores + 2 * causal + 4 * states}


# Largest relative error (2-norm) of any output against the same path in 64 bits, over all cases:
#   bfloat16   EMA 1.66e-3 (the rounding of y, dx), SSD 3.2e-3 (carried states and weighted operands rounded too)
#   float32    EMA 3.4e-7, its stages 3.2e-6 and SSD 4.8e-6 (differences of cumulative sums in the exponents)
def tolerance(case):
    ssd = case["op"].startswith("ssd")
    if case["dtype"] == "bf16":
        return {"rel": 1e-2 if ssd else 7e-3}
    return {"rel": 2e-5 if ssd else 1.2e-5 if case["op"] == "ema_stages" else 2e-6}
