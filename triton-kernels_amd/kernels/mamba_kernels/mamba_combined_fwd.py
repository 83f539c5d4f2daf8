"""The five SSD forward stages in sequence.

The reference ships the stage launchers of kernels/mamba_kernels/ without a wrapper that runs
them together (its benchmarks call mamba_ssm's mamba_chunk_scan_combined instead, e.g.
kernels/benchmarks/ema_bench.py:9); this function is that wrapper, with the argument names of
the headed entry point in kernels/ema_combined.py:100-119."""
import torch

from kernels import _lib
from kernels.mamba_kernels._shapes import NATIVE, walk_pays
from kernels.mamba_kernels.mamba_bmm import _bmm_chunk_fwd
from kernels.mamba_kernels.mamba_cumsum import _chunk_cumsum_fwd
from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd
from kernels.mamba_kernels.mamba_state_fwd import _chunk_state_fwd, chunk_state_varlen
from kernels.mamba_kernels.mamba_state_pass import _state_passing_fwd


def _chunk_state_passing_fwd(B, x, dt, dA_cumsum, initial_states=None, out_dtype=None):
    """_chunk_state_fwd followed by _state_passing_fwd (kernels/mamba_kernels/mamba_state_fwd.py:138-169,
    kernels/mamba_kernels/mamba_state_pass.py:84-115 of the reference) as one kernel that keeps the
    chunk-local states on chip, or None where that kernel does not apply (then the caller runs the two
    launchers).  Returns (states (batch, nchunks, nheads, headdim, dstate) in out_dtype: the state
    entering each chunk; final_states (batch, nheads, headdim, dstate) float32), the same values bit
    for bit as the two launchers give."""
    batch, seqlen, nheads, headdim = x.shape
    _, _, nchunks, chunk_size = dt.shape
    _, _, ngroups, dstate = B.shape
    assert nheads % ngroups == 0 and nchunks == -(-seqlen // chunk_size)
    assert B.shape == (batch, seqlen, ngroups, dstate)
    assert dt.shape == (batch, nheads, nchunks, chunk_size) and dA_cumsum.shape == dt.shape
    if initial_states is not None:
        assert initial_states.shape == (batch, nheads, headdim, dstate)
    out_dtype = torch.float32 if out_dtype is None else out_dtype
    if (chunk_size % 64 or headdim not in (64, 128) or dstate not in (64, 128)
            or x.dtype not in (torch.float32, torch.bfloat16) or out_dtype not in (torch.float32, torch.bfloat16)):
        return None
    dev = _lib.require_gpu(x, B, dt, dA_cumsum, initial_states)
    if B.dtype != x.dtype:
        B = B.to(x.dtype)
    x, xs = _lib.strided4(x)
    B, bs = _lib.strided4(B)
    dt_f = _lib.f32c(dt)
    dA_f = _lib.f32c(dA_cumsum)
    init = None if initial_states is None else _lib.f32c(initial_states)
    states = torch.empty(batch, nchunks, nheads, headdim, dstate, device=dev, dtype=out_dtype)
    final_states = torch.empty(batch, nheads, headdim, dstate, device=dev, dtype=torch.float32)
    with _lib.on_device(dev):
        _lib.check(
            _lib.lib().ssd_chunk_state_passing_fwd(*bs, *xs, _lib.dtype_code(x), dt_f.data_ptr(), dA_f.data_ptr(),
                                                   None if init is None else init.data_ptr(), states.data_ptr(),
                                                   _lib.dtype_code(states), final_states.data_ptr(), batch, seqlen,
                                                   nheads, ngroups, headdim, dstate, chunk_size,
                                                   _lib.stream_ptr(dev)),
            "ssd_chunk_state_passing_fwd")
    return states, final_states


def _carried_states(B, x, dt, dA_cumsum, initial_states, seq_idx, out_dtype):
    """(states entering each chunk, final_states) by the form that walk_pays() expects to be the faster, by the walk
    also where there is no room for the chunk-local states of the two launchers."""
    batch, seqlen, nheads, headdim = x.shape
    chunk_size, dstate = dt.shape[-1], B.shape[-1]

    def walk():
        if seq_idx is not None or out_dtype not in (torch.float32, torch.bfloat16):
            return None
        return _chunk_state_passing_fwd(B, x, dt, dA_cumsum, initial_states=initial_states, out_dtype=out_dtype)

    def two_launches():
        states = _chunk_state_fwd(B, x, dt, dA_cumsum, seq_idx=seq_idx, states_in_fp32=True)
        init = None if initial_states is None else initial_states.reshape(batch, nheads, headdim * dstate)
        states, final_states = _state_passing_fwd(states.reshape(batch, -1, nheads, headdim * dstate),
                                                  dA_cumsum[:, :, :, -1], initial_states=init, seq_idx=seq_idx,
                                                  chunk_size=chunk_size, out_dtype=out_dtype)
        return (states.reshape(batch, -1, nheads, headdim, dstate),
                final_states.reshape(batch, nheads, headdim, dstate))

    if not walk_pays(batch, nheads, seqlen, chunk_size, headdim, dstate, x.element_size()):
        try:
            return two_launches()
        except torch.cuda.OutOfMemoryError:
            pass
    return walk() or two_launches()


def _one_call(x, dt, B, C, z, chunk_size):
    """Whether the five stages run behind one entry point: one type throughout and shapes the kernels take."""
    return (x.dtype in (torch.float32, torch.bfloat16) and B.dtype == x.dtype and C.dtype == x.dtype
            and (z is None or (z.dtype == x.dtype and z.shape == x.shape))
            and dt.dtype in (torch.float32, torch.bfloat16)
            and x.shape[-1] in NATIVE and B.shape[-1] in NATIVE and chunk_size % 4 == 0 and 0 < chunk_size <= 1024)


def _combined_one_call(x, dt, A, B, C, chunk_size, D, z, dt_bias, initial_states, seq_idx, cu_seqlens, dt_softplus,
                       dt_limit, want_out_x):
    """The body of _mamba_chunk_scan_combined_fwd as one call of the library (ssd_combined_fwd): what the stage
    launchers would allocate is allocated here, and the kernels are theirs."""
    batch, seqlen, nheads, headdim = x.shape
    _, _, ngroups, dstate = B.shape
    if dt_bias is not None:
        assert dt_bias.shape == (nheads,)
    if D is not None:
        assert D.shape == (nheads, headdim) or D.shape == (nheads,)
    dev = _lib.require_gpu(x, dt, A, B, C, D, z, dt_bias, initial_states)
    ids, id_args = _lib.seq_ids(seq_idx, batch, seqlen, dev)
    x, xs = _lib.strided4(x)
    B, bs = _lib.strided4(B)
    C, cs = _lib.strided4(C)
    zs = [None, 0, 0, 0]
    if z is not None:
        z, zs = _lib.strided4(z)
    # float32 views / copies are bound to names so that they outlive the launches below
    Af, Df = _lib.f32c(A), None if D is None else _lib.f32c(D)
    bias = None if dt_bias is None else _lib.f32c(dt_bias)
    init = None if initial_states is None else _lib.f32c(initial_states)
    nchunks = -(-seqlen // chunk_size)
    walk = (seq_idx is None and chunk_size % 64 == 0
            and walk_pays(batch, nheads, seqlen, chunk_size, headdim, dstate, x.element_size()))
    f32 = dict(device=dev, dtype=torch.float32)
    dt_out = torch.empty(batch, nheads, nchunks, chunk_size, **f32)
    dA_cumsum = torch.empty(batch, nheads, nchunks, chunk_size, **f32)
    states = torch.empty(batch, nchunks, nheads, headdim, dstate, device=dev, dtype=x.dtype)
    local = None if walk else torch.empty(batch, nchunks, nheads, headdim, dstate, **f32)
    final_states = torch.empty(batch, nheads, headdim, dstate, **f32)
    cb = torch.empty(batch, nchunks, ngroups, chunk_size, chunk_size, **f32)
    out = torch.empty(batch, seqlen, nheads, headdim, device=dev, dtype=x.dtype)
    out_x = torch.empty_like(out) if z is not None and want_out_x else None
    cu = varlen = None
    if cu_seqlens is not None:
        assert cu_seqlens.shape[0] > 1 and cu_seqlens.device == dev
        cu = cu_seqlens.to(torch.int32).contiguous()
        varlen = torch.empty(cu.shape[0] - 1, nheads, headdim, dstate, device=dev, dtype=x.dtype)
    ptr = lambda t: None if t is None else t.data_ptr()
    with _lib.on_device(dev):
        _lib.check(
            _lib.lib().ssd_combined_fwd(
                *xs, _lib.dtype_code(x), dt.data_ptr(), _lib.dtype_code(dt), *dt.stride(), Af.data_ptr(), ptr(bias),
                int(bool(dt_softplus)), float(dt_limit[0]), float(min(dt_limit[1], 3.0e38)), *bs, *cs, ptr(Df),
                int(D is not None and D.dim() == 2), *zs, ptr(init), *id_args, ptr(cu),
                0 if cu is None else cu.shape[0] - 1, dt_out.data_ptr(), dA_cumsum.data_ptr(), ptr(local),
                states.data_ptr(), final_states.data_ptr(), cb.data_ptr(), out.data_ptr(), *out.stride()[:3],
                ptr(out_x), ptr(varlen), batch, seqlen, nheads, ngroups, headdim, dstate, chunk_size,
                _lib.stream_ptr(dev)),
            "ssd_combined_fwd")
    res = (out, out_x, dt_out, dA_cumsum, states, final_states)
    return res if varlen is None else res + (varlen,)


def _mamba_chunk_scan_combined_fwd(x, dt, A, B, C, chunk_size, D=None, z=None, dt_bias=None,
                                   initial_states=None, seq_idx=None, cu_seqlens=None, dt_softplus=False,
                                   dt_limit=(0.0, float("inf")), want_out_x=True):
    """Returns (out, out_x, dt_out, dA_cumsum, states, final_states), states (the state entering
    each chunk) in the dtype of C as in kernels/ema_combined.py:48-50, and as a seventh item the state
    at the end of each packed sequence when cu_seqlens is given (batch must be 1 then; the boundaries
    are the ones seq_idx marks), as kernels/ema_combined.py:56-62 of the reference does.
    want_out_x=False returns None for out_x (the result ahead of the gate), which need not be written then.
    Where walk_pays() chooses the two launchers, the chunk-local states take four bytes per state element of
    scratch; if there is no room for them, the walk runs."""
    batch, seqlen, nheads, headdim = x.shape
    _, _, ngroups, dstate = B.shape
    assert nheads % ngroups == 0
    assert B.shape == (batch, seqlen, ngroups, dstate) and C.shape == B.shape
    assert dt.shape == (batch, seqlen, nheads) and A.shape == (nheads,)
    if initial_states is not None:
        assert initial_states.shape == (batch, nheads, headdim, dstate)
    if cu_seqlens is not None:
        assert batch == 1, "passing cu_seqlens to get the varlen states is only supported if batch dimension is 1"
    if _one_call(x, dt, B, C, z, chunk_size):
        try:
            return _combined_one_call(x, dt, A, B, C, chunk_size, D, z, dt_bias, initial_states, seq_idx, cu_seqlens,
                                      dt_softplus, dt_limit, want_out_x)
        except torch.cuda.OutOfMemoryError:
            pass  # it holds everything at once (nothing is enqueued yet); the stages return their scratch one by one
    dA_cumsum, dt_out = _chunk_cumsum_fwd(dt, A, chunk_size, dt_bias=dt_bias, dt_softplus=dt_softplus,
                                          dt_limit=dt_limit)
    states, final_states = _carried_states(B, x, dt_out, dA_cumsum, initial_states, seq_idx, C.dtype)
    CB = _bmm_chunk_fwd(C, B, chunk_size, seq_idx=seq_idx, output_dtype=torch.float32)
    out, out_x = _chunk_scan_fwd(CB, x, dt_out, dA_cumsum, C, states, D=D, z=z, seq_idx=seq_idx)
    if not want_out_x:
        out_x = None
    if cu_seqlens is None:
        return out, out_x, dt_out, dA_cumsum, states, final_states
    varlen_states = chunk_state_varlen(B.squeeze(0), x.squeeze(0), dt_out.squeeze(0), dA_cumsum.squeeze(0),
                                       cu_seqlens, states.squeeze(0))
    return out, out_x, dt_out, dA_cumsum, states, final_states, varlen_states


def mamba_chunk_scan_combined_fwd(x, dt, A, B, C, chunk_size, D=None, z=None, dt_bias=None,
                                  initial_states=None, seq_idx=None, cu_seqlens=None, dt_softplus=False,
                                  dt_limit=(0.0, float("inf")), return_final_states=False,
                                  return_varlen_states=False):
    """out, then the final states and the per-sequence states as asked for, in that order
    (kernels/ema_combined.py:83-87 of the reference)."""
    if return_varlen_states:
        assert cu_seqlens is not None, "cu_seqlens must be provided if return_varlen_states is True"
    else:
        cu_seqlens = None
    out, _, _, _, _, final_states, *rest = _mamba_chunk_scan_combined_fwd(
        x, dt, A, B, C, chunk_size, D=D, z=z, dt_bias=dt_bias, initial_states=initial_states,
        seq_idx=seq_idx, cu_seqlens=cu_seqlens, dt_softplus=dt_softplus, dt_limit=dt_limit, want_out_x=False)
    res = (out,) + ((final_states,) if return_final_states else ()) + tuple(rest)
    return res if len(res) > 1 else out
