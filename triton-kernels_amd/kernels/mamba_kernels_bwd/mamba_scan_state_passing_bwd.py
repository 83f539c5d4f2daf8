"""SSD backward: the gradient of the chunk scan with respect to the carried states and the reverse
inter-chunk recurrence, run back to back.

The reference ships the two launchers (_chunk_scan_bwd_dstates,
kernels/mamba_kernels_bwd/mamba_scan_bwd.py:91-116, and _state_passing_bwd,
kernels/mamba_kernels_bwd/mamba_state_passing_bwd_dstates.py:116-172) without a combined backward
that would call them; a caller that does so runs this function in their place."""
import torch

from kernels import _lib
from kernels.mamba_kernels._shapes import walk_pays
from kernels.mamba_kernels_bwd.mamba_scan_bwd import _chunk_scan_bwd_dstates
from kernels.mamba_kernels_bwd.mamba_state_passing_bwd_dstates import _state_passing_bwd


def _prepare(C, dA_cumsum, dout, states, dfinal_states, has_initial_states, out_dtype):
    """Checked operands and outputs of the two forms below, or None where neither applies."""
    batch, seqlen, nheads, headdim = dout.shape
    _, _, nchunks, chunk_size = dA_cumsum.shape
    _, _, ngroups, dstate = C.shape
    if (headdim != 64 or dstate != 128 or chunk_size % 64 or chunk_size < 128 or dout.dtype != torch.bfloat16
            or states.dtype != torch.bfloat16 or out_dtype not in (torch.float32, torch.bfloat16)):
        return None
    dev = _lib.require_gpu(C, dA_cumsum, dout, states, dfinal_states)
    if C.dtype != dout.dtype:
        C = C.to(dout.dtype)
    dout, ds = _lib.strided4(dout)
    C, cs = _lib.strided4(C)
    if min(ds[1:]) < 0 or min(cs[1:]) < 0:
        return None
    # dense views / copies are handed back so that they outlive the launches
    dA_f = _lib.f32c(dA_cumsum)
    st = states.contiguous()
    dfin = None if dfinal_states is None else _lib.f32c(dfinal_states)
    dstates = torch.empty(batch, nchunks, nheads, headdim, dstate, device=dev, dtype=out_dtype)
    ddA = torch.empty(batch, nheads, nchunks, device=dev, dtype=torch.float32)
    dinit = (torch.empty(batch, nheads, headdim, dstate, device=dev, dtype=torch.float32)
             if has_initial_states else None)
    dims = (batch, seqlen, nheads, ngroups, headdim, dstate, chunk_size)
    return dev, (C, cs), (dout, ds), dA_f, st, dfin, dstates, ddA, dinit, dims


def _fused(C, dA_cumsum, dout, states, dfinal_states, has_initial_states, out_dtype):
    """One kernel for both stages (the chunk's gradient stays in the accumulators), or None where
    that kernel does not apply."""
    prep = _prepare(C, dA_cumsum, dout, states, dfinal_states, has_initial_states, out_dtype)
    if prep is None:
        return None
    dev, (C, cs), (dout, ds), dA_f, st, dfin, dstates, ddA, dinit, dims = prep
    lib = _lib.lib()
    nbytes = lib.ssd_chunk_scan_state_passing_bwd_workspace_bytes(dims[0], dstates.shape[1], dims[2])
    ws = torch.empty(max(nbytes, 16), device=dev, dtype=torch.uint8)
    with _lib.on_device(dev):
        _lib.check(
            lib.ssd_chunk_scan_state_passing_bwd(*cs, *ds, _lib.dtype_code(dout), dA_f.data_ptr(), st.data_ptr(),
                                                 _lib.dtype_code(st), None if dfin is None else dfin.data_ptr(),
                                                 dstates.data_ptr(), _lib.dtype_code(dstates), ddA.data_ptr(),
                                                 None if dinit is None else dinit.data_ptr(), ws.data_ptr(), nbytes,
                                                 *dims, _lib.stream_ptr(dev)),
            "ssd_chunk_scan_state_passing_bwd")
    return dstates, ddA, dinit


def _two_launches(C, dA_cumsum, dout, states, dfinal_states, has_initial_states, out_dtype):
    """The same results from the two stages' own kernels with a float32 tensor the size of states between them
    (dstates bit for bit), or None where _fused does not apply either.  The operands are checked and converted once:
    27 us of host time a call where the two stages' own wrappers take 34."""
    prep = _prepare(C, dA_cumsum, dout, states, dfinal_states, has_initial_states, out_dtype)
    if prep is None:
        return None
    dev, (C, cs), (dout, ds), dA_f, st, dfin, dstates, ddA, dinit, dims = prep
    lib = _lib.lib()
    batch, seqlen, nheads, _, headdim, dstate, Q = dims
    nchunks, dim = dstates.shape[1], headdim * dstate
    dprev = torch.empty(dstates.shape, device=dev, dtype=torch.float32)
    nbytes = lib.ssd_state_passing_bwd_workspace_bytes(batch, nchunks, nheads, dim)
    ws = torch.empty(max(nbytes, 16), device=dev, dtype=torch.uint8)
    no_ids = (None, 0, 0)
    with _lib.on_device(dev):
        stream = _lib.stream_ptr(dev)
        _lib.check(
            lib.ssd_chunk_scan_bwd_dstates(*cs, *ds, _lib.dtype_code(dout), dA_f.data_ptr(), dprev.data_ptr(),
                                           _lib.EMA_F32, *dims, *no_ids, stream),
            "ssd_chunk_scan_bwd_dstates")
        _lib.check(
            lib.ssd_state_passing_bwd(st.data_ptr(), _lib.dtype_code(st), dA_f.data_ptr() + 4 * (Q - 1),
                                      nheads * nchunks * Q, nchunks * Q, Q, dprev.data_ptr(), _lib.EMA_F32,
                                      None if dfin is None else dfin.data_ptr(), dstates.data_ptr(),
                                      _lib.dtype_code(dstates), ddA.data_ptr(),
                                      None if dinit is None else dinit.data_ptr(), ws.data_ptr(), nbytes, batch,
                                      nchunks, nheads, dim, *no_ids, seqlen, Q, stream),
            "ssd_state_passing_bwd")
    return dstates, ddA, dinit


def _chunk_scan_state_passing_bwd(C, dA_cumsum, dout, states, dfinal_states=None, seq_idx=None,
                                  has_initial_states=None, dstates_dtype=None):
    """C (batch, seqlen, ngroups, dstate), dA_cumsum (batch, nheads, nchunks, chunk_size), dout
    (batch, seqlen, nheads, headdim), states (batch, nchunks, nheads, headdim, dstate): the state
    entering each chunk, dfinal_states (batch, nheads, headdim, dstate) or None.  Returns what
    _state_passing_bwd returns, shaped like states: (dstates, the gradient of each chunk's local
    state; ddA_chunk_cumsum (batch, nheads, nchunks); dinitial_states or None).  The gradient with
    respect to the entering states that _chunk_scan_bwd_dstates would return travels between the
    two stages in float32 and is not returned."""
    batch, seqlen, nheads, headdim = dout.shape
    _, _, nchunks, chunk_size = dA_cumsum.shape
    _, _, ngroups, dstate = C.shape
    assert nheads % ngroups == 0 and nchunks == -(-seqlen // chunk_size)
    assert C.shape == (batch, seqlen, ngroups, dstate)
    assert dA_cumsum.shape == (batch, nheads, nchunks, chunk_size)
    assert states.shape == (batch, nchunks, nheads, headdim, dstate)
    if dfinal_states is not None:
        assert dfinal_states.shape == (batch, nheads, headdim, dstate)
    out_dtype = dstates_dtype if dstates_dtype is not None else states.dtype
    if seq_idx is None:
        walk = walk_pays(batch, nheads, seqlen, chunk_size, headdim, dstate, dout.element_size(), backward=True)
        args = (C, dA_cumsum, dout, states, dfinal_states, has_initial_states, out_dtype)
        both = None
        if not walk:
            try:
                both = _two_launches(*args)
            except torch.cuda.OutOfMemoryError:  # no room for the float32 tensor between the two: the walk needs none
                walk = True
        if walk:
            both = _fused(*args)
        if both is not None:
            return both
    dim = headdim * dstate
    dprev = _chunk_scan_bwd_dstates(C, dA_cumsum, dout, seq_idx=seq_idx, dtype=torch.float32)
    dfin = None if dfinal_states is None else dfinal_states.reshape(batch, nheads, dim)
    dstates, ddA, dinit = _state_passing_bwd(states.reshape(batch, nchunks, nheads, dim), dA_cumsum[..., -1],
                                             dprev.reshape(batch, nchunks, nheads, dim), dfinal_states=dfin,
                                             seq_idx=seq_idx, has_initial_states=has_initial_states,
                                             dstates_dtype=out_dtype, chunk_size=chunk_size)
    dstates = dstates.reshape(batch, nchunks, nheads, headdim, dstate)
    return dstates, ddA, None if dinit is None else dinit.reshape(batch, nheads, headdim, dstate)
