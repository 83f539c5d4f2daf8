"""The combined forward forms dt, dA, the chunk-local states and C . B in one launch where the states are passed on by a
launch of their own, but for many float32 states of hdim 128: everything it returns is, bit for bit, what the stage
launchers return one after the other."""
import pytest
import torch

from parity_util import announce
from test_gpu_ssd_packed import pack_ids

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


@pytest.mark.parametrize("dtype,dt_dtype", [(F32, F32), (BF16, F32), (BF16, BF16)])
@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("b,L,nh,g,P,N,Q", [(1, 1, 1, 1, 64, 64, 4), (2, 65, 3, 1, 64, 128, 64), (1, 257, 6, 2, 128, 64, 128),
                                            (3, 511, 5, 5, 64, 128, 256), (1, 700, 2, 1, 128, 128, 200), (1, 1500, 4, 2, 64, 64, 1024),
                                            # float32: three launches again, the last block count of one and the first of three
                                            (14, 2000, 5, 1, 128, 128, 512), (16, 2000, 4, 2, 128, 64, 512), (13, 2000, 5, 1, 128, 128, 512)])
def test_front_equals_the_stages(b, L, nh, g, P, N, Q, packed, dtype, dt_dtype, device, monkeypatch):
    from kernels.mamba_kernels import mamba_combined_fwd as M
    from kernels.mamba_kernels.mamba_bmm import _bmm_chunk_fwd
    from kernels.mamba_kernels.mamba_cumsum import _chunk_cumsum_fwd
    from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd
    from kernels.mamba_kernels.mamba_state_fwd import _chunk_state_fwd
    from kernels.mamba_kernels.mamba_state_pass import _state_passing_fwd

    announce(f"front b{b} L{L} nh{nh} g{g} P{P} N{N} Q{Q} packed {packed} {dtype} dt {dt_dtype}")
    monkeypatch.setattr(M, "walk_pays", lambda *a: False)
    gen = torch.Generator(device=device).manual_seed(L + Q)
    r = lambda *s: torch.randn(*s, generator=gen, device=device)
    x, B, C, dt = r(b, L, nh, P).to(dtype), r(b, L, g, N).to(dtype), r(b, L, g, N).to(dtype), r(b, L, nh).to(dt_dtype)
    wide = torch.zeros(b, L, nh + 3, device=device, dtype=dt_dtype)  # (dt as a slice of a projection)
    wide[..., 2:2 + nh] = dt
    dt = wide[..., 2:2 + nh]
    A, bias = -torch.rand(nh, generator=gen, device=device) - 0.1, r(nh)
    seq = (pack_ids(b, L, Q, seed=L) if L > 1 else torch.zeros(b, L, dtype=torch.int32)).to(device) if packed else None
    out, _, dt_out, dA, states, final = M._mamba_chunk_scan_combined_fwd(x, dt, A, B, C, Q, dt_bias=bias, seq_idx=seq,
                                                                        dt_softplus=True, dt_limit=(0.01, 3.0))
    dA_s, dt_s = _chunk_cumsum_fwd(dt, A, Q, dt_bias=bias, dt_softplus=True, dt_limit=(0.01, 3.0))
    assert torch.equal(dt_out, dt_s) and torch.equal(dA, dA_s)
    local = _chunk_state_fwd(B, x, dt_s, dA_s, seq_idx=seq, states_in_fp32=True)
    prev, fin = _state_passing_fwd(local.reshape(b, -1, nh, P * N), dA_s[..., -1], seq_idx=seq, chunk_size=Q, out_dtype=dtype)
    assert torch.equal(states.reshape(prev.shape), prev) and torch.equal(final.reshape(fin.shape), fin)
    cb = _bmm_chunk_fwd(C, B, Q, seq_idx=seq, output_dtype=F32)
    assert torch.equal(out, _chunk_scan_fwd(cb, x, dt_s, dA_s, C, states, seq_idx=seq)[0])
