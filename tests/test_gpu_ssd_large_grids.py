"""The kernels that only take over where there are many workgroups (pairs of heads in the 256-row chunk scan, one tile
per chunk in the chunk scan and dx), with the options a mixer layer brings: packed ids, a ragged last chunk, D in both
shapes, the gate, float32 and bfloat16 states, groups, and operands that are slices of a wider projection.  The batch is as large as the
rules ask for; the oracle looks at its first, middle and last element."""
import pytest
import torch

from oracle import ssd_oracle as S
from parity_util import announce, check_close
from test_gpu_ssd_packed import pack_ids
from test_gpu_ssd_tiles import one_tile_batch

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


def _slice_of_wider(t, left=64, right=32):
    """The same values as a slice along the flattened (heads, features) axis of a wider tensor."""
    b, L = t.shape[:2]
    inner = t[0, 0].numel()
    wide = torch.full((b, L, left + inner + right), float("nan"), dtype=t.dtype, device=t.device)
    v = wide[..., left:left + inner].unflatten(-1, t.shape[2:])
    v.copy_(t)
    assert not v.is_contiguous() and v.stride(2) == t.shape[3]
    return v


def _operands(b, L, nh, P, g, N, Q, dtype, states_dtype, seed):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen)
    nc = -(-L // Q)
    x, z, BC = r(b, L, nh, P).to(dtype), r(b, L, nh, P).to(dtype), r(b, L, g, N).to(dtype)
    dA, dt = S.chunk_cumsum(torch.rand(b, L, nh, generator=gen) * 0.2, -torch.rand(nh, generator=gen) * 0.1, Q)
    cb = r(b, nc, g, Q, Q) * 0.3
    states = r(b, nc, nh, P, N).to(states_dtype)
    return x, z, BC, dt, dA, cb, states


def _check_scan(b, L, nh, P, g, N, Q, dtype, states_dtype, D, gate, packed, views, device):
    from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd

    x, z, C, dt, dA, cb, states = _operands(b, L, nh, P, g, N, Q, dtype, states_dtype, seed=L + Q + N + nh)
    z = z if gate else None
    seq = pack_ids(b, L, Q, seed=L) if packed else None
    d = lambda t: None if t is None else t.to(device)
    xd, zd, Cd = d(x), d(z), d(C)
    if views:
        xd, Cd, zd = _slice_of_wider(xd), _slice_of_wider(Cd), None if z is None else _slice_of_wider(zd, 128, 8)
    out, out_x = _chunk_scan_fwd(d(cb), xd, d(dt), d(dA), Cd, d(states), D=d(D), z=zd, seq_idx=d(seq))
    assert torch.isfinite(out.float()).all()
    some = sorted({0, b // 2, b - 1})  # (the last row of a packed batch is a single sequence)
    pick = lambda t: None if t is None else t[some]
    ref, ref_x = S.chunk_scan(pick(cb), pick(x), pick(dt), pick(dA), pick(C), pick(states), D=D, z=pick(z),
                              round_to=None if dtype == F32 else dtype, seq_idx=pick(seq))
    if packed:  # the ids matter
        plain = S.chunk_scan(pick(cb), pick(x), pick(dt), pick(dA), pick(C), pick(states), D=D, z=pick(z))[0]
        assert (plain - ref).abs().max() > 1
    check_close("out", out[some], ref, dtype, regrouped=True)
    if gate:
        check_close("out_x", out_x[some], ref_x, dtype, regrouped=True)
    else:
        assert out_x is None


@pytest.mark.parametrize("D", [None, "head", "feature"])
@pytest.mark.parametrize("gate,packed,views", [(False, False, False), (True, False, True), (True, True, False),
                                               (False, True, True)])
@pytest.mark.parametrize("N,Q,L,nh,g,states_dtype", [(128, 256, 300, 4, 1, BF16), (64, 256, 512, 4, 2, F32),
                                                     (128, 512, 700, 4, 2, F32), (64, 512, 1024, 2, 1, BF16)])
def test_pairs_of_heads_in_the_256_row_scan(N, Q, L, nh, g, states_dtype, gate, packed, views, D, device):
    P = 64
    tiles = -(-L // Q) * (Q // 256)
    b = -(-512 // (tiles * (nh // 2)))  # pairs of heads from 512 workgroups on
    announce(f"paired scan b{b} L{L} nh{nh} g{g} N{N} Q{Q} states {states_dtype} D {D} gate {gate} packed {packed} "
             f"views {views}")
    gen = torch.Generator().manual_seed(1)
    Dt = None if D is None else torch.randn(nh, generator=gen) if D == "head" else torch.randn(nh, P, generator=gen)
    _check_scan(b, L, nh, P, g, N, Q, BF16, states_dtype, Dt, gate, packed, views, device)


@pytest.mark.parametrize("D", [None, "feature"])
@pytest.mark.parametrize("gate,packed,views", [(True, True, False), (False, True, True), (True, False, True)])
@pytest.mark.parametrize("nh,g,P,N,dtype,states_dtype", [(4, 1, 64, 128, BF16, F32), (4, 2, 64, 64, BF16, BF16),
                                                         (2, 1, 128, 128, BF16, F32), (3, 1, 64, 128, F32, F32),
                                                         (2, 2, 128, 64, F32, F32)])
@pytest.mark.parametrize("Q,L", [(128, 257), (128, 161), (64, 190)])
def test_one_tile_scan_options(Q, L, nh, g, P, N, dtype, states_dtype, gate, packed, views, D, device):
    b = one_tile_batch(Q, L, nh, P, dtype)
    announce(f"one-tile scan b{b} L{L} nh{nh} g{g} P{P} N{N} Q{Q} {dtype} states {states_dtype} D {D} gate {gate} "
             f"packed {packed} views {views}")
    Dt = None if D is None else torch.randn(nh, P, generator=torch.Generator().manual_seed(1))
    _check_scan(b, L, nh, P, g, N, Q, dtype, states_dtype, Dt, gate, packed, views, device)


@pytest.mark.parametrize("D", [None, "head", "feature"])
@pytest.mark.parametrize("packed,views", [(True, False), (True, True), (False, True)])
@pytest.mark.parametrize("nh,g,N,states_dtype", [(4, 1, 128, F32), (4, 2, 64, BF16)])
@pytest.mark.parametrize("Q,L", [(128, 257), (128, 161), (64, 190)])
def test_one_tile_dx_options(Q, L, nh, g, N, states_dtype, packed, views, D, device):
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_chunk_state_bwd_dx import _chunk_scan_chunk_state_bwd_dx

    P = 64
    b = one_tile_batch(Q, L, nh, P, BF16)
    announce(f"one-tile dx b{b} L{L} nh{nh} g{g} N{N} Q{Q} dstates {states_dtype} D {D} packed {packed} views {views}")
    x, dout, B, dt, dA, cb, ds = _operands(b, L, nh, P, g, N, Q, BF16, states_dtype, seed=L + Q + N)
    gen = torch.Generator().manual_seed(1)
    Dt = None if D is None else torch.randn(nh, generator=gen) if D == "head" else torch.randn(nh, P, generator=gen)
    seq = pack_ids(b, L, Q, seed=L) if packed else None
    d = lambda t: None if t is None else t.to(device)
    xd, dd, Bd = d(x), d(dout), d(B)
    if views:
        xd, dd, Bd = _slice_of_wider(xd), _slice_of_wider(dd, 128, 8), _slice_of_wider(Bd)
    dx, ddt, dD = _chunk_scan_chunk_state_bwd_dx(xd, d(dt), d(dA), Bd, d(cb), dd, d(ds), D=d(Dt), seq_idx=d(seq))
    assert torch.isfinite(dx.float()).all() and torch.isfinite(ddt).all()
    some = sorted({0, b // 2, b - 1})
    pick = lambda t: None if t is None else t[some]
    ref = S.chunk_scan_chunk_state_bwd_dx(pick(x), pick(dt), pick(dA), pick(B), pick(cb), pick(dout), pick(ds), D=Dt,
                                          round_to=BF16, seq_idx=pick(seq))
    if packed:
        plain = S.chunk_scan_chunk_state_bwd_dx(pick(x), pick(dt), pick(dA), pick(B), pick(cb), pick(dout), pick(ds), D=Dt)
        assert (plain[0] - ref[0]).abs().max() > 0.3
    check_close("dx", dx[some], ref[0], BF16, regrouped=True)
    check_close("ddt", ddt[some], ref[1], BF16, loose=True)
    if D is not None:
        prod = dout.float() * x.float()
        check_close("dD", dD, prod.sum((0, 1)) if D == "feature" else prod.sum((0, 1, 3)), F32)
