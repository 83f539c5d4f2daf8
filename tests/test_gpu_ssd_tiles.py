"""The chunk scan in one tile per chunk (chunks of 64 and 128 rows) and the choice between the state walk and
the two launchers, at the sizes where they can go wrong."""
import pytest
import torch

from kernels.mamba_kernels._shapes import walk_pays
from oracle import ssd_oracle as S
from parity_util import announce, check_close

F32, BF16 = torch.float32, torch.bfloat16


def one_tile_batch(Q, L, nh, P, dtype):
    """The batch at which the kernels of one tile per chunk take over: more than 128 chunks in float32; in bfloat16 384
    single heads of 128 features or pairs of heads of 64, more than 512 pairs with chunks of 64 rows."""
    from_ = 129 if dtype == F32 else 513 if Q == 64 and P == 64 else 384
    return -(-from_ // (-(-L // Q) * (nh // 2 if P == 64 and dtype == BF16 else nh)))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["decay", "rise", "mixed"])
@pytest.mark.parametrize("nh,g,P,dtype", [(4, 1, 64, BF16), (6, 3, 64, BF16), (2, 1, 128, BF16), (3, 1, 64, F32),
                                          (2, 2, 128, F32)])
@pytest.mark.parametrize("Q,L", [(128, 257), (128, 128), (128, 33), (64, 190), (64, 64), (64, 1)])
def test_chunk_scan_one_tile_vs_oracle(Q, L, nh, g, P, dtype, kind, device):
    """L one row past a chunk, exact and shorter than a 32-row block; dA falling, rising and both (the weights
    then take the exact form everywhere)."""
    from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd

    announce(f"chunk scan Q={Q} L={L} nh={nh} g={g} P={P} {dtype} {kind}")
    N = 64 if P == 128 else 128
    b = one_tile_batch(Q, L, nh, P, dtype)
    gen = torch.Generator().manual_seed(Q + L + nh)
    r = lambda *s: torch.randn(*s, generator=gen)
    x, C, z = r(b, L, nh, P).to(dtype), r(b, L, g, N).to(dtype), r(b, L, nh, P).to(dtype)
    dt = torch.rand(b, L, nh, generator=gen) * 0.5
    A = -torch.rand(nh, generator=gen) - 0.1
    if kind == "rise":
        A = -A
    elif kind == "mixed":
        dt = dt - 0.25
    dA, dto = S.chunk_cumsum(dt, A, Q)
    nc = -(-L // Q)
    cb = r(b, nc, g, Q, Q) * 0.3
    states = r(b, nc, nh, P, N).to(dtype)
    D = r(nh)
    for zz in (None, z):
        ref, ref_x = S.chunk_scan(cb, x, dto, dA, C, states, D=D, z=zz, round_to=dtype)
        got, got_x = _chunk_scan_fwd(*(t.to(device) for t in (cb, x, dto, dA, C, states)), D=D.to(device),
                                     z=None if zz is None else zz.to(device))
        check_close("out", got, ref, dtype, regrouped=True)
        if zz is not None:
            check_close("out_x", got_x, ref_x, dtype, regrouped=True)


@pytest.mark.gpu
@pytest.mark.parametrize("nchunks", [1, 4, 5, 8, 9, 17])
def test_state_passing_turns(nchunks, device):
    """Chunk counts around one and two turns of the prefetch, plain and packed, both directions."""
    from kernels.mamba_kernels.mamba_state_pass import _state_passing_fwd
    from kernels.mamba_kernels_bwd.mamba_state_passing_bwd_dstates import _state_passing_bwd

    announce(f"state passing, {nchunks} chunks")
    b, nh, dim, Q = 2, 3, 200, 4
    L = nchunks * Q - 1
    gen = torch.Generator().manual_seed(nchunks)
    st, dout = torch.randn(b, nchunks, nh, dim, generator=gen), torch.randn(b, nchunks, nh, dim, generator=gen)
    da = -torch.rand(b, nh, nchunks, generator=gen)
    ids = (torch.rand(b, L, generator=gen) < 0.15).to(torch.int32).cumsum(1, dtype=torch.int32)
    d = lambda t: t.to(device)
    for seq in (None, ids):
        kw = {} if seq is None else dict(seq_idx=seq, chunk_size=Q)
        dkw = {} if seq is None else dict(seq_idx=d(seq), chunk_size=Q)
        ref, rfin = S.state_passing(st, da, **kw)
        got, fin = _state_passing_fwd(d(st), d(da), out_dtype=F32, **dkw)
        check_close("states", got, ref, F32)
        check_close("final", fin, rfin, F32)
        rd, rdda, _ = S.state_passing_bwd(ref, da, dout, **kw)
        gd, gdda, _ = _state_passing_bwd(d(ref), d(da), d(dout), dstates_dtype=F32, **dkw)
        check_close("dstates", gd, rd, F32)
        check_close("ddA", gdda, rdda, F32)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])  # bfloat16: eight elements per thread backward
@pytest.mark.parametrize("nchunks", [4, 5, 8, 9])
def test_state_passing_with_the_chip_filled(nchunks, dtype, device):
    """More workgroups than the form with two turns of loads under way takes, plain and packed, both directions."""
    from kernels.mamba_kernels.mamba_state_pass import _state_passing_fwd
    from kernels.mamba_kernels_bwd.mamba_state_passing_bwd_dstates import _state_passing_bwd

    announce(f"state passing, 1040 heads, {nchunks} chunks {dtype}")
    b, nh, dim, Q = 2, 520, 16, 4
    L = nchunks * Q - 1
    gen = torch.Generator().manual_seed(nchunks)
    st, dout = (torch.randn(b, nchunks, nh, dim, generator=gen).to(dtype) for _ in range(2))
    da = -torch.rand(b, nh, nchunks, generator=gen)
    ids = (torch.rand(b, L, generator=gen) < 0.15).to(torch.int32).cumsum(1, dtype=torch.int32)
    d = lambda t: t.to(device)
    for seq in (None, ids):
        kw = {} if seq is None else dict(seq_idx=seq, chunk_size=Q)
        dkw = {} if seq is None else dict(seq_idx=d(seq), chunk_size=Q)
        ref, rfin = S.state_passing(st.float(), da, **kw)
        got, fin = _state_passing_fwd(d(st), d(da), out_dtype=dtype, **dkw)
        check_close("states", got, ref, dtype)
        check_close("final", fin, rfin, F32)
        carried = ref.to(dtype)
        rd, rdda, _ = S.state_passing_bwd(carried.float(), da, dout.float(), **kw)
        gd, gdda, _ = _state_passing_bwd(d(carried), d(da), d(dout), dstates_dtype=dtype, **dkw)
        check_close("dstates", gd, rd, dtype)
        check_close("ddA", gdda, rdda, F32)


def test_walk_choice():
    """Few heads or long chunks: the two launchers; a head per compute unit: the walk."""
    assert not walk_pays(1, 32, 4096, 256, 64, 128, 2)
    assert not walk_pays(1, 4, 512, 64, 64, 64, 4)
    assert walk_pays(8, 32, 8192, 256, 64, 128, 2) and walk_pays(8, 32, 8192, 256, 64, 128, 2, backward=True)
    assert walk_pays(4, 32, 512, 64, 64, 128, 2)
    for heads in (8, 64, 128):  # up to a workgroup per compute unit more heads never turn the walk away
        assert walk_pays(1, heads, 8192, 256, 64, 128, 2) <= walk_pays(1, 2 * heads, 8192, 256, 64, 128, 2)
    # 256 heads fill the chip; a few more make the walk take twice as long, many more make up for it
    assert walk_pays(1, 256, 8192, 256, 64, 128, 2) and not walk_pays(1, 264, 8192, 256, 64, 128, 2)
    assert walk_pays(1, 512, 8192, 256, 64, 128, 2)


@pytest.mark.parametrize("heads,L,Q,P,N,itemsize,backward,walk,pair", [  # measured on an MI355X, us
    (192, 500, 512, 64, 128, 2, False, 12.9, 21.1),  # one chunk: nothing to spread, eight stages in a row either way
    (16, 500, 512, 64, 64, 2, False, 9.0, 13.3),
    (192, 1024, 512, 64, 128, 2, False, 20.2, 25.4),
    (192, 500, 512, 128, 64, 2, False, 15.0, 20.2),
    (128, 500, 512, 64, 128, 2, True, 14.8, 19.6),
    (64, 8192, 64, 128, 128, 2, False, 393, 267),
    (128, 8192, 64, 64, 128, 4, False, 579, 431),
    (32, 8192, 256, 64, 128, 2, False, 126, 31),
    (192, 8192, 256, 64, 128, 2, False, 124, 147),
    (264, 8192, 256, 64, 128, 2, False, 235, 201),
    (512, 8192, 256, 64, 128, 2, False, 256, 358),
    (768, 8192, 256, 64, 128, 2, False, 371, 538),
    (128, 8192, 256, 64, 128, 2, True, 151, 117),
    (192, 8192, 256, 64, 128, 2, True, 154, 167),
    (512, 2048, 64, 64, 64, 4, False, 174, 220),
    (32, 2048, 256, 128, 128, 4, False, 207, 39),
])
def test_walk_choice_against_measured_times(heads, L, Q, P, N, itemsize, backward, walk, pair):
    """What the rule takes is never more than 12 % (the error of its estimates) behind the other form."""
    taken = walk if walk_pays(1, heads, L, Q, P, N, itemsize, backward=backward) else pair
    assert taken <= 1.12 * min(walk, pair)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("P,N", [(64, 64), (128, 128), (64, 128)])
def test_varlen_states_at_stage_edges(P, N, dtype, device):
    """Sequences that end one row into a chunk, on and around the 64-row stages, and an empty one."""
    from kernels.ema_chunk_state import chunk_state_varlen

    announce(f"varlen stages P={P} N={N} {dtype}")
    Q, nh, g = 256, 4, 2
    cu = torch.tensor([0, 1, 64, 129, 129, 257, 320, 511, 577], dtype=torch.int32)
    L = int(cu[-1])
    gen = torch.Generator().manual_seed(9)
    r = lambda *s: torch.randn(*s, generator=gen)
    x, B = r(L, nh, P).to(dtype), r(L, g, N).to(dtype)
    dA, dt = S.chunk_cumsum(torch.rand(1, L, nh, generator=gen) * 0.5, -torch.rand(nh, generator=gen), Q)
    prev = r(-(-L // Q), nh, P, N).to(dtype)
    ref = S.chunk_state_varlen(B, x, dt[0], dA[0], cu, prev, dtype)
    got = chunk_state_varlen(*(t.to(device) for t in (B, x, dt[0], dA[0], cu, prev)))
    check_close("varlen states", got, ref, dtype, regrouped=True)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("Q,length", [(64, 7), (256, 7), (64, 70), (256, 70)])  # float32 takes the matrix units in the last
def test_varlen_states_of_many_sequences(Q, length, dtype, device):
    from kernels.ema_chunk_state import chunk_state_varlen

    announce(f"varlen states of 260 sequences of about {length}, Q={Q} {dtype}")
    nseq, nh, g, P, N = 260, 4, 2, 64, 64
    gen = torch.Generator().manual_seed(length)
    cu = torch.randint(1, 2 * length, (nseq + 1,), generator=gen).cumsum(0).to(torch.int32)
    cu -= cu[0].clone()
    cu[-1] = max(int(cu[-1]), nseq * length)
    L = int(cu[-1])
    r = lambda *s: torch.randn(*s, generator=gen)
    x, B = r(L, nh, P).to(dtype), r(L, g, N).to(dtype)
    dA, dt = S.chunk_cumsum(torch.rand(1, L, nh, generator=gen) * 0.5, -torch.rand(nh, generator=gen), Q)
    prev = r(-(-L // Q), nh, P, N).to(dtype)
    ref = S.chunk_state_varlen(B, x, dt[0], dA[0], cu, prev, dtype)
    got = chunk_state_varlen(*(t.to(device) for t in (B, x, dt[0], dA[0], cu, prev)))
    check_close("varlen states", got, ref, dtype, regrouped=True)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["decay", "rise", "mixed"])
@pytest.mark.parametrize("nh,g,N", [(4, 1, 128), (6, 3, 64)])
@pytest.mark.parametrize("Q,L", [(128, 257), (128, 128), (128, 33), (64, 190), (64, 64), (64, 1)])
def test_dx_one_tile_vs_oracle(Q, L, nh, g, N, kind, device):
    """Pairs of bfloat16 heads: dx, ddt and dD (all its slots) at the same edges, the ddt of rows past the end zero."""
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_chunk_state_bwd_dx import _chunk_scan_chunk_state_bwd_dx

    announce(f"dx Q={Q} L={L} nh={nh} g={g} N={N} {kind}")
    P, dtype = 64, BF16
    b = one_tile_batch(Q, L, nh, P, dtype)
    gen = torch.Generator().manual_seed(Q + L + nh)
    r = lambda *s: torch.randn(*s, generator=gen)
    x, dout, B = r(b, L, nh, P).to(dtype), r(b, L, nh, P).to(dtype), r(b, L, g, N).to(dtype)
    dt = torch.rand(b, L, nh, generator=gen) * 0.5
    A = -torch.rand(nh, generator=gen) - 0.1
    if kind == "rise":
        A = -A
    elif kind == "mixed":
        dt = dt - 0.25
    dA, dto = S.chunk_cumsum(dt, A, Q)
    nc = -(-L // Q)
    cb = r(b, nc, g, Q, Q) * 0.3
    if L % Q:  # what lies past the sequence must not be looked at
        cb[:, -1, :, L % Q:, :] = float("nan")
    ref_cb = torch.nan_to_num(cb)
    ds = r(b, nc, nh, P, N).to(dtype)
    d = lambda t: t.to(device)
    for D in (None, r(nh), r(nh, P)):
        ref = S.chunk_scan_chunk_state_bwd_dx(x, dto, dA, B, ref_cb, dout, ds, D=D, round_to=dtype)
        got = _chunk_scan_chunk_state_bwd_dx(d(x), d(dto), d(dA), d(B), d(cb), d(dout), d(ds),
                                             D=None if D is None else d(D))
        check_close("dx", got[0], ref[0], dtype, regrouped=True)
        check_close("ddt", got[1], ref[1], dtype, loose=True)
        if D is not None:
            check_close("dD", got[2], ref[2], F32)


@pytest.mark.gpu
@pytest.mark.parametrize("b,nh", [(1, 4), (128, 8)])  # single heads, and 1024 pairs of heads
def test_chunk_scan_of_rows_far_apart(b, nh, device):
    """x, z and C whose positions lie megabytes apart (position-major tensors of a large batch): strides only change
    addresses, so the result is that of contiguous copies bit for bit."""
    from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd

    announce(f"chunk scan, rows far apart, b{b} nh{nh}")
    L, P, N, Q, far = 300, 64, 128, 256, 1 << 21
    gen = torch.Generator(device=device).manual_seed(3)
    r = lambda *s: torch.randn(*s, generator=gen, device=device)
    x, z, C = r(b, L, nh, P).to(BF16), r(b, L, nh, P).to(BF16), r(b, L, 1, N).to(BF16)
    buf = torch.empty(L, far, device=device, dtype=BF16)
    size = b * nh * P
    views = []
    for i, t in enumerate((x, z, C)):
        v = buf[:, i * size: i * size + t[:, 0].numel()].view(L, b, *t.shape[2:]).transpose(0, 1)
        views.append(v.copy_(t))
        assert v.stride(1) == far
    dA = (-torch.rand(b, nh, 2, Q, generator=gen, device=device) * 0.2).cumsum(-1)
    cb, states, dt = r(b, 2, 1, Q, Q), r(b, 2, nh, P, N).to(BF16), torch.rand(b, nh, 2, Q, generator=gen, device=device)
    D = r(nh)
    want = _chunk_scan_fwd(cb, x, dt, dA, C, states, D=D, z=z)
    got = _chunk_scan_fwd(cb, views[0], dt, dA, views[2], states, D=D, z=views[1])
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
