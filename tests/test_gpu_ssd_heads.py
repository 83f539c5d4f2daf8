"""The kernels that walk the heads of a group (bfloat16, hdim 64, chunks of 256 rows), at the edges of their strips of 16
rows, with each way of dealing the heads to workgroups (one head each, a share of one set, shares that run over several
sets) and each form of the decay: one that falls (its factors apart), one that falls steeply inside a strip, one that
rises.  The oracle looks at the first, a middle and the last element of the batch."""
import pytest
import torch

from oracle import ssd_oracle as S
from parity_util import announce, check_close
from test_gpu_ssd_packed import pack_ids

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16
P, Q = 64, 256

# (batch, seqlen, nheads, ngroups, dstate): 72 heads of all (batch, chunk) pairs; 276, two to a workgroup; 688 in shares of
# four; 1200 and 3210 dealt evenly; groups that do not divide evenly
DEALS = [(2, 527, 12, 1, 128), (23, 289, 6, 2, 128), (43, 512, 8, 1, 64), (100, 700, 4, 1, 128), (107, 513, 10, 1, 64),
         (3, 271, 11, 1, 128)]


def _decay(kind, b, L, nh, seed):
    gen = torch.Generator().manual_seed(seed)
    dt = torch.rand(b, L, nh, generator=gen) * 0.5
    A = -torch.rand(nh, generator=gen) * 4 - 0.1
    if kind == "steep":
        A = A * 30
    elif kind == "rising":
        A = -A * 0.05
    elif kind == "mixed":  # up and down, and one head that falls throughout
        dt[..., 1:] -= 0.25
    return S.chunk_cumsum(dt, A, Q)


def _inputs(b, L, nh, g, N, kind, seed):
    gen = torch.Generator().manual_seed(seed)
    r = lambda *s: torch.randn(*s, generator=gen)
    nc = -(-L // Q)
    dA, dt = _decay(kind, b, L, nh, seed)
    cb = r(b, nc, g, Q, Q) * 0.3
    if L % Q:  # what lies past the sequence must not be looked at
        cb[:, -1, :, L % Q:, :] = float("nan")
        dA[:, :, -1, L % Q:] = dA[:, :, -1, L % Q - 1:L % Q]
    x, y = r(b, L, nh, P).to(BF16), r(b, L, nh, P).to(BF16)
    return x, y, r(b, L, g, N).to(BF16), dt, dA, cb, r(b, nc, nh, P, N).to(BF16), r(nh)


def _some(b):
    rows = sorted({0, b // 2, b - 1})
    return rows, lambda t: None if t is None else t[rows]


def _check_scan(case, kind, skip, gate, packed, device):
    from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd

    b, L, nh, g, N = case
    announce(f"scan by heads {case} {kind} skip {skip} gate {gate} packed {packed}")
    x, z, C, dt, dA, cb, states, D = _inputs(b, L, nh, g, N, kind, seed=L + nh)
    z, D = z if gate else None, D if skip else None
    seq = pack_ids(b, L, Q, seed=L) if packed else None
    d = lambda t: None if t is None else t.to(device)
    out, out_x = _chunk_scan_fwd(d(cb), d(x), d(dt), d(dA), d(C), d(states), D=d(D), z=d(z), seq_idx=d(seq))
    rows, pick = _some(b)
    ref, ref_x = S.chunk_scan(torch.nan_to_num(pick(cb)), pick(x), pick(dt), pick(dA), pick(C), pick(states), D=D, z=pick(z),
                              round_to=BF16, seq_idx=pick(seq))
    check_close("out", out[rows], ref, BF16, regrouped=True)
    if gate:
        check_close("out_x", out_x[rows], ref_x, BF16, regrouped=True)


@pytest.mark.parametrize("skip,gate,packed", [(False, False, False), (True, False, True), (True, True, False), (False, True, True)])
@pytest.mark.parametrize("case", DEALS)
def test_scan_deals_and_options(case, skip, gate, packed, device):
    _check_scan(case, "falling", skip, gate, packed, device)


@pytest.mark.parametrize("gate", [False, True])
@pytest.mark.parametrize("kind", ["falling", "steep", "rising", "mixed"])
@pytest.mark.parametrize("L", [257, 271, 272, 273, 289, 511])
def test_scan_strip_edges(L, kind, gate, device):
    _check_scan((26, L, 6, 1, 128), kind, True, gate, False, device)


def _check_dx(case, kind, skip, packed, device):
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_chunk_state_bwd_dx import _chunk_scan_chunk_state_bwd_dx

    b, L, nh, g, N = case
    announce(f"dx by heads {case} {kind} skip {skip} packed {packed}")
    x, dout, B, dt, dA, cb, ds, D = _inputs(b, L, nh, g, N, kind, seed=L + nh)
    D = D if skip else None
    seq = pack_ids(b, L, Q, seed=L) if packed else None
    d = lambda t: None if t is None else t.to(device)
    dx, ddt, dD = _chunk_scan_chunk_state_bwd_dx(d(x), d(dt), d(dA), d(B), d(cb), d(dout), d(ds), D=d(D), seq_idx=d(seq))
    rows, pick = _some(b)
    ref = S.chunk_scan_chunk_state_bwd_dx(pick(x), pick(dt), pick(dA), pick(B), torch.nan_to_num(pick(cb)), pick(dout), pick(ds),
                                          D=D, round_to=BF16, seq_idx=pick(seq))
    check_close("dx", dx[rows], ref[0], BF16, regrouped=True)
    check_close("ddt", ddt[rows], ref[1], BF16, loose=True)
    if skip:
        check_close("dD", dD, (dout.float() * x.float()).sum((0, 1, 3)), F32)


@pytest.mark.parametrize("skip,packed", [(False, False), (True, True)])
@pytest.mark.parametrize("case", DEALS)
def test_dx_deals_and_options(case, skip, packed, device):
    _check_dx(case, "falling", skip, packed, device)


@pytest.mark.parametrize("kind", ["falling", "steep", "rising", "mixed"])
@pytest.mark.parametrize("L", [1, 15, 17, 255, 272, 289])
def test_dx_strip_edges(L, kind, device):
    _check_dx((2, L, 36, 1, 128), kind, True, False, device)


def _check_ddA(case, kind, device):
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_bwd_da import _chunk_scan_bwd_ddAcs_stable

    b, L, nh, g, N = case
    announce(f"ddA by heads {case} {kind}")
    x, dout, _, dt, dA, cb, _, _ = _inputs(b, L, nh, g, N, kind, seed=L + nh)
    d = lambda t: t.to(device)
    got = _chunk_scan_bwd_ddAcs_stable(d(x), d(dt), d(dA), d(dout), d(cb))
    rows, pick = _some(b)
    ref = S.chunk_scan_bwd_ddAcs_stable(pick(x), pick(dt), pick(dA), pick(dout), torch.nan_to_num(pick(cb)))
    # (float32 throughout: products of bfloat16 values are exact in it)
    check_close("ddA_cumsum (causal term)", got[rows], ref, F32)


# (beyond 256 heads the ddA walk takes more than 768 where they divide well: 1743 a set each, 816 in four shares a set, 2700
# dealt evenly; the general kernel 1600 and 1664)
@pytest.mark.parametrize("case", DEALS + [(100, 257, 8, 1, 128), (52, 300, 16, 1, 128), (135, 270, 10, 1, 128),
                                          (83, 700, 7, 1, 64), (51, 250, 16, 1, 128)])
def test_ddA_deals(case, device):
    _check_ddA(case, "falling", device)


@pytest.mark.parametrize("kind", ["falling", "steep", "rising", "mixed"])
@pytest.mark.parametrize("L", [1, 15, 17, 255, 272, 289])
def test_ddA_strip_edges(L, kind, device):
    _check_ddA((2, L, 4, 1, 128), kind, device)


def _unaligned(t):
    """The same values where the walks do not take them: the general kernels run."""
    return torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)


def _ddA_float64(x, dt, dA, dout, cb):
    b, L, nh, p = x.shape
    chunks = lambda t: t.double().reshape(b, L // Q, Q, nh, p).permute(0, 1, 3, 2, 4).contiguous()
    dA, dt = dA.double().permute(0, 2, 1, 3), dt.double().permute(0, 2, 1, 3)
    w = chunks(dout) @ chunks(x).transpose(-1, -2).contiguous() * cb.double().repeat_interleave(nh // cb.shape[2], 2)
    w = (w * torch.exp((dA[..., :, None] - dA[..., None, :]).clamp(max=0)) * dt[..., None, :]).tril(-1)
    delta = w.sum(-2) - w.sum(-1)
    return (delta.cumsum(-1) - delta).permute(0, 2, 1, 3)


@pytest.mark.parametrize("rate,shift", [(1.0, -2.0), (1.6, 2.0), (2.5, 2.0), (16.0, -2.0), (16.0, 0.0), (16.0, 2.0)])
def test_ddA_is_as_exact_as_the_general_kernel(rate, shift, device):
    """float32 results against float64, with A in [-rate, -1] and dt about softplus(shift).  Each kernel rounds a weight a
    few times and adds up the same weights, so their errors agree but for the luck of a seed, 0.8 to 1.27 in the norm: over
    the 12 seeds 0.76 to 1.04, and 0.2 to 1.06 in the largest.  Exponents of up to 40 of both signs in place of one small one,
    which __expf rounds by 6e-8 of the exponent, show as 1.3 in the norm and 2 and more in the largest."""
    from kernels.mamba_kernels.mamba_bmm import _bmm_chunk_fwd
    from kernels.mamba_kernels.mamba_cumsum import _chunk_cumsum_fwd
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_bwd_da import _chunk_scan_bwd_ddAcs_stable

    announce(f"ddA error rate {rate} shift {shift}")
    b, L, nh, N = 3, 2048, 8, 128
    norm, most = [], []
    for seed in range(100, 112):
        gen = torch.Generator(device=device).manual_seed(seed)
        r = lambda *s: torch.randn(*s, generator=gen, device=device)
        x, dout, B, C = (r(b, L, n, p).to(BF16) for n, p in ((nh, P), (nh, P), (1, N), (1, N)))
        A = -torch.exp(torch.rand(nh, generator=gen, device=device) * torch.tensor(rate).log().item())
        dA, dt = _chunk_cumsum_fwd(torch.nn.functional.softplus(r(b, L, nh) * 0.5 + shift), A, Q)
        cb = _bmm_chunk_fwd(C, B, Q, output_dtype=F32)
        ref = _ddA_float64(x, dt, dA, dout, cb)
        err = [_chunk_scan_bwd_ddAcs_stable(x, t, dA, dout, cb).double() - ref for t in (dt, _unaligned(dt))]
        norm.append([(e.norm() / ref.norm()).item() for e in err])
        most.append([(e.abs().max() / ref.abs().max()).item() for e in err])
    walk, general = (sum(c) / len(c) for c in zip(*norm))
    walk_most, general_most = (sum(c) / len(c) for c in zip(*most))
    print(f"  norm {general:.2e} / {walk:.2e}, largest {general_most:.2e} / {walk_most:.2e}", flush=True)
    assert walk <= 1.15 * general and walk_most <= 1.5 * general_most


# ---- forms of the decay that the split has to keep its hands off

WALKS = {"scan": (26, 512, 6, 1, 128), "dx": (6, 512, 6, 1, 128), "ddA": (2, 512, 6, 1, 128)}


def _run(name, ops, dt, dA, device, ref=None):
    """The stage's results on the device, or the oracle's for the batch elements that it looks at."""
    x, y, BC, cb, states = ops
    if ref is None:
        from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd
        from kernels.mamba_kernels_bwd.mamba_chunk_scan_bwd_da import _chunk_scan_bwd_ddAcs_stable
        from kernels.mamba_kernels_bwd.mamba_chunk_scan_chunk_state_bwd_dx import _chunk_scan_chunk_state_bwd_dx

        x, y, BC, cb, states, dt, dA = (t.to(device) for t in (x, y, BC, cb, states, dt, dA))
        if name == "scan":
            return [("out", _chunk_scan_fwd(cb, x, dt, dA, BC, states, z=y)[0], BF16)]
        if name == "dx":
            dx, ddt, _ = _chunk_scan_chunk_state_bwd_dx(x, dt, dA, BC, cb, y, states)
            return [("dx", dx, BF16), ("ddt", ddt, BF16)]
        return [("ddA", _chunk_scan_bwd_ddAcs_stable(x, dt, dA, y, cb), F32)]
    x, y, BC, cb, states, dt, dA = (t[ref] for t in (x, y, BC, torch.nan_to_num(cb), states, dt, dA))
    if name == "scan":
        return [S.chunk_scan(cb, x, dt, dA, BC, states, z=y, round_to=BF16)[0]]
    if name == "dx":
        return list(S.chunk_scan_chunk_state_bwd_dx(x, dt, dA, BC, cb, y, states, round_to=BF16)[:2])
    return [S.chunk_scan_bwd_ddAcs_stable(x, dt, dA, y, cb)]


def _compare(name, got, ref, rows, pick=lambda t: t):
    for (what, g, dtype), r in zip(got, ref):
        check_close(f"{name} {what}", pick(g[rows]), pick(r), dtype, regrouped=dtype == BF16, loose=what == "ddt")


@pytest.mark.parametrize("drop", [30.0, 1000.0])
@pytest.mark.parametrize("name", list(WALKS))
def test_small_rises_are_clamped(name, drop, device):
    """dA falls once and then rises by 9e-7 of itself per position, 2.3e-4 of itself in a chunk: every weight behind
    the fall is that of exp(0)."""
    case = WALKS[name]
    announce(f"{name} with small rises behind {drop}")
    x, y, BC, dt, dA, cb, states, _ = _inputs(*case, "falling", seed=5)
    dA = (-drop * (1 - 9e-7 * torch.arange(Q))).expand(dA.shape).clone()
    dA[..., 0] = 0
    ops = (x, y, BC, cb, states)
    rows, _ = _some(case[0])
    _compare(name, _run(name, ops, dt, dA, device), _run(name, ops, dt, dA, device, ref=rows), rows)


@pytest.mark.parametrize("rate", [0.1, 4.0, 30.0])
@pytest.mark.parametrize("name", list(WALKS))
def test_steps_of_zero(name, rate, device):
    """A tenth of the steps is 0: the library's own sums rise by their rounding between some of them."""
    from kernels.mamba_kernels.mamba_cumsum import _chunk_cumsum_fwd

    case = WALKS[name]
    b, L, nh, _, _ = case
    announce(f"{name} with steps of zero, rate {rate}")
    x, y, BC, _, _, cb, states, _ = _inputs(*case, "falling", seed=6)
    gen = torch.Generator().manual_seed(7)
    dt = torch.rand(b, L, nh, generator=gen) * (torch.rand(b, L, nh, generator=gen) > 0.1)
    dA, dt = (t.cpu() for t in _chunk_cumsum_fwd(dt.to(device), torch.full((nh,), -rate, device=device), Q))
    assert (dA[..., 1:] > dA[..., :-1]).any()
    ops = (x, y, BC, cb, states)
    rows, _ = _some(b)
    _compare(name, _run(name, ops, dt, dA, device), _run(name, ops, dt, dA, device, ref=rows), rows)


@pytest.mark.parametrize("L", [257, 263, 271, 272, 290, 400, 511])
def test_ddA_looks_at_nothing_past_the_sequence(L, device):
    """dt, dA and cb past the sequence are NaN or infinite; a last position with an infinite dt, which no weight uses.
    The general kernel does the same."""
    case = (2, L, 6, 1, 128)
    announce(f"ddA with anything past position {L}")
    x, y, BC, dt, dA, cb, states, _ = _inputs(*case, "falling", seed=L)
    ops, rows, n = (x, y, BC, cb, states), [0, 1], L % Q
    ref = _run("ddA", ops, dt, dA, device, ref=rows)
    for junk in (float("nan"), float("inf"), -float("inf"), 1e30):
        cb[:, -1, :, n:, :] = junk
        cb[:, -1, :, :, n:] = junk
        dA[:, :, -1, n:] = junk
        dt[:, :, -1, n:] = junk
        for last in (0.5, float("inf")):
            dt[:, :, -1, n - 1] = last
            for steps in (dt.to(device), _unaligned(dt.to(device))):
                got = _run("ddA", ops, steps, dA, device)
                _compare("ddA", got, ref, rows, lambda t: t[:, :, :-1])
                _compare("ddA", got, ref, rows, lambda t: t[:, :, -1, :n])
                assert torch.isfinite(got[0][1]).all()


@pytest.mark.parametrize("at", [4, 100, 252])
@pytest.mark.parametrize("name", list(WALKS))
def test_infinite_decay_and_infinite_steps(name, at, device):
    """dA of -inf from some position on lets nothing through from before it, and positions behind it see each other
    whole; an infinite dt reaches the rows behind it only."""
    case = WALKS[name]
    announce(f"{name} with dA = -inf or dt = inf from position {at}")
    x, y, BC, dt, dA, cb, states, _ = _inputs(*case, "falling", seed=at)
    ops, rows = (x, y, BC, cb, states), _some(case[0])[0]
    cut, far = dA.clone(), dA.clone()
    cut[:, ::2, :, at:], far[:, ::2, :, at:] = -float("inf"), -3e4
    _compare(name, _run(name, ops, dt, cut, device), _run(name, ops, dt, far, device, ref=rows), rows)
    inf, zero = dt.clone(), dt.clone()
    inf[:, 1::2, :, at], zero[:, 1::2, :, at] = float("inf"), 0
    got, ref = _run(name, ops, inf, dA, device), _run(name, ops, zero, dA, device, ref=rows)
    if name == "dx":  # dt scales the position's own row
        keep = torch.arange(case[1]) % Q != at
        pick = lambda t: t[:, keep] if t.shape[1] == case[1] else t
    else:
        before = lambda t, dim: t.unflatten(dim, (-1, Q)).narrow(dim + 1, 0, at)
        pick = lambda t: before(t, 1) if name == "scan" else t[..., :at]
    _compare(name, got, ref, rows, pick)


# two shares of a set of sixteen heads, four; dealt evenly, the set changes inside the loop; a set each (ddA: the ones behind)
@pytest.mark.parametrize("kind", ["steep", "rising", "mixed"])
@pytest.mark.parametrize("case", [(52, 300, 16, 1, 128), (107, 513, 10, 1, 64), (100, 257, 8, 1, 128),
                                  (51, 250, 16, 1, 128), (135, 270, 10, 1, 128), (83, 700, 7, 1, 64)])
def test_every_decay_in_workgroups_of_several_heads(case, kind, device):
    _check_scan(case, kind, True, False, False, device)
    _check_scan(case, kind, False, True, False, device)
    _check_dx(case, kind, True, False, device)
    _check_ddA(case, kind, device)


# ---- rows

def _rows_apart(t, stride):
    """The same values, `stride` elements from row to row."""
    b, L, nh, p = t.shape
    v = torch.empty((b * L - 1) * stride + nh * p, dtype=t.dtype, device=t.device).as_strided(t.shape, (L * stride, stride, p, 1))
    return v.copy_(t)


# rows of a wider projection; the longest rows that the walks take (2^23 - 8 elements) and the first that they do not
@pytest.mark.parametrize("stride", [66 * 64 + 1024, 2 ** 23 - 8, 2 ** 23])
@pytest.mark.parametrize("L", [256, 250])
def test_rows_apart(L, stride, device):
    from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_bwd_da import _chunk_scan_bwd_ddAcs_stable
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_chunk_state_bwd_dx import _chunk_scan_chunk_state_bwd_dx

    announce(f"rows {stride} elements apart, L {L}")
    x, y, BC, dt, dA, cb, states, D = _inputs(1, L, 66, 1, 128, "falling", seed=L)
    cb = torch.nan_to_num(cb)  # (the general dx looks at it past the sequence)
    ref, ref_x = S.chunk_scan(cb, x, dt, dA, BC, states, D=D, z=y, round_to=BF16)
    ref_dx, ref_ddt, _ = S.chunk_scan_chunk_state_bwd_dx(x, dt, dA, BC, cb, y, states, D=D, round_to=BF16)
    ref_ddA = S.chunk_scan_bwd_ddAcs_stable(x, dt, dA, y, cb)
    x, y, BC, dt, dA, cb, states, D = (t.to(device) for t in (x, y, BC, dt, dA, cb, states, D))
    apart = lambda t: _rows_apart(t, stride)
    xa, ya, Ba, dxa = apart(x), apart(y), apart(BC), apart(torch.zeros_like(x))
    out, out_x = _chunk_scan_fwd(cb, xa, dt, dA, Ba, states, D=D, z=ya)
    dx, ddt, dD = _chunk_scan_chunk_state_bwd_dx(xa, dt, dA, Ba, cb, ya, states, D=D, dx=dxa)
    ddA = _chunk_scan_bwd_ddAcs_stable(xa, dt, dA, ya, cb)
    assert dx.data_ptr() == dxa.data_ptr()
    for name, got, want in (("out", out, ref), ("out_x", out_x, ref_x), ("dx", dx, ref_dx)):
        check_close(name, got, want, BF16, regrouped=True)
    check_close("ddt", ddt, ref_ddt, BF16, loose=True)
    check_close("ddA", ddA, ref_ddA, F32)
    if stride < 2 ** 23:  # the same kernels as for dense rows
        same = _chunk_scan_chunk_state_bwd_dx(x, dt, dA, BC, cb, y, states, D=D)
        for got, want in ((out, _chunk_scan_fwd(cb, x, dt, dA, BC, states, D=D, z=y)[0]), (dx, same[0]), (ddt, same[1]),
                          (dD, same[2]), (ddA, _chunk_scan_bwd_ddAcs_stable(x, dt, dA, y, cb))):
            assert torch.equal(got, want)


# batch * chunks * heads up to which the header promises the same bits for states of either type
@pytest.mark.parametrize("name,b,gate", [("scan", 32, False), ("scan", 8, True), ("dx", 8, False)])
def test_states_of_either_type_give_the_same_bits(name, b, gate, device):
    from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_chunk_state_bwd_dx import _chunk_scan_chunk_state_bwd_dx

    announce(f"{name} of {8 * b} heads, gate {gate}, states of either type")
    x, y, BC, dt, dA, cb, states, D = (t.to(device) for t in _inputs(b, 300, 4, 1, 128, "falling", seed=b))
    cb = torch.nan_to_num(cb)
    if name == "scan":
        got = [_chunk_scan_fwd(cb, x, dt, dA, BC, s, D=D, z=y if gate else None) for s in (states, states.float())]
    else:
        got = [_chunk_scan_chunk_state_bwd_dx(x, dt, dA, BC, cb, y, s, D=D) for s in (states, states.float())]
    for a, c in zip(*got):
        assert a is None and c is None or torch.equal(a, c)
