"""The forward over a few rows, the one-launch packing of coefficients and the split per-row dots, at the sizes
where they can go wrong."""
import pytest
import torch

from oracle import ema_oracle as O
from parity_util import announce, check_close

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


@pytest.mark.parametrize("form", ["log_decay", "probability"])
@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("b,nh,d", [(1, 1, 8), (3, 2, 264)])
@pytest.mark.parametrize("L", [1, 7, 8, 9, 15, 16, 17])  # the turn of eight rows and the last row count taken
def test_short_forward_vs_oracle(L, b, nh, d, dtype, form, device):
    from kernels.ema_seq import ema_seq_fwd

    announce(f"short forward L={L} b={b} nh={nh} d={d} {dtype} {form}")
    gen = torch.Generator().manual_seed(L * 31 + d)
    x = torch.randn(b, L, nh, d, generator=gen).to(dtype)
    coef = torch.rand(b, L, nh, generator=gen)
    coef = -2 * coef if form == "log_decay" else coef
    flat = lambda t: t.permute(0, 2, 1, 3).reshape(b * nh, L, d)
    cf = coef.permute(0, 2, 1).reshape(b * nh, L)
    for init in (None, torch.randn(b, nh, d, generator=gen)):
        ref = O.ema_seq_loop(flat(x.float()), cf, form, None if init is None else init.reshape(b * nh, d))
        ref = ref[0] if isinstance(ref, tuple) else ref
        y, final, prev = ema_seq_fwd(coef.to(device), x.to(device), form,
                                     initial_states=None if init is None else init.to(device))
        check_close("y", flat(y), ref, dtype)
        check_close("final", final.reshape(b * nh, d), ref[:, -1], F32)
        entering = torch.zeros(b * nh, 1, d) if init is None else init.reshape(b * nh, 1, d)
        assert torch.equal(prev.cpu(), entering)


@pytest.mark.parametrize("form", ["log_decay", "probability"])
@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
def test_short_forward_against_the_tile_kernel(dtype, form, device):
    """Rows 1 to 8 are the tile kernel's bit for bit (the first group of rows of a wave); those beyond, which it forms
    from the group's product and sum, agree to rounding."""
    from kernels.ema_seq import ema_seq_fwd

    b, L, nh, d = 2, 17, 3, 520
    gen = torch.Generator(device=device).manual_seed(2)
    x = torch.randn(b, L, nh, d, generator=gen, device=device).to(dtype)
    coef = torch.rand(b, L, nh, generator=gen, device=device)
    coef = -coef if form == "log_decay" else coef
    tile, _, _ = ema_seq_fwd(coef, x, form)
    short, _, _ = ema_seq_fwd(coef[:, :16], x[:, :16], form)
    assert torch.equal(short[:, :8], tile[:, :8])
    check_close("rows 9 to 16", short[:, 8:], tile[:, 8:16].cpu(), dtype)


@pytest.mark.parametrize("form", ["log_decay", "probability"])
@pytest.mark.parametrize("layout", ["flat", "headed", "permuted", "expanded"])
def test_packing_in_one_launch_equals_tensor_operations(layout, form, device):
    """int32 ids take the one-launch packing, int64 ids the tensor operations: same outputs, same gradients,
    for every layout of the coefficient and of the ids."""
    from kernels.ema_seq import ema_seq_scan

    announce(f"packing {layout} {form}")
    b, L, nh, d = 2, 150, 3, 16
    gen = torch.Generator().manual_seed(5)
    base = torch.rand(b, L, nh, generator=gen)
    base = -base if form == "log_decay" else base
    x = torch.randn(b, L, nh, d, generator=gen)
    if layout == "flat":
        base, x = base[..., 0].contiguous(), x[:, :, 0].contiguous()
    ids = (torch.rand(b, L, generator=gen) < 0.1).to(torch.int32).cumsum(1, dtype=torch.int32)
    dy = torch.randn(x.shape, generator=gen)
    res = []
    for id_type in (torch.int32, torch.int64):
        if layout == "permuted":
            leaf = base.permute(2, 0, 1).contiguous().to(device).requires_grad_()
            coef, seq = leaf.permute(1, 2, 0), ids.t().contiguous().to(device, id_type).t()
        elif layout == "expanded":
            leaf = base[..., :1].contiguous().to(device).requires_grad_()
            coef, seq = leaf.expand(b, L, nh), ids[:1].to(device, id_type).expand(b, L)
        else:
            leaf = base.to(device).requires_grad_()
            coef, seq = leaf, ids.to(device, id_type)
        xg = x.to(device).requires_grad_()
        y, final = ema_seq_scan(coef, xg, form=form, return_final_states=True, seq_idx=seq)
        seq = seq if layout == "expanded" else seq.zero_()  # the ids are the caller's again after the forward
        torch.autograd.backward((y, final), (dy.to(device), torch.ones_like(final)))
        res.append((y.detach(), final.detach(), xg.grad, leaf.grad))
    for name, a, c in zip(("y", "final", "dx", "dcoef"), *res):
        check_close(name, a, c.cpu(), F32)


@pytest.mark.parametrize("dtype", [F32, BF16], ids=["f32", "bf16"])
@pytest.mark.parametrize("N,L,T,Q", [(1, 64, 64, 64), (2, 130, 72, 128), (1, 500, 8, 512), (3, 2048, 1032, 1000)])
def test_row_dots_and_column_sums_split_over_workgroups(N, L, T, Q, dtype, device):
    """Few chunks: several workgroups per chunk (rows past the end, a span that does not divide the chunk)."""
    from kernels.ema_kernels.ema_state_fwd import _ema_chunk_state_fwd
    from kernels.ema_kernels_bwd.ema_chunk_scan_bwd_dc import _ema_chunk_scan_bwd_dC
    from kernels.ema_kernels_bwd.ema_chunk_state_bwd_db import _ema_chunk_state_bwd_db
    from kernels.ema_kernels_bwd.ema_scan_bwd import _ema_chunk_scan_bwd_dstates
    from parity_util import flat_case, oracle_intermediates

    announce(f"split dots N={N} L={L} T={T} Q={Q} {dtype}")
    A, X, dy = flat_case(N, L, T, 3, dtype)
    o = oracle_intermediates(A, X, dy, Q)
    d = lambda t: t.to(device)
    # the states are bfloat16 sums of the inputs held in float32: the float32 bar applies to all of these
    check_close("states", _ema_chunk_state_fwd(d(X), d(o["cs"])), O.chunk_state(X.float(), o["cs"]), F32)
    check_close("dstates", _ema_chunk_scan_bwd_dstates(d(o["cs"]), d(dy)), o["ds"], F32)
    check_close("db", _ema_chunk_state_bwd_db(d(X), d(o["cs"]), d(o["g"])), O.bwd_db(X.float(), o["cs"], o["g"]), F32)
    check_close("dc", _ema_chunk_scan_bwd_dC(d(o["prev"]), d(o["cs"]), d(dy)),
                O.bwd_dc(o["prev"], o["cs"], dy.float()), F32)


@pytest.mark.parametrize("C", [1, 7, 8, 9, 16, 17, 25])  # the turns of eight chunks of the inter-chunk recurrences
def test_state_passing_turns(C, device):
    from kernels.ema_kernels.ema_state_pass import _ema_state_passing_fwd
    from kernels.ema_kernels_bwd.ema_state_passing_bwd_dstates import _ema_state_passing_bwd

    announce(f"state passing, {C} chunks")
    gen = torch.Generator().manual_seed(C)
    N, T = 3, 260
    st, ds = torch.randn(N, C, T, generator=gen), torch.randn(N, C, T, generator=gen)
    cs_last = -torch.rand(N, C, generator=gen)
    d = lambda t: t.to(device)
    prev, final = O.state_passing(st, cs_last)
    got_prev, got_final = _ema_state_passing_fwd(d(st), d(cs_last), out_dtype=F32)
    check_close("prev", got_prev, prev, F32)
    check_close("final", got_final, final, F32)
    g, ddA = O.state_passing_bwd(prev, cs_last, ds)
    got = _ema_state_passing_bwd(d(prev), d(cs_last), d(ds))
    check_close("g", got[0], g, F32)
    check_close("ddA_chunk", got[1], ddA, F32)


@pytest.mark.parametrize("C", [1, 8, 9, 17, 31, 32, 33])  # more than 1024 workgroups: guarded loads up to 31 chunks
def test_state_passing_backward_with_the_chip_filled(C, device):
    from kernels.ema_kernels_bwd.ema_state_passing_bwd_dstates import _ema_state_passing_bwd

    announce(f"state passing backward, 1100 sequences, {C} chunks")
    gen = torch.Generator().manual_seed(C)
    N, T = 1100, 12
    prev, ds = torch.randn(N, C, T, generator=gen), torch.randn(N, C, T, generator=gen)
    cs_last = -torch.rand(N, C, generator=gen)
    g, ddA = O.state_passing_bwd(prev, cs_last, ds)
    got = _ema_state_passing_bwd(*(t.to(device) for t in (prev, cs_last, ds)))
    check_close("g", got[0], g, F32)
    check_close("ddA_chunk", got[1], ddA, F32)
