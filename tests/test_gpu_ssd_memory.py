"""The two launchers hold the chunk-local states in float32; a call that fits without them must not fail for it."""
import contextlib

import pytest
import torch

from oracle import ssd_oracle as S
from parity_util import announce, check_close

pytestmark = pytest.mark.gpu

F32, BF16 = torch.float32, torch.bfloat16


@contextlib.contextmanager
def room_for(nbytes, device):
    """Lets torch's allocator take about nbytes more than is held now (results of an earlier call, which may lie in
    larger blocks, should be gone)."""
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(device).total_memory
    torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved(device) + nbytes) / total, device)
    try:
        yield
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, device)


def on_host(results):
    return [None if t is None else t.cpu() for t in results]


@pytest.mark.parametrize("dt_dtype", [F32, torch.float16], ids=["one-call", "stages"])  # float16 dt goes stage by stage
def test_forward_without_room_for_the_local_states(dt_dtype, device):
    from kernels.mamba_kernels._shapes import walk_pays
    from kernels.mamba_kernels.mamba_combined_fwd import _mamba_chunk_scan_combined_fwd

    b, L, nh, P, g, N, Q = 1, 16384, 32, 64, 1, 128, 64
    announce(f"ssd forward without room for {nh * L // Q * P * N * 4 >> 20} MiB, dt {dt_dtype}")
    assert not walk_pays(b, nh, L, Q, P, N, 2)
    x, dt, A, B, C, _, _ = S.make_inputs(b, L, nh, P, g, N, seed=3, dtype=BF16)
    args = [t.to(device) for t in (x, dt.to(dt_dtype), A, B, C)]
    free = on_host(_mamba_chunk_scan_combined_fwd(*args, Q))
    kept = sum(t.numel() * t.element_size() for t in free if t is not None) + L * Q * 4  # and the bmm
    with room_for(kept + (96 << 20), device):  # less than the 256 MiB of the local states
        tight = _mamba_chunk_scan_combined_fwd(*args, Q)
        torch.cuda.synchronize()
    for name, a, c in zip(("out", "out_x", "dt", "dA", "states", "final"), free, tight):
        assert (a is None and c is None) or torch.equal(a, c.cpu()), name


def test_packed_forward_without_room_for_everything_at_once(device):
    """A packed batch has no walk: the chunk-local states must be gone before the chunk scan takes its memory."""
    from kernels.mamba_kernels.mamba_combined_fwd import _mamba_chunk_scan_combined_fwd

    b, L, nh, P, g, N, Q = 1, 16384, 32, 64, 1, 128, 256
    announce("ssd packed forward without room for everything at once")
    x, dt, A, B, C, _, z = S.make_inputs(b, L, nh, P, g, N, seed=3, dtype=BF16, with_z=True)
    ids = torch.arange(L, dtype=torch.int32).div(5000, rounding_mode="floor").int()[None]
    args = [t.to(device) for t in (x, dt, A, B, C)]
    kw = dict(z=z.to(device), seq_idx=ids.to(device))
    free = on_host(_mamba_chunk_scan_combined_fwd(*args, Q, **kw))
    size = lambda t: t.numel() * t.element_size()
    kept = sum(size(t) for t in free) + L * Q * 4  # 64 + 64 MiB of out and out_x, 32 of the states, 16 of the bmm
    with room_for(kept + (24 << 20), device):      # less than the 64 MiB of the local states beside all of them
        tight = _mamba_chunk_scan_combined_fwd(*args, Q, **kw)
        torch.cuda.synchronize()
    for name, a, c in zip(("out", "out_x", "dt", "dA", "states", "final"), free, tight):
        assert torch.equal(a, c.cpu()), name


def test_backward_without_room_for_the_gradient_between_the_stages(device):
    from kernels.mamba_kernels._shapes import walk_pays
    from kernels.mamba_kernels_bwd.mamba_scan_state_passing_bwd import _chunk_scan_state_passing_bwd

    b, L, nh, P, g, N, Q = 1, 32768, 32, 64, 1, 128, 128
    announce(f"ssd backward without room for {nh * L // Q * P * N * 4 >> 20} MiB")
    assert not walk_pays(b, nh, L, Q, P, N, 2, backward=True)
    gen = torch.Generator(device=device).manual_seed(4)
    r = lambda *s: torch.randn(*s, generator=gen, device=device)
    C, dout = r(b, L, g, N).to(BF16), r(b, L, nh, P).to(BF16)
    dA = -torch.rand(b, nh, L // Q, Q, generator=gen, device=device).cumsum(-1) * 0.05
    states = r(b, L // Q, nh, P, N).to(BF16)
    free = on_host(_chunk_scan_state_passing_bwd(C, dA, dout, states))
    with room_for(states.numel() * 2 + (64 << 20), device):  # less than the 256 MiB of the float32 tensor
        tight = _chunk_scan_state_passing_bwd(C, dA, dout, states)
        torch.cuda.synchronize()
    assert torch.equal(free[0], tight[0].cpu())
    check_close("ddA", tight[1], free[1], F32)
