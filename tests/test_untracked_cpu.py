"""When a call without gradients may go past the autograd functions.  The kernel is stood in for by a copy made through
ctypes, which no tracer sees either."""
import ctypes

import pytest
import torch
import torch.autograd.forward_ad as fwAD

from kernels import _lib


@pytest.fixture
def copied(monkeypatch):
    def ema_seq_fwd(coef, x, form="log_decay", initial_states=None, **_):
        y = torch.empty_like(x)
        ctypes.memmove(y.data_ptr(), x.data_ptr(), x.numel() * x.element_size())
        return y, torch.empty(x.shape[0], x.shape[-1]), torch.empty(x.shape[0], 1, x.shape[-1])

    monkeypatch.setattr("kernels.ema_seq.ema_seq_fwd", ema_seq_fwd)


def _calls():
    from kernels.ema_kernels.ema_combined_fwd import ema_matmul_scan_combined
    from kernels.ema_seq import ema_seq_scan

    return {"combined": lambda a, x: ema_matmul_scan_combined(a, x, 128), "sequence": lambda a, x: ema_seq_scan(a, x)}


@pytest.mark.parametrize("off", [torch.no_grad, torch.inference_mode])
@pytest.mark.parametrize("name", ["combined", "sequence"])
def test_traced_calls_run_the_kernel_again(name, off, copied):
    call = _calls()[name]
    a = torch.zeros(2, 5)
    with off():
        traced = torch.jit.trace(call, (a, torch.ones(2, 5, 8)), check_trace=False)
        for v in (10.0, 20.0):
            x = torch.full((2, 5, 8), v)
            assert torch.equal(traced(a, x), x)


@pytest.mark.parametrize("off", [torch.no_grad, torch.inference_mode])
@pytest.mark.parametrize("name", ["combined", "sequence"])
def test_tensors_left_over_from_a_transform_are_taken(name, off, copied):
    """torch.func.grad leaves a wrapper round a tensor that outlives it, which has no memory of its own."""
    left = []

    def f(x):
        left.append(x)
        return (x * x).sum()

    a, x = torch.zeros(2, 5), torch.arange(80.0).view(2, 5, 8)
    torch.func.grad(f)(x)
    with off():
        assert torch.equal(_calls()[name](a, left[0]), x)


def test_untracked():
    seen = []

    def look(x):
        seen.append(_lib.untracked())
        return x + 1

    x = torch.ones(3)
    look(x)
    with torch.inference_mode():
        look(x)
    with torch.no_grad():
        look(x)
        with fwAD.dual_level():
            look(fwAD.make_dual(x, torch.ones(3)))
        torch.func.vmap(look)(x)
        torch.jit.trace(look, x, check_trace=False)
        look(x)
    assert seen == [False, True, True, False, False, False, True]
