"""Calls that nothing can differentiate through skip the autograd functions: the same bits as with gradients on, and what
an autograd function refuses (forward-mode tangents, transforms) is refused as before.  A traced call runs the kernel on
every replay."""
import pytest
import torch
import torch.autograd.forward_ad as fwAD

pytestmark = pytest.mark.gpu


def _calls():
    from kernels.ema_kernels.ema_combined_fwd import ema_matmul_scan_combined
    from kernels.ema_seq import ema_seq_scan

    return {"combined": lambda a, x: ema_matmul_scan_combined(a, x, 128),
            "sequence": lambda a, x: ema_seq_scan(a, x)}


@pytest.mark.parametrize("name", ["combined", "sequence"])
@pytest.mark.parametrize("L", [1, 200])
def test_same_bits_and_no_graph(name, L, device):
    call = _calls()[name]
    x, a = torch.randn(2, L, 3, 64, device=device, requires_grad=True), -torch.rand(2, L, 3, device=device)
    y = call(a, x)
    assert y.requires_grad
    for off in (torch.no_grad, torch.inference_mode):
        with off():
            z = call(a, x)
        assert not z.requires_grad and torch.equal(z, y)


@pytest.mark.parametrize("name", ["combined", "sequence"])
def test_tangents_and_transforms_are_refused(name, device):
    call = _calls()[name]
    x, a = torch.randn(2, 5, 3, 64, device=device), -torch.rand(2, 5, 3, device=device)
    with torch.no_grad():
        with fwAD.dual_level(), pytest.raises(NotImplementedError, match="jvp"):
            call(a, fwAD.make_dual(x, torch.ones_like(x)))
        with pytest.raises(RuntimeError, match="setup_context"):
            torch.func.vmap(call)(a[None], x[None])


@pytest.mark.parametrize("name", ["combined", "sequence"])
def test_traced_calls_run_the_kernel_again(name, device):
    call = _calls()[name]
    r = lambda: (-torch.rand(2, 5, 3, device=device), torch.randn(2, 5, 3, 64, device=device))
    with torch.no_grad():
        traced = torch.jit.trace(call, r(), check_trace=False)
        for _ in range(2):
            a, x = r()
            assert torch.equal(traced(a, x), call(a, x))


@pytest.mark.parametrize("name", ["combined", "sequence"])
def test_tensors_left_over_from_a_transform_are_taken(name, device):
    """torch.func.grad leaves wrappers round tensors that outlive it; either operand, or both."""
    call, left = _calls()[name], []

    def f(*tensors):
        left.extend(tensors)
        return sum(t.sum() for t in tensors)

    a, x = -torch.rand(2, 5, 3, device=device), torch.randn(2, 5, 3, 64, device=device)
    torch.func.grad(f, argnums=(0, 1))(a, x)
    with torch.no_grad():
        y = call(a, x)
        for coef, operand in ((a, left[1]), (left[0], x), left):
            assert torch.equal(call(coef, operand), y)
