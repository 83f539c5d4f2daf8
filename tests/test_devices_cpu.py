"""Every tensor whose address reaches a kernel must be on the GPU of the others and of the shape the kernel assumes.
Fake tensors stand for those on the GPU, so that the refusals (which come ahead of any use of an address) can be
exercised without one."""
import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

F32, BF16 = torch.float32, torch.bfloat16
b, L, nh, P, g, N, Q = 1, 128, 2, 64, 1, 128, 64
nc = L // Q


def ssd_combined(o):
    from kernels.mamba_kernels.mamba_combined_fwd import _mamba_chunk_scan_combined_fwd
    _mamba_chunk_scan_combined_fwd(o("x", b, L, nh, P, dtype=BF16), o("dt", b, L, nh), o("A", nh),
                                   o("B", b, L, g, N, dtype=BF16), o("C", b, L, g, N, dtype=BF16), Q, D=o("D", nh),
                                   z=o("z", b, L, nh, P, dtype=BF16), dt_bias=o("dt_bias", nh),
                                   initial_states=o("initial_states", b, nh, P, N))


def ssd_cumsum(o):
    from kernels.mamba_kernels.mamba_cumsum import _chunk_cumsum_fwd
    _chunk_cumsum_fwd(o("dt", b, L, nh), o("A", nh), Q, dt_bias=o("dt_bias", nh))


def ssd_scan(o):
    from kernels.mamba_kernels.mamba_scan_fwd import _chunk_scan_fwd
    _chunk_scan_fwd(o("cb", b, nc, g, Q, Q), o("x", b, L, nh, P), o("dt", b, nh, nc, Q), o("dA", b, nh, nc, Q),
                    o("C", b, L, g, N), o("states", b, nc, nh, P, N), D=o("D", nh), z=o("z", b, L, nh, P))


def ssd_state_passing(o):
    from kernels.mamba_kernels.mamba_state_pass import _state_passing_fwd
    _state_passing_fwd(o("states", b, nc, nh, P * N), o("dA", b, nh, nc), initial_states=o("initial_states", b, nh, P * N))


def ssd_walk(o):
    from kernels.mamba_kernels.mamba_combined_fwd import _chunk_state_passing_fwd
    _chunk_state_passing_fwd(o("B", b, L, g, N), o("x", b, L, nh, P), o("dt", b, nh, nc, Q), o("dA", b, nh, nc, Q),
                             initial_states=o("initial_states", b, nh, P, N))


def ssd_dx(o):
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_chunk_state_bwd_dx import _chunk_scan_chunk_state_bwd_dx
    _chunk_scan_chunk_state_bwd_dx(o("x", b, L, nh, P), o("dt", b, nh, nc, Q), o("dA", b, nh, nc, Q), o("B", b, L, g, N),
                                   o("cb", b, nc, g, Q, Q), o("dout", b, L, nh, P), o("dstates", b, nc, nh, P, N),
                                   D=o("D", nh), dx=o("dx", b, L, nh, P))


def ssd_db(o):
    from kernels.mamba_kernels_bwd.mamba_chunk_state_bwd_db import _chunk_state_bwd_db
    _chunk_state_bwd_db(o("x", b, L, nh, P), o("dt", b, nh, nc, Q), o("dA", b, nh, nc, Q), o("dstates", b, nc, nh, P, N),
                        B=o("B", b, L, g, N), ngroups=g)


def ssd_dc(o):
    from kernels.mamba_kernels_bwd.mamba_chunk_scan_bwd_dc import _chunk_scan_bwd_dC
    _chunk_scan_bwd_dC(o("states", b, nc, nh, P, N), o("dA", b, nh, nc, Q), o("dout", b, L, nh, P), C=o("C", b, L, g, N),
                       ngroups=g)


def ssd_state_passing_bwd(o):
    from kernels.mamba_kernels_bwd.mamba_state_passing_bwd_dstates import _state_passing_bwd
    _state_passing_bwd(o("states", b, nc, nh, P * N), o("dA", b, nh, nc), o("dout", b, nc, nh, P * N),
                       dfinal_states=o("dfinal_states", b, nh, P * N))


def ssd_walk_bwd(o):
    from kernels.mamba_kernels_bwd.mamba_scan_state_passing_bwd import _chunk_scan_state_passing_bwd
    _chunk_scan_state_passing_bwd(o("C", b, L, g, N, dtype=BF16), o("dA", b, nh, 1, L), o("dout", b, L, nh, P, dtype=BF16),
                                  o("states", b, 1, nh, P, N, dtype=BF16), dfinal_states=o("dfinal_states", b, nh, P, N))


def ema_seq(o):
    from kernels.ema_seq import ema_seq_fwd
    ema_seq_fwd(o("coef", b, L, nh), o("x", b, L, nh, P), initial_states=o("initial_states", b, nh, P))


def ema_seq_backward(o):
    from kernels.ema_seq import ema_seq_bwd
    ema_seq_bwd(o("dy", b, L, nh, P), o("x", b, L, nh, P), o("coef", b, L, nh), o("prev128", b * nh, 1, P),
                dfinal_states=o("dfinal_states", b, nh, P))


def ema_backward(o):
    from kernels.ema_kernels_bwd.ema_combined_bwd import _ema_chunk_scan_combined_bwd
    _ema_chunk_scan_combined_bwd(o("dout", b, L, nh, P), o("x", b, L, nh, P), o("A", b, L, nh), L,
                                 prev128=o("prev128", b * nh, 1, P))


CALLS = {
    ssd_combined: ("D", "z", "dt_bias", "initial_states", "B", "C", "A", "dt"), ssd_cumsum: ("dt_bias", "A"),
    ssd_scan: ("D", "z", "states", "cb"), ssd_state_passing: ("initial_states", "dA"), ssd_walk: ("initial_states", "B"),
    ssd_dx: ("D", "dx", "cb", "dstates"), ssd_db: ("B", "dstates"), ssd_dc: ("C", "dout"),
    ssd_state_passing_bwd: ("dfinal_states", "dout"), ssd_walk_bwd: ("dfinal_states", "dA", "states"),
    ema_seq: ("initial_states", "coef"), ema_seq_backward: ("dfinal_states", "coef", "prev128"),
    ema_backward: ("prev128", "A"),
}


@pytest.mark.parametrize("call,name", [(c, n) for c, names in CALLS.items() for n in names],
                         ids=lambda v: v if isinstance(v, str) else v.__name__)
def test_a_tensor_left_on_the_host_is_refused(call, name):
    seen = []

    def operand(which, *shape, dtype=F32):
        seen.append(which)
        return torch.empty(*shape, dtype=dtype, device="cpu" if which == name else "cuda:0")

    with FakeTensorMode(), pytest.raises(AssertionError, match="same device"):
        call(operand)
    assert name in seen


@pytest.mark.parametrize("wrong,shape", [("C", (1, 256, g, N)), ("C", (2, 192, g, N)), ("dA", (1, nh, 2, 128)),
                                         ("dA", (1, nh, 1, 256)), ("dA", (2, nh, 3, 128))])
def test_reverse_walk_refuses_operands_of_other_shapes(wrong, shape):
    """The kernels index C and dA_cumsum by dout's batch, length and heads."""
    from kernels.mamba_kernels_bwd.mamba_scan_state_passing_bwd import _chunk_scan_state_passing_bwd

    shapes = dict(C=(2, 256, g, N), dA=(2, nh, 2, 128))
    shapes[wrong] = shape
    with FakeTensorMode(), pytest.raises(AssertionError):
        o = lambda *s, dtype=BF16: torch.empty(*s, dtype=dtype, device="cuda:0")
        _chunk_scan_state_passing_bwd(o(*shapes["C"]), o(*shapes["dA"], dtype=F32), o(2, 256, nh, P),
                                      o(2, shapes["dA"][2], nh, P, N))


@pytest.mark.parametrize("wrong,shape", [("B", (1, 256, g, N)), ("B", (2, 192, g, N)), ("dt", (2, nh, 2, 64)),
                                         ("dt", (1, nh, 4, 64)), ("init", (1, nh, P, N))])
def test_state_walk_refuses_operands_of_other_shapes(wrong, shape):
    from kernels.mamba_kernels.mamba_combined_fwd import _chunk_state_passing_fwd

    shapes = dict(B=(2, 256, g, N), dt=(2, nh, 4, 64), init=(2, nh, P, N))
    shapes[wrong] = shape
    with FakeTensorMode(), pytest.raises(AssertionError):
        o = lambda *s: torch.empty(*s, device="cuda:0")
        _chunk_state_passing_fwd(o(*shapes["B"]), o(2, 256, nh, P), o(*shapes["dt"]), o(2, nh, 4, 64),
                                 initial_states=o(*shapes["init"]))
