"""Head sizes and state sizes outside what the SSD kernels take natively.

The kernels are built for headdim and dstate in {64, 128} (the Mamba-2 shapes).  The reference's
own tests and benchmarks also call its Mamba launchers on the EMA problem written as an SSD
one, with dstate = 1 and head sizes from 8 to 512 (kernels/tests/ema/test_ema_state_fwd.py:108-141,
kernels/benchmarks/ema/scan_fwd/scan_fwd_bench.py:20-68).  Those shapes are brought to a native
one around the same kernels:

  * a head wider than 128 is cut into sub-heads of 64 features: the recurrence treats the
    features of a head independently and only shares dt, A and D among them, so the sub-heads
    repeat those and per-head gradients are summed over them (views, no copy of x);
  * a narrower head is padded with zero features, a smaller state with zero state components;
    both contribute exact zeros and are cut off again.

The native shapes take none of this."""
import torch
import torch.nn.functional as F

NATIVE = (64, 128)


class Plan:
    def __init__(self, headdim, dstate=None):
        self.hd, self.ds = headdim, dstate
        if headdim in NATIVE:
            self.P, self.split = headdim, 1
        elif headdim < 64:
            self.P, self.split = 64, 1
        elif headdim < 128:
            self.P, self.split = 128, 1
        else:
            self.P, self.split = 64, -(-headdim // 64)
        self.hd_pad = self.P * self.split
        if dstate is None or dstate in NATIVE:
            self.N = dstate
        elif dstate < 64:
            self.N = 64
        elif dstate < 128:
            self.N = 128
        else:
            raise NotImplementedError(f"dstate {dstate} is larger than the SSD kernels take (128)")

    @property
    def native(self):
        return self.split == 1 and self.P == self.hd and self.N == self.ds

    # ---- tensors with a feature axis last: x, z, dout, out, dx (b, L, nh, hd)
    def x(self, t):
        if t is None:
            return None
        if self.hd_pad != self.hd:
            t = F.pad(t, (0, self.hd_pad - self.hd))
        b, L, nh, _ = t.shape
        return t.reshape(b, L, nh * self.split, self.P)

    def x_back(self, t):
        if t is None:
            return None
        b, L, nhs, _ = t.shape
        return t.reshape(b, L, nhs // self.split, self.hd_pad)[..., : self.hd]

    # ---- per-head arrays: dt / dA_cumsum (b, nh, C, Q), dA_chunk (b, nh, C), A / D (nh,)
    def per_head(self, t, axis=1):
        return t if t is None or self.split == 1 else t.repeat_interleave(self.split, dim=axis)

    def per_head_sum(self, t, axis=1):
        if t is None or self.split == 1:
            return t
        shape = list(t.shape)
        shape[axis: axis + 1] = [shape[axis] // self.split, self.split]
        return t.reshape(shape).sum(axis + 1)

    def D(self, D):
        if D is None:
            return None
        if D.dim() == 1:
            return self.per_head(D, 0)
        if self.hd_pad != self.hd:
            D = F.pad(D, (0, self.hd_pad - self.hd))
        return D.reshape(D.shape[0] * self.split, self.P)

    def dD_back(self, dD, D):
        if dD is None:
            return None
        if D.dim() == 1:
            return self.per_head_sum(dD, 0)
        return dD.reshape(D.shape[0], self.hd_pad)[:, : self.hd]

    # ---- B, C, dB, dC (b, L, g, ds)
    def bc(self, t):
        return t if t is None or self.N == self.ds else F.pad(t, (0, self.N - self.ds))

    def bc_back(self, t):
        return t if t is None or self.N == self.ds else t[..., : self.ds]

    # ---- states (b, C, nh, hd, ds)
    def states(self, t):
        if t is None:
            return None
        if self.N != self.ds or self.hd_pad != self.hd:
            t = F.pad(t, (0, self.N - self.ds, 0, self.hd_pad - self.hd))
        b, C, nh = t.shape[:3]
        return t.reshape(b, C, nh * self.split, self.P, self.N)

    def states_back(self, t):
        if t is None:
            return None
        b, C, nhs = t.shape[:3]
        return t.reshape(b, C, nhs // self.split, self.hd_pad, self.N)[..., : self.hd, : self.ds]


def walk_pays(batch, nheads, seqlen, chunk, headdim, dstate, itemsize, backward=False):
    """Whether the kernel in which one workgroup per (batch, head) walks the whole sequence is faster than
    the two launchers it stands for, which spread the chunks over the chip and carry the chunk-local states
    through memory in float32 (4 * batch * nheads * nchunks * headdim * dstate bytes of scratch, which the walk
    does not need).  Both give the same states bit for bit.

    The walk is a serial chain of 64-row stages, a workgroup per compute unit: 256 heads at a time, and its time
    does not depend on how many of them there are.  The two launchers are bound by the chain of stages inside one
    chunk while there are few heads, by the bytes they move (6 TB/s) and, in float32, by their matrix instructions.
    The coefficients are fitted to 1840 measured points (MI355X; 2 to 768 heads, seqlen 500 to 8192, chunk 64 to
    512, all four head and state sizes) with a root mean square error of 4 to 12 %.  Some of them, walk / two
    launchers in us, hdim 64, dstate 128:
      bfloat16 forward,  chunk 256, seqlen 8192:  32 heads 126 /  31, 128 heads 123 / 102, 192 heads 124 / 147,
                                                  256 heads 129 / 187, 264 heads 235 / 201, 320 heads 236 / 244,
                                                  512 heads 256 / 358, 768 heads 371 / 538
                         chunk  64, seqlen  500:  32 heads  14 /  12,  64 heads  14 /  16
                         chunk 512, seqlen  500:  32 heads  12 /  15, 192 heads  13 /  21
      bfloat16 backward, chunk 256, seqlen 8192: 128 heads 151 / 117, 192 heads 154 / 167, 264 heads 291 / 223
      float32 forward,   chunk 256, seqlen 2048:  32 heads 131 /  25, 256 heads 138 / 132, 384 heads 266 / 191.
    Backward the two launchers take the host 25 us a call and the walk 20, so that a walk of less is kept."""
    heads = batch * nheads
    stages = -(-seqlen // 64)
    nchunks = -(-seqlen // chunk)
    rounds = -(-heads // 256)
    state = headdim * dstate
    rel = state / 8192
    inner = -(-min(chunk, seqlen) // 64)  # stages of one chunk
    # carried states: written forward; read and written backward
    nbytes = heads * (nchunks * state * (8 + itemsize * (2 if backward else 1)) + seqlen * headdim * itemsize)
    work = heads * seqlen * rel * 1e-6
    if itemsize == 4:
        walk_us = 5.8 + rounds * (stages * (0.41 + 2.95 * rel) + nchunks * 0.88 * rel)
        pair_us = 5.5 + inner * (0.46 + 2.18 * rel) + nchunks * 0.11 + nbytes / 6.7e6 + 97 * work
        if rel > 1:  # 128 x 128: fewer workgroups per compute unit
            pair_us += heads * nchunks * 0.0144
    else:
        if headdim == 64 and dstate == 128:  # rows copied straight into LDS; other shapes go through registers
            walk_us = 6.6 + rounds * (stages * 0.96 + nchunks * 0.9) if backward else \
                5.0 + rounds * (stages * 0.87 + nchunks * 0.48)
        else:
            walk_us = 5.3 + rounds * (stages * (0.15 + 0.85 * rel) + nchunks * 0.81 * rel)
        if backward:
            pair_us = 9.5 + inner * 0.75 + nchunks * 0.17 + nbytes / 5.9e6 + 7.9 * work
        else:
            pair_us = 5.3 + inner * (0.73 + 0.32 * rel) + nchunks * 0.1 + nbytes / 6.1e6 + 5.3 * work
    return walk_us < (max(pair_us, 25.0) if backward else pair_us)
