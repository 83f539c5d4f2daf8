// Argument checks and small helpers shared by the translation units behind include/ssd_hip.h.
#pragma once
#include <hip/hip_runtime.h>

#include "../../include/ssd_hip.h"
#include "launch_facts.h"
#include "ssd_kernels.h"

using namespace ssd;

namespace {

#define SSD_TRY(expr)            \
  do {                           \
    int _s = (expr);             \
    if (_s != SSD_OK) return _s; \
  } while (0)

inline int launched() { return hipGetLastError() == hipSuccess ? SSD_OK : SSD_ERR_LAUNCH; }
inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }
inline int esize(int dtype) { return dtype == SSD_BF16 ? 2 : 4; }
inline int check_dtype(int dtype) { return (dtype == SSD_F32 || dtype == SSD_BF16) ? SSD_OK : SSD_ERR_DTYPE; }

// A tensor read or written in 16-byte pieces along its dense last axis of `inner` elements.
int check_vec(const void* p, int64_t sb, int64_t sl, int64_t sh, int dtype, int64_t inner) {
  if (!p) return SSD_ERR_NULL;
  const int epl = 16 / esize(dtype);
  if (inner % epl || sb % epl || sl % epl || sh % epl) return SSD_ERR_ALIGN;
  if (reinterpret_cast<uintptr_t>(p) % 16) return SSD_ERR_ALIGN;
  return SSD_OK;
}
int check_f32(const void* p) {
  if (!p) return SSD_ERR_NULL;
  return reinterpret_cast<uintptr_t>(p) % 16 ? SSD_ERR_ALIGN : SSD_OK;
}

// The kernels that copy their operands straight into LDS form 32-bit unsigned byte offsets from
// the strides: tensors addressed with a negative stride go to the register-staged kernels.
inline bool forward_strides(const Strides3& s) { return s.sb >= 0 && s.sl >= 0 && s.sh >= 0; }

// A carried-state tensor is float32 or of the inputs' type (16-byte aligned either way).
int check_state(const void* p, int state_dtype, int dtype) {
  if (state_dtype != SSD_F32 && state_dtype != dtype) return SSD_ERR_DTYPE;
  return check_f32(p);
}

struct Dims {
  int64_t batch, L, nh, g, P, N, Q, C;
};
int check_dims(int64_t batch, int64_t L, int64_t nh, int64_t g, int64_t P, int64_t N, int64_t Q, Dims* d) {
  if (batch <= 0 || L <= 0 || nh <= 0 || g <= 0 || Q <= 0) return SSD_ERR_SHAPE;
  if (nh % g) return SSD_ERR_SHAPE;
  if (Q > 1024 || Q % 4) return SSD_ERR_UNSUPPORTED;
  if (batch > (1 << 20) || nh > (1 << 16) || L > ((int64_t)1 << 30)) return SSD_ERR_SHAPE;
  *d = Dims{batch, L, nh, g, P, N, Q, (L + Q - 1) / Q};
  if (batch * nh * d->C > ((int64_t)1 << 28)) return SSD_ERR_SHAPE;
  return SSD_OK;
}
inline bool dim_ok(int64_t v) { return v == 64 || v == 128; }
// The state-passing entries take the chunking only to locate the last position of each chunk of
// a packed batch; without seq_idx both numbers are ignored.
inline int check_seq_chunks(const int32_t* seq_idx, int64_t seqlen, int64_t chunk, int64_t nchunks) {
  if (!seq_idx) return SSD_OK;
  if (seqlen <= 0 || chunk <= 0 || seqlen > ((int64_t)1 << 30)) return SSD_ERR_SHAPE;
  return (seqlen + chunk - 1) / chunk == nchunks ? SSD_OK : SSD_ERR_SHAPE;
}
inline SeqIdx as_seq(const int32_t* p, int64_t sb, int64_t sl) { return SeqIdx{p, sb, sl}; }
constexpr int kLdsBytes = 160 * 1024;  // LDS of one CU
// Workgroups from which the one-tile kernels of chunks of 64 and 128 rows pay in bfloat16 (one and a half for each
// of 256 compute units; measured at the rules that use it), and for pairs of heads and chunks of 64 rows, where the
// 64-row kernels have only twice the workgroups: from where those no longer run at once, three on each compute unit
// in the chunk scan and four in dx.
constexpr int64_t kMidWorkgroups = 384, kMidScanPairs64 = 385, kMidDxPairs64 = 513;
// Workgroups of float32 chunks of 128 rows up to which both workgroups of the 64-row kernel run at once.
constexpr int64_t kBoth64Row = 128;

// How the kernels that walk the heads deal them to their workgroups, one to a compute unit: each of `sets` (batch, chunk,
// group) sets of `per` heads to `splits` workgroups of its own, or (splits = 0) all heads evenly to 256.  What the heads of a
// set share is fetched again by every workgroup that has some of them, at about the cost of one and a quarter heads: the
// estimates are rounds x (heads of a workgroup and one fetch), and heads with a fetch for each set they can touch.
// us by splits / evenly: scan 9 sets of 32 19.4 / 26.8, 60 of 6 19.9 / 27.7, 64 of 15 29.6 / 31.3, 320 of 10 97 / 88, 384 of 6
// 78 / 72; with gate 192 of 13 113 / 106; dx 320 of 10 124 / 116.
struct HeadsDeal {
  unsigned workgroups;
  int units, splits;
  int64_t cost;  // the estimate, in quarters of a head
};
// Rows they take: 32-bit byte offsets within eight rows, and of a row within a chunk.
inline bool heads_rows(const Strides3& s) { return forward_strides(s) && s.sl < (int64_t(1) << 23); }
// dA and dt are copied in 16-byte pieces.
inline bool heads_vectors(const float* dt, const float* dA) {
  return (reinterpret_cast<uintptr_t>(dt) | reinterpret_cast<uintptr_t>(dA)) % 16 == 0;
}
inline HeadsDeal heads_deal(int64_t sets, int64_t per) {
  const int64_t units = sets * per, each = (units + 255) / 256;  // (units: up to 2^28, see check_dims)
  int64_t splits = 0, least = 4 * each + 5 * ((each - 2 + per) / per + 1);
  if (units <= 256) return HeadsDeal{(unsigned)units, (int)units, (int)per, 9};
  for (int64_t s = 1; s <= per && sets * (s - 1) < 1024; ++s) {
    const int64_t cost = (sets * s + 255) / 256 * (4 * ((per + s - 1) / s) + 5);
    if (cost < least) least = cost, splits = s;
  }
  return HeadsDeal{splits ? (unsigned)(sets * splits) : 256u, (int)units, (int)splits, least};
}
// Whether that estimate is below one of the kernels of one head (or pair) per workgroup: those take `head` for each 256 heads,
// `turn` for each 768, which is how many run at once, and `base`, in 32nds of a head of the walk.  A walk whose heads do not
// divide well, or that fetches what a set shares too often, is behind them at any size (dx of 347 sets of four heads 59 / 68
// us).  Fitted to 148 to 161 points a stage, sets of 1 to 64 heads, 257 to 7100 heads, each in both kernels: where it chooses
// the walk that is 8 % behind at one of the 615 points (scan, 1884 heads in groups of six) and 2 to 4 % at five.
inline bool heads_pay(const HeadsDeal& deal, int head, int turn, int base) {
  return 8 * deal.cost <= head * ((deal.units + 255) / 256) + turn * ((deal.units + 767) / 768) + base;
}

template <typename K>
int allow_smem(K kernel, int bytes) {
  if (bytes <= 64 * 1024) return SSD_OK;
  return launch_facts::smem(reinterpret_cast<const void*>(kernel), bytes) ? SSD_OK : SSD_ERR_LAUNCH;
}

// Calls f.template run<T, P, N>() for the runtime (dtype, hdim, dstate).
template <typename F>
int dispatch_tpn(int dtype, int64_t P, int64_t N, F f) {
  if (dtype == SSD_BF16) {
    if (P == 64 && N == 64) return f.template run<bf16_t, 64, 64>();
    if (P == 64 && N == 128) return f.template run<bf16_t, 64, 128>();
    if (P == 128 && N == 64) return f.template run<bf16_t, 128, 64>();
    return f.template run<bf16_t, 128, 128>();
  }
  if (P == 64 && N == 64) return f.template run<float, 64, 64>();
  if (P == 64 && N == 128) return f.template run<float, 64, 128>();
  if (P == 128 && N == 64) return f.template run<float, 128, 64>();
  return f.template run<float, 128, 128>();
}

}  // namespace
