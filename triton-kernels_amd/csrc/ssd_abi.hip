// C ABI of the SSD stages other than the chunk scan (ssd_scan_abi.hip): argument validation and kernel launches.
// Declarations and the reference launcher each entry point replaces are in include/ssd_hip.h.
#include "../../include/ssd_hip.h"

#include <type_traits>

#include "ema_gemm_kernels.h"
#include "ssd_heads_kernels.h"
#include "ssd_host.h"
#include "ssd_kernels.h"

using namespace ssd;

namespace {

template <int MODE>
struct StateLaunch {
  const void *x, *B;
  Strides3 sx, sB;
  const float *dt, *dA;
  void* states;
  int states_dtype;
  Dims d;
  SeqIdx seq;
  hipStream_t st;
  template <typename T, int P, int N>
  int run() const {
    if constexpr (!std::is_same<T, float>::value)
      if (states_dtype != SSD_F32) return run_as<T, P, N, T>();
    return run_as<T, P, N, float>();
  }
  template <typename T, int P, int N, typename TO>
  int run_as() const {
    auto kernel = ssd_chunk_state_kernel<T, P, N, MODE, TO>;
    constexpr int smem = StateSmem<T, P, N>::kBytes;
    SSD_TRY(allow_smem(kernel, smem));
    hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.C * d.nh)), dim3(256), smem, st, (const T*)x, sx,
                       (const T*)B, sB, dt, dA, (TO*)states, (int)d.nh, (int)(d.nh / d.g), (int)d.L, (int)d.Q,
                       (int)d.C, seq);
    return launched();
  }
};

// The stages ahead of the state passing in one launch (ssd_front_kernel).
struct FrontLaunch {
  const void *x, *B, *C;
  Strides3 sx, sB, sC;
  const void* dt;
  int dt_dtype;
  Strides3 sd;
  const float *A, *bias;
  float *dA, *dt_out;
  int softplus;
  float dt_min, dt_max;
  float *states, *cb;
  Dims d;
  SeqIdx seq;
  hipStream_t st;
  template <typename T, int P, int N>
  int run() const {
    return dt_dtype == SSD_BF16 ? run_as<T, P, N, bf16_t>() : run_as<T, P, N, float>();
  }
  template <typename T, int P, int N, typename TD>
  int run_as() const {
    auto kernel = ssd_front_kernel<T, P, N, TD>;
    const int smem = front_smem_bytes<T, P, N>((int)d.Q);
    SSD_TRY(allow_smem(kernel, smem));
    const int tiles = (int)((d.Q + 63) / 64);
    const int64_t nstate = d.batch * d.C * d.nh, grid = nstate + d.batch * d.C * d.g * tiles * tiles;
    if (grid > 0x7fffffff) return SSD_ERR_SHAPE;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), smem, st, (const T*)x, sx, (const T*)B, sB, (const T*)C, sC,
                       DtSource<TD>{(const TD*)dt, sd, A, bias, dA, dt_out, softplus, dt_min, dt_max}, states, cb, (int)d.nh,
                       (int)d.g, (int)d.L, (int)d.Q, (int)d.C, (int)nstate, tiles, seq);
    return launched();
  }
};

struct WalkLaunch {
  const void *x, *B;
  Strides3 sx, sB;
  const float *dt, *dA, *initial;
  void* out;
  int out_dtype;
  float* final_states;
  Dims d;
  hipStream_t st;
  template <typename T, int P, int N>
  int run() const {
    if (out_dtype == SSD_BF16) return run_as<T, P, N, bf16_t>();
    return run_as<T, P, N, float>();
  }
  template <typename T, int P, int N, typename TO>
  int run_as() const {
#ifndef SSD_WALK_DMA  // 0: development builds without the kernel that copies its rows straight into LDS
#define SSD_WALK_DMA 1
#endif
    // (the kernel keeps the byte offset of a row inside a stage in 32 bits)
    if constexpr (SSD_WALK_DMA && std::is_same<T, bf16_t>::value && P == 64 && N == 128) {
      if (forward_strides(sx) && forward_strides(sB) && sx.sl < (int64_t(1) << 24) && sB.sl < (int64_t(1) << 24)) {
        auto kernel = ssd_state_walk_dma_kernel<TO>;
        constexpr int smem = WalkDmaSmem::kBytes;
        SSD_TRY(allow_smem(kernel, smem));
        hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.nh)), dim3(512), smem, st, (const bf16_t*)x, sx,
                           (const bf16_t*)B, sB, dt, dA, initial, (TO*)out, final_states, (int)d.nh, (int)(d.nh / d.g),
                           (int)d.L, (int)d.Q, (int)d.C);
        return launched();
      }
    }
#ifndef SSD_WALK_NSPLIT  // 2: two workgroups per (b, h), half the state columns each (measured no faster: x crosses the L2 twice)
#define SSD_WALK_NSPLIT 1
#endif
    constexpr int NSPLIT = (SSD_WALK_NSPLIT == 2 && ((P / 32) * (N / 64)) % 4 == 0 && P * N <= 64 * 128) ? 2 : 1;
    auto kernel = ssd_state_walk_kernel<T, P, N, TO, NSPLIT>;
    constexpr int smem = WalkSmem<T, P, N / NSPLIT>::kBytes;
    SSD_TRY(allow_smem(kernel, smem));
    hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.nh * NSPLIT)), dim3(256), smem, st, (const T*)x, sx,
                       (const T*)B, sB, dt, dA, initial, (TO*)out, final_states, (int)d.nh, (int)(d.nh / d.g),
                       (int)d.L, (int)d.Q, (int)d.C);
    return launched();
  }
};

// Number of per-wave slots the dx kernels of a shape write per (batch, chunk, head): 256-row super-tiles have four waves,
// or eight where the walk over the heads may run (the others then zero what they do not use).
struct DxSlots {
  int64_t Q;
  template <typename T, int P, int N>
  static bool wide(int64_t Q) {
    return Q % 256 == 0 && WideSmem<T, P, N>::kBytes <= kLdsBytes;
  }
  template <typename T, int P, int N>
  int run() const {
    if (std::is_same<T, bf16_t>::value && P == 64 && Q == 256) return DxHeadsSmem<N>::kSlots;
    return wide<T, P, N>(Q) ? (int)(4 * (Q / 256)) : (int)(4 * ((Q + 63) / 64));
  }
};

struct DxLaunch {
  const float* cb;
  const void *x, *dout, *B;
  Strides3 sx, sd, sB, sdx;
  const float *dt, *dA;
  const void* dstates;
  int states_dtype;
  const float* D;
  int d_has_hdim;
  void* dx;
  float* ddt;
  Dims d;
  SeqIdx seq;
  float* dD_part;
  hipStream_t st;
  template <typename T, int P, int N>
  int run() const {
    if constexpr (!std::is_same<T, float>::value)
      if (states_dtype != SSD_F32) return run_as<T, P, N, T>();
    return run_as<T, P, N, float>();
  }
  template <typename T, int P, int N, typename TS, int ST>
  int launch_mid() const {
    auto kernel = ssd_chunk_scan_bwd_dx_mid_kernel<T, P, N, TS, ST>;
    constexpr int smem = MidSmem<T, 2 * P, N, ST>::bytes_for(2);
    SSD_TRY(allow_smem(kernel, smem));
    hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.C * (d.nh / 2))), dim3(256), smem, st, cb, (const T*)x, sx,
                       (const T*)dout, sd, dt, dA, (const T*)B, sB, (const TS*)dstates, D, d_has_hdim, (T*)dx, sdx, ddt,
                       (int)d.nh, (int)(d.nh / d.g), (int)d.g, (int)d.L, (int)d.C, seq, dD_part, 4 * (ST / 64));
    return launched();
  }
  template <typename T, int P, int N, typename TS>
  int run_as() const {
    if constexpr (std::is_same<T, bf16_t>::value && std::is_same<TS, bf16_t>::value && P == 64) {
      // The walk over the heads, where its deal pays.  The 256-row kernel / the walk, us, dstate 128: 128 heads of all (batch,
      // chunk) pairs 16.9 / 14.1, 256 19.2 / 15.3, 512 27 / 22, 3072 121 / 91; behind are 417 in groups of three 23.4 / 25.3,
      // 1388 of four 59 / 68, and at dstate 64 1430 of five 50 / 57, 1885 of five 68 / 75, 3444 of four
      // 124 / 137.  Up to 64 heads, where the walk would be faster too (15 / 12.5), the results have the same bits for states
      // of either type, which the header promises that far.
      const int64_t units = d.batch * d.C * d.nh;
      const HeadsDeal deal = heads_deal(d.batch * d.C * d.g, d.nh / d.g);
      const bool pays = units > 64 && heads_pay(deal, 32, 28, 16);
      if (d.Q == 256 && pays && !(D && d_has_hdim) && heads_vectors(dt, dA) && heads_rows(sx) && heads_rows(sd) && heads_rows(sdx)) {
        auto kernel = deal.splits ? ssd_chunk_scan_bwd_dx_heads_kernel<N, false> : ssd_chunk_scan_bwd_dx_heads_kernel<N, true>;
        constexpr int smem = DxHeadsSmem<N>::kBytes;
        static_assert(smem <= kLdsBytes, "the heads under way must fit the LDS of a compute unit");
        SSD_TRY(allow_smem(kernel, smem));
        hipLaunchKernelGGL(kernel, dim3(deal.workgroups), dim3(512), smem, st, cb, (const T*)x, sx,
                           (const T*)dout, sd, dt, dA, (const T*)B, sB, (const TS*)dstates, D, (T*)dx, sdx, ddt,
                           (int)d.nh, (int)(d.nh / d.g), (int)d.g, (int)d.L, (int)d.C, deal.units, deal.splits, seq, dD_part);
        return launched();
      }
    }
    constexpr int wide_smem = WideSmem<T, P, N>::kBytes;
    if (DxSlots::wide<T, P, N>(d.Q)) {  // (it must also fit the LDS of a CU)
      auto kernel = ssd_chunk_scan_bwd_dx_wide_kernel<T, P, N, TS>;
      SSD_TRY(allow_smem(kernel, wide_smem));
      const int stiles = (int)(d.Q / 256);
      hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.C * d.nh * stiles)), dim3(256), wide_smem, st, cb,
                         (const T*)x, sx, (const T*)dout, sd, dt, dA, (const T*)B, sB, (const TS*)dstates, D,
                         d_has_hdim, (T*)dx, sdx, ddt, (int)d.nh, (int)(d.nh / d.g), (int)d.g, (int)d.L, (int)d.Q,
                         (int)d.C, stiles, seq, dD_part, DxSlots{d.Q}.template run<T, P, N>());
      return launched();
    }
    if constexpr (P == 64 && sizeof(T) == 2) {
      // Chunks of 64 or 128 rows with two adjacent dense heads of a group per workgroup, rows at 32-bit byte offsets,
      // and enough of them.  The 64-row kernel / this one, us, dstate 128, inputs from memory: b8 nh32 L8192 chunk
      // 128 443 / 279, chunk 64 352 / 274; chunk 128 384 pairs 22.3 / 20.0, 512 25.5 / 22.4; chunk 64 384 pairs
      // 11.5 / 12.3, 512 13.0 / 14.0, 576 17.0 / 14.2; b1 nh8 L2000 chunk 64 dstate 64 (128 pairs) 6.6 / 7.7.
      auto near = [&](const Strides3& s) { return forward_strides(s) && s.sl * d.Q < (int64_t(1) << 28); };
      const bool dense = sx.sh == P && sd.sh == P && sdx.sh == P && (d.nh / d.g) % 2 == 0;
      const int64_t pairs = d.batch * d.C * (d.nh / 2);
      if (dense && near(sx) && near(sd) && near(sB) && near(sdx)) {
        if (d.Q == 128 && pairs >= kMidWorkgroups) return launch_mid<T, P, N, TS, 128>();
        if (d.Q == 64 && pairs >= kMidDxPairs64) return launch_mid<T, P, N, TS, 64>();
      }
    }
    auto kernel = ssd_chunk_scan_bwd_dx_kernel<T, P, N, TS>;
    constexpr int smem = ScanSmem<T, P, N>::kBytes;
    SSD_TRY(allow_smem(kernel, smem));
    const int mtiles = (int)((d.Q + 63) / 64);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.C * d.nh * mtiles)), dim3(256), smem, st, cb,
                       (const T*)x, sx, (const T*)dout, sd, dt, dA, (const T*)B, sB, (const TS*)dstates, D, d_has_hdim,
                       (T*)dx, sdx, ddt, (int)d.nh, (int)(d.nh / d.g), (int)d.g, (int)d.L, (int)d.Q, (int)d.C, mtiles,
                       seq, dD_part);
    return launched();
  }
};

template <int MODE>
struct GroupLaunch {
  const void* a;
  Strides3 sa;
  const void* s;
  int s_dtype;
  const float *dt, *dA;
  const void* bc;
  Strides3 sbc;
  float *out, *ddA;
  Dims d;
  SeqIdx seq;
  hipStream_t st;
  template <typename T, int P, int N>
  int run() const {
    if constexpr (!std::is_same<T, float>::value)
      if (s_dtype != SSD_F32) return run_as<T, P, N, T>();
    return run_as<T, P, N, float>();
  }
  template <typename T, int P, int N, typename TS>
  int run_as() const {
#ifndef SSD_GROUP_DMA  // 0: development builds without the kernel that copies its operands straight into LDS
#define SSD_GROUP_DMA 1
#endif
    if constexpr (SSD_GROUP_DMA && std::is_same<T, bf16_t>::value && std::is_same<TS, bf16_t>::value && P == 64 && N == 128) {
      // (the kernel keeps the byte offset of a row inside a chunk in 32 bits)
      if (d.Q % 64 == 0 && !seq.p && forward_strides(sa) && forward_strides(sbc) && d.Q * sa.sl < (int64_t(1) << 30)) {
        auto kernel = ssd_group_grad_dma_kernel<MODE>;
        constexpr int smem = GroupDmaSmem::kBytes;
        SSD_TRY(allow_smem(kernel, smem));
        const int mtiles = (int)(d.Q / 64);
        if (d.batch * d.C * d.g * mtiles > 0x7fffffff) return SSD_ERR_SHAPE;
        hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.C * d.g * mtiles)), dim3(256), smem, st, (const bf16_t*)a,
                           sa, (const bf16_t*)s, dt, dA, (const bf16_t*)bc, sbc, out, ddA, (int)d.nh, (int)(d.nh / d.g),
                           (int)d.g, (int)d.L, (int)d.Q, (int)d.C, mtiles);
        return launched();
      }
    }
    auto kernel = ssd_group_grad_kernel<T, P, N, MODE, TS>;
    constexpr int smem = GroupSmem<T, P, N>::kBytes;
    SSD_TRY(allow_smem(kernel, smem));
    const int mtiles = (int)((d.Q + 63) / 64);
    if (d.batch * d.C * d.g * mtiles > 0x7fffffff) return SSD_ERR_SHAPE;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.C * d.g * mtiles)), dim3(256), smem, st, (const T*)a, sa,
                       (const TS*)s, dt, dA, (const T*)bc, sbc, out, ddA, (int)d.nh, (int)(d.nh / d.g), (int)d.g, (int)d.L,
                       (int)d.Q, (int)d.C, mtiles, seq);
    return launched();
  }
};

int launch_row_cumsum(float* v, int64_t Q, int64_t rows, hipStream_t st) {
  hipLaunchKernelGGL(ssd_row_cumsum_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, st, v, (int)Q, rows);
  return launched();
}

// Whether the state-passing kernels keep two turns of chunks under way: where there is more than one turn and the
// workgroups leave the chip latency bound, up to four on each of 256 compute units with four state elements per
// thread (two with eight, which hold twice the registers).  One turn / two, us, 40 chunks: 64 workgroups 12.8 / 9.3
// (backward 26.2 / 18.6), 384 20.2 / 18.5 (40.6 / 35.4), 1024 44.7 / 45.5 (65.4 / 64.7); 8 chunks: 192 workgroups
// 4.9 / 4.4, 4096 41.9 / 44.9 (61.1 / 65.1).  Eight elements, backward, 40 chunks: 512 workgroups 41.7 / 38.3, 768 53 / 63.
inline bool passing_ahead(int64_t nchunks, int64_t workgroups, int per_thread) {
  return nchunks > 4 && workgroups * per_thread <= 4 * 1024;
}

template <typename T, typename TO, int K>
int launch_bmm(const void* a, Strides3 sa, const void* bm, Strides3 sb, void* out, const Dims& d, SeqIdx seq,
               hipStream_t st) {
  auto kernel = ssd_bmm_kernel<T, TO, K>;
  constexpr int smem = bmm_smem_bytes<T, K>();
  SSD_TRY(allow_smem(kernel, smem));
  const int tiles = (int)((d.Q + 63) / 64);
  const int64_t grid = d.batch * d.C * d.g * tiles * tiles;
  if (grid > 0x7fffffff) return SSD_ERR_SHAPE;
  hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), smem, st, (const T*)a, sa, (const T*)bm, sb, (TO*)out,
                     (int)d.g, (int)d.L, (int)d.Q, (int)d.C, tiles, seq);
  return launched();
}

}  // namespace

extern "C" {

int ssd_chunk_cumsum_fwd(const void* dt, int dt_dtype, int64_t dt_sb, int64_t dt_sl, int64_t dt_sh,
                         const float* A, const float* dt_bias, float* dA_cumsum, float* dt_out,
                         int64_t batch, int64_t seqlen, int64_t nheads, int64_t chunk, int dt_softplus,
                         float dt_min, float dt_max, void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, 1, 0, 0, chunk, &d));
  SSD_TRY(check_dtype(dt_dtype));
  if (!dt || !A || !dA_cumsum || !dt_out) return SSD_ERR_NULL;
  const Strides3 sd{dt_sb, dt_sl, dt_sh};
  // heads per workgroup: a power of two up to 8 (32-byte pieces of dt rows; more heads per workgroup
  // leave too few workgroups to hide their latency) whose Q x HT tile stays within 64 KB of LDS
  int HT = 8;
  while (HT > 1 && (HT / 2 >= nheads || (int64_t)HT * (chunk + 1) * 4 > 64 * 1024)) HT /= 2;
  const int hgroups = (int)((nheads + HT - 1) / HT);
  const int64_t blocks = batch * d.C * hgroups;
  if (blocks > 0x7fffffff) return SSD_ERR_SHAPE;
  const unsigned grid = (unsigned)blocks;
  const int smem = HT * (int)(chunk + 1) * 4;
  if (dt_dtype == SSD_BF16)
    hipLaunchKernelGGL(ssd_cumsum_kernel<bf16_t>, dim3(grid), dim3(256), smem, as_stream(stream), (const bf16_t*)dt,
                       sd, A, dt_bias, dA_cumsum, dt_out, (int)nheads, (int)seqlen, (int)chunk, (int)d.C, dt_softplus,
                       dt_min, dt_max, HT, hgroups);
  else
    hipLaunchKernelGGL(ssd_cumsum_kernel<float>, dim3(grid), dim3(256), smem, as_stream(stream), (const float*)dt, sd,
                       A, dt_bias, dA_cumsum, dt_out, (int)nheads, (int)seqlen, (int)chunk, (int)d.C, dt_softplus,
                       dt_min, dt_max, HT, hgroups);
  return launched();
}

int ssd_chunk_state_fwd(const void* B, int64_t b_sb, int64_t b_sl, int64_t b_sg, const void* x,
                        int64_t x_sb, int64_t x_sl, int64_t x_sh, int dtype, const float* dt,
                        const float* dA_cumsum, float* states, int64_t batch, int64_t seqlen,
                        int64_t nheads, int64_t ngroups, int64_t hdim, int64_t dstate, int64_t chunk,
                        const int32_t* seq_idx, int64_t seq_sb, int64_t seq_sl, void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  if (!dim_ok(hdim) || !dim_ok(dstate)) return SSD_ERR_UNSUPPORTED;
  SSD_TRY(check_vec(x, x_sb, x_sl, x_sh, dtype, hdim));
  SSD_TRY(check_vec(B, b_sb, b_sl, b_sg, dtype, dstate));
  if (!dt || !dA_cumsum) return SSD_ERR_NULL;
  SSD_TRY(check_f32(states));
  return dispatch_tpn(dtype, hdim, dstate,
                      StateLaunch<0>{x, B, Strides3{x_sb, x_sl, x_sh}, Strides3{b_sb, b_sl, b_sg}, dt, dA_cumsum,
                                     states, SSD_F32, d, as_seq(seq_idx, seq_sb, seq_sl), as_stream(stream)});
}

int ssd_chunk_state_passing_fwd(const void* B, int64_t b_sb, int64_t b_sl, int64_t b_sg, const void* x,
                                int64_t x_sb, int64_t x_sl, int64_t x_sh, int dtype, const float* dt,
                                const float* dA_cumsum, const float* initial, void* out, int out_dtype,
                                float* final_states, int64_t batch, int64_t seqlen, int64_t nheads,
                                int64_t ngroups, int64_t hdim, int64_t dstate, int64_t chunk, void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  SSD_TRY(check_dtype(out_dtype));
  if (!dim_ok(hdim) || !dim_ok(dstate) || chunk % 64) return SSD_ERR_UNSUPPORTED;
  SSD_TRY(check_vec(x, x_sb, x_sl, x_sh, dtype, hdim));
  SSD_TRY(check_vec(B, b_sb, b_sl, b_sg, dtype, dstate));
  SSD_TRY(check_f32(dt));  // fetched in 16-byte pieces
  SSD_TRY(check_f32(dA_cumsum));
  SSD_TRY(check_f32(out));
  SSD_TRY(check_f32(final_states));
  if (initial) SSD_TRY(check_f32(initial));
  return dispatch_tpn(dtype, hdim, dstate,
                      WalkLaunch{x, B, Strides3{x_sb, x_sl, x_sh}, Strides3{b_sb, b_sl, b_sg}, dt, dA_cumsum, initial,
                                 out, out_dtype, final_states, d, as_stream(stream)});
}

int ssd_state_passing_fwd(const float* states, const float* dA_chunk, int64_t da_sb, int64_t da_sh,
                          int64_t da_sc, const float* initial, void* out, int out_dtype, float* final_states,
                          int64_t batch, int64_t nchunks, int64_t nheads, int64_t dim, const int32_t* seq_idx,
                          int64_t seq_sb, int64_t seq_sl, int64_t seqlen, int64_t chunk, void* stream) {
  if (batch <= 0 || nchunks <= 0 || nheads <= 0 || dim <= 0) return SSD_ERR_SHAPE;
  if (dim % 4) return SSD_ERR_ALIGN;
  if (!dA_chunk) return SSD_ERR_NULL;
  SSD_TRY(check_dtype(out_dtype));
  SSD_TRY(check_seq_chunks(seq_idx, seqlen, chunk, nchunks));
  SSD_TRY(check_f32(states));
  SSD_TRY(check_f32(out));
  SSD_TRY(check_f32(final_states));
  if (initial) SSD_TRY(check_f32(initial));
  // four elements per thread: 16-byte loads of the float32 states, 8-byte stores of a bfloat16 out
  // (eight per thread, which makes those stores 16 bytes, measured 8 % slower here)
  const int tiles = (int)((dim + 1023) / 1024);
  const int64_t grid = batch * nheads * tiles;
  if (grid > 0x7fffffff || dim > (1 << 24)) return SSD_ERR_SHAPE;
  const bool ahead = passing_ahead(nchunks, grid, 4);
#define SSD_SP_LAUNCH(TO, AHEAD)                                                                                   \
  hipLaunchKernelGGL((ssd_state_passing_kernel<TO, 4, AHEAD>), dim3((unsigned)grid), dim3(256), 0, as_stream(stream), states, \
                     dA_chunk, da_sb, da_sh, da_sc, initial, (TO*)out, final_states, (int)nheads, (int)nchunks,      \
                     (int)dim, tiles, as_seq(seq_idx, seq_sb, seq_sl), (int)seqlen, (int)chunk)
  if (out_dtype == SSD_BF16 && ahead) SSD_SP_LAUNCH(bf16_t, true);
  else if (out_dtype == SSD_BF16) SSD_SP_LAUNCH(bf16_t, false);
  else if (ahead) SSD_SP_LAUNCH(float, true);
  else SSD_SP_LAUNCH(float, false);
#undef SSD_SP_LAUNCH
  return launched();
}

int ssd_bmm_chunk_fwd(const void* a, int64_t a_sb, int64_t a_sl, int64_t a_sg, const void* bm,
                      int64_t b_sb, int64_t b_sl, int64_t b_sg, int dtype, void* out, int out_dtype,
                      int64_t batch, int64_t seqlen, int64_t ngroups, int64_t k, int64_t chunk,
                      const int32_t* seq_idx, int64_t seq_sb, int64_t seq_sl, void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, ngroups, ngroups, 0, k, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  SSD_TRY(check_dtype(out_dtype));
  if (!dim_ok(k)) return SSD_ERR_UNSUPPORTED;
  if (out_dtype != SSD_F32 && out_dtype != dtype) return SSD_ERR_DTYPE;
  SSD_TRY(check_vec(a, a_sb, a_sl, a_sg, dtype, k));
  SSD_TRY(check_vec(bm, b_sb, b_sl, b_sg, dtype, k));
  if (!out) return SSD_ERR_NULL;
  const Strides3 sa{a_sb, a_sl, a_sg}, sb{b_sb, b_sl, b_sg};
  hipStream_t st = as_stream(stream);
  const SeqIdx seq = as_seq(seq_idx, seq_sb, seq_sl);
  if (dtype == SSD_BF16) {
    if (out_dtype == SSD_F32)
      return k == 64 ? launch_bmm<bf16_t, float, 64>(a, sa, bm, sb, out, d, seq, st)
                     : launch_bmm<bf16_t, float, 128>(a, sa, bm, sb, out, d, seq, st);
    return k == 64 ? launch_bmm<bf16_t, bf16_t, 64>(a, sa, bm, sb, out, d, seq, st)
                   : launch_bmm<bf16_t, bf16_t, 128>(a, sa, bm, sb, out, d, seq, st);
  }
  return k == 64 ? launch_bmm<float, float, 64>(a, sa, bm, sb, out, d, seq, st)
                 : launch_bmm<float, float, 128>(a, sa, bm, sb, out, d, seq, st);
}

int ssd_chunk_scan_bwd_dstates(const void* C, int64_t c_sb, int64_t c_sl, int64_t c_sg, const void* dout,
                               int64_t d_sb, int64_t d_sl, int64_t d_sh, int dtype, const float* dA_cumsum,
                               void* dprev_states, int states_dtype, int64_t batch, int64_t seqlen,
                               int64_t nheads, int64_t ngroups, int64_t hdim, int64_t dstate, int64_t chunk,
                               const int32_t* seq_idx, int64_t seq_sb, int64_t seq_sl, void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  if (!dim_ok(hdim) || !dim_ok(dstate)) return SSD_ERR_UNSUPPORTED;
  SSD_TRY(check_vec(dout, d_sb, d_sl, d_sh, dtype, hdim));
  SSD_TRY(check_vec(C, c_sb, c_sl, c_sg, dtype, dstate));
  if (!dA_cumsum) return SSD_ERR_NULL;
  SSD_TRY(check_state(dprev_states, states_dtype, dtype));
  return dispatch_tpn(dtype, hdim, dstate,
                      StateLaunch<1>{dout, C, Strides3{d_sb, d_sl, d_sh}, Strides3{c_sb, c_sl, c_sg}, dA_cumsum,
                                     dA_cumsum, dprev_states, states_dtype, d, as_seq(seq_idx, seq_sb, seq_sl),
                                     as_stream(stream)});
}

size_t ssd_state_passing_bwd_workspace_bytes(int64_t batch, int64_t nchunks, int64_t nheads, int64_t dim) {
  if (batch <= 0 || nchunks <= 0 || nheads <= 0 || dim <= 0) return 0;
  const int64_t tiles = (dim + 1023) / 1024;
  return (size_t)(batch * nheads * nchunks * tiles * 4) * sizeof(float);
}

int ssd_state_passing_bwd(const void* states, int states_dtype, const float* dA_chunk, int64_t da_sb, int64_t da_sh,
                          int64_t da_sc, const void* dout, int dout_dtype, const float* dfinal, void* dstates,
                          int dstates_dtype,
                          float* ddA_chunk, float* dinit, void* workspace, size_t workspace_bytes,
                          int64_t batch, int64_t nchunks, int64_t nheads, int64_t dim, const int32_t* seq_idx,
                          int64_t seq_sb, int64_t seq_sl, int64_t seqlen, int64_t chunk, void* stream) {
  if (batch <= 0 || nchunks <= 0 || nheads <= 0 || dim <= 0) return SSD_ERR_SHAPE;
  if (dim % 4) return SSD_ERR_ALIGN;
  if (!dA_chunk || !ddA_chunk) return SSD_ERR_NULL;
  SSD_TRY(check_seq_chunks(seq_idx, seqlen, chunk, nchunks));
  const SeqIdx seq = as_seq(seq_idx, seq_sb, seq_sl);
  SSD_TRY(check_dtype(states_dtype));
  SSD_TRY(check_dtype(dout_dtype));
  SSD_TRY(check_dtype(dstates_dtype));
  SSD_TRY(check_f32(states));
  SSD_TRY(check_f32(dout));
  SSD_TRY(check_f32(dstates));
  SSD_TRY(check_f32(workspace));
  if (dfinal) SSD_TRY(check_f32(dfinal));
  if (dinit) SSD_TRY(check_f32(dinit));
  if (workspace_bytes < ssd_state_passing_bwd_workspace_bytes(batch, nchunks, nheads, dim)) return SSD_ERR_SHAPE;
  // eight elements per thread when every state-sized tensor is bfloat16 (16-byte accesses)
  const bool wide = states_dtype == SSD_BF16 && dout_dtype == SSD_BF16 && dstates_dtype == SSD_BF16 && dim % 8 == 0;
  const int per_block = wide ? 2048 : 1024;
  const int tiles = (int)((dim + per_block - 1) / per_block);
  const int64_t grid = batch * nheads * tiles;
  if (grid > 0x7fffffff || dim > (1 << 24)) return SSD_ERR_SHAPE;
  hipStream_t st = as_stream(stream);
  float* part = static_cast<float*>(workspace);
  // the three tensors are float32 or bfloat16 independently of each other
  // (packed, the form with two turns also requests a turn past the end: it needs more than two turns to pay)
  const bool ahead = passing_ahead(seq.p ? nchunks - 4 : nchunks, grid, wide ? 8 : 4);
  auto launch = [&](auto ts, auto td, auto tg, auto elements) {
    using TS = decltype(ts);
    using TD = decltype(td);
    using TG = decltype(tg);
    constexpr int E = decltype(elements)::value;
    auto kernel = seq.p ? (ahead ? ssd_state_passing_bwd_kernel<TS, TD, TG, E, true, true>
                                 : ssd_state_passing_bwd_kernel<TS, TD, TG, E, false, true>)
                        : (ahead ? ssd_state_passing_bwd_kernel<TS, TD, TG, E, true, false>
                                 : ssd_state_passing_bwd_kernel<TS, TD, TG, E, false, false>);
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(256), 0, st,
                       (const TS*)states, dA_chunk, da_sb, da_sh, da_sc, (const TD*)dout, dfinal, (TG*)dstates, part,
                       dinit, (int)nheads, (int)nchunks, (int)dim, tiles, seq, (int)seqlen, (int)chunk);
  };
  using Four = std::integral_constant<int, 4>;
  using Eight = std::integral_constant<int, 8>;
  auto pick_g = [&](auto ts, auto td) {
    if (dstates_dtype == SSD_BF16) launch(ts, td, bf16_t(), Four());
    else launch(ts, td, float(), Four());
  };
  auto pick_d = [&](auto ts) {
    if (dout_dtype == SSD_BF16) pick_g(ts, bf16_t());
    else pick_g(ts, float());
  };
  if (wide) launch(bf16_t(), bf16_t(), bf16_t(), Eight());
  else if (states_dtype == SSD_BF16) pick_d(bf16_t());
  else pick_d(float());
  SSD_TRY(launched());
  const int64_t total = batch * nheads * nchunks;
  hipLaunchKernelGGL(ssd_state_passing_bwd_finish_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                     part, dA_chunk, da_sb, da_sh, da_sc, ddA_chunk, (int)nheads, (int)nchunks, tiles * 4,
                     dinit ? 1 : 0, total, seq, (int)seqlen, (int)chunk);
  return launched();
}

size_t ssd_chunk_scan_state_passing_bwd_workspace_bytes(int64_t batch, int64_t nchunks, int64_t nheads) {
  if (batch <= 0 || nchunks <= 0 || nheads <= 0) return 0;
  return (size_t)(batch * nheads * nchunks * 8) * sizeof(float);  // a partial dot per wave
}

int ssd_chunk_scan_state_passing_bwd(const void* C, int64_t c_sb, int64_t c_sl, int64_t c_sg, const void* dout,
                                     int64_t d_sb, int64_t d_sl, int64_t d_sh, int dtype, const float* dA_cumsum,
                                     const void* states, int states_dtype, const float* dfinal, void* dstates,
                                     int dstates_dtype, float* ddA_chunk, float* dinit, void* workspace,
                                     size_t workspace_bytes, int64_t batch, int64_t seqlen, int64_t nheads,
                                     int64_t ngroups, int64_t hdim, int64_t dstate, int64_t chunk, void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  SSD_TRY(check_dtype(states_dtype));
  SSD_TRY(check_dtype(dstates_dtype));
  // what the kernel is written for: its tiles and its three state buffers in LDS have these sizes
  if (dtype != SSD_BF16 || states_dtype != SSD_BF16 || hdim != 64 || dstate != 128 || chunk % 64 || chunk < 128)
    return SSD_ERR_UNSUPPORTED;
  SSD_TRY(check_vec(dout, d_sb, d_sl, d_sh, dtype, hdim));
  SSD_TRY(check_vec(C, c_sb, c_sl, c_sg, dtype, dstate));
  SSD_TRY(check_f32(dA_cumsum));  // fetched in 16-byte pieces
  SSD_TRY(check_f32(states));
  SSD_TRY(check_f32(dstates));
  SSD_TRY(check_f32(workspace));
  if (!ddA_chunk) return SSD_ERR_NULL;
  if (dfinal) SSD_TRY(check_f32(dfinal));
  if (dinit) SSD_TRY(check_f32(dinit));
  if (workspace_bytes < ssd_chunk_scan_state_passing_bwd_workspace_bytes(batch, d.C, nheads)) return SSD_ERR_SHAPE;
  const Strides3 sd{d_sb, d_sl, d_sh}, sc{c_sb, c_sl, c_sg};
  // (the kernel keeps the byte offset of a row inside a stage in 32 bits)
  if (!forward_strides(sd) || !forward_strides(sc) || sd.sl >= (int64_t(1) << 24) || sc.sl >= (int64_t(1) << 24))
    return SSD_ERR_UNSUPPORTED;
  if (batch * nheads > 0x7fffffff) return SSD_ERR_SHAPE;
  hipStream_t st = as_stream(stream);
  float* part = static_cast<float*>(workspace);
  constexpr int smem = WalkBwdDmaSmem::kBytes;
  auto launch = [&](auto tg) -> int {
    using TG = decltype(tg);
    auto kernel = ssd_state_walk_bwd_dma_kernel<TG>;
    SSD_TRY(allow_smem(kernel, smem));
    hipLaunchKernelGGL(kernel, dim3((unsigned)(batch * nheads)), dim3(512), smem, st, (const bf16_t*)dout, sd,
                       (const bf16_t*)C, sc, dA_cumsum, (const bf16_t*)states, dfinal, (TG*)dstates, part, dinit,
                       (int)nheads, (int)(nheads / ngroups), (int)seqlen, (int)chunk, (int)d.C);
    return launched();
  };
  SSD_TRY(dstates_dtype == SSD_BF16 ? launch(bf16_t()) : launch(float()));
  // ddA_chunk[b,h,c] = exp(dA_cumsum[b,h,c,chunk-1]) * the sum of the eight partial dots
  const int64_t total = batch * nheads * d.C;
  hipLaunchKernelGGL(ssd_state_passing_bwd_finish_kernel, dim3((unsigned)((total + 255) / 256)), dim3(256), 0, st,
                     part, dA_cumsum + (chunk - 1), nheads * d.C * chunk, d.C * chunk, chunk, ddA_chunk, (int)nheads,
                     (int)d.C, 8, dinit ? 1 : 0, total, as_seq(nullptr, 0, 0), (int)seqlen, (int)chunk);
  return launched();
}

int ssd_chunk_state_bwd_db(const void* x, int64_t x_sb, int64_t x_sl, int64_t x_sh, int dtype,
                           const float* dt, const float* dA_cumsum, const void* dstates, int states_dtype,
                           const void* B, int64_t b_sb, int64_t b_sl, int64_t b_sg, float* dB, float* ddA_cumsum,
                           int64_t batch, int64_t seqlen, int64_t nheads, int64_t ngroups, int64_t hdim,
                           int64_t dstate, int64_t chunk, const int32_t* seq_idx, int64_t seq_sb, int64_t seq_sl,
                           void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  if (!dim_ok(hdim) || !dim_ok(dstate)) return SSD_ERR_UNSUPPORTED;
  SSD_TRY(check_vec(x, x_sb, x_sl, x_sh, dtype, hdim));
  if (!dB) return SSD_ERR_NULL;
  SSD_TRY(check_f32(dt));  // fetched in 16-byte pieces
  SSD_TRY(check_f32(dA_cumsum));
  SSD_TRY(check_state(dstates, states_dtype, dtype));
  if (B && !ddA_cumsum) return SSD_ERR_NULL;
  if (B) SSD_TRY(check_vec(B, b_sb, b_sl, b_sg, dtype, dstate));
  hipStream_t st = as_stream(stream);
  SSD_TRY(dispatch_tpn(dtype, hdim, dstate,
                       GroupLaunch<0>{x, Strides3{x_sb, x_sl, x_sh}, dstates, states_dtype, dt, dA_cumsum, B,
                                      Strides3{b_sb, b_sl, b_sg}, dB, ddA_cumsum, d,
                                      as_seq(seq_idx, seq_sb, seq_sl), st}));
  if (!B) return SSD_OK;
  return launch_row_cumsum(ddA_cumsum, chunk, batch * nheads * d.C, st);
}

int ssd_chunk_scan_bwd_dc(const void* dout, int64_t d_sb, int64_t d_sl, int64_t d_sh, int dtype,
                          const float* dA_cumsum, const void* prev_states, int states_dtype, const void* C,
                          int64_t c_sb,
                          int64_t c_sl, int64_t c_sg, float* dC, float* ddA_cumsum_prev, int64_t batch,
                          int64_t seqlen, int64_t nheads, int64_t ngroups, int64_t hdim, int64_t dstate,
                          int64_t chunk, const int32_t* seq_idx, int64_t seq_sb, int64_t seq_sl, void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  if (!dim_ok(hdim) || !dim_ok(dstate)) return SSD_ERR_UNSUPPORTED;
  SSD_TRY(check_vec(dout, d_sb, d_sl, d_sh, dtype, hdim));
  if (!dC) return SSD_ERR_NULL;
  SSD_TRY(check_f32(dA_cumsum));  // fetched in 16-byte pieces
  SSD_TRY(check_state(prev_states, states_dtype, dtype));
  if (C && !ddA_cumsum_prev) return SSD_ERR_NULL;
  if (C) SSD_TRY(check_vec(C, c_sb, c_sl, c_sg, dtype, dstate));
  return dispatch_tpn(dtype, hdim, dstate,
                      GroupLaunch<1>{dout, Strides3{d_sb, d_sl, d_sh}, prev_states, states_dtype, dA_cumsum, dA_cumsum,
                                     C,
                                     Strides3{c_sb, c_sl, c_sg}, dC, ddA_cumsum_prev, d,
                                     as_seq(seq_idx, seq_sb, seq_sl), as_stream(stream)});
}

int ssd_chunk_scan_chunk_state_bwd_dx(const float* cb, const void* x, int64_t x_sb, int64_t x_sl, int64_t x_sh,
                                      const void* dout, int64_t d_sb, int64_t d_sl, int64_t d_sh, int dtype,
                                      const float* dt, const float* dA_cumsum, const void* B, int64_t b_sb,
                                      int64_t b_sl, int64_t b_sg, const void* dstates, int states_dtype, const float* D,
                                      int d_has_hdim, void* dx, int64_t dx_sb, int64_t dx_sl, int64_t dx_sh,
                                      float* ddt, int64_t batch, int64_t seqlen, int64_t nheads,
                                      int64_t ngroups, int64_t hdim, int64_t dstate, int64_t chunk,
                                      const int32_t* seq_idx, int64_t seq_sb, int64_t seq_sl, float* dD_partial,
                                      void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  if (!dim_ok(hdim) || !dim_ok(dstate)) return SSD_ERR_UNSUPPORTED;
  if (dD_partial && !D) return SSD_ERR_NULL;
  if (dD_partial) SSD_TRY(check_f32(dD_partial));
  SSD_TRY(check_vec(x, x_sb, x_sl, x_sh, dtype, hdim));
  SSD_TRY(check_vec(dout, d_sb, d_sl, d_sh, dtype, hdim));
  SSD_TRY(check_vec(dx, dx_sb, dx_sl, dx_sh, dtype, hdim));
  SSD_TRY(check_vec(B, b_sb, b_sl, b_sg, dtype, dstate));
  if (!dt || !dA_cumsum || !ddt) return SSD_ERR_NULL;
  SSD_TRY(check_f32(cb));
  SSD_TRY(check_state(dstates, states_dtype, dtype));
  if (batch * d.C * nheads * ((chunk + 63) / 64) > 0x7fffffff) return SSD_ERR_SHAPE;
  return dispatch_tpn(dtype, hdim, dstate,
                      DxLaunch{cb, x, dout, B, Strides3{x_sb, x_sl, x_sh}, Strides3{d_sb, d_sl, d_sh},
                               Strides3{b_sb, b_sl, b_sg}, Strides3{dx_sb, dx_sl, dx_sh}, dt, dA_cumsum, dstates,
                               states_dtype, D,
                               d_has_hdim, dx, ddt, d, as_seq(seq_idx, seq_sb, seq_sl), dD_partial,
                               as_stream(stream)});
}

int64_t ssd_chunk_scan_chunk_state_bwd_dx_dD_slots(int dtype, int64_t hdim, int64_t dstate, int64_t chunk) {
  if (check_dtype(dtype) != SSD_OK || !dim_ok(hdim) || !dim_ok(dstate)) return 0;
  if (chunk <= 0 || chunk > 1024 || chunk % 4) return 0;
  return dispatch_tpn(dtype, hdim, dstate, DxSlots{chunk});
}

static size_t ddAcs_part_floats(const Dims& d) {
  const int64_t MT = (d.Q + ema::kBM - 1) / ema::kBM;
  return (size_t)(d.batch * d.nh * d.C * MT * d.Q);
}

size_t ssd_chunk_scan_bwd_ddAcs_workspace_bytes(int64_t batch, int64_t seqlen, int64_t nheads, int64_t chunk) {
  Dims d;
  if (check_dims(batch, seqlen, nheads, 1, 0, 0, chunk, &d) != SSD_OK) return 0;
  return (ddAcs_part_floats(d) + (size_t)(batch * nheads * d.C * chunk)) * sizeof(float);
}

int ssd_chunk_scan_bwd_ddAcs(const void* x, int64_t x_sb, int64_t x_sl, int64_t x_sh, const void* dout,
                             int64_t d_sb, int64_t d_sl, int64_t d_sh, int dtype, const float* dt,
                             const float* dA_cumsum, const float* cb, float* ddA_cumsum, void* workspace,
                             size_t workspace_bytes, int64_t batch, int64_t seqlen, int64_t nheads,
                             int64_t ngroups, int64_t hdim, int64_t chunk, void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, 0, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  if (hdim <= 0 || hdim > (1 << 16)) return SSD_ERR_SHAPE;
  SSD_TRY(check_vec(x, x_sb, x_sl, x_sh, dtype, hdim));
  SSD_TRY(check_vec(dout, d_sb, d_sl, d_sh, dtype, hdim));
  if (!dt || !dA_cumsum || !cb || !ddA_cumsum) return SSD_ERR_NULL;
  SSD_TRY(check_f32(workspace));
  if (workspace_bytes < ssd_chunk_scan_bwd_ddAcs_workspace_bytes(batch, seqlen, nheads, chunk)) return SSD_ERR_SHAPE;
  hipStream_t st = as_stream(stream);
  if ((chunk == 64 || chunk == 128 || chunk == 256) && dim_ok(hdim)) {
    // one workgroup per (b, c, h) does everything, prefix sum included
    const int64_t wgs = batch * nheads * d.C;
    if (wgs > 0x7fffffff) return SSD_ERR_SHAPE;
    const Strides3 sx{x_sb, x_sl, x_sh}, sd{d_sb, d_sl, d_sh};
    const int hpg = (int)(nheads / ngroups);
#define SSD_DDA_LAUNCH(T, P)                                                                                    \
  do {                                                                                                          \
    auto kernel = ssd_ddA_causal_kernel<T, P>;                                                                  \
    constexpr int smem = DdaSmem<T, P>::kBytes;                                                                 \
    SSD_TRY(allow_smem(kernel, smem));                                                                          \
    hipLaunchKernelGGL(kernel, dim3((unsigned)wgs), dim3(256), smem, st, (const T*)x, sx, (const T*)dout, sd,  \
                       dt, dA_cumsum, cb, ddA_cumsum, (int)nheads, hpg, (int)ngroups, (int)seqlen, (int)chunk,  \
                       (int)d.C);                                                                               \
  } while (0)
    if (dtype == SSD_BF16 && hdim == 64 && chunk == 256) {
      // The walk over the heads: where each has a compute unit to itself, and from where the other kernel, 768 of whose
      // workgroups run at once, needs a second turn, if the deal pays next to its turns.  The other kernel / the walk, us,
      // inputs in turn: 64 heads of all (batch, chunk) pairs 13.2 / 10.0, 256 15.3 / 12.7; 264 15.9 / 16.5, 512 19.1 / 19.4,
      // 640 20.5 / 22.6, 768 22.4 / 27.0; 800 30 / 27, 1024 34 / 29; 1280 36.3 / 37.1, 1536 40.6 / 43.3; 1568 47 / 41; 2272 of
      // sixteen 53 / 56, 2250 of ten 55 / 59; 3072 77 / 70, 8192 186 / 155.
      // Relative error against float64, the other kernel / the walk, A in [-16, -1], b1 nh32 L4096, mean of 12 seeds: dt =
      // softplus(n/2 - 2) 8.8e-7 / 7.6e-7, softplus(n/2) 1.23e-6 / 9.6e-7, softplus(n/2 + 2) 9.1e-7 / 9.4e-7.
      const HeadsDeal deal = heads_deal(batch * d.C * ngroups, hpg);
      const bool pays = wgs <= 256 || (wgs > 768 && heads_pay(deal, 38, 0, 16));
      if (pays && heads_vectors(dt, dA_cumsum) && reinterpret_cast<uintptr_t>(ddA_cumsum) % 16 == 0 && heads_rows(sx) && heads_rows(sd)) {
        constexpr int smem = DdaHeadsSmem::kBytes;
        static_assert(smem <= kLdsBytes, "the heads under way must fit the LDS of a compute unit");
        auto kernel = deal.splits ? ssd_ddA_heads_kernel<false> : ssd_ddA_heads_kernel<true>;
        SSD_TRY(allow_smem(kernel, smem));
        hipLaunchKernelGGL(kernel, dim3(deal.workgroups), dim3(512), smem, st, (const bf16_t*)x,
                           sx, (const bf16_t*)dout, sd, dt, dA_cumsum, cb, ddA_cumsum, (int)nheads, hpg, (int)ngroups,
                           (int)seqlen, (int)d.C, deal.units, deal.splits);
        return launched();
      }
    }
    if (dtype == SSD_BF16) {
      if (hdim == 64) SSD_DDA_LAUNCH(bf16_t, 64);
      else SSD_DDA_LAUNCH(bf16_t, 128);
    } else {
      if (hdim == 64) SSD_DDA_LAUNCH(float, 64);
      else SSD_DDA_LAUNCH(float, 128);
    }
#undef SSD_DDA_LAUNCH
    return launched();
  }
  float* part = static_cast<float*>(workspace);
  float* rowsum = part + ddAcs_part_floats(d);
  const int MT = (int)((d.Q + ema::kBM - 1) / ema::kBM);
  const int64_t grid = batch * nheads * d.C * MT;
  if (grid > 0x7fffffff) return SSD_ERR_SHAPE;
  const ema::SeqStrides sx{x_sb, x_sl, x_sh}, sd{d_sb, d_sl, d_sh};
  const int hpg = (int)(nheads / ngroups);
  if (dtype == SSD_BF16)
    hipLaunchKernelGGL((ema::da_gemm_kernel<bf16_t>), dim3((unsigned)grid), dim3(256), 0, st, (const bf16_t*)x, sx,
                       (const bf16_t*)dout, sd, dA_cumsum, part, rowsum, (int)nheads, (int)seqlen, (int)hdim,
                       (int)chunk, (int)d.C, MT, dt, cb, hpg, (int)ngroups);
  else
    hipLaunchKernelGGL((ema::da_gemm_kernel<float>), dim3((unsigned)grid), dim3(256), 0, st, (const float*)x, sx,
                       (const float*)dout, sd, dA_cumsum, part, rowsum, (int)nheads, (int)seqlen, (int)hdim,
                       (int)chunk, (int)d.C, MT, dt, cb, hpg, (int)ngroups);
  SSD_TRY(launched());
  const int64_t total = batch * nheads * d.C;
  hipLaunchKernelGGL(ema::da_finish_kernel<ema::kBM>, dim3((unsigned)((total + 3) / 4)), dim3(256), 0, st, part,
                     rowsum, (const float*)nullptr, 0, (const int*)nullptr, ddA_cumsum, (int)chunk, MT, total);
  return launched();
}

namespace {
// The states at the sequence ends in float32 or, with states_dtype bfloat16, rounded to it.
int varlen_states(const void* B, int64_t b_sl, int64_t b_sg, const void* x, int64_t x_sl, int64_t x_sh, int dtype,
                  const float* dt, const float* dA_cumsum, const void* chunk_states, int states_dtype,
                  const int32_t* cu_seqlens, void* states, int out_dtype, int64_t nseq, int64_t seqlen,
                  int64_t nheads, int64_t ngroups, int64_t hdim, int64_t dstate, int64_t chunk, void* stream) {
  Dims d;
  SSD_TRY(check_dims(1, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  if (nseq <= 0 || nseq > 65535 || hdim <= 0 || dstate <= 0 || hdim > 4096 || dstate > 4096) return SSD_ERR_SHAPE;
  if (states_dtype != SSD_F32 && states_dtype != dtype) return SSD_ERR_DTYPE;
  if (out_dtype != SSD_F32 && out_dtype != states_dtype) return SSD_ERR_DTYPE;
  if (!B || !x || !dt || !dA_cumsum || !chunk_states || !cu_seqlens || !states) return SSD_ERR_NULL;
  const int64_t tiles = ((hdim + 63) / 64) * ((dstate + 63) / 64);
  const dim3 grid((unsigned)tiles, (unsigned)nseq, (unsigned)nheads);
  const int hpg = (int)(nheads / ngroups);
  // The matrix kernel takes whole 64 x 64 tiles of the state and rows in 16-byte pieces; anything else is
  // multiplied out in float32.  So are float32 inputs where the workgroups fill the chip and the rows up to a sequence's
  // end, about half a chunk or the sequence, leave its stages of 64 rows mostly empty: the float32 matrix
  // instructions are no faster there and work for the padding.  Multiplied out / matrix, us, float32, 24 heads, 6000
  // positions: 1200 sequences hdim 64 dstate 64 chunk 64 273 / 319; 60 sequences hdim 128 dstate 128 chunk 64 67 / 77,
  // chunk 256 99 / 95; 6 sequences chunk 64 16.4 / 12.5 (bfloat16, 1200 sequences 387 / 313).
  const bool padded = dtype == SSD_F32 && tiles * nseq * nheads > 1024 && (seqlen / nseq < 64 || chunk / 2 < 64);
  const bool mma = !padded && hdim % 64 == 0 && dstate % 64 == 0 && check_vec(x, 0, x_sl, x_sh, dtype, hdim) == SSD_OK &&
                   check_vec(B, 0, b_sl, b_sg, dtype, dstate) == SSD_OK;
#define SSD_VARLEN_LAUNCH(T, TS, TO)                                                                                   \
  hipLaunchKernelGGL((mma ? ssd_chunk_state_varlen_mma_kernel<T, TS, TO> : ssd_chunk_state_varlen_kernel<T, TS, TO>),  \
                     grid, dim3(256), 0, as_stream(stream), (const T*)x, x_sl, x_sh, (const T*)B, b_sl, b_sg, dt,      \
                     dA_cumsum, (const TS*)chunk_states, cu_seqlens, (TO*)states, (int)seqlen, (int)nheads, hpg,       \
                     (int)hdim, (int)dstate, (int)chunk, (int)d.C)
  if (dtype != SSD_BF16) SSD_VARLEN_LAUNCH(float, float, float);
  else if (states_dtype != SSD_BF16) SSD_VARLEN_LAUNCH(bf16_t, float, float);
  else if (out_dtype == SSD_BF16) SSD_VARLEN_LAUNCH(bf16_t, bf16_t, bf16_t);
  else SSD_VARLEN_LAUNCH(bf16_t, bf16_t, float);
#undef SSD_VARLEN_LAUNCH
  return launched();
}
}  // namespace

int ssd_chunk_state_varlen(const void* B, int64_t b_sl, int64_t b_sg, const void* x, int64_t x_sl, int64_t x_sh,
                           int dtype, const float* dt, const float* dA_cumsum, const void* chunk_states,
                           int states_dtype, const int32_t* cu_seqlens, float* states, int64_t nseq, int64_t seqlen, int64_t nheads,
                           int64_t ngroups, int64_t hdim, int64_t dstate, int64_t chunk, void* stream) {
  return varlen_states(B, b_sl, b_sg, x, x_sl, x_sh, dtype, dt, dA_cumsum, chunk_states, states_dtype, cu_seqlens,
                       states, SSD_F32, nseq, seqlen, nheads, ngroups, hdim, dstate, chunk, stream);
}

int ssd_combined_fwd(const void* x, int64_t x_sb, int64_t x_sl, int64_t x_sh, int dtype, const void* dt, int dt_dtype,
                     int64_t dt_sb, int64_t dt_sl, int64_t dt_sh, const float* A, const float* dt_bias,
                     int dt_softplus, float dt_min, float dt_max, const void* B, int64_t b_sb, int64_t b_sl,
                     int64_t b_sg, const void* C, int64_t c_sb, int64_t c_sl, int64_t c_sg, const float* D,
                     int d_has_hdim, const void* z, int64_t z_sb, int64_t z_sl, int64_t z_sh, const float* initial,
                     const int32_t* seq_idx, int64_t seq_sb, int64_t seq_sl, const int32_t* cu_seqlens, int64_t nseq,
                     float* dt_out, float* dA_cumsum, float* local_states, void* states, float* final_states,
                     float* cb, void* out, int64_t o_sb, int64_t o_sl, int64_t o_sh, void* out_x, void* varlen_out,
                     int64_t batch, int64_t seqlen, int64_t nheads, int64_t ngroups, int64_t hdim, int64_t dstate,
                     int64_t chunk, void* stream) {
  // everything that a stage would refuse, before the first one is enqueued
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  SSD_TRY(check_dtype(dt_dtype));
  if (!dim_ok(hdim) || !dim_ok(dstate)) return SSD_ERR_UNSUPPORTED;
  // the walk knows no packed batches and takes whole 64-row stages
  if (!local_states && (seq_idx || chunk % 64)) return SSD_ERR_UNSUPPORTED;
  if (varlen_out && (batch != 1 || nseq <= 0 || nseq > 65535)) return SSD_ERR_SHAPE;
  if (varlen_out && !cu_seqlens) return SSD_ERR_NULL;
  if (!dt || !A) return SSD_ERR_NULL;
  SSD_TRY(check_vec(x, x_sb, x_sl, x_sh, dtype, hdim));
  SSD_TRY(check_vec(B, b_sb, b_sl, b_sg, dtype, dstate));
  SSD_TRY(check_vec(C, c_sb, c_sl, c_sg, dtype, dstate));
  SSD_TRY(check_vec(out, o_sb, o_sl, o_sh, dtype, hdim));
  if (z) SSD_TRY(check_vec(z, z_sb, z_sl, z_sh, dtype, hdim));
  if (out_x && reinterpret_cast<uintptr_t>(out_x) % 16) return SSD_ERR_ALIGN;
  for (const void* p : {(const void*)dt_out, (const void*)dA_cumsum, (const void*)states, (const void*)final_states, (const void*)cb})
    SSD_TRY(check_f32(p));
  if (local_states) SSD_TRY(check_f32(local_states));
  if (initial) SSD_TRY(check_f32(initial));
  const int64_t C_ = d.C, tiles = (chunk + 63) / 64;
  if (batch * C_ * nheads * tiles > 0x7fffffff || batch * C_ * (nheads + ngroups * tiles * tiles) > 0x7fffffff ||
      batch * nheads * ((hdim * dstate + 1023) / 1024) > 0x7fffffff)
    return SSD_ERR_SHAPE;
  // In one launch the blocks of C . B run with the registers of the states.  Of float32 states of hdim 128 those leave one
  // workgroup to a compute unit at dstate 128 (262 registers; C . B alone two) and three at dstate 64 (144; alone four), and
  // where there are many of both C . B is faster in a launch of its own.  The whole forward, us, apart / in one launch: dstate
  // 128, 256 heads of all (batch, chunk) pairs with 4096 blocks 312 / 321, with 16384 1099 / 1165, with 65536 1846 / 2157, 512
  // heads with 2048 218 / 218, 64 with 4096 213 / 187; dstate 64, 256 heads with 4096 248 / 241, with 16384 892 / 902, with 65536
  // 1357 / 1451, 2048 heads with 2048 235 / 235, with 8192 296 / 305.  Other types and sizes are level or gain.
  const bool apart = dtype == SSD_F32 && hdim == 128 && batch * C_ * nheads >= 256 &&
                     batch * C_ * ngroups * tiles * tiles >= (dstate == 128 ? 3584 : 8192);
  if (local_states) {
    if (apart) {
      SSD_TRY(ssd_chunk_cumsum_fwd(dt, dt_dtype, dt_sb, dt_sl, dt_sh, A, dt_bias, dA_cumsum, dt_out, batch, seqlen,
                                   nheads, chunk, dt_softplus, dt_min, dt_max, stream));
      SSD_TRY(ssd_chunk_state_fwd(B, b_sb, b_sl, b_sg, x, x_sb, x_sl, x_sh, dtype, dt_out, dA_cumsum, local_states,
                                  batch, seqlen, nheads, ngroups, hdim, dstate, chunk, seq_idx, seq_sb, seq_sl, stream));
    } else SSD_TRY(dispatch_tpn(dtype, hdim, dstate,
                         FrontLaunch{x, B, C, Strides3{x_sb, x_sl, x_sh}, Strides3{b_sb, b_sl, b_sg}, Strides3{c_sb, c_sl, c_sg},
                                     dt, dt_dtype, Strides3{dt_sb, dt_sl, dt_sh}, A, dt_bias, dA_cumsum, dt_out, dt_softplus,
                                     dt_min, dt_max, local_states, cb, d, as_seq(seq_idx, seq_sb, seq_sl), as_stream(stream)}));
    SSD_TRY(ssd_state_passing_fwd(local_states, dA_cumsum + (chunk - 1), nheads * C_ * chunk, C_ * chunk, chunk,
                                  initial, states, dtype, final_states, batch, C_, nheads, hdim * dstate, seq_idx,
                                  seq_sb, seq_sl, seqlen, chunk, stream));
  } else {
    SSD_TRY(ssd_chunk_cumsum_fwd(dt, dt_dtype, dt_sb, dt_sl, dt_sh, A, dt_bias, dA_cumsum, dt_out, batch, seqlen,
                                 nheads, chunk, dt_softplus, dt_min, dt_max, stream));
    SSD_TRY(ssd_chunk_state_passing_fwd(B, b_sb, b_sl, b_sg, x, x_sb, x_sl, x_sh, dtype, dt_out, dA_cumsum, initial,
                                        states, dtype, final_states, batch, seqlen, nheads, ngroups, hdim, dstate,
                                        chunk, stream));
  }
  if (!local_states || apart)  // (last: the chunk scan reads it next)
    SSD_TRY(ssd_bmm_chunk_fwd(C, c_sb, c_sl, c_sg, B, b_sb, b_sl, b_sg, dtype, cb, SSD_F32, batch, seqlen, ngroups,
                              dstate, chunk, seq_idx, seq_sb, seq_sl, stream));
  SSD_TRY(ssd_chunk_scan_fwd(cb, x, x_sb, x_sl, x_sh, z, z_sb, z_sl, z_sh, dtype, dt_out, dA_cumsum, C, c_sb, c_sl,
                             c_sg, states, dtype, D, d_has_hdim, out, o_sb, o_sl, o_sh, out_x, batch, seqlen, nheads,
                             ngroups, hdim, dstate, chunk, seq_idx, seq_sb, seq_sl, stream));
  if (!varlen_out) return SSD_OK;
  return varlen_states(B, b_sl, b_sg, x, x_sl, x_sh, dtype, dt_out, dA_cumsum, states, dtype, cu_seqlens, varlen_out,
                       dtype, nseq, seqlen, nheads, ngroups, hdim, dstate, chunk, stream);
}

#ifdef SSD_TIMING
// Development aid, only in builds with -DSSD_TIMING: installs the per-workgroup timestamp buffer.
int ssd_debug_set_timing(void* buf) {
  return hipMemcpyToSymbol(HIP_SYMBOL(ssd::g_ssd_timing), &buf, sizeof(buf)) == hipSuccess ? 0 : -6;
}
#endif

}  // extern "C"
