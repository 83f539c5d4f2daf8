// The chunk scan's entry point (include/ssd_hip.h) and its choice of kernel.  A translation unit of its own: the
// 256-row kernel for pairs of heads works at the register limit, and how many of its values the compiler spills
// depends on what else the unit holds (68 bytes per lane next to all the other stages, 8 here).
#include <type_traits>

#include "ssd_heads_kernels.h"
#include "ssd_host.h"

namespace {

struct ScanLaunch {
  const float* cb;
  const void *x, *z, *C;
  Strides3 sx, sz, sC, so;
  const float *dt, *dA;
  const void* prev;
  int prev_dtype;
  const float* D;
  int d_has_hdim;
  void *out, *out_x;
  Dims d;
  SeqIdx seq;
  hipStream_t st;
  template <typename T, int P, int N>
  int run() const {
    if constexpr (!std::is_same<T, float>::value)
      if (prev_dtype != SSD_F32) return run_as<T, P, N, T>();
    return run_as<T, P, N, float>();
  }
  template <typename T, int P, int N, typename TS, int HP>
  int launch_wide() const {
    auto kernel = ssd_chunk_scan_wide_kernel<T, P, N, TS, HP>;
    constexpr int smem = WideSmem<T, P * HP, N>::bytes_for(HP);
    SSD_TRY(allow_smem(kernel, smem));
    const int stiles = (int)(d.Q / 256);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.C * (d.nh / HP) * stiles)), dim3(256), smem, st, cb,
                       (const T*)x, sx, (const T*)z, sz, dt, dA, (const T*)C, sC, (const TS*)prev, D, d_has_hdim,
                       (T*)out, so, (T*)out_x, (int)d.nh, (int)(d.nh / d.g), (int)d.g, (int)d.L, (int)d.Q, (int)d.C,
                       stiles, seq);
    return launched();
  }
  template <typename T, int P, int N, typename TS, int HP, int ST>
  int launch_mid() const {
    auto kernel = ssd_chunk_scan_mid_kernel<T, P, N, TS, HP, ST>;
    constexpr int smem = MidSmem<T, P * HP, N, ST>::bytes_for(HP);
    static_assert(smem <= kLdsBytes, "the tile must fit the LDS of a compute unit");
    SSD_TRY(allow_smem(kernel, smem));
    hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.C * (d.nh / HP))), dim3(256), smem, st, cb,
                       (const T*)x, sx, (const T*)z, sz, dt, dA, (const T*)C, sC, (const TS*)prev, D, d_has_hdim,
                       (T*)out, so, (T*)out_x, (int)d.nh, (int)(d.nh / d.g), (int)d.g, (int)d.L, (int)d.C, seq);
    return launched();
  }
  // Whether a chunk's rows sit at 32-bit byte offsets from its first one.
  bool near(const Strides3& s) const { return forward_strides(s) && d.Q * s.sl < (int64_t(1) << 28); }
  // Chunks of 64 or 128 rows in one tile.  Two adjacent heads of a group per workgroup where they are adjacent
  // in memory too (dense heads of 64 features): they share the fragments of cb and the rows of C.  A single
  // bfloat16 head of 64 features leaves each wave one column block for the weights it forms, and the 64-row
  // kernel is the faster one (17 heads, L 4096, b2, chunk 128: 29.0 against 32.4 us); so it is while the workgroups
  // do not fill the chip.  The 64-row kernel / this one, us at dstate 128, inputs from memory:
  //   bfloat16 hdim 64, pairs   chunk 128: 64 pairs 8.0 / 9.6, 384 20.5 / 17.3, 512 27.5 / 18.8; b8 nh32 L8192 437 / 260
  //                             chunk 64: 384 pairs 10.0 / 11.3, 416 14.1 / 11.5; b8 nh32 L8192 334 / 240
  //   bfloat16 hdim 128         chunk 128: 384 20.9 / 17.4, 1024 51 / 39; chunk 64: 384 10.5 / 10.8, 576 16.8 / 13.9
  //   float32 chunk 128         hdim 64: 16 11.3 / 15.8, 128 14.8 / 17.1, 192 19.0 / 17.6, 1024 74 / 54; hdim 128:
  //                             128 20.4 / 24.4, 192 36 / 26 (two workgroups of 64 rows are the shorter chain while
  //                             both run at once); chunk 64: level up to 128, hdim 64 256 11.8 / 10.5, 1024 31 / 25
  template <typename T, int P, int N, typename TS, int ST>
  int launch_mid_pairs(bool* taken) const {
    *taken = true;
    if constexpr (sizeof(T) == 2) {
      constexpr int HP = P == 64 ? 2 : 1;
      const bool pairs = sx.sh == P && so.sh == P && (!z || sz.sh == P) && (d.nh / d.g) % 2 == 0;
      constexpr int64_t from = HP == 2 && ST == 64 ? kMidScanPairs64 : kMidWorkgroups;
      if ((HP == 1 || pairs) && d.batch * d.C * (d.nh / HP) >= from) return launch_mid<T, P, N, TS, HP, ST>();
      *taken = false;
      return SSD_OK;
    } else {
      if (ST == 64 || d.batch * d.C * d.nh > kBoth64Row) return launch_mid<T, P, N, TS, 1, ST>();
      *taken = false;
      return SSD_OK;
    }
  }
  template <int N, bool GATED>
  int launch_heads(const HeadsDeal& deal) const {
    auto kernel = deal.splits ? ssd_chunk_scan_heads_kernel<N, GATED, false> : ssd_chunk_scan_heads_kernel<N, GATED, true>;
    constexpr int smem = ScanHeadsSmem<N, GATED>::kBytes;
    static_assert(smem <= kLdsBytes, "the heads under way must fit the LDS of a compute unit");
    SSD_TRY(allow_smem(kernel, smem));
    hipLaunchKernelGGL(kernel, dim3(deal.workgroups), dim3(512), smem, st, cb, (const bf16_t*)x, sx,
                       (const bf16_t*)z, sz, dt, dA, (const bf16_t*)C, sC, (const bf16_t*)prev, D, (bf16_t*)out, so,
                       (bf16_t*)out_x, (int)d.nh, (int)(d.nh / d.g), (int)d.g, (int)d.L, (int)d.C, deal.units, deal.splits, seq);
    return launched();
  }
  template <typename T, int P, int N, typename TS>
  int run_as() const {
    if constexpr (std::is_same<T, bf16_t>::value && std::is_same<TS, bf16_t>::value && P == 64) {
      // The walk over the heads, from where a workgroup has two of them or a gate hides the fetch of what they share,
      // and groups have three heads or more.  The 256-row kernel / the walk, us, dstate 128: without gate 256 heads of
      // all (batch, chunk) pairs 14.7 / 16.2, 288 20.9 / 19.4, 512 23.2 / 21.3, 1536 57 / 41; 512 groups of two heads 44 / 53,
      // of three 66 / 62; with gate 16 heads 16.0 / 16.8, 64 16.9 / 17.2, 128 19.6 / 18.2, 256 22.4 / 19.1.  (The
      // header promises the same bits for states of either type up to these lines.)  And where its deal pays: 725 heads
      // in groups of five 28.2 / 31.5, 1860 of three 66 / 71, with gate 465 of five 28.5 / 30.6.
      const int64_t units = d.batch * d.C * d.nh;
      const HeadsDeal deal = heads_deal(d.batch * d.C * d.g, d.nh / d.g);
      const bool pays = units > (z ? 64 : 256) && d.nh / d.g >= 3 && heads_pay(deal, 44, 8, 28);
      if (d.Q == 256 && pays && !(D && d_has_hdim) && heads_vectors(dt, dA) && heads_rows(sx) && heads_rows(so) &&
          (!z || heads_rows(sz)))
        return z ? launch_heads<N, true>(deal) : launch_heads<N, false>(deal);
    }
    constexpr int wide_smem = WideSmem<T, P, N>::kBytes;
    if (d.Q % 256 == 0 && wide_smem <= kLdsBytes) {  // 256-row super-tiles, no barrier inside the k loop
      // Two adjacent heads of a group per workgroup where they are adjacent in memory too (dense
      // heads of 64 features): they share the fragments of cb and the rows of C.  Their first x tile
      // is read at 32-bit byte offsets; single heads take any stride.
      if constexpr (P == 64 && WideSmem<T, 128, N>::bytes_for(2) <= kLdsBytes / 2) {
        // Pairs take 256 registers, two workgroups per compute unit: with fewer than 512 of them most waves a
        // compute unit could hold are missing, and single heads (twice the workgroups) are faster.  Pairs /
        // single heads, us, with gate, nh32 dstate 128 chunk 256: L2048 29.0 / 18.9, L4096 37.3 / 30.7, L8192
        // (512 pairs) 47.5 / 57.6.
        const bool dense = sx.sh == P && so.sh == P && (!z || sz.sh == P);
        const bool offsets32 = sx.sl >= 0 && sx.sl <= (int64_t(1) << 32) / (256 * (int64_t)sizeof(T));
        if (dense && offsets32 && (d.nh / d.g) % 2 == 0 && d.batch * d.C * (d.nh / 2) * (d.Q / 256) >= 512)
          return launch_wide<T, P, N, TS, 2>();
      }
      return launch_wide<T, P, N, TS, 1>();
    }
    const bool close = near(sx) && near(sC) && near(so) && (!z || near(sz));
    if ((d.Q == 64 || d.Q == 128) && close) {
      bool taken;
      const int status = d.Q == 128 ? launch_mid_pairs<T, P, N, TS, 128>(&taken) : launch_mid_pairs<T, P, N, TS, 64>(&taken);
      if (taken) return status;
    }
    auto kernel = ssd_chunk_scan_kernel<T, P, N, TS>;
    constexpr int smem = ScanSmem<T, P, N>::kBytes;
    SSD_TRY(allow_smem(kernel, smem));
    const int mtiles = (int)((d.Q + 63) / 64);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(d.batch * d.C * d.nh * mtiles)), dim3(256), smem, st, cb,
                       (const T*)x, sx, (const T*)z, sz, dt, dA, (const T*)C, sC, (const TS*)prev, D, d_has_hdim,
                       (T*)out, so, (T*)out_x, (int)d.nh, (int)(d.nh / d.g), (int)d.g, (int)d.L, (int)d.Q, (int)d.C, mtiles,
                       seq);
    return launched();
  }
};

}  // namespace

extern "C" {

int ssd_chunk_scan_fwd(const float* cb, const void* x, int64_t x_sb, int64_t x_sl, int64_t x_sh,
                       const void* z, int64_t z_sb, int64_t z_sl, int64_t z_sh, int dtype,
                       const float* dt, const float* dA_cumsum, const void* C, int64_t c_sb, int64_t c_sl,
                       int64_t c_sg, const void* prev_states, int states_dtype, const float* D, int d_has_hdim,
                       void* out, int64_t o_sb, int64_t o_sl, int64_t o_sh, void* out_x, int64_t batch,
                       int64_t seqlen, int64_t nheads, int64_t ngroups, int64_t hdim, int64_t dstate,
                       int64_t chunk, const int32_t* seq_idx, int64_t seq_sb, int64_t seq_sl, void* stream) {
  Dims d;
  SSD_TRY(check_dims(batch, seqlen, nheads, ngroups, hdim, dstate, chunk, &d));
  SSD_TRY(check_dtype(dtype));
  if (!dim_ok(hdim) || !dim_ok(dstate)) return SSD_ERR_UNSUPPORTED;
  SSD_TRY(check_vec(x, x_sb, x_sl, x_sh, dtype, hdim));
  SSD_TRY(check_vec(out, o_sb, o_sl, o_sh, dtype, hdim));
  SSD_TRY(check_vec(C, c_sb, c_sl, c_sg, dtype, dstate));
  if (z) SSD_TRY(check_vec(z, z_sb, z_sl, z_sh, dtype, hdim));
  if (out_x && reinterpret_cast<uintptr_t>(out_x) % 16) return SSD_ERR_ALIGN;
  if (!dt || !dA_cumsum) return SSD_ERR_NULL;
  SSD_TRY(check_f32(cb));
  SSD_TRY(check_state(prev_states, states_dtype, dtype));
  if (batch * d.C * nheads * ((chunk + 63) / 64) > 0x7fffffff) return SSD_ERR_SHAPE;
  return dispatch_tpn(dtype, hdim, dstate,
                      ScanLaunch{cb, x, z, C, Strides3{x_sb, x_sl, x_sh}, Strides3{z_sb, z_sl, z_sh},
                                 Strides3{c_sb, c_sl, c_sg}, Strides3{o_sb, o_sl, o_sh}, dt, dA_cumsum,
                                 prev_states, states_dtype, D, d_has_hdim, out, out_x, d,
                                 as_seq(seq_idx, seq_sb, seq_sl),
                                 as_stream(stream)});
}

}  // extern "C"
