// Kernels of the Mamba-2 SSD stages that walk the heads of a group (gfx950, wave64): bfloat16, hdim 64, chunks of
// 256 rows.
//
// What a (batch, chunk, group) shares between its heads stays in registers for the whole walk: each of eight waves
// owns two strips of 16 rows, the pieces of cb that belong to them (96 registers) and, where the stage needs them, their
// rows of B or C.  What belongs to one head arrives by copies from global memory straight into LDS, one to two heads
// ahead, so that a head costs its own bytes and one barrier, and no load waits inside it.  A workgroup is alone on its
// compute unit.  (Strips, not blocks of 32 rows: those would take 128 registers of cb next to 64 of operands and
// accumulators, which spills.)
//
// The per-head kernels these stand beside fetch cb and the rows of B / C once per head or pair of heads, a fragment at a
// time, and wait for each.  Here a head's copies alone run at 5.0 to 5.2 TB/s; what keeps the kernels from that is the
// serial chain of a head (copies landed, factors, products, sums) at two waves per SIMD.  Times below are us by the kernel
// of one head or pair and here, at b8 nh32 L8192 dstate 128 of the three walks one after another on inputs in turn, the
// others of a kernel by itself.
#pragma once
#include "ssd_kernels.h"

namespace ssd {

using ema::floatx4;
typedef unsigned u32x2_t __attribute__((ext_vector_type(2)));

// 16 x 16 blocks of a product, 32 contraction steps at once: lane l holds steps 8 (l / 16) .. of row or column l % 16 of
// either operand, register v of the result is row 4 (l / 16) + v of column l % 16.
__device__ __forceinline__ void mma16(const Vec16<bf16_t>& a, const Vec16<bf16_t>& b, floatx4& acc) {
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a.raw, b.raw, acc, 0, 0, 0);
}

// The lowest value of this lane and those before it.
__device__ __forceinline__ float running_min(float v) {
  auto with = [](float v, int other) { return fminf(v, __int_as_float(other)); };
  auto bits = [](float v) { return __float_as_int(v); };
  v = with(v, __builtin_amdgcn_update_dpp(bits(v), bits(v), 0x111, 0xf, 0xf, false));  // row_shr:1
  v = with(v, __builtin_amdgcn_update_dpp(bits(v), bits(v), 0x112, 0xf, 0xf, false));
  v = with(v, __builtin_amdgcn_update_dpp(bits(v), bits(v), 0x114, 0xf, 0xf, false));
  v = with(v, __builtin_amdgcn_update_dpp(bits(v), bits(v), 0x118, 0xf, 0xf, false));
  v = with(v, __builtin_amdgcn_update_dpp(bits(v), bits(v), 0x142, 0xa, 0xf, false));  // row_bcast:15 into rows 1 and 3
  v = with(v, __builtin_amdgcn_update_dpp(bits(v), bits(v), 0x143, 0xc, 0xf, false));  // row_bcast:31 into rows 2 and 3
  return v;
}

struct HeadsTile {
  static constexpr int Q = 256, P = 64;                      // rows of a chunk, features of a head
  static constexpr int kRows = Q * P * (int)sizeof(bf16_t);  // a head's rows of x, dout or z
  static constexpr int kVec = 2 * Q * (int)sizeof(float);    // its dA and dt
  // Strips of 16 rows of a wave: w and 15 - w.  Along the causal triangle they have 9 pieces of 16 x 32 together,
  // whatever w.
  static __device__ __forceinline__ int strip(int wave, int i) { return i == 0 ? wave : 15 - wave; }
  // Factors of the positions: a wave's strips see 288 of them together.
  static constexpr int kFactors = 8 * 288 * (int)sizeof(float);

  // Rows of 128 bytes in LDS that are read both transposed (per half wave 32 adjacent bytes of rows r .. r + 3 and
  // r + 8 .. r + 11) and a row per lane: piece j of 16 bytes of row r sits in slot j ^ key(r), which spreads either over
  // the whole bank period of 256 bytes.
  static __device__ __forceinline__ int key(int r) { return (r & 2) | ((r >> 1) & 4) | ((r >> 2) & 1); }

  // Copies 8 * COPIES rows of a tensor, row0 .. of the chunk, to dst (128 bytes a row, pieces placed by key); rows at
  // or past `limit` repeat the last one.  row0 is a multiple of 8.
  template <int COPIES>
  static __device__ __forceinline__ void copy_rows(const bf16_t* g, int row_stride, int row0, int limit,
                                                   unsigned char* dst, int lane) {
#pragma unroll
    for (int j = 0; j < COPIES; ++j) {
      const int r = lane >> 3, r0 = min(row0 + 8 * j, limit - 1);
      const unsigned at = __umul24((unsigned)min(r, limit - 1 - r0), (unsigned)row_stride * 2u) + 16u * ((lane & 7) ^ key(row0 + 8 * j + r));
      copy16_to_lds(g + (int64_t)r0 * row_stride, at, dst + j * 1024);
    }
  }

  // Whether dA falls along the chunk as far as this lane's four positions (a; `next` is the one behind them) tell, and
  // is finite: what is past the sequence does not count.  ROUNDED, for weights that are rounded to bfloat16 (2^-9): up to
  // 2^-11 above the lowest value so far still falls.  Where steps of 0 lie among the others a sum over the lanes rises by
  // its rounding in most chunks (10 % of the steps: in 82 %), and taking those as they are defined costs ddA 171 -> 214 us.
  template <bool ROUNDED>
  static __device__ __forceinline__ bool falls(const float4& a, float next, int lane, int limit) {
    constexpr float kRise = ROUNDED ? 0x1p-13f : 0.f;  // (of a step within the lane, and from the lowest of all before it)
    auto step = [](float x, float y) { return y <= x + kRise; };  // (not met by a NaN)
    const float low = ROUNDED ? running_min(fminf(fminf(a.x, a.y), fminf(a.z, a.w))) : a.w;
    if (limit == Q)  // (no short circuits: they would be branches)
      return step(a.x, a.y) & step(a.y, a.z) & step(a.z, a.w) & step(low, next) & (fabsf(a.x) < 1e30f) & (fabsf(a.w) < 1e30f);
    const float v[4] = {a.x, a.y, a.z, low}, w[4] = {a.y, a.z, a.w, next};
    bool r = (4 * lane >= limit) | (fabsf(a.x) < 1e30f);
#pragma unroll
    for (int i = 0; i < 4; ++i) r &= (4 * lane + i + 1 >= limit) | (step(v[i], w[i]) & (fabsf(w[i]) < 1e30f));
    return r;
  }

  // dt of this lane's four positions, 0 past the sequence whatever dt holds there.
  static __device__ __forceinline__ float4 weights_of_time(const float* dts, int lane, int limit) {
    const float4 t = *reinterpret_cast<const float4*>(dts + 4 * lane);
    if (limit == Q) return t;
    const int left = limit - 4 * lane;
    return make_float4(left > 0 ? t.x : 0.f, left > 1 ? t.y : 0.f, left > 2 ? t.z : 0.f, left > 3 ? t.w : 0.f);
  }
  static __device__ __forceinline__ bool finite(const float4& t) {
    return (fabsf(t.x) < 1e30f) & (fabsf(t.y) < 1e30f) & (fabsf(t.z) < 1e30f) & (fabsf(t.w) < 1e30f);
  }

  // The transposed operand: features 16 pb + l % 16 of positions 8 (l / 16) .. + 7 of 32, by two transposing reads (each
  // group of 16 lanes reads four rows of 16 features).
  struct Transposed {
    int lo, hi, flip;  // (elements)
    __device__ __forceinline__ explicit Transposed(int lane) {
      const int i16 = lane & 15, row = 8 * (lane >> 4) + (i16 >> 2), piece = (i16 & 3) >> 1;
      lo = row * P + 8 * (piece ^ (key(row) & 1)) + 4 * (i16 & 1);
      hi = (row + 4) * P + 8 * (piece ^ (key(row + 4) & 1)) + 4 * (i16 & 1);
      flip = 8 * (key(row) & 6);  // (the same for both: rows four apart differ in bit 0 of the key)
    }
    __device__ __forceinline__ Vec16<bf16_t> read(const bf16_t* tile, int pb) const {
      typedef __attribute__((address_space(3))) ema::bf16x4 lds_bf16x4;
      const int f = (16 * pb) ^ flip;
      const ema::bf16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(tile + lo + f));
      const ema::bf16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)(tile + hi + f));
      Vec16<bf16_t> r;
      r.raw = __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7);
      return r;
    }
  };
};

// A workgroup's share of the heads of all (batch, chunk, group) sets; a unit is one head, those of a set in a row.  Either
// each set is dealt to `splits` workgroups of its own, or all units evenly (EVEN, see heads_deal): a workgroup that never
// changes its set keeps everything that belongs to the set out of the loop (chunk scan, 256 sets of 32: 168 against 188 us).
// Within a set the heads are taken in turn from one that differs from workgroup to workgroup: the rows of a head are a part
// of each row of the tensors, and workgroups that walked the heads in step would all fetch from the same part of the memory
// channels at a time.
template <bool EVEN>
struct HeadsWalk {
  int unit, end, seed;       // the unit under way and the one past the last
  int per, ngroups, C;       // heads of a group
  int first, count, turn, k;  // the set's heads that are the workgroup's, the one it begins with, how many are done
  int g, c, b;
  __device__ __forceinline__ HeadsWalk(int wg, int wgs, int units, int splits, int per_, int ngroups_, int C_)
      : seed(5 * wg), per(per_), ngroups(ngroups_), C(C_) {
    const int set = EVEN ? 0 : wg / splits, part = EVEN ? wg : wg - set * splits, parts = EVEN ? wgs : splits;
    const int64_t dealt = EVEN ? units : per;
    unit = __builtin_amdgcn_readfirstlane(set * per + (int)(dealt * part / parts));
    end = __builtin_amdgcn_readfirstlane(set * per + (int)(dealt * (part + 1) / parts));
    open();
  }
  __device__ __forceinline__ void open() {
    auto scalar = [](int v) { return __builtin_amdgcn_readfirstlane(v); };  // (quotients are formed in vector registers)
    const int set = scalar(unit / per);
    first = unit - set * per;
    count = min(per - first, end - unit);
    turn = scalar(seed % count);
    k = 0;
    const int chunk = scalar(set / ngroups);
    g = set - chunk * ngroups;
    b = scalar(chunk / C);
    c = chunk - b * C;
  }
  __device__ __forceinline__ bool done() const { return unit >= end; }
  __device__ __forceinline__ int head() const {  // of the tensor
    const int h = k + turn;
    return g * per + first + (h < count ? h : h - count);
  }
  __device__ __forceinline__ void next() {
    ++unit, ++k;
    if (EVEN && k == count && !done()) open();
  }
};

__device__ __forceinline__ void load8(float* r, const float* p) {
  const float4 a = *reinterpret_cast<const float4*>(p), b = *reinterpret_cast<const float4*>(p + 4);
  r[0] = a.x, r[1] = a.y, r[2] = a.z, r[3] = a.w, r[4] = b.x, r[5] = b.y, r[6] = b.z, r[7] = b.w;
}

// Waits until at most n of the wave's requests (copies, stores) are outstanding, n the same for the whole wave: the
// first of the listed counts (falling) that n allows, or none.
template <int FIRST, int... REST>
__device__ __forceinline__ void wait_outstanding(int n) {
  if (n >= FIRST) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(FIRST) : "memory");
  else if constexpr (sizeof...(REST) > 0) wait_outstanding<REST...>(n);
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Two blocks of 16 features of a row in the accumulator layout (a lane holds four adjacent ones of each, the four
// groups of 16 lanes four apart) as 16 adjacent bytes per lane: lane group q receives features 8 (q / 2) .. + 7 of block
// q % 2.
__device__ __forceinline__ Vec16<bf16_t> join_quads(const floatx4& a, const floatx4& b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef bf16_t b16x2 __attribute__((ext_vector_type(2)));
  typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
  auto pack = [](float x, float y) {
    const f32x2 p = {x, y};
    return __builtin_bit_cast(unsigned, __builtin_convertvector(p, b16x2));
  };
  const u32x2_t s0 = __builtin_amdgcn_permlane16_swap(pack(a[0], a[1]), pack(b[0], b[1]), false, false);
  const u32x2_t s1 = __builtin_amdgcn_permlane16_swap(pack(a[2], a[3]), pack(b[2], b[3]), false, false);
  const u32x4 q = {s0[0], s1[0], s0[1], s1[1]};
  Vec16<bf16_t> r;
  r.raw = __builtin_bit_cast(ema::bf16x8, q);
  return r;
}

// The 128-byte rows of a strip, lane (l16, q) holding piece `lo` of the first half of row l16 and piece `hi` of the
// second (join_quads), stored eight whole rows at a time: the lanes 8 .. 15 of each group trade their first half for the
// second half of the row eight above.  at(r): byte offset of this lane's piece in row r of the strip; rows at or past
// `rows` are left out.
template <typename F>
__device__ __forceinline__ void store_strip(bf16_t* g, const Vec16<bf16_t>& lo, const Vec16<bf16_t>& hi, int l16,
                                            int rows, F at) {
  typedef int i32x4 __attribute__((ext_vector_type(4)));
  const bool upper = l16 >= 8;
  const i32x4 a = __builtin_bit_cast(i32x4, lo.raw), b = __builtin_bit_cast(i32x4, hi.raw);
  i32x4 first, second;
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int t = __builtin_amdgcn_update_dpp(0, upper ? a[k] : b[k], 0x128, 0xf, 0xf, false);  // row_ror:8
    first[k] = upper ? t : a[k];
    second[k] = upper ? b[k] : t;
  }
  Vec16<bf16_t> o;
  const int r = l16 & 7;
  o.raw = __builtin_bit_cast(ema::bf16x8, first);
  if (r < rows) store16_stream(at_bytes(g, at(r)), o);
  o.raw = __builtin_bit_cast(ema::bf16x8, second);
  if (r + 8 < rows) store16_stream(at_bytes(g, at(r + 8)), o);
}

// ------------------------------------------------------------------------------------
// chunk_scan (ssd_chunk_scan_kernel).  b8 nh32 L8192 295 -> 185 (4.0 TB/s of its 742 MB), by itself 244 -> 168 (406 -> 283
// with gate and out_x), b4 nh24 L8192 95 -> 68, b1 nh32 L4096 23.2 -> 21.2 (gate 31 -> 27).  On the way, by itself:
// 230 with heads in step and rows stored in 64-byte halves, 195 with the heads in turn, 184 with whole rows stored, 165 with a
// piece's LDS reads ahead of the products of the one before.  Of the 185, the copies and stores alone take 150 and the rest
// alone 128.
// ------------------------------------------------------------------------------------
template <int N, bool GATED>
struct ScanHeadsSmem : HeadsTile {
  static constexpr int R = GATED ? 2 : 3;  // heads in LDS
  static constexpr int kState = P * N * (int)sizeof(bf16_t);
  static constexpr int kHead = kRows + kState + kVec;
  static constexpr int kBytes = R * kHead + kFactors + (GATED ? kRows : 0);
};

template <int N, bool GATED, bool EVEN>
__global__ __launch_bounds__(512, 2) void ssd_chunk_scan_heads_kernel(
    const float* __restrict__ cb, const bf16_t* __restrict__ x, Strides3 sx, const bf16_t* __restrict__ z, Strides3 sz,
    const float* __restrict__ dt, const float* __restrict__ dA_cs, const bf16_t* __restrict__ Cm, Strides3 sC,
    const bf16_t* __restrict__ prev, const float* __restrict__ D, bf16_t* __restrict__ out, Strides3 so,
    bf16_t* __restrict__ out_x, int nh, int heads_per_group, int ngroups, int L, int C, int units, int splits, SeqIdx seq) {
  using S = ScanHeadsSmem<N, GATED>;
  using T = bf16_t;
  constexpr int P = S::P, Q = S::Q, R = S::R, NK = N / 32;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  HeadsWalk<EVEN> now(xcd_local_index((int)blockIdx.x, (int)gridDim.x), (int)gridDim.x, units, splits, heads_per_group, ngroups, C);
  HeadsWalk<EVEN> ahead = now;  // the head whose copies are requested next
  // the wave's strips of rows, their pieces of 32 positions up to the diagonal, their factors of the positions
  int r0[2], steps[2];
  float* fk[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) r0[j] = 16 * S::strip(wave, j), steps[j] = (r0[j] >> 5) + 1;
  fk[1] = reinterpret_cast<float*>(smem + R * S::kHead) + wave * 288;
  fk[0] = fk[1] + 32 * steps[1];
  unsigned char* gate = smem + R * S::kHead + S::kFactors + wave * (32 * P * (int)sizeof(T));

  // ---- the copies of a head: four of its rows per wave and instruction, its state, dA and dt.  What depends on the
  // lane is formed anew for each head (from `ln`, which the compiler cannot follow through the loop): the registers
  // are taken by what the heads share.
  constexpr int kXCopies = 4, kSCopies = S::kState / 8192, kCopies = kXCopies + kSCopies, kZCopies = 4;
  static_assert(8 * 8 * kXCopies == Q && 8 * 1024 * kSCopies == S::kState, "eight waves bring a head");
  constexpr int SP = N / 8;  // pieces of a row of the state
  auto state_key = [](int r) { return N == 128 ? r & 15 : (r >> 1) & 7; };
  auto vec_at = [&](const HeadsWalk<EVEN>& w) { return (((int64_t)w.b * nh + w.head()) * C + w.c) * Q; };
  auto request = [&](int u, int ln) {  // the copies of the head ahead into place u
    const HeadsWalk<EVEN>& w = ahead;
    const int h = w.head();
    unsigned char* base = smem + u * S::kHead;
    S::template copy_rows<kXCopies>(x + w.b * sx.sb + (int64_t)w.c * Q * sx.sl + h * sx.sh, (int)sx.sl, 32 * wave,
                                    min(Q, L - w.c * Q), base + kXCopies * wave * 1024, ln);
    const T* sg = prev + (((int64_t)w.b * C + w.c) * nh + h) * (P * N);
    const int r = ln / SP;  // row of the state within an instruction's
#pragma unroll
    for (int j = 0; j < kSCopies; ++j) {
      const int row0 = (kSCopies * wave + j) * (64 / SP);
      copy16_to_lds(sg + row0 * N, (unsigned)(r * N + 8 * ((ln % SP) ^ state_key(row0 + r))) * (unsigned)sizeof(T),
                    base + S::kRows + (kSCopies * wave + j) * 1024);
    }
    if (wave < 2)
      copy16_to_lds((wave == 0 ? dA_cs : dt) + vec_at(w), 16u * (unsigned)ln, base + S::kRows + S::kState + wave * 1024);
    ahead.next();
  };
  request(0, lane);
  if (R == 3 && !ahead.done()) request(1, lane);

  // What the heads of a set share: the rows of C, and of cb from the first position on (entries past the diagonal zero).
  // Waited for where they are loaded: no other wait for ordinary loads falls into the loop.
  Vec16<T> cf[2][NK];
  float cb0[4][8], cb1[8][8];
  bool live[2];
  int limit = 0, stores = 0;
  auto load_shared = [&]() {
    int ln = lane;
    asm volatile("" : "+v"(ln));
    limit = min(Q, L - now.c * Q);
    // stores of a head that can still be outstanding (a ragged chunk leaves some out: none are allowed for)
    stores = limit < Q ? 0 : GATED && out_x ? 8 : 4;
    const ChunkSeq sq = chunk_seq(seq, now.b, now.c, Q);
    const int e0 = 8 * (ln >> 4);
    const T* Cg = Cm + now.b * sC.sb + (int64_t)now.c * Q * sC.sl + now.g * sC.sh + e0;
    const float* cbg = cb + (((int64_t)now.b * C + now.c) * ngroups + now.g) * (Q * Q);
    auto load_cb = [&](float* w, const float* row, int k, int m) {
      const float4 lo = *reinterpret_cast<const float4*>(row + k), hi = *reinterpret_cast<const float4*>(row + k + 4);
      w[0] = lo.x, w[1] = lo.y, w[2] = lo.z, w[3] = lo.w, w[4] = hi.x, w[5] = hi.y, w[6] = hi.z, w[7] = hi.w;
#pragma unroll
      for (int e = 0; e < 8; ++e) w[e] = k + e0 + e > m ? 0.f : w[e];
    };
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int m = r0[j] + (ln & 15);
      const T* crow = Cg + (int64_t)min(m, limit - 1) * sC.sl;
#pragma unroll
      for (int i = 0; i < NK; ++i) cf[j][i] = load16(crow + 32 * i);
      live[j] = !sq.on() || sq.at(min(m, limit - 1)) == sq.entering(now.c);
      // (pieces past the diagonal are inside the chunk's block of cb too, and cleared by the mask)
      const float* cbrow = cbg + (int64_t)m * Q + e0;
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        if (j == 1) load_cb(cb1[t], cbrow, 32 * t, m);
        else if (t < 4) load_cb(cb0[t], cbrow, 32 * t, m);
      }
    }
#pragma unroll
    for (int i = 0; i < NK; ++i) asm volatile("" : "+v"(cf[0][i].raw), "+v"(cf[1][i].raw));
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        asm volatile("" : "+v"(cb1[t][e]));
        if (t < 4) asm volatile("" : "+v"(cb0[t][e]));
      }
  };

  if (!EVEN) load_shared();
  for (int u = 0; !now.done(); now.next(), u = u + 1 < R ? u + 1 : 0) {
    if (EVEN && now.k == 0) load_shared();
    const int64_t b = now.b;
    const int c = now.c, h = now.head();
    const bool more = now.unit + R - 1 < now.end;
    // a head's copies have landed once only what was requested behind them is outstanding: the copies of the next
    // head (R = 3) and the stores of the heads in between
    if constexpr (R == 3) {
      wait_outstanding<kCopies + 8, kCopies + 4, 8, kCopies, 4>((now.unit + 1 < now.end ? kCopies : 0) + stores * min(now.k, 2));
    } else {
      wait_outstanding<8, 4>(now.k > 0 ? stores : 0);
    }
    __syncthreads();  // every wave's part of the head is there; every wave is done with the head before
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int l16 = ln & 15, quad = ln >> 4;
    const HeadsTile::Transposed tr(ln);
    if constexpr (GATED)  // the wave's own rows of the gate
#pragma unroll
      for (int j = 0; j < 2; ++j)
        S::template copy_rows<kZCopies / 2>(z + b * sz.sb + (int64_t)c * Q * sz.sl + h * sz.sh, (int)sz.sl, r0[j], limit, gate + j * 2048, ln);
    if (more) request(u > 0 ? u - 1 : R - 1, ln);  // (the place of the head before)
    const unsigned char* base = smem + u * S::kHead;
    const T* Xs = reinterpret_cast<const T*>(base);
    const float* dAs = reinterpret_cast<const float*>(base + S::kRows + S::kState);
    const float* dts = dAs + Q;

    // The weight of (m, k) is cb times exp(dA_m - dA_k) dt_k.  Where dA falls along the chunk the decay is split at
    // the middle r of the strip of rows into a factor of k and one of the row, which is left for the end: one product
    // per weight.  Positions below the strip have factors of at most 1; those inside it stay within e^40 both ways,
    // or the strip's last piece takes its weights as they are defined.  Where dA rises anywhere all pieces do, the
    // exponent clamped at 0.
    const float4 ak = *reinterpret_cast<const float4*>(dAs + 4 * ln);
    const float4 tk = S::weights_of_time(dts, ln, limit);
    const float an = dAs[min(4 * ln + 4, Q - 1)];
    const bool split = __builtin_amdgcn_ballot_w64(S::template falls<true>(ak, an, ln, limit) & S::finite(tk)) == ~0ull;
    float am[2], ar[2];
    bool narrow[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      am[j] = dAs[r0[j] + l16];
      const float a0 = dAs[r0[j]], a1 = dAs[min(r0[j] + 7, limit - 1)], a2 = dAs[min(r0[j] + 15, limit - 1)];
      narrow[j] = __builtin_amdgcn_readfirstlane(a0 - a1 <= 40.f && a1 - a2 <= 40.f);
      ar[j] = narrow[j] ? a1 : a0;
      const float4 f = make_float4(__expf(fminf(ar[j] - ak.x, 40.f)) * tk.x, __expf(fminf(ar[j] - ak.y, 40.f)) * tk.y,
                                   __expf(fminf(ar[j] - ak.z, 40.f)) * tk.z, __expf(fminf(ar[j] - ak.w, 40.f)) * tk.w);
      if (4 * ln < 32 * steps[j]) *reinterpret_cast<float4*>(fk[j] + 4 * ln) = f;
    }
    // ---- state . C, features in the rows of the product: a lane's values belong to its row of each strip
    floatx4 acc[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) acc[j][pb] = floatx4{0.f, 0.f, 0.f, 0.f};
    // (rows of the state start at multiples of their length: the piece is chosen by flipping bits of the address)
    const unsigned piece0 = u * S::kHead + S::kRows + (l16 * N + 8 * (quad ^ state_key(l16))) * sizeof(T);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) {
        const Vec16<T> sf = load16(reinterpret_cast<const T*>(smem + (piece0 ^ (64u * ks)) + 16 * pb * N * sizeof(T)));
        mma16(sf, cf[0][ks], acc[0][pb]);
        mma16(sf, cf[1][ks], acc[1][pb]);
      }
    float scale[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float enter = live[j] ? __expf(split ? ar[j] : am[j]) : 0.f;
      scale[j] = split ? __expf(am[j] - ar[j]) : 1.f;
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) acc[j][pb] *= enter;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // the wave's own factors are visible to its own reads

    // ---- the causal sum
    if (split) {
      // what a piece needs from LDS, requested a piece ahead
      struct Piece {
        Vec16<T> xf[4];
        float4 f1[2], f0[2];
      };
      auto fetch = [&](Piece& p, int t) {
#pragma unroll
        for (int k = 0; k < 2; ++k) p.f1[k] = *reinterpret_cast<const float4*>(fk[1] + 32 * t + 8 * quad + 4 * k);
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) p.xf[pb] = tr.read(Xs + 32 * t * P, pb);
        if (t < 4)
#pragma unroll
          for (int k = 0; k < 2; ++k) p.f0[k] = *reinterpret_cast<const float4*>(fk[0] + 32 * t + 8 * quad + 4 * k);
      };
      auto weights = [&](const float* w, const float4* f) {
        const float t[8] = {w[0] * f[0].x, w[1] * f[0].y, w[2] * f[0].z, w[3] * f[0].w,
                            w[4] * f[1].x, w[5] * f[1].y, w[6] * f[1].z, w[7] * f[1].w};
        Vec16<T> wf;
        wf.set_all(t);
        return wf;
      };
      const int end0 = steps[0] - !narrow[0], end1 = steps[1] - !narrow[1];
      Piece piece[2];
      fetch(piece[0], 0);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        if (t >= 4 && t >= end1) break;  // (a strip of the lower half has five pieces or more)
        const Piece& p = piece[t & 1];
        if (t < 7) fetch(piece[(t + 1) & 1], t + 1);
        const Vec16<T> w1 = weights(cb1[t], p.f1);
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) mma16(p.xf[pb], w1, acc[1][pb]);
        if (t < 4 && t < end0) {
          const Vec16<T> w0 = weights(cb0[t & 3], p.f0);
#pragma unroll
          for (int pb = 0; pb < 4; ++pb) mma16(p.xf[pb], w0, acc[0][pb]);
        }
      }
    }
    // weights as they are defined: last pieces along which dA falls steeply, or all of them
    if (!(split && narrow[0] && narrow[1]))
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) acc[j][pb] *= scale[j];
      scale[j] = 1.f;
      const int begin = split ? steps[j] - !narrow[j] : 0;
#pragma unroll
      for (int t = 0; t < 4 + 4 * j; ++t) {
        if (t < begin || t >= steps[j]) continue;
        float ak[8], tk[8], w[8];
        load8(ak, dAs + 32 * t + 8 * quad), load8(tk, dts + 32 * t + 8 * quad);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float f = (j == 1 ? cb1[t][e] : cb0[t & 3][e]) * __expf(fminf(am[j] - ak[e], 0.f)) * tk[e];
          w[e] = 32 * t + 8 * quad + e > r0[j] + l16 ? 0.f : f;
        }
        Vec16<T> wf;
        wf.set_all(w);
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) mma16(tr.read(Xs + 32 * t * P, pb), wf, acc[j][pb]);
      }
    }
    // ---- row factor, skip, gate; whole rows out
    const int64_t row0 = b * so.sb + (int64_t)c * Q * so.sl + h * so.sh;
    const float Dh = D ? D[h] : 0.f;
    if constexpr (GATED) wait_outstanding<kCopies>(more ? kCopies : 0);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int m = r0[j] + l16;
      auto at = [&](int r) {
        return __umul24((unsigned)(r0[j] + r), (unsigned)so.sl * 2u) + 64u * (l16 >> 3) + 32u * (quad & 1) + 16u * (quad >> 1);
      };
      if (D) {
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) {
          const int piece = 8 * ((2 * pb + (quad >> 1)) ^ S::key(l16)) + 4 * (quad & 1);
          const ema::bf16x4 xv = *reinterpret_cast<const ema::bf16x4*>(Xs + m * P + piece);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[j][pb][e] = fmaf(Dh, (float)xv[e], acc[j][pb][e] * scale[j]);
        }
        scale[j] = 1.f;
      }
      floatx4 zs[4];
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) {  // features 16 pb + 4 quad ..
        const int piece = 8 * ((2 * pb + (quad >> 1)) ^ S::key(l16)) + 4 * (quad & 1);
        acc[j][pb] *= scale[j];
        if constexpr (GATED) {
          const ema::bf16x4 zv = *reinterpret_cast<const ema::bf16x4*>(reinterpret_cast<const T*>(gate) + (16 * j + l16) * P + piece);
#pragma unroll
          for (int e = 0; e < 4; ++e) zs[pb][e] = (float)zv[e] / (1.f + __expf(-(float)zv[e]));
        }
      }
      if constexpr (GATED) {
        if (out_x) store_strip(out_x + row0, join_quads(acc[j][0], acc[j][1]), join_quads(acc[j][2], acc[j][3]), l16, limit - r0[j], at);
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) acc[j][pb] *= zs[pb];
      }
      store_strip(out + row0, join_quads(acc[j][0], acc[j][1]), join_quads(acc[j][2], acc[j][3]), l16, limit - r0[j], at);
    }
  }
}

// Sums after a trade of registers between halves or quarters of a wave.  swap16(a, b): of two lane groups side by side
// (0 and 1, 2 and 3) the even one receives the sum of both's a, the odd one that of both's b; swap32(a, b): the lower half
// receives the sum of both halves' a, the upper that of both's b.
__device__ __forceinline__ float sum_of(u32x2_t s) {
  const unsigned a = s[0], b = s[1];
  return __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
}
__device__ __forceinline__ float swap16_sum(float a, float b) {
  return sum_of(__builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false));
}
__device__ __forceinline__ float swap32_sum(float a, float b) {
  return sum_of(__builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a), __builtin_bit_cast(unsigned, b), false, false));
}
// Sum over the four groups of 16 lanes, in every lane.
__device__ __forceinline__ float quad_sum(float v) {
  v = swap16_sum(v, v);
  return swap32_sum(v, v);
}
// Sum over the 16 lanes of a group, in every lane.
__device__ __forceinline__ float row16_sum(float v) {
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x128, 0xf, 0xf, false));  // row_ror:8
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x124, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x122, 0xf, 0xf, false));
  v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x121, 0xf, 0xf, false));
  return v;
}

// ------------------------------------------------------------------------------------
// dx / ddt / the partial sums of dD (ssd_chunk_scan_bwd_dx_kernel): the mirror image of the chunk scan.  The strips'
// positions run from the chunk's end to the diagonal, the weights are columns of cb.  b8 nh32 L8192 317 -> 246 (4.2 TB/s of its
// 1030 MB), by itself 304 -> 233 (with D 365 -> 258), b4 nh24 L8192 121 -> 91, b1 nh32 L4096 27 -> 22.  Of the 246, the copies
// and stores alone take 201 and the rest alone 153.
// ------------------------------------------------------------------------------------
template <int N>
struct DxHeadsSmem : HeadsTile {
  static constexpr int R = 2;  // heads in LDS
  static constexpr int kState = P * N * (int)sizeof(bf16_t);
  static constexpr int kHead = kRows + kState + kVec;
  static constexpr int kBytes = R * kHead + kFactors + kRows;  // + the waves' own rows of x
  static constexpr int kSlots = 8;                             // partial sums of dD per head: one a wave
};

template <int N, bool EVEN>
__global__ __launch_bounds__(512, 2) void ssd_chunk_scan_bwd_dx_heads_kernel(
    const float* __restrict__ cb, const bf16_t* __restrict__ x, Strides3 sx, const bf16_t* __restrict__ dout, Strides3 sd,
    const float* __restrict__ dt, const float* __restrict__ dA_cs, const bf16_t* __restrict__ Bm, Strides3 sB,
    const bf16_t* __restrict__ dstates, const float* __restrict__ D, bf16_t* __restrict__ dx, Strides3 sdx,
    float* __restrict__ ddt, int nh, int heads_per_group, int ngroups, int L, int C, int units, int splits, SeqIdx seq,
    float* __restrict__ dD_part) {
  using S = DxHeadsSmem<N>;
  using T = bf16_t;
  constexpr int P = S::P, Q = S::Q, R = S::R, NK = N / 32;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  HeadsWalk<EVEN> now(xcd_local_index((int)blockIdx.x, (int)gridDim.x), (int)gridDim.x, units, splits, heads_per_group, ngroups, C);
  HeadsWalk<EVEN> ahead = now;  // the head whose copies are requested next
  // the wave's strips of rows, their pieces of 32 positions from the end to the diagonal, their factors
  int r0[2], steps[2];
  float* fk[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) r0[j] = 16 * S::strip(wave, j), steps[j] = 8 - (r0[j] >> 5);
  float* factors = reinterpret_cast<float*>(smem + R * S::kHead) + wave * 288;
  fk[0] = factors - 32 * (8 - steps[0]);
  fk[1] = factors + 32 * steps[0] - 32 * (8 - steps[1]);
  unsigned char* own = smem + R * S::kHead + S::kFactors + wave * (32 * P * (int)sizeof(T));

  constexpr int kXCopies = 4, kSCopies = S::kState / 8192, kCopies = kXCopies + kSCopies;
  static_assert(8 * 8 * kXCopies == Q && 8 * 1024 * kSCopies == S::kState, "eight waves bring a head");
  constexpr int SP = N / 8;  // pieces of a row of the state
  auto state_key = [](int r) { return N == 128 ? r & 15 : (r >> 1) & 7; };
  auto vec_at = [&](const HeadsWalk<EVEN>& w) { return (((int64_t)w.b * nh + w.head()) * C + w.c) * Q; };
  auto request = [&](int u, int ln) {  // the copies of the head ahead into place u
    const HeadsWalk<EVEN>& w = ahead;
    const int h = w.head();
    unsigned char* base = smem + u * S::kHead;
    S::template copy_rows<kXCopies>(dout + w.b * sd.sb + (int64_t)w.c * Q * sd.sl + h * sd.sh, (int)sd.sl, 32 * wave,
                                    min(Q, L - w.c * Q), base + kXCopies * wave * 1024, ln);
    const T* sg = dstates + (((int64_t)w.b * C + w.c) * nh + h) * (P * N);
    const int r = ln / SP;
#pragma unroll
    for (int j = 0; j < kSCopies; ++j) {
      const int row0 = (kSCopies * wave + j) * (64 / SP);
      copy16_to_lds(sg + row0 * N, (unsigned)(r * N + 8 * ((ln % SP) ^ state_key(row0 + r))) * (unsigned)sizeof(T),
                    base + S::kRows + (kSCopies * wave + j) * 1024);
    }
    if (wave < 2)
      copy16_to_lds((wave == 0 ? dA_cs : dt) + vec_at(w), 16u * (unsigned)ln, base + S::kRows + S::kState + wave * 1024);
    ahead.next();
  };
  request(0, lane);

  // What the heads of a set share: the rows of B, and the columns of cb from the last position on (entries before the
  // diagonal or past the sequence zero).
  Vec16<T> bf[2][NK];
  float cb0[8][8], cb1[4][8];
  bool live[2];
  int limit = 0, stores = 0;
  auto load_shared = [&]() {
    int ln = lane;
    asm volatile("" : "+v"(ln));
    limit = min(Q, L - now.c * Q);
    // stores of a head that can still be outstanding (a ragged chunk leaves some out: none are allowed for)
    stores = limit < Q ? 0 : dD_part ? 7 : 6;
    const ChunkSeq sq = chunk_seq(seq, now.b, now.c, Q);
    const int e0 = 8 * (ln >> 4);
    const T* Bg = Bm + now.b * sB.sb + (int64_t)now.c * Q * sB.sl + now.g * sB.sh + e0;
    const float* cbg = cb + (((int64_t)now.b * C + now.c) * ngroups + now.g) * (Q * Q);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int m = r0[j] + (ln & 15);
      const T* brow = Bg + (int64_t)min(m, limit - 1) * sB.sl;
#pragma unroll
      for (int i = 0; i < NK; ++i) bf[j][i] = load16(brow + 32 * i);
      live[j] = !sq.on() || sq.at(min(m, limit - 1)) == sq.at(limit - 1);
      const float* cbcol = cbg + e0 * Q + m;
#pragma unroll
      for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int k = 32 * (7 - t) + e;
          if (j == 0) cb0[t][e] = cbcol[k * Q];
          else if (t < 4) cb1[t][e] = cbcol[k * Q];
        }
#pragma unroll
      for (int t = 0; t < 8; ++t)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const int k = 32 * (7 - t) + e + e0;
          const bool in = k >= m && k < limit;
          if (j == 0) cb0[t][e] = in ? cb0[t][e] : 0.f;
          else if (t < 4) cb1[t][e] = in ? cb1[t][e] : 0.f;
        }
    }
#pragma unroll
    for (int i = 0; i < NK; ++i) asm volatile("" : "+v"(bf[0][i].raw), "+v"(bf[1][i].raw));
#pragma unroll
    for (int t = 0; t < 8; ++t)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        asm volatile("" : "+v"(cb0[t][e]));
        if (t < 4) asm volatile("" : "+v"(cb1[t][e]));
      }
  };

  if (!EVEN) load_shared();
  for (int u = 0; !now.done(); now.next(), u ^= 1) {
    if (EVEN && now.k == 0) load_shared();
    const int64_t b = now.b;
    const int c = now.c, h = now.head();
    const bool more = now.unit + 1 < now.end;
    wait_outstanding<7, 6>(now.k > 0 ? stores : 0);
    __syncthreads();  // every wave's part of the head is there; every wave is done with the head before
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int l16 = ln & 15, quad = ln >> 4;
    const HeadsTile::Transposed tr(ln);
#pragma unroll
    for (int j = 0; j < 2; ++j)  // the wave's own rows of x
      S::template copy_rows<kXCopies / 2>(x + b * sx.sb + (int64_t)c * Q * sx.sl + h * sx.sh, (int)sx.sl, r0[j], limit, own + j * 2048, ln);
    if (more) request(u ^ 1, ln);
    const unsigned char* base = smem + u * S::kHead;
    const T* Ds = reinterpret_cast<const T*>(base);
    const float* dAs = reinterpret_cast<const float*>(base + S::kRows + S::kState);
    const float* dts = dAs + Q;

    // The weight of (m, k) is cb[k][m] exp(dA_k - dA_m), split as in the chunk scan.
    const float4 ak = *reinterpret_cast<const float4*>(dAs + 4 * ln);
    const float an = dAs[min(4 * ln + 4, Q - 1)], a_end = dAs[Q - 1];
    const bool split = __builtin_amdgcn_ballot_w64(S::template falls<true>(ak, an, ln, limit)) == ~0ull;
    float am[2], ar[2];
    bool narrow[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      am[j] = dAs[r0[j] + l16];
      const float a0 = dAs[r0[j]], a1 = dAs[min(r0[j] + 7, limit - 1)], a2 = dAs[min(r0[j] + 15, limit - 1)];
      narrow[j] = __builtin_amdgcn_readfirstlane(a0 - a1 <= 40.f && a1 - a2 <= 40.f);
      ar[j] = narrow[j] ? a1 : a2;
      const float4 f = make_float4(__expf(fminf(ak.x - ar[j], 40.f)), __expf(fminf(ak.y - ar[j], 40.f)),
                                   __expf(fminf(ak.z - ar[j], 40.f)), __expf(fminf(ak.w - ar[j], 40.f)));
      if (4 * ln >= 32 * (8 - steps[j])) *reinterpret_cast<float4*>(fk[j] + 4 * ln) = f;
    }
    // ---- dstates . B, features in the rows of the product: a lane's values belong to its row of each strip
    floatx4 acc[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) acc[j][pb] = floatx4{0.f, 0.f, 0.f, 0.f};
    const unsigned piece0 = u * S::kHead + S::kRows + (l16 * N + 8 * (quad ^ state_key(l16))) * sizeof(T);
#pragma unroll
    for (int ks = 0; ks < NK; ++ks)
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) {
        const Vec16<T> sf = load16(reinterpret_cast<const T*>(smem + (piece0 ^ (64u * ks)) + 16 * pb * N * sizeof(T)));
        mma16(sf, bf[0][ks], acc[0][pb]);
        mma16(sf, bf[1][ks], acc[1][pb]);
      }
    float scale[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float enter = live[j] ? __expf(fminf(a_end - (split ? ar[j] : am[j]), 0.f)) : 0.f;
      scale[j] = split ? __expf(ar[j] - am[j]) : 1.f;
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) acc[j][pb] *= enter;
    }
    __builtin_amdgcn_s_waitcnt(0xc07f);  // the wave's own factors are visible to its own reads

    // ---- the causal sum
    if (split) {
      struct Piece {
        Vec16<T> xf[4];
        float4 f0[2], f1[2];
      };
      auto fetch = [&](Piece& p, int t) {
        const int k = 32 * (7 - t);
#pragma unroll
        for (int q = 0; q < 2; ++q) p.f0[q] = *reinterpret_cast<const float4*>(fk[0] + k + 8 * quad + 4 * q);
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) p.xf[pb] = tr.read(Ds + k * P, pb);
        if (t < 4)
#pragma unroll
          for (int q = 0; q < 2; ++q) p.f1[q] = *reinterpret_cast<const float4*>(fk[1] + k + 8 * quad + 4 * q);
      };
      auto weights = [&](const float* w, const float4* f) {
        const float t[8] = {w[0] * f[0].x, w[1] * f[0].y, w[2] * f[0].z, w[3] * f[0].w,
                            w[4] * f[1].x, w[5] * f[1].y, w[6] * f[1].z, w[7] * f[1].w};
        Vec16<T> wf;
        wf.set_all(t);
        return wf;
      };
      const int end0 = steps[0] - !narrow[0], end1 = steps[1] - !narrow[1];
      Piece piece[2];
      fetch(piece[0], 0);
#pragma unroll
      for (int t = 0; t < 8; ++t) {
        if (t >= 4 && t >= end0) break;  // (a strip of the upper half has five pieces or more)
        const Piece& p = piece[t & 1];
        if (t < 7) fetch(piece[(t + 1) & 1], t + 1);
        const Vec16<T> w0 = weights(cb0[t], p.f0);
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) mma16(p.xf[pb], w0, acc[0][pb]);
        if (t < 4 && t < end1) {
          const Vec16<T> w1 = weights(cb1[t & 3], p.f1);
#pragma unroll
          for (int pb = 0; pb < 4; ++pb) mma16(p.xf[pb], w1, acc[1][pb]);
        }
      }
    }
    // weights as they are defined: first pieces along which dA falls steeply, or all of them
    if (!(split && narrow[0] && narrow[1]))
#pragma unroll
    for (int j = 0; j < 2; ++j) {
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) acc[j][pb] *= scale[j];
      scale[j] = 1.f;
      const int begin = split ? steps[j] - !narrow[j] : 0;
#pragma unroll
      for (int t = 0; t < 8 - 4 * j; ++t) {
        if (t < begin || t >= steps[j]) continue;
        const int k0 = 32 * (7 - t);
        float ak[8], w[8];
        load8(ak, dAs + k0 + 8 * quad);
#pragma unroll
        for (int e = 0; e < 8; ++e)  // (the exponent is at most 0 and cb 0 where the weight is none)
          w[e] = (j == 0 ? cb0[t][e] : cb1[t & 3][e]) * __expf(fminf(ak[e] - am[j], 0.f));
        Vec16<T> wf;
        wf.set_all(w);
#pragma unroll
        for (int pb = 0; pb < 4; ++pb) mma16(tr.read(Ds + k0 * P, pb), wf, acc[j][pb]);
      }
    }
    // ---- row factor, the sums over the features, dt, skip; whole rows out
    const float Dh = D ? D[h] : 0.f;
    T* dxg = dx + b * sdx.sb + (int64_t)c * Q * sdx.sl + h * sdx.sh;
    float* ddtp = ddt + vec_at(now);
    wait_outstanding<kCopies>(more ? kCopies : 0);
    floatx4 dsum[4];
#pragma unroll
    for (int pb = 0; pb < 4; ++pb) dsum[pb] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int m = r0[j] + l16;
      auto at = [&](int r) {
        return __umul24((unsigned)(r0[j] + r), (unsigned)sdx.sl * 2u) + 64u * (l16 >> 3) + 32u * (quad & 1) + 16u * (quad >> 1);
      };
      const float dtm = dts[m];
      float dot = 0.f;
#pragma unroll
      for (int pb = 0; pb < 4; ++pb) {  // features 16 pb + 4 quad ..
        const int piece = 8 * ((2 * pb + (quad >> 1)) ^ S::key(l16)) + 4 * (quad & 1);
        acc[j][pb] *= scale[j];
        const ema::bf16x4 xv = *reinterpret_cast<const ema::bf16x4*>(reinterpret_cast<const T*>(own) + (16 * j + l16) * P + piece);
#pragma unroll
        for (int e = 0; e < 4; ++e) dot = fmaf(acc[j][pb][e], (float)xv[e], dot);
        acc[j][pb] *= dtm;
        if (D) {
          const ema::bf16x4 dv = *reinterpret_cast<const ema::bf16x4*>(Ds + m * P + piece);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            acc[j][pb][e] = fmaf(Dh, (float)dv[e], acc[j][pb][e]);
            dsum[pb][e] = fmaf(m < limit ? (float)dv[e] : 0.f, (float)xv[e], dsum[pb][e]);
          }
        }
      }
      dot = quad_sum(dot);
      store_strip(dxg, join_quads(acc[j][0], acc[j][1]), join_quads(acc[j][2], acc[j][3]), l16, limit - r0[j], at);
      if (quad == 0) ddtp[m] = m < limit ? dot : 0.f;
    }
    if (dD_part) {
      floatx4 mine = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int pb = 0; pb < 4; ++pb)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float t = row16_sum(dsum[pb][e]);
          mine[e] = l16 == pb ? t : mine[e];
        }
      if (l16 < 4)
        *reinterpret_cast<floatx4*>(dD_part + (((b * C + c) * nh + h) * (int64_t)S::kSlots + wave) * P + 16 * l16 + 4 * quad) = mine;
    }
  }
}

// ------------------------------------------------------------------------------------
// Gradient of the causal term with respect to the per-position dA (ssd_ddA_causal_kernel): with
//   W[m][n] = <dout[m], x[n]> * dt_n * cb[m][n] * exp(min(dA_m - dA_n, 0))   for n < m < limit,
// ddA[j] = sum_{i < j} (colsum_i - rowsum_i).  A strip's blocks of 16 x 16 up to the diagonal one; the row sums stay in
// registers, the column sums of a wave meet those of the others in LDS, and one wave, a head later, forms the prefix
// sum.  b8 nh32 L8192 213 -> 196 (3.1 TB/s of its 600 MB), by itself 186 -> 155, b1 nh32 L2048 15.3 -> 12.7.  Of the 196, the
// copies alone take 116 and the rest alone 131.
// ------------------------------------------------------------------------------------
struct DdaHeadsSmem : HeadsTile {
  static constexpr int R = 3;                                // heads in LDS, of x, dA and dt
  static constexpr int kHead = kRows + kVec;
  static constexpr int kSums = 8 * Q * (int)sizeof(float);   // a wave's sums of columns less those of its rows, each
  static constexpr int kBytes = R * kHead + kRows + kFactors + 2 * kSums;  // + dout, the sums of two heads
};

template <bool EVEN>
__global__ __launch_bounds__(512, 2) void ssd_ddA_heads_kernel(
    const bf16_t* __restrict__ x, Strides3 sx, const bf16_t* __restrict__ dout, Strides3 sd, const float* __restrict__ dt,
    const float* __restrict__ dA_cs, const float* __restrict__ cb, float* __restrict__ ddA, int nh, int heads_per_group,
    int ngroups, int L, int C, int units, int splits) {
  using S = DdaHeadsSmem;
  using T = bf16_t;
  constexpr int P = S::P, Q = S::Q;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  HeadsWalk<EVEN> now(xcd_local_index((int)blockIdx.x, (int)gridDim.x), (int)gridDim.x, units, splits, heads_per_group, ngroups, C);
  HeadsWalk<EVEN> ahead = now;  // the head whose copies are requested next
  // the wave's strips: number `strip`, rows 16 strip .., as many blocks of columns below the diagonal one
  int strip[2];
  float* fk[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) strip[j] = S::strip(wave, j);
  unsigned char* own = smem + S::R * S::kHead;  // dout, each row read by one wave only
  fk[1] = reinterpret_cast<float*>(own + S::kRows) + wave * 288;
  fk[0] = fk[1] + 16 * (strip[1] + 1);
  auto sums = [&](int i) { return reinterpret_cast<float*>(own + S::kRows + S::kFactors + (i & 1) * S::kSums); };

  auto vec_at = [&](const HeadsWalk<EVEN>& w) { return (((int64_t)w.b * nh + w.head()) * C + w.c) * Q; };
  HeadsWalk<EVEN> ahead_own = now;  // the head whose rows of dout are requested next: one ahead, where the others are two
  auto request = [&](int u, int ln) {
    const HeadsWalk<EVEN>& w = ahead;
    unsigned char* base = smem + u * S::kHead;
    S::copy_rows<4>(x + w.b * sx.sb + (int64_t)w.c * Q * sx.sl + w.head() * sx.sh, (int)sx.sl, 32 * wave, min(Q, L - w.c * Q),
                    base + 4 * wave * 1024, ln);
    if (wave < 2) copy16_to_lds((wave == 0 ? dA_cs : dt) + vec_at(w), 16u * (unsigned)ln, base + S::kRows + wave * 1024);
    ahead.next();
  };
  auto request_own = [&](int ln) {
    const HeadsWalk<EVEN>& w = ahead_own;
    const T* dg = dout + w.b * sd.sb + (int64_t)w.c * Q * sd.sl + w.head() * sd.sh;
#pragma unroll
    for (int j = 0; j < 2; ++j) S::copy_rows<2>(dg, (int)sd.sl, 16 * strip[j], min(Q, L - w.c * Q), own + strip[j] * 2048, ln);
    ahead_own.next();
  };
  request(0, lane);
  request_own(lane);
  if (!ahead.done()) request(1, lane);

  // What the heads of a set share: the blocks of cb in the accumulator layout (rows 4 (l / 16) .. + 3, column l % 16),
  // rows past the sequence zero, and the diagonal ones as they are.
  float cb0[7][4], cb1[15][4], cbd[2][4];
  int limit = 0;
  auto load_shared = [&]() {
    int ln = lane;
    asm volatile("" : "+v"(ln));
    limit = min(Q, L - now.c * Q);
    const float* cbg = cb + (((int64_t)now.b * C + now.c) * ngroups + now.g) * (Q * Q);
    const int col = ln & 15, row = 4 * (ln >> 4);
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const float* p = cbg + (16 * strip[j] + row) * Q + col;
#pragma unroll
      for (int nb = 0; nb < 15; ++nb)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          if (j == 1) cb1[nb][v] = p[v * Q + 16 * nb];
          else if (nb < 7) cb0[nb][v] = p[v * Q + 16 * nb];
        }
#pragma unroll
      for (int v = 0; v < 4; ++v) cbd[j][v] = p[v * Q + 16 * strip[j]];
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const bool in = 16 * strip[j] + row + v < limit;
#pragma unroll
        for (int nb = 0; nb < 15; ++nb) {
          if (j == 1) cb1[nb][v] = in ? cb1[nb][v] : 0.f;
          else if (nb < 7) cb0[nb][v] = in ? cb0[nb][v] : 0.f;
        }
      }
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
#pragma unroll
      for (int nb = 0; nb < 15; ++nb) {
        asm volatile("" : "+v"(cb1[nb][v]));
        if (nb < 7) asm volatile("" : "+v"(cb0[nb][v]));
      }
      asm volatile("" : "+v"(cbd[0][v]), "+v"(cbd[1][v]));
    }
  };

  // delta_i = colsum_i - rowsum_i; ddA[j] = sum_{i<j} delta_i: one wave, four positions per lane
  // (0 past the sequence, where the sums hold whatever dt and dA do)
  int64_t before = 0;  // where the head before has its dA
  int rows_before = 0;  // its positions
  auto finish = [&](int i) {
    const float* s = sums(i);
    floatx4 t[8];
#pragma unroll
    for (int w = 0; w < 8; ++w) t[w] = *reinterpret_cast<const floatx4*>(s + w * Q + 4 * lane);
    floatx4 d = ((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]));
#pragma unroll
    for (int k = 0; k < 4; ++k) d[k] = 4 * lane + k < rows_before ? d[k] : 0.f;
    const float local = (d[0] + d[1]) + (d[2] + d[3]);
    float4 o;
    o.x = wave_inclusive_scan(local) - local;
    o.y = o.x + d[0], o.z = o.y + d[1], o.w = o.z + d[2];
    *reinterpret_cast<float4*>(ddA + before + 4 * lane) = o;
  };

  int i = 0;
  if (!EVEN) load_shared();
  for (int u = 0; !now.done(); now.next(), ++i, u = u + 1 < S::R ? u + 1 : 0) {
    if (EVEN && now.k == 0) load_shared();
    // the head's rows have landed once only x of the next head, requested behind them, is outstanding
    wait_outstanding<4>(now.unit + 1 < now.end ? 4 : 0);
    __syncthreads();  // every wave's part of the head is there; every wave is done with the head before
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int l16 = ln & 15, quad = ln >> 4;
    const unsigned char* base = smem + u * S::kHead;
    const T* Xs = reinterpret_cast<const T*>(base);
    const float* dAs = reinterpret_cast<const float*>(base + S::kRows);
    const float* dts = dAs + Q;
    float* colsum = sums(i) + wave * Q;
    // the rows of dout go to registers and their place to the next head's
    Vec16<T> df[2][2];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        df[j][ks] = load16(reinterpret_cast<const T*>(own) + (16 * strip[j] + l16) * P + 8 * ((4 * ks + quad) ^ S::key(l16)));
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(df[0][0].raw), "+v"(df[0][1].raw), "+v"(df[1][0].raw), "+v"(df[1][1].raw)::"memory");
    if (!ahead_own.done()) request_own(ln);
    if (!ahead.done()) request(u > 0 ? u - 1 : S::R - 1, ln);  // (the place of the head before)
    if (i > 0 && wave == (i & 7)) finish(i - 1);
    before = vec_at(now), rows_before = limit;

    // Below a strip the decay is split at its first row r into a factor of the column, exp(r - dA_n) dt_n, and one of the
    // row, exp(dA_m - r).  Neither exponent is larger than their sum where dA falls, so the two are no less exact than
    // the one they stand for (__expf is off by about 6e-8 of its exponent).  The diagonal block, where a split would need
    // exponents of both signs, takes its weights as they are defined.
    const float4 ak = *reinterpret_cast<const float4*>(dAs + 4 * ln);
    const float4 tk = S::weights_of_time(dts, ln, limit);
    const float an = dAs[min(4 * ln + 4, Q - 1)];
    const bool split = __builtin_amdgcn_ballot_w64(S::falls<false>(ak, an, ln, limit) & S::finite(tk)) == ~0ull;
    float em[2][4];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r0 = 16 * strip[j];
      const float ar = dAs[min(r0, limit - 1)];  // (the factors of strips past the sequence meet zeros, and must be finite)
      const float4 f = make_float4(__expf(fminf(ar - ak.x, 0.f)) * tk.x, __expf(fminf(ar - ak.y, 0.f)) * tk.y,
                                   __expf(fminf(ar - ak.z, 0.f)) * tk.z, __expf(fminf(ar - ak.w, 0.f)) * tk.w);
      if (4 * ln < r0) *reinterpret_cast<float4*>(fk[j] + 4 * ln) = f;
      const float4 am = *reinterpret_cast<const float4*>(dAs + r0 + 4 * quad);
      em[j][0] = am.x, em[j][1] = am.y, em[j][2] = am.z, em[j][3] = am.w;
    }
    const int x_lane = l16 * P + 8 * (quad ^ S::key(l16));  // (the second half of the features: bit 2 of the piece)
    auto x_frag = [&](int nb, int ks) { return load16(Xs + (16 * nb) * P + (x_lane ^ (32 * ks))); };
    auto product = [&](int j, const Vec16<T>* xf) {
      floatx4 acc = {0.f, 0.f, 0.f, 0.f};
      mma16(df[j][0], xf[0], acc);
      mma16(df[j][1], xf[1], acc);
      return acc;
    };
    floatx4 rows[2];
    rows[0] = rows[1] = floatx4{0.f, 0.f, 0.f, 0.f};
    __builtin_amdgcn_s_waitcnt(0xc07f);  // the wave's own factors are visible to its own reads

    // column sums of block nb over the lane's rows; of the diagonal blocks
    float col[16], diag[2] = {0.f, 0.f};
#pragma unroll
    for (int nb = 0; nb < 16; ++nb) col[nb] = 0.f;
    floatx4 exact[2];  // row sums that the row factor does not apply to
    // ---- the diagonal blocks
    {
      const Vec16<T> xd0[2] = {x_frag(strip[0], 0), x_frag(strip[0], 1)}, xd1[2] = {x_frag(strip[1], 0), x_frag(strip[1], 1)};
      const floatx4 d[2] = {product(0, xd0), product(1, xd1)};
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int n = 16 * strip[j] + l16;
        const float an = dAs[n], tn = n < limit ? dts[n] : 0.f;
#pragma unroll
        for (int v = 0; v < 4; ++v) {  // (selects, so that no product past the diagonal or the sequence is met)
          const float f = d[j][v] * cbd[j][v] * tn * __expf(fminf(em[j][v] - an, 0.f));
          exact[j][v] = ((l16 < 4 * quad + v) & (4 * quad + v < limit - 16 * strip[j])) ? f : 0.f;
          diag[j] += exact[j][v];
          em[j][v] = __expf(fminf(em[j][v] - dAs[16 * strip[j]], 0.f));
        }
      }
    }
    if (split) {
      auto block = [&](int j, const floatx4& acc, const float* w, float gn) {
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float u = acc[v] * w[v];
          rows[j][v] = fmaf(u, gn, rows[j][v]);
          s = fmaf(u, em[j][v], s);
        }
        return s * gn;
      };
      // the blocks two ahead with their reads and one ahead with their products
      struct Piece {
        Vec16<T> xf[2];
        float g0, g1;
      };
      auto fetch = [&](Piece& p, int nb) {
        p.xf[0] = x_frag(nb, 0), p.xf[1] = x_frag(nb, 1);
        p.g1 = fk[1][16 * nb + l16];
        if (nb < 7) p.g0 = fk[0][16 * nb + l16];
      };
      Piece piece[2];
      fetch(piece[0], 0);
      fetch(piece[1], 1);
      floatx4 p0 = product(0, piece[0].xf), p1 = product(1, piece[0].xf);
      float g0 = piece[0].g0, g1 = piece[0].g1;
#pragma unroll
      for (int nb = 0; nb < 15; ++nb) {
        if (nb >= 8 && nb >= strip[1]) break;  // (the strips of the lower half have eight blocks or more)
        fetch(piece[nb & 1], nb + 2 < 16 ? nb + 2 : 15);
        const floatx4 n1 = product(1, piece[(nb + 1) & 1].xf);
        floatx4 n0;
        if (nb < 6) n0 = product(0, piece[(nb + 1) & 1].xf);
        const float m0 = piece[(nb + 1) & 1].g0, m1 = piece[(nb + 1) & 1].g1;
        col[nb] = block(1, p1, cb1[nb], g1);
        if (nb < 7 && nb < strip[0]) col[nb] += block(0, p0, cb0[nb < 7 ? nb : 0], g0);
        p1 = n1, g1 = m1;
        if (nb < 6) p0 = n0, g0 = m0;
      }
    } else {  // where dA rises: weights as they are defined
      const float4 a0 = *reinterpret_cast<const float4*>(dAs + 16 * strip[0] + 4 * quad);
      const float4 a1 = *reinterpret_cast<const float4*>(dAs + 16 * strip[1] + 4 * quad);
      auto block = [&](int j, const floatx4& acc, const float* w, const float4& am, float an, float tn) {
        const float m[4] = {am.x, am.y, am.z, am.w};
        float s = 0.f;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          const float f = acc[v] * w[v] * tn * __expf(fminf(m[v] - an, 0.f));
          const float u = 4 * quad + v < limit - 16 * strip[j] ? f : 0.f;
          exact[j][v] += u;
          s += u;
        }
        return s;
      };
#pragma unroll
      for (int nb = 0; nb < 15; ++nb) {
        if (nb >= 8 && nb >= strip[1]) break;
        const Vec16<T> xf[2] = {x_frag(nb, 0), x_frag(nb, 1)};
        const float an = dAs[16 * nb + l16], tn = dts[16 * nb + l16];
        col[nb] = block(1, product(1, xf), cb1[nb], a1, an, tn);
        if (nb < 7 && nb < strip[0]) col[nb] += block(0, product(0, xf), cb0[nb < 7 ? nb : 0], a0, an, tn);
      }
    }
    diag[0] = quad_sum(diag[0]), diag[1] = quad_sum(diag[1]);
#pragma unroll
    for (int q = 0; q < 4; ++q) {  // the sums of four blocks over the groups of 16 lanes: lane group q holds block 4 i + q
      const float lo = swap16_sum(col[4 * q], col[4 * q + 1]), hi = swap16_sum(col[4 * q + 2], col[4 * q + 3]);
      colsum[64 * q + ln] = swap32_sum(lo, hi);
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
      if (quad == j) colsum[16 * strip[j] + l16] += diag[j];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      float4 r;
      r.x = row16_sum(fmaf(rows[j][0], em[j][0], exact[j][0])), r.y = row16_sum(fmaf(rows[j][1], em[j][1], exact[j][1]));
      r.z = row16_sum(fmaf(rows[j][2], em[j][2], exact[j][2])), r.w = row16_sum(fmaf(rows[j][3], em[j][3], exact[j][3]));
      if (l16 == 0) {
        float4* own_rows = reinterpret_cast<float4*>(colsum + 16 * strip[j] + 4 * quad);
        const float4 t = *own_rows;
        *own_rows = make_float4(t.x - r.x, t.y - r.y, t.z - r.z, t.w - r.w);
      }
    }
  }
  __syncthreads();
  if (wave == 0) finish(i - 1);
}

}  // namespace ssd
