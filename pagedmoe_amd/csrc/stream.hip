// Expert GEMMs for few rows per expert: every weight byte streamed once
// through registers into bf16 MFMA, activations held in registers.
//
// Replaces the per-expert quantized_matmul calls of the reference's grouped
// path (streaming.py:789-836) between the decode GEMV (one to a few rows an
// expert, decode.hip) and the prefill GEMMs (128-row tiles, prefill.hip).
// These sizes are bound by the weight stream, so the kernel is built around
// it:
//
//   * The reduction is cut into NSL slices of G quantization groups
//     (stream_cut), one wave each; a wave keeps its slice of the tile's 16 or 32 activation
//     rows in registers as MFMA operands for as long as the tile lasts, and
//     its inner loop only loads weights: tiles of 16 weight rows, a ring of
//     them in flight, read as 16-byte (4-bit) or 12-byte (6-bit) pieces,
//     64 or 48 contiguous bytes of each of 16 rows an instruction.
//   * Weights go into the MFMA as bf16 (128 + q), one and/or per pair
//     (gemv_common.h's form; the dequantized operand of prefill.hip takes 2.9
//     vector instructions a value, this 0.9): each group's product is scaled by
//     its s in fp32, and (b - 128 s) * sum(x) is added by one fp32 MFMA per
//     four groups, so no operand is rounded to bf16 but x itself.
//   * The slices' fp32 partial sums meet in LDS once per step of four weight
//     tiles (double buffered, one LDS-only barrier, loads stay in flight
//     across it).  With one or two tiles a step, 16 columns stored at a time
//     and 64-bit vector addresses, Qwen3-Next shapes took 169 us a layer at
//     24 tokens and 415 at 1000, against 138 and 405.
//   * Work is the flat list (row tile, step), cut into equal contiguous
//     ranges, one per resident block: every block streams the same number of
//     bytes whatever the expert loads are.
//
// Measured (Qwen3-235B shapes, 100 tokens, every expert active): gate/up 694
// -> 186 us (4.9 TB/s of weights), down 395 -> 103 us (4.4 TB/s) against the
// GEMV, which repeats its dot products for every row of an expert; the same
// loads without arithmetic, reduction and stores take 160 and 82 us.  8 waves
// a CU at 256 registers: x takes 128 of them at 32 rows.  Only the 14-group
// slices spill, around the weight loop, not in it.
#include <algorithm>
#include <type_traits>

#include "gemv_common.h"
#include "pmoe_internal.h"
#include "pmoe_kernels.h"
#include "route_common.h"

namespace pmoe {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x2_a4 __attribute__((ext_vector_type(2), aligned(4)));
typedef uint32_t u32x3_a4 __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kStreamRows = 32;   // rows of a dispatch tile
constexpr int kCols = 16;         // weight rows (output columns) of a weight tile
constexpr int kTiles = 4;         // weight tiles of a step (one reduction and barrier)
constexpr int kPart = 256;        // floats of a 16 x 16 partial, in lane order

struct StreamArgs {
  const uint8_t* slab;
  int64_t expert_bytes;
  const int32_t* order;
  const int4* tiles;      // {slot, first row, expert rows, expert offset}
  const int32_t* n_tiles;
  const uint16_t* act;    // gate/up: x [n, hidden]; down: h [rows, inter], sorted
  int kk;                 // flat rows per token (gate/up activation gather)
  int cols;               // reduction length
  int out_cols;
  QProj p0, p1;
  void* out;              // gate/up: h (sorted rows); down: y (flat rows)
  int out_vec;            // bf16 out is 8-byte aligned
};

// One weight tile of a wave's slice: 16 rows x G groups.  The words stay in
// the vectors they are loaded as, so that a ring register is never copied
// (a copy at the end of a loop trip waits for the load into it).
template <int BITS, int G>
struct WTile {
  static constexpr int kV = BITS == 4 ? G / 2 : G;
  static constexpr int kRegs = BITS == 4 ? 2 * G : 3 * G;
  using V = std::conditional_t<BITS == 4, u32x4, u32x3_a4>;
  static constexpr int kS4 = G / 8;               // scale words: vectors of 4,
  static constexpr int kSR = (G % 8) / 2;         // then one of the 0-3 left
  static_assert(G % 2 == 0, "scales are read as whole words");
  using R = std::conditional_t<kSR == 1, uint32_t,
                               std::conditional_t<kSR == 2, u32x2_a4, u32x3_a4>>;
  V w[kV];
  u32x4_a4 s4[kS4 ? kS4 : 1], b4[kS4 ? kS4 : 1];
  R sr, br;
  __device__ __forceinline__ uint32_t word(int i) const {
    return BITS == 4 ? w[i >> 2][i & 3] : w[i / 3][i % 3];
  }
  __device__ __forceinline__ uint32_t s(int i) const {
    return i < 4 * kS4 ? s4[i < 4 * kS4 ? i >> 2 : 0][i & 3] : rest(sr, i - 4 * kS4);
  }
  __device__ __forceinline__ uint32_t b(int i) const {
    return i < 4 * kS4 ? b4[i < 4 * kS4 ? i >> 2 : 0][i & 3] : rest(br, i - 4 * kS4);
  }
  static __device__ __forceinline__ uint32_t rest(const R& r, int i) {
    if constexpr (kSR == 1)
      return r;
    else
      return r[i];
  }
  // Opaque to the optimiser: without this, unpacking moves to the end of the
  // loop trip that loaded the words and waits for them there.
  __device__ __forceinline__ void pin() {
#pragma unroll
    for (int i = 0; i < kS4; ++i) asm volatile("" : "+v"(s4[i]), "+v"(b4[i]));
    if constexpr (kSR != 0) asm volatile("" : "+v"(sr), "+v"(br));
#pragma unroll
    for (int i = 0; i < kV; ++i) asm volatile("" : "+v"(w[i]));
  }
};

// Lane l of the tile owns weight row l % 16 and quarter kq = l / 16 of each
// group's 64 values.  4-bit: a load covers two groups, 16 bytes a lane, the
// lower lanes holding the first group's two halves and the upper lanes the
// second's; unpack_pair trades words between the wave's halves so that each
// register then holds one group.  6-bit: 12 bytes a lane and group.
// Addresses are a buffer resource over the expert's slot, a lane offset and a
// scalar offset per tile (no vector arithmetic, no address registers).
template <int BITS, int G>
__device__ __forceinline__ void load_tile(WTile<BITS, G>& t, __amdgpu_buffer_rsrc_t slot,
                                          uint32_t w_off, uint32_t w, uint32_t s_off, uint32_t s,
                                          uint32_t b) {
  using T = WTile<BITS, G>;
#pragma unroll
  for (int i = 0; i < T::kV; ++i) {
    if constexpr (BITS == 4)
      t.w[i] = __builtin_amdgcn_raw_buffer_load_b128(slot, w_off + 64 * i, w, 0);
    else
      t.w[i] = __builtin_amdgcn_raw_buffer_load_b96(slot, w_off + 48 * i, w, 0);
  }
#pragma unroll
  for (int i = 0; i < T::kS4; ++i) {
    t.s4[i] = __builtin_amdgcn_raw_buffer_load_b128(slot, s_off + 16 * i, s, 0);
    t.b4[i] = __builtin_amdgcn_raw_buffer_load_b128(slot, s_off + 16 * i, b, 0);
  }
  if constexpr (T::kSR == 3) {
    t.sr = __builtin_amdgcn_raw_buffer_load_b96(slot, s_off + 16 * T::kS4, s, 0);
    t.br = __builtin_amdgcn_raw_buffer_load_b96(slot, s_off + 16 * T::kS4, b, 0);
  } else if constexpr (T::kSR == 2) {
    t.sr = __builtin_amdgcn_raw_buffer_load_b64(slot, s_off + 16 * T::kS4, s, 0);
    t.br = __builtin_amdgcn_raw_buffer_load_b64(slot, s_off + 16 * T::kS4, b, 0);
  } else if constexpr (T::kSR == 1) {
    t.sr = __builtin_amdgcn_raw_buffer_load_b32(slot, s_off + 16 * T::kS4, s, 0);
    t.br = __builtin_amdgcn_raw_buffer_load_b32(slot, s_off + 16 * T::kS4, b, 0);
  }
}

// First of the 16 values of a group that lane quarter kq holds: after the
// exchange of unpack_pair the quarters hold values 0-15, 32-47, 16-31 and
// 48-63 of a 4-bit group; a 6-bit group's are in order.
template <int BITS>
__device__ __forceinline__ int quarter_k(int kq) {
  return BITS == 4 ? ((kq & 1) << 5) | ((kq >> 1) << 4) : kq << 4;
}

// The wave's slice of 16 activation rows, as MFMA A operands in the weight
// words' value order, and sum(x) of group 4 q + kq of the lane's row.
template <int G>
struct XTile {
  u32x4 a[G][2];
  float sum[(G + 3) / 4];
};

// The first `repeat` groups are the slice before's too and count as zero here.
template <int BITS, int G>
__device__ __forceinline__ void load_x(XTile<G>& x, const uint16_t* src, int kq, int repeat) {
  constexpr uint32_t kOnes = 0x3F803F80u;
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int c = 0; c < 2; ++c)
      x.a[g][c] = *reinterpret_cast<const u32x4*>(src + 64 * g + 8 * c);
#pragma unroll
  for (int q = 0; q < (G + 3) / 4; ++q) x.sum[q] = 0.0f;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const uint32_t keep = g < repeat ? 0u : ~0u;
    float s = 0.0f;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const u32x4 d = x.a[g][c] & keep;
      s = dot2(d[3], kOnes, dot2(d[2], kOnes, dot2(d[1], kOnes, dot2(d[0], kOnes, s))));
      if constexpr (BITS == 4)  // pairs (x_i, x_{i+4}), as nib_pair unpacks
        x.a[g][c] = u32x4{__builtin_amdgcn_perm(d[2], d[0], 0x05040100u),
                          __builtin_amdgcn_perm(d[2], d[0], 0x07060302u),
                          __builtin_amdgcn_perm(d[3], d[1], 0x05040100u),
                          __builtin_amdgcn_perm(d[3], d[1], 0x07060302u)};
      else
        x.a[g][c] = d;
    }
    s = s + xor_lane<32>(s);
    s = s + xor_lane<16>(s);
    if (kq == (g & 3)) x.sum[g >> 2] = s;
  }
}

__device__ __forceinline__ uint32_t mov_k43() {
  uint32_t k;
  asm("v_mov_b32 %0, 0x43004300" : "=v"(k));
  return k;
}

// 8 values of a 4-bit word / half of a 6-bit quarter as the bf16 operand.
__device__ __forceinline__ bf16x8 op4(uint32_t w, uint32_t k43) {
  return __builtin_bit_cast(bf16x8, u32x4{nib_pair<0>(w, k43), nib_pair<1>(w, k43),
                                          nib_pair<2>(w, k43), nib_pair<3>(w, k43)});
}

template <int C>
__device__ __forceinline__ bf16x8 op6(const u32x3_a4& w, uint32_t k43) {
  u32x4 o;
#pragma unroll
  for (int p = 0; p < 4; ++p) {
    const int bit = 12 * (4 * C + p), wi = bit >> 5, sh = bit & 31;
    uint32_t f;
    if (sh + 12 <= 32)
      f = w[wi] >> sh;
    else
      f = __builtin_amdgcn_alignbit(w[wi + 1], w[wi], sh);
    o[p] = and_or(f, 0x3Fu, and_or(f << 10, 0x003F0000u, k43));
  }
  return __builtin_bit_cast(bf16x8, o);
}

// bf16 half (odd ? high : low) of a word as float, the half picked per lane.
__device__ __forceinline__ float pick_half(uint32_t w, bool odd) {
  return __uint_as_float(odd ? (w & 0xFFFF0000u) : (w << 16));
}

// acc[mt] = x_mt . dequantized tile over the slice.
template <int BITS, int G, int MT>
__device__ __forceinline__ void tile_mfma(WTile<BITS, G>& t, const XTile<G> (&x)[MT], int kq,
                                          f32x4 (&acc)[MT]) {
  t.pin();
  const uint32_t k43 = mov_k43();
  // (b - 128 s) sum(x): K = 4 groups a step, lane quarter kq holding group
  // 4 q + kq of both operands
#pragma unroll
  for (int q = 0; q < (G + 3) / 4; ++q) {
    constexpr int kWords = G / 2;
    const bool two = 2 * q + 1 < kWords;
    const int hi = two ? 2 * q + 1 : 2 * q;
    const uint32_t sw = (kq & 2) ? t.s(hi) : t.s(2 * q);
    const uint32_t bw = (kq & 2) ? t.b(hi) : t.b(2 * q);
    const float s = pick_half(sw, kq & 1), b = pick_half(bw, kq & 1);
    float c = __builtin_fmaf(-128.0f, s, b);
    if (!two && (kq & 2)) c = 0.0f;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      acc[mt] = __builtin_amdgcn_mfma_f32_16x16x4f32(x[mt].sum[q], c, q ? acc[mt] : f32x4{}, 0, 0,
                                                     0);
  }
#pragma unroll
  for (int g = 0; g < G; ++g) {
    bf16x8 b0, b1;
    if constexpr (BITS == 4) {
      const int p = g >> 1;
      // groups 2p, 2p+1: the upper lanes' words of the first chunk half
      // trade places with the lower lanes' of the second
      const auto r0 = __builtin_amdgcn_permlane32_swap(t.w[p][0], t.w[p][2], false, false);
      const auto r1 =
          __builtin_amdgcn_permlane32_swap(t.w[p][1], t.w[p][3], false, false);
      b0 = op4(r0[g & 1], k43);
      b1 = op4(r1[g & 1], k43);
    } else {
      b0 = op6<0>(t.w[g], k43);
      b1 = op6<1>(t.w[g], k43);
    }
    const float s = __uint_as_float((g & 1) ? (t.s(g >> 1) & 0xFFFF0000u) : (t.s(g >> 1) << 16));
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f32x4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8, x[mt].a[g][0]), b0, f32x4{}, 0, 0, 0);
      d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, x[mt].a[g][1]), b1, d,
                                                  0, 0, 0);
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[mt][r] = __builtin_fmaf(s, d[r], acc[mt][r]);
    }
  }
}

// z, or NaN where v holds an infinity or a NaN.
__device__ __forceinline__ float finite_or_nan(const f32x4& v, float z) {
#pragma unroll
  for (int i = 0; i < 4; ++i) z = __builtin_fmaf(v[i], 0.0f, z);
  return z;
}

// A block's current tile.
struct Seg {
  __amdgpu_buffer_rsrc_t slot;  // the expert's weights
  int p0, m;                    // first sorted row, rows
};

template <int BITS, int G, int NSL, bool DUAL, bool F32>
struct StreamKernel {
  static constexpr int kThreads = 64 * NSL;
  static constexpr int kMaxMT = G <= 8 ? 2 : 1;  // 32 rows of x fit next to the ring
  static constexpr int kStepCols = kTiles * kCols / (DUAL ? 2 : 1);  // output columns a step
  // Partials of one weight tile: [row tile][slice][16 x 16]; the pad puts the
  // tiles that 16 neighbouring threads of the reduction read on other banks.
  static constexpr int kTilePart = kMaxMT * NSL * kPart + 16;
  static constexpr int kLds = 2 * kTiles * kTilePart;
  using Out = std::conditional_t<F32, float, uint16_t>;

  // Weight tiles in flight: what fits in 256 registers next to x.
  template <int MT>
  static constexpr int ring() {
    constexpr int room = 256 - (BITS == 4 ? 56 : 72) - MT * (8 * G + (G + 3) / 4 + 4);
    return 4 * (WTile<BITS, G>::kRegs + G) <= room ? 4 : 2;
  }

  // Steps [st0, st1) of rows [r0, r0 + 16 MT) of the segment.  Tile t of a
  // step: gate (even t) or up rows of 16 columns, or 16 down rows.
  template <int MT>
  static __device__ __forceinline__ void run(const StreamArgs& a, const Seg& sg, int r0, int st0,
                                             int st1, float* part, int& buf,
                                             const int32_t* s_row, uint32_t* s_odd) {
    constexpr int E = ring<MT>();
    const int lane = threadIdx.x & 63;
    const int slice = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, kq = lane >> 4;
    const int m = sg.m - r0;
    const uint32_t row_bytes = uint32_t(a.cols) * BITS / 8;
    const uint32_t groups = uint32_t(a.cols) / 64;
    // first group of the slice: the last slices of an uneven cut move back to
    // end with the row
    const int g0 = min(slice * G, int(groups) - G);
    const uint32_t w_off = row * row_bytes + kq * (BITS == 4 ? 16 : 12);
    const uint32_t s_off = row * groups * 2;
    WTile<BITS, G> W[E];
    // tile t0 + e of a step into ring entry e (t0 even)
    auto load = [&](int e, int t0, int step) {
      const QProj& q = DUAL && (e & 1) ? a.p1 : a.p0;
      const uint32_t r = (step * (kStepCols / kCols) + (DUAL ? (t0 + e) >> 1 : t0 + e)) * kCols;
      const uint32_t g = g0 * 2 + r * groups * 2;
      load_tile<BITS, G>(W[e], sg.slot, w_off,
                         uint32_t(q.w) + g0 * (64 * BITS / 8) + r * row_bytes, s_off,
                         uint32_t(q.s) + g, uint32_t(q.b) + g);
    };
    int ar[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int r = sg.p0 + r0 + min(16 * mt + row, m - 1);  // rows past the tile: its last row
      ar[mt] = DUAL ? a.order[r] / a.kk : r;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) load(e, 0, st0);
    __builtin_amdgcn_sched_barrier(0);
    XTile<G> x[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      load_x<BITS, G>(x[mt], a.act + size_t(ar[mt]) * a.cols + g0 * 64 + quarter_k<BITS>(kq), kq,
                      slice * G - g0);
    // Everything so far has arrived (the activations, requested last, are
    // needed at once): with nothing pending on entry, the compiler's wait
    // counts at the loop head are those of the steady state.  Left pending
    // in an order of the compiler's choosing, it waited there for the whole
    // ring on every trip.
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    for (int st = st0; st < st1; ++st) {
      float* pb = part + buf * (kTiles * kTilePart);
      const int next = min(st + 1, st1 - 1);  // past the range: the last step's again, unused
      // One trip per ring length: each tile of a trip keeps its registers.
#pragma unroll 1
      for (int t0 = 0; t0 < kTiles; t0 += E) {
        const int tn = t0 + E < kTiles ? t0 + E : 0;
        const int sn = t0 + E < kTiles ? st : next;
#pragma unroll
        for (int e = 0; e < E; ++e) {
          f32x4 acc[MT];
          tile_mfma<BITS, G, MT>(W[e], x, kq, acc);
          __builtin_amdgcn_sched_barrier(0);
          load(e, tn, sn);
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              pb[(t0 + e) * kTilePart + (mt * NSL + slice) * kPart + 64 * r + lane] = acc[mt][r];
        }
      }
      block_lds_sync();
      // Sum the slices: 4 columns of a row a thread, neighbouring threads
      // along the row.
      constexpr int kQuads = kStepCols / 4;
      int tid = threadIdx.x;
      asm volatile("" : "+v"(tid));  // opaque: addresses recomputed here, not held across the loop
      float odd = 0.0f;  // NaN once an output is infinite or NaN (redo_range)
      for (int i = tid; i < MT * 16 * kQuads; i += kThreads) {
        const int c4 = i % kQuads, j = i / kQuads;
        const int mt = j >> 4;
        const int rr = 16 * mt + 4 * (j & 3) + ((j >> 2) & 3);
        if (rr >= m) continue;
        const float* q = pb + (DUAL ? 2 : 1) * (c4 >> 2) * kTilePart + mt * NSL * kPart +
                         64 * ((j >> 2) & 3) + 16 * (j & 3) + 4 * (c4 & 3);
        f32x4 v = *reinterpret_cast<const f32x4*>(q);
#pragma unroll
        for (int sl = 1; sl < NSL; ++sl) v += *reinterpret_cast<const f32x4*>(q + sl * kPart);
        odd = finite_or_nan(v, DUAL ? 0.0f : odd);
        if constexpr (DUAL) {
          // Branched on between the two sums, not once after the loop: with
          // both sums' reads in flight the longest slices spill.
          if (odd != 0.0f) *s_odd = 1;
          f32x4 u = *reinterpret_cast<const f32x4*>(q + kTilePart);
#pragma unroll
          for (int sl = 1; sl < NSL; ++sl)
            u += *reinterpret_cast<const f32x4*>(q + kTilePart + sl * kPart);
          if (finite_or_nan(u, 0.0f) != 0.0f) *s_odd = 1;
#pragma unroll
          for (int c = 0; c < 4; ++c) v[c] = silu_fast(v[c]) * u[c];
        }
        const int orow = DUAL ? sg.p0 + r0 + rr : s_row[r0 + rr];
        Out* dst = static_cast<Out*>(a.out) + size_t(orow) * a.out_cols + st * kStepCols + 4 * c4;
        if constexpr (F32) {
          *reinterpret_cast<f32x4*>(dst) = v;
        } else {
          const u32x2 o = {uint32_t(f2bf(v[0])) | uint32_t(f2bf(v[1])) << 16,
                           uint32_t(f2bf(v[2])) | uint32_t(f2bf(v[3])) << 16};
          if (DUAL || a.out_vec) {
            *reinterpret_cast<u32x2*>(dst) = o;
          } else {
            dst[0] = Out(o[0]), dst[1] = Out(o[0] >> 16);
            dst[2] = Out(o[1]), dst[3] = Out(o[1] >> 16);
          }
        }
      }
      if (!DUAL && odd != 0.0f) *s_odd = 1;
      buf ^= 1;
    }
  }
};

// One weight row times one activation row, group by group: lanes take a group
// each, weights dequantized before the product.
template <int BITS>
__device__ __forceinline__ float plain_dot(const uint32_t* w, const uint16_t* s, const uint16_t* b,
                                           const uint16_t* x, int groups) {
  float p = 0.0f;
  for (int g = threadIdx.x & 63; g < groups; g += 64) {
    const float sg = bf16f(s[g]), bg = bf16f(b[g]);
    uint64_t bits = 0;
    int have = 0, wi = g * (2 * BITS);
#pragma unroll 1
    for (int k = 0; k < 64; ++k) {
      if (have < BITS) bits |= uint64_t(w[wi++]) << have, have += 32;
      const float q = float(uint32_t(bits) & ((1u << BITS) - 1));
      bits >>= BITS, have -= BITS;
      p = __builtin_fmaf(bf16f(x[64 * g + k]), __builtin_fmaf(sg, q, bg), p);
    }
  }
  return wave_sum_bfly(p);
}

// Row tiles of a block's range of the flat list [u, u1): the tile and its steps
// at u, and u past them.
struct Part {
  int slot, p0, m, st0, st1;
};

__device__ __forceinline__ Part next_part(const StreamArgs& a, int n_st, int64_t& u, int64_t u1) {
  typedef const __attribute__((address_space(4))) int32_t ConstI32;
  const int tile = int(u / n_st);
  Part t;
  t.st0 = int(u - int64_t(tile) * n_st);
  t.st1 = int(min(int64_t(n_st), t.st0 + (u1 - u)));
  u += t.st1 - t.st0;
  ConstI32* tl = (ConstI32*)(a.tiles + tile);
  const int first = tl[1];
  t.slot = tl[0];
  t.p0 = tl[3] + first;
  t.m = min(kStreamRows, tl[2] - first);
  return t;
}

// The outputs of a block's range that came out infinite or NaN once more, with
// plain products: (128 + q) x and 128 s sum(x) of an x above ~1e34 overflow
// where (s q + b) x does not, and those of an infinity cancel to NaN.  (An
// overflow on the way always reaches the output.  Scaling such rows in
// registers cost the loops spills, a flag a tile 1-2% of a layer.)  Rows with a
// NaN are left as they are.  Waves take 64 columns of a row at a time.
template <int BITS, int NSL, int STEP_COLS, bool DUAL, bool F32>
__device__ __forceinline__ void redo_range(const StreamArgs& a, int n_st, int64_t u, int64_t u1) {
  using Out = std::conditional_t<F32, float, uint16_t>;
  constexpr uint32_t kInf = F32 ? 0x7F800000u : 0x7F80u;
  const int lane = threadIdx.x & 63;
  const int groups = a.cols / 64;
  const size_t row_bytes = size_t(a.cols) * BITS / 8;
#pragma unroll 1
  while (u < u1) {
    const Part t = next_part(a, n_st, u, u1);
    if (t.slot < 0) continue;
    const uint8_t* slot = a.slab + size_t(t.slot) * size_t(a.expert_bytes);
#pragma unroll 1
    for (int p = t.p0; p < t.p0 + t.m; ++p) {
      const int flat = a.order[p];
      const uint16_t* x = a.act + size_t(DUAL ? flat / a.kk : p) * a.cols;
      Out* out = static_cast<Out*>(a.out) + size_t(DUAL ? p : flat) * a.out_cols;
      bool nan = false;
      for (int k = lane; k < a.cols; k += 64) nan |= (x[k] & 0x7FFFu) > 0x7F80u;
      if (__ballot(nan)) continue;
      const int c1 = t.st1 * STEP_COLS;
#pragma unroll 1
      for (int c0 = t.st0 * STEP_COLS + int(threadIdx.x & ~63u); c0 < c1; c0 += 64 * NSL) {
        const uint32_t v =
            c0 + lane < c1
                ? reinterpret_cast<const std::conditional_t<F32, uint32_t, uint16_t>*>(out)[c0 + lane]
                : 0u;
#pragma unroll 1
        for (uint64_t odd = __ballot((v & kInf) == kInf); odd; odd &= odd - 1) {
          const int c = c0 + __builtin_ctzll(odd);
          auto dot = [&](const QProj& q) {
            return plain_dot<BITS>(
                reinterpret_cast<const uint32_t*>(slot + q.w + c * row_bytes),
                reinterpret_cast<const uint16_t*>(slot + q.s) + size_t(c) * groups,
                reinterpret_cast<const uint16_t*>(slot + q.b) + size_t(c) * groups, x, groups);
          };
          float y = dot(a.p0);
          if constexpr (DUAL) y = silu_fast(y) * dot(a.p1);
          if (lane) continue;
          if constexpr (F32)
            out[c] = y;
          else
            out[c] = f2bf(y);
        }
      }
    }
  }
}

template <int BITS, int G, int NSL, bool DUAL, bool F32>
__global__ __launch_bounds__(64 * NSL, 2) void stream_kernel(const StreamArgs a) {
  using K = StreamKernel<BITS, G, NSL, DUAL, F32>;
  typedef const __attribute__((address_space(4))) int32_t ConstI32;
  __shared__ __attribute__((aligned(16))) float part[K::kLds];
  __shared__ int32_t s_row[2][kStreamRows];
  __shared__ uint32_t s_odd;  // an output of this block is not finite
  const int n_st = a.out_cols / K::kStepCols;
  const int64_t total = int64_t(*(ConstI32*)a.n_tiles) * n_st;
  const int64_t u0 = total * blockIdx.x / gridDim.x;
  const int64_t u1 = total * (blockIdx.x + 1) / gridDim.x;
  int buf = 0, par = 0;
  if (threadIdx.x == 0) s_odd = 0;  // seen by all from the first step's barrier
  for (int64_t u = u0; u < u1;) {
    const Part t = next_part(a, n_st, u, u1);
    const int st0 = t.st0, st1 = t.st1, slot = t.slot;
    Seg sg;
    sg.p0 = t.p0;
    sg.m = t.m;
    sg.slot = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<uint8_t*>(a.slab) + size_t(max(slot, 0)) * size_t(a.expert_bytes), 0,
        uint32_t(a.expert_bytes), 0x00027000);
    if (slot < 0) {  // not resident: exact zero rows of y (streaming.py:715-719)
      if constexpr (!DUAL) {
        const int nc = (st1 - st0) * K::kStepCols;
        for (int i = threadIdx.x; i < sg.m * nc; i += K::kThreads) {
          const int r = i / nc;
          static_cast<typename K::Out*>(
              a.out)[size_t(a.order[sg.p0 + r]) * a.out_cols + st0 * K::kStepCols + (i - r * nc)] = 0;
        }
      }
      continue;
    }
    if constexpr (!DUAL) {
      // output rows, read by the reduction after the first step's barrier;
      // two buffers, as the last step's readers may still hold the other
      if (int(threadIdx.x) < sg.m) s_row[par][threadIdx.x] = a.order[sg.p0 + threadIdx.x];
    }
    if constexpr (K::kMaxMT == 2) {
      if (sg.m > 16)
        K::template run<2>(a, sg, 0, st0, st1, part, buf, s_row[par], &s_odd);
      else
        K::template run<1>(a, sg, 0, st0, st1, part, buf, s_row[par], &s_odd);
    } else {
      for (int r0 = 0; r0 < sg.m; r0 += 16)
        K::template run<1>(a, sg, r0, st0, st1, part, buf, s_row[par], &s_odd);
    }
    par ^= 1;
  }
  block_lds_sync();
  if (__builtin_amdgcn_readfirstlane(s_odd)) {
    __builtin_amdgcn_s_waitcnt(0);  // this wave's stores, then every wave's
    __syncthreads();
    redo_range<BITS, NSL, K::kStepCols, DUAL, F32>(a, n_st, u0, u1);
  }
}

// Slices of a reduction of `cols` values: {groups a slice, slices}, or zeros
// where there is no cut.  The fewest waves whose x fits next to the ring at 32
// rows (6 or 8 groups); beyond 64 groups 8 waves of 10, 12 or 14, at 16 rows a
// pass.  Scales and biases are read as words, two groups each, so the count
// has to be even; and a row is at least a slice.  An uneven cut reads the
// groups its last slices share from L2 and multiplies them by zero: at most
// 1.4 times the arithmetic (34 groups, the first count of 8 waves).
struct Cut {
  int g, nsl;
};

Cut stream_cut(int cols) {
  const int n = cols / 64;
  if (cols % 128 || n < 6 || n > 112) return {0, 0};
  for (int nsl = 1; nsl <= 8; nsl *= 2)
    if (n <= 8 * nsl) return {n <= 6 * nsl ? 6 : 8, nsl};
  return {n <= 80 ? 10 : n <= 96 ? 12 : 14, 8};
}

// Blocks: every CU filled with 8 waves (two a SIMD).
constexpr int kCus = 256;

template <int BITS, bool DUAL, bool F32>
int launch_stream(const StreamArgs& a, hipStream_t st) {
  const Cut c = stream_cut(a.cols);
#define PMOE_CASE(G, NSL)                                                              \
  if (c.g == G && c.nsl == NSL) {                                                      \
    stream_kernel<BITS, G, NSL, DUAL, F32><<<kCus * (8 / NSL), 64 * NSL, 0, st>>>(a);       \
    PMOE_LAUNCH_CHECK("stream_kernel");                                                \
    return PMOE_OK;                                                                    \
  }
  PMOE_CASE(6, 1)
  PMOE_CASE(8, 1)
  PMOE_CASE(6, 2)
  PMOE_CASE(8, 2)
  PMOE_CASE(6, 4)
  PMOE_CASE(8, 4)
  PMOE_CASE(6, 8)
  PMOE_CASE(8, 8)
  if constexpr (BITS == 4) {
    PMOE_CASE(10, 8)
    PMOE_CASE(12, 8)
    PMOE_CASE(14, 8)
  }
#undef PMOE_CASE
  return fail(PMOE_EINVAL, "stream: unsupported reduction length");
}

}  // namespace

int stream_tile_rows() { return kStreamRows; }

// Shapes with a cut for both reductions, in slots that the buffer loads can
// address: a resource spans one slot (32-bit offsets; what lies outside reads
// as zero), so every component has to lie inside the slot's stride, on whole
// words.
bool stream_covers(const pmoe_geom* g, const void* slab) {
  const Cut gu = stream_cut(g->hidden), dn = stream_cut(g->inter);
  if (!gu.g || !dn.g || (g->bits == 6 && (gu.g > 8 || dn.g > 8))) return false;
  if (g->expert_bytes >= (int64_t(1) << 31)) return false;
  uintptr_t at = reinterpret_cast<uintptr_t>(slab) | uintptr_t(g->expert_bytes);
  const int64_t vals = int64_t(g->hidden) * g->inter;
  for (int c = 0; c < PMOE_NCOMP; ++c) {
    const int64_t bytes = c % 3 ? vals / 64 * 2 : vals * g->bits / 8;
    if (g->off[c] < 0 || g->off[c] + bytes > g->expert_bytes) return false;
    at |= uintptr_t(g->off[c]);
  }
  return at % 4 == 0;
}

int stream_experts(const pmoe_geom* g, const uint8_t* slab, const uint16_t* x, int n, int kk,
                   const int32_t* order, const int4* tiles, const int32_t* n_tiles, uint16_t* h,
                   void* y, int y_f32, hipStream_t st) {
  PMOE_REQUIRE(stream_covers(g, slab), "stream: unsupported shape");
  StreamArgs a{};
  a.slab = slab;
  a.expert_bytes = g->expert_bytes;
  a.order = order;
  a.tiles = tiles;
  a.n_tiles = n_tiles;
  a.act = x;
  a.kk = kk;
  a.cols = g->hidden;
  a.out_cols = g->inter;
  a.p0 = {g->off[PMOE_GATE_W], g->off[PMOE_GATE_S], g->off[PMOE_GATE_B]};
  a.p1 = {g->off[PMOE_UP_W], g->off[PMOE_UP_S], g->off[PMOE_UP_B]};
  a.out = h;
  a.out_vec = 1;
  {
    ProfScope prof_scope(K_PREFILL_GATEUP, st);
    const int rc = g->bits == 4 ? launch_stream<4, true, false>(a, st)
                                : launch_stream<6, true, false>(a, st);
    if (rc) return rc;
  }
  a.act = h;
  a.kk = 1;
  a.cols = g->inter;
  a.out_cols = g->hidden;
  a.p0 = a.p1 = {g->off[PMOE_DOWN_W], g->off[PMOE_DOWN_S], g->off[PMOE_DOWN_B]};
  a.out = y;
  a.out_vec = (reinterpret_cast<uintptr_t>(y) & 7) == 0;
  ProfScope prof_scope(K_PREFILL_DOWN, st);
  if (y_f32)
    return g->bits == 4 ? launch_stream<4, false, true>(a, st)
                        : launch_stream<6, false, true>(a, st);
  return g->bits == 4 ? launch_stream<4, false, false>(a, st)
                      : launch_stream<6, false, false>(a, st);
}

}  // namespace pmoe
