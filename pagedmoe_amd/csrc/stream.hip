// Expert GEMMs for few rows per expert: every weight byte streamed once
// through registers into bf16 MFMA, activations held in registers.
//
// Replaces the per-expert quantized_matmul calls of the reference's grouped
// path (streaming.py:789-836) between the decode GEMV (one to a few rows an
// expert, decode.hip) and the prefill GEMMs (128-row tiles, prefill.hip).
// These sizes are bound by the weight stream, so the kernel is built around
// it:
//
//   * The reduction is cut into NSL slices of G quantization groups, one
//     wave each; a wave keeps its slice of the tile's 16 or 32 activation
//     rows in registers as MFMA operands for as long as the tile lasts, and
//     its inner loop only loads weights: tiles of 16 weight rows, a ring of
//     them in flight, read as 16-byte (4-bit) or 12-byte (6-bit) pieces,
//     64 or 48 contiguous bytes of each of 16 rows an instruction.
//   * Weights go into the MFMA as bf16 (128 + q), one and/or per pair
//     (gemv_common.h's form; the dequantized operand of prefill.hip takes 2.9
//     vector instructions a value, this 0.9): each group's product is scaled by
//     its s in fp32, and (b - 128 s) * sum(x) is added by one fp32 MFMA per
//     four groups, so no operand is rounded to bf16 but x itself.
//   * The slices' fp32 partial sums meet in LDS once per 16 columns (double
//     buffered, one LDS-only barrier, loads stay in flight across it).
//   * Work is the flat list (tile, 16-column block), cut into equal
//     contiguous ranges, one per resident block: every block streams the
//     same number of bytes whatever the expert loads are.
//
// Measured (Qwen3-235B shapes, 100 tokens, every expert active): gate/up 694
// -> 187 us (4.8 TB/s of weights), down 395 -> 109 us (4.2 TB/s) against the
// GEMV, which repeats its dot products for every row of an expert; the same
// loads without arithmetic, reduction and stores take 157 and 82 us.  8 waves
// a CU at 256 registers: x takes 128 of them at 32 rows.
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
typedef uint32_t u32x3_a4 __attribute__((ext_vector_type(3), aligned(4)));
typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kStreamRows = 32;   // rows of a dispatch tile
constexpr int kCols = 16;         // weight rows (output columns) of a step
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
  int out_vec;            // out is 16-byte aligned
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
  static constexpr int kS3 = (G % 8) / 2 == 3;    // then one of 3
  static_assert(kS4 * 8 + kS3 * 6 == G, "groups a slice: 8 i or 8 i + 6");
  V w[kV];
  u32x4_a4 s4[kS4 ? kS4 : 1], b4[kS4 ? kS4 : 1];
  u32x3_a4 s3, b3;
  __device__ __forceinline__ uint32_t word(int i) const {
    return BITS == 4 ? w[i >> 2][i & 3] : w[i / 3][i % 3];
  }
  __device__ __forceinline__ uint32_t s(int i) const {
    return i < 4 * kS4 ? s4[i < 4 * kS4 ? i >> 2 : 0][i & 3] : s3[i - 4 * kS4];
  }
  __device__ __forceinline__ uint32_t b(int i) const {
    return i < 4 * kS4 ? b4[i < 4 * kS4 ? i >> 2 : 0][i & 3] : b3[i - 4 * kS4];
  }
  // Opaque to the optimiser: without this, unpacking moves to the end of the
  // loop trip that loaded the words and waits for them there.
  __device__ __forceinline__ void pin() {
#pragma unroll
    for (int i = 0; i < kS4; ++i) asm volatile("" : "+v"(s4[i]), "+v"(b4[i]));
    if constexpr (kS3) asm volatile("" : "+v"(s3), "+v"(b3));
#pragma unroll
    for (int i = 0; i < kV; ++i) asm volatile("" : "+v"(w[i]));
  }
};

// Lane l of the tile owns weight row l % 16 and quarter kq = l / 16 of each
// group's 64 values.  4-bit: a load covers two groups, 16 bytes a lane, the
// lower lanes holding the first group's two halves and the upper lanes the
// second's; unpack_pair trades words between the wave's halves so that each
// register then holds one group.  6-bit: 12 bytes a lane and group.
template <int BITS, int G>
__device__ __forceinline__ void load_tile(WTile<BITS, G>& t, const uint8_t* w, uint32_t w_off,
                                          const uint8_t* s, const uint8_t* b, uint32_t s_off) {
  using T = WTile<BITS, G>;
#pragma unroll
  for (int i = 0; i < T::kV; ++i)
    t.w[i] = *reinterpret_cast<const typename T::V*>(w + w_off + (BITS == 4 ? 64 : 48) * i);
#pragma unroll
  for (int i = 0; i < T::kS4; ++i) {
    t.s4[i] = *reinterpret_cast<const u32x4_a4*>(s + s_off + 16 * i);
    t.b4[i] = *reinterpret_cast<const u32x4_a4*>(b + s_off + 16 * i);
  }
  if constexpr (T::kS3) {
    t.s3 = *reinterpret_cast<const u32x3_a4*>(s + s_off + 16 * T::kS4);
    t.b3 = *reinterpret_cast<const u32x3_a4*>(b + s_off + 16 * T::kS4);
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

template <int BITS, int G>
__device__ __forceinline__ void load_x(XTile<G>& x, const uint16_t* src, int kq) {
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
    float s = 0.0f;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const u32x4 d = x.a[g][c];
      s = dot2(d[3], kOnes, dot2(d[2], kOnes, dot2(d[1], kOnes, dot2(d[0], kOnes, s))));
      if constexpr (BITS == 4)  // pairs (x_i, x_{i+4}), as nib_pair unpacks
        x.a[g][c] = u32x4{__builtin_amdgcn_perm(d[2], d[0], 0x05040100u),
                          __builtin_amdgcn_perm(d[2], d[0], 0x07060302u),
                          __builtin_amdgcn_perm(d[3], d[1], 0x05040100u),
                          __builtin_amdgcn_perm(d[3], d[1], 0x07060302u)};
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

// A block's current tile.
struct Seg {
  const uint8_t* base;  // the expert's slot
  int p0, m;            // first sorted row, rows
};

template <int BITS, int G, int NSL, bool DUAL, bool F32>
struct StreamKernel {
  static constexpr int NP = DUAL ? 2 : 1;
  static constexpr int kThreads = 64 * NSL;
  static constexpr int kMaxMT = G <= 8 ? 2 : 1;  // 32 rows of x fit next to the ring
  static constexpr int kLds = 2 * NP * kMaxMT * NSL * kPart;
  // Output tile: two groups of 64 columns, rows padded by 16 bytes.
  using Out = std::conditional_t<F32, float, uint16_t>;
  static constexpr int kOutRows = 16 * kMaxMT;
  static constexpr int kOutPitch = 64 + 16 / int(sizeof(Out));

  // Weight tiles in flight: what fits in 256 registers next to x.
  template <int MT>
  static constexpr int ring() {
    constexpr int per = WTile<BITS, G>::kRegs + G;
    constexpr int room = 256 - (BITS == 4 ? 48 : MT == 1 ? 52 : 64) - MT * (8 * G + (G + 3) / 4) - NP * MT * 4;
    constexpr int r = room / per;
    constexpr int c = r > 4 ? 4 : r;
    return c < NP ? NP : c / NP * NP;
  }

  // Columns [ct0, ct1) (units of 16) of rows [r0, r0 + 16 MT) of the segment.
  template <int MT>
  static __device__ __forceinline__ void run(const StreamArgs& a, const Seg& sg, int r0, int ct0,
                                             int ct1, float* part, int& buf, Out* ot,
                                             const int32_t* s_row) {
    constexpr int E = ring<MT>();
    constexpr int SR = E / NP;  // steps in flight
    const int lane = threadIdx.x & 63;
    const int slice = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, kq = lane >> 4;
    const int m = sg.m - r0;
    const uint32_t row_bytes = uint32_t(a.cols) * BITS / 8;
    const uint32_t groups = uint32_t(a.cols) / 64;
    const uint32_t w_off = row * row_bytes + kq * (BITS == 4 ? 16 : 12);
    const uint32_t s_off = row * groups * 2;
    const uint8_t* wb[2];
    const uint8_t* sb[2];
    const uint8_t* bb[2];
#pragma unroll
    for (int p = 0; p < NP; ++p) {
      const QProj& q = p ? a.p1 : a.p0;
      wb[p] = sg.base + q.w + slice * (G * 64 * BITS / 8);
      sb[p] = sg.base + q.s + slice * (G * 2);
      bb[p] = sg.base + q.b + slice * (G * 2);
    }
    WTile<BITS, G> W[E];
    auto load = [&](int e, int ct) {
      const int p = e % NP;
      load_tile<BITS, G>(W[e], wb[p] + size_t(ct) * kCols * row_bytes, w_off,
                         sb[p] + size_t(ct) * kCols * groups * 2,
                         bb[p] + size_t(ct) * kCols * groups * 2, s_off);
    };
    int ar[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int r = sg.p0 + r0 + min(16 * mt + row, m - 1);  // rows past the tile: its last row
      ar[mt] = DUAL ? a.order[r] / a.kk : r;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) load(e, min(ct0 + e / NP, ct1 - 1));
    __builtin_amdgcn_sched_barrier(0);
    XTile<G> x[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      load_x<BITS, G>(x[mt], a.act + size_t(ar[mt]) * a.cols + slice * (G * 64) +
                                 quarter_k<BITS>(kq), kq);
    // Everything so far has arrived (the activations, requested last, are
    // needed at once): with nothing pending on entry, the compiler's wait
    // counts at the loop head are those of the steady state.  Left pending
    // in an order of the compiler's choosing, it waited there for the whole
    // ring on every trip.
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
    __builtin_amdgcn_sched_barrier(0);
    for (int c = ct0; c < ct1; c += SR) {
#pragma unroll
      for (int v = 0; v < SR; ++v) {
        // past the range: the last column again, the same values to the
        // same place (an exit here would cost register copies that wait for
        // the ring)
        const int ct = min(c + v, ct1 - 1);
        float* pb = part + buf * (NP * kMaxMT * NSL * kPart);
#pragma unroll
        for (int p = 0; p < NP; ++p) {
          f32x4 acc[MT];
          tile_mfma<BITS, G, MT>(W[v * NP + p], x, kq, acc);
          __builtin_amdgcn_sched_barrier(0);
          load(v * NP + p, min(ct + SR, ct1 - 1));
          __builtin_amdgcn_sched_barrier(0);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              pb[((p * kMaxMT + mt) * NSL + slice) * kPart + 64 * r + lane] = acc[mt][r];
        }
        block_lds_sync();
        // the step before this one completed a 64-column group: it goes out
        if ((ct & 3) == 0 && ct != ct0) flush(a, sg, r0, m, (ct >> 2) - 1, ct0, ct1, ot, s_row);
        // Sum the slices into the output tile.  Rows past the tile repeat its
        // last row and are never stored; threads beyond the outputs repeat
        // the first ones'.
        constexpr int J = MT * 256 > kThreads ? MT * 256 / kThreads : 1;
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int e = (int(threadIdx.x) + j * kThreads) % (MT * 256);
          const int mt = e >> 8;
          float v[2];
#pragma unroll
          for (int p = 0; p < NP; ++p) {
            const float* q = pb + (p * kMaxMT + mt) * NSL * kPart + (e & 255);
            v[p] = q[0];
#pragma unroll
            for (int sl = 1; sl < NSL; ++sl) v[p] += q[sl * kPart];
          }
          const float o = DUAL ? silu_fast(v[0]) * v[1] : v[0];
          Out* d = ot + (ct & 4) / 4 * (kOutRows * kOutPitch) +
                   (16 * mt + 4 * ((e >> 4) & 3) + ((e >> 6) & 3)) * kOutPitch +
                   (ct & 3) * kCols + (e & 15);
          if constexpr (F32)
            *d = o;
          else
            *d = f2bf(o);
        }
        buf ^= 1;
      }
    }
    block_lds_sync();
    flush(a, sg, r0, m, (ct1 - 1) >> 2, ct0, ct1, ot, s_row);
  }

  // Rows [0, m) of the 64-column group gi of the output tile, its columns
  // within [ct0, ct1), as 16-byte pieces of whole lines.  (Stored by the step,
  // 16 columns at a time, the short stores took a tenth of the gate/up
  // launch: loads and stores share one counter, so the loads behind a store
  // wait for its acknowledgement.)
  static __device__ __forceinline__ void flush(const StreamArgs& a, const Seg& sg, int r0, int m,
                                               int gi, int ct0, int ct1, const Out* ot,
                                               const int32_t* s_row) {
    constexpr int kPieces = 64 * sizeof(Out) / 16;
    constexpr int kVals = 16 / sizeof(Out);
    const Out* src = ot + (gi & 1) * (kOutRows * kOutPitch);
    for (int i = threadIdx.x; i < m * kPieces; i += kThreads) {
      const int r = i / kPieces, pc = i % kPieces;
      const int ct = 4 * gi + pc / (kPieces / 4);
      if (ct < ct0 || ct >= ct1) continue;
      const int orow = DUAL ? sg.p0 + r0 + r : s_row[r0 + r];
      Out* dst = static_cast<Out*>(a.out) + size_t(orow) * a.out_cols + 64 * gi + kVals * pc;
      const Out* q = src + r * kOutPitch + kVals * pc;
      if (a.out_vec)
        *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(q);
      else
#pragma unroll
        for (int j = 0; j < kVals; ++j) dst[j] = q[j];
    }
  }
};

template <int BITS, int G, int NSL, bool DUAL, bool F32>
__global__ __launch_bounds__(64 * NSL, 2) void stream_kernel(const StreamArgs a) {
  using K = StreamKernel<BITS, G, NSL, DUAL, F32>;
  typedef const __attribute__((address_space(4))) int32_t ConstI32;
  __shared__ float part[K::kLds];
  __shared__ __attribute__((aligned(16))) typename K::Out ot[2 * K::kOutRows * K::kOutPitch];
  __shared__ int32_t s_row[2][kStreamRows];
  const int n_ct = a.out_cols / kCols;
  const int64_t total = int64_t(*(ConstI32*)a.n_tiles) * n_ct;
  const int64_t u1 = total * (blockIdx.x + 1) / gridDim.x;
  int64_t u = total * blockIdx.x / gridDim.x;
  int buf = 0, par = 0;
  while (u < u1) {
    const int tile = int(u / n_ct);
    const int ct0 = int(u - int64_t(tile) * n_ct);
    const int ct1 = int(min(int64_t(n_ct), ct0 + (u1 - u)));
    u += ct1 - ct0;
    ConstI32* tl = (ConstI32*)(a.tiles + tile);
    const int slot = tl[0], first = tl[1], cnt = tl[2], off = tl[3];
    Seg sg;
    sg.p0 = off + first;
    sg.m = min(kStreamRows, cnt - first);
    sg.base = a.slab + size_t(max(slot, 0)) * size_t(a.expert_bytes);
    if (slot < 0) {  // not resident: exact zero rows of y (streaming.py:715-719)
      if constexpr (!DUAL) {
        const int nc = (ct1 - ct0) * kCols;
        for (int i = threadIdx.x; i < sg.m * nc; i += K::kThreads) {
          const int r = i / nc;
          const size_t o = size_t(a.order[sg.p0 + r]) * a.out_cols + ct0 * kCols + (i - r * nc);
          if constexpr (F32)
            static_cast<float*>(a.out)[o] = 0.0f;
          else
            static_cast<uint16_t*>(a.out)[o] = 0;
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
        K::template run<2>(a, sg, 0, ct0, ct1, part, buf, ot, s_row[par]);
      else
        K::template run<1>(a, sg, 0, ct0, ct1, part, buf, ot, s_row[par]);
    } else {
      for (int r0 = 0; r0 < sg.m; r0 += 16)
        K::template run<1>(a, sg, r0, ct0, ct1, part, buf, ot, s_row[par]);
    }
    par ^= 1;
  }
}

// Slices of a reduction of `cols` values: {groups a slice, slices}, or zeros.
struct Cut {
  int g, nsl;
};

Cut stream_cut(int cols) {
  switch (cols) {
    case 512: return {8, 1};
    case 1024: return {8, 2};
    case 1536: return {6, 4};
    case 2048: return {8, 4};
    case 4096: return {8, 8};
    case 7168: return {14, 8};
    default: return {0, 0};
  }
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
  PMOE_CASE(8, 1)
  PMOE_CASE(8, 2)
  PMOE_CASE(6, 4)
  PMOE_CASE(8, 4)
  PMOE_CASE(8, 8)
  if constexpr (BITS == 4) {
    PMOE_CASE(14, 8)
  }
#undef PMOE_CASE
  return fail(PMOE_EINVAL, "stream: unsupported reduction length");
}

}  // namespace

int stream_tile_rows() { return kStreamRows; }

bool stream_covers(const pmoe_geom* g) {
  const Cut gu = stream_cut(g->hidden), dn = stream_cut(g->inter);
  return gu.g && dn.g && (g->bits == 4 || (gu.g <= 8 && dn.g <= 8));
}

int stream_experts(const pmoe_geom* g, const uint8_t* slab, const uint16_t* x, int n, int kk,
                   const int32_t* order, const int4* tiles, const int32_t* n_tiles, uint16_t* h,
                   void* y, int y_f32, hipStream_t st) {
  PMOE_REQUIRE(stream_covers(g), "stream: unsupported shape");
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
  a.out_vec = (reinterpret_cast<uintptr_t>(y) & 15) == 0;
  ProfScope prof_scope(K_PREFILL_DOWN, st);
  if (y_f32)
    return g->bits == 4 ? launch_stream<4, false, true>(a, st)
                        : launch_stream<6, false, true>(a, st);
  return g->bits == 4 ? launch_stream<4, false, false>(a, st)
                      : launch_stream<6, false, false>(a, st);
}

}  // namespace pmoe
