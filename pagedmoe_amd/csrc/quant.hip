// Affine group quantization format: quantize and dequantize kernels.
//
// Format (safetensors_index.py:8-25, bench/slab_probe.py:82): weight u32
// [rows, cols*bits/32] holding a little-endian bit stream per row (value i at
// stream bits [i*bits, i*bits+bits)), scales and biases bf16 [rows,
// cols/group], w = s*q + b.  A group of 64 values is 64*bits/32 whole words
// (8 for 4-bit, 12 for 6-bit) and rows are whole groups, so both kernels work
// on the flat list of groups: 8 lanes a group, 8 values a lane, a wave's 8
// groups contiguous in every array.
//
// Both are bound by HBM.  24576 x 4096, 4-bit: quantize 511 -> 88 us (5.2 TB/s),
// dequant 84 -> 56 us (4.6 TB/s), against one thread a group, whose loads and
// stores each touched one line a lane and whose quantize read its group twice
// and divided per value.
#include "pmoe_internal.h"

namespace pmoe {

namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Minimum and maximum over aligned groups of 8 lanes.
__device__ __forceinline__ void minmax8(float& lo, float& hi) {
  lo = fminf(lo, xor_lane<1>(lo)), hi = fmaxf(hi, xor_lane<1>(hi));
  lo = fminf(lo, xor_lane<2>(lo)), hi = fmaxf(hi, xor_lane<2>(hi));
  lo = fminf(lo, xor_lane<4>(lo)), hi = fmaxf(hi, xor_lane<4>(hi));
}

// VEC: w is 16-byte aligned.
template <int BITS, bool VEC>
__global__ __launch_bounds__(256) void quantize_kernel(const float* __restrict__ w, size_t groups,
                                                       uint32_t* __restrict__ q,
                                                       uint16_t* __restrict__ scales,
                                                       uint16_t* __restrict__ biases) {
  constexpr float kTop = float((1 << BITS) - 1);
  const size_t gid = size_t(blockIdx.x) * 32 + (threadIdx.x >> 3);
  const int sub = threadIdx.x & 7;
  const float* src = w + (gid < groups ? gid : groups - 1) * 64 + sub * 8;
  float v[8];
  if constexpr (VEC) {
    const f32x4 a = *reinterpret_cast<const f32x4*>(src);
    const f32x4 b = *reinterpret_cast<const f32x4*>(src + 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = a[i], v[i + 4] = b[i];
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = src[i];
  }
  float lo = v[0], hi = v[0];
#pragma unroll
  for (int i = 1; i < 8; ++i) lo = fminf(lo, v[i]), hi = fmaxf(hi, v[i]);
  minmax8(lo, hi);
  const float scale = (hi - lo) / kTop;
  uint16_t sb = f2bf(scale);
  if (bf16f(sb) == 0.0f) sb = 0x3F80;  // zero scale -> 1.0
  const uint16_t bb = f2bf(lo);
  const float s = bf16f(sb), b = bf16f(bb);
  // rint((x - b) / s) by the reciprocal, with the division where that could
  // differ.  In and near the code range |quotient| < 64, and the product is
  // within 4 ulp (2e-5) of the rounded quotient; further out both clamp to
  // the same end.  So only a product within 1e-4 of a half (one in 5000) or
  // a non-finite one (a scale or value that is not finite, or a denormal
  // scale) needs the division.
  const float r = __builtin_amdgcn_rcpf(s);
  float qf[8];
  bool redo = false;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float t = (v[i] - b) * r;
    qf[i] = __builtin_rintf(t);
    redo |= !(fabsf(t - qf[i]) < 0.4999f);
  }
  if (redo) {
#pragma unroll
    for (int i = 0; i < 8; ++i) qf[i] = __builtin_rintf((v[i] - b) / s);
  }
  uint32_t word = 0, next = 0;  // the lane's 32 or 48 bits
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t qi = uint32_t(fminf(fmaxf(qf[i], 0.0f), kTop));
    const int pos = i * BITS;
    if (pos < 32) word |= qi << pos;
    if (pos + BITS > 32) next |= pos < 32 ? qi >> (32 - pos) : qi << (pos - 32);
  }
  if (gid >= groups) return;
  if constexpr (BITS == 4) {
    q[gid * 8 + sub] = word;
  } else {
    uint16_t* dst = reinterpret_cast<uint16_t*>(q) + (gid * 8 + sub) * 3;
    dst[0] = uint16_t(word);
    dst[1] = uint16_t(word >> 16);
    dst[2] = uint16_t(next);
  }
  if (sub == 0) {
    scales[gid] = sb;
    biases[gid] = bb;
  }
}

// VEC: out is 16-byte aligned.
template <int BITS, bool VEC>
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t* __restrict__ q,
                                                      const uint16_t* __restrict__ scales,
                                                      const uint16_t* __restrict__ biases,
                                                      size_t groups, uint16_t* __restrict__ out) {
  const size_t gid = size_t(blockIdx.x) * 32 + (threadIdx.x >> 3);
  const int sub = threadIdx.x & 7;
  if (gid >= groups) return;
  uint64_t bits;  // the lane's 8 values
  if constexpr (BITS == 4) {
    bits = q[gid * 8 + sub];
  } else {
    // 48 bits from byte 6 sub of the group: within words 3 sub / 2 and the next
    const uint32_t* src = q + gid * 12 + (3 * sub >> 1);
    bits = (uint64_t(src[0]) | uint64_t(src[1]) << 32) >> (16 * (sub & 1));
  }
  const float s = bf16f(scales[gid]), b = bf16f(biases[gid]);
  uint32_t o[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t q0 = uint32_t(bits >> (2 * i * BITS)) & ((1u << BITS) - 1);
    const uint32_t q1 = uint32_t(bits >> ((2 * i + 1) * BITS)) & ((1u << BITS) - 1);
    o[i] = uint32_t(f2bf(__builtin_fmaf(s, float(q0), b))) |
           uint32_t(f2bf(__builtin_fmaf(s, float(q1), b))) << 16;
  }
  uint16_t* dst = out + gid * 64 + sub * 8;
  if constexpr (VEC) {
    *reinterpret_cast<u32x4*>(dst) = u32x4{o[0], o[1], o[2], o[3]};
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) dst[2 * i] = uint16_t(o[i]), dst[2 * i + 1] = uint16_t(o[i] >> 16);
  }
}

// A launch holds at most 2^32 - 1 threads, 8 to a group: longer arrays go out
// in several.  go(first group, groups, blocks).
template <class Go>
void each_launch(size_t groups, Go go) {
  constexpr size_t kMost = size_t(1) << 28;
  for (size_t g0 = 0; g0 < groups; g0 += kMost) {
    const size_t n = groups - g0 < kMost ? groups - g0 : kMost;
    go(g0, n, unsigned((n + 31) / 32));
  }
}

}  // namespace

int quantize(const float* w, int rows, int cols, int bits, int group, uint32_t* q,
             uint16_t* scales, uint16_t* biases, hipStream_t st) {
  PMOE_REQUIRE(w && q && scales && biases, "quantize: null pointer");
  PMOE_REQUIRE(group == 64, "quantize: only group size 64 is supported");
  PMOE_REQUIRE(bits == 4 || bits == 6, "quantize: bits must be 4 or 6");
  PMOE_REQUIRE(rows >= 0 && cols > 0 && cols % 64 == 0, "quantize: cols must be a multiple of 64");
  const size_t n = size_t(rows) * (cols / 64);
  if (n == 0) return PMOE_OK;
  const bool vec = reinterpret_cast<uintptr_t>(w) % 16 == 0;
  auto go = [&](auto kernel) {
    each_launch(n, [&](size_t g0, size_t groups, unsigned blocks) {
      kernel<<<blocks, 256, 0, st>>>(w + g0 * 64, groups, q + g0 * (2 * bits), scales + g0,
                                     biases + g0);
    });
  };
  if (bits == 4)
    vec ? go(quantize_kernel<4, true>) : go(quantize_kernel<4, false>);
  else
    vec ? go(quantize_kernel<6, true>) : go(quantize_kernel<6, false>);
  PMOE_LAUNCH_CHECK("quantize_kernel");
  return PMOE_OK;
}

int dequant(const uint32_t* q, const uint16_t* scales, const uint16_t* biases, int rows,
            int cols, int bits, int group, uint16_t* out, hipStream_t st) {
  PMOE_REQUIRE(q && scales && biases && out, "dequant: null pointer");
  PMOE_REQUIRE(group == 64, "dequant: only group size 64 is supported");
  PMOE_REQUIRE(bits == 4 || bits == 6, "dequant: bits must be 4 or 6");
  PMOE_REQUIRE(rows >= 0 && cols > 0 && cols % 64 == 0, "dequant: cols must be a multiple of 64");
  const size_t n = size_t(rows) * (cols / 64);
  if (n == 0) return PMOE_OK;
  const bool vec = reinterpret_cast<uintptr_t>(out) % 16 == 0;
  auto go = [&](auto kernel) {
    each_launch(n, [&](size_t g0, size_t groups, unsigned blocks) {
      kernel<<<blocks, 256, 0, st>>>(q + g0 * (2 * bits), scales + g0, biases + g0, groups,
                                     out + g0 * 64);
    });
  };
  if (bits == 4)
    vec ? go(dequant_kernel<4, true>) : go(dequant_kernel<4, false>);
  else
    vec ? go(dequant_kernel<6, true>) : go(dequant_kernel<6, false>);
  PMOE_LAUNCH_CHECK("dequant_kernel");
  return PMOE_OK;
}

}  // namespace pmoe

extern "C" int pmoe_quantize(const float* w, int rows, int cols, int bits, int group, uint32_t* q,
                             uint16_t* scales, uint16_t* biases, void* stream) {
  pmoe::clear_error();
  return pmoe::quantize(w, rows, cols, bits, group, q, scales, biases,
                        static_cast<hipStream_t>(stream));
}

extern "C" int pmoe_dequant(const uint32_t* q, const uint16_t* scales, const uint16_t* biases,
                            int rows, int cols, int bits, int group, uint16_t* out, void* stream) {
  pmoe::clear_error();
  return pmoe::dequant(q, scales, biases, rows, cols, bits, group, out,
                       static_cast<hipStream_t>(stream));
}
