// GPU quantizer: one wave per (row, group). Each lane owns value pairs (2 l, 2 l + 1) + 128 j of the group, so the
// packed byte of a pair is formed in one lane. With no clip grid the result is bit-identical to the canonical
// absmax quantizer (reference lowbit/quant.py:23-35): scale = fp16(amax / 7) with a correctly rounded fp32 division,
// q = clamp(round_half_even(w / fp32(scale)), -8, 7). With a grid it follows the reference's clip search
// (lowbit/ops.py:98-112): per candidate a, scale = fp16(fp32(amax * a) / 7), zero -> 1, squared error summed in
// fp32 (wave-tree order), strictly better replaces the best so ties keep the earlier candidate.
#include "kernels.hpp"

namespace lowbit {

namespace {

template <int kDtype>
__device__ __forceinline__ float load_w(const void* w, size_t i) {
  if (kDtype == 0) return reinterpret_cast<const float*>(w)[i];
  if (kDtype == 1) return (float)reinterpret_cast<const f16*>(w)[i];
  const uint32_t b = reinterpret_cast<const uint16_t*>(w)[i];
  return __builtin_bit_cast(float, b << 16);
}

__device__ __forceinline__ float quantize_one(float v, float scf) {
  return fminf(fmaxf(__builtin_rintf(v / scf), -8.0f), 7.0f);
}

}  // namespace

constexpr int kMaxPairsPerLane = 8;     // groups up to 1024 values

template <int kDtype>
__global__ __launch_bounds__(256) void quantize_kernel(const void* __restrict__ w, uint8_t* __restrict__ packed,
                                                       f16* __restrict__ scales, int N, int K, int G, ClipGrid grid) {
  const int lane = threadIdx.x & 63;
  const size_t group = (size_t)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int KG = K / G;
  if (group >= (size_t)N * KG) return;
  const size_t n = group / KG, g = group % KG;
  const size_t base = n * K + g * G;
  const int npairs = G / 2;
  float v0[kMaxPairsPerLane], v1[kMaxPairsPerLane];
  float amax = 0.f;
#pragma unroll
  for (int j = 0; j < kMaxPairsPerLane; ++j) {
    const int p = lane + 64 * j;
    v0[j] = v1[j] = 0.f;
    if (p < npairs) {
      v0[j] = load_w<kDtype>(w, base + 2 * p);
      v1[j] = load_w<kDtype>(w, base + 2 * p + 1);
      amax = fmaxf(amax, fmaxf(fabsf(v0[j]), fabsf(v1[j])));
    }
  }
  amax = wave_max(amax);
  const int ncand = grid.n > 0 ? grid.n : 1;
  f16 best_sc = (f16)1.0f;
  float best_err = 0.f;
  for (int ci = 0; ci < ncand; ++ci) {
    const float a = grid.n > 0 ? grid.a[ci] : 1.0f;
    const float num = a != 1.0f ? amax * a : amax;
    f16 sc = (f16)(num / 7.0f);
    if (sc == (f16)0.0f) sc = (f16)1.0f;
    if (grid.n == 0) {
      best_sc = sc;
      break;
    }
    const float scf = (float)sc;
    float err = 0.f;
#pragma unroll
    for (int j = 0; j < kMaxPairsPerLane; ++j) {
      if (lane + 64 * j < npairs) {
        const float e0 = quantize_one(v0[j], scf) * scf - v0[j];
        const float e1 = quantize_one(v1[j], scf) * scf - v1[j];
        err += e0 * e0 + e1 * e1;
      }
    }
    err = wave_sum(err);
    if (ci == 0 || err < best_err) {
      best_err = err;
      best_sc = sc;
    }
  }
  const float scf = (float)best_sc;
#pragma unroll
  for (int j = 0; j < kMaxPairsPerLane; ++j) {
    const int p = lane + 64 * j;
    if (p < npairs) {
      const uint32_t u0 = (uint32_t)(int)(quantize_one(v0[j], scf) + 8.0f);
      const uint32_t u1 = (uint32_t)(int)(quantize_one(v1[j], scf) + 8.0f);
      packed[base / 2 + p] = (uint8_t)(u0 | (u1 << 4));
    }
  }
  if (lane == 0) scales[group] = best_sc;
}

// Groups of 32, 64 and 128 values: LPG = 4, 8 or 16 lanes a group, 8 consecutive values a lane, so that a wave quantizes
// 16, 8 or 4 groups at once from 16-byte loads. The same bits as quantize_kernel: its lane l holds values 2 l and 2 l + 1,
// so a lane here holds the pairs of one of its quads; their squared errors are added as wave_sum adds that quad, the rest
// of its tree is the same tree over the lanes here, and its idle lanes add zeros.
// The clip search evaluates v / scale for every value and candidate. A quotient is formed from the reciprocal y = RN(1 /
// scale), one division per lane and candidate: q0 = RN(v y), r = v - q0 scale, q = RN(q0 + r y), Markstein's correction
// (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", IBM J. Res. Dev. 34, 1990).
// It is the correctly rounded quotient: the scale is an fp16 value, so its 11 bits make r exact and keep v / scale at least
// 2^-12 ulp away from every rounding boundary, far more than the ~2^-22 ulp that y's error can move the sum by; an infinite
// scale, whose reciprocal says nothing, and a group whose largest quotient overflows (a clip factor near 0 on weights near
// fp32's largest; q0 would be infinite and r not a number) take the division itself.
// Bound: vector instructions (8 per value and candidate; the division took ~10 by itself). 11008 x 2048 fp16, 11
// candidates, MI355X: quantize_kernel 207 us, 63 here.
template <int kDtype>
__device__ __forceinline__ void load8(const void* w, size_t i, float (&v)[8]) {
  if constexpr (kDtype == 0) {
    const f32x4 a = reinterpret_cast<const f32x4*>(w)[i / 4], b = reinterpret_cast<const f32x4*>(w)[i / 4 + 1];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = a[e], v[4 + e] = b[e];
  } else {
    const u32x4 t = load16(reinterpret_cast<const uint16_t*>(w) + i);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      if constexpr (kDtype == 1) {
        v[2 * e] = (float)as_f16x2(t[e])[0];
        v[2 * e + 1] = (float)as_f16x2(t[e])[1];
      } else {
        v[2 * e] = __builtin_bit_cast(float, t[e] << 16);
        v[2 * e + 1] = __builtin_bit_cast(float, t[e] & 0xFFFF0000u);
      }
    }
  }
}

template <int kDtype, int LPG>
__global__ __launch_bounds__(256) void quantize_groups(const void* __restrict__ w, uint32_t* __restrict__ packed,
                                                       f16* __restrict__ scales, long lanes, ClipGrid grid) {
  const long gid = (long)blockIdx.x * 256 + threadIdx.x;
  const bool live = gid < lanes;                            // a group's lanes are live together
  float v[8];
  load8<kDtype>(w, 8 * (size_t)(live ? gid : 0), v);
  // over the lanes of a group: after the quad steps every quad is uniform, after lane ^ 7 every eight
  auto over_group = [](float x, auto op) {
    x = op(x, dpp<kQuadSwap1>(x));
    x = op(x, dpp<kQuadSwap2>(x));
    if (LPG >= 8) x = op(x, dpp<kRowHalfMirror>(x));
    if (LPG >= 16) x = op(x, dpp<kRowMirror>(x));
    return x;
  };
  float amax = 0.f;
#pragma unroll
  for (int e = 0; e < 8; e += 2) amax = fmaxf(amax, fmaxf(fabsf(v[e]), fabsf(v[e + 1])));
  amax = over_group(amax, [](float a, float b) { return fmaxf(a, b); });
  auto quantize8 = [&](float scf, auto each) {              // each(e, quantized value), e = 0..7
    const float y = 1.0f / scf;
    if (__any(__builtin_isinf(scf) || __builtin_isinf(amax * y))) {
#pragma unroll
      for (int e = 0; e < 8; ++e) each(e, quantize_one(v[e], scf));
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float q0 = v[e] * y, r = fmaf(-q0, scf, v[e]);
        each(e, fminf(fmaxf(__builtin_rintf(fmaf(r, y, q0)), -8.0f), 7.0f));
      }
    }
  };
  const int ncand = grid.n > 0 ? grid.n : 1;
  f16 best_sc = (f16)1.0f;
  float best_err = 0.f;
  for (int ci = 0; ci < ncand; ++ci) {
    const float a = grid.n > 0 ? grid.a[ci] : 1.0f;
    const float num = a != 1.0f ? amax * a : amax;
    f16 sc = (f16)(num / 7.0f);
    if (sc == (f16)0.0f) sc = (f16)1.0f;
    if (grid.n == 0) {
      best_sc = sc;
      break;
    }
    const float scf = (float)sc;
    float d[8];
    quantize8(scf, [&](int e, float q) { d[e] = q * scf - v[e]; });
    float pair[4];                                          // as quantize_kernel's multiply and fused multiply-add round it
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float e1 = d[2 * e + 1];
      pair[e] = fmaf(d[2 * e], d[2 * e], e1 * e1);
      asm("" : "+v"(pair[e]));                              // (not fused into the sums below)
    }
    const float err = over_group((pair[0] + pair[1]) + (pair[2] + pair[3]), [](float x, float z) { return x + z; });
    if (ci == 0 || err < best_err) {
      best_err = err;
      best_sc = sc;
    }
  }
  if (!live) return;
  const float scf = (float)best_sc;
  uint32_t word = 0;
  quantize8(scf, [&](int e, float q) { word |= (uint32_t)(int)(q + 8.0f) << (4 * e); });
  packed[gid] = word;
  if (gid % LPG == 0) scales[gid / LPG] = best_sc;
}

namespace {
template <int kDtype>
hipError_t launch_groups(const void* w, uint8_t* packed, f16* scales, long lanes, int G, const ClipGrid& grid,
                         hipStream_t st) {
  const dim3 gr((unsigned)((lanes + 255) / 256)), block(256);
  uint32_t* words = reinterpret_cast<uint32_t*>(packed);
  if (G == 32) return launch(quantize_groups<kDtype, 4>, gr, block, 0, st, w, words, scales, lanes, grid);
  if (G == 64) return launch(quantize_groups<kDtype, 8>, gr, block, 0, st, w, words, scales, lanes, grid);
  return launch(quantize_groups<kDtype, 16>, gr, block, 0, st, w, words, scales, lanes, grid);
}
}  // namespace

hipError_t quantize_launch(const void* w, int dtype, uint8_t* packed, f16* scales, int N, int K, int G,
                           const ClipGrid& grid, hipStream_t st) {
  const size_t groups = (size_t)N * (K / G);
  // other group sizes, and tensors that 16-byte loads or 4-byte stores do not fit, take the kernel of a wave per group
  if ((G == 32 || G == 64 || G == 128) && (reinterpret_cast<uintptr_t>(w) & 15) == 0 &&
      (reinterpret_cast<uintptr_t>(packed) & 3) == 0) {
    const long lanes = (long)groups * (G / 8);
    switch (dtype) {
      case 0: return launch_groups<0>(w, packed, scales, lanes, G, grid, st);
      case 1: return launch_groups<1>(w, packed, scales, lanes, G, grid, st);
      default: return launch_groups<2>(w, packed, scales, lanes, G, grid, st);
    }
  }
  dim3 gr((unsigned)((groups + 3) / 4)), block(256);
  switch (dtype) {
    case 0: return launch(quantize_kernel<0>, gr, block, 0, st, w, packed, scales, N, K, G, grid);
    case 1: return launch(quantize_kernel<1>, gr, block, 0, st, w, packed, scales, N, K, G, grid);
    default: return launch(quantize_kernel<2>, gr, block, 0, st, w, packed, scales, N, K, G, grid);
  }
}

}  // namespace lowbit
