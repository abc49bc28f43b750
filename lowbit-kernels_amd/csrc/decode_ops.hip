// Decode-step neighbours of the W4A16 projections in a Qwen2 decoder layer, so that one layer is nine launches
// instead of the ~50 the stock PyTorch modules issue per token: RMSNorm, RoPE fused with the KV-cache write, and
// causal GQA attention over the cache. Each follows the arithmetic of the module it replaces (transformers
// Qwen2RMSNorm, apply_rotary_pos_emb + StaticCache.update, scaled_dot_product_attention with a causal mask), with
// the same fp16 roundings where the torch ops round.
#include <algorithm>
#include <cfloat>
#include <climits>

#include "kernels.hpp"

namespace lowbit {

namespace {

constexpr int kHeadDim = kAttnHeadDim;

__device__ __forceinline__ float block_sum(float v, float* red) {    // all threads of the block get the total
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[wave] = v;
  __syncthreads();
  float t = 0.f;
  for (int i = 0; i < nw; ++i) t += red[i];
  return t;
}

}  // namespace

// out[m] = w * fp16(x[m] / sqrt(mean(x[m]^2) + eps)), one block per row (Qwen2RMSNorm: the normalisation in fp32,
// rounded to fp16, then the fp16 product with the weight). The first kNormPieces 16-byte pieces of x and w per thread
// (H <= 8192 at 256 threads) are loaded once, before the block reduction, and kept in registers for the output: one
// memory round trip instead of two; longer rows reload the rest.
constexpr int kNormPieces = 4;
__global__ __launch_bounds__(256) void rmsnorm_kernel(const f16* __restrict__ x, const f16* __restrict__ w,
                                                      f16* __restrict__ out, int H, float eps) {
  __shared__ float red[4];
  const size_t row = (size_t)blockIdx.x * H;
  const int step = blockDim.x * 8;
  u32x4 xv[kNormPieces], wv[kNormPieces];
#pragma unroll
  for (int c = 0; c < kNormPieces; ++c) {
    const int i = threadIdx.x * 8 + c * step;
    if (i < H) {
      xv[c] = *reinterpret_cast<const u32x4*>(x + row + i);
      wv[c] = *reinterpret_cast<const u32x4*>(w + i);
    }
  }
  float ss = 0.f;
  auto add_squares = [&](const u32x4& v) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f16x2 p = as_f16x2(v[j]);
      ss = fmaf((float)p[0], (float)p[0], ss);
      ss = fmaf((float)p[1], (float)p[1], ss);
    }
  };
#pragma unroll
  for (int c = 0; c < kNormPieces; ++c)
    if (threadIdx.x * 8 + c * step < H) add_squares(xv[c]);
  for (int i = threadIdx.x * 8 + kNormPieces * step; i < H; i += step) add_squares(*reinterpret_cast<const u32x4*>(x + row + i));
  const float r = rsqrtf(block_sum(ss, red) / (float)H + eps);
  auto store_norm = [&](int i, const u32x4& v, const u32x4& g) {
    *reinterpret_cast<u32x4*>(out + row + i) = rms_apply8(v, g, r);
  };
#pragma unroll
  for (int c = 0; c < kNormPieces; ++c) {
    const int i = threadIdx.x * 8 + c * step;
    if (i < H) store_norm(i, xv[c], wv[c]);
  }
  for (int i = threadIdx.x * 8 + kNormPieces * step; i < H; i += step)
    store_norm(i, *reinterpret_cast<const u32x4*>(x + row + i), *reinterpret_cast<const u32x4*>(w + i));
}

// qkv [M][(Hq + 2 Hkv) D] (the fused projection's output, bias included) -> q_out [M][Hq][D] with RoPE; k (with
// RoPE) and v written to k_cache / v_cache [Hkv][L][D] at row positions[m]. One thread per (token, head, dim pair
// (i, i + 64)), RoPE by rope_pair. permuted: qkv holds each head's rows in the RoPE-permuted order (rope_row), as the
// fused decoder's W4A16 q|k|v projection writes them.
__global__ __launch_bounds__(256) void rope_kv_kernel(const f16* __restrict__ qkv, const int64_t* __restrict__ pos,
                                                      const float* __restrict__ inv_freq, f16* __restrict__ q_out,
                                                      f16* __restrict__ k_cache, f16* __restrict__ v_cache, int M,
                                                      int Hq, int Hkv, int L, bool permuted) {
  const int heads = Hq + 2 * Hkv;
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  const int i = gid & 63, h = (gid >> 6) % heads, m = (gid >> 6) / heads;
  if (m >= M) return;
  const int64_t p = pos[m];
  if (p < 0 || p >= L) return;                               // the host checks positions; never write out of bounds
  const f16* src = qkv + ((size_t)m * heads + h) * kHeadDim;
  const int s1 = permuted ? rope_row(i) : i, s2 = permuted ? rope_row(i) + 8 : i + 64;   // dims i and i + 64
  if (h >= Hq + Hkv) {                                       // v: plain copy into the cache
    f16* dst = v_cache + ((size_t)(h - Hq - Hkv) * L + p) * kHeadDim;
    dst[i] = src[s1];
    dst[i + 64] = src[s2];
    return;
  }
  f16 o1, o2;
  rope_pair(src[s1], src[s2], p, inv_freq[i], o1, o2);
  f16* dst = h < Hq ? q_out + ((size_t)m * Hq + h) * kHeadDim : k_cache + ((size_t)(h - Hq) * L + p) * kHeadDim;
  dst[i] = o1;
  dst[i + 64] = o2;
}

// Causal GQA attention for M query tokens at positions pos[m] over the cache rows 0 .. pos[m]:
// out[m][h * D + d] = sum_j softmax_j(scale * q[m][h] . k[j]) v[j][d], KV head h / (Hq / Hkv) for query head h.
// One block of W waves per (token, group of G consecutive query heads of one KV head): G = Hq / Hkv shares every K/V
// read among the heads; G = 1 gives Hq / Hkv times more blocks (decode steps, where M Hkv blocks cannot fill the
// chip). Lane l always owns dims 8 (l % 16) .. + 7 and key row-group l / 16: each 16-byte K and V load of a wave
// reads four whole cache rows, the lane's slice of q stays in registers, a score is a 16-lane DPP sum, and the
// probabilities never leave the lane that multiplies them into V. Waves take blocks of KB keys; the row groups and
// the waves are merged at the end (lane shuffles, then LDS).
// When (token, group) blocks alone cannot fill the chip (a decode step), the keys are also split into P partitions
// of CH keys (grid.y): each block writes its partial (max, sum, unnormalized output) to the workspace and
// attention_combine, launched next, merges the P partials in partition order (merge_partitions). A merge by the last
// block to arrive (agent-coherent partial stores, an arrival counter per (token, group)) measured slower in graph
// decode (3B: 1.139 against 1.124 ms/token): phase stamps put 1.8 us on the arrival count alone, the P blocks of a
// (token, group) incrementing one counter, and 2.6 us on the last block's merge, against ~3 us for the key loop.
// Output dim d of one (block, head) from the P <= kAttnMaxParts partial records (kAttnRec floats) at float index `first`,
// `stride` floats apart: max over partitions, then the rescaled sums in partition order (partitions that saw no key
// hold max = -inf and are skipped; partition 0 always holds key 0). The loops run to the compile-time bound, so all
// the loads are requested before the first is used.
__device__ __forceinline__ float merge_partitions(__amdgpu_buffer_rsrc_t pr, int first, int stride, int P, int d) {
  float pm[kAttnMaxParts], ps[kAttnMaxParts], po[kAttnMaxParts];
#pragma unroll
  for (int p = 0; p < kAttnMaxParts; ++p) {
    const int at = 4 * (first + p * stride);
    const bool live = p < P;
    pm[p] = live ? load_partial(pr, at) : -INFINITY;
    ps[p] = live ? load_partial(pr, at + 4) : 0.f;
    po[p] = live ? load_partial(pr, at + 4 * (4 + d)) : 0.f;
  }
  float gm = -INFINITY;
#pragma unroll
  for (int p = 0; p < kAttnMaxParts; ++p) gm = fmaxf(gm, pm[p]);
  float num = 0.f, den = 0.f;
#pragma unroll
  for (int p = 0; p < kAttnMaxParts; ++p) {
    if (pm[p] == -INFINITY) continue;
    const float f = expf(pm[p] - gm);
    num = fmaf(f, po[p], num);
    den = fmaf(f, ps[p], den);
  }
  return num / den;
}

// the block bx of (token, head group)s, partition pid of P, whose partial goes to records `rec` ..
template <int G, int KB>
__device__ __forceinline__ void attend_heads(const f16* __restrict__ q, const f16* __restrict__ k_cache,
                                             const f16* __restrict__ v_cache, const int64_t* __restrict__ pos,
                                             f16* __restrict__ out, int Hq, int Hkv, int L, float scale, int CH,
                                             float* __restrict__ part, uint8_t* smem, int bx, int pid, int P, size_t rec) {
  constexpr int NI = KB / 4;                                 // 16-byte loads per lane and step, per K and per V
  const int groups = Hq / G;
  const int m = bx / groups, h0 = (bx % groups) * G, hk = h0 / (Hq / Hkv);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), W = blockDim.x >> 6;
  const int rg = lane >> 4, dl = (lane & 15) * 8;          // key row-group, first dim of the lane's slice
  const int64_t pm = pos[m];
  const int nkeys = (int)min((int64_t)L, pm + 1), last = nkeys - 1;
  const int kbeg = pid * CH, kend = pid == P - 1 ? nkeys : min(nkeys, kbeg + CH);   // this block's keys
  u32x4 qv[G];
#pragma unroll
  for (int g = 0; g < G; ++g) qv[g] = *reinterpret_cast<const u32x4*>(q + ((size_t)m * Hq + h0 + g) * kHeadDim + dl);
  const f16* kb = k_cache + (size_t)hk * L * kHeadDim + dl;
  const f16* vb = v_cache + (size_t)hk * L * kHeadDim + dl;
  float mx[G], sum[G], o[G][8];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    mx[g] = -INFINITY;
    sum[g] = 0.f;
#pragma unroll
    for (int d = 0; d < 8; ++d) o[g][d] = 0.f;
  }
  for (int base = kbeg + wave * KB; base < kend; base += KB * W) {
    // step keys base + 4 i + rg, i < NI (rows past the end are clamped and masked)
    u32x4 kq[NI], vq[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) kq[i] = *reinterpret_cast<const u32x4*>(kb + (size_t)min(base + 4 * i + rg, last) * kHeadDim);
#pragma unroll
    for (int i = 0; i < NI; ++i) vq[i] = *reinterpret_cast<const u32x4*>(vb + (size_t)min(base + 4 * i + rg, last) * kHeadDim);
    __builtin_amdgcn_sched_barrier(0);                      // every load requested before the first is used
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float s[NI];
      float bm = -INFINITY;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        float a = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) a = dot2(as_f16x2(qv[g][e]), as_f16x2(kq[i][e]), a);
        a = row_sum(a) * scale;                              // the key's score, in all 16 lanes of the row group
        s[i] = base + 4 * i + rg < kend ? a : -INFINITY;
        bm = fmaxf(bm, s[i]);
      }
      bm = fmaxf(bm, __shfl_xor(bm, 16, 64));
      bm = fmaxf(bm, __shfl_xor(bm, 32, 64));                // the step's max over all its keys
      const float nm = fmaxf(mx[g], bm);
      const float corr = __expf(mx[g] - nm);                 // 0 on the first step (mx = -inf)
      float ps = 0.f;
#pragma unroll
      for (int d = 0; d < 8; ++d) o[g][d] *= corr;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const float pj = __expf(s[i] - nm);                  // 0 for masked keys
        ps += pj;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f16x2 v2 = as_f16x2(vq[i][e]);
          o[g][2 * e] = fmaf(pj, (float)v2[0], o[g][2 * e]);
          o[g][2 * e + 1] = fmaf(pj, (float)v2[1], o[g][2 * e + 1]);
        }
      }
      ps += __shfl_xor(ps, 16, 64);                           // + the other row groups' keys: the step's total
      ps += __shfl_xor(ps, 32, 64);
      sum[g] = sum[g] * corr + ps;
      mx[g] = nm;
    }
  }
  // merge the four row groups (lanes l, l ^ 16, l ^ 32, l ^ 48 hold the same dims), then the waves through LDS
  float* st = reinterpret_cast<float*>(smem);                // [W][G] (max, sum)
  float* os = st + W * G * 2;                                // [W][G][D]
#pragma unroll
  for (int g = 0; g < G; ++g) {
#pragma unroll
    for (int d = 0; d < 8; ++d) {
      o[g][d] += __shfl_xor(o[g][d], 16, 64);
      o[g][d] += __shfl_xor(o[g][d], 32, 64);
    }
    if (lane == 0) {
      st[(wave * G + g) * 2] = mx[g];
      st[(wave * G + g) * 2 + 1] = sum[g];
    }
    if (rg == 0) {
#pragma unroll
      for (int d = 0; d < 8; ++d) os[(wave * G + g) * kHeadDim + dl + d] = o[g][d];
    }
  }
  __syncthreads();
  // partial of this block: G records (max, sum, then the unnormalized output)
  float* mine = part + rec * kAttnRec;
  for (int idx = threadIdx.x; idx < G * kHeadDim; idx += blockDim.x) {
    const int g = idx / kHeadDim, d = idx % kHeadDim;
    float gm = -INFINITY;
    for (int w = 0; w < W; ++w) gm = fmaxf(gm, st[(w * G + g) * 2]);
    float num = 0.f, den = 0.f;
    for (int w = 0; w < W; ++w) {
      const float wm = st[(w * G + g) * 2];
      if (wm == -INFINITY) continue;                          // a wave that saw no key
      const float f = expf(wm - gm);
      num = fmaf(f, os[(w * G + g) * kHeadDim + d], num);
      den = fmaf(f, st[(w * G + g) * 2 + 1], den);
    }
    if (P == 1) {
      out[((size_t)m * Hq + h0 + g) * kHeadDim + d] = (f16)(num / den);
    } else {
      mine[g * kAttnRec + 4 + d] = num;
      if (d == 0) {
        mine[g * kAttnRec] = gm;
        mine[g * kAttnRec + 1] = den;
      }
    }
  }
}

template <int G, int KB>
__global__ __launch_bounds__(G == 1 && KB == 32 ? 1024 : 512) void attention_kernel(
    const f16* __restrict__ q, const f16* __restrict__ k_cache, const f16* __restrict__ v_cache,
    const int64_t* __restrict__ pos, f16* __restrict__ out, int Hq, int Hkv, int L, float scale, int CH,
    float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  args_in_sgprs(q, k_cache, v_cache, pos, out, Hq, Hkv, L, CH, part, (int)blockDim.x);
  attend_heads<G, KB>(q, k_cache, v_cache, pos, out, Hq, Hkv, L, scale, CH, part, smem, blockIdx.x, blockIdx.y, gridDim.y,
                      (size_t)(blockIdx.x * gridDim.y + blockIdx.y) * G);
}

// out[m][h][d] from the P <= kAttnMaxParts partials of attention_kernel or attention_mfma (merge_partitions), launched
// after it
__global__ __launch_bounds__(256) void attention_combine(const float* __restrict__ part, f16* __restrict__ out,
                                                         int blocks, int G, int P, int Hq) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= blocks * G * kHeadDim) return;
  const int b = idx / (G * kHeadDim), g = (idx / kHeadDim) % G, d = idx % kHeadDim;
  const int groups = Hq / G, m = b / groups, h = (b % groups) * G + g;
  const __amdgpu_buffer_rsrc_t pr = make_rsrc(part, (uint32_t)(blocks * P * G * kAttnRec * 4));
  out[((size_t)m * Hq + h) * kHeadDim + d] =
      (f16)merge_partitions(pr, b * P * G * kAttnRec + g * kAttnRec, G * kAttnRec, P, d);
}

// The key partitions of a call whose kernel is chosen on the device, by the keys attended (attention_select). The caller's
// bound on the keys sizes the launch and may lie far above them (a captured step's bound is its cache), and a kernel that
// is the better one on long contexts is not on the short ones at a conversation's start. The last token's position stands
// for all; any choice is right for any positions. keys < from: attend_heads (by_head) or attend_mfma with up to `few`
// partitions, else attend_prompt with up to `many`. The partials lie as [token][KV head][partition of `room`][head of the
// KV head] records.
struct AttnSplit {
  int from, few, many, by_head, room;
};
// keys a partition of attend_heads takes, in four waves of 32
__device__ __forceinline__ int attn_head_keys(int keys, int few) { return ((keys + few - 1) / few + 127) & ~127; }
__device__ __forceinline__ int attn_parts(const AttnSplit& sp, int keys) {
  if (keys >= sp.from) return min(sp.many, (keys + kAttnPromptMinKeys - 1) / kAttnPromptMinKeys);
  if (!sp.by_head) return keys <= kAttnMinKeys ? 1 : min(sp.few, (keys + 31) / 32);
  const int ch = attn_head_keys(keys, sp.few);
  return (keys + ch - 1) / ch;
}
__device__ __forceinline__ int attn_keys(const int64_t* __restrict__ pos, int M, int L) {
  return max(1, (int)min((int64_t)L, pos[M - 1] + 1));
}

// attention_combine for up to kAttnManyParts partitions, their records room for sp.room: one block per (token, head), a
// thread per dim; the partitions' weights exp(max - overall max) are evaluated once, a thread each, and shared through LDS
// (attention_combine has every thread evaluate them all, which its at most 16 partitions hide behind one round trip). Of
// many tokens the loads of the first 16 partitions go out with the position's, before the partitions' number is known:
// those that were not written hold anything and are left out (200 tokens on 1000 keys 19.4 -> 17.9 us with the attention;
// of one token, where most are cold, 12.1 -> 12.9 on 3000). One partition has written out itself.
__global__ __launch_bounds__(kHeadDim) void attention_combine_many(const float* __restrict__ part,
                                                                   const int64_t* __restrict__ pos, f16* __restrict__ out,
                                                                   int M, int Hq, int Hkv, int L, AttnSplit sp) {
  __shared__ float s_max[kAttnManyParts], s_f[kAttnManyParts], s_sum[kAttnManyParts];
  const int m = blockIdx.x / Hq, hd = blockIdx.x % Hq, G = Hq / Hkv, d = threadIdx.x;
  const float* rec = part + ((size_t)(m * Hkv + hd / G) * sp.room * G + hd % G) * kAttnRec;
  const int step = G * kAttnRec;                            // from one partition's record to the next one's
  float v[16], pm = -INFINITY, ps = 0.f;
  auto load_first = [&](int parts) {
    if (d < parts) {
      pm = rec[(size_t)d * step];
      ps = rec[(size_t)d * step + 1];
    }
#pragma unroll
    for (int u = 0; u < 16; ++u) v[u] = u < parts ? rec[(size_t)u * step + 4 + d] : 0.f;
  };
  if (!sp.by_head) load_first(sp.room);
  const int P = attn_parts(sp, attn_keys(pos, M, L));
  if (P == 1) return;
  if (sp.by_head) load_first(P);
  if (d < P) s_max[d] = pm;
  __syncthreads();
  float gm = -INFINITY;
  for (int p = 0; p < P; ++p) gm = fmaxf(gm, s_max[p]);
  if (d < P) {
    const float f = pm == -INFINITY ? 0.f : expf(pm - gm);   // (a partition that saw no key)
    s_f[d] = f;
    s_sum[d] = f * ps;
  }
  __syncthreads();
  float num = 0.f, den = 0.f;
  for (int p0 = 0; p0 < P; p0 += 16) {                       // 16 loads in flight
    if (p0 > 0) {
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = p0 + u < P ? rec[(size_t)(p0 + u) * step + 4 + d] : 0.f;
    }
#pragma unroll
    for (int u = 0; u < 16; ++u)
      if (p0 + u < P) {
        num = fmaf(s_f[p0 + u], v[u], num);
        den += s_sum[p0 + u];
      }
  }
  out[(size_t)blockIdx.x * kHeadDim + d] = (f16)(num / den);
}

// Causal GQA attention on MFMA for multi-token steps and prompts (same contract as attention_kernel): one wave per
// (KV head, 16 query rows, key partition), the query rows of a KV head numbered row = token * G + head-in-group.
// Per block of 32 keys (v_mfma_f32_16x16x32_f16):
//   S^T = K Q^T: A = 16 keys x 32 dims (lane (r, c): key kb + 8 (r / 4) + r % 4 + 4 t, 16 bytes of its row), B = the
//   wave's 16 query rows x 32 dims (held in registers), two key tiles t x four 32-dim steps; the key order is chosen so
//   that lane (r, c) ends up with the scores of query row r at keys kb + 8 c .. kb + 8 c + 7;
//   online softmax per query row (max and sum over the four lanes r, r + 16, r + 32, r + 48), masked past the row's
//   position; the probabilities, split into an fp16 head and an fp16 remainder (together exact to ~2^-22), are the
//   B operands of the next product (two MFMAs per dim tile, so the weights carry fp32 accuracy as in
//   attention_kernel);
//   O^T += V^T P^T: A = 16 dims x 32 keys of V^T, which the wave writes to its own LDS from its 8 KB of V rows
//   (4 keys x 8 dims per lane, packed into 8-byte rows of V^T) and reads back as 16-byte fragments; eight dim tiles.
// A wave touches only its own LDS, in order, so no barrier is needed. With P > 1 each wave writes the partial (max,
// sum, unnormalized output) of its rows in attention_kernel's layout and attention_combine merges them.
constexpr int kAttnVtPitch = 80;                            // bytes per dim row of the staged V^T (64 + 16 padding)

// a wave's work: (KV head, row tile) unit, partition pid of P (records of PS), with kHeadDim * kAttnVtPitch bytes of LDS at vt
__device__ __forceinline__ void attend_mfma(const f16* __restrict__ q, const f16* __restrict__ k_cache,
                                            const f16* __restrict__ v_cache, const int64_t* __restrict__ pos,
                                            f16* __restrict__ out, int M, int Hq, int Hkv, int L, float scale,
                                            float* __restrict__ part, uint8_t* vt, int unit, int pid, int P, int PS) {
  const int G = Hq / Hkv;
  const int hk = unit % Hkv, tile = unit / Hkv;
  const int lane = threadIdx.x & 63, r = lane & 15, c = lane >> 4;
  // this lane's query row (as the B column r)
  const int row = 16 * tile + r, m = row / G, g = row - m * G;
  const bool live = m < M;
  const int pr = live ? (int)min((int64_t)L - 1, pos[m]) : -1;  // last key the row attends
  int wmax = pr;                                               // the wave's last key
  wmax = max(wmax, __shfl_xor(wmax, 1, 64));
  wmax = max(wmax, __shfl_xor(wmax, 2, 64));
  wmax = max(wmax, __shfl_xor(wmax, 4, 64));
  wmax = max(wmax, __shfl_xor(wmax, 8, 64));
  // the P partitions split the keys this wave attends (not the caller's bound on them) in whole 32-key blocks
  const int ch = ((wmax + 1 + P - 1) / P + 31) / 32 * 32;
  const int kbeg = pid * ch, kend = min(wmax + 1, kbeg + ch);
  const __amdgpu_buffer_rsrc_t qr = make_rsrc(q, (uint32_t)M * (uint32_t)Hq * kHeadDim * 2u);
  const int qoff = live ? ((m * Hq + hk * G + g) * kHeadDim + 8 * c) * 2 : kOutOfRange;
  f16x8 qf[4];
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) qf[ks] = __builtin_bit_cast(f16x8, buffer_load16(qr, qoff + 64 * ks));
  const f16* kh = k_cache + (size_t)hk * L * kHeadDim;
  const f16* vh = v_cache + (size_t)hk * L * kHeadDim;
  const int kr = 8 * (r >> 2) + (r & 3);                      // key of A row r in tile 0 (tile 1: + 4)
  float mx = -INFINITY, lsum = 0.f;
  f32x4 o[8];
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) o[dt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // K and V rows are read in whole 32-key blocks, clamped to the wave's last attended key: rows past it may never
  // have been written (NaN or Inf in an uninitialized cache), and a masked key's weight 0 times NaN is still NaN in
  // the P V product
  for (int kb = kbeg; kb < kend; kb += 32) {
    u32x4 kf[2][4], vf[2][4];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      const f16* krow = kh + (size_t)min(kb + kr + 4 * t, wmax) * kHeadDim + 8 * c;
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) kf[t][ks] = *reinterpret_cast<const u32x4*>(krow + 32 * ks);
    }
#pragma unroll
    for (int u = 0; u < 2; ++u)                               // V rows kb + 4 (lane % 8) + j, dims 8 (lane / 8 + 8 u)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        vf[u][j] = *reinterpret_cast<const u32x4*>(vh + (size_t)min(kb + 4 * (lane & 7) + j, wmax) * kHeadDim +
                                                   8 * ((lane >> 3) + 8 * u));
    f32x4 st[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      st[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
        st[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, kf[t][ks]), qf[ks], st[t], 0, 0, 0);
    }
    // V^T rows (dim) x 4 keys per lane into the wave's LDS
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int d0 = 8 * ((lane >> 3) + 8 * u);
#pragma unroll
      for (int e = 0; e < 4; ++e) {                           // dims d0 + 2 e, d0 + 2 e + 1
        const uint32_t a0 = vf[u][0][e], a1 = vf[u][1][e], a2 = vf[u][2][e], a3 = vf[u][3][e];
        // v_perm picks bytes of {a1, a0}: 0x05040100 the low halves (a0, a1), 0x07060302 the high halves
        const uint2 lo = make_uint2(__builtin_amdgcn_perm(a1, a0, 0x05040100u),
                                    __builtin_amdgcn_perm(a3, a2, 0x05040100u));
        const uint2 hi = make_uint2(__builtin_amdgcn_perm(a1, a0, 0x07060302u),
                                    __builtin_amdgcn_perm(a3, a2, 0x07060302u));
        *reinterpret_cast<uint2*>(vt + (d0 + 2 * e) * kAttnVtPitch + 8 * (lane & 7)) = lo;
        *reinterpret_cast<uint2*>(vt + (d0 + 2 * e + 1) * kAttnVtPitch + 8 * (lane & 7)) = hi;
      }
    }
    // scores of row r at keys kb + 8 c + i (i = 4 t + v), masked past the row's position and the partition
    float sc[8], bm = -INFINITY;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int key = kb + 8 * c + i;
      sc[i] = key <= pr && key < kend ? st[i >> 2][i & 3] * scale : -INFINITY;
      bm = fmaxf(bm, sc[i]);
    }
    bm = fmaxf(bm, __shfl_xor(bm, 16, 64));
    bm = fmaxf(bm, __shfl_xor(bm, 32, 64));
    const float nm = fmaxf(mx, bm);
    const float corr = nm == -INFINITY ? 1.f : __expf(mx - nm);   // 0 on the first block with a key
    f16x8 ph, pl;                                           // p = ph + pl to ~2^-22: fp32-accurate weights
    float ps = 0.f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float pj = nm == -INFINITY ? 0.f : __expf(sc[i] - nm);
      ps += pj;
      ph[i] = (f16)pj;
      pl[i] = (f16)(pj - (float)ph[i]);
    }
    lsum = lsum * corr + ps;
    mx = nm;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      const f16x8 va = *reinterpret_cast<const f16x8*>(vt + (16 * dt + r) * kAttnVtPitch + 16 * c);
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, ph, o[dt] * corr, 0, 0, 0);
      o[dt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(va, pl, o[dt], 0, 0, 0);
    }
  }
  lsum += __shfl_xor(lsum, 16, 64);
  lsum += __shfl_xor(lsum, 32, 64);
  if (!live) return;
  // lane (r, c) holds O^T[16 dt + 4 c + v][row r]
  if (P == 1) {
    f16* dst = out + ((size_t)m * Hq + hk * G + g) * kHeadDim + 4 * c;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      const f16x2 lo = {(f16)(o[dt][0] / lsum), (f16)(o[dt][1] / lsum)};
      const f16x2 hi = {(f16)(o[dt][2] / lsum), (f16)(o[dt][3] / lsum)};
      *reinterpret_cast<uint2*>(dst + 16 * dt) = make_uint2(as_u32(lo), as_u32(hi));
    }
    return;
  }
  float* mine = part + (((size_t)(m * Hkv + hk) * PS + pid) * G + g) * kAttnRec;
  if (c == 0) {
    mine[0] = mx;
    mine[1] = lsum;
  }
#pragma unroll
  for (int dt = 0; dt < 8; ++dt) *reinterpret_cast<f32x4*>(mine + 4 + 16 * dt + 4 * c) = o[dt];
}

__global__ __launch_bounds__(64) void attention_mfma(const f16* __restrict__ q, const f16* __restrict__ k_cache,
                                                     const f16* __restrict__ v_cache, const int64_t* __restrict__ pos,
                                                     f16* __restrict__ out, int M, int Hq, int Hkv, int L, float scale,
                                                     float* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) uint8_t vt[kHeadDim * kAttnVtPitch];
  args_in_sgprs(q, k_cache, v_cache, pos, out, M, Hq, Hkv, L, part);
  attend_mfma(q, k_cache, v_cache, pos, out, M, Hq, Hkv, L, scale, part, vt, blockIdx.x, blockIdx.y, gridDim.y, gridDim.y);
}

// Causal GQA attention for prompts and long steps (the contract of attention_mfma): a workgroup of four waves takes
// 32 RG query rows of one KV head (row = token * G + head-in-group) and walks the keys in blocks of 32 KG that its waves
// share through LDS; a wave owns 32 rows (row group wave % RG) and 32 keys of every block (key group wave / RG), and the
// key groups' sums are merged at the end. Per block and wave (v_mfma_f32_32x32x16_f16, lane l: j = l % 32, h = l / 32):
//   S^T = K Q^T: A = 32 keys x 16 dims from LDS, B = the wave's 32 rows (registers). Lane (j, h) holds row j's scores of
//   keys 8 (v / 4) + 4 h + v % 4, v = 0..15: two lanes a row.
//   Online softmax in base 2 against a reference that follows the running maximum only when a score exceeds it by more
//   than a lag, so that the 64 accumulator registers are rescaled in the first blocks only and no lane exchange is
//   needed in the others. The weights are split into an fp16 head and an fp16 remainder, together good to ~2^-22 of a
//   weight while the remainder is a normal fp16 number and to half of fp16's smallest subnormal, 2^-25, below. They are
//   therefore evaluated as 2^(score - reference + 15 - lag), with the maximum between 2^(15 - lag) and 2^15 (the factor
//   cancels against their sum), so that what is cut off lies below 2^-39 of the largest weight at a lag of 1 and 2^-32 at
//   8: a long tail of small weights keeps its sum. (Evaluated as 2^(score - reference), 64000 weights of 2^-26 vanished
//   beside a weight of 1.) A lag of 1 rescales more often, which costs 1-2% with few rows and 13% with many (3000 tokens
//   83 us against 73): the few rows whose other kernel is attention_kernel, with fp32 weights, take 1, the others, whose
//   other kernel is attention_mfma, with weights of at most 1 and the same split, 8.
//   O^T += V^T P^T: B = the weights as the lane holds them, i.e. contraction index 8 h + i of step s is key
//   16 s + 8 (i / 4) + 4 h + i % 4; A = V^T from LDS by transposing reads (ds_read_b64_tr_b16).
// K and V go from memory straight to LDS, one block ahead (K two: a block's scores are multiplied while the vector unit
// evaluates the weights of the block before), with one barrier per block.
// attention_mfma has a wave of 16 rows load its own K and V and wait for them in every block: L2 latency and reads bound
// it. Here 32 RG rows share them; what is left is the matrix cores (three products per score and dim, the weights being
// split), about level with the softmax's vector instructions, at two waves per SIMD (188 registers, 64 KB of LDS a
// workgroup at KG = 2). Against 64 rows (RG = KG = 2), 128 rows (RG = 4, KG = 1) lengthen the serial walk of the last
// rows: 3000 tokens 97 us against 81 (before K's second block ahead and the transposing reads), 700 tokens 27 against
// 21; 32 rows (KG = 4) double the L2 reads (126 us) and win only where 64 rows leave CUs idle.
// MI355X, 16 query / 2 KV heads, graph-timed, us (attention_mfma -> this): 3000 tokens 283 -> 73, 700 tokens 34.5 -> 17.1,
// 300 tokens 16.1 -> 11.4, 128 tokens 10.9 -> 8.7; 512 tokens on 4096 cached 203 -> 51, 128 on 8000 125 -> 39 (KG = 4; 70 and 49
// with KG = 2); 28 / 4 heads, 2048 tokens 230 -> 63.
constexpr float kAttnLagFew = 1.f, kAttnLag = 8.f;

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));

// a workgroup's work: bx of tiles * Hkv, partition pid of P (records of PS); FEW: below kAttnMfmaMinRows rows; one: the last
// key of a one-token call, where the caller has read it, else -1
template <int RG, int KG, bool FEW>
__device__ __forceinline__ void attend_prompt(const f16* __restrict__ q, const f16* __restrict__ k_cache,
                                              const f16* __restrict__ v_cache, const int64_t* __restrict__ pos,
                                              f16* __restrict__ out, int M, int Hq, int Hkv, int L, float scale, int tiles,
                                              float* __restrict__ part, uint8_t* smem, int bx, int pid, int P, int PS, int one) {
  static_assert(RG * KG == 4, "four waves");
  constexpr int kRows = 32 * RG, kKeys = 32 * KG;         // query rows of the workgroup, keys of a block
  constexpr int kBuf = kKeys * kHeadDim * 2;                  // bytes of a block's K, and of its V
  constexpr int NP = kKeys / 16;                              // 16-byte pieces a thread loads of K, and of V
  // smem: [2][K block, V block]
  int* s_max = reinterpret_cast<int*>(smem);                  // the waves' last keys, before the first block is staged
  const int G = Hq / Hkv;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;
  // longest tiles first; every second round of workgroups in reverse, so that a CU's two workgroups add up alike
  const int hk = bx % Hkv, idx = bx / Hkv, per = max(1, 256 / Hkv), rnd = idx / per;
  const int at = rnd & 1 ? rnd * per + min(per, tiles - rnd * per) - 1 - (idx - rnd * per) : idx;
  const int tile = tiles - 1 - at;
  const int rgrp = wave % RG, kgrp = wave / RG;               // the wave's rows, and its keys of a block
  const int row = kRows * tile + 32 * rgrp + j, m = row / G, g = row - m * G;
  const bool live = m < M;
  int pr, wmax, wmin, gmax;                                   // the last keys: the row's, the wave's largest and least, all
  if (one >= 0) {                                             // one token, whose position the caller has read
    pr = live ? one : -1;
    wmax = rgrp == 0 ? one : -1;
    wmin = rgrp == 0 ? one : INT_MAX;
    gmax = one;
  } else {
    pr = live ? (int)min((int64_t)L - 1, pos[m]) : -1;
    wmax = pr;
    wmin = live ? pr : INT_MAX;
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) {
      wmax = max(wmax, __shfl_xor(wmax, o, 64));
      wmin = min(wmin, __shfl_xor(wmin, o, 64));
    }
    wmax = __builtin_amdgcn_readfirstlane(wmax);
    wmin = __builtin_amdgcn_readfirstlane(wmin);
    if (lane == 0) s_max[wave] = wmax;
    __syncthreads();
    gmax = max(max(s_max[0], s_max[1]), max(s_max[2], s_max[3]));
    __syncthreads();
  }
  const int ch = ((gmax + 1 + P - 1) / P + kKeys - 1) / kKeys * kKeys;
  const int kbeg = pid * ch, kend = min(gmax + 1, kbeg + ch);
  // q of row j, dims 16 ks + 8 h .. + 7; a negative scale is moved into q (exact), so that score order is weight order
  const uint32_t flip = scale < 0.f ? 0x80008000u : 0u;
  // base-2 score scale; held above 0, so that a masked score of -inf stays -inf (scale 0: every weight is 2^~0 = 1)
  const float c2 = fabsf(scale) * 1.44269504088896340736f < FLT_MIN ? FLT_MIN : fabsf(scale) * 1.44269504088896340736f;
  f16x8 qf[8];
  const f16* qrow = q + ((size_t)min(m, M - 1) * Hq + hk * G + g) * kHeadDim + 8 * h;
#pragma unroll
  for (int ks = 0; ks < 8; ++ks) {
    u32x4 t = load16(qrow + 16 * ks);
#pragma unroll
    for (int e = 0; e < 4; ++e) t[e] ^= flip;
    qf[ks] = __builtin_bit_cast(f16x8, t);
  }
  const uint8_t* kh = reinterpret_cast<const uint8_t*>(k_cache + (size_t)hk * L * kHeadDim);
  const uint8_t* vh = reinterpret_cast<const uint8_t*>(v_cache + (size_t)hk * L * kHeadDim);
  // K and V rows go straight to LDS as they are, 256 bytes each: this thread's pieces are 16 bytes of keys tid / 16 + 16 u,
  // slot tid % 16 of the row, whose 16-byte pieces are permuted by the key: K's so that the 32 rows of a fragment read
  // meet different banks, V's so that the four rows of a transposing read do. Rows past the last attended key (never
  // written, maybe NaN) are clamped to it: their weight 0 must meet finite values
  const int kk = tid >> 4, kp = tid & 15;
  const uint32_t dst = lds_addr(smem) + 1024 * wave;
  auto load = [&](const uint8_t* rows, int kb, int piece, uint32_t at) {   // (a block past the last one: the last key)
    const int k0 = min(kb, gmax), lim = gmax - k0;
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(rows + (size_t)k0 * 256, kBuf);
#pragma unroll
    for (int u = 0; u < NP; ++u) dma16(rs, min(kk + 16 * u, lim) * 256 + 16 * piece, dst + at + 4096 * u);
  };
  auto vswz = [](int key) { return 4 * (key & 3) + 2 * ((key >> 2) & 1); };
  auto load_k = [&](int kb, uint32_t base) { load(kh, kb, kp ^ kk, base); };
  auto load_v = [&](int kb, uint32_t base) { load(vh, kb, kp ^ vswz(kk), base + kBuf); };
  // LDS offsets in a buffer. Both permutations are an exclusive-or of address bits 4..7 applied to the running offset, so
  // one register holds each family. K: row 32 kgrp + j, pieces 2 s + h. V: transposing 8-byte reads (16 lanes i get column
  // i of the 4 keys x 16 dims whose 8-byte pieces they address): key 4 h + i / 4, dims 16 (l / 16 % 2) + 4 (i % 4)
  const uint32_t kr = (32 * kgrp + j) * 256 + 16 * (h ^ (j & 15));
  const int vk = 4 * h + ((lane & 15) >> 2), vp = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
  const uint32_t vr = kBuf + (32 * kgrp + vk) * 256 + 16 * (vp ^ vswz(vk)) + 8 * (lane & 1);
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  auto v_frag = [&](uint32_t at) {                            // keys at .. and at + 8 rows, this lane's dim
    typedef __attribute__((address_space(3))) s16x4* lds_ptr;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(smem + at));
    const s16x4 c = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(smem + at + 2048));
    return __builtin_bit_cast(f16x8, __builtin_shufflevector(a, c, 0, 1, 2, 3, 4, 5, 6, 7));
  };
  constexpr float lag = FEW ? kAttnLagFew : kAttnLag;
  float ref = -INFINITY, lsum = 0.f;                          // reference (base 2), the lane's share of the weights' sum
  f32x16 o[4];
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int v = 0; v < 16; ++v) o[dt][v] = 0.f;

  const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16 st = zero;                                           // scores of the wave's 32 keys of a block
  auto scores = [&](uint32_t base, int s0, int s1) {          // dims 16 s0 .. 16 s1 of them
#pragma unroll
    for (int s = s0; s < s1; ++s)
      st = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const f16x8*>(smem + ((kr + base) ^ (32 * s))), qf[s], st,
                                                  0, 0, 0);
  };
  // one block: the weights of its scores, the weights times V and the next block's scores (its K lies in the other
  // buffer), whose products run while the vector unit evaluates the weights
  auto block = [&](uint32_t base, int kb) {                   // kb: the wave's first key
    if (kb + 31 > min(wmin, kend - 1)) {                      // some row attends part of these keys only (uniform)
      const int last = min(pr, kend - 1) - kb - 4 * h;        // a key at or below it counts
#pragma unroll
      for (int v = 0; v < 16; ++v)
        if (8 * (v >> 2) + (v & 3) > last) st[v] = -INFINITY;
    }
    float bm = st[0];
#pragma unroll
    for (int v = 1; v < 16; ++v) bm = fmaxf(bm, st[v]);
    if (__any(bm * c2 > ref + lag)) {                    // (uniform; either lane of a row)
      const float nm = fmaxf(ref, fmaxf(bm, __shfl_xor(bm, 32, 64)) * c2);   // -inf while the row has seen no key
      const float corr = nm == -INFINITY ? 1.f : __builtin_amdgcn_exp2f(ref - nm);
      ref = nm;
      lsum *= corr;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) o[dt] *= corr;
    }
    const float sub = ref == -INFINITY ? 0.f : ref - (15.f - lag);
    const f32x16 sc = st;
    st = zero;
#pragma unroll
    for (int s = 0; s < 2; ++s) {                             // 16 keys: head and remainder of their weights, then V
      u32x4 ph, pl;
      float ps[2] = {0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const f32x2 p = {__builtin_amdgcn_exp2f(fmaf(sc[8 * s + 2 * i], c2, -sub)),
                         __builtin_amdgcn_exp2f(fmaf(sc[8 * s + 2 * i + 1], c2, -sub))};
        ps[0] += p[0];
        ps[1] += p[1];
        const f16x2 head = __builtin_convertvector(p, f16x2);
        const f32x2 rest = {p[0] - (float)head[0], p[1] - (float)head[1]};
        ph[i] = as_u32(head);
        pl[i] = as_u32(__builtin_convertvector(rest, f16x2));
      }
      lsum += ps[0] + ps[1];
      scores(base ^ (2 * kBuf), 4 * s, 4 * s + 4);            // (past the last block: of stale K, never used)
      f16x8 va[4];
#pragma unroll
      for (int dt = 0; dt < 4; ++dt) va[dt] = v_frag(((vr + base) ^ (64 * dt)) + 4096 * s);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[dt], __builtin_bit_cast(f16x8, ph), o[dt], 0, 0, 0);
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[dt], __builtin_bit_cast(f16x8, pl), o[dt], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  // buffer b holds block i's V and block i + 1's K is in the other one, whose V slot takes block i + 1 at the end; the K
  // of block i + 2 replaces that of block i, whose scores are in registers
  if (kbeg < kend) {
    load_k(kbeg, 0);
    load_k(kbeg + kKeys, 2 * kBuf);
    load_v(kbeg, 0);
  }
  lds_wait_barrier<0>();
  if (kbeg < kend) scores(0, 0, 8);
  lds_barrier();                                              // every wave has read the first K
  uint32_t b = 0;
  for (int kb = kbeg; kb < kend; kb += kKeys, b ^= 2 * kBuf) {
    const bool more = kb + kKeys < kend;
    if (more) {
      load_k(kb + 2 * kKeys, b);
      load_v(kb + kKeys, b ^ (2 * kBuf));
    }
    block(b, kb + 32 * kgrp);
    lds_wait_barrier<0>();                                    // the K and V requested above are visible
  }
  lsum += __shfl_xor(lsum, 32, 64);
  if constexpr (KG > 1) {                                     // the key groups' sums, through LDS, into key group 0
    constexpr int kRec = 66 * 64 * 4;                         // a wave's sums, reference and weight sum
    float* mine = reinterpret_cast<float*>(smem + (size_t)((kgrp - 1) * RG + rgrp) * kRec) + lane;
    if (kgrp > 0) {
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) mine[64 * (16 * dt + v)] = o[dt][v];
      mine[64 * 64] = ref;
      mine[65 * 64] = lsum;
    }
    lds_barrier();
    if (kgrp > 0) return;
    for (int g2 = 1; g2 < KG; ++g2) {
      const float* theirs = reinterpret_cast<const float*>(smem + (size_t)((g2 - 1) * RG + rgrp) * kRec) + lane;
      const float r2 = theirs[64 * 64], nm = fmaxf(ref, r2);
      const float c0 = ref == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(ref - nm);
      const float c1 = r2 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(r2 - nm);
      ref = nm;
      lsum = lsum * c0 + theirs[65 * 64] * c1;
#pragma unroll
      for (int dt = 0; dt < 4; ++dt)
#pragma unroll
        for (int v = 0; v < 16; ++v) o[dt][v] = o[dt][v] * c0 + theirs[64 * (16 * dt + v)] * c1;
    }
  }
  if (!live) return;
  // lane (j, h) holds O^T[32 dt + 8 (v / 4) + 4 h + v % 4][row j]
  if (P == 1) {
    f16* dst = out + ((size_t)m * Hq + hk * G + g) * kHeadDim + 4 * h;
#pragma unroll
    for (int dt = 0; dt < 4; ++dt)
#pragma unroll
      for (int v = 0; v < 16; v += 4) {
        const f16x2 lo = {(f16)(o[dt][v] / lsum), (f16)(o[dt][v + 1] / lsum)};
        const f16x2 hi = {(f16)(o[dt][v + 2] / lsum), (f16)(o[dt][v + 3] / lsum)};
        *reinterpret_cast<uint2*>(dst + 32 * dt + 2 * v) = make_uint2(as_u32(lo), as_u32(hi));
      }
    return;
  }
  // the record's maximum and sum are natural-base ones: ref / log2(e)
  float* mine = part + (((size_t)(m * Hkv + hk) * PS + pid) * G + g) * kAttnRec;
  if (h == 0) {
    mine[0] = ref * 0.69314718055994530942f;
    mine[1] = lsum;
  }
#pragma unroll
  for (int dt = 0; dt < 4; ++dt)
#pragma unroll
    for (int v = 0; v < 16; v += 4)
      *reinterpret_cast<f32x4*>(mine + 4 + 32 * dt + 2 * v + 4 * h) = f32x4{o[dt][v], o[dt][v + 1], o[dt][v + 2], o[dt][v + 3]};
}

template <int RG, int KG>
__global__ __launch_bounds__(256, 2) void attention_prompt(const f16* __restrict__ q, const f16* __restrict__ k_cache,
                                                           const f16* __restrict__ v_cache,
                                                           const int64_t* __restrict__ pos, f16* __restrict__ out, int M,
                                                           int Hq, int Hkv, int L, float scale, int tiles,
                                                           float* __restrict__ part) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  args_in_sgprs(q, k_cache, v_cache, pos, out, M, Hq, Hkv, L, tiles, part);
  attend_prompt<RG, KG, false>(q, k_cache, v_cache, pos, out, M, Hq, Hkv, L, scale, tiles, part, smem, blockIdx.x, blockIdx.y,
                        gridDim.y, gridDim.y, -1);
}

// attend_prompt, or with fewer than sp.from keys attend_heads (HEADS) or attend_mfma, in workgroups of four waves: the work
// of either is numbered along blockIdx.x, partitions slowest, and workgroups past it end at once. Beside launching one of
// the kernels by the bound, us on an 8192-row cache with the bound at 8192 (attention_kernel or attention_mfma / attend_prompt
// alone / this): one token, 16 / 2 heads at position 200 8.7 / 13.6 / 7.3, at 700 11.2 / 13.5 / 8.4, 3000 12.2 / 14.2 /
// 12.5, 8000 17.2 / 15.0 / 15.4; 28 / 4 heads 10.1 / 13.8 / 7.9, 12.3 / 14.1 / 9.1, 14.9 / 14.7 / 12.2, 28.8 / 16.4 /
// 16.8; 16 tokens, 16 / 2 heads 8.1 / 13.4 / 7.2, 10.2 / 13.9 / 9.4, 15.8 / 15.1 / 13.7, 29.5 / 17.7 / 17.5. Prompts of
// 50 .. 200 tokens whose bound is a 4096-row cache: 64 tokens 9.3 / 13.1 / 7.5, on 200 cached 10.7 / 13.3 / 11.5, on 1500
// 18.6 / 15.1 / 14.7.
template <int RG, int KG, bool HEADS>
__global__ __launch_bounds__(256, 2) void attention_select(const f16* __restrict__ q, const f16* __restrict__ k_cache,
                                                           const f16* __restrict__ v_cache,
                                                           const int64_t* __restrict__ pos, f16* __restrict__ out, int M,
                                                           int Hq, int Hkv, int L, float scale, int tiles,
                                                           float* __restrict__ part, AttnSplit sp) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  args_in_sgprs(q, k_cache, v_cache, pos, out, M, Hq, Hkv, L, tiles, part, sp.from, sp.few, sp.many);
  const int keys = __builtin_amdgcn_readfirstlane(attn_keys(pos, M, L)), P = attn_parts(sp, keys);
  if (keys >= sp.from) {
    const int n = tiles * Hkv, pid = blockIdx.x / n;
    if (pid < P)
      attend_prompt<RG, KG, HEADS>(q, k_cache, v_cache, pos, out, M, Hq, Hkv, L, scale, tiles, part, smem, blockIdx.x - pid * n,
                            pid, P, sp.room, HEADS && M == 1 ? keys - 1 : -1);
  } else if constexpr (HEADS) {
    const int n = M * Hq, pid = blockIdx.x / n;
    const int bx = blockIdx.x - pid * n, G = Hq / Hkv;        // (token, head)
    if (pid < P)
      attend_heads<1, 32>(q, k_cache, v_cache, pos, out, Hq, Hkv, L, scale, attn_head_keys(keys, sp.few), part, smem, bx,
                          pid, P, ((size_t)(bx / G) * sp.room + pid) * G + bx % G);
  } else {
    // as many waves a CU as attention_mfma's workgroups of one would put there: two, in one workgroup where no more fit
    constexpr int NW = KG == 4 ? 2 : 1;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), unit = NW * blockIdx.x + wave;
    const int n = (M * (Hq / Hkv) + 15) / 16 * Hkv, pid = unit / n;
    if (wave < NW && pid < P)
      attend_mfma(q, k_cache, v_cache, pos, out, M, Hq, Hkv, L, scale, part, smem + wave * kHeadDim * kAttnVtPitch,
                  unit - pid * n, pid, P, sp.room);
  }
}

// fp16 GEMV for the (tied) lm_head, M <= 4: y[m][n] = fp16(sum_k x[m][k] W[n][k]), W fp16 [N][K] row-major, fp32
// accumulation. A bandwidth kernel: the workgroup stages x[M][K] in LDS once (one barrier), then each wave streams
// RW weight rows with 16-byte non-temporal loads (lane l takes k = 512 c + 8 l .. + 7 of chunk c, so every load is
// one contiguous 1 KB), kHeadChunks chunks of every row in flight, dot2 against x from LDS, and a wave reduction per
// row. Two rows per wave, four chunks each (MI355X graph, 3 cold copies of the 151936 x 2048 Qwen2.5 head): 94.3 us
// (6.6 TB/s) against 102.3 for 8 rows and two chunks, 99.0 for 4 and two, 96.2 for one row and four; same bits.
constexpr int kHeadChunks = 4;

// The greedy pick's order on (fp16 logit, index) as one 64-bit key, larger = picked, as torch.argmax picks: the larger
// value (-0 equal to +0, a NaN above every number), then the smaller index. Zero is below every key.
__device__ __forceinline__ uint64_t pick_key(uint16_t b, int idx) {
  uint32_t k;
  if ((b & 0x7FFFu) > 0x7C00u) {
    k = 0x10000u;                                            // NaN
  } else {
    if (b == 0x8000u) b = 0;                                 // -0 ties with +0
    k = (b & 0x8000u) ? (~b & 0xFFFFu) : (b | 0x8000u);      // fp16 order as unsigned order
  }
  return ((uint64_t)k << 32) | (uint32_t)(0xFFFFFFFFu - (uint32_t)idx);
}

// PICK (M = 1): each workgroup also writes the key of its largest logit (as stored, fp16) to pick[blockIdx.x], for
// head_pick_kernel
template <int M, int RW, int CH = kHeadChunks, bool PICK = false>
__global__ __launch_bounds__(256) void gemv_f16_kernel(const f16* __restrict__ x, const f16* __restrict__ w,
                                                       f16* __restrict__ y, int N, int K, uint64_t* __restrict__ pick,
                                                       int mrows) {
  static_assert(!PICK || M == 1, "the greedy pick takes one row");
  // M rows compiled in, mrows <= M of them real (x staged and y stored for those; the rest computes on stale LDS)
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  u32x4* xs = reinterpret_cast<u32x4*>(smem);               // [M][K / 8]
  // wave through readfirstlane: the row buffer resource below is then known uniform and stays in scalar registers
  // (from a per-lane value every weight load becomes a waterfall loop)
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kp = K >> 3;                                     // 16-byte pieces per row
  for (int i = threadIdx.x; i < mrows * kp; i += blockDim.x) xs[i] = *reinterpret_cast<const u32x4*>(x + 8 * (size_t)i);
  __syncthreads();
  const int n0 = (blockIdx.x * 4 + wave) * RW;
  if (!PICK && n0 >= N) return;                             // (PICK: every wave reaches the barrier below; one past N
                                                             // reads nothing and stores nothing)
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(w + (size_t)min(n0, N) * K, (uint32_t)(max(0, min(RW, N - n0)) * K * 2));
  float acc[RW][M];
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) acc[r][m] = 0.f;
  const int nc = (kp + 63) >> 6;                             // 512-k chunks
  for (int c0 = 0; c0 < nc; c0 += CH) {
    u32x4 wv[CH][RW];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int p = 64 * (c0 + u) + lane;                    // this lane's piece of the chunk
#pragma unroll
      for (int r = 0; r < RW; ++r) wv[u][r] = buffer_load16_nt(wr, p < kp ? 2 * (r * K + 8 * p) : kOutOfRange);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
      const int p = 64 * (c0 + u) + lane;
      if (p >= kp) break;
#pragma unroll
      for (int m = 0; m < M; ++m) {
        const u32x4 xv = xs[m * kp + p];
#pragma unroll
        for (int r = 0; r < RW; ++r)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[r][m] = dot2(as_f16x2(wv[u][r][e]), as_f16x2(xv[e]), acc[r][m]);
      }
    }
  }
  uint64_t best = 0;
#pragma unroll
  for (int r = 0; r < RW; ++r)
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const float v = wave_sum(acc[r][m]);
      if (lane == 0 && n0 + r < N && m < mrows) {
        const f16 h = (f16)v;
        y[(size_t)m * N + n0 + r] = h;
        if constexpr (PICK) {
          const uint64_t kv = pick_key(__builtin_bit_cast(uint16_t, h), n0 + r);
          best = kv > best ? kv : best;
        }
      }
    }
  if constexpr (PICK) {
    __shared__ uint64_t red[4];
    if (lane == 0) red[wave] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
      for (int v = 1; v < 4; ++v) best = red[v] > best ? red[v] : best;
      pick[blockIdx.x] = best;
    }
  }
}

// The greedy pick and its feedback, one workgroup: the largest of the head workgroups' keys (pick[0 .. n)) gives the
// index; tokens[0] = index, positions[0] += 1 (positions may be null), out[*out_count] = index while *out_count <
// out_cap and *out_count + 1 (out_count may be null), and h_out[0 .. H) = embed row index (embed may be null): the next
// step's input, so that a one-token step needs no embedding gather of its own
constexpr int kPickThreads = 1024;
__global__ __launch_bounds__(kPickThreads) void head_pick_kernel(const uint64_t* __restrict__ pick, int n,
                                                                 int64_t* tokens, int64_t* positions, int64_t* out,
                                                                 int out_cap, int* out_count,
                                                                 const f16* __restrict__ embed, int H, f16* h_out) {
  __shared__ uint64_t red[kPickThreads / 64];
  __shared__ int s_idx;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  uint64_t best = 0;
  for (int i0 = tid; i0 < n; i0 += 8 * kPickThreads) {      // eight loads in flight per thread
    uint64_t v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = i0 + u * kPickThreads < n ? pick[i0 + u * kPickThreads] : 0;
#pragma unroll
    for (int u = 0; u < 8; ++u) best = v[u] > best ? v[u] : best;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const uint64_t o = __shfl_xor(best, off, 64);
    best = o > best ? o : best;
  }
  if (lane == 0) red[wave] = best;
  __syncthreads();
  if (tid == 0) {
    for (int v = 1; v < kPickThreads / 64; ++v) best = red[v] > best ? red[v] : best;
    const int idx = (int)(0xFFFFFFFFu - (uint32_t)best);
    s_idx = idx;
    tokens[0] = idx;
    if (positions) positions[0] += 1;
    if (out_count) {
      const unsigned c = (unsigned)*out_count;               // (a count past INT_MAX stays out of range)
      if (c < (unsigned)out_cap) out[c] = idx;
      *out_count = (int)(c + 1u);
    }
  }
  if (embed == nullptr) return;                              // (uniform)
  __syncthreads();
  const u32x4* src = reinterpret_cast<const u32x4*>(embed + (size_t)s_idx * H);
  for (int i = tid; i < (H >> 3); i += kPickThreads) reinterpret_cast<u32x4*>(h_out)[i] = src[i];
}

constexpr int kHeadRows = 2;                                // RW: rows per wave (4 waves a workgroup)

// fp16-weight MFMA GEMV for the head beyond 8 rows (up to 64: MT 16-row activation tiles), where the dot2 kernel above
// turns ALU-bound. Each wave owns one 16-row tile of W, the MFMA's A; the workgroup's four waves share x, the B. Both
// stream through LDS in 128-k chunks by direct-to-LDS loads, D chunks deep: a wave-load takes 256 contiguous
// bytes of each of 4 rows, non-temporal for W, where the fragments read from memory directly (lane (r, q) its own row) took
// 64 bytes of 16 rows, half of each 128-byte line. A row's sixteen 16-byte blocks are permuted by the row (block b at
// b ^ f16w_swz(row % 16)), so a fragment's rows meet different banks; lane (r, q) takes block 4 q + s as k-step s. One
// barrier a chunk: it makes the next chunk's x visible and frees the slot consumed before; loads complete in issue order,
// so waiting for all but the newest D - 2 chunks' loads means that the chunk has landed. Rows past N and M read
// zeros. Lane l holds y[16 mt + l % 16][16 t + 4 (l / 16) + v], v = 0..3.
// Bound: HBM. 151936 x 2048 head (622 MB, 3 cold copies), MI355X, us (direct fragments -> this; hipBLASLt): 16 rows
// 134 -> 104 (205), 32 rows 145 -> 114 (147), 48 rows 156 -> 133 (144), 64 rows 166 -> 144 (154); one more slot at 16
// rows, which costs the second workgroup per CU, 110.
// Slots: two workgroups share a CU at up to 32 rows (80 and 72 KB of LDS), one at more (84 and 96 KB). There, weights of
// more than one workgroup a CU whose chunks are few, so that the pipeline's start and end count, take two slots and so
// two workgroups a CU (f16w_short). us at 48 and 64 rows, two slots / three: 151936 x 128 15.6 and 17.8 / 24.0 and 27.2, x
// 512 34.8 and 39.1 / 44.0 and 49.1, x 1024 62 and 67 / 69 and 79, x 1536 92 and 100 / 100 and 111, x 2048 134 and 141 / 130
// and 142; 18944 x 1024 11.6 and 12.7 / 13.2 and 14.9; but 2048 x 2048 13.0 and 13.6 / 10.0 and 11.4.
constexpr int f16w_slots(int MT) { return MT == 1 ? 4 : 3; }
constexpr bool f16w_short(int N, int K) { return N > 64 * 256 && K <= 1536; }
constexpr int f16w_swz(int r) { return ((r & 3) << 2) | (r >> 2); }
template <int MT, int D>
__global__ __launch_bounds__(256) void gemm_f16w_rows_kernel(const f16* __restrict__ x, const f16* __restrict__ w,
                                                             f16* __restrict__ y, int M, int N, int K) {
  constexpr int kTile = 16 * 256;                           // bytes of 16 rows of a chunk
  constexpr int kSlot = (4 + MT) * kTile;                   // a chunk: the waves' W tiles, then x
  constexpr int kLoads = 4 + MT;                            // a wave's loads of a chunk
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4, KC = K >> 7;
  const int n0 = 16 * (blockIdx.x * 4 + wave);
  const int rows = max(0, min(16, N - n0));
  // (hipcc multiplies 64-bit sizes in vector registers; the resource of a direct-to-LDS load must be scalar)
  const uint64_t first = (uint64_t)min(n0, N) * (uint64_t)K;
  const uint64_t first_s = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(first >> 32)) << 32) |
                           (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)first);
  const __amdgpu_buffer_rsrc_t wr = make_rsrc(w + first_s, (uint32_t)__builtin_amdgcn_readfirstlane(rows * K * 2));
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(x, (uint32_t)(M * K * 2));
  // W load u of a wave: rows 4 u + lane / 16, slot lane % 16 of the row. x load mt: row 16 mt + tid / 16, slot tid % 16
  int woff[4], xoff[MT];
#pragma unroll
  for (int u = 0; u < 4; ++u) woff[u] = 2 * ((4 * u + q) * K + 8 * (r ^ f16w_swz(4 * u + q)));
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int row = 16 * mt + (tid >> 4);
    xoff[mt] = row < M ? 2 * (row * K + 8 * ((tid & 15) ^ f16w_swz(tid >> 4))) : kOutOfRange - 256 * KC;
  }
  const uint32_t base = lds_addr(smem);
  auto issue = [&](int d, int c) {                          // kLoads loads, always (chunks past the end read zeros)
    const bool live = c < KC;
    const uint32_t at = base + d * kSlot;
#pragma unroll
    for (int u = 0; u < 4; ++u) dma16_nt(wr, live ? woff[u] + 256 * c : kOutOfRange, at + wave * kTile + 1024 * u);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) dma16(xr, live ? xoff[mt] + 256 * c : kOutOfRange, at + (4 + mt) * kTile + 1024 * wave);
  };
#pragma unroll
  for (int d = 0; d < D - 1; ++d) issue(d, d);
  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < KC; c0 += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      const int c = c0 + d;
      if (c < KC) {                                         // uniform: every wave runs the same chunks
        lds_wait_barrier<(D - 2) * kLoads>();               // chunk c has landed in every wave; slot c - 1 is free
        issue((d + D - 1) % D, c + D - 1);
        const uint8_t* slot = smem + d * kSlot;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const int at = 256 * r + 16 * ((4 * q + s) ^ f16w_swz(r));
          const f16x8 a = *reinterpret_cast<const f16x8*>(slot + wave * kTile + at);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            const f16x8 b = *reinterpret_cast<const f16x8*>(slot + (4 + mt) * kTile + at);
            acc[mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, acc[mt], 0, 0, 0);
          }
        }
      }
    }
  }
  vm_drain();                                               // no load into LDS is left in flight
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = 16 * mt + r, n = n0 + 4 * q;
    if (m < M && n < N) {
      f16* dst = y + (size_t)m * N + n;
      if (n + 4 <= N && (reinterpret_cast<uintptr_t>(dst) & 7) == 0) {
        const f16x2 lo = {(f16)acc[mt][0], (f16)acc[mt][1]}, hi = {(f16)acc[mt][2], (f16)acc[mt][3]};
        *reinterpret_cast<uint2*>(dst) = make_uint2(as_u32(lo), as_u32(hi));
      } else {
#pragma unroll
        for (int v = 0; v < 4; ++v)
          if (n + v < N) dst[v] = (f16)acc[mt][v];
      }
    }
  }
}

template <int MT, int D>
hipError_t launch_f16w_rows(const f16* x, const f16* w, f16* y, int M, int N, int K, hipStream_t st) {
  constexpr size_t lds = (size_t)D * (4 + MT) * 16 * 256;
  if (lds > 65536) {
    static std::atomic<uint64_t> done{0};
    if (hipError_t e = allow_lds_once(done, gemm_f16w_rows_kernel<MT, D>, lds)) return e;
  }
  return launch(gemm_f16w_rows_kernel<MT, D>, dim3((unsigned)((N + 63) / 64)), dim3(256), lds, st, x, w, y, M, N, K);
}

hipError_t gemm_f16w_rows_launch(const f16* x, const f16* w, f16* y, int M, int N, int K, hipStream_t st) {
  switch ((M + 15) / 16) {
    case 1: return launch_f16w_rows<1, f16w_slots(1)>(x, w, y, M, N, K, st);
    case 2: return launch_f16w_rows<2, f16w_slots(2)>(x, w, y, M, N, K, st);
    case 3:
      if (f16w_short(N, K)) return launch_f16w_rows<3, 2>(x, w, y, M, N, K, st);
      return launch_f16w_rows<3, f16w_slots(3)>(x, w, y, M, N, K, st);
    default:
      if (f16w_short(N, K)) return launch_f16w_rows<4, 2>(x, w, y, M, N, K, st);
      return launch_f16w_rows<4, f16w_slots(4)>(x, w, y, M, N, K, st);
  }
}

namespace {
template <int M, int RW, int CH>
hipError_t launch_head(const f16* x, const f16* w, f16* y, int mrows, int N, int K, hipStream_t st) {
  const dim3 grid((unsigned)((N + 4 * RW - 1) / (4 * RW))), block(256);
  return launch(gemv_f16_kernel<M, RW, CH>, grid, block, (size_t)M * K * 2, st, x, w, y, N, K, nullptr, mrows);
}
}  // namespace

hipError_t gemv_f16_launch(const f16* x, const f16* w, f16* y, int M, int N, int K, hipStream_t st) {
  switch (M) {
    case 1: return launch_head<1, kHeadRows, kHeadChunks>(x, w, y, 1, N, K, st);
    case 2: return launch_head<2, kHeadRows, kHeadChunks>(x, w, y, 2, N, K, st);
    case 3: return launch_head<3, kHeadRows, kHeadChunks>(x, w, y, 3, N, K, st);
    case 4: return launch_head<4, kHeadRows, kHeadChunks>(x, w, y, 4, N, K, st);
    // more rows: 8 weight rows per wave, two chunks in flight (the head, 3 cold copies: 8 rows 119.5 us against
    // 126.6 for 4 per wave and 163.7 for 2; hipBLASLt 203.6). The MFMA kernel would take 101 there, but up to 8 rows a
    // row has the bits it has alone
    default: {
      const bool x_fits = (size_t)M * K * 2 <= 65536;      // the dot2 kernels stage x whole
      if (M <= 8 && x_fits) return launch_head<8, 8, 2>(x, w, y, M, N, K, st);
      if (K % 128) return x_fits && M <= 16 ? launch_head<16, 8, 2>(x, w, y, M, N, K, st) : hipErrorInvalidValue;
      return gemm_f16w_rows_launch(x, w, y, M, N, K, st);
    }
  }
}

int head_pick_parts(int N) { return (N + 4 * kHeadRows - 1) / (4 * kHeadRows); }

hipError_t head_pick_launch(const f16* x, const f16* w, f16* y, int N, int K, uint64_t* pick, int64_t* tokens,
                            int64_t* positions, int64_t* out, int out_cap, int* out_count, const f16* embed, f16* h_out,
                            hipStream_t st) {
  const int parts = head_pick_parts(N);
  if (hipError_t e = launch(gemv_f16_kernel<1, kHeadRows, kHeadChunks, true>, dim3(parts), dim3(256), (size_t)K * 2, st,
                            x, w, y, N, K, pick, 1))
    return e;
  return launch(head_pick_kernel, dim3(1), dim3(kPickThreads), 0, st, pick, parts, tokens, positions, out, out_cap,
                out_count, embed, K, h_out);
}

hipError_t rmsnorm_launch(const f16* x, const f16* w, f16* out, int M, int H, float eps, hipStream_t st) {
  return launch(rmsnorm_kernel, dim3(M), dim3(256), 0, st, x, w, out, H, eps);
}

// table[m][i] = fp16 (cos, sin) of positions[m] * inv_freq[i] (rope_cos_sin): the RoPE factors of a step, shared by
// every head and layer; the multi-row q|k|v GEMMs read them in their store
__global__ __launch_bounds__(256) void rope_table_kernel(const int64_t* __restrict__ pos, const float* __restrict__ inv_freq,
                                                         uint32_t* __restrict__ table, int M) {
  const int gid = blockIdx.x * blockDim.x + threadIdx.x;
  if (gid >= M * 64) return;
  f16 c, s;
  rope_cos_sin(pos[gid >> 6], inv_freq[gid & 63], c, s);
  table[gid] = as_u32(f16x2{c, s});
}

hipError_t rope_table_launch(const int64_t* pos, const float* inv_freq, uint32_t* table, int M, hipStream_t st) {
  return launch(rope_table_kernel, dim3((unsigned)((M * 64 + 255) / 256)), dim3(256), 0, st, pos, inv_freq, table, M);
}

hipError_t rope_kv_launch(const f16* qkv, const int64_t* pos, const float* inv_freq, f16* q_out, f16* k_cache,
                          f16* v_cache, int M, int Hq, int Hkv, int L, bool permuted, hipStream_t st) {
  const long threads = (long)M * (Hq + 2 * Hkv) * 64;
  return launch(rope_kv_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, qkv, pos, inv_freq, q_out,
                k_cache, v_cache, M, Hq, Hkv, L, permuted);
}

namespace {
// combine = false: the partials are left for the caller (their count in *parts; with one partition the kernel writes
// out itself and *parts is 1)
template <int G, int KB>
hipError_t launch_attention(const f16* q, const f16* k, const f16* v, const int64_t* pos, f16* out, int M, int Hq,
                            int Hkv, int L, int max_keys, float scale, void* ws, size_t ws_bytes, hipStream_t st,
                            int max_parts = kAttnMaxParts, bool combine = true, int* parts = nullptr) {
  const int max_waves = (G == 1 && KB == 32) ? 16 : 8;
  const long blocks = (long)M * (Hq / G);
  // key partitions: when the (token, group) blocks cannot fill the chip, split the keys so that about
  // kAttnTargetBlocks blocks run, each with at least kAttnMinKeys keys, within the workspace
  int P = 1;
  if (ws && ws_bytes > kAttnCounterBytes && blocks < kAttnTargetBlocks && max_keys >= kAttnMinSplitKeys) {
    P = (int)std::min<long>({(kAttnTargetBlocks + blocks - 1) / blocks, (max_keys + kAttnMinKeys - 1) / kAttnMinKeys,
                             (long)max_parts});
    const size_t per = (size_t)blocks * G * kAttnRec * sizeof(float);
    P = (int)std::max<size_t>(1, std::min<size_t>((size_t)P, (ws_bytes - kAttnCounterBytes) / per));
  }
  const int CH = ((max_keys + P - 1) / P + KB - 1) / KB * KB;   // keys per partition, whole steps
  P = (max_keys + CH - 1) / CH;
  int waves = 1;                                              // enough waves to give each one step of keys
  while (waves < max_waves && waves * KB < CH) waves *= 2;
  // prefill-sized launches (many blocks) take at most 4 waves per block: merging 8 waves' partial outputs through LDS
  // costs more than the keys they share out (measured: 3B prompt of 512 tokens 58 -> 48 us, 7B 99 -> 70 us)
  if (blocks * P >= kAttnManyBlocks && waves > 4) waves = 4;
  const size_t lds = (size_t)waves * G * 2 * 4 + (size_t)waves * G * kHeadDim * 4;
  float* part = ws ? reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + kAttnCounterBytes) : nullptr;
  if (parts) *parts = P;
  hipError_t e = launch(attention_kernel<G, KB>, dim3((unsigned)blocks, P), dim3(64 * waves), lds, st, q, k, v, pos,
                        out, Hq, Hkv, L, scale, CH, part);
  if (e != hipSuccess || P == 1 || !combine) return e;
  const long threads = (long)M * Hq * kHeadDim;
  return launch(attention_combine, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, part, out, (int)blocks, G,
                P, Hq);
}
// multi-token steps and prompts on MFMA: one wave per (KV head, 16 query rows, key partition); partitions while the
// waves number fewer than kAttnMfmaTargetWaves, at most one per kAttnMinKeys of max_keys, within the workspace (each
// wave splits the keys its rows actually attend, so a bound well above the real count costs nothing)
hipError_t launch_attention_mfma(const f16* q, const f16* k, const f16* v, const int64_t* pos, f16* out, int M,
                                 int Hq, int Hkv, int L, int max_keys, float scale, void* ws, size_t ws_bytes,
                                 hipStream_t st) {
  const int G = Hq / Hkv;
  const long waves = (long)((M * G + 15) / 16) * Hkv;
  int P = 1;
  if (ws && ws_bytes > kAttnCounterBytes && waves < kAttnMfmaTargetWaves && max_keys >= 2 * kAttnMinKeys) {
    P = (int)std::min<long>({(kAttnMfmaTargetWaves + waves - 1) / waves, (max_keys + kAttnMinKeys - 1) / kAttnMinKeys,
                             (long)kAttnMaxParts});
    const size_t per = (size_t)M * Hkv * G * kAttnRec * sizeof(float);
    P = (int)std::max<size_t>(1, std::min<size_t>((size_t)P, (ws_bytes - kAttnCounterBytes) / per));
  }
  // the partials after the workspace's first kAttnCounterBytes (unused, kept for the layout)
  float* part = ws ? reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + kAttnCounterBytes) : nullptr;
  hipError_t e = launch(attention_mfma, dim3((unsigned)waves, P), dim3(64), 0, st, q, k, v, pos, out, M, Hq, Hkv, L,
                        scale, part);
  if (e != hipSuccess || P == 1) return e;
  const long threads = (long)M * Hq * kHeadDim;
  return launch(attention_combine, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, part, out, M * Hkv, G, P,
                Hq);
}
template <int RG, int KG>
constexpr size_t prompt_lds() {
  return std::max<size_t>((size_t)2 * 2 * 32 * KG * kHeadDim * 2, (size_t)(KG - 1) * RG * 66 * 256);
}
// key partitions of attend_prompt while its workgroups number fewer than `target`, at most one per kAttnPromptMinKeys of
// max_keys, within the workspace (a workgroup splits the keys its rows actually attend)
template <int RG, int KG>
int prompt_parts(int M, int Hq, int Hkv, int max_keys, const void* ws, size_t ws_bytes, long target) {
  const long wgs = ((long)M * (Hq / Hkv) + 32 * RG - 1) / (32 * RG) * Hkv;
  if (!ws || ws_bytes <= kAttnCounterBytes || wgs >= target || max_keys < 2 * kAttnPromptMinKeys) return 1;
  // (a workgroup of KG = 4 has its CU to itself: one round of them)
  const long P = std::min<long>({KG == 4 ? std::max(1L, 256 / wgs) : (target + wgs - 1) / wgs, (max_keys + kAttnPromptMinKeys - 1) / kAttnPromptMinKeys,
                                 (long)kAttnManyParts});
  const size_t per = (size_t)M * Hq * kAttnRec * sizeof(float);
  return (int)std::max<size_t>(1, std::min<size_t>((size_t)P, (ws_bytes - kAttnCounterBytes) / per));
}
float* attn_partials(void* ws) {
  return ws ? reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + kAttnCounterBytes) : nullptr;
}
// prompts whose keys number few: one workgroup per (KV head, 64 query rows, key partition)
hipError_t launch_attention_prompt(const f16* q, const f16* k, const f16* v, const int64_t* pos, f16* out, int M, int Hq,
                                   int Hkv, int L, int max_keys, float scale, void* ws, size_t ws_bytes, hipStream_t st) {
  const int G = Hq / Hkv;
  const int tiles = (int)(((long)M * G + 63) / 64);
  const int P = max_keys < kAttnPromptSplitKeys ? 1 : prompt_parts<2, 2>(M, Hq, Hkv, max_keys, ws, ws_bytes, 512);
  static_assert(prompt_lds<2, 2>() <= 65536 && kAttnPromptLongKeys / kAttnPromptMinKeys <= kAttnMaxParts, "");
  hipError_t e = launch(attention_prompt<2, 2>, dim3((unsigned)(tiles * Hkv), P), dim3(256), prompt_lds<2, 2>(), st, q, k, v,
                        pos, out, M, Hq, Hkv, L, scale, tiles, attn_partials(ws));
  if (e != hipSuccess || P == 1) return e;
  const long threads = (long)M * Hq * kHeadDim;
  return launch(attention_combine, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, st, attn_partials(ws), out, M * Hkv,
                G, P, Hq);
}
// attention_select: the launch holds both kernels' workgroups
template <int RG, int KG, bool HEADS>
hipError_t launch_attention_select(const f16* q, const f16* k, const f16* v, const int64_t* pos, f16* out, int M,
                                   int Hq, int Hkv, int L, int max_keys, float scale, void* ws, size_t ws_bytes,
                                   hipStream_t st, long target, int from) {
  const int G = Hq / Hkv;
  const int tiles = (int)(((long)M * G + 32 * RG - 1) / (32 * RG));
  AttnSplit sp{from, 1, prompt_parts<RG, KG>(M, Hq, Hkv, max_keys, ws, ws_bytes, target), HEADS, 1};
  const long units = HEADS ? (long)M * Hq : ((long)M * G + 15) / 16 * Hkv, room = HEADS ? kAttnSelectBlocks : kAttnMfmaTargetWaves;
  const int few_keys = std::min(max_keys, from - 1), least = HEADS ? 128 : kAttnMinKeys;
  if (ws && ws_bytes > kAttnCounterBytes && units < room && few_keys >= 2 * least) {
    const size_t per = (size_t)M * Hq * kAttnRec * sizeof(float);
    sp.few = (int)std::min<long>({(room + units - 1) / units, (few_keys + least - 1) / least,
                                  (long)(HEADS ? kAttnManyParts : kAttnMaxParts), (long)((ws_bytes - kAttnCounterBytes) / per)});
    sp.few = std::max(sp.few, 1);
  }
  sp.room = std::max(sp.few, sp.many);
  constexpr size_t lds = prompt_lds<RG, KG>();
  static_assert(lds >= (size_t)2 * kHeadDim * kAttnVtPitch, "attend_mfma's V");
  const long few_blocks = HEADS || KG != 4 ? units * sp.few : (units * sp.few + 1) / 2;
  if (lds > 65536) {
    static std::atomic<uint64_t> done{0};
    if (hipError_t e = allow_lds_once(done, attention_select<RG, KG, HEADS>, lds)) return e;
  }
  hipError_t e = launch(attention_select<RG, KG, HEADS>, dim3((unsigned)std::max((long)tiles * Hkv * sp.many, few_blocks)),
                        dim3(256), lds, st, q, k, v, pos, out, M, Hq, Hkv, L, scale, tiles, attn_partials(ws), sp);
  if (e != hipSuccess || sp.room == 1) return e;
  return launch(attention_combine_many, dim3((unsigned)(M * Hq)), dim3(kHeadDim), 0, st, attn_partials(ws), pos, out, M, Hq,
                Hkv, L, sp);
}
// Which kernel serves a call. attend_prompt shares K and V among a KV head's rows and splits the keys over the chip up to
// kAttnManyParts ways, where attention_kernel has every query head read them on its own and attention_mfma's waves load
// theirs unshared, both at most 16 ways; its prologue and merge cost more. Its figures here are with a bound equal to the
// keys (others -> it).
//   Few rows (below kAttnPromptMinRows per KV head) from 2048 keys and M Hq keys of 80 K, one token from 128 K (the others
//   can leave its merge to the o projection): us, one token, 28 / 4 heads, 3000 keys 16.7 -> 12.1, 16000 45 -> 19, 24000
//   65 -> 22; 12 / 2 heads 12000 18.3 -> 16.5; 4 tokens of 16 / 2 heads on 6000 23.4 -> 14.7; 16 on 3000 16.1 -> 14.1
//   (1500: 11.2 against 11.9). With one query head per KV head there is nothing to share below 16 rows (one token, 16 / 16
//   heads on 16000 keys 29.9 -> 32.9; 2 heads per KV head 26.2 -> 22.9), and steps of 64 or more (token, KV head)s below 32
//   rows keep attention_kernel. A workspace of fewer than 16 partitions keeps the others, too: that of 4 MB which the
//   Python binding gives serves M Hq <= 496.
//   More rows, us: 65 to 128 keys, which attention_mfma splits and attend_prompt need not (16 / 2 heads, 64 tokens on 64
//   cached 9.0 -> 8.5, 128 tokens 10.6 -> 8.5; up to 64 keys neither does, 64 tokens 5.5 -> 7.7). Up to 383, where
//   attend_prompt's one walk of the keys grows with them and the other's with the rows, from M Hq of 4 keys + 256 (16 / 2
//   heads, 64 tokens on 128 cached 9.2 -> 9.4, 80 on 128 10.4 -> 10.1, 64 on 256 10.3 -> 11.0, 128 on 128 12.9 -> 10.1; 12 /
//   2, 86 on 128 9.9 -> 10.1, 107 on 128 10.5 -> 10.1; 28 / 4, 64 on 128 11.5 -> 9.5). Beyond, from M Hq keys of 700 K (48
//   tokens on 512 cached 11.0 -> 11.9, on 1500 16.4 -> 14.8; 64 on 512 12.2 level, on 1000 15.8 -> 14.6; 4 / 4 heads, 384
//   on 64 12.6 -> 13.1, on 128 13.7 -> 13.1).
// attn_bound_from: the keys from which a call's bound on them lets attend_prompt serve few rows (0: never), attn_prompt_bound
// whether it lets it serve more. attn_keys_from: the keys from which, in attention_select, it then does (one token 50 K Hq
// keys, few rows 76 K M Hq keys, up to 383 rows 2048 keys, beyond 192: where the two bodies crossed in sweeps of 200 ..
// 16000 keys on 4096- to 16384-row caches).
bool attn_prompt_bound(long work, int max_keys) {
  if (max_keys >= kAttnPromptSplitKeys) return work * max_keys >= kAttnPromptWork;
  return max_keys > 64 && (max_keys <= 128 || work >= 4L * max_keys + 256);
}
int attn_bound_from(int M, int Hq, int Hkv, size_t ws_bytes) {
  const int G = Hq / Hkv;
  const long rows = (long)M * G, work = (long)M * Hq;
  if (G == 1 && rows < 16) return 0;
  if (rows < kAttnMfmaMinRows && (long)M * Hkv >= 64) return 0;
  if (ws_bytes < kAttnCounterBytes + (size_t)16 * M * Hq * kAttnRec * sizeof(float)) return 0;
  return (int)std::max<long>(kAttnLongKeys, ((M == 1 ? kAttnLongWorkOne : kAttnLongWork) + work - 1) / work);
}
int attn_keys_from(int M, int Hq, int Hkv) {
  const long rows = (long)M * (Hq / Hkv), work = (long)M * Hq;
  if (rows >= kAttnPromptMinRows) return kAttnPromptKeysFrom;
  if (rows >= kAttnMfmaMinRows) return kAttnRowsKeysFrom;
  return (int)(((M == 1 ? kAttnOneWorkFrom : kAttnFewWorkFrom) + work - 1) / work);
}
}  // namespace

hipError_t attention_launch(const f16* q, const f16* k, const f16* v, const int64_t* pos, f16* out, int M, int Hq,
                            int Hkv, int L, int max_keys, float scale, void* ws, size_t ws_bytes, hipStream_t st) {
  const long rows = (long)M * (Hq / Hkv);
  if (!ws) ws_bytes = 0;
  const int from = attn_keys_from(M, Hq, Hkv);
  if (rows >= kAttnPromptMinRows) {
    if (!attn_prompt_bound((long)M * Hq, max_keys))
      return launch_attention_mfma(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
    // M tokens attend M keys at least, unless they share positions; a bound of more may lie far above them
    const bool sure = M >= from, wide = (rows + 63) / 64 * Hkv < kAttnPromptWide;
    if (max_keys < kAttnPromptLongKeys || (sure && !wide && prompt_parts<2, 2>(M, Hq, Hkv, max_keys, ws, ws_bytes, 512) == 1))
      return launch_attention_prompt(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
    if (wide)
      return launch_attention_select<1, 4, false>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st, 512, sure ? 1 : from);
    return launch_attention_select<2, 2, false>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st, 512, sure ? 1 : from);
  }
  const int bound_from = attn_bound_from(M, Hq, Hkv, ws_bytes);
  if (bound_from > 0 && max_keys >= bound_from) {
    if (rows < kAttnMfmaMinRows)
      return launch_attention_select<2, 2, true>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st, 256, from);
    // 64 rows a workgroup up to 128 rows, 32 beyond (28 / 4 heads, 32 tokens on 24000, in a workspace that holds their
    // partitions: 43 us against 53; 16 / 2, 16 on 24000: 24 against 27)
    if (rows <= 128)
      return launch_attention_select<2, 2, false>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st, 256, from);
    return launch_attention_select<1, 4, false>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st, 256, from);
  }
  if (rows >= kAttnMfmaMinRows)
    return launch_attention_mfma(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
  if ((long)M * Hkv < 64)                                     // few tokens: one query head per block, short steps
    return launch_attention<1, 32>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
  switch (Hq / Hkv) {
    case 1: return launch_attention<1, 64>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
    case 2: return launch_attention<2, 64>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
    case 4: return launch_attention<4, 32>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
    case 6: return launch_attention<6, 32>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
    case 7: return launch_attention<7, 32>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
    case 8: return launch_attention<8, 32>(q, k, v, pos, out, M, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t attention_partials_launch(const f16* q, const f16* k, const f16* v, const int64_t* pos, f16* out, int Hq,
                                     int Hkv, int L, int max_keys, float scale, void* ws, size_t ws_bytes, int* parts,
                                     hipStream_t st) {
  // one token: the decode kernel with one query head per block (the MFMA kernel takes 32 or more rows per KV head)
  if (Hq / Hkv >= kAttnMfmaMinRows || Hkv >= 64) return hipErrorInvalidValue;
  // a bound of a long cache: merged here, into out, as attention_launch does; the partials then follow out in the workspace
  const size_t xbytes = (size_t)Hq * kHeadDim * sizeof(f16);
  const int bound_from = ws_bytes > xbytes ? attn_bound_from(1, Hq, Hkv, ws_bytes - xbytes) : 0;
  if (bound_from > 0 && max_keys >= bound_from) {
    *parts = 1;
    return launch_attention_select<2, 2, true>(q, k, v, pos, out, 1, Hq, Hkv, L, max_keys, scale,
                                               static_cast<uint8_t*>(ws) + xbytes, ws_bytes - xbytes, st, 256,
                                               attn_keys_from(1, Hq, Hkv));
  }
  return launch_attention<1, 32>(q, k, v, pos, out, 1, Hq, Hkv, L, max_keys, scale, ws, ws_bytes, st, kAttnXMaxParts,
                                 false, parts);
}

}  // namespace lowbit
