// Prefill GEMM on the MFMA layout, M > 64: y[M, N] = x[M, K] . dequant(W)^T with v_mfma_f32_16x16x32_f16, reading
// the int4 weights directly (no fp16 copy of W). The reference's prefill dequantizes into an fp16 W and calls cuBLAS
// (lowbit/ops.py:126-135,163-178); this kernel computes the same products without writing W out.
//
// Operands (lane l, r = l % 16, q = l / 16), as in the skinny kernel:
//   A (16 weight rows x 32 k): lane l's 16-byte piece of a 1 KB block holds row r, k = 128 c + 32 q + 8 s + 0..7 in
//     word s, which feeds k-step s. Each word is decoded to (u - 8) exactly in fp16 and multiplied by the row's fp16
//     group scale with one rounding, so A holds exactly the dequantized weights of the reference's rule.
//   B (32 k x 16 activation rows): x[m0 + 16 mt + r][128 c + 32 q + 8 s + 0..7], 16 bytes from LDS.
//   D: lane l holds y[m0 + 16 mt + r][16 t + 4 q + v], v = 0..3.
//
// Workgroup: 4 waves, each owning PT 16-row tiles (64 PT weight rows per workgroup) against 16 MT activation rows. Every
// wave decodes only its own rows, so no weight is decoded twice in a workgroup; a 128-k chunk of x goes straight from
// memory to LDS (direct-to-LDS loads, no registers) and is shared by the waves, double buffered. LDS rows are 256 bytes,
// their 16-byte blocks permuted by the row (xswz: block b of row m at b ^ xswz(m % 16)), so that a fragment's 16 rows
// meet different banks. Rows past N and activation rows past M read zeros or are never stored.
//
// Pipeline: the chunk is walked in groups of two activation tiles; while a group's 2 PT MFMAs run, the next group's B
// fragments are read and a share of the next k-step's A fragments decoded, across the chunk's end too, and one barrier per
// chunk, which waits for x alone, leaves the weights of the chunk after next in flight. The version before (chunk decoded
// whole, fragment reads waited for as they were issued, x through registers, a barrier that drained every load) left the
// matrix cores 31% busy at 2048 x 3584 x 18944; this one keeps them 45-50% busy there, at the clock that the power limit
// leaves (1.8-2.0 GHz; MFMAs with the decode's vector instructions between them and nothing else reach 1.6 PFLOP/s).
// MI355X, graph-timed, cold weights, one run, rows x K x N, us (before -> now, dequantize + hipBLASLt): 128 x 3584 x 18944
// 42.8 -> 36.8 (67.3); 333 x 2048 x 11008 34.4 -> 32.2 (43.5); 333 x 11008 x 2048 49.1 -> 37.0 (55.1); 512 x 18944 x 3584
// 111 -> 87 (204); 700 x 2048 x 22016 90 -> 75 (106); 1000 x 3584 x 18944 184 -> 140 (161); 2048 x 3584 x 18944 334 -> 258
// (341).
// Not kept: the same loop on 32x32x16 MFMAs (271-294 at 2048 x 3584 x 18944, more power per product), 8 tiles x 4
// per wave (registers spill; the compiler moves accumulators between register files at 16), 8-wave workgroups.
//
// Work items: the tiles that fill whole rounds of the chip one workgroup each, the rest with K split S ways
// (plan_gemm_prefill), activation groups fastest, then row groups, and the workgroup -> item map puts consecutive items
// on the same XCD (workgroup i runs on XCD i % 8), so the workgroups that share weight rows share that XCD's L2. The
// splits of a tile write fp32 partials to the workspace (agent-coherent stores); the last to arrive on the tile's counter
// adds them in split order and resets the counter, as in the skinny kernel.
#include <algorithm>
#include <climits>
#include <type_traits>
#include <utility>

#include "kernels.hpp"

namespace lowbit {

namespace {

// f(integral_constant 0) .. f(integral_constant N - 1)
template <int... I, typename F>
__device__ __forceinline__ void unrolled_seq(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unrolled(F&& f) {
  unrolled_seq(std::make_integer_sequence<int, N>{}, f);
}

constexpr int xswz(int r) { return ((r & 3) << 2) | (r >> 2); }

}  // namespace

template <int MT, int PT, bool ROPE>
__global__ __launch_bounds__(256, 2) void gemm_prefill(
    const f16* __restrict__ x, const uint8_t* __restrict__ w, const f16* __restrict__ s, f16* y, int M, int N, int K,
    int G, int S, int MG, int full, int items, uint32_t* __restrict__ ctr, float* __restrict__ part, Epilogue epi) {
  constexpr int kXBuf = 16 * MT * 256;                      // one staged chunk of x
  constexpr int kRows = 64 * PT;                            // weight rows per workgroup
  args_in_sgprs(x, w, s, y, M, N, K, G, S, MG, full, items, ctr, part, epi.aux);
  constexpr int kThreads = 256;
  constexpr int XP = 16 * MT * 16 / kThreads;               // 16-byte x pieces per thread and chunk
  static_assert(XP >= 1 && XP * kThreads == 16 * MT * 16, "x pieces must divide evenly");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;

  // workgroup -> work item: first `full` whole tiles, then the others S splits each; consecutive items on one XCD (full
  // is a multiple of 8 unless it is all the tiles or none)
  const bool whole = (int)blockIdx.x < full;
  const int b0 = whole ? blockIdx.x : blockIdx.x - full, n_items = whole ? full : items - full;
  const int per = n_items >> 3, rem = n_items & 7, xcd = b0 & 7, idx = b0 >> 3;
  const int item = xcd < rem ? xcd * (per + 1) + idx : rem * (per + 1) + (xcd - rem) * per + idx;
  if (whole) S = 1;
  const int sp = item % S, tile = whole ? item : full + item / S, mg = tile % MG, ng = tile / MG;
  const int m0 = 16 * MT * mg, n0 = kRows * ng;
  const int ntiles = (N + 15) >> 4, KC = K >> 7, KG = K / G, cpg = G >> 7;
  const int cb = (int)((int64_t)KC * sp / S), ce = (int)((int64_t)KC * (sp + 1) / S);
  const int nsteps = ce - cb;
  const size_t tile_bytes = (size_t)8 * K;

  // Weight rows past N read other rows' nibbles or zeros; their scales lie past the end (zeros) and their outputs are not
  // stored. The uniform part of an offset is in the resource's base, so one register serves all tiles. Chunks past the
  // range are clamped to its last one and never consumed.
  const uint8_t* wp[PT];
  int wrows[PT], tc[PT];                                    // (uniform)
#pragma unroll
  for (int i = 0; i < PT; ++i) {
    const int t = n0 / 16 + PT * wave + i;
    tc[i] = min(t, ntiles - 1);
    wrows[i] = t < ntiles ? min(16, N - 16 * t) : 0;
    wp[i] = w + tc[i] * tile_bytes;
  }
  const int woff = 64 * r + 16 * q, soff = 2 * r * KG;
  // piece tid + kThreads u of a staged chunk is slot p % 16 of row p / 16, which holds the row's 16-byte block
  // slot ^ xswz(row % 16) (kThreads is a multiple of 256, so that block is the same for every u); each u has a resource
  // of its own, from its first row's chunk to the end of x (rows past M read zeros)
  const int xoff = ((tid >> 4) * K + 8 * ((tid & 15) ^ xswz((tid >> 4) & 15))) * 2;
  const uint32_t xdst = lds_addr(smem) + 1024 * wave;

  u32x4 rw[2][PT];
  uint32_t rs[2][PT];
  const uint32_t gmagic = cpg == 1 ? 0u : (uint32_t)(0xFFFFFFFFu / (uint32_t)cpg) + 1u;   // c / cpg == mulhi(c, gmagic)
  auto issue_w = [&](int d, int chunk) {                    // 2 PT loads (lds_wait_barrier counts them)
    const int c = min(chunk, ce - 1);
    const int g = cpg == 1 ? c : (int)__umulhi((uint32_t)c, gmagic);
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      const int at = c * wrows[i] * 64;                     // (weights are re-read by other m-groups: default policy)
      rw[d][i] = buffer_load16(make_rsrc(wp[i] + at, (uint32_t)(wrows[i] * (K / 2) - at)), woff);
      const int sat = 16 * tc[i] * KG + g;
      rs[d][i] = buffer_load2(make_rsrc(s + sat, (uint32_t)(N * KG - sat) * 2u), soff);
    }
  };
  // the activation rows of a full tile share one resource, the row part of the offset in a scalar register; the last,
  // ragged tile takes one per u, cut off at the end of x (a scalar offset past the end would escape the bounds check)
  const bool ragged = m0 + 16 * MT > M;
  const uint8_t* xtile = reinterpret_cast<const uint8_t*>(x) + (size_t)m0 * K * 2;
  const int ustep = kThreads / 8 * K;                       // bytes from one u's rows to the next one's
  const __amdgpu_buffer_rsrc_t xr = make_rsrc(xtile, (uint32_t)(16 * MT * K * 2));
  auto issue_x = [&](int b, int c) __attribute__((always_inline)) {   // chunk c of x straight into LDS buffer b
    if (!ragged) {
      int at = 256 * c;
#pragma unroll
      for (int u = 0; u < XP; ++u, at += ustep) dma16_s(xr, xoff, at, xdst + b * kXBuf + 16 * kThreads * u);
    } else {
#pragma unroll
      for (int u = 0; u < XP; ++u) {
        const int left = max(0, M - m0 - kThreads / 16 * u) * 2 * K - 256 * c;
        dma16(make_rsrc(xtile + (size_t)u * ustep + 256 * c, (uint32_t)max(0, left)), xoff,
              xdst + b * kXBuf + 16 * kThreads * u);
      }
    }
  };

  f32x4 acc[PT][MT];
#pragma unroll
  for (int i = 0; i < PT; ++i)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[i][mt] = f32x4{0.f, 0.f, 0.f, 0.f};

  const f16x2 m1032 = {(f16)-1032.0f, (f16)-1032.0f}, m72 = {(f16)-72.0f, (f16)-72.0f};
  const f16x2 inv16 = {(f16)0.0625f, (f16)0.0625f};
  const DecodeRegs dc = decode_regs();                      // masks and magic in registers: v_and_or_b32
  int xrd[4];                                               // lane (r, q): block 4 q + st of row r
#pragma unroll
  for (int st = 0; st < 4; ++st) xrd[st] = 256 * r + 16 * ((4 * q + st) ^ xswz(r));
  auto decode = [&](int d, int i, int st) {                 // (u - 8) exact, times the scale: one rounding
    const f16 sv = __builtin_bit_cast(f16, (uint16_t)rs[d][i]);
    const f16x2 sc = {sv, sv};
    const uint32_t wd = rw[d][i][st], w8 = wd >> 8;
    const f16x2 p0 = (as_f16x2((wd & dc.lo) | dc.magic) + m1032) * sc;
    const f16x2 p1 = (as_f16x2((wd & dc.hi) | dc.magic) * inv16 + m72) * sc;
    const f16x2 p2 = (as_f16x2((w8 & dc.lo) | dc.magic) + m1032) * sc;
    const f16x2 p3 = (as_f16x2((w8 & dc.hi) | dc.magic) * inv16 + m72) * sc;
    return __builtin_bit_cast(f16x8, u32x4{as_u32(p0), as_u32(p1), as_u32(p2), as_u32(p3)});
  };
  // One chunk as 4 MT / 2 groups of two activation tiles: while a group's 2 PT MFMAs run, the next group's two B fragments
  // are read and a share of the next k-step's A fragments decoded, across the chunk's end too. Chunk j's x sits in LDS
  // buffer j % 2, its weights in slot j % 2. The slot is refilled two chunks ahead when its last k-step has been decoded;
  // before the last group, when every B fragment of the chunk has been read, one barrier makes the next chunk's x
  // visible (the wait leaves the 2 PT newer weight loads in flight) and frees this chunk's buffer for the x two chunks
  // ahead. The count relies on those loads, which are the compiler's own, being there: they are while the chunk they
  // fetch is consumed, and where it is past the range (the last two chunks), the wait is for everything. (Left
  // to itself hipcc waits for every pair of fragment reads right after issuing it.)
  constexpr int GP = MT / 2, DPG = (PT + GP - 1) / GP;      // groups per k-step, decodes per group
  f16x8 a[2][PT], bx[2][2];
  auto chunk = [&](int j, auto slot) __attribute__((always_inline)) {
    constexpr int d = decltype(slot)::value;
    unrolled<4 * GP>([&](auto gi) __attribute__((always_inline)) {   // (a plain loop of this size is not unrolled)
      constexpr int g = decltype(gi)::value, st = g / GP, mp = g % GP, nst = (g + 1) / GP % 4, nmp = (g + 1) % GP;
      constexpr bool last = g + 1 == 4 * GP;
      if constexpr (g == 3 * GP) issue_w(d, cb + j + 2);
      if constexpr (last) {
        if (j + 2 < nsteps) {
          lds_wait_barrier<2 * PT>();
          issue_x(d, cb + j + 2);
        } else {
          lds_wait_barrier<0>();
        }
      }
#pragma unroll
      for (int e = 0; e < 2; ++e)
        bx[(g + 1) & 1][e] =
            *reinterpret_cast<const f16x8*>(smem + (last ? d ^ 1 : d) * kXBuf + 4096 * (2 * nmp + e) + xrd[nst]);
#pragma unroll
      for (int i = DPG * mp; i < DPG * mp + DPG && i < PT; ++i) a[(st + 1) & 1][i] = decode(st == 3 ? d ^ 1 : d, i, (st + 1) & 3);
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int i = 0; i < PT; ++i)
          acc[i][2 * mp + e] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[st & 1][i], bx[g & 1][e], acc[i][2 * mp + e], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);    // 2 LDS reads, then 2 vector instructions to each MFMA
#pragma unroll
      for (int u = 0; u < 2 * PT; ++u) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 2, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  issue_w(0, cb);
  issue_x(0, cb);
  issue_w(1, cb + 1);
  if (nsteps > 1) {
    issue_x(1, cb + 1);
    lds_wait_barrier<2 * PT + XP>();                        // chunk 0 of x has landed
  } else {
    lds_wait_barrier<0>();
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) bx[0][e] = *reinterpret_cast<const f16x8*>(smem + 4096 * e + xrd[0]);
#pragma unroll
  for (int i = 0; i < PT; ++i) a[0][i] = decode(0, i, 0);
  int j0 = 0;
  for (; j0 + 2 <= nsteps; j0 += 2) {
    chunk(j0, std::integral_constant<int, 0>{});
    chunk(j0 + 1, std::integral_constant<int, 1>{});
  }
  if (j0 < nsteps) chunk(j0, std::integral_constant<int, 0>{});
  vm_drain();                                               // no load into LDS is left in flight

  if (S > 1) {
    // fp32 partials of the tile, [split][fragment][thread] 16 bytes each: every store and load is one contiguous KB a wave
    constexpr int kFrag = 16 * kThreads, kPart = PT * MT * kFrag;
    const __amdgpu_buffer_rsrc_t pr =
        make_rsrc(reinterpret_cast<uint8_t*>(part) + (size_t)(tile - full) * S * kPart, (uint32_t)(S * kPart));
#pragma unroll
    for (int i = 0; i < PT; ++i)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) store_partial4(pr, sp * kPart + (i * MT + mt) * kFrag + 16 * tid, acc[i][mt]);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);               // the partials' stores stay before the wait
    __builtin_amdgcn_s_waitcnt(0);                          // every partial acknowledged: visible to all XCDs
    __builtin_amdgcn_s_barrier();
    int& s_last = *reinterpret_cast<int*>(smem);            // (the x buffers are free)
    uint32_t* count = ctr + (tile - full);
    if (tid == 0) {
      const uint32_t prev = __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s_last = prev == (uint32_t)(S - 1);
    }
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_s_barrier();
    __atomic_signal_fence(__ATOMIC_SEQ_CST);               // the partials' loads stay after the count
    if (!s_last) return;
    if (tid == 0) __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the sum in split order; the loads of 8 fragments (all of them in small tiles) go out before the first add
    constexpr int kBatch = PT * MT < 8 ? PT * MT : 8;
#pragma unroll
    for (int f0 = 0; f0 < PT * MT; f0 += kBatch) {
      f32x4 sum[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) sum[u] = f32x4{0.f, 0.f, 0.f, 0.f};
      f32x4 v[kBatch];
#pragma unroll
      for (int u = 0; u < kBatch; ++u) v[u] = load_partial4(pr, (f0 + u) * kFrag + 16 * tid);
      for (int k = 1; k <= S; ++k) {                        // the next split's are requested before this one's are added
        f32x4 nv[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; ++u)
          nv[u] = load_partial4(pr, k < S ? k * kPart + (f0 + u) * kFrag + 16 * tid : kOutOfRange);
#pragma unroll
        for (int u = 0; u < kBatch; ++u) {
          sum[u] += v[u];
          v[u] = nv[u];
        }
      }
#pragma unroll
      for (int u = 0; u < kBatch; ++u) acc[(f0 + u) / MT][(f0 + u) % MT] = sum[u];
    }
  }
  if constexpr (ROPE) {                                     // per tile: the MT column tiles' loads and RoPE, then stores
#pragma unroll
    for (int i = 0; i < PT; ++i) {
      Out4 out[MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) {
        const int m = m0 + 16 * mt + r, n = n0 + 16 * (PT * wave + i) + 4 * q;
        const f32x4 v = acc[i][mt];                         // partner rows 8 + 4 q + v sit 32 lanes on (q + 2)
        const f32x4 up = {shfl_down32(v[0]), shfl_down32(v[1]), shfl_down32(v[2]), shfl_down32(v[3])};
        out[mt] = q < 2 && m < M && n < N ? rope_qkv_out4(epi, m, n, v, up) : Out4{};
      }
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) store_rope4(out[mt]);
    }
    return;
  }
  // The tile's fp16 values through LDS, so that y and the bias / residual move in 16-byte pieces of contiguous rows: a
  // lane holds 4 rows n of one m, and storing those 8 bytes as they are makes every wave-store 16 rows of 32 bytes (at
  // 2048 x 16384 outputs the stores alone took 35 us a round of tiles). Rows are padded by 32 bytes: the 16 rows x 32
  // bytes of a wave's write then meet different banks.
  constexpr int kPitch = 2 * kRows + 32;
  typedef f16 row8 __attribute__((ext_vector_type(8), aligned(2)));   // 8 values of a row, at any 2-byte address
  lds_barrier();                                            // (s_last has been read)
#pragma unroll
  for (int i = 0; i < PT; ++i)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const f32x4 v = acc[i][mt];
      const f16x2 lo = {(f16)v[0], (f16)v[1]}, hi = {(f16)v[2], (f16)v[3]};
      *reinterpret_cast<uint2*>(smem + (16 * mt + r) * kPitch + 32 * (PT * wave + i) + 8 * q) = make_uint2(as_u32(lo), as_u32(hi));
    }
  lds_barrier();
  if (epi.mode == kEpiSiluMul) {                            // 8 outputs from a 16-row tile's 8 gate and 8 up values (all
    constexpr int kPcs = kRows / 16;                        // lanes busy: in the registers' layout half of them hold up)
    const int ny = N / 2;                                   // (N % 16 == 0)
    for (int p = tid; p < 16 * MT * kPcs; p += kThreads) {
      const int row = p / kPcs, m = m0 + row, n = n0 / 2 + 8 * (p % kPcs);
      if (m >= M || n >= ny) continue;
      const u32x4* src = reinterpret_cast<const u32x4*>(smem + row * kPitch + 32 * (p % kPcs));
      const u32x4 gv = src[0], uv = src[1];
      u32x4 o;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const f16x2 g2 = as_f16x2(gv[e]), u2 = as_f16x2(uv[e]);
        o[e] = as_u32(f16x2{silu_mul((float)g2[0], (float)u2[0]), silu_mul((float)g2[1], (float)u2[1])});
      }
      f16* dst = y + (size_t)m * ny + n;
      *reinterpret_cast<row8*>(dst) = __builtin_bit_cast(f16x8, o);
    }
    return;
  }
  // 8 values a piece, at any 2-byte address (global memory takes dwordx4 accesses at those), then the values past the last
  // whole piece of the rows. Single values wherever a piece is not 16-byte aligned, as this kernel stored them before: 333
  // rows of 2048 x 11004 37 us, 32.3 now; 512 of 3584 x 18941 85 -> 77; 2048 of 1024 x 4100 37 -> 26 (a width of 11008
  // 32.3 both ways). The rows' ends inside the loop, with a residual: 40.5 us where they now take 36.
  constexpr int kPcs = kRows / 8;
  const bool aux = epi.mode == kEpiBias || epi.mode == kEpiResidual;
  auto add_at = [&](int m, int n) { return epi.mode == kEpiBias ? epi.aux + n : epi.aux + (size_t)m * N + n; };
  for (int p = tid; p < 16 * MT * kPcs; p += kThreads) {
    const int row = p / kPcs, m = m0 + row, n = n0 + 8 * (p % kPcs);
    if (m >= M || n + 8 > N) continue;
    f16x8 v = *reinterpret_cast<const f16x8*>(smem + row * kPitch + 16 * (p % kPcs));
    if (aux) v += *reinterpret_cast<const row8*>(add_at(m, n));
    *reinterpret_cast<row8*>(y + (size_t)m * N + n) = v;
  }
  const int nw = N & ~7;
  if (nw < N && n0 + kRows > nw)
    for (int p = tid; p < 16 * MT * 8; p += kThreads) {
      const int row = p >> 3, m = m0 + row, n = nw + (p & 7);
      if (m >= M || n >= N) continue;
      const f16 v = *reinterpret_cast<const f16*>(smem + row * kPitch + 2 * (n - n0));
      y[(size_t)m * N + n] = aux ? v + *add_at(m, n) : v;
    }
}

namespace {

template <int MT, int PT>
hipError_t launch_prefill(const GemvArgs& a, const PrefillPlan& p, uint32_t* ctr, float* part) {
  // two x buffers; the output tile of the epilogue takes their place
  constexpr size_t shmem = std::max((size_t)2 * 16 * MT * 256, (size_t)16 * MT * (128 * PT + 32));
  static_assert(shmem <= 65536, "above the default dynamic LDS limit");
  // the RoPE epilogue is its own instantiation: its registers would cost every other epilogue occupancy
  auto kern = a.epi.mode == kEpiRopeQKV ? gemm_prefill<MT, PT, true> : gemm_prefill<MT, PT, false>;
  return launch(kern, dim3(p.items), dim3(256), shmem, a.stream, a.x, a.w, a.s, a.y, a.M, a.N, a.K, a.G, p.S, p.MG, p.full,
                p.items, ctr, part, a.epi);
}

// The tile shapes built, and what a launch of each costs (us): `groups` workgroups share a CU (registers, LDS); `base` for
// a launch; a workgroup takes `alone` per 128-k chunk, or a CU's resident ones `each` per chunk and workgroup when that is
// more; a K split costs `split` and `per_mb` per MB of partials. Fitted to an MI355X sweep (graph-timed, cold weights, 65
// to 2048 rows of 12 Qwen2.5-0.5B .. 7B projections, 1 to 8 splits; the fit's error is 10-15%); the cheapest plan by
// the fitted constants was 2.5% slower than the sweep's best on average and 26% at worst. `alone` of the 64-row shapes was
// raised from the fit's 0.74 and 0.66 afterwards, by the points named here and without taking those two figures again: a
// workgroup that has its CU to itself and walks all of K waits for its weights (0.86 .. 0.9 a chunk), so two splits beat it
// (2048 x 2048 at 512 rows 17.0 -> 14.2, 2048 x 2560 at 300 17.0 -> 14.2, 3584 x 4608 at 333
// 28.1 -> 25.1, 3584 x 3584 at 400 27.8 -> 24.9, 1536 x 2048 at 512 13.0 -> 12.1).
struct PrefillShape {
  int MT, PT, groups;
  float base, alone, each, split, per_mb;
};
constexpr PrefillShape kPrefillShapes[] = {
    {8, 2, 2, 4.8f, 1.20f, 0.93f, 4.4f, 0.30f},             // 128 activation rows x 128 weight rows
    {6, 4, 2, 6.8f, 1.41f, 1.25f, 6.9f, 0.24f},             // 96 x 256
    {4, 2, 4, 4.2f, 0.88f, 0.56f, 2.7f, 0.31f},             // 64 x 128
    {4, 1, 4, 2.5f, 0.88f, 0.385f, 2.0f, 0.38f},            // 64 x 64
};
constexpr int kCUs = 256;

struct PrefillCount {
  long tiles, full, rest;
  int S;
};

// the tiles of a shape, those that fill whole rounds, and the split of the others: at most `S`, within K and the workspace
PrefillCount count_prefill(const PrefillShape& c, int M, int N, int KC, int S, bool all, size_t part_bytes) {
  PrefillCount n;
  n.tiles = (long)((M + 16 * c.MT - 1) / (16 * c.MT)) * ((N + 64 * c.PT - 1) / (64 * c.PT));
  const long slots = (long)kCUs * c.groups;
  n.full = all ? 0 : n.tiles / slots * slots;
  n.rest = n.tiles - n.full;
  n.S = std::min({S, KC, kMaxSplits});
  const size_t tile_bytes = (size_t)16 * c.MT * 64 * c.PT * sizeof(float);   // fp32 partials of a tile
  if (n.rest > 0) n.S = (int)std::min<size_t>((size_t)n.S, part_bytes / (tile_bytes * n.rest));
  if (n.rest == 0 || n.rest > (long)(kCounterBytes / 4)) n.S = 1;   // one arrival counter a tile
  if (n.S <= 1) n.S = 1, n.full = n.tiles, n.rest = 0;
  return n;
}

float prefill_cost(const PrefillShape& c, const PrefillCount& n, int KC) {
  const long slots = (long)kCUs * c.groups;
  auto rounds = [&](long items) {                           // us per chunk of `items` workgroups
    const long last = items % slots;
    return (items / slots) * std::max(c.alone, c.groups * c.each) +
           (last ? std::max(c.alone, ((last + kCUs - 1) / kCUs) * c.each) : 0.f);
  };
  float t = c.base + KC * rounds(n.full);
  if (n.rest > 0) {
    const float mb = (float)n.S * n.rest * (16 * c.MT * 64 * c.PT * 4) * 1e-6f;
    t += KC * rounds(n.rest * n.S) / n.S + c.split + c.per_mb * mb;
  }
  return t;
}

}  // namespace

// Launch shape: the cheapest of the tile shapes and of 1, 2, 3, 4, 6, 8 splits (at least 4 chunks each) of the tiles that
// do not fill a round. The tuning override selects the shape (waves_per_group: 1 or 2 = 64 x 128, 4 or 8 = 128 x 128) and
// the split of all tiles (k_splits).
PrefillPlan plan_gemm_prefill(int M, int N, int K, size_t workspace_bytes) {
  const GemvOverride o = gemv_override();
  const int KC = K / 128;
  const size_t part_bytes = workspace_bytes > kCounterBytes ? workspace_bytes - kCounterBytes : 0;
  PrefillPlan p;
  float best = -1.f;
  for (const PrefillShape& c : kPrefillShapes) {
    if (o.waves > 0 && (c.PT != 2 || c.MT != (o.waves >= 4 ? 8 : 4))) continue;
    for (int S : {1, 2, 3, 4, 6, 8}) {
      if (o.splits > 0 ? S != 1 : S > 1 && KC < 4 * S) continue;
      const PrefillCount n = count_prefill(c, M, N, KC, o.splits > 0 ? o.splits : S, o.splits > 0, part_bytes);
      const float t = prefill_cost(c, n, KC);
      if (best >= 0.f && t >= best) continue;
      best = t;
      p.MT = c.MT;
      p.PT = c.PT;
      p.MG = (M + 16 * c.MT - 1) / (16 * c.MT);
      p.S = n.S;
      p.full = (int)n.full;
      p.items = (int)(n.full + n.rest * n.S);
    }
  }
  return p;
}

hipError_t gemm_prefill_launch(const GemvArgs& a, void* workspace, size_t workspace_bytes) {
  const PrefillPlan p = plan_gemm_prefill(a.M, a.N, a.K, workspace ? workspace_bytes : 0);
  uint32_t* ctr = static_cast<uint32_t*>(workspace);
  float* part = workspace ? reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + kCounterBytes) : nullptr;
  if (p.MT == 8) return launch_prefill<8, 2>(a, p, ctr, part);
  if (p.MT == 6) return launch_prefill<6, 4>(a, p, ctr, part);
  return p.PT == 2 ? launch_prefill<4, 2>(a, p, ctr, part) : launch_prefill<4, 1>(a, p, ctr, part);
}

}  // namespace lowbit
