// Paged decode / prefill attention for gfx950.
//
// A query row is one token (batch * q_len rows).  One workgroup handles one
// (row, KV head, context split); all GQA query heads of the KV head are computed
// together, so each K/V page is read from HBM once.  The host picks the number of
// splits S: 1 whenever rows * kv_heads already fills the GPU (then the workgroup
// writes the final output and nothing goes through global memory), otherwise a
// few splits whose (max, sum, O) partials a small merge kernel combines.
//
// fp16 pools, head_dim 128 (Llama-3 / Qwen2 shapes), 8 wavefronts per workgroup:
//   * the split's context is cut into 32-token blocks dealt round-robin to the
//     wavefronts; a wavefront issues every K and V load of its block up front
//     (8 KiB of K and 8 KiB of V in flight, no branches: tiles past the end are
//     clamped to a valid page and masked);
//   * S = Q K^T on MFMA 16x16x32 f16: A = the group's query heads padded to 16
//     rows, B = a 16-token tile of K read straight from its page (token rows of
//     256 B); fp32 accumulate;
//   * softmax in base 2 (scale*log2(e) folded into the scores): exact within the
//     block, online (running max / rescale) across a wavefront's blocks; the row
//     max over a tile's 16 token lanes is a DPP reduction (no LDS round trips) and
//     the rescale factors are read out of their lane as scalars;
//   * O = P V on VALU: a lane owns 8 contiguous head dims of 4 token rows of each
//     tile (1 KiB contiguous per load instruction); P comes from the score lanes by
//     ds_bpermute shuffles, in fp16 with two heads per dword (l sums the same
//     rounded values); the four token groups are summed once at the end;
//   * the 8 wavefronts merge (max, sum, O) through LDS with log-sum-exp weights.
// Prefill (q_len > 1) on fp16 pools runs attn_prefill_f16_d128 instead: 64 or 128 query
// vectors of a sequence per workgroup over its blocks, both products on MFMA.
// fp32 pools and other head sizes (tiny-model parity path) use a VALU kernel over
// 128-token chunks: a context of one chunk is written out directly, more chunks leave
// partials for the same merge kernel.
//
// Reference semantics: cacheir/backends/triton_kernels.py:174-217 (paged gather
// pool[page_table[b, t // P], kvh, t % P], GQA kvh = h // (Hq/Hkv), positions
// t < seq_len) and cacheir/runtime/cpu.py:342-377 (softmax(q.k * scale) v,
// prefill causal mask).
#include "common.hpp"

#include <float.h>
#include <math.h>

#include <atomic>
#include <mutex>

namespace cir {
namespace {

template <int CTRL>
__device__ __forceinline__ float dpp_mov(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, false));
}
// Max over the 16 lanes of each DPP row (lanes 16r .. 16r+15): swap neighbours, swap
// pairs, mirror the half rows, mirror the rows; every lane ends with its row's max.
__device__ __forceinline__ float row16_max(float v) {
  v = fmaxf(v, dpp_mov<0xB1>(v));   // quad_perm [1,0,3,2]
  v = fmaxf(v, dpp_mov<0x4E>(v));   // quad_perm [2,3,0,1]
  v = fmaxf(v, dpp_mov<0x141>(v));  // row_half_mirror
  v = fmaxf(v, dpp_mov<0x140>(v));  // row_mirror
  return v;
}
// The same pattern as a sum: lane 16r of each row ends with the row's total (the
// other lanes too, summed in another order).
__device__ __forceinline__ float row16_sum(float v) {
  v += dpp_mov<0xB1>(v);
  v += dpp_mov<0x4E>(v);
  v += dpp_mov<0x141>(v);
  v += dpp_mov<0x140>(v);
  return v;
}
// Sums over the four rows of four values at once, by gfx950's lane-swap instructions
// (no LDS): v_permlane16_swap(a, b) leaves rows (a0, b0, a2, b2) and (a1, b1, a3, b3),
// v_permlane32_swap(x, y) leaves (x0, x1, y0, y1) and (x2, x3, y2, y3).  Row k of the
// result holds the total of v[k], summed (r0 + r1) + (r2 + r3) in every lane.
__device__ __forceinline__ float swap_sum16(float a, float b) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b),
                                                  false, false);
  const uint32_t r0 = r[0], r1 = r[1];  // (bit_cast of a vector element lvalue reads element 0)
  return __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ float rows_sum4(const float (&v)[4]) {
  const float ab = swap_sum16(v[0], v[1]), cd = swap_sum16(v[2], v[3]);
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, ab), __builtin_bit_cast(uint32_t, cd),
                                                  false, false);
  const uint32_t r0 = r[0], r1 = r[1];
  return __builtin_bit_cast(float, r0) + __builtin_bit_cast(float, r1);
}

// 8 wavefronts of 32-token steps measured best on MI355X at config 4 (batch 32,
// 2048 tokens), against 64-token steps, 16 wavefronts of 16 tokens and a
// double-buffered pipeline.  A long streaming read peaks at ~7.0 TB/s on this part;
// a loads-only copy of this kernel's access pattern (same grid, pages and per-lane
// addresses) takes 47.4 us at config 4 (5.7 TB/s), and the kernel 50.0 us.
constexpr int kTiles = 2;             // 16-token MFMA tiles per wavefront step
constexpr int kBlock = 16 * kTiles;   // tokens per wavefront step
constexpr int kWaves = 8;             // wavefronts per workgroup (fp16 path)
constexpr int kChunk = 128;  // tokens per partial in the generic path
// Page-table entries a workgroup keeps in LDS (2 KiB at 8 wavefronts): one per thread, since every thread fills
// one entry (a split whose pages exceed the thread count reads the table directly); the row sort of the
// longest-first dispatch also ranks one row per thread in this array.
constexpr int kPtCache = 64 * kWaves;
constexpr int kMinSplitTokens = 256;
constexpr float kLog2e = 1.4426950408889634f;

// Tokens visible to query row `row`, clamped to what the page table can address.
__device__ __forceinline__ int visible_len(const int32_t* lens, int row, int q_len, int max_ctx) {
  const int b = row / q_len;
  const int s = row - b * q_len;
  return min(lens[b] - q_len + s + 1, max_ctx);
}

// ----------------------------------------------------------------------------
// fp16 pools, head_dim 128.  G = query heads per KV head (1..8).
// Fused decode input (optional): the QKV projection's fp32 split-k partials
// [splits][batch][(Hq + 2 Hkv) D] instead of a finished q.  The workgroup then sums
// its heads' partials, applies RoPE to q and k, appends the new k and v to their page
// and keeps q in LDS -- the work of the QKV epilogue kernel, in the same order and
// precision, for one (row, KV head) at a time.
struct QkvIn {
  const float* part;        // null: q is read from `q`
  int splits;
  const float* inv_freq;    // [D/2]
  const int32_t* positions; // [batch]: position of the new token
};

// Splits of the QKV partials a fused workgroup loads before its first K/V block;
// more splits are loaded when summed.
constexpr int kSumUnroll = 8;

// FUSED: q comes from the QKV partials in `qkv` (decode, q_len 1), else from `q`.
template <int G, bool FUSED>
__global__ __launch_bounds__(64 * kWaves) void attn_f16_d128(
    const f16* __restrict__ q, f16* __restrict__ kp, f16* __restrict__ vp,
    const int32_t* __restrict__ pt, const int32_t* __restrict__ lens, f16* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, int q_len, int Hq, int Hkv, int P, int max_pages,
    int S, float scale_log2, int sort_rows, QkvIn qkv) {
  constexpr int D = 128;
  __shared__ float sm_m[kWaves][16];
  __shared__ float sm_l[kWaves][16];
  __shared__ float sm_o[kWaves][G][D];
  __shared__ __align__(16) f16 sm_q[G][D];
  __shared__ __align__(16) f16 sm_kn[D];  // fused: the new token's k and v
  __shared__ __align__(16) f16 sm_vn[D];
  __shared__ int sm_pt[kPtCache];

  const int split = blockIdx.x, kvh = blockIdx.y;
  // Rows in decreasing order of context (sort_rows: decode, rows <= one per thread, more
  // workgroups than CUs): workgroups are dispatched in blockIdx order as CUs free up,
  // so the longest rows start first and the short ones fill in behind them (longest
  // processing time first) instead of a long row starting last and running alone.
  // Row t's rank counts the rows longer than it, ties broken by index.
  int row = blockIdx.z;
  if (sort_rows) {
    const int n = gridDim.z, t = threadIdx.x;
    const int lt = t < n ? lens[t] : 0;
    sm_pt[t] = lt;  // (the page-table cache is filled later)
    __syncthreads();
    if (t < n) {
      int rank = 0;
      for (int j = 0; j < n; ++j) {
        const int lj = sm_pt[j];
        rank += (lj > lt || (lj == lt && j < t)) ? 1 : 0;
      }
      if (rank == (int)blockIdx.z) sm_m[0][0] = __builtin_bit_cast(float, t);
    }
    __syncthreads();
    row = __builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, sm_m[0][0]));
    __syncthreads();  // sm_pt and sm_m are written again below
  }
  // readfirstlane: the wavefront index is uniform, so block indices and page-table
  // lookups stay scalar (s_load, their own counter) instead of vector loads that
  // would retire in order behind the K/V loads in flight.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int li = lane & 15;  // score column (token in tile) / Q row (head in group)
  const int lg = lane >> 4;  // k-group of the MFMA operands; token group for P V
  const int L = visible_len(lens, row, q_len, max_pages * P);
  const int nblk = L > 0 ? (L + kBlock - 1) / kBlock : 0;
  const int per = (nblk + S - 1) / S;
  const int b0 = split * per, b1 = min(nblk, b0 + per);
  const int b = row / q_len;
  const int32_t* ptrow = pt + (size_t)b * max_pages;

  // One block of K/V operands (kTiles 16-token tiles) for one wavefront.
  struct Blk {
    f16x8 k[kTiles][4], v[kTiles][4];
  };
  // Issue every K load, then every V load, of block `blk` (K first: the scores need
  // only K, so they start while V is still arriving).  Tiles past the end re-read
  // the block's first tile (masked in the scores).
  // This split's page-table entries, cached in LDS when they fit (filled before the
  // first workgroup barrier; until then lookups read the table directly).
  const int pg0 = (b0 * kBlock) / P;
  const int pg1 = min(max_pages, (b1 * kBlock + P - 1) / P);
  const bool pt_cached = pg1 - pg0 <= kPtCache;
  bool pt_ready = false;
  auto page_of = [&](int t) __attribute__((always_inline)) {
    const int pi = t / P;
    return (pt_ready && pt_cached) ? __builtin_amdgcn_readfirstlane(sm_pt[pi - pg0]) : ptrow[pi];
  };
  auto page_bases = [&](size_t (&base)[kTiles], int blk) __attribute__((always_inline)) {
    const int tb = blk * kBlock;
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      const int tj = tb + 16 * j;
      const int tv = tj < L ? tj : tb;
      const int page = page_of(tv);
      base[j] = (((size_t)page * Hkv + kvh) * P + (tv % P)) * D;
    }
  };
  auto load_k = [&](Blk& o, int blk) __attribute__((always_inline)) {
    size_t base[kTiles];
    page_bases(base, blk);
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      const f16* krow = kp + base[j] + (size_t)li * D + 8 * lg;
#pragma unroll
      for (int s = 0; s < 4; ++s) o.k[j][s] = *reinterpret_cast<const f16x8*>(krow + 32 * s);
    }
  };
  auto load_v = [&](Blk& o, int blk) __attribute__((always_inline)) {
    size_t base[kTiles];
    page_bases(base, blk);
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      const f16* vrow = vp + base[j] + 8 * li;
#pragma unroll
      for (int u = 0; u < 4; ++u) o.v[j][u] = *reinterpret_cast<const f16x8*>(vrow + (size_t)(4 * u + lg) * D);
    }
  };
  auto load_block = [&](Blk& o, int blk) __attribute__((always_inline)) {
    load_k(o, blk);
    load_v(o, blk);
  };
  // Issue order: load counters retire in order, so waiting for one load waits for every
  // load issued before it.  q (or the fused prologue's partials) and the page-table
  // entries for the LDS cache go out first, the first K/V block after them, and in a
  // workgroup with blocks every thread issues the same loads (indices clamped, results
  // unused where out of range), so the compiler's waits before the LDS fill and the
  // prologue's arithmetic count the block's loads out instead of waiting for them.
  //
  // Q as the MFMA A operand: row li = head kvh*G + li (zero rows past G); element e
  // of step s is head dim 32*s + 8*lg + e, the same mapping the K loads use.
  f16x8 qa[4];
  if constexpr (!FUSED) {
    const f16* qrow = q + ((size_t)row * Hq + (size_t)kvh * G + (li < G ? li : 0)) * D + 8 * lg;
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const f16x8 v = *reinterpret_cast<const f16x8*>(qrow + 32 * s);
      qa[s] = (li < G) ? v : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }

  // Fused decode input: q, k, v of this row and KV head.  Work items are column pairs:
  // RoPE pair i of q head hh (hh < G) or of k (hh == G), then pairs of v (hh == G + 1).
  // The split whose blocks hold the new token (the writer) also computes its k and v:
  // they go to LDS, the wavefront whose block holds the token patches them into its
  // registers, and the writer appends them to the pool at the very end (a store
  // completes after loads issued later and would hold up every wait behind it), so
  // no ordering between the append and any load of that page line is needed.  The
  // first kSumUnroll splits of an item are loaded up front; more when it is summed.
  constexpr int kHalf = D / 2;
  constexpr int kItems = ((G + 2) * kHalf + 64 * kWaves - 1) / (64 * kWaves);  // per thread
  const int pos = FUSED ? qkv.positions[b] : 0;
  const bool writer = FUSED && split == min(S - 1, (pos / kBlock) / max(per, 1));
  const int items = writer ? (G + 2) * kHalf : G * kHalf;
  const int N = (Hq + 2 * Hkv) * D;
  const size_t plane = (size_t)gridDim.z * N;
  const float* prow = FUSED ? qkv.part + (size_t)row * N : nullptr;
  auto item_col = [&](int it) __attribute__((always_inline)) -> size_t {  // first column of item it
    const int hh = it / kHalf, i = it - hh * kHalf;
    return (hh < G ? ((size_t)kvh * G + hh) * D : (size_t)(Hq + (hh - G) * Hkv) * D + (size_t)kvh * D) + 2 * i;
  };
  float xa[kItems][kSumUnroll], xb[kItems][kSumUnroll], fr[kItems];
  if constexpr (FUSED) {
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
      const int it = min((int)threadIdx.x + k * 64 * kWaves, items - 1);
      const float* p = prow + item_col(it);
#pragma unroll
      for (int s = 0; s < kSumUnroll; ++s) {
        const float* ps = p + (size_t)(s < qkv.splits ? s : 0) * plane;
        xa[k][s] = ps[0];
        xb[k][s] = ps[1];
      }
      fr[k] = qkv.inv_freq[it % kHalf];
    }
  }
  // Sums each item's partials in split order (bitwise as the QKV epilogue kernel),
  // applies RoPE and puts q (and the writer's k and v) in LDS.
  auto prologue = [&]() __attribute__((always_inline)) {
    auto sum = [&](const float (&t)[kSumUnroll], size_t col) __attribute__((always_inline)) {
      float v = t[0];
#pragma unroll
      for (int s = 1; s < kSumUnroll; ++s)
        if (s < qkv.splits) v += t[s];
      for (int s = kSumUnroll; s < qkv.splits; ++s) v += prow[(size_t)s * plane + col];
      return v;
    };
#pragma unroll
    for (int k = 0; k < kItems; ++k) {
      const int it = threadIdx.x + k * 64 * kWaves;
      if (it >= items) continue;
      const int hh = it / kHalf, i = it - hh * kHalf;
      const size_t col = item_col(it);
      const float x0 = sum(xa[k], col), x1 = sum(xb[k], col + 1);
      f16x2 y;
      if (hh <= G) {  // q or k: RoPE
        float sn, cs;
        sincosf((float)pos * fr[k], &sn, &cs);
        // The QKV epilogue kernel's operations: each FMA written out, rounded to fp32 before the fp16 conversion.
        y = f16x2{static_cast<f16>(as_f32_value(fmaf(x0, cs, -(x1 * sn)))),
                  static_cast<f16>(as_f32_value(fmaf(x0, sn, x1 * cs)))};
      } else {
        y = f16x2{static_cast<f16>(x0), static_cast<f16>(x1)};
      }
      f16* dst = hh < G ? &sm_q[hh][2 * i] : (hh == G ? &sm_kn[2 * i] : &sm_vn[2 * i]);
      *reinterpret_cast<f16x2*>(dst) = y;
    }
  };

  // The first block's K/V do not depend on q: issue them before the workgroup barrier
  // and the fused prologue's arithmetic.  A wavefront without a block of its own loads
  // block b0 and drops it.
  Blk A;
  int blk = b0 + wave;
  if (b0 < b1) {  // uniform: pg0 .. pg1 - 1 and block b0 exist
    const int ptv = ptrow[pg0 + min((int)threadIdx.x, pg1 - pg0 - 1)];
    load_block(A, blk < b1 ? blk : b0);
    // Every thread writes (entries past the split's pages are never read): a store under
    // a condition would let the compiler sink the load below the block's loads.
    sm_pt[threadIdx.x] = ptv;
    if constexpr (FUSED) prologue();
  } else if (writer) {
    prologue();
  }
  if constexpr (FUSED) {
    __syncthreads();  // publishes q, the new k and v and the page-table cache
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const f16x8 v = *reinterpret_cast<const f16x8*>(&sm_q[li < G ? li : 0][8 * lg + 32 * s]);
      qa[s] = (li < G) ? v : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  } else if (pt_cached) {
    __syncthreads();  // publishes the page-table cache
  }
  pt_ready = true;

  float m[4], lsum[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    m[r] = -INFINITY;
    lsum[r] = 0.f;
  }
  float acc[G][8];
#pragma unroll
  for (int h = 0; h < G; ++h)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[h][e] = 0.f;

  // Scores of block `blk`: sc[j][r] = S[head 4*lg + r][token tb + 16*j + li] (log2 units).
  auto scores = [&](const Blk& o, int blk, f32x4 (&sc)[kTiles]) __attribute__((always_inline)) {
    const int tb = blk * kBlock;
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      f32x4 c = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f32_16x16x32_f16(qa[s], o.k[j][s], c, 0, 0, 0);
      const bool valid = tb + 16 * j + li < L;
#pragma unroll
      for (int r = 0; r < 4; ++r) sc[j][r] = valid ? c[r] * scale_log2 : -INFINITY;
    }
  };
  // Online softmax update with the block's scores, then O += P V.
  auto softmax_pv = [&](const Blk& o, f32x4 (&sc)[kTiles]) __attribute__((always_inline)) {
    float alpha[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float bm = sc[0][r];
#pragma unroll
      for (int j = 1; j < kTiles; ++j) bm = fmaxf(bm, sc[j][r]);
      bm = row16_max(bm);
      const float mn = fmaxf(m[r], bm);  // finite: token tb is always visible
      // hardware exp2 (the library exp2f adds range steps that only matter below 2^-126, where p rounds to 0 in fp16):
      // config-4 attention 48.6 -> 47.8 us, config 5 203.7 -> 199.4 (two alternated bench runs on one box)
      alpha[r] = __builtin_amdgcn_exp2f(m[r] - mn);
      float ps = 0.f;
#pragma unroll
      for (int j = 0; j < kTiles; ++j) {
        // P V takes p in fp16 (two heads per shuffled dword); l sums the same rounded p.
        const float p = static_cast<float>(static_cast<f16>(__builtin_amdgcn_exp2f(sc[j][r] - mn)));
        sc[j][r] = p;
        ps += p;
      }
      lsum[r] = lsum[r] * alpha[r] + ps;
      m[r] = mn;
    }
    // fp16 p of heads (4g, 4g+1) and (4g+2, 4g+3), g = lane / 16, packed for the shuffles.
    uint32_t pk[kTiles][2];
#pragma unroll
    for (int j = 0; j < kTiles; ++j)
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const f16x2 two = {static_cast<f16>(sc[j][2 * q]), static_cast<f16>(sc[j][2 * q + 1])};
        pk[j][q] = __builtin_bit_cast(uint32_t, two);
      }
    // Rescale O, then O += P V.  Head h's alpha / p live in lanes 16*(h/4).., register h%4.
#pragma unroll
    for (int h = 0; h < G; ++h) {
      const float a = __builtin_bit_cast(
          float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, alpha[h & 3]), 16 * (h >> 2)));  // uniform
#pragma unroll
      for (int e = 0; e < 8; ++e) acc[h][e] *= a;
    }
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int tok = 4 * u + lg;
        float vf[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) vf[e] = static_cast<float>(o.v[j][u][e]);
#pragma unroll
        for (int h2 = 0; h2 < (G + 1) / 2; ++h2) {
          const uint32_t pp = static_cast<uint32_t>(__shfl(static_cast<int>(pk[j][h2 & 1]), tok + 16 * (h2 >> 1), 64));
          const f16x2 p2 = __builtin_bit_cast(f16x2, pp);
          const float p0 = static_cast<float>(p2.x), p1 = static_cast<float>(p2.y);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[2 * h2][e] = fmaf(p0, vf[e], acc[2 * h2][e]);
          if (2 * h2 + 1 < G) {
#pragma unroll
            for (int e = 0; e < 8; ++e) acc[2 * h2 + 1][e] = fmaf(p1, vf[e], acc[2 * h2 + 1][e]);
          }
        }
      }
    }
  };

  // Register patch of the new token (fused): every tile whose rows include it -- its
  // own and any past-the-end tile re-reading the block's first tile -- takes the k row
  // (lanes li == row) and the v row (lanes lg == row % 4, element row / 4).  Selects,
  // not conditional writes: registers take no runtime index.
  auto patch_k = [&](Blk& o, int blk) __attribute__((always_inline)) {
    const int tb = blk * kBlock;
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      const int r = pos - ((tb + 16 * j < L) ? tb + 16 * j : tb);
      const bool hit = r >= 0 && r < 16 && li == r;
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        const f16x8 n = *reinterpret_cast<const f16x8*>(&sm_kn[32 * s + 8 * lg]);
        o.k[j][s] = hit ? n : o.k[j][s];
      }
    }
  };
  auto patch_v = [&](Blk& o, int blk) __attribute__((always_inline)) {
    const int tb = blk * kBlock;
#pragma unroll
    for (int j = 0; j < kTiles; ++j) {
      const int r = pos - ((tb + 16 * j < L) ? tb + 16 * j : tb);
      const bool hit = r >= 0 && r < 16 && lg == (r & 3);
      const f16x8 n = *reinterpret_cast<const f16x8*>(&sm_vn[8 * li]);
#pragma unroll
      for (int u = 0; u < 4; ++u) o.v[j][u] = (hit && u == (r >> 2)) ? n : o.v[j][u];
    }
  };

  // Rotating pipeline: the next block's K is loaded into the K registers as soon as
  // this block's scores have read them, and its V once P V has read this block's V,
  // so every wavefront keeps loads in flight while it computes.  The last block is
  // peeled off, which keeps the steady-state loads unconditional (load counters
  // retire in order; a conditional load would make every wait a full drain).
  {
    const int nb = blk < b1 ? (b1 - blk + kWaves - 1) / kWaves : 0;
    if (nb > 0) {
      // The block holding a fused call's new token (its wavefront in the writer split):
      // its k and v rows are patched into the registers.
      const int blk_new = pos / kBlock;
      const int patch_blk = (writer && blk_new >= b0 && blk_new < b1 && (blk_new - b0) % kWaves == wave) ? blk_new : -1;
      f32x4 sc[kTiles];
      for (int t = 0; t + 1 < nb; ++t, blk += kWaves) {
        if (blk == patch_blk) patch_k(A, blk);
        scores(A, blk, sc);
        load_k(A, blk + kWaves);
        __builtin_amdgcn_sched_barrier(0);
        if (blk == patch_blk) patch_v(A, blk);
        softmax_pv(A, sc);
        load_v(A, blk + kWaves);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (blk == patch_blk) {
        patch_k(A, blk);
        patch_v(A, blk);
      }
      scores(A, blk, sc);
      softmax_pv(A, sc);
    }
  }

  // Wavefront totals: O over the 4 token groups (row k of each 4-value sum holds
  // acc[h][4 * half + k], so every lane writes one), l over the 16 lanes of a row.
#pragma unroll
  for (int h = 0; h < G; ++h)
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const float v[4] = {acc[h][4 * half], acc[h][4 * half + 1], acc[h][4 * half + 2], acc[h][4 * half + 3]};
      sm_o[wave][h][8 * li + 4 * half + lg] = rows_sum4(v);
    }
#pragma unroll
  for (int r = 0; r < 4; ++r) lsum[r] = row16_sum(lsum[r]);

  if (li == 0) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      sm_m[wave][4 * lg + r] = m[r];
      sm_l[wave][4 * lg + r] = lsum[r];
    }
  }
  __syncthreads();

  // Merge the wavefronts: one thread per (head, dim).
  for (int idx = threadIdx.x; idx < G * D; idx += 64 * kWaves) {
    const int h = idx / D, d = idx - h * D;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) M = fmaxf(M, sm_m[w][h]);
    float den = 0.f, o = 0.f;
    if (M != -INFINITY) {
#pragma unroll
      for (int w = 0; w < kWaves; ++w) {
        const float f = exp2f(sm_m[w][h] - M);
        den = fmaf(sm_l[w][h], f, den);
        o = fmaf(sm_o[w][h][d], f, o);
      }
    }
    const int head = kvh * G + h;
    if (S == 1) {
      out[((size_t)row * Hq + head) * D + d] = static_cast<f16>(den > 0.f ? o / den : 0.f);
    } else {
      part_o[(((size_t)row * Hq + head) * S + split) * D + d] = o;
      if (d == 0) {
        float* ml = part_ml + (((size_t)row * Hq + head) * S + split) * 2;
        ml[0] = M;
        ml[1] = den;
      }
    }
  }
  if (writer && (int)threadIdx.x < kHalf) {  // the KV append (fused): k and v pair t, whole rows
    const int page_idx = pos / P;
    const int slot = page_idx < max_pages ? ptrow[page_idx] : -1;
    if (slot >= 0) {
      const size_t at = (((size_t)slot * Hkv + kvh) * P + (pos - page_idx * P)) * D + 2 * threadIdx.x;
      *reinterpret_cast<uint32_t*>(kp + at) = *reinterpret_cast<const uint32_t*>(&sm_kn[2 * threadIdx.x]);
      *reinterpret_cast<uint32_t*>(vp + at) = *reinterpret_cast<const uint32_t*>(&sm_vn[2 * threadIdx.x]);
    }
  }
}

// ----------------------------------------------------------------------------
// Prefill (q_len > 1), fp16 pools, head_dim 128, G <= 8.  The query vectors of one
// sequence and KV head (vector v = t * G + g over its q_len new tokens) form 32-vector
// tiles, one per wavefront.  A workgroup of VW * CW wavefronts holds VW tiles; its CW
// groups take turns of NB 32-token blocks of the context, so a stage of NB * CW blocks
// feeds all of them, and merge (max, sum, O) through LDS at the end.
//   * Staging: K and V rows go from their pages to LDS by DMA (16 bytes a lane, no
//     registers), one stage ahead, one barrier per stage.  Each stage has an array of
//     its own, so the compiler does not make the reads of one wait for the DMA into
//     another.  16-byte chunk c of a K row r sits in slot c ^ (r % 16), of a V row in slot
//     c ^ (4 (r % 4) + r / 4 % 4): the reads below then cover all banks evenly.
//   * S^T = K Q^T on MFMA 32x32x16 f16: lane q + 32h ends with S[q][8j + 4h + e].
//   * O^T = V^T P^T: the B operand is P as the lanes hold it (8 tokens 8j + 4h ..), and
//     V^T's A operand takes the same token order by gfx950's transposing LDS read
//     (ds_read_b64_tr_b16: 16 lanes read 4 token rows of 16 dims and each gets 4 tokens of
//     one dim), so neither product exchanges lanes and the softmax rescale is per lane.
// Causal mask per query vector, applied only to blocks a wavefront's first query does not
// see whole; softmax in base 2 with p rounded to fp16 for P V and l summing the rounded p;
// the rescale is skipped when no running max moved; a wavefront skips the blocks past its
// last token.  The longest tiles are dispatched first, so a causal grid of several rounds
// balances itself.
//
// What bounds it: 32 vectors x 32 tokens cost a wavefront 512 matrix cycles, ~450 VALU
// cycles of softmax and 16 KiB of LDS reads (128 of the CU's LDS cycles), and the time is
// what these do not overlap: by counters (2 x 509 tokens after 3500) the matrix cores are
// busy 27% of the cycles, VALU 38%, both at once 12%, so half of them nothing issues, with
// two wavefronts per SIMD between the barriers and 224 workgroups on 256 CUs; no LDS
// conflicts, K/V read from HBM once.  The earlier kernel (16 vectors per wavefront: twice the LDS bytes per product;
// V transposed by 2-byte LDS writes) was bound by LDS.  Measured (us, before -> now): 2 x
// 509 tokens after 3500 (28/4 heads) 178 -> 84, 2048 after 6000 (32/8) 625 -> 271 (870
// TFLOP/s), a 2048-token prompt 102 -> 57, 8 x 512 tokens 54 -> 41, 10 tokens after 5000
// (28/4) 209 -> 19.  NB = 2 (one max, one rescale and one barrier per 64 tokens of a
// wavefront) against 1: 2048 after 6000 280 -> 251.
constexpr int kPfVec = 32;  // query vectors per wavefront (one 32-wide MFMA tile)

typedef float f32x16 __attribute__((ext_vector_type(16)));

// Transposing LDS read: see the kernel's header.
__device__ __forceinline__ f16x4 lds_read_tr(const uint8_t* p) {
  typedef __fp16 h4 __attribute__((ext_vector_type(4)));
  const h4 v = __builtin_amdgcn_ds_read_tr16_b64_v4f16((__attribute__((address_space(3))) h4*)(p));
  return __builtin_bit_cast(f16x4, v);
}
// This wavefront's DMA has landed, then every wavefront's.  The wait is the builtin, not asm: the compiler counts it,
// and then puts no wait of its own (which would cover the next stage's DMA too) before the reads of the landed stage.
__device__ __forceinline__ void dma_wait_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0x70);  // vmcnt(0), lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <int VW, int CW, int NB>
__global__ __launch_bounds__(64 * VW * CW, 2) void attn_prefill_f16_d128(
    const f16* __restrict__ q, const f16* __restrict__ kp, const f16* __restrict__ vp,
    const int32_t* __restrict__ pt, const int32_t* __restrict__ lens, f16* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml, int q_len, int Hq, int Hkv, int P, int max_pages, int S,
    float scale_log2) {
  constexpr int D = 128;
  constexpr int W = VW * CW;
  constexpr int kTok = kBlock * NB * CW;   // tokens per stage
  constexpr int kHalf = kTok * D * 2;      // bytes of K (then V) in a stage
  constexpr int kRows = kTok / W; // rows of K and of V a wavefront brings in (within one page: kRows | 16)
  static_assert(kRows == 8 || kRows == 16, "a wavefront's rows lie in one page");
  __shared__ __align__(16) uint8_t st0[2 * kHalf];
  __shared__ __align__(16) uint8_t st1[2 * kHalf];
  __shared__ float sm_ml[CW > 1 ? CW : 1][VW][2][64];
  const int kvh = blockIdx.x % Hkv, b = blockIdx.x / Hkv;
  const int tile = gridDim.y - 1 - blockIdx.y;  // the longest contexts first
  const int split = blockIdx.z;
  const int G = Hq / Hkv;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int vw = wave % VW, cw = wave / VW;
  const int l32 = lane & 31, h = lane >> 5;
  const int nvec = q_len * G;
  const int L = lens[b];
  const int Lc = min(L, max_pages * P);  // keys the page table can address
  const int past = L - q_len;            // context before the new tokens
  const int32_t* ptrow = pt + (size_t)b * max_pages;
  // Last key position query vector v sees (negative: none, its output is zero).
  auto pos_of = [&](int v) __attribute__((always_inline)) { return min(past + v / G, Lc - 1); };
  const int tv0 = tile * kPfVec * VW;                   // the workgroup's first vector
  const int tv1 = min(nvec, tv0 + kPfVec * VW) - 1;     // and its last
  const int nblk = pos_of(tv1) >= 0 ? pos_of(tv1) / kBlock + 1 : 0;  // blocks the last token sees
  const int nst = (nblk + NB * CW - 1) / (NB * CW), per = (nst + S - 1) / S;
  const int s0 = min(nst, split * per), s1 = min(nst, s0 + per);     // this split's stages
  const int v0 = tv0 + kPfVec * vw;                     // this wavefront's first vector
  const int wlast = min(nvec - 1, v0 + kPfVec - 1);
  const int wblk = (v0 < nvec && pos_of(wlast) >= 0) ? pos_of(wlast) / kBlock + 1 : 0;  // uniform

  // DMA of stage st: this wavefront's rows kRows * wave .. of the stage, 4 rows per instruction (lane / 16 = row,
  // lane % 16 = LDS slot).  Rows past the context re-read its last token (masked; p = 0 meets finite values).
  const int drow = kRows * wave + (lane >> 4), dslot = lane & 15;
  int page = 0, prow = 0;  // the page of its rows of the stage to issue next, and the page's first position
  auto fetch_page = [&](int st) __attribute__((always_inline)) {
    const int i = min(st * kTok + kRows * wave, Lc - 1) / P;
    page = ptrow[i];
    prow = i * P;
  };
  auto issue = [&](uint8_t* buf, int st) __attribute__((always_inline)) {
    const size_t base = ((size_t)page * Hkv + kvh) * P * D;
    const rsrc_t rk = make_rsrc(kp + base, (uint32_t)P * 2 * D), rv = make_rsrc(vp + base, (uint32_t)P * 2 * D);
    const int row0 = st * kTok - prow, last = Lc - 1 - prow;
#pragma unroll
    for (int u = 0; u < kRows / 4; ++u) {
      const int r = drow + 4 * u;
      const uint32_t at = (uint32_t)min(row0 + r, last) * 2 * D;
      buf16_to_lds(rk, buf + (kRows * wave + 4 * u) * 2 * D, at + 16 * (dslot ^ (r & 15)), 0);
      buf16_to_lds(rv, buf + kHalf + (kRows * wave + 4 * u) * 2 * D,
                   at + 16 * (dslot ^ (((r & 3) << 2) | ((r >> 2) & 3))), 0);
    }
  };

  // Q^T as the B operand (zero past the last vector); a negative scale is folded into q's sign, so the running max
  // can be taken before scaling.
  f16x8 qb[8];
  const int vq = v0 + l32;
  const bool live = vq < nvec;
  const int qpos = pos_of(live ? vq : nvec - 1);
  const int qmin = pos_of(min(v0, nvec - 1));  // the wavefront's first query position (the least)
  const float sc = fabsf(scale_log2);
  {
    const int vv = live ? vq : 0;
    const int t = vv / G, g = vv - t * G;
    const f16* qrow = q + (((size_t)b * q_len + t) * Hq + (size_t)kvh * G + g) * D + 8 * h;
    const uint32_t flip = scale_log2 < 0.f ? 0x80008000u : 0u;
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const u32x4 x = *reinterpret_cast<const u32x4*>(qrow + 16 * s) ^ flip;
      qb[s] = live ? __builtin_bit_cast(f16x8, x) : f16x8{0, 0, 0, 0, 0, 0, 0, 0};
    }
  }

  const float one = as_f32_value(1.f);
  bool huge = false;             // uniform: some query's |m| is 2^24 or more
  float m = -INFINITY, l = 0.f;  // query l32: running max (both lanes of the query), this lane's share of the sum
  f32x16 acc[D / 32];            // O[query l32][32 dt + 8 j + 4 h + e], element 4 j + e
#pragma unroll
  for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[dt][r] = 0.f;

  // Byte offsets of this lane's reads inside a stage.
  const int krow = (kBlock * NB * cw + l32) * 2 * D, kx = 16 * (h ^ (l32 & 15));
  const int ti = lane & 15, sub = (lane >> 4) & 1;
  int vo[2];
#pragma unroll
  for (int a = 0; a < 2; ++a)
    vo[a] = kHalf + (kBlock * NB * cw + 8 * a + 4 * h + (ti >> 2)) * 2 * D +
            16 * ((2 * sub + ((ti & 3) >> 1)) ^ (2 * a + h)) + 8 * (ti & 1);

  // This wavefront's NB blocks of a stage, from block `blk` on.
  auto blocks = [&](const uint8_t* buf, int blk) __attribute__((always_inline)) {
    f32x16 c[NB];
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      f16x8 ka[8];
#pragma unroll
      for (int s = 0; s < 8; ++s)
        ka[s] = *reinterpret_cast<const f16x8*>(buf + krow + j * kBlock * 2 * D + (kx ^ (32 * s)));
#pragma unroll
      for (int r = 0; r < 16; ++r) c[j][r] = 0.f;
#pragma unroll
      for (int s = 0; s < 8; ++s) c[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ka[s], qb[s], c[j], 0, 0, 0);
    }
    f16x8 va[NB][D / 32][2];
    auto load_v = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          const uint8_t* pv = buf + 64 * (dt ^ (ti >> 2)) + (2 * j + ks) * 16 * 2 * D;
          const f16x4 lo = lds_read_tr(pv + vo[0]), hi = lds_read_tr(pv + vo[1]);
          va[j][dt][ks] = f16x8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
    };
    load_v(0);  // V^T of the first block goes to registers before the softmax, which hides the LDS latency
    __builtin_amdgcn_sched_barrier(0);
    if ((blk + NB) * kBlock - 1 > qmin) {  // uniform: some query of the wavefront does not see all the blocks
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          c[j][r] = ((blk + j) * kBlock + 8 * (r >> 2) + 4 * h + (r & 3) <= qpos) ? c[j][r] : -INFINITY;
    }
    float mx = c[0][0];
#pragma unroll
    for (int r = 1; r < 16 * NB; ++r) mx = fmaxf(mx, c[r >> 4][r & 15]);
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64)) * sc;
    // (m follows the running max exactly, so the largest p is exactly one: letting it lag by up to 2^8 to save most
    // rescales took 5% off the time and added 3-5% to the error.)
    // A query that has seen no key yet keeps m = -inf and subtracts 0 instead: its p and alpha are exp2(-inf) = 0
    // (not the NaN of -inf - -inf).
    if (__builtin_amdgcn_ballot_w64(mx > m) != 0) {  // uniform
      const float mn = fmaxf(m, mx);
      const float alpha = __builtin_amdgcn_exp2f(m - (mn == -INFINITY ? 0.f : mn));
      l *= alpha;
      m = mn;
      huge = __builtin_amdgcn_ballot_w64(fabsf(m) >= 0x1p24f && m != -INFINITY) != 0;
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt) acc[dt] *= alpha;
    }
    // p = exp2(c sc - m) by one FMA.  m is the rounded product, so the largest p is 2^r with r the rounding error of
    // m, up to half an ulp: a factor that all p of the query share, until p leaves fp16.  From |m| = 2^24 on (r up to
    // one) the difference is taken of the rounded products instead, which makes it exactly zero at the maximum.
    float ms = m == -INFINITY ? 0.f : m, pc = sc;
    if (__builtin_expect(huge, 0)) {
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) c[j][r] = as_f32_value(c[j][r] * sc) - ms;
      ms = 0.f;
      pc = 1.f;
    }
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      float ps = 0.f;
      f16x8 pa[2];
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        pa[r >> 3][r & 7] = static_cast<f16>(__builtin_amdgcn_exp2f(fmaf(c[j][r], pc, -ms)));
        // l sums the rounded p; the multiply by one (opaque) makes it one v_fma_mix_f32 reading the fp16 value
        ps = fmaf(static_cast<float>(pa[r >> 3][r & 7]), one, ps);
      }
      if (j > 0 && blk + j >= wblk) break;  // uniform: past the wavefront's last token (p = 0 would meet its values)
      l += ps;
      if (j > 0) load_v(j);
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int dt = 0; dt < D / 32; ++dt)
          acc[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(va[j][dt][ks], pa[ks], acc[dt], 0, 0, 0);
    }
  };
  // Stage st: wait for its DMA, issue the next stage into the buffer that stage st - 1 has just left, multiply.
  auto step = [&](const uint8_t* cur, uint8_t* other, int st) __attribute__((always_inline)) {
    dma_wait_barrier();
    if (st + 1 < s1) {
      issue(other, st + 1);
      fetch_page(min(st + 2, s1 - 1));
    }
    const int blk = (st * CW + cw) * NB;
    if (blk < wblk) blocks(cur, blk);
  };
  if (s0 < s1) {
    fetch_page(s0);
    issue(st0, s0);
    fetch_page(min(s0 + 1, s1 - 1));
    for (int st = s0;;) {  // uniform
      step(st0, st1, st);
      if (++st >= s1) break;
      step(st1, st0, st);
      if (++st >= s1) break;
    }
  }
  l += __shfl_xor(l, 32, 64);

  // Merge the CW groups in order: groups 1.. park (max, sum, O) in the stage buffers.
  if constexpr (CW > 1) {
    dma_wait_barrier();  // every DMA has landed, every wavefront has read its last stage
    constexpr int kWaveO = 64 * 64 * 4;            // O of one wavefront
    constexpr int kPer = 2 * kHalf / kWaveO;       // wavefronts per stage buffer
    static_assert((CW - 1) * VW <= 2 * kPer, "parked outputs fit the first two buffers");
    auto park = [&](int g, int v) __attribute__((always_inline)) -> float* {
      const int i = (g - 1) * VW + v;
      return reinterpret_cast<float*>((i < kPer ? st0 : st1) + (i % kPer) * kWaveO) + lane;
    };
    if (cw > 0) {
      float* o = park(cw, vw);
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[(16 * dt + r) * 64] = acc[dt][r];
      sm_ml[cw][vw][0][lane] = m;
      sm_ml[cw][vw][1][lane] = l;
    }
    __syncthreads();
    if (cw > 0) return;
#pragma unroll
    for (int g = 1; g < CW; ++g) {
      const float* o = park(g, vw);
      const float mg = sm_ml[g][vw][0][lane], lg = sm_ml[g][vw][1][lane];
      const float mn = fmaxf(m, mg), ms = mn == -INFINITY ? 0.f : mn;
      const float fa = __builtin_amdgcn_exp2f(m - ms), fb = __builtin_amdgcn_exp2f(mg - ms);
      m = mn;
      l = fmaf(l, fa, lg * fb);
#pragma unroll
      for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[dt][r] = fmaf(acc[dt][r], fa, o[(16 * dt + r) * 64] * fb);
    }
  }
  if (!live) return;
  const int t = vq / G, g = vq - t * G;
  const size_t head = ((size_t)b * q_len + t) * Hq + (size_t)kvh * G + g;
  if (S == 1) {
    f16* po = out + head * D + 4 * h;
    const float inv = l > 0.f ? 1.f / l : 0.f;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f16x4*>(po + 32 * dt + 8 * j) =
            f16x4{static_cast<f16>(acc[dt][4 * j] * inv), static_cast<f16>(acc[dt][4 * j + 1] * inv),
                  static_cast<f16>(acc[dt][4 * j + 2] * inv), static_cast<f16>(acc[dt][4 * j + 3] * inv)};
  } else {
    float* po = part_o + (head * S + split) * D + 4 * h;
#pragma unroll
    for (int dt = 0; dt < D / 32; ++dt)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(po + 32 * dt + 8 * j) =
            f32x4{acc[dt][4 * j], acc[dt][4 * j + 1], acc[dt][4 * j + 2], acc[dt][4 * j + 3]};
    if (h == 0) {
      float* ml = part_ml + (head * S + split) * 2;
      ml[0] = m;
      ml[1] = l;
    }
  }
}

// ----------------------------------------------------------------------------
// Generic kernel (fp32 or fp16 pools, any page size, head_dim <= 256): four wavefronts
// per (128-token chunk, KV head, row).  LPT lanes (D <= 4 LPT) hold four dims each of a
// token's K and V rows, so a wavefront takes TPW = 64 / LPT tokens per load and kGenU
// loads of each in flight; the score of a token is summed over its LPT lanes by DPP and
// stays in their registers, where P V needs it, so nothing but the wavefronts' (max, sum,
// O) goes through LDS.  kGenHeads query heads of the group share each load.  One chunk
// (NC == 1) writes the output itself; more leave partials for attn_merge.  These launches
// are bound by latency (page entry, then K and V): the tiny model's decode attention took
// 23.5 us with one wavefront per chunk, a token per lane and the dims in turn.
constexpr int kGenWaves = 4;
constexpr int kGenU = 8;
constexpr int kGenHeads = 4;

// Four consecutive values as fp32 (VEC: one vector load; else one by one, zero past n).
template <bool VEC>
__device__ __forceinline__ f32x4 load_dims(const float* p, int n) {
  if constexpr (VEC) return *reinterpret_cast<const f32x4*>(p);
  f32x4 v;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] = e < n ? p[e] : 0.f;
  return v;
}
template <bool VEC>
__device__ __forceinline__ f32x4 load_dims(const f16* p, int n) {
  f32x4 v;
  if constexpr (VEC) {
    const f16x4 t = *reinterpret_cast<const f16x4*>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = static_cast<float>(t[e]);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = e < n ? static_cast<float>(p[e]) : 0.f;
  }
  return v;
}

template <typename T, int LPT, bool VEC>
__global__ __launch_bounds__(64 * kGenWaves) void attn_chunk_generic(
    const T* __restrict__ q, const T* __restrict__ kp, const T* __restrict__ vp,
    const int32_t* __restrict__ pt, const int32_t* __restrict__ lens, T* __restrict__ out,
    float* __restrict__ part_o, float* __restrict__ part_ml,
    int q_len, int Hq, int Hkv, int D, int P, int max_pages, int NC, float scale_log2) {
  constexpr int TPW = 64 / LPT;
  __shared__ float sm_m[kGenWaves][kGenHeads], sm_l[kGenWaves][kGenHeads];
  __shared__ __align__(16) float sm_o[kGenWaves][kGenHeads][4 * LPT];
  const int chunk = blockIdx.x, kvh = blockIdx.y, row = blockIdx.z;
  const int L = visible_len(lens, row, q_len, max_pages * P);
  const int t0 = chunk * kChunk;
  const int G = Hq / Hkv;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int d0 = 4 * (lane & (LPT - 1)), grp = lane / LPT;
  const int nd = max(0, min(4, D - d0));  // this lane's dims (none: it repeats dim 0 and drops out by zeros)
  const int n = max(0, min(L, t0 + kChunk) - t0);
  const int32_t* ptrow = pt + (size_t)(row / q_len) * max_pages;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  for (int h0 = 0; h0 < G; h0 += kGenHeads) {  // uniform
    const int nh = min(kGenHeads, G - h0);
    const size_t head0 = (size_t)row * Hq + (size_t)kvh * G + h0;
    f32x4 qv[kGenHeads], o[kGenHeads];
    float m[kGenHeads], l[kGenHeads];
#pragma unroll
    for (int h = 0; h < kGenHeads; ++h) {
      const f32x4 t = load_dims<VEC>(q + (head0 + min(h, nh - 1)) * D + (nd ? d0 : 0), nd);
      qv[h] = nd ? t : zero;
      o[h] = zero;
      m[h] = -FLT_MAX;  // finite: a score of -inf then weighs exp2(-inf) = 0 even where it stands alone
      l[h] = 0.f;
    }
    for (int j0 = wave * TPW; j0 < n; j0 += kGenU * kGenWaves * TPW) {  // uniform; tokens j0 + i * kGenWaves * TPW + grp
      f32x4 kv[kGenU], vv[kGenU];
      bool in[kGenU];
#pragma unroll
      for (int i = 0; i < kGenU; ++i) {
        const int j = j0 + i * kGenWaves * TPW + grp;
        in[i] = j < n;
        const int t = t0 + (in[i] ? j : 0);  // tokens past the chunk re-read its first one (p = 0)
        const size_t at = (((size_t)ptrow[t / P] * Hkv + kvh) * P + t % P) * D + (nd ? d0 : 0);
        const f32x4 a = load_dims<VEC>(kp + at, nd), c = load_dims<VEC>(vp + at, nd);
        kv[i] = nd ? a : zero;
        vv[i] = in[i] ? c : zero;
      }
#pragma unroll
      for (int h = 0; h < kGenHeads; ++h) {
        if (h >= nh) break;
        float s[kGenU], mx = m[h];
#pragma unroll
        for (int i = 0; i < kGenU; ++i) {
          float dot = 0.f;
#pragma unroll
          for (int e = 0; e < 4; ++e) dot = fmaf(qv[h][e], kv[i][e], dot);
          dot = row16_sum(dot);
          if constexpr (LPT >= 32) dot += __shfl_xor(dot, 16, 64);
          if constexpr (LPT >= 64) dot += __shfl_xor(dot, 32, 64);
          s[i] = in[i] ? dot * scale_log2 : -INFINITY;
          mx = fmaxf(mx, s[i]);
        }
        if constexpr (LPT <= 16) mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        if constexpr (LPT <= 32) mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float a = exp2f(m[h] - mx);
        l[h] *= a;
        o[h] *= a;
        m[h] = mx;
#pragma unroll
        for (int i = 0; i < kGenU; ++i) {
          const float p = exp2f(s[i] - mx);
          l[h] += p;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[h][e] = fmaf(p, vv[i][e], o[h][e]);
        }
      }
    }
    // Sum the TPW token groups of the wavefront, then merge the wavefronts in order.
#pragma unroll
    for (int h = 0; h < kGenHeads; ++h) {
#pragma unroll
      for (int off = LPT; off < 64; off <<= 1) {
        l[h] += __shfl_xor(l[h], off, 64);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[h][e] += __shfl_xor(o[h][e], off, 64);
      }
      if (grp == 0) *reinterpret_cast<f32x4*>(&sm_o[wave][h][d0]) = o[h];
      if (lane == 0) {
        sm_m[wave][h] = m[h];
        sm_l[wave][h] = l[h];
      }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < nh * D; idx += 64 * kGenWaves) {
      const int h = idx / D, d = idx - h * D;
      float M = sm_m[0][h];
#pragma unroll
      for (int w = 1; w < kGenWaves; ++w) M = fmaxf(M, sm_m[w][h]);
      float den = 0.f, acc = 0.f;
#pragma unroll
      for (int w = 0; w < kGenWaves; ++w) {
        const float f = exp2f(sm_m[w][h] - M);
        den = fmaf(sm_l[w][h], f, den);
        acc = fmaf(sm_o[w][h][d], f, acc);
      }
      // No weight at all: no tokens (the output is 0), or scores of -inf alone (NaN, as a softmax over them gives).
      const bool none = den == 0.f, nan = none && n > 0;
      if (NC == 1) {
        out[(head0 + h) * D + d] = from_f32<T>(as_f32_value(acc * (nan ? NAN : none ? 0.f : 1.f / den)));
      } else {
        part_o[((head0 + h) * NC + chunk) * D + d] = acc;
        if (d == 0) {
          float* ml = part_ml + ((head0 + h) * NC + chunk) * 2;
          ml[0] = none ? -INFINITY : M;
          ml[1] = nan ? 1.f : den;
        }
      }
    }
    __syncthreads();  // the next heads write the same arrays
  }
}

// ----------------------------------------------------------------------------
// Merge S partials of one (row, head): out = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s.
// Latency-bound (a few KiB per workgroup), so no load waits for another: thread s
// reads split s's (m, l), the weights 2^(m_s - M) go through LDS, and each output
// element's S partials are loaded 8 at a time before they are summed.  Sums run in
// split order, as the serial form for S > kMergeFast does.  A row whose scores are all
// -inf (every M -inf, some l > 0: the generic kernel's partials) gives NaN, as a softmax
// over them does; one without tokens (every l 0) gives 0.  o * inv is rounded to fp32
// before the fp16 conversion (as_f32_value: no single-rounding mixed-precision multiply),
// the same two roundings the O projection's merge (qgemm.hip, attn_merged_chunk) makes.
constexpr int kMergeFast = 128;
template <typename T>
__global__ __launch_bounds__(128) void attn_merge(const float* __restrict__ part_o, const float* __restrict__ part_ml,
                                                  T* __restrict__ out, int Hq, int D, int S) {
  const int head = blockIdx.x, row = blockIdx.y;
  const float* ml = part_ml + ((size_t)row * Hq + head) * S * 2;
  if (S <= kMergeFast) {
    __shared__ float sw[kMergeFast], sl[kMergeFast], smax[2];
    const int t = threadIdx.x;
    const float mv = t < S ? ml[2 * t] : -INFINITY;
    const float lv = t < S ? ml[2 * t + 1] : 0.f;
    const float wm = wave_max(mv);
    if ((t & 63) == 0) smax[t >> 6] = wm;
    __syncthreads();
    const float M = fmaxf(smax[0], smax[1]);
    sw[t] = (t < S && M != -INFINITY) ? exp2f(mv - M) : 0.f;
    sl[t] = lv;
    __syncthreads();
    float den = 0.f;
    if (M != -INFINITY)
      for (int s = 0; s < S; ++s) den = fmaf(sl[s], sw[s], den);
    float inv = den > 0.f ? 1.f / den : 0.f;
    if (M == -INFINITY)
      for (int s = 0; s < S; ++s) inv = sl[s] > 0.f ? NAN : inv;
    const float* po = part_o + ((size_t)row * Hq + head) * S * D;
    for (int d = t; d < D; d += 128) {
      float o = 0.f;
      for (int s0 = 0; s0 < S; s0 += 8) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = po[(size_t)min(s0 + j, S - 1) * D + d];
#pragma unroll
        for (int j = 0; j < 8; ++j)
          if (s0 + j < S) o = fmaf(v[j], sw[s0 + j], o);
      }
      out[((size_t)row * Hq + head) * D + d] = from_f32<T>(as_f32_value(o * inv));
    }
    return;
  }
  float M = -INFINITY;
  for (int s = 0; s < S; ++s) M = fmaxf(M, ml[2 * s]);
  float den = 0.f;
  if (M != -INFINITY)
    for (int s = 0; s < S; ++s) den = fmaf(ml[2 * s + 1], exp2f(ml[2 * s] - M), den);
  float inv = den > 0.f ? 1.f / den : 0.f;
  if (M == -INFINITY)
    for (int s = 0; s < S; ++s) inv = ml[2 * s + 1] > 0.f ? NAN : inv;
  const float* po = part_o + ((size_t)row * Hq + head) * S * D;
  for (int d = threadIdx.x; d < D; d += blockDim.x) {
    float o = 0.f;
    if (M != -INFINITY)
      for (int s = 0; s < S; ++s) o = fmaf(po[(size_t)s * D + d], exp2f(ml[2 * s] - M), o);
    out[((size_t)row * Hq + head) * D + d] = from_f32<T>(as_f32_value(o * inv));
  }
}

int max_splits(int max_context) { return max(1, (max_context + kMinSplitTokens - 1) / kMinSplitTokens); }

int generic_chunks(int max_context) { return max(1, (max_context + kChunk - 1) / kChunk); }

// Splits for the fp16 path: about one workgroup per CU (256 / (rows * kv_heads)),
// at most 8.  Measured at 2048 tokens of context, 32/8 heads (attention + merge):
// batch 1 best at 8 splits (13.1 us; 16 splits 14.8, 64 splits 34), batch 4 at 4-8,
// batch 8 at 4 (19.7 us; 8 splits 25.3), batch 16 at 2 (29.5 us; 1 split 32.8,
// 4 splits 33.9), batch 32 at 1.  More splits add per-workgroup fixed cost (page
// table, q, first load latency, the 8-wavefront merge) and a longer merge.
int choose_splits(int rows, int Hkv, int max_context) {
  const long groups = (long)rows * Hkv;
  const int want = (int)min(8L, max(1L, 256 / groups));
  return max(1, min(want, max_splits(max_context)));
}

// The MFMA kernel serves fp16 pools with head_dim 128, pages of a multiple of 16
// tokens and up to 8 query heads per KV head; everything else runs the generic kernel.
bool mfma_path(int kv_dtype, int D, int P, int G) { return kv_dtype == CIR_F16 && D == 128 && P % 16 == 0 && G <= 8; }

// Context splits of a launch: about one workgroup per CU on the MFMA path, one
// partial per 128-token chunk on the generic path.
int launch_splits(int rows, int Hkv, int max_ctx, bool mfma) {
  return mfma ? choose_splits(rows, Hkv, max_ctx) : generic_chunks(max_ctx);
}

// Bytes of split partials (O, then (max, sum)) a launch writes: none when it runs
// unsplit (one chunk on the generic path) and the kernel writes the output itself.
size_t partial_bytes(int rows, int Hq, int D, int S) {
  if (S == 1) return 0;
  return (size_t)rows * Hq * S * ((size_t)D + 2) * sizeof(float);
}

// Compute units of the current device, looked up once per device.
int device_cus() {
  static std::atomic<int> cus[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int n = cus[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
    cus[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}

// Prefill launch: wavefronts on query tiles x wavefronts sharing their context, tiles per (sequence, KV head) and
// context splits.  A sequence of more than 64 vectors has the same bits in every batch up to kPfSplitTokens of table; else
// the batch, the table's width and the CUs decide too, and a row's last bits may differ between batches and widths.
// Measured on MI355X, us per launch (32/8 heads unless said):
//   * up to kPfSplitTokens of table a workgroup walks few stages and its start and merge dominate: four wavefronts, two
//     workgroups per CU, no merge (8 x 512 tokens 39.7 against 51.2 with 8 wavefronts, 5 x 301 at 28/4 15.1 against 20.4).
//   * longer contexts: 8 wavefronts in two context groups (2 x 509 tokens after 3500 at 28/4: 78.6 against 94.8 with
//     four wavefronts in one group); four in one group again once the grid keeps every CU's two workgroups busy for more than one round
//     (2 x 2048 tokens: 89.0 against 98.3); 64-vector tiles in four context groups where 128-vector tiles leave half
//     of the CUs idle (4 x 400 tokens after 1000 at 8/8: 23.5 against 28.9, 100 after 3000: 24.3 against 28.5).
//   * a sequence of up to 64 vectors, at any length: four context groups, or two once the grid exceeds the CUs, since the
//     128 KiB of LDS of four leave one workgroup per CU (64 x 4 tokens after 100 7.8 / 13.8, after 500 24.2 / 31.2, after
//     1500 66 / 72, 128 x 2 after 900 82.7 / 99.3; in smaller grids 1 x 2 after 900 18.0 / 16.4), or its splits fill
//     three quarters of them (16 x 5 after 1050 19.3 / 20.7, 8 x 5 after 4500 29.2 / 31.4; on fewer workgroups 3 x 5
//     after 1500 18.8 / 17.0; with more tiles 8 x 30 after 4500 54.3 / 46.4).
//   * a grid below one workgroup per CU splits long contexts, by the table's capacity, into pieces of about
//     kPfSplitTokens / 2 (of that capacity: a context that fills half its table is cut twice as fine), if the caller
//     gave a workspace for the partials (may_split).  The host does not see the lengths, so a short context in a wide
//     table pays the merge launch for nothing: 1 x 5 tokens in a table of 2048, split against unsplit, after 100 10.5 /
//     7.7, after 600 11.7 / 12.6, after 1500 13.2 / 22.1.
struct PrefillPlan {
  int vec_waves, ctx_waves, tiles, splits;
};
constexpr int kPfSplitTokens = 1024;
PrefillPlan prefill_plan(int batch, int q_len, int Hkv, int G, int max_ctx, bool may_split) {
  const int nvec = q_len * G;
  const long seqs = (long)Hkv * batch, cus = device_cus();
  const long groups4 = (nvec + 4 * kPfVec - 1) / (4 * kPfVec) * seqs;  // workgroups at 128 vectors each
  const bool longctx = max_ctx > kPfSplitTokens;
  PrefillPlan p;
  p.vec_waves = (nvec <= 2 * kPfVec || (longctx && 2 * groups4 <= cus)) ? 2 : 4;
  p.tiles = (nvec + kPfVec * p.vec_waves - 1) / (kPfVec * p.vec_waves);
  p.splits = longctx && may_split ? (int)max(1L, min(2L * max_ctx / kPfSplitTokens, cus / (p.tiles * seqs))) : 1;
  const long wgs = p.tiles * seqs * p.splits;
  if (p.vec_waves == 2) p.ctx_waves = (p.splits > 1 ? p.tiles == 1 && wgs >= 3 * cus / 4 : wgs > cus) ? 2 : 4;
  else p.ctx_waves = longctx && groups4 < 3 * cus ? 2 : 1;
  return p;
}

int launch_attention(const void* q, const void* k_pool, const void* v_pool, const int32_t* page_table,
                     const int32_t* seq_lens, void* out, void* workspace, size_t workspace_bytes,
                     int batch, int q_len, int Hq, int Hkv, int D, int P, int max_pages, float scale,
                     int kv_dtype, void* stream, QkvIn qkv = QkvIn{nullptr, 0, nullptr, nullptr},
                     bool merge = true, bool exact_workspace = false, bool prefill_splits = false) {
  CIR_CHECK_ARG(batch >= 0 && q_len >= 1, "attention: batch must be >= 0 and q_len >= 1");
  if (batch == 0) return 0;
  CIR_CHECK_ARG((q || qkv.part) && k_pool && v_pool && page_table && seq_lens && out, "attention: null pointer");
  CIR_CHECK_ARG(Hkv > 0 && Hq > 0 && Hq % Hkv == 0, "attention: num_heads (%d) must be a multiple of num_kv_heads (%d)", Hq, Hkv);
  CIR_CHECK_ARG(D > 0 && D <= 256, "attention: head_dim %d out of range (1..256)", D);
  CIR_CHECK_ARG(P > 0 && max_pages > 0, "attention: page_size and max_pages must be positive");
  CIR_CHECK_ARG(kv_dtype == CIR_F16 || kv_dtype == CIR_F32, "attention: kv_dtype must be CIR_F16 or CIR_F32");
  const int rows = batch * q_len;
  const int max_ctx = max_pages * P;
  CIR_CHECK_ARG(rows <= 65535 && Hkv <= 65535, "attention: grid too large");
  const float scale_log2 = scale * kLog2e;
  const int G = Hq / Hkv;
  hipStream_t s = as_stream(stream);
  const bool mfma = mfma_path(kv_dtype, D, P, G);
  // The prefill kernel's DMA takes 16-byte groups of the pools by 32-bit offsets inside a page; pools on other addresses
  // (or pages of 4 GiB a head) run the decode kernel over the rows, which reads them by plain loads.
  const bool prefill = mfma && q_len > 1 && P < (1 << 24) &&
                       (reinterpret_cast<uintptr_t>(k_pool) | reinterpret_cast<uintptr_t>(v_pool)) % 16 == 0;
  const int S = mfma && q_len > 1 ? 1 : launch_splits(rows, Hkv, max_ctx, mfma);
  // The advertised size (cir_paged_attention_workspace_bytes) covers any split count;
  // the static-scratch and split-prefill entry points check the bytes this launch writes instead.
  PrefillPlan pl{};
  if (prefill) pl = prefill_plan(batch, q_len, Hkv, G, max_ctx, prefill_splits);
  const size_t need = !exact_workspace ? cir_paged_attention_workspace_bytes(rows, Hq, D, max_ctx)
                      : prefill        ? partial_bytes(rows, Hq, D, pl.splits)
                                       : partial_bytes(rows, Hq, D, S);
  CIR_CHECK_ARG((workspace || need == 0) && workspace_bytes >= need,
                "attention: workspace too small (%zu < %zu)", workspace_bytes, need);
  CIR_CHECK_ARG(!qkv.part || (mfma && q_len == 1 && qkv.splits >= 1 && qkv.inv_freq && qkv.positions),
                "attention: the fused QKV input needs decode (q_len 1), fp16 pools, head_dim 128, page_size %% 16 == 0, "
                "num_heads/num_kv_heads <= 8 and inv_freq/positions");
  CIR_CHECK_ARG(merge || (mfma && S > 1), "attention: unmerged partials need the fp16 decode path with > 1 split");
  float* part_o = static_cast<float*>(workspace);
  float* part_ml = part_o + (size_t)rows * Hq * S * D;
  dim3 grid(S, Hkv, rows);
  if (prefill) {  // query tiles over each sequence's blocks
    const dim3 pgrid(Hkv * batch, pl.tiles, pl.splits);
    const auto kernel = pl.vec_waves == 2
                            ? (pl.ctx_waves == 4 ? attn_prefill_f16_d128<2, 4, 1> : attn_prefill_f16_d128<2, 2, 1>)
                            : (pl.ctx_waves == 2 ? attn_prefill_f16_d128<4, 2, 2> : attn_prefill_f16_d128<4, 1, 2>);
    part_ml = part_o + (size_t)rows * Hq * pl.splits * D;
    kernel<<<pgrid, 64 * pl.vec_waves * pl.ctx_waves, 0, s>>>(
        static_cast<const f16*>(q), static_cast<const f16*>(k_pool), static_cast<const f16*>(v_pool), page_table,
        seq_lens, static_cast<f16*>(out), part_o, part_ml, q_len, Hq, Hkv, P, max_pages, pl.splits,
        scale_log2 == 0.f ? FLT_MIN : scale_log2);  // (a masked score is -inf: -inf * 0 would be NaN)
    const int st = launch_status();
    if (st || pl.splits == 1) return st;
    attn_merge<f16><<<dim3(Hq, rows), 128, 0, s>>>(part_o, part_ml, static_cast<f16*>(out), Hq, D, pl.splits);
    return launch_status();
  }
  if (mfma) {
    // Longest rows first when the workgroups outnumber the CUs (they then run in rounds).
    const int sort_rows = q_len == 1 && rows <= 64 * kWaves && (long)S * Hkv * rows > device_cus();
    auto kq = static_cast<const f16*>(q);
    auto kk = static_cast<f16*>(const_cast<void*>(k_pool));
    auto kv = static_cast<f16*>(const_cast<void*>(v_pool));
    auto ko = static_cast<f16*>(out);
#define CIR_ATT_CASE(g)                                                                                             \
  case g:                                                                                                           \
    if (qkv.part)                                                                                                   \
      attn_f16_d128<g, true><<<grid, 64 * kWaves, 0, s>>>(kq, kk, kv, page_table, seq_lens, ko, part_o, part_ml,   \
                                                           q_len, Hq, Hkv, P, max_pages, S, scale_log2,          \
                                                           sort_rows, qkv);                                        \
    else                                                                                                            \
      attn_f16_d128<g, false><<<grid, 64 * kWaves, 0, s>>>(kq, kk, kv, page_table, seq_lens, ko, part_o, part_ml,  \
                                                            q_len, Hq, Hkv, P, max_pages, S, scale_log2,         \
                                                            sort_rows, qkv);                                       \
    break;
    switch (G) {
      CIR_ATT_CASE(1) CIR_ATT_CASE(2) CIR_ATT_CASE(3) CIR_ATT_CASE(4)
      CIR_ATT_CASE(5) CIR_ATT_CASE(6) CIR_ATT_CASE(7) CIR_ATT_CASE(8)
    }
#undef CIR_ATT_CASE
    const int st = launch_status();
    if (st || S == 1 || !merge) return st;
  } else {
    // Vector loads of four dims need rows on whole, aligned groups of four.
    const bool vec = D % 4 == 0 && (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k_pool) |
                                    reinterpret_cast<uintptr_t>(v_pool)) % 16 == 0;
    auto go = [&]<typename T, int LPT, bool VEC>() {
      attn_chunk_generic<T, LPT, VEC><<<grid, 64 * kGenWaves, 0, s>>>(
          static_cast<const T*>(q), static_cast<const T*>(k_pool), static_cast<const T*>(v_pool), page_table, seq_lens,
          static_cast<T*>(out), part_o, part_ml, q_len, Hq, Hkv, D, P, max_pages, S, scale_log2);
    };
    auto by_dim = [&]<typename T, bool VEC>() {
      if (D <= 64) go.template operator()<T, 16, VEC>();
      else if (D <= 128) go.template operator()<T, 32, VEC>();
      else go.template operator()<T, 64, VEC>();
    };
    if (kv_dtype == CIR_F16) vec ? by_dim.template operator()<f16, true>() : by_dim.template operator()<f16, false>();
    else vec ? by_dim.template operator()<float, true>() : by_dim.template operator()<float, false>();
    const int st = launch_status();
    if (st || S == 1) return st;
  }
  dim3 mgrid(Hq, rows);
  if (kv_dtype == CIR_F16) {
    attn_merge<f16><<<mgrid, 128, 0, s>>>(part_o, part_ml, static_cast<f16*>(out), Hq, D, S);
  } else {
    attn_merge<float><<<mgrid, 128, 0, s>>>(part_o, part_ml, static_cast<float*>(out), Hq, D, S);
  }
  return launch_status();
}

}  // namespace
}  // namespace cir

extern "C" size_t cir_paged_attention_workspace_bytes(int rows, int num_heads, int head_dim, int max_context) {
  if (rows <= 0 || num_heads <= 0 || head_dim <= 0) return 0;
  // Partial O and (max, sum) per (row, head, split), sized for the larger split count of the two paths.
  const int a = cir::max_splits(max_context), c = cir::generic_chunks(max_context);
  const size_t s = (size_t)(a > c ? a : c);
  return (size_t)rows * num_heads * s * ((size_t)head_dim + 2) * sizeof(float);
}

extern "C" int cir_paged_decode_attention(const void* q, const void* k_pool, const void* v_pool,
                                          const int32_t* page_table, const int32_t* seq_lens, void* out,
                                          void* workspace, size_t workspace_bytes, int batch, int num_heads,
                                          int num_kv_heads, int head_dim, int page_size, int max_pages, float scale,
                                          int kv_dtype, void* stream) {
  return cir::launch_attention(q, k_pool, v_pool, page_table, seq_lens, out, workspace, workspace_bytes, batch, 1,
                               num_heads, num_kv_heads, head_dim, page_size, max_pages, scale, kv_dtype, stream);
}

extern "C" int cir_paged_decode_splits(int batch, int num_heads, int num_kv_heads, int head_dim, int page_size,
                                       int max_pages, int kv_dtype) {
  if (batch <= 0 || num_heads <= 0 || num_kv_heads <= 0 || page_size <= 0 || max_pages <= 0) return 0;
  const bool mfma = num_heads % num_kv_heads == 0 &&
                    cir::mfma_path(kv_dtype, head_dim, page_size, num_heads / num_kv_heads);
  return cir::launch_splits(batch, num_kv_heads, max_pages * page_size, mfma);
}

extern "C" int cir_paged_prefill_attention(const void* q, const void* k_pool, const void* v_pool,
                                           const int32_t* page_table, const int32_t* seq_lens, void* out,
                                           void* workspace, size_t workspace_bytes, int batch, int q_len,
                                           int num_heads, int num_kv_heads, int head_dim, int page_size,
                                           int max_pages, float scale, int kv_dtype, void* stream) {
  return cir::launch_attention(q, k_pool, v_pool, page_table, seq_lens, out, workspace, workspace_bytes, batch,
                               q_len, num_heads, num_kv_heads, head_dim, page_size, max_pages, scale, kv_dtype,
                               stream);
}

extern "C" size_t cir_paged_prefill_split_bytes(int batch, int q_len, int num_heads, int num_kv_heads, int head_dim,
                                                int page_size, int max_pages, int kv_dtype) {
  if (batch <= 0 || q_len <= 1 || num_heads <= 0 || num_kv_heads <= 0 || page_size <= 0 || max_pages <= 0 ||
      num_heads % num_kv_heads)
    return 0;
  const int G = num_heads / num_kv_heads;
  if (!cir::mfma_path(kv_dtype, head_dim, page_size, G)) return 0;
  const cir::PrefillPlan p = cir::prefill_plan(batch, q_len, num_kv_heads, G, max_pages * page_size, true);
  return cir::partial_bytes(batch * q_len, num_heads, head_dim, p.splits);
}

extern "C" int cir_paged_prefill_attention_split(const void* q, const void* k_pool, const void* v_pool,
                                                 const int32_t* page_table, const int32_t* seq_lens, void* out,
                                                 void* workspace, size_t workspace_bytes, int batch, int q_len,
                                                 int num_heads, int num_kv_heads, int head_dim, int page_size,
                                                 int max_pages, float scale, int kv_dtype, void* stream) {
  return cir::launch_attention(q, k_pool, v_pool, page_table, seq_lens, out, workspace, workspace_bytes, batch,
                               q_len, num_heads, num_kv_heads, head_dim, page_size, max_pages, scale, kv_dtype,
                               stream, cir::QkvIn{nullptr, 0, nullptr, nullptr}, true, true, true);
}

extern "C" int cir_paged_decode_attention_qkv(const float* qkv_partial, int splits, const float* inv_freq,
                                              const int32_t* positions, void* k_pool, void* v_pool,
                                              const int32_t* page_table, const int32_t* seq_lens, void* out,
                                              void* workspace, size_t workspace_bytes, int batch, int num_heads,
                                              int num_kv_heads, int head_dim, int page_size, int max_pages,
                                              float scale, void* stream) {
  CIR_CHECK_ARG(batch == 0 || qkv_partial, "attention_qkv: null qkv_partial");
  return cir::launch_attention(nullptr, k_pool, v_pool, page_table, seq_lens, out, workspace, workspace_bytes, batch,
                               1, num_heads, num_kv_heads, head_dim, page_size, max_pages, scale, CIR_F16, stream,
                               cir::QkvIn{qkv_partial, splits, inv_freq, positions});
}

extern "C" int cir_paged_decode_attention_qkv_parts(const float* qkv_partial, int splits, const float* inv_freq,
                                                    const int32_t* positions, void* k_pool, void* v_pool,
                                                    const int32_t* page_table, const int32_t* seq_lens, void* workspace,
                                                    size_t workspace_bytes, int batch, int num_heads, int num_kv_heads,
                                                    int head_dim, int page_size, int max_pages, float scale,
                                                    void* stream) {
  CIR_CHECK_ARG(batch == 0 || qkv_partial, "attention_qkv_parts: null qkv_partial");
  // `out` is never written on this path; the workspace pointer stands in for the non-null check.
  return cir::launch_attention(nullptr, k_pool, v_pool, page_table, seq_lens, workspace, workspace, workspace_bytes,
                               batch, 1, num_heads, num_kv_heads, head_dim, page_size, max_pages, scale, CIR_F16,
                               stream, cir::QkvIn{qkv_partial, splits, inv_freq, positions}, false);
}


// ----------------------------------------------------------------------------
// Decode attention that allocates nothing (cir_paged_decode_attention_noalloc).
// The split partials go to `scratch`, a device array of fixed size that every call
// on a GPU shares.  Host code never passes the array's name to a kernel (on the
// host it is only a stand-in for the symbol): its device address is looked up once
// per device with hipGetSymbolAddress and kept in g_scratch_ptr.
static constexpr size_t kScratchBytes = CIR_ATTENTION_NOALLOC_MAX_BYTES;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace cir {
namespace {

constexpr int kMaxDevices = 64;
std::atomic<void*> g_scratch_ptr[kMaxDevices];
std::mutex g_scratch_mu;

// Device address of `scratch` on the current device (looked up on the first call
// for that device, with that device current).
int scratch_on_current_device(void** out) {
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) {
    set_error("attention_noalloc: hipGetDevice failed: %s", hipGetErrorString(e));
    return static_cast<int>(e);
  }
  if (dev < 0 || dev >= kMaxDevices) {
    set_error("attention_noalloc: device %d beyond the %d devices the library tracks", dev, kMaxDevices);
    return static_cast<int>(hipErrorInvalidDevice);
  }
  void* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
  if (!p) {
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    p = g_scratch_ptr[dev].load(std::memory_order_relaxed);
    if (!p) {
      e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
      if (e != hipSuccess || !p) {
        set_error("attention_noalloc: hipGetSymbolAddress(scratch) failed on device %d: %s", dev,
                  hipGetErrorString(e));
        return static_cast<int>(e != hipSuccess ? e : hipErrorInvalidSymbol);
      }
      g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
  }
  *out = p;
  return 0;
}

}  // namespace
}  // namespace cir

extern "C" int cir_paged_decode_attention_noalloc(const void* q, const void* k_pool, const void* v_pool,
                                                  const int32_t* page_table, const int32_t* seq_lens, void* out,
                                                  int batch, int num_heads, int num_kv_heads, int head_dim,
                                                  int page_size, int max_pages, float scale, int kv_dtype,
                                                  void* stream) {
  CIR_CHECK_ARG(batch >= 0, "attention_noalloc: batch must be >= 0");
  if (batch == 0) return 0;
  CIR_CHECK_ARG(num_kv_heads > 0 && num_heads > 0 && num_heads % num_kv_heads == 0,
                "attention_noalloc: num_heads (%d) must be a multiple of num_kv_heads (%d)", num_heads, num_kv_heads);
  CIR_CHECK_ARG(head_dim > 0 && head_dim <= 256, "attention_noalloc: head_dim %d out of range (1..256)", head_dim);
  CIR_CHECK_ARG(page_size > 0 && max_pages > 0, "attention_noalloc: page_size and max_pages must be positive");
  CIR_CHECK_ARG(batch <= 65535, "attention_noalloc: grid too large");
  const bool mfma = cir::mfma_path(kv_dtype, head_dim, page_size, num_heads / num_kv_heads);
  const int S = cir::launch_splits(batch, num_kv_heads, max_pages * page_size, mfma);
  const size_t need = cir::partial_bytes(batch, num_heads, head_dim, S);
  CIR_CHECK_ARG(need <= kScratchBytes,
                "attention_noalloc: the split partials need %zu bytes, more than the %zu bytes of static scratch "
                "(batch %d, %d heads, head_dim %d, %d splits); use cir_paged_decode_attention with a workspace",
                need, kScratchBytes, batch, num_heads, head_dim, S);
  void* ws = nullptr;
  const int st = cir::scratch_on_current_device(&ws);
  if (st) return st;
  return cir::launch_attention(q, k_pool, v_pool, page_table, seq_lens, out, ws, kScratchBytes, batch, 1, num_heads,
                               num_kv_heads, head_dim, page_size, max_pages, scale, kv_dtype, stream,
                               cir::QkvIn{nullptr, 0, nullptr, nullptr}, true, true);
}
