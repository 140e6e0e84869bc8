// Large-m GEMM (qgemm_xl_kernel, m > 32): a workgroup of W wavefronts owns a contiguous run
// of up to W/H pairs of 16-column weight tiles (gate/up pairs for SwiGLU), 16*MT activation
// rows and one k-split; H wavefronts share a pair, MT/H row tiles each.
//   * Activations: a quad (128 columns of k) at a time to LDS by buffer DMA, NS - 1 quads ahead
//     of the one being multiplied, NS stages, each an array of its own (the compiler then lets
//     the reads of one run while DMA fills the others), one barrier per quad.
//   * Weights: each wavefront loads its pair's codes and scales straight to registers, NS quads
//     ahead, and converts the fragments of block j + 1 between the MFMAs of block j (of the
//     next quad's block 0 during block 3), so no conversion stands between barrier and MFMA.
//   * The order of instructions is pinned (see `sweep`): a step issues its two MFMAs, then the
//     scale FMAs of the step before, and reads the activations of the step seven later.  Left
//     alone the compiler puts each MFMA's FMAs right behind it with eight wait states between,
//     and nothing overlaps within a wavefront.
//   * Two wavefronts per SIMD: one issues a VALU instruction every four cycles at most, two
//     together one every two, and the MFMAs of one run under the FMAs of the other.
//   * Exact weights and per-block fp32 scales as in the m <= 32 kernel, the quads and blocks of
//     a split in order, so a split's partials are the same bits at every m > 16.
// What bounds it, by the launches' counters: over many workgroups the issue of VALU and MFMA
// instructions, which overlap too little (Q4_0 28672 x 4096 + SwiGLU at m = 2048: VALU 70% of
// the cycles, matrix cores 40%, both at once 15%, so 95% busy; 6.9 VALU instructions an MFMA,
// most of them the scale FMAs and conversions).  In one round at m <= 128 latency and an uneven
// share: Q8_0 37888 x 3584 at 128 VALU 48%, matrix cores 22%, both 8%, neither 38%; the L1
// refuses requests 31% of the cycles, HBM gives each byte once (152 MB in 62 us), and of ten
// wavefronts two SIMDs hold three and two hold two.  Measured against the kernels before (us;
// the compiler's order, the row formats' activation sums repeated by every wavefront, fixed
// 128-column groups or runs on four wavefronts; the builds timed in turn): Q4_0 28672 x 4096 +
// SwiGLU at m = 77 65.4 -> 40.5, 128 64.7 -> 48.6, 2048 540-548 -> 545-548 (882 TFLOP/s); Q8_0
// 37888 x 3584 at 77 67.4 -> 49.7, 128 66.9 -> 58.1, 2048 715-729 -> 692-704; int4 rows
// 28672 x 4096 at 77 40.1 -> 31.4, 2048 804 -> 459-469; Q4_0 4096 x 14336 and store at 77 32.7
// -> 24.3.
// EPI 0: fp32 split-k partials part[split][m][n]; EPI 1: SwiGLU over interleaved gate/up tiles
// (one split), out[m][N/2] in type TO; EPI 2: greedy-head candidates (one split), the best
// column of each pair and row: value in part, index in act (as int), at [m][run * W/H + pair].
#include "qgemm.hpp"

namespace cir {
namespace {

template <int FMT>
inline constexpr int kXlLB = layout_fmt(FMT) == CIR_Q4_0 ? 1 : 2;  // 16-byte loads of codes per lane, tile and quad

template <int FMT, int MT, int H, int W, int EPI, typename TO>
__global__ __launch_bounds__(64 * W, 2) void qgemm_xl_kernel(const f16* __restrict__ x, int ldx,
                                                          const uint8_t* __restrict__ wq,
                                                          const uint16_t* __restrict__ wd, float* __restrict__ part,
                                                          TO* __restrict__ act, int M, int N, int K, int nq) {
  constexpr int LB = kXlLB<FMT>;
  constexpr bool kRow = is_row_fmt(FMT);
  constexpr int NA = MT / H;                 // row tiles of a wavefront
  constexpr int NS = H == 2 ? 3 : 2;         // stages of activations, and of weights in registers
  constexpr int NI = (4 * MT + W - 1) / W;   // its DMA instructions per quad
  constexpr int RL = 2 * (LB + (kRow ? 0 : 1));  // its weight loads per quad
  constexpr int SR = (MT + W - 1) / W;       // row tiles whose sums it takes (row formats)
  static_assert(MT % H == 0 && (H == 1 || H == 2), "whole row shares");
  static_assert(NI + 2 * RL < 64, "vmcnt range");
  __shared__ __align__(16) uint8_t sa[16 * MT * 256];
  __shared__ __align__(16) uint8_t sb[16 * MT * 256];
  __shared__ __align__(16) uint8_t sc[NS == 3 ? 16 * MT * 256 : 16];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63, li = lane & 15, lg = lane >> 4;
  const int KQ = K / 128, NTILES = (N + 15) / 16, NP = (NTILES + 1) / 2;
  const int p0 = (int)((long)blockIdx.x * NP / gridDim.x);
  const int cnt = (int)((long)(blockIdx.x + 1) * NP / gridDim.x) - p0;  // 1 .. W/H pairs (host-checked)
  const int split = blockIdx.y, q0 = split * nq;
  const int nqs = min(nq, KQ - q0);  // quads of this split (the last may hold fewer)
  const int m0 = blockIdx.z * 16 * MT;
  const int pw = wave / H;
  const bool own = pw < cnt;
  const int nt = 2 * (p0 + min(pw, cnt - 1));  // this wavefront's first tile
  const int a0 = (wave % H) * NA;               // and row tile

  // Activation DMA: instruction i (0 .. 4*MT-1) fills KiB i of a stage, rows 4i + lane/16; 16-byte chunk g of row r sits
  // in slot g ^ (r & 15), so the 16 rows of a fragment read hit 16 different slots.  Every wavefront issues NI (past the
  // last: the last again, the same bytes to the same place), so the waits can count.  Rows past M re-read row M-1.
  // Offsets are 32 bits from the row block's first row and, for the weights, from the run's first tile (xl_fits).
  const int mrows = min(16 * MT, M - m0);
  const rsrc_t rx = make_rsrc(x + (size_t)m0 * ldx, (uint32_t)mrows * (uint32_t)ldx * 2u);
  uint32_t xoff[NI];
#pragma unroll
  for (int u = 0; u < NI; ++u) {
    const int r = 4 * min(wave * NI + u, 4 * MT - 1) + (lane >> 4);
    xoff[u] = (uint32_t)min(r, mrows - 1) * (uint32_t)ldx * 2u + 16u * ((lane & 15) ^ (r & 15));
  }
  auto dma = [&](uint8_t* st, int i) __attribute__((always_inline)) {
    const uint32_t off = 256u * (uint32_t)__builtin_amdgcn_readfirstlane(q0 + min(i, nqs - 1));
#pragma unroll
    for (int u = 0; u < NI; ++u) buf16_to_lds(rx, st + min(wave * NI + u, 4 * MT - 1) * 1024, xoff[u], off);
  };

  // Weight loads of quad i (clamped to the last) into ring slot i % NS.
  const int run_tiles = min(2 * cnt, NTILES - 2 * p0);
  const size_t tile0 = (size_t)(2 * p0) * KQ;
  const rsrc_t rw = make_rsrc(wq + tile0 * 1024 * LB, (uint32_t)run_tiles * KQ * 1024u * LB);
  const rsrc_t rd = make_rsrc(kRow ? wd : wd + tile0 * 64, kRow ? 0u : (uint32_t)run_tiles * KQ * 128u);
  const uint32_t vw = (uint32_t)lane * 16u * LB, vd = (uint32_t)li * 8u;
  uint32_t tb[2];
#pragma unroll
  for (int b = 0; b < 2; ++b) tb[b] = (uint32_t)(min(nt + b, NTILES - 1) - 2 * p0) * KQ + q0;
  struct Raw {
    uint4 w[2][LB];
    uint2 d[2];
  };
  Raw raw[NS];
  auto load_w = [&](Raw& o, int i) __attribute__((always_inline)) {
    const uint32_t q = (uint32_t)__builtin_amdgcn_readfirstlane(min(i, nqs - 1));
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int c = 0; c < LB; ++c) o.w[b][c] = buf16(rw, vw + 16u * c, (tb[b] + q) * 1024u * LB);
      if constexpr (!kRow) o.d[b] = buf8(rd, vd, (tb[b] + q) * 128u);
    }
  };

  f16x8 wb[2][2];  // [block parity][tile]: converted fragments
  float dj[2][2];
  auto convert = [&](const Raw& o, int j, int b) __attribute__((always_inline)) {
    if constexpr (layout_fmt(FMT) == CIR_Q4_0) {
      const uint4 v = o.w[b][0];
      wb[j & 1][b] = dq_q4((j == 0) ? v.x : (j == 1) ? v.y : (j == 2) ? v.z : v.w);
    } else {
      const uint4 v = o.w[b][j >> 1];
      wb[j & 1][b] = dq_q8((j & 1) ? v.z : v.x, (j & 1) ? v.w : v.y);
    }
    if constexpr (!kRow) {
      const uint32_t dw = (j < 2) ? o.d[b].x : o.d[b].y;
      dj[j & 1][b] = as_f32_value(
          static_cast<float>(__builtin_bit_cast(f16, (uint16_t)((j & 1) ? (dw >> 16) : (dw & 0xFFFFu)))));
    }
  };

  f32x4 acc[NA][2], c[2][2], sx[SR];
#pragma unroll
  for (int a = 0; a < SR; ++a) sx[a] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < NA; ++a) acc[a][0] = acc[a][1] = f32x4{0.f, 0.f, 0.f, 0.f};
  int xo[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) xo[j] = a0 * 4096 + li * 256 + (((4 * j + lg) ^ li) << 4);

  // One quad from stage `st`: step t = (block t / NA, row tile t % NA).  `cur` holds its codes, `next` the next quad's.
  constexpr int T = 4 * NA, R = 8;  // steps; activation fragments in registers (LDS latency ~240 cycles)
  auto sweep = [&](const uint8_t* st, const Raw& cur, const Raw& next) __attribute__((always_inline)) {
    f16x8 xr[R];
    auto read_x = [&](int t) __attribute__((always_inline)) {
      xr[t % R] = *reinterpret_cast<const f16x8*>(st + (t % NA) * 4096 + xo[t / NA]);
    };
    auto fmas = [&](int t) __attribute__((always_inline)) {
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          acc[t % NA][b][r] = fmaf(dj[(t / NA) & 1][b], c[t & 1][b][r], acc[t % NA][b][r]);
    };
#pragma unroll
    for (int t = 0; t < R - 1; ++t)
      if (t < T) read_x(t);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int j = t / NA, a = t % NA;
      if (t + R - 1 < T) read_x(t + R - 1);
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        if constexpr (kRow) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xr[t % R], wb[j & 1][b], acc[a][b], 0, 0, 0);
        else c[t & 1][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(xr[t % R], wb[j & 1][b], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!kRow) {
        if (t > 0) fmas(t - 1);
      }
      // fragments of the next block, one tile in each of two steps (the block before used that set; its last FMAs, which
      // read its scales, went out in step a = 0)
      if (a == 1 || (a == 2 && NA > 2)) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
          if (NA == 2 || b == a - 1) j < 3 ? convert(cur, j + 1, b) : convert(next, 0, b);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (!kRow) fmas(T - 1);
  };
  static_assert(NA >= 2, "a block's last scale FMAs go out in the next block's first step, before its set is rewritten");
  // Row formats: the activation sums of row tiles wave * SR .. (the MFMA against ones leaves each row's sum in the
  // accumulators' layout).
  auto row_sum = [&](const uint8_t* st) __attribute__((always_inline)) {
    const f16x8 ones = {1, 1, 1, 1, 1, 1, 1, 1};
#pragma unroll
    for (int a = 0; a < SR; ++a)
      if (wave * SR + a < MT) {
#pragma unroll
        for (int j = 0; j < 4; ++j)
          sx[a] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
              *reinterpret_cast<const f16x8*>(st + (wave * SR + a - a0) * 4096 + xo[j]), ones, sx[a], 0, 0, 0);
      }
  };

  // Wait until at most N of this wavefront's loads are in flight, then for every wavefront (the builtin, so the
  // compiler counts it and adds no wait of its own before the reads).
  auto arrive = [&]<int V>() __attribute__((always_inline)) {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((V & 15) | 0x70 | ((V >> 4) << 14));  // vmcnt(V), lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto pin = []() __attribute__((always_inline)) { __builtin_amdgcn_sched_barrier(0); };
  auto multiply = [&]<int S>(const uint8_t* cur) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    if (own) sweep(cur, raw[S], raw[(S + 1) % NS]);
    if constexpr (kRow) row_sum(cur);
  };
  // Quad i: its activations are in `cur`; quad i + NS - 1's go to `far`, which quad i - 1 has left; quad i + NS's weights
  // replace quad i's.  Newer than quad i's activations: NS - 1 quads' weight loads and NS - 2 quads' DMA.  A load that
  // nothing reads would be dropped, and a wait that counts it would let the DMA it is there for stay in flight: `hold`
  // reads the ring slots that no quad does, so whatever the compiler peels or unrolls, each counted load is issued.
  constexpr int kNewer = (NS - 2) * NI + (NS - 1) * RL;
  auto step = [&]<int S>(const uint8_t* cur, uint8_t* far, int i) __attribute__((always_inline)) {
    arrive.template operator()<kNewer>();
    dma(far, i + NS - 1);
    multiply.template operator()<S>(cur);
    load_w(raw[S], i + NS);
    pin();
  };
  auto hold = [](const Raw& o) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int c = 0; c < LB; ++c) asm volatile("" ::"v"(o.w[b][c].x), "v"(o.w[b][c].y), "v"(o.w[b][c].z), "v"(o.w[b][c].w));
      if constexpr (!kRow) asm volatile("" ::"v"(o.d[b].x), "v"(o.d[b].y));
    }
  };
  load_w(raw[0], 0);
  pin();
  dma(sa, 0);
  pin();
  load_w(raw[1], 1);
  pin();
  if constexpr (NS == 3) {
    dma(sb, 1);
    pin();
    load_w(raw[2], 2);
    pin();
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) convert(raw[0], 0, b);
  int i = 0;
  // Rounds of NS whole steps (past the last quad they load and DMA it again, which nothing uses), then the quads left,
  // all on their way: no condition stands around an issue in the loop, else the compiler counts waits for paths that
  // skip it and drains the DMA before every read.  Without a round nothing carries the loads issued above (the compiler
  // moves some into the loop's way in), so the waits of the quads left count none of them.
  auto rest = [&]<int V>(int i) __attribute__((always_inline)) {
    if (i > 0) arrive.template operator()<V>();
    else arrive.template operator()<0>();
  };
  if constexpr (NS == 3) {
#pragma nounroll
    for (; i + 3 <= nqs; i += 3) {  // uniform
      step.template operator()<0>(sa, sc, i);
      step.template operator()<1>(sb, sa, i + 1);
      step.template operator()<2>(sc, sb, i + 2);
    }
    if (i < nqs) {
      rest.template operator()<kNewer>(i);
      multiply.template operator()<0>(sa);
      if (i + 1 < nqs) {
        rest.template operator()<RL>(i);  // newer: the weights of quad i + 2
        multiply.template operator()<1>(sb);
      } else {
        hold(raw[1]);
      }
    } else {
      hold(raw[0]);
      hold(raw[1]);
    }
    hold(raw[2]);
  } else {
#pragma nounroll
    for (; i + 2 <= nqs; i += 2) {
      step.template operator()<0>(sa, sb, i);
      step.template operator()<1>(sb, sa, i + 1);
    }
    if (i < nqs) {
      rest.template operator()<kNewer>(i);
      multiply.template operator()<0>(sa);
    } else {
      hold(raw[0]);
    }
    hold(raw[1]);
  }
  if constexpr (kAccScale<FMT> != 1.f) {
#pragma unroll
    for (int a = 0; a < NA; ++a) acc[a][0] *= kAccScale<FMT>, acc[a][1] *= kAccScale<FMT>;
  }
  if constexpr (kRow) {  // w = (c - zp) * s, so y = s * (sum x c + (c0 - zp) * sum x)
    float* sums = reinterpret_cast<float*>(sa);
    arrive.template operator()<0>();  // every read and DMA of sa is over
#pragma unroll
    for (int a = 0; a < SR; ++a)
      if (wave * SR + a < MT && li == 0) *reinterpret_cast<f32x4*>(sums + (wave * SR + a) * 16 + 4 * lg) = sx[a];
    __syncthreads();
    const float* rscale = reinterpret_cast<const float*>(wd);
    const float* roff = rscale + (size_t)NTILES * 16;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int n = min(nt + b, NTILES - 1) * 16 + li;
      const float s = rscale[n], o = roff[n];
#pragma unroll
      for (int a = 0; a < NA; ++a) {
        const f32x4 rs = *reinterpret_cast<const f32x4*>(sums + (a0 + a) * 16 + 4 * lg);
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[a][b][r] = s * fmaf(o, rs[r], acc[a][b][r]);
      }
    }
  }
  if constexpr (EPI == 2) {
    // The best (value, column) of the pair's 32 columns per row; a wavefront without a pair leaves neutral candidates.
    float* cand_v = part;
    int* cand_i = reinterpret_cast<int*>(act);
    const int WT = gridDim.x * (W / H), at = blockIdx.x * (W / H) + pw;
#pragma unroll
    for (int a = 0; a < NA; ++a)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float bv = -INFINITY;
        int bi = 0x7fffffff;
#pragma unroll
        for (int b = 0; b < 2; ++b) {
          const int n = (nt + b) * 16 + li;
          if (own && nt + b < NTILES && n < N) argmax_better(bv, bi, acc[a][b][r], n);
        }
        // the 16 lanes of this row group (same lg) hold 16 different columns
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) {
          const float ov = __shfl_xor(bv, off, 64);
          const int oi = __shfl_xor(bi, off, 64);
          argmax_better(bv, bi, ov, oi);
        }
        const int m = m0 + 16 * (a0 + a) + 4 * lg + r;
        if (li == 0 && m < M) {
          cand_v[(size_t)m * WT + at] = bv;
          cand_i[(size_t)m * WT + at] = bi;
        }
      }
    return;
  }
  if (!own) return;
  if constexpr (EPI == 1) {
    const int inter = N / 2;
    const int col = (nt >> 1) * 16 + li;
    if (nt + 1 < NTILES && col < inter) {
#pragma unroll
      for (int a = 0; a < NA; ++a)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = m0 + 16 * (a0 + a) + 4 * lg + r;
          const float g = acc[a][0][r], u = acc[a][1][r];
          if (m < M) act[(size_t)m * inter + col] = static_cast<TO>(as_f32_value((g / (1.0f + expf(-g))) * u));
        }
    }
  } else {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const int n = (nt + b) * 16 + li;
      if (nt + b < NTILES && n < N) {
#pragma unroll
        for (int a = 0; a < NA; ++a)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int m = m0 + 16 * (a0 + a) + 4 * lg + r;
            if (m < M) part[((size_t)split * M + m) * N + n] = acc[a][b][r];
          }
      }
    }
  }
}

// The geometry of a launch (us measured on MI355X):
//   * one block of 64, 96 or 128 rows (m <= 128) whose columns one round of workgroups over the 256 CUs holds in runs of
//     at most 5 pairs: such runs, as many as there are CUs (at most one pair each), two wavefronts per pair (H = 2); 10
//     wavefronts where a run holds 5 (a fifth pair split over 8 took 10 us more at Q8_0 gate|up 37888 x 3584, m = 128).
//     96-row blocks: Q4_0 gate|up 28672 x 4096 at m = 77 37.6 against 46.3.
//   * more columns (n > 40960 at one split): four wavefronts per workgroup, each a pair over all rows (H = 1), several
//     workgroups per CU.  A head's logits, 128256 x 4096, with 5 pairs to a workgroup of 10 wavefronts against this: Q4_0
//     m = 33 156 / 93, 64 172 / 108, 128 262 / 191; Q8_0 177 / 132, 187 / 140, 286 / 216; int4 131 / 80, 143 / 95, 213 / 170;
//     Q4_0 SwiGLU 45056 x 4096 at 64 73 / 44.  (57344 x 4096 and 151936 x 1024 alike; at 81920, whose last round of runs
//     is full, 0.75-1.12 times.)  Within one round the runs win: Q4_0 40960 x 4096 at 64 44 against 49.
//   * more than 128 rows in a grid of at most one workgroup per CU: H = 2 in runs of 4 pairs.
//   * more rows in a larger grid: H = 1 over 128 rows, two workgroups per CU: a converted fragment feeds 8 MFMAs instead
//     of 4 (Q4_0 gate|up at m = 2048 522 against 620, int4 rows 443 against 510; while at m = 512 the 192 workgroups of
//     Q4_0 QKV 6144 x 4096 take 44.6 with eight wavefronts, 50.6 with four).
//   * the greedy head (EPI 2), in runs of 4 pairs at any m (the candidates' count): H = 1 past 96 rows as above, at 65-96
//     rows for 8-bit codes past one workgroup per CU, at up to 64 rows past two (Q8_0: one).  H = 2 against H = 1, Q8_0
//     128256 x 4096 at m = 33 172 / 137, 64 174 / 143, 96 207 / 178, 40960 x 4096 at 64 80 / 65; int8 rows 128256 x 4096 at
//     64 137 / 130, 96 193 / 163; Q4_0 at 33 113 / 104, 64 116 / 109.  H = 2 stays for 4-bit codes at 65-96 rows (40960 x
//     4096: Q4_0 72 against 76, int4 62 against 66) and below those counts (Q4_0 28672 x 4096 at 64 39 against 43).
template <int FMT, int EPI, typename TO>
int launch_xl(const f16* x, int ldx, const uint8_t* wq, const uint16_t* wd, float* part, TO* act, int M, int N, int K,
              int splits, hipStream_t s) {
  const int nq = (K / 128 + splits - 1) / splits;
  const int np = ((N + 15) / 16 + 1) / 2, groups = (np + 3) / 4;
  auto go = [&]<int MT, int H, int W>(int runs) {
    const dim3 grid(runs, splits, (M + 16 * MT - 1) / (16 * MT));
    qgemm_xl_kernel<FMT, MT, H, W, EPI, TO><<<grid, 64 * W, 0, s>>>(x, ldx, wq, wd, part, act, M, N, K, nq);
  };
  const bool fill = (long)groups * splits * ((M + 127) / 128) > kCUs;
  if constexpr (EPI == 2) {
    constexpr bool k8 = layout_fmt(FMT) == CIR_Q8_0;
    if (M > 96 && fill) go.template operator()<8, 1, 4>(groups);
    else if (M > 96) go.template operator()<8, 2, 8>(groups);
    else if (M > 64) {
      if constexpr (k8) {
        if (fill) go.template operator()<6, 1, 4>(groups);
      }
      if (!k8 || !fill) go.template operator()<6, 2, 8>(groups);
    } else if (groups > (FMT == CIR_Q8_0 ? 1 : 2) * kCUs) go.template operator()<4, 1, 4>(groups);
    else go.template operator()<4, 2, 8>(groups);
    return 4 * groups;
  } else {
    if (M > 128) {
      if (fill) go.template operator()<8, 1, 4>(groups);
      else go.template operator()<8, 2, 8>(groups);
      return 0;
    }
    const int runs = kCUs / splits < np ? kCUs / splits : np;  // one round, at most one pair each
    auto by_rows = [&]<int H, int W>(int n_runs) {
      if (M <= 64) go.template operator()<4, H, W>(n_runs);
      else if (M <= 96) go.template operator()<6, H, W>(n_runs);
      else go.template operator()<8, H, W>(n_runs);
    };
    if (np <= 4 * runs) by_rows.template operator()<2, 8>(runs);
    else if (np <= 5 * runs) by_rows.template operator()<2, 10>(runs);
    else by_rows.template operator()<1, 4>(groups);
    return 0;
  }
}

}  // namespace

template <int FMT>
void launch_qgemm_xl(const f16* x, int ldx, const uint8_t* wq, const uint16_t* wd, float* part, int M, int N, int K,
                     int splits, hipStream_t s) {
  launch_xl<FMT, 0, float>(x, ldx, wq, wd, part, nullptr, M, N, K, splits, s);
}
template <int FMT>
void launch_qgemm_xl_swiglu(const f16* x, int ldx, const uint8_t* wq, const uint16_t* wd, void* act, int odt, int M,
                            int N, int K, hipStream_t s) {
  if (odt == CIR_F16) launch_xl<FMT, 1, f16>(x, ldx, wq, wd, nullptr, static_cast<f16*>(act), M, N, K, 1, s);
  else launch_xl<FMT, 1, float>(x, ldx, wq, wd, nullptr, static_cast<float*>(act), M, N, K, 1, s);
}
template <int FMT>
int launch_qgemm_xl_argmax(const f16* x, int ldx, const uint8_t* wq, const uint16_t* wd, float* cand_v, int* cand_i,
                           int M, int N, int K, hipStream_t s) {
  return launch_xl<FMT, 2, float>(x, ldx, wq, wd, cand_v, reinterpret_cast<float*>(cand_i), M, N, K, 1, s);
}
#define CIR_XL(F)                                                                                                  \
  template void launch_qgemm_xl<F>(const f16*, int, const uint8_t*, const uint16_t*, float*, int, int, int, int,   \
                                   hipStream_t);                                                                   \
  template void launch_qgemm_xl_swiglu<F>(const f16*, int, const uint8_t*, const uint16_t*, void*, int, int, int,  \
                                          int, hipStream_t);                                                       \
  template int launch_qgemm_xl_argmax<F>(const f16*, int, const uint8_t*, const uint16_t*, float*, int*, int, int, \
                                         int, hipStream_t);
CIR_XL(CIR_Q4_0)
CIR_XL(CIR_Q8_0)
CIR_XL(CIR_I4_ROW)
CIR_XL(CIR_I8_ROW)
#undef CIR_XL

}  // namespace cir
