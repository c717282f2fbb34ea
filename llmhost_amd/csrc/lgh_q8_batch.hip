// Q8_0 head over several tokens for gfx950 (crates/llm-engine/src/
// weights.rs:194-227 with tokens > 1): one pass over the weights per 64 tokens.
//
// The GEMV (lgh_gemv.hip) runs one grid row per token and so moves the whole
// matrix once per token.  Here 16 weight rows x up to 64 tokens share one pass,
// with the block dots on the int8 matrix cores:
//   * A operand (16 rows x 64 elements = one block pair): lane l holds bytes
//     16 g .. 16 g + 15 (g = l / 16) of row l % 16's 64 bytes of the pair --
//     the natural order of the weights, one 128-bit load per lane, no shuffle;
//   * v_mfma_i32_16x16x64_i8 sums over both blocks of the pair, so each block's
//     dot takes the operand with the other block's lanes zeroed (lanes g < 2
//     hold the first block): two MFMAs of 4 passes a pair, what two 16x16x32
//     would take, and every result is one exact block dot;
//   * the terms (f32(dot) * sw) * sa are added in block order within a quad of
//     blocks (weights.rs:206-212), the last product fused into the addition, two
//     quads to a chunk, and the chunks' sums in two sums in turn; rows of more than
//     80 blocks are summed so in groups of 64 blocks.  Relative error (2-norms)
//     against 64 bits, here and of the GEMV's partial sums: K=1536 7.0e-8, 6.9e-8;
//     K=4128 8.1e-8, 8.4e-8; K=8192 8.3e-8, 8.6e-8; K=16384 9.2e-8, 9.4e-8
//     (without the groups 8.4e-8, 9.8e-8 and 1.2e-7 at the last three).
// A wave owns 16 rows and walks them chunk by chunk (4.3 KB of weights); the 8
// waves of a workgroup share the activations, staged in LDS KS blocks at a
// time.  HBM-bound: norm + head, K=1536, N=65536 (107 MB), M = 2 / 16 / 32 / 64:
// 30.9 / 216 / 434 / 882 -> 24.0 / 24.6 / 27.5 / 39.0 us with the image launch
// (~4 us); at 64 tokens the folds (12 VALU operations per MFMA) weigh as much
// as the stream.  Measured against it: weight loads with the streaming hint
// 31.0 us (a load takes 64-byte halves of 16 rows' lines, and the hint lets the
// other half go before the next load asks for it); a K slice per wave with the
// activations in registers 37 us; two or four chunks in flight 24.8-28.5 us;
// without the limit to 128 registers 41 / 47 us at 48 / 64 tokens (34 / 39).
#include <algorithm>

#include "lgh_device.h"
#include "lgh_internal.h"

namespace lgh {

namespace {

struct Q8MmaArgs {
  const int8_t *qs;    // [n][bpr][32], natural order
  const uint16_t *sc;  // f16 scales [n][bpr]
  const uint8_t *ci;   // activation codes image [mt][2 pq][64][16], MmaOrder::kPair
  const float *si;     // activation scales image [mt][pq][16][4]
  float *y;            // [m][n]
  int n, bpr, m, mt, pq;
  int vec4;            // n % 4 == 0 and y 16-byte aligned
};

constexpr int kChunk = 8;   // blocks of a chunk
constexpr int kGroup = 64;  // blocks of a group of chunks
constexpr int kLong = 80;   // rows of more blocks are summed by groups

// Weights of one chunk of 16 rows: four block pairs, two block scales.
struct Q8Chunk {
  uint4 w[kChunk / 2];
  uint16_t s[2];
};

// Requests of the chunk at block kb0: lane l = row l % 16, bytes 16 (l / 16) of
// each pair, and the scales of row l / 4, blocks 2 (l % 4) and the next; blocks
// past the row read 0.
__device__ __forceinline__ void q8_load(__amdgpu_buffer_rsrc_t wr, __amdgpu_buffer_rsrc_t sr, int bpr, int kb0,
                                        Q8Chunk &c) {
  const int lane = threadIdx.x & (kWave - 1), lr = lane & 15, g = lane >> 4;
#pragma unroll
  for (int e = 0; e < 2; e++) {
    const int kb = kb0 + 2 * (lane & 3) + e;
    c.s[e] = buf_load_u16(sr, kb < bpr ? static_cast<uint32_t>((lane >> 2) * bpr + kb) * 2u : kOOB);
  }
#pragma unroll
  for (int p = 0; p < kChunk / 2; p++) {
    const int kb = kb0 + 2 * p;
    c.w[p] = buf_load16(
        wr, kb + (g >> 1) < bpr ? static_cast<uint32_t>(lr * bpr + kb) * 32u + 16u * static_cast<uint32_t>(g) : kOOB);
  }
}

// TT 16-token tiles, W waves, KS blocks of activations in LDS.  LONG: rows of
// more than kLong blocks, whose chunks are summed group by group.
template <int TT, int W, int KS, bool LONG>
__global__ __launch_bounds__(W * kWave) __attribute__((amdgpu_waves_per_eu(4))) void q8_mma_kernel(Q8MmaArgs a) {
  static_assert(KS % kChunk == 0, "whole chunks per stage");
  constexpr int THREADS = W * kWave;
  constexpr int kRow = 16;  // scales of a block in s_sw
  __shared__ __align__(16) uint4 s_b[TT][KS / 2][kWave];
  __shared__ __align__(16) float4 s_sa[TT][KS / 4][16];
  __shared__ __align__(16) float s_sw[W][kChunk * kRow];
  const int tid = threadIdx.x, lane = tid & (kWave - 1), wave = uniform(tid / kWave);
  const int lr = lane & 15, g = lane >> 4;
  const int bpr = a.bpr;
  const int row0 = (static_cast<int>(blockIdx.x) * W + wave) * 16;
  const int rows = uniform(max(0, min(16, a.n - row0)));
  const size_t blk0 = rows > 0 ? static_cast<size_t>(row0) * bpr : 0;
  const auto wr = make_rsrc(a.qs + blk0 * 32, static_cast<uint32_t>(rows * bpr) * 32u);
  const auto sr = make_rsrc(a.sc + blk0, static_cast<uint32_t>(rows * bpr) * 2u);
  const auto cr = make_rsrc(a.ci, static_cast<uint32_t>(a.mt * 2 * a.pq) * 1024u);
  const auto ar = make_rsrc(a.si, static_cast<uint32_t>(a.mt * a.pq) * 256u);

  float acc[2][TT][4];  // sums of every other chunk, in turns
  // LONG: the sums of the groups before; of four token tiles in LDS, where the
  // registers are used up and two workgroups a CU still fit.
  constexpr bool kTotLds = LONG && TT == 4;
  __shared__ float s_tot[kTotLds ? TT * 4 : 1][kTotLds ? THREADS : 1];
  float r_tot[LONG && !kTotLds ? TT : 1][4];
  auto tot = [&](int tt, int v) -> float & {
    if constexpr (kTotLds)
      return s_tot[tt * 4 + v][tid];
    else
      return r_tot[tt][v];
  };
#pragma unroll
  for (int tt = 0; tt < TT; tt++)
#pragma unroll
    for (int v = 0; v < 4; v++) {
      acc[0][tt][v] = acc[1][tt][v] = 0.0f;
      if constexpr (LONG) tot(tt, v) = 0.0f;
    }

  // A stage's activations, every load of a tile before its first LDS write.
  // Pairs and quads past the row's image hold 0: whole chunks are computed, and
  // their weights and scales read 0 too, but 0 * a stale inf would not be 0.
  auto stage = [&](int s0) {
    constexpr int NB = (KS / 2 * kWave + THREADS - 1) / THREADS, NS = (KS / 4 * 16 + THREADS - 1) / THREADS;
#pragma unroll
    for (int tt = 0; tt < TT; tt++) {
      uint4 b[NB];
      float4 f[NS];
#pragma unroll
      for (int u = 0; u < NB; u++) {
        const int i = tid + u * THREADS;
        b[u] = buf_load16(cr, s0 / 2 + i / kWave < 2 * a.pq
                                  ? static_cast<uint32_t>((tt * 2 * a.pq + s0 / 2) * kWave + i) * 16u
                                  : kOOB);
      }
#pragma unroll
      for (int u = 0; u < NS; u++) {
        const int i = tid + u * THREADS;
        f[u] = buf_load_f4(
            ar, s0 / 4 + i / 16 < a.pq ? static_cast<uint32_t>((tt * a.pq + s0 / 4) * 16 + i) * 16u : kOOB);
      }
#pragma unroll
      for (int u = 0; u < NB; u++)
        if (tid + u * THREADS < KS / 2 * kWave) s_b[tt][0][tid + u * THREADS] = b[u];
#pragma unroll
      for (int u = 0; u < NS; u++)
        if (tid + u * THREADS < KS / 4 * 16) s_sa[tt][0][tid + u * THREADS] = f[u];
    }
  };

  // The first chunk's weights go out behind the first stage's activations and
  // are in flight across the barrier.  From there a chunk's registers are
  // refilled as soon as it is done, past the row with nothing: the loop has no
  // branch around its loads, so the compiler counts them.
  Q8Chunk c;
  stage(0);
  q8_load(wr, sr, bpr, 0, c);
  __syncthreads();
  for (int s0 = 0;;) {
    const int sblk = min(KS, bpr - s0);  // blocks of this stage
    for (int kc = 0; kc < sblk; kc += kChunk) {
      float *tsw = s_sw[wave];  // written and read by this wave only, in order
#pragma unroll
      for (int e = 0; e < 2; e++) tsw[(2 * (lane & 3) + e) * kRow + (lane >> 2)] = h2f(c.s[e]);
      float cs[2][TT][4];  // the two quads' sums
#pragma unroll
      for (int tt = 0; tt < TT; tt++)
#pragma unroll
        for (int v = 0; v < 4; v++) cs[0][tt][v] = cs[1][tt][v] = 0.0f;
#pragma unroll
      for (int j = 0; j < kChunk; j++) {
        const bool mine = (g >> 1) == (j & 1);
        const uint4 w = c.w[j / 2];
        const v4i wa = {mine ? static_cast<int>(w.x) : 0, mine ? static_cast<int>(w.y) : 0,
                        mine ? static_cast<int>(w.z) : 0, mine ? static_cast<int>(w.w) : 0};
        const float4 sw = *reinterpret_cast<const float4 *>(&tsw[j * kRow + 4 * g]);
#pragma unroll
        for (int tt = 0; tt < TT; tt++) {
          const v4i wb = *reinterpret_cast<const v4i *>(&s_b[tt][kc / 2 + j / 2][lane]);
          const v4i zero = {0, 0, 0, 0};
          const v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(wa, wb, zero, 0, 0, 0);
          const float sa = reinterpret_cast<const float *>(&s_sa[tt][kc / 4 + j / 4][lr])[j & 3];
          float(&o)[4] = cs[j / 4][tt];
          o[0] = fmaf(static_cast<float>(d[0]) * sw.x, sa, o[0]);
          o[1] = fmaf(static_cast<float>(d[1]) * sw.y, sa, o[1]);
          o[2] = fmaf(static_cast<float>(d[2]) * sw.z, sa, o[2]);
          o[3] = fmaf(static_cast<float>(d[3]) * sw.w, sa, o[3]);
        }
      }
#pragma unroll
      for (int tt = 0; tt < TT; tt++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
          const float t = acc[1][tt][v] + (cs[0][tt][v] + cs[1][tt][v]);
          acc[1][tt][v] = acc[0][tt][v];
          acc[0][tt][v] = t;
        }
      if constexpr (LONG) {
        if ((s0 + kc) % kGroup == kGroup - kChunk) {  // uniform: a group is done
#pragma unroll
          for (int tt = 0; tt < TT; tt++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
              tot(tt, v) += acc[0][tt][v] + acc[1][tt][v];
              acc[0][tt][v] = acc[1][tt][v] = 0.0f;
            }
        }
      }
      q8_load(wr, sr, bpr, s0 + kc + kChunk, c);
    }
    s0 += KS;
    if (s0 >= bpr) break;  // uniform
    __syncthreads();       // every wave is done with the stage
    stage(s0);
    __syncthreads();
  }

  // D layout: token tt * 16 + lr, rows 4 g + v.
#pragma unroll
  for (int tt = 0; tt < TT; tt++) {
    const int t = tt * 16 + lr;
    if (t >= a.m || 4 * g >= rows) continue;
    float *y = a.y + static_cast<size_t>(t) * a.n + row0 + 4 * g;
    float o[4];
#pragma unroll
    for (int v = 0; v < 4; v++) {
      o[v] = acc[0][tt][v] + acc[1][tt][v];
      if constexpr (LONG) o[v] += tot(tt, v);
    }
    if (a.vec4 && 4 * g + 3 < rows) {
      *reinterpret_cast<float4 *>(y) = make_float4(o[0], o[1], o[2], o[3]);
    } else {
#pragma unroll
      for (int v = 0; v < 4; v++)
        if (4 * g + v < rows) y[v] = o[v];
    }
  }
}

template <int TT, int KS>
hipError_t launch_tt(const Q8MmaArgs &a, hipStream_t st) {
  constexpr int W = 8;
  const unsigned wgs = static_cast<unsigned>((a.n + 16 * W - 1) / (16 * W));
  if (a.bpr > kLong)
    hipLaunchKernelGGL((q8_mma_kernel<TT, W, KS, true>), dim3(wgs), dim3(W * kWave), 0, st, a);
  else
    hipLaunchKernelGGL((q8_mma_kernel<TT, W, KS, false>), dim3(wgs), dim3(W * kWave), 0, st, a);
  return hipGetLastError();
}

}  // namespace

// One pass costs about as much as the matrix's stream plus a chain of one load
// round trip per chunk of a row (~1 us each) behind the image launch; a GEMV
// row per token costs its share of the stream each.  So the bytes that the pass
// saves have to be worth the chain: measured crossings at K=1024, N=32003
// (35 MB) between 2 and 3 tokens (13.4 against 13.0 us, 18.7 against 13), at
// K=1536, N=65536 below 2 (30.9 against 24.0 us), at K=2048, N=12000 (26 MB)
// between 4 and 5 (17.5 against 17.9 us, 21.5).  Where the GEMV has a multiple of 8
// workgroups a token (of 8 waves: N < 12288, a multiple of 256), all tokens'
// workgroups of a row group run on one XCD and find its share of a matrix of up
// to 18 MiB in its L2, so that a token costs about half: crossings at N=8192, K=512 /
// 1024 / 1536 / 2048 at 16 / 13 / 9 / 7 tokens (8.2 / 10.6 / 14.0 / 17.2 us), where
// N=8456 has them at 10 / 7 / 6 / 6.  Fewer rows leave most CUs without a workgroup.
// Rows longer than one launch of the GEMV covers stay with its K ranges, whose
// sums are closer to the 64-bit result there.
bool q8_batch_wanted(const lgh_q8 *w, size_t tokens) {
  if (tokens < 2 || w->bpr == 0 || w->k > kQ8GemvMaxK || w->n < 8192) return false;
  const size_t chunks = (w->bpr + kChunk - 1) / kChunk, bytes = w->n * w->bpr * 34;
  const Q4GemvPlan p = plan_q4_gemv(w->n, w->bpr, 1, false);
  const bool in_l2 = p.W == 8 && p.wgs_per_mat % 8 == 0 && bytes <= (size_t{18} << 20);
  const size_t chain = in_l2 ? std::min(32 + 16 * chunks, 96 + 2 * chunks) : 32 + 8 * chunks;
  return (tokens - 1) * bytes >= chain << 20;
}

hipError_t launch_q8_mma(const lgh_q8 *w, const uint8_t *codes, const float *scales, float *y, size_t m,
                         hipStream_t st) {
  if (m == 0 || w->n == 0) return hipSuccess;
  if (m > 64 || w->bpr == 0) return hipErrorInvalidValue;
  const Q8MmaArgs a{w->qs, w->sc, codes, scales, y, static_cast<int>(w->n), static_cast<int>(w->bpr),
                    static_cast<int>(m), static_cast<int>((m + 15) / 16), static_cast<int>((w->bpr + 3) / 4),
                    (w->n % 4 == 0 && (reinterpret_cast<uintptr_t>(y) & 15u) == 0) ? 1 : 0};
  // Activations staged whole up to K = 2048 for one or two token tiles; three
  // and four stage 16 blocks at a time, which leaves room for four workgroups
  // on a CU (64 tokens, K=1536, N=65536: 32 blocks 50.3 us, 16 blocks 40.0).
  switch (a.mt) {
    case 1: return launch_tt<1, 64>(a, st);
    case 2: return launch_tt<2, 64>(a, st);
    case 3: return launch_tt<3, 16>(a, st);
    default: return launch_tt<4, 16>(a, st);
  }
}

}  // namespace lgh
