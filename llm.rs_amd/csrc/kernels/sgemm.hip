// sgemm.hip - skinny GEMM (short prompts, batched decode) for gfx950.
//
// Reference: the Q4/Q8 x Q8_0 block loop of CpuBackend::matmul_transposed
// per activation row (cpu.rs:90-110; kernel_avx2 cpu.rs:888-941):
// y[t][n] = (...((0 + isum_0 s_0) + isum_1 s_1) + ...), s_b = d_w[n,b] * d_a[t,b],
// isum_b the exact int32 dot of the block's weight and activation codes.
// Every output's terms are added in block order, so the results are
// bit-identical to the reference's for the same activation codes.
//
// What bounds it: few rows leave few output tiles (N / 16 x M / 16 of them,
// 256 for a 4096-row projection of up to 16 tokens on 256 CUs), so a wave
// that walks a whole row of blocks alone has neither the bytes in flight nor
// the issue slots to stream the weights.  Only the additions have an order:
// the terms isum_b * s_b do not.  So a workgroup of eight waves takes 16 R
// rows x 16 tokens (R = 1, 2, 4) and a wave the terms of 16 rows and an
// eighth / quarter / half of each round of 64 / R blocks; the terms pass
// through 64 KB of LDS, four blocks of one output per 16-byte chunk, and
// every thread adds its own outputs' terms in block order.  The order thus
// costs one dependent add per block (K / 32 of them) and no hand-over
// between waves.
//
// Per four blocks and 16 x 16 tile: one v_mfma_i32_16x16x32_i8 per block
// gives its exact sums, one v_mfma_f32_16x16x1_4b_f32 every scale product
// d_w * d_a as a single IEEE product (lane 16 b + i supplies row / token i of
// block b; block b's products sit in registers 4 b .. 4 b + 3 in the layout
// of the block sums).  A wave loads the eight blocks of a step from 16 rows as
// they lie in memory, 128 contiguous bytes per row, and turns them through
// its own LDS so that lane (r, g) (r = lane % 16, g = lane / 16) holds block
// g of row r; a 4x4 dword transpose across the lane groups
// (v_permlane32_swap, v_permlane16_swap) then gives lane group g dword g of
// each of four blocks - its MFMA operand (Q4: the nibbles unpacked to q - 8;
// Q8: dwords g and g + 4).  The activation codes are stored in the operand
// order itself (act_offset), 1 KB of consecutive bytes per load.  Loads in
// which neighbouring lanes read different rows bounded the kernel before: the
// L1 serves one line per lane then, and the same kernel with row-strided
// weight and activation loads took 34 us for the 8B gate|up at 16 rows
// against 21.
//
// Workgroups are dealt to the XCDs so that the token tiles of one row set run
// on one XCD back to back: the weights come from HBM about once and the other
// token tiles read them from its L2.
//
// Measured (8B widths, Q4_0, us per launch; before: one wave per 16 rows with
// row-strided loads): 16 rows Q|K|V 12 -> 7.6, O and down in the mean 14.5 -> 9.8
// (5.5 and 14.1); 23 rows Q|K|V 15.1 -> 10.7, O and down 30.5 -> 13.8 (7.6 and 20.0).
// gate|up goes to the wide kernels below (before 35.7, split 21.4, wide 18.6 at 16
// rows).  The rounds' phases (loads, products, LDS, adds) overlap only across the
// two workgroups of a CU.

#include <type_traits>

#include "common.h"
#include "exact_math.h"
#include "gemm_common.h"
#include "gemv_core.h"
#include "../kernel_args.h"

using namespace llmrs;

namespace {

typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int kSgThreads = kSgemmThreads;   // eight waves
constexpr int kSgWaves = kSgThreads / LLMRS_WAVE;
constexpr int kStep = 8;                    // blocks of one wave per round

// In: lane group g holds the four dwords of its block g.  Out: x[j] = dword
// g of block j.  v_permlane32_swap(a, b) exchanges the upper half of a with
// the lower half of b; v_permlane16_swap the odd 16-lane rows of a with the
// even rows of b.
__device__ __forceinline__ void transpose4(unsigned x[4]) {
  auto p = __builtin_amdgcn_permlane32_swap(x[0], x[2], false, false);
  x[0] = p[0];
  x[2] = p[1];
  p = __builtin_amdgcn_permlane32_swap(x[1], x[3], false, false);
  x[1] = p[0];
  x[3] = p[1];
  p = __builtin_amdgcn_permlane16_swap(x[0], x[1], false, false);
  x[0] = p[0];
  x[1] = p[1];
  p = __builtin_amdgcn_permlane16_swap(x[2], x[3], false, false);
  x[2] = p[0];
  x[3] = p[1];
}

// A wave's loads of eight blocks of 16 weight rows: the codes as they lie in
// memory (lanes 8 i .. 8 i + 7 the 128 bytes of row i, or lanes 16 i .. of 256
// bytes for Q8) and the scales of blocks g and 4 + g of row r.
template <int WT>
struct SgWeights {
  static constexpr int WL = WT == WT_Q8H ? 4 : 2;  // 1 KB loads
  u32x4 w[WL];
  unsigned dw[2];                                  // raw
};
// And of 16 tokens: token r's operands and its scales of blocks g and 4 + g.
struct SgTokens {
  u32x4 x[2][2];  // [run of four blocks][half]
  float da[2];
};

// Blocks b0 .. b0 + 7; runs of four past the row end clamped to its last one
// (nb is a multiple of 4), never added; rows clamped to the last row.
template <int WT>
__device__ __forceinline__ void load_weights(SgWeights<WT>& G, const SgemmArgs& a, int b0, int row0, int nb, int lane) {
  constexpr int BCH = WT == WT_Q8H ? 2 : 1;  // 16-byte chunks per block
  constexpr int RCH = kStep * BCH;           // chunks of a row's eight blocks
#pragma unroll
  for (int j = 0; j < SgWeights<WT>::WL; ++j) {
    const int q = LLMRS_WAVE * j + lane, c = q % RCH;
    const int row = min(row0 + q / RCH, a.N - 1), blk = min(b0 + c / BCH, nb - 1);
    G.w[j] = *(const u32x4*)(a.wq + ((size_t)row * nb + blk) * (16 * BCH) + 16 * (c % BCH));
  }
  const size_t wi = (size_t)min(row0 + (lane & 15), a.N - 1) * nb + (lane >> 4);
#pragma unroll
  for (int u = 0; u < 2; ++u) G.dw[u] = load_scale<WT>(a.ws, wi + min(b0 + 4 * u, nb - 4));
}
__device__ __forceinline__ void load_tokens(SgTokens& G, const SgemmArgs& a, int b0, int tile, int nb, int lane) {
#pragma unroll
  for (int u = 0; u < 2; ++u) {
    const int b = min(b0 + 4 * u, nb - 4);
    const u32x4* p = (const u32x4*)(a.xq + (size_t)tile * 16 * a.K + (size_t)b * 512) + lane;
    G.x[u][0] = p[0];
    G.x[u][1] = p[LLMRS_WAVE];
    G.da[u] = a.xd[(size_t)tile * 16 * nb + b * 16 + lane];
  }
}

// The weights of a step through the wave's own LDS (1 KB per load), in which
// the codes change from memory order (row, chunk) to one row per lane: chunk c
// of row i sits at c ^ (i & 7) of its row, so that 16 rows' chunks spread over
// the banks.
template <int WT>
__device__ __forceinline__ void stage_weights(const SgWeights<WT>& G, u32x4* stage, int lane) {
  constexpr int RCH = kStep * (WT == WT_Q8H ? 2 : 1);
#pragma unroll
  for (int j = 0; j < SgWeights<WT>::WL; ++j) {
    const int q = LLMRS_WAVE * j + lane, i = q / RCH, c = q % RCH;
    stage[i * RCH + (c ^ (i & 7))] = G.w[j];
  }
}

// Four blocks' weights as MFMA operands (dwords lo[j], hi[j] of block j) and
// the scale of block g.
struct SgOperands {
  unsigned lo[4], hi[4];
  float dw;
};
template <int WT>
__device__ __forceinline__ void unpack_weights(const SgWeights<WT>& G, const u32x4* stage, int u, int lane,
                                               SgOperands& op) {
  constexpr int BCH = WT == WT_Q8H ? 2 : 1, RCH = kStep * BCH;
  const int r = lane & 15, g = lane >> 4;
  op.dw = wscale<WT>(G.dw[u]);
  const u32x4 w0 = stage[r * RCH + (((4 * u + g) * BCH) ^ (r & 7))];
#pragma unroll
  for (int j = 0; j < 4; ++j) op.lo[j] = w0[j];
  transpose4(op.lo);
  if constexpr (WT == WT_Q8H) {
    const u32x4 w1 = stage[r * RCH + (((4 * u + g) * BCH + 1) ^ (r & 7))];
#pragma unroll
    for (int j = 0; j < 4; ++j) op.hi[j] = w1[j];
    transpose4(op.hi);
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      op.hi[j] = nib_s8((op.lo[j] >> 4) & 0x0F0F0F0Fu);
      op.lo[j] = nib_s8(op.lo[j] & 0x0F0F0F0Fu);
    }
  }
}

// Four blocks' terms isum_b * (d_w d_a) of a 16 x 16 tile, each operation
// rounded as the reference rounds it: t[b][i] is row 4 g + i, token r of block
// b.  Every MFMA is issued before the first result is read.
__device__ __forceinline__ void block_terms(const SgOperands& op, const SgTokens& G, int u, float (&t)[4][4]) {
  const v16f sc = __builtin_amdgcn_mfma_f32_16x16x1f32(op.dw, G.da[u], v16f{}, 0, 0, 0);
  i32x4 isum[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const unsigned b0 = G.x[u][j >> 1][2 * (j & 1)], b1 = G.x[u][j >> 1][2 * (j & 1) + 1];
    const long op_a = (long)((unsigned long long)op.lo[j] | ((unsigned long long)op.hi[j] << 32));
    const long op_b = (long)((unsigned long long)b0 | ((unsigned long long)b1 << 32));
    isum[j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(op_a, op_b, i32x4{0, 0, 0, 0}, 0, 0, 0);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) t[j][i] = (float)isum[j][i] * sc[4 * j + i];
}

// Element 32 run + j of token t's SwiGLU product m (j = lane % 32: a 32-lane
// group holds one Q8_0 block of m): the f32 value (test probes) and its code.
__device__ __forceinline__ void swiglu_out(const SgemmArgs& a, int t, int run, int j, float m) {
  float amax = fabsf(m);
#pragma unroll
  for (int o = 16; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 32));
  const float d = amax / 127.0f;
  const float inv = amax == 0.0f ? 0.0f : 1.0f / d;
  if (t < a.M) {
    const int F = a.N / 2;
    if (a.y) a.y[(size_t)t * a.ldy + 32 * run + j] = m;
    a.yq[act_row(t, F, a.layout) + act_offset(32 * run + j, a.layout)] =
        amax == 0.0f ? (int8_t)0 : (int8_t)q8_code(m, inv);
    if (j == 0) a.yd[act_scale_row(t, F / 32, a.layout) + act_scale_offset(run, a.layout)] = amax == 0.0f ? 0.0f : d;
  }
}

template <int WT, int EPI, int R>
__device__ __forceinline__ void sgemm_impl(const SgemmArgs& a) {
  constexpr int KP = kSgWaves / R;            // waves that share a row tile's blocks
  constexpr int ROUND = KP * kStep;           // blocks per round
  constexpr int QUADS = ROUND / 4;
  constexpr int OUT = R * 256;                // outputs of the workgroup
  constexpr int PER = OUT > kSgThreads ? OUT / kSgThreads : 1;  // per adding thread
  static_assert(EPI != EPI_SILU || R == 4, "SwiGLU: a run of 32 gate and 32 up rows per workgroup");
  // four blocks' terms of output o = 256 rt + 64 i + lane (row 16 rt +
  // 4 (lane / 16) + i, token lane % 16) at s_t[quad * OUT + o]
  __shared__ f32x4 s_t[QUADS * OUT];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4, rt = w % R, kp = w / R;
  const int nb = a.K >> 5, nt = (a.M + 15) >> 4, nrow = (a.N + 16 * R - 1) / (16 * R);
  const int slot = blockIdx.x >> 3, ty = slot % nt, tx = (slot / nt) * 8 + (blockIdx.x & 7);
  if (tx >= nrow) return;
  const int row0 = tx * 16 * R + 16 * rt;

  float acc[PER];
#pragma unroll
  for (int p = 0; p < PER; ++p) acc[p] = 0.0f;
  SgWeights<WT> W;
  SgTokens X;
  load_weights<WT>(W, a, kp * kStep, row0, nb, lane);
  load_tokens(X, a, kp * kStep, ty, nb, lane);
  for (int base = 0; base < nb; base += ROUND) {
    if (base + kp * kStep < nb) {
      u32x4* stage = (u32x4*)&s_t[2 * kp * OUT + rt * 256];  // the place of the wave's own terms
      stage_weights<WT>(W, stage, lane);
      SgOperands op[2];  // both read before the terms take the place
#pragma unroll
      for (int u = 0; u < 2; ++u) unpack_weights<WT>(W, stage, u, lane, op[u]);
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float t[4][4];
        block_terms(op[u], X, u, t);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          s_t[(2 * kp + u) * OUT + rt * 256 + i * 64 + lane] = f32x4{t[0][i], t[1][i], t[2][i], t[3][i]};
      }
    }
    load_weights<WT>(W, a, base + ROUND + kp * kStep, row0, nb, lane);
    load_tokens(X, a, base + ROUND + kp * kStep, ty, nb, lane);
    __syncthreads();
    if (OUT >= kSgThreads || tid < OUT) {  // cpu.rs:930-935, in block order
      const int nq = min(QUADS, (nb - base) >> 2);
      if (nq == QUADS) {
#pragma unroll
        for (int q = 0; q < QUADS; ++q)
#pragma unroll
          for (int p = 0; p < PER; ++p) {
            const f32x4 v = s_t[q * OUT + p * kSgThreads + tid];
            acc[p] = acc[p] + v[0];
            acc[p] = acc[p] + v[1];
            acc[p] = acc[p] + v[2];
            acc[p] = acc[p] + v[3];
          }
      } else {
        for (int q = 0; q < nq; ++q)
#pragma unroll
          for (int p = 0; p < PER; ++p) {
            const f32x4 v = s_t[q * OUT + p * kSgThreads + tid];
            acc[p] = acc[p] + v[0];
            acc[p] = acc[p] + v[1];
            acc[p] = acc[p] + v[2];
            acc[p] = acc[p] + v[3];
          }
      }
    }
    __syncthreads();
  }

  float* s_o = (float*)s_t;
  if constexpr (EPI == EPI_SILU) {
    // outputs tid and tid + 512 of a thread are a gate row and its up row
    // (layer.rs:72-79); m by token into LDS, then Q8_0 of each token's run
    const float gv = acc[0], uv = acc[PER - 1];
    const float mv = (gv / (1.0f + exact_expf(-gv))) * uv;  // glibc expf (exact_math.h)
    s_o[r * 33 + 16 * (tid >> 8) + 4 * g + ((tid >> 6) & 3)] = mv;
    __syncthreads();
    swiglu_out(a, 16 * ty + (tid >> 5), tx, tid & 31, s_o[(tid >> 5) * 33 + (tid & 31)]);
  } else {
    // rows of one token side by side, for whole-line stores
    constexpr int LD = 16 * R + 1;
    if (OUT >= kSgThreads || tid < OUT) {
#pragma unroll
      for (int p = 0; p < PER; ++p) {
        const int o = p * kSgThreads + tid;
        s_o[r * LD + 16 * (o >> 8) + 4 * g + ((o >> 6) & 3)] = acc[p];
      }
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < PER; ++p) {
      const int o = p * kSgThreads + tid, t = 16 * ty + o / (16 * R), n = tx * 16 * R + o % (16 * R);
      if (o < OUT && t < a.M && n < a.N) {
        float v = s_o[(o / (16 * R)) * LD + o % (16 * R)];
        if (EPI == EPI_RESID) v = v + a.res[(size_t)t * a.N + n];  // layer.rs:386,403
        a.y[(size_t)t * a.ldy + n] = v;
      }
    }
  }
}

// ---- wide layers -------------------------------------------------------------
// Where 64-row sets fill the chip (gate|up, the head of a batch), a wave keeps
// 16 rows x 16 TT tokens to itself and adds its terms in block order in
// registers, with no hand-over through LDS.  A workgroup of four waves (64
// rows) streams eight blocks a stage: weights, activation codes (shared by the
// waves) and scales go to LDS by direct loads, two or three stages ahead, so
// that the loads in flight cover the memory's latency without registers; the
// matrix instructions run one product ahead of the arithmetic.  The serial
// chain of a stage (LDS reads, transposes, products, additions: 0.7 us for one
// token tile) bounds it while a SIMD holds one or two waves.
// Measured, split kernel -> wide (us under a kernel trace, about 1 more than
// without): 8B gate|up 16 rows 22.6 -> 20.1 (66 MB: 3.3 TB/s; Q8_0 27.2 -> 23.2), 32
// rows 40.9 -> 29.7 (45.8 -> 32.8), 48 rows 60.4 (tile GEMM 55.1) -> 39.6; 1B gate|up
// 64 rows 25.2 -> 18.1; a 32000-row head of 16 sequences 21.7 -> 18.8.
template <int WT, int TT>
struct WideStage {
  static constexpr int RC = kStep * (WT == WT_Q8H ? 2 : 1);  // 16-byte chunks of a row
  static constexpr int SD = WT == WT_Q4F ? 8 : 4;            // scale dwords of a row (f16: two scales each)
  static constexpr int X = 0;                                // codes [TT][4 KB]
  static constexpr int DA = X + TT * 4096;                   // scales [TT][8 blocks][16 tokens]
  static constexpr int W = DA + TT * 512;                    // codes [64 rows][RC]
  static constexpr int DW = W + 64 * RC * 16;                // scales [64 rows][SD]
  static constexpr int BYTES = DW + 64 * SD * 4;
  static constexpr int LOADS = TT + 1 + RC / 4 + SD / 4;     // per wave
  static constexpr int N = WT == WT_Q8H || TT == 3 ? 3 : 4;  // buffers
  static_assert(N * BYTES <= 80 * 1024, "two workgroups per CU");
};

template <int WT, int EPI, int TT>
__device__ __forceinline__ void wide_impl(const SgemmArgs& a, uint8_t* lds) {
  typedef WideStage<WT, TT> S;
  constexpr int BCH = WT == WT_Q8H ? 2 : 1, RC = S::RC, SD = S::SD;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int nb = a.K >> 5, nst = (nb + kStep - 1) / kStep;
  const int nt = (a.M + 16 * TT - 1) / (16 * TT), nrow = (a.N + 63) / 64;
  const int slot = blockIdx.x >> 3, ty = slot % nt, tx = (slot / nt) * 8 + (blockIdx.x & 7);
  if (tx >= nrow) return;
  const int tile0 = ty * TT, tiles = (a.M + 15) >> 4, n0 = tx * 64;

  // Stage st into its buffer.  Rows past N and token tiles past M are the last
  // one again, blocks past the row's end (nb is a multiple of 4) a valid run;
  // none of them is added or stored.
  const uint8_t* wbase = a.wq + (size_t)n0 * nb * (16 * BCH);
  const uint8_t* dbase = (const uint8_t*)a.ws + (size_t)n0 * nb * (SD / 2);
  unsigned woff[RC / 4], doff[SD / 4];  // of the lane's chunk c of row i, at c ^ (i & 7), and its scales
  int wblk[RC / 4], dblk[SD / 4];       // their first block in a stage
#pragma unroll
  for (int j = 0; j < RC / 4; ++j) {
    const int p = 64 * j + lane, i = p / RC, c = (p % RC) ^ (i & 7);
    woff[j] = (unsigned)(min(n0 + 16 * w + i, a.N - 1) - n0) * (unsigned)(nb * 16 * BCH) + 16 * c;
    wblk[j] = c / BCH;
  }
#pragma unroll
  for (int j = 0; j < SD / 4; ++j) {
    const int p = 64 * j + lane;
    doff[j] = (unsigned)(min(n0 + 16 * w + p / SD, a.N - 1) - n0) * (unsigned)(nb * SD / 2) + 4 * (p % SD);
    dblk[j] = (p % SD) * (8 / SD);
  }
  constexpr int DV = (TT + 1) / 2;  // waves that cover the 32 TT chunks of d_a; the others repeat them
  const int dq = 64 * (w % DV) + lane;
  auto load_stage = [&](int st) {
    uint8_t* base = lds + (st % S::N) * S::BYTES;
    const int b0 = st * kStep;
    auto load = [&](bool part) {
#pragma unroll
      for (int t = 0; t < TT; ++t) {
        const size_t tile = min(tile0 + t, tiles - 1);
        load_lds16(a.xq + (tile * 16 * a.K + (size_t)b0 * 512) + (unsigned)(16 * (part ? tid & 127 : tid)),
                   base + S::X + t * 4096 + 1024 * w);
      }
      if (dq / 32 < TT) {
        const size_t tile = min(tile0 + dq / 32, tiles - 1);
        load_lds16(a.xd + (size_t)b0 * 16 + tile * 16 * nb + 4 * (dq & (part ? 15 : 31)),
                   base + S::DA + 1024 * (w % DV));
      }
#pragma unroll
      for (int j = 0; j < RC / 4; ++j) {
        const int back = part ? max(b0 + wblk[j] - (nb - 1), 0) : 0;
        load_lds16(wbase + (size_t)b0 * (16 * BCH) + (woff[j] - (unsigned)(16 * BCH * back)),
                   base + S::W + (16 * w * RC + 64 * j) * 16);
      }
#pragma unroll
      for (int j = 0; j < SD / 4; ++j) {
        const int back = part ? max(b0 + dblk[j] - (nb - 8 / SD), 0) : 0;
        load_lds4(dbase + (size_t)b0 * (SD / 2) + (doff[j] - (unsigned)(SD / 2 * back)),
                  base + S::DW + (16 * w * SD + 64 * j) * 4);
      }
    };
    if (b0 + kStep <= nb) load(false);
    else load(true);
  };

  float acc[TT][4];
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[t][i] = 0.0f;

  // The first 4 NU blocks of a stage: products q = TT u + t, token tile t of
  // blocks 4 u .. 4 u + 3.  The matrix instructions of product q + 1 are issued
  // before the arithmetic of q, and its operands read another one before.
  auto compute = [&](const uint8_t* base, auto nu) {
    constexpr int NU = decltype(nu)::value, Q = NU * TT;
    const u32x4* sw = (const u32x4*)(base + S::W) + (16 * w + r) * RC;
    const uint8_t* sd = base + S::DW + (16 * w + r) * SD * 4;
    SgOperands op[NU];
    SgTokens X[3];
    auto tokens = [&](int q) {
      const u32x4* sx = (const u32x4*)(base + S::X + (q % TT) * 4096 + (q / TT) * 2048);
      X[q % 3].x[0][0] = sx[lane];
      X[q % 3].x[0][1] = sx[64 + lane];
      X[q % 3].da[0] = ((const float*)(base + S::DA + (q % TT) * 512))[64 * (q / TT) + lane];
    };
    tokens(0);
    if (Q > 1) tokens(1);
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const u32x4 w0 = sw[((4 * u + g) * BCH) ^ (r & 7)];
#pragma unroll
      for (int j = 0; j < 4; ++j) op[u].lo[j] = w0[j];
      transpose4(op[u].lo);
      if constexpr (WT == WT_Q8H) {
        const u32x4 w1 = sw[((4 * u + g) * BCH + 1) ^ (r & 7)];
#pragma unroll
        for (int j = 0; j < 4; ++j) op[u].hi[j] = w1[j];
        transpose4(op[u].hi);
      } else {  // 16 (q - 8) in a byte's upper half (gemm_common.h)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          op[u].hi[j] = (op[u].lo[j] & 0xF0F0F0F0u) ^ 0x80808080u;
          op[u].lo[j] = ((op[u].lo[j] << 4) & 0xF0F0F0F0u) ^ 0x80808080u;
        }
      }
      op[u].dw = wscale<WT>(WT == WT_Q4F ? ((const unsigned*)sd)[4 * u + g] : ((const uint16_t*)sd)[4 * u + g]);
    }
    v16f sc[2];
    i32x4 isum[2][4];
    auto issue = [&](int q) {
      const SgTokens& x = X[q % 3];
      const SgOperands& o = op[q / TT];
      sc[q % 2] = __builtin_amdgcn_mfma_f32_16x16x1f32(o.dw, x.da[0], v16f{}, 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const long oa = (long)((unsigned long long)o.lo[j] | ((unsigned long long)o.hi[j] << 32));
        const long ob = (long)((unsigned long long)x.x[0][j >> 1][2 * (j & 1)] |
                               ((unsigned long long)x.x[0][j >> 1][2 * (j & 1) + 1] << 32));
        isum[q % 2][j] = __builtin_amdgcn_mfma_i32_16x16x32_i8(oa, ob, i32x4{0, 0, 0, 0}, 0, 0, 0);
      }
      pin(sc[q % 2]);
#pragma unroll
      for (int j = 0; j < 4; ++j) pin(isum[q % 2][j]);
    };
    issue(0);
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      if (q + 2 < Q) tokens(q + 2);
      if (q + 1 < Q) {
        pin(X[(q + 1) % 3].da[0]);
        pin(X[(q + 1) % 3].x[0][0]);
        pin(X[(q + 1) % 3].x[0][1]);
        issue(q + 1);
      }
      __builtin_amdgcn_sched_barrier(0);
      float (&s)[4] = acc[q % TT];
      pin(sc[q % 2]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        pin(isum[q % 2][j]);
#pragma unroll
        for (int i = 0; i < 4; ++i) s[i] = s[i] + (float)isum[q % 2][j][i] * sc[q % 2][4 * j + i];  // cpu.rs:930-935
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) pin(s[i]);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

  for (int st = 0; st < S::N - 1 && st < nst; ++st) load_stage(st);
  for (int st = 0; st < nst; ++st) {
    // This wave's loads of stage st, then everyone's; the barrier also ends the
    // reads of stage st - 1, whose buffer the next loads take.
    if (st + S::N - 1 <= nst) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S::N - 2) * S::LOADS) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (st + S::N - 1 < nst) load_stage(st + S::N - 1);
    const uint8_t* base = lds + (st % S::N) * S::BYTES;
    if ((st + 1) * kStep <= nb) compute(base, std::integral_constant<int, 2>{});
    else compute(base, std::integral_constant<int, 1>{});
  }
  if (WT != WT_Q8H) {  // the Q4 codes were 16 times theirs
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int i = 0; i < 4; ++i) acc[t][i] = acc[t][i] * 0.0625f;
  }

  // token t's 64 rows side by side
  constexpr int LD = 65;
  float* s_o = (float*)lds;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) s_o[(16 * t + r) * LD + 16 * w + 4 * g + i] = acc[t][i];
  __syncthreads();
  bool redo = false;  // this lane met a total that is not finite
  if constexpr (EPI == EPI_SILU) {
    // 32 gate rows, then their up rows (layer.rs:72-79)
#pragma unroll
    for (int p = 0; p < 2 * TT; ++p) {
      const int t = 8 * p + (tid >> 5), j = tid & 31;
      const float gv = s_o[t * LD + j], uv = s_o[t * LD + 32 + j];
      if (WT != WT_Q8H) redo |= !is_finite(gv) || !is_finite(uv);
      const float mv = (gv / (1.0f + exact_expf(-gv))) * uv;  // glibc expf (exact_math.h)
      swiglu_out(a, 16 * tile0 + t, tx, j, mv);
    }
  } else {
#pragma unroll
    for (int p = 0; p < 4 * TT; ++p) {
      const int lt = 4 * p + w, t = 16 * tile0 + lt, n = n0 + lane;
      if (t < a.M && n < a.N) {
        float v = s_o[lt * LD + lane];
        const bool ok = WT == WT_Q8H || is_finite(v);
        redo |= !ok;
        if (EPI == EPI_RESID && ok) v = v + a.res[(size_t)t * a.N + n];  // layer.rs:386,403
        if (EPI != EPI_RESID || ok) a.y[(size_t)t * a.ldy + n] = v;     // may be the residual's place
      }
    }
  }
  if constexpr (WT != WT_Q8H) {
    // Those outputs again by the plain block loop (gemm_common.h).  The
    // arguments are read anew, so that the loops above need not hold them.
    if (__any(redo)) {
      const SgemmArgs* ka = (const SgemmArgs*)__builtin_amdgcn_kernarg_segment_ptr();
      asm volatile("" : "+s"(ka));
#pragma unroll 1
      for (int p = 0; p < (EPI == EPI_SILU ? 2 : 4) * TT; ++p) {
        if constexpr (EPI == EPI_SILU) {
          const int lt = 8 * p + (tid >> 5), j = tid & 31, t = 16 * tile0 + lt;
          float gv = s_o[lt * LD + j], uv = s_o[lt * LD + 32 + j];
          if (t < ka->M && !is_finite(gv)) gv = q4_block_loop<WT, kActMfma>(*ka, t, n0 + j);
          if (t < ka->M && !is_finite(uv)) uv = q4_block_loop<WT, kActMfma>(*ka, t, n0 + 32 + j);
          swiglu_out(*ka, t, tx, j, (gv / (1.0f + exact_expf(-gv))) * uv);
        } else {
          const int lt = 4 * p + w, t = 16 * tile0 + lt, n = n0 + lane;
          if (t < ka->M && n < ka->N && !is_finite(s_o[lt * LD + lane])) {
            float v = q4_block_loop<WT, kActMfma>(*ka, t, n);
            if (EPI == EPI_RESID) v = v + ka->res[(size_t)t * ka->N + n];
            ka->y[(size_t)t * ka->ldy + n] = v;
          }
        }
      }
    }
  }
}

}  // namespace

// Kernels: sgemm_<weights>_<epilogue>_r<row tiles per workgroup>.
#define LLMRS_SGEMM(name, WT, EPI, R) \
  extern "C" __global__ __launch_bounds__(kSgThreads, 4) void name(SgemmArgs a) { sgemm_impl<WT, EPI, R>(a); }
#define LLMRS_SGEMM_WT(tag, WT)                      \
  LLMRS_SGEMM(sgemm_##tag##_store_r1, WT, EPI_STORE, 1) \
  LLMRS_SGEMM(sgemm_##tag##_store_r2, WT, EPI_STORE, 2) \
  LLMRS_SGEMM(sgemm_##tag##_store_r4, WT, EPI_STORE, 4) \
  LLMRS_SGEMM(sgemm_##tag##_resid_r1, WT, EPI_RESID, 1) \
  LLMRS_SGEMM(sgemm_##tag##_resid_r2, WT, EPI_RESID, 2) \
  LLMRS_SGEMM(sgemm_##tag##_resid_r4, WT, EPI_RESID, 4) \
  LLMRS_SGEMM(sgemm_##tag##_silu_r4, WT, EPI_SILU, 4)
LLMRS_SGEMM_WT(q4h, WT_Q4H)
LLMRS_SGEMM_WT(q4f, WT_Q4F)
LLMRS_SGEMM_WT(q8h, WT_Q8H)

// Kernels: sgemm_<weights>_<epilogue>_w<token tiles per workgroup>.
#define LLMRS_WIDE(name, WT, EPI, TT)                                                  \
  extern "C" __global__ __launch_bounds__(kWideThreads, 2) void name(SgemmArgs a) {    \
    __shared__ __align__(16) uint8_t wide_lds[WideStage<WT, TT>::N * WideStage<WT, TT>::BYTES]; \
    wide_impl<WT, EPI, TT>(a, wide_lds);                                               \
  }
#define LLMRS_WIDE_TT(tag, WT, TT)                            \
  LLMRS_WIDE(sgemm_##tag##_store_w##TT, WT, EPI_STORE, TT)    \
  LLMRS_WIDE(sgemm_##tag##_resid_w##TT, WT, EPI_RESID, TT)    \
  LLMRS_WIDE(sgemm_##tag##_silu_w##TT, WT, EPI_SILU, TT)
LLMRS_WIDE_TT(q4h, WT_Q4H, 1)
LLMRS_WIDE_TT(q4h, WT_Q4H, 2)
LLMRS_WIDE_TT(q4h, WT_Q4H, 3)
LLMRS_WIDE_TT(q4f, WT_Q4F, 1)
LLMRS_WIDE_TT(q4f, WT_Q4F, 2)
LLMRS_WIDE_TT(q4f, WT_Q4F, 3)
LLMRS_WIDE_TT(q8h, WT_Q8H, 1)
LLMRS_WIDE_TT(q8h, WT_Q8H, 2)
