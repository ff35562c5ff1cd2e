// prefill.hip - batched prompt processing (prefill) for gfx950.
//
// Reference: LlamaModel::forward over a chunk of M tokens (model.rs:17-49,
// layer.rs:373-406; the prompt step of main.rs:134-190).  The reference's
// M > 1 GEMM quantises every activation row to Q8_0 and runs the Q4 x Q8
// block loop per output element (cpu.rs:90-110, kernel_avx2 cpu.rs:888-941):
//   y[t][r] = (...((0 + isum_0 * s_0) + isum_1 * s_1) + ...),  s_b = d_w[r,b] * d_a[t,b]
// with isum_b the exact int32 dot product of one 32-element block.
//
// gemm_*: per 32-element block and 32 x 32 (token x row) tile, one
// v_mfma_i32_32x32x32_i8 gives every isum_b exactly, and one two-block
// v_mfma_f32_32x32x1_2b_f32 per token tile gives the scales
// s_b = d_w * d_a of both row tiles, each as a single IEEE product (round to
// nearest even, the same value as the reference's f32 multiply).  Lane
// 32 blk + i supplies row / column i of block blk, and block blk's results
// sit in registers 16 blk .. 16 blk + 15 in the layout of a one-block
// 32 x 32 MFMA (checked on the device), so no operand is wasted.  The epilogue per element and
// block is then the reference's own two roundings, total = total + isum * s,
// in block order, so every output is bit-identical to the reference for
// identical activation codes.
//
// Three VALU operations per element and block (convert, multiply, add) bound
// the kernel: at the 8B gate|up shape with 2048 tokens the VALU issues on 94 %
// of its cycles and the matrix cores work on 24 %.  So everything else is kept
// off the VALU.  Workgroup tile 128 tokens x 128 rows, four waves of 64 x 64
// (2 x 2 MFMA tiles).  Operands reach LDS four blocks at a time by direct
// loads (no registers, no LDS writes), double-buffered: a stage's loads are in
// flight while the one before is computed.  Q4 codes stay packed until the
// operand is read: lanes 0..31 of a wave take a block's low nibbles, the
// others the high ones, as 16 (q - 8) in the upper half of a byte - a shift
// and one three-input operation per dword.  The factor 16 only moves the
// exponent of sums and totals and is taken out at the end; a wave in which it
// may have carried one past the largest float redoes those outputs without it
// (gemm_common.h).  The check is one FMA per output (8B, 2048 tokens, without /
// with it in turn: gate|up 919 - 927 / 892 - 913 us, down 430 - 434 / 421 - 428).
// Within a wave the matrix instructions run one tile ahead of the arithmetic.
// Measured (8B, 2048 tokens, us; before: codes through registers, unpacked
// when written to LDS, matrix results read as soon as issued): gate|up 1066 ->
// 867 (555 TOP/s), down 492 -> 412, O 161 -> 139, Q|K|V 244 -> 186; 1B, 700
// tokens: gate|up 160 -> 128, down 232 -> 163.  Eight waves of 64 x 32 (four a
// SIMD) were no faster (down 440, O 137), nor were sums started at 1.5 * 2^23
// so that a subtraction replaces the convert (gate|up 859).
//
// 128 x 128 tiles leave CUs idle when the rows or tokens are few (96 of them
// for 700 tokens and 2048 rows), and the K blocks of an output cannot be split
// (their additions have an order).  64 x 128 (a wave: one token tile, two row
// tiles) and 64 x 64 (one tile, its scales two blocks at a time) give more and
// shorter chains, in stages of eight blocks; gemm_plan (runtime.cpp) picks one.
// 1B, 700 tokens, us: down 163 -> 74, O 55 -> 24, Q|K|V 43 -> 33.
#include "attn_core.h"
#include "exact_math.h"
#include "gemm_common.h"
#include "gemv_core.h"

using namespace llmrs;

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v32f __attribute__((ext_vector_type(32)));

namespace {

// LDS of one pipeline stage (bytes) of a workgroup's 64 TT tokens x 64 RT rows,
// KB blocks of BCH weight chunks.  Codes in 16-byte chunks as they lie in
// memory, one row (token) after the other: chunk c of row i at
// i * C + (c ^ swizzle<C>(i)), C chunks per row.  The lanes of a wave's direct
// load fill 64 consecutive chunks, whole rows of a stage, so the global reads
// are runs of 64 to 256 bytes; a half-wave's operand read (one chunk of 32
// rows) takes 16 rows' chunks from 16 different places of a 256-byte window.
// Then f32 scales d_w [KB][SW] and d_a [KB][SA] (rows padded by 4).
template <int TT, int RT, int KB, int BCH>
struct GemmStage {
  static constexpr int BM = 64 * TT, BN = 64 * RT;
  static constexpr int AC = 2 * KB, RC = BCH * KB;  // chunks of a token / row
  static constexpr int A = 0;
  static constexpr int B = A + AC * BM * 16;
  static constexpr int DW = B + RC * BN * 16;
  static constexpr int SW = BN + 4, SA = BM + 4;
  static constexpr int DA = DW + KB * SW * 4;
  static constexpr int BYTES = DA + KB * SA * 4;
  static_assert(2 * BYTES == gemm_lds_bytes(TT, RT, KB, BCH), "GEMM LDS size");
};

template <int C>
__device__ __forceinline__ int swizzle(int row) {
  return C == 16 ? row & 15 : C == 8 ? (row >> 1) & 7 : (row >> 2) & 3;
}

// MFMA operands of one block for a wave's TT x RT tiles: codes (Q4: the raw
// 16 bytes of the lane's row until unpacked) and the operands of the two-block
// scale MFMA, whose block blk comes from lanes 32 blk..: with two row tiles d_a
// of the lane's token in each token tile and d_w of its row in row tile `half`;
// with one, of its token and row in block b + half.
template <int TT, int RT>
struct GemmOps {
  v4i A[TT], B[RT];
  float da[TT], dw;
};

// The lane's 16 Q4 codes as int8 16 (q - 8): q ^ 8 in the upper nibble of a
// byte.  sh = 4 takes the low nibbles (codes 0..15), 0 the high (16..31).
__device__ __forceinline__ v4i q4_bytes16(v4i w, int sh) {
  v4i r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = (int)((((unsigned)w[i] << sh) & 0xF0F0F0F0u) ^ 0x80808080u);
  return r;
}

}  // namespace

// First token and row of this workgroup's tile (PrefillGemmArgs::group_m).
// Both steps are bijections on [0, tiles): the XCD deal when the tile count
// is a multiple of 8, the grouped walk for any grid.
template <int BM, int BN>
__device__ __forceinline__ void gemm_tile(const PrefillGemmArgs& a, int& m0, int& n0) {
  const int gx = gridDim.x, gy = gridDim.y, T = gx * gy;
  if (a.group_m <= 0) {
    m0 = blockIdx.y * BM;
    n0 = blockIdx.x * BN;
    return;
  }
  int t = blockIdx.x + blockIdx.y * gx;
  if ((T & 7) == 0) t = (t & 7) * (T >> 3) + (t >> 3);
  const int gsz = a.group_m * gx, g = t / gsz, fm = g * a.group_m;
  const int gm = min(gy - fm, a.group_m), r = t - g * gsz;
  m0 = (fm + r % gm) * BM;
  n0 = (r / gm) * BN;
}

template <int WT, int EPI, int TT, int RT>
__device__ __forceinline__ void gemm_impl(const PrefillGemmArgs& a, uint8_t* lds) {
  constexpr int BCH = WT == WT_Q8H ? 2 : 1;  // 16-byte chunks per weight block
  constexpr int KB = gemm_stage_blocks(TT, RT, BCH);
  typedef GemmStage<TT, RT, KB, BCH> S;
  typedef GemmOps<TT, RT> Ops;
  constexpr int T = kGemmThreads;
  constexpr int AL = S::AC * S::BM / T, BL = S::RC * S::BN / T;  // chunks per thread
  constexpr int SAL = KB * S::BM / T, SWL = KB * S::BN / T;      // scales per thread
  constexpr int NTB = TT * RT;                                   // a wave's tiles per block
  constexpr int AHEAD = NTB == 1 ? 2 : 1;                        // blocks whose operands are read ahead
  static_assert(EPI != EPI_SILU || RT == 2, "SwiGLU: a gate and an up tile per wave");
  static_assert(RT == 2 || TT == 1, "scale pairs: two row tiles or two blocks");
  const int lane = lane_id(), tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(wave_id());
  const int half = lane >> 5, col = lane & 31;
  int m0, n0;
  gemm_tile<S::BM, S::BN>(a, m0, n0);
  const int wm = (wave >> 1) * 32 * TT, wn = (wave & 1) * 32 * RT;
  const int nb = a.K >> 5;
  const int nfull = nb / KB, rest = nb % KB;

  // ---- staging: codes straight to LDS, scales through registers -------------
  // Load j of a wave fills chunks T j + 64 wave + lane: chunk p belongs to row
  // p / C and holds chunk (p % C) ^ swizzle(row) of it (the same for every j).
  const int8_t* xbase = a.xq + (size_t)m0 * a.K;
  const uint8_t* wbase = a.wq + (size_t)n0 * nb * (16 * BCH);
  const int ac = (tid % S::AC) ^ swizzle<S::AC>(tid / S::AC);
  const int bc = (tid % S::RC) ^ swizzle<S::RC>(tid / S::RC);
  unsigned aoff[AL], boff[BL];  // bytes from the tile's first row, block 0
#pragma unroll
  for (int j = 0; j < AL; ++j)
    aoff[j] = (unsigned)(min(m0 + (T * j + tid) / S::AC, a.M - 1) - m0) * (unsigned)a.K;
#pragma unroll
  for (int j = 0; j < BL; ++j)
    boff[j] = (unsigned)(min(n0 + (T * j + tid) / S::RC, a.N - 1) - n0) * (unsigned)(nb * 16 * BCH);
  const int srow = tid / KB, sblk = tid % KB;  // scales: row srow + T / KB j, block sblk
  unsigned rdw[SWL];
  float rda[SAL];
  auto load_stage = [&](int b0, uint8_t* base) {
    // blocks past the row's end (a last partial stage): its last block again
    const int ab = min(b0 + ac / 2, nb - 1) * 32 + 16 * (ac & 1);
    const int bb = min(b0 + bc / BCH, nb - 1) * (16 * BCH) + 16 * (bc % BCH);
#pragma unroll
    for (int j = 0; j < AL; ++j) load_lds16(xbase + (aoff[j] + (unsigned)ab), base + S::A + (T * j + 64 * wave) * 16);
#pragma unroll
    for (int j = 0; j < BL; ++j) load_lds16(wbase + (boff[j] + (unsigned)bb), base + S::B + (T * j + 64 * wave) * 16);
    const int blk = min(b0 + sblk, nb - 1);
#pragma unroll
    for (int j = 0; j < SWL; ++j) {
      const size_t si = (size_t)min(n0 + srow + T / KB * j, a.N - 1) * nb + blk;
      rdw[j] = WT == WT_Q4F ? ((const unsigned*)a.ws)[si] : ((const uint16_t*)a.ws)[si];
    }
#pragma unroll
    for (int j = 0; j < SAL; ++j) rda[j] = a.xd[(size_t)min(m0 + srow + T / KB * j, a.M - 1) * nb + blk];
  };
  auto store_scales = [&](uint8_t* base) {
#pragma unroll
    for (int j = 0; j < SWL; ++j) ((float*)(base + S::DW))[sblk * S::SW + srow + T / KB * j] = wscale<WT>(rdw[j]);
#pragma unroll
    for (int j = 0; j < SAL; ++j) ((float*)(base + S::DA))[sblk * S::SA + srow + T / KB * j] = rda[j];
  };

  // ---- compute -------------------------------------------------------------
  const int tok = wm + col, row = wn + col;  // of tile 0; tile t's swizzles are the same
  auto load_codes = [&](const uint8_t* base, int b, Ops& o) {
#pragma unroll
    for (int t = 0; t < TT; ++t)
      o.A[t] = *(const v4i*)(base + S::A + ((tok + 32 * t) * S::AC + ((2 * b + half) ^ swizzle<S::AC>(tok))) * 16);
#pragma unroll
    for (int r = 0; r < RT; ++r) {
      const int c = BCH == 2 ? 2 * b + half : b;
      o.B[r] = *(const v4i*)(base + S::B + ((row + 32 * r) * S::RC + (c ^ swizzle<S::RC>(row))) * 16);
    }
  };
  auto load_scales = [&](const uint8_t* base, int b, Ops& o) {
#pragma unroll
    for (int t = 0; t < TT; ++t) o.da[t] = ((const float*)(base + S::DA))[b * S::SA + tok + 32 * t];
    o.dw = ((const float*)(base + S::DW))[b * S::SW + row + (RT == 2 ? 32 * half : 0)];
  };
  auto load_ops = [&](const uint8_t* base, int b, Ops& o) {
    load_codes(base, b, o);
    if (RT == 2) load_scales(base, b, o);
    else if (b % 2 == 0) load_scales(base, b + half, o);
  };
  const int sh = half ? 0 : 4;
  auto unpack = [&](Ops& o) {
    if (WT != WT_Q8H) {
#pragma unroll
      for (int r = 0; r < RT; ++r) o.B[r] = q4_bytes16(o.B[r], sh);
    }
  };
  auto scales = [&](const Ops& o, int t) {
    return __builtin_amdgcn_mfma_f32_32x32x1f32(o.da[t], o.dw, v32f{}, 0, 0, 0);
  };
  auto sums = [&](const Ops& o, int t, int r) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(o.A[t], o.B[r], v16i{}, 0, 0, 0);
  };

  v16f acc[TT][RT];
#pragma unroll
  for (int t = 0; t < TT; ++t)
#pragma unroll
    for (int r = 0; r < RT; ++r) acc[t][r] = v16f{};

  // The next stage's loads are in flight while this one is computed; each
  // wave waits for its own before the barrier that hands the buffer over.
  auto hand_over = [&](int st, bool more) {
    if (more) store_scales(lds + ((st + 1) & 1) * S::BYTES);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };
  load_stage(0, lds);
  hand_over(-1, true);
  for (int st = 0; st < nfull; ++st) {
    const bool more = (st + 1) * KB < nb;
    if (more) load_stage((st + 1) * KB, lds + ((st + 1) & 1) * S::BYTES);
    const uint8_t* base = lds + (st & 1) * S::BYTES;
    // The stage's tiles k = NTB b + RT t + r, pipelined within the wave: the
    // block sums of tile k + 1 are issued before the arithmetic of tile k, and
    // the next pair's scales between the last products that read this pair's
    // and the additions, so no result is waited for.  pin() and the fences keep
    // this order: left to itself the compiler issues a stage's matrix
    // instructions together and spills their results.
    Ops o[AHEAD + 1];
    v16i P[2];
#pragma unroll
    for (int b = 0; b < AHEAD; ++b) {
      load_ops(base, b, o[b]);
      unpack(o[b]);
    }
    v32f SC = scales(o[0], 0);  // of tiles k and k + 1, k even
    P[0] = sums(o[0], 0, 0);
    pin(SC);
    pin(P[0]);
#pragma unroll
    for (int k = 0; k < NTB * KB; ++k) {
      const int b = k / NTB, t = (k % NTB) / RT, r = k % RT, kn = k + 1, tn = (kn % NTB) / RT;
      const bool next = kn < NTB * KB, ahead = b + AHEAD < KB;
      Ops& on = o[(kn / NTB) % (AHEAD + 1)];
      Ops& oa = o[(b + AHEAD) % (AHEAD + 1)];
      if (k % NTB == 0 && ahead) load_ops(base, b + AHEAD, oa);
      if (next) {
        pin(on.A[tn]);
        P[kn % 2] = sums(on, tn, kn % RT);
        pin(P[kn % 2]);
      }
      __builtin_amdgcn_sched_barrier(0);
      pin(P[k % 2]);
      v16f f;
#pragma unroll
      for (int i = 0; i < 16; ++i) f[i] = (float)P[k % 2][i];
#pragma unroll
      for (int i = 0; i < 16; ++i) f[i] = f[i] * SC[16 * (k % 2) + i];  // cpu.rs:913,932: total += isum * (d_w * d_a)
      pin(f);
      __builtin_amdgcn_sched_barrier(0);
      if (k % 2 == 1 && next) {
        pin(on.da[tn]);
        SC = scales(on, tn);
        pin(SC);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[t][r][i] = acc[t][r][i] + f[i];
      pin(acc[t][r]);
      if (k % NTB == NTB / 2 - (NTB == 2) && ahead) {
        unpack(oa);
#pragma unroll
        for (int q = 0; q < RT; ++q) pin(oa.B[q]);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    hand_over(st, more);
  }
  const uint8_t* tail = lds + (nfull & 1) * S::BYTES;
  for (int b = 0; b < rest; ++b) {
    Ops o;
    load_codes(tail, b, o);
    load_scales(tail, b, o);
    unpack(o);
#pragma unroll
    for (int t = 0; t < TT; ++t) {
      const v32f sc = scales(o, t);
#pragma unroll
      for (int r = 0; r < RT; ++r) {
        const v16i p = sums(o, t, r);
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][r][i] = acc[t][r][i] + (float)p[i] * sc[16 * r + i];
      }
    }
  }
  if (WT != WT_Q8H) {  // the Q4 codes were 16 times theirs
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 16; ++i) acc[t][r][i] = acc[t][r][i] * 0.0625f;
  }

  // Epilogues.  Register i of a tile holds token 8 (i / 4) + 4 half + i % 4
  // and row col.  Where a wave holds totals that are not finite (gemm_common.h),
  // those outputs take the plain block loop.
  bool redo_any = false;
  if constexpr (WT != WT_Q8H) {
    float z = 0.0f;  // stays 0 while every total is finite
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int i = 0; i < 16; ++i) z = __builtin_fmaf(acc[t][r][i], 0.0f, z);
    redo_any = __any(z != 0.0f);
  }
  auto token = [&](int t, int i) { return m0 + wm + 32 * t + 8 * (i / 4) + 4 * half + (i % 4); };
  if constexpr (EPI == EPI_SILU) {
    // rows n0+wn .. +31 are gate, +32 .. +63 the matching up rows
    // (layer.rs:72-79); m index j = (n0+wn)/2 + col.
    const int run = (n0 + wn) / 64, j = run * 32 + col;
    auto out = [&](int m, float g, float u) {
      const float mv = (g / (1.0f + exact_expf(-g))) * u;  // glibc expf (exact_math.h)
      float amax = fabsf(mv);
#pragma unroll
      for (int o = 16; o > 0; o >>= 1) amax = fmaxf(amax, __shfl_xor(amax, o, 32));
      const float d = amax / 127.0f;
      const float inv = amax == 0.0f ? 0.0f : 1.0f / d;
      if (m < a.M && n0 + wn < a.N) {
        if (a.y) a.y[(size_t)m * a.ldy + j] = mv;
        a.yq[act_row(m, a.N / 2, a.layout) + act_offset(j, a.layout)] =
            amax == 0.0f ? (int8_t)0 : (int8_t)q8_code(mv, inv);
        if (col == 0)
          a.yd[act_scale_row(m, a.N / 64, a.layout) + act_scale_offset(run, a.layout)] = amax == 0.0f ? 0.0f : d;
      }
    };
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
      for (int i = 0; i < 16; ++i) out(token(t, i), acc[t][0][i], acc[t][1][i]);
    if constexpr (WT != WT_Q8H) {
      if (redo_any) {  // over what was written: the tokens of register 16 t + i
        unsigned redo = 0;
#pragma unroll
        for (int t = 0; t < TT; ++t)
#pragma unroll
          for (int i = 0; i < 16; ++i)
            if (__any(!(is_finite(acc[t][0][i]) && is_finite(acc[t][1][i])))) redo |= 1u << (16 * t + i);
        const int gr = min(n0 + wn + col, a.N - 1), ur = min(n0 + wn + 32 + col, a.N - 1);
#pragma unroll 1
        for (; redo; redo &= redo - 1) {
          const int k = __builtin_ctz(redo), m = token(k >> 4, k & 15), mc = min(m, a.M - 1);
          out(m, q4_block_loop<WT, kActNatural>(a, mc, gr), q4_block_loop<WT, kActNatural>(a, mc, ur));
        }
      }
    }
  } else {
    auto out = [&](int m, int n, float v) {
      if (EPI == EPI_RESID) v = v + a.res[(size_t)m * a.N + n];  // layer.rs:386,403
      a.y[(size_t)m * a.ldy + n] = v;
    };
    if (!redo_any) {
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int r = 0; r < RT; ++r)
            if (token(t, i) < a.M && n0 + row + 32 * r < a.N) out(token(t, i), n0 + row + 32 * r, acc[t][r][i]);
    } else if constexpr (WT != WT_Q8H) {
      unsigned long long redo = 0;  // this lane's: bit RT (16 t + i) + r
#pragma unroll
      for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int i = 0; i < 16; ++i)
#pragma unroll
          for (int r = 0; r < RT; ++r)
            if (token(t, i) < a.M && n0 + row + 32 * r < a.N) {
              if (is_finite(acc[t][r][i])) out(token(t, i), n0 + row + 32 * r, acc[t][r][i]);
              else redo |= 1ull << (RT * (16 * t + i) + r);
            }
#pragma unroll 1
      for (; redo; redo &= redo - 1) {
        const int k = __builtin_ctzll(redo), i = k / RT, m = token(i >> 4, i & 15), n = n0 + row + 32 * (k % RT);
        out(m, n, q4_block_loop<WT, kActNatural>(a, m, n));
      }
    }
  }
}

// Kernels: gemm_<weights>_<epilogue>_<tokens>x<rows>; dynamic LDS of two stages.
#define LLMRS_GEMM(name, WT, EPI, TT, RT)                                         \
  extern "C" __global__ __launch_bounds__(kGemmThreads, 2) void name(PrefillGemmArgs a) { \
    extern __shared__ __align__(16) uint8_t gemm_lds[];                            \
    gemm_impl<WT, EPI, TT, RT>(a, gemm_lds);                                      \
  }
#define LLMRS_GEMM_WT(tag, WT)                                  \
  LLMRS_GEMM(gemm_##tag##_store_128x128, WT, EPI_STORE, 2, 2)   \
  LLMRS_GEMM(gemm_##tag##_resid_128x128, WT, EPI_RESID, 2, 2)   \
  LLMRS_GEMM(gemm_##tag##_silu_128x128, WT, EPI_SILU, 2, 2)     \
  LLMRS_GEMM(gemm_##tag##_store_64x128, WT, EPI_STORE, 1, 2)    \
  LLMRS_GEMM(gemm_##tag##_resid_64x128, WT, EPI_RESID, 1, 2)    \
  LLMRS_GEMM(gemm_##tag##_silu_64x128, WT, EPI_SILU, 1, 2)      \
  LLMRS_GEMM(gemm_##tag##_store_64x64, WT, EPI_STORE, 1, 1)     \
  LLMRS_GEMM(gemm_##tag##_resid_64x64, WT, EPI_RESID, 1, 1)
LLMRS_GEMM_WT(q4h, WT_Q4H)
LLMRS_GEMM_WT(q4f, WT_Q4F)
LLMRS_GEMM_WT(q8h, WT_Q8H)

// Per-row RMSNorm + Q8_0 (w != null) or plain Q8_0 (w == null): the GEMV
// prologue's arithmetic (same summation order), one workgroup per row, so a
// row gets the same codes here as in the decode path.
extern "C" __global__ __launch_bounds__(kThreads) void prefill_rows_q8(PrefillRowArgs r) {
  extern __shared__ __align__(16) uint8_t smem[];
  __shared__ float s_red[kWaves];
  GemvArgs g{};
  g.k = r.dim;
  g.x = r.x;
  g.norm_w = r.w;
  g.eps = r.eps;
  const int nb = r.dim >> 5;
  int8_t* s_q = (int8_t*)smem;
  float* s_d = (float*)(smem + r.dim);
  int* s_off = (int*)(smem + r.dim + 4 * nb);
  const int row = blockIdx.x;
  if (r.w) load_activation<PRO_NORM, false, false>(g, row, s_q, s_d, s_off, s_red);
  else load_activation<PRO_QUANT, false, false>(g, row, s_q, s_d, s_off, s_red);
  __syncthreads();
  if (r.layout == kActNatural) {
    const i32x4* src = (const i32x4*)s_q;
    i32x4* dst = (i32x4*)(r.xq + (size_t)row * r.dim);
    for (int i = threadIdx.x; i < r.dim / 16; i += kThreads) dst[i] = src[i];
  } else {
    int8_t* dst = r.xq + act_row(row, r.dim, r.layout);
    for (int i = 4 * threadIdx.x; i < r.dim; i += 4 * kThreads)  // aligned runs of 4 stay together
      *(unsigned*)(dst + act_offset(i, r.layout)) = *(const unsigned*)(s_q + i);
  }
  float* xd = r.xd + act_scale_row(row, nb, r.layout);
  for (int b = threadIdx.x; b < nb; b += kThreads) xd[act_scale_offset(b, r.layout)] = s_d[b];
}

// RoPE of q and k (cpu.rs:326-357, per head, position start_pos + t) and the
// K/V append (layer.rs:219-246): one thread per (token, head, pair).
extern "C" __global__ __launch_bounds__(256) void prefill_rope_kv(PrefillRopeArgs r) {
  const int mid = r.hd / 2;
  const int heads = r.nq + 2 * r.nkv;
  const long total = (long)r.M * heads * mid;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const int j = (int)(i % mid);
    const int h = (int)((i / mid) % heads);
    const int t = (int)(i / ((long)mid * heads));
    const int pos = r.start_pos + t;
    const float* src = r.qkv + (size_t)t * r.qkv_rows + (size_t)h * r.hd;
    const float c = r.rope_cos[(size_t)pos * mid + j], s = r.rope_sin[(size_t)pos * mid + j];
    if (h < r.nq) {
      const float re = src[j], im = src[j + mid];
      float* q = r.q + (size_t)t * r.nq * r.hd + (size_t)h * r.hd;
      q[j] = re * c - im * s;
      q[j + mid] = re * s + im * c;
    } else if (h < r.nq + r.nkv) {
      const int g = h - r.nq;
      const float re = src[j], im = src[j + mid];
      const float k0 = re * c - im * s, k1 = re * s + im * c;
      const size_t o = ((size_t)g * r.max_seq + pos) * r.hd;
      if (r.kv16) {
        ((uint16_t*)r.kc)[o + j] = f2h(k0);
        ((uint16_t*)r.kc)[o + j + mid] = f2h(k1);
      } else {
        ((float*)r.kc)[o + j] = k0;
        ((float*)r.kc)[o + j + mid] = k1;
      }
    } else {
      const int g = h - r.nq - r.nkv;
      const size_t o = ((size_t)g * r.max_seq + pos) * r.hd;
      if (r.kv16) {  // blocked V layout (v_offset)
        const size_t hb = (size_t)g * r.max_seq * r.hd;
        ((uint16_t*)r.vc)[hb + v_offset(pos, j, r.hd, true)] = f2h(src[j]);
        ((uint16_t*)r.vc)[hb + v_offset(pos, j + mid, r.hd, true)] = f2h(src[j + mid]);
      } else {
        ((float*)r.vc)[o + j] = src[j];
        ((float*)r.vc)[o + j + mid] = src[j + mid];
      }
    }
  }
}

// Causal prefill attention (layer.rs:248-326): one workgroup per (32-query
// tile, query head).  Per key tile (64 positions for an f16 cache, 32 for
// f32): scores in 2 x 4 register blocks (f32 q times the stored K, staged in
// LDS in the cache's type), online softmax per query row (16-lane
// reductions), P.V in 2 x (HD/16) blocks; the causal mask keeps key
// j <= start_pos + t (layer.rs:264-266).  ctx is written as f32 and as Q8_0.
template <int HD, bool KV16>
__device__ __forceinline__ void attn_prefill_impl(const PrefillAttnArgs& a) {
  typedef typename KvType<KV16>::T kv_t;
  constexpr int QT = 32, KT = KV16 ? 64 : 32;
  constexpr int KPT = KT / 16;       // keys per thread in the score block
  constexpr int DPT = HD / 16;       // head dims per thread in P.V
  constexpr int KS = HD + (KV16 ? 8 : 4);  // padded LDS row (elements)
  __shared__ __align__(16) float s_q[QT][HD + 4];
  __shared__ __align__(16) kv_t s_k[KT][KS];
  __shared__ __align__(16) kv_t s_v[KT][KS];
  __shared__ float s_p[QT][KT + 4];

  const int tid = threadIdx.x;
  const int q0 = blockIdx.x * QT, h = blockIdx.y;
  const int g = h / (a.nq / a.nkv);
  const int qi = tid / 16, ki = tid % 16;  // rows 2qi, 2qi+1; keys KPT*ki..; dims DPT*ki..
  const int qdim = a.nq * HD;
  const kv_t* kc = (const kv_t*)a.kc + (size_t)g * a.max_seq * HD;
  const kv_t* vc = (const kv_t*)a.vc + (size_t)g * a.max_seq * HD;

  for (int i = tid; i < QT * HD; i += 256) {
    const int r = i / HD, d = i % HD;
    const int t = min(q0 + r, a.M - 1);
    s_q[r][d] = a.q[(size_t)t * qdim + (size_t)h * HD + d];
  }
  float m[2], l[2], o[2][DPT];
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    m[r] = -INFINITY;
    l[r] = 0.0f;
#pragma unroll
    for (int e = 0; e < DPT; ++e) o[r][e] = 0.0f;
  }
  // keys up to the last query's position
  const int kend = a.start_pos + min(q0 + QT, a.M);
  for (int k0 = 0; k0 < kend; k0 += KT) {
    __syncthreads();
#pragma unroll 2
    for (int i = tid; i < KT * HD; i += 256) {
      const int r = i / HD, d = i % HD;
      const int t = min(k0 + r, kend - 1);
      s_k[r][d] = kc[(size_t)t * HD + d];
      s_v[r][d] = vc[v_offset(t, d, HD, KV16)];
    }
    __syncthreads();
    float sc[2][KPT];
#pragma unroll
    for (int r = 0; r < 2; ++r)
#pragma unroll
      for (int c = 0; c < KPT; ++c) sc[r][c] = 0.0f;
#pragma unroll 2
    for (int d = 0; d < HD; d += 4) {
      f32x4 qv[2];
#pragma unroll
      for (int r = 0; r < 2; ++r) qv[r] = *(const f32x4*)&s_q[2 * qi + r][d];
#pragma unroll
      for (int c = 0; c < KPT; ++c) {
        const kv_t* kr = &s_k[KPT * ki + c][d];
        const float k0f = kv_to_f<KV16>(kr[0]), k1f = kv_to_f<KV16>(kr[1]);
        const float k2f = kv_to_f<KV16>(kr[2]), k3f = kv_to_f<KV16>(kr[3]);
#pragma unroll
        for (int r = 0; r < 2; ++r) {
          float s2 = sc[r][c];
          s2 = __builtin_fmaf(qv[r].x, k0f, s2);
          s2 = __builtin_fmaf(qv[r].y, k1f, s2);
          s2 = __builtin_fmaf(qv[r].z, k2f, s2);
          s2 = __builtin_fmaf(qv[r].w, k3f, s2);
          sc[r][c] = s2;
        }
      }
    }
    // mask, online softmax per query row (16 lanes share a row pair)
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const int qpos = a.start_pos + q0 + 2 * qi + r;
      float rmax = -INFINITY;
#pragma unroll
      for (int c = 0; c < KPT; ++c) {
        const int kpos = k0 + KPT * ki + c;
        sc[r][c] = (kpos <= qpos && kpos < kend) ? sc[r][c] * a.scale : -INFINITY;
        rmax = fmaxf(rmax, sc[r][c]);
      }
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) rmax = fmaxf(rmax, __shfl_xor(rmax, off, 16));
      const float mnew = fmaxf(m[r], rmax);
      const float corr = (m[r] == -INFINITY) ? 0.0f : expf(m[r] - mnew);
      float psum = 0.0f;
#pragma unroll
      for (int c = 0; c < KPT; ++c) {
        const float p = (sc[r][c] == -INFINITY) ? 0.0f : expf(sc[r][c] - mnew);
        s_p[2 * qi + r][KPT * ki + c] = p;
        psum += p;
      }
#pragma unroll
      for (int off = 8; off > 0; off >>= 1) psum += __shfl_xor(psum, off, 16);
      l[r] = l[r] * corr + psum;
      m[r] = mnew;
#pragma unroll
      for (int e = 0; e < DPT; ++e) o[r][e] = o[r][e] * corr;
    }
    __syncthreads();
    // P.V: rows 2qi.., dims DPT*ki..
    const int kvalid = min(KT, kend - k0);
#pragma unroll 4
    for (int kk = 0; kk < kvalid; ++kk) {
      const float p0 = s_p[2 * qi][kk], p1 = s_p[2 * qi + 1][kk];
      const kv_t* vr = &s_v[kk][DPT * ki];
#pragma unroll
      for (int e = 0; e < DPT; ++e) {
        const float vv = kv_to_f<KV16>(vr[e]);
        o[0][e] = __builtin_fmaf(p0, vv, o[0][e]);
        o[1][e] = __builtin_fmaf(p1, vv, o[1][e]);
      }
    }
  }
  // ctx rows (f32 and Q8_0): a 32-dim block spans 32/DPT threads of a row.
  constexpr int TPB = 32 / DPT;
#pragma unroll
  for (int r = 0; r < 2; ++r) {
    const int t = q0 + 2 * qi + r;
    float v[DPT];
    float amax = 0.0f;
#pragma unroll
    for (int e = 0; e < DPT; ++e) {
      v[e] = o[r][e] / l[r];
      amax = fmaxf(amax, fabsf(v[e]));
    }
#pragma unroll
    for (int off = TPB / 2; off > 0; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, TPB));
    const float d = amax / 127.0f;
    const float inv = amax == 0.0f ? 0.0f : 1.0f / d;
    if (t < a.M) {
      const size_t base = (size_t)t * qdim + (size_t)h * HD + DPT * ki;
#pragma unroll
      for (int e = 0; e < DPT; ++e) {
        if (a.ctx) a.ctx[base + e] = v[e];
        a.ctx_q[act_row(t, qdim, a.ctx_layout) + act_offset(h * HD + DPT * ki + e, a.ctx_layout)] =
            amax == 0.0f ? (int8_t)0 : (int8_t)q8_code(v[e], inv);
      }
      if ((ki % TPB) == 0)
        a.ctx_d[act_scale_row(t, qdim / 32, a.ctx_layout) +
                act_scale_offset((h * HD + DPT * ki) / 32, a.ctx_layout)] = amax == 0.0f ? 0.0f : d;
    }
  }
}

// Causal prefill attention on the matrix cores, f16 K/V cache.  One
// workgroup of 8 waves per (32-query tile, KV group): wave w takes query head
// g * n_rep + w % 4 (+4, +8, ... for larger groups) and key stream w / 4,
// which covers the even or odd key tiles, so the four heads share each
// staged K/V tile and the two streams halve the serial path of long tiles.
// Per key tile of 32:
//   S^T = K Q^T        (v_mfma_f32_32x32x16_f16; q split into f16 hi + lo,
//                       so the products carry ~22 bits of q, as in f32)
//   online softmax      one query per lane column: row max / sum over the
//                       lane's 16 keys and its partner lane's 16; exp as
//                       exp2 of log2(e)-scaled scores
//   O^T += V^T P^T      (P split into f16 hi + lo; keys taken in the order
//                       the S^T registers hold them, V^T staged to match)
// The two streams' (max, sum, O) are merged through LDS at the end.  The
// causal mask keeps key j <= start_pos + t (layer.rs:264-266).  Query tiles
// run longest-first.  ctx is written as Q8_0 (and f32 when asked).
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

template <int HD>
struct AttnMfmaLds {
  static constexpr int KT = 32;                 // keys per tile
  static constexpr int KROW = HD * 2 + 16;      // padded K row (bytes)
  static constexpr int VROW = KT * 2 + 8;       // padded V^T row (bytes)
  static constexpr int K = 0;
  static constexpr int V = K + KT * KROW;
  static constexpr int TILE = V + HD * VROW;    // one staged tile
  static constexpr int BYTES = 2 * TILE;        // the even and odd tiles
  // merge area (reuses the tiles): per head, lane: 16 O values of one pass + m, l
  static constexpr int MERGE = 4 * 64 * 18 * 4;
  static_assert(MERGE <= BYTES, "merge area fits in the tile buffers");
};

template <int HD>
__device__ __forceinline__ void attn_prefill_mfma_impl(const PrefillAttnArgs& a) {
  typedef AttnMfmaLds<HD> LY;
  constexpr int NS = HD / 16, ND = HD / 32, KT = LY::KT;
  constexpr float kLog2e = 1.4426950408889634f;
  __shared__ __align__(16) uint8_t lds[LY::BYTES];
  const int lane = lane_id(), wave = wave_id(), tid = threadIdx.x;
  const int h2 = lane >> 5, col = lane & 31;
  const int hw = wave & 3, stream = wave >> 2;
  const int q0 = (gridDim.x - 1 - blockIdx.x) * 32, g = blockIdx.y;  // longest tiles first
  const int n_rep = a.nq / a.nkv;
  const int qdim = a.nq * HD;
  const uint16_t* kc = (const uint16_t*)a.kc + (size_t)g * a.max_seq * HD;
  const uint16_t* vc = (const uint16_t*)a.vc + (size_t)g * a.max_seq * HD;
  const int kend = a.start_pos + min(q0 + 32, a.M);  // keys [0, kend)
  const int ntile = (kend + KT - 1) / KT;
  const int npair = (ntile + 1) / 2;
  const int myq = q0 + col;
  const int qpos = a.start_pos + myq;
  const float sl2 = a.scale * kLog2e;

  for (int rp = 0; rp < n_rep; rp += 4) {
    const int r = rp + hw;
    const bool active = r < n_rep;  // wave-uniform
    const int h = g * n_rep + min(r, n_rep - 1);
    v8h qh[NS], ql[NS];
    {
      const float* qrow = a.q + (size_t)min(myq, a.M - 1) * qdim + (size_t)h * HD;
#pragma unroll
      for (int sl = 0; sl < NS; ++sl) {
        const f32x4 x0 = *(const f32x4*)(qrow + 16 * sl + 8 * h2);
        const f32x4 x1 = *(const f32x4*)(qrow + 16 * sl + 8 * h2 + 4);
        const float xv[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const _Float16 hi = (_Float16)xv[j];
          qh[sl][j] = hi;
          ql[sl][j] = (_Float16)(xv[j] - (float)hi);
        }
      }
    }
    v16f o[ND];
#pragma unroll
    for (int d = 0; d < ND; ++d) o[d] = v16f{};
    float m = -INFINITY, l = 0.0f;  // m in the log2 domain

    // K rows [key][HD] and V^T [HD][key] of tile pair (2i, 2i+1): thread
    // chunk c < 2 * 32 * HD / 8 = (tile c / (32 HD / 8), then key and 8-dim
    // part of K, or dim and 8-key block of the blocked V); keys clamped
    // (those past kend are masked below).  Loaded a pair ahead.
    constexpr int CPT = 2 * KT * HD / 8 / 512;
    u32x4 rk[CPT], rv[CPT];
    auto fetch = [&](int pr) {
#pragma unroll
      for (int j = 0; j < CPT; ++j) {
        const int c = tid + 512 * j;
        const int t = c / (KT * HD / 8), cc = c % (KT * HD / 8);
        const int key = cc / (HD / 8), part = cc % (HD / 8);
        rk[j] = *(const u32x4*)(kc + (size_t)min((2 * pr + t) * KT + key, kend - 1) * HD + part * 8);
        const int vb = cc / HD, vd = cc % HD;
        rv[j] = *(const u32x4*)(vc + v_offset(min((2 * pr + t) * KT + 8 * vb, kend - 1) & ~7, vd, HD, true));
      }
    };
    fetch(0);
    for (int pr = 0; pr < npair; ++pr) {
      __syncthreads();  // the previous pair is consumed
#pragma unroll
      for (int j = 0; j < CPT; ++j) {
        const int c = tid + 512 * j;
        const int t = c / (KT * HD / 8), cc = c % (KT * HD / 8);
        const int key = cc / (HD / 8), part = cc % (HD / 8);
        uint8_t* tb = lds + t * LY::TILE;
        *(u32x4*)(tb + LY::K + key * LY::KROW + part * 16) = rk[j];
        const int vb = cc / HD, vd = cc % HD;  // keys 8 vb .. 8 vb + 7 of dim vd
        uint2* vdst = (uint2*)(tb + LY::V + vd * LY::VROW + vb * 16);
        vdst[0] = make_uint2(rv[j].x, rv[j].y);
        vdst[1] = make_uint2(rv[j].z, rv[j].w);
      }
      __syncthreads();
      if (pr + 1 < npair) fetch(pr + 1);
      const int kt = 2 * pr + stream;
      if (!active || kt >= ntile) continue;
      const uint8_t* tb = lds + stream * LY::TILE;
      // S^T: lane holds keys kt*32 + 8(i/4) + 4 h2 + i%4 for query col
      v16f st = v16f{};
#pragma unroll
      for (int sl = 0; sl < NS; ++sl) {
        const v8h kop = *(const v8h*)(tb + LY::K + col * LY::KROW + (16 * sl + 8 * h2) * 2);
        st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kop, qh[sl], st, 0, 0, 0);
        st = __builtin_amdgcn_mfma_f32_32x32x16_f16(kop, ql[sl], st, 0, 0, 0);
      }
      float p[16];
      float mloc = -INFINITY;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int key = kt * KT + 8 * (i / 4) + 4 * h2 + (i % 4);
        p[i] = key <= qpos ? st[i] * sl2 : -INFINITY;
        mloc = fmaxf(mloc, p[i]);
      }
      mloc = fmaxf(mloc, __shfl_xor(mloc, 32));
      // The stream's first tile holds a key <= qpos for every query (key 0
      // or, for stream 1, key 32 <= qpos whenever that tile is reached with
      // an unmasked key); a fully masked tile keeps mn = m.
      const float mn = fmaxf(m, mloc);
      const float corr = mn == -INFINITY ? 1.0f : __builtin_amdgcn_exp2f(m - mn);
      float lsum = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        p[i] = mn == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(p[i] - mn);
        lsum += p[i];
      }
      lsum += __shfl_xor(lsum, 32);
      l = l * corr + lsum;
      m = mn;
#pragma unroll
      for (int d = 0; d < ND; ++d)
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] *= corr;
      // O^T += V^T P^T over the two 16-key slices
#pragma unroll
      for (int s2 = 0; s2 < 2; ++s2) {
        v8h ph, pl;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const float x = p[8 * s2 + j];
          const _Float16 hi = (_Float16)x;
          ph[j] = hi;
          pl[j] = (_Float16)(x - (float)hi);
        }
#pragma unroll
        for (int d = 0; d < ND; ++d) {
          const uint8_t* vrow = tb + LY::V + (32 * d + col) * LY::VROW;
          const v4h v0 = *(const v4h*)(vrow + (16 * s2 + 4 * h2) * 2);
          const v4h v1 = *(const v4h*)(vrow + (16 * s2 + 8 + 4 * h2) * 2);
          const v8h vop = v8h{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vop, ph, o[d], 0, 0, 0);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vop, pl, o[d], 0, 0, 0);
        }
      }
    }
    // Merge stream 1 into stream 0 through LDS, one 32-dim block at a time.
    float* mg = (float*)lds + (hw * 64 + lane) * 18;
    float m1 = -INFINITY, l1 = 0.0f, c0 = 1.0f, c1 = 0.0f;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      __syncthreads();  // tiles (or the previous block) consumed
      if (stream == 1) {
#pragma unroll
        for (int i = 0; i < 16; ++i) mg[i] = o[d][i];
        mg[16] = m;
        mg[17] = l;
      }
      __syncthreads();
      if (stream == 0) {
        if (d == 0) {
          m1 = mg[16];
          l1 = mg[17];
          const float mm = fmaxf(m, m1);  // finite: stream 0 saw key 0
          c0 = __builtin_amdgcn_exp2f(m - mm);
          c1 = m1 == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(m1 - mm);
          l = l * c0 + l1 * c1;
        }
#pragma unroll
        for (int i = 0; i < 16; ++i) o[d][i] = o[d][i] * c0 + mg[i] * c1;
      }
    }
    __syncthreads();  // merge reads done before the next pass stages tiles
    if (!active || stream != 0) continue;
    // o[d][i] = O[query col][dim 32 d + 8 (i/4) + 4 h2 + i%4] * l
    const float inv_l = 1.0f / l;
    const bool write = myq < a.M;
    const size_t base = (size_t)min(myq, a.M - 1) * qdim + (size_t)h * HD;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
      float v[16];
      float amax = 0.0f;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        v[i] = o[d][i] * inv_l;
        amax = fmaxf(amax, fabsf(v[i]));
      }
      amax = fmaxf(amax, __shfl_xor(amax, 32));
      const float dq = amax / 127.0f;
      const float inv = amax == 0.0f ? 0.0f : 1.0f / dq;
      if (write) {
#pragma unroll
        for (int gq = 0; gq < 4; ++gq) {
          const size_t e = base + 32 * d + 8 * gq + 4 * h2;
          unsigned w = 0;
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            const int q8 = amax == 0.0f ? 0 : q8_code(v[4 * gq + c], inv);
            w |= ((unsigned)q8 & 0xFFu) << (8 * c);
          }
          *(unsigned*)(a.ctx_q + act_row(myq, qdim, a.ctx_layout) +
                       act_offset(h * HD + 32 * d + 8 * gq + 4 * h2, a.ctx_layout)) = w;
          if (a.ctx) *(f32x4*)(a.ctx + e) = f32x4{v[4 * gq], v[4 * gq + 1], v[4 * gq + 2], v[4 * gq + 3]};
        }
        if (h2 == 0)
          a.ctx_d[act_scale_row(myq, qdim / 32, a.ctx_layout) + act_scale_offset(h * HD / 32 + d, a.ctx_layout)] =
              amax == 0.0f ? 0.0f : dq;
      }
    }
  }
}

// Causal prefill attention on the matrix cores, f32 K/V cache: one workgroup of
// four waves per (32-query tile, query head), wave w taking key tiles w, w + 4,
// ... of 32 keys, so a wave works without barriers until the four streams'
// (max, sum, O) are merged through LDS.  Everything stays f32:
//   S^T = K Q^T        v_mfma_f32_32x32x2f32: lane (col, half) holds dims
//                       half * HD/2 .. of key / query col, so step s takes dims
//                       s and HD/2 + s; two sums of half the steps each, which
//                       rounds less than one long one
//   online softmax      one query per lane column, as in the f16 kernel
//   O^T += V^T P^T      register i of S^T holds keys 8 (i/4) + i%4 (lower half)
//                       and + 4 (upper half): step i takes those two
// K rows are read as 16-byte pieces of a lane's own row and V as whole lines; V
// is requested before the scores and the next K after them, so a tile's 2 HD/2
// matrix instructions (64 cycles each) cover the reads.  They bound it: 700 rows
// of the 1B shape need 14 us at the f32 matrix rate and take 51, 2048 rows 319
// (the longest query tile's streams end last); the vector kernel's dots
// and P.V (four multiply-adds per LDS read) took 104 and 655.  Distance from
// 64-bit sums as a share of the vector kernel's (30 seeds a shape), with one
// sum / two: 16 rows after 17 1.03 / 0.94 (head_dim 64), 1.01 / 0.80 (128); 32
// rows 1.01 / 0.99, 1.01 / 0.87; 64 rows 0.97 / 0.94, 0.99 / 0.85; 700 rows (3
// seeds) 0.66 / 0.65, 0.71 / 0.63.  Times are the same.
template <int HD>
__device__ __forceinline__ void attn_prefill_f32_impl(const PrefillAttnArgs& a) {
  constexpr int ND = HD / 32, HH = HD / 2, KT = 32, NSTR = 4;
  __shared__ float s_o[NSTR][16 * ND][LLMRS_WAVE];
  __shared__ float s_ml[NSTR][2][LLMRS_WAVE];
  const int lane = lane_id();
  const int w = __builtin_amdgcn_readfirstlane(wave_id());
  const int h2 = lane >> 5, col = lane & 31;
  const int q0 = (gridDim.x - 1 - blockIdx.x) * 32, h = blockIdx.y;  // longest tiles first
  const int g = h / (a.nq / a.nkv), qdim = a.nq * HD;
  const float* kc = (const float*)a.kc + (size_t)g * a.max_seq * HD;
  const float* vc = (const float*)a.vc + (size_t)g * a.max_seq * HD;
  const int kend = a.start_pos + min(q0 + 32, a.M);  // keys [0, kend)
  const int ntile = (kend + KT - 1) / KT;
  const int myq = q0 + col, qpos = a.start_pos + myq;

  float q[HH], k[HH], v[ND][16];
  auto load_row = [&](const float* row, float (&x)[HH]) {
#pragma unroll
    for (int j = 0; j < HH / 4; ++j) {
      const f32x4 t = *(const f32x4*)(row + HH * h2 + 4 * j);
#pragma unroll
      for (int c = 0; c < 4; ++c) x[4 * j + c] = t[c];
    }
  };
  auto load_k = [&](int kt) { load_row(kc + (size_t)min(kt * KT + col, kend - 1) * HD, k); };
  load_row(a.q + (size_t)min(myq, a.M - 1) * qdim + (size_t)h * HD, q);
  if (w < ntile) load_k(w);
  v16f o[ND];
#pragma unroll
  for (int d = 0; d < ND; ++d) o[d] = v16f{};
  float m = -INFINITY, l = 0.0f;
  for (int kt = w; kt < ntile; kt += NSTR) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = min(kt * KT + 8 * (i / 4) + 4 * h2 + (i % 4), kend - 1);
#pragma unroll
      for (int d = 0; d < ND; ++d) v[d][i] = vc[(size_t)key * HD + 32 * d + col];
    }
    v16f st = v16f{}, st1 = v16f{};
#pragma unroll
    for (int s = 0; s < HH / 2; ++s) {
      st = __builtin_amdgcn_mfma_f32_32x32x2f32(k[s], q[s], st, 0, 0, 0);
      st1 = __builtin_amdgcn_mfma_f32_32x32x2f32(k[HH / 2 + s], q[HH / 2 + s], st1, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) st[i] = st[i] + st1[i];
    if (kt + NSTR < ntile) load_k(kt + NSTR);
    float p[16];
    float mloc = -INFINITY;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int key = kt * KT + 8 * (i / 4) + 4 * h2 + (i % 4);
      p[i] = key <= qpos && key < kend ? st[i] * a.scale : -INFINITY;
      mloc = fmaxf(mloc, p[i]);
    }
    mloc = fmaxf(mloc, __shfl_xor(mloc, 32));
    const float mn = fmaxf(m, mloc);  // -inf while every key so far is masked
    const float corr = m == -INFINITY ? 0.0f : expf(m - mn);
    float lsum = 0.0f;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      p[i] = p[i] == -INFINITY ? 0.0f : expf(p[i] - mn);
      lsum += p[i];
    }
    lsum += __shfl_xor(lsum, 32);
    l = l * corr + lsum;
    m = mn;
#pragma unroll
    for (int d = 0; d < ND; ++d) {
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d][i] *= corr;
#pragma unroll
      for (int i = 0; i < 16; ++i) o[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[d][i], p[i], o[d], 0, 0, 0);
    }
  }
#pragma unroll
  for (int d = 0; d < ND; ++d)
#pragma unroll
    for (int i = 0; i < 16; ++i) s_o[w][16 * d + i][lane] = o[d][i];
  s_ml[w][0][lane] = m;
  s_ml[w][1][lane] = l;
  __syncthreads();
  // Wave d merges and writes dims 32 d ..: register i is dim 8 (i/4) + 4 h2 + i%4.
  if (w >= ND) return;
  float mm = -INFINITY, c[NSTR];
#pragma unroll
  for (int s = 0; s < NSTR; ++s) mm = fmaxf(mm, s_ml[s][0][lane]);  // finite: key 0 is seen
  l = 0.0f;
#pragma unroll
  for (int s = 0; s < NSTR; ++s) {
    const float ms = s_ml[s][0][lane];
    c[s] = ms == -INFINITY ? 0.0f : expf(ms - mm);
    l += s_ml[s][1][lane] * c[s];
  }
  float x[16], amax = 0.0f;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    float t = 0.0f;
#pragma unroll
    for (int s = 0; s < NSTR; ++s) t += s_o[s][16 * w + i][lane] * c[s];
    x[i] = t / l;
    amax = fmaxf(amax, fabsf(x[i]));
  }
  amax = fmaxf(amax, __shfl_xor(amax, 32));
  const float dq = amax / 127.0f;
  const float inv = amax == 0.0f ? 0.0f : 1.0f / dq;
  if (myq >= a.M) return;
#pragma unroll
  for (int gq = 0; gq < 4; ++gq) {
    const int e = h * HD + 32 * w + 8 * gq + 4 * h2;
    unsigned word = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int q8 = amax == 0.0f ? 0 : q8_code(x[4 * gq + b], inv);
      word |= ((unsigned)q8 & 0xFFu) << (8 * b);
    }
    *(unsigned*)(a.ctx_q + act_row(myq, qdim, a.ctx_layout) + act_offset(e, a.ctx_layout)) = word;
    if (a.ctx)
      *(f32x4*)(a.ctx + (size_t)myq * qdim + e) = f32x4{x[4 * gq], x[4 * gq + 1], x[4 * gq + 2], x[4 * gq + 3]};
  }
  if (h2 == 0)
    a.ctx_d[act_scale_row(myq, qdim / 32, a.ctx_layout) + act_scale_offset(h * HD / 32 + w, a.ctx_layout)] =
        amax == 0.0f ? 0.0f : dq;
}

extern "C" __global__ __launch_bounds__(256, 2) void attn_prefill_mfma_hd64_f32(PrefillAttnArgs a) {
  attn_prefill_f32_impl<64>(a);
}
extern "C" __global__ __launch_bounds__(256, 1) void attn_prefill_mfma_hd128_f32(PrefillAttnArgs a) {
  attn_prefill_f32_impl<128>(a);
}

extern "C" __global__ __launch_bounds__(512) void attn_prefill_mfma_hd64(PrefillAttnArgs a) {
  attn_prefill_mfma_impl<64>(a);
}
extern "C" __global__ __launch_bounds__(512) void attn_prefill_mfma_hd128(PrefillAttnArgs a) {
  attn_prefill_mfma_impl<128>(a);
}

#define LLMRS_ATTN_PREFILL(name, HD, KV16)                                        \
  extern "C" __global__ __launch_bounds__(256) void name(PrefillAttnArgs a) {   \
    attn_prefill_impl<HD, KV16>(a);                                             \
  }
LLMRS_ATTN_PREFILL(attn_prefill_hd64_f32, 64, false)
LLMRS_ATTN_PREFILL(attn_prefill_hd64_f16, 64, true)
LLMRS_ATTN_PREFILL(attn_prefill_hd128_f32, 128, false)
LLMRS_ATTN_PREFILL(attn_prefill_hd128_f16, 128, true)
