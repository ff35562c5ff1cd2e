// runtime.cpp - device context, module loading, allocator, errors, helpers.
#include <dlfcn.h>
#include <immintrin.h>

#include <cmath>
#include <cstdlib>
#include <cstring>
#include <filesystem>
#include <functional>
#include <initializer_list>
#include <thread>

#include "../kernel_args.h"
#include "internal.h"

namespace llmrs {

namespace {
thread_local std::string g_last_error;
Context* g_ctx = nullptr;

std::string library_dir() {
  Dl_info info;
  if (dladdr((void*)&library_dir, &info) && info.dli_fname) {
    return std::filesystem::path(info.dli_fname).parent_path().string();
  }
  return ".";
}
}  // namespace

void fail(int code, const std::string& msg) { throw Error(code, msg); }
void set_last_error(const std::string& msg) { g_last_error = msg; }

std::recursive_mutex& api_mutex() {
  static std::recursive_mutex m;
  return m;
}

Context& ctx() {
  if (!g_ctx) fail(LLMRS_E_NOINIT, "llmrs_init has not been called");
  return *g_ctx;
}

hipFunction_t kernel(const std::string& name, dim3 block) {
  Context& c = ctx();
  auto it = c.kernels.find(name);
  if (it == c.kernels.end()) {
    for (hipModule_t m : c.modules) {
      KernelInfo k;
      if (hipModuleGetFunction(&k.f, m, name.c_str()) == hipSuccess && k.f) {
        LLMRS_HIP(hipFuncGetAttribute(&k.max_threads, HIP_FUNC_ATTRIBUTE_MAX_THREADS_PER_BLOCK, k.f));
        it = c.kernels.emplace(name, k).first;
        break;
      }
      (void)hipGetLastError();  // not in this module
    }
    if (it == c.kernels.end()) {
      fail(LLMRS_E_MODULE, "kernel not found in any loaded hsaco: " + name);
    }
  }
  const long threads = (long)block.x * block.y * block.z;
  LLMRS_REQUIRE(threads <= it->second.max_threads, LLMRS_E_INVALID,
                name + ": " + std::to_string(threads) + " threads per workgroup, compiled for at most " +
                    std::to_string(it->second.max_threads));
  return it->second.f;
}

void fetch(void* dst, const void* src, size_t bytes, std::initializer_list<const int*> ints, int* out) {
  Context& c = ctx();
  if (bytes > kFetchBytes) {
    LLMRS_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, c.stream));
    bytes = 0;
  }
  int* host_ints = (int*)(c.host_out + kFetchBytes);
  if (bytes || ints.size()) {
    PublishArgs a{src, c.host_out, bytes, {}, host_ints};
    size_t i = 0;
    for (const int* p : ints) a.ints[i++] = p;
    const size_t wgs = (bytes / 16 + 255) / 256;
    launch("publish", dim3((unsigned)std::max<size_t>(1, std::min<size_t>(wgs, 256))), dim3(256), 0, c.stream, a);
  }
  LLMRS_HIP(hipStreamSynchronize(c.stream));
  if (bytes) std::memcpy(dst, c.host_out, bytes);
  if (ints.size()) std::memcpy(out, host_ints, ints.size() * sizeof(int));
}

bool xcd_dealt_mod8(unsigned gx, unsigned gy) {
  const size_t n = (size_t)gx * gy;
  int* d = nullptr;
  LLMRS_HIP(hipMalloc(&d, n * sizeof(int)));
  std::vector<int> h(n);
  hipError_t e = hipSuccess;
  void* args[] = {&d};
  e = hipModuleLaunchKernel(kernel("xcc_ids", dim3(64)), gx, gy, 1, 64, 1, 1, 0, ctx().stream, args, nullptr);
  if (e == hipSuccess) e = hipMemcpyAsync(h.data(), d, n * sizeof(int), hipMemcpyDeviceToHost, ctx().stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx().stream);
  (void)hipFree(d);
  LLMRS_HIP(e);
  for (size_t i = 8; i < n; ++i)
    if (h[i] != h[i % 8]) return false;
  return true;
}

int gemm_group_m() {
  // 4 token tiles per group: on the 8B shapes at M = 2048 this cuts the
  // gate|up GEMM's L2 fetches 2.7x against row-major (8 is close, 2 and 16
  // fetch 1.5x and 2.1x more than 4)
  static const int g = [] {
    const char* v = std::getenv("LLMRS_GEMM_GROUP");
    return (v && *v) ? std::atoi(v) : 4;
  }();
  return g;
}

const char* wt_tag(int wt) {
  switch (wt) {
    case WT_Q4H: return "q4h";
    case WT_Q4F: return "q4f";
    case WT_Q8H: return "q8h";
  }
  fail(LLMRS_E_DTYPE, "unknown weight type");
}

// Rows per wave-unit R and 64-block chunks per unit U follow the shape: U = 2
// when the row splits into whole 128-block chunks, R = 2 for the narrow
// (n <= 8192) projections so that more waves share them.  The SwiGLU tile is
// 64 rows per workgroup (8-wave workgroups looping over the tiles, one per
// CU, when the tiles outnumber the CUs); other kinds deal R-row groups to
// waves, capped at
// LLMRS_GEMV_WG_PER_CU (default 2, the best of 1/2/4/8 measured on the 8B
// decode) workgroups per CU, beyond which waves loop.
GemvPlan gemv_plan(int wt, const std::string& kind, int n, int k, int num_cus) {
  const int nb = k / 32;
  int U = (nb % 128 == 0) ? 2 : 1;
  const char* eu = std::getenv("LLMRS_GEMV_U");
  if (eu && (std::atoi(eu) == 1 || std::atoi(eu) == 2)) U = std::atoi(eu);
  int R = 4;
  if (kind == "norm_store" || kind == "q8_resid" || kind == "nq_store" || kind == "q8b_store" ||
      kind == "q8b_resid") {
    R = 2;
    const char* er = std::getenv("LLMRS_GEMV_R");
    if (er && (std::atoi(er) == 2 || std::atoi(er) == 4)) R = std::atoi(er);
  }
  int waves = 4;
  if (kind == "q8_nq") {  // 32-row tiles, one per 8-wave workgroup (gemv_w8.hip)
    R = 2;
    waves = 8;
  }
  // SwiGLU with the RMSNorm prologue, more 64-row tiles than CUs: 8-wave
  // workgroups, one per CU (LLMRS_GEMV_SILU_W8=0/1 forces either)
  const char* es = std::getenv("LLMRS_GEMV_SILU_W8");
  const bool silu_w8 = kind == "norm_silu" && (es && *es ? std::atoi(es) == 1 : n / 64 > num_cus);
  if (silu_w8) waves = 8;
  // Workgroups per CU (measured on MI355X): 1 for the RMSNorm-prologue
  // store GEMV (Q|K|V: 8B 14 MB, 70B 47 MB) and for matrices under 24 MB -
  // fewer, longer-lived workgroups keep the activation loads from queueing
  // behind as many weight requests - and 2 otherwise.
  const double wbytes = (double)n * k * (wt == WT_Q8H ? 34.0 : wt == WT_Q4F ? 20.0 : 18.0) / 32.0;
  const char* ew = std::getenv("LLMRS_GEMV_WG_PER_CU");
  const bool store = kind == "norm_store" || kind == "nq_store";
  const int per_cu = ew && *ew ? std::max(1, std::atoi(ew)) : (store || silu_w8 || wbytes < 24e6 ? 1 : 2);
  const long cap = (long)std::max(1, num_cus) * per_cu;
  GemvPlan p;
  p.name = std::string("gemv_") + wt_tag(wt) + "_" + kind + "_r" + std::to_string(R) + "u" +
           std::to_string(U) + (waves == 8 ? "_w8" : "");
  p.threads = 64 * waves;
  // tiled epilogues: whole 64-row SwiGLU tiles or 32-row next-norm tiles
  const int tile = (kind == "norm_silu" || kind == "nq_silu" || kind == "q8b_silu") ? 64 : kind == "q8_nq" ? 32 : 0;
  long wgs;
  if (tile) {
    wgs = (n + tile - 1) / tile;
  } else {
    const long nrg = (n + R - 1) / R;
    wgs = (nrg + waves - 1) / waves;
  }
  p.grid = (unsigned)std::max<long>(1, std::min(wgs, cap));
  p.lds = llmrs::gemv_lds_bytes(tile, n, k, R, (int)p.grid, waves);
  return p;
}

// Whether m rows can run on the skinny GEMM: whole 128-element runs and up to
// 160 rows.
bool sgemm_serves(size_t m, size_t k) { return m <= 160 && k % 128 == 0; }

namespace {
struct GemmTile {
  int tt, rt;         // 64 tt tokens x 64 rt rows
  double lone, pair;  // time per block of 32: one workgroup on a CU, two
};
constexpr GemmTile kGemmTiles[] = {{2, 2, 2.9, 4.4}, {1, 2, 1.65, 2.5}, {1, 1, 1.0, 1.4}};

// The tile for m tokens x n rows, and its time per block of 32.  It follows
// from how the tiles fill the CUs: a CU works on two workgroups at once, and a
// lone one takes more than half the time of a pair (nothing covers its waves'
// latencies).  In units of a lone 64 x 64 tile's block (0.21 us) the tiles took
// the times above; the tile with the smallest sum over the fullest CU is
// taken.  8B down, us for 128 x 128 / 64 x 128 / 64 x 64: 256 rows 269 / 154 /
// 94, 1024 rows 297 / 237 / 255, 2048 rows 423 / 452 / 492; 1B O at 1500 rows
// 57 / 43 / 39, gate|up 231 / 245.
const GemmTile& gemm_tile(const std::string& epi, int m, int n, int num_cus, double* units) {
  const GemmTile* best = nullptr;
  for (const GemmTile& t : kGemmTiles) {
    if (epi == "silu" && t.rt == 1) continue;  // a gate and an up run of 32 per wave
    const long token_tiles = (m + 64 * t.tt - 1) / (64 * t.tt);
    if (t.tt == 1 && token_tiles > 65535) continue;  // past a grid's second dimension
    const long wgs = token_tiles * ((n + 64 * t.rt - 1) / (64 * t.rt));
    const long per_cu = (wgs + num_cus - 1) / num_cus;
    const double u = (double)(per_cu / 2) * t.pair + (double)(per_cu % 2) * t.lone;
    if (best && u >= *units) continue;
    best = &t;
    *units = u;
  }
  return *best;
}
}  // namespace

GemmPlan gemm_tile_plan(int wt, const std::string& epi, int m, int n, int tt, int rt) {
  const int bm = 64 * tt, bn = 64 * rt, bch = wt == WT_Q8H ? 2 : 1;
  GemmPlan p;
  p.name = std::string("gemm_") + wt_tag(wt) + "_" + epi + "_" + std::to_string(bm) + "x" + std::to_string(bn);
  p.grid = dim3((unsigned)((n + bn - 1) / bn), (unsigned)((m + bm - 1) / bm));
  p.lds = gemm_lds_bytes(tt, rt, gemm_stage_blocks(tt, rt, bch), bch);
  return p;
}

GemmPlan gemm_plan(int wt, const std::string& epi, int m, int n, int num_cus) {
  double units = 0;
  const GemmTile& t = gemm_tile(epi, m, n, num_cus, &units);
  return gemm_tile_plan(wt, epi, m, n, t.tt, t.rt);
}

// Either grid of the skinny GEMM deals eight row sets at a time, one per XCD,
// each over its token tiles.
static unsigned sgemm_deal(long rows, long tokens) { return (unsigned)(8 * tokens * ((rows + 7) / 8)); }

SgemmPlan sgemm_split_plan(int wt, const std::string& epi, int m, int n, int R) {
  SgemmPlan p;
  p.name = std::string("sgemm_") + wt_tag(wt) + "_" + epi + "_r" + std::to_string(R);
  p.grid = sgemm_deal(((long)n + 16 * R - 1) / (16 * R), (m + 15) / 16);
  p.threads = kSgemmThreads;
  return p;
}

SgemmPlan sgemm_wide_plan(int wt, const std::string& epi, int m, int n, int tt) {
  SgemmPlan p;
  p.name = std::string("sgemm_") + wt_tag(wt) + "_" + epi + "_w" + std::to_string(tt);
  p.grid = sgemm_deal(((long)n + 63) / 64, (m + 16 * tt - 1) / (16 * tt));
  p.threads = kWideThreads;
  return p;
}

// The skinny GEMM's kernel for m rows (16-token tiles) x n weight rows, and its
// time per block of 32 in gemm_tile's units; the 3 to 5 us that every launch takes
// besides are left out of all estimates.  The split kernels spread any shape over
// the chip: 0.0070 per token tile and num_cus weight rows.  Their row tiles per
// workgroup (R = 1, 2 or 4 tiles of 16 rows; eight waves share them) are the most
// that still leave every CU two workgroups, since a workgroup's rows share its
// activation loads; SwiGLU runs always span four.  The wide kernels (64 rows x 1, 2
// or 3 token tiles, a wave's tiles its own) win where that grid fills the chip, by
// the same sum over the fullest CU as the tile GEMM's.  Both sides, Q4_0, us under a
// kernel trace: 8B O r1 / r2 / w1 / w2 at 16 rows 6.9 / 8.8 / 14.4 / 19.4, 32 rows 9.2 / 9.2 /
// 14.4 / 20.2, 64 rows 15.8 / 13.8 / 15.3 / 21.2; 8B gate|up r4 / w1 / w2 / w3 at 16 rows
// 22.6 / 20.1 / 28.1 / 37.8, 32 rows 40.9 / 35.0 / 29.7 / 38.6, 48 rows 60.4 / 50.5 / 53.8 /
// 39.6; 1B gate|up at 64 rows 25.2 / 22.0 / 18.1 / 24.3.  The rule is not the best at every
// shape: 1B gate|up at 32 rows takes w2 (13.6) where w1 takes 12.3, a 1024 x 1024
// layer at 144 rows r1 (8.3) where r2 takes 5.4; over 400 shapes (16 to 160 rows, 17
// [n, k], all weight types) its kernel is 3.6 % slower than the best one (geometric
// mean).
SgemmPlan sgemm_plan(int wt, const std::string& epi, int m, int n, int num_cus) {
  const long nt = (m + 15) / 16;
  int R = 4;
  if (epi != "silu")
    while (R > 1 && ((long)n + 16 * R - 1) / (16 * R) * nt < 2 * num_cus) R /= 2;
  SgemmPlan p = sgemm_split_plan(wt, epi, m, n, R);
  p.units = 0.0070 * n / num_cus * nt;
  static const struct {
    double lone, pair;
  } kWide[] = {{0.40, 0.68}, {0.64, 1.0}, {0.95, 1.37}};
  const long rows = (n + 63) / 64;
  for (int tt = 1; tt <= (wt == WT_Q8H ? 2 : 3); ++tt) {  // three token tiles of Q8: one workgroup per CU
    const long tokens = (nt + tt - 1) / tt, per_cu = (rows * tokens + num_cus - 1) / num_cus;
    const double u = (double)(per_cu / 2) * kWide[tt - 1].pair + (double)(per_cu % 2) * kWide[tt - 1].lone;
    if (u >= p.units) continue;
    p = sgemm_wide_plan(wt, epi, m, n, tt);
    p.units = u;
  }
  return p;
}

// Whether the skinny GEMM is the faster one for m rows that it can run.  Where
// the estimates are close it is, by up to 5 %, and up to 22 % for SwiGLU, whose
// epilogue a tile's wave runs on 32 tokens at once; Q8_0's skinny kernels take
// about 10 % longer than the estimate, which is Q4's, and its tiles do not.
// Short rows (K = 1024) leave too little to pay for the skinny kernels' longer
// start.  Skinny / tile under a kernel trace, us: 8B gate|up at 64 rows 54.0 /
// 56.2, 96 rows 75.4 / 76.0; 8B O at 128 rows 20.4 / 28.9, 160 rows 29.6 / 31.7;
// 70B O at 112 rows 48.1 / 55.1; 8B Q|K|V in Q8_0 at 128 rows 28.3 / 26.4; 8192 x
// 1024 at 128 rows (a whole call) 12.5 / 11.8.  Over 400 shapes (16 to 160 rows, 17
// [n, k], all weight types) the kernel taken is 0.15 % slower than the better of
// the two (geometric mean), 0.43 % with the plain comparison.
bool sgemm_faster(int wt, const std::string& epi, int m, int n, int k, int num_cus) {
  if (!sgemm_serves((size_t)m, (size_t)k)) return false;
  double units = 0;
  (void)gemm_tile(epi, m, n, num_cus, &units);
  const double margin = k < 2048 ? 1.0 : epi == "silu" ? 1.22 : 1.05;
  return sgemm_plan(wt, epi, m, n, num_cus).units * (wt == WT_Q8H ? 1.10 : 1.0) < units * margin;
}

// ---- allocator -------------------------------------------------------------
void* Allocator::alloc(size_t bytes) {
  size_t sz = align_up(bytes ? bytes : 1, 256);
  if (sz > (1u << 20)) {  // round large requests to 1/8 octave to improve reuse
    size_t p = 1;
    while (p < sz) p <<= 1;
    size_t step = std::max<size_t>(p / 8, 256);
    sz = align_up(sz, step);
  }
  auto it = free_.find(sz);
  void* ptr = nullptr;
  if (it != free_.end()) {
    ptr = it->second;
    free_.erase(it);
  } else {
    hipError_t e = hipMalloc(&ptr, sz);
    if (e != hipSuccess) {
      (void)hipGetLastError();
      trim();
      e = hipMalloc(&ptr, sz);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      fail(LLMRS_E_OOM, "hipMalloc of " + std::to_string(sz) + " bytes failed");
    }
  }
  live_[ptr] = sz;
  return ptr;
}

void Allocator::release(void* p) {
  if (!p) return;
  auto it = live_.find(p);
  if (it == live_.end()) return;
  free_.emplace(it->second, p);
  live_.erase(it);
}

void Allocator::trim() {
  for (auto& kv : free_) (void)hipFree(kv.second);
  free_.clear();
}

// ---- host helpers ----------------------------------------------------------
uint16_t host_f2h(float f) { return _cvtss_sh(f, _MM_FROUND_TO_NEAREST_INT); }
float host_h2f(uint16_t h) { return _cvtsh_ss(h); }

bool scales_fit_f16(const float* scales, size_t count) {
  for (size_t i = 0; i < count; ++i) {
    float back = host_h2f(host_f2h(scales[i]));
    if (!(back == scales[i]) && !(std::isnan(back) && std::isnan(scales[i]))) return false;
  }
  return true;
}

void parallel_for(size_t n, int threads, const std::function<void(size_t, size_t)>& fn) {
  if (threads <= 0) threads = (int)std::max(1u, std::thread::hardware_concurrency());
  if (n < 2 || threads == 1) {
    if (n) fn(0, n);
    return;
  }
  size_t nt = std::min<size_t>((size_t)threads, n);
  size_t chunk = (n + nt - 1) / nt;
  std::vector<std::thread> ts;
  for (size_t t = 0; t < nt; ++t) {
    size_t b = t * chunk, e = std::min(n, b + chunk);
    if (b >= e) break;
    ts.emplace_back(fn, b, e);
  }
  for (auto& t : ts) t.join();
}

// Reference nibble order: byte i of a block = e[2i] | e[2i+1] << 4
// (tensor.rs:125-131).  Device order: byte i = e[i] | e[i+16] << 4, so that
// the low nibbles of a dword are four consecutive elements.
void repack_q4_rows(const uint8_t* qs, const float* scales, size_t rows, size_t k, int wt,
                    const std::vector<size_t>& row_map, uint8_t* dst_codes, uint8_t* dst_scales) {
  const size_t nb = k / 32;
  parallel_for(rows, 0, [&](size_t r0, size_t r1) {
    uint8_t e[32];
    for (size_t r = r0; r < r1; ++r) {
      const size_t dr = row_map.empty() ? r : row_map[r];
      for (size_t b = 0; b < nb; ++b) {
        const uint8_t* src = qs + r * (k / 2) + b * 16;
        for (int i = 0; i < 16; ++i) {
          e[2 * i] = src[i] & 0x0F;
          e[2 * i + 1] = src[i] >> 4;
        }
        uint8_t* dst = dst_codes + (dr * nb + b) * 16;
        for (int i = 0; i < 16; ++i) dst[i] = (uint8_t)(e[i] | (e[i + 16] << 4));
        const float s = scales[r * nb + b];
        if (wt == WT_Q4F) {
          std::memcpy(dst_scales + (dr * nb + b) * 4, &s, 4);
        } else {
          const uint16_t h = host_f2h(s);
          std::memcpy(dst_scales + (dr * nb + b) * 2, &h, 2);
        }
      }
    }
  });
}

void repack_q8_rows(const int8_t* qs, const float* scales, size_t rows, size_t k,
                    const std::vector<size_t>& row_map, uint8_t* dst_codes, uint8_t* dst_scales) {
  const size_t nb = k / 32;
  parallel_for(rows, 0, [&](size_t r0, size_t r1) {
    for (size_t r = r0; r < r1; ++r) {
      const size_t dr = row_map.empty() ? r : row_map[r];
      std::memcpy(dst_codes + dr * k, qs + r * k, k);
      for (size_t b = 0; b < nb; ++b) {
        const uint16_t h = host_f2h(scales[r * nb + b]);
        std::memcpy(dst_scales + (dr * nb + b) * 2, &h, 2);
      }
    }
  });
}

void rope_table(size_t pos0, size_t npos, int hd, float theta, float* cos_out, float* sin_out) {
  const int mid = hd / 2;
  std::vector<float> inv(mid);
  for (int j = 0; j < mid; ++j) {
    float freq_idx = ((float)j * 2.0f) / (float)hd;
    inv[j] = 1.0f / std::pow(theta, freq_idx);
  }
  for (size_t p = 0; p < npos; ++p)
    for (int j = 0; j < mid; ++j) {
      float a = (float)(pos0 + p) * inv[j];
      cos_out[p * mid + j] = std::cos(a);
      sin_out[p * mid + j] = std::sin(a);
    }
}

}  // namespace llmrs

using namespace llmrs;

extern "C" {

const char* llmrs_last_error(void) { return g_last_error.c_str(); }

int llmrs_init(int device_ordinal, const char* hsaco_dir) {
  return guard([&] {
    if (g_ctx) return;
    int count = 0;
    LLMRS_HIP(hipGetDeviceCount(&count));
    LLMRS_REQUIRE(device_ordinal >= 0 && device_ordinal < count, LLMRS_E_INVALID,
                  "no such HIP device: " + std::to_string(device_ordinal));
    auto* c = new Context();
    try {
      c->device = device_ordinal;
      LLMRS_HIP(hipSetDevice(device_ordinal));
      hipDeviceProp_t prop;
      LLMRS_HIP(hipGetDeviceProperties(&prop, device_ordinal));
      c->num_cus = prop.multiProcessorCount;
      LLMRS_HIP(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
      LLMRS_HIP(hipHostMalloc((void**)&c->host_out, kFetchBytes + 64, hipHostMallocDefault));
      // the no-allocation entry point's scratch, resolved with the device
      // current; a failure is reported by that entry point, not by init
      try {
        c->noalloc_scratch = noalloc_scratch_address();
      } catch (const Error& e) {
        c->noalloc_scratch = nullptr;
        c->noalloc_error = e.what();
      }
      std::string dir = hsaco_dir ? std::string(hsaco_dir) : library_dir();
      for (const char* name : {"gemv", "gemv_w8", "attention", "exact", "ops", "prefill", "sample", "sgemm"}) {
        std::string path = dir + "/" + name + ".hsaco";
        LLMRS_REQUIRE(std::filesystem::exists(path), LLMRS_E_MODULE, "missing code object " + path);
        hipModule_t m = nullptr;
        hipError_t e = hipModuleLoad(&m, path.c_str());
        if (e != hipSuccess)
          fail(LLMRS_E_MODULE, "hipModuleLoad(" + path + "): " + hipGetErrorString(e));
        c->modules.push_back(m);
      }
    } catch (...) {
      for (hipModule_t m : c->modules) (void)hipModuleUnload(m);
      if (c->stream) (void)hipStreamDestroy(c->stream);
      if (c->host_out) (void)hipHostFree(c->host_out);
      delete c;
      throw;
    }
    g_ctx = c;
  });
}

int llmrs_shutdown(void) {
  return guard([&] {
    if (!g_ctx) return;
    (void)hipStreamSynchronize(g_ctx->stream);
    g_ctx->alloc.trim();
    for (hipModule_t m : g_ctx->modules) (void)hipModuleUnload(m);
    (void)hipStreamDestroy(g_ctx->stream);
    (void)hipHostFree(g_ctx->host_out);
    delete g_ctx;
    g_ctx = nullptr;
  });
}

int llmrs_device(void) { return LLMRS_DEVICE_HIP; }
const char* llmrs_name(void) { return "Hip"; }

int llmrs_sync(void) {
  return guard([&] { LLMRS_HIP(hipStreamSynchronize(ctx().stream)); });
}

int llmrs_num_cus(void) { return g_ctx ? g_ctx->num_cus : 0; }

}  // extern "C"
