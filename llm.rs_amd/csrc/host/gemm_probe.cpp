// gemm_probe.cpp - test probes of the several-row GEMMs: which kernel a shape
// takes, and one launch of a given kernel.
#include <cstring>

#include "../kernel_args.h"
#include "internal.h"

using namespace llmrs;

namespace {

// A buffer of the caching allocator for the length of a call.
struct Scratch {
  void* p;
  explicit Scratch(size_t bytes) : p(ctx().alloc.alloc(bytes)) {}
  ~Scratch() { ctx().alloc.release(p); }
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
};

int weight_of(const char* tag) {
  for (int wt : {WT_Q4H, WT_Q4F, WT_Q8H})
    if (!std::strcmp(tag, wt_tag(wt))) return wt;
  fail(LLMRS_E_DTYPE, std::string("unknown weight type ") + tag);
}

void require_epilogue(const std::string& epi, size_t n) {
  LLMRS_REQUIRE(epi == "store" || epi == "resid" || epi == "silu", LLMRS_E_INVALID, "epilogue: store, resid or silu");
  LLMRS_REQUIRE(epi != "silu" || n % 64 == 0, LLMRS_E_INVALID, "silu: rows in runs of 64");
}

void require_shape(size_t m, size_t n, size_t k) {
  LLMRS_REQUIRE(m >= 1 && m <= 65535 * 128 && n >= 1 && n <= (1u << 24) && k >= 32 && k <= 32768 && k % 32 == 0,
                LLMRS_E_INVALID, "shape out of range");
}

}  // namespace

extern "C" {

int llmrs_probe_gemm_plan(const char* weight, const char* epi, size_t m, size_t n, size_t k, int num_cus, char* name,
                          uint32_t grid[2]) {
  return guard([&] {
    LLMRS_REQUIRE(weight && epi && name && grid && num_cus > 0, LLMRS_E_INVALID, "bad argument");
    require_epilogue(epi, n);
    require_shape(m, n, k);
    const int wt = weight_of(weight);
    std::string s;
    if (sgemm_faster(wt, epi, (int)m, (int)n, (int)k, num_cus)) {
      const SgemmPlan p = sgemm_plan(wt, epi, (int)m, (int)n, num_cus);
      s = p.name;
      grid[0] = p.grid;
      grid[1] = 1;
    } else {
      const GemmPlan p = gemm_plan(wt, epi, (int)m, (int)n, num_cus);
      s = p.name;
      grid[0] = p.grid.x;
      grid[1] = p.grid.y;
    }
    LLMRS_REQUIRE(s.size() < 64, LLMRS_E_INVALID, "kernel name too long");
    std::memcpy(name, s.c_str(), s.size() + 1);
  });
}

int llmrs_probe_gemm(const llmrs_tensor* a, const llmrs_tensor* w, const llmrs_tensor* res, const char* epi,
                     const char* variant, int order, float* y, int8_t* yq, float* yd) {
  return guard([&] {
    LLMRS_REQUIRE(a && w && epi && variant && y, LLMRS_E_INVALID, "null argument");
    LLMRS_REQUIRE(a->dtype == LLMRS_F32 && a->dims.size() == 2 && w->wt >= 0 && w->dims.size() == 2 &&
                      a->dims[1] == w->dims[1],
                  LLMRS_E_INVALID, "a [m, k] in f32 and a quantised w [n, k]");
    const size_t m = a->dims[0], k = a->dims[1], n = w->dims[0];
    const std::string e(epi), v(variant);
    const bool silu = e == "silu", resid = e == "resid", skinny = v[0] == 'r' || v[0] == 'w';
    require_epilogue(e, n);
    require_shape(m, n, k);
    LLMRS_REQUIRE(m <= 65535, LLMRS_E_INVALID, "too many rows for a probe");
    LLMRS_REQUIRE(!silu || (yq && yd && (order == kActNatural || (order == kActMfma && n / 2 % 128 == 0))),
                  LLMRS_E_INVALID, "silu: codes, scales and an operand order that its row length allows");
    LLMRS_REQUIRE(!resid || (res && res->dtype == LLMRS_F32 && res->dims == std::vector<size_t>({m, n})),
                  LLMRS_E_INVALID, "resid: an f32 tensor [m, n]");
    SgemmPlan sp;
    GemmPlan gp;
    if (skinny) {
      LLMRS_REQUIRE(k % 128 == 0, LLMRS_E_INVALID, "the skinny GEMM takes whole runs of 128 elements");
      const int c = v.size() == 2 ? v[1] - '0' : 0;
      LLMRS_REQUIRE(v[0] == 'r' ? c == 1 || c == 2 || c == 4 : c >= 1 && c <= 3, LLMRS_E_INVALID, "unknown variant " + v);
      sp = v[0] == 'r' ? sgemm_split_plan(w->wt, e, (int)m, (int)n, c) : sgemm_wide_plan(w->wt, e, (int)m, (int)n, c);
      (void)kernel(sp.name);  // fails where there is none
    } else {
      LLMRS_REQUIRE(v == "128x128" || v == "64x128" || v == "64x64", LLMRS_E_INVALID, "unknown variant " + v);
      gp = gemm_tile_plan(w->wt, e, (int)m, (int)n, v == "128x128" ? 2 : 1, v == "64x64" ? 1 : 2);
      (void)kernel(gp.name);
    }
    hipStream_t s = ctx().stream;
    const int act = skinny ? kActMfma : kActNatural;
    const size_t rows = act_rows(m), out = silu ? n / 2 : n;
    Scratch xq(rows * k), xd(rows * (k / 32) * 4), dy(m * out * 4);
    Scratch dq(silu ? rows * out : 1), dd(silu ? rows * (out / 32) * 4 : 1);
    PrefillRowArgs r{(const float*)a->data, nullptr, (int8_t*)xq.p, (float*)xd.p, (int)m, (int)k, 0.0f, act};
    launch("prefill_rows_q8", dim3((unsigned)m), dim3(256), gemv_act_lds_host((int)k), s, r);
    if (resid) LLMRS_HIP(hipMemcpyAsync(dy.p, res->data, m * n * 4, hipMemcpyDeviceToDevice, s));
    const float* rp = resid ? (const float*)dy.p : nullptr;
    int8_t* qp = silu ? (int8_t*)dq.p : nullptr;
    float* dp = silu ? (float*)dd.p : nullptr;
    if (skinny) {
      SgemmArgs g{(int8_t*)xq.p, (float*)xd.p, (const uint8_t*)w->data, w->scales, (float*)dy.p, rp, qp, dp,
                  (int)m, (int)n, (int)k, (int)out, order};
      launch(sp.name, dim3(sp.grid), dim3(sp.threads), 0, s, g);
    } else {
      PrefillGemmArgs g{(int8_t*)xq.p, (float*)xd.p, (const uint8_t*)w->data, w->scales, (float*)dy.p, rp, qp, dp,
                        (int)m, (int)n, (int)k, (int)out, gemm_group_m(), order};
      launch(gp.name, gp.grid, dim3(kGemmThreads), gp.lds, s, g);
    }
    fetch(y, dy.p, m * out * 4);
    if (!silu) return;
    std::vector<int8_t> hq(rows * out);
    std::vector<float> hd(rows * out / 32);
    fetch(hq.data(), dq.p, hq.size());
    fetch(hd.data(), dd.p, hd.size() * 4);
    for (size_t t = 0; t < m; ++t) {
      for (size_t i = 0; i < out; ++i) yq[t * out + i] = hq[act_row(t, out, order) + act_offset((int)i, order)];
      for (size_t b = 0; b < out / 32; ++b)
        yd[t * (out / 32) + b] = hd[act_scale_row(t, out / 32, order) + act_scale_offset((int)b, order)];
    }
  });
}

}  // extern "C"
