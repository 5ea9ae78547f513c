// Plain bf16 GEMM entry points over the MFMA core:
//   C = alpha * op(A) op(B) + beta * C     (fp32 accumulation, C bf16 or fp32)
// with K optionally split into segments (K-concatenated operands).
#include "gemm_core.h"

namespace mla {
namespace gemm {
namespace {

int run(int64_t M, int64_t N, int nseg, const Segment* segs, int la, int lb, void* C, int64_t ldc,
        int c_dtype, float alpha, float beta, void* ws, size_t ws_bytes, void* stream) {
  ML_CHECK(M > 0 && N > 0 && M < (1LL << 31) && N < (1LL << 31), "gemm: bad M=%lld N=%lld",
           (long long)M, (long long)N);
  ML_CHECK(la == kKMajor || la == kMNMajor, "gemm: bad A layout %d", la);
  ML_CHECK(lb == kKMajor || lb == kMNMajor, "gemm: bad B layout %d", lb);
  ML_CHECK(C != nullptr && ldc >= N, "gemm: bad C (ldc %lld < N %lld)", (long long)ldc,
           (long long)N);
  // the bf16 store epilogue writes rows of 8 columns as 16-byte vectors
  ML_CHECK(c_dtype != ML_BF16 || (ldc % 8 == 0 && aligned16(C)),
           "gemm: a bf16 C needs ldc a multiple of 8 and a 16-byte aligned base (ldc %lld)",
           (long long)ldc);
  hipStream_t st = (hipStream_t)stream;
  // r4 is the faster engine when A is K-major, the big engine otherwise
  if (la == kKMajor) {
    float* w = static_cast<float*>(ws);
    if (c_dtype == ML_F32)
      return run_product((int)M, (int)N, nseg, segs, lb, static_cast<float*>(C), ldc, alpha, beta,
                         w, ws_bytes, st);
    if (c_dtype == ML_BF16)
      return run_product((int)M, (int)N, nseg, segs, lb, static_cast<bf16*>(C), ldc, alpha, beta,
                         w, ws_bytes, st);
  } else {
    Problem pb;
    int rc = make_problem<BigCfg>(pb, (int)M, (int)N, nseg, segs, la, lb, 0);
    if (rc) return rc;
    if (c_dtype == ML_F32) return launch_store<float>(pb, la, lb, C, ldc, alpha, beta, st);
    if (c_dtype == ML_BF16) return launch_store<bf16>(pb, la, lb, C, ldc, alpha, beta, st);
  }
  set_error("gemm: C dtype %d not supported (fp32 or bf16)", c_dtype);
  return ML_ERR_INVALID;
}

// Split-K / tile-shape variant (cfg 0: 256x256, 1: 256x32, 2: 64x256).
template <class C, typename TC>
int run_splitk_cfg(const Problem& pb, int la, int lb, float* ws, TC* out, int64_t ldo, float alpha,
                   float beta, hipStream_t st) {
  if (la == kKMajor && lb == kKMajor) return launch_splitk<C, kKMajor, kKMajor, TC>(pb, ws, out, ldo, alpha, beta, st);
  if (la == kKMajor && lb == kMNMajor) return launch_splitk<C, kKMajor, kMNMajor, TC>(pb, ws, out, ldo, alpha, beta, st);
  if (la == kMNMajor && lb == kKMajor) return launch_splitk<C, kMNMajor, kKMajor, TC>(pb, ws, out, ldo, alpha, beta, st);
  return launch_splitk<C, kMNMajor, kMNMajor, TC>(pb, ws, out, ldo, alpha, beta, st);
}

template <class C>
int run_splitk(int64_t M, int64_t N, const Segment& seg, int la, int lb, int ksplit, void* C_,
               int64_t ldc, int c_dtype, float alpha, float beta, void* ws, size_t ws_bytes,
               hipStream_t st) {
  Problem pb;
  int rc = make_problem<C>(pb, (int)M, (int)N, 1, &seg, la, lb, 0, ksplit);
  if (rc) return rc;
  ML_CHECK(ws && ws_bytes >= splitk_ws_bytes(pb), "gemm: split-K workspace too small (%zu < %zu)",
           ws_bytes, splitk_ws_bytes(pb));
  float* w = static_cast<float*>(ws);
  if (c_dtype == ML_F32)
    return run_splitk_cfg<C, float>(pb, la, lb, w, static_cast<float*>(C_), ldc, alpha, beta, st);
  if (c_dtype == ML_BF16)
    return run_splitk_cfg<C, bf16>(pb, la, lb, w, static_cast<bf16*>(C_), ldc, alpha, beta, st);
  set_error("gemm: C dtype %d not supported (fp32 or bf16)", c_dtype);
  return ML_ERR_INVALID;
}

// The same for the r4 engine's tiles (A K-major); one split stores C directly.
template <class C>
int run_splitk_r4(int64_t M, int64_t N, const Segment& seg, int la, int lb, int ksplit, void* C_,
                  int64_t ldc, int c_dtype, float alpha, float beta, void* ws, size_t ws_bytes,
                  hipStream_t st) {
  ML_CHECK(la == kKMajor, "gemm: this tile takes a K-major A");
  ML_CHECK(c_dtype == ML_F32 || c_dtype == ML_BF16, "gemm: C dtype %d not supported (fp32 or bf16)",
           c_dtype);
  ML_CHECK(c_dtype != ML_BF16 || (ldc % 8 == 0 && aligned16(C_)),
           "gemm: a bf16 C needs ldc a multiple of 8 and a 16-byte aligned base (ldc %lld)",
           (long long)ldc);
  Problem pb;
  int rc = make_problem<C>(pb, (int)M, (int)N, 1, &seg, la, lb, 0, ksplit);
  if (rc) return rc;
  if (pb.ksplit == 1)
    return c_dtype == ML_F32 ? launch_store<float, C>(pb, la, lb, C_, ldc, alpha, beta, st)
                             : launch_store<bf16, C>(pb, la, lb, C_, ldc, alpha, beta, st);
  ML_CHECK(ws && ws_bytes >= splitk_ws_bytes(pb), "gemm: split-K workspace too small (%zu < %zu)",
           ws_bytes, splitk_ws_bytes(pb));
  float* w = static_cast<float*>(ws);
  auto go = [&](auto* out) {
    using TC = std::remove_pointer_t<decltype(out)>;
    return lb == kKMajor
               ? launch_splitk<C, kKMajor, kKMajor, TC>(pb, w, out, ldc, alpha, beta, st)
               : launch_splitk<C, kKMajor, kMNMajor, TC>(pb, w, out, ldc, alpha, beta, st);
  };
  return c_dtype == ML_F32 ? go(static_cast<float*>(C_)) : go(static_cast<bf16*>(C_));
}

}  // namespace
}  // namespace gemm
}  // namespace mla

using namespace mla;

extern "C" int ml_gemm_bf16(int64_t M, int64_t N, int64_t K, const void* A, int64_t lda,
                            int a_layout, const void* B, int64_t ldb, int b_layout, void* C,
                            int64_t ldc, int c_dtype, float alpha, float beta, void* stream) {
  ML_CHECK(K >= 0 && K < (1LL << 31), "gemm: bad K=%lld", (long long)K);
  gemm::Segment s{{static_cast<const bf16*>(A), lda}, {static_cast<const bf16*>(B), ldb}, (int)K};
  return gemm::run(M, N, 1, &s, a_layout, b_layout, C, ldc, c_dtype, alpha, beta, nullptr, 0,
                   stream);
}

extern "C" int ml_gemm_bf16_segments(int64_t M, int64_t N, int nseg, const int64_t* k_lens,
                                     const void* const* a_ptrs, const int64_t* ldas,
                                     const void* const* b_ptrs, const int64_t* ldbs, int a_layout,
                                     int b_layout, void* C, int64_t ldc, int c_dtype, float alpha,
                                     float beta, void* stream) {
  return ml_gemm_bf16_segments_ws(M, N, nseg, k_lens, a_ptrs, ldas, b_ptrs, ldbs, a_layout,
                                  b_layout, C, ldc, c_dtype, alpha, beta, nullptr, 0, stream);
}

extern "C" size_t ml_gemm_bf16_segments_workspace_bytes(int64_t M, int64_t N, int nseg,
                                                        const int64_t* k_lens) {
  if (M <= 0 || N <= 0 || M >= (1LL << 31) || N >= (1LL << 31) || !k_lens) return 0;
  int64_t kt = 0;
  for (int s = 0; s < nseg; ++s) {
    if (k_lens[s] < 0 || k_lens[s] >= (1LL << 31)) return 0;
    kt += (k_lens[s] + gemm::kBK - 1) / gemm::kBK;
  }
  return kt < (1LL << 31) ? gemm::product_ws_bytes((int)M, (int)N, (int)kt) : 0;
}

extern "C" int ml_gemm_bf16_segments_ws(int64_t M, int64_t N, int nseg, const int64_t* k_lens,
                                        const void* const* a_ptrs, const int64_t* ldas,
                                        const void* const* b_ptrs, const int64_t* ldbs,
                                        int a_layout, int b_layout, void* C, int64_t ldc,
                                        int c_dtype, float alpha, float beta, void* workspace,
                                        size_t workspace_bytes, void* stream) {
  ML_CHECK(nseg >= 1 && nseg <= gemm::kMaxSeg, "gemm: 1..%d segments supported (got %d)",
           gemm::kMaxSeg, nseg);
  ML_CHECK(k_lens && a_ptrs && ldas && b_ptrs && ldbs, "gemm: null segment arrays");
  gemm::Segment segs[gemm::kMaxSeg];
  for (int s = 0; s < nseg; ++s) {
    ML_CHECK(k_lens[s] >= 0 && k_lens[s] < (1LL << 31), "gemm: bad K segment %d", s);
    segs[s] = gemm::Segment{{static_cast<const bf16*>(a_ptrs[s]), ldas[s]},
                            {static_cast<const bf16*>(b_ptrs[s]), ldbs[s]}, (int)k_lens[s]};
  }
  return gemm::run(M, N, nseg, segs, a_layout, b_layout, C, ldc, c_dtype, alpha, beta, workspace,
                   workspace_bytes, stream);
}

extern "C" int ml_gemm_bf16_segments_group(int count, const int64_t* M, const int64_t* N,
                                           const int* nseg, const int64_t* k_lens,
                                           const void* const* a_ptrs, const int64_t* ldas,
                                           const void* const* b_ptrs, const int64_t* ldbs,
                                           int b_layout, void* const* C, const int64_t* ldc,
                                           int c_dtype, float alpha, float beta, void* stream) {
  ML_CHECK(count >= 1 && count <= gemm::kMaxGroup, "gemm group: 1..%d products (got %d)",
           gemm::kMaxGroup, count);
  ML_CHECK(M && N && nseg && k_lens && a_ptrs && ldas && b_ptrs && ldbs && C && ldc,
           "gemm group: null argument arrays");
  ML_CHECK(b_layout == gemm::kKMajor || b_layout == gemm::kMNMajor, "gemm group: bad B layout");
  gemm::Problem pbs[gemm::kMaxGroup];
  gemm::Segment segs[gemm::kMaxGroup][gemm::kMaxSeg];
  int ms[gemm::kMaxGroup], ns[gemm::kMaxGroup], kts[gemm::kMaxGroup];
  int base = 0;
  for (int g = 0; g < count; ++g) {
    ML_CHECK(M[g] > 0 && N[g] > 0 && M[g] < (1LL << 31) && N[g] < (1LL << 31),
             "gemm group: bad M=%lld N=%lld (product %d)", (long long)M[g], (long long)N[g], g);
    ML_CHECK(C[g] != nullptr && ldc[g] >= N[g], "gemm group: bad C (product %d)", g);
    ML_CHECK(c_dtype != ML_BF16 || (ldc[g] % 8 == 0 && aligned16(C[g])),
             "gemm group: a bf16 C needs ldc a multiple of 8 and a 16-byte aligned base "
             "(product %d, ldc %lld)", g, (long long)ldc[g]);
    ML_CHECK(nseg[g] >= 1 && nseg[g] <= gemm::kMaxSeg, "gemm group: 1..%d segments (product %d)",
             gemm::kMaxSeg, g);
    for (int s = 0; s < nseg[g]; ++s) {
      const int q = base + s;
      ML_CHECK(k_lens[q] >= 0 && k_lens[q] < (1LL << 31), "gemm group: bad K segment %d", q);
      segs[g][s] = gemm::Segment{{static_cast<const bf16*>(a_ptrs[q]), ldas[q]},
                              {static_cast<const bf16*>(b_ptrs[q]), ldbs[q]}, (int)k_lens[q]};
    }
    ms[g] = (int)M[g];
    ns[g] = (int)N[g];
    kts[g] = gemm::segment_ktiles(nseg[g], segs[g]);
    base += nseg[g];
  }
  const bool small = gemm::plan_products(count, ms, ns, kts, false).tile == 128;
  for (int g = 0; g < count; ++g) {
    const int rc = small ? gemm::make_problem<gemm::R4SCfg>(pbs[g], ms[g], ns[g], nseg[g], segs[g],
                                                            gemm::kKMajor, b_layout, 0)
                         : gemm::make_problem<gemm::R4Cfg>(pbs[g], ms[g], ns[g], nseg[g], segs[g],
                                                           gemm::kKMajor, b_layout, 0);
    if (rc) return rc;
  }
  hipStream_t st = (hipStream_t)stream;
  auto go = [&](auto tc) {
    using TC = decltype(tc);
    return small ? gemm::launch_store_group<gemm::R4SCfg, TC>(pbs, count, b_layout, C, ldc, alpha,
                                                              beta, st)
                 : gemm::launch_store_group<gemm::R4Cfg, TC>(pbs, count, b_layout, C, ldc, alpha,
                                                             beta, st);
  };
  if (c_dtype == ML_BF16) return go(bf16{});
  if (c_dtype == ML_F32) return go(float{});
  set_error("gemm group: C dtype %d not supported (fp32 or bf16)", c_dtype);
  return ML_ERR_INVALID;
}

extern "C" size_t ml_gemm_splitk_workspace_bytes(int64_t M, int64_t N, int64_t K, int ksplit) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int64_t total = (K + gemm::kBK - 1) / gemm::kBK;
  const int64_t ks = ksplit < 1 ? 1 : ksplit;
  const int64_t kps = (total + ks - 1) / ks;
  const int64_t splits = (total + kps - 1) / kps;
  return (size_t)(splits * M * N) * sizeof(float);
}

extern "C" int ml_gemm_bf16_splitk(int64_t M, int64_t N, int64_t K, const void* A, int64_t lda,
                                   int a_layout, const void* B, int64_t ldb, int b_layout, void* C,
                                   int64_t ldc, int c_dtype, float alpha, float beta, int tile_cfg,
                                   int ksplit, void* workspace, size_t workspace_bytes,
                                   void* stream) {
  ML_CHECK(M > 0 && N > 0 && M < (1LL << 31) && N < (1LL << 31), "gemm: bad M=%lld N=%lld",
           (long long)M, (long long)N);
  ML_CHECK(K > 0 && K < (1LL << 31), "gemm: bad K=%lld", (long long)K);
  ML_CHECK(a_layout == gemm::kKMajor || a_layout == gemm::kMNMajor, "gemm: bad A layout");
  ML_CHECK(b_layout == gemm::kKMajor || b_layout == gemm::kMNMajor, "gemm: bad B layout");
  ML_CHECK(C != nullptr && ldc >= N, "gemm: bad C");
  ML_CHECK(ksplit >= 1, "gemm: ksplit must be >= 1");
  gemm::Segment s{{static_cast<const bf16*>(A), lda}, {static_cast<const bf16*>(B), ldb}, (int)K};
  hipStream_t st = (hipStream_t)stream;
  auto go = [&](auto fn) {
    return fn(M, N, s, a_layout, b_layout, ksplit, C, ldc, c_dtype, alpha, beta, workspace,
              workspace_bytes, st);
  };
  switch (tile_cfg) {
    case 0: return go(gemm::run_splitk<gemm::BigCfg>);
    case 1: return go(gemm::run_splitk<gemm::TallCfg>);
    case 2: return go(gemm::run_splitk<gemm::WideCfg>);
    case 3: return go(gemm::run_splitk_r4<gemm::R4SCfg>);
    case 4: return go(gemm::run_splitk_r4<gemm::R4Cfg>);
    default:
      set_error("gemm: tile_cfg must be 0 (256x256), 1 (256x32), 2 (64x256), 3 (128x128) or 4 "
                "(256x256, K-major A)");
      return ML_ERR_INVALID;
  }
}
