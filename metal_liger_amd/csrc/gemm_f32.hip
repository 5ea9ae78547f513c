// fp32 GEMM on the matrix cores (v_mfma_f32_32x32x2_f32, full fp32
// products and sums) for the fp32 forms of the LoRA and fused linear
// cross-entropy ops (the reference runs them in whatever float dtype the
// model has, ops/fused_lora.py:69-82, ops/fused_linear_cross_entropy.py:108):
//
//   C[M, N] = alpha * sum_seg op(A_s) op(B_s) + beta * C      (all fp32)
//
// Operand layouts as in the bf16 engine: K-major element (r, k) at
// p[r * ld + k], MN-major at p[k * ld + r]; K may be a list of up to 8
// segments with their own pointers (K-concatenated operands).
//
// Tiles: 4 waves (2 x 2) share a BM x BN tile, a wave owns (BM / 2) x (BN / 2)
// of it as MFMA tiles of 32 x 32; k-tiles of BK are staged global -> registers
// -> LDS (two stages). LDS holds each operand as BK k-planes of BM (BN)
// values, with a pitch that spreads both the stores (4 consecutive k of a
// K-major row, or 4 consecutive rows of an MN-major k-plane) and the fragment
// reads (32 consecutive rows of one plane per half-wave) over the banks. Rows
// past M / N re-read the last row (never stored); k past a segment's end is
// zero-filled.
//
// Bound by the fp32 matrix cores (157 TFLOP/s; one MFMA takes 64 cycles of a
// SIMD) where the tiles fill the chip, and by latency where they do not: a
// wave with no other wave beside it waits for every k-tile's loads. Products
// here are often small ([1000, 2048] x 2048, or N = one LoRA rank), so:
//   * 64 x 64 tiles, four blocks per CU, unless 128 x 128 tiles alone give
//     two blocks per CU (they read half as much per product): [1000, 2048] x
//     2064 as 512 small tiles takes 110 us, as 128 large ones 200; [2048,
//     2048] x 2064, 1024 tiles, 196 us (88 TFLOP/s; the matrix cores 70%
//     busy) against 207;
//   * K split over blocks until there are two blocks per CU, at least
//     kMinSplitTiles k-tiles each: fp32 partials in the caller's workspace,
//     summed in split order by a second kernel (deterministic). Without a
//     workspace there is no split. [1000, 16] x 2048: 12 + 4 us against 100.
// A LoRA projection of [1000, 2048] to 2048, forward and backward: 1099 us of
// GPU time as 128 x 128 tiles without a split, 278 us.
#include <algorithm>

#include "common.h"

namespace mla {
namespace gemmf32 {
namespace {

typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
// four consecutive floats at any float address (global loads need no more)
typedef float f32x4_u __attribute__((ext_vector_type(4), aligned(4)));

constexpr int kThreads = 256;
constexpr int kMaxSeg = 8;
constexpr int kMaxSplit = 32;
constexpr int kMinSplitTiles = 4;
enum : int { kKMajor = 0, kMNMajor = 1 };

// One operand's staged k-tile: ROWS rows x BK k.
template <int L, int ROWS, int BK>
struct Stage {
  // K-major stores: lanes cover BK / 4 groups of 4 planes x 64 / (BK / 4)
  // rows, so 4 planes have to move the bank by the rows per group. MN-major
  // stores and reads are consecutive; the pitch only keeps 16-byte alignment.
  static constexpr int kPitch = ROWS + (L == kKMajor ? (BK == 16 ? 4 : 2) : 4);
  static constexpr int kFloats = BK * kPitch;
  static constexpr int kVecs = ROWS * BK / 4 / kThreads;  // float4 per thread
  static_assert(kVecs * 4 * kThreads == ROWS * BK, "whole float4s per thread");

  // K-major: thread t covers row t / (BK / 4) + ..., k 4 (t % (BK / 4)) .. + 3.
  // MN-major: k-plane t / (ROWS / 4) + ..., rows 4 (t % (ROWS / 4)) .. + 3.
  static __device__ __forceinline__ void load(f32x4_t (&v)[kVecs], const float* p, int64_t ld,
                                              int row0, int rows, int k0, int klen) {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      if constexpr (L == kKMajor) {
        constexpr int G = BK / 4;
        int r = row0 + t / G + kThreads / G * i;
        r = r < rows ? r : rows - 1;
        const int k = k0 + 4 * (t % G);
        const float* q = p + (int64_t)r * ld + k;
        if (k + 4 <= klen) {
          v[i] = *reinterpret_cast<const f32x4_u*>(q);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[i][e] = (k + e < klen) ? q[e] : 0.f;
        }
      } else {
        constexpr int G = ROWS / 4;
        const int k = k0 + t / G + kThreads / G * i;
        const int r = row0 + 4 * (t % G);
        const float* q = p + (int64_t)k * ld;
        if (k >= klen) {
          v[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        } else if (r + 4 <= rows) {
          v[i] = *reinterpret_cast<const f32x4_u*>(q + r);
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) v[i][e] = q[r + e < rows ? r + e : rows - 1];
        }
      }
    }
  }

  static __device__ __forceinline__ void store(const f32x4_t (&v)[kVecs], float* lds) {
    const int t = threadIdx.x;
#pragma unroll
    for (int i = 0; i < kVecs; ++i) {
      if constexpr (L == kKMajor) {
        constexpr int G = BK / 4;
        const int r = t / G + kThreads / G * i;
        const int k = 4 * (t % G);
#pragma unroll
        for (int e = 0; e < 4; ++e) lds[(k + e) * kPitch + r] = v[i][e];
      } else {
        constexpr int G = ROWS / 4;
        const int k = t / G + kThreads / G * i;
        *reinterpret_cast<f32x4_t*>(lds + k * kPitch + 4 * (t % G)) = v[i];
      }
    }
  }
};

struct Seg {
  const float* a;
  const float* b;
  int64_t lda, ldb;
  int k_len;
};

struct Prob {
  int M, N, nseg;
  Seg seg[kMaxSeg];
  float* C;
  int64_t ldc;
  float alpha, beta;
  float* partial;  // [nsplit][M][N] when nsplit > 1 (C, alpha, beta: the reduction's)
  int nsplit;
};

template <int BM, int BN, int BK, int LA, int LB>
__global__ __launch_bounds__(kThreads) void gemm_f32_kernel(const Prob pb) {
  using SA = Stage<LA, BM, BK>;
  using SB = Stage<LB, BN, BK>;
  constexpr int TM = BM / 64, TN = BN / 64;  // MFMA tiles per wave
  __shared__ __attribute__((aligned(16))) float lds[2][SA::kFloats + SB::kFloats];
  const int tiles_m = (pb.M + BM - 1) / BM;
  const int tm = blockIdx.x % tiles_m, tn = blockIdx.x / tiles_m;
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = (wave >> 1) * (BM / 2), wn = (wave & 1) * (BN / 2);
  f32x16_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

  // k-tiles [kt, kt_end) of the concatenated segments are this split's
  int nk = 0;
  for (int s = 0; s < pb.nseg; ++s) nk += (pb.seg[s].k_len + BK - 1) / BK;
  int kt = (int)((int64_t)nk * blockIdx.y / pb.nsplit);
  const int kt_end = (int)((int64_t)nk * (blockIdx.y + 1) / pb.nsplit);
  if (kt < kt_end) {
    int seg = 0, k0 = kt;
    for (;; ++seg) {
      const int n = (pb.seg[seg].k_len + BK - 1) / BK;
      if (k0 < n) break;
      k0 -= n;
    }
    k0 *= BK;
    f32x4_t ra[SA::kVecs], rb[SB::kVecs];
    auto load = [&]() {
      const Seg& sg = pb.seg[seg];
      SA::load(ra, sg.a, sg.lda, m0, pb.M, k0, sg.k_len);
      SB::load(rb, sg.b, sg.ldb, n0, pb.N, k0, sg.k_len);
    };
    auto advance = [&]() {
      k0 += BK;
      if (k0 >= pb.seg[seg].k_len) {
        k0 = 0;
        do {
          ++seg;
        } while (seg < pb.nseg && pb.seg[seg].k_len == 0);
      }
    };
    load();
    SA::store(ra, lds[0]);
    SB::store(rb, lds[0] + SA::kFloats);
    __syncthreads();
    for (int buf = 0; kt < kt_end; ++kt, buf ^= 1) {
      const bool more = kt + 1 < kt_end;
      if (more) {
        advance();
        load();
      }
      const float* As = lds[buf] + (lane >> 5) * SA::kPitch + wm + (lane & 31);
      const float* Bs = lds[buf] + SA::kFloats + (lane >> 5) * SB::kPitch + wn + (lane & 31);
#pragma unroll
      for (int ks = 0; ks < BK; ks += 2) {
        float a[TM], b[TN];
#pragma unroll
        for (int i = 0; i < TM; ++i) a[i] = As[ks * SA::kPitch + 32 * i];
#pragma unroll
        for (int j = 0; j < TN; ++j) b[j] = Bs[ks * SB::kPitch + 32 * j];
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[j], acc[i][j], 0, 0, 0);
      }
      if (more) {
        SA::store(ra, lds[buf ^ 1]);
        SB::store(rb, lds[buf ^ 1] + SA::kFloats);
      }
      __syncthreads();
    }
  }
  const bool split = pb.nsplit > 1;
  float* out = split ? pb.partial + (int64_t)blockIdx.y * pb.M * pb.N : pb.C;
  const int64_t ldo = split ? pb.N : pb.ldc;
  const float alpha = split ? 1.f : pb.alpha, beta = split ? 0.f : pb.beta;
  // element v of tile (i, j): row wm + 32 i + 8 (v / 4) + 4 (lane / 32) + v % 4,
  // column wn + 32 j + lane % 32
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + wn + 32 * j + (lane & 31);
      if (n >= pb.N) continue;
#pragma unroll
      for (int v = 0; v < 16; ++v) {
        const int m = m0 + wm + 32 * i + 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        if (m < pb.M) {
          float* c = out + (int64_t)m * ldo + n;
          float o = alpha * acc[i][j][v];
          if (beta != 0.f) o += beta * *c;
          *c = o;
        }
      }
    }
}

// C = alpha * (sum of the partials in split order) + beta * C.
__global__ __launch_bounds__(kThreads) void reduce_f32_kernel(const float* __restrict__ partial,
                                                              int nsplit, int64_t M, int64_t N,
                                                              float* __restrict__ C, int64_t ldc,
                                                              float alpha, float beta) {
  const int64_t n_all = M * N;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < n_all;
       i += (int64_t)gridDim.x * kThreads) {
    float sum = 0.f;
#pragma unroll 8
    for (int s = 0; s < nsplit; ++s) sum += partial[s * n_all + i];
    float* c = C + i / N * ldc + i % N;
    float o = alpha * sum;
    if (beta != 0.f) o += beta * *c;
    *c = o;
  }
}

struct Choice {
  bool big;    // 128 x 128 tiles (else 64 x 64)
  int nsplit;  // K splits, given a workspace
};

// k_len: the summed K of all segments (its k-tiles, to within a rounding per
// segment).
Choice choose(int64_t M, int64_t N, int64_t k_len) {
  const int64_t cus = num_cus();
  const int64_t big = ((M + 127) / 128) * ((N + 127) / 128);
  if (big >= 2 * cus) return {true, 1};
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64);
  const int64_t most = k_len / (32 * kMinSplitTiles);
  const int64_t want = std::min<int64_t>({2 * cus / tiles, most, kMaxSplit});
  return {false, (int)std::max<int64_t>(want, 1)};
}

}  // namespace
}  // namespace gemmf32
}  // namespace mla

using namespace mla;

extern "C" size_t ml_gemm_f32_workspace_bytes(int64_t M, int64_t N, int64_t K) {
  if (M <= 0 || N <= 0 || K <= 0) return 0;
  const int nsplit = gemmf32::choose(M, N, K).nsplit;
  return nsplit > 1 ? (size_t)nsplit * M * N * sizeof(float) : 0;
}

extern "C" int ml_gemm_f32_segments_ws(int64_t M, int64_t N, int nseg, const int64_t* k_lens,
                                       const void* const* a_ptrs, const int64_t* ldas,
                                       const void* const* b_ptrs, const int64_t* ldbs,
                                       int a_layout, int b_layout, float* C, int64_t ldc,
                                       float alpha, float beta, void* workspace,
                                       size_t workspace_bytes, void* stream) {
  using namespace gemmf32;
  ML_CHECK(M > 0 && N > 0 && M < (1LL << 31) && N < (1LL << 31), "gemm f32: bad M=%lld N=%lld",
           (long long)M, (long long)N);
  ML_CHECK(nseg >= 1 && nseg <= kMaxSeg, "gemm f32: 1..%d segments supported (got %d)", kMaxSeg,
           nseg);
  ML_CHECK(k_lens && a_ptrs && ldas && b_ptrs && ldbs, "gemm f32: null segment arrays");
  ML_CHECK(a_layout == kKMajor || a_layout == kMNMajor, "gemm f32: bad A layout %d", a_layout);
  ML_CHECK(b_layout == kKMajor || b_layout == kMNMajor, "gemm f32: bad B layout %d", b_layout);
  ML_CHECK(C != nullptr && ldc >= N, "gemm f32: bad C (ldc %lld < N %lld)", (long long)ldc,
           (long long)N);
  Prob pb{};
  pb.M = (int)M;
  pb.N = (int)N;
  pb.nseg = nseg;
  pb.C = C;
  pb.ldc = ldc;
  pb.alpha = alpha;
  pb.beta = beta;
  int64_t k_sum = 0;
  for (int s = 0; s < nseg; ++s) {
    ML_CHECK(k_lens[s] >= 0 && k_lens[s] < (1LL << 31), "gemm f32: bad K segment %d", s);
    Seg& g = pb.seg[s];
    g.a = static_cast<const float*>(a_ptrs[s]);
    g.b = static_cast<const float*>(b_ptrs[s]);
    g.lda = ldas[s];
    g.ldb = ldbs[s];
    g.k_len = (int)k_lens[s];
    k_sum += k_lens[s];
    if (g.k_len == 0) continue;
    ML_CHECK(g.a && g.b, "gemm f32: null operand in segment %d", s);
    ML_CHECK(a_layout == kKMajor ? g.lda >= g.k_len : g.lda >= M,
             "gemm f32: A leading dimension %lld too small in segment %d", (long long)g.lda, s);
    ML_CHECK(b_layout == kKMajor ? g.ldb >= g.k_len : g.ldb >= N,
             "gemm f32: B leading dimension %lld too small in segment %d", (long long)g.ldb, s);
  }
  const Choice ch = choose(M, N, k_sum);
  const bool split = ch.nsplit > 1 && workspace != nullptr &&
                     workspace_bytes >= (size_t)ch.nsplit * M * N * sizeof(float);
  pb.nsplit = split ? ch.nsplit : 1;
  pb.partial = static_cast<float*>(workspace);
  const int64_t bt = ch.big ? 128 : 64;
  const int64_t tiles = ((M + bt - 1) / bt) * ((N + bt - 1) / bt);
  ML_CHECK(tiles <= 0x7fffffffLL, "gemm f32: too many tiles");
  hipStream_t st = (hipStream_t)stream;
  const dim3 grid((unsigned)tiles, (unsigned)pb.nsplit);
#define ML_GF(LA, LB)                                                              \
  if (ch.big)                                                                      \
    gemm_f32_kernel<128, 128, 16, LA, LB><<<grid, kThreads, 0, st>>>(pb);          \
  else                                                                             \
    gemm_f32_kernel<64, 64, 32, LA, LB><<<grid, kThreads, 0, st>>>(pb)
  if (a_layout == kKMajor && b_layout == kKMajor) {
    ML_GF(kKMajor, kKMajor);
  } else if (a_layout == kKMajor) {
    ML_GF(kKMajor, kMNMajor);
  } else if (b_layout == kKMajor) {
    ML_GF(kMNMajor, kKMajor);
  } else {
    ML_GF(kMNMajor, kMNMajor);
  }
#undef ML_GF
  ML_LAUNCH_CHECK();
  if (split) {
    const int64_t blocks = std::min<int64_t>((M * N + kThreads - 1) / kThreads, 8 * num_cus());
    reduce_f32_kernel<<<dim3((unsigned)blocks), kThreads, 0, st>>>(pb.partial, pb.nsplit, M, N, C,
                                                                   ldc, alpha, beta);
    ML_LAUNCH_CHECK();
  }
  return ML_OK;
}

extern "C" int ml_gemm_f32_segments(int64_t M, int64_t N, int nseg, const int64_t* k_lens,
                                    const void* const* a_ptrs, const int64_t* ldas,
                                    const void* const* b_ptrs, const int64_t* ldbs, int a_layout,
                                    int b_layout, float* C, int64_t ldc, float alpha, float beta,
                                    void* stream) {
  return ml_gemm_f32_segments_ws(M, N, nseg, k_lens, a_ptrs, ldas, b_ptrs, ldbs, a_layout,
                                 b_layout, C, ldc, alpha, beta, nullptr, 0, stream);
}
