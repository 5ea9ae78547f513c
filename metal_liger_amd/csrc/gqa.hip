// Key / value heads of grouped-query attention repeated for the query heads
// that share them, and the gradients' way back, for gfx950: what
// transformers' repeat_kv does with expand + reshape (a strided copy each for
// k and v, a strided reduction each in the backward).
//
// HBM-bound: every input read once, every output written once, k and v in one
// launch. A thread moves one 16-byte vector of a row to (from) the `groups`
// heads, so the source is read once instead of once per copy, and the 16
// threads of a 128-wide bf16 row keep each access 256 bytes long. The gradients
// are written as [B, S, H, D], the layout of the projections they go to, so
// that no copy follows. At [4, 8, 2048, 128] bf16 and 2 groups: 52 -> 18 us
// forward, 55 us with the copy behind it -> 18 us backward (5.6 TB/s).
#include "common.h"

namespace mla {
namespace gqa {
namespace {

constexpr int kMaxTensors = 2;

struct Tensor {
  const void* x;
  void* y;
  int B, H, S, D;  // H: key / value heads
  int64_t xb, xh, xs, yb, yh, ys;  // strides in elements; D dense
};
struct Args {
  Tensor t[kMaxTensors];
  int groups;
};

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// y[b, h groups + g, s] = x[b, h, s]
template <typename T>
__global__ __launch_bounds__(256) void expand_kernel(const Args a) {
  constexpr int V = vec16<T>();
  const Tensor& t = a.t[blockIdx.y];
  const int dv = t.D / V;
  const int64_t total = (int64_t)t.B * t.H * t.S * dv;
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < total;
       q += (int64_t)gridDim.x * 256) {
    const int d = (int)(q % dv) * V;
    const int64_t row = q / dv, bh = row / t.S;
    const int s = (int)(row - bh * t.S), b = (int)(bh / t.H), h = (int)(bh - (int64_t)b * t.H);
    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(
        static_cast<const T*>(t.x) + b * t.xb + h * t.xh + s * t.xs + d));
    T* y = static_cast<T*>(t.y) + b * t.yb + (int64_t)h * a.groups * t.yh + s * t.ys + d;
    for (int g = 0; g < a.groups; ++g) *reinterpret_cast<u32x4*>(y + g * t.yh) = v;
  }
}

// y[b, h, s] = sum over g of x[b, h groups + g, s], in fp32, rounded once
template <typename T>
__global__ __launch_bounds__(256) void reduce_kernel(const Args a) {
  constexpr int V = vec16<T>();
  const Tensor& t = a.t[blockIdx.y];
  const int dv = t.D / V;
  const int64_t total = (int64_t)t.B * t.H * t.S * dv;
  for (int64_t q = (int64_t)blockIdx.x * 256 + threadIdx.x; q < total;
       q += (int64_t)gridDim.x * 256) {
    const int d = (int)(q % dv) * V;
    const int64_t row = q / dv, bs = row / t.H;
    const int h = (int)(row - bs * t.H), b = (int)(bs / t.S), s = (int)(bs - (int64_t)b * t.S);
    const T* x = static_cast<const T*>(t.x) + b * t.xb + (int64_t)h * a.groups * t.xh + s * t.xs + d;
    float sum[V];
    load_n_nt<T, V>(x, sum);
    for (int g = 1; g < a.groups; ++g) {
      float v[V];
      load_n_nt<T, V>(x + g * t.xh, v);
#pragma unroll
      for (int k = 0; k < V; ++k) sum[k] += v[k];
    }
    store_n<T, V>(static_cast<T*>(t.y) + b * t.yb + h * t.yh + s * t.ys + d, sum);
  }
}

int run(bool expand, int count, const void* const* x, void* const* y, const int64_t* geometry,
        int64_t groups, int dtype, hipStream_t st) {
  ML_CHECK(count >= 1 && count <= kMaxTensors, "kv heads: 1..%d tensors (got %d)", kMaxTensors,
           count);
  ML_CHECK(x && y && geometry, "kv heads: null argument arrays");
  ML_CHECK(groups >= 1 && groups < (1 << 20), "kv heads: bad group count %lld", (long long)groups);
  ML_CHECK(dtype == ML_F32 || dtype == ML_BF16 || dtype == ML_F16, "kv heads: dtype %d", dtype);
  const int64_t es = dtype == ML_F32 ? 4 : 2, V = 16 / es;
  Args a{};
  a.groups = (int)groups;
  int64_t most = 0;
  for (int i = 0; i < count; ++i) {
    const int64_t* g = geometry + 10 * i;  // B, H, S, D, x strides b h s, y strides b h s
    for (int k = 0; k < 4; ++k)
      ML_CHECK(g[k] >= 0 && g[k] < (1LL << 31), "kv heads: bad size of tensor %d", i);
    ML_CHECK(g[3] % V == 0, "kv heads: head size must be a multiple of 16 bytes (got %lld)",
             (long long)g[3]);
    for (int k = 4; k < 10; ++k)
      ML_CHECK(g[k] >= 0 && g[k] % V == 0, "kv heads: strides must be multiples of 16 bytes");
    const int64_t n = g[0] * g[1] * g[2];
    ML_CHECK(n < (1LL << 40), "kv heads: tensor %d too large", i);
    ML_CHECK(n == 0 || g[3] == 0 || (x[i] && y[i] && aligned16(x[i]) && aligned16(y[i])),
             "kv heads: null or misaligned pointer of tensor %d", i);
    a.t[i] = Tensor{x[i], y[i], (int)g[0], (int)g[1], (int)g[2], (int)g[3],
                    g[4], g[5], g[6], g[7], g[8], g[9]};
    most = n * (g[3] / V) > most ? n * (g[3] / V) : most;
  }
  if (most == 0) return ML_OK;
  int64_t blocks = (most + 255) / 256;
  blocks = blocks < 16384 ? blocks : 16384;
  const dim3 grid((unsigned)blocks, (unsigned)count);
  auto go = [&](auto v) {
    using T = decltype(v);
    if (expand) expand_kernel<T><<<grid, 256, 0, st>>>(a);
    else reduce_kernel<T><<<grid, 256, 0, st>>>(a);
  };
  if (dtype == ML_F32) go(float{});
  else if (dtype == ML_BF16) go(bf16{});
  else go(f16{});
  ML_LAUNCH_CHECK();
  return ML_OK;
}

}  // namespace
}  // namespace gqa
}  // namespace mla

extern "C" int ml_kv_expand(int count, const void* const* x, void* const* y,
                            const int64_t* geometry, int64_t groups, int dtype, void* stream) {
  return mla::gqa::run(true, count, x, y, geometry, groups, dtype, (hipStream_t)stream);
}

extern "C" int ml_kv_reduce(int count, const void* const* x, void* const* y,
                            const int64_t* geometry, int64_t groups, int dtype, void* stream) {
  return mla::gqa::run(false, count, x, y, geometry, groups, dtype, (hipStream_t)stream);
}
