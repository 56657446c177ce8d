// nm_dense_gemv.hip — y = W x for one row of activations and a dense [n, K]
// weight with unit column stride (the output head of a decode step), fp16 and
// bf16 (nm_dense_gemv, include/nmsparse_hip.h).
//
// Bound by the weight stream, read once. A wave computes R rows at a time: the
// row's 16-byte words lie over the lanes (512 elements per load), x stays in
// registers for all of the wave's rows, and the R rows' loads, about 16 in all
// for any K, are requested together and a step ahead of their use. Waves take
// neighbouring rows, so the launch reads the matrix front to back. One sum over
// the lanes per row (DPP), no LDS, no split of K.
// Measured in a graph over fresh weights (the BLAS library's one-row product in
// parentheses): 128256 x 4096 159 us, 6.6 TB/s (188); 151936 x 5120 236 us (309);
// 151936 x 1024 51 us (61).
#include "nm_gemv_kernel.h"

namespace nm_hip {
namespace {

constexpr int kDenseMaxK = 8192;
constexpr int kDenseBlocks = 512;  // two workgroups per CU

// NI: 16-byte words of a row per lane; R: rows per step.
template <int DT, int NI, int R>
__global__ __launch_bounds__(kBlock) void nm_dense_gemv_kernel(const void* __restrict__ x, const void* __restrict__ wgt,
                                                              long long row_stride, void* __restrict__ y, int n,
                                                              int K) {
  using E = Elem<DT>;
  typedef typename E::scalar T;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)));
  const int step = (int)gridDim.x * (kBlock / 64) * R;
  const T* __restrict__ w = static_cast<const T*>(wgt);
  int off[NI];
  u32x4 xr[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int k = 512 * i + 8 * lane;
    off[i] = k < K ? k : 0;  // lanes past the row read its start and multiply it by nothing
    const u32x4 v = *reinterpret_cast<const u32x4*>(static_cast<const T*>(x) + off[i]);
    xr[i] = k < K ? v : u32x4{0u, 0u, 0u, 0u};
  }
  auto load = [&](u32x4 (&d)[R][NI], int r0) {
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const T* row = w + (long long)min(r0 + r, n - 1) * row_stride;
#pragma unroll
      for (int i = 0; i < NI; ++i) d[r][i] = load16<true>(reinterpret_cast<const u32x4*>(row + off[i]));
    }
  };
  auto finish = [&](const u32x4 (&d)[R][NI], int r0) {
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = 0.0f;
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      float xf[8];
      const u32x4 xw[1] = {xr[i]};
      E::unpack(xw, xf);
      const bool in = 512 * i + 8 * lane < K;
#pragma unroll
      for (int r = 0; r < R; ++r) {
        float wf[8];
        const u32x4 ww[1] = {in ? d[r][i] : u32x4{0u, 0u, 0u, 0u}};
        E::unpack(ww, wf);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[r] = __builtin_fmaf(wf[e], xf[e], acc[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = wave_sum(acc[r]);
    if (lane == 0)
#pragma unroll
      for (int r = 0; r < R; ++r)
        if (r0 + r < n) static_cast<T*>(y)[r0 + r] = E::from_f32(acc[r]);
  };
  u32x4 a[R][NI], b[R][NI];
  int r = wave * R;
  if (r >= n) return;
  load(a, r);
  for (; r < n; r += 2 * step) {  // loads past the last row read it again
    load(b, r + step);
    finish(a, r);
    if (r + step >= n) break;
    load(a, r + 2 * step);
    finish(b, r + step);
  }
}

typedef void (*DenseFn)(const void*, const void*, long long, void*, int, int);
template <int DT>
DenseFn dense_fn(int ni) {
  if (ni <= 1) return &nm_dense_gemv_kernel<DT, 1, 8>;
  if (ni <= 2) return &nm_dense_gemv_kernel<DT, 2, 8>;
  if (ni <= 4) return &nm_dense_gemv_kernel<DT, 4, 4>;
  if (ni <= 6) return &nm_dense_gemv_kernel<DT, 6, 2>;
  if (ni <= 8) return &nm_dense_gemv_kernel<DT, 8, 2>;
  if (ni <= 10) return &nm_dense_gemv_kernel<DT, 10, 2>;
  return &nm_dense_gemv_kernel<DT, 16, 1>;
}
inline int dense_rows(int ni) { return ni <= 2 ? 8 : (ni <= 4 ? 4 : (ni <= 10 ? 2 : 1)); }

}  // namespace
}  // namespace nm_hip

using namespace nm_hip;

extern "C" int nm_dense_gemv(int dtype, const void* x, const void* weight, long long row_stride, void* y, int n, int K,
                             void* stream) {
  if (dtype != NM_DTYPE_F16 && dtype != NM_DTYPE_BF16) return NM_ERR_BAD_CONFIG;
  if (n <= 0 || K <= 0 || K % 8 != 0 || K > kDenseMaxK || row_stride < K || row_stride % 8 != 0 ||
      n > 0x7fffffff - 4 * kDenseBlocks * (kBlock / 64) * 8)
    return NM_ERR_BAD_SHAPE;
  if (!x || !weight || !y) return NM_ERR_NULL_POINTER;
  if ((((uintptr_t)x | (uintptr_t)weight) & 15u) != 0) return NM_ERR_MISALIGNED;
  const int ni = (K + 511) / 512, rows = dense_rows(ni);
  const int need = (n + rows * (kBlock / 64) - 1) / (rows * (kBlock / 64));  // workgroups of one step
  const DenseFn fn = dtype == NM_DTYPE_F16 ? dense_fn<NM_DTYPE_F16>(ni) : dense_fn<NM_DTYPE_BF16>(ni);
  hipLaunchKernelGGL(fn, dim3((unsigned)(need < kDenseBlocks ? need : kDenseBlocks)), dim3(kBlock), 0,
                     static_cast<hipStream_t>(stream), x, weight, row_stride, y, n, K);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? NM_OK : (int)e;
}
