// nm_norm.hip — the residual add and the RMSNorm behind it, for the rows of a
// prompt in one pass: s = round_T(x + d), out = round_T(s / rms(s) * weight),
// fp16 and bf16 (nm_add_rms_norm, include/nmsparse_hip.h).
//
// Bound by memory: two rows read, two written. A workgroup owns a row; its
// 16-byte words stay in registers between the add, the sum of squares (one
// exchange through LDS) and the scaled store, so nothing is read twice. The
// arithmetic is PyTorch's add, then its fused rms_norm: fp32, one rounding each.
// Graph replay, fp16, the two calls in parentheses: 500 x 4096 3.7 us, 4.4 TB/s
// out of the caches (8.8); 1500 x 5120 9.9 (17.0); 20 x 4096 2.4 (6.3).
#include "nm_gemv_kernel.h"

namespace nm_hip {
namespace {

constexpr int kNormMaxDim = 8192;

// NI: 16-byte words of a row per lane.
template <int DT, int NI>
__global__ __launch_bounds__(kBlock) void nm_add_rms_norm_kernel(const u32x4* __restrict__ x,
                                                                const u32x4* __restrict__ d,
                                                                const u32x4* __restrict__ weight, float eps,
                                                                u32x4* __restrict__ sum, u32x4* __restrict__ out,
                                                                int words) {
  using E = Elem<DT>;
  typedef typename E::scalar T;
  typedef T t8 __attribute__((ext_vector_type(8)));
  __shared__ float part[kBlock / 64];
  const int tid = threadIdx.x;
  const size_t row = (size_t)blockIdx.x * (size_t)words;
  u32x4 xw[NI], dw[NI], ww[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int c = min(tid + i * kBlock, words - 1);  // lanes past the row read its last word, unused
    xw[i] = x[row + c];
    dw[i] = d[row + c];
    ww[i] = weight[c];
  }
  float v[NI][8], ssq = 0.0f;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const u32x4 a[1] = {xw[i]}, b[1] = {dw[i]};
    float p[8], q[8];
    E::unpack(a, p);
    E::unpack(b, q);
    t8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = E::from_f32(p[e] + q[e]);
    const u32x4 s[1] = {__builtin_bit_cast(u32x4, r)};
    E::unpack(s, v[i]);
    if (tid + i * kBlock < words) {
      sum[row + tid + i * kBlock] = s[0];
#pragma unroll
      for (int e = 0; e < 8; ++e) ssq = __builtin_fmaf(v[i][e], v[i][e], ssq);
    }
  }
  ssq = wave_sum(ssq);
  if ((tid & 63) == 0) part[tid >> 6] = ssq;
  __syncthreads();
  float t = 0.0f;
#pragma unroll
  for (int i = 0; i < kBlock / 64; ++i) t += part[i];
  const float scale = rsqrtf(t / (float)(words * 8) + eps);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const u32x4 a[1] = {ww[i]};
    float g[8];
    E::unpack(a, g);
    t8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = E::from_f32(v[i][e] * scale * g[e]);
    if (tid + i * kBlock < words) out[row + tid + i * kBlock] = __builtin_bit_cast(u32x4, r);
  }
}

typedef void (*NormFn)(const u32x4*, const u32x4*, const u32x4*, float, u32x4*, u32x4*, int);
template <int DT>
NormFn norm_fn(int words) {
  if (words <= kBlock) return &nm_add_rms_norm_kernel<DT, 1>;
  if (words <= 2 * kBlock) return &nm_add_rms_norm_kernel<DT, 2>;
  if (words <= 3 * kBlock) return &nm_add_rms_norm_kernel<DT, 3>;
  return &nm_add_rms_norm_kernel<DT, 4>;
}

}  // namespace
}  // namespace nm_hip

using namespace nm_hip;

extern "C" int nm_add_rms_norm(int dtype, const void* x, const void* d, const void* weight, float eps, void* sum,
                               void* out, int rows, int dim, void* stream) {
  if (dtype != NM_DTYPE_F16 && dtype != NM_DTYPE_BF16) return NM_ERR_BAD_CONFIG;
  if (rows <= 0 || dim <= 0 || dim % 8 != 0 || dim > kNormMaxDim) return NM_ERR_BAD_SHAPE;
  if (!x || !d || !weight || !sum || !out) return NM_ERR_NULL_POINTER;
  if ((((uintptr_t)x | (uintptr_t)d | (uintptr_t)weight | (uintptr_t)sum | (uintptr_t)out) & 15u) != 0)
    return NM_ERR_MISALIGNED;
  const NormFn fn = dtype == NM_DTYPE_F16 ? norm_fn<NM_DTYPE_F16>(dim / 8) : norm_fn<NM_DTYPE_BF16>(dim / 8);
  hipLaunchKernelGGL(fn, dim3((unsigned)rows), dim3(kBlock), 0, static_cast<hipStream_t>(stream),
                     static_cast<const u32x4*>(x), static_cast<const u32x4*>(d), static_cast<const u32x4*>(weight), eps,
                     static_cast<u32x4*>(sum), static_cast<u32x4*>(out), dim / 8);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? NM_OK : (int)e;
}
