// nm_attention.hip — the attention of one decode token over the transposed
// static caches, in one launch (nm_attention_decode, include/nmsparse_hip.h):
//
//   out[h, :] = softmax_p( q[h, :] . K[:, p] / sqrt(hd) ) V[:, p]^T,  p <= pos
//
// for grouped query heads (g = n_heads / kv_heads per key/value head), fp16
// and bf16, read from the layouts the q/k/v launch writes: K [kv_heads, >= hd,
// S], V [kv_heads, hd, S] (positions contiguous). It replaces a batched
// product over all S positions, a softmax and a second batched product.
//
//  * A workgroup (256 lanes = 4 wave64) owns one key/value head and a split of
//    PW consecutive positions for all g query heads; splits past pos end at
//    once, so the work follows the position and not the cache length. At
//    decode contexts the caches are a few MB: the launch is bound by latency,
//    so every load of a split is requested before the first is waited for.
//  * Scores on the matrix cores: A = the queries (g rows of 16), B = K through
//    LDS, read transposed (ds_read_b64_tr_b16: rows are head dimensions, the
//    columns positions, as the weights of the matrix-core SpMM); each wave 16
//    positions per block. Scale, mask and softmax in fp32 registers.
//  * Values on the matrix cores too: V is stored with the positions contiguous,
//    which is the B operand of [16 heads x PW] x [PW x hd] as it lies: a lane's
//    16 B of V go from memory to the operand without LDS. Each wave owns hd / 4
//    output columns, so no sum crosses waves. Probabilities enter as the
//    element type, unnormalised (largest 1), and their fp32 sum divides the
//    result (the library path rounds scores and normalised probabilities).
//  * Measured (graph replay): 32 heads over 8, 512 of 640 positions 6.6 us where
//    the three library kernels took 25.2 (kernel times 12.6 + 6.2 + 6.4); 40
//    heads, 4001 of 4096 (16.4 MB) 10.4 against 37.4. An empty kernel replays at
//    1.6 us; the rest is one memory round trip for the loads, the softmax's
//    barriers and, with several splits, the handoff (2 us).
//  * More than one split: each leaves its fp32 output rows, row maxima and
//    sums in the workspace; the last to arrive at the head (the GEMV's split-K
//    handoff: agent-scope atomics, no fence) merges them in split order. The
//    result does not depend on the arrival order.
#include <math.h>

#include "nm_mfma.h"

namespace nm_hip {
namespace {

constexpr int kAttnMaxGroup = 16;  // query heads per key/value head: the MFMA's rows

constexpr int kAgentLoad = 16;     // buffer cache policy: sc1, an agent-scope load

struct AttnArgs {
  const void* q;          // [kv_heads * g, hd], rows q_stride elements apart
  const void* k;          // [kv_heads, >= hd, S], heads k_head elements apart
  const void* v;          // [kv_heads, hd, S], heads v_head elements apart
  void* out;              // [kv_heads * g, hd] contiguous
  const long long* pos;   // device: the last position attended to
  float* part;            // [kv_heads, splits, g, hd] unnormalised outputs
  float* ml;              // [kv_heads, splits, 2, g] row maxima (base-2 exponents), sums
  uint32_t* tickets;      // [kv_heads]
  long long q_stride, k_head, v_head;
  int S, g, kvh, splits, eager;
  float scale;            // log2(e) / sqrt(hd)
};

template <class F>
__device__ inline float row16(float v, F f) {  // f over the 16 lanes of a row, to all of them
  v = f(v, dpp<0xB1>(v));
  v = f(v, dpp<0x4E>(v));
  v = f(v, dpp<0x141>(v));
  return f(v, dpp<0x140>(v));
}
// A maximum that keeps NaN (a NaN score makes its whole row NaN, as softmax does).
__device__ inline float max_nan(float a, float b) { return a > b || a != a ? a : b; }

template <int DT, int HD, int NPB>
__global__ __launch_bounds__(kBlock) void nm_attention_kernel(AttnArgs a) {
  using E = Elem<DT>;
  typedef typename E::scalar T;
  constexpr int PW = 64 * NPB;          // positions per split
  constexpr int LPR = PW / 8;           // 16-B slots per LDS row of K
  constexpr int RPI = kBlock / LPR;     // K rows per load
  constexpr int NK = HD / RPI;          // K loads per lane
  constexpr int KQ = HD / 32;           // MFMA steps over the head dimension
  constexpr int DB = HD / 64;           // 16-column output blocks per wave
  constexpr int KP = PW / 32;           // MFMA steps over the positions
  constexpr int PSTR = PW + 8;          // LDS row stride of the probabilities
  static_assert(RPI % 4 == 0 && NK >= 1, "K tile shape");
  __shared__ __attribute__((aligned(16))) T ks[HD * PW];
  __shared__ __attribute__((aligned(16))) T ps[16 * PSTR];
  __shared__ __attribute__((aligned(16))) float wmax[4][16], wsum[4][16];
  __shared__ int is_last;

  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lg = lane >> 4, li = lane & 15;
  const int kh = (int)blockIdx.x % a.kvh, split = (int)blockIdx.x / a.kvh;
  const int p0 = split * PW;
  // The position, as a vector load (in order with the loads below, where a
  // scalar one would have every argument wait for it). The first round of
  // workgroups (eager splits) requests its loads before it has arrived; those
  // past the position then read for nothing, at most one round's worth. Later
  // splits wait for it.
  int zero = 0;
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+v"(zero));
#endif
  const long long pos_v = a.pos[zero];
  // n = min(max(pos + 1, 0), S): the positions attended to
  auto count = [&](long long p) {
    return __builtin_amdgcn_readfirstlane((int)(p < 0 ? 0 : (p >= a.S ? a.S : p + 1)));
  };
  if (split >= a.eager && p0 >= max(count(pos_v), 1)) return;

  // 1. Every load of the split: the queries, K, then V (positions past the
  //    cache read its last 8; they are masked).
  const T* __restrict__ q = static_cast<const T*>(a.q) + (size_t)(kh * a.g + min(li, a.g - 1)) * (size_t)a.q_stride;
  u32x4 qr[KQ];
#pragma unroll
  for (int i = 0; i < KQ; ++i) qr[i] = *reinterpret_cast<const u32x4*>(q + 32 * i + 8 * lg);
  // LDS row r keeps its 16-B slot c at c ^ 2 (r & 3): the four rows that a
  // transposed read takes then lie in four bank groups.
  const int krow = tid / LPR, kslot = tid % LPR;
  const T* __restrict__ k = static_cast<const T*>(a.k) + (size_t)kh * (size_t)a.k_head + min(p0 + 8 * kslot, a.S - 8);
  u32x4 kr[NK];
#pragma unroll
  for (int i = 0; i < NK; ++i)
    kr[i] = *reinterpret_cast<const u32x4*>(k + (size_t)(krow + i * RPI) * (size_t)a.S);
  const T* __restrict__ v =
      static_cast<const T*>(a.v) + (size_t)kh * (size_t)a.v_head + (size_t)(wave * (HD / 4) + li) * (size_t)a.S;
  u32x4 vr[DB][KP];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int i = 0; i < KP; ++i)
      vr[d][i] = *reinterpret_cast<const u32x4*>(v + (size_t)(16 * d) * (size_t)a.S + min(p0 + 32 * i + 8 * lg, a.S - 8));
  __builtin_amdgcn_sched_barrier(0);
  const int n = count(pos_v);
  const int active = n > 0 ? (n + PW - 1) / PW : 1;
  if (split >= active) return;

  // 2. K to LDS; the queries' operand (rows past g zero).
#pragma unroll
  for (int i = 0; i < NK; ++i)
    *reinterpret_cast<u32x4*>(&ks[(krow + i * RPI) * PW + 8 * (kslot ^ (2 * (krow & 3)))]) = kr[i];
  s8 qa[KQ];
#pragma unroll
  for (int i = 0; i < KQ; ++i) qa[i] = __builtin_bit_cast(s8, li < a.g ? qr[i] : u32x4{0u, 0u, 0u, 0u});
  __syncthreads();

  // 3. Scores: the wave's NPB blocks of 16 positions; lane: position li of the
  //    block, heads 4 lg .. + 3. In base-2 exponents, -inf past the position.
  float sc[NPB][4];
  const int rr = 8 * lg + (li >> 2);
#pragma unroll
  for (int b = 0; b < NPB; ++b) {
    const int c0 = 16 * (wave * NPB + b);
    const int slot = c0 / 8 + ((li & 3) >> 1);
    const T* kp = &ks[rr * PW + 8 * (slot ^ (2 * (rr & 3))) + 4 * (li & 1)];
    s4 lo[KQ], hi[KQ];
#pragma unroll
    for (int i = 0; i < KQ; ++i) {
      lo[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(kp + 32 * i * PW));
      hi[i] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(kp + (32 * i + 4) * PW));
    }
    __builtin_amdgcn_sched_barrier(0);  // one LDS round trip per block, not one per step
    f4 acc = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int i = 0; i < KQ; ++i) {
      const s8 kb = {lo[i][0], lo[i][1], lo[i][2], lo[i][3], hi[i][0], hi[i][1], hi[i][2], hi[i][3]};
      acc = mfma16x16x32<DT>(qa[i], kb, acc);
    }
    const bool ok = p0 + c0 + li < n;
#pragma unroll
    for (int j = 0; j < 4; ++j) sc[b][j] = ok ? acc[j] * a.scale : -INFINITY;
  }

  // 4. Softmax over the split: row maxima, then probabilities and their sums
  //    (the four rows of a lane together: one LDS round trip).
  float rowmax[4], rowsum[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    rowmax[j] = sc[0][j];
#pragma unroll
    for (int b = 1; b < NPB; ++b) rowmax[j] = max_nan(rowmax[j], sc[b][j]);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) rowmax[j] = row16(rowmax[j], [](float x, float y) { return max_nan(x, y); });
  if (li == 0) *reinterpret_cast<float4*>(&wmax[wave][4 * lg]) = make_float4(rowmax[0], rowmax[1], rowmax[2], rowmax[3]);
  __syncthreads();
  float4 wm[4];
#pragma unroll
  for (int w = 0; w < 4; ++w) wm[w] = *reinterpret_cast<const float4*>(&wmax[w][4 * lg]);
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    auto at = [&](int w) { return j == 0 ? wm[w].x : (j == 1 ? wm[w].y : (j == 2 ? wm[w].z : wm[w].w)); };
    rowmax[j] = max_nan(max_nan(at(0), at(1)), max_nan(at(2), at(3)));
    rowsum[j] = 0.0f;
#pragma unroll
    for (int b = 0; b < NPB; ++b) {
      const float p = __builtin_amdgcn_exp2f(sc[b][j] - rowmax[j]);
      rowsum[j] += p;
      ps[(4 * lg + j) * PSTR + 16 * (wave * NPB + b) + li] = E::from_f32(p);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) rowsum[j] = row16(rowsum[j], [](float x, float y) { return x + y; });
  if (li == 0) *reinterpret_cast<float4*>(&wsum[wave][4 * lg]) = make_float4(rowsum[0], rowsum[1], rowsum[2], rowsum[3]);
  __syncthreads();

  // 5. Positions of the last split past the end weigh zero; their values are
  //    cleared too, so that whatever the cache holds there (NaN) stays out.
  if (p0 + PW > n) {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int left = n - (p0 + 32 * i + 8 * lg);  // valid positions of the lane's 8
      u32x4 keep;
#pragma unroll
      for (int e = 0; e < 4; ++e) keep[e] = (left > 2 * e ? 0xffffu : 0u) | (left > 2 * e + 1 ? 0xffff0000u : 0u);
#pragma unroll
      for (int d = 0; d < DB; ++d) vr[d][i] &= keep;
    }
  }

  // 6. Values: rows 4 lg .. + 3 (heads), column li of the wave's blocks.
  f4 o[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d) o[d] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < KP; ++i) {
    const s8 pa = __builtin_bit_cast(s8, *reinterpret_cast<const u32x4*>(&ps[li * PSTR + 32 * i + 8 * lg]));
#pragma unroll
    for (int d = 0; d < DB; ++d) o[d] = mfma16x16x32<DT>(pa, __builtin_bit_cast(s8, vr[d][i]), o[d]);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int h = 4 * lg + j;
    rowsum[j] = (wsum[0][h] + wsum[1][h]) + (wsum[2][h] + wsum[3][h]);
  }
  T* __restrict__ out = static_cast<T*>(a.out) + (size_t)kh * (size_t)(a.g * HD);
  const int col = wave * (HD / 4) + li;
  if (active == 1) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (4 * lg + j < a.g)
#pragma unroll
        for (int d = 0; d < DB; ++d) out[(4 * lg + j) * HD + col + 16 * d] = E::from_f32(o[d][j] / rowsum[j]);
    return;
  }

  // 7. Handoff (as nm_gemv_kernel): publish, count, the last arrival merges.
  const int gh = a.g * HD;
  float* part = a.part + (size_t)kh * (size_t)a.splits * (size_t)gh;
  float* ml = a.ml + (size_t)kh * (size_t)a.splits * (size_t)(2 * a.g);
#pragma unroll
  for (int j = 0; j < 4; ++j)
    if (4 * lg + j < a.g) {
      float* pp = part + (size_t)split * (size_t)gh + (4 * lg + j) * HD + col;
#pragma unroll
      for (int d = 0; d < DB; ++d)
        __hip_atomic_store(pp + 16 * d, o[d][j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      if (wave == 0 && li == 0) {
        float* mp = ml + (size_t)split * (size_t)(2 * a.g) + 4 * lg + j;
        __hip_atomic_store(mp, rowmax[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(mp + a.g, rowsum[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const uint32_t prev = __hip_atomic_fetch_add(&a.tickets[kh], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    is_last = (prev == (uint32_t)(active - 1)) ? 1 : 0;
  }
  __syncthreads();
  if (!is_last) return;

  // 8. Merge. Lane (sg, e) sums outputs 4 e .. + 3 over the splits sg, sg + SG,
  //    ...: SG lanes share a quad where the g hd / 4 quads leave lanes idle. 16
  //    lanes per head turn the splits' maxima and sums into weights (in LDS,
  //    over K's tile: the plan bounds 2 splits g + 1024 floats by its size)
  //    while the first partials are on their way. All reads are coherent at
  //    agent scope (sc1, as the scalar atomic loads), 16 B each.
  const int quads = gh / 4;  // a multiple of 16
  const int SG = quads >= kBlock ? 1 : kBlock / quads;
  const int sg = SG > 1 ? tid / quads : 0;
  const int e0 = SG > 1 ? tid - sg * quads : tid;
  constexpr int NF = NPB == 1 ? 8 : 16;  // partials in flight per lane
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(part, 0, a.splits * gh * 4, 0x00020000);
  u32x4 t[NF];
  auto load = [&](int e, int s) {
#pragma unroll
    for (int i = 0; i < NF; ++i)
      t[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, (min(s + i * SG, active - 1) * gh + 4 * min(e, quads - 1)) * 4, 0,
                                                   kAgentLoad);
  };
  const int mh = min(tid >> 4, a.g - 1), mr = tid & 15;
  const bool own = (tid >> 4) < a.g;  // lanes past the heads load (no branch around the loads) and write nothing
  constexpr int NM = 4;               // 64 splits' maxima and sums in flight
  float m4[NM], s4_[NM];
  auto load_ml = [&](int s) {
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      const float* mp = ml + (size_t)min(s + 16 * i, active - 1) * (size_t)(2 * a.g) + mh;
      m4[i] = __hip_atomic_load(mp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      s4_[i] = __hip_atomic_load(mp + a.g, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  };
  load_ml(mr);
  load(e0, sg);
  float* wt = reinterpret_cast<float*>(ks);
  float* ls = wt + active * a.g;
  float m = -INFINITY;
  for (int s = mr; s < active; s += 16 * NM) {
    if (s != mr) load_ml(s);
#pragma unroll
    for (int i = 0; i < NM; ++i) {
      m = max_nan(m, m4[i]);
      if (own && s + 16 * i < active) {
        wt[(s + 16 * i) * a.g + mh] = m4[i];
        ls[(s + 16 * i) * a.g + mh] = s4_[i];
      }
    }
  }
  m = row16(m, [](float x, float y) { return max_nan(x, y); });
  float sum = 0.0f;
  for (int s = mr; s < active; s += 16) {
    const float e = __builtin_amdgcn_exp2f(wt[s * a.g + mh] - m);
    sum += e * ls[s * a.g + mh];
  }
  sum = row16(sum, [](float x, float y) { return x + y; });
  const float inv = 1.0f / sum;
  if (own)  // the weights take the sums' place (each lane its own splits')
    for (int s = mr; s < active; s += 16) ls[s * a.g + mh] = __builtin_amdgcn_exp2f(wt[s * a.g + mh] - m) * inv;
  __syncthreads();
  auto store = [&](int e, const f4& x) {
    typedef T t4 __attribute__((ext_vector_type(4)));
    t4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = E::from_f32(x[i]);
    *reinterpret_cast<t4*>(out + 4 * e) = r;
  };
  f4* sums = reinterpret_cast<f4*>(wt + ((2 * active * a.g + 3) & ~3));  // [256], where lanes share quads
  for (int e = e0; e < (SG > 1 ? quads : (quads + kBlock - 1) / kBlock * kBlock); e += SG > 1 ? quads : kBlock) {
    const float* we = ls + 4 * min(e, quads - 1) / HD;
    f4 x = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int s = sg; s < active; s += NF * SG) {
      if (s != sg || e != e0) load(e, s);
#pragma unroll
      for (int i = 0; i < NF; ++i) {
        const int si = s + i * SG;
        const float wv = we[min(si, active - 1) * a.g];
        const f4 p = __builtin_bit_cast(f4, t[i]);
#pragma unroll
        for (int c = 0; c < 4; ++c) x[c] = si < active ? __builtin_fmaf(p[c], wv, x[c]) : x[c];
      }
    }
    if (SG > 1) {
      sums[tid] = x;
    } else if (e < quads) {
      store(e, x);
    }
  }
  if (SG > 1) {
    __syncthreads();
    if (tid < quads) {
      f4 x = sums[tid];
      for (int i = 1; i < SG; ++i) x += sums[i * quads + tid];
      store(tid, x);
    }
  }
  if (tid == 0) __hip_atomic_store(&a.tickets[kh], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

constexpr int kAttnCUs = 256;  // workgroups of one round

struct AttnPlan {
  int npb, splits;
  size_t ml_off, workspace;
};

// Positions per split (64, 128 or 256; `span` forces one), from graph-replay
// sweeps (us a launch at spans 64 / 128 / 256, 32 heads over 8 but where
// stated): a cache of one span needs no merge (128 positions 6.1 / 4.1 / 5.6);
// past it the loads of a split are one round trip whatever its size, so the
// smallest split wins until its merge reads more than 16 of them (640
// positions 6.6 / 7.5 / 9.1, 1024 7.4 / 7.7 / 9.1, 2048 9.9 / 8.5 / 9.5, 4096
// with 40 heads 16.4 / 11.4 / 10.4, 8192 22.9 / 14.0 / 13.3).
constexpr int kAttnMaxMerge = 16;

int make_attn_plan(int n_heads, int kv_heads, int head_dim, int cache_len, int span, AttnPlan* p) {
  if (n_heads <= 0 || kv_heads <= 0 || n_heads % kv_heads != 0 || cache_len < 8 || cache_len % 8 != 0)
    return NM_ERR_BAD_SHAPE;
  if (head_dim != 64 && head_dim != 128) return NM_ERR_BAD_SHAPE;
  const int g = n_heads / kv_heads;
  if (g > kAttnMaxGroup || kv_heads > kMaxTickets) return NM_ERR_BAD_SHAPE;
  if (span != 0 && span != 64 && span != 128 && span != 256) return NM_ERR_BAD_CONFIG;
  for (int npb = 1; npb <= 4; npb *= 2) {
    const int pw = 64 * npb;
    if (span != 0 && pw != span) continue;
    const long long splits = ((long long)cache_len + pw - 1) / pw;
    if (8LL * splits * g + 4096 + 16 > 2LL * head_dim * pw) continue;  // merge weights and sums over K's tile
    if (span == 0 && npb < 4 && (splits > kAttnMaxMerge || (npb == 1 && cache_len <= 128 && cache_len > 64))) continue;
    if (splits * kv_heads > 0x7fffffffLL) return NM_ERR_BAD_SHAPE;
    p->npb = npb;
    p->splits = (int)splits;
    const size_t rows = (size_t)kv_heads * (size_t)splits * (size_t)g;
    p->ml_off = (size_t)NM_TICKET_BYTES + rows * (size_t)head_dim * sizeof(float);
    p->workspace = p->ml_off + rows * 2 * sizeof(float);
    return NM_OK;
  }
  return NM_ERR_BAD_SHAPE;
}

typedef void (*AttnFn)(AttnArgs);
#define NM_ATTN_ROW(DT)                                                                              \
  {{&nm_attention_kernel<DT, 64, 1>, &nm_attention_kernel<DT, 64, 2>, &nm_attention_kernel<DT, 64, 4>}, \
   {&nm_attention_kernel<DT, 128, 1>, &nm_attention_kernel<DT, 128, 2>, &nm_attention_kernel<DT, 128, 4>}}
const AttnFn kAttnKernels[2][2][3] = {NM_ATTN_ROW(NM_DTYPE_F16), NM_ATTN_ROW(NM_DTYPE_BF16)};
#undef NM_ATTN_ROW

}  // namespace
}  // namespace nm_hip

using namespace nm_hip;

extern "C" {

size_t nm_attention_decode_workspace_bytes(int n_heads, int kv_heads, int head_dim, int cache_len, int span) {
  AttnPlan p;
  return make_attn_plan(n_heads, kv_heads, head_dim, cache_len, span, &p) == NM_OK ? p.workspace : 0;
}

int nm_attention_decode(int dtype, const void* q, long long q_row_stride, const void* k_cache_t,
                        long long k_head_stride, const void* v_cache_t, long long v_head_stride, void* out,
                        const long long* pos, void* workspace, size_t workspace_bytes, int n_heads, int kv_heads,
                        int head_dim, int cache_len, int span, void* stream) {
  if (dtype != NM_DTYPE_F16 && dtype != NM_DTYPE_BF16) return NM_ERR_BAD_CONFIG;
  AttnPlan p;
  const int rc = make_attn_plan(n_heads, kv_heads, head_dim, cache_len, span, &p);
  if (rc != NM_OK) return rc;
  if (!q || !k_cache_t || !v_cache_t || !out || !pos || !workspace) return NM_ERR_NULL_POINTER;
  const long long row = (long long)head_dim * cache_len;
  if (q_row_stride < head_dim || k_head_stride < row || v_head_stride < row) return NM_ERR_BAD_SHAPE;
  if (q_row_stride % 8 != 0 || k_head_stride % 8 != 0 || v_head_stride % 8 != 0 ||
      ((uintptr_t)q | (uintptr_t)k_cache_t | (uintptr_t)v_cache_t | (uintptr_t)out) % 16 != 0 ||
      (uintptr_t)workspace % 256 != 0)
    return NM_ERR_MISALIGNED;
  if (workspace_bytes < p.workspace) return NM_ERR_WORKSPACE;
  AttnArgs a;
  memset(&a, 0, sizeof(a));
  a.q = q;
  a.k = k_cache_t;
  a.v = v_cache_t;
  a.out = out;
  a.pos = pos;
  a.part = reinterpret_cast<float*>(static_cast<char*>(workspace) + NM_TICKET_BYTES);
  a.ml = reinterpret_cast<float*>(static_cast<char*>(workspace) + p.ml_off);
  a.tickets = static_cast<uint32_t*>(workspace);
  a.q_stride = q_row_stride;
  a.k_head = k_head_stride;
  a.v_head = v_head_stride;
  a.S = cache_len;
  a.g = n_heads / kv_heads;
  a.kvh = kv_heads;
  a.splits = p.splits;
  a.eager = kAttnCUs / kv_heads;
  a.scale = 1.44269504088896340736f / sqrtf((float)head_dim);
  const AttnFn fn = kAttnKernels[dtype == NM_DTYPE_F16 ? 0 : 1][head_dim / 128][p.npb / 2];
  hipLaunchKernelGGL(fn, dim3((unsigned)(p.splits * kv_heads)), dim3(kBlock), 0, static_cast<hipStream_t>(stream), a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? NM_OK : (int)e;
}

}  // extern "C"
