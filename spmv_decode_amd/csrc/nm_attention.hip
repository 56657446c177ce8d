// nm_attention.hip — attention over the transposed static caches
// (include/nmsparse_hip.h): one decode token in one launch
// (nm_attention_decode), and a whole prompt (nm_prefill_rope,
// nm_attention_prefill; at the end of this file). The decode token:
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
//    once, so the work follows the position. PW follows the cache length
//    (make_attn_plan): an early position of a long cache runs in the few large
//    splits that its end needs. At decode contexts the caches are a few MB: the
//    launch is bound by latency, so every load of a split is requested before
//    the first is waited for.
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
#include <float.h>
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
// What the scores of a split or block are taken relative to: its maximum m, and
// a finite number where every score is -inf. Their probabilities are then 0
// (exp2(-inf - -inf) is NaN), so other positions keep their softmax; a row of
// nothing but -inf ends as 0 / 0.
__device__ inline float exp_base(float m) { return fmaxf(m, -FLT_MAX); }

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
    const float base = exp_base(rowmax[j]);
#pragma unroll
    for (int b = 0; b < NPB; ++b) {
      const float p = __builtin_amdgcn_exp2f(sc[b][j] - base);
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

// ---------------------------------------------------------------------------
// A whole prompt (nm_prefill_rope, nm_attention_prefill): the rotary embedding
// with the cache writes, and causal attention of every position over the
// caches.
// ---------------------------------------------------------------------------
struct RopeArgs {
  const void *q, *k, *v;            // [P, heads * hd], rows *_stride elements apart
  long long q_stride, k_stride, v_stride;
  const void *q_norm, *k_norm;      // optional [hd] per-head RMSNorm weights
  const float2* rope;               // [>= P, hd / 2] (cos, sin)
  void* q_out;                      // [P, n_heads, hd]
  void* k_cache;                    // [kv_heads, >= hd, S]
  void* v_cache;                    // [kv_heads, hd, S]
  long long k_head, v_head;
  float eps;
  int P, nh, kvh, S;
};

// A workgroup takes 64 positions of one head: blockIdx.y < nh a query head
// (norm, rotation, to q_out), then the key heads (the same, transposed into the
// cache through LDS) and the value heads (transposed only). Lane (row, part)
// holds a quarter of a row's head. One pass over q, k and v where the norms, the
// casts, the complex product and the strided cache copies took twelve launches
// per layer. Bound by its launch and one memory round trip.
template <int DT, int HD>
__global__ __launch_bounds__(kBlock) void nm_prefill_rope_kernel(RopeArgs a) {
  using E = Elem<DT>;
  typedef typename E::scalar T;
  constexpr int Q = HD / 4;        // elements per lane
  constexpr int TS = 64 + 8;       // LDS row stride of the transposed tile
  __shared__ __attribute__((aligned(16))) T tile[HD * TS];
  const int tid = threadIdx.x, row = tid >> 2, part = tid & 3;
  const int p0 = (int)blockIdx.x * 64, head = (int)blockIdx.y;
  const int pos = min(p0 + row, a.P - 1);
  const int kind = head < a.nh ? 0 : (head < a.nh + a.kvh ? 1 : 2);
  const int hi = kind == 0 ? head : (kind == 1 ? head - a.nh : head - a.nh - a.kvh);
  const T* src = static_cast<const T*>(kind == 0 ? a.q : (kind == 1 ? a.k : a.v)) +
                 (long long)pos * (kind == 0 ? a.q_stride : (kind == 1 ? a.k_stride : a.v_stride)) + hi * HD + part * Q;
  u32x4 raw[Q / 8];
#pragma unroll
  for (int i = 0; i < Q / 8; ++i) raw[i] = *reinterpret_cast<const u32x4*>(src + 8 * i);
  float x[Q];
#pragma unroll
  for (int i = 0; i < Q / 8; ++i) {
    const u32x4 one[1] = {raw[i]};
    float f[8];
    E::unpack(one, f);
#pragma unroll
    for (int e = 0; e < 8; ++e) x[8 * i + e] = f[e];
  }
  const T* norm = static_cast<const T*>(kind == 0 ? a.q_norm : a.k_norm);
  if (kind < 2) {
    if (norm) {
      float s = 0.0f;
#pragma unroll
      for (int e = 0; e < Q; ++e) s = __builtin_fmaf(x[e], x[e], s);
      s += dpp<0xB1>(s);
      s += dpp<0x4E>(s);  // the row's four lanes
      const float r = rsqrtf(s / (float)HD + a.eps);
#pragma unroll
      for (int e = 0; e < Q; ++e) x[e] *= r * E::to_f32(norm[part * Q + e]);
    }
    const float2* cs = a.rope + (size_t)pos * (HD / 2) + part * (Q / 2);
#pragma unroll
    for (int e = 0; e < Q / 2; ++e) {
      const float2 c = cs[e];
      const float x0 = x[2 * e], x1 = x[2 * e + 1];
      x[2 * e] = x0 * c.x - x1 * c.y;
      x[2 * e + 1] = x0 * c.y + x1 * c.x;
    }
  }
  typedef T t8 __attribute__((ext_vector_type(8)));
  if (kind == 0) {
    if (p0 + row >= a.P) return;
    T* out = static_cast<T*>(a.q_out) + ((long long)pos * a.nh + hi) * HD + part * Q;
#pragma unroll
    for (int i = 0; i < Q / 8; ++i) {
      t8 v;
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = E::from_f32(x[8 * i + e]);
      *reinterpret_cast<t8*>(out + 8 * i) = v;
    }
    return;
  }
#pragma unroll
  for (int e = 0; e < Q; ++e) tile[(part * Q + e) * TS + row] = E::from_f32(x[e]);
  __syncthreads();
  T* cache = static_cast<T*>(kind == 1 ? a.k_cache : a.v_cache) + (long long)hi * (kind == 1 ? a.k_head : a.v_head);
#pragma unroll
  for (int i = 0; i < HD / 32; ++i) {  // 8 positions of a dimension per lane
    const int d = i * 32 + (tid >> 3), p = 8 * (tid & 7);
    T* dst = cache + (long long)d * a.S + p0 + p;
    if (p0 + p + 8 <= a.P) {  // S and so every row of the cache is a multiple of 8 (host)
      *reinterpret_cast<u32x4*>(dst) = *reinterpret_cast<const u32x4*>(&tile[d * TS + p]);
    } else {
      for (int e = 0; e < 8; ++e)
        if (p0 + p + e < a.P) dst[e] = tile[d * TS + p + e];
    }
  }
}

struct PrefillArgs {
  const void* q;   // [P, n_heads, hd]
  const void* k;   // [kv_heads, >= hd, S]
  const void* v;   // [kv_heads, hd, S]
  void* out;       // [P, n_heads, hd]
  long long k_head, v_head;
  int P, nh, kvh, g, S, tiles;
  float scale;     // log2(e) / sqrt(hd)
};

// A workgroup takes 64 positions of one query head, 16 per wave, and goes over
// the cached positions up to its last in blocks of 64: scores as in
// nm_attention_kernel (K through LDS, read transposed), a running maximum and
// sum per row, values from LDS rows of positions; the next block's K and V are
// requested before the current one is multiplied. Workgroups of one key/value
// head share an XCD's L2 (id modulo kv_heads), the longest rows first. The
// library's fused kernel with its transposes took 41.6 us for 500 positions of 32
// heads over 8 (128 workgroups), this one takes 22.5; at 128 / 1024 / 8000
// positions 17.5 / 59.7 / 1388 and 9.1 / 42.9 / 1229.
template <int DT, int HD>
__global__ __launch_bounds__(kBlock) void nm_attention_prefill_kernel(PrefillArgs a) {
  using E = Elem<DT>;
  typedef typename E::scalar T;
  constexpr int PB = 64;
  constexpr int NK = HD / 32;   // 16-B loads per lane of K (and of V)
  constexpr int KQ = HD / 32;   // MFMA steps over the head dimension
  constexpr int DB = HD / 16;   // 16-column output blocks
  constexpr int VS = PB + 8, PSTR = PB + 8;
  __shared__ __attribute__((aligned(16))) T ks[HD * PB];
  __shared__ __attribute__((aligned(16))) T vs[HD * VS];
  __shared__ __attribute__((aligned(16))) T ps[4][16 * PSTR];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, lg = lane >> 4, li = lane & 15;
  const int id = (int)blockIdx.x;
  const int kh = id % a.kvh, head = kh * a.g + (id / a.kvh) % a.g, qt = a.tiles - 1 - id / a.nh;
  const int r0 = qt * PB + 16 * wave;  // the wave's first position

  u32x4 qr[KQ];
  const T* q = static_cast<const T*>(a.q) + ((long long)min(r0 + li, a.P - 1) * a.nh + head) * HD;
#pragma unroll
  for (int i = 0; i < KQ; ++i) qr[i] = *reinterpret_cast<const u32x4*>(q + 32 * i + 8 * lg);
  const int krow = tid >> 3, kslot = tid & 7;  // 16 B of row krow + 32 i
  const T* kb = static_cast<const T*>(a.k) + (long long)kh * a.k_head;
  const T* vb = static_cast<const T*>(a.v) + (long long)kh * a.v_head;
  u32x4 kr[NK], vr[NK];
  auto load = [&](int blk) {
    const int p = min(blk * PB + 8 * kslot, a.S - 8);
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      kr[i] = *reinterpret_cast<const u32x4*>(kb + (long long)(krow + 32 * i) * a.S + p);
      vr[i] = *reinterpret_cast<const u32x4*>(vb + (long long)(krow + 32 * i) * a.S + p);
    }
  };
  load(0);
  f4 o[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d) o[d] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  float m[4], l[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) m[j] = -INFINITY, l[j] = 0.0f;
  const int rr = 8 * lg + (li >> 2);

  for (int blk = 0; blk <= qt; ++blk) {
    __syncthreads();  // the previous block's reads are done
    const int left = a.P - (blk * PB + 8 * kslot);  // cached positions past the prompt stay out of the sums
    u32x4 keep;
#pragma unroll
    for (int e = 0; e < 4; ++e) keep[e] = (left > 2 * e ? 0xffffu : 0u) | (left > 2 * e + 1 ? 0xffff0000u : 0u);
#pragma unroll
    for (int i = 0; i < NK; ++i) {
      const int r = krow + 32 * i;
      *reinterpret_cast<u32x4*>(&ks[r * PB + 8 * (kslot ^ (2 * (r & 3)))]) = kr[i];
      *reinterpret_cast<u32x4*>(&vs[r * VS + 8 * kslot]) = vr[i] & keep;
    }
    __syncthreads();
    if (blk < qt) load(blk + 1);

    float sc[4][4];  // [16-position block][row 4 lg + j]
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int slot = 2 * b + ((li & 3) >> 1);
      const T* kp = &ks[rr * PB + 8 * (slot ^ (2 * (rr & 3))) + 4 * (li & 1)];
      f4 acc = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int i = 0; i < KQ; ++i) {
        const s4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(kp + 32 * i * PB));
        const s4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(kp + (32 * i + 4) * PB));
        const s8 kf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        acc = mfma16x16x32<DT>(__builtin_bit_cast(s8, qr[i]), kf, acc);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        sc[b][j] = blk < qt || 16 * b + li <= 16 * wave + 4 * lg + j ? acc[j] * a.scale : -INFINITY;
    }
    float alpha[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      float mx = max_nan(max_nan(sc[0][j], sc[1][j]), max_nan(sc[2][j], sc[3][j]));
      mx = max_nan(m[j], row16(mx, [](float x, float y) { return max_nan(x, y); }));
      const float base = exp_base(mx);
      alpha[j] = __builtin_amdgcn_exp2f(m[j] - base);  // 0 at the first block
      m[j] = mx;
      float s = 0.0f;
#pragma unroll
      for (int b = 0; b < 4; ++b) {
        const float p = __builtin_amdgcn_exp2f(sc[b][j] - base);
        s += p;
        ps[wave][(4 * lg + j) * PSTR + 16 * b + li] = E::from_f32(p);
      }
      l[j] = l[j] * alpha[j] + row16(s, [](float x, float y) { return x + y; });
    }
#pragma unroll
    for (int d = 0; d < DB; ++d)
#pragma unroll
      for (int j = 0; j < 4; ++j) o[d][j] *= alpha[j];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int i = 0; i < PB / 32; ++i) {
      const s8 pa = __builtin_bit_cast(s8, *reinterpret_cast<const u32x4*>(&ps[wave][li * PSTR + 32 * i + 8 * lg]));
#pragma unroll
      for (int d = 0; d < DB; ++d)
        o[d] = mfma16x16x32<DT>(
            pa, __builtin_bit_cast(s8, *reinterpret_cast<const u32x4*>(&vs[(16 * d + li) * VS + 32 * i + 8 * lg])), o[d]);
    }
    __builtin_amdgcn_wave_barrier();
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = r0 + 4 * lg + j;
    if (r >= a.P) continue;
    T* out = static_cast<T*>(a.out) + ((long long)r * a.nh + head) * HD + li;
    const float inv = 1.0f / l[j];
#pragma unroll
    for (int d = 0; d < DB; ++d) out[16 * d] = E::from_f32(o[d][j] * inv);
  }
}

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

int nm_prefill_rope(int dtype, const void* q, long long q_row_stride, const void* k, long long k_row_stride,
                    const void* v, long long v_row_stride, const void* q_norm, const void* k_norm, float eps,
                    const float* rope_table, int P, int n_heads, int kv_heads, int head_dim, void* q_out,
                    void* k_cache_t, long long k_head_stride, void* v_cache_t, long long v_head_stride, int cache_len,
                    void* stream) {
  if (dtype != NM_DTYPE_F16 && dtype != NM_DTYPE_BF16) return NM_ERR_BAD_CONFIG;
  if (P <= 0 || n_heads <= 0 || kv_heads <= 0 || (head_dim != 64 && head_dim != 128) || cache_len < P ||
      cache_len % 8 != 0 || n_heads + 2LL * kv_heads > 65535)
    return NM_ERR_BAD_SHAPE;
  const long long qd = (long long)n_heads * head_dim, kd = (long long)kv_heads * head_dim;
  const long long row = (long long)head_dim * cache_len;
  if (q_row_stride < qd || k_row_stride < kd || v_row_stride < kd || k_head_stride < row || v_head_stride < row)
    return NM_ERR_BAD_SHAPE;
  if (!q || !k || !v || !rope_table || !q_out || !k_cache_t || !v_cache_t) return NM_ERR_NULL_POINTER;
  if (((q_row_stride | k_row_stride | v_row_stride | k_head_stride | v_head_stride) & 7) != 0 ||
      ((uintptr_t)q | (uintptr_t)k | (uintptr_t)v | (uintptr_t)q_out | (uintptr_t)k_cache_t | (uintptr_t)v_cache_t) %
              16 != 0 ||
      (uintptr_t)rope_table % 8 != 0)
    return NM_ERR_MISALIGNED;
  if ((q_norm || k_norm) && !(eps >= 0.0f)) return NM_ERR_BAD_EPILOGUE;
  RopeArgs a;
  memset(&a, 0, sizeof(a));
  a.q = q, a.k = k, a.v = v;
  a.q_stride = q_row_stride, a.k_stride = k_row_stride, a.v_stride = v_row_stride;
  a.q_norm = q_norm, a.k_norm = k_norm, a.eps = eps;
  a.rope = reinterpret_cast<const float2*>(rope_table);
  a.q_out = q_out, a.k_cache = k_cache_t, a.v_cache = v_cache_t;
  a.k_head = k_head_stride, a.v_head = v_head_stride;
  a.P = P, a.nh = n_heads, a.kvh = kv_heads, a.S = cache_len;
  typedef void (*Fn)(RopeArgs);
  const Fn fns[2][2] = {{&nm_prefill_rope_kernel<NM_DTYPE_F16, 64>, &nm_prefill_rope_kernel<NM_DTYPE_F16, 128>},
                        {&nm_prefill_rope_kernel<NM_DTYPE_BF16, 64>, &nm_prefill_rope_kernel<NM_DTYPE_BF16, 128>}};
  hipLaunchKernelGGL(fns[dtype == NM_DTYPE_F16 ? 0 : 1][head_dim / 128],
                     dim3((unsigned)((P + 63) / 64), (unsigned)(n_heads + 2 * kv_heads)), dim3(kBlock), 0,
                     static_cast<hipStream_t>(stream), a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? NM_OK : (int)e;
}

int nm_attention_prefill(int dtype, const void* q, const void* k_cache_t, long long k_head_stride,
                         const void* v_cache_t, long long v_head_stride, void* out, int P, int n_heads, int kv_heads,
                         int head_dim, int cache_len, void* stream) {
  if (dtype != NM_DTYPE_F16 && dtype != NM_DTYPE_BF16) return NM_ERR_BAD_CONFIG;
  if (P <= 0 || n_heads <= 0 || kv_heads <= 0 || n_heads % kv_heads != 0 || (head_dim != 64 && head_dim != 128) ||
      cache_len < P || cache_len % 8 != 0)
    return NM_ERR_BAD_SHAPE;
  const long long row = (long long)head_dim * cache_len, tiles = (P + 63) / 64;
  if (k_head_stride < row || v_head_stride < row || tiles * n_heads > 0x7fffffffLL) return NM_ERR_BAD_SHAPE;
  if (!q || !k_cache_t || !v_cache_t || !out) return NM_ERR_NULL_POINTER;
  if (((k_head_stride | v_head_stride) & 7) != 0 ||
      ((uintptr_t)q | (uintptr_t)k_cache_t | (uintptr_t)v_cache_t | (uintptr_t)out) % 16 != 0)
    return NM_ERR_MISALIGNED;
  PrefillArgs a;
  memset(&a, 0, sizeof(a));
  a.q = q, a.k = k_cache_t, a.v = v_cache_t, a.out = out;
  a.k_head = k_head_stride, a.v_head = v_head_stride;
  a.P = P, a.nh = n_heads, a.kvh = kv_heads, a.g = n_heads / kv_heads, a.S = cache_len, a.tiles = (int)tiles;
  a.scale = 1.44269504088896340736f / sqrtf((float)head_dim);
  typedef void (*Fn)(PrefillArgs);
  const Fn fns[2][2] = {
      {&nm_attention_prefill_kernel<NM_DTYPE_F16, 64>, &nm_attention_prefill_kernel<NM_DTYPE_F16, 128>},
      {&nm_attention_prefill_kernel<NM_DTYPE_BF16, 64>, &nm_attention_prefill_kernel<NM_DTYPE_BF16, 128>}};
  hipLaunchKernelGGL(fns[dtype == NM_DTYPE_F16 ? 0 : 1][head_dim / 128], dim3((unsigned)(tiles * n_heads)),
                     dim3(kBlock), 0, static_cast<hipStream_t>(stream), a);
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? NM_OK : (int)e;
}

}  // extern "C"
