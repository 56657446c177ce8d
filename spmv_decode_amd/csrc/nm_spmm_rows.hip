// nm_spmm_rows.hip — the matrix-core product for more rows than one tile of
// nm_spmm_mc.hip (long prompts, large batches): out_i[b, :] = W_i x[b, :] for n
// products of the same activations, fp16 and bf16 (nm_spmm_rows,
// include/nmsparse_hip.h).
//
// A gather launch writes the activations of every product in MFMA operand
// order (nm_spmm_mc.hip: fragments of 16 rows x 32 compressed columns, 1 KB
// each); the product launch is a GEMM of them and the packed weights.
//
//  * A workgroup (256 lanes = 4 wave64, one workgroup per CU) owns a tile of
//    128 rows x 128 outputs over one split of the compressed columns; a wave 64
//    x 64 of it, 16 fp32 accumulator blocks. Per 64 compressed columns a CU then
//    reads 64 KB of operands from LDS and writes 32 KB into it, 768 cycles of
//    its LDS against 512 of its matrix cores: the larger the wave's tile, the
//    fewer reads per multiply, and 64 x 64 is what the registers hold beside
//    two sets of operands.
//  * Chunks of 64 compressed columns (16 KB of weights, 16 KB of activations)
//    go from memory into a ring of 5 LDS stages (global_load_lds_dwordx4),
//    three in flight. The loads are issued in inline asm, addresses in one
//    scalar base per chunk and constant lane offsets: they have no register
//    results, and the compiler, which would otherwise wait for every DMA in
//    flight before each LDS read that it cannot tell apart, keeps exact counts
//    for the reads. Each wave waits for its own loads of a chunk (vmcnt), and
//    a barrier in the middle of the previous chunk releases it to all, so the
//    operands of the next multiplies are read while the current ones run.
//  * Weights are read transposed (ds_read_b64_tr_b16) from rows of 256 B whose
//    16-B slots are XOR-swizzled by 2 (row & 3): the four rows of one read lie
//    in four bank groups.
//  * Split-K as nm_spmm_mc.hip: fp32 partials, an arrival counter per tile, the
//    last arrival adds them in split order.
#include "nm_mfma.h"
#include "nm_spmm_mc.h"

namespace nm_hip {
namespace {

constexpr int kCK = 64;                     // compressed columns per chunk
constexpr int kBM = 128, kBN = 128;         // tile: rows x outputs
constexpr int kStages = 5;
constexpr int kWBytes = kCK * kBN * 2;      // weights of a stage
constexpr int kABytes = kBM * kCK * 2;      // activations of a stage
constexpr int kStage = kWBytes + kABytes;
constexpr int kOps = 8;                     // DMA instructions per wave per chunk
constexpr int kAgentScope = 16;             // buffer cache policy: sc1
static_assert(kBM == kRowsTile && kBN == kRowsTile, "tile shape");
static_assert(kStages * kStage <= 160 * 1024, "LDS");
static_assert(kStages * kOps < 64, "vmcnt is a 6-bit counter");

// One DMA of 1 KB: lane l's 16 B at base + off to LDS byte lds + 16 l (M0, which
// the compiler is told it loses; the warning is that nothing restores it).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base)
               : "m0", "memory");
#endif
}
#pragma clang diagnostic pop

// This wave's loads but for the last VM have landed and its LDS reads but for
// the last LGKM have returned; then the workgroup's barrier.
template <int VM, int LGKM>
__device__ __forceinline__ void wait_barrier() {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(%1)\n\ts_barrier" ::"n"(VM), "n"(LGKM) : "memory");
#endif
}

typedef __attribute__((address_space(3))) char lds_char;

// The sums of a workgroup's tile of BM rows, wave w the 64 x 64 block of row
// block w % (BM / 64) and column block w / (BM / 64), to the output or, split,
// through the partials; lds is free (its first word is used).
template <int DT, int BM>
__device__ __forceinline__ void finish_tile(const SpmmArgs& a, f4 (&acc)[4][4], char* lds, int tile, int mtile, int mt,
                                            int split) {
  using E = Elem<DT>;
  typedef typename E::scalar T;
  constexpr int kPartBytes = BM * kBN * 4;  // a split's partial tile
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lg = lane >> 4, li = lane & 15;
  const int wm = wave % (BM / 64), wn = wave / (BM / 64);
  // acc[i][j][e]: batch row row0 + 16 i, output column col0 + 16 j + e.
  const int row0 = mtile * BM + wm * 64 + li;
  const int col0 = tile * kBN + wn * 64 + 4 * lg;
  const int ticket = tile * mt + mtile;
  if (a.splits > 1) {
    // A split's partial tile is stored as the accumulators lie, 16 B per lane:
    // block i, j of wave w at ((w * 16 + 4 i + j) * 64 + lane) * 16 bytes. Stores and loads are coherent at agent scope (sc1), as the 4-byte
    // atomics of the other kernels; those, 64 of them per lane in 64-B pieces,
    // took 9 us (2 splits) to 17 us (4).
    int& is_last = *reinterpret_cast<int*>(lds);
    const size_t tiles = (size_t)a.tiles * (size_t)mt * (kPartBytes / 4);
    float* part = a.partial + (size_t)ticket * (kPartBytes / 4);
    auto rsrc = [&](int sp) {
      return __builtin_amdgcn_make_buffer_rsrc(part + (size_t)sp * tiles, 0, kPartBytes, 0x00020000);
    };
    const int off = (wave * 16 * 64 + lane) * 16;
    {
      const auto rs = rsrc(split);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, acc[i][j]), rs, off + (4 * i + j) * 1024, 0,
                                                 kAgentScope);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tid == 0) {
      const uint32_t prev = __hip_atomic_fetch_add(&a.tickets[ticket], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      is_last = (prev == (uint32_t)(a.splits - 1)) ? 1 : 0;
    }
    __syncthreads();
    if (!is_last) return;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    for (int sp = 0; sp < a.splits; ++sp) {
      const auto rs = rsrc(sp);
      u32x4 t[4][4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          t[i][j] = __builtin_amdgcn_raw_buffer_load_b128(rs, off + (4 * i + j) * 1024, 0, kAgentScope);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] += __builtin_bit_cast(f4, t[i][j]);
    }
  }
  typedef T t4 __attribute__((ext_vector_type(4)));
  T* __restrict__ out = static_cast<T*>(a.out);
#pragma unroll
  for (int i = 0; i < 4; ++i)
    if (row0 + 16 * i < a.batch)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        t4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = E::from_f32(acc[i][j][e]);
        *reinterpret_cast<t4*>(out + (long long)(row0 + 16 * i) * a.out_row_stride + col0 + 16 * j) = v;
      }
  if (a.splits > 1 && tid == 0) __hip_atomic_store(&a.tickets[ticket], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int DT>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void nm_spmm_rows_kernel(McGroupArgs g,
                                                                                                      int mt) {
  using E = Elem<DT>;
  typedef typename E::scalar T;
  __shared__ __attribute__((aligned(16))) char lds[kStages * kStage];

  // Workgroups go round-robin to the 8 XCDs; workgroup b takes the l-th of all
  // tiles, l counting through one XCD's share before the next's, row tiles
  // fastest: the row tiles of one output tile then run on one XCD at about the
  // same time, and its weights come from HBM once.
  const int total = (int)gridDim.x, xcd = (int)blockIdx.x & 7, per = total >> 3, extra = total & 7;
  const int blk = xcd * per + min(xcd, extra) + ((int)blockIdx.x >> 3);
  int gi = 0;
#pragma unroll
  for (int j = 1; j < kMcMaxGroup; ++j) gi += (j < g.n && blk >= g.first[j]) ? 1 : 0;
  const SpmmArgs& a = g.p[gi];
  const int l0 = blk - g.first[gi];
  const int mtile = l0 % mt, tile = (l0 / mt) % a.tiles, split = l0 / mt / a.tiles;

  const int h = a.h, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lg = lane >> 4, li = lane & 15;
  const int wm = wave & 1, wn = wave >> 1;  // the wave's 64 x 64 quarter
  const int c0 = split * a.rows_per_split;
  const int cw = min(a.rows_per_split, a.w - c0);
  const int nch = (cw + kCK - 1) / kCK;
  const int rem = cw - (nch - 1) * kCK;  // columns of the last chunk
  const int rbk = (int)a.x_row_stride;   // 16-row blocks of the gathered activations
  const int rb0 = mtile * (kBM / 16);

  // DMA addresses. Weights: lane tid fills slot tid % 16 of row tid / 16 + 16 i
  // (i < 4), which holds column slot (tid % 16) ^ 2 (row & 3); the last chunk's
  // rows past the split read its last row. Activations: fragment wave + 4 i of
  // the chunk's 16 (K step f / 8, row block f % 8; blocks past the batch read
  // its last).
  const int wrow = tid >> 4;
  const int gcol = tile * kBN + 8 * ((tid & 15) ^ (2 * (wrow & 3)));
  uint32_t woff[4], wlast[4], aoff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    woff[i] = (uint32_t)(((size_t)(wrow + 16 * i) * (size_t)h + (size_t)gcol) * 2);
    wlast[i] = (uint32_t)(((size_t)min(wrow + 16 * i, rem - 1) * (size_t)h + (size_t)gcol) * 2);
    const int f = wave + 4 * i;
    aoff[i] = (uint32_t)(((f >> 3) * rbk + min(rb0 + (f & 7), rbk - 1)) * 1024 + lane * 16);
  }
  const char* wbase = static_cast<const char*>(a.mat_data) + (size_t)c0 * (size_t)h * 2;
  const char* abase = static_cast<const char*>(a.x) + (size_t)(c0 / kCK) * (size_t)rbk * 2048;
  const size_t wstep = (size_t)kCK * (size_t)h * 2, astep = (size_t)rbk * 2048;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_char*)lds;
  const uint32_t ldsw = lds0 + (uint32_t)wave * 1024;
  // A chunk's loads go out in two halves of kOps / 2, the weights, then the
  // activations. Every step issues the same number (a static vmcnt count); steps
  // past the last chunk read it again.
  struct Source {
    const char *w, *a;
    bool last;
  };
  auto source = [&](int k) {
    const int kk = min(k, nch - 1);
    return Source{wbase + (size_t)kk * wstep, abase + (size_t)kk * astep, kk == nch - 1};
  };
  auto load_w = [&](const Source& c, int s, int i) {
    dma16(c.w, c.last ? wlast[i] : woff[i], ldsw + (uint32_t)(s * kStage + i * 4096));
  };
  auto load_a = [&](const Source& c, int s, int i) {
    dma16(c.a, aoff[i], ldsw + (uint32_t)(s * kStage + kWBytes + i * 4096));
  };

  f4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  struct Operands {
    s8 a[4];
    s4 lo[4], hi[4];
  };
  const int rr = 8 * lg + (li >> 2);
  const char* arow = lds + kWBytes + wm * 4096 + lane * 16;
  const char* wcol[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int slot = wn * 8 + 2 * j + ((li & 3) >> 1);
    wcol[j] = lds + rr * 256 + (slot ^ (2 * (rr & 3))) * 16 + (li & 1) * 8;
  }
  constexpr int kReads = 12;  // LDS reads of one operand set
  auto read = [&](Operands& o, int s, int ks, int t) {
    if (t < 4) {
      o.a[t] = *reinterpret_cast<const s8*>(arow + s * kStage + ks * 8192 + t * 1024);
    } else {
      const char* p = wcol[(t - 4) / 2] + s * kStage + ks * 8192;
      if (t % 2 == 0)
        o.lo[(t - 4) / 2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p);
      else
        o.hi[(t - 4) / 2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p + 4 * 256));
    }
  };
  // Half a chunk: 16 multiplies of `cur`, between them (pinned: issued together
  // they would hold up the multiplies behind them) the reads of the next
  // operands and four DMAs.
  auto half = [&](const Operands& cur, auto&& next, auto&& dma) {
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const int i = t % 4, j = t / 4;
      const s8 b = {cur.lo[j][0], cur.lo[j][1], cur.lo[j][2], cur.lo[j][3],
                    cur.hi[j][0], cur.hi[j][1], cur.hi[j][2], cur.hi[j][3]};
      acc[i][j] = mfma16x16x32<DT>(b, cur.a[i], acc[i][j]);  // transposed: a lane gets 4 adjacent outputs
      if (t < kReads) next(t);
      if (i == 1) dma(j);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // The ragged last chunk's rows past the split hold its last row: cleared once
  // it has landed.
  auto clear = [&](int s) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (wrow + 16 * i >= rem)
        *reinterpret_cast<u32x4*>(lds + s * kStage + (wrow + 16 * i) * 256 + (tid & 15) * 16) = u32x4{0u, 0u, 0u, 0u};
    wait_barrier<63, 0>();
  };

#pragma unroll
  for (int s = 0; s < kStages - 1; ++s) {
    const Source c = source(s);
#pragma unroll
    for (int i = 0; i < 4; ++i) load_w(c, s, i);
    if (s < kStages - 2)
#pragma unroll
      for (int i = 0; i < 4; ++i) load_a(c, s, i);
  }
  wait_barrier<(kStages - 3) * kOps + kOps / 2, 0>();
  if (nch == 1 && rem < kCK) clear(0);
  Operands o0, o1;
#pragma unroll
  for (int t = 0; t < kReads; ++t) read(o0, 0, 0, t);
  auto none = [](int) {};
  Source fill = source(kStages - 2);
  for (int k0 = 0;; k0 += kStages) {
#pragma unroll
    for (int s = 0; s < kStages; ++s) {
      const int k = k0 + s;
      half(o0, [&](int t) { read(o1, s, 1, t); }, [&](int i) { load_a(fill, (s + kStages - 2) % kStages, i); });
      if (k + 1 == nch) goto done;
      // Chunk k + 1 has landed; every wave is past its reads of chunk k - 1,
      // whose stage the next loads fill.
      wait_barrier<(kStages - 3) * kOps, kReads>();
      if (k + 2 == nch && rem < kCK) clear((s + 1) % kStages);
      fill = source(k + kStages - 1);
      half(o1, [&](int t) { read(o0, (s + 1) % kStages, 0, t); },
           [&](int i) { load_w(fill, (s + kStages - 1) % kStages, i); });
    }
  }
done:
  half(o1, none, none);
  wait_barrier<0, 0>();  // no DMA into this workgroup's LDS outlives it; its first word is free

  finish_tile<DT, kBM>(a, acc, lds, tile, mtile, mt, split);
}

// The same with tiles of 256 rows: 512 lanes = 8 wave64, two per SIMD, each 64 x
// 64. Against two 128-row tiles a CU reads the weights once instead of twice
// from memory (48 KB into LDS per 64 compressed columns where they take 64), and
// one wave's LDS reads and waits run under the other's multiplies. A step is 32
// compressed columns (8 KB of weights, 16 KB of activations) in a ring of 6
// stages, at least three steps in flight: before step k every wave's loads of
// step k + 1 have landed and its reads of step k - 1, whose stage the loads of
// step k + 5 then fill, have been multiplied.
// Graph replay, gathers included, against the 128-row tiles (us): Llama-3.1-8B
// gate and up at 200 / 500 / 1024 rows 46 / 83 / 155 (56 / 105 / 175), q, k and v at
// 1024 rows 45 (59); a split deep product of few rows stays with those (down at 200
// rows 47 against 43).
constexpr int kTallBM = kRowsTallTile, kTallCK = 32, kTallStages = 6;
constexpr int kTallW = kTallCK * kBN * 2;                // weights of a stage
constexpr int kTallStage = kTallW + kTallBM * kTallCK * 2;
constexpr int kTallOps = 3;                              // DMA instructions per wave per step
static_assert(kTallStages * kTallStage <= 160 * 1024 && kTallStages % 2 == 0, "LDS ring");

template <int DT>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void nm_spmm_rows_tall_kernel(
    McGroupArgs g, int mt) {
  __shared__ __attribute__((aligned(16))) char lds[kTallStages * kTallStage];

  // Tiles in the order of nm_spmm_rows_kernel.
  const int total = (int)gridDim.x, xcd = (int)blockIdx.x & 7, per = total >> 3, extra = total & 7;
  const int blk = xcd * per + min(xcd, extra) + ((int)blockIdx.x >> 3);
  int gi = 0;
#pragma unroll
  for (int j = 1; j < kMcMaxGroup; ++j) gi += (j < g.n && blk >= g.first[j]) ? 1 : 0;
  const SpmmArgs& a = g.p[gi];
  const int l0 = blk - g.first[gi];
  const int mtile = l0 % mt, tile = (l0 / mt) % a.tiles, split = l0 / mt / a.tiles;

  const int h = a.h, tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63, lg = lane >> 4, li = lane & 15;
  const int wm = wave & 3, wn = wave >> 2;  // the wave's 64 x 64 block
  const int c0 = split * a.rows_per_split;
  const int cw = min(a.rows_per_split, a.w - c0);
  const int nch = (cw + kCK - 1) / kCK;  // chunks of two steps
  const int rem = cw - (nch - 1) * kCK;  // columns of the last chunk
  const int rbk = (int)a.x_row_stride;
  const int rb0 = mtile * (kTallBM / 16);

  // DMA addresses, as nm_spmm_rows_kernel's: lane tid fills slot tid % 16 of
  // weight row tid / 16; a wave fills activation fragments wave and wave + 8.
  const int wrow = tid >> 4;
  const int gcol = tile * kBN + 8 * ((tid & 15) ^ (2 * (wrow & 3)));
  uint32_t woff[2], wlast[2];  // of a chunk's two steps
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int row = q * kTallCK + wrow;
    woff[q] = (uint32_t)(((size_t)row * (size_t)h + (size_t)gcol) * 2);
    wlast[q] = (uint32_t)(((size_t)min(row, rem - 1) * (size_t)h + (size_t)gcol) * 2);
  }
  uint32_t aoff[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) aoff[i] = (uint32_t)(min(rb0 + wave + 8 * i, rbk - 1) * 1024 + lane * 16);
  const char* wbase = static_cast<const char*>(a.mat_data) + (size_t)c0 * (size_t)h * 2;
  const char* abase = static_cast<const char*>(a.x) + (size_t)(c0 / kTallCK) * (size_t)rbk * 1024;
  const size_t wstep = (size_t)kCK * (size_t)h * 2, astep = (size_t)rbk * 1024;
  const uint32_t ldsw = (uint32_t)(uintptr_t)(lds_char*)lds + (uint32_t)wave * 1024;
  // DMA i (0 the weights, 1 and 2 the activations) of step q of chunk c into
  // stage s; chunks past the last read it again (a static vmcnt count).
  auto load = [&](int c, int q, int s, int i) {
    const int cc = min(c, nch - 1);
    if (i == 0)
      dma16(wbase + (size_t)cc * wstep, cc == nch - 1 ? wlast[q] : woff[q], ldsw + (uint32_t)(s * kTallStage));
    else
      dma16(abase + (size_t)(2 * cc + q) * astep, aoff[i - 1],
            ldsw + (uint32_t)(s * kTallStage + kTallW + (i - 1) * 8192));
  };

  f4 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  struct Operands {
    s8 a[4];
    s4 lo[4], hi[4];
  };
  const int rr = 8 * lg + (li >> 2);
  const char* arow = lds + kTallW + wm * 4096 + lane * 16;
  const char* wcol[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int slot = wn * 8 + 2 * j + ((li & 3) >> 1);
    wcol[j] = lds + rr * 256 + (slot ^ (2 * (rr & 3))) * 16 + (li & 1) * 8;
  }
  constexpr int kReads = 12;
  auto read = [&](Operands& o, int s, int t) {
    if (t < 4) {
      o.a[t] = *reinterpret_cast<const s8*>(arow + s * kTallStage + t * 1024);
    } else {
      const char* p = wcol[(t - 4) / 2] + s * kTallStage;
      if (t % 2 == 0)
        o.lo[(t - 4) / 2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p);
      else
        o.hi[(t - 4) / 2] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)(p + 4 * 256));
    }
  };
  auto clear = [&](int s, int q) {  // weight rows of the ragged last chunk past the split
    if (q * kTallCK + wrow >= rem)
      *reinterpret_cast<u32x4*>(lds + s * kTallStage + wrow * 256 + (tid & 15) * 16) = u32x4{0u, 0u, 0u, 0u};
    wait_barrier<63, 0>();
  };
  auto step = [&](const Operands& cur, auto&& next, auto&& dma) {
#pragma unroll
    for (int t = 0; t < 16; ++t) {
      const int i = t % 4, j = t / 4;
      const s8 b = {cur.lo[j][0], cur.lo[j][1], cur.lo[j][2], cur.lo[j][3],
                    cur.hi[j][0], cur.hi[j][1], cur.hi[j][2], cur.hi[j][3]};
      acc[i][j] = mfma16x16x32<DT>(b, cur.a[i], acc[i][j]);
      if (t < kReads) next(t);
      if (i == 1 && j < kTallOps) dma(j);
      __builtin_amdgcn_sched_barrier(0);
    }
  };

#pragma unroll
  for (int s = 0; s < kTallStages - 1; ++s)
#pragma unroll
    for (int i = 0; i < kTallOps; ++i) load(s / 2, s % 2, s, i);
  wait_barrier<(kTallStages - 2) * kTallOps, 0>();
  if (nch == 1 && rem < kTallCK) clear(0, 0);
  Operands o0, o1;
#pragma unroll
  for (int t = 0; t < kReads; ++t) read(o0, 0, t);
  auto none = [](int) {};
  for (int k0 = 0;; k0 += kTallStages / 2) {
#pragma unroll
    for (int s = 0; s < kTallStages; s += 2) {
      const int c = k0 + s / 2;
      wait_barrier<(kTallStages - 3) * kTallOps, kReads>();
      if (c + 1 == nch && rem < kCK) clear(s + 1, 1);
      step(o0, [&](int t) { read(o1, s + 1, t); }, [&](int i) { load(c + 2, 1, (s + 5) % kTallStages, i); });
      if (c + 1 == nch) goto done;
      wait_barrier<(kTallStages - 3) * kTallOps, kReads>();
      if (c + 2 == nch && rem < kTallCK) clear((s + 2) % kTallStages, 0);
      step(o1, [&](int t) { read(o0, (s + 2) % kTallStages, t); }, [&](int i) { load(c + 3, 0, s, i); });
    }
  }
done:
  step(o1, none, none);
  wait_barrier<0, 0>();  // no DMA into this workgroup's LDS outlives it; its first word is free
  finish_tile<DT, kTallBM>(a, acc, lds, tile, mtile, mt, split);
}
}  // namespace

// Launch the product over the gathered activations; dtype fp16 or bf16, every
// h a multiple of 128, bm rows per tile (kRowsTile or kRowsTallTile), blocks the
// sum of tiles x mt x splits.
void launch_rows_product(int dtype, const McGroupArgs& g, int bm, int mt, int blocks, hipStream_t st) {
  const bool f16 = dtype == NM_DTYPE_F16;
  if (bm == kRowsTallTile)
    hipLaunchKernelGGL(
        (f16 ? nm_spmm_rows_tall_kernel<NM_DTYPE_F16> : nm_spmm_rows_tall_kernel<NM_DTYPE_BF16>), dim3(blocks),
        dim3(512), 0, st, g, mt);
  else
    hipLaunchKernelGGL((f16 ? nm_spmm_rows_kernel<NM_DTYPE_F16> : nm_spmm_rows_kernel<NM_DTYPE_BF16>), dim3(blocks),
                       dim3(256), 0, st, g, mt);
}

}  // namespace nm_hip
