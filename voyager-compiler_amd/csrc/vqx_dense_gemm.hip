// Dense bf16 product of two K-major matrices, fp32 accumulation:
//   out[b, m, n] = sum_k A[b, m, k] * B[b, n, k]  (+ bias[n]),  bf16 out.
// The block-coded products (vqx_mx_gemm.hip) run here once both operands are
// plain bf16 with K contiguous: decoded weights ([N][K], decoded once) and
// activations decoded by the streaming pass.
//
// A workgroup of 256 threads computes 128 x BN outputs: 4 waves, one per
// SIMD, each 64 x BN / 2 as 32 x 32 v_mfma_f32_32x32x16_bf16 tiles.  K
// advances by BK per step through a ring of LDS stages, filled by buffer
// loads that write LDS directly: no register staging, and a step's fills are
// in flight for kStages - 1 steps.  A step is BK / 16 slices of 16; while a
// slice computes, the next one's fragments are read from LDS, one read
// behind each MFMA, and a step's fills are spread over BK / 16 - 1 slices
// (issued together they stall the wave: 2048 x 11008 x 4096 180 -> 169 us).
// One barrier per step, before its last slice.  The results are staged
// through LDS so that every store instruction writes whole rows of the tile,
// non-temporally: written straight from the accumulators (32-byte pieces of
// 32 rows, through the L2 that holds the operands) 2048 x 11008 x 4096 took
// 173 us instead of 158, and the attention scores 101 instead of 70.
//
// Three shapes (us; 1000 x 4096 x 4096 / 2048 x 11008 x 4096 / 32 products of
// 2048 x 2048 x 128; launches on one set of buffers, in parentheses rotating
// over 600 MB of them, all on one box; boxes differ by 10%, and the pairs of
// figures elsewhere in this file are each from one box, on one set):
//   kWide   BN 256, BK 64, 3 stages of 48 KiB:   41 (56) / 147 (171) / 103 (102)
//   kNarrow BN 128, BK 64, 3 stages of 32 KiB:   31 (41) / 169 (202) / 131 (131)
//   kShort  BN 256, BK 32, 3 stages of 24 KiB, two workgroups per CU (one
//           loads while the other stores):       53 (78) / 182 (212) /  75 (81)
// What bounds kWide (2048 x 11008 x 4096, 688 tiles = 2.69 rounds of the
// CUs): per step and CU 1024 cycles of MFMA against 1152 of LDS (96 KiB of
// fragment reads, 48 KiB of fills, 128 B per cycle) and 768 of the vector
// memory path; by counters (2048 x 4096 x 11008) the MFMA pipe is busy 77% of
// the cycles, at the 1.6 GHz the power limit leaves (141 us).  A 256 x 256 tile of 8
// waves reads less LDS per product and keeps the pipe 85% busy at 8192^3, but
// at 1.4 GHz, and leaves 1.34 rounds here: 166 to 184 us.
//
// Products with too few tiles for the CUs split K (plan_dense): the pieces
// leave fp32 sums in a caller-owned workspace, which dense_reduce_kernel adds
// in a fixed order.
#include "vqx_kernels.h"

namespace vqx {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(3))) const u32x4 lds_cu32x4;

constexpr int kBM = 128;
constexpr int kBand = 8;  // row tiles walked together

template <int BN, int BK, int OCC>
struct Shape {
  static constexpr int kBN = BN, kBK = BK, kOcc = OCC, kStages = 3;  // OCC: workgroups per CU
  static constexpr int kFN = BN / 64;                                // 32-column blocks per wave
  static constexpr int kRow = 2 * BK, kRows = 1024 / kRow;           // bytes of a stage row; rows per 1 KiB fill
  static constexpr int kStA = kBM * kRow, kStB = BN * kRow;          // bytes per stage
  static constexpr int kFillA = kBM / 4 / kRows, kFillB = BN / 4 / kRows, kFills = kFillA + kFillB;  // per wave, step
  static constexpr int kSlices = BK / 16, kFillSlices = kSlices - 1;
  static constexpr int kTileF32 = kBM * BN;                          // fp32 sums of one tile
  static constexpr int kOutRow = 2 * BN + 16;                        // bytes of a staged output row (padded)
  static constexpr int kLds = kStages * (kStA + kStB);
  static_assert(kBM * kOutRow <= kLds, "the output staging fits the stages");
};
typedef Shape<256, 64, 1> kWide;
typedef Shape<128, 64, 1> kNarrow;
typedef Shape<256, 32, 2> kShort;

// LDS slot (of 16 bytes) of chunk c in stage row r: 16 consecutive rows meet
// 16 distinct slots of the 64 banks for any one chunk (64-deep rows are half
// of the banks long, 32-deep ones a quarter), so fragment reads and fills are
// conflict free.
template <int BK>
__device__ __forceinline__ int slot(int c, int r) {
  return BK == 64 ? c ^ (r & 7) ^ ((r >> 3) & 7) : c ^ ((r >> 2) & 3);
}

struct DenseArgs {
  const uint16_t* a;
  const uint16_t* b;
  const uint16_t* bias;
  uint16_t* out;
  float* ws;
  int64_t a_bstride, b_bstride;  // elements between batch items
  uint32_t lda, ldb;             // bytes between rows
  int M, N, K, tm, tn, tiles, splits;
};

// Tile -> (batch item, first row, first column): within an item, bands of
// kBand row tiles, row tiles fastest, so the tiles that run together on an
// XCD share both row slabs of A and column slabs of B in its L2.
struct TilePos {
  int64_t b;
  int m0, n0;
};

template <int kBN>
__device__ __forceinline__ TilePos tile_pos(int tile, const DenseArgs& p) {
  const int per = p.tm * p.tn;
  const int b = tile / per, t = tile - b * per;
  const int band = t / (kBand * p.tn), r = t - band * (kBand * p.tn);
  const int rows = p.tm - band * kBand < kBand ? p.tm - band * kBand : kBand;
  return {b, (band * kBand + r % rows) * kBM, (r / rows) * kBN};
}

// Up to eight columns of a row of any alignment: through the L2, which joins
// the pieces of a line (scores of 1333 x 1333: 39 us, non-temporally 52).
__device__ __forceinline__ void store_any(uint16_t* o, int n, u32x4 v) {
  if (n >= 8) {
    __builtin_memcpy(o, &v, 16);
    return;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (e < n) o[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
}

__device__ __forceinline__ float bias_at(const uint16_t* bias, int n, int N) { return n < N ? bf2f(bias[n]) : 0.0f; }

template <int N>
__device__ __forceinline__ void wait_fills() {  // all but the last N loads of this wave have landed
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

// The barrier and the compiler fences around it: LDS is written by loads the
// compiler does not order against its reads.
__device__ __forceinline__ void stage_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}

template <int I>
struct Int {
  static constexpr int value = I;
};

template <typename S>
__global__ __launch_bounds__(256, S::kOcc) void dense_gemm_kernel(DenseArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)  // address-space casts and builtins the host pass does not take
  constexpr int kBN = S::kBN, kBK = S::kBK, kStages = S::kStages, kFN = S::kFN, kRow = S::kRow, kRows = S::kRows;
  constexpr int kStA = S::kStA, kStB = S::kStB, kFillA = S::kFillA, kFillB = S::kFillB, kFills = S::kFills;
  constexpr int kSlices = S::kSlices, kFillSlices = S::kFillSlices, kOutRow = S::kOutRow;
  constexpr int kMfmas = 2 * kFN;  // per slice
  __shared__ __attribute__((aligned(1024))) uint8_t lds[S::kLds];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1, lr = lane & 31, lk = lane >> 5;

  // workgroups go to the XCDs in turn; within each full round of 256, an XCD
  // takes 32 consecutive units (they share slabs of A and B in its L2)
  const int units = gridDim.x, bid = blockIdx.x;
  const int round = bid & ~255, w = bid & 255;
  const int cnt = units - round < 256 ? units - round : 256;
  const int unit = cnt % 8 == 0 ? round + (w & 7) * (cnt / 8) + (w >> 3) : bid;
  // unit = split * tiles + tile: the pieces of one tile run far apart, the
  // tiles of one k range together
  const int split = unit / p.tiles, tile = unit - split * p.tiles;
  const TilePos pos = tile_pos<kBN>(tile, p);
  const int nk = p.K / kBK;
  const int k0 = (int)((int64_t)nk * split / p.splits), n = (int)((int64_t)nk * (split + 1) / p.splits) - k0;

  // A fill covers kRows stage rows of kRow bytes: lane l writes LDS slot
  // l % (64 / kRows) of row l / (64 / kRows) (the hardware places lanes 16
  // bytes apart) and reads the chunk that belongs there (slot() is its own
  // inverse).  Rows past the end read the last row (their results are not
  // stored).
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.a + pos.b * p.a_bstride), 0, (int)((uint32_t)(p.M - 1) * p.lda + 2u * (uint32_t)p.K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.b + pos.b * p.b_bstride), 0, (int)((uint32_t)(p.N - 1) * p.ldb + 2u * (uint32_t)p.K), 0x00020000);
  constexpr int kLanes = 64 / kRows;  // lanes per row
  uint32_t va[kFillA], vb[kFillB];
#pragma unroll
  for (int i = 0; i < kFillA; ++i) {
    const int r = wave * (kBM / 4) + kRows * i + lane / kLanes, m = pos.m0 + r < p.M ? pos.m0 + r : p.M - 1;
    va[i] = (uint32_t)m * p.lda + 16u * (uint32_t)slot<kBK>(lane % kLanes, r);
  }
#pragma unroll
  for (int i = 0; i < kFillB; ++i) {
    const int r = wave * (kBN / 4) + kRows * i + lane / kLanes, c = pos.n0 + r < p.N ? pos.n0 + r : p.N - 1;
    vb[i] = (uint32_t)c * p.ldb + 16u * (uint32_t)slot<kBK>(lane % kLanes, r);
  }
  auto fill = [&](int i, int ks, int st) {
    if (i < kFillA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          ra, (lds_void*)(lds + st * kStA + (wave * (kBM / 4) + kRows * i) * kRow), 16, va[i], (k0 + ks) * kRow, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rb, (lds_void*)(lds + kStages * kStA + st * kStB + (wave * (kBN / 4) + kRows * (i - kFillA)) * kRow), 16,
          vb[i - kFillA], (k0 + ks) * kRow, 0, 0);
  };

  // Fragment of 32-row block i, slice kk: chunk 2 kk + lk of row 32 i + lr.
  // slot() of a 64-deep row takes row bits 3-5: block i flips chunk bit 2.
  const uint32_t base = (uint32_t)(uintptr_t)(lds_void*)lds;
  uint32_t fa[kSlices], fb[kSlices];
#pragma unroll
  for (int v = 0; v < kSlices; ++v) {
    const uint32_t s = (uint32_t)slot<kBK>(2 * v + lk, lr) << 4;
    fa[v] = base + (uint32_t)((wm * 64 + lr) * kRow) + s;
    fb[v] = base + (uint32_t)(kStages * kStA + (wn * (kBN / 2) + lr) * kRow) + s;
  }
  auto flip = [](int kk, int i) { return kBK == 64 ? kk ^ (2 * (i & 1)) : kk; };
  f32x16 acc[2][kFN];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < kFN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  bf16x8 A[2][2], B[2][kFN];  // fragments: the slice that computes, the slice being read
  // read t of slice kk: A0, B0, B1 .., A1 (the order the MFMAs need them)
  auto read = [&](int t, int buf, int kk, int st) {
    if (t == 0 || t == kFN + 1) {
      const int i = t != 0;
      A[buf][i] = __builtin_bit_cast(bf16x8, *(lds_cu32x4*)(size_t)(fa[flip(kk, i)] + i * 32 * kRow + st * kStA));
    } else {
      const int j = t - 1;
      B[buf][j] = __builtin_bit_cast(bf16x8, *(lds_cu32x4*)(size_t)(fb[flip(kk, j)] + j * 32 * kRow + st * kStB));
    }
  };

#pragma unroll
  for (int s = 0; s < kStages; ++s)
    if (s < n) {
#pragma unroll
      for (int i = 0; i < kFills; ++i) fill(i, s, s);
    }
  if (n >= kStages) wait_fills<(kStages - 1) * kFills>();
  else wait_fills<0>();
  stage_barrier();
#pragma unroll
  for (int t = 0; t < kFN + 2; ++t) read(t, 0, 0, 0);

  // Slice KK: the MFMAs on fragment buffer KK & 1; behind each, a fragment
  // read of slice KK + 1 (stage rst) into the other buffer and the step fills
  // that fall there: a step's fills go behind evenly spaced MFMAs of the
  // kFillSlices slices that start with the last one (part Q of them).
  auto slice = [&](auto KK, int rst, bool reads, bool fills, int fks, int fst, auto Q) {
    constexpr int kk = decltype(KK)::value, cb = kk & 1, nb = 1 - cb, q = decltype(Q)::value;
#pragma unroll
    for (int t = 0; t < kMfmas; ++t) {
      acc[t / kFN][t % kFN] =
          __builtin_amdgcn_mfma_f32_32x32x16_bf16(B[cb][t % kFN], A[cb][t / kFN], acc[t / kFN][t % kFN], 0, 0, 0);
      if (reads && t < kFN + 2) read(t, nb, (kk + 1) % kSlices, rst);
      if (fills) {
#pragma unroll
        for (int d = 0; d < kFills; ++d)
          if (d * kMfmas * kFillSlices / kFills == t + q * kMfmas) fill(d, fks, fst);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Step ks in stage ST.  The barrier before the last slice says that every
  // wave has read the last fragments of stage ST (so step ks + kStages may
  // fill it) and that the fills of step ks + 1 have landed.  In a FULL step
  // ks + 2 * kStages <= n at the loop's head, so every fill and read happens:
  // no branches.  (Whole slices with and without fills for the other steps
  // copy accumulators where they join: kShort spills, kWide 165 -> 186 us.)
  auto step = [&](int ks, auto ST, auto FULL) {
    constexpr int st = decltype(ST)::value, next = (st + 1) % kStages, prev = (st + kStages - 1) % kStages;
    constexpr bool full = decltype(FULL)::value != 0;
    if constexpr (kSlices == 4) {
      const bool fprev = ks > 0 && (full || ks + kStages - 1 < n);  // the rest of the fills the step before began
      slice(Int<0>{}, st, true, fprev, ks + kStages - 1, prev, Int<1>{});
      slice(Int<1>{}, st, true, fprev, ks + kStages - 1, prev, Int<2>{});
    }
    slice(Int<kSlices - 2>{}, st, true, false, 0, 0, Int<kFillSlices>{});
    if (full || ks + kStages - 1 < n) wait_fills<(kStages - 2) * kFills>();
    else wait_fills<0>();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    stage_barrier();
    slice(Int<kSlices - 1>{}, next, full || ks + 1 < n, full || ks + kStages < n, ks + kStages, st, Int<0>{});
  };
  int ks = 0;
  for (; ks + 2 * kStages <= n; ks += kStages) {
    step(ks, Int<0>{}, Int<1>{});
    step(ks + 1, Int<1>{}, Int<1>{});
    step(ks + 2, Int<2>{}, Int<1>{});
  }
  for (; ks < n; ks += kStages) {
    step(ks, Int<0>{}, Int<0>{});
    if (ks + 1 < n) step(ks + 1, Int<1>{}, Int<0>{});
    if (ks + 2 < n) step(ks + 2, Int<2>{}, Int<0>{});
  }

  // Accumulator layout: lane (lr, lk) of block (i, j) holds row 32 i + lr,
  // columns 32 j + 8 g + 4 lk + e in element 4 g + e.
  if (p.splits > 1) {  // fp32 sums in this order, whole lines per store
    f32x4* const ws = reinterpret_cast<f32x4*>(p.ws + (int64_t)unit * S::kTileF32) + wave * (S::kTileF32 / 16) + lane;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < kFN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          ws[((i * kFN + j) * 4 + g) * 64] =
              f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
    return;
  }
  if (p.bias) {
#pragma unroll
    for (int j = 0; j < kFN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const float b = bias_at(p.bias, pos.n0 + wn * (kBN / 2) + j * 32 + 8 * (e >> 2) + 4 * lk + (e & 3), p.N);
        acc[0][j][e] += b;
        acc[1][j][e] += b;
      }
  }
  // the last step's barrier lies before its last slice, whose fragments were
  // read before it: no wave reads the stages any more
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < kFN; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const f32x16& v = acc[i][j];
        *reinterpret_cast<u32x2*>(lds + (wm * 64 + i * 32 + lr) * kOutRow +
                                  2 * (wn * (kBN / 2) + j * 32 + 8 * g + 4 * lk)) =
            u32x2{pack_bf16x2(v[4 * g], v[4 * g + 1]), pack_bf16x2(v[4 * g + 2], v[4 * g + 3])};
      }
  __syncthreads();
  constexpr int kChunks = kBN / 8, kRowsOut = 256 / kChunks;  // 16-byte chunks per row; rows per round of the workgroup
  const int c = threadIdx.x % kChunks, nn = pos.n0 + c * 8;
  uint16_t* const ob = p.out + pos.b * (int64_t)p.M * p.N;
  const bool rows16 = (p.N & 7) == 0 && ((uintptr_t)p.out & 15) == 0;  // every row 16-byte aligned
#pragma unroll
  for (int q = 0; q < kBM / kRowsOut; ++q) {
    const int r = q * kRowsOut + threadIdx.x / kChunks, m = pos.m0 + r;
    const u32x4 v = *reinterpret_cast<const u32x4*>(lds + r * kOutRow + c * 16);
    if (m < p.M && nn < p.N) {
      uint16_t* const o = ob + (int64_t)m * p.N + nn;
      if (rows16) st_nt(reinterpret_cast<u32x4*>(o), v);
      else store_any(o, p.N - nn, v);
    }
  }
#endif
}

// The split tiles' sums: each thread adds four columns of one row over the
// pieces, in the order of the k ranges, and stores them as bf16.
template <typename S>
__global__ __launch_bounds__(256) void dense_reduce_kernel(DenseArgs p) {
  constexpr int kQuads = S::kTileF32 / 4, kFN = S::kFN;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int tile = (int)(t / kQuads), q = (int)(t % kQuads);
  const int lane = q & 63, blk = (q >> 6) % (8 * kFN), wave = q / (512 * kFN);
  const int i = blk / (4 * kFN), j = (blk >> 2) % kFN, g = blk & 3;
  const TilePos pos = tile_pos<S::kBN>(tile, p);
  const int m = pos.m0 + (wave >> 1) * 64 + i * 32 + (lane & 31);
  const int n = pos.n0 + (wave & 1) * (S::kBN / 2) + j * 32 + 8 * g + 4 * (lane >> 5);
  if (m >= p.M || n >= p.N) return;
  const f32x4* src = reinterpret_cast<const f32x4*>(p.ws) + (int64_t)tile * kQuads + q;
  const int64_t step = (int64_t)p.tiles * kQuads;
  f32x4 s = src[0];
  for (int k = 1; k < p.splits; ++k) s += src[k * step];
  uint16_t* const o = p.out + (pos.b * p.M + m) * (int64_t)p.N + n;
  if (p.bias) {
#pragma unroll
    for (int e = 0; e < 4; ++e) s[e] += bias_at(p.bias, n + e, p.N);
  }
  const u32x2 v = {pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3])};
  if (n + 4 <= p.N) {
    __builtin_memcpy(o, &v, 8);
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (n + e < p.N) o[e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
  }
}

// The shape and K splits of a product: the least of this estimate (us),
// fitted to measurements on one MI355X.  A full machine takes 0.82 us per
// step on kWide and 0.45 on kNarrow; a unit's start and output 3 and 2.5; a
// split 4 for the second launch and 0.2 per MB of fp32 sums.  Measured on one
// set of buffers / rotating over 600 MB / estimated: 1000 x 4096 x 4096 kNarrow
// 31 / 41 / 31, kWide in 2 pieces 41 / 46 / 40; 512 x 4096 x 4096 kNarrow in 2
// pieces 24 / 31 / 24, kWide in 4 27 / 32 / 27; 333 x 4096 x 11008 kWide in 5
// pieces 38 / 49 / 42, kNarrow in 2 39 / 58 / 48; 2048 x 11008 x 4096 kWide
// 147 / 171 / 166, kNarrow 169 / 202 / 188.
// Products of K <= 128 are bound by the output: kShort (the attention scores
// 75 us against 103 and 131), or kNarrow while its tiles are one round of the
// CUs (one 2048 x 2048 x 128 6.5 us against 7.8, 12 x 197 x 197 x 64 5.4
// against 7.6; at 180 kShort tiles, 12 x 577 x 577 x 64, 11.2 against 11.0).
enum ShapeId : int { kShapeWide = 0, kShapeNarrow = 1, kShapeShort = 2 };

struct Plan {
  int shape, splits;
  int64_t tiles;
};

template <typename S>
int64_t tiles_of(int64_t batch, int64_t M, int64_t N) {
  return batch * ((M + kBM - 1) / kBM) * ((N + S::kBN - 1) / S::kBN);
}

Plan plan_dense(int64_t batch, int64_t M, int64_t N, int64_t K, bool may_split) {
  const int64_t nk = K / 64, cus = num_cus();
  if (K <= 128) {
    const int64_t narrow = tiles_of<kNarrow>(batch, M, N);
    if (narrow <= cus) return {kShapeNarrow, 1, narrow};
    return {kShapeShort, 1, tiles_of<kShort>(batch, M, N)};
  }
  Plan best{kShapeWide, 1, 0};
  double cost = 0.0;
  for (int shape = kShapeWide; shape <= kShapeNarrow; ++shape) {
    const bool wide = shape == kShapeWide;
    const int64_t tiles = wide ? tiles_of<kWide>(batch, M, N) : tiles_of<kNarrow>(batch, M, N);
    const double mb = (wide ? kWide::kTileF32 : kNarrow::kTileF32) * 4.0e-6;
    for (int s = 1; s <= (may_split ? 16 : 1) && (s == 1 || 4 * s <= nk); ++s) {
      const double rounds = (double)((tiles * s + cus - 1) / cus), steps = (double)((nk + s - 1) / s);
      const double c = rounds * (wide ? 0.82 * steps + 3.0 : 0.45 * steps + 2.5) +
                       (s > 1 ? 4.0 + 0.2 * mb * (double)(tiles * s) : 0.0);
      if (best.tiles == 0 || c < cost) {
        best = {shape, s, tiles};
        cost = c;
      }
    }
  }
  return best;
}

template <typename S>
int launch_dense(const DenseArgs& p, hipStream_t st) {
  hipLaunchKernelGGL(dense_gemm_kernel<S>, dim3((unsigned)(p.tiles * p.splits)), dim3(256), 0, st, p);
  const int rc = check_launch("dense_gemm_kernel");
  if (rc || p.splits == 1) return rc;
  hipLaunchKernelGGL(dense_reduce_kernel<S>, dim3((unsigned)(p.tiles * (S::kTileF32 / 4 / 256))), dim3(256), 0, st, p);
  return check_launch("dense_reduce_kernel");
}

}  // namespace

bool dense_gemm_takes(int64_t batch, int64_t M, int64_t N, int64_t K) {
  return K % 64 == 0 && batch >= 1 && M >= 1 && N >= 1 && K >= 64 && batch <= INT32_MAX && M <= INT32_MAX &&
         N <= INT32_MAX && K <= INT32_MAX && tiles_of<kNarrow>(1, M, N) <= INT32_MAX &&
         tiles_of<kNarrow>(batch, M, N) <= INT32_MAX / 256;  // the launches' grids fit 32 bits
}

int64_t dense_gemm_workspace(int64_t batch, int64_t M, int64_t N, int64_t K) {
  const Plan d = plan_dense(batch, M, N, K, true);
  const int64_t tile = (d.shape == kShapeNarrow ? kNarrow::kTileF32 : kWide::kTileF32) * (int64_t)sizeof(float);
  return d.splits > 1 ? d.tiles * d.splits * tile : 0;
}

int dense_gemm(const uint16_t* a, int64_t lda, int64_t a_bstride, const uint16_t* b, int64_t ldb, int64_t b_bstride,
               const uint16_t* bias, uint16_t* out, int64_t batch, int64_t M, int64_t N, int64_t K, void* workspace,
               int64_t workspace_bytes, hipStream_t st) {
  if (!dense_gemm_takes(batch, M, N, K)) return set_error(kErrInvalid, "dense_gemm: unsupported shape");
  const int64_t need = dense_gemm_workspace(batch, M, N, K);
  const bool split = need > 0 && workspace && workspace_bytes >= need;  // without a workspace: whole tiles
  if (split && !aligned(workspace, 16)) return set_error(kErrInvalid, "dense_gemm: workspace must be 16-byte aligned");
  const Plan d = plan_dense(batch, M, N, K, split);
  DenseArgs p;
  p.a = a;
  p.b = b;
  p.bias = bias;
  p.out = out;
  p.ws = static_cast<float*>(workspace);
  p.a_bstride = a_bstride;
  p.b_bstride = b_bstride;
  p.lda = (uint32_t)(2 * lda);
  p.ldb = (uint32_t)(2 * ldb);
  p.M = (int)M;
  p.N = (int)N;
  p.K = (int)K;
  p.tm = (int)((M + kBM - 1) / kBM);
  p.tn = (int)(d.shape == kShapeNarrow ? (N + kNarrow::kBN - 1) / kNarrow::kBN : (N + kWide::kBN - 1) / kWide::kBN);
  p.tiles = (int)d.tiles;
  p.splits = d.splits;
  if (d.shape == kShapeNarrow) return launch_dense<kNarrow>(p, st);
  return d.shape == kShapeShort ? launch_dense<kShort>(p, st) : launch_dense<kWide>(p, st);
}

}  // namespace vqx
