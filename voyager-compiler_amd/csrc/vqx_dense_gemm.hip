// Dense bf16 product of two K-major matrices, fp32 accumulation:
//   out[b, m, n] = sum_k A[b, m, k] * B[b, n, k]  (+ bias[n]),  bf16 out.
// The block-coded products (vqx_mx_gemm.hip) run here once both operands are
// plain bf16 with K contiguous: decoded weights ([N][K], decoded once) and
// activations decoded by the streaming pass.
//
// A workgroup of 256 threads computes 128 x 256 outputs: 4 waves, one per
// SIMD, each 64 x 128 as 2 x 4 v_mfma_f32_32x32x16_bf16 tiles (128 fp32
// accumulators).  K advances by 64 per step through a ring of three LDS
// stages (48 KiB each), filled by buffer loads that write LDS directly: no
// register staging, and the fill of step s + 3 is issued while steps s and
// s + 1 compute.  A step is four 16-deep slices; while slice i computes, the
// fragments of slice i + 1 are read from LDS, one read behind each MFMA, and
// the twelve fills of a step are spread over three slices (issued together
// they stall the wave: 2048 x 11008 x 4096 180 -> 169 us).  One barrier per
// step, before its last slice.
//
// What bounds it (2048 x 11008 x 4096, 688 tiles = 2.69 rounds of the CUs):
// per step and CU 1024 cycles of MFMA against 1152 of LDS (96 KiB of fragment
// reads, 48 KiB of fills, 128 B per cycle) and 768 of the vector memory path.
// A 256 x 256 tile of 8 waves reads less LDS per product and keeps the MFMA
// pipe 85% busy at 8192^3, but clocks 1.4 GHz at the power limit and leaves
// 1.34 rounds here: 184 us, 166 to 182 with the last round split along K.
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

constexpr int kBM = 128, kBN = 256, kBK = 64;  // tile and k per step
constexpr int kStages = 3;
constexpr int kStA = kBM * kBK * 2, kStB = kBN * kBK * 2;  // bytes per stage
constexpr int kFillA = kBM / 32, kFillB = kBN / 32;        // 1 KiB fills per wave and step
constexpr int kFills = kFillA + kFillB;
constexpr int kFillSlices = 3;                             // slices the fills are spread over
constexpr int kBand = 8;                                   // row tiles walked together
constexpr int kTileF32 = kBM * kBN;                        // fp32 sums of one tile

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

__device__ __forceinline__ TilePos tile_pos(int tile, const DenseArgs& p) {
  const int per = p.tm * p.tn;
  const int b = tile / per, t = tile - b * per;
  const int band = t / (kBand * p.tn), r = t - band * (kBand * p.tn);
  const int rows = p.tm - band * kBand < kBand ? p.tm - band * kBand : kBand;
  return {b, (band * kBand + r % rows) * kBM, (r / rows) * kBN};
}

// Eight output columns n .. n + 7 of row m.  N % 8 == 0 with a 16-byte
// aligned output is one aligned store; otherwise the store is unaligned, and
// element by element past the last whole 8.
__device__ __forceinline__ void store8(uint16_t* out, int n, int N, u32x4 v) {
  if (n + 8 <= N) {
    __builtin_memcpy(out + n, &v, 16);
    return;
  }
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (n + e < N) out[n + e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
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

__global__ __launch_bounds__(256, 1) void dense_gemm_kernel(DenseArgs p) {
#if defined(__HIP_DEVICE_COMPILE__)  // address-space casts and builtins the host pass does not take
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kStages * (kStA + kStB)];
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
  const TilePos pos = tile_pos(tile, p);
  const int nk = p.K / kBK;
  const int k0 = (int)((int64_t)nk * split / p.splits), n = (int)((int64_t)nk * (split + 1) / p.splits) - k0;

  // Fill i of a wave covers 8 tile rows of 128 bytes: lane l writes LDS slot
  // l & 7 of row l >> 3 (the hardware places lanes 16 bytes apart), and reads
  // the chunk that belongs there, slot ^ (row & 7) ^ ((row >> 3) & 7).  Rows
  // past the end read the last row (their results are not stored).
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.a + pos.b * p.a_bstride), 0, (int)((uint32_t)(p.M - 1) * p.lda + 2u * (uint32_t)p.K), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.b + pos.b * p.b_bstride), 0, (int)((uint32_t)(p.N - 1) * p.ldb + 2u * (uint32_t)p.K), 0x00020000);
  uint32_t va[kFillA], vb[kFillB];
#pragma unroll
  for (int i = 0; i < kFillA; ++i) {
    const int r = wave * (kBM / 4) + 8 * i + (lane >> 3), m = pos.m0 + r < p.M ? pos.m0 + r : p.M - 1;
    va[i] = (uint32_t)m * p.lda + 16u * (uint32_t)((lane & 7) ^ (r & 7) ^ ((r >> 3) & 7));
  }
#pragma unroll
  for (int i = 0; i < kFillB; ++i) {
    const int r = wave * (kBN / 4) + 8 * i + (lane >> 3), c = pos.n0 + r < p.N ? pos.n0 + r : p.N - 1;
    vb[i] = (uint32_t)c * p.ldb + 16u * (uint32_t)((lane & 7) ^ (r & 7) ^ ((r >> 3) & 7));
  }
  auto fill = [&](int i, int ks, int st) {
    if (i < kFillA)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, (lds_void*)(lds + st * kStA + (wave * (kBM / 4) + 8 * i) * 128), 16,
                                               va[i], (k0 + ks) * 128, 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rb, (lds_void*)(lds + kStages * kStA + st * kStB + (wave * (kBN / 4) + 8 * (i - kFillA)) * 128), 16,
          vb[i - kFillA], (k0 + ks) * 128, 0, 0);
  };

  // Fragment reads: row lr of 32-row block i, chunk 2 kk + lk, in slot
  // (2 kk) ^ (4 (i & 1)) ^ x.  16 consecutive rows meet 16 distinct (row
  // parity, slot) pairs: no bank conflicts.
  const uint32_t x = (uint32_t)(lk ^ (lr & 7) ^ (lr >> 3)), base = (uint32_t)(uintptr_t)(lds_void*)lds;
  uint32_t fa[4], fb[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    fa[v] = base + (uint32_t)(wm * 64 + lr) * 128u + (((2u * v) ^ x) << 4);
    fb[v] = base + (uint32_t)kStages * kStA + (uint32_t)(wn * 128 + lr) * 128u + (((2u * v) ^ x) << 4);
  }
  f32x16 acc[2][4];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  bf16x8 A[2][2], B[2][4];  // fragments: the slice that computes, the slice being read
  // read t of slice kk: A0, B0 .. B3, A1 (the order the MFMAs need them)
  auto read = [&](int t, int buf, int kk, int st) {
    if (t == 0 || t == 5) {
      const int i = t == 5;
      A[buf][i] = __builtin_bit_cast(bf16x8, *(lds_cu32x4*)(size_t)(fa[kk ^ (2 * i)] + i * 4096 + st * kStA));
    } else {
      const int j = t - 1;
      B[buf][j] = __builtin_bit_cast(bf16x8, *(lds_cu32x4*)(size_t)(fb[kk ^ (2 * (j & 1))] + j * 4096 + st * kStB));
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
  for (int t = 0; t < 6; ++t) read(t, 0, 0, 0);

  // Slice KK: 8 MFMAs on fragment buffer KK & 1; behind each, a fragment read
  // of slice KK + 1 (stage rst) into the other buffer and the step fills that
  // fall there: fill d of a step goes behind MFMA 8/4 d of the kFillSlices
  // slices that start with slice 3 (part Q of them).
  auto slice = [&](auto KK, int rst, bool reads, bool fills, int fks, int fst, auto Q) {
    constexpr int kk = decltype(KK)::value, cb = kk & 1, nb = 1 - cb, q = decltype(Q)::value;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      acc[t >> 2][t & 3] =
          __builtin_amdgcn_mfma_f32_32x32x16_bf16(B[cb][t & 3], A[cb][t >> 2], acc[t >> 2][t & 3], 0, 0, 0);
      if (reads && t < 6) read(t, nb, (kk + 1) & 3, rst);
      if (fills) {
#pragma unroll
        for (int d = 0; d < kFills; ++d)
          if (d * 8 * kFillSlices / kFills == t + q * 8) fill(d, fks, fst);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Step ks in stage ST.  The barrier before slice 3 says that every wave has
  // read the last fragments of stage ST (so step ks + 3 may fill it) and that
  // the fills of step ks + 1 have landed.  In a FULL step ks + 2 * kStages <=
  // n at the loop's head, so every fill and read happens: no branches.
  auto step = [&](int ks, auto ST, auto FULL) {
    constexpr int st = decltype(ST)::value, next = (st + 1) % kStages, prev = (st + kStages - 1) % kStages;
    constexpr bool full = decltype(FULL)::value != 0;
    const bool fprev = ks > 0 && (full || ks + kStages - 1 < n);  // the rest of the fills begun in slice 3 before
    slice(Int<0>{}, st, true, fprev, ks + kStages - 1, prev, Int<1>{});
    slice(Int<1>{}, st, true, fprev, ks + kStages - 1, prev, Int<2>{});
    slice(Int<2>{}, st, true, false, 0, 0, Int<3>{});
    if (full) wait_fills<(kStages - 2) * kFills>();
    else wait_fills<0>();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    stage_barrier();
    slice(Int<3>{}, next, full || ks + 1 < n, full || ks + kStages < n, ks + kStages, st, Int<0>{});
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
    f32x4* const ws = reinterpret_cast<f32x4*>(p.ws + (int64_t)unit * kTileF32) + wave * 2048 + lane;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          ws[((i * 4 + j) * 4 + g) * 64] =
              f32x4{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
    return;
  }
  uint16_t* const ob = p.out + pos.b * (int64_t)p.M * p.N;
#pragma unroll
  for (int j = 0; j < 4; ++j)
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      const int n4 = pos.n0 + wn * 128 + j * 32 + 8 * g + 4 * lk;
      float bs[8] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
      if (p.bias) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          bs[e] = bias_at(p.bias, n4 + e, p.N);
          bs[4 + e] = bias_at(p.bias, n4 + 8 + e, p.N);
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const f32x16& c = acc[i][j];
        // the halves of the wave trade quads: lanes 0-31 get columns 8 g ..
        // 8 g + 7, lanes 32-63 the next eight
        const auto s0 = __builtin_amdgcn_permlane32_swap(
            pack_bf16x2(c[4 * g] + bs[0], c[4 * g + 1] + bs[1]), pack_bf16x2(c[4 * g + 4] + bs[4], c[4 * g + 5] + bs[5]),
            false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(
            pack_bf16x2(c[4 * g + 2] + bs[2], c[4 * g + 3] + bs[3]),
            pack_bf16x2(c[4 * g + 6] + bs[6], c[4 * g + 7] + bs[7]), false, false);
        const int m = pos.m0 + wm * 64 + i * 32 + lr;
        if (m < p.M) store8(ob + (int64_t)m * p.N, pos.n0 + wn * 128 + j * 32 + 8 * (g + lk), p.N, u32x4{s0[0], s1[0], s0[1], s1[1]});
      }
    }
#endif
}

// The split tiles' sums: each thread adds four columns of one row over the
// pieces, in the order of the k ranges, and stores them as bf16.
__global__ __launch_bounds__(256) void dense_reduce_kernel(DenseArgs p) {
  constexpr int kQuads = kTileF32 / 4;
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int tile = (int)(t / kQuads), q = (int)(t % kQuads);
  const int lane = q & 63, blk = (q >> 6) & 31, wave = q >> 11;
  const int i = blk >> 4, j = (blk >> 2) & 3, g = blk & 3;
  const TilePos pos = tile_pos(tile, p);
  const int m = pos.m0 + (wave >> 1) * 64 + i * 32 + (lane & 31);
  const int n = pos.n0 + (wave & 1) * 128 + j * 32 + 8 * g + 4 * (lane >> 5);
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

// K splits of a product, from measurement (one MI355X): a step takes 0.86 us
// on a CU, a unit's start and epilogue about 4 steps, a split about 5 for the
// second launch and 0.06 steps per piece for its fp32 sums.  333 x 4096 x
// 11008: 5 splits 47 us, 4 splits 50; 512 x 4096 x 4096: 3 or 4 splits 29 us;
// 1000 x 4096 x 4096: 2 splits and whole tiles both 42 us.
int plan_dense(int64_t tiles, int64_t nk) {
  const int64_t cus = num_cus();
  int best = 1;
  double cost = 0.0;
  for (int s = 1; s <= 16 && 4 * s <= nk; ++s) {
    const int64_t rounds = (tiles * s + cus - 1) / cus;
    const double c = (double)rounds * ((double)((nk + s - 1) / s) + 4.0) + (s > 1 ? 5.0 + 0.06 * (double)(tiles * s) : 0.0);
    if (s == 1 || c < cost) {
      best = s;
      cost = c;
    }
  }
  return best;
}

int64_t dense_tiles(int64_t batch, int64_t M, int64_t N) {
  return batch * ((M + kBM - 1) / kBM) * ((N + kBN - 1) / kBN);
}

}  // namespace

bool dense_gemm_takes(int64_t batch, int64_t M, int64_t N, int64_t K) {
  return K % kBK == 0 && batch >= 1 && M >= 1 && N >= 1 && K >= kBK && M <= INT32_MAX && N <= INT32_MAX &&
         K <= INT32_MAX && dense_tiles(batch, M, N) <= INT32_MAX / 16;
}

int64_t dense_gemm_workspace(int64_t batch, int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = dense_tiles(batch, M, N);
  const int s = plan_dense(tiles, K / kBK);
  return s > 1 ? tiles * s * kTileF32 * (int64_t)sizeof(float) : 0;
}

int dense_gemm(const uint16_t* a, int64_t lda, int64_t a_bstride, const uint16_t* b, int64_t ldb, int64_t b_bstride,
               const uint16_t* bias, uint16_t* out, int64_t batch, int64_t M, int64_t N, int64_t K, void* workspace,
               int64_t workspace_bytes, hipStream_t st) {
  if (!dense_gemm_takes(batch, M, N, K)) return set_error(kErrInvalid, "dense_gemm: unsupported shape");
  DenseArgs p;
  p.a = a;
  p.b = b;
  p.bias = bias;
  p.out = out;
  p.a_bstride = a_bstride;
  p.b_bstride = b_bstride;
  p.lda = (uint32_t)(2 * lda);
  p.ldb = (uint32_t)(2 * ldb);
  p.M = (int)M;
  p.N = (int)N;
  p.K = (int)K;
  p.tm = (int)((M + kBM - 1) / kBM);
  p.tn = (int)((N + kBN - 1) / kBN);
  const int64_t tiles = dense_tiles(batch, M, N);
  p.tiles = (int)tiles;
  p.splits = 1;
  p.ws = nullptr;
  const int64_t need = dense_gemm_workspace(batch, M, N, K);
  if (need > 0 && workspace && workspace_bytes >= need) {  // without a workspace: whole tiles
    if (!aligned(workspace, 16)) return set_error(kErrInvalid, "dense_gemm: workspace must be 16-byte aligned");
    p.splits = plan_dense(tiles, K / kBK);
    p.ws = static_cast<float*>(workspace);
  }
  hipLaunchKernelGGL(dense_gemm_kernel, dim3((unsigned)(tiles * p.splits)), dim3(256), 0, st, p);
  int rc = check_launch("dense_gemm_kernel");
  if (rc || p.splits == 1) return rc;
  hipLaunchKernelGGL(dense_reduce_kernel, dim3((unsigned)(tiles * (kTileF32 / 4 / 256))), dim3(256), 0, st, p);
  return check_launch("dense_reduce_kernel");
}

}  // namespace vqx
