// Block-scaled product with both operands decoded on the fly:
//   out[b, m, n] = sum_k A'[b, m, k] * B'[b, k, n]  (+ bias[n]),  bf16 out,
// where each operand X' is the decode linear_mx / matmul_mx apply before
// their dense product (src/voyager_compiler/ops/quantized.py:313-326 and
// :388-398): X' = bf16(code[trunc(X)] * scale[block of k]) with the code
// lookup and the scale each optional.  X holds bf16 values or integer-valued
// bf16 code indices; the scales are bf16, one per block of `bs` along K.
// This is the path of the converted models' operands that are not a
// 16-level weight with blocks of 64 (that one runs vqx_nf4_gemm.hip with a
// packed weight): int6 / nf4_6 attention operands coded on both sides, int8
// weights with blocks of 16, activations coded with input_code / input_scale.
//
// bf16 MFMA (v_mfma_f32_32x32x16_bf16), fp32 accumulation.  A workgroup of
// 256 threads computes a 128 x 128 tile; wave w owns the 64 x 64 block at
// rows 64 (w >> 1), columns 64 (w & 1).  The K loop steps by 64.  Each step
// the raw operand bytes of step s + 2 are loaded into registers (two register
// sets, so a load has two steps to land), those of step s + 1 are decoded and
// written to the other of two LDS stages, and the MFMAs of step s read their
// fragments from the current stage; one barrier per step.  Two workgroups fit
// a CU (72 KiB of LDS each), so one's decode runs under the other's MFMAs.
//  * K-major operands ([rows][K], A always): 16-byte loads, 8 lanes per
//    128-byte row; each 8-value chunk shares one scale (the block size is a
//    power of two >= 8).
//  * An N-major right operand ([K][N], matmul_mx's "ck" layout): each thread
//    loads 4 k rows x 8 columns, decodes them with the 8 columns' scales (one
//    16-byte load) and transposes them with v_perm into 8 column rows of 4 k,
//    written as 8-byte LDS stores.
//  * Code lookups: the decode of a pattern depends only on its sign and on
//    its magnitude clamped to [0x3F7F, 0x4381] (every |v| < 1 truncates to
//    index 0 like 0.996; |v| >= 258, Inf and NaN are outside any table of up
//    to 256 entries), so each workgroup tabulates 2 x 1027 decoded bf16 values
//    in LDS once and a lookup is a clamp and one 2-byte LDS read.  An index
//    outside the table (the reference raises IndexError) decodes to NaN.
// Tiles are numbered batch-major, then by row tile, then by column tile, and
// handed out so each XCD runs a contiguous range (whole row slabs of A, and
// for batched attention products whole heads, stay in its L2).
#include <type_traits>

#include "vqx_kernels.h"

namespace vqx {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kTK = 64;  // k per step
constexpr uint32_t kCodeLo = 0x3F7Fu, kCodeHi = 0x4381u;
constexpr int kCodeSpan = (int)(kCodeHi - kCodeLo) + 1;  // entries per sign
constexpr int kMaxCode = 256;

enum Dec : int { kPlain = 0, kScale = 1, kCode = 2, kCodeScale = 3 };

struct MxOpArgs {
  const uint16_t* data;
  const uint16_t* scale;
  const uint16_t* code;
  int64_t bstride, ld, sbstride, sld;
  int32_t code_len, bs_shift;  // block size = 1 << bs_shift
};

// byte offset of 16-byte chunk c (0..7) of row r in a [rows][64] bf16 tile;
// the slot is c ^ (r & 7) ^ ((r >> 3) & 7).  Fragment reads (16 aligned
// consecutive rows, one chunk) meet 16 distinct (row parity, slot) pairs and
// row-wise 16-byte writes 16 distinct pairs per 16 lanes, so both are
// conflict free; the N-major operand's 8-byte column writes meet at most two
// lanes per bank group.
__device__ __forceinline__ uint32_t swz(uint32_t r, uint32_t c) {
  return r * 128u + ((c ^ (r & 7u) ^ ((r >> 3) & 7u)) << 4);
}

__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Decoded bf16 value of code pattern h through the LDS table.
__device__ __forceinline__ uint32_t code_value(const uint16_t* tab, uint32_t h) {
  uint32_t a = h & 0x7FFFu;
  a = a < kCodeLo ? kCodeLo : (a > kCodeHi ? kCodeHi : a);
  return tab[a - kCodeLo + ((h >> 15) & 1u) * (uint32_t)kCodeSpan];
}

// The table: entry e of sign s is the decode of the bf16 pattern
// s << 15 | (kCodeLo + e), the reference's code[index.to(long)] (trunc
// toward zero, a negative index counting from the end).
template <int THREADS>
__device__ void build_code_table(uint16_t* tab, const uint16_t* code, int len) {
  for (int e = threadIdx.x; e < 2 * kCodeSpan; e += THREADS) {
    const uint32_t s = e >= kCodeSpan ? 1u : 0u;
    const uint32_t h = (s << 15) | (kCodeLo + (uint32_t)(e - (int)s * kCodeSpan));
    const float t = __builtin_truncf(u2f(h << 16));
    const bool ok = t >= -(float)len && t < (float)len;
    const int i = ok ? (int)t : 0;
    tab[e] = ok ? code[i < 0 ? i + len : i] : (uint16_t)0x7FC0u;
  }
}

// Decode one dword (two bf16 patterns, low half first) with scales s0 / s1.
template <int D>
__device__ __forceinline__ uint32_t decode2(uint32_t w, float s0, float s1, const uint16_t* tab) {
  if constexpr (D == kPlain) {
    return w;
  } else if constexpr (D == kScale) {
    return pack_bf16x2(u2f(w << 16) * s0, u2f(w & 0xFFFF0000u) * s1);
  } else {
    const uint32_t lo = code_value(tab, w & 0xFFFFu), hi = code_value(tab, w >> 16);
    if constexpr (D == kCode) return lo | (hi << 16);
    else return pack_bf16x2(u2f(lo << 16) * s0, u2f(hi << 16) * s1);
  }
}

__device__ __forceinline__ float bf_lo(uint32_t w) { return u2f(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return u2f(w & 0xFFFF0000u); }

// One operand's raw bytes of one step: up to four 16-byte chunks and their scales.
struct Raw {
  u32x4 v[4];
  u32x4 s;  // K-major: s[q] low half = scale of chunk q; N-major: the 8 columns' scales
  int in;   // k values of the chunks inside K (values past K must decode to zero)
};

// 16 bytes from a 2-byte aligned address (rows whose length is not a multiple
// of 8 values): one load instruction, which takes any alignment.
__device__ __forceinline__ u32x4 load16_any(const char* p) {
  u32x4 v;
  __builtin_memcpy(&v, __builtin_assume_aligned(p, 2), 16);
  return v;
}

// The values of v from element n (0..7) on, zeros behind them.
__device__ __forceinline__ u32x4 shift_down(u32x4 v, int n) {
  const uint64_t lo = v.x | ((uint64_t)v.y << 32), hi = v.z | ((uint64_t)v.w << 32);
  const int b = 16 * (n & 3);
  const uint64_t l = n & 4 ? hi : lo, h = n & 4 ? 0 : hi;
  const uint64_t rl = b ? (l >> b) | (h << (64 - b)) : l, rh = h >> b;
  return {(uint32_t)rl, (uint32_t)(rl >> 32), (uint32_t)rh, (uint32_t)(rh >> 32)};
}

// Mask of dword j (values 2 j, 2 j + 1) of a chunk with n valid values.
__device__ __forceinline__ uint32_t valid_mask(int n, int j) {
  return n >= 2 * j + 2 ? 0xFFFFFFFFu : (n == 2 * j + 1 ? 0xFFFFu : 0u);
}

// K-major staging of ROWS tile rows (A, or B stored [N][K]) by THREADS
// threads: chunk q of thread t is chunk t % 8 of tile row t / 8 + q THREADS / 8.
// Loads are never skipped (a branch around a load makes the compiler wait for
// every load in flight at the join): past the last row the last row is read,
// past K the last 8 values, and in a checked step the values past K are zeroed
// after the decode.  ANY: K and the row stride may be any (K >= 8), else both
// are multiples of 8 and rows 16-byte aligned.  Addresses are a uniform base (the batch item) plus 32-bit byte
// offsets; LDS addresses are precomputed.
template <int D, int ROWS, int THREADS, bool ANY>
struct KMajor {
  static constexpr int kCh = ROWS * 8 / THREADS;  // chunks per thread
  static_assert(kCh >= 1 && kCh <= 4, "chunks per thread");
  const char* base;   // data of the batch item
  const char* sbase;  // scales of the batch item
  uint32_t off[kCh];  // byte offset of the thread's chunk in step 0, per row
  uint32_t soff[kCh];
  uint32_t lds[kCh];  // LDS byte offset of the thread's chunks in a stage
  int sh;

  __device__ __forceinline__ void init(const MxOpArgs& o, int64_t b, int r0, int rows_valid) {
    const int t = threadIdx.x;
    base = reinterpret_cast<const char*>(o.data + b * o.bstride);
    if constexpr (D == kScale || D == kCodeScale) sbase = reinterpret_cast<const char*>(o.scale + b * o.sbstride);
#pragma unroll
    for (int q = 0; q < kCh; ++q) {
      int r = r0 + (t >> 3) + (THREADS / 8) * q;
      r = r < rows_valid ? r : rows_valid - 1;
      off[q] = 2u * ((uint32_t)r * (uint32_t)o.ld + (uint32_t)(t & 7) * 8u);
      if constexpr (D == kScale || D == kCodeScale) soff[q] = 2u * (uint32_t)r * (uint32_t)o.sld;
      lds[q] = swz((t >> 3) + (THREADS / 8) * q, t & 7);
    }
    sh = o.bs_shift;
  }
  template <bool CHECK>
  __device__ __forceinline__ void load(Raw& x, int ks, int K) {
    const int k = ks * kTK + (threadIdx.x & 7) * 8;
    int kl = k;
    x.in = 8;
    if constexpr (CHECK) {
      x.in = K - k;  // 8 or more: all; K % 8 == 0 without ANY: all or none
      kl = k < K - 8 ? k : K - 8;
    }
    const uint32_t kb = 2u * (uint32_t)(kl - (int)(threadIdx.x & 7) * 8);
    const int ksc = ANY && CHECK && k < K ? k : kl;  // a chunk wholly past K takes any scale
#pragma unroll
    for (int q = 0; q < kCh; ++q) {
      if constexpr (ANY) x.v[q] = load16_any(base + (off[q] + kb));
      else x.v[q] = *reinterpret_cast<const u32x4*>(base + (off[q] + kb));
      if constexpr (D == kScale || D == kCodeScale)
        x.s[q] = *reinterpret_cast<const uint16_t*>(sbase + (soff[q] + 2u * (uint32_t)(ksc >> sh)));
    }
  }
  // decode and write to the stage; in a checked step chunks past K are
  // written as zeros
  template <bool CHECK>
  __device__ __forceinline__ void store(const Raw& x, uint8_t* stage, const uint16_t* tab) {
#pragma unroll
    for (int q = 0; q < kCh; ++q) {
      const float s = bf_lo(x.s[q]);
      u32x4 d, v = x.v[q];
      if constexpr (ANY && CHECK) {
        if (x.in < 8) v = shift_down(v, (8 - x.in) & 7);  // loaded from K - 8 on
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        d[j] = decode2<D>(v[j], s, s, tab);
        if constexpr (CHECK) d[j] = ANY ? d[j] & valid_mask(x.in, j) : (x.in > 0 ? d[j] : 0u);
      }
      *reinterpret_cast<u32x4*>(stage + lds[q]) = d;
    }
  }
};

// N-major staging of COLS tile columns (B stored [K][N]): a 64-deep step is
// 16 blocks of 4 k rows by COLS / 8 blocks of 8 columns; thread t < 2 COLS
// loads block (k rows 4 (t / (COLS / 8)) .. +3, columns 8 (t % (COLS / 8))
// .. +7) (past N the last 8 columns, past K the last 4 rows, zeroed after the
// load in a checked step), decodes it with the 8 columns' scales and
// transposes it into 8 column rows of 4 k.
template <int D, int COLS, int THREADS>
struct NMajor {
  static constexpr int kOct = COLS / 8;  // column blocks per k-row block
  static_assert(2 * COLS <= THREADS, "one block per thread");
  const char* base;
  const char* sbase;
  uint32_t coff;   // byte offset of the thread's first column (clamped)
  uint32_t ldb;    // bytes between k rows
  uint32_t sldb;   // bytes between block rows of the scales
  int sh;

  __device__ __forceinline__ static bool active() { return 2 * COLS == THREADS || (int)threadIdx.x < 2 * COLS; }

  __device__ __forceinline__ void init(const MxOpArgs& o, int64_t b, int n0, int N) {
    const int t = threadIdx.x;
    int n = n0 + (t % kOct) * 8;
    n = n < N ? n : N - 8;
    base = reinterpret_cast<const char*>(o.data + b * o.bstride);
    if constexpr (D == kScale || D == kCodeScale) sbase = reinterpret_cast<const char*>(o.scale + b * o.sbstride);
    coff = 2u * (uint32_t)n;
    ldb = 2u * (uint32_t)o.ld;
    sldb = 2u * (uint32_t)o.sld;
    sh = o.bs_shift;
  }
  template <bool CHECK>
  __device__ __forceinline__ void load(Raw& x, int ks, int K) {
    if (!active()) return;
    int k = ks * kTK + ((int)threadIdx.x / kOct) * 4;
    x.in = 8;
    if constexpr (CHECK) {
      x.in = k < K ? 8 : 0;  // K % 8 == 0: the four rows are all in or all out
      k = x.in ? k : K - 4;
    }
    const uint32_t r0 = (uint32_t)k * ldb + coff;
#pragma unroll
    for (int i = 0; i < 4; ++i) x.v[i] = *reinterpret_cast<const u32x4*>(base + (r0 + (uint32_t)i * ldb));
    if constexpr (D == kScale || D == kCodeScale)
      x.s = *reinterpret_cast<const u32x4*>(sbase + ((uint32_t)(k >> sh) * sldb + coff));
  }
  template <bool CHECK>
  __device__ __forceinline__ void store(const Raw& x, uint8_t* stage, const uint16_t* tab) {
    if (!active()) return;
    const int t = threadIdx.x, o = t % kOct, kq = t / kOct;
    u32x4 d[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        d[i][j] = decode2<D>(x.v[i][j], bf_lo(x.s[j]), bf_hi(x.s[j]), tab);
        if constexpr (CHECK) d[i][j] = x.in ? d[i][j] : 0u;
      }
    // column 2 j takes the low halves of dword j of rows 0..3, column 2 j + 1
    // the high halves
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x2 ev = {__builtin_amdgcn_perm(d[1][j], d[0][j], 0x05040100u),
                        __builtin_amdgcn_perm(d[3][j], d[2][j], 0x05040100u)};
      const u32x2 od = {__builtin_amdgcn_perm(d[1][j], d[0][j], 0x07060302u),
                        __builtin_amdgcn_perm(d[3][j], d[2][j], 0x07060302u)};
      *reinterpret_cast<u32x2*>(stage + swz(8 * o + 2 * j, kq >> 1) + 8 * (kq & 1)) = ev;
      *reinterpret_cast<u32x2*>(stage + swz(8 * o + 2 * j + 1, kq >> 1) + 8 * (kq & 1)) = od;
    }
  }
};

// Output of one wave's (32 FM) x 64 block, staged through LDS: the wave
// writes its bf16 results (bias added) as rows of 144 bytes (64 values and
// 16 bytes of padding, which spreads a column of 32 rows over the banks)
// into its own region, then stores 8 whole 128-byte row segments per
// instruction (16 bytes a lane, non-temporal: the output is not read again
// by this kernel).  The accumulator layout has each lane hold 4 consecutive
// columns of 32 different rows, which would otherwise make every store
// instruction write 16-byte pieces of 32 rows.
constexpr int kOutRow = 144;  // bytes per staged row

template <int FM>
__device__ __forceinline__ void store_block(f32x16 (&acc)[FM][2], uint8_t* region, const uint16_t* __restrict__ bias,
                                            uint16_t* __restrict__ ob, int M, int N, int mrow0, int ncol0) {
  const int lane = threadIdx.x & 63, lr = lane & 31, lk = lane >> 5;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int c = j * 32 + 8 * g + 4 * lk;  // column within the block
      if (bias) {
        const int n = ncol0 + c < N ? ncol0 + c : N - 4;  // N % 4 == 0
        const u32x2 bb = *reinterpret_cast<const u32x2*>(bias + n);
#pragma unroll
        for (int i = 0; i < FM; ++i) {
          acc[i][j][4 * g] += bf_lo(bb.x);
          acc[i][j][4 * g + 1] += bf_hi(bb.x);
          acc[i][j][4 * g + 2] += bf_lo(bb.y);
          acc[i][j][4 * g + 3] += bf_hi(bb.y);
        }
      }
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const u32x2 o = {pack_bf16x2(acc[i][j][4 * g], acc[i][j][4 * g + 1]),
                         pack_bf16x2(acc[i][j][4 * g + 2], acc[i][j][4 * g + 3])};
        *reinterpret_cast<u32x2*>(region + (i * 32 + lr) * kOutRow + c * 2) = o;
      }
    }
  wave_lds_sync();
  const int c = (lane & 7) * 8, n = ncol0 + c;
#pragma unroll
  for (int q = 0; q < FM * 4; ++q) {
    const int r = q * 8 + (lane >> 3), m = mrow0 + r;
    const u32x4 v = *reinterpret_cast<const u32x4*>(region + r * kOutRow + c * 2);
    if (m >= M || n >= N) continue;
    uint16_t* dst = ob + (int64_t)m * N + n;
    if ((N & 7) == 0) {
      st_nt(reinterpret_cast<u32x4*>(dst), v);
    } else {  // rows are only 8-byte aligned; the last chunk may be half inside
      *reinterpret_cast<u32x2*>(dst) = u32x2{v.x, v.y};
      if (n + 4 < N) *reinterpret_cast<u32x2*>(dst + 4) = u32x2{v.z, v.w};
    }
  }
}

// Tile shapes: TM x TN outputs per workgroup of THREADS threads; the waves
// form a (TM / WROWS) x (TN / 64) grid, each owning WROWS x 64 outputs as
// (WROWS / 32) x 2 MFMA tiles of 32 x 32.
//   128 x 128, 256 threads: 64 x 64 per wave, two workgroups per CU;
//   256 x 128, 512 threads: 64 x 64 per wave, one workgroup per CU: three
//                           quarters of the 128 x 128 tile's decode per
//                           product.
// (256 x 256 with 128 x 64 per wave needs more than the 256 registers a wave
// has at two waves per SIMD: its accumulators alone take 128.)
template <int TM, int TN>
struct Shape {
  static constexpr int kThreads = (TM == 128 && TN == 128) ? 256 : 512;  // as in the launch bounds below
  static constexpr int kWavesN = TN / 64;
  static constexpr int kWavesM = kThreads / 64 / kWavesN;
  static constexpr int kWRows = TM / kWavesM;
  static constexpr int kFM = kWRows / 32;
  static constexpr int kStageA = TM * kTK * 2, kStageB = TN * kTK * 2;
};

template <int DA, int DB, bool BK, int TM, int TN, bool ANY>
__global__ __launch_bounds__((TM == 128 && TN == 128) ? 256 : 512, 2) void mx_gemm_kernel(
    MxOpArgs a, MxOpArgs b, const uint16_t* __restrict__ bias, uint16_t* __restrict__ out, int M, int N, int K, int tm,
    int tn, int ntiles) {
  using S = Shape<TM, TN>;
  constexpr int kThreads = S::kThreads, kFM = S::kFM, kStageA = S::kStageA, kStageB = S::kStageB;
  __shared__ __attribute__((aligned(16))) uint8_t lds[2 * (kStageA + kStageB)];
  static_assert(kThreads / 64 * kFM * 32 * kOutRow <= 2 * (kStageA + kStageB), "output staging fits the stages");
  uint8_t* const la = lds;
  uint8_t* const lb = lds + 2 * kStageA;
  __shared__ uint16_t ta[DA >= kCode ? 2 * kCodeSpan : 1];
  __shared__ uint16_t tb[DB >= kCode ? 2 * kCodeSpan : 1];

  const int bid = blockIdx.x;
  const int per_xcd = (ntiles + 7) / 8;
  const int tile = ntiles % 8 == 0 ? (bid & 7) * per_xcd + (bid >> 3) : bid;
  const int per_batch = tm * tn;
  const int64_t bi = tile / per_batch;
  const int rem = tile - (int)bi * per_batch;
  const int m0 = (rem / tn) * TM, n0 = (rem % tn) * TN;

  if constexpr (DA >= kCode) build_code_table<kThreads>(ta, a.code, a.code_len);
  if constexpr (DB >= kCode) build_code_table<kThreads>(tb, b.code, b.code_len);
  if constexpr (DA >= kCode || DB >= kCode) __syncthreads();

  KMajor<DA, TM, kThreads, ANY> sa;
  sa.init(a, bi, m0, M);
  typename std::conditional<BK, KMajor<DB, TN, kThreads, ANY>, NMajor<DB, TN, kThreads>>::type sb;
  sb.init(b, bi, n0, N);

  const int nk = (K + kTK - 1) / kTK;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave / S::kWavesN, wn = wave % S::kWavesN, lr = lane & 31, lk = lane >> 5;

  f32x16 acc[kFM][2];
#pragma unroll
  for (int i = 0; i < kFM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;

  auto compute = [&](uint32_t sta, uint32_t stb) {
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      bf16x8 fb[2];
#pragma unroll
      for (int j = 0; j < 2; ++j)
        fb[j] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(lb + stb + swz(wn * 64 + j * 32 + lr, kk * 2 + lk)));
#pragma unroll
      for (int i = 0; i < kFM; ++i) {
        const bf16x8 fa = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const u32x4*>(la + sta + swz(wm * S::kWRows + i * 32 + lr, kk * 2 + lk)));
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fb[j], fa, acc[i][j], 0, 0, 0);
      }
    }
  };

  // step s lives in registers ra/rb[s % 2] and in LDS stage s % 2
  Raw ra[2], rb[2];
  sa.template load<true>(ra[0], 0, K);
  sb.template load<true>(rb[0], 0, K);
  if (nk > 1) {
    sa.template load<true>(ra[1], 1, K);
    sb.template load<true>(rb[1], 1, K);
  }
  sa.template store<true>(ra[0], la, ta);
  sb.template store<true>(rb[0], lb, tb);
  if (nk > 2) {
    sa.template load<true>(ra[0], 2, K);
    sb.template load<true>(rb[0], 2, K);
  }
  lds_barrier();

  // FULL: ks + 3 < nk and step ks + 3 lies wholly inside K (so do the steps
  // before it), so the step stores and loads unconditionally and without
  // range checks: no branch in the steady state, and the compiler waits only
  // for the loads of the step it decodes, not for those issued after them
  auto step = [&](int ks, auto par, auto full) {
    constexpr int P = decltype(par)::value;  // ks % 2
    constexpr bool kFull = decltype(full)::value;
    compute(P * kStageA, P * kStageB);
    if (kFull || ks + 1 < nk) {
      sa.template store<!kFull>(ra[1 - P], la + (1 - P) * kStageA, ta);
      sb.template store<!kFull>(rb[1 - P], lb + (1 - P) * kStageB, tb);
    }
    lds_barrier();
    if (kFull || ks + 3 < nk) {
      sa.template load<!kFull>(ra[1 - P], ks + 3, K);
      sb.template load<!kFull>(rb[1 - P], ks + 3, K);
    }
  };
  const std::integral_constant<int, 0> p0;
  const std::integral_constant<int, 1> p1;
  const std::true_type all;
  const std::false_type checked;
  const int nfull = K / kTK;  // steps wholly inside K
  int ks = 0;
  for (; ks + 4 < nfull; ks += 2) {
    step(ks, p0, all);
    step(ks + 1, p1, all);
  }
  for (; ks < nk; ks += 2) {
    step(ks, p0, checked);
    if (ks + 1 < nk) step(ks + 1, p1, checked);
  }

  // every wave has passed the last step's barrier: the stages are free for
  // the output staging
  store_block<kFM>(acc, lds + wave * (kFM * 32 * kOutRow), bias, out + bi * (int64_t)M * N, M, N,
                   m0 + wm * S::kWRows, n0 + wn * 64);
}

// Decode passes: an operand that many output tiles read, decoded once into
// dense bf16 ahead of the product.  The code table in LDS has one entry per
// index from -len - 1 to len, the first and last (clamped to by everything
// outside, NaN too) decoding to NaN: built from 2 len + 2 reads, where the
// product kernel's table by bit pattern (2054 entries, fewer instructions per
// lookup) took most of the pass (333 x 11008 activations 8.0 us).
struct CodeLookup {
  const uint16_t* tab;
  float lo, hi;
  int off;
  __device__ __forceinline__ uint32_t operator()(uint32_t h) const {
    const float v = __builtin_fminf(__builtin_fmaxf(u2f(h << 16), lo), hi);
    return tab[(int)v + off];
  }
};

template <int D>
__device__ __forceinline__ CodeLookup make_lookup(uint16_t* tab, const MxOpArgs& o) {
  const int len = o.code_len;
  if constexpr (D >= kCode) {
    for (int e = threadIdx.x; e < 2 * len + 2; e += 256) {
      const int i = e - len - 1;
      tab[e] = i >= -len && i < len ? o.code[i < 0 ? i + len : i] : (uint16_t)0x7FC0u;
    }
    __syncthreads();
  }
  return {tab, -(float)(len + 1), (float)len, len + 1};
}

template <int D>
__device__ __forceinline__ uint32_t decode_pair(uint32_t w, float s0, float s1, const CodeLookup& lk) {
  if constexpr (D == kPlain) {
    return w;
  } else if constexpr (D == kScale) {
    return pack_bf16x2(bf_lo(w) * s0, bf_hi(w) * s1);
  } else {
    const uint32_t lo = lk(w & 0xFFFFu), hi = lk(w >> 16);
    if constexpr (D == kCode) return lo | (hi << 16);
    else return pack_bf16x2(u2f(lo << 16) * s0, u2f(hi << 16) * s1);
  }
}

typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));

// Up to n values from p, zeros behind them.
__device__ __forceinline__ u32x4 load8(const uint16_t* p, int n) {
  if (n >= 8) return load16_any(reinterpret_cast<const char*>(p));
  u32x4 v = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < 8; ++e)
    if (e < n) v[e >> 1] |= (uint32_t)p[e] << (16 * (e & 1));
  return v;
}

// Decode in the operand's own layout.  Item b of the operand is [R][C] (row
// stride o.ld, any alignment), out is [items][R][CP] contiguous with CP >= C
// a multiple of 8, zeros past C; KMAJ: C = K, blocks along C; else R = K,
// blocks along R.  Each thread decodes 8 consecutive values of a row per
// iteration.  NT: non-temporal loads and stores, for the product that decodes
// its other operand itself (P V of 2048 tokens 92 -> 85 us: P streams past
// the decoded V); the dense product finds plainly stored operands in the
// caches (scores of 2048 tokens 110 -> 90 us, 1000 x 4096 x 4096 41 -> 35).
template <int D, bool KMAJ, bool NT>
__global__ __launch_bounds__(256) void mx_decode_kernel(MxOpArgs o, uint16_t* __restrict__ out, int R, int C, int CP,
                                                        uint32_t chunks) {
  __shared__ uint16_t tab[D >= kCode ? 2 * kMaxCode + 2 : 1];
  const CodeLookup lk = make_lookup<D>(tab, o);
  const uint32_t cpr = (uint32_t)CP / 8u;
  for (uint32_t i = blockIdx.x * 256u + threadIdx.x; i < chunks; i += gridDim.x * 256u) {
    const uint32_t row = i / cpr;  // over all items
    const int c = (int)(i - row * cpr) * 8;
    const uint32_t bi = row / (uint32_t)R;
    const int r = (int)(row - bi * (uint32_t)R);
    const int n = C - c;  // values of the chunk inside the row
    u32x4 d = {0u, 0u, 0u, 0u};
    if (n > 0) {
      const uint16_t* src = o.data + (int64_t)bi * o.bstride + (int64_t)r * o.ld + c;
      const u32x4 v =
          NT && n >= 8 ? __builtin_nontemporal_load(reinterpret_cast<const u32x4_any*>(src)) : load8(src, n);
      u32x4 sc = {0u, 0u, 0u, 0u};
      float s = 1.0f;
      if constexpr (D == kScale || D == kCodeScale) {
        const uint16_t* sp = o.scale + (int64_t)bi * o.sbstride;
        if constexpr (KMAJ) s = bf_lo(sp[(int64_t)r * o.sld + (c >> o.bs_shift)]);
        else sc = load8(sp + (int64_t)(r >> o.bs_shift) * o.sld + c, n);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        d[j] = decode_pair<D>(v[j], KMAJ ? s : bf_lo(sc[j]), KMAJ ? s : bf_hi(sc[j]), lk) & valid_mask(n, j);
    }
    u32x4* const dst = reinterpret_cast<u32x4*>(out + (int64_t)row * CP + c);
    if constexpr (NT) st_nt(dst, d);
    else *dst = d;
  }
}

// Decode with a transpose: item b of the operand is [R][C] (row stride o.ld,
// any alignment), out is [items][C][RP] contiguous with RP >= R, zeros past R.
// SROW: the scales' blocks run along R (an N-major operand: R = K), one scale
// row per block; else along C (a K-major weight laid out by rows of K).  A
// workgroup turns a 64 x 64 tile: a thread loads 8 columns of two rows, pairs
// them by column and writes 8 dwords to LDS (row c of the tile holds 64 r in
// eight 16-byte slots, slot s at s ^ (c >> 3): at most two lanes a bank), then
// four threads write each column's 128 bytes.
template <int D, bool SROW>
__global__ __launch_bounds__(256) void mx_turn_kernel(MxOpArgs o, uint16_t* __restrict__ out, int R, int C, int RP,
                                                      int tr, int tc) {
  __shared__ uint16_t tab[D >= kCode ? 2 * kMaxCode + 2 : 1];
  __shared__ __attribute__((aligned(16))) uint32_t tile[64 * 32];
  const CodeLookup lk = make_lookup<D>(tab, o);
  const int b = blockIdx.x / (tr * tc), rem = blockIdx.x - b * (tr * tc);
  const int r0 = rem / tc * 64, c0 = rem % tc * 64;
  const uint16_t* data = o.data + (int64_t)b * o.bstride;
  const uint16_t* scale = nullptr;
  if constexpr (D == kScale || D == kCodeScale) scale = o.scale + (int64_t)b * o.sbstride;
  const int rp = threadIdx.x >> 3, cc = (threadIdx.x & 7) * 8;  // row pair, first column in the tile
  const int n = C - (c0 + cc);
  u32x4 d[2];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int r = r0 + 2 * rp + h;
    d[h] = u32x4{0u, 0u, 0u, 0u};
    if (r < R && n > 0) {
      const u32x4 v = load8(data + (int64_t)r * o.ld + c0 + cc, n);
      u32x4 sc = {0u, 0u, 0u, 0u};
      float s = 1.0f;
      if constexpr (D == kScale || D == kCodeScale) {
        if constexpr (SROW) sc = load8(scale + (int64_t)(r >> o.bs_shift) * o.sld + c0 + cc, n);
        else s = bf_lo(scale[(int64_t)r * o.sld + ((c0 + cc) >> o.bs_shift)]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) d[h][j] = decode_pair<D>(v[j], SROW ? bf_lo(sc[j]) : s, SROW ? bf_hi(sc[j]) : s, lk);
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    uint32_t* t = tile + (cc + 2 * j) * 32 + ((((uint32_t)rp >> 2) ^ ((uint32_t)cc >> 3)) << 2) + (rp & 3);
    t[0] = __builtin_amdgcn_perm(d[1][j], d[0][j], 0x05040100u);
    t[32] = __builtin_amdgcn_perm(d[1][j], d[0][j], 0x07060302u);
  }
  __syncthreads();
  const int c = threadIdx.x >> 2;
  if (c0 + c >= C) return;
  uint16_t* orow = out + ((int64_t)b * C + c0 + c) * RP;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int s = (threadIdx.x & 3) * 2 + h, r = r0 + s * 8;
    const u32x4 v = *reinterpret_cast<const u32x4*>(tile + c * 32 + ((s ^ (c >> 3)) << 2));
    if (r + 8 <= RP) {
      __builtin_memcpy(__builtin_assume_aligned(orow + r, 2), &v, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (r + e < RP) orow[r + e] = (uint16_t)(v[e >> 1] >> (16 * (e & 1)));
    }
  }
}

// Products of few rows with an N-major right operand (a decode step's
// attention: one query row against the K^T or V cache, [K][N] as quantize_mx
// writes it), both decoded on the fly.  Bound by the one read of the right
// operand and, per CU, by its decode (about 4 VALU per value): a workgroup of
// 256 threads owns 8 LN columns of an item; its 256 / LN groups of LN lanes
// each take a run of consecutive k rows, a lane 8 columns (one 16-byte load
// per row, eight rows in flight; the scales are loaded when the block
// changes).  LN = 8 reads whole 128-byte lines of a k row; LN = 2, for
// products whose columns would leave CUs idle (P V: 128 columns an item),
// spreads an item over more workgroups, placed on one XCD, whose L2 serves the
// rest of each line.  The groups' fp32 sums are added across the lanes, then
// the waves, in a fixed order; nothing is split over workgroups.
// Measured, 32 x [1, 128] x [128, 1999] and 32 x [1, 1999] x [1999, 128]:
// 10.5 + 11 us (16 MB each); turning the cache and running the dense product
// took 21 + 27, one workgroup of 1024 threads per 64 columns 14.5 + 16.7.
constexpr int kGemvA = 16384;  // decoded left values a workgroup can hold

template <int CTRL>
__device__ __forceinline__ float add_dpp(float v) {
  return v + u2f((uint32_t)__builtin_amdgcn_update_dpp(0, (int)f2u(v), CTRL, 0xF, 0xF, false));
}

// Sum of v over the lanes that hold the same columns (lane % LN), everywhere.
template <int LN>
__device__ __forceinline__ float add_groups(float v) {
#if defined(__HIP_DEVICE_COMPILE__)
  v = add_dpp<0x128>(v);  // row_ror:8
  if constexpr (LN == 2) {
    v = add_dpp<0x124>(v);  // row_ror:4
    v = add_dpp<0x4E>(v);   // quad_perm: lane ^ 2
  }
  auto s = __builtin_amdgcn_permlane16_swap(f2u(v), f2u(v), false, false);
  v = u2f(s[0]) + u2f(s[1]);
  s = __builtin_amdgcn_permlane32_swap(f2u(v), f2u(v), false, false);
  v = u2f(s[0]) + u2f(s[1]);
#endif
  return v;
}

template <int DB, int MR, int LN>
__global__ __launch_bounds__(256) void mx_gemv_kernel(MxOpArgs a, MxOpArgs b, uint16_t* __restrict__ out, int M, int N,
                                                      int K, int tn, int batch) {
  constexpr int kGroups = 256 / LN, kCols = 8 * LN;
  __shared__ uint16_t tab[2 * kMaxCode + 2];
  __shared__ uint16_t as[kGemvA];
  __shared__ float part[MR][4][kCols];
  // an item's tiles on one XCD (workgroups go to the eight in turn)
  const int j8 = blockIdx.x >> 3;
  const bool turn = (batch & 7) == 0;
  const int64_t bi = turn ? (j8 / tn) * 8 + (blockIdx.x & 7) : blockIdx.x / tn;
  const int n0 = (turn ? j8 % tn : blockIdx.x % tn) * kCols;

  const int kg = threadIdx.x / LN, c = n0 + (threadIdx.x % LN) * 8, nv = N - c;
  const int run = (K + kGroups - 1) / kGroups;
  int k = kg * run;
  const int kend = k + run < K ? k + run : K;
  const uint16_t* bd = b.data + bi * b.bstride + c;
  const uint16_t* sp = b.scale ? b.scale + bi * b.sbstride + c : nullptr;
  u32x4 v[8];  // the first rows are under way while the left rows are decoded
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = k + i < kend ? load8(bd + (int64_t)(k + i) * b.ld, nv) : u32x4{0u, 0u, 0u, 0u};

  u32x4 sc = {0u, 0u, 0u, 0u};
  int blk = -1;
  if constexpr (DB == kScale || DB == kCodeScale) {
    if (k < kend) {
      blk = k >> b.bs_shift;
      sc = load8(sp + (int64_t)blk * b.sld, nv);
    }
  }

  // the left rows, decoded as the reference's operand: bf16 values
  const uint16_t* asc = a.scale ? a.scale + bi * a.sbstride : nullptr;
  for (int m = 0; m < M; ++m)
    for (int i = threadIdx.x * 8; i < K; i += 256 * 8) {
      const u32x4 w = load8(a.data + bi * a.bstride + (int64_t)m * a.ld + i, K - i);
      const float s = asc ? bf2f(asc[(int64_t)m * a.sld + (i >> a.bs_shift)]) : 1.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        if (i + e >= K) break;
        float x = bf2f((w[e >> 1] >> (16 * (e & 1))) & 0xFFFFu);
        if (a.code) {
          const float t = __builtin_truncf(x);
          const bool ok = t >= -(float)a.code_len && t < (float)a.code_len;
          const int j = ok ? (int)t : 0;
          x = ok ? bf2f(a.code[j < 0 ? j + a.code_len : j]) : __builtin_nanf("");
        }
        as[m * K + i + e] = (uint16_t)f2bf(x * s);  // without scales: x * 1
      }
    }
  const int len = b.code_len;
  if constexpr (DB >= kCode) {
    for (int e = threadIdx.x; e < 2 * len + 2; e += 256) {
      const int i = e - len - 1;
      tab[e] = i >= -len && i < len ? b.code[i < 0 ? i + len : i] : (uint16_t)0x7FC0u;
    }
  }
  __syncthreads();
  const CodeLookup lk{tab, -(float)(len + 1), (float)len, len + 1};
  float acc[MR][8];
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[m][e] = 0.0f;
  while (k < kend) {
    u32x4 nx[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      nx[i] = k + 8 + i < kend ? load8(bd + (int64_t)(k + 8 + i) * b.ld, nv) : u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (k + i >= kend) break;
      if constexpr (DB == kScale || DB == kCodeScale) {
        if (((k + i) >> b.bs_shift) != blk) {
          blk = (k + i) >> b.bs_shift;
          sc = load8(sp + (int64_t)blk * b.sld, nv);
        }
      }
      float x[MR];
#pragma unroll
      for (int m = 0; m < MR; ++m) x[m] = m < M ? bf2f(as[m * K + k + i]) : 0.0f;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t d = decode_pair<DB>(v[i][j], bf_lo(sc[j]), bf_hi(sc[j]), lk);
#pragma unroll
        for (int m = 0; m < MR; ++m) {
          acc[m][2 * j] += x[m] * bf_lo(d);
          acc[m][2 * j + 1] += x[m] * bf_hi(d);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = nx[i];
    k += 8;
  }
#pragma unroll
  for (int m = 0; m < MR; ++m)
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const float t = add_groups<LN>(acc[m][e]);
      if ((threadIdx.x & 63) < LN) part[m][threadIdx.x >> 6][(threadIdx.x % LN) * 8 + e] = t;
    }
  __syncthreads();
  for (int i = threadIdx.x; i < M * kCols; i += 256) {
    const int m = i / kCols, col = i % kCols;
    const float t = (part[m][0][col] + part[m][1][col]) + (part[m][2][col] + part[m][3][col]);
    if (n0 + col < N) out[((int64_t)bi * M + m) * N + n0 + col] = (uint16_t)f2bf(t);
  }
}

template <int DA, int DB, bool BK, int TM, int TN, bool ANY = false>
int launch_one(const MxOpArgs& a, const MxOpArgs& b, const uint16_t* bias, uint16_t* out, int M, int N, int K,
               int batch, hipStream_t stream) {
  const int tm = (M + TM - 1) / TM, tn = (N + TN - 1) / TN;
  const int64_t ntiles = (int64_t)batch * tm * tn;
  if (ntiles > INT32_MAX) return set_error(kErrInvalid, "mx_gemm: too many tiles");
  hipLaunchKernelGGL((mx_gemm_kernel<DA, DB, BK, TM, TN, ANY>), dim3((unsigned)ntiles), dim3(Shape<TM, TN>::kThreads), 0,
                     stream, a, b, bias, out, M, N, K, tm, tn, (int)ntiles);
  return check_launch("mx_gemm_kernel");
}

// The tile, from measurement (LLaMA-7B shapes on one MI355X): 256 x 128
// for products with N > 128 and K > 128 that still give every CU a tile
// (2048 x 11008 x 4096: 253 against 282 us), else 128 x 128 (two
// workgroups per CU: the attention products, K = 128 or N = 128, run 9% and
// 6% faster on it).
enum TileKind : int { kT128 = 0, kT256x128 = 1 };

int pick_tile(int64_t batch, int64_t M, int64_t N, int64_t K) {
  if (N <= 128 || K <= 128) return kT128;
  const int64_t tiles = batch * ((M + 255) / 256) * ((N + 127) / 128);
  return tiles >= num_cus() ? kT256x128 : kT128;
}

template <int DA, int DB, bool BK>
int launch_tile(int tile, const MxOpArgs& a, const MxOpArgs& b, const uint16_t* bias, uint16_t* out, int M, int N,
                int K, int batch, hipStream_t stream) {
  if (tile == kT256x128) return launch_one<DA, DB, BK, 256, 128>(a, b, bias, out, M, N, K, batch, stream);
  return launch_one<DA, DB, BK, 128, 128>(a, b, bias, out, M, N, K, batch, stream);
}

template <int DA, int DB>
int launch_layout(bool bk, int tile, const MxOpArgs& a, const MxOpArgs& b, const uint16_t* bias, uint16_t* out, int M,
                  int N, int K, int batch, hipStream_t stream) {
  return bk ? launch_tile<DA, DB, true>(tile, a, b, bias, out, M, N, K, batch, stream)
            : launch_tile<DA, DB, false>(tile, a, b, bias, out, M, N, K, batch, stream);
}

template <int DA>
int launch_b(int db, bool bk, int tile, const MxOpArgs& a, const MxOpArgs& b, const uint16_t* bias, uint16_t* out,
             int M, int N, int K, int batch, hipStream_t stream) {
  switch (db) {
    case kPlain: return launch_layout<DA, kPlain>(bk, tile, a, b, bias, out, M, N, K, batch, stream);
    case kScale: return launch_layout<DA, kScale>(bk, tile, a, b, bias, out, M, N, K, batch, stream);
    case kCode: return launch_layout<DA, kCode>(bk, tile, a, b, bias, out, M, N, K, batch, stream);
    default: return launch_layout<DA, kCodeScale>(bk, tile, a, b, bias, out, M, N, K, batch, stream);
  }
}

int dec_of(const MxOperand& o) { return (o.code ? kCode : kPlain) | (o.scale ? kScale : kPlain); }

// The kernels address each matrix (and its scales) of a batch item with
// 32-bit byte offsets from the item's base.
constexpr int64_t kMaxItemBytes = (int64_t)1 << 32;

// any: the operand may have any alignment and strides (else 16-byte aligned
// data, strides and N-major scales, as the N-major staging reads them).
int check_operand(const MxOperand& o, const char* name, bool k_major_only, int64_t K, int64_t cols, bool any = false) {
  if (!o.data || !aligned(o.data, any ? 2 : 16))
    return set_error(kErrInvalid, "%s: data must be a 16-byte aligned pointer", name);
  if (k_major_only && !o.k_major) return set_error(kErrInvalid, "%s: the left operand is K-major ([M][K])", name);
  const int64_t need = o.k_major ? K : cols;
  if (o.ld < need || (!any && o.ld % 8)) return set_error(kErrInvalid, "%s: ld %lld must be >= %lld and a multiple of 8", name,
                                                          (long long)o.ld, (long long)need);
  if (o.batch_stride < 0 || (!any && o.batch_stride % 8))
    return set_error(kErrInvalid, "%s: batch_stride must be >= 0 and a multiple of 8", name);
  const int64_t span = o.k_major ? (cols - 1) * o.ld + K : (K - 1) * o.ld + cols;
  if (2 * span >= kMaxItemBytes)
    return set_error(kErrInvalid, "%s: one batch item spans more than 4 GiB", name);
  if (o.code && (o.code_len < 1 || o.code_len > kMaxCode))
    return set_error(kErrInvalid, "%s: code_len %d outside 1..%d", name, (int)o.code_len, kMaxCode);
  if (o.scale) {
    if (o.block_size < 8 || (o.block_size & (o.block_size - 1)))
      return set_error(kErrInvalid, "%s: block_size %d must be a power of two >= 8", name, (int)o.block_size);
    const int64_t nkb = (K + o.block_size - 1) / o.block_size;
    if (o.scale_batch_stride < 0) return set_error(kErrInvalid, "%s: scale_batch_stride must be >= 0", name);
    const int64_t sspan = o.k_major ? (cols - 1) * o.scale_ld + nkb : (nkb - 1) * o.scale_ld + cols;
    if (2 * sspan >= kMaxItemBytes)
      return set_error(kErrInvalid, "%s: one batch item's scales span more than 4 GiB", name);
    if (o.k_major) {
      if (o.scale_ld < nkb) return set_error(kErrInvalid, "%s: scale_ld must be >= %lld", name, (long long)nkb);
    } else {
      if (o.scale_ld < cols ||
          (!any && (!aligned(o.scale, 16) || o.scale_ld % 8 || o.scale_batch_stride % 8)))
        return set_error(kErrInvalid,
                         "%s: N-major scales need a 16-byte aligned pointer, scale_ld >= %lld and strides that are "
                         "multiples of 8",
                         name, (long long)cols);
    }
  }
  return kOk;
}

MxOpArgs args_of(const MxOperand& o) {
  MxOpArgs r;
  r.data = static_cast<const uint16_t*>(o.data);
  r.scale = static_cast<const uint16_t*>(o.scale);
  r.code = static_cast<const uint16_t*>(o.code);
  r.bstride = o.batch_stride;
  r.ld = o.ld;
  r.sbstride = o.scale_batch_stride;
  r.sld = o.scale_ld;
  r.code_len = o.code ? o.code_len : 0;
  r.bs_shift = o.scale ? __builtin_ctz((unsigned)o.block_size) : 0;
  return r;
}

}  // namespace

int mx_gemm(const MxOperand& a, const MxOperand& b, const uint16_t* bias, uint16_t* out, int64_t batch, int64_t M,
            int64_t N, int64_t K, bool any, hipStream_t stream) {
  if (batch < 1 || M < 1 || N < 1 || K < 1) return set_error(kErrInvalid, "mx_gemm: empty product");
  if (!any && K % 8) return set_error(kErrInvalid, "mx_gemm: K (%lld) must be a multiple of 8", (long long)K);
  if (any && (K < 8 || !b.k_major)) return set_error(kErrInvalid, "mx_gemm: K-major operands with K >= 8 needed");
  if (N % 4) return set_error(kErrInvalid, "mx_gemm: N (%lld) must be a multiple of 4", (long long)N);
  if (!b.k_major && N % 8) return set_error(kErrInvalid, "mx_gemm: an N-major right operand needs N %% 8 == 0");
  if (M > INT32_MAX || N > INT32_MAX || K > INT32_MAX) return set_error(kErrInvalid, "mx_gemm: dimension too large");
  int rc = check_operand(a, "mx_gemm A", true, K, M, any);
  if (rc) return rc;
  rc = check_operand(b, "mx_gemm B", false, K, N, any);
  if (rc) return rc;
  if (!out || !aligned(out, 8)) return set_error(kErrInvalid, "mx_gemm: out must be 8-byte aligned");
  if (bias && !aligned(bias, 8)) return set_error(kErrInvalid, "mx_gemm: bias must be 8-byte aligned");
  if (batch > INT32_MAX) return set_error(kErrInvalid, "mx_gemm: batch too large");
  // nothing to decode and K contiguous on both sides: the dense product (from
  // four of its 64-deep steps; below that its pipeline does not fill)
  if (!any && dec_of(a) == kPlain && dec_of(b) == kPlain && b.k_major && K >= 256 && dense_gemm_takes(batch, M, N, K))
    return dense_gemm(static_cast<const uint16_t*>(a.data), a.ld, a.batch_stride, static_cast<const uint16_t*>(b.data),
                      b.ld, b.batch_stride, bias, out, batch, M, N, K, nullptr, 0, stream);
  const MxOpArgs aa = args_of(a), bb = args_of(b);
  const int db = dec_of(b);
  if (any) {
    if (db != kPlain) return set_error(kErrInvalid, "mx_gemm: a plain right operand needed for operands of any K");
    switch (dec_of(a)) {
      case kPlain: return launch_one<kPlain, kPlain, true, 128, 128, true>(aa, bb, bias, out, (int)M, (int)N, (int)K, (int)batch, stream);
      case kScale: return launch_one<kScale, kPlain, true, 128, 128, true>(aa, bb, bias, out, (int)M, (int)N, (int)K, (int)batch, stream);
      case kCode: return launch_one<kCode, kPlain, true, 128, 128, true>(aa, bb, bias, out, (int)M, (int)N, (int)K, (int)batch, stream);
      default: return launch_one<kCodeScale, kPlain, true, 128, 128, true>(aa, bb, bias, out, (int)M, (int)N, (int)K, (int)batch, stream);
    }
  }
  const bool bk = b.k_major != 0;
  const int tile = pick_tile(batch, M, N, K);
  const int iM = (int)M, iN = (int)N, iK = (int)K, ib = (int)batch;
  switch (dec_of(a)) {
    case kPlain: return launch_b<kPlain>(db, bk, tile, aa, bb, bias, out, iM, iN, iK, ib, stream);
    case kScale: return launch_b<kScale>(db, bk, tile, aa, bb, bias, out, iM, iN, iK, ib, stream);
    case kCode: return launch_b<kCode>(db, bk, tile, aa, bb, bias, out, iM, iN, iK, ib, stream);
    default: return launch_b<kCodeScale>(db, bk, tile, aa, bb, bias, out, iM, iN, iK, ib, stream);
  }
}

template <int D, bool NT>
int launch_decode_nt(bool kmaj, const MxOpArgs& o, uint16_t* out, int R, int C, int CP, uint32_t chunks,
                     hipStream_t stream) {
  const dim3 grid(grid_for(chunks, 256, 8)), block(256);
  if (kmaj) hipLaunchKernelGGL((mx_decode_kernel<D, true, NT>), grid, block, 0, stream, o, out, R, C, CP, chunks);
  else hipLaunchKernelGGL((mx_decode_kernel<D, false, NT>), grid, block, 0, stream, o, out, R, C, CP, chunks);
  return check_launch("mx_decode_kernel");
}

template <int D>
int launch_decode(bool kmaj, bool nt, const MxOpArgs& o, uint16_t* out, int R, int C, int CP, uint32_t chunks,
                  hipStream_t stream) {
  return nt ? launch_decode_nt<D, true>(kmaj, o, out, R, C, CP, chunks, stream)
            : launch_decode_nt<D, false>(kmaj, o, out, R, C, CP, chunks, stream);
}

template <int D>
int launch_turn(bool srow, const MxOpArgs& o, uint16_t* out, int R, int C, int RP, int64_t batch, hipStream_t stream) {
  const int tr = (RP + 63) / 64, tc = (C + 63) / 64;
  const dim3 grid((unsigned)(batch * tr * tc));
  if (srow) hipLaunchKernelGGL((mx_turn_kernel<D, true>), grid, dim3(256), 0, stream, o, out, R, C, RP, tr, tc);
  else hipLaunchKernelGGL((mx_turn_kernel<D, false>), grid, dim3(256), 0, stream, o, out, R, C, RP, tr, tc);
  return check_launch("mx_turn_kernel");
}

// x decoded into dense bf16: in its own layout (turn 0, rows padded with zeros
// to out_ld, a multiple of 8), or with its two dims swapped (turn 1).
int mx_decode(const MxOperand& x, int64_t batch, int64_t rows, int64_t K, uint16_t* out, int64_t out_ld, bool turn,
              bool nt, bool any, hipStream_t stream) {
  if (batch < 1 || rows < 1 || K < 1) return set_error(kErrInvalid, "mx_decode: empty operand");
  int rc = check_operand(x, "mx_decode", false, K, rows, any);
  if (rc) return rc;
  const int64_t R = x.k_major ? rows : K, C = x.k_major ? K : rows, ol = turn ? R : C;
  if (!out || !aligned(out, 16)) return set_error(kErrInvalid, "mx_decode: out must be 16-byte aligned");
  if (out_ld < ol || (!turn && out_ld % 8))
    return set_error(kErrInvalid, "mx_decode: out_ld %lld for rows of %lld", (long long)out_ld, (long long)ol);
  if (R > INT32_MAX || C > INT32_MAX || out_ld > INT32_MAX - 64 || batch * R > INT32_MAX)
    return set_error(kErrInvalid, "mx_decode: operand too large");
  const MxOpArgs o = args_of(x);
  const int d = dec_of(x), iR = (int)R, iC = (int)C, il = (int)out_ld;
  const bool km = x.k_major != 0;
  if (turn) {
    if (batch * ((out_ld + 63) / 64) * ((C + 63) / 64) > INT32_MAX)
      return set_error(kErrInvalid, "mx_decode: operand too large");
    switch (d) {
      case kPlain: return launch_turn<kPlain>(!km, o, out, iR, iC, il, batch, stream);
      case kScale: return launch_turn<kScale>(!km, o, out, iR, iC, il, batch, stream);
      case kCode: return launch_turn<kCode>(!km, o, out, iR, iC, il, batch, stream);
      default: return launch_turn<kCodeScale>(!km, o, out, iR, iC, il, batch, stream);
    }
  }
  const int64_t chunks = batch * R * (out_ld / 8);
  if (chunks > INT32_MAX) return set_error(kErrInvalid, "mx_decode: operand too large");
  switch (d) {
    case kPlain: return launch_decode<kPlain>(km, nt, o, out, iR, iC, il, (uint32_t)chunks, stream);
    case kScale: return launch_decode<kScale>(km, nt, o, out, iR, iC, il, (uint32_t)chunks, stream);
    case kCode: return launch_decode<kCode>(km, nt, o, out, iR, iC, il, (uint32_t)chunks, stream);
    default: return launch_decode<kCodeScale>(km, nt, o, out, iR, iC, il, (uint32_t)chunks, stream);
  }
}

template <int DB, int MR>
int launch_gemv(const MxOpArgs& a, const MxOpArgs& b, uint16_t* out, int64_t batch, int M, int N, int K,
                hipStream_t stream) {
  // whole lines of a k row when that gives every CU a workgroup
  if (batch * ((N + 63) / 64) >= num_cus()) {
    const int tn = (N + 63) / 64;
    hipLaunchKernelGGL((mx_gemv_kernel<DB, MR, 8>), dim3((unsigned)(batch * tn)), dim3(256), 0, stream, a, b, out, M, N,
                       K, tn, (int)batch);
  } else {
    const int tn = (N + 15) / 16;
    hipLaunchKernelGGL((mx_gemv_kernel<DB, MR, 2>), dim3((unsigned)(batch * tn)), dim3(256), 0, stream, a, b, out, M, N,
                       K, tn, (int)batch);
  }
  return check_launch("mx_gemv_kernel");
}

int mx_gemv(const MxOperand& a, const MxOperand& b, uint16_t* out, int64_t batch, int64_t M, int64_t N, int64_t K,
            hipStream_t stream) {
  if (batch < 1 || M < 1 || N < 1 || K < 1) return set_error(kErrInvalid, "mx_gemv: empty product");
  if (M > 4 || M * K > kGemvA)
    return set_error(kErrInvalid, "mx_gemv: at most 4 rows and %d left values", kGemvA);
  if (b.k_major) return set_error(kErrInvalid, "mx_gemv: the right operand is N-major ([K][N])");
  int rc = check_operand(a, "mx_gemv A", true, K, M, true);
  if (rc) return rc;
  rc = check_operand(b, "mx_gemv B", false, K, N, true);
  if (rc) return rc;
  if (!out || !aligned(out, 2)) return set_error(kErrInvalid, "mx_gemv: null or misaligned out");
  if (N > INT32_MAX - 64 || batch * ((N + 15) / 16) > INT32_MAX)
    return set_error(kErrInvalid, "mx_gemv: dimension too large");
  const MxOpArgs aa = args_of(a), bb = args_of(b);
  const int iM = (int)M, iN = (int)N, iK = (int)K;
  switch (dec_of(b)) {
#define VQX_GEMV(D)                                                                        \
  return M == 1 ? launch_gemv<D, 1>(aa, bb, out, batch, iM, iN, iK, stream)                \
                : launch_gemv<D, 4>(aa, bb, out, batch, iM, iN, iK, stream);
    case kPlain: VQX_GEMV(kPlain)
    case kScale: VQX_GEMV(kScale)
    case kCode: VQX_GEMV(kCode)
    default: VQX_GEMV(kCodeScale)
#undef VQX_GEMV
  }
}

}  // namespace vqx
