// BF16 GEMM tiles on v_mfma_f32_32x32x16_bf16 (FP32 accumulate) for the
// learned per-element smoother: forward layers, backward data and weight
// gradients, split-K partial sums, column sums and the Adam step. No
// reference counterpart (the reference has no learned components).
//
// Operand layout of v_mfma_f32_32x32x16_bf16 (C[32x32] += A[32x16] B[16x32],
// wave64): lane l supplies eight A values of row l%32 and eight B values of
// column l%32, the K slice 8*(l/32)..8*(l/32)+7; it holds
// c[r] = C[8*(r/4) + 4*(l/32) + r%4][l%32]. A and B take the same K slice per
// lane, so the product does not depend on how the hardware orders K inside it.
//
// Tiles: 128x128 per workgroup of four wavefronts (2x2, 64x64 each = 2x2
// MFMA blocks), BK = 64, two LDS buffers with register prefetch of the next
// K tile, two workgroups per CU (the layers have 512 to 1024 tiles).
// What bounds it: the LDS reads of a K tile take as long as its MFMAs, and with
// two workgroups per CU little covers a tile's first loads and its epilogue.
//
// Operands reach LDS as [row][k] (row stride BK + 8 entries) whatever their
// layout in HBM: a K-contiguous operand is copied with 16-byte loads and
// stores; of a row-contiguous one (the transposed operands of the backward
// products) each thread loads a 4 x 4 patch, four 8-byte loads, transposes it
// with byte permutes and stores four 8-byte pieces.
//
// Whole calls, ten in a replayed graph, 32,768 rows, microseconds; before: BK = 32,
// four workgroups per CU, transposed operands stored to LDS two bytes at a time,
// each chunk's load and each result's store under a branch of its own:
//   layer        896->256    256->256    256->512   | 256->125    256->343    1000->1001
//   forward       37 -> 27    22 -> 15    27 -> 25  |  20 -> 17    26 -> 25   153 -> 124
//   data          96 -> 43    44 -> 16    61 -> 22  |  38 -> 35    59 -> 49   363 -> 284
//   weight       235 -> 42   179 -> 27   182 -> 35  | 218 -> 41   224 -> 58   662 -> 246
// (left: whole vectors everywhere, gemm_vectors; right: a width that is none).
#include <algorithm>
#include <cmath>

#include "reduce.hpp"

namespace libp_amd {

typedef unsigned short u16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// float -> bf16, round to nearest even; NaN stays NaN
__device__ inline u16 f2bf(float f) {
  unsigned u = __builtin_bit_cast(unsigned, f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (u16)((u >> 16) | 0x40u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (u16)(u >> 16);
}
__device__ inline float bf2f(u16 h) { return __builtin_bit_cast(float, (unsigned)h << 16); }

constexpr int GBM = 128, GBN = 128, GBK = 64;
constexpr int GTHREADS = 256;

enum { EPI_F32_BIAS = 0, EPI_BF16_BIAS_RELU = 1, EPI_BF16_MASK = 2, EPI_F32_PARTIAL = 3 };

struct GemmArgs {
  int M, N, K;          // C is M x N, reduction over K
  const u16* A;         // TA=false: A[m*lda + k]; TA=true: A[k*lda + m]
  long lda;
  const u16* B;         // TB=false: B[n*ldb + k]; TB=true: B[k*ldb + n]
  long ldb;
  void* C;              // [M][ldc]; split s of a partial output at C + s*M*ldc (FP32)
  long ldc;
  const float* bias;    // [N] or null
  const u16* mask;      // [M][ldm] or null: output zeroed where mask <= 0
  long ldm;
  int kChunk;           // K range of one split (multiple of GBK)
  const float* rowScale = nullptr;  // EPI_F32_BIAS: C[m][n] = rowScale[m] * (A B + bias)[m][n] when set
};

// Workgroups are dispatched round-robin over the eight XCDs, each with its
// own L2. When the M tiles come in multiples of eight, the tiles are renamed
// so that the gridDim.x N tiles of one M tile run on one XCD, one after
// another: the A rows (the large operand) then reach that L2 once instead of
// once per N tile. In the same way the tiles of one K split run on one XCD
// when the splits come in multiples of eight (weight gradients: both operands'
// rows of the split are read by every tile). The tiles and their arithmetic
// are unchanged.
__device__ inline void gemm_tile(int& mt, int& nt, int& split) {
  mt = blockIdx.y, nt = blockIdx.x, split = blockIdx.z;
  if ((gridDim.z & 7) == 0) {
    const int tiles = gridDim.x * gridDim.y;
    const int b = blockIdx.x + gridDim.x * blockIdx.y + tiles * blockIdx.z, k = b >> 3, tile = k % tiles;
    split = (k / tiles) * 8 + (b & 7);
    nt = tile % gridDim.x;
    mt = tile / gridDim.x;
  } else if ((gridDim.y & 7) == 0) {
    const int b = blockIdx.x + gridDim.x * blockIdx.y;  // dispatch order within a K split
    const int k = b >> 3;
    nt = k % gridDim.x;
    mt = (k / gridDim.x) * 8 + (b & 7);
  }
}

// One operand tile in registers, on its way to LDS. No load sits under a branch, so
// the loads of the next K tile are all in flight during a tile's MFMAs. Rows past the
// end of A or B repeat the last one (their results are not stored); K entries past
// the end are zeroed on the way to LDS.
//
// In LDS the 16-byte chunk c of row n of a transposed operand sits at chunk
// c ^ (n / 16 % 4): the operand is read row by row, 32 lanes along 256 contiguous
// bytes (with eight rows per load, lanes across rows, every lane was a request of its
// own: dW of 32,768 x 896 x 256 took 67 us), and its patches, 4 rows of the tile
// apart, then meet on two lanes per bank instead of eight; the MFMA reads stay
// conflict-free.
template <bool T, int BK>
struct Tile {
  static constexpr int LD = BK + 8;                          // row stride in LDS
  static constexpr int GCH = GBM * BK * 2 / 16 / GTHREADS;  // 16-byte chunks per thread
  static __device__ inline int chunk(const int row, const int c) {
    return row * LD + ((T ? c ^ (row >> 4 & 3) : c) << 3);
  }
  u32x4 v[GCH];
  // as whole vectors: 8 bytes of a transposed operand's rows, 16 of another's
  __device__ inline void load(const u16* __restrict__ X, const long ld, const int row0, const int nrows, const int k0,
                              const int kEnd) {
    const int t = threadIdx.x;
    if (T) {  // patch i: rows k0 + 32 i + 4 (t / 32) + r, r = 0..3, columns row0 + 4 (t % 32) ..
      const u16* x = X + min(row0 + 4 * (t & 31), nrows - 4);
#pragma unroll
      for (int ir = 0; ir < 2 * GCH; ++ir) {
        const int gk = min(k0 + 32 * (ir >> 2) + 4 * (t >> 5) + (ir & 3), kEnd - 1);
        const u32x2 w = *reinterpret_cast<const u32x2*>(x + (long)gk * ld);
        v[ir >> 1][2 * (ir & 1)] = w.x;
        v[ir >> 1][2 * (ir & 1) + 1] = w.y;
      }
    } else {
#pragma unroll
      for (int i = 0; i < GCH; ++i) {
        const int c = t + GTHREADS * i;
        const int gr = min(row0 + c / (BK / 8), nrows - 1), gk = min(k0 + (c % (BK / 8)) * 8, kEnd - 8);
        v[i] = *reinterpret_cast<const u32x4*>(X + (long)gr * ld + gk);
      }
    }
  }
  // Whether load() serves this tile of an operand whose rows start on whole vectors: the
  // vectors of its contiguous dimension are whole inside it (the same for every thread).
  static __device__ inline bool whole(const int row0, const int nrows, const int k0, const int kEnd) {
    return T ? row0 + GBM <= nrows || nrows % 4 == 0 : k0 + BK <= kEnd || kEnd % 8 == 0;
  }
  // the same entries one by one; past an end the last one is read again, so that no load
  // sits under a branch
  __device__ inline void load_entries(const u16* __restrict__ X, const long ld, const int row0, const int nrows,
                                      const int k0, const int kEnd) {
    const int t = threadIdx.x;
    if (T) {
#pragma unroll
      for (int ir = 0; ir < 2 * GCH; ++ir) {
        const u16* x = X + (long)min(k0 + 32 * (ir >> 2) + 4 * (t >> 5) + (ir & 3), kEnd - 1) * ld;
        unsigned e[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) e[j] = x[min(row0 + 4 * (t & 31) + j, nrows - 1)];
        v[ir >> 1][2 * (ir & 1)] = e[0] | (e[1] << 16);
        v[ir >> 1][2 * (ir & 1) + 1] = e[2] | (e[3] << 16);
      }
    } else {
#pragma unroll
      for (int i = 0; i < GCH; ++i) {
        const int c = t + GTHREADS * i, gk = k0 + (c % (BK / 8)) * 8;
        const u16* x = X + (long)min(row0 + c / (BK / 8), nrows - 1) * ld;
        unsigned e[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = x[min(gk + j, kEnd - 1)];
#pragma unroll
        for (int j = 0; j < 8; ++j) e[j] = gk + j < kEnd ? e[j] : 0u;
        v[i] = u32x4{e[0] | (e[1] << 16), e[2] | (e[3] << 16), e[4] | (e[5] << 16), e[6] | (e[7] << 16)};
      }
    }
  }
  __device__ inline void store(u16* __restrict__ s, const int k0, const int kEnd) {
    const int t = threadIdx.x;
    if (k0 + BK > kEnd) {  // the last K tile of a split: entries past the end are zero
#pragma unroll
      for (int i = 0; i < GCH; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const int gk = T ? k0 + 32 * (i >> 1) + 4 * (t >> 5) + 2 * (i & 1) + h
                           : k0 + ((t + GTHREADS * i) % (BK / 8)) * 8;
          if (gk >= kEnd) v[i][2 * h] = v[i][2 * h + 1] = 0u;
        }
    }
    if (T) {  // column j of the patch: k entries of four rows, low and high halves picked by byte
#pragma unroll
      for (int ij = 0; ij < 2 * GCH; ++ij) {
        const int i = ij >> 2, j = ij & 3, d = j >> 1;
        const unsigned pick = (j & 1) ? 0x07060302u : 0x05040100u;
        u16* o = s + chunk(4 * (t & 31) + j, 4 * i + (t >> 6)) + 4 * (t >> 5 & 1);
        *reinterpret_cast<u32x2*>(o) = u32x2{__builtin_amdgcn_perm(v[2 * i][2 + d], v[2 * i][d], pick),
                                             __builtin_amdgcn_perm(v[2 * i + 1][2 + d], v[2 * i + 1][d], pick)};
      }
    } else {
#pragma unroll
      for (int i = 0; i < GCH; ++i) {
        const int c = t + GTHREADS * i;
        *reinterpret_cast<u32x4*>(s + chunk(c / (BK / 8), c % (BK / 8))) = v[i];
      }
    }
  }
};

constexpr int GCLD = GBN + 4;  // row stride of the result tile in LDS (FP32)

// VEC: every access of the product is a whole vector (gemm_vectors); the result tile
// goes through LDS, so bias, mask and C are read and written 16 bytes at a time.
// Otherwise each operand's tile takes vectors where its own rows allow them (an
// unaligned result, or the other operand, does not change that) and the result is
// written entry by entry: gathered to 128-byte runs through LDS first, 32,768 x 275 x
// 125 took 69 us (data gradient) against 60.
template <bool TA, bool TB, int EPI, bool VEC, int BK>
__global__ void __launch_bounds__(GTHREADS, BK == 32 ? 3 : 2) gemm_bf16_kernel(const GemmArgs g) {
  constexpr int LD = BK + 8;
  constexpr int ABYTES = 2 * 2 * GBM * LD * 2, CBYTES = VEC ? GBM * GCLD * 4 : 0;
  __shared__ __attribute__((aligned(16))) char smem[ABYTES > CBYTES ? ABYTES : CBYTES];
  u16* const sA = reinterpret_cast<u16*>(smem);
  u16* const sB = sA + 2 * GBM * LD;
  const int t = threadIdx.x, w = t >> 6, l = t & 63;
  const int wm = w >> 1, wn = w & 1;
  int mt, nt, split;
  gemm_tile(mt, nt, split);
  const int m0 = mt * GBM, n0 = nt * GBN;
  const int kBeg = split * g.kChunk;
  const int kEnd = min(g.K, kBeg + g.kChunk);
  const int nT = (kEnd > kBeg) ? (kEnd - kBeg + BK - 1) / BK : 0;

  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const int lr = l & 31, lc = l >> 5;
  const auto product = [&](const int buf) {
    const u16* a_s = sA + buf * GBM * LD;
    const u16* b_s = sB + buf * GBN * LD;
#pragma unroll
    for (int ks = 0; ks < BK; ks += 16) {
      bf16x8 a[2], b[2];
#pragma unroll
      for (int i = 0; i < 2; ++i)
        a[i] = *reinterpret_cast<const bf16x8*>(a_s + Tile<TA, BK>::chunk(wm * 64 + i * 32 + lr, ks / 8 + lc));
#pragma unroll
      for (int j = 0; j < 2; ++j)
        b[j] = *reinterpret_cast<const bf16x8*>(b_s + Tile<TB, BK>::chunk(wn * 64 + j * 32 + lr, ks / 8 + lc));
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    }
  };
  const bool vecA = VEC || (g.lda % 8 == 0 && ((uintptr_t)g.A & 15) == 0);
  const bool vecB = VEC || (g.ldb % 8 == 0 && ((uintptr_t)g.B & 15) == 0);
  const auto load = [&](auto& r, const u16* X, const long ld, const int row0, const int nrows, const int k0,
                        const bool vec) {
    if (VEC || (vec && r.whole(row0, nrows, k0, kEnd)))
      r.load(X, ld, row0, nrows, k0, kEnd);
    else
      r.load_entries(X, ld, row0, nrows, k0, kEnd);
  };
  if (nT > 0) {
    Tile<TA, BK> ra;
    Tile<TB, BK> rb;
    load(ra, g.A, g.lda, m0, g.M, kBeg, vecA);
    load(rb, g.B, g.ldb, n0, g.N, kBeg, vecB);
    ra.store(sA, kBeg, kEnd);
    rb.store(sB, kBeg, kEnd);
    __syncthreads();
    for (int it = 0; it + 1 < nT; ++it) {
      const int k0 = kBeg + (it + 1) * BK;
      load(ra, g.A, g.lda, m0, g.M, k0, vecA);
      load(rb, g.B, g.ldb, n0, g.N, k0, vecB);
      // all of the loads go out before the MFMAs: left to itself the scheduler spreads them
      // between, the last ones right before the stores that wait for them
      __builtin_amdgcn_sched_barrier(0);
      product(it & 1);
      ra.store(sA + ((it & 1) ^ 1) * GBM * LD, k0, kEnd);
      rb.store(sB + ((it & 1) ^ 1) * GBN * LD, k0, kEnd);
      __syncthreads();
    }
    product((nT - 1) & 1);
  }
  if constexpr (!VEC) {  // entry by entry
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int col = n0 + wn * 64 + j * 32 + lr;
        if (col >= g.N) continue;
        const float bcol = (g.bias && (EPI == EPI_F32_BIAS || EPI == EPI_BF16_BIAS_RELU)) ? g.bias[col] : 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3);
          if (row >= g.M) continue;
          const float v = acc[i][j][r];
          if (EPI == EPI_F32_BIAS) {
            const float o = v + bcol;
            reinterpret_cast<float*>(g.C)[(long)row * g.ldc + col] = g.rowScale ? g.rowScale[row] * o : o;
          } else if (EPI == EPI_BF16_BIAS_RELU) {
            reinterpret_cast<u16*>(g.C)[(long)row * g.ldc + col] = f2bf(fmaxf(v + bcol, 0.f));
          } else if (EPI == EPI_BF16_MASK) {
            const bool keep = !g.mask || bf2f(g.mask[(long)row * g.ldm + col]) > 0.f;
            reinterpret_cast<u16*>(g.C)[(long)row * g.ldc + col] = f2bf(keep ? v : 0.f);
          } else {
            reinterpret_cast<float*>(g.C)[(long)split * g.M * g.ldc + (long)row * g.ldc + col] = v;
          }
        }
      }
    return;
  }
  __syncthreads();  // the tiles have been read: the result tile takes their place

  float* const sC = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r)
        sC[(wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (l >> 5) + (r & 3)) * GCLD + wn * 64 + j * 32 + lr] = acc[i][j][r];
  __syncthreads();
  constexpr bool BF = EPI == EPI_BF16_BIAS_RELU || EPI == EPI_BF16_MASK;
  constexpr int W = BF ? 8 : 4, RC = GBN / W, STEP = GTHREADS / RC, NS = GBM / STEP;  // W columns per access
  const int cc = (t % RC) * W, r0 = t / RC;
  const int col = n0 + cc;
  if (col >= g.N) return;
  float bias[W];
#pragma unroll
  for (int e = 0; e < W; ++e)
    bias[e] = (g.bias && (EPI == EPI_F32_BIAS || EPI == EPI_BF16_BIAS_RELU)) ? g.bias[col + e] : 0.f;
  u32x4 mask[EPI == EPI_BF16_MASK ? NS : 1];
  float scale[EPI == EPI_F32_BIAS ? NS : 1];
  if (EPI == EPI_BF16_MASK && g.mask) {
#pragma unroll
    for (int k = 0; k < NS; ++k)
      mask[k] = *reinterpret_cast<const u32x4*>(g.mask + (long)min(m0 + r0 + STEP * k, g.M - 1) * g.ldm + col);
  }
  if (EPI == EPI_F32_BIAS && g.rowScale) {
#pragma unroll
    for (int k = 0; k < NS; ++k) scale[k] = g.rowScale[min(m0 + r0 + STEP * k, g.M - 1)];
  }
#pragma unroll
  for (int k = 0; k < NS; ++k) {
    const int lrow = r0 + STEP * k, row = m0 + lrow;
    float v[W];
#pragma unroll
    for (int e = 0; e < W; e += 4) {
      const f32x4 x = *reinterpret_cast<const f32x4*>(sC + lrow * GCLD + cc + e);
#pragma unroll
      for (int j = 0; j < 4; ++j) v[e + j] = x[j];
    }
    if (row < g.M) {
      if (BF) {
        unsigned o[W];
#pragma unroll
        for (int e = 0; e < W; ++e) {
          if (EPI == EPI_BF16_BIAS_RELU) {
            o[e] = f2bf(fmaxf(v[e] + bias[e], 0.f));
          } else {
            const unsigned m = mask[k][e >> 1];
            const bool keep = !g.mask || bf2f((u16)((e & 1) ? (m >> 16) : (m & 0xffffu))) > 0.f;
            o[e] = f2bf(keep ? v[e] : 0.f);
          }
        }
        *reinterpret_cast<u32x4*>(reinterpret_cast<u16*>(g.C) + (long)row * g.ldc + col) =
            u32x4{o[0] | (o[1] << 16), o[2] | (o[3] << 16), o[4] | (o[5] << 16), o[6] | (o[7] << 16)};
      } else {
        f32x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          o[e] = v[e];
          if (EPI == EPI_F32_BIAS) {
            o[e] = v[e] + bias[e];
            if (g.rowScale) o[e] = scale[k] * o[e];
          }
        }
        const long base = EPI == EPI_F32_PARTIAL ? (long)split * g.M * g.ldc : 0;
        *reinterpret_cast<f32x4*>(reinterpret_cast<float*>(g.C) + base + (long)row * g.ldc + col) = o;
      }
    }
  }
}

// Whether the VEC form serves the product: pointers and leading dimensions
// whole vectors, the vectors of the contiguous dimension whole inside the matrix.
template <bool TA, bool TB, int EPI>
static bool gemm_vectors(const GemmArgs& g) {
  const auto on16 = [](const void* p) { return ((uintptr_t)p & 15) == 0; };
  constexpr bool BF = EPI == EPI_BF16_BIAS_RELU || EPI == EPI_BF16_MASK;
  const int W = BF ? 8 : 4;
  const bool a = on16(g.A) && g.lda % 8 == 0 && (TA ? g.M % 4 == 0 : g.K % 8 == 0);
  const bool b = on16(g.B) && g.ldb % 8 == 0 && (TB ? g.N % 4 == 0 : g.K % 8 == 0);
  const bool c = on16(g.C) && g.ldc % W == 0 && g.N % W == 0 && (EPI != EPI_F32_PARTIAL || (g.M * g.ldc) % 4 == 0);
  return a && b && c && (!g.mask || (on16(g.mask) && g.ldm % 8 == 0));
}

template <bool TA, bool TB, int EPI>
static int gemm(const GemmArgs& g, int splits, void* stream, const char* where) {
  if (g.M <= 0 || g.N <= 0) return LIBP_OK;
  dim3 grid((g.N + GBN - 1) / GBN, (g.M + GBM - 1) / GBM, splits);
  // Two workgroups of BK = 64 fit a CU, three of BK = 32: the smaller step where that takes one
  // round over the 256 CUs instead of two (768 tiles: data gradient of 275 x 125 43 us against 60,
  // forward 256 -> 343 25 against 33); elsewhere it is slower (512 tiles: forward 896 -> 256 with
  // unaligned rows 136 us against 100).
  const unsigned tiles = grid.x * grid.y * grid.z;
  const auto kernel = gemm_vectors<TA, TB, EPI>(g)  ? gemm_bf16_kernel<TA, TB, EPI, true, GBK>
                      : tiles > 512 && tiles <= 768 ? gemm_bf16_kernel<TA, TB, EPI, false, 32>
                                                    : gemm_bf16_kernel<TA, TB, EPI, false, GBK>;
  hipLaunchKernelGGL(kernel, grid, dim3(GTHREADS), 0, as_stream(stream), g);
  return launch_status(where);
}

// Column sums of a BF16 [M][ld] matrix, two stages: block (x, y) sums 64 columns
// over the rows of chunk y, 8 columns (16 bytes where aligned) x 32 rows at a
// time, into P[y][col]; the second kernel sums the chunks. The loads of four
// steps are in flight together. (A thread per column over 256 rows in turn, two
// bytes per load, took 60 us for 32,768 x 256: 128 blocks of dependent loads.)
__global__ void __launch_bounds__(256) colsum_bf16_kernel(const int M, const int N, const u16* __restrict__ X,
                                                          const long ld, const int rowsPerChunk, const bool vec,
                                                          float* __restrict__ P) {
  __shared__ float s_a[32][65];
  const int t = threadIdx.x, cg = t & 7, rl = t >> 3;
  const int c0 = blockIdx.x * 64 + cg * 8;
  const int r0 = blockIdx.y * rowsPerChunk, r1 = min(M, r0 + rowsPerChunk);
  float a[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) a[j] = 0.f;
  if (vec && c0 + 8 <= N) {
    for (int r = r0 + rl; r < r1; r += 128) {
      u32x4 w[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] = *reinterpret_cast<const u32x4*>(X + (long)min(r + 32 * u, r1 - 1) * ld + c0);
#pragma unroll
      for (int u = 0; u < 4; ++u)
        if (r + 32 * u < r1)
#pragma unroll
          for (int j = 0; j < 8; ++j) a[j] += bf2f((u16)((j & 1) ? (w[u][j >> 1] >> 16) : (w[u][j >> 1] & 0xffffu)));
    }
  } else {
    for (int r = r0 + rl; r < r1; r += 32)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        if (c0 + j < N) a[j] += bf2f(X[(long)r * ld + c0 + j]);
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) s_a[rl][cg * 8 + j] = a[j];
  __syncthreads();
  if (t < 64 && blockIdx.x * 64 + t < N) {
    float v = 0.f;
#pragma unroll
    for (int r = 0; r < 32; ++r) v += s_a[r][t];
    P[(long)blockIdx.y * N + blockIdx.x * 64 + t] = v;
  }
}
// The partial sums of a weight gradient, in one launch (two of their own cost a
// launch each, ~4.7 us): blocks below sumBlocks form out[i] = sum_s P[s*n + i], s in
// order (deterministic), with eight loads in flight (32 splits of 229,376 entries
// took 30 us as a chain of dependent loads, 6 us so); the rest form 16 column sums
// each from the C <= 128 chunks of Pc, eight per segment.
__global__ void __launch_bounds__(256) weight_finish_kernel(const long n, const int S, const float* __restrict__ P,
                                                            float* __restrict__ out, const int sumBlocks, const int N,
                                                            const int C, const float* __restrict__ Pc,
                                                            float* __restrict__ db) {
  if (blockIdx.x < (unsigned)sumBlocks) {
    for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)sumBlocks * blockDim.x) {
      float a = 0.f;
      for (int s0 = 0; s0 < S; s0 += 8) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = P[(long)min(s0 + u, S - 1) * n + i];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          if (s0 + u < S) a += v[u];
      }
      out[i] = a;
    }
    return;
  }
  __shared__ float s_a[16][17];
  const int col = (blockIdx.x - sumBlocks) * 16 + (threadIdx.x & 15), seg = threadIdx.x >> 4;
  float v[8], a = 0.f;
#pragma unroll
  for (int u = 0; u < 8; ++u) v[u] = Pc[(long)min(seg + 16 * u, C - 1) * N + min(col, N - 1)];
#pragma unroll
  for (int u = 0; u < 8; ++u)
    if (seg + 16 * u < C) a += v[u];
  s_a[seg][threadIdx.x & 15] = a;
  __syncthreads();
  if (seg == 0 && col < N) {
    float b = 0.f;
#pragma unroll
    for (int k = 0; k < 16; ++k) b += s_a[k][threadIdx.x];
    db[col] = b;
  }
}

__global__ void __launch_bounds__(256) f32_to_bf16_kernel(const long n, const float* __restrict__ x,
                                                          u16* __restrict__ y) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[i] = f2bf(x[i]);
}

// Adam (Kingma & Ba 2015) on FP32 masters with a BF16 copy of the result.
// c1 = 1/(1 - beta1^t), c2 = 1/(1 - beta2^t).
__global__ void __launch_bounds__(256) adam_kernel(const int n, float* __restrict__ p, u16* __restrict__ pb,
                                                   const float* __restrict__ grad, float* __restrict__ m,
                                                   float* __restrict__ v, const float lr, const float b1,
                                                   const float b2, const float eps, const float c1, const float c2) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float gi = grad[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    const float pi = p[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
    p[i] = pi;
    if (pb) pb[i] = f2bf(pi);
  }
}

// Split-K sizing of the weight gradient (reduction over M rows): as many splits
// as give two workgroups per CU over the output tiles, of 256 rows at least and
// 64 splits at most, so that the partial sums stay few.
static void weight_splits(int M, int K, int Nout, int& S, int& kChunk) {
  const int tiles = ((K + GBN - 1) / GBN) * ((Nout + GBM - 1) / GBM);
  S = (512 + tiles - 1) / tiles;
  S = std::min(std::min(S, 64), (M + 255) / 256);
  if (S >= 8) S = S / 8 * 8;
  if (S < 1) S = 1;
  kChunk = ((M + S - 1) / S + GBK - 1) / GBK * GBK;
  if (S < 8) S = std::max(1, (M + kChunk - 1) / kChunk);  // from 8 on, trailing splits may be empty (zero partials)
}
static int colsum_chunks(int M) { return M < 256 ? 1 : (M + 255) / 256 > 128 ? 128 : (M + 255) / 256; }

}  // namespace libp_amd

using namespace libp_amd;

extern "C" int libp_mlp_linear_fwd(int M, int K, int Nout, const unsigned short* X, long ldx, const unsigned short* Wt,
                                   long ldw, const float* b, int relu, void* Y, long ldy, void* stream) {
  if (M < 0 || K <= 0 || Nout <= 0) return arg_error("mlp_linear_fwd", "bad size");
  if (!X || !Wt || !Y) return arg_error("mlp_linear_fwd", "null pointer");
  if (ldx < K || ldw < K || ldy < Nout) return arg_error("mlp_linear_fwd", "leading dimension too small");
  GemmArgs g{M, Nout, K, X, ldx, Wt, ldw, Y, ldy, b, nullptr, 0, ((K + GBK - 1) / GBK) * GBK};
  if (relu) return gemm<false, false, EPI_BF16_BIAS_RELU>(g, 1, stream, "mlp_linear_fwd");
  return gemm<false, false, EPI_F32_BIAS>(g, 1, stream, "mlp_linear_fwd");
}

extern "C" int libp_mlp_linear_fwd_scaled(int M, int K, int Nout, const unsigned short* X, long ldx,
                                          const unsigned short* Wt, long ldw, const float* b, const float* rowScale,
                                          float* Y, long ldy, void* stream) {
  if (M < 0 || K <= 0 || Nout <= 0) return arg_error("mlp_linear_fwd_scaled", "bad size");
  if (!X || !Wt || !Y || !rowScale) return arg_error("mlp_linear_fwd_scaled", "null pointer");
  if (ldx < K || ldw < K || ldy < Nout) return arg_error("mlp_linear_fwd_scaled", "leading dimension too small");
  GemmArgs g{M, Nout, K, X, ldx, Wt, ldw, Y, ldy, b, nullptr, 0, ((K + GBK - 1) / GBK) * GBK, rowScale};
  return gemm<false, false, EPI_F32_BIAS>(g, 1, stream, "mlp_linear_fwd_scaled");
}

extern "C" int libp_mlp_linear_bwd_data(int M, int K, int Nout, const unsigned short* dY, long lddy,
                                        const unsigned short* Wt, long ldw, const unsigned short* H, long ldh,
                                        unsigned short* dX, long lddx, void* stream) {
  if (M < 0 || K <= 0 || Nout <= 0) return arg_error("mlp_linear_bwd_data", "bad size");
  if (!dY || !Wt || !dX) return arg_error("mlp_linear_bwd_data", "null pointer");
  if (lddy < Nout || ldw < K || lddx < K || (H && ldh < K)) return arg_error("mlp_linear_bwd_data", "leading dimension");
  // dX[m][k] = sum_n dY[m][n] Wt[n][k]: A = dY (K-contiguous over n), B(k, n) = Wt[n*ldw + k] (transposed)
  GemmArgs g{M, K, Nout, dY, lddy, Wt, ldw, dX, lddx, nullptr, H, ldh, ((Nout + GBK - 1) / GBK) * GBK};
  return gemm<false, true, EPI_BF16_MASK>(g, 1, stream, "mlp_linear_bwd_data");
}

extern "C" long libp_mlp_ws_bytes(int M, int K, int Nout) {
  // The splits of weight_splits fall as the tiles grow, so S * Nout * K does not grow with every
  // size; what is asked for does, and a workspace of the largest call serves the smaller ones:
  // S <= one per 256 rows and 64, and S * tiles < 512 + tiles (34 MB of splits beside the result).
  const long rows = std::min(64L, (M + 255L) / 256), entries = (long)Nout * K;
  const long tiles = ((K + GBN - 1L) / GBN) * ((Nout + GBM - 1L) / GBM);
  const long splits = std::min(std::max(rows, 1L) * entries, (511 + tiles) * GBM * GBN);
  return splits * 4 + (long)colsum_chunks(M) * Nout * 4 + 256;
}

extern "C" int libp_mlp_linear_bwd_weight(int M, int K, int Nout, const unsigned short* dY, long lddy,
                                          const unsigned short* X, long ldx, float* dWt, float* db, void* ws,
                                          void* stream) {
  if (M <= 0 || K <= 0 || Nout <= 0) return arg_error("mlp_linear_bwd_weight", "bad size");
  if (!dY || !X || !dWt || !ws) return arg_error("mlp_linear_bwd_weight", "null pointer");
  if (lddy < Nout || ldx < K) return arg_error("mlp_linear_bwd_weight", "leading dimension");
  int S, kc;
  weight_splits(M, K, Nout, S, kc);
  float* P = reinterpret_cast<float*>(ws);
  // dWt[n][k] = sum_m dY[m][n] X[m][k]: A(n, m) = dY[m*lddy + n], B(k, m) = X[m*ldx + k] (both transposed)
  GemmArgs g{Nout, K, M, dY, lddy, X, ldx, P, K, nullptr, nullptr, 0, kc};
  int st = gemm<true, true, EPI_F32_PARTIAL>(g, S, stream, "mlp_linear_bwd_weight");
  if (st) return st;
  const long n = (long)Nout * K;
  const unsigned sumBlocks = stream_blocks(n, 256, 4096);
  const int C = colsum_chunks(M);
  float* Pc = P + (long)S * Nout * K;
  if (db) {
    const bool vec = (lddy % 8) == 0 && ((uintptr_t)dY & 15) == 0;
    hipLaunchKernelGGL(colsum_bf16_kernel, dim3((Nout + 63) / 64, C), dim3(256), 0, as_stream(stream), M, Nout, dY,
                       lddy, (M + C - 1) / C, vec, Pc);
  }
  hipLaunchKernelGGL(weight_finish_kernel, dim3(sumBlocks + (db ? (Nout + 15) / 16 : 0)), dim3(256), 0,
                     as_stream(stream), n, S, P, dWt, (int)sumBlocks, Nout, C, Pc, db);
  return launch_status("mlp_linear_bwd_weight");
}

extern "C" int libp_adam_step(int n, float* master, unsigned short* wbf16, const float* grad, float* m, float* v,
                              float lr, float beta1, float beta2, float eps, int step, void* stream) {
  if (n <= 0) return LIBP_OK;
  if (!master || !grad || !m || !v) return arg_error("adam_step", "null pointer");
  if (step < 1) return arg_error("adam_step", "step counts from 1");
  const float c1 = (float)(1.0 / (1.0 - std::pow((double)beta1, step)));
  const float c2 = (float)(1.0 / (1.0 - std::pow((double)beta2, step)));
  hipLaunchKernelGGL(adam_kernel, dim3(stream_blocks(n, 256, 4096)), dim3(256), 0, as_stream(stream), n, master, wbf16,
                     grad, m, v, lr, beta1, beta2, eps, c1, c2);
  return launch_status("adam_step");
}

extern "C" int libp_f32_to_bf16(long n, const float* x, unsigned short* y, void* stream) {
  if (n <= 0) return LIBP_OK;
  if (!x || !y) return arg_error("f32_to_bf16", "null pointer");
  hipLaunchKernelGGL(f32_to_bf16_kernel, dim3(stream_blocks(n, 256, 4096)), dim3(256), 0, as_stream(stream), n, x, y);
  return launch_status("f32_to_bf16");
}
