// p-multigrid intergrid transfers for hex elements (FP64 and FP32).
//
// Each transfer is three 1-D contractions with P (NqF x NqC): k, j, i for the
// restriction (okl/ellipticPreconCoarsenHex3D.okl:209-294), i, j, k for the
// prolongation (okl/ellipticPreconProlongateHex3D.okl:216-301). A workgroup takes
// NE elements. Their nodes are read and written flat (consecutive threads,
// consecutive nodes), and in a contraction a thread holds one whole line: both
// sizes are template arguments, so the line sits in registers, and the entries of
// P, the same for every lane, come through scalar loads (a coarse size known only at
// run time loads P entry by entry: 10->9 in FP32 took 45 us against 30).
//
// The form before took a NqF x NqF tile per element (the same arithmetic and order,
// bit for bit), read P from LDS for every product, left lanes idle (49 of 64 at
// NqF = 7) and had known sizes at 7->3 and 3->1 only; it is left where it is the
// faster one (mg_prolong_tile_kernel). What bounds this one: HBM (12 bytes per fine
// node with the weights, FP32), and for the restriction the latency of its
// index -> value loads. 8M fine nodes, microseconds, weighted restriction /
// prolongation before and now (in turn on one card, ten launches in a replayed graph):
//             2->1      3->1      4->2      6->4      7->3      9->8     12->9    15->11    15->14
//   FP64   107/107     60/33     56/44     69/41     52/18     63/69     57/65     57/84    66/121
//      now   28/23     31/19     32/21     39/26     38/16     53/36     44/32     42/39     58/53
//   FP32    93/102     47/32     47/41     53/35     44/11     49/46     41/38     40/43     45/65
//      now   27/18     25/14     28/15     31/18     31/12     42/24     34/21     32/23     35/29
#include <type_traits>

#include "kcommon.hpp"

namespace libp_amd {

// Elements and threads per workgroup: about 1000 nodes, and threads for all the
// fine lines of one direction where that is a multiple of a wavefront or close to it
// (7->3 at 1 element / 64 threads, 2 / 128 and 4 / 256 prolongs in 17.6, 16.7 and 16.7 us).
template <int NqF>
struct MgShape {
  static constexpr int NE = NqF <= 3 ? 32 : NqF <= 5 ? 8 : NqF <= 7 ? 4 : NqF == 8 ? 2 : 1;
  static constexpr int threads = (NqF >= 8 && NqF <= 11) || NqF == 4 ? 128 : 256;
};

// out(c, sum_m P[m][c] x[m]), six c at a time: each row of P gives six neighbouring
// entries per scalar load. One c at a time is NqF loads of a column, which the compiler
// pipelines only where the count of c has a small factor (15->14 in FP64, 1728 elements:
// 66 us as a tile, 80 so, 58 with six; 9->8 at 8 elements 6.0, 8.8 and 5.2; two, three
// or four at a time are slower at Nq >= 9, eight alike).
template <int NqF, int NqC, typename T, typename F>
__device__ inline void mg_restrict_line(const T* __restrict__ P, const T (&x)[NqF], const F& out) {
  constexpr int UC = 6;
  const auto some = [&](const int c0, auto n) {
    T res[n];
#pragma unroll
    for (int u = 0; u < n; ++u) res[u] = 0;
#pragma unroll
    for (int m = 0; m < NqF; ++m)
#pragma unroll
      for (int u = 0; u < n; ++u) res[u] += P[m * NqC + c0 + u] * x[m];
#pragma unroll
    for (int u = 0; u < n; ++u) out(c0 + u, res[u]);
  };
  if constexpr (NqC >= UC)
    for (int c = 0; c + UC <= NqC; c += UC) some(c, std::integral_constant<int, UC>());
  if constexpr (NqC % UC > 0) some(NqC - NqC % UC, std::integral_constant<int, NqC % UC>());
}

template <int NqF, int NqC, typename T>
__global__ void __launch_bounds__(MgShape<NqF>::threads)
    mg_coarsen_kernel(const int Nelements, const int* __restrict__ elementList,
                      const int* __restrict__ G2L, const T* __restrict__ P, const T* __restrict__ qf,
                      const T* __restrict__ w, T* __restrict__ qc) {
  constexpr int NE = MgShape<NqF>::NE, B = MgShape<NqF>::threads, FF = NqF * NqF, NpF = NqF * FF, NN = NE * NpF;
  constexpr int UN = (NN + B - 1) / B, R = NqF | 1;  // rows of the last contraction, odd stride
  __shared__ T s_f[NE * (NqF - 1) * (NqF - 1) * R > NN ? NE * (NqF - 1) * (NqF - 1) * R : NN];
  __shared__ T s_c[NE * (NqF - 1) * FF];
  const int t = threadIdx.x, e0 = blockIdx.x * NE, last = Nelements - 1 - e0;
  const auto element = [&](const int es) {  // a group past the end repeats its last element
    const int e = e0 + min(es, last);
    return (size_t)(elementList ? elementList[e] : e);
  };
  // index loads first, then unconditional value loads (masked nodes read entry 0 and take 0):
  // loads under (id >= 0) compile to branches that wait for each load in turn
  int ids[UN];
  T q[UN], wv[UN];
#pragma unroll
  for (int u = 0; u < UN; ++u) {
    const int n = min(t + u * B, NN - 1);
    ids[u] = __builtin_nontemporal_load(G2L + element(n / NpF) * NpF + n % NpF);
  }
#pragma unroll
  for (int u = 0; u < UN; ++u) {
    const int id = max(ids[u], 0);
    q[u] = qf[id];
    // w: the inverse-multiplicity weight of the fine residual (ellipticPreconMultiGridLevel.cpp:51),
    // applied here instead of in a separate pass (the same single rounding)
    if (w) wv[u] = w[id];
  }
#pragma unroll
  for (int u = 0; u < UN; ++u)
    if ((u + 1) * B <= NN || t + u * B < NN)
      s_f[t + u * B] = (ids[u] >= 0) ? (w ? T(1) * wv[u] * q[u] : q[u]) : T(0);
  __syncthreads();
  // k: lines (e, j, i) of s_f -> s_c[e][c][j][i]
  for (int p = t; p < NE * FF; p += B) {
    const int e = p / FF, ji = p % FF;
    T x[NqF];
#pragma unroll
    for (int m = 0; m < NqF; ++m) x[m] = s_f[e * NpF + m * FF + ji];
    mg_restrict_line<NqF, NqC>(P, x, [&](const int c, const T v) { s_c[(e * NqC + c) * FF + ji] = v; });
  }
  __syncthreads();
  // j: lines (e, k, i) of s_c -> s_f[e][k][c][i], rows of R
  for (int p = t; p < NE * NqC * NqF; p += B) {
    const int ek = p / NqF, i = p % NqF;
    T x[NqF];
#pragma unroll
    for (int m = 0; m < NqF; ++m) x[m] = s_c[ek * FF + m * NqF + i];
    mg_restrict_line<NqF, NqC>(P, x, [&](const int c, const T v) { s_f[(ek * NqC + c) * R + i] = v; });
  }
  __syncthreads();
  // i: lines (e, k, j) of s_f -> s_c, flat coarse nodes
  for (int p = t; p < NE * NqC * NqC; p += B) {
    T x[NqF];
#pragma unroll
    for (int m = 0; m < NqF; ++m) x[m] = s_f[p * R + m];
    mg_restrict_line<NqF, NqC>(P, x, [&](const int c, const T v) { s_c[p * NqC + c] = v; });
  }
  __syncthreads();
  const int NpC = NqC * NqC * NqC;
  for (int n = t; n < NE * NpC; n += B) {
    const int e = n / NpC;
    qc[element(e) * NpC + (n - e * NpC)] = s_c[n];
  }
}

template <int NqF, int NqC, typename T>
__global__ void __launch_bounds__(MgShape<NqF>::threads)
    mg_prolong_kernel(const int Nelements, const int* __restrict__ elementList,
                      const int* __restrict__ G2LC, const T* __restrict__ P, const T* __restrict__ qcIn,
                      T* __restrict__ qN) {
  constexpr int NE = MgShape<NqF>::NE, B = MgShape<NqF>::threads, FF = NqF * NqF, NpF = NqF * FF, C = NqF - 1;
  constexpr int UN = (NE * C * C * C + B - 1) / B;
  __shared__ T s_c[NE * C * NqF * NqF];  // coarse nodes, then [e][k][j fine][i fine]
  __shared__ T s_m[NE * C * C * NqF];    // [e][k][j][i fine]
  const int t = threadIdx.x, e0 = blockIdx.x * NE, last = Nelements - 1 - e0;
  const auto element = [&](const int es) {
    const int e = e0 + min(es, last);
    return (size_t)(elementList ? elementList[e] : e);
  };
  const int NpC = NqC * NqC * NqC, NC = NE * NpC;
  // index loads first, then unconditional value loads; u * B < NC is the same for every lane
  int ids[UN];
#pragma unroll
  for (int u = 0; u < UN; ++u)
    if (u * B < NC) {
      const int n = min(t + u * B, NC - 1), e = n / NpC;
      ids[u] = __builtin_nontemporal_load(G2LC + element(e) * NpC + (n - e * NpC));
    }
  T q[UN];
#pragma unroll
  for (int u = 0; u < UN; ++u)
    if (u * B < NC) q[u] = qcIn[max(ids[u], 0)];
#pragma unroll
  for (int u = 0; u < UN; ++u)
    if (t + u * B < NC) s_c[t + u * B] = (ids[u] >= 0) ? q[u] : T(0);
  __syncthreads();
  // i: lines (e, k, j) -> s_m
  for (int p = t; p < NE * NqC * NqC; p += B) {
    T o[NqF];
#pragma unroll
    for (int f = 0; f < NqF; ++f) o[f] = 0;
    for (int m = 0; m < NqC; ++m) {
      const T x = s_c[p * NqC + m];
#pragma unroll
      for (int f = 0; f < NqF; ++f) o[f] += P[f * NqC + m] * x;
    }
#pragma unroll
    for (int f = 0; f < NqF; ++f) s_m[p * NqF + f] = o[f];
  }
  __syncthreads();
  // j: lines (e, k, i) -> s_c
  for (int p = t; p < NE * NqC * NqF; p += B) {
    const int ek = p / NqF, i = p % NqF;
    T o[NqF];
#pragma unroll
    for (int f = 0; f < NqF; ++f) o[f] = 0;
    for (int m = 0; m < NqC; ++m) {
      const T x = s_m[(ek * NqC + m) * NqF + i];
#pragma unroll
      for (int f = 0; f < NqF; ++f) o[f] += P[f * NqC + m] * x;
    }
#pragma unroll
    for (int f = 0; f < NqF; ++f) s_c[ek * FF + f * NqF + i] = o[f];
  }
  __syncthreads();
  // k: lines (e, j, i) -> the E-vector; at each f a run of consecutive nodes
  for (int p = t; p < NE * FF; p += B) {
    const int e = p / FF, ji = p % FF;
    T o[NqF];
#pragma unroll
    for (int f = 0; f < NqF; ++f) o[f] = 0;
    for (int m = 0; m < NqC; ++m) {
      const T x = s_c[(e * NqC + m) * FF + ji];
#pragma unroll
      for (int f = 0; f < NqF; ++f) o[f] += P[f * NqC + m] * x;
    }
    T* out = qN + element(e) * NpF + ji;
#pragma unroll
    for (int f = 0; f < NqF; ++f) out[f * FF] = o[f];
  }
}

// The prolongation with one wavefront per element, an 8 x 8 tile of its fine nodes, each
// thread one (j, i). It keeps to itself (no barrier waits for another wave), which is
// worth more than idle lanes while the coarse tile fills at most a quarter of it: 15,625
// elements, FP64, 7->1, 7->2, 7->3 13.8, 14.8 and 16.5 us against 16.0, 17.6 and 18.4 in
// mg_prolong_kernel, but 7->5 and 7->6 26.1 and 32.9 against 24.6 and 30.2 (7->4 alike).
template <int NqC, typename T>
__global__ void __launch_bounds__(64) mg_prolong_tile_kernel(const int* __restrict__ elementList,
                                                             const int* __restrict__ G2LC, const T* __restrict__ P,
                                                             const T* __restrict__ qcIn, T* __restrict__ qN) {
  constexpr int NqF = 8;
  __shared__ T s_A[NqC][NqF][NqF];  // coarse nodes, then the planes after the j sweep
  __shared__ T s_ccf[NqC][NqC][NqF];
  __shared__ T s_P[NqF][NqF - 1];
  const size_t element = elementList ? elementList[blockIdx.x] : blockIdx.x;
  const int t = threadIdx.x, i = t % NqF, j = t / NqF;
  if (i < NqC && j < NqC) {
    // index loads first, then unconditional value loads
    int ids[NqC];
#pragma unroll
    for (int k = 0; k < NqC; ++k) ids[k] = G2LC[element * (NqC * NqC * NqC) + i + j * NqC + k * NqC * NqC];
#pragma unroll
    for (int k = 0; k < NqC; ++k) {
      const T qv = qcIn[max(ids[k], 0)];
      s_A[k][j][i] = (ids[k] >= 0) ? qv : T(0);
    }
  }
  if (t < NqF * NqC) s_P[t / NqC][t % NqC] = P[t];
  __syncthreads();
  if (j < NqC)
    for (int k = 0; k < NqC; ++k) {
      T res = 0;
      for (int m = 0; m < NqC; ++m) res += s_P[i][m] * s_A[k][j][m];
      s_ccf[k][j][i] = res;
    }
  __syncthreads();
  for (int k = 0; k < NqC; ++k) {
    T res = 0;
    for (int m = 0; m < NqC; ++m) res += s_P[j][m] * s_ccf[k][m][i];
    s_A[k][j][i] = res;
  }
  __syncthreads();
  for (int k = 0; k < NqF; ++k) {
    T res = 0;
    for (int m = 0; m < NqC; ++m) res += s_P[k][m] * s_A[m][j][i];
    qN[element * (NqF * NqF * NqF) + i + j * NqF + k * NqF * NqF] = res;
  }
}

// the kernel of coarse size nqc, NqC <= nqc < NqF
template <int NqF, int NqC, typename T, bool COARSEN>
static void launch_transfer(int nqc, int Nelements, const int* elist, const int* g2l, const T* P, const T* in,
                            const T* w, T* out, hipStream_t st) {
  if constexpr (NqC < NqF) {
    if (nqc != NqC) return launch_transfer<NqF, NqC + 1, T, COARSEN>(nqc, Nelements, elist, g2l, P, in, w, out, st);
    const dim3 grid((Nelements + MgShape<NqF>::NE - 1) / MgShape<NqF>::NE), block(MgShape<NqF>::threads);
    if constexpr (COARSEN)
      hipLaunchKernelGGL((mg_coarsen_kernel<NqF, NqC, T>), grid, block, 0, st, Nelements, elist, g2l, P, in, w, out);
    else if constexpr (NqF == 8 && NqC <= 4)
      hipLaunchKernelGGL((mg_prolong_tile_kernel<NqC, T>), dim3(Nelements), dim3(64), 0, st, elist, g2l, P, in, out);
    else
      hipLaunchKernelGGL((mg_prolong_kernel<NqF, NqC, T>), grid, block, 0, st, Nelements, elist, g2l, P, in, out);
  }
}

template <typename T, bool COARSEN>
static int transfer(int Nf, int Nc, int Nelements, const int* elist, const int* g2l, const T* P, const T* in, T* out,
                    void* stream, const T* w = nullptr) {
  if (Nelements <= 0) return LIBP_OK;
  if (Nc < 1 || Nc >= Nf || Nf > 15) return arg_error("mg_transfer", "need 1 <= Nc < Nf <= 15");
  if (!g2l || !P || !in || !out) return arg_error("mg_transfer", "null pointer");
  hipStream_t st = as_stream(stream);
  switch (Nf) {
#define LIBP_MG_CASE(NF)                                                                     \
  case NF:                                                                                   \
    launch_transfer<NF + 1, 2, T, COARSEN>(Nc + 1, Nelements, elist, g2l, P, in, w, out, st); \
    break;
    LIBP_MG_CASE(2)
    LIBP_MG_CASE(3)
    LIBP_MG_CASE(4)
    LIBP_MG_CASE(5)
    LIBP_MG_CASE(6)
    LIBP_MG_CASE(7)
    LIBP_MG_CASE(8)
    LIBP_MG_CASE(9)
    LIBP_MG_CASE(10)
    LIBP_MG_CASE(11)
    LIBP_MG_CASE(12)
    LIBP_MG_CASE(13)
    LIBP_MG_CASE(14)
    LIBP_MG_CASE(15)
#undef LIBP_MG_CASE
    default:
      return arg_error("mg_transfer", "unsupported fine degree");
  }
  return launch_status(COARSEN ? "mg_coarsen" : "mg_prolong");
}

}  // namespace libp_amd

using namespace libp_amd;

extern "C" int libp_mg_coarsen_hex_f64(int Nf, int Nc, int Nelements, const int* elementList,
                                       const int* GlobalToLocal, const double* P, const double* qf, double* qc,
                                       void* stream) {
  return transfer<double, true>(Nf, Nc, Nelements, elementList, GlobalToLocal, P, qf, qc, stream);
}
extern "C" int libp_mg_coarsen_hex_f32(int Nf, int Nc, int Nelements, const int* elementList,
                                       const int* GlobalToLocal, const float* P, const float* qf, float* qc,
                                       void* stream) {
  return transfer<float, true>(Nf, Nc, Nelements, elementList, GlobalToLocal, P, qf, qc, stream);
}
extern "C" int libp_mg_prolong_hex_f64(int Nf, int Nc, int Nelements, const int* elementList,
                                       const int* GlobalToLocalC, const double* P, const double* qc, double* qf,
                                       void* stream) {
  return transfer<double, false>(Nf, Nc, Nelements, elementList, GlobalToLocalC, P, qc, qf, stream);
}
extern "C" int libp_mg_prolong_hex_f32(int Nf, int Nc, int Nelements, const int* elementList,
                                       const int* GlobalToLocalC, const float* P, const float* qc, float* qf,
                                       void* stream) {
  return transfer<float, false>(Nf, Nc, Nelements, elementList, GlobalToLocalC, P, qc, qf, stream);
}

extern "C" int libp_mg_coarsen_weighted_hex_f64(int Nf, int Nc, int Nelements, const int* elementList,
                                                const int* GlobalToLocal, const double* P, const double* weight,
                                                const double* qf, double* qc, void* stream) {
  if (!weight) return arg_error("mg_coarsen_weighted", "null pointer");
  return transfer<double, true>(Nf, Nc, Nelements, elementList, GlobalToLocal, P, qf, qc, stream, weight);
}
extern "C" int libp_mg_coarsen_weighted_hex_f32(int Nf, int Nc, int Nelements, const int* elementList,
                                                const int* GlobalToLocal, const float* P, const float* weight,
                                                const float* qf, float* qc, void* stream) {
  if (!weight) return arg_error("mg_coarsen_weighted", "null pointer");
  return transfer<float, true>(Nf, Nc, Nelements, elementList, GlobalToLocal, P, qf, qc, stream, weight);
}
