// Matrix-free C0 hex stiffness + mass operator for gfx950.
//
// The operator of solvers/elliptic/okl/ellipticAxHex3D.okl:156-295. A workgroup
// takes NE elements and alternates two ways of holding their nodes:
//  * flat: thread t holds the nodes t, t + T, ... of the group in local order.
//    The index map, the values, the geometric factors and the result are read
//    and written this way, so every access to HBM is a run of consecutive
//    entries whatever the degree, and lanes idle only past the end of a group;
//  * pencils: a thread holds one whole line of Nq nodes along r, s or t and
//    contracts it with D. D[o][m] is then the same for every lane, so it comes
//    through scalar loads and each node costs one LDS read and one LDS write
//    per direction.
// The steps: load q (flat) -> D along r, s, t (pencils) -> the geometric factors
// (flat) -> D^T along r, s, t (pencils) -> sum and store (flat), with q, r and s
// parts in three LDS arrays; the t contraction, and every D^T, runs in place.
//
// What bounds it: HBM, 60 (lambda = 0) or 68 bytes per node in FP64. All the
// factors of a thread's nodes are requested before the first barrier, so they
// arrive while the contractions run. A thread tile per k-plane, with D in LDS
// (the form this kernel replaces), made 8 Nq LDS reads per node and left
// 64 - Nq^2 mod 64 lanes idle; here lanes idle only past the last pencil and the
// last node of a group. Partial Ax of ~10M local nodes, lambda = 1, curved boxes,
// microseconds before -> now (TB/s of those bytes now):
//   N        1        2        3        4        5        6        7
//   FP64  211->116 237->119 117->115 169->118 150->121 144->124   131
//         (6.0)    (5.9)    (6.3)    (6.1)    (6.1)    (6.0)   (the tile)
//   FP32  159->61  147->62   93->63  116->65   87->64   91->69   73->67
//   N        8        9       10       11       12       13       14
//   FP64  144->121 181->127 146->137 204->123 166->147 204->124 203->145
//         (6.1)    (6.2)    (5.8)    (6.1)    (5.5)    (5.5)    (4.8)
//   FP32   93->67   90->72   84->73  106->69  116->80  107->72  101->80
// (N = 15 FP32: 98->65; N = 7 in FP64 keeps the thread tile, see
// ax_hex_tile_kernel; N = 15 in FP64 runs on the matrix cores, ax_hex_mfma.hip.)
// At N >= 12 in FP64 the LDS of an element (53-81 KB) leaves two or three workgroups
// per CU, too few to cover the phases without loads.
//
// Further:
//  * elements run in natural order: brick or XCD-contiguous orderings that cut
//    q re-fetch were all slower (they break the sequential page streams of
//    the dominant arrays);
//  * the E-vector result is written with non-temporal stores (it is consumed
//    by the gather kernel, not re-read by this one);
//  * lambda = 0 (the Poisson operator) runs an instance that does not read wJ
//    (the reference reads it whatever lambda is): the mass term is +-0 in both,
//    so the result is the same to the bit, and the kernel streams 60 instead of
//    68 bytes per local node.
//
// The split output form (OUT = 1) serves the whole C0 operator A = Q^T A_L Q
// (ellipticOperator.cpp:29-107) without writing the full E-vector: a node
// interior to its element has exactly one copy, so its gathered row is the
// element's value itself and is stored straight into the gathered output
// (0 + a = a: bit-identical to the gather). Only the element-boundary ("face")
// nodes go to a compact face E-vector, e * Nface + faceIndex(n), which a gather
// over the shared rows alone then sums (ogs_gather_face_kernel). With PAP, the
// block also forms its share of p.Ap over the interior rows.
#include <type_traits>

#include "reduce.hpp"

namespace libp_amd {

// Elements per workgroup NE, threads T, waves per SIMD to compile for, rows of D
// per pass of a contraction's loop (UF: all of them while they fit the scalar
// registers, two or three above), the nodes of a thread whose factors are
// requested before the first barrier (GP), and whether the factors are read past the
// caches. The shapes are the fastest of a sweep at ~10M nodes, lambda 0 and 1, unless that
// one was slower than the tile at another size between 20 thousand and 55M nodes: more
// threads per element, or all of D, at Nq = 3, 6 and 7 (FP32, 14^3 elements of Nq = 3
// 4.6 -> 3.9 us, the tile 4.0; 4^3 of Nq = 7 7.3 -> 6.3, the tile 6.9).
// What is left, each against the tile:
//  * Nq = 8 in FP32, the kernel called over and over with nothing between: from 16M nodes 6 to
//    14% slower (33^3, lambda = 0, 124 us against 117). Two elements per workgroup mend
//    that (110 us) and lose where the kernel is used, between the gathers of a smoother:
//    32^3, three handles in turn, 587 us per smoothing against 580, 40^3 1191 against 1146
//    (the tile 581 and 1167; in the trace of one handle the Ax 104 us in both, the tile 120);
//  * 10^3 elements of Nq = 11 (FP64, lambda = 1) 23.2 us and 21.9: their workgroups take two
//    rounds where the tile's took one, and shapes with four workgroups per CU lose 2 to 6%
//    from 4M nodes on (likewise the PAP form of Nq = 13, 49.8 and 46.4);
//  * 0.3 us at Nq = 2 below 5000 elements.
// The rules of the sweep:
//  * T is a multiple of 256 where an element has over 64 pencils: five to seven waves
//    per workgroup spread unevenly over the four SIMDs (Nq = 12, 320 threads: 264 us
//    against 123 with 256);
//  * GP: at Nq = 14 and 15 all factors at once need over 128 registers, which leaves
//    one workgroup per CU (Nq = 14: 188 us against 124 with four of six nodes early,
//    the rest requested after the contractions);
//  * cached factor reads where a wave's requests are shorter than a cache line, which
//    several of them then share (Nq = 2 in FP32: 88 -> 61 us, Nq = 3 in FP64:
//    135 -> 120), and in FP32 wherever that measured faster at 10M and 50M nodes (up
//    to 10%; at Nq = 8 they are slower by 18% at 57M nodes).
template <int Nq, typename R>
struct AxShape;
template <int NE_, int T_, int W_, int UF_, int GP_, bool NT_>
struct AxShapeOf {
  static constexpr int NE = NE_, threads = T_, waves = W_, UF = UF_, GP = GP_;
  static constexpr bool NT = NT_;
};
constexpr int ALL = 1 << 20;
template <> struct AxShape<2, double> : AxShapeOf<32, 128, 2, 2, ALL, false> {};
template <> struct AxShape<3, double> : AxShapeOf<8, 128, 2, 3, ALL, false> {};
template <> struct AxShape<4, double> : AxShapeOf<4, 64, 2, 4, ALL, true> {};
template <> struct AxShape<5, double> : AxShapeOf<4, 256, 2, 5, ALL, true> {};
template <> struct AxShape<6, double> : AxShapeOf<4, 256, 2, 6, ALL, true> {};
template <> struct AxShape<7, double> : AxShapeOf<2, 256, 2, 7, ALL, true> {};
template <> struct AxShape<9, double> : AxShapeOf<1, 256, 2, 3, ALL, true> {};
template <> struct AxShape<10, double> : AxShapeOf<1, 256, 2, 5, ALL, true> {};
template <> struct AxShape<11, double> : AxShapeOf<1, 256, 2, 2, ALL, true> {};
template <> struct AxShape<12, double> : AxShapeOf<1, 256, 2, 3, ALL, true> {};
template <> struct AxShape<13, double> : AxShapeOf<1, 256, 2, 1, ALL, true> {};
template <> struct AxShape<14, double> : AxShapeOf<1, 512, 4, 2, 4, true> {};
template <> struct AxShape<15, double> : AxShapeOf<1, 512, 4, 1, 4, true> {};
template <> struct AxShape<16, double> : AxShapeOf<1, 512, 2, 2, ALL, true> {};  // the E-vector form only
template <> struct AxShape<2, float> : AxShapeOf<64, 128, 2, 2, ALL, false> {};
template <> struct AxShape<3, float> : AxShapeOf<16, 256, 2, 3, ALL, false> {};
template <> struct AxShape<4, float> : AxShapeOf<8, 128, 2, 4, ALL, true> {};
template <> struct AxShape<5, float> : AxShapeOf<4, 256, 2, 5, ALL, false> {};
template <> struct AxShape<6, float> : AxShapeOf<4, 256, 2, 6, ALL, false> {};
template <> struct AxShape<7, float> : AxShapeOf<4, 256, 2, 7, ALL, false> {};
template <> struct AxShape<8, float> : AxShapeOf<1, 128, 2, 2, ALL, true> {};
template <> struct AxShape<9, float> : AxShapeOf<1, 256, 2, 3, ALL, false> {};
template <> struct AxShape<10, float> : AxShapeOf<1, 256, 2, 2, ALL, false> {};
template <> struct AxShape<11, float> : AxShapeOf<1, 256, 2, 2, ALL, false> {};
template <> struct AxShape<12, float> : AxShapeOf<1, 512, 2, 2, ALL, true> {};
template <> struct AxShape<13, float> : AxShapeOf<1, 512, 2, 2, ALL, false> {};
template <> struct AxShape<14, float> : AxShapeOf<1, 256, 2, 2, ALL, false> {};
template <> struct AxShape<15, float> : AxShapeOf<1, 512, 4, 2, ALL, false> {};
template <> struct AxShape<16, float> : AxShapeOf<1, 512, 4, 4, ALL, false> {};

// The waves and GP of an instance, elsewhere those of the shape (NE and threads stay: the
// launcher counts blocks by them). At Nq = 13 the mass term takes the E-vector form past 168
// registers, two workgroups per CU; with seven of nine nodes early three fit (9^3 elements,
// lambda = 1, 34.5 -> 27.8 us, the tile 31.7; 15^3 118 -> 106). The list form keeps ALL (29^3
// 716 against 803 us), and the split form (862 against 950). At Nq = 11 the split form is faster with
// four workgroups per CU (10^3 elements, lambda 0 / 1, 27.9 / 28.9 -> 25.3 / 26.6 us, the
// tile 25.4 / 25.1; 18^3 112 / 122 -> 106 / 116), the E-vector form is not (95 -> 98).
template <int Nq, typename R, int OUT, bool LAM, bool LIST>
struct AxInstance : AxShape<Nq, R> {};
template <> struct AxInstance<13, double, 0, true, false> : AxShapeOf<1, 256, 3, 1, 7, true> {};
template <bool LAM> struct AxInstance<11, double, 1, LAM, false> : AxShapeOf<1, 256, 4, 2, 4, true> {};

// Number of element-boundary nodes of an Nq^3 element, and the position of
// node (i,j,k) among them in local order (the node index minus the interior
// nodes before it).
__host__ __device__ constexpr int hex_face_nodes(int Nq) { return Nq * Nq * Nq - (Nq - 2) * (Nq - 2) * (Nq - 2); }
__device__ inline int interior_before(int x, int Nq) { return min(max(x - 1, 0), Nq - 2); }
__device__ inline bool hex_interior(int i, int j, int k, int Nq) {
  return i > 0 && i < Nq - 1 && j > 0 && j < Nq - 1 && k > 0 && k < Nq - 1;
}
__device__ inline int hex_face_index(int i, int j, int k, int Nq) {
  const int n = i + j * Nq + k * Nq * Nq;
  const bool kin = k > 0 && k < Nq - 1, jin = j > 0 && j < Nq - 1;
  const int before = interior_before(k, Nq) * (Nq - 2) * (Nq - 2) +
                     (kin ? interior_before(j, Nq) * (Nq - 2) + (jin ? interior_before(i, Nq) : 0) : 0);
  return n - before;
}

// LDS layout of a group's nodes: rows of P entries, planes of S. Odd Nq needs no
// padding (pencils of neighbouring lanes start on different banks); for even Nq
// the paddings with the fewest conflicts over all the accesses of an element.
template <int Nq>
struct AxLds {
  static constexpr int P = (Nq == 4 || Nq == 16) ? Nq + 1 : Nq;
  static constexpr int S = Nq * P + (Nq == 8 ? 5 : Nq == 12 ? 1 : Nq == 14 ? 3 : 0);
  __device__ static inline int node(const int n) {  // node n of the group, local order
    return S == Nq * Nq ? n : (n / (Nq * Nq)) * S + (n / Nq % Nq) * P + n % Nq;
  }
  // pencil p along r (DIR 0), s (1) or t (2): its first entry and its stride
  template <int DIR>
  static constexpr int stride = DIR == 0 ? 1 : DIR == 1 ? P : S;
  template <int DIR>
  __device__ static inline int pencil(const int p) {
    if (DIR == 0) return S == Nq * P ? p * P : (p / Nq) * S + (p % Nq) * P;
    if (DIR == 1) return (p / Nq) * S + p % Nq;
    const int ji = p % (Nq * Nq);
    return (p / (Nq * Nq)) * Nq * S + (ji / Nq) * P + ji % Nq;
  }
};

// dst = D src (TR: D^T src) along one direction of the group's NE elements, by
// threads tid = 0..T-1. A thread reads its whole pencil before it writes it, so
// dst may be src. The loop over the rows of D takes UF at a time: fully unrolled
// at Nq >= 10 the rows overflow the scalar registers into vector ones.
template <int Nq, int NE, int T, int UF, int DIR, bool TR, typename R>
__device__ inline void ax_contract(const R* __restrict__ D, const R* src, R* dst, const int tid) {
#pragma clang fp contract(on)
  using L = AxLds<Nq>;
  constexpr int NP = NE * Nq * Nq, ROUNDS = (NP + T - 1) / T, st = L::template stride<DIR>;
#pragma unroll
  for (int u = 0; u < ROUNDS; ++u) {
    const int p = tid + u * T;
    if ((u + 1) * T <= NP || p < NP) {
      const int b = L::template pencil<DIR>(p);
      R x[Nq];
      if (TR) {  // out[o] = sum_m D[m][o] src[m], one row of D at a time
#pragma unroll
        for (int o = 0; o < Nq; ++o) x[o] = 0;
#pragma unroll UF
        for (int m = 0; m < Nq; ++m) {
          const R v = src[b + m * st];
#pragma unroll
          for (int o = 0; o < Nq; ++o) x[o] += D[m * Nq + o] * v;
        }
#pragma unroll
        for (int o = 0; o < Nq; ++o) dst[b + o * st] = x[o];
      } else {
#pragma unroll
        for (int m = 0; m < Nq; ++m) x[m] = src[b + m * st];
#pragma unroll UF
        for (int o = 0; o < Nq; ++o) {
          R acc = 0;
#pragma unroll
          for (int m = 0; m < Nq; ++m) acc += D[o * Nq + m] * x[m];
          dst[b + o * st] = acc;
        }
      }
    }
  }
}

// MODE 0: q is a gathered vector indexed through GlobalToLocal (-1 -> 0).
// MODE 1: q is an E-vector (element-local input, no gather).
// OUT 0: Aq is the E-vector; with PAP (MODE 0, the PCG form), each block
// also stores sum over its local nodes of q_L * (A_L q)_L, which summed over
// all blocks is p.Ap = p^T Q^T A_L Q p for a gathered q = p, and the kernel
// returns at once while scal[8] (STOP) is set. OUT 1 (MODE 0 only): interior nodes go to the
// gathered Ag, element-boundary nodes to the face E-vector Aq; PAP adds one
// partial of sum q Ag over the interior rows per block.
// LIST: the elements are elementList[0..Nelements); without it they are
// 0..Nelements-1 and the group's entries are one block with 32-bit offsets.
// A group past the end repeats its last element: the same loads, the same
// values stored by several threads of the one block.
template <int Nq, typename R, int MODE, int OUT, bool PAP, bool LAM, bool LIST>
__global__ void __launch_bounds__((AxShape<Nq, R>::threads))
    __attribute__((amdgpu_waves_per_eu((AxInstance<Nq, R, OUT, LAM, LIST>::waves))))
    ax_hex_kernel(const int Nelements, const int* __restrict__ elementList, const int* __restrict__ G2L,
                  const R* __restrict__ wJ, const R* __restrict__ ggeo, const R* __restrict__ D, const R lambda,
                  const R* __restrict__ q, R* __restrict__ Aq, R* __restrict__ Ag, double* __restrict__ pap,
                  const int* __restrict__ fslot, const double* __restrict__ scal) {
  // a*b + c contracts only within one source expression, so every
  // instantiation (E-vector, split, split with p.Ap) rounds alike: with
  // contraction across expressions the backend may fuse x*y + z*w as
  // fma(x, y, z*w) in one instantiation and fma(z, w, x*y) in another
#pragma clang fp contract(on)
  using S = AxInstance<Nq, R, OUT, LAM, LIST>;
  using L = AxLds<Nq>;
  using offset = std::conditional_t<LIST, size_t, unsigned>;
  constexpr int NE = S::NE, T = S::threads, UF = S::UF, GP = S::GP;
  constexpr int Np = Nq * Nq * Nq, NN = NE * Np, UN = (NN + T - 1) / T, SA = NE * Nq * L::S;
  // r and s pencils side by side on the two halves of the block where both fit
  constexpr bool PAIR = T % 128 == 0 && NE * Nq * Nq <= T / 2;
  __shared__ R s_q[SA], s_r[SA], s_s[SA];
  if (PAP && OUT == 0 && scal[8] != 0.0) return;  // a PCG step after convergence (STOP)
  const int t = threadIdx.x;
  const bool upper = PAIR && __builtin_amdgcn_readfirstlane(t) >= T / 2;
  const int e0 = blockIdx.x * NE;
  const int last = Nelements - 1 - e0;
  const auto load = [](const auto* p) { return S::NT ? __builtin_nontemporal_load(p) : *p; };

  // node u of this thread: n = t + u T of the group (clamped past its end), of element el
  const size_t first = LIST ? 0 : (size_t)e0;
  const int* g2lb = G2L + first * Np;
  const R* gb = ggeo + first * 6 * Np;
  const R* wb = wJ + first * Np;
  const auto in = [t](const int u) { return (u + 1) * T <= NN || t + u * T < NN; };
  offset el[UN], off[UN];
  R v[UN], G[6][UN], mass[UN];
  int ids[UN], at[UN];
#pragma unroll
  for (int u = 0; u < UN; ++u) {
    const int n = min(t + u * T, NN - 1);
    at[u] = L::node(n);
    // with NE = 1, min(0, last) is 0, but not to the compiler: at Nq >= 15 in FP32 it then keeps
    // one 32-bit offset per node beside scalar bases instead of many precomputed addresses
    // (Nq = 16: 116 registers instead of 147, 515 -> 325 us at 50M nodes); elsewhere it costs registers
    const int es = (NE > 1) ? min(n / Np, last) : (sizeof(R) == 4 && Nq >= 15) ? min(0, last) : 0;
    el[u] = LIST ? (offset)elementList[e0 + es] : (offset)es;
    off[u] = el[u] * Np + ((NE == 1) ? n : n % Np);
    if (MODE == 0) ids[u] = load(g2lb + off[u]);
    if (MODE == 1) v[u] = load(q + first * Np + off[u]);
  }
  if (MODE == 0) {
    // unconditional loads (a masked node, id -1, reads q[0] and takes 0): a load
    // under (id >= 0) compiles to a branch that waits for each load in turn
#pragma unroll
    for (int u = 0; u < UN; ++u) v[u] = q[max(ids[u], 0)];
  }
  // LAM = false (lambda = 0): wJ is not read; lambda * wJ * q is +-0 with any finite wJ
  if (LAM) {
#pragma unroll
    for (int u = 0; u < UN; ++u) mass[u] = load(wb + off[u]);
  }
  const auto loadG = [&](const int u) {
#pragma unroll
    for (int g = 0; g < 6; ++g) G[g][u] = load(gb + g * Np + (off[u] + 5 * el[u] * Np));
  };
#pragma unroll
  for (int u = 0; u < UN && u < GP; ++u) loadG(u);
#pragma unroll
  for (int u = 0; u < UN; ++u) {
    if (MODE == 0) v[u] = (ids[u] >= 0) ? v[u] : R(0);
    if (in(u)) s_q[at[u]] = v[u];
    if (LAM) mass[u] = mass[u] * lambda * v[u];
  }
  __syncthreads();

  if (PAIR) {
    if (!upper)
      ax_contract<Nq, NE, T / 2, UF, 0, false>(D, s_q, s_r, t);
    else
      ax_contract<Nq, NE, T / 2, UF, 1, false>(D, s_q, s_s, t - T / 2);
  } else {
    ax_contract<Nq, NE, T, UF, 0, false>(D, s_q, s_r, t);
    ax_contract<Nq, NE, T, UF, 1, false>(D, s_q, s_s, t);
  }
  __syncthreads();
  ax_contract<Nq, NE, T, UF, 2, false>(D, s_q, s_q, t);
#pragma unroll
  for (int u = GP; u < UN; ++u) loadG(u);
  __syncthreads();

#pragma unroll
  for (int u = 0; u < UN; ++u)
    if (in(u)) {
      const int a = at[u];
      const R qr = s_r[a], qs = s_s[a], qt = s_q[a];
      s_r[a] = G[0][u] * qr + G[1][u] * qs + G[2][u] * qt;
      s_s[a] = G[1][u] * qr + G[3][u] * qs + G[4][u] * qt;
      s_q[a] = G[2][u] * qr + G[4][u] * qs + G[5][u] * qt;
    }
  __syncthreads();

  if (PAIR) {
    if (!upper)
      ax_contract<Nq, NE, T / 2, UF, 0, true>(D, s_r, s_r, t);
    else
      ax_contract<Nq, NE, T / 2, UF, 1, true>(D, s_s, s_s, t - T / 2);
  } else {
    ax_contract<Nq, NE, T, UF, 0, true>(D, s_r, s_r, t);
    ax_contract<Nq, NE, T, UF, 1, true>(D, s_s, s_s, t);
  }
  ax_contract<Nq, NE, T, UF, 2, true>(D, s_q, s_q, t);
  __syncthreads();

  double acc = 0;
#pragma unroll
  for (int u = 0; u < UN; ++u)
    if (in(u)) {
      const int n = t + u * T, a = at[u];
      R o = s_r[a] + s_s[a];
      o = o + s_q[a];
      if (LAM) o = o + mass[u];
      const bool own = NE == 1 || n / Np <= last;  // not a repeat of the last element
      if (OUT == 0) {
        __builtin_nontemporal_store(o, Aq + first * Np + off[u]);
        if (PAP && own) acc += (double)v[u] * (double)o;
      } else {
        constexpr int Nface = hex_face_nodes(Nq);
        const int ln = (NE == 1) ? n : n % Np;
        const int i = ln % Nq, j = ln / Nq % Nq, k = ln / (Nq * Nq);
        if (hex_interior(i, j, k, Nq)) {
          if (ids[u] >= 0) Ag[ids[u]] = o;
          if (PAP && own) acc += (double)v[u] * (double)o;
        } else {
          const size_t f = (first + el[u]) * Nface + hex_face_index(i, j, k, Nq);
          if (fslot)  // slot layout: the copy's place in the row-ordered copy list
            Aq[__builtin_nontemporal_load(fslot + f)] = o;
          else
            __builtin_nontemporal_store(o, Aq + f);
        }
      }
    }
  if constexpr (PAP) {
    __shared__ double s_w[16];
    const double b = block_sum(acc, s_w);
    if (t == 0) pap[blockIdx.x] = b;
  }
}

// The FP64 operator at N = 7 as a thread tile: one 8 x 8 tile (a wavefront) per
// element, each thread holding the k-pencil q(i,j,0:7) in registers, the r and s
// contractions through LDS plane by plane, NE = 4 elements per workgroup. Here a
// wavefront is an element's plane, so the tile has neither idle lanes nor short
// requests, and it stays the faster form where operators of several handles run
// on their own streams: 48^3 elements, lambda = 0, Ax + gather of three handles in
// turn 822 us per operator against 858-875 us for every shape of the pencil kernel
// (one handle alone: 812 against 805 us, the Ax without its gather 614 against
// 587 us). Four waves per SIMD: a five-wave target (96 VGPRs) took 1168 us.
// Every element slot of a block is a real element: the launcher runs the whole
// blocks first and the remainder with NE = 1 (element offset e0); a clamped tail
// inside this kernel roughly quadruples its register use.
template <int NE, int MODE, int OUT, bool PAP, bool LAM>
__global__ void __launch_bounds__(NE * 64) __attribute__((amdgpu_waves_per_eu(4, 8)))
    ax_hex_tile_kernel(const int e0, const int* __restrict__ elementList, const int* __restrict__ G2L,
                       const double* __restrict__ wJ, const double* __restrict__ ggeo, const double* __restrict__ D,
                       const double lambda, const double* __restrict__ q, double* __restrict__ Aq,
                       double* __restrict__ Ag, double* __restrict__ pap, const int pap0,
                       const int* __restrict__ fslot, const double* __restrict__ scal) {
  // a*b + c contracts only within one source expression, so every
  // instantiation (E-vector, split, split with p.Ap) rounds alike: with
  // contraction across expressions the backend may fuse x*y + z*w as
  // fma(x, y, z*w) in one instantiation and fma(z, w, x*y) in another
#pragma clang fp contract(on)
  constexpr int Nq = 8, NqNq = 64, Np = 512, threads = NE * NqNq;
  __shared__ double s_D[Nq][Nq + 1];
  __shared__ double s_q[NE][Nq][Nq + 1];
  __shared__ double s_Gqr[NE][Nq][Nq + 1];
  __shared__ double s_Gqs[NE][Nq][Nq + 1];
  __shared__ int s_id[OUT == 1 ? NE : 1][OUT == 1 ? Nq : 1][OUT == 1 ? NqNq : 1];
  __shared__ double s_out[OUT == 1 ? NE : 1][OUT == 1 ? Nq : 1][OUT == 1 ? NqNq : 1];

  if (scal != nullptr && scal[8] != 0.0) return;  // a PCG step after convergence (STOP)
  const int t = threadIdx.x;
  const int es = (NE == 1) ? 0 : t / NqNq;
  const int ij = (NE == 1) ? t : t - es * NqNq;
  const int i = ij % Nq;
  const int j = ij / Nq;
  const int eIdx = e0 + blockIdx.x * NE + es;
  const int element = elementList ? elementList[eIdx] : eIdx;

  for (int n = t; n < NqNq; n += threads) s_D[n / Nq][n % Nq] = D[n];

  double r_q[Nq], r_Aq[Nq];
  const size_t base = (size_t)element * Np + ij;
  if (MODE == 0) {
    // all Nq index loads in flight, then all Nq value loads: the value loads are
    // unconditional (a masked node, id -1, reads q[0] and takes 0), since a load
    // under (id >= 0) compiles to a branch that waits for each load in turn
    int ids[Nq];
#pragma unroll
    for (int k = 0; k < Nq; ++k) ids[k] = __builtin_nontemporal_load(G2L + base + k * NqNq);
#pragma unroll
    for (int k = 0; k < Nq; ++k) {
      const double v = q[max(ids[k], 0)];
      r_q[k] = (ids[k] >= 0) ? v : 0.0;
      if (OUT == 1) s_id[es][k][ij] = ids[k];
    }
  } else {
#pragma unroll
    for (int k = 0; k < Nq; ++k) r_q[k] = __builtin_nontemporal_load(q + base + k * NqNq);
  }
#pragma unroll
  for (int k = 0; k < Nq; ++k) r_Aq[k] = 0;
  const double* gb = ggeo + (size_t)element * 6 * Np + ij;
  const double* wb = wJ + (size_t)element * Np + ij;
  __syncthreads();

#pragma unroll
  for (int k = 0; k < Nq; ++k) {
    const double G00 = __builtin_nontemporal_load(gb + 0 * Np + k * NqNq);
    const double G01 = __builtin_nontemporal_load(gb + 1 * Np + k * NqNq);
    const double G02 = __builtin_nontemporal_load(gb + 2 * Np + k * NqNq);
    const double G11 = __builtin_nontemporal_load(gb + 3 * Np + k * NqNq);
    const double G12 = __builtin_nontemporal_load(gb + 4 * Np + k * NqNq);
    const double G22 = __builtin_nontemporal_load(gb + 5 * Np + k * NqNq);
    // LAM = false (lambda = 0): wJ is not read; lambda * GwJ * q is +-0 with either GwJ
    const double GwJ = LAM ? __builtin_nontemporal_load(wb + k * NqNq) : 0.0;

    s_q[es][j][i] = r_q[k];
    double qt = 0;
#pragma unroll
    for (int m = 0; m < Nq; ++m) qt += s_D[k][m] * r_q[m];
    __syncthreads();

    double qr = 0, qs = 0;
#pragma unroll
    for (int m = 0; m < Nq; ++m) {
      qr += s_D[i][m] * s_q[es][j][m];
      qs += s_D[j][m] * s_q[es][m][i];
    }
    s_Gqs[es][j][i] = G01 * qr + G11 * qs + G12 * qt;
    s_Gqr[es][j][i] = G00 * qr + G01 * qs + G02 * qt;
    const double Gqt = G02 * qr + G12 * qs + G22 * qt;
    double Auk = GwJ * lambda * r_q[k];
    __syncthreads();

#pragma unroll
    for (int m = 0; m < Nq; ++m) {
      Auk += s_D[m][j] * s_Gqs[es][m][i];
      r_Aq[m] += s_D[k][m] * Gqt;
      Auk += s_D[m][i] * s_Gqr[es][j][m];
    }
    r_Aq[k] += Auk;
  }

  if (OUT == 0) {
    double* out = Aq + base;
#pragma unroll
    for (int k = 0; k < Nq; ++k) __builtin_nontemporal_store(r_Aq[k], out + k * NqNq);
    if constexpr (PAP) {
      double acc = 0;
#pragma unroll
      for (int k = 0; k < Nq; ++k) acc += (double)r_q[k] * (double)r_Aq[k];
      __shared__ double s_w[NE];
      const double b = block_sum(acc, s_w);
      if (t == 0) pap[pap0 + blockIdx.x] = b;
    }
  } else {
    // The results go through LDS first: stored with the regular pattern of the
    // E-vector store, the registers die there. Scattering straight from the
    // registers (one branch and address per k) made the compiler spill ~500
    // VGPRs at N=7.
    constexpr int Nface = hex_face_nodes(Nq);
    double acc = 0;
#pragma unroll
    for (int k = 0; k < Nq; ++k) {
      s_out[es][k][ij] = r_Aq[k];
      if (PAP) acc += hex_interior(i, j, k, Nq) ? (double)r_q[k] * (double)r_Aq[k] : 0.0;
    }
    __syncthreads();
    double* fout = Aq + (size_t)element * Nface;
    for (int k = 0; k < Nq; ++k) {
      const double v = s_out[es][k][ij];
      if (hex_interior(i, j, k, Nq)) {
        const int id = s_id[es][k][ij];
        if (id >= 0) Ag[id] = v;
      } else {
        const int fi = hex_face_index(i, j, k, Nq);
        if (fslot)  // slot layout: the copy's place in the row-ordered copy list
          Aq[__builtin_nontemporal_load(fslot + (size_t)element * Nface + fi)] = v;
        else
          __builtin_nontemporal_store(v, fout + fi);
      }
    }
    if constexpr (PAP) {
      __shared__ double s_w[NE];
      const double b = block_sum(acc, s_w);
      if (t == 0) pap[pap0 + blockIdx.x] = b;
    }
  }
}

// N = 7 in FP64 runs as a tile: NE = 4 elements per workgroup, the remainder one each
constexpr int AX_TILE_NE = 4;
template <int Nq, typename R>
constexpr bool ax_tile = Nq == 8 && sizeof(R) == 8;

template <int Nq, typename R>
static int ax_blocks(int Nelements) {
  if (Nelements <= 0) return 0;
  if constexpr (ax_tile<Nq, R>)
    return Nelements / AX_TILE_NE + Nelements % AX_TILE_NE;
  else
    return (Nelements + AxShape<Nq, R>::NE - 1) / AxShape<Nq, R>::NE;
}

template <typename R>
struct AxArgs {
  int Nelements;
  const int *elementList, *G2L;
  const R *wJ, *ggeo, *D;
  R lambda;
  const R* q;
  R *Aq, *Ag;
  double* pap;
  const int* fslot;
  const double* scal;
  hipStream_t stream;
};

template <int MODE, int OUT, bool PAP, bool LAM>
static void launch_ax_tile(const AxArgs<double>& a) {
  const int full = a.Nelements / AX_TILE_NE, rest = a.Nelements % AX_TILE_NE;
  if (full > 0)
    hipLaunchKernelGGL((ax_hex_tile_kernel<AX_TILE_NE, MODE, OUT, PAP, LAM>), dim3(full), dim3(AX_TILE_NE * 64), 0,
                       a.stream, 0, a.elementList, a.G2L, a.wJ, a.ggeo, a.D, a.lambda, a.q, a.Aq, a.Ag, a.pap, 0,
                       a.fslot, a.scal);
  if (rest > 0)
    hipLaunchKernelGGL((ax_hex_tile_kernel<1, MODE, OUT, PAP, LAM>), dim3(rest), dim3(64), 0, a.stream,
                       full * AX_TILE_NE, a.elementList, a.G2L, a.wJ, a.ggeo, a.D, a.lambda, a.q, a.Aq, a.Ag, a.pap,
                       full, a.fslot, a.scal);
}

// lambda = 0 (the Poisson operator) takes the instances that do not read wJ:
// the mass term lambda * wJ * q is +-0 in both, so the results are the same to
// the bit, and the kernel moves 8 (FP64) or 4 (FP32) bytes less per local node.
template <int Nq, typename R, int MODE, int OUT, bool PAP>
static int launch_ax(const AxArgs<R>& a, const char* where) {
  if (a.Nelements <= 0) return LIBP_OK;
  const bool lam = a.lambda != R(0);
  if constexpr (ax_tile<Nq, R>) {
    if (lam)
      launch_ax_tile<MODE, OUT, PAP, true>(a);
    else
      launch_ax_tile<MODE, OUT, PAP, false>(a);
  } else {
    const auto launch = [&](auto kernel) {
      hipLaunchKernelGGL(kernel, dim3(ax_blocks<Nq, R>(a.Nelements)), dim3(AxShape<Nq, R>::threads), 0, a.stream,
                         a.Nelements, a.elementList, a.G2L, a.wJ, a.ggeo, a.D, a.lambda, a.q, a.Aq, a.Ag, a.pap,
                         a.fslot, a.scal);
    };
    if (a.elementList && lam)
      launch(ax_hex_kernel<Nq, R, MODE, OUT, PAP, true, true>);
    else if (a.elementList)
      launch(ax_hex_kernel<Nq, R, MODE, OUT, PAP, false, true>);
    else if (lam)
      launch(ax_hex_kernel<Nq, R, MODE, OUT, PAP, true, false>);
    else
      launch(ax_hex_kernel<Nq, R, MODE, OUT, PAP, false, false>);
  }
  return launch_status(where);
}

// p.Ap from the partials of the PCG-form Ax kernel, summed in block order,
// then alpha = s[RDOTZ1] / p.Ap (linearSolverPCG.cpp:134-140).
__global__ void __launch_bounds__(1024) ax_pap_finish_kernel(const int nb, double* __restrict__ s,
                                                             const double* __restrict__ part) {
  __shared__ double s_w[16];
  if (s[8] != 0.0) return;
  // 27,648 partials at 48^3, N=7: one round of 32 loads per thread (7.3 us with 8)
  const double pap = block_sum(strided_sum<32>(part, nb), s_w);
  if (threadIdx.x == 0) {
    s[4] = pap;
    s[2] = s[0] / pap;
  }
}

// Partial Ax of p (gathered, through GlobalToLocal) into the E-vector with
// p.Ap from the local nodes and alpha (MODE 0, OUT 0, PAP).
template <int Nq>
static int launch_ax_pap(const AxArgs<double>& a, double* s) {
  const int st = launch_ax<Nq, double, 0, 0, true>(a, "pcg_ax_hex_pap");
  if (st != LIBP_OK || a.Nelements <= 0) return st;
  hipLaunchKernelGGL(ax_pap_finish_kernel, dim3(1), dim3(1024), 0, a.stream, ax_blocks<Nq, double>(a.Nelements), s,
                     (const double*)a.pap);
  return launch_status("pcg_ax_hex_pap");
}

#define LIBP_AX_CASES_1_14                                                                                       \
  LIBP_AX_CASE(1) LIBP_AX_CASE(2) LIBP_AX_CASE(3) LIBP_AX_CASE(4) LIBP_AX_CASE(5) LIBP_AX_CASE(6) LIBP_AX_CASE(7) \
  LIBP_AX_CASE(8) LIBP_AX_CASE(9) LIBP_AX_CASE(10) LIBP_AX_CASE(11) LIBP_AX_CASE(12) LIBP_AX_CASE(13)             \
  LIBP_AX_CASE(14)

template <typename R, int MODE>
static int dispatch_ax(int N, int Nelements, const int* elist, const int* g2l, const R* wJ, const R* ggeo,
                       const R* D, R lambda, const R* q, R* Aq, void* stream) {
  if (!wJ || !ggeo || !D || !q || !Aq || (MODE == 0 && !g2l)) return arg_error("ax_hex", "null pointer");
  const AxArgs<R> a{Nelements, elist, g2l, wJ, ggeo, D, lambda, q, Aq, nullptr, nullptr, nullptr, nullptr,
                    as_stream(stream)};
  switch (N) {
#define LIBP_AX_CASE(NN) \
  case NN:               \
    return launch_ax<NN + 1, R, MODE, 0, false>(a, "ax_hex");
    LIBP_AX_CASES_1_14
#undef LIBP_AX_CASE
    case 15:
      // the gathered FP64 form on the matrix cores: 13^3 elements 182 us as pencils, 116 us there
      if constexpr (MODE == 0 && sizeof(R) == 8)
        return libp_ax_hex_partial_mfma_n15(Nelements, elist, g2l, wJ, ggeo, D, lambda, q, Aq, stream);
      else
        return launch_ax<16, R, MODE, 0, false>(a, "ax_hex");
    default:
      return arg_error("ax_hex", "polynomial degree must be in [1,15]");
  }
}

}  // namespace libp_amd

using namespace libp_amd;

extern "C" int libp_ax_hex_partial_f64(int N, int Nelements, const int* elementList, const int* GlobalToLocal,
                                       const double* wJ, const double* ggeo, const double* D, double lambda,
                                       const double* q, double* AqL, void* stream) {
  return dispatch_ax<double, 0>(N, Nelements, elementList, GlobalToLocal, wJ, ggeo, D, lambda, q, AqL, stream);
}

extern "C" int libp_ax_hex_partial_f32(int N, int Nelements, const int* elementList, const int* GlobalToLocal,
                                       const float* wJ, const float* ggeo, const float* D, float lambda,
                                       const float* q, float* AqL, void* stream) {
  return dispatch_ax<float, 0>(N, Nelements, elementList, GlobalToLocal, wJ, ggeo, D, lambda, q, AqL, stream);
}

extern "C" int libp_ax_hex_local_f64(int N, int Nelements, const double* wJ, const double* ggeo, const double* D,
                                     double lambda, const double* qL, double* AqL, void* stream) {
  return dispatch_ax<double, 1>(N, Nelements, nullptr, nullptr, wJ, ggeo, D, lambda, qL, AqL, stream);
}

extern "C" int libp_ax_hex_split_blocks(int N, int Nelements) {
  switch (N) {
#define LIBP_AX_CASE(NN) \
  case NN:               \
    return ax_blocks<NN + 1, double>(Nelements);
    LIBP_AX_CASES_1_14
#undef LIBP_AX_CASE
    case 15:  // the MFMA kernel of the PCG form: one partial per element
      return Nelements;
    default:
      return -1;
  }
}

extern "C" int libp_ax_hex_face_nodes(int N) { return (N >= 1 && N <= 15) ? hex_face_nodes(N + 1) : -1; }

extern "C" int libp_ax_hex_split_f64(int N, int Nelements, const int* elementList, const int* GlobalToLocal,
                                     const double* wJ, const double* ggeo, const double* D, double lambda,
                                     const double* q, double* Aq, double* AqFace, const int* faceSlots,
                                     double* papPartials, void* stream) {
  if (!GlobalToLocal || !wJ || !ggeo || !D || !q || !Aq || !AqFace) return arg_error("ax_hex_split", "null pointer");
  const AxArgs<double> a{Nelements, elementList, GlobalToLocal, wJ, ggeo, D, lambda, q, AqFace, Aq, papPartials,
                         faceSlots, nullptr, as_stream(stream)};
  switch (N) {
#define LIBP_AX_CASE(NN)                                                          \
  case NN:                                                                        \
    return papPartials ? launch_ax<NN + 1, double, 0, 1, true>(a, "ax_hex_split") \
                       : launch_ax<NN + 1, double, 0, 1, false>(a, "ax_hex_split");
    LIBP_AX_CASES_1_14
#undef LIBP_AX_CASE
    default:
      return arg_error("ax_hex_split", "polynomial degree must be in [1,14]");
  }
}

namespace libp_amd {
// ax_hex_mfma.hip: the N=15 MFMA kernel in its PCG form (p.Ap partials, STOP)
int launch_ax_mfma_n15_pap(int Nelements, const int* elementList, const int* G2L, const double* wJ,
                           const double* ggeo, const double* D, double lambda, const double* p, double* AqL,
                           double* part, const double* scal, hipStream_t st);
}  // namespace libp_amd

extern "C" int libp_pcg_ax_hex_pap_f64(int N, int Nelements, const int* elementList, const int* GlobalToLocal,
                                       const double* wJ, const double* ggeo, const double* D, double lambda,
                                       const double* p, double* AqL, double* papPartials, double* scalars,
                                       void* stream) {
  if (!GlobalToLocal || !wJ || !ggeo || !D || !p || !AqL || !papPartials || !scalars)
    return arg_error("pcg_ax_hex_pap", "null pointer");
  hipStream_t st = as_stream(stream);
  const AxArgs<double> a{Nelements, elementList, GlobalToLocal, wJ, ggeo, D, lambda, p, AqL, nullptr, papPartials,
                         nullptr, scalars, st};
  switch (N) {
#define LIBP_AX_CASE(NN) \
  case NN:               \
    return launch_ax_pap<NN + 1>(a, scalars);
    LIBP_AX_CASES_1_14
#undef LIBP_AX_CASE
    case 15: {  // the FP64 MFMA kernel, one element (and one partial) per workgroup
      if (Nelements <= 0) return LIBP_OK;
      const int rc = launch_ax_mfma_n15_pap(Nelements, elementList, GlobalToLocal, wJ, ggeo, D, lambda, p, AqL,
                                            papPartials, scalars, st);
      if (rc != LIBP_OK) return rc;
      hipLaunchKernelGGL(ax_pap_finish_kernel, dim3(1), dim3(1024), 0, st, Nelements, scalars,
                         (const double*)papPartials);
      return launch_status("pcg_ax_hex_pap");
    }
    default:
      return arg_error("pcg_ax_hex_pap", "polynomial degree must be in [1,15]");
  }
}

namespace libp_amd {
unsigned gather_jacobi_blocks(int Nrows);  // ogs.hip
int launch_gather_jacobi_fold(int Nrows, const int* rowStarts, const int* colIds, const double* AqL,
                              const double* invDiag, const double* p, double* x, double* r, double* z,
                              const double* s, double* part, int nbAx, const double* papPart, hipStream_t st);
int launch_update_p_fold(int N, int first, const double* z, double* p, const double* prev, double* cur, int nb,
                         const double* part, hipStream_t st);  // linalg.hip
}  // namespace libp_amd

extern "C" int libp_pcg_jacobi_iteration_folds(int N, int Nelements, int Nrows) {
  const int nbAx = libp_ax_hex_split_blocks(N, Nelements);
  return Nelements > 0 && Nrows > 0 && nbAx > 0 && nbAx <= PCG_FOLD_MAX && gather_jacobi_blocks(Nrows) <= PCG_FOLD_MAX;
}

// Three launches per iteration: each sum of partials is formed by the kernel that needs it.
// Small solves are bound by the latency of their launches (8^3 elements, N = 4: 2.8 + 5.1 +
// 3.4 + 6.1 + 3.5 us in five; 3.9 + 4.8 + 6.5 us in three). PCG_FOLD_MAX partials are what
// a block of 256 threads sums with four loads each; past it (16^3 elements at N = 4,
// 524,288 rows) the finishers' 7 us are a small share of an iteration and every block
// would read more than 8 KB of partials.
extern "C" int libp_pcg_jacobi_iteration_f64(int N, int Nelements, const int* elementList, const int* GlobalToLocal,
                                             const double* wJ, const double* ggeo, const double* D, double lambda,
                                             int Nrows, const int* rowStarts, const int* colIds,
                                             const double* invDiag, int it, double* p, double* AqL, double* x,
                                             double* r, double* z, double* papPartials, double* gatherPartials,
                                             double* states, void* stream) {
  if (!GlobalToLocal || !wJ || !ggeo || !D || !rowStarts || !colIds || !invDiag || !p || !AqL || !x || !r || !z ||
      !papPartials || !gatherPartials || !states || it < 0)
    return arg_error("pcg_jacobi_iteration", "null pointer or negative iteration");
  if (((uintptr_t)z & 15) || ((uintptr_t)p & 15)) return arg_error("pcg_jacobi_iteration", "p and z must be 16-byte aligned");
  if (!libp_pcg_jacobi_iteration_folds(N, Nelements, Nrows))
    return arg_error("pcg_jacobi_iteration", "degree out of range or too many partial sums");
  hipStream_t st = as_stream(stream);
  double* cur = states + 16 * (it & 1);
  int rc = launch_update_p_fold(Nrows, it == 0, z, p, states + 16 * ((it + 1) & 1), cur,
                                (int)gather_jacobi_blocks(Nrows), gatherPartials, st);
  if (rc != LIBP_OK) return rc;
  const AxArgs<double> a{Nelements, elementList, GlobalToLocal, wJ, ggeo, D, lambda, p, AqL, nullptr, papPartials,
                         nullptr, cur, st};
  switch (N) {
#define LIBP_AX_CASE(NN)                                                   \
  case NN:                                                                 \
    rc = launch_ax<NN + 1, double, 0, 0, true>(a, "pcg_jacobi_iteration"); \
    break;
    LIBP_AX_CASES_1_14
#undef LIBP_AX_CASE
    default:
      rc = launch_ax_mfma_n15_pap(Nelements, elementList, GlobalToLocal, wJ, ggeo, D, lambda, p, AqL, papPartials, cur,
                                  st);
  }
  if (rc != LIBP_OK) return rc;
  return launch_gather_jacobi_fold(Nrows, rowStarts, colIds, AqL, invDiag, p, x, r, z, cur, gatherPartials,
                                   libp_ax_hex_split_blocks(N, Nelements), papPartials, st);
}
