// Fused explicit step: the per-step Domain_d sequence regrouped into four
// kernels with one grid-wide dependency between each pair.
//
//   F1 element pass   x gather -> J -> vol                      (CalcElemVol)
//   F2 node pass      CSR sum of vol -> V_n, ANP ratio V_n/V0_n, nodal mass
//                                                  (CalcNodalVol,
//                                                   CalcNodalMassFromVol,
//                                                   calcElemPressure nodes)
//   F3 element pass   J and dH recomputed from x, strain rate and spin from
//                     the predicted v, ANP pressure, Jaumann + J2 return,
//                     internal and hourglass forces (f_elem - f_hg), added per
//                     node of the work-group's element cluster in LDS -> one
//                     partial sum per (cluster, node) slot
//                                                  (calcElemJAndDerivatives,
//                                                   calcElemStrainRates,
//                                                   calcElemPressure,
//                                                   CalcStressStrain,
//                                                   calcElemForces,
//                                                   calcElemHourglassForces)
//   F4 node pass      sum of the node's slots, acceleration, BCs,
//                     Chung-Hulbert correction, position update and the
//                     next step's prediction   (assemblyForces, calcAccel,
//                                                   ImposeBCA/BCV,
//                                                   UpdateCorrection*,
//                                                   UpdatePrediction)
//
// Meshes of at most 256 element clusters in FP64, 512 in FP32-mixed, take two
// kernels per step instead (paired passes; run_paired has the exceptions): F2
// becomes part of F3's staging, and F4 and the next F1 one cluster pass.  FP64
// meshes whose clusters share no node take all steps of a run but the last in
// one kernel (solo pass, run_solo).
//
// Every expression is the one of the per-step kernels, so the FP64 fused path
// differs from the per-step path only in the order of the nodal force sums:
// the hourglass force is subtracted per element instead of after the
// element-force sum, and a node's element forces are added per cluster
// (ascending element within a cluster, clusters in order) instead of in one
// ascending run.
//
// Device inputs beyond the per-step state:
//   nodel_pk[nnz]  packed CSR entry (element << 3) | local node
//   bc_word[N]     0, or (index into bc_val << 3) | mask (per-node Dirichlet data)
//   anp_ratio[N]   V_n / V0_n,   vsum0[N] = V0_n (constant after init)
#pragma once

#include "wfx_cluster.hpp"
#include "wfx_contact.hpp"
#include "wfx_kernels.hpp"
#include "wfx_launch.hpp"
#include "wfx_slots.hpp"

namespace wfx {
namespace {

// CSR entries fetched per batch of independent loads in the node passes
constexpr int kChunk = 8;  // also the width of the padded first-entries table
// Element-node rows of the per-step thermal rates (dTedt), tiled in blocks of
// 64 elements [E/64][n][64] so that a wavefront's rows are contiguous.
__device__ __forceinline__ long fidx(int row, long e, long Es, int nrow) {
  return (e >> 6) * ((long)nrow * 64) + (long)row * 64 + (e & 63);
}
// Data a pass reads or writes once per step (stress, strain, yield stress; F2's
// tables).  NT: non-temporal accesses keep these out of the way of what the
// gathers and the next pass read again; else the next step finds them in the
// last-level cache (wfx_ctx::stream_step says which).
template <bool NT, typename T>
__device__ __forceinline__ void st_stream(T *p, T v) {
  if constexpr (NT) __builtin_nontemporal_store(v, p);
  else *p = v;
}
template <bool NT, typename T>
__device__ __forceinline__ T ld_stream(const T *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  else return *p;
}

// The nodal ANP ratio F2 leaves for the element pass: double, or (FP32-mixed)
// 1 + a float deviation
template <typename T>
__device__ __forceinline__ double anp_ratio_at(const double *ratio, int i) {
  if constexpr (std::is_same<T, double>::value) return ratio[i];
  else return 1.0 + (double)reinterpret_cast<const float *>(ratio)[i];
}

// Once per run, V0_n: CSR-ordered sum of the initial volumes (calcElemPressure
// :698-705), and the mean density of the node's elements.  Densities do not
// change during a fused run, so CalcNodalMassFromVol's sum of rho V_n / c
// over the c elements is this mean times V_n: a loop of c divisions less in
// every step's nodal sums.  (A node of no element: mean and mass 0, its empty
// sum's.)  Without rho_avg no density is read: the later passes take a uniform
// density from their arguments.
template <typename T>
__global__ __launch_bounds__(kBlock) void f0_vsum0(int N, const int *__restrict__ off,
                                                   const int *__restrict__ cnt,
                                                   const int *__restrict__ nodel_pk,
                                                   const T *__restrict__ vol0, const T *__restrict__ rho,
                                                   double *__restrict__ vsum0, double *__restrict__ rho_avg) {
  int i = gtid();
  if (i >= N) return;
  int o = off[i], c = cnt[i];
  double s0 = 0.0, r = 0.0;
  for (int k = 0; k < c; ++k) {
    const int e = nodel_pk[o + k] >> 3;
    s0 += (double)vol0[e];
    if (rho_avg) r += (double)rho[e];
  }
  if (vsum0) vsum0[i] = s0;
  if (rho_avg) rho_avg[i] = c > 0 ? r / (double)c : 0.0;
}

// F2: nodal volume sum in CSR order; ratio for the ANP pressure and nodal
// mass (the nodal volume field itself is written once per run, in phase 5).
template <typename T, int BS, bool NT>
__global__ __launch_bounds__(BS) void f2_nodal(int N, int nodxelem, const int *__restrict__ off,
                                                   const int *__restrict__ cnt,
                                                   const int *__restrict__ nodel_pk,
                                                   const int *__restrict__ pad,
                                                   const T *__restrict__ vol,
                                                   const double *__restrict__ rho_avg,
                                                   const double *__restrict__ vsum0,
                                                   double *__restrict__ ratio,
                                                   double *__restrict__ mdiag, double rho_u, CflReduce cr,
                                                   const T *__restrict__ rho) {
  // per-step CFL time step: one more block reduces it beside the nodes, which do
  // not need it (a kernel of its own took 3 us and its launch)
  const int nb = gridDim.x - (cr.cfl > 0.0 ? 1 : 0);
  if ((int)blockIdx.x == nb) {
    cfl_reduce<BS>(cr, rho, true);
    return;
  }
  int i = xcd_block(nb) * BS + threadIdx.x;
  if (i >= N) return;
  const int c = ld_stream<NT>(&cnt[i]), o = c > kChunk ? off[i] : 0;
  // The table, count and V0_n are read once per step (4M FP64 hexahedra 68.4
  // us with plain loads, 60.8 with NT; 1.1M FP32-mixed 14.7 and 16.9).  The ratio
  // is stored plainly: the element pass gathers it next.
  // CSR entries are taken eight at a time with independent loads, then
  // summed in CSR order (the order of the reference's serial loop); the
  // first eight come from the padded [8][N] table.
  const double v0 = ld_stream<NT>(&vsum0[i]);
  const double rho_n = rho_u > 0.0 ? rho_u : ld_stream<NT>(&rho_avg[i]);
  double s = 0.0;
  for (int k = 0; k < c; k += kChunk) {
    int e[kChunk];
    double vv[kChunk];
#pragma unroll
    for (int j = 0; j < kChunk; ++j)
      e[j] = (k == 0) ? (ld_stream<NT>(&pad[(long)j * N + i]) >> 3) : ((k + j < c) ? (nodel_pk[o + k + j] >> 3) : -1);
    // every load is issued (entries past the count read the chunk's first
    // element) and only the node's own entries are added: conditional loads
    // would each be waited for on their own
#pragma unroll
    for (int j = 0; j < kChunk; ++j) vv[j] = (double)vol[e[j] >= 0 ? e[j] : e[0]];
#pragma unroll
    for (int j = 0; j < kChunk; ++j)
      if (k + j < c) s += vv[j];
  }
  // the ANP ratio V_n / V0_n: FP64 stores it; FP32-mixed stores its
  // deviation from 1 as a float in the same buffer (the element pass adds the
  // 1 back; the deviation keeps the float's relative precision)
  if constexpr (std::is_same<T, double>::value) ratio[i] = s / v0;
  else reinterpret_cast<float *>(ratio)[i] = (float)(s / v0 - 1.0);
  double vn = s;
  vn *= 1.0 / nodxelem;  // 4 or 8: exact
  st_stream<NT>(&mdiag[i], vn * rho_n);
}

// Nodes with many elements (tetrahedral meshes: about 23 per node) are
// summed by kF2Lanes lanes each: lane q takes the node's CSR entries q,
// q + kF2Lanes, ... in order, kF2Width at a time with every load issued, and
// the lanes' partial sums are combined by a butterfly, which leaves the same
// total in every lane.  V0_n goes through the same function, so the ANP ratio
// is exactly 1 wherever vol equals vol0.  val(e) gives entry e's term.
constexpr int kF2Lanes = 8, kF2Width = 4;
template <int L, typename F>
__device__ __forceinline__ double lane_csr_sum(int o, int c, int q, const int *__restrict__ nodel_pk, F val) {
  constexpr int W = kF2Width;
  double s = 0.0;
  for (int k0 = 0; k0 < c; k0 += W * L) {
    int e[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const int k = k0 + q + j * L;
      e[j] = nodel_pk[o + (k < c ? k : c - 1)] >> 3;
    }
    double v[W];
#pragma unroll
    for (int j = 0; j < W; ++j) v[j] = val(e[j]);
#pragma unroll
    for (int j = 0; j < W; ++j)
      if (k0 + q + j * L < c) s += v[j];
  }
#pragma unroll
  for (int m = 1; m < L; m <<= 1) s += __shfl_xor(s, m, L);
  return s;
}

// V0_n with kF2Lanes lanes per node (grid of N * kF2Lanes threads)
template <typename T>
__global__ __launch_bounds__(kBlock) void f0_vsum0_lanes(int N, const int *__restrict__ off,
                                                         const int *__restrict__ cnt,
                                                         const int *__restrict__ nodel_pk,
                                                         const T *__restrict__ vol0, const T *__restrict__ rho,
                                                         double *__restrict__ vsum0,
                                                         double *__restrict__ rho_avg) {
  constexpr int L = kF2Lanes;
  const long g = (long)xcd_block() * kBlock + threadIdx.x;
  const long n = g / L;
  const int q = (int)(g % L), i = (int)(n < N ? n : N - 1);  // every lane reaches the butterfly
  const int o = off[i], c = cnt[i];
  const double s0 = lane_csr_sum<L>(o, c, q, nodel_pk, [&](int e) { return (double)vol0[e]; });
  double r = 0.0;
  if (rho_avg) r = lane_csr_sum<L>(o, c, q, nodel_pk, [&](int e) { return (double)rho[e]; });
  if (q == 0 && n < N) {
    if (vsum0) vsum0[i] = s0;
    if (rho_avg) rho_avg[i] = c > 0 ? r / (double)c : 0.0;
  }
}

// F2 with kF2Lanes lanes per node: the nodal volume sum, ANP ratio and mass
// of f2_nodal
template <typename T, int BS>
__global__ __launch_bounds__(BS) void f2_nodal_lanes(int N, int nodxelem, const int *__restrict__ off,
                                                     const int *__restrict__ cnt,
                                                     const int *__restrict__ nodel_pk,
                                                     const T *__restrict__ vol,
                                                     const double *__restrict__ rho_avg,
                                                     const double *__restrict__ vsum0,
                                                     double *__restrict__ ratio, double *__restrict__ mdiag,
                                                     double rho_u, CflReduce cr, const T *__restrict__ rho) {
  constexpr int L = kF2Lanes;
  const int nb = gridDim.x - (cr.cfl > 0.0 ? 1 : 0);  // as in f2_nodal
  if ((int)blockIdx.x == nb) {
    cfl_reduce<BS>(cr, rho, true);
    return;
  }
  const long g = (long)xcd_block(nb) * BS + threadIdx.x;
  const long n = g / L;
  const int q = (int)(g % L), i = (int)(n < N ? n : N - 1);  // every lane reaches the butterflies
  const int o = off[i], c = cnt[i];
  // loaded with the offsets, not after the sum
  const double v0 = vsum0[i], rho_n = rho_u > 0.0 ? rho_u : rho_avg[i];
  const double s = lane_csr_sum<L>(o, c, q, nodel_pk, [&](int e) { return (double)vol[e]; });
  if (q != 0 || n >= N) return;
  if constexpr (std::is_same<T, double>::value) ratio[i] = s / v0;
  else reinterpret_cast<float *>(ratio)[i] = (float)(s / v0 - 1.0);
  mdiag[i] = s * (1.0 / nodxelem) * rho_n;
}

struct FusedParams {
  double dt;
  MatParams mp;
  PressParams pp;     // pp.full handled as in k_pressure_elem
  int need_jlocal;    // J_local = vol/vol0 enters the pressure
  double av_al, av_be;  // artificial viscosity (calcArtificialViscosity); both zero: none
  void *avq;          //   its diagonal stress term per element (T[E]), for the sigma field
  double hg_coeff, cs0;
  double rho_u;       // > 0: every element density equals it (no density loads)
  const double *dtp;  // non-null: the step's dt from the device (per-step CFL time step)
  double plheat_frac; // thermal coupling: fraction of plastic work into heat
  double k_T, cp_T;   //   conductivity and specific heat (rates when mp.Tn is set)
  // thermal expansion (with thermal coupling; texp null: none): exp_T, the
  // element means of the last rates (from F1), and where this step's rates
  // go: flat index flat_base[e] + a below N, divided by the node's mass
  double exp_T;
  const void *texp;
  void *dte_flat;
  const int *flat_base;
  const double *mdiag;
  // store the element outputs no later pass of the step reads (pressure,
  // yield stress, plastic heat, viscosity term): on a run's last step
  int write_out;
};

// dH(d,a) = adj(J)(d,:) . dN_a/dxi from the cofactor matrix C (adj = C^T),
// written exactly as calcElemJAndDerivatives does (Domain_d.C:1843-1850,
// :1866-1887).  a is a compile-time constant after unrolling.
template <typename T, int NN>
__device__ __forceinline__ T shape_dH(const T (&C)[3][3], int d, int a) {
  const T a0 = C[0][d], a1 = C[1][d], a2 = C[2][d];
  if constexpr (NN == 8) {
    const T q = T(0.125);
    switch (a) {
      case 0: return q * (-a0 - a1 - a2);
      case 1: return q * (a0 - a1 - a2);
      case 2: return q * (a0 + a1 - a2);
      case 3: return q * (-a0 + a1 - a2);
      case 4: return q * (-a0 - a1 + a2);
      case 5: return q * (a0 - a1 + a2);
      case 6: return q * (a0 + a1 + a2);
      default: return q * (-a0 + a1 + a2);
    }
  } else {
    switch (a) {
      case 0: return -a0 - a1 - a2;
      case 1: return a0;
      case 2: return a1;
      default: return a2;
    }
  }
}

// Walsh modes of a hexahedron's nodal values y[a] (local order of
// Domain_d.C:1313-1346): m[k] = sum_a y[a] prod_{i in k} s_i(a), the bits of
// k naming the natural directions (1 xi, 2 eta, 4 zeta) and s_i(a) = +-1 the
// sign of node a's natural coordinate (the table of Domain_d.C:1824-1826).
// m[1], m[2], m[4] are the sums calcElemJAndDerivatives weighs with 0.125
// (the rows of J for positions, of the velocity gradient in natural
// coordinates for velocities); m[6], m[5], m[3], m[7] are the hourglass
// amplitudes of Gamma rows 0..3 (Mechanical.f90:259-263: eta zeta, xi zeta,
// xi eta, xi eta zeta).  Three butterfly stages over the nodes in binary
// position order (local 0, 1, 3, 2, 4, 5, 7, 6); m[0] is not formed.
template <typename T>
__device__ __forceinline__ void hexa_modes(const T (&y)[8], T (&m)[8]) {
  const T a0 = y[1] + y[0], b0 = y[1] - y[0], a1 = y[2] + y[3], b1 = y[2] - y[3];
  const T a2 = y[5] + y[4], b2 = y[5] - y[4], a3 = y[6] + y[7], b3 = y[6] - y[7];
  const T c0 = a1 + a0, d0 = a1 - a0, c1 = b1 + b0, d1 = b1 - b0;
  const T c2 = a3 + a2, d2 = a3 - a2, c3 = b3 + b2, d3 = b3 - b2;
  m[0] = T(0);
  m[4] = c2 - c0;
  m[1] = c3 + c1;
  m[5] = c3 - c1;
  m[2] = d2 + d0;
  m[6] = d2 - d0;
  m[3] = d3 + d1;
  m[7] = d3 - d1;
}
// The inverse: nodal values z[a] = sum_k q[k] prod_{i in k} s_i(a) for
// mode coefficients q[1..7] (q[0] = 0), the same three stages in reverse.
template <typename T>
__device__ __forceinline__ void hexa_synthesis(const T (&q)[8], T (&z)[8]) {
  const T u0 = -q[4], u4 = q[4], u1 = q[1] - q[5], u5 = q[1] + q[5];
  const T u2 = q[2] - q[6], u6 = q[2] + q[6], u3 = q[3] - q[7], u7 = q[3] + q[7];
  const T v0 = u0 - u2, v2 = u0 + u2, v1 = u1 - u3, v3 = u1 + u3;
  const T v4 = u4 - u6, v6 = u4 + u6, v5 = u5 - u7, v7 = u5 + u7;
  z[0] = v0 - v1;
  z[1] = v0 + v1;
  z[3] = v2 - v3;
  z[2] = v2 + v3;
  z[4] = v4 - v5;
  z[5] = v4 + v5;
  z[7] = v6 - v7;
  z[6] = v6 + v7;
}

// Cofactors C (adj(J) = C^T, Matrix.h:694-727) and the Sarrus determinant
// (Matrix.h:610-615) of J.  FP64 without contraction: the same roundings as
// the per-step Jacobian kernel, so that an element's volume at rest equals
// its initial volume bit for bit (the ANP ratio is then exactly 1 there).
#define WFX_COFACTORS(J, C, detJ)                                                                         \
  C[0][0] = (J[1][1] * J[2][2] - J[1][2] * J[2][1]);                                                        \
  C[0][1] = -(J[1][0] * J[2][2] - J[1][2] * J[2][0]);                                                       \
  C[0][2] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]);                                                        \
  C[1][0] = -(J[0][1] * J[2][2] - J[0][2] * J[2][1]);                                                       \
  C[1][1] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]);                                                        \
  C[1][2] = -(J[0][0] * J[2][1] - J[0][1] * J[2][0]);                                                       \
  C[2][0] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]);                                                        \
  C[2][1] = -(J[0][0] * J[1][2] - J[0][2] * J[1][0]);                                                       \
  C[2][2] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]);                                                        \
  detJ = J[0][0] * J[1][1] * J[2][2] - J[0][0] * J[1][2] * J[2][1] - J[0][1] * J[1][0] * J[2][2] +          \
         J[0][1] * J[1][2] * J[2][0] + J[0][2] * J[1][0] * J[2][1] - J[0][2] * J[1][1] * J[2][0];
template <typename T>
__device__ __forceinline__ void cofactors(const T (&J)[3][3], T (&C)[3][3], T &detJ) {
  if constexpr (std::is_same<T, double>::value) {
#pragma clang fp contract(off)
    WFX_COFACTORS(J, C, detJ)
  } else {
    WFX_COFACTORS(J, C, detJ)
  }
}
#undef WFX_COFACTORS

// pow(vol, 0.6666666) of the hourglass coefficient (Mechanical.f90:299).
// FP64: vol^(2/3) exp(-d ln vol) with d = 2/3 - 0.6666666.  r = cbrt(vol), its
// square in two parts and the residual vol - r^3 give vol^(2/3) to half a unit
// in the last place; |d ln vol| < 5e-6, so that three terms of the exponential
// leave 2e-23.  The library's pow carries a double-double logarithm and
// exponential one after the other: 1450 of the 13200 cycles of the element
// pass's chain on an idle chip; cbrt and log are shorter and independent of
// each other.  Error of 8.4M volumes over 1e-30..1e30 against long double: largest
// 0.50 ulp, mean 0.25 (pow 1.34 and 0.34).  Other volumes
// (not positive, not finite, out of the float reciprocal's range) take pow.
// FP32-mixed: the hardware base-2 logarithm and exponential.
__device__ __forceinline__ double pow_hg(double vol) {
  constexpr double d = 6.666666666858372e-08;
  const double r = cbrt(vol), y = d * log(vol);
  const double h = r * r, l = fma(r, r, -h);
  const double res = fma(-r, l, fma(-r, h, vol));
  const double t = (2.0 / 3.0) * res * (double)__builtin_amdgcn_rcpf((float)vol) - y * (1.0 - y * (0.5 - y * (1.0 / 6.0)));
  return h + fma(h, t, l);
}
template <typename T>
__device__ __forceinline__ T vol_pow_hg(T vol) {
  if constexpr (std::is_same<T, double>::value) {
    if (vol >= 1e-30 && vol <= 1e30) return pow_hg(vol);
    return pow(vol, 0.6666666);
  } else {
    return exp2f(0.6666666f * log2f(vol));
  }
}

// The cluster's slots staged in LDS by the element pass: positions (double),
// predicted velocities (T), ANP ratio as F2 stored it (double, or the float
// deviation from 1) and node ids, [field][slot_cap].
template <typename T, int NN>
struct SlotLds {
  static constexpr int cap = slot_cap(NN);
  static constexpr int bytes = cap * (3 * 8 + 3 * (int)sizeof(T) + (int)sizeof(T) + 4);
  double *x;
  T *v, *r;
  int *node;
  __device__ explicit SlotLds(unsigned char *base)
      : x(reinterpret_cast<double *>(base)),
        v(reinterpret_cast<T *>(base + 3 * 8 * cap)),
        r(reinterpret_cast<T *>(base + (3 * 8 + 3 * (int)sizeof(T)) * cap)),
        node(reinterpret_cast<int *>(base + (3 * 8 + 4 * (int)sizeof(T)) * cap)) {}
};

// What the first part of the element chain leaves for the second: geometry,
// strain rate and spin, hourglass amplitudes, the nodal ANP average and,
// with thermal coupling, the element's temperature terms.
template <typename T, int NN, bool TH>
struct ElemGeo {
  T C[3][3];
  T detJ, volv;
  T s00, s11, s22, s01, s12, s02, w01, w12, w02;
  T hm[3][4];
  double J_avg, div_v;
  bool is_contact;
  int g[TH ? NN : 1];
  double tsum, gT0, gT1, gT2;
};

// The Jacobian of an element from its staged positions, as the per-step
// Jacobian kernel forms it (calcElemJAndDerivatives, Domain_d.C:1822-1889):
// hexahedron rows 0.125 * (the signed sum of the nodes in the reference's
// order), tetrahedron rows x_{i+1} - x_0; FP32-mixed from FP64 differences to
// node 0 narrowed to float.  FP64 without contraction, so that the volume
// at rest equals the initial volume bit for bit.
template <typename T, int NN>
__device__ __forceinline__ void staged_jacobian(const double *lx, int cap, const int (&ls)[NN], T (&J)[3][3]) {
  T X[NN][3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const double *xc = lx + c * cap;
    if constexpr (std::is_same<T, double>::value) {
#pragma unroll
      for (int a = 0; a < NN; ++a) X[a][c] = xc[ls[a]];
    } else {
      const double x0 = xc[ls[0]];
      X[0][c] = T(0);
#pragma unroll
      for (int a = 1; a < NN; ++a) X[a][c] = T(xc[ls[a]] - x0);
    }
  }
  if constexpr (std::is_same<T, double>::value) {
#pragma clang fp contract(off)
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if constexpr (NN == 8) {
        J[0][c] = T(0.125) * (-X[0][c] + X[1][c] + X[2][c] - X[3][c] - X[4][c] + X[5][c] + X[6][c] - X[7][c]);
        J[1][c] = T(0.125) * (-X[0][c] - X[1][c] + X[2][c] + X[3][c] - X[4][c] - X[5][c] + X[6][c] + X[7][c]);
        J[2][c] = T(0.125) * (-X[0][c] - X[1][c] - X[2][c] - X[3][c] + X[4][c] + X[5][c] + X[6][c] + X[7][c]);
      } else {
        J[0][c] = X[1][c] - X[0][c];
        J[1][c] = X[2][c] - X[0][c];
        J[2][c] = X[3][c] - X[0][c];
      }
    }
  } else {
#pragma unroll
    for (int c = 0; c < 3; ++c) {
      if constexpr (NN == 8) {
        J[0][c] = T(0.125) * (-X[0][c] + X[1][c] + X[2][c] - X[3][c] - X[4][c] + X[5][c] + X[6][c] - X[7][c]);
        J[1][c] = T(0.125) * (-X[0][c] - X[1][c] + X[2][c] + X[3][c] - X[4][c] - X[5][c] + X[6][c] + X[7][c]);
        J[2][c] = T(0.125) * (-X[0][c] - X[1][c] - X[2][c] - X[3][c] + X[4][c] + X[5][c] + X[6][c] + X[7][c]);
      } else {
        J[0][c] = X[1][c] - X[0][c];
        J[1][c] = X[2][c] - X[0][c];
        J[2][c] = X[3][c] - X[0][c];
      }
    }
  }
}

// The element's mean of its nodes' ANP ratios (calcElemPressure)
template <typename T, int NN>
__device__ __forceinline__ double element_ratio(const T *r, const int (&ls)[NN]) {
  double J_avg = 0.0;
#pragma unroll
  for (int a = 0; a < NN; ++a) {
    if constexpr (std::is_same<T, double>::value) J_avg += r[ls[a]];
    else J_avg += 1.0 + (double)r[ls[a]];
  }
  return J_avg / NN;
}

// F3, first part: everything that reads the staged nodal data of element
// `ls` (its nodes as slot indices): Jacobian, cofactors and determinant
// (calcElemJAndDerivatives), the velocity gradient and from it the strain
// rate and spin (calcElemStrainRates), the hourglass amplitudes, with RATIO the
// ANP average of the nodal ratios (calcElemPressure) and the contact test.
// sum_a dH(d,a) y_a = sum_i C[i][d] (0.125 m_i(y)) for a hexahedron
// (dH(d,a) = 0.125 sum_i s_i(a) C[i][d], Domain_d.C:1843-1850), and
// sum_i C[i][d] (y_{i+1} - y_0) for a tetrahedron (:1866-1887).
template <typename T, int NN, bool TH, bool RATIO>
__device__ __forceinline__ void element_geometry(const FusedParams &fp, const SlotLds<T, NN> &L,
                                                 const int (&ls)[NN], ElemGeo<T, NN, TH> &G) {
  T J[3][3];
  staged_jacobian<T, NN>(L.x, L.cap, ls, J);
  cofactors(J, G.C, G.detJ);
  const T w = (NN == 4) ? T(1.0 / 6.0) : T(8.0);
  G.volv = G.detJ * w;
  // velocity modes: Mv[i][c] = 0.125 m_i(v_c) / the tetrahedron's differences
  T Mv[3][3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    const T *vc = L.v + c * L.cap;
    if constexpr (NN == 8) {
      T y[8], m[8];
#pragma unroll
      for (int a = 0; a < 8; ++a) y[a] = vc[ls[a]];
      hexa_modes(y, m);
      Mv[0][c] = m[1];
      Mv[1][c] = m[2];
      Mv[2][c] = m[4];
      G.hm[c][0] = m[6];
      G.hm[c][1] = m[5];
      G.hm[c][2] = m[3];
      G.hm[c][3] = m[7];
    } else {
      const T v0 = vc[ls[0]];
#pragma unroll
      for (int i = 0; i < 3; ++i) Mv[i][c] = vc[ls[i + 1]] - v0;
#pragma unroll
      for (int j = 0; j < 4; ++j) G.hm[c][j] = T(0);
    }
  }
  // Gv(d,c) = sum_a dH(d,a) v_a,c up to the hexahedron's 0.125; the
  // reference's D and W (Mechanical.C:58-116): f = 1/detJ, off-diagonals
  // halved
  T Gv[3][3];
#pragma unroll
  for (int d = 0; d < 3; ++d)
#pragma unroll
    for (int c = 0; c < 3; ++c) Gv[d][c] = G.C[0][d] * Mv[0][c] + G.C[1][d] * Mv[1][c] + G.C[2][d] * Mv[2][c];
  const T f = T(1) / G.detJ;
  const T q = (NN == 8) ? T(0.125) * f : f, qh = T(0.5) * q;
  G.s00 = q * Gv[0][0];
  G.s11 = q * Gv[1][1];
  G.s22 = q * Gv[2][2];
  G.s01 = qh * (Gv[1][0] + Gv[0][1]);
  G.w01 = qh * (Gv[1][0] - Gv[0][1]);
  G.s12 = qh * (Gv[2][1] + Gv[1][2]);
  G.w12 = qh * (Gv[2][1] - Gv[1][2]);
  G.s02 = qh * (Gv[2][0] + Gv[0][2]);
  G.w02 = qh * (Gv[2][0] - Gv[0][2]);
  // div v times detJ for the pressure's stabilisation terms
  G.div_v = (NN == 8 ? 0.125 : 1.0) * ((double)Gv[0][0] + (double)Gv[1][1] + (double)Gv[2][2]);
  if constexpr (RATIO) G.J_avg = element_ratio<T, NN>(L.r, ls);
  G.is_contact = elem_in_contact<NN>(fp.pp, [&](int a) { return L.node[ls[a]]; });
  // thermal coupling (ThermalCalcs, Thermal.C:27-115): the conduction matrix
  // applied through the element's temperature gradient,
  // (Kt T)_i = sum_d dH(d,i) G_d with G_d = k_T w / detJ sum_j dH(d,j) T_j;
  // the nodal temperatures also give the rate laws' temperature (their mean)
  G.tsum = G.gT0 = G.gT1 = G.gT2 = 0.0;
  if constexpr (TH) {
#pragma unroll
    for (int a = 0; a < NN; ++a) {
      G.g[a] = L.node[ls[a]];
      const double ta = fp.mp.Tn[G.g[a]];
      G.tsum += ta;
      G.gT0 += (double)shape_dH<T, NN>(G.C, 0, a) * ta;
      G.gT1 += (double)shape_dH<T, NN>(G.C, 1, a) * ta;
      G.gT2 += (double)shape_dH<T, NN>(G.C, 2, a) * ta;
    }
    const double kf = fp.k_T / (double)G.detJ * (NN == 4 ? 1.0 / 6.0 : 8.0);
    G.gT0 *= kf;
    G.gT1 *= kf;
    G.gT2 *= kf;
  }
}

// F3, second part: thermal expansion, hourglass coefficient, ANP pressure,
// Jaumann update and J2 return (CalcStressStrain), artificial viscosity,
// the element's internal and hourglass forces (calcElemForces,
// calcElemHourglassForces: f - f_hg, what the assembly adds to each node),
// handed to sink(a, node, fx, fy, fz, thermal term).  Hexahedral element
// passes of the rate laws in FP64 keep the hourglass amplitudes and the
// cofactors in LDS across the stress update (stash: this thread's column,
// stride BS): the laws' transcendental functions otherwise push the pass
// past 256 VGPRs.
// The element's state the second part reads (CalcStressStrain's stress,
// strain, plastic strain and yield stress; the per-element plastic modulus
// of specimen batches): loaded by the work-group before it stages its
// slots, so that these loads are in flight together with the staging
template <typename T>
struct ElemState {
  T tau[6], eps[6], ep, sy0, He;
};
template <typename T, bool NT>
__device__ __forceinline__ void load_elem_state(int e, int E, const T *tau_io,
                                                const T *__restrict__ eps_io, const T *pl_strain,
                                                const T *__restrict__ sy0, const T *__restrict__ He,
                                                ElemState<T> &S) {
  const long Es = E;
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    S.tau[k] = ld_stream<NT>(&tau_io[k * Es + e]);
    S.eps[k] = ld_stream<NT>(&eps_io[k * Es + e]);
  }
  S.ep = ld_stream<NT>(&pl_strain[e]);
  S.sy0 = ld_stream<NT>(&sy0[e]);
  S.He = He ? ld_stream<NT>(&He[e]) : T(0);
}

template <typename T, int NN, int LAW>
constexpr bool kStashLDS = NN == 8 && LAW == LAW_RATE && std::is_same<T, double>::value;
// hm[3][4], c_h, C[3][3] and with thermal coupling the gradient term G[3]
template <bool TH>
constexpr int kStashVals = TH ? 25 : 22;

template <typename T, int NN, int LAW, int BS, bool TH, bool NT, class Sink>
__device__ __forceinline__ void element_material(
    int e, int E, const FusedParams &fp, T dt, ElemGeo<T, NN, TH> &G, const ElemState<T> &S,
    const T *__restrict__ vol0, const T *__restrict__ rho, const T *__restrict__ He, T *tau_out,
    T *__restrict__ eps_io, T *__restrict__ p_out, T *pl_out, bool pl_all, T *__restrict__ sigma_y,
    T *__restrict__ q_plheat, double *stash, Sink &&sink) {
  const long Es = E;
  T s00 = G.s00, s11 = G.s11, s22 = G.s22, s01 = G.s01, s12 = G.s12, s02 = G.s02;
  if constexpr (TH) {  // calcThermalExpansion (Thermal.C:164-178)
    if (fp.texp) {
      const double sh = fp.exp_T * (double)static_cast<const T *>(fp.texp)[e];
      s00 = (T)((double)s00 - sh * 1.0);
      s11 = (T)((double)s11 - sh * 1.0);
      s22 = (T)((double)s22 - sh * 1.0);
      s01 = (T)((double)s01 - sh * 0.0);
      s12 = (T)((double)s12 - sh * 0.0);
      s02 = (T)((double)s02 - sh * 0.0);
    }
  }
  const T volv = G.volv;
  T c_h = T(0);
  if constexpr (NN == 8) {
    if (fp.hg_coeff != 0.0) {
      const double rho_e = fp.rho_u > 0.0 ? fp.rho_u : (double)rho[e];
      c_h = (T)(fp.hg_coeff * rho_e * 0.25 * fp.cs0) * vol_pow_hg<T>(volv);
    }
  }
  if constexpr (kStashLDS<T, NN, LAW>) {
    double *st = stash;
    if constexpr (TH) {
      st[22 * BS] = G.gT0;
      st[23 * BS] = G.gT1;
      st[24 * BS] = G.gT2;
    }
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) st[(4 * c + j) * BS] = G.hm[c][j];
    st[12 * BS] = c_h;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) st[(13 + 3 * r + q) * BS] = G.C[r][q];
  }
  // ---- ANP pressure (calcElemPressure element part) ----------------------
  const PressParams &pp = fp.pp;
  const bool general = press_general(pp, (double)volv, G.J_avg);
  double J_local = 0.0;
  if (fp.need_jlocal || general) J_local = (double)volv / (double)vol0[e];
  const double div_v = G.div_v;
  const T pe = (T)anp_elem_pressure(
      pp, G.is_contact, general, J_local, G.J_avg, (double)volv, [&] { return (double)rho[e]; },
      [&] { return div_v; });
  if (fp.write_out) p_out[e] = pe;

  // ---- Jaumann update and J2 return (CalcStressStrain) -------------------
  const MatParams &mp = fp.mp;
  T3<T> tau = t3_from_sym(S.tau[0], S.tau[1], S.tau[2], S.tau[3], S.tau[4], S.tau[5]);
  T3<T> D = t3_from_sym(s00, s11, s22, s01, s12, s02);
  T3<T> W = t3_from_antisym(G.w01, G.w12, G.w02);
  T3<T> I = t3_identity<T>();
  T Gm = (T)mp.G;
  T3<T> Wt = t3_trans(W);
  T3<T> SRT = t3_mul(tau, Wt);
  T3<T> RS = t3_mul(W, tau);
  T3<T> cI = t3_scale(I, T(1.0 / 3.0) * t3_trace(D));
  T3<T> devD = t3_sub(D, cI);
  T3<T> A = t3_scale(devD, T(2) * Gm);
  T3<T> B = t3_add(A, SRT);
  T3<T> Cc = t3_add(B, RS);
  tau = t3_add(tau, t3_scale(Cc, dt));
  T3<T> pI = t3_scale(I, -pe);
  T3<T> st = t3_add(pI, tau);
  T3<T> s = t3_sub(st, t3_scale(I, T(1.0 / 3.0) * t3_trace(st)));
  T J2 = T(0.5) * (s.xx * s.xx + T(2) * s.xy * s.xy + T(2) * s.xz * s.xz + s.yy * s.yy +
                   T(2) * s.yz * s.yz + s.zz * s.zz);
  T sig_trial = sqrt(T(3) * J2);
  T ep = S.ep;
  // bilinear plastic modulus: per element when given (specimen batches)
  T sy, Hb = (T)mp.H;
  const bool per_elem = LAW == LAW_PLAIN && mp.model == BILINEAR && He;
  const T edot = (LAW == LAW_RATE) ? eff_strain_rate(D) : T(0);
  RateTemp rt = mp.ut;  // the rate laws' temperature factors (law_temperature on the loaded nodes)
  if constexpr (LAW == LAW_RATE) {
    if (!mp.t_uniform) {
      const double temp = TH ? G.tsum / NN : mp.Te[e];
      rt = rate_temp_at(mp, temp);
    }
  }
  RateCache<T> rc;
  if (per_elem) {
    Hb = S.He;
    sy = S.sy0 + Hb * ep;
  } else {
    sy = yield_stress<T, LAW>(mp, rt, S.sy0, ep, edot, rc);
  }
  if (fp.write_out) sigma_y[e] = sy;
  T dep = T(0);
  if (sy < sig_trial) {
    T H = per_elem ? Hb : tangent_modulus<T, LAW>(mp, rt, ep, cap_rate(mp, edot), rc);
    T dgamma = (sig_trial - sy) / (T(3) * Gm + H);
    T factor = T(1) - (T(3) * Gm * dgamma) / sig_trial;
    tau = t3_scale(s, factor);
    pl_out[e] = ep + dgamma;
    dep = dgamma;
  } else if (pl_all) {  // not in place: every element's
    pl_out[e] = ep;
  }
  T3<T> sig = t3_add(pI, tau);
  double heat = 0.0;  // thermal coupling: the element's heat per node and cp
  if constexpr (TH) {  // plastic heat source of the step
    T q = T(0);
    if (dep > T(0)) {
      const T f = dep / sy;
      q = plastic_heat<T>(sig, f * (sig.xx - T(0.5) * (sig.yy + sig.zz)), f * (sig.yy - T(0.5) * (sig.xx + sig.zz)),
                          f * (sig.zz - T(0.5) * (sig.xx + sig.yy)), T(1.5) * f * (sig.xy), T(1.5) * f * (sig.yz),
                          T(1.5) * f * (sig.xz), dt, fp.plheat_frac);
    }
    if (fp.write_out) q_plheat[e] = q;
    heat = 0.9 * (double)q * (double)volv / NN / fp.cp_T;
  }
  // ---- calcArtificialViscosity (Mechanical.C:1948-1977), after the stress
  // update as in the reference's step (Solver_explicit.C:755-757): added to
  // the diagonal stresses the forces use; kept per element for the sigma field.
  // With zero coefficients it is zero except where the volume is negative or
  // not finite, or the scan flagged the densities (0 * NaN, as in the
  // reference); an infinite diagonal strain rate already makes the diagonal
  // stresses NaN.
  if (fp.av_al != 0.0 || fp.av_be != 0.0 || pp.guard || !vol_regular((double)volv)) {
    const double rho_e = fp.rho_u > 0.0 ? fp.rho_u : (double)rho[e];
    double qs = 0.0;
    if (artificial_viscosity_q(pp.K, fp.av_al, fp.av_be, rho_e, (double)volv,
                               (double)D.xx + (double)D.yy + (double)D.zz, qs)) {
      sig.xx = (T)((double)sig.xx + qs);
      sig.yy = (T)((double)sig.yy + qs);
      sig.zz = (T)((double)sig.zz + qs);
    }
    if (fp.write_out) static_cast<T *>(fp.avq)[e] = (T)qs;
  }
  st_stream<NT>(&eps_io[0 * Es + e], S.eps[0] + D.xx * dt);
  st_stream<NT>(&eps_io[1 * Es + e], S.eps[1] + D.yy * dt);
  st_stream<NT>(&eps_io[2 * Es + e], S.eps[2] + D.zz * dt);
  st_stream<NT>(&eps_io[3 * Es + e], S.eps[3] + D.xy * dt);
  st_stream<NT>(&eps_io[4 * Es + e], S.eps[4] + D.yz * dt);
  st_stream<NT>(&eps_io[5 * Es + e], S.eps[5] + D.xz * dt);
  st_stream<NT>(&tau_out[0 * Es + e], tau.xx); st_stream<NT>(&tau_out[1 * Es + e], tau.yy);
  st_stream<NT>(&tau_out[2 * Es + e], tau.zz); st_stream<NT>(&tau_out[3 * Es + e], tau.xy);
  st_stream<NT>(&tau_out[4 * Es + e], tau.yz); st_stream<NT>(&tau_out[5 * Es + e], tau.xz);

  T C[3][3], hm[3][4];
  double gT0 = G.gT0, gT1 = G.gT1, gT2 = G.gT2;
  if constexpr (kStashLDS<T, NN, LAW>) {  // back from LDS (volatile: real loads)
    volatile double *sv = stash;
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) hm[c][j] = sv[(4 * c + j) * BS];
    c_h = sv[12 * BS];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) C[r][q] = sv[(13 + 3 * r + q) * BS];
    if constexpr (TH) {
      gT0 = sv[22 * BS];
      gT1 = sv[23 * BS];
      gT2 = sv[24 * BS];
    }
  } else {
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
      for (int q = 0; q < 3; ++q) C[r][q] = G.C[r][q];
#pragma unroll
    for (int c = 0; c < 3; ++c)
#pragma unroll
      for (int j = 0; j < 4; ++j) hm[c][j] = G.hm[c][j];
  }
  // ---- internal forces (calcElemForces, Mechanical.C:448-457) and hourglass
  // f_c(a) = w sum_d dH(d,a) sigma(d,c): the cofactors times the stress give
  // the coefficients of the linear modes, Q(i,c) = 0.125 w sum_d C[i][d]
  // sigma(d,c) (0.125 w = 1 for the hexahedron); the hourglass force
  // (fi -= f_hg, Matrices.f90:641) adds c_h times the amplitudes to the
  // hourglass modes; one synthesis per component gives the nodal forces.
  const T sg0 = sig.xx, sg1 = sig.yy, sg2 = sig.zz, sg3 = sig.xy, sg4 = sig.yz, sg5 = sig.xz;
  T Q[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    Q[i][0] = C[i][0] * sg0 + C[i][1] * sg3 + C[i][2] * sg5;
    Q[i][1] = C[i][0] * sg3 + C[i][1] * sg1 + C[i][2] * sg4;
    Q[i][2] = C[i][0] * sg5 + C[i][1] * sg4 + C[i][2] * sg2;
  }
  T fn[3][NN];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if constexpr (NN == 8) {
      T qm[8], z[8];
      qm[0] = T(0);
      qm[1] = Q[0][c];
      qm[2] = Q[1][c];
      qm[4] = Q[2][c];
      if (fp.hg_coeff != 0.0) {
        qm[6] = c_h * hm[c][0];
        qm[5] = c_h * hm[c][1];
        qm[3] = c_h * hm[c][2];
        qm[7] = c_h * hm[c][3];
      } else {
        qm[3] = qm[5] = qm[6] = qm[7] = T(0);
      }
      hexa_synthesis(qm, z);
#pragma unroll
      for (int a = 0; a < 8; ++a) fn[c][a] = z[a];
    } else {
      const T w = T(1.0 / 6.0);
      fn[c][1] = w * Q[0][c];
      fn[c][2] = w * Q[1][c];
      fn[c][3] = w * Q[2][c];
      fn[c][0] = -(fn[c][1] + fn[c][2] + fn[c][3]);
    }
  }
#pragma unroll
  for (int a = 0; a < NN; ++a) {
    // the node's thermal term times its mass: -(Kt T)_a + heat / cp
    T th = T(0);
    int node = 0;
    if constexpr (TH) {
      const T h0 = shape_dH<T, NN>(C, 0, a), h1 = shape_dH<T, NN>(C, 1, a), h2 = shape_dH<T, NN>(C, 2, a);
      th = (T)(heat - ((double)h0 * gT0 + (double)h1 * gT1 + (double)h2 * gT2));
      node = G.g[a];
    }
    sink(a, node, fn[0][a], fn[1][a], fn[2][a], th);
  }
}

// What the paired passes need beyond the four separate ones
struct PairArgs {
  const int4 *rec;       // per slot (DevMesh::srec)
  const int *sent;       //   and its node's elements [S][pw]
  const int *sbc;        //   and its boundary word
  int pw, lanes;         // lanes: summed as f2_nodal_lanes sums, else in CSR order as f2_nodal
  const void *vol;       // T[E]
  const double *vsum0, *rho_avg;
  double *ratio, *mdiag; // written by each node's first slot
  CflReduce cr;          // per-step CFL time step
};

// Where the element pass stores a slot's partial sum.  FP64 (but for the
// paired passes of small meshes, where one dependent load less counts and
// bandwidth does not): in slot order (a cluster's sums are one contiguous run; the node pass reads a node's
// slots through their ids, and moves its bytes near the copy rate anyway).
// FP32-mixed: node-major, at the slot's place in its node's slot list (the
// node pass reads a node's sums contiguously from its offset, one dependent
// load less; measured on the 200x200x100 block: node pass 154 -> 118 us,
// element pass +12 us, while FP64 loses 15 us in the element pass).
template <typename T>
constexpr bool kNodeMajor = std::is_same<T, float>::value;

// Values per element-node the element pass adds up: the force and, with
// thermal coupling, the node's thermal term
template <bool TH>
constexpr int kNodeVals = TH ? 4 : 3;

// LDS of one work-group of the element pass, in turn: the cluster's staged
// slots (SlotLds), then the element-node values (kEntStride; the last
// component without its unused cells) and, in the same space (each thread
// only ever writes its own column, and reloads its stash before it writes its
// values), the per-thread stash of the FP64 hexahedral rate-law passes.
// FP64 hexahedra: 53,256 bytes, three work-groups on a CU.
template <typename T, int NN, bool TH>
constexpr int kEntLds = ((kNodeVals<TH> - 1) * kEntStride(NN) + NN * kCluster + 1) * (int)sizeof(T);
template <typename T, int NN, int LAW, bool TH>
constexpr int kF3Vals = (kStashLDS<T, NN, LAW> && kStashVals<TH> * 8 * kCluster > kEntLds<T, NN, TH>)
                            ? kStashVals<TH> * 8 * kCluster
                            : kEntLds<T, NN, TH>;
template <typename T, int NN, int LAW, bool TH>
constexpr int kF3Lds = kF3Vals<T, NN, LAW, TH> > SlotLds<T, NN>::bytes ? kF3Vals<T, NN, LAW, TH>
                                                                        : SlotLds<T, NN>::bytes;

// The nodal volume sums of a thread's slots' nodes from the element volumes,
// with the ANP ratio as F2 leaves it and, by a node's first slot, the ratio
// and the mass stored: F2's sums in F2's orders (f2_nodal, or with lanes set
// f2_nodal_lanes: eight strided sums and their butterfly), so that paired and
// separate passes give the same bits.  In three parts, so that the entries
// are loaded with the slot records and the volumes with the nodal state: as
// one part after the staging's loads, slot after slot and with the mass
// summed from the densities, it added 6300 (hexahedra) and 12000
// (tetrahedra) cycles to the staging's 1000.
template <typename T, int NN, int SLOTS>
struct PairSum {
  // entries in flight: all of a structured hexahedral node's; up to 24 of a
  // tetrahedral one's
  static constexpr int W = NN == 8 ? 8 : 24, K = SLOTS;
  long slot[K];
  int4 en[K][W / 4];
  T v[K][W];
  double v0[K], rho_n[K];
  __device__ __forceinline__ void entries(const PairArgs &pr, int k0) {
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int h = 0; h < W / 4; ++h)
        en[k][h] = reinterpret_cast<const int4 *>(pr.sent + slot[k] * pr.pw)[min(k0 / 4 + h, pr.pw / 4 - 1)];
  }
  // vol: the volumes of the elements from the pass's first one on
  __device__ __forceinline__ void volumes(const T *vol) {
#pragma unroll
    for (int k = 0; k < K; ++k)
#pragma unroll
      for (int h = 0; h < W / 4; ++h) {
        v[k][4 * h + 0] = vol[en[k][h].x];
        v[k][4 * h + 1] = vol[en[k][h].y];
        v[k][4 * h + 2] = vol[en[k][h].z];
        v[k][4 * h + 3] = vol[en[k][h].w];
      }
  }
  __device__ __forceinline__ void nodal(const PairArgs &pr, const int4 (&rec)[K], double rho_u) {
#pragma unroll
    for (int k = 0; k < K; ++k) {
      v0[k] = pr.vsum0[rec[k].x];
      rho_n[k] = rho_u > 0.0 ? rho_u : pr.rho_avg[rec[k].x];
    }
  }
  // the nodes' sums, their further volumes from vol
  __device__ __forceinline__ void sums(const PairArgs &pr, const int4 (&rec)[K], const T *vol, double (&s)[K]) {
    double l[K][8];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      s[k] = 0.0;
#pragma unroll
      for (int j = 0; j < 8; ++j) l[k][j] = 0.0;
    }
    for (int k0 = 0;;) {
      // entries past the node's count add zero
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const int c = rec[k].w & 0xff;
        if (pr.lanes) {
#pragma unroll
          for (int j = 0; j < W; ++j) l[k][j & 7] += k0 + j < c ? (double)v[k][j] : 0.0;
        } else {
#pragma unroll
          for (int j = 0; j < W; ++j) s[k] += k0 + j < c ? (double)v[k][j] : 0.0;
        }
      }
      k0 += W;
      if (k0 >= pr.pw) break;
      entries(pr, k0);
      volumes(vol);
    }
#pragma unroll
    for (int k = 0; k < K; ++k)
      if (pr.lanes)
        s[k] = ((l[k][0] + l[k][1]) + (l[k][2] + l[k][3])) + ((l[k][4] + l[k][5]) + (l[k][6] + l[k][7]));
  }
  __device__ __forceinline__ T ratio(int k, double s) const {
    if constexpr (std::is_same<T, double>::value) return s / v0[k];
    else return (float)(s / v0[k] - 1.0);
  }
  __device__ __forceinline__ double mass(int k, double s) const { return s * (1.0 / NN) * rho_n[k]; }
};

// One slot's sums of R components: its entry groups [k0, k1), the first G of
// them in registers.  Four entries at a time with their LDS reads in flight
// together, added in order.  One entry per pass waited for two dependent LDS
// reads each time: 2800 (hexahedra) and 4900 (tetrahedra) of the 13200 and
// 11700 cycles a work-group takes on an idle chip.
template <typename T, int NN, int R, int G>
__device__ __forceinline__ void add_entries(const unsigned char *lds, const uint2 (&ew)[G], const uint2 *en, int k0, int k1,
                                            double (&acc)[R]) {
  auto add4 = [&](uint2 w) {
    T val[4][R];
#pragma unroll
    for (int h = 0; h < 4; ++h) {
      const unsigned o = h & 1 ? (h < 2 ? w.x : w.y) >> 16 : (h < 2 ? w.x : w.y) & 0xffffu;
#pragma unroll
      for (int u = 0; u < R; ++u) val[h][u] = *reinterpret_cast<const T *>(lds + o + u * (kEntStride(NN) * (int)sizeof(T)));
    }
#pragma unroll
    for (int h = 0; h < 4; ++h)
#pragma unroll
      for (int u = 0; u < R; ++u) acc[u] += (double)val[h][u];
  };
#pragma unroll
  for (int h = 0; h < G; ++h)
    if (k0 + h < k1) add4(ew[h]);
  for (int k = k0 + G; k < k1; ++k) add4(en[k]);  // more elements than the registers hold
}

// F3: one work-group per element cluster.  The work-group first stages its
// cluster's slots (the distinct nodes of its elements: positions,
// velocities, ANP ratio, ids) in LDS with one load per slot and field; each
// thread then runs the element chain of one element from LDS and leaves its
// element-node values in the same LDS; then the work-group adds them per
// cluster node (the slot's entries, ascending element, in double) and writes
// one partial sum per slot (assemblyForces, Matrices.C:42-87, for the
// cluster's share of each node).
// PAIR (small meshes, launch-bound): F2 is part of the staging, each slot's
// thread summing its node's element volumes; slots of a node in several
// clusters repeat the sum (1.7 times the work of F2), and a launch and F2's
// round trip of the ratio are saved.
template <typename T, int NN, int LAW, bool TH, bool PAIR, bool NT, int SL, int BS>
__global__ __launch_bounds__(BS) void f3_cluster(
    int E, int N, FusedParams fp, ClusterArgs ca, PairArgs pr, const double *__restrict__ x, const T *__restrict__ v,
    const double *__restrict__ ratio, const T *__restrict__ vol0, const T *__restrict__ rho,
    const T *__restrict__ sy0, const T *__restrict__ He, const T *tau_in, T *tau_out, T *__restrict__ eps_io,
    T *__restrict__ p_out, const T *pl_in, T *pl_out, T *__restrict__ sigma_y, T *__restrict__ part,
    T *__restrict__ q_plheat) {
  constexpr int R = kNodeVals<TH>;
  __shared__ __align__(16) unsigned char lds_raw[kF3Lds<T, NN, LAW, TH>];
  T *lf = reinterpret_cast<T *>(lds_raw);
  const SlotLds<T, NN> L(lds_raw);
  const int c = xcd_block(), t = threadIdx.x;
  const ClusterDesc cd = ca.desc[c];
  const int e0 = cd.e0, s0 = cd.s0, ne = cd.em & 0xffff, M = cd.em >> 16;  // M <= slot_cap(NN), checked at set-up
  const uint16_t *lo = ca.goff + cd.goff;
  const uint2 *en = ca.ent + cd.ent;  // the cluster's entry groups
  // the nodes of this thread's slots t and t + BS: first, as the
  // staging loads depend on them
  constexpr int kSl = SL;
  static_assert(kSl * BS <= slot_cap(NN) && kSl <= 2, "one or two slots per thread");
  // Every load below is issued unconditionally, threads past the cluster's
  // elements, entries or slots repeating its last one (a cluster has at
  // least one element and NN slots), so that none is waited for on its own;
  // the values are used only where they are the thread's own.
  // Loads return in order, so the order is that of the waits: the nodes of
  // this thread's slots t and t + BS (PAIR: with their elements), the
  // slot tables and the element's slots; the nodal state; the element's own
  // state last, which only the second part of the chain needs.  That is the
  // order of the paired passes, whose work-groups run alone on their CUs.  In
  // a large mesh the bytes decide and the state, most of them, is asked for
  // before the nodes' round trip (1.1M FP32-mixed hexahedra: 59.1 us with the
  // state last, 56.0 so; 4M in FP64 283 either way).
  int sn[kSl];
  int4 rec[kSl];
  bool mine[kSl];
  PairSum<T, NN, SL> ps;
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    const int j = t + k * BS, q = s0 + min(j, M - 1);
    if constexpr (PAIR) {
      rec[k] = pr.rec[q];
      sn[k] = rec[k].x;
      ps.slot[k] = q;
      mine[k] = j < M;
    } else {
      sn[k] = cd.node0 + ca.nrel[cd.nrel + min(j, M - 1)];
    }
  }
  if constexpr (PAIR) ps.entries(pr, 0);
  // The entry groups' range of the thread's own slots t and t + BS; the
  // groups themselves follow once these are here.
  uint32_t ow[kSl];  // (end << 16) | start of slots t and t + BS
  int sp[kSl];       //   and where their sums go
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    const int q = min(t + k * BS, M - 1);
    __builtin_memcpy(&ow[k], lo + q, 4);  // lo[q], lo[q + 1]
    if constexpr (kNodeMajor<T> || PAIR) sp[k] = ca.spos[s0 + q];
    else sp[k] = ca.nm ? ca.spos[s0 + q] : s0 + q;
  }
  int ls[NN];
  const int my_e = e0 + min(t, ne - 1);
  load_lslot<NN>(ca.lslot + (long)(cd.lslot + min(t, ne - 1)) * NN, ls);
  ElemState<T> S;
  if constexpr (PAIR) __builtin_amdgcn_sched_barrier(0);
  else load_elem_state<T, NT>(my_e, E, tau_in, eps_io, pl_in, sy0, He, S);
  // stage the slots: all loads first, then the LDS stores
  double sx[kSl][3];
  T sv[kSl][3], sr[kSl];
  if constexpr (PAIR) ps.volumes(static_cast<const T *>(pr.vol));
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    const int node = sn[k];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      sx[k][d] = x[(long)d * N + node];
      sv[k][d] = v[(long)d * N + node];
    }
    if constexpr (PAIR) {
    } else if constexpr (std::is_same<T, double>::value) {
      sr[k] = ratio[node];
    } else {
      sr[k] = reinterpret_cast<const float *>(ratio)[node];
    }
  }
  if constexpr (PAIR) ps.nodal(pr, rec, fp.rho_u);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (PAIR) load_elem_state<T, NT>(my_e, E, tau_in, eps_io, pl_in, sy0, He, S);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (PAIR) {
    double vs[kSl];
    ps.sums(pr, rec, static_cast<const T *>(pr.vol), vs);
#pragma unroll
    for (int k = 0; k < kSl; ++k) {
      sr[k] = ps.ratio(k, vs[k]);
      if (mine[k] && rec[k].w < 0) {
        reinterpret_cast<T *>(pr.ratio)[rec[k].x] = sr[k];
        pr.mdiag[rec[k].x] = ps.mass(k, vs[k]);
      }
    }
  }
  double dt_step = fp.dt;
  if constexpr (PAIR) {
    // every work-group reduces the step's dt for itself, since a kernel for it
    // takes 3 us and the few partials of a small mesh less than one; the first
    // work-group stores it for the later kernels
    if (pr.cr.cfl > 0.0) dt_step = cfl_reduce<BS>(pr.cr, rho, blockIdx.x == 0);
  } else {
    if (fp.dtp) dt_step = *fp.dtp;
  }
  const T dt = (T)dt_step;
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    const int j = t + k * BS;  // < slot_cap
    L.node[j] = sn[k];
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      L.x[d * L.cap + j] = sx[k][d];
      L.v[d * L.cap + j] = sv[k][d];
    }
    L.r[j] = sr[k];
  }
  __syncthreads();
  // The thread's slots' entries straight from the table: they arrive under
  // the element chain.  (Staged in LDS, the eight 16-bit reads of a slot cost
  // as many LDS passes as a third of its values.)
  constexpr int kGr = NN == 8 ? 2 : 6;  // groups held in registers
  uint2 ew[kSl][kGr];
#pragma unroll
  for (int k = 0; k < kSl; ++k)
#pragma unroll
    for (int h = 0; h < kGr; ++h) ew[k][h] = en[(ow[k] & 0xffffu) + h];
  ElemGeo<T, NN, TH> G;
  if (t < ne) element_geometry<T, NN, TH, true>(fp, L, ls, G);
  __syncthreads();  // the staged slots are read: their LDS takes the element-node values
  if (t < ne) {
    element_material<T, NN, LAW, kCluster, TH, NT>(
        e0 + t, E, fp, dt, G, S, vol0, rho, He, tau_out, eps_io, p_out, pl_out, pl_in != pl_out, sigma_y, q_plheat,
        reinterpret_cast<double *>(lds_raw) + t, [&](int a, int node, T f0, T f1, T f2, T th) {
          lf[0 * kEntStride(NN) + a * kCluster + t] = f0;
          lf[1 * kEntStride(NN) + a * kCluster + t] = f1;
          lf[2 * kEntStride(NN) + a * kCluster + t] = f2;
          if constexpr (TH) {
            lf[3 * kEntStride(NN) + a * kCluster + t] = th;
            if (fp.dte_flat) {  // this step's rate at the flat index calcThermalExpansion reads
              const long q = (long)fp.flat_base[e0 + t] + a;
              if (q < N) static_cast<T *>(fp.dte_flat)[q] = (T)((double)th / fp.mdiag[node]);
            }
          }
        });
  }
  // the zero cells lie in thread 0's column, as its stash does: it is done with it
  if (t == 0)
#pragma unroll
    for (int u = 0; u < R; ++u) lf[u * kEntStride(NN) + NN * kCluster] = T(0);
  __syncthreads();
#pragma unroll
  for (int r = 0; r < kSl; ++r) {  // M <= kSl * BS
    const int j = t + r * BS;
    if (j >= M) break;
    const int k0 = ow[r] & 0xffffu, k1 = ow[r] >> 16;
    double acc[R];
#pragma unroll
    for (int q = 0; q < R; ++q) acc[q] = 0.0;
    add_entries<T, NN, R, kGr>(lds_raw, ew[r], en, k0, k1, acc);
#pragma unroll
    for (int q = 0; q < R; ++q) part[q * ca.S + sp[r]] = (T)acc[q];  // cached: the node pass reads them next
  }
}

// One element's volume from its staged positions, the inverted-element count
// and (edges) its smallest edge
template <typename T, int NN>
__device__ __forceinline__ double element_volume(int e, const double *lx, int cap, const int (&ls)[NN], bool edges,
                                                 T *__restrict__ vol, unsigned int *__restrict__ status) {
  T J[3][3], C[3][3], det;
  staged_jacobian<T, NN>(lx, cap, ls, J);
  cofactors(J, C, det);
  const T w = (NN == 4) ? T(1.0 / 6.0) : T(8.0);
  vol[e] = det * w;  // CalcElemVol's 0 + detJ * w * 1 (the same value)
  count_inverted(det, status);
  if (!edges) return kMinEdgeInit;
  T P[4][3];  // the first four nodes, as calcMinEdgeLength takes them
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      if constexpr (std::is_same<T, double>::value) P[a][d] = lx[d * cap + ls[a]];
      else P[a][d] = T(lx[d * cap + ls[a]] - lx[d * cap + ls[0]]);
    }
  return min_edge4<T>(P);
}

// F1 as a cluster pass: one work-group per element cluster stages its
// slots' positions (and node ids when thermal expansion reads them) in LDS,
// then each thread forms its element's Jacobian from LDS (the same Jacobian
// as the element pass's): vol = detJ * w (calcElemJAndDerivatives
// determinant + CalcElemVol), the inverted-element count, with minl_part the
// work-group's smallest edge (per-step CFL time step), with texp each
// element's mean of the last step's element-node temperature rates at the
// flat indices of its node ids (calcThermalExpansion's dTdt).
template <typename T, int NN>
__global__ __launch_bounds__(kCluster) void f1_cluster(int E, ClusterArgs ca, const double *__restrict__ x, int N,
                                                       T *__restrict__ vol, double *__restrict__ minl_part,
                                                       unsigned int *__restrict__ status,
                                                       const T *__restrict__ dte_flat, T *__restrict__ texp) {
  constexpr int cap = slot_cap(NN);
  __shared__ double lx[3 * cap];
  __shared__ int lnode[cap];
  const int c = xcd_block(), t = threadIdx.x;
  const ClusterDesc cd = ca.desc[c];
  const int e0 = cd.e0, s0 = cd.s0, ne = cd.em & 0xffff, M = cd.em >> 16;  // M <= slot_cap(NN), checked at set-up
  // every load is issued unconditionally (threads past the cluster's
  // elements or slots repeat its last one), as in the element pass
  constexpr int kSl = kSlotsPerThread<NN>;
  int sn[kSl];
#pragma unroll
  for (int k = 0; k < kSl; ++k) sn[k] = cd.node0 + ca.nrel[cd.nrel + min(t + k * kCluster, M - 1)];
  int ls[NN];
  load_lslot<NN>(ca.lslot + (long)(cd.lslot + min(t, ne - 1)) * NN, ls);
  double sx[kSl][3];
#pragma unroll
  for (int k = 0; k < kSl; ++k)
#pragma unroll
    for (int d = 0; d < 3; ++d) sx[k][d] = x[(long)d * N + sn[k]];
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    const int j = t + k * kCluster;  // < slot_cap
#pragma unroll
    for (int d = 0; d < 3; ++d) lx[d * cap + j] = sx[k][d];
    lnode[j] = sn[k];
  }
  __syncthreads();
  double medge = kMinEdgeInit;
  if (t < ne) {
    const int e = e0 + t;
    if (texp) {
      double m = 0.0;
#pragma unroll
      for (int a = 0; a < NN; ++a) m += 1.0 / NN * (double)dte_flat[lnode[ls[a]]];
      texp[e] = (T)m;
    }
    medge = element_volume<T, NN>(e, lx, cap, ls, minl_part != nullptr, vol, status);
  }
  if (minl_part) {
    medge = block_extreme<kCluster, true>(medge);
    if (threadIdx.x == 0) minl_part[blockIdx.x] = medge;
  }
}

// ---- thermal coupling ------------------------------------------------------
// ThermalCalcs (Thermal.C:27-115) without contact conduction.  Element e:
// Kt(i,j) = (sum_d dH(d,i) dH(d,j)) k_T / detJ * w, element-node rate
// -(Kt T)_i / m_i + 0.9 q_plheat vol / n / (m_i cp_T) into dTedt[i][E]; the
// node pass adds a node's rates in CSR order and advances T by dt.
template <typename T, int NN>
__device__ __forceinline__ void thermal_rates(int e, long Es, const int (&g)[NN], const double (&h)[3][NN],
                                              double detJ, double vol, double q, const double *__restrict__ Tn,
                                              const double *__restrict__ mdiag, double k_T, double cp_T,
                                              T *__restrict__ dTedt, long q0, int N, T *__restrict__ dte_flat) {
  const double w = (NN == 4) ? 1.0 / 6.0 : 8.0;
  double Te[NN];
#pragma unroll
  for (int a = 0; a < NN; ++a) Te[a] = Tn[g[a]];
  const double heat = 0.9 * q;
  const double elem_pow = heat * vol;
  const double pow_per_node = elem_pow / NN;
#pragma unroll
  for (int i = 0; i < NN; ++i) {
    double acc = 0.0;
#pragma unroll
    for (int j = 0; j < NN; ++j) {
      double k = 0.0;
      k += h[0][i] * h[0][j];
      k += h[1][i] * h[1][j];
      k += h[2][i] * h[2][j];
      const double kt = k * k_T / detJ * w;
      acc += kt * Te[j];
    }
    const double m = mdiag[g[i]];
    const double m_inv = 1.0 / m;
    double r = -m_inv * acc;
    r += pow_per_node / (m * cp_T);
    dTedt[fidx(i, e, Es, NN)] = (T)r;
    if (dte_flat && q0 + i < N) dte_flat[q0 + i] = (T)r;  // the entries thermal expansion reads
  }
}

// per-step API: shape derivatives and determinant of this step's Jacobians
template <typename T, int NN>
__global__ __launch_bounds__(kBlock) void k_thermal_elem(
    int E, const int *__restrict__ elnod, const T *__restrict__ dH, const T *__restrict__ detJ,
    const T *__restrict__ vol, const T *__restrict__ q, const double *__restrict__ Tn,
    const double *__restrict__ mdiag, double k_T, double cp_T, T *__restrict__ dTedt,
    const int *__restrict__ flat_base, int N, T *__restrict__ dte_flat) {
  const int e = gtid();
  if (e >= E) return;
  int g[NN];
  double h[3][NN];
#pragma unroll
  for (int a = 0; a < NN; ++a) {
    g[a] = elnod[(long)a * E + e];
#pragma unroll
    for (int d = 0; d < 3; ++d) h[d][a] = (double)dH[(long)(d * NN + a) * E + e];
  }
  thermal_rates<T, NN>(e, E, g, h, (double)detJ[e], (double)vol[e], (double)q[e], Tn, mdiag, k_T, cp_T, dTedt,
                       dte_flat ? (long)flat_base[e] : 0L, N, dte_flat);
}

// calcThermalExpansion (Thermal.C:164-178): the strain rate loses (exp_T times
// the mean of the last step's element-node temperature rates at the flat
// indices given by the element's node ids) on its diagonal; the shear rates
// lose that times 0.
template <typename T, int NN>
__global__ __launch_bounds__(kBlock) void k_thermal_expansion(int E, const int *__restrict__ elnod,
                                                              const T *__restrict__ dte_flat, double exp_T,
                                                              T *__restrict__ sr) {
  const int e = gtid();
  if (e >= E) return;
  const long Es = E;
  double m = 0.0;
#pragma unroll
  for (int i = 0; i < NN; ++i) m += 1.0 / NN * (double)dte_flat[elnod[(long)i * Es + e]];
  const double sh = exp_T * m;
#pragma unroll
  for (int k = 0; k < 6; ++k) sr[k * Es + e] = (T)((double)sr[k * Es + e] - sh * (k < 3 ? 1.0 : 0.0));
}

// T += (sum of the node's element-node rates in CSR order) * dt; the rates
// sit in the element-force layout (fidx) and are gathered like the forces
template <typename T>
__global__ __launch_bounds__(kBlock) void k_thermal_node(int N, long Es, int nn, const int *__restrict__ off,
                                                         const int *__restrict__ cnt,
                                                         const int *__restrict__ nodel_pk,
                                                         const int *__restrict__ pad,
                                                         const T *__restrict__ dTedt, double dt,
                                                         double *__restrict__ Tn,
                                                         const double *__restrict__ qc,
                                                         const double *__restrict__ mdiag, double cp_T) {
  const int i = gtid();
  if (i >= N) return;
  const int c = cnt[i], o = c > kChunk ? off[i] : 0;
  double dTdt = 0.0;
  for (int k = 0; k < c; k += kChunk) {
    int pk[kChunk];
    double q[kChunk];
#pragma unroll
    for (int j = 0; j < kChunk; ++j)
      pk[j] = (k == 0) ? pad[(long)j * N + i] : ((k + j < c) ? nodel_pk[o + k + j] : -1);
#pragma unroll
    for (int j = 0; j < kChunk; ++j)
      q[j] = (pk[j] >= 0) ? (double)dTedt[fidx(pk[j] & 7, pk[j] >> 3, Es, nn)] : 0.0;
#pragma unroll
    for (int j = 0; j < kChunk; ++j)
      if (k + j < c) dTdt += q[j];
  }
  // with the contact heat conduction of the last contact step (Thermal.C:124)
  const double qn = qc ? qc[i] * 1.0 / (mdiag[i] * cp_T) : 0.0;
  Tn[i] += (dTdt + qn) * dt;
}

struct NodeParams {
  double dt, alpha, beta, gamma;
  double f;        // 1/(1-alpha)
  double gdt;      // gamma*dt
  double bdt2;     // beta*dt*dt
  double pred_u;   // (0.5-beta)*dt   (next prediction)
  double pred_v;   // (1-gamma)*dt
  int predict;     // run the next step's prediction
  int write_fi;    // store the internal force (last step of a run, or its reaction is recorded)
  int read_ud;     // read the predicted increment (else recomputed from v' and prev_a)
  int write_ud;    // store the increment every step (else on a run's last step only)
  int run_first, run_last;  // FP64: first / last step of a run (both: u += u_dt directly)
  double *x_start;          //   positions when the run started
  float *x_lo;              //   rounding error of the position updates since then
  int has_fe;      // external forces present
  const double *dtp;  // per-step CFL time step: the step's dt on the device
  double *vmax_part;  //   and the per-block largest predicted speed
  const double *qcont;  // contact heat conduction per node (thermal with contact), or null
  double cp_T;
  // reaction record (rz null: none): one bit per reaction node, the rank of
  // each word's first one, and the step's row of z forces (the nodal type)
  const unsigned long long *rbits;
  const int *rbase;
  void *rz;
};

// The step's z force of a reaction node into its row.  A wavefront's 64 nodes
// share one word of bits, so the test costs one scalar load; storing every
// node's force instead (and reading the reaction nodes' back) cost 24 B per
// node and step.
// (LANES: the lanes hold nodes of their own, each with its own word.)
template <typename T, bool LANES>
__device__ __forceinline__ void record_reaction(const NodeParams &np, int i, double fz) {
  if (!np.rz) return;
  const int w = LANES ? i >> 6 : __builtin_amdgcn_readfirstlane(i >> 6);
  const unsigned long long b = np.rbits[w];
  const int l = i & 63;
  if ((b >> l) & 1ull)
    static_cast<T *>(np.rz)[np.rbase[w] + __popcll(b & ((1ull << l) - 1ull))] = (T)fz;
}

// the step-length terms of NodeParams for step length dt (same expressions
// as node_params on the host)
__device__ __forceinline__ void set_step_length(NodeParams &np, double dt) {
  np.dt = dt;
  np.gdt = np.gamma * dt;
  np.bdt2 = np.beta * dt * dt;
  np.pred_u = (0.5 - np.beta) * dt;
  np.pred_v = (1.0 - np.gamma) * dt;
}

// The state of node i the nodal update reads, loaded before the node's
// partial force sums so that these loads are in flight together with them.
template <typename T, bool CONTACT>
struct NodeIn {
  T v[3], pa[3], ud[3];
  float lo[3];
  double x[3], u[3], xs[3], fe[3], cf[3], bv[3], m;
  int mask;
};
template <typename T, bool CONTACT>
__device__ __forceinline__ void load_node(int i, long Ns, const NodeParams &np, const double *__restrict__ cf,
                                          const double *__restrict__ fe, const double *__restrict__ mdiag,
                                          int word,
                                          const double *__restrict__ bc_val, const T *__restrict__ v,
                                          const T *__restrict__ prev_a, const T *__restrict__ u_dt,
                                          const double *__restrict__ x, const double *__restrict__ u,
                                          NodeIn<T, CONTACT> &s) {
  // row bases are uniform; the unsigned node index lets every row share one
  // 32-bit offset register
  const unsigned ui = (unsigned)i;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const long r = d * Ns;
    s.v[d] = (v + r)[ui];
    s.pa[d] = (prev_a + r)[ui];
    // the predicted increment is used on a run's first step only; the other
    // steps load the array's first entry in every lane instead (one cache
    // line), so that no branch holds the load: a float widened inside one
    // waits for every load issued before it
    s.ud[d] = (u_dt + (np.read_ud ? r : 0L))[np.read_ud ? ui : 0u];
    s.x[d] = (x + r)[ui];
    s.u[d] = s.xs[d] = 0.0;
    s.lo[d] = 0.0f;
    if constexpr (std::is_same<T, double>::value) {  // FP32-mixed: u from x when a run ends
      // the error term is loaded every step (a run's first ignores it): a
      // load behind a branch would have its float widened inside the branch,
      // which waits for every load issued before it
      s.lo[d] = (np.x_lo + r)[ui];
      if (np.run_last) {
        s.u[d] = (u + r)[ui];
        s.xs[d] = (np.x_start + r)[ui];
      }
    }
    s.fe[d] = np.has_fe ? (fe + r)[ui] : 0.0;
    s.cf[d] = 0.0;
    if constexpr (CONTACT) s.cf[d] = (cf + r)[ui];
  }
  s.m = mdiag[ui];
  // The boundary values here and not where they are used: six uses in a row,
  // each behind its own branch, waited for their load one after the other and
  // made the constrained nodes' wavefronts the last ones of the pass.
  s.mask = word & 7;
  s.bv[0] = s.bv[1] = s.bv[2] = 0.0;
  if (word) {
    const double *b = bc_val + 3L * (word >> 3);
    s.bv[0] = b[0];
    s.bv[1] = b[1];
    s.bv[2] = b[2];
  }
}

// The nodal update of one step for node i given its assembled internal
// force f: non-finite scrub (Solver_explicit.C:777-785), calcAccel, ImposeBCA,
// UpdateCorrectionAccVel, ImposeBCV, UpdateCorrectionPos and the next step's
// UpdatePrediction + ImposeBCV.  FP64: every nodal array is double.
// FP32-mixed: velocity, previous acceleration, increment and internal force
// are stored in float (the update itself runs in double), positions stay
// double, and u is not touched per step (recovered as x - x_start when the
// run ends).  FP64 neither: positions advance as x += u_dt, and the exact
// rounding error of each of those additions (two-sum) is accumulated in a
// float beside them, so that u = u_start + ((x - x_start) + error) when the
// run ends is the sum of the increments to a few units in the last place of
// u (x - x_start alone loses the bits of x that u does not have); a one-step
// run adds the increment to u directly.
// The predicted increment u_dt = dt (v + (0.5 - beta) dt a) of the previous
// node pass is not stored between the steps of a run: it is formed again
// from what that pass stored, v' = v + (1 - gamma) dt a (or the imposed
// velocity, which the prediction then used itself) and prev_a = a, which
// gives it up to the rounding of v'.  The first step of a run reads the
// increment UpdatePrediction left (its v may differ from an imposed v'), a
// run's last step stores the corrected increment, and with a per-step time
// step (the previous step's length predicted it) it is read and stored
// every step.
// BY: the node pass (a thread per node); the paired node pass, where several
// work-groups update the same node, only the one that owns it (own) stores
// and xn_out receives the new position in either case; or the solo pass, which
// keeps the state in s from step to step.
enum NodeBy { BY_NODE, BY_SLOT, IN_PLACE };
template <typename T, bool CFL, bool CONTACT, int BY>
__device__ __forceinline__ double node_update(
    int i, long Ns, const NodeParams &np, double (&f)[3], NodeIn<T, CONTACT> &s,
    T *__restrict__ fi, T *__restrict__ v, T *__restrict__ prev_a, T *__restrict__ u_dt, double *__restrict__ x, double *__restrict__ u,
    unsigned int *__restrict__ status, bool own, double *xn_out) {
  const bool store = BY != BY_SLOT || own;
  unsigned bad = 0;
#pragma unroll
  for (int d = 0; d < 3; ++d)
    if (!isfinite(f[d])) { f[d] = 0.0; ++bad; }
  if (bad && store) atomicAdd(status, bad);
  if (store) record_reaction<T, BY != BY_NODE>(np, i, f[2]);
  const int mask = s.mask;
  const double m = s.m;
  double vs[3];
  const unsigned ui = (unsigned)i;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const long r = d * Ns;
    T &fi_d = (fi + r)[ui], &v_d = (v + r)[ui], &pa_d = (prev_a + r)[ui], &ud_d = (u_dt + r)[ui];
    double &x_d = (x + r)[ui];
    if (np.write_fi && store) fi_d = (T)f[d];
    double a = (s.fe[d] - f[d]) / m;                    // calcAccel
    if constexpr (CONTACT) a += s.cf[d] / m;            //   + contact force
    if (mask & (1 << d)) a = 0.0;                       // ImposeBCA
    double pa = (double)s.pa[d];
    a = np.f * (a - np.alpha * pa);                     // UpdateCorrectionAccVel
    double vv = (double)s.v[d] + np.gdt * a;
    if (mask & (1 << d)) vv = s.bv[d];    // ImposeBCV
    // the previous node pass's prediction, from its v' and a
    double v0 = (double)s.v[d];
    if (!(mask & (1 << d))) v0 = v0 - np.pred_v * pa;
    double ud = np.read_ud ? (double)s.ud[d] : np.dt * (v0 + np.pred_u * pa);
    ud = ud + np.bdt2 * a;                              // UpdateCorrectionPos
    const double xo = s.x[d], xn = xo + ud;
    if constexpr (BY == IN_PLACE) s.x[d] = xn;
    else if (store) x_d = xn;
    if constexpr (BY == BY_SLOT) xn_out[d] = xn;
    if constexpr (std::is_same<T, double>::value) {
      const double bb = xn - xo;
      const double err = (xo - (xn - bb)) + (ud - bb);  // xo + ud - xn, exactly
      const double lo = (np.run_first ? 0.0 : (double)s.lo[d]) + err;
      if (!store) {
      } else if (np.run_last) {
        (u + r)[ui] = s.u[d] + (np.run_first ? ud : ((xn - s.xs[d]) + lo));
      } else {
        if (np.run_first) (np.x_start + r)[ui] = xo;
        if constexpr (BY == IN_PLACE) s.lo[d] = (float)lo;
        else (np.x_lo + r)[ui] = (float)lo;
      }
    }
    if (np.predict) {                                   // UpdatePrediction
      ud = np.dt * (vv + np.pred_u * a);
      vv = vv + np.pred_v * a;
      if (mask & (1 << d)) vv = s.bv[d];  // ImposeBCV
    }
    if constexpr (BY == IN_PLACE) {
      s.pa[d] = (T)a;
      s.v[d] = (T)vv;
    } else if (store) {
      if (np.write_ud || !np.predict) ud_d = (T)ud;
      pa_d = (T)a;
      v_d = (T)vv;
    }
    vs[d] = (double)(T)vv;
  }
  // speed of the predicted velocity, for the next step's CFL time step
  if constexpr (CFL) return sqrt(vs[0] * vs[0] + vs[1] * vs[1] + vs[2] * vs[2]);
  return 0.0;
}

// Internal force of node i (and with TH its thermal term in f[3]): the sum of
// its slots' partial sums in ascending cluster order (assemblyForces,
// Matrices.C:42-87, completed across clusters), four at a time: FP64 through
// the slot ids of the node's list, FP32-mixed directly from its offset (the
// element pass stores those sums node-major).
// W: partial sums in flight together.
template <typename T, bool TH, int W>
__device__ __forceinline__ void gather_slots(int o, int c, bool nm, const int *__restrict__ nsl, const T *__restrict__ part,
                                             long S, double (&f)[TH ? 4 : 3]) {
  constexpr int R = TH ? 4 : 3;
#pragma unroll
  for (int d = 0; d < R; ++d) f[d] = 0.0;
  // every load is issued (indices past the node's count repeat its last
  // slot) and only the node's own entries are added: conditional loads would
  // each be waited for on their own
  for (int k = 0; k < c; k += W) {
    int sl[W];
#pragma unroll
    for (int j = 0; j < W; ++j) {
      const int kk = min(k + j, c - 1);
      if (kNodeMajor<T> || nm) sl[j] = o + kk;
      else sl[j] = nsl[o + kk];
    }
    T q[W][R];
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int d = 0; d < R; ++d) q[j][d] = part[d * S + sl[j]];
#pragma unroll
    for (int j = 0; j < W; ++j)
      if (k + j < c)
#pragma unroll
        for (int d = 0; d < R; ++d) f[d] += (double)q[j][d];
  }
}

// F4: assembly and the whole nodal update of one step; CFL: dt from the
// device and each block's largest predicted speed for the next step's dt;
// TH: thermal coupling, T += (sum of the node's thermal terms) / m * dt
template <typename T, int BS, bool CFL, bool CONTACT, bool TH>
__global__ __launch_bounds__(BS) void f4_node(
    int N, NodeParams np, int nm, const double *__restrict__ cf, const int *__restrict__ nsl_off,
    const int *__restrict__ nsl, const T *__restrict__ part, long S,
    const double *__restrict__ fe, const double *__restrict__ mdiag, const int *__restrict__ bc_word,
    const double *__restrict__ bc_val, T *__restrict__ fi,
    T *__restrict__ v, T *__restrict__ prev_a, T *__restrict__ u_dt,
    double *__restrict__ x, double *__restrict__ u, unsigned int *__restrict__ status,
    double *__restrict__ Tn, RigidArgs rg) {
  NodeParams q = np;
  if constexpr (CFL) set_step_length(q, *q.dtp);
  // contact: one more block moves the rigid surfaces beside the nodes (a
  // kernel of its own took 2 us and its launch)
  int nb = gridDim.x;
  if constexpr (CONTACT) {
    nb -= rg.rn > 0 ? 1 : 0;
    if ((int)blockIdx.x == nb) {
      rigid_move(rg, q.dt);
      return;
    }
  }
  const int i = xcd_block(nb) * BS + threadIdx.x;
  double speed = 0.0;
  if (i < N) {
    // the node's slot range first: the partial sums wait for it, not for
    // the state loads behind it
    const int o = nsl_off[i], c = nsl_off[i + 1] - o;
    const int word = bc_word[i];  // and the boundary word: the boundary values wait for it
    NodeIn<T, CONTACT> st;
    load_node<T, CONTACT>(i, N, q, cf, fe, mdiag, word, bc_val, v, prev_a, u_dt, x, u, st);
    double f[TH ? 4 : 3];
    gather_slots<T, TH, 4>(o, c, nm, nsl, part, S, f);
    speed = node_update<T, CFL, CONTACT, BY_NODE>(i, N, q, *reinterpret_cast<double(*)[3]>(f), st, fi, v, prev_a, u_dt, x, u, status, true, nullptr);
    if constexpr (TH) {  // T += (dTdt + q_cont / (m cp)) dt (Thermal.C:124)
      double r = f[3] / st.m;
      if (q.qcont) r += q.qcont[i] * 1.0 / (st.m * q.cp_T);
      Tn[i] += r * q.dt;
    }
  }
  if constexpr (CFL) {
    if (q.predict) {
      speed = block_extreme<BS, false>(speed);
      if (threadIdx.x == 0) q.vmax_part[blockIdx.x] = speed;
    }
  }
}



// F4 and the next step's F1 in one cluster pass (small meshes, launch-bound):
// each work-group updates all nodes its elements touch, one per thread, so
// that it has the new positions its volumes need without waiting for other
// work-groups; a node of several clusters is updated by each of them alike
// and stored by its first slot's.  The new state goes to the other set of
// buffers, since the other work-groups still read this one (x_lo and T, which
// only the storing thread uses, stay in place).
// Bound: two dependent rounds of loads (slot record and boundary word; sums,
// state and boundary values), each near a microsecond since the last kernel's
// results lie beyond this XCD's L2, the update and the launch; not bytes.
struct NodeSet {  // the nodal arrays a paired node pass writes
  double *x;
  void *v, *pa, *ud;
};
template <typename T, int NN, bool CFL, bool CONTACT, bool TH, int SL>
__global__ __launch_bounds__(SL * kCluster) void f41_cluster(
    int N, NodeParams np, ClusterArgs ca, PairArgs pr, NodeSet out, const double *__restrict__ cf,
    const T *__restrict__ part, const double *__restrict__ fe, const double *__restrict__ mdiag,
    const double *__restrict__ bc_val, T *__restrict__ fi, const T *__restrict__ v, const T *__restrict__ prev_a,
    const T *__restrict__ u_dt, const double *__restrict__ x, unsigned int *__restrict__ status,
    double *__restrict__ Tn, T *__restrict__ vol, double *__restrict__ minl_part, RigidArgs rg) {
  constexpr int cap = SL * kCluster;
  __shared__ double lx[3 * cap];
  NodeParams q = np;
  if constexpr (CFL) set_step_length(q, *q.dtp);
  int nb = gridDim.x;
  if constexpr (CONTACT) {  // one more block, as in f4_node
    nb -= 1;
    if ((int)blockIdx.x == nb) {
      rigid_move(rg, q.dt);
      return;
    }
  }
  const int c = xcd_block(nb), t = threadIdx.x;
  const ClusterDesc cd = ca.desc[c];
  const int e0 = cd.e0, s0 = cd.s0, ne = cd.em & 0xffff, M = cd.em >> 16;  // M <= cap, checked at set-up
  // as in the element pass every load is issued unconditionally: threads past
  // the cluster's slots or elements repeat its last one and store nothing
  const int4 rec = pr.rec[s0 + min(t, M - 1)];
  const int word = pr.sbc[s0 + min(t, M - 1)];
  int ls[NN];
  load_lslot<NN>(ca.lslot + (long)(cd.lslot + min(t, ne - 1)) * NN, ls);
  const int i = rec.x;
  const bool own = t < M && rec.w < 0;
  NodeIn<T, CONTACT> st;
  load_node<T, CONTACT>(i, N, q, cf, fe, mdiag, word, bc_val, v, prev_a, u_dt, x, nullptr, st);
  double f[TH ? 4 : 3];
  // all of a node's sums in one round: up to 8 clusters meet in a corner of bricks
  if (__any(rec.z > 4)) gather_slots<T, TH, 8>(rec.y, rec.z, true, nullptr, part, ca.S, f);
  else gather_slots<T, TH, 4>(rec.y, rec.z, true, nullptr, part, ca.S, f);
  double xn[3];
  double speed = node_update<T, CFL, CONTACT, BY_SLOT>(
      i, N, q, *reinterpret_cast<double(*)[3]>(f), st, fi, static_cast<T *>(out.v), static_cast<T *>(out.pa),
      static_cast<T *>(out.ud), out.x, nullptr, status, own, xn);
#pragma unroll
  for (int d = 0; d < 3; ++d) lx[d * cap + t] = xn[d];
  if constexpr (TH) {
    if (own) {
      double r = f[3] / st.m;
      if (q.qcont) r += q.qcont[i] * 1.0 / (st.m * q.cp_T);
      Tn[i] += r * q.dt;
    }
  }
  __syncthreads();
  double medge = kMinEdgeInit;
  if (t < ne) medge = element_volume<T, NN>(e0 + t, lx, cap, ls, CFL, vol, status);
  if constexpr (CFL) {
    medge = block_extreme<cap, true>(medge);
    speed = block_extreme<cap, false>(speed);
    if (t == 0) {
      minl_part[blockIdx.x] = medge;
      q.vmax_part[blockIdx.x] = speed;
    }
  }
}

// Many steps of a mesh whose clusters share no node, in one launch: each
// work-group's elements and nodes meet no other's, so that it steps alone, the
// nodal state in registers (the thread of a slot is its node's), positions,
// volumes and ratios in LDS.  Same arithmetic in the same order as the paired
// passes, bit for bit.  The element state goes through memory as there (a
// thread reads what it wrote; the loads lead the step and are not waited for
// until the stress update).
// Bound: the chain of one element and four barriers, on one CU: latency.  The
// two launches a step and their round trips were three fifths of it.  Measured,
// us a step, launched: one hexahedron 11.5 by the paired passes, 4.7 here; 216
// hexahedra 5.9, with Johnson-Cook's law 10.4; the smallest tetrahedral cylinder 4.0.
template <typename T, int NN, int LAW>
__global__ __launch_bounds__(slot_cap(NN)) void f_solo(
    int E, int N, int nsteps, size_t rz_row, FusedParams fp, NodeParams np, ClusterArgs ca, PairArgs pr,
    double *x, T *v, T *prev_a, const T *__restrict__ u_dt, const double *__restrict__ fe,
    const double *__restrict__ bc_val, const T *__restrict__ vol0, const T *__restrict__ rho,
    const T *__restrict__ sy0, const T *__restrict__ He, T *tau, T *eps, T *pl, unsigned int *status) {
  constexpr int cap = slot_cap(NN), R = 3;
  __shared__ __align__(16) unsigned char staged[SlotLds<T, NN>::bytes];
  __shared__ __align__(16) unsigned char lds_raw[kF3Vals<T, NN, LAW, false>];  // element-node values and stash, as in F3
  __shared__ T lvol[kCluster], lpa[3 * cap];  // volumes; each thread's node's previous acceleration,
  __shared__ double lbv[3 * cap];             //   boundary values and
  __shared__ float llo[3 * cap];              //   position error terms
  const SlotLds<T, NN> L(staged);
  T *lf = reinterpret_cast<T *>(lds_raw);
  const int t = threadIdx.x;
  const ClusterDesc cd = ca.desc[blockIdx.x];
  const int e0 = cd.e0, s0 = cd.s0, ne = cd.em & 0xffff, M = cd.em >> 16;  // M <= slot_cap(NN), checked at set-up
  const uint16_t *lo = ca.goff + cd.goff;
  const uint2 *en = ca.ent + cd.ent;
  // a thread per slot; as in F3, threads past the cluster's slots or elements
  // repeat its last one
  const int j = min(t, M - 1), te = min(t, ne - 1);
  PairSum<T, NN, 1> ps;
  int ls[NN];
  load_lslot<NN>(ca.lslot + (long)(cd.lslot + te) * NN, ls);
  const int4 rec[1] = {pr.rec[s0 + j]};
  ps.slot[0] = s0 + j;
  uint32_t ow;
  __builtin_memcpy(&ow, lo + j, 4);
  const int k0 = ow & 0xffffu, k1 = ow >> 16, i = rec[0].x, mask = pr.sbc[s0 + j] & 7;
  np.predict = 1;
  np.run_last = np.write_fi = np.write_ud = 0;
  {
    NodeIn<T, false> st;
    load_node<T, false>(i, N, np, nullptr, fe, pr.mdiag, pr.sbc[s0 + j], bc_val, v, prev_a, u_dt, x, nullptr, st);
    L.node[t] = i;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      L.x[d * cap + t] = st.x[d];
      L.v[d * cap + t] = st.v[d];
      lpa[d * cap + t] = st.pa[d];
      lbv[d * cap + t] = st.bv[d];
      llo[d * cap + t] = st.lo[d];
    }
  }
  ps.nodal(pr, rec, fp.rho_u);
  constexpr int kGr = NN == 8 ? 2 : 6;
  uint2 ew[kGr];
#pragma unroll
  for (int h = 0; h < kGr; ++h) ew[h] = en[k0 + h];
  const T dt = (T)fp.dt;
  for (int step = 0; step < nsteps; ++step) {
    // opaque, or the addresses of every row and entry are kept from step to
    // step, in more registers than there are
    int e = e0 + te;
    asm volatile("" : "+v"(e));
#pragma unroll
    for (int h = 0; h < kGr; ++h) asm volatile("" : "+v"(ew[h].x), "+v"(ew[h].y));
#pragma unroll
    for (int a = 0; a < NN; ++a) asm volatile("" : "+v"(ls[a]));
    ps.entries(pr, 0);
    __syncthreads();
    ElemGeo<T, NN, false> G;
    if (t < ne) {
      element_geometry<T, NN, false, false>(fp, L, ls, G);
      count_inverted(G.detJ, status);
      lvol[t] = G.volv;
    }
    ElemState<T> S;
    load_elem_state<T, false>(e, E, tau, eps, pl, sy0, He, S);
    __syncthreads();
    double vs[1];
    ps.volumes(lvol - e0);
    ps.sums(pr, rec, lvol - e0, vs);
    L.r[t] = ps.ratio(0, vs[0]);
    const double m = ps.mass(0, vs[0]);
    __syncthreads();
    if (t < ne) {
      G.J_avg = element_ratio<T, NN>(L.r, ls);
      element_material<T, NN, LAW, kCluster, false, false>(
          e, E, fp, dt, G, S, vol0, rho, He, tau, eps, nullptr, pl, false, nullptr, nullptr,
          reinterpret_cast<double *>(lds_raw) + t, [&](int a, int, T f0, T f1, T f2, T) {
            lf[0 * kEntStride(NN) + a * kCluster + t] = f0;
            lf[1 * kEntStride(NN) + a * kCluster + t] = f1;
            lf[2 * kEntStride(NN) + a * kCluster + t] = f2;
          });
    }
    if (t == 0)  // the zero cells, as in F3
#pragma unroll
      for (int u = 0; u < R; ++u) lf[u * kEntStride(NN) + NN * kCluster] = T(0);
    __syncthreads();
    if (t < M) {
      double acc[R] = {0.0, 0.0, 0.0}, f[3];
      add_entries<T, NN, R, kGr>(lds_raw, ew, en, k0, k1, acc);
#pragma unroll
      for (int d = 0; d < 3; ++d) f[d] = 0.0 + (double)(T)acc[d];
      NodeIn<T, false> st;
      st.m = m;
      st.mask = mask;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const long r = (long)d * N;
        st.x[d] = L.x[d * cap + t];
        st.v[d] = L.v[d * cap + t];
        st.pa[d] = lpa[d * cap + t];
        st.bv[d] = lbv[d * cap + t];
        st.lo[d] = llo[d * cap + t];
        st.fe[d] = np.has_fe ? (fe + r)[(unsigned)i] : 0.0;
        st.ud[d] = T(0);
        if (np.read_ud) st.ud[d] = (u_dt + r)[(unsigned)i];
      }
      node_update<T, false, false, IN_PLACE>(i, N, np, f, st, nullptr, v, prev_a, nullptr, x, nullptr, status, true,
                                             nullptr);
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        L.x[d * cap + t] = st.x[d];
        L.v[d * cap + t] = st.v[d];
        lpa[d * cap + t] = st.pa[d];
        llo[d * cap + t] = st.lo[d];
      }
    }
    np.run_first = np.read_ud = 0;
    if (np.rz) np.rz = static_cast<char *>(np.rz) + rz_row;
  }
  if (t >= M) return;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const long r = (long)d * N;
    (x + r)[(unsigned)i] = L.x[d * cap + t];
    (v + r)[(unsigned)i] = L.v[d * cap + t];
    (prev_a + r)[(unsigned)i] = lpa[d * cap + t];
    if constexpr (std::is_same<T, double>::value) (np.x_lo + r)[(unsigned)i] = llo[d * cap + t];
  }
}

// FP32-mixed fused runs keep v, prev_a, u_dt and fi in float between steps:
// narrowed once when the run starts, widened back (and u advanced by the
// position change) when it ends.
__global__ __launch_bounds__(kBlock) void f_pack(long n3, const double *__restrict__ v,
                                                 const double *__restrict__ pa,
                                                 const double *__restrict__ ud,
                                                 const double *__restrict__ x, float *__restrict__ v32,
                                                 float *__restrict__ pa32, float *__restrict__ ud32,
                                                 double *__restrict__ x0) {
  long i = gtid();
  if (i >= n3) return;
  v32[i] = (float)v[i];
  pa32[i] = (float)pa[i];
  ud32[i] = (float)ud[i];
  x0[i] = x[i];
}
__global__ __launch_bounds__(kBlock) void f_unpack(long n3, const float *__restrict__ v32,
                                                   const float *__restrict__ pa32,
                                                   const float *__restrict__ ud32,
                                                   const float *__restrict__ fi32,
                                                   const double *__restrict__ x,
                                                   const double *__restrict__ x0, double *__restrict__ v,
                                                   double *__restrict__ pa, double *__restrict__ a,
                                                   double *__restrict__ ud, double *__restrict__ fi,
                                                   double *__restrict__ u) {
  long i = gtid();
  if (i >= n3) return;
  v[i] = v32[i];
  pa[i] = a[i] = pa32[i];
  ud[i] = ud32[i];
  fi[i] = fi32[i];
  u[i] = u[i] + (x[i] - x0[i]);
}

// sigma = -p I + tau (CalcStressStrain :1766), for the field after a fused run
// (+ the step's artificial-viscosity term, calcArtificialViscosity, when avq)
// With zero viscosity coefficients (av_all false) the term is read only for
// the elements the element pass wrote it for: negative or non-finite volume
// in the last step (vol holds that step's volumes), or all under the guard.
template <typename T>
__global__ __launch_bounds__(kBlock) void f_sigma(int E, const T *__restrict__ p,
                                                  const T *__restrict__ tau, const T *__restrict__ avq,
                                                  const T *__restrict__ vol, int av_all,
                                                  T *__restrict__ sigma) {
  int e = gtid();
  if (e >= E) return;
  const long Es = E;
  T pe = p[e];
  T3<T> I = t3_identity<T>();
  T3<T> pI = t3_scale(I, -pe);
  T3<T> t = t3_from_sym(tau[0 * Es + e], tau[1 * Es + e], tau[2 * Es + e], tau[3 * Es + e], tau[4 * Es + e],
                        tau[5 * Es + e]);
  T3<T> s = t3_add(pI, t);
  if ((av_all || !vol_regular((double)vol[e])) && avq[e] != T(0)) {
    const double qs = (double)avq[e];
    s.xx = (T)((double)s.xx + qs);
    s.yy = (T)((double)s.yy + qs);
    s.zz = (T)((double)s.zz + qs);
  }
  sigma[0 * Es + e] = s.xx; sigma[1 * Es + e] = s.yy; sigma[2 * Es + e] = s.zz;
  sigma[3 * Es + e] = s.xy; sigma[4 * Es + e] = s.yz; sigma[5 * Es + e] = s.xz;
}

// Contact launchers (internal to each translation unit; the per-step API
// reaches them through the wrappers of wfx_k64.hip).
hipError_t launch_ext_face_areas(wfx_ctx *c, hipStream_t s) {
  const auto &ct = c->contact;
  hipLaunchKernelGGL(k_ext_face_areas, dim3(nblocks(ct.next)), dim3(kBlock), 0, s, ct.next, ct.ext_nodes,
                     ct.afc_off, ct.afc_face, ct.ext_face, c->N, c->nd.x, ct.node_area);
  return hipGetLastError();
}
hipError_t launch_elem_length(wfx_ctx *c, hipStream_t s) {
  hipLaunchKernelGGL(k_elem_length, dim3(nblocks(c->E)), dim3(kBlock), 0, s, c->E, c->N, c->ms.elnod, c->nd.x,
                     c->contact.elem_length);
  return hipGetLastError();
}
// CalcContactForces with the predicted velocities v (T: the fused FP32 path's
// narrowed copy) and the host's dt or the device's (per-step CFL)
template <typename T>
hipError_t launch_contact(wfx_ctx *c, const T *v, bool device_dt, hipStream_t s) {
  const auto &ct = c->contact;
  ContactParams cp{ct.rt,        ct.rnode,  ct.rnormal, ct.rpplane, ct.rtri, ct.rmesh,
                   c->prm.mat.E, ct.pf,     ct.mu_sta,  ct.mu_dyn,  c->prm.dt,
                   device_dt ? c->scalars + kCflDt : nullptr,
                   ct.heat_cond, ct.T_const, c->nd.T, c->thermal.on ? ct.q_cont : nullptr};
  hipLaunchKernelGGL((k_contact<T>), dim3(nblocks(ct.next)), dim3(kBlock), 0, s, ct.next, ct.ext_nodes, c->N, cp,
                     c->nd.x, v, c->nd.mdiag, c->ms.nodel_offset, c->ms.nodel_count, c->ms.nodel, ct.elem_length,
                     ct.node_area, ct.contforce, ct.ut_prev, ct.mesh_in_contact, ct.cfn);
  return hipGetLastError();
}
inline RigidArgs rigid_args(const wfx_ctx *c, bool move) {
  const auto &ct = c->contact;
  return RigidArgs{move ? ct.rn : 0, ct.rt, ct.rnode, ct.rvel, ct.rtri, ct.rnormal, ct.rpplane};
}
hipError_t launch_rigid_update(wfx_ctx *c, bool device_dt, hipStream_t s) {
  hipLaunchKernelGGL(k_rigid_update, dim3(1), dim3(kBlock), 0, s, rigid_args(c, true), c->prm.dt,
                     device_dt ? c->scalars + kCflDt : nullptr);
  return hipGetLastError();
}

}  // namespace

// Whether what is launched on s is recorded, not run.  The null stream cannot be
// captured (and asking about it fails while another thread captures).
inline bool is_capturing(hipStream_t s) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return s != nullptr && hipStreamIsCapturing(s, &st) == hipSuccess && st != hipStreamCaptureStatusNone;
}
// Whether the passes read the nodal mean densities
inline bool reads_means(const wfx_ctx *c) { return !(c->rho_uniform > 0.0); }
// V0_n (v0) and, where they are read, the nodal mean densities
template <typename T>
hipError_t launch_run_sums(wfx_ctx *c, bool v0, hipStream_t s) {
  double *const avg = reads_means(c) ? c->nd.rho_avg : nullptr;
  if (c->f2_lanes) {
    hipLaunchKernelGGL((f0_vsum0_lanes<T>), dim3(nblocks((long)c->N * kF2Lanes)), dim3(kBlock), 0, s, c->N,
                       c->ms.nodel_offset, c->ms.nodel_count, c->ms.nodel_pk, elem<T>(c).vol0, elem<T>(c).rho,
                       v0 ? c->nd.voln0_sum : (double *)nullptr, avg);
  } else {
    hipLaunchKernelGGL((f0_vsum0<T>), dim3(nblocks(c->N)), dim3(kBlock), 0, s, c->N, c->ms.nodel_offset,
                       c->ms.nodel_count, c->ms.nodel_pk, elem<T>(c).vol0, elem<T>(c).rho,
                       v0 ? c->nd.voln0_sum : (double *)nullptr, avg);
  }
  if (avg && !is_capturing(s)) c->rho_avg_valid = true;
  return hipGetLastError();
}
template <typename T>
hipError_t launch_vsum0(wfx_ctx *c, hipStream_t s) {
  return launch_run_sums<T>(c, true, s);
}

inline NodeParams node_params(wfx_ctx *c, int predict) {
  const auto &P = c->prm;
  NodeParams np;
  np.dt = P.dt;
  np.alpha = P.alpha;
  np.beta = P.beta;
  np.gamma = P.gamma;
  np.f = 1.0 / (1.0 - P.alpha);
  np.gdt = P.gamma * P.dt;
  np.bdt2 = P.beta * P.dt * P.dt;
  np.pred_u = (0.5 - P.beta) * P.dt;
  np.pred_v = (1.0 - P.gamma) * P.dt;
  np.predict = predict;
  np.write_fi = c->fused_write_fi;
  np.read_ud = c->fused_read_ud;
  np.write_ud = c->fused_write_ud;
  np.run_first = c->fused_run_first;
  np.run_last = c->fused_run_last;
  np.x_start = c->x_start;
  np.x_lo = c->x_lo;
  np.has_fe = c->has_fe;
  np.dtp = nullptr;
  np.vmax_part = nullptr;
  np.qcont = (c->thermal.on && c->contact.on) ? c->contact.q_cont : nullptr;
  np.cp_T = c->thermal.cp_T;
  np.rbits = c->react_bits;
  np.rbase = c->react_base;
  np.rz = c->fused_rz;
  return np;
}

// dt of step `step` of a run from the partial extremes (per-step CFL time step)
inline CflReduce cfl_args(const wfx_ctx *c, double cfl, int nmin, int step) {
  return CflReduce{cfl,  c->prm.mat.K, c->cfl_part,   c->cfl_part + c->cfl_cap_min, nmin, c->cfl_nvmax,
                   step, c->scalars,   (step >= 0 && step < c->dt_cap) ? c->dt_hist : nullptr};
}

template <typename T>
hipError_t launch_thermal(wfx_ctx *c, hipStream_t s);

// Launch one phase (1..4) of a fused step on the current state with block
// size BS; launch_fused_phase picks BS from the context (autotuned or 256).
template <typename T, int NN, bool PAIR, bool NT, int SL, int BS>
auto f3_pick(bool rate, bool th) {
  return rate ? (th ? f3_cluster<T, NN, LAW_RATE, true, PAIR, NT, SL, BS> : f3_cluster<T, NN, LAW_RATE, false, PAIR, NT, SL, BS>)
              : (th ? f3_cluster<T, NN, LAW_PLAIN, true, PAIR, NT, SL, BS> : f3_cluster<T, NN, LAW_PLAIN, false, PAIR, NT, SL, BS>);
}
template <typename T, bool PAIR, bool NT>
auto f3_pick(int n, bool one_slot, bool rate, bool th) {
  if (n == 4) return f3_pick<T, 4, PAIR, NT, 1, kCluster>(rate, th);
  if constexpr (PAIR) {
    // a thread per slot: one work-group on a CU, the second slot's loads and
    // sums would only lengthen its chain
    return one_slot ? f3_pick<T, 8, PAIR, NT, 1, kCluster>(rate, th) : f3_pick<T, 8, PAIR, NT, 1, 2 * kCluster>(rate, th);
  } else {
    return f3_pick<T, 8, PAIR, NT, 2, kCluster>(rate, th);
  }
}

// the fused path's nodal arrays in the element real type
template <typename T>
void fused_node_arrays(wfx_ctx *c, T *&v, T *&pa, T *&ud, T *&fi) {
  if constexpr (std::is_same<T, double>::value) {
    v = c->nd.v; pa = c->nd.prev_a; ud = c->nd.u_dt; fi = c->nd.fi;
  } else {
    v = c->v32; pa = c->pa32; ud = c->ud32; fi = c->fi32;
  }
}
template <typename T>
FusedParams element_params(wfx_ctx *c, const double *dtp) {
  auto &el = elem<T>(c);
  const auto &P = c->prm;
  const auto &st = P.stab;
  FusedParams fp;
  fp.dt = P.dt;
  fp.mp = mat_params(c);
  fp.pp = press_params(c);
  fp.need_jlocal = press_needs_jlocal(fp.pp);
  fp.av_al = st.artifvisc0;
  fp.av_be = st.artifvisc1;
  fp.avq = el.avq;
  fp.hg_coeff = (c->n == 8) ? st.hg_coeff : 0.0;
  fp.cs0 = P.mat.cs0;
  fp.rho_u = c->rho_uniform;
  fp.dtp = dtp;
  fp.plheat_frac = c->thermal.plheat_frac;
  fp.k_T = c->thermal.k_T;
  fp.cp_T = c->thermal.cp_T;
  const bool texp = c->thermal.on && c->thermal.exp_T != 0.0;
  fp.exp_T = c->thermal.exp_T;
  fp.texp = texp ? el.texp : nullptr;
  fp.dte_flat = texp ? el.dte_flat : nullptr;
  fp.flat_base = c->ms.flat_base;
  fp.mdiag = c->nd.mdiag;
  fp.write_out = c->fused_write_out;
  return fp;
}
// F3 (PAIR: with F2 in its staging); dtp: the step's dt on the device, or null
template <typename T, bool PAIR>
hipError_t launch_element_pass(wfx_ctx *c, const double *dtp, const PairArgs &pr, hipStream_t s) {
  auto &el = elem<T>(c);
  T *vN, *paN, *udN, *fiN;
  fused_node_arrays<T>(c, vN, paN, udN, fiN);
  const FusedParams fp = element_params<T>(c, dtp);
  const bool rate = law_class(fp.mp.model) == LAW_RATE, th = c->thermal.on;
  auto kern = f3_pick<T, PAIR, true>(c->n, c->one_slot, rate, th);
  if constexpr (!PAIR)
    if (!c->stream_step) kern = f3_pick<T, false, false>(c->n, false, rate, th);
  const int bs = PAIR && c->n == 8 && !c->one_slot ? 2 * kCluster : kCluster;
  hipLaunchKernelGGL(kern, dim3(c->ms.ncl), dim3(bs), 0, s, c->E, c->N, fp, cluster_args(c), pr, c->nd.x, vN,
                     c->nd.anp_ratio, el.vol0, el.rho, el.sy0, el.He, el.tau,
                     c->fused_tau_out ? (T *)c->fused_tau_out : el.tau, el.eps, el.p, el.pl_strain,
                     c->fused_pl_out ? (T *)c->fused_pl_out : el.pl_strain, el.sigma_y, el.part, c->thermal.on ? el.q_plheat : (T *)nullptr);
  return hipGetLastError();
}

// F1, with the edge minima of the per-step CFL time step when cfl
template <typename T>
hipError_t launch_volumes(wfx_ctx *c, bool cfl, hipStream_t s) {
  auto &el = elem<T>(c);
  const bool texp = c->thermal.on && c->thermal.exp_T != 0.0;
  auto kern = c->n == 8 ? f1_cluster<T, 8> : f1_cluster<T, 4>;
  hipLaunchKernelGGL(kern, dim3(c->ms.ncl), dim3(kCluster), 0, s, c->E, cluster_args(c), c->nd.x, c->N, el.vol,
                     cfl ? c->cfl_part : (double *)nullptr, c->status, el.dte_flat, texp ? el.texp : (T *)nullptr);
  return hipGetLastError();
}

// ---- paired passes: two kernels per step ------------------------------------
template <typename T>
PairArgs pair_args(wfx_ctx *c, int step) {
  PairArgs pr{};
  pr.rec = c->ms.srec;
  pr.sent = c->ms.sent;
  pr.pw = c->ms.pw;
  pr.lanes = c->f2_lanes;
  pr.vol = elem<T>(c).vol;
  pr.vsum0 = c->nd.voln0_sum;
  pr.rho_avg = c->nd.rho_avg;
  pr.sbc = c->ms.sbc;
  pr.ratio = c->nd.anp_ratio;
  pr.mdiag = c->nd.mdiag;
  pr.cr = cfl_args(c, c->prm.cfl, c->ms.ncl, step);
  return pr;
}

// nodal sums and element pass of one step (F2 + F3), and the contact forces
template <typename T>
hipError_t launch_pair_element(wfx_ctx *c, int step, hipStream_t s) {
  const bool cfl = c->prm.cfl > 0.0;
  if (cfl && c->contact.on) {  // calcMinEdgeLength also refreshes the element heights contact uses
    hipError_t e = launch_elem_length(c, s);
    if (e != hipSuccess) return e;
  }
  hipError_t e = launch_element_pass<T, true>(c, nullptr, pair_args<T>(c, step), s);
  if (e != hipSuccess || !c->contact.on) return e;
  T *vN, *paN, *udN, *fiN;
  fused_node_arrays<T>(c, vN, paN, udN, fiN);
  return launch_contact<T>(c, vN, cfl, s);
}

template <typename T, int NN, bool CFL, bool CT, int SL>
auto f41_pick(bool th) {
  return th ? f41_cluster<T, NN, CFL, CT, true, SL> : f41_cluster<T, NN, CFL, CT, false, SL>;
}
template <typename T, int NN, int SL>
auto f41_pick(bool cfl, bool ct, bool th) {
  return cfl ? (ct ? f41_pick<T, NN, true, true, SL>(th) : f41_pick<T, NN, true, false, SL>(th))
             : (ct ? f41_pick<T, NN, false, true, SL>(th) : f41_pick<T, NN, false, false, SL>(th));
}

// the context's nodal arrays and the other set change places
template <typename T>
void pair_swap(wfx_ctx *c) {
  std::swap(c->nd.x, c->x_b);
  auto swap_t = [](T *&a, void *&b) {
    T *q = a;
    a = static_cast<T *>(b);
    b = q;
  };
  if constexpr (std::is_same<T, double>::value) {
    swap_t(c->nd.v, c->v_b); swap_t(c->nd.prev_a, c->pa_b); swap_t(c->nd.u_dt, c->ud_b);
  } else {
    swap_t(c->v32, c->v_b); swap_t(c->pa32, c->pa_b); swap_t(c->ud32, c->ud_b);
  }
}

// node pass of one step and the next one's volumes (F4 + F1), the rigid
// surfaces' motion; the nodal arrays change places
template <typename T>
hipError_t launch_pair_node(wfx_ctx *c, hipStream_t s) {
  const bool cfl = c->prm.cfl > 0.0, ct = c->contact.on, th = c->thermal.on;
  auto &el = elem<T>(c);
  T *vN, *paN, *udN, *fiN;
  fused_node_arrays<T>(c, vN, paN, udN, fiN);
  NodeParams np = node_params(c, 1);
  np.dtp = cfl ? c->scalars + kCflDt : nullptr;
  np.vmax_part = c->cfl_part + c->cfl_cap_min;
  auto kern = c->n == 4      ? f41_pick<T, 4, 1>(cfl, ct, th)
              : c->one_slot ? f41_pick<T, 8, 1>(cfl, ct, th)
                            : f41_pick<T, 8, 2>(cfl, ct, th);
  hipLaunchKernelGGL(kern, dim3(c->ms.ncl + (ct ? 1 : 0)), dim3(c->one_slot ? kCluster : slot_cap(c->n)), 0, s, c->N, np, cluster_args(c), pair_args<T>(c, -1),
                     NodeSet{c->x_b, c->v_b, c->pa_b, c->ud_b}, c->contact.contforce, el.part, c->nd.fe,
                     c->nd.mdiag, c->bc_tab, fiN, vN, paN, udN, c->nd.x, c->status, c->nd.T, el.vol, c->cfl_part,
                     rigid_args(c, ct));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  if (cfl) c->cfl_nvmax = c->ms.ncl;
  pair_swap<T>(c);
  return hipSuccess;
}

// Step k by the paired passes from one step record to the next (the adjoint's
// recomputation, FP64): the nodal arrays, stress and plastic strain are read
// in `in` and written in `out`, the step's internal force, mass and nodal
// ratios go to `in`, so that nothing is copied.  first: the step's volumes are
// not there yet.
template <typename T>
hipError_t launch_recorded_step(wfx_ctx *c, int k, bool first, const StepRecord &in, const StepRecord &out,
                                hipStream_t s) {
  static_assert(std::is_same<T, double>::value, "the records hold doubles");
  auto &el = c->e64;
  DevNode nd = c->nd;
  double *x_b = c->x_b, *tau = el.tau, *ep = el.pl_strain;
  void *v_b = c->v_b, *pa_b = c->pa_b;
  c->nd.x = in.x; c->nd.v = in.v; c->nd.prev_a = in.pa;
  c->nd.fi = in.fi; c->nd.mdiag = in.m; c->nd.anp_ratio = in.r;
  c->x_b = out.x; c->v_b = out.v; c->pa_b = out.pa;
  el.tau = in.tau; el.pl_strain = in.ep;
  c->fused_tau_out = out.tau; c->fused_pl_out = out.ep;
  c->fused_write_out = 0;
  c->fused_read_ud = (k == 0 || c->prm.cfl > 0.0) ? 1 : 0;
  c->fused_write_ud = c->prm.cfl > 0.0 ? 1 : 0;
  c->fused_run_first = k == 0 ? 1 : 0;
  c->fused_run_last = 0;
  hipError_t e = first ? launch_volumes<T>(c, c->prm.cfl > 0.0, s) : hipSuccess;
  if (e == hipSuccess) e = launch_pair_element<T>(c, k, s);
  if (e == hipSuccess) e = launch_pair_node<T>(c, s);
  c->fused_write_out = c->fused_read_ud = c->fused_write_ud = c->fused_run_first = c->fused_run_last = 1;
  c->fused_tau_out = c->fused_pl_out = nullptr;
  el.tau = tau; el.pl_strain = ep;
  nd.u_dt = c->nd.u_dt;  // the increment's two buffers stay where the step left them
  c->nd = nd;
  c->x_b = x_b; c->v_b = v_b; c->pa_b = pa_b;
  return e;
}

template <typename T, int BS, bool CFL, bool CT>
auto f4_pick(bool th) {
  return th ? f4_node<T, BS, CFL, CT, true> : f4_node<T, BS, CFL, CT, false>;
}

template <typename T, int BS>
hipError_t launch_fused_phase_bs(wfx_ctx *c, int phase, int predict, int step, hipStream_t s) {
  // per-step CFL time step inside a run; otherwise (step < 0) the host's dt
  const bool cfl = step >= 0 && c->prm.cfl > 0.0;
  const double *dtp = cfl ? c->scalars + kCflDt : nullptr;
  auto &el = elem<T>(c);
  const auto &st = c->prm.stab;
  const int N = c->N, E = c->E;
  const int gN = (N + BS - 1) / BS;
  T *vN, *paN, *udN, *fiN;
  fused_node_arrays<T>(c, vN, paN, udN, fiN);
  const ClusterArgs ca = cluster_args(c);
  if (phase == 1) {
    hipError_t e = launch_volumes<T>(c, cfl, s);
    if (e != hipSuccess) return e;
    // calcMinEdgeLength also refreshes the element heights contact uses
    if (cfl && c->contact.on) return launch_elem_length(c, s);
  } else if (phase == 2) {
    // outside a run: after the densities changed, and in a capture, whose replays
    // may follow another change (a run forms the means when it starts)
    if (step < 0 && reads_means(c) && (!c->rho_avg_valid || is_capturing(s))) {
      hipError_t e = launch_run_sums<T>(c, false, s);
      if (e != hipSuccess) return e;
    }
    const CflReduce cr = cfl_args(c, cfl ? c->prm.cfl : 0.0, c->ms.ncl, step);
    const int more = cfl ? 1 : 0;
    if (c->f2_lanes) {
      const int gL = (int)(((long)N * kF2Lanes + BS - 1) / BS);
      hipLaunchKernelGGL((f2_nodal_lanes<T, BS>), dim3(gL + more), dim3(BS), 0, s, N, c->n, c->ms.nodel_offset,
                         c->ms.nodel_count, c->ms.nodel_pk, el.vol, c->nd.rho_avg, c->nd.voln0_sum, c->nd.anp_ratio,
                         c->nd.mdiag, c->rho_uniform, cr, el.rho);
    } else {
      auto kern = c->stream_step ? f2_nodal<T, BS, true> : f2_nodal<T, BS, false>;
      hipLaunchKernelGGL(kern, dim3(gN + more), dim3(BS), 0, s, N, c->n, c->ms.nodel_offset,
                         c->ms.nodel_count, c->ms.nodel_pk, c->ms.nodel_pad, el.vol, c->nd.rho_avg, c->nd.voln0_sum,
                         c->nd.anp_ratio, c->nd.mdiag, c->rho_uniform, cr, el.rho);
    }
  } else if (phase == 3) {
    hipError_t e = launch_element_pass<T, false>(c, dtp, PairArgs{}, s);
    if (e != hipSuccess) return e;
    // contact forces after the element forces, before the assembly
    if (c->contact.on) return launch_contact<T>(c, vN, cfl, s);
  } else if (phase == 4) {
    NodeParams np = node_params(c, predict);
    np.dtp = dtp;
    np.vmax_part = cfl ? c->cfl_part + c->cfl_cap_min : nullptr;
    if (cfl && predict) c->cfl_nvmax = gN;
    const bool ct = c->contact.on, th = c->thermal.on;
    auto kern = cfl ? (ct ? f4_pick<T, BS, true, true>(th) : f4_pick<T, BS, true, false>(th))
                    : (ct ? f4_pick<T, BS, false, true>(th) : f4_pick<T, BS, false, false>(th));
    const RigidArgs rg = rigid_args(c, ct && step >= 0);  // the rigid surfaces move after the position update
    hipLaunchKernelGGL(kern, dim3(gN + (rg.rn > 0 ? 1 : 0)), dim3(BS), 0, s, N, np, ca.nm, c->contact.contforce, c->ms.nsl_off, c->ms.nsl,
                       el.part, c->ms.nslot, c->nd.fe, c->nd.mdiag, c->bc_word, c->bc_tab, fiN, vN,
                       paN, udN, c->nd.x, c->nd.u, c->status, c->nd.T, rg);
  } else if (phase == 5) {
    const bool av = st.artifvisc0 != 0.0 || st.artifvisc1 != 0.0 || press_params(c).guard;
    hipLaunchKernelGGL((f_sigma<T>), dim3(nblocks(E)), dim3(kBlock), 0, s, E, el.p, el.tau, el.avq, el.vol,
                       (int)av, el.sigma);
    // the nodal volumes no step reads, once per run: the same CSR-order sum
    // and division as CalcNodalVol, so the field equals the per-step API's
    hipLaunchKernelGGL((k_nodal_vol<T>), dim3(nblocks(N)), dim3(kBlock), 0, s, N, c->ms.nodel_offset,
                       c->ms.nodel_count, c->ms.nodel_pad, c->ms.nodel_pk, el.vol, c->nd.voln, c->n);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

// step >= 0: step index within a run (per-step CFL slots); -1: host dt
template <typename T>
hipError_t launch_fused_phase(wfx_ctx *c, int phase, int predict, hipStream_t s, int step) {
  const int bs = (phase >= 1 && phase <= 4) ? c->fused_bs[phase] : 256;
  switch (bs) {
    case 64: return launch_fused_phase_bs<T, 64>(c, phase, predict, step, s);
    case 128: return launch_fused_phase_bs<T, 128>(c, phase, predict, step, s);
    case 512: return launch_fused_phase_bs<T, 512>(c, phase, predict, step, s);
    default: return launch_fused_phase_bs<T, 256>(c, phase, predict, step, s);
  }
}

// Per-step CFL time step at the start of a run: the predicted velocities'
// per-block largest speeds for the first step's dt; packed: a fused run's
// velocities as its node passes store them (FP32-mixed: the float copy, as
// the later steps' speeds are taken)
template <typename T>
hipError_t launch_cfl_begin(wfx_ctx *c, hipStream_t s, bool packed) {
  if (packed && !std::is_same<T, double>::value)
    hipLaunchKernelGGL((k_cfl_max_speed<float>), dim3(nblocks(c->N)), dim3(kBlock), 0, s, c->N, c->v32,
                       c->cfl_part + c->cfl_cap_min);
  else
    hipLaunchKernelGGL((k_cfl_max_speed<double>), dim3(nblocks(c->N)), dim3(kBlock), 0, s, c->N, c->nd.v,
                       c->cfl_part + c->cfl_cap_min);
  c->cfl_nvmax = nblocks(c->N);
  return hipGetLastError();
}

// The time step of one per-step API step (after the prediction and the
// Jacobians, Solver_explicit.C:576-600) into the dt slot.
template <typename T>
hipError_t launch_cfl_step(wfx_ctx *c, int step, hipStream_t s) {
  hipError_t e = launch_cfl_begin<T>(c, s, false);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_cfl_min_edge, dim3(nblocks(c->E)), dim3(kBlock), 0, s, c->E, c->N, c->ms.elnod, c->nd.x,
                     c->cfl_part);
  hipLaunchKernelGGL((k_cfl_reduce<T>), dim3(1), dim3(kCflReduceBlock), 0, s,
                     cfl_args(c, c->prm.cfl, nblocks(c->E), -1), elem<T>(c).rho);
  return hipGetLastError();
}

// ThermalCalcs of one per-step API step: element rates from the stored
// Jacobians, then the nodal update with the host's dt.  (The fused path
// folds both into its element and node passes.)
template <typename T>
hipError_t launch_thermal(wfx_ctx *c, hipStream_t s) {
  auto &el = elem<T>(c);
  const auto &th = c->thermal;
  auto kern = c->n == 8 ? k_thermal_elem<T, 8> : k_thermal_elem<T, 4>;
  const bool texp = th.on && th.exp_T != 0.0;
  hipLaunchKernelGGL(kern, dim3(nblocks(c->E)), dim3(kBlock), 0, s, c->E, c->ms.elnod, el.dH, el.detJ, el.vol,
                     el.q_plheat, c->nd.T, c->nd.mdiag, th.k_T, th.cp_T, el.dTedt, c->ms.flat_base, c->N,
                     texp ? el.dte_flat : (T *)nullptr);
  hipLaunchKernelGGL((k_thermal_node<T>), dim3(nblocks(c->N)), dim3(kBlock), 0, s, c->N, (long)c->E, c->n,
                     c->ms.nodel_offset, c->ms.nodel_count, c->ms.nodel_pk, c->ms.nodel_pad, el.dTedt, c->prm.dt,
                     c->nd.T, c->contact.on ? c->contact.q_cont : (const double *)nullptr, c->nd.mdiag, th.cp_T);
  return hipGetLastError();
}

// calcThermalExpansion of one per-step API step (no-op at exp_T = 0)
template <typename T>
hipError_t launch_thermal_expansion(wfx_ctx *c, hipStream_t s) {
  auto &el = elem<T>(c);
  if (c->thermal.exp_T == 0.0 || !el.dte_flat) return hipSuccess;
  auto kern = c->n == 8 ? k_thermal_expansion<T, 8> : k_thermal_expansion<T, 4>;
  hipLaunchKernelGGL(kern, dim3(nblocks(c->E)), dim3(kBlock), 0, s, c->E, c->ms.elnod, el.dte_flat, c->thermal.exp_T,
                     el.str_rate);
  return hipGetLastError();
}

// FP32-mixed runs keep the nodal velocity, previous acceleration and
// increment in float between the two; no-ops for FP64.
template <typename T>
hipError_t launch_fused_pack(wfx_ctx *c, hipStream_t s) {
  if constexpr (!std::is_same<T, double>::value) {
    const long n3 = 3L * c->N;
    hipLaunchKernelGGL(f_pack, dim3(nblocks(n3)), dim3(kBlock), 0, s, n3, c->nd.v, c->nd.prev_a, c->nd.u_dt,
                       c->nd.x, c->v32, c->pa32, c->ud32, c->x_start);
  }
  return hipGetLastError();
}
template <typename T>
hipError_t launch_fused_unpack(wfx_ctx *c, hipStream_t s) {
  if constexpr (!std::is_same<T, double>::value) {
    const long n3 = 3L * c->N;
    hipLaunchKernelGGL(f_unpack, dim3(nblocks(n3)), dim3(kBlock), 0, s, n3, c->v32, c->pa32, c->ud32, c->fi32,
                       c->nd.x, c->x_start, c->nd.v, c->nd.prev_a, c->nd.a, c->nd.u_dt, c->nd.fi, c->nd.u);
  }
  return hipGetLastError();
}

// The nodal arrays change places in every paired step but a run's last, whose
// node pass updates them in place; the first step's does too where that makes
// the changes even, so that a run ends in the arrays it started in (a captured
// run has their addresses in its kernels).
inline bool step_in_place(bool pair, int k, int nsteps) {
  return !pair || k + 1 == nsteps || (k == 0 && nsteps % 2 == 0);
}

// A failed launch leaves the nodal arrays in their places
template <typename T>
struct NodalPlaces {
  wfx_ctx *c;
  double *x;
  explicit NodalPlaces(wfx_ctx *c_) : c(c_), x(c_->nd.x) {}
  ~NodalPlaces() {
    if (c->nd.x != x) pair_swap<T>(c);
  }
};

// Steps [k, k + n) of a run, n > 0 and none of them the last, by the solo pass;
// rz: the first one's reaction record, or null
template <typename T>
hipError_t launch_solo_steps(wfx_ctx *c, int k, int n, void *rz, hipStream_t s) {
  static_assert(std::is_same<T, double>::value, "run_solo: FP64 only (a template, so that only its unit holds the kernels)");
  auto &el = elem<T>(c);
  T *vN, *paN, *udN, *fiN;
  fused_node_arrays<T>(c, vN, paN, udN, fiN);
  FusedParams fp = element_params<T>(c, nullptr);
  fp.write_out = 0;
  NodeParams np = node_params(c, 1);
  np.write_fi = np.write_ud = np.run_last = 0;
  np.run_first = np.read_ud = k == 0 ? 1 : 0;
  np.rz = rz;
  const bool rate = law_class(fp.mp.model) == LAW_RATE;
  auto kern = c->n == 8 ? (rate ? f_solo<T, 8, LAW_RATE> : f_solo<T, 8, LAW_PLAIN>)
                        : (rate ? f_solo<T, 4, LAW_RATE> : f_solo<T, 4, LAW_PLAIN>);
  hipLaunchKernelGGL(kern, dim3(c->ms.ncl), dim3(slot_cap(c->n)), 0, s, c->E, c->N, n, (size_t)c->react_n * sizeof(T), fp, np,
                     cluster_args(c), pair_args<T>(c, -1), c->nd.x, vN, paN, udN, c->nd.fe, c->bc_tab, el.vol0, el.rho,
                     el.sy0, el.He, el.tau, el.eps, el.pl_strain, c->status);
  return hipGetLastError();
}

// Step k of a run of nsteps; have_vol: the step before left this one's
// volumes (and whether this one leaves the next one's).  rz: the step's
// reaction record, or null.  ev: an event before each pass (separate passes).
template <typename T>
hipError_t launch_run_step(wfx_ctx *c, int k, int nsteps, bool pair, bool &have_vol, void *rz, hipStream_t s,
                           hipEvent_t *ev) {
  // the internal force and the element outputs are observed after the run
  c->fused_write_fi = (k + 1 == nsteps) ? 1 : 0;
  c->fused_write_out = (k + 1 == nsteps) ? 1 : 0;
  // the increment is predicted again from v' and prev_a after the first
  // step, unless each step has its own length
  c->fused_read_ud = (k == 0 || c->prm.cfl > 0.0) ? 1 : 0;
  c->fused_write_ud = c->prm.cfl > 0.0 ? 1 : 0;
  c->fused_run_first = k == 0 ? 1 : 0;
  c->fused_run_last = k + 1 == nsteps ? 1 : 0;
  const bool in_place = step_in_place(pair, k, nsteps);
  hipError_t e = hipSuccess;
  for (int ph = 1; ph <= 4 && e == hipSuccess; ++ph) {
    if (ev) e = hipEventRecord(ev[4 * k + ph - 1], s);
    if (e != hipSuccess || (ph == 1 && have_vol) || (ph == 2 && pair)) continue;
    c->fused_rz = ph == 4 ? rz : nullptr;
    if (ph == 1 && pair) e = launch_volumes<T>(c, c->prm.cfl > 0.0, s);
    else if (ph == 3 && pair) e = launch_pair_element<T>(c, k, s);
    else if (ph == 4 && !in_place) e = launch_pair_node<T>(c, s);
    else e = launch_fused_phase<T>(c, ph, k + 1 < nsteps, s, k);
  }
  have_vol = !in_place;
  c->fused_rz = nullptr;
  c->fused_write_fi = c->fused_write_out = c->fused_read_ud = c->fused_write_ud = 1;
  c->fused_run_first = c->fused_run_last = 1;
  return e;
}

template <typename T>
hipError_t launch_fused_steps(wfx_ctx *c, int nsteps, double *hist, hipStream_t s, hipEvent_t *ev) {
  const ReactRecord rec(c, hist, nsteps, sizeof(T));
  {
    hipError_t e = launch_fused_pack<T>(c, s);
    if (e != hipSuccess) return e;
  }
  if (c->prm.cfl > 0.0) {
    hipError_t e = launch_cfl_begin<T>(c, s, true);
    if (e != hipSuccess) return e;
  }
  const bool pair = run_paired(c) && !ev;  // with events the four passes run separately
  const NodalPlaces<T> places(c);
  bool have_vol = false;
  int k = 0;
  if constexpr (std::is_same<T, double>::value)
    while (!ev && run_solo(c) && k + 1 < nsteps) {  // all steps but the last
      // up to the row at which the reaction record is full
      int n = std::min(nsteps - 1 - k, kSoloSteps);
      if (rec.hist) n = std::min(n, c->react_rows - k % c->react_rows);
      hipError_t e = launch_solo_steps<T>(c, k, n, rec.row(k), s);
      k += n;
      if (e == hipSuccess && rec.full(k - 1)) e = launch_reaction_rows<T>(c, rec, k - 1, s);
      if (e != hipSuccess) return e;
    }
  for (; k < nsteps; ++k) {
    if (c->contact.on && (c->contact.step_count + k) % 10 == 0) {
      hipError_t e = launch_ext_face_areas(c, s);  // every 10 steps, at the step's start
      if (e != hipSuccess) return e;
    }
    const hipError_t e = launch_run_step<T>(c, k, nsteps, pair, have_vol, rec.row(k), s, ev);
    if (e != hipSuccess) return e;
    if (ev && k + 1 == nsteps) {
      hipError_t e = hipEventRecord(ev[4 * nsteps], s);
      if (e != hipSuccess) return e;
    }
    if (rec.full(k)) {
      hipError_t e = launch_reaction_rows<T>(c, rec, k, s);
      if (e != hipSuccess) return e;
    }
  }
  {
    hipError_t e = launch_fused_unpack<T>(c, s);
    if (e != hipSuccess) return e;
  }
  return launch_fused_phase<T>(c, 5, 0, s, -1);
}

}  // namespace wfx
