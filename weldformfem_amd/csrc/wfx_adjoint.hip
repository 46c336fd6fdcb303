// Hand-written adjoint of the explicit step with checkpointing.
//
// The step map differentiated here is the fused step (wfx_step_fused) seen
// from one step boundary to the next.  The state at boundary k is
//   Z_k = (x_k, v'_k, ud_k, pa_{k-1}, tau_k, ep_k)
// with v'_k and ud_k the predicted velocity (boundary values imposed) and
// displacement increment of step k, pa_{k-1} the previous corrected
// acceleration.  Within step k (Solver_explicit.C:524-978):
//   element pass   vol, dH, D, W, p(r), Jaumann + radial return, forces   (wfx_adjoint.hpp)
//   node pass      r_i = S_i / S0_i, m_i = (S_i / n) * mean rho_i, S_i = sum vol_e
//                  fi = sum_e fnet, a = (fe - fi)/m, a = 0 where v is prescribed
//                  a'' = (a - alpha pa)/(1 - alpha), v'' = BCV(v' + gamma dt a'')
//                  ud' = ud + beta dt^2 a'', x_{k+1} = x_k + ud', pa_k = a''
//                  ud_{k+1} = dt (v'' + (0.5 - beta) dt a''),
//                  v'_{k+1} = BCV(v'' + (1 - gamma) dt a'')
// The loss cotangent enters through the reaction history R_{k,g} = sum over
// group g of fi_z after assembly.
//
// Forward: the fused step is run as usual and the state is stored every K
// steps (checkpoints).  Backward: for each segment, last first, the state is
// restored from its checkpoint, the K steps are recomputed while their
// inputs (x, v', tau, ep) and node-pass values (fi, m, r) are recorded, and
// the segment is then reversed step by step with two kernels, each one
// work-group per element cluster over the nodes its elements touch (slots), as
// the paired forward passes:
//   a_element  node: the later step's position and velocity cotangents gathered
//              from the clusters' sums, then the node-pass reverse
//              (prediction, correction, BC masks, accel, reaction cotangent ->
//              fi and m cotangents); element reverse (recomputes the element
//              forward first); its position, velocity and ratio cotangents
//              summed per slot
//   a_volume   node: the ratio cotangents gathered, volume cotangent; element
//              volume cotangent -> positions, summed per slot
// A node of several clusters is worked on by each of them alike and stored by
// its first slot's, to a second set of buffers since the others still read.
// All adjoint arithmetic is FP64; the forward runs in the context's precision.
#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "../../include/wfx.h"
#include "wfx_adjoint.hpp"
#include "wfx_internal.hpp"
#include "wfx_kernels.hpp"
#include "wfx_launch.hpp"
#include "wfx_slots.hpp"

namespace wfx {

struct Adjoint {
  int nsteps = 0, every = 0, nck = 0, ng = 0, N = 0, E = 0, n = 0, precision = 0;
  bool recorded = false;
  size_t ck_stride = 0, slot_stride = 0;
  std::vector<void *> mem;
  double *ck = nullptr, *slot = nullptr, *hist = nullptr, *hbar = nullptr;
  double *bars[2] = {nullptr, nullptr};  // the state cotangents [x v ud pa][3][N], two sets
  double *taub = nullptr, *epb = nullptr, *mb = nullptr;
  double *p1[2] = {nullptr, nullptr}, *p2 = nullptr;  // per-slot sums (SlotSums)
  double *volb = nullptr, *grad = nullptr;
  double *sy0d = nullptr, *Hd = nullptr, *rhod = nullptr, *rho_avg = nullptr, *sums = nullptr;
  int *rgroup = nullptr;
  std::vector<std::pair<void *, size_t>> final_bufs;
  std::vector<void *> final_saved;
  // per-step CFL time step: each step's dt (device and host), the node and
  // element shares of its cotangent, and the arg-min edge / arg-max speed
  bool cfl = false;
  double *dts = nullptr, *dtb = nullptr, *cfl_loc = nullptr;
  double *lawc = nullptr;  // rate laws at per-element temperatures: their constants per element [5][E]
  std::vector<double> dts_h;
};

void adjoint_free(wfx_ctx *c) {
  if (!c->adj) return;
  for (void *p : c->adj->mem) (void)hipFree(p);
  for (void *p : c->adj->final_saved) (void)hipFree(p);
  delete c->adj;
  c->adj = nullptr;
}

namespace {

constexpr int kB = 256;
inline int nb(long n) { return (int)((n + kB - 1) / kB); }
__device__ __forceinline__ long tid() { return (long)blockIdx.x * blockDim.x + threadIdx.x; }

// ---- state transfer --------------------------------------------------------
// checkpoint [x 3N][v 3N][ud 3N][pa 3N][tau 6E][ep E] (ud is read back by
// the run's first step only: the later ones form it from v and pa)
template <typename T>
__global__ void k_ck_save(long N, long E, const double *x, const T *v, const T *ud, const T *pa, const T *tau,
                          const T *ep, double *dst) {
  long i = tid();
  const long n3 = 3 * N;
  if (i < n3) dst[i] = x[i];
  else if (i < 2 * n3) dst[i] = (double)v[i - n3];
  else if (i < 3 * n3) dst[i] = (double)ud[i - 2 * n3];
  else if (i < 4 * n3) dst[i] = (double)pa[i - 3 * n3];
  else if (i < 4 * n3 + 6 * E) dst[i] = (double)tau[i - 4 * n3];
  else if (i < 4 * n3 + 7 * E) dst[i] = (double)ep[i - 4 * n3 - 6 * E];
}
template <typename T>
__global__ void k_ck_load(long N, long E, const double *src, double *x, T *v, T *ud, T *pa, T *tau, T *ep) {
  long i = tid();
  const long n3 = 3 * N;
  if (i < n3) x[i] = src[i];
  else if (i < 2 * n3) v[i - n3] = (T)src[i];
  else if (i < 3 * n3) ud[i - 2 * n3] = (T)src[i];
  else if (i < 4 * n3) pa[i - 3 * n3] = (T)src[i];
  else if (i < 4 * n3 + 6 * E) tau[i - 4 * n3] = (T)src[i];
  else if (i < 4 * n3 + 7 * E) ep[i - 4 * n3 - 6 * E] = (T)src[i];
}
// step record [x 3N][v 3N][fi 3N][m N][r N][tau 6E][ep E][pa 3N]; the first
// part before the step's kernels, the node-pass values after them
template <typename T>
__global__ void k_rec_pre(long N, long E, const double *x, const T *v, const T *tau, const T *ep, const T *pa,
                          double *dst) {
  long i = tid();
  const long n3 = 3 * N, o = 11 * N;
  if (i < n3) dst[i] = x[i];
  else if (i < 2 * n3) dst[i] = (double)v[i - n3];
  else if (i < 2 * n3 + 6 * E) dst[o + i - 2 * n3] = (double)tau[i - 2 * n3];
  else if (i < 2 * n3 + 7 * E) dst[o + i - 2 * n3] = (double)ep[i - 2 * n3 - 6 * E];
  else if (i < 3 * n3 + 7 * E) dst[o + i - 2 * n3] = (double)pa[i - 2 * n3 - 7 * E];
}
// (the ANP ratio as the fused node pass leaves it: double, or for FP32-mixed
// 1 + a float deviation in the same buffer)
template <typename T>
__global__ void k_rec_post(long N, const T *fi, const double *m, const double *r, double *dst) {
  long i = tid();
  const long n3 = 3 * N;
  if (i < n3) dst[6 * N + i] = (double)fi[i];
  else if (i < n3 + N) dst[9 * N + i - n3] = m[i - n3];
  else if (i < n3 + 2 * N) {
    const long k = i - n3 - N;
    if constexpr (std::is_same<T, double>::value) dst[10 * N + k] = r[k];
    else dst[10 * N + k] = 1.0 + (double)reinterpret_cast<const float *>(r)[k];
  }
}

__global__ void k_zero(long n, double *p) {
  long i = tid();
  if (i < n) p[i] = 0.0;
}

// element parameters in FP64 and per-node mean density
template <typename T>
__global__ void k_prep_elem(int E, const T *sy0, const T *He, double H, const T *rho, double *sy0d,
                            double *Hd, double *rhod) {
  int e = (int)tid();
  if (e >= E) return;
  sy0d[e] = (double)sy0[e];
  Hd[e] = He ? (double)He[e] : H;
  rhod[e] = (double)rho[e];
}
__global__ void k_prep_node(int N, const int *off, const int *cnt, const int *pk, const double *rhod,
                            double *rho_avg) {
  int i = (int)tid();
  if (i >= N) return;
  double s = 0.0;
  for (int k = 0; k < cnt[i]; ++k) s += rhod[pk[off[i] + k] >> 3];
  rho_avg[i] = cnt[i] > 0 ? s / cnt[i] : 0.0;
}

struct NodeAdj {
  double dt, alpha, beta, gamma;
  int has_fe, ng;
};

// the state cotangents [3][N] at a step boundary
struct Bars {
  double *x, *v, *ud, *pa;
};

// the slots' lists and the sums over them: P1 [7][S] of a_element (position,
// velocity, ratio), P2 [3][S] of a_volume (position); a slot's place is its own
// index or, node-major (nm), its place in its node's list
struct SlotSums {
  const int *nsl_off, *nsl, *spos;
  int nm, shift;  // shift: the entry table's byte offsets are for 4-byte values (1) or doubles (0)
  long S;
};
__device__ __forceinline__ int slot_at(const SlotSums &q, int o) { return q.nm ? o : q.nsl[o]; }
__device__ __forceinline__ bool first_slot(const SlotSums &q, int o, int slot) {
  return q.nm ? q.spos[slot] == o : q.nsl[o] == slot;
}

// node-pass reverse of step k for node i; Z-bar of boundary k+1 in, of
// boundary k out (partial: the element sums of this step are added by the
// next earlier step's call).  dtbar (per-step CFL time step): the node's share
// of the step length's cotangent, from vv = v' + gamma dt ac, ud = ud + beta
// dt^2 ac and the prediction ud' = dt (vv + (0.5 - beta) dt ac), v'' = vv +
// (1 - gamma) dt ac, with ac the corrected acceleration (1/(1-alpha)) (a - alpha pa)
struct NodeBack {
  double x[3], v[3], ud[3], pa[3], fib[3], mb, dtb;
};
struct NodeVals {
  double x[3], v[3], fi[3], fe[3], xb[3], vb[3], ud[3], pab[3], pa[3], m, r;
  int mask, rg;
};
__device__ __forceinline__ void load_node_vals(int i, long Ns, long Es, const NodeAdj &P, const double *rec,
                                               const double *fe, const int *bc_word, const int *rgroup, bool cfl,
                                               const Bars &in, NodeVals &s) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const long id = d * Ns + i;
    s.x[d] = rec[id];
    s.v[d] = rec[3 * Ns + id];
    s.fi[d] = rec[6 * Ns + id];
    s.pa[d] = cfl ? rec[11 * Ns + 7 * Es + id] : 0.0;
    s.fe[d] = P.has_fe ? fe[id] : 0.0;
    s.xb[d] = in.x[id];
    s.vb[d] = in.v[id];
    s.ud[d] = in.ud[id];
    s.pab[d] = in.pa[id];
  }
  s.m = rec[9 * Ns + i];
  s.r = rec[10 * Ns + i];
  s.mask = bc_word[i] & 7;
  s.rg = rgroup[i];
}
// the sums of one slot: position, velocity (P1) and position (P2)
__device__ __forceinline__ void load_sums(const SlotSums &q, const double *P1, const double *P2, int at,
                                          double (&p)[9]) {
#pragma unroll
  for (int u = 0; u < 6; ++u) p[u] = P1[u * q.S + at];
#pragma unroll
  for (int u = 0; u < 3; ++u) p[6 + u] = P2[u * q.S + at];
}
__device__ __forceinline__ void node_reverse(const NodeAdj &P, const NodeVals &s, double hbar, bool cfl,
                                             const double (&dx)[3], const double (&dv)[3], NodeBack &B) {
  const double m = s.m, dt = P.dt, ia = 1.0 / (1.0 - P.alpha);
  double mbar = 0.0, dtbar = 0.0;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const bool free_d = !((s.mask >> d) & 1);
    const double vp = s.vb[d] + dv[d], udp = s.ud[d], pa_in = s.pab[d], xbar = s.xb[d] + dx[d];
    const double vpm = free_d ? vp : 0.0;
    const double vpp = dt * udp + vpm;       // v'' after its boundary values
    const double vppr = free_d ? vpp : 0.0;  // v'' before them
    const double app = dt * dt * (0.5 - P.beta) * udp + (1.0 - P.gamma) * dt * vpm + pa_in +
                       P.gamma * dt * vppr + P.beta * dt * dt * xbar;
    B.x[d] = xbar;
    B.ud[d] = xbar;
    B.v[d] = vppr;
    B.pa[d] = -P.alpha * ia * app;
    const double abar = free_d ? app * ia : 0.0;
    const double a = (s.fe[d] - s.fi[d]) / m;
    B.fib[d] = -abar / m + (d == 2 ? hbar : 0.0);
    mbar -= abar * a / m;
    if (cfl) {
      const double ac = ia * ((free_d ? a : 0.0) - P.alpha * s.pa[d]);
      const double vv = free_d ? s.v[d] + P.gamma * dt * ac : s.v[d];  // an imposed v' is its value
      dtbar += udp * (vv + 2.0 * (0.5 - P.beta) * dt * ac) + vpm * (1.0 - P.gamma) * ac +
               vppr * P.gamma * ac + xbar * 2.0 * P.beta * dt * ac;
    }
  }
  B.mb = mbar;
  B.dtb = dtbar;
}

// Per-step CFL time step dt = cfl m / (cs + v), m the smallest edge of the
// first four nodes of every element (calcMinEdgeLength's edges, Domain_d.C:
// 2224-2260) and v the largest speed of the predicted velocities
// (Solver_explicit.C:576-600), both at the step's start.  One block finds an
// element edge of length m and a node of speed v (ties: the lowest index)
// from the step record: loc = {m, 6 e + edge, v, node}.
constexpr int kCflB = 1024;
__device__ const int kEdgePairs[6][2] = {{1, 0}, {2, 0}, {3, 0}, {2, 1}, {3, 1}, {3, 2}};
__global__ __launch_bounds__(kCflB) void a_cfl_locate(int E, int N, const int *elnod, const double *rec,
                                                       double *loc) {
  __shared__ double sv[kCflB];
  __shared__ long si[kCflB];
  const long Ns = N, Es = E;
  const double *x = rec, *v = rec + 3 * Ns;
  const int t = threadIdx.x;
  double m = 1.0e300;
  long mi = -1;
  for (int e = t; e < E; e += kCflB) {
    double P[4][3];
    for (int a = 0; a < 4; ++a) {
      const int g = elnod[a * Es + e];
      for (int c = 0; c < 3; ++c) P[a][c] = x[c * Ns + g];
    }
    for (int q = 0; q < 6; ++q) {
      const int a = kEdgePairs[q][0], b = kEdgePairs[q][1];
      const double ex = P[a][0] - P[b][0], ey = P[a][1] - P[b][1], ez = P[a][2] - P[b][2];
      const double len = sqrt(ex * ex + ey * ey + ez * ez);
      if (len < m) { m = len; mi = 6L * e + q; }
    }
  }
  double vm = -1.0;
  long vi = -1;
  for (int i = t; i < N; i += kCflB) {
    const double vx = v[i], vy = v[Ns + i], vz = v[2 * Ns + i];
    const double sp = sqrt(vx * vx + vy * vy + vz * vz);
    if (sp > vm) { vm = sp; vi = i; }
  }
  // (value, index) extremes over the block, the lower index on ties
  for (int pass = 0; pass < 2; ++pass) {
    const bool mn = pass == 0;
    sv[t] = mn ? m : vm;
    si[t] = mn ? mi : vi;
    __syncthreads();
    for (int h = kCflB / 2; h > 0; h >>= 1) {
      if (t < h) {
        const double a = sv[t], b = sv[t + h];
        const long ia = si[t], ib = si[t + h];
        const bool take = ib >= 0 && (ia < 0 || (mn ? (b < a || (b == a && ib < ia)) : (b > a || (b == a && ib < ia))));
        if (take) { sv[t] = b; si[t] = ib; }
      }
      __syncthreads();
    }
    if (t == 0) {
      loc[mn ? 0 : 2] = sv[0];
      loc[mn ? 1 : 3] = (double)si[0];
    }
    __syncthreads();
  }
}

// The step length's cotangent (node and element shares summed in a fixed
// order) passed on through dt = cfl m / (cs + v): dm-bar = dt-bar dt / m to the
// two nodes of the edge found, dv-bar = -dt-bar dt^2 / (cfl m) to the node found
// (cs + v = cfl m / dt).
__global__ __launch_bounds__(kCflB) void a_cfl_apply(int N, int E, double dt, double cfl, const double *dtb,
                                                      const double *loc, const int *elnod, const double *rec,
                                                      double *xb, double *vb) {
  __shared__ double sh[kCflB];
  const long Ns = N, Es = E;
  const int t = threadIdx.x;
  double s = 0.0;
  for (long k = t; k < Ns + Es; k += kCflB) s += dtb[k];
  sh[t] = s;
  __syncthreads();
  for (int h = kCflB / 2; h > 0; h >>= 1) {
    if (t < h) sh[t] += sh[t + h];
    __syncthreads();
  }
  if (t != 0) return;
  const double dtbar = sh[0], m = loc[0], vmax = loc[2];
  const long mi = (long)loc[1], vi = (long)loc[3];
  if (mi >= 0 && m > 0.0) {
    const long e = mi / 6;
    const int q = (int)(mi % 6);
    const int ga = elnod[kEdgePairs[q][0] * Es + e], gb = elnod[kEdgePairs[q][1] * Es + e];
    const double mbar = dtbar * dt / m;
    for (int c = 0; c < 3; ++c) {
      const double dx = rec[c * Ns + ga] - rec[c * Ns + gb];
      xb[c * Ns + ga] += mbar * dx / m;
      xb[c * Ns + gb] -= mbar * dx / m;
    }
  }
  if (vi >= 0 && vmax > 0.0 && m > 0.0) {
    const double vbar = -dtbar * dt * dt / (cfl * m);
    for (int c = 0; c < 3; ++c) vb[c * Ns + vi] += vbar * rec[3 * Ns + c * Ns + vi] / vmax;
  }
}

// The rate laws' temperature factors of each element at its own temperature
// (per-element temperatures, fixed during a run), as the forward forms them:
// Johnson-Cook 1 - T_h^m (Material.cuh:379-384); GMT at T clamped to
// [T_min, T_max]: C1 exp(C2 T), exp(C2 T), n1 T + n2, m1 T + m2, I1 T + I2
// (Material.cuh:441-444, :465-472).  lawc [5][E].
__global__ void k_law_temps(int E, int law, const double *Te, double T_t, double T_m, double mj, double C1,
                            double C2, double n1, double n2, double m1, double m2, double I1, double I2,
                            double T_min, double T_max, double *lawc) {
  int e = (int)tid();
  if (e >= E) return;
  const double T = Te[e];
  if (law == 2) {
    lawc[e] = 1.0 - pow((T - T_t) / (T_m - T_t), mj);
  } else {
    const double Tc = T < T_min ? T_min : (T > T_max ? T_max : T);
    lawc[e] = C1 * exp(C2 * Tc);
    lawc[E + e] = exp(C2 * Tc);
    lawc[2L * E + e] = n1 * Tc + n2;
    lawc[3L * E + e] = m1 * Tc + m2;
    lawc[4L * E + e] = I1 * Tc + I2;
  }
}

// Sums of R components per slot of the work-group's cluster from the
// element-node values in LDS (kEntStride), to P[R][S] (the element pass's sums)
template <int NN, int R>
__device__ __forceinline__ void slot_sums(const unsigned char *lds, const ClusterArgs &ca, const SlotSums &q,
                                          const ClusterDesc &cd, double *P) {
  const int s0 = cd.s0, M = cd.em >> 16;
  const uint16_t *lo = ca.goff + cd.goff;
  const uint2 *en = ca.ent + cd.ent;
  for (int j = threadIdx.x; j < M; j += kCluster) {
    const int at = q.nm ? q.spos[s0 + j] : s0 + j;
    double acc[R];
#pragma unroll
    for (int u = 0; u < R; ++u) acc[u] = 0.0;
    const int k1 = lo[j + 1];
    for (int k = lo[j]; k < k1; ++k) {
      const uint2 w = en[k];
      double v[4][R];
#pragma unroll
      for (int h = 0; h < 4; ++h) {
        const unsigned o = ((h < 2 ? w.x : w.y) >> (16 * (h & 1)) & 0xffffu) << q.shift;
#pragma unroll
        for (int u = 0; u < R; ++u)
          v[h][u] = *reinterpret_cast<const double *>(lds + o + u * (kEntStride(NN) * 8));
      }
#pragma unroll
      for (int h = 0; h < 4; ++h)
#pragma unroll
        for (int u = 0; u < R; ++u) acc[u] += v[h][u];
    }
#pragma unroll
    for (int u = 0; u < R; ++u) P[u * q.S + at] = acc[u];
  }
}

// The reverse step's first kernel.  LDS: the slots' nodal data (x, v', r and
// the fi cotangent), then the 7 n element-node values; 127 KB (hexahedra), so
// that every component is summed in one round: one work-group on a CU, which
// its registers (256 and 224 accumulation registers: the element's forward and
// reverse live together) allow no more of anyway.
// Before (node, element, node, element and node kernels with the element-node
// values in memory, 30^3 hexahedra): 5.0 + 17.7 + 6.0 + 9.9 + 8.0 us.
template <int NN>
__global__ __launch_bounds__(kCluster) void a_element(
    int E, int N, NodeAdj P, adj::ElemConst K, ClusterArgs ca, SlotSums q, const double *rec, const double *fe,
    const int *bc_word, const int *rgroup, const double *hbar_k, Bars in, Bars out, const double *P1in,
    const double *P2in, int pending, double *mb, double *dtb_n, const double *sy0d, const double *Hd,
    const double *rhod, double *taub, double *epb, double *P1, double *volb, double *grad, double *dtb_e,
    const double *lawc) {
  constexpr int cap = slot_cap(NN), kSl = kSlotsPerThread<NN>;
  __shared__ __align__(16) double lds[6 * kEntStride(NN) + NN * kCluster + 1];
  static_assert(10 * cap <= 6 * kEntStride(NN) + NN * kCluster, "the staged slots fit");
  const int c = xcd_block(), t = threadIdx.x;
  const ClusterDesc cd = ca.desc[c];
  const int e0 = cd.e0, s0 = cd.s0, ne = cd.em & 0xffff, M = cd.em >> 16;
  const long Es = E, Ns = N;
  const double *tau = rec + 11 * Ns, *ep = tau + 6 * Es;
  const int e = e0 + min(t, ne - 1);
  int ls[NN];
  load_lslot<NN>(ca.lslot + (long)(cd.lslot + min(t, ne - 1)) * NN, ls);
  int node[kSl], o[kSl], n[kSl];
#pragma unroll
  for (int k = 0; k < kSl; ++k) node[k] = ca.snode[s0 + min(t + k * kCluster, M - 1)];
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    o[k] = q.nsl_off[node[k]];
    n[k] = q.nsl_off[node[k] + 1] - o[k];
  }
  // every slot's loads before the first slot's arithmetic: the nodal values
  // and the first four of the later step's element sums (clusters in order)
  NodeVals nv[kSl];
  double p[kSl][4][9];
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    load_node_vals(node[k], Ns, Es, P, rec, fe, bc_word, rgroup, dtb_n != nullptr, in, nv[k]);
    if (pending)
#pragma unroll
      for (int g = 0; g < 4; ++g) load_sums(q, P1in, P2in, slot_at(q, o[k] + min(g, n[k] - 1)), p[k][g]);
  }
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    const int j = t + k * kCluster, i = node[k];
    const bool own = j < M && first_slot(q, o[k], s0 + min(j, M - 1));
    double dx[3] = {0.0, 0.0, 0.0}, dv[3] = {0.0, 0.0, 0.0};
    if (pending)
      for (int h = 0;;) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
          if (h + g < n[k])
#pragma unroll
            for (int u = 0; u < 3; ++u) {
              dx[u] += p[k][g][u] + p[k][g][6 + u];
              dv[u] += p[k][g][3 + u];
            }
        h += 4;
        if (h >= n[k]) break;
#pragma unroll
        for (int g = 0; g < 4; ++g) load_sums(q, P1in, P2in, slot_at(q, o[k] + min(h + g, n[k] - 1)), p[k][g]);
      }
    NodeBack B;
    node_reverse(P, nv[k], nv[k].rg >= 0 ? hbar_k[nv[k].rg] : 0.0, dtb_n != nullptr, dx, dv, B);
    if (own) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const long id = d * Ns + i;
        out.x[id] = B.x[d];
        out.v[id] = B.v[d];
        out.ud[id] = B.ud[d];
        out.pa[id] = B.pa[d];
      }
      mb[i] = B.mb;
      if (dtb_n) dtb_n[i] = B.dtb;
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      lds[d * cap + j] = nv[k].x[d];
      lds[(3 + d) * cap + j] = nv[k].v[d];
      lds[(7 + d) * cap + j] = B.fib[d];
    }
    lds[6 * cap + j] = nv[k].r;
  }
  __syncthreads();
  adj::ElemIn<NN> ei;
  double fb[NN][3];
#pragma unroll
  for (int a = 0; a < NN; ++a) {
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      ei.X[a][d] = lds[d * cap + ls[a]];
      ei.V[a][d] = lds[(3 + d) * cap + ls[a]];
      fb[a][d] = lds[(7 + d) * cap + ls[a]];
    }
    ei.r[a] = lds[6 * cap + ls[a]];
  }
  __syncthreads();
  if (t < ne) {
    if (lawc) {  // the element's own temperature factors
      if (K.law == 2) {
        K.jsoft = lawc[e];
      } else {
        K.ga = lawc[e];
        K.gexp = lawc[E + e];
        K.gn = lawc[2L * E + e];
        K.gm = lawc[3L * E + e];
        K.gi = lawc[4L * E + e];
      }
    }
    double tb[6];
    for (int k = 0; k < 6; ++k) {
      ei.tau[k] = tau[k * Es + e];
      tb[k] = taub[k * Es + e];
    }
    ei.ep = ep[e];
    ei.rho = rhod[e];
    ei.sy0 = sy0d[e];
    ei.H = Hd[e];
    adj::ElemFwd<NN> F;
    adj::elem_forward<NN>(K, ei, F);
    adj::ElemBar<NN> B;
    adj::elem_reverse<NN>(K, ei, F, fb, tb, epb[e], B);
    for (int k = 0; k < 6; ++k) taub[k * Es + e] = B.tau[k];
    epb[e] = B.ep;
    volb[e] = B.volb;
    if (dtb_e) dtb_e[e] = B.dt;
    // rows: the law's two parameters (bilinear sy0, H; Hollomon Kh, mh;
    // Johnson-Cook A, B; GMT C1, n2), hg
    grad[e] += K.law == 1 ? B.Kh : B.sy0;
    grad[Es + e] += K.law == 1 ? B.mh : B.H;
    grad[2 * Es + e] += B.hg;
#pragma unroll
    for (int a = 0; a < NN; ++a) {
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        lds[d * kEntStride(NN) + a * kCluster + t] = B.X[a][d];
        lds[(3 + d) * kEntStride(NN) + a * kCluster + t] = B.V[a][d];
      }
      lds[6 * kEntStride(NN) + a * kCluster + t] = B.r[a];
    }
  }
  if (t < 7) lds[t * kEntStride(NN) + NN * kCluster] = 0.0;
  __syncthreads();
  slot_sums<NN, 7>(reinterpret_cast<const unsigned char *>(lds), ca, q, cd, P1);
}

// The reverse step's second kernel: the nodes' volume cotangents w (the ratio
// cotangents over S0_i, and the mass cotangent through rho V / n), each
// element's volume cotangent to its positions
template <int NN>
__global__ __launch_bounds__(kCluster) void a_volume(int E, int N, ClusterArgs ca, SlotSums q, const double *rec,
                                                     const double *P1, const double *vsum0, const double *mb,
                                                     const double *rho_avg, const double *volb, double *P2) {
  constexpr int cap = slot_cap(NN), kSl = kSlotsPerThread<NN>;
  __shared__ __align__(16) double lds[2 * kEntStride(NN) + NN * kCluster + 1];
  const int c = xcd_block(), t = threadIdx.x;
  const ClusterDesc cd = ca.desc[c];
  const int e0 = cd.e0, s0 = cd.s0, ne = cd.em & 0xffff, M = cd.em >> 16;
  const long Ns = N;
  const int e = e0 + min(t, ne - 1);
  int ls[NN];
  load_lslot<NN>(ca.lslot + (long)(cd.lslot + min(t, ne - 1)) * NN, ls);
  double vb = volb[e];
  // as in a_element: every slot's loads first
  int node[kSl], o[kSl], n[kSl];
#pragma unroll
  for (int k = 0; k < kSl; ++k) node[k] = ca.snode[s0 + min(t + k * kCluster, M - 1)];
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    o[k] = q.nsl_off[node[k]];
    n[k] = q.nsl_off[node[k] + 1] - o[k];
  }
  double x[kSl][3], v0[kSl], mbk[kSl], ra[kSl], p[kSl][4];
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
#pragma unroll
    for (int d = 0; d < 3; ++d) x[k][d] = rec[d * Ns + node[k]];
    v0[k] = vsum0[node[k]];
    mbk[k] = mb[node[k]];
    ra[k] = rho_avg[node[k]];
#pragma unroll
    for (int g = 0; g < 4; ++g) p[k][g] = P1[6 * q.S + slot_at(q, o[k] + min(g, n[k] - 1))];
  }
#pragma unroll
  for (int k = 0; k < kSl; ++k) {
    const int j = t + k * kCluster;
    double rs = 0.0;
    for (int h = 0;;) {
#pragma unroll
      for (int g = 0; g < 4; ++g)
        if (h + g < n[k]) rs += p[k][g];
      h += 4;
      if (h >= n[k]) break;
#pragma unroll
      for (int g = 0; g < 4; ++g) p[k][g] = P1[6 * q.S + slot_at(q, o[k] + min(h + g, n[k] - 1))];
    }
#pragma unroll
    for (int d = 0; d < 3; ++d) lds[d * cap + j] = x[k][d];
    lds[3 * cap + j] = rs / v0[k] + mbk[k] * ra[k] / NN;
  }
  __syncthreads();
  double X[NN][3];
#pragma unroll
  for (int a = 0; a < NN; ++a) {
#pragma unroll
    for (int d = 0; d < 3; ++d) X[a][d] = lds[d * cap + ls[a]];
    vb += lds[3 * cap + ls[a]];
  }
  __syncthreads();
  if (t < ne) {
    double Xb[NN][3];
    adj::vol_reverse<NN>(X, vb, Xb);
#pragma unroll
    for (int a = 0; a < NN; ++a)
#pragma unroll
      for (int d = 0; d < 3; ++d) lds[d * kEntStride(NN) + a * kCluster + t] = Xb[a][d];
  }
  if (t < 3) lds[t * kEntStride(NN) + NN * kCluster] = 0.0;
  __syncthreads();
  slot_sums<NN, 3>(reinterpret_cast<const unsigned char *>(lds), ca, q, cd, P2);
}

// parameter gradients: one work-group per parameter row, fixed order; for
// the bilinear law the tangent-modulus row is converted from H to Et on the
// way (H = E Et/(E - Et), dH/dEt = (E + H)^2 / E^2)
__global__ void a_reduce(int E, double Emod, int bilinear, const double *grad, const double *Hd, double *gEt,
                         double *out) {
  __shared__ double sh[1024];
  const int row = blockIdx.x;
  double s = 0.0;
  for (int e = threadIdx.x; e < E; e += blockDim.x) {
    double g = grad[(long)row * E + e];
    if (row == 1) {
      if (bilinear) {
        const double f = (Emod + Hd[e]) / Emod;
        g *= f * f;
      }
      gEt[e] = g;
    }
    s += g;
  }
  sh[threadIdx.x] = s;
  __syncthreads();
  for (int k = blockDim.x / 2; k > 0; k >>= 1) {
    if ((int)threadIdx.x < k) sh[threadIdx.x] += sh[threadIdx.x + k];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[row] = sh[0];
}

}  // namespace

std::vector<std::pair<void *, size_t>> fused_state_buffers(wfx_ctx *c);

}  // namespace wfx

using namespace wfx;

#define REQUIRE(cond, code, msg)        \
  do {                                  \
    if (!(cond)) {                      \
      wfx::set_error(msg);              \
      return code;                      \
    }                                   \
  } while (0)
#define LAUNCH(expr) WFX_CHECK_HIP(expr)

static hipStream_t as_stream(wfx_stream s) { return (hipStream_t)s; }

template <typename T>
static hipError_t node_arrays(wfx_ctx *c, T **v, T **ud, T **pa, T **fi) {
  if constexpr (std::is_same<T, double>::value) {
    *v = c->nd.v; *ud = c->nd.u_dt; *pa = c->nd.prev_a; *fi = c->nd.fi;
  } else {
    *v = c->v32; *ud = c->ud32; *pa = c->pa32; *fi = c->fi32;
  }
  return hipSuccess;
}

template <typename T>
static DevElem<T> &el_of(wfx_ctx *c);
template <> DevElem<double> &el_of<double>(wfx_ctx *c) { return c->e64; }
template <> DevElem<float> &el_of<float>(wfx_ctx *c) { return c->e32; }

static int check_supported(wfx_ctx *c) {
  const Stab &s = c->prm.stab;
  REQUIRE(c->prm.mat.model == WFX_BILINEAR || c->prm.mat.model == WFX_HOLLOMON ||
              c->prm.mat.model == WFX_JOHNSON_COOK || c->prm.mat.model == WFX_GMT,
          WFX_ERR_STATE, "the adjoint supports the bilinear, Hollomon, Johnson-Cook and GMT materials");
  // thermal coupling one way: the temperatures follow the mechanics, which do
  // not read them when the law ignores temperature and nothing expands, so
  // the mechanical adjoint is the whole one
  REQUIRE(!c->thermal.on || ((c->prm.mat.model == WFX_BILINEAR || c->prm.mat.model == WFX_HOLLOMON) &&
                             c->thermal.exp_T == 0.0),
          WFX_ERR_STATE,
          "the adjoint covers thermal coupling only with a law that ignores temperature and no thermal expansion");
  REQUIRE(!c->contact.on, WFX_ERR_STATE, "the adjoint does not cover contact");
  REQUIRE(s.alpha_free == 0.0 && s.log_factor == 0.0 && s.J_min == 0.0 && s.hg_coeff_free == 0.0 &&
              s.pspg_scale == 0.0 && s.p_pspg_bulkfac == 0.0 && s.av_coeff_div == 0.0 && s.av_coeff_bulk == 0.0 &&
              s.artifvisc0 == 0.0 && s.artifvisc1 == 0.0,
          WFX_ERR_STATE, "the adjoint supports the ANP pressure without stabilisation terms");
  return WFX_OK;
}

static int adj_alloc(wfx_ctx *c, int nsteps, int every) {
  const long N = c->N, E = c->E, n = c->n;
  const int ng = c->ngroups > 0 ? c->ngroups : 1;
  const int nck = (nsteps + every - 1) / every;
  Adjoint *B = c->adj;
  const bool reuse = B && B->nsteps == nsteps && B->every == every && B->ng == ng && B->N == N && B->E == E &&
                     B->precision == c->precision;  // same run shape (identification loops)
  if (!reuse) {
    adjoint_free(c);
    Adjoint *A = new Adjoint();
    c->adj = A;
    A->nsteps = nsteps; A->every = every; A->nck = nck; A->ng = ng;
    A->N = (int)N; A->E = (int)E; A->n = (int)n; A->precision = c->precision;
    A->ck_stride = 12 * N + 7 * E;
    A->slot_stride = 14 * N + 7 * E;
    hipError_t err = hipSuccess;
    auto get = [&](double **p, size_t count) {
      if (err != hipSuccess) return;
      void *q = nullptr;
      err = hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(double));
      if (err == hipSuccess) { A->mem.push_back(q); *p = (double *)q; }
    };
    get(&A->ck, A->ck_stride * nck);
    get(&A->slot, A->slot_stride * (every + 1));  // and the state after a segment's last step
    get(&A->hist, (size_t)nsteps * ng);
    get(&A->hbar, (size_t)nsteps * ng);
    const long S = c->ms.nslot;
    get(&A->bars[0], 12 * N); get(&A->bars[1], 12 * N);
    get(&A->taub, 6 * E); get(&A->epb, E); get(&A->mb, N);
    get(&A->p1[0], 7 * S); get(&A->p1[1], 7 * S); get(&A->p2, 3 * S); get(&A->volb, E); get(&A->grad, 3 * E);
    get(&A->sy0d, E); get(&A->Hd, E); get(&A->rhod, E); get(&A->rho_avg, N); get(&A->sums, 8 + E);
    get(&A->dts, nsteps); get(&A->dtb, N + E); get(&A->cfl_loc, 8); get(&A->lawc, 5 * E);
    // summed whole (a_cfl_apply), but written for the nodes of some cluster only:
    // a node of no element has no share
    if (err == hipSuccess) err = hipMemset(A->dtb, 0, (size_t)(N + E) * sizeof(double));
    if (err == hipSuccess) {
      void *q = nullptr;
      err = hipMalloc(&q, std::max<long>(N, 1) * sizeof(int));
      if (err == hipSuccess) { A->mem.push_back(q); A->rgroup = (int *)q; }
    }
    // buffers saved at the end of the forward run and restored after the backward
    if (err == hipSuccess) A->final_bufs = fused_state_buffers(c);
    for (size_t k = 0; k < A->final_bufs.size() && err == hipSuccess; ++k) {
      void *q = nullptr;
      err = hipMalloc(&q, A->final_bufs[k].second);
      if (err == hipSuccess) A->final_saved.push_back(q);
    }
    if (err != hipSuccess) {
      adjoint_free(c);
      WFX_CHECK_HIP(err);
    }
  }
  Adjoint *A = c->adj;
  A->recorded = false;
  // node -> reaction group (each node in at most one group)
  std::vector<int> rg(N, -1);
  for (int g = 0; g + 1 < (int)c->react_off_h.size(); ++g)
    for (int k = c->react_off_h[g]; k < c->react_off_h[g + 1]; ++k) {
      const int node = c->react_h[k];
      if (rg[node] != -1) {
        set_error("the adjoint needs every reaction node in at most one group, once");
        return WFX_ERR_STATE;
      }
      rg[node] = g;
    }
  WFX_CHECK_HIP(hipMemcpy(A->rgroup, rg.data(), N * sizeof(int), hipMemcpyHostToDevice));
  return WFX_OK;
}

template <typename T>
static hipError_t save_ck(wfx_ctx *c, int idx, hipStream_t st) {
  Adjoint *A = c->adj;
  T *v, *ud, *pa, *fi;
  node_arrays<T>(c, &v, &ud, &pa, &fi);
  auto &el = el_of<T>(c);
  const long N = c->N, E = c->E;
  hipLaunchKernelGGL((k_ck_save<T>), dim3(nb(A->ck_stride)), dim3(kB), 0, st, N, E, c->nd.x, v, ud, pa, el.tau,
                     el.pl_strain, A->ck + (size_t)idx * A->ck_stride);
  return hipGetLastError();
}

template <typename T>
static hipError_t load_ck(wfx_ctx *c, int idx, hipStream_t st) {
  Adjoint *A = c->adj;
  T *v, *ud, *pa, *fi;
  node_arrays<T>(c, &v, &ud, &pa, &fi);
  auto &el = el_of<T>(c);
  const long N = c->N, E = c->E;
  hipLaunchKernelGGL((k_ck_load<T>), dim3(nb(A->ck_stride)), dim3(kB), 0, st, N, E,
                     A->ck + (size_t)idx * A->ck_stride, c->nd.x, v, ud, pa, el.tau, el.pl_strain);
  return hipGetLastError();
}

// one fused step (phases 1..4); rec != nullptr records its inputs and node
// values.  As in a fused run, only the run's first step reads the predicted
// increment (the node pass forms it again from v' and prev_a after that), so
// a segment recomputed from its checkpoint repeats the forward bit for bit.
// With the per-step CFL time step (step k >= 0) each step forms its dt on the
// device as a fused run does, and reads and stores the increment every step.
template <typename T>
static hipError_t fused_step(wfx_ctx *c, int predict, int k, bool last, double *rec, hipStream_t st) {
  T *v, *ud, *pa, *fi;
  node_arrays<T>(c, &v, &ud, &pa, &fi);
  auto &el = el_of<T>(c);
  const long N = c->N, E = c->E;
  const bool cfl = c->adj->cfl;
  if (rec) {
    hipLaunchKernelGGL((k_rec_pre<T>), dim3(nb(9 * N + 7 * E)), dim3(kB), 0, st, N, E, c->nd.x, v, el.tau,
                       el.pl_strain, pa, rec);
  }
  c->fused_read_ud = (k == 0 || cfl) ? 1 : 0;
  c->fused_run_first = k == 0 ? 1 : 0;
  c->fused_run_last = last ? 1 : 0;
  c->fused_write_ud = cfl ? 1 : 0;
  hipError_t e = hipSuccess;
  for (int ph = 1; ph <= 4 && e == hipSuccess; ++ph) e = launch_fused_phase<T>(c, ph, predict, st, cfl ? k : -1);
  c->fused_read_ud = c->fused_write_ud = c->fused_run_first = c->fused_run_last = 1;
  if (e != hipSuccess) return e;
  if (rec) {
    hipLaunchKernelGGL((k_rec_post<T>), dim3(nb(5 * N)), dim3(kB), 0, st, N, fi, c->nd.mdiag, c->nd.anp_ratio,
                       rec);
  }
  return hipGetLastError();
}

// The two sets of nodal arrays in the places they had (a run of paired steps
// ends so by itself; a failed one, or one record by record, does not)
struct KeepPlaces {
  wfx_ctx *c;
  double *x, *v, *pa, *ud, *x_b;
  float *v32, *pa32, *ud32;
  void *v_b, *pa_b, *ud_b;
  explicit KeepPlaces(wfx_ctx *q)
      : c(q), x(q->nd.x), v(q->nd.v), pa(q->nd.prev_a), ud(q->nd.u_dt), x_b(q->x_b), v32(q->v32), pa32(q->pa32),
        ud32(q->ud32), v_b(q->v_b), pa_b(q->pa_b), ud_b(q->ud_b) {}
  ~KeepPlaces() {
    c->nd.x = x; c->nd.v = v; c->nd.prev_a = pa; c->nd.u_dt = ud; c->x_b = x_b;
    c->v32 = v32; c->pa32 = pa32; c->ud32 = ud32;
    c->v_b = v_b; c->pa_b = pa_b; c->ud_b = ud_b;
  }
};

template <typename T>
static int adjoint_forward(wfx_ctx *c, int nsteps, bool want_hist, hipStream_t st) {
  Adjoint *A = c->adj;
  LAUNCH(launch_vsum0<T>(c, st));
  LAUNCH(launch_update_prediction(c, st));
  for (int d = 0; d < 3; ++d) LAUNCH(launch_impose(c, d, false, st));
  LAUNCH(launch_fused_pack<T>(c, st));
  if (A->cfl) LAUNCH(launch_cfl_begin<T>(c, st, true));
  const ReactRecord rec(c, want_hist ? A->hist : nullptr, nsteps, sizeof(T));
  const KeepPlaces places(c);
  const bool pair = run_paired(c);
  bool have_vol = false;
  for (int k = 0; k < nsteps; ++k) {
    if (k % A->every == 0) LAUNCH(save_ck<T>(c, k / A->every, st));
    LAUNCH(launch_run_step<T>(c, k, nsteps, pair, have_vol, rec.row(k), st, nullptr));
    if (rec.full(k)) LAUNCH(launch_reaction_rows<T>(c, rec, k, st));
  }
  LAUNCH(launch_fused_unpack<T>(c, st));
  LAUNCH(launch_fused_phase<T>(c, 5, 0, st, -1));
  LAUNCH(launch_copy(c->nd.prev_a, c->nd.a, 3L * c->N, st));
  for (size_t k = 0; k < A->final_bufs.size(); ++k)
    WFX_CHECK_HIP(hipMemcpyAsync(A->final_saved[k], A->final_bufs[k].first, A->final_bufs[k].second,
                                 hipMemcpyDeviceToDevice, st));
  return WFX_OK;
}

template <typename T>
static int adjoint_backward(wfx_ctx *c, hipStream_t st) {
  Adjoint *A = c->adj;
  const int N = c->N, E = c->E, n = c->n;
  auto &el = el_of<T>(c);
  const auto &P = c->prm;
  hipLaunchKernelGGL(k_zero, dim3(nb(12L * N)), dim3(kB), 0, st, 12L * N, A->bars[0]);
  hipLaunchKernelGGL(k_zero, dim3(nb(6L * E)), dim3(kB), 0, st, 6L * E, A->taub);
  hipLaunchKernelGGL(k_zero, dim3(nb(E)), dim3(kB), 0, st, (long)E, A->epb);
  hipLaunchKernelGGL(k_zero, dim3(nb(3L * E)), dim3(kB), 0, st, 3L * E, A->grad);
  hipLaunchKernelGGL((k_prep_elem<T>), dim3(nb(E)), dim3(kB), 0, st, E, el.sy0, el.He, P.mat.H, el.rho, A->sy0d,
                     A->Hd, A->rhod);
  hipLaunchKernelGGL(k_prep_node, dim3(nb(N)), dim3(kB), 0, st, N, c->ms.nodel_offset, c->ms.nodel_count,
                     c->ms.nodel_pk, A->rhod, A->rho_avg);
  LAUNCH(hipGetLastError());
  adj::ElemConst K{P.dt, P.mat.G, P.mat.K, P.mat.cs0, P.stab.hg_coeff, n == 8};
  if (P.mat.model == WFX_HOLLOMON) {
    K.law = 1;
    K.Kh = P.mat.Kh;
    K.mh = P.mat.mh;
    K.eps0 = P.mat.eps0;
    K.eps1 = P.mat.eps1;
    K.sy0m = P.mat.sy0;
  } else if (P.mat.model == WFX_JOHNSON_COOK) {
    K.law = 2;
    K.jB = P.mat.B;
    K.jn = P.mat.n;
    K.jC = P.mat.C;
    K.jeps0 = P.mat.eps_0;
    // the softening factor 1 - T_h^m of the uniform temperature (Material.cuh:379-384)
    K.jsoft = 1.0 - pow((P.mat.temp - P.mat.T_t) / (P.mat.T_m - P.mat.T_t), P.mat.m);
    K.jcap = P.mat.max_edot;
    K.Emod = P.mat.E;
  } else if (P.mat.model == WFX_GMT) {
    K.law = 3;
    // the temperature factors at the clamped uniform temperature (Material.cuh:441-444, :465-472)
    const double Tc = std::min(std::max(P.mat.temp, P.mat.T_min), P.mat.T_max);
    K.gexp = exp(P.mat.C2 * Tc);
    K.ga = P.mat.C1 * exp(P.mat.C2 * Tc);
    K.gn = P.mat.n1 * Tc + P.mat.n2;
    K.gm = P.mat.m1 * Tc + P.mat.m2;
    K.gi = P.mat.I1 * Tc + P.mat.I2;
    K.ge_min = P.mat.e_min;
    K.ge_max = P.mat.e_max;
    K.ger_min = P.mat.er_min;
    K.ger_max = P.mat.er_max;
    K.jcap = P.mat.max_edot;
  }
  // per-element temperatures: the rate laws' factors of every element
  const double *lawc = nullptr;
  if (c->temp_e && (K.law == 2 || K.law == 3)) {
    const Material &M = P.mat;
    hipLaunchKernelGGL(k_law_temps, dim3(nb(E)), dim3(kB), 0, st, E, K.law, c->temp_e, M.T_t, M.T_m, M.m, M.C1,
                       M.C2, M.n1, M.n2, M.m1, M.m2, M.I1, M.I2, M.T_min, M.T_max, A->lawc);
    LAUNCH(hipGetLastError());
    lawc = A->lawc;
  }
  // the recomputed steps read the nodal mean densities of the present densities
  if (!(c->rho_uniform > 0.0) && !c->rho_avg_valid) LAUNCH(launch_vsum0<T>(c, st));
  NodeAdj NP{P.dt, P.alpha, P.beta, P.gamma, c->has_fe, A->ng};
  const ClusterArgs ca = cluster_args(c);
  const SlotSums sums{c->ms.nsl_off, c->ms.nsl, c->ms.spos, c->ms.spos != nullptr, c->precision == WFX_FP64 ? 0 : 1,
                      c->ms.nslot};
  auto bars = [&](int k) {
    double *b = A->bars[k];
    return Bars{b, b + 3L * N, b + 6L * N, b + 9L * N};
  };
  const KeepPlaces places(c);
  auto record = [&](int j) {
    double *p = A->slot + (size_t)j * A->slot_stride;
    const long n3 = 3L * N, o = 11L * N;
    return StepRecord{p, p + n3, p + o + 7L * E, p + 2 * n3, p + 9L * N, p + 10L * N, p + o, p + o + 6L * E};
  };
  int cur = 0, pending = 0;
  for (int seg = A->nck - 1; seg >= 0; --seg) {
    const int k0 = seg * A->every, k1 = std::min(A->nsteps, k0 + A->every);
    LAUNCH(load_ck<T>(c, seg, st));
    if (A->cfl) LAUNCH(launch_cfl_begin<T>(c, st, true));  // the first recomputed step's largest speed
    if constexpr (std::is_same<T, double>::value) {
      if (run_paired(c)) {
        // the checkpoint's state into the first record, then from record to record
        const StepRecord r0 = record(0);
        hipLaunchKernelGGL((k_rec_pre<T>), dim3(nb(9L * N + 7L * E)), dim3(kB), 0, st, N, E, c->nd.x, c->nd.v, el.tau,
                           el.pl_strain, c->nd.prev_a, r0.x);
        LAUNCH(hipGetLastError());
        for (int k = k0; k < k1; ++k)
          LAUNCH(launch_recorded_step<T>(c, k, k == k0, record(k - k0), record(k - k0 + 1), st));
      }
    }
    if (!std::is_same<T, double>::value || !run_paired(c))
      for (int k = k0; k < k1; ++k)
        LAUNCH(fused_step<T>(c, k + 1 < A->nsteps, k, k + 1 == A->nsteps, A->slot + (size_t)(k - k0) * A->slot_stride,
                             st));
    for (int k = k1 - 1; k >= k0; --k) {
      const double *rec = A->slot + (size_t)(k - k0) * A->slot_stride;
      if (A->cfl) NP.dt = K.dt = A->dts_h[k];
      double *dtb_n = A->cfl ? A->dtb : nullptr, *dtb_e = A->cfl ? A->dtb + N : nullptr;
      const Bars in = bars(cur), out = bars(1 - cur);
      if (n == 8) {
        hipLaunchKernelGGL((a_element<8>), dim3(c->ms.ncl), dim3(kCluster), 0, st, E, N, NP, K, ca, sums, rec,
                           c->nd.fe, c->bc_word, A->rgroup, A->hbar + (size_t)k * A->ng, in, out, A->p1[1 - cur],
                           A->p2, pending, A->mb, dtb_n, A->sy0d, A->Hd, A->rhod, A->taub, A->epb, A->p1[cur],
                           A->volb, A->grad, dtb_e, lawc);
        hipLaunchKernelGGL((a_volume<8>), dim3(c->ms.ncl), dim3(kCluster), 0, st, E, N, ca, sums, rec, A->p1[cur],
                           c->nd.voln0_sum, A->mb, A->rho_avg, A->volb, A->p2);
      } else {
        hipLaunchKernelGGL((a_element<4>), dim3(c->ms.ncl), dim3(kCluster), 0, st, E, N, NP, K, ca, sums, rec,
                           c->nd.fe, c->bc_word, A->rgroup, A->hbar + (size_t)k * A->ng, in, out, A->p1[1 - cur],
                           A->p2, pending, A->mb, dtb_n, A->sy0d, A->Hd, A->rhod, A->taub, A->epb, A->p1[cur],
                           A->volb, A->grad, dtb_e, lawc);
        hipLaunchKernelGGL((a_volume<4>), dim3(c->ms.ncl), dim3(kCluster), 0, st, E, N, ca, sums, rec, A->p1[cur],
                           c->nd.voln0_sum, A->mb, A->rho_avg, A->volb, A->p2);
      }
      cur = 1 - cur;  // the cotangents and sums just written are the next step's inputs
      pending = 1;
      if (A->cfl) {  // the step length's dependence on x and v' at the step's start
        hipLaunchKernelGGL(a_cfl_locate, dim3(1), dim3(kCflB), 0, st, E, N, c->ms.elnod, rec, A->cfl_loc);
        hipLaunchKernelGGL(a_cfl_apply, dim3(1), dim3(kCflB), 0, st, N, E, A->dts_h[k], P.cfl, A->dtb, A->cfl_loc,
                           c->ms.elnod, rec, out.x, out.v);
      }
      LAUNCH(hipGetLastError());
    }
  }
  // the forward run's final state again
  for (size_t k = 0; k < A->final_bufs.size(); ++k)
    WFX_CHECK_HIP(hipMemcpyAsync(A->final_bufs[k].first, A->final_saved[k], A->final_bufs[k].second,
                                 hipMemcpyDeviceToDevice, st));
  LAUNCH(launch_copy(c->nd.prev_a, c->nd.a, 3L * c->N, st));
  hipLaunchKernelGGL(a_reduce, dim3(3), dim3(1024), 0, st, E, P.mat.E, P.mat.model == WFX_BILINEAR ? 1 : 0,
                     A->grad, A->Hd, A->sums + 8, A->sums);
  LAUNCH(hipGetLastError());
  return WFX_OK;
}

int wfx_adjoint_forward(wfx_ctx *c, int nsteps, int checkpoint_every, double *reaction_hist, wfx_stream s) {
  REQUIRE(c, WFX_ERR_ARG, "null context");
  REQUIRE(c->has_mesh && c->initialized, WFX_ERR_STATE, "call wfx_init first");
  REQUIRE(nsteps > 0 && checkpoint_every > 0, WFX_ERR_ARG, "nsteps and checkpoint_every must be positive");
  int rc = check_supported(c);
  if (rc) return rc;
  rc = adj_alloc(c, nsteps, checkpoint_every);
  if (rc) return rc;
  if (reaction_hist) {
    rc = ensure_react_ring(c);
    if (rc) return rc;
  }
  hipStream_t st = as_stream(s);
  Adjoint *A = c->adj;
  A->cfl = c->prm.cfl > 0.0;
  // each step's dt goes to the adjoint's own record (the per-step CFL reduction writes dt_hist[step])
  double *hist_keep = c->dt_hist;
  const int cap_keep = c->dt_cap;
  c->dt_hist = A->dts;
  c->dt_cap = nsteps;
  rc = c->precision == WFX_FP64 ? adjoint_forward<double>(c, nsteps, reaction_hist != nullptr, st)
                                : adjoint_forward<float>(c, nsteps, reaction_hist != nullptr, st);
  c->dt_hist = hist_keep;
  c->dt_cap = cap_keep;
  if (rc) return rc;
  c->fused_stale = true;
  if (A->cfl) {  // the host's dt follows the run's last step, as after a fused run
    A->dts_h.resize(nsteps);
    WFX_CHECK_HIP(hipMemcpyAsync(A->dts_h.data(), A->dts, nsteps * sizeof(double), hipMemcpyDeviceToHost, st));
    WFX_CHECK_HIP(hipStreamSynchronize(st));
    c->prm.dt = A->dts_h.back();
  }
  if (reaction_hist) {
    const size_t bytes = (size_t)nsteps * c->adj->ng * sizeof(double);
    if (c->ngroups > 0) WFX_CHECK_HIP(hipMemcpyAsync(reaction_hist, c->adj->hist, bytes, hipMemcpyDeviceToHost, st));
    else std::fill(reaction_hist, reaction_hist + (size_t)nsteps * c->adj->ng, 0.0);
  }
  WFX_CHECK_HIP(hipStreamSynchronize(st));
  c->adj->recorded = true;
  return WFX_OK;
}

int wfx_adjoint_backward(wfx_ctx *c, const double *reaction_hist_bar, double *grad, double *grad_sy0_elem,
                         double *grad_Et_elem, double *grad_hg_elem, wfx_stream s) {
  REQUIRE(c, WFX_ERR_ARG, "null context");
  REQUIRE(c->adj && c->adj->recorded, WFX_ERR_STATE, "call wfx_adjoint_forward first");
  REQUIRE(reaction_hist_bar && grad, WFX_ERR_ARG, "null argument");
  Adjoint *A = c->adj;
  REQUIRE(A->N == c->N && A->E == c->E && A->precision == c->precision, WFX_ERR_STATE,
          "mesh changed since wfx_adjoint_forward");
  REQUIRE(c->ngroups > 0, WFX_ERR_STATE, "no reaction nodes: the loss has no input");
  REQUIRE(A->ng == c->ngroups, WFX_ERR_STATE, "reaction groups changed since wfx_adjoint_forward");
  REQUIRE(A->cfl == (c->prm.cfl > 0.0), WFX_ERR_STATE, "the time-step rule changed since wfx_adjoint_forward");
  int rc = check_supported(c);
  if (rc) return rc;
  hipStream_t st = as_stream(s);
  WFX_CHECK_HIP(hipMemcpyAsync(A->hbar, reaction_hist_bar, (size_t)A->nsteps * A->ng * sizeof(double),
                               hipMemcpyHostToDevice, st));
  double *hist_keep = c->dt_hist;
  const int cap_keep = c->dt_cap;
  c->dt_hist = A->dts;
  c->dt_cap = A->nsteps;
  const double dt_keep = c->prm.dt;
  rc = c->precision == WFX_FP64 ? adjoint_backward<double>(c, st) : adjoint_backward<float>(c, st);
  c->dt_hist = hist_keep;
  c->dt_cap = cap_keep;
  c->prm.dt = dt_keep;
  if (rc) return rc;
  WFX_CHECK_HIP(hipMemcpyAsync(grad, A->sums, 3 * sizeof(double), hipMemcpyDeviceToHost, st));
  // per-element gradients: device rows in the stored (cluster) order, handed
  // back in the original element order
  const size_t E = (size_t)c->E, eb = E * sizeof(double);
  double *outs[3] = {grad_sy0_elem, grad_Et_elem, grad_hg_elem};
  const double *srcs[3] = {A->grad, A->sums + 8, A->grad + 2 * E};
  std::vector<double> rows[3];
  for (int k = 0; k < 3; ++k)
    if (outs[k]) {
      rows[k].resize(E);
      WFX_CHECK_HIP(hipMemcpyAsync(rows[k].data(), srcs[k], eb, hipMemcpyDeviceToHost, st));
    }
  WFX_CHECK_HIP(hipStreamSynchronize(st));
  for (int k = 0; k < 3; ++k)
    if (outs[k])
      for (size_t e = 0; e < E; ++e) outs[k][e] = rows[k][c->el_o2s[e]];
  return WFX_OK;
}

int wfx_adjoint_release(wfx_ctx *c) {
  REQUIRE(c, WFX_ERR_ARG, "null context");
  adjoint_free(c);
  return WFX_OK;
}
