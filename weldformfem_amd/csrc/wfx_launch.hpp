// Declarations of the kernel launchers.  The precision-dependent ones are
// defined (explicit specialisations) in wfx_k64.hip (double) and wfx_k32.hip
// (float); the nodal ones, which are precision independent, in wfx_k64.hip.
#pragma once

#include "wfx_internal.hpp"

namespace wfx {

template <typename T> hipError_t launch_elem_jacobians(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_elem_vol(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_elem_density(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_init_elem(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_scan_elem(wfx_ctx *c, unsigned long long *scan, hipStream_t s);
template <typename T> hipError_t launch_nodal_vol(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_nodal_mass(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_strain_rates(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_pressure(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_node_sums(wfx_ctx *c, hipStream_t s);  // CalcNodalVol, CalcNodalMassFromVol, ANP ratios
template <typename T> hipError_t launch_pressure_elem(wfx_ctx *c, hipStream_t s);  // the element part alone
template <typename T> hipError_t launch_stress_strain(wfx_ctx *c, double dt, hipStream_t s);
template <typename T> hipError_t launch_artificial_viscosity(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_elem_forces(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_hourglass(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_assembly(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_energies(wfx_ctx *c, double *dev_out2, double *partial, hipStream_t s);

#define WFX_DECLARE_SPECIALISATIONS(T)                                                          \
  template <> hipError_t launch_elem_jacobians<T>(wfx_ctx *, hipStream_t);                       \
  template <> hipError_t launch_elem_vol<T>(wfx_ctx *, hipStream_t);                             \
  template <> hipError_t launch_elem_density<T>(wfx_ctx *, hipStream_t);                         \
  template <> hipError_t launch_init_elem<T>(wfx_ctx *, hipStream_t);                            \
  template <> hipError_t launch_scan_elem<T>(wfx_ctx *, unsigned long long *, hipStream_t);      \
  template <> hipError_t launch_nodal_vol<T>(wfx_ctx *, hipStream_t);                            \
  template <> hipError_t launch_nodal_mass<T>(wfx_ctx *, hipStream_t);                           \
  template <> hipError_t launch_strain_rates<T>(wfx_ctx *, hipStream_t);                         \
  template <> hipError_t launch_pressure<T>(wfx_ctx *, hipStream_t);                             \
  template <> hipError_t launch_node_sums<T>(wfx_ctx *, hipStream_t);                            \
  template <> hipError_t launch_pressure_elem<T>(wfx_ctx *, hipStream_t);                        \
  template <> hipError_t launch_stress_strain<T>(wfx_ctx *, double, hipStream_t);                \
  template <> hipError_t launch_artificial_viscosity<T>(wfx_ctx *, hipStream_t);                 \
  template <> hipError_t launch_elem_forces<T>(wfx_ctx *, hipStream_t);                          \
  template <> hipError_t launch_hourglass<T>(wfx_ctx *, hipStream_t);                            \
  template <> hipError_t launch_assembly<T>(wfx_ctx *, hipStream_t);                             \
  template <> hipError_t launch_energies<T>(wfx_ctx *, double *, double *, hipStream_t);
WFX_DECLARE_SPECIALISATIONS(double)
WFX_DECLARE_SPECIALISATIONS(float)

// ev (optional, 4 * nsteps + 1 events): recorded before each phase of each
// step and after the last, for per-phase durations of a run
template <typename T>
hipError_t launch_fused_steps(wfx_ctx *c, int nsteps, double *hist, hipStream_t s, hipEvent_t *ev);

// The reaction record of a run of nsteps steps into hist (null, or no
// reaction group: nothing is recorded): the node pass of step k fills row(k),
// and where full(k) holds launch_reaction_rows sums the rows filled since
// the last time.
struct ReactRecord {
  const wfx_ctx *c;
  double *hist;
  int nsteps;
  size_t es;  // bytes of a recorded value
  ReactRecord(const wfx_ctx *c_, double *hist_, int nsteps_, size_t es_)
      : c(c_), hist(c_->ngroups > 0 && c_->react_ring ? hist_ : nullptr), nsteps(nsteps_), es(es_) {}
  void *row(int k) const {
    return hist ? static_cast<char *>(c->react_ring) + (size_t)(k % c->react_rows) * c->react_n * es : nullptr;
  }
  bool full(int k) const { return hist && (k + 1 == nsteps || (k + 1) % c->react_rows == 0); }
  int first(int k) const { return k / c->react_rows * c->react_rows; }  // the step of the ring's first row
};
template <typename T> hipError_t launch_reaction_rows(wfx_ctx *c, const ReactRecord &r, int k, hipStream_t s);
extern template hipError_t launch_reaction_rows<double>(wfx_ctx *, const ReactRecord &, int, hipStream_t);
extern template hipError_t launch_reaction_rows<float>(wfx_ctx *, const ReactRecord &, int, hipStream_t);
// row k of the record from nd.fi (per-step path)
hipError_t launch_reaction_gather(wfx_ctx *c, double *row, hipStream_t s);
// the context's ring of recorded rows, allocated once per set of reaction nodes
int ensure_react_ring(wfx_ctx *c);

// Whether a run takes the paired passes.  Thermal expansion does not: its
// flat array divides by the masses the paired element pass is still forming.
// Nor do FP32-mixed hexahedra in more than 256 clusters with thermal coupling or
// the per-step CFL time step.  Above 256, two of the 512-thread work-groups have to
// share a CU: the coupled element pass holds 136 registers a thread, more than
// the 128 that leave room for two; the time step's reduction is repeated by every
// work-group.  us per step in graph replay, paired / separate, 333 and 474
// clusters: coupling 26.4 / 23.3 and 28.2 / 25.2, time step 24.9 / 22.5 and 26.4 /
// 24.0, both with Johnson-Cook's law 36.1 / 27.6 and 38.2 / 29.2; neither 19.3 / 20.5
// and 20.6 / 22.0.  (Tetrahedra, 366 and 504 clusters: coupling 16.3 / 16.4 and 17.6 /
// 17.1, time step 18.0 / 17.3 and 19.3 / 18.0, but launched one by one 17.3 / 18.9,
// 17.7 / 18.0, 19.3 / 18.7 and 19.7 / 22.6.)
constexpr int kPairAlways = 256;
inline bool run_paired(const wfx_ctx *c) {
  if (!c->pair || (c->thermal.on && c->thermal.exp_T != 0.0)) return false;
  return c->precision == 0 || c->n == 4 || c->ms.ncl <= kPairAlways || !(c->thermal.on || c->prm.cfl > 0.0);
}
// Whether a run takes the solo pass for all its steps but the last: a paired one
// (whose tables it reads; every node then has a slot, so that as many slots as
// nodes means no node of two clusters: meshes of up to 256 connected elements, or
// many such) in which nothing outside the nodes and elements moves with the steps.  FP64 only: its unit contracts
// within expressions; in the FP32-mixed unit the contractions the compiler picks
// depend on the kernel around them, and a float rounded otherwise shows in the
// results.
inline bool run_solo(const wfx_ctx *c) {
  return c->precision == 0 && run_paired(c) && c->ms.nslot == c->N && !c->contact.on && !c->thermal.on &&
         !(c->prm.cfl > 0.0);
}
constexpr int kSoloSteps = 512;  // of one launch: a few milliseconds
template <typename T>
hipError_t launch_run_step(wfx_ctx *c, int k, int nsteps, bool pair, bool &have_vol, void *rz, hipStream_t s,
                           hipEvent_t *ev);
extern template hipError_t launch_run_step<double>(wfx_ctx *, int, int, bool, bool &, void *, hipStream_t, hipEvent_t *);
extern template hipError_t launch_run_step<float>(wfx_ctx *, int, int, bool, bool &, void *, hipStream_t, hipEvent_t *);
struct StepRecord {  // one step of the adjoint's record
  double *x, *v, *pa, *fi, *m, *r, *tau, *ep;
};
template <typename T>
hipError_t launch_recorded_step(wfx_ctx *c, int k, bool first, const StepRecord &in, const StepRecord &out,
                                hipStream_t s);
extern template hipError_t launch_recorded_step<double>(wfx_ctx *, int, bool, const StepRecord &, const StepRecord &,
                                                        hipStream_t);

template <typename T> hipError_t launch_vsum0(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_fused_phase(wfx_ctx *c, int phase, int predict, hipStream_t s, int step);
template <typename T> hipError_t launch_cfl_step(wfx_ctx *c, int step, hipStream_t s);
template <typename T> hipError_t launch_thermal(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_thermal_expansion(wfx_ctx *c, hipStream_t s);
extern template hipError_t launch_thermal_expansion<double>(wfx_ctx *, hipStream_t);
extern template hipError_t launch_thermal_expansion<float>(wfx_ctx *, hipStream_t);
extern template hipError_t launch_thermal<double>(wfx_ctx *, hipStream_t);
extern template hipError_t launch_thermal<float>(wfx_ctx *, hipStream_t);
extern template hipError_t launch_cfl_step<double>(wfx_ctx *, int, hipStream_t);
extern template hipError_t launch_cfl_step<float>(wfx_ctx *, int, hipStream_t);
extern template hipError_t launch_fused_steps<double>(wfx_ctx *, int, double *, hipStream_t, hipEvent_t *);
extern template hipError_t launch_fused_steps<float>(wfx_ctx *, int, double *, hipStream_t, hipEvent_t *);
extern template hipError_t launch_vsum0<double>(wfx_ctx *, hipStream_t);
extern template hipError_t launch_vsum0<float>(wfx_ctx *, hipStream_t);
extern template hipError_t launch_fused_phase<double>(wfx_ctx *, int, int, hipStream_t, int);
extern template hipError_t launch_fused_phase<float>(wfx_ctx *, int, int, hipStream_t, int);
template <typename T> hipError_t launch_fused_pack(wfx_ctx *c, hipStream_t s);
template <typename T> hipError_t launch_cfl_begin(wfx_ctx *c, hipStream_t s, bool packed);
extern template hipError_t launch_cfl_begin<double>(wfx_ctx *, hipStream_t, bool);
extern template hipError_t launch_cfl_begin<float>(wfx_ctx *, hipStream_t, bool);
template <typename T> hipError_t launch_fused_unpack(wfx_ctx *c, hipStream_t s);
extern template hipError_t launch_fused_pack<double>(wfx_ctx *, hipStream_t);
extern template hipError_t launch_fused_pack<float>(wfx_ctx *, hipStream_t);
extern template hipError_t launch_fused_unpack<double>(wfx_ctx *, hipStream_t);
extern template hipError_t launch_fused_unpack<float>(wfx_ctx *, hipStream_t);

hipError_t launch_update_prediction(wfx_ctx *c, hipStream_t s);
hipError_t launch_copy(const double *src, double *dst, long n, hipStream_t s);
hipError_t launch_impose(wfx_ctx *c, int dim, bool accel, hipStream_t s);
hipError_t launch_calc_accel(wfx_ctx *c, hipStream_t s);
hipError_t launch_correction_accvel(wfx_ctx *c, hipStream_t s);
hipError_t launch_correction_pos(wfx_ctx *c, hipStream_t s);
hipError_t launch_node_step(wfx_ctx *c, bool predict, hipStream_t s);
hipError_t launch_reaction(wfx_ctx *c, int dim, double *dev_out, hipStream_t s);
hipError_t launch_min_edge(wfx_ctx *c, double *partial, double *dev_out, hipStream_t s);
int min_edge_partial_count(wfx_ctx *c);

// rigid-surface contact, per-step API (wfx_k64.hip)
hipError_t contact_face_areas(wfx_ctx *c, hipStream_t s);
hipError_t contact_elem_length(wfx_ctx *c, hipStream_t s);
hipError_t contact_forces(wfx_ctx *c, hipStream_t s);
hipError_t contact_rigid_update(wfx_ctx *c, double dt, hipStream_t s);

// device buffers a fused run writes (saved and restored around autotuning
// and around the adjoint's recomputation)
std::vector<std::pair<void *, size_t>> fused_state_buffers(wfx_ctx *c);
void adjoint_free(wfx_ctx *c);

// Fills device buffers with a 4-byte word each (8-byte values for a double
// fill) in one launch.
struct FillList {
  static constexpr int kMost = 24;
  int count = 0;
  struct {
    void *p;
    size_t words;          // 4-byte words
    unsigned lo, hi;       // even and odd words
  } buf[kMost];
  void add(void *p, size_t bytes, unsigned word = 0) { add2(p, bytes, word, word); }
  void add2(void *p, size_t bytes, unsigned lo, unsigned hi) {
    if (p && bytes) buf[count++] = {p, bytes / 4, lo, hi};
  }
  void add_value(void *p, size_t n, double v, bool f32) {
    union { double d; float f; unsigned u[2]; } b;
    if (f32) {
      b.f = (float)v;
      add(p, n * 4, b.u[0]);
    } else {
      b.d = v;
      add2(p, n * 8, b.u[0], b.u[1]);
    }
  }
};
hipError_t launch_fill(const FillList &f, hipStream_t s);

// A real field's transfer: host [cnt][rows] double, device [rows][cnt]
// (spin: 3 device rows for host columns 3..5 of 6, the others zero), float
// when f32; perm maps a host item to its device column (null: the same).
// The device must be current and idle; both return when the transfer is over.
struct FieldMove {
  void *dev;
  long cnt;
  int rows, spin, f32;
  const int *perm;    // on the device
  const int *perm_h;  // the same on the host
};
int field_to_host(wfx_ctx *c, const FieldMove &f, double *host);
int field_from_host(wfx_ctx *c, const FieldMove &f, const double *host);
// a context comes and goes: the transfers' pinned memory goes with the last one
void staging_open();
void staging_close();
void frames_free(wfx_ctx *c);
void frames_join(wfx_ctx *c);

}  // namespace wfx
