// Internal declarations of libflurry_hip: the context and the launchers the
// C-ABI layer (fhip_api.hip) drives.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>

#include <map>
#include <string>
#include <vector>

#include "fhip_physics.hpp"
#include "flurry_hip.h"

namespace fhip {

struct Sizes {
  int D, N, P, S, F, Ff, E, nRK, nFaces, nFaceFpts;
  long long nS() const { return (long long)S * E * N; }  // doubles in one [S][E][N] array
  long long nF() const { return (long long)F * E * N; }
};

// Face flux points grouped for coalesced access: every face flux point has
// a left point index (fpt*E+ele), a right one (or -1) and a kind.
struct FaceTables {
  int* ptL = nullptr;   // [nFaceFpts]
  int* ptR = nullptr;   // [nFaceFpts], -1 on boundaries
  int* bc = nullptr;    // [nFaceFpts], -1 interior
};

// Per-kernel timing with HIP events recorded on the context's stream around
// each launch; nothing synchronises until the times are read (or the event
// pool is full), so timing runs inside the timed region itself.
struct Timer {
  std::map<std::string, std::pair<double, long long>> acc;  // total ms, launches
  std::vector<hipEvent_t> pool;
  std::vector<std::pair<const char*, size_t>> pending;       // name, index of start event
  size_t used = 0;
};

// Debug aid: with FHIP_POISON_ALLOC=1 in the environment every device
// allocation of the library is filled with 0xFF bytes (NaN in FP64/FP32, -1 in
// int32), so that a read of memory no kernel has written shows up as NaN.
inline bool poison_alloc() {
  static const bool on = [] {
    const char* v = std::getenv("FHIP_POISON_ALLOC");
    return v && v[0] == '1';
  }();
  return on;
}
inline void poison_fill(void* p, size_t bytes) {
  if (!(poison_alloc() && p && bytes)) return;
  (void)hipMemset(p, 0xFF, bytes);
  (void)hipDeviceSynchronize();
}

// f(l) for the non-zeros a[l] of a dense operator's k entries, ascending, until one
// returns false; false then.  Mostly zeros: eight at a time (the sign bit out of the
// way), since set-up of a small mesh is largely these scans.
template <class F>
inline bool each_nonzero(const double* a, int k, F&& f) {
  for (int l0 = 0; l0 < k; l0 += 8) {
    const int m8 = std::min(8, k - l0);
    unsigned long long v[8] = {}, any = 0;
    std::memcpy(v, a + l0, m8 * sizeof(double));
    for (unsigned long long x : v) any |= x << 1;
    if (!any) continue;
    for (int l = l0; l < l0 + m8; l++)
      if (a[l] != 0.0 && !f(l)) return false;
  }
  return true;
}
inline long long count_nonzeros(const double* a, long long k) {
  long long n = 0;
  for (long long l = 0; l < k; l++) n += a[l] != 0.0;
  return n;
}

// A dense operator kept as its non-zero entries, row by row: q entries (padded
// with zero weights) in each of `groups` partial sums, idx the row of the
// operand.  q == 0: too many non-zeros per row, applied dense.
struct RowOp {
  int m = 0, groups = 1, q = 0;
  int* idx = nullptr;     // [m][groups][q]
  double* w = nullptr;    // [m][groups][q]
};

struct Ctx {
  Sizes z;
  fhip_params prm;
  Phys ph;
  int device = 0;
  hipStream_t stream = nullptr;

  // operators
  double *sf = nullptr, *grad = nullptr, *efn = nullptr, *corr = nullptr, *corru = nullptr, *ws = nullptr,
         *wf = nullptr;
  // the same operators by their non-zeros: extrapolation, gradient of all
  // directions, gradient correction, normal-flux extrapolation and divergence
  // over the stacked directions, divergence correction (staged path)
  RowOp r_sf, r_grad, r_corru, r_efn, r_div, r_corr;
  void* row_mem = nullptr;  // their tables
  // 1-D tensor-product factors for the fused path (see fhip_fused.hip)
  double* tp = nullptr;
  // metrics
  double *jginv = nullptr, *detj = nullptr, *norm = nullptr, *da = nullptr;
  FaceTables ft;
  // face-fpt order used by the staged kernels (natural) and original face ids
  std::vector<int> h_ptL, h_ptR;
  // state and work arrays (FlurryPP layouts)
  double *U = nullptr, *U0 = nullptr, *Uf = nullptr, *Fs = nullptr, *dU = nullptr, *dUf = nullptr,
         *dUc = nullptr, *disFn = nullptr, *Fn = nullptr, *divF = nullptr, *waveSp = nullptr, *eleDt = nullptr,
         *faceFn = nullptr, *src = nullptr, *Uacc = nullptr;
  double* d_dt = nullptr;       // device copy of params->dt
  double* partial = nullptr;    // reduction scratch
  int* flag = nullptr;          // state-check flag
  double h_dt = 0;
  int iter = 0;
  bool timing = false;
  Timer timer;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  // captured RK steps (fused path), by graph_slot: with P-multigrid source,
  // keeping divF_spts[0], FP64, mixed, mixed with BF16 hi+lo, mixed with BF16
  // hi+mid+lo, U at the flux points in the second copy (fused_flipped).  A graph
  // holds the device pointers of the moment it was captured: drop them
  // whenever an array they use is (re)allocated.
  hipGraphExec_t graph[32] = {};
  static int graph_slot(bool src, bool keep, int precision, bool flipped) {
    return ((flipped * 4 + precision) * 2 + keep) * 2 + src;
  }
  // mixed path: BF16 pieces of the matrix-core z contractions (0: none)
  int bf16 = 0;
  unsigned long long graph_gen = 0;  // bumped by drop_graphs: graphs over several contexts check it
  void drop_graphs() {
    graph_gen++;
    bool any = false;
    for (auto& g : graph) any = any || g != nullptr;
    if (any) (void)hipStreamSynchronize(stream);  // no replay still in flight
    for (auto& g : graph) {
      if (g) (void)hipGraphExecDestroy(g);
      g = nullptr;
    }
  }
  bool fused_ok = false;
  bool use_graphs = true;
  bool batched = false;  // several meshes or a boundary-state table
  void* fused = nullptr;  // FusedState (fhip_fused.hip)
};

void timer_resolve(Ctx& c);

// Launch helper: brackets one kernel launch with timing events when enabled.
struct Launch {
  Ctx& c;
  const char* name;
  size_t slot = 0;
  Launch(Ctx& c_, const char* n) : c(c_), name(n) {
    if (!c.timing) return;
    Timer& t = c.timer;
    if (t.used + 2 > 8192) timer_resolve(c);
    while (t.pool.size() < t.used + 2) {
      hipEvent_t e;
      (void)hipEventCreate(&e);
      t.pool.push_back(e);
    }
    slot = t.used;
    t.used += 2;
    (void)hipEventRecord(t.pool[slot], c.stream);
  }
  ~Launch() {
    if (!c.timing) return;
    (void)hipEventRecord(c.timer.pool[slot + 1], c.stream);
    c.timer.pending.push_back({name, slot});
  }
};

// staged path (fhip_staged.hip)
void staged_setup(Ctx& c, const fhip_desc* d);  // the operators' non-zeros
void staged_release(Ctx& c);
void staged_extrapolate_u(Ctx& c);
void staged_wave_speed(Ctx& c);
void staged_residual(Ctx& c, int step);
void staged_time_step_a(Ctx& c, int step, double rk, bool src);
void staged_time_step_b(Ctx& c, int step, bool src);
void copy_array(Ctx& c, double* dst, const double* src, long long n);
void calc_dt(Ctx& c, bool refresh);
// C[m][E*N] = A[m][k] B[k][E*N] (+ C when beta): an operator applied to every
// element and field of a FlurryPP-layout array
void op_apply(Ctx& c, const char* name, int m, int k, const double* A, const double* B, double* C, bool beta);
void sub_array(Ctx& c, double* out, const double* a, const double* b, long long n);  // out = a; out -= b
void add_array(Ctx& c, double* y, const double* x, long long n);                     // y += x
void residual_norm(Ctx& c, int res_type, double* out_host);
// The same without allocating: partial sums in a static device array of
// kNoAllocScratch doubles per GPU (std::length_error beyond it).
constexpr long long kNoAllocScratch = 16384;  // 128 KiB per GPU
constexpr unsigned kResBlocks = 512;  // blocks of the residual norm's grid, at least (bounds its partial sums)
constexpr int kNoAllocMaxDevices = 64;
void residual_norm_noalloc(Ctx& c, int res_type, double* out_host);
double* noalloc_scratch(int device);  // device address of that GPU's scratch array
int check_state(Ctx& c);

// fused path (fhip_fused.hip)
bool fused_setup(Ctx& c, const fhip_desc* d);  // false: configuration not covered
void fused_release(Ctx& c);
// import U, wave speeds [and the P-multigrid source], extrapolate U to the faces
void fused_begin(Ctx& c, bool mixed, bool src = false);
void fused_end(Ctx& c);                // after steps: export U, divF_spts[0], wave speeds and dt
// (keep: write divF_spts[0] at the first stage; steps whose residual nothing
// reads skip it)
// (make_src, where fused_em_source_in_step: the source less this step's first
// residual becomes the source, as fused_em_residual's 1 before the step)
void fused_rk_step(Ctx& c, bool refresh, bool mixed, bool keep = true, bool make_src = false);
bool fused_em_source_in_step(const Ctx& c);
// Inviscid runs: whether U at the flux points lies in the second of its two copies
// (after an odd number of stages since the call's start); a replayed step's flip.
bool fused_flipped(const Ctx& c);
void fused_set_flipped(Ctx& c, bool flipped);
bool fused_step_flips(const Ctx& c);
// P-multigrid cycle on element-major levels: work arrays and the FAS source
// allocated; the start of a cycle; the residual (no source)
// and the wave speeds, the residual written (how) 0: into divF_spts[0],
// 1: subtracted from the source in place, 2: plus the source into
// divF_spts[0]; the source on or off for the RK
// update; U, divF_spts[0] or the source (which 0, 1, 2); a cycle's results
// written back to FlurryPP's layout; the transfers into the coarse level c (U,
// source, sol) and into the upper level up (U += P (U_c - sol_c)), with U at the
// flux points there.
void fused_em_prepare(Ctx& c, bool mixed);
void fused_em_begin(Ctx* const* coarse, int nc, Ctx* const* fine, int nf, bool mixed);
void fused_em_residual(Ctx& c, bool mixed, int how = 0);
void fused_em_set_src(Ctx& c, bool on);
double* fused_em_array(Ctx& c, int which);
void fused_em_end(Ctx* const* coarse, int nc, Ctx* const* fine, int nf, bool stepped);
// (restriction into the coarse elements [e0, e0 + ne) from the fine rows Uf,
// divFf of those elements)
void pmg_restrict_em(Ctx& c, bool mixed, long long e0, long long ne, int Sf, const double* R, const double* Uf,
                     const double* divFf, double* solc);
void pmg_prolong_em(Ctx& up, bool mixed, int Sc, const double* Pm, const double* Uc, const double* solc, bool extrap);
void fused_residual(Ctx& c, bool mixed);  // divF_spts[0] and wave speeds of the current U
// block sizes of the fused kernels (extrapolate, face_inviscid, volume, face_boundary, rk)
void fused_autotune(Ctx& c, bool mixed, int* out);
void fused_set_blocks(Ctx& c, bool mixed, const int* nt);
void fused_get_blocks(Ctx& c, bool mixed, int* out);
void fused_mesh_residuals(Ctx& c, int type, double* out);  // out [nMesh][N]
int fused_n_meshes(Ctx& c);
void fused_set_active(Ctx& c, const int* active);

}  // namespace fhip

struct fhip_ctx {
  fhip::Ctx c;
};
