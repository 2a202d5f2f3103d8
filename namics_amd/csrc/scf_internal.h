// Host-side internals shared by the C ABI (scf_api.hip) and the request
// server (scf_server.hip): the system handle and the helpers that build it.
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/namics_scf.h"
#include "scf_device.h"
#include "scf_kernels.h"
#include "scf_spec.h"

// 2-gradient tiles are faster while a call has no more systems than the
// lattice has 700 + 24000 / N sites (scf_system::mode_among; N segments in
// all its chains): tiles take one system after another, 2.5 us per segment and
// a fixed part for launches and the passes around the chains.  Batches of n
// solves of 3 evaluations, one workgroup each against tiles, ms:
//   100 x 100, N = 8     n = 3   2.5   1.8   n = 5   3.0   3.0
//   100 x 100, N = 20    n = 5   4.3   3.6   n = 7   4.8   5.0
//   128 x 256, N = 20    n = 16 18.7  16.4   n = 24 23.9  24.6
//   97 x 102, N = 100    n = 8  13.8  10.3   n = 12 14.9  15.4
//   128 x 256, N = 100   n = 32 69.8  61.1   n = 45 63.7  68.2
//   128 x 200, N = 400   n = 30 152   118    n = 40 145   144
constexpr int kTileSites = 700, kTileFixed = 24000;

// One SCF system: its parsed input, device description and HBM arena.
struct scf_system {
  nscf::SystemSpec spec;
  nscf::DevSys h;              // host copy holding device pointers
  nscf::DevSys *d = nullptr;   // device copy
  nscf::DevSys **d_list = nullptr;
  char *arena = nullptr;
  size_t arena_bytes = 0;
  hipStream_t stream = nullptr;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  hipGraphExec_t graph_exec = nullptr;    // captured grid-path iteration
  hipGraphExec_t graph_exec32 = nullptr;  // the same with FP32 propagators (mixed precision)
  bool use_graph = true;
  int mode = SCF_MODE_AUTO;
  int tuned_mode = SCF_MODE_AUTO;  // the autotuner's choice for this shape (used under AUTO)
  int nb = 0;            // workgroups of the grid path
  int gf_rows = 0;       // end-point rows (of M sites) the arena holds: chain length x components, or
                         // fewer with the input's save_memory
  int m_alloc = 0;       // DIIS history the arena was sized for
  size_t lds_bytes = 0;  // dynamic LDS the fused path asks for (0: rows in HBM)
  bool have_results = false;
  bool owns_stream = true;  // false when a server lends its stream
  char *region = nullptr;   // arena placed in a caller's device region (not owned)
  std::vector<nscf::BranchPlan> plans;  // row schedules of the branched molecules (h.branch points here)

  bool newton() const { return spec.solver.method != nscf::SOLVER_DIIS; }
  // destroys the captured grid-path iterations (both precisions)
  void drop_graphs() {
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    if (graph_exec32) (void)hipGraphExecDestroy(graph_exec32);
    graph_exec = graph_exec32 = nullptr;
  }
  bool branched() const {
    for (auto &m : spec.mol)
      if (m.scheduled()) return true;
    return false;
  }

  // 2- and 3-gradient systems whose results depend on ghost values the
  // reference computes over its flattened arrays: charged systems (the
  // potential reads densities on ghosts) and surface boundaries (a surface
  // ghost keeps its own value).  They run one workgroup per system with the
  // chains over every site (chain_literal).
  bool has_ring() const {
    for (auto &m : spec.mol)
      if (m.ring) return true;
    return false;
  }
  bool literal() const {
    if (spec.lat.gradients < 2) return false;
    if (spec.charged) return true;
    for (int d = 0; d < 6; d++)
      if (spec.lat.bc[d] == nscf::BC_SURFACE) return true;
    return false;
  }

  int effective_mode() const {
    if (mode != SCF_MODE_AUTO) return mode;
    // branched molecules and dendrimers run their row schedules on the grid path
    if (branched()) return SCF_MODE_GRID;
    // charged systems solve the potential in the one-workgroup kernels
    if (spec.charged || literal() || has_ring()) return SCF_MODE_FUSED;
    // checkpointed end-point storage runs on the strip chains or the grid path
    if (h.ckpt > 1 && h.strip_sx == 0) return SCF_MODE_GRID;
    if (tuned_mode != SCF_MODE_AUTO) return tuned_mode;
    bool markov2 = false;  // second-order chains run on the fused path only
    for (auto &m : spec.mol) markov2 = markov2 || m.markov == 2;
    return spec.lat.gradients == 3 && !markov2 ? SCF_MODE_GRID : SCF_MODE_FUSED;
  }

  // The mode of this system when a call solves or evaluates n systems.  A
  // 2-gradient lattice whose rows do not fit LDS (from about 9800 sites off
  // the strip path) runs its chains as tiles over many workgroups
  // (scf_tile2d.h) while the call is small: one after another, such systems
  // take the time of their launches each, while one launch of a workgroup per
  // system takes 4 ns per site and contour index whatever their number up to
  // one per CU.  Alone, per evaluation: 101 x 128, N = 100: 5.14 -> 0.38
  // ms; 128 x 256, N = 400: 49.5 -> 1.09 ms.  Lattices with their rows in LDS
  // stay with one workgroup each: tiles would be 1.4 to 4 times faster alone,
  // but a served or batched system gives the bits it gives alone, and there
  // one workgroup per system has many times the throughput.
  //
  // Branched molecules on a 1-gradient lattice whose rows fit LDS run their
  // schedule in one workgroup (chain_branched) instead of one launch per row
  // operation, however many systems there are: 60 layers, 20 segments, about
  // 100 operations: 0.27 -> 0.06 ms per evaluation.  Not with checkpoints (a
  // linear molecule's save_memory): there the linear chains of one workgroup
  // store every row, and the arena holds the checkpoints only.
  int mode_among(int n) const {
    const int m = effective_mode();
    if (mode == SCF_MODE_AUTO && m == SCF_MODE_GRID && h.branch_lds && h.ckpt <= 1 &&
        tuned_mode != SCF_MODE_GRID && h.precision == SCF_PREC_FP64)
      return SCF_MODE_FUSED;
    const bool tiles = m == SCF_MODE_FUSED && mode == SCF_MODE_AUTO && tuned_mode == SCF_MODE_AUTO && h.tile2 &&
                       h.strip_sx == 0 && h.wave2 == 0 && !h.use_lds && h.precision == SCF_PREC_FP64;
    if (!tiles) return m;
    long long N = 0;
    for (auto &mol : spec.mol) N += mol.chainlength;
    return n * (kTileSites * N + kTileFixed) <= N * spec.lat.MX * spec.lat.MY ? SCF_MODE_GRID : m;
  }
};

namespace nscf {

int fail(int code, const std::string &msg);
int hip_fail(hipError_t e, const char *where);

#define HIP_TRY(expr)                                 \
  do {                                                \
    hipError_t _e = (expr);                           \
    if (_e != hipSuccess) return hip_fail(_e, #expr); \
  } while (0)

// Where build() places a system's arena: its own allocation (default), a
// caller's device region of `capacity` bytes, or nowhere (dry: compute the
// footprint only, into scf_system::arena_bytes).
struct Placement {
  char *region = nullptr;
  size_t capacity = 0;
  bool dry = false;
};

int validate(const SystemSpec &s, std::string &why);
int build(scf_system *S, const Placement *pl = nullptr);
int upload_solver(scf_system *S);
int read_scalars(const scf_system *S, DevScalars &sc);
int grid_solve(scf_system *S, scf_solve_info *info);
// Newton-Krylov solve of a pseudohessian / hessian input (scf_newton.hip)
int newton_solve(scf_system *S, scf_solve_info *info);
// LBFGS solve of an input with `method : LBFGS` (scf_newton.hip)
int lbfgs_solve(scf_system *S, scf_solve_info *info);
// Broyden rank-reduction solve of an input with `method : BRR` (scf_newton.hip)
int brr_solve(scf_system *S, scf_solve_info *info);
double wall_clock_khz();
size_t lds_limit();
void plan_layout(scf_system *S, int want_sx, int registers);
void plan_tuned(scf_system *S);
std::string shape_key(const scf_system *S);
// End-point rows kept with checkpoint interval K (K <= 1: all N rows): the
// checkpoints 0, K, 2K, ... plus a buffer for the rows of one segment.
int ckpt_rows(int N, int K);
// Checkpoint interval for the input's save_memory (0: every row): about
// sqrt(2 N) rows kept for the longest chain that asks for it, as the
// reference plans them (src/molecule.cpp:174-191), on a uniform grid.
int save_memory_interval(const SystemSpec &s);
// SCF_OK when the system's options (precision, checkpoints) run on the
// given layout, else SCF_E_UNSUPPORTED with the reason.
int check_layout(const scf_system *S, int mode, int strip_sx);
// Job queue: check that `slots` (nslots x chain systems) can share one
// launch, set the carry maps between chain positions, and return the
// workgroup size and dynamic LDS the launch needs.
int prepare_jobs(scf_system *const *slots, int nslots, int chain, int *threads, size_t *lds);
// Device job records -> caller results; t0 = the earliest solve start.
void convert_job_records(const JobRecord *h, size_t n, unsigned long long t0, scf_job_result *results);

}  // namespace nscf
