// libjja: MI355X (gfx950) kernels and device plan for the semi-implicit RCSJ
// time evolution of Josephson junction arrays.
//
// One workgroup integrates one column (problem w) of one circuit for a whole
// chunk of steps: columns never exchange data, so a launch needs no grid-wide
// synchronisation. Per step (stencil 3 shown; time_evolution.py:523-580):
//
//   junctions  x_j = eta - Is + Ic sin(2 th1 - th2) + c1 th1 + c2 th2
//              u_j = x_j / c0_j - ths_j                            (scratch)
//   faces      b_f = sum_j A_fj u_j - 2 pi f_f                      (LDS)
//   solve      J = K^-1 b : staged forward/backward triangular solves (LDS)
//   junctions  y_j = sum_f A_fj J_f ; th_new = (y - x) / c0 ; I = y + Is
//
// The face vector lives in LDS for the whole step. The oldest phase slot of the
// history holds x between the junction passes, then the new phase, so the
// state is stencil_width-1 vectors per column. The junction pass that finishes
// step t also prepares step t+1. Arithmetic of the step expressions follows the
// reference's operation order (no FMA contraction; a division by c0 is a
// product with the reciprocal 1/c0), so results agree with the CPU scheme to
// the rounding of sin, of those quotients and of the linear solve.
//
// This file holds the general kernels, the plan and the C API. Columns that fit stay on
// chip for a whole launch in kernels of their own, chosen at launch for the usual step
// (stencil 3, no voltage sources, noise from Philox at a given amplitude or none):
// jja_resident.hip (small columns), jja_wide.hip (large lattices, one workgroup),
// jja_slab.hip (lattices in row slabs) and jja_domain.hip (other circuits in subdomains).
//
// The solve is a linear program of slices whose addresses do not depend on any
// data: each thread prefetches the entries of the next slice (also across the
// phase barriers, which only order LDS traffic) while it processes the current
// one, so global-memory latency overlaps the LDS gathers and reductions.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/jja.h"
#include "jja_device.h"
#include "jja_domain.h"
#include "jja_resident.h"
#include "jja_wide.h"
#include "jja_slab.h"

// Device scratch of jja_solve_noalloc (a global face store for its columns):
// 2^21 doubles (16 MiB) per GPU, held until the process ends. Calls on one
// GPU share it; calls that overlap on one GPU race.
constexpr int64_t kScratchDoubles = int64_t{1} << 21;
static __device__ __align__(256) double scratch[kScratchDoubles];

namespace {

thread_local std::string g_error;

int fail(int code, const std::string& msg) {
  g_error = msg;
  return code;
}

#define JJA_HIP(expr)                                                              \
  do {                                                                             \
    hipError_t e_ = (expr);                                                        \
    if (e_ != hipSuccess)                                                          \
      return fail(JJA_EHIP, std::string(#expr) + ": " + hipGetErrorString(e_));   \
  } while (0)
// PAIR: a work item is a pair of columns (2q, 2q+1; the last one alone when W is
// odd), its barrier words those of the pair.
template <int BS, int SW, bool PAIR>
__global__ __launch_bounds__(BS) void evolve_split_kernel(const DevProblem* __restrict__ probs,
                                                          const jja_problem_run* __restrict__ runs,
                                                          const WorkItem* __restrict__ work,
                                                          int32_t n_steps, int64_t step0, uint32_t* ctrs,
                                                          int32_t* err, uint32_t wait_limit) {
  extern __shared__ double split_lds[];
  __shared__ int32_t stopped;
  if (threadIdx.x == 0) stopped = 0;
  __syncthreads();
  const WorkItem wi = work[blockIdx.x];
  const DevProblem& P = probs[wi.problem];
  const jja_problem_run& R = runs[wi.problem];
  const int64_t w = wi.column / P.parts;
  const int32_t part = wi.column % P.parts;
  if constexpr (PAIR) {
    const int64_t wa = 2 * w;
    const bool two = wa + 1 < R.W;
    const SplitStore za = split_store(P, gblw(R.zbuf), wa, part, ctrs, wi, err, wait_limit, &stopped, BS,
                                        (LAS double*)split_lds);
    SplitStore zb = za;
    if (two) zb.p = za.p + (static_cast<size_t>(P.Nf) + P.max_stage_rows);
    evolve_steps_pair<BS, SW>(P, R, wa, two, za, zb, n_steps, step0);
  } else {
    const SplitStore zs = split_store(P, gblw(R.zbuf), w, part, ctrs, wi, err, wait_limit, &stopped, BS,
                                        (LAS double*)split_lds);
    evolve_steps<BS, SW>(P, R, w, zs, n_steps, step0);
  }
}

// One workgroup per work item (problem, column). STORE: 0 face stores in LDS,
// 1 in global memory, 2 either, as each problem's index width says (a batch of
// small and large circuits in one launch).
template <int BS, int SW, int STORE>
__global__ __launch_bounds__(BS) void evolve_kernel(const DevProblem* __restrict__ probs,
                                                    const jja_problem_run* __restrict__ runs,
                                                    const WorkItem* __restrict__ work,
                                                    int32_t n_steps, int64_t step0) {
  extern __shared__ double lds[];
  const WorkItem wi = work[blockIdx.x];
  const DevProblem& P = probs[wi.problem];
  const jja_problem_run& R = runs[wi.problem];
  if constexpr (STORE == 2) {
    if (P.index_bytes == 4)
      evolve_column<BS, SW, true>(P, R, wi.column, lds, n_steps, step0);
    else
      evolve_column<BS, SW, false>(P, R, wi.column, lds, n_steps, step0);
  } else {
    evolve_column<BS, SW, STORE == 1>(P, R, wi.column, lds, n_steps, step0);
  }
}

template <int BS, bool GLOBAL>
__global__ __launch_bounds__(BS) void adjoint_kernel(const DevProblem* __restrict__ probs,
                                                     const jja_adjoint_run* __restrict__ runs,
                                                     const WorkItem* __restrict__ work, int64_t k_hi,
                                                     int64_t k_lo) {
  extern __shared__ double lds[];
  const WorkItem wi = work[blockIdx.x];
  const DevProblem& P = probs[wi.problem];
  const jja_adjoint_run& A = runs[wi.problem];
  const int64_t w = wi.column;
  FaceStore<GLOBAL> zs;
  if constexpr (GLOBAL)
    zs.p = gblw(A.zbuf) + static_cast<size_t>(w) * (static_cast<size_t>(P.Nf) + P.max_stage_rows);
  else
    zs.p = lds;
  zs.vt = threadIdx.x;
  zs.vbs = BS;
  if constexpr (!GLOBAL) init_store(P, lds, threadIdx.x, BS);
  adjoint_steps<BS>(P, A, w, zs, k_hi, k_lo);
}

template <int BS, bool PAIR>
__global__ __launch_bounds__(BS) void adjoint_split_kernel(const DevProblem* __restrict__ probs,
                                                           const jja_adjoint_run* __restrict__ runs,
                                                           const WorkItem* __restrict__ work, int64_t k_hi,
                                                           int64_t k_lo, uint32_t* ctrs, int32_t* err,
                                                           uint32_t wait_limit) {
  extern __shared__ double split_lds[];
  __shared__ int32_t stopped;
  if (threadIdx.x == 0) stopped = 0;
  __syncthreads();
  const WorkItem wi = work[blockIdx.x];
  const DevProblem& P = probs[wi.problem];
  const jja_adjoint_run& A = runs[wi.problem];
  const int64_t w = wi.column / P.parts;
  const int32_t part = wi.column % P.parts;
  if constexpr (PAIR) {
    const int64_t wa = 2 * w;
    const bool two = wa + 1 < A.W;
    const SplitStore za = split_store(P, gblw(A.zbuf), wa, part, ctrs, wi, err, wait_limit, &stopped, BS,
                                        (LAS double*)split_lds);
    SplitStore zb = za;
    if (two) zb.p = za.p + (static_cast<size_t>(P.Nf) + P.max_stage_rows);
    adjoint_steps_pair<BS>(P, A, wa, two, za, zb, k_hi, k_lo);
  } else {
    const SplitStore zs = split_store(P, gblw(A.zbuf), w, part, ctrs, wi, err, wait_limit, &stopped, BS,
                                        (LAS double*)split_lds);
    adjoint_steps<BS>(P, A, w, zs, k_hi, k_lo);
  }
}

// After a launch whose parts keep their junctions on chip: once a wait has given up (err),
// what the launch left in a column does not look valid, every value becomes NaN, and the
// host is told through pinned memory, which it reads without waiting (jja_plan_poll). A kernel of
// its own, one workgroup a column: the same in the step kernels cost them 1 to 3% in
// spilled scalar registers (256x256, 16 columns), this one some two microseconds a launch.
constexpr int kSpoilBlock = 256;
__global__ __launch_bounds__(kSpoilBlock) void evolve_spoil_kernel(const jja_problem_run* __restrict__ runs, int32_t Nj,
                                                                   const int32_t* __restrict__ err, int32_t* host_err,
                                                                   int32_t n_steps, int64_t step0) {
  if (!err[0]) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) __hip_atomic_store(host_err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const jja_problem_run& R = runs[0];
  const size_t stride = static_cast<size_t>(R.W) * Nj, col = static_cast<size_t>(blockIdx.x) * Nj;
  const double bad = __builtin_nan("");
  for (int32_t j = threadIdx.x; j < Nj; j += kSpoilBlock) R.theta[col + j] = R.theta[stride + col + j] = bad;
  for (int64_t i = 0; i < n_steps; ++i) {
    const int64_t at = step0 + i - R.slot_t0;
    const int32_t tho = R.th_slot ? R.th_slot[at] : -1, Io = R.I_slot ? R.I_slot[at] : -1;
    for (int32_t j = threadIdx.x; j < Nj; j += kSpoilBlock) {
      if (tho >= 0) R.th_out[tho * stride + col + j] = bad;
      if (Io >= 0) R.I_out[Io * stride + col + j] = bad;
    }
  }
}

__global__ __launch_bounds__(kSpoilBlock) void adjoint_spoil_kernel(const jja_adjoint_run* __restrict__ runs, int32_t Nj,
                                                                    int32_t Nf, const int32_t* __restrict__ err,
                                                                    int32_t* host_err) {
  if (!err[0]) return;
  if (blockIdx.x == 0 && threadIdx.x == 0) __hip_atomic_store(host_err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  const jja_adjoint_run& A = runs[0];
  const size_t stride = static_cast<size_t>(A.W) * Nj, w = blockIdx.x;
  const double bad = __builtin_nan("");
  for (int32_t j = threadIdx.x; j < Nj; j += kSpoilBlock)
    A.grad_Ic[w * Nj + j] = A.grad_Is[w * Nj + j] = A.lam[w * Nj + j] = A.lam[stride + w * Nj + j] = bad;
  for (int32_t f = threadIdx.x; f < Nf; f += kSpoilBlock) A.grad_f[w * Nf + f] = bad;
}

// n[col][f] = -sum_j A[f,j] rint(theta_j / 2pi) (time_evolution.py:734-755): one
// workgroup per phase vector, one thread per face position (a workgroup takes
// the slots of all parts of a split plan in turn).
template <int BS>
__global__ __launch_bounds__(BS) void vortex_kernel(const DevProblem* __restrict__ probs, int32_t p,
                                                    const double* __restrict__ theta,
                                                    int32_t* __restrict__ n_out) {
  const DevProblem& P = probs[p];
  const int64_t col = blockIdx.x;
  const GAS double* __restrict__ th = gbl(theta) + col * P.Nj;
  const int64_t vbs = static_cast<int64_t>(P.parts) * BS;
  for (int32_t part = 0; part < P.parts; ++part) {
    const int32_t vt = part * BS + static_cast<int32_t>(threadIdx.x);
    int64_t acc = 0;
    for (int32_t k = 0; k < P.n_face_slices; ++k) {
      const jja_slice m = load_rec(P.face_slices, k);
      const GAS int32_t* __restrict__ code = gbl(P.face_code) + m.base + vt;
      for (int32_t it = 0; it < m.n_iter; ++it) {
        const int32_t cd = code[it * vbs];
        if (cd < 0) continue;
        const int64_t kk = static_cast<int64_t>(rint(th[cd >> 1] / kTwoPi));
        acc += (cd & 1) ? kk : -kk;
      }
      if (m.flags & JJA_SLICE_FINISH) {
        const int32_t pos = gbl(P.slice_rows)[m.rowbase + vt];
        if (pos >= 0) gblw(n_out)[col * P.Nf + gbl(P.face_of_pos)[pos]] = static_cast<int32_t>(acc);
        acc = 0;
      }
    }
  }
}

// K x = b for `cols` right-hand sides with problem p's solve program: one
// workgroup per column loads b into the face store by solve position (and the
// first stage's scratch, which equals b), runs the staged forward and backward
// solves, and writes x back in face order. b and x are [cols][Nf] with leading
// dimensions ldb and ldx.
template <int BS, bool GLOBAL>
__global__ __launch_bounds__(BS) void spd_solve_kernel(const DevProblem* __restrict__ probs, int32_t p,
                                                       const double* __restrict__ b, int64_t ldb,
                                                       double* __restrict__ x, int64_t ldx, double* zbuf) {
  extern __shared__ double lds[];
  const DevProblem& P = probs[p];
  const int64_t col = blockIdx.x;
  FaceStore<GLOBAL> zs;
  if constexpr (GLOBAL)
    zs.p = gblw(zbuf) + col * (static_cast<int64_t>(P.Nf) + P.max_stage_rows);
  else
    zs.p = lds;
  zs.vt = threadIdx.x;
  zs.vbs = BS;
  const GAS double* __restrict__ bc = gbl(b) + col * ldb;
  GAS double* __restrict__ xc = gblw(x) + col * ldx;
  const GAS int32_t* __restrict__ fop = gbl(P.face_of_pos);
  if constexpr (!GLOBAL) init_store(P, lds, threadIdx.x, BS);
  for (int32_t q = threadIdx.x; q < P.Nf; q += BS) {
    const double v = bc[fop[q]];
    zs.wr(GLOBAL ? q : store_address(P, q), v);
    if (q < P.copy_rows) zs.wr(P.Nf + q, v);
  }
  zs.sync();
  solve_face_system(P, zs);
  zs.sync();
  for (int32_t q = threadIdx.x; q < P.Nf; q += BS) xc[fop[q]] = zs.rd(GLOBAL ? q : store_address(P, q));
}

struct Plan {
  int device = 0;
  std::vector<void*> allocations;
  std::vector<DevProblem> problems;
  std::vector<int64_t> lds_bytes;     // per problem; 0 for a global face store
  std::vector<int64_t> zbuf_doubles;  // per problem; 0 for an LDS face store
  std::vector<int64_t> cost;          // per problem: entries one step of a column reads
  std::vector<int32_t> max_cols;      // per problem: the most columns a run may have
  DevProblem* d_problems = nullptr;
  jja_problem_run* d_runs = nullptr;
  WorkItem* d_work = nullptr;
  size_t work_cap = 0;
  int64_t lds_limit = 0;
  int32_t block_size = 1024;
  int32_t stencil_width = 3;
  jja_adjoint_run* d_adj = nullptr;
  int32_t parts = 1;                 // workgroups per column (block_size is one workgroup's)
  bool pairs = false;                // split launches work two columns per work item
  uint32_t* d_ctrs = nullptr;        // split launches: barrier words per column (counter, XCD set)
  size_t ctr_cap = 0;
  int32_t* d_err = nullptr;          // split launches: [0] a column barrier gave up,
                                     // [1] workgroups whose column ran on one XCD
  int32_t n_cu = 0;                  // compute units of the device
  uint32_t wait_limit = kWaitLimit;  // split launches: polls before a column barrier gives up
  // columns in parts that keep their junctions on chip (one problem; row slabs or
  // subdomains): the device tables and kernels, dynamic LDS doubles, and each
  // part's sequence number of its last step [max_columns][parts], kept on the device
  // so that a launch replayed from a graph counts on
  const void* d_parts = nullptr;
  const void* parts_evolve = nullptr;
  const void* parts_adjoint = nullptr;
  int64_t parts_lds = 0;
  bool parts_only = false;           // subdomains: there is no other way to solve
  uint32_t* d_parts_seq = nullptr;
  // those launches' report to the host: pinned, 1 once a wait has given up
  int32_t* host_err = nullptr;
  // every problem's tables for the kernel that holds a large lattice column in the
  // registers of one workgroup, or NULL; its dynamic LDS bytes
  const WideDev* d_wide = nullptr;
  int64_t wide_lds = 0;
  int64_t split_lds = 0;             // split launches: dynamic LDS bytes (part-local lattice solves)
  // what the device copies of the launch descriptors hold: a launch uploads
  // only what changed since the previous one
  std::vector<jja_problem_run> h_runs;
  std::vector<jja_adjoint_run> h_adj;
  std::vector<WorkItem> h_work;
  bool runs_valid = false, adj_valid = false, work_valid = false;
  // what the launch being prepared reads: the arrays above, or a captured launch's own
  const jja_problem_run* use_runs = nullptr;
  const jja_adjoint_run* use_adj = nullptr;
  const WorkItem* use_work = nullptr;
  // A launch recorded into a graph reads descriptors and work items that never change:
  // a replay must find those of its capture, whatever eager launches did meanwhile.
  // Equal contents are kept once; chunks are freed with the plan.
  struct Kept {
    std::vector<char> host;
    void* dev;
  };
  std::vector<Kept> kept;
  char* kept_chunk = nullptr;
  size_t kept_left = 0, kept_bytes = 0;
  // the stream of the previous launch and an event recorded after it
  hipEvent_t done = nullptr;
  hipStream_t last_stream = nullptr;
  bool launched = false;
  // per kernel: the dynamic LDS limit set on it, and its resident workgroups per CU
  std::vector<std::pair<const void*, int>> lds_attr;
  std::vector<std::pair<const void*, int>> per_cu;
};

// The sine matrix of n modes in DstShape's layout, and T_n's eigenvalues
// 4 sin^2(pi (k + 1) / (2 (n + 1))); angles reduced to a period in integers
std::vector<double> dst_table(int32_t n) {
  const DstShape D(n);
  std::vector<double> t(static_cast<size_t>(D.entries()), 0.0);
  const double pi = 3.14159265358979323846, norm = std::sqrt(2.0 / (n + 1));
  for (size_t e = 0; e < t.size(); ++e) {
    const int64_t l = e % kWave, par = e / kWave % 2, k = e / (2 * kWave) % D.steps, b = e / (2 * kWave) / D.steps;
    const int64_t j = 2 * (16 * b + l % 16) + par, i = 4 * k + l / 16;
    if (i >= D.h || j >= n) continue;
    const int64_t m = (i + 1) * (j + 1) % (2 * (static_cast<int64_t>(n) + 1));
    if (m % (n + 1) == 0) continue;  // the sine of a multiple of pi
    const double v = norm * std::sin(pi * static_cast<double>(m) / (n + 1));
    t[e] = 2 * i + 1 == n ? 0.5 * v : v;
  }
  return t;
}

std::vector<double> dst_eigenvalues(int32_t n) {
  std::vector<double> mu(n);
  for (int32_t k = 0; k < n; ++k) {
    const double s = std::sin(3.14159265358979323846 * (k + 1) / (2.0 * (n + 1)));
    mu[k] = 4.0 * s * s;
  }
  return mu;
}

// The tables of a lattice of at most 16 by 16 faces (TileShape)
std::vector<double> tile_table(int32_t R, int32_t C, double g, double gc) {
  constexpr int32_t T = TileShape::kTable;
  std::vector<double> t(3 * T, 0.0);
  const double pi = 3.14159265358979323846;
  const std::vector<double> mc = dst_eigenvalues(C), mr = dst_eigenvalues(R);
  for (int32_t e = 0; e < T; ++e) {
    const int32_t i = 4 * (e / kWave) + e % kWave / 16, j = e % 16;  // row of a step's operand and of a result register
    for (int32_t side = 0; side < 2; ++side) {
      const int32_t n = side ? R : C, m = (i + 1) * (j + 1) % (2 * (n + 1));
      if (i < n && j < n && m % (n + 1) != 0)
        t[side * T + e] = std::sqrt(2.0 / (n + 1)) * std::sin(pi * static_cast<double>(m) / (n + 1));
    }
    if (i < R && j < C) t[2 * T + e] = 1.0 / (g * mr[i] + gc * mc[j]);
  }
  return t;
}

template <typename T>
int upload(Plan* plan, const T* host, size_t n, const T** out) {
  *out = nullptr;
  if (n == 0) return JJA_OK;
  if (!host) return fail(JJA_EINVAL, "jja_plan_create: missing array");
  void* d = nullptr;
  JJA_HIP(hipMalloc(&d, n * sizeof(T)));
  plan->allocations.push_back(d);
  JJA_HIP(hipMemcpy(d, host, n * sizeof(T), hipMemcpyHostToDevice));
  *out = static_cast<const T*>(d);
  return JJA_OK;
}

// Whether a plan of this problem alone is asked for row slabs.
bool wants_slabs(const jja_problem_desc& d) {
  return d.lattice_slabs && d.lattice_rows && d.lattice_gc > 0.0 && d.n_junctions > 0 && d.parts >= 2 && d.block_size == d.parts * kPartBlock;
}

// The slab form of a split lattice problem, where it asks for it and fits.
int create_slabs(Plan* plan, const jja_problem_desc& d) {
  if (!wants_slabs(d)) return JJA_OK;
  SlabHost h;
  if (!build_slabs(d, plan->parts, kSplitLdsMax, &h)) return JJA_OK;
  const int32_t per = (std::max(h.d.pairs, h.d.faces) + kPartBlock - 1) / kPartBlock;
  const std::vector<double> table = dst_table(d.lattice_cols);
  int rc;
  if ((rc = upload(plan, h.pair.data(), h.pair.size(), &h.d.pair))) return rc;
  if ((rc = upload(plan, h.pair_code.data(), h.pair_code.size(), &h.d.pair_code))) return rc;
  if ((rc = upload(plan, h.face_code.data(), h.face_code.size(), &h.d.face_code))) return rc;
  if ((rc = upload(plan, h.face_id.data(), h.face_id.size(), &h.d.face_id))) return rc;
  if ((rc = upload(plan, h.face_at.data(), h.face_at.size(), &h.d.face_at))) return rc;
  if ((rc = upload(plan, h.face_pos.data(), h.face_pos.size(), &h.d.face_pos))) return rc;
  if ((rc = upload(plan, table.data(), table.size(), &h.d.table))) return rc;
  if ((rc = upload(plan, h.inv.data(), h.inv.size(), &h.d.inv))) return rc;
  if ((rc = upload(plan, h.spike.data(), h.spike.size(), &h.d.spike))) return rc;
  if ((rc = upload(plan, h.reduced.data(), h.reduced.size(), &h.d.reduced))) return rc;
  const std::vector<double> ends(static_cast<size_t>(d.max_columns) * 2 * h.d.ends_rows * d.lattice_cols, 0.0);
  const std::vector<uint32_t> flags(static_cast<size_t>(d.max_columns) * plan->parts * h.d.mode_waves, 0u);
  const double* e = nullptr;
  const uint32_t* f = nullptr;
  if ((rc = upload(plan, ends.data(), ends.size(), &e))) return rc;
  if ((rc = upload(plan, flags.data(), flags.size(), &f))) return rc;
  h.d.ends = const_cast<double*>(e);
  h.d.flags = const_cast<uint32_t*>(f);
  const SlabDev* dev = nullptr;
  if ((rc = upload(plan, &h.d, 1, &dev))) return rc;
  plan->d_parts = dev;
  plan->parts_evolve = slab_evolve_kernel(per);
  plan->parts_adjoint = slab_adjoint_kernel(per);
  plan->parts_lds = 8 * slab_lds_doubles(h.d, d.lattice_cols);
  return JJA_OK;
}

// The tables of jja_wide.hip, where every problem of the plan takes that form: lattices
// whose padded four-product solve does not fit in LDS. Where that fits, the kernel with
// its phases in memory is the faster one (one column a CU, 200 columns with noise: 57x57
// 26.2 us a step against 30.2, 64x64 30.8 against 32.1); where it does not, this one
// (72x72 39.1 against 50.8, 100x100 62.9 against 83.8).
int create_wide(Plan* plan, const jja_problem_desc* descs, int32_t n) {
  if (plan->parts != 1 || plan->stencil_width != 3 || plan->block_size <= kResidentBlock) return JJA_OK;
  std::vector<WideHost> h(n);
  int64_t lds = 0;
  for (int32_t i = 0; i < n; ++i) {
    if (!descs[i].lattice_rows || !(descs[i].lattice_gc > 0.0) || plan->problems[i].lat_ld || plan->problems[i].index_bytes != 2 ||
        !build_wide(descs[i], plan->lds_limit, &h[i]))
      return JJA_OK;
    lds = std::max(lds, 8 * wide_lds_doubles(h[i].d, descs[i].n_junctions));
  }
  std::vector<WideDev> dev(n);
  for (int32_t i = 0; i < n; ++i) {
    WideHost& v = h[i];
    const std::vector<double> table = dst_table(descs[i].lattice_cols);
    int rc;
    if ((rc = upload(plan, v.junc_code.data(), v.junc_code.size(), &v.d.junc_code))) return rc;
    if ((rc = upload(plan, v.face_code.data(), v.face_code.size(), &v.d.face_code))) return rc;
    if ((rc = upload(plan, table.data(), table.size(), &v.d.table))) return rc;
    if ((rc = upload(plan, v.inv.data(), v.inv.size(), &v.d.inv))) return rc;
    if ((rc = upload(plan, v.spike.data(), v.spike.size(), &v.d.spike))) return rc;
    if ((rc = upload(plan, v.reduced.data(), v.reduced.size(), &v.d.reduced))) return rc;
    dev[i] = v.d;
  }
  plan->wide_lds = lds;
  return upload(plan, dev.data(), dev.size(), &plan->d_wide);
}

// The subdomains of a problem that has them (validated).
int create_domains(Plan* plan, const jja_problem_desc& d) {
  if (!d.domains) return JJA_OK;
  const jja_domains& s = *d.domains;
  const size_t G = s.parts, np = G * s.pairs, nf = G * s.faces;
  DomainDev v{};
  v.parts = s.parts;
  v.pairs = s.pairs;
  v.faces = s.faces;
  v.n_gamma = s.n_gamma;
  v.sources = s.sources;
  v.n_published = s.n_published;
  v.val_bytes = static_cast<int32_t>(s.n_entries * static_cast<int64_t>(sizeof(double)));
  std::vector<uint32_t> pc(2 * np), fc(4 * nf), at(nf);
  for (size_t i = 0; i < pc.size(); ++i) pc[i] = s.pair_code[2 * i] | static_cast<uint32_t>(s.pair_code[2 * i + 1]) << 16;
  for (size_t i = 0; i < fc.size(); ++i) fc[i] = s.face_code[2 * i] | static_cast<uint32_t>(s.face_code[2 * i + 1]) << 16;
  for (size_t i = 0; i < nf; ++i) at[i] = s.face_used[i] ? static_cast<uint32_t>(i % s.faces) : 0xffffffffu;
  int rc;
  if ((rc = upload(plan, s.pair, np, &v.pair))) return rc;
  if ((rc = upload(plan, pc.data(), pc.size(), &v.pair_code))) return rc;
  if ((rc = upload(plan, fc.data(), fc.size(), &v.face_code))) return rc;
  if ((rc = upload(plan, at.data(), at.size(), &v.face_at))) return rc;
  if ((rc = upload(plan, s.face_id, nf, &v.face_id))) return rc;
  v.face_pos = v.face_id;  // solve positions are in circuit order
  if ((rc = upload(plan, s.pub_ptr, G + 1, &v.pub_ptr))) return rc;
  if ((rc = upload(plan, s.pub_at, static_cast<size_t>(s.n_published), &v.pub_at))) return rc;
  if ((rc = upload(plan, s.source, static_cast<size_t>(s.n_gamma) * s.sources, &v.source))) return rc;
  if ((rc = upload(plan, s.records, static_cast<size_t>(s.n_records), &v.solve_slices))) return rc;
  if ((rc = upload(plan, s.wave_ptr, 2 * G * (kPartBlock / kWave + 1), &v.wave_ptr))) return rc;
  if ((rc = upload(plan, s.slice_rows, static_cast<size_t>(s.n_slice_rows), &v.slice_rows))) return rc;
  if ((rc = upload(plan, s.ent_val, static_cast<size_t>(s.n_entries), &v.ent_val))) return rc;
  const uint16_t* off = nullptr;
  if ((rc = upload(plan, s.ent_off, static_cast<size_t>(s.n_index), &off))) return rc;
  v.ent_off = off;
  const std::vector<double> pub(static_cast<size_t>(d.max_columns) * 2 * s.n_published, 0.0);
  const std::vector<uint32_t> flags(static_cast<size_t>(d.max_columns) * G * (kPartBlock / kWave), 0u);
  const double* e = nullptr;
  const uint32_t* f = nullptr;
  if ((rc = upload(plan, pub.data(), pub.size(), &e))) return rc;
  if ((rc = upload(plan, flags.data(), flags.size(), &f))) return rc;
  v.pub = const_cast<double*>(e);
  v.flags = const_cast<uint32_t*>(f);
  const DomainDev* dev = nullptr;
  if ((rc = upload(plan, &v, 1, &dev))) return rc;
  const int32_t per = (std::max(v.pairs, v.faces) + kPartBlock - 1) / kPartBlock;
  plan->d_parts = dev;
  plan->parts_evolve = domain_evolve_kernel(per);
  plan->parts_adjoint = domain_adjoint_kernel(per);
  plan->parts_lds = 8 * domain_lds_doubles(v);
  plan->parts_only = true;
  return JJA_OK;
}

void free_plan(Plan* plan) {
  for (void* p : plan->allocations) (void)hipFree(p);
  if (plan->host_err) (void)hipHostFree(plan->host_err);
  if (plan->done) (void)hipEventDestroy(plan->done);
  delete plan;
}

// Launches of a plan share its device descriptors, so they run on one stream
// at a time: a launch on another stream waits for nothing and is refused while
// the previous launch has not finished.
int claim_stream(Plan* plan, hipStream_t stream) {
  if (!plan->launched || stream == plan->last_stream) return JJA_OK;
  const hipError_t e = hipEventQuery(plan->done);
  if (e == hipErrorNotReady)
    return fail(JJA_EBUSY, "the plan's previous launch, on another stream, has not finished");
  if (e != hipSuccess) return fail(JJA_EHIP, std::string("hipEventQuery: ") + hipGetErrorString(e));
  return JJA_OK;
}

// Whether `stream` is being captured into a graph.
int capture_state(hipStream_t stream, bool* capturing) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  JJA_HIP(hipStreamIsCapturing(stream, &status));
  *capturing = status != hipStreamCaptureStatusNone;
  return JJA_OK;
}

// Split launches that meet at column barriers are not captured: their barrier words are
// cleared by a memset, and they need the cooperative launch.
int refuse_capture(const char* who) {
  return fail(JJA_EUNSUPPORTED, std::string(who) + ": a launch with column barriers cannot be captured into a graph");
}

int mark_launched(Plan* plan, hipStream_t stream) {
  JJA_HIP(hipEventRecord(plan->done, stream));
  plan->last_stream = stream;
  plan->launched = true;
  return JJA_OK;
}

// Copies n host descriptors to the plan's device array when they differ from
// what it holds (pageable source: staged before the call returns, ordered after
// earlier work on the stream).
template <typename T>
int upload_if_changed(T* dev, const T* host, size_t n, std::vector<T>& shadow, bool& valid, hipStream_t stream) {
  if (valid && shadow.size() == n && std::memcmp(shadow.data(), host, n * sizeof(T)) == 0) return JJA_OK;
  JJA_HIP(hipMemcpyAsync(dev, host, n * sizeof(T), hipMemcpyHostToDevice, stream));
  shadow.assign(host, host + n);
  valid = true;
  return JJA_OK;
}

// This thread may allocate and copy beside a stream that is being captured.
struct BesideCapture {
  hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
  BesideCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
  ~BesideCapture() { (void)hipThreadExchangeStreamCaptureMode(&mode); }
};

// A device copy of `bytes` of host data that stays as it is until the plan is destroyed,
// made outside the graph being captured.
constexpr size_t kKeptChunk = size_t{1} << 16, kKeptLimit = size_t{1} << 26;
int keep_copy(Plan* plan, const void* host, size_t bytes, const void** out) {
  for (const Plan::Kept& k : plan->kept)
    if (k.host.size() == bytes && std::memcmp(k.host.data(), host, bytes) == 0) {
      *out = k.dev;
      return JJA_OK;
    }
  const size_t room = (bytes + 255) & ~size_t{255};
  if (plan->kept_bytes + room > kKeptLimit)
    return fail(JJA_ENOMEM, "the plan's captured launches hold " + std::to_string(plan->kept_bytes) +
                                " bytes of descriptors; destroy the plan to free them");
  const BesideCapture beside;
  if (room > plan->kept_left) {
    const size_t chunk = std::max(room, kKeptChunk);
    void* d = nullptr;
    if (hipMalloc(&d, chunk) != hipSuccess) return fail(JJA_ENOMEM, "captured launch: device allocation failed");
    plan->allocations.push_back(d);
    plan->kept_chunk = static_cast<char*>(d);
    plan->kept_left = chunk;
  }
  void* const d = plan->kept_chunk;
  hipStream_t side = nullptr;
  JJA_HIP(hipStreamCreateWithFlags(&side, hipStreamNonBlocking));
  hipError_t e = hipMemcpyAsync(d, host, bytes, hipMemcpyHostToDevice, side);
  if (e == hipSuccess) e = hipStreamSynchronize(side);
  (void)hipStreamDestroy(side);
  if (e != hipSuccess) return fail(JJA_EHIP, std::string("captured launch: copy of its descriptors: ") + hipGetErrorString(e));
  try {
    const char* first = static_cast<const char*>(host);
    plan->kept.push_back({std::vector<char>(first, first + bytes), d});
  } catch (const std::bad_alloc&) {
    return fail(JJA_ENOMEM, "captured launch: out of host memory");
  }
  plan->kept_chunk += room;
  plan->kept_left -= room;
  plan->kept_bytes += room;
  *out = d;
  return JJA_OK;
}

// The device array a launch reads n descriptors from: the plan's, brought up to date, or
// a copy of the launch's own when it is captured.
template <typename T>
int stage(Plan* plan, T* dev, const T* host, size_t n, std::vector<T>& shadow, bool& valid, hipStream_t stream,
          bool capturing, const T** use) {
  if (capturing) return keep_copy(plan, host, n * sizeof(T), reinterpret_cast<const void**>(use));
  *use = dev;
  return upload_if_changed(dev, host, n, shadow, valid, stream);
}

// Raise a kernel's dynamic LDS limit to at least lds bytes. The limit belongs
// to the kernel on a device, not to a plan, so the largest value any plan has
// asked for is kept process-wide and never lowered (a plan that set a smaller
// one would otherwise break a later launch of another plan).
int raise_lds_attr(const void* kern, int lds) {
  static std::mutex mu;
  static std::vector<std::pair<std::pair<int, const void*>, int>> limits;
  int dev = 0;
  JJA_HIP(hipGetDevice(&dev));
  std::lock_guard<std::mutex> lock(mu);
  for (auto& a : limits)
    if (a.first.first == dev && a.first.second == kern) {
      if (a.second >= lds) return JJA_OK;
      JJA_HIP(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
      a.second = lds;
      return JJA_OK;
    }
  JJA_HIP(hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
  limits.push_back({{dev, kern}, lds});
  return JJA_OK;
}

// The dynamic LDS limit of a kernel with a dynamic LDS face store.
int set_lds_limit(Plan* plan, const void* kern, int lds) {
  for (auto& a : plan->lds_attr)
    if (a.first == kern) {
      if (a.second >= lds) return JJA_OK;
      if (int rc = raise_lds_attr(kern, lds)) return rc;
      a.second = lds;
      return JJA_OK;
    }
  hipFuncAttributes attr;
  JJA_HIP(hipFuncGetAttributes(&attr, kern));
  // the solve reads LDS at the plan's absolute byte offsets: the dynamic LDS
  // array must start at address 0, i.e. the kernel must have no static LDS
  if (attr.sharedSizeBytes != 0) return fail(JJA_EUNSUPPORTED, "kernel with a dynamic LDS face store has static LDS");
  if (int rc = raise_lds_attr(kern, lds)) return rc;
  plan->lds_attr.push_back({kern, lds});
  return JJA_OK;
}

bool pow2_le(int32_t g, int32_t limit) { return g >= 1 && g <= limit && (g & (g - 1)) == 0; }

int32_t parts_of(const jja_problem_desc& d) { return d.parts > 0 ? d.parts : 1; }

// The problems of one plan share the stencil width and the workgroup size
// (block_size / parts); the part count may differ between problems, but if any
// column is split, every problem keeps its face store in global memory (one
// launch runs them all).
int check_plan_shapes(int32_t n, const jja_problem_desc* descs) {
  bool split = false;
  for (int32_t p = 0; p < n; ++p) split = split || parts_of(descs[p]) > 1;
  for (int32_t p = 0; p < n; ++p) {
    const jja_problem_desc& d = descs[p];
    if (d.stencil_width != descs[0].stencil_width)
      return fail(JJA_EINVAL, "jja_plan_create: all problems of a plan need the same stencil width");
    if (parts_of(d) <= 0 || d.block_size % parts_of(d) ||
        d.block_size / parts_of(d) != descs[0].block_size / parts_of(descs[0]))
      return fail(JJA_EINVAL, "jja_plan_create: all problems of a plan need the same block_size/parts");
    if (split && d.index_bytes != 4)
      return fail(JJA_EINVAL, "jja_plan_create: with a split column, every problem needs the global face store");
    // subdomains are built for a plan's only problem, and nothing else solves there
    if (d.domains && (n != 1 || d.lattice_rows != 0 || d.n_faces <= 0 || d.n_junctions <= 0))
      return fail(JJA_EINVAL, "jja_plan_create: domains need a plan of one problem with junctions and faces, "
                              "without a lattice solve");
    if ((d.column_pairs != 0) != (descs[0].column_pairs != 0))
      return fail(JJA_EINVAL, "jja_plan_create: column_pairs must be the same for every problem of a plan");
  }
  return JJA_OK;
}

// Every index of a problem's subdomains.
int validate_domains(const jja_problem_desc& d) {
  const jja_domains& s = *d.domains;
  auto bad = [](const char* what) { return fail(JJA_EINVAL, std::string("jja_plan_create: subdomains: ") + what); };
  const int32_t G = s.parts, waves = kPartBlock / kWave;
  if (G < 2 || G != parts_of(d) || d.block_size != G * kPartBlock || d.index_bytes != 4 || d.column_pairs ||
      d.n_solve_slices || d.face_copy_rows || d.stencil_width != 3)
    return bad("layout of the problem");
  if (s.pairs < 1 || s.faces < 1 || s.n_gamma < 1 || s.sources < 1 || s.n_published < 1 || s.n_records < 1 ||
      s.pairs > kDomainPairs * kPartBlock || s.faces > kDomainPairs * kPartBlock)
    return bad("sizes");
  const int64_t addresses = 2 * static_cast<int64_t>(s.faces) + s.n_gamma;
  if (8 * (addresses + 2 * static_cast<int64_t>(s.pairs) + 1) > kSplitLdsMax) return bad("LDS");
  if (!s.pair || !s.pair_code || !s.face_code || !s.face_id || !s.face_used || !s.pub_ptr || !s.pub_at || !s.source ||
      !s.records || !s.wave_ptr || !s.slice_rows || !s.ent_val || !s.ent_off)
    return bad("missing array");
  for (int32_t q = 0; q < d.n_faces; ++q)
    if (d.face_of_pos[q] != q) return bad("solve positions must be in circuit order");
  for (int64_t i = 0; i < static_cast<int64_t>(G) * s.pairs; ++i) {
    const int32_t e = s.pair[i];
    if (e == -1) continue;
    const int32_t q = e >> 4, m = e & 3;
    if (e < 0 || m == 0 || 2 * q >= d.n_junctions || ((m & 2) && 2 * q + 1 >= d.n_junctions)) return bad("pair");
    for (int32_t c = 0; c < 4; ++c)
      if (s.pair_code[4 * i + c] != 0xffff && (s.pair_code[4 * i + c] >> 1) >= s.faces) return bad("pair code");
  }
  for (int64_t i = 0; i < static_cast<int64_t>(G) * s.faces; ++i) {
    if (s.face_id[i] < -1 || s.face_id[i] >= d.n_faces || (s.face_id[i] >= 0 && !s.face_used[i])) return bad("face");
    for (int32_t c = 0; c < 8; ++c)
      if (s.face_code[8 * i + c] != 0xffff && (s.face_code[8 * i + c] >> 1) >= 2 * s.pairs) return bad("face code");
  }
  if (s.pub_ptr[0] != 0 || s.pub_ptr[G] != s.n_published) return bad("published ranges");
  for (int32_t p = 0; p < G; ++p)
    if (s.pub_ptr[p + 1] < s.pub_ptr[p]) return bad("published ranges");
  for (int32_t i = 0; i < s.n_published; ++i)
    if (s.pub_at[i] < 0 || s.pub_at[i] >= s.faces) return bad("published face");
  for (int64_t i = 0; i < static_cast<int64_t>(s.n_gamma) * s.sources; ++i)
    if (s.source[i] < -1 || s.source[i] >= s.n_published) return bad("source");
  if (s.n_entries < kMaxIter * kWave || s.n_entries * 8 >= (int64_t{1} << 31) || s.n_index < kMaxIter * kWave)
    return bad("record arrays");
  for (int32_t pr = 0; pr < 2 * G; ++pr) {
    const int32_t* wp = s.wave_ptr + static_cast<int64_t>(pr) * (waves + 1);
    int32_t barriers = -1;
    for (int32_t w = 0; w < waves; ++w) {
      if (wp[w] < 0 || wp[w + 1] > s.n_records || wp[w + 1] - wp[w] < 4 || (wp[w + 1] - wp[w] - 4) % 3)
        return bad("wave program");
      int32_t nb = 0;
      for (int32_t k = wp[w]; k < wp[w + 1]; ++k) {
        const jja_slice& m = s.records[k];
        const int32_t g = m.flags & 0xff, rows = m.flags >> 16;
        if (!pow2_le(g, kWave) || m.n_iter < 0 || m.n_iter > kMaxIter || rows < 0 || rows > kWave / g || m.r0 != 0 ||
            (m.flags & (0xe000 | JJA_SLICE_NARROW | JJA_SLICE_WG_BARRIER)))
          return bad("record fields");
        if (m.base < 0 || (m.base % 2) || m.base + kMaxIter * kWave > s.n_entries || m.ibase < 0 || (m.ibase % 8) ||
            m.ibase + kMaxIter * kWave > s.n_index || m.rowbase < 0 || m.rowbase + kWave / g > s.n_slice_rows)
          return bad("record data");
        if (k >= wp[w + 1] - 4) continue;  // loaded ahead, never executed
        nb += (m.flags & JJA_SLICE_BARRIER) != 0;
        for (int32_t i = 0; i < rows; ++i)
          if (s.slice_rows[m.rowbase + i] < -1 || s.slice_rows[m.rowbase + i] >= addresses) return bad("record row");
        for (int64_t e = m.ibase; e < m.ibase + kMaxIter * kWave; ++e)
          if (s.ent_off[e] >= addresses) return bad("record index");
      }
      if (barriers < 0) barriers = nb;
      if (nb != barriers) return bad("wave programs disagree on their barriers");
    }
  }
  return JJA_OK;
}

// Every index the kernels follow is checked here, once, on the host.
int validate(const jja_problem_desc& d) {
  const int32_t Nj = d.n_junctions, Nf = d.n_faces, BS = d.block_size, ms = d.max_stage_rows;
  if (Nj < 0 || Nf < 0 || (Nj == 0 && Nf == 0) || d.stencil_width < 3 || d.stencil_width > 5 || d.n_face_slices < 0 ||
      d.n_solve_slices < 0 || ms < 0)
    return fail(JJA_EINVAL, "jja_plan_create: bad sizes");
  const int32_t parts = d.parts > 0 ? d.parts : 1;
  if (!pow2_le(parts, 32)) return fail(JJA_EINVAL, "jja_plan_create: parts must be a power of two <= 32");
  const int32_t wg = BS / parts;
  if (BS % parts || (wg != 64 && wg != 128 && wg != 256 && wg != 512 && wg != 1024))
    return fail(JJA_EINVAL, "jja_plan_create: block_size/parts must be 64, 128, 256, 512 or 1024");
  if (parts > 1 && d.index_bytes != 4)
    return fail(JJA_EINVAL, "jja_plan_create: a column split over workgroups needs the global face store");
  if (d.column_pairs != 0 && (d.column_pairs != 1 || parts < 2 || wg > 512))
    return fail(JJA_EINVAL, "jja_plan_create: column_pairs needs split columns (parts >= 2) and workgroups "
                            "of at most 512 threads");
  if (d.max_columns < 1 || d.max_columns > (1 << 20))
    return fail(JJA_EINVAL, "jja_plan_create: max_columns must be 1 .. 2^20");
  if (d.cpr_terms < 0 || d.cpr_terms > JJA_CPR_MAX_TERMS)
    return fail(JJA_EINVAL, "jja_plan_create: cpr_terms must be 0 .. " + std::to_string(JJA_CPR_MAX_TERMS));
  if (Nj > 0 && (!d.Ic || !d.Rv || !d.coef || !d.junc_code))
    return fail(JJA_EINVAL, "jja_plan_create: missing junction arrays");
  for (int64_t e = 0; e < 2 * static_cast<int64_t>(Nj); ++e)
    if (d.junc_code[e] < -1 || (d.junc_code[e] >> 1) >= Nf)
      return fail(JJA_EINVAL, "junc_code out of range");
  if (Nf == 0)
    return (d.n_face_slices || d.n_solve_slices || d.lattice_rows) ? fail(JJA_EINVAL, "slices without faces")
                                                                   : JJA_OK;
  if (!d.face_of_pos || !d.face_code || !d.face_slices || !d.slice_rows ||
      (d.n_solve_slices && (!d.solve_slices || !d.ent_val || !d.ent_off)))
    return fail(JJA_EINVAL, "jja_plan_create: missing face or solve arrays");
  if (d.index_bytes != 2 && d.index_bytes != 4) return fail(JJA_EINVAL, "index_bytes must be 2 or 4");
  if (d.index_bytes == 2 && static_cast<int64_t>(Nf) + ms > 65536)
    return fail(JJA_EINVAL, "face vector exceeds 16-bit indices");
  if (static_cast<int64_t>(Nf) + ms > INT32_MAX) return fail(JJA_EINVAL, "face vector too large");
  std::vector<char> seen(Nf, 0);
  for (int32_t q = 0; q < Nf; ++q) {
    const int32_t f = d.face_of_pos[q];
    if (f < 0 || f >= Nf || seen[f]) return fail(JJA_EINVAL, "face_of_pos is not a permutation");
    seen[f] = 1;
  }
  auto check_slice = [&](const jja_slice& m, int64_t n_ent, bool paired) -> int {
    const int32_t G = m.flags & 0xff;
    if (!pow2_le(G, std::min(64, BS))) return fail(JJA_EINVAL, "slice lanes per row must be a power of two <= 64");
    if (m.n_iter < 0 || m.n_iter > kMaxIter) return fail(JJA_EINVAL, "slice n_iter must be 0..8");
    // face records: n_iter*BS codes; solve records: ceil(n_iter/2) pairs of BS doubles
    const int64_t extent = paired ? 2 * static_cast<int64_t>((m.n_iter + 1) / 2) * BS
                                  : static_cast<int64_t>(m.n_iter) * BS;
    if (m.base < 0 || m.base + extent > n_ent) return fail(JJA_EINVAL, "slice entries out of range");
    if (m.rowbase < 0 || m.rowbase + BS / G > d.n_slice_rows) return fail(JJA_EINVAL, "slice rows out of range");
    if ((m.flags >> 16) < 0 || (m.flags >> 16) > BS / G) return fail(JJA_EINVAL, "slice row count out of range");
    if (m.flags & 0xf800) return fail(JJA_EINVAL, "unknown slice flags");
    return JJA_OK;
  };
  for (int32_t k = 0; k < d.n_face_slices; ++k) {
    const jja_slice& m = d.face_slices[k];
    if (int rc = check_slice(m, d.n_face_entries, false)) return rc;
    if ((m.flags & 0xff) != 1) return fail(JJA_EINVAL, "face slices use one lane per row");
    if (m.n_iter > kFaceIter) return fail(JJA_EINVAL, "face slices hold at most 4 codes per thread");
    for (int32_t i = 0; i < BS; ++i) {
      const int32_t r = d.slice_rows[m.rowbase + i];
      if (r < -1 || r >= Nf) return fail(JJA_EINVAL, "face slice row out of range");
    }
    for (int64_t e = m.base; e < m.base + static_cast<int64_t>(m.n_iter) * BS; ++e)
      if (d.face_code[e] < -1 || (d.face_code[e] >> 1) >= Nj) return fail(JJA_EINVAL, "face_code out of range");
  }
  if (d.lattice_rows != 0) {
    const int64_t R = d.lattice_rows, C = d.lattice_cols, H = (C + 1) / 2, ES = H + (H & 1);
    if (R < 2 || C < 2 || R * C != Nf) return fail(JJA_EINVAL, "lattice rows * columns must equal n_faces (>= 2 each)");
    if (d.column_pairs) return fail(JJA_EINVAL, "a lattice solve does not pair columns");
    if (!d.lattice_sine || !d.lattice_inv) return fail(JJA_EINVAL, "jja_plan_create: missing lattice tables");
    if (d.n_solve_slices != 0 || d.face_copy_rows != 0)
      return fail(JJA_EINVAL, "a lattice solve has no solve records and no face copy rows");
    const int64_t B = std::max<int64_t>(1, std::min<int64_t>(R, int64_t{JJA_LATTICE_TRI_THREADS} * parts / C));
    const int64_t EF = d.index_bytes == 4 ? (ES + 3) & ~int64_t{3} : ES;
    if (ms < (Nf & 1) + std::max(2 * R * EF, 4 * B * C))
      return fail(JJA_EINVAL, "max_stage_rows too small for the lattice solve");
    if (!(d.lattice_g > 0.0) || !std::isfinite(d.lattice_g)) return fail(JJA_EINVAL, "lattice_g must be finite and > 0");
    if (!(d.lattice_gc >= 0.0) || !std::isfinite(d.lattice_gc))
      return fail(JJA_EINVAL, "lattice_gc must be finite and > 0, or 0 where it is not given");
    return JJA_OK;
  }
  if (d.domains) return validate_domains(d);
  // solve programs: one per wave of 64 lanes; each runs a multiple of three
  // records and loads four more ahead, all of which must be in range
  const int32_t NW = BS / kWave;
  const int32_t* wp = d.solve_wave_ptr;
  if (!wp || wp[0] != 0 || wp[NW] != d.n_solve_slices)
    return fail(JJA_EINVAL, "solve_wave_ptr must cover the solve records");
  if (d.n_entries < kMaxIter * kWave || d.n_index < kMaxIter * kWave)
    return fail(JJA_EINVAL, "solve arrays too short");
  if (d.n_entries * static_cast<int64_t>(sizeof(double)) >= (int64_t{1} << 31))
    return fail(JJA_EUNSUPPORTED, "solve values of one problem exceed 2 GiB");
  if (d.face_copy_rows < 0 || d.face_copy_rows > Nf || d.face_copy_rows > ms)
    return fail(JJA_EINVAL, "face_copy_rows out of range");
  const int64_t lds_end = static_cast<int64_t>(Nf) + ms;
  int32_t barriers = -1;
  std::string seq0;  // column ('c') and workgroup ('w') barriers of wave 0, in order
  for (int32_t w = 0; w < NW; ++w) {
    if (wp[w + 1] - wp[w] < 4 || (wp[w + 1] - wp[w] - 4) % 3)
      return fail(JJA_EINVAL, "a wave program needs a record count divisible by 3 and 4 lookahead records");
    int32_t nb = 0;
    std::string seq;
    for (int32_t k = wp[w]; k < wp[w + 1]; ++k) {
      const jja_slice& m = d.solve_slices[k];
      const int32_t G = m.flags & 0xff, rows = m.flags >> 16;
      if (!pow2_le(G, kWave)) return fail(JJA_EINVAL, "solve record lanes per row must be a power of two <= 64");
      if (m.n_iter < 0 || m.n_iter > kMaxIter || rows < 0 || rows > kWave / G || (m.flags & 0xe000))
        return fail(JJA_EINVAL, "solve record fields out of range");
      if ((m.flags & JJA_SLICE_NARROW) && (d.index_bytes != 4 || (m.flags & JJA_SLICE_BLOCK)))
        return fail(JJA_EINVAL, "NARROW solve records need 4-byte indices and an off-block phase");
      if (m.base < 0 || (m.base % 2) || m.base + kMaxIter * kWave > d.n_entries || m.ibase < 0 ||
          (m.ibase % (16 / d.index_bytes)) || m.ibase + kMaxIter * kWave > d.n_index || m.rowbase < 0 ||
          m.rowbase + kWave / G > d.n_slice_rows)
        return fail(JJA_EINVAL, "solve record data out of range or misaligned");
      if (k >= wp[w + 1] - 4) continue;  // lookahead only: loaded, never executed
      if (m.flags & JJA_SLICE_BARRIER) {
        ++nb;
        seq.push_back('c');
      } else if (m.flags & JJA_SLICE_WG_BARRIER) {
        seq.push_back('w');
      }
      const bool block = m.flags & JJA_SLICE_BLOCK;
      for (int32_t i = 0; i < rows; ++i) {
        const int32_t r = d.slice_rows[m.rowbase + i];
        if (r == -1) continue;
        if (r < 0 || r >= Nf || (!block && (r - m.r0 < 0 || r - m.r0 >= ms)))
          return fail(JJA_EINVAL, "solve slice row out of range");
      }
      if (m.flags & JJA_SLICE_NARROW) {
        // lane base, then two 16-bit offsets per word
        const uint32_t* ip = static_cast<const uint32_t*>(d.ent_off) + m.ibase;
        for (int32_t l = 0; l < kWave; ++l) {
          uint32_t dmax = 0;
          for (int32_t q = 0; q < kMaxIter / 2; ++q) {
            const uint32_t wd = ip[kWave + 4 * l + q];
            dmax = std::max(dmax, std::max(wd & 0xffffu, wd >> 16));
          }
          if (static_cast<int64_t>(ip[l]) + dmax >= lds_end) return fail(JJA_EINVAL, "solve LDS offset out of range");
        }
      } else if (block && d.index_bytes == 4) {
        // one word per lane: base | len << 28; entries base + i*G, i < len
        for (int32_t l = 0; l < kWave; ++l) {
          const uint32_t wd = static_cast<const uint32_t*>(d.ent_off)[m.ibase + l];
          const int64_t len = wd >> 28, base = wd & 0x0FFFFFFFu;
          if (len > kMaxIter || (len > 0 && base + (len - 1) * G >= lds_end))
            return fail(JJA_EINVAL, "solve LDS offset out of range");
        }
      } else {
        for (int64_t e = m.ibase; e < m.ibase + kMaxIter * kWave; ++e) {
          const int64_t ix = d.index_bytes == 2 ? static_cast<const uint16_t*>(d.ent_off)[e]
                                                : static_cast<const uint32_t*>(d.ent_off)[e];
          if (ix >= lds_end) return fail(JJA_EINVAL, "solve LDS offset out of range");
        }
      }
    }
    if (barriers < 0) barriers = nb;
    if (nb != barriers) return fail(JJA_EINVAL, "wave programs disagree on their barrier count");
    // every wave meets the same barriers in the same order (a workgroup
    // barrier is a __syncthreads of its workgroup, and so is part of a column one)
    if (w == 0)
      seq0 = seq;
    else if (seq != seq0)
      return fail(JJA_EINVAL, "wave programs disagree on their barrier sequence");
  }
  return JJA_OK;
}

template <int BS, int SW, int STORE>
int launch_evolve(Plan* plan, const WorkItem* work, int32_t n_work, int64_t lds, int32_t n_steps,
                  int64_t step0, hipStream_t stream) {
  auto* kern = evolve_kernel<BS, SW, STORE>;
  if (int rc = set_lds_limit(plan, reinterpret_cast<const void*>(kern), static_cast<int>(lds))) return rc;
  hipLaunchKernelGGL(kern, dim3(n_work), dim3(BS), static_cast<size_t>(lds), stream,
                     plan->d_problems, plan->use_runs, work, n_steps, step0);
  JJA_HIP(hipGetLastError());
  return JJA_OK;
}

template <int BS, bool GLOBAL>
int launch_adjoint(Plan* plan, const WorkItem* work, int32_t n_work, int64_t lds, int64_t k_hi,
                   int64_t k_lo, hipStream_t stream) {
  auto* kern = adjoint_kernel<BS, GLOBAL>;
  if (int rc = set_lds_limit(plan, reinterpret_cast<const void*>(kern), static_cast<int>(lds))) return rc;
  hipLaunchKernelGGL(kern, dim3(n_work), dim3(BS), static_cast<size_t>(lds), stream,
                     plan->d_problems, plan->use_adj, work, k_hi, k_lo);
  JJA_HIP(hipGetLastError());
  return JJA_OK;
}

template <int BS>
int launch_vortex(Plan* plan, int32_t p, const double* theta, int32_t cols, int32_t* n_out,
                  hipStream_t stream) {
  hipLaunchKernelGGL(vortex_kernel<BS>, dim3(cols), dim3(BS), 0, stream, plan->d_problems, p, theta,
                     n_out);
  JJA_HIP(hipGetLastError());
  return JJA_OK;
}

// Copies the work items of one launch to the plan's array (sized at plan
// creation) when they differ from what it holds, or to a captured launch's own.
int upload_work(Plan* plan, const std::vector<WorkItem>& work, hipStream_t stream, bool capturing) {
  if (work.size() > plan->work_cap) return fail(JJA_EINVAL, "launch has more work items than the plan was sized for");
  return stage(plan, plan->d_work, work.data(), work.size(), plan->h_work, plan->work_valid, stream, capturing,
               &plan->use_work);
}

template <int BS, int STORE>
int launch_evolve_sw(Plan* plan, const WorkItem* work, int32_t n, int64_t lds, int32_t n_steps,
                     int64_t step0, hipStream_t stream) {
  switch (plan->stencil_width) {
    case 3: return launch_evolve<BS, 3, STORE>(plan, work, n, lds, n_steps, step0, stream);
    case 4: return launch_evolve<BS, 4, STORE>(plan, work, n, lds, n_steps, step0, stream);
    default: return launch_evolve<BS, 5, STORE>(plan, work, n, lds, n_steps, step0, stream);
  }
}

// How a launch can keep every column's state on chip (jja_resident.hip): the
// junction pairs each thread keeps in registers, 0 for the state in LDS, or -1 when
// some problem needs the general kernels. *lds receives the dynamic LDS bytes of
// the widest column.
int resident_layout(const Plan* plan, int64_t* lds) {
  if (plan->stencil_width != 3 || plan->block_size > kResidentBlock) return -1;
  const int32_t BS = plan->block_size;
  int32_t form = 1;
  for (const DevProblem& d : plan->problems) {
    if (d.index_bytes != 2) return -1;
    const int32_t need = std::max(((d.Nj + 1) / 2 + BS - 1) / BS, (d.n_face_slices + kResidentFaces - 1) / kResidentFaces);
    if (need > kResidentPairs && d.n_face_slices > kResidentRecords) return -1;
    form = form == 0 || need > kResidentPairs ? 0 : std::max(form, need);
  }
  *lds = 8;
  for (const DevProblem& d : plan->problems) {
    // the face vector's store, then u (registers) or two phases per junction and,
    // when each junction has its own 1/c0, u
    const int64_t arrays = form > 0 ? 1 : d.coef_si == 0 ? 2 : 3;
    *lds = std::max(*lds, 8 * (d.store_doubles + arrays * 2 * ((static_cast<int64_t>(d.Nj) + 1) / 2)));
  }
  return *lds <= plan->lds_limit ? form : -1;
}

// The resident kernels take the usual step: stencil 3, no voltage sources, noise
// from Philox with a given amplitude or none.
bool resident_runs(const Plan* plan, const jja_problem_run* runs) {
  for (size_t p = 0; p < plan->problems.size(); ++p)
    if (!runs[p].Vs.zero || runs[p].noise || (!runs[p].T.zero && !runs[p].sigma.base)) return false;
  return true;
}

template <typename... Args>
int launch_resident(Plan* plan, const void* kern, int32_t n, int64_t lds, hipStream_t stream, Args... args) {
  if (!kern) return fail(JJA_EUNSUPPORTED, "no resident kernel for this workgroup size");
  if (int rc = set_lds_limit(plan, kern, static_cast<int>(lds))) return rc;
  void* argv[] = {static_cast<void*>(&args)...};
  JJA_HIP(hipLaunchKernel(kern, dim3(n), dim3(plan->block_size), argv, static_cast<size_t>(lds), stream));
  return JJA_OK;
}

int launch_resident_evolve(Plan* plan, int32_t n, int form, int64_t lds, int32_t n_steps, int64_t step0,
                           hipStream_t stream) {
  const DevProblem* probs = plan->d_problems;
  const jja_problem_run* runs = plan->use_runs;
  const WorkItem* work = plan->use_work;
  return launch_resident(plan, resident_evolve_kernel(plan->block_size, form), n, lds, stream, probs, runs, work, n_steps,
                         step0);
}

int launch_resident_adjoint(Plan* plan, int32_t n, int form, int64_t lds, int64_t k_hi, int64_t k_lo,
                            hipStream_t stream) {
  const DevProblem* probs = plan->d_problems;
  const jja_adjoint_run* runs = plan->use_adj;
  const WorkItem* work = plan->use_work;
  return launch_resident(plan, resident_adjoint_kernel(plan->block_size, form), n, lds, stream, probs, runs, work, k_hi,
                         k_lo);
}

// Those also take the default current-phase relation alone, and inputs that are one
// value for all junctions or lie one after the other.
bool wide_runs(const Plan* plan, const jja_problem_run* runs) {
  if (!plan->d_wide || !resident_runs(plan, runs)) return false;
  auto plain = [](const jja_source& s) { return s.zero || s.s_i == 0 || s.s_i == 1; };
  for (size_t p = 0; p < plan->problems.size(); ++p)
    if (plan->problems[p].cpr_terms || !plain(runs[p].Is) || !plain(runs[p].f) || (!runs[p].T.zero && !plain(runs[p].sigma))) return false;
  return true;
}

int launch_wide(Plan* plan, const jja_problem_run* host_runs, int32_t n, int32_t n_steps, int64_t step0,
                hipStream_t stream) {
  bool gauss = false, uniform = true;
  for (size_t p = 0; p < plan->problems.size(); ++p) {
    const bool noisy = !host_runs[p].T.zero;
    gauss = gauss || noisy;
    uniform = uniform && plan->problems[p].coef_si == 0 && (!noisy || host_runs[p].sigma.s_i == 0);
  }
  const void* kern = wide_evolve_kernel(gauss, uniform);
  if (int rc = set_lds_limit(plan, kern, static_cast<int>(plan->wide_lds))) return rc;
  const DevProblem* probs = plan->d_problems;
  const jja_problem_run* runs = plan->use_runs;
  const WorkItem* work = plan->use_work;
  const WideDev* tables = plan->d_wide;
  void* argv[] = {&probs, &runs, &work, &tables, &n_steps, &step0};
  JJA_HIP(hipLaunchKernel(kern, dim3(n), dim3(kWideBlock), argv, static_cast<size_t>(plan->wide_lds), stream));
  return JJA_OK;
}

template <int STORE>
int launch_evolve_bs(Plan* plan, const WorkItem* work, int32_t n, int64_t lds, int32_t n_steps,
                     int64_t step0, hipStream_t stream) {
  switch (plan->block_size) {
    case 64: return launch_evolve_sw<64, STORE>(plan, work, n, lds, n_steps, step0, stream);
    case 128: return launch_evolve_sw<128, STORE>(plan, work, n, lds, n_steps, step0, stream);
    case 256: return launch_evolve_sw<256, STORE>(plan, work, n, lds, n_steps, step0, stream);
    case 512: return launch_evolve_sw<512, STORE>(plan, work, n, lds, n_steps, step0, stream);
    default: return launch_evolve_sw<1024, STORE>(plan, work, n, lds, n_steps, step0, stream);
  }
}

// The work items of a launch, largest problems first: workgroups are
// dispatched in index order as compute units free up, so this is a
// longest-first list schedule of uneven problems (the sort is stable: the
// columns of a problem, and problems of equal cost, keep their order).
void order_work(const Plan* plan, std::vector<WorkItem>& work) {
  std::stable_sort(work.begin(), work.end(), [plan](const WorkItem& a, const WorkItem& b) {
    return plan->cost[a.problem] > plan->cost[b.problem];
  });
}

// Work items of a split launch, from one item per column: every part of every
// column (its problem's part count), each column with its own barrier counter
// (slot). All workgroups of a cooperative launch are resident at once, so the
// order only decides placement: workgroups go to the eight XCDs in turn by
// block index (block b on XCD b mod 8), and the columns are packed onto the
// XCDs (largest part count first, each to the XCD with the most free blocks)
// so that the parts of a column share one L2. If a column does not fit, the
// items stay in column order.
std::vector<WorkItem> split_work(const Plan* plan, std::vector<WorkItem> cols) {
  order_work(plan, cols);
  constexpr size_t kXcd = 8;
  const size_t nc = cols.size();
  size_t total = 0;
  for (const WorkItem& c : cols) total += static_cast<size_t>(plan->problems[c.problem].parts);
  std::vector<WorkItem> out(total);
  // free block indices of each XCD, in ascending order
  std::vector<std::vector<size_t>> slots(kXcd);
  for (size_t b = 0; b < total; ++b) slots[b % kXcd].push_back(b);
  std::vector<size_t> next(kXcd, 0);
  std::vector<size_t> order(nc);
  for (size_t c = 0; c < nc; ++c) order[c] = c;
  std::stable_sort(order.begin(), order.end(), [&](size_t a, size_t b) {
    return plan->problems[cols[a].problem].parts > plan->problems[cols[b].problem].parts;
  });
  bool packed = true;
  for (size_t c : order) {
    const size_t G = static_cast<size_t>(plan->problems[cols[c].problem].parts);
    size_t best = kXcd;
    for (size_t x = 0; x < kXcd; ++x)
      if (slots[x].size() - next[x] >= G && (best == kXcd || slots[x].size() - next[x] > slots[best].size() - next[best]))
        best = x;
    if (best == kXcd) {
      packed = false;
      break;
    }
    for (size_t g = 0; g < G; ++g)
      out[slots[best][next[best]++]] = {cols[c].problem, static_cast<int32_t>(cols[c].column * G + g),
                                        static_cast<int32_t>(c)};
  }
  if (!packed) {
    out.clear();
    for (size_t c = 0; c < nc; ++c) {
      const int32_t G = plan->problems[cols[c].problem].parts;
      for (int32_t g = 0; g < G; ++g)
        out.push_back({cols[c].problem, cols[c].column * G + g, static_cast<int32_t>(c)});
    }
  }
  return out;
}

// Work items of a problem with W columns: one per column, or one per pair of
// columns (the last one alone when W is odd) in a plan with column pairs.
int32_t items_of(const Plan* plan, int32_t W) { return plan->pairs ? (W + 1) / 2 : W; }

// Barrier words of n work items (arrival counter, XCD set), zeroed on the
// stream before a split launch (the array is sized at plan creation).
int reset_counters(Plan* plan, size_t n, hipStream_t stream) {
  n *= 2;
  if (n > plan->ctr_cap) return fail(JJA_EINVAL, "launch has more columns than the plan was sized for");
  JJA_HIP(hipMemsetAsync(plan->d_ctrs, 0, n * sizeof(uint32_t), stream));
  return JJA_OK;
}

// Cooperative launch of a split kernel: all n workgroups resident at once (the
// column barriers need every part of a column running), or an error. Each
// workgroup gets lds_bytes of dynamic LDS.
template <typename... Args>
int launch_cooperative(Plan* plan, const void* kern, int BS, int32_t n, int64_t lds_bytes, hipStream_t stream,
                       Args... args) {
  const int lds = static_cast<int>(lds_bytes);
  int per_cu = -1;
  for (const auto& a : plan->per_cu)
    if (a.first == kern) per_cu = a.second;
  if (lds > 0)
    if (int rc = raise_lds_attr(kern, lds)) return rc;
  if (per_cu < 0) {
    JJA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kern, BS, static_cast<size_t>(lds)));
    plan->per_cu.push_back({kern, per_cu});
  }
  if (static_cast<int64_t>(per_cu) * plan->n_cu < n)
    return fail(JJA_EUNSUPPORTED, "split launch of " + std::to_string(n) + " workgroups; the device holds " +
                                      std::to_string(static_cast<int64_t>(per_cu) * plan->n_cu) + " at once");
  void* argv[] = {static_cast<void*>(&args)...};
  // a graph takes the plain launch: its workgroups fit on the device together (above)
  bool capturing = false;
  if (int rc = capture_state(stream, &capturing)) return rc;
  if (capturing) {
    JJA_HIP(hipLaunchKernel(kern, dim3(n), dim3(BS), argv, static_cast<size_t>(lds), stream));
    return JJA_OK;
  }
  JJA_HIP(hipLaunchCooperativeKernel(kern, dim3(n), dim3(BS), argv, static_cast<size_t>(lds), stream));
  return JJA_OK;
}

template <int BS>
int launch_evolve_split_bs(Plan* plan, int32_t n, int32_t n_steps, int64_t step0, hipStream_t stream) {
  const DevProblem* probs = plan->d_problems;
  const jja_problem_run* runs = plan->use_runs;
  const WorkItem* work = plan->use_work;
  const void* kern = plan->pairs ? reinterpret_cast<const void*>(evolve_split_kernel<BS, 3, BS <= 512>)
                                 : reinterpret_cast<const void*>(evolve_split_kernel<BS, 3, false>);
  return launch_cooperative(plan, kern, BS, n, plan->split_lds, stream, probs, runs, work, n_steps, step0, plan->d_ctrs,
                            plan->d_err, plan->wait_limit);
}

int launch_evolve_split(Plan* plan, int32_t n, int32_t n_steps, int64_t step0, hipStream_t stream) {
  if (plan->stencil_width != 3) return fail(JJA_EUNSUPPORTED, "split columns: stencil width 3 only");
  switch (plan->block_size) {
    case 256: return launch_evolve_split_bs<256>(plan, n, n_steps, step0, stream);
    case 512: return launch_evolve_split_bs<512>(plan, n, n_steps, step0, stream);
    case 1024: return launch_evolve_split_bs<1024>(plan, n, n_steps, step0, stream);
    default: return fail(JJA_EUNSUPPORTED, "split columns: workgroups of 256, 512 or 1024 threads");
  }
}

// Whether a run can go to the kernels that keep each part's junctions on chip: the
// usual step (stencil 3, no voltage sources, noise from Philox with a given
// amplitude or none).
bool parts_run(const Plan* plan, const jja_problem_run& r) {
  return plan->d_parts && plan->stencil_width == 3 && r.Vs.zero && !r.noise && (r.T.zero || r.sigma.base);
}

int launch_evolve_parts(Plan* plan, int32_t n, int32_t n_steps, int64_t step0, hipStream_t stream) {
  const DevProblem* probs = plan->d_problems;
  const jja_problem_run* runs = plan->use_runs;
  const WorkItem* work = plan->use_work;
  const void* tables = plan->d_parts;
  if (int rc = launch_cooperative(plan, plan->parts_evolve, plan->block_size, n, plan->parts_lds, stream, probs, runs, work,
                                  tables, n_steps, step0, plan->d_parts_seq, plan->d_err, plan->wait_limit))
    return rc;
  hipLaunchKernelGGL(evolve_spoil_kernel, dim3(n / plan->parts), dim3(kSpoilBlock), 0, stream, runs,
                     plan->problems[0].Nj, plan->d_err, plan->host_err, n_steps, step0);
  JJA_HIP(hipGetLastError());
  return JJA_OK;
}

int launch_adjoint_parts(Plan* plan, int32_t n, int64_t k_hi, int64_t k_lo, hipStream_t stream) {
  const DevProblem* probs = plan->d_problems;
  const jja_adjoint_run* runs = plan->use_adj;
  const WorkItem* work = plan->use_work;
  const void* tables = plan->d_parts;
  if (int rc = launch_cooperative(plan, plan->parts_adjoint, plan->block_size, n, plan->parts_lds, stream, probs, runs, work,
                                  tables, k_hi, k_lo, plan->d_parts_seq, plan->d_err, plan->wait_limit))
    return rc;
  hipLaunchKernelGGL(adjoint_spoil_kernel, dim3(n / plan->parts), dim3(kSpoilBlock), 0, stream, runs,
                     plan->problems[0].Nj, plan->problems[0].Nf, plan->d_err, plan->host_err);
  JJA_HIP(hipGetLastError());
  return JJA_OK;
}

template <int BS>
int launch_adjoint_split_bs(Plan* plan, int32_t n, int64_t k_hi, int64_t k_lo, hipStream_t stream) {
  const DevProblem* probs = plan->d_problems;
  const jja_adjoint_run* runs = plan->use_adj;
  const WorkItem* work = plan->use_work;
  const void* kern = plan->pairs ? reinterpret_cast<const void*>(adjoint_split_kernel<BS, BS <= 512>)
                                 : reinterpret_cast<const void*>(adjoint_split_kernel<BS, false>);
  return launch_cooperative(plan, kern, BS, n, plan->split_lds, stream, probs, runs, work, k_hi, k_lo, plan->d_ctrs,
                            plan->d_err, plan->wait_limit);
}

int launch_adjoint_split(Plan* plan, int32_t n, int64_t k_hi, int64_t k_lo, hipStream_t stream) {
  switch (plan->block_size) {
    case 256: return launch_adjoint_split_bs<256>(plan, n, k_hi, k_lo, stream);
    case 512: return launch_adjoint_split_bs<512>(plan, n, k_hi, k_lo, stream);
    case 1024: return launch_adjoint_split_bs<1024>(plan, n, k_hi, k_lo, stream);
    default: return fail(JJA_EUNSUPPORTED, "split columns: workgroups of 256, 512 or 1024 threads");
  }
}

template <bool GLOBAL>
int launch_adjoint_bs(Plan* plan, const WorkItem* work, int32_t n, int64_t lds, int64_t k_hi,
                      int64_t k_lo, hipStream_t stream) {
  switch (plan->block_size) {
    case 64: return launch_adjoint<64, GLOBAL>(plan, work, n, lds, k_hi, k_lo, stream);
    case 128: return launch_adjoint<128, GLOBAL>(plan, work, n, lds, k_hi, k_lo, stream);
    case 256: return launch_adjoint<256, GLOBAL>(plan, work, n, lds, k_hi, k_lo, stream);
    case 512: return launch_adjoint<512, GLOBAL>(plan, work, n, lds, k_hi, k_lo, stream);
    default: return launch_adjoint<1024, GLOBAL>(plan, work, n, lds, k_hi, k_lo, stream);
  }
}

template <int BS>
int launch_spd_solve(Plan* plan, int32_t p, const double* b, int64_t ldb, double* x, int64_t ldx,
                     int32_t cols, double* zbuf, hipStream_t stream) {
  const bool global = plan->zbuf_doubles[p] > 0;
  const int lds = global ? 8 : static_cast<int>(std::max<int64_t>(plan->lds_bytes[p], 8));
  const void* kern = global ? reinterpret_cast<const void*>(spd_solve_kernel<BS, true>)
                            : reinterpret_cast<const void*>(spd_solve_kernel<BS, false>);
  if (int rc = set_lds_limit(plan, kern, lds)) return rc;
  if (global)
    hipLaunchKernelGGL((spd_solve_kernel<BS, true>), dim3(cols), dim3(BS), static_cast<size_t>(lds), stream,
                       plan->d_problems, p, b, ldb, x, ldx, zbuf);
  else
    hipLaunchKernelGGL((spd_solve_kernel<BS, false>), dim3(cols), dim3(BS), static_cast<size_t>(lds), stream,
                       plan->d_problems, p, b, ldb, x, ldx, zbuf);
  JJA_HIP(hipGetLastError());
  return JJA_OK;
}

// scratch's device address on each GPU, taken once per device with that device
// current (the array's name is a host-side stand-in, not a device address)
constexpr int kMaxDevices = 64;
double* g_scratch_ptr[kMaxDevices] = {};
std::mutex g_scratch_mu;

int scratch_ptr(int device, double** out) {
  if (device < 0 || device >= kMaxDevices) return fail(JJA_EINVAL, "jja_solve_noalloc: device index out of range");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[device]) {
    int cur = -1;
    JJA_HIP(hipGetDevice(&cur));
    if (cur != device) return fail(JJA_EINVAL, "jja_solve_noalloc: the plan's device is not the current device");
    void* ptr = nullptr;
    JJA_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return fail(JJA_EHIP, "jja_solve_noalloc: no device address for the scratch array");
    g_scratch_ptr[device] = static_cast<double*>(ptr);
  }
  *out = g_scratch_ptr[device];
  return JJA_OK;
}

}  // namespace

extern "C" {

const char* jja_last_error(void) { return g_error.c_str(); }

int jja_plan_validate(int32_t n_problems, const jja_problem_desc* descs) {
  if (n_problems <= 0 || !descs) return fail(JJA_EINVAL, "jja_plan_validate: invalid arguments");
  if (int rc = check_plan_shapes(n_problems, descs)) return rc;
  for (int32_t p = 0; p < n_problems; ++p)
    if (int rc = validate(descs[p])) return rc;
  return JJA_OK;
}

int jja_slabs_fit(const jja_problem_desc* d) {
  if (!d) return fail(JJA_EINVAL, "jja_slabs_fit: invalid arguments");
  try {
    if (int rc = check_plan_shapes(1, d)) return rc;
    if (int rc = validate(*d)) return rc;
    return wants_slabs(*d) && slabs_fit(*d, d->parts, kSplitLdsMax) ? 1 : 0;
  } catch (const std::bad_alloc&) {
    return fail(JJA_ENOMEM, "jja_slabs_fit: out of host memory");
  }
}

int jja_plan_create(int32_t n_problems, const jja_problem_desc* descs, jja_plan** out) {
  if (!out || n_problems <= 0 || !descs) return fail(JJA_EINVAL, "jja_plan_create: invalid arguments");
  *out = nullptr;
  if (int rc = check_plan_shapes(n_problems, descs)) return rc;
  Plan* plan = new Plan();
  plan->parts = 1;
  for (int32_t p = 0; p < n_problems; ++p) plan->parts = std::max(plan->parts, parts_of(descs[p]));
  plan->pairs = descs[0].column_pairs != 0;
  plan->block_size = descs[0].block_size / parts_of(descs[0]);
  plan->stencil_width = descs[0].stencil_width;
  int rc = JJA_OK;
  hipDeviceProp_t prop;
  if (hipGetDevice(&plan->device) != hipSuccess ||
      hipGetDeviceProperties(&prop, plan->device) != hipSuccess) {
    delete plan;
    return fail(JJA_EHIP, "jja_plan_create: no HIP device");
  }
  plan->lds_limit = static_cast<int64_t>(prop.sharedMemPerBlock);
  plan->n_cu = prop.multiProcessorCount;
  for (int32_t p = 0; p < n_problems && rc == JJA_OK; ++p) {
    const jja_problem_desc& d = descs[p];
    rc = validate(d);
    if (rc) break;
    DevProblem dp{};
    dp.Nj = d.n_junctions;
    dp.Nf = d.n_faces;
    dp.sw = d.stencil_width;
    dp.BS = d.block_size;
    dp.parts = parts_of(d);
    dp.n_face_slices = d.n_face_slices;
    dp.n_solve_slices = d.n_solve_slices;
    dp.max_stage_rows = d.max_stage_rows;
    dp.copy_rows = d.face_copy_rows;
    dp.index_bytes = d.index_bytes;
    dp.val_bytes = static_cast<int32_t>(d.n_entries * static_cast<int64_t>(sizeof(double)));
    dp.cpr_terms = d.cpr_terms;
    for (int k = 0; k < JJA_CPR_MAX_TERMS; ++k) dp.cpr_coef[k] = d.cpr_coef[k];
    if (d.lattice_rows) {
      const int32_t R = d.lattice_rows, C = d.lattice_cols, H = (C + 1) / 2;
      dp.lat_rows = R;
      dp.lat_cols = C;
      dp.lat_es = H + (H & 1);
      dp.lat_ef = d.index_bytes == 4 ? (dp.lat_es + 3) & ~3 : dp.lat_es;
      // a split column solves its tridiagonal systems part by part in LDS
      // when a part's modes and block ends fit
      const int32_t np = parts_of(d);
      if (np > 1) {
        const int32_t mp = 2 * ((H + np - 1) / np);  // mode pairs (i, C-1-i) per part, two slots each
        const int32_t bp = std::max(1, std::min(R, JJA_LATTICE_TRI_THREADS / mp));
        const int64_t need = (static_cast<int64_t>(R) * mp + 4 * static_cast<int64_t>(bp) * mp) * 8;
        if (need <= kSplitLdsMax) {
          dp.lat_mp = mp;
          dp.lat_bp = bp;
          plan->split_lds = std::max(plan->split_lds, need);
        }
      }
      dp.lat_cp = (C + JJA_LATTICE_CHUNK - 1) / JJA_LATTICE_CHUNK * JJA_LATTICE_CHUNK;
      dp.lat_t0 = static_cast<int64_t>(d.n_faces) + (d.n_faces & 1);
      dp.lat_g = d.lattice_g;
      if ((rc = upload(plan, d.lattice_sine, static_cast<size_t>(dp.lat_es) * dp.lat_cp, &dp.lat_sine))) break;
      {
        // mode j of row i at i*CP + (j & 1)*(CP/2) + j/2 (CP is a multiple of 14, so even)
        const size_t cp = dp.lat_cp, half = cp / 2, n = static_cast<size_t>(dp.lat_es) * cp;
        std::vector<double> split(n);
        for (size_t i = 0; i < static_cast<size_t>(dp.lat_es); ++i)
          for (size_t j = 0; j < cp; ++j) split[i * cp + (j & 1) * half + j / 2] = d.lattice_sine[i * cp + j];
        if ((rc = upload(plan, split.data(), n, &dp.lat_sine_p))) break;
      }
      if ((rc = upload(plan, d.lattice_inv, static_cast<size_t>(R) * dp.lat_cp, &dp.lat_inv))) break;
      // padded LDS form: the table's steps and their mirrors stay inside a side of
      // 8 elements or more; rows of 32 k + 4 doubles put the 16 rows of a tile on all banks
      const DstShape dc(C), dr(R);
      const int32_t ld = dc.padded() + 4;
      const int64_t buf = static_cast<int64_t>(dr.padded()) * ld;
      const int64_t tables = dc.entries() + (R == C ? 0 : dr.entries());
      const bool solve_in_modes = d.lattice_gc > 0.0;  // both factors known
      if (solve_in_modes && d.index_bytes == 2 && R <= TileShape::kSide && C <= TileShape::kSide) {
        dp.lat_tile = 1;
        dp.lat_ld = TileShape::kLd;
        dp.lat_buf = TileShape::kSide * TileShape::kLd;
        dp.lat_tab = 2 * dp.lat_buf;
        dp.store_doubles = dp.lat_tab + 3 * TileShape::kTable;
        const std::vector<double> t = tile_table(R, C, d.lattice_g, d.lattice_gc);
        if ((rc = upload(plan, t.data(), t.size(), &dp.lat_table))) break;
      } else if (solve_in_modes && d.index_bytes == 2 && R >= 8 && C >= 8 && 8 * (2 * buf + tables) <= plan->lds_limit) {
        dp.lat_ld = ld;
        dp.lat_buf = static_cast<int32_t>(buf);
        dp.lat_tab = static_cast<int32_t>(2 * buf);
        dp.store_doubles = static_cast<int32_t>(2 * buf + tables);
        std::vector<double> t = dst_table(C), lam(static_cast<size_t>(buf), 0.0);
        if (R != C) {
          const std::vector<double> tr = dst_table(R);
          t.insert(t.end(), tr.begin(), tr.end());
        }
        const std::vector<double> mc = dst_eigenvalues(C), mr = dst_eigenvalues(R);
        for (size_t i = 0; i < static_cast<size_t>(R); ++i)
          for (size_t j = 0; j < static_cast<size_t>(C); ++j)
            lam[i * ld + j] = 1.0 / (d.lattice_g * mr[i] + d.lattice_gc * mc[j]);
        if ((rc = upload(plan, t.data(), t.size(), &dp.lat_table))) break;
        if ((rc = upload(plan, lam.data(), lam.size(), &dp.lat_lam))) break;
      }
    }
    const size_t Nj = d.n_junctions, Nf = d.n_faces;
    if ((rc = upload(plan, d.Ic, Nj, &dp.Ic))) break;
    if ((rc = upload(plan, d.Rv, Nj, &dp.Rv))) break;
    if ((rc = upload(plan, d.coef, Nj * d.stencil_width, &dp.coef))) break;
    dp.coef_si = 0;  // every coefficient row one value (uniform R and C): read one address
    for (int32_t k = 0; k < d.stencil_width && !dp.coef_si; ++k)
      for (size_t j = 1; j < Nj; ++j)
        if (d.coef[k * Nj + j] != d.coef[k * Nj]) {
          dp.coef_si = 1;
          break;
        }
    {
      std::vector<double> rc0(Nj);
      for (size_t j = 0; j < Nj; ++j) rc0[j] = 1.0 / d.coef[j];
      if ((rc = upload(plan, rc0.data(), Nj, &dp.rc0))) break;
    }
    // incidence codes and face rows by store address
    auto address = [&](int32_t q) { return dp.lat_ld ? q / dp.lat_cols * dp.lat_ld + q % dp.lat_cols : q; };
    {
      std::vector<int32_t> code(d.junc_code, d.junc_code + 2 * Nj);
      for (int32_t& c : code)
        if (c >= 0) c = 2 * address(c >> 1) + (c & 1);
      if ((rc = upload(plan, code.data(), code.size(), &dp.junc_code))) break;
    }
    if (Nf) {
      if ((rc = upload(plan, d.face_of_pos, Nf, &dp.face_of_pos))) break;
      if ((rc = upload(plan, d.face_slices, static_cast<size_t>(d.n_face_slices), &dp.face_slices))) break;
      if ((rc = upload(plan, d.solve_slices, static_cast<size_t>(d.n_solve_slices), &dp.solve_slices))) break;
      if ((rc = upload(plan, d.solve_wave_ptr, static_cast<size_t>(d.block_size / kWave + 1), &dp.wave_ptr))) break;
      if ((rc = upload(plan, d.face_code, static_cast<size_t>(d.n_face_entries), &dp.face_code))) break;
      if ((rc = upload(plan, d.slice_rows, static_cast<size_t>(d.n_slice_rows), &dp.slice_rows))) break;
      dp.face_addr = dp.slice_rows;
      if (dp.lat_ld) {
        std::vector<int32_t> at(d.slice_rows, d.slice_rows + d.n_slice_rows);
        for (int32_t& q : at)
          if (q >= 0) q = address(q);
        if ((rc = upload(plan, at.data(), at.size(), &dp.face_addr))) break;
      }
      {
        // face index of every row slot a face record finishes (the flux input)
        std::vector<int32_t> fid(static_cast<size_t>(d.n_slice_rows), -1);
        for (int32_t k = 0; k < d.n_face_slices; ++k) {
          const jja_slice& m = d.face_slices[k];
          if (!(m.flags & JJA_SLICE_FINISH)) continue;
          for (int32_t i = 0; i < (m.flags >> 16); ++i) {
            const int32_t pos = d.slice_rows[m.rowbase + i];
            if (pos >= 0) fid[static_cast<size_t>(m.rowbase) + i] = d.face_of_pos[pos];
          }
        }
        if ((rc = upload(plan, fid.data(), fid.size(), &dp.face_fid))) break;
      }
      if ((rc = upload(plan, d.ent_val, static_cast<size_t>(d.n_entries), &dp.ent_val))) break;
      if (d.index_bytes == 2) {
        const uint16_t* o = nullptr;
        if ((rc = upload(plan, static_cast<const uint16_t*>(d.ent_off), static_cast<size_t>(d.n_index), &o))) break;
        dp.ent_off = o;
      } else {
        const uint32_t* o = nullptr;
        if ((rc = upload(plan, static_cast<const uint32_t*>(d.ent_off), static_cast<size_t>(d.n_index), &o))) break;
        dp.ent_off = o;
      }
    }
    {
      static const double zeros[8] = {0, 0, 0, 0, 0, 0, 0, 0};
      if ((rc = upload(plan, zeros, 8, &dp.zero))) break;
    }
    if (!dp.lat_ld) dp.store_doubles = (d.n_faces + d.max_stage_rows + 1) & ~1;
    plan->problems.push_back(dp);
    plan->lds_bytes.push_back(d.index_bytes == 2 ? static_cast<int64_t>(dp.store_doubles) * 8 : 0);
    // work of one column step in factor-entry units (a lattice solve: its multiply-adds)
    const int64_t solve_work = d.lattice_rows ? static_cast<int64_t>(d.n_faces) * (d.lattice_cols + 1) : d.n_entries;
    plan->cost.push_back(solve_work + d.n_face_entries + 8 * static_cast<int64_t>(d.n_junctions));
    plan->zbuf_doubles.push_back(d.index_bytes == 2 ? 0 : static_cast<int64_t>(d.n_faces) + d.max_stage_rows);
    plan->max_cols.push_back(d.max_columns);
  }
  if (rc == JJA_OK) {
    const DevProblem* dprob = nullptr;
    rc = upload(plan, plan->problems.data(), plan->problems.size(), &dprob);
    plan->d_problems = const_cast<DevProblem*>(dprob);
  }
  // launch descriptors, work lists and barrier words for the largest runs
  // the descriptors allow: launches allocate nothing
  size_t items = 0, blocks = 0;
  for (size_t p = 0; p < plan->max_cols.size(); ++p) {
    const size_t it = static_cast<size_t>(items_of(plan, plan->max_cols[p]));
    items += it;
    blocks += it * static_cast<size_t>(plan->problems[p].parts);
  }
  auto alloc = [&](size_t bytes, void** out) {
    if (rc != JJA_OK) return;
    void* d = nullptr;
    if (hipMalloc(&d, bytes) != hipSuccess) {
      rc = fail(JJA_ENOMEM, "jja_plan_create: device allocation failed");
      return;
    }
    plan->allocations.push_back(d);
    *out = d;
  };
  alloc(sizeof(jja_problem_run) * n_problems, reinterpret_cast<void**>(&plan->d_runs));
  alloc(sizeof(jja_adjoint_run) * n_problems, reinterpret_cast<void**>(&plan->d_adj));
  alloc(sizeof(WorkItem) * blocks, reinterpret_cast<void**>(&plan->d_work));
  plan->work_cap = blocks;
  if (plan->parts > 1) {
    alloc(2 * sizeof(uint32_t) * items, reinterpret_cast<void**>(&plan->d_ctrs));
    plan->ctr_cap = 2 * items;
  }
  if (rc == JJA_OK && n_problems == 1) rc = descs[0].domains ? create_domains(plan, descs[0]) : create_slabs(plan, descs[0]);
  if (rc == JJA_OK && plan->d_parts) {
    const std::vector<uint32_t> seq(static_cast<size_t>(descs[0].max_columns) * plan->parts, 0u);
    const uint32_t* d = nullptr;
    rc = upload(plan, seq.data(), seq.size(), &d);
    plan->d_parts_seq = const_cast<uint32_t*>(d);
    if (rc == JJA_OK && hipHostMalloc(reinterpret_cast<void**>(&plan->host_err), sizeof(int32_t), hipHostMallocMapped) != hipSuccess)
      rc = fail(JJA_ENOMEM, "jja_plan_create: pinned host allocation failed");
    if (rc == JJA_OK) *plan->host_err = 0;
  }
  if (rc == JJA_OK) rc = create_wide(plan, descs, n_problems);
  if (rc == JJA_OK && hipEventCreateWithFlags(&plan->done, hipEventDisableTiming) != hipSuccess)
    rc = fail(JJA_EHIP, "jja_plan_create: hipEventCreateWithFlags failed");
  if (rc == JJA_OK && plan->parts > 1) {
    void* d = nullptr;
    if (hipMalloc(&d, 2 * sizeof(int32_t)) != hipSuccess || hipMemset(d, 0, 2 * sizeof(int32_t)) != hipSuccess) {
      rc = fail(JJA_ENOMEM, "jja_plan_create: device allocation failed");
    } else {
      plan->allocations.push_back(d);
      plan->d_err = static_cast<int32_t*>(d);
    }
  }
  if (rc != JJA_OK) {
    free_plan(plan);
    return rc;
  }
  *out = reinterpret_cast<jja_plan*>(plan);
  return JJA_OK;
}

int jja_plan_status(jja_plan* p) {
  Plan* plan = reinterpret_cast<Plan*>(p);
  if (!plan) return fail(JJA_EINVAL, "jja_plan_status: invalid arguments");
  if (!plan->d_err) return JJA_OK;
  int32_t e = 0;
  JJA_HIP(hipMemcpy(&e, plan->d_err, sizeof(e), hipMemcpyDeviceToHost));
  if (!e) return JJA_OK;
  JJA_HIP(hipMemset(plan->d_err, 0, sizeof(int32_t)));
  if (plan->host_err) __atomic_store_n(plan->host_err, 0, __ATOMIC_RELAXED);
  return fail(JJA_EHIP, "a column barrier of a split launch gave up waiting; its results are invalid");
}

int jja_plan_poll(jja_plan* p) {
  Plan* plan = reinterpret_cast<Plan*>(p);
  if (!plan) return fail(JJA_EINVAL, "jja_plan_poll: invalid arguments");
  if (!plan->host_err || !__atomic_load_n(plan->host_err, __ATOMIC_RELAXED)) return JJA_OK;
  return jja_plan_status(p);
}

int64_t jja_plan_one_xcd_parts(jja_plan* p) {
  Plan* plan = reinterpret_cast<Plan*>(p);
  if (!plan) return fail(JJA_EINVAL, "jja_plan_one_xcd_parts: invalid arguments");
  if (!plan->d_err) return 0;
  int32_t n = 0;
  JJA_HIP(hipMemcpy(&n, plan->d_err + 1, sizeof(n), hipMemcpyDeviceToHost));
  JJA_HIP(hipMemset(plan->d_err + 1, 0, sizeof(int32_t)));
  return n;
}

int jja_plan_set_wait_limit(jja_plan* p, uint32_t polls) {
  Plan* plan = reinterpret_cast<Plan*>(p);
  if (!plan) return fail(JJA_EINVAL, "jja_plan_set_wait_limit: invalid arguments");
  plan->wait_limit = polls;
  return JJA_OK;
}

int jja_plan_destroy(jja_plan* p) {
  if (!p) return JJA_OK;
  free_plan(reinterpret_cast<Plan*>(p));
  return JJA_OK;
}

int64_t jja_plan_lds_bytes(const jja_plan* p, int32_t i) {
  const Plan* plan = reinterpret_cast<const Plan*>(p);
  if (!plan || i < 0 || i >= static_cast<int32_t>(plan->lds_bytes.size())) return 0;
  return plan->lds_bytes[i] <= plan->lds_limit ? plan->lds_bytes[i] : 0;
}

int64_t jja_plan_zbuf_doubles(const jja_plan* p, int32_t i) {
  const Plan* plan = reinterpret_cast<const Plan*>(p);
  if (!plan || i < 0 || i >= static_cast<int32_t>(plan->zbuf_doubles.size())) return 0;
  return plan->zbuf_doubles[i];
}

int jja_evolve(jja_plan* p, const jja_problem_run* runs, int32_t n_steps, int64_t step0,
               void* stream_ptr) {
  Plan* plan = reinterpret_cast<Plan*>(p);
  if (!plan || !runs || n_steps < 0 || step0 < 0) return fail(JJA_EINVAL, "jja_evolve: invalid arguments");
  if (n_steps == 0) return JJA_OK;
  const int32_t np = static_cast<int32_t>(plan->problems.size());
  std::vector<WorkItem> work, work_g;
  int64_t lds = 0;
  for (int32_t i = 0; i < np; ++i) {
    const jja_problem_run& r = runs[i];
    if (plan->problems[i].Nj == 0)
      return fail(JJA_EINVAL, "jja_evolve: problem " + std::to_string(i) + " is a matrix plan without junctions");
    if (r.W <= 0 || !r.theta) return fail(JJA_EINVAL, "jja_evolve: run needs W > 0 and theta");
    if (r.W > plan->max_cols[i])
      return fail(JJA_EINVAL, "jja_evolve: problem " + std::to_string(i) + " has more columns than its max_columns");
    if (r.dt <= 0) return fail(JJA_EINVAL, "jja_evolve: dt must be positive");
    if (plan->parts_only && !parts_run(plan, r))
      return fail(JJA_EUNSUPPORTED, "jja_evolve: subdomains take no voltage sources, given normals or varying temperature");
    if (!r.Is.base || !r.Vs.base || !r.f.base || !r.T.base)
      return fail(JJA_EINVAL, "jja_evolve: every source needs a base array");
    if (!r.Vs.zero && !r.theta_s) return fail(JJA_EINVAL, "jja_evolve: non-zero Vs needs theta_s");
    const bool global = plan->zbuf_doubles[i] > 0;
    if (global && !r.zbuf)
      return fail(JJA_EINVAL, "jja_evolve: problem " + std::to_string(i) + " needs a global face store (zbuf)");
    // an LDS face store's junction pass writes u for its face phase (a split
    // plan's columns all use the global store, faceless ones included)
    if (!global && plan->parts == 1 && !r.u)
      return fail(JJA_EINVAL, "jja_evolve: problem " + std::to_string(i) + " (LDS face store) needs u");
    if (!global && plan->lds_bytes[i] > plan->lds_limit)
      return fail(JJA_EUNSUPPORTED, "jja_evolve: face vector of problem " + std::to_string(i) +
                                        " needs " + std::to_string(plan->lds_bytes[i]) +
                                        " bytes of LDS; limit " + std::to_string(plan->lds_limit));
    if (!global) lds = std::max(lds, plan->lds_bytes[i]);
    for (int32_t w = 0; w < items_of(plan, r.W); ++w) (global ? work_g : work).push_back({i, w});
  }
  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  bool capturing = false;
  if (int rc = capture_state(stream, &capturing)) return rc;
  if (capturing && plan->parts > 1 && !parts_run(plan, runs[0])) return refuse_capture("jja_evolve");
  if (int rc = capturing ? JJA_OK : claim_stream(plan, stream)) return rc;
  if (int rc = stage(plan, plan->d_runs, runs, static_cast<size_t>(np), plan->h_runs, plan->runs_valid, stream, capturing,
                     &plan->use_runs))
    return rc;
  int rc = JJA_OK;
  if (plan->parts > 1) {
    // every problem of a split plan has the global face store (validated; a
    // circuit without faces has none and needs none): all columns, one launch
    work.insert(work.end(), work_g.begin(), work_g.end());
    const std::vector<WorkItem> split = split_work(plan, work);
    if ((rc = upload_work(plan, split, stream, capturing))) return rc;
    if (parts_run(plan, runs[0]))
      rc = launch_evolve_parts(plan, static_cast<int32_t>(split.size()), n_steps, step0, stream);
    else if ((rc = reset_counters(plan, work.size(), stream)))
      return rc;
    else
      rc = launch_evolve_split(plan, static_cast<int32_t>(split.size()), n_steps, step0, stream);
  } else {
    // one launch: a kernel for one kind of face store, or one that takes either
    const int32_t n_lds = static_cast<int32_t>(work.size()), n_g = static_cast<int32_t>(work_g.size());
    work.insert(work.end(), work_g.begin(), work_g.end());
    order_work(plan, work);
    if ((rc = upload_work(plan, work, stream, capturing))) return rc;
    if (lds < 8) lds = 8;
    const int32_t n = n_lds + n_g;
    int64_t resident_lds = 0;
    const int form = n_g == 0 && resident_runs(plan, runs) ? resident_layout(plan, &resident_lds) : -1;
    if (form >= 0)
      rc = launch_resident_evolve(plan, n, form, resident_lds, n_steps, step0, stream);
    else if (n_g == 0 && wide_runs(plan, runs))
      rc = launch_wide(plan, runs, n, n_steps, step0, stream);
    else if (n_g == 0)
      rc = launch_evolve_bs<0>(plan, plan->use_work, n, lds, n_steps, step0, stream);
    else if (n_lds == 0)
      rc = launch_evolve_bs<1>(plan, plan->use_work, n, 8, n_steps, step0, stream);
    else
      rc = launch_evolve_bs<2>(plan, plan->use_work, n, lds, n_steps, step0, stream);
  }
  if (rc) return rc;
  return capturing ? JJA_OK : mark_launched(plan, stream);  // nothing has been launched yet
}

int jja_adjoint(jja_plan* p, const jja_adjoint_run* runs, int64_t k_hi, int64_t k_lo, void* stream_ptr) {
  Plan* plan = reinterpret_cast<Plan*>(p);
  if (!plan || !runs || k_lo < 0 || k_hi < k_lo) return fail(JJA_EINVAL, "jja_adjoint: invalid arguments");
  if (plan->stencil_width != 3) return fail(JJA_EUNSUPPORTED, "jja_adjoint: stencil width 3 only");
  for (const DevProblem& P : plan->problems)
    if (P.cpr_terms != 0) return fail(JJA_EUNSUPPORTED, "jja_adjoint: the default current-phase relation only");
  const int32_t np = static_cast<int32_t>(plan->problems.size());
  std::vector<WorkItem> work, work_g;
  int64_t lds = 0;
  for (int32_t i = 0; i < np; ++i) {
    const jja_adjoint_run& r = runs[i];
    if (r.W <= 0 || !r.hist || !r.lam || !r.u || !r.grad_Ic || !r.grad_Is || !r.grad_f)
      return fail(JJA_EINVAL, "jja_adjoint: run needs W > 0, hist, lam, u and the gradient arrays");
    if (r.W > plan->max_cols[i])
      return fail(JJA_EINVAL, "jja_adjoint: problem " + std::to_string(i) + " has more columns than its max_columns");
    if (r.hist_m0 > k_lo - 2) return fail(JJA_EINVAL, "jja_adjoint: hist must start at k_lo - 2 or earlier");
    if (r.g && (!r.g_slot || r.g_lo < r.slot_t0 || r.g_hi < r.g_lo))
      return fail(JJA_EINVAL, "jja_adjoint: g needs g_slot covering [g_lo, g_hi)");
    const bool global = plan->zbuf_doubles[i] > 0;
    if (global && !r.zbuf)
      return fail(JJA_EINVAL, "jja_adjoint: problem " + std::to_string(i) + " needs a global face store (zbuf)");
    if (!global && plan->lds_bytes[i] > plan->lds_limit)
      return fail(JJA_EUNSUPPORTED, "jja_adjoint: face vector of problem " + std::to_string(i) + " exceeds LDS");
    if (!global) lds = std::max(lds, plan->lds_bytes[i]);
    for (int32_t w = 0; w < items_of(plan, r.W); ++w) (global ? work_g : work).push_back({i, w});
  }
  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  bool capturing = false;
  if (int rc = capture_state(stream, &capturing)) return rc;
  if (capturing && plan->parts > 1 && !plan->d_parts) return refuse_capture("jja_adjoint");
  if (int rc = capturing ? JJA_OK : claim_stream(plan, stream)) return rc;
  if (int rc = stage(plan, plan->d_adj, runs, static_cast<size_t>(np), plan->h_adj, plan->adj_valid, stream, capturing,
                     &plan->use_adj))
    return rc;
  int rc = JJA_OK;
  if (plan->parts > 1) {
    work.insert(work.end(), work_g.begin(), work_g.end());
    const std::vector<WorkItem> split = split_work(plan, work);
    if ((rc = upload_work(plan, split, stream, capturing))) return rc;
    if (plan->d_parts)
      rc = launch_adjoint_parts(plan, static_cast<int32_t>(split.size()), k_hi, k_lo, stream);
    else if ((rc = reset_counters(plan, work.size(), stream)))
      return rc;
    else
      rc = launch_adjoint_split(plan, static_cast<int32_t>(split.size()), k_hi, k_lo, stream);
  } else {
    const int32_t n_lds = static_cast<int32_t>(work.size()), n_g = static_cast<int32_t>(work_g.size());
    order_work(plan, work);
    order_work(plan, work_g);
    work.insert(work.end(), work_g.begin(), work_g.end());
    if ((rc = upload_work(plan, work, stream, capturing))) return rc;
    if (lds < 8) lds = 8;
    int64_t resident_lds = 0;
    const int form = n_lds && !n_g ? resident_layout(plan, &resident_lds) : -1;
    if (form >= 0)
      rc = launch_resident_adjoint(plan, n_lds, form, resident_lds, k_hi, k_lo, stream);
    else if (n_lds)
      rc = launch_adjoint_bs<false>(plan, plan->use_work, n_lds, lds, k_hi, k_lo, stream);
    if (!rc && n_g) rc = launch_adjoint_bs<true>(plan, plan->use_work + n_lds, n_g, 8, k_hi, k_lo, stream);
  }
  if (rc) return rc;
  return capturing ? JJA_OK : mark_launched(plan, stream);  // nothing has been launched yet
}

int jja_solve(jja_plan* p, int32_t i, const double* b, int64_t ldb, double* x, int64_t ldx, int32_t cols,
              double* zbuf, void* stream_ptr) {
  Plan* plan = reinterpret_cast<Plan*>(p);
  if (!plan || i < 0 || i >= static_cast<int32_t>(plan->problems.size()) || cols < 0 || (cols && (!b || !x)))
    return fail(JJA_EINVAL, "jja_solve: invalid arguments");
  const DevProblem& P = plan->problems[i];
  if (P.parts != 1) return fail(JJA_EUNSUPPORTED, "jja_solve: the plan's columns are split over workgroups");
  if (ldb < P.Nf || ldx < P.Nf) return fail(JJA_EINVAL, "jja_solve: leading dimension below n");
  if (cols == 0 || P.Nf == 0) return JJA_OK;
  const bool global = plan->zbuf_doubles[i] > 0;
  if (global && !zbuf) return fail(JJA_EINVAL, "jja_solve: the problem needs a global face store (zbuf)");
  if (!global && plan->lds_bytes[i] > plan->lds_limit)
    return fail(JJA_EUNSUPPORTED, "jja_solve: the face vector exceeds LDS");
  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  switch (plan->block_size) {
    case 64: return launch_spd_solve<64>(plan, i, b, ldb, x, ldx, cols, zbuf, stream);
    case 128: return launch_spd_solve<128>(plan, i, b, ldb, x, ldx, cols, zbuf, stream);
    case 256: return launch_spd_solve<256>(plan, i, b, ldb, x, ldx, cols, zbuf, stream);
    case 512: return launch_spd_solve<512>(plan, i, b, ldb, x, ldx, cols, zbuf, stream);
    default: return launch_spd_solve<1024>(plan, i, b, ldb, x, ldx, cols, zbuf, stream);
  }
}

int jja_solve_noalloc(jja_plan* p, int32_t i, const double* b, int64_t ldb, double* x, int64_t ldx,
                      int32_t cols, void* stream_ptr) {
  Plan* plan = reinterpret_cast<Plan*>(p);
  if (!plan || i < 0 || i >= static_cast<int32_t>(plan->problems.size()) || cols < 0)
    return fail(JJA_EINVAL, "jja_solve_noalloc: invalid arguments");
  double* zbuf = nullptr;
  if (plan->zbuf_doubles[i] > 0 && cols > 0) {
    const int64_t need = static_cast<int64_t>(cols) * plan->zbuf_doubles[i];
    if (need > kScratchDoubles)
      return fail(JJA_EINVAL, "jja_solve_noalloc: " + std::to_string(cols) + " columns need " + std::to_string(need) +
                                  " doubles of scratch; the limit is " + std::to_string(kScratchDoubles));
    if (int rc = scratch_ptr(plan->device, &zbuf)) return rc;
  }
  return jja_solve(p, i, b, ldb, x, ldx, cols, zbuf, stream_ptr);
}

int jja_vortex(jja_plan* p, int32_t i, const double* theta, int32_t cols, int32_t* n_out,
               void* stream_ptr) {
  Plan* plan = reinterpret_cast<Plan*>(p);
  if (!plan || i < 0 || i >= static_cast<int32_t>(plan->problems.size()) || !theta || !n_out || cols < 0)
    return fail(JJA_EINVAL, "jja_vortex: invalid arguments");
  if (cols == 0 || plan->problems[i].Nf == 0) return JJA_OK;
  hipStream_t stream = static_cast<hipStream_t>(stream_ptr);
  switch (plan->block_size) {
    case 64: return launch_vortex<64>(plan, i, theta, cols, n_out, stream);
    case 128: return launch_vortex<128>(plan, i, theta, cols, n_out, stream);
    case 256: return launch_vortex<256>(plan, i, theta, cols, n_out, stream);
    case 512: return launch_vortex<512>(plan, i, theta, cols, n_out, stream);
    default: return launch_vortex<1024>(plan, i, theta, cols, n_out, stream);
  }
}

}  // extern "C"
