// jja_part_kernels.h -- step kernels of columns worked by several workgroups that
// each keep their own junctions on chip and exchange a few face values once a step.
// What a part holds (PartTables) and the rest of the step are the same for every way
// to solve the face system in parts; the Solver holds the LDS arrays and solves:
//   u    junction values the face sums read, by pair slot: 2 * slot + member
//   in   face sums, written at the faces' addresses
//   out  the solution, read at the junctions' codes and the faces' addresses
// head() issues loads that solve() needs before the face sums. seqs: every part's
// sequence number of its last step; all parts of a column run the same steps, so they
// agree, and each advances its own at the end of a launch.
#ifndef JJA_PART_KERNELS_H
#define JJA_PART_KERNELS_H

#include "jja_device.h"
#include "jja_parts.h"

namespace {

// One face of a part: its sum's codes into the junction values (two to a word, W
// words), where the sum goes and the face's index (-1: its flux is another part's).
template <int W>
struct PartFace {
  uint32_t code[W], at;
  int32_t id;
};

template <int W>
__device__ __forceinline__ PartFace<W> part_face(const PartTables& T, int32_t part, int32_t slot) {
  // loaded without a branch (a slot past the last reads the last), so that the loads of
  // all slots are in flight together
  PartFace<W> f;
  const int64_t at = static_cast<int64_t>(part) * T.faces + min(slot, T.faces - 1);
#pragma unroll
  for (int i = 0; i < W; i += 2) {
    const vuint2 c = gbl(reinterpret_cast<const vuint2*>(T.face_code + W * at + i))[0];
    f.code[i] = c.x;
    f.code[i + 1] = c.y;
  }
  f.at = gbl(T.face_at)[at];
  f.id = gbl(T.face_id)[at];
  if (slot >= T.faces) {
    f.at = 0xffffffffu;
    f.id = -1;
  }
  return f;
}

template <int W>
__device__ __forceinline__ double face_sum(const PartFace<W>& f, const LAS double* U) {
  double uv[2 * W], acc = 0.0;
#pragma unroll
  for (int i = 0; i < 2 * W; ++i) uv[i] = U[code_address((f.code[i >> 1] >> (16 * (i & 1))) & 0xffffu)];
#pragma unroll
  for (int i = 0; i < 2 * W; ++i) acc = acc + signed_value(uv[i], (f.code[i >> 1] >> (16 * (i & 1))) & 0xffffu);
  return acc;
}

// NP: junction pairs a thread holds in registers (phases and right-hand sides; with
// few pairs also their constant inputs).
template <class Solver, int NP>
__global__ __launch_bounds__(kPartBlock) void evolve_parts_kernel(const DevProblem* __restrict__ probs,
                                                         const jja_problem_run* __restrict__ runs,
                                                         const WorkItem* __restrict__ work,
                                                         const typename Solver::Dev* __restrict__ tables, int32_t n_steps,
                                                         int64_t step0, uint32_t* seqs, int32_t* err,
                                                         uint32_t wait_limit) {
  extern __shared__ double lds[];
  constexpr int BS = kPartBlock, FW = Solver::kFaceWords;
  constexpr bool KEEP = NP <= 2;
  constexpr int NF = NP;
  WorkItem wi = work[blockIdx.x];
  wi.problem = __builtin_amdgcn_readfirstlane(wi.problem);
  wi.column = __builtin_amdgcn_readfirstlane(wi.column);
  const DevProblem& P = probs[wi.problem];
  const jja_problem_run& R = runs[wi.problem];
  const typename Solver::Dev& S = tables[wi.problem];
  const int64_t w = wi.column / S.parts;
  const int32_t tid0 = threadIdx.x, tid = tid0;
  const int32_t part = wi.column % S.parts;
  const uint32_t seq0 = __builtin_amdgcn_readfirstlane(gbl(seqs)[wi.column]);  // before the solver's barrier
  const Solver solver(P, S, w, part, lds, err, wait_limit, tid, BS);
  LAS double *const U = solver.u, *const face_in = solver.in, *const face_out = solver.out;
  const int32_t Nj = P.Nj;
  const size_t stride = static_cast<size_t>(R.W) * Nj, col = static_cast<size_t>(w) * Nj;
  GAS double* const even = gblw(R.theta) + col;  // phases of even and odd steps
  GAS double* const odd = even + stride;
  const uint32_t noise_col = static_cast<uint32_t>(R.column_offset + w);
  const GAS double* Icp = gbl(R.Ic ? R.Ic : P.Ic);
  const bool gauss = !R.T.zero, is_zero = R.Is.zero;
  const bool uni = P.coef_si == 0;
  double rc0 = 0.0, c1 = 0.0, c2 = 0.0;
  if (uni) {
    rc0 = rc0_at(P, 0);
    c1 = coef_at(P, 1, 0);
    c2 = coef_at(P, 2, 0);
  }
  const bool keep_is = KEEP && R.Is.s_t == 0;
  const GAS double* const th1 = (step0 & 1) ? even : odd;   // theta_{step0-1}
  const GAS double* const th2 = (step0 & 1) ? odd : even;   // theta_{step0-2}

  // pair slot k*BS + tid; pe: pair * 16 + present bits + 4 * owner bits
  const GAS int32_t* list = gbl(S.pair) + static_cast<int64_t>(part) * S.pairs;
  const GAS uint32_t* codes = gbl(S.pair_code) + static_cast<int64_t>(part) * S.pairs * 2;
  double x[NP][2], tp[NP][2], ic[KEEP ? NP : 1][2], is[KEEP ? NP : 1][2];
  int32_t pe[NP];
  uint32_t jc[KEEP ? NP : 1][2];
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    const int32_t slot = k * BS + tid;
    pe[k] = slot < S.pairs ? max(list[slot], 0) : 0;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int32_t j = min(2 * (pe[k] >> 4) + m, Nj - 1);
      tp[k][m] = th1[j];
      x[k][m] = th2[j];
      if constexpr (KEEP) {
        jc[k][m] = pe[k] ? codes[2 * slot + m] : 0xffffffffu;
        ic[k][m] = Icp[j];
        is[k][m] = gbl(R.Is.base)[w * R.Is.s_w + j * R.Is.s_i];
      }
    }
  }
  PartFace<FW> face[NF];
  double fx[NF];
  const bool keep_f = KEEP && R.f.s_t == 0;
  if constexpr (KEEP) {
    const TermView fv = term_view(R.f, !R.f.zero, P.zero, w, R.f.t0);
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      face[k] = part_face<FW>(S, part, k * BS + tid);
      fx[k] = face[k].id >= 0 ? fv.p[face[k].id * fv.si] : 0.0;
    }
  }

  // x of step t from theta_{t-1} = a and theta_{t-2} = c, and u for the face sums
  auto prepare = [&](int slot, int m, int32_t j, double a, double c, double icj, double isj, double sg, double z) {
    double r0 = rc0, k1 = c1, k2 = c2;
    if (!uni) {
      r0 = rc0_at(P, j);
      k1 = coef_at(P, 1, j);
      k2 = coef_at(P, 2, j);
    }
    const double X = icj * cpr_sum(P, 2.0 * a - c) + k1 * a + k2 * c;
    double eta = 0.0;
    if (gauss) eta = sg * z;
    const double xn = is_zero ? eta + X : (eta - isj) + X;
    U[2 * slot + m] = xn * r0;
    return xn;
  };
  {
    const TermView isv = term_view(R.Is, true, P.zero, w, step0);
    const TermView sgv = term_view(R.sigma, gauss, P.zero, w, step0);
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      if (!pe[k]) continue;
      const int32_t q = pe[k] >> 4;
      double z[2] = {0.0, 0.0};
      if (gauss)
        normal_pair(R.seed, static_cast<uint32_t>(2 * q), noise_col, static_cast<uint64_t>(step0), &z[0], &z[1]);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int32_t j = min(2 * q + m, Nj - 1);
        x[k][m] = prepare(k * BS + tid, m, j, tp[k][m], x[k][m], Icp[j], term_at(isv, j), term_at(sgv, j), z[m]);
      }
    }
  }
  for (int32_t n = 0; n < n_steps; ++n) {
    const int64_t t = step0 + n;
    const int32_t again = wi.problem + opaque_zero();
    const DevProblem& P = probs[again];
    const jja_problem_run& R = runs[again];
    const typename Solver::Dev& S = tables[again];
    const int32_t tid = opaque(tid0);
    {
      const TermView fv = term_view(R.f, !R.f.zero, P.zero, w, t);
      double fq[NF];
#pragma unroll
      for (int k = 0; k < NF; ++k) {
        if constexpr (!KEEP) face[k] = part_face<FW>(S, part, k * BS + tid);
        fq[k] = KEEP ? fx[k] * fv.amp : 0.0;
        if (!keep_f) fq[k] = term_at(fv, max(face[k].id, 0));  // used by faces that have one
      }
      typename Solver::Head head;
      solver.head(S, tid, head);
      lds_barrier();
#pragma unroll
      for (int k = 0; k < NF; ++k)
        if (face[k].at != 0xffffffffu)
          face_in[face[k].at] = face_sum(face[k], U) - (face[k].id >= 0 ? kTwoPi * fq[k] : 0.0);
      lds_barrier();
      solver.solve(P, S, seq0 + 1u + static_cast<uint32_t>(n), tid, BS, head);
    }
    // finish step t, prepare step t + 1
    const bool prep = n + 1 < n_steps;
    const int32_t tho = R.th_slot ? gbl(R.th_slot)[t - R.slot_t0] : -1;
    const int32_t Io = R.I_slot ? gbl(R.I_slot)[t - R.slot_t0] : -1;
    GAS double* th_out = tho >= 0 ? gblw(R.th_out) + static_cast<size_t>(tho) * stride + col : nullptr;
    GAS double* I_out = Io >= 0 ? gblw(R.I_out) + static_cast<size_t>(Io) * stride + col : nullptr;
    const TermView ist = term_view(R.Is, true, P.zero, w, t);
    const TermView isn = term_view(R.Is, prep, P.zero, w, t + 1);
    const TermView sgn = term_view(R.sigma, gauss && prep, P.zero, w, t + 1);
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      if (pe[k]) {
        const int32_t q = pe[k] >> 4, slot = k * BS + tid;
        double icj[2], isj[2], sg[2], z[2] = {0.0, 0.0};
        uint32_t code[2];
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const int32_t j = min(2 * q + m, Nj - 1);
          if constexpr (KEEP) {
            code[m] = jc[k][m];
            icj[m] = ic[k][m];
            isj[m] = keep_is ? is[k][m] * isn.amp : term_at(isn, j);
          } else {
            code[m] = codes[2 * slot + m];
            icj[m] = Icp[j];
            isj[m] = term_at(isn, j);
          }
          sg[m] = term_at(sgn, j);
        }
        if (gauss && prep)
          normal_pair(R.seed, static_cast<uint32_t>(2 * q), noise_col, static_cast<uint64_t>(t + 1), &z[0], &z[1]);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const int32_t j = min(2 * q + m, Nj - 1);
          const uint32_t ca = code[m] & 0xffffu, cb = code[m] >> 16;
          const double za = face_out[code_address(ca)], zb = face_out[code_address(cb)];
          const double y = signed_value(za, ca) + signed_value(zb, cb);
          const double t0 = (y - x[k][m]) * (uni ? rc0 : rc0_at(P, j));
          const bool owner = (pe[k] >> (2 + m)) & 1;
          if (owner && th_out) th_out[j] = t0;
          if (owner && I_out) I_out[j] = y + term_at(ist, j);
          if (prep) {
            x[k][m] = prepare(slot, m, j, t0, tp[k][m], icj[m], isj[m], sg[m], z[m]);
          } else if (owner) {
            // the launch's last step: theta_{t-1} and theta_t to the history ring
            ((t & 1) ? even : odd)[j] = tp[k][m];
            ((t & 1) ? odd : even)[j] = t0;
          }
          tp[k][m] = t0;
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if (threadIdx.x == 0) gblw(seqs)[wi.column] = seq0 + static_cast<uint32_t>(n_steps);
}

// The adjoint sweep (adjoint_steps) of a part: with few pairs a thread keeps
// lambda_k, the partial sum of lambda_{k-1}, both gradients and the phases of two
// steps of its junctions in registers for the whole launch; with more, lambda alone.
template <class Solver, int NP>
__global__ __launch_bounds__(kPartBlock) void adjoint_parts_kernel(const DevProblem* __restrict__ probs,
                                                          const jja_adjoint_run* __restrict__ runs,
                                                          const WorkItem* __restrict__ work,
                                                          const typename Solver::Dev* __restrict__ tables, int64_t k_hi, int64_t k_lo,
                                                          uint32_t* seqs, int32_t* err, uint32_t wait_limit) {
  extern __shared__ double lds[];
  constexpr int BS = kPartBlock, FW = Solver::kFaceWords;
  constexpr bool KEEP = NP <= 2;
  constexpr int NF = NP, N = KEEP ? NP : 1, K = KEEP ? NF : 1;
  WorkItem wi = work[blockIdx.x];
  wi.problem = __builtin_amdgcn_readfirstlane(wi.problem);
  wi.column = __builtin_amdgcn_readfirstlane(wi.column);
  const DevProblem& P = probs[wi.problem];
  const jja_adjoint_run& A = runs[wi.problem];
  const typename Solver::Dev& S = tables[wi.problem];
  const int64_t w = wi.column / S.parts;
  const int32_t tid0 = threadIdx.x, tid = tid0;
  const int32_t part = wi.column % S.parts;
  const uint32_t seq0 = __builtin_amdgcn_readfirstlane(gbl(seqs)[wi.column]);  // before the solver's barrier
  const Solver solver(P, S, w, part, lds, err, wait_limit, tid, BS);
  LAS double *const U = solver.u, *const face_in = solver.in, *const face_out = solver.out;
  const int32_t Nj = P.Nj;
  const AdjCol C = adjoint_column(P, A, w);
  GAS double* const gIc = gblw(A.grad_Ic) + static_cast<size_t>(w) * Nj;
  GAS double* const gIs = gblw(A.grad_Is) + static_cast<size_t>(w) * Nj;
  GAS double* const gf = gblw(A.grad_f) + static_cast<size_t>(w) * P.Nf;
  // solve position of a face of this part whose gradient it adds, or -1
  auto position = [&](int32_t slot) {
    return slot < S.faces ? gbl(S.face_pos)[static_cast<int64_t>(part) * S.faces + slot] : -1;
  };
  const bool uni = P.coef_si == 0;
  double rc0 = 0.0, c1 = 0.0, c2 = 0.0;
  if (uni) {
    rc0 = rc0_at(P, 0);
    c1 = coef_at(P, 1, 0);
    c2 = coef_at(P, 2, 0);
  }
  auto history = [&](int64_t m, int32_t j) { return C.hist[static_cast<size_t>(m - C.hist_m0) * C.stride + j]; };
  const GAS int32_t* list = gbl(S.pair) + static_cast<int64_t>(part) * S.pairs;
  const GAS uint32_t* codes = gbl(S.pair_code) + static_cast<int64_t>(part) * S.pairs * 2;
  double la[NP][2], lb[NP][2], ic[N][2], ai[N][2], as[N][2], h1[N][2], h2[N][2];
  int32_t pe[NP];
  uint32_t jc[N][2];
#pragma unroll
  for (int k = 0; k < NP; ++k) {
    const int32_t slot = k * BS + tid;
    pe[k] = slot < S.pairs ? max(list[slot], 0) : 0;
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int32_t j = min(2 * (pe[k] >> 4) + m, Nj - 1);
      la[k][m] = (C.lam + (k_hi & 1) * C.stride)[j];
      if (A.prime) la[k][m] = la[k][m] + adj_g(A, C, k_hi, j);
      lb[k][m] = (C.lam + ((k_hi - 1) & 1) * C.stride)[j];
      if constexpr (KEEP) {
        jc[k][m] = pe[k] ? codes[2 * slot + m] : 0xffffffffu;
        ic[k][m] = C.Ic[j];
        ai[k][m] = gIc[j];
        as[k][m] = gIs[j];
        h1[k][m] = history(k_hi - 1, j);
        h2[k][m] = history(k_hi - 2, j);
      }
      if (pe[k]) U[2 * slot + m] = la[k][m] * (uni ? rc0 : rc0_at(P, j));
    }
  }
  PartFace<FW> face[K];
  double af[K];
  int32_t fp[K];
  if constexpr (KEEP) {
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      face[k] = part_face<FW>(S, part, k * BS + tid);
      fp[k] = position(k * BS + tid);
      af[k] = fp[k] >= 0 ? gf[fp[k]] : 0.0;
    }
  }
  for (int64_t t = k_hi; t >= k_lo; --t) {
    const int32_t again = wi.problem + opaque_zero();
    const DevProblem& P = probs[again];
    const jja_adjoint_run& A = runs[again];
    const typename Solver::Dev& S = tables[again];
    const int32_t tid = opaque(tid0);
    typename Solver::Head head;
    solver.head(S, tid, head);
    lds_barrier();
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      const PartFace<FW> f = KEEP ? face[KEEP ? k : 0] : part_face<FW>(S, part, k * BS + tid);
      if (f.at != 0xffffffffu) face_in[f.at] = face_sum(f, U);
    }
    lds_barrier();
    solver.solve(P, S, seq0 + 1u + static_cast<uint32_t>(k_hi - t), tid, BS, head);
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      if constexpr (KEEP) {
        if (fp[k] >= 0) af[k] = af[k] - kTwoPi * face_out[face[k].at];
      } else {
        const int32_t p = position(k * BS + tid);
        if (p >= 0) gf[p] = gf[p] - kTwoPi * face_out[part_face<FW>(S, part, k * BS + tid).at];
      }
    }
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      if (pe[k]) {
        const int32_t q = pe[k] >> 4, slot = k * BS + tid;
        double nh[2] = {0.0, 0.0};
        if (KEEP && t > k_lo) {
#pragma unroll
          for (int m = 0; m < 2; ++m) nh[m] = history(t - 3, min(2 * q + m, Nj - 1));
        }
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const int32_t j = min(2 * q + m, Nj - 1);
          double r0 = rc0, k1 = c1, k2 = c2, t1, t2, icj, gi, gs;
          uint32_t code;
          if (!uni) {
            r0 = rc0_at(P, j);
            k1 = coef_at(P, 1, j);
            k2 = coef_at(P, 2, j);
          }
          if constexpr (KEEP) {
            code = jc[k][m];
            icj = ic[k][m];
            gi = ai[k][m];
            gs = as[k][m];
            t1 = h1[k][m];
            t2 = h2[k][m];
          } else {
            code = codes[2 * slot + m];
            icj = C.Ic[j];
            gi = gIc[j];
            gs = gIs[j];
            t1 = history(t - 1, j);
            t2 = history(t - 2, j);
          }
          const double gj = adj_g(A, C, t - 1, j);
          const uint32_t ca = code & 0xffffu, cb = code >> 16;
          const double za = face_out[code_address(ca)], zb = face_out[code_address(cb)];
          const double y = signed_value(za, ca) + signed_value(zb, cb);
          const double mu = (y - la[k][m]) * r0;
          double sn, cs;
          jja_sincos(2.0 * t1 - t2, &sn, &cs);
          const double av = 2.0 * icj * cs + k1, bv = k2 - icj * cs;
          const double l1 = (lb[k][m] + av * mu) + gj;
          lb[k][m] = bv * mu;
          la[k][m] = l1;
          U[2 * slot + m] = l1 * r0;
          const bool owner = (pe[k] >> (2 + m)) & 1;
          if constexpr (KEEP) {
            ai[k][m] = gi + sn * mu;
            as[k][m] = gs - mu;
            h1[k][m] = t2;
            h2[k][m] = nh[m];
          } else if (owner) {
            gIc[j] = gi + sn * mu;
            gIs[j] = gs - mu;
          }
          if (t == k_lo && owner) {
            // lambda_{k_lo - 1} complete, the partial sum of lambda_{k_lo - 2}
            (C.lam + ((k_lo - 1) & 1) * C.stride)[j] = l1;
            (C.lam + (k_lo & 1) * C.stride)[j] = lb[k][m];
            C.u[j] = l1 * r0;
            if constexpr (KEEP) {
              gIc[j] = ai[k][m];
              gIs[j] = as[k][m];
            }
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  if constexpr (KEEP) {
#pragma unroll
    for (int k = 0; k < NF; ++k)
      if (fp[k] >= 0) gf[fp[k]] = af[k];
  }
  if (threadIdx.x == 0) gblw(seqs)[wi.column] = seq0 + static_cast<uint32_t>(k_hi - k_lo + 1);
}

}  // namespace

#endif  // JJA_PART_KERNELS_H
