// Step kernels of columns small enough that one workgroup holds their whole
// state: each thread keeps the phases and right-hand sides of its junction
// pairs in registers for all steps of a launch, the junction values the face
// phase sums lie in LDS beside the face vector, and the codes of both
// incidence products are read once per launch.
//
// What bounds a small column is latency: with the state in global memory each
// step waits for a write of u, the face records, their codes, the gathers of u
// and the junction pass's own loads in turn, five to seven round trips of about
// a microsecond. Here a step touches LDS only (and global memory for stored
// steps and for inputs that vary in time). Measured with the padded lattice solve,
// us a step: 12x9, 64 columns 9.9 before, 4.7 (with one wave's solve 3.5 now); 37x53, 96
// columns 23.0 before, 13.4 now.
#include "jja_resident.h"

#include "jja_device.h"

namespace {

// NP > 0: every thread keeps NP junction pairs in registers. NP 0: phases and
// right-hand sides lie in LDS and the threads loop over the pairs.
template <int BS, int NP>
__global__ __launch_bounds__(BS) void evolve_resident_kernel(const DevProblem* __restrict__ probs,
                                                             const jja_problem_run* __restrict__ runs,
                                                             const WorkItem* __restrict__ work, int32_t n_steps,
                                                             int64_t step0) {
  extern __shared__ double lds[];
  constexpr bool REG = NP > 0;
  constexpr int N = REG ? NP : 1;
  constexpr int NF = REG ? kResidentFaces * NP : kResidentRecords;
  const int32_t problem = __builtin_amdgcn_readfirstlane(work[blockIdx.x].problem);
  const int64_t w = __builtin_amdgcn_readfirstlane(work[blockIdx.x].column);
  const DevProblem& P = probs[problem];
  const jja_problem_run& R = runs[problem];
  const int32_t tid0 = threadIdx.x, tid = tid0;
  const int32_t Nj = P.Nj, Nf = P.Nf, pairs = (Nj + 1) >> 1;
  FaceStore<false> zs;
  zs.p = lds;
  zs.vt = tid;
  zs.vbs = BS;
  init_store(P, lds, tid, BS);
  // after the face vector and its scratch: u when every 1/c0 is its own (else
  // the face phase forms x * 1/c0), x and theta_{t-1} of the LDS form
  LAS double* const base = (LAS double*)lds + P.store_doubles;
  const bool uni = P.coef_si == 0;
  LAS double* const X = base;
  LAS double* const TP = X + 2 * pairs;
  LAS double* const U = REG ? base : (uni ? X : TP + 2 * pairs);
  const size_t stride = static_cast<size_t>(R.W) * Nj, col = static_cast<size_t>(w) * Nj;
  GAS double* th = gblw(R.theta) + col;
  GAS double* const even = th;          // phases of even and odd steps
  GAS double* const odd = th + stride;
  const uint32_t noise_col = static_cast<uint32_t>(R.column_offset + w);
  const GAS double* Icp = gbl(R.Ic ? R.Ic : P.Ic);
  const bool gauss = !R.T.zero, is_zero = R.Is.zero;
  double rc0 = 0.0, c1 = 0.0, c2 = 0.0;
  if (uni) {
    rc0 = rc0_at(P, 0);
    c1 = coef_at(P, 1, 0);
    c2 = coef_at(P, 2, 0);
  }
  const bool keep_is = REG && R.Is.s_t == 0, keep_f = R.f.s_t == 0;

  // junction pairs (2q, 2q+1), q = k*BS + tid
  double x[N][2], tp[N][2], ic[N][2], is[N][2];
  uint32_t jc[N][2];
  const GAS double* const th1 = (step0 & 1) ? even : odd;   // theta_{step0-1}
  const GAS double* const th2 = (step0 & 1) ? odd : even;   // theta_{step0-2}
  if constexpr (REG) {
#pragma unroll
    for (int k = 0; k < N; ++k)
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int32_t j = min(2 * (k * BS + tid) + m, Nj - 1);
        const vint2 c = gbl(reinterpret_cast<const vint2*>(P.junc_code))[j];
        jc[k][m] = pack_codes(c.x, c.y);
        tp[k][m] = th1[j];
        x[k][m] = th2[j];
        ic[k][m] = Icp[j];
        is[k][m] = R.Is.base ? gbl(R.Is.base)[w * R.Is.s_w + j * R.Is.s_i] : 0.0;
      }
  }
  // face records: codes of u, the position written and the face's flux
  uint32_t fc[NF][2], fpos[NF], finish = 0;
  int32_t ffid[NF];
  double fx[NF];
  const int32_t nrec = P.n_face_slices;
#pragma unroll
  for (int k = 0; k < NF; ++k) {
    // past the last record (a circuit without faces has none, and no list)
    FaceRec r{{-1, -1, -1, -1}, -1, -1, false};
    if (k < nrec) face_rec_load(P, k, true, tid, BS, r);
    fc[k][0] = pack_codes(r.cd[0], r.cd[1]);
    fc[k][1] = pack_codes(r.cd[2], r.cd[3]);
    fpos[k] = r.pos < 0 ? 0xffffffffu : static_cast<uint32_t>(r.pos);
    finish |= r.finish ? 1u << k : 0u;
    ffid[k] = r.fid;
    const TermView fv = term_view(R.f, !R.f.zero, P.zero, w, R.f.t0);
    fx[k] = r.fid >= 0 ? fv.p[r.fid * fv.si] : 0.0;
  }

  // x of step t from theta_{t-1} = a and theta_{t-2} = b, and u for the face phase
  auto prepare = [&](int32_t j, double a, double b, double icj, double isj, double sg, double z) {
    double r0 = rc0, k1 = c1, k2 = c2;
    if (!uni) {
      r0 = rc0_at(P, j);
      k1 = coef_at(P, 1, j);
      k2 = coef_at(P, 2, j);
    }
    const double S = icj * cpr_sum(P, 2.0 * a - b) + k1 * a + k2 * b;
    double eta = 0.0;
    if (gauss) eta = sg * z;
    const double xn = is_zero ? eta + S : (eta - isj) + S;
    if constexpr (REG) {
      U[j] = xn * r0;
    } else {
      X[j] = xn;
      if (!uni) U[j] = xn * r0;
    }
    return xn;
  };
  auto first = [&](int k, int32_t q) {
    const TermView isv = term_view(R.Is, true, P.zero, w, step0);
    const TermView sgv = term_view(R.sigma, gauss, P.zero, w, step0);
    double z[2] = {0.0, 0.0};
    if (gauss)
      normal_pair(R.seed, static_cast<uint32_t>(2 * q), noise_col, static_cast<uint64_t>(step0), &z[0], &z[1]);
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int32_t j = 2 * q + m;
      if (j >= Nj) break;
      const double a = REG ? tp[k][m] : th1[j], b = REG ? x[k][m] : th2[j];
      const double xn = prepare(j, a, b, Icp[j], term_at(isv, j), term_at(sgv, j), z[m]);
      if constexpr (REG)
        x[k][m] = xn;
      else
        TP[j] = a;
    }
  };
  if constexpr (REG) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      if (k * BS + tid < pairs) first(k, k * BS + tid);
  } else {
    for (int32_t q = tid; q < pairs; q += BS) first(0, q);
  }
  for (int32_t n = 0; n < n_steps; ++n) {
    const int64_t t = step0 + n;
    const int32_t again = problem + opaque_zero();
    const DevProblem& P = probs[again];
    const jja_problem_run& R = runs[again];
    const int32_t tid = opaque(tid0);
    zs.vt = tid;
    if (Nf > 0) {
      const TermView fv = term_view(R.f, !R.f.zero, P.zero, w, t);
      double fq[NF];
#pragma unroll
      for (int k = 0; k < NF; ++k) {
        fq[k] = fx[k] * fv.amp;
        if (!keep_f) fq[k] = ffid[k] >= 0 ? term_at(fv, ffid[k]) : 0.0;
      }
      lds_barrier();
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < NF; ++k) {
        if (k >= nrec) break;
        double uv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) uv[i] = U[code_address((fc[k][i >> 1] >> (16 * (i & 1))) & 0xffffu)];
        if (!REG && uni) {
#pragma unroll
          for (int i = 0; i < 4; ++i) uv[i] = uv[i] * rc0;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = acc + signed_value(uv[i], (fc[k][i >> 1] >> (16 * (i & 1))) & 0xffffu);
        if (finish >> k & 1u) {
          if (fpos[k] != 0xffffffffu) {
            const int32_t pos = static_cast<int32_t>(fpos[k]);
            acc = acc - kTwoPi * fq[k];
            zs.wr(pos, acc);
            if (pos < P.copy_rows) zs.wr(Nf + pos, acc);
          }
          acc = 0.0;
        }
      }
      lds_barrier();
      solve_face_system(P, zs);
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
    auto finish_pair = [&](int k, int32_t q) {
      // the loads of both junctions first, then the pair's Philox draw
      double xo[2], tm[2], icj[2], isj[2], sg[2], z[2] = {0.0, 0.0};
      uint32_t code[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int32_t j = min(2 * q + m, Nj - 1);
        if constexpr (REG) {
          xo[m] = x[k][m];
          tm[m] = tp[k][m];
          code[m] = jc[k][m];
          icj[m] = ic[k][m];
          isj[m] = keep_is ? is[k][m] * isn.amp : term_at(isn, j);
        } else {
          const vint2 c = gbl(reinterpret_cast<const vint2*>(P.junc_code))[j];
          code[m] = pack_codes(c.x, c.y);
          icj[m] = Icp[j];
          isj[m] = term_at(isn, j);
          xo[m] = X[j];
          tm[m] = TP[j];
        }
        sg[m] = term_at(sgn, j);
      }
      if (gauss && prep)
        normal_pair(R.seed, static_cast<uint32_t>(2 * q), noise_col, static_cast<uint64_t>(t + 1), &z[0], &z[1]);
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int32_t j = 2 * q + m;
        if (j >= Nj) break;
        const uint32_t ca = code[m] & 0xffffu, cb = code[m] >> 16;
        const double za = zs.gather(code_address(ca)), zb = zs.gather(code_address(cb));
        const double y = signed_value(za, ca) + signed_value(zb, cb);
        const double t0 = (y - xo[m]) * (uni ? rc0 : rc0_at(P, j));
        if (th_out) th_out[j] = t0;
        if (I_out) I_out[j] = y + term_at(ist, j);
        if (prep) {
          const double xn = prepare(j, t0, tm[m], icj[m], isj[m], sg[m], z[m]);
          if constexpr (REG) {
            x[k][m] = xn;
            tp[k][m] = t0;
          } else {
            TP[j] = t0;
          }
        } else {
          // the launch's last step: theta_{t-1} and theta_t to the history ring
          ((t & 1) ? even : odd)[j] = tm[m];
          ((t & 1) ? odd : even)[j] = t0;
        }
      }
    };
    if constexpr (REG) {
#pragma unroll
      for (int k = 0; k < N; ++k) {
        if (k * BS + tid < pairs) finish_pair(k, k * BS + tid);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      for (int32_t q = tid; q < pairs; q += BS) finish_pair(0, q);
    }
  }
}

// The adjoint sweep (adjoint_steps) of a column. NP > 0: lambda_k, the partial sum
// of lambda_{k-1}, both gradients and the phases of two steps stay in registers for
// the whole launch; NP 0: both lambdas lie in LDS.
template <int BS, int NP>
__global__ __launch_bounds__(BS) void adjoint_resident_kernel(const DevProblem* __restrict__ probs,
                                                              const jja_adjoint_run* __restrict__ runs,
                                                              const WorkItem* __restrict__ work, int64_t k_hi,
                                                              int64_t k_lo) {
  extern __shared__ double lds[];
  constexpr bool REG = NP > 0;
  constexpr int N = REG ? NP : 1;
  constexpr int NF = REG ? kResidentFaces * NP : kResidentRecords;
  const int32_t problem = __builtin_amdgcn_readfirstlane(work[blockIdx.x].problem);
  const int64_t w = __builtin_amdgcn_readfirstlane(work[blockIdx.x].column);
  const DevProblem& P = probs[problem];
  const jja_adjoint_run& A = runs[problem];
  const int32_t tid0 = threadIdx.x, tid = tid0;
  const int32_t Nj = P.Nj, Nf = P.Nf, pairs = (Nj + 1) >> 1;
  FaceStore<false> zs;
  zs.p = lds;
  zs.vt = tid;
  zs.vbs = BS;
  init_store(P, lds, tid, BS);
  const bool uni = P.coef_si == 0;
  LAS double* const X = (LAS double*)lds + P.store_doubles;   // lambda_k, then the partial sum
  LAS double* const B = X + 2 * pairs;
  LAS double* const U = REG || uni ? X : B + 2 * pairs;
  const AdjCol C = adjoint_column(P, A, w);
  GAS double* const gIc = gblw(A.grad_Ic) + static_cast<size_t>(w) * Nj;
  GAS double* const gIs = gblw(A.grad_Is) + static_cast<size_t>(w) * Nj;
  GAS double* const gf = gblw(A.grad_f) + static_cast<size_t>(w) * Nf;
  double rc0 = 0.0, c1 = 0.0, c2 = 0.0;
  if (uni) {
    rc0 = rc0_at(P, 0);
    c1 = coef_at(P, 1, 0);
    c2 = coef_at(P, 2, 0);
  }
  auto history = [&](int64_t m, int32_t j) { return C.hist[static_cast<size_t>(m - C.hist_m0) * C.stride + j]; };
  const GAS double* const lam_k = C.lam + (k_hi & 1) * C.stride;
  const GAS double* const lam_p = C.lam + ((k_hi - 1) & 1) * C.stride;
  double la[N][2], lb[N][2], ic[N][2], ai[N][2], as[N][2], h1[N][2], h2[N][2];
  uint32_t jc[N][2];
  auto begin = [&](int k, int32_t q) {
#pragma unroll
    for (int m = 0; m < 2; ++m) {
      const int32_t j = 2 * q + m;
      if (j >= Nj) break;
      double l = lam_k[j];
      if (A.prime) l = l + adj_g(A, C, k_hi, j);
      const double u = l * (uni ? rc0 : rc0_at(P, j));
      if constexpr (REG) {
        const vint2 c = gbl(reinterpret_cast<const vint2*>(P.junc_code))[j];
        jc[k][m] = pack_codes(c.x, c.y);
        la[k][m] = l;
        lb[k][m] = lam_p[j];
        ic[k][m] = C.Ic[j];
        ai[k][m] = gIc[j];
        as[k][m] = gIs[j];
        h1[k][m] = history(k_hi - 1, j);
        h2[k][m] = history(k_hi - 2, j);
        U[j] = u;
      } else {
        X[j] = l;
        B[j] = lam_p[j];
        if (!uni) U[j] = u;
      }
    }
  };
  if constexpr (REG) {
#pragma unroll
    for (int k = 0; k < N; ++k)
      if (k * BS + tid < pairs) begin(k, k * BS + tid);
  } else {
    for (int32_t q = tid; q < pairs; q += BS) begin(0, q);
  }
  uint32_t fc[NF][2], fpos[NF], finish = 0;
  const int32_t nrec = P.n_face_slices;
#pragma unroll
  for (int k = 0; k < NF; ++k) {
    FaceRec r{{-1, -1, -1, -1}, -1, -1, false};
    if (k < nrec) face_rec_load(P, k, true, tid, BS, r);
    fc[k][0] = pack_codes(r.cd[0], r.cd[1]);
    fc[k][1] = pack_codes(r.cd[2], r.cd[3]);
    fpos[k] = r.pos < 0 ? 0xffffffffu : static_cast<uint32_t>(r.pos);
    finish |= r.finish ? 1u << k : 0u;
  }
  for (int64_t t = k_hi; t >= k_lo; --t) {
    const int32_t again = problem + opaque_zero();
    const DevProblem& P = probs[again];
    const jja_adjoint_run& A = runs[again];
    const int32_t tid = opaque(tid0);
    zs.vt = tid;
    if (Nf > 0) {
      lds_barrier();
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < NF; ++k) {
        if (k >= nrec) break;
        double uv[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) uv[i] = U[code_address((fc[k][i >> 1] >> (16 * (i & 1))) & 0xffffu)];
        if (!REG && uni) {
#pragma unroll
          for (int i = 0; i < 4; ++i) uv[i] = uv[i] * rc0;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) acc = acc + signed_value(uv[i], (fc[k][i >> 1] >> (16 * (i & 1))) & 0xffffu);
        if (finish >> k & 1u) {
          if (fpos[k] != 0xffffffffu) {
            const int32_t pos = static_cast<int32_t>(fpos[k]);
            zs.wr(pos, acc);
            if (pos < P.copy_rows) zs.wr(Nf + pos, acc);
          }
          acc = 0.0;
        }
      }
      lds_barrier();
      solve_face_system(P, zs);
      for (int32_t p = tid; p < Nf; p += BS) gf[p] = gf[p] - kTwoPi * zs.rd(store_address(P, p));
    }
    auto sweep = [&](int k, int32_t q) {
      double t1[2], t2[2], nh[2] = {0.0, 0.0}, icj[2], gi[2], gs[2], lk[2], lp[2];
      uint32_t code[2];
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int32_t j = min(2 * q + m, Nj - 1);
        if constexpr (REG) {
          code[m] = jc[k][m];
          t1[m] = h1[k][m];
          t2[m] = h2[k][m];
          icj[m] = ic[k][m];
          gi[m] = ai[k][m];
          gs[m] = as[k][m];
          lk[m] = la[k][m];
          lp[m] = lb[k][m];
          if (t > k_lo) nh[m] = history(t - 3, j);
        } else {
          const vint2 c = gbl(reinterpret_cast<const vint2*>(P.junc_code))[j];
          code[m] = pack_codes(c.x, c.y);
          t1[m] = history(t - 1, j);
          t2[m] = history(t - 2, j);
          icj[m] = C.Ic[j];
          gi[m] = gIc[j];
          gs[m] = gIs[j];
          lk[m] = X[j];
          lp[m] = B[j];
        }
      }
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const int32_t j = 2 * q + m;
        if (j >= Nj) break;
        double r0 = rc0, k1 = c1, k2 = c2;
        if (!uni) {
          r0 = rc0_at(P, j);
          k1 = coef_at(P, 1, j);
          k2 = coef_at(P, 2, j);
        }
        const double gj = adj_g(A, C, t - 1, j);
        const uint32_t ca = code[m] & 0xffffu, cb = code[m] >> 16;
        const double za = zs.gather(code_address(ca)), zb = zs.gather(code_address(cb));
        const double y = signed_value(za, ca) + signed_value(zb, cb);
        const double mu = (y - lk[m]) * r0;
        double sn, cs;
        jja_sincos(2.0 * t1[m] - t2[m], &sn, &cs);
        const double av = 2.0 * icj[m] * cs + k1, bv = k2 - icj[m] * cs;
        const double gn = gi[m] + sn * mu, sm = gs[m] - mu, part = bv * mu;
        const double l1 = (lp[m] + av * mu) + gj;
        if constexpr (REG) {
          la[k][m] = l1;
          lb[k][m] = part;
          ai[k][m] = gn;
          as[k][m] = sm;
          h1[k][m] = t2[m];
          h2[k][m] = nh[m];
          U[j] = l1 * r0;
        } else {
          X[j] = l1;
          B[j] = part;
          if (!uni) U[j] = l1 * r0;
        }
        if (!REG || t == k_lo) {
          gIc[j] = gn;
          gIs[j] = sm;
        }
        if (t == k_lo) {
          // lambda_{k_lo - 1} complete, the partial sum of lambda_{k_lo - 2}
          (C.lam + ((k_lo - 1) & 1) * C.stride)[j] = l1;
          (C.lam + (k_lo & 1) * C.stride)[j] = part;
          C.u[j] = l1 * r0;
        }
      }
    };
    if constexpr (REG) {
#pragma unroll
      for (int k = 0; k < N; ++k) {
        if (k * BS + tid < pairs) sweep(k, k * BS + tid);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      for (int32_t q = tid; q < pairs; q += BS) sweep(0, q);
    }
  }
}

template <int BS>
const void* evolve_of(int pairs) {
  switch (pairs) {
    case 1: return reinterpret_cast<const void*>(evolve_resident_kernel<BS, 1>);
    case 2: return reinterpret_cast<const void*>(evolve_resident_kernel<BS, 2>);
    case 3: return reinterpret_cast<const void*>(evolve_resident_kernel<BS, 3>);
    default: return reinterpret_cast<const void*>(evolve_resident_kernel<BS, 0>);
  }
}

template <int BS>
const void* adjoint_of(int pairs) {
  switch (pairs) {
    case 1: return reinterpret_cast<const void*>(adjoint_resident_kernel<BS, 1>);
    case 2: return reinterpret_cast<const void*>(adjoint_resident_kernel<BS, 2>);
    case 3: return reinterpret_cast<const void*>(adjoint_resident_kernel<BS, 3>);
    default: return reinterpret_cast<const void*>(adjoint_resident_kernel<BS, 0>);
  }
}

}  // namespace

const void* resident_evolve_kernel(int block_size, int pairs) {
  switch (block_size) {
    case 64: return evolve_of<64>(pairs);
    case 128: return evolve_of<128>(pairs);
    case 256: return evolve_of<256>(pairs);
    case 512: return evolve_of<512>(pairs);
    default: return nullptr;
  }
}

const void* resident_adjoint_kernel(int block_size, int pairs) {
  switch (block_size) {
    case 64: return adjoint_of<64>(pairs);
    case 128: return adjoint_of<128>(pairs);
    case 256: return adjoint_of<256>(pairs);
    case 512: return adjoint_of<512>(pairs);
    default: return nullptr;
  }
}
