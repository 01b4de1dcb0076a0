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
// steps and for inputs that vary in time).
#include "jja_resident.h"

#include "jja_device.h"

namespace {

// +-v by the sign bit of an incidence code; 0 for an empty slot
__device__ __forceinline__ double signed_value(double v, uint32_t code) {
  const long long b = __builtin_bit_cast(long long, v) ^ (static_cast<long long>(code & 1u) << 63);
  return code == 0xffffu ? 0.0 : __builtin_bit_cast(double, b);
}
__device__ __forceinline__ uint32_t code_address(uint32_t code) { return code == 0xffffu ? 0u : code >> 1; }
__device__ __forceinline__ uint32_t pack_codes(int32_t a, int32_t b) {
  return static_cast<uint32_t>(a & 0xffff) | (static_cast<uint32_t>(b & 0xffff) << 16);
}

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
  const WorkItem wi = work[blockIdx.x];
  const DevProblem& P = probs[wi.problem];
  const jja_problem_run& R = runs[wi.problem];
  const int64_t w = wi.column;
  const int tid = threadIdx.x;
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

template <int BS>
const void* kernel_of(int pairs) {
  switch (pairs) {
    case 1: return reinterpret_cast<const void*>(evolve_resident_kernel<BS, 1>);
    case 2: return reinterpret_cast<const void*>(evolve_resident_kernel<BS, 2>);
    default: return reinterpret_cast<const void*>(evolve_resident_kernel<BS, 0>);
  }
}

}  // namespace

const void* resident_evolve_kernel(int block_size, int pairs) {
  switch (block_size) {
    case 64: return kernel_of<64>(pairs);
    case 128: return kernel_of<128>(pairs);
    case 256: return kernel_of<256>(pairs);
    case 512: return kernel_of<512>(pairs);
    case 1024: return pairs ? nullptr : kernel_of<1024>(0);
    default: return nullptr;
  }
}
