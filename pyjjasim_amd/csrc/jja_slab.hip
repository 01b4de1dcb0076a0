// Step kernels of lattice columns cut into row slabs, one workgroup each: a column
// of a few thousand to some ten thousand junctions then uses many compute units.
//
// Face row r couples to rows r - 1 and r + 1 only, and the sine transform along a
// row is local to it, so a part keeps the junctions its rows touch (the ones
// between two parts in both, which see the same bits), forms its face sums,
// transforms its rows and solves its own block of every mode's tridiagonal system,
// all in LDS. With w the solution of the own block alone, the rows of the whole
// system are x_l = w_l + V_l x_below + V_{s-1-l} x_above (V the block's response to
// its neighbour's row, a table), and the parts' first and last rows x are fixed
// linear combinations of every part's first and last w (a table, the inverse of the
// reduced system of the end rows; Wang, ACM TOMS 7 (1981) 170-183). The parts exchange those two
// rows, 2 C doubles each, and nothing else: one meeting a step, where a solve that
// splits rows for the transform and modes for the recurrence needs four to six and
// moves the whole face vector through memory twice. The inverse transform runs on
// the own rows and both neighbours' rows (x_below and x_above), so the junction
// pass needs no exchange either.
//
// The meeting: the wave that holds 32 modes publishes their end rows with
// device-scope stores, waits for them to be acknowledged and sets its own flag to
// the step's sequence number; the waves holding the same modes in the other parts
// poll those flags and read the rows. No counter, no workgroup barrier around it,
// and no cache write-back or invalidation: only the end rows pass between parts.
// Two buffers by parity suffice: a part writes a buffer again only after every
// part has published the step in between, which it does after reading.
#include "jja_slab.h"

#include <algorithm>
#include <cmath>

#include "jja_device.h"

namespace {

// Rows 0 .. rows - 1 of src times the sine matrix into dst (rows of ld doubles, on
// the matrix cores as dst_product<false>; row tiles past the last row read it again
// and are not stored). The table lies in LDS, or in memory with four steps loaded
// ahead.
template <class F>
__device__ __forceinline__ void slab_transform(const LAS double* src, LAS double* dst, F table, int32_t C, int32_t rows,
                                               int32_t ld, int32_t tid, int32_t nt) {
  constexpr bool LOCAL = std::is_same<F, const LAS double*>::value;
  constexpr int U = LOCAL ? 2 : 4;
  const DstShape D(C);
  const int lane = tid & (kWave - 1), lr = lane & 15, lk = lane >> 4;
  const int32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), NW = nt / kWave;
  const int32_t tasks = D.pairs * ((rows + 15) >> 4);
  for (int32_t task = wave, mb = wave, ob = 0; task < tasks; task += NW, mb += NW) {
    while (mb >= D.pairs) {
      mb -= D.pairs;
      ob += 16;
    }
    F f = table + mb * D.steps * 2 * kWave + lane;
    const int32_t row = min(ob + lr, rows - 1) * ld;
    const LAS double* s0 = src + row + lk;
    const LAS double* s1 = src + row + (C - 1 - lk);
    vdouble4 ae{0.0, 0.0, 0.0, 0.0}, ao{0.0, 0.0, 0.0, 0.0};
    double v[U][2];
    if constexpr (!LOCAL) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int32_t at = 2 * min(u, D.steps - 1) * kWave;
        v[u][0] = f[at];
        v[u][1] = f[at + kWave];
      }
    }
    for (int32_t k = 0; k < D.steps; k += U) {
      double p[U], q[U], vn[U][2];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        p[u] = s0[4 * u];
        q[u] = s1[-4 * u];
        if constexpr (LOCAL) {
          v[u][0] = f[(2 * u) * kWave];
          v[u][1] = f[(2 * u + 1) * kWave];
        } else {
          const int32_t at = 2 * min(k + U + u, D.steps - 1) * kWave;
          vn[u][0] = f[at];
          vn[u][1] = f[at + kWave];
        }
      }
      s0 += 4 * U;
      s1 -= 4 * U;
      if constexpr (LOCAL) f += 2 * U * kWave;
#pragma unroll
      for (int u = 0; u < U; ++u) {
        if (!LOCAL && k + u >= D.steps) break;   // steps are even, a batch holds four
        const double e = p[u] + q[u], d = p[u] - q[u];
        ae = __builtin_amdgcn_mfma_f64_16x16x4f64(e, v[u][0], ae, 0, 0, 0);
        ao = __builtin_amdgcn_mfma_f64_16x16x4f64(d, v[u][1], ao, 0, 0, 0);
      }
      if constexpr (!LOCAL) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
          v[u][0] = vn[u][0];
          v[u][1] = vn[u][1];
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int32_t o = ob + lk + 4 * r;
      if (o < rows) *reinterpret_cast<LAS vdouble2*>(dst + o * ld + 2 * (16 * mb + lr)) = vdouble2{ae[r], ao[r]};
    }
  }
}

// What one workgroup of a slab launch works on, and its LDS arrays.
struct Slab {
  int32_t part, s, r0, C, ld, parts;
  LAS double *Z, *Y, *inv;        // face rows, their transform (and before it the junction values), pivots
  const LAS double* table;
  GAS double* ends;               // this column's [2][parts][2][C]
  uint32_t* flags;                // this column's [parts][mode_waves]
  uint32_t wait_limit;
  int32_t* err;
  volatile int32_t* stopped;
};

__device__ __forceinline__ Slab slab_of(const DevProblem& P, const SlabDev& S, int64_t column, int32_t part, double* lds,
                                        int32_t* err, uint32_t wait_limit, volatile int32_t* stopped, int32_t tid, int32_t nt) {
  Slab b;
  b.part = part;
  b.parts = S.parts;
  b.s = S.base + (part < S.extra ? 1 : 0);
  b.r0 = part * S.base + min(part, S.extra);
  b.C = P.lat_cols;
  b.ld = S.ld;
  b.Z = (LAS double*)lds;
  b.Y = b.Z + S.buf;
  LAS double* next = b.Y + max(S.buf, 2 * S.pairs);
  b.inv = next;
  if (S.inv_lds) next += S.rows * b.C;
  b.table = next;
  const int32_t entries = DstShape(b.C).entries();
  b.ends = gblw(S.ends) + column * (4 * S.parts * static_cast<int64_t>(b.C));
  b.flags = S.flags + column * (S.parts * S.mode_waves);
  b.wait_limit = wait_limit;
  b.err = err;
  b.stopped = stopped;
  for (int32_t i = tid; i < S.buf + max(S.buf, 2 * S.pairs); i += nt) b.Z[i] = 0.0;
  if (S.inv_lds)
    for (int32_t i = tid; i < S.rows * b.C; i += nt) b.inv[i] = gbl(S.inv)[i];
  if (S.table_lds)
    for (int32_t i = tid; i < entries; i += nt) next[i] = gbl(S.table)[i];
  if (tid == 0) *stopped = 0;
  __syncthreads();
  return b;
}

// K^-1 of the column's face sums: in Z's rows 1 .. s on entry, the solution in rows
// 0 .. s + 1 on exit (a neighbour's row below the first or above the last face row
// is zero). seq: the step's sequence number.
__device__ __forceinline__ void slab_solve(const DevProblem& P, const SlabDev& S, const Slab& b, uint32_t seq, int32_t tid,
                                           int32_t nt) {
  constexpr int TB = 8;  // rows or terms loaded together
  const int32_t s = b.s, C = b.C, ld = b.ld, G = b.parts;
  if (S.table_lds)
    slab_transform<const LAS double*>(b.Z, b.Y, b.table, C, s + 2, ld, tid, nt);
  else
    slab_transform<const GAS double*>(b.Z, b.Y, gbl(S.table), C, s + 2, ld, tid, nt);
  lds_barrier();
  const int32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid & (kWave - 1);
  if (wave < S.mode_waves) {
    // two lanes a mode: both run the own block's recurrences (the same values), one
    // then takes the row below, the other the row above
    const int32_t k = min(tid >> 1, C - 1), side = tid & 1;
    const bool live = (tid >> 1) < C;
    const double g = P.lat_g;
    const GAS double* ginv = gbl(S.inv) + k;
    const LAS double* linv = b.inv + k;
    LAS double* y = b.Y + ld + k;
    double d = 0.0;
    for (int32_t l0 = 0; l0 < s; l0 += TB) {
      double v[TB], iv[TB];
#pragma unroll
      for (int q = 0; q < TB; ++q) {
        const int32_t l = min(l0 + q, s - 1);
        v[q] = y[l * ld];
        iv[q] = S.inv_lds ? linv[l * C] : ginv[l * C];
      }
#pragma unroll
      for (int q = 0; q < TB; ++q)
        if (l0 + q < s) {
          d = __builtin_fma(g, d, v[q]) * iv[q];
          y[(l0 + q) * ld] = d;
        }
    }
    const double last = d;
    double x = 0.0;
    for (int32_t l0 = s - 1; l0 >= 0; l0 -= TB) {
      double v[TB], iv[TB];
#pragma unroll
      for (int q = 0; q < TB; ++q) {
        const int32_t l = max(l0 - q, 0);
        v[q] = y[l * ld];
        iv[q] = S.inv_lds ? linv[l * C] : ginv[l * C];
      }
#pragma unroll
      for (int q = 0; q < TB; ++q)
        if (l0 - q >= 0) {
          x = __builtin_fma(g * iv[q], x, v[q]);
          y[(l0 - q) * ld] = x;
        }
    }
    // publish the end rows, wait for the other parts'
    const int64_t step = (seq & 1u) ? 2 * static_cast<int64_t>(G) * C : 0;
    GAS double* e = b.ends + step + k;
    if (live)
      __hip_atomic_store(reinterpret_cast<unsigned long long*>((double*)(e + (2 * b.part + side) * C)),
                         __builtin_bit_cast(unsigned long long, side ? last : x), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(kWaitVmem);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (lane == 0)
      __hip_atomic_store(b.flags + b.part * S.mode_waves + wave, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!*b.stopped) {
      const uint32_t* f = b.flags + min(lane, G - 1) * S.mode_waves + wave;
      uint32_t spins = 0;
      while (true) {
        const uint32_t v = __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__all(static_cast<int32_t>(v - seq) >= 0)) break;
        if (++spins > b.wait_limit) {
          // gives up for the rest of the launch; the host reports it
          *b.stopped = 1;
          __hip_atomic_store(b.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
    }
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    // four rows from all parts' end rows: the lower lane takes the last row of the
    // part below and this part's first, the upper lane this part's last row and the
    // first of the part above. Both neighbours form a row by the same sum, so the
    // junctions between two parts, which both keep, see the same bits in both (with
    // bits of their own the copies would drift apart like two separate junctions).
    const int32_t outer = side ? 2 * b.part + 2 : 2 * b.part - 1, own = 2 * b.part + side;
    const bool edge = outer < 0 || outer >= 2 * G;  // beyond the lattice: zero
    const GAS double* ro = gbl(S.reduced) + static_cast<int64_t>(edge ? own : outer) * 2 * G * C + k;
    const GAS double* rw = gbl(S.reduced) + static_cast<int64_t>(own) * 2 * G * C + k;
    double no = 0.0, nw = 0.0;
    for (int32_t i0 = 0; i0 < 2 * G; i0 += 4) {
      double ev[4], co[4], cw[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        ev[q] = __builtin_bit_cast(
            double, __hip_atomic_load(reinterpret_cast<unsigned long long*>((double*)(e + (i0 + q) * C)), __ATOMIC_RELAXED,
                                      __HIP_MEMORY_SCOPE_AGENT));
        co[q] = ro[(i0 + q) * C];
        cw[q] = rw[(i0 + q) * C];
      }
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        no = __builtin_fma(co[q], ev[q], no);
        nw = __builtin_fma(cw[q], ev[q], nw);
      }
    }
    if (edge) no = 0.0;
    const double swapped = dpp_f64<0xB1, 0xf>(no);  // quad_perm [1, 0, 3, 2]: the mode's other lane
    const double below = side ? swapped : no, above = side ? no : swapped;
    const GAS double* V = gbl(S.spike) + (s > S.base ? static_cast<int64_t>(S.rows) * C : 0) + k;
    for (int32_t l0 = 1 + side; l0 < s - 1; l0 += 2 * TB) {
      double v[TB], va[TB], vb[TB];
#pragma unroll
      for (int q = 0; q < TB; ++q) {
        const int32_t l = min(l0 + 2 * q, s - 1);
        v[q] = y[l * ld];
        va[q] = V[l * C];
        vb[q] = V[(s - 1 - l) * C];
      }
#pragma unroll
      for (int q = 0; q < TB; ++q)
        if (l0 + 2 * q < s - 1) y[(l0 + 2 * q) * ld] = __builtin_fma(va[q], below, __builtin_fma(vb[q], above, v[q]));
    }
    y[(side ? s - 1 : 0) * ld] = nw;
    b.Y[(side ? s + 1 : 0) * ld + k] = no;
  }
  lds_barrier();
  if (S.table_lds)
    slab_transform<const LAS double*>(b.Y, b.Z, b.table, C, s + 2, ld, tid, nt);
  else
    slab_transform<const GAS double*>(b.Y, b.Z, gbl(S.table), C, s + 2, ld, tid, nt);
  lds_barrier();
}

// One face of the part's own rows: its sum's codes into the junction values, where
// the sum goes and the face's index.
struct SlabFace {
  uint32_t code[2], at;
  int32_t id;
};

__device__ __forceinline__ SlabFace slab_face(const SlabDev& S, const Slab& b, int32_t slot) {
  SlabFace f{{0xffffffffu, 0xffffffffu}, 0xffffffffu, -1};
  if (slot < b.s * b.C) {
    const int64_t at = static_cast<int64_t>(b.part) * S.faces + slot;
    const vuint2 c = gbl(reinterpret_cast<const vuint2*>(S.face_code))[at];
    f.code[0] = c.x;
    f.code[1] = c.y;
    f.at = gbl(S.face_at)[at];
    f.id = gbl(S.face_id)[at];
  }
  return f;
}

__device__ __forceinline__ double face_sum(const SlabFace& f, const LAS double* U) {
  double uv[4], acc = 0.0;
#pragma unroll
  for (int i = 0; i < 4; ++i) uv[i] = U[code_address((f.code[i >> 1] >> (16 * (i & 1))) & 0xffffu)];
#pragma unroll
  for (int i = 0; i < 4; ++i) acc = acc + signed_value(uv[i], (f.code[i >> 1] >> (16 * (i & 1))) & 0xffffu);
  return acc;
}

// NP: junction pairs a thread holds in registers (phases and right-hand sides; with
// few pairs also their constant inputs).
template <int BS, int NP>
__global__ __launch_bounds__(BS) void evolve_slab_kernel(const DevProblem* __restrict__ probs,
                                                         const jja_problem_run* __restrict__ runs,
                                                         const WorkItem* __restrict__ work,
                                                         const SlabDev* __restrict__ slabs, int32_t n_steps,
                                                         int64_t step0, uint32_t seq0, int32_t* err,
                                                         uint32_t wait_limit) {
  extern __shared__ double lds[];
  __shared__ volatile int32_t stopped;
  constexpr bool KEEP = NP <= 2;
  constexpr int NF = kSlabFacesPerPair * NP;
  WorkItem wi = work[blockIdx.x];
  wi.problem = __builtin_amdgcn_readfirstlane(wi.problem);
  wi.column = __builtin_amdgcn_readfirstlane(wi.column);
  const DevProblem& P = probs[wi.problem];
  const jja_problem_run& R = runs[wi.problem];
  const SlabDev& S = slabs[wi.problem];
  const int64_t w = wi.column / S.parts;
  const int32_t tid0 = threadIdx.x, tid = tid0;
  const Slab b = slab_of(P, S, w, wi.column % S.parts, lds, err, wait_limit, &stopped, tid, BS);
  LAS double* const U = b.Y;
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
  const GAS int32_t* list = gbl(S.pair) + static_cast<int64_t>(b.part) * S.pairs;
  const GAS uint32_t* codes = gbl(S.pair_code) + static_cast<int64_t>(b.part) * S.pairs * 2;
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
  SlabFace face[NF];
  double fx[NF];
  const bool keep_f = KEEP && R.f.s_t == 0;
  if constexpr (KEEP) {
    const TermView fv = term_view(R.f, !R.f.zero, P.zero, w, R.f.t0);
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      face[k] = slab_face(S, b, k * BS + tid);
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
    const SlabDev& S = slabs[again];
    const int32_t tid = opaque(tid0);
    {
      const TermView fv = term_view(R.f, !R.f.zero, P.zero, w, t);
      double fq[NF];
#pragma unroll
      for (int k = 0; k < NF; ++k) {
        if constexpr (!KEEP) face[k] = slab_face(S, b, k * BS + tid);
        fq[k] = KEEP ? fx[k] * fv.amp : 0.0;
        if (!keep_f) fq[k] = face[k].id >= 0 ? term_at(fv, face[k].id) : 0.0;
      }
      lds_barrier();
#pragma unroll
      for (int k = 0; k < NF; ++k)
        if (face[k].at != 0xffffffffu) b.Z[face[k].at] = face_sum(face[k], U) - kTwoPi * fq[k];
      lds_barrier();
    }
    slab_solve(P, S, b, seq0 + 1u + static_cast<uint32_t>(n), tid, BS);
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
          const double za = b.Z[code_address(ca)], zb = b.Z[code_address(cb)];
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
}

// The adjoint sweep (adjoint_steps) of a part: with few pairs a thread keeps
// lambda_k, the partial sum of lambda_{k-1}, both gradients and the phases of two
// steps of its junctions in registers for the whole launch; with more, lambda alone.
template <int BS, int NP>
__global__ __launch_bounds__(BS) void adjoint_slab_kernel(const DevProblem* __restrict__ probs,
                                                          const jja_adjoint_run* __restrict__ runs,
                                                          const WorkItem* __restrict__ work,
                                                          const SlabDev* __restrict__ slabs, int64_t k_hi, int64_t k_lo,
                                                          uint32_t seq0, int32_t* err, uint32_t wait_limit) {
  extern __shared__ double lds[];
  __shared__ volatile int32_t stopped;
  constexpr bool KEEP = NP <= 2;
  constexpr int NF = kSlabFacesPerPair * NP, N = KEEP ? NP : 1, K = KEEP ? NF : 1;
  WorkItem wi = work[blockIdx.x];
  wi.problem = __builtin_amdgcn_readfirstlane(wi.problem);
  wi.column = __builtin_amdgcn_readfirstlane(wi.column);
  const DevProblem& P = probs[wi.problem];
  const jja_adjoint_run& A = runs[wi.problem];
  const SlabDev& S = slabs[wi.problem];
  const int64_t w = wi.column / S.parts;
  const int32_t tid0 = threadIdx.x, tid = tid0;
  const Slab b = slab_of(P, S, w, wi.column % S.parts, lds, err, wait_limit, &stopped, tid, BS);
  LAS double* const U = b.Y;
  const int32_t Nj = P.Nj;
  const AdjCol C = adjoint_column(P, A, w);
  GAS double* const gIc = gblw(A.grad_Ic) + static_cast<size_t>(w) * Nj;
  GAS double* const gIs = gblw(A.grad_Is) + static_cast<size_t>(w) * Nj;
  GAS double* const gf = gblw(A.grad_f) + static_cast<size_t>(w) * P.Nf + static_cast<size_t>(b.r0) * b.C;
  const bool uni = P.coef_si == 0;
  double rc0 = 0.0, c1 = 0.0, c2 = 0.0;
  if (uni) {
    rc0 = rc0_at(P, 0);
    c1 = coef_at(P, 1, 0);
    c2 = coef_at(P, 2, 0);
  }
  auto history = [&](int64_t m, int32_t j) { return C.hist[static_cast<size_t>(m - C.hist_m0) * C.stride + j]; };
  const GAS int32_t* list = gbl(S.pair) + static_cast<int64_t>(b.part) * S.pairs;
  const GAS uint32_t* codes = gbl(S.pair_code) + static_cast<int64_t>(b.part) * S.pairs * 2;
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
  SlabFace face[K];
  double af[K];
  if constexpr (KEEP) {
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      face[k] = slab_face(S, b, k * BS + tid);
      af[k] = k * BS + tid < b.s * b.C ? gf[k * BS + tid] : 0.0;
    }
  }
  for (int64_t t = k_hi; t >= k_lo; --t) {
    const int32_t again = wi.problem + opaque_zero();
    const DevProblem& P = probs[again];
    const jja_adjoint_run& A = runs[again];
    const SlabDev& S = slabs[again];
    const int32_t tid = opaque(tid0);
    lds_barrier();
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      const SlabFace f = KEEP ? face[KEEP ? k : 0] : slab_face(S, b, k * BS + tid);
      if (f.at != 0xffffffffu) b.Z[f.at] = face_sum(f, U);
    }
    lds_barrier();
    slab_solve(P, S, b, seq0 + 1u + static_cast<uint32_t>(k_hi - t), tid, BS);
#pragma unroll
    for (int k = 0; k < NF; ++k) {
      if constexpr (KEEP) {
        if (face[k].at != 0xffffffffu) af[k] = af[k] - kTwoPi * b.Z[face[k].at];
      } else {
        const int32_t slot = k * BS + tid;
        if (slot < b.s * b.C) gf[slot] = gf[slot] - kTwoPi * b.Z[slab_face(S, b, slot).at];
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
          const double za = b.Z[code_address(ca)], zb = b.Z[code_address(cb)];
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
      if (k * BS + tid < b.s * b.C) gf[k * BS + tid] = af[k];
  }
}

// the tables are formed in extended precision: their rounding is that of one value
using real = long double;

std::vector<real> thomas_inverse(real diag, real g, int32_t s) {
  std::vector<real> inv(s);
  real piv = diag;
  for (int32_t l = 0; l < s; ++l) {
    inv[l] = 1.0 / piv;
    piv = diag - g * g * inv[l];
  }
  return inv;
}

// g A^-1 e_0 for the block of s rows
std::vector<real> spike_of(const std::vector<real>& inv, real g, int32_t s) {
  std::vector<real> v(s);
  real d = 0.0;
  for (int32_t l = 0; l < s; ++l) v[l] = d = ((l == 0 ? g : 0.0) + g * d) * inv[l];
  for (int32_t l = s - 2; l >= 0; --l) v[l] += g * inv[l] * v[l + 1];
  return v;
}

// Inverse of the n x n matrix a in place (Gauss-Jordan, partial pivoting).
void invert(std::vector<real>& a, int32_t n) {
  std::vector<real> r(static_cast<size_t>(n) * n, 0.0);
  for (int32_t i = 0; i < n; ++i) r[static_cast<size_t>(i) * n + i] = 1.0;
  for (int32_t c = 0; c < n; ++c) {
    int32_t p = c;
    for (int32_t i = c + 1; i < n; ++i)
      if (std::fabs(a[static_cast<size_t>(i) * n + c]) > std::fabs(a[static_cast<size_t>(p) * n + c])) p = i;
    for (int32_t j = 0; j < n && p != c; ++j) {
      std::swap(a[static_cast<size_t>(p) * n + j], a[static_cast<size_t>(c) * n + j]);
      std::swap(r[static_cast<size_t>(p) * n + j], r[static_cast<size_t>(c) * n + j]);
    }
    const real d = 1.0 / a[static_cast<size_t>(c) * n + c];
    for (int32_t j = 0; j < n; ++j) {
      a[static_cast<size_t>(c) * n + j] *= d;
      r[static_cast<size_t>(c) * n + j] *= d;
    }
    for (int32_t i = 0; i < n; ++i) {
      const real f = a[static_cast<size_t>(i) * n + c];
      if (i == c || f == 0.0) continue;
      for (int32_t j = 0; j < n; ++j) {
        a[static_cast<size_t>(i) * n + j] -= f * a[static_cast<size_t>(c) * n + j];
        r[static_cast<size_t>(i) * n + j] -= f * r[static_cast<size_t>(c) * n + j];
      }
    }
  }
  a = r;
}

}  // namespace

int64_t slab_lds_doubles(const SlabDev& d, int32_t cols) {
  return static_cast<int64_t>(d.buf) + std::max(d.buf, 2 * d.pairs) + (d.inv_lds ? static_cast<int64_t>(d.rows) * cols : 0) +
         (d.table_lds ? DstShape(cols).entries() : 0);
}

bool build_slabs(const jja_problem_desc& desc, int32_t parts, int64_t lds_bytes, SlabHost* out) {
  const int32_t R = desc.lattice_rows, C = desc.lattice_cols, Nj = desc.n_junctions, G = parts;
  if (R < 2 * G || C < 8 || G < 2) return false;  // two rows a part: its first and its last
  SlabDev& d = out->d;
  d.parts = G;
  d.base = R / G;
  d.extra = R % G;
  d.rows = d.base + (d.extra ? 1 : 0);
  d.ld = DstShape(C).padded() + 4;
  d.buf = (d.rows + 2) * d.ld;
  d.mode_waves = (2 * C + 63) / 64;
  d.faces = d.rows * C;
  if (d.buf > 32767 || 64 * d.mode_waves > kSlabBlock) return false;
  auto first_row = [&](int32_t p) { return p * d.base + std::min(p, d.extra); };
  auto part_of = [&](int32_t r) {
    const int32_t big = d.extra * (d.base + 1);
    return r < big ? r / (d.base + 1) : d.extra + (r - big) / d.base;
  };
  // junctions of every part: those with a face in its rows; the owner holds the
  // lowest of them
  std::vector<std::vector<int32_t>> mask(G, std::vector<int32_t>((Nj + 1) / 2, 0));
  for (int32_t j = 0; j < Nj; ++j) {
    int32_t rows[2] = {-1, -1}, n = 0, pos[2] = {-1, -1};
    for (int32_t i = 0; i < 2; ++i) {
      const int32_t c = desc.junc_code[2 * j + i];
      if (c < 0) continue;
      pos[n] = c >> 1;
      rows[n++] = (c >> 1) / C;
    }
    if (n == 2 && std::abs(pos[0] - pos[1]) != C && !(rows[0] == rows[1] && std::abs(pos[0] - pos[1]) == 1)) return false;
    int32_t owner = 0;
    if (n) owner = part_of(n == 2 ? std::min(rows[0], rows[1]) : rows[0]);
    auto put = [&](int32_t p) { mask[p][j / 2] |= (1 << (j & 1)) | (p == owner ? 4 << (j & 1) : 0); };
    put(owner);
    for (int32_t i = 0; i < n; ++i)
      if (part_of(rows[i]) != owner) put(part_of(rows[i]));
  }
  d.pairs = 0;
  for (int32_t p = 0; p < G; ++p) {
    int32_t n = 0;
    for (int32_t v : mask[p]) n += v != 0;
    d.pairs = std::max(d.pairs, n);
  }
  if (2 * d.pairs > 32767 || Nj >= (1 << 27)) return false;
  out->pair.assign(static_cast<size_t>(G) * d.pairs, -1);
  out->pair_code.assign(2 * static_cast<size_t>(G) * d.pairs, 0xffffffffu);
  out->face_id.assign(static_cast<size_t>(G) * d.faces, -1);
  out->face_at.assign(static_cast<size_t>(G) * d.faces, 0);
  out->face_code.assign(2 * static_cast<size_t>(G) * d.faces, 0xffffffffu);
  for (int32_t p = 0; p < G; ++p) {
    const int32_t r0 = first_row(p), s = d.base + (p < d.extra ? 1 : 0);
    std::vector<int32_t> count(static_cast<size_t>(s) * C, 0);
    std::vector<uint16_t> fcode(static_cast<size_t>(s) * C * 4, 0xffffu);
    int32_t slot = 0;
    for (int32_t q = 0; q < (Nj + 1) / 2; ++q) {
      if (!mask[p][q]) continue;
      out->pair[static_cast<size_t>(p) * d.pairs + slot] = q * 16 + mask[p][q];
      for (int32_t m = 0; m < 2; ++m) {
        if (!(mask[p][q] >> m & 1)) continue;
        uint32_t word = 0;
        for (int32_t i = 0; i < 2; ++i) {
          const int32_t c = desc.junc_code[2 * (2 * q + m) + i];
          uint32_t code = 0xffffu;
          if (c >= 0) {
            const int32_t row = (c >> 1) / C - r0, cl = (c >> 1) % C;
            if (row < -1 || row > s) return false;
            code = static_cast<uint32_t>(2 * ((row + 1) * d.ld + cl) + (c & 1));
            if (row >= 0 && row < s) {
              int32_t& n = count[static_cast<size_t>(row) * C + cl];
              if (n == 4) return false;
              fcode[(static_cast<size_t>(row) * C + cl) * 4 + n++] = static_cast<uint16_t>(2 * (2 * slot + m) + (c & 1));
            }
          }
          word |= code << (16 * i);
        }
        out->pair_code[2 * (static_cast<size_t>(p) * d.pairs + slot) + m] = word;
      }
      ++slot;
    }
    for (int32_t e = 0; e < s * C; ++e) {
      const size_t at = static_cast<size_t>(p) * d.faces + e;
      out->face_at[at] = static_cast<uint32_t>((e / C + 1) * d.ld + e % C);
      out->face_id[at] = desc.face_of_pos[r0 * C + e];
      for (int32_t i = 0; i < 2; ++i)
        out->face_code[2 * at + i] = fcode[4 * static_cast<size_t>(e) + 2 * i] |
                                     static_cast<uint32_t>(fcode[4 * static_cast<size_t>(e) + 2 * i + 1]) << 16;
    }
  }
  // per mode: the own block's pivots and responses, and the reduced system
  const real pi = 3.14159265358979323846264338328L, g = desc.lattice_g;
  out->inv.assign(static_cast<size_t>(d.rows) * C, 0.0);
  out->spike.assign(2 * static_cast<size_t>(d.rows) * C, 0.0);
  out->reduced.assign(static_cast<size_t>(G) * 4 * G * C, 0.0);
  for (int32_t k = 0; k < C; ++k) {
    const real h = std::sin(pi * (k + 1) / (2 * static_cast<real>(C + 1))), diag = 2 * g + desc.lattice_gc * 4 * h * h;
    const std::vector<real> inv = thomas_inverse(diag, g, d.rows);
    std::vector<real> v[2];
    for (int32_t i = 0; i < 2; ++i) {
      const int32_t s = std::min(d.base + i, d.rows);
      v[i] = spike_of(inv, g, s);
      for (int32_t l = 0; l < s; ++l) out->spike[(static_cast<size_t>(i) * d.rows + l) * C + k] = static_cast<double>(v[i][l]);
    }
    for (int32_t l = 0; l < d.rows; ++l) out->inv[static_cast<size_t>(l) * C + k] = static_cast<double>(inv[l]);
    // unknowns 2p, 2p + 1: the first and last row of part p
    const int32_t n = 2 * G;
    std::vector<real> m(static_cast<size_t>(n) * n, 0.0);
    for (int32_t p = 0; p < G; ++p) {
      const std::vector<real>& vp = v[p < d.extra ? 1 : 0];
      const int32_t s = d.base + (p < d.extra ? 1 : 0);
      for (int32_t e = 0; e < 2; ++e) {
        real* row = &m[static_cast<size_t>(2 * p + e) * n];
        const int32_t l = e ? s - 1 : 0;
        row[2 * p + e] = 1.0;
        if (p > 0) row[2 * p - 1] -= vp[l];
        if (p + 1 < G) row[2 * p + 2] -= vp[s - 1 - l];
      }
    }
    invert(m, n);
    for (size_t i = 0; i < m.size(); ++i) out->reduced[i * C + k] = static_cast<double>(m[i]);
  }
  // LDS: the pivots, then the sine table, where there is room
  d.inv_lds = d.table_lds = 0;
  if (8 * slab_lds_doubles(d, C) > lds_bytes) return false;
  d.inv_lds = 1;
  if (8 * slab_lds_doubles(d, C) > lds_bytes) d.inv_lds = 0;
  d.table_lds = 1;
  if (8 * slab_lds_doubles(d, C) > lds_bytes) d.table_lds = 0;
  return true;
}

const void* slab_evolve_kernel(int pairs) {
  if (pairs <= 1) return reinterpret_cast<const void*>(evolve_slab_kernel<kSlabBlock, 1>);
  if (pairs <= 2) return reinterpret_cast<const void*>(evolve_slab_kernel<kSlabBlock, 2>);
  if (pairs <= 3) return reinterpret_cast<const void*>(evolve_slab_kernel<kSlabBlock, 3>);
  if (pairs <= 5) return reinterpret_cast<const void*>(evolve_slab_kernel<kSlabBlock, 5>);
  return pairs <= kSlabPairs ? reinterpret_cast<const void*>(evolve_slab_kernel<kSlabBlock, kSlabPairs>) : nullptr;
}

const void* slab_adjoint_kernel(int pairs) {
  if (pairs <= 1) return reinterpret_cast<const void*>(adjoint_slab_kernel<kSlabBlock, 1>);
  if (pairs <= 2) return reinterpret_cast<const void*>(adjoint_slab_kernel<kSlabBlock, 2>);
  if (pairs <= 3) return reinterpret_cast<const void*>(adjoint_slab_kernel<kSlabBlock, 3>);
  if (pairs <= 5) return reinterpret_cast<const void*>(adjoint_slab_kernel<kSlabBlock, 5>);
  return pairs <= kSlabPairs ? reinterpret_cast<const void*>(adjoint_slab_kernel<kSlabBlock, kSlabPairs>) : nullptr;
}
