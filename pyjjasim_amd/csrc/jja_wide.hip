// Step kernel of large lattice columns that one workgroup holds whole: the two values
// a junction keeps from step to step lie in registers (kWidePairs pairs a thread, 160 of
// its 256 registers), the face vector twice in LDS.
//
// With the phases in memory such a column moves 50 bytes a junction and step (243 MB for
// 256 columns of 100x100, more than the L2 holds), and that bounds the step: without
// noise, sine and solve it still took 53 of 90 us. Here a step reads the critical
// currents, sources and codes, 24 bytes, most of them from the L2. What bounds it now,
// 100x100 with noise, in cycles of one CU: 70,000 of junction pass (300 vector
// instructions a pair, two waves a SIMD), 41,000 of the two transforms (12,000 of them
// matrix instructions on each SIMD; the rest waits for the table and LDS), 18,000 of the
// tridiagonal systems and 17,000 of face sums (mostly latency of the L2). Measured, us a
// step, 256 columns: 100x100 89.5 before, 62.0 now; 70x70 50.5 before, 37.9 now.
#include "jja_wide.h"

#include <algorithm>

#include "jja_device.h"
#include "jja_rowparts.h"

namespace {

typedef double vdouble16 __attribute__((ext_vector_type(16)));

// at_offset for data that no other column reads: it does not displace the tables that
// all columns share from the L2.
template <class T>
__device__ __forceinline__ T stream_offset(const GAS T* base, uint32_t bytes) {
  return __builtin_nontemporal_load(reinterpret_cast<const GAS T*>(reinterpret_cast<const GAS char*>(base) + bytes));
}

// The transforms here are those of jja_rowdst.h (whose header says why they are as they
// are) without its blocks of four rows: with that code in this kernel, which holds 160
// registers of state, its forms spilled 46 to 138 registers.
//
// The table's values of four steps are loaded together, a batch ahead of the products
// (and the next task's first ones before the last steps of a task): they come from the
// L2, which answers in 1000 to 2000 cycles here, and the matrix pipe works on a batch
// of two waves for 2000.
constexpr int kWideBatch = 4;
struct WideBatch {
  double v[kWideBatch][2];
};
__device__ __forceinline__ void wide_fetch(const GAS double* f, int32_t k, int32_t stored, WideBatch& b) {
#pragma unroll
  for (int u = 0; u < kWideBatch; ++u) {
    const int32_t at = 2 * min(k + u, stored - 1) * kWave;
    b.v[u][0] = f[at];
    b.v[u][1] = f[at + kWave];
  }
}

// The products of one task; v holds its first batch and receives that of the next.
template <bool TWO>
__device__ __forceinline__ void wide_products(const GAS double* f, const GAS double* next, int32_t stored, int32_t steps,
                                              const LAS double* a0, const LAS double* a1, const LAS double* b0,
                                              const LAS double* b1, WideBatch& v, vdouble4& ae, vdouble4& ao, vdouble4& be,
                                              vdouble4& bo) {
  constexpr int U = kWideBatch;
  WideBatch vn;
  double x[4], nx[4];  // the operands of a step, loaded a step ahead
  auto load = [&](int u, double (&o)[4]) __attribute__((always_inline)) {
    o[0] = a0[4 * u];
    o[1] = a1[-4 * u];
    if constexpr (TWO) {
      o[2] = b0[4 * u];
      o[3] = b1[-4 * u];
    }
  };
  auto step = [&](int u) __attribute__((always_inline)) {
    ae = __builtin_amdgcn_mfma_f64_16x16x4f64(x[0] + x[1], v.v[u][0], ae, 0, 0, 0);
    ao = __builtin_amdgcn_mfma_f64_16x16x4f64(x[0] - x[1], v.v[u][1], ao, 0, 0, 0);
    if constexpr (TWO) {
      be = __builtin_amdgcn_mfma_f64_16x16x4f64(x[2] + x[3], v.v[u][0], be, 0, 0, 0);
      bo = __builtin_amdgcn_mfma_f64_16x16x4f64(x[2] - x[3], v.v[u][1], bo, 0, 0, 0);
    }
  };
  load(0, x);
  int32_t k = 0;
  for (; k + U <= steps; k += U) {
    const bool more = k + U < steps;
    wide_fetch(more ? f : next, more ? k + U : 0, stored, vn);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u + 1 < U) {
        load(u + 1, nx);
      } else {
        const int32_t on = more ? 4 * U : 0;
        a0 += on;
        a1 -= on;
        b0 += on;
        b1 -= on;
        load(0, nx);
      }
      __builtin_amdgcn_sched_barrier(0);
      step(u);
#pragma unroll
      for (int i = 0; i < (TWO ? 4 : 2); ++i) x[i] = nx[i];
    }
    v = vn;
  }
  if (k < steps) {
    wide_fetch(next, 0, stored, vn);
#pragma unroll
    for (int u = 0; u < U - 1; ++u)
      if (k + u < steps) {
        if (u) load(u, x);
        step(u);
      }
    v = vn;
  }
}

// Rows of src times the sine matrix into dst, after a barrier; a task is one block of
// 16 modes of each parity for one or two blocks of 16 rows, whose products share the
// table's values.
__device__ __forceinline__ void wide_transform(const LAS double* src, LAS double* dst, const GAS double* table, int32_t C,
                                               int32_t rows, int32_t ld, int32_t tid) {
  const DstShape D(C);
  const int lane = tid & (kWave - 1), lr = lane & 15, lk = lane >> 4;
  const int32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), NW = kWideBlock / kWave;
  const int32_t blocks = (rows + 15) >> 4, steps = (D.h + 3) >> 2;
  const int32_t each = D.pairs * ((blocks + 1) >> 1) >= NW ? 2 : 1;
  const int32_t tasks = D.pairs * ((blocks + each - 1) / each);
  int32_t mb = wave, ob = 0;
  auto settle = [&]() {
    while (mb >= D.pairs) {
      mb -= D.pairs;
      ob += 16 * each;
    }
  };
  settle();
  const GAS double* f = table + mb * D.steps * 2 * kWave + lane;
  WideBatch v;
  wide_fetch(f, 0, D.steps, v);
  lds_barrier();
  for (int32_t task = wave; task < tasks; task += NW) {
    const int32_t mine = mb, row = ob;
    mb += NW;
    settle();
    const GAS double* next = table + mb * D.steps * 2 * kWave + lane;
    const bool two = each == 2 && row + 16 < rows;
    const int32_t rowa = min(row + lr, rows - 1) * ld, rowb = min(row + 16 + lr, rows - 1) * ld;
    const LAS double* a0 = src + rowa + lk;
    const LAS double* a1 = src + rowa + (C - 1 - lk);
    const LAS double* b0 = src + rowb + lk;
    const LAS double* b1 = src + rowb + (C - 1 - lk);
    vdouble4 ae{0.0, 0.0, 0.0, 0.0}, ao = ae, be = ae, bo = ae;
    if (two)
      wide_products<true>(f, next, D.steps, steps, a0, a1, b0, b1, v, ae, ao, be, bo);
    else
      wide_products<false>(f, next, D.steps, steps, a0, a1, b0, b1, v, ae, ao, be, bo);
    f = next;
    if (16 * mine + lr < D.h) {
      LAS double* d = dst + 2 * (16 * mine + lr);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int32_t o = row + lk + 4 * r;
        if (o < rows) *reinterpret_cast<LAS vdouble2*>(d + o * ld) = vdouble2{ae[r], ao[r]};
        if (two && o + 16 < rows) *reinterpret_cast<LAS vdouble2*>(d + (o + 16) * ld) = vdouble2{be[r], bo[r]};
      }
    }
  }
}

// The tridiagonal systems of all modes, in place in y (row l of mode k at l * ld + k):
// the threads of a mode take a part of its rows each and keep them in registers
// (Wang's partition as in the row slabs; `ends` takes the parts' end rows in LDS, from
// their own blocks and then of the whole system). Tables of a part have kWideRows rows,
// zero past its own: what is read past a part's end (the next part's row) counts for
// nothing without a test.
__device__ __forceinline__ void wide_tridiagonal(const DevProblem& P, const WideDev& S, LAS double* yy, LAS double* ends,
                                                 int32_t C, int32_t ld, int32_t part, int32_t k) {
  constexpr int N = kWideRows, H = N / 2;
  const bool live = part < S.parts;
  part = live ? part : 0;
  const int32_t rows = S.rows, s = S.base + (part < S.extra ? 1 : 0);
  const int32_t n = 2 * S.parts;
  const uint32_t lane = 8 * static_cast<uint32_t>((s > S.base ? N * C : 0) + k);
  const double g = P.lat_g;
  LAS double* y = yy + (part * S.base + min(part, S.extra)) * ld + k;
  LAS double* own = ends + 2 * part * C + k;
  double x[N];
  {
    double iv[N], d = 0.0;
#pragma unroll
    for (int l = 0; l < N; ++l) iv[l] = at_offset(gbl(S.inv) + l * C, lane);
    lds_barrier();
#pragma unroll
    for (int l = 0; l < N; ++l) x[l] = y[min(l, rows - 1) * ld];
#pragma unroll
    for (int l = 0; l < N; ++l) x[l] = d = __builtin_fma(g, d, x[l]) * iv[l];
    double last = x[N - 1];
#pragma unroll
    for (int l = N - 2; l >= 0; --l) {
      if (l >= rows - 2) last = l == s - 1 ? x[l] : last;
      x[l] = __builtin_fma(g * iv[l], x[l + 1], x[l]);
    }
    if (live) {
      own[0] = x[0];
      own[C] = last;
    }
  }
  {
    // chunks of four end rows, the coefficients two chunks ahead (zero past the last)
    const uint32_t at = 8 * static_cast<uint32_t>(2 * part * S.ends * C + k);
    double first = 0.0, last = 0.0, c[2][4][2];
    auto fetch = [&](double (&to)[4][2], int32_t i0) __attribute__((always_inline)) {
      i0 = min(i0, S.ends - 4);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        to[q][0] = at_offset(gbl(S.reduced) + (i0 + q) * C, at);
        to[q][1] = at_offset(gbl(S.reduced) + (S.ends + i0 + q) * C, at);
      }
    };
    auto add = [&](double (&from)[4][2], int32_t i0) __attribute__((always_inline)) {
      double e[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) e[q] = ends[min(i0 + q, n - 1) * C + k];
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        first = __builtin_fma(from[q][0], e[q], first);
        last = __builtin_fma(from[q][1], e[q], last);
      }
    };
    fetch(c[0], 0);
    fetch(c[1], 4);
    lds_barrier();
    for (int32_t i0 = 0; i0 < S.ends; i0 += 8) {
      add(c[0], i0);
      fetch(c[0], i0 + 8);
      if (i0 + 4 < S.ends) {
        add(c[1], i0 + 4);
        fetch(c[1], i0 + 12);
      }
    }
    if (live) {
      own[n * C] = first;
      own[(n + 1) * C] = last;
    }
  }
  double vb[H], va[H];
#pragma unroll
  for (int i = 0; i < H; ++i) {
    vb[i] = at_offset(gbl(S.spike) + i * C, lane);
    va[i] = at_offset(gbl(S.spike) + (2 * N + i) * C, lane);
  }
  lds_barrier();
  if (live) {
    const double below = part ? own[(n - 1) * C] : 0.0, above = part + 1 < S.parts ? own[(n + 2) * C] : 0.0;
#pragma unroll
    for (int l = 0; l < N; ++l) {
      x[l] = __builtin_fma(vb[l % H], below, __builtin_fma(va[l % H], above, x[l]));
      if (l + H < N) {
        vb[l] = at_offset(gbl(S.spike) + (H + l) * C, lane);
        va[l] = at_offset(gbl(S.spike) + (2 * N + H + l) * C, lane);
      }
      if (l < rows - 1 || (l == rows - 1 && l < s)) y[l * ld] = x[l];
    }
  }
}

// Difference of the two doubles a code names.
__device__ __forceinline__ double coded_difference(const LAS double* lds, uint32_t code) {
  return lds[code & 0xffffu] - lds[code >> 16];
}

// What a pair reads of memory in a pass (UNI: the coefficients and the noise amplitude
// are one value each and are not among it).
template <bool UNI>
struct WideInput {
  vuint2 code;
  double ic[2], is[2], more[UNI ? 1 : 2][4];
};

// One pass over the thread's pairs: UPDATE finishes step t (else its phases come from
// memory), and step t + 1 is prepared. The work on a pair is one straight run of
// instructions, so that its three sine and cosine evaluations share the polynomials'
// constants, with the next pair's inputs loaded at its start. `out` steps (stored, or
// the launch's last) then write their values.
template <bool GAUSS, bool UNI, bool UPDATE>
__device__ __forceinline__ void wide_pass(const DevProblem& P, const jja_problem_run& R, const WideDev& S, LAS double* Z,
                                          vdouble16 (&state)[kWideGroups], int64_t w, int32_t tid, bool prep, int64_t t) {
  constexpr int BS = kWideBlock;
  const int32_t Nj = P.Nj, pairs = (Nj + 1) >> 1;
  LAS double* const U = Z + S.buf + 2;
  const uint32_t noise_col = static_cast<uint32_t>(R.column_offset + w);
  const GAS double* Icp = gbl(R.Ic ? R.Ic : P.Ic);
  // a source marked zero is left out of the step, whatever its values
  const TermView isn = term_view(R.Is, prep && !R.Is.zero, P.zero, w, t + 1);
  const TermView sgn = term_view(R.sigma, GAUSS && prep && !R.T.zero, P.zero, w, t + 1);
  const double rc0 = rc0_at(P, 0), c1 = coef_at(P, 1, 0), c2 = coef_at(P, 2, 0), sg0 = sgn.p[0] * sgn.amp;
  const size_t stride = static_cast<size_t>(R.W) * Nj, col = static_cast<size_t>(w) * Nj;
  GAS double* const even = gblw(R.theta) + col;  // phases of even and odd steps
  GAS double* const odd = even + stride;
  const int32_t tho = UPDATE && R.th_slot ? gbl(R.th_slot)[t - R.slot_t0] : -1;
  const int32_t Io = UPDATE && R.I_slot ? gbl(R.I_slot)[t - R.slot_t0] : -1;
  const bool out = UPDATE && (tho >= 0 || Io >= 0 || !prep);
  const int32_t ks = S.k, k0 = S.k0, p0 = S.p0;
  auto pair_of = [&](int32_t k) { return k * BS + tid + (k < k0 ? 0 : p0 - k0 * BS); };
  const uint32_t is_step = isn.si ? 8u : 0u, sg_step = sgn.si ? 8u : 0u, c_step = P.coef_si ? 8u : 0u;
  auto load = [&](int32_t q, WideInput<UNI>& in) __attribute__((always_inline)) {
    q = min(q, pairs - 1);
    const uint32_t j = 2 * static_cast<uint32_t>(q), j1 = min(j + 1, static_cast<uint32_t>(Nj - 1));
    if (UPDATE) in.code = at_offset(gbl(reinterpret_cast<const vuint2*>(S.junc_code)), 4 * j);
    in.ic[0] = at_offset(Icp, 8 * j);
    in.ic[1] = at_offset(Icp, 8 * j1);
    in.is[0] = stream_offset(isn.p, is_step * j);
    in.is[1] = stream_offset(isn.p, is_step * j1);
    if constexpr (!UNI) {
#pragma unroll
      for (int m = 0; m < 2; ++m) {
        const uint32_t i = m ? j1 : j;
        in.more[m][0] = at_offset(gbl(P.rc0), c_step * i);
        in.more[m][1] = at_offset(gbl(P.coef) + P.Nj, c_step * i);
        in.more[m][2] = at_offset(gbl(P.coef) + 2 * static_cast<int64_t>(P.Nj), c_step * i);
        in.more[m][3] = GAUSS ? at_offset(sgn.p, sg_step * i) : 0.0;
      }
    }
  };
  WideInput<UNI> in;
  load(pair_of(0), in);
#pragma unroll
  for (int v = 0; v < kWideGroups; ++v) {
#pragma unroll 1
    for (int32_t i = 0; i < 4; ++i) {
      const int32_t k = 4 * v + i;
      if (k >= ks) break;
      const WideInput<UNI> now = in;
      const int32_t q = pair_of(k);
      load(pair_of(k + 1), in);
      if (q < (k < k0 ? p0 : pairs)) {
        double z[2] = {0.0, 0.0}, xs[2], as[2], cs[2], us[2], ys[2];
        if constexpr (!UPDATE) {
          // the phases of the two steps before
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            const int32_t j = min(2 * q + m, Nj - 1);
            as[m] = ((t & 1) ? odd : even)[j];
            cs[m] = ((t & 1) ? even : odd)[j];
          }
        }
        if constexpr (GAUSS)
          normal_pair(R.seed, 2 * static_cast<uint32_t>(q), noise_col, static_cast<uint64_t>(t + 1), &z[0], &z[1]);
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          const double r0 = UNI ? rc0 : now.more[m][0];
          if constexpr (UPDATE) {
            ys[m] = coded_difference(Z, now.code[m]);
            as[m] = (ys[m] - state[v][4 * i + m]) * r0;
            cs[m] = state[v][4 * i + 2 + m];
          }
          double X = 0.0;
          if constexpr (GAUSS) X = (UNI ? sg0 : now.more[m][3] * sgn.amp) * z[m];
          X = __builtin_fma(-now.is[m], isn.amp, X);
          X = __builtin_fma(UNI ? c1 : now.more[m][1], as[m], X);
          X = __builtin_fma(UNI ? c2 : now.more[m][2], cs[m], X);
          xs[m] = __builtin_fma(now.ic[m], jja_sin(__builtin_fma(2.0, as[m], -cs[m])), X);
          us[m] = xs[m] * r0;
        }
        if (k < k0) {
          U[2 * q] = us[0];
          U[2 * q + 1] = us[1];
        }
#pragma unroll
        for (int m = 0; m < 2; ++m) {
          state[v][4 * i + m] = xs[m];
          state[v][4 * i + 2 + m] = as[m];
        }
        if (out) {
          const TermView ist = term_view(R.Is, Io >= 0, P.zero, w, t);
#pragma unroll
          for (int m = 0; m < 2; ++m) {
            const int32_t j = 2 * q + m;
            if (j >= Nj) break;  // an odd count's last junction has no partner
            if (tho >= 0) gblw(R.th_out)[static_cast<size_t>(tho) * stride + col + j] = as[m];
            if (Io >= 0) gblw(R.I_out)[static_cast<size_t>(Io) * stride + col + j] = ys[m] + term_at(ist, j);
            if (!prep) {
              ((t & 1) ? even : odd)[j] = cs[m];
              ((t & 1) ? odd : even)[j] = as[m];
            }
          }
        }
      }
    }
  }
}

// GAUSS: some problem has noise; UNI: the coefficients and noise amplitude of each
// are one value for all junctions.
template <bool GAUSS, bool UNI>
__global__ __launch_bounds__(kWideBlock) void evolve_wide_kernel(const DevProblem* __restrict__ probs,
                                                                 const jja_problem_run* __restrict__ runs,
                                                                 const WorkItem* __restrict__ work,
                                                                 const WideDev* __restrict__ tables, int32_t n_steps,
                                                                 int64_t step0) {
  extern __shared__ double lds[];
  constexpr int BS = kWideBlock;
  constexpr int NF = kWidePairs;   // face addresses a thread has at most
  WorkItem wi = work[blockIdx.x];
  wi.problem = __builtin_amdgcn_readfirstlane(wi.problem);
  wi.column = __builtin_amdgcn_readfirstlane(wi.column);
  const int64_t w = wi.column;
  const int32_t tid0 = threadIdx.x;
  LAS double* const Z = (LAS double*)lds;
  const int32_t C = probs[wi.problem].lat_cols;
  const int32_t part0 = tid0 / C;
  // part and mode of the thread in the tridiagonal systems
  const uint32_t home = static_cast<uint32_t>(part0) << 16 | static_cast<uint32_t>(tid0 - part0 * C);
  // row and column of the thread's first face address
  const uint32_t start = static_cast<uint32_t>(tid0 / tables[wi.problem].ld) << 16 |
                         static_cast<uint32_t>(tid0 % tables[wi.problem].ld);
  // the zero that codes name, and the row past the last that short parts read
  for (int32_t i = tid0; i < tables[wi.problem].lds; i += BS) Z[i] = 0.0;
  lds_barrier();

  // element 4 i + {0, 1, 2, 3} of group v: x of both members of pair slot 4 v + i,
  // then their phases of the step before. The loop over a group is not unrolled (the
  // elements are picked by register index): unrolled, the pass would be larger than
  // the instruction cache.
  vdouble16 state[kWideGroups];
  wide_pass<GAUSS, UNI, false>(probs[wi.problem], runs[wi.problem], tables[wi.problem], Z, state, w, tid0, true, step0 - 1);
  for (int32_t n = 0; n < n_steps; ++n) {
    const int64_t t = step0 + n;
    const int32_t again = wi.problem + opaque_zero();
    const DevProblem& P = probs[again];
    const jja_problem_run& R = runs[again];
    const WideDev& S = tables[again];
    const int32_t tid = opaque(tid0);
    const int32_t ld = S.ld, buf = S.buf, part = static_cast<int32_t>(home >> 16), mode = static_cast<int32_t>(home & 0xffffu);
    // face sums in two rounds, each with the junction values of one in LDS
    {
      uint32_t code[NF];
      double flux[NF];  // the second half is loaded when the first is used
      auto codes = [&](int which) __attribute__((always_inline)) {
        const GAS uint32_t* c = gbl(S.face_code) + which * buf;
#pragma unroll
        for (int b = 0; b < NF; ++b) code[b] = at_offset(c, 4 * static_cast<uint32_t>(min(tid + b * BS, buf - 1)));
      };
      codes(0);
      const TermView fv = term_view(R.f, !R.f.zero, P.zero, w, t);
      const double amp = kTwoPi * fv.amp;
      const uint32_t one = fv.si ? 0xffffffffu : 0u;
      // byte offsets of the faces' flux inputs, from one address of the thread to the next
      uint32_t at[NF];
      {
        int32_t c = static_cast<int32_t>(start & 0xffffu), id = static_cast<int32_t>(start >> 16) * S.f_row + c * S.f_col;
        const int32_t dr = BS / ld, dc = BS - dr * ld;
#pragma unroll
        for (int b = 0; b < NF; ++b) {
          at[b] = one & (8 * static_cast<uint32_t>(min(id, P.Nf - 1)));
          c += dc;
          id += dr * S.f_row + dc * S.f_col;
          const bool wrap = c >= ld;
          c -= wrap ? ld : 0;
          id += wrap ? S.f_row - ld * S.f_col : 0;
        }
      }
#pragma unroll
      for (int b = 0; b < NF / 2; ++b) flux[b] = at_offset(fv.p, at[b]);
      lds_barrier();
#pragma unroll
      for (int b = 0; b < NF; ++b)
        if (tid + b * BS < buf) Z[tid + b * BS] = coded_difference(Z, code[b]);
      codes(1);
      lds_barrier();
      LAS double* const U = Z + buf + 2;
      const int32_t pairs = (P.Nj + 1) >> 1, ks = S.k, k0 = S.k0, p0 = S.p0;
      const double rc0 = UNI ? rc0_at(P, 0) : 0.0;
#pragma unroll
      for (int k = 0; k < kWidePairs; ++k) {
        const int32_t q = (k - k0) * BS + tid;
        if (k >= k0 && k < ks && q < pairs - p0) {
          const int32_t j = 2 * (q + p0);
          U[2 * q] = state[k / 4][4 * (k % 4)] * (UNI ? rc0 : rc0_at(P, j));
          U[2 * q + 1] = state[k / 4][4 * (k % 4) + 1] * (UNI ? rc0 : rc0_at(P, min(j + 1, P.Nj - 1)));
        }
      }
      if (S.j0 & 1) {
        // the pair across the rounds: its second member, past the round's own
#pragma unroll
        for (int k = 0; k < kWidePairs; ++k)
          if (k == k0 - 1 && k * BS + tid == p0 - 1)
            U[2 * (pairs - p0)] = state[k / 4][4 * (k % 4) + 1] * (UNI ? rc0 : rc0_at(P, S.j0));
      }
      lds_barrier();
#pragma unroll
      for (int b = NF / 2; b < NF; ++b) flux[b] = at_offset(fv.p, at[b]);
#pragma unroll
      for (int b = 0; b < NF; ++b)
        if (tid + b * BS < buf)
          Z[tid + b * BS] = __builtin_fma(-amp, flux[b], Z[tid + b * BS] + coded_difference(Z, code[b]));
    }
    LAS double* const Y = Z + buf + 2;
    wide_transform(Z, Y, gbl(S.table), C, P.lat_rows, ld, tid);
    wide_tridiagonal(P, S, Y, Z, C, ld, part, mode);
    wide_transform(Y, Z, gbl(S.table), C, P.lat_rows, ld, tid);
    lds_barrier();
    wide_pass<GAUSS, UNI, true>(P, R, S, Z, state, w, tid, n + 1 < n_steps, t);
  }
}

}  // namespace

int64_t wide_lds_doubles(const WideDev& d, int32_t n_junctions) {
  const int64_t pairs = (static_cast<int64_t>(n_junctions) + 1) / 2;
  return d.buf + 2 + std::max<int64_t>({d.buf + (d.extra ? d.ld : 0), 2 * d.p0, 2 * (pairs - d.p0) + 1});
}

bool build_wide(const jja_problem_desc& desc, int64_t lds_bytes, WideHost* out) {
  const int32_t R = desc.lattice_rows, C = desc.lattice_cols, Nj = desc.n_junctions, Nf = desc.n_faces;
  const int32_t pairs = (Nj + 1) / 2;
  if (R < 2 || C < 8 || C > kWideBlock || pairs > kWidePairs * kWideBlock) return false;
  WideDev& d = out->d;
  d.parts = std::max(1, std::min({kWideBlock / C, R / 4, kWideParts}));
  d.base = R / d.parts;
  d.extra = R % d.parts;
  d.rows = d.base + (d.extra ? 1 : 0);
  if (d.rows > kWideRows) return false;
  // the first round ends before a junction that would be a face's second of a sign
  struct Face {
    int32_t j[2][2] = {{-1, -1}, {-1, -1}};  // [round][sign]
  };
  std::vector<Face> face(Nf);
  int32_t round = 0;
  d.j0 = Nj;
  for (int32_t j = 0; j < Nj; ++j) {
    const int32_t* c = desc.junc_code + 2 * j;
    if (c[0] >= 0 && c[1] >= 0 && ((c[0] ^ c[1]) & 1) == 0) return false;  // the junction's own code: one of each sign
    for (int32_t i = 0; i < 2; ++i) {
      if (c[i] < 0 || face[c[i] >> 1].j[round][c[i] & 1] < 0) continue;
      if (round) return false;
      round = 1;
      d.j0 = j;
    }
    for (int32_t i = 0; i < 2; ++i)
      if (c[i] >= 0) face[c[i] >> 1].j[round][c[i] & 1] = j;
  }
  d.p0 = (d.j0 + 1) / 2;
  d.k0 = (d.p0 + kWideBlock - 1) / kWideBlock;
  d.k = d.k0 + (pairs - d.p0 + kWideBlock - 1) / kWideBlock;
  if (d.k > kWidePairs) return false;
  // rows 4 doubles (mod 8) apart: the 16 rows of a product's operand, four elements
  // each, then lie in different banks
  const int32_t even = 2 * ((C + 1) / 2);
  d.ld = even + (12 - even % 8) % 8;
  d.buf = R * d.ld;
  if (8 * wide_lds_doubles(d, Nj) > lds_bytes) {
    d.ld = even;
    d.buf = R * d.ld;
  }
  if (8 * wide_lds_doubles(d, Nj) > lds_bytes || d.buf > kWidePairs * kWideBlock ||
      wide_lds_doubles(d, Nj) > 65535 || 4 * d.parts * C > d.buf)
    return false;
  d.lds = static_cast<int32_t>(wide_lds_doubles(d, Nj));
  const uint32_t zero = static_cast<uint32_t>(d.buf);
  // LDS index of junction j's value in its round: a pair across both rounds has its
  // second member after the second round's own
  auto value = [&](int32_t j, int32_t in_round) -> uint32_t {
    if (j < 0) return zero;
    const int32_t at = !in_round ? j : j < 2 * d.p0 ? 2 * (pairs - d.p0) : j - 2 * d.p0;
    return static_cast<uint32_t>(d.buf + 2 + at);
  };
  out->face_code.assign(2 * static_cast<size_t>(d.buf), zero | zero << 16);
  // face index of row r and column c: r * f_row + c * f_col
  d.f_row = R > 1 ? desc.face_of_pos[C] : 0;
  d.f_col = desc.face_of_pos[1];
  for (int32_t e = 0; e < Nf; ++e)
    if (desc.face_of_pos[e] != e / C * d.f_row + e % C * d.f_col) return false;
  for (int32_t e = 0; e < Nf; ++e) {
    const int32_t at = e / C * d.ld + e % C;
    for (int32_t r = 0; r < 2; ++r)
      out->face_code[static_cast<size_t>(r) * d.buf + at] = value(face[e].j[r][0], r) | value(face[e].j[r][1], r) << 16;
  }
  out->junc_code.assign(2 * static_cast<size_t>(pairs), zero | zero << 16);
  for (int32_t j = 0; j < Nj; ++j) {
    uint32_t at[2] = {zero, zero};
    for (int32_t i = 0; i < 2; ++i) {
      const int32_t c = desc.junc_code[2 * j + i];
      if (c >= 0) at[c & 1] = static_cast<uint32_t>(((c >> 1) / C) * d.ld + (c >> 1) % C);
    }
    out->junc_code[j] = at[0] | at[1] << 16;
  }
  std::vector<double> inv, spike, reduced;
  row_part_tables(R, C, d.parts, desc.lattice_g, desc.lattice_gc, &inv, &spike, &reduced);
  d.ends = (2 * d.parts + 3) / 4 * 4;
  out->reduced.assign(2 * static_cast<size_t>(d.parts) * d.ends * C, 0.0);
  for (int32_t e = 0; e < 2 * d.parts; ++e)
    std::copy_n(&reduced[static_cast<size_t>(e) * 2 * d.parts * C], 2 * static_cast<size_t>(d.parts) * C,
                &out->reduced[static_cast<size_t>(e) * d.ends * C]);
  const size_t table = static_cast<size_t>(kWideRows) * C;
  out->inv.assign(2 * table, 0.0);
  out->spike.assign(4 * table, 0.0);
  for (int32_t type = 0; type < 2; ++type) {
    const int32_t s = std::min(d.base + type, d.rows);
    for (int32_t l = 0; l < s; ++l)
      for (int32_t k = 0; k < C; ++k) {
        const size_t at = type * table + static_cast<size_t>(l) * C + k;
        out->inv[at] = inv[static_cast<size_t>(l) * C + k];
        out->spike[at] = spike[(static_cast<size_t>(type) * d.rows + l) * C + k];
        out->spike[2 * table + at] = spike[(static_cast<size_t>(type) * d.rows + s - 1 - l) * C + k];
      }
  }
  return true;
}

const void* wide_evolve_kernel(bool gauss, bool uniform) {
  if (gauss)
    return uniform ? reinterpret_cast<const void*>(evolve_wide_kernel<true, true>)
                   : reinterpret_cast<const void*>(evolve_wide_kernel<true, false>);
  return uniform ? reinterpret_cast<const void*>(evolve_wide_kernel<false, true>)
                 : reinterpret_cast<const void*>(evolve_wide_kernel<false, false>);
}
