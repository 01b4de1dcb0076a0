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
//
// What bounds a step of few junctions a part is latency (one 100x100 column in 16 parts,
// 39,000 cycles: junction pass 9000, transforms 7000, recurrences 3000, meeting and
// reduced system 18,000, of which the other parts' rows alone take two accesses of about
// 4000 to the memory side of the caches); of large parts (256x256 in 16, 150,000 cycles)
// the junction pass 48,000, the transforms 40,000 and the meeting with the reduced
// system's four rows of coefficients a mode 35,000. Measured, us a step before (one
// workgroup, or 4 parts with column barriers for 256x256) and now: 100x100, one column 77,
// 16.1; 64x64, 32 columns 38, 11.1; 256x256, 16 columns 186, 66.5.
#include "jja_slab.h"

#include <algorithm>

#include "jja_part_kernels.h"
#include "jja_rowdst.h"
#include "jja_rowparts.h"

namespace {

// Rows 0 .. rows - 1 of src times the sine matrix into dst (rows of ld doubles, on
// the matrix cores as dst_product<false>; row tiles past the last row read it again
// and are not stored). The table lies in LDS, or in memory with four steps loaded
// ahead. row_transform, which large slabs take, is no better for a table in LDS (100x100
// in 16 slabs: 4400 cycles against 3600).
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

// An end row's value as another part published it.
__device__ __forceinline__ double end_row(const GAS double* at) {
  return __builtin_bit_cast(
      double, __hip_atomic_load(reinterpret_cast<unsigned long long*>(const_cast<double*>((const double*)at)),
                                __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// AHEAD: the reduced system's first coefficients and the responses are loaded before the
// wait for the other parts, and eight end rows at once after it. With nine pairs a thread
// (large lattices, 255 modes: four rows of 32 coefficients a mode) that shortens wait and
// reduced system from 48,000 to 33,000 cycles; with few modes the loads only delay the
// polls (one 100x100 column in 16 parts: 16.5 us a step against 17.6), and four end rows
// at a time with their coefficients are enough. A table in memory then also takes
// row_transform, which reads it once for a slab's 16 rows and the border rows (both
// transforms together 57,000 cycles before, 40,000 now); the kernels with few pairs keep
// their inputs in the registers that it needs.
template <bool AHEAD>
struct SlabSolver {
  using Dev = SlabDev;
  static constexpr int kFaceWords = 2;
  int32_t part, s, C, ld, parts;
  LAS double *in, *out, *u;       // face rows Z (both); junction values in the rows' transform Y
  LAS double* inv;                // pivots
  const LAS double* table;
  GAS double* ends;               // this column's [2][ends_rows][C]
  uint32_t* flags;                // this column's [parts][mode_waves]
  uint32_t wait_limit;
  int32_t* err;
  volatile LAS int32_t* stopped;

  __device__ __forceinline__ SlabSolver(const DevProblem& P, const SlabDev& S, int64_t column, int32_t part_, double* lds,
                                        int32_t* err_, uint32_t wait_limit_, int32_t tid, int32_t nt)
      : part(part_), s(S.base + (part_ < S.extra ? 1 : 0)), C(P.lat_cols), ld(S.ld), parts(S.parts),
        wait_limit(wait_limit_), err(err_) {
    in = out = (LAS double*)lds;
    u = in + S.buf;
    LAS double* next = u + max(S.buf, 2 * S.pairs);
    inv = next;
    if (S.inv_lds) next += S.rows * C;
    table = next;
    const int32_t entries = S.table_lds ? DstShape(C).entries() : 0;
    stopped = (volatile LAS int32_t*)(next + entries);
    ends = gblw(S.ends) + column * (2 * S.ends_rows * static_cast<int64_t>(C));
    flags = S.flags + column * (parts * S.mode_waves);
    for (int32_t i = tid; i < S.buf + max(S.buf, 2 * S.pairs); i += nt) in[i] = 0.0;
    if (S.inv_lds)
      for (int32_t i = tid; i < S.rows * C; i += nt) inv[i] = gbl(S.inv)[i];
    for (int32_t i = tid; i < entries; i += nt) next[i] = gbl(S.table)[i];
    if (tid == 0) *stopped = 0;
    __syncthreads();
  }

  struct Head {};
  __device__ __forceinline__ void head(const SlabDev&, int32_t, Head&) const {}
  __device__ __forceinline__ void solve(const DevProblem& P, const SlabDev& S, uint32_t seq, int32_t tid, int32_t nt,
                                        Head&) const;
};

// K^-1 of the column's face sums: in rows 1 .. s on entry, the solution in rows
// 0 .. s + 1 on exit (a neighbour's row below the first or above the last face row
// is zero). seq: the step's sequence number.
template <bool AHEAD>
__device__ __forceinline__ void SlabSolver<AHEAD>::solve(const DevProblem& P, const SlabDev& S, uint32_t seq, int32_t tid,
                                                  int32_t nt, Head&) const {
  constexpr int TB = 8;                // rows loaded together
  constexpr int RB = 4;                // end rows whose coefficients are loaded together
  const int32_t G = parts;
  LAS double *const Z = in, *const Y = u;
  if (S.table_lds)
    slab_transform<const LAS double*>(Z + ld, Y + ld, table, C, s, ld, tid, nt);
  else if constexpr (AHEAD)
    row_transform<false>(Z + ld, Y + ld, gbl(S.table), C, s, ld, tid, nt);
  else
    slab_transform<const GAS double*>(Z + ld, Y + ld, gbl(S.table), C, s, ld, tid, nt);
  lds_barrier();
  const int32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid & (kWave - 1);
  if (wave < S.mode_waves) {
    // two lanes a mode: both run the own block's recurrences (the same values), one
    // then takes the row below, the other the row above
    const int32_t k = min(tid >> 1, C - 1), side = tid & 1;
    const bool live = (tid >> 1) < C;
    const double g = P.lat_g;
    const GAS double* ginv = gbl(S.inv) + k;
    const LAS double* linv = inv + k;
    LAS double* y = Y + ld + k;
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
    const int64_t step = (seq & 1u) ? static_cast<int64_t>(S.ends_rows) * C : 0;
    GAS double* e = ends + step + k;
    if (live)
      __hip_atomic_store(reinterpret_cast<unsigned long long*>((double*)(e + (2 * part + side) * C)),
                         __builtin_bit_cast(unsigned long long, side ? last : x), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(kWaitVmem);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (lane == 0)
      __hip_atomic_store(flags + part * S.mode_waves + wave, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the reduced system's coefficients (zero past the last end row) and the responses
    const int32_t outer = side ? 2 * part + 2 : 2 * part - 1, own = 2 * part + side;
    const bool edge = outer < 0 || outer >= 2 * G;  // beyond the lattice: zero
    const int32_t E = S.ends_rows;
    const uint32_t at_outer = 8u * static_cast<uint32_t>((edge ? own : outer) * E * C + k);
    const uint32_t at_own = 8u * static_cast<uint32_t>(own * E * C + k);
    struct Chunk {
      double outer[RB], own[RB];
    } c[2];
    auto coefficients = [&](Chunk& to, int32_t i0) __attribute__((always_inline)) {
      i0 = min(i0, E - RB);
#pragma unroll
      for (int q = 0; q < RB; ++q) {
        to.outer[q] = at_offset(gbl(S.reduced) + (i0 + q) * C, at_outer);
        to.own[q] = at_offset(gbl(S.reduced) + (i0 + q) * C, at_own);
      }
    };
    const GAS double* V = gbl(S.spike) + (s > S.base ? static_cast<int64_t>(S.rows) * C : 0);
    double va[TB], vb[TB];
    auto responses = [&](int32_t l0) __attribute__((always_inline)) {
#pragma unroll
      for (int q = 0; q < TB; ++q) {
        const int32_t l = min(l0 + side + 2 * q, s - 1);
        va[q] = V[l * C + k];
        vb[q] = V[(s - 1 - l) * C + k];
      }
    };
    if constexpr (AHEAD) {
      coefficients(c[0], 0);
      coefficients(c[1], RB);
      responses(1);
    }
    if (!*stopped) {
      const uint32_t* f = flags + min(lane, G - 1) * S.mode_waves + wave;
      uint32_t spins = 0;
      while (true) {
        const uint32_t v = __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__all(static_cast<int32_t>(v - seq) >= 0)) break;
        if (++spins > wait_limit) {
          // gives up for the rest of the launch; a kernel after it (evolve_spoil_kernel) tells the host
          // and spoils the results
          *stopped = 1;
          __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
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
    double no = 0.0, nw = 0.0;
    if constexpr (AHEAD) {
      for (int32_t i0 = 0; i0 < E; i0 += 2 * RB) {
        double ev[2 * RB];
#pragma unroll
        for (int q = 0; q < 2 * RB; ++q) ev[q] = end_row(e + min(i0 + q, E - 1) * C);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          if (i0 + h * RB < E) {
#pragma unroll
            for (int q = 0; q < RB; ++q) {
              no = __builtin_fma(c[h].outer[q], ev[h * RB + q], no);
              nw = __builtin_fma(c[h].own[q], ev[h * RB + q], nw);
            }
            coefficients(c[h], i0 + (h + 2) * RB);
          }
        }
      }
    } else {
      const GAS double* ro = gbl(S.reduced) + static_cast<int64_t>(edge ? own : outer) * E * C + k;
      const GAS double* rw = gbl(S.reduced) + static_cast<int64_t>(own) * E * C + k;
      for (int32_t i0 = 0; i0 < E; i0 += RB) {
        double ev[RB], co[RB], cw[RB];
#pragma unroll
        for (int q = 0; q < RB; ++q) {
          ev[q] = end_row(e + (i0 + q) * C);
          co[q] = ro[(i0 + q) * C];
          cw[q] = rw[(i0 + q) * C];
        }
#pragma unroll
        for (int q = 0; q < RB; ++q) {
          no = __builtin_fma(co[q], ev[q], no);
          nw = __builtin_fma(cw[q], ev[q], nw);
        }
      }
      responses(1);
    }
    if (edge) no = 0.0;
    const double swapped = dpp_f64<0xB1, 0xf>(no);  // quad_perm [1, 0, 3, 2]: the mode's other lane
    const double below = side ? swapped : no, above = side ? no : swapped;
    for (int32_t l0 = 1; l0 + side < s - 1; l0 += 2 * TB) {
      double v[TB];
#pragma unroll
      for (int q = 0; q < TB; ++q) v[q] = y[min(l0 + side + 2 * q, s - 1) * ld];
#pragma unroll
      for (int q = 0; q < TB; ++q) {
        const int32_t l = l0 + side + 2 * q;
        if (l < s - 1) y[l * ld] = __builtin_fma(va[q], below, __builtin_fma(vb[q], above, v[q]));
      }
      if (l0 + 2 * TB < s - 1) responses(l0 + 2 * TB);
    }
    y[(side ? s - 1 : 0) * ld] = nw;
    Y[(side ? s + 1 : 0) * ld + k] = no;
  }
  if (AHEAD && !S.table_lds) {
    row_transform<true>(Y, Z, gbl(S.table), C, s + 2, ld, tid, nt);
  } else {
    lds_barrier();
    if (S.table_lds)
      slab_transform<const LAS double*>(Y, Z, table, C, s + 2, ld, tid, nt);
    else if constexpr (!AHEAD)
      slab_transform<const GAS double*>(Y, Z, gbl(S.table), C, s + 2, ld, tid, nt);
  }
  lds_barrier();
}

}  // namespace

int64_t slab_lds_doubles(const SlabDev& d, int32_t cols) {
  return static_cast<int64_t>(d.buf) + std::max(d.buf, 2 * d.pairs) + (d.inv_lds ? static_cast<int64_t>(d.rows) * cols : 0) +
         (d.table_lds ? DstShape(cols).entries() : 0) + 1;
}

namespace {

// The parts' junctions and faces and what LDS holds: everything but the tables.
bool cut_slabs(const jja_problem_desc& desc, int32_t parts, int64_t lds_bytes, SlabHost* out) {
  const int32_t R = desc.lattice_rows, C = desc.lattice_cols, Nj = desc.n_junctions, G = parts;
  // two rows a part: its first and its last; more columns, rows or junctions fit in no way
  if (R < 2 * G || C < 8 || G < 2 || 2 * C > kPartBlock || R / G > 32767 || Nj >= (1 << 27)) return false;
  SlabDev& d = out->d;
  d.parts = G;
  d.base = R / G;
  d.extra = R % G;
  d.rows = d.base + (d.extra ? 1 : 0);
  d.ld = DstShape(C).padded() + 4;
  d.buf = (d.rows + 2) * d.ld;
  d.mode_waves = (2 * C + 63) / 64;
  d.faces = d.rows * C;
  if (d.buf > 32767 || 64 * d.mode_waves > kPartBlock) return false;
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
  d.ends_rows = (2 * G + 3) / 4 * 4;
  if (2 * d.pairs > 32767 || std::max(d.pairs, d.faces) > kSlabPairs * kPartBlock) return false;
  // LDS: the pivots, then the sine table, where there is room
  d.inv_lds = d.table_lds = 0;
  if (8 * slab_lds_doubles(d, C) > lds_bytes) return false;
  d.inv_lds = 1;
  if (8 * slab_lds_doubles(d, C) > lds_bytes) d.inv_lds = 0;
  d.table_lds = 1;
  if (8 * slab_lds_doubles(d, C) > lds_bytes) d.table_lds = 0;
  out->pair.assign(static_cast<size_t>(G) * d.pairs, -1);
  out->pair_code.assign(2 * static_cast<size_t>(G) * d.pairs, 0xffffffffu);
  out->face_id.assign(static_cast<size_t>(G) * d.faces, -1);
  out->face_at.assign(static_cast<size_t>(G) * d.faces, 0xffffffffu);
  out->face_pos.assign(static_cast<size_t>(G) * d.faces, -1);
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
      out->face_pos[at] = r0 * C + e;
      out->face_at[at] = static_cast<uint32_t>((e / C + 1) * d.ld + e % C);
      out->face_id[at] = desc.face_of_pos[r0 * C + e];
      for (int32_t i = 0; i < 2; ++i)
        out->face_code[2 * at + i] = fcode[4 * static_cast<size_t>(e) + 2 * i] |
                                     static_cast<uint32_t>(fcode[4 * static_cast<size_t>(e) + 2 * i + 1]) << 16;
    }
  }
  return true;
}

}  // namespace

bool slabs_fit(const jja_problem_desc& desc, int32_t parts, int64_t lds_bytes) {
  SlabHost h;
  return cut_slabs(desc, parts, lds_bytes, &h);
}

bool build_slabs(const jja_problem_desc& desc, int32_t parts, int64_t lds_bytes, SlabHost* out) {
  if (!cut_slabs(desc, parts, lds_bytes, out)) return false;
  const int32_t R = desc.lattice_rows, C = desc.lattice_cols, G = parts;
  SlabDev& d = out->d;
  std::vector<double> reduced;
  row_part_tables(R, C, G, desc.lattice_g, desc.lattice_gc, &out->inv, &out->spike, &reduced);
  out->reduced.assign(2 * static_cast<size_t>(G) * d.ends_rows * C, 0.0);
  for (int32_t r = 0; r < 2 * G; ++r)
    std::copy_n(&reduced[2 * static_cast<size_t>(r) * G * C], 2 * static_cast<size_t>(G) * C,
                &out->reduced[static_cast<size_t>(r) * d.ends_rows * C]);
  return true;
}

const void* slab_evolve_kernel(int pairs) {
  if (pairs <= 1) return reinterpret_cast<const void*>(evolve_parts_kernel<SlabSolver<false>, 1>);
  if (pairs <= 2) return reinterpret_cast<const void*>(evolve_parts_kernel<SlabSolver<false>, 2>);
  if (pairs <= 3) return reinterpret_cast<const void*>(evolve_parts_kernel<SlabSolver<false>, 3>);
  if (pairs <= 5) return reinterpret_cast<const void*>(evolve_parts_kernel<SlabSolver<false>, 5>);
  return pairs <= kSlabPairs ? reinterpret_cast<const void*>(evolve_parts_kernel<SlabSolver<true>, kSlabPairs>) : nullptr;
}

const void* slab_adjoint_kernel(int pairs) {
  if (pairs <= 1) return reinterpret_cast<const void*>(adjoint_parts_kernel<SlabSolver<false>, 1>);
  if (pairs <= 2) return reinterpret_cast<const void*>(adjoint_parts_kernel<SlabSolver<false>, 2>);
  if (pairs <= 3) return reinterpret_cast<const void*>(adjoint_parts_kernel<SlabSolver<false>, 3>);
  if (pairs <= 5) return reinterpret_cast<const void*>(adjoint_parts_kernel<SlabSolver<false>, 5>);
  return pairs <= kSlabPairs ? reinterpret_cast<const void*>(adjoint_parts_kernel<SlabSolver<false>, kSlabPairs>) : nullptr;
}
