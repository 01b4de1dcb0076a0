// jja_rowdst.h -- sine transform of a few lattice rows in LDS on the matrix cores, for
// the kernels that keep row slabs on chip (jja_slab.hip).
#ifndef JJA_ROWDST_H
#define JJA_ROWDST_H

#include "jja_device.h"

namespace {

// The table's values of four steps are loaded together, a batch ahead of the products
// (and the next task's first ones before the last steps of a task): in memory they come
// from the L2, which answers in 1000 to 2000 cycles under load, and the matrix pipe works
// on a batch of two waves for 2000. The operands from LDS are loaded a step ahead.
constexpr int kDstBatch = 4;
struct DstBatch {
  double v[kDstBatch][2];
};
template <class F>
__device__ __forceinline__ void dst_fetch(F f, int32_t k, int32_t stored, DstBatch& b) {
#pragma unroll
  for (int u = 0; u < kDstBatch; ++u) {
    const int32_t at = 2 * min(k + u, stored - 1) * kWave;
    b.v[u][0] = f[at];
    b.v[u][1] = f[at + kWave];
  }
}

// Addresses of a lane's operands in each block of rows, from the row's start and end.
struct DstRows {
  const LAS double *up, *down;
};

// The products of one task: NB blocks of 16 rows and, TAIL, one of four rows (the
// 4x4x4 instruction, a quarter of the time; its operands and results lie in the lanes
// as those of the large one, by row lane / 16 of the result, lane % 4 of the operand).
// v holds the first batch and receives that of the next task.
template <int NB, bool TAIL, class F>
__device__ __forceinline__ void dst_products(F f, F next, int32_t stored, int32_t steps, DstRows (&in)[NB + TAIL],
                                             DstBatch& v, vdouble4 (&even)[2], vdouble4 (&odd)[2], double& te, double& to) {
  constexpr int U = kDstBatch, N = NB + TAIL;
  DstBatch vn;
  double x[N][2], nx[N][2];
  auto load = [&](int u, double (&o)[N][2]) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < N; ++b) {
      o[b][0] = in[b].up[4 * u];
      o[b][1] = in[b].down[-4 * u];
    }
  };
  auto step = [&](int u) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      even[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[b][0] + x[b][1], v.v[u][0], even[b], 0, 0, 0);
      odd[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(x[b][0] - x[b][1], v.v[u][1], odd[b], 0, 0, 0);
    }
    if constexpr (TAIL) {
      te = __builtin_amdgcn_mfma_f64_4x4x4f64(x[NB][0] + x[NB][1], v.v[u][0], te, 0, 0, 0);
      to = __builtin_amdgcn_mfma_f64_4x4x4f64(x[NB][0] - x[NB][1], v.v[u][1], to, 0, 0, 0);
    }
  };
  load(0, x);
  int32_t k = 0;
  for (; k + U <= steps; k += U) {
    const bool more = k + U < steps;
    dst_fetch(more ? f : next, more ? k + U : 0, stored, vn);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (u + 1 < U) {
        load(u + 1, nx);
      } else {
        const int32_t on = more ? 4 * U : 0;
#pragma unroll
        for (int b = 0; b < N; ++b) {
          in[b].up += on;
          in[b].down -= on;
        }
        load(0, nx);
      }
      __builtin_amdgcn_sched_barrier(0);
      step(u);
#pragma unroll
      for (int b = 0; b < N; ++b) {
        x[b][0] = nx[b][0];
        x[b][1] = nx[b][1];
      }
    }
    v = vn;
  }
  if (k < steps) {
    dst_fetch(next, 0, stored, vn);
#pragma unroll
    for (int u = 0; u < U - 1; ++u)
      if (k + u < steps) {
        if (u) load(u, x);
        step(u);
      }
    v = vn;
  }
}

// Rows of src times the sine matrix into dst (rows of ld doubles; BARRIER: after a
// barrier, with the table's first values loaded before it). A task is one block of 16
// modes of each parity for one or two blocks of 16 rows, whose products share the
// table's values. Up to four rows past the last block go with it where tasks have one
// block, and are tasks of their own where they have two (three blocks' operands at once
// take too many registers).
template <bool BARRIER, class F>
__device__ __forceinline__ void row_transform(const LAS double* src, LAS double* dst, F table, int32_t C, int32_t rows,
                                              int32_t ld, int32_t tid, int32_t nt) {
  const DstShape D(C);
  const int lane = tid & (kWave - 1), lr = lane & 15, lk = lane >> 4;
  const int32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), NW = nt / kWave;
  const int32_t steps = (D.h + 3) >> 2, over = rows & 15;
  const int32_t blocks = (rows >> 4) + (over > 4 ? 1 : 0);
  const bool tail = over > 0 && over <= 4;
  const int32_t each = D.pairs * ((blocks + 1) >> 1) >= NW ? 2 : 1;
  const bool join = tail && each == 1 && blocks > 0;
  const int32_t full = (blocks + each - 1) / each, tasks = D.pairs * (full + (tail && !join ? 1 : 0));
  int32_t mb = wave, group = 0;
  auto settle = [&]() {
    while (mb >= D.pairs) {
      mb -= D.pairs;
      ++group;
    }
  };
  settle();
  F f = table + mb * D.steps * 2 * kWave + lane;
  DstBatch v;
  dst_fetch(f, 0, D.steps, v);
  if constexpr (BARRIER) lds_barrier();
  for (int32_t task = wave; task < tasks; task += NW) {
    const int32_t mine = mb, first = group * each, row = 16 * first;
    const int32_t nb = max(min(each, blocks - first), 0);
    const bool with = nb == 0 || (join && group == full - 1);
    mb += NW;
    settle();
    F next = table + mb * D.steps * 2 * kWave + lane;
    auto rows_at = [&](int32_t r) {
      const int32_t at = min(r, rows - 1) * ld;
      return DstRows{src + at + lk, src + at + (C - 1 - lk)};
    };
    vdouble4 even[2], odd[2];
    even[0] = even[1] = odd[0] = odd[1] = vdouble4{0.0, 0.0, 0.0, 0.0};
    double te = 0.0, to = 0.0;
    if (nb == 2) {
      DstRows in[2] = {rows_at(row + lr), rows_at(row + 16 + lr)};
      dst_products<2, false, F>(f, next, D.steps, steps, in, v, even, odd, te, to);
    } else if (nb == 1 && !with) {
      DstRows in[1] = {rows_at(row + lr)};
      dst_products<1, false, F>(f, next, D.steps, steps, in, v, even, odd, te, to);
    } else {
      const DstRows t = rows_at(16 * blocks + (lane & 3));
      if (nb == 1) {
        DstRows in[2] = {rows_at(row + lr), t};
        dst_products<1, true, F>(f, next, D.steps, steps, in, v, even, odd, te, to);
      } else {
        DstRows in[1] = {t};
        dst_products<0, true, F>(f, next, D.steps, steps, in, v, even, odd, te, to);
      }
    }
    f = next;
    if (16 * mine + lr < D.h) {
      LAS double* d = dst + 2 * (16 * mine + lr);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int32_t o = row + lk + 4 * r;
        if (nb >= 1 && o < rows) *reinterpret_cast<LAS vdouble2*>(d + o * ld) = vdouble2{even[0][r], odd[0][r]};
        if (nb == 2 && o + 16 < rows) *reinterpret_cast<LAS vdouble2*>(d + (o + 16) * ld) = vdouble2{even[1][r], odd[1][r]};
      }
      const int32_t o = 16 * blocks + lk;
      if (with && o < rows) *reinterpret_cast<LAS vdouble2*>(d + o * ld) = vdouble2{te, to};
    }
  }
}

}  // namespace

#endif  // JJA_ROWDST_H
