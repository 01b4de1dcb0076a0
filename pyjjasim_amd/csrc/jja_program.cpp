// Wave programs of subdomains from phases given as rows (host code; domain_plan.py).
//
// The records are those of the solve programs in solver_plan.py with 2-byte indices:
// rows of a phase with the same lanes per row go, longest first, into chains of 64 / G
// rows, chains to the least-loaded wave, longest first. A plan of 32 parts has 64
// programs of some 30,000 entries each; forming them row by row here takes a tenth of
// what as many rounds of small array operations took in Python (60x60 honeycomb array:
// 175 ms of a plan of 285).

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <functional>
#include <new>
#include <queue>
#include <utility>
#include <vector>

#include "../../include/jja.h"

namespace {

constexpr int32_t kLanes = 64, kIter = 8;

struct Chain {
  int32_t g, rows, records, n_iter;
  int64_t first, rowbase;  // record number, row slot
};

struct Input {
  const int64_t* phase_ptr;
  const int32_t* flags;
  const int32_t* rows;
  const int64_t* row_ptr;
  const int32_t* idx;
  const double* val;
};

struct Output {
  jja_slice* records;
  double* ent_val;
  uint16_t* ent_off;
  int32_t* slice_rows;
};

// Chains of a phase; the data of its records and their row slots when `out` is given.
void phase_chains(const Input& in, int32_t phase, int64_t& n_rec, int64_t& n_row, const Output* out,
                  std::vector<Chain>& chains) {
  const int64_t r0 = in.phase_ptr[phase], r1 = in.phase_ptr[phase + 1];
  auto length = [&](int64_t r) { return in.row_ptr[r + 1] - in.row_ptr[r]; };
  std::vector<int64_t> by_lanes[7];
  for (int64_t r = r0; r < r1; ++r) {
    const int64_t need = std::max<int64_t>(1, (length(r) + kIter - 1) / kIter);
    int32_t lg = 0;
    while ((int64_t{1} << lg) < need && lg < 6) ++lg;
    by_lanes[lg].push_back(r);
  }
  chains.clear();
  for (int32_t lg = 0; lg < 7; ++lg) {
    std::vector<int64_t>& sel = by_lanes[lg];
    std::stable_sort(sel.begin(), sel.end(), [&](int64_t a, int64_t b) { return length(a) > length(b); });
    const int32_t g = 1 << lg, per = kLanes / g;
    for (size_t s = 0; s < sel.size(); s += per) {
      Chain c;
      c.g = g;
      c.rows = static_cast<int32_t>(std::min<size_t>(per, sel.size() - s));
      c.n_iter = static_cast<int32_t>((length(sel[s]) + g - 1) / g);  // the longest row's
      c.records = std::max(1, (c.n_iter + kIter - 1) / kIter);
      c.first = n_rec;
      c.rowbase = n_row;
      n_rec += c.records;
      n_row += per;
      chains.push_back(c);
      if (!out) continue;
      for (int32_t i = 0; i < per; ++i) {
        const bool row = i < c.rows;
        out->slice_rows[c.rowbase + i] = row ? in.rows[sel[s + i]] : -1;
        if (!row) continue;
        const int64_t e0 = in.row_ptr[sel[s + i]], n = length(sel[s + i]);
        for (int64_t e = 0; e < n; ++e) {
          const int64_t k = e / g, rec = c.first + k / kIter, it = k % kIter, lane = i * g + e % g;
          out->ent_val[512 * rec + (it / 2) * 128 + 2 * lane + it % 2] = in.val[e0 + e];
          out->ent_off[512 * rec + 8 * lane + it] = static_cast<uint16_t>(in.idx[e0 + e]);
        }
      }
    }
  }
}

}  // namespace

extern "C" int jja_domain_programs(int32_t n_programs, int32_t waves, const int32_t* program_ptr, const int64_t* phase_ptr,
                                   const int32_t* flags, const int32_t* rows, const int64_t* row_ptr, const int32_t* idx,
                                   const double* val, int64_t* sizes, jja_slice* records, int32_t* wave_ptr,
                                   double* ent_val, uint16_t* ent_off, int32_t* slice_rows) {
  if (n_programs < 0 || waves < 1 || !program_ptr || !phase_ptr || !flags || !rows || !row_ptr || !idx || !val || !sizes)
    return JJA_EINVAL;
  const bool fill = records != nullptr;
  if (fill && (!wave_ptr || !ent_val || !ent_off || !slice_rows)) return JJA_EINVAL;
  const Input in{phase_ptr, flags, rows, row_ptr, idx, val};
  const Output out{records, ent_val, ent_off, slice_rows};
  try {
    if (fill) {
      std::fill_n(ent_val, sizes[1], 0.0);
      std::fill_n(ent_off, sizes[1], uint16_t{0});
      std::fill_n(slice_rows, kLanes, -1);
    }
    const jja_slice noop{0, 0, 0, 0, 0, 1};
    int64_t n_data = 1, n_row = kLanes, n_out = 0;  // block 0 and the first row slots: the no-op's
    std::vector<Chain> chains;
    std::vector<int32_t> order;
    std::vector<std::vector<jja_slice>> program(waves);
    for (int32_t p = 0; p < n_programs; ++p) {
      for (auto& w : program) w.clear();
      for (int32_t ph = program_ptr[p]; ph < program_ptr[p + 1]; ++ph) {
        phase_chains(in, ph, n_data, n_row, fill ? &out : nullptr, chains);
        order.resize(chains.size());
        for (size_t i = 0; i < order.size(); ++i) order[i] = static_cast<int32_t>(i);
        std::stable_sort(order.begin(), order.end(), [&](int32_t a, int32_t b) { return chains[a].records > chains[b].records; });
        using Load = std::pair<int64_t, int32_t>;
        std::priority_queue<Load, std::vector<Load>, std::greater<Load>> loads;
        std::vector<size_t> start(waves);
        for (int32_t w = 0; w < waves; ++w) {
          loads.push({0, w});
          start[w] = program[w].size();
        }
        for (int32_t i : order) {
          const Chain& c = chains[i];
          const Load least = loads.top();
          loads.pop();
          loads.push({least.first + c.records, least.second});
          for (int32_t k = 0; k < c.records; ++k) {
            const int64_t base = 512 * (c.first + k);
            const int32_t fl = c.g | flags[ph] | (c.rows << 16) | (k == c.records - 1 ? JJA_SLICE_FINISH : 0);
            program[least.second].push_back(
                {base, base, static_cast<int32_t>(c.rowbase), 0, std::min(kIter, c.n_iter - k * kIter), fl});
          }
        }
        for (int32_t w = 0; w < waves; ++w) {
          if (program[w].size() == start[w]) program[w].push_back(noop);
          program[w].back().flags |= JJA_SLICE_BARRIER;
        }
      }
      for (int32_t w = 0; w < waves; ++w) {
        // the kernel runs records in threes and loads four more ahead
        std::vector<jja_slice>& r = program[w];
        r.insert(r.end(), (3 - r.size() % 3) % 3 + 4, noop);
        if (fill) {
          wave_ptr[static_cast<int64_t>(p) * (waves + 1) + w] = static_cast<int32_t>(n_out);
          std::copy(r.begin(), r.end(), records + n_out);
        }
        n_out += static_cast<int64_t>(r.size());
      }
      if (fill) wave_ptr[static_cast<int64_t>(p) * (waves + 1) + waves] = static_cast<int32_t>(n_out);
    }
    sizes[0] = n_out;
    sizes[1] = 512 * n_data;
    sizes[2] = n_row;
  } catch (const std::bad_alloc&) {
    return JJA_ENOMEM;
  }
  return JJA_OK;
}
