// jja_wide.h -- large lattice columns whose junctions stay in the registers of one
// workgroup (jja_wide.hip), as the plan and the launch code see them.
#ifndef JJA_WIDE_H
#define JJA_WIDE_H

#include <cstdint>
#include <vector>

#include "../../include/jja.h"

// Threads of a workgroup, and the junction pairs each can hold: four to a group.
constexpr int kWideBlock = 512;
constexpr int kWideGroups = 5;
constexpr int kWidePairs = 4 * kWideGroups;

// Most rows a thread solves of a mode's tridiagonal system, and parts of a mode.
constexpr int kWideRows = 20;
constexpr int kWideParts = 16;

// One problem as the kernel sees it (device pointers). LDS holds the face vector
// (rows of ld doubles, buf in all), two doubles of zero, then the junction values of
// one round of the face sums or the other copy of the face vector. Junctions below j0
// form the first round, the others the second; a face has at most one of each sign in
// each. Pair slots k * kWideBlock + thread: k < k0 for the pairs that start below j0,
// then the others. Codes are two 16-bit LDS indices of doubles (added, subtracted; the
// zero where there is none).
struct WideDev {
  int32_t j0, p0, k0, k;             // p0 = ceil(j0 / 2) pairs in the first k0 of k slots a thread
  int32_t ld, buf, lds;              // lds: doubles of LDS in all
  int32_t parts, base, extra;        // row parts of the modes' recurrences: base rows, the first `extra` one more
  int32_t rows;                      // the most rows a part has (at most kWideRows)
  const uint32_t* junc_code;         // [2 pairs]: the two faces
  const uint32_t* face_code;         // [2][buf]: a round's two junctions, by face address
  const double* table;               // sine table of C modes (DstShape)
  const double* inv;                 // [2][kWideRows][C] inverse pivots of a part's own block, parts of base and
                                     // base + 1 rows
  const double* spike;               // [2][2][kWideRows][C] responses to the row below and the row above, likewise
  int32_t ends;                      // 2 parts rounded up to a multiple of four
  int32_t f_row, f_col;              // face index of row r and column c: r * f_row + c * f_col
  const double* reduced;             // [2 parts][ends][C] first and last rows of the parts from their own blocks'
};

struct WideHost {
  WideDev d{};
  std::vector<uint32_t> junc_code, face_code;
  std::vector<double> inv, spike, reduced;
};

// Dynamic LDS doubles of a workgroup.
int64_t wide_lds_doubles(const WideDev& d, int32_t n_junctions);

// The tables of a lattice problem, or false when it does not fit this form.
bool build_wide(const jja_problem_desc& desc, int64_t lds_bytes, WideHost* out);

// The kernel for problems some of which have noise (gauss), all with one value for all
// junctions of each coefficient and of the noise amplitude (uniform) or not.
const void* wide_evolve_kernel(bool gauss, bool uniform);

#endif  // JJA_WIDE_H
