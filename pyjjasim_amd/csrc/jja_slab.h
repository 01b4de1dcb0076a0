// jja_slab.h -- lattice columns cut into row slabs (jja_slab.hip), as the plan and
// the launch code see them.
#ifndef JJA_SLAB_H
#define JJA_SLAB_H

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/jja.h"
#include "jja_parts.h"

// Most junction pairs a thread holds.
constexpr int kSlabPairs = 9;

// One problem's slabs as the kernels see them (device pointers). Part p works on
// the face rows r0 = p * base + min(p, extra) .. r0 + s - 1, s = base + (p < extra),
// and on every junction one of them touches; its local rows are 0 (the row below),
// 1 .. s and s + 1 (the row above), each of ld doubles.
struct SlabDev : PartTables {
  int32_t base, extra, rows;             // rows: the most rows a part has
  int32_t ld, buf;                       // doubles per local row, doubles of one local face array
  int32_t table_lds;                     // the sine table lies in LDS (else it is read from memory)
  int32_t mode_waves;                    // waves that hold the modes (two lanes each)
  int32_t inv_lds;                       // the pivots lie in LDS
  int32_t ends_rows;                     // 2 parts rounded up to a multiple of four
  const double* table;                   // sine table of C modes (DstShape)
  const double* inv;                     // [rows][C] inverse pivots of a part's own block
  const double* spike;                   // [2][rows][C]: response to the row below, parts of base and base + 1 rows
  const double* reduced;                 // [2 parts][ends_rows][C]: first and last rows of the parts from their own blocks'
  double* ends;                          // [columns][2][ends_rows][C] end rows of a step, two of a part
  uint32_t* flags;                       // [columns][parts][mode_waves] sequence number of the last end rows
};

// Host arrays of the same, built from a descriptor.
struct SlabHost {
  SlabDev d{};
  std::vector<int32_t> pair, face_id, face_pos;
  std::vector<uint32_t> pair_code, face_code, face_at;
  std::vector<double> inv, spike, reduced;
};

// Doubles of dynamic LDS one workgroup of a slab launch takes.
int64_t slab_lds_doubles(const SlabDev& d, int32_t cols);

// Whether the lattice problem can be cut into `parts` slabs: every junction joins
// neighbours, no face has more than four, the slabs fit in LDS, a thread's registers and
// local indices. build_slabs cuts it and makes the tables.
bool slabs_fit(const jja_problem_desc& desc, int32_t parts, int64_t lds_bytes);
bool build_slabs(const jja_problem_desc& desc, int32_t parts, int64_t lds_bytes, SlabHost* out);

// Kernels (workgroups of kPartBlock threads) whose threads hold at most `pairs`
// junction pairs each, or NULL.
const void* slab_evolve_kernel(int pairs);
const void* slab_adjoint_kernel(int pairs);

#endif  // JJA_SLAB_H
