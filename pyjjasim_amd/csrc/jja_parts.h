// jja_parts.h -- what a workgroup of a column worked in parts holds, as the plan and
// the kernels (jja_part_kernels.h) see it.
#ifndef JJA_PARTS_H
#define JJA_PARTS_H

#include <cstdint>

// Threads of a workgroup.
constexpr int kPartBlock = 512;

// Junctions and faces of every part (device pointers). A part has `pairs` slots for
// junction pairs and `faces` slots for faces; the kernels keep both in registers,
// slot k * kPartBlock + thread.
struct PartTables {
  int32_t parts, pairs, faces, pad_;
  const int32_t* pair;        // [parts][pairs]: pair * 16 + present bits + 4 * owner bits, or -1
  const uint32_t* pair_code;  // [parts][pairs][2]: two incidence codes of each member
  const uint32_t* face_code;  // [parts][faces][words]: codes of junction values, two to a word
  const uint32_t* face_at;    // [parts][faces]: address of the face, or 0xffffffff
  const int32_t* face_id;     // [parts][faces]: face index (flux input), or -1
  const int32_t* face_pos;    // [parts][faces]: solve position of a face whose gradient the part adds, or -1
};

#endif  // JJA_PARTS_H
