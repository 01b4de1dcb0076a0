// jja_resident.h -- kernels that keep a column's whole state on chip
// (jja_resident.hip), as the launch code sees them.
#ifndef JJA_RESIDENT_H
#define JJA_RESIDENT_H

// Most threads of a workgroup, junction pairs a thread may keep in registers, face
// records (of up to four junctions) it then keeps per pair, and face records of the
// form that keeps the state in LDS.
constexpr int kResidentBlock = 512;
constexpr int kResidentPairs = 3;
constexpr int kResidentFaces = 2;
constexpr int kResidentRecords = 8;

// Kernel address for workgroups of `block_size` threads that keep `pairs`
// junction pairs each in registers (0: the state in LDS), or NULL when there is
// none. Arguments: those of evolve_kernel and adjoint_kernel.
const void* resident_evolve_kernel(int block_size, int pairs);
const void* resident_adjoint_kernel(int block_size, int pairs);

#endif  // JJA_RESIDENT_H
