// jja_domain.h -- columns of any circuit worked as subdomains (jja_domain.hip), as
// the plan and the launch code see them.
#ifndef JJA_DOMAIN_H
#define JJA_DOMAIN_H

#include <cstdint>

#include "../../include/jja.h"
#include "jja_parts.h"

// Most junction pairs (and faces) a thread holds.
constexpr int kDomainPairs = 4;

// One problem's subdomains as the kernels see them (device pointers): jja_domains
// with the exchange buffers. A face's address is its place in the part's face
// vector; LDS holds the face sums, then the solution, then the separator faces'.
struct DomainDev : PartTables {
  int32_t n_gamma, sources, n_published, val_bytes;
  const int32_t* pub_ptr;         // [parts + 1]
  const int32_t* pub_at;          // [n_published]
  const int32_t* source;          // [n_gamma][sources]
  const jja_slice* solve_slices;
  const int32_t* wave_ptr;        // [parts][2][waves + 1]
  const int32_t* slice_rows;
  const double* ent_val;
  const void* ent_off;
  double* pub;                    // [columns][2][n_published]
  uint32_t* flags;                // [columns][parts][waves] sequence number a wave published last
};

// Doubles of dynamic LDS one workgroup takes.
inline int64_t domain_lds_doubles(const DomainDev& d) {
  return 2 * static_cast<int64_t>(d.faces) + d.n_gamma + 2 * static_cast<int64_t>(d.pairs) + 1;
}

// Kernels (workgroups of kPartBlock threads) whose threads hold at most `pairs`
// junction pairs and faces each, or NULL.
const void* domain_evolve_kernel(int pairs);
const void* domain_adjoint_kernel(int pairs);

#endif  // JJA_DOMAIN_H
