// jja_device.h -- device code of the step kernels: the problem as the device
// sees it, the face stores, the solvers of the face system, the face phase, the
// junction pass and the adjoint step. Included by the .hip files that define
// kernels.
#ifndef JJA_DEVICE_H
#define JJA_DEVICE_H

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdint>
#include <type_traits>

#include "../../include/jja.h"
#include "jja_math.h"

namespace {


constexpr double kTwoPi = 6.283185307179586;  // 2 * np.pi
constexpr int kMaxIter = 8;                   // entries per lane and solve record
constexpr int kFaceIter = 4;                  // junction codes per thread and face record
constexpr int kFaceGroup = 4;                 // face records whose loads are issued together
constexpr int kWave = 64;                     // lanes of a wavefront (solve records are per wave)
// buffer resource word 3 for gfx9-family raw buffers (no format conversion),
// and a byte offset beyond any resource range (ranges stay below 2^31)
constexpr int kBufferWord3 = 0x00020000;
constexpr uint32_t kOutOfRange = 0x80000000u;

// Pointers read out of the descriptor structs are generic; casting them to the
// global (1) or constant (4) address space lets the compiler use global and
// scalar loads instead of flat ones, which would also stall on LDS traffic.
#define GAS __attribute__((address_space(1)))
#define CAS __attribute__((address_space(4)))
#define LAS __attribute__((address_space(3)))
template <typename T>
__device__ __forceinline__ const GAS T* gbl(const T* p) {
  return (const GAS T*)p;
}
template <typename T>
__device__ __forceinline__ GAS T* gblw(T* p) {
  return (GAS T*)p;
}

typedef double vdouble2 __attribute__((ext_vector_type(2)));
typedef double vdouble4 __attribute__((ext_vector_type(4)));
typedef uint32_t vuint2 __attribute__((ext_vector_type(2)));
typedef uint32_t vuint4 __attribute__((ext_vector_type(4)));
typedef int32_t vint2 __attribute__((ext_vector_type(2)));

struct RecWords {
  vuint4 a, b;
};
static_assert(sizeof(RecWords) == sizeof(jja_slice), "record layout");

// Uniform load of one program record through the scalar cache.
__device__ __forceinline__ jja_slice load_rec(const jja_slice* prog, int32_t k) {
  const CAS vuint4* q = (const CAS vuint4*)(prog + k);
  RecWords w;
  w.a = q[0];
  w.b = q[1];
  return __builtin_bit_cast(jja_slice, w);
}

// Device-resident description of one circuit (all pointers device memory).
struct DevProblem {
  int32_t Nj, Nf, sw, BS;
  int32_t n_face_slices, n_solve_slices, max_stage_rows, copy_rows;
  int32_t index_bytes;
  int32_t val_bytes;        // bytes of ent_val (below 2^31: the solve reads it through a buffer resource)
  const double* Ic;
  const double* Rv;
  const double* coef;
  const int32_t* junc_code;
  const int32_t* face_of_pos;
  const jja_slice* face_slices;
  const jja_slice* solve_slices;
  const int32_t* face_code;
  const int32_t* slice_rows;
  const double* ent_val;
  const void* ent_off;      // LDS indices: uint16 (face store in LDS) or uint32 (in global memory)
  const int32_t* wave_ptr;  // [BS/64 + 1]
  const double* zero;       // 8 zero doubles: absent input terms read here
  const int32_t* face_fid;  // [n_slice_rows]: face index of a face record's row slot, or -1
  int32_t parts;            // workgroups per column (1, or more with a global face store)
  int32_t coef_si;          // junction stride of coef: 1, or 0 when every row is one value
  const double* rc0;        // [Nj] 1 / c0 (stride coef_si)
  int32_t cpr_terms;        // 0: Ic sin(arg); else Ic * sum_k cpr_coef[k] sin((k+1) arg)
  double cpr_coef[JJA_CPR_MAX_TERMS];
  // lattice solve (lat_rows 0: the staged factor program solves K)
  int32_t lat_rows, lat_cols;  // R, C: faces at positions r*C + c
  int32_t lat_es, lat_cp;      // folded row length ES (even) and sine-table row stride CP
  int32_t lat_ef;              // folded rows stored per row: ES (LDS store), ES rounded up to 4 (global)
  int32_t lat_mp, lat_bp;      // split column: modes per part and blocks per mode of the part-local
                               // tridiagonal solve in LDS (lat_mp 0: the column-wide one)
  int32_t lat_tile;            // both sides at most 16: one wave solves (solve_lattice_tile)
  int64_t lat_t0;              // store offset of the folded rows (even: 16-byte loads)
  const double* lat_sine;      // [ES][CP]
  const double* lat_sine_p;    // [ES][2][CP/2]: the same table, even and odd modes apart (matrix-core B operands)
  const double* lat_inv;       // [R][CP] inverse Thomas pivots
  double lat_g;
  // LDS store of a lattice whose padded form fits (lat_ld 0: it does not): two
  // copies of the face vector with rows of lat_ld doubles, the second at
  // lat_buf, then the sine tables of both sides at lat_tab (DstShape)
  int32_t lat_ld, lat_buf, lat_tab;
  int32_t store_doubles;       // LDS store: doubles a column's store takes
  const double* lat_table;     // the sine tables (C's, then R's unless R == C); lat_tile: TileShape's
  const double* lat_lam;       // [padded rows][lat_ld] inverse eigenvalues, 0 in the padding
  const int32_t* face_addr;    // [n_slice_rows]: store address of a face record's row slot
};

// The sine matrix of n modes as operands of v_mfma_f64_16x16x4f64: modes of one
// parity in blocks of 16, the folded index i in steps of 4 (an even count). Lane l
// of (pair of blocks b, step k, parity p) holds S[4k + l/16][2 (16 b + l%16) + p]
// at ((b * steps + k) * 2 + p) * 64 + l, 0 past the matrix; the middle element of
// an odd n, which the fold adds to itself, is halved.
struct DstShape {
  int32_t n, h, pairs, steps;
  __host__ __device__ __forceinline__ explicit DstShape(int32_t modes)
      : n(modes), h((modes + 1) >> 1), pairs((h + 15) >> 4), steps((((h + 3) >> 2) + 1) & ~1) {}
  __host__ __device__ __forceinline__ int32_t entries() const { return pairs * steps * 2 * 64; }
  // rows or columns that outputs of all blocks take
  __host__ __device__ __forceinline__ int32_t padded() const { return 32 * pairs; }
};

// Tables of a lattice of at most 16 by 16 faces in LDS: the sine matrices of C and R
// modes as operands of four steps, lane l of step s S[4 s + l / 16][l % 16], and the
// inverse eigenvalues as results, register r of lane l row l / 16 + 4 r, column l % 16;
// zero past the lattice. Rows of 20 doubles put the 16 rows of an operand on all banks.
struct TileShape {
  static constexpr int32_t kSide = 16, kLd = 20, kTable = 256;
};

// Store address of solve position q (an LDS store; the global one is linear).
__device__ __forceinline__ int32_t store_address(const DevProblem& P, int32_t q) {
  if (!P.lat_ld) return q;
  const int32_t r = q / P.lat_cols;
  return r * P.lat_ld + (q - r * P.lat_cols);
}

// The current-phase relation's sum at one argument: sin(arg) for the default
// relation, else sum_k a_k sin((k+1) arg) accumulated in ascending k (each
// (k+1) arg formed as one product, as numpy forms k * theta).
__device__ __forceinline__ double cpr_sum(const DevProblem& P, double arg) {
  if (P.cpr_terms == 0) return jja_sin(arg);
  double acc = P.cpr_coef[0] * jja_sin(arg);
  for (int k = 1; k < P.cpr_terms; ++k) acc = acc + P.cpr_coef[k] * jja_sin(static_cast<double>(k + 1) * arg);
  return acc;
}

// Stencil coefficient k of junction j (an identical value for every junction
// is read from one address).
__device__ __forceinline__ double coef_at(const DevProblem& P, int k, int32_t j) {
  return gbl(P.coef)[static_cast<int64_t>(k) * P.Nj + static_cast<int64_t>(j) * P.coef_si];
}
// 1 / c0 of junction j: the step divides by c0 as a product with its
// reciprocal (within one rounding of the quotient)
__device__ __forceinline__ double rc0_at(const DevProblem& P, int32_t j) {
  return gbl(P.rc0)[static_cast<int64_t>(j) * P.coef_si];
}

// A value the compiler must assume changed: what is computed from it inside a loop
// is then formed there instead of being hoisted into registers that live through
// the whole loop (addresses of every array and constants spill otherwise).
__device__ __forceinline__ int32_t opaque(int32_t v) {
  __asm__ volatile("" : "+v"(v));
  return v;
}
// The same for a wave-uniform value: a zero to add to an index.
__device__ __forceinline__ int32_t opaque_zero() {
  int32_t z = 0;
  __asm__ volatile("" : "+s"(z));
  return z;
}

// A value at a byte offset from a wave-uniform base.
template <class T>
__device__ __forceinline__ T at_offset(const GAS T* base, uint32_t bytes) {
  return *reinterpret_cast<const GAS T*>(reinterpret_cast<const GAS char*>(base) + bytes);
}

// 16-bit incidence codes (2 * address + sign, 0xffff empty) of the kernels that
// keep them in registers, two to a word: +-v by the sign bit, 0 for an empty slot
__device__ __forceinline__ double signed_value(double v, uint32_t code) {
  const long long b = __builtin_bit_cast(long long, v) ^ (static_cast<long long>(code & 1u) << 63);
  return code == 0xffffu ? 0.0 : __builtin_bit_cast(double, b);
}
__device__ __forceinline__ uint32_t code_address(uint32_t code) { return code == 0xffffu ? 0u : code >> 1; }
__device__ __forceinline__ uint32_t pack_codes(int32_t a, int32_t b) {
  return static_cast<uint32_t>(a & 0xffff) | (static_cast<uint32_t>(b & 0xffff) << 16);
}

struct WorkItem {
  int32_t problem;
  int32_t column;  // column (times the problem's parts, plus the part, in a split launch)
  int32_t slot;    // the column's barrier counter in a split launch
};

// Workgroup barrier that orders LDS traffic only: global loads in flight (the
// prefetched solve entries) stay in flight across it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Philox4x32-10 (Salmon et al., SC'11) + Box-Muller for the junction pair
// (j, j+1), j even; counter (j>>1, w, step, 0), key = seed.
__device__ __forceinline__ void normal_pair(uint64_t seed, uint32_t j, uint32_t w, uint64_t step,
                                            double* z0, double* z1) {
  uint32_t c0 = j >> 1, c1 = w, c2 = static_cast<uint32_t>(step), c3 = 0u;
  uint32_t k0 = static_cast<uint32_t>(seed), k1 = static_cast<uint32_t>(seed >> 32);
  // an empty statement that the compiler must assume changes the key: the
  // round keys are then formed here (two scalar adds per round) instead of
  // being hoisted out of the junction loop as 20 live scalar registers, which
  // spilled to vector lanes and cost 22 v_readlane per pair
  __asm__ volatile("" : "+s"(k0), "+s"(k1));
#pragma unroll
  for (int r = 0; r < 10; ++r) {
    const uint64_t p0 = static_cast<uint64_t>(0xD2511F53u) * c0;
    const uint64_t p1 = static_cast<uint64_t>(0xCD9E8D57u) * c2;
    // a ^ b ^ c in one instruction
    c0 = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(p1 >> 32), c1, k0, 0x96);
    c2 = __builtin_amdgcn_bitop3_b32(static_cast<uint32_t>(p0 >> 32), c3, k1, 0x96);
    c1 = static_cast<uint32_t>(p1);
    c3 = static_cast<uint32_t>(p0);
    k0 += 0x9E3779B9u;
    k1 += 0xBB67AE85u;
  }
  // u1 = (a + 1) 2^-53 and u2 = b 2^-53, a and b the upper 53 bits of (c1, c0) and
  // (c3, c2): all sums below are exact
  const double k53 = JJA_K(0x1.0p-53), k32 = JJA_K(0x1.0p-32);
  const double u1 = fma(static_cast<double>(c1), k32, fma(static_cast<double>(c0 >> 11), k53, k53));
  const double u2 = fma(static_cast<double>(c3), k32, static_cast<double>(c2 >> 11) * k53);
  // sqrt(-2 log u1) by Goldschmidt's iteration from the estimate of its reciprocal
  // root; u1 = 1 gives 1e-150 for 0
  const double x = fmax(2.0 * jja_neg_log(u1), 1e-300);
  const double e = __builtin_amdgcn_rsq(x);
  double g = x * e, h = 0.5 * e;
  const double c = fma(-h, g, 0.5);
  g = fma(g, c, g);
  h = fma(h, c, h);
  const double rho = fma(fma(-g, g, x), h, g);
  double sn, cs;
  jja_sincos_turn(u2, &sn, &cs);
  *z0 = rho * cs;
  *z1 = rho * sn;
}

// One 64-bit DPP move (two 32-bit halves); rows outside ROW_MASK and lanes
// without a source read 0.
template <int CTRL, int ROW_MASK>
__device__ __forceinline__ double dpp_f64(double v) {
  const long long b = __builtin_bit_cast(long long, v);
  const int lo = __builtin_amdgcn_update_dpp(0, static_cast<int>(b), CTRL, ROW_MASK, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, static_cast<int>(b >> 32), CTRL, ROW_MASK, 0xf, true);
  return __builtin_bit_cast(double, static_cast<long long>(static_cast<unsigned>(lo)) |
                                        (static_cast<long long>(hi) << 32));
}

// Sum over each aligned group of G lanes (G a power of two <= 64), left in the
// group's last lane. Fixed order (shift-add within 16-lane rows, then row
// broadcasts), so the bits do not depend on anything but the inputs.
__device__ __forceinline__ double group_sum_last(double v, int G) {
  if (G >= 2) v += dpp_f64<0x111, 0xf>(v);   // row_shr:1
  if (G >= 4) v += dpp_f64<0x112, 0xf>(v);   // row_shr:2
  if (G >= 8) v += dpp_f64<0x114, 0xf>(v);   // row_shr:4
  if (G >= 16) v += dpp_f64<0x118, 0xf>(v);  // row_shr:8
  if (G >= 32) v += dpp_f64<0x142, 0xa>(v);  // row_bcast:15 into rows 1, 3
  if (G >= 64) v += dpp_f64<0x143, 0xc>(v);  // row_bcast:31 into rows 2, 3
  return v;
}

// Where a column keeps its face vector z (by solve position) and the stage
// scratch t after it, and which threads work on the column. FaceStore<false>:
// the workgroup's LDS, addressed by the plan's 16-bit indices as absolute LDS
// addresses (the evolve and adjoint kernels have no static LDS, checked on the
// host before every launch). FaceStore<true>: a per-column array in global
// memory for circuits whose face vector does not fit in LDS, addressed by
// 32-bit indices. SplitStore: the global array of a column that several
// workgroups (its parts) share. The arithmetic on the values is the same in all.
//
// vt and vbs are the thread's index within the column and the column's thread
// count (threadIdx.x and the block size, or part * blockDim + threadIdx.x and
// parts * blockDim). sync() orders all memory between the column's threads;
// barrier() orders the face vector only (the solve's phase boundaries).
template <bool GLOBAL>
struct FaceStore;

template <>
struct FaceStore<false> {
  static constexpr bool kGlobal = false;
  double* p;
  int32_t vt, vbs;
  __device__ __forceinline__ double rd(int64_t i) const { return p[i]; }
  __device__ __forceinline__ double gather(uint32_t i) const {
    return *reinterpret_cast<const LAS double*>(static_cast<uintptr_t>(i) << 3);
  }
  __device__ __forceinline__ void wr(int64_t i, double v) const { p[i] = v; }
  // elements i and i+1 (i even) in one 16-byte load
  __device__ __forceinline__ vdouble2 rd2(int64_t i) const {
    return *reinterpret_cast<const LAS vdouble2*>(static_cast<uintptr_t>(i) << 3);
  }
  // orders LDS traffic only: global loads in flight stay in flight
  __device__ __forceinline__ void barrier() const { lds_barrier(); }
  __device__ __forceinline__ void wg_barrier() const { lds_barrier(); }
  __device__ __forceinline__ void sync() const { __syncthreads(); }
};

template <>
struct FaceStore<true> {
  static constexpr bool kGlobal = true;
  GAS double* p;
  int32_t vt, vbs;
  __device__ __forceinline__ double rd(int64_t i) const { return p[i]; }
  __device__ __forceinline__ double gather(uint32_t i) const { return p[i]; }
  __device__ __forceinline__ void wr(int64_t i, double v) const { p[i] = v; }
  __device__ __forceinline__ vdouble2 rd2(int64_t i) const {
    return *reinterpret_cast<const GAS vdouble2*>(p + i);
  }
  __device__ __forceinline__ void barrier() const { __syncthreads(); }
  __device__ __forceinline__ void wg_barrier() const { __syncthreads(); }
  __device__ __forceinline__ void sync() const { __syncthreads(); }
};

// Dynamic LDS a split workgroup may take for its part of a lattice solve (the
// workgroup's 160 KiB less room for its static variables)
constexpr int64_t kSplitLdsMax = 163840 - 256;

// Default polls of one column barrier before a workgroup gives up (each poll
// sleeps briefly; far longer than any phase of a step takes).
constexpr uint32_t kWaitLimit = 1u << 21;
// s_waitcnt immediate (gfx9 encoding) that waits for vmcnt 0 only: expcnt and
// lgkmcnt fields at their maxima
constexpr int kWaitVmem = 0x0F70;

// The XCD (accelerator complex die) the calling wave runs on: hardware
// register XCC_ID, bits 3:0.
__device__ __forceinline__ uint32_t xcd_id() {
  return __builtin_amdgcn_s_getreg((3 << 11) | 20) & 15u;
}

struct SplitStore {
  static constexpr bool kGlobal = true;
  GAS double* p;
  int32_t vt, vbs;
  uint32_t* ctr;         // the column's arrival counter, zero at launch
  uint32_t* xcds;        // bit x set by each part running on XCD x, zero at launch
  uint32_t parts;
  uint32_t wait_limit;   // polls before a wait gives up
  int32_t* err;          // [0] set when a wait gave up; [1] counts one-XCD workgroups
  int32_t* stopped;      // this workgroup's flag (LDS): it no longer waits
  mutable uint32_t gen;  // arrivals to wait for (thread 0)
  mutable bool one_xcd;  // every part of the column shares this XCD's L2 (thread 0)
  LAS double* lds;       // this workgroup's dynamic LDS (the part-local tridiagonal solve)
  __device__ __forceinline__ double rd(int64_t i) const { return p[i]; }
  __device__ __forceinline__ double gather(uint32_t i) const { return p[i]; }
  __device__ __forceinline__ void wr(int64_t i, double v) const { p[i] = v; }
  __device__ __forceinline__ vdouble2 rd2(int64_t i) const {
    return *reinterpret_cast<const GAS vdouble2*>(p + i);
  }
  // Every wave waits for its own memory operations (stores reach the L2,
  // which the L1 writes through to), the workgroup meets, and thread 0 alone
  // arrives on the column's counter, polls it with relaxed loads (an acquire
  // per poll would invalidate caches under the working workgroups) and
  // acquires once at device scope (the invalidation covers the compute unit's
  // other waves); then the workgroup meets again.
  //   Parts on several XCDs (separate L2s) release at device scope before the
  // arrival: an L2 write-back. Parts on one XCD skip it: their stores already
  // meet in that XCD's L2. The parts publish their XCDs at launch
  // (split_store); each workgroup reads the column's set after its first
  // barrier, which always releases.
  //   A wait that gives up sets err and stops this workgroup's waits for the
  // rest of the launch (its results are then invalid, and the host reports
  // the error).
  __device__ __forceinline__ void sync() const {
    if (parts == 1) {  // a column of one workgroup (in a launch with split columns)
      __syncthreads();
      return;
    }
    __builtin_amdgcn_s_waitcnt(kWaitVmem);
    __syncthreads();
    if (threadIdx.x == 0 && !*stopped) {
      gen += parts;
      if (one_xcd)
        __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      else
        __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
      uint32_t spins = 0;
      while (__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < gen) {
        if (++spins > wait_limit) {
          *stopped = 1;
          __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          break;
        }
        __builtin_amdgcn_s_sleep(2);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
      // after the first barrier every part has published its XCD
      if (gen == parts && !*stopped) {
        one_xcd = __builtin_popcount(__hip_atomic_load(xcds, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 1;
        if (one_xcd) __hip_atomic_fetch_add(err + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
    __syncthreads();
  }
  __device__ __forceinline__ void barrier() const { sync(); }
  // the waves of this workgroup only (a part-local phase: its rows' readers
  // and writers are all in this workgroup)
  __device__ __forceinline__ void wg_barrier() const { __syncthreads(); }
};

// Entries of one solve record for one lane, held in registers: 8 values and
// their indices (two 16-bit halves per word, or one 32-bit index per word).
template <bool GLOBAL>
struct SliceRegs {
  double v[kMaxIter];
  uint32_t idx[GLOBAL ? kMaxIter : kMaxIter / 2];
  int32_t row;
};

template <bool GLOBAL>
__device__ __forceinline__ uint32_t slice_index(const SliceRegs<GLOBAL>& r, int i) {
  if constexpr (GLOBAL)
    return r.idx[i];
  else
    return (r.idx[i / 2] >> (16 * (i % 2))) & 0xffffu;
}

// Face-store index of entry i of a record. In a global store a block-phase
// record's lane reads consecutive scratch rows: its word (idx[0]) is
// base | len << 28, and entry i is base + i*G for i < len, else 0 (a padding
// entry: its value is zero). LDS stores keep explicit indices: there the
// decode costs more than the index bytes it saves.
template <bool GLOBAL>
__device__ __forceinline__ uint32_t record_index(const SliceRegs<GLOBAL>& r, int32_t flags, int i) {
  if (GLOBAL && (flags & JJA_SLICE_BLOCK)) {
    const uint32_t w = r.idx[0];
    const uint32_t G = static_cast<uint32_t>(flags & 0xff);
    return static_cast<uint32_t>(i) < (w >> 28) ? (w & 0x0FFFFFFFu) + static_cast<uint32_t>(i) * G : 0u;
  }
  // a NARROW off-block record of a global store: lane base (idx[0]) plus a
  // 16-bit offset (two per word in idx[1..4])
  if (GLOBAL && (flags & JJA_SLICE_NARROW))
    return r.idx[0] + ((r.idx[1 + i / 2] >> (16 * (i % 2))) & 0xffffu);
  return slice_index(r, i);
}

// Issue the loads of one solve record: always the same vector loads, each a
// scalar base (from the record) plus a per-lane offset that does not change
// between records, so no address arithmetic runs per record.
// The record values go through a buffer resource over ent_val: a value pair at
// or past the record's iteration count is read at an offset beyond the
// resource's range, which returns zeros without a memory access, so a short
// record moves only the bytes it uses and every record issues the same loads.
template <class D>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t value_resource(const D& P) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<double*>(P.ent_val), 0, P.val_bytes, kBufferWord3);
}

template <bool GLOBAL, class D>
__device__ __forceinline__ void load_slice(const D& P, __amdgpu_buffer_rsrc_t vres,
                                           const jja_slice& m, int lane, SliceRegs<GLOBAL>& r) {
  const int lg = __builtin_ctz(static_cast<unsigned>(m.flags & 0xff));
  const uint32_t voff = static_cast<uint32_t>(m.base) * 8u + static_cast<uint32_t>(lane) * 16u;
  // the raw row; whether this lane's slot holds one is decided when the record
  // is processed (a select here would wait for the load)
  r.row = gbl(P.slice_rows)[m.rowbase + (lane >> lg)];
#pragma unroll
  for (int q = 0; q < kMaxIter / 2; ++q) {
    const uint32_t off = 2 * q < m.n_iter ? voff + q * 16u * kWave : kOutOfRange;
    const vdouble2 d = __builtin_bit_cast(
        vdouble2, __builtin_amdgcn_raw_buffer_load_b128(vres, static_cast<int>(off), 0, 0));
    r.v[2 * q] = d.x;
    r.v[2 * q + 1] = d.y;
  }
  if (GLOBAL && (m.flags & JJA_SLICE_BLOCK)) {
    // implicit indices: one word per lane
    r.idx[0] = gbl(static_cast<const uint32_t*>(P.ent_off) + m.ibase)[lane];
  } else if (GLOBAL && (m.flags & JJA_SLICE_NARROW)) {
    // lane base, then 8 16-bit offsets in one 16-byte load
    const uint32_t* ip = static_cast<const uint32_t*>(P.ent_off) + m.ibase;
    r.idx[0] = gbl(ip)[lane];
    const vuint4 o = gbl(reinterpret_cast<const vuint4*>(ip + kWave))[lane];
    r.idx[1] = o.x;
    r.idx[2] = o.y;
    r.idx[3] = o.z;
    r.idx[4] = o.w;
  } else if constexpr (GLOBAL) {
    const GAS vuint4* __restrict__ op =
        gbl(reinterpret_cast<const vuint4*>(static_cast<const uint32_t*>(P.ent_off) + m.ibase)) + 2 * lane;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const vuint4 o = op[q];
      r.idx[4 * q] = o.x;
      r.idx[4 * q + 1] = o.y;
      r.idx[4 * q + 2] = o.z;
      r.idx[4 * q + 3] = o.w;
    }
  } else {
    const vuint4 o = *(gbl(reinterpret_cast<const vuint4*>(static_cast<const uint16_t*>(P.ent_off) + m.ibase)) + lane);
    r.idx[0] = o.x;
    r.idx[1] = o.y;
    r.idx[2] = o.z;
    r.idx[3] = o.w;
  }
}

// Gather, accumulate, and (flag FINISH) reduce and write one record's rows.
template <class Z>
__device__ __forceinline__ void process_slice(const Z& zs, int32_t Nf, int lane, const jja_slice& m,
                                              const SliceRegs<Z::kGlobal>& r, double& acc) {
  // iterations at or past the record's count have zero values and index 0:
  // their gathers read one broadcast address and contribute exact zeros
  double zv[kMaxIter];
#pragma unroll
  for (int i = 0; i < kMaxIter; ++i) zv[i] = zs.gather(record_index(r, m.flags, i));
#pragma unroll
  for (int i = 0; i < kMaxIter; ++i) acc = __builtin_fma(r.v[i], zv[i], acc);
  if (m.flags & JJA_SLICE_FINISH) {
    const int G = m.flags & 0xff;
    acc = group_sum_last(acc, G);
    const int slot = lane >> __builtin_ctz(static_cast<unsigned>(G));
    if (slot < (m.flags >> 16) && r.row >= 0 && (lane & (G - 1)) == G - 1) {
      if (m.flags & JJA_SLICE_BLOCK)
        zs.wr(r.row, acc);
      else
        zs.wr(Nf + r.row - m.r0, zs.rd(r.row) - acc);
    }
    acc = 0.0;
  }
  if (m.flags & JJA_SLICE_BARRIER)
    zs.barrier();
  else if (m.flags & JJA_SLICE_WG_BARRIER)
    zs.wg_barrier();
}

// The whole forward + backward solve. Each wave walks its own record program,
// software-pipelined in three register buffers used in turn: the loads of
// records k+1 and k+2 are in flight while record k is processed (the
// scheduling barriers keep the compiler from hoisting a record's LDS address
// use above the next record's loads, which would make it wait for all loads),
// and descriptors are read ahead. A wave's executed record count is a multiple
// of three and four never-executed records follow it, so the loop has a single
// exit and every lookahead load stays inside the program. Waves meet only at
// BARRIER records (one per phase, the same number in every wave). D: a problem, or
// anything with its program's arrays.
// solve_head issues the loads of a program's first two records, which a caller may do
// early (before a barrier or a wait) to hide their latency.
template <bool GLOBAL>
struct SolveHead {
  SliceRegs<GLOBAL> A, B;
};

template <class D>
__device__ __forceinline__ int32_t program_start(const D& P, int32_t vt) {
  const CAS int32_t* wp = (const CAS int32_t*)(P.wave_ptr) + __builtin_amdgcn_readfirstlane(vt / kWave);
  return __builtin_amdgcn_readfirstlane(wp[0]);
}

template <class D, bool GLOBAL>
__device__ __forceinline__ void solve_head(const D& P, int32_t vt, SolveHead<GLOBAL>& h) {
  const int lane = vt & (kWave - 1);
  const jja_slice* __restrict__ prog = P.solve_slices + program_start(P, vt);
  const __amdgpu_buffer_rsrc_t vres = value_resource(P);
  load_slice(P, vres, load_rec(prog, 0), lane, h.A);
  load_slice(P, vres, load_rec(prog, 1), lane, h.B);
  __builtin_amdgcn_sched_barrier(0);
}

template <class D, class Z>
__device__ __forceinline__ void solve_tail(const D& P, const Z& zs, SolveHead<Z::kGlobal>& h) {
  constexpr bool GLOBAL = Z::kGlobal;
  const int lane = zs.vt & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(zs.vt / kWave);
  const CAS int32_t* wp = (const CAS int32_t*)(P.wave_ptr) + wave;
  const int32_t k0 = __builtin_amdgcn_readfirstlane(wp[0]);
  const int32_t nk = __builtin_amdgcn_readfirstlane(wp[1]) - k0 - 4;
  const jja_slice* __restrict__ prog = P.solve_slices + k0;
  jja_slice m0 = load_rec(prog, 0), m1 = load_rec(prog, 1), m2 = load_rec(prog, 2);
  const __amdgpu_buffer_rsrc_t vres = value_resource(P);
  SliceRegs<GLOBAL>&A = h.A, &B = h.B;
  SliceRegs<GLOBAL> C;
  double acc = 0.0;
  for (int32_t k = 0; k < nk; k += 3) {
    const jja_slice m3 = load_rec(prog, k + 3);
    load_slice(P, vres, m2, lane, C);
    __builtin_amdgcn_sched_barrier(0);
    process_slice(zs, P.Nf, lane, m0, A, acc);
    const jja_slice m4 = load_rec(prog, k + 4);
    load_slice(P, vres, m3, lane, A);
    __builtin_amdgcn_sched_barrier(0);
    process_slice(zs, P.Nf, lane, m1, B, acc);
    const jja_slice m5 = load_rec(prog, k + 5);
    load_slice(P, vres, m4, lane, B);
    __builtin_amdgcn_sched_barrier(0);
    process_slice(zs, P.Nf, lane, m2, C, acc);
    m0 = m3;
    m1 = m4;
    m2 = m5;
  }
}

template <class D, class Z>
__device__ __forceinline__ void solve(const D& P, const Z& zs) {
  SolveHead<Z::kGlobal> h;
  solve_head(P, zs.vt, h);
  solve_tail(P, zs, h);
}

// ------------------------------------------------------------ lattice solve
// The face matrix of a rectangular lattice of R x C faces (positions r*C + c)
// with one junction weight per direction is the Kronecker sum
// g (T_R (x) I_C) + g_c (I_R (x) T_C), T_n = tridiag(-1, 2, -1), so
// K^-1 = (I (x) S) M^-1 (I (x) S) with the orthonormal symmetric sine matrix S
// (DST-I) and M tridiagonal along r for each sine mode (Hockney, J. ACM 12
// (1965) 95-113). Per step: fold every row (S[C-1-i][j] = (-1)^j S[i][j]),
// transform (out[r][j] = sum_{i<H} F_j[r][i] S[i][j], H = ceil(C/2)), one
// tridiagonal solve per mode along r, then fold and transform again. Each
// transform output is summed in a fixed order (one thread in ascending i with
// fused multiply-adds in LDS; one matrix-core chain in a global store) and each
// block of a mode's recurrence runs in one thread with a blocking fixed by R, C
// and the part count, so results do not depend on the block size or the launch
// length; the two face stores agree to rounding.

// Stores the lattice solve runs on: one workgroup's (LDS or global) and a
// split column's (global, column barriers)
template <class Z>
struct RunsLattice {
  static constexpr bool value = false;
};
template <bool G>
struct RunsLattice<FaceStore<G>> {
  static constexpr bool value = true;
};
template <>
struct RunsLattice<SplitStore> {
  static constexpr bool value = true;
};

// elements of the fold each thread loads before it computes (global store)
constexpr int kFoldBatch = 4;

// E[r][i] = v[r][i] + v[r][C-1-i], O[r][i] = v[r][i] - v[r][C-1-i] for i < H
// (the middle of an odd row pairs with itself: E = v, O = 0) and 0 for
// H <= i < EF (EF = lat_ef). An LDS store keeps them by row (EF = ES; E at
// lat_t0 + r*ES + i, O at lat_t0 + (R + r)*ES + i: a lane reads 16 bytes of its
// own row per load). A global store keeps them in blocks of four i by row
// (EF = ES rounded up to 4; E at lat_t0 + ((i/4)*R + r)*4 + i%4, O at
// lat_t0 + R*EF + the same): a matrix-core operand, 16 rows x 4 i, is 512
// contiguous bytes, and a wave of the fold reads 32-byte runs of 16 rows.
// Either way element e of the loop lands at lat_t0 + e and lat_t0 + R*EF + e.
template <class Z>
__device__ __forceinline__ void lattice_fold(const DevProblem& P, const Z& zs) {
  constexpr int KB = Z::kGlobal ? kFoldBatch : 1;
  const int32_t R = P.lat_rows, C = P.lat_cols, ES = P.lat_es, H = (C + 1) >> 1;
  const int32_t n = R * P.lat_ef;
  const int64_t e0 = P.lat_t0, o0 = P.lat_t0 + static_cast<int64_t>(R) * P.lat_ef;
  // KB elements per thread at a time: all their loads are issued first
  for (int32_t e = zs.vt; e < n; e += KB * zs.vbs) {
    double x[KB], y[KB];
    int32_t ii[KB];
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      const int32_t ek = min(e + k * zs.vbs, n - 1);
      int32_t r, i;
      if constexpr (Z::kGlobal) {
        const int32_t blk = (ek >> 2) / R;
        r = (ek >> 2) - blk * R;
        i = 4 * blk + (ek & 3);
      } else {
        r = ek / ES;
        i = ek - r * ES;
      }
      ii[k] = i;
      // a padding slot (i >= H) reads the row's first element and drops it
      const int64_t row = static_cast<int64_t>(r) * C;
      const int32_t ic = i < H ? i : 0;
      x[k] = zs.rd(row + ic);
      y[k] = zs.rd(row + (C - 1 - ic));
    }
#pragma unroll
    for (int k = 0; k < KB; ++k) {
      const int32_t ek = e + k * zs.vbs;
      if (ek >= n) break;
      const int32_t i = ii[k];
      double a = 0.0, b = 0.0;
      if (i < H) {
        if (2 * i + 1 == C) {
          a = x[k];
        } else {
          a = x[k] + y[k];
          b = x[k] - y[k];
        }
      }
      zs.wr(e0 + ek, a);
      zs.wr(o0 + ek, b);
    }
  }
}

// out[r][j] = sum_{i<ES} (j even ? E : O)[r][i] S[i][j] into the face vector
// of an LDS store. A wave takes 64 rows (one per lane) and JJA_LATTICE_CHUNK
// consecutive modes from an even j0, so a mode's parity is its slot's; the
// table's values are wave-uniform scalar loads. Each output adds its terms in
// ascending i with fused multiply-adds.
template <class Z>
__device__ __forceinline__ void lattice_transform_lds(const DevProblem& P, const Z& zs) {
  constexpr int MC = JJA_LATTICE_CHUNK;
  const int32_t R = P.lat_rows, C = P.lat_cols, ES = P.lat_es, CP = P.lat_cp;
  const int lane = zs.vt & (kWave - 1);
  const int32_t wave = __builtin_amdgcn_readfirstlane(zs.vt / kWave);
  const int32_t NW = zs.vbs / kWave;
  const int32_t nrb = (R + kWave - 1) / kWave, tasks = nrb * (CP / MC);
  const CAS double* __restrict__ S = (const CAS double*)P.lat_sine;
  for (int32_t task = wave; task < tasks; task += NW) {
    const int32_t rb = task % nrb, j0 = (task / nrb) * MC;
    const int32_t r = rb * kWave + lane;
    const int64_t e = P.lat_t0 + static_cast<int64_t>(r < R ? r : R - 1) * ES;
    const int64_t o = e + static_cast<int64_t>(R) * ES;
    double acc[MC];
#pragma unroll
    for (int q = 0; q < MC; ++q) acc[q] = 0.0;
    for (int32_t i = 0; i < ES; i += 2) {
      const vdouble2 ev = zs.rd2(e + i), ov = zs.rd2(o + i);
      const CAS double* s0 = S + static_cast<int64_t>(i) * CP + j0;
      const CAS double* s1 = s0 + CP;
#pragma unroll
      for (int q = 0; q < MC; ++q) {
        acc[q] = __builtin_fma((q & 1) ? ov.x : ev.x, s0[q], acc[q]);
        acc[q] = __builtin_fma((q & 1) ? ov.y : ev.y, s1[q], acc[q]);
      }
    }
    if (r < R) {
      const int64_t row = static_cast<int64_t>(r) * C;
#pragma unroll
      for (int q = 0; q < MC; ++q)
        if (j0 + q < C) zs.wr(row + j0 + q, acc[q]);
    }
  }
}

// The solve of an LDS store with room for padding: both sides of the lattice by
// sine transforms, X = S_R ((S_R B S_C) / lambda) S_C with lambda = g mu_R +
// g_c mu_C, as four products on the matrix cores between two copies of the face
// vector. A wave takes 16 x 16 tiles of v_mfma_f64_16x16x4f64 (lane l holds
// A[l%16][l/16] and B[l/16][l%16], result register q D[l/16 + 4q][l%16]): one
// operand comes from the sine table in LDS, the other is the sum (even modes) or
// difference (odd modes) of two mirrored elements, folded as they are read
// (S[n-1-i][j] = (-1)^j S[i][j]); a wave takes an even and an odd block of modes
// together. Rows and columns are padded to whole blocks of zeros, so nothing is
// clamped or masked.
//   Small lattices are bound by latency: one wave issues an instruction in 4 to 8
// cycles, so what counts is the instructions of a stage and the number of
// barriers (four here, against ten with folds, transforms of the rows only and
// blocked recurrences along them).

// dst[r][j] = sum_i src[r][i] S[i][j] (LEFT false), or dst[i][c] = lam[i][c]
// sum_r S[i][r] src[r][c] (LEFT true; lam may be NULL)
template <bool LEFT>
__device__ __forceinline__ void dst_product(const LAS double* src, LAS double* dst, const LAS double* table,
                                            const GAS double* lam, int32_t n, int32_t other, int32_t ld, int32_t tid,
                                            int32_t nt) {
  const DstShape D(n);
  const int lane = tid & (kWave - 1), lr = lane & 15, lk = lane >> 4;
  const int32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), NW = nt / kWave;
  const int32_t tasks = D.pairs * ((other + 15) >> 4);
  // task = block of the other side * pairs + mode pair, split by subtraction (a
  // division costs more than the few rounds)
  for (int32_t task = wave, mb = wave, ob = 0; task < tasks; task += NW, mb += NW) {
    while (mb >= D.pairs) {
      mb -= D.pairs;
      ob += 16;
    }
    const LAS double* f = table + mb * D.steps * 2 * kWave + lane;
    // element i of the folded side at s0 + i * si, its mirror at s1 - i * si
    const int32_t si = LEFT ? ld : 1, o = LEFT ? ob + lr : (ob + lr) * ld;
    const LAS double* s0 = src + o + lk * si;
    const LAS double* s1 = src + o + (n - 1 - lk) * si;
    const int32_t out = LEFT ? 2 * (16 * mb + lk) * ld + ob + lr : (ob + lk) * ld + 2 * (16 * mb + lr);
    double scale[4][2];
    if (LEFT && lam) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        scale[r][0] = lam[out + 8 * r * ld];
        scale[r][1] = lam[out + (8 * r + 1) * ld];
      }
    }
    vdouble4 ae{0.0, 0.0, 0.0, 0.0}, ao{0.0, 0.0, 0.0, 0.0};
    for (int32_t k = 0; k < D.steps; k += 2) {
      double p[2], q[2], v[2][2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        p[u] = s0[4 * u * si];
        q[u] = s1[-4 * u * si];
        v[u][0] = f[(2 * u) * kWave];
        v[u][1] = f[(2 * u + 1) * kWave];
      }
      s0 += 8 * si;
      s1 -= 8 * si;
      f += 4 * kWave;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const double e = p[u] + q[u], d = p[u] - q[u];
        if constexpr (LEFT) {
          ae = __builtin_amdgcn_mfma_f64_16x16x4f64(v[u][0], e, ae, 0, 0, 0);
          ao = __builtin_amdgcn_mfma_f64_16x16x4f64(v[u][1], d, ao, 0, 0, 0);
        } else {
          ae = __builtin_amdgcn_mfma_f64_16x16x4f64(e, v[u][0], ae, 0, 0, 0);
          ao = __builtin_amdgcn_mfma_f64_16x16x4f64(d, v[u][1], ao, 0, 0, 0);
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if constexpr (LEFT) {
        dst[out + 8 * r * ld] = lam ? ae[r] * scale[r][0] : ae[r];
        dst[out + (8 * r + 1) * ld] = lam ? ao[r] * scale[r][1] : ao[r];
      } else {
        *reinterpret_cast<LAS vdouble2*>(dst + out + 4 * r * ld) = vdouble2{ae[r], ao[r]};
      }
    }
  }
}

// K^-1 for a lattice of at most 16 by 16 faces: Z <- S_R (lam o (S_R Z S_C)) S_C by one
// wave, without barriers between the four products. The result of a product lies in the
// lanes as the operand B of the next (register r of the result is step r's operand), so
// the three products that sum over rows follow each other in registers, and only the
// last, over columns, takes its operand through LDS. The chain of 16 matrix
// instructions is 1200 cycles; four products shared by the workgroup's waves, halved by
// parity, spend longer at their barriers (64 columns of 12x9, thermal: 4.67 us a step,
// now 3.46).
__device__ __forceinline__ void solve_lattice_tile(const DevProblem& P, const FaceStore<false>& zs) {
  constexpr int32_t N = TileShape::kSide, LD = TileShape::kLd, T = TileShape::kTable;
  if (zs.vt < kWave) {
    const int32_t R = P.lat_rows, C = P.lat_cols;
    const int32_t lane = zs.vt, lr = lane & 15, lk = lane >> 4;
    LAS double* z = (LAS double*)zs.p;
    LAS double* t = z + P.lat_buf;
    const LAS double* tab = z + P.lat_tab + lane;
    double x[4], sc[4], sr[4], lam[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      // past the lattice the tables are zero: any finite operand will do
      x[s] = z[min(lr, R - 1) * LD + min(4 * s + lk, C - 1)];
      sc[s] = tab[s * kWave];
      sr[s] = tab[T + s * kWave];
      lam[s] = tab[2 * T + s * kWave];
    }
    vdouble4 a{0.0, 0.0, 0.0, 0.0}, b = a, c = a, d = a;
#pragma unroll
    for (int s = 0; s < 4; ++s) a = __builtin_amdgcn_mfma_f64_16x16x4f64(x[s], sc[s], a, 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 4; ++s) b = __builtin_amdgcn_mfma_f64_16x16x4f64(sr[s], a[s], b, 0, 0, 0);
#pragma unroll
    for (int s = 0; s < 4; ++s) c = __builtin_amdgcn_mfma_f64_16x16x4f64(sr[s], b[s] * lam[s], c, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) t[(lk + 4 * r) * LD + lr] = c[r];
    // one wave's LDS accesses stay in order
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = t[lr * LD + 4 * s + lk];
#pragma unroll
    for (int s = 0; s < 4; ++s) d = __builtin_amdgcn_mfma_f64_16x16x4f64(x[s], sc[s], d, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (lk + 4 * r < R && lr < C) z[(lk + 4 * r) * LD + lr] = d[r];
  }
  static_assert(N * N == T, "a table of four steps of 64 lanes");
  zs.barrier();
}

__device__ __forceinline__ void solve_lattice_padded(const DevProblem& P, const FaceStore<false>& zs) {
  if (P.lat_tile) return solve_lattice_tile(P, zs);
  const int32_t R = P.lat_rows, C = P.lat_cols, ld = P.lat_ld;
  LAS double* z = (LAS double*)zs.p;
  LAS double* t = z + P.lat_buf;
  const LAS double* tc = z + P.lat_tab;
  const LAS double* tr = R == C ? tc : tc + DstShape(C).entries();
  dst_product<false>(z, t, tc, nullptr, C, R, ld, zs.vt, zs.vbs);
  zs.barrier();
  dst_product<true>(t, z, tr, gbl(P.lat_lam), R, C, ld, zs.vt, zs.vbs);
  zs.barrier();
  dst_product<true>(z, t, tr, nullptr, R, C, ld, zs.vt, zs.vbs);
  zs.barrier();
  dst_product<false>(t, z, tc, nullptr, C, R, ld, zs.vt, zs.vbs);
  zs.barrier();
}

// Zeros in both copies of the face vector (their padding stays zero) and the sine
// tables: every kernel with an LDS store, before it writes its first face value.
__device__ __forceinline__ void init_store(const DevProblem& P, double* lds, int32_t tid, int32_t nt) {
  if (!P.lat_ld) return;
  for (int32_t i = tid; i < P.lat_tab; i += nt) lds[i] = 0.0;
  for (int32_t i = P.lat_tab + tid; i < P.store_doubles; i += nt) lds[i] = gbl(P.lat_table)[i - P.lat_tab];
  __syncthreads();
}

// The same sums for a global store, on the matrix cores: for each parity p,
// out[r][2m+p] = sum_i F_p[r][i] S[i][2m+p] (F_0 = E, F_1 = O) is a product
// of an R x ES and an ES x (modes of parity p) matrix. A wave takes a tile of
// 32 rows x 32 modes of one parity as 2 x 2 blocks of 16 x 16 and runs
// v_mfma_f64_16x16x4f64 over i in steps of 4; lane l holds A[i][k] =
// F[r0 + l%16][i0 + l/16] and B[k][j] = S[i0 + l/16][2(m0 + l%16) + p], and
// result register q of lane l is D[l/16 + 4q][l%16]. E and O are kept in
// blocks of four i by row, so each A load is 512 contiguous bytes; B comes from
// the table with even and odd modes apart (lat_sine_p), four 128-byte rows.
// kMfmaBatch steps of loads are issued before their products. Rows and modes
// past the lattice load clamped (finite) operands and are not stored; the
// folded rows are zero for i >= H, and table rows past ES are read clamped.
// The matrix cores round differently from a chain of fused multiply-adds: the
// two stores agree to rounding.
constexpr int kMfmaBatch = 4;
constexpr int kMfmaRowBlocks = 2;   // 16-row blocks per wave tile
constexpr int kMfmaModeBlocks = 2;  // 16-mode blocks per wave tile
template <class Z>
__device__ __forceinline__ void lattice_transform_mfma(const DevProblem& P, const Z& zs) {
  constexpr int U = kMfmaBatch, NR = kMfmaRowBlocks, NC = kMfmaModeBlocks;
  constexpr int TR = 16 * NR, TC = 16 * NC;  // tile rows, tile modes (of one parity)
  const int32_t R = P.lat_rows, C = P.lat_cols, ES = P.lat_es, EF = P.lat_ef, CP = P.lat_cp;
  const int lane = zs.vt & (kWave - 1);
  const int32_t wave = __builtin_amdgcn_readfirstlane(zs.vt / kWave);
  const int32_t NW = zs.vbs / kWave;
  const int32_t n_even = (C + 1) >> 1, n_odd = C >> 1;
  const int32_t nrt = (R + TR - 1) / TR, nte = (n_even + TC - 1) / TC, nto = (n_odd + TC - 1) / TC;
  const int32_t tasks = nrt * (nte + nto);
  const int lr = lane & 15, lk = lane >> 4;
  const GAS double* __restrict__ S = gbl(P.lat_sine_p);
  const int32_t half = CP >> 1;
  for (int32_t task = wave; task < tasks; task += NW) {
    const int32_t rt = task % nrt, mt = task / nrt;
    const int par = mt < nte ? 0 : 1;
    const int32_t m0 = TC * (par ? mt - nte : mt);
    const int32_t r0 = TR * rt;
    // operand addresses of this lane (clamped into the lattice)
    const GAS double* fa[NR];
    const GAS double* sb[NC];
#pragma unroll
    for (int b = 0; b < NR; ++b) {
      const int32_t r = min(r0 + 16 * b + lr, R - 1);
      fa[b] = zs.p + P.lat_t0 + static_cast<int64_t>(par) * EF * R + 4 * r + lk;
    }
#pragma unroll
    for (int c = 0; c < NC; ++c) sb[c] = S + par * half + min(m0 + 16 * c + lr, half - 1);
    vdouble4 acc[NR][NC];
#pragma unroll
    for (int b = 0; b < NR; ++b)
#pragma unroll
      for (int c = 0; c < NC; ++c) acc[b][c] = vdouble4{0.0, 0.0, 0.0, 0.0};
    for (int32_t i0 = 0; i0 < EF; i0 += 4 * U) {
      double av[U][NR], bv[U][NC];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int32_t i4 = i0 + 4 * u;                     // this step's first i (a multiple of 4)
        const int32_t blk = min(i4, EF - 4) >> 2;
        const int32_t ic = min(i4 + lk, ES - 1);
#pragma unroll
        for (int b = 0; b < NR; ++b) {
          const double v = fa[b][static_cast<int64_t>(blk) * R * 4];
          av[u][b] = i4 < EF ? v : 0.0;
        }
#pragma unroll
        for (int c = 0; c < NC; ++c) bv[u][c] = sb[c][static_cast<int64_t>(ic) * CP];
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int b = 0; b < NR; ++b)
#pragma unroll
          for (int c = 0; c < NC; ++c)
            acc[b][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[u][b], bv[u][c], acc[b][c], 0, 0, 0);
    }
#pragma unroll
    for (int b = 0; b < NR; ++b)
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const int32_t j = 2 * (m0 + 16 * c + lr) + par;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int32_t r = r0 + 16 * b + lk + 4 * q;
          if (r < R && j < C) zs.wr(static_cast<int64_t>(r) * C + j, acc[b][c][q]);
        }
      }
  }
}

template <class Z>
__device__ __forceinline__ void lattice_transform(const DevProblem& P, const Z& zs) {
  if constexpr (Z::kGlobal)
    lattice_transform_mfma(P, zs);
  else
    lattice_transform_lds(P, zs);
}

// Mode k's tridiagonal solve along r, in place in the face vector. Both
// sweeps are first-order linear recurrences with the multiplier
// a_r = g inv_r: forward d_r = (y_r + g d_{r-1}) inv_r = y_r inv_r + a_r d_{r-1},
// backward x_r = d_r - ((-g) inv_r) x_{r+1} = d_r + a_r x_{r+1}. The rows of a
// mode are cut into B blocks (B from R, C and the part count only, so results
// do not depend on the block size): each block runs its recurrence from a
// zero start while keeping the running product of its multipliers, and then
// adds its product times the value carried in from the blocks before it. A
// block's thread chains those blocks' (value, product) ends itself, in block
// order, so each carry is the same sum whoever forms it, and no phase or
// barrier is spent on a separate chain. Three phases: forward from zero;
// forward carries, then backward from zero on the same rows; backward carries.
constexpr int kTriRows = 8;  // rows (or block ends) held in registers at a time
// blocks per mode: JJA_LATTICE_TRI_THREADS per part of the column, over C
__device__ __forceinline__ int32_t lattice_blocks(const DevProblem& P) {
  return max(1, min(P.lat_rows, JJA_LATTICE_TRI_THREADS * P.parts / P.lat_cols));
}

// The value carried into block b of mode k: dir +1 chains the ends of blocks
// 0 .. b-1 upward (cin = endp cin + endv from 0), dir -1 the ends of blocks
// B-1 .. b+1 downward.
template <class Z>
__device__ __forceinline__ double lattice_carry(const Z& zs, int32_t C, int32_t B, int64_t endv, int64_t endp,
                                                int32_t b, int32_t k, int dir) {
  constexpr int TB = kTriRows;
  const int32_t n = dir > 0 ? b : B - 1 - b, first = dir > 0 ? 0 : B - 1;
  double cin = 0.0;
  for (int32_t i0 = 0; i0 < n; i0 += TB) {
    double ev[TB], ep[TB];
#pragma unroll
    for (int q = 0; q < TB; ++q) {
      const int64_t at = static_cast<int64_t>(first + dir * min(i0 + q, n - 1)) * C + k;
      ev[q] = zs.rd(endv + at);
      ep[q] = zs.rd(endp + at);
    }
#pragma unroll
    for (int q = 0; q < TB; ++q)
      if (i0 + q < n) cin = __builtin_fma(ep[q], cin, ev[q]);
  }
  return cin;
}

// The tridiagonal solves of a split column with each part's modes in its own
// LDS, followed by the second fold. Part p takes the mode pairs (i, C-1-i) for
// i in [p*MH, p*MH + MH) (MH = lat_mp / 2; the middle mode of an odd C has no
// partner) with all R rows (Y[r][slot]: the lower modes in slots 0..nh-1, their
// partners after them; R*lat_mp doubles), cuts each mode into BP = lat_bp
// blocks and runs the same blocked recurrences as lattice_tridiag between
// workgroup barriers; the block ends (forward and backward, value and product,
// 4*BP*lat_mp doubles) stay in LDS, so no column barrier is needed inside.
// Holding both modes of a pair, the part then writes their folded rows
// (E = x_i + x_{C-1-i}, O = x_i - x_{C-1-i}, the same sums as lattice_fold) in
// the global store's blocked layout, in place of a separate fold pass.
__device__ __forceinline__ void lattice_tridiag_parts(const DevProblem& P, const SplitStore& zs) {
  constexpr int TB = kTriRows;
  const int32_t R = P.lat_rows, C = P.lat_cols, CP = P.lat_cp, MP = P.lat_mp, B = P.lat_bp;
  const int32_t H = (C + 1) >> 1, EF = P.lat_ef, MH = MP >> 1;
  const int32_t nt = static_cast<int32_t>(blockDim.x), tid = static_cast<int32_t>(threadIdx.x);
  const int32_t part = __builtin_amdgcn_readfirstlane(zs.vt / nt);
  const int64_t e0 = P.lat_t0, o0 = P.lat_t0 + static_cast<int64_t>(R) * EF;
  // folded-row padding (H <= i < EF) is zero; part 0 writes it
  if (part == 0)
    for (int32_t e = tid; e < R * (EF - H); e += nt) {
      const int32_t i = H + e / R, r = e - (e / R) * R;
      const int64_t at = (static_cast<int64_t>(i >> 2) * R + r) * 4 + (i & 3);
      zs.wr(e0 + at, 0.0);
      zs.wr(o0 + at, 0.0);
    }
  const int32_t i0 = part * MH, nh = min(MH, H - i0);
  if (nh <= 0) return;  // a part past the last pair (the whole workgroup)
  const int32_t nu = (2 * (i0 + nh - 1) + 1 == C) ? nh - 1 : nh;  // partners (the middle has none)
  const int32_t nm = nh + nu;
  auto mode = [&](int32_t kk) { return kk < nh ? i0 + kk : C - 1 - (i0 + kk - nh); };
  const GAS double* __restrict__ inv = gbl(P.lat_inv);
  const double g = P.lat_g;
  const int32_t m = (R + B - 1) / B;
  LAS double* Y = zs.lds;
  LAS double* fv = Y + static_cast<int32_t>(R) * MP;
  LAS double* fp = fv + B * MP;
  LAS double* bv = fp + B * MP;
  LAS double* bp = bv + B * MP;
  for (int32_t e = tid; e < R * nm; e += nt) {
    const int32_t r = e / nm, kk = e - r * nm;
    Y[r * MP + kk] = zs.rd(static_cast<int64_t>(r) * C + mode(kk));
  }
  __syncthreads();
  auto sweep = [&](int32_t kk, int32_t first, int32_t count, int32_t dir, auto&& f) {
    const int32_t k = mode(kk);
    for (int32_t c0 = 0; c0 < count; c0 += TB) {
      double y[TB], a[TB];
#pragma unroll
      for (int q = 0; q < TB; ++q) {
        const int32_t r = first + dir * min(c0 + q, count - 1);
        y[q] = Y[r * MP + kk];
        a[q] = inv[static_cast<int64_t>(r) * CP + k];
      }
#pragma unroll
      for (int q = 0; q < TB; ++q)
        if (c0 + q < count) f(first + dir * (c0 + q), y[q], a[q]);
    }
  };
  // the value carried into block b (dir +1: from blocks 0..b-1, upward; dir
  // -1: from blocks B-1..b+1, downward), chained in block order
  auto carry = [&](const LAS double* ev, const LAS double* ep, int32_t b, int32_t kk, int dir) {
    const int32_t n = dir > 0 ? b : B - 1 - b, first = dir > 0 ? 0 : B - 1;
    double cin = 0.0;
    for (int32_t i = 0; i < n; ++i) {
      const int32_t at = (first + dir * i) * MP + kk;
      cin = __builtin_fma(ep[at], cin, ev[at]);
    }
    return cin;
  };
  // forward from zero
  for (int32_t e = tid; e < B * nm; e += nt) {
    const int32_t b = e / nm, kk = e - b * nm, r0 = b * m, n = min(m, R - r0);
    double d = 0.0, pr = 1.0;
    if (n > 0)
      sweep(kk, r0, n, 1, [&](int32_t r, double y, double iv) {
        d = __builtin_fma(g, d, y) * iv;
        pr = pr * (g * iv);
        Y[r * MP + kk] = d;
      });
    fv[b * MP + kk] = d;
    fp[b * MP + kk] = pr;
  }
  __syncthreads();
  // forward carries, then backward from zero (the same thread's rows)
  for (int32_t e = tid; e < B * nm; e += nt) {
    const int32_t b = e / nm, kk = e - b * nm, r0 = b * m, n = min(m, R - r0);
    double x = 0.0, pr = 1.0;
    if (n > 0) {
      if (b > 0) {
        const double cin = carry(fv, fp, b, kk, 1);
        double pf = 1.0;
        sweep(kk, r0, n, 1, [&](int32_t r, double y, double iv) {
          pf = pf * (g * iv);
          Y[r * MP + kk] = __builtin_fma(pf, cin, y);
        });
      }
      sweep(kk, r0 + n - 1, n, -1, [&](int32_t r, double dv, double iv) {
        const double a = g * iv;
        x = __builtin_fma(a, x, dv);
        pr = pr * a;
        Y[r * MP + kk] = x;
      });
    }
    bv[b * MP + kk] = x;
    bp[b * MP + kk] = pr;
  }
  __syncthreads();
  // backward carries (the last block has none)
  for (int32_t e = tid; e < B * nm; e += nt) {
    const int32_t b = e / nm, kk = e - b * nm, r0 = b * m, n = min(m, R - r0);
    if (n <= 0 || b == B - 1) continue;
    const double cin = carry(bv, bp, b, kk, -1);
    double pr = 1.0;
    sweep(kk, r0 + n - 1, n, -1, [&](int32_t r, double x, double iv) {
      pr = pr * (g * iv);
      Y[r * MP + kk] = __builtin_fma(pr, cin, x);
    });
  }
  __syncthreads();
  // the pairs' folded rows into the global store's blocked layout
  for (int32_t e = tid; e < R * nh; e += nt) {
    const int32_t r = e / nh, j = e - r * nh, i = i0 + j;
    const double x = Y[r * MP + j];
    double a = x, b = 0.0;
    if (2 * i + 1 != C) {
      const double y = Y[r * MP + nh + j];
      a = x + y;
      b = x - y;
    }
    const int64_t at = (static_cast<int64_t>(i >> 2) * R + r) * 4 + (i & 3);
    zs.wr(e0 + at, a);
    zs.wr(o0 + at, b);
  }
}

template <class Z>
__device__ __forceinline__ void lattice_tridiag(const DevProblem& P, const Z& zs) {
  if constexpr (std::is_same<Z, SplitStore>::value) {
    if (P.lat_mp) {
      lattice_tridiag_parts(P, zs);
      return;
    }
  }
  constexpr int TB = kTriRows;
  const int32_t R = P.lat_rows, C = P.lat_cols, CP = P.lat_cp;
  const GAS double* __restrict__ inv = gbl(P.lat_inv);
  const double g = P.lat_g;
  const int32_t B = lattice_blocks(P), m = (R + B - 1) / B;
  // forward and backward block ends (value, product) in the free folded-row
  // area: the second phase reads forward ends while other blocks write their
  // backward ends
  const int64_t fv = P.lat_t0, fp = fv + static_cast<int64_t>(B) * C;
  const int64_t bv = fp + static_cast<int64_t>(B) * C, bp = bv + static_cast<int64_t>(B) * C;
  auto zi = [&](int32_t r, int32_t k) { return static_cast<int64_t>(r) * C + k; };
  // one pass over `count` rows of mode k from `first` in direction dir (+1
  // up, -1 down): f(r, y, a) for each row, rows loaded TB at a time
  auto sweep = [&](int32_t k, int32_t first, int32_t count, int32_t dir, auto&& f) {
    for (int32_t c0 = 0; c0 < count; c0 += TB) {
      double y[TB], a[TB];
#pragma unroll
      for (int q = 0; q < TB; ++q) {
        const int32_t r = first + dir * min(c0 + q, count - 1);
        y[q] = zs.rd(zi(r, k));
        a[q] = inv[static_cast<int64_t>(r) * CP + k];
      }
#pragma unroll
      for (int q = 0; q < TB; ++q)
        if (c0 + q < count) f(first + dir * (c0 + q), y[q], a[q]);
    }
  };
  // forward from zero (an empty block at the end passes its carry through:
  // value 0, product 1)
  for (int32_t e = zs.vt; e < B * C; e += zs.vbs) {
    const int32_t b = e / C, k = e - b * C, r0 = b * m, n = min(m, R - r0);
    double d = 0.0, pr = 1.0;
    if (n > 0)
      sweep(k, r0, n, 1, [&](int32_t r, double y, double iv) {
        d = __builtin_fma(g, d, y) * iv;
        pr = pr * (g * iv);
        zs.wr(zi(r, k), d);
      });
    zs.wr(fv + e, d);
    zs.wr(fp + e, pr);
  }
  zs.barrier();
  // forward carries into the rows, then backward from zero, top row down (the
  // same thread wrote the rows it reads back)
  for (int32_t e = zs.vt; e < B * C; e += zs.vbs) {
    const int32_t b = e / C, k = e - b * C, r0 = b * m, n = min(m, R - r0);
    double x = 0.0, pr = 1.0;
    if (n > 0) {
      if (b > 0) {
        const double cin = lattice_carry(zs, C, B, fv, fp, b, k, 1);
        double pf = 1.0;
        sweep(k, r0, n, 1, [&](int32_t r, double y, double iv) {
          pf = pf * (g * iv);
          zs.wr(zi(r, k), __builtin_fma(pf, cin, y));
        });
      }
      sweep(k, r0 + n - 1, n, -1, [&](int32_t r, double dv, double iv) {
        const double a = g * iv;
        x = __builtin_fma(a, x, dv);
        pr = pr * a;
        zs.wr(zi(r, k), x);
      });
    }
    zs.wr(bv + e, x);
    zs.wr(bp + e, pr);
  }
  zs.barrier();
  // backward carries into the rows
  for (int32_t e = zs.vt; e < B * C; e += zs.vbs) {
    const int32_t b = e / C, k = e - b * C, r0 = b * m, n = min(m, R - r0);
    if (n <= 0 || b == B - 1) continue;
    const double cin = lattice_carry(zs, C, B, bv, bp, b, k, -1);
    double pr = 1.0;
    sweep(k, r0 + n - 1, n, -1, [&](int32_t r, double x, double iv) {
      pr = pr * (g * iv);
      zs.wr(zi(r, k), __builtin_fma(pr, cin, x));
    });
  }
}

template <class Z>
__device__ __forceinline__ void solve_lattice(const DevProblem& P, const Z& zs) {
  // a split column's part-local tridiagonal solve also writes the second fold
  bool folded = false;
  if constexpr (std::is_same<Z, SplitStore>::value) folded = P.lat_mp != 0;
  lattice_fold(P, zs);
  zs.barrier();
  lattice_transform(P, zs);
  zs.barrier();
  lattice_tridiag(P, zs);
  zs.barrier();
  if (!folded) {
    lattice_fold(P, zs);
    zs.barrier();
  }
  lattice_transform(P, zs);
  zs.barrier();
}

// K^-1 b of the face vector in place: the lattice solve or the factor program.
template <class Z>
__device__ __forceinline__ void solve_face_system(const DevProblem& P, const Z& zs) {
  if constexpr (RunsLattice<Z>::value) {
    if (P.lat_rows) {
      if constexpr (!Z::kGlobal) {
        if (P.lat_ld) {
          solve_lattice_padded(P, zs);
          return;
        }
      }
      solve_lattice(P, zs);
      return;
    }
  }
  solve(P, zs);
}

// Two columns of one problem through the same record (their face stores za and
// zb): each column's gathers, sums and writes are exactly those of
// process_slice, so each column's results are bit-identical to a solve of its
// own; the record's values and indices are loaded once for both.
template <class Z>
__device__ __forceinline__ void process_slice_pair(const Z& za, const Z& zb, int32_t Nf, int lane,
                                                   const jja_slice& m, const SliceRegs<Z::kGlobal>& r,
                                                   double& acca, double& accb) {
  double va[kMaxIter], vb[kMaxIter];
#pragma unroll
  for (int i = 0; i < kMaxIter; ++i) {
    const uint32_t ix = record_index(r, m.flags, i);
    va[i] = za.gather(ix);
    vb[i] = zb.gather(ix);
  }
#pragma unroll
  for (int i = 0; i < kMaxIter; ++i) {
    acca = __builtin_fma(r.v[i], va[i], acca);
    accb = __builtin_fma(r.v[i], vb[i], accb);
  }
  if (m.flags & JJA_SLICE_FINISH) {
    const int G = m.flags & 0xff;
    acca = group_sum_last(acca, G);
    accb = group_sum_last(accb, G);
    const int slot = lane >> __builtin_ctz(static_cast<unsigned>(G));
    if (slot < (m.flags >> 16) && r.row >= 0 && (lane & (G - 1)) == G - 1) {
      if (m.flags & JJA_SLICE_BLOCK) {
        za.wr(r.row, acca);
        zb.wr(r.row, accb);
      } else {
        za.wr(Nf + r.row - m.r0, za.rd(r.row) - acca);
        zb.wr(Nf + r.row - m.r0, zb.rd(r.row) - accb);
      }
    }
    acca = 0.0;
    accb = 0.0;
  }
  if (m.flags & JJA_SLICE_BARRIER)
    za.barrier();
  else if (m.flags & JJA_SLICE_WG_BARRIER)
    za.wg_barrier();
}

// solve() for two columns that share one set of threads and one barrier (za's).
template <class Z>
__device__ __forceinline__ void solve_pair(const DevProblem& P, const Z& za, const Z& zb) {
  constexpr bool GLOBAL = Z::kGlobal;
  const int lane = za.vt & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(za.vt / kWave);
  const CAS int32_t* wp = (const CAS int32_t*)(P.wave_ptr) + wave;
  const int32_t k0 = __builtin_amdgcn_readfirstlane(wp[0]);
  const int32_t nk = __builtin_amdgcn_readfirstlane(wp[1]) - k0 - 4;
  const jja_slice* __restrict__ prog = P.solve_slices + k0;
  jja_slice m0 = load_rec(prog, 0), m1 = load_rec(prog, 1), m2 = load_rec(prog, 2);
  const __amdgpu_buffer_rsrc_t vres = value_resource(P);
  SliceRegs<GLOBAL> A, B, C;
  load_slice(P, vres, m0, lane, A);
  load_slice(P, vres, m1, lane, B);
  double acca = 0.0, accb = 0.0;
  for (int32_t k = 0; k < nk; k += 3) {
    const jja_slice m3 = load_rec(prog, k + 3);
    load_slice(P, vres, m2, lane, C);
    __builtin_amdgcn_sched_barrier(0);
    process_slice_pair(za, zb, P.Nf, lane, m0, A, acca, accb);
    const jja_slice m4 = load_rec(prog, k + 4);
    load_slice(P, vres, m3, lane, A);
    __builtin_amdgcn_sched_barrier(0);
    process_slice_pair(za, zb, P.Nf, lane, m1, B, acca, accb);
    const jja_slice m5 = load_rec(prog, k + 5);
    load_slice(P, vres, m4, lane, B);
    __builtin_amdgcn_sched_barrier(0);
    process_slice_pair(za, zb, P.Nf, lane, m2, C, acca, accb);
    m0 = m3;
    m1 = m4;
    m2 = m5;
  }
}

// One input term of one column at one step: element i is p[i * si] * amp.
// amp is exactly 1 for a term without amplitude; a term that is absent reads
// an exact +0.0 from the plan's zero page (si = 0), which leaves every sum it
// enters bit-identical to skipping it.
struct TermView {
  const GAS double* p;
  int64_t si;
  double amp;
};

__device__ __forceinline__ TermView term_view(const jja_source& s, bool present, const double* zero,
                                              int64_t w, int64_t t) {
  TermView v{gbl(zero), 0, 1.0};
  if (present && s.base) {
    const int64_t tt = t - s.t0;
    v.p = gbl(s.base) + w * s.s_w + tt * s.s_t;
    v.si = s.s_i;
    if (s.amp) v.amp = gbl(s.amp)[w * s.a_w + tt * s.a_t];
  }
  return v;
}

__device__ __forceinline__ double term_at(const TermView& v, int32_t i) {
  return v.p[static_cast<int64_t>(i) * v.si] * v.amp;
}

// Face phase: b_p = sum +-u_j in ascending j, minus 2 pi f (time_evolution.py:560-569).
// A face longer than one record continues in the next record (flag FINISH on
// its last one). Records go in groups of kFaceGroup: the code, row and face
// loads of the group are issued together, then its u gathers and flux values,
// so a group costs two memory round trips.
struct FaceRec {
  int32_t cd[kFaceIter];  // +-junction codes, -1 past the face's length
  int32_t pos;            // store address written at FINISH, or -1
  int32_t fid;            // face index of that position (flux input), or -1
  bool finish;
};

__device__ __forceinline__ void face_rec_load(const DevProblem& P, int32_t k, bool present, int tid,
                                              int32_t vbs, FaceRec& r) {
  const jja_slice m = load_rec(P.face_slices, k);
  const bool live = present && tid < (m.flags >> 16);
  const GAS int32_t* __restrict__ code = gbl(P.face_code) + m.base + tid;
#pragma unroll
  for (int i = 0; i < kFaceIter; ++i) r.cd[i] = (live && i < m.n_iter) ? code[i * vbs] : -1;
  r.finish = present && (m.flags & JJA_SLICE_FINISH);
  const bool rowed = live && r.finish;
  r.pos = rowed ? gbl(P.face_addr)[m.rowbase + tid] : -1;
  r.fid = rowed ? gbl(P.face_fid)[m.rowbase + tid] : -1;
}

// The junction values u_j the face phase sums: u itself (an LDS store's
// evolution, whose junction pass writes u, and the adjoint), or, for a global
// store, formed from the step's x as the junction pass would have: x_j / c0 (a
// product with the reciprocal), less theta_s with voltage sources; one write
// stream fewer per junction. rc0u is 1/c0 when every junction has the same
// (read once).
struct JuncSource {
  const GAS double* v;
  const GAS double* ths;
  bool scaled;
  double rc0u;
};

// MODE 0: u itself; 1: x / c0 with one c0; 2: x / c0 per junction; 3: x / c0
// per junction less theta_s
template <int MODE>
__device__ __forceinline__ double junc_value(const DevProblem& P, const JuncSource& s, int32_t j) {
  if constexpr (MODE == 0) return s.v[j];
  if constexpr (MODE == 1) return s.v[j] * s.rc0u;
  if constexpr (MODE == 2) return s.v[j] * rc0_at(P, j);
  return s.v[j] * rc0_at(P, j) - s.ths[j];
}

template <int BS, int MODE, class Z>
__device__ __forceinline__ void face_phase_impl(const DevProblem& P, const jja_source* f, const JuncSource& us,
                                                const Z& zs, int64_t w, int64_t t) {
  const int tid = zs.vt;
  // flux of face q at this step is fv.p[q * fv.si] * fv.amp; an absent flux
  // reads an exact zero, and acc - 2 pi * 0 leaves acc unchanged
  const TermView fv = term_view(f ? *f : jja_source{}, f && !f->zero, P.zero, w, t);
  double acc = 0.0;
  const int32_t n = P.n_face_slices;
  for (int32_t k = 0; k < n; k += kFaceGroup) {
    FaceRec r[kFaceGroup];
#pragma unroll
    for (int g = 0; g < kFaceGroup; ++g)
      face_rec_load(P, k + g < n ? k + g : k, k + g < n, tid, zs.vbs, r[g]);
    double uu[kFaceGroup][kFaceIter], fq[kFaceGroup];
#pragma unroll
    for (int g = 0; g < kFaceGroup; ++g) {
#pragma unroll
      for (int i = 0; i < kFaceIter; ++i)
        uu[g][i] = r[g].cd[i] >= 0 ? junc_value<MODE>(P, us, r[g].cd[i] >> 1) : 0.0;
      fq[g] = r[g].fid >= 0 ? term_at(fv, r[g].fid) : 0.0;
    }
#pragma unroll
    for (int g = 0; g < kFaceGroup; ++g) {
#pragma unroll
      for (int i = 0; i < kFaceIter; ++i)
        if (r[g].cd[i] >= 0) acc = (r[g].cd[i] & 1) ? acc - uu[g][i] : acc + uu[g][i];
      if (r[g].finish) {
        if (r[g].pos >= 0) {
          acc = acc - kTwoPi * fq[g];
          zs.wr(r[g].pos, acc);
          if (r[g].pos < P.copy_rows) zs.wr(P.Nf + r[g].pos, acc);  // first stage: scratch = b
        }
        acc = 0.0;
      }
    }
  }
}

template <int BS, class Z>
__device__ __forceinline__ void face_phase(const DevProblem& P, const jja_source* f, JuncSource us, const Z& zs,
                                           int64_t w, int64_t t) {
  if (!us.scaled) {
    face_phase_impl<BS, 0>(P, f, us, zs, w, t);
  } else if (us.ths) {
    face_phase_impl<BS, 3>(P, f, us, zs, w, t);
  } else if (P.coef_si == 0) {
    us.rc0u = rc0_at(P, 0);
    face_phase_impl<BS, 1>(P, f, us, zs, w, t);
  } else {
    face_phase_impl<BS, 2>(P, f, us, zs, w, t);
  }
}

// Everything one junction pass needs that is the same for all its junctions.
struct JunctionStep {
  GAS double* th_n;            // slot of step t: holds x_t, receives theta_t
  const GAS double* th_k[4];   // theta_{tx-1-k}, k = 0..S-1 (k = 0 unused with UPDATE)
  GAS double* th_x;            // slot of step tx: receives x_tx
  GAS double* ths;             // voltage-source phase (NULL without Vs)
  GAS double* u;               // LDS store: receives u = x_tx/c0 - theta_s (global store: NULL)
  GAS double* th_out;          // stored theta_t row or NULL
  GAS double* I_out;           // stored current row or NULL
  TermView Is_t, Vs_t;         // step t (update)
  TermView Is_x, sig_x;        // step tx (prep); sig_x is sigma, or T when from_T
  const GAS double* noise;     // reference normals of step tx, or NULL
  const GAS double* Ic;        // critical currents (the run's, else the plan's)
  bool is_zero, t_zero, from_T;
  double dt;
  uint64_t seed;
  uint32_t noise_col;
  uint64_t tx;
  int32_t vt, vbs;             // the thread's index in the column, the column's thread count
};

// ---------------------------------------------------------------- general
// One junction, all options: with UPDATE finish step t (time_evolution.py:
// 560-580): y = A^T J from the face vector, theta_t = (y - x)/c0, stored
// outputs, theta_s += Vs dt; with PREP form x of step tx (time_evolution.py:
// 533-558) and write x to the history slot, and for an LDS store u = x/c0 -
// theta_s to the scratch (a global store's face phase forms u from x). All
// loads are issued before any arithmetic.
template <int SW, bool UPDATE, bool PREP, class Z>
__device__ __forceinline__ void junction_one(const DevProblem& P, const JunctionStep& J,
                                             const Z& zs, int32_t j, double zj) {
  const double rc0 = rc0_at(P, j);
  vint2 code{-1, -1};
  double xo = 0.0, isn = 0.0, thsv = 0.0, vsv = 0.0;
  if (UPDATE) {
    code = gbl(reinterpret_cast<const vint2*>(P.junc_code))[j];
    xo = J.th_n[j];
    if (J.I_out) isn = term_at(J.Is_t, j);
    if (J.ths) vsv = term_at(J.Vs_t, j);
  }
  if (J.ths) thsv = J.ths[j];
  double t[4] = {0.0, 0.0, 0.0, 0.0}, c[SW], Ic = 0.0, isx = 0.0, sg = 0.0, rv = 0.0;
  if (PREP) {
#pragma unroll
    for (int k = UPDATE ? 1 : 0; k < SW - 1; ++k) t[k] = J.th_k[k][j];
    Ic = J.Ic[j];
#pragma unroll
    for (int k = 1; k < SW; ++k) c[k] = coef_at(P, k, j);
    isx = term_at(J.Is_x, j);
    sg = term_at(J.sig_x, j);
    if (J.from_T) rv = gbl(P.Rv)[j];
    if (J.noise) zj = J.noise[j];
  }
  if (UPDATE) {
    double y = 0.0;
    if (code.x >= 0) y = (code.x & 1) ? y - zs.rd(code.x >> 1) : y + zs.rd(code.x >> 1);
    if (code.y >= 0) y = (code.y & 1) ? y - zs.rd(code.y >> 1) : y + zs.rd(code.y >> 1);
    t[0] = (y - xo) * rc0;
    J.th_n[j] = t[0];
    if (J.th_out) J.th_out[j] = t[0];
    if (J.I_out) J.I_out[j] = y + isn;
    if (J.ths) {
      thsv += vsv * J.dt;
      J.ths[j] = thsv;
    }
  }
  if (PREP) {
    double X;
    if constexpr (SW == 3) {
      X = Ic * cpr_sum(P, 2.0 * t[0] - t[1]) + c[1] * t[0] + c[2] * t[1];
    } else if constexpr (SW == 4) {
      X = Ic * cpr_sum(P, 3.0 * t[0] - 3.0 * t[1] + t[2]) + c[1] * t[0] + c[2] * t[1] + c[3] * t[2];
    } else {
      X = Ic * cpr_sum(P, 4.0 * t[0] - 6.0 * t[1] + 4.0 * t[2] - t[3]) + c[1] * t[0] + c[2] * t[1] +
          c[3] * t[2] + c[4] * t[3];
    }
    double eta = 0.0;
    if (!J.t_zero) eta = (J.from_T ? sqrt(2.0 * sg * rv) : sg) * zj;
    const double x = J.is_zero ? eta + X : (eta - isx) + X;
    J.th_x[j] = x;
    if constexpr (!Z::kGlobal) {
      double uj = x * rc0;
      if (J.ths) uj = uj - thsv;
      J.u[j] = uj;
    }
  }
}

// Deviate of this lane's junction from a Philox pair computed by another lane
// of the wave: lane `src` holds (z0, z1) for junctions (2i, 2i+1); `second`
// picks z1.
__device__ __forceinline__ double take_normal(double z0, double z1, int src, bool second) {
  const long long b0 = __builtin_bit_cast(long long, z0), b1 = __builtin_bit_cast(long long, z1);
  const int a = src << 2;
  const int lo0 = __builtin_amdgcn_ds_bpermute(a, static_cast<int>(b0));
  const int hi0 = __builtin_amdgcn_ds_bpermute(a, static_cast<int>(b0 >> 32));
  const int lo1 = __builtin_amdgcn_ds_bpermute(a, static_cast<int>(b1));
  const int hi1 = __builtin_amdgcn_ds_bpermute(a, static_cast<int>(b1 >> 32));
  const int lo = second ? lo1 : lo0, hi = second ? hi1 : hi0;
  return __builtin_bit_cast(double, static_cast<long long>(static_cast<unsigned>(lo)) |
                                        (static_cast<long long>(hi) << 32));
}

// Normals for the junctions k*BS + tid and (k+1)*BS + tid of this lane. Each
// Philox pair (junctions 2i, 2i+1) is drawn once: lanes 0..31 of a wave draw
// the 32 pairs its 64 junctions of iteration k form, lanes 32..63 those of
// iteration k+1, and every lane then fetches its own deviate. All lanes of the
// wave take part, whether or not their junctions exist.
template <int BS>
__device__ __forceinline__ void wave_normals(const JunctionStep& J, int32_t k, double& zA, double& zB) {
  const int lane = J.vt & 63;
  const int32_t wave_base = J.vt - lane;
  const int32_t it = lane < 32 ? k : k + 1;
  const int32_t j_even = it * J.vbs + wave_base + 2 * (lane & 31);
  double z0, z1;
  normal_pair(J.seed, static_cast<uint32_t>(j_even), J.noise_col, J.tx, &z0, &z1);
  zA = take_normal(z0, z1, lane >> 1, lane & 1);
  zB = take_normal(z0, z1, 32 + (lane >> 1), lane & 1);
}

// The junction pass, general form: thread tid takes junctions k*BS + tid
// (consecutive lanes, consecutive junctions), two iterations at a time.
template <int BS, int SW, bool UPDATE, bool PREP, class Z>
__device__ __forceinline__ void junction_loop(const DevProblem& P, const JunctionStep& J, const Z& zs) {
  const int32_t Nj = P.Nj;
  const int32_t tid = J.vt, vbs = J.vbs;
  const bool gauss = PREP && !J.t_zero && !J.noise;
  for (int32_t k = 0; k * vbs < Nj; k += 2) {
    double zA = 0.0, zB = 0.0;
    if (gauss) wave_normals<BS>(J, k, zA, zB);
    const int32_t jA = k * vbs + tid, jB = jA + vbs;
    if (jA < Nj) junction_one<SW, UPDATE, PREP, Z>(P, J, zs, jA, zA);
    // keep the two junctions apart: interleaving them would double the live
    // registers and spill
    __builtin_amdgcn_sched_barrier(0);
    if (jB < Nj) junction_one<SW, UPDATE, PREP, Z>(P, J, zs, jB, zB);
  }
}

// ------------------------------------------------------------ common step
// The usual step (stencil 3, no voltage sources, nothing stored at step t,
// noise amplitude given per junction, Philox or no noise): the same
// arithmetic as junction_one, each lane taking a junction pair, with the loads
// of both junctions issued first and the pair's Philox draw computed while
// they are in flight. (Loading the next pair's face codes an iteration ahead,
// so that the face-store gathers could go out with the other loads, made the
// split kernel spill and was 3.6% slower on SquareArray(512,512).)
struct JFast {
  vint2 code;
  double rc0, xo, t2, c1, c2, Ic, isx, sg;
};

// UNI: 1/c0, c1, c2 and sigma are one value each (uniform R and C, constant
// T): read once before the loop (scalar registers), not per junction
template <bool UNI>
__device__ __forceinline__ void jfast_load(const DevProblem& P, const JunctionStep& J, int32_t j, JFast& L) {
  L.code = gbl(reinterpret_cast<const vint2*>(P.junc_code))[j];
  L.xo = J.th_n[j];
  L.t2 = J.th_k[1][j];
  L.Ic = J.Ic[j];
  L.isx = term_at(J.Is_x, j);
  if constexpr (!UNI) {
    L.rc0 = rc0_at(P, j);
    L.c1 = coef_at(P, 1, j);
    L.c2 = coef_at(P, 2, j);
    L.sg = term_at(J.sig_x, j);
  }
}

template <class Z>
__device__ __forceinline__ void jfast_compute(const DevProblem& P, const JunctionStep& J, const Z& zs, int32_t j,
                                              const JFast& L, double z) {
  double y = 0.0;
  if (L.code.x >= 0) y = (L.code.x & 1) ? y - zs.rd(L.code.x >> 1) : y + zs.rd(L.code.x >> 1);
  if (L.code.y >= 0) y = (L.code.y & 1) ? y - zs.rd(L.code.y >> 1) : y + zs.rd(L.code.y >> 1);
  const double t1 = (y - L.xo) * L.rc0;
  J.th_n[j] = t1;
  const double X = L.Ic * cpr_sum(P, 2.0 * t1 - L.t2) + L.c1 * t1 + L.c2 * L.t2;
  double eta = 0.0;
  if (!J.t_zero) eta = L.sg * z;
  const double x = J.is_zero ? eta + X : (eta - L.isx) + X;
  J.th_x[j] = x;
  if constexpr (!Z::kGlobal) J.u[j] = x * L.rc0;
}

template <int BS, bool UNI, class Z>
__device__ __forceinline__ void junction_loop_fast(const DevProblem& P, const JunctionStep& J, const Z& zs) {
  const int32_t Nj = P.Nj;
  double u_rc0 = 0.0, u_c1 = 0.0, u_c2 = 0.0, u_sg = 0.0;
  if constexpr (UNI) {
    u_rc0 = rc0_at(P, 0);
    u_c1 = coef_at(P, 1, 0);
    u_c2 = coef_at(P, 2, 0);
    u_sg = term_at(J.sig_x, 0);
  }
  const int32_t tid = J.vt, vbs = J.vbs;
  const int32_t last = Nj - 1;
  const bool gauss = !J.t_zero;
  // a lane takes the junction pair (2q, 2q+1): its own Philox draw gives both
  // deviates (the pair's counter, as in the general loop); a pair past the
  // end (odd Nj) reads the last junction and does not use it
  for (int32_t q = tid; 2 * q < Nj; q += vbs) {
    const int32_t jA = 2 * q, jB = jA + 1;
    JFast A, B;
    jfast_load<UNI>(P, J, jA, A);
    jfast_load<UNI>(P, J, min(jB, last), B);
    if constexpr (UNI) {
      A.rc0 = B.rc0 = u_rc0;
      A.c1 = B.c1 = u_c1;
      A.c2 = B.c2 = u_c2;
      A.sg = B.sg = u_sg;
    }
    __builtin_amdgcn_sched_barrier(0);
    // the Philox draw runs while the loads are in flight
    double zA = 0.0, zB = 0.0;
    if (gauss) normal_pair(J.seed, static_cast<uint32_t>(jA), J.noise_col, J.tx, &zA, &zB);
    jfast_compute(P, J, zs, jA, A, zA);
    if (jB < Nj) jfast_compute(P, J, zs, jB, B, zB);
  }
}

// Set up and run one junction pass (finish step t if `update`, prepare step tx
// if `prep`) for column w.
template <int BS, int SW, class Z>
__device__ __forceinline__ void junction_pass(const DevProblem& P, const jja_problem_run& R,
                                              GAS double* __restrict__ th, GAS double* __restrict__ ths,
                                              GAS double* __restrict__ u, const Z& zs,
                                              int64_t w, size_t slot_stride, int64_t t, bool update,
                                              int64_t tx, bool prep, uint32_t noise_col) {
  constexpr int32_t S = SW - 1;
  auto slot = [&](int64_t m) -> size_t {
    int64_t r = m % S;
    return static_cast<size_t>(r < 0 ? r + S : r) * slot_stride;
  };
  JunctionStep J;
  J.vt = zs.vt;
  J.vbs = zs.vbs;
  J.th_n = th + slot(t);
#pragma unroll
  for (int k = 0; k < 4; ++k) J.th_k[k] = th + (k < S ? slot(tx - 1 - k) : 0);
  J.th_x = th + slot(tx);
  J.ths = ths;
  J.u = u;
  const size_t col = static_cast<size_t>(w) * P.Nj;
  const int32_t tho = (update && R.th_slot) ? gbl(R.th_slot)[t - R.slot_t0] : -1;
  const int32_t Io = (update && R.I_slot) ? gbl(R.I_slot)[t - R.slot_t0] : -1;
  J.th_out = tho >= 0 ? gblw(R.th_out) + static_cast<size_t>(tho) * slot_stride + col : nullptr;
  J.I_out = Io >= 0 ? gblw(R.I_out) + static_cast<size_t>(Io) * slot_stride + col : nullptr;
  J.Is_t = term_view(R.Is, update, P.zero, w, t);
  J.Vs_t = term_view(R.Vs, update && ths, P.zero, w, t);
  J.Is_x = term_view(R.Is, prep, P.zero, w, tx);
  J.t_zero = R.T.zero;
  J.from_T = !R.sigma.base;
  J.sig_x = term_view(J.from_T ? R.T : R.sigma, prep && !R.T.zero, P.zero, w, tx);
  J.noise = (prep && !R.T.zero && R.noise)
                ? gbl(R.noise) + static_cast<size_t>(tx - R.noise_t0) * slot_stride + col
                : nullptr;
  J.Ic = gbl(R.Ic ? R.Ic : P.Ic);
  J.is_zero = R.Is.zero;
  J.dt = R.dt;
  J.seed = R.seed;
  J.noise_col = noise_col;
  J.tx = static_cast<uint64_t>(tx);
  const bool fast = SW == 3 && update && prep && !ths && !J.th_out && !J.I_out && !J.noise && !J.from_T;
  if (fast && P.coef_si == 0 && J.sig_x.si == 0) junction_loop_fast<BS, true, Z>(P, J, zs);
  else if (fast) junction_loop_fast<BS, false, Z>(P, J, zs);
  else if (update && prep) junction_loop<BS, SW, true, true, Z>(P, J, zs);
  else if (update) junction_loop<BS, SW, true, false, Z>(P, J, zs);
  else if (prep) junction_loop<BS, SW, false, true, Z>(P, J, zs);
}

// The face phase's junction values of step t: x_t, in history slot t mod
// (SW - 1), written by the junction pass before it.
__device__ __forceinline__ JuncSource step_source(const GAS double* th, const GAS double* ths,
                                                 size_t slot_stride, int SW, int64_t t) {
  return JuncSource{th + static_cast<size_t>(t % (SW - 1)) * slot_stride, ths, true, 0.0};
}

// n_steps steps of column w of one problem, by the threads the store names.
template <int BS, int SW, class Z>
__device__ __forceinline__ void evolve_steps(const DevProblem& P, const jja_problem_run& R, int64_t w,
                                             const Z& zs, int32_t n_steps, int64_t step0) {
  const size_t slot_stride = static_cast<size_t>(R.W) * P.Nj;
  GAS double* __restrict__ th = gblw(R.theta) + static_cast<size_t>(w) * P.Nj;
  GAS double* __restrict__ ths = R.theta_s ? gblw(R.theta_s) + static_cast<size_t>(w) * P.Nj : nullptr;
  GAS double* __restrict__ u = Z::kGlobal ? nullptr : gblw(R.u) + static_cast<size_t>(w) * P.Nj;
  const uint32_t noise_col = static_cast<uint32_t>(R.column_offset + w);

  junction_pass<BS, SW>(P, R, th, ths, u, zs, w, slot_stride, step0, false, step0, true, noise_col);
  zs.sync();
  for (int32_t n = 0; n < n_steps; ++n) {
    const int64_t t = step0 + n;
    if (P.Nf > 0) {  // a circuit without faces has nothing to solve (K is 0 x 0)
      face_phase<BS>(P, &R.f, Z::kGlobal ? step_source(th, ths, slot_stride, SW, t) : JuncSource{u, nullptr, false, 0.0},
                     zs, w, t);
      zs.barrier();
      solve_face_system(P, zs);
    }
    // finish step t and prepare step t+1 in one pass
    junction_pass<BS, SW>(P, R, th, ths, u, zs, w, slot_stride, t, true, t + 1, n + 1 < n_steps, noise_col);
    zs.sync();
  }
}

// Columns wa and wa+1 (two) or wa alone of one problem, worked by one set of
// threads: the face phases and junction passes run column by column, the solve
// streams each record once for both, and za's barriers serve both.
template <int BS, int SW>
__device__ __forceinline__ void evolve_steps_pair(const DevProblem& P, const jja_problem_run& R, int64_t wa,
                                                  bool two, const SplitStore& za, const SplitStore& zb,
                                                  int32_t n_steps, int64_t step0) {
  const size_t slot_stride = static_cast<size_t>(R.W) * P.Nj;
  const int64_t wb = wa + 1;
  const size_t ca = static_cast<size_t>(wa) * P.Nj, cb = two ? static_cast<size_t>(wb) * P.Nj : ca;
  // column b's arrays alias column a's when it is alone (and are then unused)
  GAS double* tha = gblw(R.theta) + ca;
  GAS double* thb = gblw(R.theta) + cb;
  GAS double* thsa = R.theta_s ? gblw(R.theta_s) + ca : nullptr;
  GAS double* thsb = R.theta_s ? gblw(R.theta_s) + cb : nullptr;
  const uint32_t na = static_cast<uint32_t>(R.column_offset + wa), nb = static_cast<uint32_t>(R.column_offset + wb);

  junction_pass<BS, SW>(P, R, tha, thsa, nullptr, za, wa, slot_stride, step0, false, step0, true, na);
  if (two) junction_pass<BS, SW>(P, R, thb, thsb, nullptr, zb, wb, slot_stride, step0, false, step0, true, nb);
  za.sync();
  for (int32_t n = 0; n < n_steps; ++n) {
    const int64_t t = step0 + n;
    if (P.Nf > 0) {
      face_phase<BS>(P, &R.f, step_source(tha, thsa, slot_stride, SW, t), za, wa, t);
      if (two) face_phase<BS>(P, &R.f, step_source(thb, thsb, slot_stride, SW, t), zb, wb, t);
      za.barrier();
      if (two)
        solve_pair(P, za, zb);
      else
        solve(P, za);
    }
    const bool prep = n + 1 < n_steps;
    junction_pass<BS, SW>(P, R, tha, thsa, nullptr, za, wa, slot_stride, t, true, t + 1, prep, na);
    if (two) junction_pass<BS, SW>(P, R, thb, thsb, nullptr, zb, wb, slot_stride, t, true, t + 1, prep, nb);
    za.sync();
  }
}

// Column w of one problem in one workgroup: face vector by solve position,
// stage scratch after it.
template <int BS, int SW, bool GLOBAL>
__device__ __forceinline__ void evolve_column(const DevProblem& P, const jja_problem_run& R, int64_t w,
                                              double* lds, int32_t n_steps, int64_t step0) {
  FaceStore<GLOBAL> zs;
  if constexpr (GLOBAL)
    zs.p = gblw(R.zbuf) + static_cast<size_t>(w) * (static_cast<size_t>(P.Nf) + P.max_stage_rows);
  else
    zs.p = lds;
  zs.vt = threadIdx.x;
  zs.vbs = BS;
  if constexpr (!GLOBAL) init_store(P, lds, threadIdx.x, BS);
  evolve_steps<BS, SW>(P, R, w, zs, n_steps, step0);
}

// A column shared by P.parts workgroups (part `part` of the work item's column
// w): face vector in global memory, a column barrier wherever the one-workgroup
// kernel has a workgroup barrier.
__device__ __forceinline__ SplitStore split_store(const DevProblem& P, GAS double* zbuf, int64_t w,
                                                  int32_t part, uint32_t* ctrs, const WorkItem& wi,
                                                  int32_t* err, uint32_t wait_limit, int32_t* stopped,
                                                  int BS, LAS double* lds) {
  SplitStore zs;
  zs.p = zbuf + static_cast<size_t>(w) * (static_cast<size_t>(P.Nf) + P.max_stage_rows);
  zs.vt = part * BS + static_cast<int32_t>(threadIdx.x);
  zs.vbs = P.parts * BS;
  zs.ctr = ctrs + 2 * static_cast<int64_t>(wi.slot);
  zs.xcds = zs.ctr + 1;
  zs.parts = static_cast<uint32_t>(P.parts);
  zs.wait_limit = wait_limit;
  zs.err = err;
  zs.stopped = stopped;
  zs.gen = 0;
  zs.one_xcd = false;
  zs.lds = lds;
  if (threadIdx.x == 0 && P.parts > 1)
    __hip_atomic_fetch_or(zs.xcds, 1u << xcd_id(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return zs;
}

// ------------------------------------------------------------------ adjoint
// Adjoint of theta_k wherever a run stores it: lam[m mod 2].
struct AdjCol {
  GAS double* lam;  // slot m mod 2 at lam + (m & 1) * stride
  const GAS double* g;  // this column of the upstream gradient (slot s at g + s * stride)
  GAS double* u;
  const GAS double* hist;
  int64_t hist_m0;
  size_t stride;
  const GAS double* Ic;
};

__device__ __forceinline__ double adj_g(const jja_adjoint_run& A, const AdjCol& C, int64_t m, int32_t j) {
  if (!A.g || m < A.g_lo || m >= A.g_hi) return 0.0;
  const int32_t sl = gbl(A.g_slot)[m - A.slot_t0];
  return sl >= 0 ? C.g[static_cast<size_t>(sl) * C.stride + j] : 0.0;
}

// lambda_k += g_k (complete) and u = lambda_k / c0: the first step of a sweep.
template <class Z>
__device__ __forceinline__ void adjoint_prime(const DevProblem& P, const jja_adjoint_run& A,
                                              const AdjCol& C, const Z& zs, int64_t k) {
  GAS double* __restrict__ lk = C.lam + (k & 1) * C.stride;
  for (int32_t j = zs.vt; j < P.Nj; j += zs.vbs) {
    const double l = lk[j] + adj_g(A, C, k, j);
    lk[j] = l;
    C.u[j] = l * rc0_at(P, j);
  }
}

// After the solve of step k (face vector J' = K^-1 A D lambda_k in LDS):
// mu_k = (A^T J' - lambda_k)/c0 and the updates of lambda_{k-1}, lambda_{k-2}
// and of the gradients; then lambda_{k-1} gets g_{k-1} and u = lambda_{k-1}/c0
// prepares step k-1.
template <class Z>
__device__ __forceinline__ void adjoint_junctions(const DevProblem& P, const jja_adjoint_run& A,
                                                  const AdjCol& C, const Z& zs, int64_t k, int64_t w) {
  const int32_t Nj = P.Nj;
  const GAS vint2* __restrict__ jcode = gbl(reinterpret_cast<const vint2*>(P.junc_code));
  GAS double* __restrict__ lk = C.lam + (k & 1) * C.stride;
  GAS double* __restrict__ lk1 = C.lam + ((k - 1) & 1) * C.stride;
  const GAS double* __restrict__ h1 = C.hist + static_cast<size_t>(k - 1 - C.hist_m0) * C.stride;
  const GAS double* __restrict__ h2 = C.hist + static_cast<size_t>(k - 2 - C.hist_m0) * C.stride;
  GAS double* __restrict__ gIc = gblw(A.grad_Ic) + static_cast<size_t>(w) * Nj;
  GAS double* __restrict__ gIs = gblw(A.grad_Is) + static_cast<size_t>(w) * Nj;
  for (int32_t j = zs.vt; j < Nj; j += zs.vbs) {
    const vint2 code = jcode[j];
    const double rc0 = rc0_at(P, j), c1 = coef_at(P, 1, j), c2 = coef_at(P, 2, j);
    const double lam = lk[j], lprev = lk1[j], t1 = h1[j], t2 = h2[j], Ic = C.Ic[j];
    const double gj = adj_g(A, C, k - 1, j);
    const double gi = gIc[j], gs = gIs[j];
    double y = 0.0;
    if (code.x >= 0) y = (code.x & 1) ? y - zs.rd(code.x >> 1) : y + zs.rd(code.x >> 1);
    if (code.y >= 0) y = (code.y & 1) ? y - zs.rd(code.y >> 1) : y + zs.rd(code.y >> 1);
    const double mu = (y - lam) * rc0;
    double sn, cs;
    jja_sincos(2.0 * t1 - t2, &sn, &cs);
    const double a = 2.0 * Ic * cs + c1, b = c2 - Ic * cs;
    gIc[j] = gi + sn * mu;
    gIs[j] = gs - mu;
    lk[j] = b * mu;  // slot k mod 2 now holds lambda_{k-2}'s partial sum
    const double l1 = (lprev + a * mu) + gj;
    lk1[j] = l1;
    C.u[j] = l1 * rc0;
  }
}

// The column of work item wi: lambda, history, gradients and upstream
// gradient of column w.
__device__ __forceinline__ AdjCol adjoint_column(const DevProblem& P, const jja_adjoint_run& A, int64_t w) {
  const size_t stride = static_cast<size_t>(A.W) * P.Nj;
  const size_t col = static_cast<size_t>(w) * P.Nj;
  AdjCol C;
  C.lam = gblw(A.lam) + col;
  C.g = A.g ? gbl(A.g) + col : nullptr;
  C.u = gblw(A.u) + col;
  C.hist = gbl(A.hist) + col;
  C.hist_m0 = A.hist_m0;
  C.stride = stride;
  C.Ic = gbl(A.Ic ? A.Ic : P.Ic);
  return C;
}

// Steps k_hi down to k_lo of the adjoint sweep of column w.
template <int BS, class Z>
__device__ __forceinline__ void adjoint_steps(const DevProblem& P, const jja_adjoint_run& A, int64_t w,
                                              const Z& zs, int64_t k_hi, int64_t k_lo) {
  const AdjCol C = adjoint_column(P, A, w);
  GAS double* __restrict__ gf = gblw(A.grad_f) + static_cast<size_t>(w) * P.Nf;
  if (A.prime) adjoint_prime(P, A, C, zs, k_hi);
  zs.sync();
  for (int64_t k = k_hi; k >= k_lo; --k) {
    if (P.Nf > 0) {
      face_phase<BS>(P, nullptr, JuncSource{C.u, nullptr, false, 0.0}, zs, w, k);
      zs.barrier();
      solve_face_system(P, zs);
    }
    for (int32_t p = zs.vt; p < P.Nf; p += zs.vbs)
      gf[p] = gf[p] - kTwoPi * zs.rd(Z::kGlobal ? p : store_address(P, p));
    adjoint_junctions(P, A, C, zs, k, w);
    zs.sync();
  }
}

// adjoint_steps for columns wa and wa+1 (two) or wa alone, on one set of
// threads: per-column face phases and junction updates, one shared solve, za's
// barriers.
template <int BS>
__device__ __forceinline__ void adjoint_steps_pair(const DevProblem& P, const jja_adjoint_run& A, int64_t wa,
                                                   bool two, const SplitStore& za, const SplitStore& zb,
                                                   int64_t k_hi, int64_t k_lo) {
  const int64_t wb = two ? wa + 1 : wa;
  const AdjCol Ca = adjoint_column(P, A, wa), Cb = adjoint_column(P, A, wb);
  // column b's gradient aliases column a's when it is alone (and is then unused)
  GAS double* gfa = gblw(A.grad_f) + static_cast<size_t>(wa) * P.Nf;
  GAS double* gfb = gblw(A.grad_f) + static_cast<size_t>(wb) * P.Nf;
  if (A.prime) {
    adjoint_prime(P, A, Ca, za, k_hi);
    if (two) adjoint_prime(P, A, Cb, zb, k_hi);
  }
  za.sync();
  for (int64_t k = k_hi; k >= k_lo; --k) {
    if (P.Nf > 0) {
      face_phase<BS>(P, nullptr, JuncSource{Ca.u, nullptr, false, 0.0}, za, wa, k);
      if (two) face_phase<BS>(P, nullptr, JuncSource{Cb.u, nullptr, false, 0.0}, zb, wb, k);
      za.barrier();
      if (two)
        solve_pair(P, za, zb);
      else
        solve(P, za);
    }
    for (int32_t p = za.vt; p < P.Nf; p += za.vbs) gfa[p] = gfa[p] - kTwoPi * za.rd(p);
    if (two)
      for (int32_t p = zb.vt; p < P.Nf; p += zb.vbs) gfb[p] = gfb[p] - kTwoPi * zb.rd(p);
    adjoint_junctions(P, A, Ca, za, k, wa);
    if (two) adjoint_junctions(P, A, Cb, zb, k, wb);
    za.sync();
  }
}

}  // namespace

#endif  // JJA_DEVICE_H
