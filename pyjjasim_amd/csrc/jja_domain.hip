// Step kernels of split columns of any circuit as subdomains, one workgroup each.
//
// The staged factor of a split column streams all its entries through every column
// and meets at a column barrier per stage: 535 us a step for 25,000 faces in one
// workgroup, 210 in eight, more beyond. Subdomains (domain_plan.py) meet once: each
// part eliminates its interior faces onto the separator faces it borders (two
// phases of dense rows), publishes those contributions, sums everybody's for each
// separator face, and computes the separator rows it borders and its interior
// (three phases). The operators of a part are a few hundred kilobytes to two
// megabytes streamed from the L2 every step, which bounds large parts; small ones
// are bound by the phases' latency and the meeting.
//
// Measured, us a step in one workgroup before (with the state in memory) and now: honeycomb
// 30x30, 64 columns 41, 18.4 in 4 parts; triangular 80x80, 4 columns 535, 42 in 32;
// triangular 20x20, 8 columns 35, 11.4 in 8.
//
// The meeting is that of the row slabs (jja_slab.hip): published values and the
// waves' flags are device-scope accesses, buffered by the step's parity.
#include "jja_domain.h"

#include "jja_part_kernels.h"

namespace {

constexpr int kPartWaves = kPartBlock / kWave;

// A record program as solve() walks it; rows and indices are LDS addresses.
struct Program {
  static constexpr int32_t Nf = 0;  // an off-block record's row is updated in place
  int32_t val_bytes;
  const jja_slice* solve_slices;
  const int32_t* slice_rows;
  const double* ent_val;
  const void* ent_off;
  const int32_t* wave_ptr;
};

struct DomainSolver {
  using Dev = DomainDev;
  static constexpr int kFaceWords = 4;
  LAS double *in, *out, *gamma, *u;
  int32_t part;
  uint32_t need;                  // flags lane + 64 i this wave waits for
  GAS double* pub;                // this column's [2][n_published]
  uint32_t* flags;                // this column's [parts][waves]
  uint32_t wait_limit;
  int32_t* err;
  volatile LAS int32_t* stopped;

  __device__ __forceinline__ DomainSolver(const DevProblem&, const DomainDev& S, int64_t column, int32_t part_, double* lds,
                                          int32_t* err_, uint32_t wait_limit_, int32_t tid, int32_t nt)
      : part(part_), need(0), wait_limit(wait_limit_), err(err_) {
    in = (LAS double*)lds;
    out = in + S.faces;
    gamma = out + S.faces;
    u = gamma + S.n_gamma;
    stopped = (volatile LAS int32_t*)(u + 2 * S.pairs);
    pub = gblw(S.pub) + column * 2 * S.n_published;
    flags = S.flags + column * (S.parts * kPartWaves);
    for (int32_t i = tid; i < 2 * S.faces + S.n_gamma + 2 * S.pairs; i += nt) in[i] = 0.0;
    // flag f is wave f % waves of part f / waves; waves past a part's published
    // values have none
    const int32_t lane = tid & (kWave - 1);
    for (int32_t i = 0; i * kWave < S.parts * kPartWaves; ++i) {
      const int32_t f = lane + kWave * i, p = f / kPartWaves, wv = f % kPartWaves;
      if (p < S.parts && wv * kWave < gbl(S.pub_ptr)[p + 1] - gbl(S.pub_ptr)[p]) need |= 1u << i;
    }
    if (tid == 0) *stopped = 0;
    __syncthreads();
  }

  using Head = SolveHead<false>;
  __device__ __forceinline__ Program program(const DomainDev& S, int32_t which) const {
    return Program{S.val_bytes, S.solve_slices, S.slice_rows, S.ent_val, S.ent_off,
                   S.wave_ptr + (2 * part + which) * (kPartWaves + 1)};
  }
  __device__ __forceinline__ void head(const DomainDev& S, int32_t tid, Head& h) const {
    solve_head(program(S, 0), tid, h);
  }

  // K^-1 of the column's face sums: at the faces' addresses in `in` on entry (a
  // separator face's sum is spread over the parts that hold its junctions), the
  // solution in `out` on exit.
  __device__ __forceinline__ void solve(const DevProblem&, const DomainDev& S, uint32_t seq, int32_t tid, int32_t nt,
                                        Head& h) const {
    FaceStore<false> zs;
    zs.p = (double*)in;
    zs.vt = tid;
    zs.vbs = nt;
    solve_tail(program(S, 0), zs, h);
    const int32_t wave = __builtin_amdgcn_readfirstlane(tid / kWave), lane = tid & (kWave - 1);
    const int32_t p0 = gbl(S.pub_ptr)[part], n = gbl(S.pub_ptr)[part + 1] - p0;
    GAS double* const buf = pub + ((seq & 1u) ? S.n_published : 0);
    for (int32_t i = tid; i < n; i += nt)
      __hip_atomic_store(reinterpret_cast<unsigned long long*>((double*)(buf + p0 + i)),
                         __builtin_bit_cast(unsigned long long, in[gbl(S.pub_at)[p0 + i]]), __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    __builtin_amdgcn_s_waitcnt(kWaitVmem);
    __atomic_signal_fence(__ATOMIC_SEQ_CST);
    if (lane == 0)
      __hip_atomic_store(flags + part * kPartWaves + wave, seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // the second program's first records arrive during the wait
    solve_head(program(S, 1), tid, h);
    // one wave watches the flags (eight would contend for them)
    if (wave == 0 && !*stopped) {
      uint32_t spins = 0;
      while (true) {
        bool ready = true;
        for (int32_t i = 0; i * kWave < S.parts * kPartWaves; ++i)
          if (need >> i & 1u) {
            const uint32_t v = __hip_atomic_load(flags + lane + kWave * i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ready = ready && static_cast<int32_t>(v - seq) >= 0;
          }
        if (__all(ready)) break;
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
    lds_barrier();
    // every separator face's right-hand side, its parts' contributions in order
    for (int32_t g = tid; g < S.n_gamma; g += nt) {
      double acc = 0.0;
      for (int32_t i = 0; i < S.sources; ++i) {
        const int32_t src = gbl(S.source)[g * S.sources + i];
        if (src >= 0)
          acc = acc + __builtin_bit_cast(
                          double, __hip_atomic_load(reinterpret_cast<unsigned long long*>((double*)(buf + src)),
                                                    __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
      }
      gamma[g] = acc;
    }
    lds_barrier();
    solve_tail(program(S, 1), zs, h);
  }
};

}  // namespace

const void* domain_evolve_kernel(int pairs) {
  if (pairs <= 1) return reinterpret_cast<const void*>(evolve_parts_kernel<DomainSolver, 1>);
  if (pairs <= 2) return reinterpret_cast<const void*>(evolve_parts_kernel<DomainSolver, 2>);
  return pairs <= kDomainPairs ? reinterpret_cast<const void*>(evolve_parts_kernel<DomainSolver, kDomainPairs>) : nullptr;
}

const void* domain_adjoint_kernel(int pairs) {
  if (pairs <= 1) return reinterpret_cast<const void*>(adjoint_parts_kernel<DomainSolver, 1>);
  if (pairs <= 2) return reinterpret_cast<const void*>(adjoint_parts_kernel<DomainSolver, 2>);
  return pairs <= kDomainPairs ? reinterpret_cast<const void*>(adjoint_parts_kernel<DomainSolver, kDomainPairs>) : nullptr;
}
