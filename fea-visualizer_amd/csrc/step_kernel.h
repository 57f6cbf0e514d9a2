// step_kernel.h -- persistent, cooperative time-stepping kernel (included by
// two translation units per exchange mode, without and with rows in LDS:
// step_plain.hip, step_coherent.hip, step_fenced.hip and step_plain_rows.hip,
// step_coherent_rows.hip, step_fenced_rows.hip).
//
// One launch advances every instance of a batch by `nsteps` implicit time
// steps.  The grid is split into teams (contiguous workgroup ranges); a team
// owns a list of instances and walks them one after the other.  Inside a team
// each workgroup owns a contiguous block of CSR rows, and the team meets at a
// barrier between phases.
//
// Memory model.  On gfx950 a device-scope fence is a whole-L2 write-back plus
// invalidate (buffer_wbl2 sc1 / buffer_inv sc1) that the L2 serialises across
// workgroups, so a fenced barrier costs ~35 ns per participating workgroup.
// Two exchange modes serve teams of more than one workgroup:
//  - coherent (no fences): every value that one workgroup writes during the
//    launch and another reads later (state, solution, residual, Krylov
//    vectors, partial sums) is stored and loaded device-coherently (agent-
//    scope atomic accesses: global_load/store sc1).  A barrier is then: every
//    wave waits for its stores to complete (s_waitcnt 0 -- the release the
//    memory model would emit for such data, without the cache-wide
//    write-back), s_barrier, and the workgroup stores its partial dot
//    products coherently into its own record.  Best when a workgroup's rows fit
//    its LDS row cache and the phases are latency-bound;
//  - fenced: ordinary cached accesses for all data; one wave writes the L2
//    back before the workgroup's arrival and invalidates once the barrier has
//    completed.  Best when phases stream megabytes between barriers.
// In both, each 64-bit partial carries the barrier's epoch tag in its lowest
// mantissa bit, so the partials are also the arrival signal: readers poll the
// values themselves, and arrivals never contend on one address.  Read-only
// data (pattern, matrices, preconditioner) uses ordinary cached loads.  A
// one-workgroup team needs none of this and runs the plain variant.
//
// Rows in LDS.  While a workgroup's rows fit two per lane, its Krylov sweeps
// keep their vectors in registers and LDS, and its neighbours' products come
// in words that carry their own epoch (exchange words), polled together with
// the iteration's sums: between two barriers nothing else is loaded
// (krylov_pcg_rows, krylov_bicgstab_rows).
//
// Reductions: partials are four-way buffered by epoch in the records and
// always summed in a fixed order, so results are deterministic and every
// workgroup takes the same decisions.  One wave of a workgroup, the control
// wave, publishes, polls and advances the scalars while the others take the
// exchange words.
//
// Per step and instance (the reference's CPUSolver::advance_time,
// src/FEM/CPUSolver.cpp:64-147, re-expressed as fused phases):
//   R    right-hand side (FP64) incl. the Gray-Scott reaction, the initial
//        residual r = b - S x0 (FP64), r -> inner precision
//   I    CG start: w = S D^-1 r, <r, D^-1 r>, <D^-1 r, w>
//   C    one Chronopoulos-Gear PCG iteration per barrier: p, s = S p, xi, r
//        updated for own rows; w = S D^-1 r_new with the neighbours' r_new
//        recomputed from the double-buffered r, w, s of the previous
//        iteration; <r,u>, <u,w>, <r,r>
//        (classic two-phase CG and BiCGSTAB are also available)
//   Res  FP64 refinement residual r = b - S64 (x + xi), next sweep while
//        |r| >= tol |b|
//   U    state update (heat: u = x; wave: v = x, u += dt v; Gray-Scott: u,v;
//        Newmark: u, v, a) and the instability rule (CPUSolver.cpp:41-48)
// Vectors are [rows][k] with the right-hand side fastest, so the k lanes of a
// row gather one contiguous span per neighbour.
#pragma once

#include "femhip_internal.h"
#include "femhip_step.h"

#include <cfloat>

#ifndef FEMHIP_TEAM_BLOCK
#define FEMHIP_TEAM_BLOCK 256  // kBlock: one-workgroup teams, and the streaming engine's phases
#endif

namespace femhip {

namespace {

// Phases and drivers are inlined: called, they take the instance, the team and
// the row pool by pointers into LDS and scratch, and an iteration spends most
// of its time on those.
#define FEM_INLINE __device__ __attribute__((always_inline)) inline

// Threads per workgroup of this translation unit's stepping kernel (team_block).
constexpr int kTB = FEMHIP_TEAM_BLOCK;

// Every barrier wait is bounded by the team's wait_ticks (wall_clock64 ticks
// at 100 MHz; 4 s unless the caller set another limit): a longer wait aborts
// the launch.  It cannot happen in a correct run.

struct Shared {
  double wred[kTB / kWave][kMaxRed];
  double red[kMaxRed];     // reduced values of the last barrier
  double gamma[kMaxK];     // CG: <r,z>;  BiCGSTAB: rho
  double alpha[kMaxK];
  double beta[kMaxK];
  double omega[kMaxK];
  double thr[kMaxK];       // tol^2 |b|^2
  double ithr[kMaxK];      // inner stopping threshold of the sweep
  double bb[kMaxK];
  int active[kMaxK];
  int uni;                 // uniform control value broadcast
  int redo;                // refinement: repeat the residual pass
  int bkd;                 // BiCGSTAB: a scalar of this iteration broke down
  int reset[kMaxK];        // refinement: drop the correction xi of column j
};

// Shared of a stepping workgroup: also what its team barriers need.
struct TeamShared : Shared {
  double ig[kMaxK], ia[kMaxK];  // CG: 1 / gamma and 1 / alpha
  int tmo;                      // a wait of this workgroup ended without its value (never reset)
};

// Lane of the control wave (negative elsewhere): the last wave, which adds up
// the workgroup's sums, publishes them, polls the other ranks' and advances
// the scalars.  Rows fill a workgroup from its first wave, so in all but full
// workgroups the control wave has none of its own.
FEM_INLINE int ctl() { return (int)threadIdx.x - (kTB - kWave); }

// Pointers loaded from the instance table are generic; casting them to the
// global address space lets the compiler emit global_load/store instead of
// flat accesses.
#define GA __attribute__((address_space(1)))
template <typename T>
FEM_INLINE T GA* gp(T* p) { return (T GA*)p; }
template <typename T>
FEM_INLINE const T GA* gp(const T* p) { return (const T GA*)p; }

// Exchange modes of a launch (template parameter C):
//   kPlain     every team is one workgroup: nothing is shared across CUs;
//   kCoherent  data exchanged between the workgroups of a team is stored and
//              loaded device-coherently (below), barriers need no fence;
//   kFenced    data uses ordinary cached accesses; a barrier arrival first
//              writes the L2 back (release) and the workgroup invalidates its
//              caches once the barrier completes (acquire).  Costlier per
//              barrier, but every vector access stays cached: the mode for
//              teams whose phases stream megabytes between barriers.
constexpr int kPlain = 0, kCoherent = 1, kFenced = 2;

// Device-coherent (C == kCoherent) or plain access to data exchanged between
// the workgroups of a team.
template <int C, typename T>
FEM_INLINE T ld(const T* p) {
  if constexpr (C == kCoherent) return __hip_atomic_load(gp(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else return *gp(p);
}
template <int C, typename T>
FEM_INLINE void st(T* p, T v) {
  if constexpr (C == kCoherent) __hip_atomic_store(gp(p), v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *gp(p) = v;
}


// Rank of this workgroup inside its team, ordered so that ranks on the same
// XCD (workgroups are dealt round-robin over the 8 XCDs) own adjacent row
// blocks and share halo rows in their XCD's L2.
FEM_INLINE int xcd_rank(int l, int g) {
  int x = l & 7, base = 0;
  for (int y = 0; y < x; y++) base += (g - y + 7) >> 3;
  return base + (l >> 3);
}

// Tag a partial sum for barrier epoch e: its lowest mantissa bit becomes
// (e >> 2) & 1.  The change is at most one unit in the last place and is the
// same on every workgroup, so reductions stay deterministic and every
// workgroup takes the same decisions.
FEM_INLINE double tag_value(double v, unsigned e) {
  const unsigned long long b = (unsigned long long)__double_as_longlong(v);
  return __longlong_as_double((long long)((b & ~1ull) | (unsigned long long)((e >> 2) & 1u)));
}
FEM_INLINE bool has_tag(double v, unsigned e) {
  return ((unsigned long long)__double_as_longlong(v) & 1ull) == (unsigned long long)((e >> 2) & 1u);
}

// Values every barrier of a K-column instance writes per buffer.  A barrier
// reducing fewer values pads with tagged zeros: otherwise entries last
// written eight epochs earlier (same buffer, same tag) would look current.
template <int K>
constexpr int kPadVals = 4 * K;

// A double of another lane: rotated by N within its row of 16 lanes (DPP), or
// both halves of the lane pairs 16 or 32 apart added up (permlane swaps).
template <int N>
FEM_INLINE double row_rotated(double v) {
  int lo = __double2loint(v), hi = __double2hiint(v);
  lo = __builtin_amdgcn_update_dpp(lo, lo, 0x120 | N, 0xf, 0xf, false);
  hi = __builtin_amdgcn_update_dpp(hi, hi, 0x120 | N, 0xf, 0xf, false);
  return __hiloint2double(hi, lo);
}
template <int N>
FEM_INLINE double pair_sum(double v) {
  const unsigned lo = (unsigned)__double2loint(v), hi = (unsigned)__double2hiint(v);
  if constexpr (N == 16) {
    const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
  } else {
    const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    return __hiloint2double((int)b[0], (int)a[0]) + __hiloint2double((int)b[1], (int)a[1]);
  }
}

// Sum over the lanes of a wave with equal lane % G (G a power of two), in
// every lane, in a fixed order.  Register moves only: the same sums by
// __shfl_xor are LDS permutes, 12 dependent ones per value at G = 1, which
// cost a barrier of six values 1.0 us of 2.8 (two workgroups, no other work).
template <int G>
FEM_INLINE double wave_sum(double v) {
  if constexpr (G <= 8) v += row_rotated<8>(v);
  if constexpr (G <= 4) v += row_rotated<4>(v);
  if constexpr (G <= 2) v += row_rotated<2>(v);
  if constexpr (G <= 1) v += row_rotated<1>(v);
  if constexpr (G <= 16) v = pair_sum<16>(v);
  if constexpr (G <= 32) v = pair_sum<32>(v);
  return v;
}

// Per-lane partial sums -> this workgroup's share at q*K + j, written by the
// control wave.  A one-workgroup team keeps it in LDS (sh.red).  Larger teams first wait
// until every wave's stores of the phase are complete, then store the share
// tagged and coherently into buffer e & 3 of their record: the tagged values
// are the arrival signal.  DRAIN false: no other workgroup reads what the
// phase stored except through words that carry their own tag (exchange
// words), so nothing is waited for or written back first.
template <int K, int NS, int C, bool DRAIN = true>
FEM_INLINE void block_partials(const double (&acc)[NS], Shared& sh, double* dst, unsigned e) {
  static_assert(NS * K <= kPadVals<K> && kPadVals<K> <= kWave, "reduction wider than the record");
  const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x / kWave;
#pragma unroll
  for (int q = 0; q < NS; q++) {
    const double v = wave_sum<K>(acc[q]);
    if (lane < K) sh.wred[wave][q * K + lane] = v;
  }
  if constexpr (C != kPlain && DRAIN) __builtin_amdgcn_s_waitcnt(0);  // the phase's stores have completed
  __syncthreads();
  const int cl = ctl();
  if (cl < 0) return;
  // release: write the phase's data back from this XCD's L2 before arriving
  if constexpr (C == kFenced && DRAIN) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  double s = 0.0;
  if (cl < NS * K) {
    constexpr int W = kTB / kWave;
    double v[W];
#pragma unroll
    for (int w = 0; w < W; w++) v[w] = sh.wred[w][cl];
#pragma unroll
    for (int h = W / 2; h > 0; h >>= 1)
#pragma unroll
      for (int w = 0; w < h; w++) v[w] += v[w + h];
    s = v[0];
  }
  if constexpr (C != kPlain) {
    if (cl < kPadVals<K>) st<kCoherent>(dst + cl, tag_value(s, e));  // the team's record in global memory
  } else if (cl < NS * K) {
    dst[cl] = s;  // sh.red in LDS
  }
}

FEM_INLINE bool aborted(const Team& T) {
  return __hip_atomic_load(T.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
}

FEM_INLINE void raise_abort(const Team& T) {
  if (ctl() == 0) __hip_atomic_fetch_or(T.abort_flag, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Re-load a word until arrived(word).  Sets *to on a timeout or when another
// workgroup aborted.
template <typename W, typename F>
FEM_INLINE W wait_word(const Team& T, const W* p, F arrived, int* to) {
  long long t0 = 0;
  int spins = 0;
  while (true) {
    const W v = ld<kCoherent>(p);
    if (arrived(v)) return v;
    if (T.wait_ticks <= 0) {  // zero limit: no waiting at all
      *to = 1;
      return v;
    }
    __builtin_amdgcn_s_sleep(1);
    if ((++spins & 63) == 0) {  // the clock is read only in long waits
      const long long now = wall_clock64();
      if (spins == 64) t0 = now;
      if (aborted(T) || now - t0 > T.wait_ticks) {
        *to = 1;
        return v;
      }
    }
  }
}
FEM_INLINE double wait_value(const Team& T, const double* p, unsigned e, int* to) {
  return wait_word(T, p, [e](double v) { return has_tag(v, e); }, to);
}

// Exchange words: a value of the inner precision (or an FP64 one) as one 32-bit
// half per 64-bit word, the other half of the word holding the epoch of the
// barrier it is published for.  A reader polls the words themselves, together
// with the sums of that barrier, so the value needs no wait for its store, no
// fence, and no load after the barrier.
typedef unsigned long long xword;
template <typename V>
constexpr int kXW = (int)sizeof(V) / 4;
template <typename V>
FEM_INLINE void put_words(xword* x, size_t o, V v, unsigned tag) {
  const xword hi = (xword)tag << 32;
  if constexpr (sizeof(V) == 4) {
    st<kCoherent>(x + o, hi | (unsigned)__float_as_int(v));
  } else {
    st<kCoherent>(x + 2 * o, hi | (unsigned)__double2loint(v));
    st<kCoherent>(x + 2 * o + 1, hi | (unsigned)__double2hiint(v));
  }
}
template <typename V>
struct XWords {
  xword w[kXW<V>];
};
template <typename V>
FEM_INLINE void load_words(const xword* x, size_t o, XWords<V>& v) {
#pragma unroll
  for (int i = 0; i < kXW<V>; i++) v.w[i] = ld<kCoherent>(x + kXW<V> * o + i);
}
template <typename V>
FEM_INLINE V take_words(const Team& T, const xword* x, size_t o, XWords<V>& v, unsigned tag, int* to) {
#pragma unroll
  for (int i = 0; i < kXW<V>; i++)
    if ((unsigned)(v.w[i] >> 32) != tag)
      v.w[i] = wait_word(T, x + kXW<V> * o + i, [tag](xword w) { return (unsigned)(w >> 32) == tag; }, to);
  if constexpr (sizeof(V) == 4) return __int_as_float((int)(unsigned)v.w[0]);
  else return __hiloint2double((int)(unsigned)v.w[1], (int)(unsigned)v.w[0]);
}

// Rank w's record of barrier buffer buf, and group w's (two-level reductions).
FEM_INLINE double* team_record(const Team& T, int buf, int w) {
  return T.slots + ((size_t)buf * T.buf_records + w) * T.rec_vals;
}
FEM_INLINE double* group_record(const Team& T, int buf, int w) {
  return T.groups + ((size_t)buf * T.buf_records + w) * T.rec_vals;
}

constexpr int pow2_at_least(int n) {
  int p = 1;
  while (p < n) p <<= 1;
  return p;
}

// Control wave: wait for the NV tagged values of `count` adjacent records and
// sum them in a fixed order: lane (q, c) sums records c, c + chunks, ... with
// kR loads in flight, then the lanes that hold the same value q are added up
// (wave_sum), so every lane returns the sum of value lane % VP.  One wave
// polls: the sums meet in registers, with no LDS round or workgroup barrier
// before the scalars.
template <int NV>
FEM_INLINE double sum_records(const Team& T, unsigned e, const double* rec, int count, int* to) {
  constexpr int VP = pow2_at_least(NV);
  constexpr int chunks = kWave / VP;
  const int q = ctl() & (VP - 1), c = ctl() / VP;
  double s = 0.0;
  if (q < NV) {
    constexpr int kR = 8;
    for (int w0 = c; w0 < count && !*to; w0 += kR * chunks) {
      double v[kR];
#pragma unroll
      for (int i = 0; i < kR; i++) {
        const int w = w0 + i * chunks;
        if (i * chunks < count) v[i] = ld<kCoherent>(rec + (size_t)(w < count ? w : w0) * T.rec_vals + q);
      }
#pragma unroll
      for (int i = 0; i < kR; i++) {
        const int w = w0 + i * chunks;
        if (w < count) {
          if (!has_tag(v[i], e)) v[i] = wait_value(T, rec + (size_t)w * T.rec_vals + q, e, to);
          s += v[i];
        }
      }
    }
  }
  return wave_sum<VP>(s);
}

// The control wave's part of a barrier whose partials are published: the sums
// of all ranks into sh.red.  Flat: every workgroup sums all records.  In two
// levels: the first rank of each kGroup ranks sums its group's records and
// publishes the sum as the group's record, and every workgroup sums those.
template <int K, int NV>
FEM_INLINE void collect(const Team& T, int rank, unsigned e, TeamShared& sh) {
  const int cl = ctl(), buf = e & 3;
  int to = 0;
  double s;
  if (T.allpoll) {
    s = sum_records<NV>(T, e, team_record(T, buf, 0), T.size, &to);
  } else {
    const int g = rank / kGroup;
    if (rank == g * kGroup) {
      s = sum_records<NV>(T, e, team_record(T, buf, rank), min(kGroup, T.size - rank), &to);
      if (cl < kPadVals<K>) st<kCoherent>(group_record(T, buf, g) + cl, tag_value(cl < NV ? s : 0.0, e));
    }
    s = sum_records<NV>(T, e, group_record(T, buf, 0), (T.size + kGroup - 1) / kGroup, &to);
  }
  if (cl < NV) sh.red[cl] = s;
  if (to) sh.tmo = 1;
}

// Run scalars() in the control wave on the sums its lanes have stored to
// sh.red.  Lane j reads what other lanes of the wave wrote: the fence keeps
// the compiler from moving those loads before the stores (the wave's LDS
// accesses complete in program order).
template <typename F>
FEM_INLINE void run_scalars(F scalars) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  scalars();
}

// Reduction + barrier: acc -> team sums in sh.red[q*K + j], handed to
// scalars(), which the control wave (whose lanes wrote them) runs; every wave
// returns once all ranks have arrived and the scalars are in LDS.  Returns
// false when the launch must stop.
template <int K, int NS, int C, typename F>
FEM_INLINE bool team_reduce(const double (&acc)[NS], const Team& T, int rank, unsigned& e, TeamShared& sh, F scalars) {
  e++;
  // a one-workgroup team (also inside a multi-workgroup launch) reduces in LDS
  if (C == kPlain || T.size == 1) {
    block_partials<K, NS, kPlain>(acc, sh, sh.red, e);
    if (ctl() >= 0) run_scalars(scalars);
    __syncthreads();
    return true;
  }
  block_partials<K, NS, C>(acc, sh, team_record(T, e & 3, rank), e);
  if (ctl() >= 0) {
    collect<K, NS * K>(T, rank, e, sh);
    // acquire: drop cached copies of data other workgroups wrote this phase
    if constexpr (C == kFenced) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    run_scalars(scalars);
  }
  __syncthreads();
  if (sh.tmo) {
    raise_abort(T);
    return false;
  }
  return true;
}

struct NoHalo {
  FEM_INLINE void take(const Team&, unsigned, int*) {}
};

// team_reduce of a phase that stored nothing but exchange words: meanwhile the
// other waves take the words of this barrier's epoch that the next phase needs.
template <int K, int NS, int C, typename H, typename F>
FEM_INLINE bool rows_reduce(const double (&acc)[NS], const Team& T, int rank, unsigned& e, TeamShared& sh, H&& halo,
                            F scalars) {
  e++;
  if (C == kPlain || T.size == 1) {
    block_partials<K, NS, kPlain>(acc, sh, sh.red, e);
    if (ctl() >= 0) run_scalars(scalars);
    __syncthreads();
    return true;
  }
  block_partials<K, NS, C, false>(acc, sh, team_record(T, e & 3, rank), e);
  if (ctl() >= 0) {
    collect<K, NS * K>(T, rank, e, sh);
    run_scalars(scalars);
  } else {
    int to = 0;
    halo.take(T, e, &to);
    if (to) sh.tmo = 1;
  }
  __syncthreads();
  if (sh.tmo) {
    raise_abort(T);
    return false;
  }
  return true;
}

// Plain barrier: K (ignored) values per workgroup are the arrival signal.
template <int K, int C>
FEM_INLINE bool team_barrier(const Team& T, int rank, unsigned& e, TeamShared& sh) {
  if (C == kPlain || T.size == 1) {
    __syncthreads();
    return true;
  }
  const double acc[1] = {0.0};
  return team_reduce<K, 1, C>(acc, T, rank, e, sh, [] {});
}

template <typename TI>
FEM_INLINE TI to_ti(double v) { return (TI)v; }

// Chronopoulos-Gear update of one entry, shared by the owner and by
// neighbours recomputing it (identical operations, identical rounding).
template <typename TI>
FEM_INLINE TI cg_s(TI w, TI s, TI be, bool first) { return first ? w : (w + be * s); }
template <typename TI>
FEM_INLINE TI cg_r(TI r, TI sv, TI al) { return r - al * sv; }

// ---------------------------------------------------------------------------
// Phases.  Lane layout: column jr = tid % K, rows tid / K + m * (kTB / K).
//
// Row gathers are unrolled by kU with clamped (always in-bounds) indices, so a
// row's loads are all in flight before the first is consumed; the masked
// accumulation keeps the sequential summation order.
// ---------------------------------------------------------------------------

constexpr int kU = 8;

template <typename A>
FEM_INLINE void acc_add(A& acc, const A& t) { acc += t; }

struct D2 {
  double a, b;
  __device__ D2& operator+=(const D2& o) {
    a += o.a;
    b += o.b;
    return *this;
  }
};
struct D3 {
  double a, b, c;
  __device__ D3& operator+=(const D3& o) {
    a += o.a;
    b += o.b;
    c += o.c;
    return *this;
  }
};

// sum over s in [lo, hi) of f(s), in ascending s; U entries in flight
template <int U = kU, typename A, typename F>
FEM_INLINE A row_gather(int lo, int hi, A zero, F f) {
  A acc = zero;
  for (int s0 = lo; s0 < hi; s0 += U) {
    A t[U];
#pragma unroll
    for (int u = 0; u < U; u++) t[u] = f(min(s0 + u, hi - 1));
#pragma unroll
    for (int u = 0; u < U; u++)
      if (s0 + u < hi) acc_add(acc, t[u]);
  }
  return acc;
}

// Entries in flight for gathers that load five or more values per entry.
constexpr int kUWide = 4;

// Hold a loaded value here: what stands before is issued before, and its use
// stands after.
FEM_INLINE void hold(int& v) { asm volatile("" : "+v"(v)); }
FEM_INLINE void hold(float& v) { asm volatile("" : "+v"(v)); }
FEM_INLINE void hold(double& v) { asm volatile("" : "+v"(v)); }

// sum over s in [lo, hi) of use(v), v = the N values that load(s, column, v)
// fetches, in ascending s.  In stages, each with the loads of kU entries in
// flight: the columns, then the values.  Left to the compiler the entries were
// loaded one after the other in the 512-thread variants: at two waves per SIMD
// it takes back any order that lengthens live ranges once the scalar registers
// spill.  ms that way and in stages: BiCGSTAB on 489,000 rows x 16 columns 113
// and 52 (3 steps of 40 iterations), 100 meshes of 1,521 rows x 16 10.9 and 7.4,
// CG on 40,000 rows of a Delaunay mesh 27.3 and 23.9.
template <int N, typename TI, typename L, typename F>
FEM_INLINE TI col_gather(const int GA* ci, int lo, int hi, L load, F use) {
  TI acc = (TI)0;
  for (int s0 = lo; s0 < hi; s0 += kU) {
    int c[kU];
#pragma unroll
    for (int u = 0; u < kU; u++) c[u] = ci[min(s0 + u, hi - 1)];
#pragma unroll
    for (int u = 0; u < kU; u++) hold(c[u]);
    TI v[kU][N];
#pragma unroll
    for (int u = 0; u < kU; u++) load(min(s0 + u, hi - 1), c[u], v[u]);
#pragma unroll
    for (int u = 0; u < kU; u++)
#pragma unroll
      for (int i = 0; i < N; i++) hold(v[u][i]);
#pragma unroll
    for (int u = 0; u < kU; u++) {
      const TI t = use(v[u]);
      if (s0 + u < hi) acc += t;
    }
  }
  return acc;
}

template <int K, typename TI, int C, int NA>
FEM_INLINE void phase_rhs(const Inst& I, int row_lo, int row_hi, TI* r, int step, double (&acc)[NA]) {
  static_assert(NA >= 3, "phase_rhs sums three values");
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI* xi = (TI*)I.xi;
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const double inv_dt = 1.0 / I.dt;
  const bool warm = I.warm != 0;
  // predictor order this step: 2 x_n - x_{n-1} once the previous solution is
  // known, 3 x_n - 3 x_{n-1} + x_{n-2} once two are, 4 x_n - 6 x_{n-1} +
  // 4 x_{n-2} - x_{n-3} once three are
  // (the guess gathered from the history levels here: quartic at most)
  const int lv = warm ? min(min(I.extrap, kPersistentExtrap), I.hist + step) : 0;
  const bool ex = lv > 0;
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  const double GA* M64 = gp(I.M64);
  const double GA* K64 = gp(I.K64);
  const double GA* S64 = gp(I.S64);
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const int lo = rp[row], hi = rp[row + 1];
    const size_t o = (size_t)row * K + jr;
    double b = 0.0, sx = 0.0, x0 = 0.0;
    switch (I.eq) {
      case EQ_HEAT:
      case EQ_ADVDIFF:
      case EQ_GS: {  // b = (M/dt) u                                  CPUSolver.cpp:78,96
        // Gray-Scott: b_u = (M/dt)u - uvv + F(1-u); b_v = (M/dt)v + uvv - (F+k)v   CPUSolver.cpp:134,137
        const D2 g = row_gather(lo, hi, D2{0.0, 0.0}, [&](int s) {
          const size_t oc = (size_t)ci[s] * K + jr;
          const double uc = ld<C>(I.u + oc);
          const double xc = lv == 4   ? 5.0 * (uc - ld<C>(I.h3 + oc)) + 10.0 * (ld<C>(I.v + oc) - ld<C>(I.a + oc)) +
                                            ld<C>(I.h4 + oc)
                            : lv == 3 ? 4.0 * (uc + ld<C>(I.v + oc)) - 6.0 * ld<C>(I.a + oc) - ld<C>(I.h3 + oc)
                            : lv == 2 ? 3.0 * (uc - ld<C>(I.a + oc)) + ld<C>(I.v + oc)
                            : ex      ? 2.0 * uc - ld<C>(I.a + oc)
                                      : uc;
          return D2{M64[s] * uc, warm ? S64[(size_t)s * kv + vj] * xc : 0.0};
        });
        b = g.a * inv_dt;
        if (I.eq == EQ_GS) {
          const double uu = ld<C>(I.u + (size_t)row * K), vv = ld<C>(I.u + (size_t)row * K + 1);
          const double uvv = uu * (vv * vv);
          const double f = (jr == 0) ? (-uvv + I.p3 * (1.0 - uu)) : (uvv - (I.p3 + I.p4) * vv);
          const double w = I.weighting ? gp(I.lumped)[row] : 1.0;
          b += w * f;
        }
        sx = g.b;
        const double uo = ld<C>(I.u + o);
        x0 = !warm     ? 0.0
             : lv == 4 ? 5.0 * (uo - ld<C>(I.h3 + o)) + 10.0 * (ld<C>(I.v + o) - ld<C>(I.a + o)) + ld<C>(I.h4 + o)
             : lv == 3 ? 4.0 * (uo + ld<C>(I.v + o)) - 6.0 * ld<C>(I.a + o) - ld<C>(I.h3 + o)
             : lv == 2 ? 3.0 * (uo - ld<C>(I.a + o)) + ld<C>(I.v + o)
             : ex      ? 2.0 * uo - ld<C>(I.a + o)
                       : uo;
      } break;
      case EQ_WAVE: {  // b = (M/dt) v - c^2 K u                    CPUSolver.cpp:114
        const D3 g = row_gather(lo, hi, D3{0.0, 0.0, 0.0}, [&](int s) {
          const size_t oc = (size_t)ci[s] * K + jr;
          const double vc = ld<C>(I.v + oc);
          const double xc = ex ? 2.0 * vc - ld<C>(I.a + oc) : vc;
          return D3{M64[s] * vc, K64[s] * ld<C>(I.u + oc), warm ? S64[(size_t)s * kv + vj] * xc : 0.0};
        });
        b = g.a * inv_dt - I.p1 * I.p1 * g.b;
        sx = g.c;
        const double vo = ld<C>(I.v + o);
        x0 = warm ? (ex ? 2.0 * vo - ld<C>(I.a + o) : vo) : 0.0;
      } break;
      case EQ_NEWMARK: {  // b = -c^2 K (u + dt v + (1/2 - beta) dt^2 a)
        // guess: the acceleration extrapolated (a_{n-1} in h3, a_{n-2} in h4)
        const double h = (0.5 - I.p2) * I.dt * I.dt;
        const D2 g = row_gather(lo, hi, D2{0.0, 0.0}, [&](int s) {
          const size_t oc = (size_t)ci[s] * K + jr;
          const double ac = ld<C>(I.a + oc);
          const double xc = lv == 2 ? 3.0 * (ac - ld<C>(I.h3 + oc)) + ld<C>(I.h4 + oc)
                            : ex    ? 2.0 * ac - ld<C>(I.h3 + oc)
                                    : ac;
          return D2{K64[s] * (ld<C>(I.u + oc) + I.dt * ld<C>(I.v + oc) + h * ac),
                    warm ? S64[(size_t)s * kv + vj] * xc : 0.0};
        });
        b = -I.p1 * I.p1 * g.a;
        sx = g.b;
        const double ao = ld<C>(I.a + o);
        x0 = !warm     ? 0.0
             : lv == 2 ? 3.0 * (ao - ld<C>(I.h3 + o)) + ld<C>(I.h4 + o)
             : ex      ? 2.0 * ao - ld<C>(I.h3 + o)
                       : ao;
      } break;
      default: {  // EQ_SOLVE: b supplied, x holds the guess
        b = gp(I.b)[o];
        if (warm)
          sx = row_gather(lo, hi, 0.0, [&](int s) {
            return S64[(size_t)s * kv + vj] * ld<C>(I.x + (size_t)ci[s] * K + jr);
          });
        x0 = warm ? ld<C>(I.x + o) : 0.0;
      } break;
    }
    const double r64 = b - sx;
    gp(I.b)[o] = b;
    st<C>(I.x + o, x0);
    const TI rr = to_ti<TI>(r64);
    st<C>(r + o, rr);
    st<C>(xi + o, (TI)0);
    acc[0] += b * b;
    acc[1] += r64 * r64;
    // BiCGSTAB starts from rho = <r, r>; CG from <r, D^-1 r>
    acc[2] += (I.krylov == 1) ? (double)rr * (double)rr : (double)rr * (double)(dinv[(size_t)row * kv + vj] * rr);
  }
}

// Predictor weights on (x_n, x_{n-1}, ..., x_{n-4}) for order lv: the
// alternating binomial coefficients of row lv + 1, 0 (1), 1 (2, -1),
// 2 (3, -3, 1), 3 (4, -6, 4, -1), 4 (5, -10, 10, -5, 1).
FEM_INLINE void pred_weights(int lv, double& w0, double& w1, double& w2, double& w3, double& w4) {
  w0 = lv + 1.0;
  w1 = lv == 4 ? -10.0 : lv == 3 ? -6.0 : lv == 2 ? -3.0 : lv == 1 ? -1.0 : 0.0;
  w2 = lv == 4 ? 10.0 : lv == 3 ? 4.0 : lv == 2 ? 1.0 : 0.0;
  w3 = lv == 4 ? -5.0 : lv == 3 ? -1.0 : 0.0;
  w4 = lv == 4 ? 1.0 : 0.0;
}

// The same weights for any order up to kMaxExtrap: w[j] = (-1)^j C(lv + 1, j + 1)
// on x_{n-j} (lv = 0: x_n), zero beyond the order.
FEM_INLINE void pred_weights_n(int lv, double (&w)[kMaxExtrap + 1]) {
  double c = 1.0;
  for (int j = 0; j <= kMaxExtrap; j++) {
    if (j <= lv) {
      c = c * (double)(lv + 1 - j) / (double)(j + 1);
      w[j] = (j & 1) ? -c : c;
    } else {
      w[j] = 0.0;
    }
  }
}

// Row cache: a workgroup's entries as (column, S_ij D^-1_jj) pairs, for teams
// whose rows fit kCacheP per lane and kCacheE entries but whose halo does not
// fit beside them (Rows below): rows of scattered numbering.  The gathers go
// to memory with the columns known.
template <typename TI>
struct RowCache {
  int col[kCacheP][kCacheE][kTB];
  TI val[kCacheP][kCacheE][kTB];
};

// A workgroup's rows while they fit kCacheP per lane and kCacheE entries each
// (fill_rows): per lane the entries' places and weights S_ij D^-1_jj, and a
// staging area for the vector its phases gather: its own rows' values, written
// from registers, and those of the rows of other workgroups that its rows read
// (the halo, listed by k_halo when the plan is built).  The gathers read LDS.
// Gathered from memory, each of a row's ~7 neighbours costs three coherent
// loads per iteration, which bypass the CU's own cache.  The halo's Krylov
// vectors are kept beside the staging area and advanced by their owner's
// operations, so that only the product of an iteration is exchanged.  All of
// it lives in one LDS pool; the parts are sized by the rows the team deals
// its workgroups.
#define LA __attribute__((address_space(3)))
template <typename TI>
struct Rows {
  unsigned short LA* col;  // [passes][kCacheE][kTB]: place of the entry's value in the staging area
  TI LA* val;              // [passes][kCacheE][kTB]
  unsigned char LA* hv;    // staging area: own values, then the halo's
  const int LA* list;      // [nhalo] halo rows, ascending
  int nhalo;
  int own;                 // values of the own rows: rows x columns
  int nx;                  // halo values: nhalo x columns
  int nvals;               // own + nx
  int res;                 // FP64 vectors the residual pass can stage: the candidate, and the history part
};

template <int C, typename TI>
constexpr int rows_pool() {
  return C == kPlain ? rows_pool_bytes(kTB, (int)sizeof(TI)) : kTeamPool;
}

// The halo's values are handled by the waves before the control wave, from the
// last lane down (the row lanes come first): a lane takes values halo_lane,
// halo_lane + kHaloLanes, ... , all of its own column.
constexpr int kHaloLanes = kTB - kWave;
template <int K>
FEM_INLINE int halo_lane() {
  const int t = (int)threadIdx.x;
  return t < kHaloLanes ? (kHaloLanes - 1 - t) / K * K + t % K : INT32_MAX;
}

// Stage f(offset) of the halo's values into hv + own, kS of a lane's values in
// flight at a time (indices clamped, not guarded: a branch around a value's
// loads would wait for them).
template <int K, typename V, typename TI, typename F>
FEM_INLINE void stage_halo(const Rows<TI>& R, V LA* hv, F f) {
  constexpr int kS = 4;
  for (int t0 = halo_lane<K>(); t0 < R.nx; t0 += kS * kHaloLanes) {
    size_t o[kS];
    V v[kS];
#pragma unroll
    for (int u = 0; u < kS; u++) {
      const int t = t0 + u * kHaloLanes < R.nx ? t0 + u * kHaloLanes : t0;
      o[u] = (size_t)R.list[t / K] * K + t % K;
    }
#pragma unroll
    for (int u = 0; u < kS; u++) v[u] = f(o[u]);
#pragma unroll
    for (int u = 0; u < kS; u++)
      if (t0 + u * kHaloLanes < R.nx) hv[R.own + t0 + u * kHaloLanes] = v[u];
  }
}

// Take the exchange words of all halo values tagged `tag` into dst.
template <int K, typename V, typename TI>
FEM_INLINE void take_halo(const Team& T, const Rows<TI>& R, const xword* x, V LA* dst, unsigned tag, int* to) {
  constexpr int kS = 4;
  for (int t0 = halo_lane<K>(); t0 < R.nx && !*to; t0 += kS * kHaloLanes) {
    int o[kS];
    XWords<V> v[kS];
#pragma unroll
    for (int u = 0; u < kS; u++) {
      const int t = t0 + u * kHaloLanes < R.nx ? t0 + u * kHaloLanes : t0;
      o[u] = R.list[t / K] * K + t % K;
    }
#pragma unroll
    for (int u = 0; u < kS; u++) load_words<V>(x, o[u], v[u]);
#pragma unroll
    for (int u = 0; u < kS; u++)
      if (t0 + u * kHaloLanes < R.nx) dst[t0 + u * kHaloLanes] = take_words<V>(T, x, o[u], v[u], tag, to);
  }
}
template <int K, typename TI>
struct TakeHalo {
  const Rows<TI>& R;
  const xword* x;
  TI LA* dst;
  FEM_INLINE void take(const Team& T, unsigned tag, int* to) { take_halo<K, TI>(T, R, x, dst, tag, to); }
};

// A lane's entries of its rows, in registers for a sweep: read from the pool
// each iteration they were two of the three LDS reads per entry.
template <typename TI>
struct RowCells {
  unsigned short col[kCacheP][kCacheE];
  TI val[kCacheP][kCacheE];
};
template <int K, typename TI>
FEM_INLINE void load_cells(const Rows<TI>& R, int row0, int row_hi, RowCells<TI>& c) {
#pragma unroll
  for (int q = 0; q < kCacheP; q++)
#pragma unroll
    for (int e = 0; e < kCacheE; e++) {
      c.col[q][e] = 0;
      c.val[q][e] = (TI)0;
      if (row0 + q * (kTB / K) >= row_hi) continue;
      const int at = (q * kCacheE + e) * kTB + (int)threadIdx.x;
      c.col[q][e] = R.col[at];
      c.val[q][e] = R.val[at];
    }
}
// sum over the entries of this lane's row of pass q of weight x staged value
template <typename TI>
FEM_INLINE TI cells_gather(const RowCells<TI>& c, const TI LA* hv, int q) {
  TI g[kCacheE], acc = (TI)0;
#pragma unroll
  for (int e = 0; e < kCacheE; e++) g[e] = hv[c.col[q][e]];
#pragma unroll
  for (int e = 0; e < kCacheE; e++) acc += c.val[q][e] * g[e];
  return acc;
}
template <typename TI>
FEM_INLINE TI rows_gather(const Rows<TI>& R, const TI LA* hv, int q) {
  const int at = q * kCacheE * kTB + (int)threadIdx.x;
  TI g[kCacheE], acc = (TI)0;
#pragma unroll
  for (int e = 0; e < kCacheE; e++) g[e] = hv[R.col[at + e * kTB]];
#pragma unroll
  for (int e = 0; e < kCacheE; e++) acc += R.val[at + e * kTB] * g[e];
  return acc;
}

// One row of the FP64 residual pass of a fused step: S c, M c and S h, with
// c = x + xi the candidate solution (xi dropped for a column restarted from x)
// and h the next initial guess's history part.  HM: 0 no history part,
// 1 h gathered from hvec, 2 h formed from the history levels u, a, v, h3.
template <int HM, int K, typename TI, int C>
FEM_INLINE D3 res_gather_fused(const Inst& I, int lo, int hi, int jr, int vj,
                                                                     bool drop, int lvn, double w1, double w2,
                                                                     double w3, double w4) {
  const int kv = I.kv;
  const TI* xi = (const TI*)I.xi;
  const int GA* __restrict__ ci = gp(I.ci);
  const double GA* S64 = gp(I.S64);
  const double GA* M64 = gp(I.M64);
  return row_gather<kUWide>(lo, hi, D3{0.0, 0.0, 0.0}, [&](int s) {
    const size_t oc = (size_t)ci[s] * K + jr;
    const double sv = S64[(size_t)s * kv + vj];
    const double xc = ld<C>(I.x + oc) + (drop ? 0.0 : (double)ld<C>(xi + oc));
    double hv = 0.0;
    if constexpr (HM == 1) hv = ld<C>(I.hvec + oc);
    if constexpr (HM == 2)
      hv = w1 * ld<C>(I.u + oc) + (lvn >= 2 ? w2 * ld<C>(I.a + oc) : 0.0) +
           (lvn >= 3 ? w3 * ld<C>(I.v + oc) : 0.0) + (lvn >= 4 ? w4 * ld<C>(I.h3 + oc) : 0.0);
    return D3{sv * xc, M64[s] * xc, sv * hv};
  });
}

// FP64 residual of x + xi into r (inner precision); acc: <r, r>, <r, D^-1 r>.
// hpre != nullptr: the next step's update is fused with its right-hand side
// and takes, should this pass turn out to be the last of the step, what it
// needs from here instead of gathering the candidate solution c = x + xi:
// the next right-hand side b = M c / dt (+ the Gray-Scott reaction at c)
// into xnext and the next initial residual b - (w0 S c + S h) into hpre
// (lvn: the next step's predictor order; hready: the update of this step
// formed h in hvec).
template <int K, typename TI, int C>
FEM_INLINE void phase_res(const Inst& I, int row_lo, int row_hi, TI* r,
                                                                const Shared& sh, double (&acc)[2], int lvn = 0,
                                                                double* hpre = nullptr, bool hready = false) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI* xi = (TI*)I.xi;
  // a column whose sweep produced non-finite values restarts from x alone
  const bool drop = sh.reset[jr] != 0;
  // Eigen: rhs == 0 -> x = 0, so the next update sees a zero solution
  const bool zero = sh.bb[jr] == 0.0;
  const bool warm = I.warm != 0;
  const double inv_dt = 1.0 / I.dt;
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  const double GA* S64 = gp(I.S64);
  double w0, w1, w2, w3, w4;
  pred_weights(lvn, w0, w1, w2, w3, w4);
  const bool want_h = hpre && lvn > 0;
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    const double bo = gp(I.b)[o];
    const TI dj = dinv[(size_t)row * kv + vj];  // loaded before the stores below (one completion counter)
    double sx;
    if (hpre) {
      const int lo = rp[row], hi = rp[row + 1];
      const D3 g = !want_h   ? res_gather_fused<0, K, TI, C>(I, lo, hi, jr, vj, drop, lvn, w1, w2, w3, w4)
                   : !hready ? res_gather_fused<2, K, TI, C>(I, lo, hi, jr, vj, drop, lvn, w1, w2, w3, w4)
                             : res_gather_fused<1, K, TI, C>(I, lo, hi, jr, vj, drop, lvn, w1, w2, w3, w4);
      sx = g.a;
      const double su = zero ? 0.0 : g.a;
      double bn = (zero ? 0.0 : g.b) * inv_dt;
      if (I.eq == EQ_GS) {  // CPUSolver.cpp:134,137 at the candidate
        auto cand = [&](int j) -> double {  // species j of this row
          const size_t oj = (size_t)row * K + j;
          return sh.bb[j] == 0.0 ? 0.0 : ld<C>(I.x + oj) + (sh.reset[j] ? 0.0 : (double)ld<C>(xi + oj));
        };
        double uu, vv;
        if constexpr (K == 2) {  // the row's other species is the pair lane
          const double xo = cand(jr);
          const double xp = __shfl_xor(xo, 1, kWave);
          uu = jr == 0 ? xo : xp;
          vv = jr == 0 ? xp : xo;
        } else {
          uu = cand(0);
          vv = cand(1);
        }
        const double uvv = uu * (vv * vv);
        const double fr = (jr == 0) ? (-uvv + I.p3 * (1.0 - uu)) : (uvv - (I.p3 + I.p4) * vv);
        bn += (I.weighting ? gp(I.lumped)[row] : 1.0) * fr;
      }
      gp(I.xnext)[o] = bn;
      st<C>(hpre + o, bn - (warm ? w0 * su + (want_h ? g.c : 0.0) : 0.0));
    } else {
      sx = row_gather(rp[row], rp[row + 1], 0.0, [&](int s) {
        const size_t oc = (size_t)ci[s] * K + jr;
        return S64[(size_t)s * kv + vj] * (ld<C>(I.x + oc) + (drop ? 0.0 : (double)ld<C>(xi + oc)));
      });
    }
    const double r64 = bo - sx;
    const TI rr = to_ti<TI>(r64);
    st<C>(r + o, rr);
    if (drop) st<C>(xi + o, (TI)0);
    acc[0] += r64 * r64;
    acc[1] += (I.krylov == 1) ? (double)rr * (double)rr : (double)rr * (double)(dj * rr);
  }
}

// Pipelined CG start: fold x += xi; w = S D^-1 r; <r, D^-1 r>, <D^-1 r, w>.
template <int K, typename TI, int C>
FEM_INLINE void phase_pcg_init(const Inst& I, int row_lo, int row_hi, const TI* rc, TI* wc, double (&acc)[2]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI* xi = (TI*)I.xi;
  const TI GA* S = gp((const TI*)I.Si);
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    const double xo = ld<C>(I.x + o), xio = (double)ld<C>(xi + o);
    const TI ro = ld<C>(rc + o);
    const TI uo = dinv[(size_t)row * kv + vj] * ro;  // loaded before the stores below
    const TI wa = col_gather<3, TI>(ci, rp[row], rp[row + 1], [&](int s, int c, TI (&v)[3]) {
      v[0] = S[(size_t)s * kv + vj];
      v[1] = dinv[(size_t)c * kv + vj];
      v[2] = ld<C>(rc + (size_t)c * K + jr);
    }, [&](const TI (&v)[3]) { return v[0] * (v[1] * v[2]); });
    st<C>(I.x + o, xo + xio);
    st<C>(xi + o, (TI)0);
    st<C>(wc + o, wa);
    acc[0] += (double)ro * (double)uo;
    acc[1] += (double)uo * (double)wa;
  }
}

// One Chronopoulos-Gear iteration (see file header).
template <int K, typename TI, int C>
FEM_INLINE void phase_pcg_iter(const Inst& I, int row_lo, int row_hi, const TI* rc, const TI* wc, const TI* sc,
                               TI* rn, TI* wn, TI* sn, bool first, const Shared& sh, double (&acc)[3]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI* xi = (TI*)I.xi;
  TI GA* p = gp((TI*)I.p0);  // own rows only
  const TI GA* S = gp((const TI*)I.Si);
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const TI al = to_ti<TI>(sh.alpha[jr]);
  const TI be = first ? (TI)0 : to_ti<TI>(sh.beta[jr]);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  const TI* sg = first ? rc : sc;  // no s yet: any values (cg_s leaves them out)
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    const TI ro = ld<C>(rc + o);
    const TI wo = ld<C>(wc + o);
    const TI so = first ? (TI)0 : ld<C>(sc + o);
    const TI po = first ? (TI)0 : p[o];
    const TI xio = ld<C>(xi + o);
    const TI wa = col_gather<5, TI>(ci, rp[row], rp[row + 1], [&](int s, int c, TI (&v)[5]) {
      const size_t oc = (size_t)c * K + jr;
      v[0] = S[(size_t)s * kv + vj];
      v[1] = dinv[(size_t)c * kv + vj];
      v[2] = ld<C>(wc + oc);
      v[3] = ld<C>(sg + oc);
      v[4] = ld<C>(rc + oc);
    }, [&](const TI (&v)[5]) { return v[0] * (v[1] * cg_r<TI>(v[4], cg_s<TI>(v[2], v[3], be, first), al)); });
    const TI d = dinv[(size_t)row * kv + vj];
    const TI uo = d * ro;
    const TI pn = first ? uo : (uo + be * po);
    const TI sv = cg_s<TI>(wo, so, be, first);
    const TI rr = cg_r<TI>(ro, sv, al);
    p[o] = pn;
    st<C>(xi + o, xio + al * pn);
    st<C>(sn + o, sv);
    st<C>(rn + o, rr);
    st<C>(wn + o, wa);
    const TI un = d * rr;
    acc[0] += (double)rr * (double)un;
    acc[1] += (double)un * (double)wa;
    acc[2] += (double)rr * (double)rr;
  }
}

// Classic CG phase A: p = z + beta p_old (z = D^-1 r), q = S p, <p, q>.
// Neighbour p values are recomputed from r and p_old, so p needs no barrier of
// its own.  On the first iteration of a sweep the pending correction is folded.
template <int K, typename TI, int C>
FEM_INLINE void phase_cg_a(const Inst& I, int row_lo, int row_hi, const TI* r, const TI* pold, TI* pnew,
                           bool first, const Shared& sh, double (&acc)[1]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI GA* q = gp((TI*)I.q);  // own rows only
  TI* xi = (TI*)I.xi;
  const TI GA* S = gp((const TI*)I.Si);
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const TI bj = first ? (TI)0 : to_ti<TI>(sh.beta[jr]);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  const TI* pg = first ? r : pold;  // no p yet: any values, left out below
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    if (first) {
      st<C>(I.x + o, ld<C>(I.x + o) + (double)ld<C>(xi + o));
      st<C>(xi + o, (TI)0);
    }
    const TI qa = col_gather<4, TI>(ci, rp[row], rp[row + 1], [&](int s, int c, TI (&v)[4]) {
      const size_t oc = (size_t)c * K + jr;
      v[0] = S[(size_t)s * kv + vj];
      v[1] = dinv[(size_t)c * kv + vj];
      v[2] = ld<C>(r + oc);
      v[3] = ld<C>(pg + oc);
    }, [&](const TI (&v)[4]) {
      const TI zc = v[1] * v[2];
      return v[0] * (first ? zc : (zc + bj * v[3]));
    });
    const TI zo = dinv[(size_t)row * kv + vj] * ld<C>(r + o);
    const TI pn = first ? zo : (zo + bj * ld<C>(pold + o));
    st<C>(pnew + o, pn);
    q[o] = qa;
    acc[0] += (double)pn * (double)qa;
  }
}

// Classic CG phase B: xi += alpha p, r -= alpha q, <r, D^-1 r>, <r, r>.
template <int K, typename TI, int C>
FEM_INLINE void phase_cg_b(const Inst& I, int row_lo, int row_hi, TI* r, const TI* p, const Shared& sh,
                           double (&acc)[2]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI* xi = (TI*)I.xi;
  const TI GA* q = gp((const TI*)I.q);
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const TI al = to_ti<TI>(sh.alpha[jr]);
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    st<C>(xi + o, ld<C>(xi + o) + al * ld<C>(p + o));
    const TI rr = ld<C>(r + o) - al * q[o];
    st<C>(r + o, rr);
    acc[0] += (double)rr * (double)(dinv[(size_t)row * kv + vj] * rr);
    acc[1] += (double)rr * (double)rr;
  }
}

// BiCGSTAB (right Jacobi preconditioning) phase P:
// p = r + beta (p_old - omega v_old); v = S D^-1 p; <rh, v>.
template <int K, typename TI, int C>
FEM_INLINE void phase_bi_p(const Inst& I, int row_lo, int row_hi, const TI* r, const TI* pold, TI* pnew,
                           const TI* vold, TI* vnew, bool first, const Shared& sh, double (&acc)[1]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI GA* rh = gp((TI*)I.rh);  // own rows only
  TI* xi = (TI*)I.xi;
  const TI GA* S = gp((const TI*)I.Si);
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const TI be = first ? (TI)0 : to_ti<TI>(sh.beta[jr]);
  const TI om = first ? (TI)0 : to_ti<TI>(sh.omega[jr]);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  const TI *pg = first ? r : pold, *vg = first ? r : vold;  // no p, v yet: any values, left out below
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    const TI ro = ld<C>(r + o);
    if (first) {
      st<C>(I.x + o, ld<C>(I.x + o) + (double)ld<C>(xi + o));
      st<C>(xi + o, (TI)0);
      rh[o] = ro;
    }
    const TI va = col_gather<5, TI>(ci, rp[row], rp[row + 1], [&](int s, int c, TI (&v)[5]) {
      const size_t oc = (size_t)c * K + jr;
      v[0] = S[(size_t)s * kv + vj];
      v[1] = dinv[(size_t)c * kv + vj];
      v[2] = ld<C>(r + oc);
      v[3] = ld<C>(pg + oc);
      v[4] = ld<C>(vg + oc);
    }, [&](const TI (&v)[5]) { return v[0] * (v[1] * (first ? v[2] : (v[2] + be * (v[3] - om * v[4])))); });
    const TI pn = first ? ro : (ro + be * (ld<C>(pold + o) - om * ld<C>(vold + o)));
    st<C>(pnew + o, pn);
    st<C>(vnew + o, va);
    acc[0] += (double)(first ? ro : rh[o]) * (double)va;
  }
}

// BiCGSTAB phase S: s = r - alpha v; t = S D^-1 s; <t,s>, <t,t>, <s,s>.
template <int K, typename TI, int C>
FEM_INLINE void phase_bi_s(const Inst& I, int row_lo, int row_hi, const TI* r, const TI* vnew, const Shared& sh,
                           double (&acc)[3]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI GA* sv = gp((TI*)I.s);  // own rows only
  TI GA* tv = gp((TI*)I.t);  // own rows only
  const TI GA* S = gp((const TI*)I.Si);
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const TI al = to_ti<TI>(sh.alpha[jr]);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    const TI so = ld<C>(r + o) - al * ld<C>(vnew + o);
    const TI ta = col_gather<4, TI>(ci, rp[row], rp[row + 1], [&](int s, int c, TI (&v)[4]) {
      const size_t oc = (size_t)c * K + jr;
      v[0] = S[(size_t)s * kv + vj];
      v[1] = dinv[(size_t)c * kv + vj];
      v[2] = ld<C>(r + oc);
      v[3] = ld<C>(vnew + oc);
    }, [&](const TI (&v)[4]) { return v[0] * (v[1] * (v[2] - al * v[3])); });
    sv[o] = so;
    tv[o] = ta;
    acc[0] += (double)ta * (double)so;
    acc[1] += (double)ta * (double)ta;
    acc[2] += (double)so * (double)so;
  }
}

// BiCGSTAB phase X: xi += D^-1 (alpha p + omega s); r = s - omega t; <rh,r>, <r,r>.
template <int K, typename TI, int C>
FEM_INLINE void phase_bi_x(const Inst& I, int row_lo, int row_hi, TI* r, const TI* p, const Shared& sh,
                           double (&acc)[2]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI* xi = (TI*)I.xi;
  const TI GA* rh = gp((const TI*)I.rh);
  const TI GA* sv = gp((const TI*)I.s);
  const TI GA* tv = gp((const TI*)I.t);
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const TI al = to_ti<TI>(sh.alpha[jr]);
  const TI om = to_ti<TI>(sh.omega[jr]);
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    const TI d = dinv[(size_t)row * kv + vj];
    st<C>(xi + o, ld<C>(xi + o) + d * (al * ld<C>(p + o) + om * sv[o]));
    const TI rr = sv[o] - om * tv[o];
    st<C>(r + o, rr);
    acc[0] += (double)rh[o] * (double)rr;
    acc[1] += (double)rr * (double)rr;
  }
}

// Fill the row cache for this workgroup's rows.  Whether the team caches is
// decided from quantities all its workgroups share.
template <int K, typename TI>
FEM_INLINE bool fill_cache(const Inst& I, int row_lo, int row_hi, int rows_per_wg, RowCache<TI>& RC) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  const TI GA* S = gp((const TI*)I.Si);
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  const bool ok = (rows_per_wg + RPP - 1) / RPP <= kCacheP && I.max_row <= kCacheE;
  if (ok) {
    for (int q = 0; q < kCacheP; q++) {
      const int row = row_lo + (int)threadIdx.x / K + q * RPP;
      int lo = 0, hi = 0;
      if (row < row_hi) {
        lo = rp[row];
        hi = rp[row + 1];
      }
      for (int e = 0; e < kCacheE; e++) {
        const int s = lo + e;
        const bool v = s < hi;
        const int c = v ? ci[s] : (row < row_hi ? row : 0);
        RC.col[q][e][threadIdx.x] = c;
        RC.val[q][e][threadIdx.x] = v ? S[(size_t)s * kv + vj] * dinv[(size_t)c * kv + vj] : (TI)0;
      }
    }
  }
  __syncthreads();
  return ok;
}

// Pipelined CG start from the cache (same arithmetic as phase_pcg_init).
template <int K, typename TI, int C>
FEM_INLINE void phase_pcg_init_c(const Inst& I, int row_lo, int row_hi, const TI* rc, TI* wc,
                                 const RowCache<TI>& RC, double (&acc)[2]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI* xi = (TI*)I.xi;
  const TI GA* dinv = gp((const TI*)I.dinvi);
  for (int q = 0; q < kCacheP; q++) {
    const int row = row_lo + (int)threadIdx.x / K + q * RPP;
    if (row >= row_hi) break;
    const size_t o = (size_t)row * K + jr;
    const double xo = ld<C>(I.x + o), xio = (double)ld<C>(xi + o);
    const TI ro = ld<C>(rc + o);
    const TI uo = dinv[(size_t)row * kv + vj] * ro;  // loaded before the stores below
    TI g[kCacheE];
#pragma unroll
    for (int e = 0; e < kCacheE; e++) g[e] = ld<C>(rc + (size_t)RC.col[q][e][threadIdx.x] * K + jr);
    TI wa = (TI)0;
#pragma unroll
    for (int e = 0; e < kCacheE; e++) wa += RC.val[q][e][threadIdx.x] * g[e];
    st<C>(I.x + o, xo + xio);
    st<C>(xi + o, (TI)0);
    st<C>(wc + o, wa);
    acc[0] += (double)ro * (double)uo;
    acc[1] += (double)uo * (double)wa;
  }
}

// One Chronopoulos-Gear iteration from the cache (same arithmetic as phase_pcg_iter).
template <int K, typename TI, int C>
FEM_INLINE void phase_pcg_iter_c(const Inst& I, int row_lo, int row_hi, const TI* rc, const TI* wc, const TI* sc,
                                 TI* rn, TI* wn, TI* sn, bool first, const Shared& sh, const RowCache<TI>& RC,
                                 double (&acc)[3]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI* xi = (TI*)I.xi;
  TI GA* p = gp((TI*)I.p0);  // own rows only
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const TI al = to_ti<TI>(sh.alpha[jr]);
  const TI be = first ? (TI)0 : to_ti<TI>(sh.beta[jr]);
  for (int q = 0; q < kCacheP; q++) {
    const int row = row_lo + (int)threadIdx.x / K + q * RPP;
    if (row >= row_hi) break;
    const size_t o = (size_t)row * K + jr;
    const TI ro = ld<C>(rc + o);
    const TI wo = ld<C>(wc + o);
    const TI so = first ? (TI)0 : ld<C>(sc + o);
    const TI po = first ? (TI)0 : p[o];
    const TI xio = ld<C>(xi + o);
    TI gr[kCacheE], gw[kCacheE], gs[kCacheE];
#pragma unroll
    for (int e = 0; e < kCacheE; e++) {
      const size_t oc = (size_t)RC.col[q][e][threadIdx.x] * K + jr;
      gr[e] = ld<C>(rc + oc);
      gw[e] = ld<C>(wc + oc);
      gs[e] = first ? (TI)0 : ld<C>(sc + oc);
    }
    TI wa = (TI)0;
#pragma unroll
    for (int e = 0; e < kCacheE; e++)
      wa += RC.val[q][e][threadIdx.x] * cg_r<TI>(gr[e], cg_s<TI>(gw[e], gs[e], be, first), al);
    const TI d = dinv[(size_t)row * kv + vj];
    const TI uo = d * ro;
    const TI pn = first ? uo : (uo + be * po);
    const TI sv = cg_s<TI>(wo, so, be, first);
    const TI rr = cg_r<TI>(ro, sv, al);
    p[o] = pn;
    st<C>(xi + o, xio + al * pn);
    st<C>(sn + o, sv);
    st<C>(rn + o, rr);
    st<C>(wn + o, wa);
    const TI un = d * rr;
    acc[0] += (double)rr * (double)un;
    acc[1] += (double)un * (double)wa;
    acc[2] += (double)rr * (double)rr;
  }
}

// BiCGSTAB phase P from the cache.
template <int K, typename TI, int C>
FEM_INLINE void phase_bi_p_c(const Inst& I, int row_lo, int row_hi, const TI* r, const TI* pold, TI* pnew,
                             const TI* vold, TI* vnew, bool first, const Shared& sh, const RowCache<TI>& RC,
                             double (&acc)[1]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  TI GA* rh = gp((TI*)I.rh);  // own rows only
  TI* xi = (TI*)I.xi;
  const TI be = first ? (TI)0 : to_ti<TI>(sh.beta[jr]);
  const TI om = first ? (TI)0 : to_ti<TI>(sh.omega[jr]);
  for (int q = 0; q < kCacheP; q++) {
    const int row = row_lo + (int)threadIdx.x / K + q * RPP;
    if (row >= row_hi) break;
    const size_t o = (size_t)row * K + jr;
    const TI ro = ld<C>(r + o);
    if (first) {
      st<C>(I.x + o, ld<C>(I.x + o) + (double)ld<C>(xi + o));
      st<C>(xi + o, (TI)0);
      rh[o] = ro;
    }
    TI gr[kCacheE], gp_[kCacheE], gv[kCacheE];
#pragma unroll
    for (int e = 0; e < kCacheE; e++) {
      const size_t oc = (size_t)RC.col[q][e][threadIdx.x] * K + jr;
      gr[e] = ld<C>(r + oc);
      gp_[e] = first ? (TI)0 : ld<C>(pold + oc);
      gv[e] = first ? (TI)0 : ld<C>(vold + oc);
    }
    TI va = (TI)0;
#pragma unroll
    for (int e = 0; e < kCacheE; e++)
      va += RC.val[q][e][threadIdx.x] * (first ? gr[e] : (gr[e] + be * (gp_[e] - om * gv[e])));
    const TI pn = first ? ro : (ro + be * (ld<C>(pold + o) - om * ld<C>(vold + o)));
    st<C>(pnew + o, pn);
    st<C>(vnew + o, va);
    acc[0] += (double)(first ? ro : rh[o]) * (double)va;
  }
}

// BiCGSTAB phase S from the cache.
template <int K, typename TI, int C>
FEM_INLINE void phase_bi_s_c(const Inst& I, int row_lo, int row_hi, const TI* r, const TI* vnew, const Shared& sh,
                             const RowCache<TI>& RC, double (&acc)[3]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  TI GA* sv = gp((TI*)I.s);  // own rows only
  TI GA* tv = gp((TI*)I.t);  // own rows only
  const TI al = to_ti<TI>(sh.alpha[jr]);
  for (int q = 0; q < kCacheP; q++) {
    const int row = row_lo + (int)threadIdx.x / K + q * RPP;
    if (row >= row_hi) break;
    const size_t o = (size_t)row * K + jr;
    const TI so = ld<C>(r + o) - al * ld<C>(vnew + o);
    TI gr[kCacheE], gv[kCacheE];
#pragma unroll
    for (int e = 0; e < kCacheE; e++) {
      const size_t oc = (size_t)RC.col[q][e][threadIdx.x] * K + jr;
      gr[e] = ld<C>(r + oc);
      gv[e] = ld<C>(vnew + oc);
    }
    TI ta = (TI)0;
#pragma unroll
    for (int e = 0; e < kCacheE; e++) ta += RC.val[q][e][threadIdx.x] * (gr[e] - al * gv[e]);
    sv[o] = so;
    tv[o] = ta;
    acc[0] += (double)ta * (double)so;
    acc[1] += (double)ta * (double)ta;
    acc[2] += (double)so * (double)so;
  }
}

// Fill the pool for this workgroup's rows of a team-instance.  Rows are owned
// by the same lane for the whole launch, and the inner-precision matrix and
// preconditioner do not change during it.  Unused entries point at the row
// itself with weight 0, so the unrolled gather is branch-free and every place
// is valid.  Whether the team keeps its rows this way is decided from
// quantities all its workgroups share -- the rows each is dealt, the
// instance's longest row, and whether every halo fits (halo->ok) -- so all
// agree: the pipelined CG then starts inside the update phase, one barrier
// fewer, and a team whose workgroups disagreed would wait at different
// barriers.  A one-workgroup team has no halo.
template <int K, typename TI, int C>
FEM_INLINE bool fill_rows(const Inst& I, const Team& T, const HaloRef* halo, int rank, int row_lo, int row_hi,
                          int rows_per_wg, unsigned char LA* pool, Rows<TI>& R) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  const TI GA* S = gp((const TI*)I.Si);
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  const int passes = (rows_per_wg + RPP - 1) / RPP;
  if (passes > kCacheP || I.max_row > kCacheE) return false;
  const bool lone = C == kPlain || T.size == 1;
  HaloRef H{};
  if (!lone) {
    if (!halo || !I.xch) return false;
    H = *halo;
    if (!H.ok) return false;
  }
  const int cells = passes * kCacheE * kTB;
  R.val = (TI LA*)pool;
  R.col = (unsigned short LA*)(R.val + cells);
  R.nhalo = lone ? 0 : gp(H.n)[rank];
  R.own = (row_hi - row_lo) * K;
  R.nx = R.nhalo * K;
  R.nvals = R.own + R.nx;
  int LA* list = (int LA*)(pool + rows_pool<C, TI>()) - R.nhalo;
  R.list = list;
  R.hv = pool + rows_cells_bytes(passes, kTB, (int)sizeof(TI));
  if (!lone) {
    const int GA* src = gp(H.list) + (size_t)rank * H.cap;
    for (int t = threadIdx.x; t < R.nhalo; t += kTB) list[t] = src[t];
    // exchange words of an earlier launch carry epochs this one will use (the
    // first barrier, before any word is polled, waits for these stores)
    const size_t nk = (size_t)I.n * K;
    for (int arr = 0; arr < 3; arr++) {
      const int per = arr < 2 ? kXW<TI> : kXW<double>;
      xword* at = I.xch + arr * nk * kXW<TI> + (size_t)row_lo * K * per;
      for (int t = threadIdx.x; t < R.own * per; t += kTB) st<kCoherent>(at + t, (xword)0);
    }
  }
  // what the residual pass may stage, the same for all workgroups of the team
  {
    const int most = H.max_n;
    const int bytes = rows_pool<C, TI>() - rows_cells_bytes(passes, kTB, (int)sizeof(TI)) - 4 * most;
    const int vals = (rows_per_wg + most) * K;
    R.res = 16 * vals <= bytes ? 2 : 8 * vals <= bytes ? 1 : 0;
  }
  const unsigned short GA* places = gp(H.place) + (size_t)rank * H.place_n;
  for (int q = 0; q < passes; q++) {
    const int row = row_lo + (int)threadIdx.x / K + q * RPP;
    int lo = 0, hi = 0;
    if (row < row_hi) {
      lo = rp[row];
      hi = rp[row + 1];
    }
    const int self = row < row_hi ? row - row_lo : 0;
    // all entries' loads in flight at once: indices clamped to the row, not
    // guarded entry by entry (12 us of a launch with 512 rows per workgroup)
    int c[kCacheE], place[kCacheE];
    TI v[kCacheE];
    if (hi > lo) {
#pragma unroll
      for (int e = 0; e < kCacheE; e++) {
        const int s = min(lo + e, hi - 1);
        c[e] = ci[s];
        v[e] = S[(size_t)s * kv + vj];
        place[e] = lone ? 0 : (int)places[(q * kCacheE + e) * kTB + (int)threadIdx.x];
      }
#pragma unroll
      for (int e = 0; e < kCacheE; e++) v[e] *= dinv[(size_t)c[e] * kv + vj];
    }
#pragma unroll
    for (int e = 0; e < kCacheE; e++) {
      const bool on = lo + e < hi;
      const int at = (q * kCacheE + e) * kTB + (int)threadIdx.x;
      R.col[at] = (unsigned short)((!on ? self : lone ? c[e] - row_lo : place[e]) * K + jr);
      R.val[at] = on ? v[e] : (TI)0;
    }
  }
  __syncthreads();
  return true;
}

// phase_res for rows in the pool: x + xi (and, for the fused step, the next
// guess's history part) is staged once per row read, and the lanes gather it
// from LDS.  The matrix rows are read from memory, the first pass's while the
// staging loads are in flight.  Same per-row arithmetic as phase_res; for the
// fused step with lvn > 0, hvec holds the history part (hready).  The
// candidate is exchanged in words tagged for the reduction that ends this
// phase (epoch `tag`): no barrier separates it from the sweep before.
template <int K, typename TI, int C>
FEM_INLINE void phase_res_rows(const Inst& I, const Team& T, int row_lo, int row_hi, TI* r, TeamShared& sh,
                               const Rows<TI>& R, double (&acc)[2], int lvn, double* hpre, unsigned tag) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  TI* xi = (TI*)I.xi;
  const bool drop = sh.reset[jr] != 0;
  const bool zero = sh.bb[jr] == 0.0;
  const bool warm = I.warm != 0;
  const double inv_dt = 1.0 / I.dt;
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const int GA* __restrict__ rp = gp(I.rp);
  const double GA* S64 = gp(I.S64);
  const double GA* M64 = gp(I.M64);
  const bool want_h = hpre && lvn > 0;
  const double w0 = lvn + 1.0;  // pred_weights
  double LA* cv = (double LA*)R.hv;
  double LA* hc = cv + R.nvals;  // the history part behind the candidate (Rows::res)
  struct Row {
    double s[kCacheE], m[kCacheE], b;
    TI d;
  };
  auto load = [&](int row, Row& w) {
    if (row >= row_hi) return;
    const int lo = rp[row], hi = rp[row + 1];
    if (hi > lo) {  // a vertex without triangles has no entries
#pragma unroll
      for (int e = 0; e < kCacheE; e++) {
        const int s = min(lo + e, hi - 1);  // past the row's end: its weights are 0 below
        w.s[e] = S64[(size_t)s * kv + vj];
        w.m[e] = hpre ? M64[s] : 0.0;
      }
    }
#pragma unroll
    for (int e = 0; e < kCacheE; e++)
      if (lo + e >= hi) w.s[e] = w.m[e] = 0.0;
    w.b = gp(I.b)[(size_t)row * K + jr];
    w.d = dinv[(size_t)row * kv + vj];
  };
  const int row0 = row_lo + (int)threadIdx.x / K;
  Row w;
  load(row0, w);
  const bool share = C != kPlain && T.size > 1;
  xword* xc = I.xch + 2 * (size_t)I.n * K * kXW<TI>;
  for (int row = row0; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    const int at = (row - row_lo) * K + jr;
    const double c = ld<C>(I.x + o) + (drop ? 0.0 : (double)ld<C>(xi + o));
    if (share) put_words<double>(xc, o, c, tag);
    cv[at] = c;
    if (want_h) hc[at] = ld<C>(I.hvec + o);
  }
  if (want_h) stage_halo<K>(R, hc, [&](size_t oc) { return ld<C>(I.hvec + oc); });
  int to = 0;
  if constexpr (C != kPlain) take_halo<K, double>(T, R, xc, cv + R.own, tag, &to);
  if (to) sh.tmo = 1;  // the reduction that ends the phase sees it and stops
  __syncthreads();
  for (int row = row0, q = 0; row < row_hi; row += RPP, q++) {
    if (q > 0) load(row, w);
    const size_t o = (size_t)row * K + jr;
    const int at = q * kCacheE * kTB + (int)threadIdx.x;
    double sc = 0.0, mc = 0.0, sh_ = 0.0;
#pragma unroll
    for (int e = 0; e < kCacheE; e++) {
      const int place = R.col[at + e * kTB];
      const double c = cv[place];
      sc += w.s[e] * c;
      if (hpre) mc += w.m[e] * c;
      if (want_h) sh_ += w.s[e] * hc[place];
    }
    if (hpre) {
      const double su = zero ? 0.0 : sc;
      double bn = (zero ? 0.0 : mc) * inv_dt;
      if (I.eq == EQ_GS) {  // CPUSolver.cpp:134,137 at the candidate
        const int own = (row - row_lo) * K;
        const double uu = sh.bb[0] == 0.0 ? 0.0 : cv[own];
        const double vv = K < 2 || sh.bb[K < 2 ? 0 : 1] == 0.0 ? 0.0 : cv[own + (K < 2 ? 0 : 1)];
        const double uvv = uu * (vv * vv);
        const double fr = (jr == 0) ? (-uvv + I.p3 * (1.0 - uu)) : (uvv - (I.p3 + I.p4) * vv);
        bn += (I.weighting ? gp(I.lumped)[row] : 1.0) * fr;
      }
      gp(I.xnext)[o] = bn;
      st<C>(hpre + o, bn - (warm ? w0 * su + (want_h ? sh_ : 0.0) : 0.0));
    }
    const double r64 = w.b - sc;
    const TI rr = to_ti<TI>(r64);
    st<C>(r + o, rr);
    if (drop) st<C>(xi + o, (TI)0);
    acc[0] += r64 * r64;
    acc[1] += (I.krylov == 1) ? (double)rr * (double)rr : (double)rr * (double)(w.d * rr);
  }
}

// State update and the instability rule (CPUSolver.cpp:41-48, widened to
// flag NaN/Inf separately).
// With lvn >= 0 (heat, advection-diffusion, Gray-Scott), also the next
// step's initial guess of predictor order lvn into xnext, from this row's own
// history: the next right-hand side then gathers one vector for S x0.
template <int K, typename TI, int C>
FEM_INLINE void phase_update(const Inst& I, int row_lo, int row_hi, const Shared& sh, int* flags, int step,
                             int lvn = -1) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  TI* xi = (TI*)I.xi;
  int f = 0;
  double* traj = nullptr;  // trajectory record of this step, if any
  if (I.traj && (step + 1) % I.traj_every == 0)
    traj = I.traj + (size_t)((step + 1) / I.traj_every - 1) * I.n * K;
  const bool first_order = I.eq == EQ_HEAT || I.eq == EQ_ADVDIFF || I.eq == EQ_GS;
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    // every load of the row first: loads and stores share one completion
    // counter, so a load issued after a store also waits for the store
    double xf = ld<C>(I.x + o) + (double)ld<C>(xi + o);
    const double uo = ld<C>(I.u + o);
    const double ao = (first_order ? I.extrap >= 2 : I.eq == EQ_NEWMARK) ? ld<C>(I.a + o) : 0.0;
    const double vo = (first_order ? I.extrap >= 3 : (I.eq == EQ_WAVE || I.eq == EQ_NEWMARK)) ? ld<C>(I.v + o) : 0.0;
    const double ho = (first_order ? I.extrap >= 4 : (I.eq == EQ_NEWMARK && I.extrap >= 2)) ? ld<C>(I.h3 + o) : 0.0;
    if (sh.bb[jr] == 0.0) xf = 0.0;  // Eigen: rhs == 0 -> x = 0
    st<C>(I.x + o, xf);
    st<C>(xi + o, (TI)0);
    double c1 = xf, c2 = 0.0, up = xf;  // up: new primary variable
    switch (I.eq) {
      case EQ_HEAT:
      case EQ_ADVDIFF:
      case EQ_GS:
        if (I.extrap) {  // history for the predictor: x_{n-4} <- x_{n-3} <- x_{n-2} <- x_{n-1} <- x_n
          if (I.extrap >= 4) st<C>(I.h4 + o, ho);
          if (I.extrap >= 3) st<C>(I.h3 + o, vo);
          if (I.extrap >= 2) st<C>(I.v + o, ao);
          st<C>(I.a + o, uo);
          if (lvn >= 0 && I.xnext) {
            double w0, w1, w2, w3, w4;
            pred_weights(lvn, w0, w1, w2, w3, w4);
            gp(I.xnext)[o] = w0 * xf + w1 * uo + w2 * ao + w3 * vo + w4 * ho;
          }
        }
        st<C>(I.u + o, xf);
        break;
      case EQ_WAVE: {
        if (I.extrap) st<C>(I.a + o, vo);
        st<C>(I.v + o, xf);
        const double un = uo + xf * I.dt;  // CPUSolver.cpp:118
        st<C>(I.u + o, un);
        c2 = un;
        up = un;
      } break;
      case EQ_NEWMARK: {
        const double dt = I.dt, be = I.p2, ga = I.p3;
        const double ut = uo + dt * vo + (0.5 - be) * dt * dt * ao;
        const double un = ut + be * dt * dt * xf;
        const double vn = vo + dt * ((1.0 - ga) * ao + ga * xf);
        st<C>(I.u + o, un);
        st<C>(I.v + o, vn);
        if (I.extrap >= 2) st<C>(I.h4 + o, ho);  // acceleration history for the predictor
        if (I.extrap >= 1) st<C>(I.h3 + o, ao);
        st<C>(I.a + o, xf);
        c1 = un;
        c2 = vn;
        up = un;
      } break;
      default:
        break;
    }
    if (traj) gp(traj)[o] = up;
    if (c1 > 1e4 || c2 > 1e4) f |= ST_UNSTABLE;
    if (!isfinite(c1) || !isfinite(c2)) f |= ST_NONFINITE;
  }
  if (f) atomicOr(flags, f);
}

// The state update of step `step` and the right-hand side of step + 1 as one
// phase (heat, advection-diffusion, Gray-Scott: the new state is the
// solution).  Neighbours are gathered only through x + xi, which no
// workgroup writes in this phase; everything written belongs to the
// workgroup's own rows: the state and predictor history, b, r, and the next
// initial guess in xnext, which phase_install moves into x (xi = 0) after the
// barrier.  The history part of S x0 comes from hpre (phase_res or
// phase_hpre of this step); lvn is the next step's predictor order.  pre:
// the last residual pass of this step already formed b (in xnext) and the
// initial residual r (in hpre), so no neighbour state is gathered.  lvh > 0:
// also the history part of the initial guess after that into hvec.
// R (with pre; pipelined CG, rows in the pool): also the start of that CG,
// w = S D^-1 r into wq from the neighbours' r in hpre, so the sweep needs no
// start phase of its own; acc[3] then sums <D^-1 r, w>.
template <int K, typename TI, int C, bool START>
FEM_INLINE void phase_update_rhs(const Inst& I, int row_lo, int row_hi, TI* r, const Shared& sh, int* flags, int step,
                                 int lvn, int lvh, bool pre, const Rows<TI>* R, TI* wq, double (&acc)[4]) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  const TI* xi = (const TI*)I.xi;
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const double inv_dt = 1.0 / I.dt;
  const bool warm = I.warm != 0;
  double w0, w1, w2, w3, w4;
  pred_weights(lvn, w0, w1, w2, w3, w4);
  double h0, h1, h2, h3, h4;  // lvh: the step after this one (its history combination goes to hvec)
  pred_weights(lvh, h0, h1, h2, h3, h4);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  const double GA* M64 = gp(I.M64);
  const double GA* S64 = gp(I.S64);
  int f = 0;
  double* traj = nullptr;  // trajectory record of this step, if any
  if (I.traj && (step + 1) % I.traj_every == 0)
    traj = I.traj + (size_t)((step + 1) / I.traj_every - 1) * I.n * K;
  // this step's solution of column j at offset idx (Eigen: rhs == 0 -> x = 0)
  auto xn_at = [&](size_t idx, int j) -> double {
    return sh.bb[j] == 0.0 ? 0.0 : ld<C>(I.x + idx) + (double)ld<C>(xi + idx);
  };
  if constexpr (!START) R = nullptr;
  TI LA* hv = R ? (TI LA*)R->hv : nullptr;
  if (R) {
    stage_halo<K>(*R, hv, [&](size_t oc) { return to_ti<TI>(ld<C>(I.hpre + oc)); });
    for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP)
      hv[(row - row_lo) * K + jr] = to_ti<TI>(ld<C>(I.hpre + (size_t)row * K + jr));
    __syncthreads();
  }
  int q = 0;  // pass over the workgroup's rows
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP, q++) {
    const size_t o = (size_t)row * K + jr;
    // every load of the row first: loads and stores share one completion
    // counter, so a load issued after a store also waits for the store
    const double xn = xn_at(o, jr);
    const double uo = ld<C>(I.u + o);
    const double ao = I.extrap >= 2 ? ld<C>(I.a + o) : 0.0;
    const double vo = I.extrap >= 3 ? ld<C>(I.v + o) : 0.0;
    const double ho = I.extrap >= 4 ? ld<C>(I.h3 + o) : 0.0;
    // ---- next right-hand side: b = (M/dt) x_n (+ Gray-Scott reaction), r = b - S x0
    double b, r64;
    TI wa = (TI)0;  // S D^-1 r (with R)
    if (pre) {      // both formed by the last residual pass of this step
      b = gp(I.xnext)[o];
      r64 = ld<C>(I.hpre + o);
      if (R) wa = rows_gather(*R, (const TI LA*)hv, q);
    } else {
      const D2 g = row_gather(rp[row], rp[row + 1], D2{0.0, 0.0}, [&](int s) {
        const double xc = xn_at((size_t)ci[s] * K + jr, jr);
        return D2{M64[s] * xc, warm ? S64[(size_t)s * kv + vj] * xc : 0.0};
      });
      b = g.a * inv_dt;
      if (I.eq == EQ_GS) {  // CPUSolver.cpp:134,137 with the new state
        const double uu = xn_at((size_t)row * K, 0), vv = xn_at((size_t)row * K + 1, 1);
        const double uvv = uu * (vv * vv);
        const double fr = (jr == 0) ? (-uvv + I.p3 * (1.0 - uu)) : (uvv - (I.p3 + I.p4) * vv);
        const double w = I.weighting ? gp(I.lumped)[row] : 1.0;
        b += w * fr;
      }
      r64 = b - (warm ? w0 * g.b + (lvn > 0 ? gp(I.hpre)[o] : 0.0) : 0.0);
    }
    const TI dj = dinv[(size_t)row * kv + vj];
    const double x0 = warm ? w0 * xn + w1 * uo + w2 * ao + w3 * vo + w4 * ho : 0.0;
    const TI rr = to_ti<TI>(r64);
    // ---- update: state and history x_{n-3} <- x_{n-2} <- x_{n-1} <- x_n (own row)
    if (I.extrap >= 4) st<C>(I.h4 + o, ho);
    if (I.extrap >= 3) st<C>(I.h3 + o, vo);
    if (I.extrap >= 2) st<C>(I.v + o, ao);
    if (I.extrap >= 1) st<C>(I.a + o, uo);
    st<C>(I.u + o, xn);
    // the shifted history is x_n, x_{n-1}, x_{n-2}, x_{n-3}
    if (lvh > 0) st<C>(I.hvec + o, h1 * xn + h2 * uo + h3 * ao + h4 * vo);
    if (traj) gp(traj)[o] = xn;
    if (xn > 1e4) f |= ST_UNSTABLE;
    if (!isfinite(xn)) f |= ST_NONFINITE;
    gp(I.b)[o] = b;
    gp(I.xnext)[o] = x0;
    st<C>(r + o, rr);
    if (R) st<C>(wq + o, wa);
    acc[0] += b * b;
    acc[1] += r64 * r64;
    const TI uz = dj * rr;
    acc[2] += (I.krylov == 1) ? (double)rr * (double)rr : (double)rr * (double)uz;
    if (R) acc[3] += (double)uz * (double)wa;
  }
  if (f) atomicOr(flags, f);
}

// Own rows: x = xnext, xi = 0 (the initial guess phase_update_rhs prepared).
template <int K, typename TI, int C>
FEM_INLINE void phase_install(const Inst& I, int row_lo, int row_hi) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  TI* xi = (TI*)I.xi;
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    st<C>(I.x + o, gp(I.xnext)[o]);
    st<C>(xi + o, (TI)0);
  }
}

// The history part of the next step's initial residual (as phase_res does)
// for a step that ran no refinement sweep.
template <int K, typename TI, int C>
FEM_INLINE void phase_hpre(const Inst& I, int row_lo, int row_hi, int lvn, bool hready) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  double w0, w1, w2, w3, w4;
  pred_weights(lvn, w0, w1, w2, w3, w4);
  const int GA* __restrict__ rp = gp(I.rp);
  const int GA* __restrict__ ci = gp(I.ci);
  const double GA* S64 = gp(I.S64);
  for (int row = row_lo + (int)threadIdx.x / K; row < row_hi; row += RPP) {
    const size_t o = (size_t)row * K + jr;
    if (hready) {
      gp(I.hpre)[o] = row_gather(rp[row], rp[row + 1], 0.0, [&](int s) {
        return S64[(size_t)s * kv + vj] * ld<C>(I.hvec + (size_t)ci[s] * K + jr);
      });
      continue;
    }
    gp(I.hpre)[o] = row_gather<kUWide>(rp[row], rp[row + 1], 0.0, [&](int s) {
      const size_t oc = (size_t)ci[s] * K + jr;
      const double hv = w1 * ld<C>(I.u + oc) + (lvn >= 2 ? w2 * ld<C>(I.a + oc) : 0.0) +
                        (lvn >= 3 ? w3 * ld<C>(I.v + oc) : 0.0) + (lvn >= 4 ? w4 * ld<C>(I.h3 + oc) : 0.0);
      return S64[(size_t)s * kv + vj] * hv;
    });
  }
}

// ---------------------------------------------------------------------------
// Krylov drivers (uniform control flow across the team)
// ---------------------------------------------------------------------------

// The control wave's scalars of the pipelined CG (K <= 64 columns, one lane
// each).  Start: gamma = <r, D^-1 r>, delta = <D^-1 r, w>.
template <int K>
FEM_INLINE void pcg_start(TeamShared& sh) {
  const int j = ctl();
  if (j >= K) return;
  const double g = sh.red[j], d = sh.red[K + j];
  sh.gamma[j] = g;
  sh.alpha[j] = (sh.active[j] && d != 0.0) ? g / d : 0.0;
  sh.beta[j] = 0.0;
}
// While an iteration's phase runs: 1 / gamma and 1 / alpha, so that one
// division is left after its reduction.
template <int K>
FEM_INLINE void pcg_inverses(TeamShared& sh) {
  const int j = ctl();
  if (j < 0 || j >= K) return;
  sh.ig[j] = 1.0 / sh.gamma[j];
  sh.ia[j] = 1.0 / sh.alpha[j];
}
// After an iteration's reduction: the next alpha and beta, and the stop vote.
template <int K>
FEM_INLINE void pcg_scalars(const Inst& I, TeamShared& sh, int it_s, int its) {
  const int j = ctl();
  bool done = true;
  if (j < K) {
    const double g = sh.red[j], d = sh.red[K + j], rr = sh.red[2 * K + j];
    done = !sh.active[j] || rr < sh.ithr[j] || !(rr == rr);
    double be = 0.0, al = 0.0;
    if (!done && sh.gamma[j] != 0.0 && sh.alpha[j] != 0.0) {
      be = g * sh.ig[j];
      const double den = d - be * g * sh.ia[j];
      al = (den != 0.0) ? g / den : 0.0;
    }
    sh.beta[j] = be;
    sh.alpha[j] = al;
    sh.gamma[j] = g;
  }
  const bool alldone = __all(done);
  if (j == 0) sh.uni = alldone || it_s >= I.max_inner || its >= I.max_iters;
}

// Pipelined (Chronopoulos-Gear) PCG on the current sweep; r starts in I.r.
template <int K, typename TI, int C>
FEM_INLINE bool krylov_pcg(const Inst& I, const Team& T, int rank, unsigned& e, TeamShared& sh, int row_lo, int row_hi,
                           int& its, const RowCache<TI>* RC) {
  TI* rb[2] = {(TI*)I.r, (TI*)I.z};
  TI* wb[2] = {(TI*)I.q, (TI*)I.rh};
  TI* sb[2] = {(TI*)I.s, (TI*)I.t};
  int par = 0;
  {
    double acc[2] = {0.0, 0.0};
    if (RC) phase_pcg_init_c<K, TI, C>(I, row_lo, row_hi, rb[0], wb[0], *RC, acc);
    else phase_pcg_init<K, TI, C>(I, row_lo, row_hi, rb[0], wb[0], acc);
    if (!team_reduce<K, 2, C>(acc, T, rank, e, sh, [&] { pcg_start<K>(sh); })) return false;
  }
  int it_s = 0;
  bool first = true;
  while (true) {
    double acc[3] = {0.0, 0.0, 0.0};
    pcg_inverses<K>(sh);
    if (RC)
      phase_pcg_iter_c<K, TI, C>(I, row_lo, row_hi, rb[par], wb[par], sb[par], rb[par ^ 1], wb[par ^ 1], sb[par ^ 1],
                                 first, sh, *RC, acc);
    else
      phase_pcg_iter<K, TI, C>(I, row_lo, row_hi, rb[par], wb[par], sb[par], rb[par ^ 1], wb[par ^ 1], sb[par ^ 1],
                               first, sh, acc);
    par ^= 1;
    first = false;
    it_s++;
    its++;
    if (!team_reduce<K, 3, C>(acc, T, rank, e, sh, [&] { pcg_scalars<K>(I, sh, it_s, its); })) return false;
    if (sh.uni) break;
  }
  return true;
}

// The same with the rows in the pool.  A lane's entries of x, r, w, s, p stay
// in registers for the sweep, and the halo's r, s, w in LDS: its new r and s
// are formed by the owner's operations, so per iteration only w is exchanged,
// in words polled together with the iteration's sums (double-buffered by
// epoch: a workgroup that has passed a barrier may publish the next w while
// another still takes this one).  xi goes to memory when the sweep ends.
// started: the update phase already formed w = S D^-1 r and the start
// scalars (x holds the initial guess, xi = 0).
// Latency-bound: publishing the sums, polling them and the words (~1.5 us), the
// scalars, and the LDS gather.  Device time of a run over its iterations, the
// residuals and right-hand sides included (us; three coherent loads per entry
// from memory, and now): 3,969 FP64 rows 6.3 -> 3.1; 39,601 rows 7.3 -> 4.3;
// 259,000 rows 12.2 -> 5.1; BiCGSTAB on 261,000 rows 48 -> 16.  An iteration of
// the loop alone (140 against 40 in one sweep): 2.7, 3.0, 4.1 and 10.4.
template <int K, typename TI, int C>
FEM_INLINE bool krylov_pcg_rows(const Inst& I, const Team& T, int rank, unsigned& e, TeamShared& sh, int row_lo,
                                int row_hi, int& its, const Rows<TI>& R, bool started) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  const TI* rg = (const TI*)I.r;
  const TI* wg = (const TI*)I.q;
  TI* xi = (TI*)I.xi;
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const bool share = C != kPlain && T.size > 1;  // other workgroups read this one's rows
  const size_t xn = (size_t)I.n * K * kXW<TI>;   // words of one exchange buffer
  TI LA* hv = (TI LA*)R.hv;     // r: own rows, halo
  TI LA* hr = hv + R.own;
  TI LA* hs = hv + R.nvals;     // the halo's s and w
  TI LA* hw = hs + R.nx;
  const int row0 = row_lo + (int)threadIdx.x / K;
  RowCells<TI> cells;
  load_cells<K>(R, row0, row_hi, cells);
  TI r[kCacheP], w[kCacheP], s[kCacheP], p[kCacheP], x[kCacheP], d[kCacheP];
#pragma unroll
  for (int q = 0; q < kCacheP; q++) {
    r[q] = w[q] = s[q] = p[q] = x[q] = d[q] = (TI)0;
    const int row = row0 + q * RPP;
    if (row >= row_hi) continue;
    const size_t o = (size_t)row * K + jr;
    r[q] = ld<C>(rg + o);
    d[q] = dinv[(size_t)row * kv + vj];
    if (started) w[q] = ld<C>(wg + o);
  }
  stage_halo<K>(R, hv, [&](size_t oc) { return ld<C>(rg + oc); });
  if (started) {
    stage_halo<K>(R, hw - R.own, [&](size_t oc) { return ld<C>(wg + oc); });
  } else {
    double xo[kCacheP];
#pragma unroll
    for (int q = 0; q < kCacheP; q++) {
      const int row = row0 + q * RPP;
      if (row >= row_hi) continue;
      const size_t o = (size_t)row * K + jr;
      xo[q] = ld<C>(I.x + o) + (double)ld<C>(xi + o);
      hv[(row - row_lo) * K + jr] = r[q];
    }
    __syncthreads();
    xword* xw = I.xch + ((e + 1) & 1) * xn;
    double acc[2] = {0.0, 0.0};
#pragma unroll
    for (int q = 0; q < kCacheP; q++) {
      const int row = row0 + q * RPP;
      if (row >= row_hi) continue;
      const size_t o = (size_t)row * K + jr;
      st<C>(I.x + o, xo[q]);
      w[q] = cells_gather(cells, (const TI LA*)hv, q);
      if (share) put_words<TI>(xw, o, w[q], e + 1);
      const TI uo = d[q] * r[q];
      acc[0] += (double)r[q] * (double)uo;
      acc[1] += (double)uo * (double)w[q];
    }
    if (!rows_reduce<K, 2, C>(acc, T, rank, e, sh, TakeHalo<K, TI>{R, xw, hw}, [&] { pcg_start<K>(sh); }))
      return false;
  }
  int it_s = 0;
  bool first = true;
  while (true) {
    const TI al = to_ti<TI>(sh.alpha[jr]);
    const TI be = first ? (TI)0 : to_ti<TI>(sh.beta[jr]);
    pcg_inverses<K>(sh);
    for (int t = halo_lane<K>(); t < R.nx; t += kHaloLanes) {
      const TI sv = cg_s<TI>(hw[t], first ? (TI)0 : hs[t], be, first);
      hs[t] = sv;
      hr[t] = cg_r<TI>(hr[t], sv, al);
    }
#pragma unroll
    for (int q = 0; q < kCacheP; q++) {
      const int row = row0 + q * RPP;
      if (row >= row_hi) continue;
      const TI uo = d[q] * r[q];
      p[q] = first ? uo : (uo + be * p[q]);
      s[q] = cg_s<TI>(w[q], s[q], be, first);
      r[q] = cg_r<TI>(r[q], s[q], al);
      x[q] = x[q] + al * p[q];
      hv[(row - row_lo) * K + jr] = r[q];
    }
    __syncthreads();
    xword* xw = I.xch + ((e + 1) & 1) * xn;
    double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
    for (int q = 0; q < kCacheP; q++) {
      const int row = row0 + q * RPP;
      if (row >= row_hi) continue;
      w[q] = cells_gather(cells, (const TI LA*)hv, q);
      if (share) put_words<TI>(xw, (size_t)row * K + jr, w[q], e + 1);
      const TI un = d[q] * r[q];
      acc[0] += (double)r[q] * (double)un;
      acc[1] += (double)un * (double)w[q];
      acc[2] += (double)r[q] * (double)r[q];
    }
    first = false;
    it_s++;
    its++;
    if (!rows_reduce<K, 3, C>(acc, T, rank, e, sh, TakeHalo<K, TI>{R, xw, hw},
                              [&] { pcg_scalars<K>(I, sh, it_s, its); }))
      return false;
    if (sh.uni) break;
  }
#pragma unroll
  for (int q = 0; q < kCacheP; q++) {
    const int row = row0 + q * RPP;
    if (row < row_hi) st<C>(xi + (size_t)row * K + jr, x[q]);
  }
  return true;
}

template <int K, typename TI, int C>
FEM_INLINE bool krylov_cg_classic(const Inst& I, const Team& T, int rank, unsigned& e, TeamShared& sh, int row_lo,
                                  int row_hi, int& its) {
  TI* r = (TI*)I.r;
  TI* pa = (TI*)I.p0;
  TI* pb = (TI*)I.p1b;
  int it_s = 0;
  bool first = true;
  while (true) {
    {
      double acc[1] = {0.0};
      phase_cg_a<K, TI, C>(I, row_lo, row_hi, r, pa, pb, first, sh, acc);
      const bool ok = team_reduce<K, 1, C>(acc, T, rank, e, sh, [&] {
        const int j = ctl();
        if (j >= K) return;
        const double pq = sh.red[j];
        sh.alpha[j] = (sh.active[j] && pq != 0.0) ? sh.gamma[j] / pq : 0.0;
      });
      if (!ok) return false;
    }
    {
      double acc[2] = {0.0, 0.0};
      phase_cg_b<K, TI, C>(I, row_lo, row_hi, r, pb, sh, acc);
      it_s++;
      its++;
      const bool ok = team_reduce<K, 2, C>(acc, T, rank, e, sh, [&] {
        const int j = ctl();
        bool done = true;
        if (j < K) {
          const double rz = sh.red[j], rr = sh.red[K + j];
          const double g = sh.gamma[j];
          sh.beta[j] = (g != 0.0) ? rz / g : 0.0;
          sh.gamma[j] = rz;
          done = !sh.active[j] || rr < sh.ithr[j] || !(rr == rr);
        }
        const bool alldone = __all(done);
        if (j == 0) sh.uni = alldone || it_s >= I.max_inner || its >= I.max_iters;
      });
      if (!ok) return false;
    }
    if (sh.uni) break;
    first = false;
    TI* tmp = pa;
    pa = pb;
    pb = tmp;
  }
  return true;
}

// BiCGSTAB's scalars after phases P, S and X (control wave).
template <int K>
FEM_INLINE void bi_alpha(TeamShared& sh) {
  const int j = ctl();
  if (j >= K) return;
  const double rv = sh.red[j];
  const double a = (sh.active[j] && rv != 0.0) ? sh.gamma[j] / rv : 0.0;
  // near-breakdown: a step the inner precision cannot represent restarts the sweep
  const bool fine = fabs(a) < 1e30;
  sh.alpha[j] = fine ? a : 0.0;
  if (!fine) sh.bkd = 1;
}
template <int K>
FEM_INLINE void bi_omega(TeamShared& sh) {
  const int j = ctl();
  if (j >= K) return;
  const double ts = sh.red[j], tt = sh.red[K + j], ss = sh.red[2 * K + j];
  const double om = (sh.active[j] && tt > 0.0 && !(ss < sh.ithr[j])) ? ts / tt : 0.0;
  const bool fine = fabs(om) < 1e30;
  sh.omega[j] = fine ? om : 0.0;
  if (!fine) sh.bkd = 1;
}
template <int K>
FEM_INLINE void bi_beta(const Inst& I, TeamShared& sh, int it_s, int its) {
  const int j = ctl();
  bool done = true, brk = false;
  if (j < K) {
    const double rho_new = sh.red[j], rr = sh.red[K + j];
    done = !sh.active[j] || rr < sh.ithr[j] || !(rr == rr);
    if (!done) {
      const double om = sh.omega[j], rho = sh.gamma[j];
      const double be = (om == 0.0 || rho == 0.0) ? 0.0 : (rho_new / rho) * (sh.alpha[j] / om);
      if (be == 0.0 || !(fabs(be) < 1e30)) brk = true;  // breakdown: restart the sweep
      else sh.beta[j] = be;
    }
    sh.gamma[j] = rho_new;
  }
  const bool alldone = __all(done), anybrk = __any(brk);
  if (j == 0) {
    sh.uni = alldone || anybrk || sh.bkd || it_s >= I.max_inner || its >= I.max_iters;
    sh.bkd = 0;
  }
}

template <int K, typename TI, int C>
FEM_INLINE bool krylov_bicgstab(const Inst& I, const Team& T, int rank, unsigned& e, TeamShared& sh, int row_lo,
                                int row_hi, int& its, const RowCache<TI>* RC) {
  TI* r = (TI*)I.r;
  TI* pa = (TI*)I.p0;
  TI* pb = (TI*)I.p1b;
  TI* va = (TI*)I.v0;
  TI* vb = (TI*)I.v1;
  int it_s = 0;
  bool first = true;
  if (ctl() == 0) sh.bkd = 0;
  while (true) {
    {
      double acc[1] = {0.0};
      if (RC) phase_bi_p_c<K, TI, C>(I, row_lo, row_hi, r, pa, pb, va, vb, first, sh, *RC, acc);
      else phase_bi_p<K, TI, C>(I, row_lo, row_hi, r, pa, pb, va, vb, first, sh, acc);
      if (!team_reduce<K, 1, C>(acc, T, rank, e, sh, [&] { bi_alpha<K>(sh); })) return false;
    }
    {
      double acc[3] = {0.0, 0.0, 0.0};
      if (RC) phase_bi_s_c<K, TI, C>(I, row_lo, row_hi, r, vb, sh, *RC, acc);
      else phase_bi_s<K, TI, C>(I, row_lo, row_hi, r, vb, sh, acc);
      if (!team_reduce<K, 3, C>(acc, T, rank, e, sh, [&] { bi_omega<K>(sh); })) return false;
    }
    {
      double acc[2] = {0.0, 0.0};
      phase_bi_x<K, TI, C>(I, row_lo, row_hi, r, pb, sh, acc);
      it_s++;
      its++;
      if (!team_reduce<K, 2, C>(acc, T, rank, e, sh, [&] { bi_beta<K>(I, sh, it_s, its); })) return false;
    }
    if (sh.uni) break;
    first = false;
    TI* tmp = pa;
    pa = pb;
    pb = tmp;
    tmp = va;
    va = vb;
    vb = tmp;
  }
  return true;
}

// The same with the rows in the pool: x, r, r-hat, p, v, s, t of a lane stay
// in registers, and the halo's r, p, v in LDS, advanced by the owner's
// operations: v and t are exchanged (a full barrier lies between a word's last
// reader and its next write, so each has one buffer).
template <int K, typename TI, int C>
FEM_INLINE bool krylov_bicgstab_rows(const Inst& I, const Team& T, int rank, unsigned& e, TeamShared& sh, int row_lo,
                                     int row_hi, int& its, const Rows<TI>& R) {
  constexpr int RPP = kTB / K;
  const int jr = threadIdx.x % K;
  const int kv = I.kv, vj = (kv == 1) ? 0 : jr;
  const TI* rg = (const TI*)I.r;
  TI* xi = (TI*)I.xi;
  const TI GA* dinv = gp((const TI*)I.dinvi);
  const bool share = C != kPlain && T.size > 1;
  xword* xv = I.xch;                                   // v
  xword* xt = I.xch + (size_t)I.n * K * kXW<TI>;       // t
  TI LA* hv = (TI LA*)R.hv;     // staging: p, then s
  TI LA* hx = hv + R.own;       // its halo part
  TI LA* hr = hv + R.nvals;     // the halo's r (t between phases S and X), p, v
  TI LA* hp = hr + R.nx;
  TI LA* hvv = hp + R.nx;
  const int row0 = row_lo + (int)threadIdx.x / K;
  RowCells<TI> cells;
  load_cells<K>(R, row0, row_hi, cells);
  TI r[kCacheP], rh[kCacheP], p[kCacheP], v[kCacheP], s[kCacheP], t[kCacheP], x[kCacheP], d[kCacheP];
#pragma unroll
  for (int q = 0; q < kCacheP; q++) {
    r[q] = rh[q] = p[q] = v[q] = s[q] = t[q] = x[q] = d[q] = (TI)0;
    const int row = row0 + q * RPP;
    if (row >= row_hi) continue;
    const size_t o = (size_t)row * K + jr;
    r[q] = ld<C>(rg + o);
    d[q] = dinv[(size_t)row * kv + vj];
    const double xo = ld<C>(I.x + o) + (double)ld<C>(xi + o);
    st<C>(I.x + o, xo);
    rh[q] = r[q];
  }
  stage_halo<K>(R, hr - R.own, [&](size_t oc) { return ld<C>(rg + oc); });
  int it_s = 0;
  bool first = true;
  if (ctl() == 0) sh.bkd = 0;
  while (true) {
    {  // P: p = r + beta (p - omega v); v = S D^-1 p; <rh, v>
      const TI be = first ? (TI)0 : to_ti<TI>(sh.beta[jr]);
      const TI om = first ? (TI)0 : to_ti<TI>(sh.omega[jr]);
      for (int i = halo_lane<K>(); i < R.nx; i += kHaloLanes) {
        const TI pc = first ? hr[i] : (hr[i] + be * (hp[i] - om * hvv[i]));
        hp[i] = pc;
        hx[i] = pc;
      }
#pragma unroll
      for (int q = 0; q < kCacheP; q++) {
        const int row = row0 + q * RPP;
        if (row >= row_hi) continue;
        p[q] = first ? r[q] : (r[q] + be * (p[q] - om * v[q]));
        hv[(row - row_lo) * K + jr] = p[q];
      }
      __syncthreads();
      double acc[1] = {0.0};
#pragma unroll
      for (int q = 0; q < kCacheP; q++) {
        const int row = row0 + q * RPP;
        if (row >= row_hi) continue;
        v[q] = cells_gather(cells, (const TI LA*)hv, q);
        if (share) put_words<TI>(xv, (size_t)row * K + jr, v[q], e + 1);
        acc[0] += (double)rh[q] * (double)v[q];
      }
      if (!rows_reduce<K, 1, C>(acc, T, rank, e, sh, TakeHalo<K, TI>{R, xv, hvv}, [&] { bi_alpha<K>(sh); }))
        return false;
    }
    {  // S: s = r - alpha v; t = S D^-1 s; <t,s>, <t,t>, <s,s>
      const TI al = to_ti<TI>(sh.alpha[jr]);
      for (int i = halo_lane<K>(); i < R.nx; i += kHaloLanes) hx[i] = hr[i] - al * hvv[i];
#pragma unroll
      for (int q = 0; q < kCacheP; q++) {
        const int row = row0 + q * RPP;
        if (row >= row_hi) continue;
        s[q] = r[q] - al * v[q];
        hv[(row - row_lo) * K + jr] = s[q];
      }
      __syncthreads();
      double acc[3] = {0.0, 0.0, 0.0};
#pragma unroll
      for (int q = 0; q < kCacheP; q++) {
        const int row = row0 + q * RPP;
        if (row >= row_hi) continue;
        t[q] = cells_gather(cells, (const TI LA*)hv, q);
        if (share) put_words<TI>(xt, (size_t)row * K + jr, t[q], e + 1);
        acc[0] += (double)t[q] * (double)s[q];
        acc[1] += (double)t[q] * (double)t[q];
        acc[2] += (double)s[q] * (double)s[q];
      }
      if (!rows_reduce<K, 3, C>(acc, T, rank, e, sh, TakeHalo<K, TI>{R, xt, hr}, [&] { bi_omega<K>(sh); }))
        return false;
    }
    {  // X: xi += D^-1 (alpha p + omega s); r = s - omega t; <rh,r>, <r,r>
      const TI al = to_ti<TI>(sh.alpha[jr]);
      const TI om = to_ti<TI>(sh.omega[jr]);
      for (int i = halo_lane<K>(); i < R.nx; i += kHaloLanes) hr[i] = hx[i] - om * hr[i];
      double acc[2] = {0.0, 0.0};
#pragma unroll
      for (int q = 0; q < kCacheP; q++) {
        if (row0 + q * RPP >= row_hi) continue;
        x[q] = x[q] + d[q] * (al * p[q] + om * s[q]);
        r[q] = s[q] - om * t[q];
        acc[0] += (double)rh[q] * (double)r[q];
        acc[1] += (double)r[q] * (double)r[q];
      }
      it_s++;
      its++;
      if (!rows_reduce<K, 2, C>(acc, T, rank, e, sh, NoHalo{}, [&] { bi_beta<K>(I, sh, it_s, its); })) return false;
    }
    if (sh.uni) break;
    first = false;
  }
#pragma unroll
  for (int q = 0; q < kCacheP; q++) {
    const int row = row0 + q * RPP;
    if (row < row_hi) st<C>(xi + (size_t)row * K + jr, x[q]);
  }
  return true;
}

// Variants that keep the row cache: plans of multi-workgroup teams none of
// which has its rows in the pool, in the mode such teams take (they do not
// stream).
template <int KR, int C, bool ROWS>
constexpr bool row_cache() {
  return !ROWS && KR != 2 && C == kCoherent;
}

// All steps of one instance by one team.  KR: 0 pipelined CG, 1 BiCGSTAB,
// 2 classic CG (one Krylov method per kernel keeps register pressure down).
// ROWS: instances whose rows fit keep them in the pool; a plan without any
// runs the variant that leaves those paths out (with them the gathering
// phases of 16 columns spill 100 registers).
// last: the team's last instance, whose last step nothing follows.
// Returns false when the launch aborts.
template <int K, typename TI, int KR, int C, bool ROWS>
FEM_INLINE bool run_instance(const Inst& I, const Team& T, const HaloRef* halo, int rank, unsigned& e, TeamShared& sh,
                             unsigned char LA* pool, RowCache<TI>* RC, int nsteps, bool last) {
  const int n = I.n;
  const int rows_per_wg = (n + T.size - 1) / T.size;
  const int row_lo = min(n, rank * rows_per_wg);
  const int row_hi = min(n, row_lo + rows_per_wg);
  Rows<TI> R{};
  bool cached = false;
  if constexpr (ROWS) cached = fill_rows<K, TI, C>(I, T, halo, rank, row_lo, row_hi, rows_per_wg, pool, R);
  if constexpr (!row_cache<KR, C, ROWS>()) RC = nullptr;
  else if (!fill_cache<K, TI>(I, row_lo, row_hi, rows_per_wg, *RC)) RC = nullptr;
  long long its_total = 0, sweeps_total = 0;
  int status = 0;
  TI* r0 = (TI*)I.r;
  // first-order equations: the update of one step and the right-hand side of
  // the next share a phase (phase_update_rhs); have_rhs: this step's
  // right-hand side is already formed and reduced (sh.red)
  // (each barrier has one call site: inlined copies of the wait loops spill)
  const bool fuse_eq = (I.eq == EQ_HEAT || I.eq == EQ_ADVDIFF || I.eq == EQ_GS) && I.xnext && I.hpre;
  bool have_rhs = false;  // the previous step's update is pending: it runs with this step's right-hand side
  bool rhs_pre = false;   // ... and the previous step's last residual pass formed its products
  for (int step = 0; step < nsteps; step++) {
    const bool fuse_next = fuse_eq && step + 1 < nsteps;
    const int lvn = (fuse_next && I.warm) ? min(I.extrap, I.hist + step + 1) : 0;  // next step's predictor order
    // ---- R: right-hand side and initial residual (after the previous step's
    // update, in the same phase, when that was deferred)
    // the pipelined CG of the first sweep starts in the update phase (from
    // the initial residuals the last residual pass stored)
    const bool started = ROWS && KR == 0 && have_rhs && rhs_pre && cached;
    int sweeps = 0, its = 0;
    // Whether a sweep follows, and its inner threshold, are decided in the
    // control wave (one lane per column) together with the state they depend
    // on: here for the first sweep, after the last residual pass of a sweep
    // for the next.
    auto next_sweep = [&](int sweeps_done) {
      const int j = ctl();
      const bool act = j < K && sh.active[j];
      const bool go = __any(act) && sweeps_done < I.max_sweeps && its < I.max_iters;
      if (go && j < K) {
        // FP32 sweeps reduce the residual by inner_tol; an FP64 inner
        // solve goes straight to the final tolerance.
        const double rs = sh.ithr[j];
        sh.ithr[j] = (sizeof(TI) == 4) ? fmax(I.inner_tol2 * rs, sh.thr[j]) : sh.thr[j];
      }
      if (j == 0) sh.uni = go;
    };
    {
      double acc[4] = {0.0, 0.0, 0.0, 0.0};
      if (have_rhs)
        phase_update_rhs<K, TI, C, ROWS && KR == 0>(I, row_lo, row_hi, r0, sh, I.status, step - 1,
                                   I.warm ? min(I.extrap, I.hist + step) : 0, I.hvec ? lvn : 0, rhs_pre,
                                   started ? &R : nullptr, (TI*)I.q, acc);
      else
        phase_rhs<K, TI, C>(I, row_lo, row_hi, r0, step, acc);
      const bool ok = team_reduce<K, 4, C>(acc, T, rank, e, sh, [&] {
        const int j = ctl();
        if (j < K) {
          const double bb = sh.red[j], rr = sh.red[K + j], g = sh.red[2 * K + j];
          sh.bb[j] = bb;
          sh.thr[j] = fmax(I.tol2 * bb, DBL_MIN);
          const bool act = (bb != 0.0) && (rr >= sh.thr[j]);
          sh.active[j] = act;
          sh.gamma[j] = g;
          sh.ithr[j] = rr;  // residual^2 at sweep start
          sh.reset[j] = 0;
          if (started) {  // as pcg_start
            const double d = sh.red[3 * K + j];
            sh.alpha[j] = (act && d != 0.0) ? g / d : 0.0;
            sh.beta[j] = 0.0;
          }
        }
        next_sweep(0);
      });
      if (!ok) return false;
    }
    const bool hready = have_rhs && I.hvec;  // the update above formed hvec
    // the residual pass over rows in the pool: all workgroups of the team
    // agree (each publishes the candidate the others take)
    const bool want_h = fuse_next && lvn > 0;
    const bool res_rows = cached && (!want_h || hready) && R.res >= (want_h ? 2 : 1);
    // own rows only: the phases up to the next barrier read no other row's x
    if (have_rhs) phase_install<K, TI, C>(I, row_lo, row_hi);
    while (sh.uni) {
      bool ok;
      if constexpr (KR == 2) {
        ok = krylov_cg_classic<K, TI, C>(I, T, rank, e, sh, row_lo, row_hi, its);
      } else {
        auto general = [&] {
          if constexpr (KR == 1) return krylov_bicgstab<K, TI, C>(I, T, rank, e, sh, row_lo, row_hi, its, RC);
          else return krylov_pcg<K, TI, C>(I, T, rank, e, sh, row_lo, row_hi, its, RC);
        };
        if constexpr (!ROWS) ok = general();
        else if (!cached) ok = general();
        else if constexpr (KR == 1) ok = krylov_bicgstab_rows<K, TI, C>(I, T, rank, e, sh, row_lo, row_hi, its, R);
        else ok = krylov_pcg_rows<K, TI, C>(I, T, rank, e, sh, row_lo, row_hi, its, R, started && sweeps == 0);
      }
      if (!ok) return false;
      // ---- Res: FP64 residual of x + xi.  A column whose residual is not
      // finite (the sweep broke down in the inner precision) drops its
      // correction and takes the residual of x alone.
      for (int pass = 0; pass < 2; pass++) {
        double acc[2] = {0.0, 0.0};
        if (ROWS && res_rows) {
          if constexpr (ROWS)
            phase_res_rows<K, TI, C>(I, T, row_lo, row_hi, r0, sh, R, acc, lvn, fuse_next ? I.hpre : nullptr, e + 1);
        } else {
          // the sweep over rows in the pool ended without a barrier after its xi
          if (ROWS && cached && pass == 0 && !team_barrier<K, C>(T, rank, e, sh)) return false;
          phase_res<K, TI, C>(I, row_lo, row_hi, r0, sh, acc, lvn, fuse_next ? I.hpre : nullptr, hready);
        }
        const bool ok = team_reduce<K, 2, C>(acc, T, rank, e, sh, [&] {
          const int j = ctl();
          bool redo_j = false;
          if (j < K) {
            const bool bad = !(sh.red[j] <= DBL_MAX);  // NaN or infinite
            redo_j = bad && !sh.reset[j];
            sh.reset[j] = bad;
          }
          const bool redo = __any(redo_j) && pass == 0;
          if (!redo) {  // the sweep's last pass: its state, then the next sweep's decision
            if (j < K) {
              sh.reset[j] = 0;
              const double rr = sh.red[j];
              sh.active[j] = (sh.bb[j] != 0.0) && (rr >= sh.thr[j]) && (rr == rr);
              sh.gamma[j] = sh.red[K + j];
              sh.ithr[j] = rr;
            }
            next_sweep(sweeps + 1);
          }
          if (j == 0) sh.redo = redo;
        });
        if (!ok) return false;
        if (!sh.redo) break;
      }
      sweeps++;
    }
    // ---- U: state update
    int notconv = 0;
    for (int j = 0; j < K; j++) notconv |= sh.active[j];
    if (notconv) status |= ST_NOT_CONVERGED;
    if (rank == 0 && threadIdx.x < K) {
      const double bb = sh.bb[threadIdx.x];
      I.last_res[threadIdx.x] = bb > 0.0 ? sqrt(sh.ithr[threadIdx.x] / bb) : 0.0;
    }
    its_total += its;
    sweeps_total += sweeps;
    bool barrier;
    if (fuse_next) {
      // ---- U deferred: it runs with the next step's right-hand side.  With
      // no FP64 residual this step, form the history term here and share the
      // installed x before neighbours gather it.
      if (sweeps == 0 && lvn > 0) phase_hpre<K, TI, C>(I, row_lo, row_hi, lvn, hready);
      barrier = sweeps == 0 && have_rhs;
      have_rhs = true;
      rhs_pre = sweeps > 0;
    } else {
      phase_update<K, TI, C>(I, row_lo, row_hi, sh, I.status, step);
      barrier = !last || step + 1 < nsteps;  // the next step (or the team's next instance) gathers the new state
      have_rhs = false;
    }
    if (barrier && !team_barrier<K, C>(T, rank, e, sh)) return false;
  }
  if (rank == 0 && threadIdx.x == 0) {
    I.counters[0] += its_total;
    I.counters[1] += sweeps_total;
    I.counters[2] += nsteps;
    if (status) atomicOr(I.status, status);
    if (I.hist_dev) *I.hist_dev = min(4, I.hist_raw + nsteps);
  }
  return true;
}

// ---------------------------------------------------------------------------
// The kernel
// ---------------------------------------------------------------------------

template <int K, typename TI, int KR, int C, bool ROWS>
__global__ void __launch_bounds__(kTB) k_step(const Team* __restrict__ teams, const int* __restrict__ wg_team,
                                                const Inst* __restrict__ insts, const int* __restrict__ team_inst,
                                                int nsteps) {
  __shared__ TeamShared sh;
  __shared__ __attribute__((aligned(16))) unsigned char pool[ROWS ? rows_pool<C, TI>() : row_cache<KR, C, ROWS>() ? sizeof(RowCache<TI>) : 16];
  // The instance record lives in LDS while it runs: its fields are read in
  // every phase, and a global load of one would wait for every store the
  // workgroup still has in flight (loads and stores share one counter).
  __shared__ Inst sI;
  static_assert(sizeof(Inst) % sizeof(int) == 0, "Inst copied as ints");
  const int tid_team = wg_team[blockIdx.x];
  if (tid_team < 0) return;
  const Team T = teams[tid_team];
  const int l = (int)blockIdx.x - T.first_wg;
  const int rank = xcd_rank(l, T.size);
  if (threadIdx.x == 0) sh.tmo = 0;
  unsigned e = 0;  // barrier epoch, identical across the team
  for (int qi = T.inst_begin; qi < T.inst_end; qi++) {
    __syncthreads();  // the previous instance's readers are done
    const int* src = (const int*)(insts + team_inst[qi]);
    for (int w = threadIdx.x; w < (int)(sizeof(Inst) / sizeof(int)); w += kTB) ((int*)&sI)[w] = src[w];
    __syncthreads();
    // predictor history held in device memory: every workgroup of the team
    // reads it here, before the instance's first barrier; rank 0 stores the
    // new count after the last one (run_instance)
    if (threadIdx.x == 0 && sI.hist_dev) {
      const int held = *sI.hist_dev;
      sI.hist_raw = held;
      sI.hist = min(held, sI.extrap);
    }
    __syncthreads();
    if (sI.n <= 0) continue;
    if (!run_instance<K, TI, KR, C, ROWS>(sI, T, T.halo ? T.halo + qi : nullptr, rank, e, sh, (unsigned char LA*)pool,
                                              (RowCache<TI>*)pool, nsteps, qi + 1 == T.inst_end))
      return;
  }
}

// Instantiation for (columns, inner precision, Krylov method) in exchange
// mode C; no rows variant of classic CG.
template <int C, bool ROWS, int K, typename TI>
const void* pick_kr(int kr) {
  switch (kr) {
    case 0: return (const void*)k_step<K, TI, 0, C, ROWS>;
    case 1: return (const void*)k_step<K, TI, 1, C, ROWS>;
    case 2: if constexpr (!ROWS) return (const void*)k_step<K, TI, 2, C, false>; else return nullptr;
    default: return nullptr;
  }
}

template <int C, bool ROWS>
const void* pick_for_mode(int k, int fp32, int kr) {
  switch (k) {
    case 1: return fp32 ? pick_kr<C, ROWS, 1, float>(kr) : pick_kr<C, ROWS, 1, double>(kr);
    case 2: return fp32 ? pick_kr<C, ROWS, 2, float>(kr) : pick_kr<C, ROWS, 2, double>(kr);
    case 4: return fp32 ? pick_kr<C, ROWS, 4, float>(kr) : pick_kr<C, ROWS, 4, double>(kr);
    case 16: return fp32 ? pick_kr<C, ROWS, 16, float>(kr) : pick_kr<C, ROWS, 16, double>(kr);
    default: return nullptr;
  }
}

}  // namespace
}  // namespace femhip
