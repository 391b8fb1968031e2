// events.hpp -- the tree events that move state between slots, as device
// functions shared by the per-wave event kernel and the integrator's
// operation-graph mode.  Internal: not part of the C ABI.
#pragma once
#include <hip/hip_runtime.h>
#include <cstddef>

#include "../../include/gal_ode.h"
#include "../../include/gal_tree.h"
#include "physics.hpp"

namespace gal {

// State that passes between operations of a graph, on whichever XCD they run,
// is read and written at device scope (SHARED): past the XCD's own cache, so
// that handing an operation on takes a wait for the writes and no cache
// maintenance.  A release fence writes the whole cache back and an acquire
// drops it, the cooling table with it: some 14 us for each operation that ends.
template <bool SHARED, class T>
__device__ __forceinline__ T load_state_word(const T* p) {
  if constexpr (SHARED) return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else return *p;
}
template <bool SHARED, class T>
__device__ __forceinline__ void store_state_word(T* p, T v) {
  if constexpr (SHARED) __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  else *p = v;
}

// Apply one event to the state y (SoA, leading dimension ld) and the
// per-slot step sizes:
//  GAL_OP_PROMOTE: the galaxy in slot a, and its step size, move into the
//    parent's slot b (node_evolver/standard.F90:1241-1327);
//  GAL_OP_MERGE_GALAXY: satellite a merges into host b with the simple mass
//    movements (satellites/merging/mass_movements/simple.F90:208-290):
//    satellite gas and stars to the host spheroid, and in a major merger the
//    host disk joins them; the satellite's hot-halo reservoirs and black hole
//    join the host's.
// Both slots are read whole before anything is written: taken variable by
// variable, each read waited behind the write before it, some 30 trips to
// memory in a row for an event on a tree's main branch.
template <bool SHARED>
__device__ inline void apply_event(int kind, size_t a, size_t b, int ld, double* __restrict__ y,
                                   double* __restrict__ h_step, double major_ratio) {
  auto get = [&](int v, size_t s) { return load_state_word<SHARED>(y + (size_t)v * ld + s); };
  auto put = [&](int v, size_t s, double x) { store_state_word<SHARED>(y + (size_t)v * ld + s, x); };
  if (kind != GAL_OP_PROMOTE && kind != GAL_OP_MERGE_GALAXY) return;
  double ya[kNV], yb[kNV];
#pragma unroll
  for (int v = 0; v < kNV; ++v) ya[v] = get(v, a);
  if (kind == GAL_OP_PROMOTE) {
    const double h = load_state_word<SHARED>(h_step + a);
#pragma unroll
    for (int v = 0; v < kNV; ++v) put(v, b, ya[v]);
    store_state_word<SHARED>(h_step + b, h);
    return;
  }
#pragma unroll
  for (int v = 0; v < kNV; ++v) yb[v] = get(v, b);
  const double m_sat = ya[GAL_V_DISK_MASS_GAS] + ya[GAL_V_DISK_MASS_STELLAR] + ya[GAL_V_SPHEROID_MASS_GAS] +
                       ya[GAL_V_SPHEROID_MASS_STELLAR];
  const double m_host = yb[GAL_V_DISK_MASS_GAS] + yb[GAL_V_DISK_MASS_STELLAR] + yb[GAL_V_SPHEROID_MASS_GAS] +
                        yb[GAL_V_SPHEROID_MASS_STELLAR];
  const bool major = m_sat > 0.0 && m_host > 0.0 && fmin(m_sat, m_host) >= major_ratio * fmax(m_sat, m_host);
  struct Move { int from, to; };
  // satellite disk and spheroid -> host spheroid
  constexpr Move sat_moves[] = {
      {GAL_V_DISK_MASS_GAS, GAL_V_SPHEROID_MASS_GAS},
      {GAL_V_DISK_ABUNDANCES_GAS, GAL_V_SPHEROID_ABUNDANCES_GAS},
      {GAL_V_DISK_MASS_STELLAR, GAL_V_SPHEROID_MASS_STELLAR},
      {GAL_V_DISK_ABUNDANCES_STELLAR, GAL_V_SPHEROID_ABUNDANCES_STELLAR},
      {GAL_V_DISK_MASS_STELLAR_FORMED, GAL_V_SPHEROID_MASS_STELLAR_FORMED},
      {GAL_V_DISK_ANGULAR_MOMENTUM, GAL_V_SPHEROID_ANGULAR_MOMENTUM},
      {GAL_V_SPHEROID_MASS_GAS, GAL_V_SPHEROID_MASS_GAS},
      {GAL_V_SPHEROID_ABUNDANCES_GAS, GAL_V_SPHEROID_ABUNDANCES_GAS},
      {GAL_V_SPHEROID_MASS_STELLAR, GAL_V_SPHEROID_MASS_STELLAR},
      {GAL_V_SPHEROID_ABUNDANCES_STELLAR, GAL_V_SPHEROID_ABUNDANCES_STELLAR},
      {GAL_V_SPHEROID_MASS_STELLAR_FORMED, GAL_V_SPHEROID_MASS_STELLAR_FORMED},
      {GAL_V_SPHEROID_ANGULAR_MOMENTUM, GAL_V_SPHEROID_ANGULAR_MOMENTUM},
      // the satellite's circumgalactic reservoirs and black hole
      {GAL_V_HOT_MASS, GAL_V_HOT_MASS},
      {GAL_V_HOT_ABUNDANCES, GAL_V_HOT_ABUNDANCES},
      {GAL_V_HOT_ANGULAR_MOMENTUM, GAL_V_HOT_ANGULAR_MOMENTUM},
      {GAL_V_HOT_OUTFLOWED_MASS, GAL_V_HOT_OUTFLOWED_MASS},
      {GAL_V_HOT_OUTFLOWED_ANGULAR_MOMENTUM, GAL_V_HOT_OUTFLOWED_ANGULAR_MOMENTUM},
      {GAL_V_HOT_OUTFLOWED_ABUNDANCES, GAL_V_HOT_OUTFLOWED_ABUNDANCES},
      {GAL_V_HOT_UNACCRETED_MASS, GAL_V_HOT_UNACCRETED_MASS},
      {GAL_V_HOT_UNACCRETED_ABUNDANCES, GAL_V_HOT_UNACCRETED_ABUNDANCES},
      {GAL_V_HOT_ENERGY_RADIATED, GAL_V_HOT_ENERGY_RADIATED},
      {GAL_V_BH_MASS, GAL_V_BH_MASS},
  };
#pragma unroll
  for (const Move& m : sat_moves) {
    yb[m.to] += ya[m.from];
    ya[m.from] = 0.0;
  }
  // the satellite's stripped gas joins the host's outflowed reservoir, as
  // hot_halo/standard/_class.F90:532-597 moves it after each satellite
  // evolve (here at the merger: mass and metals; its angular momentum,
  // M_stripped J_host/M_host there, is not carried)
  yb[GAL_V_HOT_OUTFLOWED_MASS] += ya[GAL_V_HOT_STRIPPED_MASS];
  ya[GAL_V_HOT_STRIPPED_MASS] = 0.0;
  yb[GAL_V_HOT_OUTFLOWED_ABUNDANCES] += ya[GAL_V_HOT_STRIPPED_ABUNDANCES];
  ya[GAL_V_HOT_STRIPPED_ABUNDANCES] = 0.0;
  constexpr Move host_moves[] = {
      {GAL_V_DISK_MASS_GAS, GAL_V_SPHEROID_MASS_GAS},
      {GAL_V_DISK_ABUNDANCES_GAS, GAL_V_SPHEROID_ABUNDANCES_GAS},
      {GAL_V_DISK_MASS_STELLAR, GAL_V_SPHEROID_MASS_STELLAR},
      {GAL_V_DISK_ABUNDANCES_STELLAR, GAL_V_SPHEROID_ABUNDANCES_STELLAR},
      {GAL_V_DISK_MASS_STELLAR_FORMED, GAL_V_SPHEROID_MASS_STELLAR_FORMED},
      {GAL_V_DISK_ANGULAR_MOMENTUM, GAL_V_SPHEROID_ANGULAR_MOMENTUM},
  };
  if (major) {
#pragma unroll
    for (const Move& m : host_moves) {
      yb[m.to] += yb[m.from];
      yb[m.from] = 0.0;
    }
  }
  // what changed: the moves' ends, and the disk of a host in a major merger
#pragma unroll
  for (const Move& m : sat_moves) {
    put(m.from, a, ya[m.from]);
    put(m.to, b, yb[m.to]);
  }
  put(GAL_V_HOT_STRIPPED_MASS, a, ya[GAL_V_HOT_STRIPPED_MASS]);
  put(GAL_V_HOT_STRIPPED_ABUNDANCES, a, ya[GAL_V_HOT_STRIPPED_ABUNDANCES]);
  if (major) {
#pragma unroll
    for (const Move& m : host_moves) put(m.from, b, yb[m.from]);
  }
}

// A forest's operations as a dependency graph for one persistent launch of
// the integrator.  ops is the device copy of the schedule's operations,
// indexed as in the schedule; the graph holds n of them (becoming a
// satellite changes no state and is left out).  Operation k touches slot
// ops[k].a (and ops[k].b for events); it waits on the previous operation on
// each slot it touches, and next_a[k], next_b[k] are the operations that
// follow it on those slots (-1: none).  npred[k] counts the links still
// unfinished.  The lane that counts an operation to zero runs it next itself,
// with no way through the list and no wait for another lane to look there;
// where it makes two ready, the second is appended to ready[], from which idle
// lanes claim entries in order.  tail[0] counts the appends and tail[1] the
// chained operations: each operation is one or the other, so the list ends at
// n - tail[1] when all are done.  Entries not yet written hold -1.
struct OpGraph {
  int n = 0;                               // operations in the graph
  const gal_schedule_op* ops = nullptr;    // the schedule's operations (device)
  const int* next_a = nullptr;
  const int* next_b = nullptr;
  int* npred = nullptr;
  int* ready = nullptr;
  unsigned int* tail = nullptr;            // two counts, 8-byte aligned
  double major_ratio = 0.25;
};

__device__ __forceinline__ int graph_ready_entry(const OpGraph& g, int j) {
  return __hip_atomic_load(&g.ready[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Appended and chained operations so far, in one word.
__device__ __forceinline__ unsigned long long graph_progress(const OpGraph& g) {
  return __hip_atomic_load((const unsigned long long*)g.tail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Every store this wave has issued has reached the device's memory.
__device__ __forceinline__ void stores_done() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_waitcnt(0);
}

// Operation k has finished and its writes are done: count it off its
// successors na and nb (-1: none).  A successor counted to zero is run next by
// the lane that did so: it is returned, and never enters the ready list.  With
// two of them the second is appended to the list.
__device__ inline int graph_release(const OpGraph& g, int k, int na, int nb) {
  // both at once, one that is missing as an addition of 0 to the operation's
  // own count
  const int left_a = __hip_atomic_fetch_add(&g.npred[na < 0 ? k : na], na < 0 ? 0 : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int left_b = __hip_atomic_fetch_add(&g.npred[nb < 0 ? k : nb], nb < 0 ? 0 : -1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const bool ready_a = na >= 0 && left_a == 1, ready_b = nb >= 0 && left_b == 1;
  if (ready_a && ready_b) {
    const unsigned int pos = __hip_atomic_fetch_add(g.tail, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (pos < (unsigned int)g.n) __hip_atomic_store(&g.ready[pos], nb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (ready_a || ready_b) (void)__hip_atomic_fetch_add(g.tail + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  return ready_a ? na : (ready_b ? nb : -1);
}

}  // namespace gal
