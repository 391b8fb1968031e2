// gal_ode.hip -- batched node-ODE evolution on MI355X (gfx950) and its C ABI.
//
// A group of 64 nodes is served by one workgroup of four waves, one wave on
// each SIMD of a CU and one lane position per node.  A persistent grid of
// groups claims nodes from a global counter (one atomic per refill) and
// integrates each from t_start to t_end with the Cash-Karp (4,5) pair, the
// scaled error norm and step controller, the driver loop and the node-evolver
// trial loop of the reference:
//   trial loop    node_evolver/standard.F90:587-740
//   solve         numerical/ODE_solver/solver.F90:492-691
//   driver        external/gslODEInitVal2/driver2.c:148-250
//   evolve/step   GSL 2.6 gsl_odeiv2_evolve_apply + rkck (published method)
//   controller    external/gslODEInitVal2/cscal2.c:93-169
// When a lane's node finishes it claims the next one, so lanes stay busy
// while step counts differ by two orders of magnitude between nodes.
//
// Schedule.  The lanes of a group advance in lockstep, one Cash-Karp attempt
// per trip: the derivative at (t, y) -- dydt at the new point (the reference's
// dydt_out, reused as the next k1), k1 of a freshly claimed node, or k1 after a
// trial restart -- then the five stages of k2..k6, the solution, its error norm
// and the controller.  Every lane spends six RHS evaluations per trip whatever
// it is doing, and the RHS never diverges by stage.
//
// Memory.  State is structure-of-arrays in HBM (y[v*ld + i]); it is read once
// when a node is claimed and written once when it finishes.  In between the
// integrator's state is in registers and in the group's LDS (see group_wave).
#include <hip/hip_runtime.h>
#include <cstddef>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <cmath>
#include <algorithm>
#include <mutex>

#include "../../include/gal_ode.h"
#include "../../include/gal_tree.h"
#include "constants.hpp"
#include "physics.hpp"
#include "integrator.hpp"
#include "batch.hpp"
#include "events.hpp"
#include "group_rhs.hpp"

#include <hipcub/device/device_radix_sort.hpp>

using namespace gal;

namespace {

struct EvolveArgs {
  int n, ld;
  int n_claim;  // claims are limited to n_claim entries of order[] (n when order is null)
  const int* n_claim_dev;  // if set, the limit is read from device memory instead
  double* y;
  const double* np;
  const double* t_start;
  const double* t_end;
  double* h_step;
  double* scale;
  int* status;
  long long* counters;
  const int* order;
  unsigned int* work;
  const double* P;
  const double* tab;
  DerivedConstants D;
  CoolingDesc cd;
  double eps_abs, eps_rel;
  int flags, mode;
  // Wall-time limit of the launch in ticks of the GPU's constant-rate
  // realtime counter (0: none).  An attempt that would start after it
  // returns the node with errorStatusXCPU and its state untouched.
  unsigned long long wall_ticks;
  // Operation-graph mode (kernel parameter GRAPH): lanes claim entries of
  // the graph's ready list (a.work counts the claims) instead of nodes.  A
  // lane whose claimed entry stays unwritten while no operation is appended
  // for stall_ticks gives up, sets *graph_error and leaves, so that a
  // malformed graph ends the launch instead of holding it.
  OpGraph g;
  int* graph_error;
  unsigned long long stall_ticks;
};

// An index the compiler computes addresses from but does not fold.
__device__ __forceinline__ int opaque(int index) {
  asm volatile("" : "+v"(index));
  return index;
}

// Claim one node index per requesting lane with a single atomic per wave.
__device__ __forceinline__ int wave_claim(bool want, unsigned int* work, int n, const int* order) {
  const unsigned long long mask = __ballot(want);
  int idx = -1;
  if (mask) {
    const int lane = __lane_id();
    const int leader = __ffsll((long long)mask) - 1;
    const int cnt = __popcll(mask);
    unsigned int base = 0;
    if (lane == leader) base = atomicAdd(work, (unsigned int)cnt);
    base = __shfl(base, leader);
    const unsigned long long below = lane ? (mask & ((1ull << lane) - 1ull)) : 0ull;
    const unsigned int mine = base + (unsigned int)__popcll(below);
    if (want && mine < (unsigned int)n) idx = order ? order[mine] : (int)mine;
  }
  return idx;
}

template <bool SHARED>
__device__ __forceinline__ void write_counters(const EvolveArgs& a, int node, long long na, long long nc,
                                               long long nr) {
  if (a.counters) {
    store_state_word<SHARED>(a.counters + node, na);
    store_state_word<SHARED>(a.counters + (size_t)a.n + node, nc);
    store_state_word<SHARED>(a.counters + 2 * (size_t)a.n + node, nr);
  }
}

// What a lane of the cooling wave keeps about the node it claimed last.
struct ClaimState {
  // graph mode: the operation in hand and its successors, the one to run after
  // it, and the claimed entry of the ready list with what it last read
  int op = -1, next_a = -1, next_b = -1, next = -1, pend = -1, peek = -1;
  unsigned long long wait_progress = ~0ull;   // progress seen while waiting on the entry
  unsigned long long wait_since = 0ull;
};
// Claims, then the rounds of an attempt: the time part alone (new nodes), the derivative at its
// start, then the stages 0-4 that give k2-k6.
enum : int { kClaims = -3, kTimeOnly = -2, kFirst = -1, kLast = 4 };
// By stage 0-3: the next stage's time.
__constant__ const double kNextTime[kLast] = {ck::a3, ck::a4, ck::a5, ck::a6};
// What steers a lane, as bits of one register: booleans of their own cost three
// scalar instructions each wherever two paths of the round meet.
struct LaneFlags {
  enum : unsigned {
    kActive = 1u,        // has a node
    kWant = 2u,          // wants one
    kEval = 4u,          // the coming derivative is one it needs
    kPost = 8u,          // an accepted state awaits the post-step fixes
    kDecide = 16u,       // an attempt awaits the controller
    kFinalStep = 32u,    // its step ends the interval
    kFetch = 64u,        // its state is to be loaded
    kFresh = 128u,       // its node was claimed just now
    kStepping = 256u,    // in an attempt
    kForbidden = 512u,   // the attempt's state is negative where it may not be
    kNeedFix = 1024u     // and where the post-step fixes apply
  };
  unsigned bits;
  __device__ __forceinline__ bool has(unsigned f) const { return (bits & f) != 0u; }
  __device__ __forceinline__ void set(unsigned f) { bits |= f; }
  __device__ __forceinline__ void clear(unsigned f) { bits &= ~f; }
};
enum : int { kNoClaim = -1, kExhausted = -2 };   // codes of the claim vector beside a node index

// Claim a node's interval for each lane that wants one (cooling wave) and
// publish it, or why there is none, in the claim vectors of the exchange
// area.
template <bool GRAPH>
__device__ __forceinline__ void claim_nodes(const EvolveArgs& a, int n_claim, bool want, bool idle, ClaimState& c,
                                            double* __restrict__ C) {
  auto publish = [&](int node, double t0, double t1, const double* np, size_t stride) {
    C[kXClaimNode * kGroupNodes] = (double)node;
    C[kXClaimT0 * kGroupNodes] = t0;
    C[kXClaimT1 * kGroupNodes] = t1;
    C[kXClaimStep * kGroupNodes] = load_state_word<GRAPH>(a.h_step + node);
#pragma unroll
    for (int k = 0; k < GAL_NPARAM_NODE; ++k) C[(kXClaimPar + k) * kGroupNodes] = np[k * stride];
  };
  C[kXClaimNode * kGroupNodes] = (double)kNoClaim;
  if constexpr (GRAPH) {
    // The operation that the lane's last one made ready, else a claimed entry
    // of the ready list once it is written; events are applied on the spot.
    // An entry is looked at here only by a group with nothing else to do: one
    // with nodes under way read it during its last evaluation.
    if (idle && c.pend >= 0) c.peek = graph_ready_entry(a.g, c.pend);
    bool again = true;
    while (again) {
      const bool need = want && c.pend < 0 && c.next < 0;
      if (__any(need)) {
        const int j = wave_claim(need, a.work, a.g.n, nullptr);
        if (need) {
          if (j < 0) {
            want = false;
            C[kXClaimNode * kGroupNodes] = (double)kExhausted;
          } else {
            c.pend = j;
            c.peek = graph_ready_entry(a.g, j);
            c.wait_progress = ~0ull;
          }
        }
      }
      if (want) {
        int k = c.next;
        c.next = -1;
        if (k < 0 && c.pend >= 0 && c.peek >= 0) {
          k = c.peek;
          c.pend = c.peek = -1;
        }
        if (k >= 0) {
          const gal_schedule_op* o = a.g.ops + k;
          const int kind = o->kind;
          c.next_a = a.g.next_a[k];
          c.next_b = a.g.next_b[k];
          if (kind != GAL_OP_EVOLVE) {
            apply_event<true>(kind, (size_t)o->a, (size_t)o->b, a.ld, a.y, a.h_step, a.g.major_ratio);
            stores_done();
            c.next = graph_release(a.g, k, c.next_a, c.next_b);
          } else {
            c.op = k;
            publish(o->a, o->t0, o->t1, o->node_par, 1);
            want = false;
          }
        } else if (idle) {
          const unsigned long long progress = graph_progress(a.g);
          const unsigned long long now = wall_clock64();
          // the list ends at what is never chained past it
          bool over = c.pend >= a.g.n - (int)(progress >> 32);
          if (progress != c.wait_progress) {
            c.wait_progress = progress;
            c.wait_since = now;
          } else if (now - c.wait_since > a.stall_ticks) {
            __hip_atomic_store(a.graph_error, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            over = true;
          }
          if (over) {
            want = false;
            c.pend = c.peek = -1;
            C[kXClaimNode * kGroupNodes] = (double)kExhausted;
          }
        }
      }
      again = __any(want && c.pend < 0);
    }
  } else {
    // an order entry outside the batch (a plan the caller did not let finish)
    // ends this lane's claims instead of addressing past it
    const int claimed = wave_claim(want, a.work, n_claim, a.order);
    if (want) {
      if (claimed < 0 || claimed >= a.n) C[kXClaimNode * kGroupNodes] = (double)kExhausted;
      else publish(claimed, a.t_start[claimed], a.t_end[claimed], a.np + claimed, (size_t)a.ld);
    }
  }
}

// Persistent integrator: a workgroup of four waves serves 64 nodes, one per
// lane position, and group_rhs.hpp deals the RHS out over the waves.  The
// integrator's state is split by variable: wave w (of the first three) owns
// variables [10 w, 10 w + 10) of every node -- state, stage derivatives and
// error scales -- and forms their stage inputs, solution and error norm.  What
// steers a node (times, step size, trial, flags) is held by all four waves
// alike: each runs the same code on the same published values, so they agree
// without a message.  The cooling wave owns no variables and does what needs
// one wave: claims, statuses, counters, the wall clock.
//
// The step controller's pow is not on the path: whether a step is accepted
// follows from the error norm alone, and the derivative at the new point does
// not depend on the step size, so the time wave computes the next step size
// during that evaluation (which also decides a step-size underflow).
//
// One instance of this per wave of the group: a lone wave issues one
// instruction every 4.6 cycles whatever it is (a dependent FP64 FMA costs no
// more than an independent one, and a move of half a constant as much as
// either), so what there is to save is instructions on the chain that crosses
// the waves.  An attempt's six evaluations are some 14.6 of its 18.7 us; the
// rest is between them, where each owner forms ten variables one by one.
// With a loop of its own a wave keeps the constants of its own transcendental
// functions in registers across the integration.  Between two evaluations
// every value that is carried round the loop and set on more than one path
// costs a move on each: the state at the start of the step is therefore kept
// in LDS, a lane's booleans share one register, and there is one loop with one
// evaluation in it and one exit.
//
// Measured on the stiffest node of 100,000 isolated halos (3701 attempts): 18.7
// us an attempt, 22.6 us with the state in registers and nested loops, and 43
// us with one wave for the whole RHS, or two waves that split it in halves.
//
template <int WAVE, bool GRAPH>
__device__ __forceinline__ void group_wave(const EvolveArgs& a, double* __restrict__ X,
                                           const GroupConstants& constants, int* __restrict__ norm_flags,
                                           int* __restrict__ flags, int& wall_expired) {
  // in registers for the whole integration, as far as this wave uses them
  const GroupConstants G = constants;
  constexpr int wave = WAVE;
  constexpr bool owner = wave < kOwnerWaves;
  constexpr int v0 = owner ? wave * kOwned : 0;    // first owned variable
  const int lane = threadIdx.x & (kGroupNodes - 1);
  double* __restrict__ XY = X + (kXState + v0) * kGroupNodes;   // owned rows (owners only)
  double* __restrict__ XG = X + (kXGalaxy + v0) * kGroupNodes;
  double* __restrict__ XH = X + (kXHalo + v0) * kGroupNodes;
  // bases of their own: an offset past 64 KiB would cost an addition per access
  double* __restrict__ XK = X + opaque((kXStage + v0) * kGroupNodes);
  double* __restrict__ X0 = X + opaque((kXStart + v0) * kGroupNodes);
  double* __restrict__ F = X + opaque(kXFar * kGroupNodes);
  auto time_vectors = [&](int which) { return F + (kFarTime + which * kTimeVectors) * kGroupNodes; };
  const int mode = a.mode;
  const int ops = mode == GAL_PHYSICS_STANDARD ? (int)a.P[GAL_P_OPERATORS] : 0;
  const bool reuse = (a.flags & GAL_FLAG_REUSE_STEP_SIZE) != 0;
  const bool enforce = (a.flags & GAL_FLAG_ENFORCE_NON_NEGATIVITY) != 0;
  const bool scales_given = (a.flags & GAL_FLAG_SCALES_PROVIDED) != 0;
  // owned variables that may not be negative, and those the post-step fixes
  constexpr unsigned nonneg = kNonNegative >> v0;
  const bool galaxy_fix = a.P[GAL_P_POST_STEP_ZERO_NEGATIVE_MASSES] != 0.0;
  const unsigned fixable =
      (mode == GAL_PHYSICS_TEST ? 0u : kPostStepHalo | (galaxy_fix ? kPostStepGalaxy : 0u)) >> v0;

  // steering, alike in all four waves
  NodePar np{};
  int node = -1, trial = 0;
  LaneFlags s{LaneFlags::kWant};
  double t = 0.0, t0 = 0.0, t1 = 0.0, h = 0.0, h0 = 0.0, h_node = 0.0, sign = 1.0;
  double rmax = 0.0;       // error norm of the attempt
  bool time_stale = false;
  int round = 0;
  int tb = 0;              // which time part is the coming stage's
  // owners
  double abs_tol[kOwned];    // absolute tolerance times the error scale
#pragma unroll
  for (int i = 0; i < kOwned; ++i) abs_tol[i] = 0.0;
  // derivative of a stage, and the state at the start of the step
  auto K = [&](int stage, int i) -> double& { return XK[((stage == 4 ? 1 : stage) * kNV + i) * kGroupNodes]; };
  auto Y0 = [&](int i) -> double& { return X0[i * kGroupNodes]; };
  // cooling wave
  ClaimState claim;
  long long n_attempt = 0, n_accept = 0, n_rhs = 0;
  const int n_claim = a.n_claim_dev ? *a.n_claim_dev : a.n_claim;
  const unsigned long long t_launch = a.wall_ticks ? wall_clock64() : 0ull;

  // The first step of a trial (solver.F90:537-555)
  auto start_trial = [&](double step_size) {
    double xs = t1 - t0;
    if (step_size > 0.0) xs = fmin(step_size, xs);
    h = xs;
    h0 = xs;
    t = t0;
    s.set(LaneFlags::kEval);
  };
  // Results of a lane's interval (cooling wave); its state is stored by the
  // owners beforehand, and in graph mode its successors are released.
  auto finish = [&](bool done, double h_out, bool write_h, int status) {
    if (wave == kCoolingWave && done) {
      if (write_h) store_state_word<GRAPH>(a.h_step + node, h_out);
      store_state_word<GRAPH>(a.status + node, status);
      write_counters<GRAPH>(a, node, n_attempt, n_accept, n_rhs);
    }
    if constexpr (GRAPH) {
      stores_done();
      __syncthreads();
      if (wave == kCoolingWave && done) claim.next = graph_release(a.g, claim.op, claim.next_a, claim.next_b);
    }
    if (done) {
      s.clear(LaneFlags::kActive);
      s.set(LaneFlags::kWant);
    }
  };
  // The reference's negative-value fixes on the published state of the given
  // lanes (rare): one wave fixes, the owners take their variables back.
  auto fix_published = [&](bool lanes, auto&& take) {
    if (wave == kCoolingWave && lanes) post_step(constants.P, constants.D, np, mode, t, X + kXState * kGroupNodes, kGroupNodes);
    __syncthreads();
    if (owner && lanes) {
#pragma unroll
      for (int i = 0; i < kOwned; ++i) take(i, XY[i * kGroupNodes]);
    }
  };

  auto norm = [&]() {
    ErrorNorm e;
    e.rmax = rmax;
    e.forbidden = s.has(LaneFlags::kForbidden);
    return e;
  };
  // The sums over the older stage derivatives, formed beside the RHS; each is
  // completed once the newest derivative is known, with its coefficient bn.
  auto older_terms = [&](int ph, double (&y)[kOwned], double (&sp)[kOwned], double& bn) {
    if constexpr (owner) {
#pragma clang fp contract(off)
      bn = 0.0;
#pragma unroll
      for (int i = 0; i < kOwned; ++i) y[i] = Y0(i);
      if (ph == 0) {
        bn = ck::b32;
#pragma unroll
        for (int i = 0; i < kOwned; ++i) sp[i] = ck::b31 * K(0, i);
      } else if (ph == 1) {
        bn = ck::b43;
#pragma unroll
        for (int i = 0; i < kOwned; ++i) sp[i] = fma(ck::b41, K(0, i), ck::b42 * K(1, i));
      } else if (ph == 2) {
        bn = ck::b54;
#pragma unroll
        for (int i = 0; i < kOwned; ++i) sp[i] = fma(ck::b53, K(2, i), fma(ck::b52, K(1, i), ck::b51 * K(0, i)));
      } else if (ph == 3) {
        bn = ck::b65;
#pragma unroll
        for (int i = 0; i < kOwned; ++i)
          sp[i] = fma(ck::b64, K(3, i), fma(ck::b63, K(2, i), fma(ck::b61, K(0, i), ck::b62 * K(1, i))));
      } else if (ph == kLast) {
#pragma unroll
        for (int i = 0; i < kOwned; ++i) sp[i] = fma(ck::c4, K(3, i), fma(ck::c1, K(0, i), ck::c3 * K(2, i)));
      } else {
        // not used, and set so that nothing is carried from round to round
#pragma unroll
        for (int i = 0; i < kOwned; ++i) sp[i] = 0.0;
      }
    }
  };

  // One RHS evaluation per trip.  What follows an evaluation of the stages 0-3,
  // four of an attempt's six, touches none of the steering; everything rarer
  // sits in branches that leave the state in the registers where it was.
  int ph = kClaims;
  for (;;) {
    if (ph == kClaims) {
      // ---- claims, and the state the next derivative is taken at -------------
      bool begun = false;
      while (__any(s.has(LaneFlags::kWant))) {
        double* C = time_vectors(tb ^ 1);
        if (wave == kCoolingWave) claim_nodes<GRAPH>(a, n_claim, s.has(LaneFlags::kWant), !__any(s.has(LaneFlags::kActive)), claim, C);
        __syncthreads();
        const int code = (int)C[kXClaimNode * kGroupNodes];
        begun = s.has(LaneFlags::kWant) && code >= 0;
        if (code == kExhausted) s.clear(LaneFlags::kWant);
        if (begun) {
          node = code;
          t0 = C[kXClaimT0 * kGroupNodes];
          t1 = C[kXClaimT1 * kGroupNodes];
          h_node = C[kXClaimStep * kGroupNodes];
          np = load_node_par(C + kXClaimPar * kGroupNodes, kGroupNodes, 0);
          s = LaneFlags{LaneFlags::kActive | LaneFlags::kFetch | LaneFlags::kFresh};
          trial = 0;
          n_attempt = n_accept = n_rhs = 0;
          start_trial(reuse ? h_node : -1.0);
          sign = h > 0.0 ? 1.0 : -1.0;
          if (t0 == t1) s.clear(LaneFlags::kEval);
          if (owner && scales_given) {
#pragma unroll
            for (int i = 0; i < kOwned; ++i) abs_tol[i] = a.eps_abs * a.scale[(size_t)(v0 + i) * a.ld + node];
          }
        }
        if (__any(s.has(LaneFlags::kActive))) break;
        __syncthreads();   // the claim vectors are free again
        // graph mode: lanes wait on ready-list entries; poll again after a pause
        if (__any(s.has(LaneFlags::kWant))) __builtin_amdgcn_s_sleep(8);
      }
      if (!__any(s.has(LaneFlags::kActive))) break;
      if (owner && s.has(LaneFlags::kFetch)) {
#pragma unroll
        for (int i = 0; i < kOwned; ++i) XY[i * kGroupNodes] = Y0(i) = load_state_word<GRAPH>(a.y + (size_t)(v0 + i) * a.ld + node);
      }
      s.clear(LaneFlags::kFetch);
      // The time part of the derivative was computed ahead for lanes that go
      // on; for new ones an extra round computes it (all lanes; the others'
      // comes out as it was).
      ph = time_stale || __any(begun) ? kTimeOnly : kFirst;
      time_stale = false;
    }
    ++round;
    __syncthreads();   // stage state and time part published
    if (ph == kFirst && !scales_given && owner && __any(s.has(LaneFlags::kFresh))) {
      double ys[kNV], s30[kNV];
      load_state(X, ys);
      const TimePart T = load_time_part(time_vectors(tb));
      scales_of_halo(G.P, G.D, T.mass, T.r_vir, T.v_vir, galaxy_radius(T, ys[GAL_V_SPIN_ANGULAR_MOMENTUM]).r, ys, s30);
      if (s.has(LaneFlags::kFresh)) {
#pragma unroll
        for (int i = 0; i < kOwned; ++i) {
          const double sc = mode == GAL_PHYSICS_TEST ? 1.0 : rounded(s30[v0 + i]);
          abs_tol[i] = a.eps_abs * sc;
          if (a.scale) store_state_word<GRAPH>(a.scale + (size_t)(v0 + i) * a.ld + node, sc);
        }
      }
    }
    double y[kOwned], sp[kOwned], bn;
    if constexpr (wave == kTimeWave) {
      older_terms(ph, y, sp, bn);   // its own work waits for nobody, so these come first
      // the time of the next stage, or after the last one of the point that
      // the step leads to if it is accepted
      double tn = t;
      if (ph == kFirst) {
        const double hn = s.has(LaneFlags::kDecide) ? hadjust_step(norm(), kRkckOrder, h0) : h0;
        F[kFarStep * kGroupNodes] = hn;
        const double dt = t1 - t;
        const double hs = ((dt >= 0.0 && hn > dt) || (dt < 0.0 && hn < dt)) ? dt : hn;
        tn = t + ck::a2 * hs;
      } else if (ph == kLast) {
        if (!s.has(LaneFlags::kEval)) tn = s.has(LaneFlags::kFinalStep) ? t1 : t + h0;
      } else if (ph != kTimeOnly) {
        tn = t + kNextTime[ph] * h0;
      }
      store_time_part(time_part(G.P, G.D, G.C, np, tn), time_vectors(tb ^ 1));
      if (ph != kTimeOnly && mode == GAL_PHYSICS_STANDARD) time_wave_rhs(X, F, flags, round);
    } else if (ph != kTimeOnly) {
      if constexpr (wave == kGalaxyWave) {
        galaxy_wave_rhs(G, mode, ops, np, X, F, time_vectors(tb), flags, round);
      } else if (mode == GAL_PHYSICS_STANDARD) {
        if constexpr (wave == kProfileWave) profile_wave_rhs(G, ops, X, F, time_vectors(tb), flags, round);
        if constexpr (wave == kCoolingWave) cooling_wave_rhs(G, a.tab, np, X, F, time_vectors(tb), flags, round);
      }
      if constexpr (wave == kCoolingWave) {
        if (GRAPH && ph == kLast) claim.peek = graph_ready_entry(a.g, claim.pend >= 0 ? claim.pend : 0);
        if (ph == kFirst && a.wall_ticks && lane == 0) wall_expired = wall_clock64() - t_launch > a.wall_ticks;
      }
    }
    if constexpr (wave != kTimeWave) older_terms(ph, y, sp, bn);
    __syncthreads();   // derivatives published
    tb ^= 1;
    double kn[kOwned];
    if (owner) {
      // all reads in flight before the first sum; a half that has no part of a
      // variable's derivative is not read
      double fh[kOwned];
#pragma unroll
      for (int i = 0; i < kOwned; ++i) kn[i] = (kGalaxyVars >> (v0 + i)) & 1u ? XG[i * kGroupNodes] : 0.0;
#pragma unroll
      for (int i = 0; i < kOwned; ++i) fh[i] = (kHaloVars >> (v0 + i)) & 1u ? XH[i * kGroupNodes] : 0.0;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < kOwned; ++i) {
        if (!((kGalaxyVars >> (v0 + i)) & 1u)) kn[i] = fh[i];
        else if ((kHaloVars >> (v0 + i)) & 1u) kn[i] += fh[i];
      }
    }
    if (ph >= 0 && ph < kLast) {
      // the next stage's input y + h (older terms + newest)
      if (owner) {
#pragma clang fp contract(off)
#pragma unroll
        for (int i = 0; i < kOwned; ++i) XY[i * kGroupNodes] = fma(h0, fma(bn, kn[i], sp[i]), y[i]);
#pragma unroll
        for (int i = 0; i < kOwned; ++i) K(ph + 1, i) = kn[i];
      }
      ++ph;
    } else if (ph == kTimeOnly) {
      ph = kFirst;
    } else if (ph == kFirst) {
      const bool evaluated = s.has(LaneFlags::kEval), zero_length = s.has(LaneFlags::kFresh) && !evaluated;
      if (owner && evaluated) {
#pragma unroll
        for (int i = 0; i < kOwned; ++i) K(0, i) = kn[i];
      }
      if (wave == kCoolingWave && evaluated) ++n_rhs;
      // GSL_CONTINUE: the post-step fixes leave the derivative as it is
      const bool fix = s.has(LaneFlags::kPost) && s.has(LaneFlags::kNeedFix);
      if (__any(fix)) fix_published(fix, [&](int i, double v) { Y0(i) = v; });
      const double hn = F[kFarStep * kGroupNodes];
      bool failed = false;
      if (s.has(LaneFlags::kDecide)) {
        if (hadjust_kind(norm()) == kHadjDec) {
          const double t_adv = s.has(LaneFlags::kFinalStep) ? t1 : t + h0;
          if (fabs(hn) < fabs(h0) && t_adv + hn != t_adv) h0 = hn;   // rejected: retry, same k1
          else failed = true;                                         // step size underflow
        } else {
          h = hn;
          h0 = hn;
        }
      }
      s.clear(LaneFlags::kEval | LaneFlags::kPost | LaneFlags::kFresh | LaneFlags::kDecide | LaneFlags::kStepping |
              LaneFlags::kFinalStep);
      // nothing to integrate (standard.F90:580): success, timeStep -1
      if (__any(zero_length)) finish(zero_length, -1.0, true, GAL_STATUS_SUCCESS);
      if (__any(failed)) {
        // node-evolver trial loop (standard.F90:657-692)
        bool rescued = false;
        if (enforce) {
          if (owner) {
            bool any = false;
#pragma unroll
            for (int i = 0; i < kOwned; ++i) any |= Y0(i) < 0.0 && ((nonneg >> i) & 1u);
            norm_flags[wave * kGroupNodes + lane] = any ? 4 : 0;
          }
          __syncthreads();
#pragma unroll
          for (int w = 0; w < kOwnerWaves; ++w) rescued |= (norm_flags[w * kGroupNodes + lane] & 4) != 0;
          rescued = rescued && failed;
          if (owner && rescued) {
#pragma unroll
            for (int i = 0; i < kOwned; ++i)
              store_state_word<GRAPH>(a.y + (size_t)(v0 + i) * a.ld + node,
                                      Y0(i) < 0.0 && ((nonneg >> i) & 1u) ? 0.0 : Y0(i));
          }
          if (__any(rescued)) finish(rescued, h_node / (double)(1 << trial), true, GAL_STATUS_SUCCESS);
        }
        const bool retry = failed && !rescued;
        bool spent = false;
        if (retry) {
          spent = ++trial >= 8;
          if (!spent) {
            s.set(LaneFlags::kFetch);
            start_trial(reuse ? h_node / (double)(1 << trial) : -1.0);
          }
        }
        // all trials failed: state restored, errorStatusUnderflow (standard.F90:715-718)
        if (__any(spent)) finish(spent, 0.0, false, GAL_STATUS_UNDERFLOW);
      }
      // Wall-time limit (node_evolver/standard.F90:693-705 and the RHS's own
      // check, standard.F90:860-866): the nodes return errorStatusXCPU with
      // their state as it came in.
      if (a.wall_ticks && wall_expired && __any(s.has(LaneFlags::kActive))) {
        finish(s.has(LaneFlags::kActive), 0.0, false, GAL_STATUS_XCPU);
        s.clear(LaneFlags::kEval | LaneFlags::kFetch);
      }
      const bool stepping = s.has(LaneFlags::kActive) && !s.has(LaneFlags::kEval);
      if (__any(stepping)) {
        // gsl_odeiv2_evolve_apply: clip the step to reach t1 exactly
        const double dt = t1 - t;
        if (stepping) {
          s.set(LaneFlags::kStepping);
          if ((dt >= 0.0 && h0 > dt) || (dt < 0.0 && h0 < dt)) {
            h0 = dt;
            s.set(LaneFlags::kFinalStep);
          }
          if (wave == kCoolingWave) {
            ++n_attempt;
            n_rhs += 5;
          }
        }
        if (owner) {
#pragma clang fp contract(off)
#pragma unroll
          for (int i = 0; i < kOwned; ++i) XY[i * kGroupNodes] = fma(h0, ck::b21 * K(0, i), Y0(i));
        }
        ph = 0;
      } else {
        time_stale = true;
        ph = kClaims;
      }
    } else {
      // ---- k6 is in kn: solution, error norm, controller ---------------------
      double yn[kOwned];
      if (owner) {
        double e_max = ErrorNorm{}.rmax;
        bool forbidden = false;
        unsigned negative = 0u;
#pragma unroll
        for (int i = 0; i < kOwned; ++i) {
#pragma clang fp contract(off)
          yn[i] = fma(h0, fma(ck::c6, kn[i], sp[i]), y[i]);
          const double ye =
              h0 * fma(ck::ec6, kn[i],
                       fma(ck::ec5, K(4, i), fma(ck::ec4, K(3, i), fma(ck::ec3, K(2, i), ck::ec1 * K(0, i)))));
          e_max = fmax(e_max, error_ratio(a.eps_rel, yn[i], ye, abs_tol[i]));
          forbidden = forbidden || (enforce && ((nonneg >> i) & 1u) && yn[i] < 0.0);
          negative |= yn[i] < 0.0 ? 1u << i : 0u;
        }
        // The next derivative is taken at the new state; a lane whose attempt
        // is rejected does not need one, so it is published without a choice.
#pragma unroll
        for (int i = 0; i < kOwned; ++i) XY[i * kGroupNodes] = yn[i];
        F[(kFarNorm + wave) * kGroupNodes] = e_max;
        norm_flags[wave * kGroupNodes + lane] = (forbidden ? 1 : 0) | ((negative & fixable) ? 2 : 0);
      }
      __syncthreads();   // error norms and new state published
      rmax = ErrorNorm{}.rmax;
      int seen = 0;
#pragma unroll
      for (int w = 0; w < kOwnerWaves; ++w) {
        const double r = F[(kFarNorm + w) * kGroupNodes];
        rmax = fmax(rmax, r);
        seen |= norm_flags[w * kGroupNodes + lane];
      }
      s.clear(LaneFlags::kForbidden | LaneFlags::kNeedFix);
      if (seen & 1) s.set(LaneFlags::kForbidden);
      if (seen & 2) s.set(LaneFlags::kNeedFix);
      const bool stepping = s.has(LaneFlags::kStepping);
      const bool accepted = stepping && hadjust_kind(norm()) != kHadjDec;
      const bool final_step = s.has(LaneFlags::kFinalStep), need_fix = s.has(LaneFlags::kNeedFix);
      bool done = false;
      if (stepping) s.set(LaneFlags::kDecide);
      if (accepted) {
        if (wave == kCoolingWave) ++n_accept;
        t = final_step ? t1 : t + h0;
        done = !(sign * (t1 - t) > 0.0);
        if (done) s.clear(LaneFlags::kDecide);
        else s.set(LaneFlags::kEval | LaneFlags::kPost);
      }
      if (__any(done)) {
        if (__any(done && need_fix)) {
          fix_published(done && need_fix, [&](int i, double v) { yn[i] = v; });
        }
        if (owner && done) {
#pragma unroll
          for (int i = 0; i < kOwned; ++i) store_state_word<GRAPH>(a.y + (size_t)(v0 + i) * a.ld + node, yn[i]);
        }
        // odeSolverSolve returns xStep = driver h (solver.F90:593)
        double h_out = h;
        if (wave == kCoolingWave && done && !final_step) h_out = hadjust_step(norm(), kRkckOrder, h0);
        finish(done, h_out, true, GAL_STATUS_SUCCESS);
      }
      if (owner && accepted) {
#pragma unroll
        for (int i = 0; i < kOwned; ++i) Y0(i) = yn[i];
      }
      ph = kClaims;
    }
  }
}

template <bool GRAPH>
__global__ __launch_bounds__(kGroupNodes * kGroupWaves, 1) void evolve_kernel(EvolveArgs a) {
  extern __shared__ double exchange[];
  __shared__ GroupConstants constants;
  __shared__ int norm_flags[kOwnerWaves * kGroupNodes];   // bit 0: forbidden, bit 1: post-step needed, bit 2: rescue
  __shared__ int wall_expired;
  __shared__ int flags[kSignals];
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kGroupNodes));
  double* X = exchange + (threadIdx.x & (kGroupNodes - 1));
  if (threadIdx.x < kSignals) flags[threadIdx.x] = 0;
  for (int k = wave; k < 2 * kNV; k += kGroupWaves) X[(kXGalaxy + k) * kGroupNodes] = 0.0;
  {
    // the derived constants and the table's grid are read from the kernel's
    // argument segment, which its one argument starts
    const char* args = (const char*)__builtin_amdgcn_kernarg_segment_ptr();
    const double* d = (const double*)(args + offsetof(EvolveArgs, D));
    const double* c = (const double*)(args + offsetof(EvolveArgs, cd));
    constexpr int threads = kGroupNodes * kGroupWaves;
    for (int k = threadIdx.x; k < GAL_NPARAM; k += threads) constants.P[k] = a.P[k];
    for (int k = threadIdx.x; k < (int)(sizeof(constants.D) / 8); k += threads) ((double*)&constants.D)[k] = d[k];
    for (int k = threadIdx.x; k < (int)(sizeof(constants.C) / 8); k += threads) ((double*)&constants.C)[k] = c[k];
  }
  __syncthreads();
  if (wave == kGalaxyWave) group_wave<kGalaxyWave, GRAPH>(a, X, constants, norm_flags, flags, wall_expired);
  else if (wave == kProfileWave) group_wave<kProfileWave, GRAPH>(a, X, constants, norm_flags, flags, wall_expired);
  else if (wave == kTimeWave) group_wave<kTimeWave, GRAPH>(a, X, constants, norm_flags, flags, wall_expired);
  else group_wave<kCoolingWave, GRAPH>(a, X, constants, norm_flags, flags, wall_expired);
}

__global__ void reset_counter_kernel(unsigned int* w) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *w = 0u;
}

// One lane per node and 2600 instructions a wave (2164 vector, 401 scalar)
// with 38 doubles of a node in and 30 out: a million nodes take 116 to 132 us,
// 4.1 to 4.7 TB/s, and 100,000 17 us, in which a wave issues vector instructions for 31 %
// of its time and waits for memory or an issue slot for 63 %.  The whole RHS
// in one lane wants more than 200 registers, so two waves share a SIMD: with
// 128 registers a wave (four to a SIMD) it spills and takes 210 us, with 168
// 149 us.  Single waves as workgroups spread a small batch over more CUs than
// groups of four do (123 us and 17 us).
constexpr int kRhsThreads = 64, kRhsWavesPerSimd = 2;
__global__ __launch_bounds__(kRhsThreads, kRhsWavesPerSimd) void rhs_kernel(int n, int ld, const double* __restrict__ t, const double* __restrict__ y,
                           const double* __restrict__ npa, double* __restrict__ dydt, const double* __restrict__ P,
                           const double* __restrict__ tab, DerivedConstants D, CoolingDesc cd, int mode) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double yy[kNV], f[kNV];
#pragma unroll
  for (int v = 0; v < kNV; ++v) yy[v] = y[v * (size_t)ld + i];
  const NodePar np = load_node_par(npa, ld, i);
  rhs(P, D, tab, cd, mode, np, t[i], yy, f);
#pragma unroll
  for (int v = 0; v < kNV; ++v) dydt[v * (size_t)ld + i] = f[v];
}

__global__ void hadjust_kernel(int n, int dim, int ord, double eps_abs, double eps_rel, double a_y, double a_dydt,
                               const double* __restrict__ y, const double* __restrict__ yerr,
                               const double* __restrict__ yp, const double* __restrict__ scale,
                               const int* __restrict__ nonneg, double* __restrict__ h, int* __restrict__ result) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  ErrorNorm en;
  const double h_old = h[i];
  for (int v = 0; v < dim; ++v) {
    const size_t k = v * (size_t)n + i;
    error_norm_add(en, eps_abs, eps_rel, a_y, a_dydt, h_old, y[k], yerr[k], yp[k], scale[k], nonneg[k] != 0);
  }
  double hh = h_old;
  result[i] = hadjust_decide(en, ord, hh);
  h[i] = hh;
}

// Stiffness probe for the claim order: one RHS evaluation per node at its
// start point; cost key = |t_end - t_start| / sqrt(tau), tau = the shortest
// e-folding time min_v (|y_v| + scale_v) / |dy_v/dt|.  Only the order in
// which lanes claim nodes depends on it, never a result.
__global__ __launch_bounds__(kRhsThreads, kRhsWavesPerSimd) void cost_probe_kernel(int n_items, const int* __restrict__ subset, int ld, const double* __restrict__ y,
                                  const double* __restrict__ npa, const double* __restrict__ t_start,
                                  const double* __restrict__ t_end, const double* __restrict__ scale_in,
                                  const double* __restrict__ P, const double* __restrict__ tab, DerivedConstants D,
                                  CoolingDesc cd, int mode, int scales_given, const int* __restrict__ n_valid,
                                  float* __restrict__ key, int* __restrict__ index) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n_items) return;
  if (n_valid && j >= *n_valid) {
    // beyond the count the caller's list is unset: sorted last, never claimed
    key[j] = -1.0f;
    index[j] = 0;
    return;
  }
  const int i = subset ? subset[j] : j;
  double yy[kNV], f[kNV], sc[kNV];
#pragma unroll
  for (int v = 0; v < kNV; ++v) yy[v] = y[v * (size_t)ld + i];
  const NodePar np = load_node_par(npa, ld, i);
  const double t0 = t_start[i];
  if (scales_given) {
#pragma unroll
    for (int v = 0; v < kNV; ++v) sc[v] = scale_in[v * (size_t)ld + i];
  } else if (mode == GAL_PHYSICS_TEST) {
#pragma unroll
    for (int v = 0; v < kNV; ++v) sc[v] = 1.0;
  } else {
    scales(P, D, np, t0, yy, sc);
  }
  rhs(P, D, tab, cd, mode, np, t0, yy, f);
  double tau = 1.0e30;
#pragma unroll
  for (int v = 0; v < kNV; ++v) {
    const double r = fabs(f[v]);
    const double tv = (fabs(yy[v]) + fabs(sc[v])) / r;
    tau = (r > 0.0 && tv < tau) ? tv : tau;
  }
  const double k = fabs(t_end[i] - t0) * rsqrt(fmax(tau, 1.0e-30));
  key[j] = (float)fmin(k, 3.0e38);
  index[j] = i;
}

// LDS of a group of nodes: one group fills a CU's 160 KiB.
constexpr size_t kExchangeBytes = sizeof(double) * kXVectors * kGroupNodes;
static_assert(kExchangeBytes + sizeof(GroupConstants) + 1024 <= 163840, "a group must fit 160 KiB");

hipError_t set_lds_attributes() {
  for (const void* f : {(const void*)evolve_kernel<false>, (const void*)evolve_kernel<true>}) {
    const hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kExchangeBytes);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace

// ============================================================================
// C ABI
// ============================================================================
static int half_power_code(double alpha) {
  const double a2 = 2.0 * alpha;
  if (a2 == std::floor(a2) && std::fabs(a2) <= 16.0) return (int)a2;
  return kNoHalfPower;
}

static void derive_constants(const double* p, DerivedConstants& D) {
  const double om = p[GAL_P_OMEGA_MATTER], ol = p[GAL_P_OMEGA_DARK_ENERGY], h0 = p[GAL_P_HUBBLE_CONSTANT];
  D.om = om;
  D.ol = ol;
  D.a3_norm = om / ol;
  D.sinh_arg = 1.5 * std::sqrt(ol) * h0 / kMpcPerKmsToGyr;
  const double rho_crit0 = 3.0 * h0 * h0 / (8.0 * kPi * kGravity);
  D.rvir_coeff = 3.0 / (4.0 * kPi * rho_crit0);
  const double ar = 1.0 / (1.0 + p[GAL_P_REDSHIFT_REIONIZATION]);
  D.a3_reion = ar * ar * ar;
  D.f_baryon = p[GAL_P_OMEGA_BARYON] / om;
  D.inv_200 = 1.0 / 200.0;
  D.inv_sqrt_200 = 1.0 / std::sqrt(200.0);
  D.ln_200 = std::log(200.0);
  D.v_fb_disk = p[GAL_P_FB_DISK_VELOCITY];
  D.sqrt_v_fb_disk = std::sqrt(D.v_fb_disk);
  D.ln_v_fb_disk = std::log(D.v_fb_disk);
  D.v_fb_sph = p[GAL_P_FB_SPHEROID_VELOCITY];
  D.sqrt_v_fb_sph = std::sqrt(D.v_fb_sph);
  D.ln_v_fb_sph = std::log(D.v_fb_sph);
  D.n2_sf_disk = half_power_code(p[GAL_P_SF_DISK_EXPONENT_VELOCITY]);
  D.n2_sf_sph = half_power_code(p[GAL_P_SF_SPHEROID_EXPONENT_VELOCITY]);
  D.n2_fb_disk = half_power_code(p[GAL_P_FB_DISK_EXPONENT]);
  D.n2_fb_sph = half_power_code(p[GAL_P_FB_SPHEROID_EXPONENT]);
  D.t_vir_per_v2 = 0.5 * kAtomicMassUnit * kMeanAtomicMassPrimordial * kKilo * kKilo / kBoltzmann;
  D.cs2_per_t = 5.0 / 3.0 * kBoltzmann / (kMeanAtomicMassPrimordial * kAtomicMassUnit) / (kKilo * kKilo);
  D.cs2_sph = D.cs2_per_t * p[GAL_P_BH_TEMPERATURE_SPHEROID];
  D.m_edd_per_mass = 4.0 * kPi * kGravitySI * kMassHydrogenAtom * kGigaYear / kThomson / kSpeedLight;
  const double unit = kErgs * kGigaYear / kMassSolar / (kKilo * kKilo);
  // (M/1e9)^0.9 (Mdot/(k M))^1.2 = 1e9^-0.9 k^-1.2 M^-0.3 Mdot^1.2
  const double ln_common = -0.9 * std::log(1.0e9) - 1.2 * std::log(D.m_edd_per_mass);
  D.ln_jet_kerr = 42.7 * std::log(10.0) + std::log(unit) + ln_common;
  D.ln_jet_schw = 41.7 * std::log(10.0) + std::log(unit) + ln_common;
  D.cool_k_pre = p[GAL_P_DEGREES_OF_FREEDOM] / 2.0 * kBoltzmann / kErgs / kGigaYear;
  D.unit_energy = kMassSolar * kKilo * kKilo / kErgs / kGigaYear;
  const double mpc_cm = kHecto * kMegaParsec;
  D.nh_coeff = kMassSolar / kMassHydrogenAtom / (mpc_cm * mpc_cm * mpc_cm);
  D.inv_eff_sf_disk = p[GAL_P_SF_DISK_EFFICIENCY] != 0.0 ? 1.0 / p[GAL_P_SF_DISK_EFFICIENCY] : 0.0;
  D.inv_eff_sf_sph = p[GAL_P_SF_SPHEROID_EFFICIENCY] != 0.0 ? 1.0 / p[GAL_P_SF_SPHEROID_EFFICIENCY] : 0.0;
  D.inv_tmin_fb_disk = 1.0 / p[GAL_P_FB_DISK_TIMESCALE_MINIMUM];
  D.inv_tmin_fb_sph = 1.0 / p[GAL_P_FB_SPHEROID_TIMESCALE_MINIMUM];
  D.inv_core = 1.0 / p[GAL_P_CORE_RADIUS_OVER_VIRIAL];
  D.inv_cs2_sph = D.cs2_sph > 0.0 ? 1.0 / D.cs2_sph : 0.0;
  const double bhl_unit = kKilo * kGigaYear / kMegaParsec * 4.0 * kPi;
  D.bhl_sph_coeff = D.cs2_sph > 0.0 ? p[GAL_P_BH_ENHANCEMENT_SPHEROID] * bhl_unit * kGravity * kGravity /
                                          (D.cs2_sph * std::sqrt(D.cs2_sph))
                                    : 0.0;
  D.jeans_coeff = D.cs2_sph > 0.0 ? kGravity / D.cs2_sph : 0.0;
  D.h0_gyr = h0 / kMpcPerKmsToGyr;
  D.inv_one_minus_j_loss = 1.0 / (1.0 - p[GAL_P_FRACTION_LOSS_ANGULAR_MOMENTUM]);
  // Ciotti & Ostriker wind coupling (black_holes/winds/Ciotti2009.F90:156-175):
  // P_ISM / P_wind = 3 (3/2) k T_ISM v_wind Gyr / (m_H c^2 Mpc) * M_gas / (r eff Mdot)
  {
    constexpr double kVelocityWind = 1.0e4, kTemperatureISM = 1.0e4;  // km/s, K
    D.wind_pressure_ratio = 3.0 * 1.5 * kBoltzmann * kTemperatureISM * kGigaYear * (kVelocityWind * kKilo) /
                            (kMassHydrogenAtom * kSpeedLight * kSpeedLight * kMegaParsec);
  }
}

extern "C" {

int gal_ode_version(void) { return 10000; }

int gal_ode_device_check(int* n_devices, int* n_cus) {
  int nd = 0;
  if (hipGetDeviceCount(&nd) != hipSuccess || nd < 1) {
    if (n_devices) *n_devices = 0;
    return GAL_E_NODEVICE;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, 0) != hipSuccess) return GAL_E_HIP;
  if (n_devices) *n_devices = nd;
  if (n_cus) *n_cus = prop.multiProcessorCount;
  if (std::strncmp(prop.gcnArchName, "gfx950", 6) != 0) return GAL_E_NODEVICE;
  return GAL_OK;
}

int gal_ode_batch_create(int n_max, double tol_abs, double tol_rel, int flags, gal_ode_batch** out) {
  if (!out || n_max < 0) return GAL_E_INVALID;
  if (tol_abs < 0.0 || tol_rel < 0.0 || (tol_abs <= 0.0 && tol_rel <= 0.0)) return GAL_E_INVALID;
  *out = nullptr;
  int nd = 0, ncu = 0;
  int rc = gal_ode_device_check(&nd, &ncu);
  if (rc != GAL_OK) return rc;
  gal_ode_batch* h = new gal_ode_batch();
  h->n_max = n_max;
  h->tol_abs = tol_abs;
  h->tol_rel = tol_rel;
  h->flags = flags;
  if (hipGetDevice(&h->device) != hipSuccess) {
    delete h;
    return GAL_E_HIP;
  }
  h->n_cus = ncu;
  {
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, h->device) == hipSuccess && khz > 0)
      h->wall_clock_hz = 1.0e3 * khz;
    else
      (void)hipGetLastError();
  }
  const size_t nm = (size_t)std::max(n_max, 1);
  if (hipMalloc(&h->d_params, sizeof(double) * GAL_NPARAM) != hipSuccess ||
      hipMalloc(&h->d_table, sizeof(double) * GAL_COOLING_NT_MAX * GAL_COOLING_NZ_MAX) != hipSuccess ||
      hipMalloc(&h->d_work, sizeof(unsigned int)) != hipSuccess ||
      hipMalloc(&h->d_order, sizeof(int) * nm) != hipSuccess || hipMalloc(&h->d_index, sizeof(int) * nm) != hipSuccess ||
      hipMalloc(&h->d_key, sizeof(float) * nm) != hipSuccess ||
      hipMalloc(&h->d_key_sorted, sizeof(float) * nm) != hipSuccess) {
    gal_ode_batch_destroy(h);
    return GAL_E_NOMEM;
  }
  if (hipcub::DeviceRadixSort::SortPairsDescending(nullptr, h->sort_temp_bytes, h->d_key, h->d_key_sorted,
                                                   h->d_index, h->d_order, (int)nm) != hipSuccess ||
      hipMalloc(&h->d_sort_temp, std::max<size_t>(h->sort_temp_bytes, 16)) != hipSuccess) {
    gal_ode_batch_destroy(h);
    return GAL_E_NOMEM;
  }
  // Set on every handle creation (on the current device): no process-wide
  // state, and cheap.
  if (set_lds_attributes() != hipSuccess) {
    (void)hipGetLastError();
    gal_ode_batch_destroy(h);
    return GAL_E_HIP;
  }
  *out = h;
  return GAL_OK;
}

static void free_staging(gal_ode_batch* h) {
  hipFree(h->d_y); hipFree(h->d_np); hipFree(h->d_t0); hipFree(h->d_t1); hipFree(h->d_h);
  hipFree(h->d_scale); hipFree(h->d_status); hipFree(h->d_counters);
  h->d_y = h->d_np = h->d_t0 = h->d_t1 = h->d_h = h->d_scale = nullptr;
  h->d_status = nullptr;
  h->d_counters = nullptr;
}

int gal_ode_batch_destroy(gal_ode_batch* h) {
  if (!h) return GAL_E_INVALID;
  hipFree(h->d_params);
  hipFree(h->d_table);
  hipFree(h->d_work);
  hipFree(h->d_order);
  hipFree(h->d_index);
  hipFree(h->d_key);
  hipFree(h->d_key_sorted);
  hipFree(h->d_sort_temp);
  free_staging(h);
  delete h;
  return GAL_OK;
}

static bool physics_valid(const double* params) {
  const int mode = (int)params[GAL_P_PHYSICS_MODE];
  if (mode < GAL_PHYSICS_STANDARD || mode > GAL_PHYSICS_TEST) return false;
  if (!(params[GAL_P_OMEGA_MATTER] > 0.0) || !(params[GAL_P_OMEGA_DARK_ENERGY] > 0.0) ||
      !(params[GAL_P_HUBBLE_CONSTANT] > 0.0) || !(params[GAL_P_FB_DISK_VELOCITY] > 0.0) ||
      !(params[GAL_P_FB_SPHEROID_VELOCITY] > 0.0) || !(params[GAL_P_FB_DISK_TIMESCALE_MINIMUM] > 0.0) ||
      !(params[GAL_P_FB_SPHEROID_TIMESCALE_MINIMUM] > 0.0) || !(params[GAL_P_CORE_RADIUS_OVER_VIRIAL] > 0.0) ||
      !(params[GAL_P_FRACTION_LOSS_ANGULAR_MOMENTUM] < 1.0) || !(params[GAL_P_OPERATORS] >= 0.0) ||
      !(params[GAL_P_OPERATORS] <= 15.0))
    return false;
  return true;
}

int gal_ode_batch_set_physics(gal_ode_batch* h, const double* params, int n_params) {
  if (!h || !params || n_params != GAL_NPARAM) return GAL_E_INVALID;
  if (!physics_valid(params)) return GAL_E_INVALID;
  std::memcpy(h->params, params, sizeof(double) * GAL_NPARAM);
  derive_constants(h->params, h->D);
  HIP_TRY(hipMemcpy(h->d_params, h->params, sizeof(double) * GAL_NPARAM, hipMemcpyHostToDevice));
  h->have_physics = true;
  return GAL_OK;
}

static bool cooling_table_valid(const double* ln_lambda, int n_t, double d_ln_t, int n_z, double d_ln_z) {
  return ln_lambda && n_t >= 2 && n_z >= 2 && n_t <= GAL_COOLING_NT_MAX && n_z <= GAL_COOLING_NZ_MAX &&
         d_ln_t > 0.0 && d_ln_z > 0.0;
}

static void cooling_desc(CoolingDesc& c, int n_t, double ln_t_min, double d_ln_t, int n_z, double ln_z_min,
                         double d_ln_z) {
  c.n_t = n_t;
  c.n_z = n_z;
  c.ln_t_min = ln_t_min;
  c.d_ln_t = d_ln_t;
  c.inv_d_ln_t = 1.0 / d_ln_t;
  c.ln_z_min = ln_z_min;
  c.d_ln_z = d_ln_z;
  c.inv_d_ln_z = 1.0 / d_ln_z;
  c.t_min = std::exp(ln_t_min);
  c.t_max = std::exp(ln_t_min + d_ln_t * (n_t - 1));
  c.z_min = std::exp(ln_z_min);
  c.z_max = std::exp(ln_z_min + d_ln_z * (n_z - 1));
}

int gal_ode_batch_set_cooling_table(gal_ode_batch* h, const double* ln_lambda, int n_t, double ln_t_min,
                                    double d_ln_t, int n_z, double ln_z_min, double d_ln_z) {
  if (!h || !cooling_table_valid(ln_lambda, n_t, d_ln_t, n_z, d_ln_z)) return GAL_E_INVALID;
  cooling_desc(h->cd, n_t, ln_t_min, d_ln_t, n_z, ln_z_min, d_ln_z);
  HIP_TRY(hipMemcpy(h->d_table, ln_lambda, sizeof(double) * n_t * n_z, hipMemcpyHostToDevice));
  h->have_table = true;
  return GAL_OK;
}

int gal_ode_batch_set_launch(gal_ode_batch* h, int nodes_per_block, int blocks_per_cu) {
  if (!h) return GAL_E_INVALID;
  if (nodes_per_block != 64) return GAL_E_INVALID;
  // kept and reported only: launch_evolve has one shape
  if (blocks_per_cu < 1 || blocks_per_cu > 4) return GAL_E_INVALID;
  h->nodes_per_block = nodes_per_block;
  h->blocks_per_cu = blocks_per_cu;
  return GAL_OK;
}

int gal_ode_batch_set_wall_limit(gal_ode_batch* h, double seconds) {
  if (!h || !(seconds == seconds)) return GAL_E_INVALID;
  if (seconds > 0.0 && !(h->wall_clock_hz > 0.0)) return GAL_E_HIP;
  h->wall_limit_s = seconds > 0.0 ? seconds : 0.0;
  return GAL_OK;
}

int gal_ode_batch_set_graph_stall_limit(gal_ode_batch* h, double seconds) {
  if (!h || !(seconds == seconds)) return GAL_E_INVALID;
  h->graph_stall_s = seconds > 0.0 ? seconds : 60.0;
  return GAL_OK;
}

int gal_ode_batch_set_rhs_waves(gal_ode_batch* h, int waves) {
  if (!h || (waves != 1 && waves != 2)) return GAL_E_INVALID;
  h->rhs_waves = waves;
  return GAL_OK;
}

int gal_ode_batch_get_launch(gal_ode_batch* h, int* nodes_per_block, int* blocks_per_cu, int* rhs_waves) {
  if (!h) return GAL_E_INVALID;
  if (nodes_per_block) *nodes_per_block = h->nodes_per_block;
  if (blocks_per_cu) *blocks_per_cu = h->blocks_per_cu;
  if (rhs_waves) *rhs_waves = h->rhs_waves;
  return GAL_OK;
}

extern "C++" {
template <bool GRAPH = false>
static int launch_evolve(gal_ode_batch* h, const EvolveArgs& args, hipStream_t s) {
  // a combination that is documented as refused; the kernel would run alike
  if (h->rhs_waves == 2 && h->blocks_per_cu > 2) return GAL_E_INVALID;
  // one group of nodes fills a CU, and a lone group per CU is claimed from
  // until the last node is out
  const int blocks = std::max(1, h->n_cus);
  hipLaunchKernelGGL(reset_counter_kernel, dim3(1), dim3(64), 0, s, args.work);
  hipLaunchKernelGGL((evolve_kernel<GRAPH>), dim3(blocks), dim3(kGroupNodes * kGroupWaves), kExchangeBytes, s, args);
  HIP_TRY(hipGetLastError());
  return GAL_OK;
}
}  // extern "C++"

static int make_args(gal_ode_batch* h, int n, int ld, double* y, const double* node_par, const double* t_start,
                     const double* t_end, double* h_step, double* scale, int* status, int64_t* counters,
                     EvolveArgs& a) {
  if (!h || n < 0 || n > h->n_max || ld < n) return GAL_E_INVALID;
  if (!h->have_physics || !h->have_table) return GAL_E_INVALID;
  if (n > 0 && (!y || !node_par || !t_start || !t_end || !h_step || !status)) return GAL_E_INVALID;
  if ((h->flags & GAL_FLAG_SCALES_PROVIDED) && !scale) return GAL_E_INVALID;
  a.n = n;
  a.n_claim = n;
  a.ld = ld;
  a.y = y;
  a.np = node_par;
  a.t_start = t_start;
  a.t_end = t_end;
  a.h_step = h_step;
  a.scale = scale;
  a.status = status;
  a.counters = reinterpret_cast<long long*>(counters);
  a.order = nullptr;
  a.n_claim_dev = nullptr;
  a.work = h->d_work;
  a.P = h->d_params;
  a.tab = h->d_table;
  a.D = h->D;
  a.cd = h->cd;
  a.eps_abs = h->tol_abs;
  a.eps_rel = h->tol_rel;
  a.flags = h->flags;
  a.mode = (int)h->params[GAL_P_PHYSICS_MODE];
  a.wall_ticks = 0;
  if (h->wall_limit_s > 0.0)
    a.wall_ticks = (unsigned long long)std::max(1.0, std::min(h->wall_limit_s * h->wall_clock_hz, 1.0e18));
  return GAL_OK;
}

int gal_ode_batch_evolve_d(gal_ode_batch* h, int n, int ld, double* y, const double* node_par,
                           const double* t_start, const double* t_end, double* h_step, double* scale, int* status,
                           int64_t* counters, void* stream) {
  return gal_ode_evolve_subset(h, n, ld, y, node_par, t_start, t_end, h_step, scale, status, counters, nullptr, n,
                               (hipStream_t)stream);
}

int gal_ode_batch_evolve_h(gal_ode_batch* h, int n, double* y, const double* node_par, const double* t_start,
                           const double* t_end, double* h_step, double* scale, int* status, int64_t* counters) {
  if (!h || n < 0 || n > h->n_max) return GAL_E_INVALID;
  if (n == 0) return GAL_OK;
  if (!y || !node_par || !t_start || !t_end || !h_step || !status) return GAL_E_INVALID;
  if (!h->d_y) {
    const size_t nm = (size_t)h->n_max;
    if (hipMalloc(&h->d_y, sizeof(double) * GAL_NVAR * nm) != hipSuccess ||
        hipMalloc(&h->d_np, sizeof(double) * GAL_NPARAM_NODE * nm) != hipSuccess ||
        hipMalloc(&h->d_t0, sizeof(double) * nm) != hipSuccess ||
        hipMalloc(&h->d_t1, sizeof(double) * nm) != hipSuccess ||
        hipMalloc(&h->d_h, sizeof(double) * nm) != hipSuccess ||
        hipMalloc(&h->d_scale, sizeof(double) * GAL_NVAR * nm) != hipSuccess ||
        hipMalloc(&h->d_status, sizeof(int) * nm) != hipSuccess ||
        hipMalloc(&h->d_counters, sizeof(long long) * 3 * nm) != hipSuccess) {
      free_staging(h);
      return GAL_E_NOMEM;
    }
  }
  const size_t nn = (size_t)n;
  HIP_TRY(hipMemcpy(h->d_y, y, sizeof(double) * GAL_NVAR * nn, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(h->d_np, node_par, sizeof(double) * GAL_NPARAM_NODE * nn, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(h->d_t0, t_start, sizeof(double) * nn, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(h->d_t1, t_end, sizeof(double) * nn, hipMemcpyHostToDevice));
  HIP_TRY(hipMemcpy(h->d_h, h_step, sizeof(double) * nn, hipMemcpyHostToDevice));
  if ((h->flags & GAL_FLAG_SCALES_PROVIDED) && scale)
    HIP_TRY(hipMemcpy(h->d_scale, scale, sizeof(double) * GAL_NVAR * nn, hipMemcpyHostToDevice));
  int rc = gal_ode_batch_evolve_d(h, n, n, h->d_y, h->d_np, h->d_t0, h->d_t1, h->d_h, h->d_scale, h->d_status,
                                  counters ? reinterpret_cast<int64_t*>(h->d_counters) : nullptr, nullptr);
  if (rc != GAL_OK) return rc;
  HIP_TRY(hipDeviceSynchronize());
  HIP_TRY(hipMemcpy(y, h->d_y, sizeof(double) * GAL_NVAR * nn, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(h_step, h->d_h, sizeof(double) * nn, hipMemcpyDeviceToHost));
  HIP_TRY(hipMemcpy(status, h->d_status, sizeof(int) * nn, hipMemcpyDeviceToHost));
  if (scale) HIP_TRY(hipMemcpy(scale, h->d_scale, sizeof(double) * GAL_NVAR * nn, hipMemcpyDeviceToHost));
  if (counters) HIP_TRY(hipMemcpy(counters, h->d_counters, sizeof(long long) * 3 * nn, hipMemcpyDeviceToHost));
  return GAL_OK;
}

int gal_ode_rhs_d(gal_ode_batch* h, int n, int ld, const double* t, const double* y, const double* node_par,
                  double* dydt, void* stream) {
  if (!h || n < 0 || ld < n || !h->have_physics || !h->have_table) return GAL_E_INVALID;
  if (n == 0) return GAL_OK;
  if (!t || !y || !node_par || !dydt) return GAL_E_INVALID;
  const int threads = kRhsThreads;
  hipLaunchKernelGGL(rhs_kernel, dim3((n + threads - 1) / threads), dim3(threads), 0, (hipStream_t)stream, n, ld, t,
                     y, node_par, dydt, (const double*)h->d_params, (const double*)h->d_table, h->D, h->cd,
                     (int)h->params[GAL_P_PHYSICS_MODE]);
  HIP_TRY(hipGetLastError());
  return GAL_OK;
}

int gal_ode_hadjust_d(int n, int dim, int ord, double eps_abs, double eps_rel, double a_y, double a_dydt,
                      const double* y, const double* yerr, const double* yp, const double* scale,
                      const int* is_non_negative, double* h, int* result, void* stream) {
  if (n < 0 || dim < 1 || ord < 1) return GAL_E_INVALID;
  if (n == 0) return GAL_OK;
  if (!y || !yerr || !yp || !scale || !is_non_negative || !h || !result) return GAL_E_INVALID;
  const int threads = 256;
  hipLaunchKernelGGL(hadjust_kernel, dim3((n + threads - 1) / threads), dim3(threads), 0, (hipStream_t)stream, n, dim,
                     ord, eps_abs, eps_rel, a_y, a_dydt, y, yerr, yp, scale, is_non_negative, h, result);
  HIP_TRY(hipGetLastError());
  return GAL_OK;
}

int gal_ode_batch_autotune(gal_ode_batch* h, int n, int ld, double* y, const double* node_par,
                           const double* t_start, const double* t_end, double* h_step, double* scale, int* status,
                           void* stream, int* best_nodes_per_block, int* best_blocks_per_cu) {
  // The kernel runs alike at every admitted shape: there is nothing to time.
  if (!h || n <= 0 || n > h->n_max || ld < n || !h->have_physics || !h->have_table) return GAL_E_INVALID;
  if (!y || !node_par || !t_start || !t_end || !h_step) return GAL_E_INVALID;
  (void)scale; (void)status; (void)stream;
  h->nodes_per_block = 64;
  h->blocks_per_cu = 1;
  h->rhs_waves = 2;
  if (best_nodes_per_block) *best_nodes_per_block = h->nodes_per_block;
  if (best_blocks_per_cu) *best_blocks_per_cu = h->blocks_per_cu;
  return GAL_OK;
}

}  // extern "C"

// ============================================================================
// Allocation-free evolve
// ============================================================================
// The handle path keeps physics parameters, the cooling table and the claim
// counter in device buffers that gal_ode_batch_create allocates.  Callers
// that cannot allocate (code under graph capture, serving loops, harnesses
// that forbid hipMalloc) use gal_ode_evolve_static_d instead: its scratch is
// this file-scope array, one copy per GPU, held for the life of the process:
//   [0, 8)                         claim counter
//   [8, 8 + 8*GAL_NPARAM)          physics parameters
//   then                           cooling table, up to NT_MAX x NZ_MAX doubles
// Every call on a GPU reuses that GPU's copy; calls that overlap on one GPU
// race on it.
namespace {
constexpr size_t kStaticTableDoubles = (size_t)GAL_COOLING_NT_MAX * GAL_COOLING_NZ_MAX;
constexpr size_t kStaticScratchDoubles = 1 + GAL_NPARAM + kStaticTableDoubles;
constexpr int kMaxDevices = 64;
std::mutex g_static_mutex;
void* g_static_scratch[kMaxDevices] = {};
int g_static_cus[kMaxDevices] = {};
}  // namespace

static __device__ __align__(256) double scratch[kStaticScratchDoubles];

// Once per device, with that device current: the device address of this
// device's copy of the scratch array (the array's name is a host-side
// stand-in, not a device address), the CU count and the LDS attribute of the
// kernel the entry point launches.
static int static_scratch(int device, void** ptr, int* n_cus) {
  if (device < 0 || device >= kMaxDevices) return GAL_E_INVALID;
  std::lock_guard<std::mutex> lock(g_static_mutex);
  if (!g_static_scratch[device]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) {
      (void)hipGetLastError();
      return GAL_E_HIP;
    }
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1)
      return GAL_E_HIP;
    if (set_lds_attributes() != hipSuccess) {
      (void)hipGetLastError();
      return GAL_E_HIP;
    }
    g_static_cus[device] = cus;
    g_static_scratch[device] = p;
  }
  *ptr = g_static_scratch[device];
  *n_cus = g_static_cus[device];
  return GAL_OK;
}

extern "C" int gal_ode_evolve_static_d(const double* params, int n_params, const double* ln_lambda, int n_t,
                                       double ln_t_min, double d_ln_t, int n_z, double ln_z_min, double d_ln_z,
                                       double tol_abs, double tol_rel, int flags, int n, int ld, double* y,
                                       const double* node_par, const double* t_start, const double* t_end,
                                       double* h_step, double* scale, int* status, int64_t* counters, void* stream) {
  if (!params || n_params != GAL_NPARAM || !physics_valid(params)) return GAL_E_INVALID;
  if (!cooling_table_valid(ln_lambda, n_t, d_ln_t, n_z, d_ln_z)) {
    if (ln_lambda && ((size_t)n_t * (size_t)n_z > kStaticTableDoubles))
      fprintf(stderr, "gal_ode_evolve_static_d: cooling table %d x %d exceeds the %d x %d of the static scratch\n",
              n_t, n_z, GAL_COOLING_NT_MAX, GAL_COOLING_NZ_MAX);
    return GAL_E_INVALID;
  }
  if (tol_abs < 0.0 || tol_rel < 0.0 || (tol_abs <= 0.0 && tol_rel <= 0.0)) return GAL_E_INVALID;
  if (n < 0 || ld < n) return GAL_E_INVALID;
  if (n == 0) return GAL_OK;
  if (!y || !node_par || !t_start || !t_end || !h_step || !status) return GAL_E_INVALID;
  if ((flags & GAL_FLAG_SCALES_PROVIDED) && !scale) return GAL_E_INVALID;
  int device = 0;
  HIP_TRY(hipGetDevice(&device));
  void* base = nullptr;
  int n_cus = 0;
  int rc = static_scratch(device, &base, &n_cus);
  if (rc != GAL_OK) return rc;
  hipStream_t s = (hipStream_t)stream;
  unsigned int* work = reinterpret_cast<unsigned int*>(base);
  double* d_params = reinterpret_cast<double*>(base) + 1;
  double* d_table = d_params + GAL_NPARAM;
  HIP_TRY(hipMemcpyAsync(d_params, params, sizeof(double) * GAL_NPARAM, hipMemcpyHostToDevice, s));
  HIP_TRY(hipMemcpyAsync(d_table, ln_lambda, sizeof(double) * (size_t)n_t * n_z, hipMemcpyHostToDevice, s));
  EvolveArgs a{};
  a.n = n;
  a.n_claim = n;
  a.ld = ld;
  a.y = y;
  a.np = node_par;
  a.t_start = t_start;
  a.t_end = t_end;
  a.h_step = h_step;
  a.scale = scale;
  a.status = status;
  a.counters = reinterpret_cast<long long*>(counters);
  a.order = nullptr;             // claims in node order
  a.n_claim_dev = nullptr;
  a.work = work;
  a.P = d_params;
  a.tab = d_table;
  derive_constants(params, a.D);
  cooling_desc(a.cd, n_t, ln_t_min, d_ln_t, n_z, ln_z_min, d_ln_z);
  a.eps_abs = tol_abs;
  a.eps_rel = tol_rel;
  a.flags = flags;
  a.mode = (int)params[GAL_P_PHYSICS_MODE];
  a.wall_ticks = 0;
  // one group of nodes per CU; no workspace beyond the scratch
  hipLaunchKernelGGL(reset_counter_kernel, dim3(1), dim3(64), 0, s, work);
  hipLaunchKernelGGL((evolve_kernel<false>), dim3(n_cus), dim3(kGroupNodes * kGroupWaves), kExchangeBytes, s, a);
  HIP_TRY(hipGetLastError());
  return GAL_OK;
}

// Claim order of an evolve: every node's cost estimate, sorted so that the
// costliest nodes are claimed first (their chains then overlap the bulk).
// Writes h->d_order on stream s.
static int plan_claim_order(gal_ode_batch* h, int n_subset, const int* subset, int ld, const double* y,
                            const double* node_par, const double* t_start, const double* t_end, const double* scale,
                            const int* n_subset_dev, hipStream_t s) {
  const int threads = kRhsThreads;
  hipLaunchKernelGGL(cost_probe_kernel, dim3((n_subset + threads - 1) / threads), dim3(threads), 0, s, n_subset,
                     subset, ld, y, node_par, t_start, t_end, scale, (const double*)h->d_params,
                     (const double*)h->d_table, h->D, h->cd, (int)h->params[GAL_P_PHYSICS_MODE],
                     (h->flags & GAL_FLAG_SCALES_PROVIDED) ? 1 : 0, n_subset_dev, h->d_key, h->d_index);
  HIP_TRY(hipGetLastError());
  size_t tb = h->sort_temp_bytes;
  HIP_TRY(hipcub::DeviceRadixSort::SortPairsDescending(h->d_sort_temp, tb, h->d_key, h->d_key_sorted, h->d_index,
                                                       h->d_order, n_subset, 0, 32, s));
  return GAL_OK;
}

int gal_ode_evolve_subset(gal_ode_batch* h, int n, int ld, double* y, const double* node_par, const double* t_start,
                          const double* t_end, double* h_step, double* scale, int* status, int64_t* counters,
                          const int* subset, int n_subset, hipStream_t s, const int* n_subset_dev) {
  EvolveArgs a;
  int rc = make_args(h, n, ld, y, node_par, t_start, t_end, h_step, scale, status, counters, a);
  if (rc != GAL_OK) return rc;
  if (n_subset < 0 || n_subset > n || (subset == nullptr && n_subset != n)) return GAL_E_INVALID;
  if (n_subset == 0) return GAL_OK;
  a.n_claim = n_subset;
  a.n_claim_dev = n_subset_dev;   // when set, n_subset is the list's capacity
  a.order = subset;
  h->plan_y = nullptr;            // an evolve of its own replaces any pending plan
  if (h->flags & GAL_FLAG_COST_ORDER) {
    rc = plan_claim_order(h, n_subset, subset, ld, y, node_par, t_start, t_end, scale, n_subset_dev, s);
    if (rc != GAL_OK) return rc;
    a.order = h->d_order;
  }
  return launch_evolve(h, a, s);
}

int gal_ode_batch_plan_d(gal_ode_batch* h, int n, int ld, const double* y, const double* node_par,
                         const double* t_start, const double* t_end, const double* scale, void* stream) {
  if (!h || n < 0 || n > h->n_max || ld < n) return GAL_E_INVALID;
  if (!h->have_physics || !h->have_table || !(h->flags & GAL_FLAG_COST_ORDER)) return GAL_E_INVALID;
  if (n > 0 && (!y || !node_par || !t_start || !t_end || ((h->flags & GAL_FLAG_SCALES_PROVIDED) && !scale)))
    return GAL_E_INVALID;
  h->plan_y = nullptr;
  if (n > 0) {
    const int rc = plan_claim_order(h, n, nullptr, ld, y, node_par, t_start, t_end, scale, nullptr, (hipStream_t)stream);
    if (rc != GAL_OK) return rc;
  }
  h->plan_y = y;
  h->plan_n = n;
  h->plan_ld = ld;
  return GAL_OK;
}

int gal_ode_batch_evolve_planned_d(gal_ode_batch* h, int n, int ld, double* y, const double* node_par,
                                   const double* t_start, const double* t_end, double* h_step, double* scale,
                                   int* status, int64_t* counters, void* stream) {
  if (!h || !y || h->plan_y != y || h->plan_n != n || h->plan_ld != ld) return GAL_E_INVALID;
  h->plan_y = nullptr;   // a plan serves one evolve
  EvolveArgs a;
  const int rc = make_args(h, n, ld, y, node_par, t_start, t_end, h_step, scale, status, counters, a);
  if (rc != GAL_OK) return rc;
  if (n == 0) return GAL_OK;
  a.n_claim = n;
  a.n_claim_dev = nullptr;
  a.order = h->d_order;
  return launch_evolve(h, a, (hipStream_t)stream);
}

int gal_ode_evolve_graph(gal_ode_batch* h, int ld, double* y, double* h_step, double* scale, int* status,
                         const gal::OpGraph& g, int* graph_error, hipStream_t s) {
  if (!h || ld < 1 || ld > h->n_max || g.n < 0 || !graph_error) return GAL_E_INVALID;
  if (g.n == 0) return GAL_OK;
  if (!g.ops || !g.next_a || !g.next_b || !g.npred || !g.ready || !g.tail) return GAL_E_INVALID;
  EvolveArgs a;
  // the per-node arrays of the node mode are unused: intervals and halo
  // parameters come with each operation
  const double* unused = &g.ops->t0;
  int rc = make_args(h, ld, ld, y, unused, unused, unused, h_step, scale, status, nullptr, a);
  if (rc != GAL_OK) return rc;
  a.g = g;
  a.graph_error = graph_error;
  // a claimed entry may wait for the whole remaining critical path, but
  // not for the handle's stall limit (a minute by default) in which no
  // operation anywhere becomes ready
  const double hz = h->wall_clock_hz > 0.0 ? h->wall_clock_hz : 1.0e8;
  a.stall_ticks = (unsigned long long)std::min(std::max(h->graph_stall_s * hz, 1.0), 1.0e18);
  return launch_evolve<true>(h, a, s);
}
