// group_rhs.hpp -- the RHS of a group of 64 nodes computed by the four waves
// of a workgroup, one wave on each SIMD of a CU.  Internal.
//
// A node's Cash-Karp attempts are a serial chain of RHS evaluations, and a
// wave64 FP64 instruction takes its issue cycles whether one lane or all 64
// are active, so the time of a stiff node -- and of every launch, which lasts
// as long as its stiffest node -- is the chain of instructions from one
// barrier to the next, through whichever waves it crosses: the waves issue
// vector instructions in 35 % of their time and wait, for each other, LDS and
// the cooling table, in 45 %.  The blocks of physics.hpp are dealt out by what
// they wait for:
//   galaxy wave   the galaxy half, then the CGM outer radius;
//   profile wave  hot-halo profile, ISCO, spheroid accretion, then the mean
//                 radius of the hot gas, then the spheroid's rates, the black
//                 hole's spin and its winds;
//   time wave     the part that depends on the time alone, of the *next*
//                 stage (its time is known ahead of its state), and the step
//                 controller's pow; then the radiated energy;
//   cooling wave  cooling function and time, then cooling radius and hot-mode
//                 accretion, then jet power and net cooling: the serial chain
//                 that nothing takes off the path.
// They meet in a barrier when the stage state is published and when the
// derivatives are.  In between a value goes from the wave that computes it to
// the ones that need it by a flag in LDS (Signal below): barriers there made
// every wave wait for the slowest at each of them, 8800 cycles an evaluation
// for 6300 cycles of work in the busiest wave.
//
// All exchange goes through LDS vectors of 64 doubles, one per lane
// (conflict-free), each written by one wave.  The stage state, the time parts,
// the halves of the derivative, the error norms, the step size and the claims
// are read on the far side of a barrier.  The kMid vectors are written and
// read within one evaluation, with no barrier between: a wave reads one only
// after it has awaited the signal that is named beside it.
#pragma once
#include <hip/hip_runtime.h>

#include "physics.hpp"

namespace gal {

constexpr int kGroupNodes = 64;
enum : int { kGalaxyWave = 0, kProfileWave = 1, kTimeWave = 2, kCoolingWave = 3, kGroupWaves = 4 };

// The integrator's variables are owned by three of the waves, ten each; the
// cooling wave, the longest of an RHS, owns none.
constexpr int kOwnerWaves = 3, kOwned = kNV / kOwnerWaves;
static_assert(kOwned * kOwnerWaves == kNV, "owners must tile the state");

constexpr int kTimeVectors = (int)(sizeof(TimePart) / sizeof(double));
constexpr int kMidVectors = 10;

// Stages whose derivatives are kept: k1, k2 (whose place k5 takes once the last
// stage input no longer needs it), k3 and k4.  k6 is consumed as it is produced.
constexpr int kStages = 4;

// LDS of a group, in vectors of 64 doubles.
enum : int {
  kXState = 0,                              // stage state
  kXGalaxy = kXState + kNV,                 // galaxy half of the derivative
  kXHalo = kXGalaxy + kNV,                  // hot-halo half
  kXStage = kXHalo + kNV,                   // stage derivatives, each kNV vectors
  kXStart = kXStage + kStages * kNV,        // state at the start of the step
  kXFar = kXStart + kNV,                    // what follows, counted from here
  kXVectors = kXFar + 2 * kTimeVectors + kMidVectors + kOwnerWaves + 1
};
enum : int {
  kFarTime = 0,                             // TimePart of this stage and of the next
  kFarMid = kFarTime + 2 * kTimeVectors,    // published within an evaluation
  kFarNorm = kFarMid + kMidVectors,         // each owner's error norm
  kFarStep = kFarNorm + kOwnerWaves,        // step size chosen by the controller
  // published within an evaluation, by the profile wave:
  kMidRho0 = kFarMid, kMidRhoOut,             // kProfileReady
  kMidEffThin, kMidEddCap, kMidMdotSph,       // kAccretorReady
  kMidInvRMean,                               // kMeanRadiusReady
  // and by the cooling wave:
  kMidLambda, kMidNhPerRho, kMidNallPerNh,    // kCoolingFunctionReady
  kMidMdot,                                   // kAccretionReady
  kMidEnd,
  // claimed nodes, in the time part that is not in use
  kXClaimNode = 0, kXClaimT0, kXClaimT1, kXClaimStep, kXClaimPar
};
static_assert(kMidEnd - kFarMid == kMidVectors, "count the published values");
static_assert(kXClaimPar + GAL_NPARAM_NODE <= kTimeVectors, "a claim must fit a time part");

// The copy of the parameters that the RHS reads.
struct GroupConstants {
  double P[GAL_NPARAM];
  DerivedConstants D;
  CoolingDesc C;
};

// Variables whose derivative has a part in each half; the other entries of
// the exchange area stay zero.
constexpr unsigned var_bits(std::initializer_list<int> vars) {
  unsigned m = 0;
  for (int v : vars) m |= 1u << v;
  return m;
}
constexpr unsigned kGalaxyVars =
    var_bits({GAL_V_HOT_MASS, GAL_V_HOT_ABUNDANCES, GAL_V_HOT_ANGULAR_MOMENTUM, GAL_V_HOT_OUTFLOWED_MASS,
              GAL_V_HOT_OUTFLOWED_ANGULAR_MOMENTUM, GAL_V_HOT_OUTFLOWED_ABUNDANCES, GAL_V_HOT_UNACCRETED_MASS,
              GAL_V_HOT_UNACCRETED_ABUNDANCES, GAL_V_HOT_OUTER_RADIUS, GAL_V_HOT_STRIPPED_MASS,
              GAL_V_HOT_STRIPPED_ABUNDANCES, GAL_V_DISK_MASS_STELLAR, GAL_V_DISK_MASS_STELLAR_FORMED,
              GAL_V_DISK_ABUNDANCES_STELLAR, GAL_V_DISK_MASS_GAS, GAL_V_DISK_ABUNDANCES_GAS,
              GAL_V_DISK_ANGULAR_MOMENTUM, GAL_V_SPHEROID_MASS_STELLAR, GAL_V_SPHEROID_MASS_STELLAR_FORMED,
              GAL_V_SPHEROID_ABUNDANCES_STELLAR, GAL_V_SPHEROID_MASS_GAS, GAL_V_SPHEROID_ABUNDANCES_GAS,
              GAL_V_SPHEROID_ANGULAR_MOMENTUM, GAL_V_SPIN_ANGULAR_MOMENTUM, GAL_V_SATELLITE_BOUND_MASS});
constexpr unsigned kHaloVars =
    var_bits({GAL_V_HOT_MASS, GAL_V_HOT_ABUNDANCES, GAL_V_HOT_ANGULAR_MOMENTUM, GAL_V_HOT_OUTFLOWED_MASS,
              GAL_V_HOT_OUTFLOWED_ANGULAR_MOMENTUM, GAL_V_HOT_OUTFLOWED_ABUNDANCES, GAL_V_HOT_STRIPPED_MASS,
              GAL_V_HOT_STRIPPED_ABUNDANCES, GAL_V_HOT_ENERGY_RADIATED, GAL_V_DISK_MASS_GAS,
              GAL_V_DISK_ABUNDANCES_GAS, GAL_V_DISK_ANGULAR_MOMENTUM, GAL_V_SPHEROID_MASS_GAS,
              GAL_V_SPHEROID_ABUNDANCES_GAS, GAL_V_SPHEROID_ANGULAR_MOMENTUM, GAL_V_BH_MASS, GAL_V_BH_SPIN});

// What one wave tells others within an evaluation, as the number of the
// evaluation (a round counts up alike in all waves).  A wave publishes its
// vectors, then the flag; LDS keeps one wave's operations in order, and the
// fences keep the compiler to it.  Every wait ends: a flag is set by a wave of
// the same workgroup that runs the same rounds, and the waits form no cycle
// (profile -> cooling -> profile's last part; profile -> galaxy; cooling -> time).
enum Signal : int { kProfileReady = 0, kAccretorReady, kMeanRadiusReady, kCoolingFunctionReady, kAccretionReady, kSignals };

__device__ __forceinline__ void signal(int* __restrict__ flags, Signal s, int round) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if ((threadIdx.x & (kGroupNodes - 1)) == 0)
    __hip_atomic_store(flags + s, round, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ void await(int* __restrict__ flags, Signal s, int round) {
  while (__builtin_amdgcn_readfirstlane(
             __hip_atomic_load(flags + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) != round) {
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Work that follows a signal stays behind it: without this the compiler
// mixes later arithmetic in before the signal and delays who waits for it.
__device__ __forceinline__ double after_signal(double x) {
  asm volatile("" : "+v"(x) : : "memory");
  return x;
}

__device__ __forceinline__ TimePart load_time_part(const double* __restrict__ X) {
  double v[kTimeVectors];
#pragma unroll
  for (int k = 0; k < kTimeVectors; ++k) v[k] = X[k * kGroupNodes];
  return __builtin_bit_cast(TimePart, v);
}

__device__ __forceinline__ void store_time_part(const TimePart& T, double* __restrict__ X) {
  struct Values { double v[kTimeVectors]; };
  const Values w = __builtin_bit_cast(Values, T);
#pragma unroll
  for (int k = 0; k < kTimeVectors; ++k) X[k * kGroupNodes] = w.v[k];
}

__device__ __forceinline__ void load_state(const double* __restrict__ X, double (&y)[kNV]) {
#pragma unroll
  for (int v = 0; v < kNV; ++v) y[v] = X[(kXState + v) * kGroupNodes];
}

// X: this lane's column of the group's LDS; F: the part of it from kXFar on;
// time: this stage's time part.
__device__ __forceinline__ void galaxy_wave_rhs(const GroupConstants& G, int mode, int ops, const NodePar& np,
                                                double* __restrict__ X, double* __restrict__ F,
                                  const double* __restrict__ time, int* __restrict__ flags, int round) {
  double y[kNV], f[kNV];
  load_state(X, y);
#pragma unroll
  for (int v = 0; v < kNV; ++v) f[v] = 0.0;
  const TimePart T = load_time_part(time);
  if (mode == GAL_PHYSICS_TEST) {
    test_rates(T.time, y, f);
  } else {
    const bool box = mode == GAL_PHYSICS_BOX;
    galaxy_rates(G.P, G.D, ops, box, np, T, y, f);
    if (!box && (ops & GAL_OPERATOR_CGM_OUTER_RADIUS)) {
      await(flags, kProfileReady, round);
      outer_radius_rates(G.P, np, T, F[kMidRho0 * kGroupNodes], F[kMidRhoOut * kGroupNodes], y, f);
    }
  }
#pragma unroll
  for (int v = 0; v < kNV; ++v)
    if ((kGalaxyVars >> v) & 1u) X[(kXGalaxy + v) * kGroupNodes] = f[v];
}

// Of the hot-halo half, the profile wave writes the variables of the spheroid,
// the outflow and the black hole's spin, the time wave the radiated energy and
// the cooling wave the others.
constexpr unsigned kSpheroidVars =
    var_bits({GAL_V_HOT_OUTFLOWED_MASS, GAL_V_HOT_OUTFLOWED_ANGULAR_MOMENTUM, GAL_V_HOT_OUTFLOWED_ABUNDANCES,
              GAL_V_SPHEROID_MASS_GAS, GAL_V_SPHEROID_ABUNDANCES_GAS, GAL_V_SPHEROID_ANGULAR_MOMENTUM, GAL_V_BH_SPIN});
constexpr unsigned kCoolingVars = kHaloVars & ~kSpheroidVars & ~(1u << GAL_V_HOT_ENERGY_RADIATED);

__device__ __forceinline__ void profile_wave_rhs(const GroupConstants& G, int ops, double* __restrict__ X,
                                                 double* __restrict__ F, const double* __restrict__ time,
                                                 int* __restrict__ flags, int round) {
  auto Y = [&](int v) { return X[(kXState + v) * kGroupNodes]; };
  const TimePart T = load_time_part(time);
  const double m_hot = Y(GAL_V_HOT_MASS), r_out = Y(GAL_V_HOT_OUTER_RADIUS), m_bh = Y(GAL_V_BH_MASS);
  const double mg_s = Y(GAL_V_SPHEROID_MASS_GAS), ms_s = Y(GAL_V_SPHEROID_MASS_STELLAR);
  const double j_s = Y(GAL_V_SPHEROID_ANGULAR_MOMENTUM), zg_s = Y(GAL_V_SPHEROID_ABUNDANCES_GAS);
  const double y_spin = Y(GAL_V_BH_SPIN), r_bh = Y(GAL_V_BH_RADIAL_POSITION);
  const GalaxyRadius galaxy = galaxy_radius(T, Y(GAL_V_SPIN_ANGULAR_MOMENTUM));
  HotProfile p = hot_profile(T, m_hot, r_out);
  F[kMidRho0 * kGroupNodes] = p.rho0;
  F[kMidRhoOut * kGroupNodes] = p.rho_out;
  signal(flags, kProfileReady, round);
  const BlackHole b = black_hole(G.P, G.D, galaxy, m_bh, after_signal(y_spin), after_signal(r_bh), mg_s);
  F[kMidEffThin * kGroupNodes] = b.eff_thin;
  F[kMidEddCap * kGroupNodes] = b.edd_cap;
  F[kMidMdotSph * kGroupNodes] = b.mdot_sph;
  signal(flags, kAccretorReady, round);
  p.uo = after_signal(p.uo);
  F[kMidInvRMean * kGroupNodes] = hot_inv_mean_radius(T, p);
  signal(flags, kMeanRadiusReady, round);
  SpheroidShares q = spheroid_shares(G.P, G.D, ops, b, m_bh, after_signal(mg_s), ms_s, j_s, zg_s, galaxy.r);
  q.inv_mg = after_signal(q.inv_mg);
  q.inv_mt = after_signal(q.inv_mt);
  q.inv_m_bh = after_signal(q.inv_m_bh);
  double f[kNV];
#pragma unroll
  for (int v = 0; v < kNV; ++v) f[v] = 0.0;
  await(flags, kAccretionReady, round);
  spheroid_rates(G.P, G.D, T, b, q, F[kMidMdot * kGroupNodes], m_bh, mg_s, ms_s, j_s, zg_s, galaxy.r, f);
#pragma unroll
  for (int v = 0; v < kNV; ++v)
    if ((kSpheroidVars >> v) & 1u) X[(kXHalo + v) * kGroupNodes] = f[v];
}

// The time wave's share of this stage's derivative, after the next stage's
// time part.
__device__ __forceinline__ void time_wave_rhs(double* __restrict__ X, double* __restrict__ F,
                                              int* __restrict__ flags, int round) {
  await(flags, kCoolingFunctionReady, round);
  X[(kXHalo + GAL_V_HOT_ENERGY_RADIATED) * kGroupNodes] =
      radiated_energy(F[kMidLambda * kGroupNodes], F[kMidNhPerRho * kGroupNodes], F[kMidNallPerNh * kGroupNodes],
                      X[(kXState + GAL_V_HOT_MASS) * kGroupNodes], X[(kXState + GAL_V_HOT_OUTER_RADIUS) * kGroupNodes]);
}

__device__ __forceinline__ void cooling_wave_rhs(const GroupConstants& G, const double* __restrict__ tab,
                                                 const NodePar& np, double* __restrict__ X, double* __restrict__ F,
                                                 const double* __restrict__ time, int* __restrict__ flags, int round) {
  auto Y = [&](int v) { return X[(kXState + v) * kGroupNodes]; };
  const TimePart T = load_time_part(time);
  const double m_hot = Y(GAL_V_HOT_MASS), r_out = Y(GAL_V_HOT_OUTER_RADIUS), z_hot = Y(GAL_V_HOT_ABUNDANCES);
  const double j_hot = Y(GAL_V_HOT_ANGULAR_MOMENTUM), m_bh = Y(GAL_V_BH_MASS), y_spin = Y(GAL_V_BH_SPIN);
  const CoolingTime c = cooling_time(G.D, tab, G.C, T, m_hot, z_hot, r_out);
  F[kMidLambda * kGroupNodes] = c.lambda_cool;
  F[kMidNhPerRho * kGroupNodes] = c.nh_per_rho;
  F[kMidNallPerNh * kGroupNodes] = c.nall_per_nh;
  signal(flags, kCoolingFunctionReady, round);
  await(flags, kProfileReady, round);
  const double rho0 = F[kMidRho0 * kGroupNodes];
  HotAccretion s = hot_accretion(G.P, G.D, T, c, rho0, F[kMidRhoOut * kGroupNodes], m_hot, r_out, m_bh);
  s.bondi = after_signal(s.bondi);
  await(flags, kAccretorReady, round);
  const double eff_thin = F[kMidEffThin * kGroupNodes];
  accretion_rate(s, eff_thin, F[kMidEddCap * kGroupNodes], F[kMidMdotSph * kGroupNodes]);
  F[kMidMdot * kGroupNodes] = s.mdot;
  signal(flags, kAccretionReady, round);
  const double p_jet = jet_power(G.D, after_signal(s.mdot), m_bh, y_spin);
  double f[kNV];
#pragma unroll
  for (int v = 0; v < kNV; ++v) f[v] = 0.0;
  f[GAL_V_BH_MASS] += black_hole_growth(s.mdot, p_jet, eff_thin, m_bh);
  await(flags, kMeanRadiusReady, round);
  cooling_rates(G.P, np, T, s, p_jet, c.inv_m_hot, rho0, F[kMidInvRMean * kGroupNodes], m_hot, z_hot, j_hot, r_out,
                m_bh, f);
#pragma unroll
  for (int v = 0; v < kNV; ++v)
    if ((kCoolingVars >> v) & 1u) X[(kXHalo + v) * kGroupNodes] = f[v];
}

}  // namespace gal
