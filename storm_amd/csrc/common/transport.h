// Per-packet IMC transport on a Cartesian mesh in cell-local coordinates.
//
// One function, compiled for gfx950 (the transport kernels) and for the host
// (the bit-exact replay used by the tests), advances one packet through up to
// `max_segments` segments.  A segment is one call of the reference's
// RadiationIMC::step (radiation/RadiationIMC.hpp:1700-1881), counted like
// cellsStepsCounters (MonteCarloManagerSerial.hpp:302-303):
//   * in a random-walk cell, a random-walk step if the packet is deep enough
//     (tryRandomWalkStep, :1065-1276);
//   * else in a DDMC cell, a discrete-diffusion step (tryDDMCStep, :1415-1612);
//   * else analytic tracking: the distance to the nearest cell face, to the
//     next effective-scatter event and to census is compared, the packet
//     moves, its weight is attenuated by the continuous absorption factor, the
//     absorbed energy and the time-integrated radiation energy are tallied in
//     the cell, and the event is applied (face crossing with the manager's
//     cell move or boundary call, MonteCarloManagerSerial.hpp:318-357;
//     isotropic redirection; census).  Roulette below 1e-3 of the step's
//     starting weight (1e-4 in a random-walk step) deposits the rest.
//
// Layout decisions (MI355X): the position is the fraction of the cell width
// on each axis (u in [0,1]^3), so a face crossing sets one coordinate to 0 or
// 1 exactly instead of nudging by 1e-8 as the FP64 reference does; the
// direction is a unit vector; times are carried as path lengths in cm
// (time * c).  The Real type is float for the mixed engine (deterministic own
// math, fixed-point tallies) and double for the plain FP64 engine.
#pragma once

#include <stdint.h>
#include <math.h>
#include "constants.h"
#include "fixed.h"
#include "fpmath.h"
#include "hd.h"
#include "mathpolicy.h"
#include "philox.h"

namespace storm {

// Packed cell coordinates: i (12 bits) | j (10 bits) | k (10 bits).
STORM_HD uint32_t pack_ijk(uint32_t i, uint32_t j, uint32_t k) { return (i << 20) | (j << 10) | k; }
STORM_HD uint32_t ijk_i(uint32_t p) { return p >> 20; }
STORM_HD uint32_t ijk_j(uint32_t p) { return (p >> 10) & 0x3ffu; }
STORM_HD uint32_t ijk_k(uint32_t p) { return p & 0x3ffu; }

// Multigroup spectrum as seen by the transport (groups < 2: gray).  Photon
// energies are in keV.  A packet of energy E in cell c sees
//   sigma_a(c, E) = sigma_a(c, 1 keV) * max(E, e_lo)^(-nu_pow)
// (the cell table then holds f sigma_a(c, 1 keV) and (1-f) sigma_a(c, 1 keV))
// and re-emits after an effective scatter at an energy drawn from the cell's
// emission CDF: cdf[c*(groups+1) + g] over the group bounds, linear within a
// group (DensmoreOpacity::GetThermalEnergy, examples/densmore2012/DensmoreOpacity.hpp:66-77).
template <typename Real>
struct SpectrumView {
  int32_t groups;
  Real nu_pow;
  Real e_lo, e_hi;     // bounds[0], bounds[groups]
  const Real *bounds;  // groups + 1
  const Real *cdf;     // per cell, groups + 1, cdf[0] = 0 and cdf[groups] = 1
  const Real *sig_s;   // per cell scattering opacity (gray)
  int32_t eg;          // 1: tally the path integral per cell and group (withEgTimeAvg)
};

// RadiationOpacityModel::findGroup (radiation/RadiationOpacityModel.hpp:76-86):
// the first group whose upper bound lies above E, else the last.
template <typename Real>
STORM_HD int32_t group_of(Real e, const Real *bounds, int32_t groups) {
  int32_t lo = 0, hi = groups - 1;
  while (lo < hi) {
    const int32_t mid = (lo + hi) >> 1;
    if (e < bounds[mid + 1]) hi = mid;
    else lo = mid + 1;
  }
  return lo;
}

// The draw for the unbiased rounding of a per-group path integral: a hash of
// the packet, its stream position, the cell and the group.
STORM_HD uint32_t group_tally_draw(uint32_t id, uint32_t ctr, uint32_t cell, int32_t g) {
  uint32_t h = id * 0x85EBCA6Bu ^ (ctr + 0x2F1B9A3Du) * 0xC2B2AE35u ^ cell * 0x27D4EB2Du ^
               static_cast<uint32_t>(g) * 0x165667B1u;
  h ^= h >> 16;
  h *= 0x7FEB352Du;
  h ^= h >> 15;
  return h >> 8;
}

// Energy (keV) at the quantile `u` of a normalised group CDF, linear within
// the group (LinearInterpolation, utils/LinearInterpolation.hpp:17-42, of
// the CDF onto the bounds).
template <typename Real>
STORM_HD Real spectrum_quantile(const Real *cdf, const Real *bounds, int32_t groups, Real u) {
  // smallest i in [1, groups] with cdf[i] > u
  int32_t lo = 0, hi = groups;
  while (hi - lo > 1) {
    const int32_t mid = (lo + hi) >> 1;
    if (cdf[mid] > u) hi = mid;
    else lo = mid;
  }
  const Real c0 = cdf[hi - 1], c1 = cdf[hi];
  const Real b0 = bounds[hi - 1], b1 = bounds[hi];
  const Real t = c1 > c0 ? (u - c0) / (c1 - c0) : Real(0.5);
  const Real e = b0 + t * (b1 - b0);
  return e < b0 ? b0 : (e > b1 ? b1 : e);
}

// Mesh as seen by the transport: per-axis widths (cm), the fate of a packet
// at each box face (order x-, x+, y-, y+, z-, z+) and the spectrum.
template <typename Real>
struct MeshView {
  int32_t nx, ny, nz;
  uint32_t escape_mask;  // bit f set: box face f removes the packet (else it reflects)
  // the cell widths and their reciprocals, interleaved (width_pairs), axis
  // x then y then z: index i along axis a at width_at(m, a, i)
  const Real *width;
  SpectrumView<Real> spec;
};

// (width, 1 / width) of index i along axis a
template <typename Real>
STORM_HD const Real *width_at(const MeshView<Real> &m, int a, uint32_t i) {
  const uint32_t off = a == 0 ? 0u : (a == 1 ? static_cast<uint32_t>(m.nx) : static_cast<uint32_t>(m.nx + m.ny));
  return m.width + 2u * (off + i);
}

// Host: widths w[0..n) and their reciprocals, interleaved into out[0..2n).
// The reciprocal is the one IEEE division a segment would otherwise do on
// entering the cell, so the tracking is unchanged bit for bit.
template <typename Real>
inline void width_pairs(const Real *w, int n, Real *out) {
  for (int i = 0; i < n; ++i) {
    out[2 * i] = w[i];
    out[2 * i + 1] = Real(1) / w[i];
  }
}

template <typename Real>
STORM_HD uint32_t flat_cell(const MeshView<Real> &m, uint32_t ijk) {
  return (ijk_i(ijk) * static_cast<uint32_t>(m.ny) + ijk_j(ijk)) * static_cast<uint32_t>(m.nz) + ijk_k(ijk);
}

// Per-cell opacities used by a segment (cm^-1):
//   sig_abs = f * sigma_a              continuous absorption (weight attenuation)
//   sig_ev  = sigma_s + (1-f)*sigma_a  effective-scatter event opacity
//   inv_ev  = 1 / sig_ev (0 where sig_ev is 0), for the event distance
//   r_acc   no packet closer than this to a face of the cell takes a random
//           walk or a DDMC step (accel_radius; 0: it has to be tried)
// 16 bytes in the mixed engine: one load.
template <typename Real>
struct alignas(4 * sizeof(Real)) CellXS {
  Real sig_abs, sig_ev, inv_ev, r_acc;
};

template <typename Real>
STORM_HD CellXS<Real> make_xs(Real sig_abs, Real sig_ev) {
  CellXS<Real> x;
  x.sig_abs = sig_abs;
  x.sig_ev = sig_ev;
  x.inv_ev = sig_ev > Real(0) ? Real(1) / sig_ev : Real(0);
  x.r_acc = Real(0);
  return x;
}

// Per-cell data of the diffusion accelerations:
//   flags   bit 0 random-walk cell, bit 1 DDMC cell
//   sig_t   sigma_a + sigma_s (cm^-1); multigroup: the Planck mean of
//           sigma_a(E) + sigma_s over the diffusive groups (the walk's
//           particle threshold opacity)
//   rate    DDMC leak rate per face / c (cm^-1), order x-, x+, y-, y+, z-, z+
//   total   sum of rate
//   gcut    multigroup: the diffusive groups are 0 .. gcut-1
//   sig_d   opacity of the walk's diffusion coefficient, D = c / (3 sig_d)
//           (gray: sig_t; multigroup: the Planck-weighted harmonic mean of
//           sigma_a(E) + sigma_s over the diffusive groups)
//   sig_abs multigroup: f times the Planck mean of sigma_a(E) over the
//           diffusive groups, the continuous absorption during a walk
//   up_rate multigroup: (1 - f) sigma_a,mean (1 - gamma) (cm^-1), the rate of
//           re-emission above the diffusive groups, which ends a walk
//   e_cut   multigroup: lower bound (keV) of group gcut; packets at or above
//           it do not walk (+inf gray)
//   ddmc_sig_t  DDMC: sigma_P + sigma_s, the Planck-mean total opacity (the
//           particle threshold's opacity; equal to sig_t in a gray problem)
//   ddmc_abs    DDMC in a multigroup problem: f sigma_P, the continuous
//           absorption during a DDMC step (a gray step uses the cell's own);
//           with ddmc_multigroup_pgrw f sigma_A of the diffusive groups
//   ddmc_e_cut  DDMC with ddmc_multigroup_pgrw: lower bound (keV) of the
//           first non-diffusive group; packets at or above it take no DDMC
//           step (+inf otherwise)
// (precomputeRandomWalkData, radiation/RadiationIMC.hpp:983-1063;
// precomputeDDMCData without ddmcUseMultigroupPGRW, :1282-1351)
template <typename Real>
struct CellAccel {
  Real sig_t;
  Real total;
  Real rate[6];
  uint32_t flags;
  uint32_t gcut;
  Real sig_d;
  Real sig_abs;
  Real up_rate;
  Real e_cut;
  Real ddmc_sig_t;
  Real ddmc_abs;
  Real ddmc_e_cut;
};

// Random-walk tables (see random_walk.h) and the particle thresholds.
template <typename Real>
struct AccelView {
  const CellAccel<Real> *cell;  // null: no random walk and no DDMC in this problem
  const Real *rw;           // [rw::kAllSize]: the tables (rw::tables_at)
  Real rw_particle_tau;    // rwMinParticleOpticalDepth
  Real ddmc_particle_tau;  // ddmcMinParticleOpticalDepth
};

// CellXS::r_acc of a cell: both accelerations ask for a distance Ro to the
// nearest face with Ro sigma >= tau (sigma and tau the method's own), so none
// applies below the smaller tau / sigma of the methods the cell is flagged
// for.  Less 1e-5 of it, far above the rounding of the product that decides.
template <typename Real>
STORM_HD Real accel_radius(const CellAccel<Real> &a, Real rw_tau, Real ddmc_tau) {
  Real r = MathPolicy<Real>::inf();
  auto lower = [&r](Real tau, Real sigma) {
    const Real t = tau / sigma * Real(1 - 1e-5);
    if (!(t > Real(0))) r = Real(0);  // a threshold at or below 0, or no number: always try
    else r = t < r ? t : r;
  };
  if ((a.flags & 1u) && a.sig_t > Real(0)) lower(rw_tau, a.sig_t);
  if (a.flags & 2u) lower(ddmc_tau, a.ddmc_sig_t);
  return r;
}

template <typename Real>
struct Packet {
  Real u[3];      // position as a fraction of the cell width per axis
  Real s;         // path length left in the step, cm (= timeLeft * c)
  Real o[3];      // unit direction
  Real wmin;      // roulette threshold, 1e-3 of the weight at step start
  double w;       // weight, erg
  uint32_t ijk;   // packed cell coordinates
  uint32_t id;    // packet id within the step (keys the random stream)
  uint32_t ctr;   // Philox blocks consumed by transport so far
  uint32_t flags;
  Real nu;        // photon energy, keV (multigroup; 0 when gray)
};

// Scalars shared by every packet of a step.
struct StepConsts {
  uint64_t seed;
  uint32_t step;
  int32_t eq;      // energy quantum exponent, Q = 2^eq erg
  int32_t et;      // path-integral quantum exponent, 2^et erg*cm
};

enum TransportOutcome : int { kAlive = 0, kCensus = 1, kGone = 2, kEscaped = 3 };

}  // namespace storm

#include "random_walk.h"

namespace storm {

// ---------------------------------------------------------------- transport
// Component access by a runtime axis without indexing a local array (a
// runtime index into a register array would put it in scratch memory).
template <typename T>
STORM_HD T sel3(int a, T x, T y, T z) {
  return a == 0 ? x : (a == 1 ? y : z);
}
template <typename T>
STORM_HD void put3(int a, T &x, T &y, T &z, T v) {
  x = a == 0 ? v : x;
  y = a == 1 ? v : y;
  z = a == 2 ? v : z;
}

// Cell-local coordinates are fractions of the cell width.  A float moved by
// less than half a unit in its last place keeps its value, and near u = 1
// that unit is 2^-24 of the width: in an optically thick cell a collision
// flight is far shorter.  A packet lying on a face (after a reflection, say)
// would then stay pinned there, at distance 0 from the face, never eligible
// for the random walk, and with its time budget no longer decreasing either
// once a flight is below the budget's own unit: a history without end (the
// FP64 reference pins the same way once a flight is below the unit of its
// absolute coordinates).  So a packet on a face that moves inward by less
// than a unit is taken one unit inside (the smallest normal number above 0
// on the lower face), far below the cell size but enough for the random walk
// to take over in such a cell; elsewhere a sub-unit move of `delta` is taken
// as one whole unit with probability |delta| / unit (from 8 random bits
// `r8`), so that the expected move is exact.
STORM_HD float move_coord(float u, float n, float delta, uint32_t r8) {
  if (n != u || delta == 0.0f) return n;
  if (delta > 0.0f ? !(u < 1.0f) : !(u > 0.0f)) return n;
  if (u == 0.0f) return 1.17549435e-38f;
  if (u == 1.0f) return 0.99999994f;
  uint32_t b;
  __builtin_memcpy(&b, &u, sizeof(b));
  b = delta > 0.0f ? b + 1u : b - 1u;
  float next;
  __builtin_memcpy(&next, &b, sizeof(next));
  const float unit = delta > 0.0f ? next - u : u - next;
  const float p = (delta > 0.0f ? delta : -delta) / unit;
  return (static_cast<float>(r8) + 0.5f) * 0.00390625f < p ? next : u;
}

// The next representable number above a positive x.
STORM_HD float next_above(float x) {
  uint32_t b;
  __builtin_memcpy(&b, &x, sizeof(b));
  ++b;
  __builtin_memcpy(&x, &b, sizeof(x));
  return x;
}
STORM_HD double next_above(double x) {
  uint64_t b;
  __builtin_memcpy(&b, &x, sizeof(b));
  ++b;
  __builtin_memcpy(&x, &b, sizeof(x));
  return x;
}

// Sink interface (duck-typed):
//   visit(cell, dep_limbs, path_limbs, segments)  (Real = float) or
//   visit_fp(cell, dep, path, segments)           (Real = double): a cell visit ends
//   roulette(cell, weight)                          Real = float: weight rouletted into the material
//   escape_fx(cell, weight) / escape_fp(...)        the packet leaves the problem (mixed / FP64)
//   rw_step() / ddmc_step()                         acceleration counters
// The mixed engine tallies the path integral only in cells without
// absorption: elsewhere it equals the absorbed energy divided by f sigma_a
// (both are sums of w (1 - e^{-x}) over the same segments), which the
// postStep evaluates from the exact deposit tally.
//
// Tracker<Real, F> holds one packet's history between segments, so that a
// kernel can advance a packet one segment at a time and give an idle lane a
// new packet (transport_packet below runs a whole pass of one packet).
// F selects the code compiled in: kFeatAccel (random walk and DDMC) and
// kFeatMultigroup; a problem without them runs a leaner kernel with the same
// results.
//
// A segment is written so that what its three kinds of step (analytic, random
// walk, DDMC) and its ways to end a cell visit (face, census, roulette,
// escape) have in common stands once, outside the branches that differ: the
// lanes of a wavefront take different kinds, and a wavefront runs every branch
// that one of its lanes takes.  The transport is bound by these instructions
// (82% of the vector issue slots on the 64^3 cube; a history alone in its
// wavefront runs at its instruction count too), so the tail that closes a
// visit, the random numbers, the logarithm, the attenuation and the new
// direction are each in the code once.
enum : uint32_t { kFeatAccel = 1u, kFeatMultigroup = 2u, kFeatAll = 3u };

// Kinds of step, what ends a segment, and how it ends the visit of its cell.
enum : int { kStepAnalytic = 0, kStepWalk = 1, kStepDdmc = 2 };
enum : int { kEvFace = 0, kEvCollide = 1, kEvCensus = 2, kEvLeak = 3, kEvReemit = 4 };
enum : int { kEndNone = 0, kEndCross = 1, kEndCensus = 2, kEndRoulette = 3, kEndEscape = 4 };

// The part of a packet's history that does not depend on the mesh: weight,
// path integral, photon energy and the opacities of its cell.  In the mixed
// engine the weight is in quanta of the step (a power of two times erg, so
// every product and comparison rounds as it does in erg) and the weight the
// visit began with is the integer it is then.
template <typename Real, uint32_t F>
struct PacketState {
  using M = MathPolicy<Real>;
  static constexpr bool fixed_point = sizeof(Real) == 4;
  static constexpr bool multigroup = (F & kFeatMultigroup) != 0u;

  Real o0, o1, o2, s, wmin, nu;
  Real cell_sig_abs, cell_sig_ev, inv_sig_ev, r_acc;
  Real cell_sig_s, nu_fac;  // multigroup: the cell's scattering opacity, E^-nu_pow of the packet
  double w, path_int;
  double w_enter;    // FP64 engine: weight when the current cell visit began
  uint64_t n_enter;  // mixed engine: the same, in quanta
  uint32_t ctr, cell, visit_segs, id;
  int outcome;
  // per-group tally (multigroup with withEgTimeAvg): the packet's group and
  // the part of the visit's path integral already handed to it
  int32_t grp;
  double eg_mark;

  STORM_HD static bool is_mg(const SpectrumView<Real> &sp) { return multigroup && sp.groups >= 2; }
  STORM_HD static bool eg_track(const SpectrumView<Real> &sp) { return is_mg(sp) && sp.eg != 0; }

  STORM_HD void begin_packet(const Packet<Real> &p, const SpectrumView<Real> &sp, const StepConsts &k) {
    s = p.s;
    ctr = p.ctr;
    id = p.id;
    nu = p.nu;
    if constexpr (fixed_point) {
      const double q = fpm::pow2d(-k.eq);
      w = p.w * q;
      wmin = static_cast<Real>(static_cast<double>(p.wmin) * q);
      n_enter = fx::to_u64(floor(w));
    } else {
      w = p.w;
      wmin = p.wmin;
      w_enter = w;
    }
    grp = 0;
    eg_mark = 0.0;
    path_int = 0.0;  // sum of w * (1 - e^{-x}) / sig_abs over the visit, quanta (erg in FP64) times cm
    visit_segs = 0;
    outcome = kAlive;
    set_energy(sp);
  }

  // Writes the state back; a packet still alive closes its visit so that the
  // next pass starts clean.
  template <typename Sink>
  STORM_HD void end_packet(Packet<Real> &p, const SpectrumView<Real> &sp, const StepConsts &k, Sink &sink) {
    if (outcome == kAlive) end_visit(kEndCross, sp, k, sink);
    p.o[0] = o0;
    p.o[1] = o1;
    p.o[2] = o2;
    p.s = s;
    if constexpr (fixed_point) {
      const double q = fpm::pow2d(k.eq);
      p.w = w * q;
      p.wmin = static_cast<Real>(static_cast<double>(wmin) * q);
    } else {
      p.w = w;
      p.wmin = wmin;
    }
    p.ctr = ctr;
    p.id = id;
    p.nu = nu;
  }

  // The mixed engine tallies the path integral only where postStep cannot
  // derive it from the deposit (gray cells without absorption).
  STORM_HD bool derive_pint(const SpectrumView<Real> &sp) const {
    return fixed_point && !is_mg(sp) && cell_sig_abs > Real(0);
  }

  // Hands the path integral since the last call to the packet's group
  // (RadiationIMC.hpp:1166-1173, 1485-1492, 1802-1809): at the end of each
  // visit and before the photon energy changes.
  template <typename Sink>
  STORM_HD void group_split(const SpectrumView<Real> &sp, const StepConsts &k, Sink &sink) {
    if constexpr (multigroup) {
      if (eg_track(sp)) {
        double v = path_int - eg_mark;
        if constexpr (fixed_point) v *= fpm::pow2d(k.eq);
        if (v > 0.0) sink.group_path(cell, grp, v, k, group_tally_draw(id, ctr, cell, grp));
        eg_mark = path_int;
      }
    }
  }

  // Closes the visit of the current cell: tallies its deposit, path integral
  // and segments and applies what `how` says to the weight.  The weight goes
  // on as a multiple of the quantum; at the end of the step it does so in both
  // engines, so that population control can work in exact integers.
  template <typename Sink>
  STORM_HD void end_visit(int how, const SpectrumView<Real> &sp, const StepConsts &k, Sink &sink) {
    group_split(sp, k, sink);
    if constexpr (multigroup) eg_mark = 0.0;
    if constexpr (fixed_point) {
      // roulette cuts the weight to whole quanta, the rest round it
      const uint64_t n = fx::carry_round_q(w, how == kEndRoulette ? 0u : n_enter, fx::carry_draw(id, ctr, cell));
      fx::Limbs e{0u, 0u};
      if (!derive_pint(sp)) {
        // the rounding draw: a hash of the packet, its stream position and
        // the cell (no random-stream draw, so the history is unchanged)
        uint32_t h = id * 0x9E3779B1u ^ (ctr + 0x7F4A7C15u) * 0x85EBCA77u ^ cell * 0xC2B2AE3Du;
        h ^= h >> 15;
        h *= 0x2C1B3C6Du;
        h ^= h >> 12;
        const double y = path_int * fpm::pow2d(k.eq - k.et), fl = floor(y);
        const double u = static_cast<double>(h >> 8) * 0x1p-24;
        e = fx::limbs_of_value(fx::to_u64(u < y - fl ? fl + 1.0 : fl));
      }
      sink.visit(cell, fx::limbs_of_value(n_enter - n), e, visit_segs);
      n_enter = n;
      if (how == kEndRoulette) sink.roulette(cell, w * fpm::pow2d(k.eq));
      if (how == kEndEscape) sink.escape_fx(cell, w * fpm::pow2d(k.eq));
      if (how == kEndRoulette || how == kEndEscape) w = 0.0;
    } else {
      if (how == kEndCensus) w = fx::carry_round(w, w_enter, k.eq, id, ctr, cell);
      sink.visit_fp(cell, w_enter - (how == kEndRoulette ? 0.0 : w), path_int, visit_segs);
      if (how == kEndEscape) sink.escape_fp(cell, w);
      if (how == kEndRoulette || how == kEndEscape) w = 0.0;
      w_enter = w;
    }
    if (how == kEndCensus) outcome = kCensus;
    if (how == kEndRoulette) outcome = kGone;
    if (how == kEndEscape) outcome = kEscaped;
    visit_segs = 0;
    path_int = 0.0;
  }

  // multigroup: what depends on the photon energy alone
  STORM_HD void set_energy(const SpectrumView<Real> &sp) {
    if constexpr (multigroup) {
      if (sp.groups >= 2) {
        // clampFrequencyToBounds (RadiationIMC.hpp:868-872) and E^-nu_pow
        const Real e = nu < sp.e_lo ? sp.e_lo : (nu > sp.e_hi ? sp.e_hi : nu);
        nu_fac = M::exp(-sp.nu_pow * M::log(e));
        if (sp.eg) grp = group_of<Real>(e, sp.bounds, sp.groups);
      }
    }
  }

  // from the cell's gray opacities `x` and scattering opacity `sig_s`
  // (multigroup only)
  STORM_HD void set_opacity(const SpectrumView<Real> &sp, const CellXS<Real> &x, Real sig_s) {
    cell_sig_abs = x.sig_abs;
    cell_sig_ev = x.sig_ev;
    inv_sig_ev = x.inv_ev;
    r_acc = x.r_acc;
    if constexpr (multigroup) {
      cell_sig_s = Real(0);
      if (sp.groups >= 2) {
        cell_sig_s = sig_s;
        cell_sig_abs = x.sig_abs * nu_fac;
        cell_sig_ev = cell_sig_s + x.sig_ev * nu_fac;
        inv_sig_ev = cell_sig_ev > Real(0) ? M::recip_any(cell_sig_ev) : Real(0);
      }
    }
  }

  // continuous absorption over a path d (cm); `tally_free` adds w * d to the
  // path integral when nothing is absorbed (the analytic step and DDMC do,
  // the random-walk step does not, RadiationIMC.hpp:1163-1165)
  STORM_HD void absorb(const SpectrumView<Real> &sp, Real sig_abs, Real d, bool tally_free) {
    const Real xabs = sig_abs * d;
    const Real frac = -M::expm1_neg(-xabs);
    const double w0 = w;
    w = w0 - w0 * static_cast<double>(frac);
    // the mixed engine derives the path integral of absorbing gray cells
    // from their deposit (see end_visit)
    if (derive_pint(sp)) return;
    if (xabs >= Real(1e-12)) {
      path_int += w0 * static_cast<double>(frac / sig_abs);
    } else if (tally_free) {
      path_int += w0 * static_cast<double>(d);
    } else if (sig_abs > Real(0)) {
      path_int += w0 * static_cast<double>(frac / sig_abs);
    }
  }

  // A new photon energy from the cell's emission spectrum: over all of it
  // after an effective scatter (RadiationIMC.hpp:1843-1852; gcut = 0), above
  // the diffusive groups 0 .. gcut-1 where a walk ends by re-emission
  // (:1237-1252).
  STORM_HD void new_energy(const SpectrumView<Real> &sp, Real u, uint32_t gcut) {
    const int32_t G = sp.groups;
    const Real *cdfc = sp.cdf + static_cast<size_t>(cell) * static_cast<size_t>(G + 1);
    if (gcut) {
      const Real lo = cdfc[gcut];
      if (lo < Real(1)) {
        nu = spectrum_quantile<Real>(cdfc, sp.bounds, G, lo + u * (Real(1) - lo));
      } else {
        nu = next_above(sp.bounds[gcut]);
      }
      nu = nu < sp.e_lo ? sp.e_lo : (nu > sp.e_hi ? sp.e_hi : nu);
    } else {
      nu = spectrum_quantile<Real>(cdfc, sp.bounds, G, u);
    }
    set_energy(sp);
  }
};

template <typename Real, uint32_t F = kFeatAll>
struct Tracker : PacketState<Real, F> {
  using Base = PacketState<Real, F>;
  using M = MathPolicy<Real>;
  using Base::fixed_point;
  using Base::multigroup;
  using Base::o0;
  using Base::o1;
  using Base::o2;
  using Base::s;
  using Base::w;
  using Base::wmin;
  using Base::nu;
  using Base::ctr;
  using Base::id;
  using Base::cell;
  using Base::outcome;
  using Base::cell_sig_abs;
  using Base::cell_sig_ev;
  using Base::cell_sig_s;
  using Base::inv_sig_ev;

  Real u0, u1, u2;
  Real io0, io1, io2;  // 1/|o| per axis (+inf along an axis the packet does not move on)
  // the current cell's widths and their reciprocals
  Real cw0, cw1, cw2, icw0, icw1, icw2;
  uint32_t ijk;

  STORM_HD void begin(const Packet<Real> &p, const MeshView<Real> &m, const CellXS<Real> *xs, const StepConsts &k) {
    u0 = p.u[0];
    u1 = p.u[1];
    u2 = p.u[2];
    o0 = p.o[0];
    o1 = p.o[1];
    o2 = p.o[2];
    io0 = o0 != Real(0) ? Real(1) / (o0 > Real(0) ? o0 : -o0) : M::inf();
    io1 = o1 != Real(0) ? Real(1) / (o1 > Real(0) ? o1 : -o1) : M::inf();
    io2 = o2 != Real(0) ? Real(1) / (o2 > Real(0) ? o2 : -o2) : M::inf();
    ijk = p.ijk;
    cell = flat_cell(m, ijk);
    const Real *p0 = width_at(m, 0, ijk_i(ijk));
    const Real *p1 = width_at(m, 1, ijk_j(ijk));
    const Real *p2 = width_at(m, 2, ijk_k(ijk));
    cw0 = p0[0];
    icw0 = p0[1];
    cw1 = p1[0];
    icw1 = p1[1];
    cw2 = p2[0];
    icw2 = p2[1];
    this->begin_packet(p, m.spec, k);
    this->set_opacity(m.spec, xs[cell], Base::is_mg(m.spec) ? m.spec.sig_s[cell] : Real(0));
  }

  template <typename Sink>
  STORM_HD void end(Packet<Real> &p, const MeshView<Real> &m, const StepConsts &k, Sink &sink) {
    this->end_packet(p, m.spec, k, sink);
    p.u[0] = u0;
    p.u[1] = u1;
    p.u[2] = u2;
    p.ijk = ijk;
  }

  // One segment of the history (a random-walk step, a DDMC step or an
  // analytic step to the next face, scatter or census event); returns the
  // outcome, kAlive while the packet goes on.
  template <typename Sink>
  STORM_HD int segment(const MeshView<Real> &m, const CellXS<Real> *xs, const AccelView<Real> &acc,
                       const StepConsts &k, Sink &sink) {
    const PacketStream rs = PacketStream::make(k.seed, id, k.step, kTagTransport);
    const bool mg = Base::is_mg(m.spec);
    ++this->visit_segs;

    // ---------------- which kind of step
    // A cell's r_acc is a radius below which neither acceleration applies
    // (+inf in a cell without them), so that a packet near a face reads
    // nothing of its cell's acceleration data, and one in a cell without them
    // does not work out its distance either (in the FP64 engine 20 of 470
    // vector instructions a segment, 5% of the transport of 1-D slabs of thin
    // cells: 1.46 against 1.39 ms for 2.9e7 segments in passes).
    int step = kStepAnalytic;
    Real Ro = Real(0);
    if constexpr ((F & kFeatAccel) != 0u) {
      if (acc.cell && this->r_acc < M::inf()) {
        // distance to the nearest face (computeMinDistanceToFaces, :956-969)
        const Real a0 = u0 * cw0, b0 = (Real(1) - u0) * cw0;
        const Real a1 = u1 * cw1, b1 = (Real(1) - u1) * cw1;
        const Real a2 = u2 * cw2, b2 = (Real(1) - u2) * cw2;
        const Real m0 = a0 < b0 ? a0 : b0, m1 = a1 < b1 ? a1 : b1, m2 = a2 < b2 ? a2 : b2;
        Ro = m0 < m1 ? m0 : m1;
        Ro = m2 < Ro ? m2 : Ro;
        if (Ro >= this->r_acc) {
          const CellAccel<Real> &ca = acc.cell[cell];
          // multigroup: the partial-gray walk, for packets in the diffusive groups only (:1094-1114)
          if ((ca.flags & 1u) && (!mg || nu < ca.e_cut) && Ro > Real(0) && ca.sig_t > Real(0) &&
              Ro * ca.sig_t >= acc.rw_particle_tau)
            step = kStepWalk;
          else if ((ca.flags & 2u) && ca.total > Real(0) && Ro * ca.ddmc_sig_t >= acc.ddmc_particle_tau &&
                   (!multigroup || nu < ca.ddmc_e_cut))
            step = kStepDdmc;
        }
      }
    }

    // ---------------- analytic: the nearest face along the direction (+inf
    // along an axis the packet does not move on); ties go to the lower axis
    int fax = 0;
    bool up = false, outside = false;
    Real d = Real(0), nw = Real(0), niw = Real(0), nsig_s = Real(0);
    CellXS<Real> nxs{};
    if (step == kStepAnalytic) {
      auto face_dist = [](Real ua, Real oa, Real wa, Real ioa) {
        Real frac = oa > Real(0) ? (Real(1) - ua) : ua;
        Real t = frac * wa * ioa;
        return oa != Real(0) ? t : M::inf();
      };
      const Real d0 = face_dist(u0, o0, cw0, io0), d1 = face_dist(u1, o1, cw1, io1),
                 d2 = face_dist(u2, o2, cw2, io2);
      int sax = 1;
      Real dsecond = d1;
      d = d0;
      if (d1 < d0) {
        fax = 1;
        sax = 0;
        d = d1;
        dsecond = d0;
      }
      if (d2 < d) {
        sax = fax;
        dsecond = d;
        fax = 2;
        d = d2;
      } else if (d2 < dsecond) {
        sax = 2;
        dsecond = d2;
      }
      if constexpr (fixed_point) {
        // Two faces within 1e-6 of each other along the path (an edge or corner
        // crossing): decide which one is hit first in FP64.
        if (dsecond < M::inf() && dsecond - d <= Real(1e-6) * dsecond) {
          auto dist64 = [&](int a) {
            double oa = static_cast<double>(sel3(a, o0, o1, o2));
            double ua = static_cast<double>(sel3(a, u0, u1, u2));
            double fr = oa > 0.0 ? (1.0 - ua) : ua;
            return fr * static_cast<double>(sel3(a, cw0, cw1, cw2)) / (oa > 0.0 ? oa : -oa);
          };
          double dA = dist64(fax), dB = dist64(sax);
          if (dB < dA) {
            fax = sax;
            d = static_cast<Real>(dB);
          }
        }
      }
      up = sel3(fax, o0, o1, o2) > Real(0);
      // The neighbour across it (this cell again when the face is on the box
      // boundary): its data is loaded now and used only if the segment ends on
      // that face, so that the load latency overlaps the random numbers and
      // the attenuation below.
      outside = load_neighbour(fax, up, m, xs, nxs, nw, niw, nsig_s);
    }

    // ---------------- random numbers: one Philox block, block ctr (two for a
    // random-walk step and a multigroup re-emission)
    Philox4 r = rs.block(ctr++);
    const Real xi = M::uniform(r.v[0]);
    // -ln xi, the free flight of the analytic and DDMC steps; the walk's leak
    // time inverts -ln(1 - xi)
    const Real nlog = -M::log_unit(step == kStepWalk ? Real(1) - xi : xi);

    // ---------------- the event (d: its distance)
    int ev = kEvFace;
    Real sig_abs = cell_sig_abs;
    Philox4 r2{};  // of a walk, its second block
    if (step == kStepAnalytic) {
      // Event: face < scatter < census on ties, as the reference's min_element.
      const Real dcol = cell_sig_ev > Real(0) ? nlog * inv_sig_ev : M::inf();
      if (dcol < d) {
        ev = kEvCollide;
        d = dcol;
      }
    } else if ((F & kFeatAccel) != 0u && step == kStepWalk) {
      // random-walk step (tryRandomWalkStep)
      const CellAccel<Real> &ca = acc.cell[cell];
      r2 = rs.block(ctr++);
      const Real tauLeak = rw::sample_leak_time<Real>(rw::tables_at(acc.rw), xi, nlog);
      // tLeak = tau Ro^2 / D with D = c / (3 sig_d): as a path, tau Ro^2 3 sig_d
      d = tauLeak * Ro * Ro * (Real(3) * (mg ? ca.sig_d : ca.sig_t));
      ev = kEvLeak;
      if (mg) {
        sig_abs = ca.sig_abs;
        // re-emission above the diffusive groups (:1126-1131); leak, census,
        // upscatter, ties in that order (:1133-1152)
        if (ca.up_rate > Real(0)) {
          const Real sUp = (-M::log(M::uniform(r2.v[2]))) / ca.up_rate;
          if (sUp < d && sUp < s) {
            ev = kEvReemit;
            d = sUp;
          }
        }
      }
    } else if constexpr ((F & kFeatAccel) != 0u) {
      // DDMC step (tryDDMCStep; in a multigroup problem with the Planck-mean
      // data and the photon energy kept, as the reference does without
      // ddmcUseMultigroupPGRW)
      const CellAccel<Real> &ca = acc.cell[cell];
      d = nlog / ca.total;
      ev = kEvLeak;
      if constexpr (multigroup) sig_abs = ca.ddmc_abs;
    }
    // census: before a face or a scatter (s < d), before a walk's leak (s < d),
    // or with a DDMC leak (s <= d)
    if (s < d || (step == kStepDdmc && s == d)) {
      ev = kEvCensus;
      d = s;
    }

    this->absorb(m.spec, sig_abs, d, step != kStepWalk);
    s = ev == kEvCensus ? Real(0) : s - d;
    if (s < Real(0)) s = Real(0);
    if constexpr ((F & kFeatAccel) != 0u) {
      if (step == kStepWalk) sink.rw_step();
      if (step == kStepDdmc) sink.ddmc_step();
    }

    // ---------------- roulette (RadiationIMC.hpp:1812-1820): the remaining
    // weight goes to the material
    int end = ev == kEvCensus ? kEndCensus : kEndNone;
    bool turn = false;
    if (w < static_cast<double>(step == kStepWalk ? wmin * Real(0.1) : wmin)) {
      end = kEndRoulette;
    } else if (step == kStepAnalytic) {
      // Move (the face axis is set exactly).
      const Real m0 = o0 * d * icw0, m1 = o1 * d * icw1, m2 = o2 * d * icw2;
      Real n0 = u0 + m0, n1 = u1 + m1, n2 = u2 + m2;
      n0 = n0 < Real(0) ? Real(0) : (n0 > Real(1) ? Real(1) : n0);
      n1 = n1 < Real(0) ? Real(0) : (n1 > Real(1) ? Real(1) : n1);
      n2 = n2 < Real(0) ? Real(0) : (n2 > Real(1) ? Real(1) : n2);
      if constexpr (fixed_point) {
        if (n0 == u0 || n1 == u1 || n2 == u2) {
          // the low 8 bits of these words are not used by the uniforms
          n0 = move_coord(u0, n0, m0, r.v[1] & 0xffu);
          n1 = move_coord(u1, n1, m1, r.v[2] & 0xffu);
          n2 = move_coord(u2, n2, m2, r.v[3] & 0xffu);
        }
      }
      u0 = n0;
      u1 = n1;
      u2 = n2;
      if (ev == kEvCollide) {
        // scatter: isotropic redirection (RadiationIMC.hpp:1827-1874)
        turn = true;
        // an effective (absorption + re-emission) scatter takes a new energy,
        // an elastic one (probability sigma_s / event opacity) keeps it
        if (mg && !(M::uniform(r.v[1]) * cell_sig_ev < cell_sig_s)) ev = kEvReemit;
      } else if (ev == kEvFace) {
        // on the neighbour's side of the face, or on this cell's own
        put3<Real>(fax, u0, u1, u2, up != outside ? Real(0) : Real(1));
        end = kEndCross;
        if (outside) {
          if ((m.escape_mask >> (2 * fax + (up ? 1 : 0))) & 1u) {
            end = kEndEscape;  // REMOVE: the weight leaves the problem
          } else {
            // specular reflection on the box face (BoundaryCondition.hpp:87-108)
            end = kEndNone;
            put3<Real>(fax, o0, o1, o2, -sel3(fax, o0, o1, o2));
          }
        }
      }
    } else if ((F & kFeatAccel) != 0u && step == kStepWalk) {
      // new position on the sphere (leak) or inside it (census)
      Real dir[3];
      isotropic_dir<Real>(M::uniform(r.v[1]), M::uniform(r.v[2]), dir);
      Real disp = Ro;
      if (ev != kEvLeak) {
        const Real sig_d = mg ? acc.cell[cell].sig_d : acc.cell[cell].sig_t;
        const Real tauPos = d / (Real(3) * sig_d * Ro * Ro);
        disp = Ro * rw::sample_radius<Real>(rw::tables_at(acc.rw), tauPos, M::uniform(r.v[3]));
      }
      if (disp > Ro) disp = Ro;
      const Real c0 = u0, c1 = u1, c2 = u2;
      // nudge toward the cell centre (RadiationIMC.hpp:1214-1215)
      Real n0 = (c0 + disp * dir[0] * icw0) * Real(1 - 1e-6) + Real(1e-6) * Real(0.5);
      Real n1 = (c1 + disp * dir[1] * icw1) * Real(1 - 1e-6) + Real(1e-6) * Real(0.5);
      Real n2 = (c2 + disp * dir[2] * icw2) * Real(1 - 1e-6) + Real(1e-6) * Real(0.5);
      for (int guard = 0; guard < 2000; ++guard) {
        bool inside = n0 >= Real(0) && n0 <= Real(1) && n1 >= Real(0) && n1 <= Real(1) && n2 >= Real(0) &&
                      n2 <= Real(1);
        if (inside) break;
        disp = disp * Real(0.99);
        n0 = c0 + disp * dir[0] * icw0;
        n1 = c1 + disp * dir[1] * icw1;
        n2 = c2 + disp * dir[2] * icw2;
      }
      u0 = n0 < Real(0) ? Real(0) : (n0 > Real(1) ? Real(1) : n0);
      u1 = n1 < Real(0) ? Real(0) : (n1 > Real(1) ? Real(1) : n1);
      u2 = n2 < Real(0) ? Real(0) : (n2 > Real(1) ? Real(1) : n2);
      turn = true;
      r.v[2] = r2.v[0];
      r.v[3] = r2.v[1];
    } else if constexpr ((F & kFeatAccel) != 0u) {
      if (ev == kEvLeak) {
        // DDMC leak through a face chosen in proportion to its rate
        const CellAccel<Real> &ca = acc.cell[cell];
        Real pick = M::uniform(r.v[1]) * ca.total;
        int face = -1, lastf = -1;
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
        for (int f = 0; f < 6; ++f) {
          if (ca.rate[f] > Real(0)) {
            lastf = f;
            pick -= ca.rate[f];
            if (face < 0 && pick <= Real(0)) face = f;
          }
        }
        if (face < 0) face = lastf;
        fax = face >> 1;
        up = (face & 1) != 0;
        // placed at the face centroid (:1588), in the neighbour
        u0 = u1 = u2 = Real(0.5);
        put3<Real>(fax, u0, u1, u2, up ? Real(0) : Real(1));
        turn = true;
        end = kEndCross;
        load_neighbour(fax, up, m, xs, nxs, nw, niw, nsig_s);
      }
    }

    // ---------------- new direction: isotropic about z, or (a DDMC leak)
    // mu = sqrt(U) about the outward normal, basis as in :1565-1586
    if (turn) {
      const bool ddmc = (F & kFeatAccel) != 0u && step == kStepDdmc;
      const Real ua = M::uniform(r.v[2]), ub = M::uniform(r.v[3]);
      const Real mu = ddmc ? M::sqrt_unit(ua) : Real(2) * ua - Real(1);
      const Real st2 = Real(1) - mu * mu;
      const Real st = M::sqrt_unit(st2 > Real(0) ? st2 : Real(0));
      Real sp, cp;
      M::sincos2pi(ub, sp, cp);
      const Real x = st * cp, y = st * sp;
      o0 = x;
      o1 = y;
      o2 = mu;
      if (ddmc) {
        const Real n = up ? mu : -mu, t = up ? y : -y;
        if (fax == 0) {          // e1 = y, e2 = n x y = sg z
          o0 = n;
          o1 = x;
          o2 = t;
        } else if (fax == 1) {   // e1 = x, e2 = n x x = -sg z
          o1 = n;
          o2 = -t;
        } else {                 // e1 = x, e2 = n x x = sg y
          o1 = t;
          o2 = n;
        }
      }
      // (a component is 0 or at least 2^-40: no subnormal reciprocal)
      io0 = o0 != Real(0) ? M::recip(o0 > Real(0) ? o0 : -o0) : M::inf();
      io1 = o1 != Real(0) ? M::recip(o1 > Real(0) ? o1 : -o1) : M::inf();
      io2 = o2 != Real(0) ? M::recip(o2 > Real(0) ? o2 : -o2) : M::inf();
    }
    if constexpr (multigroup) {
      if (ev == kEvReemit && end == kEndNone) {
        this->group_split(m.spec, k, sink);
        const bool walk = (F & kFeatAccel) != 0u && step == kStepWalk;
        // a walk's draw is in its second block, a scatter takes another block
        const Philox4 re = rs.block(walk ? ctr - 1u : ctr);
        if (!walk) ++ctr;
        this->new_energy(m.spec, M::uniform(walk ? re.v[3] : re.v[0]), walk ? acc.cell[cell].gcut : 0u);
        this->set_opacity(m.spec, xs[cell], m.spec.sig_s[cell]);
      }
    }

    // ---------------- the visit's end
    if (end != kEndNone) {
      this->end_visit(end, m.spec, k, sink);
      if (end == kEndCross) {
        neighbour(fax, up, m, cell, ijk);
        put3<Real>(fax, cw0, cw1, cw2, nw);
        put3<Real>(fax, icw0, icw1, icw2, niw);
        this->set_opacity(m.spec, nxs, nsig_s);
      }
    }
    return outcome;
  }

  STORM_HD static uint32_t axis_index(int a, uint32_t code) {
    return sel3<uint32_t>(a, ijk_i(code), ijk_j(code), ijk_k(code));
  }
  // whether face `fax`/`up` of the current cell is on the box boundary
  STORM_HD bool on_box(int fax, bool up, const MeshView<Real> &m) const {
    const uint32_t n = static_cast<uint32_t>(sel3<int32_t>(fax, m.nx, m.ny, m.nz));
    return axis_index(fax, ijk) == (up ? n - 1u : 0u);
  }
  // moves the index `c` and the packed coordinates `code` of a cell across its face
  STORM_HD static void neighbour(int fax, bool up, const MeshView<Real> &m, uint32_t &c, uint32_t &code) {
    const uint32_t snz = static_cast<uint32_t>(m.nz);
    const uint32_t cstride = sel3<uint32_t>(fax, static_cast<uint32_t>(m.ny) * snz, snz, 1u);
    const uint32_t istride = sel3<uint32_t>(fax, 1u << 20, 1u << 10, 1u);
    c = up ? c + cstride : c - cstride;
    code = up ? code + istride : code - istride;
  }
  // the data of the cell across face `fax`/`up` (of this one where the face
  // is on the box): opacities, and width and its reciprocal along the axis.
  // Returns whether the face is on the box.
  STORM_HD bool load_neighbour(int fax, bool up, const MeshView<Real> &m, const CellXS<Real> *xs, CellXS<Real> &nxs,
                               Real &nw, Real &niw, Real &nsig_s) const {
    uint32_t c = cell, code = ijk;
    neighbour(fax, up, m, c, code);
    const bool out = on_box(fax, up, m);
    c = out ? cell : c;
    code = out ? ijk : code;
    nxs = xs[c];
    const Real *nwp = width_at(m, fax, axis_index(fax, code));
    nw = nwp[0];
    niw = nwp[1];
    if (Base::is_mg(m.spec)) nsig_s = m.spec.sig_s[c];
    return out;
  }
};

// The tracker of a mesh type (the polyhedral mesh's is in unstructured.h).
template <typename Real, uint32_t F, typename MeshT>
struct TrackerOf {
  using type = Tracker<Real, F>;
};

// One transport pass of a packet: at most `max_segments` segments, then the
// packet is written back (alive, in census, absorbed or escaped).
template <typename Real, uint32_t F = kFeatAll, typename Sink>
STORM_HD int transport_packet(Packet<Real> &p, const MeshView<Real> &m, const CellXS<Real> *xs,
                              const AccelView<Real> &acc, const StepConsts &k, int max_segments, Sink &sink) {
  Tracker<Real, F> t;
  t.begin(p, m, xs, k);
  for (int seg = 0; seg < max_segments && t.outcome == kAlive; ++seg) t.segment(m, xs, acc, k, sink);
  t.end(p, m, k, sink);
  return t.outcome;
}

}  // namespace storm
