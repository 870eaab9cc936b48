// Per-packet IMC transport on a mesh of convex polyhedral cells (a Voronoi
// tessellation, or any mesh flattened to per-cell face tables), shared by
// the gfx950 kernels and the CPU replay.
//
// The physics of a segment is the Cartesian tracker's (transport.h):
// RadiationIMC::step (radiation/RadiationIMC.hpp:1700-1881), the random walk
// (tryRandomWalkStep, :1065-1276) and DDMC (tryDDMCStep, :1415-1612).  What
// changes is the geometry, which follows the reference's general-face code:
//   * distance to the nearest face: the smallest non-negative
//     (d_f - n_f . x) / (n_f . o) over the faces moving outward
//     (Particle::distanceToNearestFace, particle/Particle.hpp:188-279);
//   * the random walk's sphere radius: the smallest plane distance
//     d_f - n_f . x (computeMinDistanceToFaces, RadiationIMC.hpp:956-969);
//     after a walk the position is nudged towards the mesh point by 1e-6
//     and the displacement shrunk by 0.99 while outside a face (:1211-1228);
//   * a DDMC leak through face f lands on the face centroid with
//     mu = sqrt(U) about the outward normal in the basis of :1561-1586;
//   * a box face removes or reflects the packet (escape mask per side).
//
// Layout (MI355X): a packet's position is kept relative to its cell's mesh
// point (the Voronoi generator), so FP32 carries it to ~1e-7 of the cell
// size; crossing a face adds the face's frame shift (mesh point of the cell
// minus that of the neighbour).  Each face is 16 bytes of plane in FP32
// (normal, offset in the cell's frame) and 32 of link (neighbour and its
// faces, frame shift).
#pragma once

#include <stdint.h>
#include <math.h>
#include "hd.h"
#include "transport.h"

namespace storm {

template <typename Real>
struct UFace {
  Real n[3];     // outward unit normal
  Real d;        // plane offset in the cell's frame: n . x = d on the face
  int32_t nbr;   // neighbour cell, or -1 - box side (x-, x+, y-, y+, z-, z+)
  Real sh[3];    // mesh point of this cell minus that of the neighbour (0 on the box)
};

// The transport's two halves of a face: the plane, which every segment reads
// for every face of its cell, and what only the face it leaves through needs,
// with the neighbour's own planes [pbeg, pend) so that they are read without
// looking them up in between.  A cell's planes are filled up to a multiple of
// kFaceBatch with planes that nothing ever reaches (n = 0, d = +inf), so that
// they are read and tried kFaceBatch at a time with no test for the last one;
// links stand in the same places.
constexpr uint32_t kFaceBatch = 3;
template <typename Real>
struct alignas(4 * sizeof(Real)) UPlane {
  Real n[3], d;
};
template <typename Real>
struct alignas(16) ULink {
  int32_t nbr;
  uint32_t pbeg, pend;
  Real sh[3];
};

template <typename Real>
struct UMeshView {
  uint32_t ncells;
  uint32_t escape_mask;            // bit s: box side s removes the packet (else it reflects)
  const uint32_t *face_start;      // ncells + 1
  const uint32_t *plane_start;     // ncells + 1
  const UPlane<Real> *plane;       // per face, filled up (kFaceBatch)
  const ULink<Real> *link;         // per plane
  uint32_t tame;                   // 1: every |d| lies in [2^-30, 2^50] (nearest_face)
  const Real *face_centroid;       // 3 per face, in the cell's frame (DDMC leaks)
  const Real *ddmc_rate;           // per face, leak rate / c (cm^-1); null without DDMC
  SpectrumView<Real> spec;
};

// A tetrahedron of a cell's fan decomposition: the mesh point (the frame's
// origin) and a triangle of a face fan, a, b, c in the cell's frame; `cum`
// the cell's cumulative volume fraction up to and including it.
template <typename Real>
struct UTet {
  Real cum;
  Real a[3], b[3], c[3];
};

// A triangle of a source face's fan, vertices in the cell's frame; `cum` the
// face's cumulative area fraction.
template <typename Real>
struct UTri {
  Real cum;
  Real a[3], b[3], c[3];
};

// A boundary source face: its cell, its triangles and its packets
// [first, first + count) of the step's boundary packets.
struct USource {
  uint32_t cell;
  uint32_t tri_start, tri_count;
  uint32_t first, count;
  int32_t xhi;  // 1: an x+ face (packets enter along -x)
};

// Stochastic rounding of a sub-unit move of an absolute coordinate: when
// x + delta rounds back to x, take one unit in the direction of delta with
// probability |delta| / unit (8 random bits), so the expected move is exact
// and a packet resting on a face of a very opaque cell leaves it.
STORM_HD float ulp_step(float x, bool upward) {
  if (x == 0.0f) return upward ? 1.17549435e-38f : -1.17549435e-38f;  // the smallest normal number
  uint32_t b;
  __builtin_memcpy(&b, &x, sizeof(b));
  const bool positive = (b >> 31) == 0u;
  b = positive == upward ? b + 1u : b - 1u;
  float y;
  __builtin_memcpy(&y, &b, sizeof(y));
  return y;
}
STORM_HD float umove_coord(float x, float nx, float delta, uint32_t r8) {
  if (nx != x || delta == 0.0f) return nx;
  const float up = ulp_step(x, delta > 0.0f);
  const float unit = delta > 0.0f ? up - x : x - up;
  const float p = (delta > 0.0f ? delta : -delta) / unit;
  return (static_cast<float>(r8) + 0.5f) * 0.00390625f < p ? up : x;
}

// The faces of a cell are read kFaceBatch at a time (the loads of a batch
// overlap; one face per turn waits for its load every time), in one pass that
// gives the random walk's radius and the analytic step's nearest face alike.
// The pass keeps the smallest distance and the second smallest; which face
// the second belongs to matters only when the two nearly tie, and then the
// faces are gone through again (resolve_tie).

template <typename Real, uint32_t F = kFeatAll>
struct UTracker : PacketState<Real, F> {
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

  Real x0, x1, x2;
  uint32_t pbeg, pend;  // the current cell's planes

  STORM_HD void begin(const Packet<Real> &p, const UMeshView<Real> &m, const CellXS<Real> *xs, const StepConsts &k) {
    x0 = p.u[0];
    x1 = p.u[1];
    x2 = p.u[2];
    o0 = p.o[0];
    o1 = p.o[1];
    o2 = p.o[2];
    cell = p.ijk;
    pbeg = m.plane_start[cell];
    pend = m.plane_start[cell + 1u];
    this->begin_packet(p, m.spec, k);
    this->set_opacity(m.spec, xs[cell], Base::is_mg(m.spec) ? m.spec.sig_s[cell] : Real(0));
  }

  template <typename Sink>
  STORM_HD void end(Packet<Real> &p, const UMeshView<Real> &m, const StepConsts &k, Sink &sink) {
    this->end_packet(p, m.spec, k, sink);
    p.u[0] = x0;
    p.u[1] = x1;
    p.u[2] = x2;
    p.ijk = cell;
  }

  // Whether (a0, a1, a2) lies within every face plane of the cell.
  STORM_HD bool inside(const UMeshView<Real> &m, Real a0, Real a1, Real a2) const {
    bool in = true;
    for (uint32_t f = pbeg; f < pend && in; f += kFaceBatch) {
      UPlane<Real> pl[kFaceBatch];
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
      for (uint32_t j = 0; j < kFaceBatch; ++j) pl[j] = m.plane[f + j];
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
      for (uint32_t j = 0; j < kFaceBatch; ++j)
        in = in && pl[j].n[0] * a0 + pl[j].n[1] * a1 + pl[j].n[2] * a2 <= pl[j].d;
    }
    return in;
  }

  // Two faces at (nearly) the smallest distance: the nearest and the next one
  // in the order of the faces, and, in the mixed engine, when they are within
  // 1e-6 along the path (an edge or a vertex), the choice between them in FP64.
  STORM_HD void resolve_tie(const UMeshView<Real> &m, Real &d, uint32_t &fa) const {
    Real dsecond = M::inf();
    uint32_t fb = pbeg;
    d = M::inf();
    fa = pbeg;
    for (uint32_t f = pbeg; f < pend; ++f) {
      const UPlane<Real> fc = m.plane[f];
      const Real den = fc.n[0] * o0 + fc.n[1] * o1 + fc.n[2] * o2;
      if (!(den > Real(0))) continue;
      Real t = (fc.d - (fc.n[0] * x0 + fc.n[1] * x1 + fc.n[2] * x2)) / den;
      t = t > Real(0) ? t : Real(0);
      if (t < d) {
        dsecond = d;
        fb = fa;
        d = t;
        fa = f;
      } else if (t < dsecond) {
        dsecond = t;
        fb = f;
      }
    }
    if (fixed_point && dsecond < M::inf() && dsecond - d <= Real(1e-6) * dsecond) {
      auto dist64 = [&](uint32_t f) {
        const UPlane<Real> fc = m.plane[f];
        const double den = static_cast<double>(fc.n[0]) * o0 + static_cast<double>(fc.n[1]) * o1 +
                           static_cast<double>(fc.n[2]) * o2;
        const double num = static_cast<double>(fc.d) - (static_cast<double>(fc.n[0]) * x0 +
                                                        static_cast<double>(fc.n[1]) * x1 +
                                                        static_cast<double>(fc.n[2]) * x2);
        const double t = num / den;
        return t > 0.0 ? t : 0.0;
      };
      const double dA = dist64(fa), dB = dist64(fb);
      if (dB < dA) {
        fa = fb;
        d = static_cast<Real>(dB);
      }
    }
  }

  template <typename Sink>
  STORM_HD int segment(const UMeshView<Real> &m, const CellXS<Real> *xs, const AccelView<Real> &acc,
                       const StepConsts &k, Sink &sink) {
    const PacketStream rs = PacketStream::make(k.seed, id, k.step, kTagTransport);
    const bool mg = Base::is_mg(m.spec);
    ++this->visit_segs;

    // ---------------- the distance to the nearest face plane
    // (computeMinDistanceToFaces), and along the direction to the nearest
    // face and the next one for ties
    Real Ro = M::inf();
    Real d = M::inf(), dsecond = M::inf();
    uint32_t fa = 0u;
    for (uint32_t f = pbeg; f < pend; f += kFaceBatch) {
      UPlane<Real> pl[kFaceBatch];
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
      for (uint32_t j = 0; j < kFaceBatch; ++j) pl[j] = m.plane[f + j];
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
#endif
      for (uint32_t j = 0; j < kFaceBatch; ++j) {
        const UPlane<Real> &fc = pl[j];
        const Real dist = fc.d - (fc.n[0] * x0 + fc.n[1] * x1 + fc.n[2] * x2);
        if constexpr ((F & kFeatAccel) != 0u) Ro = dist < Ro ? dist : Ro;
        const Real den = fc.n[0] * o0 + fc.n[1] * o1 + fc.n[2] * o2;
        // 0 where the packet sits on or beyond the face.  On a tame mesh a
        // positive distance is above 2^-56 (it is a multiple of a unit of d)
        // and a denominator below 2^-60 only ever makes a face too far to
        // matter, so the short division is exact where it counts.
        const Real a = dist > Real(0) ? dist : Real(0);
        Real t = m.tame ? M::div_tame(a, den) : a / den;
        t = den > Real(0) ? t : M::inf();
        fa = t < d ? f + j : fa;
        dsecond = M::median(d, dsecond, t);
        d = t < d ? t : d;
      }
    }

    // ---------------- which kind of step (CellXS::r_acc as on the Cartesian mesh)
    int step = kStepAnalytic;
    if constexpr ((F & kFeatAccel) != 0u) {
      if (!(Ro > Real(0))) Ro = Real(0);
      if (acc.cell && Ro >= this->r_acc) {
        const CellAccel<Real> ca = acc.cell[cell];
        const bool walk = ((ca.flags & 1u) != 0u) & (!mg | (nu < ca.e_cut)) & (Ro > Real(0)) &
                          (ca.sig_t > Real(0)) & (Ro * ca.sig_t >= acc.rw_particle_tau);
        const bool ddmc = ((ca.flags & 2u) != 0u) & (ca.total > Real(0)) &
                          (Ro * ca.ddmc_sig_t >= acc.ddmc_particle_tau) & (!multigroup | (nu < ca.ddmc_e_cut)) &
                          (m.ddmc_rate != nullptr);
        if (walk) step = kStepWalk;
        else if (ddmc)
          step = kStepDdmc;
      }
    }
    ULink<Real> ln{};
    if (step == kStepAnalytic) {
      // (also when no face lies ahead, or a denominator was too small a number)
      if (fixed_point && !(dsecond - d > Real(1e-6) * dsecond)) resolve_tie(m, d, fa);
      ln = m.link[fa];
    }

    // ---------------- random numbers (as Tracker::segment)
    Philox4 r = rs.block(ctr++);
    const Real xi = M::uniform(r.v[0]);
    const Real nlog = -M::log_unit(step == kStepWalk ? Real(1) - xi : xi);

    // ---------------- the event (d: its distance)
    int ev = kEvFace;
    Real sig_abs = cell_sig_abs;
    Philox4 r2{};
    if (step == kStepAnalytic) {
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
      d = tauLeak * Ro * Ro * (Real(3) * (mg ? ca.sig_d : ca.sig_t));
      ev = kEvLeak;
      if (mg) {
        sig_abs = ca.sig_abs;
        if (ca.up_rate > Real(0)) {
          const Real sUp = (-M::log(M::uniform(r2.v[2]))) / ca.up_rate;
          if (sUp < d && sUp < s) {
            ev = kEvReemit;
            d = sUp;
          }
        }
      }
    } else if constexpr ((F & kFeatAccel) != 0u) {
      // DDMC step (tryDDMCStep)
      const CellAccel<Real> &ca = acc.cell[cell];
      d = nlog / ca.total;
      ev = kEvLeak;
      if constexpr (multigroup) sig_abs = ca.ddmc_abs;
    }
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

    int end = ev == kEvCensus ? kEndCensus : kEndNone;
    bool turn = false;
    Real fn0 = Real(0), fn1 = Real(0), fn2 = Real(0);  // DDMC: the leak face's normal
    if (w < static_cast<double>(step == kStepWalk ? wmin * Real(0.1) : wmin)) {
      end = kEndRoulette;
    } else if (step == kStepAnalytic) {
      const Real m0 = o0 * d, m1 = o1 * d, m2 = o2 * d;
      Real n0 = x0 + m0, n1 = x1 + m1, n2 = x2 + m2;
      if constexpr (fixed_point) {
        if (n0 == x0 || n1 == x1 || n2 == x2) {
          n0 = umove_coord(x0, n0, m0, r.v[1] & 0xffu);
          n1 = umove_coord(x1, n1, m1, r.v[2] & 0xffu);
          n2 = umove_coord(x2, n2, m2, r.v[3] & 0xffu);
        }
      }
      x0 = n0;
      x1 = n1;
      x2 = n2;
      if (ev == kEvCollide) {
        turn = true;
        if (mg && !(M::uniform(r.v[1]) * cell_sig_ev < cell_sig_s)) ev = kEvReemit;
      } else if (ev == kEvCensus) {
      } else if (ln.nbr >= 0) {
        end = kEndCross;
      } else if ((m.escape_mask >> static_cast<uint32_t>(-1 - ln.nbr)) & 1u) {
        end = kEndEscape;
      } else {
        // specular reflection on the box face (BoundaryCondition.hpp:87-108)
        const UPlane<Real> fc = m.plane[fa];
        const Real on = o0 * fc.n[0] + o1 * fc.n[1] + o2 * fc.n[2];
        o0 -= Real(2) * on * fc.n[0];
        o1 -= Real(2) * on * fc.n[1];
        o2 -= Real(2) * on * fc.n[2];
      }
    } else if ((F & kFeatAccel) != 0u && step == kStepWalk) {
      Real dir[3];
      isotropic_dir<Real>(M::uniform(r.v[1]), M::uniform(r.v[2]), dir);
      Real disp = Ro;
      if (ev != kEvLeak) {
        const Real sig_d = mg ? acc.cell[cell].sig_d : acc.cell[cell].sig_t;
        const Real tauPos = d / (Real(3) * sig_d * Ro * Ro);
        disp = Ro * rw::sample_radius<Real>(rw::tables_at(acc.rw), tauPos, M::uniform(r.v[3]));
      }
      if (disp > Ro) disp = Ro;
      const Real c0 = x0, c1 = x1, c2 = x2;
      // nudge towards the mesh point, the frame's origin (:1214-1215)
      Real n0 = (c0 + disp * dir[0]) * Real(1 - 1e-6);
      Real n1 = (c1 + disp * dir[1]) * Real(1 - 1e-6);
      Real n2 = (c2 + disp * dir[2]) * Real(1 - 1e-6);
      for (int guard = 0; guard < 2000; ++guard) {
        if (inside(m, n0, n1, n2)) break;
        disp = disp * Real(0.99);
        n0 = c0 + disp * dir[0];
        n1 = c1 + disp * dir[1];
        n2 = c2 + disp * dir[2];
      }
      x0 = n0;
      x1 = n1;
      x2 = n2;
      turn = true;
      r.v[2] = r2.v[0];
      r.v[3] = r2.v[1];
    } else if ((F & kFeatAccel) != 0u && ev == kEvLeak) {
      // DDMC leak through a face chosen in proportion to its rate
      Real pick = M::uniform(r.v[1]) * acc.cell[cell].total;
      uint32_t face = 0xFFFFFFFFu, lastf = 0xFFFFFFFFu;
      const uint32_t fbeg = m.face_start[cell], fend = m.face_start[cell + 1u];
      for (uint32_t f = fbeg; f < fend; ++f) {
        const Real rt = m.ddmc_rate[f];
        if (rt > Real(0)) {
          lastf = f;
          pick -= rt;
          if (face == 0xFFFFFFFFu && pick <= Real(0)) face = f;
        }
      }
      if (face == 0xFFFFFFFFu) face = lastf;
      const UPlane<Real> fc = m.plane[pbeg + (face - fbeg)];
      fn0 = fc.n[0];
      fn1 = fc.n[1];
      fn2 = fc.n[2];
      ln = m.link[pbeg + (face - fbeg)];
      // on the face centroid (:1588), then into the neighbour
      x0 = m.face_centroid[3 * face];
      x1 = m.face_centroid[3 * face + 1];
      x2 = m.face_centroid[3 * face + 2];
      turn = true;
      end = kEndCross;
    }

    // ---------------- new direction: isotropic, or (a DDMC leak) mu = sqrt(U)
    // about the outward normal, basis as in :1565-1586
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
        const Real nx = fn0, ny = fn1, nz = fn2;
        const bool hx = (nx < Real(0) ? -nx : nx) < Real(0.9);
        // helper (1,0,0) or (0,1,0), e1 = helper - (helper . n) n, e2 = n x e1
        Real e10 = (hx ? Real(1) : Real(0)) - (hx ? nx : ny) * nx;
        Real e11 = (hx ? Real(0) : Real(1)) - (hx ? nx : ny) * ny;
        Real e12 = -(hx ? nx : ny) * nz;
        const Real e1n = M::sqrt(e10 * e10 + e11 * e11 + e12 * e12);
        if (e1n > Real(0)) {
          e10 /= e1n;
          e11 /= e1n;
          e12 /= e1n;
        }
        const Real e20 = ny * e12 - nz * e11, e21 = nz * e10 - nx * e12, e22 = nx * e11 - ny * e10;
        Real d0 = mu * nx + x * e10 + y * e20;
        Real d1 = mu * ny + x * e11 + y * e21;
        Real d2 = mu * nz + x * e12 + y * e22;
        const Real dn = M::sqrt(d0 * d0 + d1 * d1 + d2 * d2);
        if (dn > Real(0)) {
          d0 /= dn;
          d1 /= dn;
          d2 /= dn;
        }
        o0 = d0;
        o1 = d1;
        o2 = d2;
      }
    }
    if constexpr (multigroup) {
      if (ev == kEvReemit && end == kEndNone) {
        this->group_split(m.spec, k, sink);
        const bool walk = (F & kFeatAccel) != 0u && step == kStepWalk;
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
        x0 += ln.sh[0];
        x1 += ln.sh[1];
        x2 += ln.sh[2];
        cell = static_cast<uint32_t>(ln.nbr);
        pbeg = ln.pbeg;
        pend = ln.pend;
        this->set_opacity(m.spec, xs[cell], mg ? m.spec.sig_s[cell] : Real(0));
      }
    }
    return outcome;
  }
};

template <typename Real, uint32_t F>
struct TrackerOf<Real, F, UMeshView<Real>> {
  using type = UTracker<Real, F>;
};

template <typename Real, uint32_t F = kFeatAll, typename Sink>
STORM_HD int transport_packet(Packet<Real> &p, const UMeshView<Real> &m, const CellXS<Real> *xs,
                              const AccelView<Real> &acc, const StepConsts &k, int max_segments, Sink &sink) {
  UTracker<Real, F> t;
  t.begin(p, m, xs, k);
  for (int seg = 0; seg < max_segments && t.outcome == kAlive; ++seg) t.segment(m, xs, acc, k, sink);
  t.end(p, m, k, sink);
  return t.outcome;
}

}  // namespace storm
