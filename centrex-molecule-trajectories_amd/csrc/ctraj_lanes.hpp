// ctraj_lanes.hpp -- persistent lane-refill walker for beamlines with one lens.
//
// In the ES-lens beamline most molecules stop inside the lens after a variable number of steps,
// so a wavefront that walks 64 molecules start to finish keeps most lanes idle while its longest
// survivor crosses the lens.  Here a wavefront instead keeps its lanes busy:
//   * lanes are in one of the phases NEED (no molecule), LENS (integrating), POST (left the lens,
//     elements after it still to walk) or DONE;
//   * every iteration advances all LENS lanes by one integration step;
//   * when at least `refill_min` lanes are NEED/POST (or none is in the lens), a convergent refill
//     section walks the POST lanes to their end, records finished molecules, and hands NEED lanes
//     new molecule indices from the wavefront's claim [next, end), refilled in chunks from a global
//     atomic counter; new molecules walk the elements before the lens and the lens entrance.
// Each molecule's arithmetic is exactly the one of walk() in ctraj_device.hpp, so results are
// bit-identical to the simple kernel and the oracle; only the order of work changes.
#pragma once

#include "ctraj_device.hpp"

namespace ctraj {

enum : int { PH_NEED = 0, PH_LENS = 1, PH_POST = 2, PH_DONE = 3 };

struct LaneMol {
  MState m;
  int64_t gidx;
  WsRef wsb;  // LDS spline of the molecule's state
  int st;
  int label;
  uint32_t status;
  int phase;
  int fin;  // 1: finished molecule waiting to be recorded; 2: same, stopped by the lens bore
  // lens integration state
  int i, nfull;
  double h, hp, dzs, r2;  // current step, final partial step, z advance per full step, x^2 + y^2
};

// ---- circular apertures, the common case arranged for few instructions ----
// A face costs 45 VALU instructions as walk_plain writes it (14 of them the division by vz, 10 the products with
// the zero components of the acceleration), and a wavefront runs nearly every face of the beamline.  With
// a = (0, -g, 0) and faces, z, vz and g of moderate size (walk_tame_elems on the host, walk_tame per molecule) the
// same values come from 22:
//   * every face's time (zf - z) / vz by the operations of the compiled division, of which the reciprocal's are made
//     once for all faces (nothing needs its scaling: a face is nonzero, so zf - z is zero or at least 2^-160);
//   * 0 dt^2 / 2 and 0 dt add +0, which changes only a -0;
//   * (a dt^2) / 2 is exact and goes with its sum into one fused operation; dt = 0 adds zeros (velocities are
//     finite), where the plain drift leaves the molecule as it is.
// The zeros matter to a -0 only, so walk_tame sends x, y, vx, vy or t = -0 the plain way (none of them becomes -0
// on the way: a sum is -0 only where both terms are).
// 5 10^7 molecules without a lens: 682 -> 581 us (4.1 TB/s of inputs).
constexpr double kWalkLo = 0x1p-100, kWalkHi = 0x1p100;

__host__ __device__ __forceinline__ bool walk_tame_value(double v) {
  const double a = __builtin_fabs(v);
  return a >= kWalkLo && a < kWalkHi;
}

// The element table's part of the condition: circular apertures (elements in between are not looked at) and lens
// entrances on faces of moderate size, g moderate or zero.
inline bool walk_tame_elems(const ctraj_elem *e, int n, double g) {
  bool ok = g == 0.0 || walk_tame_value(g);
  for (int i = 0; i < n; ++i) ok = ok && walk_tame_value(e[i].z0) && walk_tame_value(e[i].z1);
  return ok;
}

__device__ __forceinline__ uint32_t high_word(double v) { return (uint32_t)((uint64_t)__double_as_longlong(v) >> 32); }
// false for -0 (and the smallest negative numbers)
__device__ __forceinline__ bool not_neg_zero(double v) { return high_word(v) != 0x80000000u; }
// Finite, so that v dt is 0 where dt is, and not -0, in one instruction (v_cmp_class: negative normal and denormal
// numbers, +0, positive ones).
__device__ __forceinline__ bool velocity_tame(double v) { return __builtin_amdgcn_class(v, 0x1d8); }

// The molecule's part: its acceleration is (0, -g, 0) (the caller's knowledge).
__device__ __forceinline__ bool walk_tame(const MState &m) {
  return walk_tame_value(m.vz) & ((m.z == 0.0) | walk_tame_value(m.z)) & not_neg_zero(m.x) & not_neg_zero(m.y) &
         not_neg_zero(m.t) & velocity_tame(m.vx) & velocity_tame(m.vy);
}

// 1 / v to within an ulp (v moderate).
__device__ __forceinline__ double recip(double v) {
  double y = __builtin_amdgcn_rcp(v);
  y = __builtin_fma(__builtin_fma(-v, y, 1.0), y, y);
  return __builtin_fma(__builtin_fma(-v, y, 1.0), y, y);
}

// Drift of a tame molecule to the plane zf (iv = recip(vz)); the acceleration stays (0, -g, 0).
__device__ __forceinline__ void drift_tame(MState &m, double zf, double iv, double g) {
  const double a = zf - m.z, q = a * iv;
  const double dt = __builtin_fma(__builtin_fma(-m.vz, q, a), iv, q);
  m.x = m.x + m.vx * dt;
  m.y = __builtin_fma(0.5, (-g) * (dt * dt), m.y + m.vy * dt);
  m.z = m.z + m.vz * dt;
  m.vy = m.vy + (-g) * dt;
  m.t = m.t + dt;
}

// A queue entry's molecule in registers of its own, before a walk.  The entry is read in 16-byte pieces, and this
// compiler (ROCm 7.2) may keep two fields of one piece together as one value through the walk's loop; its register
// coalescer has then lost track of one of them, which the loop overwrote (k_batch_post counted molecules twice).  An
// empty asm on the fields does not separate them for certain, a move that the compiler cannot join does.  The build
// has the machine code verified (build.py), which reports the fault.
__device__ __forceinline__ void own_registers(MState &m) {
  const auto own = [](double &v) {
    double r;
    asm("v_mov_b64 %0, %1" : "=v"(r) : "v"(v));
    v = r;
  };
  own(m.x); own(m.y); own(m.z); own(m.vx); own(m.vy); own(m.vz); own(m.t);
}

// walk_plain over circular apertures for a tame molecule.
template <bool SE>
__device__ __forceinline__ bool walk_circ_tame(const ctraj_elem *__restrict__ elems, int e0, int e1, double g, MState &m,
                                               double iv, int &label, WalkCounters &wc) {
  for (int e = e0; e < e1; ++e) {
    const ctraj_elem E = elem_get<SE>(elems, e);
    const int lhit = SE ? stop_label(E.label_hit) : E.label_hit;
    const double thr2 = E.p[1];
    drift_tame(m, E.z0, iv, g);
    ++wc.faces;
    if (beyond_r2(m.x, m.y, thr2)) { label = lhit; return false; }
    drift_tame(m, E.z1, iv, g);
    ++wc.faces;
    if (beyond_r2(m.x, m.y, thr2)) { label = lhit; return false; }
  }
  return true;
}

// Walk elements [e0, e1) (no lens among them) from the molecule's current row.  Returns false if
// the molecule stopped (label set).
template <int KM = KM_ALL, bool SE = false>
__device__ __forceinline__ bool walk_plain(const ctraj_elem *__restrict__ elems, int e0, int e1, double g, MState &m,
                                           int &label, WalkCounters &wc) {
  NullSink sk;
  for (int e = e0; e < e1; ++e) {
    const ctraj_elem E = elem_get<SE>(elems, e);
    const int lhit = SE ? stop_label(E.label_hit) : E.label_hit;
    if (E.kind == CTRAJ_CIRC) {
      const double thr2 = E.p[1];  // the squared-radius threshold of d/2 (beyond_r2)
      drift_dt(m, time_to(m, E.z0), g);
      ++wc.faces;
      if (beyond_r2(m.x, m.y, thr2)) { label = lhit; return false; }
      drift_dt(m, time_to(m, E.z1), g);
      ++wc.faces;
      if (beyond_r2(m.x, m.y, thr2)) { label = lhit; return false; }
    } else if ((KM & KM_RECT) && E.kind == CTRAJ_RECT) {
      const double x1 = E.p[0], x2 = E.p[1], y1 = E.p[2], y2 = E.p[3];
      drift_dt(m, time_to(m, E.z0), g);
      ++wc.faces;
      if (!((x1 < m.x && m.x < x2) && (y1 < m.y && m.y < y2))) { label = lhit; return false; }
      drift_dt(m, time_to(m, E.z1), g);
      ++wc.faces;
      if (!((x1 < m.x && m.x < x2) && (y1 < m.y && m.y < y2))) { label = lhit; return false; }
    } else if ((KM & KM_PLATES) && E.kind == CTRAJ_PLATES) {
      const double x1 = E.p[0], x2 = E.p[1];
      drift_dt(m, time_to(m, E.z0), g);
      ++wc.faces;
      if (!(x1 < m.x && m.x < x2)) { label = lhit; return false; }
      double dt = time_to(m, E.z1);
      double xe = m.x;
      if (dt != 0.0) xe = (m.x + m.vx * dt) + (m.ax * (dt * dt)) * 0.5;
      const bool inside = (x1 < xe && xe < x2);
      if (!inside) {
        if (m.vx < 0.0) dt = (x1 - m.x) / m.vx;
        else if (m.vx > 0.0) dt = (x2 - m.x) / m.vx;
      }
      drift_dt(m, dt, g);
      ++wc.faces;
      if (!inside) { label = lhit; return false; }
    }
  }
  (void)sk;
  return true;
}

}  // namespace ctraj
