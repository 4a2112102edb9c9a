// adjoint.hip -- sigmoid-smoothed detected flux and its discrete adjoint (gfx950).
//
// k_smooth<GRAD> walks 64 molecules per wavefront work item through the beamline without stopping
// them.  Each circular-aperture face multiplies the molecule's weight by sigmoid((r - rho)/s); the
// lens is integrated with the same classical RK4 (and the same FMA sequence) as the propagation
// kernels.  With GRAD the wavefront then runs the reverse sweep:
//   * aperture faces: the sigmoid factor's derivative and the adjoint of the ballistic drift;
//   * lens: the adjoint of the final partial step (with d/dh, which carries d/d(vz)), then, for each
//     checkpoint segment (last first), the segment's steps recomputed from the checkpoint and the
//     adjoint of each full step applied backwards, accumulating d/dV through the field scale;
//   * the mean axial speed collects the adjoint of vz.
// Per-parameter sums are reduced over the wavefront (xor butterfly) at wave-uniform points and
// written per work item; k_smooth_reduce adds the items of each parameter set in a fixed order,
// so J and the gradient do not depend on scheduling.
//
// Workspace of one wavefront (doubles, lane-minor so that every access is one 512-byte row):
//   faces [n_face_slots][4][64]   state (x, y, vx, vy) on each aperture face and lens entrance
//   ends  [n_lens][4][64]         lens state before the final partial step
//   ckpt  [n_ck_slots][4][64]     lens state before full steps 0, K, 2K, ...
//   sub   [ceil(K/kSub)][4][64]   state every kSub steps of the segment being reversed (K > kSub)
// and, in LDS, a [kSub][4][64] window of recomputed step inputs per wavefront.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "ctraj_device.hpp"
#include "ctraj_internal.hpp"
#include "ctraj_wave.hpp"

using namespace ctraj;

namespace {

struct SmoothArgs {
  const double *x, *y, *vx, *vy, *eps;
  const double *params;           // [n_cfg][n_params]
  double *partial;                // [n_items][n_params + 1]: gradient sums, then the J sum
  double *ws;                     // workspace, ws_stride doubles per wavefront
  unsigned long long *n_capped;   // may be null
  unsigned long long *next;       // items handed out beyond each wavefront's first (zeroed before the launch)
  int64_t n, items_per_cfg, n_items, ws_stride;
  double z_src, sigma_vz, inv_s;
  int n_params, K, max_steps, ck_per_lens, off_end, off_ck, off_sub;  // offsets in rows of 256 doubles
  int rec_lds;                  // LDS offset (doubles) of the per-wavefront recompute windows
};

// Inside a checkpoint segment the reverse sweep works in windows of kSub steps: a segment of more
// than one window is recomputed once to store the state every kSub steps (HBM rows, cache-resident),
// then each window, last first, is recomputed into the wavefront's LDS slice and reversed.  With
// K <= kSub a segment is one window: 1 - 1/kSub forward steps are recomputed per step.
constexpr int kSub = 4;

// sigmoid(w) and 1 - sigmoid(w) without cancellation.
__device__ __forceinline__ void sigmoid2(double w, double &phi, double &omphi) {
  const double e = exp(-__builtin_fabs(w));
  const double q = 1.0 / (1.0 + e);
  const double eq = e * q;
  phi = w >= 0.0 ? q : eq;
  omphi = w >= 0.0 ? eq : q;
}

// Ballistic drift by tau under a = (0, -g): the propagation kernels' drift with the stored
// acceleration (0, -g, 0) (x gains + (0 * tau^2) * 0.5 = +0 there, which changes nothing).
__device__ __forceinline__ void drift_g(double &x, double &y, double vx, double &vy, double tau, double g) {
  x = x + vx * tau;
  y = (y + vy * tau) + ((-g) * (tau * tau)) * 0.5;
  vy = vy + (-g) * tau;
}

// Adjoint of drift_g given the state after the drift (vx, vy_after): updates (vbx, vby) in place
// (pbx, pby pass through) and returns d/dtau.
__device__ __forceinline__ double drift_g_adj(double vx, double vy_after, double g, double tau, double pbx,
                                              double pby, double &vbx, double &vby) {
  const double taubar = (pbx * vx + pby * vy_after) - g * vby;
  vbx = vbx + tau * pbx;
  vby = vby + tau * pby;
  return taubar;
}

// A value that is the same in every lane, as a scalar register pair.  FP64 arithmetic has no scalar
// unit, so the lens constants formed from a parameter set (20 doubles) would otherwise hold 40 vector
// registers of every lane.
__device__ __forceinline__ double uniform_f64(double v) {
  return __longlong_as_double((long long)uniform_u64((unsigned long long)__double_as_longlong(v)));
}

__device__ __forceinline__ HexK uniform_hex_k(double ks, double h) {
  const HexK k = hex_k(ks, h);
  return HexK{uniform_f64(k.h), uniform_f64(k.hh), uniform_f64(k.c3), uniform_f64(k.c4), uniform_f64(k.cx),
              uniform_f64(k.kh6)};
}

// One lens of one parameter set.  FOLD (hex_folds(ks)): slopes are s = W' p + (0, gk), gk = -g/ks, and the
// step constants are hex_k(ks, h); otherwise slopes are accelerations and the constants hex_k(1, h).
struct LensK {
  WsRef wsb;
  double umax, cu;
  double kf;  // the step constants' scale: ks (FOLD) or 1
  double sl;  // slope per W': 1 (FOLD) or ks
  double gs;  // the slope's constant part: gk (FOLD) or -g
  double c2;  // 2 cu sl: d(slope scale)/d(r2) = c2/2 dW'/du
  HexK hk;    // of the full step
};

template <bool FOLD>
__device__ __forceinline__ void smooth_slope(const LensK &L, double x, double y, double r2, double &sx, double &sy) {
  if constexpr (FOLD) {
    slope_hex_k(L.wsb, L.umax, L.cu, L.gs, x, y, r2, sx, sy);
  } else {
    const double f = wspline_eval(L.wsb, L.umax, r2 * L.cu) * L.sl;  // force_hex_r2
    sx = f * x;
    sy = __builtin_fma(f, y, L.gs);
  }
}

// The forward sweep's lens step and its recomputation in the reverse sweep (one function, so that a
// recomputed state equals the forward state bit for bit): the propagation kernels' folded hexapole step,
// or their plain RK4 step where the force scale does not fold.
template <bool FOLD>
__device__ __forceinline__ void smooth_step(const LensK &L, const HexK &K, double &x, double &y, double &vx, double &vy) {
  rk4_expanded(
      K, [&](double px, double py, double pr2, double &sx, double &sy) { smooth_slope<FOLD>(L, px, py, pr2, sx, sy); }, x,
      y, vx, vy, __builtin_fma(x, x, y * y));
}

// The slope scale and its derivatives at r2: w = sl W'(u), u = min(cu r2, umax); dw = 2 dw/dr2 (0 where u
// is clamped); gv = V dw/dV per unit sl (ks and cu are both proportional to V): W' + u dW'/du.
template <bool FOLD>
__device__ __forceinline__ void hex_eval_d(const LensK &L, double r2, double &w, double &dw, double &gv) {
  const double u0 = r2 * L.cu;
  const double u = clamp_to(u0, L.umax);
  const unsigned k = (unsigned)(int)u;
  const double s = __builtin_amdgcn_fract(u);
  const dbl2_t ab = L.wsb.ab[k];
  const double c = L.wsb.c[k];
  const double t = __builtin_fma(ab.x, s, ab.y);
  const double P = __builtin_fma(t, s, c);
  double dP = __builtin_fma(ab.x, s, t);
  if (u0 > L.umax) dP = 0.0;
  w = FOLD ? P : P * L.sl;
  dw = L.c2 * dP;
  gv = __builtin_fma(u0, dP, P);
}

// Jacobian of one stage slope s = w(r2) p + const, transposed (it is symmetric: w I + dw p p^T), applied
// to the slope's adjoint (sbx, sby); Vbar gathers the slope's dependence on V.
__device__ __forceinline__ void slope_adj(double w, double dw, double gv, double px, double py, double sbx, double sby,
                                          double &pbx, double &pby, double &Vbar) {
  const double q = __builtin_fma(px, sbx, py * sby);
  const double dq = dw * q;
  Vbar = __builtin_fma(q, gv, Vbar);
  pbx = __builtin_fma(w, sbx, dq * px);
  pby = __builtin_fma(w, sby, dq * py);
}

// Reverse of one RK4 step with constants K from input state (x, y, vx, vy): the transposed derivative of
// rk4_expanded's own form,
//   x2 = x + h/2 v,  x3 = x2 + c3 s1,  x4 = (x + h v) + c4 s2,
//   x' = (x + h v) + cx (s1 + s2 + s3),  v' = v + kh6 (s1 + 2 s2 + 2 s3 + s4),
// which needs no stage velocities (52 operations on the adjoint where the classical stages take 85).
// In: (pbx, pby, vbx, vby) = adjoint of the step's output.  Out: adjoint of its input.  Vbar gathers
// V/sl d/dV; with WANT_H the derivative with respect to h is returned.
// The sums of products are fused multiply-adds (the gradient is checked against the CPU adjoint to a
// tolerance, not bit for bit).
template <bool FOLD, bool WANT_H>
__device__ __forceinline__ double rk4_adjoint(const LensK &L, const HexK &K, double x, double y, double vx, double vy,
                                              double &pbx, double &pby, double &vbx, double &vby, double &Vbar) {
  double w1, d1, g1, w2, d2, g2, w3, d3, g3, w4, d4, g4;
  hex_eval_d<FOLD>(L, __builtin_fma(x, x, y * y), w1, d1, g1);
  const double s1x = w1 * x, s1y = __builtin_fma(w1, y, L.gs);
  const double p2x = __builtin_fma(K.hh, vx, x), p2y = __builtin_fma(K.hh, vy, y);
  hex_eval_d<FOLD>(L, __builtin_fma(p2x, p2x, p2y * p2y), w2, d2, g2);
  const double s2x = w2 * p2x, s2y = __builtin_fma(w2, p2y, L.gs);
  const double p3x = __builtin_fma(K.c3, s1x, p2x), p3y = __builtin_fma(K.c3, s1y, p2y);
  hex_eval_d<FOLD>(L, __builtin_fma(p3x, p3x, p3y * p3y), w3, d3, g3);
  const double xvx = __builtin_fma(K.h, vx, x), xvy = __builtin_fma(K.h, vy, y);
  const double p4x = __builtin_fma(K.c4, s2x, xvx), p4y = __builtin_fma(K.c4, s2y, xvy);
  hex_eval_d<FOLD>(L, __builtin_fma(p4x, p4x, p4y * p4y), w4, d4, g4);

  const double s4bx = K.kh6 * vbx, s4by = K.kh6 * vby;
  double pb4x, pb4y, pb3x, pb3y, pb2x, pb2y, pb1x, pb1y;
  slope_adj(w4, d4, g4, p4x, p4y, s4bx, s4by, pb4x, pb4y, Vbar);
  const double e1x = __builtin_fma(K.cx, pbx, s4bx), e1y = __builtin_fma(K.cx, pby, s4by);
  const double e2x = e1x + s4bx, e2y = e1y + s4by;
  slope_adj(w3, d3, g3, p3x, p3y, e2x, e2y, pb3x, pb3y, Vbar);
  const double s2bx = __builtin_fma(K.c4, pb4x, e2x), s2by = __builtin_fma(K.c4, pb4y, e2y);
  slope_adj(w2, d2, g2, p2x, p2y, s2bx, s2by, pb2x, pb2y, Vbar);
  const double s1bx = __builtin_fma(K.c3, pb3x, e1x), s1by = __builtin_fma(K.c3, pb3y, e1y);
  slope_adj(w1, d1, g1, x, y, s1bx, s1by, pb1x, pb1y, Vbar);
  const double xvbx = pbx + pb4x, xvby = pby + pb4y, x2bx = pb2x + pb3x, x2by = pb2y + pb3y;
  double hbar = 0.0;
  if constexpr (WANT_H) {
    const double s3x = w3 * p3x, s3y = __builtin_fma(w3, p3y, L.gs);
    const double s4x = w4 * p4x, s4y = __builtin_fma(w4, p4y, L.gs);
    const double S3x = (s1x + s2x) + s3x, S3y = (s1y + s2y) + s3y;
    const double kh = L.kf * K.h;
    hbar = (pbx * (vx + (kh / 3.0) * S3x) + pby * (vy + (kh / 3.0) * S3y)) +
           (L.kf * kSixth) * (vbx * ((S3x + s2x) + (s3x + s4x)) + vby * ((S3y + s2y) + (s3y + s4y))) +
           0.5 * ((x2bx * vx + x2by * vy) + kh * (pb3x * s1x + pb3y * s1y)) +
           (pb4x * (vx + kh * s2x) + pb4y * (vy + kh * s2y));
  }
  pbx = (xvbx + x2bx) + pb1x;
  pby = (xvby + x2by) + pb1y;
  vbx = __builtin_fma(K.hh, x2bx, __builtin_fma(K.h, xvbx, vbx));
  vby = __builtin_fma(K.hh, x2by, __builtin_fma(K.h, xvby, vby));
  return hbar;
}

// Lane j of the wavefront owns accumulators for parameters j, j + 64, j + 128.
__device__ __forceinline__ void acc_add(double &a0, double &a1, double &a2, int p, int lane, double v) {
  if ((p & 63) == lane) {
    const int b = p >> 6;
    if (b == 0) a0 += v;
    else if (b == 1) a1 += v;
    else a2 += v;
  }
}

__device__ __forceinline__ double *row(double *W, int slot, int lane) { return W + (size_t)slot * 256 + lane; }

__device__ __forceinline__ void put4(double *W, int slot, int lane, double a, double b, double c, double d) {
  double *r = row(W, slot, lane);
  r[0] = a;
  r[64] = b;
  r[128] = c;
  r[192] = d;
}

__device__ __forceinline__ void get4(const double *W, int slot, int lane, double &a, double &b, double &c, double &d) {
  const double *r = W + (size_t)slot * 256 + lane;
  a = r[0];
  b = r[64];
  c = r[128];
  d = r[192];
}

// z of the exit face of an element (CIRC: z1; LENS: its z0 parameter + L); z_src before the first.
__device__ __forceinline__ double exit_z(const KBeam &B, const double *P, int e, int pidx_e, double z_src) {
  if (e < 0) return z_src;
  const ctraj_elem E = elem_at(B.elems, e);
  if (E.kind == CTRAJ_LENS) return uniform_f64(P[pidx_e + 1]) + E.p[3];
  return E.z1;
}

__device__ __forceinline__ int n_params_of(const ctraj_elem &E) { return E.kind == CTRAJ_LENS ? 2 : 1; }

__device__ __forceinline__ int wave_max(int v) {
  for (int o = 1; o < 64; o <<= 1) v = max(v, __shfl_xor(v, o, 64));
  return __builtin_amdgcn_readfirstlane(v);
}

__device__ __forceinline__ LensK smooth_lens(const ctraj_elem &E, const Tables &T, double scale, double g) {
  LensK L;
  const double ks = E.p[4] * scale, cu = E.p[5] * scale;
  const bool fold = hex_folds(ks);
  L.wsb = ws_of(T, 0);
  L.umax = T.umax;
  L.cu = uniform_f64(cu);
  L.kf = uniform_f64(fold ? ks : 1.0);
  L.sl = uniform_f64(fold ? 1.0 : ks);
  L.gs = uniform_f64(fold ? -g / ks : -g);
  L.c2 = uniform_f64((2.0 * L.sl) * cu);
  L.hk = uniform_hex_k(L.kf, E.p[2]);
  return L;
}

// Where a wavefront keeps what the reverse sweep of one lens needs (workspace rows), and its LDS window.
struct LensStore {
  double *W;
  int end, ck, sub;  // rows: the state before the partial step, checkpoints, states every kSub steps
  int K;
  lds_double *rec;
};

// Forward through one lens: nfull full steps (per lane; nmax is the wavefront's largest), then the partial
// step hp.  The step loop and its counters are wave-uniform, so every checkpoint is one coalesced row.
template <bool GRAD, bool FOLD>
__device__ __forceinline__ void lens_forward(const LensK &L, const LensStore &S, int lane, bool ok, int nfull, int nmax,
                                             double hp, double &x, double &y, double &vx, double &vy) {
  int next = 0, slot = S.ck;
  for (int s = 0; s < nmax; ++s) {
    const bool mark = GRAD && s == next;
    if (s < nfull) {
      if constexpr (GRAD) {
        if (mark) put4(S.W, slot, lane, x, y, vx, vy);
      }
      smooth_step<FOLD>(L, L.hk, x, y, vx, vy);
    }
    if (mark) {
      next += S.K;
      ++slot;
    }
  }
  if (ok) {
    if constexpr (GRAD) put4(S.W, S.end, lane, x, y, vx, vy);
    smooth_step<FOLD>(L, hex_k(L.kf, hp), x, y, vx, vy);
  }
}

// Reverse through one lens; returns d/dhp.
template <bool FOLD>
__device__ __forceinline__ double lens_reverse(const LensK &L, const LensStore &S, int lane, bool ok, int nfull, int nmax,
                                               double hp, double &pbx, double &pby, double &vbx, double &vby,
                                               double &Vbar) {
  double x = 0.0, y = 0.0, vx = 0.0, vy = 0.0, hbar = 0.0;
  if (ok) {
    get4(S.W, S.end, lane, x, y, vx, vy);
    hbar = rk4_adjoint<FOLD, true>(L, hex_k(L.kf, hp), x, y, vx, vy, pbx, pby, vbx, vby, Vbar);
  }
  if (nmax == 0) return hbar;
  for (int sg = (nmax - 1) / S.K; sg >= 0; --sg) {
    const int s0 = sg * S.K, s1 = min(s0 + S.K, nmax);
    const int nsub = (s1 - s0 + kSub - 1) / kSub;
    if (s0 < nfull) get4(S.W, S.ck + sg, lane, x, y, vx, vy);
    if (nsub > 1) {  // the state every kSub steps of the segment
      for (int q = 0; q < nsub; ++q) {
        const int t0 = s0 + q * kSub;
        if (t0 < nfull) put4(S.W, S.sub + q, lane, x, y, vx, vy);
        if (q + 1 < nsub)
          for (int s = t0; s < t0 + kSub; ++s)
            if (s < nfull) smooth_step<FOLD>(L, L.hk, x, y, vx, vy);
      }
    }
    // windows, last first: recompute into LDS (the last state stays in registers), then reverse
    for (int q = nsub - 1; q >= 0; --q) {
      const int t0 = s0 + q * kSub, t1 = min(t0 + kSub, s1);
      if (nsub > 1 && t0 < nfull) get4(S.W, S.sub + q, lane, x, y, vx, vy);
      for (int s = t0; s < t1 - 1; ++s) {
        if (s < nfull) {
          lds_double *r = S.rec + (s - t0) * 256;
          r[0] = x;
          r[64] = y;
          r[128] = vx;
          r[192] = vy;
          smooth_step<FOLD>(L, L.hk, x, y, vx, vy);
        }
      }
      for (int s = t1 - 1; s >= t0; --s) {
        if (s < nfull) {
          if (s < t1 - 1) {
            const lds_double *r = S.rec + (s - t0) * 256;
            x = r[0];
            y = r[64];
            vx = r[128];
            vy = r[192];
          }
          (void)rk4_adjoint<FOLD, false>(L, L.hk, x, y, vx, vy, pbx, pby, vbx, vby, Vbar);
        }
      }
    }
  }
  return hbar;
}

// What bounds it: VALU issue.  With GRAD a lens step costs 74 VALU instructions forward, 3/4 of that again
// to recompute, and 143 to reverse (169 with the stage velocities formed), at four wavefronts per SIMD:
// 128 registers (46 spilled, none inside a step loop) and 8 KB of window each, so that 16 wavefronts share
// one 24 KB table per CU; with the lens constants in vector registers (233) and 16 KB windows it was two.
// 10^6 molecules, one parameter set, K = 64: 5.5 -> 3.0 ms (the four wavefronts and the shorter reverse
// step 5.5 -> 3.84, items from a counter -> 3.1); 16 sets of 100,003, K = 8: 7.35 -> 5.1 ms.  Without
// GRAD 115 registers hold four wavefronts; five, six and eight (96, 80, 64 registers, no spill in the step
// loop) measured the same or slower (1.69, 1.70, 1.76 ms against 1.70 for 12 x 2 10^5 molecules; 2.05
// with a fixed share per wavefront).
template <bool GRAD>
__global__ void __launch_bounds__(GRAD ? 1024 : 512) k_smooth(KBeam B, KTab KT, SmoothArgs A) {
  extern __shared__ __attribute__((aligned(16))) double lds[];
  const Tables T = stage_tables(lds, KT);
  __syncthreads();
  const int lane = lane_id();
  const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t wpb = blockDim.x >> 6;
  const int64_t gwave = (int64_t)blockIdx.x * wpb + wave;
  const int64_t nwaves = (int64_t)gridDim.x * wpb;
  double *W = GRAD ? A.ws + gwave * A.ws_stride : nullptr;
  LensStore S{W, 0, 0, A.off_sub, A.K, nullptr};
  if constexpr (GRAD) S.rec = (lds_double *)(lds + A.rec_lds) + wave * (kSub * 256) + lane;
  const double g = B.g;
  const int np = A.n_params;
  unsigned long long capped = 0;

  // A SIMD issues its oldest ready wavefront first, so with a fixed share per wavefront the oldest of a
  // SIMD's four finished in half the time of the youngest, which then ran alone (1e6 molecules: 1.7 to 3.4 ms,
  // wavefronts alive 63 % of the kernel's time); items taken from a counter keep all of them busy to the end.
  for (int64_t item = gwave; item < A.n_items;) {
    const int64_t cfg = item / A.items_per_cfg;
    const int64_t i = (item - cfg * A.items_per_cfg) * 64 + lane;
    const double *P = A.params + cfg * np;
    double x = 0.0, y = 0.0, vx = 0.0, vy = 0.0, vz = 1.0;
    bool ok = false;
    if (i < A.n) {
      x = A.x[i];
      y = A.y[i];
      vx = A.vx[i];
      vy = A.vy[i];
      vz = P[np - 1] + A.sigma_vz * A.eps[i];
      ok = vz > 0.0;
      if (!ok) vz = 1.0;
    }
    double Jw = ok ? 1.0 : 0.0;  // product of the sigmoid factors
    double zc = A.z_src;
    int fslot = 0, lens = 0, pidx = 0;

    // ---------------- forward ----------------
    for (int e = 0; e < B.n_elems; ++e) {
      const ctraj_elem E = elem_at(B.elems, e);
      if (E.kind == CTRAJ_CIRC) {
        const double r = P[pidx];
        const int nf = E.z1 > E.z0 ? 2 : 1;
        for (int f = 0; f < nf; ++f) {
          const double zf = f ? E.z1 : E.z0;
          if (ok) {
            drift_g(x, y, vx, vy, (zf - zc) / vz, g);
            if constexpr (GRAD) put4(W, fslot, lane, x, y, vx, vy);
            double phi, om;
            sigmoid2((r - __builtin_sqrt(x * x + y * y)) * A.inv_s, phi, om);
            Jw = Jw * phi;
          }
          zc = zf;
          ++fslot;
        }
        pidx += 1;
      } else {  // CTRAJ_LENS
        const double V = uniform_f64(P[pidx]), z0 = uniform_f64(P[pidx + 1]);
        const double scale = V / E.p[7];
        const LensK L = smooth_lens(E, T, scale, g);
        const double h = E.p[2], Ll = E.p[3];
        if (!(scale >= 0.0)) {  // a negative or NaN field scale has no table: the set contributes 0
          ok = false;
          Jw = 0.0;
        }
        int nfull = 0;
        double hp = 0.0;
        if (ok) {
          drift_g(x, y, vx, vy, (z0 - zc) / vz, g);
          if constexpr (GRAD) put4(W, fslot, lane, x, y, vx, vy);
          uint32_t st = 0;
          nfull = rk4_full_steps(Ll, vz, h, A.max_steps, st);
          capped += (st & CTRAJ_ST_CAPPED) ? 1u : 0u;
          hp = Ll / vz - (double)nfull * h;
        }
        const int nmax = wave_max(nfull);
        S.end = A.off_end + lens;
        S.ck = A.off_ck + lens * A.ck_per_lens;
        if (hex_folds(E.p[4] * scale)) lens_forward<GRAD, true>(L, S, lane, ok, nfull, nmax, hp, x, y, vx, vy);
        else lens_forward<GRAD, false>(L, S, lane, ok, nfull, nmax, hp, x, y, vx, vy);
        zc = z0 + Ll;
        ++fslot;
        ++lens;
        pidx += 2;
      }
    }

    double a0 = 0.0, a1 = 0.0, a2 = 0.0;
    if constexpr (GRAD) {
      // ---------------- reverse ----------------
      double pbx = 0.0, pby = 0.0, vbx = 0.0, vby = 0.0, vzbar = 0.0;
      double zexit_bar = 0.0;  // adjoint of the exit z of the element before the current one
      for (int e = B.n_elems - 1; e >= 0; --e) {
        const ctraj_elem E = elem_at(B.elems, e);
        pidx -= n_params_of(E);
        const int pprev = e > 0 ? pidx - n_params_of(elem_at(B.elems, e - 1)) : 0;
        const double zprev = exit_z(B, P, e - 1, pprev, A.z_src);
        if (E.kind == CTRAJ_CIRC) {
          const double r = P[pidx];
          const int nf = E.z1 > E.z0 ? 2 : 1;
          double rbar = 0.0, zfrom_bar = 0.0;
          for (int f = nf - 1; f >= 0; --f) {
            --fslot;
            const double zf = f ? E.z1 : E.z0;
            const double zfrom = f ? E.z0 : zprev;
            if (ok) {
              double fx, fy, fvx, fvy;
              get4(W, fslot, lane, fx, fy, fvx, fvy);
              const double rho = __builtin_sqrt(fx * fx + fy * fy);
              double phi, om;
              sigmoid2((r - rho) * A.inv_s, phi, om);
              const double wbar = Jw * om;
              rbar = rbar + wbar * A.inv_s;
              if (rho > 0.0) {
                const double rb = -(wbar * A.inv_s) / rho;
                pbx = pbx + rb * fx;
                pby = pby + rb * fy;
              }
              const double tau = (zf - zfrom) / vz;
              const double taubar = drift_g_adj(fvx, fvy, g, tau, pbx, pby, vbx, vby);
              vzbar = vzbar - (taubar * tau) / vz;
              if (f == 0) zfrom_bar = -taubar / vz;
            }
          }
          acc_add(a0, a1, a2, pidx, lane, wave_sum(rbar));
          zexit_bar = zfrom_bar;
        } else {  // CTRAJ_LENS
          const double V = uniform_f64(P[pidx]), z0 = uniform_f64(P[pidx + 1]);
          const double scale = V / E.p[7];
          const LensK L = smooth_lens(E, T, scale, g);
          const double h = E.p[2], Ll = E.p[3];
          double Vbar = 0.0, z0bar = zexit_bar, zfrom_bar = 0.0;
          --lens;
          --fslot;
          int nfull = 0;
          double hp = 0.0;
          if (ok) {
            uint32_t st = 0;
            nfull = rk4_full_steps(Ll, vz, h, A.max_steps, st);
            hp = Ll / vz - (double)nfull * h;
          }
          const int nmax = wave_max(nfull);
          S.end = A.off_end + lens;
          S.ck = A.off_ck + lens * A.ck_per_lens;
          const double hbar =
              hex_folds(E.p[4] * scale)
                  ? lens_reverse<true>(L, S, lane, ok, nfull, nmax, hp, pbx, pby, vbx, vby, Vbar)
                  : lens_reverse<false>(L, S, lane, ok, nfull, nmax, hp, pbx, pby, vbx, vby, Vbar);
          if (ok) {
            Vbar = (Vbar * L.sl) * (1.0 / V);
            vzbar = vzbar - hbar * ((Ll / vz) / vz);  // hp = L/vz - nfull h
            // drift from the previous exit to the lens entrance z0
            double ex, ey, evx, evy;
            get4(W, fslot, lane, ex, ey, evx, evy);
            const double tau = (z0 - zprev) / vz;
            const double taubar = drift_g_adj(evx, evy, g, tau, pbx, pby, vbx, vby);
            vzbar = vzbar - (taubar * tau) / vz;
            z0bar = z0bar + taubar / vz;
            zfrom_bar = -taubar / vz;
          }
          acc_add(a0, a1, a2, pidx, lane, wave_sum(Vbar));
          acc_add(a0, a1, a2, pidx + 1, lane, wave_sum(z0bar));
          zexit_bar = zfrom_bar;
        }
      }
      acc_add(a0, a1, a2, np - 1, lane, wave_sum(vzbar));  // d vz / d mu = 1
    }
    acc_add(a0, a1, a2, np, lane, wave_sum(Jw));
    double *out = A.partial + item * (int64_t)(np + 1);
    if (lane <= np) out[lane] = a0;
    if (64 + lane <= np) out[64 + lane] = a1;
    if (128 + lane <= np) out[128 + lane] = a2;
    unsigned long long t = 0;
    if (lane == 0) t = atomicAdd(A.next, 1ull);
    item = nwaves + (int64_t)uniform_u64(t);
  }
  if (A.n_capped) {
    const double c = wave_sum((double)capped);
    if (lane == 0 && c > 0.0) atomicAdd(A.n_capped, (unsigned long long)c);
  }
}

// J[c] = (sum of item J sums) / n and grad[c][j] = (sum of item sums) / n, each over the items of
// parameter set c = blockIdx.x in a fixed order (strided per thread, then a fixed LDS tree).  One
// workgroup per sum, j = blockIdx.y (the last is J): a workgroup's time is the latency of its strided
// loads, so one workgroup for all seven sums of 10^6 molecules took 64 us.
__global__ void __launch_bounds__(256) k_smooth_reduce(const double *partial, int64_t items_per_cfg, int np, double inv_n,
                                                       double *J, double *grad) {
  __shared__ double red[256];
  const int64_t c = blockIdx.x;
  const int j = (int)blockIdx.y;
  if (j < np && !grad) return;
  const double *base = partial + c * items_per_cfg * (int64_t)(np + 1) + j;
  double s = 0.0;
  for (int64_t it = threadIdx.x; it < items_per_cfg; it += blockDim.x) s += base[it * (np + 1)];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int w = blockDim.x >> 1; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    if (j == np) J[c] = red[0] * inv_n;
    else grad[c * np + j] = red[0] * inv_n;
  }
}

}  // namespace

// ---------------------------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------------------------
static int smooth_layout(ctraj_ctx *c, int *np, int *n_faces, int *n_lens, double *theta) {
  if (!c->have_beamline) return fail(c, CTRAJ_ESTATE, "no beamline set");
  int p = 0, nf = 0, nl = 0;
  for (const ctraj_elem &E : c->h_elems) {
    if (E.kind == CTRAJ_CIRC) {
      if (theta) theta[p] = E.p[0];
      p += 1;
      nf += E.z1 > E.z0 ? 2 : 1;
    } else if (E.kind == CTRAJ_LENS) {
      if (E.force != CTRAJ_FORCE_WSPLINE_HEX || E.integrator != CTRAJ_INTEG_RK4)
        return fail(c, CTRAJ_EINVAL, "smooth objective: lenses must use the hexapole W' spline and classical RK4");
      if (!(E.p[7] != 0.0)) return fail(c, CTRAJ_EINVAL, "smooth objective: lens V (p[7]) must be nonzero");
      if (theta) {
        theta[p] = E.p[7];
        theta[p + 1] = E.z0;
      }
      p += 2;
      nf += 1;
      nl += 1;
    } else {
      return fail(c, CTRAJ_EINVAL, "smooth objective: only circular apertures and lenses are supported");
    }
  }
  *np = p + 1;
  *n_faces = nf;
  *n_lens = nl;
  return CTRAJ_OK;
}

// Whether b holds `bytes`, or could be replaced by a buffer that does.  Where memory is short it stays as it is: a
// caller that can do with less does not give up what it has, nor other contexts their kept blocks, call after call.
static bool extra_buf(ctraj_ctx *c, ctraj_devbuf &b, size_t bytes) {
  if (b.p && b.bytes >= bytes) return true;
  size_t free_b = 0, total = 0;
  void *p = nullptr;
  if (hipMemGetInfo(&free_b, &total) != hipSuccess || free_b < bytes || hipMalloc(&p, bytes) != hipSuccess) {
    (void)hipGetLastError();
    return false;
  }
  if (b.p && (hipStreamSynchronize(c->stream) != hipSuccess || hipFree(b.p) != hipSuccess)) {
    (void)hipGetLastError();
    (void)hipFree(p);
    return false;
  }
  b.p = p;
  b.bytes = bytes;
  return true;
}

extern "C" {

int32_t ctraj_smooth_params(ctraj_ctx *c, int32_t *n_params, double *theta) {
  if (!c || !n_params) return fail(c, CTRAJ_EINVAL, "null argument");
  int np, nf, nl;
  const int rc = smooth_layout(c, &np, &nf, &nl, theta);
  if (rc != CTRAJ_OK) return rc;
  *n_params = np;
  return CTRAJ_OK;
}

int32_t ctraj_smooth_objective(ctraj_ctx *c, const ctraj_smooth *s) {
  if (!c || !s) return fail(c, CTRAJ_EINVAL, "null argument");
  HIPCHK(c, hipSetDevice(c->device));
  int np, nf, nl;
  int rc = smooth_layout(c, &np, &nf, &nl, nullptr);
  if (rc != CTRAJ_OK) return rc;
  if (s->n_params != np)
    return fail(c, CTRAJ_EINVAL, "n_params is " + std::to_string(s->n_params) + ", the beamline has " + std::to_string(np));
  if (np + 1 > 192) return fail(c, CTRAJ_EINVAL, "smooth objective: at most 191 parameters");
  if (s->n <= 0) return fail(c, CTRAJ_EINVAL, "n must be > 0");
  if (s->n_cfg < 1) return fail(c, CTRAJ_EINVAL, "n_cfg must be >= 1");
  if (!s->x || !s->y || !s->vx || !s->vy || !s->eps || !s->params || !s->J)
    return fail(c, CTRAJ_EINVAL, "source arrays, params and J are required");
  if (!(s->softness > 0.0)) return fail(c, CTRAJ_EINVAL, "softness must be > 0");
  if (s->ckpt_every < 1) return fail(c, CTRAJ_EINVAL, "ckpt_every must be >= 1");
  if (s->max_steps < 1) return fail(c, CTRAJ_EINVAL, "max_steps must be >= 1");
  const bool grad = s->grad != nullptr;
  const int block_req = s->block;
  if (block_req % 64 || block_req < 0 || block_req > 512)
    return fail(c, CTRAJ_EINVAL, "block must be a multiple of 64 up to 512");
  if (nl > 0 && (!c->d_ws || c->ws_states < 1)) return fail(c, CTRAJ_ESTATE, "no W' spline set");

  KTab kt = ctx_ktab(c);
  kt.ws_states = nl > 0 ? 1 : 0;  // state 0 only
  kt.rt_total = 0;
  const size_t lds_tab = ktab_lds_bytes(kt);
  // with gradients each wavefront keeps a recompute window in LDS beside the tables
  const size_t lds_wave = grad ? (size_t)kSub * 256 * sizeof(double) : 0;
  int block = block_req ? block_req : 256;
  if (grad && !block_req) {
    // 16 wavefronts fit beside one state's 24 KB table, fewer beside a longer one.  Where there are fewer work items
    // than that for every CU, a workgroup has one CU's share of them: a wavefront's time is then its serial steps,
    // which take twice as long where four share a SIMD and the other CUs are idle.  One set, K = 8, workgroups of 16
    // wavefronts -> here, us: 1000 molecules 766 -> 452, 16 384 902 -> 499, 65 536 963 -> 550, 131 072 1036 -> 709
    const int64_t items = (s->n + 63) / 64 * s->n_cfg;
    block = 64 * (int)std::min<int64_t>(16, (items + c->n_cu - 1) / c->n_cu);
    while (block > 64 && lds_tab + (size_t)(block / 64) * lds_wave > (size_t)c->lds_max) block -= 64;
  }
  const size_t lds = lds_tab + (size_t)(block / 64) * lds_wave;
  const void *kern = grad ? (const void *)k_smooth<true> : (const void *)k_smooth<false>;
  if ((rc = lds_limit(c, kern, lds)) != CTRAJ_OK) return rc;
  if ((rc = block_ok(c, kern, block)) != CTRAJ_OK) return rc;

  SmoothArgs A{};
  A.x = s->x; A.y = s->y; A.vx = s->vx; A.vy = s->vy; A.eps = s->eps;
  A.params = s->params;
  A.n_capped = reinterpret_cast<unsigned long long *>(s->n_capped);
  A.n = s->n;
  A.items_per_cfg = (s->n + 63) / 64;
  A.n_items = A.items_per_cfg * s->n_cfg;
  A.z_src = s->z_src;
  A.sigma_vz = s->sigma_vz;
  A.inv_s = 1.0 / s->softness;
  A.n_params = np;
  A.max_steps = s->max_steps;
  A.off_end = nf;
  A.off_ck = nf + nl;
  // rows of 256 doubles per wavefront with checkpoints every K steps
  auto layout = [&](int K) {
    A.K = K;
    A.ck_per_lens = (s->max_steps + K - 1) / K;
    A.off_sub = A.off_ck + nl * A.ck_per_lens;
    A.ws_stride = (int64_t)(A.off_sub + (K > kSub ? (K + kSub - 1) / kSub : 0)) * 256;
  };
  A.rec_lds = (int)(lds_tab / sizeof(double));

  const int wpb = block / 64;
  int grid = grid_for(c, kern, block, lds, A.n_items * 64, 0);
  if (grad) {
    // Checkpoints every kSub steps leave one window per segment and the fewest steps to recompute; the
    // store then grows with the steps of the lens (1.1 GB for 4096 wavefronts and 520 steps), so it is
    // taken while it stays within 2 GiB and can be had, and the caller's interval otherwise
    const int64_t dense_max = (int64_t)2 << 30, ws_max = (int64_t)4 << 30, grain = (int64_t)64 << 20;
    const auto per_block = [&] { return A.ws_stride * 8 * wpb; };
    // keep the checkpoint/recompute store within 4 GiB
    const auto bound = [&] { grid = (int)std::min<int64_t>(grid, std::max<int64_t>(1, ws_max / per_block())); };
    bool dense = false;
    if (s->ckpt_every > kSub) {
      layout(kSub);
      dense = per_block() * grid <= dense_max &&
              extra_buf(c, c->sm_ws, (size_t)((per_block() * grid + grain - 1) / grain * grain));
    }
    if (!dense) {
      layout(s->ckpt_every);
      bound();
      const int64_t most = per_block() * grid;
      const int64_t bytes = s->ckpt_every > kSub ? most : (most + grain - 1) / grain * grain;
      if ((rc = ensure_buf(c, c->sm_ws, (size_t)bytes)) != CTRAJ_OK) return rc;
    }
    A.ws = (double *)c->sm_ws.p;
  }
  // the item counter's 256 bytes, then the partial sums
  if ((rc = ensure_buf(c, c->sm_part, 256 + (size_t)A.n_items * (np + 1) * sizeof(double))) != CTRAJ_OK) return rc;
  A.next = (unsigned long long *)c->sm_part.p;
  A.partial = (double *)((char *)c->sm_part.p + 256);
  if ((rc = ctraj_fill_i64(c, (int64_t *)A.next, 0, 1)) != CTRAJ_OK) return rc;

  const KBeam B = make_kbeam(c->d_elems, c->h_elems.data(), c->n_elems, c->phys);
  if (grad)
    hipLaunchKernelGGL(k_smooth<true>, dim3(grid), dim3(block), lds, c->stream, B, kt, A);
  else
    hipLaunchKernelGGL(k_smooth<false>, dim3(grid), dim3(block), lds, c->stream, B, kt, A);
  HIPCHK(c, hipGetLastError());
  hipLaunchKernelGGL(k_smooth_reduce, dim3(s->n_cfg, np + 1), dim3(256), 0, c->stream, (const double *)A.partial,
                     A.items_per_cfg, np, 1.0 / (double)s->n, s->J, s->grad);
  HIPCHK(c, hipGetLastError());
  return CTRAJ_OK;
}

}  // extern "C"
