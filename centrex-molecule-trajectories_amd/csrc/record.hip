// record.hip -- z-grid samples of many molecules (post_processing.py:20-140), in three kernels and a plan.
//
// A sample needs the rows of the molecule's trajectory next to its z and nothing of the other samples, so the
// walk and the sampling are separate: k_zrows walks one molecule per lane and stores its rows, k_zfaces and k_zlens
// take one sample per lane, outside and inside the lens.  What bounds them: k_zrows one molecule's serial lens
// steps, the others the bytes they write (48 per sample).  In one kernel the lane that walks writes its molecule's
// samples between its steps, from as few wavefronts as there are molecules: 37 000 x 2501 samples, 4.45 GB,
// 1.94 ms; here 0.24 + 0.87 + 0.45 (a fill of the same buffer takes 0.87).  Sampling in one kernel took 1.6 to 2.8 ms:
// with the force tables in LDS, or the lens's rows and force in the same loop (150 registers a lane), too few
// wavefronts are in flight for the loads, which wait behind the wavefront's own stores.
// k_zplan decides on the device whether they are the form for these molecules; if not, they return at once and the
// one-kernel form, which is launched last in any case, takes all of them.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <string>

#include "ctraj_device.hpp"
#include "ctraj_internal.hpp"
#include "ctraj_record.hpp"
#include "ctraj_sinks.hpp"
#include "ctraj_wave.hpp"

using namespace ctraj;

namespace {

// A molecule's rows: those at element faces, with the lens exit and once more the last row of all, with all ten
// fields; and of the rows inside the lens x, y, vx and vy (z, t and the acceleration follow from the row's number
// and position, lens_rk4).  Arrays of one value per molecule are interleaved over the 64 molecules of a wavefront.
struct ZRows {
  int4 *hdr;                 // [n] face rows up to the lens entrance, lens rows, full lens steps, face rows | state << 16
                             //     (< 0: odd); face row nb is the lens exit where the molecule got there
  int64_t *lens_at;          // [n] place of the first lens row
  double *face;              // [n / 64][n_face][10][64]; the last row at the number of face rows
  double2 *lens;             // [cap_rows][2]: molecule-major (a molecule's rows contiguous) or interleaved
  unsigned long long *used;  // lens rows given out
  const uint32_t *go;        // 0: every slot is left to the one-kernel form (k_zplan)
  uint32_t *odd;             // [0] count or ZGRID_ALL, [1 ...] slots left to the one-kernel form
  int n_face;
  int64_t cap_rows;
  int64_t s0, n;             // this slice's slots
};

// Whether a lens step of dz takes a molecule at z forward, at a step that its z resolves.
__device__ __forceinline__ bool moves_on(double dz, double z) {
  return dz > 1e-9 * __builtin_fabs(z) && dz > 1e-100 && dz < 1e100;
}

template <bool MOL>
struct RowStore {
  static constexpr bool kRows = true, kLensRows = true;
  const ZRows *Z;
  double *face;  // this lane's column
  double2 *lens = nullptr;
  int64_t at = 0;
  int nf = 0, nb = -1, nl = 0, nfull = 0;
  bool odd = false;

  __device__ __forceinline__ void put(const MState &m) {
    double *p = face + (size_t)nf * 640;
    p[0] = m.x; p[64] = m.y; p[128] = m.z; p[192] = m.vx; p[256] = m.vy; p[320] = m.vz;
    p[384] = m.ax; p[448] = m.ay; p[512] = m.az; p[576] = m.t;
  }
  __device__ __forceinline__ void row(const MState &m) {
    put(m);
    ++nf;
  }
  // Room for the lens rows of the wavefront's lanes that are here: each its own number (molecule-major), or as
  // many each as the longest (interleaved).  A molecule that is not moving forward at a step that its z
  // resolves or that finds no room left is odd: k_zplan has seen to it that there is room and that there are no such
  // molecules, except where an axial acceleration changes vz before the lens.
  __device__ __forceinline__ bool lens_begin(const MState &m, int n_full, double dz) {
    nb = nf;
    nfull = n_full;
    odd = !moves_on(dz, m.z) || (int64_t)n_full >= Z->cap_rows;
    const uint32_t rows = odd ? 0u : (uint32_t)n_full + 1u;
    // over the lanes here, bit by bit: the sum of rows (below this lane, and of all), or the largest
    uint64_t among = __builtin_amdgcn_ballot_w64(true);
    const bool first = lanes_below(among) == 0;
    uint32_t below = 0, total = 0, most = 0;
    for (int b = 31; b >= 0; --b) {
      const uint64_t has = __builtin_amdgcn_ballot_w64((rows >> b) & 1u);
      if constexpr (MOL) {
        below += (uint32_t)lanes_below(has) << b;
        total += (uint32_t)__popcll(has) << b;
      } else if (has & among) {
        most |= 1u << b;
        among &= has;
      }
    }
    const uint32_t want = MOL ? total : most * 64u;
    unsigned long long base = 0;
    if (first) base = atomicAdd(Z->used, (unsigned long long)want);
    base = uniform_u64(base);  // of the first lane here
    if (base + want > (unsigned long long)Z->cap_rows) odd = true;
    at = (int64_t)base + (MOL ? below : (uint32_t)lane_id());
    lens = Z->lens + 2 * at;
    return !odd;
  }
  __device__ __forceinline__ void lens_row(int j, double x, double y, double vx, double vy) {
    nl = j;
    lens[0] = make_double2(x, y);
    lens[1] = make_double2(vx, vy);
    lens += MOL ? 2 : 128;
  }
  __device__ __forceinline__ void lens_end(const MState &m) { row(m); }
};

// A value that the whole wavefront reads: through the constant address space it is a scalar load, which does not
// wait behind the wavefront's stores (vector memory operations complete in order) and takes no vector registers.
// What it reads was written by an earlier kernel.
template <bool UNIFORM, class T>
__device__ __forceinline__ T load(const T *p) {
#if defined(__HIP_DEVICE_COMPILE__)
  if constexpr (UNIFORM) return *(const __attribute__((address_space(4))) T *)p;
#endif
  return *p;
}

template <int FORCE, bool MOL, int KM>
__global__ void __launch_bounds__(KM == KM_CIRC ? 512 : 256) k_zrows(KBeam B, KTab KT, ctraj_record RC, ZRows Z) {
  extern __shared__ __attribute__((aligned(16))) double lds[];
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  if (load<true>(Z.go) == 0) return;
  const Tables T = stage_tables(lds, KT);
  __syncthreads();
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < Z.n; k += stride) {
    const int64_t s = Z.s0 + k;
    const int64_t i = RC.index ? RC.index[s] : s;
    MState m;
    m.x = RC.in.x[i];
    m.y = RC.in.y[i];
    m.z = RC.in.z ? RC.in.z[i] : RC.z_const;
    m.vx = RC.in.vx[i];
    m.vy = RC.in.vy[i];
    m.vz = RC.in.vz[i];
    m.t = RC.in.t ? RC.in.t[i] : RC.t_const;
    m.ax = RC.a0[0] ? RC.a0[0][i] : 0.0;
    m.ay = RC.a0[1] ? RC.a0[1][i] : -B.g;
    m.az = RC.a0[2] ? RC.a0[2][i] : 0.0;
    const int st = RC.state ? min((int)RC.state[i], B.n_states - 1) : 0;
    int label;
    uint32_t status = 0;
    WalkCounters wc{0u, 0u};
    RowStore<MOL> sk;
    sk.Z = &Z;
    sk.face = Z.face + (size_t)(k >> 6) * Z.n_face * 640 + (k & 63);
    walk<FORCE, CTRAJ_INTEG_RK4, RowStore<MOL>, KM>(B.elems, B.n_elems, T, B.g, B.cap, st, B.label_detected, m, label,
                                                    status, wc, sk);
    sk.put(m);  // the last row
    if (sk.odd) Z.odd[1 + atomicAdd(&Z.odd[0], 1u)] = (uint32_t)s;
    Z.hdr[k] = make_int4(sk.nb < 0 ? sk.nf : sk.nb, sk.nl, sk.nfull, sk.odd ? -1 : sk.nf | st << 16);
    Z.lens_at[k] = sk.at;
    if (RC.n_rows) RC.n_rows[s] = 0;  // k_zfaces and k_zlens count
    if (RC.label) RC.label[s] = label;
  }
}

// A state's force table read through the caches ([seg][4] = {A, B, C, 0}): a sample evaluates the force once, and
// four states' tables in LDS would leave a CU eight wavefronts.
struct WsMem {
  struct Pair {
    const double *p;
    __device__ __forceinline__ dbl2_t operator[](unsigned k) const { return *reinterpret_cast<const dbl2_t *>(p + 4 * (size_t)k); }
  } ab;
  struct One {
    const double *p;
    __device__ __forceinline__ double operator[](unsigned k) const { return p[4 * (size_t)k + 2]; }
  } c;
};

template <int FORCE>
__device__ __forceinline__ void lens_force(const Force<FORCE> &F, const WsMem &ws, double umax, double x, double y,
                                           double &ax, double &ay) {
  if constexpr (FORCE == CTRAJ_FORCE_WSPLINE_HEX)
    force_hex_r2(ws, umax, F.ks, F.cu, F.g, x, y, __builtin_fma(x, x, y * y), ax, ay);
  else
    force_lin(ws, umax, F.ks, F.cu, F.g, x, y, ax, ay);
}

__device__ __forceinline__ void ahead(MState &o, double zk) {
  const double dt = (zk - o.z) / o.vz;
  const double dt2 = dt * dt;
  o.x = (o.x + o.vx * dt) + (o.ax * dt2) / 2.0;
  o.y = (o.y + o.vy * dt) + (o.ay * dt2) / 2.0;
  o.vx = o.vx + o.ax * dt;
  o.vy = o.vy + o.ay * dt;
  o.vz = o.vz + o.az * dt;
  o.t = o.t + dt;
}

// The grid: z_k, and how many of the cap samples lie at or before (LE) or before z (z_k does not fall with k).
struct Grid {
  double z_start, z_step;
  int cap;
  __device__ __forceinline__ double at(int k) const { return z_start + (double)k * z_step; }
  template <bool LE>
  __device__ __forceinline__ bool in(int k, double z) const { return LE ? at(k) <= z : at(k) < z; }
  template <bool LE>
  __device__ __forceinline__ int upto(double z) const {
    const double e = (z - z_start) / z_step;
    int n = e > 0.0 ? (e < (double)cap ? (int)e : cap) : 0;
    while (n < cap && in<LE>(n, z)) ++n;
    while (n > 0 && !in<LE>(n - 1, z)) --n;
    return n;
  }
};

template <bool UNIFORM>
__device__ __forceinline__ int4 load_hdr(const int4 *p) {
  const int *q = reinterpret_cast<const int *>(p);
  return make_int4(load<UNIFORM>(q), load<UNIFORM>(q + 1), load<UNIFORM>(q + 2), load<UNIFORM>(q + 3));
}

// The face rows of one molecule (U: the same molecule in every lane).
template <bool U>
struct Faces {
  const double *p;
  int nb, nl, nfull, nf;
  __device__ __forceinline__ Faces(const ZRows &Z, int64_t k, const int4 &H)
      : p(Z.face + (size_t)(k >> 6) * Z.n_face * 640 + (k & 63)), nb(H.x), nl(H.y), nfull(H.z), nf(H.w & 0xffff) {}
  __device__ __forceinline__ double z(int q) const { return load<U>(p + (size_t)q * 640 + 128); }
  template <bool V = U>
  __device__ __forceinline__ MState get(int q) const {
    const double *a = p + (size_t)q * 640;
    MState m;
    m.x = load<V>(a); m.y = load<V>(a + 64); m.z = load<V>(a + 128);
    m.vx = load<V>(a + 192); m.vy = load<V>(a + 256); m.vz = load<V>(a + 320);
    m.ax = load<V>(a + 384); m.ay = load<V>(a + 448); m.az = load<V>(a + 512); m.t = load<V>(a + 576);
    return m;
  }
};

// The samples go by ZGridSinkT's rule, which decides each from the first row at or beyond its z and the next one:
// so a molecule's samples fall into runs, those before its first row, one exactly there, those decided at each
// face row, those inside the lens (k_zlens's), and those that no row reaches.
enum : int { RUN_BEFORE, RUN_FIRST, RUN_FACE, RUN_LENS, RUN_NONE };

template <bool U>
struct Runs {
  const Faces<U> &M;
  const Grid &G;
  double z1, dt;  // the lens end and step
  int kind, q, hi;  // the run, its face row and the sample after its last
  double z_last, zr, zn;  // the z of the last row, of this row and of the next (NaN: none, or none that can matter)
  MState prev;   // the row before this one; the last row before the first

  __device__ __forceinline__ Runs(const Faces<U> &m, const Grid &g, double z1_, double dt_) : M(m), G(g), z1(z1_), dt(dt_) {
    kind = RUN_BEFORE;
    q = 0;
    z_last = M.z(M.nf);
    hi = G.template upto<false>(M.z(0));
    zr = zn = nan64();
    prev = M.get(M.nf);
  }
  __device__ __forceinline__ double lens_z(int j) const {
    if (j > M.nfull) return z1;
    const double *e = M.p + (size_t)(M.nb - 1) * 640;  // the entrance
    return __builtin_fma((double)j, load<U>(e + 320) * dt, load<U>(e + 128));
  }
  __device__ __forceinline__ double lens_z_max() const {
    const double a = lens_z(M.nl);
    if (M.nl <= M.nfull || M.nfull == 0) return a;
    const double b = lens_z(M.nfull);
    return b > a ? b : a;
  }
  // the next run that holds a sample at or after lo
  __device__ __forceinline__ void next(int lo) {
    do {
      if (kind == RUN_BEFORE) {
        kind = RUN_FIRST;
        if (hi < G.cap && G.at(hi) == M.z(0)) ++hi;
        continue;
      }
      ++q;  // past the lens, row nb is its exit
      if (M.nl > 0 && q == M.nb) {
        kind = RUN_LENS;
        hi = max(hi, G.template upto<true>(lens_z_max()));
      } else if (q < M.nf) {
        kind = RUN_FACE;
        zr = M.z(q);
        hi = max(hi, G.template upto<true>(zr));
        if (hi > lo) {
          prev = M.get(q - 1);
          // of the rows after the entrance only the lens end of a lens without a full step can lie before it
          if (M.nl > 0 && q == M.nb - 1) zn = M.nl == 1 && M.nfull == 0 ? z1 : nan64();
          else zn = q + 1 < M.nf ? M.z(q + 1) : nan64();
        }
      } else {
        kind = RUN_NONE;
        hi = G.cap;
        return;
      }
    } while (hi <= lo);
  }
  // sample i of this run, not inside the lens; false: the rule gives none
  __device__ __forceinline__ bool sample(int i, MState &o) const {
    const double zk = G.at(i);
    if (kind == RUN_NONE || (kind == RUN_BEFORE ? z_last < zk : zk > z_last)) return false;
    const bool exact = kind == RUN_FIRST || (kind == RUN_FACE && (zk == zr || zk == zn));
    if (exact) {  // row q + 1 after the entrance: the lens exit, or the last row where the bore stopped it there
      o = M.template get<false>(kind == RUN_FIRST ? 0 : zk == zr ? q : q + 1);
    } else {
      o = prev;
      ahead(o, zk);
    }
    return true;
  }
};

// Write 64 samples of one molecule, a lane each, the first n of them, through LDS (so: 192 pairs), in stores
// that cover 1 KB each without gaps.
__device__ __forceinline__ void store_block(double2 *so, double2 *dst, int n, const MState &o) {
  const int lane = lane_id();
  so[3 * lane] = make_double2(o.x, o.y);
  so[3 * lane + 1] = make_double2(o.vx, o.vy);
  so[3 * lane + 2] = make_double2(o.vz, o.t);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int p = 0; p < 3; ++p)
    if (p * 64 + lane < 3 * n) dst[p * 64 + lane] = so[p * 64 + lane];
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ void count_written(int32_t *n_rows, int64_t s, int written) {
  if (!n_rows) return;
  for (int o = 32; o > 0; o >>= 1) written += __shfl_xor(written, o);
  if (lane_id() == 0 && written) atomicAdd(&n_rows[s], written);
}

__device__ __forceinline__ MState no_sample() {
  MState o;
  o.x = o.y = o.z = o.vx = o.vy = o.vz = o.ax = o.ay = o.az = o.t = nan64();
  return o;
}

__device__ __forceinline__ void store_field(const ctraj_record &RC, int i, int64_t s, const MState &o) {
  const size_t a = (size_t)i * RC.n + s, fs = (size_t)RC.cap * RC.n;
  RC.buf[a] = o.x; RC.buf[a + fs] = o.y; RC.buf[a + 2 * fs] = o.vx;
  RC.buf[a + 3 * fs] = o.vy; RC.buf[a + 4 * fs] = o.vz; RC.buf[a + 5 * fs] = o.t;
}

// The samples outside the lens.  MOL, buf[slot][k][6]: a wavefront takes `tile` samples of one molecule, 64 at a
// time and a lane each; else, buf[f][k][slot], `tile` samples of 64 molecules, a molecule per lane.
template <bool MOL>
__global__ void __launch_bounds__(256) k_zfaces(KBeam B, ctraj_record RC, ZRows Z, int lens_e, int tile) {
  __shared__ double2 s_out[MOL ? 4 : 1][192];
  if (load<true>(Z.go) == 0) return;
  const ctraj_elem &E = B.elems[lens_e];
  const double z1 = load<true>(&E.z1), dt = load<true>(&E.p[2]);
  const Grid G{RC.z_start, RC.z_step, RC.cap};
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int tiles = (RC.cap + tile - 1) / tile;
  const int64_t items = (MOL ? Z.n : (Z.n + 63) >> 6) * tiles, stride = (int64_t)gridDim.x * 4;
  for (int64_t w = (int64_t)blockIdx.x * 4 + wave; w < items; w += stride) {
    const int64_t grp = w / tiles;
    const int i0 = (int)(w - grp * tiles) * tile, i1 = min(i0 + tile, RC.cap);
    const int64_t k = MOL ? grp : grp * 64 + lane;
    if (k >= Z.n) continue;
    const int4 H = load_hdr<MOL>(Z.hdr + k);
    if (H.w < 0) continue;
    const int64_t s = Z.s0 + k;
    const Faces<MOL> M(Z, k, H);
    Runs<MOL> R(M, G, z1, dt);
    if (R.hi <= i0) R.next(i0);
    int written = 0;
    if constexpr (MOL) {
      for (int lo = i0; lo < i1;) {  // a run's samples in blocks of 64
        const int hi = min(R.hi, i1);
        if (R.kind != RUN_LENS) {
          for (int b = lo; b < hi; b += 64) {
            MState o = no_sample();
            if (b + lane < hi && R.sample(b + lane, o)) ++written;
            store_block(s_out[wave], reinterpret_cast<double2 *>(RC.buf) + ((size_t)s * RC.cap + b) * 3, min(64, hi - b), o);
          }
        }
        lo = hi;
        if (lo < i1) R.next(lo);
      }
      count_written(RC.n_rows, s, written);
    } else {
      for (int i = i0; i < i1; ++i) {
        if (R.hi <= i) R.next(i);
        if (R.kind == RUN_LENS) continue;
        MState o = no_sample();
        if (R.sample(i, o)) ++written;
        store_field(RC, i, s, o);
      }
      if (RC.n_rows && written) atomicAdd(&RC.n_rows[s], written);
    }
  }
}

// The samples inside the lens, of one molecule a wavefront or of 64, as k_zfaces.
template <int FORCE, bool MOL>
__global__ void __launch_bounds__(256) k_zlens(KBeam B, KTab KT, ctraj_record RC, ZRows Z, int lens_e, int tile) {
  __shared__ double2 s_out[MOL ? 4 : 1][192];
  if (load<true>(Z.go) == 0) return;
  const ctraj_elem &E = B.elems[lens_e];
  const Force<FORCE> F = make_force<FORCE>(E, B.g);
  const double z1 = E.z1, R2 = E.p[1], h = E.p[2], L = E.p[3];
  const Grid G{RC.z_start, RC.z_step, RC.cap};
  const int lane = lane_id(), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int tiles = (RC.cap + tile - 1) / tile;
  const int64_t items = (MOL ? Z.n : (Z.n + 63) >> 6) * tiles, stride = (int64_t)gridDim.x * 4;
  for (int64_t w = (int64_t)blockIdx.x * 4 + wave; w < items; w += stride) {
    const int64_t grp = w / tiles;
    const int i0 = (int)(w - grp * tiles) * tile, i1 = min(i0 + tile, RC.cap);
    const int64_t k = MOL ? grp : grp * 64 + lane;
    if (k >= Z.n) continue;
    const int4 H = load_hdr<MOL>(Z.hdr + k);
    if (H.w < 0 || H.y == 0) continue;
    const int64_t s = Z.s0 + k;
    const Faces<MOL> M(Z, k, H);
    const double *in = M.p + (size_t)(M.nb - 1) * 640;
    const double z_in = load<MOL>(in + 128), vz = load<MOL>(in + 320), t_in = load<MOL>(in + 576);
    const double dz = vz * h, inv_dz = 1.0 / dz, z_last = M.z(M.nf);
    const int n = min(M.nl, M.nfull);
    const auto lens_z = [&](int j) { return j <= M.nfull ? __builtin_fma((double)j, dz, z_in) : z1; };
    double top = lens_z(M.nl);
    if (M.nl > M.nfull && M.nfull > 0) top = lens_z(M.nfull) > top ? lens_z(M.nfull) : top;
    // the run: past what the rows up to the entrance decide
    int lo = G.template upto<false>(M.z(0));
    if (lo < G.cap && G.at(lo) == M.z(0)) ++lo;
    for (int q = 1; q < M.nb; ++q) lo = max(lo, G.template upto<true>(M.z(q)));
    const int hi = min(G.template upto<true>(top), i1);
    lo = max(lo, i0);
    const double zn = M.nb + 1 < M.nf ? M.z(M.nb + 1) : nan64();  // the row after the exit
    const double *ws = KT.ws + (size_t)(H.w >> 16) * KT.ws_nseg * 4;
    const WsMem W{{ws}, {ws}};
    const double2 *lens = Z.lens + 2 * load<MOL>(Z.lens_at + k);
    const auto sample = [&](int i, MState &o) {
      const double zk = G.at(i);
      if (zk > z_last) return false;
      // the first lens row with z >= zk: the uniform steps' z does not fall from one to the next, so the first
      // of them is found from an estimate, whose error the two loops take out
      double e = __builtin_ceil((zk - z_in) * inv_dz);
      e = e > 1.0 ? e : 1.0;
      int j = e < (double)n ? (int)e : max(n, 1);
      while (j > 1 && lens_z(j - 1) >= zk) --j;
      while (j <= n && !(lens_z(j) >= zk)) ++j;
      j = min(j, n + 1);
      bool exact = lens_z(j) == zk;
      if (!exact) {
        exact = (j < M.nl ? lens_z(j + 1) : zn) == zk;
        j += exact ? 1 : -1;
      }
      if (j == 0 || j > M.nl) {
        o = M.template get<false>(j == 0 ? M.nb - 1 : M.nb + 1);
      } else {
        const double2 *p = lens + (size_t)(j - 1) * (MOL ? 2 : 128);
        const double2 a = p[0], b = p[1];
        o.x = a.x; o.y = a.y; o.vx = b.x; o.vy = b.y; o.vz = vz;
        o.z = lens_z(j);
        if (j <= M.nfull) o.t = __builtin_fma((double)j, h, t_in);
        else o.t = __builtin_fma((double)M.nfull, h, t_in) + (L / vz - (double)M.nfull * h);
        o.ax = 0.0;
        o.ay = -B.g;
        o.az = 0.0;
        if (j <= M.nfull || __builtin_fma(o.x, o.x, o.y * o.y) > R2)
          lens_force<FORCE>(F, W, KT.umax, o.x, o.y, o.ax, o.ay);
      }
      if (!exact) ahead(o, zk);
      return true;
    };
    int written = 0;
    if constexpr (MOL) {
      for (int b = lo; b < hi; b += 64) {
        MState o = no_sample();
        if (b + lane < hi && sample(b + lane, o)) ++written;
        store_block(s_out[wave], reinterpret_cast<double2 *>(RC.buf) + ((size_t)s * RC.cap + b) * 3, min(64, hi - b), o);
      }
      count_written(RC.n_rows, s, written);
    } else {
      for (int i = lo; i < hi; ++i) {
        MState o = no_sample();
        if (sample(i, o)) ++written;
        store_field(RC, i, s, o);
      }
      if (RC.n_rows && written) atomicAdd(&RC.n_rows[s], written);
    }
  }
}

// What a run of the three kernels is for, decided before it: that the lens rows of every slice have room, that every
// molecule can be sampled by them, and that the lens rows of all are within the bounds in which they are the faster
// form (zgrid_in_two).  One workgroup a slice; the last to end decides.
struct ZPlan {
  uint32_t go, done, bad;
  unsigned long long rows;
};

struct ZPlanArgs {
  ZPlan *plan;
  unsigned long long *used;  // [slices]
  uint32_t *odd;
  int64_t slice, cap_rows;
  double h, z0;  // the lens step and entrance
  float steps;   // L / h: a molecule's steps are this over its vz
  double lo, hi;
};

template <bool MOL>
__global__ void __launch_bounds__(1024) k_zplan(ctraj_record RC, ZPlanArgs A) {
  __shared__ unsigned long long s_rows;
  __shared__ uint32_t s_bad;
  if (threadIdx.x == 0) s_rows = 0, s_bad = 0;
  __syncthreads();
  const int64_t s0 = (int64_t)blockIdx.x * A.slice, n = min(A.slice, RC.n - s0);
  unsigned long long sum = 0;
  bool bad = false;
  constexpr int AT_ONCE = 16;  // loads in flight: the workgroup is alone on its CU
  for (int64_t k0 = threadIdx.x; k0 - threadIdx.x < n; k0 += AT_ONCE * 1024) {
    double vz[AT_ONCE];
    int64_t at[AT_ONCE];
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u) at[u] = s0 + min(k0 + u * 1024, n - 1);
    if (RC.index) {
#pragma unroll
      for (int u = 0; u < AT_ONCE; ++u) at[u] = RC.index[at[u]];
    }
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u) vz[u] = RC.in.vz[at[u]];
#pragma unroll
    for (int u = 0; u < AT_ONCE; ++u) {
      const bool here = k0 + u * 1024 < n, ok = moves_on(vz[u] * A.h, A.z0);
      uint32_t rows = here && ok ? (uint32_t)fminf(A.steps * __builtin_amdgcn_rcpf((float)vz[u]), 0x1p24f) + 2u : 0u;
      bad = bad || (here && !ok);
      if constexpr (!MOL) {  // padded to the longest of the 64
        for (int o = 32; o > 0; o >>= 1) rows = max(rows, (uint32_t)__shfl_xor((int)rows, o));
      }
      sum += rows;
    }
  }
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
  if (lane_id() == 0) atomicAdd(&s_rows, sum);
  if (bad) s_bad = 1;
  __syncthreads();
  if (threadIdx.x != 0) return;
  A.used[blockIdx.x] = 0;
  uint32_t no = s_bad | (uint32_t)(s_rows > (unsigned long long)A.cap_rows);
  unsigned long long rows = s_rows;
  if (gridDim.x > 1) {
    atomicAdd(&A.plan->rows, rows);
    if (no) atomicOr(&A.plan->bad, 1u);
    __threadfence();
    if (atomicAdd(&A.plan->done, 1u) != gridDim.x - 1) return;
    __threadfence();
    rows = atomicAdd(&A.plan->rows, 0ull);
    no = atomicOr(&A.plan->bad, 0u);
  }
  const bool go = !no && (double)rows >= A.lo && (double)rows <= A.hi;
  A.plan->go = go;
  A.odd[0] = go ? 0u : ZGRID_ALL;
}

__global__ void __launch_bounds__(64) k_zclear(ZPlan *plan) {
  if (threadIdx.x == 0) plan->done = 0, plan->bad = 0, plan->rows = 0;
}

using RowsFn = void (*)(KBeam, KTab, ctraj_record, ZRows);
using FaceFn = void (*)(KBeam, ctraj_record, ZRows, int, int);
using LensFn = void (*)(KBeam, KTab, ctraj_record, ZRows, int, int);

template <int F>
RowsFn rows_kernel(bool mol, bool circ) {
  if (mol) return circ ? k_zrows<F, true, KM_CIRC> : k_zrows<F, true, KM_ALL>;
  return circ ? k_zrows<F, false, KM_CIRC> : k_zrows<F, false, KM_ALL>;
}

// Molecules walked and sampled at a time, and the lens rows kept for them (512 MiB): 409 of a molecule's own
// number each, or 512 where they are padded to the longest of 64
constexpr int64_t SLICE_MOL = ZGRID_SLICE_MOL, SLICE_FIELD = ZGRID_SLICE_FIELD;

}  // namespace

namespace ctraj {

int record_zgrid(ctraj_ctx *c, const ctraj_record &RC, int lens_e, bool circ_only, const KBeam &B, const KTab &kt,
                 size_t lds, const ZGridSteps &steps, ZGridPlan &plan) {
  plan = ZGridPlan{};
  const bool mol = RC.mode == CTRAJ_REC_ZGRID_MOL, hex = c->force == CTRAJ_FORCE_WSPLINE_HEX;
  const RowsFn kr = hex ? rows_kernel<CTRAJ_FORCE_WSPLINE_HEX>(mol, circ_only)
                        : rows_kernel<CTRAJ_FORCE_WSPLINE_LIN>(mol, circ_only);
  const FaceFn kf = mol ? k_zfaces<true> : k_zfaces<false>;
  const LensFn kl = hex ? (mol ? k_zlens<CTRAJ_FORCE_WSPLINE_HEX, true> : k_zlens<CTRAJ_FORCE_WSPLINE_HEX, false>)
                        : (mol ? k_zlens<CTRAJ_FORCE_WSPLINE_LIN, true> : k_zlens<CTRAJ_FORCE_WSPLINE_LIN, false>);
  const int n_face = 3 + 2 * c->n_elems;  // the start, two per element, the lens exit, the last
  // a slice's face rows stay below an eighth of a GiB
  const int64_t slice = std::min<int64_t>({RC.n, mol ? SLICE_MOL : SLICE_FIELD, std::max<int64_t>(64, ((int64_t)1 << 27) / (n_face * 80) & ~63LL)});
  const int64_t pad = (slice + 63) & ~(int64_t)63;
  ZRows Z{};
  Z.n_face = n_face;
  Z.cap_rows = std::min<int64_t>(ZGRID_ROWS, pad * ZGRID_ROWS_EACH);
  size_t at = 0;
  const auto place = [&](size_t bytes) {
    const size_t p = at;
    at += (bytes + 255) & ~(size_t)255;
    return p;
  };
  const int64_t slices = (RC.n + slice - 1) / slice;
  const size_t p_plan = place(sizeof(ZPlan)), p_used = place(8 * (size_t)slices),
               p_odd = place(4 * ((size_t)RC.n + 1)), p_hdr = place(16 * (size_t)pad), p_at = place(8 * (size_t)pad), p_face = place((size_t)pad * n_face * 80),
               p_lens = place((size_t)Z.cap_rows * 32);
  void *ws = nullptr;
  int rc = lds_limit(c, (const void *)kr, lds);
  if (rc) return rc;
  if (ctraj_scratch_alloc(c, at, &ws) != CTRAJ_OK) {
    (void)hipGetLastError();
    return CTRAJ_OK;  // plan.ws stays null: the one-kernel form needs no memory
  }
  char *w = (char *)ws;
  unsigned long long *used = (unsigned long long *)(w + p_used);
  ZPlan *zp = (ZPlan *)(w + p_plan);
  Z.go = &zp->go;
  Z.odd = (uint32_t *)(w + p_odd);
  Z.hdr = (int4 *)(w + p_hdr);
  Z.lens_at = (int64_t *)(w + p_at);
  Z.face = (double *)(w + p_face);
  Z.lens = (double2 *)(w + p_lens);
  // the walk: few wavefronts, spread over the CUs, unless one workgroup's tables fill a CU's LDS
  const int most = circ_only ? 512 : 256;
  int block = 64;
  while (block < most && (int64_t)block * c->n_cu * std::max<int64_t>(1, (int64_t)c->lds_max / (int64_t)std::max<size_t>(lds, 1)) < slice)
    block *= 2;
  const int tile = mol ? 512 : 16;
  const int tiles = (RC.cap + tile - 1) / tile;
  const ctraj_elem &lens = c->h_elems[lens_e];
  const ZPlanArgs plan_args{zp, used, Z.odd, slice, Z.cap_rows, lens.p[2], lens.z0, (float)(lens.p[3] / lens.p[2]),
                            steps.lo * (double)RC.n, steps.hi * (double)RC.n};
  if (slices > 1) hipLaunchKernelGGL(k_zclear, dim3(1), dim3(64), 0, c->stream, zp);
  if (mol) hipLaunchKernelGGL(k_zplan<true>, dim3((int)slices), dim3(1024), 0, c->stream, RC, plan_args);
  else hipLaunchKernelGGL(k_zplan<false>, dim3((int)slices), dim3(1024), 0, c->stream, RC, plan_args);
  hipError_t e = hipGetLastError();
  // grids for a whole slice (each asks the runtime for the occupancy, some 8 us, more than a launch)
  const int64_t items = (mol ? slice : (slice + 63) >> 6) * tiles;
  const dim3 gr(grid_for(c, (const void *)kr, block, lds, slice, 0)), gf(grid_for(c, (const void *)kf, 256, 0, items * 64, 0)),
      gl(grid_for(c, (const void *)kl, 256, 0, items * 64, 0));
  for (int64_t s0 = 0; s0 < RC.n && e == hipSuccess; s0 += slice) {
    Z.s0 = s0;
    Z.used = used + s0 / slice;
    Z.n = std::min(slice, RC.n - s0);
    hipLaunchKernelGGL(kr, gr, dim3(block), lds, c->stream, B, kt, RC, Z);
    hipLaunchKernelGGL(kf, gf, dim3(256), 0, c->stream, B, RC, Z, lens_e, tile);
    hipLaunchKernelGGL(kl, gl, dim3(256), 0, c->stream, B, kt, RC, Z, lens_e, tile);
    e = hipGetLastError();
  }
  if (e != hipSuccess) {
    (void)ctraj_scratch_free(c, ws);
    return hipfail(c, e, "record_zgrid");
  }
  plan.ws = ws;
  plan.odd = Z.odd;
  return CTRAJ_OK;
}

}  // namespace ctraj
