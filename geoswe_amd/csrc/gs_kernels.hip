// gs_kernels.hip -- MI355X (gfx950) kernels and C ABI of the fused finite-volume step.
//
// Dense layout: one wavefront owns a strip of 64 contiguous columns (60 written, two
// halo lanes on each side) and sweeps it down `tile_rows` rows. Each x-face is computed
// once and carried in registers from one row to the next; each y-face is computed once
// by the lane left of it and handed to the lane on its right with a cross-lane shuffle.
// Ghost cells are never stored: the stencil loads synthesise them from the boundary
// kinds. The residual, rain, Euler update, friction, wet/dry rule, stage boundary,
// running max and the next step's CFL wave speed are one pass; the last workgroup turns
// the wave-speed maximum into the next dt on the device (no host synchronisation).
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include <type_traits>

#include "gs_common.h"
#include "gs_wave.h"

namespace gs {

thread_local char g_err[512] = "";

// clock set-up kernels (one thread)
__global__ void k_clock_reset(GsClock* c, double t0) {
  c->t = t0;
  c->dt = 0.0;
  c->t_end = INFINITY;
  c->dt_max = 0.0;
  c->eta64 = 0.0;
  c->nsteps = 0;
  c->max_steps = INT64_MAX;
  c->lam_acc = 0ull;
  c->lam_bits = 0ull;
  c->blocks_done = 0u;
  c->status = 0;
  c->dt32 = 0.0f;
  c->rain32 = 0.0f;
  c->eta32 = 0.0f;
  c->rain_idx = 0;
  c->use_host_dt = 0;
  c->run_mode = 0;
  // the padding too, so that a clock's bytes are a function of its history alone
  for (int i = 0; i < 6; ++i) c->pad_[i] = 0;
}

__global__ void k_clock_target(GsClock* c, Plan p, double t_end, double dt_max, long long max_steps,
                               int run_mode) {
  c->t_end = t_end;
  c->dt_max = dt_max;
  c->max_steps = max_steps < 0 ? INT64_MAX : c->nsteps + max_steps;
  c->run_mode = run_mode;
  c->status &= ~GS_ST_DONE;
  const ClockIn k = clock_read(c);
  ForcIn f;
  forcing_read(p, k.t, f);
  plan_dt(c, p, k, f, c->lam_bits);
}

__global__ void k_clock_dt(GsClock* c, Plan p, double dt) {
  const ClockIn k = clock_read(c);
  ForcIn f;
  forcing_read(p, k.t, f);
  plan_host_dt(c, p, k, f, dt);
}


// ---------------------------------------------------------------------------
// dense layout
// ---------------------------------------------------------------------------
constexpr int kOut = 60;      // columns written per strip (lanes 2..61)
constexpr int kMaxWaves = 8;  // most strips per workgroup
constexpr int kBlock = 64 * kMaxWaves;

// T is the arithmetic type, S the type of the planes in memory (S = float with T = double:
// float32 planes stepped with float64 arithmetic, each value rounded once when it is stored).
template <typename T, typename S = T>
struct DenseK {
  int nx, ny, bc_x, bc_y, tile_rows, ncs, nrs, ntiles;
  int64_t pitch;
  S* buf[2][3];
  const S* bed;
  const uint8_t* flags;
  const S* ntab;
  int n_classes;
  const S* n_field;
  S* max_h;
  const uint8_t* cls;   // per-cell class plane (ids 0..255), or NULL: the flags' class bits
  T* rhs[3];
  int which;
  Phys<T> P;
  int rain_mode;  // 0 none, 1 uniform, 2 gridded
  int wave;       // kWave* flags of P
  const S* rain_frames;
  int64_t frame_stride, rain_pitch;
  int stage;
  GsClock* clock;
  Plan plan;
};

// Ghost synthesis (bc.py:50-98 state, solver.py:1466-1484 bed). Rows/columns outside the
// interior map to the interior cell the boundary kind copies; `zero` for 'fall';
// `flip` negates the normal momentum for 'wall'.
__device__ __forceinline__ int map_state(int i, int n, int bc, bool& zero, bool& flip) {
  if (i >= 0 && i < n) return i;
  switch (bc) {
    case GS_BC_PERIODIC: return i < 0 ? i + n : i - n;
    case GS_BC_WALL: flip = true; return i < 0 ? -1 - i : 2 * n - 1 - i;
    case GS_BC_FALL: zero = true; return i < 0 ? 0 : n - 1;
    default: return i < 0 ? 0 : n - 1;
  }
}
__device__ __forceinline__ int map_bed(int i, int n, int bc) {
  if (i >= 0 && i < n) return i;
  if (bc == GS_BC_PERIODIC) return i < 0 ? i + n : i - n;
  return i < 0 ? 0 : n - 1;
}

// Column part of the ghost map, fixed for a lane over the whole sweep.
struct ColMap {
  int mj, mjb;     // state column, bed column
  bool zero, flip;
};
__device__ __forceinline__ ColMap col_map(int c, int ny, int bc) {
  ColMap m;
  m.zero = false;
  m.flip = false;
  m.mj = map_state(c, ny, bc, m.zero, m.flip);
  m.mjb = map_bed(c, ny, bc);
  return m;
}

// What a tile's rows read besides the kernel argument.
template <typename T, typename S>
struct DenseTile {
  const S* qi[3];
  S* qo[3];
  const S* frame;      // gridded rain frame of this step
  const T* ntab;       // Manning n per class (LDS)
  T rain, eta, n0;     // n0: the Manning n of a domain with no classes
  int c;               // the lane's column
  bool col_ok;         // the lane writes its cell
  bool edge;           // the tile's stencils reach ghost rows or columns
  ColMap cm;
};

// One row of a lane's column as it lies in memory. The loads of a row are issued one row ahead of
// its use; what the row then needs (the ghost rules, a conversion) waits until then.
template <typename S>
struct RawRow {
  S h, hu, hv;
};

template <typename O, typename T, typename S>
__device__ __forceinline__ void load_q(const DenseK<T, S>& a, const DenseTile<T, S>& x, int i, RawRow<S>& r) {
  int mi = i;
  if (x.edge) {
    bool zx = false, fx = false;
    mi = map_state(i, a.nx, a.bc_x, zx, fx);
  }
  const int64_t row = (int64_t)mi * a.pitch;
  const O off = (O)(uint32_t)x.cm.mj * (O)sizeof(S);
  r.h = row_at(row_base(x.qi[0] + row), off);
  r.hu = row_at(row_base(x.qi[1] + row), off);
  r.hv = row_at(row_base(x.qi[2] + row), off);
}
// The cell's state from the loaded row i.
template <typename T, typename S>
__device__ __forceinline__ void use_q(const DenseK<T, S>& a, const DenseTile<T, S>& x, int i, const RawRow<S>& r, T& h,
                                      T& hu, T& hv) {
  h = (T)r.h;
  hu = (T)r.hu;
  hv = (T)r.hv;
  if (x.edge) {
    bool zx = false, fx = false;
    (void)map_state(i, a.nx, a.bc_x, zx, fx);
    if (fx) hu = -hu;
    if (x.cm.flip) hv = -hv;
    if (zx || x.cm.zero) { h = T(0); hu = T(0); hv = T(0); }
  }
}

template <typename O, typename T, typename S>
__device__ __forceinline__ S load_b(const DenseK<T, S>& a, const DenseTile<T, S>& x, int i) {
  const int mi = x.edge ? map_bed(i, a.nx, a.bc_x) : i;
  return row_at(row_base(a.bed + (int64_t)mi * a.pitch), (O)(uint32_t)x.cm.mjb * (O)sizeof(S));
}

// What a cell's update reads from its planes. Lanes that write nothing read nothing. LEAN: the
// domain has no flags, Manning, class and running-max plane and no gridded rain. The residual
// (MODE 0) takes the flags alone: its launch fills in neither the rain nor the Manning table.
template <int MODE, bool LEAN, typename T, typename S>
__device__ __forceinline__ void cell_inputs(const DenseK<T, S>& a, const DenseTile<T, S>& x, int i, T& rh, T& rhu,
                                            T& rhv, T& rr0, T& n, uint8_t& fl) {
  fl = 0;
  rr0 = rh;
  n = T(0);
  if (LEAN) {
    rr0 = rr0 + x.rain;   // + 0 without rain: rh is not -0
    n = x.n0;
    return;
  }
  const int64_t idx = (int64_t)i * a.pitch + x.c;
  if (a.flags) {
    if (x.col_ok) fl = a.flags[idx];
    if (fl & GS_FLAG_INACTIVE) { rh = T(0); rhu = T(0); rhv = T(0); }
    rr0 = rh;
  }
  if constexpr (MODE == 0) return;
  if (a.rain_mode == 1) {
    rr0 = rr0 + x.rain;
  } else if (a.rain_mode == 2) {
    if (x.col_ok) rr0 = rr0 + (T)x.frame[(int64_t)i * a.rain_pitch + x.c];
  }
  if (a.flags && (fl & GS_FLAG_INACTIVE)) rr0 = rh;
  if (a.P.friction) {
    if (a.n_field || a.cls) {
      if (x.col_ok) n = a.n_field ? (T)a.n_field[idx] : x.ntab[a.cls[idx]];
    } else {
      n = x.ntab[fl & GS_FLAG_CLASS_MASK];
    }
  }
}

// The same planes and the running maximum for one row, loaded a row ahead through buffers that start
// at the tile: a plane that is not there reads 0 on every lane, without a branch, and a row's lookups
// do not wait for the loads of the next row's state, as loads made at their use did (1021^2 with
// flags, gridded rain and running maximum, 10 steps: 305 us against 323).
template <typename S>
struct CellRow {
  uint8_t fl, cl;
  S rain, n, mh;
};
template <typename T, typename S>
struct CellBufs {
  RowBuf fl, cl, rain, n, mh;
  uint32_t c1, cs, no_fl, no_cl, no_rain, no_n, no_mh, pitch, rain_pitch;   // c1, cs: the lane's offsets
  __device__ __forceinline__ CellBufs(const DenseK<T, S>& a, const DenseTile<T, S>& x, int i0) {
    const int64_t base = (int64_t)i0 * a.pitch;
    fl = row_buf(a.flags + base);
    cl = row_buf(a.cls + base);
    rain = row_buf(x.frame + (int64_t)i0 * a.rain_pitch);
    n = row_buf(a.n_field + base);
    mh = row_buf(a.max_h + base);
    no_fl = a.flags ? 0u : kNoLane;
    no_cl = a.P.friction && a.cls && !a.n_field ? 0u : kNoLane;
    no_rain = a.rain_mode == 2 ? 0u : kNoLane;
    no_n = a.P.friction && a.n_field ? 0u : kNoLane;
    no_mh = a.max_h ? 0u : kNoLane;
    c1 = x.col_ok ? (uint32_t)x.c : kNoLane;
    cs = x.col_ok ? (uint32_t)x.c * (uint32_t)sizeof(S) : kNoLane;
    pitch = (uint32_t)a.pitch;
    rain_pitch = (uint32_t)a.rain_pitch * (uint32_t)sizeof(S);
  }
  __device__ __forceinline__ void load(int r, CellRow<S>& o) const {   // row i0 + r
    const uint32_t at = (uint32_t)r * pitch;
    row_load(fl, c1 | no_fl, at, o.fl);
    row_load(cl, c1 | no_cl, at, o.cl);
    row_load(rain, cs | no_rain, (uint32_t)r * rain_pitch, o.rain);
    row_load(n, cs | no_n, at * (uint32_t)sizeof(S), o.n);
    row_load(mh, cs | no_mh, at * (uint32_t)sizeof(S), o.mh);
  }
};
// cell_inputs from a row loaded ahead.
template <typename T, typename S>
__device__ __forceinline__ void use_cell(const DenseK<T, S>& a, const DenseTile<T, S>& x, const CellRow<S>& o, T& rh,
                                         T& rhu, T& rhv, T& rr0, T& n) {
  const lmask off = lm_of((o.fl & GS_FLAG_INACTIVE) != 0);
  T rain = a.rain_mode == 1 ? x.rain : (T)o.rain;   // 0 where there is none: rh is not -0
  if (lm_any(off)) {
    rh = lm_sel(off, T(0), rh);
    rhu = lm_sel(off, T(0), rhu);
    rhv = lm_sel(off, T(0), rhv);
    rain = lm_sel(off, T(0), rain);
  }
  rr0 = rh + rain;
  n = T(0);
  if (a.P.friction) n = a.n_field ? (T)o.n : x.ntab[a.cls ? o.cl : (o.fl & GS_FLAG_CLASS_MASK)];
}

template <bool LEAN, typename O, typename T, typename S>
__device__ __forceinline__ void cell_store(const DenseK<T, S>& a, const DenseTile<T, S>& x, int i, S h, S hu, S hv) {
  const int64_t row = (int64_t)i * a.pitch;
  const O out = (O)(uint32_t)x.c * (O)sizeof(S);
  GS_G S* r0 = row_base(x.qo[0] + row);
  GS_G S* r1 = row_base(x.qo[1] + row);
  GS_G S* r2 = row_base(x.qo[2] + row);
  if (x.col_ok) {
    if (!LEAN && a.max_h && h > a.max_h[row + x.c]) a.max_h[row + x.c] = h;
    row_at(r0, out) = h;
    row_at(r1, out) = hu;
    row_at(r2, out) = hv;
  }
}

// Rows i0 .. i_end-1 of a tile by the wavefront forms (gs_wave.h). Returns the first row that it
// leaves to dense_rows_general: one whose stencil or update holds an operand outside their
// bounds, before anything of that row is written; i_end where there is none.
template <typename T, int MODE, bool LEAN, typename S, typename O>
__device__ __forceinline__ int dense_rows(const DenseK<T, S>& a, const DenseTile<T, S>& x, const WaveC<T>& w, int i0,
                                          int i_end, lam_t<T>& lam) {
  // lanes whose cell is written, whose y-face is used and whose cell a used face reads
  const lmask act = lm_of(x.col_ok);
  const lmask yuse = act | (act >> 1), cuse = yuse | (act << 1);
  lmask odd = 0;
  const Lanes ln = lanes_of(threadIdx.x & 63);

  const S sm2 = load_b<O>(a, x, i0 - 2), sm1 = load_b<O>(a, x, i0 - 1), s0 = load_b<O>(a, x, i0),
          s1 = load_b<O>(a, x, i0 + 1);
  RawRow<S> rP, rC, rN;   // rN: the next row of the state, and sp2 the bed of the row after it
  load_q<O>(a, x, i0 - 1, rP);
  load_q<O>(a, x, i0, rC);
  load_q<O>(a, x, i0 + 1, rN);
  S sp2 = load_b<O>(a, x, i0 + 2);
  const T bm2 = (T)sm2, bm1 = (T)sm1;
  T b0 = (T)s0, bp1 = (T)s1;
  T hP, huP, hvP, uP, vP, hC, huC, hvC, uC, vC;
  use_q<T>(a, x, i0 - 1, rP, hP, huP, hvP);
  use_q<T>(a, x, i0, rC, hC, huC, hvC);
  lmask dryP, dryC;
  prims_w<T>(hP, huP, hvP, vabs(bm2) + vabs(bm1), cuse, w, uP, vP, dryP, odd);
  prims_w<T>(hC, huC, hvC, vabs(b0) + vabs(bp1), cuse, w, uC, vC, dryC, odd);
  const T zxP = w.hdx * ((T(0.5) * (b0 - bm2)) * w.ix);
  T zxC = w.hdx * ((T(0.5) * (bp1 - bm1)) * w.ix);
  FaceProd<T> fx;   // the x-face below the current row
  face_w<T>(bm1, b0, zxP, zxC, hP, hC, uP, vP, uC, vC, dryP, dryC, act, w.ix, w, fx, odd);

  // where the written lanes' results go (offsets of 32 bits within the tile)
  const RowBuf st0 = row_buf(x.qo[0] + (int64_t)i0 * a.pitch), st1 = row_buf(x.qo[1] + (int64_t)i0 * a.pitch),
                  st2 = row_buf(x.qo[2] + (int64_t)i0 * a.pitch);
  const uint32_t lane_st = x.col_ok ? (uint32_t)x.c * (uint32_t)sizeof(S) : kNoLane;
  const uint32_t pitch_st = (uint32_t)a.pitch * (uint32_t)sizeof(S);
  constexpr bool AHEAD = !LEAN && MODE == 1 && sizeof(O) == 4;   // the cells' other planes, one row ahead
  const CellBufs<T, S> cb(a, x, i0);
  CellRow<S> cr;
  if (AHEAD) cb.load(0, cr);
  take_loaded(rN.h, rN.hu, rN.hv, sp2);   // nothing is in flight when the rows begin

  // one row; false if it is left to the general functions
  auto row = [&](int i) __attribute__((always_inline)) -> bool {
    T hN, huN, hvN;
    RawRow<S> r = rN;
    S sb = sp2;
    take_loaded(r.h, r.hu, r.hv, sb);
    const int ipf = min(i + 2, i_end);   // the last rows load again what they have
    load_q<O>(a, x, ipf, rN);
    sp2 = load_b<O>(a, x, ipf + 1);
    use_q<T>(a, x, i + 1, r, hN, huN, hvN);
    const T bp2 = (T)sb;

    T uN, vN;
    lmask dryN;
    prims_w<T>(hN, huN, hvN, bp2, cuse, w, uN, vN, dryN, odd);
    // y faces of row i: lane computes its upper face (c, c+1)
    const T bl = lane_get(ln.dn, b0), br = lane_get(ln.up, b0);
    const T zy = w.hdy * ((T(0.5) * (br - bl)) * w.iy);
    const T hR = lane_get(ln.up, hC), uR = lane_get(ln.up, uC), vR = lane_get(ln.up, vC);
    const T zyR = lane_get(ln.up, zy);
    const T zxN = w.hdx * ((T(0.5) * (bp2 - b0)) * w.ix);
    FaceProd<T> fn, fy;
    face_w<T>(b0, br, zy, zyR, hC, hR, vC, uC, vR, uR, dryC, lm_upper(dryC), yuse, w.iy, w, fy, odd);
    const T lFh = lane_get(ln.dn, fy.Fh), lFN = lane_get(ln.dn, fy.FN), lFT = lane_get(ln.dn, fy.FT), lsR = lane_get(ln.dn, fy.sR);
    face_w<T>(b0, bp1, zxC, zxN, hC, hN, uC, vC, uN, vN, dryC, dryN, act, w.ix, w, fn, odd);
    T rh, rhu, rhv, rr0, n;
    uint8_t fl;
    sum_faces<T>(fn, fx, fy, lFh, lFN, lFT, lsR, rh, rhu, rhv);
    S mh = S(0);
    if (AHEAD) {
      use_cell<T, S>(a, x, cr, rh, rhu, rhv, rr0, n);
      fl = cr.fl;
      mh = cr.mh;
      cb.load(min(i + 1, i_end - 1) - i0, cr);
    } else {
      cell_inputs<MODE, LEAN, T>(a, x, i, rh, rhu, rhv, rr0, n, fl);
    }
    if (MODE == 0) {
      if (lm_any(odd)) return false;
      if (x.col_ok) {
        const int64_t idx = (int64_t)i * a.pitch + x.c;
        a.rhs[0][idx] = rh;
        a.rhs[1][idx] = rhu;
        a.rhs[2][idx] = rhv;
      }
    } else {
      T h, hu, hv, speed;
      update_w<T>(hC, huC, hvC, rr0, rhu, rhv, n, act, a.P, w, h, hu, hv, speed, odd);
      if (sizeof(O) == 8 && lm_any(odd)) return false;
      bool quick = sizeof(S) == sizeof(T) && (w.flags & kWaveLam);
      if (!LEAN && a.flags) {
        const lmask stage = lm_of((fl & GS_FLAG_STAGE) != 0);
        if (lm_any(stage)) {
          quick = false;
          const T hs = x.eta - b0;
          h = lm_sel(stage, hs > T(0) ? hs : T(0), h);
          hu = lm_sel(stage, T(0), hu);
          hv = lm_sel(stage, T(0), hv);
        }
      }
      // the stored values (one rounding each when S is narrower than T) are the state the
      // running max and the next step's wave speed see
      const S hS = (S)h, huS = (S)hu, hvS = (S)hv;
      const lam_t<T> key = quick ? lam_key_w<T>(speed) : lam_key<T>((T)hS, (T)huS, (T)hvS, a.P);
      if (sizeof(O) == 8) {
        cell_store<LEAN, O>(a, x, i, hS, huS, hvS);
        if (x.col_ok && (LEAN || !(fl & GS_FLAG_CFL_SKIP))) lam = key > lam ? key : lam;
      } else {
        // a row with an odd lane is left through the same stores, each lane's out of range, so
        // that every way to the next row's loads holds the same stores
        const bool left = lm_any(odd);
        const uint32_t at = lane_st | (left ? kNoLane : 0u), row_st = (uint32_t)(i - i0) * pitch_st;
        if (AHEAD) row_store(cb.mh, at | cb.no_mh | (hS > mh ? 0u : kNoLane), row_st, hS);
        row_store(st0, at, row_st, hS);
        row_store(st1, at, row_st, huS);
        row_store(st2, at, row_st, hvS);
        if (left) return false;
        if (x.col_ok && (LEAN || !(fl & GS_FLAG_CFL_SKIP))) lam = key > lam ? key : lam;
      }
    }

    // slide the window one row down
    hC = hN; huC = huN; hvC = hvN; uC = uN; vC = vN; zxC = zxN; dryC = dryN;
    b0 = bp1; bp1 = bp2;
    fx = fn;
    return true;
  };
  // two rows per trip, so that half of the window's moves are names instead
  int i = i0;
  while (i < i_end) {
    if (!row(i)) break;
    if (++i == i_end) break;
    if (!row(i)) break;
    ++i;
  }
  return i;
}

// The same rows by the general functions of gs_device.h, for every operand.
template <typename T, int MODE, bool LEAN, typename S, typename O>
__device__ __forceinline__ void dense_rows_general(const DenseK<T, S>& a, const DenseTile<T, S>& x, T dt, int i0,
                                                   int i_end, lam_t<T>& lam) {
  const Phys<T>& P = a.P;
  const T ix = P.inv_dx, iy = P.inv_dy, hdx = P.half_dx, hdy = P.half_dy, g = P.g, hm = P.h_min;
  const T bm2 = (T)load_b<O>(a, x, i0 - 2), bm1 = (T)load_b<O>(a, x, i0 - 1);
  T b0 = (T)load_b<O>(a, x, i0), bp1 = (T)load_b<O>(a, x, i0 + 1);
  RawRow<S> r;
  T hP, huP, hvP, uP, vP, hC, huC, hvC, uC, vC;
  load_q<O>(a, x, i0 - 1, r);
  use_q<T>(a, x, i0 - 1, r, hP, huP, hvP);
  prims(hP, huP, hvP, hm, uP, vP);
  const T gzxP = (T(0.5) * (b0 - bm2)) * ix;
  load_q<O>(a, x, i0, r);
  use_q<T>(a, x, i0, r, hC, huC, hvC);
  prims(hC, huC, hvC, hm, uC, vC);
  T gzxC = (T(0.5) * (bp1 - bm1)) * ix;
  FaceProd<T> fx;
  face_prod<T>(bm1, b0, gzxP, gzxC, hP, hC, uP, vP, uC, vC, hdx, ix, g, hm, fx);
  for (int i = i0; i < i_end; ++i) {
    const T bp2 = (T)load_b<O>(a, x, i + 2);
    T hN, huN, hvN, uN, vN;
    load_q<O>(a, x, i + 1, r);
    use_q<T>(a, x, i + 1, r, hN, huN, hvN);
    prims(hN, huN, hvN, hm, uN, vN);
    const T gzxN = (T(0.5) * (bp2 - b0)) * ix;
    const T bl = lane_lower(b0), br = lane_upper(b0);
    const T gzy = (T(0.5) * (br - bl)) * iy;
    const T hR = lane_upper(hC), uR = lane_upper(uC), vR = lane_upper(vC);
    const T gzyR = lane_upper(gzy);
    FaceProd<T> fn, fy;
    face_prod<T>(b0, bp1, gzxC, gzxN, hC, hN, uC, vC, uN, vN, hdx, ix, g, hm, fn);
    face_prod<T>(b0, br, gzy, gzyR, hC, hR, vC, uC, vR, uR, hdy, iy, g, hm, fy);
    const T lFh = lane_lower(fy.Fh), lFN = lane_lower(fy.FN), lFT = lane_lower(fy.FT), lsR = lane_lower(fy.sR);
    T rh, rhu, rhv, rr0, n;
    uint8_t fl;
    sum_faces<T>(fn, fx, fy, lFh, lFN, lFT, lsR, rh, rhu, rhv);
    cell_inputs<MODE, LEAN, T>(a, x, i, rh, rhu, rhv, rr0, n, fl);
    if (MODE == 0) {
      if (x.col_ok) {
        const int64_t idx = (int64_t)i * a.pitch + x.c;
        a.rhs[0][idx] = rh;
        a.rhs[1][idx] = rhu;
        a.rhs[2][idx] = rhv;
      }
    } else {
      S hS = S(0), huS = S(0), hvS = S(0);
      if (x.col_ok) {
        T h, hu, hv;
        update<T>(hC, huC, hvC, rr0, rhu, rhv, dt, n, P, h, hu, hv);
        if (fl & GS_FLAG_STAGE) {
          const T hs = x.eta - b0;
          h = hs > T(0) ? hs : T(0);
          hu = T(0);
          hv = T(0);
        }
        hS = (S)h;
        huS = (S)hu;
        hvS = (S)hv;
        if (!(fl & GS_FLAG_CFL_SKIP)) {
          const lam_t<T> key = lam_key<T>((T)hS, (T)huS, (T)hvS, P);
          lam = key > lam ? key : lam;
        }
      }
      cell_store<LEAN, O>(a, x, i, hS, huS, hvS);
    }
    hC = hN; huC = huN; hvC = hvN; uC = uN; vC = vN; gzxC = gzxN;
    b0 = bp1; bp1 = bp2;
    fx = fn;
  }
}

// MODE 0: residual into a.rhs; MODE 1: fused step. LEAN: see cell_inputs. O: byte offset of a column (row_at).
// The lean float64 sweeps are held to 128 VGPRs, 4 wavefronts per SIMD instead of 3 (a few registers
// spilled outside the row loop): 1537 x 2111 float64 466 against 475 us, 1999 x 2003 float64 on
// float32 planes 569 against 591, both for 6 steps.
template <typename T, int MODE, bool LEAN, typename S, typename O>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(LEAN ? (sizeof(T) == 4 ? 6 : 4) : 1)))
void k_dense_sweep(DenseK<T, S> a) {
  int par = 0;
  T dt = T(0);
  DenseTile<T, S> x;
  x.rain = T(0);
  x.eta = T(0);
  int ridx = 0;
  if (MODE == 1) {
    const GsClock* c = a.clock;
    if (c->status & GS_ST_DONE) return;  // the whole grid sees the same clock
    par = (int)(c->nsteps & 1);
    ridx = c->rain_idx;
    if (sizeof(T) == 4) {
      dt = (T)c->dt32;
      x.rain = a.rain_mode == 1 ? (T)c->rain32 : T(0);
      x.eta = (T)c->eta32;
    } else {
      dt = (T)c->dt;
      x.rain = a.rain_mode == 1 ? (T)a.plan.rain_rate[ridx] : T(0);
      x.eta = (T)c->eta64;
    }
  } else {
    par = a.which;
  }
  x.n0 = T(0);
  x.ntab = nullptr;
  if (LEAN) {
    if (a.P.friction) x.n0 = (T)a.ntab[0];
  } else if (MODE == 1) {
    __shared__ T s_ntab[GS_MAX_CLASSES];
    for (int k = (int)threadIdx.x; k < a.n_classes; k += (int)blockDim.x) s_ntab[k] = (T)a.ntab[k];
    __syncthreads();
    x.ntab = s_ntab;
  }

  // the buffers by value: an index into the argument's table at run time would put it in
  // private memory
  for (int k = 0; k < 3; ++k) {
    x.qi[k] = par ? a.buf[1][k] : a.buf[0][k];
    x.qo[k] = par ? a.buf[0][k] : a.buf[1][k];
  }
  x.frame = (MODE == 1 && a.rain_mode == 2) ? a.rain_frames + (int64_t)ridx * a.frame_stride : nullptr;

  // XCD-aware order: workgroups are dealt round-robin to the 8 XCDs; give each XCD a
  // contiguous range of tiles so neighbouring strips share that XCD's L2.
  const unsigned nb = gridDim.x, b = blockIdx.x;
  const unsigned qd = nb / 8u, rm = nb % 8u, xcd = b % 8u, kk = b / 8u;
  const unsigned lb = (xcd < rm) ? xcd * (qd + 1u) + kk : rm * (qd + 1u) + (xcd - rm) * qd + kk;
  const int lane = threadIdx.x & 63;
  // the wavefront index as a scalar: tile, rows and row addresses are then uniform values
  const int tile = (int)(lb * (blockDim.x >> 6)) + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  lam_t<T> lam = 0;

  if (tile < a.ntiles) {
    const int rs = __builtin_amdgcn_readfirstlane(tile / a.ncs), cs = tile - rs * a.ncs;
    x.c = cs * kOut + lane - 2;
    const int cl = x.c < -2 ? -2 : (x.c > a.ny + 1 ? a.ny + 1 : x.c);   // loads stay within one ghost pair
    int i = rs * a.tile_rows;
    const int i_end = min(i + a.tile_rows, a.nx);
    x.col_ok = (lane >= 2) && (lane < 2 + kOut) && (x.c < a.ny);
    x.edge = cs == 0 || (cs + 1) * kOut + 2 > a.ny || i < 2 || i_end + 2 > a.nx;
    x.cm = col_map(cl, a.ny, a.bc_y);
    if (a.wave & kWaveFast) {
      const WaveC<T> w = wave_consts<T>(a.P, dt, a.wave);
      DenseTile<T, S> xv = x;
      xv.rain = vreg(x.rain);
      xv.n0 = vreg(x.n0);
      i = __builtin_amdgcn_readfirstlane(dense_rows<T, MODE, LEAN, S, O>(a, xv, w, i, i_end, lam));
    }
    if (i < i_end) dense_rows_general<T, MODE, LEAN, S, O>(a, x, dt, i, i_end, lam);
  }
  if (MODE == 1) grid_reduce_and_plan(lam, a.clock, a.plan, true);
}

// CFL wave speed of the current dense state, then plan dt (no time advance).
template <typename T, typename S = T>
__global__ __launch_bounds__(256) void k_dense_cfl(DenseK<T, S> a) {
  const int par = (int)(a.clock->nsteps & 1);
  S* const* q = a.buf[par];
  lam_t<T> lam = 0;
  const int64_t n = (int64_t)a.nx * a.ny;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
       k += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = k / a.ny, j = k - i * a.ny;
    const int64_t idx = i * a.pitch + j;
    if (a.flags && (a.flags[idx] & GS_FLAG_CFL_SKIP)) continue;
    const lam_t<T> l = lam_key<T>((T)q[0][idx], (T)q[1][idx], (T)q[2][idx], a.P);
    lam = l > lam ? l : lam;
  }
  grid_reduce_and_plan(lam, a.clock, a.plan, false);
}

// Rows per tile. A tile costs about 1.3 rows beside its own (the rows above it, the first x-face),
// so tall tiles do the least work; but a wavefront takes about 1.4 us per row by itself, so a grid
// that does not fill the GPU several times over wants short ones, and as many wavefronts as there
// are SIMDs. Measured best heights (float32): 1 row on 128^2 and 256^2, 3 on 500 x 517, 5 on
// 1024^2, 6-12 on 2000^2, 16 on 4096^2, 24-32 on 8192 x 8000, 32-64 on 640 M cells; float64 within
// 4 % of its best at the same heights. 1.5 (cells/65536)^0.4 follows them. (With at least 16 rows
// always, 500 x 517 took 30 us a step against 13.2, 1024^2 33 us against 21.) The bands are then
// made even.
static int pick_tile_rows(int nx, int ny, int req) {
  if (req > 0) return req;
  const double cells = (double)nx * (double)ny;
  int rows = (int)(1.5 * pow(cells / 65536.0, 0.4) + 0.5);
  rows = rows < 1 ? 1 : (rows > 64 ? 64 : rows);
  const int bands = (nx + rows - 1) / rows;
  return (nx + bands - 1) / bands;
}

// Wavefronts per workgroup: 8 for the short tiles of small float32 grids, else 4. Each workgroup
// makes two atomics on the clock's line, which the line takes one after the other (5.8 ns each):
// 1024^2 in 5-row tiles 21.0 us with 8 against 25.1 us with 4. Grids of more tiles hide them, and
// a workgroup of 4 fills the last free wavefront slots better (8192 x 8000: 577 against 592 us);
// so do the 12 resident wavefronts of a float64 CU.
static int tile_waves(int ntiles, size_t arith) {
  return arith == 4 && ntiles < 16384 ? kMaxWaves : 4;
}

template <typename T, typename S = T>
static int build_dense(const GsDense* d, const GsPhys* p, const GsForcing& f, GsClock* clk, DenseK<T, S>& a,
                       bool need_clock) {
  if (!d) return fail(GS_E_ARG, "dense descriptor is NULL");
  if (d->nx < 4 || d->ny < 4) return fail(GS_E_RANGE, "dense grid needs nx, ny >= 4 (got %d x %d)", d->nx, d->ny);
  if (d->pitch < d->ny) return fail(GS_E_ARG, "pitch %lld < ny %d", (long long)d->pitch, d->ny);
  if ((int64_t)d->nx * d->pitch > ((int64_t)1 << 40)) return fail(GS_E_RANGE, "grid too large");
  if (d->bc_x < 0 || d->bc_x > 3 || d->bc_y < 0 || d->bc_y > 3) return fail(GS_E_ARG, "bad boundary kind");
  if (!d->bed) return fail(GS_E_ARG, "bed is NULL");
  for (int s = 0; s < 2; ++s)
    for (int k = 0; k < 3; ++k)
      if (!d->q[s][k]) return fail(GS_E_ARG, "state plane q[%d][%d] is NULL", s, k);
  int rc = check_phys(p);
  if (rc) return rc;
  rc = check_forcing(f);
  if (rc) return rc;
  if (p->friction && !d->ntab && !d->n_field) return fail(GS_E_ARG, "friction needs ntab or n_field");
  if (need_clock && !clk) return fail(GS_E_ARG, "clock is NULL");
  memset(&a, 0, sizeof a);
  a.nx = d->nx;
  a.ny = d->ny;
  a.bc_x = d->bc_x;
  a.bc_y = d->bc_y;
  a.pitch = d->pitch;
  a.ncs = (d->ny + kOut - 1) / kOut;
  a.tile_rows = pick_tile_rows(d->nx, d->ny, d->tile_rows);
  a.nrs = (d->nx + a.tile_rows - 1) / a.tile_rows;
  if ((int64_t)a.ncs * a.nrs > (int64_t)INT32_MAX / 2) return fail(GS_E_RANGE, "too many tiles");
  a.ntiles = a.ncs * a.nrs;
  for (int s = 0; s < 2; ++s)
    for (int k = 0; k < 3; ++k) a.buf[s][k] = (S*)d->q[s][k];
  a.bed = (const S*)d->bed;
  a.flags = d->flags;
  a.ntab = (const S*)d->ntab;
  a.n_classes = d->ntab ? (p->n_classes > 0 ? p->n_classes : 1) : 0;
  a.n_field = (const S*)d->n_field;
  a.cls = d->cls;
  a.max_h = (S*)d->max_h;
  a.P = make_phys<T>(*p, d->dx, d->dy);
  a.wave = wave_flags<T>(a.P, false);
  a.rain_mode = f.n_rain > 0 ? (f.rain_gridded ? 2 : 1) : 0;
  a.rain_frames = (const S*)f.rain_frames;
  a.frame_stride = f.rain_frame_stride;
  a.rain_pitch = f.rain_row_pitch;
  a.stage = f.n_stage > 0;
  a.clock = clk;
  a.plan = make_plan(*p, f);
  return GS_OK;
}

// Tiles of 2 GiB or more (per plane) take the sweep with 64-bit offsets.
template <typename T, typename S>
static bool wide_rows(const DenseK<T, S>& a) {
  const int64_t pitch = a.rain_mode == 2 && a.rain_pitch > a.pitch ? a.rain_pitch : a.pitch;
  return pitch * (int64_t)sizeof(S) >= ((int64_t)1 << 31) / a.tile_rows;
}

template <typename T, typename S = T>
static int dense_step_t(const GsDense* d, const GsPhys* p, GsForcing f, GsClock* clk, hipStream_t s) {
  DenseK<T, S> a;
  int rc = build_dense<T, S>(d, p, f, clk, a, true);
  if (rc) return rc;
  const int waves = tile_waves(a.ntiles, sizeof(T));
  const dim3 grid((unsigned)((a.ntiles + waves - 1) / waves)), block(64 * waves);
  const bool lean = !a.flags && !a.n_field && !a.cls && !a.max_h && a.rain_mode != 2;
  if (wide_rows(a)) hipLaunchKernelGGL((k_dense_sweep<T, 1, false, S, uint64_t>), grid, block, 0, s, a);
  else if (lean) hipLaunchKernelGGL((k_dense_sweep<T, 1, true, S, uint32_t>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_dense_sweep<T, 1, false, S, uint32_t>), grid, block, 0, s, a);
  GS_HIP(hipGetLastError(), "k_dense_sweep launch");
  return GS_OK;
}

template <typename T, typename S = T>
static int dense_residual_t(const GsDense* d, const GsPhys* p, int which, void* r0, void* r1, void* r2,
                            hipStream_t s) {
  GsForcing f;
  memset(&f, 0, sizeof f);
  DenseK<T, S> a;
  int rc = build_dense<T, S>(d, p, f, nullptr, a, false);
  if (rc) return rc;
  if (which < 0 || which > 1) return fail(GS_E_ARG, "which must be 0 or 1");
  if (!r0 || !r1 || !r2) return fail(GS_E_ARG, "residual planes are NULL");
  a.which = which;
  a.rhs[0] = (T*)r0;
  a.rhs[1] = (T*)r1;
  a.rhs[2] = (T*)r2;
  // MODE 0 writes qout = buf[which ^ 1] never; buf[par ^ 1] is unused there
  const int waves = tile_waves(a.ntiles, sizeof(T));
  const dim3 grid((unsigned)((a.ntiles + waves - 1) / waves)), block(64 * waves);
  if (wide_rows(a)) hipLaunchKernelGGL((k_dense_sweep<T, 0, false, S, uint64_t>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((k_dense_sweep<T, 0, false, S, uint32_t>), grid, block, 0, s, a);
  GS_HIP(hipGetLastError(), "k_dense_sweep(residual) launch");
  return GS_OK;
}

template <typename T, typename S = T>
static int dense_cfl_t(const GsDense* d, const GsPhys* p, GsForcing f, GsClock* clk, hipStream_t s) {
  DenseK<T, S> a;
  int rc = build_dense<T, S>(d, p, f, clk, a, true);
  if (rc) return rc;
  const int64_t n = (int64_t)a.nx * a.ny;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL((k_dense_cfl<T, S>), dim3((unsigned)blocks), dim3(256), 0, s, a);
  GS_HIP(hipGetLastError(), "k_dense_cfl launch");
  return GS_OK;
}

}  // namespace gs

using namespace gs;

extern "C" {

int gs_version(void) { return GS_ABI_VERSION; }
const char* gs_last_error(void) { return g_err; }

int gs_get_device_count(int* n) {
  if (!n) return fail(GS_E_ARG, "n is NULL");
  GS_HIP(hipGetDeviceCount(n), "hipGetDeviceCount");
  return GS_OK;
}
int gs_set_device(int dev) {
  GS_HIP(hipSetDevice(dev), "hipSetDevice");
  return GS_OK;
}

int gs_malloc(void** ptr, size_t bytes) {
  if (!ptr) return fail(GS_E_ARG, "ptr is NULL");
  *ptr = nullptr;
  if (bytes == 0) bytes = 256;
  GS_HIP(hipMalloc(ptr, bytes), "hipMalloc");
  return GS_OK;
}
int gs_free(void* ptr) {
  if (ptr) GS_HIP(hipFree(ptr), "hipFree");
  return GS_OK;
}
int gs_memcpy_h2d(void* dst, const void* src, size_t bytes, void* stream) {
  if (!bytes) return GS_OK;
  GS_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t)stream), "hipMemcpyAsync h2d");
  return GS_OK;
}
int gs_memcpy_d2h(void* dst, const void* src, size_t bytes, void* stream) {
  if (!bytes) return GS_OK;
  GS_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, (hipStream_t)stream), "hipMemcpyAsync d2h");
  return GS_OK;
}
int gs_memcpy_d2d(void* dst, const void* src, size_t bytes, void* stream) {
  if (!bytes) return GS_OK;
  GS_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToDevice, (hipStream_t)stream), "hipMemcpyAsync d2d");
  return GS_OK;
}
int gs_memcpy2d(void* dst, size_t dpitch, const void* src, size_t spitch, size_t width, size_t height, int kind,
                void* stream) {
  hipMemcpyKind k = kind == 1 ? hipMemcpyHostToDevice : (kind == 2 ? hipMemcpyDeviceToHost : hipMemcpyDeviceToDevice);
  if (kind < 1 || kind > 3) return fail(GS_E_ARG, "memcpy2d kind must be 1, 2 or 3");
  if (!width || !height) return GS_OK;
  GS_HIP(hipMemcpy2DAsync(dst, dpitch, src, spitch, width, height, k, (hipStream_t)stream), "hipMemcpy2DAsync");
  return GS_OK;
}
int gs_memset(void* dst, int value, size_t bytes, void* stream) {
  if (!bytes) return GS_OK;
  GS_HIP(hipMemsetAsync(dst, value, bytes, (hipStream_t)stream), "hipMemsetAsync");
  return GS_OK;
}
int gs_stream_create(void** stream) {
  if (!stream) return fail(GS_E_ARG, "stream is NULL");
  hipStream_t s;
  GS_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking), "hipStreamCreate");
  *stream = (void*)s;
  return GS_OK;
}
int gs_stream_destroy(void* stream) {
  if (stream) GS_HIP(hipStreamDestroy((hipStream_t)stream), "hipStreamDestroy");
  return GS_OK;
}
int gs_stream_synchronize(void* stream) {
  GS_HIP(hipStreamSynchronize((hipStream_t)stream), "hipStreamSynchronize");
  return GS_OK;
}
int gs_event_create(void** ev) {
  if (!ev) return fail(GS_E_ARG, "ev is NULL");
  hipEvent_t e;
  GS_HIP(hipEventCreate(&e), "hipEventCreate");
  *ev = (void*)e;
  return GS_OK;
}
int gs_event_destroy(void* ev) {
  if (ev) GS_HIP(hipEventDestroy((hipEvent_t)ev), "hipEventDestroy");
  return GS_OK;
}
int gs_event_record(void* ev, void* stream) {
  GS_HIP(hipEventRecord((hipEvent_t)ev, (hipStream_t)stream), "hipEventRecord");
  return GS_OK;
}
int gs_event_elapsed_ms(float* ms, void* start, void* stop) {
  if (!ms) return fail(GS_E_ARG, "ms is NULL");
  GS_HIP(hipEventElapsedTime(ms, (hipEvent_t)start, (hipEvent_t)stop), "hipEventElapsedTime");
  return GS_OK;
}

int gs_clock_reset(GsClock* clock_dev, double t0, void* stream) {
  if (!clock_dev) return fail(GS_E_ARG, "clock is NULL");
  hipLaunchKernelGGL(k_clock_reset, dim3(1), dim3(1), 0, (hipStream_t)stream, clock_dev, t0);
  GS_HIP(hipGetLastError(), "k_clock_reset launch");
  return GS_OK;
}

int gs_clock_set_target(GsClock* clock_dev, double t_end, double dt_max, int64_t max_steps, const GsPhys* phys,
                        GsForcing forc, void* stream) {
  if (!clock_dev) return fail(GS_E_ARG, "clock is NULL");
  int rc = check_phys(phys);
  if (rc) return rc;
  rc = check_forcing(forc);
  if (rc) return rc;
  const int run_mode = isfinite(t_end) ? 1 : 0;
  hipLaunchKernelGGL(k_clock_target, dim3(1), dim3(1), 0, (hipStream_t)stream, clock_dev, make_plan(*phys, forc),
                     t_end, dt_max, (long long)max_steps, run_mode);
  GS_HIP(hipGetLastError(), "k_clock_target launch");
  return GS_OK;
}

int gs_clock_set_dt(GsClock* clock_dev, double dt, const GsPhys* phys, GsForcing forc, void* stream) {
  if (!clock_dev) return fail(GS_E_ARG, "clock is NULL");
  if (!(dt >= 0.0) || isinf(dt)) return fail(GS_E_ARG, "dt must be finite and >= 0");
  int rc = check_phys(phys);
  if (rc) return rc;
  rc = check_forcing(forc);
  if (rc) return rc;
  hipLaunchKernelGGL(k_clock_dt, dim3(1), dim3(1), 0, (hipStream_t)stream, clock_dev, make_plan(*phys, forc), dt);
  GS_HIP(hipGetLastError(), "k_clock_dt launch");
  return GS_OK;
}

int gs_dense_step(const GsDense* d, const GsPhys* phys, GsForcing forc, GsClock* clock_dev, void* stream) {
  if (!d) return fail(GS_E_ARG, "dense descriptor is NULL");
  if (d->dtype == GS_F32) return dense_step_t<float>(d, phys, forc, clock_dev, (hipStream_t)stream);
  if (d->dtype == GS_F64) return dense_step_t<double>(d, phys, forc, clock_dev, (hipStream_t)stream);
  if (d->dtype == GS_F32X64) return dense_step_t<double, float>(d, phys, forc, clock_dev, (hipStream_t)stream);
  return fail(GS_E_DTYPE, "unsupported dtype %d", d->dtype);
}

int gs_dense_residual(const GsDense* d, const GsPhys* phys, int which, void* rhs0, void* rhs1, void* rhs2,
                      void* stream) {
  if (!d) return fail(GS_E_ARG, "dense descriptor is NULL");
  if (d->dtype == GS_F32) return dense_residual_t<float>(d, phys, which, rhs0, rhs1, rhs2, (hipStream_t)stream);
  if (d->dtype == GS_F64) return dense_residual_t<double>(d, phys, which, rhs0, rhs1, rhs2, (hipStream_t)stream);
  if (d->dtype == GS_F32X64)
    return dense_residual_t<double, float>(d, phys, which, rhs0, rhs1, rhs2, (hipStream_t)stream);
  return fail(GS_E_DTYPE, "unsupported dtype %d", d->dtype);
}

int gs_dense_cfl(const GsDense* d, const GsPhys* phys, GsForcing forc, GsClock* clock_dev, void* stream) {
  if (!d) return fail(GS_E_ARG, "dense descriptor is NULL");
  if (d->dtype == GS_F32) return dense_cfl_t<float>(d, phys, forc, clock_dev, (hipStream_t)stream);
  if (d->dtype == GS_F64) return dense_cfl_t<double>(d, phys, forc, clock_dev, (hipStream_t)stream);
  if (d->dtype == GS_F32X64) return dense_cfl_t<double, float>(d, phys, forc, clock_dev, (hipStream_t)stream);
  return fail(GS_E_DTYPE, "unsupported dtype %d", d->dtype);
}

}  // extern "C"
