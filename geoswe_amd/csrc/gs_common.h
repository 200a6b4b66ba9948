// gs_common.h -- pieces shared by the layout kernels: error reporting, the device-side
// step scheduler (the reference's host dt arithmetic moved onto the GPU) and the
// last-workgroup grid reduction of the CFL wave speed.
#pragma once

#include <hip/hip_runtime.h>

#include <math.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

#include "gs_device.h"

namespace gs {

// ---------------------------------------------------------------------------
// error reporting
// ---------------------------------------------------------------------------
extern thread_local char g_err[512];

static inline int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof g_err, fmt, ap);
  va_end(ap);
  return code;
}

static inline int hip_fail(hipError_t e, const char* what) {
  snprintf(g_err, sizeof g_err, "%s: %s", what, hipGetErrorString(e));
  return -(int)e;
}

#define GS_HIP(call, what)                       \
  do {                                           \
    hipError_t _e = (call);                      \
    if (_e != hipSuccess) return hip_fail(_e, what); \
  } while (0)

// ---------------------------------------------------------------------------
// device-side scheduling (Solver2D.run / cfl_dt host arithmetic, on the device)
// ---------------------------------------------------------------------------
struct Plan {
  double cfl, dmin, lam_floor;
  int n_rain, n_stage;
  const double* rain_t;
  const double* rain_rate;
  const double* rain_cap;
  const double* stage_t;
  const double* stage_v;
};

static inline Plan make_plan(const GsPhys& p, const GsForcing& f) {
  Plan pl;
  pl.cfl = p.cfl;
  pl.dmin = p.dmin;
  pl.lam_floor = p.lam_floor;
  pl.n_rain = f.n_rain;
  pl.n_stage = f.n_stage;
  pl.rain_t = f.rain_t;
  pl.rain_rate = f.rain_rate;
  pl.rain_cap = f.rain_cap;
  pl.stage_t = f.stage_t;
  pl.stage_v = f.stage_v;
  return pl;
}

// The number of entries of a[lo, hi) that `before` holds for, plus lo (it holds for a prefix of the
// ascending table). Eight probes a round: a table of 400 takes 3 rounds of loads, where halving
// took 9, and the last workgroup of a step waits for each round.
template <typename F>
__device__ __forceinline__ int table_count(const double* a, int lo, int hi, F before) {
  while (lo < hi) {
    const int step = (hi - lo + 8) / 9;
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = a[min(lo + (k + 1) * step, hi) - 1];
    int c = 0;
#pragma unroll
    for (int k = 0; k < 8; ++k) c += (lo + (k + 1) * step <= hi && c == k && before(v[k])) ? 1 : 0;
    const int end = lo + (c + 1) * step - 1;   // the first probe that fails, if there is one
    if (c < 8 && end < hi) hi = end;
    lo += c * step;
  }
  return lo;
}

// bisect_right(a, x) - 1, clamped to [0, n-1] (forcing.py:198-199)
__device__ __forceinline__ int seg_index(const double* a, int n, double x) {
  const int idx = table_count(a, 0, n, [x](double v) { return !(x < v); }) - 1;
  return idx < 0 ? 0 : idx;
}

// The stage table around time t: what StageBoundary.stage_at_time (forcing.py:315-347) needs at a
// time a little later, loaded before that time is known.
struct StageSpot {
  int k;                        // entries before t
  double t0, t1, t2, s0, s1, s2;   // entries k-1, k and k+1, as far as there are
  double t_first, s_first, t_last, s_last;
};
__device__ __forceinline__ void stage_spot(const double* ts, const double* sv, int n, double t, StageSpot& s) {
  s.t_first = ts[0];
  s.s_first = sv[0];
  s.t_last = ts[n - 1];
  s.s_last = sv[n - 1];
  s.k = table_count(ts, 0, n, [t](double v) { return v < t; });
  const int i0 = max(s.k - 1, 0), i1 = min(s.k, n - 1), i2 = min(s.k + 1, n - 1);
  s.t0 = ts[i0];
  s.t1 = ts[i1];
  s.t2 = ts[i2];
  s.s0 = sv[i0];
  s.s1 = sv[i1];
  s.s2 = sv[i2];
}
__device__ __forceinline__ double stage_at(const StageSpot& s, const double* ts, const double* sv, int n, double t) {
  if (t <= s.t_first) return s.s_first;
  if (t >= s.t_last) return s.s_last;
  // bisect_left in the entries at hand, else in the table (where t has passed the next entry but
  // one, or lies before the spot's time)
  double t0, t1, s0, s1;
  if (s.k >= 1 && s.k < n && s.t0 < t && t <= s.t1) {
    t0 = s.t0; t1 = s.t1; s0 = s.s0; s1 = s.s1;
  } else if (s.k + 1 < n && s.t1 < t && t <= s.t2) {
    t0 = s.t1; t1 = s.t2; s0 = s.s1; s1 = s.s2;
  } else {
    const int i = table_count(ts, 0, n, [t](double v) { return v < t; });
    t0 = ts[i - 1]; t1 = ts[i]; s0 = sv[i - 1]; s1 = sv[i];
  }
  const double w = (t - t0) / (t1 - t0);
  return s0 + w * (s1 - s0);
}

// What the next step's plan reads of the clock.
struct ClockIn {
  double t, dt, t_end, dt_max;
  int64_t nsteps, max_steps;
  int status, run_mode;
};
__device__ __forceinline__ ClockIn clock_read(const GsClock* c) {
  return {c->t, c->dt, c->t_end, c->dt_max, c->nsteps, c->max_steps, c->status, c->run_mode};
}

// Forcing values of the step that starts at t with step dt.
struct ForcIn {
  int ridx;
  double rate, cap;
  StageSpot stage;
};
__device__ __forceinline__ void forcing_read(const Plan& p, double t, ForcIn& f) {
  f.ridx = 0;
  if (p.n_rain > 0) f.ridx = seg_index(p.rain_t, p.n_rain, t);
  if (p.n_stage > 0) stage_spot(p.stage_t, p.stage_v, p.n_stage, t, f.stage);
  if (p.n_rain > 0) {
    f.rate = p.rain_rate[f.ridx];
    f.cap = p.rain_cap[f.ridx];
  }
}
__device__ __forceinline__ void plan_forcing(GsClock* c, const Plan& p, const ForcIn& f, double t, double dt) {
  c->rain_idx = f.ridx;
  c->rain32 = p.n_rain > 0 ? (float)f.rate : 0.0f;
  if (p.n_stage > 0) {
    const double e = stage_at(f.stage, p.stage_t, p.stage_v, p.n_stage, t + dt);
    c->eta64 = e;
    c->eta32 = (float)e;
  }
}

// dt from the wave speed of the current state (solver.py:2657-2666) and, in run mode,
// the rain-film cap, dt_max and the clip to t_end (solver.py:2990-2999, 3005-3027).
// k: the clock, at the state's time and step count; f: forcing_read of that time.
__device__ __forceinline__ void plan_dt(GsClock* c, const Plan& p, const ClockIn& k, const ForcIn& f, uint64_t lam_bits) {
  int st = k.status & ~GS_ST_DONE;
  double lam = __longlong_as_double((long long)lam_bits);
  if (!(lam == lam) || isinf(lam)) {
    c->status = st | GS_ST_NONFINITE | GS_ST_DONE;
    return;
  }
  if (lam < p.lam_floor) lam = p.lam_floor;
  double dt = p.cfl * p.dmin / (lam + 1.0e-12);
  if (k.run_mode) {
    if (p.n_rain > 0 && f.cap < dt) dt = f.cap;
    if (k.dt_max > 0.0 && dt > k.dt_max) dt = k.dt_max;
    if (k.t + dt > k.t_end) dt = k.t_end - k.t;
    if (!(k.t < k.t_end - 1.0e-12)) st |= GS_ST_DONE;
  }
  if (k.nsteps >= k.max_steps) st |= GS_ST_DONE;
  c->dt = dt;
  c->dt32 = (float)dt;
  c->use_host_dt = 0;
  c->status = st;
  plan_forcing(c, p, f, k.t, dt);
}

// A dt that the host gives (gs_clock_set_dt, or next_dt of the step before).
__device__ __forceinline__ void plan_host_dt(GsClock* c, const Plan& p, const ClockIn& k, const ForcIn& f, double dt) {
  c->dt = dt;
  c->dt32 = (float)dt;
  c->use_host_dt = 1;
  int st = k.status & ~GS_ST_DONE;
  if ((st & GS_ST_NONFINITE) || k.nsteps >= k.max_steps) st |= GS_ST_DONE;
  c->status = st;
  plan_forcing(c, p, f, k.t, dt);
}

// Called by the last workgroup of a step (advance) or of a CFL pass. k: the clock before it; the
// forcing tables are searched while the grid's maximum is on its way. next_dt > 0: the next step's dt,
// given by the host (as gs_clock_set_dt would after the step).
__device__ __forceinline__ void plan_finish(GsClock* c, const Plan& p, ClockIn k, bool advance, double next_dt = 0.0) {
  const uint64_t lam = __hip_atomic_load(&c->lam_acc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (advance) {
    k.t = k.t + k.dt;
    k.nsteps = k.nsteps + 1;
  }
  ForcIn f;
  forcing_read(p, k.t, f);
  if (advance) {
    c->t = k.t;
    c->nsteps = k.nsteps;
  }
  c->lam_bits = lam;
  c->lam_acc = 0ull;
  c->blocks_done = 0u;
  if (next_dt > 0.0) {
    const double l = __longlong_as_double((long long)lam);
    if (!(l == l) || isinf(l)) k.status |= GS_ST_NONFINITE;
    plan_host_dt(c, p, k, f, next_dt);
  } else {
    plan_dt(c, p, k, f, lam);
  }
}

// Neighbour-lane values for the y-faces: lane l receives lane l+1's value (lane_upper)
// or lane l-1's (lane_lower); the end lanes keep their own. The shuffle runs on the LDS
// crossbar, beside the VALU work of the faces: DPP wavefront shifts (one VALU move per 32
// bits plus hazard waits) made the VALU-bound sweeps 1-6 % slower on MI355X.
template <typename T> __device__ __forceinline__ T lane_upper(T x) { return __shfl_down(x, 1, 64); }
template <typename T> __device__ __forceinline__ T lane_lower(T x) { return __shfl_up(x, 1, 64); }

// The maximum of a wavefront's keys, in every lane (64 bits) or as a uniform value (32 bits: six
// DPP steps, which leave the maximum in the last lane).
__device__ __forceinline__ uint64_t wave_max(uint64_t v) {
  for (int off = 32; off > 0; off >>= 1) {
    const uint64_t o = __shfl_xor(v, off, 64);
    v = o > v ? o : v;
  }
  return v;
}
template <int CTRL, int ROWS>
__device__ __forceinline__ uint32_t dpp_max(uint32_t v) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROWS, 0xf, false);
  return o > v ? o : v;
}
__device__ __forceinline__ uint32_t wave_max(uint32_t v) {
  v = dpp_max<0x111, 0xf>(v);   // row_shr 1, 2, 4, 8: lane 15 of each row has the row's maximum
  v = dpp_max<0x112, 0xf>(v);
  v = dpp_max<0x114, 0xf>(v);
  v = dpp_max<0x118, 0xf>(v);
  v = dpp_max<0x142, 0xa>(v);   // row_bcast 15 into rows 1 and 3
  v = dpp_max<0x143, 0xc>(v);   // row_bcast 31 into rows 2 and 3
  return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}

// Use an atomic's returned value: the wave waits until the atomic has been performed, and
// the compiler moves no memory access across this point.
__device__ __forceinline__ void await_atomic(uint64_t v) { __asm__ volatile("" ::"v"(v) : "memory"); }

// Block reduction of a per-thread wave-speed (IEEE bits, order independent) and the
// last-workgroup-done hand-off of the grid maximum to plan_finish. Only atomics cross
// workgroups here (the state a workgroup stores is read by the next launch), so the
// hand-off orders atomics and nothing else: thread 0 folds the workgroup's maximum into
// the clock and waits until that atomic has been performed before it counts the
// workgroup done, so the count that reveals the last workgroup follows every maximum, and
// the last workgroup reads the total with a device-scope atomic load. A release on the
// count would also write back the XCD's L2 (its dirty state lines) once per workgroup,
// which cost 10 % of the coastal step at one workgroup per four tiles.
//
// The barrier orders LDS alone (the state's stores are not waited for, the kernel's end does that),
// and the first wavefront goes on alone. Only the last workgroup reads the rest of the clock: a load
// of the line that the atomics are queueing for waits in their queue (with one in every workgroup a
// 2048^2 coastal step took 69 us instead of 40).
template <typename K>
__device__ __forceinline__ void grid_reduce_and_plan(K key, GsClock* c, const Plan& p, bool advance,
                                                     double next_dt = 0.0) {
  __shared__ K s_w[16];
  const K top = wave_max(key);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) s_w[wave] = top;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  if (threadIdx.x != 0) return;
  K m = 0;
  const int nw = (blockDim.x + 63) >> 6;
  for (int w = 0; w < nw; ++w) m = s_w[w] > m ? s_w[w] : m;
  if (m)
    await_atomic(__hip_atomic_fetch_max(&c->lam_acc, lam_key_bits64(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  const unsigned int prev = __hip_atomic_fetch_add(&c->blocks_done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (prev == gridDim.x - 1) plan_finish(c, p, clock_read(c), advance, next_dt);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
template <typename T>
static inline Phys<T> make_phys(const GsPhys& p, double dx, double dy) {
  Phys<T> P;
  P.g = (T)p.g;
  P.h_min = (T)p.h_min;
  P.h_cfl = (T)p.h_cfl;
  P.vcap = (T)p.vcap;
  P.has_vcap = isfinite(p.vcap) && p.vcap > 0.0;
  P.inv_dx = (T)(1.0 / dx);
  P.inv_dy = (T)(1.0 / dy);
  // the reference kernel recomputes dx = 1/inv_dx in T (rhs_cuda.py:928-929)
  P.half_dx = T(0.5) * (T(1) / P.inv_dx);
  P.half_dy = T(0.5) * (T(1) / P.inv_dy);
  P.friction = p.friction;
  P.quadratic = p.quadratic;
  P.keep_h = p.keep_h;
  P.cfl_l2 = p.cfl_l2;
  return P;
}

// gs_flat_step (pre: NULL, or the three planes of gs_flat_step_pre) whose plan takes `next_dt` for the
// step after it if that is positive. smp: NULL, or depths of the step's input state to sample.
struct FlatSample {
  const int64_t* ids;
  int n;
  void* out;
};
int flat_step_next(const GsFlat* f, const GsPhys* phys, const GsForcing& forc, GsClock* clock_dev, void* const* pre,
                   double next_dt, const FlatSample* smp, void* stream);

static inline int check_phys(const GsPhys* p) {
  if (!p) return fail(GS_E_ARG, "phys is NULL");
  if (!(p->g > 0.0) || !(p->h_min > 0.0) || !(p->cfl > 0.0) || !(p->dmin > 0.0))
    return fail(GS_E_ARG, "phys: g, h_min, cfl and dmin must be positive");
  if (p->friction && (p->n_classes < 1 || p->n_classes > GS_MAX_CLASSES))
    return fail(GS_E_ARG, "phys: n_classes must be in [1, %d] with friction on (got %d)", GS_MAX_CLASSES,
                p->n_classes);
  return GS_OK;
}

static inline int check_forcing(const GsForcing& f) {
  if (f.n_rain < 0 || f.n_stage < 0) return fail(GS_E_ARG, "forcing: negative table size");
  if (f.n_rain > 0 && (!f.rain_t || !f.rain_rate || !f.rain_cap))
    return fail(GS_E_ARG, "forcing: rain tables are NULL");
  if (f.rain_gridded && (f.n_rain < 1 || !f.rain_frames))
    return fail(GS_E_ARG, "forcing: gridded rain needs frames");
  if (f.n_stage > 0 && (!f.stage_t || !f.stage_v)) return fail(GS_E_ARG, "forcing: stage tables are NULL");
  return GS_OK;
}


}  // namespace gs
