// gs_flat.hip -- compressed active-cell ("flat") layout of the fused finite-volume step.
//
// Stored cells are the active set dilated by two cells (4-neighbour cross), laid out in
// row-major padded (i, j) order like the reference's CompressedMesh2D
// (src/geoswe/compressed_mesh.py:139-157, compressed_rhs.py:241-369). Because of the
// ring-2 dilation, the +-1 and +-2 neighbours along j of an active cell are the flat ids
// k+-1, k+-2; the rows i+-1, i+-2 sit at offsets that are constant over a run of
// consecutive active cells, so the kernel reads a small run table instead of a per-cell
// neighbour table. Cells in no run are the frozen ring: never written, identical in both
// state buffers.
//
// A wavefront pass covers 64 consecutive flat ids and writes the middle 60 (the chunk
// stride of the run index). Each lane evaluates its two x-faces with gathered neighbours and its
// upper y-face with the lane above; the lower y-face comes from the lane below by a
// cross-lane shuffle. The face arithmetic is gs_device.h's, shared with the dense sweep,
// so the residual is bitwise the dense one.
#include <atomic>
#include <mutex>
#include <vector>

#include "gs_common.h"
#include "gs_wave.h"

namespace gs {

constexpr int kFOut = 60;     // flat ids written per wavefront (lanes 2..61)
constexpr int kFBlock = 256;
// Wavefronts (tiles in flight) per workgroup of a sweep. Each workgroup ends with two atomics on
// the clock's cache line, which serialize at about 6 ns each: eight wavefronts halve them (2048^2
// coastal domain, 6-row tiles: 43.1 against 44.5 us per step; 2-row tiles: 57.7 against 81 us). Float64
// sweeps fit three wavefronts per SIMD, which workgroups of eight would leave at two.
template <typename T>
constexpr int kSweepWaves = sizeof(T) == 4 ? 8 : 4;
template <typename T>
constexpr int kSBlock = 64 * kSweepWaves<T>;

// One domain, as its kernels read it; also a member's view in the ensemble's table, of which
// gs_ens_run_noalloc keeps a promised number in a fixed scratch: what belongs to one launch alone is
// in FlatLaunch.
template <typename T>
struct FlatK {
  int64_t n;
  int n_runs, nyp, ngh;
  int wave;         // kWave* flags of P; 0 too where a tile's rows may span 2 GiB
  int64_t nchunks;
  T* buf[2][3];
  const T* bed;
  const uint8_t* flags;
  const T* ntab;
  int n_classes;
  const T* n_field;
  T* max_h;
  const uint8_t* cls;   // per-cell class plane (ids 0..255), or NULL: the flags' class bits
  T* rhs[3];
  int which;
  const int64_t* run_k0;
  const int32_t* run_len;
  const int32_t* run_i;
  const int32_t* run_j0;
  const int32_t* run_d;
  const int32_t* chunk_run;
  Phys<T> P;
  int rain_mode;
  const T* rain_frames;
  int64_t frame_stride, rain_pitch;
  GsClock* clock;
  Plan plan;
  T* pre[3];        // nullable: pre-friction h, hu, hv of active cells (adjoint recomputation)
  int64_t n_tiles;  // row-sweep tiles (0: chunk traversal)
  const int64_t* tile_e0;
  const int32_t* tile_irc;
  const uint64_t* ent;
  const T* sponge;  // nullable [N][2] (keep, amb) of GS_FLAG_FORCE cells
  const T* clamp;   // nullable [N] h_max of GS_FLAG_FORCE cells
  const T* infil;   // nullable [32] infiltration rate per Manning class
  const T* drain;   // nullable [N] karst target depth of GS_FLAG_FORCE cells
  const uint8_t* ga_cls;  // Green-Ampt / drain-tau (nullable tables, see the ABI header)
  const T* ga_ks;
  const T* ga_psi;
  const T* ga_dth;
  T* ga_F;
  const T* ga_fmax;
  const T* ga_inv_tau;
  const int32_t* rain_lookup;  // rain_mode 3: native-table column of each cell
  int64_t n_rmode;             // ring modes of the cached replay (top of the step)
  const int64_t* rmode_ids;
  const int64_t* rmode_nb;
  const uint8_t* rmode_kind;
  T rmode_eta;
  int64_t n_fring;  // forced cells of the ring (stored, not active): sponge, clamp, gauge ring
  const int64_t* fring;
  const int32_t* fring_row;  // nullable: gauge-ring row of each entry, -1 for none
  int ring_ng, ring_nt;
  const T* ring_bed;
  const T* ring_w;
  const double* ring_t;
  const T* ring_stage;
};

// What one launch of a step adds.
template <typename T>
struct FlatLaunch {
  double next_dt = 0.0;               // > 0: the dt that the step's plan takes for the step after it
  const int64_t* smp_ids = nullptr;   // lean sweep: depths of the step's input state at smp_n ids into smp_out
  T* smp_out = nullptr;
  int smp_n = 0;
  unsigned ring_blocks = 0;           // first workgroups of a sweep that take the ring cells (a multiple of 8, 0: none)
};


// What a wavefront reads whole by scalar loads: the mesh tables (tiles and their rows) and the
// descriptor itself. No kernel that reads them writes them.
#define GS_C __attribute__((address_space(4)))
template <typename P>
__device__ __forceinline__ const GS_C P* cp(const GS_G P* p) {
  return (const GS_C P*)(uint64_t)p;
}

// Read a value that the launch never writes through the constant address space: a
// uniform address then gives scalar loads. The host pass sees an ordinary read.
template <typename U>
__device__ __forceinline__ U const_read(const U* p) {
#if defined(__HIP_DEVICE_COMPILE__)
  return *(const __attribute__((address_space(4))) U*)p;
#else
  return *p;
#endif
}

// Everything one chunk pass reads, as values: the state buffers picked for this step (a
// runtime index into the argument's buffer table would put the table in private memory and
// every state access behind a generic pointer), the mesh arrays, the clock's per-step
// values and the physics scalars. Filled from the kernel argument (plain step) or from
// the member table (ensemble).
template <typename T>
struct FlatCtx {
  const GS_G T* qi0;
  const GS_G T* qi1;
  const GS_G T* qi2;
  GS_G T* qo0;
  GS_G T* qo1;
  GS_G T* qo2;
  const GS_G T* bed;
  const GS_G uint8_t* flags;
  const GS_G T* n_field;
  GS_G T* max_h;
  const GS_G uint8_t* cls;
  GS_G T* rhs0;
  GS_G T* rhs1;
  GS_G T* rhs2;
  GS_G T* pre0;
  GS_G T* pre1;
  GS_G T* pre2;
  const GS_G int64_t* run_k0;
  const GS_G int32_t* run_len;
  const GS_G int32_t* run_i;
  const GS_G int32_t* run_j0;
  const GS_G int32_t* run_d;
  const GS_G int32_t* chunk_run;
  const GS_G int64_t* tile_e0;
  const GS_G int32_t* tile_irc;
  const GS_G uint64_t* ent;
  const GS_G T* sponge;
  const GS_G T* clamp;
  const GS_G T* infil;
  const GS_G T* drain;
  const GS_G uint8_t* ga_cls;
  const GS_G T* ga_ks;
  const GS_G T* ga_psi;
  const GS_G T* ga_dth;
  GS_G T* ga_F;
  const GS_G T* ga_fmax;
  const GS_G T* ga_inv_tau;
  const GS_G int32_t* rain_lookup;
  const GS_G T* frame;   // gridded rain frame of this step (rain_mode 2)
  const T* ntab;         // Manning n per class (LDS copy or the member's table)
  const GS_C FlatK<T>* k;   // the descriptor itself, for cold()
  int64_t n, rain_pitch;
  int n_runs, ngh, rain_mode, wave;
  T dt, rain_u, eta;
  Phys<T> P;
};

// Device buffers are global memory; the explicit address space lets the compiler use global
// (not generic) accesses for pointers that come from device memory (the member table).
template <typename P>
__device__ __forceinline__ GS_G P* gp(P* p) {
  return (GS_G P*)p;
}

// The clock's per-step values for one domain (read once per launch, or once per member
// switch in the ensemble).
template <typename T>
struct FlatClk {
  bool live;        // false when the clock says the run is done
  int par;          // input buffer (MODE 1: nsteps & 1; MODE 0: the residual selector)
  T dt, rain_u, eta;
  const GS_G T* frame;
};

template <typename T, int MODE>
__device__ __forceinline__ FlatClk<T> flat_clock(const FlatK<T>& a) {
  FlatClk<T> k;
  k.live = true;
  k.par = MODE == 1 ? 0 : a.which;
  k.dt = T(0);
  k.rain_u = T(0);
  k.eta = T(0);
  k.frame = nullptr;
  if (MODE == 1) {
    // one line, read whole before the first branch on it; uniform values, in scalar registers
    const GS_G GsClock* c = gp(a.clock);
    const int st = c->status, ridx = __builtin_amdgcn_readfirstlane(c->rain_idx);
    const int64_t ns = c->nsteps;
    const T dt = sizeof(T) == 4 ? (T)c->dt32 : (T)c->dt, eta = sizeof(T) == 4 ? (T)c->eta32 : (T)c->eta64;
    const T rain = sizeof(T) == 4 ? (T)c->rain32 : T(0);
    k.par = __builtin_amdgcn_readfirstlane((int)(ns & 1));
    if (st & GS_ST_DONE) {
      k.live = false;
      return k;
    }
    k.dt = sreg(dt);
    k.rain_u = sizeof(T) == 4 ? sreg(rain) : a.rain_mode == 1 ? sreg((T)gp(a.plan.rain_rate)[ridx]) : T(0);
    k.eta = sreg(eta);
    if (a.rain_mode >= 2) k.frame = gp(a.rain_frames) + (int64_t)ridx * a.frame_stride;
  }
  return k;
}

// The step context: the layout of `a` with the buffers the clock values pick.
template <typename T, int MODE>
__device__ __forceinline__ void flat_ctx(const FlatK<T>& a, const FlatClk<T>& k, FlatCtx<T>& x) {
  const bool in1 = k.par != 0;
  const bool out1 = MODE == 1 ? !in1 : true;   // MODE 0 writes no state
  x.qi0 = gp(in1 ? a.buf[1][0] : a.buf[0][0]);
  x.qi1 = gp(in1 ? a.buf[1][1] : a.buf[0][1]);
  x.qi2 = gp(in1 ? a.buf[1][2] : a.buf[0][2]);
  x.qo0 = gp(out1 ? a.buf[1][0] : a.buf[0][0]);
  x.qo1 = gp(out1 ? a.buf[1][1] : a.buf[0][1]);
  x.qo2 = gp(out1 ? a.buf[1][2] : a.buf[0][2]);
  x.bed = gp(a.bed);
  x.flags = gp(a.flags);
  x.n_field = gp(a.n_field);
  x.cls = gp(a.cls);
  x.max_h = gp(a.max_h);
  x.rhs0 = gp(a.rhs[0]);
  x.rhs1 = gp(a.rhs[1]);
  x.rhs2 = gp(a.rhs[2]);
  x.pre0 = gp(a.pre[0]);
  x.pre1 = gp(a.pre[1]);
  x.pre2 = gp(a.pre[2]);
  x.run_k0 = gp(a.run_k0);
  x.run_len = gp(a.run_len);
  x.run_i = gp(a.run_i);
  x.run_j0 = gp(a.run_j0);
  x.run_d = gp(a.run_d);
  x.chunk_run = gp(a.chunk_run);
  x.tile_e0 = gp(a.tile_e0);
  x.tile_irc = gp(a.tile_irc);
  x.ent = gp(a.ent);
  x.sponge = gp(a.sponge);
  x.clamp = gp(a.clamp);
  x.infil = gp(a.infil);
  x.drain = gp(a.drain);
  x.ga_cls = gp(a.ga_cls);
  x.ga_ks = gp(a.ga_ks);
  x.ga_psi = gp(a.ga_psi);
  x.ga_dth = gp(a.ga_dth);
  x.ga_F = gp(a.ga_F);
  x.ga_fmax = gp(a.ga_fmax);
  x.ga_inv_tau = gp(a.ga_inv_tau);
  x.rain_lookup = gp(a.rain_lookup);
  x.frame = k.frame;
  x.ntab = a.ntab;
  x.n = a.n;
  x.rain_pitch = a.rain_pitch;
  x.n_runs = a.n_runs;
  x.ngh = a.ngh;
  x.rain_mode = a.rain_mode;
  x.wave = a.wave;
  x.dt = k.dt;
  x.rain_u = k.rain_u;
  x.eta = k.eta;
  x.P = a.P;
}

// The context with the pointers and physics scalars that a row needs seldom or late read from the
// descriptor again (scalar loads that hit the scalar cache; a caller pays for what it uses). Held
// through the row loop they were spilled to vector lanes, 450 lane reads for each two rows of the
// extended sweep.
template <typename T>
__device__ __forceinline__ const GS_C FlatK<T>* cold_ptr(const GS_C FlatK<T>* k) {
#if defined(__HIP_DEVICE_COMPILE__)
  asm volatile("" : "+s"(k));
#endif
  return k;
}
template <typename T>
__device__ __forceinline__ FlatCtx<T> cold(const FlatCtx<T>& x) {
  const GS_C FlatK<T>* k = cold_ptr<T>(x.k);
  FlatCtx<T> y = x;
  y.n_field = gp((T*)k->n_field);
  y.cls = gp((uint8_t*)k->cls);
  y.max_h = gp((T*)k->max_h);
  y.pre0 = gp((T*)k->pre[0]);
  y.pre1 = gp((T*)k->pre[1]);
  y.pre2 = gp((T*)k->pre[2]);
  y.sponge = gp((T*)k->sponge);
  y.clamp = gp((T*)k->clamp);
  y.infil = gp((T*)k->infil);
  y.drain = gp((T*)k->drain);
  y.ga_cls = gp((uint8_t*)k->ga_cls);
  y.ga_ks = gp((T*)k->ga_ks);
  y.ga_psi = gp((T*)k->ga_psi);
  y.ga_dth = gp((T*)k->ga_dth);
  y.ga_F = gp((T*)k->ga_F);
  y.ga_fmax = gp((T*)k->ga_fmax);
  y.ga_inv_tau = gp((T*)k->ga_inv_tau);
  y.rain_lookup = gp((int32_t*)k->rain_lookup);
  y.wave = k->wave;
  y.P = const_read((const Phys<T>*)(uint64_t)&k->P);
  return y;
}
template <typename T>
__device__ __forceinline__ const GS_C FlatK<T>* kernel_arg() {   // a kernel whose first argument is a FlatK<T>
#if defined(__HIP_DEVICE_COMPILE__)
  return (const GS_C FlatK<T>*)__builtin_amdgcn_kernarg_segment_ptr();
#else
  return nullptr;
#endif
}

// The next_dt of a kernel whose arguments are a FlatK<T> and a FlatLaunch<T>, read where it is used
// (held through the row loop it cost the lean sweep spilled lanes: 290 lane reads instead of 219).
template <typename T>
__device__ __forceinline__ double next_dt_arg() {
#if defined(__HIP_DEVICE_COMPILE__)
  static_assert(sizeof(FlatK<T>) % alignof(FlatLaunch<T>) == 0, "the second argument follows the first");
  return ((const GS_C FlatLaunch<T>*)(cold_ptr<T>(kernel_arg<T>()) + 1))->next_dt;
#else
  return 0.0;
#endif
}

// One wavefront pass over flat ids chunk*60-2 .. chunk*60+61: the residual (MODE 0) or the
// fused update (MODE 1) of the 60 middle ids, folding their CFL speed bits into lam.
// Every lane of the wavefront must call it (cross-lane shuffles).
// Element at byte offset `off` of an array segment that starts at `row` (uniform).
template <typename P>
__device__ __forceinline__ const GS_G P& gat(const GS_G P* row, uint32_t off) {
  return *(const GS_G P*)((const GS_G char*)row + off);
}
template <typename P>
__device__ __forceinline__ GS_G P& gat(GS_G P* row, uint32_t off) {
  return *(GS_G P*)((GS_G char*)row + off);
}

// Sponge band then stage clamp on a GS_FLAG_FORCE cell, after the update, the stage and the
// running max (sponge_band, compressed_solver.py:1320-1326: h*keep then + amb, two roundings;
// stage_clamp_flat, 424-440). keep = 1, amb = 0, h_max = +inf leave a cell unchanged.
template <typename T>
__device__ __forceinline__ void sponge_cell(T kp, T am, T& h, T& hu, T& hv) {
  h = h * kp + am;
  hu = hu * kp;
  hv = hv * kp;
}
template <typename T>
__device__ __forceinline__ void clamp_cell(T hx, T& h, T& hu, T& hv) {
  if (h > hx) {
    const T ratio = hx / h;
    h = hx;
    hu = hu * ratio;
    hv = hv * ratio;
  }
}
template <typename T>
__device__ __forceinline__ void drain_cell(T ht, T& h, T& hu, T& hv) {
  if (h > ht) {
    const T r = h > T(1e-12) ? ht / h : T(0);
    h = ht;
    hu = hu * r;
    hv = hv * r;
  }
}
// Constant-rate infiltration of one active cell (infiltrate_flat): nothing below h_min.
template <typename T>
__device__ __forceinline__ void infil_cell(T rate, T dt, T hmin, T& h, T& hu, T& hv) {
  if (!(h < hmin)) {
    const T dh = rate * dt;
    T hn = h - dh;
    hn = hn < T(0) ? T(0) : hn;
    const T r = hn / h;
    h = hn;
    hu = hu * r;
    hv = hv * r;
  }
}
// exp(x) in float64 from IEEE +, -, *, rint and ldexp only, so that it is the oracle's
// exp_ieee bit for bit: Cody-Waite reduction x = k ln2 + r (ln2 split in a 32-bit head, so
// k*LN2_HI is exact, and a tail), exp(r) on |r| <= ln2/2 by the degree-13 Taylor polynomial in
// Horner form, scaled by 2^k. It replaces the fast exponential of the reference's drain decay
// (float64 state; float32 state uses exp_ieee_f below).
__device__ __forceinline__ double exp_ieee(double x) {
  if (!(x == x)) return x;
  if (x > 709.8) return __builtin_inf();
  if (x < -745.2) return 0.0;
  const double kf = rint(x * 1.44269504088896338700e+00);
  const double r = (x - kf * 6.93147180369123816490e-01) - kf * 1.90821492927058770002e-10;
  double p = 1.6059043836821613e-10;
  p = p * r + 2.08767569878681e-09;
  p = p * r + 2.505210838544172e-08;
  p = p * r + 2.755731922398589e-07;
  p = p * r + 2.7557319223985893e-06;
  p = p * r + 2.48015873015873e-05;
  p = p * r + 0.0001984126984126984;
  p = p * r + 0.001388888888888889;
  p = p * r + 0.008333333333333333;
  p = p * r + 0.041666666666666664;
  p = p * r + 0.16666666666666666;
  p = p * r + 0.5;
  p = p * r + 1.0;
  p = p * r + 1.0;
  return ldexp(p, (int)kf);
}

// The float32 form: ln2 split in a 15-bit head (k*LN2_HI exact for |k| < 512) and a tail, a
// degree-7 Taylor polynomial (truncation below 5e-9 relative), every operation in float32.
__device__ __forceinline__ float exp_ieee_f(float x) {
  if (!(x == x)) return x;
  if (x > 88.73f) return __builtin_inff();
  if (x < -103.98f) return 0.0f;
  const float kf = rintf(x * 1.4426950216293335f);
  const float r = (x - kf * 0.693145751953125f) - kf * 1.428606765330187e-06f;
  float p = 0.00019841270113829523f;
  p = p * r + 0.0013888889225199819f;
  p = p * r + 0.008333333767950535f;
  p = p * r + 0.0416666679084301f;
  p = p * r + 0.1666666716337204f;
  p = p * r + 0.5f;
  p = p * r + 1.0f;
  p = p * r + 1.0f;
  return ldexpf(p, (int)kf);
}

// What the forcings of every active cell read: its infiltration rate, and with GA its Green-Ampt and
// drain-tau values (0 where there are none). Loaded ahead of the update, all at once: at their use,
// behind the branches on the rate, K and h, seven loads waited for one another, and the whole forcing
// tail on 121 M cells took 2.44 ms per step against 2.01 (10 steps on 1500^2: 484 us against 451).
template <typename T>
struct ForceIn {
  T rate, K, psi, dth, F0, fmax, inv_tau;
};
template <typename T, bool GA>
__device__ __forceinline__ ForceIn<T> force_load(const FlatCtx<T>& x, uint8_t fg, int64_t base, uint32_t off,
                                                 uint32_t ob) {
  ForceIn<T> v = {T(0), T(0), T(0), T(0), T(0), T(0), T(0)};
  if (GA && x.ga_ks) {
    const int c = gat(x.ga_cls + base, ob);
    v.F0 = gat(x.ga_F + base, off);
    if (x.ga_fmax) v.fmax = gat(x.ga_fmax + base, off);
    if (x.ga_inv_tau) v.inv_tau = gat(x.ga_inv_tau + base, off);
    v.K = x.ga_ks[c];
    v.psi = x.ga_psi[c];
    v.dth = x.ga_dth[c];
  } else if (GA && x.ga_inv_tau) {
    v.inv_tau = gat(x.ga_inv_tau + base, off);
  }
  if (x.infil) v.rate = x.infil[x.cls ? gat(x.cls + base, ob) : (fg & GS_FLAG_CLASS_MASK)];
  return v;
}

// Green-Ampt infiltration then drain-tau of one active cell (ga_drain_flat).
template <typename T>
__device__ __forceinline__ void ga_cell(const FlatCtx<T>& x, const ForceIn<T>& v, int64_t base, uint32_t off, T& h,
                                        T& hu, T& hv) {
  if (h <= T(0)) return;
  T scale = T(1);
  if (v.K > T(0)) {
    const T KsDt = v.K * x.dt;
    const T head = v.psi + h;
    const T a = v.F0 + KsDt;
    const T disc = a * a + ((T(4) * KsDt) * head) * v.dth;
    const T F1 = T(0.5) * (a + sqrt(disc > T(0) ? disc : T(0)));   // fmax(disc, 0): NaN gives 0
    T dF = F1 - v.F0;
    dF = dF > T(0) ? dF : T(0);
    if (dF > h) dF = h;
    if (x.ga_fmax) {
      const T room = v.fmax - v.F0;
      if (dF > room) dF = room > T(0) ? room : T(0);
    }
    const T hn = h - dF;
    scale = scale * (hn / h);
    h = hn;
    gat(x.ga_F + base, off) = v.F0 + dF;
  }
  if (v.inv_tau > T(0) && h > T(0)) {
    const T arg = (-x.dt) * v.inv_tau;
    T decay;
    if constexpr (sizeof(T) == 4) decay = exp_ieee_f(arg);
    else decay = exp_ieee(arg);
    scale = scale * decay;
    h = h * decay;
  }
  hu = hu * scale;
  hv = hv * scale;
}

// The forcings after the running max, in the reference's order: infiltration (every active
// cell, by Manning class), the sponge of a GS_FLAG_FORCE cell, (the gauge ring: ring cells
// only, in the ring pass), Green-Ampt and drain-tau (every active cell), then the clamp and
// the karst drain of a GS_FLAG_FORCE cell. GA = false leaves Green-Ampt out of the code (the
// plain sweep's instantiation, which has no register to spare for it).
template <typename T, bool GA>
__device__ __forceinline__ void active_force(const FlatCtx<T>& x, const ForceIn<T>& v, uint8_t fg, int64_t base,
                                             uint32_t off, T& h, T& hu, T& hv) {
  if (x.infil) infil_cell<T>(v.rate, x.dt, x.P.h_min, h, hu, hv);
  const bool fc = (fg & GS_FLAG_FORCE) != 0;
  if (fc && x.sponge)
    sponge_cell<T>(gat(x.sponge + 2 * base, 2 * off), gat(x.sponge + 2 * base + 1, 2 * off), h, hu, hv);
  if (GA && (x.ga_ks || x.ga_inv_tau)) ga_cell<T>(x, v, base, off, h, hu, hv);
  if (fc && x.clamp) clamp_cell<T>(gat(x.clamp + base, off), h, hu, hv);
  if (fc && x.drain) drain_cell<T>(gat(x.drain + base, off), h, hu, hv);
}

template <typename T, int MODE>
__device__ __forceinline__ void flat_chunk(const FlatCtx<T>& x, int64_t chunk, int lane, lam_t<T>& lam) {
  const FlatCtx<T>& a = x;
  const Phys<T>& P = a.P;
  const T ix = P.inv_dx, iy = P.inv_dy, hdx = P.half_dx, hdy = P.half_dy, g = P.g, hm = P.h_min;
  const int64_t k = chunk * kFOut + lane - 2;
  const int64_t kl = k < 0 ? 0 : (k >= a.n ? a.n - 1 : k);
  // this lane's cell (needed by every lane for the y-face shuffles)
  const T hC = x.qi0[kl], huC = x.qi1[kl], hvC = x.qi2[kl];
  const T bC = a.bed[kl];
  T uC, vC;
  prims(hC, huC, hvC, hm, uC, vC);
  const T bl = lane_lower(bC), br = lane_upper(bC);
  const T gzy = (T(0.5) * (br - bl)) * iy;
  // upper y-face (k, k+1)
  const T hR = lane_upper(hC), uR = lane_upper(uC), vR = lane_upper(vC);
  const T gzyR = lane_upper(gzy);
  Face<T> fy;
  face<T>(bC, br, gzy, gzyR, hC, hR, vC, uC, vR, uR, hdy, g, hm, fy);
  const T yFhB = lane_lower(fy.Fh), yFNB = lane_lower(fy.FN), yFTB = lane_lower(fy.FT);
  const T ysRB = lane_lower(fy.srcR);
  const int ygB = lane_lower((int)fy.gate);

  // run of this cell
  int r = -1;
  if (lane >= 2 && lane < 2 + kFOut && k < a.n) {
    int rr = a.chunk_run[chunk];
    while (rr < a.n_runs && a.run_k0[rr] + a.run_len[rr] <= k) ++rr;
    if (rr < a.n_runs && a.run_k0[rr] <= k) r = rr;
  }
  if (r < 0) return;
  const GS_G int32_t* d = a.run_d + 4 * (int64_t)r;
  const int64_t kE = k + d[0], kW = k + d[1], kEE = k + d[2], kWW = k + d[3];
  const T bE = a.bed[kE], bW = a.bed[kW], bEE = a.bed[kEE], bWW = a.bed[kWW];
  const T hE = x.qi0[kE], huE = x.qi1[kE], hvE = x.qi2[kE];
  const T hW = x.qi0[kW], huW = x.qi1[kW], hvW = x.qi2[kW];
  T uE, vE, uW, vW;
  prims(hE, huE, hvE, hm, uE, vE);
  prims(hW, huW, hvW, hm, uW, vW);
  const T gzxC = (T(0.5) * (bE - bW)) * ix;
  const T gzxE = (T(0.5) * (bEE - bC)) * ix;
  const T gzxW = (T(0.5) * (bC - bWW)) * ix;
  Face<T> fr, fl;
  face<T>(bC, bE, gzxC, gzxE, hC, hE, uC, vC, uE, vE, hdx, g, hm, fr);
  face<T>(bW, bC, gzxW, gzxC, hW, hC, uW, vW, uC, vC, hdx, g, hm, fl);
  T rh = T(0), rhu = T(0), rhv = T(0);
  if (fr.gate) {
    rh = rh - fr.Fh * ix;
    rhu = rhu - fr.FN * ix;
    rhv = rhv - fr.FT * ix;
    rhu = rhu - fr.srcL * ix;
  }
  if (fl.gate) {
    rh = rh + fl.Fh * ix;
    rhu = rhu + fl.FN * ix;
    rhv = rhv + fl.FT * ix;
    rhu = rhu + fl.srcR * ix;
  }
  if (fy.gate) {
    rh = rh - fy.Fh * iy;
    rhu = rhu - fy.FT * iy;
    rhv = rhv - fy.FN * iy;
    rhv = rhv - fy.srcL * iy;
  }
  if (ygB) {
    rh = rh + yFhB * iy;
    rhu = rhu + yFTB * iy;
    rhv = rhv + yFNB * iy;
    rhv = rhv + ysRB * iy;
  }
  if (MODE == 0) {
    a.rhs0[k] = rh;
    a.rhs1[k] = rhu;
    a.rhs2[k] = rhv;
    return;
  }
  const uint8_t fg = a.flags ? a.flags[k] : (uint8_t)0;
  T rr0 = rh;
  if (a.rain_mode == 1) {
    rr0 = rr0 + x.rain_u;
  } else if (a.rain_mode == 2) {
    const int64_t ii = (int64_t)a.run_i[r] - a.ngh;
    const int64_t jj = (int64_t)a.run_j0[r] + (k - a.run_k0[r]) - a.ngh;
    rr0 = rr0 + x.frame[ii * a.rain_pitch + jj];
  } else if (a.rain_mode == 3) {
    rr0 = rr0 + x.frame[x.rain_lookup[k]];
  }
  if (a.pre0) {   // the first three statements of update(), kept for its reverse
    a.pre0[k] = hC + x.dt * rr0;
    a.pre1[k] = huC + x.dt * rhu;
    a.pre2[k] = hvC + x.dt * rhv;
  }
  T n = T(0);
  if (P.friction) n = a.n_field ? a.n_field[k] : x.ntab[a.cls ? a.cls[k] : (fg & GS_FLAG_CLASS_MASK)];
  T h, hu, hv;
  update<T>(hC, huC, hvC, rr0, rhu, rhv, x.dt, n, P, h, hu, hv);
  if (fg & GS_FLAG_STAGE) {
    const T hs = x.eta - bC;
    h = hs > T(0) ? hs : T(0);
    hu = T(0);
    hv = T(0);
  }
  if (a.max_h && h > a.max_h[k]) a.max_h[k] = h;
  active_force<T, true>(x, force_load<T, true>(x, fg, k, 0u, 0u), fg, k, 0u, h, hu, hv);
  x.qo0[k] = h;
  x.qo1[k] = hu;
  x.qo2[k] = hv;
  if (!(fg & GS_FLAG_CFL_SKIP)) {
    const lam_t<T> lb_ = lam_key<T, true>(h, hu, hv, P);
    lam = lb_ > lam ? lb_ : lam;
  }
}

// Lane `lane`'s cell in one window row of a sweep tile (entry e = first stored id, stored
// mask, active mask): the stored cells of a row are consecutive flat ids, so the lane's cell
// is the row's first id (uniform across the wavefront) plus the number of stored lanes below
// it. The byte offset of that count is returned; accesses add it to the row's start.
template <typename T>
__device__ __forceinline__ uint32_t sweep_lane(const GS_C uint64_t* e, int lane, int64_t& base, bool& st) {
  const uint64_t sm = e[1];
  base = (int64_t)e[0];
  const unsigned below =
      __builtin_amdgcn_mbcnt_hi((unsigned)(sm >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)sm, 0u));
  st = ((sm >> lane) & 1ull) != 0ull;
  return below * (uint32_t)sizeof(T);
}

// State and bed of a lane's cell; lanes on unstored cells read nothing and hold zeros
// (their faces are never used: every face an active cell needs has its stencil stored).
template <typename T>
__device__ __forceinline__ void sweep_q(const FlatCtx<T>& x, int64_t base, uint32_t off, bool st, T& h, T& hu,
                                        T& hv) {
  h = T(0);
  hu = T(0);
  hv = T(0);
  if (st) {
    h = gat(x.qi0 + base, off);
    hu = gat(x.qi1 + base, off);
    hv = gat(x.qi2 + base, off);
  }
}

template <typename T>
__device__ __forceinline__ T sweep_b(const FlatCtx<T>& x, int64_t base, uint32_t off, bool st) {
  T b = T(0);
  if (st) b = gat(x.bed + base, off);
  return b;
}

// The cell of an active lane after its update, in the reference's order: the stage, the running
// max and the forcings (what LEAN leaves out is not there).
template <typename T, bool EXT, bool LEAN>
__device__ __forceinline__ void finish_cell(const FlatCtx<T>& x, const ForceIn<T>& v, uint8_t fg, int64_t base,
                                            uint32_t off, T b, T& h, T& hu, T& hv) {
  if (fg & GS_FLAG_STAGE) {
    const T hs = x.eta - b;
    h = hs > T(0) ? hs : T(0);
    hu = T(0);
    hv = T(0);
  }
  if (!LEAN) {
    if (x.max_h && h > gat(x.max_h + base, off)) gat(x.max_h + base, off) = h;
    active_force<T, EXT>(x, v, fg, base, off, h, hu, hv);
  }
}

// The tallest tile that flat_rows takes: its rows are addressed with 32-bit offsets.
constexpr int kWaveRows = 1024;

// The rows of a sweep. The lean sweeps have an instantiation of each: in the lean row the general wave
// speed beside the quick one cost the L-inf steps 1 to 2 % (2048^2, 20 steps: 764 us against 755). The
// others decide by the descriptor, in a branch that a forcing takes anyway.
enum {
  kRowsQuick,    // wavefront forms, with the L-inf wave speed that the update has made (kWaveLam)
  kRowsAny,      // wavefront forms, any wave speed (the L2 norm, a CFL floor above h_min)
  kRowsGeneral,  // the general functions alone
};
template <bool LEAN>
constexpr int kRowsOf = LEAN ? kRowsQuick : kRowsAny;

// One row of a sweep tile.
struct FlatRow {
  uint32_t row;        // its first stored id, from the tile's first one (uniform)
  uint64_t st, act;    // stored and active lanes
  uint32_t below;      // stored lanes below this one: with `row` the lane's id where it is stored
};
__device__ __forceinline__ FlatRow flat_row(const GS_C uint64_t* e, uint32_t g0) {
  FlatRow r;
  r.row = (uint32_t)e[0] - g0;
  r.st = e[1];
  r.act = e[2];
  r.below = __builtin_amdgcn_mbcnt_hi((unsigned)(r.st >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)r.st, 0u));
  return r;
}

// Rows 0 .. nr-1 of a tile by the wavefront forms (gs_wave.h): every face is evaluated once, the
// x-face below a row is carried from the row above, the y-face below a lane comes from the lane
// below by shuffle, and the residual terms are added in the dense sweep's order, so all traversals
// give the same bits. Returns the first row that it leaves to flat_rows_general (one that holds
// an operand outside their bounds, before anything of it is written), nr where there is none.
// A row's state, flags and rain are loaded one row ahead of their use, its bed two rows ahead and
// its entry before that. Lanes on unstored cells read 0: no face that an active cell uses reads
// them.
template <typename T, bool PRE, bool EXT, bool LEAN, int ROWS>
__device__ __forceinline__ int flat_rows(const FlatCtx<T>& x, const WaveC<T>& w, const GS_C uint64_t* E, int i0, int nr,
                                         int c0, int lane, lam_t<T>& lam) {
  constexpr uint32_t es = (uint32_t)sizeof(T);
  lmask odd = 0;
  lam_t<T> top = 0;   // the tile's own maximum: what the caller holds need not stay in a register
  const Lanes ln = lanes_of(lane);
  const int64_t g0 = (int64_t)E[0];   // ids of a tile's rows ascend
  const uint32_t g0l = (uint32_t)g0;
  const RowBuf qi0 = row_buf(x.qi0 + g0), qi1 = row_buf(x.qi1 + g0), qi2 = row_buf(x.qi2 + g0),
               bed = row_buf(x.bed + g0), qo0 = row_buf(x.qo0 + g0), qo1 = row_buf(x.qo1 + g0),
               qo2 = row_buf(x.qo2 + g0);
  // flags and gridded rain are read as 0 where there are none, without a branch
  const bool gridded = x.rain_mode == 2;
  const lmask flagged = x.flags ? lm_every() : lm_none(), rained = gridded ? lm_every() : lm_none();
  const RowBuf flg = row_buf(x.flags + g0);
  const RowBuf rnb = row_buf(x.frame + (int64_t)(i0 - x.ngh) * x.rain_pitch + (c0 - x.ngh) - 1);   // from lane -1
  const T rain = vreg(x.rain_mode == 1 ? x.rain_u : T(0));
  const uint32_t rain_row = (uint32_t)x.rain_pitch * es;
  auto load_q = [&](const FlatRow& r, T& h, T& hu, T& hv) __attribute__((always_inline)) {
    const uint32_t off = lm_lane(r.st) ? r.below * es : kNoLane;
    row_load(qi0, off, r.row * es, h);
    row_load(qi1, off, r.row * es, hu);
    row_load(qi2, off, r.row * es, hv);
  };
  auto load_b = [&](const FlatRow& r, T& b) __attribute__((always_inline)) {
    row_load(bed, lm_lane(r.st) ? r.below * es : kNoLane, r.row * es, b);
  };
  // a row's flags and rain, on its active lanes
  auto load_c = [&](const FlatRow& r, int k, uint8_t& fg, T& rn) __attribute__((always_inline)) {
    row_load(flg, lm_lane(r.act & flagged) ? r.below : kNoLane, r.row, fg);
    row_load(rnb, lm_lane(r.act & rained) ? (uint32_t)ln.up * (es / 4u) : kNoLane, (uint32_t)k * rain_row, rn);
  };

  T b0, bp1, hC, huC, hvC, uC, vC, zxC;
  T sh, shu, shv, sb, srn;   // loaded ahead: the next row's state and rain, the bed of the one after it
  uint8_t sfl;               // and the next row's flags
  lmask dryC;
  FaceProd<T> fx;            // the x-face below the current row
  FlatRow eC = flat_row(E + 6, g0l), eN = flat_row(E + 9, g0l), eF = flat_row(E + 12, g0l);
  {
    const FlatRow e0 = flat_row(E, g0l), e1 = flat_row(E + 3, g0l);
    T bm2, bm1, hP, huP, hvP, uP, vP;
    load_b(e0, bm2);
    load_b(e1, bm1);
    load_b(eC, b0);
    load_b(eN, bp1);
    load_q(e1, hP, huP, hvP);
    load_q(eC, hC, huC, hvC);
    load_q(eN, sh, shu, shv);
    load_b(eF, sb);
    load_c(eC, 0, sfl, srn);
    lmask dryP;
    prims_w<T>(hP, huP, hvP, vabs(bm2) + vabs(bm1), e1.st, w, uP, vP, dryP, odd);
    prims_w<T>(hC, huC, hvC, vabs(b0) + vabs(bp1), eC.st, w, uC, vC, dryC, odd);
    const T zxP = w.hdx * ((T(0.5) * (b0 - bm2)) * w.ix);
    zxC = w.hdx * ((T(0.5) * (bp1 - bm1)) * w.ix);
    face_w<T>(bm1, b0, zxP, zxC, hP, hC, uP, vP, uC, vC, dryP, dryC, eC.act, w.ix, w, fx, odd);
    take_loaded(sh, shu, shv, sb);   // nothing is in flight when the rows begin
  }

  // one row; false if it is left to the general functions
  auto row = [&](int r) __attribute__((always_inline)) -> bool {
    T hN = sh, huN = shu, hvN = shv, bp2 = sb;
    take_loaded(hN, huN, hvN, bp2);
    const FlatRow e2 = eF;   // row r + 2
    load_q(e2, sh, shu, shv);
    eF = flat_row(E + 3 * min(r + 5, nr + 3), g0l);   // row r + 3; the last rows read again what they have
    T uN, vN;
    lmask dryN;
    prims_w<T>(hN, huN, hvN, bp2, eN.st, w, uN, vN, dryN, odd);
    // y faces of the row: each lane computes its upper face (j, j+1)
    const T bl = lane_get(ln.dn, b0), br = lane_get(ln.up, b0);
    const T zy = w.hdy * ((T(0.5) * (br - bl)) * w.iy);
    const T hR = lane_get(ln.up, hC), uR = lane_get(ln.up, uC), vR = lane_get(ln.up, vC);
    const T zyR = lane_get(ln.up, zy);
    const T zxN = w.hdx * ((T(0.5) * (bp2 - b0)) * w.ix);
    const lmask act = eC.act;
    FaceProd<T> fn, fy;
    face_w<T>(b0, br, zy, zyR, hC, hR, vC, uC, vR, uR, dryC, lm_upper(dryC), act | lm_upper(act), w.iy, w, fy, odd);
    const T lFh = lane_get(ln.dn, fy.Fh), lFN = lane_get(ln.dn, fy.FN), lFT = lane_get(ln.dn, fy.FT),
            lsR = lane_get(ln.dn, fy.sR);
    load_b(eF, sb);
    face_w<T>(b0, bp1, zxC, zxN, hC, hN, uC, vC, uN, vN, dryC, dryN, act | eN.act, w.ix, w, fn, odd);
    T rh, rhu, rhv;
    sum_faces<T>(fn, fx, fy, lFh, lFN, lFT, lsR, rh, rhu, rhv);

    const uint8_t fg = sfl;
    T rr0 = rh + (rain + srn);   // one of them is 0, or both: rh is never -0, and + 0 changes nothing
    const lmask stage = act & lm_of((fg & GS_FLAG_STAGE) != 0), cfl = act & lm_of(!(fg & GS_FLAG_CFL_SKIP));
    const int64_t gC = g0 + eC.row;
    T n = T(0);
    if (LEAN) {
      if (x.P.friction) n = x.ntab[fg & GS_FLAG_CLASS_MASK];
    } else {
      const FlatCtx<T> y = cold(x);
      if (EXT && x.rain_mode == 3 && lm_lane(act)) rr0 = rh + x.frame[gat(y.rain_lookup + gC, eC.below * 4u)];
      if (EXT ? y.P.friction : x.P.friction) {
        if (y.n_field || y.cls) {
          if (lm_lane(act)) n = y.n_field ? gat(y.n_field + gC, eC.below * es) : x.ntab[gat(y.cls + gC, eC.below)];
        } else {
          n = x.ntab[fg & GS_FLAG_CLASS_MASK];
        }
      }
    }
    load_c(eN, r + 1, sfl, srn);
    ForceIn<T> fin;
    if (!LEAN) {
      const FlatCtx<T> y = cold(x);
      if (lm_lane(act)) fin = force_load<T, EXT>(y, fg, gC, eC.below * es, eC.below);
    }
    T h, hu, hv, speed;
    // the extended sweep has no scalar registers for the physics switches either (held, they cost 20 lane
    // reads more in float32 and 144 in float64: 2500^2 with the forcing tail 87 us per step against 86)
    if constexpr (EXT) update_w<T>(hC, huC, hvC, rr0, rhu, rhv, n, act, cold(x).P, w, h, hu, hv, speed, odd);
    else update_w<T>(hC, huC, hvC, rr0, rhu, rhv, n, act, x.P, w, h, hu, hv, speed, odd);
    const bool left = lm_any(odd);
    if (PRE) {   // the first three statements of update(), kept for its reverse
      const FlatCtx<T> y = cold(x);
      if (lm_lane(act) && !left) {
        gat(y.pre0 + gC, eC.below * es) = hC + w.dt * rr0;
        gat(y.pre1 + gC, eC.below * es) = huC + w.dt * rhu;
        gat(y.pre2 + gC, eC.below * es) = hvC + w.dt * rhv;
      }
    }
    lam_t<T> key;
    if (LEAN) {
      if (lm_any(stage)) {   // |eta| < 2^30 here, and beds are below 2^20
        h = lm_sel(stage, pos_w(x.eta - b0), h);
        hu = lm_sel(stage, T(0), hu);
        hv = lm_sel(stage, T(0), hv);
        if (ROWS == kRowsQuick) speed = speed_w<T>(h, hu, hv, w);
      }
      if constexpr (ROWS == kRowsQuick) key = lam_key_w<T>(speed);
      else key = lam_key<T, true>(h, hu, hv, cold(x).P);
    } else {
      const FlatCtx<T> y = cold(x);
      if (lm_lane(act) && !left) finish_cell<T, EXT, LEAN>(y, fin, fg, gC, eC.below * es, b0, h, hu, hv);
      speed = speed_w<T>(h, hu, hv, w);
      key = lam_key_w<T>(speed);
      if (!(y.wave & kWaveLam) || lm_any(act & lm_not(lm_lt(speed, kMaxSpeed<T>))))
        key = lam_key<T, true>(h, hu, hv, cold(x).P);
    }
    // in a row with an odd lane every lane's store is out of range, so that every way to the next
    // row's loads holds the same stores
    const uint32_t so = (lm_lane(act) ? eC.below * es : kNoLane) | (left ? kNoLane : 0u);
    row_store(qo0, so, eC.row * es, h);
    row_store(qo1, so, eC.row * es, hu);
    row_store(qo2, so, eC.row * es, hv);
    if (left) return false;
    if (lm_lane(cfl)) top = key > top ? key : top;

    // slide the window one row down
    hC = hN; huC = huN; hvC = hvN; uC = uN; vC = vN; zxC = zxN; dryC = dryN;
    b0 = bp1; bp1 = bp2;
    fx = fn;
    eC = eN; eN = e2;
    return true;
  };
  int r = 0;   // two rows per trip: half of the window's moves are names instead
  while (r < nr) {
    if (!row(r)) break;
    if (++r == nr) break;
    if (!row(r)) break;
    ++r;
  }
  lam = top > lam ? top : lam;
  return r;
}

// The same rows by the general functions of gs_device.h, for every operand. HOT: nothing ran before
// them, so the context is taken as it is.
template <typename T, bool PRE, bool EXT, bool LEAN, bool HOT>
__device__ __forceinline__ void flat_rows_general(const FlatCtx<T>& hot, const GS_C uint64_t* E, int i0, int nr, int c0,
                                                  int lane, lam_t<T>& lam) {
  const FlatCtx<T> x = HOT ? hot : cold(hot);
  const Phys<T>& P = x.P;
  const T ix = P.inv_dx, iy = P.inv_dy, hdx = P.half_dx, hdy = P.half_dy, g = P.g, hm = P.h_min;
  bool sm2, sm1, sC, sN;
  int64_t gm2, gm1, gC, gN;   // first flat id of rows i-2, i-1, i, i+1 (uniform)
  const uint32_t om2 = sweep_lane<T>(E, lane, gm2, sm2);
  const uint32_t om1 = sweep_lane<T>(E + 3, lane, gm1, sm1);
  uint32_t oC = sweep_lane<T>(E + 6, lane, gC, sC);
  uint32_t oN = sweep_lane<T>(E + 9, lane, gN, sN);
  const T bm2 = sweep_b(x, gm2, om2, sm2), bm1 = sweep_b(x, gm1, om1, sm1);
  T b0 = sweep_b(x, gC, oC, sC), bp1 = sweep_b(x, gN, oN, sN);
  T hP, huP, hvP, uP, vP;
  sweep_q(x, gm1, om1, sm1, hP, huP, hvP);
  prims(hP, huP, hvP, hm, uP, vP);
  const T gzxP = (T(0.5) * (b0 - bm2)) * ix;
  T hC, huC, hvC, uC, vC;
  sweep_q(x, gC, oC, sC, hC, huC, hvC);
  prims(hC, huC, hvC, hm, uC, vC);
  T gzxC = (T(0.5) * (bp1 - bm1)) * ix;
  FaceProd<T> fx;
  face_prod<T>(bm1, b0, gzxP, gzxC, hP, hC, uP, vP, uC, vC, hdx, ix, g, hm, fx);

  for (int r = 0; r < nr; ++r) {
    const GS_C uint64_t* Er = E + 3 * (r + 2);   // this row's entry
    bool sNN;
    int64_t gNN;
    const uint32_t oNN = sweep_lane<T>(Er + 6, lane, gNN, sNN);
    const T bp2 = sweep_b(x, gNN, oNN, sNN);
    T hN, huN, hvN, uN, vN;
    sweep_q(x, gN, oN, sN, hN, huN, hvN);
    prims(hN, huN, hvN, hm, uN, vN);
    const T gzxN = (T(0.5) * (bp2 - b0)) * ix;
    FaceProd<T> fn, fy;
    face_prod<T>(b0, bp1, gzxC, gzxN, hC, hN, uC, vC, uN, vN, hdx, ix, g, hm, fn);
    const T bl = lane_lower(b0), br = lane_upper(b0);
    const T gzy = (T(0.5) * (br - bl)) * iy;
    const T hR = lane_upper(hC), uR = lane_upper(uC), vR = lane_upper(vC);
    const T gzyR = lane_upper(gzy);
    face_prod<T>(b0, br, gzy, gzyR, hC, hR, vC, uC, vR, uR, hdy, iy, g, hm, fy);
    const T lFh = lane_lower(fy.Fh), lFN = lane_lower(fy.FN), lFT = lane_lower(fy.FT), lsR = lane_lower(fy.sR);
    T rh, rhu, rhv;
    sum_faces<T>(fn, fx, fy, lFh, lFN, lFT, lsR, rh, rhu, rhv);

    if ((Er[2] >> lane) & 1ull) {   // an active cell: lanes 2..61 only
      const uint32_t ob = oC / (uint32_t)sizeof(T);   // byte offset in a 1-byte plane
      const uint8_t fg = x.flags ? gat(x.flags + gC, ob) : (uint8_t)0;
      T rr0 = rh;
      if (x.rain_mode == 1) {
        rr0 = rr0 + x.rain_u;
      } else if (x.rain_mode == 2) {
        rr0 = rr0 + x.frame[(int64_t)(i0 + r - x.ngh) * x.rain_pitch + (c0 + lane - x.ngh)];
      } else if (EXT && x.rain_mode == 3) {
        rr0 = rr0 + x.frame[gat(x.rain_lookup + gC, (oC / (uint32_t)sizeof(T)) * 4u)];
      }
      if (PRE) {
        gat(x.pre0 + gC, oC) = hC + x.dt * rr0;
        gat(x.pre1 + gC, oC) = huC + x.dt * rhu;
        gat(x.pre2 + gC, oC) = hvC + x.dt * rhv;
      }
      T n = T(0);
      if (P.friction)
        n = (!LEAN && x.n_field) ? gat(x.n_field + gC, oC)
                                 : x.ntab[(!LEAN && x.cls) ? gat(x.cls + gC, ob) : (fg & GS_FLAG_CLASS_MASK)];
      T h, hu, hv;
      update<T>(hC, huC, hvC, rr0, rhu, rhv, x.dt, n, P, h, hu, hv);
      ForceIn<T> fin;
      if (!LEAN) fin = force_load<T, EXT>(x, fg, gC, oC, ob);
      finish_cell<T, EXT, LEAN>(x, fin, fg, gC, oC, b0, h, hu, hv);
      gat(x.qo0 + gC, oC) = h;
      gat(x.qo1 + gC, oC) = hu;
      gat(x.qo2 + gC, oC) = hv;
      if (!(fg & GS_FLAG_CFL_SKIP)) {
        const lam_t<T> lb_ = lam_key<T, true>(h, hu, hv, P);
        lam = lb_ > lam ? lb_ : lam;
      }
    }

    // slide the window one row down
    hC = hN; huC = huN; hvC = hvN; uC = uN; vC = vN; gzxC = gzxN;
    b0 = bp1; bp1 = bp2;
    fx = fn;
    gC = gN; oC = oN; gN = gNN; oN = oNN; sN = sNN;
  }
}

// A tile's place: its first row, rows and column, and the entry of row i0 - 2.
struct TileHead {
  int i0, nr, c0;
  const GS_C uint64_t* E;
};
template <typename T>
__device__ __forceinline__ TileHead tile_head(const GS_C FlatK<T>* k, int64_t t) {
  const GS_C int32_t* irc = cp(gp((int32_t*)k->tile_irc)) + 3 * t;
  return {irc[0], irc[1], irc[2], cp(gp((uint64_t*)k->ent)) + 3 * cp(gp((int64_t*)k->tile_e0))[t]};
}

// One row-sweep tile: the fused update of the active lanes of rows i0 .. i0+nr-1 of one
// 64-column window. Every lane of the wavefront must call it. PRE: also write the pre-friction
// state (the adjoint's recomputation); a separate instantiation keeps those pointers out of the
// plain step's scalar registers. LEAN: the domain has no per-cell Manning field or class plane, no
// running maximum and no active-cell forcing, so none of their pointers is held (the host checks
// that they are all null).
template <typename T, bool PRE, bool EXT, bool LEAN = false, int ROWS = kRowsOf<LEAN>>
__device__ __forceinline__ void flat_tile(const FlatCtx<T>& x, const TileHead& h, int lane, lam_t<T>& lam) {
  const int i0 = h.i0, nr = h.nr, c0 = h.c0;
  const GS_C uint64_t* E = h.E;
  int r = 0;
  if constexpr (ROWS != kRowsGeneral) {
    constexpr int forms = ROWS == kRowsQuick ? kWaveFast | kWaveLam : kWaveFast;
    if ((x.wave & forms) == forms && vabs(x.eta) < T(0x1p30) && nr <= kWaveRows) {
      const WaveC<T> w = wave_consts<T>(x.P, x.dt, x.wave);
      r = __builtin_amdgcn_readfirstlane(flat_rows<T, PRE, EXT, LEAN, ROWS>(x, w, E, i0, nr, c0, lane, lam));
    }
  }
  if (r < nr) flat_rows_general<T, PRE, EXT, LEAN, ROWS == kRowsGeneral>(x, E + 3 * r, i0 + r, nr - r, c0, lane, lam);
}

// Workgroup b's place in an XCD-major order: workgroups are dealt round-robin to the 8
// XCDs, so giving each XCD a contiguous range of wavefronts (hence of chunks in every
// pass) keeps the rows i+-1 that a chunk gathers mostly in that XCD's L2.
__device__ __forceinline__ unsigned xcd_rank(unsigned b, unsigned nb) {
  const unsigned qd = nb / 8u, rm = nb % 8u, xcd = b % 8u, kk = b / 8u;
  return xcd * qd + min(xcd, rm) + kk;   // the first rm XCDs have one more
}

// One step of one flat domain on a resident grid, each wavefront striding over chunks.
template <typename T, int MODE>
__global__ __launch_bounds__(kFBlock) void k_flat_step(FlatK<T> a, double next_dt) {
  const FlatClk<T> ck = flat_clock<T, MODE>(a);
  if (!ck.live) return;   // the whole grid sees the same clock
  FlatCtx<T> x;
  flat_ctx<T, MODE>(a, ck, x);
  __shared__ T s_ntab[GS_MAX_CLASSES];
  if (MODE == 1)
    for (int k = (int)threadIdx.x; k < a.n_classes; k += (int)blockDim.x) s_ntab[k] = a.ntab[k];
  __syncthreads();
  x.ntab = s_ntab;
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * (kFBlock / 64);
  lam_t<T> lam = 0;
  for (int64_t chunk = (int64_t)xcd_rank(blockIdx.x, gridDim.x) * (kFBlock / 64) + (threadIdx.x >> 6);
       chunk < a.nchunks; chunk += nwaves)
    flat_chunk<T, MODE>(x, chunk, lane, lam);
  if (MODE == 1) grid_reduce_and_plan(lam, a.clock, a.plan, true, next_dt);
}

// The forcings on the ring cells of the band (stored, not active): out = force(in), one thread per
// listed id, by `blocks` workgroups. The step itself only reads these cells, from the input buffer,
// so the two never touch the same word.
template <typename T>
__device__ __forceinline__ void ring_cells(const FlatK<T>& a, const FlatCtx<T>& x, unsigned block, unsigned blocks) {
  const bool sp = x.sponge != nullptr, cl = x.clamp != nullptr;
  const GS_G int64_t* ids = gp(a.fring);
  const GS_G int32_t* rows = gp(a.fring_row);
  // gauge stage weights at the step's start time (uniform: every thread takes the same path)
  T wa = T(0), wb = T(0);
  int ti = 0;
  if (rows) {
    const double* tc = a.ring_t;
    const double t = gp(a.clock)->t;
    // bisect_left: the number of samples below t
    ti = table_count(tc, 0, a.ring_nt, [t](double v) { return v < t; }) - 1;
    if (ti > a.ring_nt - 2) ti = a.ring_nt - 2;
    if (ti < 0) ti = 0;
    double wt = (t - tc[ti]) / (tc[ti + 1] - tc[ti] + 1.0e-12);
    wt = wt < 1.0 ? wt : 1.0;
    wt = wt > 0.0 ? wt : 0.0;
    wa = (T)(1.0 - wt);
    wb = (T)wt;
  }
  for (int64_t i = (int64_t)block * blockDim.x + threadIdx.x; i < a.n_fring; i += (int64_t)blocks * blockDim.x) {
    const int64_t k = ids[i];
    T h = x.qi0[k], hu = x.qi1[k], hv = x.qi2[k];
    const bool fc = x.flags != nullptr && (x.flags[k] & GS_FLAG_FORCE);
    if (fc && sp) sponge_cell<T>(x.sponge[2 * k], x.sponge[2 * k + 1], h, hu, hv);
    const int r = rows ? rows[i] : -1;
    if (r >= 0) {
      const GS_G T* w = gp(a.ring_w) + (int64_t)r * a.ring_ng;
      const GS_G T* S = gp(a.ring_stage);
      T eta = T(0);
      for (int g = 0; g < a.ring_ng; ++g) {
        const T sg = S[(int64_t)g * a.ring_nt + ti] * wa + S[(int64_t)g * a.ring_nt + ti + 1] * wb;
        eta = eta + w[g] * sg;
      }
      const T d = eta - gp(a.ring_bed)[r];
      h = d > T(0) ? d : T(0);   // fmaxf(0, d): NaN gives 0
      hu = T(0);
      hv = T(0);
    }
    if (fc && cl) clamp_cell<T>(x.clamp[k], h, hu, hv);
    if (fc && x.drain) drain_cell<T>(x.drain[k], h, hu, hv);
    x.qo0[k] = h;
    x.qo1[k] = hu;
    x.qo2[k] = hv;
  }
}

// Launched just before the chunk traversal on the same stream: it reads the clock the step will read.
template <typename T>
__global__ __launch_bounds__(kFBlock) void k_flat_ring_force(FlatK<T> a) {
  const FlatClk<T> ck = flat_clock<T, 1>(a);
  if (!ck.live) return;
  FlatCtx<T> x;
  flat_ctx<T, 1>(a, ck, x);
  ring_cells<T>(a, x, blockIdx.x, gridDim.x);
}

// One step of one flat domain by row-sweep tiles, one wavefront per tile in band-major tile
// order and XCD-major wavefront order. What bounds it is the issue of vector instructions (about
// 400 per row, 0.8 of the cycles) and, on a domain of one round of tiles, the slowest tile. The
// float32 steps are held to 80 VGPRs (6 wavefronts per SIMD), where no row reloads a spilled
// register. LEAN (a domain with no per-cell Manning field or class plane, running maximum or
// active-cell forcing) drops those paths. us per step, general functions with 4-row tiles before
// and wavefront forms now: 2048^2 coastal domain (lean) 63 and 38, 1500^2 with the forcing tail
// (below) 69 and 45.
template <typename T, bool PRE, bool LEAN = false, int ROWS = kRowsOf<LEAN>>
__global__ __launch_bounds__(kSBlock<T>) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 6 : 1))) void k_flat_sweep(FlatK<T> a, FlatLaunch<T> l) {
  // What waits on nothing but the argument is asked for first: the tile's place, the Manning table
  // and the clock. Each wavefront keeps its own copy of the table, so that none waits for another
  // (2048^2 coastal step: 38.4 us against 39.5; the extended sweep, with fewer registers to spare,
  // gained nothing from it and keeps the shorter form).
  const GS_C FlatK<T>* k = kernel_arg<T>();
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const unsigned rb = LEAN || PRE ? 0u : l.ring_blocks;
  const bool ring = blockIdx.x < rb;
  const int64_t nwaves = (int64_t)(gridDim.x - rb) * kSweepWaves<T>;
  int64_t t = (int64_t)xcd_rank(blockIdx.x - rb, gridDim.x - rb) * kSweepWaves<T> + wv;
  TileHead h = tile_head<T>(k, !ring && t < a.n_tiles ? t : a.n_tiles - 1);   // (a ring workgroup's is not used)
  __shared__ T s_ntab[kSweepWaves<T>][GS_MAX_CLASSES];
  const T n_mine = lane < a.n_classes ? gp(a.ntab)[lane] : T(0);
  const FlatClk<T> ck = flat_clock<T, 1>(a);
  if (LEAN && l.smp_n > 0 && blockIdx.x == gridDim.x - 1 && wv == 0) {
    const GS_G T* h0 = gp(ck.par ? a.buf[1][0] : a.buf[0][0]);
    for (int i = lane; i < l.smp_n; i += 64) gp(l.smp_out)[i] = h0[gp(l.smp_ids)[i]];
  }
  if (!ck.live) return;   // the whole grid sees the same clock
  FlatCtx<T> x;
  flat_ctx<T, 1>(a, ck, x);
  x.k = k;
  s_ntab[wv][lane] = n_mine;
  for (int c = lane + 64; c < a.n_classes; c += 64) s_ntab[wv][c] = gp(a.ntab)[c];
  x.ntab = s_ntab[wv];
  lam_t<T> lam = 0;
  // PRE (the adjoint's recomputation) also compiles the extended forcings in unless it is LEAN, so
  // that a replay reads rain through the per-cell lookup exactly as the forward run's extended sweep
  if (ring) ring_cells<T>(a, x, blockIdx.x, rb);
  while (!ring && t < a.n_tiles) {
    flat_tile<T, PRE, PRE && !LEAN, LEAN, ROWS>(x, h, lane, lam);
    t += nwaves;
    if (t < a.n_tiles) h = tile_head<T>(cold_ptr<T>(k), t);
  }
  grid_reduce_and_plan(lam, a.clock, a.plan, true, next_dt_arg<T>());
}

// The sweep with the extended forcings compiled in: Green-Ampt infiltration, drain-tau and
// rain read through a per-cell lookup into a native-grid table (launched only when one of
// them is set).
template <typename T>
__global__ __launch_bounds__(kSBlock<T>) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 6 : 1))) void k_flat_sweep_ext(FlatK<T> a, FlatLaunch<T> l) {
  const FlatClk<T> ck = flat_clock<T, 1>(a);
  if (!ck.live) return;
  FlatCtx<T> x;
  flat_ctx<T, 1>(a, ck, x);
  x.k = kernel_arg<T>();
  __shared__ T s_ntab[GS_MAX_CLASSES];
  for (int k = (int)threadIdx.x; k < a.n_classes; k += (int)blockDim.x) s_ntab[k] = a.ntab[k];
  __syncthreads();
  x.ntab = s_ntab;
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const unsigned rb = l.ring_blocks;
  const bool ring = blockIdx.x < rb;
  const int64_t nwaves = (int64_t)(gridDim.x - rb) * kSweepWaves<T>;
  lam_t<T> lam = 0;
  if (ring) ring_cells<T>(a, x, blockIdx.x, rb);
  for (int64_t t = (int64_t)xcd_rank(blockIdx.x - rb, gridDim.x - rb) * kSweepWaves<T> + wv; !ring && t < a.n_tiles;
       t += nwaves)
    flat_tile<T, false, true>(x, tile_head<T>(cold_ptr<T>(x.k), t), lane, lam);
  grid_reduce_and_plan(lam, a.clock, a.plan, true, next_dt_arg<T>());
}

// The ring modes of the cached replay on the step's input state, before the step reads
// it: each listed ring cell is overwritten from its active neighbour (extrapolate), with
// still water (stage), or with still-water depth and the neighbour's velocity. Only ring
// cells are written and only active cells (which nothing writes here) are read from.
template <typename T>
__global__ __launch_bounds__(kFBlock) void k_flat_ring_mode(FlatK<T> a) {
  const FlatClk<T> ck = flat_clock<T, 1>(a);
  if (!ck.live) return;
  FlatCtx<T> x;
  flat_ctx<T, 1>(a, ck, x);
  GS_G T* q0 = (GS_G T*)x.qi0;
  GS_G T* q1 = (GS_G T*)x.qi1;
  GS_G T* q2 = (GS_G T*)x.qi2;
  const GS_G int64_t* ids = gp(a.rmode_ids);
  const GS_G int64_t* nbs = gp(a.rmode_nb);
  const GS_G uint8_t* kind = gp(a.rmode_kind);
  for (int64_t i = (int64_t)blockIdx.x * kFBlock + threadIdx.x; i < a.n_rmode; i += (int64_t)gridDim.x * kFBlock) {
    const int64_t k = ids[i];
    const int kd = kind[i];
    if (kd == 0) {
      const int64_t nb = nbs[i];
      q0[k] = q0[nb];
      q1[k] = q1[nb];
      q2[k] = q2[nb];
      continue;
    }
    const T d = a.rmode_eta - x.bed[k];
    const T h = d > T(0) ? d : T(0);
    T hu = T(0), hv = T(0);
    if (kd == 2) {
      const int64_t nb = nbs[i];
      const T hn = q0[nb];
      const T inv = hn > a.P.h_min ? T(1) / hn : T(0);
      hu = h * (q1[nb] * inv);
      hv = h * (q2[nb] * inv);
    }
    q0[k] = h;
    q1[k] = hu;
    q2[k] = hv;
  }
}

// CFL wave speed of the current flat state over active cells, then plan dt.
template <typename T>
__global__ __launch_bounds__(kFBlock) void k_flat_cfl(FlatK<T> a) {
  const int par = (int)(a.clock->nsteps & 1);
  T* const* q = a.buf[par];
  lam_t<T> lam = 0;
  for (int64_t r = (int64_t)blockIdx.x * (kFBlock / 64) + (threadIdx.x >> 6); r < a.n_runs;
       r += (int64_t)gridDim.x * (kFBlock / 64)) {
    const int64_t k0 = a.run_k0[r];
    const int len = a.run_len[r];
    for (int t = threadIdx.x & 63; t < len; t += 64) {
      const int64_t k = k0 + t;
      if (a.flags && (a.flags[k] & GS_FLAG_CFL_SKIP)) continue;
      const lam_t<T> l = lam_key<T, true>(q[0][k], q[1][k], q[2][k], a.P);
      lam = l > lam ? l : lam;
    }
  }
  grid_reduce_and_plan(lam, a.clock, a.plan, false);
}

template <typename T>
static int build_flat(const GsFlat* f, const GsPhys* p, const GsForcing& fo, GsClock* clk, FlatK<T>& a,
                      bool need_clock) {
  if (!f) return fail(GS_E_ARG, "flat descriptor is NULL");
  if (f->n_stored < 1 || f->n_stored > ((int64_t)1 << 40)) return fail(GS_E_RANGE, "n_stored out of range");
  if (f->n_runs < 0) return fail(GS_E_ARG, "n_runs < 0");
  if (f->n_runs > 0 && (!f->run_k0 || !f->run_len || !f->run_i || !f->run_j0 || !f->run_d || !f->chunk_run))
    return fail(GS_E_ARG, "run tables are NULL");
  if (f->n_tiles < 0) return fail(GS_E_ARG, "n_tiles < 0");
  if (f->n_tiles > 0 && (!f->tile_e0 || !f->tile_irc || !f->ent)) return fail(GS_E_ARG, "tile tables are NULL");
  if (f->n_force_ring < 0 || f->n_force_ring > f->n_stored) return fail(GS_E_RANGE, "n_force_ring out of range");
  if (f->n_ring_mode < 0 || f->n_ring_mode > f->n_stored) return fail(GS_E_RANGE, "n_ring_mode out of range");
  if (f->n_ring_mode > 0 && (!f->ring_mode_ids || !f->ring_mode_nb || !f->ring_mode_kind))
    return fail(GS_E_ARG, "ring mode arrays are NULL");
  if (f->ga_ks && (!f->ga_cls || !f->ga_psi || !f->ga_dth || !f->ga_F))
    return fail(GS_E_ARG, "Green-Ampt needs the soil class, psi, dth and F arrays");
  if (f->n_force_ring > 0 && !f->force_ring) return fail(GS_E_ARG, "force_ring is NULL");
  if (f->n_force_ring > 0 && !f->sponge && !f->clamp && !f->drain && !f->force_ring_row)
    return fail(GS_E_ARG, "force_ring lists cells but no sponge, clamp, drain or gauge ring is set");
  if (f->force_ring_row && (f->ring_ng < 1 || f->ring_nt < 2 || !f->ring_bed || !f->ring_w || !f->ring_t ||
                            !f->ring_stage))
    return fail(GS_E_ARG, "gauge ring: needs >= 1 gauge, >= 2 time samples and its bed, weight, time and stage "
                "arrays");
  if (!f->bed) return fail(GS_E_ARG, "bed is NULL");
  for (int s = 0; s < 2; ++s)
    for (int k = 0; k < 3; ++k)
      if (!f->q[s][k]) return fail(GS_E_ARG, "state q[%d][%d] is NULL", s, k);
  int rc = check_phys(p);
  if (rc) return rc;
  rc = check_forcing(fo);
  if (rc) return rc;
  if (p->friction && !f->ntab && !f->n_field) return fail(GS_E_ARG, "friction needs ntab or n_field");
  if (need_clock && !clk) return fail(GS_E_ARG, "clock is NULL");
  memset(&a, 0, sizeof a);
  a.n = f->n_stored;
  a.n_runs = f->n_runs;
  a.nyp = f->nyp;
  a.ngh = f->ngh;
  a.nchunks = (f->n_stored + kFOut - 1) / kFOut;
  for (int s = 0; s < 2; ++s)
    for (int k = 0; k < 3; ++k) a.buf[s][k] = (T*)f->q[s][k];
  a.bed = (const T*)f->bed;
  a.flags = f->flags;
  a.ntab = (const T*)f->ntab;
  a.n_classes = f->ntab ? (p->n_classes > 0 ? p->n_classes : 1) : 0;
  a.n_field = (const T*)f->n_field;
  a.max_h = (T*)f->max_h;
  a.cls = f->cls;
  a.run_k0 = f->run_k0;
  a.run_len = f->run_len;
  a.run_i = f->run_i;
  a.run_j0 = f->run_j0;
  a.run_d = f->run_d;
  a.chunk_run = f->chunk_run;
  a.n_tiles = f->n_tiles;
  a.tile_e0 = f->tile_e0;
  a.tile_irc = f->tile_irc;
  a.ent = f->ent;
  a.sponge = (const T*)f->sponge;
  a.clamp = (const T*)f->clamp;
  a.infil = (const T*)f->infil;
  a.drain = (const T*)f->drain;
  a.ga_cls = f->ga_cls;
  a.ga_ks = (const T*)f->ga_ks;
  a.ga_psi = (const T*)f->ga_psi;
  a.ga_dth = (const T*)f->ga_dth;
  a.ga_F = (T*)f->ga_F;
  a.ga_fmax = (const T*)f->ga_fmax;
  a.ga_inv_tau = (const T*)f->ga_inv_tau;
  a.n_fring = f->n_force_ring;
  a.fring = f->force_ring;
  a.fring_row = f->force_ring_row;
  a.ring_ng = f->ring_ng;
  a.ring_nt = f->ring_nt;
  a.ring_bed = (const T*)f->ring_bed;
  a.ring_w = (const T*)f->ring_w;
  a.ring_t = f->ring_t;
  a.ring_stage = (const T*)f->ring_stage;
  a.P = make_phys<T>(*p, f->dx, f->dy);
  // the wavefront forms address a tile's rows and their stencil with 32-bit offsets
  const int64_t span = (kWaveRows + 4) * (int64_t)sizeof(T);
  a.wave = (int64_t)f->nyp * span < ((int64_t)1 << 31) && fo.rain_row_pitch * span < ((int64_t)1 << 31)
               ? wave_flags<T>(a.P, true)
               : 0;
  a.rain_mode = fo.n_rain > 0 ? (fo.rain_gridded ? (f->rain_lookup ? 3 : 2) : 1) : 0;
  a.rain_lookup = f->rain_lookup;
  a.n_rmode = f->n_ring_mode;
  a.rmode_ids = f->ring_mode_ids;
  a.rmode_nb = f->ring_mode_nb;
  a.rmode_kind = f->ring_mode_kind;
  a.rmode_eta = (T)f->ring_mode_eta;
  a.rain_frames = (const T*)fo.rain_frames;
  a.frame_stride = fo.rain_frame_stride;
  a.rain_pitch = fo.rain_row_pitch;
  a.clock = clk;
  a.plan = make_plan(*p, fo);
  return GS_OK;
}

// Workgroups of a one-wavefront-per-item kernel that are resident at once on the current
// device (cached per device and kernel); the grid never exceeds the work.
template <typename F>
static unsigned resident_grid(F kern, std::atomic<int>* cache, int64_t items, int block = kFBlock) {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) dev = -1;
  int per = (dev >= 0 && dev < 64) ? cache[dev].load(std::memory_order_relaxed) : 0;
  if (per <= 0) {
    int occ = 0, cus = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, kern, block, 0) != hipSuccess) occ = 4;
    if (dev < 0 || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) cus = 256;
    per = (occ > 0 ? occ : 1) * (cus > 0 ? cus : 1);
    if (dev >= 0 && dev < 64) cache[dev].store(per, std::memory_order_relaxed);
  }
  const int64_t need = (items + block / 64 - 1) / (block / 64);
  return (unsigned)(need < per ? (need > 0 ? need : 1) : per);
}

template <typename T, int MODE>
static unsigned flat_grid(int64_t nchunks) {
  static std::atomic<int> cache[64];
  return resident_grid(k_flat_step<T, MODE>, cache, nchunks);
}

// The sweeps launch one wavefront per tile: the hardware then keeps every SIMD fed until the last
// tile, where a resident grid striding over the tiles leaves a partial last round and ends all its
// workgroups at once, whose atomics then queue with nothing beside them (one wavefront per tile
// against the resident grid: 1536^2 adjoint with its 80 sweeps 10.85 against 11.48 ms, 2048^2 lean
// 43.1 against 43.5 us per step, 1500^2 with the forcing tail 64.1 against 65.7).
template <typename T>
static unsigned sweep_grid(int64_t ntiles) {
  return (unsigned)((ntiles + kSweepWaves<T> - 1) / kSweepWaves<T>);
}

// The domain may take the LEAN sweep: nothing it would skip is set.
template <typename T>
static bool flat_lean(const FlatK<T>& a) {
  return !a.n_field && !a.cls && !a.max_h && !a.sponge && !a.clamp && !a.infil && !a.drain;
}

// The step takes the extended sweep.
template <typename T>
static bool flat_ext(const FlatK<T>& a) {
  return a.ga_ks || a.ga_inv_tau || a.rain_mode == 3;
}

// The ring cells by workgroups of the sweep itself, ahead of its tiles (a launch of their own took
// 8 us beside a 46 us sweep: 1500^2 with the forcing tail 547 -> 484 us for 10 steps); the lean sweep,
// which only a gauge ring by itself would bring here, has no register for them. 0: a launch of their
// own, or none to force.
template <typename T>
static unsigned sweep_ring_blocks(const FlatK<T>& a) {
  if (a.n_fring <= 0 || a.n_tiles <= 0 || a.pre[0] || !(flat_ext(a) || !flat_lean(a))) return 0;
  const int64_t nb = (a.n_fring + kSBlock<T> - 1) / kSBlock<T>;
  return (unsigned)(((nb < 1024 ? nb : 1024) + 7) / 8 * 8);
}

// Its rows, where they may take the wavefront forms, know the wave speed from the update.
template <typename T>
static bool flat_quick(const FlatK<T>& a) {
  return !(a.wave & kWaveFast) || (a.wave & kWaveLam);
}

// The rows of the lean and the plain sweep for `a`. The general functions alone where the forms may not
// be taken at all (h_min below 2^-21 in float32), and for a float64 step of up to one wavefront per
// SIMD, which is one tile's latency (us per lean step with and without the forms: 64^2 14.0 and 12.8,
// 150^2 14.2 and 13.1, 400^2 of 864 tiles 18.2 and 17.8; but 500^2 of 1230 tiles 20.7 and 20.7, 700^2 of 2250
// 23.8 and 25.1). The extended sweep gains nothing from it: 400^2 with the forcing tail 22.8 us against 21.5.
template <typename T>
static int sweep_rows_kind(const FlatK<T>& a) {
  if (!(a.wave & kWaveFast) || (sizeof(T) == 8 && a.n_tiles <= 1024)) return kRowsGeneral;
  return flat_quick(a) ? kRowsQuick : kRowsAny;
}

template <typename T, bool PRE>
static auto lean_sweep(const FlatK<T>& a) -> void (*)(FlatK<T>, FlatLaunch<T>) {
  switch (sweep_rows_kind(a)) {
    case kRowsGeneral: return k_flat_sweep<T, PRE, true, kRowsGeneral>;
    case kRowsAny: return k_flat_sweep<T, PRE, true, kRowsAny>;
    default: return k_flat_sweep<T, PRE, true, kRowsQuick>;
  }
}
template <typename T>
static auto plain_sweep(const FlatK<T>& a) -> void (*)(FlatK<T>, FlatLaunch<T>) {
  return sweep_rows_kind(a) == kRowsGeneral ? k_flat_sweep<T, false, false, kRowsGeneral> : k_flat_sweep<T, false, false>;
}
// Each one's number, for a cache by kernel.
template <typename T>
static int sweep_slot(const FlatK<T>& a) {
  return (flat_ext(a) ? 6 : flat_lean(a) ? 0 : 3) + sweep_rows_kind(a);
}

// The launch gs_flat_step makes for `a` (without the pre-friction state): which kernel, its
// grid and the kernel's resident grid on this device.
template <typename T>
static void flat_launch_choice(const FlatK<T>& a, int* kernel, int64_t* blocks, int64_t* resident) {
  static std::atomic<int> cache[9][64];
  if (a.n_tiles <= 0) {
    *kernel = 0;
    *blocks = flat_grid<T, 1>(a.nchunks);
    *resident = *blocks;
    return;
  }
  auto kern = flat_ext(a) ? k_flat_sweep_ext<T> : flat_lean(a) ? lean_sweep<T, false>(a) : plain_sweep(a);
  *kernel = flat_ext(a) ? 2 : 1;
  *blocks = sweep_grid<T>(a.n_tiles) + sweep_ring_blocks(a);
  *resident = resident_grid(kern, cache[sweep_slot(a)], a.n_tiles, kSBlock<T>);
}

// The fused step: row-sweep tiles when the descriptor has them, else chunks of the run table.
template <typename T>
static int flat_step_launch(const FlatK<T>& a, FlatLaunch<T> l, hipStream_t s) {
  if (a.n_rmode > 0) {
    const int64_t nb = (a.n_rmode + kFBlock - 1) / kFBlock;
    hipLaunchKernelGGL((k_flat_ring_mode<T>), dim3((unsigned)(nb < 1024 ? nb : 1024)), dim3(kFBlock), 0, s, a);
    GS_HIP(hipGetLastError(), "k_flat_ring_mode launch");
  }
  const bool ext = flat_ext(a);
  l.ring_blocks = sweep_ring_blocks(a);
  if (a.n_fring > 0 && l.ring_blocks == 0) {
    const int64_t nb = (a.n_fring + kFBlock - 1) / kFBlock;
    hipLaunchKernelGGL((k_flat_ring_force<T>), dim3((unsigned)(nb < 1024 ? nb : 1024)), dim3(kFBlock), 0, s, a);
    GS_HIP(hipGetLastError(), "k_flat_ring_force launch");
  }
  if (a.n_tiles > 0 && a.pre[0] && !ext && flat_lean(a)) {
    // 1536^2 adjoint: 33.5 us against the general pre-friction sweep's 36
    hipLaunchKernelGGL((lean_sweep<T, true>(a)), dim3(sweep_grid<T>(a.n_tiles)), dim3(kSBlock<T>), 0, s, a, l);
    GS_HIP(hipGetLastError(), "k_flat_sweep(pre, lean) launch");
  } else if (a.n_tiles > 0 && a.pre[0]) {
    hipLaunchKernelGGL((k_flat_sweep<T, true>), dim3(sweep_grid<T>(a.n_tiles)), dim3(kSBlock<T>), 0, s, a, l);
    GS_HIP(hipGetLastError(), "k_flat_sweep(pre) launch");
  } else if (a.n_tiles > 0 && ext) {
    hipLaunchKernelGGL((k_flat_sweep_ext<T>), dim3(sweep_grid<T>(a.n_tiles) + l.ring_blocks), dim3(kSBlock<T>), 0, s, a, l);
    GS_HIP(hipGetLastError(), "k_flat_sweep_ext launch");
  } else if (a.n_tiles > 0 && flat_lean(a)) {
    hipLaunchKernelGGL((lean_sweep<T, false>(a)), dim3(sweep_grid<T>(a.n_tiles)), dim3(kSBlock<T>), 0, s, a, l);
    GS_HIP(hipGetLastError(), "k_flat_sweep(lean) launch");
  } else if (a.n_tiles > 0) {
    hipLaunchKernelGGL(plain_sweep(a), dim3(sweep_grid<T>(a.n_tiles) + l.ring_blocks), dim3(kSBlock<T>), 0, s, a, l);
    GS_HIP(hipGetLastError(), "k_flat_sweep launch");
  } else {
    hipLaunchKernelGGL((k_flat_step<T, 1>), dim3(flat_grid<T, 1>(a.nchunks)), dim3(kFBlock), 0, s, a, l.next_dt);
    GS_HIP(hipGetLastError(), "k_flat_step launch");
  }
  return GS_OK;
}

// Depth of the current state at listed flat ids (gauges), read after a step.
template <typename T>
__global__ void k_flat_sample(FlatK<T> a, const int64_t* ids, int n, T* out) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int par = (int)(a.clock->nsteps & 1);
  out[t] = a.buf[par][0][ids[t]];
}

template <typename T>
static int flat_step_t(const GsFlat* f, const GsPhys* p, GsForcing fo, GsClock* clk, hipStream_t s,
                       void* pre0 = nullptr, void* pre1 = nullptr, void* pre2 = nullptr, double next_dt = 0.0,
                       const FlatSample* smp = nullptr) {
  FlatK<T> a;
  int rc = build_flat<T>(f, p, fo, clk, a, true);
  if (rc) return rc;
  FlatLaunch<T> l;
  l.next_dt = next_dt;
  if ((pre0 || pre1 || pre2) && !(pre0 && pre1 && pre2)) return fail(GS_E_ARG, "pre: all three planes or none");
  if (pre0 && a.n_tiles == 0)
    return fail(GS_E_ARG, "the pre-friction state is written by the row-sweep traversal only (n_tiles > 0)");
  a.pre[0] = (T*)pre0;
  a.pre[1] = (T*)pre1;
  a.pre[2] = (T*)pre2;
  if (smp && a.n_tiles > 0 && a.n_rmode == 0 && !pre0 && !flat_ext(a) && flat_lean(a)) {
    // by a wavefront of the sweep, on its way (not where a ring mode overwrites cells of the sweep's
    // input ahead of it)
    l.smp_ids = smp->ids;
    l.smp_n = smp->n;
    l.smp_out = (T*)smp->out;
  } else if (smp) {
    hipLaunchKernelGGL(k_flat_sample<T>, dim3((unsigned)((smp->n + 255) / 256)), dim3(256), 0, s, a, smp->ids, smp->n,
                       (T*)smp->out);
    GS_HIP(hipGetLastError(), "k_flat_sample launch");
  }
  return flat_step_launch<T>(a, l, s);
}

template <typename T>
static int flat_residual_t(const GsFlat* f, const GsPhys* p, int which, void* r0, void* r1, void* r2,
                           hipStream_t s) {
  GsForcing fo;
  memset(&fo, 0, sizeof fo);
  FlatK<T> a;
  int rc = build_flat<T>(f, p, fo, nullptr, a, false);
  if (rc) return rc;
  if (which < 0 || which > 1) return fail(GS_E_ARG, "which must be 0 or 1");
  if (!r0 || !r1 || !r2) return fail(GS_E_ARG, "residual arrays are NULL");
  a.which = which;
  a.rhs[0] = (T*)r0;
  a.rhs[1] = (T*)r1;
  a.rhs[2] = (T*)r2;
  hipLaunchKernelGGL((k_flat_step<T, 0>), dim3(flat_grid<T, 0>(a.nchunks)), dim3(kFBlock), 0, s, a, 0.0);
  GS_HIP(hipGetLastError(), "k_flat_step(residual) launch");
  return GS_OK;
}

template <typename T>
static int flat_cfl_t(const GsFlat* f, const GsPhys* p, GsForcing fo, GsClock* clk, hipStream_t s) {
  FlatK<T> a;
  int rc = build_flat<T>(f, p, fo, clk, a, true);
  if (rc) return rc;
  int64_t blocks = ((int64_t)a.n_runs + 3) / 4;
  if (blocks < 1) blocks = 1;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL((k_flat_cfl<T>), dim3((unsigned)blocks), dim3(kFBlock), 0, s, a);
  GS_HIP(hipGetLastError(), "k_flat_cfl launch");
  return GS_OK;
}


// ---------------------------------------------------------------------------
// batched ensemble: every member's sweep tiles in one launch, per-member clocks
// ---------------------------------------------------------------------------
template <typename T>
struct EnsK {
  const FlatK<T>* __restrict__ mem;   // member views (device)
  const int64_t* __restrict__ tile0;  // [n_members + 1] first global tile of each member
  int n_members;
  int tpp;                            // consecutive tiles per wavefront pass
  int64_t ntiles;                     // total tiles
  unsigned* done;                     // workgroups finished in this launch
};

// Fold a wavefront's CFL speed bits of member m into that member's clock (lane 0 waits
// until its atomic has been performed, as grid_reduce_and_plan's thread 0 does).
template <typename T>
__device__ __forceinline__ void ens_flush(const EnsK<T>& e, int m, lam_t<T> lam) {
  lam = wave_max(lam);
  if (m >= 0 && (threadIdx.x & 63) == 0 && lam)
    await_atomic(__hip_atomic_fetch_max(&e.mem[m].clock->lam_acc, lam_key_bits64(lam), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}

// The member that owns global tile gc (tile0: the members' tile prefix, n + 1 entries).
__device__ __forceinline__ int ens_member_of(const int64_t* tile0, int n, int64_t gc) {
  int lo = 0, hi = n;
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (const_read(tile0 + mid) <= gc) lo = mid;
    else hi = mid;
  }
  return lo;
}

// One step of every live member. The global tile space is the members' sweep tiles end to
// end; a wavefront takes `tpp` consecutive tiles per pass and strides by the grid (the
// autotuner usually picks one wavefront per tile, as the plain sweep launches), finding a
// tile's member by bisection of the tile prefix and reading the member's view and clock
// values from the member table with scalar loads. A wavefront folds its speed maximum into
// a member's clock when it leaves the member; its last maximum goes through the
// workgroup's thread 0, which folds the workgroup's maxima (one atomic per member) before
// counting the workgroup done. The last workgroup to finish plans each member's next dt
// from its own maximum (plan_finish), as the plain step's last workgroup does for its
// single domain; the hand-off orders atomics only, as grid_reduce_and_plan's does.
// KIND kEnsExt compiles the extended forcings (Green-Ampt, drain-tau, rain through a
// per-cell lookup) in; kEnsPlain leaves them out; kEnsLean also leaves out the per-cell
// Manning field, the running maximum and the active-cell forcings (every member has none
// of them), and its float32 build is held to 96 VGPRs (5 wavefronts per SIMD, nothing spilled; at
// 80 and 6 the row loop reloads, and 16 members of 256 to 1024 cells a side took 90 us per step at
// 8 rows a tile against 84).
// kEnsLeanAny is kEnsLean where some member's wave speed is not the quick one (kRowsAny).
enum { kEnsPlain = 0, kEnsExt = 1, kEnsLean = 2, kEnsLeanAny = 3 };

// The members' clock statuses side by side, for one copy to the host.
template <typename T>
__global__ void k_ens_status(const FlatK<T>* mem, int n, int* out) {
  for (int m = blockIdx.x * blockDim.x + threadIdx.x; m < n; m += gridDim.x * blockDim.x) out[m] = mem[m].clock->status;
}

template <typename T, int KIND>
__global__ __launch_bounds__(kFBlock) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 && KIND >= kEnsLean ? 5 : 1)))
void k_ens_step(EnsK<T> e, const FlatK<T>* __restrict__ mem, const int64_t* __restrict__ tile0) {
  const int lane = threadIdx.x & 63;
  const int64_t nwaves = (int64_t)gridDim.x * (kFBlock / 64);
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int64_t wave = (int64_t)xcd_rank(blockIdx.x, gridDim.x) * (kFBlock / 64) + wv;
  const int64_t tpp = e.tpp;
  // the Manning table of the wavefront's member: a lookup beside the row's loads in flight must not
  // wait for them, as one in global memory would
  __shared__ T s_ntab[kFBlock / 64][GS_MAX_CLASSES];
  int m = -1;          // the member whose maximum `lam` holds
  lam_t<T> lam = 0;
  for (int64_t base = wave * tpp; base < e.ntiles; base += nwaves * tpp) {
    const int64_t stop = base + tpp < e.ntiles ? base + tpp : e.ntiles;
    for (int64_t gc = base; gc < stop; ++gc) {
      // the tile's member, its view and clock values, looked up per tile so that none of
      // them is held across tiles
      const int mt = ens_member_of(tile0, e.n_members, gc);
      if (mt != m) {
        ens_flush(e, m, lam);
        lam = 0;
        m = mt;
        const T* nt = const_read(&mem[mt].ntab);
        for (int k = lane; k < const_read(&mem[mt].n_classes); k += 64) s_ntab[wv][k] = gp(nt)[k];
      }
      const FlatK<T> v = const_read(mem + mt);
      const FlatClk<T> ck = flat_clock<T, 1>(v);
      if (!ck.live) continue;
      FlatCtx<T> x;
      flat_ctx<T, 1>(v, ck, x);
      x.k = cp((const GS_G FlatK<T>*)(mem + mt));
      x.ntab = s_ntab[wv];
      flat_tile<T, false, KIND == kEnsExt, (KIND >= kEnsLean), KIND == kEnsLean ? kRowsQuick : kRowsAny>(
          x, tile_head<T>(x.k, gc - const_read(tile0 + mt)), lane, lam);
    }
  }
  __shared__ int s_m[kFBlock / 64];
  __shared__ uint64_t s_l[kFBlock / 64];
  __shared__ int s_last;
  const uint64_t lw = lam_key_bits64(wave_max(lam));
  if (lane == 0) {
    s_m[wv] = m;
    s_l[wv] = lw;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 0; w < kFBlock / 64; ++w) {
      const int mw = s_m[w];
      const uint64_t l = s_l[w];
      if (mw < 0 || !l) continue;
      if (w + 1 < kFBlock / 64 && s_m[w + 1] == mw) {   // the next wave's member: fold into its slot
        s_l[w + 1] = s_l[w + 1] > l ? s_l[w + 1] : l;
        continue;
      }
      await_atomic(__hip_atomic_fetch_max(&e.mem[mw].clock->lam_acc, l, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    }
    const unsigned prev = __hip_atomic_fetch_add(e.done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    s_last = (prev == gridDim.x - 1) ? 1 : 0;
  }
  __syncthreads();
  if (!s_last) return;
  for (int mm = threadIdx.x; mm < e.n_members; mm += blockDim.x) {
    GsClock* c = e.mem[mm].clock;
    const ClockIn k = clock_read(c);
    if (k.status & GS_ST_DONE) continue;
    plan_finish(c, e.mem[mm].plan, k, true);
  }
  if (threadIdx.x == 0) __hip_atomic_store(e.done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <typename T>
static auto ens_kernel(int kind) -> void (*)(EnsK<T>, const FlatK<T>*, const int64_t*) {
  switch (kind) {
    case kEnsExt: return k_ens_step<T, kEnsExt>;
    case kEnsLean: return k_ens_step<T, kEnsLean>;
    case kEnsLeanAny: return k_ens_step<T, kEnsLeanAny>;
    default: return k_ens_step<T, kEnsPlain>;
  }
}

template <typename T>
static int ens_occupancy(int kind) {
  int occ = 0;
  const hipError_t h = hipOccupancyMaxActiveBlocksPerMultiprocessor(&occ, ens_kernel<T>(kind), kFBlock, 0);
  if (h != hipSuccess || occ < 1) occ = 1;
  return occ;
}

// The instantiation the members need: extended if any member has an extended forcing, lean
// if every member may take the lean sweep, else plain.
template <typename T>
static int ens_kind(const FlatK<T>* views, int n) {
  bool lean = true, quick = true;
  for (int m = 0; m < n; ++m) {
    if (flat_ext(views[m])) return kEnsExt;
    lean = lean && flat_lean(views[m]);
    quick = quick && flat_quick(views[m]);
  }
  return !lean ? kEnsPlain : quick ? kEnsLean : kEnsLeanAny;
}

template <typename T>
static void ens_launch_kind(int kind, int64_t blocks, hipStream_t s, const EnsK<T>& k) {
  hipLaunchKernelGGL((ens_kernel<T>(kind)), dim3((unsigned)blocks), dim3(kFBlock), 0, s, k, k.mem, k.tile0);
}

int flat_step_next(const GsFlat* f, const GsPhys* phys, const GsForcing& forc, GsClock* clock_dev, void* const* pre,
                   double next_dt, const FlatSample* smp, void* stream) {
  if (!f) return fail(GS_E_ARG, "flat descriptor is NULL");
  void *p0 = pre ? pre[0] : nullptr, *p1 = pre ? pre[1] : nullptr, *p2 = pre ? pre[2] : nullptr;
  if (pre && (!p0 || !p1 || !p2)) return fail(GS_E_ARG, "pre arrays are NULL");
  const hipStream_t s = (hipStream_t)stream;
  if (f->dtype == GS_F64) return flat_step_t<double>(f, phys, forc, clock_dev, s, p0, p1, p2, next_dt, smp);
  if (f->dtype == GS_F32) return flat_step_t<float>(f, phys, forc, clock_dev, s, p0, p1, p2, next_dt, smp);
  return fail(GS_E_DTYPE, "unsupported dtype %d", f->dtype);
}

}  // namespace gs

using namespace gs;

extern "C" {

int gs_flat_step(const GsFlat* f, const GsPhys* phys, GsForcing forc, GsClock* clock_dev, void* stream) {
  if (!f) return fail(GS_E_ARG, "flat descriptor is NULL");
  if (f->dtype == GS_F32) return flat_step_t<float>(f, phys, forc, clock_dev, (hipStream_t)stream);
  if (f->dtype == GS_F64) return flat_step_t<double>(f, phys, forc, clock_dev, (hipStream_t)stream);
  return fail(GS_E_DTYPE, "unsupported dtype %d", f->dtype);
}

int gs_flat_residual(const GsFlat* f, const GsPhys* phys, int which, void* rhs0, void* rhs1, void* rhs2,
                     void* stream) {
  if (!f) return fail(GS_E_ARG, "flat descriptor is NULL");
  if (f->dtype == GS_F32) return flat_residual_t<float>(f, phys, which, rhs0, rhs1, rhs2, (hipStream_t)stream);
  if (f->dtype == GS_F64) return flat_residual_t<double>(f, phys, which, rhs0, rhs1, rhs2, (hipStream_t)stream);
  return fail(GS_E_DTYPE, "unsupported dtype %d", f->dtype);
}

int gs_flat_cfl(const GsFlat* f, const GsPhys* phys, GsForcing forc, GsClock* clock_dev, void* stream) {
  if (!f) return fail(GS_E_ARG, "flat descriptor is NULL");
  if (f->dtype == GS_F32) return flat_cfl_t<float>(f, phys, forc, clock_dev, (hipStream_t)stream);
  if (f->dtype == GS_F64) return flat_cfl_t<double>(f, phys, forc, clock_dev, (hipStream_t)stream);
  return fail(GS_E_DTYPE, "unsupported dtype %d", f->dtype);
}

int gs_flat_launch_info(const GsFlat* f, const GsPhys* phys, GsForcing forc, int* kernel, int64_t* blocks,
                        int64_t* resident) {
  using namespace gs;
  if (!f || !kernel || !blocks || !resident) return fail(GS_E_ARG, "gs_flat_launch_info: NULL argument");
  if (f->dtype == GS_F32) {
    FlatK<float> a;
    const int rc = build_flat<float>(f, phys, forc, nullptr, a, false);
    if (rc) return rc;
    flat_launch_choice<float>(a, kernel, blocks, resident);
  } else if (f->dtype == GS_F64) {
    FlatK<double> a;
    const int rc = build_flat<double>(f, phys, forc, nullptr, a, false);
    if (rc) return rc;
    flat_launch_choice<double>(a, kernel, blocks, resident);
  } else {
    return fail(GS_E_DTYPE, "unsupported dtype %d", f->dtype);
  }
  return GS_OK;
}

int gs_flat_step_pre(const GsFlat* f, const GsPhys* phys, GsForcing forc, GsClock* clock_dev, void* pre0,
                     void* pre1, void* pre2, void* stream) {
  using namespace gs;
  if (!pre0 || !pre1 || !pre2) return fail(GS_E_ARG, "pre arrays are NULL");
  if (!f) return fail(GS_E_ARG, "flat descriptor is NULL");
  if (f->dtype == GS_F64)
    return flat_step_t<double>(f, phys, forc, clock_dev, (hipStream_t)stream, pre0, pre1, pre2);
  if (f->dtype == GS_F32)
    return flat_step_t<float>(f, phys, forc, clock_dev, (hipStream_t)stream, pre0, pre1, pre2);
  return fail(GS_E_DTYPE, "unsupported dtype %d", f->dtype);
}

int gs_flat_sample(const GsFlat* f, const GsClock* clock_dev, const int64_t* ids, int n, void* out, void* stream) {
  using namespace gs;
  if (!f || !clock_dev || (n > 0 && (!ids || !out))) return fail(GS_E_ARG, "NULL argument");
  if (n < 0) return fail(GS_E_ARG, "n < 0");
  if (n == 0) return GS_OK;
  GsPhys p;
  memset(&p, 0, sizeof p);
  p.g = 9.81; p.h_min = 1e-6; p.h_cfl = 1e-6; p.cfl = 0.5; p.dmin = 1.0; p.n_classes = 1;
  GsForcing fo;
  memset(&fo, 0, sizeof fo);
  const unsigned nb = (unsigned)((n + 255) / 256);
  if (f->dtype == GS_F64) {
    FlatK<double> a;
    int rc = build_flat<double>(f, &p, fo, (GsClock*)clock_dev, a, true);
    if (rc) return rc;
    hipLaunchKernelGGL(k_flat_sample<double>, dim3(nb), dim3(256), 0, (hipStream_t)stream, a, ids, n, (double*)out);
  } else {
    FlatK<float> a;
    int rc = build_flat<float>(f, &p, fo, (GsClock*)clock_dev, a, true);
    if (rc) return rc;
    hipLaunchKernelGGL(k_flat_sample<float>, dim3(nb), dim3(256), 0, (hipStream_t)stream, a, ids, n, (float*)out);
  }
  GS_HIP(hipGetLastError(), "k_flat_sample launch");
  return GS_OK;
}


}  // extern "C"

// ---------------------------------------------------------------------------
// ensemble host object
// ---------------------------------------------------------------------------
struct GsEns {
  int dtype = 0;
  int n = 0;
  void* mem = nullptr;          // device FlatK<T>[n]
  int64_t* tile0 = nullptr;     // device [n + 1]
  unsigned* done = nullptr;     // device counter; the members' statuses (gs_ens_status) from byte 256
  int64_t ntiles = 0;
  int blocks = 0;               // 0: one occupancy wave of the device
  int tpp = 1;
  int cus = 256;
  int occ = 1;                  // resident k_ens_step workgroups per CU
  int kind = 0;                 // k_ens_step instantiation (kEnsPlain / kEnsExt / kEnsLean)
  std::vector<GsFlat> flat;
  std::vector<GsClock*> clocks;
  hipStream_t gstream = nullptr;
  hipEvent_t ev_in = nullptr, ev_out = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  int g_batch = 0, g_blocks = -1, g_tpp = -1;
};

namespace gs {

// Member m's view for k_ens_step, with the checks of what the ensemble step supports.
template <typename T>
static int ens_member_view(const GsFlat* members, const GsPhys* phys, const GsForcing* forcings,
                           GsClock* const* clocks, int m, FlatK<T>& v) {
  const int rc = build_flat<T>(&members[m], &phys[m], forcings[m], clocks[m], v, true);
  if (rc) {
    char msg[512];
    snprintf(msg, sizeof msg, "%s", g_err);
    return fail(rc, "member %d: %s", m, msg);
  }
  if (v.n_runs > 0 && v.n_tiles < 1) return fail(GS_E_ARG, "member %d has active cells but no row-sweep tiles", m);
  if (v.n_rmode > 0) return fail(GS_E_ARG, "member %d has ring modes; the ensemble step does not apply them", m);
  if (v.n_fring > 0)
    return fail(GS_E_ARG, "member %d forces ring cells (gauge ring, or sponge or clamp outside the active set); the ensemble "
                "step updates active cells only", m);
  return GS_OK;
}

// Grid of one k_ens_step launch: `blocks` resident workgroups (0: one occupancy wave of the
// device), never more than the tiles need.
static int64_t ens_grid(int64_t blocks, int occ, int cus, int64_t ntiles, int tpp) {
  if (blocks <= 0) blocks = (int64_t)occ * cus;
  const int64_t need = (ntiles + 4LL * tpp - 1) / (4LL * tpp);
  if (blocks > need) blocks = need;
  return blocks < 1 ? 1 : blocks;
}

template <typename T>
static int ens_build_views(GsEns* e, const GsFlat* members, const GsPhys* phys, const GsForcing* forcings) {
  std::vector<FlatK<T>> views((size_t)e->n);
  std::vector<int64_t> c0((size_t)e->n + 1, 0);
  for (int m = 0; m < e->n; ++m) {
    const int rc = ens_member_view<T>(members, phys, forcings, e->clocks.data(), m, views[m]);
    if (rc) return rc;
    c0[m + 1] = c0[m] + views[m].n_tiles;
  }
  e->ntiles = c0[e->n];
  e->kind = ens_kind<T>(views.data(), e->n);
  e->occ = ens_occupancy<T>(e->kind);
  // until a launch shape is set: one wavefront per tile, as the plain sweep (16 members of 256 to
  // 1024 cells a side, tiles of 7 rows: 84 us per step; the resident grid's two rounds: 91)
  const int64_t per_tile = (e->ntiles + 3) / 4;
  e->blocks = (int)(per_tile < (1 << 24) ? per_tile : (1 << 24));
  GS_HIP(hipMalloc(&e->mem, sizeof(FlatK<T>) * (size_t)e->n), "ensemble views");
  GS_HIP(hipMalloc((void**)&e->tile0, sizeof(int64_t) * ((size_t)e->n + 1)), "ensemble tile table");
  GS_HIP(hipMalloc((void**)&e->done, 256 + 4 * (size_t)e->n), "ensemble counter");
  GS_HIP(hipMemcpy(e->mem, views.data(), sizeof(FlatK<T>) * (size_t)e->n, hipMemcpyHostToDevice), "views h2d");
  GS_HIP(hipMemcpy(e->tile0, c0.data(), sizeof(int64_t) * ((size_t)e->n + 1), hipMemcpyHostToDevice),
         "tile table h2d");
  GS_HIP(hipMemset(e->done, 0, 256), "counter clear");
  return GS_OK;
}

template <typename T>
static int ens_launch(GsEns* e, hipStream_t s) {
  EnsK<T> k;
  k.mem = (const FlatK<T>*)e->mem;
  k.tile0 = e->tile0;
  k.n_members = e->n;
  k.tpp = e->tpp;
  k.ntiles = e->ntiles;
  k.done = e->done;
  const int64_t blocks = ens_grid(e->blocks, e->occ, e->cus, e->ntiles, e->tpp);
  ens_launch_kind<T>(e->kind, blocks, s, k);
  GS_HIP(hipGetLastError(), "k_ens_step launch");
  return GS_OK;
}

static int ens_step(GsEns* e, hipStream_t s) {
  return e->dtype == GS_F64 ? ens_launch<double>(e, s) : ens_launch<float>(e, s);
}

static void ens_drop_graph(GsEns* e) {
  if (e->exec) (void)hipGraphExecDestroy(e->exec);
  if (e->graph) (void)hipGraphDestroy(e->graph);
  e->exec = nullptr;
  e->graph = nullptr;
  e->g_batch = 0;
}

static int ens_capture(GsEns* e, int batch) {
  ens_drop_graph(e);
  GS_HIP(hipStreamBeginCapture(e->gstream, hipStreamCaptureModeThreadLocal), "begin capture");
  int rc = GS_OK;
  for (int i = 0; i < batch && rc == GS_OK; ++i) rc = ens_step(e, e->gstream);
  hipGraph_t g = nullptr;
  const hipError_t ee = hipStreamEndCapture(e->gstream, &g);
  if (rc) {
    if (g) (void)hipGraphDestroy(g);
    return rc;
  }
  if (ee != hipSuccess) return hip_fail(ee, "end capture");
  e->graph = g;
  GS_HIP(hipGraphInstantiate(&e->exec, e->graph, nullptr, nullptr, 0), "graph instantiate");
  e->g_batch = batch;
  e->g_blocks = e->blocks;
  e->g_tpp = e->tpp;
  return GS_OK;
}

}  // namespace gs

extern "C" {

int gs_ens_create(const GsFlat* members, const GsPhys* phys, const GsForcing* forcings, GsClock* const* clocks,
                  int n_members, GsEns** out) {
  using namespace gs;
  if (!out) return fail(GS_E_ARG, "out is NULL");
  *out = nullptr;
  if (n_members < 1 || n_members > (1 << 20)) return fail(GS_E_RANGE, "n_members must be in 1..2^20");
  if (!members || !phys || !forcings || !clocks) return fail(GS_E_ARG, "member arrays are NULL");
  const int dt = members[0].dtype;
  if (dt != GS_F32 && dt != GS_F64) return fail(GS_E_DTYPE, "unsupported dtype %d", dt);
  for (int m = 0; m < n_members; ++m) {
    if (members[m].dtype != dt) return fail(GS_E_DTYPE, "member %d dtype differs from member 0", m);
    if (!clocks[m]) return fail(GS_E_ARG, "clock of member %d is NULL", m);
  }
  GsEns* e = new GsEns();
  e->dtype = dt;
  e->n = n_members;
  e->flat.assign(members, members + n_members);
  e->clocks.assign(clocks, clocks + n_members);
  int dev = 0;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&e->cus, hipDeviceAttributeMultiprocessorCount, dev);
  if (e->cus < 1) e->cus = 256;
  int rc = dt == GS_F64 ? ens_build_views<double>(e, members, phys, forcings)
                        : ens_build_views<float>(e, members, phys, forcings);
  if (rc == GS_OK) {
    hipError_t h = hipStreamCreateWithFlags(&e->gstream, hipStreamNonBlocking);
    if (h == hipSuccess) h = hipEventCreateWithFlags(&e->ev_in, hipEventDisableTiming);
    if (h == hipSuccess) h = hipEventCreateWithFlags(&e->ev_out, hipEventDisableTiming);
    if (h != hipSuccess) rc = hip_fail(h, "ensemble stream/events");
  }
  if (rc) {
    gs_ens_destroy(e);
    return rc;
  }
  *out = e;
  return GS_OK;
}

int gs_ens_status(GsEns* e, int* status, void* stream) {
  using namespace gs;
  if (!e || !status) return fail(GS_E_ARG, "gs_ens_status: NULL argument");
  hipStream_t s = (hipStream_t)stream;
  int* d = (int*)((char*)e->done + 256);
  const dim3 grid((unsigned)((e->n + 63) / 64)), block(64);
  if (e->dtype == GS_F64) hipLaunchKernelGGL(k_ens_status<double>, grid, block, 0, s, (const FlatK<double>*)e->mem, e->n, d);
  else hipLaunchKernelGGL(k_ens_status<float>, grid, block, 0, s, (const FlatK<float>*)e->mem, e->n, d);
  GS_HIP(hipGetLastError(), "k_ens_status launch");
  GS_HIP(hipMemcpyAsync(status, d, sizeof(int) * (size_t)e->n, hipMemcpyDeviceToHost, s), "ensemble status d2h");
  GS_HIP(hipStreamSynchronize(s), "ensemble status");
  return GS_OK;
}
int gs_ens_destroy(GsEns* e) {
  if (!e) return GS_OK;
  gs::ens_drop_graph(e);
  if (e->gstream) (void)hipStreamSynchronize(e->gstream);
  if (e->ev_in) (void)hipEventDestroy(e->ev_in);
  if (e->ev_out) (void)hipEventDestroy(e->ev_out);
  if (e->gstream) (void)hipStreamDestroy(e->gstream);
  if (e->mem) (void)hipFree(e->mem);
  if (e->tile0) (void)hipFree(e->tile0);
  if (e->done) (void)hipFree(e->done);
  delete e;
  return GS_OK;
}

int gs_ens_set_launch(GsEns* e, int blocks, int tiles_per_pass) {
  using namespace gs;
  if (!e) return fail(GS_E_ARG, "ensemble is NULL");
  if (blocks < 0 || blocks > (1 << 24)) return fail(GS_E_RANGE, "blocks must be in 0..2^24");
  if (tiles_per_pass < 1 || tiles_per_pass > 64) return fail(GS_E_RANGE, "tiles_per_pass must be in 1..64");
  e->blocks = blocks;
  e->tpp = tiles_per_pass;
  return GS_OK;
}

int gs_ens_get_launch(const GsEns* e, int* blocks, int* tiles_per_pass, int64_t* total_tiles) {
  using namespace gs;
  if (!e) return fail(GS_E_ARG, "ensemble is NULL");
  if (blocks) {
    int b = e->blocks;
    if (b == 0) b = e->occ * e->cus;
    *blocks = b;
  }
  if (tiles_per_pass) *tiles_per_pass = e->tpp;
  if (total_tiles) *total_tiles = e->ntiles;
  return GS_OK;
}

int gs_ens_step(GsEns* e, void* stream) {
  using namespace gs;
  if (!e) return fail(GS_E_ARG, "ensemble is NULL");
  return ens_step(e, (hipStream_t)stream);
}

int gs_ens_run(GsEns* e, int64_t nsteps, int graph_batch, void* stream) {
  using namespace gs;
  if (!e) return fail(GS_E_ARG, "ensemble is NULL");
  if (nsteps < 0) return fail(GS_E_ARG, "nsteps < 0");
  hipStream_t s = (hipStream_t)stream;
  if (graph_batch <= 0 || nsteps < graph_batch) {
    for (int64_t i = 0; i < nsteps; ++i) {
      const int rc = ens_step(e, s);
      if (rc) return rc;
    }
    return GS_OK;
  }
  if (graph_batch > 100000) return fail(GS_E_RANGE, "graph_batch too large");
  GS_HIP(hipEventRecord(e->ev_in, s), "event record");
  GS_HIP(hipStreamWaitEvent(e->gstream, e->ev_in, 0), "stream wait");
  if (!e->exec || e->g_batch != graph_batch || e->g_blocks != e->blocks || e->g_tpp != e->tpp) {
    const int rc = ens_capture(e, graph_batch);
    if (rc) return rc;
  }
  const int64_t reps = nsteps / graph_batch, rest = nsteps % graph_batch;
  for (int64_t r = 0; r < reps; ++r) GS_HIP(hipGraphLaunch(e->exec, e->gstream), "graph launch");
  for (int64_t i = 0; i < rest; ++i) {
    const int rc = ens_step(e, e->gstream);
    if (rc) return rc;
  }
  GS_HIP(hipEventRecord(e->ev_out, e->gstream), "event record");
  GS_HIP(hipStreamWaitEvent(s, e->ev_out, 0), "stream wait");
  return GS_OK;
}

int gs_ens_autotune(GsEns* e, int trial_steps, void* stream, double* best_ms) {
  using namespace gs;
  if (!e) return fail(GS_E_ARG, "ensemble is NULL");
  if (trial_steps < 1 || trial_steps > 10000) return fail(GS_E_RANGE, "trial_steps must be in 1..10000");
  hipStream_t s = (hipStream_t)stream;
  const size_t es = e->dtype == GS_F64 ? 8 : 4;
  GS_HIP(hipStreamSynchronize(s), "sync");
  // snapshot: the current state buffer, the running max, the Green-Ampt cumulative
  // infiltration and the clock of every member (everything a step writes)
  constexpr int kSnap = 5;
  auto plane = [&](int m, int par, int k) -> void* {
    return k < 3 ? e->flat[m].q[par][k] : (k == 3 ? e->flat[m].max_h : e->flat[m].ga_F);
  };
  std::vector<GsClock> clk((size_t)e->n);
  std::vector<void*> snap;
  int rc = GS_OK;
  auto cleanup = [&]() {
    for (void* p : snap) (void)hipFree(p);
    snap.clear();
  };
  for (int m = 0; m < e->n && rc == GS_OK; ++m) {
    hipError_t h = hipMemcpy(&clk[m], e->clocks[m], sizeof(GsClock), hipMemcpyDeviceToHost);
    if (h != hipSuccess) { rc = hip_fail(h, "clock d2h"); break; }
    const int par = (int)(clk[m].nsteps & 1);
    const size_t bytes = (size_t)e->flat[m].n_stored * es;
    for (int k = 0; k < kSnap && rc == GS_OK; ++k) {
      const void* src = plane(m, par, k);
      void* p = nullptr;
      if (src) {
        h = hipMalloc(&p, bytes);
        if (h == hipSuccess) h = hipMemcpy(p, src, bytes, hipMemcpyDeviceToDevice);
        if (h != hipSuccess) rc = hip_fail(h, "autotune snapshot");
      }
      snap.push_back(p);
    }
  }
  if (rc) { cleanup(); return rc; }
  auto restore = [&]() -> int {
    for (int m = 0; m < e->n; ++m) {
      const int par = (int)(clk[m].nsteps & 1);
      const size_t bytes = (size_t)e->flat[m].n_stored * es;
      for (int k = 0; k < kSnap; ++k) {
        void* dst = plane(m, par, k);
        void* p = snap[(size_t)m * kSnap + k];
        if (dst && p) GS_HIP(hipMemcpyAsync(dst, p, bytes, hipMemcpyDeviceToDevice, s), "restore");
      }
      GS_HIP(hipMemcpyAsync(e->clocks[m], &clk[m], sizeof(GsClock), hipMemcpyHostToDevice, s), "clock restore");
    }
    GS_HIP(hipStreamSynchronize(s), "sync");
    return GS_OK;
  };
  const int occ = e->occ;
  // resident grids of 1, 2, occ/2 and occ workgroups per CU, and (last) one wavefront per
  // tile, which the launch reaches by capping a larger grid at the tiles' need
  int per_cu[5] = {1, 2, occ > 1 ? occ / 2 : 1, occ, 0};
  const int64_t per_tile = (e->ntiles + 3) / 4;
  const int tpps[2] = {1, 2};
  hipEvent_t t0 = nullptr, t1 = nullptr;
  (void)hipEventCreate(&t0);
  (void)hipEventCreate(&t1);
  double best = 1e300;
  int best_b = e->blocks, best_c = e->tpp;
  for (int a = 0; a < 5 && rc == GS_OK; ++a) {
    bool dup = false;
    for (int b = 0; b < a; ++b) dup = dup || per_cu[b] == per_cu[a];
    if (a < 4 && (dup || per_cu[a] > occ)) continue;
    if (a == 4 && per_tile <= (int64_t)occ * e->cus) continue;   // already a resident grid
    for (int c = 0; c < 2 && rc == GS_OK; ++c) {
      if (a == 4 && c > 0) continue;
      e->blocks = a < 4 ? per_cu[a] * e->cus : (int)(per_tile < 0x7fffffff ? per_tile : 0x7fffffff);
      e->tpp = tpps[c];
      rc = restore();
      if (!rc) rc = ens_step(e, s);   // warm-up
      if (!rc && hipEventRecord(t0, s) != hipSuccess) rc = fail(GS_E_STATE, "event record failed");
      for (int i = 0; i < trial_steps && !rc; ++i) rc = ens_step(e, s);
      if (!rc && hipEventRecord(t1, s) != hipSuccess) rc = fail(GS_E_STATE, "event record failed");
      if (!rc && hipEventSynchronize(t1) != hipSuccess) rc = fail(GS_E_STATE, "event sync failed");
      float ms = 0.0f;
      if (!rc && hipEventElapsedTime(&ms, t0, t1) == hipSuccess && ms / trial_steps < best) {
        best = ms / trial_steps;
        best_b = e->blocks;
        best_c = e->tpp;
      }
    }
  }
  (void)hipEventDestroy(t0);
  (void)hipEventDestroy(t1);
  e->blocks = best_b;
  e->tpp = best_c;
  const int rc2 = restore();
  cleanup();
  if (rc) return rc;
  if (rc2) return rc2;
  if (best_ms) *best_ms = best;
  return GS_OK;
}


}  // extern "C"

// ---------------------------------------------------------------------------
// the ensemble run with no allocation
// ---------------------------------------------------------------------------
// The device memory k_ens_step needs beyond the members' own buffers (the last-workgroup
// counter, the tile prefix and the member views) for gs_ens_run_noalloc, which allocates
// nothing: layout [counter, 256 B][tile prefix (n + 1) x int64, padded to 256 B][views].
// Every device holds its own copy at its own address (looked up per device); host code uses
// that address, never the array's name.
constexpr size_t kScratchBytes = 256 * 1024;
static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace gs {

constexpr int kScratchDevices = 64;
static std::mutex g_scratch_mu;                    // guards the table and the host staging copy
static void* g_scratch_dev[kScratchDevices];       // scratch's address on each device
alignas(256) static unsigned char g_scratch_host[kScratchBytes];   // what a call copies into scratch

// The address of `scratch` on the current device; the caller holds g_scratch_mu.
static int scratch_addr(void** out) {
  int dev = 0;
  GS_HIP(hipGetDevice(&dev), "hipGetDevice");
  if (dev < 0 || dev >= kScratchDevices) return fail(GS_E_RANGE, "device %d: the scratch table covers %d devices", dev,
                                                     kScratchDevices);
  if (!g_scratch_dev[dev]) {
    void* p = nullptr;
    GS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "hipGetSymbolAddress(scratch)");
    if (!p) return fail(GS_E_STATE, "hipGetSymbolAddress(scratch) returned NULL");
    g_scratch_dev[dev] = p;
  }
  *out = g_scratch_dev[dev];
  return GS_OK;
}

constexpr size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

// Bytes of scratch the no-allocation run needs for n members (0 if they do not fit).
template <typename T>
static constexpr size_t noalloc_bytes(int n) {
  const size_t need = align256(256 + 8 * ((size_t)n + 1)) + sizeof(FlatK<T>) * (size_t)n;
  return need <= kScratchBytes ? need : 0;
}
static_assert(noalloc_bytes<float>(409) && noalloc_bytes<double>(384), "the members that the ABI promises");

template <typename T>
static int ens_run_noalloc_t(const GsFlat* members, const GsPhys* phys, const GsForcing* forcings,
                             GsClock* const* clocks, int n, int64_t nsteps, hipStream_t s) {
  const size_t need = noalloc_bytes<T>(n);
  if (!need) {
    int cap = 0;
    while (noalloc_bytes<T>(cap + 1)) ++cap;
    return fail(GS_E_RANGE, "gs_ens_run_noalloc: %d members exceed the %zu-byte scratch (at most %d members of "
                "this dtype)", n, kScratchBytes, cap);
  }
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  void* base = nullptr;
  int rc = scratch_addr(&base);
  if (rc) return rc;
  const size_t off_tile = 256, off_views = align256(256 + 8 * ((size_t)n + 1));
  memset(g_scratch_host, 0, off_views);            // the counter starts at zero
  int64_t* c0 = (int64_t*)(g_scratch_host + off_tile);
  FlatK<T>* views = (FlatK<T>*)(g_scratch_host + off_views);
  c0[0] = 0;
  for (int m = 0; m < n; ++m) {
    new (&views[m]) FlatK<T>();
    rc = ens_member_view<T>(members, phys, forcings, clocks, m, views[m]);
    if (rc) return rc;
    c0[m + 1] = c0[m] + views[m].n_tiles;
  }
  const int kind = ens_kind<T>(views, n);
  // steps of an earlier call on this stream may still read the scratch: let them finish
  // before it is overwritten (a synchronous copy, so the host staging is free on return)
  GS_HIP(hipStreamSynchronize(s), "hipStreamSynchronize");
  GS_HIP(hipMemcpy(base, g_scratch_host, need, hipMemcpyHostToDevice), "scratch h2d");
  EnsK<T> k;
  k.mem = (const FlatK<T>*)((unsigned char*)base + off_views);
  k.tile0 = (const int64_t*)((unsigned char*)base + off_tile);
  k.n_members = n;
  k.tpp = 1;
  k.ntiles = c0[n];
  k.done = (unsigned*)base;
  const int64_t blocks = (k.ntiles + 3) / 4 > 0 ? (k.ntiles + 3) / 4 : 1;   // one wavefront per tile
  for (int64_t i = 0; i < nsteps; ++i) {
    ens_launch_kind<T>(kind, blocks, s, k);
    GS_HIP(hipGetLastError(), "k_ens_step launch");
  }
  return GS_OK;
}

}  // namespace gs

extern "C" {

int gs_ens_run_noalloc(const GsFlat* members, const GsPhys* phys, const GsForcing* forcings, GsClock* const* clocks,
                       int n_members, int64_t nsteps, void* stream) {
  using namespace gs;
  if (n_members < 1) return fail(GS_E_RANGE, "gs_ens_run_noalloc: n_members must be >= 1");
  if (!members || !phys || !forcings || !clocks) return fail(GS_E_ARG, "gs_ens_run_noalloc: member arrays are NULL");
  if (nsteps < 0) return fail(GS_E_ARG, "gs_ens_run_noalloc: nsteps < 0");
  const int dt = members[0].dtype;
  if (dt != GS_F32 && dt != GS_F64) return fail(GS_E_DTYPE, "unsupported dtype %d", dt);
  for (int m = 0; m < n_members; ++m) {
    if (members[m].dtype != dt) return fail(GS_E_DTYPE, "member %d dtype differs from member 0", m);
    if (!clocks[m]) return fail(GS_E_ARG, "clock of member %d is NULL", m);
  }
  hipStream_t s = (hipStream_t)stream;
  return dt == GS_F64 ? ens_run_noalloc_t<double>(members, phys, forcings, clocks, n_members, nsteps, s)
                      : ens_run_noalloc_t<float>(members, phys, forcings, clocks, n_members, nsteps, s);
}

}  // extern "C"
