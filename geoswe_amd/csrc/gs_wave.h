// gs_wave.h -- the step arithmetic of gs_device.h for a whole wavefront at a time: the same
// IEEE results bit for bit, in far fewer issue cycles.
//
// The sweeps are bound by VALU issue, not by memory, and the instructions do not cost the
// same. Measured on MI355X (one instruction kind at a time, eight chains per lane, eight
// wavefronts per SIMD), in cycles of a SIMD per wave-instruction: 2.4 for add, mul and fma on
// vector registers and literals; 4.3 for min, max, med3, compare, select, div_scale, div_fmas,
// div_fixup and for any of the former with a scalar-register operand; 8.3 for rcp, rsq, sqrt.
// So the row below
//   * takes quotients as rcp + fma without the scaling and fix-up instructions (20 cycles
//     against 36), one reciprocal for all quotients of a denominator, and roots from one rsq
//     and four fast instructions (18 against 35);
//   * decides per wavefront, with scalar branches on lane masks, what the scalar code decides
//     per lane: dry cells, dry faces, one-sided fluxes and gated faces cost selects only in
//     wavefronts that hold one;
//   * folds the reconstruction's nested min and max into max3 (rounding is monotonic, so
//     max(RN(a - c), RN(b - c)) = RN(max(a, b) - c));
//   * keeps the scalars of the physics in vector registers.
// The short quotients and roots need operands away from the ends of the exponent range. That is
// ensured by one test per row (`sane`: |u| + |v| + (|b| + |h|)/1024 < 1024), which bounds
// everything the faces form, and by the dry test that the flux makes in any case; the bounds
// are derived where they are used. Operands outside them are collected in a mask (`odd`); a
// wavefront that finds one gives the row, before it writes anything of it, to the general
// functions of gs_device.h, so every input, non-finite ones included, has the same result as
// there.
//
// Every function here must be called by all 64 lanes of a wavefront with uniform control flow.
// The host build (one lane, masks are bools) serves the CPU comparison with gs_device.h.
#pragma once

#include <type_traits>

#include "gs_device.h"

// device buffers are global memory: an explicit address space gives global (not generic) accesses
#if defined(__HIPCC__)
#define GS_G __attribute__((address_space(1)))
#else
#define GS_G
#endif

namespace gs {

// ---------------------------------------------------------------------------
// lane masks: one bit per lane in a scalar register pair on the device
// ---------------------------------------------------------------------------
#if defined(__HIP_DEVICE_COMPILE__)
typedef uint64_t lmask;
// predicates of the compare builtins (ordered unless noted)
enum { kGT = 2, kGE = 3, kLT = 4, kLE = 5, kORD = 7 };
__device__ __forceinline__ lmask lm_gt(float a, float b) { return __builtin_amdgcn_fcmpf(a, b, kGT); }
__device__ __forceinline__ lmask lm_ge(float a, float b) { return __builtin_amdgcn_fcmpf(a, b, kGE); }
__device__ __forceinline__ lmask lm_lt(float a, float b) { return __builtin_amdgcn_fcmpf(a, b, kLT); }
__device__ __forceinline__ lmask lm_le(float a, float b) { return __builtin_amdgcn_fcmpf(a, b, kLE); }
__device__ __forceinline__ lmask lm_gt(double a, double b) { return __builtin_amdgcn_fcmp(a, b, kGT); }
__device__ __forceinline__ lmask lm_ge(double a, double b) { return __builtin_amdgcn_fcmp(a, b, kGE); }
__device__ __forceinline__ lmask lm_lt(double a, double b) { return __builtin_amdgcn_fcmp(a, b, kLT); }
__device__ __forceinline__ lmask lm_le(double a, double b) { return __builtin_amdgcn_fcmp(a, b, kLE); }
// neither is NaN
__device__ __forceinline__ lmask lm_ord(float a, float b) { return __builtin_amdgcn_fcmpf(a, b, kORD); }
__device__ __forceinline__ lmask lm_ord(double a, double b) { return __builtin_amdgcn_fcmp(a, b, kORD); }
__device__ __forceinline__ lmask lm_of(bool c) { return __ballot(c); }
__device__ __forceinline__ lmask lm_none() { return 0ull; }
__device__ __forceinline__ lmask lm_every() { return ~0ull; }
__device__ __forceinline__ lmask lm_not(lmask m) { return ~m; }
__device__ __forceinline__ bool lm_any(lmask m) { return m != 0ull; }
__device__ __forceinline__ bool lm_lane(lmask m) { return __builtin_amdgcn_inverse_ballot_w64(m); }
// Neighbour-lane values for the y-faces (lane l receives lane l+1's or lane l-1's value; what
// the end lanes receive is not used) by the LDS crossbar, beside the VALU work of the faces, with
// the source lanes' byte addresses kept in two registers.
struct Lanes {
  int up, dn;
};
__device__ __forceinline__ Lanes lanes_of(int lane) { return {((lane + 1) & 63) * 4, ((lane - 1) & 63) * 4}; }
__device__ __forceinline__ float lane_get(int at, float x) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(at, __float_as_int(x)));
}
__device__ __forceinline__ double lane_get(int at, double x) {
  const uint64_t b = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)(uint32_t)b);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)(uint32_t)(b >> 32));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// A row's start as a value of its own: an access then adds its 32-bit lane offset to a scalar
// base. Left to itself the compiler hoists (plane + lane offset) into vector registers and adds
// the row to it with a 64-bit vector add per access.
template <typename P>
__device__ __forceinline__ GS_G P* row_base(P* p) {
  GS_G P* q = (GS_G P*)p;
  __asm__("" : "+s"(q));
  return q;
}
// One row of a tile through a buffer that starts at the tile: a lane at offset kNoLane stores
// nothing and loads 0, by the bounds check of the buffer. There is no branch around the access, so
// that the wait for the next row's loads, which are older than this row's stores, need not count on
// the stores having been made.
constexpr uint32_t kNoLane = 0xFFFFFFF0u;
typedef __amdgpu_buffer_rsrc_t RowBuf;
template <typename P>
__device__ __forceinline__ RowBuf row_buf(P* p) {
  const uint64_t a = (uint64_t)p;   // uniform; made so for the compiler too
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)a), hi = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), 0, 0x80000000, 0x00020000);
}
__device__ __forceinline__ void row_store(RowBuf r, uint32_t lane_off, uint32_t row_off, float v) {
  __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, lane_off, row_off, 0);
}
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ void row_store(RowBuf r, uint32_t lane_off, uint32_t row_off, double v) {
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, v), r, lane_off, row_off, 0);
}
__device__ __forceinline__ void row_load(RowBuf r, uint32_t lane_off, uint32_t row_off, float& v) {
  v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, lane_off, row_off, 0));
}
__device__ __forceinline__ void row_load(RowBuf r, uint32_t lane_off, uint32_t row_off, double& v) {
  v = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, lane_off, row_off, 0));
}
__device__ __forceinline__ void row_load(RowBuf r, uint32_t lane_off, uint32_t row_off, uint8_t& v) {
  v = __builtin_amdgcn_raw_buffer_load_b8(r, lane_off, row_off, 0);
}
// Four loaded values moved out of the registers they were loaded into, before the loads of the
// next row into those registers: the wait that this implies is for loads a row old, where the
// copies that the compiler makes otherwise wait for the loads just issued.
__device__ __forceinline__ void take_loaded(float& a, float& b, float& c, float& d) {
  float w, x, y, z;
  __asm__ volatile("v_mov_b32 %0, %4\n\tv_mov_b32 %1, %5\n\tv_mov_b32 %2, %6\n\tv_mov_b32 %3, %7"
                   : "=&v"(w), "=&v"(x), "=&v"(y), "=&v"(z) : "v"(a), "v"(b), "v"(c), "v"(d) : "memory");
  a = w;
  b = x;
  c = y;
  d = z;
}
__device__ __forceinline__ void take_loaded(double& a, double& b, double& c, double& d) {
  __asm__ volatile("" : "+v"(a), "+v"(b), "+v"(c), "+v"(d)::"memory");
}
// the mask of each lane's upper neighbour (lane l gets bit l + 1; the top lane's is not used)
__device__ __forceinline__ lmask lm_upper(lmask m) { return m >> 1; }
// A uniform value in scalar registers.
__device__ __forceinline__ float sreg(float x) { return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x))); }
__device__ __forceinline__ double sreg(double x) {
  const uint64_t b = (uint64_t)__double_as_longlong(x);
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)b), hi = __builtin_amdgcn_readfirstlane((uint32_t)(b >> 32));
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// The value itself, for a rare branch: what is computed from it is not moved out of the row loop,
// where it would hold a register.
__device__ __forceinline__ float here(float x) {
  asm volatile("" : "+v"(x));
  return x;
}
__device__ __forceinline__ double here(double x) {
  asm volatile("" : "+v"(x));
  return x;
}
// A uniform value in a vector register: fast instructions that read a scalar register run at half
// rate.
__device__ __forceinline__ float vreg(float x) {
  float y;
  __asm__("v_mov_b32 %0, %1" : "=v"(y) : "s"(x));
  return y;
}
__device__ __forceinline__ double vreg(double x) { return x; }
// min and max without the quieting instruction per operand that the builtins carry for values
// from another basic block (no signalling NaN is of interest here)
__device__ __forceinline__ float min_w(float a, float b) {
  float r;
  __asm__("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float max_w(float a, float b) {
  float r;
  __asm__("v_max_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float min_abs_w(float a, float b) {
  float r;
  __asm__("v_min_f32 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float max_abs_w(float a, float b) {
  float r;
  __asm__("v_max_f32 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ float pos_w(float a) {   // max(a, 0)
  float r;
  __asm__("v_max_f32 %0, 0, %1" : "=v"(r) : "v"(a));
  return r;
}
__device__ __forceinline__ float pos_neg_w(float a, float b) {   // max(-a, b, 0)
  float r;
  __asm__("v_max3_f32 %0, -%1, %2, 0" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double min_w(double a, double b) {
  double r;
  __asm__("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double max_w(double a, double b) {
  double r;
  __asm__("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double min_abs_w(double a, double b) {
  double r;
  __asm__("v_min_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double max_abs_w(double a, double b) {
  double r;
  __asm__("v_max_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(a), "v"(b));
  return r;
}
__device__ __forceinline__ double pos_w(double a) {
  double r;
  __asm__("v_max_f64 %0, 0, %1" : "=v"(r) : "v"(a));
  return r;
}
__device__ __forceinline__ double pos_neg_w(double a, double b) {
  return pos_w(max_w(-a, b));
}
__device__ __forceinline__ float rcp_approx(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double rcp_approx(double x) { return __builtin_amdgcn_rcp(x); }
__device__ __forceinline__ float rsq_approx(float x) { return __builtin_amdgcn_rsqf(x); }
__device__ __forceinline__ double rsq_approx(double x) { return __builtin_amdgcn_rsq(x); }
#else
typedef bool lmask;
GS_HD lmask lm_of(bool c) { return c; }
template <typename T> GS_HD lmask lm_gt(T a, T b) { return a > b; }
template <typename T> GS_HD lmask lm_ge(T a, T b) { return a >= b; }
template <typename T> GS_HD lmask lm_lt(T a, T b) { return a < b; }
template <typename T> GS_HD lmask lm_le(T a, T b) { return a <= b; }
template <typename T> GS_HD lmask lm_ord(T a, T b) { return a == a && b == b; }
GS_HD lmask lm_none() { return false; }
GS_HD lmask lm_every() { return true; }
GS_HD lmask lm_not(lmask m) { return !m; }
GS_HD bool lm_any(lmask m) { return m; }
GS_HD bool lm_lane(lmask m) { return m; }
GS_HD lmask lm_upper(lmask m) { return m; }
struct Lanes {
  int up, dn;
};
GS_HD Lanes lanes_of(int) { return {0, 0}; }
template <typename T> GS_HD T lane_get(int, T x) { return x; }
template <typename P> GS_HD GS_G P* row_base(P* p) { return (GS_G P*)p; }
typedef void* RowBuf;
constexpr uint32_t kNoLane = 0xFFFFFFF0u;
template <typename P> GS_HD RowBuf row_buf(P* p) { return (void*)p; }
template <typename T> GS_HD void row_store(RowBuf, uint32_t, uint32_t, T) {}
template <typename T> GS_HD void row_load(RowBuf, uint32_t, uint32_t, T&) {}
template <typename T> GS_HD void take_loaded(T&, T&, T&, T&) {}
template <typename T> GS_HD T vreg(T x) { return x; }
template <typename T> GS_HD T sreg(T x) { return x; }
template <typename T> GS_HD T here(T x) { return x; }
template <typename T> GS_HD T min_w(T a, T b) { return vmin(a, b); }
template <typename T> GS_HD T max_w(T a, T b) { return vmax(a, b); }
template <typename T> GS_HD T min_abs_w(T a, T b) { return vmin(vabs(a), vabs(b)); }
template <typename T> GS_HD T max_abs_w(T a, T b) { return vmax(vabs(a), vabs(b)); }
template <typename T> GS_HD T pos_w(T a) { return a > T(0) ? a : T(0); }
template <typename T> GS_HD T pos_neg_w(T a, T b) { return pos_w(vmax(-a, b)); }
// the CPU comparison may put any value within the hardware's error here
#ifndef GS_HOST_RCP
#define GS_HOST_RCP(x) (decltype(x)(1) / (x))
#define GS_HOST_RSQ(x) (decltype(x)(1) / vsqrt(x))
#endif
template <typename T> GS_HD T rcp_approx(T x) { return GS_HOST_RCP(x); }
template <typename T> GS_HD T rsq_approx(T x) { return GS_HOST_RSQ(x); }
#endif

template <typename T> GS_HD T lm_sel(lmask m, T a, T b) { return lm_lane(m) ? a : b; }

GS_HD float vfma(float a, float b, float c) { return fmaf(a, b, c); }
GS_HD double vfma(double a, double b, double c) { return fma(a, b, c); }

// ---------------------------------------------------------------------------
// quotients and roots away from the ends of the exponent range
// ---------------------------------------------------------------------------
// 1/b. float32: one Newton step on v_rcp_f32, correctly rounded (gs_crmath.h). float64: the two
// steps of the compiler's own division, RN(1/b) but for a few b beside a midpoint.
GS_HD float recip_w(float b) { return cr_recip_refine(b, rcp_approx(b)); }
GS_HD double recip_w(double b) {
  double y = rcp_approx(b);
  y = vfma(vfma(-b, y, 1.0), y, y);
  return vfma(vfma(-b, y, 1.0), y, y);
}
// RN(a/b) with y = recip_w(b), for a = +-0 or |a| large enough that a - b*q is exact and the
// quotient normal (Markstein; the remainder is formed negated so that a = -0 gives -0 for b > 0;
// over a negative denominator a zero's sign is not kept).
template <typename T>
GS_HD T quot_w(T a, T b, T y) {
  const T q = a * y;
  return vfma(-vfma(b, q, -a), y, q);
}
// RN(a/d) for a = 1 or 2 and d >= 1. The float64 reciprocal is not RN(1/d) for every d (not, on the
// device, for 0.15 % of the significands within 2^12 ulps below 2), so it takes the quotient's
// correction, as the division of the general functions does.
GS_HD float unit_quot_w(float a, float d) { return a * recip_w(d); }
GS_HD double unit_quot_w(double a, double d) { return quot_w(a, d, recip_w(d)); }
// RN(sqrt(x)) from y = v_rsq_f32(x): s = x*y, then one correction by the exact remainder
// (x - s*s)*(y/2). Over every float32 x >= 2^-96 the device result equals the general root's
// (the crmath check's third test). float64: the compiler's own sequence without its scaling.
GS_HD float root_from_rsq(float x, float y) {
  const float s = x * y;
  return vfma(vfma(-s, s, x), 0.5f * y, s);
}
GS_HD double root_from_rsq(double x, double y) {
  double s = x * y, h = 0.5 * y;
  const double e = vfma(-h, s, 0.5);
  s = vfma(s, e, s);
  h = vfma(h, e, h);
  s = vfma(vfma(-s, s, x), h, s);
  return vfma(vfma(-s, s, x), h, s);
}
template <typename T> GS_HD T root_w(T x) { return root_from_rsq(x, rsq_approx(x)); }
// x below `root` takes the general root (0 excepted); numerators below `num_tiny` the general
// quotient, where a remainder could be inexact; quotients of operands in [lo, hi] are safe
template <typename T> struct Range;
template <> struct Range<float> {
  GS_HD static float root() { return 0x1p-96f; }
  GS_HD static float num_tiny() { return 0x1p-80f; }
  GS_HD static float lo() { return 0x1p-60f; }
  GS_HD static float hi() { return 0x1p60f; }
};
template <> struct Range<double> {
  GS_HD static double root() { return 0x1p-700; }
  GS_HD static double num_tiny() { return 0x1p-700; }
  GS_HD static double lo() { return 0x1p-400; }
  GS_HD static double hi() { return 0x1p400; }
};
// RN(sqrt(x)) with sqrt(0) = 0 (x >= 0, not in (0, root()))
template <typename T>
GS_HD T root0_w(T x) {
  return root_from_rsq(x, rsq_approx(max_w(x, Range<T>::root())));
}

#if defined(__HIPCC__)
// Element at byte offset `off` of a row that starts at `row` (uniform): the row's address stays
// in scalar registers and the lane adds a 32-bit offset, so an access costs no vector address
// arithmetic. O is uint32_t unless a row spans 4 GiB or more.
template <typename P, typename O>
__device__ __forceinline__ GS_G P& row_at(GS_G P* row, O off) {
  // a value of its own, widened beside the access: a widening hoisted out of the row loop would
  // make the lane's address a 64-bit vector add
  if (sizeof(O) == 4) __asm__("" : "+v"(off));
  typedef typename std::conditional<std::is_const<P>::value, const char, char>::type B;
  return *(GS_G P*)((GS_G B*)row + off);
}
#endif

// ---------------------------------------------------------------------------
// the uniform scalars of a row
// ---------------------------------------------------------------------------
template <typename T>
struct WaveC {
  T g, hg, hm, ix, iy, hdx, hdy, dt, vcap;
  int flags;       // kWave*
  lmask not_wet;   // all lanes unless kWaveWet is set
};

// What the host finds of the physics scalars (wave_flags), for every row of a launch:
enum {
  // the short forms may be used at all: g <= 16, h_min in [floor, 1] and a cell size within 2^+-40;
  // a sane row then has velocities below 2^10, depths and beds below 2^20, celerities below 2^12
  // and every product of a face below 2^100
  kWaveFast = 1,
  // h_min >= 2^-21 and g*h_min >= 2^-20, so that a wet face's celerities are at least 2^-10
  kWaveWet = 2,
  // the L-inf wave speed with a CFL floor that the division does not see (lam_key_w)
  kWaveLam = 4,
};
inline float wave_floor(float) { return 0x1p-21f; }
inline double wave_floor(double) { return 0x1p-36; }
template <typename T>
inline int wave_flags(const Phys<T>& P, bool flat) {
  const double hm = (double)P.h_min, g = (double)P.g, ix = (double)P.inv_dx, iy = (double)P.inv_dy;
  const double lo = (double)wave_floor(T(0));
  if (!(g > 0.0 && g <= 16.0 && hm >= lo && hm <= 1.0 && ix >= 0x1p-40 && ix <= 0x1p40 && iy >= 0x1p-40 &&
        iy <= 0x1p40))
    return 0;
  int f = kWaveFast;
  if (hm >= 0x1p-21 && g * hm >= 0x1p-20) f |= kWaveWet;
  if (g * hm >= (sizeof(T) == 4 ? 0x1p-20 : 0x1p-40) && !P.cfl_l2 && (flat ? P.h_cfl <= P.h_min : P.h_cfl == P.h_min)) f |= kWaveLam;
  return f;
}
template <typename T>
GS_HD WaveC<T> wave_consts(const Phys<T>& P, T dt, int flags) {
  WaveC<T> w;
  w.g = vreg(P.g);
  w.hg = vreg(T(0.5) * P.g);
  w.hm = P.h_min;
  w.ix = vreg(P.inv_dx);
  w.iy = vreg(P.inv_dy);
  w.hdx = vreg(P.half_dx);
  w.hdy = vreg(P.half_dy);
  w.dt = vreg(dt);
  w.vcap = sreg(P.has_vcap ? P.vcap : T(INFINITY));
  w.flags = flags;
  w.not_wet = (flags & kWaveWet) ? lm_none() : lm_every();
  return w;
}

// ---------------------------------------------------------------------------
// primitive velocities of a row, its wet/dry mask and its sanity
// ---------------------------------------------------------------------------
// Lanes where x or y is not 0 but too small for the short quotient.
template <typename T>
GS_HD lmask tiny_num(T x, T y, lmask use) {
  lmask m = (lm_lt(vabs(x), Range<T>::num_tiny()) | lm_lt(vabs(y), Range<T>::num_tiny())) & use;
  if (lm_any(m))   // zeros (still water) are in order
    m = m & lm_of((x != T(0) && vabs(x) < Range<T>::num_tiny()) || (y != T(0) && vabs(y) < Range<T>::num_tiny()));
  return m;
}

// `use`: the lanes whose cells matter (the others may hold anything after this). `dry`: lanes
// with h < h_min. `odd` gathers the lanes that make the row not sane, with the bed `b` of the
// row that was read beside it.
template <typename T>
GS_HD void prims_w(T h, T hu, T hv, T b, lmask use, const WaveC<T>& w, T& u, T& v, lmask& dry, lmask& odd) {
  const lmask wet = lm_gt(h, w.hm);
  dry = lm_none();
  const lmask tiny = tiny_num<T>(hu, hv, use);
  if (!lm_any(lm_not(wet) & use)) {
    const T y = recip_w(h);
    u = quot_w(hu, h, y);
    v = quot_w(hv, h, y);
  } else {
    dry = lm_lt(h, w.hm);
    const T hs = max_w(h, w.hm);
    const T y = recip_w(hs);
    u = lm_sel(wet, quot_w(hu, hs, y), T(0));
    v = lm_sel(wet, quot_w(hv, hs, y), T(0));
  }
  if (lm_any(tiny)) {
    // Momenta that friction has all but stopped: the division itself. Their rows must not go to the
    // general functions: a few hundred of 36 000 window rows of a 2048^2 coastal domain hold one
    // after 200 steps, and with all tiles in one round the slowest tile is the step (50.0 against
    // 42.5 us).
    const lmask wet1 = lm_gt(h, w.hm);
    u = lm_sel(wet1, vdiv(here(hu), max_w(h, w.hm)), T(0));
    v = lm_sel(wet1, vdiv(here(hv), max_w(h, w.hm)), T(0));
  }
  const T s = (vabs(u) + vabs(v)) + (vabs(b) + vabs(h)) * T(0x1p-10);
  odd = odd | (lm_not(lm_lt(s, T(1024))) & use);
}

// ---------------------------------------------------------------------------
// HLLC
// ---------------------------------------------------------------------------
// The star state (or, with S = 0 and a = b = 1, the one-sided flux) of the side chosen.
template <typename T>
GS_HD void hllc_flux_w(T S, T SM, T uN, T uT, T hh, T a, T b, const WaveC<T>& w, T& Fh, T& FN, T& FT) {
  const T hs = hh * quot_w(a, b, recip_w(b));
  const T huN = hh * uN;
  const T F_N = huN * uN + (w.hg * hh) * hh;
  Fh = huN + S * (hs - hh);
  FN = F_N + S * (hs * SM - huN);
  FT = huN * uT + S * (hs * uT - hh * uT);
}

// hllc() of gs_device.h for a sane row (hL, hR >= 0 and not NaN); `use`: the lanes whose face
// matters.
//
// All faces wet (both depths above h_min): a = sqrt(g h) >= 2^-10 while |u| < 2^10,
// so u - a differs from u by at least 2^-11; S, S - u and u - S are multiples of 2^-36 where they
// are small; SL < 0 <= SM (or SM < 0 < SR) makes |S - SM| >= 2^-36; the numerator of SM is 0 or
// at least 2^-91 and its denominator, a sum of two terms of one sign, at least 2^-31 (above the
// 1e-14 of the general function), their quotient 0 or at least 2^-103: every quotient and root
// is in range (in float64, whose bounds are finer, all the more).
template <typename T>
GS_HD void hllc_w(T hL, T uNL, T uTL, T hR, T uNR, T uTR, lmask use, const WaveC<T>& w, T& Fh, T& FN, T& FT,
                  lmask& odd) {
  const lmask dryL = lm_le(hL, w.hm), dryR = lm_le(hR, w.hm);
  const T xL = w.g * hL, xR = w.g * hR;
  if (!lm_any(((dryL | dryR) & use) | w.not_wet)) {
    const T aL = root_w(xL), aR = root_w(xR);
    const T U = uNL + uNR;
    const T u_st = vfma(T(0.5), U, aL) - aR;
    const T a_st = pos_w(vfma(T(0.5), aL + aR, T(0.25) * (uNL - uNR)));
    const T SL = min_w(uNL - aL, u_st - a_st);
    const T SR = max_w(uNR + aR, u_st + a_st);
    const T p = uNR - SR, m = uNL - SL;
    const T denom = hR * p - hL * m;
    const T SM = quot_w((SL * hR) * p - (SR * hL) * m, denom, recip_w(denom));
    lmask lft = lm_ge(SM, T(0));
    const lmask star = lm_lt(SL * SR, T(0));   // SL <= SR always: SL < 0 < SR
    if (!lm_any(lm_not(star) & use)) {
      const T S = lm_sel(lft, SL, SR), uN = lm_sel(lft, uNL, uNR);
      hllc_flux_w(S, SM, uN, lm_sel(lft, uTL, uTR), lm_sel(lft, hL, hR), S - uN, (S - SM) + T(1.0e-30), w, Fh, FN,
                  FT);
    } else {
      // SL >= 0: the left flux; SR < 0 with SM < 0: the right one; else a star state
      const lmask c1 = lm_ge(SL, T(0)), c3 = lm_ge(SR, T(0));
      const lmask one = c1 | (lm_not(lft) & lm_not(c3));
      lft = lft | c1;
      const T S = lm_sel(lft, SL, SR), uN = lm_sel(lft, uNL, uNR);
      hllc_flux_w(lm_sel(one, T(0), S), SM, uN, lm_sel(lft, uTL, uTR), lm_sel(lft, hL, hR),
                  lm_sel(one, T(1), S - uN), lm_sel(one, T(1), (S - SM) + T(1.0e-30)), w, Fh, FN, FT);
    }
    return;
  }
  // Some lane's face is dry on a side: the same without branches. A depth of exactly 0 keeps the
  // bounds (with hL = 0, SM = SL up to rounding: SL >= 0 is the one-sided flux, SL < 0 the right
  // star state with S - u = SR - uR >= a); a film between 0 and h_min does not, and its operands
  // are tested.
  const T aL = root0_w(xL), aR = root0_w(xR);
  const T U = uNL + uNR;
  const T u_st = vfma(T(0.5), U, aL) - aR;
  const T a_st = pos_w(vfma(T(0.5), aL + aR, T(0.25) * (uNL - uNR)));
  const lmask both = dryL & dryR;
  T SL = lm_sel(dryL, vfma(T(-2), aR, uNR), min_w(uNL - aL, u_st - a_st));
  T SR = lm_sel(dryR, vfma(T(2), aL, uNL), max_w(uNR + aR, u_st + a_st));
  SL = lm_sel(both, T(0), SL);
  SR = lm_sel(both, T(0), SR);
  const T p = uNR - SR, m = uNL - SL;
  const T denom = hR * p - hL * m;
  const T num = (SL * hR) * p - (SR * hL) * m;
  const lmask big = lm_gt(vabs(denom), T(1.0e-14));
  const T SM = lm_sel(big, quot_w(num, denom, recip_w(denom)), T(0.5) * U);
  const lmask c1 = lm_ge(SL, T(0)), c2 = lm_ge(SM, T(0)), c3 = lm_ge(SR, T(0));
  const lmask one = c1 | (lm_not(c2) & lm_not(c3));
  const lmask lft = c1 | c2;
  const T S = lm_sel(lft, SL, SR), uN = lm_sel(lft, uNL, uNR);
  const T a = lm_sel(one, T(1), S - uN), b = lm_sel(one, T(1), (S - SM) + T(1.0e-30));
  const lmask part = ((dryL & lm_gt(hL, T(0))) | (dryR & lm_gt(hR, T(0)))) & use;
  if (lm_any(part | w.not_wet)) {
    const lmask bad = lm_lt(min_abs_w(a, b), Range<T>::lo()) | lm_gt(max_abs_w(a, b), Range<T>::hi()) |
                      lm_of((xL != T(0) && xL < Range<T>::root()) || (xR != T(0) && xR < Range<T>::root()) ||
                            (num != T(0) && vabs(num) < Range<T>::num_tiny()));
    odd = odd | (bad & use);
  }
  hllc_flux_w(lm_sel(one, T(0), S), SM, uN, lm_sel(lft, uTL, uTR), lm_sel(lft, hL, hR), a, b, w, Fh, FN, FT);
}

// ---------------------------------------------------------------------------
// one face per lane, as the products its cells add: flux and sources times inv_d, zero where
// both cells are dry
// ---------------------------------------------------------------------------
template <typename T>
struct FaceProd {
  T Fh, FN, FT, sL, sR;
};

// face() of gs_device.h. zL, zhR: half_d times the bed gradients of L and R. dryL, dryR: lanes
// whose cells have h < h_min. The sign of a zero in a product does not matter: the residual sums
// start at +0 and never hold -0.
template <typename T>
GS_HD void face_w(T bL, T bR, T zL, T zhR, T hL, T hR, T uNL, T uTL, T uNR, T uTR, lmask dryL, lmask dryR, lmask use,
                  T inv, const WaveC<T>& w, FaceProd<T>& f, lmask& odd) {
  const T z = T(0);
  const T db = bR - bL;
  const T zR = db - zhR;
  const T zf0 = pos_w(db);
  const T dzc = zR - zL;
  const T dz = db - dzc;
  const T etaR = hR + db;
  const T D = etaR - hL;
  const T headL = zf0 - hL, headR = zf0 - etaR;
  // detaL = max(0, min(dz, D)) and detaR = max(0, min(-dz, -D)) = max(0, -max(dz, D));
  // max(0, (hL + detaL) - zf0) = max(0, hL - zf0, (hL + min(dz, D)) - zf0)
  const T hLf = pos_neg_w(headL, (hL + min_w(dz, D)) - zf0);
  const T hRf = pos_neg_w(headR, (etaR - max_w(dz, D)) - zf0);
  T cL = dzc, cR = -dzc;
  if (lm_any((dryL | dryR) & use)) {
    // the head alone where the other cell is dry; nothing where both are (every product of a
    // sane row is finite)
    cL = lm_sel(dryR, T(INFINITY), cL);
    cR = lm_sel(dryL, T(INFINITY), cR);
    inv = lm_sel(dryL & dryR, z, inv);
  }
  const T sL = (w.hg * (hLf + hL)) * (zf0 - pos_w(min_w(cL, headL)));
  const T sR = (w.hg * (hRf + hR)) * ((zf0 - pos_w(min_w(cR, headR))) - db);
  T Fh, FN, FT;
  hllc_w(hLf, uNL, uTL, hRf, uNR, uTR, use, w, Fh, FN, FT, odd);
  f.Fh = Fh * inv;
  f.FN = FN * inv;
  f.FT = FT * inv;
  f.sL = sL * inv;
  f.sR = sR * inv;
}

// The four faces of a cell in the reference's order. A face gated off (both cells dry) adds
// zeros: the sums start at +0 and IEEE addition yields -0 only from two -0 terms, so they never
// hold -0, and x + 0 = x - 0 = x for every other x.
template <typename T>
GS_HD void sum_faces(const FaceProd<T>& up, const FaceProd<T>& dn, const FaceProd<T>& right,
                                          T lFh, T lFN, T lFT, T lsR, T& rh, T& rhu, T& rhv) {
  rh = T(0); rhu = T(0); rhv = T(0);
  rh = rh - up.Fh;
  rhu = rhu - up.FN;
  rhv = rhv - up.FT;
  rhu = rhu - up.sL;
  rh = rh + dn.Fh;
  rhu = rhu + dn.FN;
  rhv = rhv + dn.FT;
  rhu = rhu + dn.sR;
  rh = rh - right.Fh;
  rhu = rhu - right.FT;
  rhv = rhv - right.FN;
  rhv = rhv - right.sL;
  rh = rh + lFh;
  rhu = rhu + lFT;
  rhv = rhv + lFN;
  rhv = rhv + lsR;
}

// face() as the products its cells add, zero where it is gated off.
template <typename T>
GS_HD void face_prod(T bL, T bR, T gzL, T gzR, T hL, T hR, T uNL, T uTL, T uNR, T uTR, T half,
                                          T inv, T g, T hm, FaceProd<T>& f) {
  Face<T> q;
  face<T>(bL, bR, gzL, gzR, hL, hR, uNL, uTL, uNR, uTR, half, g, hm, q);
  f.Fh = q.gate ? q.Fh * inv : T(0);
  f.FN = q.gate ? q.FN * inv : T(0);
  f.FT = q.gate ? q.FT * inv : T(0);
  f.sL = q.gate ? q.srcL * inv : T(0);
  f.sR = q.gate ? q.srcR * inv : T(0);
}

template <typename T>
constexpr T kMaxSpeed = T(0x1p40);

// ---------------------------------------------------------------------------
// update
// ---------------------------------------------------------------------------
// update() of gs_device.h for the lanes `act` of a wavefront (the others' results are not used).
// `speed`: max(|hu|, |hv|)/h + sqrt(g h) of every such lane with h >= h_min, 0 of the others.
//
// One test of the final speed stands for the operands: where a depth, a momentum or an
// intermediate is not finite, or too large for a quotient, the speed is not below 2^40 (NaN
// included: the maximum drops one NaN of two, but with friction both momenta are then NaN, by the
// speed that scales them, and without it they are tested). Small momenta need no test: below 2^-100
// their square vanishes beside any square that matters.
template <typename T>
GS_HD void update_w(T q0, T q1, T q2, T rr0, T r1, T r2, T n, lmask act, const Phys<T>& P, const WaveC<T>& w, T& h,
                    T& hu, T& hv, T& speed, lmask& odd) {
  h = q0 + w.dt * rr0;
  hu = q1 + w.dt * r1;
  hv = q2 + w.dt * r2;
  const lmask dry = lm_lt(h, w.hm);
  const lmask live = act & lm_not(dry);
  const T hs = max_w(h, w.hm);
  const T yh = recip_w(hs);
  if (P.friction) {
    const T u = quot_w(hu, hs, yh);
    const T v = quot_w(hv, hs, yh);
    const T m2 = u * u + v * v;
    T modU = root0_w(m2);
    const T h43 = pow_m43(hs);
    // one branch for what few rows hold: velocities below 2^-48, which take the general root (still
    // water, 0, is in order), and those above the cap
    lmask creep = lm_lt(m2, Range<T>::root()) & live;
    if (lm_any(creep | (lm_gt(modU, w.vcap) & live))) {
      creep = creep & lm_gt(m2, T(0));
      if (lm_any(creep)) modU = lm_sel(creep, vsqrt(here(m2)), modU);
      const lmask fastw = lm_gt(modU, w.vcap) & live;
      if (lm_any(fastw)) {
        const T n_cri = vsqrt(vdiv(T(1), (((T(1.0e-10) + here(w.dt)) * P.g) * h43) * (modU + T(1.0e-30))));
        n = lm_sel(fastw & lm_gt(n_cri, n), n_cri, n);
      }
    }
    const T Cf = ((w.g * n) * n) * h43;
    T alpha;
    if (P.quadratic) {
      // alpha = 2 / (sqrt(1 + 2*two) + 1); doubled where (2*dt)*Cf would overflow, so that it does
      // here too
      const T dtCf = w.dt * Cf;
      const T two = (dtCf + dtCf) * modU;
      alpha = unit_quot_w(T(2), root_w(vfma(T(2), two, T(1))) + T(1));
    } else {
      const T d = T(1) + (w.dt * Cf) * modU;
      alpha = unit_quot_w(T(1), d);
      odd = odd | (lm_gt(d, Range<T>::hi()) & live);   // alpha may be subnormal
    }
    hu = hu * alpha;
    hv = hv * alpha;
  } else {
    odd = odd | (lm_not(lm_ord(hu, hv)) & live);
  }
  speed = quot_w(max_abs_w(hu, hv), hs, yh) + root_w(w.g * h);
  odd = odd | (lm_not(lm_lt(speed, kMaxSpeed<T>)) & live);
  if (lm_any(dry & act)) {
    h = lm_sel(dry, P.keep_h ? pos_w(h) : T(0), h);
    hu = lm_sel(dry, T(0), hu);
    hv = lm_sel(dry, T(0), hv);
    speed = lm_sel(dry, T(0), speed);
  }
}

// The wave speed of a state that the update did not make (a stage, a forcing): the same expression.
// Not below kMaxSpeed on a wet lane: one that this form does not serve (a NaN momentum beside a
// finite one among them, which the maximum alone would drop).
template <typename T>
GS_HD T speed_w(T h, T hu, T hv, const WaveC<T>& w) {
  const T hs = max_w(h, w.hm);
  const T speed = quot_w(max_abs_w(hu, hv), hs, recip_w(hs)) + root_w(w.g * h);
  return lm_sel(lm_lt(h, w.hm), T(0), lm_sel(lm_ord(hu, hv), speed, T(INFINITY)));
}

#if defined(__HIPCC__)
// lam_key() of gs_device.h from update_w's speed, for a row that nothing changed since and where
// kWaveLam is set. A velocity too small for an exact quotient vanishes beside the celerity.
template <typename T>
__device__ __forceinline__ lam_t<T> lam_key_w(T speed) {
  if constexpr (sizeof(T) == 4) return (lam_t<T>)__float_as_uint((float)speed);
  else return (lam_t<T>)__double_as_longlong((double)speed);
}
#endif

}  // namespace gs
