// CPU comparison of the wavefront forms of the step arithmetic (gs_wave.h, built for one lane)
// with the general functions (gs_device.h): wherever the wavefront forms do not report an operand
// outside their bounds, every result has the general function's value. The hardware reciprocal and
// reciprocal root are replaced by the correctly rounded values moved by -1, 0 or +1 ulp (0 for the
// root, whose one correction is checked against the hardware on the GPU). Test infrastructure only.
#include <math.h>
#include <stdint.h>
#include <stdio.h>
#include <string.h>

static uint64_t g_state = 88172645463325252ull;
static uint64_t rnd() {
  g_state ^= g_state << 13;
  g_state ^= g_state >> 7;
  g_state ^= g_state << 17;
  return g_state;
}
static double uni(double a, double b) { return a + (b - a) * (double)(rnd() >> 11) * 0x1p-53; }

static float host_rcp(float x) {
  const float y = 1.0f / x;
  if (!(fabsf(y) < 1e30f) || y == 0.0f) return y;
  const int k = (int)(rnd() % 3) - 1;
  const float z = k == 0 ? y : nextafterf(y, k > 0 ? INFINITY : -INFINITY);
  const double ulp = fabs((double)nextafterf(y, INFINITY) - (double)y);
  // within 1 ulp of 1/x; and not the one such pair that the refinement does not round correctly,
  // which the hardware does not produce (the GPU's check of every reciprocal)
  const bool ones = (__builtin_bit_cast(uint32_t, x) & 0x7FFFFFu) == 0x7FFFFFu;
  return !ones && fabs((double)z - 1.0 / (double)x) <= ulp ? z : y;
}
// float64 approximations of 24 bits, as the hardware's
static double bits24(double y) {
  int e;
  if (!isfinite(y)) return y;
  const double m = frexp(y, &e);
  return ldexp((double)(float)m, e);
}
static double host_rcp(double x) { return bits24(1.0 / x); }
static float host_rsq(float x) { return (float)(1.0 / sqrt((double)x)); }
static double host_rsq(double x) { return bits24(1.0 / sqrt(x)); }
#define GS_HOST_RCP(x) host_rcp(x)
#define GS_HOST_RSQ(x) host_rsq(x)

#include "../../geoswe_amd/csrc/gs_wave.h"

using namespace gs;

static long g_bad = 0;
template <typename T>
static void same(const char* what, T a, T b) {
  if (a == b || (a != a && b != b)) return;
  if (++g_bad <= 10) printf("MISMATCH float%d %s: %.17g against %.17g\n", (int)sizeof(T) * 8, what, (double)a, (double)b);
}

// a value of a kind: ordinary, tiny, huge or not finite
template <typename T>
static T special() {
  const bool f = sizeof(T) == 4;
  const double v[] = {0.0, -0.0, f ? 1e-45 : 5e-324, f ? 1e-38 : 1e-308, f ? 1e-30 : 1e-200, 1e-24, 1e-16, 1e-12,
                      1e-6, 1e-7, 1e-5, 1.0, 1e3, 1e4, 1e7, 1e12, f ? 1e30 : 1e200, f ? 3e38 : 1e308, INFINITY, NAN};
  const double s = v[rnd() % (sizeof v / sizeof v[0])];
  return (T)((rnd() & 1) ? s : -s);
}

template <typename T>
static Phys<T> phys(T hm, int quad) {
  Phys<T> P;
  memset(&P, 0, sizeof P);
  P.g = T(9.81);
  P.h_min = hm;
  P.h_cfl = hm;
  P.vcap = T(15);
  P.inv_dx = T(1) / T(3);
  P.inv_dy = T(1) / T(2.5);
  P.half_dx = T(0.5) * (T(1) / P.inv_dx);
  P.half_dy = T(0.5) * (T(1) / P.inv_dy);
  P.friction = 1;
  P.quadratic = quad;
  P.keep_h = 1;
  P.has_vcap = 1;
  return P;
}

struct Count {
  long n = 0, odd = 0;
};

// regime: 0 wet, 1 films and dry cells on rough beds, 2 fast flow, 3 still water, 4 special values
template <typename T>
static T depth(int r) {
  switch (r) {
    case 0: return (T)uni(0.05, 5.0);
    case 1: return rnd() % 4 == 0 ? T(0) : (T)pow(10.0, uni(-9, 0));
    case 2: return (T)uni(1e-4, 10.0);
    case 3: return (T)uni(0.1, 2.0);
    default: return rnd() % 2 ? special<T>() : (T)uni(0.0, 2.0);
  }
}
template <typename T>
static T momentum(int r, T h) {
  switch (r) {
    case 0: return (T)(h * uni(-2, 2));
    case 1: return h > T(0) ? (T)(h * uni(-1, 1) * pow(10.0, uni(-4, 0))) : T(0);
    case 2: return (T)(h * uni(-40, 40));
    case 3: return T(0);
    default: return rnd() % 2 ? special<T>() : (T)uni(-2.0, 2.0);
  }
}

template <typename T>
static void run(int regime, T hm, long n, Count& faces, Count& updates) {
  for (long k = 0; k < n; ++k) {
    const Phys<T> P = phys<T>(hm, (int)(rnd() & 1));
    const T dt = (T)uni(1e-3, 2.0);
    const WaveC<T> w = wave_consts<T>(P, dt, wave_flags<T>(P, false));
    T h[2], hu[2], hv[2], u[2], v[2], gu, gv, b[4];
    lmask dry[2], odd = false;
    for (int i = 0; i < 4; ++i) b[i] = regime == 4 && rnd() % 8 == 0 ? special<T>() : (T)uni(-1.0, regime == 1 ? 3.0 : -0.5);
    for (int i = 0; i < 2; ++i) {
      h[i] = depth<T>(regime);
      hu[i] = momentum<T>(regime, h[i]);
      hv[i] = momentum<T>(regime, h[i]);
      prims_w<T>(h[i], hu[i], hv[i], vabs(b[i]) + vabs(b[i + 2]), true, w, u[i], v[i], dry[i], odd);
      prims(h[i], hu[i], hv[i], hm, gu, gv);
      if (!odd) {
        same("u", u[i], gu);
        same("v", v[i], gv);
      }
      u[i] = gu;
      v[i] = gv;
    }
    // bed gradients of the two cells, and the face
    const T gz0 = (T(0.5) * (b[1] - b[2])) * P.inv_dx, gz1 = (T(0.5) * (b[3] - b[0])) * P.inv_dx;
    FaceProd<T> f;
    Face<T> q;
    face_w<T>(b[0], b[1], P.half_dx * gz0, P.half_dx * gz1, h[0], h[1], u[0], v[0], u[1], v[1], dry[0], dry[1], true,
              w.ix, w, f, odd);
    face<T>(b[0], b[1], gz0, gz1, h[0], h[1], u[0], v[0], u[1], v[1], P.half_dx, P.g, hm, q);
    faces.n++;
    faces.odd += odd;
    if (!odd) {
      same("Fh", f.Fh, q.gate ? q.Fh * P.inv_dx : T(0));
      same("FN", f.FN, q.gate ? q.FN * P.inv_dx : T(0));
      same("FT", f.FT, q.gate ? q.FT * P.inv_dx : T(0));
      same("sL", f.sL, q.gate ? q.srcL * P.inv_dx : T(0));
      same("sR", f.sR, q.gate ? q.srcR * P.inv_dx : T(0));
    }
    // the update from a residual of the regime's size
    const T r0 = regime == 4 ? special<T>() : (T)(uni(-0.2, 0.2) * h[0]);
    const T r1 = regime == 3 ? T(0) : (regime == 4 ? special<T>() : (T)(uni(-1, 1) * h[0]));
    const T r2 = regime == 3 ? T(0) : (T)(uni(-1, 1) * pow(10.0, uni(-20, 0)));
    const T nn = (T)uni(0.0, 0.12);
    T oh, ohu, ohv, speed, eh, ehu, ehv;
    lmask uodd = false;
    update_w<T>(h[0], hu[0], hv[0], r0, r1, r2, nn, true, P, w, oh, ohu, ohv, speed, uodd);
    update<T>(h[0], hu[0], hv[0], r0, r1, r2, dt, nn, P, eh, ehu, ehv);
    updates.n++;
    updates.odd += uodd;
    if (!uodd) {
      same("h", oh, eh);
      same("hu", ohu, ehu);
      same("hv", ohv, ehv);
      if (eh >= hm) {
        const T au = vabs(ehu), av = vabs(ehv);
        same("speed", speed, (au > av ? au : av) / eh + vsqrt(P.g * eh));
      } else {
        same("speed", speed, T(0));
      }
    }
  }
}

int main() {
  const char* names[] = {"wet", "films and dry cells", "fast", "still", "special values"};
  int rc = 0;
  for (int r = 0; r < 5; ++r) {
    Count f32f, f32u, f64f, f64u, f64sf, f64su;
    run<float>(r, 1e-6f, 1000000, f32f, f32u);
    run<double>(r, 1e-6, 300000, f64f, f64u);
    run<double>(r, 1e-10, 300000, f64sf, f64su);
    const double o[] = {(double)f32f.odd / f32f.n, (double)f32u.odd / f32u.n, (double)f64f.odd / f64f.n,
                        (double)f64u.odd / f64u.n, (double)f64sf.odd / f64sf.n, (double)f64su.odd / f64su.n};
    printf("%s: left to the general functions: float32 faces %.2g updates %.2g, float64 %.2g %.2g, small h_min %.2g %.2g\n",
           names[r], o[0], o[1], o[2], o[3], o[4], o[5]);
    // the states of a flood stay with the wavefront forms
    if (r < 4)
      for (double x : o) rc |= x > 1e-3;
  }
  // scalars outside the bounds never take them
  Phys<float> P = phys<float>(1e-6f, 1);
  P.g = 20.0f;
  rc |= wave_flags<float>(P, false) != 0;
  P = phys<float>(1e-9f, 1);
  rc |= wave_flags<float>(P, false) != 0;
  printf("mismatches %ld\n", g_bad);
  return rc || g_bad ? 1 : 0;
}
