// CPU comparison of update_w and speed_w (gs_wave.h, built for one lane) with the general functions
// (gs_device.h), over the physics that wave_check.cpp holds fixed: friction on and off, both
// friction formulas, with and without the velocity cap and the kept film, steps of 1 ms to 3 h,
// Manning numbers and momenta of every size, and values that are not finite in the momenta of
// dry cells as of wet ones. Test infrastructure only.
#define main wave_check_main
#include "wave_check.cpp"
#undef main

template <typename T>
static double log_uni(double lo, double hi) { return pow(10.0, uni(lo, hi)); }

// kind: 0 flood, 1 creeping films, 2 special values in the momenta, 3 special values anywhere
template <typename T>
static void updates(int kind, long n, Count& c) {
  for (long k = 0; k < n; ++k) {
    Phys<T> P = phys<T>(rnd() % 4 == 0 ? T(1e-3) : T(1e-6), (int)(rnd() & 1));
    P.friction = (int)(rnd() % 3 != 0);
    P.keep_h = (int)(rnd() & 1);
    P.has_vcap = (int)(rnd() & 1);
    if (rnd() % 4 == 0) P.vcap = (T)log_uni<T>(-25, 2);
    const T dt = (T)log_uni<T>(-3, 4);
    const WaveC<T> w = wave_consts<T>(P, dt, wave_flags<T>(P, false));
    T h = rnd() % 4 == 0 ? T(0) : (T)log_uni<T>(-8, 1), hu, hv;
    switch (kind) {
      case 0: hu = (T)(h * uni(-3, 3)); hv = (T)(h * uni(-3, 3)); break;
      case 1: hu = (T)(h * uni(-1, 1) * log_uni<T>(-25, -8)); hv = rnd() & 1 ? T(0) : (T)(h * uni(-1, 1) * log_uni<T>(-25, -8)); break;
      default: hu = rnd() & 1 ? special<T>() : (T)uni(-2, 2); hv = rnd() & 1 ? special<T>() : (T)uni(-2, 2); break;
    }
    T r0 = (T)(uni(-0.2, 1.0) * log_uni<T>(-8, -3)), r1 = T(0), r2 = T(0);
    if (kind == 0) r1 = (T)(uni(-1, 1) * h), r2 = (T)(uni(-1, 1) * h);
    if (kind == 3) {
      if (rnd() % 4 == 0) h = special<T>();
      if (rnd() % 4 == 0) r0 = special<T>();
      if (rnd() % 4 == 0) r1 = special<T>();
    }
    T nn = kind == 3 && rnd() % 4 == 0 ? vabs(special<T>()) : (T)(rnd() % 8 == 0 ? 0.0 : log_uni<T>(-3, 0));
    if (kind > 1 && rnd() % 4 == 0) nn = (T)log_uni<T>(3, sizeof(T) == 4 ? 19 : 154);   // n^2 up to the largest number
    T oh, ohu, ohv, speed, eh, ehu, ehv;
    lmask odd = false;
    update_w<T>(h, hu, hv, r0, r1, r2, nn, true, P, w, oh, ohu, ohv, speed, odd);
    update<T>(h, hu, hv, r0, r1, r2, dt, nn, P, eh, ehu, ehv);
    c.n++;
    c.odd += odd;
    if (odd) continue;
    const long before = g_bad;
    same("h", oh, eh);
    same("hu", ohu, ehu);
    same("hv", ohv, ehv);
    T want = T(0);
    if (!(eh < P.h_min)) {   // lam_key's speed: a NaN component leaves a NaN speed or a general one
      const T au = vabs(ehu), av = vabs(ehv);
      want = (au != au || av != av) ? T(NAN) : (au > av ? au : av) / eh + vsqrt(P.g * eh);
    }
    same("speed", speed, want);
    // a state that the update did not make
    const T sw = speed_w<T>(eh, ehu, ehv, w);
    if (sw < kMaxSpeed<T>) same("speed_w", sw, want);
    if (g_bad != before && g_bad < 12)
      printf("  kind %d friction %d quadratic %d dt %.9g n %.9g vcap %d %.9g: h %.17g hu %.17g hv %.17g r %.17g %.17g\n",
             kind, P.friction, P.quadratic, (double)dt, (double)nn, P.has_vcap, (double)P.vcap, (double)h, (double)hu,
             (double)hv, (double)r0, (double)r1);
  }
}

int main() {
  const char* names[] = {"flood", "creeping films", "special momenta", "special values"};
  int rc = 0;
  for (int k = 0; k < 4; ++k) {
    Count f, d;
    updates<float>(k, 2000000, f);
    updates<double>(k, 1000000, d);
    const double of = (double)f.odd / f.n, od = (double)d.odd / d.n;
    printf("%s: left to the general functions: float32 %.2g float64 %.2g; mismatches so far %ld\n", names[k], of, od, g_bad);
    if (k < 2) rc |= of > 1e-3 || od > 1e-3;   // the states of a flood stay with the wavefront forms
  }
  printf("mismatches %ld\n", g_bad);
  return rc || g_bad ? 1 : 0;
}
