// CPU check of the slot form of the FP64 histogram kernel's fixed-point floor
// (fix_slot, fix_slot_from_rsq in softx-d-16-00083_amd/csrc/xs_fixbin.h):
// squared distances in units of (2 bins)^2, a window offset folded into the
// sum, reciprocal square roots perturbed to v_rsq_f64's documented worst
// accuracy.  Wherever the low word passes, the AND of the high word must give
// the slot of the reference expression (unsigned)(sqrt(s) / bin).  A band
// without a margin must fail on the same samples.
#include <cmath>
#include <cstdio>
#include <random>

#include "xs_fixbin.h"
#include "xs_hist_plan.h"

using namespace xs::hist;

static unsigned long long fast, doubtful, wrong;

static void one(double t, double bin, long double e, int32_t off, const FixSlot &fs) {
  const double r = t * bin;                        // a distance, binned by the reference
  const uint32_t want = (uint32_t)(r / bin);
  const double h = 0.5 * (1.0 / bin) * r, s = h * h;  // (r / 2 bins)^2
  const double y = (double)((1.0L + e) / sqrtl((long double)s));
  uint32_t lo;
  const uint32_t at = fix_slot_from_rsq(s, y, fs.m, lo) & (65536 * 4 - 4);
  if (lo <= fs.lm1)
    ++doubtful;
  else if (at == (want + (uint32_t)off) << 2)
    ++fast;
  else
    ++wrong;
}

int main() {
  std::mt19937_64 rng(11);
  std::uniform_real_distribution<double> u(0.0, 1.0);
  std::uniform_real_distribution<long double> ed(-0x1p-23L, 0x1p-23L);
  int bad = 0;
  for (uint32_t nh : {64u, 8192u, 97251u, 700000u, 3000000u})
    for (double bin : {0.005, 0.0173, 1.0 / 3.0})
      for (int w = 0; w < 4; ++w) {
        // windows from bin 0 and from further up
        const uint32_t B = nh > 40000 ? (uint32_t)((nh - 32768.0) * w / 3.0) : 0;
        const uint32_t top = nh - B < 32768 ? nh - B : 32768;
        const int32_t off = -(int32_t)B;
        const FixSlot fs = fix_slot(band_for(nh), off);
        const FixSlot none{0x1p18 + (double)off, 0u};
        unsigned long long naive = 0;
        fast = doubtful = wrong = 0;
        for (int i = 0; i < 100000; ++i) one(B + u(rng) * (top - 1) + 0.5, bin, ed(rng), off, fs);
        const unsigned long long uniform_doubtful = doubtful;
        for (int i = 0; i < 4000; ++i) {
          const uint32_t k = B + 1 + (uint32_t)(u(rng) * (top - 2));
          for (int p = 16; p <= 48; p += 4)
            for (int sg = -1; sg <= 1; ++sg)
              for (long double e : {-0x1p-23L, 0x1p-23L, 0.0L}) {
                const double t = k + sg * std::ldexp(1.0, -p);
                one(t, bin, e, off, fs);
                const unsigned long long w0 = wrong;
                one(t, bin, e, off, none);
                naive += wrong - w0;
                wrong = w0;
              }
        }
        if (wrong || fast < 100000 || uniform_doubtful > 1000) {
          std::printf("nhist %u bin %g B %u: fast %llu doubtful %llu (%llu uniform) wrong %llu\n", nh,
                      bin, B, fast, doubtful, uniform_doubtful, wrong);
          bad = 1;
        }
        if (nh >= 97251 && naive == 0) {
          std::printf("a band without margin passed: nhist %u bin %g\n", nh, bin);
          bad = 1;
        }
      }
  // zero, negative and non-finite squared distances are doubtful
  const FixSlot fs = fix_slot(band_for(97251), -1000);
  for (double s : {0.0, -0x1p-60, (double)INFINITY, (double)NAN}) {
    uint32_t lo;
    fix_slot_from_rsq(s, 1.0 / std::sqrt(s), fs.m, lo);
    if (lo > fs.lm1) bad = 1;
  }
  std::printf(bad ? "FAIL\n" : "OK\n");
  return bad;
}
