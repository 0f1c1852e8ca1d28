// drag_vanishes (gpu-comcot_amd/csrc/fastdiv.h): wherever it holds, the
// friction terms X - FF P and X / (1 + FF) of the momentum equations give X
// itself.  Random fluxes, depths from 1 up and coefficients, with X drawn
// around both of its bounds, zeros among them; FF as the oracle computes it.
// Prints the number of cases where it held and of those where a term moved X.
#include <stdio.h>

#include <random>

#include "../gpu-comcot_amd/csrc/detmath.h"
#include "../gpu-comcot_amd/csrc/fastdiv.h"

int main() {
  std::mt19937_64 rng(7);
  auto logu = [&](double lo, double hi) {
    return (float)exp2(std::uniform_real_distribution<double>(lo, hi)(rng));
  };
  const float steps[] = {1.0f, 1.5f, 511.99997f, 512.0f, 512.00006f};
  long long held = 0, moved = 0;
  for (long long k = 0; k < 4000000; ++k) {
    const float kf = logu(-16, 2), df = k % 16 == 0 ? steps[k / 16 % 5] : logu(0, 14);
    const float w = df * df * (df >= 512.0f ? 8.0f : 1.0f), kf26 = gc::kDragScale * kf;
    // |P| + |Q| around the bound on FF, split anyhow (k % 7 == 0: far below)
    const float sum = w / kf26 * (k % 7 == 0 ? logu(-140, 0) : logu(-6, 0.01));
    const float part = std::uniform_real_distribution<float>(0, 1)(rng);
    const float p = (k & 1 ? -1.0f : 1.0f) * (k % 11 == 0 ? sum : sum * part), q = sum - fabsf(p);
    const float x = k % 13 == 0 ? p : (k & 2 ? -1.0f : 1.0f) * kf26 * (fabsf(p) + fabsf(q)) * fabsf(p) / w * logu(-0.01, 3);
    if (!gc::drag_vanishes(kf26, p, q, df, x)) continue;
    ++held;
    const float ff = kf * sqrtf(p * p + q * q) / gcdet::powf_det(df, 2.3333333f);
    if (x - ff * p != x || 1.0f + ff != 1.0f) ++moved;
  }
  printf("%lld %lld\n", held, moved);
}
