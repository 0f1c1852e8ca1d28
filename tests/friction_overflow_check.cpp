// drag_vanishes (gpu-comcot_amd/csrc/fastdiv.h) at fluxes, depths and
// coefficients whose friction leaves the range of a float, as a run that has
// blown up brings them: infinities, NaN and squares that overflow.  Wherever it
// holds, X - FF P and 1 + FF have to be X and 1 there too.  Prints the number
// of cases where it held and of those where a term moved X.
#include <stdio.h>

#include "../gpu-comcot_amd/csrc/detmath.h"
#include "../gpu-comcot_amd/csrc/fastdiv.h"

int main() {
  const float inf = INFINITY, nan = NAN;
  const float flux[] = {0.0f, 1e-30f, 1.0f, 1e6f, 1e10f, 1.5e19f, 3e19f, 1e25f, 1e30f, 3e38f, inf, nan};
  const float depth[] = {1.0f, 100.0f, 4000.0f, 7e5f, 1e6f, 1e10f, 1e14f, 1e16f, 1e18f, 3e19f, 1e30f, 3e38f, inf, nan};
  const float left[] = {0.0f, 1e-20f, 1.0f, 1e10f, 1e20f, 1e30f, 3e38f, inf, nan};
  const float coef[] = {0.0f, 1e-40f, 1e-20f, 1e-6f, 3e-3f, 1.0f, 1e12f, 1e30f, 3e38f, inf, nan};
  long long held = 0, moved = 0;
  for (float kf : coef)
    for (float p0 : flux)
      for (float q0 : flux)
        for (float df : depth)
          for (float x0 : left)
            for (int sign = 0; sign < 8; ++sign) {
              const float p = sign & 1 ? -p0 : p0, q = sign & 2 ? -q0 : q0, x = sign & 4 ? -x0 : x0;
              if (!gc::drag_vanishes(gc::drag_scaled(kf), p, q, df, x)) continue;
              ++held;
              const float ff = kf * sqrtf(p * p + q * q) / gcdet::powf_det(df, 2.3333333f);
              if (x - ff * p != x || 1.0f + ff != 1.0f) ++moved;
            }
  printf("%lld %lld\n", held, moved);
}
