// The index arithmetic of BC7's pixel pass (fastc_amd/csrc/bc7_index.h) on the
// host, over every squared endpoint distance.  Prints the number of values
// checked; exits with 1 at the first that is wrong.
#include <stdio.h>

#include "../../fastc_amd/csrc/bc7_index.h"

using namespace fh::bc7;

static int fail(const char *what, int a, int b, int c) {
  printf("%s: %d %d %d\n", what, a, b, c);
  return 1;
}

int main() {
  static const int kWeights[3][16] = {
      {0, 21, 43, 64},
      {0, 9, 18, 27, 37, 46, 55, 64},
      {0, 4, 9, 13, 17, 21, 26, 30, 34, 38, 43, 47, 51, 55, 60, 64}};
  long long n = 0;
  for (int t = 0; t < 3; t++)
    for (int j = 0; j < 4 << t; j++, n++)
      if ((int)weight_of(weight_fn(4 << t), j) != kWeights[t][j])
        return fail("weight", 4 << t, j, 0);
  const int top = 4 * 255 * 255;
  for (int l = 1; l <= top; l++) {
    // the Newton step from every start within 2 ulp
    const float want = (float)(1.0 / (64.0 * l));
    for (host_rcp_ulps = -2; host_rcp_ulps <= 2; host_rcp_ulps++, n++)
      if (scaled_rcp(l) != want) return fail("reciprocal", l, host_rcp_ulps, 0);
    // both bounds around every step, and beyond either end
    for (int kf = 3; kf <= 15; kf = 2 * kf + 1)
      for (int k = 0; k <= kf; k++)
        for (int o = -2; o <= 2; o++, n++) {
          const long long d = (long long)k * l / kf + o;
          if (d < -top || d > top) continue;
          const long long c = d < 0 ? 0 : (d > l ? l : d);
          uint32_t j1, j2;
          index_bounds((int)(64 * d), want, (float)kf, j1, j2);
          // the reference's own float quotient names the same indices
          const float r = (float)c / (float)l * (float)kf;
          if (floorf(r) != (float)(c * kf / l) || ceilf(r) != (float)((c * kf + l - 1) / l))
            return fail("reference", l, (int)d, kf);
          if (j1 != c * kf / l) return fail("floor", l, (int)d, kf);
          if (j2 != (c * kf + l - 1) / l) return fail("ceiling", l, (int)d, kf);
        }
  }
  printf("%lld checked\n", n);
  return 0;
}
