// Which config an exact linear call of a given size runs (host code): a cost model of the
// kernels' tiles, for shapes and row counts no tuning table covers.
//
// Every candidate's time is t = fixed + rounds * (round + step * K / 1024) + byte * MB, with
// rounds = cdiv(workgroups, 256) rounds of one workgroup per CU and MB the weight digits in
// 1e6 bytes: the rounds carry the work of a workgroup (its K steps and its fixed phases), the
// last term the weight stream where that is longer. The coefficients (us) are least-squares fits
// of the relative error to graph-replay timings on MI355X of each candidate at 133 (M, N, K)
// grids x 5 (F = 14, 3 dots: 845 sizes, F = 15, 4 dots: 665), M = 1..4096, N = 512..16384, K =
// 512..12288, weights rotated. The picked candidate then takes 1.026x (3 dots) and 1.018x
// (4 dots) the time of the best of all 50 measured at that size on average, 1.13x and 1.10x at
// the 95th percentile; the fixed configs by row count it replaces took 2.1x on average at M >= 96.

#include <cmath>

#include "exact_gemm_common.h"

namespace {

constexpr int64_t kAnyRows = int64_t(1) << 40;

struct Candidate {
  bool one_launch;   // digitize inside the GEMM launch
  int64_t max_rows;  // taken up to this many rows
  int32_t bm, bn, bk, waves, stages;
  float fixed, round, step, byte;
};

constexpr Candidate kThreeDots[] = {
    {false, kAnyRows, 16, 16, 128, 8, 1, 2.613f, 0.168f, 0.647f, 0.079f},
    {false, kAnyRows, 16, 16, 128, 16, 1, 2.163f, 0.626f, 0.580f, 0.085f},
    {false, kAnyRows, 16, 32, 128, 4, 1, 3.180f, 0.000f, 0.995f, 0.096f},
    {false, kAnyRows, 16, 32, 128, 8, 1, 2.473f, 0.495f, 0.713f, 0.109f},
    {false, kAnyRows, 32, 16, 128, 8, 1, 2.557f, 0.264f, 0.924f, 0.068f},
    {false, kAnyRows, 32, 32, 128, 4, 1, 3.513f, 0.269f, 1.348f, 0.083f},
    {false, kAnyRows, 32, 32, 128, 8, 1, 2.829f, 0.534f, 1.335f, 0.088f},
    {false, kAnyRows, 32, 128, 64, 4, 4, 4.248f, 0.686f, 3.728f, 0.070f},
    {false, kAnyRows, 64, 16, 128, 8, 1, 2.600f, 0.880f, 1.651f, 0.062f},
    {false, kAnyRows, 64, 32, 128, 8, 1, 3.098f, 1.498f, 1.979f, 0.082f},
    {false, kAnyRows, 64, 64, 256, 8, 2, 0.620f, 4.043f, 2.847f, 0.082f},
    {false, kAnyRows, 64, 96, 256, 8, 2, 0.720f, 5.185f, 3.511f, 0.091f},
    {false, kAnyRows, 64, 128, 128, 8, 2, 2.362f, 2.235f, 4.255f, 0.100f},
    {false, kAnyRows, 64, 192, 128, 8, 2, 0.160f, 5.749f, 5.710f, 0.121f},
    {false, kAnyRows, 128, 128, 128, 8, 2, 0.000f, 7.254f, 6.593f, 0.077f},
    {false, kAnyRows, 128, 192, 128, 8, 2, 0.000f, 9.454f, 9.756f, 0.044f},
    {true, 4, 16, 16, 128, 8, 1, 3.162f, 0.460f, 1.367f, 0.000f},
    {true, 64, 16, 16, 128, 8, 1, 2.742f, 0.532f, 1.882f, 0.000f},
    {true, 4, 16, 16, 128, 16, 1, 2.584f, 1.550f, 0.939f, 0.034f},
    {true, 64, 16, 16, 128, 16, 1, 2.480f, 1.242f, 1.584f, 0.000f},
    {true, 4, 16, 32, 128, 8, 1, 2.365f, 1.263f, 1.515f, 0.060f},
    {true, 64, 16, 32, 128, 8, 1, 2.253f, 1.041f, 2.180f, 0.047f},
    {true, 4, 16, 32, 128, 16, 1, 0.000f, 3.970f, 1.381f, 0.065f},
    {true, 64, 16, 32, 128, 16, 1, 0.936f, 2.753f, 1.987f, 0.052f},
    {true, 4, 16, 64, 128, 8, 1, 0.000f, 3.714f, 2.001f, 0.095f},
    {true, 64, 16, 64, 128, 8, 1, 1.487f, 2.136f, 2.986f, 0.079f},
};

constexpr Candidate kFourDots[] = {
    {false, kAnyRows, 16, 16, 128, 8, 1, 2.696f, 0.185f, 0.681f, 0.076f},
    {false, kAnyRows, 16, 16, 128, 16, 1, 2.250f, 0.692f, 0.623f, 0.076f},
    {false, kAnyRows, 16, 32, 128, 4, 1, 3.320f, 0.017f, 1.017f, 0.101f},
    {false, kAnyRows, 16, 32, 128, 8, 1, 2.796f, 0.331f, 0.989f, 0.107f},
    {false, kAnyRows, 32, 16, 128, 8, 1, 2.748f, 0.424f, 0.984f, 0.076f},
    {false, kAnyRows, 32, 32, 128, 4, 1, 3.677f, 0.593f, 1.410f, 0.080f},
    {false, kAnyRows, 32, 32, 128, 8, 1, 2.565f, 1.044f, 1.381f, 0.086f},
    {false, kAnyRows, 32, 128, 64, 4, 4, 6.230f, 1.777f, 4.229f, 0.052f},
    {false, kAnyRows, 64, 16, 128, 8, 1, 2.682f, 1.097f, 1.656f, 0.051f},
    {false, kAnyRows, 64, 32, 128, 8, 1, 0.356f, 4.160f, 2.531f, 0.090f},
    {false, kAnyRows, 64, 64, 256, 8, 2, 0.642f, 6.476f, 3.169f, 0.071f},
    {false, kAnyRows, 64, 96, 256, 8, 2, 0.703f, 8.977f, 3.897f, 0.073f},
    {false, kAnyRows, 64, 128, 128, 8, 2, 0.000f, 8.989f, 5.086f, 0.072f},
    {false, kAnyRows, 64, 192, 128, 8, 2, 0.000f, 12.544f, 6.816f, 0.086f},
    {false, kAnyRows, 128, 128, 128, 8, 2, 0.000f, 16.151f, 8.685f, 0.042f},
    {true, 4, 16, 16, 128, 8, 1, 3.047f, 0.801f, 1.440f, 0.000f},
    {true, 64, 16, 16, 128, 8, 1, 2.635f, 0.992f, 1.898f, 0.000f},
    {true, 4, 16, 16, 128, 16, 1, 2.414f, 2.021f, 1.209f, 0.007f},
    {true, 64, 16, 16, 128, 16, 1, 1.762f, 2.505f, 1.660f, 0.000f},
    {true, 4, 16, 32, 128, 8, 1, 2.816f, 1.105f, 1.504f, 0.066f},
    {true, 64, 16, 32, 128, 8, 1, 2.154f, 1.603f, 2.127f, 0.048f},
    {true, 4, 16, 32, 128, 16, 1, 1.483f, 3.549f, 1.327f, 0.075f},
    {true, 64, 16, 32, 128, 16, 1, 1.175f, 3.178f, 2.134f, 0.046f},
    {true, 4, 16, 64, 128, 8, 1, 0.000f, 4.249f, 1.990f, 0.092f},
    {true, 64, 16, 64, 128, 8, 1, 0.000f, 4.341f, 2.965f, 0.084f},
};

double cost(const Candidate& c, int64_t m, int64_t n, int64_t k, int sk) {
  const double kp = (double)cdiv<int64_t>(k, 64) * 64;
  const double rounds = std::ceil((double)cdiv<int64_t>(m, c.bm) * (double)cdiv<int64_t>(n, c.bn) * sk / 256.0);
  double t = c.fixed + rounds * (c.round + c.step * kp / sk / 1024.0) + c.byte * 2.0 * (double)n * kp / 1e6;
  if (!c.one_launch) t += 2.9 + (double)m * kp / 1.1e6;                      // digitize: its launch, then its bytes
  if (sk > 1) t += 2.6 + (double)m * (double)n * 8.0 * sk * 2.0 / 5e6;       // partials written and read, finalize
  return t;
}

}  // namespace

extern "C" int vxa_exact_linear_pick(int64_t m, int64_t n, int64_t k, int trunc, int one_launch_ok, int32_t* cfg,
                                     int* one_launch) {
  if (m < 0 || n < 0 || k < 0 || !cfg || !one_launch) return VXA_ERR_ARG;
  const Candidate* set = trunc ? kThreeDots : kFourDots;
  const int count = trunc ? (int)(sizeof(kThreeDots) / sizeof(Candidate)) : (int)(sizeof(kFourDots) / sizeof(Candidate));
  const Candidate* best = nullptr;
  double best_t = 0;
  int best_sk = 1;
  for (int i = 0; i < count; ++i) {
    const Candidate& c = set[i];
    if (m > c.max_rows || (c.one_launch && (!one_launch_ok || k > 32768))) continue;
    if (c.one_launch && i > 0 && set[i - 1].max_rows >= m && set[i - 1].one_launch && set[i - 1].bn == c.bn &&
        set[i - 1].waves == c.waves)
      continue;  // the same config's coefficients for fewer rows apply
    // K splits of the K-split kernel while its grid leaves CUs idle, at least 512 columns each
    const bool splits = c.bm >= 64 && c.waves == 8 && c.stages == 2;
    const double tiles = (double)cdiv<int64_t>(m, c.bm) * (double)cdiv<int64_t>(n, c.bn);
    for (int sk = 1; sk <= 4; sk *= 2) {
      if (sk > 1 && (!splits || k / sk < 512 || tiles * sk > 640)) break;
      const double t = cost(c, m, n, k, sk);
      if (!best || t < best_t) {
        best = &c;
        best_t = t;
        best_sk = sk;
      }
    }
  }
  cfg[0] = best->bm;
  cfg[1] = best->bn;
  cfg[2] = best->bk;
  cfg[3] = best->waves;
  cfg[4] = best->stages;
  cfg[5] = 8;
  cfg[6] = best_sk;
  *one_launch = best->one_launch ? 1 : 0;
  return VXA_OK;
}
