// Which config an exact linear call of a given size runs (host code): a cost model of the
// kernels' tiles, for shapes and row counts no tuning table covers.
//
// Every candidate's time is the larger of
//   fixed + ceil(r) * (round + step * K / 1024) + byte * MB   and   r * (many_round + many_step * K / 1024)
// with r = workgroups / 256, the rounds of one workgroup per CU, and MB the weight digits in 1e6
// bytes. A round carries the work of a workgroup (its fixed phases and its K steps), MB the weight
// stream where that is longer. Over many rounds a partly filled last one counts by its share, and a
// round takes longer: these kernels are power-bound and the chip then holds a lower clock. The
// coefficients (us) are least-squares fits of the relative error to graph-replay timings on MI355X
// of each candidate at 979 sizes (F = 14, 3 dots) and 749 (F = 15, 4 dots), M = 1..8192, N =
// 512..24576, K = 512..12288, weights rotated. Digitize and GEMM of the picked candidate take
// 1.023x (3 dots) and 1.017x (4 dots) the time of the best of all configs measured at that size on
// average, 1.11x and 1.10x at the 95th percentile (1.009x and 1.006x on average from 1024 rows
// up); the fixed configs by row count that it replaces took 1.8x below 96 rows and 1.9x from there
// to 1024. 1531 rows of fp16 through 5136 x 2600: 163.6 -> 66 us.

#include <algorithm>
#include <cmath>

#include "exact_gemm_common.h"

namespace {

constexpr int64_t kAnyRows = int64_t(1) << 40;

struct Candidate {
  bool one_launch;   // digitize inside the GEMM launch
  int64_t max_rows;  // taken up to this many rows
  int32_t bm, bn, bk, waves, stages;
  float fixed, round, step, byte, many_round, many_step;
};

constexpr Candidate kThreeDots[] = {
    {false, kAnyRows, 16, 16, 128, 8, 1, 2.552f, 0.184f, 0.665f, 0.078f, 0.000f, 0.000f},
    {false, kAnyRows, 16, 16, 128, 16, 1, 2.087f, 0.653f, 0.600f, 0.084f, 0.000f, 0.000f},
    {false, kAnyRows, 16, 32, 128, 4, 1, 3.172f, 0.000f, 0.993f, 0.097f, 0.000f, 0.000f},
    {false, kAnyRows, 16, 32, 128, 8, 1, 2.357f, 0.560f, 0.727f, 0.110f, 0.000f, 0.000f},
    {false, kAnyRows, 32, 16, 128, 8, 1, 2.501f, 0.263f, 0.937f, 0.072f, 0.000f, 0.000f},
    {false, kAnyRows, 32, 32, 128, 4, 1, 3.454f, 0.278f, 1.363f, 0.083f, 0.000f, 0.000f},
    {false, kAnyRows, 32, 32, 128, 8, 1, 2.770f, 0.547f, 1.349f, 0.090f, 0.000f, 0.000f},
    {false, kAnyRows, 32, 128, 64, 4, 4, 4.235f, 0.700f, 3.702f, 0.075f, 0.000f, 0.000f},
    {false, kAnyRows, 64, 16, 128, 8, 1, 2.574f, 0.885f, 1.635f, 0.071f, 0.000f, 0.000f},
    {false, kAnyRows, 64, 32, 128, 8, 1, 3.070f, 1.508f, 1.964f, 0.088f, 0.000f, 0.000f},
    {false, kAnyRows, 64, 64, 256, 8, 2, 1.380f, 3.691f, 2.462f, 0.105f, 3.125f, 4.133f},
    {false, kAnyRows, 64, 96, 256, 8, 2, 1.597f, 4.612f, 3.265f, 0.105f, 4.820f, 5.091f},
    {false, kAnyRows, 64, 128, 128, 8, 2, 2.814f, 1.997f, 4.068f, 0.106f, 2.032f, 5.394f},
    {false, kAnyRows, 64, 192, 128, 8, 2, 0.893f, 5.164f, 5.574f, 0.126f, 5.558f, 7.819f},
    {false, kAnyRows, 128, 128, 128, 8, 2, 0.000f, 7.203f, 6.340f, 0.076f, 6.508f, 9.486f},
    {false, kAnyRows, 128, 192, 128, 8, 2, 0.000f, 9.423f, 9.631f, 0.046f, 10.047f, 13.239f},
    {true, 4, 16, 16, 128, 8, 1, 3.162f, 0.460f, 1.367f, 0.000f, 0.000f, 0.000f},
    {true, 64, 16, 16, 128, 8, 1, 2.764f, 0.527f, 1.874f, 0.000f, 0.000f, 0.000f},
    {true, 4, 16, 16, 128, 16, 1, 2.584f, 1.550f, 0.939f, 0.034f, 0.000f, 0.000f},
    {true, 64, 16, 16, 128, 16, 1, 2.447f, 1.253f, 1.593f, 0.000f, 0.000f, 0.000f},
    {true, 4, 16, 32, 128, 8, 1, 2.365f, 1.263f, 1.515f, 0.060f, 0.000f, 0.000f},
    {true, 64, 16, 32, 128, 8, 1, 2.231f, 1.054f, 2.186f, 0.046f, 0.000f, 0.000f},
    {true, 4, 16, 32, 128, 16, 1, 0.000f, 3.970f, 1.381f, 0.065f, 0.000f, 0.000f},
    {true, 64, 16, 32, 128, 16, 1, 0.833f, 2.820f, 2.003f, 0.052f, 0.000f, 0.000f},
    {true, 4, 16, 64, 128, 8, 1, 0.000f, 3.714f, 2.001f, 0.095f, 0.000f, 0.000f},
    {true, 64, 16, 64, 128, 8, 1, 1.345f, 2.256f, 2.989f, 0.080f, 0.000f, 0.000f},
    {true, 4, 16, 48, 128, 8, 1, 2.955f, 0.000f, 1.563f, 0.098f, 0.000f, 0.000f},
    {true, 64, 16, 48, 128, 8, 1, 3.128f, 0.000f, 1.981f, 0.091f, 0.000f, 0.000f},
    {true, 4, 16, 80, 128, 8, 1, 0.906f, 2.809f, 2.485f, 0.083f, 0.000f, 0.000f},
    {true, 64, 16, 80, 128, 8, 1, 0.700f, 3.839f, 2.744f, 0.080f, 0.000f, 0.000f},
    {true, 4, 16, 96, 128, 8, 1, 0.956f, 2.951f, 2.959f, 0.085f, 0.000f, 0.000f},
    {true, 64, 16, 96, 128, 8, 1, 0.898f, 4.277f, 3.108f, 0.082f, 0.000f, 0.000f},
};

constexpr Candidate kFourDots[] = {
    {false, kAnyRows, 16, 16, 128, 8, 1, 2.696f, 0.185f, 0.681f, 0.076f, 0.000f, 0.000f},
    {false, kAnyRows, 16, 16, 128, 16, 1, 2.250f, 0.692f, 0.623f, 0.076f, 0.000f, 0.000f},
    {false, kAnyRows, 16, 32, 128, 4, 1, 3.320f, 0.017f, 1.017f, 0.101f, 0.000f, 0.000f},
    {false, kAnyRows, 16, 32, 128, 8, 1, 2.796f, 0.331f, 0.989f, 0.107f, 0.000f, 0.000f},
    {false, kAnyRows, 32, 16, 128, 8, 1, 2.748f, 0.424f, 0.984f, 0.076f, 0.000f, 0.000f},
    {false, kAnyRows, 32, 32, 128, 4, 1, 3.677f, 0.593f, 1.410f, 0.080f, 0.000f, 0.000f},
    {false, kAnyRows, 32, 32, 128, 8, 1, 2.565f, 1.044f, 1.381f, 0.086f, 0.000f, 0.000f},
    {false, kAnyRows, 32, 128, 64, 4, 4, 6.186f, 1.870f, 4.159f, 0.056f, 0.000f, 0.000f},
    {false, kAnyRows, 64, 16, 128, 8, 1, 2.682f, 1.097f, 1.656f, 0.051f, 0.000f, 0.000f},
    {false, kAnyRows, 64, 32, 128, 8, 1, 0.356f, 4.160f, 2.531f, 0.090f, 0.000f, 0.000f},
    {false, kAnyRows, 64, 64, 256, 8, 2, 1.475f, 6.174f, 2.634f, 0.098f, 5.679f, 4.238f},
    {false, kAnyRows, 64, 96, 256, 8, 2, 1.536f, 8.496f, 3.598f, 0.088f, 8.938f, 5.258f},
    {false, kAnyRows, 64, 128, 128, 8, 2, 0.499f, 8.739f, 4.730f, 0.085f, 8.142f, 6.367f},
    {false, kAnyRows, 64, 192, 128, 8, 2, 0.514f, 12.199f, 6.618f, 0.093f, 12.964f, 8.679f},
    {false, kAnyRows, 128, 128, 128, 8, 2, 0.000f, 16.201f, 8.395f, 0.029f, 15.379f, 11.051f},
    {true, 4, 16, 16, 128, 8, 1, 3.047f, 0.801f, 1.440f, 0.000f, 0.000f, 0.000f},
    {true, 64, 16, 16, 128, 8, 1, 2.635f, 0.992f, 1.898f, 0.000f, 0.000f, 0.000f},
    {true, 4, 16, 16, 128, 16, 1, 2.414f, 2.021f, 1.209f, 0.007f, 0.000f, 0.000f},
    {true, 64, 16, 16, 128, 16, 1, 1.762f, 2.505f, 1.660f, 0.000f, 0.000f, 0.000f},
    {true, 4, 16, 32, 128, 8, 1, 2.816f, 1.105f, 1.504f, 0.066f, 0.000f, 0.000f},
    {true, 64, 16, 32, 128, 8, 1, 2.154f, 1.603f, 2.127f, 0.048f, 0.000f, 0.000f},
    {true, 4, 16, 32, 128, 16, 1, 1.483f, 3.549f, 1.327f, 0.075f, 0.000f, 0.000f},
    {true, 64, 16, 32, 128, 16, 1, 1.175f, 3.178f, 2.134f, 0.046f, 0.000f, 0.000f},
    {true, 4, 16, 64, 128, 8, 1, 0.000f, 4.249f, 1.990f, 0.092f, 0.000f, 0.000f},
    {true, 64, 16, 64, 128, 8, 1, 0.000f, 4.341f, 2.965f, 0.084f, 0.000f, 0.000f},
    {true, 4, 16, 48, 128, 8, 1, 2.062f, 1.507f, 1.458f, 0.097f, 0.000f, 0.000f},
    {true, 64, 16, 48, 128, 8, 1, 1.807f, 2.413f, 1.759f, 0.089f, 0.000f, 0.000f},
    {true, 4, 16, 80, 128, 8, 1, 0.701f, 3.394f, 2.462f, 0.083f, 0.000f, 0.000f},
    {true, 64, 16, 80, 128, 8, 1, 0.780f, 4.421f, 2.662f, 0.081f, 0.000f, 0.000f},
    {true, 4, 16, 96, 128, 8, 1, 1.050f, 2.564f, 3.130f, 0.086f, 0.000f, 0.000f},
    {true, 64, 16, 96, 128, 8, 1, 0.940f, 4.488f, 3.203f, 0.082f, 0.000f, 0.000f},
};

double cost(const Candidate& c, int64_t m, int64_t n, int64_t k, int sk) {
  const double kp = (double)cdiv<int64_t>(k, 64) * 64;
  const double rounds = (double)cdiv<int64_t>(m, c.bm) * (double)cdiv<int64_t>(n, c.bn) * sk / 256.0;
  const double steps = kp / sk / 1024.0;
  double t = std::max(c.fixed + std::ceil(rounds) * (c.round + c.step * steps) + c.byte * 2.0 * (double)n * kp / 1e6,
                      rounds * (c.many_round + c.many_step * steps));
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
    const bool wide = c.one_launch && (c.bn == 48 || c.bn == 80 || c.bn == 96);
    if (wide && k > 4096) continue;  // its x registers end there
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
