// Instances of the band cost kernel for uint16 volumes.
#include "sgm_internal.h"

namespace sgm {

static constexpr bool OUT16 = true;

template <int LANES, int R, int WORDS, bool DIFF>
static int launch_band_t(hipStream_t st, const PathJobs &jobs, const BandArgs &A) {
  constexpr int waves = 4;
  const unsigned blocks = (unsigned)((A.total + waves - 1) / waves);
  band_cost_kernel<LANES, R, WORDS, DIFF, OUT16><<<blocks, waves * 64, 0, st>>>(jobs, A);
  return launch_check("band cost kernel");
}

int launch_band16(hipStream_t st, int Dp, int words, bool diff, const PathJobs &jobs, const BandArgs &A) {
  int lanes = 0, R = 0;
  if (excess_shape(Dp, lanes, R)) {
#define CASE(L, RR)                                                        \
  if (lanes == L && R == RR) {                                             \
    if (words == 1)                                                        \
      return diff ? launch_band_t<L, RR, 1, true>(st, jobs, A)             \
                  : launch_band_t<L, RR, 1, false>(st, jobs, A);           \
    return diff ? launch_band_t<L, RR, 2, true>(st, jobs, A)               \
                : launch_band_t<L, RR, 2, false>(st, jobs, A);             \
  }
    CASE(16, 4) CASE(16, 8) CASE(16, 12) CASE(16, 16) CASE(16, 20)
    CASE(32, 12) CASE(32, 16) CASE(32, 20) CASE(64, 12) CASE(64, 16)
#undef CASE
  }
  return fail(SGM_ERR_INVALID_ARGUMENT, "no band cost kernel for %d padded disparities", Dp);
}

}  // namespace sgm
