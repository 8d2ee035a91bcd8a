// Instances and launches of the compact plan's whole-image line sweeps.
#include "sgm_internal.h"
#include "sgm_compact.h"
#include "sgm_compact_lines.h"

namespace sgm {

template <int LANES, int R>
static int launch_compact_lines_t(hipStream_t st, int phase, const CompactJobs &J,
                                  const CompactLineArgs &A) {
  const unsigned blocks = (unsigned)((A.total + 3) / 4);
  if (phase == ESGM_CANDIDATES)
    compact_line_kernel<LANES, R, ESGM_CANDIDATES><<<blocks, 256, 0, st>>>(J, A);
  else if (phase == ESGM_SUMS)
    compact_line_kernel<LANES, R, ESGM_SUMS><<<blocks, 256, 0, st>>>(J, A);
  else
    compact_line_kernel<LANES, R, ESGM_VERIFY><<<blocks, 256, 0, st>>>(J, A);
  return launch_check("compact line sweep kernel");
}

int launch_compact_lines(sgm_context *ctx, int lanes, int R, int phase, const CompactJobs &J,
                         const CompactLineArgs &A) {
  static const char *names[3] = {"compact proposals", "compact sums", "compact verify"};
  ProfileScope ps(ctx, names[phase]);
#define CASE(L, RR) \
  if (lanes == L && R == RR) return launch_compact_lines_t<L, RR>(ctx->stream, phase, J, A);
  CASE(16, 4) CASE(16, 8) CASE(32, 8) CASE(64, 8)
#undef CASE
  return fail(SGM_ERR_INVALID_ARGUMENT, "no compact line sweep of %d x %d disparities", lanes, R);
}

}  // namespace sgm
