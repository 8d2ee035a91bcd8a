// Instances and launches of the excess-plane sweeps.
#include "sgm_internal.h"

namespace sgm {

template <int LANES, int R, int CB, bool PAIR>
static int launch_excess_t(hipStream_t st, bool nt, const PathJobs &jobs, const ExcessArgs &A) {
  constexpr int waves = 4;
  const unsigned blocks = (unsigned)((A.total + waves - 1) / waves);
  if (nt) excess_kernel<LANES, R, CB, PAIR, true, false><<<blocks, waves * 64, 0, st>>>(jobs, A);
  else excess_kernel<LANES, R, CB, PAIR, false, false><<<blocks, waves * 64, 0, st>>>(jobs, A);
  return launch_check("excess sweep kernel");
}

template <int LANES, int R>
static int launch_excess_r(hipStream_t st, int cost_bytes, bool pairs, bool nt,
                           const PathJobs &jobs, const ExcessArgs &A) {
  if (cost_bytes == 1)
    return pairs ? launch_excess_t<LANES, R, 1, true>(st, nt, jobs, A)
                 : launch_excess_t<LANES, R, 1, false>(st, nt, jobs, A);
  return pairs ? launch_excess_t<LANES, R, 2, true>(st, nt, jobs, A)
               : launch_excess_t<LANES, R, 2, false>(st, nt, jobs, A);
}

int launch_excess(sgm_context *ctx, int Dp, int cost_bytes, bool nt, const PathJobs &jobs,
                  const ExcessArgs &A, hipStream_t stream) {
  ProfileScope ps(ctx, "path_excess");
  if (A.total <= 0) return SGM_OK;
  hipStream_t st = stream ? stream : ctx->stream;
  int lanes = 0, R = 0;
  if (excess_shape(Dp, lanes, R)) {
    if (A.narrow && narrow_shape(Dp, lanes, R)) {
#define CASE(L, RR)                                                          \
  if (lanes == L && R == RR)                                                 \
    return cost_bytes == 1 ? launch_excess_t<L, RR, 1, false>(st, nt, jobs, A) \
                           : launch_excess_t<L, RR, 2, false>(st, nt, jobs, A);
      CASE(32, 4) CASE(64, 4) CASE(64, 8)
#undef CASE
    }
    const bool pairs = A.pairs != 0;
#define CASE(L, RR) \
  if (lanes == L && R == RR) return launch_excess_r<L, RR>(st, cost_bytes, pairs, nt, jobs, A);
    CASE(16, 4) CASE(16, 8) CASE(16, 12) CASE(16, 16) CASE(16, 20)
    CASE(32, 12) CASE(32, 16) CASE(32, 20) CASE(64, 12) CASE(64, 16)
#undef CASE
  }
  return fail(SGM_ERR_INVALID_ARGUMENT, "no excess sweep for %d padded disparities", Dp);
}

}  // namespace sgm
