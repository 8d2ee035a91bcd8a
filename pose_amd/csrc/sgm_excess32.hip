// Instances and launches of the excess-plane sweeps and the winner search with
// path costs and aggregates in 32 bits (uint16 costs, four planes).
#include "sgm_internal.h"

namespace sgm {

template <int LANES, int R, bool NT>
static void launch_excess32_t(hipStream_t st, const PathJobs &jobs, const ExcessArgs &A) {
  const unsigned blocks = (unsigned)((A.total + 3) / 4);
  if (A.pairs) excess_kernel<LANES, R, 2, true, NT, true><<<blocks, 256, 0, st>>>(jobs, A);
  else excess_kernel<LANES, R, 2, false, NT, true><<<blocks, 256, 0, st>>>(jobs, A);
}

int launch_excess32(sgm_context *ctx, int Dp, bool nt, const PathJobs &jobs, const ExcessArgs &A) {
  ProfileScope ps(ctx, "path_excess");
  if (A.total <= 0) return SGM_OK;
  int lanes = 0, R = 0;
  if (A.planes == 4 && excess_shape(Dp, lanes, R)) {
#define CASE(L, RR)                                                   \
  if (lanes == L && R == RR) {                                        \
    if (nt) launch_excess32_t<L, RR, true>(ctx->stream, jobs, A);     \
    else launch_excess32_t<L, RR, false>(ctx->stream, jobs, A);       \
    return launch_check("32-bit excess sweep kernel");                \
  }
    CASE(16, 4) CASE(16, 8) CASE(16, 12) CASE(16, 16) CASE(16, 20)
    CASE(32, 12) CASE(32, 16) CASE(32, 20) CASE(64, 12) CASE(64, 16)
#undef CASE
  }
  return fail(SGM_ERR_INVALID_ARGUMENT, "no 32-bit excess sweep for %d padded disparities", Dp);
}

int launch_winner32(sgm_context *ctx, int Dp, bool nt, const PathJobs &jobs, const WinnerArgs &A,
                    int w, int h, int njobs) {
  ProfileScope ps(ctx, "path_winner");
  const unsigned px = kWinnerPixels * kWinnerWaves;
  const dim3 grid((unsigned)(w + px - 1) / px, (unsigned)h, (unsigned)njobs);
  constexpr int threads = 64 * kWinnerWaves;
  int lanes = 0, R = 0;
  if (excess_shape(Dp, lanes, R)) {
#define CASE(L, RR)                                                                        \
  if (lanes == L && R == RR) {                                                             \
    if (nt) winner32_kernel<L, RR, true><<<grid, threads, 0, ctx->stream>>>(jobs, A);      \
    else winner32_kernel<L, RR, false><<<grid, threads, 0, ctx->stream>>>(jobs, A);        \
    return launch_check("32-bit winner kernel");                                           \
  }
    CASE(16, 4) CASE(16, 8) CASE(16, 12) CASE(16, 16) CASE(16, 20)
    CASE(32, 12) CASE(32, 16) CASE(32, 20) CASE(64, 12) CASE(64, 16)
#undef CASE
  }
  return fail(SGM_ERR_INVALID_ARGUMENT, "no 32-bit winner search for %d padded disparities", Dp);
}

}  // namespace sgm
