// Instances and launches of the winner search over excess planes.
#include "sgm_internal.h"

namespace sgm {

template <int LANES, int R, int CB, int NPL, int G>
static int launch_winner_t(hipStream_t st, bool nt, dim3 grid, const PathJobs &jobs,
                           const WinnerArgs &A, int job0) {
  constexpr int threads = 64 * kWinnerWaves;
  if (nt) winner_kernel<LANES, R, CB, NPL, G, true><<<grid, threads, 0, st>>>(jobs, A, job0);
  else winner_kernel<LANES, R, CB, NPL, G, false><<<grid, threads, 0, st>>>(jobs, A, job0);
  return launch_check("winner kernel");
}

template <int LANES, int R>
static int launch_winner_r(hipStream_t st, int cost_bytes, int planes, int largest, bool nt,
                           dim3 grid, const PathJobs &jobs, const WinnerArgs &A, int job0) {
  // two planes are added as bytes where their sum fits one (P2 <= 127)
  const bool two = 2 * largest <= 255;
  if (planes == 8) {
    if (cost_bytes == 2) return launch_winner_t<LANES, R, 2, 8, 1>(st, nt, grid, jobs, A, job0);
    if (two) return launch_winner_t<LANES, R, 1, 8, 2>(st, nt, grid, jobs, A, job0);
    return launch_winner_t<LANES, R, 1, 8, 1>(st, nt, grid, jobs, A, job0);
  }
  if (cost_bytes == 2) return launch_winner_t<LANES, R, 2, 4, 1>(st, nt, grid, jobs, A, job0);
  if (two) return launch_winner_t<LANES, R, 1, 4, 2>(st, nt, grid, jobs, A, job0);
  return launch_winner_t<LANES, R, 1, 4, 1>(st, nt, grid, jobs, A, job0);
}

int launch_winner(sgm_context *ctx, int Dp, int cost_bytes, int planes, int largest, bool nt,
                  const PathJobs &jobs, const WinnerArgs &A, int w, int h, int njobs, bool narrow,
                  hipStream_t stream) {
  ProfileScope ps(ctx, "path_winner");
  hipStream_t st = stream ? stream : ctx->stream;
  int lanes = 0, R = 0;
  if ((planes != 4 && planes != 8) || !excess_shape(Dp, lanes, R))
    return fail(SGM_ERR_INVALID_ARGUMENT, "no winner search over %d planes of %d disparities",
                planes, Dp);
  // rows of 20 bytes a lane are split (PlaneRow) where the sweeps have that shape too;
  // narrow sweeps leave 320 disparities in order
  int narrow_lanes, narrow_R;
  if (narrow && R == 20 && narrow_shape(Dp, narrow_lanes, narrow_R)) {
    lanes = 32;
    R = 16;
  }
  constexpr int kMaxZ = 65535;  // grid z limit: jobs in slices
  for (int z0 = 0; z0 < njobs; z0 += kMaxZ) {
    const unsigned px = kWinnerPixels * kWinnerWaves;
    const dim3 grid((unsigned)(w + px - 1) / px, (unsigned)h, (unsigned)std::min(kMaxZ, njobs - z0));
    int rc = SGM_ERR_INVALID_ARGUMENT;
#define CASE(L, RR)            \
  if (lanes == L && R == RR)   \
    rc = launch_winner_r<L, RR>(st, cost_bytes, planes, largest, nt, grid, jobs, A, z0);
    CASE(16, 4) CASE(16, 8) CASE(16, 12) CASE(16, 16) CASE(16, 20)
    CASE(32, 12) CASE(32, 16) CASE(32, 20) CASE(64, 12) CASE(64, 16)
#undef CASE
    if (rc) return rc;
  }
  return SGM_OK;
}

}  // namespace sgm
