// Census transform + texture mask (CensusSgm.java:523-555), rectangular window.
//
// A thread takes four neighbouring pixels, so a window row of all four is a few
// dwords from LDS and every byte is taken out once; the window is a template
// parameter, so each cell of a pixel costs a compare into the carry, an add with
// carry that shifts it into the descriptor (cells in reverse window order: the
// last bit first), and a minimum and a maximum shared by two cells.  Bound by
// VALU at about 3.2 instructions per cell and pixel, small images by the one
// round of loads of the tile.  Measured, both images of a pair, against a thread
// per pixel and a window known only at run time (12 instructions): 9x7 window
// 160x120 7.5 -> 6.8 us, 640x480 20 -> 10.7, 1600x1067 83 -> 33; 11x11 window
// 1201x801 106 -> 49.
#include "sgm_internal.h"

namespace sgm {

constexpr int kCensusPx = 4, kCensusW = 64, kCensusH = 16;

// d = 2 * d + (v < c)
__device__ __forceinline__ void census_bit(uint32_t &d, uint32_t v, uint32_t c) {
  asm("v_cmp_lt_u32_e32 vcc, %1, %2\n\tv_addc_co_u32_e32 %0, vcc, %0, %0, vcc"
      : "+v"(d)
      : "v"(v), "v"(c)
      : "vcc");
}

// SUMS: window sums of g and g^2 as well (ZNCC costs).
template <int WW, int WH, bool SUMS>
__global__ __launch_bounds__(256) void census_kernel(CensusJobs jobs) {
  constexpr int RX = WW / 2, RY = WH / 2, CELLS = WW * WH;
  constexpr int WORDS = (CELLS - 1 + 63) / 64, ND = (WW + kCensusPx - 1 + 3) / 4;
  constexpr int PITCH = kCensusW / 4 + 3;  // dwords
  const CensusJob &J = jobs.job[blockIdx.z];
  const int w = J.w, h = J.h;
  const int x0 = blockIdx.x * kCensusW, y0 = blockIdx.y * kCensusH;
  if (x0 >= w || y0 >= h) return;
  __shared__ uint32_t tile[kCensusH + WH - 1][PITCH];
  // The tile, all of a thread's loads in flight at once: 64 columns, then the
  // WW - 1 further ones.  Outside the image any pixel does (only windows that
  // are not inside see it).
  constexpr int ROWS = kCensusH + WH - 1, N0 = (ROWS + 3) / 4, N1 = (ROWS + 15) / 16;
  const int lane = lane_id(), wave = threadIdx.x >> 6;
  auto pixel = [&](int col, int row) {
    const int gx = min(max(x0 - RX + col, 0), w - 1), gy = min(max(y0 - RY + row, 0), h - 1);
    return J.gray[(size_t)gy * w + gx];
  };
  uint8_t in0[N0], in1[N1];
#pragma unroll
  for (int i = 0; i < N0; i++) in0[i] = pixel(lane, wave + 4 * i);
#pragma unroll
  for (int i = 0; i < N1; i++) in1[i] = pixel(64 + lane % 16, threadIdx.x / 16 + 16 * i);
#pragma unroll
  for (int i = 0; i < N0; i++)
    if (wave + 4 * i < ROWS) reinterpret_cast<uint8_t *>(tile[wave + 4 * i])[lane] = in0[i];
#pragma unroll
  for (int i = 0; i < N1; i++) {
    const int row = threadIdx.x / 16 + 16 * i;
    if (lane % 16 < WW - 1 && row < ROWS)
      reinterpret_cast<uint8_t *>(tile[row])[64 + lane % 16] = in1[i];
  }
  __syncthreads();
  const int tx = threadIdx.x % (kCensusW / kCensusPx), ty = threadIdx.x / (kCensusW / kCensusPx);
  const int x = x0 + tx * kCensusPx, y = y0 + ty;
  if (x >= w || y >= h) return;

  uint32_t c[kCensusPx], d[kCensusPx][2 * WORDS], lo[kCensusPx], hi[kCensusPx];
  int s1[kCensusPx], s2[kCensusPx];
  const uint8_t *mid = reinterpret_cast<const uint8_t *>(tile[ty + RY]) + tx * kCensusPx + RX;
#pragma unroll
  for (int j = 0; j < kCensusPx; j++) {
    c[j] = lo[j] = hi[j] = mid[j];
    s1[j] = s2[j] = 0;
#pragma unroll
    for (int i = 0; i < 2 * WORDS; i++) d[j][i] = 0;
  }
#pragma unroll
  for (int yy = WH - 1; yy >= 0; yy--) {
    uint32_t raw[ND], v[4 * ND];
#pragma unroll
    for (int i = 0; i < ND; i++) raw[i] = tile[ty + yy][tx + i];
#pragma unroll
    for (int i = 0; i < 4 * ND; i++) v[i] = raw[i / 4] >> (i % 4 * 8) & 0xFFu;
#pragma unroll
    for (int j = 0; j < kCensusPx; j++) {
#pragma unroll
      for (int xx = WW - 1; xx >= 0; xx--) {
        const int at = yy * WW + xx, centre = RY * WW + RX;
        if (SUMS) {
          s1[j] += (int)v[xx + j];
          s2[j] += (int)(v[xx + j] * v[xx + j]);
        }
        if (at != centre) census_bit(d[j][(at - (at > centre ? 1 : 0)) / 32], v[xx + j], c[j]);
      }
#pragma unroll
      for (int xx = 0; xx + 1 < WW; xx += 2) {
        lo[j] = min(min(lo[j], v[xx + j]), v[xx + 1 + j]);
        hi[j] = max(max(hi[j], v[xx + j]), v[xx + 1 + j]);
      }
      lo[j] = min(lo[j], v[WW - 1 + j]);
      hi[j] = max(hi[j], v[WW - 1 + j]);
    }
  }

  const size_t n = (size_t)w * h, p = (size_t)y * w + x;
  const int count = min(kCensusPx, w - x);
  uint32_t mask[kCensusPx];
#pragma unroll
  for (int j = 0; j < kCensusPx; j++) {
    const bool interior = x + j >= RX && x + j < w - RX && y >= RY && y < h - RY;
    if (!interior) {
#pragma unroll
      for (int i = 0; i < 2 * WORDS; i++) d[j][i] = 0;
      s1[j] = s2[j] = 0;
    }
    bool m = false;
    if (j < count) {
      if (J.mask_in) m = J.mask_in[p + j] != 0;
      else m = interior && hi[j] - lo[j] >= 4 && (J.valid == nullptr || J.valid[p + j] != 0);
    }
    mask[j] = m;
    // One-word descriptors use at most 62 bits; bit 63 carries texture&valid so a
    // sweep can test a target's usability from its descriptor alone.
    if (WORDS == 1) d[j][1] |= mask[j] << 31;
  }
  if (J.stats && p < 16)
    for (int j = 0; j < count && p + j < 16; j++) J.stats[p + j] = 0ULL;
  // rows of whole groups of four: one store per plane where its base allows
  const bool whole = (w & 3) == 0;
  auto bytes = [&](uint8_t *out, uint32_t v) {
    if (!out) return;
    if (whole && ((uintptr_t)out & 3) == 0) {
      *reinterpret_cast<uint32_t *>(out + p) = v;
    } else {
      for (int j = 0; j < count; j++) out[p + j] = (uint8_t)(v >> (8 * j));
    }
  };
  bytes(J.reasons, 0x01010101u);
  bytes(J.boundary, 0u);
  bytes(J.gray_copy, c[0] | (c[1] << 8) | (c[2] << 16) | (c[3] << 24));
  bytes(J.mask, mask[0] | (mask[1] << 8) | (mask[2] << 16) | (mask[3] << 24));
  if (J.gm) {
    if (whole && ((uintptr_t)J.gm & 7) == 0) {
      *reinterpret_cast<uint2 *>(J.gm + p) =
          make_uint2(c[0] | (mask[0] << 8) | (c[1] << 16) | (mask[1] << 24),
                     c[2] | (mask[2] << 8) | (c[3] << 16) | (mask[3] << 24));
    } else {
#pragma unroll
      for (int j = 0; j < kCensusPx; j++)
        if (j < count) J.gm[p + j] = (uint16_t)(c[j] | (mask[j] << 8));
    }
  }
#pragma unroll
  for (int i = 0; i < WORDS; i++) {
    uint64_t *out = J.desc + (size_t)i * n;
    if (whole && ((uintptr_t)out & 15) == 0) {
      uint4 *to = reinterpret_cast<uint4 *>(out + p);
      to[0] = make_uint4(d[0][2 * i], d[0][2 * i + 1], d[1][2 * i], d[1][2 * i + 1]);
      to[1] = make_uint4(d[2][2 * i], d[2][2 * i + 1], d[3][2 * i], d[3][2 * i + 1]);
    } else {
#pragma unroll
      for (int j = 0; j < kCensusPx; j++)
        if (j < count) out[p + j] = (uint64_t)d[j][2 * i] | ((uint64_t)d[j][2 * i + 1] << 32);
    }
  }
  if (SUMS && J.wsum) {
#pragma unroll
    for (int j = 0; j < kCensusPx; j++)
      if (j < count) {
        J.wsum[p + j] = s1[j];
        J.wsum2[p + j] = s2[j];
      }
  }
}

int launch_census(sgm_context *ctx, const CensusJobs &jobs, int njobs, int w, int h,
                  const sgm_params *p) {
  ProfileScope ps(ctx, "census");
  const dim3 grid((w + kCensusW - 1) / kCensusW, (h + kCensusH - 1) / kCensusH, njobs);
  bool sums = false;
  for (int i = 0; i < njobs; i++) sums |= jobs.job[i].wsum != nullptr;
#define CASE(A, B)                                                             \
  if (p->window_w == A && p->window_h == B) {                                  \
    if (sums) census_kernel<A, B, true><<<grid, 256, 0, ctx->stream>>>(jobs);  \
    else census_kernel<A, B, false><<<grid, 256, 0, ctx->stream>>>(jobs);      \
    return launch_check("census kernel");                                      \
  }
#define ROW(A) CASE(A, 3) CASE(A, 5) CASE(A, 7) CASE(A, 9) CASE(A, 11)
  ROW(3) ROW(5) ROW(7) ROW(9) ROW(11)
#undef ROW
#undef CASE
  return fail(SGM_ERR_INVALID_ARGUMENT, "no census kernel for a %dx%d window", p->window_w,
              p->window_h);
}

}  // namespace sgm
