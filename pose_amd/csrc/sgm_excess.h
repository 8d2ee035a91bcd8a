// Path sweeps over excess planes, several scan lines per wave.
//
// The path cost of a cell is its matching cost plus an excess,
//   L_r(p, k) = C(p, k) + e_r(p, k),
//   e_r(p, k) = min(L_r(p-r, k), L_r(p-r, k+-1) + P1, min_k L_r(p-r, k) + P2') - min_k L_r(p-r, k),
// with 0 <= e_r <= P2' <= P2 (edge-adaptive P2', 0 where the path starts).  So
// wherever P2 <= 255 a direction's whole contribution to the aggregate
//   S(p, k) = P * C(p, k) + sum_r e_r(p, k)
// is one byte per cell, for any matching cost: excess_kernel stores e_r of
// every direction in plane r (plane k of pixel p: the Dp bytes at
// (planes * p + k) * Dp), and winner_kernel adds the planes and selects.  The
// directions only read C, so one launch carries all of them, and the winner
// search has no recurrence: it runs at streaming speed over independent pixels.
//
// Wave shape.  A line takes LANES = 16, 32 or 64 lanes of R disparities, so a
// wave sweeps 64 / LANES neighbouring lines.  A step's fixed part (wave minimum,
// neighbour lanes, penalty) then serves up to four lines, and the minimum over
// 16 lanes is four DPP steps that leave the result in every lane: no scalar
// round trip.  VALU instructions per line and pixel step of one direction (from
// the assembly): 53 with one line per wave and a lane group of 4, 23 here at
// 256 disparities; 45 and 8 at 64.
//
// Measured against one launch per seven directions and a fused last sweep with
// one line per wave (both matching directions, census 9x7; cost and census kernels
// of that time on both sides): 640x480 D=64
// 653 -> 304 us a pair, 1600x1067 D=256 4.03 -> 3.11 ms with pair sweeps (4.24
// with one plane per path: at that size HBM traffic decides, 26 or 19 bytes per
// cell), 2901x2175 D=350 24.7 -> 18.6 ms; FP32 ZNCC 1600x1067 D=192 against
// paired aggregates 7.24 -> 5.31 ms.
//
// A dword of four cells c0..c3 is held as the packed pairs E = (c0, c2) and
// O = (c1, c3), which cost one instruction each to take out of bytes and one
// to put back; the neighbours k+-1 of an E pair are O pairs and the reverse.
// Packed minima of three come from v_pk_minimum3_f16: all values are
// non-negative and below 0x7C00, where the order of half floats is that of
// their bits (subnormals are kept: the kernels run in the default f16 mode).
//
// Volume codes of this schedule: an invalid cell holds 254 (uint8) or 0x8800
// (uint16), a pad cell (k >= D) 255 or 0x8FFF.  Widened, invalid cells enter
// the recurrence as the reference's 512 (2048), pads as 771 (4095): more than
// the largest minimum (512, 2048) plus P2, so pads never win a minimum and need
// no mask.
#pragma once

namespace sgm {

constexpr int kMaxExcessDirs = 8;
constexpr uint32_t kExcessInf = 0x70007000u;
// buffer range of the excess sweeps' accesses and the offset of a dropped one
// (further planes and row tails lie behind it, below 2^31)
constexpr uint32_t kExcessRange = 0x7F000000u;
constexpr int kExcessDrop = 0x7F000000;

// Lanes per line and disparities per lane for a padded row of Dp cells (Dp a
// multiple of 64, at most 1024); false: no shape.  R divides Dp, so a lane lies
// wholly inside the row or wholly past it.
inline bool excess_shape(int Dp, int &lanes, int &R) {
  static const int8_t lanes_of[17] = {0,  16, 16, 16, 16, 16, 32, 32, 32,
                                      64, 32, 64, 64, 64, 64, 64, 64};
  static const int8_t R_of[17] = {0, 4, 8, 12, 16, 20, 12, 16, 16, 12, 20, 16, 12, 16, 16, 16, 16};
  const int u = Dp / 64;
  if (u < 1 || u > 16 || Dp % 64) return false;
  lanes = lanes_of[u];
  R = R_of[u];
  return true;
}

// The same with more lanes of fewer cells, for single planes of long images: a step of
// a line is sooner done (0.18 against 0.28 us at 256 disparities), for more
// instructions a cell.
// false: none for these rows, lanes and R stay.
inline bool narrow_shape(int Dp, int &lanes, int &R) {
  const int u = Dp / 64;
  if (u < 2 || u > 8) return false;
  lanes = u == 2 ? 32 : 64;
  R = u <= 4 ? 4 : 8;
  return true;
}

struct ExcessArgs {
  int ndirs, total;      // directions (or pairs), wave slots over all of them
  int planes;            // plane rows per pixel
  int pairs;             // each entry sweeps a direction and its opposite
  int narrow;            // narrow_shape
  int p1, p2, edge;
  int njobs;
  int dx[kMaxExcessDirs], dy[kMaxExcessDirs], begin[kMaxExcessDirs];
  int split[kMaxExcessDirs];  // two by-value jobs: waves of job 0
  // jobs in a device table: first wave of each job by line class
  const int *wave_begin[3];
  const int *order;      // dispatch order of the wave slots (optional)
};

struct WinnerArgs {
  int paths;             // directions summed in the planes
  double uniq;
};

// The volumes and sizes of a job as wave-uniform values (a job picked from
// either argument space comes through vector loads).
struct ExcessJob {
  const uint8_t *cost;
  uint8_t *planes;
  const uint16_t *gm;
  int w, h, Dp;
};
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }
template <typename T>
__device__ __forceinline__ T *uniform(T *p) {
  const uint64_t v = (uint64_t)p;
  return (T *)(((uint64_t)(uint32_t)uniform((int)(uint32_t)(v >> 32)) << 32) |
               (uint32_t)uniform((int)(uint32_t)v));
}
__device__ __forceinline__ ExcessJob excess_job(const PathJob &J) {
  return {uniform((const uint8_t *)J.cost), uniform((uint8_t *)J.sum), uniform(J.gm), uniform(J.w),
          uniform(J.h), uniform(J.Dp)};
}

template <int N, int POL>
__device__ __forceinline__ void bload_dwords(uint32_t *dst, __amdgpu_buffer_rsrc_t r, int off) {
  if constexpr (N == 1) {
    dst[0] = __builtin_amdgcn_raw_buffer_load_b32(r, off, 0, POL);
  } else if constexpr (N == 2) {
    const v2u32 t = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, POL);
    dst[0] = t.x;
    dst[1] = t.y;
  } else if constexpr (N == 3) {
    const v3u32 t = __builtin_amdgcn_raw_buffer_load_b96(r, off, 0, POL);
    dst[0] = t.x;
    dst[1] = t.y;
    dst[2] = t.z;
  } else {
    const v4u32 t = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, POL);
    dst[0] = t.x;
    dst[1] = t.y;
    dst[2] = t.z;
    dst[3] = t.w;
    if constexpr (N > 4) bload_dwords<N - 4, POL>(dst + 4, r, off + 16);
  }
}

template <int N, int POL>
__device__ __forceinline__ void bstore_dwords(const uint32_t *src, __amdgpu_buffer_rsrc_t r,
                                              int off) {
  if constexpr (N == 1) {
    __builtin_amdgcn_raw_buffer_store_b32(src[0], r, off, 0, POL);
  } else if constexpr (N == 2) {
    __builtin_amdgcn_raw_buffer_store_b64(v2u32{src[0], src[1]}, r, off, 0, POL);
  } else if constexpr (N == 3) {
    __builtin_amdgcn_raw_buffer_store_b96(v3u32{src[0], src[1], src[2]}, r, off, 0, POL);
  } else {
    __builtin_amdgcn_raw_buffer_store_b128(v4u32{src[0], src[1], src[2], src[3]}, r, off, 0, POL);
    if constexpr (N > 4) bstore_dwords<N - 4, POL>(src + 4, r, off + 16);
  }
}

// A lane's R bytes of a plane row of LANES * R: at l * R, but 20 bytes take two
// accesses, which side by side would each cover parts of every 64-byte granule, so
// there the row holds the first 16 bytes of all lanes and then their last 4.
// 2000x1400 D=320, 20 bytes side by side against this: a plane per path 10.6 -> 6.1
// ms and its winner search 3.2 -> 2.5, a plane per pair 5.9 -> 5.2 and 1.8 -> 1.5.
template <int LANES, int R>
struct PlaneRow {
  static constexpr bool SPLIT = R == 20;
  static constexpr int ND = R / 4, HEAD = SPLIT ? 4 : ND;
  static __device__ __forceinline__ int head(int l) { return l * HEAD * 4; }
  // bytes from the head to the tail
  static __device__ __forceinline__ int tail(int l) { return SPLIT ? (LANES - l) * 16 + l * 4 : 0; }
  template <int POL>
  static __device__ __forceinline__ void load(uint32_t *dst, __amdgpu_buffer_rsrc_t r, int off,
                                              int tail) {
    bload_dwords<HEAD, POL>(dst, r, off);
    if constexpr (SPLIT) bload_dwords<1, POL>(dst + 4, r, off + tail);
  }
  template <int POL>
  static __device__ __forceinline__ void store(const uint32_t *src, __amdgpu_buffer_rsrc_t r,
                                               int off, int tail) {
    bstore_dwords<HEAD, POL>(src, r, off);
    if constexpr (SPLIT) bstore_dwords<1, POL>(src + 4, r, off + tail);
  }
};

// Minimum of three packed pairs; every half non-negative and below 0x7C00.
__device__ __forceinline__ uint32_t pk_min3(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_pk_minimum3_f16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
  return r;
}
// a * b + c on packed uint16, modulo 2^16 or saturating; b is uniform.
__device__ __forceinline__ uint32_t pk_mad(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_pk_mad_u16 %0, %1, %2, %3" : "=v"(r) : "v"(a), "s"(b), "v"(c));
  return r;
}
__device__ __forceinline__ uint32_t pk_mad_sat(uint32_t a, uint32_t b, uint32_t c) {
  uint32_t r;
  asm("v_pk_mad_u16 %0, %1, %2, %3 clamp" : "=v"(r) : "v"(a), "s"(b), "v"(c));
  return r;
}
__device__ __forceinline__ uint32_t pk_sub_sat(uint32_t a, uint32_t b) {
  return as_u32(__builtin_elementwise_sub_sat(as_pk(a), as_pk(b)));
}
// Bytes 1 and 3 of a dword as a packed pair (bytes 0 and 2: & 0x00FF00FF).
__device__ __forceinline__ uint32_t odd_bytes(uint32_t v) {
  return as_u32(as_pk(v) >> (unsigned short)8);
}

// Lane l <- lane l-1 / l+1 of the same line; the first / last lane of a line
// takes `fill`.
template <int LANES>
__device__ __forceinline__ uint32_t line_shr1(uint32_t v, uint32_t fill, bool first) {
  if constexpr (LANES == 16)
    return (uint32_t)__builtin_amdgcn_update_dpp((int)fill, (int)v, 0x111, 0xF, 0xF, false);
  const uint32_t t = (uint32_t)dpp_shr1((int)v, (int)fill);
  return LANES == 64 ? t : first ? fill : t;
}
template <int LANES>
__device__ __forceinline__ uint32_t line_shl1(uint32_t v, uint32_t fill, bool last) {
  if constexpr (LANES == 16)
    return (uint32_t)__builtin_amdgcn_update_dpp((int)fill, (int)v, 0x101, 0xF, 0xF, false);
  const uint32_t t = (uint32_t)dpp_shl1((int)v, (int)fill);
  return LANES == 64 ? t : last ? fill : t;
}

// Unsigned minimum over the lanes of each line, left in all of them.
template <int LANES>
__device__ __forceinline__ uint32_t line_min(uint32_t v) {
#define SGM_LINE_MIN(ctrl) \
  v = min(v, (uint32_t)__builtin_amdgcn_update_dpp(-1, (int)v, ctrl, 0xF, 0xF, false));
  SGM_LINE_MIN(0xB1)
  SGM_LINE_MIN(0x4E)
  SGM_LINE_MIN(0x141)
  SGM_LINE_MIN(0x140)
#undef SGM_LINE_MIN
  if constexpr (LANES >= 32) {
    const auto s = __builtin_amdgcn_permlane16_swap(v, v, false, false);
    v = min((uint32_t)s[0], (uint32_t)s[1]);
  }
  if constexpr (LANES == 64) {
    const auto s = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    v = min((uint32_t)s[0], (uint32_t)s[1]);
  }
  return v;
}
template <int LANES>
__device__ __forceinline__ uint32_t line_min_pk(uint32_t v) {
  return line_min<LANES>(min(v & 0xFFFFu, v >> 16));
}

// Lane j of each row of 16 lanes, in every lane of the row.
template <int J>
__device__ __forceinline__ uint32_t row_lane(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x150 + J, 0xF, 0xF, true);
}

// Costs of one lane's R cells: raw volume dwords to the pairs of the recurrence
// (E at 2 * i, O at 2 * i + 1 of dword i).  `beyond`: all ones in lanes past
// the padded row, whose loads return zero.
template <int LANES, int R, int CB>
__device__ __forceinline__ void excess_costs(const uint32_t *raw, uint32_t beyond, uint32_t *c) {
#pragma unroll
  for (int i = 0; i < R / 4; i++) {
    if constexpr (CB == 1) {
      const uint32_t v = LANES > 16 ? raw[i] | beyond : raw[i];
      const uint32_t e = v & 0x00FF00FFu, o = odd_bytes(v);
      // 254 -> 512, 255 -> 771: + 258 times the excess over 253
      c[2 * i] = pk_mad(pk_sub_sat(e, 0x00FD00FDu), 0x01020102u, e);
      c[2 * i + 1] = pk_mad(pk_sub_sat(o, 0x00FD00FDu), 0x01020102u, o);
    } else {
      const uint32_t lo = LANES > 16 ? raw[2 * i] | beyond : raw[2 * i];
      const uint32_t hi = LANES > 16 ? raw[2 * i + 1] | beyond : raw[2 * i + 1];
      c[2 * i] = __builtin_amdgcn_perm(hi, lo, 0x05040100u) & 0x0FFF0FFFu;
      c[2 * i + 1] = __builtin_amdgcn_perm(hi, lo, 0x07060302u) & 0x0FFF0FFFu;
    }
  }
}

// The path costs of one pixel of a line and their minimum (splat).
template <int R>
struct ExcessState {
  uint32_t L[R / 2], minpk;
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int i = 0; i < R / 2; i++) L[i] = 0u;
    minpk = 0u;
  }
  // min(L - min L, 255), and back from its bytes
  __device__ __forceinline__ void offsets(uint32_t *m) const {
#pragma unroll
    for (int i = 0; i < R / 2; i++) m[i] = pk_min(L[i] - minpk, 0x00FF00FFu);
  }
  __device__ __forceinline__ void restore(const uint32_t *bytes) {
#pragma unroll
    for (int d = 0; d < R / 4; d++) {
      L[2 * d] = bytes[d] & 0x00FF00FFu;
      L[2 * d + 1] = odd_bytes(bytes[d]);
    }
    minpk = 0u;
  }
};

// The same in 32 bits, cells in ascending order, for 32-bit aggregates: twice the
// arithmetic of the packed pairs, still HBM-bound over uint16 costs.  Eight paths
// of 1024x768 D=128, both matching directions, in pairs: 0.88 ms and the winner
// search 0.18, against 3.4 ms of sequential 32-bit sweeps.
template <int R>
struct WideState {
  int L[R], least;
  __device__ __forceinline__ void clear() {
#pragma unroll
    for (int j = 0; j < R; j++) L[j] = 0;
    least = 0;
  }
  __device__ __forceinline__ void offsets(uint32_t *m) const {
#pragma unroll
    for (int i = 0; i < R / 2; i++) {
      const int j = (i >> 1) * 4 + (i & 1);
      m[i] = (uint32_t)min(L[j] - least, 255) | ((uint32_t)min(L[j + 2] - least, 255) << 16);
    }
  }
  __device__ __forceinline__ void restore(const uint32_t *bytes) {
#pragma unroll
    for (int j = 0; j < R; j++) L[j] = (int)(bytes[j / 4] >> (j % 4 * 8) & 0xFFu);
    least = 0;
  }
};

// One pixel step: `c` the pixel's costs, `p2` its packed penalty P2' (0: the
// path starts here, every excess is 0).  Leaves the pixel's excesses in `e`.
template <int LANES, int R>
__device__ __forceinline__ void excess_step(ExcessState<R> &s, const uint32_t *c, uint32_t p2,
                                            uint32_t p1, bool first, bool last, uint32_t *e) {
  constexpr int ND = R / 4;
  const uint32_t mp2 = s.minpk + p2;
  uint32_t q[R / 2];
#pragma unroll
  for (int i = 0; i < R / 2; i++) q[i] = s.L[i] + p1;
  const uint32_t in_lo = line_shr1<LANES>(q[2 * ND - 1], kExcessInf, first);
  const uint32_t in_hi = line_shl1<LANES>(q[0], kExcessInf, last);
  uint32_t least[R / 2];
#pragma unroll
  for (int i = 0; i < ND; i++) {
    const uint32_t qe = q[2 * i], qo = q[2 * i + 1];
    const uint32_t below = __builtin_amdgcn_alignbit(qo, i ? q[2 * i - 1] : in_lo, 16);
    const uint32_t above = __builtin_amdgcn_alignbit(i + 1 < ND ? q[2 * i + 2] : in_hi, qe, 16);
    const uint32_t te = pk_min3(pk_min(s.L[2 * i], mp2), below, qo);
    const uint32_t to = pk_min3(pk_min(s.L[2 * i + 1], mp2), above, qe);
    e[2 * i] = te - s.minpk;
    e[2 * i + 1] = to - s.minpk;
  }
#pragma unroll
  for (int i = 0; i < R / 2; i++) {
    s.L[i] = c[i] + e[i];
    least[i] = s.L[i];
  }
#pragma unroll
  for (int n = R / 2; n > 1; n = (n + 2) / 3) {
#pragma unroll
    for (int i = 0; 3 * i < n; i++) {
      if (3 * i + 2 < n) least[i] = pk_min3(least[3 * i], least[3 * i + 1], least[3 * i + 2]);
      else if (3 * i + 1 < n) least[i] = pk_min(least[3 * i], least[3 * i + 1]);
      else least[i] = least[3 * i];
    }
  }
  const uint32_t m = line_min_pk<LANES>(least[0]);
  s.minpk = m | (m << 16);
}

template <int LANES, int R>
__device__ __forceinline__ void excess_step(WideState<R> &s, const uint32_t *c, uint32_t p2,
                                            uint32_t p1, bool first, bool last, uint32_t *e) {
  const int step = (int)(p1 & 0xFFFFu), cap = s.least + (int)(p2 & 0xFFFFu);
  const int below = (int)line_shr1<LANES>((uint32_t)s.L[R - 1], kExcessInf, first);
  const int above = (int)line_shl1<LANES>((uint32_t)s.L[0], kExcessInf, last);
  int x[R];
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int side = min(j ? s.L[j - 1] : below, j + 1 < R ? s.L[j + 1] : above) + step;
    x[j] = min(min(s.L[j], cap), side) - s.least;
  }
  int least = (int)kExcessInf;
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int i = (j >> 2) * 2 + (j & 1);
    s.L[j] = (int)(j & 2 ? c[i] >> 16 : c[i] & 0xFFFFu) + x[j];
    least = min(least, s.L[j]);
  }
#pragma unroll
  for (int i = 0; i < R / 2; i++) {
    const int j = (i >> 1) * 4 + (i & 1);
    e[i] = (uint32_t)x[j] | ((uint32_t)x[j + 2] << 16);
  }
  s.least = (int)line_min<LANES>((uint32_t)least);
}

// StereoCost.pathP2 for every |dI|, as a packed pair (P2 and the edge scale are
// at most 255, so 32 bits hold the product).
__device__ __forceinline__ void build_p2_pairs(uint32_t *tab, int p1, int p2, int edge) {
  for (int d = threadIdx.x; d < 256; d += 256) {
    int v = p2;
    if (edge != 0) v = max(p1 + 1, (int)((unsigned)(p2 * edge) / (unsigned)(edge + d)));
    tab[d] = (uint32_t)v | ((uint32_t)v << 16);
  }
}

// The 64 / LANES neighbouring lines of a wave: line0, line0 + 1, .. of direction
// (dx, dy), one per LANES lanes.  Rows of the wave are addressed from its lowest
// start pixel; a lane's offset in them is fixed along the line.
template <int LANES, int R, int CB, bool NT>
struct ExcessLines {
  static constexpr int ND = R / 4;
  static constexpr int POL = NT ? POL_NT : POL_DEFAULT;

  const ExcessJob J;
  const uint32_t *tab;
  int len, maxlen, minlen;      // this lane's line, longest and shortest of the wave
  int p0, step;                 // first pixel of this lane's line, pixels per step
  int coff, poff, ptail;        // this lane's offsets in the wave's cost / plane rows
  const uint8_t *crow;          // the wave's cost and plane rows of step 0
  uint8_t *prow;
  ptrdiff_t cstep, pstep;
  uint32_t p1pk, beyond;
  bool first, last;
  __amdgpu_buffer_rsrc_t gm;

  __device__ __forceinline__ ExcessLines(const ExcessJob &J_, const ExcessArgs &A, int dx, int dy,
                                         int line0, int plane, const uint32_t *tab_)
      : J(J_), tab(tab_) {
    const int lane = lane_id(), l = lane % LANES;
    const int line = line0 + lane / LANES;
    const int lines = dy == 0 ? J.h : dx == 0 ? J.w : J.w + J.h - 1;
    int x = 0, y = 0;
    len = 0;
    if (line < lines) line_start(line, dx, dy, J.w, J.h, x, y, len);
    p0 = y * J.w + x;
    step = dy * J.w + dx;
    int base = __builtin_amdgcn_readlane(p0, 0);
    maxlen = minlen = __builtin_amdgcn_readlane(len, 0);
#pragma unroll
    for (int g = 1; g < 64 / LANES; g++) {
      const int n = __builtin_amdgcn_readlane(len, g * LANES);
      if (n > 0) base = min(base, __builtin_amdgcn_readlane(p0, g * LANES));
      maxlen = max(maxlen, n);
      minlen = min(minlen, n);
    }
    const int rel = len > 0 ? p0 - base : 0;
    const bool inside = l * R < J.Dp;
    coff = inside ? (rel * J.Dp + l * R) * CB : kExcessDrop;
    poff = inside ? rel * A.planes * J.Dp + PlaneRow<LANES, R>::head(l) : kExcessDrop;
    ptail = PlaneRow<LANES, R>::tail(l);
    cstep = (ptrdiff_t)step * J.Dp * CB;
    pstep = (ptrdiff_t)step * J.Dp * A.planes;
    crow = J.cost + (ptrdiff_t)base * J.Dp * CB;
    prow = J.planes + ((ptrdiff_t)base * A.planes + plane) * J.Dp;
    p1pk = splat16((uint32_t)A.p1);
    beyond = inside ? 0u : ~0u;
    first = l == 0;
    last = l == LANES - 1;
    gm = make_rsrc(J.gm, (uint32_t)J.w * (uint32_t)J.h * 2u);
  }

  __device__ __forceinline__ void load(uint32_t *dst, const uint8_t *row, bool in) const {
    bload_dwords<ND * CB, POL_DEFAULT>(dst, make_rsrc(row, kExcessRange), in ? coff : kExcessDrop);
  }
  __device__ __forceinline__ void store(const uint32_t *src, uint8_t *row, bool in) const {
    PlaneRow<LANES, R>::template store<POL>(src, make_rsrc(row, kExcessRange),
                                            in ? poff : kExcessDrop, ptail);
  }
  // gray | mask << 8 of the pixel of step s (0, an unusable pixel, off the line)
  __device__ __forceinline__ int pixel(int s) const {
    return s >= 0 && s < len
               ? (int)__builtin_amdgcn_raw_buffer_load_b16(gm, (p0 + s * step) * 2, 0, 0)
               : 0;
  }
  // packed P2' of a step from pixel `gp` to pixel `g`
  __device__ __forceinline__ uint32_t penalty(int g, int gp) const {
    const uint32_t v = tab[abs((g & 0xFF) - (gp & 0xFF))];
    return (gp >> 8) ? v : 0u;
  }
  template <class State>
  __device__ __forceinline__ void advance(State &s, const uint32_t *c, uint32_t p2,
                                          uint32_t *e) const {
    excess_step<LANES, R>(s, c, p2, p1pk, first, last, e);
  }
};

template <int R>
__device__ __forceinline__ void excess_bytes(const uint32_t *e, uint32_t *out) {
#pragma unroll
  for (int i = 0; i < R / 4; i++) out[i] = e[2 * i] | (e[2 * i + 1] << 8);
}

// One direction per line, excesses to plane `plane`.  The costs of W steps
// ahead are in flight.
template <int LANES, int R, int CB, bool NT, class State>
struct ExcessSweep : ExcessLines<LANES, R, CB, NT> {
  using Base = ExcessLines<LANES, R, CB, NT>;
  using Base::Base;
  using Base::ND;
  static constexpr int W = R * CB <= 8 ? 16 : 8;

  const uint8_t *ld;            // wave row of the next loaded step
  uint8_t *st;                  // wave row of the next stored step
  uint32_t cb[W][ND * CB];
  uint32_t meta;                // packed P2' of step (lane % W) of the window
  State state;

  template <bool MASKED, int JJ>
  __device__ __forceinline__ void one(int s) {
    uint32_t c[R / 2], e[R / 2], out[ND];
    excess_costs<LANES, R, CB>(cb[JJ], this->beyond, c);
    this->load(cb[JJ], ld, !MASKED || s + W < this->len);
    ld += this->cstep;
    this->advance(state, c, row_lane<JJ>(meta), e);
    excess_bytes<R>(e, out);
    this->store(out, st, !MASKED || s < this->len);
    st += this->pstep;
  }

  template <bool MASKED, int... JJ>
  __device__ __forceinline__ void window(int w0, std::integer_sequence<int, JJ...>) {
    const int s = w0 + W + lane_id() % W;
    const int g = this->pixel(s), gp = this->pixel(s - 1);
    (one<MASKED, JJ>(w0 + JJ), ...);
    meta = this->penalty(g, gp);
  }

  __device__ __forceinline__ void run() {
    const int s = lane_id() % W;
    const int g = this->pixel(s), gp = this->pixel(s - 1);
    ld = this->crow;
    st = this->prow;
#pragma unroll
    for (int j = 0; j < W; j++) {
      this->load(cb[j], ld, j < this->len);
      ld += this->cstep;
    }
    meta = this->penalty(g, gp);
    state.clear();
    int w0 = 0;
    // every line of the wave covers the window and the loads ahead of it
    for (; w0 + 2 * W <= this->minlen; w0 += W)
      window<false>(w0, std::make_integer_sequence<int, W>());
    for (; w0 < this->maxlen; w0 += W) window<true>(w0, std::make_integer_sequence<int, W>());
  }
};

// Both directions of a line, the sum of their excesses to plane `plane`
// (2 * P2 <= 255): half the planes, so 3.25 bytes of traffic per cell and pair
// where two single sweeps and the winner search move 4 and read one plane
// more.  The forward direction is swept twice: first only for its state at
// the start of every segment of SEG steps, then segment by segment from the
// line's end, its excesses in registers, right before the backward direction
// takes the same segment.  A state is kept as bytes min(L - min L, 255), which
// is all the recurrence can tell apart when P2 <= 255; it lies in the plane row
// of the segment's first pixel until the sums overwrite it.
template <int LANES, int R, int CB, bool NT, class State>
struct PairSweep : ExcessLines<LANES, R, CB, NT> {
  using Base = ExcessLines<LANES, R, CB, NT>;
  using Base::Base;
  using Base::ND;
  static constexpr int SEG = R * CB <= 16 ? 8 : 4;

  const uint8_t *ld;
  uint8_t *st;
  uint32_t cb[SEG][ND * CB], ef[SEG][ND];
  uint32_t mf, mb;              // packed P2' of step (lane % SEG), forward and backward
  State fwd, bwd;

  __device__ __forceinline__ void keep_state(bool in) {
    uint32_t m[R / 2], out[ND];
    fwd.offsets(m);
    excess_bytes<R>(m, out);
    this->store(out, st, in);
  }

  __device__ __forceinline__ void keep_load(uint32_t *kept, bool in) const {
    PlaneRow<LANES, R>::template load<POL_DEFAULT>(kept, make_rsrc(st, kExcessRange),
                                                   in ? this->poff : kExcessDrop, this->ptail);
  }

  template <int JJ>
  __device__ __forceinline__ void ahead(int s) {
    uint32_t c[R / 2], e[R / 2];
    excess_costs<LANES, R, CB>(cb[JJ], this->beyond, c);
    this->load(cb[JJ], ld, s + SEG < this->len);
    ld += this->cstep;
    this->advance(fwd, c, row_lane<JJ>(mf), e);
  }
  template <int JJ>
  __device__ __forceinline__ void again() {
    uint32_t c[R / 2], e[R / 2];
    excess_costs<LANES, R, CB>(cb[JJ], this->beyond, c);
    this->advance(fwd, c, row_lane<JJ>(mf), e);
    excess_bytes<R>(e, ef[JJ]);
  }
  template <int JJ>
  __device__ __forceinline__ void back(int s) {
    uint32_t c[R / 2], e[R / 2], out[ND];
    excess_costs<LANES, R, CB>(cb[JJ], this->beyond, c);
    this->load(cb[JJ], ld, s >= SEG && s - SEG < this->len);
    ld -= this->cstep;
    this->advance(bwd, c, row_lane<JJ>(mb), e);
    excess_bytes<R>(e, out);
#pragma unroll
    for (int i = 0; i < ND; i++) out[i] += ef[JJ][i];
    this->store(out, st, s < this->len);
    st -= this->pstep;
  }
  template <int... JJ>
  __device__ __forceinline__ void all_ahead(int s0, std::integer_sequence<int, JJ...>) {
    (ahead<JJ>(s0 + JJ), ...);
  }
  template <int... JJ>
  __device__ __forceinline__ void all_again(std::integer_sequence<int, JJ...>) {
    (again<JJ>(), ...);
  }
  template <int... JJ>
  __device__ __forceinline__ void all_back(int s0, std::integer_sequence<int, JJ...>) {
    (back<SEG - 1 - JJ>(s0 + SEG - 1 - JJ), ...);
  }

  __device__ __forceinline__ void run() {
    using Steps = std::make_integer_sequence<int, SEG>;
    const int nseg = (this->maxlen + SEG - 1) / SEG;
    const int i = lane_id() % SEG;
    // forward, for the states at the segment starts (segment 0 starts the path)
    ld = this->crow;
#pragma unroll
    for (int j = 0; j < SEG; j++) {
      this->load(cb[j], ld, j < this->len);
      ld += this->cstep;
    }
    mf = this->penalty(this->pixel(i), this->pixel(i - 1));
    fwd.clear();
    st = this->prow;
    for (int k = 0; k + 1 < nseg; k++) {
      const int s = (k + 1) * SEG + i;
      const int g = this->pixel(s), gp = this->pixel(s - 1);
      all_ahead(k * SEG, Steps());
      mf = this->penalty(g, gp);
      st += SEG * this->pstep;
      keep_state((k + 1) * SEG < this->len);
    }
    // the slots hold the last segment's costs
    bwd.clear();
    int s0 = (nseg - 1) * SEG;
    int g = this->pixel(s0 + i), gp = this->pixel(s0 + i - 1), gn = this->pixel(s0 + i + 1);
    ld = this->crow + (ptrdiff_t)(s0 - 1) * this->cstep;
    uint32_t kept[ND];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the kept states are in memory
    keep_load(kept, s0 < this->len);
    for (; s0 >= 0; s0 -= SEG) {
      mf = this->penalty(g, gp);
      mb = this->penalty(g, gn);
      // (lanes past the padded row keep no bytes: a pad's, not the minimum's)
      if constexpr (LANES > 16) {
#pragma unroll
        for (int i = 0; i < ND; i++) kept[i] |= this->beyond;
      }
      fwd.restore(kept);
      // the next segment's state and pixels, one segment ahead
      st = this->prow + (ptrdiff_t)(s0 - SEG) * this->pstep;
      keep_load(kept, s0 >= SEG && s0 - SEG < this->len);
      const int s = s0 - SEG + i;
      g = this->pixel(s);
      gp = this->pixel(s - 1);
      gn = this->pixel(s + 1);
      all_again(Steps());
      st = this->prow + (ptrdiff_t)(s0 + SEG - 1) * this->pstep;
      all_back(s0, Steps());
    }
  }
};

// All directions of all jobs (two by value or a device table), one wave per 64 / LANES
// lines.  HBM-bound at large volumes (2 bytes per cell and direction), bound
// by the recurrence's instructions where the volumes fit the caches.
// WIDE: path costs in 32 bits.
template <int LANES, int R, int CB, bool PAIR, bool NT, bool WIDE>
__global__ __launch_bounds__(256) void excess_kernel(PathJobs jobs, ExcessArgs A) {
  __shared__ uint32_t tab[256];
  build_p2_pairs(tab, A.p1, A.p2, A.edge);
  __syncthreads();
  const int slot = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) +
                                                  (int)(threadIdx.x >> 6));
  if (slot >= A.total) return;
  const int wave = A.order ? __builtin_amdgcn_readfirstlane(A.order[slot]) : slot;
  int k = 0, dx = A.dx[0], dy = A.dy[0], begin = A.begin[0], split = A.split[0];
#pragma unroll
  for (int i = 1; i < kMaxExcessDirs; i++) {
    if (i < A.ndirs && wave >= A.begin[i]) {
      k = i;
      dx = A.dx[i];
      dy = A.dy[i];
      begin = A.begin[i];
      split = A.split[i];
    }
  }
  int local = wave - begin, ji = 0;
  if (jobs.table) {
    const int *wb = dy == 0 ? A.wave_begin[0] : dx == 0 ? A.wave_begin[1] : A.wave_begin[2];
    ji = __builtin_amdgcn_readfirstlane(find_job(wb, A.njobs, local));
    local -= wb[ji];
  } else if (A.njobs > 1 && local >= split) {
    ji = 1;
    local -= split;
  }
  const ExcessJob J = excess_job(jobs.table ? jobs.table[ji] : jobs.local[ji & 1]);
  using State = std::conditional_t<WIDE, WideState<R>, ExcessState<R>>;
  if constexpr (PAIR)
    PairSweep<LANES, R, CB, NT, State>(J, A, dx, dy, local * (64 / LANES), k, tab).run();
  else
    ExcessSweep<LANES, R, CB, NT, State>(J, A, dx, dy, local * (64 / LANES), k, tab).run();
}

// ---------------------------------------------------------------------------
// Winner search over the planes: S = paths * C + sum of NPL planes, then the
// winner, runner-up, neighbours and selection of CensusSgm.java:460-515.  One
// wave per 64 pixels of a row, 64 / LANES pixels at a time; the pixels' summaries are
// collected in LDS and selected 64 at once (select_flush).
// G: planes added bytewise before they are widened (their largest sum fits a
// byte).
template <int LANES, int R, int CB, int NPL, int G, bool NT>
struct WinnerSearch {
  static constexpr int ND = R / 4, NL = 64 / LANES;
  static constexpr int POL = NT ? POL_NT : POL_DEFAULT;
  struct Row {
    uint32_t c[ND * CB], pl[NPL][ND];
  };

  static __device__ __forceinline__ void load(Row &r, const uint8_t *cost, const uint8_t *planes,
                                              int coff, int poff, int tail, int Dp) {
    bload_dwords<ND * CB, POL>(r.c, make_rsrc(cost, kExcessRange), coff);
    const __amdgpu_buffer_rsrc_t rs = make_rsrc(planes, kExcessRange);
#pragma unroll
    for (int k = 0; k < NPL; k++)
      PlaneRow<LANES, R>::template load<POL>(r.pl[k], rs, poff + k * Dp, tail);
  }

  // Aggregates of one lane's cells, invalid and pad cells 0xFFFF.
  static __device__ __forceinline__ void sums(const Row &r, uint32_t beyond, uint32_t paths,
                                              uint32_t *S) {
#pragma unroll
    for (int i = 0; i < ND; i++) {
      uint32_t e = 0, o = 0;
#pragma unroll
      for (int k = 0; k < NPL; k += G) {
        uint32_t v = r.pl[k][i];
#pragma unroll
        for (int j = 1; j < G; j++) v += r.pl[k + j][i];
        e += v & 0x00FF00FFu;
        o += odd_bytes(v);
      }
      uint32_t ce, co, me, mo;  // costs, and non-zero where the cell is not valid
      if constexpr (CB == 1) {
        const uint32_t v = LANES > 16 ? r.c[i] | beyond : r.c[i];
        ce = v & 0x00FF00FFu;
        co = odd_bytes(v);
        me = pk_sub_sat(ce, 0x00FD00FDu);
        mo = pk_sub_sat(co, 0x00FD00FDu);
      } else {
        const uint32_t lo = LANES > 16 ? r.c[2 * i] | beyond : r.c[2 * i];
        const uint32_t hi = LANES > 16 ? r.c[2 * i + 1] | beyond : r.c[2 * i + 1];
        ce = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
        co = __builtin_amdgcn_perm(hi, lo, 0x07060302u);
        me = pk_sub_sat(ce, 0x7FFF7FFFu);
        mo = pk_sub_sat(co, 0x7FFF7FFFu);
      }
      S[2 * i] = pk_mad_sat(me, ~0u, pk_mad(ce, paths, e));
      S[2 * i + 1] = pk_mad_sat(mo, ~0u, pk_mad(co, paths, o));
    }
  }

  static __device__ __forceinline__ uint32_t least(const uint32_t *v) {
    uint32_t m = v[0];
#pragma unroll
    for (int i = 1; i < R / 2; i++) m = pk_min(m, v[i]);
    return line_min_pk<LANES>(m);
  }

  // Byte of cell k of a line's pixel in the wave's aggregate rows in LDS.
  static __device__ __forceinline__ int cell_byte(int k) {
    return (k & ~3) * 2 + (k & 1) * 4 + (k & 2);
  }
};

constexpr int kWinnerPixels = 64;  // pixels per wave of the winner search
constexpr int kWinnerWaves = 4;

template <int LANES, int R, int CB, int NPL, int G, bool NT>
__global__ __launch_bounds__(64 * kWinnerWaves) void winner_kernel(PathJobs jobs, WinnerArgs A,
                                                                   int job0) {
  using WS = WinnerSearch<LANES, R, CB, NPL, G, NT>;
  constexpr int NL = 64 / LANES, NP = R / 2;
  __shared__ __align__(16) uint8_t cells[kWinnerWaves][64 * R * 2];
  __shared__ uint32_t found[kWinnerWaves][3][kWinnerPixels];
  const int wv = threadIdx.x >> 6;
  const int ji = job0 + (int)blockIdx.z;
  const PathJob J = jobs.table ? jobs.table[ji] : jobs.local[ji & 1];
  const ExcessJob V = excess_job(J);
  const int y = blockIdx.y;
  const int x0 = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWinnerWaves + wv) * kWinnerPixels);
  if (y >= V.h || x0 >= V.w) return;
  const int count = min(kWinnerPixels, V.w - x0);
  const int lane = lane_id(), g = lane / LANES, l = lane % LANES;
  const int Dp = V.Dp, D = J.D;
  const bool inside = l * R < Dp;
  const uint32_t beyond = inside ? 0u : ~0u, paths = splat16((uint32_t)A.paths);
  const uint8_t *cost = V.cost + ((size_t)y * V.w + x0) * Dp * CB;
  const uint8_t *planes = V.planes + ((size_t)y * V.w + x0) * Dp * NPL;
  const int coff = inside ? (g * Dp + l * R) * CB : kExcessDrop;
  const int poff = inside ? g * NPL * Dp + PlaneRow<LANES, R>::head(l) : kExcessDrop;
  const int tail = PlaneRow<LANES, R>::tail(l);
  uint32_t kpk[NP];
#pragma unroll
  for (int i = 0; i < NP; i++) {
    const int k = l * R + (i >> 1) * 4 + (i & 1);
    kpk[i] = (uint32_t)k | ((uint32_t)(k + 2) << 16);
  }
  uint8_t *row = cells[wv];
  const int own = lane * R * 2, line = g * LANES * R * 2;
  typename WS::Row cur;
  WS::load(cur, cost, planes, g < count ? coff : kExcessDrop, g < count ? poff : kExcessDrop, tail,
           Dp);
  for (int i = 0; i < count; i += NL) {
    uint32_t S[NP];
    WS::sums(cur, beyond, paths, S);
    cost += NL * Dp * CB;
    planes += NL * Dp * NPL;
    const bool next = i + NL + g < count;
    WS::load(cur, cost, planes, next ? coff : kExcessDrop, next ? poff : kExcessDrop, tail, Dp);
#pragma unroll
    for (int j = 0; j < NP; j += 2)
      *reinterpret_cast<uint2 *>(row + own + 4 * j) = make_uint2(S[j], S[j + 1]);
    const uint32_t value = WS::least(S), vpk = value | (value << 16);
    uint32_t t[NP];
#pragma unroll
    for (int j = 0; j < NP; j++) t[j] = pk_mad_sat(pk_sub(S[j], vpk), ~0u, kpk[j]);
    const uint32_t best = WS::least(t);  // the first k of the smallest aggregate
    const uint32_t bm1 = splat16(best - 1u);
#pragma unroll
    for (int j = 0; j < NP; j++)  // cells within one of the winner: 0xFFFF
      t[j] = pk_mad_sat(pk_sub_sat(0x00030003u, pk_sub(kpk[j], bm1)), ~0u, S[j]);
    const uint32_t second = WS::least(t);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (l == 0) {
      const bool any = value != 0xFFFFu;
      const int b = (int)best;
      auto at = [&](int k) {
        return (uint32_t)*reinterpret_cast<const uint16_t *>(row + line + WS::cell_byte(k));
      };
      uint32_t f0 = 0u, f1 = 0u, f2 = 0xFFFFFFFFu;
      if (any) {
        const uint32_t before = b > 0 ? at(b - 1) : 0xFFFFu;
        const uint32_t after = b + 1 < D ? at(b + 1) : 0xFFFFu;
        const uint32_t flags = (at(0) != 0xFFFFu ? 1u : 0u) | (at(D - 1) != 0xFFFFu ? 2u : 0u);
        f0 = (uint32_t)(b + 1) | (flags << 13);
        f1 = value | (second << 16);
        f2 = before | (after << 16);
      }
      found[wv][0][i + g] = f0;
      found[wv][1][i + g] = f1;
      found[wv][2][i + g] = f2;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  DeferredPk d{0u, 0u, 0u};
  d.f0 = found[wv][0][lane];
  d.f1 = found[wv][1][lane];
  d.f2 = found[wv][2][lane];
  PathArgs P;
  P.dx = 1;
  P.dy = 0;
  P.uniq = A.uniq;
  select_flush(make_flush_args(J, P), d.view(), count, 0, x0, y);
}

// The same over four planes and uint16 costs with the aggregates in 32 bits.
// HBM-bound: 6 bytes per cell.
template <int LANES, int R, bool NT>
__global__ __launch_bounds__(64 * kWinnerWaves) void winner32_kernel(PathJobs jobs, WinnerArgs A) {
  using WS = WinnerSearch<LANES, R, 2, 4, 1, NT>;
  constexpr int NL = 64 / LANES;
  constexpr uint32_t none = 0x7FFFFFFFu;
  __shared__ __align__(16) uint32_t cells[kWinnerWaves][64 * R];
  __shared__ int found[kWinnerWaves][6][kWinnerPixels];
  const int wv = threadIdx.x >> 6;
  const PathJob J = jobs.local[blockIdx.z & 1];
  const ExcessJob V = excess_job(J);
  const int y = blockIdx.y;
  const int x0 = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * kWinnerWaves + wv) * kWinnerPixels);
  if (y >= V.h || x0 >= V.w) return;
  const int count = min(kWinnerPixels, V.w - x0);
  const int lane = lane_id(), g = lane / LANES, l = lane % LANES;
  const int Dp = V.Dp, D = J.D;
  const bool inside = l * R < Dp;
  const uint32_t beyond = inside ? 0u : ~0u;
  const uint8_t *cost = V.cost + ((size_t)y * V.w + x0) * Dp * 2;
  const uint8_t *planes = V.planes + ((size_t)y * V.w + x0) * Dp * 4;
  const int coff = inside ? (g * Dp + l * R) * 2 : kExcessDrop;
  const int poff = inside ? g * 4 * Dp + PlaneRow<LANES, R>::head(l) : kExcessDrop;
  const int tail = PlaneRow<LANES, R>::tail(l);
  uint32_t *own = cells[wv] + lane * R;
  const uint32_t *line = cells[wv] + g * LANES * R;
  typename WS::Row cur;
  WS::load(cur, cost, planes, g < count ? coff : kExcessDrop, g < count ? poff : kExcessDrop, tail,
           Dp);
  for (int i = 0; i < count; i += NL) {
    uint32_t S[R];  // invalid and pad cells: none
    uint32_t value = none;
#pragma unroll
    for (int j = 0; j < R; j++) {
      const uint32_t raw = LANES > 16 ? cur.c[j / 2] | beyond : cur.c[j / 2];
      const uint32_t c = j % 2 ? raw >> 16 : raw & 0xFFFFu;
      uint32_t e = 0;
#pragma unroll
      for (int k = 0; k < 4; k++) e += cur.pl[k][j / 4] >> (j % 4 * 8) & 0xFFu;
      S[j] = c & 0x8000u ? none : (uint32_t)A.paths * c + e;
      value = min(value, S[j]);
    }
    cost += NL * Dp * 2;
    planes += NL * Dp * 4;
    const bool next = i + NL + g < count;
    WS::load(cur, cost, planes, next ? coff : kExcessDrop, next ? poff : kExcessDrop, tail, Dp);
#pragma unroll
    for (int j = 0; j < R; j += 4)
      *reinterpret_cast<uint4 *>(own + j) = make_uint4(S[j], S[j + 1], S[j + 2], S[j + 3]);
    value = line_min<LANES>(value);
    uint32_t best = none;  // the first k of the smallest aggregate
#pragma unroll
    for (int j = 0; j < R; j++) best = min(best, S[j] == value ? (uint32_t)(l * R + j) : none);
    best = line_min<LANES>(best);
    uint32_t second = none;  // beyond one of the winner
#pragma unroll
    for (int j = 0; j < R; j++)
      second = min(second, (uint32_t)(l * R + j) - best + 1u < 3u ? none : S[j]);
    second = line_min<LANES>(second);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (l == 0) {
      const bool any = value != none;
      const int b = any ? (int)best : -1;
      auto at = [&](int k) { return k >= 0 && k < D && line[k] != none ? (int)line[k] : -1; };
      int *f = &found[wv][0][i + g];
      f[0] = b;
      f[kWinnerPixels] = (int)value;
      f[2 * kWinnerPixels] = (int)second;
      f[3 * kWinnerPixels] = any ? at(b - 1) : -1;
      f[4 * kWinnerPixels] = any ? at(b + 1) : -1;
      f[5 * kWinnerPixels] = any ? (at(0) >= 0 ? 1 : 0) | (at(D - 1) >= 0 ? 2 : 0) : 0;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
  WinnerView v;
  v.best = found[wv][0][lane];
  v.value = found[wv][1][lane];
  v.second = found[wv][2][lane];
  v.before = found[wv][3][lane];
  v.after = found[wv][4][lane];
  v.flags = found[wv][5][lane];
  PathArgs P;
  P.dx = 1;
  P.dy = 0;
  P.uniq = A.uniq;
  select_flush(make_flush_args(J, P), v, count, 0, x0, y);
}

}  // namespace sgm
