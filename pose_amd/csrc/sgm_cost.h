// Cost volume of the census-family costs (StereoCost.value modes 0..2,
// StereoCost.java:50-74; validity test of the reference's `costs` kernel,
// GpuStereo.java:706-731), several row segments per wave.
//
// A row segment takes LANES lanes of R disparities (the shapes of sgm_excess.h),
// each lane holding its R target descriptors in registers.  One pixel step
// moves the targets by one column: every lane passes its end target to the
// next lane (DPP) and one new target enters, so a target is loaded once per
// segment.  A cell costs its Hamming distance (two instructions per 32 bits)
// and a quarter of the packing of four cells; whether the target is usable is a
// byte mask that slides with the targets and picks the invalid code with one
// v_bfi per four cells.  Bound by these instructions at small ranges, by the
// volume's HBM write at large ones.  Measured against one thread per four cells
// with its targets read from L2 (cost volume alone, both matching directions):
// AD-census 11x11 1201x801 D=97 754 -> 175 us, census 5x5 1200x900 D=700 2806 ->
// 479 us, uint16 census 9x7 1024x768 D=128 385 -> 85 us; against a sliding
// window with one segment per wave: census 9x7 640x480 D=64 45 -> 20 us,
// 1600x1067 D=256 302 -> 246 us, 2901x2175 D=350 1866 -> 1387 us (3.5 TB/s), with
// stores past the caches (where the sweeps' volumes exceed 1 GiB) 202 and 969 us;
// below that size the sweeps want the costs in them (640x480: 252 -> 284 us a pair).
// The 20 bytes of a lane at 16 x 20 and 32 x 20 take two stores that each cover parts
// of a 64-byte granule, so there the caches join them: 2000x1400 D=320 0.72 -> 0.60 ms.
#pragma once

namespace sgm {

struct BandArgs {
  int njobs, total;      // jobs, waves over all jobs
  int split;             // two by-value jobs: waves of job 0
  const int *wave_begin; // jobs in a device table: first wave of each job
  int seg;               // pixels per row segment
  int gradient;          // difference of the gray gradients instead of the grays
  int stream;            // volumes far beyond the caches: the stores pass them by
  // AD-census, census-gradient: value = (wa * ham + wb * min(difference, cap) + half) / den as
  // a multiplication by `magic` and a shift (band_division)
  uint32_t wa, wb, half, cap, magic;
  int shift;
  uint32_t inv, pad;     // stored codes of an invalid and of a pad cell
};

inline int band_segments(int w, int seg) { return (w + seg - 1) / seg; }

// Exact n / den for 0 <= n < 2^31 as (n * magic) >> (32 + shift).
inline void band_division(uint32_t den, uint32_t &magic, int &shift) {
  int l = 0;
  while (((uint64_t)1 << l) < den) l++;  // 2^l >= den
  shift = l > 0 ? l - 1 : 0;
  magic = (uint32_t)(((((uint64_t)1 << (32 + shift)) + den - 1) / den));
}

// DIFF: AD-census or census-gradient (BandArgs::gradient).
// REV: target x + d, the window slides towards lower disparities.
template <int LANES, int R, int WORDS, bool DIFF, bool OUT16, bool REV>
struct BandCost {
  static constexpr int ND = R / 4, W = R == 4 ? 8 : R == 20 ? 10 : R;
  struct Target {
    uint32_t d[2 * WORDS];
    uint32_t aux;
  };

  const PathJob &J;
  const BandArgs &A;
  int lane, l, y, x0, len;      // this lane's segment
  uint32_t padm[ND];            // bytes of cells k < D
  Target win[R];
  uint32_t keep[ND];            // bytes of usable targets
  // reference pixel of step (lane % 16 % W) and the target entering after it
  uint32_t ra[2 * WORDS], raux, rok;
  Target in;
  uint32_t in_keep;

  __device__ __forceinline__ BandCost(const PathJob &J_, const BandArgs &A_, int task)
      : J(J_), A(A_) {
    lane = lane_id();
    l = lane % LANES;
    const int t = task + lane / LANES, nseg = (J.w + A.seg - 1) / A.seg;
    y = t / nseg;
    x0 = (t - y * nseg) * A.seg;
    len = y < J.h ? min(A.seg, J.w - x0) : 0;
    if (len <= 0) y = 0;
#pragma unroll
    for (int i = 0; i < ND; i++) {
      padm[i] = 0;
#pragma unroll
      for (int b = 0; b < 4; b++) padm[i] |= l * R + 4 * i + b < J.D ? 0xFFu << (8 * b) : 0u;
    }
  }

  // Difference input of a pixel: its gray value, or both gray differences
  // offset to be non-negative.
  __device__ __forceinline__ uint32_t aux_of(const uint8_t *gray, size_t p) const {
    if (!A.gradient) return gray[p];
    const int gx = (int)gray[p + 1] - (int)gray[p - 1];
    const int gy = (int)gray[p + J.w] - (int)gray[p - J.w];
    return (uint32_t)(gx + 256) | ((uint32_t)(gy + 256) << 16);
  }

  // Target of column t: usable inside [rx, w - rx) and textured.
  __device__ __forceinline__ uint32_t fetch(Target &T, int t) const {
    const bool inside = len > 0 && t >= J.rx && t < J.w - J.rx && y >= J.ry && y < J.h - J.ry;
    const size_t n = (size_t)J.w * J.h, q = inside ? (size_t)y * J.w + t : 0;
#pragma unroll
    for (int i = 0; i < WORDS; i++) {
      const uint64_t d = J.desc_b[i * n + q];
      T.d[2 * i] = (uint32_t)d;
      T.d[2 * i + 1] = (uint32_t)(d >> 32);
    }
    if constexpr (WORDS == 1) T.d[1] |= 0x80000000u;  // bit 63 is the mask
    T.aux = 0u;
    if (DIFF && inside) T.aux = aux_of(J.gray_b, q);
    return inside && J.mask_b[q] ? 0xFFu : 0u;
  }

  // Reference pixel of step s and the target entering after it.
  __device__ __forceinline__ void meta(int w0) {
    const int s = w0 + (lane & 15) % W, x = x0 + s;
    const bool ok = s < len && x >= J.rx && x < J.w - J.rx && y >= J.ry && y < J.h - J.ry;
    const size_t n = (size_t)J.w * J.h, p = ok ? (size_t)y * J.w + x : 0;
#pragma unroll
    for (int i = 0; i < WORDS; i++) {
      const uint64_t d = J.desc_a[i * n + p];
      ra[2 * i] = (uint32_t)d;
      ra[2 * i + 1] = (uint32_t)(d >> 32);
    }
    if constexpr (WORDS == 1) ra[1] |= 0x80000000u;
    raux = 0u;
    if (DIFF && ok) raux = aux_of(J.gray, p);
    rok = ok && J.mask[p] ? ~0u : 0u;
    in_keep = fetch(in, REV ? x + 1 + J.minD + LANES * R - 1 : x + 1 - J.minD);
  }

  __device__ __forceinline__ uint32_t cell(const Target &T, const uint32_t *a, uint32_t aux) const {
    uint32_t ham = 0;
#pragma unroll
    for (int i = 0; i < 2 * WORDS; i++) ham += __builtin_popcount(T.d[i] ^ a[i]);
    if constexpr (!DIFF) return ham;
    const uint32_t diff = __builtin_amdgcn_sad_u16(T.aux, aux, 0u);
    const uint32_t v = ham * A.wa + min(diff, A.cap) * A.wb + A.half;
    return __umulhi(v, A.magic) >> A.shift;
  }

  static __device__ __forceinline__ uint32_t pass(uint32_t end, uint32_t fill, bool edge) {
    return REV ? line_shl1<LANES>(end, fill, edge) : line_shr1<LANES>(end, fill, edge);
  }

  template <int JJ>
  __device__ __forceinline__ void one(int s, uint8_t *row, int off, bool edge) {
    uint32_t a[2 * WORDS];
#pragma unroll
    for (int i = 0; i < 2 * WORDS; i++) a[i] = row_lane<JJ>(ra[i]);
    const uint32_t aux = !DIFF ? 0u : row_lane<JJ>(raux);
    const uint32_t ok = row_lane<JJ>(rok);
    uint32_t out[OUT16 ? 2 * ND : ND];
#pragma unroll
    for (int i = 0; i < ND; i++) {
      uint32_t v[4];
#pragma unroll
      for (int b = 0; b < 4; b++) v[b] = cell(win[4 * i + b], a, aux);
      const uint32_t use = keep[i] & padm[i] & ok;
      if constexpr (!OUT16) {
        const uint32_t codes = (A.inv & padm[i]) | (A.pad & ~padm[i]);
        const uint32_t c = v[0] | (v[1] << 8) | ((v[2] | (v[3] << 8)) << 16);
        out[i] = (c & use) | (codes & ~use);
      } else {
#pragma unroll
        for (int h = 0; h < 2; h++) {
          const uint32_t sel = h ? 0x03030202u : 0x01010000u;
          const uint32_t u = __builtin_amdgcn_perm(0u, use, sel);
          const uint32_t pm = __builtin_amdgcn_perm(0u, padm[i], sel);
          const uint32_t codes = (A.inv & pm) | (A.pad & ~pm);
          out[2 * i + h] = ((v[2 * h] | (v[2 * h + 1] << 16)) & u) | (codes & ~u);
        }
      }
    }
    const __amdgpu_buffer_rsrc_t to = make_rsrc(row, kExcessRange);
    const int at = s < len ? off : kExcessDrop;
    if (R != 20 && A.stream) bstore_dwords<OUT16 ? 2 * ND : ND, POL_NT>(out, to, at);
    else bstore_dwords<OUT16 ? 2 * ND : ND, POL_DEFAULT>(out, to, at);
    // the targets move by one column
    Target e;
    const Target &end = win[REV ? 0 : R - 1];
#pragma unroll
    for (int i = 0; i < 2 * WORDS; i++) e.d[i] = pass(end.d[i], row_lane<JJ>(in.d[i]), edge);
    e.aux = !DIFF ? 0u : pass(end.aux, row_lane<JJ>(in.aux), edge);
    const uint32_t k = REV ? pass(keep[0] & 0xFFu, row_lane<JJ>(in_keep), edge)
                           : pass(keep[ND - 1] >> 24, row_lane<JJ>(in_keep), edge);
    if constexpr (REV) {
#pragma unroll
      for (int j = 0; j + 1 < R; j++) win[j] = win[j + 1];
      win[R - 1] = e;
#pragma unroll
      for (int i = 0; i < ND; i++)
        keep[i] = (keep[i] >> 8) | ((i + 1 < ND ? keep[i + 1] : k) << 24);
    } else {
#pragma unroll
      for (int j = R - 1; j > 0; j--) win[j] = win[j - 1];
      win[0] = e;
#pragma unroll
      for (int i = ND - 1; i >= 0; i--)
        keep[i] = (keep[i] << 8) | (i > 0 ? keep[i - 1] >> 24 : k);
    }
  }

  template <int... JJ>
  __device__ __forceinline__ void steps(int w0, const uint8_t *base, int off, bool edge,
                                        std::integer_sequence<int, JJ...>) {
    (one<JJ>(w0 + JJ,
             const_cast<uint8_t *>(base) + (size_t)(w0 + JJ) * J.Dp * (OUT16 ? 2 : 1), off, edge),
     ...);
  }

  __device__ __forceinline__ void run() {
    const bool inside = l * R < J.Dp;
    const int ob = OUT16 ? 2 : 1;
    // rows of the wave start at its first segment; the others lie behind it
    const int p = y * J.w + x0, p_first = __builtin_amdgcn_readfirstlane(p);
    const int off = inside && len > 0 ? ((p - p_first) * J.Dp + l * R) * ob : kExcessDrop;
    const uint8_t *base = uniform((const uint8_t *)J.cost_out) + (size_t)p_first * J.Dp * ob;
    const bool edge = REV ? l == LANES - 1 : l == 0;
#pragma unroll
    for (int i = 0; i < ND; i++) keep[i] = 0;
#pragma unroll
    for (int j = 0; j < R; j++) {
      const int k = l * R + j;
      keep[j >> 2] |= fetch(win[j], REV ? x0 + J.minD + k : x0 - J.minD - k) << (8 * (j & 3));
    }
    for (int w0 = 0; w0 < A.seg; w0 += W) {
      if (__builtin_amdgcn_ballot_w64(w0 < len) == 0) break;
      meta(w0);
      steps(w0, base, off, edge, std::make_integer_sequence<int, W>());
    }
  }
};

template <int LANES, int R, int WORDS, bool DIFF, bool OUT16>
__global__ __launch_bounds__(256) void band_cost_kernel(PathJobs jobs, BandArgs A) {
  const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * (blockDim.x >> 6) +
                                                  (int)(threadIdx.x >> 6));
  if (wave >= A.total) return;
  int local = wave, ji = 0;
  if (jobs.table) {
    ji = __builtin_amdgcn_readfirstlane(find_job(A.wave_begin, A.njobs, wave));
    local -= A.wave_begin[ji];
  } else if (A.njobs > 1 && wave >= A.split) {
    ji = 1;
    local -= A.split;
  }
  PathJob J = jobs.table ? jobs.table[ji] : jobs.local[ji & 1];
  J.desc_a = uniform(J.desc_a);
  J.desc_b = uniform(J.desc_b);
  J.mask = uniform(J.mask);
  J.mask_b = uniform(J.mask_b);
  J.gray = uniform(J.gray);
  J.gray_b = uniform(J.gray_b);
  J.w = uniform(J.w);
  J.h = uniform(J.h);
  J.D = uniform(J.D);
  J.Dp = uniform(J.Dp);
  J.minD = uniform(J.minD);
  J.rx = uniform(J.rx);
  J.ry = uniform(J.ry);
  const int task = local * (64 / LANES);
  if (uniform(J.reverse)) BandCost<LANES, R, WORDS, DIFF, OUT16, true>(J, A, task).run();
  else BandCost<LANES, R, WORDS, DIFF, OUT16, false>(J, A, task).run();
}

}  // namespace sgm
