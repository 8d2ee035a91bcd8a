// Whole-image sweeps of the compact plan (sgm_compact.h), several lines per wave.
//
// The passes and their results are those of compact_segment with costs computed
// on the fly; a line takes LANES lanes of R disparities and a wave 64 / LANES
// neighbouring lines, with the packed recurrence of sgm_excess.h (whole numbers;
// the largest sum, 512 + 3 * P2, fits for P2 <= kCompactLineP2).  A line's target
// descriptors are loaded side by side and turned through LDS: read lane by lane
// (R descriptors each, 64 cache lines an instruction) the L1 cache was the bound,
// 7.3 ms against 3.8 for the verification pass below.  Cells lie in ascending
// columns for both matching directions, so neither needs its own code.
//
// The proposal pass runs every direction in one launch (a direction writes only
// its own proposals); the verification pass too, adding with 32-bit atomics on
// packed pairs: a cell's sum stays within 16 bits (paths * (512 + P2)), a pad
// cell's would not and is left out, so no half carries.  Both are bound by VALU,
// 120 instructions a wave and step, 190 with two proposals, issued at about 85%
// of the rate.  The sum pass accumulates, so direction by direction, and its one
// or two waves per SIMD are bound by their own issue; four pixels' proposals are
// looked up together.  Measured at 1600x1067 D=256, two proposals per path,
// against one line per wave, 32-bit integers and one direction per launch:
// proposals 16.6 -> 5.2 ms, sums 18.3 -> 9.0, verification 10.5 -> 3.3.
#pragma once

namespace sgm {

constexpr int kCompactLineP2 = 9216;  // 512 + 3 * P2, the largest sum, stays below 0x7000

struct CompactLineArgs {
  int ndirs, total, njobs;
  int p1, p2, edge;
  int C, pool;
  int dx[kMaxExcessDirs], dy[kMaxExcessDirs], index[kMaxExcessDirs];
  int begin[kMaxExcessDirs], split[kMaxExcessDirs];
  int first;             // sum pass: the first direction stores, the others add
};

template <int LANES, int R, int PH>
struct CompactLine {
  static constexpr int NP = R / 2, W = 8;
  static constexpr int NB = 4;  // sum pass: pixels whose proposals are looked up together
  static constexpr int PL = LANES == 16 ? 2 : 1;  // proposals per lane (at most 32 per pixel)

  const CompactJob &J;
  const CompactLineArgs &A;
  const uint32_t *tab;
  int lane, l, len, maxlen, x0, y0, dx, dy, p0, step, direction;
  bool first, last;
  int flip;  // cells lie in ascending columns: cell of disparity k is k ^ flip
  uint32_t p1pk, kpk[NP], inv[NP], keep[NP];
  __amdgpu_buffer_rsrc_t gm, db;
  // steps between a target's load and its use: the sum pass has one or two waves
  // per SIMD to hide the latency behind
  static constexpr int AHEAD = PH == ESGM_SUMS ? 2 : 1;
  uint32_t tw[AHEAD][2 * R];    // targets as loaded: chunks i * LANES + l of the line's
  uint32_t rd[2 * R];           // this step's, the lane's own, ascending columns
  uint4 *stage;                 // this line's LDS room for them
  int put_at[R / 2], get_at;
  uint32_t ma_lo, ma_hi, mok, mp2;
  // sum pass: this line's LDS rows, NB each of kRow cells after kEdge: path costs
  // (zero past either end of the range), and those of valid cells off the
  // proposals (else 0xFFFF)
  static constexpr int kEdge = 8, kRow = LANES * R + 2 * kEdge;
  uint16_t *cells, *open;
  struct Sums {
    int cand[PL], v[PL][3];
  } ahead[NB];
  int outside;                  // bound so far of pixel l of the NB
  int lead;                     // pixels from the wave's lowest start pixel
  int base;                     // that start pixel

  __device__ __forceinline__ CompactLine(const CompactJob &J_, const CompactLineArgs &A_, int k,
                                         int line0, const uint32_t *tab_)
      : J(J_), A(A_), tab(tab_) {
    lane = lane_id();
    l = lane % LANES;
    dx = A.dx[0];
    dy = A.dy[0];
    direction = A.index[0];
#pragma unroll
    for (int i = 1; i < kMaxExcessDirs; i++)
      if (i == k) {
        dx = A.dx[i];
        dy = A.dy[i];
        direction = A.index[i];
      }
    const int line = line0 + lane / LANES;
    const int lines = dy == 0 ? J.h : dx == 0 ? J.w : J.w + J.h - 1;
    x0 = y0 = 0;
    len = 0;
    if (line < lines) line_start(line, dx, dy, J.w, J.h, x0, y0, len);
    p0 = y0 * J.w + x0;
    step = dy * J.w + dx;
    maxlen = __builtin_amdgcn_readlane(len, 0);
#pragma unroll
    for (int g = 1; g < 64 / LANES; g++)
      maxlen = max(maxlen, __builtin_amdgcn_readlane(len, g * LANES));
    first = l == 0;
    last = l == LANES - 1;
    p1pk = splat16((uint32_t)A.p1);
    flip = J.reverse ? 0 : LANES * R - 1;
    const uint32_t pad = 512u + (uint32_t)A.p2;
#pragma unroll
    for (int i = 0; i < NP; i++) {
      const int c0 = l * R + (i >> 1) * 4 + (i & 1);
      const int k0 = c0 ^ flip, k1 = (c0 + 2) ^ flip;
      kpk[i] = (uint32_t)k0 | ((uint32_t)k1 << 16);
      keep[i] = (k0 < J.D ? 0xFFFFu : 0u) | (k1 < J.D ? 0xFFFF0000u : 0u);
      inv[i] = (k0 < J.D ? 512u : pad) | ((k1 < J.D ? 512u : pad) << 16);
    }
#pragma unroll
    for (int i = 0; i < R / 2; i++) {
      const int q = i * LANES + l;
      put_at[i] = q / (R / 2) * (R / 2 + 1) + q % (R / 2);
    }
    get_at = l * (R / 2 + 1);
    const uint32_t n = (uint32_t)J.w * (uint32_t)J.h;
    gm = make_rsrc(J.gm, n * 2u);
    db = make_rsrc(J.desc_b, n * 8u);
  }

  // Targets of step s: LANES * R descriptors in ascending columns, 16 bytes a
  // lane side by side (outside the array: 0).
  __device__ __forceinline__ void load_targets(uint32_t *to, int s) {
    const int sc = min(s, max(len - 1, 0));
    const int t = x0 + sc * dx + (J.reverse ? J.minD : -J.minD - (LANES * R - 1));
    const int off = (int)(((uint32_t)(y0 + sc * dy) * (uint32_t)J.w + (uint32_t)(t + 2 * l)) * 8u);
#pragma unroll
    for (int i = 0; i < R / 2; i++) bload_dwords<4, POL_DEFAULT>(to + 4 * i, db, off + i * LANES * 16);
  }
  // Hands every lane the R descriptors of its own disparities, through LDS: a
  // lane's rows lie R / 2 + 1 (odd) chunks apart, so neither side meets a bank
  // twice.  The wave's LDS accesses run in order.
  __device__ __forceinline__ void turn_targets(const uint32_t *v) {
#pragma unroll
    for (int i = 0; i < R / 2; i++)
      stage[put_at[i]] = make_uint4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
    lds_turn();
#pragma unroll
    for (int i = 0; i < R / 2; i++) {
      const uint4 c = stage[get_at + i];
      rd[4 * i] = c.x;
      rd[4 * i + 1] = c.y;
      rd[4 * i + 2] = c.z;
      rd[4 * i + 3] = c.w;
    }
    lds_turn();
  }

  // Proposal arrays of the wave's pixels at step s, addressed from its lowest one.
  __device__ __forceinline__ __amdgpu_buffer_rsrc_t row_of(const uint16_t *p, int each, int s) const {
    return make_rsrc(uniform(p) + (int64_t)(base + s * step) * each, kExcessRange);
  }

  // Sum pass: proposals, their sums so far and the bounds of steps s .. s + NB - 1.
  __device__ __forceinline__ void load_sums(int s) {
#pragma unroll
    for (int b = 0; b < NB; b++) {
      Sums &q = ahead[b];
      const __amdgpu_buffer_rsrc_t cr = row_of(J.cand, A.C, s + b), sr = row_of(J.sums, 3 * A.C, s + b);
#pragma unroll
      for (int u = 0; u < PL; u++) {
        const int t = l + u * LANES;
        const int off = t < A.C && s + b < len ? (lead * A.C + t) * 2 : kExcessDrop;
        q.cand[u] = __builtin_amdgcn_raw_buffer_load_b16(cr, off, 0, 0);
#pragma unroll
        for (int o = 0; o < 3; o++)
          q.v[u][o] = A.first ? 0 : (int)__builtin_amdgcn_raw_buffer_load_b16(
                                        sr, off == kExcessDrop ? off : 3 * off + 2 * o, 0, 0);
      }
    }
    outside = 0;
    if (!A.first && l < NB && s + l < len) outside = J.outside[p0 + (s + l) * step];
  }

  // Reference pixels and penalties of the window [w0, w0 + W), one per lane % W.
  struct Raw {
    int g, gp;
    uint64_t a;
    bool inside;
  };
  __device__ __forceinline__ Raw meta_load(int w0) const {
    const int s = w0 + (lane & 15) % W;
    const bool in = s < len;
    const int p = p0 + (in ? s : 0) * step;
    const int x = x0 + s * dx, y = y0 + s * dy;
    Raw r;
    r.g = __builtin_amdgcn_raw_buffer_load_b16(gm, p * 2, 0, 0);
    r.gp = in && s > 0 ? (int)__builtin_amdgcn_raw_buffer_load_b16(gm, (p - step) * 2, 0, 0) : 0;
    r.a = J.desc_a[p];
    r.inside = in && x >= J.rx && x < J.w - J.rx && y >= J.ry && y < J.h - J.ry;
    return r;
  }
  __device__ __forceinline__ void meta_finish(const Raw &r) {
    const uint32_t v = tab[abs((r.g & 0xFF) - (r.gp & 0xFF))];
    mp2 = (r.gp >> 8) ? v : 0u;
    mok = r.inside && (r.g >> 8) ? ~0u : 0u;
    ma_lo = (uint32_t)r.a;
    ma_hi = (uint32_t)(r.a >> 32) | 0x80000000u;
  }

  // Costs of the step's pixel and, per pair, which cells are valid.
  template <int JJ>
  __device__ __forceinline__ void costs(int s, uint32_t *c, uint32_t *valid) {
    // (the flag bit is set in both descriptors of a valid cell)
    const uint32_t alo = row_lane<JJ>(ma_lo), ahi = row_lane<JJ>(ma_hi);
    // disparities whose target lies in [rx, w - rx), within the range
    const int x = x0 + s * dx;
    const int ka = max(0, J.reverse ? J.rx - J.minD - x : x - J.minD - (J.w - J.rx - 1));
    const int kb = min(J.D - 1, J.reverse ? J.w - J.rx - 1 - J.minD - x : x - J.minD - J.rx);
    const uint32_t lo = splat16((uint32_t)ka);
    const int span = row_lane<JJ>(mok) ? kb - ka : -1;  // < 0: none
#pragma unroll
    for (int i = 0; i < NP; i++) {
      uint32_t ham[2], high[2];
#pragma unroll
      for (int h = 0; h < 2; h++) {
        const int j = (i >> 1) * 4 + (i & 1) + 2 * h;
        const uint32_t dl = rd[2 * j], dh = rd[2 * j + 1];
        ham[h] = __builtin_popcount(dl ^ alo) + __builtin_popcount(dh ^ ahi);
        high[h] = dh;
      }
      c[i] = ham[0] | (ham[1] << 16);
      valid[i] = __builtin_amdgcn_perm(high[1], high[0], 0x0B0B0909u);  // their flags, spread
    }
    if (__builtin_amdgcn_ballot_w64(span != LANES * R - 1)) {
      const uint32_t sp = splat16(span < 0 ? 0u : (uint32_t)span);
#pragma unroll
      for (int i = 0; i < NP; i++) {
        // 0 where ka <= k <= kb
        const uint32_t t = pk_min(pk_sub_sat(pk_sub(kpk[i], lo), sp), 0x00010001u);
        valid[i] &= span < 0 ? 0u : pk_sub(t, 0x00010001u);
      }
    }
#pragma unroll
    for (int i = 0; i < NP; i++) c[i] = (c[i] & valid[i]) | (inv[i] & ~valid[i]);
  }

  // Separated proposals of the pixel (Lm: path costs, invalid cells 0xFFFF): the
  // least cost and its first disparity as one 32-bit key.
  __device__ __forceinline__ void propose(uint32_t *Lm, int s) {
    uint32_t chosen[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      chosen[q] = 65535u;
      if (q < A.pool) {
        uint32_t key = ~0u;
#pragma unroll
        for (int i = 0; i < NP; i++)
          key = min(min(key, (Lm[i] << 16) | (kpk[i] & 0xFFFFu)),
                    (Lm[i] & 0xFFFF0000u) | (kpk[i] >> 16));
        key = line_min<LANES>(key);
        if (key < 0xFFFF0000u) chosen[q] = key & 0xFFFFu;
        if (q + 1 < A.pool) {
          const uint32_t bm1 = splat16((key & 0xFFFFu) - 1u);
#pragma unroll
          for (int i = 0; i < NP; i++)
            Lm[i] = pk_mad_sat(pk_sub_sat(0x00030003u, pk_sub(kpk[i], bm1)), ~0u, Lm[i]);
        }
      }
    }
    if (l < A.pool && s < len) {
      const uint32_t mine = l == 0 ? chosen[0] : l == 1 ? chosen[1] : l == 2 ? chosen[2] : chosen[3];
      J.cand[(size_t)(p0 + s * step) * A.C + direction * A.pool + l] = (uint16_t)mine;
    }
  }

  static __device__ __forceinline__ void lds_turn() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }

  // Sum pass: the step's rows, in ascending columns.
  __device__ __forceinline__ void keep_rows(int b, const uint32_t *L, const uint32_t *Lm) {
    uint2 *own = reinterpret_cast<uint2 *>(cells + b * kRow + kEdge + l * R);
    uint2 *off = reinterpret_cast<uint2 *>(open + b * kRow + kEdge + l * R);
#pragma unroll
    for (int i = 0; i < NP; i += 2) {
      const uint32_t e = L[i] & keep[i], o = L[i + 1] & keep[i + 1];
      own[i / 2] = make_uint2(__builtin_amdgcn_perm(o, e, 0x05040100u),
                              __builtin_amdgcn_perm(o, e, 0x07060302u));
      off[i / 2] = make_uint2(__builtin_amdgcn_perm(Lm[i + 1], Lm[i], 0x05040100u),
                              __builtin_amdgcn_perm(Lm[i + 1], Lm[i], 0x07060302u));
    }
  }

  // Adds the path costs at the proposals of steps s .. s + NB - 1 and the least
  // ones off them.
  __device__ __forceinline__ void add_sums(int s) {
    Sums q[NB];
    const int before = outside;
#pragma unroll
    for (int b = 0; b < NB; b++) q[b] = ahead[b];
    load_sums(s + NB);
    lds_turn();
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
      for (int u = 0; u < PL; u++) {
        // no proposal (or none of this lane's): the zeros before the range
        const int k = q[b].cand[u];
        const bool some = k < J.D && l + u * LANES < A.C;
        const int c = b * kRow + (some ? kEdge + (k ^ flip) : 1);
        const int below = cells[c - 1], above = cells[c + 1];
        q[b].v[u][0] += J.reverse ? below : above;
        q[b].v[u][1] += cells[c];
        q[b].v[u][2] += J.reverse ? above : below;
        open[c - 1] = open[c] = open[c + 1] = 0xFFFFu;
        if (!some) q[b].cand[u] = 65535;
      }
    lds_turn();
    uint32_t lower[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const uint2 *off = reinterpret_cast<const uint2 *>(open + b * kRow + kEdge + l * R);
      uint32_t m = ~0u;
#pragma unroll
      for (int i = 0; i < NP / 2; i++) {
        const uint2 v = off[i];
        m = pk_min(m, pk_min(v.x, v.y));
      }
      lower[b] = m;
    }
#pragma unroll
    for (int b = 0; b < NB; b++) lower[b] = line_min_pk<LANES>(lower[b]);
    lds_turn();
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const __amdgpu_buffer_rsrc_t sr = row_of(J.sums, 3 * A.C, s + b);
#pragma unroll
      for (int u = 0; u < PL; u++) {
        const int off = q[b].cand[u] < J.D && s + b < len ? (lead * A.C + l + u * LANES) * 6 : kExcessDrop;
#pragma unroll
        for (int o = 0; o < 3; o++)
          __builtin_amdgcn_raw_buffer_store_b16((uint16_t)q[b].v[u][o], sr, off + 2 * o, 0, 0);
      }
    }
    if (l < NB && s + l < len) {
      const uint32_t mine = l == 0 ? lower[0] : l == 1 ? lower[1] : l == 2 ? lower[2] : lower[3];
      J.outside[p0 + (s + l) * step] =
          (uint16_t)(mine == 0xFFFFu ? 65535 : min(65535, before + (int)mine));
    }
  }

  // Adds the path costs of a pixel that is verified in this group.
  __device__ __forceinline__ void add_verified(const uint32_t *L, int sl) {
    const int lanes = J.Dp / R, own = l ^ (flip / R);  // verify_cell's layout
    if (sl >= J.lo && sl < J.hi && own < lanes) {
      uint32_t *row = reinterpret_cast<uint32_t *>(J.verify + (size_t)(sl - J.lo) * J.Dp) + own;
#pragma unroll
      for (int i = 0; i < NP; i++)
        __hip_atomic_fetch_add(row + i * lanes, L[i] & keep[i], __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
    }
  }

  ExcessState<R> state;
  int slots;

  template <int JJ>
  __device__ __forceinline__ void one(int s) {
    uint32_t c[NP], valid[NP], e[NP];
    costs<JJ>(s, c, valid);
    turn_targets(tw[(JJ + 1) % AHEAD]);
    load_targets(tw[(JJ + 1) % AHEAD], s + 1 + AHEAD);
    const uint32_t p2 = row_lane<JJ>(mp2);
    excess_step<LANES, R>(state, c, p2, p1pk, first, last, e);
    if constexpr (PH == ESGM_VERIFY) {
      const int sl = (int)row_lane<JJ>((uint32_t)slots);
      add_verified(state.L, s < len ? sl : -1);
    } else {
      uint32_t Lm[NP];
#pragma unroll
      for (int i = 0; i < NP; i++) Lm[i] = state.L[i] | ~valid[i];
      if constexpr (PH == ESGM_CANDIDATES) {
        propose(Lm, s);
      } else {
        keep_rows(JJ % NB, state.L, Lm);
        if constexpr (JJ % NB == NB - 1) add_sums(s - (NB - 1));
      }
    }
  }
  template <int... JJ>
  __device__ __forceinline__ void window(int w0, std::integer_sequence<int, JJ...>) {
    const Raw next = meta_load(w0 + W);
    int snext = -1;
    if constexpr (PH == ESGM_VERIFY) {
      const int s = w0 + W + (lane & 15) % W;
      if (s < len) snext = J.slot[p0 + s * step];
    }
    (one<JJ>(w0 + JJ), ...);
    meta_finish(next);
    slots = snext;
  }

  __device__ __forceinline__ void run() {
    meta_finish(meta_load(0));
    slots = -1;
    if constexpr (PH == ESGM_VERIFY) {
      const int s = (lane & 15) % W;
      if (s < len) slots = J.slot[p0 + s * step];
    }
    load_targets(tw[0], 0);
    turn_targets(tw[0]);
#pragma unroll
    for (int j = 1; j <= AHEAD; j++) load_targets(tw[j % AHEAD], j);
    if constexpr (PH == ESGM_SUMS) {
      for (int i = l; i < NB * kRow; i += LANES) cells[i] = 0;
      lds_turn();
      // (the lines of a wave that exist lie before those that do not)
      base = __builtin_amdgcn_readlane(p0, 0);
#pragma unroll
      for (int g = 1; g < 64 / LANES; g++) {
        const int other = __builtin_amdgcn_readlane(p0, g * LANES);
        if (__builtin_amdgcn_readlane(len, g * LANES) > 0) base = min(base, other);
      }
      lead = p0 - base;
      load_sums(0);
    }
    state.clear();
    for (int w0 = 0; w0 < maxlen; w0 += W) window(w0, std::make_integer_sequence<int, W>());
  }
};

template <int LANES, int R, int PH>
__global__ __launch_bounds__(256, PH == ESGM_SUMS ? 2 : 4) void compact_line_kernel(CompactJobs jobs, CompactLineArgs A) {
  using Sweep = CompactLine<LANES, R, PH>;
  __shared__ uint32_t tab[256];
  __shared__ uint4 targets[4][64 * (R / 2 + 1)];
  constexpr int kLine = Sweep::kRow * Sweep::NB, kRows = PH == ESGM_SUMS ? 64 / LANES * kLine : 8;
  __shared__ __align__(16) uint16_t rows[PH == ESGM_SUMS ? 4 : 1][2][kRows];
  build_p2_pairs(tab, A.p1, A.p2, A.edge);
  const int wv = (int)(threadIdx.x >> 6), lane = lane_id();
  __syncthreads();
  const int wave = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + wv);
  if (wave >= A.total) return;
  int k = 0, begin = A.begin[0], split = A.split[0];
#pragma unroll
  for (int i = 1; i < kMaxExcessDirs; i++)
    if (i < A.ndirs && wave >= A.begin[i]) {
      k = i;
      begin = A.begin[i];
      split = A.split[i];
    }
  int local = wave - begin;
  const bool second = A.njobs > 1 && local >= split;
  if (second) local -= split;
  const CompactJob J = second ? jobs.job[1] : jobs.job[0];
  Sweep sweep(J, A, k, local * (64 / LANES), tab);
  sweep.stage = targets[wv] + lane / LANES * LANES * (R / 2 + 1);
  if (PH == ESGM_SUMS) {
    sweep.cells = rows[wv][0] + lane / LANES * kLine;
    sweep.open = rows[wv][1] + lane / LANES * kLine;
  }
  sweep.run();
}

}  // namespace sgm
