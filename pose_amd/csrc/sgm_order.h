// Dispatch orders of a launch's waves, longest first (host code only).
#pragma once

#include <string.h>

#include <algorithm>
#include <vector>

namespace sgm {

constexpr int kMaxOrderDirs = 8;

inline int lines_of(int cls, int w, int h) { return cls == 0 ? h : cls == 1 ? w : w + h - 1; }
inline int lines_along(int dx, int dy, int w, int h) {
  return lines_of(dy == 0 ? 0 : dx == 0 ? 1 : 2, w, h);
}

// Length of line `line` of direction (dx, dy) in a w x h image, in the line
// enumeration of line_start.
inline int line_length(int dx, int dy, int line, int w, int h) {
  if (dy == 0) return w;
  if (dx == 0) return h;
  const int x = line < w ? line : (dx > 0 ? 0 : w - 1);
  const int y = line < w ? (dy > 0 ? 0 : h - 1) : (dy > 0 ? line - w + 1 : h - 2 - (line - w));
  return std::min(dx > 0 ? w - x : x + 1, dy > 0 ? h - y : y + 1);
}

// Longest of the `per` lines of wave `wave`.
inline int wave_length(int dx, int dy, int wave, int per, int w, int h) {
  const int lines = lines_along(dx, dy, w, h);
  int n = 0;
  for (int l = wave * per; l < std::min(lines, (wave + 1) * per); l++)
    n = std::max(n, line_length(dx, dy, l, w, h));
  return n;
}

// The indices of `len` by length, longest first, equal lengths in index order.
inline void longest_first(const std::vector<int> &len, int maxlen, std::vector<int> &order) {
  // counting sort
  std::vector<int> start((size_t)maxlen + 2, 0);
  for (int n : len) start[maxlen - n + 1]++;  // bucket maxlen - n: longest first
  for (int i = 1; i <= maxlen + 1; i++) start[i] += start[i - 1];
  order.assign(len.size(), 0);
  for (size_t g = 0; g < len.size(); g++) order[start[maxlen - len[g]]++] = (int)g;
}

// The waves of a launch over a w x h pair: nd matching directions, every
// direction (dx[k], dy[k]) with `per` neighbouring lines a wave, split[k] waves
// of each matching direction from begin[k] on.  An order holds for these
// waves alone: launches of equally many directions (four paths, or the pairs of
// eight) number theirs differently, so all of it is compared.
struct WaveLayout {
  int w, h, nd, per, ndirs, total;
  int dx[kMaxOrderDirs], dy[kMaxOrderDirs];
  int begin[kMaxOrderDirs], split[kMaxOrderDirs];
  bool operator==(const WaveLayout &o) const { return memcmp(this, &o, sizeof o) == 0; }
};

inline WaveLayout wave_layout(int ndirs, const int *dx, const int *dy, int w, int h, int nd,
                              int per) {
  WaveLayout L;
  memset(&L, 0, sizeof L);
  L.w = w;
  L.h = h;
  L.nd = nd;
  L.per = per;
  L.ndirs = ndirs;
  for (int k = 0; k < ndirs; k++) {
    L.dx[k] = dx[k];
    L.dy[k] = dy[k];
    L.split[k] = (lines_along(dx[k], dy[k], w, h) + per - 1) / per;
    L.begin[k] = L.total;
    L.total += nd * L.split[k];
  }
  return L;
}

// The waves of `L`, longest first.
inline void wave_order(const WaveLayout &L, std::vector<int> &order) {
  std::vector<int> len((size_t)L.total);
  for (int k = 0; k < L.ndirs; k++)
    for (int m = 0; m < L.nd; m++)
      for (int l = 0; l < L.split[k]; l++)
        len[(size_t)L.begin[k] + (size_t)m * L.split[k] + l] =
            wave_length(L.dx[k], L.dy[k], l, L.per, L.w, L.h);
  longest_first(len, std::max(L.w, L.h), order);
}

}  // namespace sgm
