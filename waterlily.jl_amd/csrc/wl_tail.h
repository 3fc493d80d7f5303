// Where the coarse tail's levels lie in the LDS: the offsets its kernels use and the bytes its
// launches ask for, from one place.  Plain C++ (the host's launches, the kernels and a CPU test
// include it).
#pragma once
#include <cstddef>
#include <cstdint>

namespace wl {

struct TailLv {           // one level of k_mg_tail_fast; built on the host, read with scalar loads
  int N0, N1, N2;
  int s1, s2, n, cm;
  int lx, ly;             // log2 of the threads along x (pairs) and y
  int oL, oD, oI;         // LDS element offsets: L (D arrays of n), D, 1/D ...
  int oR, oX, oE;         // ... r, x, ϵ
  int small;              // run by the first wave alone
};
// The image (L, D, 1/D of every level) first, rounded up to whole vectors of 4 elements (it is copied
// in by them: *nimg), then each level's r, x and ϵ.  lv[k].n is set; returns the elements in all.
inline int tail_fast_layout(int D, TailLv* lv, int levels, int* nimg) {
  int o = 0;
  for (int k = 0; k < levels; ++k) {
    TailLv& q = lv[k];
    q.oL = o;
    q.oD = o + D * q.n;
    q.oI = q.oD + q.n;
    o = q.oI + q.n;
  }
  o = (o + 3) & ~3;
  *nimg = o;
  for (int k = 0; k < levels; ++k) {
    TailLv& q = lv[k];
    q.oR = o;
    q.oX = o + q.n;
    q.oE = q.oX + q.n;
    o = q.oE + q.n;
  }
  return o;
}
// The elements the levels take whose cells sum to n: by k_mg_tail_lds, level by level (L, x, r, ϵ, D,
// 1/D), and by k_mg_tail_fast
inline int64_t tail_general_elems(int D, int64_t n) { return (D + 5) * n; }
inline int64_t tail_fast_elems(int D, int64_t n) { return (((D + 2) * n + 3) & ~int64_t(3)) + 3 * n; }
// What a tail launch over such levels asks for, in bytes
inline size_t tail_lds_bytes(int D, int64_t n, bool fast, size_t elem) {
  return (size_t)(fast ? tail_fast_elems(D, n) : tail_general_elems(D, n)) * elem;
}

}  // namespace wl
