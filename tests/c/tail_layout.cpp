// The coarse tail's LDS layout (csrc/wl_tail.h) against the bytes its launches ask for, over the level
// sizes of hierarchies in 2D and 3D: prints how many lie past the request or overlap.
#include <cstdio>
#include <vector>

#include "wl_tail.h"

int main() {
  long bad = 0, seen = 0, padded = 0;
  for (int D = 2; D <= 3; ++D)
    for (int a = 4; a <= 26; ++a)
      for (int b = 4; b <= 26; ++b)
        for (int c = D == 3 ? 4 : 1; c <= (D == 3 ? 26 : 1); ++c) {
          int N[3] = {a, b, c};
          std::vector<wl::TailLv> lv;
          long n = 0;
          for (bool more = true; more && lv.size() < 11;) {
            wl::TailLv q = {};
            q.n = N[0] * N[1] * N[2];
            n += q.n;
            lv.push_back(q);
            more = false;
            for (int d = 0; d < D; ++d)
              if (N[d] % 2 == 0 && N[d] > 4) N[d] = 1 + N[d] / 2, more = true;
          }
          int nimg = 0;
          const long total = wl::tail_fast_layout(D, lv.data(), (int)lv.size(), &nimg);
          const long asked = (long)(wl::tail_lds_bytes(D, n, true, sizeof(float)) / sizeof(float));
          long at = 0;  // the arrays follow each other, the second part on a whole vector
          for (const wl::TailLv& q : lv) {
            bad += q.oL != at || q.oD != at + D * q.n || q.oI != q.oD + q.n;
            at = q.oI + q.n;
          }
          bad += nimg < at || nimg > at + 3 || nimg % 4 != 0;
          padded += nimg != at;
          at = nimg;
          for (const wl::TailLv& q : lv) {
            bad += q.oR != at || q.oX != at + q.n || q.oE != q.oX + q.n;
            at = q.oE + q.n;
          }
          bad += at != total || at > asked;
          bad += wl::tail_lds_bytes(D, n, false, sizeof(float)) / sizeof(float) < (size_t)((D + 5) * n);
          ++seen;
        }
  std::printf("%ld of %ld, %s\n", bad, seen, padded ? "some padded" : "none padded");
  return 0;
}
