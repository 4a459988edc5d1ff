// Host-only check of the grouped order of a causal whole-row grid (whole_item's group,
// attn_fwd_split.h): over a range of heads, query blocks and group sizes, every (b, h, query
// block) is an item exactly once, an XCD (block id mod 8) has whole heads of its own, and
// within a group its query blocks run from the heaviest to the lightest, every head's before
// any head's next.  Prints "ok <cases>" or the first failure.
#include <cstdio>
#include <vector>

#include "attn_fwd_split.h"

int main() {
  int cases = 0;
  for (int hx = 2; hx <= 33; ++hx)
    for (int nq = 1; nq <= 33; nq += nq < 6 ? 1 : 9)
      for (int group = 2; group <= 9; ++group, ++cases) {
        const int n_bh = 8 * hx;
        std::vector<int> seen((size_t)n_bh * nq, 0);
        std::vector<int> last(8, -1), first_head(8, -1);  // the XCD's last block and group
        for (int blk = 0; blk < n_bh * nq; ++blk) {
          const ta::WorkItem w = ta::whole_item(blk, n_bh, nq, 1, true, group);
          const int x = blk & 7;
          bool ok = w.bh >= x * hx && w.bh < (x + 1) * hx && w.qt >= 0 && w.qt < nq && w.slot == -1 &&
                    w.t_beg == 0 && w.t_end == -1;
          if (ok) {
            const int g = (w.bh - x * hx) / group;
            if (g != first_head[x]) {
              ok = g == first_head[x] + 1 && w.qt == nq - 1;  // groups in order, heaviest first
            } else {
              ok = w.qt == last[x] || w.qt == last[x] - 1;
            }
            first_head[x] = g;
            last[x] = w.qt;
            ok = ok && ++seen[(size_t)w.bh * nq + w.qt] == 1;
          }
          if (!ok) {
            printf("FAIL heads %d blocks %d group %d: block %d is (%d, %d)\n", n_bh, nq, group, blk, w.bh, w.qt);
            return 1;
          }
        }
        // n_bh * nq items, each once
      }
  printf("ok %d\n", cases);
  return 0;
}
