// The longest-first launch order (csrc/mask.h: launch_order, rank_order): every
// (slice, unit) served once, units in falling order, and, where the order pins
// slices to XCDs, each slice on one XCD and every XCD with the same number of
// slices (packed sequences of 8 n heads: of every sequence), and the units of
// one packed sequence's slice spread over the 4 shader engines that an XCD's
// workgroups go round.  Built and run by
// tests/test_launch_order.py; exits non-zero on the first violation.
#include <cstdio>
#include <cstring>
#include <map>
#include <vector>

#include "mask.h"

using namespace chia;

int main(int argc, char** argv) {
  const bool planted = argc > 1 && !std::strcmp(argv[1], "planted");
  long checked = 0;
  int bad = 0;
  for (int batch : {1, 2, 3, 5, 7, 8})
    for (int heads : {1, 2, 3, 4, 8, 12, 16, 24, 32, 40})
      for (int res : {1, 2, 3, 4})
        for (int units : {1, 2, 3, 7, 16, 33})
          for (bool packed : {false, true}) {
            const int slices = batch * heads * res;
            LaunchOrder o = launch_order(true, slices, heads, res, packed);
            if (planted && o.shift == 3 && packed) o.hs -= 1;  // neighbouring runs overlap
            std::vector<char> seen((size_t)slices * units, 0);
            std::map<int, int> xcd_of;
            std::vector<int> engine((size_t)slices * 4, 0);  // [slice][turn of 4 in its XCD] -> units
            const bool by_seq = packed && heads % 8 == 0 && res == 1;
            std::map<std::pair<int, int>, int> per_xcd;  // (XCD, sequence) -> slices
            int last = units;
            for (int x = 0; x < slices * units; ++x) {
              const SliceUnit su = rank_order(x, o, units);
              ++checked;
              if (su.slice < 0 || su.slice >= slices || su.unit < 0 || su.unit >= units) { ++bad; continue; }
              char& s = seen[(size_t)su.slice * units + su.unit];
              if (s++) ++bad;
              if (x % 8 == 0 && su.unit > last) ++bad;
              if (x % 8 == 0) last = su.unit;
              if (o.shift == 3) {
                if (xcd_of.count(su.slice) && xcd_of[su.slice] != x % 8) ++bad;
                if (!xcd_of.count(su.slice)) ++per_xcd[{x % 8, by_seq ? su.slice / heads : 0}];
                xcd_of[su.slice] = x % 8;
                ++engine[(size_t)su.slice * 4 + x / 8 % 4];
              }
            }
            if (o.shift == 3) {
              const int each = by_seq ? heads / 8 : slices / 8;
              for (auto& kv : per_xcd)
                if (kv.second != each) ++bad;
            }
            // a slice's turns come round every hx (-1: its rank starts one on), but
            // for one skipped turn every hx ranks
            if (o.shift == 3 && packed)
              for (int n : engine)
                if (n > (units + 3) / 4 + 1 + units / o.hx) ++bad;
            if (bad && !planted) {
              std::printf("violation: batch %d heads %d residues %d units %d packed %d\n", batch, heads, res, units, packed);
              return 1;
            }
          }
  std::printf("%ld workgroups checked, %s\n", checked, bad ? "planted mistake caught" : "0 violations");
  return planted ? (bad ? 0 : 1) : 0;
}
