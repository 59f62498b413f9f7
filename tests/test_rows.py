"""The rows that a thread of a reduction reads ahead in a pass that also writes its rows: the thread's
own, so that none is read while another thread writes it."""
import host_build

PROGRAM = r"""
#include <cstdio>
#include <vector>
#include "lsx_rows.hpp"
int main() {
  const int BS = 8, R = 4;
  for (long n = 1; n <= 300; ++n)
    for (int nb = 1; nb <= 12; ++nb) {
      std::vector<long> owner(n, -1);
      for (int pass = 0; pass < 2; ++pass)  // who writes a row, then who reads it
        for (int b = 0; b < nb; ++b)
          for (int t = 0; t < BS; ++t) {
            long lo, hi;
            lsx::chunk_of(n, b, nb, &lo, &hi);
            for (long i = lo + t; i < hi; i += R * BS)
              for (int r = 0; r < R; ++r) {
                if (pass == 0 && i + r * BS < hi) owner[i + r * BS] = b * BS + t;
                if (pass == 1 && owner[lsx::row_ahead(i, r * BS, hi)] != b * BS + t) return 1;
              }
          }
      for (long o : owner)
        if (o < 0) return 2;  // every row is someone's
    }
  std::printf("ok\n");
}
"""


def test_rows_read_ahead_are_the_threads_own(tmp_path):
    host_build.run(tmp_path, PROGRAM)
