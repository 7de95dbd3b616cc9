// Host check of the shape of the Clifford measurement loop
// (qibojit_amd/csrc/qj_cliff_plan.h): what rows_shape accepts must fit the LDS
// of a compute unit with the kernel's arrays counted one by one, and nothing
// that fits may be refused.
#include <cstdio>

#include "../../qibojit_amd/csrc/qj_cliff_plan.h"

using namespace qj;

template <bool SYM>
static int check(int n, int S, int cus, size_t cu_lds) {
  RowsPlan p;
  const bool got = rows_shape<SYM>(n, S, cus, cu_lds, &p);
  const size_t nw = (n + 31) / 32, C = 2 * (size_t)n + S;
  if (p.R != 1 && p.R != 2 && p.R != 4 && p.R != 8) return 1;
  if ((size_t)p.G * p.R < nw || (nw > 8 && p.R != 1)) return 1;
  // counters, qubits, draws, four words; rows of both halves; two copies of a row
  const size_t fixed = kRowsWaves * p.R * 16 + kRowsThreads * 4 + (SYM ? 1 : kRowsThreads) + 4 * 4;
  const size_t used = fixed + 2 * C * p.R * 4 + 2 * (2 * ((C + 63) / 64)) * 4;
  const bool fits = used <= cu_lds && p.G <= cus && p.G <= 256;
  // up to 16 bytes of padding may be refused
  const bool wrong = got ? !fits : fits && used + 16 <= cu_lds;
  if (wrong) std::printf("FAIL sym=%d n=%d S=%d cus=%d lds=%zu of %zu\n", (int)SYM, n, S, cus, used, cu_lds);
  return wrong;
}

int main() {
  int bad = 0;
  const size_t full = 160 * 1024;
  for (int n = 1; n <= 9000; ++n) {
    bad += check<false>(n, 1, 256, full);
    bad += check<true>(n, n + 1, 256, full);
  }
  for (int n : {1, 31, 32, 33, 64, 65, 128, 129, 200, 256, 257, 1000, 7000})
    for (int m = 1; m <= 20000; ++m) {
      bad += check<true>(n, m + 1, 256, full);
      bad += check<true>(n, m + 1, 32, 65536);
    }
  return bad != 0;
}
