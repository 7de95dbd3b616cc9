// Shape of the one-launch measurement loop (qj_cliff_rows.h) for a tableau:
// words of rows per workgroup, workgroups and LDS.  Host arithmetic only, so
// that it can be checked without a device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

namespace qj {

constexpr int kRowsThreads = 512;
constexpr int kRowsWaves = kRowsThreads / 64;

// The fixed LDS of a workgroup, beside the dynamic part (RowsPlan::lds).
template <int R, bool SYM>
struct RowsShared {
  uint4 cnt[kRowsWaves * R];
  int q[kRowsThreads];                     // the next steps' qubits
  int best, ok, fetched;
  uint32_t par;
  uint8_t draw[SYM ? 1 : kRowsThreads];    // and random bits
};

struct RowsPlan {
  int R, G, dw;  // words of rows per workgroup, workgroups, LDS words of a row
  size_t lds;    // dynamic LDS
};

template <bool SYM>
constexpr size_t rows_fixed_lds(int R) {
  return R == 1 ? sizeof(RowsShared<1, SYM>) : R == 2 ? sizeof(RowsShared<2, SYM>)
       : R == 4 ? sizeof(RowsShared<4, SYM>) : sizeof(RowsShared<8, SYM>);
}

// n qubits, S sign columns: one workgroup up to 256 qubits (no exchange, R = 1,
// 2, 4 or 8), else 32 rows each.  False unless every workgroup is resident and
// its slice fits `cu_lds` bytes together with the fixed part.
template <bool SYM>
inline bool rows_shape(int n, int S, int cus, size_t cu_lds, RowsPlan* p) {
  const int nw = (n + 31) / 32;
  p->R = 1;
  if (nw <= 8)
    while (p->R < nw) p->R *= 2;
  p->G = (nw + p->R - 1) / p->R;
  const int64_t C = 2 * (int64_t)n + S;
  p->dw = (int)(2 * ((C + 63) / 64));
  p->lds = ((size_t)2 * C * p->R + 2 * (size_t)p->dw) * sizeof(uint32_t);
  return p->G <= cus && p->G <= 256 && p->lds + rows_fixed_lds<SYM>(p->R) <= cu_lds;
}

}  // namespace qj
