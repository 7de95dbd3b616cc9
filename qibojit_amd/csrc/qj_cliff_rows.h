// Measurement loop of a stabilizer tableau held in LDS, one launch for all
// measured qubits.  Included by qj_clifford.hip inside its namespace.
//
// Workgroup g owns 32 R destabilizer rows j and the stabilizer rows n + j of
// the same j, every column of them as R words each (the stabilizer words are
// shifted so that both halves line up).  The row products of a random
// outcome then need nothing from other rows but row p, and one measured
// qubit costs two waits for other workgroups, one after the other:
//  * every workgroup posts its first stabilizer row with x_q = 1 (the row's
//    bits, gathered by ballots, and its index), or the parity of the
//    selected stabilizer signs when it has none;
//  * every workgroup reads all headers; the lowest index is p, and its bits
//    come from the slot of the workgroup that posted it.
// Every posted 64-bit word carries the step in its upper half, so a reader
// waits for the words themselves: no fence, and the slots of a step are free
// again two steps later (a workgroup posts step s + 1 only after it has read
// all of step s).  The launch is cooperative, so every workgroup is resident
// and every wait ends; the waits are bounded regardless, and a loop that
// gave up reports -1 random outcomes.
//
// Symbolic form (SYM): S = m + 1 sign columns instead of one, column j the
// coefficient of the j-th random outcome (measurement_forms); the tableau is
// not written back.
//
// What bounds it: a chain of m dependent steps, each two cross-XCD round trips
// (about 2.5 us together) and the update of a workgroup's slice in LDS.  The launch-
// per-phase loop took 7-8 launches per qubit.  All qubits of a random Clifford
// state, per qubit: 1.8 us at 100 qubits (one workgroup; 6.8 by columns), 3.3 at
// 300, 4.25 at 1000 (32 workgroups; 26), 7.0 at 4000.  Two or four words of rows per
// workgroup (fewer, larger) made a gate list and 1000 measured qubits 5.33 and 6.9
// ms instead of 5.19.
constexpr int kRowsMaxSpins = 1 << 22;

typedef unsigned long long post_t;

__device__ __forceinline__ void post_word(post_t* p, uint32_t tag, uint32_t v) {
  __hip_atomic_store(p, ((post_t)tag << 32) | v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits until *p carries `tag`; false after kRowsMaxSpins reads.
__device__ __forceinline__ bool await_word(post_t* p, uint32_t tag, uint32_t* v) {
  for (int i = 0; i < kRowsMaxSpins; ++i) {
    const post_t x = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if ((uint32_t)(x >> 32) == tag) {
      *v = (uint32_t)x;
      return true;
    }
  }
  return false;
}

// (a0, a1) += (b0, b1): 2-bit counters mod 4, one per bit position.
__device__ __forceinline__ void count_add(uint32_t& a0, uint32_t& a1, uint32_t b0, uint32_t b1) {
  a1 ^= b1 ^ (a0 & b0);
  a0 ^= b0;
}

// Barrier that orders LDS only: posts, samples and forms stay in flight across
// it (no thread of the workgroup reads another's global words).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// v of the lane ROR places on within its row of 16 lanes.
template <int ROR>
__device__ __forceinline__ uint32_t row_rotate(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x120 + ROR, 0xf, 0xf, true);
}
template <int ROR>
__device__ __forceinline__ void count_add_rotated(uint32_t& c0, uint32_t& c1) {
  const uint32_t b0 = row_rotate<ROR>(c0), b1 = row_rotate<ROR>(c1);
  count_add(c0, c1, b0, b1);
}
// Counters of the two halves of 32 lanes (HALVES) or of neighbouring rows of
// 16 lanes added: the swapped pair holds one side's values in each result.
template <bool HALVES>
__device__ __forceinline__ void count_add_swapped(uint32_t& c0, uint32_t& c1) {
  const auto x0 = HALVES ? __builtin_amdgcn_permlane32_swap(c0, c0, false, false)
                         : __builtin_amdgcn_permlane16_swap(c0, c0, false, false);
  const auto x1 = HALVES ? __builtin_amdgcn_permlane32_swap(c1, c1, false, false)
                         : __builtin_amdgcn_permlane16_swap(c1, c1, false, false);
  c0 = x0[0];
  c1 = x1[0];
  count_add(c0, c1, x0[1], x1[1]);
}
// Counters summed over the lanes l, l + STEP, l + 2 STEP, ... of the SPAN
// lanes that hold different ones (the wave repeats them beyond).
template <int STEP, int SPAN>
__device__ __forceinline__ void count_lanes(uint32_t& c0, uint32_t& c1) {
  if (STEP <= 1 && SPAN > 1) count_add_rotated<1>(c0, c1);
  if (STEP <= 2 && SPAN > 2) count_add_rotated<2>(c0, c1);
  if (STEP <= 4 && SPAN > 4) count_add_rotated<4>(c0, c1);
  if (STEP <= 8 && SPAN > 8) count_add_rotated<8>(c0, c1);
  if (STEP <= 16 && SPAN > 16) count_add_swapped<false>(c0, c1);
  if (STEP <= 32 && SPAN > 32) count_add_swapped<true>(c0, c1);
}

// Exponents of i of the products of row p (masks mx, mz of its bits of a
// column pair) with 32 rows (X, Z) into their counters: A marks the rows that
// anticommute with it there, f those of them with exponent +1 (the cases of
// k_cliff_rowsum_sliced without branches).
__device__ __forceinline__ void count_product(uint32_t mx, uint32_t mz, uint32_t X, uint32_t Z, uint32_t& c0,
                                              uint32_t& c1) {
  const uint32_t A = (Z & mx) ^ (X & mz);
  const uint32_t f = (mz & (Z ^ ~mx)) | (~mz & X);
  c1 ^= A & ~(c0 ^ f);
  c0 ^= A;
}

struct RowsArgs {
  const uint32_t* tab;
  uint32_t* out;          // not SYM: the tableau again where its one workgroup writes it, else null
  int64_t ws;
  int n, m, S;            // qubits, measured qubits, sign columns
  const int32_t* qubits;
  const uint8_t* draws;   // not SYM
  post_t* hdr;            // [2][G]
  post_t* data;           // [2][G][dw]
  int dw;                 // 64-bit data words of a slot = LDS words of a row
  uint32_t* stage;        // not SYM: [2][2n + 1][G * R] destabilizer, stabilizer words
  uint32_t* scratch;      // not SYM: [G][dw + 1] partial scratch rows, sign last
  int32_t* det_any;       // not SYM: whether a determined outcome set the scratch row
  int32_t* sample;        // not SYM: [m]
  uint8_t* forms;         // SYM: [m][m + 1], zeroed
  int32_t* nrandom;
};

// Word w of a tableau column from its destabilizer words de and stabilizer
// words st (nw each): the latter start at bit n.  Bit 2n, the scratch row's, is
// `sum`, or stays what it is in `old` unless it was `set`.
__device__ __forceinline__ uint32_t merged_word(const uint32_t* de, const uint32_t* st, int nw, int n, int64_t w,
                                                bool set, uint32_t sum, uint32_t old) {
  uint32_t v = 0;
  if (w < nw) v = de[w] & rows_below(w, n);
  // stabilizer rows n + i, i = 32 w - n + bit
  const int64_t i0 = w * 32 - n;
  if (i0 > -32) {
    uint64_t pair = 0;
    const int64_t f = i0 >> 5;  // floor
    if (f >= 0 && f < nw) pair = st[f];
    if (f + 1 < nw) pair |= (uint64_t)st[f + 1] << 32;
    v |= (uint32_t)(pair >> (i0 & 31)) & rows_below(w, 2 * (int64_t)n) & ~rows_below(w, n);
  }
  const int64_t s2 = 2 * (int64_t)n;
  if (w == (s2 >> 5)) v |= (set ? sum : (old >> (s2 & 31)) & 1u) << (s2 & 31);
  return v;
}

template <int R, bool SYM>
__global__ __launch_bounds__(kRowsThreads) void k_cliff_measure_rows(RowsArgs a) {
  extern __shared__ uint32_t rows_lds[];
  __shared__ RowsShared<R, SYM> sh;
  const int t = (int)threadIdx.x, lane = t & 63, wave = t >> 6;
  const int g = (int)blockIdx.x, G = (int)gridDim.x;
  const int n = a.n, C = 2 * n + a.S, w0 = g * R, nw = (n + 31) >> 5;
  uint32_t* DE = rows_lds;
  uint32_t* ST = DE + (size_t)C * R;
  uint32_t* rowp = ST + (size_t)C * R;
  uint32_t* scr = rowp + a.dw;
  const int nchunk = (C + 63) >> 6;  // 2 * nchunk == dw
  {
    // eight words of each half in flight per thread: a column's words are one
    // stride of the tableau apart, so every load is a memory round trip
    constexpr int U = 8;
    const int sh = n & 31;
    for (int e0 = t; e0 < C * R; e0 += U * kRowsThreads) {
      uint32_t d[U], lo[U], hi[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * kRowsThreads, c = e / R, w = w0 + e % R;
        d[u] = lo[u] = hi[u] = 0;
        if (e < C * R && c <= 2 * n && w < nw) {
          const uint32_t* col = a.tab + (int64_t)c * a.ws;
          const int64_t f = ((int64_t)n + (int64_t)w * 32) >> 5;  // bits n+32w .. n+32w+31 of the column
          d[u] = col[w];
          lo[u] = col[f];
          if (f + 1 < a.ws) hi[u] = col[f + 1];
        }
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int e = e0 + u * kRowsThreads;
        if (e >= C * R) break;
        const uint32_t mask = rows_below(w0 + e % R, n);
        DE[e] = d[u] & mask;
        ST[e] = (uint32_t)((((uint64_t)hi[u] << 32) | lo[u]) >> sh) & mask;
      }
    }
  }
  int count = 0;
  bool det_any = false, ok = true;
  uint32_t scr_sign = 0;
  int drawn = 0;  // random outcomes before sh.draw[0]
  lds_barrier();
  for (int i = 0; i < a.m; ++i) {
    const uint32_t tag = (uint32_t)i + 1;
    if ((i & (kRowsThreads - 1)) == 0) {  // uniform; the barrier above closed the last reads
      sh.q[t] = i + t < a.m ? a.qubits[i + t] : 0;
      if (!SYM) sh.draw[t] = count + t < a.m ? a.draws[count + t] : 0;
      drawn = count;
      lds_barrier();
    }
    const int q = sh.q[i & (kRowsThreads - 1)];
    const uint32_t draw = SYM ? 0u : (sh.draw[count - drawn] & 1u);
    uint32_t hD[R], hS[R];
    int cand = -1;
    uint32_t par = 0;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      hD[r] = DE[q * R + r];
      hS[r] = ST[q * R + r];
      if (hS[r] && cand < 0) cand = r * 32 + __builtin_ctz(hS[r]);
      par ^= hD[r] & ST[2 * n * R + r];
    }
    par = (uint32_t)__builtin_popcount(par) & 1u;
    post_t* hdr = a.hdr + (size_t)(i & 1) * G;
    post_t* data = a.data + (size_t)(i & 1) * G * a.dw;
    if (cand >= 0) {
      const int r0 = cand >> 5, b0 = cand & 31;
      for (int ch = wave; ch < nchunk; ch += kRowsWaves) {
        const int c = ch * 64 + lane;
        const uint64_t bits = __ballot(c < C && ((ST[(c < C ? c : 0) * R + r0] >> b0) & 1u));
        if (lane < 2) {
          const uint32_t v = (uint32_t)(bits >> (32 * lane));
          rowp[2 * ch + lane] = v;
          if (G > 1) post_word(data + (size_t)g * a.dw + 2 * ch + lane, tag, v);
        }
      }
    } else if (SYM) {  // partial forms: parity of every sign column over the selected rows
      for (int ch = wave; ch < (a.S + 63) >> 6; ch += kRowsWaves) {
        const int j = ch * 64 + lane;
        uint32_t v = 0;
        if (j < a.S)
#pragma unroll
          for (int r = 0; r < R; ++r) v ^= hD[r] & ST[(2 * n + j) * R + r];
        const uint64_t bits = __ballot(__builtin_popcount(v) & 1);
        if (lane < 2) {
          const uint32_t x = (uint32_t)(bits >> (32 * lane));
          rowp[2 * ch + lane] = x;
          if (G > 1) post_word(data + (size_t)g * a.dw + 2 * ch + lane, tag, x);
        }
      }
    }
    if (G > 1) {
      if (t == 0) post_word(hdr + g, tag, cand >= 0 ? (uint32_t)(w0 * 32 + cand + 1) : par << 31);
      if (wave == 0) {
        int best = 0x7fffffff;
        uint32_t px = 0;
        bool got = true;
        for (int b = lane; b < G; b += 64) {
          uint32_t v = 0;
          got = got && await_word(hdr + b, tag, &v);
          const int idx = (int)(v & 0x7fffffffu);
          if (idx && idx - 1 < best) best = idx - 1;
          px ^= v >> 31;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
          best = min(best, __shfl_xor(best, off, 64));
          px ^= (uint32_t)__shfl_xor((int)px, off, 64);
        }
        const bool all = __all(got);
        if (lane == 0) {
          sh.best = best;
          sh.par = px;
          sh.ok = all;
          sh.fetched = 1;
        }
      }
    }
    lds_barrier();
    int best = cand >= 0 ? cand : 0x7fffffff;
    uint32_t parity = par;
    if (G > 1) {
      best = sh.best;
      parity = sh.par;
      ok = sh.ok;
      if (!ok) break;  // uniform
    }
    if (best != 0x7fffffff) {
      const int owner = best / (32 * R), pr = (best >> 5) % R;
      const uint32_t pbit = 1u << (best & 31);
      const bool mine = owner == g;
      if (!mine) {
        bool got = true;
        for (int w = t; w < 2 * nchunk; w += kRowsThreads) {
          uint32_t v = 0;
          got = got && await_word(data + (size_t)owner * a.dw + w, tag, &v);
          rowp[w] = v;
        }
        if (!got) sh.fetched = 0;
        lds_barrier();
        ok = sh.fetched;
        if (!ok) break;  // uniform
      }
      const int r = t % R;
      uint32_t hd = 0, hs = 0;
#pragma unroll
      for (int x = 0; x < R; ++x)
        if (x == r) {
          hd = hD[x];
          hs = hS[x];
        }
      const bool own = mine && r == pr;
      if (own) hs &= ~pbit;
      uint32_t d0 = 0, d1 = 0, s0 = 0, s1 = 0;
      if (hd | hs | (uint32_t)own) {
        for (int e = t; e < n * R; e += kRowsThreads) {
          const int k = e / R;
          const int xe = e, ze = (n + k) * R + r;
          const uint32_t mx = 0u - ((rowp[k >> 5] >> (k & 31)) & 1u);
          const uint32_t mz = 0u - ((rowp[(n + k) >> 5] >> ((n + k) & 31)) & 1u);
          uint32_t X = DE[xe], Z = DE[ze], Y = ST[xe], V = ST[ze];
          count_product(mx, mz, X, Z, d0, d1);
          count_product(mx, mz, Y, V, s0, s1);
          X ^= hd & mx;
          Z ^= hd & mz;
          Y ^= hs & mx;
          V ^= hs & mz;
          if (own) {  // row p - n <- row p, row p <- z_q
            X = (X & ~pbit) | (mx & pbit);
            Z = (Z & ~pbit) | (mz & pbit);
            Y &= ~pbit;
            V = (V & ~pbit) | (k == q ? pbit : 0u);
          }
          DE[xe] = X;
          DE[ze] = Z;
          ST[xe] = Y;
          ST[ze] = V;
        }
      }
      count_lanes<R, 64>(d0, d1);
      count_lanes<R, 64>(s0, s1);
      if (lane < R) sh.cnt[wave * R + lane] = make_uint4(d0, d1, s0, s1);
      lds_barrier();
      ++count;
      {
        // every wave adds the waves' counters: lane l those of rows l % R
        const uint4 v = sh.cnt[lane % (kRowsWaves * R)];
        d0 = v.x;
        d1 = v.y;
        s0 = v.z;
        s1 = v.w;
        count_lanes<R, kRowsWaves * R>(d0, d1);
        count_lanes<R, kRowsWaves * R>(s0, s1);
        for (int e = t; e < a.S * R; e += kRowsThreads) {
          const int j = e / R, c = 2 * n + j, se = c * R + r;
          const uint32_t bp = (rowp[c >> 5] >> (c & 31)) & 1u;
          const uint32_t rp = bp ? ~0u : 0u, odd = j == 0 ? ~0u : 0u;
          uint32_t x = DE[se];
          const uint32_t ev = x ^ rp ^ (j == 0 ? d1 : 0u);
          x = (x & ~hd) | (hd & ~d0 & ev) | (hd & d0 & odd);
          uint32_t y = ST[se];
          const uint32_t ew = y ^ rp ^ (j == 0 ? s1 : 0u);
          y = (y & ~hs) | (hs & ~s0 & ew) | (hs & s0 & odd);
          if (own) {
            x = (x & ~pbit) | (bp ? pbit : 0u);
            const bool set = SYM ? j == count : draw != 0;
            y = (y & ~pbit) | (set ? pbit : 0u);
          }
          DE[se] = x;
          ST[se] = y;
        }
      }
      if (g == 0 && t == 0) {
        if (SYM) a.forms[(size_t)i * (a.m + 1) + count] = 1;
        else a.sample[i] = (int32_t)draw;
      }
    } else if (SYM) {
      if (g == 0) {  // form of the determined outcome: the partial forms' sum
        bool got = true;
        for (int w = t; w < (a.S + 31) >> 5; w += kRowsThreads) {
          uint32_t sum = rowp[w];
          for (int b = 1; b < G; ++b) {
            uint32_t v = 0;
            got = got && await_word(data + (size_t)b * a.dw + w, tag, &v);
            sum ^= v;
          }
          for (int j = 0; j < 32 && 32 * w + j < a.S; ++j)
            a.forms[(size_t)i * (a.m + 1) + 32 * w + j] = (uint8_t)((sum >> j) & 1u);
        }
        if (!got) sh.fetched = 0;
      }
    } else {
      det_any = true;
      scr_sign = par;
      for (int ch = wave; ch < nchunk; ch += kRowsWaves) {
        const int c = ch * 64 + lane;
        uint32_t v = 0;
        if (c < 2 * n)
#pragma unroll
          for (int r = 0; r < R; ++r) v ^= hD[r] & ST[c * R + r];
        const uint64_t bits = __ballot(__builtin_popcount(v) & 1);
        if (lane < 2) scr[2 * ch + lane] = (uint32_t)(bits >> (32 * lane));
      }
      if (g == 0 && t == 0) a.sample[i] = (int32_t)parity;
    }
    lds_barrier();  // the step's words, counters and sh are read before the next writes
    if (SYM && G > 1 && g == 0) {
      ok = sh.fetched;
      lds_barrier();  // read before the next step sets it
      if (!ok) break;   // uniform
    }
  }
  if (!SYM && a.out) {
    const int64_t W = (2 * (int64_t)n + 1 + 31) / 32;
    for (int64_t e = t; e < (2 * (int64_t)n + 1) * W; e += kRowsThreads) {
      const int64_t c = e / W, w = e - c * W;
      const int word = c == 2 * n ? 0 : (int)(c >> 5), sh = c == 2 * n ? 0 : (int)(c & 31);
      const uint32_t sum = det_any ? (c == 2 * n ? scr_sign : scr[word] >> sh) & 1u : 0u;
      uint32_t* p = a.out + c * a.ws + w;
      *p = merged_word(DE + c * R, ST + c * R, R, n, w, det_any, sum, *p);
    }
  } else if (!SYM) {
    const int nwp = G * R;
    for (int e = t; e < (2 * n + 1) * R; e += kRowsThreads) {
      const int c = e / R, w = w0 + e % R;
      a.stage[(size_t)c * nwp + w] = DE[e];
      a.stage[((size_t)(2 * n + 1) + c) * nwp + w] = ST[e];
    }
    for (int w = t; w < a.dw; w += kRowsThreads) a.scratch[(size_t)g * (a.dw + 1) + w] = det_any ? scr[w] : 0u;
    if (t == 0) a.scratch[(size_t)g * (a.dw + 1) + a.dw] = scr_sign;
    if (g == 0 && t == 0) a.det_any[0] = det_any;
  }
  // a workgroup that gave up stops posting, so workgroup 0 gives up too
  if (g == 0 && t == 0) a.nrandom[0] = ok ? count : -1;
}

// Tableau words from the staged rows: thread per (column, word).  The scratch
// row is the sum of the workgroups' partial rows (eight loads of the chain at a
// time: 188 partial rows, 6000 qubits, one by one took 100 us), or stays what it was.
__global__ void k_cliff_merge_rows(uint32_t* __restrict__ tab, int n, int64_t ws, int64_t W, RowsArgs a, int G,
                                   int R) {
  const int64_t C = 2 * (int64_t)n + 1;
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= C * W) return;
  const int64_t c = e / W, w = e - c * W;
  const int nwp = G * R;
  const int64_t s2 = 2 * (int64_t)n;
  uint32_t sum = 0;
  if (w == (s2 >> 5) && a.det_any[0]) {
    constexpr int U = 8;
    const int word = c == s2 ? a.dw : (int)(c >> 5), sh = c == s2 ? 0 : (int)(c & 31);
    const uint32_t* p = a.scratch + word;
    int g = 0;
    for (; g + U <= G; g += U) {
      uint32_t x[U];
#pragma unroll
      for (int u = 0; u < U; ++u) x[u] = p[(size_t)(g + u) * (a.dw + 1)];
#pragma unroll
      for (int u = 0; u < U; ++u) sum ^= x[u];
    }
    for (; g < G; ++g) sum ^= p[(size_t)g * (a.dw + 1)];
    sum = (sum >> sh) & 1u;
  }
  uint32_t* out = tab + c * ws + w;
  *out = merged_word(a.stage + c * nwp, a.stage + (C + c) * nwp, nwp, n, w, a.det_any[0], sum, *out);
}
