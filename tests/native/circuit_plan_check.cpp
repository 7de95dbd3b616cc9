// Host check of the gate-list planner (qibojit_amd/csrc/qj_circuit.hip).
// Random gate lists go through qj_run_gates; the entry points it calls are
// replaced by ones that carry out their documented semantics
// (include/qjhip.h) on host memory, and the state they leave is compared
// with the gates applied one by one in the order of the list.  Exit status 0
// when every case agrees; prints one line per case.
#include <cstdarg>
#include <cstdio>
#include <random>

#include "../../qibojit_amd/csrc/qj_circuit.hip"

namespace qj {
int set_error(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vprintf(fmt, ap);
  va_end(ap);
  printf("\n");
  return code;
}
// The rule of the launch (qj_tile.hip) on 256 CUs.
bool tile_per_cu(u64 ntiles) { return ntiles <= 256; }
int tile_register_bits(int dtype, int maxk, bool one_per_cu) {
  const int most = dtype == QJ_COMPLEX128 ? 4 : 5;
  const int bits = std::max(maxk, dtype == QJ_COMPLEX128 && one_per_cu ? 3 : 4);
  return bits <= most ? bits : 0;
}
}  // namespace qj

static int g_permuted = 0, g_segments = 0;

// Register layouts of the pass's plan (0 where the LDS kernel runs it).
static int segments(int dtype, int nq, int low, const int32_t* high, int nhigh, const int32_t* source_bits,
                    const qj_tile_op* ops, int nops, const char* data) {
  int maxk = 0, spos[kRegMaxBits];
  for (int o = 0; o < nops; ++o)
    if (ops[o].kind == QJ_TILE_DENSE) maxk = std::max(maxk, ops[o].k);
  RegPlanIn in;
  std::memset(&in, 0, sizeof(in));
  in.TB = low + nhigh;
  in.NRB = tile_register_bits(dtype, maxk, tile_per_cu(u64(1) << (nq - in.TB)));
  if (!in.NRB) return 0;
  in.S = dtype == QJ_COMPLEX64 ? 5 : 4;
  in.esize = (int)elem_size(dtype);
  const int nout = nq - in.TB;
  in.ga = (nout + 1) / 2;
  in.gb = nout - in.ga;
  for (int b = 0; b < in.TB; ++b) in.gpos[b] = b < low ? b : high[b - low];
  for (int b = 0; source_bits && b < in.TB; ++b) spos[b] = source_bits[in.gpos[b]];
  in.spos = source_bits ? spos : nullptr;
  in.ops = ops;
  in.nops = nops;
  in.data = data;
  in.lds_cap = kRegPlanLds;
  std::vector<char> plan;
  return reg_plan(in, plan) ? reinterpret_cast<const RegHead*>(plan.data())->nseg : 0;
}

template <typename R>
static int host_pass(const void* source, const int32_t* source_bits, void* state, int nq, int low, const int32_t* high,
                     int nhigh, const qj_tile_op* ops, int nops, const char* data) {
  const u64 n = u64(1) << nq;
  std::vector<int> tile;
  for (int b = 0; b < low; ++b) tile.push_back(b);
  for (int j = 0; j < nhigh; ++j) {
    if (j && high[j] <= high[j - 1]) return 1;
    tile.push_back(high[j]);
  }
  const int TB = (int)tile.size();
  std::vector<int> outside;
  for (int b = 0; b < nq; ++b)
    if (std::find(tile.begin(), tile.end(), b) == tile.end()) outside.push_back(b);
  std::vector<c128> x(n, 0.0);
  const cplx<R>* src = static_cast<const cplx<R>*>(source);
  cplx<R>* st = static_cast<cplx<R>*>(state);
  if (!src) x[0] = 1;
  for (u64 i = 0; src && i < n; ++i) {
    u64 j = source_bits ? 0 : i;
    for (int b = 0; source_bits && b < nq; ++b) j |= ((i >> b) & 1) << source_bits[b];
    x[i] = c128(src[j].re, src[j].im);
  }
  const int nout = (int)outside.size(), ga = (nout + 1) / 2;
  auto value = [](const cplx<R>* p) { return c128(p->re, p->im); };
  auto local = [&](u64 i) {
    u64 e = 0;
    for (int b = 0; b < TB; ++b) e |= ((i >> tile[b]) & 1) << b;
    return e;
  };
  for (int o = 0; o < nops; ++o) {
    const qj_tile_op& op = ops[o];
    auto on = [&](u64 i) {
      return (i & op.global_ctrl) == op.global_ctrl && (local(i) & op.local_ctrl) == op.local_ctrl;
    };
    if (op.kind == QJ_TILE_SWAP) {
      const u64 a = u64(1) << tile[op.target[0]], b = u64(1) << tile[op.target[1]];
      for (u64 i = 0; i < n; ++i)
        if ((i & a) && !(i & b)) std::swap(x[i], x[i ^ a ^ b]);
    } else if (op.kind == QJ_TILE_DENSE) {
      const int N = 1 << op.k;
      const cplx<R>* m = reinterpret_cast<const cplx<R>*>(data + op.offset);
      u64 mask = 0;
      for (int u = 0; u < op.k; ++u) mask |= u64(1) << tile[op.target[u]];
      for (u64 i = 0; i < n; ++i) {
        if ((i & mask) || !on(i)) continue;
        std::vector<u64> at(N, i);
        std::vector<c128> in(N);
        for (int r = 0; r < N; ++r) {
          for (int u = 0; u < op.k; ++u)
            if ((r >> (op.k - 1 - u)) & 1) at[r] |= u64(1) << tile[op.target[u]];
          in[r] = x[at[r]];
        }
        for (int r = 0; r < N; ++r) {
          c128 acc = 0;
          for (int c = 0; c < N; ++c) acc += value(m + r * N + c) * in[c];
          x[at[r]] = acc;
        }
      }
    } else if (op.kind == QJ_TILE_SCALE) {
      const c128 z = value(reinterpret_cast<const cplx<R>*>(data + op.offset));
      for (u64 i = 0; i < n; ++i)
        if (on(i)) x[i] *= z;
    } else if (op.kind == QJ_TILE_PHASE) {
      const cplx<R>* oa = reinterpret_cast<const cplx<R>*>(data + op.offset + 16);
      const cplx<R>* ob = oa + (size_t(1) << ga);
      const cplx<R>* w = ob + (size_t(1) << (nout - ga));
      for (u64 i = 0; i < n; ++i) {
        if (!on(i)) continue;
        u64 t = 0;
        for (int r = 0; r < nout; ++r) t |= ((i >> outside[r]) & 1) << r;
        c128 f = value(oa + (t & ((u64(1) << ga) - 1))) * value(ob + (t >> ga));
        for (int b = 0; b < TB; ++b)
          if ((local(i) >> b) & 1) f *= value(w + b);
        x[i] *= f;
      }
    } else {
      return 1;
    }
  }
  for (u64 i = 0; i < n; ++i) st[i] = mk<R>((R)x[i].real(), (R)x[i].imag());
  return 0;
}

extern "C" int qj_apply_tile_pass_permuted(const void* source, const int32_t* source_bits, void* state, int dtype,
                                           int nqubits, int low_bits, const int32_t* high_bits, int nhigh,
                                           const qj_tile_op* ops, int nops, const void* data, uint64_t, void*) {
  g_permuted += source_bits != nullptr;
  const char* d = static_cast<const char*>(data);
  g_segments = std::max(g_segments, segments(dtype, nqubits, low_bits, high_bits, nhigh, source_bits, ops, nops, d));
  return dtype == QJ_COMPLEX64
             ? host_pass<float>(source, source_bits, state, nqubits, low_bits, high_bits, nhigh, ops, nops, d)
             : host_pass<double>(source, source_bits, state, nqubits, low_bits, high_bits, nhigh, ops, nops, d);
}
template <typename R>
static void host_swaps(void* state, int nq, const int32_t* pairs, int npairs) {
  cplx<R>* st = static_cast<cplx<R>*>(state);
  for (int p = 0; p < npairs; ++p) {
    const u64 a = u64(1) << pairs[2 * p], b = u64(1) << pairs[2 * p + 1];
    for (u64 i = 0; i < u64(1) << nq; ++i)
      if ((i & a) && !(i & b)) std::swap(st[i], st[i ^ a ^ b]);
  }
}
extern "C" int qj_apply_bit_swaps(void* state, int dtype, int nqubits, const int32_t* pairs, int npairs, void*) {
  if (dtype == QJ_COMPLEX64) host_swaps<float>(state, nqubits, pairs, npairs);
  else host_swaps<double>(state, nqubits, pairs, npairs);
  return 0;
}
extern "C" int qj_memcpy_dtod(void* dst, const void* src, uint64_t nbytes, void*) {
  std::memcpy(dst, src, nbytes);
  return 0;
}
extern "C" int qj_initial_state(void* state, int dtype, uint64_t n, void*) {
  std::memset(state, 0, n * elem_size(dtype));
  if (dtype == QJ_COMPLEX64) static_cast<float*>(state)[0] = 1;
  else static_cast<double*>(state)[0] = 1;
  return 0;
}

// The gates one by one: target matrix under controls on explicit bits.
static void apply_gate(std::vector<c128>& x, const std::vector<int>& tg, u64 ctrl, const std::vector<c128>& m) {
  const int k = (int)tg.size(), N = 1 << k;
  u64 mask = 0;
  for (int b : tg) mask |= u64(1) << b;
  for (u64 i = 0; i < x.size(); ++i) {
    if ((i & mask) || (i & ctrl) != ctrl) continue;
    std::vector<u64> at(N, i);
    std::vector<c128> in(N);
    for (int r = 0; r < N; ++r) {
      for (int u = 0; u < k; ++u)
        if ((r >> (k - 1 - u)) & 1) at[r] |= u64(1) << tg[u];
      in[r] = x[at[r]];
    }
    for (int r = 0; r < N; ++r) {
      c128 acc = 0;
      for (int c = 0; c < N; ++c) acc += m[r * N + c] * in[c];
      x[at[r]] = acc;
    }
  }
}

static std::vector<c128> textbook(int code, const double* p) {
  const c128 i(0, 1);
  const double s = std::sqrt(0.5), pi = std::acos(-1.0);
  auto e = [&](double a) { return std::exp(i * a); };
  switch (code) {
    case QJ_GATE_SWAP: return {1, 0, 0, 0, 0, 0, 1, 0, 0, 1, 0, 0, 0, 0, 0, 1};
    case QJ_GATE_X: return {0, 1, 1, 0};
    case QJ_GATE_Y: return {0, -i, i, 0};
    case QJ_GATE_Z: return {1, 0, 0, -1};
    case QJ_GATE_H: return {s, s, s, -s};
    case QJ_GATE_S: return {1, 0, 0, i};
    case QJ_GATE_SDG: return {1, 0, 0, -i};
    case QJ_GATE_T: return {1, 0, 0, e(pi / 4)};
    case QJ_GATE_TDG: return {1, 0, 0, e(-pi / 4)};
    case QJ_GATE_SX: return {0.5 + 0.5 * i, 0.5 - 0.5 * i, 0.5 - 0.5 * i, 0.5 + 0.5 * i};
    case QJ_GATE_SXDG: return {0.5 - 0.5 * i, 0.5 + 0.5 * i, 0.5 + 0.5 * i, 0.5 - 0.5 * i};
    case QJ_GATE_RX: return {std::cos(p[0] / 2), -i * std::sin(p[0] / 2), -i * std::sin(p[0] / 2), std::cos(p[0] / 2)};
    case QJ_GATE_RY: return {std::cos(p[0] / 2), -std::sin(p[0] / 2), std::sin(p[0] / 2), std::cos(p[0] / 2)};
    case QJ_GATE_RZ: return {e(-p[0] / 2), 0, 0, e(p[0] / 2)};
    case QJ_GATE_U1: return {1, 0, 0, e(p[0])};
    case QJ_GATE_U2:
      return {e(-(p[0] + p[1]) / 2) * s, -e(-(p[0] - p[1]) / 2) * s, e((p[0] - p[1]) / 2) * s, e((p[0] + p[1]) / 2) * s};
    default: {
      const double c = std::cos(p[0] / 2), q = std::sin(p[0] / 2);
      return {e(-(p[1] + p[2]) / 2) * c, -e(-(p[1] - p[2]) / 2) * q, e((p[1] - p[2]) / 2) * q, e((p[1] + p[2]) / 2) * c};
    }
  }
}

// mix 0: everything; 1: phases and Hadamards (QFT-like); 2: swaps and few
// others; `tail`: swaps of all qubits at the end.
template <typename R>
static int check(std::mt19937_64& rng, int nq, bool density, int low, int max_high, int count, int mix, bool tail,
                 int from, double tol) {
  const int nbits = density ? 2 * nq : nq, dtype = sizeof(R) == 4 ? QJ_COMPLEX64 : QJ_COMPLEX128;
  std::uniform_real_distribution<double> U(-7.0, 7.0);
  std::normal_distribution<double> N(0.0, 1.0);
  std::vector<int32_t> recs;
  std::vector<double> params;
  const u64 n = u64(1) << nbits;
  std::vector<c128> x(n);
  std::vector<cplx<R>> src(n), st(n);
  double norm = 0;
  for (auto& v : x) {
    v = c128(N(rng), N(rng));
    norm += std::norm(v);
  }
  for (u64 i = 0; i < n; ++i) {
    x[i] /= std::sqrt(norm);
    src[i] = mk<R>((R)x[i].real(), (R)x[i].imag());
    x[i] = from == 2 ? c128(i == 0 ? 1 : 0) : c128(src[i].re, src[i].im);
    st[i] = from == 0 ? src[i] : mk<R>((R)7, (R)-7);
  }
  auto push = [&](int code, std::vector<int> q, int nt, const std::vector<double>& p) {
    recs.push_back(code);
    recs.push_back(nt);
    recs.push_back((int)q.size() - nt);
    for (int v : q) recs.push_back(v);
    params.insert(params.end(), p.begin(), p.end());
    std::vector<c128> m;
    if (code <= QJ_GATE_DENSE_BITS)
      for (size_t j = 0; j < p.size(); j += 2) m.push_back(c128(p[j], p[j + 1]));
    else
      m = textbook(code, p.data());
    const int top = nbits - 1;
    std::vector<int> tg;
    u64 ctrl = 0;
    for (int j = 0; j < (int)q.size(); ++j)
      if (j < nt) tg.push_back(top - q[j]);
      else ctrl |= u64(1) << (top - q[j]);
    apply_gate(x, tg, ctrl, m);
    if (!density || code == QJ_GATE_DENSE_BITS) return;
    for (int& b : tg) b -= nq;
    for (c128& v : m) v = std::conj(v);
    apply_gate(x, tg, ctrl >> nq, m);
  };
  const int kmax = std::min({QJ_TILE_MAX_K, max_high > 0 ? max_high : low, nq});
  for (int g = 0; g < count; ++g) {
    std::vector<int> q(nq);
    for (int b = 0; b < nq; ++b) q[b] = b;
    std::shuffle(q.begin(), q.end(), rng);
    const int pick = mix == 0 ? (int)(rng() % 10) : mix == 1 ? 10 : 11;
    if (pick == 0) {  // a dense matrix, sometimes on bits of both halves
      const bool raw = rng() % 2;
      const int k = 1 + (int)(rng() % (raw ? std::min(kmax, nbits) : kmax));
      std::vector<int> t(raw ? nbits : nq);
      for (int b = 0; b < (int)t.size(); ++b) t[b] = b;
      std::shuffle(t.begin(), t.end(), rng);
      const int nc = (int)t.size() > k ? (int)(rng() % 2) : 0;
      t.resize(k + nc);
      std::vector<double> p(size_t(2) << (2 * k));
      for (double& v : p) v = N(rng) / std::sqrt((double)(2 << k));
      push(raw ? QJ_GATE_DENSE_BITS : QJ_GATE_DENSE, t, k, p);
    } else if (pick == 1) {  // a diagonal matrix of phases
      const c128 a = std::polar(1.0, U(rng)), b = std::polar(1.0, U(rng));
      push(QJ_GATE_DENSE, {q[0]}, 1, {a.real(), a.imag(), 0, 0, 0, 0, b.real(), b.imag()});
    } else if (pick == 2 || (pick == 11 && rng() % 2)) {  // one swap or a run of them
      const int m = 1 + (int)(rng() % (nq / 2 + 1));
      for (int j = 0; j < m && 2 * j + 1 < nq; ++j) push(QJ_GATE_SWAP, {q[2 * j], q[2 * j + 1]}, 2, {});
    } else {
      int code = QJ_GATE_X + (int)(rng() % (QJ_GATE_LAST - QJ_GATE_X + 1));
      if (pick == 10) {
        const int phases[] = {QJ_GATE_U1, QJ_GATE_U1, QJ_GATE_Z, QJ_GATE_T, QJ_GATE_RZ, QJ_GATE_S, QJ_GATE_H};
        code = phases[rng() % 7];
      }
      const int np = nparams_of(code);
      std::vector<double> p(np);
      for (double& v : p) v = U(rng);
      int nc = (int)(rng() % 3);
      if (pick == 10) nc = code == QJ_GATE_H ? 0 : 1 + (int)(rng() % 4 == 0);
      q.resize(1 + std::min(nc, nq - 1));
      push(code, q, 1, p);
    }
  }
  if (tail)
    for (int q = 0; q < nq / 2; ++q) push(QJ_GATE_SWAP, {q, nq - 1 - q}, 2, {});
  g_permuted = 0;
  int32_t planned = 0, only = 0;
  const void* source = from == 1 ? src.data() : nullptr;
  int rc = qj_run_gates(source, from != 0, st.data(), dtype, nq, density, low, max_high, recs.data(), (int64_t)recs.size(),
                        params.data(), (int64_t)params.size(), &planned, nullptr);
  if (!rc)
    rc = qj_run_gates(source, from != 0, nullptr, dtype, nq, density, low, max_high, recs.data(), (int64_t)recs.size(),
                      params.data(), (int64_t)params.size(), &only, nullptr);
  double err = 0, scale = 0;
  for (u64 i = 0; i < n; ++i) {
    err = std::max(err, std::abs(c128(st[i].re, st[i].im) - x[i]));
    scale = std::max(scale, std::abs(x[i]));
  }
  const bool pass = rc == 0 && err <= tol * scale && planned == only;
  std::printf("%s %s nq=%d density=%d low=%d high=%d gates=%d mix=%d tail=%d from=%d passes=%d/%d permuted=%d err=%.2e\n",
              pass ? "ok" : "FAIL", sizeof(R) == 4 ? "c64" : "c128", nq, (int)density, low, max_high, count, mix,
              (int)tail, from, planned, only, g_permuted, err / scale);
  return pass ? 0 : 1;
}

// Layers of one-target dense gates: the runs of a pass share register sets, so
// its 12 or 13 bits take one set per 3 or 4 of them and at most two more (the
// loads and the stores keep six bits on a wave's lanes).
static int layers(int nq, int dtype, int low, int per_set) {
  std::vector<int32_t> recs;
  std::vector<double> params;
  for (int g = 0; g < 10 * nq; ++g) {
    recs.insert(recs.end(), {g % 3 ? QJ_GATE_RX : QJ_GATE_U3, 1, 0, g % nq});
    params.insert(params.end(), g % 3 ? 1 : 3, 0.1 * g);
  }
  std::vector<double> st(size_t(2) << nq);
  g_segments = 0;
  const int rc = qj_run_gates(nullptr, 1, st.data(), dtype, nq, 0, low, 7, recs.data(), (int64_t)recs.size(),
                              params.data(), (int64_t)params.size(), nullptr, nullptr);
  const int limit = (low + 7 + per_set - 1) / per_set + 2;
  const bool pass = rc == 0 && g_segments > 0 && g_segments <= limit;
  std::printf("%s layers nq=%d dtype=%d segments=%d of at most %d\n", pass ? "ok" : "FAIL", nq, dtype, g_segments,
              limit);
  return pass ? 0 : 1;
}

int main() {
  std::mt19937_64 rng(20250117);
  int bad = 0;
  for (int rep = 0; rep < 8; ++rep)
    for (int from = 0; from < 3; ++from)
      for (int mix = 0; mix < 3; ++mix) {
        const bool tail = rng() % 2;
        const int count = 1 + (int)(rng() % 60);
        const int tiny = 1 + (int)(rng() % 3);
        bad += check<double>(rng, tiny, false, tiny, 0, count, mix, tail, from, 1e-10);
        bad += check<double>(rng, 8, false, 2, 5, count, mix, tail, from, 1e-10);
        bad += check<double>(rng, 9, false, 1, 3, count, mix, tail, from, 1e-10);
        bad += check<double>(rng, 10, false, 3, 6, count, mix, tail, from, 1e-10);
        bad += check<float>(rng, 9, false, 4, 5, count, mix, tail, from, 1e-3);
        bad += check<double>(rng, 4, true, 2, 4, count, mix, tail, from, 1e-10);
        bad += check<double>(rng, 5, true, 3, 5, count, mix, tail, from, 1e-10);
      }
  for (int nq : {12, 13, 14}) bad += layers(nq, QJ_COMPLEX128, 5, 3);
  for (int nq : {13, 14}) bad += layers(nq, QJ_COMPLEX64, 6, 4);
  return bad ? 1 : 0;
}
