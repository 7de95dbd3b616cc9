// Fused execution of a gate list: the planner between gate records and tile
// passes.
//
// A gate becomes one op of three kinds: dense (a matrix on up to five target
// bits under control bits), phase (a one-target diagonal of modulus 1: exp(i
// (c0 + theta bit)) under controls) or swap.  Ops are taken into passes by
// list scheduling: a pass goes through the pending ops in order and takes
// every one that fits its tile and commutes with all it has left behind, so
// a pass also collects the later layers its bits allow (a two-layer 26-qubit
// ansatz runs in 6 passes, not the 12 of cutting the list in order).  Two ops
// commute when neither changes a bit (dense and swap targets) that the
// other one reads or changes; controls and phases only read.  Inside a pass,
// phase ops under one control set merge (a controlled phase without constant
// is symmetric in its two bits and may be re-rooted on the shared one: a QFT
// ladder becomes one op), and the ops are ordered so that as many dense
// targets as possible share the kernel's register bits.
//
// A circuit that ends with swaps of many bits (a QFT) and starts from another
// buffer has them moved to its front: SWAPs G = G' SWAPs with the bits of G
// exchanged, and the first pass, which reads that buffer anyway, reads it
// permuted (|0...0> is its own permutation).  The first tile then also holds
// the bits that are lowest in the source, so that its loads are whole lines.
// A 30-qubit complex64 QFT went from 19.5 to 17.1 ms, a 28-qubit complex128 one
// from 9.3 to 7.65; with 12 to 20 qubits it takes as long or up to 12% less.
//
// A pass is closed when its plan would outgrow the kernel's LDS share, counted
// item by item as the plan is laid out (what a merged phase adds, not what it
// would take alone): with a rough budget of 12 of the 15 KiB a 32-qubit
// complex128 QFT took one pass more (175 instead of 155 ms), and 20 qubits, 600
// gates 0.82 instead of 0.68 ms.
//
// The same steps in Python, cutting the list in order, took about 8 us a gate,
// more than the device needed: 20 qubits, 600 gates 5.3 -> 1.07 ms; the two-layer
// 26-qubit ansatz and its energy 5.9 -> 4.65 ms; two layers of a noisy 12-qubit
// density matrix 1.83 -> 1.17 ms.
#include <algorithm>
#include <cmath>
#include <complex>
#include <cstring>
#include <new>
#include <vector>

#include "qj_common.h"
#include "qj_tile_reg.h"

namespace qj {
namespace {

typedef std::complex<double> c128;

struct GateOp {
  int kind;              // QJ_TILE_DENSE, QJ_TILE_PHASE or QJ_TILE_SWAP
  int k;                 // targets (dense, swap)
  int tg[QJ_TILE_MAX_K]; // target bits, first = matrix MSB
  u64 ctrl;              // control bits
  u64 X, Z;              // bits changed, bits only read
  size_t mat;            // dense: first entry in the pool
  double c0, th;         // phase
  int tb;                // phase: bit of th, or -1
};

// An op of a pass; a phase item may hold several merged ops.
struct Item {
  GateOp op;
  std::vector<std::pair<int, double>> th;  // phase: (bit, angle), ascending insertion order
};

struct Run {
  const void* source;
  void* state;
  int dtype, nbits, low, max_high;
  bool from_source, plan_only, one_per_cu;
  hipStream_t stream;
  std::vector<c128> pool;
  std::vector<GateOp> ops;  // in circuit order
  std::vector<int32_t> source_bits;  // state bit -> source bit, where swaps moved to the front
  int npasses = 0;
};

u64 bit(int b) { return u64(1) << b; }

void set_masks(GateOp& op) {
  op.X = op.Z = 0;
  if (op.kind == QJ_TILE_PHASE) {
    op.Z = op.ctrl | (op.tb >= 0 ? bit(op.tb) : 0);
    return;
  }
  for (int u = 0; u < op.k; ++u) op.X |= bit(op.tg[u]);
  op.Z = op.ctrl;
}

// ------------------------------------------------------------- records --
int nparams_of(int code) {
  switch (code) {
    case QJ_GATE_RX: case QJ_GATE_RY: case QJ_GATE_RZ: case QJ_GATE_U1: return 1;
    case QJ_GATE_U2: return 2;
    case QJ_GATE_U3: return 3;
    default: return 0;
  }
}

double phase_of(c128 z) { return std::atan2(z.imag(), z.real()); }

// The gate's 2x2 matrix; the parameter-free and rotation gates of qibo.
void one_qubit_matrix(int code, const double* p, c128* m) {
  const c128 i(0, 1);
  const double s = 1.0 / std::sqrt(2.0);
  auto set = [&](c128 a, c128 b, c128 c, c128 d) {
    m[0] = a;
    m[1] = b;
    m[2] = c;
    m[3] = d;
  };
  switch (code) {
    case QJ_GATE_X: set(0, 1, 1, 0); break;
    case QJ_GATE_Y: set(0, -i, i, 0); break;
    case QJ_GATE_H: set(s, s, s, -s); break;
    case QJ_GATE_SX: set(c128(0.5, 0.5), c128(0.5, -0.5), c128(0.5, -0.5), c128(0.5, 0.5)); break;
    case QJ_GATE_SXDG: set(c128(0.5, -0.5), c128(0.5, 0.5), c128(0.5, 0.5), c128(0.5, -0.5)); break;
    case QJ_GATE_RX: {
      const double c = std::cos(p[0] / 2), q = std::sin(p[0] / 2);
      set(c, c128(0, -q), c128(0, -q), c);
      break;
    }
    case QJ_GATE_RY: {
      const double c = std::cos(p[0] / 2), q = std::sin(p[0] / 2);
      set(c, -q, q, c);
      break;
    }
    case QJ_GATE_U2: {
      const c128 e = std::polar(1.0, (p[0] + p[1]) / 2), f = std::polar(1.0, (p[0] - p[1]) / 2);
      set(std::conj(e) * s, -std::conj(f) * s, f * s, e * s);
      break;
    }
    default: {  // U3
      const double c = std::cos(p[0] / 2), q = std::sin(p[0] / 2);
      const c128 e = std::polar(1.0, (p[1] + p[2]) / 2), f = std::polar(1.0, (p[1] - p[2]) / 2);
      set(std::conj(e) * c, -std::conj(f) * q, f * q, e * c);
    }
  }
}

// Angle of a diagonal one-qubit gate: diag(e^(i c0), e^(i (c0 + th))).
bool diagonal_angles(int code, const double* p, double* c0, double* th) {
  const double pi = 3.14159265358979323846;
  *c0 = 0;
  switch (code) {
    case QJ_GATE_Z: *th = pi; return true;
    case QJ_GATE_S: *th = pi / 2; return true;
    case QJ_GATE_SDG: *th = -pi / 2; return true;
    case QJ_GATE_T: *th = pi / 4; return true;
    case QJ_GATE_TDG: *th = -pi / 4; return true;
    case QJ_GATE_U1: *th = phase_of(std::polar(1.0, p[0])); return true;
    case QJ_GATE_RZ:
      *c0 = phase_of(std::polar(1.0, -p[0] / 2));
      *th = phase_of(std::polar(1.0, p[0] / 2)) - *c0;
      return true;
    default: return false;
  }
}

// One record -> an op (and, for a density matrix, its column half: the same
// gate conjugated on the column bits).
int push_record(Run& run, int nqubits, bool density, const int32_t* rec, const double* p) {
  const int code = rec[0], nt = rec[1], nc = rec[2];
  const bool raw = code == QJ_GATE_DENSE_BITS;
  GateOp op;
  std::memset(&op, 0, sizeof(op));
  op.tb = -1;
  u64 seen = 0;
  for (int j = 0; j < nt + nc; ++j) {
    const int limit = raw ? run.nbits : nqubits;
    if (rec[3 + j] < 0 || rec[3 + j] >= limit)
      return set_error(QJ_EVALUE, "run_gates: qubit %d out of range", rec[3 + j]);
    const int b = run.nbits - 1 - rec[3 + j];
    if (seen & bit(b)) return set_error(QJ_EVALUE, "run_gates: a gate acts twice on one qubit");
    seen |= bit(b);
    if (j < nt) op.tg[j] = b;
    else op.ctrl |= bit(b);
  }
  op.k = nt;
  if (code == QJ_GATE_SWAP) {
    op.kind = QJ_TILE_SWAP;
  } else if (code == QJ_GATE_DENSE || raw) {
    const size_t n = size_t(1) << (2 * nt);
    const c128* m = reinterpret_cast<const c128*>(p);
    const bool diag = nt == 1 && m[1] == 0.0 && m[2] == 0.0 && std::abs(std::abs(m[0]) - 1) < 1e-14 &&
                      std::abs(std::abs(m[3]) - 1) < 1e-14;
    if (diag) {
      op.kind = QJ_TILE_PHASE;
      op.c0 = phase_of(m[0]);
      op.th = phase_of(m[3]) - op.c0;
      op.tb = op.tg[0];
    } else {
      op.kind = QJ_TILE_DENSE;
      op.mat = run.pool.size();
      run.pool.insert(run.pool.end(), m, m + n);
    }
  } else if (diagonal_angles(code, p, &op.c0, &op.th)) {
    op.kind = QJ_TILE_PHASE;
    op.tb = op.tg[0];
  } else {
    // no rotation by an infinite angle; NaN runs through
    if ((code == QJ_GATE_RX || code == QJ_GATE_RY || code == QJ_GATE_U3) && std::isinf(p[0]))
      return set_error(QJ_EVALUE, "run_gates: rotation angle is infinite");
    c128 m[4];
    one_qubit_matrix(code, p, m);
    op.kind = QJ_TILE_DENSE;
    op.mat = run.pool.size();
    run.pool.insert(run.pool.end(), m, m + 4);
  }
  set_masks(op);
  run.ops.push_back(op);
  if (!density || raw) return QJ_OK;
  GateOp col = op;
  for (int u = 0; u < nt; ++u) col.tg[u] -= nqubits;
  col.ctrl >>= nqubits;
  if (col.tb >= 0) col.tb -= nqubits;
  col.c0 = -col.c0;
  col.th = -col.th;
  if (col.kind == QJ_TILE_DENSE) {
    const size_t n = size_t(1) << (2 * nt);
    col.mat = run.pool.size();
    for (size_t j = 0; j < n; ++j) run.pool.push_back(std::conj(run.pool[op.mat + j]));
  }
  set_masks(col);
  run.ops.push_back(col);
  return QJ_OK;
}

// --------------------------------------------------------------- passes --
// LDS bytes of an item in the register kernel's plan (a dense op may also open
// a segment), and their budget: what the plan may take next to a tile, less the
// first and the last segment and three paddings.  A 32-qubit complex128 QFT needs
// nearly all of it in its last pass.
constexpr size_t kPassBudget = kRegPlanLds - 2 * sizeof(RegSeg) - 3 * 16;
bool one_factor(const Item& it) { return it.th.empty() || (it.th.size() == 1 && it.op.c0 == 0.0); }
size_t item_bytes(const Item& it, int esize) {
  const size_t head = sizeof(RegOp) + sizeof(u64);
  if (it.op.kind == QJ_TILE_SWAP) return 0;
  if (it.op.kind == QJ_TILE_DENSE) return head + sizeof(RegSeg) + (size_t(1) << (2 * it.op.k)) * esize;
  return head + (one_factor(it) ? 16 : (esize == 8 ? 100 : 84) * (size_t)esize);  // largest phase tables
}

bool symmetric(const Item& it) {
  return __builtin_popcountll(it.op.ctrl) == 1 && it.op.c0 == 0.0 && it.th.size() == 1;
}
void reroot(Item& it) {  // a controlled phase on its other bit
  const int c = __builtin_ctzll(it.op.ctrl), t = it.th[0].first;
  it.op.ctrl = bit(t);
  it.th[0].first = c;
}

// Merges phase op `p` into phase item `it` if both act under the same controls.
bool merge(Item& it, const Item& p) {
  for (int a = 0; a < 2; ++a) {
    if (a == 1 && !symmetric(it)) break;
    Item x = it;
    if (a == 1) reroot(x);
    for (int b = 0; b < 2; ++b) {
      if (b == 1 && !symmetric(p)) break;
      Item y = p;
      if (b == 1) reroot(y);
      if (x.op.ctrl != y.op.ctrl) continue;
      x.op.c0 += y.op.c0;
      for (auto& [yb, ya] : y.th) {
        bool found = false;
        for (auto& [xb, xa] : x.th)
          if (xb == yb) {
            xa += ya;
            found = true;
          }
        if (!found) x.th.push_back({yb, ya});
      }
      x.op.Z = it.op.Z | p.op.Z;
      it = std::move(x);
      return true;
    }
  }
  return false;
}

// What an LDS-kernel pass may take: its ops and matrices travel in one slot of
// the staging ring.  kLdsOthers: ops per one that needs the LDS kernel.
constexpr size_t kLdsBudget = kRingSlotBytes / 2;
constexpr int kLdsOthers = 8;

// Appends an op to a pass: phases join the latest item they can merge with
// while everything after it commutes with them.  False, and nothing is
// changed, if the pass's plan would grow over its budget.
bool add_item(std::vector<Item>& items, const GateOp& op, int esize, size_t* bytes, size_t budget) {
  Item it;
  it.op = op;
  if (op.kind == QJ_TILE_PHASE) {
    if (op.tb >= 0) it.th.push_back({op.tb, op.th});
    for (size_t j = items.size(), tries = 0; j-- > 0 && tries < 64; ++tries) {
      if (items[j].op.kind == QJ_TILE_PHASE) {
        Item old = items[j];
        if (merge(items[j], it)) {
          const size_t now = *bytes - item_bytes(old, esize) + item_bytes(items[j], esize);
          if (now > budget && now > *bytes) {
            items[j] = std::move(old);
            return false;
          }
          *bytes = now;
          return true;
        }
      }
      if (items[j].op.X & op.Z) break;
    }
  }
  const size_t more = item_bytes(it, esize);
  if (!items.empty() && more && *bytes + more > budget) return false;
  *bytes += more;
  items.push_back(std::move(it));
  return true;
}

// Orders the items so that runs of dense ops share the kernel's register
// bits (each new register set re-lays the tile out through LDS);
// the first run avoids the six lowest tile bits, which the loads keep on
// the lanes of a wave.
void order_items(std::vector<Item>& items, u64 lane_bits, int dtype, bool one_per_cu) {
  int maxk = 0;
  for (const Item& it : items) {
    if (it.op.kind == QJ_TILE_SWAP) return;  // swaps relabel bits on the way
    if (it.op.kind == QJ_TILE_DENSE) maxk = std::max(maxk, it.op.k);
  }
  const int nrb = tile_register_bits(dtype, maxk, one_per_cu);
  if (!nrb) return;  // the LDS kernel keeps no bits in registers
  std::vector<Item> out;
  out.reserve(items.size());
  std::vector<char> done(items.size(), 0);
  bool first = true;
  while (out.size() < items.size()) {
    u64 used = 0, bx = 0, bz = 0;
    const size_t before = out.size();
    for (size_t j = 0; j < items.size(); ++j) {
      if (done[j]) continue;
      const GateOp& op = items[j].op;
      bool take = !((op.X | op.Z) & bx) && !(op.X & bz);
      if (take && op.kind == QJ_TILE_DENSE) {
        take = !(first && (op.X & lane_bits)) && __builtin_popcountll(used | op.X) <= nrb;
        if (take) used |= op.X;
      }
      if (take) {
        done[j] = 1;
        out.push_back(std::move(items[j]));
      } else {
        bx |= op.X;
        bz |= op.Z;
      }
    }
    if (out.size() == before && !first) break;  // not reached: the first pending item is always takeable
    first = false;
  }
  items.swap(out);
}

template <typename R>
int emit_tile(Run& run, std::vector<Item>& items, u64 high) {
  const int low = std::min(run.low, run.nbits);
  int nhigh = __builtin_popcountll(high);
  for (int b = low; b < run.nbits && nhigh < run.max_high; ++b)  // widen with the lowest unused bits
    if (!(high & bit(b))) {
      high |= bit(b);
      ++nhigh;
    }
  ++run.npasses;
  if (run.plan_only) return QJ_OK;
  int32_t hb[64];
  int local[64], outside[64], rank[64];
  int tb = 0, nout = 0;
  for (int b = 0; b < run.nbits; ++b) {
    local[b] = rank[b] = -1;
    if (b < low || (high & bit(b))) {
      if (b >= low) hb[tb - low] = b;
      local[b] = tb++;
    } else {
      rank[b] = nout;
      outside[nout++] = b;
    }
  }
  const int ga = (nout + 1) / 2, gb = nout - ga;
  const bool permuted = run.from_source && !run.source_bits.empty();
  u64 lane_bits = 0;
  for (int b = 0, lanes = 0; b < run.nbits && lanes < 6; ++b) {
    const int sb = permuted ? run.source_bits[b] : b;  // the state bit that the source keeps at b
    if (local[sb] < 0) continue;
    lane_bits |= bit(sb);
    ++lanes;
  }
  order_items(items, lane_bits, run.dtype, run.one_per_cu);

  std::vector<qj_tile_op> ops;
  std::vector<char> data;
  ops.reserve(items.size());
  auto room = [&](size_t bytes) {
    const size_t off = data.size();
    data.resize(off + ((bytes + 15) & ~size_t(15)), 0);
    return off;
  };
  auto put = [](cplx<R>* p, c128 z) { *p = mk<R>((R)z.real(), (R)z.imag()); };
  std::vector<double> ang;
  for (const Item& it : items) {
    qj_tile_op o;
    std::memset(&o, 0, sizeof(o));
    u64 ctrl = it.op.ctrl;
    if (it.op.kind == QJ_TILE_SWAP) {
      o.kind = QJ_TILE_SWAP;
      o.k = 2;
      o.target[0] = local[it.op.tg[0]];
      o.target[1] = local[it.op.tg[1]];
      ops.push_back(o);
      continue;
    }
    if (it.op.kind == QJ_TILE_DENSE) {
      o.kind = QJ_TILE_DENSE;
      o.k = it.op.k;
      for (int u = 0; u < o.k; ++u) o.target[u] = local[it.op.tg[u]];
      const size_t n = size_t(1) << (2 * o.k);
      o.offset = room(n * sizeof(cplx<R>));
      cplx<R>* m = reinterpret_cast<cplx<R>*>(data.data() + o.offset);
      for (size_t j = 0; j < n; ++j) put(m + j, run.pool[it.op.mat + j]);
    } else if (one_factor(it)) {
      // one factor where every bit is 1
      o.kind = QJ_TILE_SCALE;
      if (!it.th.empty()) ctrl |= bit(it.th[0].first);
      o.offset = room(sizeof(cplx<R>));
      put(reinterpret_cast<cplx<R>*>(data.data() + o.offset),
          std::polar(1.0, it.th.empty() ? it.op.c0 : it.th[0].second));
    } else {
      o.kind = QJ_TILE_PHASE;
      const size_t na = size_t(1) << ga, nb = size_t(1) << gb;
      o.offset = room(16 + (na + nb + (size_t)tb) * sizeof(cplx<R>));
      const int32_t head[4] = {ga, gb, tb, 0};
      std::memcpy(data.data() + o.offset, head, sizeof(head));
      cplx<R>* tab = reinterpret_cast<cplx<R>*>(data.data() + o.offset + 16);
      // angle sums per table index, then one exponential each
      auto table = [&](cplx<R>* dst, int r0, int nr, double c0) {
        ang.assign(size_t(1) << nr, c0);
        bool any = false;
        for (const auto& [b, a] : it.th)
          if (rank[b] >= r0 && rank[b] < r0 + nr) {
            any = true;
            const size_t step = size_t(1) << (rank[b] - r0);
            for (size_t j = 0; j < ang.size(); ++j)
              if (j & step) ang[j] += a;
          }
        const c128 z0 = std::polar(1.0, c0);
        for (size_t j = 0; j < ang.size(); ++j) put(dst + j, any ? std::polar(1.0, ang[j]) : z0);
      };
      table(tab, 0, ga, it.op.c0);
      table(tab + na, ga, gb, 0.0);
      cplx<R>* w = tab + na + nb;
      ang.assign((size_t)tb, 0.0);
      for (const auto& [b, a] : it.th)
        if (local[b] >= 0) ang[local[b]] += a;
      for (int j = 0; j < tb; ++j) put(w + j, std::polar(1.0, ang[j]));
    }
    for (int b = 0; b < run.nbits; ++b)
      if (ctrl & bit(b)) {
        if (local[b] >= 0) o.local_ctrl |= bit(local[b]);
        else o.global_ctrl |= bit(b);
      }
    ops.push_back(o);
  }
  const void* src = run.from_source ? run.source : run.state;
  run.from_source = false;
  return qj_apply_tile_pass_permuted(src, permuted ? run.source_bits.data() : nullptr, run.state, run.dtype, run.nbits,
                                     low, hb, tb - low, ops.data(), (int)ops.size(), data.data(), data.size(),
                                     run.stream);
}

// The state itself before a pass that works in place.
int fill_state(Run& run) {
  if (!run.from_source) return QJ_OK;
  run.from_source = false;
  if (run.plan_only) return QJ_OK;
  const u64 n = u64(1) << run.nbits;
  if (!run.source) return qj_initial_state(run.state, run.dtype, n, run.stream);
  const int rc = qj_memcpy_dtod(run.state, run.source, n * elem_size(run.dtype), run.stream);
  if (rc || run.source_bits.empty()) return rc;
  std::vector<int32_t> pairs;
  for (int b = 0; b < run.nbits; ++b)
    if (b < run.source_bits[b]) {
      pairs.push_back(b);
      pairs.push_back(run.source_bits[b]);
    }
  return qj_apply_bit_swaps(run.state, run.dtype, run.nbits, pairs.data(), (int)pairs.size() / 2, run.stream);
}

// Moves swaps of many bits from the end of the circuit to its front (see the
// top).  Returns the bits to keep in the first tile for its loads.
u64 fold_swaps(Run& run, u64 low_mask) {
  if (!run.from_source || run.nbits > 56) return 0;
  u64 bits = 0;
  size_t j = run.ops.size();
  for (; j > 0 && run.ops[j - 1].kind == QJ_TILE_SWAP && !(run.ops[j - 1].X & bits); --j) bits |= run.ops[j - 1].X;
  if (j == 0 || __builtin_popcountll(bits & ~low_mask) <= run.max_high) return 0;
  std::vector<int32_t> to(run.nbits);
  for (int b = 0; b < run.nbits; ++b) to[b] = b;
  for (size_t i = j; i < run.ops.size(); ++i) std::swap(to[run.ops[i].tg[0]], to[run.ops[i].tg[1]]);
  u64 keep = 0;  // whole 128-byte lines of the source
  for (int b = 0; run.source && (elem_size(run.dtype) << b) < 128; ++b) keep |= bit(to[b]) & ~low_mask;
  if (__builtin_popcountll(keep) >= run.max_high) return 0;
  run.ops.resize(j);
  for (GateOp& op : run.ops) {
    if (op.kind == QJ_TILE_PHASE) {
      if (op.tb >= 0) op.tb = to[op.tb];
    } else {
      for (int u = 0; u < op.k; ++u) op.tg[u] = to[op.tg[u]];
    }
    u64 ctrl = 0;
    for (u64 m = op.ctrl; m; m &= m - 1) ctrl |= bit(to[__builtin_ctzll(m)]);
    op.ctrl = ctrl;
    set_masks(op);
  }
  if (run.source) run.source_bits = std::move(to);
  return keep;
}

// The pending ops in order: those that earlier passes left behind, then the
// ones no pass has looked at yet.
struct Pending {
  const std::vector<GateOp>& ops;
  std::vector<int> left;
  size_t next = 0;
  size_t size() const { return left.size() + (ops.size() - next); }
  int id(size_t i) const { return i < left.size() ? left[i] : (int)(next + i - left.size()); }
  const GateOp& operator[](size_t i) const { return ops[id(i)]; }
  // Drops the first n of the order but those in `keep`.
  void consume(size_t n, const std::vector<int>& keep) {
    std::vector<int> l(keep);
    if (n < left.size()) l.insert(l.end(), left.begin() + (long)n, left.end());
    else next += n - left.size();
    left.swap(l);
  }
};

// Length of the run of swaps on distinct bits that starts at pending op i.
size_t swap_run(const Pending& pend, size_t i, u64* bits) {
  *bits = 0;
  size_t j = i;
  for (; j < pend.size() && pend[j].kind == QJ_TILE_SWAP && !(pend[j].X & *bits); ++j) *bits |= pend[j].X;
  return j - i;
}

int run_pending(Run& run) {
  const int esize = (int)elem_size(run.dtype);
  const u64 low_mask = bit(std::min(run.low, run.nbits)) - 1;
  const u64 all = bit(run.nbits) - 1;
  // A dense op too wide for the register kernel (complex128, five targets) fills
  // its plan alone.  Where each tile has a CU to itself a pass that starts with
  // one goes on with the LDS kernel: it takes more of them, which saves a pass
  // and an upload each (16 of them on 16 qubits 1.88 -> 1.63 ms), and a few other
  // ops between.  With many other ops, or more tiles, a pass of its own is faster
  // (20 rotations each: 2.27 against 2.51 ms; 24 qubits: 9.8 against 17.8).
  run.one_per_cu = tile_per_cu(u64(1) << (run.nbits - std::min(run.nbits, run.low + run.max_high)));
  auto wide = [&](const GateOp& op) {
    return op.kind == QJ_TILE_DENSE && !tile_register_bits(run.dtype, op.k, run.one_per_cu);
  };
  u64 first_high = fold_swaps(run, low_mask);
  Pending pend{run.ops, {}, 0};
  std::vector<int> keep;
  std::vector<Item> items;
  while (pend.size()) {
    keep.clear();
    items.clear();
    u64 bits = 0;
    const size_t lead = swap_run(pend, 0, &bits);
    if (lead >= 2 && __builtin_popcountll(bits & ~low_mask) > run.max_high) {
      // a permutation of many bits: one exchange of tiles for the whole run
      std::vector<int32_t> pairs;
      for (size_t j = 0; j < lead; ++j) {
        pairs.push_back(pend[j].tg[0]);
        pairs.push_back(pend[j].tg[1]);
      }
      pend.consume(lead, keep);
      first_high = 0;
      int rc = fill_state(run);
      ++run.npasses;
      if (!rc && !run.plan_only)
        rc = qj_apply_bit_swaps(run.state, run.dtype, run.nbits, pairs.data(), (int)lead, run.stream);
      if (rc) return rc;
      continue;
    }
    u64 high = first_high, bx = 0, bz = 0;
    size_t bytes = 0, i = 0;
    int nwide = 0, nother = 0;  // of an LDS-kernel pass
    while (i < pend.size() && bx != all) {  // with every bit changed by an op left behind, none commutes
      const size_t nrun = swap_run(pend, i, &bits);
      const size_t n = nrun >= 2 ? nrun : 1;  // swaps of a run stay together
      bool take = true;
      u64 need = high;
      for (size_t j = i; j < i + n; ++j) {
        const GateOp& op = pend[j];
        take = take && !((op.X | op.Z) & bx) && !(op.X & bz);
        need |= op.X & ~low_mask;
      }
      take = take && __builtin_popcountll(need) <= run.max_high;
      for (size_t j = i; j < i + n; ++j) {
        const GateOp& op = pend[j];
        const bool lds = run.one_per_cu && (nwide || (items.empty() && wide(op)));
        if (lds && op.kind != QJ_TILE_SWAP) {
          if (wide(op)) nwide += take;
          else take = take && ++nother <= kLdsOthers * nwide;
        }
        // swaps take no room: a run is not cut
        take = take && add_item(items, op, esize, &bytes, lds ? kLdsBudget : kPassBudget);
        if (take) continue;
        bx |= op.X;
        bz |= op.Z;
        keep.push_back(pend.id(j));
      }
      if (take) high = need;
      i += n;
    }
    if (items.empty() && first_high) {  // a wide gate comes first: without the load's bits
      first_high = 0;
      continue;
    }
    first_high = 0;
    if (items.empty()) return set_error(QJ_EVALUE, "run_gates: a gate does not fit a tile");
    pend.consume(i, keep);
    const int rc = run.dtype == QJ_COMPLEX64 ? emit_tile<float>(run, items, high) : emit_tile<double>(run, items, high);
    if (rc) return rc;
  }
  return QJ_OK;
}

}  // namespace
}  // namespace qj

using namespace qj;

extern "C" int qj_run_gates(const void* source, int from_source, void* state, int dtype, int nqubits, int density,
                            int low_bits, int max_high, const int32_t* recs, int64_t nwords, const double* params,
                            int64_t nparams, int32_t* npasses, void* stream) {
  const int nbits = density ? 2 * nqubits : nqubits;
  if (nqubits < 1 || nbits > 62) return set_error(QJ_EVALUE, "run_gates: bad nqubits %d", nqubits);
  if (!is_complex(dtype)) return set_error(QJ_EVALUE, "run_gates: dtype must be complex64/complex128");
  if (nwords < 0 || nparams < 0 || (nwords > 0 && !recs) || (nparams > 0 && !params))
    return set_error(QJ_EVALUE, "run_gates: bad records");
  if (low_bits < 1 || low_bits > nbits || max_high < 0 || low_bits + max_high > nbits ||
      low_bits + max_high > QJ_TILE_MAX_BITS)
    return set_error(QJ_EVALUE, "run_gates: bad tile (low_bits=%d, max_high=%d)", low_bits, max_high);
  try {
    Run run;
    run.source = source;
    run.state = state;
    run.dtype = dtype;
    run.nbits = nbits;
    run.low = low_bits;
    run.max_high = max_high;
    run.plan_only = state == nullptr;
    run.from_source = from_source != 0;
    run.stream = (hipStream_t)stream;
    int64_t at = 0, par = 0;
    while (at < nwords) {
      if (nwords - at < 3) return set_error(QJ_EVALUE, "run_gates: truncated record");
      const int code = recs[at], nt = recs[at + 1], nc = recs[at + 2];
      if (code < 0 || code > QJ_GATE_LAST) return set_error(QJ_EVALUE, "run_gates: unknown gate code %d", code);
      const bool dense = code == QJ_GATE_DENSE || code == QJ_GATE_DENSE_BITS;
      const int want = code == QJ_GATE_SWAP ? 2 : 1;
      if (nc < 0 || (dense ? (nt < 1 || nt > QJ_TILE_MAX_K) : nt != want) || nt + nc > nbits ||
          (code == QJ_GATE_SWAP && nc) || nwords - at < 3 + (int64_t)nt + nc)
        return set_error(QJ_EVALUE, "run_gates: bad record at word %lld", (long long)at);
      const int64_t np = dense ? 2 * (int64_t(1) << (2 * nt)) : nparams_of(code);
      if (nparams - par < np) return set_error(QJ_EVALUE, "run_gates: too few parameters");
      const int rc = push_record(run, nqubits, density != 0, recs + at, params + par);
      if (rc) return rc;
      at += 3 + nt + nc;
      par += np;
    }
    int rc = run_pending(run);
    if (!rc) rc = fill_state(run);  // no gates at all
    if (npasses) *npasses = run.npasses;
    return rc;
  } catch (const std::bad_alloc&) {
    return set_error(QJ_EMEMORY, "run_gates: out of host memory");
  }
}
