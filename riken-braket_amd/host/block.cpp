// Gate-block planner and its C ABI (brk_block_plan_*, brk_circuit_run_blocked).
//
// The circuit's ops are walked in order with the logical -> physical qubit
// map (as brk_circuit_run_timed does).  Consecutive ops are grouped greedily;
// a local swap joins as the SWAP gate of its two physical qubits (the map
// changes for the ops after it).  This is the role of bra's BEGIN/END FUSION
// (bra/src/state.cpp:2193-2217, nompi_state.cpp:1282-1357) and of ket's
// cache-aware gate functions (gate_bitmasks.hpp:587-2134): a run of gates
// applied per group of amplitudes held near the core, with the per-gate
// arithmetic unchanged.
//
// Two groupings:
//  * steps, which the plan reports: the union of a block's qubits, together
//    with the qubits that address one 128-byte line, fits in the local bits of
//    a chunk; the local set is filled up with the lowest remaining qubits;
//  * launches, which run: only the bits that a gate flips need to be local --
//    control bits and the parity bits of diagonal gates (RZ, CZ, ...) outside
//    the chunk are the same for all its amplitudes -- and moves may run out of
//    order (launch_builder), so a launch takes the gates of two to four steps
//    (20 qubits with 10 layers of RZ and CNOT: 9 for 41).
// A group of one op, or of ops that act on a small part of the state, runs on the plain kernels.
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstring>
#include <iterator>
#include <new>
#include <utility>
#include <vector>

#include "brk_block.hpp"
#include "braket_hip.h"
#include "circuit.hpp"

namespace brk {
int fail(int status, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
}

struct brk_block_plan {
  struct step {
    unsigned first_op = 0, num_ops = 0;  // ops of the circuit covered by this step
    uint64_t local = 0;                  // the block's local qubits, 0: plain op
  };
  struct launch {
    bool plain = false;
    brk_circuit::op physical;  // the op at physical qubits (plain)
    brk::block_args args;      // the block's program
  };
  unsigned num_qubits = 0;
  int dtype = BRK_C128;
  std::vector<step> steps;
  std::vector<launch> launches;
  std::vector<unsigned> final_permutation;
};

namespace brk {

static unsigned popcount64(uint64_t x) { return (unsigned)__builtin_popcountll(x); }

// The shape of a dtype's chunks on n qubits.
struct chunk_shape {
  unsigned n, max_local;
  uint64_t line;  // the qubits addressing one 128-byte line (block_run_bytes)
  chunk_shape(unsigned n, int dtype) : n(n), max_local(block_max_local(dtype)) {
    line = (1ull << std::min(block_run_qubits(dtype), n)) - 1ull;
  }
  unsigned num_local() const { return std::min(max_local, n); }
  // a chunk is 2^L amplitudes with L >= 9 (one per thread of a workgroup at least)
  bool enabled() const { return num_local() >= (unsigned)BLOCK_THREAD_BITS; }
  bool fits(uint64_t qubits) const { return popcount64(qubits | line) <= max_local; }
};

// `qubits` filled up with the lowest others to num_local in all.
static uint64_t fill_local(uint64_t qubits, unsigned n, unsigned num_local) {
  for (unsigned q = 0; q < n && popcount64(qubits) < num_local; ++q) qubits |= 1ull << q;
  return qubits;
}

// The bits a gate flips: these have to be local.
static uint64_t mixing_bits(const gate_desc& d) { return d.mode == BLOCK_DIAG ? 0 : d.flip; }

// Groups the program's gates into passes, reordering them only where that is exact.  A segment
// takes gates whose flipped bits (at most two per gate) lie in its L - 9 group bits, diagonal
// gates, and the moves (X, CNOT, SWAP) among them, which it applies last: a gate after a move joins
// the segment if it mixes none of the move's qubits and none of its bits is one the move flips --
// a move only renames the indices such a gate acts on, so the order of the two changes no bit of
// the result.  Matrix gates flipping more bits get a pass of their own.
static void make_passes(block_program& prog, unsigned line_bits) {
  const unsigned L = prog.h.num_local;
  const unsigned gb = L > (unsigned)BLOCK_THREAD_BITS ? L - BLOCK_THREAD_BITS : 0;
  const uint32_t line = (1u << std::min(line_bits, L)) - 1u;
  prog.h.num_passes = 0;
  block_op order[BLOCK_MAX_OPS];
  uint32_t placed = 0;
  uint32_t bits = 0, moved = 0, moved_by = 0;  // group bits; bits the moves flip and test
  std::vector<uint32_t> gates, moves;
  auto pass = [&](block_pass_kind kind) -> block_pass& {
    block_pass& p = prog.passes[prog.h.num_passes++];
    p = block_pass{};
    p.kind = (uint8_t)kind;
    return p;
  };
  auto close = [&]() {
    if (gates.empty() && moves.empty()) return;
    block_pass& p = pass(BLOCK_PASS_SEGMENT);
    p.num_ops = (uint8_t)gates.size();
    p.num_moves = (uint8_t)moves.size();
    for (unsigned b = L; b-- > 0 && (unsigned)__builtin_popcount(bits) < gb;) bits |= 1u << b;
    unsigned k = 0;
    for (unsigned b = 0; b < L; ++b)
      if (bits >> b & 1u) {
        p.qubits[k] = prog.h.pos[b];
        p.group[k++] = (uint8_t)b;
      }
    // straight from or to the state where every access covers whole lines.  A segment that loads
    // and moves stores by way of LDS: another thread may not have loaded the target yet.
    if (prog.h.num_passes == 1 && !(bits & line)) p.flags |= BLOCK_PASS_LOADS;
    if (!(bits & line) && (moves.empty() || (!((moved | moved_by) & line) && !(p.flags & BLOCK_PASS_LOADS))))
      p.flags |= BLOCK_PASS_STORES;
    for (uint32_t i : gates) {  // the masks over the group index and over the thread's bits
      block_op o = prog.ops[i];
      const bool diagonal = o.kind == BLOCK_KIND_DIAG || o.kind == BLOCK_KIND_NEGATE;
      o.thread_cond = (uint16_t)(o.cond & ~bits);
      o.thread_zmask = (uint16_t)(o.zmask & ~bits);
      for (unsigned g = 0; g < k; ++g) {
        const uint32_t bit = 1u << p.group[g];
        if (!diagonal && (o.flip & bit)) o.group_flip |= (uint8_t)(1u << g);
        if ((diagonal ? o.zmask : o.sign) & bit) o.group_zmask |= (uint8_t)(1u << g);
        if (o.cond & bit) o.group_cond |= (uint8_t)(1u << g);
      }
      order[placed++] = o;
    }
    bool linear = true;
    for (uint32_t i : moves) {
      const block_op& o = prog.ops[i];
      const uint32_t tested = o.cond & (uint32_t)~o.flip;  // (a SWAP's own condition lies in its flip)
      linear &= (o.cond & o.flip) ? tested == 0 : (unsigned)__builtin_popcount(tested) <= 1;
      order[placed++] = o;
    }
    if (linear) p.flags |= BLOCK_PASS_LINEAR;
    gates.clear();
    moves.clear();
    bits = moved = moved_by = 0;
  };
  for (uint32_t i = 0; i < prog.h.num_ops; ++i) {
    const block_op& o = prog.ops[i];
    if (o.kind == BLOCK_KIND_SWAP) {
      moves.push_back(i);
      moved |= o.flip;
      moved_by |= o.cond & (uint32_t)~o.flip;
      continue;
    }
    const bool diagonal = o.kind == BLOCK_KIND_DIAG || o.kind == BLOCK_KIND_NEGATE;
    const uint32_t mixing = diagonal ? 0u : o.flip;
    const unsigned flips = (unsigned)__builtin_popcount(mixing);
    if (flips > 2 || flips > gb || (o.kind == BLOCK_KIND_MATRIX && o.sign)) {
      close();
      pass(BLOCK_PASS_SINGLE).num_ops = 1;
      order[placed++] = o;
      continue;
    }
    const bool before_moves = !(mixing & (moved | moved_by)) && !((o.cond | o.zmask) & moved);
    if (!before_moves || (unsigned)__builtin_popcount(bits | mixing) > gb) close();
    bits |= mixing;
    gates.push_back(i);
  }
  close();
  // only the last pass stores
  for (uint32_t k = 0; k + 1 < prog.h.num_passes; ++k) prog.passes[k].flags &= (uint8_t)~BLOCK_PASS_STORES;
  std::copy(order, order + placed, prog.ops);
}

static uint8_t kind_of(const gate_desc& d) {
  switch (d.mode) {
    case BLOCK_H: return BLOCK_KIND_H;
    case BLOCK_SWAP: return BLOCK_KIND_SWAP;
    case BLOCK_ESWAP: return BLOCK_KIND_ESWAP;
    case BLOCK_DIAG: return block_op_coefs(d) == 0 ? BLOCK_KIND_NEGATE : BLOCK_KIND_DIAG;
    default: break;
  }
  const double* u = d.u;
  if (u[1] == 0.0 && u[3] == 0.0 && u[5] == 0.0 && u[7] == 0.0) return BLOCK_KIND_REAL;
  if (u[1] == 0.0 && u[2] == 0.0 && u[4] == 0.0 && u[7] == 0.0) return BLOCK_KIND_X;
  return BLOCK_KIND_MATRIX;
}

static void make_block_program(const gate_desc* descs, unsigned count, unsigned n, uint64_t local, unsigned num_local,
                        unsigned line_bits, block_program* out) {
  block_program& prog = *out;
  prog.h = block_header{};
  prog.h.ops_at = (uint16_t)offsetof(block_program, ops);
  prog.h.coefs_at = (uint16_t)offsetof(block_program, coefs);
  const unsigned L = std::min(num_local, n);
  local = fill_local(local | ((1ull << std::min(line_bits, n)) - 1ull), n, L);
  unsigned r = 0, rank[64] = {};
  for (uint64_t m = local; m; m &= m - 1) {
    const unsigned q = (unsigned)__builtin_ctzll(m);
    rank[q] = r;
    prog.h.pos[r++] = (uint8_t)q;
  }
  prog.h.num_local = r;
  auto to_local = [&](uint64_t m) {
    uint32_t bits = 0;
    for (m &= local; m; m &= m - 1) bits |= 1u << rank[__builtin_ctzll(m)];
    return (uint16_t)bits;
  };
  prog.h.num_ops = count;
  unsigned coef = 0;
  for (unsigned i = 0; i < count; ++i) {
    const gate_desc& d = descs[i];
    block_op& o = prog.ops[i];
    o = block_op{};
    const bool diagonal = d.mode == BLOCK_DIAG;
    o.pair_bit = diagonal ? 0 : (uint8_t)rank[d.pair_bit];
    o.flip = to_local(d.flip);
    o.cond = to_local(d.cond);
    o.sign = to_local(d.sign);
    // the pair's first index has the pair bit clear: that bit of the sign mask never counts
    if (d.mode == BLOCK_MATRIX) o.sign &= (uint16_t)~(1u << o.pair_bit);
    o.zmask = to_local(d.zmask);
    o.outer_cond = d.cond & ~local;
    o.outer_zmask = d.zmask & ~local;
    o.kind = kind_of(d);
    o.inserted = (uint16_t)(o.cond | (diagonal ? 0u : 1u << o.pair_bit));
    o.coef = (uint16_t)coef;
    std::copy(d.u, d.u + block_op_coefs(d), prog.coefs + coef);
    coef += (unsigned)block_op_coefs(d);
  }
}

void make_adjoint_base(const gate_desc* descs, unsigned count, unsigned n, unsigned num_local, unsigned line_bits,
                       adjoint_base* out) {
  adjoint_base& prog = *out;
  prog = adjoint_base{};
  uint64_t local = (1ull << std::min(line_bits, n)) - 1ull;
  for (unsigned i = 0; i < count; ++i) local |= descs[i].qubits;
  local = fill_local(local, n, std::min(num_local, n));
  unsigned r = 0, rank[64] = {};
  for (unsigned q = 0; q < n; ++q)
    if (local >> q & 1u) {
      rank[q] = r;
      prog.pos[r++] = q;
    }
  prog.num_local = r;
  auto to_local = [&](uint64_t m) {
    uint32_t out = 0;
    for (unsigned q = 0; q < n; ++q)
      if (m >> q & 1u) out |= 1u << rank[q];
    return out;
  };
  // local index j = t + BLOCK_THREADS * k: the physical offset of the k part
  const uint32_t size = 1u << r, per = size > (uint32_t)BLOCK_THREADS ? size / BLOCK_THREADS : 1;
  for (uint32_t k = 0; k < per; ++k) {
    const uint32_t j = k << BLOCK_THREAD_BITS;
    uint64_t dep = 0;
    for (unsigned bit = 0; bit < r; ++bit)
      if (j >> bit & 1u) dep |= 1ull << prog.pos[bit];
    prog.deposit_high[k] = dep;
  }
  prog.num_ops = count;
  for (unsigned i = 0; i < count; ++i) {
    const gate_desc& d = descs[i];
    adjoint_op& o = prog.ops[i];
    o.mode = d.mode;
    o.pair_bit = d.mode == BLOCK_DIAG ? 0 : rank[d.pair_bit];
    o.flip = to_local(d.flip);
    o.cond = to_local(d.cond);
    o.sign = to_local(d.sign);
    // the pair's first index has the pair bit clear: that bit of the sign mask never counts
    if (d.mode == BLOCK_MATRIX) o.sign &= ~(1u << o.pair_bit);
    o.negate = d.mode == BLOCK_DIAG && d.u[0] == -1.0 && d.u[1] == 0.0 && d.u[2] == -1.0 && d.u[3] == 0.0;
    o.zmask = to_local(d.zmask);
    const uint32_t inserted = o.cond | (d.mode == BLOCK_DIAG ? 0u : 1u << o.pair_bit);
    o.nins = 0;
    for (unsigned bit = 0; bit < r; ++bit)
      if (inserted >> bit & 1u) o.ins[o.nins++] = bit;
    std::copy(d.u, d.u + 8, o.u);
  }
}

// The program as launch arguments (its ops fit: BLOCK_ARG_ROOM).
static void pack(const block_program& prog, block_args* out) {
  unsigned coefs = 0;
  for (unsigned i = 0; i < prog.h.num_ops; ++i) {
    const block_op& o = prog.ops[i];
    const unsigned k = o.kind == BLOCK_KIND_DIAG || o.kind == BLOCK_KIND_ESWAP ? 4
                       : o.kind == BLOCK_KIND_H || o.kind == BLOCK_KIND_SWAP || o.kind == BLOCK_KIND_NEGATE ? 0 : 8;
    coefs = std::max(coefs, o.coef + k);
  }
  out->h = prog.h;
  char* at = reinterpret_cast<char*>(out) + sizeof(block_header);
  auto put = [&](const void* from, size_t bytes) {
    std::memcpy(at, from, bytes);
    at += bytes;
  };
  put(prog.passes, sizeof(block_pass) * prog.h.num_passes);
  out->h.ops_at = (uint16_t)(at - reinterpret_cast<char*>(out));
  put(prog.ops, sizeof(block_op) * prog.h.num_ops);
  out->h.coefs_at = (uint16_t)(at - reinterpret_cast<char*>(out));
  put(prog.coefs, sizeof(double) * coefs);
}

op_dependences dependences_of(const std::vector<brk_circuit::op>& ops) {
  const size_t count = ops.size();
  op_dependences d;
  d.mask.assign(count, 0);
  d.succ.assign(count, {});
  d.indeg.assign(count, 0);
  std::vector<long> last(64, -1);
  std::vector<long> prev;
  for (size_t i = 0; i < count; ++i) {
    const auto& o = ops[i];
    for (unsigned q : o.targets) d.mask[i] |= 1ull << q;
    for (unsigned q : o.controls) d.mask[i] |= 1ull << q;
    if (o.code == BRK_OP_LOCAL_SWAP) d.mask[i] = ~0ull;  // a barrier: it moves qubits between slots
    prev.clear();
    for (unsigned q = 0; q < 64; ++q)
      if (d.mask[i] >> q & 1ull) prev.push_back(last[q]);
    std::sort(prev.begin(), prev.end());
    prev.erase(std::unique(prev.begin(), prev.end()), prev.end());
    for (long f : prev)
      if (f >= 0) {
        d.succ[(size_t)f].push_back(i);
        ++d.indeg[i];
      }
    for (unsigned q = 0; q < 64; ++q)
      if (d.mask[i] >> q & 1ull) last[q] = (long)i;
  }
  return d;
}

std::vector<size_t> block_order(const std::vector<brk_circuit::op>& ops, unsigned num_local, unsigned line_bits) {
  const size_t count = ops.size();
  op_dependences dep = dependences_of(ops);
  const std::vector<uint64_t>& mask = dep.mask;
  const std::vector<std::vector<size_t>>& succ = dep.succ;
  std::vector<unsigned>& indeg = dep.indeg;
  std::vector<size_t> ready, order;
  order.reserve(count);
  for (size_t i = 0; i < count; ++i)
    if (!indeg[i]) ready.push_back(i);
  const uint64_t line = line_bits >= 64 ? ~0ull : (1ull << line_bits) - 1ull;
  auto take = [&](size_t k) {  // schedule ready[k]
    const size_t i = ready[k];
    ready.erase(ready.begin() + (long)k);
    order.push_back(i);
    for (size_t j : succ[i])
      if (--indeg[j] == 0) ready.insert(std::lower_bound(ready.begin(), ready.end(), j), j);
  };
  // Lookahead: how many ops (at most `budget`) could run within the local qubits `loc` once
  // `first` runs, without adding qubits.
  std::vector<unsigned> tmp_deg(count, 0), stamp(count, 0);
  unsigned cur_stamp = 0;
  std::vector<size_t> pend;
  auto closure = [&](size_t first, uint64_t loc, unsigned budget) {
    ++cur_stamp;
    pend.assign(1, first);
    for (size_t r : ready)
      if (r != first && !(mask[r] & ~loc)) pend.push_back(r);
    unsigned got = 0;
    while (!pend.empty() && got < budget) {
      const size_t i = pend.back();
      pend.pop_back();
      ++got;
      for (size_t j : succ[i]) {
        if (stamp[j] != cur_stamp) {
          stamp[j] = cur_stamp;
          tmp_deg[j] = indeg[j];
        }
        if (--tmp_deg[j] == 0 && !(mask[j] & ~loc)) pend.push_back(j);
      }
    }
    return got;
  };
  while (!ready.empty()) {
    uint64_t local = line;
    unsigned taken = 0;
    while (taken < (unsigned)BLOCK_MAX_OPS && !ready.empty()) {
      // an op within the block's qubits first (the earliest); else the op whose qubits
      // let the most ops run per added qubit
      size_t best = ready.size();
      for (size_t k = 0; k < ready.size() && best == ready.size(); ++k)
        if (!(mask[ready[k]] & ~local)) best = k;
      if (best == ready.size()) {
        double best_score = -1.0;
        unsigned best_growth = 65;
        for (size_t k = 0; k < ready.size(); ++k) {
          const uint64_t m = mask[ready[k]];
          if (popcount64(local | m) > num_local) continue;
          const unsigned growth = popcount64(m & ~local);
          const double score = (double)closure(ready[k], local | m, (unsigned)BLOCK_MAX_OPS - taken) / growth;
          if (score > best_score || (score == best_score && growth < best_growth)) {
            best = k;
            best_score = score;
            best_growth = growth;
          }
        }
      }
      if (best == ready.size()) break;
      local |= mask[ready[best]];
      take(best);
      ++taken;
    }
    if (!taken) take(0);  // an op no block holds: a step of its own
  }
  return order;
}

// Op o of the circuit at physical qubits (m's lists are used again); advances the map over it.
static void place_op(const brk_circuit::op& o, permutation& perm, brk_circuit::op* m) {
  *m = o;
  if (o.code == BRK_OP_LOCAL_SWAP) {  // given at physical qubits; the map changes for the ops after it
    perm.permutate(perm.inverse[o.targets[0]], perm.inverse[o.targets[1]]);
    return;
  }
  for (auto& q : m->targets) q = perm.perm[q];
  for (auto& q : m->controls) q = perm.perm[q];
}

// The description of an op at physical qubits: the data of a local swap is a SWAP gate on its two qubits
// (swap_permutated_local_qubits.hpp:64-77).
static int describe_op(const brk_circuit::op& m, gate_desc* d) {
  return describe_physical_op(m.code == BRK_OP_LOCAL_SWAP ? (int)BRK_OP_SWAP : m.code, m.targets.data(),
                              (unsigned)m.targets.size(), m.controls.empty() ? nullptr : m.controls.data(),
                              (unsigned)m.controls.size(), m.params.data(), d);
}

// Collects ops into launches and hands each over as soon as it is complete.  A launch takes the ops
// in order, and passes over one that does not fit for later ones where that changes no bit of the
// result: a move (X, CNOT, SWAP) only renames the indices that a gate acts on, so it may pass, or be
// passed by, any gate that mixes none of the qubits they share (two qubits' H, say, may not change
// places: their roundings differ).  Launches for 200 gates, in order and so: 29 qubits 11-13 and 9-11,
// 20 qubits 9 and 7, 18 qubits 7-8 and 5-7; 20 qubits with 10 layers of RZ and CNOT 12 and 9.
// plain(op) / block(args) return a status.
template <typename Plain, typename Block>
struct launch_builder {
  // Ops passed over at most; a launch of the above circuits takes 20 to 40.
  static constexpr size_t LOOKAHEAD = 2 * BLOCK_MAX_OPS;
  struct entry {
    brk_circuit::op op;
    gate_desc desc;
  };
  chunk_shape shape;
  int dtype;
  double state_bytes;
  unsigned line_bits;
  Plain plain;
  Block block;
  // the launch in the making
  gate_desc descs[BLOCK_MAX_OPS];
  unsigned count = 0;
  uint64_t mixing = 0;
  size_t room = 0;
  double plain_bytes = 0.0;  // what the ops' plain kernels move, as state (plain_is_faster)
  std::vector<brk_circuit::op> ops;  // for their plain kernels: all of them while those are faster
  // the ops passed over: what they flip, and all that they touch; whether one of them rounds
  std::vector<entry> rest;
  uint64_t rest_mixing = 0, rest_qubits = 0;
  bool rest_rounds = false;
  std::vector<entry> pending;  // (empty but within add and flush)
  block_program prog;
  block_args args{};

  launch_builder(unsigned n, int dtype, Plain p, Block b)
      : shape(n, dtype), dtype(dtype), state_bytes((dtype == BRK_C128 ? 16.0 : 8.0) * (double)(1ull << n)),
        line_bits(block_run_qubits(dtype)), plain(p), block(b) {}
  int add(brk_circuit::op&& m, const gate_desc& d) {
    if (!shape.enabled() || !shape.fits(mixing_bits(d))) {  // too wide for a chunk
      if (int st = flush()) return st;
      return plain(m);
    }
    return place(std::move(m), d) ? emit() : BRK_OK;
  }
  int flush() {
    while (count)
      if (int st = emit()) return st;
    return BRK_OK;
  }

 private:
  // Whether the launch is complete with this op.
  bool place(brk_circuit::op&& op, const gate_desc& d) {
    const uint64_t m = mixing_bits(d);
    const bool rounds = d.mode != BLOCK_SWAP;
    const bool in_order = !(rest_mixing & d.qubits) && !(m & rest_qubits) && !(rounds && rest_rounds);
    if (in_order && shape.fits(mixing | m) && room + block_op_room(d) <= BLOCK_ARG_ROOM) {
      mixing |= m;
      room += block_op_room(d);
      if (plain_is_faster()) {  // (slower once, it stays so, and the op is not needed any more)
        plain_bytes += std::max(plain_share(d, dtype) * state_bytes + 6e6, 12e6);
        if (!count || plain_is_faster()) ops.push_back(std::move(op));
      }
      descs[count++] = d;
      return count == (unsigned)BLOCK_MAX_OPS;
    }
    rest_mixing |= m;
    rest_qubits |= d.qubits;
    rest_rounds |= rounds;
    rest.push_back({std::move(op), d});
    // (nothing passes a gate that rounds once every qubit is touched)
    return rest.size() == LOOKAHEAD || (rest_rounds && rest_qubits == (1ull << shape.n) - 1ull);
  }
  // A launch moves the whole state whatever its gates act on; their plain kernels move what they act on,
  // but no less than what passes in a kernel's 3 us (12 MB of the state), and 6 MB more each for their
  // start and end.  The line is where both take the same time: complex64 plain kernels move a state 10 %
  // slower than a launch does (2 GiB: 735 and 690 us), complex128 ones 4 % faster (4 GiB: 1360 and 1420).
  // 28 qubits complex128, launch against plain kernels: two Z with 10 controls 1.38 ms and 17 us, two X
  // with 4 controls 1.43 and 0.18 ms, two CNOT 1.42 and 1.36, H and CZ 1.45 and 1.69, four CZ 1.38 and
  // 1.34; 22 qubits: two CZ 22 and 11 us, four 23 and 27; up to 20 qubits a launch is always the faster.
  // Over 946 circuits of 2 to 8 such gates (10 to 28 qubits, both types) the choice is at most 3 % slower
  // than the other one.
  bool plain_is_faster() const {
    return plain_bytes < (dtype == BRK_C128 ? 1.08 : 0.90) * state_bytes;
  }
  int launch() {
    if (count == 1 || plain_is_faster()) {
      for (const brk_circuit::op& op : ops)
        if (int st = plain(op)) return st;
      return BRK_OK;
    }
    make_block_program(descs, count, shape.n, mixing, shape.num_local(), line_bits, &prog);
    make_passes(prog, line_bits);
    pack(prog, &args);
    return block(args);
  }
  // Runs the launch, and puts the ops passed over in the next ones; the last of these stays open.
  int emit() {
    size_t next = 0;
    bool complete = true;
    while (complete) {
      if (int st = launch()) return st;
      rest.insert(rest.end(), std::make_move_iterator(pending.begin() + next),
                  std::make_move_iterator(pending.end()));
      pending.swap(rest);
      rest.clear();
      count = 0;
      ops.clear();
      mixing = rest_mixing = rest_qubits = 0;
      room = 0;
      plain_bytes = 0.0;
      rest_rounds = false;
      complete = false;
      for (next = 0; next < pending.size() && !complete; ++next)
        complete = place(std::move(pending[next].op), pending[next].desc);
    }
    pending.clear();
    return BRK_OK;
  }
};

static int check_permutation(permutation& perm, const unsigned* given, unsigned n) {
  if (given && !perm.load(given, n))
    return fail(BRK_ERR_INVALID_ARGUMENT, "permutation is not a permutation of 0..%u", n - 1);
  return BRK_OK;
}

static int build_plan(const brk_circuit* circuit, int dtype, const unsigned* permutation_in, brk_block_plan* plan) {
  const unsigned n = circuit->num_qubits;
  plan->num_qubits = n;
  plan->dtype = dtype;
  permutation perm(n);
  if (int st = check_permutation(perm, permutation_in, n)) return st;
  const chunk_shape shape(n, dtype);
  // the step in the making
  brk_block_plan::step s;
  uint64_t qubits = 0;
  auto close_step = [&]() {
    if (!s.num_ops) return;
    if (s.num_ops > 1) s.local = fill_local(qubits | shape.line, n, shape.num_local());
    plan->steps.push_back(s);
    s = brk_block_plan::step{};
    qubits = 0;
  };
  auto plain = [&](const brk_circuit::op& m) {
    plan->launches.emplace_back();
    plan->launches.back().plain = true;
    plan->launches.back().physical = m;
    return BRK_OK;
  };
  auto block = [&](const block_args& a) {
    plan->launches.emplace_back();
    plan->launches.back().args = a;
    return BRK_OK;
  };
  launch_builder<decltype(plain), decltype(block)> b(n, dtype, plain, block);
  brk_circuit::op m;
  for (unsigned i = 0; i < circuit->ops.size(); ++i) {
    gate_desc d;
    place_op(circuit->ops[i], perm, &m);
    if (int st = describe_op(m, &d)) return st;
    if (!shape.enabled() || s.num_ops == (unsigned)BLOCK_MAX_OPS || !shape.fits(qubits | d.qubits)) close_step();
    if (!s.num_ops) s.first_op = i;
    ++s.num_ops;
    qubits |= d.qubits;
    if (int st = b.add(std::move(m), d)) return st;
  }
  close_step();
  if (int st = b.flush()) return st;
  plan->final_permutation = perm.perm;
  return BRK_OK;
}

static int run_plan(const brk_block_plan* plan, void* first, void* stream) {
  const uint64_t size = 1ull << plan->num_qubits;
  for (const auto& l : plan->launches)
    if (int st = l.plain ? apply_physical_op(l.physical, first, size, plan->dtype, stream)
                         : launch_block(l.args, first, size, plan->dtype, stream))
      return st;
  return BRK_OK;
}

int run_in_blocks(const brk_circuit* circuit, void* first, int dtype, permutation& perm, void* stream) {
  const uint64_t size = 1ull << circuit->num_qubits;
  auto plain = [&](const brk_circuit::op& m) { return apply_physical_op(m, first, size, dtype, stream); };
  auto block = [&](const block_args& a) { return launch_block(a, first, size, dtype, stream); };
  brk_circuit::op m;
  if (circuit->ops.size() <= 1 || !chunk_shape(circuit->num_qubits, dtype).enabled()) {  // nothing to collect
    for (const auto& o : circuit->ops) {
      place_op(o, perm, &m);
      if (int st = plain(m)) return st;
    }
    return BRK_OK;
  }
  launch_builder<decltype(plain), decltype(block)> b(circuit->num_qubits, dtype, plain, block);
  for (const auto& o : circuit->ops) {
    gate_desc d;
    place_op(o, perm, &m);
    if (int st = describe_op(m, &d)) return st;
    if (int st = b.add(std::move(m), d)) return st;  // (takes the op only where it keeps it)
  }
  return b.flush();
}

}  // namespace brk

using namespace brk;

extern "C" {

int brk_block_plan_create(const brk_circuit* circuit, int dtype, const unsigned* permutation, brk_block_plan** out) {
  if (!circuit || !out) return fail(BRK_ERR_INVALID_ARGUMENT, "null argument");
  if (dtype != BRK_C128 && dtype != BRK_C64) return fail(BRK_ERR_UNSUPPORTED_DTYPE, "dtype %d", dtype);
  *out = nullptr;
  auto* plan = new (std::nothrow) brk_block_plan;
  if (!plan) return fail(BRK_ERR_OUT_OF_MEMORY, "cannot allocate the plan");
  if (int st = build_plan(circuit, dtype, permutation, plan)) {
    delete plan;
    return st;
  }
  *out = plan;
  return BRK_OK;
}

int brk_block_plan_destroy(brk_block_plan* plan) {
  delete plan;
  return BRK_OK;
}

int brk_block_plan_num_steps(const brk_block_plan* plan, unsigned* num_steps) {
  if (!plan || !num_steps) return fail(BRK_ERR_INVALID_ARGUMENT, "null argument");
  *num_steps = (unsigned)plan->steps.size();
  return BRK_OK;
}

int brk_block_plan_step(const brk_block_plan* plan, unsigned i, unsigned* first_op, unsigned* num_ops,
                        unsigned* num_local, unsigned* local_qubits) {
  if (!plan) return fail(BRK_ERR_INVALID_ARGUMENT, "plan is null");
  if (i >= plan->steps.size()) return fail(BRK_ERR_INVALID_ARGUMENT, "step %u out of range", i);
  const auto& s = plan->steps[i];
  if (first_op) *first_op = s.first_op;
  if (num_ops) *num_ops = s.num_ops;
  if (num_local) *num_local = popcount64(s.local);
  if (local_qubits)
    for (uint64_t m = s.local; m; m &= m - 1) *local_qubits++ = (unsigned)__builtin_ctzll(m);
  return BRK_OK;
}

int brk_block_plan_final_permutation(const brk_block_plan* plan, unsigned* permutation) {
  if (!plan || !permutation) return fail(BRK_ERR_INVALID_ARGUMENT, "null argument");
  std::copy(plan->final_permutation.begin(), plan->final_permutation.end(), permutation);
  return BRK_OK;
}

int brk_block_plan_run(brk_block_plan* plan, void* first, void* stream) {
  if (!plan) return fail(BRK_ERR_INVALID_ARGUMENT, "plan is null");
  return run_plan(plan, first, stream);
}

int brk_circuit_block_order(const brk_circuit* circuit, unsigned num_local, unsigned line_bits, unsigned* order) {
  if (!circuit || (!order && !circuit->ops.empty())) return fail(BRK_ERR_INVALID_ARGUMENT, "null argument");
  if (num_local < 1 || num_local > 64 || line_bits > num_local)
    return fail(BRK_ERR_INVALID_ARGUMENT, "need 1 <= num_local <= 64 and line_bits <= num_local");
  const std::vector<size_t> o = block_order(circuit->ops, num_local, line_bits);
  for (size_t k = 0; k < o.size(); ++k) order[k] = (unsigned)o[k];
  return BRK_OK;
}

int brk_circuit_run_blocked(const brk_circuit* circuit, void* first, int dtype, unsigned* permutation,
                            void* stream) {
  if (!circuit) return fail(BRK_ERR_INVALID_ARGUMENT, "null argument");
  if (dtype != BRK_C128 && dtype != BRK_C64) return fail(BRK_ERR_UNSUPPORTED_DTYPE, "dtype %d", dtype);
  brk::permutation perm(circuit->num_qubits);
  if (int st = check_permutation(perm, permutation, circuit->num_qubits)) return st;
  int st = run_in_blocks(circuit, first, dtype, perm, stream);
  if (hipStreamSynchronize(reinterpret_cast<hipStream_t>(stream)) != hipSuccess && !st)
    st = fail(BRK_ERR_HIP, "hipStreamSynchronize failed");
  if (!st && permutation) std::copy(perm.perm.begin(), perm.perm.end(), permutation);
  return st;
}

}  // extern "C"
