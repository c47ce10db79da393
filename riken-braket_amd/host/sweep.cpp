// Planner of the adjoint gradient's sweeps: blocks, segments and macros (csrc/brk_sweep.hpp).
//
// A mixing gate depends on the gates before it on its qubit; a diagonal gate (phase or sign) only on
// the mixing gates before it, since diagonal gates commute.  Blocks, and the segments of a block, are
// built greedily: one qubit at a time is added to the set -- the block's local qubits, the segment's
// group -- that lets the most gates run, where gates on one qubit need it in the set and signs run
// anywhere.  On a layered ansatz that walks the light cone: a block takes a triangle or parallelogram
// of layers and qubits, a segment up to three layers of three qubits.
#include "sweep.hpp"

#include <algorithm>
#include <cstring>

namespace brk {

namespace {

// What can run next is kept by kind and place, and a look ahead goes no further than its budget, so that a
// macro or segment takes the same time in a long circuit as in a short one.  (One list of all runnable gates,
// scanned for every macro, and a copy of every gate's dependences for every segment: 66 000 RY and RX on one
// qubit 3.5 s, 80 000 RZ in a row 81 s; now 0.15 and 0.18.)
struct planner {
  const std::vector<sweep_gate>& gates;
  unsigned n;
  struct edge {
    uint32_t to;
    int32_t next;
  };
  std::vector<edge> edges;    // what depends on a gate: lists through the edges
  std::vector<int32_t> succ;  // first edge of each gate, -1: none
  std::vector<uint32_t> indeg;
  std::vector<uint32_t> open;  // the same without the signs that can run: a look ahead takes those as run
  size_t remaining;            // gates not run yet
  // runnable gates, -1: none.  Signs by distance and lower qubit, phases (with a parameter and without) by
  // qubit: the first of a list, link[] its next; a qubit's mixing gate; next[q]: the one that only signs are
  // in the way of
  std::vector<int32_t> link;
  int32_t signs[32][32];
  uint32_t signs_at[32] = {};  // the lower qubits with signs of a distance
  uint32_t distances = 0;      // the distances with signs
  int32_t phases[32], param_phases[32], mixing[32], next[32];
  uint32_t active = 0;  // qubits with one-qubit gates among these (a superset while a macro is made)
  // a look ahead: its own dependences, where its stamp is the present one
  std::vector<uint32_t> stamp, left;
  uint32_t now = 0;
  std::vector<uint32_t> base_stamp, base;
  uint32_t base_now = 0;
  std::vector<uint32_t> stack;
  std::vector<uint32_t> waiting[32];  // per qubit

  // (at most `most` of the gates that depend on i)
  template <typename F>
  void for_successors(uint32_t i, unsigned most, F f) const {
    for (int32_t e = succ[i]; e >= 0 && most--; e = edges[(size_t)e].next) f(edges[(size_t)e].to);
  }
  uint32_t qubits(const sweep_gate& g) const { return g.sign ? g.mask : 1u << g.q; }

  planner(const std::vector<sweep_gate>& g, unsigned num_qubits) : gates(g), n(num_qubits), remaining(g.size()) {
    const uint32_t count = (uint32_t)gates.size();
    succ.assign(count, -1);
    edges.reserve(4 * (size_t)count);
    indeg.assign(count, 0);
    stamp.assign(count, 0);
    left.assign(count, 0);
    base_stamp.assign(count, 0);
    base.assign(count, 0);
    link.assign(count, -1);
    for (int32_t* list : {&signs[0][0], phases, param_phases, mixing, next})
      std::fill(list, list + (list == &signs[0][0] ? 32 * 32 : 32), -1);
    std::vector<long> last_mix(n, -1);
    std::vector<std::vector<uint32_t>> since(n);  // diagonal gates on a qubit since its last mixing gate
    for (uint32_t i = 0; i < count; ++i) {
      const sweep_gate& gate = gates[i];
      auto after = [&](uint32_t j) {
        edges.push_back({i, succ[j]});
        succ[j] = (int32_t)edges.size() - 1;
        ++indeg[i];
      };
      if (gate.sign || gate.diagonal) {
        for (uint32_t m = qubits(gate); m; m &= m - 1) {
          const unsigned q = (unsigned)__builtin_ctz(m);
          if (last_mix[q] >= 0) after((uint32_t)last_mix[q]);
          since[q].push_back(i);
        }
      } else {
        for (uint32_t j : since[gate.q]) after(j);
        if (since[gate.q].empty() && last_mix[gate.q] >= 0) after((uint32_t)last_mix[gate.q]);
        since[gate.q].clear();
        last_mix[gate.q] = (long)i;
      }
    }
    open = indeg;
    for (uint32_t i = 0; i < count; ++i)
      if (!indeg[i]) runnable(i);
  }

  // Files gate i, on which nothing waits any more.
  void runnable(uint32_t i) {
    const sweep_gate& g = gates[i];
    if (g.sign) {
      const unsigned lo = (unsigned)__builtin_ctz(g.mask), d = 31u - (unsigned)__builtin_clz(g.mask) - lo;
      push(signs[d][lo], i);
      signs_at[d] |= 1u << lo;
      distances |= 1u << d;
      for_successors(i, ~0u, [&](uint32_t j) {
        if (--open[j] == 0) only_signs_before(j);  // (only mixing gates wait for a sign)
      });
    } else {
      active |= 1u << g.q;
      if (g.diagonal) push((g.param >= 0 ? param_phases : phases)[g.q], i);
      else mixing[g.q] = next[g.q] = (int32_t)i;
    }
  }
  void push(int32_t& first, uint32_t i) {
    link[i] = first;
    first = (int32_t)i;
  }
  void only_signs_before(uint32_t j) {
    active |= 1u << gates[j].q;
    next[gates[j].q] = (int32_t)j;
  }

  // Runs gate i, which its list no longer holds.
  void take(uint32_t i) {
    --remaining;
    const bool sign = gates[i].sign;  // (open counts it as run)
    for_successors(i, ~0u, [&](uint32_t j) {
      if (!sign) --open[j];
      if (--indeg[j] == 0) runnable(j);
      else if (!sign && open[j] == 0 && !gates[j].sign && !gates[j].diagonal) only_signs_before(j);
    });
  }

  bool runs_in(uint32_t i, uint32_t set) const { return gates[i].sign || (set >> gates[i].q & 1u); }

  // Puts the one-qubit gates of qubit q that can run (at most `budget` of a kind) into a list.
  void list_of(unsigned q, unsigned budget, std::vector<uint32_t>& list) const {
    for (int32_t i : {phases[q], param_phases[q]})
      for (unsigned k = budget; i >= 0 && k--; i = link[(size_t)i]) list.push_back((uint32_t)i);
    if (next[q] >= 0) list.push_back((uint32_t)next[q]);
  }

  void update_active(unsigned q) {
    if (next[q] < 0 && phases[q] < 0 && param_phases[q] < 0) active &= ~(1u << q);
  }

  // How many one-qubit gates (at most `budget`) could run within the set.
  unsigned closure(uint32_t set, unsigned budget) {
    stack.clear();
    for (uint32_t m = set & active; m; m &= m - 1) list_of((unsigned)__builtin_ctz(m), budget, stack);
    return follow(set, budget, [&](uint32_t j) { return open[j]; });
  }

  // `set` with up to `room` of the candidates added, each the one that lets the most gates (at most
  // `budget`) run.  What runs within the set is simulated once; a candidate then only follows what it
  // adds, from the gates that wait for it.
  uint32_t grow(uint32_t set, uint32_t candidates, unsigned room, unsigned budget) {
    ++base_now;
    stack.clear();
    for (unsigned q = 0; q < n; ++q) waiting[q].clear();
    for (uint32_t m = active; m; m &= m - 1) {
      const unsigned q = (unsigned)__builtin_ctz(m);
      list_of(q, budget, set >> q & 1u ? stack : waiting[q]);
    }
    run(set, budget);
    while (room--) {
      unsigned best = 0;
      unsigned qubit = 0;
      for (uint32_t m = candidates & ~set; m; m &= m - 1) {
        const unsigned q = (unsigned)__builtin_ctz(m);
        if (waiting[q].empty()) continue;
        stack = waiting[q];
        const unsigned c = follow(set | 1u << q, budget, [&](uint32_t j) { return base_of(j); });
        if (c > best) {
          best = c;
          qubit = q;
        }
      }
      if (!best) break;
      set |= 1u << qubit;
      stack.swap(waiting[qubit]);
      waiting[qubit].clear();
      run(set, budget);
    }
    return set;
  }

  uint32_t& base_of(uint32_t j) {
    if (base_stamp[j] != base_now) {
      base_stamp[j] = base_now;
      base[j] = open[j];
    }
    return base[j];
  }

  // Runs the gates on the stack and what they make runnable within the set, on `base`, until `budget`
  // one-qubit gates ran; gates on other qubits wait.
  void run(uint32_t set, unsigned budget) {
    unsigned got = 0;
    while (!stack.empty() && got < budget) {
      const uint32_t i = stack.back();
      stack.pop_back();
      if (!runs_in(i, set)) {
        waiting[gates[i].q].push_back(i);
        continue;
      }
      got += gates[i].sign ? 0 : 1;
      for_successors(i, budget, [&](uint32_t j) {
        if (--base_of(j) == 0) stack.push_back(j);
      });
    }
  }
  // How many one-qubit gates (at most `budget`) run from those on the stack within the set, with the
  // dependences that `start` gives.
  template <typename F>
  unsigned follow(uint32_t set, unsigned budget, F start) {
    ++now;
    unsigned got = 0;
    while (!stack.empty() && got < budget) {
      const uint32_t i = stack.back();
      stack.pop_back();
      if (!runs_in(i, set)) continue;
      got += gates[i].sign ? 0 : 1;
      for_successors(i, budget, [&](uint32_t j) {
        if (stamp[j] != now) {
          stamp[j] = now;
          left[j] = start(j);
        }
        if (--left[j] == 0) stack.push_back(j);
      });
    }
    stack.clear();
    return got;
  }
};

using cd = std::complex<double>;

// One macro: what can run of the gates on the group's qubits q[], or of any signs.
sweep_macro make_macro(planner& p, const unsigned (&q)[SWEEP_GROUP], bool any_signs) {
  sweep_macro mac{};
  for (int32_t& s : mac.slot) s = -1;
  uint32_t group = 0;
  for (unsigned qubit : q) group |= 1u << qubit;
  // signs: those on the group's qubits, then any others whose distance has a term (they cost nothing)
  auto take_signs = [&](uint32_t t, uint32_t lower) {
    const uint32_t d = mac.d[t];
    if (!(p.signs_at[d] &= ~lower)) p.distances &= ~(1u << d);
    for (; lower; lower &= lower - 1) {
      const unsigned lo = (unsigned)__builtin_ctz(lower);
      for (int32_t& i = p.signs[d][lo]; i >= 0; i = p.link[(size_t)i]) {
        mac.A[t] ^= 1u << lo;
        p.take((uint32_t)i);
      }
    }
  };
  for (uint32_t m = p.distances; m && mac.num_terms < (uint32_t)SWEEP_MAX_TERMS; m &= m - 1) {
    const uint32_t d = (uint32_t)__builtin_ctz(m);
    if (const uint32_t lower = any_signs ? p.signs_at[d] : p.signs_at[d] & (group | group >> d)) {
      mac.d[mac.num_terms] = d;
      take_signs(mac.num_terms++, lower);
    }
  }
  for (uint32_t t = 0; t < mac.num_terms; ++t) take_signs(t, p.signs_at[mac.d[t]]);
  // phases of the group's qubits: one product per qubit, one with a parameter among them
  cd phase[SWEEP_GROUP][2];
  for (unsigned b = 0; b < (unsigned)SWEEP_GROUP; ++b) {
    phase[b][0] = phase[b][1] = 1.0;
    auto apply = [&](uint32_t i) {
      const sweep_gate& g = p.gates[i];
      phase[b][0] *= cd(g.u[0], g.u[1]);
      phase[b][1] *= cd(g.u[6], g.u[7]);
      mac.phases = 1;
      p.take(i);
    };
    for (int32_t& i = p.phases[q[b]]; i >= 0; i = p.link[(size_t)i]) apply((uint32_t)i);
    int32_t& with_param = p.param_phases[q[b]];
    if (with_param < 0) continue;
    const uint32_t i = (uint32_t)with_param;
    with_param = p.link[i];
    const sweep_gate& g = p.gates[i];
    mac.slot[b] = g.param;
    mac.weight[b][0] = g.d[1];
    mac.weight[b][1] = g.d[7];
    mac.phase_grads |= 1u << b;
    apply(i);
  }
  // mixing gates, one per qubit
  for (unsigned b = 0; b < (unsigned)SWEEP_GROUP; ++b) {
    const int32_t i = p.mixing[q[b]];
    if (i < 0) continue;
    p.mixing[q[b]] = p.next[q[b]] = -1;
    const sweep_gate& g = p.gates[(size_t)i];
    const double* u = g.u;
    std::copy(u, u + 8, mac.matrix[b]);
    mac.mix[b] = u[1] == 0.0 && u[3] == 0.0 && u[5] == 0.0 && u[7] == 0.0   ? SWEEP_MIX_REAL
                 : u[1] == 0.0 && u[2] == 0.0 && u[4] == 0.0 && u[7] == 0.0 ? SWEEP_MIX_X
                                                                            : SWEEP_MIX_GENERAL;
    if (g.param >= 0) {
      mac.slot[SWEEP_GROUP + b] = g.param;
      const bool y_form = g.d[3] == 0.0 && g.d[5] == 0.0;  // D = [[0, a], [b, 0]], else [[0, i a], [i b, 0]]
      mac.form[b] = y_form ? SWEEP_FORM_Y : SWEEP_FORM_X;
      mac.mix_weight[b][0] = y_form ? g.d[2] : g.d[3];
      mac.mix_weight[b][1] = y_form ? g.d[4] : g.d[5];
    }
    p.take((uint32_t)i);
  }
  for (unsigned qubit : q) p.update_active(qubit);
  for (int32_t s : mac.slot) mac.any_grads |= s >= 0 ? 1u : 0u;
  // the terms' parity over the group's own bits: into the table where there is one
  for (uint32_t m = 0; m < (1u << SWEEP_GROUP); ++m) {
    uint32_t xe = 0;
    cd f = 1.0;
    for (unsigned b = 0; b < (unsigned)SWEEP_GROUP; ++b) {
      xe |= ((m >> b) & 1u) << q[b];
      f *= phase[b][(m >> b) & 1u];
    }
    uint32_t odd = 0;
    for (uint32_t t = 0; t < mac.num_terms; ++t) odd += (uint32_t)__builtin_popcount(xe & (xe >> mac.d[t]) & mac.A[t]);
    if (odd & 1u) {
      if (mac.phases) f = -f;
      else mac.uniform |= 1u << m;
    }
    mac.phase[m][0] = f.real();
    mac.phase[m][1] = f.imag();
  }
  return mac;
}

}  // namespace

int plan_sweep(const std::vector<sweep_gate>& gates, unsigned n, unsigned num_local, unsigned line_bits,
               const std::function<int(const void* program, size_t bytes)>& emit) {
  planner p(gates, n);
  const uint32_t all = n >= 32 ? ~0u : (1u << n) - 1u;
  const uint32_t line = (1u << line_bits) - 1u;
  // A segment goes on to another macro where it runs this many gates: a macro takes the time of about
  // two exchanges through LDS whatever it runs (24 qubits, 12 layers: 151 reverse macros in 58
  // segments; 178 in 56 with macros of any size).
  constexpr unsigned CHAIN_GATES = 4;
  constexpr unsigned BLOCK_GATES = 2 * SWEEP_GROUP * SWEEP_BLOCK_MACROS;  // a full block's macros run no more
  std::vector<sweep_segment> segments;
  std::vector<sweep_macro> macros;
  std::vector<char> program;
  while (p.remaining) {
    // local qubits: the line's, the greedy ones, then the lowest others
    uint32_t local = p.grow(line, all, num_local - line_bits, BLOCK_GATES);
    for (unsigned q = 0; (unsigned)__builtin_popcount(local) < num_local; ++q) local |= 1u << q;
    sweep_header h{};
    unsigned rank[32] = {}, r = 0;
    for (uint32_t m = local; m; m &= m - 1) {
      const unsigned q = (unsigned)__builtin_ctz(m);
      rank[q] = r;
      h.pos[r++] = (uint8_t)q;
    }
    segments.clear();
    macros.clear();
    while (p.remaining && macros.size() + SWEEP_MAX_MACROS <= SWEEP_BLOCK_MACROS) {
      uint32_t group = p.grow(0, local, SWEEP_GROUP, 4 * SWEEP_GROUP * SWEEP_MAX_MACROS);
      // without a gate for these qubits the block ends (signs wait for a block that needs them), or
      // only signs are left
      const bool only_signs = group == 0;
      if (only_signs && p.active != 0) break;
      // filled up with the highest local qubits: lanes then cover whole lines
      for (unsigned q = n; q-- > 0 && (unsigned)__builtin_popcount(group) < (unsigned)SWEEP_GROUP;)
        if (local >> q & 1u) group |= 1u << q;
      sweep_segment s{};
      unsigned q[SWEEP_GROUP], k = 0;
      uint32_t bits = 0;
      for (uint32_t m = group; m; m &= m - 1) {
        q[k] = (unsigned)__builtin_ctz(m);
        s.group[k] = (uint8_t)rank[q[k]];
        s.qubits[k] = (uint8_t)q[k];
        bits |= 1u << rank[q[k]];
        ++k;
      }
      do {
        macros.push_back(make_macro(p, q, only_signs));
        ++s.num_macros;
      } while (s.num_macros < SWEEP_MAX_MACROS && p.remaining && (only_signs || p.closure(group, CHAIN_GATES) >= CHAIN_GATES));
      if (!(bits & line)) s.flags = (uint8_t)(SWEEP_STORES | (segments.empty() ? SWEEP_LOADS : 0));
      segments.push_back(s);
    }
    for (size_t k = 0; k + 1 < segments.size(); ++k) segments[k].flags &= (uint8_t)~SWEEP_STORES;
    h.num_segments = (uint32_t)segments.size();
    h.num_macros = (uint32_t)macros.size();
    h.macros_at = (uint32_t)(sizeof(sweep_header) + segments.size() * sizeof(sweep_segment));
    const size_t bytes = h.macros_at + macros.size() * sizeof(sweep_macro);
    program.assign((bytes + 63) & ~(size_t)63, 0);
    std::memcpy(program.data(), &h, sizeof(h));
    std::memcpy(program.data() + sizeof(h), segments.data(), segments.size() * sizeof(sweep_segment));
    std::memcpy(program.data() + h.macros_at, macros.data(), macros.size() * sizeof(sweep_macro));
    if (int st = emit(program.data(), program.size())) return st;
  }
  return 0;
}

}  // namespace brk
