// Planner of the adjoint gradient's sweeps (csrc/brk_sweep.hpp).
#pragma once

#include <complex>
#include <cstdint>
#include <functional>
#include <vector>

#include "brk_sweep.hpp"

namespace brk {

// A gate of a sweep, in the order it is applied: a sign (Z, CZ) on the qubits of `mask`, or a 2x2
// on qubit q -- diagonal ones are phases -- with its gradient term's matrix D if it has a parameter.
struct sweep_gate {
  bool sign = false;
  bool diagonal = false;
  uint32_t mask = 0;
  unsigned q = 0;
  double u[8] = {};      // 2x2, row-major (re, im); of a phase the diagonal counts
  int param = -1;
  double d[8] = {};      // D of a gate with a parameter (reverse sweep)
};

// Plans the gates (on n qubits) into blocks over num_local local qubits, the line_bits lowest always
// among them, and hands each block's program (a multiple of 64 bytes) to emit as soon as it is made;
// a status other than BRK_OK from emit ends the plan.  The gates run in an order that keeps every
// mixing gate's place among the gates on its qubit; diagonal gates commute.
int plan_sweep(const std::vector<sweep_gate>& gates, unsigned n, unsigned num_local, unsigned line_bits,
               const std::function<int(const void* program, size_t bytes)>& emit);

// A block ends at this many macros (ordinary ones hold below 100; every macro runs a gate at least), so
// that its program has a size that does not depend on the circuit's.
constexpr size_t SWEEP_BLOCK_MACROS = 1024;
constexpr size_t SWEEP_BLOCK_BYTES =
    sizeof(sweep_header) + SWEEP_BLOCK_MACROS * (sizeof(sweep_macro) + sizeof(sweep_segment)) + 64;

// Bytes the programs of a plan of this many gates take at most: a macro and a segment for every
// gate, and a block's header and padding (every block runs at least one gate).
inline size_t sweep_program_bound(size_t gates) {
  return (gates + 1) * (sizeof(sweep_macro) + sizeof(sweep_segment) + sizeof(sweep_header) + 64);
}

}  // namespace brk
