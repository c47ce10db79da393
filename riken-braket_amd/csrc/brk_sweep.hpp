// Sweeps of the adjoint gradient over circuits of one-qubit gates and Z / CZ: the forward pass and
// the reverse sweep with its gradient terms.
//
// The sweep's results are sums, not amplitudes compared bit for bit with another path, so its
// blocks merge what commutes: all diagonal gates between two mixing gates of a qubit.  A block holds
// chunks of 2^L amplitudes (of psi, in the reverse sweep of psi and lambda) in LDS and runs
// segments: each thread takes the group of 8 amplitudes over three local bits into registers and
// runs macros on it.  A macro applies, in this order,
//   signs   Z and CZ gates on any qubits, as sign terms (d, A): the sign of an amplitude with index
//           x is the parity of popcount(x & (x >> d) & A);
//   phases  the one-qubit diagonal gates of the group's qubits, as one table of 8 factors;
//   mixing  at most one 2x2 gate on each of the group's qubits.
// In the reverse sweep the gates are the inverses, last first, and a gate with a parameter adds its
// gradient term before it is un-applied: for all phases of a macro from one product per amplitude.
//
// Planned by host/sweep.cpp.  Plain C++: included by host code compiled without HIP.
#pragma once

#include <cstdint>

namespace brk {

constexpr int SWEEP_GROUP = 3;          // group bits of a segment: 8 amplitudes per thread and state
constexpr int SWEEP_MAX_TERMS = 4;      // sign terms of a macro
constexpr int SWEEP_MAX_MACROS = 4;     // macros of a segment (its gradient sums are kept in LDS)
constexpr int SWEEP_MAX_QUBITS = 32;    // amplitude indices are 32-bit
constexpr int SWEEP_VALUES = 2 * SWEEP_GROUP;  // gradient terms of a macro: phases, then mixing gates

constexpr int SWEEP_FORWARD_LOCAL = 12;       // 512 threads; 64 KiB (c128) or 32 KiB of LDS
constexpr int SWEEP_REVERSE_LOCAL_C128 = 11;  // 256 threads; 2 x 32 KiB
constexpr int SWEEP_REVERSE_LOCAL_C64 = 12;   // 512 threads; 2 x 32 KiB

enum sweep_mix { SWEEP_MIX_NONE = 0, SWEEP_MIX_REAL = 1, SWEEP_MIX_X = 2, SWEEP_MIX_GENERAL = 3 };
enum sweep_form { SWEEP_FORM_NONE = 0, SWEEP_FORM_Y = 1, SWEEP_FORM_X = 2 };  // gradient of a mixing gate

struct sweep_macro {
  uint32_t num_terms;
  uint32_t uniform;         // bit m: parity of the terms over the group's own bits in member m (not in a table)
  uint32_t d[SWEEP_MAX_TERMS], A[SWEEP_MAX_TERMS];
  uint32_t phases;          // 1: multiply by phase[]
  uint32_t phase_grads;     // bit b: the phase of group bit b has a gradient term
  uint32_t any_grads;       // 1: the macro has gradient terms
  uint32_t mix[SWEEP_GROUP], form[SWEEP_GROUP];
  int32_t slot[8];          // parameter of value v (phases 0..2, mixing gates 3..5), -1: none
  uint32_t pad;
  double weight[SWEEP_GROUP][2];      // of a phase's sums over the members with its bit clear and set
  double mix_weight[SWEEP_GROUP][2];  // of a mixing gate's two sums
  double phase[1 << SWEEP_GROUP][2];
  double matrix[SWEEP_GROUP][8];
};

enum sweep_flags {
  SWEEP_LOADS = 1,   // the first segment: straight from the state
  SWEEP_STORES = 2   // the last segment: straight to the state
};
struct sweep_segment {
  uint8_t group[4];   // ascending local bits
  uint8_t qubits[4];  // ... and the physical qubits they are
  uint8_t flags, num_macros;  // its macros follow those of the segments before it
  uint16_t pad16;
  uint32_t pad;
};
struct sweep_header {
  uint32_t num_segments;  // they follow the header
  uint32_t macros_at;     // byte offset of the macros
  uint8_t pos[16];        // ascending physical qubits of the local bits
  uint32_t num_macros;
  uint32_t pad;
};
static_assert(sizeof(sweep_header) == 32 && sizeof(sweep_segment) == 16 && sizeof(sweep_macro) % 8 == 0, "packed");

// Launches a block (its program in device memory) on psi, and in the reverse sweep (lam not null) on
// psi and lam with the gradient terms into partials[slot * chunks + chunk].
int launch_sweep(const void* device_program, unsigned num_local, void* psi, void* lam, uint64_t size, int dtype,
                 double* partials, void* stream);

}  // namespace brk
