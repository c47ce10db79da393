// Gate blocks: runs of consecutive gates applied to one LDS-resident chunk of
// the state per workgroup.
//
// A gate is first described in physical-qubit terms (gate_desc) by the same
// code that computes the plain kernels' coefficients, so a block applies each
// gate with the plain path's arithmetic and gives bit-identical amplitudes.
// The planner (host/block.cpp) turns the descriptions of one block into a
// program over local bit positions; the kernel (brk_gates.hip) loads
// the 2^L amplitudes of a chunk, applies the program in LDS and stores them.
// Plain C++ only: included by host code compiled without HIP.
#pragma once

#include <cstddef>
#include <cstdint>

namespace brk {

constexpr int BLOCK_LDS_BYTES = 65536;            // largest chunk: 64 KiB of LDS (two workgroups per CU)
constexpr int BLOCK_THREADS = 512;
constexpr int BLOCK_MAX_LOCAL_C128 = 12;          // 2^12 x 16 B = 64 KiB
constexpr int BLOCK_MAX_LOCAL_C64 = 13;           // 2^13 x 8 B  = 64 KiB
constexpr int BLOCK_MAX_OPS = 64;
constexpr int BLOCK_THREAD_BITS = 9;              // log2(BLOCK_THREADS)

// modes of a described gate: the pair modes of the plain kernels, or diagonal
enum block_mode { BLOCK_H = 0, BLOCK_SWAP = 1, BLOCK_MATRIX = 2, BLOCK_ESWAP = 3, BLOCK_DIAG = 4 };

// One gate in physical-qubit terms.  Pair modes act on (i0, i0 ^ flip) for
// every i0 with bit pair_bit clear and all `cond` bits set; diagonal mode
// multiplies every amplitude with all `cond` bits set by u[0..1] (even parity
// of i & zmask) or u[2..3] (odd).  `sign` is the matrix mode's sign-flip
// parity mask and ESWAP's higher-qubit bit.
struct gate_desc {
  int mode;
  unsigned pair_bit;
  uint64_t flip, cond, sign, zmask;
  uint64_t qubits;  // every qubit the gate reads or writes
  double u[8];
};

// Describes an op (physical qubits; op codes of brk_op_code).  Returns
// BRK_OK, or BRK_ERR_UNSUPPORTED for ops without a description (local swap).
int describe_physical_op(int code, const unsigned* targets, unsigned num_targets, const unsigned* controls,
                         unsigned num_controls, const double* params, gate_desc* out);

// The share of the state that the gate's plain kernel reads and writes: a condition bit above the line
// boundary halves it.
double plain_share(const gate_desc& d, int dtype);

// What a block's kernel does for a gate: the described mode, with a 2x2 matrix told apart by the
// exact zeros of its coefficients (the forms of pair_math).
enum block_kind {
  BLOCK_KIND_H = 0, BLOCK_KIND_SWAP = 1, BLOCK_KIND_MATRIX = 2, BLOCK_KIND_ESWAP = 3, BLOCK_KIND_DIAG = 4,
  BLOCK_KIND_REAL = 5,   // a real 2x2 (RY, EY); off-diagonal entries under the sign mask, if any
  BLOCK_KIND_X = 6,      // [[r, i s], [i s', r']] (RX, EX); the same
  BLOCK_KIND_NEGATE = 7, // diagonal with u = (-1, -1) (Z, CZ): an exact negation on cond
  BLOCK_KIND_SIGNED = 8  // (kernels: any 2x2 under a sign mask)
};

// A gate of a block with its masks over local bit positions (bit r of a chunk index <-> physical
// qubit pos[r]).  Only the bits a pair gate flips have to be local: control bits and diagonal
// parity bits outside the chunk are the same for all its amplitudes (outer_cond: the gate acts on
// the chunk only where all these physical bits are set; outer_zmask: their parity joins zmask's).
// A single pass visits only the local indices the gate acts on: item v -> v with zeros inserted at
// the bits of `inserted` (the pair bit and the cond bits), then the cond bits set.
struct block_op {
  uint8_t kind, pair_bit;
  uint8_t group_flip, pad8;         // register segments: flip over the group index
  uint8_t group_zmask, group_cond;  // register segments: the masks' parts over the group index
                                    // (zmask, a pair gate's sign; cond),
  uint16_t coef;                    // first of its coefficients (none for H, SWAP, NEGATE)
  uint16_t flip, cond, sign, zmask;
  uint16_t inserted;
  uint16_t thread_cond, thread_zmask, pad;  // ... and over the other local bits
  uint64_t outer_cond, outer_zmask;
};
static_assert(sizeof(block_op) == 40, "read as five 64-bit words");

// A pass over the chunk.  A segment pass gives every thread one group of 2^(L - 9)
// amplitudes -- local indices that differ only in the bits group[0..] -- in registers
// and applies several gates to it: diagonal gates, and pair gates whose flipped bits
// are group bits.  Gates that only move amplitudes (X, CNOT, SWAP, local swaps) on any
// local bits come after them (num_moves ops): the segment writes its amplitudes to the
// indices they move to.  A single pass applies one gate to the chunk in LDS with a
// strided loop.  The program's ops lie in the order of its passes.
enum block_pass_kind { BLOCK_PASS_SEGMENT = 0, BLOCK_PASS_SINGLE = 1 };
enum block_pass_flags {
  BLOCK_PASS_LOADS = 1,  // the first pass: its groups come straight from the state
  BLOCK_PASS_STORES = 2, // the last pass: its groups go straight to the state
  BLOCK_PASS_LINEAR = 4  // every move is linear in the index bits (X, CNOT, SWAP: at most one local condition)
};
struct block_pass {
  uint8_t kind, num_ops, num_moves, flags;
  uint8_t group[4];   // ascending local bits of the group (L - 9 of them)
  uint8_t qubits[4];  // ... and the physical qubits they are
  uint32_t pad;
};

struct block_header {
  uint32_t num_ops;
  uint32_t num_local;   // L
  uint32_t num_passes;  // they follow the header
  uint16_t ops_at, coefs_at;  // byte offsets from the header: the ops, the coefficients (double)
  uint8_t pos[16];      // ascending physical qubits of the local bits
};
static_assert(sizeof(block_header) == 32 && sizeof(block_pass) == 16, "packed");

// A block's program with room for every block.
constexpr int BLOCK_COEFS = 8;  // at most, per op
struct block_program {
  block_header h;
  block_pass passes[BLOCK_MAX_OPS];
  block_op ops[BLOCK_MAX_OPS];
  double coefs[BLOCK_COEFS * BLOCK_MAX_OPS + BLOCK_COEFS];  // (a kernel reads 8 from any op's first one)
};

// A program packed for a launch's kernel arguments: header, passes, ops and coefficients one after
// the other.  The planner closes a block before its program outgrows them.  No device memory holds
// the program, so a run allocates, uploads and keeps nothing, and its launches can be captured.
constexpr size_t BLOCK_ARG_BYTES = 3840;
struct alignas(8) block_args {
  block_header h;
  uint8_t data[BLOCK_ARG_BYTES - sizeof(block_header)];
};
// Room the ops may take in the arguments, each itself, a pass and its coefficients (beside the
// coefficients read past the last ones).
constexpr size_t BLOCK_ARG_ROOM =
    BLOCK_ARG_BYTES - sizeof(block_header) - BLOCK_COEFS * sizeof(double);
inline int block_op_coefs(const gate_desc& d) {
  if (d.mode == BLOCK_MATRIX) return 8;
  if (d.mode == BLOCK_ESWAP) return 4;
  if (d.mode != BLOCK_DIAG) return 0;
  return d.u[0] == -1.0 && d.u[1] == 0.0 && d.u[2] == -1.0 && d.u[3] == 0.0 ? 0 : 4;
}
inline size_t block_op_room(const gate_desc& d) {
  return sizeof(block_op) + sizeof(block_pass) + sizeof(double) * (size_t)block_op_coefs(d);
}

// A gate of an adjoint block with its masks over local bit positions (every qubit local): item
// v -> j = v with zeros inserted at ins[0..nins) (ascending: the pair bit and the cond bits), then
// the cond bits set.
struct adjoint_op {
  int32_t mode;
  uint32_t pair_bit, flip, cond, sign, zmask;
  uint32_t nins;
  uint32_t ins[15];
  uint32_t group_flip, group_pair;  // register segments: flip and pair bit over the group index
  uint32_t negate;                   // diagonal with u = (-1, -1) (Z, CZ): an exact negation on cond
  uint32_t group_zmask;              // register segments: zmask over the group index, ~0 if not inside
  double u[8];
};

// Its passes: segments of several gates on a thread's group, and single gates.
struct adjoint_pass {
  int32_t kind;
  uint32_t first_op, num_ops;
  uint32_t group[4];  // ascending local bits of the group (L - 9 of them)
};

struct adjoint_base {
  uint32_t num_ops;
  uint32_t num_local;                   // L
  uint32_t num_passes;
  uint32_t pos[16];                     // ascending physical qubits of the local bits
  uint64_t deposit_high[16];            // physical offset of local index k << BLOCK_THREAD_BITS
  adjoint_pass passes[BLOCK_MAX_OPS];
  adjoint_op ops[BLOCK_MAX_OPS];
};

// Reverse sweep of the adjoint method in blocks: chunks of psi and lambda are
// held in LDS together (2^11 complex<double> or 2^12 complex<float>
// amplitudes each, 32 KiB apiece) while the block's ops -- the inverses of
// the circuit's ops, in reverse order -- are un-applied to both.  Before a
// parametric op (one target, no controls) is un-applied, its term
// 2 Re <lambda| D |psi> is summed over the chunk into
// partials[grad_slot * num_chunks + chunk] (FP64, fixed order).
constexpr int ADJ_BLOCK_LOCAL_C128 = 11;
constexpr int ADJ_BLOCK_LOCAL_C64 = 12;
constexpr int ADJ_SEGMENT_GRADIENTS = 8;  // parametric ops per register segment
// Forms of a parametric op's arithmetic, from the exact zeros of D and of the inverse op's
// 2x2: the general formulas with their zero terms left out (the same values).
//   Z: D = diag(i a, i b), the inverse op diagonal on the parity of the target
//      (RZ, EZ) or on its 1 side (U1);
//   Y: D = [[0, a], [b, 0]] real, the inverse op a real 2x2 (RY, EY);
//   X: D = [[0, i a], [i b, 0]], the inverse op [[r, i s], [i s', r']] (RX, EX).
enum adjoint_grad_kind { ADJ_GRAD_GENERAL = 0, ADJ_GRAD_Z = 1, ADJ_GRAD_Y = 2, ADJ_GRAD_X = 3 };
struct adjoint_block_program {
  adjoint_base base;                   // the inverse ops; their passes
  int32_t grad_slot[BLOCK_MAX_OPS];    // -1: no gradient term
  int32_t grad_kind[BLOCK_MAX_OPS];    // adjoint_grad_kind of a parametric op
  double d[BLOCK_MAX_OPS][8];          // D = (dU/dtheta) U^dagger, (re, im) of d00, d01, d10, d11
};
int launch_adjoint_block(const adjoint_block_program* device_program, const adjoint_block_program& program,
                         void* psi, void* lam, uint64_t size, int dtype, double* partials, void* stream);
// out[p] = scale * (sum over c of partials[p * chunks + c]) for p < rows, on the device in a
// fixed order (one workgroup per row: strided per-thread sums, then a tree).
int sum_gradient_partials(const double* partials, unsigned rows, uint64_t chunks, double scale, double* out,
                          void* stream);

// Whether the adjoint gradient runs in blocks (tuning adjoint_blocks).
bool adjoint_blocks_enabled();

// An adjoint block's gates (physical qubits of an n-qubit state): local qubits are their qubits,
// the line_bits lowest qubits, then the lowest others, num_local in all.  Makes no passes.
void make_adjoint_base(const gate_desc* descs, unsigned count, unsigned n, unsigned num_local, unsigned line_bits,
                       adjoint_base* out);

// Local qubits of a chunk for this dtype under the current tuning (block_lds).
unsigned block_max_local(int dtype);
// Number of lowest qubits every chunk keeps local (contiguous runs of block_run_bytes).
unsigned block_run_qubits(int dtype);

// Launches one block over a state of `size` amplitudes: 2^(n - L) workgroups.
int launch_block(const block_args& program, void* first, uint64_t size, int dtype, void* stream);

}  // namespace brk
