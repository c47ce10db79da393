// What brk_circuit_run and a block plan of a circuit launch, without a device: the engine's two launch
// functions are replaced by ones that print (the library's calls to them resolve to this program's).
//   block_launch_check NUM_QUBITS DTYPE < ops
// An op a line: its code, then the targets, controls and parameters, each list behind its length.
// Prints a line per launch: "block NUM_OPS" or "plain CODE", first of the run, after a line "plan" of the plan.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <iostream>
#include <vector>

#include "brk_block.hpp"
#include "circuit.hpp"

namespace brk {
int launch_block(const block_args& program, void*, uint64_t, int, void*) {
  std::printf("block %u\n", program.h.num_ops);
  return BRK_OK;
}
int apply_physical_op(const brk_circuit::op& o, void*, uint64_t, int, void*) {
  std::printf("plain %d\n", o.code);
  return BRK_OK;
}
}  // namespace brk

int main(int argc, char** argv) {
  if (argc != 3) return 2;
  const unsigned n = (unsigned)std::atoi(argv[1]);
  const int dtype = std::atoi(argv[2]);
  brk_circuit* circuit = nullptr;
  if (brk_circuit_create(n, &circuit)) return 1;
  int code;
  while (std::cin >> code) {
    std::vector<unsigned> q[2];
    std::vector<double> params;
    unsigned count;
    for (auto& list : q) {
      std::cin >> count;
      list.resize(count);
      for (unsigned& x : list) std::cin >> x;
    }
    std::cin >> count;
    params.resize(count);
    for (double& x : params) std::cin >> x;
    if (brk_circuit_add(circuit, code, q[0].data(), (unsigned)q[0].size(), q[1].data(), (unsigned)q[1].size(),
                        params.data(), (unsigned)params.size()))
      return 1;
  }
  void* const state = reinterpret_cast<void*>(4096);  // (never read)
  if (brk_circuit_run(circuit, state, dtype, nullptr, nullptr)) return 1;
  std::printf("plan\n");
  brk_block_plan* plan = nullptr;
  if (brk_block_plan_create(circuit, dtype, nullptr, &plan)) return 1;
  if (brk_block_plan_run(plan, state, nullptr)) return 1;
  brk_block_plan_destroy(plan);
  brk_circuit_destroy(circuit);
  return 0;
}
