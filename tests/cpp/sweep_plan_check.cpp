// Plans long circuits for the adjoint gradient's sweeps (riken-braket_amd/host/sweep.hpp) and reads the
// programs back: every segment's macros follow the ones before, and the macros that the segments run
// hold every gate's parameter exactly once.  No device needed.
//   sweep_plan_check chain|layers|phases NUM_GATES NUM_QUBITS NUM_LOCAL
//     chain   RY and RX in turn on the highest qubit
//     layers  RY and RZ on every qubit, then a CZ ladder, again and again
//     phases  RZ after RZ on the highest qubit, CZ between the two lowest ones in turn with them
// Prints the blocks, the macros of the largest block and the planner's seconds.
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "sweep.hpp"

using namespace brk;

static sweep_gate rotation(unsigned q, char axis, double theta, int param) {
  sweep_gate g;
  g.q = q;
  g.param = param;
  const double c = std::cos(theta / 2), s = std::sin(theta / 2);
  g.u[0] = g.u[6] = c;
  if (axis == 'z') {
    g.diagonal = true;
    g.u[1] = -s;
    g.u[7] = s;
    g.d[1] = -0.5;
    g.d[7] = 0.5;
  } else if (axis == 'y') {
    g.u[2] = -s;
    g.u[4] = s;
    g.d[2] = -0.5;
    g.d[4] = 0.5;
  } else {
    g.u[3] = g.u[5] = -s;
    g.d[3] = g.d[5] = -0.5;
  }
  return g;
}

static sweep_gate cz(unsigned a, unsigned b) {
  sweep_gate g;
  g.sign = true;
  g.mask = 1u << a | 1u << b;
  return g;
}

int main(int argc, char** argv) {
  if (argc != 5) return 2;
  const std::string kind = argv[1];
  const size_t count = std::strtoul(argv[2], nullptr, 10);
  const unsigned n = (unsigned)std::atoi(argv[3]), num_local = (unsigned)std::atoi(argv[4]), line_bits = 3;
  std::vector<sweep_gate> gates;
  int params = 0;
  while (gates.size() < count) {
    const double theta = 0.1 + 0.001 * (double)(gates.size() % 1000);
    if (kind == "chain") {
      gates.push_back(rotation(n - 1, params % 2 ? 'x' : 'y', theta, params));
      ++params;
    } else if (kind == "phases") {
      gates.push_back(rotation(n - 1, 'z', theta, params++));
      gates.push_back(cz(0, 1));
    } else {
      for (unsigned q = 0; q < n; ++q) {
        gates.push_back(rotation(q, 'y', theta, params++));
        gates.push_back(rotation(q, 'z', theta, params++));
      }
      for (unsigned q = 0; q + 1 < n; ++q) gates.push_back(cz(q, q + 1));
    }
  }
  std::vector<unsigned> seen((size_t)params, 0);
  size_t blocks = 0, largest = 0, wrong = 0, bytes_in_all = 0;
  const auto start = std::chrono::steady_clock::now();
  const int status = plan_sweep(gates, n, num_local, line_bits, [&](const void* program, size_t bytes) -> int {
    const char* p = static_cast<const char*>(program);
    sweep_header h;
    std::memcpy(&h, p, sizeof(h));
    size_t next = 0;
    for (uint32_t s = 0; s < h.num_segments; ++s) {
      sweep_segment seg;
      std::memcpy(&seg, p + sizeof(h) + s * sizeof(seg), sizeof(seg));
      const size_t first = next;
      next += seg.num_macros;
      if (seg.num_macros == 0 || next > h.num_macros) ++wrong;
      for (size_t m = first; m < next && m < h.num_macros; ++m) {
        sweep_macro mac;
        std::memcpy(&mac, p + h.macros_at + m * sizeof(mac), sizeof(mac));
        for (int32_t slot : mac.slot)
          if (slot >= 0) ++seen[(size_t)slot];
      }
    }
    if (next != h.num_macros) ++wrong;
    if (h.macros_at + (size_t)h.num_macros * sizeof(sweep_macro) > bytes || bytes % 64 != 0) ++wrong;
    if (bytes > SWEEP_BLOCK_BYTES) ++wrong;
    ++blocks;
    largest = std::max(largest, (size_t)h.num_macros);
    bytes_in_all += bytes;
    return 0;
  });
  const double seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - start).count();
  size_t missed = 0, twice = 0;
  for (unsigned k : seen) {
    missed += k == 0;
    twice += k > 1;
  }
  if (bytes_in_all > sweep_program_bound(gates.size())) ++wrong;
  std::printf("status %d blocks %zu largest %zu wrong %zu missed %zu twice %zu seconds %.3f\n", status, blocks, largest,
              wrong, missed, twice, seconds);
  return status || wrong || missed || twice;
}
