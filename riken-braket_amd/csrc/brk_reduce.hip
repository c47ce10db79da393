// FP64 reductions over a state vector: inner product, norm, spin expectation
// values, Pauli-string expectation values and the open-chain Ising energy,
// plus H|psi> for that Hamiltonian.
//
// A reduction runs on a grid that its state's size fixes -- RED_BLOCKS blocks, the
// Ising energy up to ISING_GRID a pass -- so the assignment of amplitudes to
// threads, the in-block tree and the host-side sum over the block partials (in
// block order) are the same on every call: results are bit-reproducible.  The blocks write their partials straight to pinned host
// memory (24 KB at most): a copy back costs about 10 us more per call.  Partial sums are kept in
// double whatever the element type (the reference accumulates per-thread
// partials and then std::accumulate's them, inner_product.hpp:43-55; spin
// values use long double, spin_expectation_value.hpp:31-64).
#include "brk_internal.hpp"
#include "brk_adjoint.hpp"
#include "brk_block.hpp"

#include <algorithm>
#include <cmath>
#include <complex>
#include <vector>

namespace brk {

// The items 0 .. n - 1 of a reduction, n a power of two: block b takes the tiles b, b + RED_BLOCKS, ...
// of RED_UNROLL * RED_THREADS consecutive items, a tile's loads all in flight before its first add.
// Bound: HBM reads.  A 4 GiB state's spin value (two amplitudes an item): 0.67-0.73 ms, 5.9-6.4 TB/s
// by qubit; with the unrolled items a whole grid apart, the tiles' rows in RED_UNROLL places at a
// time, 0.75-0.88 ms; one item a time that way 0.69-0.74.  (65536 blocks of one tile each: 0.66-0.68,
// but 1.5 MB of partials.)
constexpr int RED_UNROLL = 4;

template <typename Load, typename Add>
__device__ __forceinline__ void for_tiles(uint64_t n, Load load, Add add) {
  constexpr uint64_t TILE = (uint64_t)RED_UNROLL * RED_THREADS;
  for (uint64_t t = (uint64_t)blockIdx.x * TILE; t < n; t += (uint64_t)RED_BLOCKS * TILE) {
    if (t + TILE <= n) {
      decltype(load(t)) x[RED_UNROLL];
#pragma unroll
      for (int u = 0; u < RED_UNROLL; ++u) x[u] = load(t + (uint64_t)(u * RED_THREADS) + threadIdx.x);
#pragma unroll
      for (int u = 0; u < RED_UNROLL; ++u) add(x[u]);
    } else {
      for (uint64_t i = t + threadIdx.x; i < n; i += RED_THREADS) add(load(i));
    }
  }
}

// Two amplitudes of an item.
template <typename R1, typename R2>
struct amp_pair {
  cpx<R1> x;
  cpx<R2> y;
};

template <int NV>
struct dvec {
  double v[NV];
};

__device__ __forceinline__ double wave_sum(double x) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) x += __shfl_down(x, off, 64);
  return x;
}

// Reduces `acc` over the block and writes it to partial[blockIdx.x * NV + v].
template <int NV>
__device__ __forceinline__ void block_store(dvec<NV> acc, double* __restrict__ partial) {
  __shared__ double lds[RED_THREADS / 64][NV];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int v = 0; v < NV; ++v) {
    double x = wave_sum(acc.v[v]);
    if (lane == 0) lds[wave][v] = x;
  }
  __syncthreads();
  if (threadIdx.x < NV) {
    double t = 0.0;
#pragma unroll
    for (int w = 0; w < RED_THREADS / 64; ++w) t += lds[w][threadIdx.x];
    partial[(size_t)blockIdx.x * NV + threadIdx.x] = t;
  }
}

template <typename R1, typename R2>
__global__ __launch_bounds__(RED_THREADS) void k_inner(const cpx<R1>* __restrict__ a, const cpx<R2>* __restrict__ b,
                                                      uint64_t size, double* partial) {
  dvec<2> acc{{0.0, 0.0}};
  for_tiles(
      size, [&](uint64_t i) { return amp_pair<R1, R2>{a[i], b[i]}; },
      [&](const amp_pair<R1, R2>& p) {
        const double xr = p.x.re, xi = p.x.im, yr = p.y.re, yi = p.y.im;
        // conj(y) * x
        acc.v[0] += yr * xr + yi * xi;
        acc.v[1] += yr * xi - yi * xr;
      });
  block_store<2>(acc, partial);
}

template <typename R>
__global__ __launch_bounds__(RED_THREADS) void k_norm(const cpx<R>* __restrict__ a, uint64_t size, double* partial) {
  dvec<1> acc{{0.0}};
  for_tiles(
      size, [&](uint64_t i) { return a[i]; },
      [&](const cpx<R>& x) {
        const double xr = x.re, xi = x.im;
        acc.v[0] += xr * xr + xi * xi;
      });
  block_store<1>(acc, partial);
}

// Pairs of `qubit`: (Re conj(a0) a1, Im conj(a0) a1, |a0|^2 - |a1|^2).
template <typename R>
__global__ __launch_bounds__(RED_THREADS) void k_spin(const cpx<R>* __restrict__ a, uint64_t npairs, uint64_t lower,
                                                     uint64_t qmask, double* partial) {
  dvec<3> acc{{0.0, 0.0, 0.0}};
  for_tiles(
      npairs,
      [&](uint64_t g) {
        const uint64_t i0 = ((g & ~lower) << 1) | (g & lower);
        return amp_pair<R, R>{a[i0], a[i0 | qmask]};
      },
      [&](const amp_pair<R, R>& p) {
        const double r0 = p.x.re, m0 = p.x.im, r1 = p.y.re, m1 = p.y.im;
        acc.v[0] += r0 * r1 + m0 * m1;
        acc.v[1] += r0 * m1 - m0 * r1;
        acc.v[2] += (r0 * r0 + m0 * m0) - (r1 * r1 + m1 * m1);
      });
  block_store<3>(acc, partial);
}

// sum_i conj(a_i) a_{i ^ flip} (-1)^{popcount(i & sign)}
template <typename R>
__global__ __launch_bounds__(RED_THREADS) void k_pauli(const cpx<R>* __restrict__ a, uint64_t size, uint64_t flip,
                                                      uint64_t sign, double* partial) {
  struct item {
    cpx<R> x, y;
    bool odd;
  };
  dvec<2> acc{{0.0, 0.0}};
  for_tiles(
      size, [&](uint64_t i) { return item{a[i], a[i ^ flip], (__popcll(i & sign) & 1) != 0}; },
      [&](const item& p) {
        const double xr = p.x.re, xi = p.x.im, yr = p.y.re, yi = p.y.im;
        double re = xr * yr + xi * yi;
        double im = xr * yi - xi * yr;
        if (p.odd) {
          re = -re;
          im = -im;
        }
        acc.v[0] += re;
        acc.v[1] += im;
      });
  block_store<2>(acc, partial);
}

constexpr int MAX_CHAIN = 48;

struct ising_args {
  double J[MAX_CHAIN];
  double h[MAX_CHAIN];
  int n;
};

// Diagonal part of the Ising Hamiltonian at basis index k.
__device__ __forceinline__ double ising_diag(uint64_t k, const ising_args& a) {
  const uint64_t x = k ^ (k >> 1);  // bit i = b_i xor b_{i+1}
  double e = 0.0;
  for (int i = 0; i + 1 < a.n; ++i) e += ((x >> i) & 1ull) ? -a.J[i] : a.J[i];
  return e;
}

// <H> of the open-chain Ising Hamiltonian in a few passes over the state.  A pass holds chunks of
// 2^L amplitudes (64 KiB: L = 12 for c128, 13 for c64) whose L local bits are the physical qubits
// pos[]; a thread loads PER = 2^GB amplitudes differing in the GB highest local bits, adds those
// bits' X terms in registers and, in the first pass, the ZZ terms; the chunk then goes to LDS once
// and is read back in groups of PER amplitudes over the other local bits, GB bits a round.  The
// next chunk's loads are in flight during the rounds.  The first pass takes qubits 0 .. L - 1, each
// further one the 128-byte line's qubits and up to L - line others: 3 reads of a 28-qubit c128 state
// instead of the 29 of one pass per term.  Bound: HBM reads (28 qubits c128: 0.81 ms a pass, 5.3 TB/s,
// 2.4 ms in all; a pass per term took 22 ms).
// LDS addresses are XOR-swizzled so that both access shapes spread over all banks.
constexpr int ISING_THREADS = 512;
constexpr int ISING_THREAD_BITS = 9;
constexpr int ISING_GRID = 512;  // two workgroups per CU; fixed, so that the summation order is
constexpr int ISING_TABLES = MAX_CHAIN / 8;
constexpr int ISING_MAX_LOCAL = 13;

struct ising_pass {
  double J[MAX_CHAIN];
  double h2[ISING_MAX_LOCAL];      // 2 h of the qubit at a local position
  uint32_t pos[ISING_MAX_LOCAL];   // ascending; L entries
  uint32_t measure;                // local positions whose X term is added
  int n;
  int zz;                          // add the ZZ terms (the local bits are then 0 .. L - 1)
};

template <typename R>
struct ising_shape {
  static constexpr int GB = sizeof(R) == 8 ? 3 : 4;
  static constexpr int L = ISING_THREAD_BITS + GB;
};

template <typename R>
__global__ __launch_bounds__(ISING_THREADS) void k_ising(const cpx<R>* __restrict__ a, uint64_t size,
                                                        uint64_t nchunks, ising_pass P,
                                                        double* __restrict__ partial) {
  constexpr int GB = ising_shape<R>::GB, L = ising_shape<R>::L, PER = 1 << GB;
  __shared__ cpx<R> lds[1 << L];
  __shared__ double table[ISING_TABLES * 256];  // ZZ energy of a byte of the bond pattern i ^ (i >> 1)
  __shared__ double wave_sums[ISING_THREADS / 64];
  const uint32_t t = threadIdx.x;
  if (P.zz) {
    for (uint32_t e = t; e < (uint32_t)ISING_TABLES * 256; e += ISING_THREADS) {
      double v = 0.0;
      for (int b = 0; b < 8; ++b) {
        const int bond = 8 * (int)(e >> 8) + b;
        if (bond + 1 < P.n) v += ((e >> b) & 1u) ? -P.J[bond] : P.J[bond];
      }
      table[e] = v;
    }
    __syncthreads();
  }
  auto swizzle = [](uint32_t j) { return j ^ ((j >> GB) & (uint32_t)(PER - 1)); };
  uint64_t low = 0;
#pragma unroll
  for (int r = 0; r < ISING_THREAD_BITS; ++r) low |= (uint64_t)((t >> r) & 1u) << P.pos[r];
  uint64_t high[PER];
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    high[k] = 0;
#pragma unroll
    for (int g = 0; g < GB; ++g)
      if ((k >> g) & 1) high[k] |= 1ull << P.pos[ISING_THREAD_BITS + g];
  }
  auto base_of = [&](uint64_t c) {  // zeros inserted at the local positions
#pragma unroll
    for (int r = 0; r < L; ++r) {
      const uint32_t q = P.pos[r];
      c = ((c >> q) << (q + 1)) | (c & ((1ull << q) - 1ull));
    }
    return c;
  };
  cpx<R> x[PER];
  auto load = [&](uint64_t c) {
    const uint64_t b = base_of(c) | low;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const uint64_t i = b | high[k];
      x[k] = i < size ? a[i] : cpx<R>{R(0), R(0)};  // (a state smaller than a chunk)
    }
  };
  // the X terms of group bits [0, GB) of v, bit g at local position first + g
  double acc = 0.0;
  auto add_x = [&](const cpx<R> (&v)[PER], int first, uint32_t mask) {
#pragma unroll
    for (int g = 0; g < GB; ++g) {
      if (!((mask >> g) & 1u)) continue;
      double s = 0.0;
#pragma unroll
      for (int m = 0; m < PER; ++m) {
        if ((m >> g) & 1) continue;
        const cpx<R> v0 = v[m], v1 = v[m | (1 << g)];
        s = __builtin_fma((double)v0.re, (double)v1.re, s);
        s = __builtin_fma((double)v0.im, (double)v1.im, s);
      }
      acc = __builtin_fma(P.h2[first + g], s, acc);
    }
  };
  const uint32_t in_registers = P.measure >> ISING_THREAD_BITS;
  const bool rounds = (P.measure & ((1u << ISING_THREAD_BITS) - 1u)) != 0;
  uint64_t c = blockIdx.x;
  if (c < nchunks) load(c);
  for (; c < nchunks; c += gridDim.x) {
    add_x(x, ISING_THREAD_BITS, in_registers);
    if (P.zz) {
      // bond bits 0..7 depend on t alone, bits 16.. on the chunk alone
      const uint64_t i0 = (c << L) | t, d0 = i0 ^ (i0 >> 1);
      double fixed = table[d0 & 255u];
      for (int b = 2; 8 * b + 1 < P.n; ++b) fixed += table[256 * b + ((d0 >> (8 * b)) & 255u)];
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const uint64_t i = i0 | ((uint64_t)k << ISING_THREAD_BITS), d = i ^ (i >> 1);
        const double re = x[k].re, im = x[k].im;
        acc = __builtin_fma(__builtin_fma(re, re, im * im), fixed + table[256 + ((d >> 8) & 255u)], acc);
      }
    }
    if (rounds) {
#pragma unroll
      for (int k = 0; k < PER; ++k) lds[swizzle(t + ISING_THREADS * k)] = x[k];
      __syncthreads();
    }
    if (c + gridDim.x < nchunks) load(c + gridDim.x);
    if (rounds) {
#pragma unroll
      for (int first = 0; first < ISING_THREAD_BITS; first += GB) {
        uint32_t mask = (P.measure >> first) & (uint32_t)(PER - 1);
        if (first + GB > ISING_THREAD_BITS) mask &= (1u << (ISING_THREAD_BITS - first)) - 1u;  // the rest: registers
        if (!mask) continue;
        const uint32_t j = ((t >> first) << (first + GB)) | (t & ((1u << first) - 1u));
        cpx<R> v[PER];
#pragma unroll
        for (int m = 0; m < PER; ++m) v[m] = lds[swizzle(j | ((uint32_t)m << first))];
        add_x(v, first, mask);
      }
      __syncthreads();
    }
  }
  acc = wave_sum(acc);
  if ((t & 63u) == 0) wave_sums[t >> 6] = acc;
  __syncthreads();
  if (t == 0) {
    double sum = 0.0;
#pragma unroll
    for (int w = 0; w < ISING_THREADS / 64; ++w) sum += wave_sums[w];
    partial[blockIdx.x] = sum;
  }
}

template <typename R>
__global__ __launch_bounds__(256) void k_apply_ising(cpx<R>* __restrict__ out, const cpx<R>* __restrict__ psi,
                                                    uint64_t size, ising_args args) {
  const uint64_t k = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (k >= size) return;
  cpx<R> x = psi[k];
  const double e = ising_diag(k, args);
  double re = e * (double)x.re, im = e * (double)x.im;
  for (int i = 0; i < args.n; ++i) {
    cpx<R> y = psi[k ^ (1ull << i)];
    re += args.h[i] * (double)y.re;
    im += args.h[i] * (double)y.im;
  }
  out[k] = cpx<R>{(R)re, (R)im};
}

// P(qubit = 0) and P(qubit = 1): sums of |a|^2 over the two halves of the pairs
// (projective_measurement.hpp:36-72, clear.hpp zero_probability).
template <typename R>
__global__ __launch_bounds__(RED_THREADS) void k_zero_one(const cpx<R>* __restrict__ a, uint64_t npairs, uint64_t lower,
                                                         uint64_t qmask, double* partial) {
  dvec<2> acc{{0.0, 0.0}};
  for_tiles(
      npairs,
      [&](uint64_t g) {
        const uint64_t i0 = ((g & ~lower) << 1) | (g & lower);
        return amp_pair<R, R>{a[i0], a[i0 | qmask]};
      },
      [&](const amp_pair<R, R>& p) {
        acc.v[0] += (double)p.x.re * p.x.re + (double)p.x.im * p.x.im;
        acc.v[1] += (double)p.y.re * p.y.re + (double)p.y.im * p.y.im;
      });
  block_store<2>(acc, partial);
}

// Keeps the half of the pairs where the qubit equals `value`, scaled by m, and
// sets the other half to +0 (change_state_after_measuring_zero/one,
// projective_measurement.hpp:74-150; clear.hpp; set.hpp).
template <typename R, bool NT>
__global__ __launch_bounds__(256) void k_project(cpx<R>* __restrict__ a, uint64_t npairs, uint64_t lower,
                                                 uint64_t qmask, int value, R m) {
  const uint64_t g = (uint64_t)blockIdx.x * 256 + threadIdx.x;
  if (g >= npairs) return;
  const uint64_t i0 = ((g & ~lower) << 1) | (g & lower);
  const uint64_t keep = value ? (i0 | qmask) : i0, drop = value ? i0 : (i0 | qmask);
  const cpx<R> x = load_amp<NT>(a + keep);  // NT: large states stream through once
  store_amp<NT>(a + keep, cpx<R>{x.re * m, x.im * m});
  store_amp<NT>(a + drop, cpx<R>{R(0), R(0)});
}

// Sampling (generate_events.hpp:15-48).  The cumulative probability of basis
// index i is a nested left fold: the state is cut into chunks of SAMPLE_CHUNK
// amplitudes, a chunk into 16 waves, a wave into 64 threads and a thread into
// `per` consecutive amplitudes.  With S the running sum over whole chunks,
// W over the waves of the chunk, L over the threads of the wave and c over the
// thread's own amplitudes (each summed left to right from 0.0),
//   C(i) = S + (W + (L + c)).
// The last value of each level equals the next level's running sum exactly,
// so C is monotone and continuous across chunk, wave and thread boundaries:
// an index whose probability is zero repeats its predecessor's C and is
// never the first to exceed a target.  It matches a sequential scan up to
// rounding.
constexpr int SAMPLE_CHUNK = 1 << 13;
constexpr int SAMPLE_THREADS = 1024;
constexpr int SAMPLE_WAVES = SAMPLE_THREADS / 64;
constexpr int SAMPLE_PER = SAMPLE_CHUNK / SAMPLE_THREADS;  // amplitudes per thread of a whole chunk

// Where the norm of an amplitude is kept in LDS: a gap after every 8, so that the threads' reads of
// their 8 consecutive norms fall on different banks (without it 16 lanes shared each).
constexpr uint32_t norm_slot(uint32_t j) { return j + j / SAMPLE_PER; }
constexpr int SAMPLE_SLOTS = norm_slot(SAMPLE_CHUNK);
constexpr int SAMPLE_WAVE_SLOTS = norm_slot(64 * SAMPLE_PER);

__device__ inline double readlane_f64(double v, int lane) {
  const uint64_t b = (uint64_t)__double_as_longlong(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, lane);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), lane);
  return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}

// Coalesced load of one chunk's |a|^2 into LDS.  A whole chunk issues all its
// loads before the first norm is stored (eight in flight per thread).
template <typename R>
__device__ inline void load_norms(const cpx<R>* __restrict__ a, uint64_t base, uint32_t chunk, double* nrm) {
  constexpr int PER = SAMPLE_PER;
  if (chunk == (uint32_t)SAMPLE_CHUNK) {
    cpx<R> x[PER];
#pragma unroll
    for (int k = 0; k < PER; ++k) x[k] = a[base + threadIdx.x + (uint32_t)k * SAMPLE_THREADS];
#pragma unroll
    for (int k = 0; k < PER; ++k)
      nrm[norm_slot(threadIdx.x + (uint32_t)k * SAMPLE_THREADS)] =
          (double)x[k].re * x[k].re + (double)x[k].im * x[k].im;
    return;
  }
  for (uint32_t j = threadIdx.x; j < chunk; j += SAMPLE_THREADS) {
    const cpx<R> x = a[base + j];
    nrm[norm_slot(j)] = (double)x.re * x.re + (double)x.im * x.im;
  }
}

struct chunk_fold {
  double lane_before;  // L before this thread
  double wave_before;  // W before this wave
  double total;        // the chunk's sum
};

// Called by every thread after the norms are in LDS (and a barrier).
__device__ inline chunk_fold fold_chunk(const double* nrm, uint32_t chunk, uint32_t per, double* wave_sums) {
  const uint32_t first = threadIdx.x * per;
  double t = 0.0;
  for (uint32_t k = 0; k < per; ++k)
    if (first + k < chunk) t += nrm[norm_slot(first + k)];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double run = 0.0, before = 0.0;
  for (int k = 0; k < 64; ++k) {
    if (k == lane) before = run;
    run += readlane_f64(t, k);
  }
  if (lane == 0) wave_sums[wave] = run;
  __syncthreads();
  chunk_fold f{before, 0.0, 0.0};
  for (int k = 0; k < SAMPLE_WAVES; ++k) {
    if (k == wave) f.wave_before = f.total;
    f.total += wave_sums[k];
  }
  return f;
}

// The norms of one wave of a chunk: a[0 .. count) (at most 64 * per), per consecutive ones to a lane,
// zeros beyond.  The loads are coalesced and the norms change lanes in the wave's own LDS, so no
// other wave is waited for; a lane that loaded its own 128 bytes had every line fetched again by
// each of its 8 loads (100 000 events: 0.36 ms, now 0.17).
template <typename R>
__device__ __forceinline__ void wave_norms(const cpx<R>* __restrict__ a, uint32_t count, uint32_t per, double* slots,
                                           double (&p)[SAMPLE_PER]) {
  const uint32_t lane = threadIdx.x & 63u;
  auto norm = [](const cpx<R>& x) { return (double)x.re * x.re + (double)x.im * x.im; };
  if (count == 64u * SAMPLE_PER) {
    cpx<R> x[SAMPLE_PER];
#pragma unroll
    for (uint32_t u = 0; u < SAMPLE_PER; ++u) x[u] = a[u * 64u + lane];
#pragma unroll
    for (uint32_t u = 0; u < SAMPLE_PER; ++u) slots[norm_slot(u * 64u + lane)] = norm(x[u]);
  } else {
    for (uint32_t j = lane; j < count; j += 64u) slots[norm_slot(j)] = norm(a[j]);
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (uint32_t k = 0; k < SAMPLE_PER; ++k) {
    const uint32_t j = lane * per + k;
    p[k] = k < per && j < count ? slots[norm_slot(j)] : 0.0;
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

__device__ __forceinline__ uint32_t amps_of_wave(uint32_t chunk, uint32_t per, uint32_t wave) {
  const uint32_t first = wave * 64u * per;
  return first < chunk ? min(chunk - first, 64u * per) : 0u;
}

// wave_out (may be null): the 16 wave sums of every chunk as well, for k_find_events.  Bound: HBM
// reads (a 2 GiB c128 state in 0.33 ms, 6.6 TB/s; 0.45 with the workgroup's norms in one array without
// gaps).
template <typename R>
__global__ __launch_bounds__(SAMPLE_THREADS) void k_chunk_sums(const cpx<R>* __restrict__ a, uint32_t chunk,
                                                              double* __restrict__ sums,
                                                              double* __restrict__ wave_out) {
  __shared__ double slots[SAMPLE_WAVES * SAMPLE_WAVE_SLOTS];
  __shared__ double wave_sums[SAMPLE_WAVES];
  const uint32_t per = chunk >= SAMPLE_THREADS ? chunk / SAMPLE_THREADS : 1;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  double p[SAMPLE_PER];
  wave_norms(a + (uint64_t)blockIdx.x * chunk + wave * 64u * per, amps_of_wave(chunk, per, wave), per,
             slots + wave * SAMPLE_WAVE_SLOTS, p);
  double t = 0.0;
#pragma unroll
  for (int k = 0; k < SAMPLE_PER; ++k) t += p[k];  // (t + 0.0 = t: sums are never -0)
  double run = 0.0;
  for (int k = 0; k < 64; ++k) run += readlane_f64(t, k);
  if ((threadIdx.x & 63u) == 0) wave_sums[wave] = run;
  __syncthreads();
  if (threadIdx.x == 0) {
    double total = 0.0;
    for (int k = 0; k < SAMPLE_WAVES; ++k) total += wave_sums[k];
    sums[blockIdx.x] = total;
  }
  if (wave_out && threadIdx.x < SAMPLE_WAVES)
    wave_out[(uint64_t)blockIdx.x * SAMPLE_WAVES + threadIdx.x] = wave_sums[threadIdx.x];
}

// One wavefront per event, from the running sums S over whole chunks and the wave sums of
// every chunk.  The lanes find the event's chunk together (each step samples 64 points of S:
// 3 steps instead of the 14 of a binary search over 2^14 chunks), the wave of the chunk from
// its 16 sums, and only that wave's amplitudes -- 8 per lane, 8 KiB for c128 -- are read: the
// block that searched a chunk per event read and folded all 128 KiB of it.  C is monotone, so
// the first index that exceeds the target lies in the first wave whose last C does, and C is
// formed with the additions of fold_chunk: the same events bit for bit.  Bound: latency of the
// fold's 64 dependent additions, hidden by the other events' waves; 100 000 events of a 2 GiB
// c128 state take 0.17 ms (0.82 GB read, 4.8 TB/s; the search of whole chunks took 6.5 ms).
constexpr int FIND_THREADS = 256;

template <typename R>
__global__ __launch_bounds__(FIND_THREADS) void k_find_events(const cpx<R>* __restrict__ a, uint32_t chunk,
                                                             const double* __restrict__ S, uint64_t nchunks,
                                                             double total, uint64_t last_chunk,
                                                             const double* __restrict__ chunk_waves,
                                                             const double* __restrict__ canonical,
                                                             unsigned num_events, uint64_t* __restrict__ events) {
  __shared__ double slots[FIND_THREADS / 64 * SAMPLE_WAVE_SLOTS];
  const unsigned e = blockIdx.x * (FIND_THREADS / 64) + (threadIdx.x >> 6);
  if (e >= num_events) return;  // whole waves
  const unsigned lane = threadIdx.x & 63u;
  const double r = canonical[e] * total;
  // the first chunk with S > r
  uint64_t lo = 0, hi = nchunks;  // it is in [lo, hi]; hi: none before
  while (lo < hi) {
    const uint64_t step = (hi - lo + 63) / 64;
    const uint64_t at = min(lo + (lane + 1) * step, hi) - 1;
    const uint64_t over = __ballot(S[at] > r);
    if (!over) {
      lo = hi;
      break;
    }
    const unsigned f = (unsigned)__builtin_ctzll(over);
    hi = min(lo + (f + 1) * step, hi) - 1;
    lo = lo + f * step;
  }
  const uint64_t c = lo >= nchunks ? last_chunk : lo;
  const double start = c ? S[c - 1] : 0.0;
  // the first wave whose last C exceeds r, and the sum before it
  const double mine = lane < (unsigned)SAMPLE_WAVES ? chunk_waves[c * SAMPLE_WAVES + lane] : 0.0;
  double wave_before = 0.0;
  int wave = 0;
  for (; wave < SAMPLE_WAVES; ++wave) {
    const double next = wave_before + readlane_f64(mine, wave);
    if (start + next > r) break;
    wave_before = next;
  }
  const uint32_t per = chunk >= SAMPLE_THREADS ? chunk / SAMPLE_THREADS : 1;
  const uint64_t base = c * chunk;
  constexpr int PER = SAMPLE_PER;
  double p[PER];
  auto load = [&](int w) {  // the lane's probabilities in wave w (0 beyond the chunk)
    wave_norms(a + base + (uint32_t)w * 64u * per, amps_of_wave(chunk, per, (uint32_t)w), per,
               slots + (threadIdx.x >> 6) * SAMPLE_WAVE_SLOTS, p);
  };
  if (wave < SAMPLE_WAVES) {
    load(wave);
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < PER; ++k) t += p[k];  // (t + 0.0 = t: sums are never -0)
    double run = 0.0, before = 0.0;
    for (unsigned k = 0; k < 64; ++k) {
      if (k == lane) before = run;
      run += readlane_f64(t, (int)k);
    }
    double acc = 0.0;
    int found = PER;
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      acc += p[k];
      if (found == PER && start + (wave_before + (before + acc)) > r) found = k;
    }
    const uint64_t hit = __ballot(found < PER);
    if (hit) {
      if (lane == (unsigned)__builtin_ctzll(hit)) events[e] = base + ((uint32_t)wave * 64 + lane) * per + found;
      return;
    }
  }
  // none exceeds r (a target at the total): the chunk's last index of non-zero probability
  for (int w = SAMPLE_WAVES - 1; w >= 0; --w) {
    load(w);
    int last = -1;
#pragma unroll
    for (int k = 0; k < PER; ++k)
      if (p[k] > 0.0) last = k;
    const uint64_t any = __ballot(last >= 0);
    if (any) {
      if (lane == 63u - (unsigned)__builtin_clzll(any)) events[e] = base + ((uint32_t)w * 64 + lane) * per + last;
      return;
    }
  }
  if (lane == 0) events[e] = base;
}

// One block per event: the first index of chunk chunk_of[e] whose C exceeds
// target[e] (chunk_start[e] is S before the chunk).  When none does (a target
// at the total, which the host only sends for the last chunk holding
// probability), the chunk's last index of non-zero probability.
template <typename R>
__global__ __launch_bounds__(SAMPLE_THREADS) void k_chunk_search(const cpx<R>* __restrict__ a, uint32_t chunk,
                                                                const uint64_t* __restrict__ chunk_of,
                                                                const double* __restrict__ chunk_start,
                                                                const double* __restrict__ target,
                                                                uint64_t* __restrict__ events) {
  __shared__ double nrm[SAMPLE_SLOTS];
  __shared__ double wave_sums[SAMPLE_WAVES];
  __shared__ unsigned found, last_nonzero;
  const uint64_t base = chunk_of[blockIdx.x] * chunk;
  const double S = chunk_start[blockIdx.x], r = target[blockIdx.x];
  const uint32_t per = chunk >= SAMPLE_THREADS ? chunk / SAMPLE_THREADS : 1;
  if (threadIdx.x == 0) {
    found = ~0u;
    last_nonzero = 0u;
  }
  load_norms(a, base, chunk, nrm);
  __syncthreads();
  const chunk_fold f = fold_chunk(nrm, chunk, per, wave_sums);
  const uint32_t first = threadIdx.x * per;
  double c = 0.0;
  for (uint32_t k = 0; k < per && first + k < chunk; ++k) {
    const double p = nrm[norm_slot(first + k)];
    c += p;
    if (p > 0.0) atomicMax(&last_nonzero, first + k);
    if (S + (f.wave_before + (f.lane_before + c)) > r) {
      atomicMin(&found, first + k);
      break;
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) events[blockIdx.x] = base + (found != ~0u ? found : last_nonzero);
}

// Launches `launch(partial)` on the fixed reduction grid and sums the NV
// partials per block on the host.
template <int NV, typename Launch>
static int run_reduction(void* stream, Launch launch, double* out) {
  reduce_scratch* sc;
  if (int st = get_reduce_scratch(&sc)) return st;
  // the device's scratch is ours from the launch until the partials are read
  std::lock_guard<std::mutex> hold(sc->busy);
  hipStream_t s = as_stream(stream);
  launch(sc->partials, s);
  if (int st = check_launch("reduction")) return st;
  const hipError_t synced = hipStreamSynchronize(s);
  if (synced != hipSuccess) return fail(BRK_ERR_HIP, "reduction: %s", hipGetErrorString(synced));
  double sum[NV] = {};  // (not in out, which might be part of the partials for all the compiler knows: 0.3 us)
  for (int b = 0; b < RED_BLOCKS; ++b)
    for (int v = 0; v < NV; ++v) sum[v] += sc->partials[b * NV + v];
  std::copy(sum, sum + NV, out);
  return BRK_OK;
}

static int spin_raw(const void* first, uint64_t size, int dtype, unsigned qubit, double out[3], void* stream) {
  const uint64_t qmask = 1ull << qubit, lower = qmask - 1ull, npairs = size >> 1;
  return run_reduction<3>(
      stream,
      [&](double* partial, hipStream_t s) {
        if (dtype == BRK_C128)
          hipLaunchKernelGGL(k_spin<double>, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, s,
                             (const cpx<double>*)first, npairs, lower, qmask, partial);
        else
          hipLaunchKernelGGL(k_spin<float>, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, s, (const cpx<float>*)first,
                             npairs, lower, qmask, partial);
      },
      out);
}

// Per event: target r = u * total, its chunk c = the first with S[c] > r (the running
// sums S over whole chunks, computed on the host left to right), or the last chunk
// holding probability when none is (r at the total), and the running sum before c.
__global__ __launch_bounds__(256) void k_locate_events(const double* __restrict__ S, uint64_t nchunks,
                                                       double total, uint64_t last_chunk,
                                                       const double* __restrict__ canonical, unsigned num_events,
                                                       uint64_t* __restrict__ chunk_of,
                                                       double* __restrict__ chunk_start, double* __restrict__ target) {
  const unsigned e = blockIdx.x * 256 + threadIdx.x;
  if (e >= num_events) return;
  const double r = canonical[e] * total;
  uint64_t lo = 0, hi = nchunks;
  while (lo < hi) {  // upper bound: the first index with S > r
    const uint64_t mid = lo + (hi - lo) / 2;
    if (S[mid] > r) hi = mid;
    else lo = mid + 1;
  }
  const uint64_t c = lo >= nchunks ? last_chunk : lo;
  chunk_of[e] = c;
  chunk_start[e] = c ? S[c - 1] : 0.0;
  target[e] = r;
}

// Running sums over whole chunks for the no-allocation sampling entry point:
// sums[c] becomes S[c] = S[c - 1] + sums[c] (S[-1] = 0), added left to right
// exactly as brk_generate_events adds them on the host, so both give the same
// S bit for bit.  One wavefront: every lane adds the same values in the same
// order (run is uniform), lane l keeps the value after the l-th add of its
// 64-chunk window.  meta[0] = S[nchunks - 1] (the total), meta[1] = the last
// chunk whose sum is positive as an integer (-1: none, a zero-norm state).
__global__ __launch_bounds__(64) void k_running_sums(double* __restrict__ sums, uint64_t nchunks,
                                                     double* __restrict__ meta) {
  const int lane = threadIdx.x;
  double run = 0.0;
  int64_t last = -1;
  for (uint64_t base = 0; base < nchunks; base += 64) {
    const uint64_t c = base + (uint64_t)lane;
    const double v = c < nchunks ? sums[c] : 0.0;
    if (c < nchunks && v > 0.0) last = (int64_t)c;
    double mine = 0.0;
    const uint64_t left = nchunks - base;
    if (left >= 64) {
#pragma unroll
      for (int l = 0; l < 64; ++l) {
        run = run + readlane_f64(v, l);
        if (l == lane) mine = run;
      }
    } else {
      for (int l = 0; l < (int)left; ++l) {
        run = run + readlane_f64(v, l);
        if (l == lane) mine = run;
      }
    }
    if (c < nchunks) sums[c] = mine;
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    const int64_t o = __shfl_xor(last, off, 64);
    last = o > last ? o : last;
  }
  if (lane == 0) {
    meta[0] = run;
    meta[1] = (double)last;
  }
}

// Device scratch of brk_generate_events_noalloc.  Each device holds its own
// copy for the life of the process: the chunk sums (then their running sums)
// of a state of up to NOALLOC_MAX_CHUNKS chunks of SAMPLE_CHUNK amplitudes
// (2^32 amplitudes, 32 qubits in either dtype), per event its draw, chunk,
// chunk start, target and result for up to NOALLOC_MAX_EVENTS events, then
// the two values k_running_sums writes -- 6.5 MiB in all.  Every element a
// call reads is written earlier in the same call, so nothing is cleared.
// Host code never passes `scratch` itself to a kernel or a copy (on the host
// it names a stand-in, not device memory): it uses the per-device address
// noalloc_scratch() obtains from hipGetSymbolAddress.
constexpr uint64_t NOALLOC_MAX_CHUNKS = 1ull << 19;
constexpr unsigned NOALLOC_MAX_EVENTS = 1u << 16;
constexpr uint64_t NOALLOC_DOUBLES = NOALLOC_MAX_CHUNKS + 5ull * NOALLOC_MAX_EVENTS + 2;
static __device__ __align__(256) double scratch[NOALLOC_DOUBLES];

constexpr int NOALLOC_MAX_DEVICES = 64;
// One lock per device, held by a call from its first launch until its events
// are back on the host: calls on one device (from any host thread) take turns.
static std::mutex g_noalloc_busy[NOALLOC_MAX_DEVICES];
static double* g_noalloc_ptr[NOALLOC_MAX_DEVICES];  // written under g_noalloc_busy[device]

// The current device's address of `scratch`, looked up on the device's first
// call (its lock held by the caller).
static int noalloc_scratch(int device, double** out) {
  if (!g_noalloc_ptr[device]) {
    void* p = nullptr;
    const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !p)
      return fail(BRK_ERR_HIP, "hipGetSymbolAddress(scratch) on device %d: %s", device, hipGetErrorString(e));
    g_noalloc_ptr[device] = static_cast<double*>(p);
  }
  *out = g_noalloc_ptr[device];
  return BRK_OK;
}

static_assert(INNER_BLOCKS == RED_BLOCKS, "one grid");
int launch_inner_partials(const void* a, const void* b, uint64_t size, int dtype, double* partials, void* stream) {
  if (dtype == BRK_C128)
    hipLaunchKernelGGL((k_inner<double, double>), dim3(RED_BLOCKS), dim3(RED_THREADS), 0, as_stream(stream),
                       (const cpx<double>*)a, (const cpx<double>*)b, size, partials);
  else
    hipLaunchKernelGGL((k_inner<float, float>), dim3(RED_BLOCKS), dim3(RED_THREADS), 0, as_stream(stream),
                       (const cpx<float>*)a, (const cpx<float>*)b, size, partials);
  return check_launch("inner product");
}

constexpr int ROW_THREADS = 256;

__global__ __launch_bounds__(ROW_THREADS) void k_row_sums(const double* __restrict__ in, uint64_t cols,
                                                          double scale, double* __restrict__ out) {
  __shared__ double part[ROW_THREADS];
  const double* row = in + (uint64_t)blockIdx.x * cols;
  double s = 0.0;
  for (uint64_t c = threadIdx.x; c < cols; c += ROW_THREADS) s += row[c];
  part[threadIdx.x] = s;
  __syncthreads();
  for (int w = ROW_THREADS / 2; w > 0; w >>= 1) {
    if ((int)threadIdx.x < w) part[threadIdx.x] += part[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = scale * part[0];
}

int sum_gradient_partials(const double* partials, unsigned rows, uint64_t chunks, double scale, double* out,
                          void* stream) {
  if (!rows) return BRK_OK;
  if (!partials || !out || !chunks) return fail(BRK_ERR_INVALID_ARGUMENT, "gradient partials: null or empty");
  if (rows > 0x7fffffffu) return fail(BRK_ERR_INVALID_ARGUMENT, "too many gradient rows");
  hipLaunchKernelGGL(k_row_sums, dim3(rows), dim3(ROW_THREADS), 0, as_stream(stream), partials, chunks, scale, out);
  return check_launch("gradient partial sums");
}

static int make_ising_args(unsigned nq, const double* J, const double* h, ising_args* a) {
  if (nq > (unsigned)MAX_CHAIN) return fail(BRK_ERR_TOO_MANY_QUBITS, "Ising chain longer than %d", MAX_CHAIN);
  if (!J || !h) return fail(BRK_ERR_INVALID_ARGUMENT, "J or h is null");
  *a = ising_args{};
  a->n = (int)nq;
  for (unsigned i = 0; i + 1 < nq; ++i) a->J[i] = J[i];
  for (unsigned i = 0; i < nq; ++i) a->h[i] = h[i];
  return BRK_OK;
}

// <H> in passes of k_ising (terms with h = 0 are left out).  A field that is not finite multiplies its
// qubit's whole <X>, after the passes: over parts of the sum it gives 0 * inf and inf - inf.
template <typename R>
static int ising_energy(const void* first, uint64_t size, const ising_args& args, double* result, void* stream) {
  constexpr unsigned L = ising_shape<R>::L, line = sizeof(R) == 8 ? 3 : 4;  // qubits of a 128-byte line
  const unsigned n = (unsigned)args.n;
  const uint64_t nchunks = std::max<uint64_t>(1, size >> L);
  const unsigned grid = (unsigned)std::min<uint64_t>(nchunks, ISING_GRID);
  std::vector<ising_pass> passes;
  for (unsigned next = 0; next == 0 || next < n;) {
    ising_pass p{};
    p.n = args.n;
    p.zz = next == 0;
    std::copy(args.J, args.J + MAX_CHAIN, p.J);
    // the first L qubits, then the line's qubits and the next L - line ones (fewer: filled up with
    // the lowest others)
    const unsigned end = std::min(n, next == 0 ? L : next + (L - line));
    uint64_t local = next == 0 ? 0 : (1ull << line) - 1ull;
    for (unsigned q = next; q < end; ++q) local |= 1ull << q;
    for (unsigned q = 0; (unsigned)__builtin_popcountll(local) < L; ++q) local |= 1ull << q;
    unsigned r = 0;
    for (unsigned q = 0; r < L; ++q) {
      if (!(local >> q & 1ull)) continue;
      p.pos[r] = q;
      if (q >= next && q < end && args.h[q] != 0.0 && std::isfinite(2.0 * args.h[q])) {
        p.measure |= 1u << r;
        p.h2[r] = 2.0 * args.h[q];  // <X_q> = 2 sum Re conj(a0) a1
      }
      ++r;
    }
    if (p.zz || p.measure) passes.push_back(p);
    next = next == 0 ? L : end;
  }
  reduce_scratch* sc;
  if (int st = get_reduce_scratch(&sc)) return st;
  const size_t values = passes.size() * grid;
  if (values > (size_t)RED_BLOCKS * RED_MAX_VALUES) return fail(BRK_ERR_INVALID_ARGUMENT, "too many Ising passes");
  std::unique_lock<std::mutex> hold(sc->busy);
  hipStream_t s = as_stream(stream);
  int status = BRK_OK;
  for (size_t k = 0; !status && k < passes.size(); ++k) {
    hipLaunchKernelGGL(k_ising<R>, dim3(grid), dim3(ISING_THREADS), 0, s, (const cpx<R>*)first, size, nchunks,
                       passes[k], sc->partials + k * grid);
    status = check_launch("Ising energy");
  }
  const hipError_t synced = hipStreamSynchronize(s);
  if (status) return status;
  if (synced != hipSuccess) return fail(BRK_ERR_HIP, "Ising energy: %s", hipGetErrorString(synced));
  double total = 0.0;
  for (size_t k = 0; k < values; ++k) total += sc->partials[k];
  hold.unlock();
  for (unsigned q = 0; q < n; ++q) {
    if (std::isfinite(2.0 * args.h[q])) continue;
    double raw[3];
    if (int st = spin_raw(first, size, sizeof(R) == 8 ? BRK_C128 : BRK_C64, q, raw, stream)) return st;
    total += 2.0 * args.h[q] * raw[0];
  }
  *result = total;
  return BRK_OK;
}

}  // namespace brk

using namespace brk;

extern "C" {

int brk_inner_product(const void* first1, int dtype1, const void* first2, int dtype2, uint64_t size,
                      double result[2], void* stream) {
  unsigned nq;
  if (int st = check_state(first1, size, dtype1, &nq)) return st;
  if (int st = check_state(first2, size, dtype2, &nq)) return st;
  if (!result) return fail(BRK_ERR_INVALID_ARGUMENT, "result is null");
  return run_reduction<2>(
      stream,
      [&](double* partial, hipStream_t s) {
        dim3 g(RED_BLOCKS), b(RED_THREADS);
        if (dtype1 == BRK_C128 && dtype2 == BRK_C128)
          hipLaunchKernelGGL((k_inner<double, double>), g, b, 0, s, (const cpx<double>*)first1,
                             (const cpx<double>*)first2, size, partial);
        else if (dtype1 == BRK_C128)
          hipLaunchKernelGGL((k_inner<double, float>), g, b, 0, s, (const cpx<double>*)first1,
                             (const cpx<float>*)first2, size, partial);
        else if (dtype2 == BRK_C128)
          hipLaunchKernelGGL((k_inner<float, double>), g, b, 0, s, (const cpx<float>*)first1,
                             (const cpx<double>*)first2, size, partial);
        else
          hipLaunchKernelGGL((k_inner<float, float>), g, b, 0, s, (const cpx<float>*)first1,
                             (const cpx<float>*)first2, size, partial);
      },
      result);
}

int brk_fidelity(const void* first1, int dtype1, const void* first2, int dtype2, uint64_t size, double* result,
                 void* stream) {
  if (!result) return fail(BRK_ERR_INVALID_ARGUMENT, "result is null");
  double ip[2];
  if (int st = brk_inner_product(first1, dtype1, first2, dtype2, size, ip, stream)) return st;
  *result = ip[0] * ip[0] + ip[1] * ip[1];
  return BRK_OK;
}

int brk_norm2(const void* first, uint64_t size, int dtype, double* result, void* stream) {
  unsigned nq;
  if (int st = check_state(first, size, dtype, &nq)) return st;
  if (!result) return fail(BRK_ERR_INVALID_ARGUMENT, "result is null");
  return run_reduction<1>(
      stream,
      [&](double* partial, hipStream_t s) {
        if (dtype == BRK_C128)
          hipLaunchKernelGGL(k_norm<double>, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, s, (const cpx<double>*)first,
                             size, partial);
        else
          hipLaunchKernelGGL(k_norm<float>, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, s, (const cpx<float>*)first,
                             size, partial);
      },
      result);
}

int brk_spin_expectation_value(const void* first, uint64_t size, int dtype, unsigned qubit, double result[3],
                               void* stream) {
  unsigned nq;
  if (int st = check_state(first, size, dtype, &nq)) return st;
  if (!result) return fail(BRK_ERR_INVALID_ARGUMENT, "result is null");
  if (qubit >= nq) return fail(BRK_ERR_QUBIT_OUT_OF_RANGE, "qubit %u out of range for %u qubits", qubit, nq);
  double raw[3];
  if (int st = spin_raw(first, size, dtype, qubit, raw, stream)) return st;
  result[0] = raw[0];
  result[1] = raw[1];
  result[2] = raw[2] * 0.5;  // spin_expectation_value.hpp:75-76
  return BRK_OK;
}

int brk_expectation_pauli_string(const void* first, uint64_t size, int dtype, const char* pauli_string,
                                 const unsigned* qubits, unsigned num_qubits, double result[2], void* stream) {
  unsigned nq;
  if (int st = check_state(first, size, dtype, &nq)) return st;
  if (!result || !pauli_string) return fail(BRK_ERR_INVALID_ARGUMENT, "null argument");
  unsigned ops[BRK_MAX_OPERATED_QUBITS];
  unsigned cnt = 0;
  if (int st = collect_qubits(qubits, num_qubits, nq, ops, &cnt, "operated")) return st;
  uint64_t flip = 0, sign = 0;
  unsigned ny = 0;
  for (unsigned k = 0; k < num_qubits; ++k) {
    const char c = pauli_string[k];
    const uint64_t bit = 1ull << qubits[k];
    if (c == 'X') flip |= bit;
    else if (c == 'Y') { flip |= bit; sign |= bit; ++ny; }
    else if (c == 'Z') sign |= bit;
    else if (c != 'I') return fail(BRK_ERR_INVALID_ARGUMENT, "bad Pauli character '%c'", c);
  }
  if (pauli_string[num_qubits] != '\0')
    return fail(BRK_ERR_INVALID_ARGUMENT, "Pauli string length differs from the number of qubits");
  double raw[2];
  int st = run_reduction<2>(
      stream,
      [&](double* partial, hipStream_t s) {
        if (dtype == BRK_C128)
          hipLaunchKernelGGL(k_pauli<double>, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, s, (const cpx<double>*)first,
                             size, flip, sign, partial);
        else
          hipLaunchKernelGGL(k_pauli<float>, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, s, (const cpx<float>*)first,
                             size, flip, sign, partial);
      },
      raw);
  if (st) return st;
  // coefficient (-i)^{#Y} (pauli_index_coeff.hpp:32-59: -i for Y on 0, +i for Y on 1)
  std::complex<double> r{raw[0], raw[1]};
  static const std::complex<double> phases[4] = {{1, 0}, {0, -1}, {-1, 0}, {0, 1}};
  r *= phases[ny & 3u];
  result[0] = r.real();
  result[1] = r.imag();
  return BRK_OK;
}

int brk_expectation_ising(const void* first, uint64_t size, int dtype, const double* J, const double* h,
                          double* result, void* stream) {
  unsigned nq;
  if (int st = check_state(first, size, dtype, &nq)) return st;
  if (!result) return fail(BRK_ERR_INVALID_ARGUMENT, "result is null");
  ising_args a;
  if (int st = make_ising_args(nq, J, h, &a)) return st;
  if (dtype == BRK_C128) return ising_energy<double>(first, size, a, result, stream);
  return ising_energy<float>(first, size, a, result, stream);
}

int brk_apply_ising(void* out, const void* psi, uint64_t size, int dtype, const double* J, const double* h,
                    void* stream) {
  unsigned nq;
  if (int st = check_state(out, size, dtype, &nq)) return st;
  if (int st = check_state(psi, size, dtype, &nq)) return st;
  if (out == psi) return fail(BRK_ERR_INVALID_ARGUMENT, "apply_ising cannot work in place");
  ising_args a;
  if (int st = make_ising_args(nq, J, h, &a)) return st;
  uint64_t blocks = (size + 255) / 256;
  if (blocks > 0x7fffffffull) return fail(BRK_ERR_INVALID_ARGUMENT, "state too large");
  if (dtype == BRK_C128)
    hipLaunchKernelGGL(k_apply_ising<double>, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream),
                       (cpx<double>*)out, (const cpx<double>*)psi, size, a);
  else
    hipLaunchKernelGGL(k_apply_ising<float>, dim3((unsigned)blocks), dim3(256), 0, as_stream(stream),
                       (cpx<float>*)out, (const cpx<float>*)psi, size, a);
  return check_launch("apply_ising");
}

int brk_zero_one_probabilities(const void* first, uint64_t size, int dtype, unsigned qubit, double result[2],
                               void* stream) {
  unsigned nq;
  if (int st = check_state(first, size, dtype, &nq)) return st;
  if (!result) return fail(BRK_ERR_INVALID_ARGUMENT, "result is null");
  if (qubit >= nq) return fail(BRK_ERR_QUBIT_OUT_OF_RANGE, "qubit %u out of range for %u qubits", qubit, nq);
  const uint64_t qmask = 1ull << qubit, lower = qmask - 1ull, npairs = size >> 1;
  return run_reduction<2>(
      stream,
      [&](double* partial, hipStream_t s) {
        if (dtype == BRK_C128)
          hipLaunchKernelGGL(k_zero_one<double>, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, s,
                             (const cpx<double>*)first, npairs, lower, qmask, partial);
        else
          hipLaunchKernelGGL(k_zero_one<float>, dim3(RED_BLOCKS), dim3(RED_THREADS), 0, s,
                             (const cpx<float>*)first, npairs, lower, qmask, partial);
      },
      result);
}

int brk_project_qubit(void* first, uint64_t size, int dtype, unsigned qubit, int value, double multiplier,
                      void* stream) {
  unsigned nq;
  if (int st = check_state(first, size, dtype, &nq)) return st;
  if (qubit >= nq) return fail(BRK_ERR_QUBIT_OUT_OF_RANGE, "qubit %u out of range for %u qubits", qubit, nq);
  if (value != 0 && value != 1) return fail(BRK_ERR_INVALID_ARGUMENT, "value must be 0 or 1");
  const uint64_t qmask = 1ull << qubit, lower = qmask - 1ull, npairs = size >> 1;
  const uint64_t blocks = (npairs + 255) / 256;
  if (blocks > 0xffffffffull) return fail(BRK_ERR_INVALID_ARGUMENT, "state too large");
  const bool nt = size * amp_bytes(dtype) >= get_tuning().nt_min_bytes;
  hipStream_t s = as_stream(stream);
  if (dtype == BRK_C128) {
    if (nt)
      hipLaunchKernelGGL((k_project<double, true>), dim3((unsigned)blocks), dim3(256), 0, s, (cpx<double>*)first,
                         npairs, lower, qmask, value, multiplier);
    else
      hipLaunchKernelGGL((k_project<double, false>), dim3((unsigned)blocks), dim3(256), 0, s, (cpx<double>*)first,
                         npairs, lower, qmask, value, multiplier);
  } else {
    if (nt)
      hipLaunchKernelGGL((k_project<float, true>), dim3((unsigned)blocks), dim3(256), 0, s, (cpx<float>*)first,
                         npairs, lower, qmask, value, (float)multiplier);
    else
      hipLaunchKernelGGL((k_project<float, false>), dim3((unsigned)blocks), dim3(256), 0, s, (cpx<float>*)first,
                         npairs, lower, qmask, value, (float)multiplier);
  }
  return check_launch("project");
}

int brk_generate_events(const void* first, uint64_t size, int dtype, const double* canonical, unsigned num_events,
                        uint64_t* events, void* stream) {
  unsigned nq;
  if (int st = check_state(first, size, dtype, &nq)) return st;
  if (num_events == 0) return BRK_OK;
  if (!canonical || !events) return fail(BRK_ERR_INVALID_ARGUMENT, "null argument");
  const uint32_t chunk = (uint32_t)std::min<uint64_t>(size, SAMPLE_CHUNK);
  const uint64_t nchunks = size / chunk;
  if (nchunks > 0x7fffffffull) return fail(BRK_ERR_INVALID_ARGUMENT, "state too large");
  hipStream_t s = as_stream(stream);
  // device buffers: chunk sums, then their running sums | per event: draw, result | the wave sums
  // of every chunk (1/1024 of a c128 state).  Without room for the wave sums an event searches its
  // whole chunk, as in brk_generate_events_noalloc, and takes three more numbers.
  const size_t event_bytes = (sizeof(uint64_t) * 2 + sizeof(double) * 3) * num_events;
  const size_t bytes = sizeof(double) * nchunks + event_bytes;
  void* buffers = nullptr;
  bool by_wave = hipMalloc(&buffers, bytes + sizeof(double) * SAMPLE_WAVES * nchunks) == hipSuccess;
  if (!by_wave) {
    (void)hipGetLastError();
    BRK_HIP_CHECK(hipMalloc(&buffers, bytes));
  }
  double* d_sums = static_cast<double*>(buffers);
  double* d_canonical = d_sums + nchunks;
  uint64_t* d_chunk = reinterpret_cast<uint64_t*>(d_canonical + num_events);
  double* d_start = reinterpret_cast<double*>(d_chunk + num_events);
  double* d_target = d_start + num_events;
  uint64_t* d_events = reinterpret_cast<uint64_t*>(d_target + num_events);
  double* d_waves = by_wave ? reinterpret_cast<double*>(d_events + num_events) : nullptr;
  if (dtype == BRK_C128)
    hipLaunchKernelGGL(k_chunk_sums<double>, dim3((unsigned)nchunks), dim3(SAMPLE_THREADS), 0, s,
                       (const cpx<double>*)first, chunk, d_sums, d_waves);
  else
    hipLaunchKernelGGL(k_chunk_sums<float>, dim3((unsigned)nchunks), dim3(SAMPLE_THREADS), 0, s,
                       (const cpx<float>*)first, chunk, d_sums, d_waves);
  std::vector<double> sums(nchunks);
  int status = check_launch("chunk sums");
  // (while the sums are formed)
  for (unsigned e = 0; !status && e < num_events; ++e)
    if (!(canonical[e] >= 0.0 && canonical[e] < 1.0))
      status = fail(BRK_ERR_INVALID_ARGUMENT, "canonical[%u] = %g is not in [0, 1)", e, canonical[e]);
  if (!status && (hipMemcpyAsync(sums.data(), d_sums, sizeof(double) * nchunks, hipMemcpyDeviceToHost, s) != hipSuccess ||
                  hipStreamSynchronize(s) != hipSuccess))
    status = fail(BRK_ERR_HIP, "copying the chunk sums failed");
  std::vector<double> S(nchunks);  // running sum through each chunk, left to right
  double run = 0.0;
  for (uint64_t c = 0; c < nchunks; ++c) S[c] = run = run + sums[c];
  uint64_t last_chunk = nchunks;  // the last chunk holding probability
  for (uint64_t c = nchunks; c-- > 0;)
    if (sums[c] > 0.0) {
      last_chunk = c;
      break;
    }
  if (!status && last_chunk == nchunks) status = fail(BRK_ERR_INVALID_ARGUMENT, "the state has zero norm");
  if (!status) {
    // the running sums replace the chunk sums on the device; each event finds its chunk there
    if (hipMemcpyAsync(d_sums, S.data(), sizeof(double) * nchunks, hipMemcpyHostToDevice, s) != hipSuccess ||
        hipMemcpyAsync(d_canonical, canonical, sizeof(double) * num_events, hipMemcpyHostToDevice, s) !=
            hipSuccess)
      status = fail(BRK_ERR_HIP, "uploading the running sums failed");
  }
  if (!status && by_wave) {
    const unsigned per_block = FIND_THREADS / 64;
    const dim3 grid((num_events + per_block - 1) / per_block), block(FIND_THREADS);
    if (dtype == BRK_C128)
      hipLaunchKernelGGL(k_find_events<double>, grid, block, 0, s, (const cpx<double>*)first, chunk, d_sums, nchunks,
                         S[nchunks - 1], last_chunk, d_waves, d_canonical, num_events, d_events);
    else
      hipLaunchKernelGGL(k_find_events<float>, grid, block, 0, s, (const cpx<float>*)first, chunk, d_sums, nchunks,
                         S[nchunks - 1], last_chunk, d_waves, d_canonical, num_events, d_events);
    status = check_launch("find events");
  } else if (!status) {
    hipLaunchKernelGGL(k_locate_events, dim3((num_events + 255) / 256), dim3(256), 0, s, d_sums, nchunks,
                       S[nchunks - 1], last_chunk, d_canonical, num_events, d_chunk, d_start, d_target);
    status = check_launch("locate events");
    if (!status) {
      if (dtype == BRK_C128)
        hipLaunchKernelGGL(k_chunk_search<double>, dim3(num_events), dim3(SAMPLE_THREADS), 0, s,
                           (const cpx<double>*)first, chunk, d_chunk, d_start, d_target, d_events);
      else
        hipLaunchKernelGGL(k_chunk_search<float>, dim3(num_events), dim3(SAMPLE_THREADS), 0, s,
                           (const cpx<float>*)first, chunk, d_chunk, d_start, d_target, d_events);
      status = check_launch("chunk search");
    }
  }
  if (!status && (hipMemcpyAsync(events, d_events, sizeof(uint64_t) * num_events, hipMemcpyDeviceToHost, s) !=
                      hipSuccess ||
                  hipStreamSynchronize(s) != hipSuccess))
    status = fail(BRK_ERR_HIP, "copying the events failed");
  (void)hipStreamSynchronize(s);
  (void)hipFree(buffers);
  return status;
}

int brk_generate_events_noalloc(const void* first, uint64_t size, int dtype, const double* canonical,
                                unsigned num_events, uint64_t* events, void* stream) {
  unsigned nq;
  if (int st = check_state(first, size, dtype, &nq)) return st;
  if (num_events == 0) return BRK_OK;
  if (!canonical || !events) return fail(BRK_ERR_INVALID_ARGUMENT, "null argument");
  for (unsigned e = 0; e < num_events; ++e)
    if (!(canonical[e] >= 0.0 && canonical[e] < 1.0))
      return fail(BRK_ERR_INVALID_ARGUMENT, "canonical[%u] = %g is not in [0, 1)", e, canonical[e]);
  const uint32_t chunk = (uint32_t)std::min<uint64_t>(size, SAMPLE_CHUNK);
  const uint64_t nchunks = size / chunk;
  if (nchunks > NOALLOC_MAX_CHUNKS)
    return fail(BRK_ERR_INVALID_ARGUMENT,
                "brk_generate_events_noalloc takes states of at most %llu amplitudes (%llu given)",
                (unsigned long long)(NOALLOC_MAX_CHUNKS * SAMPLE_CHUNK), (unsigned long long)size);
  if (num_events > NOALLOC_MAX_EVENTS)
    return fail(BRK_ERR_INVALID_ARGUMENT, "brk_generate_events_noalloc takes at most %u events per call (%u given)",
                NOALLOC_MAX_EVENTS, num_events);
  int dev = 0;
  BRK_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= NOALLOC_MAX_DEVICES)
    return fail(BRK_ERR_INVALID_ARGUMENT, "device %d: no-allocation scratch exists for devices 0..%d", dev,
                NOALLOC_MAX_DEVICES - 1);
  std::lock_guard<std::mutex> hold(g_noalloc_busy[dev]);
  double* d_sums = nullptr;
  if (int st = noalloc_scratch(dev, &d_sums)) return st;
  double* d_canonical = d_sums + NOALLOC_MAX_CHUNKS;
  uint64_t* d_chunk = reinterpret_cast<uint64_t*>(d_canonical + NOALLOC_MAX_EVENTS);
  double* d_start = reinterpret_cast<double*>(d_chunk + NOALLOC_MAX_EVENTS);
  double* d_target = d_start + NOALLOC_MAX_EVENTS;
  uint64_t* d_events = reinterpret_cast<uint64_t*>(d_target + NOALLOC_MAX_EVENTS);
  double* d_meta = reinterpret_cast<double*>(d_events + NOALLOC_MAX_EVENTS);
  hipStream_t s = as_stream(stream);
  // every exit after the first launch waits for the stream, so the next call
  // (which takes the lock) never overlaps this call's kernels on the scratch
  auto run = [&]() -> int {
    if (dtype == BRK_C128)
      hipLaunchKernelGGL(k_chunk_sums<double>, dim3((unsigned)nchunks), dim3(SAMPLE_THREADS), 0, s,
                         (const cpx<double>*)first, chunk, d_sums, (double*)nullptr);
    else
      hipLaunchKernelGGL(k_chunk_sums<float>, dim3((unsigned)nchunks), dim3(SAMPLE_THREADS), 0, s,
                         (const cpx<float>*)first, chunk, d_sums, (double*)nullptr);
    if (int st = check_launch("chunk sums")) return st;
    hipLaunchKernelGGL(k_running_sums, dim3(1), dim3(64), 0, s, d_sums, nchunks, d_meta);
    if (int st = check_launch("running sums")) return st;
    double meta[2] = {0.0, -1.0};  // total, last chunk holding probability
    if (hipMemcpyAsync(meta, d_meta, sizeof(meta), hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return fail(BRK_ERR_HIP, "copying the running-sum total failed");
    if (meta[1] < 0.0) return fail(BRK_ERR_INVALID_ARGUMENT, "the state has zero norm");
    if (hipMemcpyAsync(d_canonical, canonical, sizeof(double) * num_events, hipMemcpyHostToDevice, s) !=
        hipSuccess)
      return fail(BRK_ERR_HIP, "uploading the draws failed");
    hipLaunchKernelGGL(k_locate_events, dim3((num_events + 255) / 256), dim3(256), 0, s, d_sums, nchunks, meta[0],
                       (uint64_t)meta[1], d_canonical, num_events, d_chunk, d_start, d_target);
    if (int st = check_launch("locate events")) return st;
    if (dtype == BRK_C128)
      hipLaunchKernelGGL(k_chunk_search<double>, dim3(num_events), dim3(SAMPLE_THREADS), 0, s,
                         (const cpx<double>*)first, chunk, d_chunk, d_start, d_target, d_events);
    else
      hipLaunchKernelGGL(k_chunk_search<float>, dim3(num_events), dim3(SAMPLE_THREADS), 0, s,
                         (const cpx<float>*)first, chunk, d_chunk, d_start, d_target, d_events);
    if (int st = check_launch("chunk search")) return st;
    if (hipMemcpyAsync(events, d_events, sizeof(uint64_t) * num_events, hipMemcpyDeviceToHost, s) != hipSuccess ||
        hipStreamSynchronize(s) != hipSuccess)
      return fail(BRK_ERR_HIP, "copying the events failed");
    return BRK_OK;
  };
  const int status = run();
  (void)hipStreamSynchronize(s);
  return status;
}

}  // extern "C"
