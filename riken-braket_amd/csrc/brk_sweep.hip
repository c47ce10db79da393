// Kernel of the adjoint gradient's sweeps (brk_sweep.hpp).
#include "brk_internal.hpp"
#include "brk_sweep.hpp"

#include <type_traits>

namespace brk {
namespace {

typedef const __attribute__((address_space(4))) char* cbytes;
typedef const __attribute__((address_space(4))) sweep_header* cheader;
typedef const __attribute__((address_space(4))) sweep_segment* csegment;
typedef const __attribute__((address_space(4))) sweep_macro* cmacro;

constexpr int GROUP = 1 << SWEEP_GROUP;

__device__ __forceinline__ float mad(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double mad(double a, double b, double c) { return __builtin_fma(a, b, c); }

// LDS slot of local index j: an XOR swizzle, so that groups over low bits spread over all banks.
__device__ __forceinline__ uint32_t sweep_slot(uint32_t j) { return j ^ ((j >> 3) & 7u) ^ ((j >> 6) & 7u); }

// The sums of v[0..7] over the wave's rows of 16 lanes, in a fixed order.  The first two steps also
// halve the number of values a lane holds: lane l of a row ends with the row's sums of values
// 4 (l & 1) + (l & 2) + {0, 1}.
__device__ __forceinline__ void row_sums(const double (&v)[8], uint32_t lane, double (&out)[2]) {
  const bool one = (lane & 1u) != 0, two = (lane & 2u) != 0;
  double r[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const double keep = one ? v[k + 4] : v[k], send = one ? v[k] : v[k + 4];
    r[k] = keep + dpp_f64<0xB1>(send);  // quad_perm [1, 0, 3, 2]
  }
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const double keep = two ? r[k + 2] : r[k], send = two ? r[k] : r[k + 2];
    double s = keep + dpp_f64<0x4E>(send);  // quad_perm [2, 3, 0, 1]
    s += dpp_f64<0x124>(s);                 // row_ror 4
    s += dpp_f64<0x128>(s);                 // row_ror 8
    out[k] = s;
  }
}

// The sign bits (bit 31) of the group's members by the macro's terms.  Member m's index is xb | xe:
// the thread's bits and the member's are disjoint, so a term's bit count is, mod 2, the thread's own
// count, plus that of xe & M with M = ((xb & A) << d) ^ ((xb >> d) & A), plus a count over xe alone
// (`uniform`, or in the phase table).
__device__ __forceinline__ void member_signs(cmacro mac, uint32_t xb, const uint32_t (&q)[SWEEP_GROUP],
                                             uint32_t (&sign)[GROUP]) {
  const uint32_t n = mac->num_terms;
  uint32_t own = 0, M = 0;
#pragma unroll
  for (uint32_t k = 0; k < (uint32_t)SWEEP_MAX_TERMS; ++k) {
    if (k >= n) break;
    const uint32_t d = mac->d[k], A = mac->A[k];
    own += __popc(xb & (xb >> d) & A);
    M ^= ((xb & A) << d) ^ ((xb >> d) & A);
  }
  sign[0] = own << 31;
#pragma unroll
  for (int b = 0; b < SWEEP_GROUP; ++b) {
    const uint32_t mb = (M >> q[b]) << 31;
#pragma unroll
    for (int m = 0; m < (1 << b); ++m) sign[m | 1 << b] = sign[m] ^ mb;
  }
}

template <typename R>
__device__ __forceinline__ cpx<R> times(cpx<R> a, cpx<R> k) {
  return {mad(a.re, k.re, -(a.im * k.im)), mad(a.re, k.im, a.im * k.re)};
}

// [[m00, m01], [m10, m11]] on the pairs of group bit B.
template <int B, typename R>
__device__ __forceinline__ void mix_pairs(cpx<R> (&x)[GROUP], uint32_t kind,
                                          const __attribute__((address_space(4))) double* u) {
  if (kind == SWEEP_MIX_REAL) {
    const R m00 = (R)u[0], m01 = (R)u[2], m10 = (R)u[4], m11 = (R)u[6];
#pragma unroll
    for (int m = 0; m < GROUP; ++m) {
      if (m & (1 << B)) continue;
      const cpx<R> a = x[m], b = x[m | 1 << B];
      x[m] = {mad(m01, b.re, m00 * a.re), mad(m01, b.im, m00 * a.im)};
      x[m | 1 << B] = {mad(m11, b.re, m10 * a.re), mad(m11, b.im, m10 * a.im)};
    }
  } else if (kind == SWEEP_MIX_X) {
    const R m00 = (R)u[0], m01 = (R)u[3], m10 = (R)u[5], m11 = (R)u[6];
#pragma unroll
    for (int m = 0; m < GROUP; ++m) {
      if (m & (1 << B)) continue;
      const cpx<R> a = x[m], b = x[m | 1 << B];
      x[m] = {mad(-m01, b.im, m00 * a.re), mad(m01, b.re, m00 * a.im)};
      x[m | 1 << B] = {mad(-m10, a.im, m11 * b.re), mad(m10, a.re, m11 * b.im)};
    }
  } else {
    const cpx<R> m00 = {(R)u[0], (R)u[1]}, m01 = {(R)u[2], (R)u[3]}, m10 = {(R)u[4], (R)u[5]}, m11 = {(R)u[6], (R)u[7]};
#pragma unroll
    for (int m = 0; m < GROUP; ++m) {
      if (m & (1 << B)) continue;
      const cpx<R> a = x[m], b = x[m | 1 << B];
      const cpx<R> p = times(a, m00), r = times(a, m10);
      x[m] = {mad(b.re, m01.re, mad(-b.im, m01.im, p.re)), mad(b.re, m01.im, mad(b.im, m01.re, p.im))};
      x[m | 1 << B] = {mad(b.re, m11.re, mad(-b.im, m11.im, r.re)), mad(b.re, m11.im, mad(b.im, m11.re, r.im))};
    }
  }
}

// The mixing gate of group bit B: its gradient term, then the gate.
//   Y form, D = [[0, a], [b, 0]]:      a Re(conj(l0) p1) + b Re(conj(l1) p0);
//   X form, D = [[0, i a], [i b, 0]]: -a Im(conj(l0) p1) - b Im(conj(l1) p0).
template <int B, typename R, bool BOTH>
__device__ __forceinline__ void mix(cpx<R> (&x)[GROUP], cpx<R> (&y)[GROUP], cmacro mac, double (&value)[8]) {
  const uint32_t kind = mac->mix[B];
  if (kind == SWEEP_MIX_NONE) return;
  if constexpr (BOTH) {
    const uint32_t form = mac->form[B];
    if (form != SWEEP_FORM_NONE) {
      double s0 = 0.0, s1 = 0.0;
      if (form == SWEEP_FORM_Y) {
#pragma unroll
        for (int m = 0; m < GROUP; ++m) {
          if (m & (1 << B)) continue;
          const cpx<R> p0 = x[m], p1 = x[m | 1 << B], l0 = y[m], l1 = y[m | 1 << B];
          s0 = mad((double)l0.re, (double)p1.re, s0);
          s0 = mad((double)l0.im, (double)p1.im, s0);
          s1 = mad((double)l1.re, (double)p0.re, s1);
          s1 = mad((double)l1.im, (double)p0.im, s1);
        }
      } else {
#pragma unroll
        for (int m = 0; m < GROUP; ++m) {
          if (m & (1 << B)) continue;
          const cpx<R> p0 = x[m], p1 = x[m | 1 << B], l0 = y[m], l1 = y[m | 1 << B];
          s0 = mad((double)l0.im, (double)p1.re, s0);
          s0 = mad(-(double)l0.re, (double)p1.im, s0);
          s1 = mad((double)l1.im, (double)p0.re, s1);
          s1 = mad(-(double)l1.re, (double)p0.im, s1);
        }
      }
      value[SWEEP_GROUP + B] = mac->mix_weight[B][0] * s0 + mac->mix_weight[B][1] * s1;
    }
  }
  mix_pairs<B>(x, kind, mac->matrix[B]);
  if constexpr (BOTH) mix_pairs<B>(y, kind, mac->matrix[B]);
}

// The macro's signs and phases: the gradient terms of the group's phases from
// t_m = -Im(conj(l_m) p_m), a product every phase of the macro shares (and a common sign leaves as it
// is), then the signed table, or the signs alone.
template <typename R, bool BOTH>
__device__ __forceinline__ void apply_diagonal(cpx<R> (&x)[GROUP], cpx<R> (&y)[GROUP], cmacro mac, uint32_t xb,
                                               const uint32_t (&q)[SWEEP_GROUP], double (&value)[8]) {
  if constexpr (BOTH) {
    if (mac->phase_grads) {
      double t[GROUP];
#pragma unroll
      for (int m = 0; m < GROUP; ++m)
        t[m] = mad((double)y[m].im, (double)x[m].re, -((double)y[m].re * (double)x[m].im));
      // sums over the members with group bit b clear and set
      const double a0 = t[0] + t[1], a1 = t[2] + t[3], a2 = t[4] + t[5], a3 = t[6] + t[7];
      const double even = (t[0] + t[2]) + (t[4] + t[6]), odd = (t[1] + t[3]) + (t[5] + t[7]);
      value[0] = mac->weight[0][0] * even + mac->weight[0][1] * odd;
      value[1] = mac->weight[1][0] * (a0 + a2) + mac->weight[1][1] * (a1 + a3);
      value[2] = mac->weight[2][0] * (a0 + a1) + mac->weight[2][1] * (a2 + a3);
    }
  }
  if (mac->num_terms == 0) {
    if (mac->phases == 0) return;
#pragma unroll
    for (int m = 0; m < GROUP; ++m) {
      const cpx<R> k = {(R)mac->phase[m][0], (R)mac->phase[m][1]};
      x[m] = times(x[m], k);
      if constexpr (BOTH) y[m] = times(y[m], k);
    }
    return;
  }
  uint32_t sign[GROUP];
  member_signs(mac, xb, q, sign);
  if (mac->phases) {
#pragma unroll
    for (int m = 0; m < GROUP; ++m) {
      const cpx<R> k = cflip(cpx<R>{(R)mac->phase[m][0], (R)mac->phase[m][1]}, sign[m]);
      x[m] = times(x[m], k);
      if constexpr (BOTH) y[m] = times(y[m], k);
    }
  } else {
    const uint32_t uniform = mac->uniform;
#pragma unroll
    for (int m = 0; m < GROUP; ++m) {
      const uint32_t s = sign[m] ^ (((uniform >> m) & 1u) << 31);
      x[m] = cflip(x[m], s);
      if constexpr (BOTH) y[m] = cflip(y[m], s);
    }
  }
}

// Bound: FP64 instructions (VALU 57 % busy in the reverse sweep, 66 % forward).  24 qubits, 12 layers
// of RY, RZ and CZ, c128: 8 reverse blocks of 0.80 ms and 8 forward blocks of 0.33 ms, against 21 of
// 0.60 ms and 17 of 0.40 ms gate by gate; 9.5 against 20.1 ms per gradient.  Fetching the next
// macro's lines ahead: 15 qubits 55 -> 38 us a reverse block (few chunks: latency), 24 qubits no change.
// One workgroup of 2^(L - 3) threads per chunk.  Two workgroups per CU (64 KiB of LDS each, plus the
// gradient sums).  The gradient terms of a segment's macros are summed over rows of 16 lanes in
// registers, kept per row in LDS (two sets in turn) and added up by a few threads after the
// segment's barrier, while the workgroup goes on.
template <typename R, int L, bool BOTH, bool NT>
__global__ __launch_bounds__(1 << (L - SWEEP_GROUP), L - SWEEP_GROUP > 8 ? 4 : 2)
void k_sweep(cpx<R>* __restrict__ psi, cpx<R>* __restrict__ lam, const void* program, double* __restrict__ partials) {
  constexpr int TB = L - SWEEP_GROUP, THREADS = 1 << TB, ROWS = THREADS / 16;
  __shared__ cpx<R> lp[1 << L], ll[BOTH ? 1 << L : 1];
  __shared__ double sums[BOTH ? 2 : 1][BOTH ? SWEEP_MAX_MACROS : 1][8][ROWS];
  const cbytes prog = (cbytes)program;
  const cheader h = (cheader)prog;
  const csegment segments = (csegment)(prog + sizeof(sweep_header));
  const cmacro macros = (cmacro)(prog + h->macros_at);
  const uint32_t t = threadIdx.x;
  const uint32_t chunk_number = (uint32_t)xcd_chunk(blockIdx.x, gridDim.x);
  uint32_t chunk = chunk_number;  // (amplitude indices are 32-bit: SWEEP_MAX_QUBITS)
#pragma unroll
  for (int r = 0; r < L; ++r) {
    const uint32_t q = h->pos[r], below = (1u << q) - 1u;
    chunk = ((chunk & ~below) << 1) | (chunk & below);
  }
  auto offset = [&](uint32_t j) {
    uint32_t o = 0;
#pragma unroll
    for (int r = 0; r < L; ++r) o |= ((j >> r) & 1u) << h->pos[r];
    return o;
  };
  // Brings a macro's lines into the scalar cache while another one runs: its fields are read in turn
  // between branches, and the programs of the chunks in flight do not fit in that cache.
  uint32_t seen = 0;
  auto fetch = [&](uint32_t i) {
    const auto* words = (const __attribute__((address_space(4))) uint32_t*)(macros + min(i, h->num_macros - 1));
#pragma unroll
    for (uint32_t k = 0; k < sizeof(sweep_macro) / 4; k += 16) seen |= words[k];
  };
  fetch(0);
  const uint32_t num_segments = h->num_segments;
  if (!(segments[0].flags & SWEEP_LOADS)) {
    const uint32_t low = chunk | offset(t);
#pragma unroll
    for (int k = 0; k < GROUP; ++k) {
      const uint32_t i = low | offset((uint32_t)k << TB);
      lp[sweep_slot(t + THREADS * k)] = load_amp<NT>(psi + i);
      if constexpr (BOTH) ll[sweep_slot(t + THREADS * k)] = load_amp<NT>(lam + i);
    }
    __syncthreads();
  }
  uint32_t first_macro = 0;  // of the segment (counted: with a number to load 24 qubits took 9.54 ms, now 9.49)
  for (uint32_t si = 0; si < num_segments; ++si) {
    const csegment seg = segments + si;
    const uint32_t flags = seg->flags, num_macros = seg->num_macros;
    const cmacro first = macros + first_macro;
    uint32_t base = t, dep[GROUP], q[SWEEP_GROUP];
    dep[0] = 0;
#pragma unroll
    for (int b = 0; b < SWEEP_GROUP; ++b) {
      const uint32_t p = seg->group[b];
      q[b] = seg->qubits[b];
      base = ((base >> p) << (p + 1)) | (base & ((1u << p) - 1u));
#pragma unroll
      for (int m = 0; m < (1 << b); ++m) dep[m | 1 << b] = dep[m] | 1u << p;
    }
    const uint32_t low = chunk | offset(base);
    uint32_t high[GROUP];
    high[0] = 0;
#pragma unroll
    for (int b = 0; b < SWEEP_GROUP; ++b)
#pragma unroll
      for (int m = 0; m < (1 << b); ++m) high[m | 1 << b] = high[m] | 1u << q[b];
    cpx<R> x[GROUP], y[GROUP];
    const uint32_t slot = sweep_slot(base);  // (the swizzle is linear)
    if (flags & SWEEP_LOADS) {
#pragma unroll
      for (int m = 0; m < GROUP; ++m) {
        x[m] = load_amp<NT>(psi + (low | high[m]));
        if constexpr (BOTH) y[m] = load_amp<NT>(lam + (low | high[m]));
      }
    } else {
#pragma unroll
      for (int m = 0; m < GROUP; ++m) {
        x[m] = lp[slot ^ sweep_slot(dep[m])];
        if constexpr (BOTH) y[m] = ll[slot ^ sweep_slot(dep[m])];
      }
    }
    for (uint32_t mi = 0; mi < num_macros; ++mi) {
      const cmacro mac = first + mi;
      fetch(first_macro + mi + 1);
      double value[8] = {};
      apply_diagonal<R, BOTH>(x, y, mac, low, q, value);
      mix<0, R, BOTH>(x, y, mac, value);
      mix<1, R, BOTH>(x, y, mac, value);
      mix<2, R, BOTH>(x, y, mac, value);
      if constexpr (BOTH) {
        if (mac->any_grads) {
          double r[2];
          row_sums(value, t & 63u, r);
          if ((t & 12u) == 0) {
            const uint32_t v = 4 * (t & 1u) + (t & 2u);
            sums[si & 1u][mi][v][t >> 4] = r[0];
            sums[si & 1u][mi][v + 1][t >> 4] = r[1];
          }
        }
      }
    }
    if (flags & SWEEP_STORES) {
#pragma unroll
      for (int m = 0; m < GROUP; ++m) {
        store_amp<NT>(psi + (low | high[m]), x[m]);
        if constexpr (BOTH) store_amp<NT>(lam + (low | high[m]), y[m]);
      }
    } else {
#pragma unroll
      for (int m = 0; m < GROUP; ++m) {
        lp[slot ^ sweep_slot(dep[m])] = x[m];
        if constexpr (BOTH) ll[slot ^ sweep_slot(dep[m])] = y[m];
      }
    }
    __syncthreads();
    if constexpr (BOTH) {
      // thread v + 8 mi: value v of macro mi
      if (t < 8 * num_macros && (t & 7u) < (uint32_t)SWEEP_VALUES) {
        const uint32_t v = t & 7u, mi = t >> 3;
        const int32_t param = first[mi].slot[v];
        if (param >= 0) {
          double sum = 0.0;
#pragma unroll
          for (int r = 0; r < ROWS; ++r) sum += sums[si & 1u][mi][v][r];
          partials[(uint64_t)param * gridDim.x + blockIdx.x] = sum;
        }
      }
    }
    first_macro += num_macros;
    if (seen == 1u) __builtin_amdgcn_s_sleep(0);  // (keeps the fetches)
    if (flags & SWEEP_STORES) return;
  }
  const uint32_t low = chunk | offset(t);
#pragma unroll
  for (int k = 0; k < GROUP; ++k) {
    const uint32_t i = low | offset((uint32_t)k << TB);
    store_amp<NT>(psi + i, lp[sweep_slot(t + THREADS * k)]);
    if constexpr (BOTH) store_amp<NT>(lam + i, ll[sweep_slot(t + THREADS * k)]);
  }
}

}  // namespace

int launch_sweep(const void* device_program, unsigned num_local, void* psi, void* lam, uint64_t size, int dtype,
                 double* partials, void* stream) {
  unsigned nq;
  if (int st = check_state(psi, size, dtype, &nq)) return st;
  const unsigned want = !lam ? SWEEP_FORWARD_LOCAL
                        : dtype == BRK_C128 ? SWEEP_REVERSE_LOCAL_C128 : SWEEP_REVERSE_LOCAL_C64;
  if (num_local != want || num_local > nq || nq > (unsigned)SWEEP_MAX_QUBITS)
    return fail(BRK_ERR_INVALID_ARGUMENT, "sweep block does not fit (%u local of %u qubits)", num_local, nq);
  const dim3 grid((unsigned)(size >> num_local)), block(1u << (num_local - SWEEP_GROUP));
  hipStream_t st = as_stream(stream);
  const bool nt = size * amp_bytes(dtype) >= get_tuning().nt_min_bytes;
  auto launch = [&](auto* p, auto* l, auto reverse_local) {
    using R = decltype(p->re);
    constexpr int REVERSE = decltype(reverse_local)::value, FORWARD = SWEEP_FORWARD_LOCAL;
    if (l && nt) hipLaunchKernelGGL((k_sweep<R, REVERSE, true, true>), grid, block, 0, st, p, l, device_program, partials);
    else if (l) hipLaunchKernelGGL((k_sweep<R, REVERSE, true, false>), grid, block, 0, st, p, l, device_program, partials);
    else if (nt) hipLaunchKernelGGL((k_sweep<R, FORWARD, false, true>), grid, block, 0, st, p, l, device_program, partials);
    else hipLaunchKernelGGL((k_sweep<R, FORWARD, false, false>), grid, block, 0, st, p, l, device_program, partials);
  };
  if (dtype == BRK_C128)
    launch((cpx<double>*)psi, (cpx<double>*)lam, std::integral_constant<int, SWEEP_REVERSE_LOCAL_C128>());
  else
    launch((cpx<float>*)psi, (cpx<float>*)lam, std::integral_constant<int, SWEEP_REVERSE_LOCAL_C64>());
  return check_launch("sweep");
}

}  // namespace brk
