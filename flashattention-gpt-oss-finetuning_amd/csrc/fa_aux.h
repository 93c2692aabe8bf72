// fa_aux.h - small work that rides on an attention kernel's launch, as workgroups after its own.
//
// Two pieces of work are too small for a launch of their own (4-6 us each, of a 70-100 us step):
//  * the gradient of the learned sink logits, the sum of the dQ kernel's partials: on the dK/dV kernel;
//  * packed rows that belong to no sequence (before the first one, after the last one and, with
//    seq_lens, between them), which no attention workgroup writes: o = 0 and lse = -inf on the
//    forward, zero dq, dk and dv on the dK/dV kernel.
// A kernel's own workgroups are [0, a.main_wgs); the ones behind them are dispatched last and run
// beside its tail.
#pragma once

#include "fa_args.h"

namespace fa {

// dsink[h] = sum over (b, 32-row block) of the partials of head h, in a fixed order (each of 256 threads
// strides over the partials in order, then the waves' sums are combined in wave order), so reruns are
// bitwise identical.  `smem`: four floats of LDS.
__device__ inline void sum_sink_logits(const Args& a, int h, float* smem) {
  const int tid = threadIdx.x;
  const int nb = a.Lp / 32;
  const int64_t n = int64_t(a.B) * nb;
  float acc = 0.f;
  if (tid < 256) {
    for (int64_t i = tid; i < n; i += 256) {
      const int64_t b = i / nb, j = i % nb;
      // row blocks past the end of a short sequence hold no partial
      if (32 * j < seq_of(a, int(b)).L) acc += a.dsink_part[(b * a.Hq + h) * nb + j];
    }
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) acc += __shfl_xor(acc, m);
    if ((tid & 63) == 0) smem[tid >> 6] = acc;
  }
  __syncthreads();
  if (tid == 0) a.dsink[h] = (smem[0] + smem[1]) + (smem[2] + smem[3]);
}

// Workgroup `wg` of a.tail_wgs: calls fill(lo, hi, first, step) for every gap's rows [lo, hi), where this
// thread takes the pieces first, first + step, ... of the gap.
template <typename F>
__device__ inline void for_gaps(const Args& a, int wg, F&& fill) {
  const int64_t first = int64_t(wg) * blockDim.x + threadIdx.x, step = int64_t(a.tail_wgs) * blockDim.x;
  const int total = a.total_rows;
  if (!a.seq_lens) {
    auto row = [&](int x) { return x < 0 ? 0 : (x > total ? total : x); };
    const int lo = row(a.cu_seqlens[0]);
    fill(0, lo, first, step);
    fill(max(lo, row(a.cu_seqlens[a.B])), total, first, step);
    return;
  }
  int end = 0;  // of the sequences so far
  for (int b = 0; b < a.B; ++b) {
    const int lo = a.cu_seqlens[b];
    fill(end, lo < total ? lo : total, first, step);
    const int s = lo < 0 ? 0 : (lo > total ? total : lo), n = a.seq_lens[b];
    const int e = n < total - s ? s + (n < 0 ? 0 : n) : total;
    end = e > end ? e : end;
  }
  fill(end, total, first, step);
}

// Rows [lo, hi) of a tensor of `heads` heads whose rows are `bytes` bytes (a multiple of 16): zeros.
__device__ inline void zero_rows(void* ptr, const int64_t (&st)[3], int heads, int bytes, int eb, int lo, int hi,
                                 int64_t first, int64_t step) {
  const int pieces = bytes / 16;
  const int64_t n = int64_t(hi - lo) * heads * pieces;
  for (int64_t u = first; u < n; u += step) {
    const int c = int(u % pieces), h = int(u / pieces % heads);
    const int64_t r = lo + u / pieces / heads;
    char* p = static_cast<char*>(ptr) + (h * st[1] + r * st[2]) * eb + 16 * c;
    *reinterpret_cast<uint4*>(p) = uint4{0u, 0u, 0u, 0u};
  }
}

// The forward's extra workgroups (`wg`: the workgroup's id); EB bytes per element of o.
template <int D, int EB>
__device__ inline void fwd_aux(const Args& a, unsigned wg) {
  for_gaps(a, int(wg - a.main_wgs), [&](int lo, int hi, int64_t first, int64_t step) {
    if (lo >= hi) return;
    zero_rows(a.o_out, a.so_out, a.Hq, D * EB, EB, lo, hi, first, step);
    for (int64_t u = first; u < int64_t(hi - lo) * a.Hq; u += step)
      a.lse_out[int64_t(u % a.Hq) * a.slse[1] + (lo + u / a.Hq) * a.slse[2]] = -__builtin_inff();
  });
}

// The dK/dV kernel's: a workgroup per head for the learned sinks (when a.dsink), then a.tail_wgs.
template <int D, int EB>
__device__ inline void bwd_aux(const Args& a, unsigned wg, float* smem) {
  int x = int(wg - a.main_wgs);
  if (a.dsink) {
    if (x < a.Hq) return sum_sink_logits(a, x, smem);
    x -= a.Hq;
  }
  for_gaps(a, x, [&](int lo, int hi, int64_t first, int64_t step) {
    if (lo >= hi) return;
    zero_rows(a.dq, a.sdq, a.Hq, D * EB, EB, lo, hi, first, step);
    zero_rows(a.dk, a.sdk, a.Hkv, D * EB, EB, lo, hi, first, step);
    zero_rows(a.dv, a.sdv, a.Hkv, D * EB, EB, lo, hi, first, step);
  });
}

// Host: workgroups behind a kernel's own `main` (a.main_wgs and a.tail_wgs are set): all of the launch's.
// Without seq_lens a packed batch usually covers every row, and its workgroups only read two offsets.
inline int64_t wgs_with_aux(Args& a, int64_t main, bool bwd) {
  a.main_wgs = unsigned(main);
  a.tail_wgs = !a.cu_seqlens ? 0 : a.seq_lens ? 256 : 64;
  return main + a.tail_wgs + (bwd && a.dsink ? a.Hq : 0);
}
inline unsigned grid_with_aux(Args& a, int64_t main, bool bwd) { return unsigned(wgs_with_aux(a, main, bwd)); }

}  // namespace fa
