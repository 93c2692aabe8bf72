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

// Calls fill(lo, hi) for every gap's rows [lo, hi) that is not empty.
template <typename F>
__device__ inline void for_gaps(const Args& a, F&& fill) {
  const int total = a.total_rows;
  auto gap = [&](int lo, int hi) {
    if (lo < hi) fill(lo, hi);
  };
  if (!a.seq_lens) {
    auto row = [&](int x) { return x < 0 ? 0 : (x > total ? total : x); };
    const int lo = row(a.cu_seqlens[0]);
    gap(0, lo);
    gap(max(lo, row(a.cu_seqlens[a.B])), total);
    return;
  }
  int end = 0;  // of the sequences so far
  for (int b = 0; b < a.B; ++b) {
    const int lo = a.cu_seqlens[b];
    gap(end, lo < total ? lo : total);
    const int s = lo < 0 ? 0 : (lo > total ? total : lo), n = a.seq_lens[b];
    const int e = n < total - s ? s + (n < 0 ? 0 : n) : total;
    end = e > end ? e : end;
  }
  gap(end, total);
}

// One thread's share of the (row, head, 16-byte piece) units of a gap in a tensor of `heads` heads of BYTES
// bytes: piece `c` of rows of a head, the head fastest.  Set up once per tensor; the loop over the units
// then divides nothing, and is bound by the stores.  4 x 4096 rows in a buffer of 65536 (Hq = 64, Hkv = 8, D = 64,
// window 128), in us, with a division and a modulo per store and 64 workgroups / with those and a launch of its own /
// now: forward 358 / 273 / 167 (96 without the unused rows, whose 403 MB take 71 at 5.7 TB/s), backward 527 / 462
// ... 502 / 354 ... 381 (264).
template <int BYTES>
struct GapUnits {
  static constexpr int P = BYTES / 16;
  int heads, c, row0, head0, drow, dhead;
  __device__ __forceinline__ GapUnits(const Args& a, int wg, int heads) : heads(heads) {
    const int t = wg * int(blockDim.x) + int(threadIdx.x), u = t / P, du = a.tail_wgs * int(blockDim.x) / P;
    c = t % P;
    row0 = u / heads;
    head0 = u % heads;
    drow = du / heads;
    dhead = du % heads;
  }
  // zeros in rows [lo, hi) of the tensor at `ptr` with strides `st` in elements of EB bytes
  template <int EB>
  __device__ __forceinline__ void zero(void* ptr, const int64_t (&st)[3], int lo, int hi) const {
    char* p = static_cast<char*>(ptr) + 16 * c;
    int h = head0;
    for (int64_t r = int64_t(lo) + row0; r < hi;) {
      *reinterpret_cast<uint4*>(p + (h * st[1] + r * st[2]) * EB) = uint4{0u, 0u, 0u, 0u};
      r += drow;
      h += dhead;
      if (h >= heads) {
        h -= heads;
        ++r;
      }
    }
  }
};

// The forward's extra workgroups (`wg`: the workgroup's id); EB bytes per element of o.
template <int D, int EB>
__device__ inline void fwd_aux(const Args& a, unsigned wg) {
  const int x = int(wg - a.main_wgs);
  const GapUnits<D * EB> o(a, x, a.Hq);
  const int first = x * int(blockDim.x) + int(threadIdx.x), step = a.tail_wgs * int(blockDim.x);
  for_gaps(a, [&](int lo, int hi) {
    o.template zero<EB>(a.o_out, a.so_out, lo, hi);
    for (int64_t r = lo + int64_t(first); r < hi; r += step)  // (rows fastest: lse is [head][row])
      for (int h = 0; h < a.Hq; ++h) a.lse_out[h * a.slse[1] + r * a.slse[2]] = -__builtin_inff();
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
  const GapUnits<D * EB> q(a, x, a.Hq), kv(a, x, a.Hkv);
  for_gaps(a, [&](int lo, int hi) {
    q.template zero<EB>(a.dq, a.sdq, lo, hi);
    kv.template zero<EB>(a.dk, a.sdk, lo, hi);
    kv.template zero<EB>(a.dv, a.sdv, lo, hi);
  });
}

// Host: workgroups behind a kernel's own `main`, 256 for the rows of no sequence: with 64 the case above takes
// 199 and 388 us, and a batch that covers every row, where they only read two offsets, is no faster (0.3%, less
// than two runs differ).  (a.main_wgs and a.tail_wgs are set): all of the launch's.
inline int64_t wgs_with_aux(Args& a, int64_t main, bool bwd) {
  a.main_wgs = unsigned(main);
  a.tail_wgs = a.cu_seqlens ? 256 : 0;
  return main + a.tail_wgs + (bwd && a.dsink ? a.Hq : 0);
}
inline unsigned grid_with_aux(Args& a, int64_t main, bool bwd) { return unsigned(wgs_with_aux(a, main, bwd)); }

}  // namespace fa
