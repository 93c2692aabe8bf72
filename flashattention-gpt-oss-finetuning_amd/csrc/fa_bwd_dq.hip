// fa_bwd_dq.hip - dQ with one tile per workgroup (16-bit inputs, no sink rows in the dQ kernel): the
// backward twin of fwd_split_kernel (fa_fwd.hip).
//
// A workgroup is 4 = wq x wh x KSP waves on one tile of 32 wq query rows x wh query heads of a KV group: wave
// (qi, hi, g) takes 32 rows of one head and every KSP-th 32-key half (half KSP s + g in step s).  Per half
// S^T = K Q^T and dP^T - delta = V dO^T - delta, P and dS elementwise, dQ^T += K^T dS^T, the mathematics of
// bwd_dq_kernel; the KSP waves' dQ are added in LDS at the end, each wave writing out a part.  delta =
// rowsum(dO o O) and the row statistics for the dK/dV kernel come from the rows in registers.  The
// tiles with the most keys are dispatched first, an XCD owns whole (batch, head set)s where their
// number allows (q_stream), and K/V halves are double-buffered in LDS by DMA, one step ahead.
//
// What it buys over bwd_dq_kernel (resident workgroups walking tiles, 64-key blocks, the next tile's rows
// stashed in LDS): 16 KB of LDS and 142 VGPRs at D = 64, three workgroups per CU instead of two, 32 KB and
// 220 at D = 128, two instead of one, and tiles of any length spread evenly.  In us, bf16, KSP = 1 / 2 / 4
// (bwd_dq_kernel): D = 64, Hq = 64, Hkv = 8, full causal L = 512 15.3 / 13.0 / 17.5 (15.2); L = 1024 27.5 /
// 25.6 / 38 (30.1); L = 4096 208 / 231 / 310 (218); L = 8192 764 / 859 / 1106 (825); Hq = 8, Hkv = 1,
// L = 2048 40 / 27 / 20 (38); D = 128, Hq = 32, Hkv = 8, L = 2048 76 / 68 (69), L = 8192 745 / 834 (836);
// B = 8, Hq = 32, Hkv = 4, L = 2048, W = 512 268 / 333 (305).  KSP = 1 gives bwd_dq_kernel's bits.
#include "fa_args.h"
#include "fa_common.h"

namespace fa {

// ROWS: more than one row tile per workgroup (wq > 1), whose waves skip halves outside their own rows.
template <typename E, int D, int KSP, bool ROWS>
__global__ __launch_bounds__(256, D == 128 || KSP == 4 ? 2 : 3) void bwd_dq_split_kernel(const Args a) {
  constexpr int KS = D / 16;
  constexpr int DB = D >= 32 ? D / 32 : 1;
  constexpr int TILE = 32 * D;              // a K or V half, swizzled row-major [key][d]
  constexpr int STAGE = KSP * 2 * TILE;     // the halves of a step: K, V of each
  constexpr int RING = 2 * STAGE;           // 16-bit units
  // dQ C tiles that a wave hands over in the merge: all but its own (db % KSP == g)
  constexpr int NM = DB < KSP ? DB : (DB / KSP) * (KSP - 1);
  constexpr int MERGE = KSP > 1 ? 4 * NM * 16 * 64 * 2 : 0;
  constexpr int CPR = D / 8;                // 16-byte chunks per K or V row
  __shared__ __attribute__((aligned(16))) uint16_t lds[RING > MERGE ? RING : MERGE];
  const int lane = threadIdx.x & 63, r32 = lane & 31, hf = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wq = ROWS ? a.wq : 1, wh = a.wh;
  const int qi = ROWS ? wave % wq : 0, hi = wave / wq % wh, g = KSP == 1 ? 0 : wave / (wq * wh);
  const int W = a.W, S = a.S;

  const int gpk = a.G / wh;
  const QStream qs = q_stream(int(a.wg_base + blockIdx.x), a.B * a.Hkv * gpk, a.cu_seqlens != nullptr);
  const int kvh = qs.stream / gpk / a.B, b = qs.stream / gpk % a.B;
  const int hw = kvh * a.G + qs.stream % gpk * wh + hi;
  const Seq sq = seq_of(a, b);
  const int L = sq.L, q0 = 32 * wq * (a.n_qtiles - 1 - qs.pos), qw = q0 + 32 * qi, q = qw + r32;
  if (q0 >= L) return;
  const Plan32 pl = plan32(q0, 32 * wq, L, W, S);
  const int nh = pl.nsink + (pl.we - pl.ws), n_steps = (nh + KSP - 1) / KSP;

  const rsrc_t rk = make_rsrc(reinterpret_cast<const char*>(a.k) + 2 * slice_off(a.sk, b, kvh, sq.row), span_bytes(L, a.sk[2], D));
  const rsrc_t rv = make_rsrc(reinterpret_cast<const char*>(a.v) + 2 * slice_off(a.sv, b, kvh, sq.row), span_bytes(L, a.sv[2], D));
  const uint32_t bk = uint32_t(2 * a.sk[2]), bv = uint32_t(2 * a.sv[2]);
  // DMA instructions of a step: D / 8 of 1 KiB per half (K, then V), shared out over the waves
  constexpr int NI = KSP * D / 8, NIW = (NI + 3) / 4;
  auto issue = [&](int step) {
    uint16_t* stage = lds + (step & 1) * STAGE;
#pragma unroll
    for (int n = 0; n < NIW; ++n) {
      const int ii = wave * NIW + n, half = ii / (D / 8), i = ii % (D / 8);
      const int is_v = i >= D / 16, p = is_v ? i - D / 16 : i;
      if (ii >= NI || step * KSP + half >= nh) continue;
      const int pos = 64 * p + lane, row = pos / CPR, col = (pos % CPR) ^ swz<D>(row);
      const int key = 32 * plan32_tile(pl, step * KSP + half) + row;
      uint16_t* dst = stage + (2 * half + is_v) * TILE + 512 * p;
      const uint32_t off = uint32_t(int64_t(key) * (is_v ? bv : bk)) + 16u * uint32_t(col);
      if (is_v) buf_dma16(rv, dst, off);
      else buf_dma16(rk, dst, off);
    }
  };
  if (n_steps > 0) issue(0);

  // the wave's rows: Q and dO operands, delta, the row statistics
  u32x4 qf[KS], dof[KS];
  float dsum = 0.f;
  {
    const rsrc_t rq = make_rsrc(reinterpret_cast<const char*>(a.q) + 2 * slice_off(a.sq, b, hw, sq.row), span_bytes(L, a.sq[2], D));
    const rsrc_t rd = make_rsrc(reinterpret_cast<const char*>(a.dout) + 2 * slice_off(a.sdo, b, hw, sq.row), span_bytes(L, a.sdo[2], D));
    const rsrc_t ro = make_rsrc(reinterpret_cast<const char*>(a.o) + 2 * slice_off(a.so, b, hw, sq.row), span_bytes(L, a.so[2], D));
    u32x4 of[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int col = hf * (D / 2) + 8 * ks;
      qf[ks] = buf_ld16(rq, uint32_t((int64_t(q) * a.sq[2] + col) * 2)) ^ a.qsign;
      dof[ks] = buf_ld16(rd, uint32_t((int64_t(q) * a.sdo[2] + col) * 2));
      of[ks] = buf_ld16(ro, uint32_t((int64_t(q) * a.so[2] + col) * 2));
    }
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) dsum = dot8<E>(dof[ks], of[ks], dsum);
  }
  const rsrc_t rl = make_rsrc(a.lse + slice_off(a.slse, b, hw, sq.row), span_f32(L, a.slse[2]));
  const float lse = buf_ldf(rl, uint32_t(int64_t(q) * a.slse[2] * 4));
  const float delta = sum_halves(dsum), ndelta = -delta;
  const float lse2 = q < L ? lse * kLog2e : __builtin_inff();
  if (g == 0 && qw < L) {
    const int64_t blk = (int64_t(b) * a.Hq + hw) * (a.Lp / 32) + qw / 32;
    if (hf == 0) {  // (rows past L: +inf and 0, so that their P and dS in the dK/dV kernel are exactly 0)
      float* st = a.delta + blk * 64;
      st[r32] = lse2;
      st[32 + r32] = ndelta;
    }
    if (a.sink_logits) {  // the learned sink's gradient, one partial per 32-row block (see bwd_dq_kernel)
      float v = q < L ? fast_exp2(a.sink_logits[hw] * kLog2e - lse2) * delta : 0.f;
#pragma unroll
      for (int m = 16; m >= 1; m >>= 1) v += __shfl_xor(v, m);
      if (lane == 0) a.dsink_part[blk] = -v;
    }
  }

  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = f32x16{};
  wait_vm_lgkm0_barrier<0>();
  for (int s = 0; s < n_steps; ++s) {
    if (s + 1 < n_steps) issue(s + 1);  // (into the stage that step s - 1 read, before the barrier)
    const int i = s * KSP + g;
    const int ks0 = i < nh ? 32 * plan32_tile(pl, i) : 0;
    if (i < nh && (!ROWS || (qw < L && wave_needs(ks0, qw, L, W, S)))) {
      const uint16_t* Kl = lds + (s & 1) * STAGE + 2 * g * TILE;
      const uint16_t* Vl = Kl + TILE;
      // masked halves start S^T from an additive bias, 0 or -inf: register e holds key ks0 + 4 hf + off(e),
      // allowed = (dq0 - off) < lim (see half_scores in fa_fwd.hip)
      f32x16 sc, dp;
      auto products = [&](const f32x16& c0) {
        f32x16 d0;
#pragma unroll
        for (int e = 0; e < 16; ++e) d0[e] = ndelta;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
          const int off = swz_off<D>(r32, hf * (D / 2) + 8 * ks);
          sc = E::mfma(lds16(Kl + off), qf[ks], ks == 0 ? c0 : sc);
          dp = E::mfma(lds16(Vl + off), dof[ks], ks == 0 ? d0 : dp);
        }
      };
      if (tile_full(ks0, qw, W, S)) {
        products(f32x16{});
      } else {
        f32x16 bias;
        const int dq0 = q - ks0 - 4 * hf;
        const int sl = S - ks0 - 4 * hf;  // keys with off < sl are sinks
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          const int off = 8 * (e / 4) + (e % 4);
          bias[e] = unsigned(dq0 - off) < (off < sl ? 0x80000000u : unsigned(W)) ? 0.f : kNegInf;
        }
        products(bias);
      }
      if constexpr (D == 64) __builtin_amdgcn_s_setprio(1);  // (as bwd_dq_kernel)
      float ds[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) ds[e] = fast_exp2(fmaf(sc[e], a.c, -lse2)) * dp[e];
      const u32x4 d0 = pack8<E>(ds), d1 = pack8<E>(ds + 8);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        acc[db] = E::mfma(tr_frag_swz<D>(Kl, 0, 32 * db, D), d0, acc[db]);
        acc[db] = E::mfma(tr_frag_swz<D>(Kl, 16, 32 * db, D), d1, acc[db]);
      }
      if constexpr (D == 64) __builtin_amdgcn_s_setprio(0);
    }
    wait_vm_lgkm0_barrier<0>();
  }

  if constexpr (KSP > 1) {  // dQ C tile db of a head's KSP waves is added up by wave db % KSP
    float* mo = reinterpret_cast<float*>(lds);  // [wave][C tile handed over][register quad][lane] x 4
    auto slot = [](int c, int from) { return DB < KSP ? c : c / KSP * (KSP - 1) + (c % KSP - from - 1 + KSP) % KSP; };
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      if (db % KSP == g) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(mo + (((wave * NM + slot(db, g)) * 4 + j) * 64 + lane) * 4) =
            f32x4{acc[db][4 * j], acc[db][4 * j + 1], acc[db][4 * j + 2], acc[db][4 * j + 3]};
    }
    __syncthreads();
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      if (db % KSP != g) continue;
#pragma unroll
      for (int gg = 0; gg < KSP; ++gg) {
        if (gg == g) continue;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const f32x4 x = *reinterpret_cast<const f32x4*>(mo + ((((gg * wh + hi) * wq + qi) * NM + slot(db, gg)) * 4 + j) * 256 + 4 * lane);
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[db][4 * j + e] += x[e];
        }
      }
    }
  }
  if (q >= L) return;
  char* dqp = reinterpret_cast<char*>(a.dq) + 2 * slice_off(a.sdq, b, hw, sq.row + q);
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    if (db % KSP != g || (D == 16 && hf == 1)) continue;
    float v[16];
#pragma unroll
    for (int e = 0; e < 16; ++e) v[e] = acc[db][e] * a.scale;
    const int d0 = 32 * db + (D >= 32 ? 16 * hf : 0);
    st16(dqp + 2 * d0, pack8<E>(v));
    st16(dqp + 2 * (d0 + 8), pack8<E>(v + 8));
  }
}

template <typename E, int D, int KSP>
static hipError_t dq_split_k(const Args& a, hipStream_t stream) {
  Args x = a;
  return launch_in_ranges(x, int64_t(a.n_qtiles) * a.B * (a.Hq / a.wh), [&](dim3 grid) {
    if constexpr (KSP < 4) {
      if (a.wq > 1) {
        hipLaunchKernelGGL((bwd_dq_split_kernel<E, D, KSP, true>), grid, dim3(256), 0, stream, x);
        return;
      }
    }
    hipLaunchKernelGGL((bwd_dq_split_kernel<E, D, KSP, false>), grid, dim3(256), 0, stream, x);
  });
}

template <typename E, int D>
static hipError_t dq_split_d(const Args& a, int ksp, hipStream_t stream) {
  if (ksp == 1) return dq_split_k<E, D, 1>(a, stream);
  if (ksp == 2) return dq_split_k<E, D, 2>(a, stream);
  if constexpr (D < 128)
    if (ksp == 4) return dq_split_k<E, D, 4>(a, stream);
  return hipErrorInvalidValue;
}

template <typename E>
static hipError_t dq_split_e(const Args& a, int D, int ksp, hipStream_t stream) {
  switch (D) {
    case 16: return dq_split_d<E, 16>(a, ksp, stream);
    case 32: return dq_split_d<E, 32>(a, ksp, stream);
    case 64: return dq_split_d<E, 64>(a, ksp, stream);
    case 128: return dq_split_d<E, 128>(a, ksp, stream);
  }
  return hipErrorInvalidValue;
}

hipError_t launch_bwd_dq_split(const Args& a, int dtype, int D, int ksp, hipStream_t stream) {
  return dtype == 1 ? dq_split_e<BF16>(a, D, ksp, stream) : dq_split_e<F16>(a, D, ksp, stream);
}

}  // namespace fa
