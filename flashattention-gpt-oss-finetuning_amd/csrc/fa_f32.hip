// fa_f32.hip - float32 inputs: forward and backward on the fp32 matrix instruction.
//
// The reference's autograd Function takes float32 q/k/v as well as 16-bit ones
// (flash_attention_gpt_oss.py:356-357: o = empty_like(q); benchmark_backward_speed.py:28-37:
// dtype "fp32").  These kernels compute that case in float32 throughout: every product runs on
// v_mfma_f32_32x32x2_f32 (exact fp32 products, fp32 sums), P and dS stay fp32, and q, k, v, o,
// dq, dk, dv are fp32 tensors.  The mathematics, masks, visit order of key tiles, workspace row
// statistics and the sink-key partial sums follow the 16-bit kernels (fa_fwd.hip, fa_bwd.hip).
//
// The instruction: a wave64 multiplies a 32x2 A tile by a 2x32 B tile into a 32x32 fp32 C tile;
// lane l (r = l % 32, h = l / 32) supplies A[r][h] and B[h][r] and holds C[crow(i, h)][r] for
// i = 0..15, crow(i, h) = 8 (i / 4) + 4 h + i % 4 -- the C layout of the 32x32x16 16-bit form.
// Two consequences, as in the 16-bit kernels:
//  * a product over a head dim of D runs as D / 2 instructions; in step t lane half h supplies
//    head-dim index h D / 2 + t, so each lane reads one contiguous half row;
//  * a C tile feeds the next product as its B operand unchanged: in step t the reduction index
//    of lane half h is crow(t, h), which is register t of every lane.
//
// What bounds them: the instruction takes 64 cycles for 4096 operations (157 TFLOP/s over the
// chip), so a 32x32 tile at D = 64 is 64 (forward), 96 (dQ) or 128 (dK/dV) of them, 4096-8192 cycles
// against a few hundred for its elementwise work: the matrix cores, once a wave's operands are at hand.
// So the tiles that the waves of a workgroup share (K and V, or a query head's Q and dO) come by
// LDS DMA, one tile ahead, and every operand is read from LDS, where it costs a small share of
// the matrix time; the waves' own rows stay in registers.  Against one wave per workgroup with
// operands straight from memory, in us (B = 1, Hq = 64, Hkv = 8, D = 64): L = 4096, W = 128, S = 4
// forward 240 -> 133, dQ 338 -> 205, dK/dV 1119 -> 253; L = 2048 full causal 1007 -> 334,
// 1390 -> 489, 4862 -> 633 (109 TFLOP/s of allowed pairs).
//
// The head-dim order of a product whose A rows are head-dim indices (O^T, dQ^T, dV^T, dK^T) is free:
// A row m of its C tile db (DB = D / 32 of them) stands for index DB m + db, so a lane reads the DB
// operands of one tile row with one LDS read of DB consecutive floats, and holds 4 DB
// consecutive outputs per four registers.
#include "fa_args.h"
#include "fa_aux.h"
#include "fa_common.h"

namespace fa {

namespace {

__device__ __forceinline__ f32x16 mfma32(float a, float b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ f32x4 mfma16(float x, float y, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(x, y, c, 0, 0, 0);
}
__device__ __forceinline__ int crow(int i, int h) { return 8 * (i >> 2) + 4 * h + (i & 3); }
__device__ __forceinline__ f32x4 ld4f(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ void st4f(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ float other_half(float x) { return __shfl_xor(x, 32); }

// 32-column C tiles of a head dim
template <int D>
constexpr int kDB = D >= 32 ? D / 32 : 1;

__device__ __forceinline__ bool allowed32(int q, int k, int W, int S) { return k <= q && (q - k < W || k < S); }

// One fp32 half row (D / 2 values starting at column h D / 2) of row `row` of a [rows][stride]
// slice, times `mul`; zeros for rows past L.
template <int D>
__device__ __forceinline__ void load_half_row(const float* base, int64_t stride, int row, int L, int h, float mul,
                                              float (&out)[D / 2]) {
  const float* p = base + int64_t(row) * stride + h * (D / 2);
#pragma unroll
  for (int u = 0; u < D / 8; ++u) {
    const f32x4 x = row < L ? ld4f(p + 4 * u) : f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) out[4 * u + j] = x[j] * mul;
  }
}

// ---- [32][D] fp32 tiles in LDS ------------------------------------------------------------------
// Row-major without padding; 16-byte chunk j of row r is stored at chunk j ^ swz32(r), so that the
// same chunk of 8 consecutive rows (a half-row read) lies in 8 different bank groups and a row
// read across lanes still covers whole rows.
template <int D>
__device__ __forceinline__ int swz32(int r) {
  return D >= 32 ? r & 7 : (r >> 1) & 3;
}
// chunk u of lane (r, h)'s half row: columns h D / 2 + 4u .. + 3 of row r
template <int D>
__device__ __forceinline__ f32x4 tile_half(const float* t, int r, int h, int u) {
  return ld4f(t + r * D + 4 * ((h * (D / 8) + u) ^ swz32<D>(r)));
}
// columns DB c .. DB c + DB - 1 of row r (D = 16 has 16 columns: lanes past them repeat the others)
template <int D>
__device__ __forceinline__ void tile_cols(const float* t, int r, int c, float (&out)[kDB<D>]) {
  const int col = D >= 32 ? kDB<D> * c : c & 15;
  const float* p = t + r * D + 4 * ((col >> 2) ^ swz32<D>(r)) + (col & 3);
  if constexpr (kDB<D> == 4) {
    const f32x4 x = ld4f(p);
#pragma unroll
    for (int db = 0; db < 4; ++db) out[db] = x[db];
  } else if constexpr (kDB<D> == 2) {
    const f32x2 x = *reinterpret_cast<const f32x2*>(p);
    out[0] = x[0];
    out[1] = x[1];
  } else {
    out[0] = *p;
  }
}
// DMA instruction p (of D / 8: 1 KiB each) of the tile at rows [row0, row0 + 32) of a slice: lane l
// loads the chunk that the swizzle places at 16-byte position 64 p + l; rows past the slice read as 0
template <int D>
__device__ __forceinline__ void dma_tile(rsrc_t rs, float* tile, int row0, int64_t stride, int p) {
  const int pos = 64 * p + int(threadIdx.x & 63), row = pos / (D / 4), chunk = (pos % (D / 4)) ^ swz32<D>(row);
  buf_dma16(rs, reinterpret_cast<uint16_t*>(tile + 256 * p), uint32_t((int64_t(row0 + row) * stride + 4 * chunk) * 4));
}
__device__ __forceinline__ rsrc_t slice_rsrc(const float* base, int L, int64_t stride, int D) {
  return make_rsrc(base, span_bytes(L, stride, D, 4));
}

// Stores a 32-row output: this lane's row at `row`, C tiles acc (A row m of tile db = column DB m +
// db) times mul.
template <int D>
__device__ __forceinline__ void store_cols(float* row, const f32x16 (&acc)[kDB<D>], int h, float mul) {
  constexpr int DB = kDB<D>;
#pragma unroll
  for (int j = 0; j < (D >= 32 ? 4 : 2); ++j) {
    float v[4 * DB];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int db = 0; db < DB; ++db) v[DB * i + db] = acc[db][4 * j + i] * mul;
#pragma unroll
    for (int x = 0; x < DB; ++x)
      st4f(row + DB * (8 * j + 4 * h) + 4 * x, f32x4{v[4 * x], v[4 * x + 1], v[4 * x + 2], v[4 * x + 3]});
  }
}

// Workgroup -> rows and heads of the query-major kernels: wq x wh waves of 32 rows x 1 head of one KV
// group (see q_stream).
struct QTile {
  int b, kvh, hq, q0, qw;
};
__device__ __forceinline__ QTile q_tile(const Args& a, unsigned wg) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int gpk = a.G / a.wh;  // head groups per KV head
  const QStream s = q_stream(int(wg), a.B * a.Hkv * gpk, a.cu_seqlens != nullptr);
  QTile t;
  t.kvh = s.stream / gpk / a.B;
  t.b = s.stream / gpk % a.B;
  t.hq = t.kvh * a.G + s.stream % gpk * a.wh + wave / a.wq;
  t.q0 = (a.n_qtiles - 1 - s.pos) * 32 * a.wq;
  t.qw = t.q0 + 32 * (wave % a.wq);
  return t;
}

// The K and V tiles of a query-major workgroup: two LDS buffers of [K, V] tiles, wave w issuing DMA
// instructions [w D / 16, (w + 1) D / 16) of the D / 4.
template <int D>
struct KvTiles {
  static constexpr int kTile = 32 * D, kBuf = 2 * kTile;
  rsrc_t rk, rv;
  int64_t sk, sv;
  float* lds;
  __device__ __forceinline__ void load(int buf, int ks0) const {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
    for (int n = 0; n < D / 16; ++n) {
      const int i = wave * (D / 16) + n;
      if (i < D / 8) dma_tile<D>(rk, lds + buf * kBuf, ks0, sk, i);
      else dma_tile<D>(rv, lds + buf * kBuf + kTile, ks0, sv, i - D / 8);
    }
  }
};

// ---------------------------------------------------------------------------------------------
// Forward: O = softmax(mask(s)) V with s = scale q.k, online softmax in the log2 domain (q is
// pre-multiplied by scale * log2(e)).
// ---------------------------------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256, 2) void fwd32_kernel(const Args a) {
  constexpr int HD = D / 2;
  constexpr int DB = kDB<D>;
  __shared__ __attribute__((aligned(16))) float lds[2 * KvTiles<D>::kBuf];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const unsigned wg = a.wg_base + blockIdx.x;
  if (wg >= a.main_wgs) return fwd_aux<D, 4>(a, wg);
  const QTile t = q_tile(a, wg);
  const Seq sq = seq_of(a, t.b);
  const int L = sq.L, W = a.W, S = a.S, hq = t.hq, b = t.b, qw = t.qw;
  if (t.q0 >= L) return;
  const float* Q = static_cast<const float*>(a.q) + slice_off(a.sq, b, hq, sq.row);
  const float* K = static_cast<const float*>(a.k) + slice_off(a.sk, b, t.kvh, sq.row);
  const float* V = static_cast<const float*>(a.v) + slice_off(a.sv, b, t.kvh, sq.row);
  const KvTiles<D> kv{slice_rsrc(K, L, a.sk[2], D), slice_rsrc(V, L, a.sv[2], D), a.sk[2], a.sv[2], lds};
  const Plan32 pl = plan32(t.q0, 32 * a.wq, L, W, S);
  const int nt = pl.nsink + (pl.we - pl.ws);
  if (nt > 0) kv.load(0, 32 * plan32_tile(pl, 0));
  const int q = qw + r;
  float qf[HD];
  load_half_row<D>(Q, a.sq[2], q, L, h, a.scale * kLog2e, qf);

  float m = kNegInf, lsum = 0.f;
  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = f32x16{};
  wait_vm_lgkm0_barrier<0>();
  for (int it = 0; it < nt; ++it) {
    // the other buffer was last read before the barrier that ended the tile before
    if (it + 1 < nt) kv.load((it + 1) & 1, 32 * plan32_tile(pl, it + 1));
    const int ks0 = 32 * plan32_tile(pl, it);
    if (qw < L && wave_needs(ks0, qw, L, W, S)) {
      const float* Kt = lds + (it & 1) * KvTiles<D>::kBuf;
      const float* Vt = Kt + KvTiles<D>::kTile;
      // S^T = K Q^T (keys x queries): lane (r, h) supplies K[ks0 + r][h HD + t]
      f32x16 s = f32x16{};
#pragma unroll
      for (int u = 0; u < D / 8; ++u) {
        const f32x4 kf = tile_half<D>(Kt, r, h, u);
#pragma unroll
        for (int j = 0; j < 4; ++j) s = mfma32(kf[j], qf[4 * u + j], s);
      }
      if (!tile_full(ks0, qw, W, S)) {
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = allowed32(q, ks0 + crow(i, h), W, S) ? s[i] : kNegInf;
      }
      float mx = s[0];
#pragma unroll
      for (int i = 1; i < 16; ++i) mx = fmaxf(mx, s[i]);
      mx = max_halves(mx);
      if (wave_any(mx > m)) {  // some row's maximum moves (otherwise the factor is 1)
        const float mnew = fmaxf(m, mx);
        const float alpha = mnew == kNegInf ? 1.f : exp2f(m - mnew);
        m = mnew;
        lsum *= alpha;
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] *= alpha;
      }
      const float ms = m == kNegInf ? 0.f : m;
      float p[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        p[i] = exp2f(s[i] - ms);
        lsum += p[i];
      }
      // O^T += V^T P^T: lane (r, h) supplies V[ks0 + crow(t, h)][DB r + db]
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float va[DB];
        tile_cols<D>(Vt, crow(i, h), r, va);
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] = mfma32(va[db], p[i], acc[db]);
      }
    }
    wait_vm_lgkm0_barrier<0>();
  }
  float lt = lsum + other_half(lsum);
  float rs = 1.f;
  if (a.sink_logits) {  // the learned sink joins the denominator (as in fwd_kernel's epilogue)
    const float sl = a.sink_logits[hq] * kLog2e;
    const float mn = fmaxf(m, sl);
    rs = m == kNegInf ? 0.f : exp2f(m - mn);
    lt = lt * rs + exp2f(sl - mn);
    m = mn;
  }
  if (q >= L) return;
  const float inv = lt > 0.f ? rs / lt : 0.f;
  store_cols<D>(static_cast<float*>(a.o_out) + slice_off(a.so_out, b, hq, sq.row + q), acc, h, inv);
  if (h == 0) a.lse_out[slice_off(a.slse, b, hq, sq.row + q)] = (m + log2f(lt)) * kLn2;
}

// ---------------------------------------------------------------------------------------------
// dQ: delta = rowsum(dO o O), P = exp2(s - lse2), dS = P (dP - delta), dQ = scale dS K.  Also
// stores the row statistics the dK/dV kernel reads (lse * log2(e), -delta per 32-row block, the
// layout of the 16-bit backward) and, with learned sinks, the per-block partials of their
// gradient.
// ---------------------------------------------------------------------------------------------
template <int D>
__global__ __launch_bounds__(256, D == 128 ? 1 : 2) void dq32_kernel(const Args a) {
  constexpr int HD = D / 2;
  constexpr int DB = kDB<D>;
  __shared__ __attribute__((aligned(16))) float lds[2 * KvTiles<D>::kBuf];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const QTile t = q_tile(a, a.wg_base + blockIdx.x);
  const Seq sq = seq_of(a, t.b);
  const int L = sq.L, W = a.W, S = a.S, hq = t.hq, b = t.b, qw = t.qw;
  if (t.q0 >= L) return;
  const float* Q = static_cast<const float*>(a.q) + slice_off(a.sq, b, hq, sq.row);
  const float* K = static_cast<const float*>(a.k) + slice_off(a.sk, b, t.kvh, sq.row);
  const float* V = static_cast<const float*>(a.v) + slice_off(a.sv, b, t.kvh, sq.row);
  const float* O = static_cast<const float*>(a.o) + slice_off(a.so, b, hq, sq.row);
  const float* dO = static_cast<const float*>(a.dout) + slice_off(a.sdo, b, hq, sq.row);
  const KvTiles<D> kv{slice_rsrc(K, L, a.sk[2], D), slice_rsrc(V, L, a.sv[2], D), a.sk[2], a.sv[2], lds};
  const Plan32 pl = plan32(t.q0, 32 * a.wq, L, W, S);
  const int nt = pl.nsink + (pl.we - pl.ws);
  if (nt > 0) kv.load(0, 32 * plan32_tile(pl, 0));
  const int q = qw + r;
  float qf[HD], dof[HD];
  load_half_row<D>(Q, a.sq[2], q, L, h, a.scale * kLog2e, qf);
  load_half_row<D>(dO, a.sdo[2], q, L, h, 1.f, dof);
  float dsum = 0.f;
  {
    float of[HD];
    load_half_row<D>(O, a.so[2], q, L, h, 1.f, of);
#pragma unroll
    for (int i = 0; i < HD; ++i) dsum = fmaf(dof[i], of[i], dsum);
  }
  const float delta = dsum + other_half(dsum);
  const float lse2 = q < L ? a.lse[slice_off(a.slse, b, hq, sq.row + q)] * kLog2e : __builtin_inff();
  if (qw < L) {
    const int64_t blk = (int64_t(b) * a.Hq + hq) * (a.Lp / 32) + qw / 32;
    if (h == 0) {
      float* st = a.delta + blk * 64;
      st[r] = lse2;
      st[32 + r] = -delta;
    }
    if (a.sink_logits) {
      float v = (q < L && h == 0) ? exp2f(a.sink_logits[hq] * kLog2e - lse2) * delta : 0.f;
#pragma unroll
      for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
      if (lane == 0) a.dsink_part[blk] = -v;
    }
  }

  f32x16 acc[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) acc[db] = f32x16{};
  wait_vm_lgkm0_barrier<0>();
  for (int it = 0; it < nt; ++it) {
    if (it + 1 < nt) kv.load((it + 1) & 1, 32 * plan32_tile(pl, it + 1));
    const int ks0 = 32 * plan32_tile(pl, it);
    if (qw < L && wave_needs(ks0, qw, L, W, S)) {
      const float* Kt = lds + (it & 1) * KvTiles<D>::kBuf;
      const float* Vt = Kt + KvTiles<D>::kTile;
      // S^T = K Q^T and dP^T - delta = V dO^T - delta (keys x queries)
      f32x16 s = f32x16{}, dp;
#pragma unroll
      for (int i = 0; i < 16; ++i) dp[i] = -delta;
#pragma unroll
      for (int u = 0; u < D / 8; ++u) {
        const f32x4 kf = tile_half<D>(Kt, r, h, u), vf = tile_half<D>(Vt, r, h, u);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          s = mfma32(kf[j], qf[4 * u + j], s);
          dp = mfma32(vf[j], dof[4 * u + j], dp);
        }
      }
      const bool full = tile_full(ks0, qw, W, S);
      float ds[16];
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float p = exp2f(s[i] - lse2);
        if (!full) p = allowed32(q, ks0 + crow(i, h), W, S) ? p : 0.f;
        ds[i] = p * dp[i];
      }
      // dQ^T += K^T dS^T: lane (r, h) supplies K[ks0 + crow(t, h)][DB r + db]
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        float ka[DB];
        tile_cols<D>(Kt, crow(i, h), r, ka);
#pragma unroll
        for (int db = 0; db < DB; ++db) acc[db] = mfma32(ka[db], ds[i], acc[db]);
      }
    }
    wait_vm_lgkm0_barrier<0>();
  }
  if (q >= L) return;
  store_cols<D>(static_cast<float*>(a.dq) + slice_off(a.sdq, b, hq, sq.row + q), acc, h, a.scale);
}

// ---------------------------------------------------------------------------------------------
// dK / dV: a workgroup owns 64 keys of one KV head; wave (kh, hh) owns the 32-key half kh and takes
// item 2s + hh of step s, an item being a (query head, 32-row block) that can see the keys: dV^T +=
// dO^T P, dK^T += Q^T dS (keys as the C columns).  A step's two items (Q and dO tiles and row
// statistics) are staged in LDS by DMA, one step ahead.  As in bwd_dkdv_kernel, a key block's steps
// can be cut into kv_split pieces, one workgroup each, and the rows past the window of a block with
// sink keys (block < nsp) go to chunk workgroups of chunk_rows rows; those and the block's own
// workgroup write fp32 sums of its sink rows, [slot][dK, dV][S][D] per (batch, KV head), slot c for
// chunk c and n_chunks for the block's own rows, and fold32_kernel adds them.
// With at most 32 sink keys the chunk workgroups are sink_chunk32's.
// ---------------------------------------------------------------------------------------------
template <int D>
constexpr int kDkdv32Slot = 2 * 32 * D + 64;  // floats of an item: Q tile, dO tile, lse2[32], -delta[32]

// Staging of the dK/dV kernel: wave w loads tile w of a step (item slot w / 2, Q or dO) and slot w % 2's
// statistics (waves w and w + 2 the same bytes to the same place).
template <int D>
struct ItemStage {
  static constexpr int SLOT = kDkdv32Slot<D>;
  const float *tensor, *stats;
  int64_t t_rs, t_hs;
  float* lds;
  int L, nblk, qb_lo, n_qb, n_items;
  __device__ __forceinline__ ItemStage(const Args& a, const Seq& sq, int b, int kvh, int qb_lo, int n_qb, int n_items, float* lds)
      : lds(lds), L(sq.L), nblk(a.Lp / 32), qb_lo(qb_lo), n_qb(n_qb), n_items(n_items) {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t_do = wave & 1;
    t_rs = t_do ? a.sdo[2] : a.sq[2];
    t_hs = t_do ? a.sdo[1] : a.sq[1];
    tensor = t_do ? static_cast<const float*>(a.dout) + slice_off(a.sdo, b, kvh * a.G, sq.row)
                  : static_cast<const float*>(a.q) + slice_off(a.sq, b, kvh * a.G, sq.row);
    stats = a.delta + (int64_t(b) * a.Hq + int64_t(kvh) * a.G) * nblk * 64;
  }
  __device__ __forceinline__ void operator()(int step) const {
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), t_slot = wave >> 1, t_do = wave & 1;
    float* st = lds + (step & 1) * 2 * SLOT;
    const int i = min(2 * step + t_slot, n_items - 1);  // (past the last item: loaded, not used)
    const int g = i / n_qb, row0 = 32 * (qb_lo + i % n_qb);
    const rsrc_t rs = slice_rsrc(tensor + g * t_hs, L, t_rs, D);
#pragma unroll
    for (int p = 0; p < D / 8; ++p) dma_tile<D>(rs, st + t_slot * SLOT + t_do * 32 * D, row0, t_rs, p);
    const int i2 = min(2 * step + (wave & 1), n_items - 1);
    const int blk = i2 / n_qb * nblk + qb_lo + i2 % n_qb;
    buf_dma4(make_rsrc(stats + int64_t(blk) * 64, 256), reinterpret_cast<uint16_t*>(st + (wave & 1) * SLOT + 64 * D),
             4u * (threadIdx.x & 63));
  }
};

// A chunk's rows against all of at most 16 KB sink keys (KB = 1, 2), by 16x16x4 products: the wave's
// matrix time is that of the keys there are, and no product is computed twice, where the 32x32x2 products
// below work for 64 keys.  Wave (kh, hh) takes rows 16 kh .. + 15 of item hh; lane (m, g) = (lane % 16,
// lane / 16) supplies row or key m and the head dims of 16-byte chunk 2 u + g % 2 of half row g / 2
// to the S and dP products, holds P and dS of keys 16 x + m at rows 4 g + e, and supplies columns NT m + t
// of those rows to dV^T += dO^T P, dK^T += Q^T dS.  Whole dK/dV, before (32x32x2 products of one 32-key
// half, S and dP computed by two waves) -> now, us: Hq = 64, Hkv = 8, L = 4096, D = 64, W = 128: S = 4
// 303 -> 253, S = 20 418 -> 327; D = 128, Hq = 32, L = 2048, W = 256, S = 4 259 -> 212 (part of it from the
// registers that the regular workgroups no longer share with that path: without sinks 224 -> 216, 214 -> 195).
// What is left of the S = 4 case's chunks, 37 us, is mostly their Q and dO (134 MB, 27 us at the rate of a copy).
// `c` is the workgroup's place among the chunk workgroups (all of block 0).
template <int D, int KB>
__device__ __forceinline__ void sink_chunk32(const Args& a, int c, float* lds) {
  constexpr int SLOT = kDkdv32Slot<D>, STAGE = 2 * SLOT, NT = D / 16;
  static_assert(4 * 8 * NT * 64 <= 2 * STAGE, "the waves' sums of 16 keys fit the stages");
  const int lane = threadIdx.x & 63, m = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kh = wave & 1, hh = wave >> 1, S = a.S;
  const int kvh = c / (a.B * a.n_chunks), b = c / a.n_chunks % a.B, chunk = c % a.n_chunks;
  const Seq sq = seq_of(a, b);
  const int lo = kv_chunk_lo(0, chunk, a.chunk_rows, sq.L, a.W), hi = kv_chunk_hi(0, chunk, a.chunk_rows, sq.L, a.W);
  if (lo >= hi) return;  // (the fold reads no slot of it)
  const int qb_lo = lo / 32, n_qb = (hi + 31) / 32 - qb_lo, n_items = a.G * n_qb;
  const ItemStage<D> issue(a, sq, b, kvh, qb_lo, n_qb, n_items, lds);
  issue(0);
  const float c2 = a.scale * kLog2e;
  float kf[KB][D / 4], vf[KB][D / 4];
  f32x4 dk[KB][NT], dv[KB][NT];
#pragma unroll
  for (int x = 0; x < KB; ++x) {
    const int key = 16 * x + m, d0 = (g >> 1) * (D / 2) + 4 * (g & 1);
    const float* K = static_cast<const float*>(a.k) + slice_off(a.sk, b, kvh, sq.row) + int64_t(key) * a.sk[2] + d0;
    const float* V = static_cast<const float*>(a.v) + slice_off(a.sv, b, kvh, sq.row) + int64_t(key) * a.sv[2] + d0;
#pragma unroll
    for (int u = 0; u < D / 16; ++u) {
      const f32x4 kx = key < S ? ld4f(K + 8 * u) : f32x4{}, vx = key < S ? ld4f(V + 8 * u) : f32x4{};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        kf[x][4 * u + j] = kx[j] * c2;
        vf[x][4 * u + j] = vx[j];
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      dk[x][t] = f32x4{};
      dv[x][t] = f32x4{};
    }
  }
  auto cols16 = [&](const float* t, int row, float (&out)[NT]) {  // columns NT m .. NT m + NT - 1
    if constexpr (NT >= 4) {
#pragma unroll
      for (int i = 0; i < NT / 4; ++i) {
        const f32x4 x = ld4f(t + row * D + 4 * ((NT / 4 * m + i) ^ swz32<D>(row)));
#pragma unroll
        for (int e = 0; e < 4; ++e) out[4 * i + e] = x[e];
      }
    } else {
      const float* p = t + row * D + 4 * ((NT * m >> 2) ^ swz32<D>(row)) + (NT * m & 3);
#pragma unroll
      for (int e = 0; e < NT; ++e) out[e] = p[e];
    }
  };
  const int steps = (n_items + 1) / 2;
  for (int s = 0; s < steps; ++s) {
    wait_vm_lgkm0_barrier<0>();  // step s has landed, and nobody reads the other stage any more
    if (s + 1 < steps) issue(s + 1);
    const int i = 2 * s + hh;
    const int r0 = 32 * (qb_lo + i % n_qb) + 16 * kh;  // this wave's first row
    if (!(i < n_items && r0 + 16 > lo && r0 < hi)) continue;
    const float* Qt = lds + (s & 1) * STAGE + hh * SLOT;
    const float* Dt = Qt + 32 * D;
    const float* st = Qt + 64 * D + 16 * kh + 4 * g;
    f32x4 sc[KB], dp[KB];
#pragma unroll
    for (int x = 0; x < KB; ++x) {
      sc[x] = f32x4{};
      dp[x] = ld4f(st + 32);
    }
#pragma unroll
    for (int u = 0; u < D / 16; ++u) {
      const f32x4 qa = tile_half<D>(Qt, 16 * kh + m, g >> 1, 2 * u + (g & 1));
      const f32x4 da = tile_half<D>(Dt, 16 * kh + m, g >> 1, 2 * u + (g & 1));
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int x = 0; x < KB; ++x) {
          sc[x] = mfma16(qa[j], kf[x][4 * u + j], sc[x]);
          dp[x] = mfma16(da[j], vf[x][4 * u + j], dp[x]);
        }
    }
    const f32x4 l4 = ld4f(st);
    float p[KB][4], ds[KB][4];
#pragma unroll
    for (int x = 0; x < KB; ++x)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool on = 16 * x + m < S && unsigned(r0 + 4 * g + e - lo) < unsigned(hi - lo);
        p[x][e] = on ? exp2f(sc[x][e] - l4[e]) : 0.f;
        ds[x][e] = p[x][e] * dp[x][e];
      }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float oa[NT], qa[NT];
      cols16(Dt, 16 * kh + 4 * g + e, oa);
      cols16(Qt, 16 * kh + 4 * g + e, qa);
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int x = 0; x < KB; ++x) {
          dv[x][t] = mfma16(oa[t], p[x][e], dv[x][t]);
          dk[x][t] = mfma16(qa[t], ds[x][e], dk[x][t]);
        }
    }
  }
  // the four waves' sums, 16 keys at a time, in order; wave w adds and stores rows [2 NT w, 2 NT (w + 1))
  // of the 8 NT [dK, dV][t][e]
#pragma unroll
  for (int x = 0; x < KB; ++x) {
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        lds[((wave * 2 * NT + t) * 4 + e) * 64 + lane] = dk[x][t][e];
        lds[((wave * 2 * NT + NT + t) * 4 + e) * 64 + lane] = dv[x][t][e];
      }
    __syncthreads();
    if (16 * x + m < S) {
      float* out = a.partial + ((int64_t(b) * a.Hkv + kvh) * (a.n_chunks + 1) + chunk) * 2 * S * D + (16 * x + m) * D;
#pragma unroll
      for (int y = 0; y < 2 * NT; ++y) {
        const int row = 2 * NT * wave + y, t = row / 4 % NT, e = row % 4;
        float v = lds[row * 64 + lane];
#pragma unroll
        for (int w = 1; w < 4; ++w) v += lds[(w * 8 * NT + row) * 64 + lane];
        out[(row / (4 * NT)) * S * D + NT * (4 * g + e) + t] = v;
      }
    }
  }
}

template <int D>
__global__ __launch_bounds__(256, D == 128 ? 1 : 2) void dkdv32_kernel(const Args a) {
  constexpr int HD = D / 2;
  constexpr int DB = kDB<D>;
  constexpr int SLOT = kDkdv32Slot<D>, STAGE = 2 * SLOT;
  static_assert(2 * STAGE >= 2 * 2 * DB * 16 * 64, "the item slots' sums fit the stages");
  __shared__ __attribute__((aligned(16))) float lds[2 * STAGE];
  const int lane = threadIdx.x & 63, r = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int kh = wave & 1, hh = wave >> 1;
  const unsigned wg = a.wg_base + blockIdx.x;
  if (wg >= a.main_wgs) return bwd_aux<D, 4>(a, wg, lds);
  const int W = a.W, S = a.S, G = a.G, ns = a.kv_split;
  const int per = a.vl_kblocks ? a.vl_kblocks : a.n_kblocks;
  const int streams = ns * a.Hkv * (a.vl_kblocks ? 1 : a.B);
  const int id = int(wg);
  int kvh, b, kblk, piece = 0, chunk = -1;
  int64_t part_slot = 0;
  if (id < streams * per) {
    const KvPiece t = kv_piece(id, streams, ns);
    piece = t.piece;
    part_slot = (int64_t(t.group) * per + t.p) * ns + piece;
    if (a.vl_kblocks) {
      kvh = t.group;
      if (!varlen_nth(a, t.p, per, kKvKeys, 1, b, kblk)) return;
    } else {
      kvh = t.group / a.B;
      b = t.group % a.B;
      kblk = t.p;
    }
  } else {
    const int n_cw = a.nsp * a.n_chunks, c = id - streams * per;
    if (S <= 16) return sink_chunk32<D, 1>(a, c, lds);
    if (S <= 32) return sink_chunk32<D, 2>(a, c, lds);
    kvh = c / (a.B * n_cw);
    b = c / n_cw % a.B;
    kblk = c % n_cw % a.nsp;
    chunk = c % n_cw / a.nsp;
  }
  const Seq sq = seq_of(a, b);
  const int L = sq.L;
  if (kKvKeys * kblk >= L) return;
  const bool is_chunk = chunk >= 0, partial_block = kblk < a.nsp;
  int lo, hi;
  if (is_chunk) {
    lo = kv_chunk_lo(kblk, chunk, a.chunk_rows, L, W);
    hi = kv_chunk_hi(kblk, chunk, a.chunk_rows, L, W);
    if (lo >= hi) return;  // (the fold reads no slot of it)
  } else {
    lo = kKvKeys * kblk;
    hi = kv_window_end(kblk, L, W);  // > lo
  }
  const int ks0 = kKvKeys * kblk + 32 * kh;  // this wave's keys
  const int key = ks0 + r;
  const bool wave_on = ks0 < L && (!is_chunk || ks0 < S);
  const int wlo = is_chunk ? lo : max(lo, ks0);

  // the steps [s_lo, s_hi) of this workgroup over the items (g, qb), qb fastest
  const int qb_lo = lo / 32, n_qb = (hi + 31) / 32 - qb_lo;
  const int n_items = G * n_qb, all_steps = (n_items + 1) / 2;
  int s_lo = 0, s_hi = all_steps;
  if (!is_chunk) {
    s_lo = int(int64_t(all_steps) * piece / ns);
    s_hi = int(int64_t(all_steps) * (piece + 1) / ns);
  }

  const ItemStage<D> issue(a, sq, b, kvh, qb_lo, n_qb, n_items, lds);
  if (s_lo < s_hi) issue(s_lo);

  const float c2 = a.scale * kLog2e;
  const float* K = static_cast<const float*>(a.k) + slice_off(a.sk, b, kvh, sq.row);
  const float* V = static_cast<const float*>(a.v) + slice_off(a.sv, b, kvh, sq.row);
  float kf[HD], vf[HD];
  load_half_row<D>(K, a.sk[2], key, L, h, c2, kf);
  load_half_row<D>(V, a.sv[2], key, L, h, 1.f, vf);
  f32x16 dk[DB], dv[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) {
    dk[db] = f32x16{};
    dv[db] = f32x16{};
  }
  // the mask as one unsigned compare, row - mref < lim (see bwd_dkdv_kernel)
  unsigned lim;
  if (is_chunk) lim = key < S ? unsigned(hi - lo) : 0u;
  else lim = key < S ? (partial_block ? unsigned(max(hi - key, 0)) : 0x80000000u) : unsigned(W);
  const int mref = is_chunk ? lo : key;

  for (int s = s_lo; s < s_hi; ++s) {
    wait_vm_lgkm0_barrier<0>();  // step s has landed, and nobody reads the other stage any more
    if (s + 1 < s_hi) issue(s + 1);
    const int i = 2 * s + hh;
    const int qr0 = 32 * (qb_lo + i % n_qb);
    if (!(wave_on && i < n_items && qr0 + 32 > wlo && qr0 < hi && kv_half_needs(qr0, ks0, L, W, S))) continue;
    const float* Qt = lds + (s & 1) * STAGE + hh * SLOT;
    const float* Dt = Qt + 32 * D;
    const float* st = Qt + 64 * D;
    // S = Q K^T and dP - delta = dO V^T - delta (queries x keys): lane (r, h) supplies rows qr0 + r
    f32x16 sc = f32x16{}, dp;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 nv = ld4f(st + 32 + 8 * j + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) dp[4 * j + e] = nv[e];
    }
#pragma unroll
    for (int u = 0; u < D / 8; ++u) {
      const f32x4 qa = tile_half<D>(Qt, r, h, u), da = tile_half<D>(Dt, r, h, u);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        sc = mfma32(qa[j], kf[4 * u + j], sc);
        dp = mfma32(da[j], vf[4 * u + j], dp);
      }
    }
    const bool full = !is_chunk && qr0 >= wlo && qr0 + 32 <= hi && tile_full(ks0, qr0, W, S);
    const int m0 = qr0 + 4 * h - mref;
    float p[16], ds[16];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const f32x4 l4 = ld4f(st + 8 * j + 4 * h);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int x = 4 * j + e;
        float pe = exp2f(sc[x] - l4[e]);
        if (!full) pe = unsigned(m0 + 8 * j + e) < lim ? pe : 0.f;
        p[x] = pe;
        ds[x] = pe * dp[x];
      }
    }
    // dV^T += dO^T P and dK^T += Q^T dS: lane (r, h) supplies dO / Q[qr0 + crow(t, h)][DB r + db]
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      float oa[DB], qa[DB];
      tile_cols<D>(Dt, crow(x, h), r, oa);
      tile_cols<D>(Qt, crow(x, h), r, qa);
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        dv[db] = mfma32(oa[db], p[x], dv[db]);
        dk[db] = mfma32(qa[db], ds[x], dk[db]);
      }
    }
  }

  // the two item slots' sums (hh = 0 gets hh = 1's), fixed order; the stages are reused
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  float* red = lds + kh * (2 * DB * 16 * 64) + lane;
  if (hh == 1) {
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        red[(db * 16 + e) * 64] = dk[db][e];
        red[((DB + db) * 16 + e) * 64] = dv[db][e];
      }
  }
  __syncthreads();
  if (hh == 1) return;
#pragma unroll
  for (int db = 0; db < DB; ++db)
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      dk[db][e] += red[(db * 16 + e) * 64];
      dv[db][e] += red[((DB + db) * 16 + e) * 64];
    }

  if (!is_chunk && ns > 1) {  // a piece: register quads in lane order, whole lines per store
    float* out = a.kv_part + part_slot * (2 * kKvKeys * 32 * DB) + kh * (DB * 16 * 64) + 4 * lane;
#pragma unroll
    for (int db = 0; db < DB; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        float* o = out + (db * 4 + j) * 256;
        st4f(o, f32x4{dk[db][4 * j], dk[db][4 * j + 1], dk[db][4 * j + 2], dk[db][4 * j + 3]});
        st4f(o + kKvKeys * 32 * DB, f32x4{dv[db][4 * j], dv[db][4 * j + 1], dv[db][4 * j + 2], dv[db][4 * j + 3]});
      }
    return;
  }
  if (key >= L) return;
  if (partial_block && key < S) {
    float* pk = a.partial + ((int64_t(b) * a.Hkv + kvh) * (a.n_chunks + 1) + (is_chunk ? chunk : a.n_chunks)) * 2 * S * D + key * D;
    float* pv = pk + S * D;
    store_cols<D>(pk, dk, h, 1.f);
    store_cols<D>(pv, dv, h, 1.f);
    return;
  }
  if (is_chunk) return;
  store_cols<D>(static_cast<float*>(a.dk) + slice_off(a.sdk, b, kvh, sq.row + key), dk, h, a.scale);
  store_cols<D>(static_cast<float*>(a.dv) + slice_off(a.sdv, b, kvh, sq.row + key), dv, h, 1.f);
}

// Adds the kv_split pieces of every key block, piece by piece in order, and writes dK and dV, or a sink
// row's sums to its block's own slot of the sink partials.  One thread per register quad of a key
// row (4 DB columns).
template <int D>
__global__ __launch_bounds__(256) void fold_pieces32_kernel(const Args a) {
  constexpr int DB = kDB<D>;
  constexpr int WGS = 2 * 2 * 4 * 64 / 256;  // [dK, dV][key half][quad][lane]
  const int per = a.vl_kblocks ? a.vl_kblocks : a.n_kblocks, ns = a.kv_split;
  const int blk = blockIdx.x / WGS, u = blockIdx.x % WGS * 256 + threadIdx.x;
  const int lane = u & 63, j = (u >> 6) & 3, kh = (u >> 8) & 1, t = u >> 9;
  int kvh, b, kblk;
  if (a.vl_kblocks) {
    kvh = blk / per;
    if (!varlen_nth(a, blk % per, per, kKvKeys, 1, b, kblk)) return;
  } else {
    kblk = blk % per;
    kvh = blk / per / a.B;
    b = blk / per % a.B;
  }
  const Seq sq = seq_of(a, b);
  const int r = lane & 31, h = lane >> 5, key = kKvKeys * kblk + 32 * kh + r;
  if (key >= sq.L || (D == 16 && j >= 2)) return;
  constexpr int HALF = kKvKeys * 32 * DB;
  const float* src = a.kv_part + int64_t(blk) * ns * (2 * HALF) + t * HALF + kh * (DB * 16 * 64) + j * 256 + 4 * lane;
  f32x4 x[DB];
#pragma unroll
  for (int db = 0; db < DB; ++db) x[db] = f32x4{0.f, 0.f, 0.f, 0.f};
  for (int s = 0; s < ns; ++s)
#pragma unroll
    for (int db = 0; db < DB; ++db) x[db] += ld4f(src + int64_t(s) * (2 * HALF) + db * 1024);
  float* dst;
  float sc = 1.f;
  if (kblk < a.nsp && key < a.S) {
    dst = a.partial + (((int64_t(b) * a.Hkv + kvh) * (a.n_chunks + 1) + a.n_chunks) * 2 + t) * a.S * D + key * D;
  } else if (t == 0) {
    dst = static_cast<float*>(a.dk) + slice_off(a.sdk, b, kvh, sq.row + key);
    sc = a.scale;
  } else {
    dst = static_cast<float*>(a.dv) + slice_off(a.sdv, b, kvh, sq.row + key);
  }
  dst += DB * (8 * j + 4 * h);
#pragma unroll
  for (int y = 0; y < DB; ++y) {
    f32x4 v;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = x[(4 * y + e) % DB][(4 * y + e) / DB] * sc;
    st4f(dst + 4 * y, v);
  }
}

// Adds the partial sums of the sink rows of the blocks below nsp, slot by slot in order
// (deterministic).  Grid (sink rows, Hkv, B): one workgroup of 128 threads per key.
template <int D>
__global__ __launch_bounds__(128) void fold32_kernel(const Args a) {
  const int kvh = blockIdx.y, b = blockIdx.z;
  const Seq sq = seq_of(a, b);
  const int key = blockIdx.x, d = threadIdx.x, kblk = key / kKvKeys;
  if (key >= sq.L || d >= D) return;
  const float* src = a.partial + (int64_t(b) * a.Hkv + kvh) * (a.n_chunks + 1) * 2 * a.S * D + key * D + d;
  const int64_t slot = int64_t(2) * a.S * D;
  // chunks that start past the sequence's end wrote nothing
  const int rows = sq.L - kv_chunk_base(kblk, sq.L, a.W);
  const int n = kv_window_end(kblk, sq.L, a.W) < sq.L ? (rows + a.chunk_rows - 1) / a.chunk_rows : 0;
  float sk = src[a.n_chunks * slot], sv = src[a.n_chunks * slot + a.S * D];
  constexpr int kBatch = 16;  // loads in flight (one at a time, c2's 62 chunks took 17 us)
  for (int c0 = 0; c0 < n; c0 += kBatch) {
    float xk[kBatch], xv[kBatch];
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      const float* p = src + min(c0 + j, n - 1) * slot;
      xk[j] = p[0];
      xv[j] = p[a.S * D];
    }
#pragma unroll
    for (int j = 0; j < kBatch; ++j) {
      sk += c0 + j < n ? xk[j] : 0.f;
      sv += c0 + j < n ? xv[j] : 0.f;
    }
  }
  static_cast<float*>(a.dk)[slice_off(a.sdk, b, kvh, sq.row + key) + d] = sk * a.scale;
  static_cast<float*>(a.dv)[slice_off(a.sdv, b, kvh, sq.row + key) + d] = sv;
}

template <int D>
hipError_t fwd_d(const Args& a, hipStream_t s) {
  Args x = a;
  return launch_in_ranges(x, wgs_with_aux(x, int64_t(a.n_qtiles) * a.B * (a.Hq / a.wh), false),
                          [&](dim3 grid) { hipLaunchKernelGGL(fwd32_kernel<D>, grid, dim3(256), 0, s, x); });
}
template <int D>
hipError_t dq_d(const Args& a, hipStream_t s) {
  Args x = a;
  return launch_in_ranges(x, int64_t(a.n_qtiles) * a.B * (a.Hq / a.wh),
                          [&](dim3 grid) { hipLaunchKernelGGL(dq32_kernel<D>, grid, dim3(256), 0, s, x); });
}
template <int D>
hipError_t dkdv_d(const Args& a, hipStream_t s) {
  const int blocks = a.Hkv * (a.vl_kblocks ? a.vl_kblocks : a.B * a.n_kblocks);
  Args x = a;
  hipError_t e = launch_in_ranges(x, wgs_with_aux(x, int64_t(a.kv_split) * blocks + a.n_chunk_wgs, true),
                                  [&](dim3 grid) { hipLaunchKernelGGL(dkdv32_kernel<D>, grid, dim3(256), 0, s, x); });
  if (e == hipSuccess && a.kv_split > 1) {
    hipLaunchKernelGGL(fold_pieces32_kernel<D>, dim3(4 * blocks), dim3(256), 0, s, a);
    e = hipGetLastError();
  }
  if (e == hipSuccess && a.nsp > 0) {
    hipLaunchKernelGGL(fold32_kernel<D>, dim3(min(a.S, kKvKeys * a.nsp), a.Hkv, a.B), dim3(128), 0, s, a);
    e = hipGetLastError();
  }
  return e;
}

}  // namespace

#define FA_F32_D(FN)                  \
  switch (D) {                        \
    case 16: return FN<16>(a, s);     \
    case 32: return FN<32>(a, s);     \
    case 64: return FN<64>(a, s);     \
    case 128: return FN<128>(a, s);   \
  }                                   \
  return hipErrorInvalidValue;

hipError_t launch_fwd_f32(const Args& a, int D, hipStream_t s) { FA_F32_D(fwd_d) }
hipError_t launch_bwd_dq_f32(const Args& a, int D, hipStream_t s) { FA_F32_D(dq_d) }
hipError_t launch_bwd_dkdv_f32(const Args& a, int D, hipStream_t s) { FA_F32_D(dkdv_d) }

}  // namespace fa
