// fa_args.h - kernel argument block shared by the C ABI (fa_capi.cpp) and the kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace fa {

// Everything a kernel needs, passed by value through the kernarg segment.  Strides are in
// elements; sequence indices are int32 (validated: L < 2^28), offsets are formed in int64.
struct Args {
  // inputs
  const void* q;
  const void* k;
  const void* v;
  const void* o;     // backward: forward output
  const void* dout;  // backward: upstream gradient
  const float* lse;  // backward: forward statistic
  // outputs
  void* o_out;       // forward
  float* lse_out;    // forward
  void* dq;
  void* dk;
  void* dv;
  // backward workspace
  float* delta;      // row statistics: [B][Hq][Lp / 32][lse * log2(e) x 32, -delta x 32] fp32, Lp = L
                     // rounded up to 32 (written by the dQ kernel, read by the dK/dV kernel)
  float* partial;    // sink-key partial sums, see fa_bwd.hip
  // learned per-head sink logits (GPT-OSS): NULL, or [Hq] fp32 logits that join every row's
  // softmax denominator without a value row
  const float* sink_logits;
  float* dsink;      // backward: [Hq] fp32 gradient of the sink logits (NULL: not computed)
  float* dsink_part; // backward workspace: [B][Hq][Lp / 32] per-32-row partial sums of dsink
  int64_t sq[3], sk[3], sv[3], so[3], sdo[3], slse[3], sdq[3], sdk[3], sdv[3], so_out[3];
  int B, Hq, Hkv, L, G, Lp;
  int W, S;          // window and sink, clamped to [0, L]
  float scale;       // softmax scale as given
  float c;           // |scale| * log2(e), kept > 0: scores enter exp2 as s * c
  uint32_t qsign;    // 0x80008000 when scale < 0: flips the sign of Q in the score product
                     // (0x80808080 for e4m3 inputs)
  float oscale;      // forward with e4m3 inputs: O is multiplied by V's dequantisation factor
  // q-major kernels (forward, dQ): a workgroup is wq x wh waves, each wave 32 rows x HPW heads
  int wq, wh;
  int n_qtiles;
  // KV-major kernel (dK/dV)
  int n_kblocks;     // ceil(L / 64)
  int nsp;           // leading 64-key blocks whose sink rows are split into chunks
  int n_chunks;      // chunks of chunk_rows query rows per chunked block (0 when nsp == 0)
  int chunk_rows;
  int n_chunk_wgs;   // B * Hkv * nsp * n_chunks
  int srows;         // sink rows stored per block in the partial sums: min(S, 64)
  // sink rows in the dQ kernel (dq_sink_mode): rows past key block 0's window add the sink keys'
  // dK/dV there
  int sink_dq;       // 1 in that mode
  float* dq_sink_part;  // [n_tiles][dK, dV][srows][D] fp32: a run's sums at the slot of its first tile
  int dq_wgs;           // the dQ kernel's grid (set for the sink fold)
  // The sliding dQ kernel (fa_bwd_slide.hip), when it runs instead of bwd_dq_kernel (dq_slide = 1),
  // and the sliding forward (fa_fwd.hip fwd_slide_kernel): their workgroups ("units") take slide_ct
  // consecutive 32-row tiles of 8 query heads; a (batch, KV head, head group of 8) has slide_ncu
  // units, in that order (chunks fastest).  In dq_sink_mode dQ unit u writes slot u of
  // dq_sink_part.
  int dq_slide;
  int slide_ct;
  int slide_ncu;
  // variable-length batches: NULL, or [B + 1] device offsets of the sequences' first rows in
  // tensors of total_rows packed rows (L is then the longest sequence, batch strides are 0)
  const int* cu_seqlens;
  int total_rows;
  // sequences with other rows between them: NULL, or [B] device lengths; sequence b is then rows
  // [cu_seqlens[b], cu_seqlens[b] + seq_lens[b])
  const int* seq_lens;
  int token_rows;    // rows of all sequences together, at most total_rows (host-side planning)
  // Packed batches: the sliding kernels' units and the dK/dV kernel's 64-key workgroups are handed
  // out over the pieces the sequences hold (varlen_nth), so no workgroup is launched for a piece
  // past a short sequence's end.  vl_units units per (KV head, head group) and vl_kblocks key
  // blocks per KV head bound those pieces; 0: the fixed-length enumeration (B x slide_ncu units,
  // B x n_kblocks blocks).
  int vl_units;
  int vl_kblocks;
  // dK/dV split (kv_split > 1, see plan_kv_split in fa_capi.cpp): every key block's steps are cut into
  // kv_split pieces, one workgroup each, whose fp32 sums go to kv_part [key block][piece][dK, dV]
  // [64 D]; bwd_dkdv_fold_kernel adds the pieces in order.
  int kv_split;
  float* kv_part;
  // a kernel's own workgroups are [0, main_wgs); the ones behind them do the work of fa_aux.h, tail_wgs of
  // them on packed rows outside every sequence
  unsigned main_wgs;
  int tail_wgs;
  // kernels with a workgroup per tile of a B x longest sequence grid: the first workgroup of this launch
  // (launch_in_ranges)
  unsigned wg_base;
};

// A grid holds fewer than 2^32 threads; a larger one is not refused, but not all of it runs (measured).
// Launches of 256-thread workgroups whose number follows B times the longest sequence (most of them empty in a
// packed batch with short ones) are cut into ranges of kRangeWgs, whole rounds of the 8 XCDs; `launch` gets a
// range's grid, with args.wg_base set.
constexpr int64_t kRangeWgs = int64_t(1) << 23;
// The other launches are refused instead.
inline bool grid_fits(int64_t wgs, int threads = 256) { return wgs * threads < int64_t(1) << 32; }
template <typename F>
inline hipError_t launch_in_ranges(Args& args, int64_t wgs, F&& launch) {
  for (int64_t lo = 0; lo < wgs; lo += kRangeWgs) {
    args.wg_base = unsigned(lo);
    launch(dim3(unsigned(wgs - lo < kRangeWgs ? wgs - lo : kRangeWgs)));
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

// Sequence b: its length and the row where it starts in the packed tensors (fixed-length
// batches: L rows from row 0 of batch b's slice).  Offsets are clamped to the tensors' rows and
// lengths to L, so malformed offsets cannot address memory outside the tensors.
struct Seq {
  int L;
  int64_t row;
};

template <typename A>
__device__ __forceinline__ Seq seq_of(const A& a, int b) {
  if (!a.cu_seqlens) return Seq{a.L, 0};
  // (both loads first: their latency is paid once)
  int lo = a.cu_seqlens[b];
  const int e = *(a.seq_lens ? a.seq_lens + b : a.cu_seqlens + b + 1);
  lo = lo < 0 ? 0 : (lo > a.total_rows ? a.total_rows : lo);
  int hi = !a.seq_lens ? e : e < a.total_rows - lo ? lo + e : a.total_rows;
  hi = hi < lo ? lo : (hi > a.total_rows ? a.total_rows : hi);
  const int n = hi - lo;
  return Seq{n < a.L ? n : a.L, lo};
}

// Packed batches: sequence b holds ceil(ceil(L_b / rows) / per) pieces of `per` blocks of `rows`
// rows, and `slots` >= their number N of workgroups enumerate them, the sequences' pieces in order
// after slots - N that have none (so that the empty ones, which exit at once, are dispatched
// first and every piece gets a place in the first round).  For the wave-uniform slot index p, sets
// b and the piece's index within its sequence and returns true, or returns false for an empty
// slot.  Wave-wide prefix sums over the sequences, 64 per round: every lane of the wave must call
// it.  (The results are made scalar so that the callers' index arithmetic stays scalar.)
template <typename A>
__device__ inline bool varlen_nth(const A& a, int p, int slots, int rows, int per, int& b, int& piece) {
  const int lane = threadIdx.x & 63;
  auto count = [&](int bb) { return bb < a.B ? ((seq_of(a, bb).L + rows - 1) / rows + per - 1) / per : 0; };
  auto prefix = [&](int n) {  // inclusive prefix sum over the wave
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int y = __shfl_up(n, o);
      if (lane >= o) n += y;
    }
    return n;
  };
  int total = 0;
  for (int b0 = 0; b0 < a.B; b0 += 64) total += __builtin_amdgcn_readfirstlane(__shfl(prefix(count(b0 + lane)), 63));
  p -= slots - total;
  if (p < 0) return false;
  int base = 0;
  for (int b0 = 0; b0 < a.B; b0 += 64) {
    const int n = count(b0 + lane);
    const int x = prefix(n);
    const int tot = __builtin_amdgcn_readfirstlane(__shfl(x, 63));
    if (p < base + tot) {
      const unsigned long long m = __ballot(base + x > p);
      const int l = __builtin_amdgcn_readfirstlane(__ffsll(m) - 1);  // the first sequence whose pieces reach past p
      b = b0 + l;
      piece = __builtin_amdgcn_readfirstlane(p - base - (__shfl(x, l) - __shfl(n, l)));
      return true;
    }
    base += tot;
  }
  return false;
}

// Workgroup id -> piece, group and key block index of a split dK/dV grid (see bwd_dkdv_kernel): `streams`
// = `ns` pieces x groups, each with one workgroup per key block.
struct KvPiece {
  int piece, group, p;
};
__device__ __forceinline__ KvPiece kv_piece(int id, int streams, int ns) {
  int stream, p;
  if (streams % 8 == 0) {  // XCD id % 8 owns streams / 8 streams
    const int spx = streams / 8, pos = id / 8;
    p = pos / spx;
    stream = id % 8 * spx + pos % spx;
  } else {
    p = id / streams;
    stream = id % streams;
  }
  return KvPiece{stream % ns, stream / ns, p};
}

// Workgroup id -> (stream, position) of the query-major kernels that run one tile per workgroup: a stream
// is one (KV head, batch, head group), positions count its row tiles from the last.  An XCD owns whole
// streams where their number allows (their tiles share K/V rows in its L2) and takes their tiles
// together, the last rows, which see the most keys, first.
// With `rotate` (a packed batch) the streams take turns: an XCD's workgroups go to its shader engines in
// turn, so where the streams of an XCD are a multiple of them, one engine would get every tile of the same
// sequences.  Full causal forward, Hq = 64, Hkv = 8, D = 64, without -> with: sequences of 1536, 1187, 640 and
// 933 rows 83 -> 66 us; of 4096, 2048, 1024, 512, 3000, 1500, 700 and 3504 rows 727 -> 413 us.
struct QStream {
  int stream, pos;
};
__device__ __forceinline__ QStream q_stream(int id, int streams, bool rotate) {
  const int spx = streams % 8 == 0 ? streams / 8 : streams;  // streams in turn
  const int i = streams % 8 == 0 ? id / 8 : id, base = streams % 8 == 0 ? id % 8 * spx : 0;
  const int pos = i / spx, s = i % spx;
  return QStream{base + (rotate ? (s + pos) % spx : s), pos};
}

// Element offset of row `row` of (batch b, head h) of a tensor with strides s[3] (a plain array
// or one read through args_fresh()).
template <typename S3>
__device__ __forceinline__ int64_t slice_off(const S3& s, int b, int h, int64_t row) {
  return int64_t(b) * s[0] + int64_t(h) * s[1] + row * s[2];
}

#if defined(__HIP_DEVICE_COMPILE__)
// The kernel's Args in the kernarg segment (constant address space), re-read at the point of
// use.  Fields read through the by-value parameter are loaded once at kernel entry and stay in
// scalar registers for the whole kernel; the many pointers and 64-bit strides that only the
// per-tile address arithmetic needs then spill scalar registers into vector lanes inside the key
// loops.  The empty asm hides where the pointer comes from, so the loads through each call's
// result are issued after the call, where the fields are used (scalar-cache hits).
using KArgs = const __attribute__((address_space(4))) Args;
__device__ __forceinline__ KArgs& args_fresh() {
  KArgs* p = (KArgs*)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(p));
  return *p;
}
#else
using KArgs = const Args;
__device__ KArgs& args_fresh();  // device code only
#endif

// Compute units of the current device (fa_capi.cpp).
int device_cus();

// Launchers (return the hipError_t of the launch; launch_bwd_dkdv also launches the sink fold).  The forward
// and dK/dV launches add the workgroups of fa_aux.h.
hipError_t launch_fwd(const Args& a, int dtype, int D, hipStream_t stream);
// e4m3 q, k, v; bf16 o; fp8_pv: P V on the fp8 MFMA as well
hipError_t launch_fwd_fp8(const Args& a, int D, int hpw, bool fp8_pv, hipStream_t stream);
// the forward with one tile per workgroup, whose keys are split over `ksp` waves: 1, 2 or 4 (D < 128);
// reads wq, wh (wq wh ksp = 4) and n_qtiles (tiles of 32 wq rows)
hipError_t launch_fwd_split(const Args& a, int dtype, int D, int hpw, int ksp, hipStream_t stream);
hipError_t launch_bwd_dq(const Args& a, int dtype, int D, int hpw, hipStream_t stream);
// dQ with one tile per workgroup, whose keys are split over `ksp` waves: 1, 2 or 4 (D < 128); no sink rows
// (sink_dq = 0); reads wq, wh (wq wh ksp = 4) and n_qtiles
hipError_t launch_bwd_dq_split(const Args& a, int dtype, int D, int ksp, hipStream_t stream);
// the sliding dQ kernel (D = 64, 16-bit, G a multiple of 8, 1 <= W <= 161, S <= 32)
hipError_t launch_bwd_dq_slide(const Args& a, int dtype, hipStream_t stream);
// the sliding forward (the same, W <= 129; reads slide_ct / slide_ncu)
hipError_t launch_fwd_slide(const Args& a, int dtype, hipStream_t stream);
hipError_t launch_bwd_dkdv(const Args& a, int dtype, int D, hipStream_t stream);
// does the 32-key dK/dV kernel serve this 16-bit backward on a device of `cus` compute units?
bool dkdv4_eligible(const Args& a, int D, int cus);
// float32 inputs (fa_f32.hip).  The dK/dV launch reads the same plan as launch_bwd_dkdv (key blocks,
// pieces, sink blocks and their chunk workgroups) and launches the folds.
hipError_t launch_fwd_f32(const Args& a, int D, hipStream_t stream);
hipError_t launch_bwd_dq_f32(const Args& a, int D, hipStream_t stream);
hipError_t launch_bwd_dkdv_f32(const Args& a, int D, hipStream_t stream);

}  // namespace fa
