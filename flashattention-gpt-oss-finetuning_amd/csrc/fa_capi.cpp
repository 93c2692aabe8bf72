// fa_capi.cpp - the C ABI declared in include/fa_gfx950.h: host-side validation, workspace
// sizing, launch-shape selection and dispatch to the gfx950 kernels.
//
// Validation mirrors the reference's checks (flash_attention_gpt_oss.py:343-354:
// causal only, shape agreement, D <= 128, Hq % Hkv == 0; benchmark_backward_speed.py:476-484)
// plus what the kernels assume (16-byte aligned rows, D in {16, 32, 64, 128}).  Nothing in
// fa_check_* touches HIP, so the checks run on machines without a GPU.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstring>

#include "../../include/fa_gfx950.h"
#include "fa_args.h"
#include "fa_plan.h"

namespace {

constexpr int64_t kMaxSeq = int64_t(1) << 28;
constexpr int kChunkRows = 64;  // query rows per sink-chunk workgroup of the dK/dV kernel

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// strides in elements of `elem_bytes` bytes: non-negative and whole 16-byte multiples
bool strides_ok(const int64_t s[3], int elem_bytes = 2) {
  const int64_t m = 16 / elem_bytes - 1;
  for (int i = 0; i < 3; ++i)
    if (s[i] < 0 || (s[i] & m) != 0) return false;
  return true;
}

bool lse_strides_ok(const int64_t s[3]) { return s[0] >= 0 && s[1] >= 0 && s[2] >= 0; }

bool aligned4(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 3u) == 0; }

// The kernels address one (batch, head) slice of a tensor with 32-bit byte offsets: its L rows
// must span fewer than 2^31 bytes.
bool slice_fits(const int64_t s[3], int L, int D, int elem_bytes) {
  return (int64_t(L - 1) * s[2] + D) * elem_bytes < (int64_t(1) << 31);
}

// bytes per element of q/k/v/o/dout/dq/dk/dv for a 16-bit or float32 call
int elem_bytes(int32_t dtype) { return dtype == FA_DTYPE_F32 ? 4 : 2; }

int check_common(int32_t B, int32_t Hq, int32_t Hkv, int32_t L, int32_t D, int32_t W, int32_t S,
                 float scale, int32_t dtype) {
  if (B < 1 || Hq < 1 || Hkv < 1 || L < 1) return FA_ERR_SHAPE;
  if (Hq % Hkv != 0) return FA_ERR_SHAPE;
  if (D != 16 && D != 32 && D != 64 && D != 128) return FA_ERR_HEAD_DIM;
  if (dtype != FA_DTYPE_BF16 && dtype != FA_DTYPE_F16 && dtype != FA_DTYPE_F32) return FA_ERR_DTYPE;
  if (W < 1 && S < 1) return FA_ERR_MASK;
  if (!std::isfinite(scale)) return FA_ERR_SCALE;
  if (int64_t(L) > kMaxSeq) return FA_ERR_OVERFLOW;
  // grid sizes of the launches must fit 32 bits
  if (int64_t(B) * Hq * ((int64_t(L) + 31) / 32) > (int64_t(1) << 31)) return FA_ERR_OVERFLOW;
  return FA_OK;
}

// Workgroup shape of the query-major kernels: wq waves along the sequence x wh waves along the
// heads, each wave 32 rows x hpw heads (hpw <= hmax); hpw * wh heads must divide the group size
// so that a workgroup never straddles two KV heads.  The forward shares each K/V fragment
// between two heads of a wave for D <= 64; the dQ kernel keeps one head per wave, which leaves
// it two waves per SIMD (measured faster at D = 64).
void choose_qmajor(int G, int hmax, int* hpw, int* wh, int* wq) {
  for (int h = hmax; h >= 1; --h)
    for (int w = 4; w >= 1; w /= 2)
      if (G % (h * w) == 0) {
        *hpw = h;
        *wh = w;
        *wq = 4 / w;
        return;
      }
  *hpw = 1;
  *wh = 1;
  *wq = 4;
}

struct SinkPlan {
  int nsp, n_chunks, srows;  // chunked blocks, chunks per block, stored sink rows per block
  int dq;                    // sink rows past block 0's window go through the dQ kernel
};

SinkPlan sink_plan(int L, int W, int S) {
  // clamp as the kernels do
  W = W < 0 ? 0 : (W > L ? L : W);
  S = S < 0 ? 0 : (S > L ? L : S);
  SinkPlan p{0, 0, 0, 0};
  p.nsp = fa::kv_sink_blocks(L, W, S);
  p.dq = fa::dq_sink_mode(L, W, S) ? 1 : 0;
  p.n_chunks = p.dq ? 0 : fa::kv_n_chunks(L, W, S, kChunkRows);
  p.srows = S < fa::kKvKeys ? S : fa::kKvKeys;
  return p;
}

// Tiles of the dQ kernel: row tiles of 32 * wq rows times head groups of wh heads (one query
// head per wave).
int64_t dq_tiles(int B, int Hq, int Hkv, int L) {
  int hpw, wh, wq;
  choose_qmajor(Hq / Hkv, 1, &hpw, &wh, &wq);
  const int64_t n_qtiles = (int64_t(L) + 32 * wq - 1) / (32 * wq);
  return n_qtiles * B * (Hq / wh);
}

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

// per-32-row-block partial sums of the learned sink logits' gradient: [B][Hq][Lp / 32] fp32
size_t dsink_part_bytes(int B, int Hq, int L) { return align256(size_t(B) * Hq * ((size_t(L) + 31) / 32) * sizeof(float)); }

// row statistics of the backward: [B][Hq][Lp / 32][lse * log2(e) x 32, -delta x 32] fp32
size_t delta_bytes(int B, int Hq, int L) {
  const size_t Lp = (size_t(L) + 31) / 32 * 32;
  return align256(size_t(B) * Hq * Lp * 2 * sizeof(float));
}

// fp32 partial sums of the sink rows: [B * Hkv][nsp][n_chunks + 1 slots][dK, dV][srows][D]
size_t partial_bytes(int B, int Hkv, int D, const SinkPlan& sp) {
  return align256(size_t(B) * Hkv * sp.nsp * (sp.n_chunks + 1) * 2 * sp.srows * D * sizeof(float));
}

// dq_sink_mode: the dQ kernel's flushed sink partials, [n_tiles][dK, dV][srows][D] fp32 (a slot
// per tile; a run of tiles writes the slot of its first tile)
size_t dq_sink_slot_bytes(int B, int Hq, int Hkv, int L, int D, const SinkPlan& sp) {
  return sp.dq ? align256(size_t(dq_tiles(B, Hq, Hkv, L)) * 2 * sp.srows * D * sizeof(float)) : 0;
}

// float32 backward: room for its sink-key partials, sized for 32-key tiles whose sink rows past the window
// are cut into chunks of 256 rows, [B * Hkv][tiles][chunks + 1][dK, dV][32][D] fp32.  The kernel keeps
// [B * Hkv][chunks + 1][dK, dV][S][D] for chunks of f32_chunk_rows rows laid out from its 64-key
// blocks' window ends, which is never more.
constexpr int kF32ChunkRows = 256;
struct F32Plan {
  int n_kt, nsp, n_chunks;
};
F32Plan f32_plan(int L, int W, int S) {
  W = W < 0 ? 0 : (W > L ? L : W);
  S = S < 0 ? 0 : (S > L ? L : S);
  F32Plan p;
  p.n_kt = (L + 31) / 32;
  const int row_end0 = fa::imin(L, 31 + fa::imax(W, 1));  // tile 0's window rows end first
  p.n_chunks = (S > 0 && row_end0 < L) ? (L - row_end0 + kF32ChunkRows - 1) / kF32ChunkRows : 0;
  p.nsp = p.n_chunks > 0 ? (S + 31) / 32 : 0;
  return p;
}
// Rows per sink-chunk workgroup of the float32 dK/dV kernel: 64, so that short workgroups even out the
// end of the launch (c2's backward with chunks of 64 / 128 / 256 rows: 502 / 509 / 596 us), or as few
// more as the room for partials needs.
int f32_chunk_rows(int L, int W, int S) {
  const F32Plan fp = f32_plan(L, W, S);
  int rows = 64;
  while (rows < kF32ChunkRows &&
         int64_t(fa::kv_n_chunks(L, W, S, rows) + 1) * S > int64_t(fp.n_chunks + 1) * 32 * fp.nsp)
    rows *= 2;
  return rows;
}
size_t f32_partial_bytes(int B, int Hkv, int D, const F32Plan& fp) {
  return align256(size_t(B) * Hkv * fp.nsp * (fp.n_chunks + 1) * 2 * 32 * D * sizeof(float));
}
// The workspace after the row statistics and the learned-sink partials: the sink-key partials
// and dQ-kernel slots of the 16-bit backward, or the float32 backward's partials (whichever is
// larger, so one size serves every dtype).
size_t partial_region_bytes(int B, int Hq, int Hkv, int L, int D, int W, int S) {
  const SinkPlan sp = sink_plan(L, W, S);
  const size_t b16 = partial_bytes(B, Hkv, D, sp) + dq_sink_slot_bytes(B, Hq, Hkv, L, D, sp);
  const size_t b32 = f32_partial_bytes(B, Hkv, D, f32_plan(L, W, S));
  return b16 > b32 ? b16 : b32;
}

void copy3(int64_t dst[3], const int64_t src[3]) {
  for (int i = 0; i < 3; ++i) dst[i] = src[i];
}

// Tiles per unit (slide_ct) of the sliding kernels, for `slots` resident units.  A fixed-length
// batch spreads its B Hkv (G / 8) n_qt tiles evenly over the slots.  A packed batch holds at most
// T = ceil(token_rows / 32) + B tiles with rows (each sequence adds at most one partial tile),
// however long its longest sequence (which sets n_qt); units past a short sequence's end exit at
// once.  Its units cut every sequence separately, so a (KV head, head group of 8) needs about
// T / ct + B / 2 units (half a unit lost per sequence on average), and ct is raised until those
// fit the slots: units that spill into a second round would double the kernel's time.
int slide_units_ct(const fa::Args& a, int64_t slots) {
  const int64_t n_qt = (int64_t(a.L) + 31) / 32;
  const int64_t hg = int64_t(a.Hkv) * (a.G / 8);
  int64_t tiles = int64_t(a.B) * n_qt;
  if (a.cu_seqlens) tiles = std::min(tiles, (int64_t(a.token_rows) + 31) / 32 + a.B);
  int64_t ct = (hg * tiles + slots - 1) / slots;
  if (a.cu_seqlens) {
    const int64_t per_group = slots / hg - a.B / 2;
    if (per_group >= 1) ct = std::max(ct, (tiles + per_group - 1) / per_group);
  }
  return int(std::max<int64_t>(ct, 1));
}

// Packed batches, the sliding kernels: units per (KV head, head group) that the sequences' rows can
// fill -- sequence b needs ceil(ceil(L_b / 32) / ct) <= L_b / (32 ct) + 1 units, so at most
// ceil(token_rows / (32 ct)) + B in all -- when fewer than B x slide_ncu (see fa::Args); 0 for a
// fixed-length batch.
int vl_units(const fa::Args& a) {
  if (!a.cu_seqlens) return 0;
  const int64_t rows_ct = 32 * int64_t(a.slide_ct);
  const int64_t bound = (int64_t(a.token_rows) + rows_ct - 1) / rows_ct + a.B;
  return bound < int64_t(a.B) * a.slide_ncu ? int(bound) : 0;
}

// The sliding dQ kernel (fa_bwd_slide.hip) serves D = 64 16-bit backwards whose KV groups hold a
// multiple of 8 query heads, with a window of 1..161 keys (at most 6 key halves of 32 in LDS) and
// at most 32 sink keys (one sink half).  Its workgroups take slide_ct consecutive 32-row tiles,
// sized so that the units with rows about fill the device once.  (Any slide_ct >= 1 fits the
// workspace: the units, B Hkv (G / 8) slide_ncu, never exceed half of bwd_dq_kernel's tiles, for
// which the dQ sink slots are sized.)
void plan_slide(fa::Args& a, int D) {
  if (D != 64 || a.G % 8 != 0 || a.W < 1 || a.W > fa::kSlideMaxW || a.S > 32 || a.L < 1) return;
  const int64_t n_qt = (int64_t(a.L) + 31) / 32;
  const int64_t ct = slide_units_ct(a, fa::device_cus());
  a.dq_slide = 1;
  a.slide_ct = int(ct);
  a.slide_ncu = int((n_qt + ct - 1) / ct);
  a.vl_units = vl_units(a);
}

// The sliding forward (fa_fwd.hip fwd_slide_kernel): the same shapes with W <= 129; two
// workgroups per CU.  Returns whether it applies (then slide_ct / slide_ncu are set).
bool plan_fwd_slide(fa::Args& a, int D, int dtype) {
  if (dtype == FA_DTYPE_F32 || D != 64 || a.G % 8 != 0 || a.W < 1 || a.W > fa::kFwdSlideMaxW || a.S > 32 ||
      a.L < 1)
    return false;
  const int64_t n_qt = (int64_t(a.L) + 31) / 32;
  const int64_t ct = slide_units_ct(a, 2 * int64_t(fa::device_cus()));
  a.slide_ct = int(ct);
  a.slide_ncu = int((n_qt + ct - 1) / ct);
  a.vl_units = vl_units(a);
  return true;
}

// Packed batches, the dK/dV kernel: key blocks per KV head that the sequences' keys can fill
// (each sequence adds at most one partial block), when fewer than B x n_kblocks (see fa::Args).
int vl_kblocks(const fa::Args& a) {
  if (!a.cu_seqlens) return 0;
  const int64_t bound = (int64_t(a.token_rows) + fa::kKvKeys - 1) / fa::kKvKeys + a.B;
  return bound < int64_t(a.B) * a.n_kblocks ? int(bound) : 0;
}

// Steps (pairs of 32-row blocks, times query heads) that the dK/dV kernel's workgroups of one (batch,
// KV head) sweep: the longest workgroup's and all of them.  Blocks whose window ends inside the
// sequence all sweep the same rows; the others sweep to the last row, one pair fewer per block.
struct KvSteps {
  double longest, total;
};
KvSteps kv_steps(double L, double W, double G) {
  const double n_kb = std::ceil(L / fa::kKvKeys);
  const double win = std::ceil((fa::kKvKeys - 1 + W) / 64.);  // pairs of a whole window
  const double n_win = std::min(n_kb, std::max(0., std::floor((L - W + 1) / fa::kKvKeys)));
  const double r = n_kb - n_win;
  return KvSteps{G * (n_win > 0 ? win : n_kb), G * (n_win * win + r * (r + 1) / 2)};
}

// Pieces per key block of the dK/dV kernel (1: unsplit) for `nseq` sequences of L rows on average and
// max_L at most on `cus` compute units: the power of two up to 32 with the least estimated time.  The kernel takes as long as its
// longest workgroup (a full causal layer's key block 0 sweeps every row, twice the average), or as
// the average work of a resident slot where that is more, or half of each, at the rate of full slots,
// where the longest starts on a full chip; splitting shortens the first, and costs
// writing and reading the pieces' fp32 sums, the launch that adds them, and the sink fold's launch
// where the dK/dV kernel would have folded (`folds`).  Measured on MI355X, in us a step: longest
// workgroups 0.55 / 0.58 / 0.8 / 1.15 at D = 16 / 32 / 64 / 128, full slots 1.3 / 1.5 / 1.14 / 1.25;
// 5 us a launch, 0.35 us per MB of sums.  Full causal D = 64, Hq = 64, Hkv = 8, dK/dV in us by pieces
// 1 / 2 / 4 / 8 / 16: L = 1024 106 / 61 / 41 / 39 / 50; L = 2048 207 / 122 / 90 / 101 / 124; L = 4096
// 434 / 298 / 302 / 321 / 386; L = 8192 1137 / 1125 / 1140 / 1198 / 1339; Hq = 8, Hkv = 1, L = 2048
// 202 / 106 / 59 / 38 / 31; D = 128, Hq = 32, Hkv = 8, L = 2048 149 / 102 / 113 / 142 / 220; with a
// window of 1024 at L = 4096 (equal workgroups) 143 / 154 / 162 / 177 / 245.
// The float32 kernel (the last four of each table): L = 2048, Hq = 64, Hkv = 8, D = 64 by pieces 1 / 2 / 4 /
// 8 / 16 1260 / 849 / 650 / 603 / 644; D = 128, Hq = 16, Hkv = 8 610 / 361 / 377 / 431 / 536.
int kv_split_pieces(bool f32, int D, int G, int Hkv, double nseq, double L, double max_L, double W, bool folds,
                    int cus) {
  const int i = (D == 16 ? 0 : D == 32 ? 1 : D == 64 ? 2 : 3) + (f32 ? 4 : 0);
  const double t_long[8] = {0.55, 0.58, 0.8, 1.15, 2.9, 2.9, 4.9, 9.3};
  const double t_slot[8] = {1.3, 1.5, 1.14, 1.25, 6.5, 6.5, 8.8, 9.6};
  const int per_cu[8] = {4, 4, 2, 1, 4, 3, 2, 1};  // resident workgroups
  const KvSteps st{kv_steps(max_L, W, G).longest, kv_steps(L, W, G).total};
  const double slot = t_slot[i] * st.total * nseq * Hkv / (double(cus) * per_cu[i]);
  const double mb = nseq * Hkv * std::ceil(L / fa::kKvKeys) * fa::kKvKeys * (D < 32 ? 32 : D) * 8 * 1e-6;  // per piece
  auto kernel_us = [&](double longest) {
    return std::max({t_long[i] * longest, slot, 0.5 * (slot + t_slot[i] * longest)});
  };
  int best = 1;
  double best_t = kernel_us(st.longest);
  for (int ns = 2; ns <= 32 && ns <= st.longest; ns *= 2) {
    const double t = kernel_us(st.longest / ns) + 5 + 0.35 * mb * ns + (folds ? 5 : 0);
    if (t < 0.95 * best_t) {
      best = ns;
      best_t = t;
    }
  }
  return best;
}

// bytes of kv_part for `blocks` key blocks (of every KV head) in `ns` pieces
size_t kv_part_bytes(int D, int64_t blocks, int ns) {
  return ns > 1 ? align256(size_t(blocks) * ns * 2 * fa::kKvKeys * (D < 32 ? 32 : D) * sizeof(float)) : 0;
}

// key blocks of every KV head that the dK/dV kernel's grid holds
int64_t kv_blocks(const fa::Args& a) {
  return int64_t(a.Hkv) * (a.vl_kblocks ? a.vl_kblocks : int64_t(a.B) * a.n_kblocks);
}

// Splits the dK/dV kernel (kv_split, kv_part) as far as the `spare` bytes of workspace at `ws` allow.
// The rows of a packed batch are taken to be spread evenly over its sequences (the host does not
// know their lengths).
void plan_kv_split(fa::Args& a, int D, bool f32, char* ws, size_t spare) {
  a.kv_split = 1;
  const int cus = fa::device_cus();
  if (!f32 && fa::dkdv4_eligible(a, D, cus)) return;
  const double rows = a.cu_seqlens ? std::min(double(a.L), std::max(1., double(a.token_rows) / a.B)) : double(a.L);
  int ns = kv_split_pieces(f32, D, a.G, a.Hkv, a.B, rows, a.L, a.W, a.sink_dq != 0, cus);
  const int64_t blocks = kv_blocks(a);
  // (the fold has up to 8 workgroups per block)
  while (ns > 1 && (kv_part_bytes(D, blocks, ns) > spare || blocks * std::max(ns, 8) > fa::kRangeWgs)) ns /= 2;
  a.kv_split = ns;
  a.kv_part = reinterpret_cast<float*>(ws);
}

// The query-major kernels with one tile per workgroup (fwd_split_kernel, bwd_dq_split_kernel): how many
// waves share a tile's keys, KSP = 1, 2 or 4 (wq, wh and n_qtiles are set).  The least estimated time, as
// for the dK/dV split: the longest tile alone on its CU, or the average work of a resident slot plus part
// of the longest tile's excess, and each workgroup's fixed time (its rows, the first keys, the merge).
struct SplitCost {
  int per_cu;          // resident workgroups (0: not built)
  double alone, full;  // us per step of a workgroup, alone on its CU and with full slots
};
int plan_split(fa::Args& a, int hpw, const SplitCost (&costs)[3], const double (&fixed)[3], double per_wg) {
  const double rows = a.cu_seqlens ? std::min(double(a.L), std::max(1., double(a.token_rows) / a.B)) : double(a.L);
  const int cus = fa::device_cus();
  // steps of one head set's tiles over `n` rows in tiles of 32 wq, for `ksp` waves on a tile's halves
  auto steps = [&](double n, int wq, int ksp, double* longest) {
    const double nt = std::ceil(n / (32 * wq));
    const double n1 = std::min(nt, std::floor((a.W - 1) / (32. * wq)) + 1);  // tiles that see key 0's half
    const double win = std::ceil((wq + std::ceil((a.W - 1) / 32.) + std::ceil(std::min(a.S, 64) / 32.)) / ksp);
    *longest = std::max(std::ceil(n1 * wq / ksp), nt > n1 ? win : 0.);
    return n1 * (n1 + 1) / 2 * wq / ksp + n1 * (ksp - 1) / (2. * ksp) + (nt - n1) * win;
  };
  int best = 0, best_wh = 0;
  double best_t = 0;
  for (int k = 0; k < 3; ++k) {
    const SplitCost& c = costs[k];
    if (!c.per_cu) continue;
    const int ksp = 1 << k;
    int wh = 4 / ksp;
    while (a.G % (hpw * wh) != 0) wh /= 2;
    const int wq = 4 / ksp / wh;
    const double streams = double(a.B) * (a.Hq / (hpw * wh)), slots = double(cus) * c.per_cu;
    double longest;
    const double slot = c.full * streams * steps(rows, wq, ksp, &longest) / slots;
    steps(a.L, wq, ksp, &longest);  // (a packed batch's longest sequence)
    const double wgs = streams * std::ceil(rows / (32 * wq));
    const double t = std::max(c.alone * longest, slot + 0.3 * std::max(0., c.full * longest - slot)) + fixed[k] +
                     per_wg * wgs / slots;
    if (!best || t < 0.97 * best_t) {
      best = ksp;
      best_wh = wh;
      best_t = t;
    }
  }
  a.wh = best_wh;
  a.wq = 4 / best / best_wh;
  a.n_qtiles = (a.L + 32 * a.wq - 1) / (32 * a.wq);
  return best;
}

// The 16-bit forward: KSP, or 0 for fwd_kernel.  The costs are measured over Hq = 8 .. 64, G = 1 .. 16,
// L = 257 .. 8192, W = 128 .. full (fwd_split_kernel's comment has the D = 64 figures; G = 1, Hq = 16,
// L = 4096 full causal: D = 64 81 / 60 / 74 for 1 / 2 / 4 waves against 88 for fwd_kernel, D = 16 at
// L = 2048 34 / 20 / 14 against 27).
// fwd_kernel keeps what it still does better: D <= 32 with one head per wave and short windows, whose
// tiles' key blocks it fetches at once (the D = 16, W = 256 default case 10.9 against 12.2 us), and D = 128
// with odd KV groups (one head per group, B = 2, Hq = 32, L = 2048 full causal 81.5 against 85 us) or with
// two rounds and more of workgroups that keep one wave per tile over long rows of equal length (B = 2, Hq = 64, Hkv = 8,
// L = 16384: W = 1024 1335 against 1376, full causal 9003 against 9309; Hq = 32, L = 4096, W = 400 46.7
// against 48.4; but W = 64 366 against 349 and 28.4 against 27.3, and one round, Hq = 64, L = 1024 full
// causal 38 against 32; sequences of 1536, 1187, 640 and 933 rows, Hq = 32, Hkv = 8, full causal 100 against 60).
int plan_fwd_split(fa::Args& a, int D, int hpw) {
  static const SplitCost costs[4][2][3] = {
      // [D][heads per wave - 1][KSP = 1, 2, 4]
      {{{7, 0.47, 1.5}, {7, 0.5, 1.5}, {7, 0.6, 1.55}}, {{4, 0.5, 1.3}, {4, 0.6, 1.4}, {4, 0.75, 1.5}}},
      {{{5, 0.5, 1.6}, {5, 0.6, 1.6}, {4, 0.8, 1.4}}, {{4, 0.63, 1.6}, {4, 0.77, 1.6}, {4, 1.0, 1.8}}},
      {{{4, 0.56, 1.34}, {4, 0.7, 1.38}, {2, 0.9, 1.15}}, {{3, 0.75, 1.57}, {3, 0.85, 1.72}, {2, 1.1, 1.43}}},
      {{{2, 0.83, 1.04}, {2, 1.2, 1.3}, {0, 0, 0}}, {{0, 0, 0}, {0, 0, 0}, {0, 0, 0}}}};
  const double fixed[3] = {3, D == 64 ? 4.5 : 3.5, 3};
  if (D <= 32 && hpw == 1 && a.W <= 320) return 0;
  if (D == 128 && a.G % 2 != 0) return 0;
  const fa::Args given = a;
  const int ksp = plan_split(a, hpw, costs[D == 16 ? 0 : D == 32 ? 1 : D == 64 ? 2 : 3][hpw - 1], fixed, hpw == 2 ? 4. : 3.);
  if (D == 128 && ksp == 1 && a.W >= 192 && !a.cu_seqlens) {
    if (int64_t(a.B) * a.L * (a.Hq / a.wh) >= int64_t(32) * a.wq * 2 * 2 * fa::device_cus()) {  // (two fit a CU)
      a = given;
      return 0;
    }
  }
  return ksp;
}

// The 16-bit dQ: KSP, or 0 for the sliding kernel's shapes and for bwd_dq_kernel, which keeps the shapes
// whose sink keys' gradients it adds up (sink_dq) and short windows at D <= 32 (D = 16, L = 4096, W = 256,
// Hq = 16: 10.0 against 11.5 us).  Costs measured as the forward's; bwd_dq_split_kernel's comment has figures.
int plan_dq_split(fa::Args& a, int D) {
  static const SplitCost costs[4][3] = {{{5, 0.42, 0.98}, {5, 0.46, 1.0}, {5, 0.6, 1.05}},
                                        {{4, 0.41, 0.93}, {4, 0.57, 1.0}, {4, 0.8, 1.15}},
                                        {{3, 0.6, 1.115}, {3, 0.75, 1.25}, {2, 1.0, 1.06}},
                                        {{2, 1.05, 1.42}, {2, 1.4, 1.56}, {0, 0, 0}}};
  const double fixed[3] = {4, 4, 4};
  if (a.sink_dq || a.dq_slide || (D <= 32 && a.W <= 320)) return 0;
  return plan_split(a, 1, costs[D == 16 ? 0 : D == 32 ? 1 : D == 64 ? 2 : 3], fixed, D <= 32 ? 3. : 4.);
}

// Where dq_sink_mode's shapes rather have the dK/dV kernel's chunk workgroups add up the sink keys'
// gradients: rows per chunk, or 0 for the dQ kernel.  A row outside key block 0's window then costs the
// dK/dV grid one short step per head, but the dQ kernel is bwd_dq_split_kernel, which holds no sink sums
// and is faster per window step -- the more so the longer the window.  Whole backward in us, dQ kernel ->
// chunks: D = 128, B = 8, Hq = 32, Hkv = 4, L = 2048, S = 16: W = 512 707 -> 649, W = 256 504 -> 456;
// B = 1, Hq = 32, Hkv = 8, L = 4096, S = 4: W = 1024 294 -> 276, W = 256 127 -> 126, but W = 128
// 102 -> 106.  D = 64, Hq = 64, Hkv = 8, L = 4096, S = 4: W = 1024 265 -> 254, but W = 512 157 -> 158.
// With few heads per group a chunk has too little work (D = 64, Hq = 16, L = 4096, W = 1024: G = 1 80 -> 88,
// G = 2 with B = 2 156.8 -> 157.7), and D <= 32 does not gain below W = 2048.  The chunks' sums lie in the room that the dQ kernel's slots have
// (a slot per 32 rows and head set: more than a chunk's, checked all the same).
int sinks_by_chunks(const fa::Args& a, int D, const SinkPlan& sp) {
  if (!sp.dq || a.G < 2) return 0;
  const int rows = D == 128 && a.W >= 256 ? 128 : D == 64 && a.W >= 1024 && a.G >= 4 ? 64 : 0;
  if (!rows) return 0;
  SinkPlan c = sp;
  c.n_chunks = fa::kv_n_chunks(a.L, a.W, a.S, rows);
  // (the dQ kernel's grid is bounded; a dK/dV launch with a chunk per B x longest sequence need not fit one grid)
  if (int64_t(a.B) * a.Hkv * c.n_chunks >= fa::kRangeWgs) return 0;
  const size_t room = partial_bytes(a.B, a.Hkv, D, sp) + dq_sink_slot_bytes(a.B, a.Hq, a.Hkv, a.L, D, sp);
  return partial_bytes(a.B, a.Hkv, D, c) <= room ? rows : 0;
}

// The kernel arguments that describe the dK/dV kernel's key blocks and sink chunks.
void set_kv_plan(fa::Args* a, int D, bool f32) {
  a->n_kblocks = (a->L + fa::kKvKeys - 1) / fa::kKvKeys;
  const SinkPlan sp = sink_plan(a->L, a->W, a->S);
  a->nsp = sp.nsp;
  if (f32) {
    a->chunk_rows = f32_chunk_rows(a->L, a->W, a->S);
    a->n_chunks = fa::kv_n_chunks(a->L, a->W, a->S, a->chunk_rows);
  } else {
    const int rows = sinks_by_chunks(*a, D, sp);
    a->sink_dq = sp.dq && !rows;
    a->chunk_rows = rows ? rows : kChunkRows;
    a->n_chunks = a->sink_dq ? 0 : fa::kv_n_chunks(a->L, a->W, a->S, a->chunk_rows);
    a->srows = sp.srows;
  }
  a->n_chunk_wgs = a->B * a->Hkv * a->nsp * a->n_chunks;
}

fa::Args base_args(int32_t B, int32_t Hq, int32_t Hkv, int32_t L, int32_t D, int32_t W, int32_t S,
                   float scale) {
  fa::Args a;
  std::memset(&a, 0, sizeof(a));
  a.B = B;
  a.Hq = Hq;
  a.Hkv = Hkv;
  a.L = L;
  a.G = Hq / Hkv;
  a.Lp = (L + 31) / 32 * 32;
  a.W = W < 0 ? 0 : (W > L ? L : W);
  a.S = S < 0 ? 0 : (S > L ? L : S);
  a.scale = scale;
  float c = std::fabs(scale) * 1.4426950408889634f;
  // A zero scale gives the uniform softmax; a tiny positive factor keeps -inf * c well defined
  // and changes no fp32 result.
  if (c < 1e-30f) c = 1e-30f;
  a.c = c;
  a.qsign = scale < 0.f ? 0x80008000u : 0u;
  (void)D;
  return a;
}

}  // namespace

// Compute units of the current device (256 on MI355X; 256 if the query fails), looked up once per
// device: launches plan with it several times a call.
int fa::device_cus() {
  static std::atomic<int> known[64];
  int dev = 0, n = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0) return 256;
  if (dev < 64 && (n = known[dev].load(std::memory_order_relaxed)) > 0) return n;
  if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) return 256;
  if (dev < 64) known[dev].store(n, std::memory_order_relaxed);
  return n;
}

extern "C" {

int fa_check_fwd(const fa_fwd_params* p) {
  if (!p) return FA_ERR_NULL;
  if (!p->q || !p->k || !p->v || !p->o || !p->lse) return FA_ERR_NULL;
  const int rc = check_common(p->batch, p->heads_q, p->heads_kv, p->seqlen, p->head_dim, p->window,
                              p->sink, p->softmax_scale, p->dtype);
  if (rc != FA_OK) return rc;
  if (!aligned16(p->q) || !aligned16(p->k) || !aligned16(p->v) || !aligned16(p->o) || !aligned4(p->lse))
    return FA_ERR_ALIGN;
  const int eb = elem_bytes(p->dtype);
  if (!strides_ok(p->q_stride, eb) || !strides_ok(p->k_stride, eb) || !strides_ok(p->v_stride, eb) ||
      !strides_ok(p->o_stride, eb) || !lse_strides_ok(p->lse_stride))
    return FA_ERR_ALIGN;
  // q, k and v are staged through buffer resources with 32-bit byte offsets inside one
  // (batch, head) slice; o and lse are written through 64-bit addresses
  const int L = p->seqlen, D = p->head_dim;
  if (!slice_fits(p->q_stride, L, D, eb) || !slice_fits(p->k_stride, L, D, eb) || !slice_fits(p->v_stride, L, D, eb))
    return FA_ERR_OVERFLOW;
  return FA_OK;
}

int fa_check_bwd(const fa_bwd_params* p) {
  if (!p) return FA_ERR_NULL;
  if (!p->q || !p->k || !p->v || !p->o || !p->dout || !p->lse || !p->dq || !p->dk || !p->dv)
    return FA_ERR_NULL;
  const int rc = check_common(p->batch, p->heads_q, p->heads_kv, p->seqlen, p->head_dim, p->window,
                              p->sink, p->softmax_scale, p->dtype);
  if (rc != FA_OK) return rc;
  const void* ptrs[] = {p->q, p->k, p->v, p->o, p->dout, p->dq, p->dk, p->dv};
  for (const void* x : ptrs)
    if (!aligned16(x)) return FA_ERR_ALIGN;
  if (!aligned4(p->lse)) return FA_ERR_ALIGN;
  const int eb = elem_bytes(p->dtype);
  if (!strides_ok(p->q_stride, eb) || !strides_ok(p->k_stride, eb) || !strides_ok(p->v_stride, eb) ||
      !strides_ok(p->o_stride, eb) || !strides_ok(p->do_stride, eb) || !lse_strides_ok(p->lse_stride) ||
      !strides_ok(p->dq_stride, eb) || !strides_ok(p->dk_stride, eb) || !strides_ok(p->dv_stride, eb))
    return FA_ERR_ALIGN;
  // every input is read through buffer resources with 32-bit byte offsets inside one
  // (batch, head) slice; dq, dk and dv are written through 64-bit addresses
  const int L = p->seqlen, D = p->head_dim;
  if (!slice_fits(p->q_stride, L, D, eb) || !slice_fits(p->do_stride, L, D, eb) || !slice_fits(p->o_stride, L, D, eb) ||
      !slice_fits(p->lse_stride, L, 1, 4) || !slice_fits(p->k_stride, L, D, eb) || !slice_fits(p->v_stride, L, D, eb))
    return FA_ERR_OVERFLOW;
  return FA_OK;
}

}  // extern "C"

namespace {

// Variable-length batches: the sequences' rows lie in one row dimension, so the batch strides are unused.
// Without `lens` sequence b is rows [cu[b], cu[b + 1]), with it [cu[b], cu[b] + lens[b]).
struct Packed {
  const int32_t* cu;
  const int32_t* lens;
  int32_t total_rows, token_rows;
};

int check_varlen(const Packed& v) {
  if (!v.cu) return FA_ERR_NULL;
  if (!aligned4(v.cu) || !aligned4(v.lens)) return FA_ERR_ALIGN;
  if (v.total_rows < 0 || v.token_rows < 0 || v.token_rows > v.total_rows) return FA_ERR_SHAPE;
  return FA_OK;
}

void set_varlen(fa::Args* a, const Packed& v) {
  a->cu_seqlens = v.cu;
  a->seq_lens = v.lens;
  a->total_rows = v.total_rows;
  a->token_rows = v.token_rows;
  for (int64_t* st : {a->sq, a->sk, a->sv, a->so, a->sdo, a->slse, a->sdq, a->sdk, a->sdv, a->so_out}) st[0] = 0;
}

int run_fwd(const fa_fwd_params* p, const float* sinks, void* stream, const Packed* packed = nullptr) {
  fa::Args a = base_args(p->batch, p->heads_q, p->heads_kv, p->seqlen, p->head_dim, p->window, p->sink,
                         p->softmax_scale);
  a.q = p->q;
  a.k = p->k;
  a.v = p->v;
  a.o_out = p->o;
  a.lse_out = p->lse;
  a.sink_logits = sinks;
  copy3(a.sq, p->q_stride);
  copy3(a.sk, p->k_stride);
  copy3(a.sv, p->v_stride);
  copy3(a.so_out, p->o_stride);
  copy3(a.slse, p->lse_stride);
  if (packed) set_varlen(&a, *packed);
  if (plan_fwd_slide(a, p->head_dim, p->dtype))
    return fa::launch_fwd_slide(a, p->dtype, static_cast<hipStream_t>(stream)) == hipSuccess ? FA_OK : FA_ERR_LAUNCH;
  const bool f32 = p->dtype == FA_DTYPE_F32;
  int hpw, wh, wq;
  choose_qmajor(a.G, p->head_dim <= 64 && !f32 ? 2 : 1, &hpw, &wh, &wq);
  a.wh = wh;
  a.wq = wq;
  a.n_qtiles = (a.L + 32 * wq - 1) / (32 * wq);
  const hipStream_t s = static_cast<hipStream_t>(stream);
  hipError_t e;
  if (f32) {
    e = fa::launch_fwd_f32(a, p->head_dim, s);
  } else if (const int ksp = plan_fwd_split(a, p->head_dim, hpw)) {
    e = fa::launch_fwd_split(a, p->dtype, p->head_dim, hpw, ksp, s);
  } else {
    e = fa::launch_fwd(a, p->dtype, p->head_dim, s);
  }
  return e == hipSuccess ? FA_OK : FA_ERR_LAUNCH;
}

int fwd_packed(const fa_fwd_params* p, const Packed& v, const float* sinks, void* stream) {
  int rc = fa_check_fwd(p);
  if (rc == FA_OK) rc = check_varlen(v);
  if (rc != FA_OK) return rc;
  if (sinks && !aligned4(sinks)) return FA_ERR_ALIGN;
  return run_fwd(p, sinks, stream, &v);  // (rows outside every sequence: o = 0, lse = -inf, see fa_aux.h)
}

// fa_fwd_fp8: e4m3 q, k, v (1-byte elements), bf16 o, D in {64, 128}, finite dequantisation factors.
int check_fwd_fp8(const fa_fwd_params* p, float qd, float kd, float vd) {
  if (!p) return FA_ERR_NULL;
  if (!p->q || !p->k || !p->v || !p->o || !p->lse) return FA_ERR_NULL;
  if (p->dtype != FA_DTYPE_FP8_E4M3) return FA_ERR_DTYPE;
  const int rc = check_common(p->batch, p->heads_q, p->heads_kv, p->seqlen, p->head_dim, p->window, p->sink,
                              p->softmax_scale, FA_DTYPE_BF16);
  if (rc != FA_OK) return rc;
  if (p->head_dim != 64 && p->head_dim != 128) return FA_ERR_HEAD_DIM;
  if (!std::isfinite(qd) || !std::isfinite(kd) || !std::isfinite(vd) || !std::isfinite(p->softmax_scale * qd * kd))
    return FA_ERR_SCALE;
  if (!aligned16(p->q) || !aligned16(p->k) || !aligned16(p->v) || !aligned16(p->o) || !aligned4(p->lse))
    return FA_ERR_ALIGN;
  if (!strides_ok(p->q_stride, 1) || !strides_ok(p->k_stride, 1) || !strides_ok(p->v_stride, 1) ||
      !strides_ok(p->o_stride) || !lse_strides_ok(p->lse_stride))
    return FA_ERR_ALIGN;
  const int L = p->seqlen, D = p->head_dim;
  if (!slice_fits(p->q_stride, L, D, 1) || !slice_fits(p->k_stride, L, D, 1) || !slice_fits(p->v_stride, L, D, 1))
    return FA_ERR_OVERFLOW;
  return FA_OK;
}

// The scores are (q_descale k_descale scale) * (q . k) over the stored e4m3 values; O is scaled
// by v_descale in the kernel's epilogue.
int run_fwd_fp8(const fa_fwd_params* p, float qd, float kd, float vd, const float* sinks, bool fp8_pv,
                void* stream) {
  const float scale = p->softmax_scale * qd * kd;
  fa::Args a = base_args(p->batch, p->heads_q, p->heads_kv, p->seqlen, p->head_dim, p->window, p->sink, scale);
  a.qsign = scale < 0.f ? 0x80808080u : 0u;
  a.oscale = vd;
  a.q = p->q;
  a.k = p->k;
  a.v = p->v;
  a.o_out = p->o;
  a.lse_out = p->lse;
  a.sink_logits = sinks;
  copy3(a.sq, p->q_stride);
  copy3(a.sk, p->k_stride);
  copy3(a.sv, p->v_stride);
  copy3(a.so_out, p->o_stride);
  copy3(a.slse, p->lse_stride);
  int hpw, wh, wq;
  choose_qmajor(a.G, p->head_dim == 64 ? 2 : 1, &hpw, &wh, &wq);
  a.wh = wh;
  a.wq = wq;
  a.n_qtiles = (a.L + 32 * wq - 1) / (32 * wq);
  const hipError_t e = fa::launch_fwd_fp8(a, p->head_dim, hpw, fp8_pv, static_cast<hipStream_t>(stream));
  return e == hipSuccess ? FA_OK : FA_ERR_LAUNCH;
}

}  // namespace

extern "C" {

int fa_fwd(const fa_fwd_params* p, void* stream) {
  const int rc = fa_check_fwd(p);
  return rc != FA_OK ? rc : run_fwd(p, nullptr, stream);
}

int fa_fwd_varlen(const fa_fwd_params* p, const int32_t* cu_seqlens, int32_t total_rows, const float* sinks,
                  void* stream) {
  return fwd_packed(p, Packed{cu_seqlens, nullptr, total_rows, total_rows}, sinks, stream);
}

int fa_fwd_ranges(const fa_fwd_params* p, const int32_t* starts, const int32_t* lens, int32_t total_rows,
                  int32_t token_rows, const float* sinks, void* stream) {
  const int rc = fa_check_fwd(p);
  if (rc != FA_OK) return rc;
  return lens ? fwd_packed(p, Packed{starts, lens, total_rows, token_rows}, sinks, stream) : FA_ERR_NULL;
}

int fa_fwd_fp8(const fa_fwd_params* p, float q_descale, float k_descale, float v_descale, const float* sinks,
               void* stream) {
  const int rc = check_fwd_fp8(p, q_descale, k_descale, v_descale);
  if (rc != FA_OK) return rc;
  if (sinks && !aligned4(sinks)) return FA_ERR_ALIGN;
  return run_fwd_fp8(p, q_descale, k_descale, v_descale, sinks, false, stream);
}

int fa_fwd_fp8_pv(const fa_fwd_params* p, float q_descale, float k_descale, float v_descale, const float* sinks,
                  void* stream) {
  const int rc = check_fwd_fp8(p, q_descale, k_descale, v_descale);
  if (rc != FA_OK) return rc;
  if (sinks && !aligned4(sinks)) return FA_ERR_ALIGN;
  return run_fwd_fp8(p, q_descale, k_descale, v_descale, sinks, true, stream);
}

int fa_fwd_sinks(const fa_fwd_params* p, const float* sinks, void* stream) {
  const int rc = fa_check_fwd(p);
  if (rc != FA_OK) return rc;
  if (!sinks) return FA_ERR_NULL;
  if (!aligned4(sinks)) return FA_ERR_ALIGN;
  return run_fwd(p, sinks, stream);
}

size_t fa_bwd_workspace_bytes(int32_t batch, int32_t heads_q, int32_t heads_kv, int32_t seqlen,
                              int32_t head_dim, int32_t window, int32_t sink) {
  if (check_common(batch, heads_q, heads_kv, seqlen, head_dim, window, sink, 1.f, FA_DTYPE_BF16) != FA_OK)
    return 0;
  return delta_bytes(batch, heads_q, seqlen) + dsink_part_bytes(batch, heads_q, seqlen) +
         partial_region_bytes(batch, heads_q, heads_kv, seqlen, head_dim, window, sink);
}

size_t fa_bwd_full_workspace_bytes(int32_t batch, int32_t heads_q, int32_t heads_kv, int32_t seqlen, int32_t head_dim,
                                   int32_t window, int32_t sink, int32_t dtype, int32_t total_rows) {
  const size_t need = fa_bwd_workspace_bytes(batch, heads_q, heads_kv, seqlen, head_dim, window, sink);
  if (need == 0) return 0;
  const bool f32 = dtype == FA_DTYPE_F32;
  fa::Args a = base_args(batch, heads_q, heads_kv, seqlen, head_dim, window, sink, 1.f);
  set_kv_plan(&a, head_dim, f32);
  if (total_rows >= 0) {
    a.cu_seqlens = &total_rows;  // (only whether there are offsets matters to the plan)
    a.token_rows = total_rows;
    a.vl_kblocks = vl_kblocks(a);
  }
  plan_kv_split(a, head_dim, f32, nullptr, SIZE_MAX);
  return need + kv_part_bytes(head_dim, kv_blocks(a), a.kv_split);
}

}  // extern "C"

namespace {

// Validates a backward call and fills the kernel arguments; returns FA_OK or an fa_status.
// packed: a packed batch (checked by the caller).
int prepare_bwd(const fa_bwd_params* p, void* workspace, size_t workspace_bytes, fa::Args* out, int* hpw,
                const Packed* packed = nullptr) {
  const int rc = fa_check_bwd(p);
  if (rc != FA_OK) return rc;
  const size_t need = fa_bwd_workspace_bytes(p->batch, p->heads_q, p->heads_kv, p->seqlen, p->head_dim,
                                             p->window, p->sink);
  if (!workspace || workspace_bytes < need || (reinterpret_cast<uintptr_t>(workspace) & 255u) != 0)
    return FA_ERR_WORKSPACE;
  fa::Args a = base_args(p->batch, p->heads_q, p->heads_kv, p->seqlen, p->head_dim, p->window, p->sink,
                         p->softmax_scale);
  a.q = p->q;
  a.k = p->k;
  a.v = p->v;
  a.o = p->o;
  a.dout = p->dout;
  a.lse = p->lse;
  a.dq = p->dq;
  a.dk = p->dk;
  a.dv = p->dv;
  copy3(a.sq, p->q_stride);
  copy3(a.sk, p->k_stride);
  copy3(a.sv, p->v_stride);
  copy3(a.so, p->o_stride);
  copy3(a.sdo, p->do_stride);
  copy3(a.slse, p->lse_stride);
  copy3(a.sdq, p->dq_stride);
  copy3(a.sdk, p->dk_stride);
  copy3(a.sdv, p->dv_stride);
  a.delta = static_cast<float*>(workspace);

  int wh, wq;
  choose_qmajor(a.G, 1, hpw, &wh, &wq);
  a.wh = wh;
  a.wq = wq;
  a.n_qtiles = (a.L + 32 * wq - 1) / (32 * wq);

  // workspace: row statistics | learned-sink partials | partial region (see partial_region_bytes)
  char* ws = static_cast<char*>(workspace);
  const size_t off_dsink = delta_bytes(a.B, a.Hq, a.L);
  a.dsink_part = reinterpret_cast<float*>(ws + off_dsink);
  a.partial = reinterpret_cast<float*>(ws + off_dsink + dsink_part_bytes(a.B, a.Hq, a.L));
  const bool f32 = p->dtype == FA_DTYPE_F32;
  set_kv_plan(&a, p->head_dim, f32);
  if (a.sink_dq)
    a.dq_sink_part = a.partial + partial_bytes(a.B, a.Hkv, p->head_dim, sink_plan(a.L, a.W, a.S)) / sizeof(float);
  if (packed) {
    set_varlen(&a, *packed);
    a.vl_kblocks = vl_kblocks(a);
  }
  if (!f32) plan_slide(a, p->head_dim);
  plan_kv_split(a, p->head_dim, f32, ws + need, workspace_bytes - need);
  *out = a;
  return FA_OK;
}

int run_dq(const fa::Args& a, const fa_bwd_params* p, int hpw, hipStream_t s) {
  fa::Args d = a;  // (the tiles of fa_bwd_dq.hip are not those that the sink fold enumerates)
  const int ksp = p->dtype == FA_DTYPE_F32 ? 0 : plan_dq_split(d, p->head_dim);
  const hipError_t e = p->dtype == FA_DTYPE_F32 ? fa::launch_bwd_dq_f32(a, p->head_dim, s)
                       : ksp                ? fa::launch_bwd_dq_split(d, p->dtype, p->head_dim, ksp, s)
                       : a.dq_slide         ? fa::launch_bwd_dq_slide(a, p->dtype, s)
                                            : fa::launch_bwd_dq(a, p->dtype, p->head_dim, hpw, s);
  return e == hipSuccess ? FA_OK : FA_ERR_LAUNCH;
}

int run_dkdv(const fa::Args& a, const fa_bwd_params* p, hipStream_t s) {
  const hipError_t e = p->dtype == FA_DTYPE_F32 ? fa::launch_bwd_dkdv_f32(a, p->head_dim, s)
                                                : fa::launch_bwd_dkdv(a, p->dtype, p->head_dim, s);
  return e == hipSuccess ? FA_OK : FA_ERR_LAUNCH;
}

int bwd_packed(const fa_bwd_params* p, const Packed& v, const float* sinks, float* dsinks, void* workspace,
               size_t workspace_bytes, void* stream) {
  fa::Args a;
  int hpw = 1;
  const int vrc = check_varlen(v);
  int rc = prepare_bwd(p, workspace, workspace_bytes, &a, &hpw, vrc == FA_OK ? &v : nullptr);
  if (rc == FA_OK) rc = vrc;
  if (rc != FA_OK) return rc;
  if (!sinks != !dsinks) return FA_ERR_NULL;
  if ((sinks && !aligned4(sinks)) || (dsinks && !aligned4(dsinks))) return FA_ERR_ALIGN;
  a.sink_logits = sinks;
  a.dsink = dsinks;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int r = run_dq(a, p, hpw, s);
  return r != FA_OK ? r : run_dkdv(a, p, s);  // (rows outside every sequence have zero gradients, see fa_aux.h)
}

}  // namespace

extern "C" {

int fa_bwd(const fa_bwd_params* p, void* workspace, size_t workspace_bytes, void* stream) {
  fa::Args a;
  int hpw = 1;
  const int rc = prepare_bwd(p, workspace, workspace_bytes, &a, &hpw);
  if (rc != FA_OK) return rc;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int r1 = run_dq(a, p, hpw, s);
  return r1 != FA_OK ? r1 : run_dkdv(a, p, s);
}

int fa_bwd_sinks(const fa_bwd_params* p, const float* sinks, float* dsinks, void* workspace, size_t workspace_bytes,
                 void* stream) {
  fa::Args a;
  int hpw = 1;
  const int rc = prepare_bwd(p, workspace, workspace_bytes, &a, &hpw);
  if (rc != FA_OK) return rc;
  if (!sinks || !dsinks) return FA_ERR_NULL;
  if (!aligned4(sinks) || !aligned4(dsinks)) return FA_ERR_ALIGN;
  a.sink_logits = sinks;
  a.dsink = dsinks;
  const hipStream_t s = static_cast<hipStream_t>(stream);
  const int r = run_dq(a, p, hpw, s);
  return r != FA_OK ? r : run_dkdv(a, p, s);
}

int fa_bwd_varlen(const fa_bwd_params* p, const int32_t* cu_seqlens, int32_t total_rows, const float* sinks,
                  float* dsinks, void* workspace, size_t workspace_bytes, void* stream) {
  return bwd_packed(p, Packed{cu_seqlens, nullptr, total_rows, total_rows}, sinks, dsinks, workspace, workspace_bytes,
                    stream);
}

int fa_bwd_ranges(const fa_bwd_params* p, const int32_t* starts, const int32_t* lens, int32_t total_rows,
                  int32_t token_rows, const float* sinks, float* dsinks, void* workspace, size_t workspace_bytes,
                  void* stream) {
  const int rc = fa_check_bwd(p);
  if (rc != FA_OK) return rc;
  if (!lens) return FA_ERR_NULL;
  return bwd_packed(p, Packed{starts, lens, total_rows, token_rows}, sinks, dsinks, workspace, workspace_bytes, stream);
}

int fa_bwd_dq(const fa_bwd_params* p, void* workspace, size_t workspace_bytes, void* stream) {
  fa::Args a;
  int hpw = 1;
  const int rc = prepare_bwd(p, workspace, workspace_bytes, &a, &hpw);
  return rc != FA_OK ? rc : run_dq(a, p, hpw, static_cast<hipStream_t>(stream));
}

int fa_bwd_dkdv(const fa_bwd_params* p, void* workspace, size_t workspace_bytes, void* stream) {
  fa::Args a;
  int hpw = 1;
  const int rc = prepare_bwd(p, workspace, workspace_bytes, &a, &hpw);
  return rc != FA_OK ? rc : run_dkdv(a, p, static_cast<hipStream_t>(stream));
}

const char* fa_strerror(int status) {
  switch (status) {
    case FA_OK: return "ok";
    case FA_ERR_NULL: return "a required pointer is NULL";
    case FA_ERR_SHAPE: return "invalid shape: batch, heads and seqlen must be >= 1 and heads_q % heads_kv == 0";
    case FA_ERR_HEAD_DIM: return "head_dim must be one of 16, 32, 64, 128 (64 or 128 for fa_fwd_fp8*)";
    case FA_ERR_DTYPE: return "dtype must be FA_DTYPE_BF16, FA_DTYPE_F16 or FA_DTYPE_F32 (FA_DTYPE_FP8_E4M3 for fa_fwd_fp8*)";
    case FA_ERR_ALIGN: return "tensors must be 16-byte aligned with non-negative strides that are multiples of 16 bytes (lse: 4-byte aligned, non-negative strides)";
    case FA_ERR_MASK: return "window < 1 and sink < 1 leave every query row fully masked";
    case FA_ERR_WORKSPACE: return "workspace is NULL, not 256-byte aligned or smaller than fa_bwd_workspace_bytes()";
    case FA_ERR_LAUNCH: return "HIP kernel launch failed";
    case FA_ERR_OVERFLOW: return "problem size exceeds the kernels' index range";
    case FA_ERR_SCALE: return "softmax_scale (and the fp8 dequantisation factors) must be finite";
    case FA_ERR_SCRATCH: return "the problem needs more backward workspace than the library's scratch buffer (FA_SCRATCH_BYTES) holds; use fa_bwd with a workspace";
  }
  return "unknown fa_status";
}

int fa_version(void) { return FA_GFX950_VERSION; }

}  // extern "C"
