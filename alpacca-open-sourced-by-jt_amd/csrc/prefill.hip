// Causal (optionally windowed) GQA prefill attention.
//
// fp16/bf16 with head_dim 64/128/256 (prefill_mfma): a flash-attention
// forward pass on v_mfma_f32_16x16x32_{f16,bf16}.  A block owns 16*NQB query
// columns per wave x 4 waves, where a column is one (token, query head) pair
// of one kv head's GQA group, so every K/V tile staged in LDS serves all the
// group's heads.  Per 64-key (32 for head_dim 256) tile each wave computes
// S^T = K Q^T (a lane owns one query column and 16 keys of each 16x16 block,
// so the softmax row max is local plus two xor shuffles), applies the causal
// mask only on tiles that straddle a row's diagonal, and accumulates
// O^T += V^T P^T with P taken straight from the score registers and V^T read
// from the row-major LDS tile with transposing reads.  K/V tiles are double
// buffered: the next tile's global loads are in flight while the current
// tile is multiplied.  One iteration's MFMA block holds PV of tile j - 1,
// the exp / convert work of tile j and QK of tile j + 1, at raised wave
// priority; the softmax max bookkeeping runs ahead of it (see grow_check).
// Tiles entirely above the diagonal are never loaded;
// tiles entirely above one wave's diagonal are skipped by that wave.  Blocks
// are mapped so that one kv head's blocks share one XCD (and its L2), with
// the latest (most expensive) column tiles launched first.  Chunks with few
// column tiles over many keys are cut along the keys as well
// (prefill_split.hip, plan_split_prefill).
//
// float32 chunks with the same head dims run prefill_f32 (prefill_f32.hip).
// Everything else (odd head dims, unaligned rows, a few float32 tokens) runs
// the split-K decode machinery in causal mode: query token t is a "sequence" whose
// visible rows are those at absolute positions <= pos0 + t (inside the
// window).
#include <math.h>
#include <string.h>

#include <algorithm>
#include <cmath>

#include "alpx_common.h"
#include "decode_internal.h"
#include "prefill_run.h"
#include "timing.h"

namespace alpx {
namespace {

template <typename T, typename TO, int D, int BK, int NQB, bool PAGED = false>
__global__ void __launch_bounds__(256, 2)
prefill_mfma(PrefillArgs a) {
  constexpr int kTileB = BK * D * (int)sizeof(T);
  constexpr int kCols = 64 * NQB;
  __shared__ __attribute__((aligned(1024))) char smem[4 * kTileB];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int kvh, ctile;
  if (!prefill_work(a, kvh, ctile)) return;
  // The heavy column tiles (late tokens, many key tiles) set the kernel's
  // end time, so of each tile and its mirror col_tiles - 1 - ctile the
  // lighter one copies both tiles' rows (each tile's rows exactly once).
  if (!PAGED && a.kn != nullptr) {
    const int mirror = a.col_tiles - 1 - ctile;
    if (ctile <= mirror) copy_tile_rows<T, D, kCols>(a, kvh, ctile, tid);
    if (ctile < mirror) copy_tile_rows<T, D, kCols>(a, kvh, mirror, tid);
  }
  auto bar = []() __attribute__((always_inline)) { __syncthreads(); };
  prefill_run<T, TO, D, BK, NQB, PAGED, kRunWrite, 4>(a, kvh, ctile, 0, -1, smem, nullptr,
                                                      nullptr, wave, tid, bar, wave, -1, false);
}

template <typename T, typename TO>
const void* pick_kernel(int D) {
  switch (D) {
    case 64: return (const void*)prefill_mfma<T, TO, 64, 64, 2>;
    case 128: return (const void*)prefill_mfma<T, TO, 128, 64, 2>;
    case 256: return (const void*)prefill_mfma<T, TO, 256, 32, 1>;
  }
  return nullptr;
}

// Paged caches: output in the cache dtype only.
template <typename T>
const void* pick_kernel_paged(int D) {
  switch (D) {
    case 64: return (const void*)prefill_mfma<T, T, 64, 64, 2, true>;
    case 128: return (const void*)prefill_mfma<T, T, 128, 64, 2, true>;
    case 256: return (const void*)prefill_mfma<T, T, 256, 32, 1, true>;
  }
  return nullptr;
}

template <typename T>
const void* pick_kernel_out(int D, int out_dtype) {
  switch (out_dtype) {
    case ALPX_F32: return pick_kernel<T, float>(D);
    case ALPX_F16: return pick_kernel<T, f16_t>(D);
    default: return pick_kernel<T, bf16_t>(D);
  }
}

}  // namespace
}  // namespace alpx

extern "C" size_t alpx_prefill_workspace_bytes(int q_tokens, int q_heads, int kv_heads,
                                               int value_dim, int kv_tokens) {
  using namespace alpx;
  if (q_tokens <= 0 || q_heads <= 0 || kv_heads <= 0 || value_dim <= 0 || kv_tokens <= 0 ||
      q_heads % kv_heads != 0)
    return 0;
  return decode_workspace(q_tokens, q_heads, kv_heads, value_dim, kv_tokens);
}

namespace {

// The window, or 0 where it reaches back past row 0 for every token (it hides
// nothing then): the kernels form its positions in 32 bits.
int live_window(int window, int64_t rel0, int q_tokens) {
  return (int64_t)window >= rel0 + q_tokens ? 0 : window;
}

// Key tiles (of `rows` rows) that column tile ct walks: tile_keys on the host.
int host_tile_keys(int q_tokens, int kv_tokens, int group, int rel0, int window, int cols_per_block,
                   int rows, int ct) {
  const int cols = q_tokens * group;
  const int col0 = ct * cols_per_block;
  const int hi = std::max(0, std::min(kv_tokens, rel0 + (std::min(col0 + cols_per_block, cols) - 1) / group + 1));
  int lo = 0;
  if (window > 0) lo = std::min(hi, std::max(0, rel0 + col0 / group - window + 1)) / rows * rows;
  return (hi - lo + rows - 1) / rows;
}

// Key splits of a chunk whose column tiles do not fill the device (see
// prefill_split): at most `splits` pieces of split_tiles key tiles each,
// splits = 0 where the chunk runs unsplit.
//
// Up to one 8-wave block per CU (kSplitBlocks), pieces of equal length.  The
// unsplit kernel then runs one 4-wave block per CU, whose time is its
// heaviest column tile's count N of key tiles (1.04 us each at head_dim
// 128, 0.77 at 64, 0.69 per 32-row tile at 256).  A piece of C tiles costs
// 0.85 C of them (its two groups walk C / 2 each, slower side by side), and
// splitting adds the combine launch and the partials' traffic: about 10
// tiles, and 6 more with a full device (half as much again in the shorter
// tiles of head_dim 256).  Measured, unsplit / split, us (32/8 heads,
// head_dim 128): 9 tokens on 512 rows 16 / 19, on 2048 42 / 19, on 8192
// 142 / 22; 77 on 8192 142 / 30; 256 on 512 21 / 24, on 2048 46 / 32; 512 on
// 512 26 / 32, on 2048 50 / 42, on 8192 149 / 80; 768 on 2048 55 / 55, on
// 8192 155 / 125 (one piece: the two groups alone).  16/2 heads, head_dim
// 256: 128 on 512 21 / 20, 512 on 2048 63 / 42, on 8192 195 / 92.
struct SplitPlan {
  int splits, split_tiles;
  size_t o_bytes, bytes;  // partial O, and all of the workspace
};
constexpr int kSplitBlocks = 256;

SplitPlan plan_split_prefill(int q_tokens, int kv_tokens, int q_heads, int kv_heads, int head_dim,
                             int64_t rel0, int window) {
  SplitPlan p = {0, 0, 0, 0};
  const bool wide = head_dim == 256;
  const int cols_per_block = wide ? 64 : 128, rows = wide ? 32 : 64;
  const int group = q_heads / kv_heads;
  const int64_t items =
      ((int64_t)q_tokens * group + cols_per_block - 1) / cols_per_block * kv_heads;
  if (items > kSplitBlocks) return p;
  const int col_tiles = (int)(items / kv_heads);
  int64_t most = 0;
  for (int ct = 0; ct < col_tiles; ++ct)
    most = std::max<int64_t>(most, host_tile_keys(q_tokens, kv_tokens, group, (int)rel0, window,
                                                  cols_per_block, rows, ct));
  // pieces of at least 256 key rows
  const int64_t pieces =
      std::max<int64_t>(1, std::min<int64_t>(kSplitBlocks / items, most * rows / 256));
  const int64_t c = std::max<int64_t>(1, (most + pieces - 1) / pieces);
  const int64_t splits = (most + c - 1) / c;
  const int64_t cost100 = (1000 + 600 * items * splits / kSplitBlocks) * (wide ? 3 : 2) / 2;
  if (100 * most - 85 * c < cost100) return p;
  p.splits = (int)splits;
  p.split_tiles = (int)c;
  const size_t slots = (size_t)(items * splits);
  p.o_bytes = slots * cols_per_block * head_dim * sizeof(float);
  p.bytes = p.o_bytes + slots * cols_per_block * sizeof(float2);
  return p;
}

// float32 chunks: prefill_f32 over whole key ranges (splits 0), over pieces
// of them, or (splits -1) the split-K decode machinery, one token per
// "sequence", which is the faster one for a few tokens on a long prefix.
// Estimated in us from measured times (32/8 heads, and 16/2 at head_dim
// 256): two blocks on a CU walk a tile each in kTilePair, one block alone
// in 0.6 of that; a split adds the combine (3 us, 6 at head_dim 256) and its
// partials' bytes at 4 TB/s; the decode machinery takes kTokenRow per (token, kv head) and
// cache row.  Measured, decode machinery / prefill_f32: head_dim 64, 1000
// tokens on 0 rows 241 / 51, 100 on 4096 204 / 48 (8 pieces), 9 on 4096
// 25 / 18 (32 pieces), 1 on 4096 12 / 12; head_dim 128, 1000 on 4096
// 3325 / 599, 4 on 1024 22 / 16, 1 on 4096 16 / 25; head_dim 256, 700 on
// 4096 1518 / 485 (4 pieces), 9 on 4096 33 / 42.
// Among the splits whose partials fit `limit` bytes: 300 tokens on 100 rows
// of 8/8 heads of 128 want 7 pieces, 9.3 MB, where the decode machinery (91
// us in place of 11) needs 8.7.
SplitPlan plan_split_f32(int q_tokens, int kv_tokens, int kv_heads, int group, int head_dim,
                         int rel0, int window, size_t limit) {
  SplitPlan p = {0, 0, 0, 0};
  const int rows = head_dim == 256 ? 16 : 32;
  const double pair_us = head_dim == 64 ? 2.2 : (head_dim == 128 ? 4.1 : 4.4);
  const double alone_us = 0.6 * pair_us;
  const double token_row_us = head_dim == 64 ? 0.06e-3 : (head_dim == 128 ? 0.12e-3 : 0.3e-3);
  const double combine_us = head_dim == 256 ? 6 : 3;
  const int col_tiles = (int)(((int64_t)q_tokens * group + 63) / 64);
  const int64_t items = (int64_t)col_tiles * kv_heads;
  const int cus = 256;
  const int first = host_tile_keys(q_tokens, kv_tokens, group, rel0, window, 64, rows, 0);
  const int last =
      host_tile_keys(q_tokens, kv_tokens, group, rel0, window, 64, rows, col_tiles - 1);
  int most = std::max(1, std::max(first, last));
  // a window's longest key range may be that of a tile in between
  if (window > 0 && items < 2 * cus)
    for (int ct = 1; ct < col_tiles - 1; ++ct)
      most = std::max(most, host_tile_keys(q_tokens, kv_tokens, group, rel0, window, 64, rows, ct));
  const double avg = std::max(1.0, 0.5 * (first + last));
  const double decode_us =
      3 + token_row_us * q_tokens * kv_heads * ((group + 15) / 16) * avg * rows;
  auto walk_us = [&](double tiles, double blocks) {  // blocks of `tiles` key tiles each
    const int per_cu = (int)std::ceil(blocks / cus);
    return tiles * ((per_cu / 2) * pair_us + (per_cu % 2) * alone_us);
  };
  double best = std::max(most * alone_us, walk_us(avg, (double)items));
  for (int pieces = 2; pieces <= 32 && items < 2 * cus; ++pieces) {
    const int c = (most + pieces - 1) / pieces;
    const int n = (most + c - 1) / c;
    const double blocks = std::min<double>(items * (double)n, items * (avg / c + 0.5));
    const double us = combine_us + blocks * 64 * head_dim * 8 / 4e6 + walk_us(c, blocks);
    const size_t slots = (size_t)items * n;
    const size_t o_bytes = slots * 64 * head_dim * sizeof(float);
    const size_t bytes = o_bytes + slots * 64 * sizeof(float2);
    if (us < best && bytes <= limit) {
      best = us;
      p = {n, c, o_bytes, bytes};
    }
  }
  if (decode_us < 1.1 * best) p = {-1, 0, 0, 0};
  return p;
}

// Kernel choice for contiguous caches.  The paired kernel gains the tail a
// heavy column tile runs alone and pays a second pipeline start (group 0)
// and the final merge.  Same-box sweep (2048 query tokens, 32/8 or 16/2
// heads, pair / single time): head_dim 128 at prefix 0, 512, 1024, 2048,
// 4096 -- 0.94, 0.98, 1.00, 1.04, 1.03; head_dim 256 at prefix 0, 2048,
// 8192 -- 0.75, 0.91, 1.04; head_dim 64 at prefix 0, 2048 -- 0.92, 0.98;
// 512 query tokens (64 pairs) 1.37; 8192 tokens at prefix 0 (four rounds
// of pairs) 1.02.  So: pairs must form one round that fills the device,
// and the heaviest column tile must walk at least R times the key tiles of
// the lightest, R = 3 at head_dim 128 and 1.8 at 64 and 256.  At head_dim
// 256 two full rounds of pairs do no worse (16/2 heads, pair / single:
// 4096 tokens at prefix 0 -- 168 / 169 us, at prefix 1024 -- 236 / 240);
// partly filled rounds do (3000 tokens at prefix 0 -- 121 / 103; 24/4
// heads, 1536 tokens -- 76 / 47), as do three (24/4 heads, 4096 tokens --
// 248 / 240).  The shared-stream kernel (one
// tile stream for both tiles of a pair, no window start inside the chunk)
// pays off at head_dim 256 with long prefixes only (2048 tokens, 16/2
// heads, shared / pair / single, us, one box: prefix 1024 -- 86.9 / 82.7 /
// 96.6, 1536 -- 101.8 / 99.4 / 113.0, 2048 -- 118.9 / 115.8 / 127.7, 8192
// -- 304.5 / 316.1 / 311.4; another box: 4096 -- 178.4 / 187.7 / 191.1;
// head_dim 128 at prefix 2048: 104.7 / 105.4 / 100.8, head_dim 64: 72.1 /
// 65.2 / 66.4), so it takes one round of pairs below a ratio of
// kSharedBelow10 / 10.
// ALPX_OVERRIDE_PREFILL_KERNEL (1 single, 2 paired, 3 shared-stream)
// overrides the choice (shared falls back to the single kernel where one
// stream cannot serve).
enum PrefillKernelChoice { kSingleKernel, kPairKernel, kSharedKernel };
constexpr int kSharedBelow10 = 16;

PrefillKernelChoice choose_prefill(int q_tokens, int kv_tokens, int kv_heads, int group, int rel0,
                                   int window, int cols_per_block, int rows, int col_tiles,
                                   int key_dim, const void* pair_kernel) {
  // both tiles of a pair walk the key rows from 0 when no window starts inside the chunk
  const bool one_stream = window <= 0 || (int64_t)window > (int64_t)rel0 + q_tokens;
  const int force = alpx::override_value(ALPX_OVERRIDE_PREFILL_KERNEL);
  if (force == 2) return kPairKernel;
  if (force == 1) return kSingleKernel;
  if (force == 3) return one_stream ? kSharedKernel : kSingleKernel;
  const int64_t pairs = (int64_t)kv_heads * ((col_tiles + 1) / 2);
  const int resident = alpx::resident_blocks(pair_kernel, 512, 0);
  if (resident <= 0) return kSingleKernel;
  const int64_t rounds = (pairs + resident - 1) / resident;
  const bool one_round = rounds == 1;
  if (pairs * 10 < rounds * resident * 9 || rounds > (key_dim == 256 ? 2 : 1))
    return kSingleKernel;
  const int first = host_tile_keys(q_tokens, kv_tokens, group, rel0, window, cols_per_block, rows, 0);
  const int last =
      host_tile_keys(q_tokens, kv_tokens, group, rel0, window, cols_per_block, rows, col_tiles - 1);
  const int64_t ratio10 = (int64_t)last * 10 / std::max(1, first);
  if (key_dim == 256 && one_round && one_stream && ratio10 < kSharedBelow10) return kSharedKernel;
  const int r10 = key_dim == 128 ? 30 : 18;  // R x 10
  return ratio10 >= r10 ? kPairKernel : kSingleKernel;
}

// Whether prefill_impl runs these operands on the MFMA kernels: fp16 /
// bf16, equal head dims of 64, 128 or 256, 16-byte aligned buffers and row
// strides (`align` ORs their addresses and byte strides), and per-tile row
// offsets that fit 32 bits.  Otherwise it takes the split-K path, which
// needs a workspace of alpx_prefill_workspace_bytes.
bool flash_operands(int dtype, int key_dim, int value_dim, uintptr_t align, int64_t kv_tokens,
                    int64_t k_pos_stride, int64_t v_pos_stride, int64_t rel0) {
  const int64_t es = (int64_t)alpx::dtype_size(dtype);
  return key_dim == value_dim &&
         (key_dim == 64 || key_dim == 128 || key_dim == 256) && (align & 15) == 0 &&
         alpx::override_value(ALPX_OVERRIDE_PREFILL_GENERIC) == 0 &&
         kv_tokens * k_pos_stride * es < ((int64_t)1 << 31) &&
         kv_tokens * v_pos_stride * es < ((int64_t)1 << 31) && rel0 < ((int64_t)1 << 30) &&
         rel0 > -((int64_t)1 << 30);
}

bool mfma_prefill_applies(int dtype, int key_dim, int value_dim, uintptr_t align,
                          int64_t kv_tokens, int64_t k_pos_stride, int64_t v_pos_stride,
                          int64_t rel0) {
  return dtype != ALPX_F32 &&
         flash_operands(dtype, key_dim, value_dim, align, kv_tokens, k_pos_stride, v_pos_stride,
                        rel0);
}

// The query prologue a prefill forms itself (alpx_attention_layer_prefill
// with no query_out): q is then the joint projection [T, Hq, 2 D].
struct QueryPrologue {
  const float* qw;
  const float2* rot;  // [T, R] (cos, sin) per token and pair
  float eps;
  int R;
};

int prefill_impl(const void* q, const void* key, const void* value, const void* gate, void* out,
                 void* workspace, size_t workspace_bytes, int q_tokens, int kv_tokens,
                 int q_heads, int kv_heads, int key_dim, int value_dim, int64_t k_pos_stride,
                 int64_t v_pos_stride, int64_t q_pos0, int window, int64_t kv_start, float scale,
                 int dtype, int out_dtype, void* stream, const int32_t* pages = nullptr,
                 int page_shift = 0, int num_pages = 0, const void* kn = nullptr,
                 const void* vn = nullptr, int64_t gate_stride = 0,
                 const QueryPrologue* qpro = nullptr) {
  using namespace alpx;
  if (!q || !key || !value || !out) return fail(ALPX_EINVAL, "alpx_prefill_causal: null buffer");
  if (!dtype_ok(dtype) || !dtype_ok(out_dtype))
    return fail(ALPX_EINVAL, "alpx_prefill_causal: unknown dtype");
  if (q_tokens <= 0 || kv_tokens <= 0 || q_heads <= 0 || kv_heads <= 0 || key_dim <= 0 ||
      value_dim <= 0)
    return fail(ALPX_EINVAL, "alpx_prefill_causal: sizes must be positive");
  if (q_heads % kv_heads != 0)
    return fail(ALPX_EINVAL, "attention query heads must be a multiple of KV heads");
  if (k_pos_stride < (int64_t)kv_heads * key_dim || v_pos_stride < (int64_t)kv_heads * value_dim)
    return fail(ALPX_EINVAL, "alpx_prefill_causal: row strides smaller than a row");
  if (q_pos0 < 0 || kv_start < 0 || window < 0)
    return fail(ALPX_EINVAL, "alpx_prefill_causal: negative position or window");
  if (!(scale > 0.0f) || !isfinite(scale))
    return fail(ALPX_EINVAL, "attention scale must be positive and finite");
  if (key_dim > 256 || value_dim > 256)
    return fail(ALPX_EUNSUPPORTED, "alpx_prefill_causal: head dims above 256 are not supported");

  window = live_window(window, q_pos0 - kv_start, q_tokens);
  hipStream_t s = (hipStream_t)stream;
  const int group = q_heads / kv_heads;
  const size_t es = dtype_size(dtype);
  // Append mode reads the chunk's rows through the cache's row strides.
  if (kn != nullptr && (k_pos_stride != (int64_t)kv_heads * key_dim ||
                        v_pos_stride != (int64_t)kv_heads * value_dim))
    return fail(ALPX_EINVAL, "alpx_prefill_append: cache rows must be contiguous");
  if (gate_stride == 0) gate_stride = value_dim;
  const int64_t q_stride = qpro != nullptr ? 2 * (int64_t)key_dim : key_dim;
  const uintptr_t align = (uintptr_t)q | (uintptr_t)(q_stride * es) | (uintptr_t)key |
                          (uintptr_t)value | (uintptr_t)gate |
                          (uintptr_t)(gate_stride * es) |
                          (uintptr_t)kn | (uintptr_t)vn | (uintptr_t)(k_pos_stride * es) |
                          (uintptr_t)(v_pos_stride * es);
  const bool mfma = mfma_prefill_applies(dtype, key_dim, value_dim, align, kv_tokens, k_pos_stride,
                                         v_pos_stride, q_pos0 - kv_start);
  if (pages != nullptr && !(mfma && out_dtype == dtype))
    return fail(ALPX_EUNSUPPORTED,
                "alpx_prefill_causal_paged: needs fp16/bf16 pages, head_dim in {64, 128, 256}, "
                "16-byte aligned rows and out_dtype == dtype");
  PrefillArgs a = {};
  a.kn = kn;
  a.vn = vn;
  a.new0 = (int)(q_pos0 - kv_start);
  a.pages = pages;
  a.page_shift = page_shift;
  a.num_pages = num_pages;
  a.ks_page = ((int64_t)1 << page_shift) * k_pos_stride;
  a.vs_page = ((int64_t)1 << page_shift) * v_pos_stride;
  a.q = q;
  a.q_stride = q_stride;
  if (qpro != nullptr) {
    a.qw = qpro->qw;
    a.q_rot = qpro->rot;
    a.q_eps = qpro->eps;
    a.q_R = qpro->R;
  }
  a.k = key;
  a.v = value;
  a.gate = gate;
  a.gate_stride = gate_stride;
  a.out = out;
  a.ks_pos = k_pos_stride;
  a.vs_pos = v_pos_stride;
  a.pos0 = q_pos0;
  a.kv_start = kv_start;
  a.window = window;
  a.q_tokens = q_tokens;
  a.kv_tokens = kv_tokens;
  a.q_heads = q_heads;
  a.kv_heads = kv_heads;
  a.group = group;
  a.scale_log2 = scale * kLog2e;
  if (mfma) {
    const int cols_per_block = key_dim == 256 ? 64 : 128;
    const int tile_rows = key_dim == 256 ? 32 : 64;
    const int col_tiles = (int)(((int64_t)q_tokens * group + cols_per_block - 1) / cols_per_block);
    const PrefillKernelChoice choice =
        pages != nullptr
            ? kSingleKernel
            : choose_prefill(q_tokens, kv_tokens, kv_heads, group, (int)(q_pos0 - kv_start), window,
                             cols_per_block, tile_rows, col_tiles, key_dim,
                             prefill_pair_kernel(dtype, key_dim, out_dtype));
    const bool pair = choice == kPairKernel, shared = choice == kSharedKernel;
    SplitPlan sp = {0, 0, 0, 0};
    if (pages == nullptr && choice == kSingleKernel && workspace != nullptr &&
        override_value(ALPX_OVERRIDE_PREFILL_KERNEL) == 0) {
      sp = plan_split_prefill(q_tokens, kv_tokens, q_heads, kv_heads, key_dim, q_pos0 - kv_start,
                              window);
      if (((uintptr_t)workspace & 15) != 0 || workspace_bytes < sp.bytes) sp.splits = 0;
    }
    const bool split = sp.splits > 0;
    a.col_tiles = col_tiles;
    const void* kernel = nullptr;
    if (split)
      kernel = prefill_split_kernel(dtype, key_dim);
    else if (pages != nullptr)
      kernel = dtype == ALPX_F16 ? pick_kernel_paged<f16_t>(key_dim)
                                 : pick_kernel_paged<bf16_t>(key_dim);
    else if (shared)
      kernel = prefill_shared_kernel(dtype, key_dim, out_dtype);
    else if (pair)
      kernel = prefill_pair_kernel(dtype, key_dim, out_dtype);
    else if (dtype == ALPX_F16)
      kernel = pick_kernel_out<f16_t>(key_dim, out_dtype);
    else
      kernel = pick_kernel_out<bf16_t>(key_dim, out_dtype);
    const bool paired = pair || shared;  // a light and a heavy column tile per block
    const int64_t items =
        (int64_t)(paired ? (a.col_tiles + 1) / 2 : a.col_tiles) * kv_heads *
        (split ? sp.splits : 1);
    a.splits = sp.splits;
    a.split_tiles = sp.split_tiles;
    a.part_o = (float*)workspace;
    a.part_st = (float2*)((char*)workspace + sp.o_bytes);
    a.per_xcd = (int)((items + kXcds - 1) / kXcds);
    TimedRegion timed(ALPX_T_PREFILL, s);
    void* args[] = {(void*)&a};
    hipError_t err = hipLaunchKernel(kernel, dim3(a.per_xcd * kXcds), dim3(paired || split ? 512 : 256),
                                     args, 0, s);
    if (err != hipSuccess)
      return fail(ALPX_EHIP, "prefill launch failed: %s", hipGetErrorString(err));
    int rc = check_launch("prefill_mfma");
    if (rc != ALPX_OK || !split) return rc;
    const void* combine = prefill_combine_kernel(dtype, key_dim, out_dtype);
    const int slices = cols_per_block / 16;  // 16-column slices per column tile
    err = hipLaunchKernel(combine, dim3(a.col_tiles * kv_heads * slices), dim3(256), args, 0, s);
    if (err != hipSuccess)
      return fail(ALPX_EHIP, "prefill combine launch failed: %s", hipGetErrorString(err));
    return check_launch("prefill_combine");
  }

  if (qpro != nullptr)  // callers check the MFMA conditions before any launch
    return fail(ALPX_EUNSUPPORTED, "fused query prologue: MFMA prefill shapes only");
  if (!workspace) return fail(ALPX_EINVAL, "alpx_prefill_causal: null workspace");
  const size_t need = decode_workspace(q_tokens, q_heads, kv_heads, value_dim, kv_tokens);
  if (workspace_bytes < need)
    return fail(ALPX_EINVAL, "decode workspace holds %zu bytes, needs %zu", workspace_bytes, need);
  if (kn != nullptr) {  // append mode off the MFMA path: the append kernel first
    const int rc = alpx_kv_append(const_cast<void*>(key), const_cast<void*>(value), kn, vn, dtype,
                                  kv_tokens, 1, kv_heads, key_dim, value_dim, q_tokens,
                                  q_pos0 - kv_start, nullptr, stream);
    if (rc != ALPX_OK) return rc;
  }
  if (dtype == ALPX_F32 && (int64_t)q_tokens * group < ((int64_t)1 << 30) &&
      flash_operands(dtype, key_dim, value_dim, align, kv_tokens, k_pos_stride, v_pos_stride,
                     q_pos0 - kv_start)) {
    const SplitPlan sp = plan_split_f32(q_tokens, kv_tokens, kv_heads, group, key_dim,
                                        (int)(q_pos0 - kv_start), window,
                                        ((uintptr_t)workspace & 15) == 0 ? workspace_bytes : 0);
    if (sp.splits >= 0) {
      const bool split = sp.splits > 0;
      a.col_tiles = (int)(((int64_t)q_tokens * group + 63) / 64);
      a.splits = sp.splits;
      a.split_tiles = sp.split_tiles;
      a.part_o = (float*)workspace;
      a.part_st = (float2*)((char*)workspace + sp.o_bytes);
      const int64_t items = (int64_t)a.col_tiles * kv_heads * (split ? sp.splits : 1);
      a.per_xcd = (int)((items + kXcds - 1) / kXcds);
      void* args[] = {(void*)&a};
      TimedRegion timed(ALPX_T_PREFILL, s);
      hipError_t err = hipLaunchKernel(prefill_f32_kernel(key_dim, out_dtype, split),
                                       dim3(a.per_xcd * kXcds), dim3(256), args, 0, s);
      if (err != hipSuccess)
        return fail(ALPX_EHIP, "prefill launch failed: %s", hipGetErrorString(err));
      const int rc = check_launch("prefill_f32");
      if (rc != ALPX_OK || !split) return rc;
      err = hipLaunchKernel(prefill_combine_kernel(dtype, key_dim, out_dtype),
                            dim3(a.col_tiles * kv_heads * 4), dim3(256), args, 0, s);
      if (err != hipSuccess)
        return fail(ALPX_EHIP, "prefill combine launch failed: %s", hipGetErrorString(err));
      return check_launch("prefill_combine");
    }
  }
  DecodeArgs d = {};
  d.q = q;
  d.k = key;
  d.v = value;
  d.seq_lens = nullptr;
  d.gate = gate;  // the combine pass applies it ([token][head][d] = [b][h][d])
  d.gate_stride = gate_stride;
  d.out = out;
  d.ks_pos = k_pos_stride;
  d.ks_b = 0;
  d.ks_h = key_dim;
  d.vs_pos = v_pos_stride;
  d.vs_b = 0;
  d.vs_h = value_dim;
  d.causal_pos0 = q_pos0;
  d.kv_start = kv_start;
  d.window = window;
  d.length = kv_tokens;
  d.batch = q_tokens;
  d.q_heads = q_heads;
  d.kv_heads = kv_heads;
  d.group = group;
  d.key_dim = key_dim;
  d.value_dim = value_dim;
  d.scale_log2 = scale * kLog2e;
  return run_decode(d, dtype, out_dtype, workspace, workspace_bytes, s, ALPX_T_PREFILL,
                    ALPX_T_AUX);
}

}  // namespace

extern "C" size_t alpx_prefill_split_bytes(int q_tokens, int kv_tokens, int q_heads, int kv_heads,
                                           int head_dim, int64_t q_pos0, int window,
                                           int64_t kv_start) {
  const int64_t rel0 = q_pos0 - kv_start;
  if (q_tokens <= 0 || kv_tokens <= 0 || q_heads <= 0 || kv_heads <= 0 ||
      q_heads % kv_heads != 0 || (head_dim != 64 && head_dim != 128 && head_dim != 256) ||
      window < 0 || rel0 >= ((int64_t)1 << 30) || rel0 <= -((int64_t)1 << 30))
    return 0;
  return plan_split_prefill(q_tokens, kv_tokens, q_heads, kv_heads, head_dim, rel0,
                            live_window(window, rel0, q_tokens))
      .bytes;
}

extern "C" size_t alpx_prefill_f32_workspace_bytes(int q_tokens, int kv_tokens, int q_heads,
                                                   int kv_heads, int key_dim, int value_dim,
                                                   int64_t q_pos0, int window, int64_t kv_start,
                                                   int* pieces) {
  const size_t need =
      alpx_prefill_workspace_bytes(q_tokens, q_heads, kv_heads, value_dim, kv_tokens);
  const int64_t rel0 = q_pos0 - kv_start;
  SplitPlan p = {-1, 0, 0, 0};
  if (need > 0 && key_dim == value_dim && (key_dim == 64 || key_dim == 128 || key_dim == 256) &&
      window >= 0 && rel0 < ((int64_t)1 << 30) && rel0 > -((int64_t)1 << 30) &&
      (int64_t)q_tokens * (q_heads / kv_heads) < ((int64_t)1 << 30))
    p = plan_split_f32(q_tokens, kv_tokens, kv_heads, q_heads / kv_heads, key_dim, (int)rel0,
                       live_window(window, rel0, q_tokens), SIZE_MAX);
  if (pieces != nullptr) *pieces = p.splits;
  return std::max(need, p.bytes);
}

extern "C" int alpx_prefill_causal(const void* q, const void* key, const void* value, void* out,
                                   void* workspace, size_t workspace_bytes, int q_tokens,
                                   int kv_tokens, int q_heads, int kv_heads, int key_dim,
                                   int value_dim, int64_t k_pos_stride, int64_t v_pos_stride,
                                   int64_t q_pos0, int window, int64_t kv_start, float scale,
                                   int dtype, int out_dtype, void* stream) {
  return prefill_impl(q, key, value, nullptr, out, workspace, workspace_bytes, q_tokens, kv_tokens,
                      q_heads, kv_heads, key_dim, value_dim, k_pos_stride, v_pos_stride, q_pos0,
                      window, kv_start, scale, dtype, out_dtype, stream);
}

extern "C" int alpx_prefill_causal_gated(const void* q, const void* key, const void* value,
                                         const void* gate, void* out, void* workspace,
                                         size_t workspace_bytes, int q_tokens, int kv_tokens,
                                         int q_heads, int kv_heads, int key_dim, int value_dim,
                                         int64_t k_pos_stride, int64_t v_pos_stride,
                                         int64_t q_pos0, int window, int64_t kv_start,
                                         float scale, int dtype, int out_dtype, void* stream) {
  if (!gate) return alpx::fail(ALPX_EINVAL, "alpx_prefill_causal_gated: null gate");
  return prefill_impl(q, key, value, gate, out, workspace, workspace_bytes, q_tokens, kv_tokens,
                      q_heads, kv_heads, key_dim, value_dim, k_pos_stride, v_pos_stride, q_pos0,
                      window, kv_start, scale, dtype, out_dtype, stream);
}

extern "C" int alpx_prefill_append(const void* q, const void* key, const void* value,
                                   void* key_cache, void* value_cache, const void* gate, void* out,
                                   void* workspace, size_t workspace_bytes, int q_tokens,
                                   int64_t capacity, int q_heads, int kv_heads, int key_dim,
                                   int value_dim, int64_t position, int window, float scale,
                                   int dtype, int out_dtype, void* stream) {
  using namespace alpx;
  if (!key || !value || !key_cache || !value_cache)
    return fail(ALPX_EINVAL, "alpx_prefill_append: null buffer");
  if (q_tokens <= 0 || capacity <= 0 || kv_heads <= 0 || key_dim <= 0 || value_dim <= 0)
    return fail(ALPX_EINVAL, "alpx_prefill_append: sizes must be positive");
  if (position < 0 || position > capacity - q_tokens)
    return fail(ALPX_ERANGE, "attention cache position exceeds capacity");
  if (position + q_tokens > INT32_MAX)
    return fail(ALPX_EUNSUPPORTED, "alpx_prefill_append: more than 2^31 - 1 cache rows");
  return prefill_impl(q, key_cache, value_cache, gate, out, workspace, workspace_bytes, q_tokens,
                      (int)(position + q_tokens), q_heads, kv_heads, key_dim, value_dim,
                      (int64_t)kv_heads * key_dim, (int64_t)kv_heads * value_dim, position, window,
                      0, scale, dtype, out_dtype, stream, nullptr, 0, 0, key, value);
}

extern "C" int alpx_attention_layer_prefill(
    const void* query_gate, const void* key, const void* value, const float* q_norm,
    const float* k_norm, void* query_out, void* key_cache, void* value_cache, void* out,
    void* workspace, size_t workspace_bytes, int dtype, int out_dtype, int64_t capacity,
    int cache_batch, int batch_index, int tokens, int q_heads, int kv_heads, int head_dim,
    int64_t position, const int* sections, double frequency_base, float eps, float scale,
    void* stream) {
  using namespace alpx;
  if (!out) return fail(ALPX_EINVAL, "alpx_attention_layer_prefill: null buffer");
  if (!dtype_ok(dtype) || !dtype_ok(out_dtype))
    return fail(ALPX_EINVAL, "alpx_attention_layer_prefill: unknown dtype");
  if (tokens <= 0 || head_dim <= 0 || kv_heads <= 0 || cache_batch <= 0)
    return fail(ALPX_EINVAL, "alpx_attention_layer_prefill: sizes must be positive");
  if (head_dim > 256)
    return fail(ALPX_EUNSUPPORTED, "alpx_prefill_causal: head dims above 256 are not supported");
  if (position + tokens > INT32_MAX)
    return fail(ALPX_EUNSUPPORTED, "alpx_attention_layer_prefill: more than 2^31 - 1 cache rows");
  // The prefill's checks that need no device work, first: a failing call
  // must not have written the caches.
  if (!workspace && !(dtype != ALPX_F32 && (head_dim == 64 || head_dim == 128 || head_dim == 256)))
    return fail(ALPX_EINVAL, "alpx_prefill_causal: null workspace");
  if (!(scale > 0.0f) || !isfinite(scale))
    return fail(ALPX_EINVAL, "attention scale must be positive and finite");
  const size_t es = dtype_size(dtype);
  const int64_t row = (int64_t)cache_batch * kv_heads * head_dim;
  const int64_t seq = (int64_t)batch_index * kv_heads * head_dim;
  const void* kseq = (const char*)key_cache + seq * es;
  const void* vseq = (const char*)value_cache + seq * es;
  const void* gate = (const char*)query_gate + head_dim * es;
  if (query_out == nullptr) {
    // The prefill forms the query rows from query_gate (its Q load runs the
    // prologue's norm and rotation); the prologue launch writes the key and
    // value rows only.  Needs the MFMA prefill and rotary pairs in whole
    // 32-channel groups; checked before any launch.
    int R = 0;
    if (!query_gate || !q_norm || bad_sections(sections, R) || R % 32 != 0 || 2 * R > head_dim ||
        !(frequency_base > 0.0) || !isfinite(frequency_base))
      return fail(ALPX_EUNSUPPORTED,
                  "alpx_attention_layer_prefill without query_out: needs rotary sections summing "
                  "to a multiple of 32 and a valid frequency base");
    const uintptr_t align = (uintptr_t)query_gate | (uintptr_t)kseq | (uintptr_t)vseq |
                            (uintptr_t)q_norm | (uintptr_t)(row * es) |
                            (uintptr_t)(2 * head_dim * es);
    if (!((dtype == ALPX_F16 || dtype == ALPX_BF16) &&
          (head_dim == 64 || head_dim == 128 || head_dim == 256) && (align & 15) == 0 &&
          override_value(ALPX_OVERRIDE_PREFILL_GENERIC) == 0 &&
          (position + tokens) * row * (int64_t)es < ((int64_t)1 << 31)))
      return fail(ALPX_EUNSUPPORTED,
                  "alpx_attention_layer_prefill without query_out: needs fp16/bf16, head_dim in "
                  "{64, 128, 256}, 16-byte aligned rows and q_norm, and a cache under 2 GiB per "
                  "tensor");
    const size_t need = (size_t)tokens * R * sizeof(float2);
    if (!workspace || workspace_bytes < need)
      return fail(ALPX_EINVAL, "alpx_attention_layer_prefill: workspace of %zu bytes, %zu needed",
                  workspace ? workspace_bytes : (size_t)0, need);
    QueryPrologue qp = {};
    qp.qw = q_norm;
    qp.rot = (const float2*)workspace;
    qp.eps = eps;
    qp.R = R;
    const int rc = attention_prologue_chunk_kv(
        query_gate, key, value, q_norm, k_norm, key_cache, value_cache, dtype, capacity,
        cache_batch, batch_index, tokens, q_heads, kv_heads, head_dim, head_dim, position,
        sections, frequency_base, eps, (float2*)workspace, stream);
    if (rc != ALPX_OK) return rc;
    // past the rotation table, workspace for a split chunk where there is any
    const size_t used = (need + 255) & ~(size_t)255;
    const bool more = workspace_bytes > used;
    return prefill_impl(query_gate, kseq, vseq, gate, out,
                        more ? (char*)workspace + used : nullptr,
                        more ? workspace_bytes - used : 0, tokens, (int)(position + tokens),
                        q_heads, kv_heads, head_dim, head_dim, row, row, position, 0, 0, scale,
                        dtype, out_dtype, stream, nullptr, 0, 0, nullptr, nullptr,
                        2 * (int64_t)head_dim, &qp);
  }
  // The query-buffer form: where the prefill will not take the MFMA
  // kernels, its split-K path needs a workspace, checked before the
  // prologue writes the caches.
  const uintptr_t qalign = (uintptr_t)query_out | (uintptr_t)(head_dim * es) | (uintptr_t)kseq |
                           (uintptr_t)vseq | (uintptr_t)gate | (uintptr_t)(2 * head_dim * es) |
                           (uintptr_t)(row * es);
  if (!mfma_prefill_applies(dtype, head_dim, head_dim, qalign, position + tokens, row, row,
                            position)) {
    const size_t need =
        alpx_prefill_workspace_bytes(tokens, q_heads, kv_heads, head_dim, (int)(position + tokens));
    if (need == 0) return fail(ALPX_EINVAL, "alpx_attention_layer_prefill: invalid sizes");
    if (!workspace || workspace_bytes < need)
      return fail(ALPX_EINVAL,
                  "alpx_attention_layer_prefill: the split-K prefill needs a workspace of %zu "
                  "bytes, %zu given (null workspace)",
                  need, workspace ? workspace_bytes : (size_t)0);
  }
  const int rc = alpx_attention_prologue_chunk(
      query_gate, key, value, q_norm, k_norm, query_out, nullptr, key_cache, value_cache, dtype,
      capacity, cache_batch, batch_index, tokens, q_heads, kv_heads, head_dim, head_dim, position,
      sections, frequency_base, eps, stream);
  if (rc != ALPX_OK) return rc;
  return prefill_impl(query_out, kseq, vseq, gate, out, workspace, workspace_bytes, tokens,
                      (int)(position + tokens), q_heads, kv_heads, head_dim, head_dim, row, row,
                      position, 0, 0, scale, dtype, out_dtype, stream, nullptr, 0, 0, nullptr,
                      nullptr, 2 * (int64_t)head_dim);
}

extern "C" int alpx_attention_layer_prefill_paged(
    const void* query_gate, const void* key, const void* value, const float* q_norm,
    const float* k_norm, void* key_pages, void* value_pages, const int32_t* block_table,
    int max_pages, int page_size, int num_pages, int batch_index, void* out, void* workspace,
    size_t workspace_bytes, int dtype, int tokens, int q_heads, int kv_heads, int head_dim,
    int64_t position, const int* sections, double frequency_base, float eps, float scale,
    void* stream) {
  using namespace alpx;
  const char* what = "alpx_attention_layer_prefill_paged";
  if (!query_gate || !key || !value || !q_norm || !k_norm || !key_pages || !value_pages ||
      !block_table || !out)
    return fail(ALPX_EINVAL, "%s: null buffer", what);
  if (!dtype_ok(dtype)) return fail(ALPX_EINVAL, "%s: unknown dtype", what);
  if (tokens <= 0 || q_heads <= 0 || kv_heads <= 0 || head_dim <= 0 || max_pages <= 0 ||
      num_pages <= 0 || batch_index < 0)
    return fail(ALPX_EINVAL, "%s: sizes must be positive", what);
  if (page_size < 64 || (page_size & (page_size - 1)) != 0)
    return fail(ALPX_EINVAL, "%s: page_size must be a power of two >= 64", what);
  if (position < 0 || position + tokens > (int64_t)max_pages * page_size)
    return fail(ALPX_ERANGE, "attention cache position exceeds capacity");
  if (!(scale > 0.0f) || !isfinite(scale))
    return fail(ALPX_EINVAL, "attention scale must be positive and finite");
  // Everything the two launches check, first: a failing call writes no page.
  int R = 0;
  if (bad_sections(sections, R) || R % 32 != 0 || 2 * R > head_dim ||
      !(frequency_base > 0.0) || !isfinite(frequency_base))
    return fail(ALPX_EUNSUPPORTED,
                "%s: needs rotary sections summing to a multiple of 32 (at most head_dim / 2) "
                "and a valid frequency base", what);
  const size_t es = dtype_size(dtype);
  const int64_t row = (int64_t)kv_heads * head_dim;
  const uintptr_t align = (uintptr_t)query_gate | (uintptr_t)key_pages | (uintptr_t)value_pages |
                          (uintptr_t)q_norm | (uintptr_t)(row * es) |
                          (uintptr_t)(2 * head_dim * es);
  if (!((dtype == ALPX_F16 || dtype == ALPX_BF16) &&
        (head_dim == 64 || head_dim == 128 || head_dim == 256) && (align & 15) == 0 &&
        override_value(ALPX_OVERRIDE_PREFILL_GENERIC) == 0 && position < ((int64_t)1 << 30) &&
        (position + tokens) * row * (int64_t)es < ((int64_t)1 << 31)))
    return fail(ALPX_EUNSUPPORTED,
                "%s: needs fp16/bf16 pages, head_dim in {64, 128, 256}, 16-byte aligned rows and "
                "q_norm, and under 2 GiB of logical rows", what);
  const size_t need = (size_t)tokens * R * sizeof(float2);
  if (!workspace || workspace_bytes < need)
    return fail(ALPX_EINVAL, "%s: workspace of %zu bytes, %zu needed", what,
                workspace ? workspace_bytes : (size_t)0, need);
  const int page_shift = __builtin_ctz((unsigned)page_size);
  const int32_t* table = block_table + (int64_t)batch_index * max_pages;
  QueryPrologue qp = {};
  qp.qw = q_norm;
  qp.rot = (const float2*)workspace;
  qp.eps = eps;
  qp.R = R;
  const int rc = attention_prologue_chunk_kv(
      query_gate, key, value, q_norm, k_norm, key_pages, value_pages, dtype,
      (int64_t)max_pages * page_size, 1, 0, tokens, q_heads, kv_heads, head_dim, head_dim,
      position, sections, frequency_base, eps, (float2*)workspace, stream, table, page_shift,
      num_pages);
  if (rc != ALPX_OK) return rc;
  return prefill_impl(query_gate, key_pages, value_pages, (const char*)query_gate + head_dim * es,
                      out, nullptr, 0, tokens, (int)(position + tokens), q_heads, kv_heads,
                      head_dim, head_dim, row, row, position, 0, 0, scale, dtype, dtype, stream,
                      table, page_shift, num_pages, nullptr, nullptr, 2 * (int64_t)head_dim, &qp);
}

extern "C" int alpx_prefill_causal_paged(const void* q, const void* key_pages,
                                         const void* value_pages, const int32_t* block_table,
                                         int max_pages, int page_size, int num_pages,
                                         int batch_index, const void* gate, void* out,
                                         int q_tokens, int kv_tokens, int q_heads, int kv_heads,
                                         int head_dim, int64_t q_pos0, int window,
                                         int64_t kv_start, float scale, int dtype, void* stream) {
  using namespace alpx;
  if (!block_table) return fail(ALPX_EINVAL, "alpx_prefill_causal_paged: null block table");
  if (max_pages <= 0 || num_pages <= 0 || batch_index < 0)
    return fail(ALPX_EINVAL, "alpx_prefill_causal_paged: sizes must be positive");
  if (page_size < 64 || (page_size & (page_size - 1)) != 0)
    return fail(ALPX_EINVAL, "alpx_prefill_causal_paged: page_size must be a power of two >= 64");
  if ((int64_t)kv_tokens > (int64_t)max_pages * page_size)
    return fail(ALPX_ERANGE, "attention cache length exceeds capacity");
  const int64_t row = (int64_t)kv_heads * head_dim;
  return prefill_impl(q, key_pages, value_pages, gate, out, nullptr, 0, q_tokens, kv_tokens,
                      q_heads, kv_heads, head_dim, head_dim, row, row, q_pos0, window, kv_start,
                      scale, dtype, dtype, stream, block_table + (int64_t)batch_index * max_pages,
                      __builtin_ctz((unsigned)page_size), num_pages);
}
