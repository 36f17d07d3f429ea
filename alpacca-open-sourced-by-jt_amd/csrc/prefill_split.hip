// Prefill of chunks whose column tiles do not fill the device: the key
// ranges are cut over more blocks, whose partial states a second launch
// merges.
#include "prefill_run.h"

namespace alpx {
namespace {

// Few column tiles over long key ranges (a short chunk on a long prefix, or
// a chunk that does not fill the device): the key tiles of every column
// tile are cut into pieces of split_tiles and each block runs one piece,
// so that the chip is filled by keys where columns cannot fill it.  The
// partial states go to global memory and prefill_combine merges them.
// Unsplit, such a chunk is bound by one block's serial walk over its key
// tiles: 77 tokens on 6011 rows (32/8 heads, head_dim 128, bf16) took 110 us
// on 24 of 256 CUs, and takes 24.5 + 5.7 us here (240 blocks of 5 or 6
// tiles per group).  What is left is the blocks' common start (8 us to the
// first tile's scores), the keys' read and 15 MB of partials each way; one
// 4-wave block per piece, twice as many pieces, measured 3 us slower.
//
// A block's eight waves are two groups of four that run the first and the
// second half of the piece's tiles, each with its own tile buffers and
// barrier (as in prefill_pair); group 1 merges group 0's state out of LDS,
// so a CU's eight waves leave one partial state rather than two.
template <typename T, int D, int BK, int NQB>
__global__ void __launch_bounds__(512, 1)
prefill_split(PrefillArgs a) {
  constexpr int kTileB = BK * D * (int)sizeof(T);
  constexpr int kCols = 64 * NQB;
  constexpr int MB = D / 16;
  static_assert(NQB * MB * 64 * 16 * 4 <= 4 * kTileB, "the partial O must fit a group's buffers");
  __shared__ __attribute__((aligned(1024))) char smem[8 * kTileB];
  __shared__ float part_st[4 * NQB * 3 * 64];
  __shared__ uint32_t gctr[2];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2;
  // kv-head-major items in 8 contiguous slices, slice x on XCD x; within a
  // kv head the column tiles of one piece are neighbours, so the blocks
  // that read the same keys run together on one XCD.
  const int b = blockIdx.x;
  const int item = (b % kXcds) * a.per_xcd + b / kXcds;
  const int per_head = a.col_tiles * a.splits;
  if (item >= a.kv_heads * per_head) return;
  const int kvh = item / per_head;
  const int piece = (item - kvh * per_head) / a.col_tiles;
  const int ctile = a.col_tiles - 1 - (item - kvh * per_head - piece * a.col_tiles);
  int lo, hi, nt;
  tile_keys<BK, kCols>(a, ctile, lo, hi, nt);
  const int tb = piece * a.split_tiles;
  if (piece > 0 && tb >= nt) return;  // this column tile has fewer pieces
  if (tid < 2) gctr[tid] = 0;
  __syncthreads();  // the group counters are zero before any group barrier
  const int te = min(tb + a.split_tiles, nt);
  const int mid = tb + (te - tb + 1) / 2;
  GroupBarrier bar{gctr + grp, 0u};
  char* gsmem = smem + grp * 4 * kTileB;
  const int gw = wave & 3, gtid = tid & 255;
  if (grp == 1 && piece == 0 && a.kn != nullptr) copy_tile_rows<T, D, kCols>(a, kvh, ctile, gtid);
  const int64_t slot = ((int64_t)kvh * a.col_tiles + ctile) * a.splits + piece;
  prefill_run<T, T, D, BK, NQB, false, kRunSplit, 4>(
      a, kvh, ctile, grp == 0 ? tb : mid, grp == 0 ? mid : te, gsmem, (float*)smem, part_st, gw,
      gtid, bar, gw, -1, false, grp == 0 ? nullptr : a.part_o + slot * kCols * D,
      grp == 0 ? nullptr : a.part_st + slot * kCols);
}

// sigmoid(g) as the kernels that the pieces stand in for form it.
template <typename T>
__device__ __forceinline__ float gate_factor(T g) {
  if constexpr (sizeof(T) == 4)
    return stable_sigmoid(g);
  else
    return fast_sigmoid(to_f32(g));
}

// Merges the pieces of prefill_split or prefill_f32: one block per (kv head,
// column tile, 16 columns), the O fragments of the 16 columns shared out over
// its four waves.  Each piece weighs 2^(mc - M), M the largest offset among
// the column's pieces that saw a key; the gate is applied before the
// rounding.
template <typename T, typename TO, int D, int BK, int NQB>
__global__ void __launch_bounds__(256)
prefill_combine(PrefillArgs a) {
  constexpr int kCols = 64 * NQB;
  constexpr int MB = D / 16;
  constexpr int MW = MB / 4;            // fragments per wave
  constexpr int kGroup = D == 256 ? 4 : 8;  // pieces whose loads are in flight together
  typedef typename Vec4<T>::type V4;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int hl = lane & 15, quad = lane >> 4;
  const int sub = blockIdx.x % (4 * NQB);  // 16-column slice of the column tile
  const int ct = blockIdx.x / (4 * NQB);   // kvh * col_tiles + ctile
  const int kvh = ct / a.col_tiles, ctile = ct - kvh * a.col_tiles;
  const int col = ctile * kCols + 16 * sub + hl;
  if (ctile * kCols + 16 * sub >= a.q_tokens * a.group) return;  // wave-uniform
  int lo, hi, nt;
  tile_keys<BK, kCols>(a, ctile, lo, hi, nt);
  const int cnt = max(1, (nt + a.split_tiles - 1) / a.split_tiles);
  const int64_t slot0 = (int64_t)ct * a.splits;
  const f32x4* po = (const f32x4*)(a.part_o + slot0 * kCols * D) + (sub * MB + w * MW) * 64 + lane;
  const float2* ps = a.part_st + slot0 * kCols + 16 * sub + hl;
  float M = -INFINITY, L = 0.f;
  f32x4 o[MW];
#pragma unroll
  for (int i = 0; i < MW; ++i) o[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < cnt; s0 += kGroup) {
    float2 st[kGroup];
    f32x4 x[kGroup][MW];
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      const int s = min(s0 + u, cnt - 1);
      st[u] = ps[(int64_t)s * kCols];
#pragma unroll
      for (int i = 0; i < MW; ++i) x[u][i] = po[(int64_t)s * (kCols * D / 4) + i * 64];
    }
    float mg = M;
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      if (s0 + u >= cnt) st[u].x = -INFINITY;
      mg = fmaxf(mg, st[u].x);
    }
    const float keep = M == -INFINITY ? 0.f : fast_exp2(M - mg);
    L *= keep;
#pragma unroll
    for (int i = 0; i < MW; ++i) o[i] *= keep;
#pragma unroll
    for (int u = 0; u < kGroup; ++u) {
      if (s0 + u >= cnt) continue;  // the last piece again: 0 times its infinities is a NaN
      const float wt = st[u].x == -INFINITY ? 0.f : fast_exp2(st[u].x - mg);
      L += wt * st[u].y;
#pragma unroll
      for (int i = 0; i < MW; ++i) o[i] += wt * x[u][i];
    }
    M = mg;
  }
  if (col >= a.q_tokens * a.group) return;
  const float inv = L > 0.f ? 1.0f / L : 0.f;
  const int tok = col / a.group, hq = kvh * a.group + (col - tok * a.group);
  const int64_t row = (int64_t)tok * a.q_heads + hq;
  const int d0 = 16 * MW * w + 4 * quad;
  TO* op = (TO*)a.out + row * D + d0;
#pragma unroll
  for (int i = 0; i < MW; ++i) {
    if (a.gate != nullptr) {
      const V4 g = *(const V4*)((const T*)a.gate + row * a.gate_stride + d0 + 16 * i);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        op[16 * i + e] = from_f32<TO>(o[i][e] * inv * gate_factor<T>(g[e]));
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) op[16 * i + e] = from_f32<TO>(o[i][e] * inv);
    }
  }
}

template <typename T>
const void* pick_split(int D) {
  switch (D) {
    case 64: return (const void*)prefill_split<T, 64, 64, 2>;
    case 128: return (const void*)prefill_split<T, 128, 64, 2>;
    case 256: return (const void*)prefill_split<T, 256, 32, 1>;
  }
  return nullptr;
}

template <typename T, typename TO>
const void* pick_combine(int D) {
  constexpr bool f32 = sizeof(T) == 4;  // the tiles of prefill_f32
  switch (D) {
    case 64: return (const void*)prefill_combine<T, TO, 64, f32 ? 32 : 64, f32 ? 1 : 2>;
    case 128: return (const void*)prefill_combine<T, TO, 128, f32 ? 32 : 64, f32 ? 1 : 2>;
    case 256: return (const void*)prefill_combine<T, TO, 256, f32 ? 16 : 32, 1>;
  }
  return nullptr;
}

template <typename T>
const void* pick_combine_out(int D, int out_dtype) {
  switch (out_dtype) {
    case ALPX_F32: return pick_combine<T, float>(D);
    case ALPX_F16: return pick_combine<T, f16_t>(D);
    default: return pick_combine<T, bf16_t>(D);
  }
}

}  // namespace

const void* prefill_split_kernel(int dtype, int head_dim) {
  return dtype == ALPX_F16 ? pick_split<f16_t>(head_dim) : pick_split<bf16_t>(head_dim);
}

const void* prefill_combine_kernel(int dtype, int head_dim, int out_dtype) {
  if (dtype == ALPX_F32) return pick_combine_out<float>(head_dim, out_dtype);
  return dtype == ALPX_F16 ? pick_combine_out<f16_t>(head_dim, out_dtype)
                           : pick_combine_out<bf16_t>(head_dim, out_dtype);
}

}  // namespace alpx
