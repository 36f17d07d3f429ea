// Causal prefill for float32 queries and caches (head_dim 64, 128 or 256),
// float32 products and sums throughout.
#include "prefill_run.h"

namespace alpx {
namespace {

// Key rows per tile: K and V tiles, double buffered, leave room for two
// blocks per CU (four at head_dim 64).
constexpr int f32_tile_keys(int d) { return d == 256 ? 16 : 32; }

// A block owns 64 query columns ((token, query head) pairs of one kv head),
// 16 per wave, on v_mfma_f32_16x16x4_f32.  As in the float32 decode, both
// products run in a permuted order that lets a lane feed what it holds:
//   S^T = K Q^T, k-step (g, j): lane (hl, quad) supplies K[row hl][16 g +
//     4 quad + j] (one 16-byte LDS read per g) and Q[column hl][same d];
//   O^T = V^T P^T, k-step (blk, i): lane supplies P[16 blk + 4 quad + i]
//     [column hl], its own score, and V[that row][16 mb + hl].
// K and V tiles go straight to LDS (row-major, 16-byte unit u of row r at
// u ^ (r mod 16) for K and u ^ 4 ((r / 4) mod 4) for V, which keeps both
// read patterns off each other's banks).
//
// Bound by the matrix cores: the f32 MFMA is 1/16 the bf16 rate, so the LDS
// reads and the softmax fit beside the other waves' products (32/8 heads,
// 1000 tokens on 4096 rows: 119 TFLOP/s at head_dim 64, 125 at 128, where
// a library product reaches 153).  1000 tokens on no prefix at head_dim 64
// take 51 us, the heaviest blocks' 32 tiles in series; the decode machinery
// (one token per "sequence", 4 of 16 MFMA columns live) took 243.  Two
// wave groups per block, each on half of its keys, measured 46 there and
// 27% slower at head_dim 128.
template <typename TO, int D, bool SPLIT>
__global__ void __launch_bounds__(256, 2)
prefill_f32(PrefillArgs a) {
  constexpr int BK = f32_tile_keys(D);
  constexpr int NB = BK / 16;
  constexpr int U = D / 4;           // 16-byte units per row
  constexpr int kRowB = D * 4;
  constexpr int kTileB = BK * kRowB;
  constexpr int kIW = BK * U / 256;  // direct-load instructions per wave per tile
  constexpr int MB = D / 16;
  __shared__ __attribute__((aligned(1024))) char smem[4 * kTileB];  // K 0, 1, V 0, 1
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int hl = lane & 15, quad = lane >> 4;
  int kvh, ctile, piece = 0;
  if constexpr (SPLIT) {
    const int item = (blockIdx.x % kXcds) * a.per_xcd + blockIdx.x / kXcds;
    const int per_head = a.col_tiles * a.splits;
    if (item >= a.kv_heads * per_head) return;
    kvh = item / per_head;
    piece = (item - kvh * per_head) / a.col_tiles;
    ctile = a.col_tiles - 1 - (item - kvh * per_head - piece * a.col_tiles);
  } else {
    if (!prefill_work(a, kvh, ctile)) return;
  }
  int lo, hi, nt;
  tile_keys<BK, 64>(a, ctile, lo, hi, nt);
  int tb = 0, te = nt;
  if constexpr (SPLIT) {
    tb = piece * a.split_tiles;
    if (piece > 0 && tb >= nt) return;  // this column tile has fewer pieces
    te = min(tb + a.split_tiles, nt);
  }

  const int G = a.group, cols = a.q_tokens * G;
  const int wcol0 = ctile * 64 + 16 * wave;
  const bool cok = wcol0 + hl < cols;
  const int col = cok ? wcol0 + hl : cols - 1;
  const int tok = col / G, hq = kvh * G + (col - tok * G);
  const int rel0 = (int)(a.pos0 - a.kv_start);
  const int wt_first = min(wcol0, cols - 1) / G, wt_last = (min(wcol0 + 16, cols) - 1) / G;
  const int qrel = rel0 + tok;  // sees keys j <= qrel (and > qrel - window)

  f32x4 qv[MB];  // Q[column][16 g + 4 quad + 0..3]
  {
    const float* qp = (const float*)a.q + ((int64_t)tok * a.q_heads + hq) * a.q_stride + 4 * quad;
#pragma unroll
    for (int g = 0; g < MB; ++g) qv[g] = *(const f32x4*)(qp + 16 * g);
  }
  f32x4 o[MB];  // O^T[d = 16 mb + 4 quad + i][column]
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) o[mb] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // m: the column's reference max (moved only when a score exceeds it by
  // more than kRescale, so P <= 2^kRescale); l: this lane's share of the sum
  float m = -INFINITY, l = 0.f;

  uint32_t kofs[kIW], vofs[kIW];
#pragma unroll
  for (int t = 0; t < kIW; ++t) {
    const int sl = (wave * kIW + t) * 64 + lane;
    const int row = sl / U, u = sl % U;
    kofs[t] = (uint32_t)((int64_t)row * a.ks_pos * 4 + 16 * (u ^ (row & 15)));
    vofs[t] = (uint32_t)((int64_t)row * a.vs_pos * 4 + 16 * (u ^ (4 * ((row >> 2) & 3))));
  }
  const float* kg = (const float*)a.k + (int64_t)kvh * D;
  const float* vg = (const float*)a.v + (int64_t)kvh * D;
  const uint32_t lbase = (uint32_t)(uintptr_t)(lds_void_t*)smem;
  auto load_tile = [&](const float* g, int64_t pos, const uint32_t (&ofs)[kIW], int t, int buf) {
    const int k0 = lo + t * BK;  // rows no column sees (at or past hi) read as zero
    const i32x4 r = rsrc_words((uint64_t)(uintptr_t)(g + (int64_t)k0 * pos),
                               (uint32_t)((int64_t)(hi - k0) * pos * 4));
    const uint32_t lds0 = lbase + buf * kTileB + wave * kIW * 1024;
#pragma unroll
    for (int i = 0; i < kIW; ++i) lds_dma16(r, lds0 + i * 1024, ofs[i]);
  };
  // V element (row 16 blk + 4 quad + i, channel 16 (4 x + y) + hl): unit
  // 16 x + 4 y + hl / 4, stored at 16 x + 4 (y ^ quad) + hl / 4
  int vadr[4];
#pragma unroll
  for (int y = 0; y < 4; ++y) vadr[y] = 4 * quad * kRowB + 64 * (y ^ quad) + 4 * hl;

  if (tb < te) {
    load_tile(kg, a.ks_pos, kofs, tb, 0);
    load_tile(vg, a.vs_pos, vofs, tb, 2);
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();
  for (int j = tb; j < te; ++j) {
    const int cur = (j - tb) & 1;
    if (j + 1 < te) {
      load_tile(kg, a.ks_pos, kofs, j + 1, cur ^ 1);
      load_tile(vg, a.vs_pos, vofs, j + 1, 2 + (cur ^ 1));
    }
    const int k0 = lo + j * BK;
    // tiles past the wave's diagonal (or before its window) hold nothing for it
    if (k0 <= rel0 + wt_last && (a.window <= 0 || k0 + BK - 1 > rel0 + wt_first - a.window)) {
      const char* kt = smem + cur * kTileB;
      const char* vt = smem + (2 + cur) * kTileB;
      f32x4 s[NB];
#pragma unroll
      for (int blk = 0; blk < NB; ++blk) s[blk] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int g = 0; g < MB; ++g) {
        f32x4 ka[NB];
#pragma unroll
        for (int blk = 0; blk < NB; ++blk)
          ka[blk] = *(const f32x4*)(kt + (16 * blk + hl) * kRowB + 16 * ((4 * g + quad) ^ hl));
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
          for (int blk = 0; blk < NB; ++blk) s[blk] = mfma16x16x4(ka[blk][e], qv[g][e], s[blk]);
      }
      const bool edge = k0 + BK - 1 > rel0 + wt_first || k0 + BK > hi ||
                        (a.window > 0 && k0 <= rel0 + wt_last - a.window);
      float mx = -INFINITY;
#pragma unroll
      for (int blk = 0; blk < NB; ++blk)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          float x = s[blk][i] * a.scale_log2;
          if (edge) {
            const int key = k0 + 16 * blk + 4 * quad + i;
            if (!(key < hi && key <= qrel && (a.window <= 0 || key > qrel - a.window)))
              x = -INFINITY;
          }
          s[blk][i] = x;
          mx = fmaxf(mx, x);
        }
      if (__ballot(mx > m + kRescale) != 0) {
        mx = fmaxf(mx, __shfl_xor(mx, 16));
        mx = fmaxf(mx, __shfl_xor(mx, 32));
        if (mx > m + kRescale) {
          const float c = fast_exp2(m - mx);  // 0 while m is -inf
          l *= c;
#pragma unroll
          for (int mb = 0; mb < MB; ++mb) o[mb] *= c;
          m = mx;
        }
      }
      // O and l take a tile's sum at a time: over a long key range that
      // halves the rounding error of adding every key to the running sum
      const float off = m == -INFINITY ? 0.f : m;
      float ps = 0.f;
#pragma unroll
      for (int blk = 0; blk < NB; ++blk)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          s[blk][i] = fast_exp2(s[blk][i] - off);
          ps += s[blk][i];
        }
      l += ps;
#pragma unroll
      for (int mb = 0; mb < MB; mb += 4) {
        f32x4 t[4];
#pragma unroll
        for (int y = 0; y < 4; ++y) t[y] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int blk = 0; blk < NB; ++blk)
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
              const float va = *(const float*)(vt + vadr[y] + (16 * blk + i) * kRowB + 64 * mb);
              t[y] = mfma16x16x4(va, s[blk][i], t[y]);
            }
        if (edge) {
          // a row that one column sees and another does not: if it holds an
          // infinity or a NaN, 0 times it must not reach the other, so each
          // token's columns take the product over their own rows alone
          bool bad = false;
#pragma unroll
          for (int y = 0; y < 4; ++y)
#pragma unroll
            for (int i = 0; i < 4; ++i) bad |= !(fabsf(t[y][i]) < INFINITY);
          if (__ballot(bad) != 0) {
#pragma unroll
            for (int y = 0; y < 4; ++y)
#pragma clang loop unroll(disable)
              for (int wt = wt_first; wt <= wt_last; ++wt) {
                f32x4 u = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int blk = 0; blk < NB; ++blk)
#pragma unroll
                  for (int i = 0; i < 4; ++i) {
                    const int key = k0 + 16 * blk + 4 * quad + i;
                    const bool seen =
                        key <= rel0 + wt && (a.window <= 0 || key > rel0 + wt - a.window);
                    const float va =
                        *(const float*)(vt + vadr[y] + (16 * blk + i) * kRowB + 64 * mb);
                    u = mfma16x16x4(seen ? va : 0.f, s[blk][i], u);
                  }
                if (tok == wt) t[y] = u;
              }
          }
        }
#pragma unroll
        for (int y = 0; y < 4; ++y) o[mb + y] += t[y];
      }
    }
    __builtin_amdgcn_s_waitcnt(0);  // the next tiles are in LDS
    __syncthreads();
  }

  l += __shfl_xor(l, 16);
  l += __shfl_xor(l, 32);
  if constexpr (SPLIT) {
    const int64_t slot = ((int64_t)kvh * a.col_tiles + ctile) * a.splits + piece;
    if (wcol0 >= cols) return;
    f32x4* po = (f32x4*)(a.part_o + slot * 64 * D) + wave * MB * 64 + lane;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) po[mb * 64] = o[mb];
    if (quad == 0) a.part_st[slot * 64 + 16 * wave + hl] = make_float2(m, l);
    return;
  }
  if (!cok) return;
  const float inv = l > 0.f ? 1.0f / l : 0.f;
  const int64_t row = (int64_t)tok * a.q_heads + hq;
  TO* op = (TO*)a.out + row * D + 4 * quad;
  const float* gp = (const float*)a.gate + row * a.gate_stride + 4 * quad;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    f32x4 r = o[mb] * inv;
    if (a.gate != nullptr) {
      const f32x4 g = *(const f32x4*)(gp + 16 * mb);
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] *= stable_sigmoid(g[i]);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) op[16 * mb + i] = from_f32<TO>(r[i]);
  }
}

template <typename TO>
const void* pick_f32(int D) {
  switch (D) {
    case 64: return (const void*)prefill_f32<TO, 64, false>;
    case 128: return (const void*)prefill_f32<TO, 128, false>;
    case 256: return (const void*)prefill_f32<TO, 256, false>;
  }
  return nullptr;
}

}  // namespace

const void* prefill_f32_kernel(int head_dim, int out_dtype, bool split) {
  if (split) {
    switch (head_dim) {
      case 64: return (const void*)prefill_f32<float, 64, true>;
      case 128: return (const void*)prefill_f32<float, 128, true>;
      case 256: return (const void*)prefill_f32<float, 256, true>;
    }
    return nullptr;
  }
  switch (out_dtype) {
    case ALPX_F32: return pick_f32<float>(head_dim);
    case ALPX_F16: return pick_f32<f16_t>(head_dim);
    default: return pick_f32<bf16_t>(head_dim);
  }
}

}  // namespace alpx
