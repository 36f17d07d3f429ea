// Prefill kernels that give a block a light and a heavy column tile of one
// kv head (prefill.hip chooses them from the causal imbalance).
#include "prefill_run.h"

namespace alpx {
namespace {

// Work of a prefill_pair block: kv head kvh and the column tiles ta (light:
// earlier tokens) and tb = col_tiles - 1 - ta (heavy; equal to ta for the
// middle tile of an odd count).  Pairs are ordered kv-head-major and cut
// into 8 contiguous slices, slice x on XCD x, so one kv head's blocks share
// one XCD's L2.
__device__ __forceinline__ bool pair_work(const PrefillArgs& a, int& kvh, int& ta, int& tb) {
  const int b = blockIdx.x;
  const int item = (b % kXcds) * a.per_xcd + b / kXcds;
  const int pairs = (a.col_tiles + 1) / 2;
  if (item >= a.kv_heads * pairs) return false;
  kvh = item / pairs;
  ta = item - kvh * pairs;
  tb = a.col_tiles - 1 - ta;
  return true;
}

// Causal imbalance removed: one block of eight waves per CU takes a light
// and a heavy column tile of one kv head.  Waves 0-3 (group 0) run the
// light tile over all its key tiles, then the heavy tile over its key
// tiles [s, nt_b); waves 4-7 (group 1) run the heavy tile over [0, s),
// with s chosen so that both groups walk about the same number of tiles.
// Each group has its own four tile buffers and its own barrier, so the two
// groups' pipelines run independently (as two co-resident blocks would);
// at the end group 0 leaves its heavy-tile partial in its LDS and group 1
// merges it into its own (one block barrier) and writes the heavy tile.
template <typename T, typename TO, int D, int BK, int NQB>
__global__ void __launch_bounds__(512, 1)
prefill_pair(PrefillArgs a) {
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
  int kvh, ta, tbt;
  if (!pair_work(a, kvh, ta, tbt)) return;
  if (tid < 2) gctr[tid] = 0;
  __syncthreads();  // the group counters are zero before any group barrier
  int lo, hi, nta = 0, ntb;
  if (ta != tbt) tile_keys<BK, kCols>(a, ta, lo, hi, nta);
  tile_keys<BK, kCols>(a, tbt, lo, hi, ntb);
  // Group 0 also pays a second pipeline start: one tile's worth.
  const int split = min(ntb, (nta + ntb + (ta != tbt ? 1 : 0) + 1) / 2);
  GroupBarrier bar{gctr + grp, 0u};
  char* gsmem = smem + grp * 4 * kTileB;
  const int gw = wave & 3, gtid = tid & 255;
  if (grp == 0) {
    // the light tile, then the heavy tile's key tiles [split, nt_b)
    if (ta != tbt) {
      if (a.kn != nullptr) copy_tile_rows<T, D, kCols>(a, kvh, ta, gtid);
      prefill_run<T, TO, D, BK, NQB, false, kRunWrite, 4>(a, kvh, ta, 0, -1, gsmem, nullptr,
                                                          nullptr, gw, gtid, bar, gw, -1, false);
    }
    prefill_run<T, TO, D, BK, NQB, false, kRunPartial, 4>(a, kvh, tbt, split, -1, gsmem,
                                                          (float*)smem, part_st, gw, gtid, bar,
                                                          gw, -1, false);
  } else {
    // the heavy tile's key tiles [0, split), merged with group 0's part
    if (a.kn != nullptr) copy_tile_rows<T, D, kCols>(a, kvh, tbt, gtid);
    prefill_run<T, TO, D, BK, NQB, false, kRunMerge, 4>(a, kvh, tbt, 0, split, gsmem,
                                                        (float*)smem, part_st, gw, gtid, bar, gw,
                                                        -1, false);
  }
}

// One K/V tile stream for a light and a heavy column tile: one block of
// eight waves per CU takes column tile ta (waves 0-3) and its mirror
// tb = col_tiles - 1 - ta (waves 4-7) of one kv head.  Without a window
// both walk the key tiles from row 0, so one set of tile buffers, loaded
// by all eight waves, serves both tiles: half the direct-load bytes per
// FLOP of two four-wave blocks, which load the same tiles separately.  The
// loads' LDS writes and texture-path time are about a fifth of the
// four-wave kernel's loop at head_dim 128, where LDS reads (K operands at
// 244 B/clk per CU, transposing V reads at 131) and those writes come
// close to the MFMA time.  The light waves stop computing after their own
// last key tile and keep loading; the middle tile of an odd count goes to
// waves 4-7 alone.
template <typename T, typename TO, int D, int BK, int NQB>
__global__ void __launch_bounds__(512, 1)
prefill_shared(PrefillArgs a) {
  constexpr int kTileB = BK * D * (int)sizeof(T);
  constexpr int kCols = 64 * NQB;
  __shared__ __attribute__((aligned(1024))) char smem[4 * kTileB];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = wave >> 2;
  int kvh, ta, tbt;
  if (!pair_work(a, kvh, ta, tbt)) return;
  int lo, hi_b, ntb;
  tile_keys<BK, kCols>(a, tbt, lo, hi_b, ntb);
  if (a.kn != nullptr && (grp == 1 || ta != tbt))
    copy_tile_rows<T, D, kCols>(a, kvh, grp == 0 ? ta : tbt, tid & 255);
  auto bar = []() __attribute__((always_inline)) { __syncthreads(); };
  prefill_run<T, TO, D, BK, NQB, false, kRunWrite, 8>(a, kvh, grp == 0 ? ta : tbt, 0, -1, smem,
                                                      nullptr, nullptr, wave & 3, tid, bar, wave,
                                                      hi_b, grp == 0 && ta == tbt);
}

template <typename T, typename TO>
const void* pick_pair(int D) {
  switch (D) {
    case 64: return (const void*)prefill_pair<T, TO, 64, 64, 2>;
    case 128: return (const void*)prefill_pair<T, TO, 128, 64, 2>;
    case 256: return (const void*)prefill_pair<T, TO, 256, 32, 1>;
  }
  return nullptr;
}

template <typename T, typename TO>
const void* pick_shared(int D) {
  switch (D) {
    case 64: return (const void*)prefill_shared<T, TO, 64, 64, 2>;
    case 128: return (const void*)prefill_shared<T, TO, 128, 64, 2>;
    case 256: return (const void*)prefill_shared<T, TO, 256, 32, 1>;
  }
  return nullptr;
}

template <typename T>
const void* pick_shared_out(int D, int out_dtype) {
  switch (out_dtype) {
    case ALPX_F32: return pick_shared<T, float>(D);
    case ALPX_F16: return pick_shared<T, f16_t>(D);
    default: return pick_shared<T, bf16_t>(D);
  }
}

template <typename T>
const void* pick_pair_out(int D, int out_dtype) {
  switch (out_dtype) {
    case ALPX_F32: return pick_pair<T, float>(D);
    case ALPX_F16: return pick_pair<T, f16_t>(D);
    default: return pick_pair<T, bf16_t>(D);
  }
}

}  // namespace

const void* prefill_pair_kernel(int dtype, int head_dim, int out_dtype) {
  return dtype == ALPX_F16 ? pick_pair_out<f16_t>(head_dim, out_dtype)
                           : pick_pair_out<bf16_t>(head_dim, out_dtype);
}

const void* prefill_shared_kernel(int dtype, int head_dim, int out_dtype) {
  return dtype == ALPX_F16 ? pick_shared_out<f16_t>(head_dim, out_dtype)
                           : pick_shared_out<bf16_t>(head_dim, out_dtype);
}

}  // namespace alpx
