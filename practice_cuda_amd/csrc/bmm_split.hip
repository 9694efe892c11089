// bmm_split.hip - the instantiations of the K-split kernel (bmm_split.h), the
// rule that sends a product to it, and the choice of its tile.
#include "bmm_split.h"

namespace pcamd {
namespace bmmp {

// 16 x 16 sub-tiles (MI x NJ) and waves of a workgroup
enum Shape { k1x2w8, k1x4w4, k1x4w8, k2x2w8, k2x4w4, k2x4w8, k4x4w4, k4x4w8 };
struct Tile { int rows, cols, threads; };
constexpr Tile kTiles[] = {{16, 32, 512}, {16, 64, 256}, {16, 64, 512}, {32, 32, 512},
                           {32, 64, 256}, {32, 64, 512}, {64, 64, 256}, {64, 64, 512}};

inline int64_t tiles(const FastArgs& a, int64_t batch, int rows, int cols) {
  return batch * ((a.m + rows - 1) / rows) * ((a.n + cols - 1) / cols);
}

// The largest tile that still gives about every CU a workgroup; with fewer
// workgroups than that the K loops of a few CUs are the whole time. Tiles
// taller than the rows there are only add loads. Eight waves per workgroup
// (twice the loads in flight, half the K steps per wave) where a CU gets one
// workgroup, four where it gets several. MI355X, block scales, us (operands
// rotating beyond the caches):
//   rows x N x K                 16x32   16x64   32x32   32x64   64x64 (8 waves / 4)
//   16 x 4096 x 4096               7.5     9.8     8.5    11.1    15.7 / 22.7
//   16 x 14336 x 4096             15.7    15.5    16.4    16.6    20.3 / 24.9  (16x64, 4 waves: 15.1)
//   128 x 2048 x 2048              6.6     6.2     5.8     7.1     9.8 / 13.7
//   512 x 1024 x 4096 (N-major)   26.2    24.0    19.2    15.5    20.7 / 29.0
//   512 x 4096 x 1024             17.8    24.3    14.1    15.5    12.0 / 11.1
inline Shape pick(const FastArgs& a, int64_t batch, int cus, bool block) {
  const int64_t enough = cus - cus / 5;
  if (a.m > 32) {
    const int64_t t = tiles(a, batch, 64, 64);
    if (t >= enough) return t <= cus ? k4x4w8 : k4x4w4;
  }
  if (a.m > 16) {
    const int64_t t = tiles(a, batch, 32, 64);
    if (t >= enough) return t <= cus ? k2x4w8 : k2x4w4;
    if (block) return k2x2w8;
  }
  if (tiles(a, batch, 16, 32) <= cus) return k1x2w8;
  return block ? k1x4w4 : k1x4w8;
}

template <bool A_K, bool B_K, int MODE>
int launch_shape(const FastArgs& a, int64_t batch, hipStream_t st) {
  constexpr bool BLOCK = MODE == 0;
  switch (pick(a, batch, device_cu_count(st), BLOCK)) {
    case k1x2w8: return launch_tile<A_K, B_K, MODE, 1, 2, 8>(a, batch, st);
    case k1x4w4:
      if constexpr (BLOCK) return launch_tile<A_K, B_K, MODE, 1, 4, 4>(a, batch, st);
      [[fallthrough]];
    case k1x4w8:
      if constexpr (!BLOCK) return launch_tile<A_K, B_K, MODE, 1, 4, 8>(a, batch, st);
      [[fallthrough]];
    case k2x2w8:
      if constexpr (BLOCK) return launch_tile<A_K, B_K, MODE, 2, 2, 8>(a, batch, st);
      [[fallthrough]];
    case k2x4w4: return launch_tile<A_K, B_K, MODE, 2, 4, 4>(a, batch, st);
    case k2x4w8: return launch_tile<A_K, B_K, MODE, 2, 4, 8>(a, batch, st);
    case k4x4w4: return launch_tile<A_K, B_K, MODE, 4, 4, 4>(a, batch, st);
    default: return launch_tile<A_K, B_K, MODE, 4, 4, 8>(a, batch, st);
  }
}

template <bool A_K, bool B_K>
int launch_mode(const FastArgs& a, int mode, int64_t batch, hipStream_t st) {
  if (mode == 1) return launch_shape<A_K, B_K, 1>(a, batch, st);
  if (mode == 2) return launch_shape<A_K, B_K, 2>(a, batch, st);
  return launch_shape<A_K, B_K, 0>(a, batch, st);
}

}  // namespace bmmp

bool bmm_split_ok(const FastArgs& a, int a_fmt, int b_fmt, bool a_k, bool b_k, int mode, int64_t batch,
                  hipStream_t st) {
  if (a_fmt != kE4M3 || b_fmt != kE4M3) return false;
  // a 16-byte piece must fit in the rows that are walked
  if (((a_k || b_k) && a.k < 16) || (!a_k && a.m < 16) || (!b_k && a.n < 16)) return false;
  // sizes rounded up to a tile, and a launch's threads, fit 32 bits (many small batches: the
  // general kernel's 128 x 128 tiles and 256 threads reach further)
  if (a.m > INT32_MAX - 64 || a.n > INT32_MAX - 64) return false;
  const bmmp::Tile t = bmmp::kTiles[bmmp::pick(a, batch, device_cu_count(st), mode == 0)];
  if (bmmp::tiles(a, batch, t.rows, t.cols) > UINT32_MAX / t.threads) return false;
  if (mode == 0) {
    if (a.qbk != 128 || a.qbm_shift < 0 || a.qbn_shift < 0) return false;
    const int64_t ra = int64_t((a.m - 1) >> a.qbm_shift) * a.ssa1, rb = int64_t((a.n - 1) >> a.qbn_shift) * a.ssb2;
    if (ra < 0 || rb < 0 || ra > UINT32_MAX || rb > UINT32_MAX) return false;
  }
  return true;
}

// Up to two 64 x 64 tiles per CU the K-split kernel is ahead of the tiled
// ones, whose few workgroups then walk K one step after the other (MI355X,
// block scales, tiled -> here, us: 16 x 14336 x 4096 50.1 -> 15.1, 16 x 1024 x
// 1024 9.9 -> 3.5, 128 x 14336 x 4096 52.3 -> 35.6, 512 x 1024 x 4096 40.3 ->
// 15.5, 512 x 4096 x 1024 12.9 -> 11.1); at four (4096 x 1024 x 512: 8.9 ->
// 13.9) it is behind: each operand byte is loaded for 64 outputs instead of
// 128 or 256.
bool bmm_split_pays(const FastArgs& a, int64_t batch, hipStream_t st) {
  return bmmp::tiles(a, batch, 64, 64) <= 2 * int64_t(device_cu_count(st));
}

int bmm_split_launch(const FastArgs& a, bool a_k, bool b_k, int mode, int64_t batch, hipStream_t st) {
  using namespace bmmp;
  if (a_k && b_k) return launch_mode<true, true>(a, mode, batch, st);
  if (a_k) return launch_mode<true, false>(a, mode, batch, st);
  if (b_k) return launch_mode<false, true>(a, mode, batch, st);
  return launch_mode<false, false>(a, mode, batch, st);
}

}  // namespace pcamd
