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

// whether the tiled kernels store a's output through LDS (their epilogue's
// conditions, bmm_wide.h)
inline bool staged_output(const FastArgs& a) {
  const bool bias16 = (a.bias_dtype == kBF16 || a.bias_dtype == kF16) && a.sbiasn == 1 && a.sbiasm % 4 == 0 &&
                      a.sbiasb % 4 == 0 && (reinterpret_cast<uintptr_t>(a.bias) & 7) == 0;
  return (a.c_dtype == kBF16 || a.c_dtype == kF16) && (a.bias == nullptr || bias16) && a.n % 8 == 0 &&
         a.scm % 8 == 0 && a.scb % 8 == 0 && (reinterpret_cast<uintptr_t>(a.c) & 15) == 0;
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

// Up to one 64 x 64 tile per CU the K-split kernel is ahead of the tiled ones,
// whose workgroups then walk K one step after the other on part of the chip;
// beyond, each operand byte is loaded for 64 outputs instead of 128. With two
// K steps there is little to split: the line is lower where the waves' sums
// meet once (channel, tensor). From 32 steps on it pays up to two tiles per CU
// when the weight comes from HBM, except where the operands' majors differ in
// block mode; so it does with at most 32 rows (smaller tiles here, padding
// there) and with outputs that the tiled kernels store element by element.
// MI355X, us with the operands in L2 / from HBM, tiled (128 x 128
// tiles) -> here, block scales and N-major B unless said:
//   16 x 14336 x 4096   30.6 / 40.2 -> 17.1 / 21.0
//   256 x 2048 x 1024    8.3 / 10.5 ->  5.8 /  6.0
//   1024 x 1024 x 256    4.7 /  5.2 ->  4.8 /  4.8   (one tile per CU; tensor 6.0 / 6.3 -> 7.0 / 6.9)
//   512 x 2048 x 4096   22.9 / 41.0 -> 19.1 / 23.3
//   128 x 14336 x 1024   8.6 / 14.8 -> 17.5 / 19.5   (1.75 per CU; K-major B 8.3 / 12.8 -> 10.9 / 12.9)
//   512 x 4096 x 4096   29.3 / 40.4 -> 52.8 / 58.4   (two; K-major B 28.2 / 37.6 -> 31.9 / 33.6,
//                       channel, K-major B 24.7 / 34.5 -> 28.5 / 28.3)
//   512 x 4096 x 256, fp32 output 21.8 -> 11.1, fp8 26.3 -> 9.3; 512 x (16 x 64 x 256) 17.1 -> 4.1
bool bmm_split_pays(const FastArgs& a, bool a_k, bool b_k, int mode, int64_t batch, hipStream_t st) {
  const int64_t t = bmmp::tiles(a, batch, 64, 64), cus = device_cu_count(st);
  const bool deep = a.k >= 32 * bmmp::BK && (mode != 0 || a_k == b_k);
  if (deep || a.m <= 32 || !bmmp::staged_output(a)) return t <= 2 * cus;
  return mode != 0 && a.k <= 2 * bmmp::BK ? 4 * t <= 3 * cus : t <= cus;
}

// Operands that the tiled kernels do not take: the general kernel is slower
// wherever it gathers bytes (rows not 16-byte aligned), folds block scales, or
// has few of its 128 x 128 tiles. On aligned rows (K no multiple of 4, or
// ragged and below 128) and more than six 64 x 64 tiles per CU it is ahead
// with one scale, and with channel scales over eight or more K steps unless
// both operands are K-major. MI355X, us, general / here, MN-major operands:
// tensor 4096 x 4096 x 1031 86.8 / 129, 2048 x 3072 x 1031 46.6 / 49.1, 2048 x 2048 x
// 1031 35.6 / 32.8, 8192 x 8192 x 64 182 / 250; channel 4096 x 4096 x 1031 138 / 155
// (K-major 1.00 : 0.89), 4096 x 4096 x 515 1 : 0.9; block 4096 x 4096 x 1031 205 / 95.
bool bmm_split_over_general(const FastArgs& a, bool a_k, bool b_k, int mode, bool aligned_rows, int64_t batch,
                            hipStream_t st) {
  if (!aligned_rows || mode == 0 || bmmp::tiles(a, batch, 64, 64) <= 6 * int64_t(device_cu_count(st))) return true;
  return mode == 1 && ((a_k && b_k) || a.k < 8 * bmmp::BK);
}

int bmm_split_launch(const FastArgs& a, bool a_k, bool b_k, int mode, int64_t batch, hipStream_t st) {
  using namespace bmmp;
  if (a_k && b_k) return launch_mode<true, true>(a, mode, batch, st);
  if (a_k) return launch_mode<true, false>(a, mode, batch, st);
  if (b_k) return launch_mode<false, true>(a, mode, batch, st);
  return launch_mode<false, false>(a, mode, batch, st);
}

}  // namespace pcamd
