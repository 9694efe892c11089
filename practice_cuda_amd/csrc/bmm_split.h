// bmm_split.h - scaled FP8 BMM for products that cannot fill the chip with
// large tiles (few rows, narrow outputs, short grids) and for operands whose
// rows are not 16-byte aligned. The kernel and its launch templates;
// bmm_split.hip instantiates them.
//
// What bounds such a product is latency, not arithmetic: a 256 x 256 tile
// walks its K steps one after the other behind a barrier each, on a few CUs.
// Here a workgroup owns a small tile (16 MI x 16 NJ outputs) and its W waves
// split K: wave w computes the whole tile over K steps w, w + W, ... Each wave
// loads its own operands into registers, one of its steps ahead, so the K loop
// loads no operand through a barrier and every wait is on the wave's own loads.
// The W partial tiles meet in LDS and are summed in a fixed order (the result
// does not depend on timing).
//
// Operands (MFMA 16x16x128, operands swapped as in the other kernels: x = B,
// y = A, a lane holds 4 consecutive outputs of one row). Both layouts go global
// -> registers -> wave-private LDS -> fragments: neighbouring lanes load
// neighbouring 16-byte pieces (K-major: 8 rows x 128 bytes per instruction).
// Loading a K-major operand straight into fragments, 16 rows x 64 bytes with
// neighbouring lanes in different rows, streamed at 7 TB/s from L2 over the
// whole chip and was the limit (16 x 4096 x 4096, 64-column tiles: 13.2 us
// against 8.2 through LDS).
//   K-major operand: fragments are two ds_read_b128 per 16 rows.
//   MN-major operand: four ds_read_b64_tr_b8 (each transposes 8 x 16 bytes).
// Loads need no alignment (global loads of 16 bytes at any byte address). A
// row's last piece, where fewer than 16 bytes are left, is loaded 16 bytes
// before the row's end and shifted down, so no load leaves the operand.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "abi_util.h"
#include "bmm_epilogue.h"
#include "bmm_fast.h"
#include "fp8_common.h"

namespace pcamd {
namespace bmmp {

typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) v2i* lds_v2i_ptr;

constexpr int BK = 128;

struct __attribute__((packed)) Bytes16 { u32x4 v; };
PCAMD_DEV u32x4 load16(const uint8_t* base, uint32_t off) { return reinterpret_cast<const Bytes16*>(base + off)->v; }

// v >> 8 n bytes of the 128-bit value (little endian), zeros from the top; n >= 0, n >= 16 gives 0
PCAMD_DEV u32x4 shift_down(u32x4 v, int n) {
  const int words = n >> 2;
  u32x4 w;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    uint32_t x = 0;
#pragma unroll
    for (int j = i; j < 4; ++j) x = words == j - i ? v[j] : x;
    w[i] = x;
  }
  u32x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    o[i] = __builtin_amdgcn_alignbyte(i < 3 ? w[i + 1] : 0u, w[i], static_cast<uint32_t>(n & 3));
  return o;
}

// One wave's operand over one K step: 16 NB rows x 128 k.
template <bool KMAJOR, int NB>
struct Operand;

template <int NB>
struct Operand<true, NB> {
  // LDS tile: [row][8 chunks of 16 bytes], chunk c of row r at c ^ swz(r)
  static constexpr int PITCH = BK;
  static constexpr int LDS = 16 * NB * PITCH;
  static constexpr int INSTS = 2 * NB;  // 8 rows x 128 bytes each
  uint32_t off[INSTS];  // byte offset of this lane's row of each instruction
  const uint8_t* base;
  uint8_t* lds;
  int k, kc, row, chunk;
  struct Regs { u32x4 v[INSTS]; };
  static PCAMD_DEV int swz(int r) { return (((r >> 1) & 1) * 5) ^ ((r >> 2) & 1); }
  // rows past the operand re-read its last row: they feed outputs that are never stored
  PCAMD_DEV Operand(const uint8_t* b, uint32_t ld, int row0, int rows, int k_, int lane, uint8_t* l)
      : base(b), lds(l), k(k_), kc(16 * (lane & 7)), row(lane >> 3), chunk(lane & 7) {
#pragma unroll
    for (int i = 0; i < INSTS; ++i) off[i] = static_cast<uint32_t>(min(row0 + 8 * i + row, rows - 1)) * ld;
  }
  PCAMD_DEV void load(Regs& r, int k0) const {
    const uint32_t kk = static_cast<uint32_t>(min(k0 + kc, k - 16));
#pragma unroll
    for (int i = 0; i < INSTS; ++i) r.v[i] = load16(base, off[i] + kk);
  }
  // `last`: the step reaches past k
  PCAMD_DEV void frags(const Regs& r, v8i (&f)[NB], int k0, bool last, int lane) const {
    const int kk = k0 + kc, sh = kk - min(kk, k - 16);
#pragma unroll
    for (int i = 0; i < INSTS; ++i) {
      u32x4 v = r.v[i];
      if (last) v = shift_down(v, sh);
      *reinterpret_cast<u32x4*>(lds + (8 * i + row) * PITCH + ((chunk ^ swz(row)) << 4)) = v;
    }
    const int g = lane >> 4, j = lane & 15, s = swz(j);
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const u32x4* p = reinterpret_cast<const u32x4*>(lds + (16 * i + j) * PITCH);
      const u32x4 x = p[(2 * g) ^ s], y = p[(2 * g + 1) ^ s];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        f[i][w] = static_cast<int>(x[w]);
        f[i][4 + w] = static_cast<int>(y[w]);
      }
    }
  }
};

template <int NB>
struct Operand<false, NB> {
  // LDS tile: [k][NB chunks of 16 bytes], chunk c of k row k at c ^ swz(k).
  // A transposing read touches 8 k rows of one chunk per 16-lane group; with
  // 64-byte rows, swz sends rows 4 apart, and the groups 16 rows apart, to
  // different 16-byte slots of the 256 bytes the LDS serves per cycle.
  static constexpr int PITCH = 16 * NB;
  static constexpr int LDS = BK * PITCH;
  static constexpr int ROWS = 64 / NB;   // k rows per load instruction
  static constexpr int INSTS = 2 * NB;
  const uint8_t* base;
  uint8_t* lds;
  uint32_t col;      // this lane's column offset (clamped into the row)
  uint32_t ld;
  int shift;         // bytes its piece lies before its columns (last column tile)
  int k, krow, chunk;
  struct Regs { u32x4 v[INSTS]; };
  static PCAMD_DEV int swz(int r) {
    const int far = ((r >> 5) ^ (r >> 6)) & 1;
    return NB == 8 ? ((r >> 1) & 3) | (far << 2) : NB == 4 ? ((r >> 2) & 1) | (far << 1) : 0;
  }
  PCAMD_DEV Operand(const uint8_t* b, uint32_t ld_, int col0, int cols, int k_, int lane, uint8_t* l)
      : base(b), lds(l), ld(ld_), k(k_), krow(lane / NB), chunk(lane % NB) {
    const int c = col0 + 16 * chunk, cc = min(c, cols - 16);
    col = static_cast<uint32_t>(cc);
    shift = c - cc;
  }
  PCAMD_DEV void load(Regs& r, int k0) const {
#pragma unroll
    for (int i = 0; i < INSTS; ++i) {
      const int kk = min(k0 + ROWS * i + krow, k - 1);
      r.v[i] = load16(base, static_cast<uint32_t>(kk) * ld + col);
    }
  }
  PCAMD_DEV void frags(const Regs& r, v8i (&f)[NB], int k0, bool last, int lane) const {
#pragma unroll
    for (int i = 0; i < INSTS; ++i) {
      const int row = ROWS * i + krow;
      u32x4 v = r.v[i];
      if (shift > 0) v = shift_down(v, shift);
      if (last && k0 + row >= k) v = u32x4{0u, 0u, 0u, 0u};
      *reinterpret_cast<u32x4*>(lds + row * PITCH + ((chunk ^ swz(row)) << 4)) = v;
    }
    const int g = lane >> 4, j = lane & 15;
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const int row = 32 * g + 8 * q + (j >> 1);
        const uint8_t* p = lds + row * PITCH + ((i ^ swz(row)) << 4) + ((j & 1) << 3);
        const v2i v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_v2i_ptr)(p));
        f[i][2 * q] = v[0];
        f[i][2 * q + 1] = v[1];
      }
  }
};

PCAMD_DEV v4f mfma(const v8i& x, const v8i& y, const v4f& c) {
  return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(x, y, c, 0, 0, 0, 0, 0, 0);
}

PCAMD_DEV float bias_at(const FastArgs& a, int64_t off) {
  if (a.bias_dtype == kF32) return static_cast<const float*>(a.bias)[off];
  if (a.bias_dtype == kBF16)
    return __uint_as_float(static_cast<uint32_t>(static_cast<const uint16_t*>(a.bias)[off]) << 16);
  return static_cast<float>(static_cast<const _Float16*>(a.bias)[off]);
}

// bias, activation and the rounding to C's type for outputs (mm, nn .. nn + 3),
// in the reference's order (kernels/bmm/per_block.py:113-137)
PCAMD_DEV void store4(const FastArgs& a, int bidx, int mm, int nn, float (&v)[4]) {
  if (mm >= a.m || nn >= a.n) return;
  const int nv = min(4, a.n - nn);
  if (a.bias) {
    const int64_t off = bidx * a.sbiasb + int64_t(mm) * a.sbiasm + int64_t(nn) * a.sbiasn;
    const uint16_t* p = static_cast<const uint16_t*>(a.bias) + off;
    if (nv == 4 && a.sbiasn == 1 && a.bias_dtype != kF32 && (reinterpret_cast<uintptr_t>(p) & 7) == 0) {
      const uint2 h = *reinterpret_cast<const uint2*>(p);
      const bool bf = a.bias_dtype == kBF16;
      v[0] += bf ? bf16_lo(h.x) : f16_lo(h.x);
      v[1] += bf ? bf16_hi(h.x) : f16_hi(h.x);
      v[2] += bf ? bf16_lo(h.y) : f16_lo(h.y);
      v[3] += bf ? bf16_hi(h.y) : f16_hi(h.y);
    } else {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r < nv) v[r] += bias_at(a, off + int64_t(r) * a.sbiasn);
    }
  }
  if (a.act == PCAMD_ACT_GELU) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = 0.5f * v[r] * (1.0f + erff(v[r] * 0.7071067811865475f));
  }
  const int64_t o = bidx * a.scb + int64_t(mm) * a.scm + nn;
  if (a.c_dtype == kBF16 || a.c_dtype == kF16) {
    const bool h = a.c_dtype == kF16;
    uint16_t* p = static_cast<uint16_t*>(a.c) + o;
    const uint2 w = make_uint2(pack16_pair<OUT16_RUNTIME>(v[0], v[1], h), pack16_pair<OUT16_RUNTIME>(v[2], v[3], h));
    if (nv == 4 && (reinterpret_cast<uintptr_t>(p) & 7) == 0) {
      *reinterpret_cast<uint2*>(p) = w;
    } else {
      const uint32_t e[4] = {w.x & 0xFFFFu, w.x >> 16, w.y & 0xFFFFu, w.y >> 16};
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r < nv) p[r] = static_cast<uint16_t>(e[r]);
    }
  } else if (a.c_dtype == kF32) {
    float* p = static_cast<float*>(a.c) + o;
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < nv) p[r] = v[r];
  } else {
    uint8_t* p = static_cast<uint8_t*>(a.c) + o;
    const float hi = a.c_dtype == kE5M2 ? 57344.0f : 448.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = clamp_sym(v[r], hi);
    const uint32_t w = a.c_dtype == kE5M2 ? hw_pack4<kE5M2>(v[0], v[1], v[2], v[3])
                                          : hw_pack4<kE4M3>(v[0], v[1], v[2], v[3]);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (r < nv) p[r] = static_cast<uint8_t>(w >> (8 * r));
  }
}

// LDS writes before it are visible to the workgroup's reads after it; loads
// from global memory stay in flight across it (__syncthreads would be as well
// for LDS alone, but leaves that to the compiler's model of global memory).
PCAMD_DEV void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// MODE: 0 block (quant-K 128), 1 channel, 2 tensor.
//
// Block mode keeps the order of the other block-scaled kernels, acc =
// fma(P_k, sa * sb, acc) over k = 0, 1, ..., so its results are theirs bit for
// bit (the product of a quantized activation equals the fused call's): each
// round, the waves put the W partials P_k into LDS and every thread folds its
// outputs over them in k order. Channel and tensor mode sum each wave's steps
// in the MFMA and meet once at the end.
template <bool A_K, bool B_K, int MODE, int MI, int NJ, int W>
__global__ __launch_bounds__(64 * W, 1) void bmm_split_kernel(FastArgs a) {
  using OA = Operand<A_K, MI>;
  using OB = Operand<B_K, NJ>;
  constexpr int TILE = MI * NJ * 1024;             // one fp32 tile
  constexpr int OPS = OA::LDS + OB::LDS;           // a wave's operands of one K step
  constexpr int STAGE = OPS > TILE ? OPS : TILE;   // ... and, after them, its partial tile
  constexpr int ROWS = 16 * MI, COLS = 16 * NJ, CH = 4 * NJ;
  constexpr int SCALES = MODE == 0 ? W * (ROWS + COLS) * 4 : 0;
  __shared__ __attribute__((aligned(16))) uint8_t smem[W * STAGE + SCALES];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane & 15, lg = lane >> 4;

  // Consecutive tiles (rows fastest) on one XCD, so the row blocks that share
  // a column panel of B read it through one L2; blockIdx % 8 picks the XCD.
  const int T = a.total_tiles, xcd = blockIdx.x & 7;
  const int pid = xcd * (T >> 3) + min(xcd, T & 7) + (blockIdx.x >> 3);
  const int bidx = __builtin_amdgcn_readfirstlane(pid / a.tiles_per_batch);
  const int tile = pid - bidx * a.tiles_per_batch;
  const int tn = __builtin_amdgcn_readfirstlane(tile / a.tiles_m);
  const int m0 = __builtin_amdgcn_readfirstlane((tile - tn * a.tiles_m) * ROWS);
  const int n0 = tn * COLS;

  uint8_t* mine = smem + wave * STAGE;
  const OA oa(a.a + bidx * a.sab, a.lda, m0, a.m, a.k, lane, mine);
  const OB ob(a.b + bidx * a.sbb, a.ldb, n0, a.n, a.k, lane, mine + OA::LDS);

  // Block scales of a K step: lane l brings row l's and column l's. Their
  // offsets within the batch's scale matrices fit 32 bits (checked on the host).
  const float* const sa_b = a.sa + bidx * a.ssab;
  const float* const sb_b = a.sb + bidx * a.ssbb;
  uint32_t sao = 0, sbo = 0;
  if constexpr (MODE == 0) {
    sao = static_cast<uint32_t>(min(m0 + min(lane, ROWS - 1), a.m - 1) >> a.qbm_shift) * static_cast<uint32_t>(a.ssa1);
    sbo = static_cast<uint32_t>(min(n0 + min(lane, COLS - 1), a.n - 1) >> a.qbn_shift) * static_cast<uint32_t>(a.ssb2);
  }
  float* const sa_l = reinterpret_cast<float*>(smem + W * STAGE);  // [W][ROWS]
  float* const sb_l = sa_l + W * ROWS;                             // [W][COLS]

  struct Step {
    typename OA::Regs ra;
    typename OB::Regs rb;
    float sa, sb;
  };
  auto load = [&](Step& s, int ks) {
    oa.load(s.ra, ks * BK);
    ob.load(s.rb, ks * BK);
    if constexpr (MODE == 0) {
      s.sa = (sa_b + int64_t(ks) * a.ssa2)[sao];
      s.sb = (sb_b + int64_t(ks) * a.ssb1)[sbo];
    }
  };
  // Tiles in LDS are row-major, 16-byte chunk c of row r at c ^ (r's low
  // bits). A thread sums and stores 4 consecutive outputs, neighbouring lanes
  // neighbouring outputs of a row: stores and bias loads cover whole row
  // pieces (in the accumulators' own layout 16 neighbouring lanes hold 16
  // rows, and each access touches 16 lines).
  auto part = [&](int w, int r, int c) -> v4f& {
    const int x = NJ == 1 ? (r >> 2) & 3 : r & (CH - 1);
    return reinterpret_cast<v4f*>(smem + w * STAGE)[r * CH + (c ^ x)];
  };
  constexpr int Q = (MI * NJ + W - 1) / W;  // groups of 4 outputs per thread
  v4f sum[Q];
#pragma unroll
  for (int q = 0; q < Q; ++q) sum[q] = v4f{0.f, 0.f, 0.f, 0.f};

  v4f acc[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};

  const int ksteps = (a.k + BK - 1) / BK;
  Step s;
  if (wave < ksteps) load(s, wave);
  for (int k0 = 0; k0 < ksteps; k0 += W) {
    const int ks = k0 + wave;
    if (ks < ksteps) {
      const bool last = (ks + 1) * BK > a.k;
      v8i fa[MI], fb[NJ];
      oa.frags(s.ra, fa, ks * BK, last, lane);
      ob.frags(s.rb, fb, ks * BK, last, lane);
      if constexpr (MODE == 0) {
        if (lane < ROWS) sa_l[wave * ROWS + lane] = s.sa;
        if (lane < COLS) sb_l[wave * COLS + lane] = s.sb;
      }
      // the operands sit in LDS and fragments now: their registers take the next step's
      if (ks + W < ksteps) load(s, ks + W);
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int i = 0; i < MI; ++i) {
          if constexpr (MODE == 0) acc[i][j] = mfma(fb[j], fa[i], v4f{0.f, 0.f, 0.f, 0.f});
          else acc[i][j] = mfma(fb[j], fa[i], acc[i][j]);
        }
      if constexpr (MODE == 0) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NJ; ++j) part(wave, 16 * i + lr, 4 * j + lg) = acc[i][j];
      }
    }
    if constexpr (MODE == 0) {
      lds_barrier();
      const int steps = min(W, ksteps - k0);
#pragma unroll
      for (int q = 0; q < Q; ++q) {
        const int item = threadIdx.x + q * 64 * W;
        if (item >= ROWS * CH) break;
        const int r = item / CH, c = item % CH;
        for (int w = 0; w < steps; ++w) {
          const v4f p = part(w, r, c);
          const float fa = sa_l[w * ROWS + r];
          const v4f fb = *reinterpret_cast<const v4f*>(sb_l + w * COLS + 4 * c);
#pragma unroll
          for (int e = 0; e < 4; ++e) sum[q][e] = fmaf(p[e], fa * fb[e], sum[q][e]);
        }
      }
      lds_barrier();  // the next round overwrites the partials
    }
  }
  if constexpr (MODE != 0) {
    lds_barrier();
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j) part(wave, 16 * i + lr, 4 * j + lg) = acc[i][j];
    lds_barrier();
  }

  float tscale = 1.0f;
  if constexpr (MODE == 2) tscale = a.scales_are_quant ? 1.0f / (a.sa[0] * a.sb[0]) : a.sa[0];
#pragma unroll
  for (int q = 0; q < Q; ++q) {
    const int item = threadIdx.x + q * 64 * W;
    if (item >= ROWS * CH) break;
    const int r = item / CH, c = item % CH;
    const int mm = m0 + r, nn = n0 + 4 * c;
    if constexpr (MODE != 0) {
      sum[q] = part(0, r, c);
#pragma unroll
      for (int w = 1; w < W; ++w) sum[q] += part(w, r, c);
    }
    float v[4] = {sum[q][0], sum[q][1], sum[q][2], sum[q][3]};
    if constexpr (MODE == 1) {
      const float sa = a.sa[bidx * a.ssab + int64_t(min(mm, a.m - 1)) * a.ssa1];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float sc = sa * a.sb[bidx * a.ssbb + int64_t(min(nn + e, a.n - 1)) * a.ssb1];
        if (a.scales_are_quant) sc = 1.0f / sc;
        v[e] *= sc;
      }
    } else if constexpr (MODE == 2) {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] *= tscale;
    }
    store4(a, bidx, mm, nn, v);
  }
}

// the launch of one tile shape: a's tile counts are set here
template <bool A_K, bool B_K, int MODE, int MI, int NJ, int W>
int launch_tile(FastArgs a, int64_t batch, hipStream_t st) {
  a.tiles_m = (a.m + 16 * MI - 1) / (16 * MI);
  a.tiles_n = (a.n + 16 * NJ - 1) / (16 * NJ);
  a.tiles_per_batch = a.tiles_m * a.tiles_n;
  a.total_tiles = static_cast<int>(a.tiles_per_batch * batch);
  bmm_split_kernel<A_K, B_K, MODE, MI, NJ, W><<<a.total_tiles, 64 * W, 0, st>>>(a);
  return check_launch("bmm_split_kernel");
}

}  // namespace bmmp
}  // namespace pcamd
