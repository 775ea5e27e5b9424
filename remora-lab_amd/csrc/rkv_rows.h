// rkv_rows.h -- the byte permutation between one page tile and its reference
// rows, in LDS, for the kernels that export, import, spill and restore pages
// (gfx950).
//
// A page tile (TT = min(32, page_tokens) slots of one page, kv head and kind)
// is two contiguous 16-byte aligned runs: codes (TT*D bytes) and scales
// (TT*D/32 f16).  Its reference rows are one contiguous run: per row D/32
// blocks of an LE f16 scale and 32 codes, 34 bytes each.  So both sides move
// in 16-byte accesses, and the rows are put together (or taken apart) in an
// LDS image of the run, 2 bytes at a time because blocks start on odd
// halfwords.  K codes are rows already; V codes are dim-major, so a lane takes
// 4 dims x 16 slots and transposes them 4x4 in registers (8 byte permutes per
// 16 codes).  One workgroup of 128 threads per tile keeps 8.5 KiB (D = 256) in
// flight, up to 16 of them per CU.  K tiles move at about the rate of a large
// copy, V tiles at half of it (rkv_append.hip has the times), likely because
// the lanes' 16 bytes lie 128 apart and each access touches a line per lane.
#pragma once

#include "rkv_launch.h"

namespace rkv {
namespace {

constexpr int kRowsThreads = 128;

// (Default cache policy on both sides: a wave's 16-byte accesses cover V
// columns half a line at a time, and nontemporal loads or stores lose the
// other half: import 13 -> 49 us with such stores, spill 131 -> 154 with such
// loads.)

template <int D>
struct RowsImage {
  static constexpr int kBytes = 34 * D;           // 32 rows of D/32 blocks
  static constexpr int kRowHalves = D / 32 * 17;  // 2-byte words of a row
};

// 4 dwords of 4 bytes each, transposed: byte i of o[j] is byte j of a[i].
__device__ __forceinline__ void transpose4x4(const uint32_t (&a)[4], uint32_t (&o)[4]) {
  const uint32_t t0 = __builtin_amdgcn_perm(a[1], a[0], 0x05010400u);
  const uint32_t t1 = __builtin_amdgcn_perm(a[3], a[2], 0x05010400u);
  const uint32_t t2 = __builtin_amdgcn_perm(a[1], a[0], 0x07030602u);
  const uint32_t t3 = __builtin_amdgcn_perm(a[3], a[2], 0x07030602u);
  o[0] = __builtin_amdgcn_perm(t1, t0, 0x05040100u);
  o[1] = __builtin_amdgcn_perm(t1, t0, 0x07060302u);
  o[2] = __builtin_amdgcn_perm(t3, t2, 0x05040100u);
  o[3] = __builtin_amdgcn_perm(t3, t2, 0x07060302u);
}

// Slot of position q of a block's scale run (scale_offset's inverse).
__device__ __forceinline__ int32_t scale_slot(int32_t TT, int32_t q) {
  return TT == 32 ? 16 * ((q >> 2) & 1) + 4 * (q >> 3) + (q & 3) : q;
}

// This thread's part of a tile: K, 16-byte chunks (row s, 16 dims); V, 16 slots
// of 4 dims (threads past the tile's D/4 * TT/16 hold none); scales, in page
// order.  Loaded apart from their way into the image, so that a caller can
// have the next tile's loads in flight.
template <int D>
struct TilePart {
  static constexpr int kChunks = 2 * D / kRowsThreads;
  static constexpr int kScales = D / kRowsThreads;
  static_assert(kChunks <= 4, "four 16-byte words per thread");
  uint4 w[4];
  uint16_t sc[kScales];
};

template <int D>
__device__ __forceinline__ TilePart<D> load_tile(const Geo &g, const uint8_t *region, int32_t kind, int32_t slot0,
                                                 int32_t TT) {
  using P = TilePart<D>;
  const int tid = threadIdx.x;
  const uint8_t *codes = region + code_offset(g, kind, slot0, 0);
  const uint16_t *scales = reinterpret_cast<const uint16_t *>(region + scale_offset(g, slot0, 0));
  P p;
  // branch-free (a thread without a part reads the tile's first bytes), so
  // that no load waits for one before it
  const int k = tid % (D / 4), h = tid / (D / 4);
  const int32_t n = TT * (D / 16);  // K chunks
  const int32_t off = kind == 0 ? 16 * tid : (h < TT / 16 ? 4 * k * TT + 16 * h : 0);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int32_t at = kind == 0 ? (i < P::kChunks && i * kRowsThreads + tid < n ? off + 16 * i * kRowsThreads : 0)
                                 : off + i * TT;
    p.w[i] = *reinterpret_cast<const uint4 *>(codes + at);
  }
#pragma unroll
  for (int i = 0; i < P::kScales; ++i) p.sc[i] = scales[min(i * kRowsThreads + tid, TT * (D / 32) - 1)];
  return p;
}

// The tile into the LDS image (halfword h of row s at s * kRowHalves + h);
// rows of slots that hold no token are whatever the page holds.  The caller's
// barrier follows.
template <int D>
__device__ __forceinline__ void tile_to_image(const TilePart<D> &p, int32_t kind, int32_t TT, uint16_t *img) {
  using P = TilePart<D>;
  constexpr int RH = RowsImage<D>::kRowHalves;
  const int tid = threadIdx.x;
  if (kind == 0) {
#pragma unroll
    for (int i = 0; i < P::kChunks; ++i) {
      const int t = i * kRowsThreads + tid;
      if (t >= TT * (D / 16)) continue;
      const int s = t / (D / 16), c = t % (D / 16);
      uint16_t *o = img + s * RH + (c >> 1) * 17 + 1 + 8 * (c & 1);
      const uint32_t ws[4] = {p.w[i].x, p.w[i].y, p.w[i].z, p.w[i].w};
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        o[2 * k] = (uint16_t)ws[k];
        o[2 * k + 1] = (uint16_t)(ws[k] >> 16);
      }
    }
  } else if (tid < (D / 4) * (TT / 16)) {
    const int k = tid % (D / 4), h = tid / (D / 4);
    uint16_t *o = img + 16 * h * RH + (k >> 3) * 17 + 1 + 2 * (k & 7);
    uint32_t w[4][4];  // [dim][slot quad]
#pragma unroll
    for (int i = 0; i < 4; ++i) w[i][0] = p.w[i].x, w[i][1] = p.w[i].y, w[i][2] = p.w[i].z, w[i][3] = p.w[i].w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t a[4] = {w[0][j], w[1][j], w[2][j], w[3][j]};
      uint32_t r[4];
      transpose4x4(a, r);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t x = r[i] ^ 0x80808080u;  // code_bias
        o[(4 * j + i) * RH] = (uint16_t)x;
        o[(4 * j + i) * RH + 1] = (uint16_t)(x >> 16);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < P::kScales; ++i) {
    const int t = i * kRowsThreads + tid;
    if (t < TT * (D / 32)) img[scale_slot(TT, t % TT) * RH + t / TT * 17] = p.sc[i];
  }
}

// The inverse, after a barrier: slots [s_lo, s_hi) of the tile from the
// image.  Slots outside the range keep their bytes.
template <int D>
__device__ __forceinline__ void image_to_tile(const Geo &g, uint8_t *region, int32_t kind, int32_t slot0, int32_t TT,
                                              int32_t s_lo, int32_t s_hi, const uint16_t *img) {
  constexpr int RH = RowsImage<D>::kRowHalves;
  const int tid = threadIdx.x;
  uint8_t *codes = region + code_offset(g, kind, slot0, 0);
  uint16_t *scales = reinterpret_cast<uint16_t *>(region + scale_offset(g, slot0, 0));
  if (kind == 0) {
    for (int t = tid; t < TT * (D / 16); t += kRowsThreads) {
      const int s = t / (D / 16), c = t % (D / 16);
      if (s < s_lo || s >= s_hi) continue;
      const uint16_t *o = img + s * RH + (c >> 1) * 17 + 1 + 8 * (c & 1);
      uint32_t w[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) w[k] = (uint32_t)o[2 * k] | ((uint32_t)o[2 * k + 1] << 16);
      reinterpret_cast<uint4 *>(codes)[t] = uint4{w[0], w[1], w[2], w[3]};
    }
  } else if (s_lo == 0 && s_hi == TT) {
    for (int t = tid; t < (D / 4) * (TT / 16); t += kRowsThreads) {
      const int k = t % (D / 4), h = t / (D / 4);
      const uint16_t *o = img + 16 * h * RH + (k >> 3) * 17 + 1 + 2 * (k & 7);
      uint32_t w[4][4];  // [dim][slot quad]
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        uint32_t a[4], r[4];
#pragma unroll
        for (int i = 0; i < 4; ++i)
          a[i] = ((uint32_t)o[(4 * j + i) * RH] | ((uint32_t)o[(4 * j + i) * RH + 1] << 16)) ^ 0x80808080u;
        transpose4x4(a, r);
#pragma unroll
        for (int i = 0; i < 4; ++i) w[i][j] = r[i];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<uint4 *>(codes + (4 * k + i) * TT + 16 * h) = uint4{w[i][0], w[i][1], w[i][2], w[i][3]};
    }
  } else {  // an edge of the range: only its slots' bytes
    const int32_t n = s_hi - s_lo;
    for (int t = tid; t < n * D; t += kRowsThreads) {
      const int s = s_lo + t % n, d = t / n;
      const uint16_t x = img[s * RH + (d >> 5) * 17 + 1 + ((d & 31) >> 1)];
      codes[d * TT + s] = (uint8_t)(x >> (8 * (d & 1))) ^ code_bias(1);
    }
  }
  for (int t = tid; t < TT * (D / 32); t += kRowsThreads) {
    const int s = scale_slot(TT, t % TT);
    if (s >= s_lo && s < s_hi) scales[t] = img[s * RH + t / TT * 17];
  }
}

// n bytes (a multiple of 8) between global memory at `p` and the 8-byte
// aligned LDS image at `lds`, 16 bytes per lane where both allow it; any
// alignment of p.
__device__ __forceinline__ void store_run(uint8_t *p, const uint8_t *lds, int32_t n) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  if (((a | (uintptr_t)n) & 15) == 0) {
    // (the image's rows start 8 bytes off a 16-byte boundary when odd rows
    // of D = 128 come first: two 8-byte LDS reads then)
    for (int32_t i = threadIdx.x; i < n / 16; i += kRowsThreads) {
      const uint2 lo = reinterpret_cast<const uint2 *>(lds)[2 * i], hi = reinterpret_cast<const uint2 *>(lds)[2 * i + 1];
      reinterpret_cast<uint4 *>(p)[i] = uint4{lo.x, lo.y, hi.x, hi.y};
    }
  } else if ((a & 7) == 0) {
    for (int32_t i = threadIdx.x; i < n / 8; i += kRowsThreads)
      reinterpret_cast<uint2 *>(p)[i] = reinterpret_cast<const uint2 *>(lds)[i];
  } else {
    for (int32_t i = threadIdx.x; i < n; i += kRowsThreads) p[i] = lds[i];
  }
}
__device__ __forceinline__ void load_run(uint8_t *lds, const uint8_t *p, int32_t n) {
  const uintptr_t a = reinterpret_cast<uintptr_t>(p);
  if (((a | (uintptr_t)n) & 15) == 0) {
    for (int32_t i = threadIdx.x; i < n / 16; i += kRowsThreads) {
      const uint4 v = reinterpret_cast<const uint4 *>(p)[i];
      reinterpret_cast<uint2 *>(lds)[2 * i] = uint2{v.x, v.y};
      reinterpret_cast<uint2 *>(lds)[2 * i + 1] = uint2{v.z, v.w};
    }
  } else if ((a & 7) == 0) {
    for (int32_t i = threadIdx.x; i < n / 8; i += kRowsThreads)
      reinterpret_cast<uint2 *>(lds)[i] = reinterpret_cast<const uint2 *>(p)[i];
  } else {
    for (int32_t i = threadIdx.x; i < n; i += kRowsThreads) lds[i] = p[i];
  }
}

}  // namespace
}  // namespace rkv
