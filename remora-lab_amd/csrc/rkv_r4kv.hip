// rkv_r4kv.hip -- R4KV page spill/restore kernels for gfx950: a device
// CRC32C (har/crates/r4kv/src/crc32c.rs) and the pack/unpack of a token
// range of Q8_0 rows between the page pool and a page payload.
//
// CRC32C.  Each wave covers a 128 KiB segment; the segments are laid out
// back from the end of the 16-byte-aligned prefix, so the first may start
// before byte 0 (those leading bytes read as zero, which leaves the raw CRC
// unchanged) and every 16-byte piece is aligned.  Lane l folds the pieces
// l, l+64, ... of its segment (Horner: shift the running value 1024 bytes,
// xor the piece's raw CRC from the slicing tables), and the lanes combine
// in a 6-level tree of shifts by 16*2^j bytes.  The four waves of a block
// hold consecutive segments: each is shifted to the block's end and xor-ed
// in LDS, and the block's value is shifted once to the end of the message
// and xor-ed into the output word.  Block 0 also adds the raw CRC of the
// unaligned tail and the init/final-xor term.  Reads stay inside [0, n).
#include <algorithm>
#include <type_traits>

#include "rkv_crc32c.h"
#include "rkv_launch.h"
#include "rkv_rows.h"

namespace rkv {
namespace {

constexpr int kCrcIter = 128;                      // pieces per lane
constexpr int64_t kCrcSeg = 16LL * 64 * kCrcIter;  // bytes per wave (128 KiB = 2^17)
constexpr int kCrcSegLog2 = 17;

__constant__ crc::Slice16 c_slice16 = crc::kSlice16;
__constant__ crc::Shift1024 c_shift1024 = crc::kShift1024;
__constant__ crc::Shifts c_shifts = crc::kShift;
__constant__ crc::ByteTable c_byte = crc::kByte;

__device__ __forceinline__ uint32_t mat_apply_dev(const crc::Mat &m, uint32_t c) {
  uint32_t r = 0;
#pragma unroll
  for (int i = 0; i < 32; ++i) r ^= m.col[i] & (0u - ((c >> i) & 1u));
  return r;
}

__global__ void zero_word_kernel(uint32_t *w) { *w = 0; }

__global__ __launch_bounds__(256) void crc32c_kernel(const uint8_t *data, int64_t n,
                                                     int64_t n_waves, uint32_t finish,
                                                     uint32_t *out) {
  __shared__ uint32_t ts[16][256];
  __shared__ uint32_t tm[4][256];
  for (int i = threadIdx.x; i < 16 * 256; i += 256) ts[i >> 8][i & 255] = c_slice16.t[i >> 8][i & 255];
  for (int i = threadIdx.x; i < 4 * 256; i += 256) tm[i >> 8][i & 255] = c_shift1024.t[i >> 8][i & 255];
  __syncthreads();
  __shared__ uint32_t wave_acc[4];
  const int wib = threadIdx.x >> 6;
  const int64_t wave = (int64_t)blockIdx.x * 4 + wib;
  const int lane = threadIdx.x & 63;
  // blocks are laid out back from the end like the waves: the last block is
  // full, the first may hold waves before the first segment (all zero)
  const int64_t n_blocks = (n_waves + 3) / 4;
  const int64_t vwave = wave - (n_blocks * 4 - n_waves);  // < 0: before byte 0
  const int64_t n16 = n & ~(int64_t)15;
  const int64_t seg = n16 - (n_waves - vwave) * kCrcSeg;
  uint32_t acc = 0;
  for (int k = 0; k < kCrcIter; ++k) {
    const int64_t p = seg + 1024 * k + 16 * lane;
    uint4 w = {0u, 0u, 0u, 0u};
    if (p >= 0) w = *reinterpret_cast<const uint4 *>(data + p);
    acc = tm[0][acc & 0xffu] ^ tm[1][(acc >> 8) & 0xffu] ^ tm[2][(acc >> 16) & 0xffu] ^ tm[3][acc >> 24];
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int q = 0; q < 16; ++q) acc ^= ts[15 - q][(ws[q >> 2] >> (8 * (q & 3))) & 0xffu];
  }
#pragma unroll
  for (int j = 0; j < 6; ++j) {
    const uint32_t other = __shfl_xor(acc, 1 << j);
    const uint32_t sh = mat_apply_dev(c_shifts.m[4 + j], acc) ^ other;
    if ((lane & (1 << j)) == 0) acc = sh;
  }
  // lane 0 holds the wave's raw CRC aligned at its segment end; the block's
  // four segments are consecutive, so wave w's value moves (3-w) segments
  if (lane == 0) {
    const int k = 3 - wib;
    if (k & 1) acc = mat_apply_dev(c_shifts.m[kCrcSegLog2], acc);
    if (k & 2) acc = mat_apply_dev(c_shifts.m[kCrcSegLog2 + 1], acc);
    wave_acc[wib] = acc;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  acc = wave_acc[0] ^ wave_acc[1] ^ wave_acc[2] ^ wave_acc[3];
  const int64_t block_end = seg + (int64_t)(4 - wib) * kCrcSeg;  // wib == 0 here
  uint64_t d = (uint64_t)(n - block_end);
  for (int j = 0; j < crc::kShiftBits && d; ++j, d >>= 1)
    if (d & 1u) acc = mat_apply_dev(c_shifts.m[j], acc);
  if (blockIdx.x == 0) {
    uint32_t t = 0;
    for (int64_t i = n16; i < n; ++i) t = c_byte.t[(t ^ data[i]) & 0xffu] ^ (t >> 8);
    acc ^= t ^ finish;
  }
  atomicXor(out, acc);
}

// Payload body of a page: for each layer of [layer_lo, layer_lo+n_layers),
// kind (K, V) and kv head, the rows of tokens [t0, t0+count) in the
// reference layout ((D/32) blocks of LE f16 scale + 32 int8).
//
// A unit is one page tile (TT = min(32, page_tokens) slots) of one stream
// (layer, kind, kv head) that the range touches; its rows are one contiguous,
// 8-byte aligned run of the body, and the byte permutation between the two
// goes through an LDS image of the run (rkv_rows.h).  A workgroup (x, kind * H
// + kv head, layer) takes tiles of its stream: pack_kernel [x*per, x*per +
// per), unpack_kernel tile x.
struct BodyMap {
  Geo g;
  int64_t layer_stride;
  int32_t layer_lo, n_layers;
  int32_t t0, count;
  int32_t tile0, n_tiles;  // page tiles touched: [tile0, tile0 + n_tiles) in units of TT
  int32_t per;             // tiles of a workgroup
  int32_t n_main;          // tiles of the workgroups before the last (see pack_kernel)
};

struct Unit {
  int32_t layer, kind, kvh;
  int32_t p0, s_lo, s_hi;  // tile start position, slots [s_lo, s_hi) in range
  int64_t body_off;        // body byte offset of the unit's first row
};

template <int D>
__device__ __forceinline__ Unit unit_of(const BodyMap &m, int32_t tile) {
  Unit r;
  const int32_t TT = tile_tokens(m.g.page_tokens);
  r.kvh = (int32_t)blockIdx.y % m.g.kv_heads;
  r.kind = (int32_t)blockIdx.y / m.g.kv_heads;
  r.layer = m.layer_lo + (int32_t)blockIdx.z;
  r.p0 = (m.tile0 + tile) * TT;
  const int32_t a = max(m.t0, r.p0), b = min(m.t0 + m.count, r.p0 + TT);
  r.s_lo = a - r.p0;
  r.s_hi = b - r.p0;
  r.body_off = ((((int64_t)blockIdx.z * 2 + r.kind) * m.g.kv_heads + r.kvh) * m.count + (a - m.t0)) *
               (2 * RowsImage<D>::kRowHalves);
  return r;
}

// The 96 header bytes, already serialized on the host.
struct Header96 {
  uint32_t w[24];
};

// The CRC polynomial with x^m for x, P(x^m) with m a power of two, is P(x)^m:
// a multiple of P with the same terms, m apart.  So the words L apart that a
// lane holds of a message (m = 32*L) can be divided by it with whole-word
// xors and no table: q_i = w_i ^ (xor of q_{i-j} over the taps j), 17 terms
// per word against 4 random LDS lookups a word and a serial chain of them.
// kTaps: 32 minus the exponents below 32.
constexpr int kTaps[17] = {4, 5, 6, 7, 9, 10, 12, 13, 14, 18, 19, 21, 22, 23, 24, 26, 32};
constexpr int kTileWords = 17;  // words of a whole tile's run per lane

// One tile: the lane's words w(i), i < 17, behind the quotient words h
// (h[31] the newest).
template <typename W>
__device__ __forceinline__ void crc_divide(uint32_t (&h)[32], W w) {
  uint32_t e[32 + kTileWords];
#pragma unroll
  for (int i = 0; i < 32; ++i) e[i] = h[i];
#pragma unroll
  for (int i = 0; i < kTileWords; ++i) {
    uint32_t q = w(i) ^ e[32 + i - kTaps[16]];
#pragma unroll
    for (int k = 15; k > 0; k -= 2)  // oldest first: the newest is just ready; 0x96: a ^ b ^ c
      q = __builtin_amdgcn_bitop3_b32(q, e[32 + i - kTaps[k]], e[32 + i - kTaps[k - 1]], 0x96);
    e[32 + i] = q;
  }
#pragma unroll
  for (int i = 0; i < 32; ++i) h[i] = e[kTileWords + i];
}

// c moved through d zero bytes, c uniform over the wave: lane l < 32 holds
// column l of every power's matrix and a row of lanes sums its 16 columns
// over DPP rotations (a serial matrix product per bit took most of a
// workgroup's tail).
__device__ __forceinline__ uint32_t wave_shift(uint32_t c, uint64_t d, int lane) {
  uint32_t col[crc::kShiftBits];
#pragma unroll
  for (int j = 0; j < crc::kShiftBits; ++j) col[j] = c_shifts.m[j].col[lane & 31];
#pragma unroll
  for (int j = 0; j < crc::kShiftBits; ++j) {
    if (!((d >> j) & 1u)) continue;
    uint32_t v = (c >> (lane & 31)) & 1u ? col[j] : 0u;
    v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xf, 0xf, false);  // row_ror:8
    v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x124, 0xf, 0xf, false);
    v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x122, 0xf, 0xf, false);
    v ^= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x121, 0xf, 0xf, false);
    c = (uint32_t)__builtin_amdgcn_readlane((int)v, 0) ^ (uint32_t)__builtin_amdgcn_readlane((int)v, 16);
  }
  return c;
}

// The launches before and behind pack_kernel: the header and a cleared CRC
// word, so that no spill relies on what another left there (captured spills
// that are replayed on two streams at once spoil each other's CRC; later ones
// must not inherit it), then the page's trailing word.  The stream orders the
// three, so that pack_kernel's xors need no order among themselves.  214 MB:
// 125.6 us with the header and the trailing word in pack_kernel (its last
// workgroup by a count), 127.3 with the first launch, 128.2 with both; a count
// with acquire-release order, which writes an XCD's L2 back once per
// workgroup, 197.6.
__global__ void spill_begin_kernel(Header96 h96, uint8_t *page_out, uint32_t *crc_word) {
  if (threadIdx.x < 24) reinterpret_cast<uint32_t *>(page_out)[threadIdx.x] = h96.w[threadIdx.x];
  if (threadIdx.x == 0) *crc_word = 0u;
}
__global__ void spill_end_kernel(const uint32_t *crc_word, uint32_t finish, uint8_t *to) {
  *reinterpret_cast<uint32_t *>(to) = *crc_word ^ finish;
}

// Spill: the body and its CRC32C in one launch.  Each tile's rows leave for
// the body from the LDS image, and the CRC is taken from the same image, so
// the body is not read back (the CRC as a second pass over a 214 MB page took
// 115 us after a 128 us pack; this launch takes 129, 3.3 TB/s of its 428 MB
// of traffic).  HBM does not bound it: unpack_kernel moves the same bytes in 89.
// The CRC is 10 us of the difference (118 against 128 us a spill without it);
// the rest is the way these workgroups move tiles, of which two tiles ahead
// (135 us), more workgroups (344 at a tile each) and fewer were slower.
// Lane t holds words t, t + L, ... of the workgroup's part of the body
// (L = TT*D/64, so a whole tile is 17 of them) and divides
// them by P(x^(32 L)) as they come (crc_divide); a partly covered first tile
// starts with zero words (which change nothing), and a partly covered last
// one gets a workgroup of its own.  At the end the lanes' remainders are a
// message of 32*L words, congruent to the part followed by as many zero
// words: it is checksummed with slicing tables, moved to the body's end
// (128*L bytes less than the part's distance from it; x has order 2^31 - 1,
// which makes a negative shift a positive one) and xor-ed into the CRC word.
template <int D, int TT>
__global__ __launch_bounds__(kRowsThreads) void pack_kernel(BodyMap m, const uint8_t *pages,
                                                            const int32_t *bt, uint8_t *page_out, int64_t body_len,
                                                            uint32_t *crc_word, int32_t *fault) {
  constexpr int kLanes = TT * D / 64;
  constexpr int RB = 2 * RowsImage<D>::kRowHalves;
  static_assert(kLanes * kTileWords * 4 == TT * RB && kLanes <= kRowsThreads, "17 words a lane");
  __shared__ __attribute__((aligned(16))) uint16_t img[2][RowsImage<D>::kBytes / 2];
  static_assert(sizeof(img) >= 33 * 4 * kLanes, "the remainders reuse the images");
  __shared__ uint32_t ts[4][256];
  __shared__ uint32_t wave_acc[kRowsThreads / 64];
  const int tid = threadIdx.x;
  for (int i = tid; i < 4 * 256; i += kRowsThreads) ts[i >> 8][i & 255] = c_slice16.t[i >> 8][i & 255];
  uint8_t *body = page_out + 96;
  int32_t j0 = (int32_t)blockIdx.x * m.per, j1 = min(j0 + m.per, m.n_main);
  if (j0 >= m.n_main) {  // the last workgroup of a stream: its partly covered last tile
    j0 = m.n_main;
    j1 = m.n_tiles;
  }
  uint32_t h[32] = {};
  int64_t end = 0;  // body offset behind the workgroup's last run
  // the pages of the workgroup's tiles, one per lane (-1: none, reported)
  const int lane = tid & 63;
  int32_t pidv = j0 + lane < j1 ? bt[(m.tile0 + j0 + lane) * TT / m.g.page_tokens] : 0;
  if (pidv < 0 || pidv >= m.g.num_pages) {
    atomicOr(fault, FAULT_BAD_PAGE);
    pidv = -1;
  }
  auto page_of = [&](int32_t j) { return __builtin_amdgcn_readlane(pidv, j - j0); };
  auto load = [&](const Unit &u, int32_t page) {
    return load_tile<D>(m.g, pages + u.layer * m.layer_stride + region_base(m.g, max(page, 0), u.kvh, u.kind), u.kind,
                        u.p0 % m.g.page_tokens, TT);
  };
  TilePart<D> part;
  if (j0 < j1) part = load(unit_of<D>(m, j0), page_of(j0));
  // (waited for here, so that inside the loop only loads with stores behind
  // them are pending)
  __builtin_amdgcn_s_waitcnt(0x0f70);
  for (int32_t j = j0; j < j1; ++j) {
    const Unit u = unit_of<D>(m, j);
    const bool ok = page_of(j) >= 0;
    uint16_t *im = img[(j - j0) & 1];
    tile_to_image<D>(part, u.kind, TT, im);
    // the next tile's loads land during this one's stores and checksums (two
    // tiles ahead measured no faster: 135 us against 130)
    if (j + 1 < j1) part = load(unit_of<D>(m, j + 1), page_of(j + 1));
    // one barrier per tile: the image of two tiles ago was read before the
    // barrier of the last
    __syncthreads();
    const int32_t nrows = u.s_hi - u.s_lo;
    uint8_t *to = body + u.body_off;
    if (ok && nrows == TT && (D == 256 || (u.body_off & 15) == 0)) {
      // straight-line, so that the wait for the next tile's loads, which are
      // older, leaves these stores in flight (a loop's count is not known: the
      // wait would take every store's round trip, 188 us)
      constexpr int kWide = TT * RB / (16 * kRowsThreads), kRest = TT * RB % (16 * kRowsThreads) / kRowsThreads;
      using Rest = typename std::conditional<kRest == 4, uint32_t,
                                             typename std::conditional<kRest == 2, uint16_t, uint8_t>::type>::type;
      static_assert(kRest == sizeof(Rest), "16-byte words and one shorter one per thread");
#pragma unroll
      for (int i = 0; i < kWide; ++i)
        reinterpret_cast<uint4 *>(to)[i * kRowsThreads + tid] = reinterpret_cast<const uint4 *>(im)[i * kRowsThreads + tid];
      constexpr int kAt = 16 * kWide * kRowsThreads / kRest;
      reinterpret_cast<Rest *>(to)[kAt + tid] = reinterpret_cast<const Rest *>(im)[kAt + tid];
    } else {
      if (ok) store_run(to, reinterpret_cast<const uint8_t *>(im) + u.s_lo * RB, nrows * RB);
      __builtin_amdgcn_s_waitcnt(0x0f70);  // vmcnt(0), which the compiler counts
    }
    if (tid < kLanes) {
      // the run's words, right-aligned in a whole tile's
      const uint32_t *w = reinterpret_cast<const uint32_t *>(im) + u.s_hi * (RB / 4) - kTileWords * kLanes + tid;
      const int32_t none = ok ? kTileWords * kLanes - nrows * (RB / 4) - tid : INT32_MAX;
      if (ok && nrows == TT)
        crc_divide(h, [&](int i) { return w[i * kLanes]; });
      else
        crc_divide(h, [&](int i) { return i * kLanes < none ? 0u : w[i * kLanes]; });
    }
    end = u.body_off + (int64_t)nrows * RB;
  }
  // remainder word i (of 32) of lane t is word i*L + t of a message that lane
  // t then checksums words 32t.. of, one pad word per 32 against bank conflicts
  __syncthreads();
  uint32_t *rem = reinterpret_cast<uint32_t *>(img);
  if (tid < kLanes) {
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      uint32_t r = 0;
#pragma unroll
      for (int k = 0; k < 17; ++k)
        if (kTaps[k] > i) r ^= h[32 + i - kTaps[k]];
      rem[i * kLanes + tid + (i * kLanes + tid) / 32] = r;
    }
  }
  __syncthreads();
  uint32_t acc = 0;
  if (tid < kLanes) {
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      acc ^= rem[33 * tid + i];
      acc = ts[3][acc & 0xffu] ^ ts[2][(acc >> 8) & 0xffu] ^ ts[1][(acc >> 16) & 0xffu] ^ ts[0][acc >> 24];
    }
  }
  // lanes: neighbours 128 * 2^k bytes apart
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    if ((1 << k) >= kLanes) continue;
    const uint32_t other = __shfl_xor(acc, 1 << k);
    const uint32_t sh = mat_apply_dev(c_shifts.m[7 + k], acc) ^ other;
    if ((lane & (1 << k)) == 0) acc = sh;
  }
  if (lane == 0) wave_acc[tid >> 6] = acc;
  __syncthreads();
  if (tid >= 64) return;
  acc = wave_acc[0];
  if (kLanes > 64) acc = mat_apply_dev(c_shifts.m[13], acc) ^ wave_acc[1];
  int64_t d = body_len - end - 128 * kLanes;
  if (d < 0) d += 0x7fffffff;
  acc = wave_shift((uint32_t)__builtin_amdgcn_readfirstlane((int)acc), j1 > j0 ? (uint64_t)d : 0, lane);
  if (tid == 0) atomicXor(crc_word, acc);
}

template <int D>
__global__ __launch_bounds__(kRowsThreads) void unpack_kernel(BodyMap m, uint8_t *pages, const int32_t *bt,
                                                              const uint8_t *body, int32_t *fault) {
  __shared__ __attribute__((aligned(16))) uint16_t img[RowsImage<D>::kBytes / 2];
  constexpr int RB = 2 * RowsImage<D>::kRowHalves;
  const int32_t TT = tile_tokens(m.g.page_tokens);
  const Unit u = unit_of<D>(m, (int32_t)blockIdx.x);
  const int32_t page = bt[u.p0 / m.g.page_tokens];
  if (page < 0 || page >= m.g.num_pages) {
    if (threadIdx.x == 0) atomicOr(fault, FAULT_BAD_PAGE);
    return;
  }
  load_run(reinterpret_cast<uint8_t *>(img) + u.s_lo * RB, body + u.body_off, (u.s_hi - u.s_lo) * RB);
  __syncthreads();
  image_to_tile<D>(m.g, pages + u.layer * m.layer_stride + region_base(m.g, page, u.kvh, u.kind), u.kind,
                   u.p0 % m.g.page_tokens, TT, u.s_lo, u.s_hi, img);
}

BodyMap body_map(const R4kvLaunch &r) {
  BodyMap m{r.g, r.layer_stride, r.layer_lo, r.n_layers, r.t0, r.count, 0, 0, 1, 0};
  const int32_t TT = tile_tokens(r.g.page_tokens);
  if (r.count > 0) {
    m.tile0 = r.t0 / TT;
    m.n_tiles = (r.t0 + r.count - 1) / TT - m.tile0 + 1;
  }
  return m;
}

}  // namespace

hipError_t launch_crc32c(const uint8_t *data, int64_t n, uint32_t *out, hipStream_t s) {
  hipLaunchKernelGGL(zero_word_kernel, dim3(1), dim3(1), 0, s, out);
  if (n <= 0) return hipGetLastError();
  const int64_t n16 = n & ~(int64_t)15;
  int64_t waves = (n16 + kCrcSeg - 1) / kCrcSeg;
  if (waves == 0) waves = 1;
  const int64_t blocks = (waves + 3) / 4;  // the kernel derives the same count
  hipLaunchKernelGGL(crc32c_kernel, dim3((unsigned)blocks), dim3(256), 0, s, data, n, waves,
                     crc::finish_term((uint64_t)n), out);
  return hipGetLastError();
}

hipError_t launch_r4kv_pack(const R4kvLaunch &r, const uint8_t *pages, const int32_t *bt,
                            uint8_t *page_out, uint32_t *crc_word, int32_t *fault, hipStream_t s) {
  BodyMap m = body_map(r);
  Header96 h;
  for (int i = 0; i < 24; ++i)
    h.w[i] = (uint32_t)r.header[4 * i] | ((uint32_t)r.header[4 * i + 1] << 8) |
             ((uint32_t)r.header[4 * i + 2] << 16) | ((uint32_t)r.header[4 * i + 3] << 24);
  const int32_t TT = tile_tokens(r.g.page_tokens);
  const int64_t streams = (int64_t)m.n_layers * 2 * r.g.kv_heads;
  const int64_t body_len = streams * m.count * (r.g.head_dim / 32 * 34);
  // a partly covered last tile behind others has a workgroup of its own
  const bool lone = m.n_tiles > 1 && (r.t0 + r.count) % TT != 0;
  m.n_main = m.n_tiles - (lone ? 1 : 0);
  // one round of seven workgroups per CU, in even shares: each reduces its
  // lanes' remainders and moves them to the body's end once.  Seven is what a
  // CU's LDS holds at D = 256, where it was measured; at D = 128 12 would fit.
  const int64_t shares = std::clamp<int64_t>(7 * kComputeUnits / streams, 1, std::max(m.n_main, 1));
  m.per = (int32_t)std::clamp<int64_t>((m.n_main + shares - 1) / shares, 1, 64);  // a lane per tile's page
  const int32_t chunks = std::max<int32_t>(1, (m.n_main + m.per - 1) / m.per) + (lone ? 1 : 0);
  const dim3 grid((unsigned)chunks, (unsigned)(2 * r.g.kv_heads), (unsigned)m.n_layers);
  const uint32_t finish = crc::finish_term((uint64_t)body_len);
  hipLaunchKernelGGL(spill_begin_kernel, dim3(1), dim3(64), 0, s, h, page_out, crc_word);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(kRowsThreads), 0, s, m, pages, bt, page_out, body_len, crc_word, fault);
  };
  if (r.g.head_dim == 256) {
    if (TT == 32) go(pack_kernel<256, 32>);
    else go(pack_kernel<256, 16>);
  } else {
    if (TT == 32) go(pack_kernel<128, 32>);
    else go(pack_kernel<128, 16>);
  }
  hipLaunchKernelGGL(spill_end_kernel, dim3(1), dim3(1), 0, s, crc_word, finish, page_out + 96 + body_len);
  return hipGetLastError();
}

hipError_t launch_r4kv_unpack(const R4kvLaunch &r, uint8_t *pages, const int32_t *bt,
                              const uint8_t *body, int32_t *fault, hipStream_t s) {
  const BodyMap m = body_map(r);
  if (m.n_tiles == 0 || m.n_layers == 0) return hipSuccess;
  const dim3 grid((unsigned)m.n_tiles, (unsigned)(2 * r.g.kv_heads), (unsigned)m.n_layers);
  if (r.g.head_dim == 256)
    hipLaunchKernelGGL(unpack_kernel<256>, grid, dim3(kRowsThreads), 0, s, m, pages, bt, body, fault);
  else
    hipLaunchKernelGGL(unpack_kernel<128>, grid, dim3(kRowsThreads), 0, s, m, pages, bt, body, fault);
  return hipGetLastError();
}

}  // namespace rkv
