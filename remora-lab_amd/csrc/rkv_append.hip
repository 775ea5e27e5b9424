// rkv_append.hip -- quantize-and-append of K/V rows into Q8_0 pages, the
// bit-exact gather/import between pages and reference rows, and a batch
// f16 encoder (gfx950).
//
// Quantization rules (bit-exact with the CPU reference): q8_quantize_values
// in rkv_device.h -- canonical (har/crates/r4kv/src/quant.rs:45-90) or
// har-serve (har/crates/har-serve/src/attention.rs:25-42).
#include <algorithm>

#include "rkv_launch.h"
#include "rkv_rows.h"

namespace rkv {

namespace {

// Eight consecutive source values (f32 or bf16) starting at element `off`.
template <bool kBf16>
__device__ inline void load_src8(const void *src, uint64_t off, float v[8]) {
  if constexpr (kBf16) {
    const uint4 w = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(src) + off);
    const uint32_t ws[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = bf16_bits_to_f32((uint16_t)(ws[i] & 0xffffu));
      v[2 * i + 1] = bf16_bits_to_f32((uint16_t)(ws[i] >> 16));
    }
  } else {
    const float4 a = *reinterpret_cast<const float4 *>(static_cast<const float *>(src) + off);
    const float4 b = *reinterpret_cast<const float4 *>(static_cast<const float *>(src) + off + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
}

// One workgroup of 256 threads appends input rows [ROWS*blockIdx.x, +ROWS)
// of kv head blockIdx.y, K and V (ROWS = 32 for large launches, 8 for small
// ones, so that a few thousand rows still spread over several workgroups per
// CU: the quantizer's VALU work, not HBM, bounds a workgroup):
//  1. each row's destination (region offset and slot; invalid rows are
//     reported and skipped, nothing is written for them);
//  2. quantize, 4 lanes per 32-value block with 8 values each (lanes of a
//     row read its values in contiguous 16-byte loads), into LDS: K and V
//     codes row-major (row stride D + 8 bytes: conflict-free for both the
//     8-byte writes here and the transposing byte reads below) and scales;
//  3. write the page bytes so that a wave's stores are contiguous whenever
//     the rows are consecutive tokens: K rows as 16-byte stores; V codes
//     (page layout [slot/TT][dim][slot%TT]) as one 4-byte store per 4 rows
//     that are 4 aligned consecutive slots of one page, lanes ordered by
//     slot group then dim (256 contiguous bytes per wave for a whole tile),
//     else byte stores; scales with lanes ordered by slot.
// Rows of a sequence whose length before them is not a multiple of 4 make
// quads that start 1..3 rows into the workgroup's: where all of them do, they
// are stored as such and only the four rows around them byte by byte.
// Row blocks go to the XCDs in chunks of kAppChunk consecutive ones, because
// a tile's 128-byte lines of V codes are then mostly put together in one L2
// (32 rows that start inside a tile share its lines with the next block, four
// 8-row blocks share a tile).  65,619 rows of 16 sequences of odd lengths
// (D 256, 2 kv heads, bf16): 59.5 us with neither, 54.8 with the chunks, 50.4
// with both; 4101 rows of 8 sequences 9.65, 8.6, 8.3; 65,536 rows that start at
// tiles 46.3 to 46.5 either way.
template <int kAppRows>
constexpr uint32_t kAppChunk = kAppRows == 32 ? 8 : 4;

template <int D, int kAppRows, bool kBf16, int kRule>
__global__ __launch_bounds__(256) void append_kernel(AppendLaunch a) {
  static_assert(kAppRows % 4 == 0 && kAppRows <= 64, "rows come in quads, resolved by wave 0");
  constexpr int NB = D / 32;
  constexpr int RS = D + 8;  // LDS row stride
  __shared__ __attribute__((aligned(16))) uint8_t codes[2][kAppRows][RS];
  __shared__ uint16_t scl[2][kAppRows][NB];
  __shared__ int64_t rbase[kAppRows];  // region offset of (page, kv head, K); -1: skip the row
  __shared__ int32_t rslot[kAppRows];
  __shared__ int32_t quad[kAppRows / 4];  // rows 4i..4i+3 are slots s..s+3 (s % 4 == 0) of one page
  __shared__ int32_t shifted;             // > 0: rows shifted..shifted+kAppRows-5 are whole such quads
  const Geo g = a.g;
  const int tid = (int)threadIdx.x;
  const int kvh = (int)blockIdx.y;
  const uint32_t x = blockIdx.x, C = kAppChunk<kAppRows>;
  const int64_t row0 = (int64_t)(x / (8 * C) * (8 * C) + x % 8 * C + x / 8 % C) * kAppRows;
  if (row0 >= a.n_rows) return;  // padding of the last chunks
  const int nr = (int)min<int64_t>(kAppRows, (int64_t)a.n_rows - row0);

  // ---- loads: lanes 0..nr-1 of wave 0 read their row's sequence and
  // position, then every thread issues its quantize tasks' source loads
  // (tasks (row, kind, block, lane), lane fastest; dtype and rule fixed at
  // compile time, rows past the last read as the last row and never
  // written), all before the first wait; the page lookup that needs the
  // position follows, so wave 0's critical path is two dependent loads
  const bool resolver = tid < 64;
  int32_t seq = -1, pos = -1;
  if (resolver && tid < nr) {
    seq = a.seq_ids[row0 + tid];
    pos = a.positions[row0 + tid];
  }
  // kWhole (32-row workgroups): one lane per (row, kind, block) task, its 32
  // values in registers (q8_quantize_block: no shuffles, one scale per
  // lane); 8-row workgroups keep 4 lanes per block so that every thread has
  // a task.  Tasks run block fastest, so consecutive lanes read consecutive
  // source bytes.
  constexpr bool kWhole = kAppRows == 32;
  constexpr int kVPL = kWhole ? 32 : 8;  // values per lane and task
  constexpr int kTasks = kAppRows * 2 * NB * (32 / kVPL);
  constexpr int kPer = kTasks / 256;
  static_assert(kTasks % 256 == 0, "every thread takes part in every task round");
  float v[kPer][kVPL];
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int t = 256 * i + tid;
    const int sub = kWhole ? 0 : t & 3;
    const int tb = kWhole ? t : t >> 2;
    const int blk = tb % NB;
    const int kind = (tb / NB) & 1;
    const int r = min(tb / NB / 2, nr - 1);
    const uint64_t off = ((uint64_t)(row0 + r) * (uint64_t)g.kv_heads + (uint64_t)kvh) * D +
                         (uint64_t)(blk * 32 + sub * 8);
#pragma unroll
    for (int e = 0; e < kVPL / 8; ++e)
      load_src8<kBf16>(kind == 0 ? a.k_src : a.v_src, off + 8 * e, &v[i][8 * e]);
  }

  // ---- rows' destinations (wave 0) --------------------------------------
  if (resolver) {
    int64_t base = -1;
    int32_t slot = 0;
    if (tid < nr) {
      if (seq < 0 || seq >= a.n_seqs) {
        if (kvh == 0) atomicOr(a.fault, FAULT_BAD_SEQ);
      } else if (pos < 0 || pos / g.page_tokens >= a.bt_stride) {
        if (kvh == 0) atomicOr(a.fault, FAULT_BAD_POSITION);
      } else {
        const int32_t page = a.bt[(int64_t)seq * a.bt_stride + pos / g.page_tokens];
        if (page < 0 || page >= g.num_pages) {
          if (kvh == 0) atomicOr(a.fault, FAULT_BAD_PAGE);
        } else {
          base = (int64_t)region_base(g, page, kvh, 0);
          slot = pos % g.page_tokens;
        }
      }
    }
    // rows 4i..4i+3 form a quad when they are 4 aligned consecutive slots of one page
    bool run = base >= 0 && slot % 4 == 0;
#pragma unroll
    for (int i = 1; i < 4; ++i) {
      const int64_t b2 = __shfl_down(base, i);
      const int32_t s2 = __shfl_down(slot, i);
      run = run && b2 == base && s2 == slot + i;
    }
    const uint64_t starts = __ballot(run);
    if (tid < kAppRows) {
      rbase[tid] = base;
      rslot[tid] = slot;
      if ((tid & 3) == 0) quad[tid >> 2] = run;
    }
    if (tid == 0) {
      constexpr uint32_t kAll = 0x11111111u >> (32 - (kAppRows - 4));
      shifted = 0;
      for (int i = 1; i < 4; ++i)
        if (((uint32_t)(starts >> i) & kAll) == kAll) shifted = i;
    }
  }

  // ---- quantize into LDS ---------------------------------------------------
#pragma unroll
  for (int i = 0; i < kPer; ++i) {
    const int t = 256 * i + tid;
    const int sub = kWhole ? 0 : t & 3;
    const int tb = kWhole ? t : t >> 2;
    const int blk = tb % NB;
    const int kind = (tb / NB) & 1;
    const int r = tb / NB / 2;
    uint16_t scale;
    if constexpr (kWhole) {
      uint32_t c[8];
      q8_quantize_block(v[i], kRule, scale, c);
      const uint32_t bias = kind == 1 ? 0x80808080u : 0u;  // V codes are stored biased (code_bias)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<uint2 *>(&codes[kind][r][blk * 32 + 8 * j]) =
            uint2{c[2 * j] ^ bias, c[2 * j + 1] ^ bias};
    } else {
      uint64_t c = q8_quantize_values<8>(v[i], kRule, scale);
      if (kind == 1) c ^= 0x8080808080808080ull;  // V codes are stored biased (code_bias)
      *reinterpret_cast<uint64_t *>(&codes[kind][r][blk * 32 + sub * 8]) = c;
    }
    if (sub == 0) scl[kind][r][blk] = scale;
  }
  __syncthreads();

  uint8_t *pages = a.pages;
  const uint64_t RB = region_bytes(g);
  // K codes: row r's D bytes at slot * D of the K region
  for (int t = tid; t < kAppRows * (D / 16); t += 256) {
    const int r = t / (D / 16), c = t % (D / 16);
    const int64_t b = rbase[r];
    if (b < 0) continue;
    // (LDS rows are 8-byte aligned: two 8-byte reads)
    const uint2 lo = *reinterpret_cast<const uint2 *>(&codes[0][r][16 * c]);
    const uint2 hi = *reinterpret_cast<const uint2 *>(&codes[0][r][16 * c + 8]);
    *reinterpret_cast<uint4 *>(pages + b + (uint64_t)rslot[r] * D + 16 * c) = uint4{lo.x, lo.y, hi.x, hi.y};
  }
  // V codes: tasks (4-row group, dim), group fastest
  // (8-row workgroups hold one such quad at most)
  const int shift = kAppRows > 8 ? shifted : 0;
  if (shift > 0) {
    constexpr int kGroups = kAppRows / 4;
    for (int t = tid; t < kGroups * D; t += 256) {
      const int q = t % kGroups, d = t / kGroups, r = 4 * q + shift;
      if (q == kGroups - 1) continue;
      uint32_t w = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) w |= (uint32_t)codes[1][r + i][d] << (8 * i);
      *reinterpret_cast<uint32_t *>(pages + rbase[r] + RB + code_offset(g, 1, rslot[r], d)) = w;
    }
    // the rows before and behind the quads, byte by byte
    for (int t = tid; t < 4 * D; t += 256) {
      const int i = t % 4, d = t / 4, r = i < shift ? i : kAppRows - 4 + i;
      if (rbase[r] >= 0) pages[rbase[r] + RB + code_offset(g, 1, rslot[r], d)] = codes[1][r][d];
    }
  } else {
    for (int t = tid; t < (kAppRows / 4) * D; t += 256) {
      const int q = t % (kAppRows / 4), d = t / (kAppRows / 4);
      const int r = 4 * q;
      uint32_t w = 0;
#pragma unroll
      for (int i = 0; i < 4; ++i) w |= (uint32_t)codes[1][r + i][d] << (8 * i);
      if (quad[q]) {
        *reinterpret_cast<uint32_t *>(pages + rbase[r] + RB + code_offset(g, 1, rslot[r], d)) = w;
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (rbase[r + i] >= 0)
            pages[rbase[r + i] + RB + code_offset(g, 1, rslot[r + i], d)] = (uint8_t)(w >> (8 * i));
      }
    }
  }
  // scales: tasks (row, block, kind), row fastest
  for (int t = tid; t < 2 * NB * kAppRows; t += 256) {
    const int r = t % kAppRows, blk = (t / kAppRows) % NB, kind = t / (kAppRows * NB);
    const int64_t b = rbase[r];
    if (b < 0) continue;
    *reinterpret_cast<uint16_t *>(pages + b + kind * RB + scale_offset(g, rslot[r], blk)) =
        scl[kind][r][blk];
  }
}

// Export (gather) and import of positions [0, len) of one sequence: one
// 128-thread workgroup per (tile of the positions, kv head), moving the tile
// through an LDS image of its rows (rkv_rows.h).  A 32,768-token sequence (D =
// 256, 2 kv heads, 17.8 MB read and 17.8 MB written per kind) took 77 us to
// gather and 62 us to import with one thread per 34-byte block and byte
// accesses.  The tile form's gather takes 8.0 us for K and 17.0 for V, its
// import 9.0 and 14.6 (kernel trace; 4.5, 2.1, 4.0 and 2.4 TB/s read and
// written): K moves at about the rate of a large copy, V, whose lanes' 16
// bytes lie 128 apart, at half of it.
template <int D>
__global__ __launch_bounds__(kRowsThreads) void gather_kernel(Geo g, const uint8_t *pages, const int32_t *bt,
                                                              int32_t len, int32_t kind, uint8_t *rows,
                                                              int32_t *fault) {
  __shared__ __attribute__((aligned(16))) uint16_t img[RowsImage<D>::kBytes / 2];
  const int32_t TT = tile_tokens(g.page_tokens), p0 = (int32_t)blockIdx.x * TT, kvh = (int32_t)blockIdx.y;
  const int32_t page = bt[p0 / g.page_tokens];
  if (page < 0 || page >= g.num_pages) {
    if (threadIdx.x == 0) atomicOr(fault, FAULT_BAD_PAGE);
    return;
  }
  tile_to_image<D>(load_tile<D>(g, pages + region_base(g, page, kvh, kind), kind, p0 % g.page_tokens, TT), kind, TT,
                   img);
  __syncthreads();
  constexpr int32_t RB = 2 * RowsImage<D>::kRowHalves;
  store_run(rows + ((int64_t)kvh * len + p0) * RB, reinterpret_cast<const uint8_t *>(img), min(TT, len - p0) * RB);
}

template <int D>
__global__ __launch_bounds__(kRowsThreads) void import_kernel(Geo g, uint8_t *pages, const int32_t *bt, int32_t len,
                                                              int32_t kind, const uint8_t *rows, int32_t *fault) {
  __shared__ __attribute__((aligned(16))) uint16_t img[RowsImage<D>::kBytes / 2];
  const int32_t TT = tile_tokens(g.page_tokens), p0 = (int32_t)blockIdx.x * TT, kvh = (int32_t)blockIdx.y;
  const int32_t page = bt[p0 / g.page_tokens];
  if (page < 0 || page >= g.num_pages) {
    if (threadIdx.x == 0) atomicOr(fault, FAULT_BAD_PAGE);
    return;
  }
  constexpr int32_t RB = 2 * RowsImage<D>::kRowHalves;
  const int32_t n = min(TT, len - p0);
  load_run(reinterpret_cast<uint8_t *>(img), rows + ((int64_t)kvh * len + p0) * RB, n * RB);
  __syncthreads();
  image_to_tile<D>(g, pages + region_base(g, page, kvh, kind), kind, p0 % g.page_tokens, TT, 0, n, img);
}

// The drop-in decode's scratch pages from contiguous K and V rows: page i
// holds tokens page_tokens*i on, and workgroup (x, 0, 0) writes the block
// table's entries, length and sequence id that the decode then reads.  (As
// three copies from host memory, a stream synchronization and an import per
// kind, a 1024-token call of 24 query and 4 kv heads took 58 us, with this
// launch 30.)
template <int D>
__global__ __launch_bounds__(kRowsThreads) void flash_import_kernel(Geo g, uint8_t *pages, const uint8_t *k_rows,
                                                                    const uint8_t *v_rows, int32_t len, int32_t *bt,
                                                                    int32_t *seq_len, int32_t *seq_id) {
  __shared__ __attribute__((aligned(16))) uint16_t img[RowsImage<D>::kBytes / 2];
  constexpr int32_t RB = 2 * RowsImage<D>::kRowHalves;
  const int32_t TT = tile_tokens(g.page_tokens), p0 = (int32_t)blockIdx.x * TT;
  const int32_t kvh = (int32_t)blockIdx.y, kind = (int32_t)blockIdx.z;
  const int32_t page = p0 / g.page_tokens, n = min(TT, len - p0);
  if (kvh == 0 && kind == 0 && threadIdx.x == 0) {
    if (p0 % g.page_tokens == 0) bt[page] = page;
    if (blockIdx.x == 0) {
      *seq_len = len;
      *seq_id = 0;
    }
  }
  if (n <= 0) return;
  load_run(reinterpret_cast<uint8_t *>(img), (kind == 0 ? k_rows : v_rows) + ((int64_t)kvh * len + p0) * RB, n * RB);
  __syncthreads();
  image_to_tile<D>(g, pages + region_base(g, page, kvh, kind), kind, p0 % g.page_tokens, TT, 0, n, img);
}

__global__ __launch_bounds__(256) void f32_to_f16_kernel(const float *in, uint16_t *out, int64_t n,
                                                         int32_t rule) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  out[i] = rule == 0 ? f16_rtne(in[i]) : f16_harserve(in[i]);
}

inline unsigned grid_for(int64_t threads) { return (unsigned)((threads + 255) / 256); }

}  // namespace

namespace {
template <int D, int ROWS>
void launch_append_r(const AppendLaunch &a, hipStream_t s) {
  const int64_t blocks = ((int64_t)a.n_rows + ROWS - 1) / ROWS, round = 8 * kAppChunk<ROWS>;
  const dim3 grid((unsigned)((blocks + round - 1) / round * round), (unsigned)a.g.kv_heads);
  if (a.src_bf16) {
    if (a.rule == 0) hipLaunchKernelGGL((append_kernel<D, ROWS, true, 0>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((append_kernel<D, ROWS, true, 1>), grid, dim3(256), 0, s, a);
  } else {
    if (a.rule == 0) hipLaunchKernelGGL((append_kernel<D, ROWS, false, 0>), grid, dim3(256), 0, s, a);
    else hipLaunchKernelGGL((append_kernel<D, ROWS, false, 1>), grid, dim3(256), 0, s, a);
  }
}
template <int D>
void launch_append_d(const AppendLaunch &a, hipStream_t s) {
  // 32-row workgroups once there are at least 8 per CU, else 8-row ones
  if ((int64_t)a.n_rows * a.g.kv_heads >= (int64_t)32 * 8 * kComputeUnits)
    launch_append_r<D, 32>(a, s);
  else
    launch_append_r<D, 8>(a, s);
}
}  // namespace

hipError_t launch_append(const AppendLaunch &a, hipStream_t s) {
  if (a.n_rows <= 0) return hipSuccess;
  if (a.g.head_dim == 256) launch_append_d<256>(a, s);
  else launch_append_d<128>(a, s);
  return hipGetLastError();
}

hipError_t launch_gather(const Geo &g, const uint8_t *pages, const int32_t *bt, int32_t len,
                         int32_t kind, uint8_t *rows, int32_t *fault, hipStream_t s) {
  if (len <= 0) return hipSuccess;
  const int32_t TT = tile_tokens(g.page_tokens);
  const dim3 grid((unsigned)((len + (int64_t)TT - 1) / TT), (unsigned)g.kv_heads);
  if (g.head_dim == 256)
    hipLaunchKernelGGL(gather_kernel<256>, grid, dim3(kRowsThreads), 0, s, g, pages, bt, len, kind, rows, fault);
  else
    hipLaunchKernelGGL(gather_kernel<128>, grid, dim3(kRowsThreads), 0, s, g, pages, bt, len, kind, rows, fault);
  return hipGetLastError();
}

hipError_t launch_import(const Geo &g, uint8_t *pages, const int32_t *bt, int32_t len,
                         int32_t kind, const uint8_t *rows, int32_t *fault, hipStream_t s) {
  if (len <= 0) return hipSuccess;
  const int32_t TT = tile_tokens(g.page_tokens);
  const dim3 grid((unsigned)((len + (int64_t)TT - 1) / TT), (unsigned)g.kv_heads);
  if (g.head_dim == 256)
    hipLaunchKernelGGL(import_kernel<256>, grid, dim3(kRowsThreads), 0, s, g, pages, bt, len, kind, rows, fault);
  else
    hipLaunchKernelGGL(import_kernel<128>, grid, dim3(kRowsThreads), 0, s, g, pages, bt, len, kind, rows, fault);
  return hipGetLastError();
}

hipError_t launch_flash_import(const Geo &g, uint8_t *pages, const uint8_t *k_rows, const uint8_t *v_rows,
                               int32_t len, int32_t *bt, int32_t *seq_len, int32_t *seq_id, hipStream_t s) {
  const int64_t tiles = ((int64_t)len + tile_tokens(g.page_tokens) - 1) / tile_tokens(g.page_tokens);
  const dim3 grid((unsigned)std::max<int64_t>(tiles, 1), (unsigned)g.kv_heads, 2);
  if (g.head_dim == 256)
    hipLaunchKernelGGL(flash_import_kernel<256>, grid, dim3(kRowsThreads), 0, s, g, pages, k_rows, v_rows, len, bt,
                       seq_len, seq_id);
  else
    hipLaunchKernelGGL(flash_import_kernel<128>, grid, dim3(kRowsThreads), 0, s, g, pages, k_rows, v_rows, len, bt,
                       seq_len, seq_id);
  return hipGetLastError();
}

namespace {
// Unpack a block-table update: `n_rows` records of [seq][W page ids] then
// the lengths of all `n_seqs` sequences.  Block i < n_rows copies record i;
// block n_rows copies the lengths.
// `packed` is the host's pinned staging buffer, read over the host link
// (no separate copy).  When every block has read it, the last one to finish
// stores `seq` to the host-visible word `done`, which tells the host that
// the buffer may be rewritten: each block counts itself in the device
// counter `count` (never reset; the launch's blocks are the counts from
// `last` - gridDim.x + 1 to `last`).
__global__ __launch_bounds__(256) void table_scatter_kernel(const int32_t *packed, int32_t n_rows,
                                                           int32_t W, int32_t n_seqs,
                                                           int32_t *tables, int32_t *lens,
                                                           unsigned long long *count,
                                                           unsigned long long last,
                                                           unsigned long long *done,
                                                           unsigned long long seq) {
  const int32_t r = blockIdx.x;
  if (r < n_rows) {
    const int32_t *rec = packed + (int64_t)r * (W + 1);
    const int32_t sq = rec[0];
    if (sq >= 0 && sq < n_seqs)  // packed by the host from its own table
      for (int32_t i = threadIdx.x; i < W; i += 256) tables[(int64_t)sq * W + i] = rec[1 + i];
  } else {
    const int32_t *src = packed + (int64_t)n_rows * (W + 1);
    for (int32_t i = threadIdx.x; i < n_seqs; i += 256) lens[i] = src[i];
  }
  // every value read above was stored, so the block's reads are done
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    if (atomicAdd(count, 1ull) == last) {
      __threadfence_system();
      __hip_atomic_store(done, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
  }
}

// Copy-on-write page copies: for each (src, dst) pair and each of `layers`
// layer arrays, page dst := page src.  A unit is one 16 KiB piece of one
// (pair, layer) page; each block walks units with a grid stride and each
// thread moves four 16-byte vectors per unit, all loads issued before the
// stores.  Pairs naming pages outside [0, num_pages) are skipped.
constexpr int32_t kCopyVecs = 4;
constexpr int32_t kCopyUnitBytes = 256 * 16 * kCopyVecs;

__global__ __launch_bounds__(256) void copy_pages_kernel(uint8_t *pages, int64_t layer_stride,
                                                         int32_t layers, int32_t num_pages,
                                                         const int32_t *pairs, int64_t page_bytes,
                                                         int32_t units_per_page, int64_t n_units) {
  for (int64_t u = blockIdx.x; u < n_units; u += gridDim.x) {
    const int64_t pl = u / units_per_page;
    const int32_t part = (int32_t)(u - pl * units_per_page);
    const int32_t layer = (int32_t)(pl % layers);
    const int64_t pair = pl / layers;
    const int32_t src = pairs[2 * pair], dst = pairs[2 * pair + 1];
    if (src < 0 || src >= num_pages || dst < 0 || dst >= num_pages) continue;
    const uint8_t *from = pages + layer * layer_stride + (int64_t)src * page_bytes;
    uint8_t *to = pages + layer * layer_stride + (int64_t)dst * page_bytes;
    const int64_t base = (int64_t)part * kCopyUnitBytes + (int64_t)threadIdx.x * 16;
    uint4 v[kCopyVecs];
#pragma unroll
    for (int32_t k = 0; k < kCopyVecs; ++k) {
      const int64_t off = base + (int64_t)k * 256 * 16;
      if (off < page_bytes) v[k] = *reinterpret_cast<const uint4 *>(from + off);
    }
#pragma unroll
    for (int32_t k = 0; k < kCopyVecs; ++k) {
      const int64_t off = base + (int64_t)k * 256 * 16;
      if (off < page_bytes) *reinterpret_cast<uint4 *>(to + off) = v[k];
    }
  }
}
}  // namespace

hipError_t launch_copy_pages(uint8_t *pages, int64_t layer_stride, int32_t layers,
                             int32_t num_pages, const int32_t *pairs, int32_t n_pairs,
                             int64_t page_bytes, hipStream_t s) {
  if (n_pairs <= 0 || layers <= 0) return hipSuccess;
  const int32_t units_per_page = (int32_t)((page_bytes + kCopyUnitBytes - 1) / kCopyUnitBytes);
  const int64_t n_units = (int64_t)n_pairs * layers * units_per_page;
  const unsigned grid = (unsigned)std::min<int64_t>(n_units, 8192);
  hipLaunchKernelGGL(copy_pages_kernel, dim3(grid), dim3(256), 0, s, pages, layer_stride, layers,
                     num_pages, pairs, page_bytes, units_per_page, n_units);
  return hipGetLastError();
}

hipError_t launch_table_scatter(const int32_t *packed, int32_t n_rows, int32_t W, int32_t n_seqs,
                                int32_t *tables, int32_t *lens, unsigned long long *count,
                                unsigned long long last, unsigned long long *done,
                                unsigned long long seq, hipStream_t s) {
  hipLaunchKernelGGL(table_scatter_kernel, dim3((unsigned)n_rows + 1), dim3(256), 0, s, packed,
                     n_rows, W, n_seqs, tables, lens, count, last, done, seq);
  return hipGetLastError();
}

hipError_t launch_f32_to_f16(const float *in, uint16_t *out, int64_t n, int32_t rule,
                             hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(f32_to_f16_kernel, dim3(grid_for(n)), dim3(256), 0, s, in, out, n, rule);
  return hipGetLastError();
}

}  // namespace rkv
