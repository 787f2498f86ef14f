// Exact-wide magnitude proofs on the device (reference
// src/core/exact_range.hpp:34-157, api_gemm.cpp:870-874):
//
// * native_axes: the per-row and per-column summaries of a 64-bit operand at
//   pack time, one launch. Row blocks give a wave to each row, column blocks
//   take 8 columns whole, so every axis's extremes, sums and centre are known
//   where its values were read: the values stay in registers (up to 2048 of a
//   row, 1024 of a column; longer axes read them again) for the deviation sums
//   around that centre, and nothing goes through partial summaries. The last
//   row block to finish writes the operand's max |x|. Few long axes, and large
//   operands, run in the tile form instead (native_axes_tiled).
// * product_axes: the cell bounds of C = A x B from A's row records and B's
//   column records, reduced per row (one wave per row) and per column (one
//   wave per column), and C's bound min(k maxA maxB, max cell).
// * proof_snapshot: the records and maxima a GEMM result keeps until its own
//   summaries are needed.
//
// The arithmetic is exact_axes.hpp's, shared with the host tests.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

#include "exact_axes.hpp"
#include "kernels.hpp"

namespace rns8x {
namespace {

using namespace xa;

typedef unsigned long long v2u64 __attribute__((ext_vector_type(2)));

constexpr int kThreads = 512, kWaves = kThreads / 64;
constexpr int kHoldRow = 16, kHoldCol = 4;  // pairs of values a lane holds
constexpr int kColsPerBlock = 8;           // 4 lanes of 2 columns; kThreads / 4 rows per load
constexpr int kRowLanes = kThreads / 4;
constexpr int64_t kMaxBlocks = 8192;       // of either kind; larger operands stride

// Merges the lanes whose index differs in bits kFrom .. 32.
template <int kFrom, bool Signed>
__device__ __forceinline__ void merge_lanes(Extremes<Signed>& e) {
#pragma unroll
  for (int m = kFrom; m < 64; m <<= 1) {
    Extremes<Signed> o;
    o.hi = __shfl_xor(e.hi, m);
    o.lo = __shfl_xor(e.lo, m);
    o.sum.lo = __shfl_xor(e.sum.lo, m);
    o.sum.hi = __shfl_xor(e.sum.hi, m);
    if constexpr (Signed) {
      o.pos.lo = __shfl_xor(e.pos.lo, m);
      o.pos.hi = __shfl_xor(e.pos.hi, m);
    }
    e.merge(o);
  }
}
template <int kFrom>
__device__ __forceinline__ void merge_lanes(Sum96& s) {
#pragma unroll
  for (int m = kFrom; m < 64; m <<= 1) {
    const u64 o = __shfl_xor(s.lo, m);
    s.add(o, __shfl_xor(s.hi, m));
  }
}

// Two neighbouring values at `off` bytes from a uniform address (16-byte
// aligned where kVec), of which the first `n` exist (0, 1, 2 or more). The
// address stays in scalar registers: eight 64-bit addresses in flight per lane
// made the column blocks spill.
template <bool kVec, typename Off>
__device__ __forceinline__ v2u64 load_pair(const uint64_t* base, Off off, int64_t n) {
  const char* const p = reinterpret_cast<const char*>(base) + off;
  v2u64 v = {0, 0};
  if (kVec && n >= 2) {
    v = *reinterpret_cast<const v2u64*>(p);
  } else {
    if (n >= 1) v[0] = *reinterpret_cast<const uint64_t*>(p);
    if (n >= 2) v[1] = *reinterpret_cast<const uint64_t*>(p + 8);
  }
  return v;
}

// What bounds this kernel is its arithmetic (about 25 operations per value and
// direction, at four waves per SIMD) and, on small operands, the latency of
// its loads and reductions. At 2048 x 2048 it takes 24 us, at 500 x 701 10 us;
// the four launches it replaces (two passes over 64 x 64 LDS tiles, each
// followed by a merge of the tiles' partials) took 14 + 6 + 11 + 5 and 20 us.
// Where that is not so, the tile form below runs (native_axes_tiled).
// kVec: 16-byte loads; kFar: 64-bit lane offsets (row strides from 2^21 on).
template <bool Signed, bool kVec, bool kFar>
__global__ __launch_bounds__(kThreads, 4) void native_axes_kernel(const uint64_t* __restrict__ src, int64_t rows,
                                                                  int64_t cols, int64_t ld, uint32_t col_blocks,
                                                                  uint32_t row_blocks,
                                                                  AxisRecord* __restrict__ out_rows,
                                                                  AxisRecord* __restrict__ out_cols,
                                                                  u64* __restrict__ words, ProofTicket* ticket) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (blockIdx.x >= col_blocks) {
    // ---- rows: one wave per row, lane l takes columns 128 j + 2 l, + 1 ----
    __shared__ u64 wave_best[kWaves];
    u64 best = 0;
    for (int64_t r = static_cast<int64_t>(blockIdx.x - col_blocks) * kWaves + wave; r < rows;
         r += static_cast<int64_t>(row_blocks) * kWaves) {
      const uint64_t* const row = src + r * ld;
      v2u64 v[kHoldRow];
      auto fetch = [&](int64_t c0) {
        const bool full = c0 + 128 * kHoldRow <= cols;
#pragma unroll
        for (int j = 0; j < kHoldRow; ++j) {
          const int64_t left = cols - (c0 + 128 * j);  // uniform, as the address but for the lane
          v[j] = load_pair<kVec>(row + c0 + 128 * j, 16u * lane, full ? 2 : left - 2 * lane);
        }
      };
      // f(u) of every value of the chunk at c0
      auto each = [&](int64_t c0, auto f) {
        if (c0 + 128 * kHoldRow <= cols) {
#pragma unroll
          for (int j = 0; j < kHoldRow; ++j) {
            f(bias(v[j][0], Signed));
            f(bias(v[j][1], Signed));
            __builtin_amdgcn_sched_barrier(0);
          }
        } else {
#pragma unroll
          for (int j = 0; j < kHoldRow; ++j) {
            const int64_t left = cols - (c0 + 128 * j);
            const int n = static_cast<int>(left < 128 ? left : 128) - 2 * lane;
            if (n > 0) f(bias(v[j][0], Signed));
            if (n > 1) f(bias(v[j][1], Signed));
          }
        }
      };
      Extremes<Signed> acc;
      for (int64_t c0 = 0; c0 < cols; c0 += 128 * kHoldRow) {
        fetch(c0);
        each(c0, [&](u64 u) { acc.add(u); });
      }
      merge_lanes<1>(acc);
      // the record is stored before the second pass and its deviation sum
      // after it: held meanwhile, its 32 registers would spill
      u64 cu;
      u128 sum;
      {
        const AxisPartial p = acc.partial(static_cast<u64>(cols));
        const AxisRecord rec = native_record(p, static_cast<u64>(cols), Signed);
        if (lane == 0) out_rows[r] = rec;
        cu = bias(static_cast<u64>(record_centre(rec)), Signed);
        sum = p.sum;
        best = rec.max_magnitude[0] > best ? rec.max_magnitude[0] : best;
      }
      Sum96 above;
      for (int64_t c0 = 0; c0 < cols; c0 += 128 * kHoldRow) {
        if (cols > 128 * kHoldRow) fetch(c0);
        each(c0, [&](u64 u) { add_above(above, u, cu); });
      }
      merge_lanes<1>(above);
      if (lane == 0)
        put_u128(out_rows[r].deviation_sum, deviation_total(above, sum, static_cast<u64>(cols), cu));
    }
    if (lane == 0) wave_best[wave] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
      for (int w = 1; w < kWaves; ++w) best = wave_best[w] > best ? wave_best[w] : best;
      // The block's maximum is in before its ticket is drawn (the wait), so
      // the block that draws the last one reads everybody's. The count wraps
      // to zero by itself: packs of one matrix that overlap (a caller's
      // error, and their maxima may mix) still draw whole multiples of
      // row_blocks, so the next pack starts from a clean ticket.
      const u64 before = __hip_atomic_fetch_max(&ticket->best, best, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      asm volatile("s_waitcnt vmcnt(0)" ::"v"(before) : "memory");
      if (atomicInc(&ticket->drawn, row_blocks - 1) == row_blocks - 1) {
        words[0] = __hip_atomic_exchange(&ticket->best, u64{0}, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        for (int i = 1; i < 8; ++i) words[i] = 0;
      }
    }
    return;
  }
  // ---- columns: 8 per block, lane l takes columns 2 (l % 4), + 1 of rows
  // kRowLanes j + 16 wave + l / 4 ----
  __shared__ AxisPartial part[kWaves][kColsPerBlock];
  __shared__ u128 dpart[kWaves][kColsPerBlock];
  __shared__ u64 centre_of[kColsPerBlock];
  __shared__ u128 sum_of[kColsPerBlock];
  // Blocks b and b + 8 run on one XCD: they take neighbouring columns, the two
  // halves of a cache line.
  const int64_t groups = (cols + kColsPerBlock - 1) / kColsPerBlock;
  const int pair = 2 * (lane & 3), rl = 16 * wave + (lane >> 2);
  for (int64_t b = blockIdx.x; b < (groups + 15) / 16 * 16; b += col_blocks) {
    const int64_t g = b / 16 * 16 + 2 * (b & 7) + (b >> 3 & 1);
    if (g >= groups) continue;
    const uint64_t* const col = src + g * kColsPerBlock;
    // (a pair past the last column reads nothing and is not stored)
    const int n = static_cast<int>(cols - g * kColsPerBlock < kColsPerBlock ? cols - g * kColsPerBlock : kColsPerBlock) - pair;
    using Off = std::conditional_t<kFar, uint64_t, uint32_t>;
    const Off off = (static_cast<Off>(rl) * static_cast<Off>(ld) + static_cast<Off>(pair)) * 8u;
    // rows of load j of the chunk at r0 that exist, from this wave's first
    auto rows_left = [&](int64_t r0, int j) {
      const int64_t left = rows - (r0 + kRowLanes * j + 16 * wave);
      return static_cast<int>(left < 16 ? left : 16);
    };
    v2u64 va[kHoldCol], vb[kHoldCol];
    auto fetch = [&](v2u64(&v)[kHoldCol], int64_t r0) {
#pragma unroll
      for (int j = 0; j < kHoldCol; ++j) {
        v[j] = load_pair<kVec>(col + (r0 + kRowLanes * j) * ld, off, (lane >> 2) < rows_left(r0, j) ? n : 0);
      }
    };
    auto each = [&](const v2u64(&v)[kHoldCol], int64_t r0, auto f) {
      if (r0 + kRowLanes * kHoldCol <= rows) {
#pragma unroll
        for (int j = 0; j < kHoldCol; ++j) {
          f(bias(v[j][0], Signed), bias(v[j][1], Signed));
          __builtin_amdgcn_sched_barrier(0);
        }
      } else {
#pragma unroll
        for (int j = 0; j < kHoldCol; ++j)
          if ((lane >> 2) < rows_left(r0, j)) f(bias(v[j][0], Signed), bias(v[j][1], Signed));
      }
    };
    // f(a, b) over the two columns' values, the next chunk's loads in flight;
    // up to two chunks stay in registers for the second sweep
    constexpr int64_t kChunk = kRowLanes * kHoldCol;
    auto sweep = [&](bool again, auto f) {
      const bool load = !again || rows > 2 * kChunk;
      if (load) fetch(va, 0);
      for (int64_t r0 = 0; r0 < rows; r0 += 2 * kChunk) {
        if (load) fetch(vb, r0 + kChunk);
        each(va, r0, f);
        if (load && r0 + 2 * kChunk < rows) fetch(va, r0 + 2 * kChunk);
        each(vb, r0 + kChunk, f);
      }
    };
    Extremes<Signed> acc[2];
    sweep(false, [&](u64 a, u64 b2) {
      acc[0].add(a);
      acc[1].add(b2);
    });
    // the lane classes' shares of the rows: partials of all waves add up, so
    // the count enters once (wave 0's partial)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      merge_lanes<4>(acc[e]);
      if (lane < 4) part[wave][pair + e] = acc[e].partial(wave == 0 ? static_cast<u64>(rows) : 0);
    }
    __syncthreads();
    const bool owner = threadIdx.x < kColsPerBlock && g * kColsPerBlock + threadIdx.x < cols;
    AxisRecord* const out = out_cols + g * kColsPerBlock + threadIdx.x;
    if (threadIdx.x < kColsPerBlock) {
      AxisPartial p = part[0][threadIdx.x];
#pragma unroll 1
      for (int w = 1; w < kWaves; ++w) partial_merge(p, part[w][threadIdx.x]);
      const AxisRecord rec = native_record(p, static_cast<u64>(rows), Signed);
      if (owner) *out = rec;
      centre_of[threadIdx.x] = bias(static_cast<u64>(record_centre(rec)), Signed);
      sum_of[threadIdx.x] = p.sum;
    }
    __syncthreads();
    const u64 cu0 = centre_of[pair], cu1 = centre_of[pair + 1];
    Sum96 above[2];
    sweep(true, [&](u64 a, u64 b2) {
      add_above(above[0], a, cu0);
      add_above(above[1], b2, cu1);
    });
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      merge_lanes<4>(above[e]);
      if (lane < 4) dpart[wave][pair + e] = above[e].value();
    }
    __syncthreads();
    if (owner) {
      u128 sum = 0;
#pragma unroll 1
      for (int w = 0; w < kWaves; ++w) sum += dpart[w][threadIdx.x];
      Sum96 total;
      total.lo = static_cast<u64>(sum);
      total.hi = static_cast<uint32_t>(sum >> 64);
      put_u128(out->deviation_sum,
               deviation_total(total, sum_of[threadIdx.x], static_cast<u64>(rows), centre_of[threadIdx.x]));
    }
  }
}

// ---- the tile form: operands with few long axes, and large ones -------------
// (native_axes_tiled says which, with both forms' times). Two passes over 64 x
// 64 tiles staged in LDS, each followed by a merge of the tiles' partials: four
// launches, but a long axis is spread over the chip, and each pass reads the
// operand once for both directions.

constexpr int kTile = 64;
constexpr int64_t kMaxGridY = 65535;
// Elements of a half-tile run read per batch: the batch's LDS reads issue
// together and one wait covers them (a rolled loop waits on every read).
constexpr int kWalkBatch = 8;

// f(elem(j)) for j in [j0, j1): whole 32-element runs (every run of a full
// tile) in batches of kWalkBatch reads, ragged ones one element at a time.
template <typename E, typename F>
__device__ __forceinline__ void walk_run(int j0, int j1, E elem, F f) {
  if (j1 - j0 == kTile / 2) {
#pragma unroll 1
    for (int b = 0; b < kTile / 2; b += kWalkBatch) {
      u64 v[kWalkBatch];
#pragma unroll
      for (int e = 0; e < kWalkBatch; ++e) v[e] = elem(j0 + b + e);
#pragma unroll
      for (int e = 0; e < kWalkBatch; ++e) f(v[e]);
    }
  } else {
    for (int j = j0; j < j1; ++j) f(elem(j));
  }
}

// One pass over the 64 x 64 tiles of a rows x cols operand (row stride ld).
// Block (x, y) takes tile column x and tile rows y, y + gridDim.y, ...; each
// lane holds its 16 elements of the next tile in registers, loaded while the
// current tile is summarized. Partials: row r of tile column x at
// row_part[x * rows + r], column c of tile row y at col_part[y * cols + c].
// Pass 1 (Dev = false) also clears the result's 8 proof words (block (0,
// 0)), which the finishing launch fills; pass 2 reads the axis centres from
// the records pass 1 finished.
template <bool Signed, bool Dev>
__global__ __launch_bounds__(256) void tiled_axes_pass(const uint64_t* __restrict__ src, int64_t rows, int64_t cols,
                                                       int64_t ld, AxisPartial* __restrict__ row_part,
                                                       AxisPartial* __restrict__ col_part,
                                                       const AxisRecord* __restrict__ row_rec,
                                                       const AxisRecord* __restrict__ col_rec, u64* __restrict__ words) {
  // the tile as 32-bit halves at a row stride of 65 words: row and column
  // reads are both free of bank conflicts
  __shared__ uint32_t tile_lo[kTile][kTile + 1], tile_hi[kTile][kTile + 1];
  __shared__ AxisPartial second[2][kTile];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t c0 = static_cast<int64_t>(blockIdx.x) * kTile;
  const int nc = static_cast<int>(cols - c0 < kTile ? cols - c0 : kTile);
  if (!Dev && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x < 8) words[threadIdx.x] = 0;
  // waves 0, 1: rows (lane = row) over column halves; waves 2, 3: columns
  // (lane = column) over row halves
  const bool by_row = wave < 2;
  const int half = wave & 1;
  i128 col_centre = 0;
  if (Dev && !by_row && lane < nc) col_centre = record_centre(col_rec[c0 + lane]);
  const int64_t tiles_y = (rows + kTile - 1) / kTile;
  // rows wave, wave + 4, ..., wave + 60 of a tile, column c0 + lane
  u64 next[kTile / 4];
  auto fetch = [&](int64_t ty) {
    const int64_t r0 = ty * kTile;
    const int nr = static_cast<int>(rows - r0 < kTile ? rows - r0 : kTile);
#pragma unroll
    for (int q = 0; q < kTile / 4; ++q) {
      const int i = wave + 4 * q;
      next[q] = lane < nc && i < nr ? src[(r0 + i) * ld + c0 + lane] : 0;
    }
  };
  if (static_cast<int64_t>(blockIdx.y) < tiles_y) fetch(blockIdx.y);
  for (int64_t ty = blockIdx.y; ty < tiles_y; ty += gridDim.y) {
    const int64_t r0 = ty * kTile;
    const int nr = static_cast<int>(rows - r0 < kTile ? rows - r0 : kTile);
    __syncthreads();  // the previous tile's readers are done
#pragma unroll
    for (int q = 0; q < kTile / 4; ++q) {
      tile_lo[wave + 4 * q][lane] = static_cast<uint32_t>(next[q]);
      tile_hi[wave + 4 * q][lane] = static_cast<uint32_t>(next[q] >> 32);
    }
    __syncthreads();
    if (ty + gridDim.y < tiles_y) fetch(ty + gridDim.y);
    const int axes = by_row ? nr : nc, len = by_row ? nc : nr;
    const int j0 = half * 32, j1 = j0 + 32 < len ? j0 + 32 : len;
    AxisPartial p = empty_partial();
    auto row_elem = [&](int j) { return (static_cast<u64>(tile_hi[lane][j]) << 32) | tile_lo[lane][j]; };
    auto col_elem = [&](int j) { return (static_cast<u64>(tile_hi[j][lane]) << 32) | tile_lo[j][lane]; };
    if (lane < axes) {
      if (!Dev) {
        PartialAcc acc;
        if (by_row)
          walk_run(j0, j1, row_elem, [&](u64 x) { acc.add(x, Signed); });
        else
          walk_run(j0, j1, col_elem, [&](u64 x) { acc.add(x, Signed); });
        p = acc.partial();
      } else {
        const i128 centre = by_row ? record_centre(row_rec[r0 + lane]) : col_centre;
        DeviationAcc acc;
        if (by_row)
          walk_run(j0, j1, row_elem, [&](u64 x) { acc.add(deviation(x, centre, Signed)); });
        else
          walk_run(j0, j1, col_elem, [&](u64 x) { acc.add(deviation(x, centre, Signed)); });
        p.sum = acc.value();
      }
    }
    if (half == 1) second[by_row ? 0 : 1][lane] = p;
    __syncthreads();
    if (half == 0 && lane < axes) {
      partial_merge(p, second[by_row ? 0 : 1][lane]);
      if (by_row)
        row_part[static_cast<int64_t>(blockIdx.x) * rows + r0 + lane] = p;
      else
        col_part[ty * cols + c0 + lane] = p;
    }
  }
}

// Merges each axis's partials (rows first, then columns): pass 1 writes the
// records and the operand's max |x| (words[0], an atomic max per block);
// pass 2 adds the deviation sums. A block takes 32 axes; its 8 thread groups
// each merge every 8th partial of them, and group 0 merges the 8 results.
template <bool Signed, bool Dev>
__global__ __launch_bounds__(256) void tiled_axes_finish(const AxisPartial* __restrict__ row_part,
                                                          const AxisPartial* __restrict__ col_part, int64_t rows,
                                                          int64_t cols, AxisRecord* __restrict__ out_rows,
                                                          AxisRecord* __restrict__ out_cols, u64* __restrict__ words) {
  constexpr int kAxes = 32, kGroups = 8;
  __shared__ AxisPartial part_of[kGroups][kAxes];
  __shared__ u64 block_max;
  const int64_t tiles_x = (cols + kTile - 1) / kTile, tiles_y = (rows + kTile - 1) / kTile;
  const int a = threadIdx.x % kAxes, g = threadIdx.x / kAxes;
  if (threadIdx.x == 0) block_max = 0;
  u64 best = 0;
  for (int64_t base = static_cast<int64_t>(blockIdx.x) * kAxes; base < rows + cols;
       base += static_cast<int64_t>(gridDim.x) * kAxes) {
    const int64_t i = base + a;
    const bool valid = i < rows + cols, is_row = i < rows;
    const int64_t axis = is_row ? i : i - rows, stride = is_row ? rows : cols, parts = is_row ? tiles_x : tiles_y;
    AxisPartial p = empty_partial();
    if (valid) {
      const AxisPartial* const part = (is_row ? row_part : col_part) + axis;
      for (int64_t t = g; t < parts; t += kGroups) {
        if (!Dev)
          partial_merge(p, part[t * stride]);
        else
          p.sum += part[t * stride].sum;
      }
    }
    __syncthreads();  // the previous round's readers are done
    part_of[g][a] = p;
    __syncthreads();
    if (g == 0 && valid) {
      for (int h = 1; h < kGroups; ++h) {
        if (!Dev)
          partial_merge(p, part_of[h][a]);
        else
          p.sum += part_of[h][a].sum;
      }
      AxisRecord* const rec = (is_row ? out_rows : out_cols) + axis;
      if (!Dev) {
        // the groups' partials start empty (hi = not_lo = 0 are neutral)
        const AxisRecord r = native_record(p, static_cast<u64>(is_row ? cols : rows), Signed);
        *rec = r;
        if (is_row) best = r.max_magnitude[0] > best ? r.max_magnitude[0] : best;
      } else {
        put_u128(rec->deviation_sum, p.sum);
      }
    }
  }
  if (!Dev) {
    if (best) atomicMax(reinterpret_cast<unsigned long long*>(&block_max), static_cast<unsigned long long>(best));
    __syncthreads();
    if (threadIdx.x == 0 && block_max)
      atomicMax(reinterpret_cast<unsigned long long*>(words), static_cast<unsigned long long>(block_max));
  }
}

struct ProductArgs {
  const AxisRecord* arows;  // m records (unused for a uniform A)
  const AxisRecord* bcols;  // n records (unused for a uniform B)
  AxisKind akind, bkind;
  const u64* amax;  // 4 words: A's bound
  const u64* bmax;  // 4 words: B's bound
  int64_t m, n;
  u64 k;
  AxisRecord* out_rows;
  AxisRecord* out_cols;
  u64* out_words;
};

__device__ __forceinline__ void wave_reduce(U256& mx, U256& sm) {
  for (int off = 32; off > 0; off >>= 1) {
    U256 om, os;
    for (int i = 0; i < 4; ++i) {
      om.w[i] = __shfl_xor(mx.w[i], off);
      os.w[i] = __shfl_xor(sm.w[i], off);
    }
    mx = max256(mx, om);
    sm = sat_add(sm, os);
  }
}

__device__ __forceinline__ void write_carried(AxisRecord* out, const U256& mx, const U256& sm) {
  AxisRecord r{};
  put_u256(r.max_magnitude, mx);
  put_u256(r.absolute_sum, sm);
  *out = r;
}

// Rows == true: one wave per row r of C, lanes over the columns; false: one
// wave per column, lanes over the rows. Each wave writes its axis's maximum
// and (saturating) sum of cell bounds.
template <bool Rows>
__global__ __launch_bounds__(256) void product_axes_kernel(ProductArgs p) {
  const int lane = threadIdx.x & 63;
  const int64_t waves = static_cast<int64_t>(gridDim.x) * (blockDim.x >> 6);
  const int64_t outer = Rows ? p.m : p.n, inner = Rows ? p.n : p.m;
  const AxisKind fixed_kind = Rows ? p.akind : p.bkind, var_kind = Rows ? p.bkind : p.akind;
  const AxisRecord* const fixed_recs = Rows ? p.arows : p.bcols;
  const AxisRecord* const var_recs = Rows ? p.bcols : p.arows;
  const U256 fixed_max = get_u256(Rows ? p.amax : p.bmax), var_max = get_u256(Rows ? p.bmax : p.amax);
  for (int64_t o = static_cast<int64_t>(blockIdx.x) * (blockDim.x >> 6) + (threadIdx.x >> 6); o < outer;
       o += waves) {
    const AxisTerms fixed = axis_terms(fixed_kind == AxisKind::Uniform ? nullptr : fixed_recs + o, fixed_kind,
                                       fixed_max, p.k);
    U256 mx = zero256(), sm = zero256();
    for (int64_t i = lane; i < inner; i += 64) {
      const AxisTerms var = axis_terms(var_kind == AxisKind::Uniform ? nullptr : var_recs + i, var_kind, var_max,
                                       p.k);
      const U256 cell = Rows ? cell_bound(fixed, var) : cell_bound(var, fixed);
      mx = max256(mx, cell);
      sm = sat_add(sm, cell);
    }
    wave_reduce(mx, sm);
    if (lane == 0) write_carried(Rows ? p.out_rows + o : p.out_cols + o, mx, sm);
  }
}

// C's bound: min(k maxA maxB, max over the row maxima); one block.
__global__ __launch_bounds__(256) void product_bound_kernel(ProductArgs p) {
  __shared__ U256 part[4];
  U256 mx = zero256();
  for (int64_t r = threadIdx.x; r < p.m; r += blockDim.x) mx = max256(mx, get_u256(p.out_rows[r].max_magnitude));
  for (int off = 32; off > 0; off >>= 1) {
    U256 o;
    for (int i = 0; i < 4; ++i) o.w[i] = __shfl_xor(mx.w[i], off);
    mx = max256(mx, o);
  }
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = mx;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < 4; ++w) mx = max256(mx, part[w]);
    const U256 outer = sat_mul(sat_mul64(p.k, get_u256(p.amax)), get_u256(p.bmax));
    put_u256(p.out_words, min256(outer, mx));
    put_u256(p.out_words + 4, zero256());
  }
}

// A result's lazy proof: A's row records, B's column records, maxA into
// words[0..3] and maxB into words[4..7].
__global__ __launch_bounds__(256) void proof_snapshot_kernel(const uint4* __restrict__ arows,
                                                             const uint4* __restrict__ bcols,
                                                             const u64* __restrict__ a_words,
                                                             const u64* __restrict__ b_words, int64_t m_chunks,
                                                             int64_t n_chunks, uint4* __restrict__ out_rows,
                                                             uint4* __restrict__ out_cols, u64* __restrict__ words) {
  const int64_t total = m_chunks + n_chunks;
  for (int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < total;
       i += static_cast<int64_t>(gridDim.x) * blockDim.x) {
    if (i < m_chunks) out_rows[i] = arows[i];
    else out_cols[i - m_chunks] = bcols[i - m_chunks];
  }
  if (blockIdx.x == 0 && threadIdx.x < 8) words[threadIdx.x] = threadIdx.x < 4 ? a_words[threadIdx.x] : b_words[threadIdx.x - 4];
}

unsigned blocks_for(int64_t items, int64_t per_block, int64_t cap) {
  int64_t b = (items + per_block - 1) / per_block;
  if (b < 1) b = 1;
  if (b > cap) b = cap;
  return static_cast<unsigned>(b);
}

}  // namespace

namespace {

hipError_t launch_tiled_axes(const uint64_t* src, int64_t rows, int64_t cols, int64_t ld, bool is_signed,
                             AxisRecord* out_rows, AxisRecord* out_cols, uint64_t* words, AxisPartial* partials,
                             hipStream_t stream) {
  const int64_t tiles_x = (cols + kTile - 1) / kTile, tiles_y = (rows + kTile - 1) / kTile;
  if (tiles_x > 0x7FFFFFFFll) return hipErrorInvalidValue;
  AxisPartial* const row_part = partials;
  AxisPartial* const col_part = partials + rows * tiles_x;
  // two tiles per block where there are enough: one loads while the other is summarized
  const int64_t gy = tiles_x * tiles_y >= 2048 ? (tiles_y + 1) / 2 : tiles_y;
  const dim3 grid(static_cast<unsigned>(tiles_x), static_cast<unsigned>(gy < kMaxGridY ? gy : kMaxGridY));
  const unsigned fin = blocks_for(rows + cols, 32, 4096);
  auto run = [&](auto sgn) {
    constexpr bool S = decltype(sgn)::value;
    hipLaunchKernelGGL((tiled_axes_pass<S, false>), grid, dim3(256), 0, stream, src, rows, cols, ld, row_part,
                       col_part, out_rows, out_cols, words);
    hipLaunchKernelGGL((tiled_axes_finish<S, false>), dim3(fin), dim3(256), 0, stream, row_part, col_part, rows,
                       cols, out_rows, out_cols, words);
    hipLaunchKernelGGL((tiled_axes_pass<S, true>), grid, dim3(256), 0, stream, src, rows, cols, ld, row_part,
                       col_part, out_rows, out_cols, words);
    hipLaunchKernelGGL((tiled_axes_finish<S, true>), dim3(fin), dim3(256), 0, stream, row_part, col_part, rows,
                       cols, out_rows, out_cols, words);
  };
  if (is_signed)
    run(std::true_type{});
  else
    run(std::false_type{});
  return hipGetLastError();
}

}  // namespace

hipError_t launch_native_axes(const void* src, int64_t rows, int64_t cols, int64_t ld, bool is_signed,
                              xa::AxisRecord* out_rows, xa::AxisRecord* out_cols, uint64_t* words,
                              ProofTicket* ticket, xa::AxisPartial* partials, hipStream_t stream) {
  if (!src || !out_rows || !out_cols || !words || !ticket || rows <= 0 || cols <= 0 || ld < cols)
    return hipErrorInvalidValue;
  const uint64_t* s = static_cast<const uint64_t*>(src);
  if (native_axes_tiled(rows, cols)) {
    if (!partials) return hipErrorInvalidValue;
    return launch_tiled_axes(s, rows, cols, ld, is_signed, out_rows, out_cols, words, partials, stream);
  }
  const unsigned rb = blocks_for(rows, kWaves, kMaxBlocks);
  // whole groups of 16 column blocks (see the kernel's numbering)
  const unsigned cb = blocks_for((cols + kColsPerBlock - 1) / kColsPerBlock, 16, kMaxBlocks / 16) * 16;
  // 32-bit lane offsets span a load's 128 rows
  const bool far = ld >= (int64_t{1} << 21);
  const bool vec = !far && (reinterpret_cast<uintptr_t>(src) & 15u) == 0 && ld % 2 == 0;
  auto run = [&](auto sgn, auto vc, auto fr) {
    hipLaunchKernelGGL((native_axes_kernel<decltype(sgn)::value, decltype(vc)::value, decltype(fr)::value>),
                       dim3(cb + rb), dim3(kThreads), 0, stream, s, rows, cols, ld, cb, rb, out_rows, out_cols, words,
                       ticket);
  };
  auto run_as = [&](auto sgn) {
    if (vec) run(sgn, std::true_type{}, std::false_type{});
    else if (!far) run(sgn, std::false_type{}, std::false_type{});
    else run(sgn, std::false_type{}, std::true_type{});
  };
  if (is_signed) run_as(std::true_type{});
  else run_as(std::false_type{});
  return hipGetLastError();
}

hipError_t launch_product_axes(const xa::AxisRecord* arows, uint32_t akind, const xa::AxisRecord* bcols,
                               uint32_t bkind, const uint64_t* a_words, const uint64_t* b_words, int64_t m,
                               int64_t n, uint64_t k, xa::AxisRecord* out_rows, xa::AxisRecord* out_cols,
                               uint64_t* out_words, hipStream_t stream) {
  if (akind > 2 || bkind > 2 || m <= 0 || n <= 0 || k == 0 || !out_rows || !out_cols || !out_words || !a_words ||
      !b_words || (akind != 2 && !arows) || (bkind != 2 && !bcols))
    return hipErrorInvalidValue;
  const ProductArgs p{arows, bcols, static_cast<AxisKind>(akind), static_cast<AxisKind>(bkind), a_words, b_words,
                      m, n, k, out_rows, out_cols, out_words};
  // four waves per block, one axis per wave
  hipLaunchKernelGGL(product_axes_kernel<true>, dim3(blocks_for(m, 4, 8192)), dim3(256), 0, stream, p);
  hipLaunchKernelGGL(product_axes_kernel<false>, dim3(blocks_for(n, 4, 8192)), dim3(256), 0, stream, p);
  hipLaunchKernelGGL(product_bound_kernel, dim3(1), dim3(256), 0, stream, p);
  return hipGetLastError();
}

hipError_t launch_proof_snapshot(const xa::AxisRecord* arows, const xa::AxisRecord* bcols, const uint64_t* a_words,
                                 const uint64_t* b_words, int64_t m, int64_t n, xa::AxisRecord* out_rows,
                                 xa::AxisRecord* out_cols, uint64_t* out_words, hipStream_t stream) {
  if (!a_words || !b_words || !out_words || m < 0 || n < 0 || (m && (!arows || !out_rows)) ||
      (n && (!bcols || !out_cols)))
    return hipErrorInvalidValue;
  constexpr int64_t kChunks = sizeof(xa::AxisRecord) / sizeof(uint4);
  hipLaunchKernelGGL(proof_snapshot_kernel, dim3(blocks_for((m + n) * kChunks, 256, 2048)), dim3(256), 0, stream,
                     reinterpret_cast<const uint4*>(arows), reinterpret_cast<const uint4*>(bcols), a_words, b_words,
                     m * kChunks, n * kChunks, reinterpret_cast<uint4*>(out_rows), reinterpret_cast<uint4*>(out_cols),
                     out_words);
  return hipGetLastError();
}

}  // namespace rns8x
