// Exact-wide magnitude proofs on the device (reference
// src/core/exact_range.hpp:34-157, api_gemm.cpp:870-874):
//
// * native_axes: the per-row and per-column summaries of a 64-bit operand at
//   pack time, one launch. Row blocks give a wave to each row, column blocks
//   take 8 columns whole, so every axis's extremes, sums and centre are known
//   where its values were read: the values stay in registers (up to 2048 of a
//   row, 1024 of a column; longer axes read them again) for the deviation sums
//   around that centre, and nothing goes through partial summaries. The last
//   row block to finish writes the operand's max |x|.
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

// 96-bit sum of 64-bit values.
struct Sum96 {
  u64 lo = 0;
  uint32_t hi = 0;
  __device__ __forceinline__ void add(u64 x, uint32_t x_hi = 0) {
    lo += x;
    hi += x_hi + (lo < x ? 1u : 0u);
  }
  __device__ __forceinline__ u128 value() const { return (static_cast<u128>(hi) << 64) | lo; }
};

// One lane's running summary over biased values u (bias(): their unsigned
// order is the order of x; at most 2^32 of them). The absolute sum comes from
// the sum of the positive parts: sum |x| = 2 sum max(x, 0) - sum x.
template <bool Signed>
struct Extremes {
  u64 hi = 0, lo = ~u64{0};
  Sum96 sum, pos;
  __device__ __forceinline__ void add(u64 u) {
    hi = u > hi ? u : hi;
    lo = u < lo ? u : lo;
    sum.add(u);
    if constexpr (Signed) pos.add(static_cast<int64_t>(u) < 0 ? u & ~(u64{1} << 63) : 0);  // x = u - 2^63
  }
  // merges the lanes whose index differs in bits kFrom .. 32
  template <int kFrom>
  __device__ __forceinline__ void merge() {
#pragma unroll
    for (int m = kFrom; m < 64; m <<= 1) {
      const u64 h = __shfl_xor(hi, m), l = __shfl_xor(lo, m);
      hi = h > hi ? h : hi;
      lo = l < lo ? l : lo;
      const u64 s = __shfl_xor(sum.lo, m);
      sum.add(s, __shfl_xor(sum.hi, m));
      if constexpr (Signed) {
        const u64 q = __shfl_xor(pos.lo, m);
        pos.add(q, __shfl_xor(pos.hi, m));
      }
    }
  }
  // of `count` values in all (this lane's are a part of them)
  __device__ __forceinline__ AxisPartial partial(u64 count) const {
    const u128 s = sum.value();
    return AxisPartial{hi, ~lo, s, Signed ? 2 * pos.value() - (s - (static_cast<u128>(count) << 63)) : s};
  }
};
// The sum of |x - c| over `count` values from sum max(x - c, 0) and the sum of
// the biased values: 2 sum max(u - cu, 0) - (sum u - count cu).
__device__ __forceinline__ u128 deviation_total(const Sum96& above, u128 sum, u64 count, u64 cu) {
  return 2 * above.value() - (sum - static_cast<u128>(count) * cu);
}
__device__ __forceinline__ void add_above(Sum96& above, u64 u, u64 cu) { above.add(u > cu ? u - cu : 0); }
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
// Only operands of few columns and more rows than a column block holds read
// worse (5000 x 300: 34 against 29 us).
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
      acc.template merge<1>();
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
      acc[e].template merge<4>();
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

hipError_t launch_native_axes(const void* src, int64_t rows, int64_t cols, int64_t ld, bool is_signed,
                              xa::AxisRecord* out_rows, xa::AxisRecord* out_cols, uint64_t* words,
                              ProofTicket* ticket, hipStream_t stream) {
  if (!src || !out_rows || !out_cols || !words || !ticket || rows <= 0 || cols <= 0 || ld < cols)
    return hipErrorInvalidValue;
  const uint64_t* s = static_cast<const uint64_t*>(src);
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
