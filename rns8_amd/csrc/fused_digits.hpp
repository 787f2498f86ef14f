// Fused native-input GEMM for results at most 16 columns wide (GEMV and
// tall-skinny products): C's residue planes straight from int64 / uint64
// device operands (reference hip_direct_gemm_native_kernels.cuh:9-193 converts
// native operands inside its tile loads; its N <= 8 GEMV is
// hip_direct_gemm_tiled_kernels.cuh:298-432).
//
// A is read once and never converted. Its 8-byte elements are base-256 digits,
// and modulo m
//   sum_k A[r][k] B[k][c] = sum_k sum_b byte_b(A[r][k]) * W[k][b],
//   W[k][b] = centered(2^(8b) B[k][c] mod m),
// so the native bytes themselves, as they lie in memory, are the int8 MFMA's A
// operand over an inner dimension 8 times as long, and only the small operand
// is converted (into 8 digit weights per element, plane and column). The
// planes and columns of the result are the N dimension: 9 planes of a GEMV
// share one 16-column MFMA. The bytes are unsigned and the MFMA's are not: all
// but a signed element's top byte have their top bit flipped (one XOR per four
// bytes) and the 128 each of them then lacks is put back through the column
// sums 128 * sum W, which the waves form with a constant A operand.
//
// What bounds this kernel is the read of A: 8192 x 1 x 8192 at 9 planes takes
// 97 us for 537 MB (5.5 TB/s; a plain read of as much reaches 5.6-5.7), 8 us
// more with the weights and the finalize; reducing every element to every
// plane's residue in registers (fused_skinny.hip) took 147 us in all, and more
// with every plane. Non-temporal loads of A: 114 against 123 us,
// but only where rows start on cache lines: a line that two steps share was
// then fetched twice (4498 x 4 x 1043 at 9 planes 26.7 us, ordinary loads 22.2;
// 989 x 10 x 6774 55.5 and 48.1); 1024 instead
// of 512 workgroups: 106 against 114; two or four lines of a row per step: 111
// and 118 (more bytes per row in flight, fewer rows).
//
// Work split: a workgroup is four waves of 32 rows of one K slice. A and the
// weights go to LDS by DMA in steps of 16 elements (whole 128-byte lines of A;
// each wave its own rows), one to three steps ahead (stages_of); one barrier
// per step publishes the shared weights. Fragments:
//   * A (MFMA src1): lane l holds row l % 16, the 16 bytes (two elements) of
//     chunk 4h + l / 16 of the 128-byte line, h the half step; the lines are
//     XOR-swizzled by row like the plane GEMM's.
//   * weights (src0): lane l holds column l % 16 of the same two elements'
//     digits, stored in lane order, 1 KB per half step and 16 columns.
// Accumulators start at kGemmAccBias; slices of at most 4096 elements keep the
// sum and its 128 * sum W correction inside 2^30. Each slice stores its
// centered residues [slice][row][16 columns x groups] in the workspace; a
// finalize adds the slices and writes C's planes. Weights and residues take at
// most kMaxPart bytes each: larger K or m run in parts.
// (A header of fused_skinny.hip, not a source: what links the kernels' objects by
// name, as the CPU fuzzers' build does, needs no further object.)
#pragma once

#include <algorithm>
#include <type_traits>

#include "dma.hpp"
#include "int_ops.hpp"
#include "kernels.hpp"
#include "plane_consts.hpp"

namespace rns8x {
namespace digits {
namespace {

constexpr int kWaves = 4;
constexpr int kThreads = 64 * kWaves;
constexpr int kStepK = 16;                  // elements per step: one 128-byte line of a row
constexpr int kWaveRows = 32, kGroupRows = kWaves * kWaveRows;
// LDS ring depth: the deepest that lets two workgroups share a CU (80 KB each)
constexpr int stages_of(int groups) { return groups <= 2 ? 4 : groups <= 4 ? 3 : 2; }
constexpr uint32_t kStepBytes = 2048;       // weights of a step and 16 columns
constexpr uint32_t kMaxGroups = 6;          // 16-column groups
constexpr int64_t kTargetGroups = 1024;
constexpr int64_t kMinSliceK = 256;
constexpr int64_t kMaxSliceK = 4096;
constexpr int64_t kMaxK = int64_t{1} << 23;
constexpr uint64_t kMaxPart = uint64_t{64} << 20;

struct DigitsArgs {
  const uint64_t* a;  // native A, m x k at row stride lda (elements), from the launch's first row
  uint32_t lda, m, k;
  const int8_t* w;    // the launch's weights: [group][step][2][64][16], group stride w_stride
  uint32_t w_stride;
  int8_t* slots;      // residues [slice][m][slot_row]
  uint32_t slot_row;
  uint32_t columns, n;  // column q is column q % n of plane q / n
  uint32_t slice0, k_slice, row_groups;
  uint32_t whole_lines;  // every row starts on a 128-byte line: a step reads whole lines once
};

// Centered residue of the 64-bit value (hi:lo) mod mc.m (pack.hip's wide
// form; a signed value is read as x ^ 2^63, the bias folded into off_i64).
template <bool Signed>
__device__ __forceinline__ uint32_t residue64(uint32_t lo, uint32_t hi, const ModulusConsts& mc) {
  if (mc.m == 256u) return lo;
  const uint32_t off = (Signed ? mc.off_i64 : mc.off_u64) - mc.half;
  const uint32_t t = __builtin_amdgcn_udot4(lo, mc.pow_lo, off, false);
  const uint32_t s = __builtin_amdgcn_udot4(Signed ? hi ^ 0x80000000u : hi, mc.pow_hi, t, false);
  return centered_byte(s, mc.pq_shift, in_vgpr(mc.half << mc.pq_shift), mc.pq_recip, 256u - mc.m);
}

// The digit weights of B rows [k0, k0 + 16 steps): thread t writes the 16
// bytes of one lane's fragment, t = ((group * steps + step) * 2 + h) * 64 +
// lane: column q = 16 group + lane % 16, elements k0 + 16 step + 2 (4h + lane /
// 16) and + 1, eight digits each. Columns past planes * n and rows past k are
// zero.
template <bool Signed>
__global__ __launch_bounds__(256) void digit_weights_kernel(const uint64_t* b, int64_t ldb, uint32_t k, uint32_t n,
                                                            uint32_t columns, uint32_t k0, uint32_t steps,
                                                            uint32_t total, int8_t* w) {
  for (uint32_t t = blockIdx.x * blockDim.x + threadIdx.x; t < total; t += gridDim.x * blockDim.x) {
    const uint32_t lane = t & 63u, h = (t >> 6) & 1u, gs = t >> 7;
    const uint32_t group = gs / steps, step = gs - group * steps;
    const uint32_t q = 16u * group + (lane & 15u);
    const uint32_t ke = k0 + kStepK * step + 2u * (4u * h + (lane >> 4));
    v4i out = {0, 0, 0, 0};
    if (q < columns) {
      const uint32_t plane = q / n, c = q - plane * n;
      const ModulusConsts& mc = plane_mod(PlaneConsts{0}, plane);
#pragma unroll
      for (uint32_t e = 0; e < 2; ++e) {
        if (ke + e >= k) continue;
        const uint64_t x = b[static_cast<int64_t>(ke + e) * ldb + c];
        const int32_t centered = static_cast<int8_t>(
            residue64<Signed>(static_cast<uint32_t>(x), static_cast<uint32_t>(x >> 32), mc));
        const uint32_t r = static_cast<uint32_t>(centered < 0 ? centered + static_cast<int32_t>(mc.m) : centered);
#pragma unroll
        for (uint32_t d = 0; d < 8; ++d) {
          const uint32_t pow = ((d < 4 ? mc.pow_lo : mc.pow_hi) >> (8u * (d & 3u))) & 0xFFu;
          const uint32_t s = r * pow + mc.half;  // < 2^16 + 2^7
          const uint32_t byte = (s - __umulhi(s, mc.recip) * mc.m - mc.half) & 0xFFu;
          out[2 * e + d / 4] |= static_cast<int>(byte << (8u * (d & 3u)));
        }
      }
    }
    *reinterpret_cast<v4i*>(w + static_cast<uint64_t>(t) * 16u) = out;
  }
}

// The plane GEMM's A swizzle: conflict-free fragment reads of 16 rows.
__device__ __forceinline__ uint32_t swizzle_line(uint32_t row, uint32_t chunk) {
  return chunk ^ ((row ^ ((row >> 3) & 1u)) & 7u);
}

template <bool Signed, int G>
__global__ __launch_bounds__(kThreads, 2) void fused_digits_kernel(DigitsArgs a) {
  constexpr int kWBlocks = (2 * G + kWaves - 1) / kWaves;  // 1 KB weight blocks per wave and step
  constexpr uint32_t kWaveA = 4096u, kStageA = kWaves * kWaveA, kStageW = kWaves * kWBlocks * 1024u;
  constexpr int kStages = stages_of(G);
  constexpr uint32_t kRingA = kStages * kStageA;
  __shared__ __attribute__((aligned(16))) int8_t lds[kStages * (kStageA + kStageW)];
  static_assert(kWaves * G * 1024 <= static_cast<int>(sizeof(lds)), "the corrections fit the ring");
  const uint32_t lane = threadIdx.x & 63u;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint32_t part = blockIdx.x / a.row_groups;  // slice within the launch
  const uint32_t row0 = (blockIdx.x - part * a.row_groups) * kGroupRows + wave * kWaveRows;
  const uint32_t rows = row0 < a.m ? min(static_cast<uint32_t>(kWaveRows), a.m - row0) : 0u;
  const uint32_t slice = a.slice0 + part;
  const uint32_t kbeg = slice * a.k_slice;
  const uint32_t steps = (min(a.k, kbeg + a.k_slice) - kbeg + kStepK - 1) / kStepK;

  // ---- DMA ------------------------------------------------------------------
  // A: load i of a step fills rows 8i .. 8i + 7 of the wave's 32; the resource
  // starts at the step's first element and ends at the last logical element of
  // the wave's last valid row. Weights: block b of a step is half b % 2 of
  // group b / 2; a wave's blocks past 2 G - 1 read nothing.
  constexpr int kABlocks = 4;
  uint32_t a_voff[kABlocks], w_voff[kWBlocks];
#pragma unroll
  for (uint32_t i = 0; i < kABlocks; ++i) {
    const uint32_t row = 8u * i + (lane >> 3);
    a_voff[i] = row * a.lda * 8u + 16u * swizzle_line(row, lane & 7u);
  }
#pragma unroll
  for (uint32_t i = 0; i < kWBlocks; ++i) {
    const uint32_t b = wave * kWBlocks + i;
    w_voff[i] = b < 2u * G ? (b >> 1) * a.w_stride + (b & 1u) * 1024u + 16u * lane : 0x80000000u;
  }
  const int8_t* a_at = reinterpret_cast<const int8_t*>(a.a + static_cast<uint64_t>(row0) * a.lda + kbeg);
  const int8_t* w_at = a.w + static_cast<uint64_t>(part) * (a.k_slice / kStepK) * kStepBytes;
  int32_t a_left = rows ? static_cast<int32_t>(((rows - 1) * a.lda + (a.k - kbeg)) * 8u) : 0;
  const uint32_t lds_a = lds_address(lds) + wave * kWaveA;
  const uint32_t lds_w = lds_address(lds) + kRingA + wave * kWBlocks * 1024u;
  auto issue = [&](uint32_t s) {
    const bool live = s < steps;
    const uint32_t stage = s % kStages;
    const v4i ra = buffer_rsrc(a_at, live ? a_left : 0);
    const v4i rw = buffer_rsrc(w_at, live ? (G - 1) * static_cast<int64_t>(a.w_stride) + kStepBytes : 0);
#pragma unroll
    for (int i = 0; i < kABlocks; ++i) {
      if (a.whole_lines) dma16_stream(lds_a + stage * kStageA + 1024u * i, a_voff[i], ra);
      else dma16(lds_a + stage * kStageA + 1024u * i, a_voff[i], ra);
    }
#pragma unroll
    for (int i = 0; i < kWBlocks; ++i) dma16(lds_w + stage * kStageW + 1024u * i, w_voff[i], rw);
    a_at += 8 * kStepK;
    w_at += kStepBytes;
    a_left = max(a_left - 8 * kStepK, 0);
  };

  // ---- loop -----------------------------------------------------------------
  v4i acc[2][G], corr[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    constexpr int kBias = static_cast<int>(kGemmAccBias);
    acc[0][g] = acc[1][g] = v4i{kBias, kBias, kBias, kBias};
    corr[g] = v4i{0, 0, 0, 0};
  }
  constexpr int kTop = static_cast<int>(Signed ? 0x00808080u : 0x80808080u);
  constexpr int kAll = static_cast<int>(0x80808080u);
  const v4i flip = {kAll, kTop, kAll, kTop};  // also the constant -128 operand of the corrections
  const uint32_t frag = (lane & 15u) * 128u;
  constexpr int kPerStep = kABlocks + kWBlocks;
#pragma unroll
  for (uint32_t s = 0; s < kStages - 1u; ++s) issue(s);
  for (uint32_t s = 0; s < steps; ++s) {
    __builtin_amdgcn_s_waitcnt(wait_vm((kStages - 2) * kPerStep));  // this wave's DMAs of step s landed
    __syncthreads();  // everybody's did, and everybody has read step s - 1
    issue(s + kStages - 1u);
    const uint32_t stage = s % kStages;
    const int8_t* const sa = lds + stage * kStageA + wave * kWaveA + frag;
    const int8_t* const sw = lds + kRingA + stage * kStageW + 16u * lane;
#pragma unroll
    for (uint32_t h = 0; h < 2; ++h) {
      const uint32_t chunk = 16u * swizzle_line(lane & 15u, 4u * h + (lane >> 4));
      const v4i a0 = *reinterpret_cast<const v4i*>(sa + chunk) ^ flip;
      const v4i a1 = *reinterpret_cast<const v4i*>(sa + 2048 + chunk) ^ flip;
      v4i w[G];
#pragma unroll
      for (int g = 0; g < G; ++g) w[g] = *reinterpret_cast<const v4i*>(sw + 2048 * g + 1024 * h);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        acc[0][g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[g], a0, acc[0][g], 0, 0, 0);
        acc[1][g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[g], a1, acc[1][g], 0, 0, 0);
      }
      // every fourth half step's column sums are this wave's
      if (wave == ((2u * s + h) & 3u)) {
#pragma unroll
        for (int g = 0; g < G; ++g) corr[g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[g], flip, corr[g], 0, 0, 0);
      }
    }
  }

  // ---- epilogue ---------------------------------------------------------------
  // corr holds -128 sum W over the wave's half steps, the same in every row;
  // acc - (the waves' corr) is bias + the slice's sum. Lane l holds columns
  // 16 g + 4 (l / 16) + e of rows l % 16 and 16 + l % 16.
  __builtin_amdgcn_s_waitcnt(wait_vm(0));  // no DMA outlives the ring
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g) *reinterpret_cast<v4i*>(lds + (wave * G + g) * 1024u + 16u * lane) = corr[g];
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g) {
    v4i sum = {0, 0, 0, 0};
#pragma unroll
    for (uint32_t v = 0; v < kWaves; ++v) sum += *reinterpret_cast<const v4i*>(lds + (v * G + g) * 1024u + 16u * lane);
    const uint32_t q0 = 16u * g + 4u * (lane >> 4);
    uint32_t r[2][4];
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) {
      const uint32_t q = q0 + e;
      // (columns past the result's: any plane)
      const ModulusConsts mc = plane_mod(PlaneConsts{0}, q < a.columns ? q / a.n : 0u);
#pragma unroll
      for (int rb = 0; rb < 2; ++rb) {
        const uint32_t u = static_cast<uint32_t>(acc[rb][g][e] - sum[e]);
        const uint32_t s = __builtin_amdgcn_udot4(u, mc.pow_lo, mc.off_acc, false);
        r[rb][e] = s - __umulhi(s, mc.recip) * mc.m - mc.half;
      }
    }
#pragma unroll
    for (uint32_t rb = 0; rb < 2; ++rb) {
      const uint32_t row = row0 + 16u * rb + (lane & 15u);
      if (row < a.m)
        *reinterpret_cast<uint32_t*>(a.slots + (static_cast<uint64_t>(slice) * a.m + row) * a.slot_row + q0) =
            pack_low_bytes(r[rb][0], r[rb][1], r[rb][2], r[rb][3]);
    }
  }
}

// Adds the slices' residues of one plane and row (thread t: row t / planes,
// plane t % planes) and writes the plane's 16-byte row, zero past column n.
__global__ __launch_bounds__(256) void digits_finalize_kernel(const int8_t* slots, uint32_t slot_row, uint32_t m,
                                                              uint32_t n, uint32_t planes, uint32_t slices,
                                                              uint64_t total, int8_t* c, int64_t pitch_c) {
  const uint64_t t = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t >= total) return;
  const uint64_t row = t / planes;
  const uint32_t plane = static_cast<uint32_t>(t - row * planes);
  const ModulusConsts& mc = plane_mod(PlaneConsts{0}, plane);
  const int8_t* const src = slots + row * slot_row + plane * n;
  uint32_t out[4] = {0, 0, 0, 0};
#pragma unroll
  for (uint32_t col = 0; col < 16; ++col) {
    if (col >= n) break;
    int32_t sum = 0;
#pragma unroll 8
    for (uint32_t s = 0; s < slices; ++s) sum += src[static_cast<uint64_t>(s) * m * slot_row + col];
    const uint32_t v = __builtin_amdgcn_udot4(static_cast<uint32_t>(sum) ^ 0x80000000u, mc.pow_lo, mc.off_i32, false);
    out[col / 4] |= ((v - __umulhi(v, mc.recip) * mc.m - mc.half) & 0xFFu) << (8u * (col & 3u));
  }
  *reinterpret_cast<uint4*>(c + plane * pitch_c + static_cast<int64_t>(row) * 16) =
      uint4{out[0], out[1], out[2], out[3]};
}

// 16-column groups of the result.
inline uint32_t groups_of(uint32_t nplanes, int64_t n) { return (nplanes * static_cast<uint32_t>(n) + 15u) / 16u; }

struct Parts {
  int64_t slices, k_slice;
  uint32_t groups;
  int64_t part_slices;  // slices whose weights the workspace holds at once
  int64_t part_rows;    // rows whose residues it holds at once
  uint64_t w_bytes, slot_bytes;
};
inline Parts split(int64_t m, int64_t n, int64_t k, uint32_t nplanes) {
  Parts p{};
  p.groups = groups_of(nplanes, n);
  const int64_t row_groups = (m + kGroupRows - 1) / kGroupRows;
  // toward kTargetGroups workgroups, slices of at least kMinSliceK elements
  p.slices = std::min((kTargetGroups + row_groups - 1) / row_groups, (k + kMinSliceK - 1) / kMinSliceK);
  p.slices = std::max(std::max<int64_t>(p.slices, 1), (k + kMaxSliceK - 1) / kMaxSliceK);
  p.k_slice = ((k + p.slices - 1) / p.slices + kStepK - 1) / kStepK * kStepK;
  p.slices = (k + p.k_slice - 1) / p.k_slice;
  const uint64_t slice_w = static_cast<uint64_t>(p.k_slice) / kStepK * kStepBytes * p.groups;
  p.part_slices = std::min<int64_t>(p.slices, std::max<int64_t>(1, static_cast<int64_t>(kMaxPart / slice_w)));
  p.w_bytes = slice_w * static_cast<uint64_t>(p.part_slices);
  const uint64_t row_bytes = static_cast<uint64_t>(p.slices) * 16u * p.groups;
  p.part_rows = std::min<int64_t>(
      row_groups * kGroupRows, std::max<int64_t>(1, static_cast<int64_t>(kMaxPart / row_bytes / kGroupRows)) * kGroupRows);
  p.slot_bytes = row_bytes * static_cast<uint64_t>(std::min(p.part_rows, m));
  return p;
}

}  // namespace

inline bool fused_digits_shape(int64_t m, int64_t n, int64_t k, uint32_t nplanes, FusedShape& out) {
  if (n <= 0 || n > 16 || m <= 0 || k <= 0 || nplanes == 0 || nplanes > kMaxPrefix) return false;
  if (m >= (int64_t{1} << 31) || k > kMaxK) return false;
  // Where this form is the faster one. Its cost grows with the 16-column groups
  // of planes x columns, the residue form's (fused_skinny.hip) with the planes.
  // Whole calls, m x n x k, residue form / this form in us:
  //   planes >= 2 groups + 1: 8192 x 1 x 8192, 9 planes 147 / 106, n = 7 148 /
  //     134; 2000 x 7 x 1000, 9 planes 50 / 22; 128 x 7 x 256, 9 planes 18.8 /
  //     17.3; 200 x 4 x 20000, 20 planes 135 / 50. Up to 4 planes this form's
  //     three launches cost more than they save (8000 x 5 x 300, 3 planes 12.8
  //     / 15.3); at 5 and 6 also below 2^18 elements of A (128 x 5 x 256,
  //     6 planes 13.9 / 14.3; but 512 x 3 x 512, 5 planes 19.1 / 13.3).
  //     Above 2^23 elements five planes' arithmetic hides behind the residue
  //     form's loads (5748 x 5 x 6620, 5 planes 79 / 89).
  //   3 groups <= 2 planes: while A is small enough to leave the residue form
  //     idle CUs and long enough to amortize the launches (2000 x 9 x 1000, 9
  //     planes 50 / 29; 2000 x 8 x 1000, 5 planes 33 / 21; but 8000 x 8 x 300,
  //     5 planes 16.6 / 17.7, 8192 x 8 x 8192, 9 planes 148 / 151, 512 x 8 x
  //     16000, 9 planes 57 / 61).
  //     Deep and large ones of five and six planes lose (1160 x 10 x 6968, 6
  //     planes 44.4 / 50.8; but 120 x 8 x 7040 45 / 28, 5041 x 7 x 1192 34 / 21).
  //   The smallest products: the residue form of at most nine planes needs no
  //     more than two launches up to 128 elements of K, this one three, so a pass
  //     of product and export is bound by the launches (1000 x 1 x 64, 7 planes
  //     14.3 / 16.0; 16 x 1 x 8, 9 planes 14.7 / 15.4; 4096 x 4 x 128, 9 planes
  //     16.4 / 16.8; but 4096 x 2 x 100, 9 planes 16.2 / 15.8, 30000 x 1 x 64, 7
  //     planes 17.5 / 15.6, 128 x 3 x 200, 8 planes 19.3 / 16.4).
  // The weights are 16 groups / m of A's bytes: with few rows per group
  // writing them costs more than it saves (9 planes: 32 x 2 x 100000 61 / 64,
  // 16 x 4 x 100000 60 / 98; 64 x 2 x 8000 53 / 17, 16 x 1 x 100000 60 / 43).
  const int64_t groups = groups_of(nplanes, n), work = m * k;
  if (m < 16 * (2 * groups - 1) || groups > kMaxGroups || nplanes < 5) return false;
  const bool few = nplanes >= 2 * groups + 1 &&
                   (nplanes >= 7 || (work >= (int64_t{1} << 18) && work <= (int64_t{1} << 23)));
  const bool mid = 3 * groups <= 2 * nplanes && k >= 512 && work >= (int64_t{1} << 18) && work <= (int64_t{1} << 23) &&
                   k <= (nplanes < 7 && work > (int64_t{1} << 22) ? 4096 : 8192);
  if (!few && !mid) return false;
  if (k <= 128 && m <= 16384 && (nplanes <= 8 || (nplanes == 9 && (groups >= 3 || k <= 32)))) return false;
  // Deeper products: the weights take 0.17 us per group and 1000 elements of K,
  // whatever m, so the residue form is the faster one of few rows (128 x 7 x
  // 200000, 9 planes 114 / 293; 128 x 4 x 65536, 9 planes 66 / 70; 800 x 7 x 32768,
  // 9 planes 87 / 104; 16 x 1 x 560000, 7 planes 109 / 134) and this one of many
  // (1200 x 4 x 65536, 9 planes 226 / 166; 512 x 2 x 100000, 9 planes 164 / 123;
  // 200 x 4 x 65536, 20 planes 145 / 90). Both sides' times, in ns: this form's
  // start, weights and read of A; the residue form's arithmetic over whole
  // workgroups of 64 rows, at least its latency, per launch of up to 18 planes.
  // Below three planes per group the weights count 15% more. Of 506 products
  // from 16384 to 600000 deep, 9 run in this form and would be 1 to 10% faster in
  // the other, 20 run in the other and would be 3 to 30% faster in this one.
  if (k > 16384) {
    if (nplanes < 7 && groups > 1) return false;
    const int64_t launches = nplanes <= 18 ? 1 : 2, planes = (nplanes + launches - 1) / launches;
    const double kd = static_cast<double>(k), md = static_cast<double>(m);
    const double weights = 12000.0 + 0.17 * static_cast<double>(groups) * kd + md * kd / 690.0;
    const double rows = static_cast<double>((m + 63) / 64 * 64);
    const double residues = static_cast<double>(launches) *
                            std::max(rows * kd * static_cast<double>(planes) / 3300.0, 10000.0 + 4200.0 * static_cast<double>(planes));
    if ((nplanes < 3 * groups ? 1.15 : 1.0) * weights >= residues) return false;
  }
  const Parts p = split(m, n, k, nplanes);
  out = FusedShape{};
  out.slices = static_cast<uint32_t>(p.slices);
  out.k_slice = p.k_slice;
  out.ws_bytes = p.w_bytes + p.slot_bytes;
  out.skinny = 2;
  return true;
}

inline hipError_t launch_fused_digits(const FusedArgs& f, hipStream_t stream) {
  const FusedShape& sh = f.shape;
  if (sh.skinny != 2 || f.ldc != 16 || f.n > 16 || f.k > kMaxK || f.lda >= (int64_t{1} << 21)) return hipErrorInvalidValue;
  const Parts p = split(f.m, f.n, f.k, f.nplanes);
  if (p.slices != sh.slices || p.k_slice != sh.k_slice || p.w_bytes + p.slot_bytes != sh.ws_bytes)
    return hipErrorInvalidValue;
  const bool sgn = f.kind == NativeKind::I64;
  int8_t* const slots = f.ws + p.w_bytes;
  for (int64_t r0 = 0; r0 < f.m; r0 += p.part_rows) {
    const uint32_t rows = static_cast<uint32_t>(std::min(p.part_rows, f.m - r0));
    for (int64_t s0 = 0; s0 < p.slices; s0 += p.part_slices) {
      const uint32_t parts = static_cast<uint32_t>(std::min(p.part_slices, p.slices - s0));
      const uint32_t steps = parts * static_cast<uint32_t>(p.k_slice / kStepK);
      const uint32_t runs = p.groups * steps * 128u;
      // the weights of these slices, unless an earlier part of the rows left them
      if (r0 == 0 || p.part_slices < p.slices) {
        const dim3 grid(std::min<uint32_t>((runs + 255u) / 256u, 8192u));
        auto weights = [&](auto s) {
          hipLaunchKernelGGL(digit_weights_kernel<decltype(s)::value>, grid, dim3(256), 0, stream,
                             static_cast<const uint64_t*>(f.b), f.ldb, static_cast<uint32_t>(f.k),
                             static_cast<uint32_t>(f.n), f.nplanes * static_cast<uint32_t>(f.n),
                             static_cast<uint32_t>(s0 * p.k_slice), steps, runs, f.ws);
        };
        if (sgn) weights(std::true_type{});
        else weights(std::false_type{});
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
      }
      DigitsArgs a{};
      a.a = static_cast<const uint64_t*>(f.a) + r0 * f.lda;
      a.lda = static_cast<uint32_t>(f.lda);
      a.m = rows;
      a.k = static_cast<uint32_t>(f.k);
      a.w_stride = steps * kStepBytes;
      a.slot_row = 16u * p.groups;
      a.columns = f.nplanes * static_cast<uint32_t>(f.n);
      a.n = static_cast<uint32_t>(f.n);
      a.slice0 = static_cast<uint32_t>(s0);
      a.k_slice = static_cast<uint32_t>(p.k_slice);
      a.row_groups = (rows + kGroupRows - 1) / kGroupRows;
      a.w = f.ws;
      a.whole_lines = (reinterpret_cast<uintptr_t>(f.a) % 128u == 0 && f.lda % kStepK == 0) ? 1u : 0u;
      a.slots = slots;
      auto run = [&](auto sg, auto g) {
        hipLaunchKernelGGL((fused_digits_kernel<decltype(sg)::value, decltype(g)::value>),
                           dim3(a.row_groups * parts), dim3(kThreads), 0, stream, a);
      };
      auto pick = [&](auto sg) {
        switch (p.groups) {
          case 1: return run(sg, std::integral_constant<int, 1>{});
          case 2: return run(sg, std::integral_constant<int, 2>{});
          case 3: return run(sg, std::integral_constant<int, 3>{});
          case 4: return run(sg, std::integral_constant<int, 4>{});
          case 5: return run(sg, std::integral_constant<int, 5>{});
          default: return run(sg, std::integral_constant<int, 6>{});
        }
      };
      if (sgn) pick(std::true_type{});
      else pick(std::false_type{});
      const hipError_t e = hipGetLastError();
      if (e != hipSuccess) return e;
    }
    const uint64_t total = static_cast<uint64_t>(rows) * f.nplanes;
    hipLaunchKernelGGL(digits_finalize_kernel, dim3(static_cast<unsigned>((total + 255) / 256)), dim3(256), 0, stream,
                       slots, 16u * p.groups, rows, static_cast<uint32_t>(f.n), f.nplanes,
                       static_cast<uint32_t>(p.slices), total, f.c + r0 * 16, f.pitch_c);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace digits
}  // namespace rns8x
