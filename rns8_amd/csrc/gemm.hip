// Plane-batched int8 MFMA GEMM for gfx950 (CDNA4).
//
// One launch computes C_p = center(A_p x B_p mod m_p) for every residue plane
// p (reference semantics: src/cpu/cpu_reference.cpp:156-206, the per-modulus
// ring GEMM with int32 accumulation reduced at least every 65536 K).
//
// Work decomposition
//   * unit = one output tile of one plane (and one K slice when split-K is
//     on). A persistent grid of workgroups (one per resident slot, a
//     multiple of 8) walks the unit list, each XCD a contiguous share, so the
//     DMA stream runs on across unit boundaries.
//   * workgroup = 4 wave64s (2 for 64x64 tiles) in a 2 x 2 (2 x 1) grid over
//     the tile. Five tile configurations (256x256, 256x128, 128x256, 128x128,
//     64x64); choose_tile takes the one predicted fastest.
//   * K is consumed in steps of 64. Both operands go global -> LDS by
//     buffer-load DMA (no VGPR staging). A is staged in chunks of two steps
//     (BM x 128, K-contiguous rows: whole cache lines; 64-byte rows asked the
//     L2 for every line twice, and the full lines took 2.4% off 4096^3 at
//     prefix 9), three chunks deep; B in steps (64 x BN, N-contiguous rows,
//     the layout it has in HBM), four deep. The DMA four steps ahead is in
//     flight while a step computes, also across the epilogue into the next
//     unit; one barrier per step.
//   * A fragments are ds_read_b128 of 16 K-contiguous bytes; B fragments are
//     gathered K-contiguous from the N-contiguous stage by ds_read_b64_tr_b8
//     (LDS transpose read), so no transpose runs on the VALU. A step's
//     fragments are read during the step before.
//   * Stage rows are XOR-swizzled in 16-byte chunks (swizzle applied on the
//     global-address side of the DMA) so every fragment read is free of bank
//     conflicts in a model of the LDS that serves 8 or 16 lanes at a time. (The
//     counters see conflicts in a third of the LDS' active cycles at 4096^3,
//     where its instructions are held up for 6% of the waves' cycles.)
//   * MFMA: v_mfma_i32_16x16x64_i8 with the B^T fragment as src0 and the A
//     fragment as src1, so each lane ends with 4 consecutive output columns
//     of one row. What bounds the large products is the power limit: with
//     random residue bytes the chip sustains 4.08-4.11 POP/s of back-to-back
//     16x16x64 MFMAs at 2.0 GHz, against 3.38-3.43 POP/s of 32x32x32 ones
//     (whose accumulator traffic per product is twice as large); with zero
//     bytes both reach 4.9. At 4096^3, 9 planes, 32x32x32 tiles took 518 us
//     (2.39 POP/s), this kernel 452 us (2.73) on the same box, at equal cycles
//     (0.90 -> 0.86 M) and a 15% higher clock. Of its time, copies without
//     the operand DMA took 358 of 460 us, without the epilogue 415.
//   * Exactness: |a*b| <= 2^14, so <= 65536 products plus a carried residue
//     fit int32. One launch covers at most 65536 K; the host issues longer K
//     as consecutive launches whose epilogues add the residue already in C.
//   * Epilogue: accumulators start at kGemmAccBias (an MFMA inline constant:
//     no accumulator writes), so each holds the biased sum the reduction
//     reads; reduction is a byte dot product plus a 24-bit reciprocal quotient
//     (full-rate VALU only); 4 residues are packed per dword, and four blocks'
//     dwords are transposed across lane groups by half-wave and row swaps
//     into 16-byte stores. Staging them through LDS instead took 13.2 k
//     cycles per 256x256 unit against 8.5 k.
//   * Split-K (few output tiles): one launch covers the
//     whole K; each slice (at most 65536 K) reduces its tile like an
//     unsplit unit and stores the centered residues to its own slot of an
//     int8 workspace; residue_finalize adds the slots and writes C
//     (deterministic, no atomics, a quarter of the bytes int32 partials
//     would move).
//   * Results at most 16 columns wide run in skinny.hip instead.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <mutex>
#include <type_traits>

#include "dma.hpp"
#include "int_ops.hpp"
#include "kernels.hpp"
#include "plane_consts.hpp"

namespace rns8x {
namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v2i __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) v2i lds_v2i;

__device__ __forceinline__ lds_v2i* as_lds_v2i(const int8_t* p) {
  return (lds_v2i*)(const_cast<int8_t*>(p));  // generic -> LDS address space
}

// Accumulator start value (tables.hpp): the MFMAs then produce u = bias + sum,
// the non-negative form the reduction reads (|sum| <= 2^30 + 128).
constexpr int kAccBias = static_cast<int>(kGemmAccBias);

// Tile configuration: kWaves waves (2 x WN) each own TM x TN blocks of 16 x 16
// outputs, so a workgroup tile is (32 TM) x (16 TN WN). K advances in steps of
// 64; A is staged in chunks of two steps.
template <int TM_, int TN_, int WN_>
struct Cfg {
  static constexpr int TM = TM_, TN = TN_, WN = WN_;
  static constexpr int kWaves = 2 * WN, kThreads = 64 * kWaves;
  static constexpr int BM = 32 * TM, BN = 16 * TN * WN, BK = 64;
  static constexpr int kBufA = BM * 2 * BK;           // A chunk: BM rows x 128 bytes
  static constexpr int kBufB = BK * BN;               // B stage: 64 k-rows x BN bytes
  static constexpr int kSlotsA = 3, kStagesB = 4;
  static constexpr int kLds = kSlotsA * kBufA + kStagesB * kBufB;
  static constexpr int kDmaA = kBufA / 2048 / kWaves; // 1 KB DMA blocks per wave and step
  static constexpr int kDmaB = kBufB / 1024 / kWaves;
  static constexpr int kGroupM = 1024 / BM;           // tile rows per L2 reuse group
  static constexpr int kChunksB = BN / 16;            // 16-byte chunks per B stage row
  static constexpr int kRowsPerBlockB = 1024 / BN;    // k rows per 1 KB B block
  static_assert(kDmaA >= 1 && kDmaA <= 4 && kDmaB >= 1 && kDmaB <= 4, "DMA blocks");
  static_assert(1024 % BN == 0 && TM % 2 == 0 && TN % 4 == 0, "tile config");
  static_assert(kLds <= 160 * 1024, "LDS per workgroup");
};

// A chunk: row-major BM x 128 bytes, whole cache lines of A. The 16-byte chunk
// index is XORed with f(row) so the ds_read_b128 fragment loads (16
// consecutive rows, one chunk per 16 lanes) are bank-conflict free for both
// 32-bank/8-lane servicing (8 consecutive rows get distinct f) and
// 64-bank/16-lane servicing (the 8 even and the 8 odd of 16 rows each do).
__device__ __forceinline__ int swizzle_a(int row, int chunk) { return chunk ^ ((row ^ ((row >> 3) & 1)) & 7); }

// B stage: row-major 64 (k) x BN bytes, N-contiguous as in global memory. A
// 16-lane transpose read touches 8 consecutive k rows of one chunk; the chunk
// index is XORed with f(k) so those rows land in distinct bank quads, and bit
// 4 of k moves the next 16 lanes' rows (k + 16, the same chunk) onto the bank
// quads the first leave free: f = 2x mod 16 + x / 4 for 16-chunk rows, f = x
// for 8-chunk ones (x = k mod 8), either XORed with that bit.
template <int BN>
__device__ __forceinline__ int swizzle_b(int k, int chunk) {
  const int x = k & 7, b4 = (k >> 4) & 1;
  if constexpr (BN == 256)
    return chunk ^ ((((2 * x) & 15) | (x >> 2)) ^ b4);
  else if constexpr (BN == 128)
    return chunk ^ (x ^ b4);
  else
    return chunk ^ (((x >> 1) ^ b4) & 3);
}

// Scheduling slots of a half-step region: kPer MFMAs, then one of the region's
// kReads LDS fragment reads, kReads times.
template <int kId, int kPer, int kReads>
__device__ __forceinline__ void sched_slots() {
  if constexpr (kReads > 0) {
    __builtin_amdgcn_sched_group_barrier(0x008, kPer, kId);  // MFMA
    __builtin_amdgcn_sched_group_barrier(0x100, 1, kId);     // DS read
    sched_slots<kId, kPer, kReads - 1>();
  }
}

// Work list of one launch: units (K slice, plane, output tile) are numbered
// slice-major, then plane, then tile; tiles run in groups of kGroupM tile
// rows. The divisors carry host-computed reciprocals (make_div_u31).
struct UnitMap {
  uint32_t units;
  uint32_t tiles_m;
  DivU31 tiles;   // tiles per plane
  DivU31 planes;  // planes
  DivU31 group;   // kGroupM * tiles_n: tiles per group of tile rows
  DivU31 rows;    // kGroupM: tile rows of a full group
  DivU31 tail;    // tile rows of the last group (tiles_m - its first row)
  uint32_t k_begin, k_stop, k_slice;
  uint32_t pairs;  // K chunks (two steps) every unit runs; past the slice's K they read zeros
  // listed launches: two words per unit, (plane << 24 | tile row) and
  // (quadrant mask << 24 | tile column), in place of the arithmetic order
  const uint32_t* list;
  // grouped launches: units are numbered task-major, task_units per task
  DivU31 task_units;
};

// Grouped launches carry their tasks' base pointers by value (kernel
// arguments are read through the scalar cache); other launches an empty
// struct.
struct TaskTable {
  TaskPtrs t[kMaxGroupTasks];
};
struct NoTaskTable {};
template <bool kGrouped>
using GroupArg = std::conditional_t<kGrouped, TaskTable, NoTaskTable>;

// floor(n / d) for n < 2^31 (make_div_u31).
__device__ __forceinline__ uint32_t div_u31(uint32_t n, DivU31 v) { return __umulhi(n << 1, v.mul) >> v.shift; }

template <typename C, int kMinBlocks, bool kListed = false, bool kGrouped = false>
__global__ __launch_bounds__(C::kThreads, kMinBlocks) void plane_gemm_kernel(GemmArgs args, PlaneConsts pc, UnitMap map,
                                                                           uint32_t accumulate,
                                                                           GroupArg<kGrouped> tasks) {
  constexpr int TM = C::TM, TN = C::TN, BM = C::BM, BN = C::BN, BK = C::BK;
  __shared__ __attribute__((aligned(16))) int8_t lds[C::kLds];

  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wave_m = wave / C::WN;
  const int wave_n = wave % C::WN;

  // ---- persistent work list ----------------------------------------------------
  // A unit is one (K slice, plane, output tile). The grid holds a few
  // workgroups per CU and each walks its units in order, so the DMA stream
  // runs on across unit boundaries: the next unit's first K tiles land while
  // the current unit's epilogue runs. Workgroups are dispatched round-robin
  // over the 8 XCDs; with a grid that is a multiple of 8, XCD x owns the
  // contiguous unit range [x*units/8, (x+1)*units/8), walked by its
  // workgroups in lock step, so concurrently running tiles are neighbours and
  // share A and B panels in that XCD's L2 (tiles are ordered within a plane
  // in groups of kGroupM tile rows).
  const uint32_t grid = gridDim.x;
  uint32_t u_first, u_step, u_end;
  if ((grid & 7u) == 0u) {
    const uint32_t xcd = blockIdx.x & 7u;
    u_first = static_cast<uint32_t>((static_cast<uint64_t>(xcd) * map.units) / 8) + (blockIdx.x >> 3);
    u_end = static_cast<uint32_t>((static_cast<uint64_t>(xcd + 1) * map.units) / 8);
    u_step = grid >> 3;
  } else {
    u_first = blockIdx.x;
    u_end = map.units;
    u_step = grid;
  }
  u_first = __builtin_amdgcn_readfirstlane(u_first);
  u_end = __builtin_amdgcn_readfirstlane(u_end);
  if (u_first >= u_end) return;  // (before any unit is decoded: a list ends with its last unit)

  // Units are decoded on the scalar unit (every value here is uniform) with
  // the host's reciprocals.
  struct Unit {
    uint32_t task, plane, slice, m0, n0, kbeg, kend, quad;
  };
  // Listed units come from a per-tile schedule: a BM x BN tile of one plane
  // whose four quadrants (2 x 2) are stored only where the mask has their bit
  // (2 * row half + column half); quadrants outside the tiles that select this
  // plane keep their contents.
  auto decode = [&](uint32_t u) {
    Unit U;
    U.task = 0;
    if constexpr (kGrouped) {
      U.task = div_u31(u, map.task_units);
      u -= U.task * map.task_units.d;
    }
    if constexpr (kListed) {
      const uint32_t w0 = map.list[2u * u], w1 = map.list[2u * u + 1u];
      U.plane = w0 >> 24;
      U.slice = 0;
      U.m0 = (w0 & 0xFFFFFFu) * BM;
      U.n0 = (w1 & 0xFFFFFFu) * BN;
      U.quad = w1 >> 24;
      U.kbeg = map.k_begin;
      U.kend = map.k_stop;
      return U;
    }
    U.quad = 0xFu;
    const uint32_t plane_slice = div_u31(u, map.tiles);
    const uint32_t pid = u - plane_slice * map.tiles.d;
    U.slice = div_u31(plane_slice, map.planes);
    U.plane = plane_slice - U.slice * map.planes.d;
    const uint32_t group = div_u31(pid, map.group);
    const uint32_t first_m = group * C::kGroupM;
    const uint32_t rem = pid - group * map.group.d;
    const DivU31 rows = first_m + C::kGroupM <= map.tiles_m ? map.rows : map.tail;
    const uint32_t tn = div_u31(rem, rows);
    U.m0 = (first_m + rem - tn * rows.d) * BM;
    U.n0 = tn * BN;
    U.kbeg = map.k_begin + U.slice * map.k_slice;
    U.kend = min(map.k_stop, U.kbeg + map.k_slice);
    return U;
  };

  // Base pointers of a unit's task (the launch's own in ungrouped launches).
  auto base_a = [&](const Unit& U) -> const int8_t* {
    if constexpr (kGrouped) return tasks.t[U.task].a;
    else return args.a;
  };
  auto base_b = [&](const Unit& U) -> const int8_t* {
    if constexpr (kGrouped) return tasks.t[U.task].b;
    else return args.b;
  };
  auto base_c = [&](const Unit& U) -> int8_t* {
    if constexpr (kGrouped) return tasks.t[U.task].c;
    else return args.c;
  };
  auto base_ws = [&](const Unit& U) -> int8_t* {
    if constexpr (kGrouped) return tasks.t[U.task].ws;
    else return args.splitk_ws;
  };

  // ---- global -> LDS by DMA ------------------------------------------------
  // buffer_load_dwordx4 ... lds writes lane l's 16 bytes to M0 + 16*l, so one
  // wave instruction fills a contiguous 1 KB block of a stage; each lane loads
  // the global bytes that belong in its slot (the LDS swizzle is applied on
  // the global side). The lane offsets are fixed; the K tile moves the
  // buffer resources. Range checks come from the resources and read zero when
  // out of range: A's covers the valid rows of the unit's row panel from the
  // current K offset on, B's the k rows [k0, min(k0 + BK, kend)) from column
  // n0 on. B columns past the padded pitch read the next k row (zero past the
  // resource): they only feed output columns >= ldc, which are never stored.
  const uint32_t lda = static_cast<uint32_t>(args.lda), ldb = static_cast<uint32_t>(args.ldb);
  const uint32_t m_rows = static_cast<uint32_t>(args.m);
  // Wave w fills the A chunk's blocks (8 rows of 128 bytes) [2 kDmaA w, 2
  // kDmaA (w + 1)), half of them in each step of the pair, and B k rows
  // [kRowsPerBlockB kDmaB w, kRowsPerBlockB kDmaB (w + 1)).
  uint32_t a_voff[2 * C::kDmaA];
  uint32_t b_voff[C::kDmaB];
#pragma unroll
  for (int i = 0; i < 2 * C::kDmaA; ++i) {
    const int row = 8 * (wave * 2 * C::kDmaA + i) + (lane >> 3);
    a_voff[i] = static_cast<uint32_t>(row) * lda + static_cast<uint32_t>(16 * swizzle_a(row, lane & 7));
  }
#pragma unroll
  for (int i = 0; i < C::kDmaB; ++i) {
    const int k = C::kRowsPerBlockB * (wave * C::kDmaB + i) + lane / C::kChunksB;
    b_voff[i] = static_cast<uint32_t>(k) * ldb + static_cast<uint32_t>(16 * swizzle_b<BN>(k, lane % C::kChunksB));
  }
  const uint32_t lds_a = lds_address(lds) + static_cast<uint32_t>(wave * 2 * C::kDmaA * 1024);
  const uint32_t lds_b = lds_address(lds) + static_cast<uint32_t>(C::kSlotsA * C::kBufA + wave * C::kDmaB * 1024);

  // DMA cursor: the K chunk whose DMA is issued next, two chunks ahead of the
  // compute position. Past a slice's K and past the last unit the resources
  // are empty (every lane reads zero), which keeps the per-step DMA count and
  // therefore the vmcnt bookkeeping uniform. The cursor steps by additions
  // and enters the next unit exactly when the compute position is two chunks
  // from the end of its own (units of one chunk: at each, the unit after the next): one wave per SIMD issues every instruction, and
  // the ~45 scalar ones of decoding a unit and rebuilding its resources at
  // every step left the matrix cores idle meanwhile.
  struct Cursor {
    const int8_t *a, *b;
    int32_t a_n;    // bytes of A from `a` to the end of the unit's valid rows (< 2^31: gemm_args_ok)
    int32_t b_rem;  // k rows left in the unit
    uint32_t b_n0;  // the unit's column offset
    int32_t dec;    // 2 BK, or 0 past the last unit (a_n and b_rem stay 0)
  };
  auto cursor_of = [&](const Unit& U, bool live) {
    const uint32_t a_rows = min(static_cast<uint32_t>(BM), m_rows - U.m0);
    Cursor c;
    c.a = base_a(U) + static_cast<uint64_t>(U.plane) * args.pitch_a + static_cast<uint64_t>(U.m0) * lda + U.kbeg;
    c.b = base_b(U) + static_cast<uint64_t>(U.plane) * args.pitch_b + static_cast<uint64_t>(U.kbeg) * ldb + U.n0;
    c.a_n = live ? static_cast<int32_t>(a_rows * lda - U.kbeg) : 0;
    c.b_rem = live ? static_cast<int32_t>(U.kend - U.kbeg) : 0;
    c.b_n0 = live ? U.n0 : 0u;
    c.dec = live ? 2 * BK : 0;
    return c;
  };
  Cursor cur = cursor_of(decode(u_first), u_first < u_end);
  const uint64_t b_step = static_cast<uint64_t>(BK) * ldb;
  auto src_a = [&]() { return buffer_rsrc(cur.a, cur.a_n); };
  auto src_b = [&](int half) {
    const int32_t rows = min(max(cur.b_rem - half * BK, 0), static_cast<int32_t>(BK));
    return buffer_rsrc(cur.b + (half ? b_step : 0u),
                       max(rows * static_cast<int32_t>(ldb) - static_cast<int32_t>(cur.b_n0), 0));
  };
  auto cursor_advance = [&]() {
    cur.a += 2 * BK;
    cur.b += 2 * b_step;
    cur.a_n = max(cur.a_n - cur.dec, 0);
    cur.b_rem = max(cur.b_rem - cur.dec, 0);
  };
  auto dma_a = [&](v4i src, uint32_t slot, int half, int i) {
    dma16_block(__builtin_amdgcn_readfirstlane(lds_a + slot), half * C::kDmaA + i, a_voff[half * C::kDmaA + i], src);
  };
  auto dma_b = [&](v4i src, uint32_t stage, int i) {
    dma16_block(__builtin_amdgcn_readfirstlane(lds_b + stage), i, b_voff[i], src);
  };

  // ---- fragments -------------------------------------------------------------
  // One MFMA covers a whole K step: lane l takes the 16 k values 16*(l >> 4) +
  // 0..15 of the stage for both operands.
  // A (MFMA src1): lane l holds row l & 15 of a 16-row block: one ds_read_b128.
  // B (MFMA src0): lane l holds column l & 15 of a 16-column block, gathered
  // by two ds_read_b64_tr_b8. In each 16-lane group g, lane j addresses the
  // 8-byte row segment (k = base + (j >> 1), columns 8*(j & 1) .. +7 of the
  // block) and lane i receives byte i & 7 of the segments of lanes
  // 2b + (i >> 3), b = 0..7: its column across 8 consecutive k.
  const int frag_row = lane & 15;
  const int frag_k = lane >> 4;
  struct Frags {
    v4i a[TM];
    v4i b[TN];
  };
  // (slots and stages are byte offsets)
  auto read_a = [&](uint32_t slot, int half, int i) {
    const int r = wave_m * (16 * TM) + 16 * i + frag_row;
    return *reinterpret_cast<const v4i*>(lds + slot + r * (2 * BK) + swizzle_a(frag_row, 4 * half + frag_k) * 16);
  };
  auto read_b = [&](uint32_t stage, int j) {
    const int8_t* const sb = lds + C::kSlotsA * C::kBufA + stage;
    const int chunk = wave_n * TN + j;
    const int k = 16 * frag_k + (frag_row >> 1);
    const int8_t* const at = sb + k * BN + swizzle_b<BN>(k, chunk) * 16 + 8 * (frag_row & 1);
    const v2i lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32(as_lds_v2i(at));
    const v2i hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32(as_lds_v2i(at + 8 * BN));  // f(k + 8) = f(k)
    return v4i{lo[0], lo[1], hi[0], hi[1]};
  };

  v4i acc[TM][TN];
  // The MFMAs of block rows [i0, i0 + TM/2) for one K step, columns in
  // alternating order so consecutive MFMAs share an operand. A unit's first
  // step starts from the bias (an inline constant, no accumulator writes).
  auto mfma_half = [&](auto first, const Frags& f, int i0) __attribute__((always_inline)) {
#pragma unroll
    for (int ii = 0; ii < TM / 2; ++ii)
#pragma unroll
      for (int jj = 0; jj < TN; ++jj) {
        const int i = i0 + ii, j = (ii & 1) ? TN - 1 - jj : jj;
        const v4i start = {kAccBias, kAccBias, kAccBias, kAccBias};
        acc[i][j] = __builtin_amdgcn_mfma_i32_16x16x64_i8(f.b[j], f.a[i], decltype(first)::value ? start : acc[i][j],
                                                          0, 0, 0);
      }
  };
  // Interleave a half step's TM/2*TN MFMAs with half of the next position's
  // fragment reads, spread over its first three quarters.
  constexpr int kMfma = TM / 2 * TN;
  constexpr int kReads = TM / 2 + TN;
  constexpr int kPerSlot = kMfma * 3 / 4 / kReads > 0 ? kMfma * 3 / 4 / kReads : 1;
  // The MFMA builtins carry no ordering of their own, so instruction
  // selection may place some of a region's MFMAs after its sched_barrier; an
  // empty asm statement that takes every accumulator (and is ordered before
  // the barrier) keeps them all inside the region.
  auto schedule_region = [&](auto id, int i0) __attribute__((always_inline)) {
    constexpr int kId = decltype(id)::value;
#pragma unroll
    for (int i = 0; i < TM / 2; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) asm volatile("" ::"a"(acc[i0 + i][j]));
    sched_slots<kId, kPerSlot, kReads>();
    if constexpr (kMfma > kPerSlot * kReads)
      __builtin_amdgcn_sched_group_barrier(0x008, kMfma - kPerSlot * kReads, kId);
    __builtin_amdgcn_sched_barrier(0);
  };

  // ---- epilogue ---------------------------------------------------------------
  // acc[i][j] register e holds u = kAccBias + C[row][col] (the accumulators
  // start at kAccBias) with
  //   row = m0 + wave_m*16*TM + 16i + (lane & 15)
  //   col = n0 + wave_n*16*TN + 16j + 4*(lane >> 4) + e.
  // Stores go through a buffer resource over the unit's tile rows, so rows
  // >= M are dropped by the range check; columns past the padded pitch (only
  // in the last tile column) get an offset beyond num_records.
  auto epilogue = [&](const Unit& U) {
    // The accumulator reads below are asm, so the compiler inserts no wait
    // states after the last MFMA for them: 24 here cover the longest
    // MFMA-write to v_accvgpr_read dependency.
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7");
    const ModulusConsts mc = plane_mod(pc, U.plane);
    const int64_t tile_rows = min(static_cast<int64_t>(BM), args.m - U.m0);
    const uint32_t lane_off =
        static_cast<uint32_t>((wave_m * (16 * TM) + frag_row) * args.ldc + wave_n * (16 * TN));
    const uint32_t row_step = static_cast<uint32_t>(16 * args.ldc);
    const bool full_cols = U.n0 + BN <= args.ldc;
    // a listed unit's wave stores its quadrant only if the mask selects it
    if (kListed && ((U.quad >> (wave_m * 2 + (wave_n >= C::WN / 2 ? 1 : 0))) & 1u) == 0u) return;
    // the unit's tile of C, or of its K slice's workspace slot
    // [slice][plane][M][ldc] (split launches never accumulate)
    int8_t* const Cp =
        args.slices <= 1
            ? base_c(U) + static_cast<int64_t>(U.plane) * args.pitch_c + U.m0 * args.ldc + U.n0
            : base_ws(U) + ((static_cast<int64_t>(U.slice) * args.nplanes + U.plane) * args.m + U.m0) * args.ldc +
                  U.n0;
    const __amdgpu_buffer_rsrc_t c_rsrc = make_rsrc(Cp, tile_rows * args.ldc - U.n0);
    const CenteredI32 kc = centered_acc_consts(mc);
    // Each lane's packed dword of block (i, j) holds 4 columns of a row. Four
    // neighbouring blocks' dwords are transposed across the four 16-lane
    // groups (two half-wave and two row swaps), so lane group g holds the 16
    // bytes of block 4q + g's row and one 16-byte store covers 64 contiguous
    // bytes of each of 16 rows.
    auto reduce = [&](auto carry, auto low_byte) {
      constexpr bool kCarry = decltype(carry)::value;
      constexpr bool kLowByte = decltype(low_byte)::value;  // m = 256: the residue is the low byte
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const uint32_t off = lane_off + static_cast<uint32_t>(i) * row_step;
        uint32_t prev[TN];
        if constexpr (kCarry) {
          // later K block: add the centered residue carried in C (|.| <= 128)
#pragma unroll
          for (int j = 0; j < TN; ++j)
            prev[j] = static_cast<uint32_t>(
                __builtin_amdgcn_raw_buffer_load_b32(c_rsrc, static_cast<int>(off + 16 * j + 4 * frag_k), 0, 0));
        }
#pragma unroll
        for (int q = 0; q < TN / 4; ++q) {
          uint32_t d[4];
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            const int j = 4 * q + jj;
            const Acc4 a4 = acc_read4(acc[i][j]);
            if constexpr (kLowByte) {
              // the bias is 0 mod 256, so u's low byte is C's, read as int8 its centered residue
              d[jj] = pack_low_bytes(a4.v[0], a4.v[1], a4.v[2], a4.v[3]);
            } else {
              uint32_t res[4];
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                uint32_t u = a4.v[e];
                if constexpr (kCarry)
                  u += static_cast<uint32_t>(static_cast<int32_t>(static_cast<int8_t>(prev[j] >> (8 * e))));
                res[e] = centered_residue_i32(u, mc, kc);
              }
              d[jj] = pack_low_bytes(res[0], res[1], res[2], res[3]);
            }
          }
          const auto s02 = __builtin_amdgcn_permlane32_swap(d[0], d[2], false, false);
          const auto s13 = __builtin_amdgcn_permlane32_swap(d[1], d[3], false, false);
          const auto t01 = __builtin_amdgcn_permlane16_swap(s02[0], s13[0], false, false);
          const auto t23 = __builtin_amdgcn_permlane16_swap(s02[1], s13[1], false, false);
          const v4i v = {static_cast<int>(t01[0]), static_cast<int>(t01[1]), static_cast<int>(t23[0]),
                         static_cast<int>(t23[1])};
          const int col = wave_n * (16 * TN) + 64 * q + 16 * frag_k;
          const bool ok = full_cols || col < static_cast<int>(args.ldc - U.n0);
          __builtin_amdgcn_raw_buffer_store_b128(
              v, c_rsrc, static_cast<int>(ok ? off + 64 * q + 16 * frag_k : 0x80000000u), 0, 0);
        }
      }
    };
    if (accumulate)
      reduce(std::true_type{}, std::false_type{});
    else if (mc.m == 256u)
      reduce(std::false_type{}, std::true_type{});
    else
      reduce(std::false_type{}, std::false_type{});
  };

  // ---- pipeline ----------------------------------------------------------------
  // Three A slots (a chunk of two K steps each) and four B stages. Stream
  // position s (the s-th K step of this workgroup's work list, across unit
  // boundaries; position s belongs to chunk s / 2) is computed from registers:
  // its fragments were read during position s-1. While it computes, the
  // fragments of position s+1 are read, the DMA of B's position s+4 goes into
  // stage s % 4 and half of A's chunk s/2 + 2 into slot (s/2 + 2) % 3; every
  // wave finished reading both before the last barrier (B's position s was
  // read during s-1, chunk s/2 - 1 during at most s-2). Before the barrier
  // that ends position s each wave waits for its DMAs of position s+2, read
  // next (issued up to position s-2, or, for the second half of an A chunk,
  // first in position s-1: then only that position's B DMAs and position s's
  // may be outstanding; older VMEM operations, the previous epilogue's stores
  // included, complete in order before them) and for its fragment reads, so
  // the barrier publishes position s+2 and retires every read of position
  // s+1. The DMAs are issued from inline asm, so the compiler tracks no LDS
  // write for them and adds no waits before the fragment reads: the explicit
  // vmcnt waits below are what orders them. They are spread over the step (A
  // DMAs in the first half, B DMAs in the second): each one holds the texture
  // path for a while, and bunching a step's DMAs stalls MFMA issue.
  constexpr int kDmaStep = C::kDmaA + C::kDmaB;
  Frags f0, f1;
  uint32_t slot0 = 0, slot1 = C::kBufA, slot2 = 2 * C::kBufA;  // chunks c, c+1, c+2 of the compute position
  uint32_t stage0 = 0, stage2 = 2 * C::kBufB;                  // B stages of the pair and of the next pair
  // (units of one chunk: the second is the next unit's)
  const bool one_chunk = map.pairs == 1u;
  auto unit_cursor = [&](uint32_t u) { return cursor_of(decode(min(u, u_end - 1)), u < u_end); };
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    const v4i sa = src_a();
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const v4i sb = src_b(half);
#pragma unroll
      for (int i = 0; i < C::kDmaA; ++i) dma_a(sa, c * C::kBufA, half, i);
#pragma unroll
      for (int i = 0; i < C::kDmaB; ++i) dma_b(sb, (2 * c + half) * C::kBufB, i);
    }
    cursor_advance();
    if (c == 0 && one_chunk) cur = unit_cursor(u_first + u_step);
  }
  __builtin_amdgcn_s_waitcnt(wait_vm(2 * kDmaStep));  // chunk 0 landed
  __syncthreads();
#pragma unroll
  for (int i = 0; i < TM; ++i) f0.a[i] = read_a(0, 0, i);
#pragma unroll
  for (int j = 0; j < TN; ++j) f0.b[j] = read_b(0, j);
  __syncthreads();  // B stage 0 is read: position 4 may overwrite it
  // K step `half` of the pair: MFMAs on `f`, the next position's fragments
  // into `fn`.
  auto step = [&](auto first, auto half_c, const Frags& f, Frags& fn) __attribute__((always_inline)) {
    constexpr int half = decltype(half_c)::value;
    constexpr int kRegionLen = TM / 2 > TN / 2 ? (TM / 2 > 4 ? TM / 2 : 4) : (TN / 2 > 4 ? TN / 2 : 4);
    const uint32_t next_slot = half ? slot1 : slot0;
    const uint32_t next_stage = half ? stage2 : stage0 + C::kBufB;
    const uint32_t dma_stage = stage0 + half * C::kBufB;
    const v4i sa = src_a(), sb = src_b(half);
#pragma unroll
    for (int t = 0; t < kRegionLen; ++t) {
      if (t < TM / 2) fn.a[t] = read_a(next_slot, half ^ 1, t);
      if (t < TN / 2) fn.b[t] = read_b(next_stage, t);
      if (t < C::kDmaA) dma_a(sa, slot2, half, t);
    }
    mfma_half(first, f, 0);
    schedule_region(std::integral_constant<int, 1>{}, 0);
#pragma unroll
    for (int t = 0; t < kRegionLen; ++t) {
      if (t < TM / 2) fn.a[TM / 2 + t] = read_a(next_slot, half ^ 1, TM / 2 + t);
      if (t < TN / 2) fn.b[TN / 2 + t] = read_b(next_stage, TN / 2 + t);
      if (t < C::kDmaB) dma_b(sb, dma_stage, t);
    }
    mfma_half(first, f, TM / 2);
    // the cursor's scalar work issues in the shadow of this region's MFMAs
    if constexpr (half == 1) cursor_advance();
    schedule_region(std::integral_constant<int, 2>{}, TM / 2);
    // the next position's fragments stay in this step
#pragma unroll
    for (int i = 0; i < TM; ++i) asm volatile("" ::"v"(fn.a[i]));
#pragma unroll
    for (int j = 0; j < TN; ++j) asm volatile("" ::"v"(fn.b[j]));
    __builtin_amdgcn_s_waitcnt(wait_vm(half ? 2 * kDmaStep : kDmaStep + C::kDmaB));
    __syncthreads();
  };
  auto pair = [&](auto first) __attribute__((always_inline)) {
    step(first, std::integral_constant<int, 0>{}, f0, f1);
    step(std::false_type{}, std::integral_constant<int, 1>{}, f1, f0);
    const uint32_t s = slot0;
    slot0 = slot1;
    slot1 = slot2;
    slot2 = s;
    stage0 ^= 2 * C::kBufB;
    stage2 ^= 2 * C::kBufB;
  };
  for (uint32_t u = u_first; u < u_end; u += u_step) {
    const Unit U = decode(u);
    const Cursor next = unit_cursor(u + (one_chunk ? 2 * u_step : u_step));
    // The cursor enters the next unit (of one-chunk units the one after it) by
    // selects at the pair two chunks before the end (a branch there makes the
    // compiler duplicate the pair and spill accumulators).
    auto enter_next = [&](bool enter) {
      cur.a = enter ? next.a : cur.a;
      cur.b = enter ? next.b : cur.b;
      cur.a_n = enter ? next.a_n : cur.a_n;
      cur.b_rem = enter ? next.b_rem : cur.b_rem;
      cur.b_n0 = enter ? next.b_n0 : cur.b_n0;
      cur.dec = enter ? next.dec : cur.dec;
    };
    uint32_t n = map.pairs;
    enter_next(n <= 2u);
    pair(std::true_type{});
    for (--n; n; --n) {
      enter_next(n == 2u);
      pair(std::false_type{});
    }
    epilogue(U);
  }
  __builtin_amdgcn_s_waitcnt(wait_vm(0));  // no DMA outlives the workgroup's LDS
}

// Zero-output tiles of a per-tile schedule: planes [0, planes) of each tile's
// rows and columns are set to 0 (reference cpu_reference.cpp:243-246). Whole
// 16-byte chunks are written: a tile's column offset is a multiple of 64, and
// the last tile column's chunks end inside the padded pitch.
__global__ __launch_bounds__(256) void zero_tiles_kernel(int8_t* c, int64_t ldc, int64_t pitch_c,
                                                         const TileFill* tiles) {
  const TileFill t = tiles[blockIdx.x];
  const uint32_t chunks = (t.cols + 15u) / 16u;
  const uint64_t per_plane = static_cast<uint64_t>(t.rows) * chunks;
  const uint64_t total = per_plane * t.planes;
  for (uint64_t i = threadIdx.x; i < total; i += blockDim.x) {
    const uint32_t p = static_cast<uint32_t>(i / per_plane);
    const uint64_t rem = i - static_cast<uint64_t>(p) * per_plane;
    const uint32_t r = static_cast<uint32_t>(rem / chunks);
    const uint32_t ch = static_cast<uint32_t>(rem - static_cast<uint64_t>(r) * chunks);
    int8_t* const dst = c + static_cast<int64_t>(p) * pitch_c + static_cast<int64_t>(t.row_off + r) * ldc + t.col_off +
                        16 * ch;
    *reinterpret_cast<v4i*>(dst) = v4i{0, 0, 0, 0};
  }
}

__global__ __launch_bounds__(256) void zero_words_kernel(uint32_t* dst, uint64_t words) {
  for (uint64_t w = static_cast<uint64_t>(blockIdx.x) * blockDim.x + threadIdx.x; w < words;
       w += static_cast<uint64_t>(gridDim.x) * blockDim.x)
    dst[w] = 0u;
}

using Cfg256x256 = Cfg<8, 8, 2>;  // one workgroup per CU (all 512 registers per lane)
using Cfg256x128 = Cfg<8, 4, 2>;  // one per CU (128 KB of LDS)
using Cfg128x256 = Cfg<4, 8, 2>;  // one per CU (112 KB)
using Cfg128x128 = Cfg<4, 4, 2>;  // two per CU
using Cfg64x64 = Cfg<2, 4, 1>;    // two waves, four workgroups per CU

template <typename Cf>
int64_t tile_count(int64_t m, int64_t n, uint32_t nplanes) {
  return ((m + Cf::BM - 1) / Cf::BM) * ((n + Cf::BN - 1) / Cf::BN) * static_cast<int64_t>(nplanes);
}

}  // namespace

namespace {

// The tile whose launch is predicted fastest. A launch costs a start plus, for
// the CU with the most units, each unit's K chunks and epilogue (workgroups
// that share a CU share its matrix cores, so their costs add). The costs, in
// 10 ns, were fitted to launches of 16 shapes from 256^3 to 4096^3 (K from 256
// to 30000, 1 to 18 planes; the measured best tile is within 3% of the choice
// at each). They trade the operand traffic per product (256x256 least) against
// the units left for the last round: 1024^3 at 9 planes ran 16.7 us with
// 256x256 tiles (144 units), 18.5 with 256x128, 15.2 with 128x128 (576); 700 x
// 700 x 3000 at 8 planes 33.0, 20.8, 22.3; one 1024^3 plane 15.6, 9.9, 7.0
// and 5.6 with 64x64; 4096^3 at 1 plane 52.8, 59.5, 65.0, 128.
GemmTile choose_tile(int64_t m, int64_t n, int64_t k_slice, int64_t plane_slices) {
  struct TileCost {
    GemmTile tile;
    int64_t bm, bn, start, chunk, unit;
  };
  constexpr TileCost kCosts[] = {
      {GemmTile::k256x256, 256, 256, 400, 150, 300}, {GemmTile::k256x128, 256, 128, 350, 84, 200},
      {GemmTile::k128x256, 128, 256, 350, 84, 200},  {GemmTile::k128x128, 128, 128, 300, 45, 100},
      {GemmTile::k64x64, 64, 64, 250, 25, 60}};
  constexpr int64_t kCus = 256;
  const int64_t chunks = (std::min<int64_t>(k_slice, kSafeKBlock) + 127) / 128;
  GemmTile best = GemmTile::k128x128;
  double best_cost = 0;
  for (const TileCost& t : kCosts) {
    const double units = static_cast<double>((m + t.bm - 1) / t.bm) * static_cast<double>((n + t.bn - 1) / t.bn) *
                         static_cast<double>(plane_slices);
    if (units > 0x7FFFFFFF) continue;  // unit numbers are 31-bit
    const double rounds = std::ceil(units / kCus);
    const double cost = static_cast<double>(t.start) + rounds * static_cast<double>(chunks * t.chunk + t.unit);
    if (best_cost == 0 || cost < best_cost) {
      best = t.tile;
      best_cost = cost;
    }
  }
  return best;
}

}  // namespace

GemmShape choose_gemm_shape(int64_t m, int64_t n, int64_t k, uint32_t nplanes) {
  // Results at most 16 columns wide: the skinny kernel (skinny.hip).
  GemmShape shape{};
  if (skinny_shape(m, n, k, nplanes, shape)) return shape;
  // K is split when 128 x 128 tiles leave the chip under-filled and K is
  // long: toward ~512 units of that size, with slices of at least 4096 K and
  // at most 65536. Each slice adds a residue tile per plane to write and sum,
  // and short slices spend a larger share in the DMA prologue and the
  // epilogue.
  shape.slices = 1;
  shape.k_slice = k;
  shape.tile = choose_tile(m, n, k, nplanes);
  if (m > 128 && n > 128 && tile_count<Cfg256x256>(m, n, nplanes) >= 256) return shape;
  const int64_t tiles = tile_count<Cfg128x128>(m, n, nplanes);
  if (tiles >= 256 || k < 8192) return shape;
  int64_t slices = std::min<int64_t>((512 + tiles - 1) / tiles, k / 4096);
  slices = std::max<int64_t>(slices, (k + kSafeKBlock - 1) / kSafeKBlock);
  if (slices <= 1) return shape;
  int64_t k_slice = (k + slices - 1) / slices;
  k_slice = (k_slice + Cfg128x128::BK - 1) / Cfg128x128::BK * Cfg128x128::BK;
  slices = (k + k_slice - 1) / k_slice;
  if (slices <= 1 || slices * tiles > 0x7FFFFFFF) return shape;
  shape.tile = choose_tile(m, n, k_slice, nplanes * slices);
  shape.slices = static_cast<uint32_t>(slices);
  shape.k_slice = k_slice;
  shape.ws_bytes = static_cast<uint64_t>(slices) * nplanes * static_cast<uint64_t>(m) * static_cast<uint64_t>(padded_ld(n));
  return shape;
}

hipError_t launch_zero_words(uint32_t* dst, uint64_t words, hipStream_t stream) {
  if (words == 0) return hipSuccess;
  if (!dst) return hipErrorInvalidValue;
  const uint64_t blocks = (words + 255) / 256;
  const unsigned grid = static_cast<unsigned>(blocks < 4096 ? blocks : 4096);
  hipLaunchKernelGGL(zero_words_kernel, dim3(grid), dim3(256), 0, stream, dst, words);
  return hipGetLastError();
}

namespace {

// Compute units of the current device (cached per device id; contexts on
// several threads may launch at once, so the cache is atomic).
int device_cu_count() {
  static std::atomic<int> cached[64] = {};
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 256;
  int cus = cached[dev].load(std::memory_order_relaxed);
  if (cus == 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    cached[dev].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

// K chunks of 128 that every unit of a launch runs.
uint32_t k_pairs(int64_t k_slice) { return static_cast<uint32_t>((k_slice + 127) / 128); }

// Ungrouped launches pass a NoTaskTable and ntasks = 1; grouped ones the
// task table and its task count (at most kMaxGroupTasks). `k_slice` is the
// K of one slice when args.slices > 1.
template <typename Cf, int kMinBlocks, bool kGrouped>
hipError_t launch_gemm_cfg(const GemmArgs& args, int64_t k_slice, const PlaneConsts& consts, hipStream_t stream,
                           const GroupArg<kGrouped>& tab, uint32_t ntasks) {
  const uint32_t tiles_m = static_cast<uint32_t>((args.m + Cf::BM - 1) / Cf::BM);
  const uint32_t tiles_n = static_cast<uint32_t>((args.ldc + Cf::BN - 1) / Cf::BN);
  const uint64_t slots = static_cast<uint64_t>(device_cu_count()) * kMinBlocks;
  // One launch per K range: the whole K split into args.slices slices, or,
  // unsplit, int32-safe blocks of 65536 whose later launches add their sum to
  // the centered residue already in C (reference cpu_reference.cpp:160-175).
  const int64_t block = args.slices > 1 ? args.k : kSafeKBlock;
  for (int64_t kb = 0; kb < args.k; kb += block) {
    const int64_t kstop = min(args.k, kb + block);
    const uint32_t accumulate = kb > 0 ? 1u : 0u;
    const int64_t ks = args.slices > 1 ? k_slice : kstop - kb;
    const uint32_t used_slices = static_cast<uint32_t>((kstop - kb + ks - 1) / ks);
    if (ks <= 0 || ks > kSafeKBlock || used_slices != args.slices) return hipErrorInvalidValue;
    const uint64_t task_units = static_cast<uint64_t>(tiles_m) * tiles_n * args.nplanes * used_slices;
    const uint64_t units = task_units * ntasks;
    if (units == 0 || units > 0x7FFFFFFFull) return hipErrorInvalidValue;
    UnitMap map{};
    map.units = static_cast<uint32_t>(units);
    map.task_units = make_div_u31(static_cast<uint32_t>(task_units));
    map.tiles_m = tiles_m;
    map.tiles = make_div_u31(tiles_m * tiles_n);
    map.planes = make_div_u31(args.nplanes);
    map.group = make_div_u31(static_cast<uint32_t>(Cf::kGroupM) * tiles_n);
    map.rows = make_div_u31(Cf::kGroupM);
    map.tail = make_div_u31(tiles_m - (tiles_m - 1) / Cf::kGroupM * Cf::kGroupM);
    map.k_begin = static_cast<uint32_t>(kb);
    map.k_stop = static_cast<uint32_t>(kstop);
    map.k_slice = static_cast<uint32_t>(ks);
    const uint64_t grid = persistent_grid(units, slots);
    map.pairs = k_pairs(ks);
    hipLaunchKernelGGL((plane_gemm_kernel<Cf, kMinBlocks, false, kGrouped>), dim3(static_cast<unsigned>(grid)),
                       dim3(Cf::kThreads), 0, stream, args, consts, map, accumulate, tab);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
    if (args.slices > 1) {
      for (uint32_t t = 0; t < ntasks; ++t) {
        int8_t* ws = args.splitk_ws;
        int8_t* c = args.c;
        if constexpr (kGrouped) {
          ws = tab.t[t].ws;
          c = tab.t[t].c;
        }
        err = launch_residue_finalize(ws, c, args.m, args.ldc, args.pitch_c, args.nplanes, args.slices, consts,
                                      stream);
        if (err != hipSuccess) return err;
      }
    }
  }
  return hipSuccess;
}

// The kernel of `shape`'s tile.
template <bool kGrouped>
hipError_t launch_tiles(const GemmShape& shape, const GemmArgs& args, const PlaneConsts& consts, hipStream_t stream,
                        const GroupArg<kGrouped>& tab, uint32_t ntasks) {
  switch (shape.tile) {
    case GemmTile::k256x256:
      return launch_gemm_cfg<Cfg256x256, 1, kGrouped>(args, shape.k_slice, consts, stream, tab, ntasks);
    case GemmTile::k256x128:
      return launch_gemm_cfg<Cfg256x128, 1, kGrouped>(args, shape.k_slice, consts, stream, tab, ntasks);
    case GemmTile::k128x256:
      return launch_gemm_cfg<Cfg128x256, 1, kGrouped>(args, shape.k_slice, consts, stream, tab, ntasks);
    case GemmTile::k128x128:
      return launch_gemm_cfg<Cfg128x128, 2, kGrouped>(args, shape.k_slice, consts, stream, tab, ntasks);
    case GemmTile::k64x64:
      return launch_gemm_cfg<Cfg64x64, 4, kGrouped>(args, shape.k_slice, consts, stream, tab, ntasks);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace

namespace {

template <typename Cf, int kMinBlocks>
hipError_t launch_listed(const GemmArgs& args, const PlaneConsts& consts, const uint32_t* d_units, uint32_t units,
                         hipStream_t stream) {
  const uint64_t slots = static_cast<uint64_t>(device_cu_count()) * kMinBlocks;
  const uint64_t grid = persistent_grid(units, slots);
  for (int64_t kb = 0; kb < args.k; kb += kSafeKBlock) {
    const int64_t kstop = min(args.k, kb + kSafeKBlock);
    UnitMap map{};
    map.units = units;
    map.k_begin = static_cast<uint32_t>(kb);
    map.k_stop = static_cast<uint32_t>(kstop);
    map.k_slice = static_cast<uint32_t>(kstop - kb);
    map.pairs = k_pairs(kstop - kb);
    map.list = d_units;
    hipLaunchKernelGGL((plane_gemm_kernel<Cf, kMinBlocks, true>), dim3(static_cast<unsigned>(grid)),
                       dim3(Cf::kThreads), 0, stream, args, consts, map, kb > 0 ? 1u : 0u, NoTaskTable{});
    const hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace

hipError_t launch_gemm_listed(const GemmArgs& args, const PlaneConsts& consts, const uint32_t* d_units,
                              uint32_t units, uint32_t edge, hipStream_t stream) {
  // the list's entries are checked against the shape and edge where it is built
  if (!gemm_args_ok(args) || args.slices != 1 || !d_units || units > 0x7FFFFFFFu) return hipErrorInvalidValue;
  if (units == 0) return hipSuccess;
  if (edge == 256) return launch_listed<Cfg256x256, 1>(args, consts, d_units, units, stream);
  if (edge == 128) return launch_listed<Cfg128x128, 2>(args, consts, d_units, units, stream);
  return hipErrorInvalidValue;
}

hipError_t launch_zero_tiles(int8_t* c, int64_t ldc, int64_t pitch_c, const TileFill* d_tiles, uint32_t count,
                             hipStream_t stream) {
  if (count == 0) return hipSuccess;
  if (!c || !d_tiles || ldc <= 0 || ldc % 16 || pitch_c < ldc || count > 0x7FFFFFFFu) return hipErrorInvalidValue;
  hipLaunchKernelGGL(zero_tiles_kernel, dim3(count), dim3(256), 0, stream, c, ldc, pitch_c, d_tiles);
  return hipGetLastError();
}

// ---- static scratch for calls that allocate nothing ---------------------------
// The split-K residues of rns8_mi355x_gemm_rns_noalloc live here instead of
// in a caller's workspace. Each device holds its own copy of the array for
// the life of the process. On the host the array's name is not a device
// address: host code uses the per-device address resolve_noalloc_scratch
// records (hipGetSymbolAddress with that device current).
static __device__ __align__(256) int8_t scratch[kNoAllocScratchBytes];

namespace {
constexpr int kMaxDevices = 64;
std::atomic<int8_t*> g_scratch[kMaxDevices] = {};
std::mutex g_scratch_mutex;
}  // namespace

hipError_t resolve_noalloc_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return hipErrorInvalidDevice;
  if (g_scratch[device].load(std::memory_order_acquire)) return hipSuccess;
  int current = -1;
  if (hipGetDevice(&current) != hipSuccess || current != device) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch[device].load(std::memory_order_acquire)) return hipSuccess;
  void* ptr = nullptr;
  const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
  if (e != hipSuccess) return e;
  if (!ptr || (reinterpret_cast<uintptr_t>(ptr) & 255u) != 0) return hipErrorInvalidSymbol;
  g_scratch[device].store(static_cast<int8_t*>(ptr), std::memory_order_release);
  return hipSuccess;
}

int8_t* noalloc_scratch(int device) {
  if (device < 0 || device >= kMaxDevices) return nullptr;
  return g_scratch[device].load(std::memory_order_acquire);
}

hipError_t launch_gemm(const GemmArgs& args, const PlaneConsts& consts, hipStream_t stream) {
  if (!gemm_args_ok(args)) return hipErrorInvalidValue;
  const GemmShape shape = choose_gemm_shape(args.m, args.n, args.k, args.nplanes);
  // the workspace was sized for the plan's slices: never use a different
  // split (an unsplit call of a split shape runs unsplit where the kernel
  // allows it)
  if (args.slices > 1 && args.slices != shape.slices) return hipErrorInvalidValue;
  if (shape.tile == GemmTile::kSkinny) {
    if (args.slices == shape.slices) return launch_skinny(args, shape, consts, stream);
    // an unsplit call (no workspace) of a shape the skinny kernel would
    // split: the 128 x 128 kernel, which takes any K in 65536 blocks
    if (args.slices != 1) return hipErrorInvalidValue;
    return launch_gemm_cfg<Cfg128x128, 2, false>(args, args.k, consts, stream, NoTaskTable{}, 1);
  }
  return launch_tiles<false>(shape, args, consts, stream, NoTaskTable{}, 1);
}

hipError_t launch_gemm_grouped(const GemmArgs& shape, const PlaneConsts& consts, const TaskPtrs* tasks,
                               uint32_t count, hipStream_t stream) {
  if (!tasks || count == 0) return hipErrorInvalidValue;
  // tile and K split for the whole group (the tasks count as extra planes);
  // never more slices than the shape's own workspaces hold
  const GemmShape g = choose_gemm_shape(shape.m, shape.n, shape.k, shape.nplanes * count);
  if (g.slices > 1 && g.slices > shape.slices) return hipErrorInvalidValue;
  for (uint32_t t = 0; t < count; ++t) {
    // every task's operands pass the same checks as an ungrouped launch
    GemmArgs a = shape;
    a.a = tasks[t].a;
    a.b = tasks[t].b;
    a.c = tasks[t].c;
    a.splitk_ws = tasks[t].ws;
    a.slices = g.tile == GemmTile::kSkinny ? shape.slices : g.slices;
    if (!gemm_args_ok(a)) return hipErrorInvalidValue;
  }
  if (g.tile == GemmTile::kSkinny) {
    // the skinny kernel fills the chip from one task's rows and K slices:
    // one launch per task, each with its own workspace
    for (uint32_t t = 0; t < count; ++t) {
      GemmArgs a = shape;
      a.a = tasks[t].a;
      a.b = tasks[t].b;
      a.c = tasks[t].c;
      a.splitk_ws = tasks[t].ws;
      const hipError_t err = launch_gemm(a, consts, stream);
      if (err != hipSuccess) return err;
    }
    return hipSuccess;
  }
  for (uint32_t first = 0; first < count; first += kMaxGroupTasks) {
    const uint32_t n = count - first < kMaxGroupTasks ? count - first : kMaxGroupTasks;
    TaskTable tab{};
    for (uint32_t t = 0; t < n; ++t) tab.t[t] = tasks[first + t];
    GemmArgs a = shape;
    a.a = a.b = nullptr;
    a.c = nullptr;
    a.splitk_ws = nullptr;
    a.slices = g.slices;
    const hipError_t err = launch_tiles<true>(g, a, consts, stream, tab, n);
    if (err != hipSuccess) return err;
  }
  return hipSuccess;
}

}  // namespace rns8x
