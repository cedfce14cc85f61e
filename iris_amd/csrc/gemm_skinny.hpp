// Shard GEMM for a few rows of A (decode-time batches, 16 or 32 rows a workgroup): C[M,N] = A[M,K] B[K,N]
// with the epilogues of the persistent kernel (gemm_all_scatter.py:209-251,
// gemm_atomics_all_reduce.py:236-248, gemm_one_shot_all_reduce.py:197-218).
//
// With so few rows the product is a stream over B: every byte of B is used
// once, the matrix cores idle, and what matters is how many bytes a CU has in
// flight and how many bytes each cache-line access of its L1 brings.  A
// workgroup of eight waves owns 16 columns of C and its waves share the K
// range out in blocks of 64, each wave two blocks in flight:
//   * B, the stream, comes in with `buffer_load ... lds`, one instruction per
//     8 rows x 128 bytes (whole cache lines: twice the bytes per line access
//     of a fetch in MFMA operand layout, 16 rows x 64 bytes), into a region of
//     LDS private to the wave, 16-byte chunks XOR-ed by the row so that the
//     operand reads are conflict-free;
//   * A, rows that every workgroup reads and L2 holds, goes into registers,
//     lanes along a row like B, and passes through 2 KiB of LDS on its way to
//     the MFMAs (a load in operand layout has neighbouring lanes in different
//     rows and merges nothing).
// A block that has been multiplied gives its place to the fetches of the one
// after next.  Two blocks a wave are enough, as three workgroups then share a
// CU: with eight (one workgroup a CU, all fetches of a K of 4096 issued before
// the first MFMA) [16,3584] x [3584,8192] took 17.6 us a pass and takes 14.1,
// [6,2560] x [2560,6208] 13.9 -> 8.9, and nothing measured is slower.  What a
// workgroup alone on its CU is bound by is the addresses: 16 clocks an
// instruction, whichever of its lanes are in range.  So up to eight rows of A
// are one instruction a block, not two ([1,1376] .. [8,4096] x [4096,1376]
// 8.6 -> 7.9 us at eight rows).
// A K too long for that is shared out over workgroups (gridDim.z of them a
// block of C), which leave their sums in the caller's workspace; the last one
// to arrive adds them up.  [2,23680] x [23680,736] 18.6 -> 11.0 us,
// [4,36864] x [36864,512] 28.8 -> 12.3.
// The waves' partial 16x16 accumulators meet in LDS; wave w then stores the
// sum on destination rank w, w+8, ...
//
// A logical tile (BLOCK_SIZE_M x BLOCK_SIZE_N, one flag) spans several such
// workgroups.  They count their arrivals in locks[tile_id]; the last one to
// arrive re-arms the counter and publishes the tile's flag.
//
// fp32 operands: the launcher counts K and the strides in 16-bit units, so a
// block of K is 32 elements of the same 128 bytes, a chunk four of them
// (gemm_kernel.hpp, Mfma<IRIS_DTYPE_F32>).  [16,4096] x [4096,4096] takes 19.1 us a
// pass, 14.1 of them B's 67 MB at the rate of a large copy.
#pragma once

#include "gemm_registry.hpp"
#include "late_tiles.hpp"

namespace iris_amd {

constexpr int SKINNY_ROWS = 16;    // rows of A per block (a workgroup takes RB blocks of them, blockIdx.y counts its share)
constexpr int SKINNY_MAX_ROWS = 32;  // rows of A a launch of single blocks can take: beyond, B is re-read too often
constexpr int SKINNY_COLS = 16;    // columns of C per workgroup
constexpr int SKINNY_MID_MAX_ROWS = 64;   // rows of A a launch of 32-row workgroups can take ...
constexpr int SKINNY_MID_MIN_K = 2048;    // ... when K is at least this long
constexpr int SKINNY_F32_MAX_ROWS = 128;  // rows of A an fp32 launch of them can take
constexpr int SKINNY_WAVES = 8;
constexpr int SKINNY_THREADS = SKINNY_WAVES * 64;
constexpr int SKINNY_BLOCK_BYTES = 2048;                  // 16 rows of A or B x 64 k
constexpr int SKINNY_UN = 2;       // K blocks whose fetches a wave has in flight
constexpr int SKINNY_MAX_SPLIT = 16;
// LDS of a workgroup of RB blocks: a block of A per wave and row block (the waves' partial accumulators, 1 KiB a
// block, take its place once the K range is done), then every wave's K blocks of B
constexpr int skinny_a_bytes(int rb) { return SKINNY_WAVES * rb * SKINNY_BLOCK_BYTES; }
constexpr int skinny_lds_bytes(int rb) { return skinny_a_bytes(rb) + SKINNY_WAVES * SKINNY_UN * SKINNY_BLOCK_BYTES; }

// Blocks of 32 rows x 32 columns a workgroup (CB = 2): shard products of up to a few hundred rows, which in the
// persistent kernel's tiles are too few to fill the chip or too short to pay for its fixed costs (its prologue, hand-over
// and flag take 3 us more than this kernel's; sharing K out over programs 4 to 6 us).  Here the eight waves share K
// inside the workgroup.  A comes in like B, by LDS-DMA, two blocks a wave in flight: 8 KiB a block of K, 128 KiB a
// workgroup, one workgroup a CU.  64 of K take 0.08 us, 0.09 on all CUs at once ([512,512], 256 workgroups: 9.0 us at K =
// 1024, 61 at 36864), and 0.048 with 112 workgroups whose operands the L2s hold.  No one unit bounds it: at [128,1376], 172 workgroups,
// a CU's L1 takes 0.73 accesses of 64 bytes a clock, an XCD's L2 gives 2.4 TB/s, half of what its channels can, and 23 % of
// its requests miss it (operands changed from launch to launch; counters at K = 4096 and 8192).
// A lane's columns are eight in a row: the block j of a row of 32 columns takes columns 8q + 4j .. + 3, so that a row
// leaves in 16-byte stores.  The cells are dealt to the XCDs in consecutive runs (the shorter direction first), so that
// each XCD's L2 fetches its share of the longer operand once.
constexpr int CELL = 32;
// LDS of a workgroup of RB x 2 blocks
constexpr int cells_lds_bytes(int rb) { return SKINNY_WAVES * SKINNY_UN * (rb + 2) * SKINNY_BLOCK_BYTES; }

// (REDUCE) four columns of the result's row m, from column n on, written through like the reference's store (".wt").
__device__ __attribute__((always_inline)) inline void store_result4(const GemmKArgs& p, int m, int n, f32x4 s) {
  const bool f32 = p.cg_dt == IRIS_DTYPE_F32, bf16 = p.cg_dt == IRIS_DTYPE_BF16;
  IRIS_GLOBAL char* d = (IRIS_GLOBAL char*)p.cg + ((int64_t)m * p.sgm + n) * (f32 ? 4 : 2);
  const u32x4 wide = __builtin_bit_cast(u32x4, s);
  const u32x2 half = bf16 ? u32x2{pack2<IRIS_DTYPE_BF16>(s[0], s[1]), pack2<IRIS_DTYPE_BF16>(s[2], s[3])}
                          : u32x2{pack2<IRIS_DTYPE_F16>(s[0], s[1]), pack2<IRIS_DTYPE_F16>(s[2], s[3])};
  if (n + 4 <= p.N) {
    if (f32 && p.sys)
      store16_any<AUX_SC0 | AUX_SC1>(d, wide);
    else if (f32)
      store16_any<AUX_SC1>(d, wide);
    else if (p.sys)
      store8_any<AUX_SC0 | AUX_SC1>(d, half);
    else
      store8_any<AUX_SC1>(d, half);
    return;
  }
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    if (n + e >= p.N) continue;
    if (f32)
      store_through((IRIS_GLOBAL unsigned int*)d + e, wide[e], p.sys != 0);
    else
      store_through((IRIS_GLOBAL unsigned short*)d + e, (unsigned short)(half[e / 2] >> (16 * (e & 1))), p.sys != 0);
  }
}

// The word of the shader engine that this workgroup runs on (late_tiles.hpp).
__device__ inline IRIS_GLOBAL int32_t* late_word(const GemmKArgs& p) {
  // (hwreg(HW_REG_HW_ID, 13, 3) and hwreg(HW_REG_XCC_ID, 0, 4))
  const int engine = __builtin_amdgcn_s_getreg(4 | 13 << 6 | (3 - 1) << 11), xcd = __builtin_amdgcn_s_getreg(20 | (4 - 1) << 11);
  return (IRIS_GLOBAL int32_t*)(p.tile_arrivals + ((xcd << 2 | (engine & 3)) & (LATE_ENGINES - 1)));
}

// Compare-and-swap that orders what this workgroup and the one it meets here have stored: `word` as it was.
__device__ inline int32_t late_swap(IRIS_GLOBAL int32_t* at, int32_t word, int32_t to) {
  __hip_atomic_compare_exchange_strong(at, &word, to, __ATOMIC_ACQ_REL, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
  return word;
}

// One lane, for a tile whose peers are late: whether this workgroup waits for it (else one that waits already takes it).
__device__ inline bool late_tile_enter(const GemmKArgs& p, int tile) {
  if (p.tile_arrivals == nullptr) return true;  // (as many as may wait have a tile each)
  IRIS_GLOBAL int32_t *at = late_word(p), *link = (IRIS_GLOBAL int32_t*)(p.locks + tile);
  const int most = late_most(p.ws);
  int32_t word = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  for (;;) {
    const bool waits = late_waits(word, most);
    if (!waits) __hip_atomic_store(link, late_left(word), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int32_t seen = late_swap(at, word, late_join(word, most, tile));
    if (seen == word) return waits;
    word = seen;
    if (!waits) __hip_atomic_store(link, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
}

// One lane, done with a late tile: the next one (plus one), or zero.
__device__ inline int late_tile_next(const GemmKArgs& p) {
  IRIS_GLOBAL int32_t* at = late_word(p);
  int32_t word = __hip_atomic_load(at, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_AGENT);
  for (;;) {
    const int tile = late_left(word);
    IRIS_GLOBAL int32_t* link = (IRIS_GLOBAL int32_t*)(p.locks + (tile ? tile - 1 : 0));
    const int32_t before = tile ? __hip_atomic_load(link, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0;
    const int32_t seen = late_swap(at, word, late_next(word, before));
    if (seen == word) {
      if (tile) __hip_atomic_store(link, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
      return tile;
    }
    word = seen;
  }
}

// AROWS: rows of A in a block, 8 or 16.
// RB: blocks of 16 rows a workgroup computes (1 for up to 32 rows; 2 up to 64
// rows of a long K, and from 17 rows on where B is large).
// CB: blocks of 16 columns, 1 or (cells: with RB 2, or a row-major B) 2.
// LOOSE: operands along K at any alignment and of any K from eight on (see Loader in gemm_kernel.hpp): a chunk that K cuts is
// fetched moved back to end there, and what it repeats is cleared in the fragments.  (us a pass, by the gathering tiles / so:
// [1,8229] x [8229,3816] 29.0 / 15.5, [15,2293] x [2293,1344] 17.0 / 9.8, [2,29690] x [29690,336] 22.3 / 11.8, [25,137] x
// [137,4864] and its reduce 17.2 / 16.8; 40 random calls of up to 32 rows 1.48x.)
// BROWS (cells, 16-bit operands): a B whose rows are its k (row-major [K, N]), in whole aligned 16-byte chunks.  A block of B lies
// in LDS as in memory, 64 k of 32 columns, and is transposed on its way to the MFMAs by ds_read_b64_tr_b16.  A row of 64
// bytes is half a cache line, so that such a block costs the L1 twice what one along K does, 1.5 times with a cell's 32 rows of
// A beside it ([95,4224] x [4224,1280] along K 9.7 us, so 12.8: 1.6 times what is above a launch's fixed 4.5).  With up to 16
// rows of A, RB is 1 ([4,1376] x [1376,4096] 8.0 -> 7.4 us, 27 random calls of 1 to 16 rows 1.08x, same bits; RB 2 fetched as many rows of A again,
// and for up to eight three times as many, all out of range).
// REDUCE (one-shot epilogue): the workgroup also reduces its block of C over all ranks.  Of its own rank's partial it needs
// what it has just computed, so it waits for no other workgroup; the peers' strips, where their signal is there by the
// last blocks of K, are fetched (wave w: rank w) under the last products and the exchange between the waves, and the sum is stored
// behind the partial.  A reduce kernel behind the product cost its launch, its gap (0.84 us) and a chain of flag, bases,
// partials and result of its own: [16,1376] x [1376,4096], 8 fp32 partials, fill of the flags included 13.2 -> 9.5 us; 64 random
// calls of up to 300 rows whose reduce is inside 1.24x, none slower.  Up to eight ranks, a wave each; where peers are late, few
// workgroups wait (late_tiles.hpp).
template <int DT, int OP, int ODT, int AROWS, int RB = 1, int CB = 1, bool LOOSE = false, bool BROWS = false, bool REDUCE = false>
__global__ __launch_bounds__(SKINNY_THREADS) __attribute__((amdgpu_waves_per_eu(2, 8))) void
gemm_skinny_kernel(const GemmKArgs p) {
  constexpr bool ATOMIC = OP == OP_ATOMIC32 || OP == OP_ATOMIC16;
  constexpr bool F32 = OP == OP_STORE32 || OP == OP_ATOMIC32;
  constexpr int UN = SKINNY_UN, AH = AROWS / 8;  // fetches of a block of A
  static_assert(AROWS == 16 || (AROWS == 8 && RB == 1), "rows of a block of A");
  static_assert(RB == 1 || RB == 2, "blocks of rows per workgroup");
  static_assert(CB == 1 || (CB == 2 && ((RB == 2 && AROWS == 16) || BROWS)), "blocks of columns per workgroup");
  static_assert(!REDUCE || !ATOMIC, "the one-shot epilogue stores");
  static_assert(!BROWS || (CB == 2 && !LOOSE && DT != IRIS_DTYPE_F32), "B by rows of k: cells of 16-bit operands");
  constexpr bool A_DMA = CB == 2;  // A in LDS, UN blocks a wave, like B
  constexpr int NB = RB * CB;
  using vec8 = typename Mfma<DT>::vec8;
  extern __shared__ __attribute__((aligned(1024))) char skinny_lds[];
  touch_args<sizeof(GemmKArgs)>();
  IRIS_LDS char* lds = (IRIS_LDS char*)skinny_lds;
  // each wave's blocks of A ([SKINNY_WAVES][RB][64] partial accumulators at the end), then each wave's UN blocks of B
  IRIS_LDS f32x4* red = (IRIS_LDS f32x4*)lds;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int lr = lane & 15, lq = lane >> 4;
  int bx = blockIdx.x, by = blockIdx.y;  // the workgroup's block of columns and of rows
  int cell = by * gridDim.x + bx;
  if constexpr (CB == 2) {
    const int round = (int)fast_div((uint32_t)bx, p.div_xcd);
    cell = (bx - round * p.num_xcds) * p.xcd_per + round;
    if (cell >= p.cells) return;
    const int outer = (int)fast_div((uint32_t)cell, p.div_inner), inner = cell - outer * p.cells_inner;
    bx = p.cells_by_row ? inner : outer;
    by = p.cells_by_row ? outer : inner;
  }
  const int n0 = bx * (SKINNY_COLS * CB);
  const int m0 = by * (SKINNY_ROWS * RB);
  IRIS_LDS char* wb = lds + (A_DMA ? SKINNY_WAVES * UN * RB * SKINNY_BLOCK_BYTES : skinny_a_bytes(RB)) + wave * (UN * CB * SKINNY_BLOCK_BYTES);
  IRIS_LDS char* wa = lds + wave * ((A_DMA ? UN : 1) * RB * SKINNY_BLOCK_BYTES);

  // Rows past the edge of either operand lie past the end of its buffer
  // descriptor and read as zero; chunks past K are parked out of range.
  constexpr int LEAD = LOOSE ? 16 : 0;  // (no offset of a chunk moved back is below zero)
  const int rows_b = min(SKINNY_COLS * CB, p.N - n0);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.b + (int64_t)n0 * p.sbn * 2 - LEAD), 0,
      (int)((BROWS ? ((int64_t)p.K - 1) * p.sbk + rows_b : ((int64_t)rows_b - 1) * p.sbn + p.K) * 2) + LEAD, 0x00020000);
  const int rows_a = min(SKINNY_ROWS * RB, p.M - m0);
  const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(p.a + (int64_t)m0 * p.sam * 2 - LEAD), 0, (int)((((int64_t)rows_a - 1) * p.sam + p.K) * 2) + LEAD, 0x00020000);
  // B: lane l of fetch j of a block brings row 8j + l/8 and lands at byte
  // l*16 of the fetch's 1 KiB, i.e. at physical chunk l%8 of that row; the
  // chunk of the row it must bring there is (l%8) ^ (row/2 % 8).
  // (CB 2: row 16j + r of the block's 32 holds column 8 (r / 4) + 4j + r % 4)
  const int brow = lane >> 3;  // + 8j
  auto b_column = [&](int j) {
    if constexpr (CB == 1) return brow + 8 * j;
    const int r = brow + 8 * (j & 1);
    return (r >> 2) * 8 + (j >> 1) * 4 + (r & 3);
  };
  const int bchunk = (lane & 7) ^ ((brow >> 1) & 7);  // rows 8j + .. : (row/2)%8 = 4j + brow/2, and 4j flips bit 2
  // A comes in the same way, but into registers, and then goes through a 2 KiB
  // region of the wave, laid out like a block of B, on its way to the MFMAs.
  // (With AROWS 8 the upper half of that region is never written; rows of the
  // product do not mix and those are not stored.)
  // The operand reads: lane l holds row l%16.  In K block kb, MFMA h (0, 1)
  // takes k = kb*64 + (l/16)*16 + h*8 .. +7 at MFMA position (l/16)*8 .. +7:
  // the same permutation of k for both operands.
  const int nb_all = (p.K + 63) / 64;
  // the blocks of K of this workgroup
  const int share = (nb_all + (int)gridDim.z - 1) / (int)gridDim.z;
  const int kb0 = blockIdx.z * share;
  const int nb = min(nb_all, kb0 + share);

  f32x4 acc[NB];  // [row block][column block]
#pragma unroll
  for (int i = 0; i < NB; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};

  u32x4 va[A_DMA ? 1 : UN][RB][AH];
  // bytes by which chunk ch of K block kb is moved back
  auto back = [&](int kb, int ch) __attribute__((always_inline)) -> uint32_t {
    return LOOSE ? (uint32_t)max(0, kb * 64 + ch * 8 + 8 - p.K) * 2 : 0u;
  };
  // fetches of K block kb into set u (blocks past the end are parked: the number of loads never changes)
  auto fetch = [&](int u, int kb) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 2 * CB; ++j) {
      if constexpr (BROWS) {
        // lane l of fetch j: columns 8 (l % 4) .. + 7 of k 16j + l / 4 (N is a multiple of eight: inside the matrix or past it)
        const int k = kb * 64 + 16 * j + (lane >> 2), col = (lane & 3) * 8;
        const bool ok = kb < nb && k < p.K && col < rows_b;
        lds_dma16(rb, wb + u * (CB * SKINNY_BLOCK_BYTES) + j * 1024, ok ? (uint32_t)(((int64_t)k * p.sbk + col) * 2) : 0x80000000u, 0);
        continue;
      }
      const int ch = bchunk ^ ((j & 1) << 2);
      const bool ok = kb < nb && kb * 64 + ch * 8 < p.K;
      const uint32_t off = (uint32_t)(((int64_t)b_column(j) * p.sbn) * 2 + kb * 128 + ch * 16) + LEAD - back(kb, ch);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(rb, (IRIS_LDS void*)(wb + u * (CB * SKINNY_BLOCK_BYTES) + j * 1024), 16,
                                               ok ? (int)off : (int)0x80000000, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < RB; ++i)
#pragma unroll
      for (int j = 0; j < AH; ++j) {
        const int ch = bchunk ^ (j << 2);
        const bool ok = kb < nb && kb * 64 + ch * 8 < p.K;
        const uint32_t off = (uint32_t)(((int64_t)(i * 16 + brow + 8 * j) * p.sam) * 2 + kb * 128 + ch * 16) + LEAD - back(kb, ch);
        if constexpr (BROWS)
          lds_dma16(ra, wa + (u * RB + i) * SKINNY_BLOCK_BYTES + j * 1024, ok ? off : 0x80000000u, 0);
        else if constexpr (A_DMA)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              ra, (IRIS_LDS void*)(wa + (u * RB + i) * SKINNY_BLOCK_BYTES + j * 1024), 16, ok ? (int)off : (int)0x80000000, 0, 0, 0);
        else
          va[u][i][j] = __builtin_amdgcn_raw_buffer_load_b128(ra, ok ? (int)off : (int)0x80000000, 0, 0);
      }
  };
  auto multiply = [&](int u, int kb) __attribute__((always_inline)) {
    // (the wave's LDS operations execute in order: these writes land after
    // the previous block's reads and before this block's)
    if constexpr (!A_DMA) {
#pragma unroll
      for (int i = 0; i < RB; ++i)
#pragma unroll
        for (int j = 0; j < AH; ++j)
          *reinterpret_cast<IRIS_LDS u32x4*>(wa + i * SKINNY_BLOCK_BYTES + j * 1024 + lane * 16) = va[u][i][j];
    }
    const IRIS_LDS char* sa = wa + (A_DMA ? u * (RB * SKINNY_BLOCK_BYTES) : 0);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int pc = (lq * 2 + h) ^ ((lr >> 1) & 7);
      vec8 fb[CB];
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        if constexpr (BROWS) {
          // Each 16 lanes read four k of the 16 columns of block j, lane l four of them of k l / 4: those of its own
          // chunk (l % 4) that are block j's.  They are handed out so that lane l holds the four k of the block's column l.
          // Twice, four k apart.  (Two of the wave's quarters meet on the same banks: 8 reads of 16 clocks a block, beside 270
          // that its fetches take.)
          typedef short s16x4 __attribute__((ext_vector_type(4)));
          const IRIS_LDS char* at = wb + u * (CB * SKINNY_BLOCK_BYTES) + (lq * 16 + h * 8 + (lr >> 2)) * 64 + (lr & 3) * 16 + j * 8;
          const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((IRIS_LDS s16x4*)at);
          const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((IRIS_LDS s16x4*)(at + 4 * 64));
          fb[j] = __builtin_bit_cast(vec8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
        } else {
          fb[j] = *reinterpret_cast<const IRIS_LDS vec8*>(wb + (u * CB + j) * SKINNY_BLOCK_BYTES + lr * 128 + pc * 16);
        }
      }
      const bool cut = LOOSE && (p.K & 7) != 0 && kb == nb_all - 1;
      const int front = lq * 2 + h == (p.K & 63) / 8 ? 8 - (p.K & 7) : 0;
      if (cut)
#pragma unroll
        for (int j = 0; j < CB; ++j) mask_tail<DT>(fb[j], front);
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        vec8 fa = *reinterpret_cast<const IRIS_LDS vec8*>(sa + i * SKINNY_BLOCK_BYTES + lr * 128 + pc * 16);
        if (cut) mask_tail<DT>(fa, front);
#pragma unroll
        for (int j = 0; j < CB; ++j) acc[i * CB + j] = Mfma<DT>::run(fb[j], fa, acc[i * CB + j]);
      }
    }
  };
  constexpr int LOADS = 2 * CB + AH * RB;  // a block's
  static_assert(LOADS * (UN - 1) <= 63, "vmcnt immediate");
  int b0 = kb0 + wave;
#pragma unroll
  for (int u = 0; u < UN; ++u) {
    fetch(u, b0 + SKINNY_WAVES * u);
    asm volatile("" ::: "memory");  // (the blocks' loads stay in this order: the waits below count them)
  }
  touch_line(p.heap_bases);  // (read by the stores)
  constexpr int ES = F32 ? 4 : 2;
  // (REDUCE) the tile that the block belongs to, and its flag as it is now
  int tile_id = 0, flag_now = 0;
  // (REDUCE) this lane's columns of each block of rank r's partial, element by element where N ends inside the four
  u32x4 strip[REDUCE ? NB : 1];
  auto fetch_strips = [&](int r) __attribute__((always_inline)) {
    const int cols = min(SKINNY_COLS * CB, p.N - n0);
    IRIS_GLOBAL char* base = rank_ptr(p, p.out, r) + ((int64_t)m0 * p.som + n0) * ES;
    const __amdgpu_buffer_rsrc_t rs =
        __builtin_amdgcn_make_buffer_rsrc((void*)base, 0, (int)((((int64_t)rows_a - 1) * p.som + cols) * ES), 0x00020000);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int row = (b / CB) * 16 + lr, col = lq * (4 * CB) + 4 * (b % CB);
      const uint32_t off = row < rows_a && col + 4 <= cols ? (uint32_t)(((int64_t)row * p.som + col) * ES) : DEAD_OFFSET;
      if constexpr (F32) {
        strip[b] = p.sys ? __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, AUX_SC0 | AUX_SC1)
                         : __builtin_amdgcn_raw_buffer_load_b128(rs, (int)off, 0, AUX_SC1);
      } else {
        const u32x2 x = p.sys ? __builtin_amdgcn_raw_buffer_load_b64(rs, (int)off, 0, AUX_SC0 | AUX_SC1)
                              : __builtin_amdgcn_raw_buffer_load_b64(rs, (int)off, 0, AUX_SC1);
        strip[b] = u32x4{x[0], x[1], 0u, 0u};
      }
      if (row < rows_a && col < cols && col + 4 > cols) {
        const IRIS_GLOBAL char* at = base + ((int64_t)row * p.som + col) * ES;
        strip[b] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int e = 0; e < 3; ++e) {
          if (col + e >= cols) continue;
          if constexpr (F32)
            strip[b][e] = load_through((const IRIS_GLOBAL unsigned int*)at + e, p.sys != 0);
          else
            strip[b][e / 2] |= (unsigned int)load_through((const IRIS_GLOBAL unsigned short*)at + e, p.sys != 0) << (16 * (e & 1));
        }
      }
    }
  };
  auto flag_of = [&]() __attribute__((always_inline)) { return (IRIS_GLOBAL int32_t*)(p.flags + tile_id); };
  if constexpr (REDUCE) {
    tile_id = tile_id_of(m0 / p.BM, n0 / p.BN, p.num_pid_m, p.num_pid_n, p.G);
    flag_now = load_through(flag_of(), p.sys != 0);
  }
  // A long range of K: as a block has been read its place takes the one UN further on, so that the fetches in
  // flight never run dry (B has landed in this wave's own region once the wave's counter says so: nobody else
  // reads or writes it).
  for (; b0 + SKINNY_WAVES * UN < nb; b0 += SKINNY_WAVES * UN) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      IRIS_WAIT_VMCNT(LOADS * (UN - 1));
      asm volatile("" ::: "memory");
      multiply(u, b0 + SKINNY_WAVES * u);
      IRIS_WAIT_LGKMCNT0();  // the reads have returned before the next fetch overwrites the region
      asm volatile("" ::: "memory");
      fetch(u, b0 + SKINNY_WAVES * (UN + u));
    }
  }
  // the last blocks: the loads behind them are all on their way
  IRIS_WAIT_VMCNT(0);
  asm volatile("" ::: "memory");
  // (REDUCE, K of one group) peers that are done: wave w fetches the strips of rank w, which arrive under the last products
  // and the exchange behind them
  bool peers_done = false;
  if constexpr (REDUCE) {
    peers_done = gridDim.z == 1 && __builtin_amdgcn_readfirstlane(flag_now) >= p.ws - 1;
    if (peers_done) {
      if (p.flag_mode & FLAG_RELEASE) acquire_at(p.sys != 0);
      if (wave < p.ws && wave != p.cur_rank) fetch_strips(wave);
    }
  }
#pragma unroll
  for (int u = 0; u < UN; ++u) multiply(u, b0 + SKINNY_WAVES * u);
  IRIS_WAIT_LGKMCNT0();
  asm volatile("" ::: "memory");

  // acc[i]: row m = i*16 + l%16 of the workgroup's rows, columns 4*(l/16) .. +3 (operands swapped, as in the
  // persistent kernel).  The waves' partial sums meet in LDS, [wave][block][lane].
  // (REDUCE: a wave's own region of B, which it has read, takes its strips and whether it saw the flag)
  if constexpr (REDUCE) {
    if (lane == 0) *(IRIS_LDS int*)(wb + NB * 1024) = peers_done;
  }
  __syncthreads();  // every wave is done with its blocks of A: the region becomes `red`
#pragma unroll
  for (int i = 0; i < NB; ++i) red[(wave * NB + i) * 64 + lane] = acc[i];
  __syncthreads();
  if constexpr (NB > 1) {
    // With several blocks every destination's wave would add up all of them:
    // first each block is summed once, in wave order, by the 8 / NB waves that
    // share it (a part of the lanes each), and left in the first wave's place.
    constexpr int WPB = SKINNY_WAVES / NB, LPW = 64 / WPB;  // waves per block, lanes of a block per wave
    const int blk = wave / WPB, l0 = (wave % WPB) * LPW;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    const bool mine = lane >= l0 && lane < l0 + LPW;
    if (mine) {
      s = red[blk * 64 + lane];
#pragma unroll
      for (int w = 1; w < SKINNY_WAVES; ++w) s += red[(w * NB + blk) * 64 + lane];  // wave order
    }
    __syncthreads();  // all partial sums have been read
    if (mine) red[blk * 64 + lane] = s;
    __syncthreads();
  }

  if constexpr (REDUCE) {
    const int seen = lane < SKINNY_WAVES ? *(IRIS_LDS int*)(wb + (lane - wave) * (UN * CB * SKINNY_BLOCK_BYTES) + NB * 1024) : 1;
    if (peers_done && __ballot(seen == 0) != 0) peers_done = false;
  }
  const bool split = gridDim.z > 1;
  if (split) {
    // K shared out over gridDim.z groups: each leaves its sum in `partials` (register order, 1 KiB a block), and
    // the last to arrive at the blocks' counter adds all of them up, in the order of K, and goes on to the
    // stores.  Nobody waits: any number of the groups can be resident.
    const uint32_t span = (uint32_t)(CB == 2 ? p.cells : (int)(gridDim.x * gridDim.y)) * (NB * 1024);  // bytes of one share's sums
    IRIS_LDS int* is_last = (IRIS_LDS int*)(lds + NB * 1024);  // (behind the blocks' sums)
    if (wave == 0) {
      f32x4 s[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        s[b] = red[b * 64 + lane];
        if constexpr (NB == 1) {
#pragma unroll
          for (int w = 1; w < SKINNY_WAVES; ++w) s[b] += red[w * 64 + lane];
        }
      }
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
          (void*)p.partials, 0, (int)(span * gridDim.z), 0x00020000);
#pragma unroll
      for (int b = 0; b < NB; ++b)
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, s[b]), rs,
                                               (int)(blockIdx.z * span + (cell * NB + b) * 1024 + lane * 16), 0, AUX_SC1);
      IRIS_WAIT_VMCNT(0);
      asm volatile("" ::: "memory");
      IRIS_GLOBAL int32_t* cnt = (IRIS_GLOBAL int32_t*)(p.locks + p.total_tiles + cell);
      int last = 0;
      if constexpr (REDUCE) flag_now = load_through(flag_of(), p.sys != 0);
      if (lane == 0) {
        last = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == (int)gridDim.z - 1;
        if (last) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
      }
      last = __builtin_amdgcn_readfirstlane(last);
      asm volatile("" ::: "memory");
      if (last) {
        constexpr int G = 8 / NB;  // shares in flight
#pragma unroll
        for (int b = 0; b < NB; ++b) s[b] = f32x4{0.f, 0.f, 0.f, 0.f};
        for (int z0 = 0; z0 < (int)gridDim.z; z0 += G) {
          u32x4 v[G][NB];
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int b = 0; b < NB; ++b)  // (shares past the last lie past the descriptor: zero)
              v[g][b] = __builtin_amdgcn_raw_buffer_load_b128(
                  rs, (int)((z0 + g) * span + (cell * NB + b) * 1024 + lane * 16), 0, AUX_SC1);
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int b = 0; b < NB; ++b) s[b] += __builtin_bit_cast(f32x4, v[g][b]);
        }
#pragma unroll
        for (int b = 0; b < NB; ++b) red[b * 64 + lane] = s[b];
      }
      if (lane == 0) *is_last = last | (REDUCE && flag_now >= p.ws - 1 ? 2 : 0);
    }
    __syncthreads();
    const int found = *is_last;
    if (!(found & 1)) return;
    if constexpr (REDUCE) {
      peers_done = (__builtin_amdgcn_readfirstlane(found) & 2) != 0;
      if (peers_done) {
        if (p.flag_mode & FLAG_RELEASE) acquire_at(p.sys != 0);
        if (wave < p.ws && wave != p.cur_rank) fetch_strips(wave);
      }
    }
  }

  const int r_begin = p.dest_all ? 0 : p.cur_rank;
  const int r_end = p.dest_all ? p.ws : p.cur_rank + 1;
  // four columns of a row, from column n on
  auto store4 = [&](IRIS_GLOBAL char* dst, int m, int n, f32x4 s) __attribute__((always_inline)) {
    if constexpr (ATOMIC) {
      // 08: add into the destination (gemm_atomics_all_reduce.py:236-248)
      if constexpr (OP == OP_ATOMIC16) {
        if (p.row_out) {
          const int valid = min(4, p.N - n);
          atomic_add16_strip<ODT>(dst + ((int64_t)m * p.som + n) * ES, s, valid, n > 0, n + valid < p.N);
          return;
        }
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n + e >= p.N) continue;
        IRIS_GLOBAL char* d = dst + ((int64_t)m * p.som + (int64_t)(n + e) * p.son) * ES;
        const float f = s[e];
        if constexpr (OP == OP_ATOMIC32)
          __hip_atomic_fetch_add((IRIS_GLOBAL float*)d, f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else
          atomic_add16_cas<ODT>((IRIS_GLOBAL unsigned short*)d, from16<ODT>(to16<ODT>(f)));
      }
    } else if (p.row_out && n + 4 <= p.N) {
      // four columns in one store (at any address: rows of an odd length are no exception)
      IRIS_GLOBAL char* d = dst + ((int64_t)m * p.som + n) * ES;
      if constexpr (F32) {
        const u32x4 v = __builtin_bit_cast(u32x4, s);
        if (p.sys)
          store16_any<AUX_SC0 | AUX_SC1>(d, v);
        else
          store16_any<AUX_SC1>(d, v);
      } else {
        const u32x2 v = {pack2<ODT>(s[0], s[1]), pack2<ODT>(s[2], s[3])};
        if (p.sys)
          store8_any<AUX_SC0 | AUX_SC1>(d, v);
        else
          store8_any<AUX_SC1>(d, v);
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (n + e >= p.N) continue;
        IRIS_GLOBAL char* d = dst + ((int64_t)m * p.som + (int64_t)(n + e) * p.son) * ES;
        const float f = s[e];
        if constexpr (F32)
          store_through((IRIS_GLOBAL unsigned int*)d, __builtin_bit_cast(unsigned int, f), p.sys != 0);
        else
          store_through((IRIS_GLOBAL unsigned short*)d, to16<ODT>(s[e]), p.sys != 0);
      }
    }
  };
  if constexpr (REDUCE) {
    // One-shot epilogue with the reduce inside (gemm_one_shot_all_reduce.py:197-271).  Wave i stores block i of the rows to
    // this rank's partial; where the peers have signalled the tile, it adds all ranks' strips up, in rank order, and stores
    // the result: what the workgroup needs of its own rank it holds, so it waits for nobody.
    const int m = m0 + wave * 16 + lr, n = n0 + lq * (4 * CB);
    const bool mine = wave < RB && m < p.M && n < p.N;
    f32x4 own[CB], sum[CB];
    if (mine) {
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        own[j] = red[(wave * CB + j) * 64 + lane];
        if (NB == 1 && !split) {
#pragma unroll
          for (int w = 1; w < SKINNY_WAVES; ++w) own[j] += red[w * 64 + lane];  // wave order
        }
      }
#pragma unroll
      for (int j = 0; j < CB; ++j) {
        if (n + 4 * j < p.N) store4((IRIS_GLOBAL char*)p.out, m, n + 4 * j, own[j]);
        if constexpr (!F32) {
          // (what the partial holds is what is added)
#pragma unroll
          for (int e = 0; e < 4; ++e) own[j][e] = from16<ODT>(to16<ODT>(own[j][e]));
        }
      }
    }
    if (peers_done) {  // (up to eight ranks, a wave each)
      if (wave < p.ws && wave != p.cur_rank) {
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          f32x4 v = __builtin_bit_cast(f32x4, strip[b]);
          if constexpr (!F32)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = from16<ODT>((unsigned short)(strip[b][e / 2] >> (16 * (e & 1))));
          *reinterpret_cast<IRIS_LDS f32x4*>(wb + b * 1024 + lane * 16) = v;
        }
      }
      __syncthreads();
      if (mine) {
#pragma unroll
        for (int j = 0; j < CB; ++j) {
          f32x4 v[SKINNY_WAVES];  // (all on their way before the first is added)
#pragma unroll
          for (int q = 0; q < SKINNY_WAVES; ++q)
            v[q] = *reinterpret_cast<const IRIS_LDS f32x4*>(wb + (q - wave) * (UN * CB * SKINNY_BLOCK_BYTES) + (wave * CB + j) * 1024 +
                                                            lane * 16);
          sum[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int q = 0; q < SKINNY_WAVES; ++q)
            if (q < p.ws) sum[j] += q == p.cur_rank ? own[j] : v[q];
        }
#pragma unroll
        for (int j = 0; j < CB; ++j)
          if (n + 4 * j < p.N) store_result4(p, m, n + 4 * j, sum[j]);
      }
    }
  } else {
  // (rank, row block) pairs over the waves
  for (int it = wave; it < (r_end - r_begin) * RB; it += SKINNY_WAVES) {
    const int r = r_begin + it / RB, i = it % RB;
    const int m = m0 + i * 16 + lr, n = n0 + lq * (4 * CB);
    if (m >= p.M || n >= p.N) continue;
    IRIS_GLOBAL char* dst = rank_ptr(p, p.out, r);
    f32x4 s[CB];
#pragma unroll
    for (int j = 0; j < CB; ++j) s[j] = red[(i * CB + j) * 64 + lane];
    if (NB == 1 && !split) {
#pragma unroll
      for (int w = 1; w < SKINNY_WAVES; ++w) s[0] += red[w * 64 + lane];  // wave order: the sum does not depend on timing
    }
    if constexpr (CB == 2 && !ATOMIC && !F32) {
      if (p.row_out && n + 8 <= p.N) {
        IRIS_GLOBAL char* d = dst + ((int64_t)m * p.som + n) * ES;
        const u32x4 v = {pack2<ODT>(s[0][0], s[0][1]), pack2<ODT>(s[0][2], s[0][3]), pack2<ODT>(s[1][0], s[1][1]),
                         pack2<ODT>(s[1][2], s[1][3])};
        if (p.sys)
          store16_any<AUX_SC0 | AUX_SC1>(d, v);
        else
          store16_any<AUX_SC1>(d, v);
        continue;
      }
    }
#pragma unroll
    for (int j = 0; j < CB; ++j)
      if (n + 4 * j < p.N) store4(dst, m, n + 4 * j, s[j]);
  }
  }
  if (p.flag_mode == 0) return;

  // The stores were write-through at the flags' scope: once every wave has
  // seen its own complete, the group's part of the tile is visible there.
  const int pid_m = m0 / p.BM, pid_n = n0 / p.BN;
  int parts = 0;  // (REDUCE) workgroups that share the tile, counted while the stores complete
  if constexpr (REDUCE) {
    constexpr int COLS = SKINNY_COLS * CB, ROWS = SKINNY_ROWS * RB;
    const int cols = min(p.N, (pid_n + 1) * p.BN) - pid_n * p.BN, rows = min(p.M, (pid_m + 1) * p.BM) - pid_m * p.BM;
    parts = ((cols + COLS - 1) / COLS) * ((rows + ROWS - 1) / ROWS);
    asm volatile("" : "+s"(parts));
  }
  IRIS_WAIT_VMCNT(0);
  __syncthreads();
  if constexpr (REDUCE) {
    // Two counts in the tile's word: the workgroups that have stored, and those of them that have reduced.  The last to
    // arrive signals the peers and, where all have reduced, consumes the flag (CAS(ws-1 -> 0), :220-234).  Else it waits for
    // the flag and reduces the tile itself, or leaves the tile to one that waits already (late_tiles.hpp).
    IRIS_LDS int* todo = (IRIS_LDS int*)lds;
    if (wave == 0) {
      int stored = 1, reduced = peers_done ? 1 : 0;
      if (parts > 1) {
        IRIS_GLOBAL int32_t* cnt = (IRIS_GLOBAL int32_t*)(p.locks + tile_id);
        int before = 0;
        if (lane == 0) before = arrive(cnt, (p.flag_mode & FLAG_RELEASE) != 0, p.sys != 0, 1 + (reduced << 16));
        before = __builtin_amdgcn_readfirstlane(before);
        stored += before & 0xFFFF;
        reduced += before >> 16;
        if (stored == parts && lane == 0) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
      }
      int late = 0;
      if (stored == parts) {
        publish_tile(p, tile_id, lane);
        if (lane == 0) {
          if (__builtin_expect(reduced < parts, 0))
            late = late_tile_enter(p, tile_id) ? tile_id + 1 : 0;
          else
            flag_add_relaxed(flag_of(), 1 - p.ws, p.sys != 0);
        }
      }
      if (lane == 0) *todo = late;
    }
    __syncthreads();
    // (the arguments are read here, from the argument block: held in scalar registers up to here they push others out)
    typedef const __attribute__((address_space(4))) GemmKArgs* KernArgPtr;
    KernArgPtr late_args = (KernArgPtr)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(late_args));
    const GemmKArgs& q = *(const GemmKArgs*)late_args;
    bool gone = false;  // (a peer that has not come within the bound: what it has not signalled is not waited for again)
    for (int late = __builtin_amdgcn_readfirstlane(*todo); __builtin_expect(late != 0, 0);) {
      __syncthreads();  // (`todo` has been read)
      if (tid == 0)
        *todo = wait_tile_flag((IRIS_GLOBAL int32_t*)(q.flags + late - 1), q.ws, q.sys != 0, gone ? 0 : q.timeout, q.status);
      __syncthreads();
      if (__builtin_amdgcn_readfirstlane(*todo)) {
        const TileCoord t = tile_map(late - 1, q.num_pid_m, q.num_pid_n, q.G);
        Item it{};
        it.lm0 = t.pid_m * q.BM;
        it.ln0 = t.pid_n * q.BN;
        it.m_end = min(q.M, it.lm0 + q.BM);
        it.n_end = min(q.N, it.ln0 + q.BN);
        constexpr int IN_DT = F32 ? IRIS_DTYPE_F32 : ODT;
        if (q.sys)
          fused_reduce_tile<IN_DT, SKINNY_THREADS, 1, true>(q, it, tid);
        else
          fused_reduce_tile<IN_DT, SKINNY_THREADS, 1, false>(q, it, tid);
      } else {
        gone = true;
      }
      if (q.tile_arrivals == nullptr) break;
      __syncthreads();
      if (tid == 0) *todo = late_tile_next(q);
      __syncthreads();
      late = __builtin_amdgcn_readfirstlane(*todo);
    }
    return;
  }
  if (wave == 0) {
    const int tile_id = tile_id_of(pid_m, pid_n, p.num_pid_m, p.num_pid_n, p.G);
    const int cols = min(p.N, (pid_n + 1) * p.BN) - pid_n * p.BN, rows = min(p.M, (pid_m + 1) * p.BM) - pid_m * p.BM;
    constexpr int COLS = SKINNY_COLS * CB;
    const int parts = ((cols + COLS - 1) / COLS) * ((rows + SKINNY_ROWS * RB - 1) / (SKINNY_ROWS * RB));
    int last = 1;
    if (parts > 1) {
      IRIS_GLOBAL int32_t* cnt = (IRIS_GLOBAL int32_t*)(p.locks + tile_id);
      if (lane == 0) {
        last = arrive(cnt, (p.flag_mode & FLAG_RELEASE) != 0, p.sys != 0) == parts - 1;
        if (last) __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // for the next launch
      }
      last = __builtin_amdgcn_readfirstlane(last);
    }
    if (last) publish_tile(p, tile_id, lane);
  }
}

// The kernel for (operand type, store op, rows of A in a block, blocks of rows and of columns a workgroup), or null.
// `loose`: for operands at any alignment.  `b_rows` (cells): for a row-major B.
// `reduce`: the build that also reduces (the one-shot epilogue).
GemmKernelFn gemm_skinny_kernel_for(int dt, int op, int arows, int rb, int cb, bool loose, bool b_rows, bool reduce);

}  // namespace iris_amd
