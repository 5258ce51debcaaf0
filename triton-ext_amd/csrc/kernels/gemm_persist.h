// Persistent 4-wavefront GEMM for aligned operands whose K is a whole number
// of 128-byte steps (KTAIL, 16-bit operands: rows 4-byte aligned, any K of
// at least two steps, read as fast::KTail describes, and C rows of any
// alignment): one workgroup per CU walks its share of the BM x BN tiles
// (256 x 256; 128 x 128 or 64 x 64 for products with fewer 256 x 256 / 128 x 128 tiles
// than CUs),
// and the LDS-DMA pipeline of gemm_fast.h runs as one continuous
// stream of (tile, K step) pairs, so the first steps of the next tile are
// loaded while the current one finishes and no tile pays a pipeline fill.
//
// Layout per workgroup: 4 wavefronts (one per SIMD) in a 2 x 2 grid, each
// owning a quarter of the tile; its accumulator blocks of 16 x 16
// (256 x 256: 64 blocks, 256 registers) live in AGPRs.  Against the
// 8-wavefront tile this reads a third less from LDS per MFMA, which the power-
// limited clock turns into speed.
//
// MFMA shape: 16x16x32 (16-bit) and 16x16x128 (fp8), not 32x32x16 / 32x32x64.
// The large products are bound by the clock the power limit leaves, and the
// 16 x 16 forms, which read and write a quarter of the accumulator per
// instruction and sum twice the K, do the same work on less: register-only
// loops on N(0,1) operands sustain 2025 against 1765 TFLOP/s (bf16) and 4360
// against 3970 (fp8).  In this kernel (32 x 32 -> 16 x 16, same box): fp16
// 4096^3 row-major B 107 -> 102 us (clock 1.75 -> 2.00 GHz, MFMA busy 64 ->
// 60%), bf16 8192^3 764 -> 721 us, 2048^3 (128 x 128) 22.8 -> 21.6 us, fp8
// 8192^3 370 -> 361 us.  Without the LDS-DMA stream (timing only) these take
// 93, 628, 19.5 and 300 us: what binds them now is that stream's power and
// its delivery, not MFMA issue (staggering reads and loads, or forcing the
// accumulators in place, moves nothing beyond 1%).
//
// The K loop is that of gemm_fast_tile_at (ring of 5 LDS slots of 256 x 128 bytes,
// B of step s+2 and A of step s+3 loaded during the second half of step s; smaller
// tiles: D stages of a whole step, both of step s+D,
// fragments one 64-byte half ahead in registers, one barrier per step), with
// s counting steps over all tiles of the workgroup.  Each operand's loads go
// through a buffer resource for the tile they belong to: base at the tile's
// first row, range ending after its last valid row, so rows past M / N read
// as zero; steps past the workgroup's last tile use an empty range.
//
// Tile order: the tiles of the transposed grid in the XCD-contiguous order of
// tile_coords, so each XCD's round of 32 concurrent tiles covers 8 column
// panels (B), kept from one round to the next, and 4 row panels (A), new in
// every round.  With inputs that are not yet in the Infinity Cache the new
// panels come from HBM, and A, loaded three steps ahead, hides that latency
// where B, two steps ahead, did not (8192^3 fp8 from HBM-resident inputs:
// 2530 -> 2290 cycles per K step; 2146 with cached inputs either way).
//
// Epilogue: the scales load just before the tile's last K step, whose loads of
// one operand (A; of 128 x 256 tiles B) are deferred so that their LDS slot
// stages the output: per 32 rows of 16 x 16 blocks the accumulators are scaled
// and rounded to bf16 / fp16 (RNE), a lane's 4 columns of a row 8 bytes in LDS;
// each wave writes its 32 x BN / 2 block to its own quarter of that slot, reads
// back whole rows (BN = 256: 4 of 256 bytes) per instruction and stores them
// through a buffer resource for C (stores past M / N are dropped).  OUT_F32 (tt.dot with its
// accumulator operand): D = A.B + C in fp32 is written straight from the
// accumulators, C's loads for the first row blocks issued before the last K
// step.  EPI: the fp8 dot's fused epilogue, likewise from the accumulators.  The first K step of each
// tile starts its MFMAs from a zero accumulator operand, so the accumulators
// are never cleared explicitly.
#pragma once

#include "gemm_fast.h"

namespace txg {

namespace persist {
constexpr int kWaves = 4;

// Chunk swizzle of a K-major B slot (row-major K x N operand) for K row k, by
// k mod 4 and bit 3 of k, for K rows of krb bytes: 256 or more, (0, 6, 12, 10)
// and 2 more (XOR) in the second 8 rows of 16; 128 (8 chunks, two rows per
// 256 bytes of banks), (0, 2, 4, 6), likewise.
__device__ __forceinline__ constexpr int kn_swz(int k, int krb) {
  const int rho = k & 3, hi = ((k >> 3) & 1) << 1;
  return (krb >= 256 ? ((rho << 1) ^ (rho << 2)) & 14 : rho << 1) ^ hi;
}

// ds_read_b64_tr_b16 at LDS pointer p.  The pointer is __restrict__ for the
// alias scope that gives the read once inlined: without one the compiler puts
// a vmcnt(0) (a drain of every operand load in flight) before this read
// whenever an LDS-DMA load is pending.  (Never as inline asm with its wait
// elsewhere: the compiler takes such a result as there at once, and copied
// fragments of a tile's first step to other registers ahead of their wait.)
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short s16x4;
__device__ __forceinline__ txd::u32x2 tr_read(const uint8_t *__restrict__ p) {
  return __builtin_bit_cast(txd::u32x2,
                            __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4 *)p));
}

// One 16 x 16 block product: 64 bytes of K of 16-bit operands (a 16-byte
// piece per lane), or the 128 bytes of a whole step of fp8 (two).
template <class C>
__device__ __forceinline__ void mfma16(txd::f32x4 &acc, const txd::i32x4 (&b)[2], const txd::i32x4 (&a)[2], int h) {
  if constexpr (C::FP8) {
    const i32x8 vb = __builtin_shufflevector(b[0], b[1], 0, 1, 2, 3, 4, 5, 6, 7);
    const i32x8 va = __builtin_shufflevector(a[0], a[1], 0, 1, 2, 3, 4, 5, 6, 7);
    acc = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(vb, va, acc, F8Code<C::EL_B_>::v, F8Code<C::EL_A_>::v, 0, 0,
                                                           0, 0);
  } else if constexpr (C::F16) {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(txd::f16x8, b[h]),
                                                 __builtin_bit_cast(txd::f16x8, a[h]), acc, 0, 0, 0);
  } else {
    acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(txd::bf16x8, b[h]),
                                                  __builtin_bit_cast(txd::bf16x8, a[h]), acc, 0, 0, 0);
  }
}

// fast::ktail_clear for this tile's fragments: lane l holds chunk 4h + l / 16
// of the step in piece h.
template <int NF>
__device__ __forceinline__ void ktail_clear(txd::i32x4 (&fr)[NF][2], int h, int g, const fast::KTail &t) {
  const bool hit = 4 * h + g == t.cp;
  int m[4];
#pragma unroll
  for (int d = 0; d < 4; ++d) m[d] = hit ? int(t.keep[d]) : -1;
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int d = 0; d < 4; ++d) fr[f][h][d] &= m[d];
}

// Buffer resource for rows r0 .. r0 + BT - 1 of an operand with `rows` rows of
// `ld_b` bytes, K step bytes kb_end: rows past the operand's end are outside
// the range.
template <int BT>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const void *base, int r0, int rows, uint32_t ld_b,
                                                            uint32_t kb_end) {
  const int valid = min(BT, rows - r0);
  return make_rsrc(static_cast<const uint8_t *>(base) + int64_t(r0) * ld_b, uint32_t(valid - 1) * ld_b + kb_end);
}
}  // namespace persist

// GROUPED: the tiles of a grouped product (tx_grouped_args with offsets;
// the m-tile prefix already written by tx_gemm_fp8_grouped_prefix), a the
// shared fields q->g: tile t of the workgroup is (problem p, m tile, n tile)
// of expert p's rows offsets[p] .. offsets[p + 1] of A, C and scale_a against
// B + p stride_b and scale_b + p stride_sb.
//
// BKN: B is row-major K x N (16-bit operands, K a whole number of steps).  A
// step of B is then 64 K rows of the tile's BN columns (2 BN bytes each),
// DMA'd into a K-major slot whose 16-byte chunk c of K row k sits at
// c ^ kn_swz(k, 2 BN), and each B fragment is two transposing LDS reads
// (ds_read_b64_tr_b16): in each 16-lane group, lane s reads 4 columns at K
// row s / 4 and lane d receives column d's 4 K values, the register layout
// the MFMA takes.  The swizzle keeps a group's 4 rows x 2 chunks on 8
// distinct 16-byte bank groups of 128 bytes, and a 32-lane half's 4 rows x
// 4 chunks on 16 of 256 bytes (for 128-byte rows, two to 256 bytes of
// banks: on 8 of 128 and on 16 half-row positions).
template <class C, int OUT = OUT_BF16, bool GROUPED = false, bool KTAIL = false, bool BKN = false, int BM = 256,
          int BN = BM, bool EPI = false>
__device__ __forceinline__ void gemm_persist(const tx_gemm_args &a, const tx_grouped_args *q = nullptr) {
  using namespace fast;
  static_assert(OUT == OUT_BF16 || (OUT == OUT_F16 && !C::FP8) || (OUT == OUT_F32 && !C::FP8),
                "bf16 output, or fp16 / fp32 (+ accumulator) out of 16-bit operands");
  static_assert(!EPI || (C::FP8 && !GROUPED && BM == 128 && BN == 128), "fused epilogue: fp8, 128 x 128");
  constexpr bool F32 = OUT == OUT_F32;
  static_assert(!KTAIL || (!C::FP8 && !GROUPED), "ragged K: 16-bit operands, one product");
  static_assert(!BKN || (!C::FP8 && !GROUPED && !KTAIL), "row-major B: 16-bit operands, whole K steps");
  static_assert(BM == BN ? BM == 256 || BM == 128 || BM == 64 : BM == 128 && BN == 256 && GROUPED,
                "tile 256, 128 or 64 square; grouped also 128 x 256");
  constexpr int NW = persist::kWaves;
  constexpr int TM = BM / 2, TN = BN / 2, FM = TM / 16, FN = TN / 16;
  // MFMAs of a K step's half (16-bit: K half h; fp8: half of the columns)
  constexpr int NM = C::FP8 ? FM * FN / 2 : FM * FN, NF = FM + FN, NR = NF;
  static_assert(!C::FP8 || BN >= 128, "fp8: at least 128 columns");
  constexpr int SBA = BM * kStep, SBB = BN * kStep;  // one operand of one K step
  constexpr int BLKA = SBA / 1024 / NW, BLKB = SBB / 1024 / NW, ND = BLKA + BLKB;
  constexpr int RW = NM >= 2 ? NM / 2 : 1;
  // Ring: 256 x 256, 5 slots of one operand of one step (B two steps ahead, A
  // three); smaller tiles, whose step is a fraction of the time a load
  // takes to arrive, D stages of a step's A and B slots, both loaded D steps
  // ahead (128 x 128: 5, 160 KiB; 64 x 64: 8, 128 KiB): against the 5-slot ring
  // fp16 640 x 2000 x 3968 (64 x 64) 51.7 -> 33.0 us, 2304 x 2304 x 4096 (128
  // x 128) 68.1 -> 59.7.  128 x 256: 3 stages, 144 KiB.
  constexpr bool STG = BM < 256;
  constexpr int D = BM != BN ? 3 : BM == 128 ? 5 : 8, STAGE = SBA + SBB;
  constexpr int kLds = STG ? D * STAGE : kSlots * SBA;
  // The epilogue stages its output in the larger slot (A's if equal), whose
  // loads of the last step wait until it is done: operand op_st.
  constexpr int op_st = BN > BM ? 1 : 0;
  constexpr bool ROWCOL = C::FP8;
  // BKN: bytes of a K row of the B tile, and K rows per 1 KiB DMA block
  constexpr int KRB = 2 * BN, RPB = 1024 / KRB, CPR = KRB / 16;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[kLds];

  // m tiles: the grouped product's real count is only on the device
  const int tiles_m = GROUPED ? q->tile_prefix[q->groups] : a.tiles_m;
  const bool use_map = GROUPED && q->tile_map && tiles_m <= q->mtiles;
  const int total = tiles_m * a.tiles_n;
  const int G = int(gridDim.x);
  const int w = int(blockIdx.x);
  // COLS: the tiles of a last round that would leave at least half of the
  // workgroups idle are cut into 2 or 4 column parts, one to a workgroup.  The
  // grouped product streams weights from HBM, and a few whole tiles alone on
  // the chip take as long as a full round of them.  (The MFMAs of the columns
  // outside a part run on zeros.)
  constexpr bool COLS = GROUPED && BM < 256;
  const int whole = COLS ? total / G * G : total, over = total - whole;
  const int parts = !COLS || over == 0 ? 1 : over * 4 <= G ? 4 : over * 2 <= G ? 2 : 1;
  const int units = whole + over * parts;
  const int T = w < units ? (units - w + G - 1) / G : 0;  // tiles (or parts) of this workgroup
  if (T == 0) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % 2, wn = wave / 2;
  constexpr int ES = C::FP8 ? 1 : 2;
  const uint32_t kb_end = uint32_t(a.K) * ES;
  const int KS = int(KTAIL ? (kb_end + kStep - 1) / kStep : kb_end / kStep);  // K steps per tile (>= 2)
  const uint32_t lda_b = uint32_t(a.lda) * ES, ldb_b = uint32_t(a.ldb) * ES;

  // Per-lane DMA offsets within a tile: row * ld + chunk for the wave's
  // first two blocks (the chunk swizzle depends on the block's parity only);
  // block j adds 8 j rows, and the K step, in the scalar offset.
  const uint32_t kch[2] = {16u * uint32_t((lane & 7) ^ ((lane >> 4) & 7)),
                           16u * uint32_t((lane & 7) ^ ((4 + (lane >> 4)) & 7))};
  // BKN block j: K rows RPB (BLKB wave + j) .. + RPB - 1 of the step, lane p
  // filling chunk position p mod CPR of row + p / CPR.  The swizzle goes by
  // the row's low two bits and bit 3, so block j shares the lane offsets of
  // block kn_rep(j), kept at kn_var(j).
  constexpr auto kn_rep = [](int j) constexpr { return BN == 256 ? (j & 1) + 4 * (j >> 2) : BN == 128 ? j & ~1 : j; };
  constexpr auto kn_var = [](int j) constexpr { return BN == 256 ? (j & 1) + 2 * (j >> 2) : BN == 128 ? j >> 1 : j; };
  constexpr int NVB = BKN && BN == 256 ? 4 : 2;
  uint32_t vo[2][NVB];
#pragma unroll
  for (int e = 0; e < 2; ++e) vo[0][e] = uint32_t(8 * (BLKA * wave + e) + (lane >> 3)) * lda_b + kch[e];
  if constexpr (BKN) {
#pragma unroll
    for (int j = 0; j < BLKB; ++j) {
      const int kr = RPB * (BLKB * wave + j) + lane / CPR;
      if (j == kn_rep(j))
        vo[1][kn_var(j)] = uint32_t(kr) * ldb_b + 16u * uint32_t((lane % CPR) ^ persist::kn_swz(kr, KRB));
    }
  } else {
#pragma unroll
    for (int e = 0; e < 2; ++e) vo[1][e] = uint32_t(8 * (BLKB * wave + e) + (lane >> 3)) * ldb_b + kch[e];
  }
  const uint32_t ld8[2] = {8u * lda_b, (BKN ? uint32_t(RPB) : 8u) * ldb_b};
  // bytes of an operand's K step in its rows
  const uint32_t kstep_b[2] = {uint32_t(kStep), BKN ? 64u * ldb_b : uint32_t(kStep)};
  // KTAIL: the lane offsets of the last K step (scalar offset - 16 there)
  const KTail kt = make_ktail(kb_end);
  uint32_t vl[2][2];
  if constexpr (KTAIL) {
    const uint32_t kb16 = kb_end & ~15u, kr = kb_end & 15u, kbz = kr ? kb16 + 16u : kb_end;
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const uint32_t cs = uint32_t(KS - 1) * kStep + kch[e];  // the lane's chunk, from the row start
#pragma unroll
      for (int op = 0; op < 2; ++op) vl[op][e] = cs >= kbz ? kOob : vo[op][e] + (cs == kb16 ? kr : 16u);
    }
  }
  using OpA = std::integral_constant<int, 0>;
  using OpB = std::integral_constant<int, 1>;
  // Tile t of the workgroup: its operands and output (for a grouped product,
  // those of its problem) and its m / n tile.
  struct TileDesc {
    const uint8_t *A, *B;
    uint8_t *out;  // C
    const float *sa, *sb;
    int rows, tm, p;
    int n0, nend;  // columns n0 .. min(nend, n0 + BN) - 1
  };
  auto desc = [&](int t) {
    TileDesc d;
    int vm, tn;
    const int u = w + t * G;
    const int tile = u < whole ? u : whole + (u - whole) / parts;
    tile_coords(tile, a.tiles_n, tiles_m, min(8, a.tiles_n), &tn, &vm);  // transposed grid
    d.n0 = tn * BN;
    d.nend = a.N;
    if (COLS && u >= whole) {
      d.n0 += (u - whole) % parts * (BN / parts);
      d.nend = min(d.nend, d.n0 + BN / parts);
    }
    d.A = static_cast<const uint8_t *>(a.A);
    d.B = static_cast<const uint8_t *>(a.B);
    d.out = static_cast<uint8_t *>(a.C);
    d.sa = a.scale_a;
    d.sb = a.scale_b;
    d.rows = a.M;
    d.tm = vm;
    d.p = 0;
    if constexpr (GROUPED) {
      int p, r0;
      if (use_map) {
        const int4 e = reinterpret_cast<const int4 *>(q->tile_map)[vm];
        p = e.x;
        r0 = e.y;
        d.rows = e.z;
        d.tm = e.w;
      } else {
        const int32_t *Tp = q->tile_prefix;
        int lo = 0, hi = q->groups - 1;  // the last problem p with Tp[p] <= vm
        while (lo < hi) {
          const int mid = (lo + hi + 1) >> 1;
          if (Tp[mid] <= vm) lo = mid;
          else hi = mid - 1;
        }
        p = lo;
        const int r1 = min(max(q->offsets[p + 1], 0), a.M);
        r0 = min(max(q->offsets[p], 0), r1);
        d.rows = r1 - r0;
        d.tm = vm - Tp[lo];
      }
      // (uniform, but loaded through vector memory: buffer resources made
      // from vector registers would turn every operand load into a loop)
      p = __builtin_amdgcn_readfirstlane(p);
      r0 = __builtin_amdgcn_readfirstlane(r0);
      d.rows = __builtin_amdgcn_readfirstlane(d.rows);
      d.tm = __builtin_amdgcn_readfirstlane(d.tm);
      d.A += int64_t(r0) * a.lda;
      d.B += int64_t(p) * q->stride_b;
      d.out += int64_t(r0) * a.ldc * 2;
      d.sa += r0;
      d.sb += int64_t(p) * q->stride_sb;
      d.p = p;
    }
    return d;
  };

  // Load cursor of one operand: the step it is at and the buffer resource of
  // that step's tile (an empty range past the last tile).  Steps advance
  // one at a time.
  // ROT: a tile's K steps run from a start of its own (by expert, spread over
  // K, so tiles that share rows of A or B stay in step) and wrap around: kp
  // is the step's place in K, k its number.  Experts' weights are read from
  // HBM, and with a row pitch of a power of two the same K step of every row
  // sits on the same few channels: 64 experts x 2048 x 4096, 256 rows in all
  // (weights alone), 131 us in step, 97 us rotated.
  constexpr bool ROT = GROUPED && BM < 256;
  struct Cursor {
    int t, k, kp;
    __amdgpu_buffer_rsrc_t rs;
  };
  auto set_tile = [&](Cursor &c, auto op_tag) {
    constexpr int op = decltype(op_tag)::value;
    c.kp = 0;
    if (c.t < T) {
      const TileDesc d = desc(c.t);
      if constexpr (ROT) c.kp = int(__umulhi(uint32_t(d.p) * 2654435769u, uint32_t(KS)));
      if constexpr (BKN && op == 1) {
        // columns n0 .. of all K rows, the range ending at the last
        // row's last column (columns past N in earlier rows read that
        // row's padding or the next row: their products are not stored)
        c.rs = make_rsrc(d.B + int64_t(d.n0) * 2, uint32_t(a.K - 1) * ldb_b + uint32_t(a.N - d.n0) * 2u);
      } else {
        c.rs = op == 0                   ? persist::tile_rsrc<BM>(d.A, d.tm * BM, d.rows, lda_b, kb_end)
               : COLS && d.n0 >= d.nend ? make_rsrc(a.B, 0u)
                                         : persist::tile_rsrc<BN>(d.B, d.n0, d.nend, ldb_b, kb_end);
      }
    } else {
      c.rs = make_rsrc(op == 0 ? a.A : a.B, 0u);
    }
  };
  auto advance = [&](Cursor &c, auto op_tag) {
    ++c.kp;
    if (ROT && c.kp == KS) c.kp = 0;
    if (++c.k == KS) {
      c.k = 0;
      ++c.t;
      set_tile(c, op_tag);
    }
  };
  auto load_op = [&](const Cursor &c, int base, auto op_tag, auto j_tag) {
    constexpr int op = decltype(op_tag)::value, j = decltype(j_tag)::value;
    constexpr int blk = op == 0 ? BLKA : BLKB;
    uint8_t *dst = lds + base + (blk * wave + j) * 1024;
    const bool lk = KTAIL && c.k == KS - 1;  // (c.k >= 1 there)
    constexpr int var = BKN && op == 1 ? kn_var(j) : j & 1;
    constexpr int past = BKN && op == 1 ? j - kn_rep(j) : j & ~1;  // blocks past the one of those offsets
    __builtin_amdgcn_raw_ptr_buffer_load_lds(c.rs, (lds_void *)dst, 16, lk ? vl[op][j & 1] : vo[op][var],
                                             uint32_t(c.kp) * kstep_b[op] + uint32_t(past) * ld8[op] -
                                                 (lk ? 16u : 0u),
                                             0, 0);
  };

  // Fragment f (A blocks 0 .. FM-1, then B blocks) is 16 rows x 128 bytes of
  // K: lane l holds row l % 16, 16-byte pieces x = 0, 1 = logical chunks
  // 4x + l / 16 (16-bit: piece x is K half x, one 16x16x32 MFMA; fp8: both
  // pieces are one 16x16x128 MFMA; the order of K inside a product is the
  // same for A and B).  Blocks 16 rows apart share the swizzle.
  const int frow = lane & 15, fg = lane >> 4;
  int ro[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x) {
    ro[0][x] = off(wm * TM + frow, 4 * x + fg);
    ro[1][x] = off(wn * TN + frow, 4 * x + fg);
  }
  // BKN: the B fragment reads' lane offsets in a slot, per 16-column block
  // fn, for K row 8 g + s / 4 (g = lane / 16, s = lane mod 16) and columns
  // 16 fn + 4 (s mod 4) .. + 3 of the wave's; half h and read r add K rows
  // 32 h + 4 r (which leave the swizzle alone).
  int bko[BKN ? FN : 1];
  if constexpr (BKN) {
    const int s16 = lane & 15, kr = 8 * fg + (s16 >> 2);
#pragma unroll
    for (int fn = 0; fn < FN; ++fn) {
      const int n = wn * TN + 16 * fn + 4 * (s16 & 3);
      bko[fn] = kr * KRB + (((n >> 3) ^ persist::kn_swz(kr, KRB)) << 4) + 8 * ((n >> 2) & 1);
    }
  }
  txd::i32x4 fr[NF][2];
  // Read piece x of fragment f of the step at LDS bytes base_a, base_b.
  auto read_piece = [&](int base_a, int base_b, auto f_tag, auto x_tag) {
    constexpr int f = decltype(f_tag)::value, x = decltype(x_tag)::value;
    if constexpr (BKN && f >= FM) {
      const uint8_t *bp = lds + (base_b + bko[f - FM]) + 32 * x * KRB;
      const txd::u32x2 lo = persist::tr_read(bp), hi = persist::tr_read(bp + 4 * KRB);
      fr[f][x] = txd::i32x4{int(lo[0]), int(lo[1]), int(hi[0]), int(hi[1])};
    } else {
      const uint8_t *Sp = lds + (f < FM ? base_a : base_b);
      const int byte = f < FM ? ro[0][x] + 2048 * f : ro[1][x] + 2048 * (f - FM);
      fr[f][x] = *reinterpret_cast<const txd::i32x4 *>(Sp + byte);
    }
  };
  // Read r of K half h (16-bit), in the order the MFMAs consume them: A0, B0,
  // A1 .. A(FM-1), B1 .. B(FN-1).
  auto read = [&](int base_a, int base_b, auto h_tag, auto r_tag) {
    constexpr int o = decltype(r_tag)::value, f = o == 0 ? 0 : o == 1 ? FM : o <= FM ? o - 1 : o;
    read_piece(base_a, base_b, std::integral_constant<int, f>{}, h_tag);
  };
  txd::f32x4 acc[FN][FM];
  // The MFMA of B block fn against A block fm on K half h (fp8: the whole
  // step); ZERO: the block's first of the tile, from a zero accumulator.
  auto mma = [&](auto h_tag, auto fn_tag, auto fm_tag, auto zero_tag) {
    constexpr int h = decltype(h_tag)::value, fn = decltype(fn_tag)::value, fm = decltype(fm_tag)::value;
    if constexpr (decltype(zero_tag)::value) acc[fn][fm] = txd::f32x4{};
    persist::mfma16<C>(acc[fn][fm], fr[FM + fn], fr[fm], h);
    // (kept in its AGPRs: left alone the ragged-K variant rotates blocks
    // through VGPRs and spills 26 of them, and the fp32 one copies them)
    if constexpr (KTAIL || (F32 && BM < 256)) asm volatile("" : "+a"(acc[fn][fm]));
  };
  using H0 = std::integral_constant<int, 0>;
  using H1 = std::integral_constant<int, 1>;

  // Prologue: steps 0, 0, 1, 1, 2 (A0 B0 A1 B1 A2) of the first tile (STG:
  // A and B of its first D steps).
  Cursor ca, cb;
  ca.t = ca.k = cb.t = cb.k = 0;
  set_tile(ca, OpA{});
  set_tile(cb, OpB{});
  static_for<STG ? D : 2>([&](auto st) {
    constexpr int la = decltype(st)::value * (STG ? STAGE : 2 * SBA), lb = la + SBA;
    static_for<BLKA>([&](auto j) { load_op(ca, la, OpA{}, j); });
    static_for<BLKB>([&](auto j) { load_op(cb, lb, OpB{}, j); });
    advance(ca, OpA{});
    advance(cb, OpB{});
  });
  if constexpr (STG) {
    wait_and_barrier<(D - 1) * ND>();
  } else {
    // (next B load: step 2, next A load: step 3)
    static_for<BLKA>([&](auto j) { load_op(ca, 4 * SBA, OpA{}, j); });
    advance(ca, OpA{});
    wait_and_barrier<2 * BLKA + BLKB>();
  }
  // The fragments a step starts with: 16-bit, its first K half; fp8, all of A
  // and the first two B blocks.
  auto read_start = [&](int base_a, int base_b) {
    if constexpr (C::FP8) {
      static_for<FM + 2>([&](auto f) {
        read_piece(base_a, base_b, f, H0{});
        read_piece(base_a, base_b, f, H1{});
      });
    } else {
      static_for<NR>([&](auto r) { read(base_a, base_b, H0{}, r); });
    }
  };
  read_start(0, SBA);

  // One K step: half 0 (reads of the rest of the step's fragments), barrier,
  // half 1 (loads of B s+2 and A s+3, reads of the first fragments of step
  // s+1).  16-bit: half h is K half h of all blocks.  fp8, whose MFMA takes
  // the whole step's K: half 0 is B blocks 0 .. FN/2-1, block by block, half 1
  // the others, A block by A block: each A block's registers are reloaded
  // with step s+1 right after its last MFMA, so fragments take 112 registers
  // (A 64, four B blocks in use and two ahead).
  // FIRST: the tile's first step
  // (MFMAs from a zero accumulator); VM: loads and stores allowed in flight
  // at the barrier (the next step's operands are older than the last VM);
  // LAST: the tile's last step, whose loads into the staging slot (op_st)
  // wait until after the epilogue, as do the reads of the
  // next step's first half (their registers hold the column scales).
  int sa = 0, sb = SBA;  // LDS bytes of step s's A and B
  auto step = [&](auto first_tag, auto vm_tag, auto last_tag) {
    constexpr int VM = decltype(vm_tag)::value;
    constexpr bool LAST = decltype(last_tag)::value;
    // those of step s+1, and of the loads (step s's, free after the barrier)
    const int na = STG ? (sa == (D - 1) * STAGE ? 0 : sa + STAGE) : sa >= 3 * SBA ? sa - 3 * SBA : sa + 2 * SBA;
    const int nb = STG ? na + SBA : sb >= 3 * SBA ? sb - 3 * SBA : sb + 2 * SBA;
    const int la = STG ? sa : sb, lb = STG ? sb : sa;
    const bool clear = KTAIL && LAST && kt.cp < 8;
    if (clear) persist::ktail_clear<NF>(fr, 0, fg, kt);
    static_for<NM>([&](auto I) {
      constexpr int i = decltype(I)::value;
      using Fn = std::integral_constant<int, i / FM>;
      using Fm = std::integral_constant<int, i % FM>;
      mma(H0{}, Fn{}, Fm{}, first_tag);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (C::FP8) {
        // B blocks 2 .. FN-1, two pieces each, over three quarters of the MFMAs
        constexpr int n = 2 * (FN - 2), r0 = spread_lo(i, n, NM * 3 / 4), r1 = spread_hi(i, n, NM * 3 / 4);
        static_for<r1 - r0>([&](auto R) {
          constexpr int r = r0 + decltype(R)::value;
          read_piece(sa, sb, std::integral_constant<int, FM + 2 + r / 2>{}, std::integral_constant<int, r % 2>{});
        });
      } else {
        constexpr int r0 = spread_lo(i, NR, RW), r1 = spread_hi(i, NR, RW);
        static_for<r1 - r0>(
            [&](auto R) { read(sa, sb, H1{}, std::integral_constant<int, r0 + decltype(R)::value>{}); });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    wait_and_barrier<VM>();
    __builtin_amdgcn_sched_barrier(0);
    if (clear) persist::ktail_clear<NF>(fr, 1, fg, kt);
    static_for<NM>([&](auto I) {
      constexpr int i = decltype(I)::value;
      constexpr int HF = FN / 2;
      if constexpr (C::FP8)
        mma(H1{}, std::integral_constant<int, HF + i % HF>{}, std::integral_constant<int, i / HF>{}, first_tag);
      else
        mma(H1{}, std::integral_constant<int, i / FM>{}, std::integral_constant<int, i % FM>{}, std::false_type{});
      __builtin_amdgcn_sched_barrier(0);
      // operand loads half a run of MFMAs away from the (16-bit) fragment reads
      constexpr auto nd = [](int j) constexpr {
        return j <= 0 ? 0 : j >= NM ? ND : (j + (C::FP8 ? 0 : NM / ND / 2)) * ND / NM;
      };
      constexpr int d0 = nd(i), d1 = nd(i + 1);
      static_for<d1 - d0>([&](auto D) {
        constexpr int d = d0 + decltype(D)::value;
        if constexpr (d < BLKB) {
          if constexpr (!LAST || op_st == 0) load_op(cb, lb, OpB{}, std::integral_constant<int, d>{});
        } else if constexpr (!LAST || op_st == 1) {
          load_op(ca, la, OpA{}, std::integral_constant<int, d - BLKB>{});
        }
      });
      if constexpr (!LAST && C::FP8) {
        // A block i / HF after its last MFMA (the second piece one MFMA on),
        // B blocks 0 and 1 in between
        constexpr int g = i / HF, j = i % HF;
        if constexpr (j == HF - 1) read_piece(na, nb, std::integral_constant<int, g>{}, H0{});
        if constexpr (j == 0 && g > 0) read_piece(na, nb, std::integral_constant<int, g - 1>{}, H1{});
        constexpr int p = HF == 4 ? (j == 1 ? g : 4) : i;  // piece p of those four
        if constexpr (p < 4)
          read_piece(na, nb, std::integral_constant<int, FM + p / 2>{}, std::integral_constant<int, p % 2>{});
        if constexpr (i == NM - 1) read_piece(na, nb, std::integral_constant<int, FM - 1>{}, H1{});
      } else if constexpr (!LAST) {
        constexpr int r0 = spread_lo(i, NR, NM), r1 = spread_hi(i, NR, NM);
        static_for<r1 - r0>(
            [&](auto R) { read(na, nb, H0{}, std::integral_constant<int, r0 + decltype(R)::value>{}); });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
    if constexpr (!LAST || op_st == 0) advance(cb, OpB{});
    if constexpr (!LAST || op_st == 1) advance(ca, OpA{});
    sa = na;
    sb = nb;
  };
  // operand loads the barrier of a step leaves in flight: those of the steps
  // past s+1
  constexpr int kAhead = STG ? (D - 2) * ND : BLKA;
  using VmStep = std::integral_constant<int, kAhead>;
  // The epilogue issues exactly kEpiStores stores per wave, then the last
  // step's deferred BLKA loads of A; the next tile's first barrier may
  // leave all of them in flight.
  // staging geometry: the wave's 32 x TN block as 32 rows of SRB bytes
  // (CH 16-byte chunks), read back SPI rows per instruction
  constexpr int SRB = 2 * TN, CH = SRB / 16, SPI = 64 / CH;
  constexpr int kEpiStores = F32 ? FM * FN : FM / 2 * (32 / SPI);
  // (EPI: the number of stores depends on the output's type and alignment;
  // none may be left, which is always safe)
  constexpr int kAfterEpi = kAhead + (EPI ? 0 : kEpiStores) + (STG ? 0 : BLKB - BLKA);
  static_assert(32 * SRB * NW <= (op_st == 0 ? SBA : SBB), "the staging fits its slot");
  using VmAfterEpi = std::integral_constant<int, (kAfterEpi < 64 ? kAfterEpi : 63)>;
  // Scale loads issued before the last step (row scales, column-scale
  // vectors) that its barrier leaves in flight with the step's own A loads.
  // F32: the tile's accumulator operand (C), 4 columns per load, is read in
  // batches of FB row blocks, 16 loads (64 x 64: 4; KTAIL, short of registers:
  // 8) each, the first before the last step.
  constexpr int FB = FM < 4 ? FM : KTAIL ? 1 : 16 / FN, NB = FM / FB;
  constexpr int kScaleLoads = ROWCOL ? FM + FN : F32 ? FB * FN : 0;
  using VmLast = std::integral_constant<int, kAhead + kScaleLoads>;
  static_assert(kAhead + kScaleLoads < 64, "vmcnt range");

  // Staging: wave w owns bytes 32 SRB w .. + 32 SRB of the slot its last
  // step's deferred loads would have filled (the same bytes those loads fill
  // once the epilogue is done, so no other wave ever touches them): 32 rows
  // of SRB bytes, 16-byte chunk c of row r at c ^ (r % CH).
  // F32 tiles below 256: K in segments of a.ksteps_split steps (0: one),
  // summed in fp32 registers in order, the rounding of a K split's planes (a
  // segment's MFMA chain is that much shorter).
  constexpr bool FOLD = F32 && BM < 256;
  txd::f32x4 sum[FOLD ? FN : 1][FOLD ? FM : 1];
  bool folded = false;
  for (int t = 0; t < T; ++t) {
    const TileDesc d = desc(t);
    const int m0 = d.tm * BM, n0 = d.n0;
    // C as a buffer: a store whose row or column block lies past M / N gets
    // an offset past the range and is dropped (N is a multiple of 8, so a
    // 16-byte column block is wholly in or out).  KTAIL: rows of C may have
    // any alignment; the buffer starts at the 16-byte boundary below C; N may
    // be any, and a block that N cuts is stored column by column.
    const uint32_t cmis = KTAIL ? uint32_t(reinterpret_cast<uintptr_t>(d.out) & 15u) : 0u;
    const __amdgpu_buffer_rsrc_t crs =
        make_rsrc(d.out - cmis, uint32_t((int64_t(d.rows - 1) * a.ldc + a.N) * (F32 ? 4 : 2)) + cmis);
    if (t == 0) step(std::true_type{}, VmStep{}, std::false_type{});
    else step(std::true_type{}, VmAfterEpi{}, std::false_type{});
    if constexpr (FOLD) {
      // K segments: at each boundary the accumulators are added to `sum`
      // and start again from zero
      const int per = a.ksteps_split > 0 ? a.ksteps_split : KS;
      folded = KS - per >= 2;
      if (folded) {
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
          for (int fm = 0; fm < FM; ++fm) sum[fn][fm] = txd::f32x4{0.f, 0.f, 0.f, 0.f};
      }
      // steps between the tile's first and last; none may end on a boundary
      // just before the last
      for (int rem = KS - 2, n = min(per - 1, rem);;) {
        for (int i = 0; i < n; ++i) step(std::false_type{}, VmStep{}, std::false_type{});
        rem -= n;
        if (rem == 0) break;
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
#pragma unroll
          for (int fm = 0; fm < FM; ++fm) sum[fn][fm] += acc[fn][fm];
        step(std::true_type{}, VmStep{}, std::false_type{});
        --rem;
        n = min(per - 1, rem);
      }
    } else {
      for (int k = 1; k < KS - 1; ++k) step(std::false_type{}, VmStep{}, std::false_type{});
    }
    // Scales load just before the last step; the compiler's wait for them after
    // it leaves that step's own loads in flight (vector-memory operations
    // complete in order).  Exactly kScaleLoads of them, between scheduling
    // barriers, since the last step's barrier counts them.  Rows past M read
    // row M - 1 and columns past N the last four; their stores are dropped.
    float sav[FM];
    txd::f32x4 sb4[FN];  // columns 16 fn + 4 g .. + 3 of the wave's
    if constexpr (ROWCOL) {
      typedef txd::f32x4 f32x4_a4 __attribute__((aligned(4)));
      const int nl = n0 + wn * TN + 4 * fg;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int fm = 0; fm < FM; ++fm) sav[fm] = d.sa[min(m0 + wm * TM + fm * 16 + frow, d.rows - 1)];
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
        sb4[fn] = *reinterpret_cast<const f32x4_a4 *>(d.sb + min(nl + 16 * fn, a.N - 4));
      __builtin_amdgcn_sched_barrier(0);
    }
    // F32: the accumulator operand through a buffer of its own (empty
    // without one), element (m, n) of row block fm and column block fn.
    txd::u32x4 cin[F32 ? 2 : 1][F32 ? FB : 1][F32 ? FN : 1];
    const __amdgpu_buffer_rsrc_t ars = make_rsrc(
        a.acc, F32 && a.acc ? uint32_t((int64_t(d.rows - 1) * a.ld_acc + a.N) * 4) : 0u);
    // byte offset of row block fm, column block fn in a matrix of ld
    // elements; past M / N, out of any range (N is a multiple of 4 here)
    auto f32_off = [&](int fm, int fn, int64_t ld) {
      const int m = m0 + wm * TM + 16 * fm + frow, n = n0 + wn * TN + 16 * fn + 4 * fg;
      return m < d.rows && n < a.N ? (uint32_t(m) * uint32_t(ld) + uint32_t(n)) * 4u : kOob;
    };
    auto load_acc = [&](auto b_tag) {
      constexpr int b = decltype(b_tag)::value;
#pragma unroll
      for (int i = 0; i < FB; ++i)
#pragma unroll
        for (int fn = 0; fn < FN; ++fn)
          cin[b % 2][i][fn] = __builtin_bit_cast(
              txd::u32x4, __builtin_amdgcn_raw_buffer_load_b128(ars, f32_off(b * FB + i, fn, a.ld_acc), 0, 0));
    };
    if constexpr (F32) {
      load_acc(std::integral_constant<int, 0>{});
      __builtin_amdgcn_sched_barrier(0);
    }
    const int stage_at = op_st == 1 ? sb : STG ? sa : sb;  // where the last step's op_st loads go
    step(std::false_type{}, VmLast{}, std::true_type{});  // the last step (KS >= 2)
    // Epilogue, per 32-row block: scale, round and stage the wave's 32 x TN
    // block (lane l: 4 columns 16 fn + 4 (l / 16) .. of row l % 16 of each 16 x
    // 16 block), then store SPI rows of SRB bytes per instruction.
    // The accumulators are read below in inline asm, for which the compiler
    // inserts no wait states after the MFMAs that write them: the last step's
    // final MFMAs stay above this point, and 32 wait states (an 8-pass MFMA's
    // result needs about 11) pass before the first read.
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (F32) {
      // D = A.B + C straight from the accumulators: 16 rows of 64 bytes per
      // store.  Batch b + 1 of C loads ahead of batch b's stores, so its wait
      // never includes them.
      static_for<NB>([&](auto b_tag) {
        constexpr int b = decltype(b_tag)::value;
        if constexpr (b + 1 < NB) {
          load_acc(std::integral_constant<int, b + 1>{});
          __builtin_amdgcn_sched_barrier(0);
        }
        static_for<FB>([&](auto i_tag) {
          constexpr int i = decltype(i_tag)::value, fm = b * FB + i;
          static_for<FN>([&](auto fn_tag) {
            constexpr int fn = decltype(fn_tag)::value;
            txd::u32x4 w;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              float v;
              asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc[fn][fm][q]));
              if constexpr (FOLD)
                if (folded) v = sum[fn][fm][q] + v;
              w[q] = __float_as_uint(a.acc ? v + __uint_as_float(cin[b % 2][i][fn][q]) : v);
            }
            __builtin_amdgcn_raw_buffer_store_b128(w, crs, f32_off(fm, fn, a.ldc), 0, 0);
          });
        });
        __builtin_amdgcn_sched_barrier(0);
      });
    }
    if constexpr (EPI) {
      // bias, activation and the output's type, from the accumulators: 4
      // columns of a row per lane and store
      const int nb = n0 + wn * TN + 4 * fg;
      txd::f32x4 bias4[FN];
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          bias4[fn][q] = a.bias && nb + 16 * fn + q < a.N ? a.bias[nb + 16 * fn + q] : 0.0f;
      with_act(a.act, [&](auto act_tag) {
        constexpr int ACT = decltype(act_tag)::value;
        static_for<FM>([&](auto fm_tag) {
          constexpr int fm = decltype(fm_tag)::value;
          const int m = m0 + wm * TM + 16 * fm + frow;
          static_for<FN>([&](auto fn_tag) {
            constexpr int fn = decltype(fn_tag)::value;
            float y[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
              float v;
              asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v) : "a"(acc[fn][fm][q]));
              y[q] = epi_act_t<ACT>(v * sav[fm] * sb4[fn][q] + bias4[fn][q]);
            }
            // (N is a multiple of 8: 4 columns are wholly in or out)
            if (m < d.rows && nb + 16 * fn < a.N) epi_store4(a, m, nb + 16 * fn, y);
          });
        });
      });
    }
    uint8_t *stg = lds + stage_at + wave * (32 * SRB);
    // The lane's staging offsets are recomputed for each tile from an opaque
    // copy of the lane index: hoisted out of the tile loop, they would hold
    // registers through the whole K loop (fp8: 238 -> 206 VGPRs).
    int el = lane;
    asm volatile("" : "+v"(el));
    const int efrow = el & 15, efg = el >> 4;
    const int srow = el / CH, schunk = el % CH;  // read-back: row SPI i + srow, chunk schunk
    const int n_st = n0 + wn * TN + 8 * schunk;
    // KTAIL: N may be any; the lanes whose 8 columns straddle it (in a last
    // column tile) store them one by one.
    const bool straddle = KTAIL && (d.nend & 7) != 0 && n0 + BN > d.nend;
    const int cols = KTAIL ? d.nend - n_st : 8;  // valid columns from n_st on
    const uint32_t coloff = n_st < d.nend && (!KTAIL || cols >= 8) ? uint32_t(n_st) * 2u + cmis : kOob;
    if constexpr (!F32 && !EPI) static_for<FM / 2>([&](auto blk_tag) {
      constexpr int blk = decltype(blk_tag)::value;
      static_for<2>([&](auto u_tag) {
        constexpr int u = decltype(u_tag)::value, fm = 2 * blk + u;
        static_for<FN>([&](auto fn_tag) {
          constexpr int fn = decltype(fn_tag)::value;
          float v[4];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            // read the accumulator where it is used (the compiler would
            // otherwise copy whole tiles out of the AGPRs at once)
            asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(v[q]) : "a"(acc[fn][fm][q]));
            if constexpr (ROWCOL) v[q] = v[q] * sav[fm] * sb4[fn][q];
          }
          const int row = 16 * u + efrow, chunk = 2 * fn + (efg >> 1);
          *reinterpret_cast<txd::u32x2 *>(stg + row * SRB + ((chunk ^ (row & (CH - 1))) << 4) + 8 * (efg & 1)) =
              OUT == OUT_F16 ? txd::u32x2{txd::pack_f16x2(v[0], v[1]), txd::pack_f16x2(v[2], v[3])}
                             : txd::u32x2{txd::pack_bf16x2(v[0], v[1]), txd::pack_bf16x2(v[2], v[3])};
        });
      });
#pragma unroll
      for (int i = 0; i < 32 / SPI; ++i) {
        const int r = SPI * i + srow;
        const txd::u32x4 w = *reinterpret_cast<const txd::u32x4 *>(stg + r * SRB + ((schunk ^ (r & (CH - 1))) << 4));
        const int m = m0 + wm * TM + blk * 32 + r;
        const uint32_t voff = (m >= d.rows || coloff == kOob) ? kOob : uint32_t(m) * uint32_t(a.ldc) * 2u + coloff;
        __builtin_amdgcn_raw_buffer_store_b128(w, crs, voff, 0, 0);
        if (straddle && cols > 0 && cols < 8 && m < d.rows) {
#pragma unroll
          for (int t = 0; t < 7; ++t)
            if (t < cols)
              __builtin_amdgcn_raw_buffer_store_b16(uint16_t(w[t / 2] >> (16 * (t & 1))), crs,
                                                    uint32_t(m) * uint32_t(a.ldc) * 2u + uint32_t(n_st + t) * 2u + cmis,
                                                    0, 0);
        }
      }
    });
    // the deferred loads (after this wave's last staging reads) and
    // the next step's first-half fragments
    __builtin_amdgcn_s_waitcnt((63 & 15) | (7 << 4) | (0 << 8) | ((63 >> 4) << 14));
    if constexpr (op_st == 0) {
      static_for<BLKA>([&](auto j) { load_op(ca, stage_at, OpA{}, j); });
      advance(ca, OpA{});
    } else {
      static_for<BLKB>([&](auto j) { load_op(cb, stage_at, OpB{}, j); });
      advance(cb, OpB{});
    }
    read_start(sa, sb);
  }
  // Drain the trailing (empty-range) loads before the workgroup's LDS is released.
  wait_and_barrier<0>();
}

}  // namespace txg
