// Prefill GEMM on gfx950: out[M,N] = X[M,K] (bf16) @ W[N,K]^T on bf16 MFMA
// (v_mfma_f32_16x16x32_bf16) for INT4 g128, INT8 per-channel and bf16 weights, with the
// prefill plan's fused epilogues.
//
//   * Block tiles from 64 x 64 to 256 x 256 (TileCfg), chosen per launch by an estimate
//     of its time (EstimateUs).  What bounds them: few rows, the weight stream and the
//     first loads' latency; many rows, the matrix pipe, which the LDS reads, the weight
//     conversions and the barriers of the k loop have to stay behind.
//   * Operands move global -> LDS by DMA (global_load_lds_dwordx4): no registers and no
//     LDS store instructions, so two or more k steps are in flight while one is
//     computed.  The ring holds the stages of X and W (per 64 k values, 128 bytes of an X
//     row and 32 B INT4, 64 B INT8 or 128 B bf16 of a W row), plus for INT4 a four-slot
//     ring of the fp16 group scales.
//   * DMA writes a wave's 64 lanes to 1 KB of consecutive LDS, so the bank layout is
//     set by which global chunk each lane fetches: 16-byte chunk c of row r sits at a
//     slot c ^ f(r) of the row (xsw, wslot), such that the 16 lanes that a 128-bit LDS read
//     serves at once (rows 0-3 and 12-15 of one k block, rows 4-11 of the next) fall into
//     distinct banks.  Conflicts counted on the 512-row 8B shapes are 0.2-1.5% of the LDS's
//     active cycles with bf16 weights, 10-16% with INT4 and 16-20% with INT8, whose 4- and
//     8-byte weight reads have them; half of the cycles before.
//   * The k loop reads the operands of one 32-value slice while the MFMAs of the slice
//     before run, also across the barrier between two steps, and converts the next
//     slice's weights between those MFMAs (one set of A registers, refilled row by row).
//     2048 x 28672 x 4096: bf16 574 -> 430 us (1.12 PFLOP/s), INT8 781 -> 460 us, INT4
//     669 -> 505 us against the loop that read, converted and multiplied in turn.
//   * Blocks are dealt to the XCDs in contiguous eighths of the tiles, so that weight and
//     row tiles are shared in one L2 (bf16 as above: 453 instead of 566 us at 128 x 256).
//   * The weight stays in its storage format in LDS.  INT4: signed nibble conversions
//     (v_cvt_off_f32_i4 gives q / 16 exactly), two packed into a register.  INT8: signed
//     byte conversions.  Both are exact in bf16.  Products are exact and accumulation is
//     fp32.  bf16: one 128-bit read, no conversion.
//   * INT4 group scales: the sums are kept in units of the running group's scale, so a
//     new group costs one multiplication by old / new scale per sum and no second set of
//     accumulators (which held the tile at 64 x 64 per wave); the last scale comes at the
//     end.  The error against 64 bits is that of the bf16 outputs (0.0061 at 512 rows,
//     before and now).
//   * Rows past the M or N edge read row 0 and are never stored.
//   * Split-K (tiles that would leave CUs idle): split s of a tile owns a contiguous
//     range of whole groups (128 k values for INT8 and bf16).  Each split block stores
//     its fp32 accumulators with device-scope stores, waits for them, and takes a ticket;
//     the last block of the tile reads the other partials back with device-scope loads
//     and sums all of them in split order (the same order whichever block is last, so
//     results do not depend on scheduling), resets the ticket and runs the epilogue.
//   * Epilogues (the op boundaries of the reference graph, model_graph_builder.cpp:
//     133-290) go through LDS: the block writes round(acc) as a bf16 tile, then every
//     thread moves 16-byte row chunks (one load of residual, one store per chunk).
//     Store; residual (out = round(res + round(acc)), Linear then Add); column split
//     (one q|k|v weight, three outputs); SiLU-Mul (tile columns [0, BN/2) are gate
//     features u, [BN/2, BN) the up rows of the same u: act = round(silu(round(gate))
//     * round(up))); q|k|v with RoPE and the KV cache write.  Chunks that cross the N
//     edge or a split column, or outputs whose rows are not 16-byte aligned, take the
//     per-element path.

#include <algorithm>
#include <type_traits>

#include "am_gemv_common.h"
#include "am_launch_timing.h"

namespace am {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8_t;
typedef __attribute__((ext_vector_type(4))) float f32x4_t;
typedef __attribute__((address_space(3))) void lvoid;

constexpr int QBK = 64;  // the k granule: a split's and a group's length are multiples of it
typedef unsigned int u32x4_t __attribute__((ext_vector_type(4)));
// Split-K partials move as 16-byte buffer loads and stores carrying the sc1 cache
// policy (bit 4 of the builtins' aux operand on gfx950): the device-coherent accesses
// the relaxed agent-scope atomics compile to, four words at a time.  The descriptor's
// last dword is the raw-buffer format word (32-bit data, no swizzle); a wave's region
// is one 64 lanes x 16 bytes record per MFMA tile of the wave.
constexpr int kCpolSc1 = 16;
constexpr int kRawBufferFlags = 0x00020000;

// Bytes of 64 k values of one weight row.
template <int WF> struct WRow;
template <> struct WRow<AM_WF_INT4> { static constexpr int kBytes = 32; };
template <> struct WRow<AM_WF_INT8> { static constexpr int kBytes = 64; };
template <> struct WRow<AM_WF_BF16> { static constexpr int kBytes = 128; };

// Block shapes.  MW x NW waves, each MT x NT MFMA tiles of 16 x 16, a k step of BK
// values, NST DMA stages, BPC resident blocks per CU to compile for.
//   Quantized weights: one wave row (MW = 1), so that each weight is converted by one wave
//   only.  LDS reads of X cost less than conversions (256 bytes against 16 weights' 28
//   VALU operations per clock and CU): 2048 x 28672 x 4096 INT4 654 -> 546 us, INT8 535 ->
//   476 us on the 128 x 256 tile.  bf16 weights need no conversion: two wave rows, which
//   read the least from LDS.  The 256 x 256 tile keeps two rows in every format (one row
//   of 16 x 2 tiles per wave does not fit the registers).
//   INT4 takes 128 k values a step where LDS allows it (half the barriers and scale
//   loads: 546 -> 505 us on the shape above).
enum Tile { kT128 = 0, kT256 = 1, kT64 = 2, kT64W = 3, kT256x256 = 4 };
template <int WF, int TILE> struct TileCfg;
//   128 x 128, 256 threads (INT4 62 KB of LDS and INT8 72 KB: two blocks per CU; bf16
//   96 KB: one)
template <int WF> struct TileCfg<WF, kT128> {
  static constexpr bool kB = WF == AM_WF_BF16;
  static constexpr int MT = kB ? 4 : 8, NT = kB ? 4 : 2, MW = kB ? 2 : 1, NW = kB ? 2 : 4, BK = 64, NST = 3, BPC = 2;
};
//   128 x 256, 512 threads, one block per CU
template <int WF> struct TileCfg<WF, kT256> {
  static constexpr bool kB = WF == AM_WF_BF16;
  static constexpr int MT = kB ? 4 : 8, NT = kB ? 4 : 2, MW = kB ? 2 : 1, NW = kB ? 4 : 8,
                       BK = WF == AM_WF_INT4 ? 128 : 64, NST = WF == AM_WF_INT8 ? 4 : 3, BPC = 1;
};
//   64 x 64 (256 threads) and 64 x 128 (512 threads) for few rows, two blocks per CU
template <int WF> struct TileCfg<WF, kT64> {
  static constexpr bool kB = WF == AM_WF_BF16;
  static constexpr int MT = kB ? 2 : 4, NT = kB ? 2 : 1, MW = kB ? 2 : 1, NW = kB ? 2 : 4,
                       BK = WF == AM_WF_INT4 ? 128 : 64, NST = WF == AM_WF_INT4 ? 3 : (WF == AM_WF_INT8 ? 6 : 4), BPC = 2;
};
template <int WF> struct TileCfg<WF, kT64W> {
  static constexpr bool kB = WF == AM_WF_BF16;
  static constexpr int MT = kB ? 2 : 4, NT = kB ? 2 : 1, MW = kB ? 2 : 1, NW = kB ? 4 : 8,
                       BK = WF == AM_WF_INT4 ? 128 : 64, NST = WF == AM_WF_INT4 ? 3 : (WF == AM_WF_INT8 ? 4 : 3), BPC = 2;
};
//   256 x 256, 512 threads, one block per CU: the fewest X and W bytes per MFMA
template <int WF> struct TileCfg<WF, kT256x256> {
  static constexpr int MT = 8, NT = 4, MW = 2, NW = 4, BK = 64, NST = WF == AM_WF_BF16 ? 2 : 3, BPC = 1;
};
template <int WF, int TILE>
struct Shape : TileCfg<WF, TILE> {
  using C = TileCfg<WF, TILE>;
  static constexpr bool kI4 = WF == AM_WF_INT4;
  static constexpr int kWaves = C::MW * C::NW;
  static constexpr int kThreads = 64 * kWaves;
  static constexpr int kBM = 16 * C::MT * C::MW, kBN = 16 * C::NT * C::NW;
  static constexpr int kXRow = C::BK * 2;                      // X row bytes per k step
  static constexpr int kRowB = WRow<WF>::kBytes * C::BK / 64;  // W row bytes per k step
  static constexpr int kXSt = kBM * kXRow;         // X bytes per stage
  static constexpr int kWSt = kBN * kRowB;         // W bytes per stage
  static constexpr int kStg = kXSt + kWSt;
  static constexpr int kScSlot = kBN * 4;          // INT4: one dword per weight row
  static constexpr int kScSlots = 4;               // groups whose scales may be in LDS
  static constexpr int kEpi = kBM * (kBN + 8) * 2;  // the epilogue's bf16 tile
  static constexpr int kRing = C::NST * kStg + (kI4 ? kScSlots * kScSlot : 0);
  static constexpr int kLds = kRing > kEpi ? kRing : kEpi;
  static constexpr int kXi = kXSt / 1024 / kWaves;  // X DMA instructions per wave per step
  static constexpr int kWi = kWSt / 1024 / kWaves;  // W DMA instructions per wave per step
  static constexpr int kLoads = kXi + kWi + (kI4 ? 1 : 0);  // + the INT4 scale dword
  static constexpr int kTiles = C::MT * C::NT;              // MFMA tiles per wave
  static constexpr int kPartWave = kTiles * 64 * 4;         // fp32 partials of a wave
  static_assert(C::BK % 64 == 0, "the loop's operand sets alternate over an even number of slices");
  static_assert(kXi >= 1 && kXi * kWaves * 1024 == kXSt, "X stage must be whole DMA instructions per wave");
  static_assert(kWi >= 1 && kWi * kWaves * 1024 == kWSt, "W stage must be whole DMA instructions per wave");
  static_assert(C::NST <= 6 && kLoads * (C::NST - 1) < 64, "the memory counter must hold the steps in flight");
  static_assert(!kI4 || C::NST <= kScSlots || C::BK == 64, "a group's scales must outlive the steps in flight");
};

// Slot of 16-byte chunk c of weight row n within the row's k-step bytes (RB of them).
template <int RB>
__device__ __forceinline__ int wslot(int n, int c) {
  if constexpr (RB == 32) return c ^ ((n >> 3) & 1);
  else if constexpr (RB == 64) return c ^ ((n >> 2) & 3);
  else return c ^ ((n >> 1) & 7);
}

// X row r's 16-byte chunk c sits at slot c ^ xsw(r) of the row: with 128-byte rows 8
// consecutive rows, and 16 rows taken as two parity classes, land in distinct LDS
// banks; with 256-byte rows all 16 do.
template <int BK>
__device__ __forceinline__ int xsw(int r) {
  if constexpr (BK == 128) return r & 15;
  else return (r >> 1) & 7;
}

enum I4Epi { kI4Store = 0, kI4Residual = 1, kI4Split = 2, kI4SiluMul = 3, kI4QkvRope = 4 };

struct I4Args {
  const uint16_t* x;  // bf16 [M][K]
  const uint8_t* w;   // [N][K]: INT4 device order (K/2 bytes a row), INT8 q+128 bytes, or bf16
  const void* s;      // INT4: fp16 scales [N][K/group]; INT8: fp32 row scales [N]; bf16: unused
  int32_t M, N, K, group;  // group: the INT4 group; 128 (the split-K unit) for INT8 and bf16
  int32_t ffn;  // SiLU-Mul: rows [0, ffn) gate, [ffn, 2 ffn) up
  uint16_t* out0;
  uint16_t* out1;
  uint16_t* out2;
  int32_t c1, c2;             // split: columns [0,c1) -> out0, [c1,c2) -> out1, [c2,N) -> out2
  const uint16_t* residual;   // [M][N] bf16, may alias out0
  int32_t vec;                // 1: 16-byte output chunks (row strides and split columns % 8 == 0, aligned)
  int32_t splits;             // k splits per tile (1: none)
  float* part;                // [tiles][splits][waves][MT NT][64] x 4 fp32 partial accumulators
  unsigned* tickets;          // [tiles], zero between launches
  // q|k|v + RoPE + KV epilogue: columns [0,c1) q -> out0 (rotated), [c1,c2) k (rotated)
  // and [c2,N) v into the cache planes at position *start + row
  const float* cos_tab;       // [cap][hd/2]
  const float* sin_tab;
  const int64_t* start;
  uint16_t* kc;
  uint16_t* vc;
  KvRows kv;
  int32_t hd, cap;
  int32_t* err;               // optional: set when a row's position is outside [0, cap)
};

// 8 bytes q+128 -> 8 bf16 values q (exact), in byte order: signed byte conversions, and
// the top halves of the fp32 bits of small integers are their bf16 encodings.
__device__ __forceinline__ bf16x8_t bytes8(uint2 v) {
  const uint32_t w[2] = {v.x ^ 0x80808080u, v.y ^ 0x80808080u};
  uint32_t d[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t word = w[i >> 1] >> (16 * (i & 1));
    const float lo = static_cast<float>(static_cast<int8_t>(word)), hi = static_cast<float>(static_cast<int8_t>(word >> 8));
    d[i] = __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
  }
  return __builtin_bit_cast(bf16x8_t, make_uint4(d[0], d[1], d[2], d[3]));
}

// signed 4-bit value of the low nibble of byte B of v, over 16 (v_cvt_off_f32_i4)
template <int B>
__device__ __forceinline__ uint32_t nibble16(uint32_t v) {
  uint32_t d;
  if constexpr (B == 0) asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(d) : "v"(v));
  else if constexpr (B == 1) asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(d) : "v"(v));
  else if constexpr (B == 2) asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(d) : "v"(v));
  else asm("v_cvt_off_f32_i4_sdwa %0, %1 dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(d) : "v"(v));
  return d;
}

constexpr uint32_t kZeroCodes = 0x88888888u;  // 8 nibbles of q = 0

// 8 nibbles q+8 in device tile order -> 8 bf16 values q / 16 (exact) in k order: the
// nibbles of k 0, 4, 1, 5 are the low halves of bytes 0..3, those of k 2, 6, 3, 7 the
// high halves.
__device__ __forceinline__ bf16x8_t unpack8(uint32_t word) {
  const uint32_t lo = word ^ kZeroCodes, hi = lo >> 4;
  const uint32_t d0 = __builtin_amdgcn_perm(nibble16<2>(lo), nibble16<0>(lo), 0x07060302u);
  const uint32_t d1 = __builtin_amdgcn_perm(nibble16<2>(hi), nibble16<0>(hi), 0x07060302u);
  const uint32_t d2 = __builtin_amdgcn_perm(nibble16<3>(lo), nibble16<1>(lo), 0x07060302u);
  const uint32_t d3 = __builtin_amdgcn_perm(nibble16<3>(hi), nibble16<1>(hi), 0x07060302u);
  return __builtin_bit_cast(bf16x8_t, make_uint4(d0, d1, d2, d3));
}

// Global -> LDS DMA of 16 (4) bytes per lane: lane L's bytes at base + off land at LDS
// byte lds + 16 (4) L.  Written as asm because the compiler counts the builtin's LDS
// write against every later LDS read and may wait for all DMA in flight before each one
// (vmcnt(0) in the k loop); the loop waits for exactly the steps it needs.  No register
// is written, and the address registers are read at issue.
__device__ __forceinline__ void dma16(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
__device__ __forceinline__ void dma4(const void* base, uint32_t off, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}

// Weight row of local tile row r.  SiLU-Mul: the first half of a tile's rows are gate
// features, the second half the up rows of the same features.  RoPE with heads wider
// than the tile: the first half of the rows lie in the first half of a head, the second
// half are their rotation partners d/2 later.
template <int EPI, int BN>
__device__ __forceinline__ int32_t wrow(const I4Args& p, int32_t tn, int32_t r) {
  if constexpr (EPI == kI4SiluMul) return r < BN / 2 ? tn * (BN / 2) + r : p.ffn + tn * (BN / 2) + (r - BN / 2);
  if constexpr (EPI == kI4QkvRope && BN < 128) {
    if (p.hd > BN) {
      const int32_t per = p.hd / BN, head = tn / per, base = head * p.hd + (tn - head * per) * (BN / 2);
      return r < BN / 2 ? base + r : base + (p.hd >> 1) + (r - BN / 2);
    }
  }
  const int32_t g = tn * BN + r;
  return g < p.N ? g : 0;
}

// Wait for this wave's LDS reads, in a form the compiler's own wait insertion sees (an asm
// wait it does not): it then knows that nothing is pending.
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xC07F); }

// Wait until at most AHEAD (<= MAX) steps of this wave's DMA are in flight, then a plain
// s_barrier, as one asm statement (no memory access moves across it; a fenced barrier
// would also wait for the younger steps' DMA).
template <int LOADS, int MAX>
__device__ __forceinline__ void wait_barrier(int ahead) {
  if constexpr (MAX > 0) {
    if (ahead >= MAX)
      asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(MAX * LOADS) : "memory");
    else
      wait_barrier<LOADS, MAX - 1>(ahead);
  } else {
    asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  }
}

template <int WF, int EPI, int TILE>
__global__ __launch_bounds__((Shape<WF, TILE>::kThreads), (Shape<WF, TILE>::BPC)) void gemm_mfma_kernel(I4Args p) {
  using S = Shape<WF, TILE>;
  constexpr int BM = S::kBM, BN = S::kBN, NST = S::NST, STG = S::kStg, MT = S::MT, NT = S::NT, NW = S::NW;
  constexpr int BK = S::BK, KK = BK / 32, XST = S::kXSt, XROW = S::kXRow, RB = S::kRowB;
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / NW, wn = wave % NW;
  // arguments of the epilogue in registers now (see the loop)
  uint16_t* out0 = p.out0;
  const uint16_t* residual = p.residual;
  asm volatile("" : "+s"(out0), "+s"(residual));

  // tile mapping: bands of 8 M-tiles, N fastest inside a band
  const int32_t tiles_m = (p.M + BM - 1) / BM;
  const int32_t tiles_n = EPI == kI4SiluMul ? p.ffn / (BN / 2) : (p.N + BN - 1) / BN;
  const int32_t tiles = tiles_m * tiles_n;
  // Block b runs on XCD b mod 8, each with an L2 of its own: XCD x takes the x-th
  // contiguous eighth of the launch's tiles, so the M tiles that share a weight tile (and
  // the N tiles that share rows of X) meet in one L2.
  const int32_t xq = gridDim.x >> 3, xr = gridDim.x & 7, xcd = blockIdx.x & 7;
  const int32_t lin = xcd * xq + min(xcd, xr) + static_cast<int32_t>(blockIdx.x >> 3);
  const int32_t bid = lin / p.splits;
  const int32_t split = lin - bid * p.splits;
  const int32_t per_band = 8 * tiles_n;
  const int32_t b0 = bid / per_band, rem = bid - b0 * per_band;
  const int32_t bands_m = min(tiles_m - b0 * 8, 8);
  const int32_t tm = b0 * 8 + rem % bands_m, tn = rem / bands_m;
  const int32_t m0 = tm * BM;

  const int32_t ng = p.K / p.group;
  const int32_t spg = p.group / BK;  // k steps per group
  // this split's groups [g0, g1) = k steps [k0, k0 + nk)
  const int32_t g0 = split * ng / p.splits, g1 = (split + 1) * ng / p.splits;
  const int32_t k0 = g0 * spg, nk = (g1 - g0) * spg;

  // ---- DMA sources of this lane ----
  // X: an instruction moves 1 KB, 1024 / XROW rows
  constexpr int XPI = 1024 / XROW, XCH = XROW / 16;
  uint32_t xsrc[S::kXi];  // byte offsets (M * K and N rows stay below 2^31 elements and bytes)
#pragma unroll
  for (int i = 0; i < S::kXi; ++i) {
    const int r = (wave * S::kXi + i) * XPI + lane / XCH;
    const int c = (lane % XCH) ^ xsw<BK>(r);
    const int32_t gr = m0 + r < p.M ? m0 + r : 0;
    xsrc[i] = static_cast<uint32_t>((static_cast<int64_t>(gr) * p.K + 8 * c) * 2);
  }
  // INT8: the fp32 scales of this lane's output columns, loaded ahead of every DMA
  float rs[NT];
  if constexpr (WF == AM_WF_INT8) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      rs[nt] = static_cast<const float*>(p.s)[wrow<EPI, BN>(p, tn, (wn * NT + nt) * 16 + (lane & 15))];
  }
  // W: instruction i of wave w fills 1 KB of the stage's W rows; lane L's 16 bytes land
  // at row (1024 (w kWi + i) + 16 L) / kRowB, slot ((16 L) mod kRowB) / 16, so it fetches
  // the chunk whose slot that is (the slot map is an XOR, its own inverse)
  const int64_t wrow_bytes = static_cast<int64_t>(p.K) / BK * RB;
  uint32_t wsrc[S::kWi];
#pragma unroll
  for (int i = 0; i < S::kWi; ++i) {
    const int o = (wave * S::kWi + i) * 1024 + 16 * lane;
    const int r = o / RB, slot = (o % RB) / 16;
    wsrc[i] = static_cast<uint32_t>(static_cast<int64_t>(wrow<EPI, BN>(p, tn, r)) * wrow_bytes + 16 * wslot<RB>(r, slot));
  }
  // INT4 scales: lane -> weight row 64 (wave % (BN / 64)) + lane (the other waves repeat
  // the same rows); the dword holding its fp16
  const int sr = (wave % (BN / 64)) * 64 + lane;
  const int64_t sbase = S::kI4 ? static_cast<int64_t>(wrow<EPI, BN>(p, tn, sr)) * ng : 0;

  const uint32_t lds0 = static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lvoid*)(lds)));
  auto issue = [&](int32_t j) {  // local step j = k step k0 + j
    const int32_t ks = k0 + j;
    const uint32_t st = lds0 + (j % NST) * STG;
    const uint8_t* xb = reinterpret_cast<const uint8_t*>(p.x) + static_cast<int64_t>(ks) * XROW;
    const uint8_t* wb = p.w + static_cast<int64_t>(ks) * RB;
#pragma unroll
    for (int i = 0; i < S::kXi; ++i) dma16(xb, xsrc[i], st + (wave * S::kXi + i) * 1024);
#pragma unroll
    for (int i = 0; i < S::kWi; ++i) dma16(wb, wsrc[i], st + XST + (wave * S::kWi + i) * 1024);
    if constexpr (S::kI4) {
      const int32_t g = ks / spg;
      const int64_t se = sbase + g;  // fp16 element; its dword, aligned down
      dma4(p.s, static_cast<uint32_t>((se * 2) & ~int64_t{3}),
           lds0 + NST * STG + (g & (S::kScSlots - 1)) * S::kScSlot + (wave % (BN / 64)) * 256);
    }
  };

  const f32x4_t zero4 = f32x4_t{0.f, 0.f, 0.f, 0.f};
  f32x4_t acc[MT][NT];
#pragma unroll
  for (int i = 0; i < MT; ++i)
#pragma unroll
    for (int j = 0; j < NT; ++j) acc[i][j] = zero4;

  // LDS read offsets of this lane (within a stage).  Lane group kb takes the 8 k values
  // 32 kk + 8 kb + ... of MFMA kk.
  const int kb = lane >> 4;
  int aoff[MT][KK], boff[NT][KK];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int r = (wm * MT + mt) * 16 + (lane & 15);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) aoff[mt][kk] = r * XROW + 16 * ((kk * 4 + kb) ^ xsw<BK>(r));
  }
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    const int n = (wn * NT + nt) * 16 + (lane & 15);
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) {
      if constexpr (WF == AM_WF_INT4)
        boff[nt][kk] = XST + n * RB + 16 * wslot<RB>(n, kk) + 4 * kb;
      else if constexpr (WF == AM_WF_INT8)
        boff[nt][kk] = XST + n * RB + 16 * wslot<RB>(n, 2 * kk + (kb >> 1)) + 8 * (kb & 1);
      else
        boff[nt][kk] = XST + n * RB + 16 * wslot<RB>(n, 4 * kk + kb);
    }
  }
  // scale of this lane's column of tile nt in group g: the half of the slot dword that
  // holds element (row * ng + g)
  // (tiles, features and heads start at even rows, so a row's parity is its lane's)
  const int soff = NST * STG + (wn * NT * 16 + (lane & 15)) * 4;
  const int shalf = lane & ng & 1;

  // Operands of one MFMA k slice: A as read, B in storage format and as bf16 (two slices)
  using RawB = std::conditional_t<WF == AM_WF_INT4, uint32_t, std::conditional_t<WF == AM_WF_INT8, uint2, uint4>>;
  uint4 oa[MT];
  RawB ob[NT];
  bf16x8_t bfr[2][NT];
  uint32_t sraw[NT];       // INT4: the group's scale dwords
  bool dead = false;       // INT4: some lane's scale of the group is zero
  float sc[NT];            // INT4: the scale the sums are in units of
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) {
    sc[nt] = 1.0f;
    sraw[nt] = 0u;
  }
  auto fetch_a = [&](const uint8_t* st, int kk, int mt) { oa[mt] = *reinterpret_cast<const uint4*>(st + aoff[mt][kk]); };
  auto fetch_b = [&](const uint8_t* st, int kk) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      if constexpr (WF == AM_WF_BF16)
        bfr[kk & 1][nt] = __builtin_bit_cast(bf16x8_t, *reinterpret_cast<const RawB*>(st + boff[nt][kk]));
      else
        ob[nt] = *reinterpret_cast<const RawB*>(st + boff[nt][kk]);
    }
  };
  auto convert = [&](int nt, int kk) {
    if constexpr (WF == AM_WF_INT4) bfr[kk & 1][nt] = unpack8(ob[nt]);
    else if constexpr (WF == AM_WF_INT8) bfr[kk & 1][nt] = bytes8(ob[nt]);
  };
  auto fetch_scales = [&](int32_t g) {
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      sraw[nt] = *reinterpret_cast<const uint32_t*>(lds + soff + nt * 64 + (g & (S::kScSlots - 1)) * S::kScSlot);
  };
  auto group_bits = [&](int32_t g, int nt) {
    return ((shalf + g) & 1) ? (sraw[nt] >> 16) : (sraw[nt] & 0xFFFFu);
  };
  // A group begins: the sums so far change to its unit; a zero scale leaves them in theirs.
  // (The smallest fp16 scale is 2^-24: sums below 2^108 stay finite in any unit.)
  auto open_group = [&](int32_t g, float (&ratio)[NT]) {
    bool zero = false;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt) {
      float s = static_cast<float>(__builtin_bit_cast(_Float16, static_cast<uint16_t>(group_bits(g, nt))));
      zero = zero || s == 0.0f;
      if (s == 0.0f) s = sc[nt];
      // sc / s: reciprocal and one correction (not where that meets an infinity)
      const float inv = __builtin_amdgcn_rcpf(s);
      float q = sc[nt] * inv;
      const float e = __builtin_fmaf(-q, s, sc[nt]);
      if (e == e) q = __builtin_fmaf(e, inv, q);
      ratio[nt] = s == sc[nt] ? 1.0f : q;
      sc[nt] = s;
    }
    dead = __builtin_amdgcn_ballot_w64(zero) != 0;
  };
  // A group of zero scale adds nothing: its codes in step j become 0 (the quantizer stores
  // 0 with such a scale, other packers may not), the first slice's in the registers they
  // were converted to and the others in the LDS words that this lane reads.  The branch,
  // which ordinary weights never take, costs up to 1% of a launch (512 x 28672 x 4096 133.8
  // -> 135.3 us); masking every conversion cost 1-6%, and a zero scale taken as 2^-60 left
  // sums of 1e-17 for rows of zero scales and overflowed above 5e21.
  auto drop_zero_scale = [&](int32_t g, int32_t j) {
    if constexpr (S::kI4) {
      if (__builtin_expect(dead, 0)) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          if ((group_bits(g, nt) & 0x7FFFu) == 0u) {
            bfr[0][nt] = bf16x8_t{};
#pragma unroll
            for (int kk = 1; kk < KK; ++kk) *reinterpret_cast<uint32_t*>(lds + (j % NST) * STG + boff[nt][kk]) = kZeroCodes;
          }
        wait_lds();
      }
    }
  };
  // MFMAs of slice kk; RESCALE: the first slice of an INT4 group.  As soon as a row of
  // tiles is issued its A registers take the operand of the next slice (kn of step sn),
  // and in the second half of the rows the next slice's weights are converted: LDS reads
  // and conversions run behind the MFMAs, kept there by the barriers to reordering.
  auto slice = [&](int kk, const uint8_t* sn, int kn, auto rescale, const float (&ratio)[NT]) {
    constexpr bool RESCALE = decltype(rescale)::value;
    fetch_b(sn, kn);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const bf16x8_t af = __builtin_bit_cast(bf16x8_t, oa[mt]);
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) {
        if constexpr (RESCALE) {
#pragma unroll
          for (int r = 0; r < 4; ++r) acc[mt][nt][r] *= ratio[nt];
        }
        acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bfr[kk & 1][nt], acc[mt][nt], 0, 0, 0);
      }
      fetch_a(sn, kn, mt);
      constexpr int H = MT / 2;
      if constexpr (WF != AM_WF_BF16) {
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          if (H + nt * H / NT == mt) convert(nt, kk + 1);
      }
      if constexpr (MT > 4 || WF != AM_WF_BF16) __builtin_amdgcn_sched_barrier(0);
    }
  };

  // prologue: steps 0 .. NST-1 in flight, then the first slice's operands
#pragma unroll
  for (int i = 0; i < NST; ++i)
    if (i < nk) issue(i);
  wait_barrier<S::kLoads, NST - 1>(nk - 1);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) fetch_a(lds, 0, mt);
  fetch_b(lds, 0);
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) convert(nt, 0);
  if constexpr (S::kI4) fetch_scales(g0);
  // no scalar load may be pending when the loop begins, or the compiler waits for all LDS
  // reads at each use in it
  __builtin_amdgcn_sched_barrier(0);
  wait_lds();
  __builtin_amdgcn_sched_barrier(0);

  // One slice of operands is read from LDS while the MFMAs of the slice before run.  The
  // last slice of a step runs after the barrier that ends the step: every wave has then
  // read all of the step, so its slot takes the DMA of step j + NST, and the next
  // step's first operands are read behind those MFMAs (after the last step: bytes of an
  // older one, never used).
  auto step = [&](int32_t j, int32_t next_group, auto first, const float (&ratio)[NT]) {
    const uint8_t* st = lds + (j % NST) * STG;
    const uint8_t* sn = lds + ((j + 1) % NST) * STG;
    slice(0, st, 1, first, ratio);
#pragma unroll
    for (int kk = 1; kk + 1 < KK; ++kk) slice(kk, st, kk + 1, std::false_type{}, ratio);
    if (j + 1 < nk) {
      wait_lds();
      wait_barrier<S::kLoads, NST - 2>(nk - 2 - j);
      if (j + NST < nk) issue(j + NST);
      if (S::kI4 && next_group >= 0) fetch_scales(next_group);
    }
    slice(KK - 1, sn, 0, std::false_type{}, ratio);
  };
  float ratio[NT];
#pragma unroll
  for (int nt = 0; nt < NT; ++nt) ratio[nt] = 1.0f;
  int32_t j = 0;
  if constexpr (S::kI4) {
    for (int32_t g = g0; g < g1; ++g) {
      open_group(g, ratio);
      drop_zero_scale(g, j);
      step(j, spg == 1 ? g + 1 : -1, std::true_type{}, ratio);
      ++j;
      for (int32_t t = 1; t < spg; ++t, ++j) {
        drop_zero_scale(g, j);
        step(j, t + 1 == spg ? g + 1 : -1, std::false_type{}, ratio);
      }
    }
  } else {
    for (; j < nk; ++j) step(j, -1, std::false_type{}, ratio);
  }
  if constexpr (S::kI4) {
    // out of the last group's unit; the operands were q / 16
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[mt][nt][r] *= 16.0f * sc[nt];
  }

  if (p.splits > 1) {
    // partial of this split: device-scope (sc1) 16-byte buffer stores of the wave's
    // region, acknowledged before the ticket
    constexpr int kTiles = S::kTiles, kWaveBytes = S::kPartWave * 4;
    auto region = [&](int32_t sp) {
      float* at = p.part + ((static_cast<int64_t>(bid) * p.splits + sp) * S::kWaves + wave) * S::kPartWave;
      return __builtin_amdgcn_make_buffer_rsrc(at, 0, kWaveBytes, kRawBufferFlags);
    };
    const __amdgpu_buffer_rsrc_t rmine = region(split);
#pragma unroll
    for (int i = 0; i < kTiles; ++i)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[i / NT][i % NT]), rmine, (i * 64 + lane) * 16, 0,
                                             kCpolSc1);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    __shared__ unsigned last;
    if (tid == 0)
      last = __hip_atomic_fetch_add(&p.tickets[bid], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) ==
             static_cast<unsigned>(p.splits - 1);
    __syncthreads();
    if (!last) return;
    // the tile's sum in split order, one row of MFMA tiles at a time (this split's own
    // partial is read back too: its registers are free for the loads in flight)
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      f32x4_t sum[NT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) sum[nt] = zero4;
#pragma unroll 2
      for (int sp = 0; sp < p.splits; ++sp) {
        const __amdgpu_buffer_rsrc_t rsrc = region(sp);
        u32x4_t v[NT];
#pragma unroll
        for (int nt = 0; nt < NT; ++nt)
          v[nt] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, ((mt * NT + nt) * 64 + lane) * 16, 0, kCpolSc1);
#pragma unroll
        for (int nt = 0; nt < NT; ++nt) sum[nt] += __builtin_bit_cast(f32x4_t, v[nt]);
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt) acc[mt][nt] = sum[nt];
    }
    if (tid == 0) __hip_atomic_store(&p.tickets[bid], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if constexpr (WF == AM_WF_INT8) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[mt][nt][r] *= rs[nt];
  }
  // ---- epilogue: round(acc) as a bf16 tile in LDS (lane holds D[4*(lane/16)+r][lane%16]
  // of each 16x16 tile), then 16-byte row chunks ----
  constexpr int TS = BN + 8;  // tile row stride in bf16 (16-byte pad)
  uint16_t* T = reinterpret_cast<uint16_t*>(lds);
  __syncthreads();  // every wave is done with the ring
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        T[((wm * MT + mt) * 16 + 4 * (lane >> 4) + r) * TS + (wn * NT + nt) * 16 + (lane & 15)] =
            f32_to_bf16_bits(acc[mt][nt][r]);
  __syncthreads();

  if constexpr (EPI == kI4QkvRope) {
    // A thread takes a chunk pair: 8 columns of the first half of a head and the 8
    // columns d/2 later (the RoPE partners), from the rounded tile.  q and k pairs are
    // rotated in fp32 from the bf16 values and rounded once (the RoPE node); k and v
    // go straight to the cache rows of their positions (the KVCacheUpdate node).
    const int32_t d = p.hd, half = d >> 1;
    // tile columns of a head or of a piece of one (wrow): the partner of a first-half
    // column lies pd / 2 columns later
    const int32_t pd = min(d, BN), ph = pd >> 1, hpt = pd >> 4;  // hpt: chunk pairs per pd columns
    const int32_t per = d / pd;                                  // pieces per head
    const int64_t start = *p.start;
    constexpr int PPR = BN / 16;  // chunk pairs per tile row (BN is a multiple of pd)
    for (int c = tid; c < BM * PPR; c += S::kThreads) {
      const int row = c / PPR, pr = c % PPR;
      const int32_t gm = m0 + row;
      const int col = (pr / hpt) * pd + (pr % hpt) * 8;  // tile column of the first-half chunk
      const int32_t piece = tn % per;                    // 0 unless the head is wider than the tile
      const int i0 = piece * ph + (pr % hpt) * 8;        // offset of the chunk inside its head
      const int32_t gn = per > 1 ? (tn / per) * d + i0 : tn * BN + col;
      if (gm >= p.M || gn >= p.N) continue;
      const uint4 a1 = *reinterpret_cast<const uint4*>(T + row * TS + col);
      const uint4 a2 = *reinterpret_cast<const uint4*>(T + row * TS + col + ph);
      const int64_t pos = start + gm;
      const bool ok = pos >= 0 && pos < p.cap;
      uint4 o1 = a1, o2 = a2;
      if (gn < p.c2 && ok) {
        const float4* cp = reinterpret_cast<const float4*>(p.cos_tab + pos * half + i0);
        const float4* sp = reinterpret_cast<const float4*>(p.sin_tab + pos * half + i0);
        const float4 c0 = cp[0], c1 = cp[1], s0 = sp[0], s1 = sp[1];
        const float cv[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
        const float sv[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
        const uint32_t w1[4] = {a1.x, a1.y, a1.z, a1.w}, w2[4] = {a2.x, a2.y, a2.z, a2.w};
        uint32_t r1[4], r2[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          uint32_t y1[2], y2[2];
#pragma unroll
          for (int hh = 0; hh < 2; ++hh) {
            const float x1 = bf16_bits_to_f32(hh ? (w1[q] >> 16) : (w1[q] & 0xFFFFu));
            const float x2 = bf16_bits_to_f32(hh ? (w2[q] >> 16) : (w2[q] & 0xFFFFu));
            const float cc = cv[2 * q + hh], sn = sv[2 * q + hh];
            float r1v, r2v;
            rope_rotate(x1, x2, cc, sn, r1v, r2v);
            y1[hh] = f32_to_bf16_bits(r1v);
            y2[hh] = f32_to_bf16_bits(r2v);
          }
          r1[q] = y1[0] | (y1[1] << 16);
          r2[q] = y2[0] | (y2[1] << 16);
        }
        o1 = make_uint4(r1[0], r1[1], r1[2], r1[3]);
        o2 = make_uint4(r2[0], r2[1], r2[2], r2[3]);
      }
      if (!ok && p.err != nullptr) *p.err = 1;
      if (gn < p.c1) {
        uint16_t* dst = out0 + static_cast<int64_t>(gm) * p.c1 + gn;
        *reinterpret_cast<uint4*>(dst) = o1;
        *reinterpret_cast<uint4*>(dst + half) = o2;
      } else if (ok) {
        const bool isk = gn < p.c2;
        const int32_t hc = isk ? gn - p.c1 : gn - p.c2;
        const int64_t row = p.kv.WriteRow(0, hc / d, pos);
        if (row >= 0) {
          uint16_t* dst = (isk ? p.kc : p.vc) + row + i0;
          *reinterpret_cast<uint4*>(dst) = o1;
          *reinterpret_cast<uint4*>(dst + half) = o2;
        }
      }
    }
    return;
  }

  if constexpr (EPI == kI4SiluMul) {
    constexpr int CPR = BN / 16;  // 16-byte output chunks per row (BN/2 features)
    constexpr int IT = BM * CPR / S::kThreads;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int c = tid + S::kThreads * i, row = c / CPR, cc = c % CPR;
      const int32_t gm = m0 + row;
      if (gm >= p.M) continue;
      const uint16_t* gt = T + row * TS + cc * 8;
      const uint16_t* ut = gt + BN / 2;
      uint16_t* o = out0 + static_cast<int64_t>(gm) * p.ffn + tn * (BN / 2) + cc * 8;
      if (p.vec) {
        const uint4 gv = *reinterpret_cast<const uint4*>(gt), uv = *reinterpret_cast<const uint4*>(ut);
        const uint32_t gw[4] = {gv.x, gv.y, gv.z, gv.w}, uw[4] = {uv.x, uv.y, uv.z, uv.w};
        uint32_t ow[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          ow[q] = f32_to_bf16_bits(silu_ref(bf16_bits_to_f32(gw[q] & 0xFFFFu)) * bf16_bits_to_f32(uw[q] & 0xFFFFu)) |
                  (static_cast<uint32_t>(
                       f32_to_bf16_bits(silu_ref(bf16_bits_to_f32(gw[q] >> 16)) * bf16_bits_to_f32(uw[q] >> 16)))
                   << 16);
        *reinterpret_cast<uint4*>(o) = make_uint4(ow[0], ow[1], ow[2], ow[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = f32_to_bf16_bits(silu_ref(bf16_bits_to_f32(gt[e])) * bf16_bits_to_f32(ut[e]));
      }
    }
    return;
  }

  constexpr int CPR = BN / 8;  // 16-byte chunks per tile row
  constexpr int IT = BM * CPR / S::kThreads;
  // residual chunks first, all loads in flight (each thread reads only the chunks it
  // writes, so an aliased residual is read before it is overwritten)
  uint4 rres[EPI == kI4Residual ? IT : 1];
  if constexpr (EPI == kI4Residual) {
    if (p.vec) {
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        const int c = tid + S::kThreads * i, row = c / CPR, cc = c % CPR;
        const int32_t gm = m0 + row, gn = tn * BN + cc * 8;
        const int64_t idx = (gm < p.M && gn + 8 <= p.N) ? static_cast<int64_t>(gm) * p.N + gn : 0;
        rres[i] = *reinterpret_cast<const uint4*>(residual + idx);
      }
    }
  }
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int c = tid + S::kThreads * i, row = c / CPR, cc = c % CPR;
    const int32_t gm = m0 + row, gn = tn * BN + cc * 8;
    if (gm >= p.M || gn >= p.N) continue;
    const uint16_t* t = T + row * TS + cc * 8;
    // destination of column gn (split: the output whose column range holds it)
    uint16_t* o = out0;
    int32_t col = gn, ld = p.N, lim = p.N;  // lim: end of the destination's columns
    if constexpr (EPI == kI4Split) {
      if (gn < p.c1) {
        ld = lim = p.c1;
      } else if (gn < p.c2) {
        o = p.out1;
        col = gn - p.c1;
        ld = p.c2 - p.c1;
        lim = p.c2;
      } else {
        o = p.out2;
        col = gn - p.c2;
        ld = p.N - p.c2;
      }
    }
    uint16_t* dst = o + static_cast<int64_t>(gm) * ld + col;
    if (p.vec && gn + 8 <= lim) {
      const uint4 tv = *reinterpret_cast<const uint4*>(t);
      uint4 ov = tv;
      if constexpr (EPI == kI4Residual) {
        const uint32_t tw[4] = {tv.x, tv.y, tv.z, tv.w}, rw[4] = {rres[i].x, rres[i].y, rres[i].z, rres[i].w};
        uint32_t ow[4];
#pragma unroll
        for (int q = 0; q < 4; ++q)
          ow[q] = f32_to_bf16_bits(bf16_bits_to_f32(rw[q] & 0xFFFFu) + bf16_bits_to_f32(tw[q] & 0xFFFFu)) |
                  (static_cast<uint32_t>(f32_to_bf16_bits(bf16_bits_to_f32(rw[q] >> 16) + bf16_bits_to_f32(tw[q] >> 16)))
                   << 16);
        ov = make_uint4(ow[0], ow[1], ow[2], ow[3]);
      }
      *reinterpret_cast<uint4*>(dst) = ov;
    } else {
      // per element: the N edge, a chunk that straddles split outputs, unaligned rows
      for (int e = 0; e < 8 && gn + e < p.N; ++e) {
        int32_t ge = gn + e;
        uint16_t* de = out0 + static_cast<int64_t>(gm) * p.N + ge;
        if constexpr (EPI == kI4Split) {
          if (ge < p.c1) de = out0 + static_cast<int64_t>(gm) * p.c1 + ge;
          else if (ge < p.c2) de = p.out1 + static_cast<int64_t>(gm) * (p.c2 - p.c1) + (ge - p.c1);
          else de = p.out2 + static_cast<int64_t>(gm) * (p.N - p.c2) + (ge - p.c2);
        }
        uint16_t v = t[e];
        if constexpr (EPI == kI4Residual)
          v = f32_to_bf16_bits(bf16_bits_to_f32(residual[static_cast<int64_t>(gm) * p.N + ge]) + bf16_bits_to_f32(v));
        *de = v;
      }
    }
  }
}

// Tiles of a launch.
template <int WF, int EPI, int TILE>
int64_t TilesOf(const I4Args& p) {
  using S = Shape<WF, TILE>;
  constexpr int64_t BN = S::kBN;
  return CeilDiv(p.M, S::kBM) * (EPI == kI4SiluMul ? p.ffn / (BN / 2) : CeilDiv(p.N, BN));
}

constexpr int64_t kTicketRegion = 4096;               // bytes at the start of the workspace
constexpr int64_t kMaxSplitTiles = kTicketRegion / 4;  // tiles of a launch that may split

// Blocks of a shape that one CU holds at once, by LDS (160 KB per CU): two for the 64-row
// tiles and the 128 x 128 INT4 and INT8 ones, one for the others.
constexpr int64_t kLdsPerCu = 160 * 1024;
template <int WF, int TILE>
constexpr int BlocksPerCu() {
  return kLdsPerCu / Shape<WF, TILE>::kLds > 1 ? static_cast<int>(kLdsPerCu / Shape<WF, TILE>::kLds) : 1;
}

// Split-K count: the largest power of two up to `most` that keeps every split at >= 8
// groups (12 beyond 4 splits) and the launch within one round of resident blocks (bpc per
// CU).  512 rows of the 8B o projection, INT4: 47 us unsplit by estimate, 36 us with 4
// splits; 64 rows of its down projection: 24 us with 8 splits of 64 x 64 tiles, 54 us with
// 4 of 128 x 128.
int SplitsFor(int64_t tiles, int64_t groups, int64_t cus, int bpc, int most) {
  if (tiles > kMaxSplitTiles) return 1;
  int s = 1;
  while (s < most && tiles * s * 2 <= bpc * cus && groups / (s * 2) >= (s < 4 ? 8 : 12)) s *= 2;
  return s;
}

// 8 splits only for the small tiles (k of 12288 and more), 2 for the bf16 128 x 256 tile
// (its 4-split launches are within 3% of two splits of 128 x 128 and take twice the
// workspace).
template <int WF, int TILE>
constexpr int MaxSplits() {
  return TILE == kT64 || TILE == kT64W ? 8 : TILE == kT256 && WF == AM_WF_BF16 ? 2 : 4;
}
constexpr int32_t kFewRows = 256;

// Workspace layout: a fixed ticket region (one u32 per tile of a splitting launch),
// then the partials.  The region's size does not depend on the launch's shape, so
// launches of different shapes can share one workspace: no launch's partials land on
// another launch's tickets.
int64_t TicketBytes(int64_t) { return kTicketRegion; }
template <int WF, int TILE>
int64_t PartialBytes(int64_t tiles, int splits) {
  using S = Shape<WF, TILE>;
  return splits > 1 ? tiles * splits * S::kWaves * S::kPartWave * 4 : 0;
}

// Splits a launch of this tile runs with the given workspace.
template <int WF, int EPI, int TILE>
int SplitsOf(const I4Args& p, const void* ws, int64_t ws_bytes) {
  if (ws == nullptr) return 1;
  const int64_t tiles = TilesOf<WF, EPI, TILE>(p);
  const int s = SplitsFor(tiles, p.K / p.group, DeviceCUs(), BlocksPerCu<WF, TILE>(), MaxSplits<WF, TILE>());
  return s > 1 && TicketBytes(tiles) + PartialBytes<WF, TILE>(tiles, s) > ws_bytes ? 1 : s;
}

template <int WF, int EPI, int TILE>
am_status_code LaunchMfma(I4Args p, void* ws, int64_t ws_bytes, hipStream_t s) {
  using S = Shape<WF, TILE>;
  static const bool lds_ok =
      hipFuncSetAttribute(reinterpret_cast<const void*>(gemm_mfma_kernel<WF, EPI, TILE>),
                          hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds) == hipSuccess;
  if (!lds_ok) return SetLastError(AM_STATUS_INTERNAL, "gemm_i4: could not set the dynamic LDS size");
  const int64_t tiles = TilesOf<WF, EPI, TILE>(p);
  const int splits = SplitsOf<WF, EPI, TILE>(p, ws, ws_bytes);
  p.splits = splits;
  if (splits > 1) {
    p.tickets = static_cast<unsigned*>(ws);
    p.part = reinterpret_cast<float*>(static_cast<uint8_t*>(ws) + TicketBytes(tiles));
  }
  const int64_t blocks = tiles * splits;
  static const char* const names[] = {"store", "residual", "split", "silu_mul", "qkv_rope_kv"};
  const char* fmt = WF == AM_WF_INT4 ? "i4" : WF == AM_WF_INT8 ? "i8" : "bf16";
  RecordLaunch(blocks, S::kThreads, S::kLds, "gemm_%s<%s,bn=%d,splits=%d>", fmt, names[EPI], S::kBN, splits);
  hipLaunchKernelGGL((gemm_mfma_kernel<WF, EPI, TILE>), dim3(static_cast<unsigned>(blocks)), dim3(S::kThreads), S::kLds,
                     s, p);
  AM_RETURN_IF_LAUNCH_FAILED("gemm_i4");
  return AM_STATUS_OK;
}

// ---- choice of the tile ----
// Estimated time of a launch in us.  Compute: rounds of resident blocks, each a split's k
// steps at the measured time of a 64-value step with the CU full (2048 x 28672 x 4096, the
// 64 x 64 tile 2048 x 4096 x 4096, divided by rounds and steps); a last round that leaves
// one block to a CU that holds two runs its steps in 0.62 of that.  Weights: read at about
// 5 TB/s.  Split merge: every partial is stored at about 5 TB/s in all, and a tile's last
// block reads all of them back at what one CU reads (75 GB/s).  On the 8B shapes from 20
// to 2048 rows the estimates fall within a tenth to a fifth of the measured times and
// order the tiles as measured, up to ties (512 rows, q|k|v INT4: 128 x 128 46 us, 128 x
// 256 45 us, 256 x 256 55 us; estimated 48, 48, 63).
//                                128x128 128x256 64x64  64x128 256x256
constexpr float kStepUs[3][5] = {{1.20f, 1.13f, 0.46f, 0.73f, 2.05f},   // INT4, by Tile
                                 {1.08f, 1.03f, 0.45f, 0.69f, 1.82f},   // INT8
                                 {0.65f, 1.01f, 0.38f, 0.71f, 1.68f}};  // bf16
template <int WF, int EPI, int TILE>
float EstimateUs(const I4Args& p, const void* ws, int64_t ws_bytes) {
  using S = Shape<WF, TILE>;
  if (p.group % S::BK != 0) return 1e30f;
  if (EPI == kI4SiluMul && p.ffn % (S::kBN / 2) != 0) return 1e30f;
  constexpr float step = kStepUs[WF == AM_WF_INT4 ? 0 : WF == AM_WF_INT8 ? 1 : 2][TILE];
  const int64_t cus = DeviceCUs(), bpc = BlocksPerCu<WF, TILE>(), tiles = TilesOf<WF, EPI, TILE>(p);
  const int splits = SplitsOf<WF, EPI, TILE>(p, ws, ws_bytes);
  const int64_t blocks = tiles * splits, slots = cus * bpc, rest = blocks % slots;
  const float rounds = static_cast<float>(blocks / slots) + (rest == 0 ? 0.0f : rest <= cus && bpc > 1 ? 0.62f : 1.0f);
  constexpr float tile = S::kBM * S::kBN * 4;
  const float merge = splits > 1 ? 2.0f + static_cast<float>(splits + 1) * tile / 75e3f + static_cast<float>(blocks) * tile / 5e6f : 0.0f;
  const float weights = static_cast<float>(p.N) * (p.K / QBK) * WRow<WF>::kBytes / 5e6f;
  return std::max(rounds * static_cast<float>(p.K / QBK) / splits * step, weights) + merge;
}

// The tile with the smallest estimate, each at the most splits that SplitsFor allows with the
// workspace (fewer splits are not weighed against them).  The 64-row tiles take part up to
// 256 rows (above, they read each weight more often than a launch of wider tiles of the same
// estimate).
template <int WF, int EPI>
am_status_code LaunchWF(const I4Args& p, void* ws, int64_t ws_bytes, hipStream_t s) {
  constexpr int kFew = EPI == kI4SiluMul ? kT64W : kT64;
  const float few = p.M <= kFewRows ? EstimateUs<WF, EPI, kFew>(p, ws, ws_bytes) : 1e30f;
  const float t128 = EstimateUs<WF, EPI, kT128>(p, ws, ws_bytes), t256 = EstimateUs<WF, EPI, kT256>(p, ws, ws_bytes),
              big = EstimateUs<WF, EPI, kT256x256>(p, ws, ws_bytes);
  const float best = std::min(std::min(few, t128), std::min(t256, big));
  if (best == few) return LaunchMfma<WF, EPI, kFew>(p, ws, ws_bytes, s);
  if (best == t256) return LaunchMfma<WF, EPI, kT256>(p, ws, ws_bytes, s);
  if (best == big) return LaunchMfma<WF, EPI, kT256x256>(p, ws, ws_bytes, s);
  return LaunchMfma<WF, EPI, kT128>(p, ws, ws_bytes, s);
}

// The weight format picks the kernel (p.group: the INT4 group, 128 otherwise).
template <int EPI>
am_status_code LaunchI4Any(const I4Args& p, int32_t fmt, void* ws, int64_t ws_bytes, hipStream_t s) {
  switch (fmt) {
    case AM_WF_INT4: return LaunchWF<AM_WF_INT4, EPI>(p, ws, ws_bytes, s);
    case AM_WF_INT8: return LaunchWF<AM_WF_INT8, EPI>(p, ws, ws_bytes, s);
    default: return LaunchWF<AM_WF_BF16, EPI>(p, ws, ws_bytes, s);
  }
}

// Split-K unit along k: the INT4 group, 128 values for INT8 and bf16 weights.
int32_t SplitUnit(const am_gfx950_weight& w) { return w.format == AM_WF_INT4 ? w.group_size : 2 * QBK; }

bool Aligned16(const void* q) { return (reinterpret_cast<uintptr_t>(q) & 15u) == 0; }

}  // namespace

// bf16 activations with INT4 weights (group % 64 == 0 and K % group == 0), INT8
// per-channel weights (K % 128 == 0) or bf16 weights (K % 128 == 0).
bool GemmI4Eligible(const am_gfx950_weight& w, int64_t m, const void* x) {
  bool fmt = false;
  int64_t row_bytes = 0;
  if (w.format == AM_WF_INT4) {
    fmt = w.scales != nullptr && w.group_size > 0 && w.group_size % QBK == 0 && w.k % w.group_size == 0;
    row_bytes = w.k / 2;
  } else if (w.format == AM_WF_INT8) {
    fmt = w.scales != nullptr && w.k % (2 * QBK) == 0;
    row_bytes = w.k;
  } else if (w.format == AM_WF_BF16) {
    fmt = w.k % (2 * QBK) == 0;
    row_bytes = 2 * w.k;
  }
  return fmt && m > 0 && m * w.k < (int64_t{1} << 31) && w.n * row_bytes < (int64_t{1} << 31) &&
         m * w.n < (int64_t{1} << 31) && (reinterpret_cast<uintptr_t>(x) & 15u) == 0;
}

// Workspace that lets a launch of this shape, or of fewer rows, split K (0: none of them
// ever splits).  Fewer rows are fewer tiles, which split more often, so the largest need is
// looked for over all of them: at 4096 x 14336 a 37-row launch runs 8 splits and one of 3072
// rows none.  Sized by the longest launch alone, a session of 4096-row chunks ran a 37-token
// prompt through two INT4 8B layers in 433 us, now 292 as with chunks of 512.  The same bound
// serves every epilogue (the SiLU-Mul tiles are never more numerous) and every weight format.
int64_t GemmI4WorkspaceBytes(int64_t m, int64_t n, int64_t k, int64_t group) {
  if (m <= 0 || n <= 0 || k <= 0 || group <= 0 || k % group != 0) return 0;
  const int64_t cus = DeviceCUs();
  int64_t best = 0;
  auto shape = [&](auto tile, auto fmt) {
    constexpr int T = decltype(tile)::value, WF = decltype(fmt)::value;
    using S = Shape<WF, T>;
    const int64_t tiles_n = CeilDiv(n, S::kBN);
    const int64_t rows = T == kT64 || T == kT64W ? std::min<int64_t>(m, kFewRows) : m;
    for (int64_t tiles = tiles_n; tiles <= CeilDiv(rows, S::kBM) * tiles_n; tiles += tiles_n) {
      const int sp = SplitsFor(tiles, k / group, cus, BlocksPerCu<WF, T>(), MaxSplits<WF, T>());
      if (sp == 1) break;  // nor do more tiles
      best = std::max(best, TicketBytes(tiles) + PartialBytes<WF, T>(tiles, sp));
    }
  };
  auto tile = [&](auto t) {
    shape(t, std::integral_constant<int, AM_WF_INT4>{});
    shape(t, std::integral_constant<int, AM_WF_INT8>{});
    shape(t, std::integral_constant<int, AM_WF_BF16>{});
  };
  tile(std::integral_constant<int, kT128>{});
  tile(std::integral_constant<int, kT256>{});
  tile(std::integral_constant<int, kT256x256>{});
  tile(std::integral_constant<int, kT64>{});
  tile(std::integral_constant<int, kT64W>{});
  return best;
}

// q|k|v GEMM with the RoPE and KVCacheUpdate nodes in the epilogue (one sequence).
am_status_code GemmI4QkvRopeKv(const void* x, int64_t m, const am_gfx950_weight& w, const am_gfx950_prefill_rope_kv& r,
                               void* q_out, void* ws, int64_t ws_bytes, hipStream_t s) {
  if (!GemmI4Eligible(w, m, x)) return SetLastError(AM_STATUS_INVALID_ARGUMENT, "gemm: unsupported shape or weight");
  AM_CHECK_ARG(ws == nullptr || (Aligned16(ws) && ws_bytes >= 0), "gemm: workspace must be 16-byte aligned");
  AM_CHECK_ARG(r.head_dim == 64 || r.head_dim == 128, "prefill q|k|v RoPE: head_dim must be 64 or 128");
  AM_CHECK_ARG(r.hq > 0 && r.hkv > 0 && r.hq % r.hkv == 0 && w.n == (r.hq + 2 * r.hkv) * r.head_dim,
               "prefill q|k|v RoPE: the weight rows must be hq + 2 hkv heads");
  AM_CHECK_ARG(r.capacity > 0 && r.max_pos >= r.capacity && r.capacity * r.head_dim < (int64_t{1} << 31),
               "prefill q|k|v RoPE: bad capacity or table length");
  AM_CHECK_ARG(q_out && r.cos_tab && r.sin_tab && r.start_pos_dev && r.k_cache && r.v_cache,
               "prefill q|k|v RoPE: null pointer");
  AM_CHECK_ARG(Aligned16(q_out) && Aligned16(r.k_cache) && Aligned16(r.v_cache) && Aligned16(r.cos_tab) &&
                   Aligned16(r.sin_tab),
               "prefill q|k|v RoPE: q, the cache planes and the tables must be 16-byte aligned");
  I4Args p{};
  p.x = static_cast<const uint16_t*>(x);
  p.w = static_cast<const uint8_t*>(w.data);
  p.s = w.scales;
  p.M = static_cast<int32_t>(m);
  p.N = static_cast<int32_t>(w.n);
  p.K = static_cast<int32_t>(w.k);
  p.group = SplitUnit(w);
  p.out0 = static_cast<uint16_t*>(q_out);
  p.c1 = static_cast<int32_t>(r.hq * r.head_dim);
  p.c2 = static_cast<int32_t>((r.hq + r.hkv) * r.head_dim);
  p.vec = 1;
  p.splits = 1;
  p.cos_tab = r.cos_tab;
  p.sin_tab = r.sin_tab;
  p.start = r.start_pos_dev;
  p.kc = static_cast<uint16_t*>(r.k_cache);
  p.vc = static_cast<uint16_t*>(r.v_cache);
  p.hd = static_cast<int32_t>(r.head_dim);
  p.cap = static_cast<int32_t>(r.capacity);
  p.err = r.err_flag;
  if (auto st = MakeKvRows(r.pages, 0, r.capacity, r.hkv, r.head_dim, &p.kv); st != AM_STATUS_OK) return st;
  if (p.kv.err == nullptr) p.kv.err = r.err_flag;
  return LaunchI4Any<kI4QkvRope>(p, w.format, ws, ws_bytes, s);
}

am_status_code GemmI4(const void* x, int64_t m, const am_gfx950_weight& w, int32_t epi, void* out0, void* out1,
                      void* out2, int64_t c1, int64_t c2, const void* residual, void* ws, int64_t ws_bytes,
                      hipStream_t s) {
  if (!GemmI4Eligible(w, m, x)) return SetLastError(AM_STATUS_INVALID_ARGUMENT, "gemm: unsupported shape or weight");
  AM_CHECK_ARG(ws == nullptr || (Aligned16(ws) && ws_bytes >= 0), "gemm: workspace must be 16-byte aligned");
  I4Args p{};
  p.x = static_cast<const uint16_t*>(x);
  p.w = static_cast<const uint8_t*>(w.data);
  p.s = w.scales;
  p.M = static_cast<int32_t>(m);
  p.N = static_cast<int32_t>(w.n);
  p.K = static_cast<int32_t>(w.k);
  p.group = SplitUnit(w);
  p.out0 = static_cast<uint16_t*>(out0);
  p.out1 = static_cast<uint16_t*>(out1);
  p.out2 = static_cast<uint16_t*>(out2);
  p.c1 = static_cast<int32_t>(c1);
  p.c2 = static_cast<int32_t>(c2);
  p.residual = static_cast<const uint16_t*>(residual);
  p.splits = 1;
  // 16-byte chunks need every output row (and the residual's) to start 16-byte aligned
  bool vec = Aligned16(out0) && (!residual || Aligned16(residual));
  switch (epi) {
    case kI4Store: vec = vec && w.n % 8 == 0; break;
    case kI4Residual: vec = vec && w.n % 8 == 0; break;
    case kI4Split:
      vec = vec && c1 % 8 == 0 && c2 % 8 == 0 && w.n % 8 == 0 && (c2 == c1 || Aligned16(out1)) &&
            (c2 == w.n || Aligned16(out2));
      break;
    default: vec = vec && (w.n / 2) % 8 == 0; break;
  }
  p.vec = vec ? 1 : 0;
  switch (epi) {
    case kI4Store: return LaunchI4Any<kI4Store>(p, w.format, ws, ws_bytes, s);
    case kI4Residual:
      AM_CHECK_ARG(residual != nullptr, "gemm: residual epilogue without a residual");
      return LaunchI4Any<kI4Residual>(p, w.format, ws, ws_bytes, s);
    case kI4Split:
      AM_CHECK_ARG(0 < c1 && c1 <= c2 && c2 <= w.n && out0 && (c2 == c1 || out1) && (c2 == w.n || out2),
                   "gemm: bad column split");
      return LaunchI4Any<kI4Split>(p, w.format, ws, ws_bytes, s);
    case kI4SiluMul:
      AM_CHECK_ARG(w.n % 128 == 0, "gemm: SiLU-Mul needs 2*ffn rows with ffn a multiple of 64");
      p.ffn = static_cast<int32_t>(w.n / 2);
      return LaunchI4Any<kI4SiluMul>(p, w.format, ws, ws_bytes, s);
    default: return SetLastError(AM_STATUS_INVALID_ARGUMENT, "gemm: unknown epilogue");
  }
}

}  // namespace am
