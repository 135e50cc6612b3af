// Expert-major grouped experts with few rows per expert (batched decode, drafted
// tokens, short prompts) on the gfx950 block-scaled matrix cores: every bank kind.
//
// Reference: affine_expert_forward_batched (src/cachalot/model/expert_affine.py:84-99),
// routed_expert_forward_sgmm / _batched (fp4_sgmm_metal.py:318-333,
// moe_prefill_batched.py:31-61), called per expert from moe_prefill_grouped.py:420-467.
// Rounding points: g = bf16(x W1), u = bf16(x W3), h = bf16(silu(min(g, L)) * clip(u,
// +-L) * w), y = bf16(h W2); the products accumulate in fp32.  Activations as two fp8
// planes per 32-element block, as in prefill_mx.hip.
//
// What bounds it: the weight bytes of the touched experts, each read once per tile of TPT
// rows, so the kernel is a weight stream.  An item is 64 weight rows (gate/up: 32 of W1 and
// the same 32 of W3; down: 64 of W2) of one tile for the whole K, and the four waves of a
// workgroup take its macros of K (MC chunks of 128) in turn, so that at any time it reads
// long contiguous runs of its rows.  (Waves owning 64 rows each, 256 per workgroup, read the
// same bytes at 4.0 against 5.3 TB/s for FP4 at 24 tokens.)  A wave keeps its next macros'
// codes in flight in registers, 16 bytes per lane and load; its share of the A planes (only
// the rows that exist) goes through an LDS ring of its own, so no wave waits for another
// until the four partial sums meet in LDS, added in wave order.  The item's scales and
// biases come as they lie, whole lines, one item ahead (4- and 8-byte loads per row and
// macro made more requests than the codes: 2-bit 1370 against 1190 us per layer at 301
// tokens, FP4 984 against 876 at 24).  The grid is what the chip holds at once, and a
// workgroup takes an equal run of the items, its ring running on across them (one
// workgroup per item: a third of the time goes to each one's start).
//
// Measured, two layers of D 4096 x F 2880, 384 experts top-6, router to combine: FP4, 24
// tokens 1225 -> 864 us (362 + 243 -> 266 + 141 us per layer for the two kernels: 5.7 and
// 5.4 TB/s); 3-bit g64, 7 tokens 1569 -> 430 us (536 + 229 -> 117 + 66).  The kernels before
// are the 16-row bf16-MFMA ones of grouped.hip.
//
// A macro is two chunks of 2- or 4-bit codes (a load covers 32 or 64 contiguous bytes per
// row and chunk) and four chunks of 3-bit codes: lane group kg then loads the whole of
// chunk 4q + kg of its row (192 contiguous bytes per row over the four groups) and twelve
// lane-group swaps (v_permlane32_swap, v_permlane16_swap) hand each chunk's four 32-code
// blocks to the four lane groups.  2-bit codes need two swaps: lane groups 0 and 1 hold
// chunk 2q, 2 and 3 chunk 2q + 1, and exchange across the wave's halves, which gives lane
// groups 0 .. 3 the blocks 0, 2, 1, 3 of the chunk; the planes store theirs in that order.
//
// The 16 A rows of an instruction.  A tile has TPT = 8 rows (4 in groups of 32); the
// affine formula s * sum(x q) + b * sum(x) needs one dot product per group, and a chunk
// holds GPC = 128 / G of them.  A row i is tile row i % TPT restricted to one group of the
// chunk (zeros elsewhere) or, with one group per chunk, to one plane: rows 0 .. 7 the hi
// plane, 8 .. 15 the lo plane, so one instruction does the work of two.  Result register
// r of lane (j, kg) is A row 4 kg + r: its group or plane is a function of kg, so each
// lane folds with one scale and one bias per weight row and chunk, acc = fma(s, d,
// fma(b, sum x, acc)), and the lane groups' parts are summed once at the end.
//
// Codes as fp4 operands: 2-bit code q is the E2M1 encoding of q / 2 (column scale 2); 3-
// and 4-bit codes are split, the low two bits so and the rest in a second instruction
// (3-bit: bit 2 as the encoding of 2.0, the same scale; 4-bit: the high pair with scale 8).
// (3-bit codes as six-bit E2M3 fields take one instruction and nine operations per 32
// codes instead of 28, but the instruction sums fp8 x fp6 products, like fp8 x fp8 ones,
// to 2^-19 of the sum of their magnitudes, against 2^-21 for fp8 x fp4.)  The order of a
// block's 32 elements along K is free as long as A has the same, so each width uses the
// order its codes spread to most cheaply (plane_pos): 2-bit codes are two masks per 16;
// 3-bit codes leave three of every four on the nibble they reach by a shift of 0, 1 or 2
// bits, and the fourth ones fill the fourth word (~55 operations in natural order).
#include <algorithm>

#include "decode_common.h"
#include "mfma_tile.h"
#include "mx_tile.h"
#include "prefill_mx.h"

namespace cachalot {
namespace {

using namespace decode;
using namespace pmx;

constexpr int SR_THREADS = 256;
constexpr int SR_WAVES = 4;
constexpr int SR_FRAGS = 4;          // 16-row weight fragments per wave (NM * NF)
constexpr uint32_t E8M0_EIGHT = 130u;

constexpr int sr_tpt(int ak) { return ak_fold(ak) && (ak_gpc(ak) == 4 || ak_bits(ak) == 3) ? 4 : 8; }

template <int AK>
struct Sr {
  static constexpr bool FOLD = ak_fold(AK);
  static constexpr int BITS = AK == AK_FP4 ? 4 : ak_bits(AK);
  static constexpr int G = ak_group(AK);
  static constexpr int GPC = ak_gpc(AK);
  static constexpr int TPT = sr_tpt(AK);                   // rows per tile
  static constexpr int PS = GPC * TPT <= 8 ? 2 : 1;        // planes apart in the A rows (2) or one after the other
  static constexpr int MC = BITS == 3 ? 4 : 2;             // chunks per macro
  static constexpr int RD = BITS == 3 || (FOLD && BITS == 4) ? 2 : 3;   // macros in flight, the one computed included
  static constexpr int CW = BITS * MC;                     // code words per lane, fragment and macro
  static constexpr int EX = FOLD ? MC : 1;                 // 16-byte loads of A scales (and sums) per macro
  static constexpr int ROWB = MC * P3_ROWB;                // one A row's macro
  static constexpr int STAGE = TPT * ROWB;
  static constexpr int ZROW = GPC > 1 ? ROWB : 0;          // a row of zeros
  // LDS: the waves' A rings, the zeros, per wave the macro's A scales [TPT][8 MC] and sums
  // [MC GPC][TPT], and two items' weight scales (and biases) as stored.  A wave's partial
  // sums (4 KiB) go into the ring stage it computed last, or have room of their own.
  static constexpr int RING = SR_WAVES * RD * STAGE;
  static constexpr int ASC = TPT * 8 * MC, SXS = FOLD ? MC * GPC * TPT * 4 : 0;
  static constexpr int WAVE = ASC + SXS;
  static constexpr int PARTW = SR_FRAGS * 4 * 64 * 4;
  static constexpr bool PART_IN_RING = STAGE >= PARTW;
  static constexpr int PART = PART_IN_RING ? 0 : SR_WAVES * PARTW;
  static constexpr int FIXED = RING + ZROW + SR_WAVES * WAVE + PART;
  static_assert(WAVE % 16 == 0, "16-byte regions");
};

typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
// A wave's macros are wave, wave + 4, ...: how many (at least one step, idle past the end).
__host__ __device__ inline int sr_steps(int nmac, int wave) {
  const int n = (nmac - wave + SR_WAVES - 1) / SR_WAVES;
  return n > 1 ? n : 1;
}

// Bytes of an item's weight scales (and biases): 64 rows.
template <int AK>
__host__ __device__ inline int sr_scale_bytes(int K) {
  return Sr<AK>::FOLD ? 2 * 64 * ((K + Sr<AK>::G - 1) / Sr<AK>::G) * 2 : 64 * (K / 32);
}

// Lanes of a wave as a 4 x 4 block transposition: w[b] of lane group a becomes w[a] of
// lane group b, for B consecutive words per block.
template <int B>
__device__ __forceinline__ void transpose_groups(uint32_t* w) {
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int i = 0; i < B; ++i) {
      auto r = __builtin_amdgcn_permlane32_swap(w[b * B + i], w[(b + 2) * B + i], false, false);
      w[b * B + i] = r[0];
      w[(b + 2) * B + i] = r[1];
    }
#pragma unroll
  for (int b = 0; b < 4; b += 2)
#pragma unroll
    for (int i = 0; i < B; ++i) {
      auto r = __builtin_amdgcn_permlane16_swap(w[b * B + i], w[(b + 1) * B + i], false, false);
      w[b * B + i] = r[0];
      w[(b + 1) * B + i] = r[1];
    }
}

// Two chunks of 2-bit codes: lane groups 0, 1 hold the halves of the first, 2, 3 of the
// second; afterwards words 0, 1 are the lane's block of the first and 2, 3 of the second.
__device__ __forceinline__ void exchange_halves(uint32_t* w) {
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    auto r = __builtin_amdgcn_permlane32_swap(w[i], w[i + 2], false, false);
    w[i] = r[0];
    w[i + 2] = r[1];
  }
}

__device__ __forceinline__ i32x8_t op4(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  return i32x8_t{(int)a, (int)b, (int)c, (int)d, 0, 0, 0, 0};
}

__device__ __forceinline__ uint32_t bfi(uint32_t mask, uint32_t a, uint32_t b) { return (a & mask) | (b & ~mask); }

// The fp4 operands of a lane's 32 codes in the order of plane_pos<BITS>: code q as the
// E2M1 encoding of q / 2, 3- and 4-bit codes split into their low two bits (lo) and the
// rest (hi: bit 2 as the encoding 0100 = 2.0; the high pair of 4-bit codes as 2-bit codes).
template <int BITS>
__device__ __forceinline__ void code_operands(const uint32_t* w, i32x8_t& lo, i32x8_t& hi) {
  constexpr uint32_t M = 0x33333333u;
  if constexpr (BITS == 2) {
    lo = op4(w[0] & M, (w[0] >> 2) & M, w[1] & M, (w[1] >> 2) & M);
  } else if constexpr (BITS == 4) {
    lo = op4(w[0] & M, w[1] & M, w[2] & M, w[3] & M);
    hi = op4((w[0] >> 2) & M, (w[1] >> 2) & M, (w[2] >> 2) & M, (w[3] >> 2) & M);
  } else {
    // codes 4t + r, r < 3, move up r bits to nibble 3t + r of the first three words
    const uint32_t x0 = bfi(0x00F00F00u, w[0] << 2, bfi(0xF00F00F0u, w[0] << 1, w[0]));
    const uint32_t x1 = bfi(0x0F00F00Fu, __builtin_amdgcn_alignbit(w[1], w[0], 30),
                            bfi(0x00F00F00u, __builtin_amdgcn_alignbit(w[1], w[0], 31), w[1]));
    const uint32_t x2 = bfi(0xF00F00F0u, __builtin_amdgcn_alignbit(w[2], w[1], 30),
                            bfi(0x0F00F00Fu, __builtin_amdgcn_alignbit(w[2], w[1], 31), w[2]));
    // codes 4t + 3 (bits 12t + 9) fill the fourth
    const uint32_t x3 = bfi(0x0F000000u, w[2] >> 5,
                            bfi(0x00F00F00u, w[2] << 3, bfi(0xF00F00F0u, w[1] << 3, w[0] >> 9)));
    lo = op4(x0 & M, x1 & M, x2 & M, x3 & M);
    constexpr uint32_t H = 0x44444444u;
    hi = op4(x0 & H, x1 & H, x2 & H, x3 & H);
  }
}

// What a wave loads of one macro into registers, in this order (after its A rows).
template <int AK>
struct SrMacro {
  uint4 ex[Sr<AK>::EX];                      // lanes 0 .. 7: A scales of row lane, 8 .. 15: sums of row lane - 8
  uint32_t codes[SR_FRAGS][Sr<AK>::CW];
};

// One workgroup takes a contiguous run of the items (tile, slice of 64 weight rows), an
// equal share of them, so the grid is what the chip holds at once and all of it ends
// together; the macros of its items are one sequence per wave, RD - 1 of them in flight
// across the items' ends.  g.recs / g.tiles_n: the tiles.
template <int AK, int NM, int NF>
__global__ void __launch_bounds__(SR_THREADS, 2) sr_kernel(MxArgs g, int slices) {
  using S = Sr<AK>;
  constexpr int TPT = S::TPT, MC = S::MC, GPC = S::GPC, G = S::G, BITS = S::BITS, PS = S::PS, RD = S::RD;
  static_assert(NM * NF == SR_FRAGS, "four fragments per wave");
  extern __shared__ __align__(16) uint8_t lds[];   // S::FIXED + 2 sr_scale_bytes
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, kg = lane >> 4;
  // this workgroup's items; neighbouring runs on one XCD
  const int xcds = 8, per = gridDim.x / xcds;
  const int run = (int)(blockIdx.x % xcds) * per + (int)blockIdx.x / xcds;
  const int64_t total = (int64_t)g.tiles_n[0] * slices;
  const int it0 = (int)(total * run / gridDim.x), it1 = (int)(total * (run + 1) / gridDim.x);
  if (it0 >= it1) return;

  uint8_t* aring = lds + wave * RD * S::STAGE;
  uint8_t* zrow = lds + S::RING;
  uint8_t* myas = zrow + S::ZROW + wave * S::WAVE;
  float* mysx = reinterpret_cast<float*>(myas + S::ASC);
  uint8_t* part0 = zrow + S::ZROW + SR_WAVES * S::WAVE;
  uint8_t* scales = part0 + S::PART;
  const int scb = sr_scale_bytes<AK>(g.K);

  const int nch = g.kch, nmac = (nch + MC - 1) / MC;
  const int mine = sr_steps(nmac, wave);
  const int groups = S::FOLD ? (g.K + G - 1) / G : g.K / 32;   // groups, or E8M0 blocks, of a weight row
  const int row_bytes = S::FOLD ? groups * G * BITS / 8 : g.K / 2;
  const int srow_bytes = S::FOLD ? groups * 2 : groups;
  constexpr int WN = 16 * NF;                          // weight rows per item and matrix
  const int tq[2] = {NM == 2 ? 0 : 3, 6};              // w1, w3 (gate/up) or w2 (down)

  // ---- the issuing side: its item, step and addresses
  constexpr int LPR = 16 * MC, RPI = 64 / LPR, NI = TPT / RPI;   // A: one instruction covers RPI rows' macros
  const int achunk = (lane >> 4) % MC;
  int i_item = it0, i_j = 0, i_tile = -1, i_rows = 1;
  const uint8_t* base = g.pool;
  const uint8_t* asrc[NI];
  const uint8_t* exsrc = nullptr;
  const bool ex_sum = S::FOLD && (lane & 8) != 0;
  const int exstep = ex_sum ? 16 * MC : 8 * MC;
  int woff[SR_FRAGS];                                  // from the slot record (< 2^31: one expert)
  auto enter_item = [&]() {
    const int tile = i_item / slices, nw0 = (i_item - tile * slices) * WN;
    if (tile != i_tile) {
      i_tile = tile;
      const int4 rec = g.recs[tile];   // expert, first row, end row, slot
      const int row0 = __builtin_amdgcn_readfirstlane(rec.y);
      i_rows = __builtin_amdgcn_readfirstlane(rec.z) - row0;
      const int slot = max(__builtin_amdgcn_readfirstlane(rec.w), 0);   // (a missing expert's results are dropped)
      base = g.pool + (int64_t)slot * g.L.record_bytes;
      // row r's 16-byte column c of a chunk sits at column c ^ (r % 16)
#pragma unroll
      for (int q = 0; q < NI; ++q) {
        const int r = q * RPI + lane / LPR;
        const int rr = row0 + min(r, i_rows - 1);
        const int src = g.a_gather ? g.a_gather[rr] : rr;
        asrc[q] = g.ap + (size_t)src * nch * P3_ROWB + (((lane & 15) ^ (r & 15)) << 4);
      }
      const int rr = row0 + min(lane & 7, i_rows - 1);
      const int src = g.a_gather ? g.a_gather[rr] : rr;
      exsrc = ex_sum ? reinterpret_cast<const uint8_t*>(g.asum + (size_t)src * nch * 4) : g.as + (size_t)src * g.sb;
    }
#pragma unroll
    for (int p = 0; p < SR_FRAGS; ++p)
      woff[p] = (int)g.L.off[tq[p / NF]] + min(nw0 + 16 * (p % NF) + i, g.N - 1) * row_bytes;
    // the item's scales as they lie, whole lines, a quarter per wave: [scales | biases][64
    // rows], or 64 rows of E8M0; wave w takes 32 rows of one kind (FP4: fragment w's 16)
    constexpr int QROWS = S::FOLD ? 32 : 16;
    const int sub = S::FOLD ? wave >> 1 : wave, kind = S::FOLD ? wave & 1 : 0;   // sub: 32 (16) of the 64 rows
    const int sm = NM == 2 ? sub * QROWS / 32 : 0, sr = sub * QROWS - sm * 32;
    const int first = min(nw0, g.N - (NM == 2 ? 32 : 64)) + sr;                  // (slices past F: rows not used)
    tile::copy_to_lds_untracked(base + g.L.off[tq[sm] + 1 + kind] + (int64_t)first * srow_bytes,
                                scales + (i_item & 1) * scb + (kind * 64 + sub * QROWS) * srow_bytes,
                                QROWS * srow_bytes, 0, 1, lane);
  };
  SrMacro<AK> ring[RD];
  auto issue = [&](uint8_t* stage, SrMacro<AK>& out) {
    if (i_j == mine) {   // the next item (past the last one: its steps again, re-reads nothing uses)
      i_j = 0;
      if (i_item + 1 < it1) {
        ++i_item;
        enter_item();
      }
    }
    const int m = min(wave + SR_WAVES * i_j, nmac - 1);
#pragma unroll
    for (int q = 0; q < NI; ++q)
      if (q * RPI < i_rows)   // uniform: rows that do not exist are not read (their results are dropped)
        tile::lds_load16_untracked(asrc[q] + (size_t)min(m * MC + achunk, nch - 1) * P3_ROWB, stage + q * 1024);
#pragma unroll
    for (int q = 0; q < S::EX; ++q)
      out.ex[q] = *reinterpret_cast<const uint4*>(exsrc + m * exstep + 16 * (ex_sum ? q : min(q, MC / 2 - 1)));
#pragma unroll
    for (int p = 0; p < SR_FRAGS; ++p) {
      if constexpr (BITS == 4) {
#pragma unroll
        for (int u = 0; u < MC; ++u) {
          const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(
              base + woff[p] + min((m * MC + u) * 64 + kg * 16, row_bytes - 16));
#pragma unroll
          for (int j = 0; j < 4; ++j) out.codes[p][4 * u + j] = v[j];
        }
      } else if constexpr (BITS == 2) {
        // half kg & 1 of chunk 2 m + (kg >> 1) (a chunk past K: the last one, not used)
        const int off = min(m * MC + (kg >> 1), nch - 1) * 32 + (kg & 1) * 16;
        const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(base + woff[p] + off);
#pragma unroll
        for (int j = 0; j < 4; ++j) out.codes[p][j] = v[j];
      } else {
        // chunk 4 m + kg of the row (a chunk past K: the last one, not used)
        const int off = min(m * MC + kg, nch - 1) * 48;
#pragma unroll
        for (int q = 0; q < 3; ++q) {
          const u32x4_a4 v = *reinterpret_cast<const u32x4_a4*>(base + woff[p] + off + 16 * q);
#pragma unroll
          for (int j = 0; j < 4; ++j) out.codes[p][4 * q + j] = v[j];
        }
      }
    }
    ++i_j;
  };

  // ---- the computing side: its item and the tile's rows
  int c_item = it0, c_j = 0, c_tile = -1, c_rows = 0, c_slot = -1, c_prow = 0;
  float c_w = 0.0f;                                    // gate/up: the lane's row weight
  uint16_t* c_y = nullptr;                             // down: the lane's output row
  // The lane's results are tile row tr x weight rows nw0 + 16 f + i (wave r finishes
  // register r); the lane groups past the tile's rows hold copies.
  const int tr = (4 * kg) % TPT + wave;
  auto enter_tile = [&](int tile) {
    c_tile = tile;
    const int4 rec = g.recs[tile];
    const int row0 = __builtin_amdgcn_readfirstlane(rec.y);
    c_rows = __builtin_amdgcn_readfirstlane(rec.z) - row0;
    c_slot = __builtin_amdgcn_readfirstlane(rec.w);
    c_prow = row0 + min(tr, c_rows - 1);
    if constexpr (NM == 2) c_w = g.row_w[c_prow];
    else c_y = g.y + ((size_t)g.row_token[c_prow] * g.k + g.row_slot[c_prow]) * g.N;
  };
  f32x4_t acc[SR_FRAGS];
#pragma unroll
  for (int p = 0; p < SR_FRAGS; ++p) acc[p] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

  // the lane's A row: tile row i % TPT for the half of the chunk that lies in the row's
  // group, the row of zeros for the other; with PS == 2 the upper rows carry the lo plane
  const int at = i % TPT, ag = i / TPT % GPC, ap = PS == 2 ? i / (TPT * GPC) % 2 : 0;
  const bool own0 = block_at<BITS>(kg >> 1) * 32 / G == ag, own1 = block_at<BITS>(2 + (kg >> 1)) * 32 / G == ag;
  const int col0 = ((8 * ap + kg) ^ at) << 4, col1 = ((8 * ap + 4 + kg) ^ at) << 4;
  const int col2 = ((8 + kg) ^ at) << 4, col3 = ((12 + kg) ^ at) << 4;
  const uint8_t* sap = myas + at * (8 * MC) + ap;
  const int dg = (4 * kg) / TPT % GPC;                         // the group of the lane's results
  const bool dlo = PS == 2 && (4 * kg) / (TPT * GPC) % 2 == 1; // they are the lo plane's (no bias term)
  const float* sxp = mysx + dg * TPT + (4 * kg) % TPT;

  // the partial sums of the waves meet; wave r finishes result register r
  auto finish_item = [&]() {
    // where wave w's partial sums go: the stage of its last step
    auto part = [&](int w) {
      if constexpr (!S::PART_IN_RING) return reinterpret_cast<float*>(part0 + w * S::PARTW);
      const int mw = sr_steps(nmac, w);
      return reinterpret_cast<float*>(lds + (w * RD + ((c_item - it0 + 1) * mw - 1) % RD) * S::STAGE);
    };
    float* own = part(wave);
#pragma unroll
    for (int p = 0; p < SR_FRAGS; ++p)
#pragma unroll
      for (int r = 0; r < 4; ++r) own[(p * 4 + r) * 64 + lane] = acc[p][r];
#pragma unroll
    for (int p = 0; p < SR_FRAGS; ++p) acc[p] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    const int tile = c_item / slices, slice = c_item - tile * slices, nw0 = slice * WN;
    if (tile != c_tile) enter_tile(tile);
    lds_sync();
    float sum[SR_FRAGS];
    const float* pw[SR_WAVES];
#pragma unroll
    for (int w = 0; w < SR_WAVES; ++w) pw[w] = part(w) + wave * 64 + lane;
#pragma unroll
    for (int p = 0; p < SR_FRAGS; ++p) {
      float t = 0.0f;
#pragma unroll
      for (int w = 0; w < SR_WAVES; ++w) t = t + pw[w][p * 4 * 64];
      // parts apart: rows [plane][group][row of the tile], four per lane group
      if constexpr (TPT == 4 && GPC * PS >= 2) t = t + xor_f<16>(t);
      if constexpr (GPC * PS * TPT == 16) t = t + xor_f<32>(t);
      sum[p] = c_slot >= 0 ? t : 0.0f;
    }
    ++c_item;   // (the barrier at the next item's first step frees the stages)
    if (tr >= c_rows || kg >= TPT / 4) return;   // the same in the 16 lanes of a row group
    if constexpr (NM == 2) {
      float hv[NF];
      float top = 0.0f;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        float gv = round_bf16(sum[f]);
        float uv = round_bf16(sum[NF + f]);
        if (g.limit > 0.0f) {
          uv = fminf(fmaxf(uv, -g.limit), g.limit);
          gv = fminf(gv, g.limit);
        }
        hv[f] = nw0 + 16 * f + i < g.N ? round_bf16((silu_f32(gv) * uv) * c_w) : 0.0f;
        top = fmaxf(top, fabsf(hv[f]));
      }
      top = mx::row16_max(top);
      const int E = plane_exp(top);
      const float inv = __uint_as_float((uint32_t)(127 - E) << 23);
      const int blk = (nw0 & ~127) / 32 + block_at<S::FOLD ? BITS : 0>((nw0 >> 5) & 3);   // the block's place
      uint8_t* dst = g.hp + ((size_t)c_prow * g.hkch + (blk >> 2)) * P3_ROWB + (blk & 3) * 32;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const float s = hv[f] * inv;
        const uint32_t hi = mx::f32_to_e4m3(s);
        const uint32_t lo = mx::f32_to_e4m3((s - mx::e4m3_to_f32(hi)) * 16.0f);
        uint8_t* p = dst + plane_pos<S::FOLD ? BITS : 0>(16 * f + i);
        p[0] = (uint8_t)hi;
        p[128] = (uint8_t)lo;
      }
      if (i == 0) {
        const uint32_t sc = (uint32_t)(E + 127) | ((uint32_t)(E + 123) << 8);
        *reinterpret_cast<uint16_t*>(g.hs + (size_t)c_prow * g.hsb + blk * 2) = (uint16_t)sc;
      }
      if constexpr (S::FOLD) {   // the sum of the 32 h values (f, then the 16 lanes)
        float hsv = 0.0f;
#pragma unroll
        for (int f = 0; f < NF; ++f) hsv = hsv + hv[f];
        hsv = row16_sum(hsv);
        if (i == 0) g.hsum[(size_t)c_prow * g.hkch * 4 + nw0 / 32] = hsv;
      }
    } else {
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        const int n = nw0 + 16 * f + i;
        if (n < g.N) c_y[n] = f32_to_bf16(sum[f]);
      }
    }
  };

  if constexpr (GPC > 1) {
    for (int z = tid; z < S::ROWB / 16; z += SR_THREADS) *reinterpret_cast<uint4*>(zrow + z * 16) = uint4{0u, 0u, 0u, 0u};
  }
  enter_item();
#pragma unroll
  for (int v = 0; v < RD - 1; ++v) issue(aring + v * S::STAGE, ring[v]);

  for (;;) {
#pragma unroll
    for (int v = 0; v < RD; ++v) {
      const int m = wave + SR_WAVES * c_j;
      // the wave's loads of macro m have landed: its last code load is consumed here, and
      // everything issued before it (the A rows among them) completes first
      asm volatile("" ::"v"(ring[v].codes[SR_FRAGS - 1][S::CW - 1]) : "memory");
      __builtin_amdgcn_s_waitcnt(0xC07F);   // lgkmcnt(0): the reads of the stage refilled below are done
      // an item's first step: every wave's quarter of its scales has landed too, and every
      // wave is past the partial sums of the item before
      if (c_j == 0) lds_sync();
      if (lane < TPT) {
#pragma unroll
        for (int q = 0; q < MC / 2; ++q) *reinterpret_cast<uint4*>(myas + lane * (8 * MC) + 16 * q) = ring[v].ex[q];
      } else if (S::FOLD && lane >= 8 && lane < 8 + TPT) {
#pragma unroll
        for (int q = 0; q < S::EX; ++q) {   // four sums of 32 per chunk -> one per group; none past K
          const bool in = m * MC + q < nch;
          const float a = in ? __uint_as_float(ring[v].ex[q].x) : 0.0f, b = in ? __uint_as_float(ring[v].ex[q].y) : 0.0f;
          const float c = in ? __uint_as_float(ring[v].ex[q].z) : 0.0f, d = in ? __uint_as_float(ring[v].ex[q].w) : 0.0f;
          float* o = mysx + q * GPC * TPT + (lane - 8);
          if constexpr (GPC == 1) {
            o[0] = (a + b) + (c + d);
          } else if constexpr (GPC == 2) {
            o[0] = a + b;
            o[TPT] = c + d;
          } else {
            o[0] = a;
            o[TPT] = b;
            o[2 * TPT] = c;
            o[3 * TPT] = d;
          }
        }
      }
      issue(aring + (v + RD - 1) % RD * S::STAGE, ring[(v + RD - 1) % RD]);
      if constexpr (BITS == 3) {
#pragma unroll
        for (int p = 0; p < SR_FRAGS; ++p) transpose_groups<BITS>(ring[v].codes[p]);
      } else if constexpr (BITS == 2) {
#pragma unroll
        for (int p = 0; p < SR_FRAGS; ++p) exchange_halves(ring[v].codes[p]);
      }
      const uint8_t* sc = scales + (c_item & 1) * scb;
      const uint8_t* arow = aring + v * S::STAGE + at * S::ROWB;
      const uint8_t* a0 = GPC == 1 || own0 ? arow : zrow;
      const uint8_t* a1 = GPC == 1 || own1 ? arow : zrow;
#pragma unroll
      for (int u = 0; u < MC; ++u) {
        const int c = m * MC + u;
        if (c >= nch) break;
        __builtin_amdgcn_sched_barrier(0);   // (chunks interleaved would spill)
        const uint4 h0 = mx::lds16(a0 + u * P3_ROWB + col0);
        const uint4 h1 = mx::lds16(a1 + u * P3_ROWB + col1);
        const i32x8_t ahi = {(int)h0.x, (int)h0.y, (int)h0.z, (int)h0.w, (int)h1.x, (int)h1.y, (int)h1.z, (int)h1.w};
        i32x8_t alo;
        uint32_t sa;
        if constexpr (PS == 1) {
          const uint4 l0 = mx::lds16(a0 + u * P3_ROWB + col2);
          const uint4 l1 = mx::lds16(a1 + u * P3_ROWB + col3);
          alo = i32x8_t{(int)l0.x, (int)l0.y, (int)l0.z, (int)l0.w, (int)l1.x, (int)l1.y, (int)l1.z, (int)l1.w};
          sa = (uint32_t)sap[(4 * u + kg) * 2] | ((uint32_t)sap[(4 * u + kg) * 2 + 1] << 8);
        } else {
          sa = sap[(4 * u + kg) * 2];
        }
        if constexpr (!S::FOLD) {
          const int blk = min(4 * c + kg, groups - 1);   // blocks past K meet zero A
          uint32_t bs[SR_FRAGS];
          i32x8_t b[SR_FRAGS];
#pragma unroll
          for (int p = 0; p < SR_FRAGS; ++p) {
            bs[p] = sc[(16 * p + i) * groups + blk];
            const uint32_t* w = ring[v].codes[p] + 4 * u;
            b[p] = op4(w[0], w[1], w[2], w[3]);
          }
#pragma unroll
          for (int p = 0; p < SR_FRAGS; ++p) acc[p] = mx::mfma_fp8_fp4<0, true>(ahi, b[p], acc[p], sa, bs[p]);
          if constexpr (PS == 1) {
#pragma unroll
            for (int p = 0; p < SR_FRAGS; ++p) acc[p] = mx::mfma_fp8_fp4<1, true>(alo, b[p], acc[p], sa, bs[p]);
          }
        } else {
          const uint16_t* s16 = reinterpret_cast<const uint16_t*>(sc) + i * groups;
          const int go = min(GPC * c + dg, groups - 1);   // groups past K meet zero A
          float sw[SR_FRAGS];
#pragma unroll
          for (int p = 0; p < SR_FRAGS; ++p) sw[p] = scale_bits_to_f32(s16[16 * p * groups + go], g.L.f16);
          constexpr uint32_t LS = mx::E8M0_TWO, HS = BITS == 4 ? E8M0_EIGHT : mx::E8M0_TWO;
          f32x4_t d[SR_FRAGS];
          // (two fragments at a time: all four's operands spill the 3-bit kernels)
#pragma unroll
          for (int pp = 0; pp < SR_FRAGS; pp += 2) {
            i32x8_t lo[2], hi[2];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
              code_operands<BITS>(ring[v].codes[pp + p] + BITS * u, lo[p], hi[p]);
              d[pp + p] = mx::mfma_fp8_fp4<0, true>(ahi, lo[p], f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, sa, LS);
            }
            if constexpr (PS == 1) {
#pragma unroll
              for (int p = 0; p < 2; ++p) d[pp + p] = mx::mfma_fp8_fp4<1, true>(alo, lo[p], d[pp + p], sa, LS);
            }
            if constexpr (BITS > 2) {
#pragma unroll
              for (int p = 0; p < 2; ++p) d[pp + p] = mx::mfma_fp8_fp4<0, true>(ahi, hi[p], d[pp + p], sa, HS);
              if constexpr (PS == 1) {
#pragma unroll
                for (int p = 0; p < 2; ++p) d[pp + p] = mx::mfma_fp8_fp4<1, true>(alo, hi[p], d[pp + p], sa, HS);
              }
            }
            __builtin_amdgcn_sched_barrier(0);
          }
          // the bias term: with the planes apart, the hi lanes take an even chunk's and the
          // lo lanes the next one's
          const bool bias_here = PS == 1 || u % 2 == 0;
          if (bias_here) {
            const int ub = PS == 1 ? u : u + (dlo ? 1 : 0);
            const int gb = min(GPC * (m * MC + ub) + dg, groups - 1);
            const float4 sx = *reinterpret_cast<const float4*>(sxp + ub * GPC * TPT);
            const float sxv[4] = {sx.x, sx.y, sx.z, sx.w};
#pragma unroll
            for (int p = 0; p < SR_FRAGS; ++p) {
              const float b = scale_bits_to_f32(s16[(64 + 16 * p) * groups + gb], g.L.f16);
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[p][r] = fmaf(sw[p], d[p][r], fmaf(b, sxv[r], acc[p][r]));
            }
          } else {
#pragma unroll
            for (int p = 0; p < SR_FRAGS; ++p)
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[p][r] = fmaf(sw[p], d[p][r], acc[p][r]);
          }
        }
      }
      if (++c_j == mine) {
        c_j = 0;
        finish_item();
        if (c_item == it1) {
          // the re-reads issued past the end (direct-to-LDS among them) land before the
          // workgroup's LDS is released
          tile::wait_vmem();
          return;
        }
      }
    }
  }
}

template <int AK>
struct SrLaunch {
  static size_t lds(int K) { return (size_t)Sr<AK>::FIXED + 2 * sr_scale_bytes<AK>(K); }
  // The issuing side may be one item ahead and no more (two items' scales in LDS): RD - 1
  // steps per item for every wave.
  static bool fits(int K) {
    const int nmac = ((K + 127) / 128 + Sr<AK>::MC - 1) / Sr<AK>::MC;
    return sr_steps(nmac, SR_WAVES - 1) >= Sr<AK>::RD - 1 && lds(K) <= 160 * 1024;
  }
  template <int NM, int NF>
  static int go(const MxArgs& a, int slices, hipStream_t s) {
    const size_t bytes = lds(a.K);
    auto k = sr_kernel<AK, NM, NF>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)bytes) != hipSuccess)
      return fail(CACHALOT_EHIP, "grouped experts (few rows): cannot grant %zu bytes of LDS", bytes);
    const int per_cu = bytes <= 80 * 1024 ? 2 : 1;   // what each of the 256 CUs holds at once
    hipLaunchKernelGGL(k, dim3(256 * per_cu), dim3(SR_THREADS), bytes, s, a, slices);
    return check_launch("sr_kernel");
  }
  static int run(const MxArgs& gu, const MxArgs& dn, hipStream_t s) {
    if (int rc = go<2, 2>(gu, gu.hkch * 4, s)) return rc;   // 32 columns of h per item
    return go<1, 4>(dn, (dn.N + 63) / 64, s);
  }
};

}  // namespace

// Rows per tile of a bank kind (the tile list's MT).
int small_rows_mt(int ak) { return sr_tpt(ak); }

template <int AK>
static bool sr_fits(int D, int F) { return SrLaunch<AK>::fits(D) && SrLaunch<AK>::fits(F); }

// A row's last chunk is read whole (2- and 3-bit codes): past a tensor's last row, where
// the row is shorter, up to 47 bytes, which must still lie inside the slot record.
bool small_rows_supported(int ak, int D, int F, const decode::Layout& L) {
  if (!(D % 128 == 0 && D >= 128 && D <= 8192 && F % 32 == 0 && F >= 32 && F <= 8192)) return false;
  const bool fold = ak_fold(ak);
  const int bits = fold ? ak_bits(ak) : 4, group = ak_group(ak);
  const int mats[3][3] = {{0, F, D}, {6, F, D}, {3, D, F}};   // w1, w3, w2: tensor, rows, K
  for (auto& m : mats) {
    const int64_t n = m[1], k = m[2], nch = (k + 127) / 128;
    const int64_t rb = fold ? (k + group - 1) / group * group * bits / 8 : k / 2;
    const int64_t code_over = bits == 4 ? 0 : nch * 16 * bits - rb;
    if (rb < 16 || L.off[m[0]] + n * rb + code_over > L.record_bytes) return false;
  }
#define CACHALOT_SR(K) \
  if (ak == (K)) return sr_fits<(K)>(D, F);
  CACHALOT_SR(AK_FP4) CACHALOT_SR(AK_Q2)
  CACHALOT_SR(ak_aff(2, 32)) CACHALOT_SR(ak_aff(2, 64))
  CACHALOT_SR(ak_aff(3, 32)) CACHALOT_SR(ak_aff(3, 64)) CACHALOT_SR(ak_aff(3, 128))
  CACHALOT_SR(ak_aff(4, 32)) CACHALOT_SR(ak_aff(4, 64)) CACHALOT_SR(ak_aff(4, 128))
#undef CACHALOT_SR
  return false;
}

int launch_small_rows(int ak, const pmx::MxArgs& gu, const pmx::MxArgs& dn, hipStream_t s) {
#define CACHALOT_SR(K) \
  if (ak == (K)) return SrLaunch<(K)>::run(gu, dn, s);
  CACHALOT_SR(AK_FP4) CACHALOT_SR(AK_Q2)
  CACHALOT_SR(ak_aff(2, 32)) CACHALOT_SR(ak_aff(2, 64))
  CACHALOT_SR(ak_aff(3, 32)) CACHALOT_SR(ak_aff(3, 64)) CACHALOT_SR(ak_aff(3, 128))
  CACHALOT_SR(ak_aff(4, 32)) CACHALOT_SR(ak_aff(4, 64)) CACHALOT_SR(ak_aff(4, 128))
#undef CACHALOT_SR
  return fail(CACHALOT_EINVAL, "grouped experts (few rows): weight kind %d", ak);
}

}  // namespace cachalot
