// Expert-major grouped experts with few rows per expert (batched decode, drafted
// tokens, short prompts) as a weight stream on the bf16 matrix cores: every bank kind.
//
// Reference: affine_expert_forward_batched (src/cachalot/model/expert_affine.py:84-99),
// routed_expert_forward_sgmm / _batched (fp4_sgmm_metal.py:318-333,
// moe_prefill_batched.py:31-61), called per expert from moe_prefill_grouped.py:420-467.
// Rounding points: g = bf16(x W1), u = bf16(x W3), h = bf16(silu(min(g, L)) * clip(u,
// +-L) * w), y = bf16(h W2); the products accumulate in fp32.
//
// What bounds it: the weight bytes of the touched experts, each read once per tile of TPT
// rows, so the kernel is a weight stream.  An item is 64 weight rows (gate/up: 32 of W1 and
// the same 32 of W3; down: 64 of W2) of one tile for the whole K, and the four waves of a
// workgroup take its macros of K (MC chunks of 128) in turn, so that at any time it reads
// long contiguous runs of its rows.  (Waves owning 64 rows each, 256 per workgroup, read the
// same bytes at 4.0 against 5.3 TB/s for FP4 at 24 tokens.)  A wave keeps its next macros'
// codes in flight in registers, 16 bytes per lane and load; its share of the A rows (only
// the rows that exist) goes through an LDS ring of its own, so no wave waits for another
// until the four partial sums meet in LDS, added in wave order.  The item's scales and
// biases come as they lie, whole lines, one item ahead (4- and 8-byte loads per row and
// macro made more requests than the codes).  A workgroup takes an equal run of the items,
// its ring running on across them (one workgroup per item: a third of the time goes to each
// one's start).  The runs are as many as the chip holds at once, or up to SR_ROUNDS times
// as many where each keeps SR_RUN items: with one round, a CU on which a kernel of another
// stream (the shared expert) still held LDS when this one came took one workgroup for the
// whole kernel, and the one left out ran after all others (2-bit, 301 tokens beside the
// shared expert, gate/up 1092 against 826 us alone).
//
// Operands.  x and h go in as the bf16 values they are and the codes as exact bf16, so
// products are exact, the sums are the instruction's fp32 sums, and an infinity or a NaN
// does what it does on the 16-row tiles of grouped.hip.  (Both as fp8 planes with fp4 codes
// on the block-scaled instruction: an element 2^13 below its block's largest loses bits,
// sums round at 2^-21 of their magnitudes, which turned one in twelve bf16 outputs against
// one in a thousand, and E4M3 has no infinity.)
//
// Measured, kernel times per layer, gate/up + down, us, 384 experts top-6: 16-row tiles ->
// planes -> here.  D 4096 x F 2880, FP4, 24 tokens: 362 + 243 -> 256 + 135 -> 258 + 144 (5.7 and
// 5.1 TB/s); 3-bit g64, 7 tokens: 536 + 229 -> 117 + 64 -> 116 + 64.  5120 x 2304, 2-bit g128, 301
// tokens beside the shared expert: 64-row tiles 1047 + 571 -> 748 to 938 + 370 -> 733 + 423 (VALU
// 68 and 59 per cent busy, matrix cores 20 and 17: issue bound, where FP4 at 31 and 15 waits for
// memory).
//
// A macro is two chunks of 2- or 4-bit codes (a load covers 32 or 64 contiguous bytes per
// row and chunk) and four chunks of 3-bit codes: lane group kg then loads the whole of
// chunk 4q + kg of its row (192 contiguous bytes per row over the four groups) and twelve
// lane-group swaps (v_permlane32_swap, v_permlane16_swap) hand each chunk's four 32-code
// blocks to the four lane groups.  2-bit codes need two swaps: lane groups 0 and 1 hold
// chunk 2q, 2 and 3 chunk 2q + 1, and exchange across the wave's halves, which gives lane
// groups 0 .. 3 the blocks 0, 2, 1, 3 of the chunk (sr_block).
//
// The 16 A rows of an instruction.  Step q of a chunk takes codes 8 q .. + 7 of each lane
// group's block, all four blocks at once.  A tile has TPT = 8 rows (4 in groups of 32 and for
// 3-bit codes, whose four-chunk macros would leave room for one workgroup per CU); the affine
// formula s * sum(x q) + b * sum(x) needs one dot product per group, and a chunk holds
// GPC = 128 / G of them.  A row i is tile row i % TPT restricted to group (i / TPT) % GPC of
// the chunk (zeros elsewhere).  Result register r of lane (j, kg) is A row 4 kg + r: its
// group is a function of kg, so each lane folds with one scale and one bias per weight row
// and chunk, acc = fma(s, d, fma(b, sum x, acc)), and the lane groups' parts are summed once
// at the end.  The order of a block's 32 elements along K is free as long as A has the same,
// so each width uses the order its codes spread to most cheaply (sr_pos, code_values).
#include <algorithm>
#include <type_traits>

#include "decode_common.h"
#include "mfma_tile.h"

namespace cachalot {
namespace {

using namespace decode;
using tile::bf16x8_t;
using tile::f32x4_t;

constexpr int SR_THREADS = 256;
constexpr int SR_WAVES = 4;
constexpr int SR_FRAGS = 4;          // 16-row weight fragments per wave (NM * NF)
constexpr int SR_ROWB = 256;         // one A row's chunk: 128 bf16

// Weight kinds: FP4, or (BITS << 8) | G for affine codes in groups of G.
constexpr int SR_FP4 = 0;
constexpr int sr_kind(int bits, int group) { return bits == 0 ? SR_FP4 : (bits << 8) | group; }
constexpr int sr_bits(int sk) { return sk == SR_FP4 ? 4 : sk >> 8; }
constexpr int sr_group(int sk) { return sk == SR_FP4 ? 128 : sk & 255; }
constexpr int sr_tpt(int sk) { return sk != SR_FP4 && (sr_group(sk) == 32 || sr_bits(sk) == 3) ? 4 : 8; }

// The order of a 32-element block of A (x and h of affine banks): the one its BITS-bit
// codes leave the spread in (code_values).  2-bit: the even elements of each 16, then the
// odd ones.  3-bit: the even elements, then the odd ones.  4-bit: elements 3j at place 2j,
// 3j + 1 at 2j + 1, and of the elements 3j + 2 the first five at 23 + 2j, the others at
// 22 + 2 (j - 5).  BITS 0 (FP4): natural.
template <int BITS>
__host__ __device__ inline int sr_pos(int n) {
  if (BITS == 2) return (n & 16) + ((n & 1) ? 8 + ((n & 15) >> 1) : (n & 15) >> 1);
  if (BITS == 3) return (n & 1) * 16 + (n >> 1);
  if (BITS == 4) {
    const int j = n / 3, r = n - 3 * j;
    return r < 2 ? 2 * j + r : j < 5 ? 23 + 2 * j : 12 + 2 * j;
  }
  return n;
}

struct SrArgs {
  const uint8_t* a;           // A rows, bf16 [source rows][kch * 128]
  int kch;                    // 128-element chunks along K
  const int32_t* a_gather;    // source row of a tile row (row_token) or null (the row itself)
  const float* asum;          // affine: sums of 32 A elements [source rows][kch * 4]
  const uint8_t* pool;
  Layout L;
  const int4* recs;           // the tiles: expert, first row, end row, slot
  const int32_t* recs_n;
  const int32_t* row_token;
  const int32_t* row_slot;
  const float* row_w;
  int K;                      // real K (D or F)
  int N;                      // weight rows per matrix (F or D)
  int k;
  float limit;
  uint16_t* h;                // gate/up: [rows][hkch * 128], columns past F zero
  int hkch;
  float* hsum;                // gate/up, affine: sums of 32 of h [rows][hkch * 4]
  uint16_t* y;                // down: [T, k, N]
};

template <int AK>
struct Sr {
  static constexpr bool FOLD = AK != SR_FP4;
  static constexpr int BITS = sr_bits(AK);
  static constexpr int G = sr_group(AK);
  static constexpr int GPC = FOLD ? 128 / G : 1;           // groups per chunk
  static constexpr int TPT = sr_tpt(AK);                   // rows per tile
  static constexpr int MC = BITS == 3 ? 4 : 2;             // chunks per macro
  static constexpr int RD = BITS == 3 || (FOLD && BITS == 4) ? 2 : 3;   // macros in flight, the one computed included
  static constexpr int CW = BITS * MC;                     // code words per lane, fragment and macro
  static constexpr int EX = FOLD ? MC : 1;                 // 16-byte loads of A sums per macro
  static constexpr int ROWB = MC * SR_ROWB;                // one A row's macro
  static constexpr int STAGE = TPT * ROWB;
  static constexpr int ZROW = GPC > 1 ? ROWB : 0;          // a row of zeros
  // LDS: the waves' A rings, the zeros, per wave the macro's sums [MC GPC][TPT], and two
  // items' weight scales (and biases) as stored.  A wave's partial sums (4 KiB) go into
  // the ring stage it computed last, or have room of their own.
  static constexpr int RING = SR_WAVES * RD * STAGE;
  static constexpr int WAVE = FOLD ? MC * GPC * TPT * 4 : 0;
  static constexpr int PARTW = SR_FRAGS * 4 * 64 * 4;
  static constexpr bool PART_IN_RING = STAGE >= PARTW;
  static constexpr int PART = PART_IN_RING ? 0 : SR_WAVES * PARTW;
  static constexpr int FIXED = RING + ZROW + SR_WAVES * WAVE + PART;
  static_assert(WAVE % 16 == 0, "16-byte regions");
};

constexpr int SR_ROUNDS = 4, SR_RUN = 16;
// Rounds of `slots` workgroups that `items` items are dealt to.
__host__ __device__ inline int sr_rounds(int64_t items, int slots) {
  const int64_t n = items / ((int64_t)slots * SR_RUN);
  return n < 1 ? 1 : n < SR_ROUNDS ? (int)n : SR_ROUNDS;
}

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

// The 32-element block of a chunk that lane group kg holds the codes of.
template <int BITS>
__device__ __forceinline__ int sr_block(int kg) {
  return BITS == 2 && (kg == 1 || kg == 2) ? 3 - kg : kg;
}

// A lane's 32 codes as exact bf16 integers in the order of sr_pos<BITS>, eight per MFMA
// step.  2-bit: spread to nibbles, E2M1 q / 2, the pair converter with scale 2 (full
// rate).  3- and 4-bit: spread to six-bit fields, E2M3 q / 8, the 32-value converter with
// scale 8 (the time of 18 instructions).
template <int BITS>
__device__ __forceinline__ void code_values(const uint32_t* w, bf16x8_t (&b)[4]) {
  if constexpr (BITS == 2) {
    constexpr uint32_t M = 0x33333333u;
#pragma unroll
    for (int s = 0; s < 4; ++s) b[s] = tile::fp4_codes_to_b((s & 1 ? w[s >> 1] >> 2 : w[s >> 1]) & M, 2.0f);
  } else {
    typedef uint32_t u32x6_t __attribute__((ext_vector_type(6)));
    u32x6_t f;
    if constexpr (BITS == 3) {
      // every second code already lies alone in a six-bit field
      constexpr uint32_t M0 = 0xC71C71C7u, M1 = 0x71C71C71u, M2 = 0x1C71C71Cu;
      const uint32_t o0 = __builtin_amdgcn_alignbit(w[1], w[0], 3), o1 = __builtin_amdgcn_alignbit(w[2], w[1], 3);
      f = u32x6_t{w[0] & M0, w[1] & M1, w[2] & M2, o0 & M0, o1 & M1, (w[2] >> 3) & M2};
    } else {
      // fields 2j (bit 12j): codes 3j, in place; fields 2j + 1: codes 3j + 1, two bits up;
      // the last ten fields (bit 132 + 6k): codes 3j + 2, from bit 68 on in place, those
      // below two bits up
      constexpr uint32_t E0 = 0x0F00F00Fu, E1 = 0xF00F00F0u, E2 = 0x00F00F00u;   // words 0, 3; 1; 2
      constexpr uint32_t O0 = 0xC03C03C0u, O1 = 0x03C03C03u, O2 = 0x3C03C03Cu;
      const uint32_t s0 = w[0] << 2, s1 = __builtin_amdgcn_alignbit(w[1], w[0], 30);
      const uint32_t s2 = __builtin_amdgcn_alignbit(w[2], w[1], 30), s3 = __builtin_amdgcn_alignbit(w[3], w[2], 30);
      f = u32x6_t{(w[0] & E0) | (s0 & O0), (w[1] & E1) | (s1 & O1), (w[2] & E2) | (s2 & O2), (w[3] & E0) | (s3 & O0),
                  (w[2] & 0xF00F00F0u) | (s0 & 0x03C03C00u) | (w[3] >> 30), (w[3] & E2) | (s1 & O2)};
    }
    typedef __attribute__((ext_vector_type(32))) __bf16 bf16x32_t;
    const bf16x32_t v = __builtin_amdgcn_cvt_scalef32_pk32_bf16_fp6(f, 8.0f);
    b[0] = __builtin_shufflevector(v, v, 0, 1, 2, 3, 4, 5, 6, 7);
    b[1] = __builtin_shufflevector(v, v, 8, 9, 10, 11, 12, 13, 14, 15);
    b[2] = __builtin_shufflevector(v, v, 16, 17, 18, 19, 20, 21, 22, 23);
    b[3] = __builtin_shufflevector(v, v, 24, 25, 26, 27, 28, 29, 30, 31);
  }
}

// A scale and a bias as stored, to fp32.  The dtype is uniform: two instructions behind a
// branch (in asm, or the compiler runs both conversions and selects: with 3- and 4-bit
// codes, whose converter leaves the fewest issue slots, 7 tokens 3-bit 212 against 195 us a
// layer; 2-bit codes measured 1 per cent the other way and keep the select).
template <int BITS>
__device__ __forceinline__ void scale_and_bias(uint32_t s, uint32_t b, bool f16, float& sw, float& bw) {
  if constexpr (BITS == 2) {
    sw = scale_bits_to_f32((uint16_t)s, f16);
    bw = scale_bits_to_f32((uint16_t)b, f16);
  } else if (f16) {
    asm("v_cvt_f32_f16 %0, %1" : "=v"(sw) : "v"(s));
    asm("v_cvt_f32_f16 %0, %1" : "=v"(bw) : "v"(b));
  } else {
    asm("v_lshlrev_b32 %0, 16, %1" : "=v"(sw) : "v"(s));
    asm("v_lshlrev_b32 %0, 16, %1" : "=v"(bw) : "v"(b));
  }
}

// What a wave loads of one macro into registers, in this order (after its A rows).
template <int AK>
struct SrMacro {
  uint4 ex[Sr<AK>::EX];                      // affine: the sums of A row lane (< TPT), four per chunk
  uint32_t codes[SR_FRAGS][Sr<AK>::CW];
};

// One workgroup takes a contiguous run of the items (tile, slice of 64 weight rows), an
// equal share of them (slots: the workgroups the chip holds at once; the runs are a whole
// number of rounds of them, so all of a round ends together); the macros of its items are
// one sequence per wave, RD - 1 of them in flight across the items' ends.
template <int AK, int NM, int NF>
__global__ void __launch_bounds__(SR_THREADS, 2) sr_kernel(SrArgs g, int slices, int slots) {
  using S = Sr<AK>;
  constexpr int TPT = S::TPT, MC = S::MC, GPC = S::GPC, G = S::G, BITS = S::BITS, RD = S::RD;
  static_assert(NM * NF == SR_FRAGS, "four fragments per wave");
  extern __shared__ __align__(16) uint8_t lds[];   // S::FIXED + 2 sr_scale_bytes
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, kg = lane >> 4;
  // this workgroup's items; neighbouring runs on one XCD
  const int64_t total = (int64_t)g.recs_n[0] * slices;
  const int runs = slots * sr_rounds(total, slots);
  const int xcds = 8, per = runs / xcds;
  const int run = (int)(blockIdx.x % xcds) * per + (int)blockIdx.x / xcds;
  if ((int)blockIdx.x >= runs) return;
  const int it0 = (int)(total * run / runs), it1 = (int)(total * (run + 1) / runs);
  if (it0 >= it1) return;

  uint8_t* aring = lds + wave * RD * S::STAGE;
  uint8_t* zrow = lds + S::RING;
  float* mysx = reinterpret_cast<float*>(zrow + S::ZROW + wave * S::WAVE);
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
        asrc[q] = g.a + (size_t)src * nch * SR_ROWB + (((lane & 15) ^ (r & 15)) << 4);
      }
      if constexpr (S::FOLD) {
        const int rr = row0 + min(lane & (TPT - 1), i_rows - 1);
        const int src = g.a_gather ? g.a_gather[rr] : rr;
        exsrc = reinterpret_cast<const uint8_t*>(g.asum + (size_t)src * nch * 4);
      }
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
        tile::lds_load16_untracked(asrc[q] + (size_t)min(m * MC + achunk, nch - 1) * SR_ROWB, stage + q * 1024);
    if constexpr (S::FOLD) {
#pragma unroll
      for (int q = 0; q < MC; ++q) out.ex[q] = *reinterpret_cast<const uint4*>(exsrc + (m * MC + q) * 16);
    }
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

  // the lane's A row: tile row i % TPT where the lane's block lies in the row's group, the
  // row of zeros elsewhere
  const int at = i % TPT, blk = sr_block<BITS>(kg);
  const bool own = blk * 32 / G == i / TPT % GPC;
  int col[4];                                                  // 16-byte columns of the four steps
#pragma unroll
  for (int q = 0; q < 4; ++q) col[q] = ((4 * blk + q) ^ at) << 4;
  const int dg = (4 * kg) / TPT % GPC;                         // the group of the lane's results
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
      // groups apart: rows [group][row of the tile], four per lane group
      if constexpr (TPT == 4 && GPC >= 2) t = t + xor_f<16>(t);
      if constexpr (GPC * TPT == 16) t = t + xor_f<32>(t);
      sum[p] = c_slot >= 0 ? t : 0.0f;
    }
    ++c_item;   // (the barrier at the next item's first step frees the stages)
    if (tr >= c_rows || kg >= TPT / 4) return;   // the same in the 16 lanes of a row group
    if constexpr (NM == 2) {
      uint16_t* dst = g.h + (size_t)c_prow * g.hkch * 128 + nw0;   // one 32-element block
      float hsv = 0.0f;
#pragma unroll
      for (int f = 0; f < NF; ++f) {
        float gv = round_bf16(sum[f]);
        float uv = round_bf16(sum[NF + f]);
        if (g.limit > 0.0f) {
          uv = fminf(fmaxf(uv, -g.limit), g.limit);
          gv = fminf(gv, g.limit);
        }
        const uint16_t hb = nw0 + 16 * f + i < g.N ? f32_to_bf16((silu_f32(gv) * uv) * c_w) : (uint16_t)0;
        dst[sr_pos<S::FOLD ? BITS : 0>(16 * f + i)] = hb;
        hsv = hsv + bf16_to_f32(hb);
      }
      if constexpr (S::FOLD) {   // the sum of the 32 h values (f, then the 16 lanes)
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
      if (S::FOLD && lane < TPT) {
#pragma unroll
        for (int q = 0; q < S::EX; ++q) {   // four sums of 32 per chunk -> one per group; none past K
          const bool in = m * MC + q < nch;
          const float a = in ? __uint_as_float(ring[v].ex[q].x) : 0.0f, b = in ? __uint_as_float(ring[v].ex[q].y) : 0.0f;
          const float c = in ? __uint_as_float(ring[v].ex[q].z) : 0.0f, d = in ? __uint_as_float(ring[v].ex[q].w) : 0.0f;
          float* o = mysx + q * GPC * TPT + lane;
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
      const uint8_t* a0 = GPC == 1 || own ? arow : zrow;
#pragma unroll
      for (int u = 0; u < MC; ++u) {
        const int c = m * MC + u;
        if (c >= nch) break;
        __builtin_amdgcn_sched_barrier(0);   // (chunks interleaved would spill)
        bf16x8_t a[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) a[q] = tile::lds_a(a0, u * SR_ROWB + col[q]);
        if constexpr (!S::FOLD) {
          const int eb = 4 * c + kg;                     // blocks past K meet zero A: any finite scale
          float es[SR_FRAGS];
#pragma unroll
          for (int p = 0; p < SR_FRAGS; ++p)
            es[p] = e8m0_to_f32(eb < groups ? sc[(16 * p + i) * groups + eb] : 127u);
#pragma unroll
          for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int p = 0; p < SR_FRAGS; ++p)
              acc[p] = tile::mfma(a[q], tile::fp4_codes_to_b(ring[v].codes[p][4 * u + q], es[p]), acc[p]);
        } else {
          const uint16_t* s16 = reinterpret_cast<const uint16_t*>(sc) + i * groups;
          const int go = min(GPC * c + dg, groups - 1);
          const bool in = GPC == 1 || GPC * c + dg < groups;   // groups past K: nothing
          const float4 sx = *reinterpret_cast<const float4*>(sxp + u * GPC * TPT);
          const float sxv[4] = {sx.x, sx.y, sx.z, sx.w};
          // (two fragments at a time, 3-bit one: more operands spill)
          constexpr int FA = BITS == 3 ? 1 : 2;
#pragma unroll
          for (int pp = 0; pp < SR_FRAGS; pp += FA) {
            bf16x8_t b[FA][4];
            f32x4_t d[FA];
#pragma unroll
            for (int p = 0; p < FA; ++p) {
              code_values<BITS>(ring[v].codes[pp + p] + BITS * u, b[p]);
              d[p] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
              for (int p = 0; p < FA; ++p) d[p] = tile::mfma(a[q], b[p][q], d[p]);
#pragma unroll
            for (int p = 0; p < FA; ++p) {
              float sw, bw;
              scale_and_bias<BITS>(s16[16 * (pp + p) * groups + go], s16[(64 + 16 * (pp + p)) * groups + go], g.L.f16,
                                   sw, bw);
              if (!in) sw = bw = 0.0f;
#pragma unroll
              for (int r = 0; r < 4; ++r) acc[pp + p][r] = fmaf(sw, d[p][r], fmaf(bw, sxv[r], acc[pp + p][r]));
            }
            __builtin_amdgcn_sched_barrier(0);
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

// x [T, D] -> rows in the order of sr_pos<BITS> and (sums != null) the sums of their
// 32-element blocks.  One thread = 8 values.
template <int BITS>
__global__ void __launch_bounds__(256) sr_rows_kernel(const uint16_t* __restrict__ x, int64_t n,
                                                      uint16_t* __restrict__ rows, float* __restrict__ sums) {
  __shared__ __align__(16) uint16_t st[2048];
  const int64_t at = (int64_t)blockIdx.x * 2048 + threadIdx.x * 8;
  const uint4 v = *reinterpret_cast<const uint4*>(x + (at < n ? at : 0));
  const uint32_t w[4] = {v.x, v.y, v.z, v.w};
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint16_t b = (uint16_t)(w[j >> 1] >> (16 * (j & 1)));
    const int e = threadIdx.x * 8 + j;
    st[(e & ~31) + sr_pos<BITS>(e & 31)] = b;
    s = s + bf16_to_f32(b);
  }
  s = s + __uint_as_float(xor1_u32(__float_as_uint(s)));
  s = s + __uint_as_float(xor2_u32(__float_as_uint(s)));
  __syncthreads();
  if (at >= n) return;
  *reinterpret_cast<uint4*>(rows + at) = *reinterpret_cast<const uint4*>(st + threadIdx.x * 8);
  if (sums != nullptr && (threadIdx.x & 3) == 0) sums[at / 32] = s;
}

template <int BITS>
int launch_sr_rows(const uint16_t* x, int64_t n, uint16_t* rows, float* sums, hipStream_t s) {
  hipLaunchKernelGGL(sr_rows_kernel<BITS>, dim3((unsigned)((n + 2047) / 2048)), dim3(256), 0, s, x, n, rows, sums);
  return check_launch("sr_rows_kernel");
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
  // max_tiles: at least the tiles there will be
  template <int NM, int NF>
  static int go(const SrArgs& a, int slices, int max_tiles, hipStream_t s) {
    const size_t bytes = lds(a.K);
    auto k = sr_kernel<AK, NM, NF>;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)bytes) != hipSuccess)
      return fail(CACHALOT_EHIP, "grouped experts (few rows): cannot grant %zu bytes of LDS", bytes);
    const int slots = 256 * (bytes <= 80 * 1024 ? 2 : 1);   // what the 256 CUs hold at once
    const int grid = slots * sr_rounds((int64_t)max_tiles * slices, slots);
    hipLaunchKernelGGL(k, dim3(grid), dim3(SR_THREADS), bytes, s, a, slices, slots);
    return check_launch("sr_kernel");
  }
  static int run(const SrArgs& gu, const SrArgs& dn, int rows, int E, hipStream_t s) {
    const int max_tiles = rows / Sr<AK>::TPT + std::min(E, rows);
    if (int rc = go<2, 2>(gu, gu.hkch * 4, max_tiles, s)) return rc;   // 32 columns of h per item
    return go<1, 4>(dn, (dn.N + 63) / 64, max_tiles, s);
  }
};

// Workspace: x in the kind's order [T][D], its sums [T][D / 32], h [rows][F_pad], its sums
// [rows][F_pad / 32] (64 bytes: a macro's sums past the last row).
struct SrWs {
  size_t x, xsum, h, hsum, total;
};
inline SrWs sr_ws(int T, int k, int D, int F) {
  const size_t rows = (size_t)T * k, fpad = (size_t)(F + 127) / 128 * 128;
  SrWs w;
  w.x = 0;
  w.xsum = w.x + align256((size_t)T * D * 2);
  w.h = w.xsum + align256((size_t)T * (D / 32) * 4 + 64);
  w.hsum = w.h + align256(rows * fpad * 2);
  w.total = w.hsum + align256(rows * (fpad / 32) * 4 + 64);
  return w;
}

}  // namespace

size_t small_rows_ws_bytes(int T, int k, int D, int F) { return sr_ws(T, k, D, F).total; }

// Rows per tile of a bank kind (the tile list's MT); bits 0: FP4.
int small_rows_mt(int bits, int group) { return sr_tpt(sr_kind(bits, group)); }

// Calls go(integral constant SK) for the kind, or returns `otherwise`.
template <typename R, typename Fn>
static R sr_dispatch(int sk, R otherwise, Fn&& go) {
#define CACHALOT_SR(K) \
  if (sk == (K)) return go(std::integral_constant<int, (K)>());
  CACHALOT_SR(SR_FP4)
  CACHALOT_SR(sr_kind(2, 32)) CACHALOT_SR(sr_kind(2, 64)) CACHALOT_SR(sr_kind(2, 128))
  CACHALOT_SR(sr_kind(3, 32)) CACHALOT_SR(sr_kind(3, 64)) CACHALOT_SR(sr_kind(3, 128))
  CACHALOT_SR(sr_kind(4, 32)) CACHALOT_SR(sr_kind(4, 64)) CACHALOT_SR(sr_kind(4, 128))
#undef CACHALOT_SR
  return otherwise;
}

// A row's last chunk is read whole (2- and 3-bit codes): past a tensor's last row, where
// the row is shorter, up to 36 bytes (3-bit, K = 128 n + 32), which must still lie inside
// the slot record.
bool small_rows_supported(int bits, int group, int D, int F, const decode::Layout& L) {
  if (!(D % 128 == 0 && D >= 128 && D <= 8192 && F % 32 == 0 && F >= 32 && F <= 8192)) return false;
  if (L.record_bytes > 0x7fffffff) return false;   // offsets inside a record are 32-bit
  const bool fold = bits != 0;
  const int mats[3][3] = {{0, F, D}, {6, F, D}, {3, D, F}};   // w1, w3, w2: tensor, rows, K
  for (auto& m : mats) {
    const int64_t n = m[1], k = m[2], nch = (k + 127) / 128;
    const int64_t rb = fold ? (k + group - 1) / group * group * bits / 8 : k / 2;
    const int64_t code_over = bits == 4 || !fold ? 0 : nch * 16 * bits - rb;
    if (rb < 16 || L.off[m[0]] + n * rb + code_over > L.record_bytes) return false;
  }
  return sr_dispatch(sr_kind(bits, group), false, [&](auto sk) {
    return SrLaunch<decltype(sk)::value>::fits(D) && SrLaunch<decltype(sk)::value>::fits(F);
  });
}

// recs: the tiles of small_rows_mt rows (tile_recs_kernel).
int launch_small_rows(int bits, int group, const uint16_t* x, int T, const uint8_t* pool, const decode::Layout& L,
                      const int4* recs, const int32_t* recs_n, const int32_t* row_token, const int32_t* row_slot,
                      const float* row_w, int D, int F, int E, int k, float limit, uint8_t* ws, uint16_t* y, hipStream_t s) {
  const SrWs w = sr_ws(T, k, D, F);
  uint16_t* xr = reinterpret_cast<uint16_t*>(ws + w.x);
  float* xsum = reinterpret_cast<float*>(ws + w.xsum);
  float* hsum = reinterpret_cast<float*>(ws + w.hsum);
  const int64_t n = (int64_t)T * D;
  const uint16_t* a = xr;
  int rc = CACHALOT_OK;
  if (bits == 2) rc = launch_sr_rows<2>(x, n, xr, xsum, s);
  else if (bits == 3) rc = launch_sr_rows<3>(x, n, xr, xsum, s);
  else if (bits == 4) rc = launch_sr_rows<4>(x, n, xr, xsum, s);
  else if (((uintptr_t)x & 15) != 0) rc = launch_sr_rows<0>(x, n, xr, nullptr, s);   // (LDS loads of 16 bytes)
  else a = x;
  if (rc) return rc;
  const int fch = (F + 127) / 128;
  const SrArgs gu{reinterpret_cast<const uint8_t*>(a), D / 128, row_token, xsum, pool, L, recs, recs_n, row_token,
                  row_slot, row_w, D, F, k, limit, reinterpret_cast<uint16_t*>(ws + w.h), fch, hsum, nullptr};
  const SrArgs dn{ws + w.h, fch, nullptr, hsum, pool, L, recs, recs_n, row_token,
                  row_slot, row_w, F, D, k, limit, nullptr, 0, nullptr, y};
  rc = sr_dispatch(sr_kind(bits, group), -1, [&](auto sk) { return SrLaunch<decltype(sk)::value>::run(gu, dn, T * k, E, s); });
  return rc >= 0 ? rc : fail(CACHALOT_EINVAL, "grouped experts (few rows): %d-bit codes in groups of %d", bits, group);
}

}  // namespace cachalot
