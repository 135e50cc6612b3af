// Router: logits -> score function -> biased top-k -> normalised weights.
//
// Reference semantics: src/cachalot/model/router_mlx.py:29-37 (DeepSeek),
// router_fused_metal.py:32-108 (fused kernels, tie rule), minimax/language.py:
// 280-292 and minimax/gpu_select.py:80-115 (sigmoid, rank order).
//
// Arithmetic contract (fixed so ids are reproducible bit for bit):
//   * D is cut into 64 contiguous chunks of D/64; lane l owns chunk l and adds
//     its bf16*bf16 products (exact in fp32) sequentially in fp32;
//   * the 64 partials are combined by the xor butterfly 1, 2, 4, 8, 16, 32
//     (pairwise summation over the chunks in natural order);
//   * logit = sum / gate_temp (fp32);
//   * score functions use only IEEE basic operations (Cody-Waite exp with
//     a degree-13 Taylor polynomial, an atanh series for log1p), so a host
//     evaluation with the same steps agrees exactly;
//   * selection = score + bias; top-k by rank counting with the order's tie rule.
//
// Kernels
//   router_scores_kernel  one wave = 4 expert rows x up to TT tokens; W row chunks
//                         are loaded once per wave and reused for TT tokens.
//   router_topk_kernel    one wave per token; k rounds of a wave-wide argmax
//                         under the order's total order (value, then index).
#include <algorithm>

#include "mx_tile.h"
#include "router_launch.h"
#include "router_math.h"
#include "topk.h"

namespace cachalot {
namespace {

// Top-k tail for one token: every workgroup counts itself finished; the last one
// selects the experts (one wave), normalises the weights, resolves the slots and
// returns the counter to zero.  Protocol: the scores are stored with agent-scope
// (write-through) stores and each wave waits for its stores to complete before
// the workgroup counts itself with a returning agent-scope add; the selecting
// wave reads the scores with agent-scope loads.  (No release/acquire fences:
// those write back / invalidate whole L2s.)
__device__ __forceinline__ void route_tail(const float* __restrict__ scores, const decode::RouteTail& tail) {
  __shared__ int last;
  __shared__ int top_i[decode::KMAX], top_s[decode::KMAX];
  __shared__ float top_v[decode::KMAX];
  __shared__ float w[decode::KMAX];
  __builtin_amdgcn_s_waitcnt(0x0F70);   // vmcnt(0): this wave's score stores are complete
  __syncthreads();
  if (threadIdx.x == 0) {
    const unsigned done = __hip_atomic_fetch_add(tail.counter, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = done == gridDim.x * gridDim.y - 1;
  }
  __syncthreads();
  if (!last || threadIdx.x >= 64) return;
  if (tail.E <= 384)
    wave_topk<6, true>(scores, tail.bias, tail.E, tail.k, tail.order, top_i, top_v, tail.slot_table, top_s);
  else
    wave_topk<16, true>(scores, tail.bias, tail.E, tail.k, tail.order, top_i, top_v, tail.slot_table, top_s);
  if (threadIdx.x == 0) normalise_weights(top_v, tail.k, tail.route_scale, tail.norm, w);
  if ((int)threadIdx.x < tail.k) {
    tail.ws_slots[threadIdx.x] = top_s[threadIdx.x];
    tail.ws_w[threadIdx.x] = w[threadIdx.x];
    if (tail.idx_out) tail.idx_out[threadIdx.x] = top_i[threadIdx.x];
    if (tail.w_out) tail.w_out[threadIdx.x] = w[threadIdx.x];
  }
  if (threadIdx.x == 0) __hip_atomic_store(tail.counter, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// One wave per expert row (lane l owns chunk l of D/64 elements), TT tokens per
// wave, blockDim / 64 waves per workgroup; optionally the top-k tail (one token).
template <int TT, int NV>
__global__ void __launch_bounds__(256) router_scores_kernel(const uint16_t* __restrict__ x,
                                                            const uint16_t* __restrict__ W, int T, int D,
                                                            int E, float gate_temp, int fn,
                                                            float* __restrict__ scores, decode::RouteTail tail,
                                                            uint8_t* __restrict__ xplanes) {
  const int lane = threadIdx.x & 63;
  const int row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (xplanes != nullptr && blockIdx.y == 0) {   // token 0 as fp8 planes for the matrix-core decode
    for (int t4 = blockIdx.x * blockDim.x + threadIdx.x; 4 * t4 < D; t4 += gridDim.x * blockDim.x)
      mx::encode_x_quad(xplanes, t4, reinterpret_cast<const uint2*>(x)[t4]);   // whole quads of lanes
  }
  if (row < E) router_row<TT, NV>(x, W, T, D, E, gate_temp, fn, scores, row, lane, tail.counter != nullptr);
  if (tail.counter != nullptr) route_tail(scores, tail);
}

// One wave per token: k rounds of a wave-wide argmax (EPT = ceil(E / 64) candidates per lane).
template <int EPT>
__global__ void __launch_bounds__(64) router_topk_kernel(const float* __restrict__ scores,
                                                         const float* __restrict__ bias,
                                                         const float* __restrict__ bias_vl,
                                                         const uint8_t* __restrict__ image_mask, int E, int k,
                                                         float route_scale, int norm, int order,
                                                         int32_t* __restrict__ idx, float* __restrict__ w) {
  __shared__ int top_i[1024];
  __shared__ float top_v[1024];
  const int t = blockIdx.x;
  const float* s = scores + (size_t)t * E;
  const float* b = (image_mask != nullptr && image_mask[t] != 0) ? bias_vl : bias;
  wave_topk<EPT>(s, b, E, k, order, top_i, top_v);
  __syncthreads();
  for (int j = threadIdx.x; j < k; j += 64) idx[(size_t)t * k + j] = top_i[j];
  if (threadIdx.x == 0) normalise_weights(top_v, k, route_scale, norm, w + (size_t)t * k);
}

// Many tokens: one workgroup = 16 TA tokens x 32 experts, each thread TA tokens (tq + 16
// a) x 2 experts (eq + 16 b).  The same arithmetic as router_row: chunk c (of 64) of every
// dot product is a sequential fp32 sum of its D/64 products in k order, and the 64 chunk
// sums meet in the pairwise tree (left + right) the xor butterfly forms, kept as a
// binary-counter stack of partial nodes per dot product.  Chunk by chunk, the x and W
// slices are staged in LDS as bf16 (double-buffered, one barrier per chunk) and read as
// 8-value runs (one 16-byte read per token or expert feeds 8 x 2 TA products); rows are
// padded to an odd number of 16-byte slots so the 16 experts a wave row reads hit distinct
// bank groups.  fma(x, w, s) equals s + x * w here: the product of two bf16 values is
// exact in fp32 (16 significant bits) unless it is below 2^-133.
//
// SP: the chunks are dealt to SP groups of 256 threads, a run of 64 / SP each (a subtree of
// the pairwise sum), whose roots meet at the end.  What bounds the kernel is the fp32
// multiply-adds, so it wants every SIMD busy: SP = 1 needs several workgroups per CU for
// that, SP = 4 one.
constexpr int RT_TB = 2;             // experts per thread (eq + 16 b)
constexpr int RT_E = 16 * RT_TB;     // experts per workgroup
constexpr int RT_MAXCH = 80;         // D / 64 <= 80 (D <= 5120)

constexpr int64_t RT_MIN_DOTS = 160 * 384;   // scores

__host__ __device__ inline int rt_stride(int ch) { return ch * 2 + ((ch / 8) % 2 == 0 ? 16 : 32); }

// Chunk c of a tile's x rows, then its W rows, as 16-byte items (rows past T / E:
// clamped, unused), and the store of those items into a staged buffer (threads past the
// last item carry it again).  Plain vectors and stores without a condition: as uint4 under
// one, the items in flight went through scratch memory, each waited for (4096 tokens x 384
// experts, unsplit: 321 us against 275 us).
typedef uint32_t rt_item __attribute__((ext_vector_type(4)));
template <int N, int TT>
__device__ __forceinline__ void rt_load(rt_item (&v)[N], const uint16_t* __restrict__ x, const uint16_t* __restrict__ W,
                                        int T, int D, int E, int t0, int e0, int c, int tid, int items, int per_row) {
  const int ch = 8 * per_row;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int it = min(tid + 256 * j, items - 1);
    const int r = it / per_row, q = it - r * per_row;
    const uint16_t* src = r < TT ? x + (size_t)min(t0 + r, T - 1) * D : W + (size_t)min(e0 + r - TT, E - 1) * D;
    v[j] = *reinterpret_cast<const rt_item*>(src + c * ch + 8 * q);
  }
}

template <int N>
__device__ __forceinline__ void rt_store(uint8_t* buf, const rt_item (&v)[N], int tid, int items, int per_row, int S) {
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int it = min(tid + 256 * j, items - 1);
    const int r = it / per_row, q = it - r * per_row;
    *reinterpret_cast<rt_item*>(buf + r * S + 16 * q) = v[j];
  }
}

// dynamic LDS = SP * 2 * (16 TA + RT_E) * rt_stride(D / 64)
template <int TA, int SP>
__global__ void __launch_bounds__(256 * SP) router_tiled_kernel(const uint16_t* __restrict__ x,
                                                                const uint16_t* __restrict__ W, int T, int D, int E,
                                                                float gate_temp, int fn,
                                                                float* __restrict__ scores) {
  constexpr int TT = 16 * TA;                 // tokens per workgroup
  constexpr int NC = CHUNKS / SP;             // chunks per group
  constexpr int LEV = NC == 64 ? 6 : 4;       // levels of a group's subtree
  static_assert(NC == 64 || NC == 16, "SP is 1 or 4");
  extern __shared__ __align__(16) uint8_t rt_lds[];
  const int grp = SP == 1 ? 0 : threadIdx.x >> 8;
  const int tid = threadIdx.x & 255;
  const int eq = tid & 15, tq = tid >> 4;
  const int t0 = blockIdx.x * TT, e0 = blockIdx.y * RT_E;
  const int per_row = D / 512;                // 16-byte items per staged row
  const int ch = 8 * per_row;                 // D / 64
  const int S = rt_stride(ch);
  const int items = (TT + RT_E) * per_row;    // x rows first, then W rows
  constexpr int MAXIT = ((TT + RT_E) * RT_MAXCH / 8 + 255) / 256;
  uint8_t* st = rt_lds + grp * 2 * (TT + RT_E) * S;
  const int c0 = grp * NC;

  float stk[LEV][TA * RT_TB];
  float node[TA * RT_TB];
  rt_item v[MAXIT];
  rt_load<MAXIT, TT>(v, x, W, T, D, E, t0, e0, c0, tid, items, per_row);
  rt_store(st, v, tid, items, per_row, S);
  __syncthreads();
  for (int c = 0; c < NC; ++c) {
    if (c + 1 < NC) rt_load<MAXIT, TT>(v, x, W, T, D, E, t0, e0, c0 + c + 1, tid, items, per_row);
    const uint8_t* buf = st + (c & 1) * (TT + RT_E) * S;
    float acc[TA * RT_TB];
#pragma unroll
    for (int p = 0; p < TA * RT_TB; ++p) acc[p] = 0.0f;
    // (a runtime loop: unrolled, the scheduled-ahead reads push the kernel to one wave per SIMD)
    for (int k8 = 0; k8 < per_row; ++k8) {
      uint4 xa[TA], wb[RT_TB];
#pragma unroll
      for (int a = 0; a < TA; ++a) xa[a] = *reinterpret_cast<const uint4*>(buf + (tq + 16 * a) * S + 16 * k8);
#pragma unroll
      for (int b = 0; b < RT_TB; ++b)
        wb[b] = *reinterpret_cast<const uint4*>(buf + (TT + eq + 16 * b) * S + 16 * k8);
#pragma unroll
      for (int h = 0; h < 4; ++h) {            // the 8 values in k order: word h, low then high half
        float xl[TA], xh[TA], wl[RT_TB], wh[RT_TB];
#pragma unroll
        for (int a = 0; a < TA; ++a) {
          const uint32_t u = h == 0 ? xa[a].x : h == 1 ? xa[a].y : h == 2 ? xa[a].z : xa[a].w;
          xl[a] = __uint_as_float(u << 16);
          xh[a] = __uint_as_float(u & 0xffff0000u);
        }
#pragma unroll
        for (int b = 0; b < RT_TB; ++b) {
          const uint32_t u = h == 0 ? wb[b].x : h == 1 ? wb[b].y : h == 2 ? wb[b].z : wb[b].w;
          wl[b] = __uint_as_float(u << 16);
          wh[b] = __uint_as_float(u & 0xffff0000u);
        }
#pragma unroll
        for (int a = 0; a < TA; ++a)
#pragma unroll
          for (int b = 0; b < RT_TB; ++b) {
            float t = acc[RT_TB * a + b];
            t = __builtin_fmaf(xl[a], wl[b], t);
            t = __builtin_fmaf(xh[a], wh[b], t);
            acc[RT_TB * a + b] = t;
          }
      }
    }
    if (c + 1 < NC) rt_store(st + ((c + 1) & 1) * (TT + RT_E) * S, v, tid, items, per_row, S);
    // merge chunk c into the tree (c is uniform: every branch below is too)
#pragma unroll
    for (int p = 0; p < TA * RT_TB; ++p) node[p] = acc[p];
    // chunk c closes the nodes of the levels below its lowest zero bit
    const int up = __builtin_ctz(~c);   // levels merged (LEV after the last chunk)
#pragma unroll
    for (int L = 0; L < LEV; ++L) {
      if (L < up) {
#pragma unroll
        for (int p = 0; p < TA * RT_TB; ++p) node[p] = stk[L][p] + node[p];
      } else if (L == up) {
#pragma unroll
        for (int p = 0; p < TA * RT_TB; ++p) stk[L][p] = node[p];
      }
    }
    __syncthreads();
  }
  // after the last chunk every level merged: node holds the group's root
  if constexpr (SP == 4) {   // (g0 + g1) + (g2 + g3), by group 0 (the staging is done with)
    float* roots = reinterpret_cast<float*>(rt_lds);   // [group][dot][thread]
#pragma unroll
    for (int p = 0; p < TA * RT_TB; ++p) roots[(grp * TA * RT_TB + p) * 256 + tid] = node[p];
    __syncthreads();
    if (grp != 0) return;
#pragma unroll
    for (int p = 0; p < TA * RT_TB; ++p) {
      const float* r = roots + p * 256 + tid;
      constexpr int G = TA * RT_TB * 256;
      node[p] = (r[0] + r[G]) + (r[2 * G] + r[3 * G]);
    }
  }
#pragma unroll
  for (int a = 0; a < TA; ++a) {
    const int t = t0 + tq + 16 * a;
    if (t >= T) continue;
#pragma unroll
    for (int b = 0; b < RT_TB; ++b) {
      const int e = e0 + eq + 16 * b;
      if (e < E) scores[(size_t)t * E + e] = score_of(node[RT_TB * a + b] / gate_temp, fn);
    }
  }
}

template <int TA, int SP>
int launch_tiled(const uint16_t* x, const uint16_t* W, int T, int D, int E, float gate_temp, int fn, float* scores,
                 hipStream_t s) {
  const size_t lds = (size_t)SP * std::max((size_t)2 * (16 * TA + RT_E) * rt_stride(D / CHUNKS),
                                           SP == 1 ? (size_t)0 : (size_t)TA * RT_TB * 256 * 4);
  auto k = router_tiled_kernel<TA, SP>;
  if (hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) !=
      hipSuccess)
    return fail(CACHALOT_EHIP, "router: cannot grant %zu bytes of LDS", lds);
  hipLaunchKernelGGL(k, dim3((T + 16 * TA - 1) / (16 * TA), (E + RT_E - 1) / RT_E), dim3(256 * SP), lds, s, x, W, T, D,
                     E, gate_temp, fn, scores);
  return check_launch("router_tiled_kernel");
}

}  // namespace

template <int TT>
static void launch_scores_tt(const uint16_t* x, const uint16_t* W, int T, int D, int E, float temp, int fn,
                             float* scores, hipStream_t s, const decode::RouteTail& tail, uint8_t* xplanes) {
  // one token: one wave per workgroup, so the E rows spread over every CU
  const int wpb = TT == 1 ? 1 : 4;
  const dim3 grid((E + wpb - 1) / wpb, (T + TT - 1) / TT), block(64 * wpb);
  switch (D) {
    case 4096: hipLaunchKernelGGL((router_scores_kernel<TT, 8>), grid, block, 0, s, x, W, T, D, E, temp, fn, scores, tail, xplanes); break;
    case 5120: hipLaunchKernelGGL((router_scores_kernel<TT, 10>), grid, block, 0, s, x, W, T, D, E, temp, fn, scores, tail, xplanes); break;
    case 7168: hipLaunchKernelGGL((router_scores_kernel<TT, 14>), grid, block, 0, s, x, W, T, D, E, temp, fn, scores, tail, xplanes); break;
    default: hipLaunchKernelGGL((router_scores_kernel<TT, 0>), grid, block, 0, s, x, W, T, D, E, temp, fn, scores, tail, xplanes); break;
  }
}

int launch_router_scores(const uint16_t* x, const uint16_t* W, int T, int D, int E, float gate_temp, int fn,
                         float* scores, hipStream_t s, const decode::RouteTail* tail, uint8_t* xplanes) {
  decode::RouteTail none{};
  // The tiled kernel from RT_MIN_DOTS scores on (384 experts: 160 tokens, 74 us on the
  // 4-token kernel against 44; 1000 tokens 410 against 95; with 8 experts, 4096 tokens, the
  // same 48 us, 16384 tokens 166 against 110).  Of 16, 32 and 64 tokens per tile with the chunks
  // split and 64 unsplit the one whose rounds of 256 workgroups take least, by what they
  // take at D = 4096 (us, router and top-k, 384 experts: measured 16 / 32 / 64 / unsplit at
  // 500 tokens 69 / 62 / 91 / 175, 1500: 149 / 163 / 173 / 193, 2049: 201 / 215 / 175 / 200, 4096:
  // 341 / 319 / 260 / 275, 8192: 673 / 632 / 511 / 477).  Unsplit, up to four workgroups share a CU,
  // and the first two of them cost little more than one.
  if ((int64_t)T * E >= RT_MIN_DOTS && D % 512 == 0 && D / CHUNKS <= RT_MAXCH) {
    const int et = (E + RT_E - 1) / RT_E;
    auto rounds = [&](int tokens) { return ((int64_t)((T + tokens - 1) / tokens) * et + 255) / 256; };
    const int64_t c16 = 26 * rounds(16) + 18, c32 = 52 * rounds(32) + 8, c64 = 84 * rounds(64) + 6;
    const int64_t whole = std::max<int64_t>(176, 68 * rounds(64) + 70);
    const int64_t least = std::min(std::min(c16, c32), std::min(c64, whole));
    if (whole == least) return launch_tiled<4, 1>(x, W, T, D, E, gate_temp, fn, scores, s);
    if (c64 == least) return launch_tiled<4, 4>(x, W, T, D, E, gate_temp, fn, scores, s);
    if (c32 == least) return launch_tiled<2, 4>(x, W, T, D, E, gate_temp, fn, scores, s);
    return launch_tiled<1, 4>(x, W, T, D, E, gate_temp, fn, scores, s);
  }
  // tokens per wave: 4 from 8 tokens on, 2 below (twice the waves for a small batch:
  // B = 4 68.4 against 70 us per batched step; at B = 32, 2 per wave lost 2.6 us)
  if (T >= 8) launch_scores_tt<4>(x, W, T, D, E, gate_temp, fn, scores, s, none, nullptr);
  else if (T >= 4) launch_scores_tt<2>(x, W, T, D, E, gate_temp, fn, scores, s, none, nullptr);
  else launch_scores_tt<1>(x, W, T, D, E, gate_temp, fn, scores, s, tail && T == 1 ? *tail : none, xplanes);
  return check_launch("router_scores_kernel");
}

}  // namespace cachalot

extern "C" int cachalot_router_topk(const uint16_t* x, const uint16_t* W, const float* bias,
                                    const float* bias_vl, const uint8_t* image_mask, int T, int D, int E,
                                    int k, int score_fn, float gate_temp, float route_scale, int norm,
                                    int order, int32_t* idx, float* w, float* scores,
                                    cachalot_stream_t stream) {
  using namespace cachalot;
  CACHALOT_REQUIRE(x && W && bias && idx && w && scores, "router: null pointer");
  CACHALOT_REQUIRE(T >= 1, "router: x must contain at least one token (T=%d)", T);
  CACHALOT_REQUIRE(D >= 128 && D % 128 == 0, "router: D=%d must be a positive multiple of 128", D);
  CACHALOT_REQUIRE(E >= 1 && E <= 1024, "router: E=%d outside 1..1024", E);
  CACHALOT_REQUIRE(k >= 1 && k <= E, "router: invalid topk=%d for %d experts", k, E);
  CACHALOT_REQUIRE(score_fn == CACHALOT_SCORE_SQRT_SOFTPLUS || score_fn == CACHALOT_SCORE_SIGMOID,
                   "router: unknown score function %d", score_fn);
  CACHALOT_REQUIRE(order == CACHALOT_ORDER_ASCENDING || order == CACHALOT_ORDER_RANK,
                   "router: unknown order %d", order);
  CACHALOT_REQUIRE(gate_temp != 0.0f, "router: gate_temp must be non-zero");
  CACHALOT_REQUIRE((image_mask == nullptr) == (bias_vl == nullptr),
                   "router: bias_vl and image_mask must be supplied together, or neither");
  hipStream_t s = (hipStream_t)stream;
  int rc = launch_router_scores(x, W, T, D, E, gate_temp, score_fn, scores, s);
  if (rc) return rc;
  if (E <= 384)
    hipLaunchKernelGGL((router_topk_kernel<6>), dim3(T), dim3(64), 0, s, scores, bias, bias_vl, image_mask, E, k,
                       route_scale, norm, order, idx, w);
  else
    hipLaunchKernelGGL((router_topk_kernel<16>), dim3(T), dim3(64), 0, s, scores, bias, bias_vl, image_mask, E, k,
                       route_scale, norm, order, idx, w);
  return check_launch("router_topk_kernel");
}
