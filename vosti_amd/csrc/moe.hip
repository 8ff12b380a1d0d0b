// A mixture of small feed-forward experts, each token through its `top` best of E: the router, the plan that sorts
// (token, choice) pairs by expert into tiles of rows, the two projections as grouped products on the matrix unit,
// and the weighted sum of a token's experts.
//
//   z = W_router h (32-bit sums of the elements' exact products);  s = softmax(z) over all experts;  the `top` largest
//   s (the lower index wins a tie);  weight_k = s_k / (sum of the chosen s + weight_eps);
//   out = sum over the chosen k, in the order they were chosen, of weight_k * W_down[e_k] act(W_up[e_k] h),
//   act(u) = max(u, 0)^2.
//
// A row of a grouped product depends on its own inputs only, and its sums have the order of this library's other
// matrix products, so a token's result does not depend on which other tokens share its tile or where the plan put it,
// and a caller may run an expert's rows through those products instead (many rows an expert) to the same bits.
#include <algorithm>

#include "common.h"
#include "lines.h"
#include "mma.h"
#include "vec.h"

#define MOE_TILE 16          // rows of a tile: pairs of one expert
#define MOE_ROUTE_TOKENS 8   // tokens a router workgroup shares an expert's weights among

// Router logits z [T, E] floats.  A workgroup of four waves takes MOE_ROUTE_TOKENS tokens and one expert; the waves
// split the row's 16-byte vectors (vector v goes to wave (v / 64) % 4, lane v % 64), a lane adds its products in ascending
// order (fused multiply-adds), a butterfly follows over the lanes and the four waves' sums are added in wave order: the
// order depends on the width alone.
// bias: one number an expert that is added to its logit (elements or floats), or null.
// EX: experts of a workgroup, one after the other on the rows it holds: with one every expert's workgroup reads a group's rows again from
// the second-level cache, which a prompt's 32 experts wait for (2,048 tokens of 4,096 entries: 37 us, with four 24); fewer tokens want the workgroups (route_launch).
template <int EX>
__global__ __launch_bounds__(256) void moe_logits_kernel(float* __restrict__ z, const elem_t* __restrict__ h, const elem_t* __restrict__ router,
                                                         int T, int W, int E, const void* __restrict__ bias, int bias_is_f32) {
  __shared__ float part[4][EX][MOE_ROUTE_TOKENS];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t0 = blockIdx.x * MOE_ROUTE_TOKENS, e0 = blockIdx.y * EX;
  if (t0 >= T) return;         // the grid is rounded up: the whole workgroup
  float acc[EX][MOE_ROUTE_TOKENS];
#pragma unroll
  for (int x = 0; x < EX; ++x)
#pragma unroll
    for (int i = 0; i < MOE_ROUTE_TOKENS; ++i) acc[x][i] = 0.f;
  const elem_t* wr = router + (int64_t)e0 * W;
  auto step = [&](int c) {
    float wv[EX][VK_VEC];
#pragma unroll
    for (int x = 0; x < EX; ++x) load_elems(wr + (int64_t)x * W + c, wv[x]);
#pragma unroll
    for (int i = 0; i < MOE_ROUTE_TOKENS; ++i) {
      float hv[VK_VEC];
      load_elems(h + (int64_t)min(t0 + i, T - 1) * W + c, hv);
#pragma unroll
      for (int x = 0; x < EX; ++x)
#pragma unroll
        for (int j = 0; j < VK_VEC; ++j) acc[x][i] = __builtin_fmaf(hv[j], wv[x][j], acc[x][i]);
    }
  };
  if constexpr (EX == 1) {
#pragma unroll 2
    for (int c = threadIdx.x * VK_VEC; c < W; c += 256 * VK_VEC) step(c);
  } else {
#pragma unroll 1
    for (int c = threadIdx.x * VK_VEC; c < W; c += 256 * VK_VEC) step(c);
  }
#pragma unroll
  for (int x = 0; x < EX; ++x)
#pragma unroll
    for (int i = 0; i < MOE_ROUTE_TOKENS; ++i) {
      const float v = wave_sum_xor(acc[x][i]);
      if (lane == 0) part[wave][x][i] = v;
    }
  __syncthreads();
  if (threadIdx.x < EX * MOE_ROUTE_TOKENS) {
    const int x = threadIdx.x / MOE_ROUTE_TOKENS, i = threadIdx.x % MOE_ROUTE_TOKENS;
    if (t0 + i < T) {
      float v = part[0][x][i];
      v = v + part[1][x][i];
      v = v + part[2][x][i];
      v = v + part[3][x][i];
      if (bias != nullptr) v = v + load_weight(bias, bias_is_f32, e0 + x);
      z[(int64_t)(t0 + i) * E + e0 + x] = v;
    }
  }
}

// LDS traffic between the lanes of a wave: what was written before is read after.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The place of the largest of v[0 .. n) over a wave (the lower index wins a tie; -inf is never the largest).
__device__ __forceinline__ int wave_argmax(const float* v, int n, int lane, float& best) {
  best = -INFINITY;
  int at = 0x7fffffff;
  for (int i = lane; i < n; i += 64) {
    const float x = v[i];
    if (x > best) { best = x; at = i; }
  }
  auto step = [&](float ov, int oe) {
    if (ov > best || (ov == best && oe < at)) { best = ov; at = oe; }
  };
  const auto as_float = [&] { return __builtin_bit_cast(float, at); };
#define ARGMAX_STEP(OFF) step(wave_partner<OFF>(best), __builtin_bit_cast(int, wave_partner<OFF>(as_float())))
  ARGMAX_STEP(32);
  ARGMAX_STEP(16);
  ARGMAX_STEP(8);
  ARGMAX_STEP(4);
  ARGMAX_STEP(2);
  ARGMAX_STEP(1);
#undef ARGMAX_STEP
  return min(at, n - 1);        // scores that are no numbers must not become an address
}

// The choice: idx [T, top] int32, wts [T, top] floats from the logits.  One wave per token, four tokens a workgroup.
// score 0: the softmax over all experts, the chosen scores divided by their sum plus weight_eps; score 1: the logistic
// function of every logit, the chosen scores as they are (the order of the scores is the order of the logits either way);
// score 2: the softmax over all experts, the chosen scores as they are.  Every weight is multiplied by `scale` at the end.
// groups > 1 with keep < groups: the experts form that many equal runs of neighbours; a group's score is its largest
// (group_score 0) or the sum of its two largest (1), and only experts of the `keep` best groups can be chosen.
// correction (score 1 only; [E] elements or floats, or null): a number an expert that joins its score for the choice, of groups
// and of experts, and not its weight.  Scores so corrected may be negative.
// scores: LDS of the workgroup, [waves][E], with a correction [waves][E] of the scores without it, then [waves][groups].
struct MoeChoice {
  int32_t* idx;
  float* wts;
  const float* logits;
  int T, E, top;
  float weight_eps;
  int score_kind, groups, keep;
  float scale;
  int group_score;
  const void* correction;
  int correction_is_f32;
};
__device__ __forceinline__ void moe_choose_token(const MoeChoice& a, float* scores, int t, int wave, int waves, int lane) {
  int32_t* idx = a.idx;
  float* wts = a.wts;
  const float* logits = a.logits;
  const int E = a.E, top = a.top, score_kind = a.score_kind, groups = a.groups, keep = a.keep, group_score = a.group_score, correction_is_f32 = a.correction_is_f32;
  const float weight_eps = a.weight_eps, scale = a.scale;
  const void* correction = a.correction;
  float* z = scores + wave * E;
  float* raw = correction != nullptr ? z + waves * E : z;
  float mx = -INFINITY;
  for (int e = lane; e < E; e += 64) {
    z[e] = logits[(int64_t)t * E + e];
    mx = fmaxf(mx, z[e]);
  }
  mx = wave_max_xor(mx);
  float sum = 0.f;
  for (int e = lane; e < E; e += 64) {
    const float p = score_kind == 1 ? 1.f / (1.f + expf(-z[e])) : expf(z[e] - mx);
    raw[e] = p;
    if (correction != nullptr) z[e] = p + load_weight(correction, correction_is_f32, e);
    sum = sum + p;
  }
  sum = score_kind == 1 ? 1.f : wave_sum_xor(sum);
  if (keep < groups) {
    // A kept group's score is marked with -inf; the experts of the others are then marked as if they had been chosen.
    float* gs = scores + (correction != nullptr ? 2 : 1) * waves * E + wave * groups;
    const int size = E / groups;
    wave_lds_fence();
    for (int g = lane; g < groups; g += 64) {
      float m = -INFINITY, second = -INFINITY;
      for (int j = 0; j < size; ++j) {
        const float v = z[g * size + j];
        second = fmaxf(second, fminf(m, v));
        m = fmaxf(m, v);
      }
      gs[g] = group_score == 1 && size > 1 ? m + second : m;
    }
    wave_lds_fence();
    for (int k = 0; k < keep; ++k) {
      float best;
      const int g = wave_argmax(gs, groups, lane, best);
      if (lane == 0) gs[g] = -INFINITY;
      wave_lds_fence();
    }
    for (int e = lane; e < E; e += 64)
      if (gs[e / size] > -INFINITY) z[e] = -INFINITY;
    wave_lds_fence();
  }
  if (correction != nullptr) wave_lds_fence();
  // The largest score `top` times; a chosen one is marked with -inf.
  float chosen_sum = 0.f;
  float my_w = 0.f;
  int my_e = 0;
  for (int k = 0; k < top; ++k) {
    float best;
    const int best_e = wave_argmax(z, E, lane, best);
    const float score = correction != nullptr ? raw[best_e] : best / sum;
    chosen_sum = chosen_sum + score;
    if (lane == k % 64 && k < 64) { my_w = score; my_e = best_e; }
    if (k >= 64 && lane == 0) { idx[(int64_t)t * top + k] = best_e; wts[(int64_t)t * top + k] = score; }
    if (lane == 0) z[best_e] = -INFINITY;
    wave_lds_fence();
  }
  const float denom = score_kind == 0 ? chosen_sum + weight_eps : 1.f;
  if (lane < top) {
    idx[(int64_t)t * top + lane] = my_e;
    wts[(int64_t)t * top + lane] = (my_w / denom) * scale;
  }
  for (int k = 64 + lane; k < top; k += 64) wts[(int64_t)t * top + k] = (wts[(int64_t)t * top + k] / denom) * scale;
}

__global__ __launch_bounds__(256) void moe_choose_kernel(MoeChoice a) {
  extern __shared__ float scores[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int t = blockIdx.x * 4 + wave;
  if (t < a.T) moe_choose_token(a, scores, t, wave, 4, lane);
}

// The plan, by one workgroup.  counts the pairs of every expert, gives expert e the rows [start_e, start_e + tile_rows *
// ceil(count_e / tile_rows)) and every pair a row among its expert's (in no fixed order: a row's result does not depend on
// its place).  row_pair [max_rows]: the pair (token * top + choice) of a row, or -1; row_token [max_rows]: the row's
// token (0 for a row without a pair); pair_row [pairs]; tile_expert [max_tiles]: the expert of a tile, or -1 beyond the
// last; expert_start [E + 1]: the first row of every expert, and the rows in use.
// order [E] or null (vk_gemm_experts): {parts before, first row, rows, expert}, an expert's rows in ceil(rows / EXPERT_PART_ROWS) parts; experts without
// rows come last.  Up to 64 experts: the ones of taller parts first, so that a launch's last workgroups are its shortest.
struct MoePlanArgs {
  const int32_t* idx;
  int32_t *row_pair, *row_token, *pair_row, *tile_expert, *expert_start;
  int pairs, top, E, max_tiles, tile_rows;
  int4* order;
};
// By all threads of a workgroup of 1,024; plan: LDS, [E] counts, then [E] cursors.
__device__ __forceinline__ void moe_make_plan(const MoePlanArgs& a, int32_t* plan) {
  int32_t* count = plan;
  int32_t* cursor = plan + a.E;
  for (int e = threadIdx.x; e < a.E; e += blockDim.x) count[e] = 0;
  for (int r = threadIdx.x; r < a.max_tiles * a.tile_rows; r += blockDim.x) {
    a.row_pair[r] = -1;
    a.row_token[r] = 0;
  }
  for (int i = threadIdx.x; i < a.max_tiles; i += blockDim.x) a.tile_expert[i] = -1;
  __syncthreads();
  for (int i = threadIdx.x; i < a.pairs; i += blockDim.x) atomicAdd(&count[a.idx[i]], 1);
  __syncthreads();
  if (a.E <= 64) {
    // One wave, an expert a lane: the tiles before an expert's are a running sum over the lanes.
    if (threadIdx.x < 64) {
      const int e = threadIdx.x;
      const int n = e < a.E ? (count[e] + a.tile_rows - 1) / a.tile_rows : 0;
      int upto = n;
#pragma unroll
      for (int off = 1; off < 64; off <<= 1) {
        const int other = __shfl_up(upto, off, VK_WAVE);
        if (e >= off) upto += other;
      }
      const int tile = upto - n;
      if (e < a.E) {
        cursor[e] = tile * a.tile_rows;
        a.expert_start[e] = tile * a.tile_rows;
        for (int j = 0; j < n; ++j) a.tile_expert[tile + j] = e;
        if (e == a.E - 1) a.expert_start[a.E] = upto * a.tile_rows;
      }
      if (a.order != nullptr) {
        const int rows = e < a.E ? count[e] : 0, parts = (rows + EXPERT_PART_ROWS - 1) / EXPERT_PART_ROWS;
        const int key = (rows > 0 ? (rows + parts - 1) / parts : 0) * 64 + 63 - e;       // different for every lane
        int rank = 0, before = 0;
#pragma unroll
        for (int i = 0; i < 64; ++i) {
          const bool ahead = __builtin_amdgcn_readlane(key, i) > key;
          rank += ahead ? 1 : 0;
          before += ahead ? __builtin_amdgcn_readlane(parts, i) : 0;
        }
        if (rank < a.E) a.order[rank] = int4{before, tile * a.tile_rows, rows, e < a.E ? e : 0};
      }
    }
  } else if (threadIdx.x == 0) {
    int tile = 0, parts = 0, busy = 0;
    for (int e = 0; e < a.E; ++e) {
      const int n = (count[e] + a.tile_rows - 1) / a.tile_rows;
      cursor[e] = tile * a.tile_rows;
      a.expert_start[e] = tile * a.tile_rows;
      for (int j = 0; j < n; ++j) a.tile_expert[tile + j] = e;
      if (a.order != nullptr && n > 0) {
        a.order[busy++] = int4{parts, tile * a.tile_rows, count[e], e};
        parts += (count[e] + EXPERT_PART_ROWS - 1) / EXPERT_PART_ROWS;
      }
      tile += n;
    }
    if (a.order != nullptr)
      for (; busy < a.E; ++busy) a.order[busy] = int4{parts, 0, 0, 0};
    a.expert_start[a.E] = tile * a.tile_rows;
  }
  __syncthreads();
  for (int i = threadIdx.x; i < a.pairs; i += blockDim.x) {
    const int row = atomicAdd(&cursor[a.idx[i]], 1);
    a.row_pair[row] = i;
    a.row_token[row] = i / a.top;
    a.pair_row[i] = row;
  }
}
__global__ __launch_bounds__(1024) void moe_plan_kernel(MoePlanArgs a) {
  extern __shared__ int32_t plan[];
  moe_make_plan(a, plan);
}

// The choice and the plan of a few tokens in one launch, a wave a token: two launches that wait for each other took 11 to 15 us for some
// hundred numbers.  The waves share one compute unit, where a choice is a chain of searches: router and plan of 64 experts in one launch
// against two, us: one choice, 16 tokens 8.5, 9.1; four, 12 tokens 10.1, 10.8, 16 11.0, 10.8; eight, 12 tokens 12.9, 13.0, 16 14.2, 13.0; beyond 16,
// with a second token a wave, 24 tokens of four 12.9, 10.8, 32 of eight 21.5, 13.0.
#define MOE_FEW_TOKENS(top) ((top) <= 4 ? 16 : 12)
__global__ __launch_bounds__(1024) void moe_choose_plan_kernel(MoeChoice c, MoePlanArgs p) {
  extern __shared__ float scores[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (wave < c.T) moe_choose_token(c, scores, wave, wave, 16, lane);
  __syncthreads();                // every choice is made and, through this compute unit's cache, to be read by all its waves
  moe_make_plan(p, reinterpret_cast<int32_t*>(scores));
}

// One tile of 16 rows and 16 output features a workgroup: out[row, f] = sum over k of x[row, k] * w[expert][f, k], in
// the order of this library's other products: the reduction axis in chunks of MOE_KC elements, a chunk's products added
// from zero over ascending slabs of 64 bytes with the weights as first operand, the chunk sums added to a zero total in
// chunk order.  The workgroup's eight waves take chunks wave, wave + 8, ... with MOE_W slabs in flight each, and the
// chunk sums meet in LDS.  UP: the rows' inputs are the tokens' (row_token) and the output is the square of max(., 0) of
// the sum rounded to the element type, as elements; else the inputs are the rows themselves and the output the sum, as
// elements.
#define MOE_KC KC
#define MOE_KC_SLABS (MOE_KC / VK_SLAB)
#define MOE_WAVES 8
#define MOE_W 4
// MODE 0: the rows themselves are the inputs (down); 1: the rows' tokens, with the squared-relu activation; 2: the rows'
// tokens, the sum as it is (an activation of two products' outputs follows in a launch of its own).
template <int MODE>
__global__ __launch_bounds__(64 * MOE_WAVES) void moe_gemm_kernel(elem_t* __restrict__ out, int64_t ldo, const elem_t* __restrict__ x, int64_t ldx,
                                                                  const elem_t* __restrict__ w, int64_t expert_stride,
                                                                  const int32_t* __restrict__ row_pair, const int32_t* __restrict__ row_token,
                                                                  const int32_t* __restrict__ tile_expert, int N, int K) {
  __shared__ f32x4 part[MOE_WAVES][64];
  const int tile = blockIdx.y;
  const int e = tile_expert[tile];
  if (e < 0) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, kq = lane >> 4;
  const int f0 = blockIdx.x * 16;
  const int row = tile * MOE_TILE + r16;
  const bool x_ok = row_pair[row] >= 0;
  constexpr bool UP = MODE != 0;
  const elem_t* xr = x + (int64_t)(UP ? row_token[row] : row) * ldx + kq * VK_VEC;
  const bool w_ok = f0 + r16 < N;
  const elem_t* wr = w + (int64_t)e * expert_stride + (int64_t)(w_ok ? f0 + r16 : 0) * K + kq * VK_VEC;
  const int nchunks = (K + MOE_KC - 1) / MOE_KC;
  const int rounds = (nchunks + MOE_WAVES - 1) / MOE_WAVES;

  frag_t wbuf[MOE_W], xbuf[MOE_W];
  auto issue = [&](int c, int s, int slot) {
    const int k = c * MOE_KC + s * VK_SLAB;
    const bool k_ok = k + kq * VK_VEC < K;
    wbuf[slot] = load_frag(wr + k, w_ok && k_ok);
    xbuf[slot] = load_frag(xr + k, x_ok && k_ok);
  };
  int c = wave;
  if (c < nchunks) {
#pragma unroll
    for (int i = 0; i < MOE_W; ++i) issue(c, i, i);
  }
  f32x4 total = {0.f, 0.f, 0.f, 0.f};
  for (int round = 0; round < rounds; ++round, c += MOE_WAVES) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    if (c < nchunks) {
      const int cn = c + MOE_WAVES;
      const bool has_next = cn < nchunks;
#pragma unroll
      for (int i = 0; i < MOE_KC_SLABS; ++i) {
        const int slot = i % MOE_W;
        const frag_t fw = wbuf[slot], fx = xbuf[slot];
        if (i + MOE_W < MOE_KC_SLABS) issue(c, i + MOE_W, slot);
        else if (has_next) issue(cn, i + MOE_W - MOE_KC_SLABS, slot);
        acc = mma_slab(fw, fx, acc);
      }
    }
    part[wave][lane] = acc;
    __syncthreads();
    if (wave == 0) {
      for (int w2 = 0; w2 < MOE_WAVES; ++w2) {
        if (round * MOE_WAVES + w2 < nchunks) {
          const f32x4 p = part[w2][lane];
          total.x = total.x + p.x; total.y = total.y + p.y; total.z = total.z + p.z; total.w = total.w + p.w;
        }
      }
    }
    __syncthreads();
  }
  // Lane l holds features f0 + 4 * (l / 16) + i for row l % 16.
  if (wave != 0 || !x_ok) return;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int f = f0 + kq * 4 + i;
    if (f >= N) continue;
    float v = total[i];
    if (MODE == 1) {
      const float rl = fmaxf(round_to_elem(v), 0.f);
      v = rl * rl;
    }
    out[(int64_t)row * ldo + f] = from_f32<elem_t>(v);
  }
}

// The same products (16-bit elements, K in whole slabs, up to MOE_LINE_CHUNKS chunks), built to keep memory busy where the kernel above
// is bound by its workgroups' starts: 64 to 128 KB of weights each behind three dependent loads, and idle waves where K has fewer than
// eight chunks.  Workgroups of a wave a chunk stay for the whole launch and take equal, contiguous shares of the (row tile, MOE_LINE_ROWS
// features) units of all tiles in use, tile by tile; a wave keeps its chunk of the tile's rows in registers; the weights come as in
// gemm_lines_kernel, a row of a chunk a load, marked as read once, into a slot a wave, or two of seven to nine chunks: what LDS has for about twelve waves a
// compute unit, which cover each other's way to memory (slots of four rows, two or three a wave, were 4 to 12 % slower); one barrier a unit, and the waves take
// turns at adding up a unit's chunk sums.  Rows without a pair are not read and not stored, features beyond N are clamped.
// What bounds it: a launch's start (expert_start, a tile's expert, its rows) where units are few, else how fast memory gives lines: 6.2 to 6.6 TB/s.
// Measured on MI355X, 32 experts, eight tokens of 4 choices, against the same stream in the operands' order straight to registers: 1,536 x
// 2,048 weights, 21 experts 28.1 -> 24.8 us, 2,048 x 1,536 31.6 -> 27.1, 3,072 x 2,048, 18 experts 48.1 -> 39.2; five chunks and more: 4,096 x 4,608, 21
// experts 147 -> 120; against the kernel above 3,072 x 4,096, 18 experts 83.9 -> 72.6, 4,608 x 4,096, 19 124 -> 110.
// WHOLE: K in whole chunks; else the pieces that the last chunk has not are its last one again, and the products are left out (a
// product with zeros would make a NaN of an infinite weight).
#ifdef VK_BF16
#define MOE_LINE_ROWS 8
#define MOE_LINE_CHUNKS 16
template <int MODE, bool WHOLE>
__global__ __launch_bounds__(64 * MOE_LINE_CHUNKS) void moe_lines_kernel(elem_t* __restrict__ out, int64_t ldo, const elem_t* __restrict__ x, int64_t ldx,
                                                                           const elem_t* __restrict__ w, int64_t expert_stride,
                                                                           const int32_t* __restrict__ row_pair, const int32_t* __restrict__ row_token,
                                                                           const int32_t* __restrict__ tile_expert, const int32_t* __restrict__ expert_start,
                                                                           int E, int N, int K, int vec, int slots) {
  constexpr int SL = MOE_KC_SLABS, R = MOE_LINE_ROWS, SLOT = R * 1024, SUMS = R / 4 * 16;
  using W = LineRows<R>;
  extern __shared__ __attribute__((aligned(16))) unsigned char lines_lds[];      // slots a wave, then the sums [2][waves][SUMS]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = blockDim.x >> 6;
  const int r16 = lane & 15, kq = lane >> 4;
  const int features = (N + R - 1) / R;
  const int64_t units = (int64_t)(expert_start[E] / MOE_TILE) * features;
  const int lo = (int)(units * blockIdx.x / gridDim.x), hi = (int)(units * (blockIdx.x + 1) / gridDim.x);
  if (lo >= hi) return;                           // the whole workgroup
  const int have = WHOLE ? SL : min(SL, (K - wave * MOE_KC) / VK_SLAB);      // slabs of this wave's chunk
  unsigned char* own = lines_lds + wave * slots * SLOT;
  f32x4* part = reinterpret_cast<f32x4*>(lines_lds + waves * slots * SLOT);
  // The units whose weights are asked for, ahead of those that are multiplied.
  int ask_u = lo, ask_tile = lo / features, ask_f = lo - ask_tile * features;
  const elem_t* expert = w + (int64_t)tile_expert[ask_tile] * expert_stride + wave * MOE_KC;
  auto ask = [&](int s) {
    W::template ask<true>(expert + (int64_t)ask_f * R * K, K, N - ask_f * R, lane, lds_offset_of(own + s * SLOT), WHOLE ? 64 : have * 4);
    ++ask_u;
    if (++ask_f == features) {
      ask_f = 0;
      ++ask_tile;
      if (ask_u < hi) expert = w + (int64_t)tile_expert[ask_tile] * expert_stride + wave * MOE_KC;
    }
  };
  frag_t rows[SL];
  bool live = false;                              // the lane's row has a pair
  auto bring = [&](int tile) {
    live = row_pair[tile * MOE_TILE + r16] >= 0;
    // The rows with a pair come first; where rows lie one after another, the last of them instead of those without (gathered, those are one token).
    const int row = tile * MOE_TILE + (MODE != 0 ? r16 : min(r16, max(__popcll(__ballot(live) & 0xFFFFu) - 1, 0)));
    const elem_t* xr = x + (int64_t)(MODE != 0 ? row_token[row] : row) * ldx + wave * MOE_KC + kq * VK_VEC;
#pragma unroll
    for (int i = 0; i < SL; ++i) rows[i] = *reinterpret_cast<const frag_t*>(xr + (WHOLE ? i : min(i, have - 1)) * VK_SLAB);
  };
  int tile = ask_tile, f = ask_f;
  for (int s = 0; s < slots; ++s)
    if (ask_u < hi) ask(s);
  bring(tile);
  int s = 0;
  for (int u = lo; u < hi; ++u) {
    // All but the slots asked for after this one's (and a store or a tile's rows, which are waited for by count as well: never too short a wait).
    const int later = ask_u - u - 1;
    __builtin_amdgcn_sched_barrier(0);
    if (later > 0) wait_vmcnt_n<R>();               // a ring has two slots at most
    else wait_vmcnt_n<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < SL; ++i)
      if (WHOLE || i < have) acc = mma_slab(W::fragment(own + s * SLOT, i, r16, kq), rows[i], acc);
    f32x4* sums = part + ((u - lo) & 1) * waves * SUMS;
    if (lane < SUMS) sums[wave * SUMS + lane] = acc;
    __builtin_amdgcn_s_waitcnt(0xC07F);           // lgkmcnt(0): the slot has been read, the sums are written
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    if (ask_u < hi) ask(s);
    s = s + 1 == slots ? 0 : s + 1;
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (wave == u % waves && lane < SUMS) {
      f32x4 total = {0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < waves; ++c) {
        const f32x4 p = sums[c * SUMS + lane];
        total.x = total.x + p.x; total.y = total.y + p.y; total.z = total.z + p.z; total.w = total.w + p.w;
      }
      if (MODE == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float rl = fmaxf(round_to_elem(total[i]), 0.f);
          total[i] = rl * rl;
        }
      }
      const int row = tile * MOE_TILE + r16, first = f * R + kq * 4;
      if (live) {
        elem_t* o = out + (int64_t)row * ldo + first;
        if (vec && first + 3 < N) {
          store_elems4(o, total);
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (first + i < N) o[i] = from_f32<elem_t>(total[i]);
        }
      }
    }
    if (++f == features) {
      f = 0;
      ++tile;
      if (u + 1 < hi) bring(tile);
    }
  }
}
// The same for one and two whole chunks and units between few and many, a unit of 16 features a workgroup, a wave a chunk, all of it asked for at once in the operands' order
// straight to registers.  What bounds it is the way to its first bytes, which here is a tile's expert and the weights behind it, with no way through LDS; and units
// of 16 features read the tile's rows half as often as those of eight.  No load is predicated.
// moe_product_kernel has both sides measured.
template <int MODE, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void moe_unit_kernel(elem_t* __restrict__ out, int64_t ldo, const elem_t* __restrict__ x, int64_t ldx,
                                                              const elem_t* __restrict__ w, int64_t expert_stride, const int32_t* __restrict__ row_pair,
                                                              const int32_t* __restrict__ row_token, const int32_t* __restrict__ tile_expert, int N, int K, int vec) {
  __shared__ f32x4 part[WAVES][64];
  const int tile = blockIdx.y, e = tile_expert[tile];
  if (e < 0) return;                              // the whole workgroup
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, kq = lane >> 4;
  const int row = tile * MOE_TILE + r16, first = blockIdx.x * 16 + kq * 4;
  const bool live = row_pair[row] >= 0;           // the lane's row has a pair
  const int64_t k0 = (int64_t)wave * MOE_KC + kq * VK_VEC;
  const elem_t* wr = w + (int64_t)e * expert_stride + (int64_t)min((int)blockIdx.x * 16 + r16, N - 1) * K + k0;
  frag_t weights[MOE_KC_SLABS], rows[MOE_KC_SLABS];
#pragma unroll
  for (int i = 0; i < MOE_KC_SLABS; ++i) weights[i] = *reinterpret_cast<const frag_t*>(wr + i * VK_SLAB);
  // As in the kernel above: instead of rows without a pair the last one with one, or, gathered, the token that the plan names there.
  const int from = MODE != 0 ? row_token[row] : tile * MOE_TILE + min(r16, max(__popcll(__ballot(live) & 0xFFFFu) - 1, 0));
  const elem_t* xr = x + (int64_t)from * ldx + k0;
#pragma unroll
  for (int i = 0; i < MOE_KC_SLABS; ++i) rows[i] = *reinterpret_cast<const frag_t*>(xr + i * VK_SLAB);
  f32x4 acc = {0.f, 0.f, 0.f, 0.f}, total = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < MOE_KC_SLABS; ++i) acc = mma_slab(weights[i], rows[i], acc);
  if constexpr (WAVES > 1) {
    part[wave][lane] = acc;
    __syncthreads();
    if (wave != 0) return;
  }
#pragma unroll
  for (int c = 0; c < WAVES; ++c) {
    const f32x4 p = WAVES > 1 ? part[c][lane] : acc;
    total.x = total.x + p.x; total.y = total.y + p.y; total.z = total.z + p.z; total.w = total.w + p.w;
  }
  if (MODE == 1) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float rl = fmaxf(round_to_elem(total[i]), 0.f);
      total[i] = rl * rl;
    }
  }
  if (!live) return;
  elem_t* o = out + (int64_t)row * ldo + first;
  if (vec && first + 3 < N) {
    store_elems4(o, total);
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (first + i < N) o[i] = from_f32<elem_t>(total[i]);
  }
}
#endif

// x <- max(x, 0)^2, element by element: the experts' activation on a product that was left as elements.  A thread
// takes a 16-byte vector (n in whole vectors).
__global__ __launch_bounds__(256) void moe_relu_square_kernel(elem_t* x, int64_t nvec) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nvec) return;
  float v[VK_VEC];
  load_elems(x + i * VK_VEC, v);
#pragma unroll
  for (int j = 0; j < VK_VEC; ++j) {
    const float rl = fmaxf(v[j], 0.f);
    v[j] = rl * rl;
  }
  store_elems(x + i * VK_VEC, v);
}

// A gated expert's activation between its two products: row r of `in` holds the gate's F outputs and, from column F on,
// the up projection's; y = g * sigmoid(slope * g) * (u + shift) with g = min(gate, limit) and u = clamp(up, -limit, limit),
// in 32-bit, as elements [rows, F].  A thread takes a 16-byte vector (F in whole vectors).
// row_pair / wts (both or neither): row r's gate and up values are multiplied by the weight of the row's (token, choice) pair
// before they are clamped, which is what an expert computes that reads its input times that weight; a row without a pair
// gives zeros.
__global__ __launch_bounds__(256) void moe_glu_kernel(elem_t* __restrict__ out, const elem_t* __restrict__ in, int64_t rows, int F, float limit,
                                                      float slope, float shift, const int32_t* __restrict__ row_pair, const float* __restrict__ wts) {
  const int per = F / VK_VEC;
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= rows * per) return;
  const int64_t r = i / per;
  const int c = (int)(i - r * per) * VK_VEC;
  float g[VK_VEC], u[VK_VEC];
  float rw = 1.f;
  if (row_pair != nullptr) {
    const int pair = row_pair[r];
    if (pair < 0) {
#pragma unroll
      for (int j = 0; j < VK_VEC; ++j) g[j] = 0.f;
      store_elems(out + r * F + c, g);
      return;
    }
    rw = wts[pair];
  }
  load_elems(in + r * 2 * F + c, g);
  load_elems(in + r * 2 * F + F + c, u);
#pragma unroll
  for (int j = 0; j < VK_VEC; ++j) {
    const float gc = fminf(g[j] * rw, limit), uc = fminf(fmaxf(u[j] * rw, -limit), limit);
    g[j] = (gc / (1.f + expf(-slope * gc))) * (uc + shift);
  }
  store_elems(out + r * F + c, g);
}

// out[t, c] = sum over k < top, ascending, of wts[t, k] * y[pair_row[t * top + k], c] (wts null: every weight 1), from zero; then + extra[t, c]
// (elements, the output of an expert that every token uses) where there is one.
__global__ __launch_bounds__(256) void moe_combine_kernel(float* __restrict__ out, const elem_t* __restrict__ y, const float* __restrict__ wts,
                                                          const int32_t* __restrict__ pair_row, int W, int top, const elem_t* __restrict__ extra) {
  const int t = blockIdx.x;
  for (int c = blockIdx.y * 256 + threadIdx.x; c < W; c += gridDim.y * 256) {
    float acc = 0.f;
    for (int k = 0; k < top; ++k)
      acc = acc + (wts != nullptr ? wts[(int64_t)t * top + k] : 1.f) * to_f32(y[(int64_t)pair_row[(int64_t)t * top + k] * W + c]);
    if (extra != nullptr) acc = acc + to_f32(extra[(int64_t)t * W + c]);
    out[(int64_t)t * W + c] = acc;
  }
}

// The same for rows of whole 16-byte vectors at 16-byte addresses, a vector a thread.
__global__ __launch_bounds__(256) void moe_combine_vec_kernel(float* __restrict__ out, const elem_t* __restrict__ y, const float* __restrict__ wts,
                                                              const int32_t* __restrict__ pair_row, int W, int top, const elem_t* __restrict__ extra) {
  const int t = blockIdx.x, c = (blockIdx.y * 256 + threadIdx.x) * VK_VEC;
  if (c >= W) return;
  float acc[VK_VEC];
#pragma unroll
  for (int j = 0; j < VK_VEC; ++j) acc[j] = 0.f;
#pragma unroll 4
  for (int k = 0; k < top; ++k) {
    float v[VK_VEC];
    load_elems(y + (int64_t)pair_row[(int64_t)t * top + k] * W + c, v);
    const float w = wts != nullptr ? wts[(int64_t)t * top + k] : 1.f;
#pragma unroll
    for (int j = 0; j < VK_VEC; ++j) acc[j] = acc[j] + w * v[j];
  }
  if (extra != nullptr) {
    float v[VK_VEC];
    load_elems(extra + (int64_t)t * W + c, v);
#pragma unroll
    for (int j = 0; j < VK_VEC; ++j) acc[j] = acc[j] + v[j];
  }
#pragma unroll
  for (int j = 0; j < VK_VEC; j += 4)
    *reinterpret_cast<f32x4*>(out + (int64_t)t * W + c + j) = f32x4{acc[j], acc[j + 1], acc[j + 2], acc[j + 3]};
}

extern "C" {

// Tiles that the plan may need for T tokens: every pair, and up to tile_rows - 1 rows of padding an expert that got any.
int vk_moe_max_tiles(int T, int top, int E, int tile_rows) {
  const int64_t pairs = (int64_t)T * top;
  const int64_t busy = std::min<int64_t>(E, pairs);
  return (int)((pairs + busy * (tile_rows - 1)) / tile_rows);
}

// logits: scratch [T, E] floats.  bias [E] (elements, or floats with bias_is_f32) or null.
static int route_launch(int32_t* idx, float* wts, float* logits, const elem_t* h, const elem_t* router, const void* bias, int bias_is_f32, int T, int W,
                        int E, int top, float weight_eps, hipStream_t st, int score_kind, int groups, int keep, float scale, int group_score, const void* correction,
                        int correction_is_f32, const MoePlanArgs& plan) {
  VK_REQUIRE(T >= 0 && W > 0 && W % VK_VEC == 0 && E > 0 && top > 0 && top <= E && E <= 4096,
             "router: bad sizes T=%d W=%d E=%d top=%d (the width in whole 16-byte vectors, at most 4096 experts)", T, W, E, top);
  VK_REQUIRE(((uintptr_t)h % 16) == 0 && ((uintptr_t)router % 16) == 0, "router: operands must be 16-byte aligned");
  VK_REQUIRE(groups > 0 && E % groups == 0 && keep > 0 && keep <= groups && top <= keep * (E / groups),
             "router: %d experts in %d groups of which %d are kept cannot give %d choices", E, groups, keep, top);
  if (T == 0) return 0;
  // Workgroup i runs on chip part i % 8: with a multiple of eight token groups a group meets every expert on the same part,
  // whose cache then holds its rows.
  const int groups_of_tokens = (T + MOE_ROUTE_TOKENS - 1) / MOE_ROUTE_TOKENS;
  const int grid_x = groups_of_tokens > 8 ? (groups_of_tokens + 7) / 8 * 8 : groups_of_tokens;
  // Four experts a workgroup from eight workgroups a compute unit on, with one each: that is where a group's rows, read again, become the longer
  // wait (one against four, with choice and plan: 256 tokens of 4,096 entries, 8 experts 10.7, 13.5 us; 32 experts, 255 and 256 tokens of
  // 4,096 11.5, 13.9, 512 15.0, 14.8; 64 experts, 256 tokens of 2,048 11.7, 12.3, 2,048 of them 46, 28).
  if (E % 4 == 0 && (int64_t)groups_of_tokens * E >= 8 * (int64_t)vk_device_cus()) moe_logits_kernel<4><<<dim3(grid_x, E / 4), 256, 0, st>>>(logits, h, router, T, W, E, bias, bias_is_f32);
  else moe_logits_kernel<1><<<dim3(grid_x, E), 256, 0, st>>>(logits, h, router, T, W, E, bias, bias_is_f32);
  if (vk_check_launch("router (logits)")) return 1;
  const MoeChoice c = {idx, wts, logits, T, E, top, weight_eps, score_kind, groups, keep, scale, group_score, correction, correction_is_f32};
  const size_t a_wave = ((correction != nullptr ? 2 : 1) * (size_t)E + (keep < groups ? groups : 0)) * sizeof(float);
  VK_REQUIRE(4 * a_wave <= 65536, "router: %d experts in %d groups are too many", E, groups);
  if (T <= MOE_FEW_TOKENS(top) && 16 * a_wave <= 65536) {
    moe_choose_plan_kernel<<<1, 1024, std::max(16 * a_wave, (size_t)2 * E * sizeof(int32_t)), st>>>(c, plan);
    return vk_check_launch("router (choice and plan)");
  }
  moe_choose_kernel<<<(T + 3) / 4, 256, 4 * a_wave, st>>>(c);
  if (vk_check_launch("router (choice)")) return 1;
  moe_plan_kernel<<<1, 1024, (size_t)2 * E * sizeof(int32_t), st>>>(plan);
  return vk_check_launch("expert plan");
}

// The router and the plan.  bias: an expert's number on its logit, which both the choice and the weights see, or null.  score_kind 0: the
// softmax over all experts, a chosen one's divided by the sum of the chosen plus weight_eps (with weight_eps 0 the softmax over the
// chosen logits alone, whatever the others are); 1: the logistic function of a chosen logit as it is; 2: the softmax over all experts as it
// is.  groups, keep: only experts of the `keep` best of that many equal groups can be chosen (1, 1: all); group_score 0: a group is worth
// its largest score, 1: the sum of its two largest.  correction (score 1, no bias; [E] elements or floats): joins the scores for the choice
// of groups and experts and not for the weights.  scale: on every weight.  tile_rows: rows of a tile of the plan (moe_plan_kernel).  order: [E][4], 16-byte aligned, or null.
int vk_moe_route_plan_ordered(int32_t* idx, float* wts, float* logits, const elem_t* h, const elem_t* router, const void* bias, int bias_is_f32,
                              const void* correction, int correction_is_f32, int T, int W, int E, int top, float weight_eps, int score_kind, int groups, int keep,
                              int group_score, float scale, int32_t* row_pair, int32_t* row_token, int32_t* pair_row, int32_t* tile_expert, int32_t* expert_start,
                              int tile_rows, int32_t* order, hipStream_t st) {
  VK_REQUIRE(score_kind >= 0 && score_kind <= 2 && (group_score == 0 || group_score == 1), "router: score kind %d, group score %d", score_kind, group_score);
  VK_REQUIRE(correction == nullptr || (bias == nullptr && score_kind == 1), "router: a correction goes with logistic scores and without a bias");
  VK_REQUIRE(T >= 0 && top > 0 && E > 0 && E <= 4096 && tile_rows > 0, "expert plan: bad sizes T=%d top=%d E=%d", T, top, E);
  VK_REQUIRE((uintptr_t)order % 16 == 0, "expert plan: the order must be 16-byte aligned");
  if (T == 0) return 0;
  const MoePlanArgs plan = {idx, row_pair, row_token, pair_row, tile_expert, expert_start, T * top, top, E, vk_moe_max_tiles(T, top, E, tile_rows), tile_rows, (int4*)order};
  return route_launch(idx, wts, logits, h, router, bias, bias_is_f32, T, W, E, top, weight_eps, st, score_kind, groups, keep, scale, group_score, correction,
                      correction_is_f32, plan);
}

int vk_moe_route_plan(int32_t* idx, float* wts, float* logits, const elem_t* h, const elem_t* router, const void* bias, int bias_is_f32,
                      const void* correction, int correction_is_f32, int T, int W, int E, int top, float weight_eps, int score_kind, int groups, int keep,
                      int group_score, float scale, int32_t* row_pair, int32_t* row_token, int32_t* pair_row, int32_t* tile_expert, int32_t* expert_start,
                      int tile_rows, hipStream_t st) {
  return vk_moe_route_plan_ordered(idx, wts, logits, h, router, bias, bias_is_f32, correction, correction_is_f32, T, W, E, top, weight_eps, score_kind, groups, keep,
                                   group_score, scale, row_pair, row_token, pair_row, tile_expert, expert_start, tile_rows, nullptr, st);
}

// An expert product of rows in tiles of 16: by the kernels for whole slabs where they take the sizes, else by the one for every K.
extern "C++" {
#ifdef VK_BF16
// Which kernel is the fastest one, by the (row tile, 16 features) units of all tiles that a launch covers.  The kernel of whole lines has a long start (the
// tiles in use, a tile's expert, its rows, a barrier a unit) and reads a tile's rows twice as often; the one for every K has eight waves whatever K.
// Measured on MI355X in recorded launches, 8 to 64 experts, 2 to 6 choices, 1 to 64 tokens; the lines lie where weights come from memory (512 MB of layers in turn).
// One and two whole chunks, a unit a workgroup over whole lines, by units: up to the compute units 0.94 to 1.18 (512 x 1,024, one token 4.7, 4.0 us), from there to 600 0.88 to 1.05, up to 1,400
// 0.74 to 0.99, then one chunk up to 4,096 0.81 to 1.02 and two up to 2,048 0.94 to 1.05, more 0.98 to 1.28.  Where the weights are in the caches (twelve layers of few experts) a unit a
// workgroup is ahead by 10 % more; the stream of such units that stayed was behind the better one by 5 to 30 % from 600 units on.
// More chunks, the kernel for every K against whole lines, us, the units in brackets.  Where units are at most half of the compute units the latter are ahead (512 x 1,536, one
// token (64) 5.3, 4.4; 512 x 2,048 (128) 5.9, 5.1; 512 x 2,560 (128) 6.2, 5.5; 256 x 3,584 (64) 7.0, 5.4; 512 x 4,096 (128) 7.5, 6.7); then
//   three: 512 x 1,536 (640) 10.7, 10.5; 1,024 x 1,536 (768) 13.5, 11.1; 2,048 x 1,536, two tokens (768) 14.0, 11.1;
//   four: 1,536 x 2,048, two tokens (576) 9.7, 10.7; 512 x 2,048 (640) 8.6, 10.1; 1,536 x 2,048 (768) 15.9, 12.2, 3,072 x 2,048, three tokens (2,304) 35.3, 28.5;
//   five: always (1,000 x 2,560 (189) 7.4, 7.2; 512 x 2,560 (480) 11.5, 10.9; 1,536 x 2,560 (576) 17.2, 13.1; in the caches 10 to 18 % the other way from 192 to 480 units);
//   six: 768 x 3,072 (288) 12.0, 11.0, 1,536 x 3,072 (384) 12.0, 11.0; seven: 1,024 x 3,584 (576) 16.2, 14.4;
//   eight: 256 x 4,096 (288) 9.9, 10.5, 384 x 4,096 (408) 16.8, 14.3; 3,072 x 4,096, eight tokens 83.9, 72.6, 24 150, 122; 6,144 x 4,096, 24 292, 239;
//   nine and more: the other kernel needs a second round: 512 x 4,608 (128) 9.7, 7.2, (576) 20.8, 16.8; at 192 to 256 units as fast, within 10 % either way;
//   a reduction that ends inside a chunk: 1,024 x 768, two (512) 6.0, 6.6, 4,096 x 768, eight 110, 55; 1,024 x 1,152, three (768) 10.0, 10.3, eight
//   28.9, 19.8; 2,048 x 2,304, one (512) 10.8, 10.9, eight 73, 53.
enum { MOE_TILES, MOE_LINES, MOE_UNITS };
static int moe_product_kernel(int chunks, bool whole, bool gathered, int64_t units) {
  if (chunks > MOE_LINE_CHUNKS) return MOE_TILES;
  if (!whole) return units >= (chunks == 1 ? (gathered ? 768 : 2304) : (chunks == 3 || chunks == 4 ? 780 : 540)) ? MOE_LINES : MOE_TILES;
  if (chunks <= 2) return units > vk_device_cus() && units < (chunks == 1 ? 4096 : 2048) ? MOE_UNITS : MOE_LINES;
  constexpr int LINES_FROM[9] = {0, 0, 0, 660, 750, 1, 260, 260, 300};
  return chunks > 8 || units >= LINES_FROM[chunks] || 2 * units <= vk_device_cus() ? MOE_LINES : MOE_TILES;
}
#endif
template <int MODE>
static int moe_product(elem_t* out, int64_t ldo, const elem_t* x, int64_t ldx, const elem_t* w, const int32_t* row_pair, const int32_t* row_token,
                       const int32_t* tile_expert, const int32_t* expert_start, int tiles, int E, int N, int K, hipStream_t st, const char* what) {
#ifdef VK_BF16
  const int chunks = (K + MOE_KC - 1) / MOE_KC, vec = ldo % 4 == 0 && (uintptr_t)out % 8 == 0;
  const int64_t units = (int64_t)tiles * ((N + 15) / 16);
  const int kernel = K % VK_SLAB == 0 && ldx % VK_VEC == 0 ? moe_product_kernel(chunks, K % MOE_KC == 0, MODE != 0, units) : MOE_TILES;
  if (kernel == MOE_UNITS) {
    const dim3 grid((N + 15) / 16, tiles);
    if (chunks == 1) moe_unit_kernel<MODE, 1><<<grid, 64, 0, st>>>(out, ldo, x, ldx, w, (int64_t)N * K, row_pair, row_token, tile_expert, N, K, vec);
    else moe_unit_kernel<MODE, 2><<<grid, 128, 0, st>>>(out, ldo, x, ldx, w, (int64_t)N * K, row_pair, row_token, tile_expert, N, K, vec);
    return vk_check_launch(what);
  }
  if (kernel == MOE_LINES) {
    // About twelve waves a compute unit, which share its LDS (measured over 544 sizes, the streams of 8, 12 and 16 waves 23.2, 22.7 and 23.0 ms, the one before them 28.8).
    static bool configured = false;
    if (!configured) {
      (void)hipFuncSetAttribute((const void*)moe_lines_kernel<MODE, true>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      (void)hipFuncSetAttribute((const void*)moe_lines_kernel<MODE, false>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
      configured = true;
    }
    const int groups = std::max(1, 12 / chunks), sums = chunks * MOE_LINE_ROWS / 4 * 16 * 2 * (int)sizeof(f32x4);
    const int slots = std::min((160 * 1024 / groups - sums) / (chunks * MOE_LINE_ROWS * 1024), 2);
    const int grid = (int)std::min<int64_t>((int64_t)tiles * ((N + MOE_LINE_ROWS - 1) / MOE_LINE_ROWS), (int64_t)vk_device_cus() * groups);
    const size_t smem = (size_t)chunks * slots * MOE_LINE_ROWS * 1024 + sums;
    if (K % MOE_KC == 0)
      moe_lines_kernel<MODE, true><<<grid, 64 * chunks, smem, st>>>(out, ldo, x, ldx, w, (int64_t)N * K, row_pair, row_token, tile_expert, expert_start, E, N, K, vec, slots);
    else
      moe_lines_kernel<MODE, false><<<grid, 64 * chunks, smem, st>>>(out, ldo, x, ldx, w, (int64_t)N * K, row_pair, row_token, tile_expert, expert_start, E, N, K, vec, slots);
    return vk_check_launch(what);
  }
#endif
  moe_gemm_kernel<MODE><<<dim3((N + 15) / 16, tiles), 64 * MOE_WAVES, 0, st>>>(out, ldo, x, ldx, w, (int64_t)N * K, row_pair, row_token, tile_expert, N, K);
  return vk_check_launch(what);
}
}  // extern "C++"

// act [max_rows, ldo] elements = relu(x[token of row] . w_up[expert of row])^2; w_up [E, N, K].
int vk_moe_up(elem_t* act, int64_t ldo, const elem_t* x, int64_t ldx, const elem_t* w_up, const int32_t* row_pair, const int32_t* row_token,
              const int32_t* tile_expert, const int32_t* expert_start, int T, int top, int E, int N, int K, hipStream_t st) {
  VK_REQUIRE(T >= 0 && top > 0 && E > 0 && N > 0 && K > 0 && K % VK_VEC == 0 && ldx % VK_VEC == 0 && ldx >= K && ldo >= N,
             "experts (up): bad sizes N=%d K=%d (K in whole 16-byte vectors)", N, K);
  VK_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)w_up % 16) == 0, "experts (up): operands must be 16-byte aligned");
  if (T == 0) return 0;
  const int tiles = vk_moe_max_tiles(T, top, E, MOE_TILE);
  VK_REQUIRE(tiles <= 65535, "experts (up): too many tiles for one launch");
  return moe_product<1>(act, ldo, x, ldx, w_up, row_pair, row_token, tile_expert, expert_start, tiles, E, N, K, st, "experts (up)");
}

// act [max_rows, ldo] elements = x[token of row] . w[expert of row], no activation; w [E, N, K].
int vk_moe_up_plain(elem_t* act, int64_t ldo, const elem_t* x, int64_t ldx, const elem_t* w, const int32_t* row_pair, const int32_t* row_token,
                    const int32_t* tile_expert, const int32_t* expert_start, int T, int top, int E, int N, int K, hipStream_t st) {
  VK_REQUIRE(T >= 0 && top > 0 && E > 0 && N > 0 && K > 0 && K % VK_VEC == 0 && ldx % VK_VEC == 0 && ldx >= K && ldo >= N,
             "experts (up): bad sizes N=%d K=%d (K in whole 16-byte vectors)", N, K);
  VK_REQUIRE(((uintptr_t)x % 16) == 0 && ((uintptr_t)w % 16) == 0, "experts (up): operands must be 16-byte aligned");
  if (T == 0) return 0;
  const int tiles = vk_moe_max_tiles(T, top, E, MOE_TILE);
  VK_REQUIRE(tiles <= 65535, "experts (up): too many tiles for one launch");
  return moe_product<2>(act, ldo, x, ldx, w, row_pair, row_token, tile_expert, expert_start, tiles, E, N, K, st, "experts (up)");
}

// out [rows, F] elements from in [rows, 2 F]: the gated activation with clamped inputs (moe_glu_kernel).
int vk_moe_glu(elem_t* out, const elem_t* in, int64_t rows, int F, float limit, float slope, float shift, hipStream_t st) {
  VK_REQUIRE(rows >= 0 && F > 0 && F % VK_VEC == 0 && limit > 0.f && ((uintptr_t)out % 16) == 0 && ((uintptr_t)in % 16) == 0,
             "experts (gated activation): bad sizes rows=%lld F=%d (whole 16-byte vectors)", (long long)rows, F);
  if (rows == 0) return 0;
  const int64_t n = rows * (F / VK_VEC);
  moe_glu_kernel<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(out, in, rows, F, limit, slope, shift, nullptr, nullptr);
  return vk_check_launch("experts (gated activation)");
}

// The same for experts that read their input times the pair's weight: row r's gate and up values are multiplied by
// wts[row_pair[r]] before the clamps (W (w h) = w (W h)); rows without a pair come out zero.
int vk_moe_glu_weighed(elem_t* out, const elem_t* in, int64_t rows, int F, float limit, float slope, float shift, const int32_t* row_pair,
                       const float* wts, hipStream_t st) {
  VK_REQUIRE(rows >= 0 && F > 0 && F % VK_VEC == 0 && limit > 0.f && ((uintptr_t)out % 16) == 0 && ((uintptr_t)in % 16) == 0,
             "experts (gated activation): bad sizes rows=%lld F=%d (whole 16-byte vectors)", (long long)rows, F);
  VK_REQUIRE(row_pair != nullptr && wts != nullptr, "experts (gated activation): the rows' pairs and weights are missing");
  if (rows == 0) return 0;
  const int64_t n = rows * (F / VK_VEC);
  moe_glu_kernel<<<(unsigned)((n + 255) / 256), 256, 0, st>>>(out, in, rows, F, limit, slope, shift, row_pair, wts);
  return vk_check_launch("experts (gated activation)");
}

// y [max_rows, N] elements = act[row] . w_down[expert of row]; w_down [E, N, K]; act rows of length lda >= K.
int vk_moe_down(elem_t* y, const elem_t* act, int64_t lda, const elem_t* w_down, const int32_t* row_pair, const int32_t* tile_expert,
                const int32_t* expert_start, int T, int top, int E, int N, int K, hipStream_t st) {
  VK_REQUIRE(T >= 0 && top > 0 && E > 0 && N > 0 && K > 0 && K % VK_VEC == 0 && lda % VK_VEC == 0 && lda >= K,
             "experts (down): bad sizes N=%d K=%d (K in whole 16-byte vectors)", N, K);
  VK_REQUIRE(((uintptr_t)act % 16) == 0 && ((uintptr_t)w_down % 16) == 0, "experts (down): operands must be 16-byte aligned");
  if (T == 0) return 0;
  const int tiles = vk_moe_max_tiles(T, top, E, MOE_TILE);
  VK_REQUIRE(tiles <= 65535, "experts (down): too many tiles for one launch");
  return moe_product<0>(y, N, act, lda, w_down, row_pair, nullptr, tile_expert, expert_start, tiles, E, N, K, st, "experts (down)");
}

int vk_moe_relu_square(elem_t* x, int64_t n, hipStream_t st) {
  VK_REQUIRE(n >= 0 && n % VK_VEC == 0 && ((uintptr_t)x % 16) == 0, "experts (activation): whole 16-byte vectors are needed");
  if (n == 0) return 0;
  const int64_t nvec = n / VK_VEC;
  moe_relu_square_kernel<<<(unsigned)((nvec + 255) / 256), 256, 0, st>>>(x, nvec);
  return vk_check_launch("experts (activation)");
}

static int combine_launch(float* out, const elem_t* y, const float* wts, const int32_t* pair_row, const elem_t* extra, int T, int W, int top,
                          hipStream_t st) {
  VK_REQUIRE(T >= 0 && W > 0 && top > 0, "experts (sum): bad sizes T=%d W=%d top=%d", T, W, top);
  if (T == 0) return 0;
  if (W % VK_VEC == 0 && (uintptr_t)out % 16 == 0 && (uintptr_t)y % 16 == 0 && (uintptr_t)extra % 16 == 0) {
    moe_combine_vec_kernel<<<dim3(T, (W / VK_VEC + 255) / 256), 256, 0, st>>>(out, y, wts, pair_row, W, top, extra);
    return vk_check_launch("experts (sum)");
  }
  const int by = std::min((W + 255) / 256, 64);
  moe_combine_kernel<<<dim3(T, by), 256, 0, st>>>(out, y, wts, pair_row, W, top, extra);
  return vk_check_launch("experts (sum)");
}

int vk_moe_combine(float* out, const elem_t* y, const float* wts, const int32_t* pair_row, int T, int W, int top, hipStream_t st) {
  return combine_launch(out, y, wts, pair_row, nullptr, T, W, top, st);
}

// The same, and extra [T, W] (elements) is added to every token's sum last.
int vk_moe_combine_add(float* out, const elem_t* y, const float* wts, const int32_t* pair_row, const elem_t* extra, int T, int W, int top,
                       hipStream_t st) {
  VK_REQUIRE(extra != nullptr, "experts (sum): the output to add is missing");
  return combine_launch(out, y, wts, pair_row, extra, T, W, top, st);
}

}  // extern "C"
