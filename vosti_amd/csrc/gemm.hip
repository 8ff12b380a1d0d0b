// out[M,N] = act[M,K] * w[N,K]^T  (weights in [out_features, in_features] layout).
//
// Reduction order, the same in every kernel of this file and for every M:
//   K is cut into chunks of 512 elements starting at 0.  Within a chunk the
//   products are accumulated from zero by mma_slab() over the chunk's slabs in
//   ascending order (weights are the first MFMA operand, activations the
//   second).  The chunk sums are then added to a zero total in ascending chunk
//   order, and the total is rounded to the element type once.
// An output element therefore never depends on M, on the other rows of its
// tile or on which kernel produced it; the choice between the kernels is a
// matter of speed only.  The reference keys its tile configuration on (N, K)
// for the same reason (kernels/triton_kernels/matmul.py:33-73,
// kernels/triton_kernels/qkv_matmul.py:24-32).
//
//   gemm_stream         M <= 64, K a multiple of 512.  Streams the weights once from HBM: persistent
//                       workgroups walk over 16-row weight tiles (one or two at a time); wave w of a
//                       workgroup's W waves takes the chunks w, w+W, ... and keeps a rolling window of
//                       slabs in flight, also across tile borders.  After each round of W chunks the chunk
//                       sums meet in LDS and are added in chunk order.  W is eight, or, up to 16 rows, the
//                       number of chunks where that is 2, 4, 5, 6, 10 or 12 (stream_waves).
//   gemm_stream_swiglu  the same for the gate/up projection with SwiGLU folded in (M <= 16).
//   gemm_lines          M <= 16, K a multiple of 512 up to 6,144, 16-bit elements: weights and activations through LDS in whole lines, tiles of eight
//                       or four weight rows, optionally SwiGLU in the epilogue (lines_rows says when).
//   gemm_rows           17 <= M <= 64, K a multiple of 512, 16-bit elements: weights and activations through LDS in whole lines, a workgroup walks all
//                       of K, optionally SwiGLU in the epilogue (rows_width says when).
//   gemm_mid            17 <= M <= 64 (more in blocks), K a multiple of 512: 64 or 32 weight rows per workgroup, weights
//                       streamed into registers, the activations of the chunks in work shared through LDS.
//   gemm_split          M <= 64, K a multiple of 512, 16-bit elements, with a workspace: a workgroup per
//                       (128 weight rows, chunk) leaves its chunk sums in the workspace, a second kernel
//                       adds them in chunk order (vk_gemm_split; vk_gemm_split_preferred says when).
//   gemm_skinny         M <= 64, any K: the same decomposition with predicated loads.
//   gemm_pipe           any M, K a multiple of two slabs (128 bytes of a row): 128x128 output tile per
//                       workgroup, 64x64 per wave, tiles straight from global memory into LDS, two
//                       stages, or four and 64 or 96 weight rows where no compute unit has more than one
//                       workgroup (pipe_fragments_in_one_round); a second accumulator set holds the total.  Optionally SwiGLU in the
//                       epilogue.
//   gemm_alternate      256 rows or more, K a multiple of 512, 16-bit elements: 256 x 192, 160 or 128 per workgroup of eight
//                       waves whose two halves take turns between LDS and the matrix unit.  Optionally SwiGLU in the epilogue
//                       (alternate_fragments says when).
//   gemm_fine           32-bit elements, more than 64 rows (32 where K is short or with SwiGLU), K as gemm_pipe: tiles of 32 x 32 to 96 x 64 or 64 x 128, the one
//                       whose launch ends first, unless larger ones of gemm_pipe fill the units (fine_takes, fine_tile).  Optionally SwiGLU in the epilogue.
//   gemm_tiled          any M and K: the same tile through registers into LDS, predicated.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "common.h"
#include "lines.h"
#include "mma.h"
#include "vec.h"

#define KC_SLABS (KC / VK_SLAB)       // 16 (bfloat16) or 32 (float)
#define SK_WAVES 8

// How a product's sums leave a kernel: whether rows take 16-byte (8-byte) stores, and an activation on the rounded sums.
#define OUT_VEC 1
#define OUT_SQUARED_RELU 2            // max(., 0)^2

__device__ __forceinline__ void store_out4(elem_t* out, int64_t ldo, int m, int n, int M, int N, f32x4 v,
                                           int form) {
  if (m >= M || n >= N) return;
  if (form & OUT_SQUARED_RELU) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float r = fmaxf(round_to_elem(v[i]), 0.f);
      v[i] = r * r;
    }
  }
  elem_t* p = out + (int64_t)m * ldo + n;
  if ((form & OUT_VEC) && n + 3 < N) {
#ifdef VK_F32
    *reinterpret_cast<f32x4*>(p) = v;
#else
    bf16x4 o;
    o[0] = (__bf16)v.x; o[1] = (__bf16)v.y; o[2] = (__bf16)v.z; o[3] = (__bf16)v.w;
    *reinterpret_cast<bf16x4*>(p) = o;
#endif
  } else {
    p[0] = from_f32<elem_t>(v.x);
    if (n + 1 < N) p[1] = from_f32<elem_t>(v.y);
    if (n + 2 < N) p[2] = from_f32<elem_t>(v.z);
    if (n + 3 < N) p[3] = from_f32<elem_t>(v.w);
  }
}

// Up to ROWS (1, 4, 8 or 16) rows of one chunk's activations as a wave's fragments, through LDS of the wave's own (CHUNK_ROWS_BYTES(ROWS)).
// The fragments' own addresses put four rows side by side in four neighbouring lanes, so that a load takes the address unit 64 clocks
// where whole lines take 16: the activations cost a launch of a few weight tiles a workgroup as much of that unit as its weights.  Here a load
// brings whole lines: eight rows of 128 bytes, four of 256, or one of 1,024.  Measured on MI355X, recorded launches with the weights of several
// layers in turn, us, against rows straight to registers: 16-bit 4,096 x 4,096, 1, 8 and 16 rows 8.9 -> 7.9, 9.3 -> 8.5, 10.8 -> 9.4; 6,144 x 4,096,
// 8 rows 14.1 -> 12.1; 2,048 x 6,144, 8 rows 11.6 -> 9.6; 1,024 x 3,072, 1 row 5.7 -> 5.2; 4,096 x 12,288, rows a chunk ahead, 1 and 16 rows
// 21.2 -> 19.3, 28.9 -> 23.4; gate/up with SwiGLU 12,288 x 4,096, 8 rows 37.7 -> 36.5; 32-bit 2,048 x 2,048, 1 and 16 rows 9.6 -> 6.2, 11.9 -> 7.3.  Over
// 315 sizes of 1 to 16 rows 5,163 -> 4,777 us in 16-bit, none more than 2 % over what it was, and 9,536 -> 8,496 in
// 32-bit.  One row as such and not as eight is 2.4 % of that (2,048 x 9,216: 13.97 -> 13.01), two to four rows as four 1.2 % (6,144 x 2,560, 2 rows 9.28 ->
// 8.98; 32-bit 24,600 x 512 11.33 -> 10.56).  Part of it is the order of the weights' loads (EARLY in the kernels).  (Weights through LDS alike do not pay: they come from
// memory, 7.1 us for 33 MB against 7.4.  Tiles of eight or four weight rows for few of them do not either: 1,024 x 2,048 4.4 -> 4.6.)
#define CHUNK_ROWS_BYTES(ROWS) ((ROWS) * KC * (int)sizeof(elem_t))
template <int ROWS>
struct ChunkRows {
  static constexpr int LOADS = CHUNK_ROWS_BYTES(ROWS) / 1024;              // of a kilobyte each
  static constexpr int PER = ROWS < 8 ? ROWS : 8, PIECES = 64 / PER;       // rows of a load, 16-byte pieces of each
  static constexpr int TURN = PER == 8 ? 1 : 4;                            // a row's pieces lie at piece ^ (row * TURN): no two rows on the same banks
  static constexpr int HALF = PER * KC * (int)sizeof(elem_t);              // eight rows, or all
  // The lane's part of a load's address, in bytes from the first row, for the rows PER h ...
  __device__ static __forceinline__ unsigned offset(int h, int64_t lda, int M, int lane) {
    const int row = lane / PIECES, piece = (lane % PIECES) ^ (row * TURN);
    return (unsigned)((min(h * PER + row, M - 1) * lda + piece * VK_VEC) * (int64_t)sizeof(elem_t));
  }
  __device__ static __forceinline__ frag_t fragment(const unsigned char* rows, int slab, int r16, int kg) {     // rows beyond ROWS repeat them
    const int r = r16 & (PER - 1), h = ROWS == 16 ? r16 >> 3 : 0, piece = slab * 4 + kg;
    return *reinterpret_cast<const frag_t*>(rows + h * HALF + (piece / PIECES) * 1024 + r * (1024 / PER) + ((piece % PIECES) ^ (r * TURN)) * 16);
  }
  __device__ static __forceinline__ unsigned char* place(unsigned char* rows, int row, int piece) {      // of one of the first eight rows
    return rows + (piece / PIECES) * 1024 + row * (1024 / PER) + ((piece % PIECES) ^ (row * TURN)) * 16;
  }
};
// Asks for them: LOADS loads.
template <int ROWS>
__device__ __forceinline__ void ask_chunk_rows(const elem_t* act, int64_t lda, int M, int lane, unsigned lds_addr) {
  using C = ChunkRows<ROWS>;
#pragma unroll
  for (int h = 0; h < (ROWS == 16 ? 2 : 1); ++h) {
    const unsigned voff = C::offset(h, lda, M, lane);
#pragma unroll
    for (int i = 0; i < C::HALF / 1024; ++i)
      pipe_load_to_lds16_sv(reinterpret_cast<const unsigned char*>(act) + i * (1024 / C::PER), voff, __builtin_amdgcn_readfirstlane(lds_addr + h * C::HALF + i * 1024));
  }
}

// The activations of a product that norms them itself: row m is (x + residual) * rsqrt(mean(.^2) + eps) * weight, the sum in 32-bit, and the sum's rounded rows
// go to `sum` (the first workgroup writes them): what vk_add_rmsnorm computes, bit for bit, its order of additions included.
struct NormArgs {
  const elem_t* residual;    // [M, K]
  elem_t* sum;               // [M, K]
  const elem_t* weight;      // [K]
  float eps;
};
// Up to ROWS rows of NW chunks by NW waves.  vk_add_rmsnorm's workgroup of four waves takes the kilobytes (groups) of a row in turn, wave q those with g % 4 ==
// q, and adds its own partial sums first: here a (row, q) pair is one wave's, all pairs in turn, a lane holding what that kernel's lane holds.
// load() reads the rows and waits for them (a weight asked for before them would have to arrive first: loads are counted in order); the weights
// are asked for next, and finish() sums, norms and puts the rows into LDS meanwhile.  A norm of its own is a launch of 3.6 us of eight rows of 4,096 and 2.6 of one
// of 1,024 between two products (normed_rows has the pairs measured).
template <int ROWS, int NW>
struct NormRows {
  static constexpr int GROUPS = NW * KC * (int)sizeof(elem_t) / 1024, Q = GROUPS < 4 ? GROUPS : 4, J = (GROUPS + 3) / 4, PAIRS = (ROWS * Q + NW - 1) / NW;
  float a[PAIRS][J][VK_VEC];
  frag_t w[PAIRS][J];
  __device__ __forceinline__ void load(const NormArgs& n, const elem_t* x, int64_t ldx, int M, int wave, int lane) {
    constexpr int K = NW * KC;
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      const int p = wave + i * NW, row = p / Q;
#pragma unroll
      for (int j = 0; j < J; ++j) {
        const int g = p % Q + 4 * j;
        if (row < M && g < GROUPS) {
          w[i][j] = *reinterpret_cast<const frag_t*>(n.weight + (g * 64 + lane) * VK_VEC);
          float b[VK_VEC];
          load_elems(x + row * ldx + (g * 64 + lane) * VK_VEC, a[i][j]);
          load_elems(n.residual + (int64_t)row * K + (g * 64 + lane) * VK_VEC, b);
#pragma unroll
          for (int e = 0; e < VK_VEC; ++e) a[i][j][e] = a[i][j][e] + b[e];
        }
      }
    }
    if (blockIdx.x == 0) {
#pragma unroll
      for (int i = 0; i < PAIRS; ++i) {
        const int p = wave + i * NW, row = p / Q;
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int g = p % Q + 4 * j;
          if (row < M && g < GROUPS) store_elems(n.sum + (int64_t)row * K + (g * 64 + lane) * VK_VEC, a[i][j]);
        }
      }
    }
  }
  // A barrier that waits for what went to LDS, and not for the loads on their way.
  __device__ static __forceinline__ void meet() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xC07F);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  }
  // red: [ROWS][4] floats of LDS; place(row, g): where the lane's 16 bytes of a row's group go.
  template <typename PLACE>
  __device__ __forceinline__ void finish(const NormArgs& n, int M, int wave, int lane, float* red, PLACE place) {
    constexpr int K = NW * KC;
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      const int p = wave + i * NW, row = p / Q;
      if (row < M) {
        float part = 0.f;
#pragma unroll
        for (int j = 0; j < J; ++j) {
          if (p % Q + 4 * j < GROUPS) {
#pragma unroll
            for (int e = 0; e < VK_VEC; ++e) part = part + a[i][j][e] * a[i][j][e];
          }
        }
        part = wave_sum_xor(part);
        if (lane == 0) red[row * 4 + p % Q] = part;
      }
    }
    meet();
#pragma unroll
    for (int i = 0; i < PAIRS; ++i) {
      const int p = wave + i * NW, row = p / Q;
      if (row < M) {
        float total = red[row * 4];
#pragma unroll
        for (int q = 1; q < Q; ++q) total = total + red[row * 4 + q];
        const float rr = rsqrtf(total / (float)K + n.eps);
#pragma unroll
        for (int j = 0; j < J; ++j) {
          const int g = p % Q + 4 * j;
          if (g < GROUPS) {
            float y[VK_VEC];
#pragma unroll
            for (int e = 0; e < VK_VEC; ++e) y[e] = (a[i][j][e] * rr) * to_f32(w[i][j][e]);
            store_elems(reinterpret_cast<elem_t*>(place(row, g)), y);
          }
        }
      }
    }
    meet();
  }
};

// ------------------------------------------------------------------ skinny
// MT: 16-row activation tiles (M <= 16*MT).  W: slabs in flight per wave.
template <int MT, int W>
__global__ __launch_bounds__(64 * SK_WAVES) void gemm_skinny_kernel(elem_t* __restrict__ out,
                                                                    const elem_t* __restrict__ act,
                                                                    const elem_t* __restrict__ w, int M, int N, int K,
                                                                    int64_t lda, int64_t ldo, int out_form) {
  static_assert(KC_SLABS % W == 0, "the window must divide a chunk");
  __shared__ f32x4 part[SK_WAVES][MT][64];

  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int n0 = blockIdx.x * 16;
  const int nchunks = (K + KC - 1) / KC;
  const int rounds = (nchunks + SK_WAVES - 1) / SK_WAVES;

  const bool wok = n0 + r16 < N;
  const elem_t* wrow = w + (int64_t)(wok ? n0 + r16 : 0) * K + kg * VK_VEC;
  const elem_t* arow[MT];
  bool aok[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int m = mt * 16 + r16;
    aok[mt] = m < M;
    arow[mt] = act + (int64_t)(aok[mt] ? m : 0) * lda + kg * VK_VEC;
  }

  frag_t wbuf[W], abuf[W][MT];
  auto issue = [&](int c, int s, int slot) {
    const int k = c * KC + s * VK_SLAB;
    const bool kok = k + kg * VK_VEC < K;
    wbuf[slot] = load_frag(wrow + k, wok && kok);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) abuf[slot][mt] = load_frag(arow[mt] + k, aok[mt] && kok);
  };

  int c = wave;
  if (c < nchunks) {
#pragma unroll
    for (int i = 0; i < W; ++i) issue(c, i, i);
  }
  f32x4 total = {0.f, 0.f, 0.f, 0.f};
  for (int round = 0; round < rounds; ++round, c += SK_WAVES) {
    f32x4 acc[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (c < nchunks) {
      const int cn = c + SK_WAVES;
      const bool has_next = cn < nchunks;
#pragma unroll
      for (int i = 0; i < KC_SLABS; ++i) {
        const int slot = i % W;
        const frag_t fw = wbuf[slot];
        frag_t fa[MT];
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) fa[mt] = abuf[slot][mt];
        if (i + W < KC_SLABS) issue(c, i + W, slot);
        else if (has_next) issue(cn, i + W - KC_SLABS, slot);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[mt] = mma_slab(fw, fa[mt], acc[mt]);
      }
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) part[wave][mt][lane] = acc[mt];
    __syncthreads();
    if (wave < MT) {
      for (int w2 = 0; w2 < SK_WAVES; ++w2) {
        if (round * SK_WAVES + w2 < nchunks) {
          const f32x4 p = part[w2][wave][lane];
          total.x = total.x + p.x; total.y = total.y + p.y; total.z = total.z + p.z; total.w = total.w + p.w;
        }
      }
    }
    __syncthreads();
  }
  if (wave < MT) store_out4(out, ldo, wave * 16 + r16, n0 + 4 * kg, M, N, total, out_form);
}

// ---------------------------------------------------------------- streaming
// The skinny kernel for K a multiple of 512, built to keep HBM busy: workgroups
// are persistent and walk over weight tiles (16 rows) with a stride of the grid;
// a wave's window of W slabs in flight runs on across tile borders, so the
// memory pipe never drains; no load is predicated (rows beyond N or M are
// clamped to the last valid row and their results dropped), because a select on
// a loaded value makes the compiler wait for it at once; and with RC > 0 a wave
// keeps the activations of its RC chunks (K <= RC * 4096) in registers for the
// whole kernel.  One barrier per round of eight chunks.
// ROWS: 1, 4, 8 or 16: the activations (one tile) come through LDS (ChunkRows): resident ones once, others a chunk ahead; 0: straight to registers.
// NORM: the rows are normed first (NormRows), K is NW chunks.
template <int MT, int W, int RC, int NT, int NW = SK_WAVES, int ROWS = 0, bool NORM = false>
__global__ __launch_bounds__(64 * NW) void gemm_stream_kernel(elem_t* __restrict__ out,
                                                                    const elem_t* __restrict__ act,
                                                                    const elem_t* __restrict__ w, int M, int N, int K,
                                                                    int64_t lda, int64_t ldo, int out_form, NormArgs norm) {
  // NT: 16-row weight tiles per workgroup.  With several activation tiles every workgroup reads all
  // activations once, M * K elements beside its 16 * NT * K weights: more weight rows per workgroup
  // keep that traffic, which comes from the second-level cache, in proportion.
  static_assert(KC_SLABS % W == 0, "the window must divide a chunk");
  // RC: chunks per wave whose activations stay in registers for the whole kernel (0: none are kept;
  // K <= RC * 8 chunks).  A chunk of one activation tile is 64 registers of 16-bit elements.
  constexpr bool RES = RC > 0;
  static_assert(RC * MT <= 2, "resident activations: at most two chunk tiles per wave");
  static_assert(NT * MT <= NW, "one wave adds up each output tile");
  __shared__ f32x4 part[2][NW][NT * MT][64];

  static_assert(ROWS == 0 || (MT == 1 && NT == 1 && RC <= 1), "one chunk tile of activations comes through LDS");
  extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];      // CHUNK_ROWS_BYTES(ROWS) a wave

  const int lane = threadIdx.x & 63, wave = ROWS ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int nchunks = K / KC;
  const int ntiles = (N + 16 * NT - 1) / (16 * NT);     // tile: NT * 16 weight rows
  // The loop over tiles written out twice (with a tile to ask for next, and without), its loads kept in the order of the slabs: a load that may or may not
  // be asked for makes the compiler wait for all of them.  16-bit 6,144 x 2,560, 16 rows 10.3 -> 9.5 us, 32-bit 2,048 x 2,048 10.0 -> 7.3; not with more
  // than eight waves of 32-bit values or two projections' windows, whose registers do not suffice (SwiGLU 17,408 x 5,120 75.8 -> 82 us).
  constexpr bool EARLY = RC == 1 && MT == 1 && (NW <= 8 || sizeof(elem_t) == 2);
  constexpr bool AHEAD = ROWS > 0 && !RES;               // a chunk's rows are asked for while the one before is computed, into registers
  unsigned char* own_rows = rows_lds + wave * CHUNK_ROWS_BYTES(ROWS);
  static_assert(!NORM || (RES && ROWS > 0 && ROWS <= 8), "rows are normed on their way through LDS");
  NormRows<NORM ? ROWS : 1, NORM ? NW : 2> normed;
  if constexpr (NORM) {
    normed.load(norm, act, lda, M, wave, lane);
    __builtin_amdgcn_sched_barrier(0);
  } else if constexpr (ROWS > 0) {
    ask_chunk_rows<ROWS>(act + (int64_t)min(wave, nchunks - 1) * KC, lda, M, lane, lds_offset_of(own_rows));
  }

  const elem_t* arow[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) arow[mt] = act + (int64_t)min(mt * 16 + r16, M - 1) * lda + kg * VK_VEC;

  frag_t wbuf[W][NT], abuf[RES ? RC * KC_SLABS : AHEAD ? 1 : W][MT];
  if (RES && ROWS == 0) {
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      const int c = min(r * NW + wave, nchunks - 1);     // beyond K: the last chunk again (not used)
#pragma unroll
      for (int s = 0; s < KC_SLABS; ++s)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
          abuf[r * KC_SLABS + s][mt] = *reinterpret_cast<const frag_t*>(arow[mt] + c * KC + s * VK_SLAB);
    }
  }
  auto issue = [&](int tile, int c, int s, int slot) {
    const int k = c * KC + s * VK_SLAB;
#pragma unroll
    for (int nt = 0; nt < NT; ++nt)
      wbuf[slot][nt] = *reinterpret_cast<const frag_t*>(w + (int64_t)min((tile * NT + nt) * 16 + r16, N - 1) * K + kg * VK_VEC + k);
    if (!RES && !AHEAD) {
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) abuf[slot][mt] = *reinterpret_cast<const frag_t*>(arow[mt] + k);
    }
  };

  int tile = blockIdx.x;
  if (tile < ntiles && wave < nchunks) {
#pragma unroll
    for (int i = 0; i < W; ++i) issue(tile, wave, i, i);
  }
  if constexpr (NORM) {
    __builtin_amdgcn_sched_barrier(0);
    normed.finish(norm, M, wave, lane, reinterpret_cast<float*>(part), [&](int row, int g) {
      constexpr int PER_CHUNK = KC * (int)sizeof(elem_t) / 1024;
      return ChunkRows<ROWS>::place(rows_lds + g / PER_CHUNK * CHUNK_ROWS_BYTES(ROWS), row, g % PER_CHUNK * 64 + lane);
    });
#pragma unroll
    for (int i = 0; i < KC_SLABS; ++i) abuf[i][0] = ChunkRows<ROWS>::fragment(own_rows, i, r16, kg);
  } else if constexpr (ROWS > 0) {
    if (wave < nchunks) {                                // a wave with a chunk has a tile: there are no more workgroups than tiles
      __builtin_amdgcn_sched_barrier(0);                 // the weights' loads stay in front of the wait that counts them
      wait_vmcnt_n<W * NT>();                            // the rows are there, the first weights on their way
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (RES) {
#pragma unroll
        for (int i = 0; i < KC_SLABS; ++i) abuf[i][0] = ChunkRows<ROWS>::fragment(own_rows, i, r16, kg);
      }
    } else {
      wait_vmcnt_n<0>();
    }
  }
  using C = ChunkRows<AHEAD ? ROWS : 1>;
  frag_t held[AHEAD ? C::LOADS : 1];
  int parity = 0;
  auto one_tile = [&](auto more_) __attribute__((always_inline)) {
    f32x4 total = {0.f, 0.f, 0.f, 0.f};
    auto round = [&](auto next_, int base, int r) __attribute__((always_inline)) {       // chunks base .. base + 7; r = base / 8 where that is a constant
      constexpr int NEXT = decltype(next_)::value;
      const int c = base + wave;
      f32x4 acc[NT][MT];
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
      if (c < nchunks) {
        // What this wave streams next: its next chunk of this tile, else its first chunk of the next tile.  A load that may or may not be asked for
        // makes the compiler wait for all of them when the chunk ends: where something always follows (NEXT) the loads are plain ones, of this
        // chunk again for the few waves that have none; a workgroup's last tile (one chunk a wave) asks for nothing.
        int nt_ = tile, nc = c + NW;
        bool ask = NEXT != 0;
        if constexpr (MT > 1) {      // loads that may not be asked for need no address of this chunk: it costs 17 to 32 rows 2 to 3 % (4,096 x 12,288, 32 rows 39.5 -> 40.5 us)
          if (nc >= nchunks) {
            nt_ = tile + gridDim.x;
            nc = wave;
          }
          ask = nt_ < ntiles;
        } else if (nc >= nchunks) {
          const bool has_next = tile + (int)gridDim.x < ntiles;
          nt_ = has_next ? tile + gridDim.x : tile;
          nc = has_next ? wave : c;
          if (NEXT == 2) ask = has_next;
        }
        if (AHEAD && ask) {
          const unsigned char* rows = reinterpret_cast<const unsigned char*>(act + (int64_t)nc * KC);
#pragma unroll
          for (int l = 0; l < C::LOADS; ++l)
            held[l] = *reinterpret_cast<const frag_t*>(rows + C::offset(l / (C::HALF / 1024), lda, M, lane) + l % (C::HALF / 1024) * (1024 / C::PER));
        }
#pragma unroll
        for (int i = 0; i < KC_SLABS; ++i) {
          const int slot = i % W;
          frag_t fw[NT], fa[MT];
#pragma unroll
          for (int nt = 0; nt < NT; ++nt) fw[nt] = wbuf[slot][nt];
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) {
            if constexpr (AHEAD) fa[mt] = C::fragment(own_rows, i, r16, kg);
            else fa[mt] = RES ? abuf[r * KC_SLABS + i][mt] : abuf[slot][mt];
          }
          if (i + W < KC_SLABS) issue(tile, c, i + W, slot);
          else if (ask) issue(nt_, nc, i + W - KC_SLABS, slot);
#pragma unroll
          for (int nt = 0; nt < NT; ++nt)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[nt][mt] = mma_slab(fw[nt], fa[mt], acc[nt][mt]);
          if (EARLY) __builtin_amdgcn_sched_barrier(0);      // the compiler would ask for the slabs of the second half when the first is done
        }
        if (AHEAD && ask) {                              // this chunk's fragments have been read: its place is free
#pragma unroll
          for (int l = 0; l < C::LOADS; ++l) *reinterpret_cast<frag_t*>(own_rows + l * 1024 + lane * 16) = held[l];
        }
      }
#pragma unroll
      for (int nt = 0; nt < NT; ++nt)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) part[parity][wave][nt * MT + mt][lane] = acc[nt][mt];
      __syncthreads();
      if (wave < NT * MT) {
        for (int w2 = 0; w2 < NW; ++w2) {
          if (base + w2 < nchunks) {
            const f32x4 p = part[parity][w2][wave][lane];
            total.x = total.x + p.x; total.y = total.y + p.y; total.z = total.z + p.z; total.w = total.w + p.w;
          }
        }
      }
      parity ^= 1;
    };
    const std::integral_constant<int, 2> maybe;
    if constexpr (RC == 1) {
      if (0 < nchunks) round(more_, 0, 0);
    } else if constexpr (RES) {
#pragma unroll
      for (int r = 0; r < RC; ++r)
        if (r * NW < nchunks) round(maybe, r * NW, r);
    } else {
      int base = 0;
      if (MT == 1 && sizeof(elem_t) == 2)                 // (elsewhere it does not pay: 32-bit 5,120 x 17,408, 1 row 102.6 -> 107.8 us; 4,096 x 4,608, 17 rows 12.8 -> 15.9)
        for (; base + NW < nchunks; base += NW) round(std::integral_constant<int, 1>(), base, 0);
      for (; base < nchunks; base += NW) round(maybe, base, 0);
    }
    if (wave < NT * MT)
      store_out4(out, ldo, (wave % MT) * 16 + r16, (tile * NT + wave / MT) * 16 + 4 * kg, M, N, total, out_form);
  };
  if constexpr (EARLY) {
    for (; tile + (int)gridDim.x < ntiles; tile += gridDim.x) one_tile(std::integral_constant<int, 1>());
    if (tile < ntiles) one_tile(std::integral_constant<int, 0>());
  } else {
    for (; tile < ntiles; tile += gridDim.x) one_tile(std::integral_constant<int, 2>());
  }
}

// The streaming kernel for the gate/up projection with the activation folded in:
// w holds I gate rows, then I up rows; a workgroup streams the gate tile and the
// matching up tile together and writes  out[m, n] = silu(g) * u  with g and u the
// two projections rounded to the element type first, which is what the separate
// GEMM and SwiGLU kernels compute (kernels/triton_kernels/silu_mul.py:64-87).
// M <= 16, K <= 4096 (activations resident in registers).
template <int W, int RC, int NW = SK_WAVES, int ROWS = 0, bool NORM = false>
__global__ __launch_bounds__(64 * NW) void gemm_stream_swiglu_kernel(elem_t* __restrict__ out,
                                                                           const elem_t* __restrict__ act,
                                                                           const elem_t* __restrict__ w, int M, int I,
                                                                           int K, int64_t lda, int64_t ldo,
                                                                           int out_form, NormArgs norm) {
  static_assert(KC_SLABS % W == 0, "the window must divide a chunk");
  static_assert(RC <= 2, "two chunks of activations stay in registers");
  __shared__ f32x4 part[2][RC][NW][2][64];      // two sets, used in turn: one barrier per tile

  static_assert(ROWS == 0 || RC == 1, "one chunk tile of activations comes through LDS");
  // As in the kernel above; two projections' windows leave fewer registers.
  constexpr bool EARLY = ROWS > 0 && NW <= 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char rows_lds[];      // CHUNK_ROWS_BYTES(ROWS) a wave
  const int lane = threadIdx.x & 63, wave = ROWS ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : threadIdx.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int nchunks = K / KC;
  const int ntiles = (I + 15) / 16;
  unsigned char* own_rows = rows_lds + wave * CHUNK_ROWS_BYTES(ROWS);
  static_assert(!NORM || (ROWS > 0 && ROWS <= 8), "rows are normed on their way through LDS");
  NormRows<NORM ? ROWS : 1, NORM ? NW : 2> normed;
  if constexpr (NORM) {
    normed.load(norm, act, lda, M, wave, lane);
    __builtin_amdgcn_sched_barrier(0);
  } else if constexpr (ROWS > 0) {
    ask_chunk_rows<ROWS>(act + (int64_t)min(wave, nchunks - 1) * KC, lda, M, lane, lds_offset_of(own_rows));
  }

  // Wave w has chunks w, w + 8, ...: RC of them (chunks beyond K are read as the last and not used).
  frag_t wg[W], wu[W], abuf[RC * KC_SLABS];
#pragma unroll
  for (int r = 0; r < (ROWS ? 0 : RC); ++r) {
    const int c = min(r * NW + wave, nchunks - 1);
    const elem_t* arow = act + (int64_t)min(r16, M - 1) * lda + kg * VK_VEC;
#pragma unroll
    for (int s = 0; s < KC_SLABS; ++s) abuf[r * KC_SLABS + s] = *reinterpret_cast<const frag_t*>(arow + c * KC + s * VK_SLAB);
  }
  // Slab g of this wave's stream over a tile: chunk (g / 16) * 8 + wave, slab g % 16 of it.
  const int my_chunks = wave < nchunks ? (nchunks - wave + NW - 1) / NW : 0;     // <= RC
  const int my_slabs = my_chunks * KC_SLABS;
  auto issue = [&](int tile, int g, int slot) {
    const int64_t row = min(tile * 16 + r16, I - 1);
    const int c = (g / KC_SLABS) * NW + wave;
    const elem_t* p = w + row * K + kg * VK_VEC + (int64_t)c * KC + (g % KC_SLABS) * VK_SLAB;
    wg[slot] = *reinterpret_cast<const frag_t*>(p);
    wu[slot] = *reinterpret_cast<const frag_t*>(p + (int64_t)I * K);
  };

  int tile = blockIdx.x;
  const bool active = my_chunks > 0;
  if (tile < ntiles && active) {
#pragma unroll
    for (int i = 0; i < W; ++i) issue(tile, i, i);
  }
  if constexpr (NORM) {
    __builtin_amdgcn_sched_barrier(0);
    normed.finish(norm, M, wave, lane, reinterpret_cast<float*>(part), [&](int row, int g) {
      constexpr int PER_CHUNK = KC * (int)sizeof(elem_t) / 1024;
      return ChunkRows<ROWS>::place(rows_lds + g / PER_CHUNK * CHUNK_ROWS_BYTES(ROWS), row, g % PER_CHUNK * 64 + lane);
    });
#pragma unroll
    for (int i = 0; i < KC_SLABS; ++i) abuf[i] = ChunkRows<ROWS>::fragment(own_rows, i, r16, kg);
  } else if constexpr (ROWS > 0) {
    if (active) {                                        // as in the kernel above
      __builtin_amdgcn_sched_barrier(0);
      wait_vmcnt_n<2 * W>();
      asm volatile("" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < KC_SLABS; ++i) abuf[i] = ChunkRows<ROWS>::fragment(own_rows, i, r16, kg);
    } else {
      wait_vmcnt_n<0>();
    }
  }
  int parity = 0;
  auto one_tile = [&](auto more_) __attribute__((always_inline)) {
    constexpr int NEXT = decltype(more_)::value;          // as in the kernel above
    const int nt = tile + gridDim.x;
    const bool ask = NEXT == 2 ? nt < ntiles : NEXT == 1;
#pragma unroll
    for (int r = 0; r < RC; ++r) {
      f32x4 ag = {0.f, 0.f, 0.f, 0.f}, au = {0.f, 0.f, 0.f, 0.f};
      if (r < my_chunks) {
#pragma unroll
        for (int i = 0; i < KC_SLABS; ++i) {
          const int slot = i % W;
          const frag_t fg = wg[slot], fu = wu[slot];
          const int g = r * KC_SLABS + i + W;             // the slab that takes this slot
          if (EARLY ? i + W < KC_SLABS : g < my_slabs) issue(tile, g, slot);
          else if (ask) issue(nt, g - my_slabs, slot);
          ag = mma_slab(fg, abuf[r * KC_SLABS + i], ag);
          au = mma_slab(fu, abuf[r * KC_SLABS + i], au);
          if (EARLY) __builtin_amdgcn_sched_barrier(0);
        }
      }
      part[parity][r][wave][0][lane] = ag;
      part[parity][r][wave][1][lane] = au;
    }
    __syncthreads();
    if (wave == 0) {       // adds up, in chunk order, and finishes the rows
      f32x4 tg = {0.f, 0.f, 0.f, 0.f}, tu = {0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < nchunks; ++c) {
        const f32x4 pg = part[parity][c / NW][c % NW][0][lane];
        const f32x4 pu = part[parity][c / NW][c % NW][1][lane];
        tg.x = tg.x + pg.x; tg.y = tg.y + pg.y; tg.z = tg.z + pg.z; tg.w = tg.w + pg.w;
        tu.x = tu.x + pu.x; tu.y = tu.y + pu.y; tu.z = tu.z + pu.z; tu.w = tu.w + pu.w;
      }
      const float g[4] = {round_to_elem(tg.x), round_to_elem(tg.y), round_to_elem(tg.z), round_to_elem(tg.w)};
      const float u[4] = {round_to_elem(tu.x), round_to_elem(tu.y), round_to_elem(tu.z), round_to_elem(tu.w)};
      f32x4 y;
      y.x = (g[0] * (1.0f / (1.0f + expf(-g[0])))) * u[0];
      y.y = (g[1] * (1.0f / (1.0f + expf(-g[1])))) * u[1];
      y.z = (g[2] * (1.0f / (1.0f + expf(-g[2])))) * u[2];
      y.w = (g[3] * (1.0f / (1.0f + expf(-g[3])))) * u[3];
      store_out4(out, ldo, r16, tile * 16 + 4 * kg, M, I, y, out_form);
    }
    parity ^= 1;
  };
  if constexpr (EARLY) {
    for (; tile + (int)gridDim.x < ntiles; tile += gridDim.x) one_tile(std::integral_constant<int, 1>());
    if (tile < ntiles) one_tile(std::integral_constant<int, 0>());
  } else {
    for (; tile < ntiles; tile += gridDim.x) one_tile(std::integral_constant<int, 2>());
  }
}

// ------------------------------------------------------------------- lines
// Up to 16 rows of 16-bit elements, K of up to twelve chunks, one a wave.  What bounds such a product is how its weights come from memory.  In the operands'
// own order (the streaming kernels) an instruction touches 16 rows, half a cache line of each: the address unit takes 64 clocks for a kilobyte, and
// a line must stay in the first cache until its other half is asked for, so that the loads cannot say that they are the only ones.  Here a load
// brings one row of a chunk, a whole kilobyte, into LDS, marked as read once: plain reads of 201 MB by 256 workgroups take 35.1 us in strides, 34.0 in pieces of
// their own and 30.3 marked so (6.6 TB/s); 64-byte pieces marked so are slower than unmarked (36.7 -> 39).  The activations come the same way, once, and stay in
// registers.  A workgroup walks over tiles of R weight rows with a ring of slots a wave; every wave waits for its own loads only, and a barrier a
// tile stands between the chunk sums and the wave (another one each tile) that adds them in chunk order, the order of every kernel here.  With the
// barrier a wave that is early cannot ask for more than its ring holds; counting arrivals in LDS instead, the last wave adding, was slower (4,096 x
// 4,096, 8 rows 8.3 -> 8.4 us, gate/up 9,728 x 2,560 18.1 -> 19.1), as were sums read four or eight at a time.
// Measured on MI355X, recorded launches with the weights of several layers in turn, us, against the streaming kernels: 1,024 x 2,048, 1 row 4.13 -> 3.22;
// 1,024 x 3,072, 8 rows 5.7 -> 4.5; 2,048 x 2,048, 8 rows 4.6 -> 4.1; 2,048 x 6,144, 1 row 8.6 -> 6.4; 5,120 x 5,120, 8 rows 15.3 -> 11.7; 6,144 x 4,096, 8 rows
// 12.2 -> 11.1; gate/up with SwiGLU 1,536 x 2,048, 8 rows 6.8 -> 5.3; 9,728 x 2,560 24.1 -> 18.2; 12,288 x 4,096 36.8 -> 34.3; 17,408 x 5,120 77.5 -> 58.3 (6.1 TB/s).
// Not in 32-bit: four to eight of a product's sixteen rows leave three quarters or half of the matrix unit unused, which a 32-bit slab cannot spare
// (2,048 x 2,048 6.4 -> 7.1).
#ifdef VK_BF16
// What a launch fixes: bytes of LDS a wave has to itself, slots in them, and how many of those lie beside the activations.
struct LinePlan {
  int own_bytes, slots, first_slots;
};
// NORM: 0, or K's chunks: the rows are normed first (NormRows).
template <int R, int ROWS, int P, int NORM = 0>
__global__ __launch_bounds__(NORM ? 64 * NORM : 768) void gemm_lines_kernel(elem_t* __restrict__ out, const elem_t* __restrict__ act, const elem_t* __restrict__ w,
                                                                            int M, int N, int K, int64_t lda, int64_t ldo, int out_form, LinePlan plan,
                                                                            NormArgs norm) {
  using W = LineRows<R>;
  using A = LineRows<ROWS>;
  constexpr int W_BYTES = R * 1024, SLOT = P * W_BYTES, L = P * R, SUMS = R / 4 * 16;      // L: loads of a slot; SUMS: lanes with sums
  constexpr int S_MAX = 63 / L < LINE_SLOTS ? 63 / L : LINE_SLOTS;                         // no more loads than their counter counts
  extern __shared__ __attribute__((aligned(16))) unsigned char lines_lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = NORM ? NORM : blockDim.x >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int S = plan.slots, step = gridDim.x, tiles = ((N + R - 1) / R - 1 - (int)blockIdx.x) / step + 1;      // of this workgroup, at least one
  unsigned char* own = lines_lds + wave * plan.own_bytes;
  f32x4* part = reinterpret_cast<f32x4*>(lines_lds + waves * plan.own_bytes);            // [2][waves][P][SUMS]
  auto slot_at = [&](int s) { return own + plan.own_bytes - (s + 1) * SLOT; };            // the first ones lie beside the activations, the others in their place
  auto ask = [&](int k, int s) {                            // the workgroup's tile k
    const int tile = (int)blockIdx.x + k * step;
    const elem_t* first = w + (int64_t)tile * R * K + wave * KC;
    const unsigned at = lds_offset_of(slot_at(s));
    W::template ask<true>(first, K, N - tile * R, lane, at);
    if constexpr (P == 2) W::template ask<true>(first + (int64_t)N * K, K, N - tile * R, lane, at + W_BYTES);
  };
  auto wait_for_all_but = [&](int slots) {                  // the loads of that many slots, asked for last, may still be on their way
    __builtin_amdgcn_sched_barrier(0);
    if (S_MAX >= 6 && slots >= 6) wait_vmcnt_n<(S_MAX >= 6 ? 6 : 0) * L>();
    else if (S_MAX >= 5 && slots == 5) wait_vmcnt_n<(S_MAX >= 5 ? 5 : 0) * L>();
    else if (S_MAX >= 4 && slots == 4) wait_vmcnt_n<(S_MAX >= 4 ? 4 : 0) * L>();
    else if (S_MAX >= 3 && slots == 3) wait_vmcnt_n<(S_MAX >= 3 ? 3 : 0) * L>();
    else if (S_MAX >= 2 && slots == 2) wait_vmcnt_n<(S_MAX >= 2 ? 2 : 0) * L>();
    else if (slots == 1) wait_vmcnt_n<L>();
    else wait_vmcnt_n<0>();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  auto lds_done = [&]() {                                   // this wave's accesses to LDS: what it has read may be overwritten, what it wrote is there
    __builtin_amdgcn_s_waitcnt(0xC07F);                    // lgkmcnt(0)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };
  const int before = min(plan.first_slots, tiles);
  static_assert(ROWS <= 8 || !NORM, "up to eight rows are normed");
  NormRows<NORM ? ROWS : 1, NORM ? NORM : 2> normed;
  if constexpr (NORM != 0) {
    normed.load(norm, act, lda, M, wave, lane);
    __builtin_amdgcn_sched_barrier(0);
    wait_vmcnt_n<0>();                                     // (a workgroup's part of the sums as well)
  } else {
    A::template ask<false>(act + wave * KC, lda, M, lane, lds_offset_of(own));
  }
#pragma unroll
  for (int s = 0; s < S_MAX; ++s)
    if (s < before) ask(s, s);
  if constexpr (NORM != 0) {
    normed.finish(norm, M, wave, lane, reinterpret_cast<float*>(part), [&](int row, int g) { return lines_lds + g * plan.own_bytes + row * 1024 + ((lane ^ A::turn(row)) * 16); });
  } else {
    wait_for_all_but(before);
  }
  frag_t rows[KC_SLABS];
#pragma unroll
  for (int i = 0; i < KC_SLABS; ++i) rows[i] = A::fragment(own, i, r16, kg);
  lds_done();
#pragma unroll
  for (int s = 0; s < S_MAX; ++s)
    if (s >= before && s < S && s < tiles) ask(s, s);
  int s = 0;
  for (int k = 0; k < tiles; ++k) {
    wait_for_all_but(min(S, tiles - k) - 1);
    const unsigned char* at = slot_at(s);
    f32x4 acc[P];
#pragma unroll
    for (int p = 0; p < P; ++p) acc[p] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < KC_SLABS; ++i)
#pragma unroll
      for (int p = 0; p < P; ++p) acc[p] = mma_slab(W::fragment(at + p * W_BYTES, i, r16, kg), rows[i], acc[p]);
    f32x4* sums = part + (k & 1) * waves * P * SUMS;
    if (lane < SUMS) {
#pragma unroll
      for (int p = 0; p < P; ++p) sums[(wave * P + p) * SUMS + lane] = acc[p];
    }
    lds_done();
    if (k + S < tiles) ask(k + S, s);
    s = s + 1 == S ? 0 : s + 1;
    __builtin_amdgcn_s_barrier();                           // (the loads that are on their way need no wait here)
    asm volatile("" ::: "memory");
    if (wave == k % waves && lane < SUMS) {                 // in chunk order; these sums' place is written again two barriers on
      const int n0 = ((int)blockIdx.x + k * step) * R;
      f32x4 total[P];
#pragma unroll
      for (int p = 0; p < P; ++p) total[p] = f32x4{0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < waves; ++c) {
#pragma unroll
        for (int p = 0; p < P; ++p) {
          const f32x4 v = sums[(c * P + p) * SUMS + lane];
          total[p].x = total[p].x + v.x; total[p].y = total[p].y + v.y; total[p].z = total[p].z + v.z; total[p].w = total[p].w + v.w;
        }
      }
      if constexpr (P == 2) {
        const float g[4] = {round_to_elem(total[0].x), round_to_elem(total[0].y), round_to_elem(total[0].z), round_to_elem(total[0].w)};
        const float u[4] = {round_to_elem(total[1].x), round_to_elem(total[1].y), round_to_elem(total[1].z), round_to_elem(total[1].w)};
        total[0].x = (g[0] * (1.0f / (1.0f + expf(-g[0])))) * u[0];
        total[0].y = (g[1] * (1.0f / (1.0f + expf(-g[1])))) * u[1];
        total[0].z = (g[2] * (1.0f / (1.0f + expf(-g[2])))) * u[2];
        total[0].w = (g[3] * (1.0f / (1.0f + expf(-g[3])))) * u[3];
      }
      store_out4(out, ldo, r16, n0 + 4 * kg, M, min(N, n0 + R), total[0], out_form);
    }
  }
}

// How gemm_lines_kernel's LDS is laid out for M rows of K and tiles of R weight rows of each projection; false: it does not take them.
static bool line_plan(int M, int K, int R, int projections, LinePlan* plan, int* lds_bytes) {
  const int waves = K / KC, rows = M == 1 ? 1 : M <= 4 ? 4 : M <= 8 ? 8 : 16;
  if (M < 1 || M > 16 || K % KC != 0 || waves < 1 || waves > 12) return false;
  const int slot = projections * R * 1024, sums = 2 * waves * projections * R / 4 * 256;
  const int most = 63 / (projections * R) < LINE_SLOTS ? 63 / (projections * R) : LINE_SLOTS;
  for (int groups = 16 / waves > 1 ? 16 / waves : 1; groups >= 1; --groups) {               // a compute unit's LDS among about 16 waves
    int own = ((160 * 1024 / groups - sums) / waves) & ~1023;
    if (own < slot || own < rows * 1024 || (groups > 1 && own < slot + rows * 1024)) continue;
    plan->slots = own / slot < most ? own / slot : most;
    if (plan->slots * slot + rows * 1024 < own) own = plan->slots * slot + rows * 1024;
    plan->own_bytes = own;
    plan->first_slots = (own - rows * 1024) / slot < plan->slots ? (own - rows * 1024) / slot : plan->slots;
    *lds_bytes = waves * own + sums;
    return true;
  }
  return false;
}
template <int R, int ROWS, int P>
static int launch_lines_of(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int form, const LinePlan& plan, int lds_bytes,
                           hipStream_t st) {
  static bool configured = false;
  if (!configured) {
    (void)hipFuncSetAttribute((const void*)gemm_lines_kernel<R, ROWS, P>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    configured = true;
  }
  const int waves = K / KC;
  static int per_cu[16] = {};                               // workgroups that a compute unit holds, by waves (which fix the LDS)
  if (per_cu[waves] == 0) {
    int held = 0;
    (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&held, gemm_lines_kernel<R, ROWS, P>, 64 * waves, lds_bytes);
    per_cu[waves] = held > 0 ? held : 1;
  }
  const int tiles = (N + R - 1) / R, resident = per_cu[waves] * vk_device_cus();
  gemm_lines_kernel<R, ROWS, P><<<tiles < resident ? tiles : resident, 64 * waves, lds_bytes, st>>>(out, act, w, M, N, K, lda, ldo, form, plan, NormArgs{});
  return vk_check_launch("gemm_lines");
}
template <int R, int P>
static int launch_lines(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int form, hipStream_t st) {
  LinePlan plan;
  int lds = 0;
  VK_REQUIRE(line_plan(M, K, R, P, &plan, &lds), "gemm: %d rows of K=%d do not fit a workgroup of %d weight rows", M, K, R);
  if (M == 1) return launch_lines_of<R, 1, P>(out, act, w, M, N, K, lda, ldo, form, plan, lds, st);
  if (M <= 4) return launch_lines_of<R, 4, P>(out, act, w, M, N, K, lda, ldo, form, plan, lds, st);
  if (M <= 8) return launch_lines_of<R, 8, P>(out, act, w, M, N, K, lda, ldo, form, plan, lds, st);
  return launch_lines_of<R, 16, P>(out, act, w, M, N, K, lda, ldo, form, plan, lds, st);
}
#endif

// ------------------------------------------------------------------- tiled
// Workgroup of four waves (2 x 2); a wave owns FN x FM tiles of 16 x 16, so the
// workgroup's tile is (32 FN) weight rows by (32 FM) activation rows.  K moves
// through LDS two slabs at a time, double-buffered; 16-byte columns of a tile
// row are XOR-swizzled by the row so that fragment reads do not collide.
#define T_ROWB 128                     // LDS bytes per tile row: two slabs
#define T_CHUNK_TILES (KC_SLABS / 2)   // K tiles (of two slabs) per chunk

template <int FN, int FM>
__global__ __launch_bounds__(256) void gemm_tiled_kernel(elem_t* __restrict__ out, const elem_t* __restrict__ act,
                                                         const elem_t* __restrict__ w, int M, int N, int K,
                                                         int64_t lda, int64_t ldo, int out_form) {
  constexpr int BN = 32 * FN, BM = 32 * FM;
  constexpr int W_BYTES = BN * T_ROWB, A_BYTES = BM * T_ROWB, BUF_BYTES = W_BYTES + A_BYTES;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];   // [buffer][w tile, act tile]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r16 = lane & 15, kg = lane >> 4;
  const int wn = wave & 1, wm = wave >> 1;
  const int n_blk = blockIdx.x * BN, m_blk = blockIdx.y * BM;
  const int nslabs = (K + VK_SLAB - 1) / VK_SLAB;
  const int ntiles = (nslabs + 1) / 2;

  // Global -> LDS mapping: thread loads 16 bytes at column c16 of rows lrow + 32*i.
  const int lrow = tid >> 3, c16 = tid & 7;
  const elem_t* gw[FN];
  const elem_t* ga[FM];
  bool gw_ok[FN], ga_ok[FM];
#pragma unroll
  for (int i = 0; i < FN; ++i) {
    const int n = n_blk + lrow + 32 * i;
    gw_ok[i] = n < N;
    gw[i] = w + (int64_t)(gw_ok[i] ? n : 0) * K + c16 * VK_VEC;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int m = m_blk + lrow + 32 * i;
    ga_ok[i] = m < M;
    ga[i] = act + (int64_t)(ga_ok[i] ? m : 0) * lda + c16 * VK_VEC;
  }

  frag_t rw[FN], ra[FM];
  auto gload = [&](int kt) {
    const int k = kt * 2 * VK_SLAB;
    const bool kok = k + c16 * VK_VEC < K;
#pragma unroll
    for (int i = 0; i < FN; ++i) rw[i] = load_frag(gw[i] + k, gw_ok[i] && kok);
#pragma unroll
    for (int i = 0; i < FM; ++i) ra[i] = load_frag(ga[i] + k, ga_ok[i] && kok);
  };
  auto lstore = [&](int buf) {
    unsigned char* base = lds + buf * BUF_BYTES;
    const int col = (c16 ^ (lrow & 7)) * 16;
#pragma unroll
    for (int i = 0; i < FN; ++i) *reinterpret_cast<frag_t*>(base + (lrow + 32 * i) * T_ROWB + col) = rw[i];
#pragma unroll
    for (int i = 0; i < FM; ++i) *reinterpret_cast<frag_t*>(base + W_BYTES + (lrow + 32 * i) * T_ROWB + col) = ra[i];
  };

  f32x4 acc[FN][FM], total[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

  gload(0);
  lstore(0);
  __syncthreads();

  for (int kt = 0; kt < ntiles; ++kt) {
    const unsigned char* base = lds + (kt & 1) * BUF_BYTES;
    if (kt + 1 < ntiles) gload(kt + 1);
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      frag_t wf[FN], af[FM];
      const int col = ((s * 4 + kg) ^ (r16 & 7)) * 16;
#pragma unroll
      for (int i = 0; i < FN; ++i)
        wf[i] = *reinterpret_cast<const frag_t*>(base + (wn * 16 * FN + i * 16 + r16) * T_ROWB + col);
#pragma unroll
      for (int j = 0; j < FM; ++j)
        af[j] = *reinterpret_cast<const frag_t*>(base + W_BYTES + (wm * 16 * FM + j * 16 + r16) * T_ROWB + col);
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) acc[i][j] = mma_slab(wf[i], af[j], acc[i][j]);
    }
    if ((kt + 1) % T_CHUNK_TILES == 0 || kt + 1 == ntiles) {
#pragma unroll
      for (int i = 0; i < FN; ++i)
#pragma unroll
        for (int j = 0; j < FM; ++j) {
          total[i][j].x = total[i][j].x + acc[i][j].x;
          total[i][j].y = total[i][j].y + acc[i][j].y;
          total[i][j].z = total[i][j].z + acc[i][j].z;
          total[i][j].w = total[i][j].w + acc[i][j].w;
          acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }
    if (kt + 1 < ntiles) lstore((kt & 1) ^ 1);
    __syncthreads();
  }

#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j)
      store_out4(out, ldo, m_blk + wm * 16 * FM + j * 16 + r16, n_blk + wn * 16 * FN + i * 16 + 4 * kg, M, N,
                 total[i][j], out_form);
}

template <int FN, int FM>
static int launch_tiled(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo,
                        int form, hipStream_t st) {
  constexpr int BN = 32 * FN, BM = 32 * FM;
  const size_t smem = 2 * (size_t)(BN + BM) * T_ROWB;
  static bool configured = false;
  if (!configured) {
    if (smem > 48 * 1024)
      (void)hipFuncSetAttribute((const void*)gemm_tiled_kernel<FN, FM>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)smem);
    configured = true;
  }
  dim3 grid((N + BN - 1) / BN, (M + BM - 1) / BM);
  VK_REQUIRE(grid.y <= 65535, "gemm: too many rows (%d)", M);
  gemm_tiled_kernel<FN, FM><<<grid, 256, smem, st>>>(out, act, w, M, N, K, lda, ldo, form);
  return vk_check_launch("gemm_tiled");
}

// --------------------------------------------------------------- pipelined
// The tiled kernel for K a multiple of 64 bytes-per-row tiles (two slabs), with
// what the other lacks to keep the MFMA units fed: tiles go from global memory
// straight into LDS (global_load_lds_dwordx4, no registers in between) and S
// stages are in flight, so a tile's latency is hidden behind the S-1 tiles
// computed meanwhile.  One barrier per K tile.  Rows beyond N or M are clamped
// (their results are dropped).  Same tile shape, swizzle and reduction order as
// gemm_tiled_kernel<4, 4>.
// With SWIGLU the weight holds N gate rows, then N up rows, and the output has N columns: a workgroup
// takes 64 gate rows and the matching 64 up rows as its 128 weight rows (the waves with wn = 0 the
// gate, those with wn = 1 the up projection), and at the end the up values pass through LDS to the
// waves that hold the gate values, which write  silu(g) * u  with g and u rounded to the element type
// first: the bits of the plain projection followed by swiglu_kernel.
// FNW: 16-row weight fragments per wave, 2 to 5: a workgroup takes 32 FNW weight rows.  4 is the square tile; 2
// gives twice the workgroups, for grids that would leave compute units with one workgroup or none; 3 and 5 are
// for grids whose last round of workgroups would otherwise run nearly empty (pipe_fragments_by_rounds).  Six
// would need more than the 256 registers of a wave.
// NWN: waves along the weight rows, two of a workgroup of four waves or four of eight, which takes 64 FNW weight rows.
// A lane's offset from its block's first row is of 32 bits: rows_far says which rows are too far apart for that.
// GROUPED: block_weights, row_pair and act_row count.
template <int S, bool WHOLE, bool SWIGLU, int FNW = 4, int NWN = 2, bool GROUPED = false>
__global__ __launch_bounds__(128 * NWN, NWN == 2 ? 2 : 1) void gemm_pipe_kernel(elem_t* __restrict__ out, const elem_t* __restrict__ act,
                                                        const elem_t* __restrict__ w, int M, int N, int K,
                                                        int64_t lda, int64_t ldo, int out_form, int band_w,
                                                        const int32_t* __restrict__ block_weights, int64_t weights_stride,
                                                        const int32_t* __restrict__ row_pair, const int32_t* __restrict__ act_row) {
  static_assert(FNW >= 2 && FNW <= 5 && (FNW == 4 || !SWIGLU), "two to five weight fragments per wave; four with SwiGLU");
  static_assert(NWN == 2 || (NWN == 4 && !SWIGLU), "two waves or four along the weight rows");
  constexpr int BN = 16 * FNW * NWN;                    // weight rows of the workgroup
  constexpr int NA = 8 / NWN, PER_TILE = FNW + NA;      // loads of activation rows, and all loads, per K tile and wave
  constexpr int W_BYTES = BN * T_ROWB, STAGE_BYTES = W_BYTES + 128 * T_ROWB;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];   // [stage][w tile, act tile]

  // The wave number as a scalar: what depends on it alone (LDS addresses, which rows a load brings)
  // then needs no vector registers.
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int wn = wave % NWN, wm = wave / NWN;
  // Workgroups start in the order of their linear index.  That order walks bands of band_w column
  // blocks: all row blocks of a band before the next band, so that a band's weights are read from HBM
  // once and found in the caches by the other row blocks (a matrix larger than the memory-side cache
  // would otherwise be streamed once per row block).
  int nb = blockIdx.x, mb = blockIdx.y;
  if (band_w < (int)gridDim.x) {
    const int lin = blockIdx.y * gridDim.x + blockIdx.x;
    const int per_band = band_w * gridDim.y;
    const int band = lin / per_band, r = lin - band * per_band;
    const int w_here = min(band_w, (int)gridDim.x - band * band_w);
    mb = r / w_here;
    nb = band * band_w + (r - mb * w_here);
  }
  // A grouped product: every block of 128 rows has a weight matrix of its own, block_weights[mb] of several that lie
  // weights_stride elements apart (a negative number: the block is not in use).
  if constexpr (GROUPED) {
    const int which = block_weights[mb];
    if (which < 0) return;
    w += (int64_t)which * weights_stride;
  }
  const int n_blk = nb * (SWIGLU ? 64 : BN), m_blk = mb * 128;
  const int ntiles = K / (2 * VK_SLAB);
  // A wave without rows (the second half of a group's last block of up to 64 rows: rows without a pair come last in a group) helps to
  // bring the tiles in and leaves the matrix unit to the others.
  const bool idle = GROUPED && NWN == 4 && row_pair != nullptr && wm == 1 && row_pair[m_blk + 64] < 0;

  // A wave-level load moves 8 rows x 128 bytes; lane i fills LDS slot i of the 1 KB block, which is
  // row i/8, physical 16-byte column i%8, i.e. logical column (i%8) ^ (i/8).
  const int lr = lane >> 3, lc = (lane & 7) ^ lr;
  // A load's address is a base that is the same for the whole workgroup (the first weight row of the
  // block, or of its up rows; the first activation row), which advances along K as a scalar, plus a
  // 32-bit offset per lane that never changes: no vector arithmetic per load.
  const unsigned char* wbase = reinterpret_cast<const unsigned char*>(w + (int64_t)min(n_blk, N - 1) * K);
  const unsigned char* ubase = reinterpret_cast<const unsigned char*>(w + (int64_t)(N + min(n_blk, N - 1)) * K);   // SWIGLU: the up rows
  // act_row: a row of the product is a row of act that the table names (below 2^31 bytes from act's first: the caller's rule).
  const bool named = GROUPED && act_row != nullptr;
  const int first_row = named ? 0 : min(m_blk, M - 1);
  auto act_off = [&](int r, int col) {         // of entry `col` of the block's row r, in bytes from the base
    const int row = min(m_blk + r, M - 1);
    return (unsigned)(((int64_t)((named ? act_row[row] : row) - first_row) * lda + col) * (int64_t)sizeof(elem_t));
  };
  const unsigned char* abase = reinterpret_cast<const unsigned char*>(act + (int64_t)first_row * lda);
  unsigned offw[FNW], offa[NA];
#pragma unroll
  for (int j = 0; j < FNW; ++j) {
    const int row = (wave * FNW + j) * 8 + lr;
    const int local = SWIGLU ? (row < 64 ? row : row - 64) : row;                 // row of the block, gate or up
    const int clamped = min(n_blk + local, N - 1) - min(n_blk, N - 1);
    offw[j] = (unsigned)(((int64_t)clamped * K + lc * VK_VEC) * (int64_t)sizeof(elem_t));
  }
#pragma unroll
  for (int j = 0; j < NA; ++j) offa[j] = act_off((wave * NA + j) * 8 + lr, lc * VK_VEC);
  const unsigned lds0 = lds_offset_of(lds);
  auto issue = [&](int kt) {                 // PER_TILE loads per wave
    const unsigned base = lds0 + (kt % S) * STAGE_BYTES;
    const int64_t kb = (int64_t)kt * 2 * VK_SLAB * (int64_t)sizeof(elem_t);
#pragma unroll
    for (int j = 0; j < FNW; ++j) {
      const bool up = SWIGLU && (wave * FNW + j) * 8 >= 64;       // a scalar: all eight rows of a load are of one kind
      pipe_load_to_lds16_sv((up ? ubase : wbase) + kb, offw[j], base + (wave * FNW + j) * 8 * T_ROWB);
    }
#pragma unroll
    for (int j = 0; j < NA; ++j) pipe_load_to_lds16_sv(abase + kb, offa[j], base + W_BYTES + (wave * NA + j) * 8 * T_ROWB);
  };

  f32x4 acc[FNW][4], total[FNW][4];
#pragma unroll
  for (int i = 0; i < FNW; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

#pragma unroll
  for (int p = 0; p < S - 1; ++p)
    if (p < ntiles) issue(p);
  if (idle) {
    for (int kt = 0; kt < ntiles; ++kt) {
      if (S == 2 || kt + 1 == ntiles) wait_vmcnt_n<0>();
      else if (S == 3 || kt + 2 == ntiles) wait_vmcnt_n<PER_TILE>();
      else wait_vmcnt_n<2 * PER_TILE>();
      __syncthreads();
      if (kt + S - 1 < ntiles) issue(kt + S - 1);
    }
    return;
  }

  auto step = [&](int kt) {
    // Tile kt has landed once at most the loads of the tiles after it are outstanding (PER_TILE per tile and wave).
    const int later = min(S - 2, ntiles - 1 - kt);
    if (later == 0) wait_vmcnt_n<0>();
    else if (later == 1) wait_vmcnt_n<PER_TILE>();
    else wait_vmcnt_n<2 * PER_TILE>();
    __syncthreads();       // every wave's part of tile kt is there; everyone is done with tile kt-1's buffer
    if (kt + S - 1 < ntiles) issue(kt + S - 1);
    const unsigned char* base = lds + (kt % S) * STAGE_BYTES;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      frag_t wf[FNW], af[4];
      const int col = ((s * 4 + kg) ^ (r16 & 7)) * 16;
#pragma unroll
      for (int i = 0; i < FNW; ++i) wf[i] = *reinterpret_cast<const frag_t*>(base + (wn * 16 * FNW + i * 16 + r16) * T_ROWB + col);
#pragma unroll
      for (int i = 0; i < 4; ++i) af[i] = *reinterpret_cast<const frag_t*>(base + W_BYTES + (wm * 64 + i * 16 + r16) * T_ROWB + col);
#pragma unroll
      for (int i = 0; i < FNW; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = mma_slab(wf[i], af[j], acc[i][j]);
    }
#ifdef VK_BF16
    // Order for the scheduler: the first slab's reads, then the second slab's reads one by one between
    // the first slab's MFMAs, so that they return while the matrix unit works.
    constexpr int BETWEEN = FNW >= 4 ? 2 : 1;                    // MFMAs between two of the second slab's reads
    __builtin_amdgcn_sched_group_barrier(0x100, FNW + 4, 0);     // the first slab's LDS reads
#pragma unroll
    for (int q = 0; q < FNW + 4; ++q) {
      __builtin_amdgcn_sched_group_barrier(0x008, BETWEEN, 0);            // MFMA
      __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                  // 1 LDS read
    }
    __builtin_amdgcn_sched_group_barrier(0x008, 8 * FNW - (FNW + 4) * BETWEEN, 0);   // the first slab's other MFMAs and the second slab's
#endif
  };
  auto close_chunk = [&]() {
#pragma unroll
    for (int i = 0; i < FNW; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        total[i][j].x = total[i][j].x + acc[i][j].x;
        total[i][j].y = total[i][j].y + acc[i][j].y;
        total[i][j].z = total[i][j].z + acc[i][j].z;
        total[i][j].w = total[i][j].w + acc[i][j].w;
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  if (WHOLE) {
    // K is whole chunks: the tiles of a chunk are written out one after the other, so that the chunk
    // sums are touched between chunks only and need not move between register files in every tile.
    for (int kt0 = 0; kt0 < ntiles; kt0 += T_CHUNK_TILES) {
#pragma unroll
      for (int u = 0; u < T_CHUNK_TILES; ++u) step(kt0 + u);
      close_chunk();
    }
  } else {
    for (int kt = 0; kt < ntiles; ++kt) {
      step(kt);
      if ((kt + 1) % T_CHUNK_TILES == 0 || kt + 1 == ntiles) close_chunk();
    }
  }

  if constexpr (SWIGLU) {
    // The two waves of a row block split the 64 output columns: the gate wave keeps columns 0..31 and
    // gets their up values, the up wave keeps columns 32..63 and gets their gate values.
    __syncthreads();            // the last tile has been read: LDS is free
    // [128 rows][16 groups of 4 columns]; a row's group g lies at place g ^ (row % 16), so that the 16 rows a
    // wave touches at once (256 bytes apart: the same banks) spread over all banks.
    f32x4* ex = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4& v = total[i][j];
        v.x = round_to_elem(v.x); v.y = round_to_elem(v.y); v.z = round_to_elem(v.z); v.w = round_to_elem(v.w);
        if ((i < 2) == (wn == 1)) ex[(wm * 64 + j * 16 + r16) * 16 + ((i * 4 + kg) ^ r16)] = v;    // what the other wave needs
      }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if ((i < 2) != (wn == 0)) continue;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const f32x4 o = ex[(wm * 64 + j * 16 + r16) * 16 + ((i * 4 + kg) ^ r16)];
        const f32x4 g = wn == 0 ? total[i][j] : o, u = wn == 0 ? o : total[i][j];
        f32x4 y;
        y.x = (g.x * (1.0f / (1.0f + expf(-g.x)))) * u.x;
        y.y = (g.y * (1.0f / (1.0f + expf(-g.y)))) * u.y;
        y.z = (g.z * (1.0f / (1.0f + expf(-g.z)))) * u.z;
        y.w = (g.w * (1.0f / (1.0f + expf(-g.w)))) * u.w;
        store_out4(out, ldo, m_blk + wm * 64 + j * 16 + r16, n_blk + i * 16 + 4 * kg, M, N, y, out_form);
      }
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < FNW; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      store_out4(out, ldo, m_blk + wm * 64 + j * 16 + r16, n_blk + wn * 16 * FNW + i * 16 + 4 * kg, M, N, total[i][j],
                 out_form);
}

// Column blocks of a band in the tile kernel (0: no bands).  64: the 512 workgroups that run at a time
// then are 8 row blocks of 64 column blocks, and the 64 of them on a chip part (workgroup i runs on part
// i % 8) are 8 row blocks of 8 column blocks: the fewest distinct tiles for its cache.  Measured on
// MI355X, gate/up with SwiGLU at 2,048 to 8,192 rows: 12,288 x 4,096 weights 950 -> 1,090 TFLOP/s,
// 25,600 x 5,120 (524 MB, more than the memory-side cache holds) 600 -> 1,040; 51 or 76 column blocks,
// which move a column block from part to part, 780 to 830.
static const int pipe_band_blocks = 64;

// Whether a grouped product of 16-bit elements and K in whole chunks goes by workgroups of 256 weight rows (launch_pipe) or of 128.
// The wide ones have one workgroup a compute unit, so that a launch of few is one round half empty where the narrow ones have two a unit,
// or one with four stages (at most one a unit: 896 sizes of 4 to 64 matrices of 20 to 200 rows, most of them wide before, 26.5 -> 23.0 ms, 22.7 with the better of
// the two everywhere); and a column block that lands on another chip part with each row block (columns that are no multiple of eight, up to 16)
// has its weights read by several.  But up to about 60 rows a matrix (M and the matrices tell: a matrix has up to 127 rows of padding)
// half of most blocks is idle, which only the wide ones leave out.  Measured on MI355X in recorded launches with the weights of
// several layers in turn, 947 sizes of 2 to 64 matrices, 40 to 4,096 tokens, rows named, narrow against wide, us: 32 matrices, 4 choices, 257
// tokens 1,536 x 1,024 25.8, 22.9; 2,048 tokens 1,536 x 1,024 50.5, 57.6, 3,072 x 2,048 163, 165, 6,144 x 4,096 594, 542; 8 matrices, 2 choices,
// 257 tokens 512 x 512 8.7, 11.7.  Rows as they lie are read by more workgroups of the narrow kernel: 2,048 tokens,
// 768 x 1,024 42.4, 35.9.  Slower by more than 3 % than the better of the two: 82 sizes, as they
// lie 94; the wide ones alone 415 and 353, the narrow ones 336 and 419.
static bool grouped_wide(int M, int N, int matrices, bool named) {
  const int64_t columns = (N + 255) / 256, groups = columns * (M / 128);
  if ((N + 127) / 128 * (int64_t)(M / 128) <= vk_device_cus()) return false;
  if (matrices > 0 && (int64_t)M + 127 <= (int64_t)matrices * (127 + 60)) return true;
  if (columns % 8 == 0 || columns > 16) return 8 * groups >= 5 * vk_device_cus();
  return !named && columns <= 4 && 2 * groups >= vk_device_cus();
}

static bool rows_far(int64_t lda, int rows = 128) { return ((rows - 1) * lda + 2 * VK_SLAB) * (int64_t)sizeof(elem_t) > (int64_t)UINT32_MAX; }

template <int S, bool SWIGLU = false, int FNW = 4, bool GROUPED = false>
static int launch_pipe(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo,
                       int form, hipStream_t st, const int32_t* block_weights = nullptr, int64_t weights_stride = 0,
                       const int32_t* row_pair = nullptr, const int32_t* act_row = nullptr, int matrices = 0) {
  constexpr int BN = SWIGLU ? 64 : 32 * FNW;                         // output columns of a workgroup
  static_assert(S >= 2 && S <= 4, "the waits count up to two tiles behind the next");
  const size_t smem = (size_t)S * (32 * FNW + 128) * T_ROWB;         // also holds the 32 KB that SWIGLU passes between waves
  static bool configured = false;
  if (!configured) {
    (void)hipFuncSetAttribute((const void*)gemm_pipe_kernel<S, true, SWIGLU, FNW, 2, GROUPED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    (void)hipFuncSetAttribute((const void*)gemm_pipe_kernel<S, false, SWIGLU, FNW, 2, GROUPED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    configured = true;
  }
  dim3 grid((N + BN - 1) / BN, (M + 127) / 128);
  VK_REQUIRE(grid.y <= 65535, "gemm: too many rows (%d)", M);
  if constexpr (GROUPED && sizeof(elem_t) == 2) {
    // A grouped product is bound by its weights' way from memory: an expert's matrix serves two or three blocks of rows where a dense
    // product's serves all of them.  Workgroups of 256 weight rows (eight waves) with three stages have two tiles of 48 KB on their way
    // a compute unit where two workgroups of 128 with two stages have two of 32, and 16 column blocks of all row blocks before the next
    // 16 keep the blocks of an expert together in time and on their chip part.  Measured on MI355X, 32 experts, before and after with the
    // idle waves: 2,048 tokens x 3 choices, 6,144 x 4,096 weights 548 -> 484 us, 4,096 x 3,072 290 -> 241; 2,445 x 4, 6,144 x 4,096 690 ->
    // 615; 700 x 3 394 -> 339; 1,360 x 3, 4,608 x 4,096 367 -> 327.  (Touching the weights' lines two to
    // eight tiles ahead instead: 548 -> 586 to 699.)
    if (K % KC == 0 && grouped_wide(M, N, matrices, act_row != nullptr)) {
      constexpr size_t wide_smem = (size_t)3 * (256 + 128) * T_ROWB;
      static bool wide = false;
      if (!wide) {
        (void)hipFuncSetAttribute((const void*)gemm_pipe_kernel<3, true, false, 4, 4, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)wide_smem);
        wide = true;
      }
      const dim3 wgrid((N + 255) / 256, grid.y);
      gemm_pipe_kernel<3, true, false, 4, 4, true><<<wgrid, 512, wide_smem, st>>>(out, act, w, M, N, K, lda, ldo, form, wgrid.x > 16 ? 16 : (int)wgrid.x, block_weights,
                                                                              weights_stride, row_pair, act_row);
      return vk_check_launch("gemm_pipe (grouped)");
    }
  }
  // No more workgroups than compute units: four stages (pipe_fragments_in_one_round says why).
  if constexpr (S == 2 && (SWIGLU || GROUPED)) {
    if ((int64_t)grid.x * grid.y <= vk_device_cus())
      return launch_pipe<4, SWIGLU, FNW, GROUPED>(out, act, w, M, N, K, lda, ldo, form, st, block_weights, weights_stride, row_pair, act_row, matrices);
  }
  const int band_w = (pipe_band_blocks > 0 && grid.y > 1 && (int)grid.x > pipe_band_blocks) ? pipe_band_blocks : (int)grid.x;
  if (K % KC == 0) gemm_pipe_kernel<S, true, SWIGLU, FNW, 2, GROUPED><<<grid, 256, smem, st>>>(out, act, w, M, N, K, lda, ldo, form, band_w, block_weights, weights_stride, row_pair, act_row);
  else gemm_pipe_kernel<S, false, SWIGLU, FNW, 2, GROUPED><<<grid, 256, smem, st>>>(out, act, w, M, N, K, lda, ldo, form, band_w, block_weights, weights_stride, row_pair, act_row);
  return vk_check_launch("gemm_pipe");
}

#ifdef VK_F32
// ------------------------------------------------------------ 32-bit tiles
// The tile kernel of 32-bit elements: K in whole pairs of slabs, 32 FM activation rows and 32 FN weight rows a workgroup of four waves (SWIGLU: 16 FN gate rows and
// their up rows, which the same wave multiplies), S stages.  Operand roles, reduction order and bits are those of gemm_tiled_kernel.
//
// What bounds it: the 32-bit matrix instruction takes 32 clocks for 2 KB of operands, so that LDS and caches are idle most of the time even with tiles of 32 x 64,
// and what a launch loses are rows of padding and the compute units that wait for the ones with a tile more.  Tiles of 128 x 128 (gemm_pipe_kernel, before) at 651 rows are 6 x 96 for
// gate/up of 6,144 x 2,048: 15 % of the rows are padding, and 576 tiles are three for some of 256 units.  Here the tile is chosen for the launch (fine_tile).  Measured on
// MI355X in recorded launches with the weights of several layers in turn, before and after, us: 651 rows, gate/up with SwiGLU 6,144 x 2,048 366 -> 260 (126 TFLOP/s), 2,048 x 6,144
// 220 -> 157, 4,096 x 2,048 126 -> 96, 2,048 x 2,048 78 -> 57; 217 rows, 3,072 x 1,024 with SwiGLU 72 -> 31, 1,024 x 3,072 69 -> 30; 434 rows, 1,024 x 1,024 40 -> 15; 2,048 rows,
// 6,144 x 2,048 721 -> 714.  The four instructions of a slab go round the tile's fragments, so that none waits for the one before it.
template <int FM, int FN, int S, bool SWIGLU, bool WHOLE>
__global__ __launch_bounds__(256) void gemm_fine_kernel(elem_t* __restrict__ out, const elem_t* __restrict__ act, const elem_t* __restrict__ w, int M, int N, int K,
                                                        int64_t lda, int64_t ldo, int out_form, int row_blocks) {
  static_assert(!SWIGLU || FN % 2 == 0, "as many gate as up fragments a wave");
  constexpr int BM = 32 * FM, BN = 32 * FN, COLS = SWIGLU ? BN / 2 : BN;
  constexpr int W_BYTES = BN * T_ROWB, STAGE_BYTES = W_BYTES + BM * T_ROWB;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];      // [S][weights, activations]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kg = lane >> 4, wn = wave & 1, wm = wave >> 1;
  const int lin = blockIdx.x, tiles = gridDim.x, part = lin & 7;
  const int tile = part * (tiles >> 3) + min(part, tiles & 7) + (lin >> 3);
  const int per_band = 8 * row_blocks, band = tile / per_band, at = tile - band * per_band;
  const int wide = min(8, (N + COLS - 1) / COLS - band * 8);
  const int mb = at / wide, nb = band * 8 + (at - mb * wide);
  const int n_blk = nb * COLS, m_blk = mb * BM, ntiles = K / (2 * VK_SLAB);

  const int lr = lane >> 3, lc = (lane & 7) ^ lr;
  const unsigned char* wbase = reinterpret_cast<const unsigned char*>(w + (int64_t)n_blk * K);
  const unsigned char* ubase = reinterpret_cast<const unsigned char*>(w + (int64_t)(N + n_blk) * K);
  const unsigned char* abase = reinterpret_cast<const unsigned char*>(act + (int64_t)m_blk * lda);
  unsigned offw[FN], offa[FM];
#pragma unroll
  for (int j = 0; j < FN; ++j) {
    const int row = (wave * FN + j) * 8 + lr;                              // of the workgroup's weight rows; a wave along them has 16 FN
    const int of_wave = row / (16 * FN), in = row - of_wave * 16 * FN;
    const int local = SWIGLU ? of_wave * 8 * FN + in % (8 * FN) : row;     // gate rows first, then their up rows
    offw[j] = (unsigned)(((int64_t)(min(n_blk + local, N - 1) - n_blk) * K + lc * VK_VEC) * (int64_t)sizeof(elem_t));
  }
#pragma unroll
  for (int j = 0; j < FM; ++j)
    offa[j] = (unsigned)(((int64_t)(min(m_blk + (wave * FM + j) * 8 + lr, M - 1) - m_blk) * lda + lc * VK_VEC) * (int64_t)sizeof(elem_t));
  const unsigned lds0 = lds_offset_of(lds);
  auto issue = [&](int kt) {
    const unsigned base = lds0 + (kt % S) * STAGE_BYTES;
    const int64_t kb = (int64_t)kt * T_ROWB;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const bool up = SWIGLU && ((wave * FN + j) * 8) % (16 * FN) >= 8 * FN;
      pipe_load_to_lds16_sv((up ? ubase : wbase) + kb, offw[j], base + (wave * FN + j) * 8 * T_ROWB);
    }
#pragma unroll
    for (int j = 0; j < FM; ++j) pipe_load_to_lds16_sv(abase + kb, offa[j], base + W_BYTES + (wave * FM + j) * 8 * T_ROWB);
  };
  f32x4 acc[FN][FM], total[FN][FM];
#pragma unroll
  for (int i = 0; i < FN; ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < S - 1; ++p)
    if (p < ntiles) issue(p);
  auto step = [&](int kt) {
    // Tile kt has landed once at most the loads of the tiles after it are outstanding.
    const int later = min(S - 2, ntiles - 1 - kt);
    if (later <= 0) wait_vmcnt_n<0>();
    else if (later == 1) wait_vmcnt_n<FM + FN>();
    else wait_vmcnt_n<2 * (FM + FN)>();
    __syncthreads();
    if (kt + S - 1 < ntiles) issue(kt + S - 1);
    const unsigned char* base = lds + (kt % S) * STAGE_BYTES;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      frag_t wf[FN], af[FM];
      const int col = ((s * 4 + kg) ^ (r16 & 7)) * 16;
#pragma unroll
      for (int i = 0; i < FN; ++i) wf[i] = *reinterpret_cast<const frag_t*>(base + (wn * 16 * FN + i * 16 + r16) * T_ROWB + col);
#pragma unroll
      for (int i = 0; i < FM; ++i) af[i] = *reinterpret_cast<const frag_t*>(base + W_BYTES + (wm * 16 * FM + i * 16 + r16) * T_ROWB + col);
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < FN; ++i)
#pragma unroll
          for (int j = 0; j < FM; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wf[i][e], af[j][e], acc[i][j], 0, 0, 0);
    }
  };
  auto close_chunk = [&]() {
#pragma unroll
    for (int i = 0; i < FN; ++i)
#pragma unroll
      for (int j = 0; j < FM; ++j) {
        total[i][j].x = total[i][j].x + acc[i][j].x;
        total[i][j].y = total[i][j].y + acc[i][j].y;
        total[i][j].z = total[i][j].z + acc[i][j].z;
        total[i][j].w = total[i][j].w + acc[i][j].w;
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  };
  // K not in whole chunks: whole ones first and what is left after them.  (Asking every tile whether it ends a chunk takes 3 to 12 % longer, 2,048 rows, 2,048 x 2,080 145 -> 130 us;
  // but with the two products of 1 x 2 fragments 2 to 7 % less.)
  constexpr bool ASK = !WHOLE && FM * FN == 2;
  const int whole = WHOLE ? ntiles : ASK ? 0 : ntiles - ntiles % T_CHUNK_TILES;
  for (int kt0 = 0; kt0 < whole; kt0 += T_CHUNK_TILES) {
#pragma unroll 2
    for (int u = 0; u < T_CHUNK_TILES; ++u) step(kt0 + u);
    close_chunk();
  }
  if (!WHOLE) {
    for (int kt = whole; kt < ntiles; ++kt) {
      step(kt);
      if ((ASK && (kt + 1) % T_CHUNK_TILES == 0) || kt + 1 == ntiles) close_chunk();
    }
  }
  const int m0 = m_blk + wm * 16 * FM + r16, n0 = n_blk + wn * (SWIGLU ? 8 : 16) * FN + 4 * kg;
#pragma unroll
  for (int i = 0; i < (SWIGLU ? FN / 2 : FN); ++i)
#pragma unroll
    for (int j = 0; j < FM; ++j) {
      f32x4 y = total[i][j];
      if constexpr (SWIGLU) {
#pragma unroll
        for (int e = 0; e < 4; ++e) y[e] = (y[e] * (1.0f / (1.0f + expf(-y[e])))) * total[i + FN / 2][j][e];
      }
      store_out4(out, ldo, m0 + j * 16, n0 + i * 16, M, N, y, out_form);
    }
}

template <int FM, int FN, int S, bool SWIGLU>
static int launch_fine(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int form, hipStream_t st) {
  constexpr int COLS = SWIGLU ? 16 * FN : 32 * FN;
  constexpr size_t smem = (size_t)S * 32 * (FM + FN) * T_ROWB;
  static_assert(S >= 2 && S <= 4, "the waits count up to two tiles behind the next");
  static bool configured = false;
  if (!configured) {
    (void)hipFuncSetAttribute((const void*)gemm_fine_kernel<FM, FN, S, SWIGLU, true>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    (void)hipFuncSetAttribute((const void*)gemm_fine_kernel<FM, FN, S, SWIGLU, false>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    configured = true;
  }
  const int row_blocks = (M + 32 * FM - 1) / (32 * FM);
  const int64_t tiles = (int64_t)row_blocks * ((N + COLS - 1) / COLS);
  VK_REQUIRE(tiles < (1 << 30), "gemm: too many rows (%d)", M);
  if (K % KC == 0) gemm_fine_kernel<FM, FN, S, SWIGLU, true><<<(unsigned)tiles, 256, smem, st>>>(out, act, w, M, N, K, lda, ldo, form, row_blocks);
  else gemm_fine_kernel<FM, FN, S, SWIGLU, false><<<(unsigned)tiles, 256, smem, st>>>(out, act, w, M, N, K, lda, ldo, form, row_blocks);
  return vk_check_launch("gemm_fine");
}
static int gemm_fine(int fm, int fn, bool swiglu, elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int form,
                     hipStream_t st) {
#define FINE(FM, FN) if (fm == FM && fn == FN) return swiglu ? launch_fine<FM, FN, 2, true>(out, act, w, M, N, K, lda, ldo, form, st) : launch_fine<FM, FN, 2, false>(out, act, w, M, N, K, lda, ldo, form, st)
  if (fm == 1 && fn == 1 && !swiglu) return launch_fine<1, 1, 3, false>(out, act, w, M, N, K, lda, ldo, form, st);
  FINE(1, 2);
  FINE(2, 2);
  FINE(3, 2);
  FINE(1, 4);
  FINE(2, 4);
#undef FINE
  return vk_fail("gemm: no tile of %d by %d fragments", fm, fn);
}
#endif

#ifdef VK_BF16
// ------------------------------------------------------------- alternating
// Tiles of 256 activation rows and 32 FNW weight rows, eight waves, a workgroup a compute unit: 16-bit elements, K in whole chunks, at least
// a tile's rows of both.  A wave has 64 activation rows and 16 FNW weight rows, in two groups of four waves, one of each a SIMD.  The groups
// take turns: while one multiplies a slab (4 FNW MFMAs a wave), the other fetches its next slab's fragments from LDS, and a barrier
// swaps them, so that a SIMD's matrix unit always has a wave whose operands are in registers.  SA (SW) K tiles of two slabs of activations (weights)
// lie in LDS or are on their way there straight from global memory, brought by group 0 (1); a tile's place is refilled as soon as both groups have
// read it.  The last block of rows or columns starts early enough to be whole: what it shares with the one before is computed twice and stored
// twice with the same bits.  Reduction order, operand roles and bits are those of gemm_pipe_kernel.
//
// What bounds it: the tile kernel asks the second-level cache for 32 KB per 2.1 MFLOP, which alone takes it 45 % of its time; 256 x 192 asks
// for 19 KB.  (256 x 256 would need 512 KB of registers for chunk sums and totals, all that a compute unit has.)  Without loads from global
// memory this kernel reaches 1,430 TFLOP/s, which is near what the chip sustains of these MFMAs (1,640).  Measured on MI355X with the weights
// of several layers in turn, tile kernel against this one, us: gate/up with SwiGLU 12,288 x 4,096, 2,048 rows 404 -> 349 (1,180 TFLOP/s), 4,096
// rows 741 -> 646 (1,280); 4,096 x 12,288, 2,048 rows 189 -> 169, 4,096 rows 364 -> 322; 6,144 x 4,096, 2,048 rows 108 -> 93; 5,120 x
// 17,408, 3,900 rows 633 -> 540 (1,290).  Over 920 sizes of 256 to 4,096 rows, weights from memory, 515 take it, 114.6 -> 104.0 ms in all (103.8 with
// the better kernel at every size).  Three of them are 5 to 8 % slower than the tile kernel (850 to 1,024 rows, 6,144 x 2,560: 38 to 39 us against 41,
// where 96 columns fill exactly one round of that), one 5 % (850 rows, 16,384 x 4,096), six 2 to 3 %; a rule that leaves these to the tile kernel
// gives up as much at others (1,300 rows, 4,096 x 2,048: 32.5 -> 30.7).
// Tried: K tiles of one slab (rows of 64 bytes, five places: half of every line that the cache sends is not asked for, 162 -> 190 us at 4,096
// rows, 6,144 x 4,096); a slab's activations read a phase ahead (5 to 15 % slower); a tile's loads in quarters, also between the MFMAs (4 %
// slower than in halves).
__device__ __forceinline__ void al_barrier() { asm volatile("s_barrier" ::: "memory"); }

template <int FNW, int SA, int SW, bool SWIGLU>
__global__ __launch_bounds__(512, 2) void gemm_alternate_kernel(elem_t* __restrict__ out, const elem_t* __restrict__ act, const elem_t* __restrict__ w,
                                                                int M, int N, int K, int64_t lda, int64_t ldo, int out_form, int row_blocks) {
  static_assert(!SWIGLU || FNW % 2 == 0, "as many gate as up fragments a wave");
  constexpr int BM = 256, BN = 32 * FNW, COLS = SWIGLU ? BN / 2 : BN;
  constexpr int A_BYTES = BM * T_ROWB, W_BYTES = BN * T_ROWB;
  constexpr int LA = BM / 32, LW = BN / 32;                // loads of 8 rows a wave and K tile: group 0's, group 1's
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];      // [SA][256 rows], [SW][BN rows]

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int group = wave >> 2, q = wave & 3;
  // Workgroup i runs on chip part i % 8.  A part takes consecutive tiles of an order that walks bands of eight column blocks, all row blocks of
  // a band before the next: the 32 tiles that a part works on at a time are four row blocks by eight column blocks (the fewest distinct rows
  // for its cache, whatever the numbers of blocks), and a band's weights come from HBM for one part or two.
  const int lin = blockIdx.x, tiles = gridDim.x, part = lin & 7;
  const int tile = part * (tiles >> 3) + min(part, tiles & 7) + (lin >> 3);
  const int per_band = 8 * row_blocks, band = tile / per_band, at = tile - band * per_band;
  const int wide = min(8, (N + COLS - 1) / COLS - band * 8);
  const int mb = at / wide, nb = band * 8 + (at - mb * wide);
  const int n_blk = min(nb * COLS, N - COLS), m_blk = min(mb * BM, M - BM);

  // A wave-level load brings 8 rows of 128 bytes: lane i fills row i / 8, place i % 8, which holds the row's 16-byte column (i % 8) ^ (i / 8).
  const int lr = lane >> 3, lc = (lane & 7) ^ lr;
  const int64_t ld = group == 0 ? lda : K;
  const unsigned voff = (unsigned)((lr * ld + lc * VK_VEC) * (int64_t)sizeof(elem_t));
  // A wave's rows lie one after the other: 64 of the activations, or 8 FNW of the weights.  With SWIGLU group g's weight rows are 8 FNW of the
  // gate and their up rows: an even wave brings gate rows, an odd one up rows.
  const int64_t row0 = group == 0 ? m_blk + q * 64 : SWIGLU ? (int64_t)(q & 1) * N + n_blk + (q >> 1) * (8 * FNW) : n_blk + q * (8 * FNW);
  const unsigned char* src = reinterpret_cast<const unsigned char*>((group == 0 ? act : w) + row0 * ld);
  const int64_t step = 8 * ld * (int64_t)sizeof(elem_t);
  const unsigned lds0 = lds_offset_of(lds) + (group == 0 ? q * LA * 8 * T_ROWB : SA * A_BYTES + q * LW * 8 * T_ROWB);
  unsigned fill = 0;                                       // the place that the next K tile to be asked for takes
  // The loads FROM .. TO of a tile of group G; the tile's last ones move on to the next tile.
  auto issue = [&](auto g_, int from, int to) __attribute__((always_inline)) {
    constexpr int G = decltype(g_)::value, L = G ? LW : LA;
#pragma unroll
    for (int j = 0; j < L; ++j)
      if (j >= from && j < to) pipe_load_to_lds16_sv(src + j * step, voff, __builtin_amdgcn_readfirstlane(lds0 + fill + j * 8 * T_ROWB));
    if (to < L) return;
    src += T_ROWB;
    fill = fill == (G ? (SW - 1) * W_BYTES : (SA - 1) * A_BYTES) ? 0 : fill + (G ? W_BYTES : A_BYTES);
  };

  f32x4 acc[FNW][4], total[FNW][4];
#pragma unroll
  for (int i = 0; i < FNW; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};

  const int frag = r16 * T_ROWB + ((kg ^ (r16 & 7)) * 16);
  const int a_at = q * 64 * T_ROWB + frag, w_at = SA * A_BYTES + group * (16 * FNW) * T_ROWB + frag;
  unsigned read_a = 0, read_w = 0;
  // Slab S of a K tile of group G: the first of a chunk starts from zero; where no tile is left to ask for, all loads that still fly are waited
  // for.  A tile is asked for in two halves where three places give the second one the time.
  auto slab = [&](auto g_, int S, bool first, bool more) __attribute__((always_inline)) {
    constexpr int G = decltype(g_)::value, L = G ? LW : LA, HALF = (G ? SW : SA) > 2 ? L / 2 : L;
    // Fetch: this slab's fragments.
    frag_t af[4], wf[FNW];
#pragma unroll
    for (int j = 0; j < 4; ++j) af[j] = *reinterpret_cast<const frag_t*>(lds + (a_at ^ (S * 64)) + read_a + j * 16 * T_ROWB);
#pragma unroll
    for (int i = 0; i < FNW; ++i) wf[i] = *reinterpret_cast<const frag_t*>(lds + (w_at ^ (S * 64)) + read_w + i * 16 * T_ROWB);
    if (S == 1) {
      read_a = read_a == (SA - 1) * A_BYTES ? 0 : read_a + A_BYTES;
      read_w = read_w == (SW - 1) * W_BYTES ? 0 : read_w + W_BYTES;
    }
    if (more && S == 0) issue(g_, 0, HALF);
    if (more && S == 1 && HALF < L) issue(g_, HALF, L);
    if (G == 1 && S == 1) {                                 // the next tile's weights are there when group 0 starts on it
      if (more) wait_vmcnt_n<(SW - 2) * LW>(); else wait_vmcnt_n<0>();
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    al_barrier();
    __builtin_amdgcn_sched_barrier(0);
    // Multiply.
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < FNW; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = mma_slab(wf[i], af[j], first ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][j]);
    __builtin_amdgcn_s_setprio(0);
    __builtin_amdgcn_sched_barrier(0);
    if (G == 0 && S == 1) {
      if (more) wait_vmcnt_n<(SA - 2) * LA>(); else wait_vmcnt_n<0>();
    }
    al_barrier();
    __builtin_amdgcn_sched_barrier(0);
  };
  auto chunk = [&](auto g_, bool last) __attribute__((always_inline)) {
    constexpr int ST = decltype(g_)::value ? SW : SA;
#pragma unroll
    for (int t = 0; t < T_CHUNK_TILES; ++t) {
      const bool more = !last || t + ST - 1 < T_CHUNK_TILES;
      slab(g_, 0, t == 0, more);
      slab(g_, 1, false, more);
    }
#pragma unroll
    for (int i = 0; i < FNW; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        total[i][j].x = total[i][j].x + acc[i][j].x;
        total[i][j].y = total[i][j].y + acc[i][j].y;
        total[i][j].z = total[i][j].z + acc[i][j].z;
        total[i][j].w = total[i][j].w + acc[i][j].w;
      }
  };
  auto walk = [&](auto g_) __attribute__((always_inline)) {
    constexpr int G = decltype(g_)::value;
#pragma unroll
    for (int p = 0; p < (G ? SW : SA) - 1; ++p) issue(g_, 0, G ? LW : LA);      // K is a chunk or more: more tiles than places
    wait_vmcnt_n<G ? (SW - 2) * LW : (SA - 2) * LA>();
    al_barrier();
    if (G == 1) al_barrier();
    for (int c = 1; c < K / KC; ++c) chunk(g_, false);
    chunk(g_, true);
    if (G == 0) al_barrier();
  };
  if (group == 0) walk(std::integral_constant<int, 0>()); else walk(std::integral_constant<int, 1>());

  const int m0 = m_blk + q * 64 + r16, n0 = n_blk + group * (SWIGLU ? 8 * FNW : 16 * FNW) + 4 * kg;
  if constexpr (SWIGLU) {
#pragma unroll
    for (int i = 0; i < FNW / 2; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = round_to_elem(total[i][j][e]), u = round_to_elem(total[i + FNW / 2][j][e]);
          y[e] = (g * (1.0f / (1.0f + expf(-g)))) * u;
        }
        store_out4(out, ldo, m0 + j * 16, n0 + i * 16, M, N, y, out_form);
      }
  } else {
#pragma unroll
    for (int i = 0; i < FNW; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) store_out4(out, ldo, m0 + j * 16, n0 + i * 16, M, N, total[i][j], out_form);
  }
}

template <int FNW, int SA, int SW, bool SWIGLU = false>
static int launch_alternate(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int form, hipStream_t st) {
  constexpr int COLS = SWIGLU ? 16 * FNW : 32 * FNW;
  constexpr size_t smem = (size_t)(SA * 256 + SW * 32 * FNW) * T_ROWB;
  VK_REQUIRE(M >= 256 && N >= COLS && K % KC == 0, "gemm: the alternating kernel takes 256 rows, %d columns and whole chunks or more", COLS);
  static bool configured = false;
  if (!configured) {
    (void)hipFuncSetAttribute((const void*)gemm_alternate_kernel<FNW, SA, SW, SWIGLU>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    configured = true;
  }
  const int row_blocks = (M + 255) / 256;
  const int64_t tiles = (int64_t)row_blocks * ((N + COLS - 1) / COLS);
  VK_REQUIRE(tiles < (1 << 30), "gemm: too many rows (%d)", M);
  if (N % 4 != 0) form &= ~OUT_VEC;       // the last block of columns begins at N - COLS: four of its columns are then no aligned vector
  gemm_alternate_kernel<FNW, SA, SW, SWIGLU><<<(unsigned)tiles, 512, smem, st>>>(out, act, w, M, N, K, lda, ldo, form, row_blocks);
  return vk_check_launch("gemm_alternate");
}
#endif

#ifdef VK_BF16
// ------------------------------------------------------------ grouped, alternating
// The experts' product by a plan's order: 16-bit elements, K in whole chunks.  A workgroup takes one part of a matrix's rows, up to 192 as they are, in
// steps of 32 (FA: 16-row fragments of a wave, one to six), and 256 weight rows (GLU: 128 of the gate and their up rows), by two groups of four waves that take
// turns as in gemm_alternate_kernel: group 0 has the first half of the rows and brings the activations, group 1 the second half and brings the weights; wave q
// of either has weight rows 64 q .. 64 q + 63.  Reduction order, operand roles and bits are those of gemm_pipe_kernel.
//
// What bounds it: an expert's matrix serves one or two parts, so that weights come from memory at 4 to 5.7 TB/s, and a part's height decides how long the
// matrix unit and LDS (4 + FA fragments for 4 FA products) are busy beside that.  Blocks of 128 rows, which this replaces, multiplied up to 64 rows
// of padding a block, brought a matrix in once a block and took LDS 8 fragments for 16 products.  Parts are levelled (193 rows: 128 and 65 at
// most, not 192 and 1), up to four rows of fragments leave LDS for a fourth tile of weights, and a matrix that serves one part passes the caches by (nt: 4,608 x 4,096, 1,360 tokens x 3
// choices of 32 268 -> 242 us; with two parts a matrix 2 to 8 % slower).  The order has the tallest parts first, as the launch's last workgroups else run alone
// (309 -> 266 us there).  Parts of a matrix lie next to each other for eight column blocks at a time: workgroup i runs on chip part i % 8, whose cache
// then has a column block's weights for all parts.  (All tiles of a matrix on one chip part instead: no gain.)
// Measured on MI355X, 32 experts, random choices, gemm_pipe_kernel's blocks against this, us: 2,048 tokens x 3, 6,144 x 4,096 465 -> 400 (with the gated activation,
// a pass of its own before, 516 -> 402), 4,096 x 3,072 277 -> 206; 2,445 x 4, 6,144 x 4,096 610 -> 533, 4,096 x 3,072 334 -> 302; 2,400 x 4, 3,072 x 2,048 194 ->
// 165; 1,334 x 4, 1,536 x 2,048 86 -> 57; 700 x 3, 6,144 x 4,096 331 -> 283 (5.7 TB/s); 8 experts, 2,048 x 2, 4,096 x 3,072 154 -> 117.
struct GluArgs {
  float limit, slope, shift;
  const int32_t* row_pair;           // both or neither
  const float* wts;
};
template <bool GLU, int FA>
__device__ __forceinline__ void experts_tile(unsigned char* lds, elem_t* __restrict__ out, const elem_t* __restrict__ act, const elem_t* __restrict__ w, int M, int N, int K,
                                             int64_t lda, int64_t ldo, int out_form, int m_blk, int n_blk, bool once, const int32_t* __restrict__ act_row,
                                             const GluArgs& glu) {
  constexpr int FNW = 4, SA = FA <= 2 || FA == 5 ? 3 : 2, SW = FA <= 4 ? 4 : 3, BN = 256;
  constexpr int A_BYTES = 32 * FA * T_ROWB, W_BYTES = BN * T_ROWB;
  constexpr int LA = FA, LW = 8;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int group = wave >> 2, q = wave & 3;
  const int lr = lane >> 3, lc = (lane & 7) ^ lr;
  const unsigned lds0 = lds_offset_of(lds) + (group == 0 ? q * LA * 8 * T_ROWB : SA * A_BYTES + q * LW * 8 * T_ROWB);
  f32x4 total[FNW][FA];
#pragma unroll
  for (int i = 0; i < FNW; ++i)
#pragma unroll
    for (int j = 0; j < FA; ++j) total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int frag = r16 * T_ROWB + ((kg ^ (r16 & 7)) * 16);
  const int a_at = group * FA * 16 * T_ROWB + frag, w_at = SA * A_BYTES + q * 64 * T_ROWB + frag;

  auto walk = [&](auto g_, auto once_) __attribute__((always_inline)) {
    constexpr bool ONCE = decltype(once_)::value;
    constexpr int G = decltype(g_)::value, L = G ? LW : LA, ST = G ? SW : SA, BYTES = G ? W_BYTES : A_BYTES, HALF = ST > 2 ? (L + 1) / 2 : L;
    unsigned voff[G ? 1 : FA];
    const unsigned char* src;
    int64_t step = 0, up = 0;
    if constexpr (G == 1) {
      src = reinterpret_cast<const unsigned char*>(w + (int64_t)(n_blk + q * (GLU ? 32 : 64)) * K);
      step = 8 * (int64_t)K * (int64_t)sizeof(elem_t);
      up = GLU ? (int64_t)(N - 32) * K * (int64_t)sizeof(elem_t) : 0;
      voff[0] = (unsigned)((lr * (int64_t)K + lc * VK_VEC) * (int64_t)sizeof(elem_t));
    } else {
      src = reinterpret_cast<const unsigned char*>(act + (act_row != nullptr ? 0 : (int64_t)m_blk * lda));
#pragma unroll
      for (int j = 0; j < FA; ++j) {
        const int row = min(m_blk + (q * FA + j) * 8 + lr, M - 1);
        voff[j] = (unsigned)(((int64_t)(act_row != nullptr ? act_row[row] : row - m_blk) * lda + lc * VK_VEC) * (int64_t)sizeof(elem_t));
      }
    }
    unsigned fill = 0, read_a = 0, read_w = 0;
    auto issue = [&](int from, int to) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < L; ++j)
        if (j >= from && j < to) {
          const unsigned at = __builtin_amdgcn_readfirstlane(lds0 + fill + j * 8 * T_ROWB);
          if constexpr (G == 1 && ONCE) pipe_load_to_lds16_once(src + j * step + (j >= 4 ? up : 0), voff[0], at);
          else if constexpr (G == 1) pipe_load_to_lds16_sv(src + j * step + (j >= 4 ? up : 0), voff[0], at);
          else pipe_load_to_lds16_sv(src, voff[j], at);
        }
      if (to < L) return;
      src += T_ROWB;
      fill = fill == (ST - 1) * BYTES ? 0 : fill + BYTES;
    };
    f32x4 acc[FNW][FA];
    auto slab = [&](int S, bool first, bool more) __attribute__((always_inline)) {
      frag_t af[FA], wf[FNW];
#pragma unroll
      for (int j = 0; j < FA; ++j) af[j] = *reinterpret_cast<const frag_t*>(lds + (a_at ^ (S * 64)) + read_a + j * 16 * T_ROWB);
#pragma unroll
      for (int i = 0; i < FNW; ++i) wf[i] = *reinterpret_cast<const frag_t*>(lds + (w_at ^ (S * 64)) + read_w + i * 16 * T_ROWB);
      if (S == 1) {
        read_a = read_a == (SA - 1) * A_BYTES ? 0 : read_a + A_BYTES;
        read_w = read_w == (SW - 1) * W_BYTES ? 0 : read_w + W_BYTES;
      }
      if (more && S == 0) issue(0, HALF);
      if (more && S == 1 && HALF < L) issue(HALF, L);
      if (G == 1 && S == 1) {
        if (more) wait_vmcnt_n<(SW - 2) * LW>(); else wait_vmcnt_n<0>();
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      al_barrier();
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int i = 0; i < FNW; ++i)
#pragma unroll
        for (int j = 0; j < FA; ++j) acc[i][j] = mma_slab(wf[i], af[j], first ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[i][j]);
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
      if (G == 0 && S == 1) {
        if (more) wait_vmcnt_n<(SA - 2) * LA>(); else wait_vmcnt_n<0>();
      }
      al_barrier();
      __builtin_amdgcn_sched_barrier(0);
    };
    auto chunk = [&](bool last) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < T_CHUNK_TILES; ++t) {
        const bool more = !last || t + ST - 1 < T_CHUNK_TILES;
        slab(0, t == 0, more);
        slab(1, false, more);
      }
#pragma unroll
      for (int i = 0; i < FNW; ++i)
#pragma unroll
        for (int j = 0; j < FA; ++j) {
          total[i][j].x = total[i][j].x + acc[i][j].x;
          total[i][j].y = total[i][j].y + acc[i][j].y;
          total[i][j].z = total[i][j].z + acc[i][j].z;
          total[i][j].w = total[i][j].w + acc[i][j].w;
        }
    };
#pragma unroll
    for (int p = 0; p < ST - 1; ++p) issue(0, L);
    wait_vmcnt_n<(ST - 2) * L>();
    al_barrier();
    if (G == 1) al_barrier();
    for (int c = 1; c < K / KC; ++c) chunk(false);
    chunk(true);
    if (G == 0) al_barrier();
  };
  if (group == 0) walk(std::integral_constant<int, 0>(), std::false_type());
  else if (once) walk(std::integral_constant<int, 1>(), std::true_type());
  else walk(std::integral_constant<int, 1>(), std::false_type());

  const int m0 = m_blk + group * FA * 16 + r16, n0 = n_blk + q * (GLU ? 32 : 64) + 4 * kg;
  if constexpr (GLU) {
#pragma unroll
    for (int j = 0; j < FA; ++j) {
      const int m = m0 + j * 16;
      float rw = 1.f;
      bool none = false;
      if (glu.wts != nullptr && m < M) {
        const int pair = glu.row_pair[m];
        none = pair < 0;
        rw = glu.wts[max(pair, 0)];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        f32x4 y;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float g = fminf(round_to_elem(total[i][j][e]) * rw, glu.limit), u = fminf(fmaxf(round_to_elem(total[i + 2][j][e]) * rw, -glu.limit), glu.limit);
          y[e] = none ? 0.f : (g / (1.f + expf(-glu.slope * g))) * (u + glu.shift);
        }
        store_out4(out, ldo, m, n0 + i * 16, M, N, y, out_form);
      }
    }
  } else {
#pragma unroll
    for (int i = 0; i < FNW; ++i)
#pragma unroll
      for (int j = 0; j < FA; ++j) store_out4(out, ldo, m0 + j * 16, n0 + i * 16, M, N, total[i][j], out_form);
  }
}

template <bool GLU>
__global__ __launch_bounds__(512, 2) void gemm_experts_kernel(elem_t* __restrict__ out, const elem_t* __restrict__ act, const elem_t* __restrict__ w, int N, int K,
                                                              int64_t lda, int64_t ldo, int out_form, const int4* __restrict__ order, int matrices,
                                                              int64_t weights_stride, const int32_t* __restrict__ act_row, GluArgs glu) {
  constexpr int COLS = GLU ? 128 : 256;
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x & 63, cols = (N + COLS - 1) / COLS, lin = blockIdx.x;
  int before = 0, first = 0, rows = 0, which = 0;
  for (int e0 = 0; e0 < matrices; e0 += 64) {
    const int4 entry = order[min(e0 + lane, matrices - 1)];
    const uint64_t begun = __ballot(e0 + lane < matrices && entry.z > 0 && entry.x * cols <= lin);
    if (begun == 0) break;
    const int from = 63 - __builtin_clzll(begun);
    before = __builtin_amdgcn_readlane(entry.x, from);
    first = __builtin_amdgcn_readlane(entry.y, from);
    rows = __builtin_amdgcn_readlane(entry.z, from);
    which = __builtin_amdgcn_readlane(entry.w, from);
    if (begun != ~0ull) break;
  }
  const int parts = (rows + EXPERT_PART_ROWS - 1) / EXPERT_PART_ROWS, o = lin - before * cols;
  if (o >= parts * cols) return;
  const int cg = o / (8 * parts), rem = o - cg * 8 * parts, wide = min(8, cols - cg * 8);
  const int r = rem / wide, nb = cg * 8 + (rem - r * wide);
  const int per = ((rows + parts - 1) / parts + 31) & ~31;
  const int count = min(per, rows - r * per);
  const int m_blk = __builtin_amdgcn_readfirstlane(first + r * per), n_blk = __builtin_amdgcn_readfirstlane(min(nb * COLS, N - COLS));
  const int M = __builtin_amdgcn_readfirstlane(m_blk + count), fa = __builtin_amdgcn_readfirstlane((count + 31) / 32);
  const elem_t* wm = w + (int64_t)which * weights_stride;
  switch (fa) {
    case 1: experts_tile<GLU, 1>(lds, out, act, wm, M, N, K, lda, ldo, out_form, m_blk, n_blk, parts == 1, act_row, glu); break;
    case 2: experts_tile<GLU, 2>(lds, out, act, wm, M, N, K, lda, ldo, out_form, m_blk, n_blk, parts == 1, act_row, glu); break;
    case 3: experts_tile<GLU, 3>(lds, out, act, wm, M, N, K, lda, ldo, out_form, m_blk, n_blk, parts == 1, act_row, glu); break;
    case 4: experts_tile<GLU, 4>(lds, out, act, wm, M, N, K, lda, ldo, out_form, m_blk, n_blk, parts == 1, act_row, glu); break;
    case 5: experts_tile<GLU, 5>(lds, out, act, wm, M, N, K, lda, ldo, out_form, m_blk, n_blk, parts == 1, act_row, glu); break;
    default: experts_tile<GLU, 6>(lds, out, act, wm, M, N, K, lda, ldo, out_form, m_blk, n_blk, parts == 1, act_row, glu); break;
  }
}

static_assert(EXPERT_PART_ROWS == 32 * 6, "six heights");
// Whether a product goes this way or by blocks of 128 rows (launch_pipe), by the workgroups that it can be expected to have: a matrix's rows, as M and the
// matrices tell them, are a part or somewhat more than their share of one.  A workgroup is alone on its compute unit and as long as all
// of K, so that few of them, or a few more than one round, lose to the smaller tiles of the other kernel; the fewer rows a matrix has, the more
// its weights' way from memory decides, which this kernel is better at.  Measured on MI355X in recorded launches with the weights of several layers in turn, 346
// sizes of 8 to 128 matrices, 32 to 1,024 rows a matrix, 256 x 1,024 to 6,144 x 4,096 weights: blocks alone 36.7 ms, parts alone 31.8, by
// this rule 31.3, with the better one everywhere 31.2; 8 matrices, 777 tokens x 2, 1,024 x 1,024 (about 45 workgroups) 14.6, 24.7 us; 16 matrices of 512 rows, 1,536 x 1,024 (312)
// 46.9, 56.7; 16 of 97, 4,096 x 3,072 (256) 117, 76; 64 of 127, 1,536 x 1,024 (402) 87, 58; one chunk, 64 of 384, 512 x 512 31.0, 33.8.  Slower by
// more than 3 % than the better one: 27 sizes, the worst 8 of 194, 4,096 x 3,072 64.9, 72.7.
static bool experts_takes(int M, int N, int K, int64_t lda, int matrices, bool gated) {
  const int columns = gated ? 128 : 256;
  if (K % KC != 0 || K == KC || N < columns || matrices < 1 || rows_far(lda, EXPERT_PART_ROWS)) return false;
  const double rows = std::max(M - 127.0 * matrices, 1.0) / matrices, units = vk_device_cus();
  const double groups = matrices * std::max(1.0, rows / EXPERT_PART_ROWS + 0.35) * ((N + columns - 1) / columns);
  if (rows < 48) return groups >= 0.4 * units;
  if (rows < 100) return groups >= 0.5 * units;
  return groups >= 0.66 * units && (groups <= units || groups >= 1.33 * units || K >= 4 * KC);
}
template <bool GLU>
static int launch_experts(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int form, const int32_t* order, int matrices,
                          int64_t weights_stride, const int32_t* act_row, const GluArgs& glu, hipStream_t st) {
  constexpr int COLS = GLU ? 128 : 256;
  constexpr int smem = (2 * 128 + 4 * 256) * T_ROWB;      // the most of the heights: two tiles of 128 rows beside four of weights
  static bool configured = false;
  if (!configured) {
    (void)hipFuncSetAttribute((const void*)gemm_experts_kernel<GLU>, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    configured = true;
  }
  if (N % 4 != 0) form &= ~OUT_VEC;
  const int64_t tiles = (int64_t)(M / 128) * ((N + COLS - 1) / COLS);
  gemm_experts_kernel<GLU><<<(unsigned)tiles, 512, smem, st>>>(out, act, w, N, K, lda, ldo, form, (const int4*)order, matrices, weights_stride, act_row, glu);
  return vk_check_launch("gemm (experts)");
}
#endif

#ifdef VK_BF16
// ---------------------------------------------------------------- few rows
// 17 to 64 rows of 16-bit elements, K in whole chunks.  The streaming kernels and the one that shares activations through LDS bring weights into
// registers in the order of the matrix unit's operands: an instruction touches 16 rows, half a cache line of each, which holds them to about 4 TB/s.  Here tiles of
// TS slabs of a row, one or two whole lines, go from memory straight into LDS, weights (read by this workgroup alone: past the caches) and activations
// alike, S of them in a ring, one barrier a tile.  A workgroup has NW waves and walks all of K; a wave has FNW x 16 weight rows, or with
// SwiGLU 16 gate rows and the 16 up rows that go with them, and all 16 FA activation rows.  Operand roles, reduction order and bits are those of
// gemm_pipe_kernel.  A row's 16-byte piece j lies at piece j ^ (row mod pieces), so that 16 rows' fragments lie on different banks.  Rows beyond N or
// M are the last one again (their results are dropped).
//
// What bounds it: memory where enough bytes are on their way (151,936 x 4,096, 17 rows: 5.9 TB/s), below that a workgroup's chain of a wait, a barrier, the
// fragments' way from LDS and the MFMAs for each tile; several workgroups a compute unit cover each other, so stages are kept to what lets three (up to 32 rows) or two
// fit a unit: six or twelve stages with fewer of them are 2 to 15 % slower.  Measured on MI355X in recorded launches with the weights
// of several layers in turn, before and after, us, 17 and 64 rows: with SwiGLU 17,408 x 5,120 89 -> 72, 101 -> 93; 9,728 x 2,560 30.6 -> 22.3, 32.9 -> 26.8; 6,144 x 2,048
// 18.1 -> 12.4, 20.8 -> 14.2; plain 7,168 x 5,120 23.2 -> 15.7, 29.9 -> 23.8; 12,288 x 4,096 24.5 -> 20.7, 33.2 -> 24.1; 32,768 x 2,048 34.6 -> 27.2, 36.6 -> 28.1.
template <int NW, int FNW, int FA, int TS, int S, bool SWIGLU>
__global__ __launch_bounds__(64 * NW) void gemm_rows_kernel(elem_t* __restrict__ out, const elem_t* __restrict__ act, const elem_t* __restrict__ w,
                                                           int M, int N, int K, int64_t lda, int64_t ldo, int out_form) {
  static_assert(!SWIGLU || FNW == 2, "a wave has its gate rows and the up rows that go with them");
  constexpr int ROWB = TS * VK_SLAB * (int)sizeof(elem_t), LOAD_ROWS = 1024 / ROWB, PIECES = ROWB / 16;
  constexpr int BN = 16 * FNW * NW, BM = 16 * FA;
  constexpr int LW = 16 * FNW / LOAD_ROWS, LA = BM / LOAD_ROWS / NW, PER_TILE = LW + LA;      // loads a tile and wave
  constexpr int STAGE = (BN + BM) * ROWB, CHUNK_TILES = KC / (TS * VK_SLAB);
  static_assert(LA * NW * LOAD_ROWS == BM, "the waves bring as many activation rows each");
  static_assert((S - 2) * PER_TILE < 64, "loads in flight are counted by six bits");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int n0 = (blockIdx.x * NW + wave) * 16 * (SWIGLU ? 1 : FNW);
  const int first = min(n0, N - 1), ntiles = K / (TS * VK_SLAB);
  // Load j of a wave's weights or activations brings LOAD_ROWS rows, a kilobyte; lane i fills piece i % PIECES of row i / PIECES.
  const int lr = lane / PIECES, lp = lane % PIECES;
  const unsigned char* wbase = reinterpret_cast<const unsigned char*>(w + (int64_t)first * K);
  const unsigned char* ubase = reinterpret_cast<const unsigned char*>(w + (int64_t)(N + first) * K);
  const unsigned char* abase = reinterpret_cast<const unsigned char*>(act);
  unsigned offw[LW], offa[LA];
#pragma unroll
  for (int j = 0; j < LW; ++j) {
    const int row = j * LOAD_ROWS + lr, local = SWIGLU ? row & 15 : row;
    offw[j] = (unsigned)(((int64_t)(min(n0 + local, N - 1) - first) * K + ((lp ^ (row & (PIECES - 1))) * VK_VEC)) * (int64_t)sizeof(elem_t));
  }
#pragma unroll
  for (int j = 0; j < LA; ++j) {
    const int row = (wave * LA + j) * LOAD_ROWS + lr;
    offa[j] = (unsigned)(((int64_t)min(row, M - 1) * lda + ((lp ^ (row & (PIECES - 1))) * VK_VEC)) * (int64_t)sizeof(elem_t));
  }
  const unsigned lds0 = lds_offset_of(lds);
  auto issue = [&](int kt, int slot) {
    const unsigned base = lds0 + slot * STAGE;
    const int64_t kb = (int64_t)kt * ROWB;
#pragma unroll
    for (int j = 0; j < LW; ++j) {
      const bool up = SWIGLU && j * LOAD_ROWS >= 16;
      pipe_load_to_lds16_once((up ? ubase : wbase) + kb, offw[j], base + (wave * LW + j) * 1024);
    }
#pragma unroll
    for (int j = 0; j < LA; ++j) pipe_load_to_lds16_sv(abase + kb, offa[j], base + BN * ROWB + (wave * LA + j) * 1024);
  };
  f32x4 acc[FNW][FA], total[FNW][FA];
#pragma unroll
  for (int i = 0; i < FNW; ++i)
#pragma unroll
    for (int j = 0; j < FA; ++j) acc[i][j] = total[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int p = 0; p < S - 1; ++p)
    if (p < ntiles) issue(p, p);
  int slot = 0, ahead = S - 1;
  for (int c = 0; c < ntiles; c += CHUNK_TILES) {
#pragma unroll
    for (int u = 0; u < CHUNK_TILES; ++u) {
      const int kt = c + u;
      // Tile kt has landed once at most the S - 2 tiles behind it are outstanding; near the end, where there are fewer, once none is.
      if (kt + S - 2 < ntiles) wait_vmcnt_n<(S - 2) * PER_TILE>();
      else wait_vmcnt_n<0>();
      __syncthreads();       // every wave's part of tile kt is there; everyone is done with tile kt - 1's place
      if (kt + S - 1 < ntiles) issue(kt + S - 1, ahead);
      const unsigned char* base = lds + slot * STAGE;
      frag_t wf[TS][FNW], af[TS][FA];
#pragma unroll
      for (int s = 0; s < TS; ++s) {
        const int col = ((s * 4 + kg) ^ (r16 & (PIECES - 1))) * 16;
#pragma unroll
        for (int i = 0; i < FNW; ++i) wf[s][i] = *reinterpret_cast<const frag_t*>(base + ((wave * FNW + i) * 16 + r16) * ROWB + col);
#pragma unroll
        for (int j = 0; j < FA; ++j) af[s][j] = *reinterpret_cast<const frag_t*>(base + (BN + j * 16 + r16) * ROWB + col);
      }
#pragma unroll
      for (int s = 0; s < TS; ++s)
#pragma unroll
        for (int i = 0; i < FNW; ++i)
#pragma unroll
          for (int j = 0; j < FA; ++j) acc[i][j] = mma_slab(wf[s][i], af[s][j], acc[i][j]);
      slot = slot + 1 == S ? 0 : slot + 1;
      ahead = ahead + 1 == S ? 0 : ahead + 1;
    }
#pragma unroll
    for (int i = 0; i < FNW; ++i)
#pragma unroll
      for (int j = 0; j < FA; ++j) {
        total[i][j].x = total[i][j].x + acc[i][j].x;
        total[i][j].y = total[i][j].y + acc[i][j].y;
        total[i][j].z = total[i][j].z + acc[i][j].z;
        total[i][j].w = total[i][j].w + acc[i][j].w;
        acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
  }
  if constexpr (SWIGLU) {
#pragma unroll
    for (int j = 0; j < FA; ++j) {
      f32x4 g = total[0][j], u = total[1][j], y;
      g.x = round_to_elem(g.x); g.y = round_to_elem(g.y); g.z = round_to_elem(g.z); g.w = round_to_elem(g.w);
      u.x = round_to_elem(u.x); u.y = round_to_elem(u.y); u.z = round_to_elem(u.z); u.w = round_to_elem(u.w);
      y.x = (g.x * (1.0f / (1.0f + expf(-g.x)))) * u.x;
      y.y = (g.y * (1.0f / (1.0f + expf(-g.y)))) * u.y;
      y.z = (g.z * (1.0f / (1.0f + expf(-g.z)))) * u.z;
      y.w = (g.w * (1.0f / (1.0f + expf(-g.w)))) * u.w;
      store_out4(out, ldo, j * 16 + r16, n0 + 4 * kg, M, N, y, out_form);
    }
  } else {
#pragma unroll
    for (int i = 0; i < FNW; ++i)
#pragma unroll
      for (int j = 0; j < FA; ++j) store_out4(out, ldo, j * 16 + r16, n0 + i * 16 + 4 * kg, M, N, total[i][j], out_form);
  }
}

template <int NW, int FNW, int FA, int TS, int S, bool SWIGLU = false>
static int launch_rows(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int form, hipStream_t st) {
  constexpr int smem = S * (16 * FNW * NW + 16 * FA) * TS * VK_SLAB * (int)sizeof(elem_t);
  static_assert(smem <= 160 * 1024, "LDS");
  static bool configured = false;
  if (!configured) {
    (void)hipFuncSetAttribute((const void*)gemm_rows_kernel<NW, FNW, FA, TS, S, SWIGLU>, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    configured = true;
  }
  constexpr int cols = 16 * NW * (SWIGLU ? 1 : FNW);
  gemm_rows_kernel<NW, FNW, FA, TS, S, SWIGLU><<<(unsigned)((N + cols - 1) / cols), 64 * NW, smem, st>>>(out, act, w, M, N, K, lda, ldo, form);
  return vk_check_launch("gemm_rows");
}

// How a product of 17 to 64 rows is cut for gemm_rows_kernel: the weight rows (with SwiGLU: gate rows) of a workgroup, or 0 where the other kernels are
// the faster ones.  The narrowest workgroups that still have enough to do are the fastest up to one or two a compute unit; then wider ones, whose
// activations serve more weights.  Measured over 240 plain sizes (N of 3,072 to 32,768, K of 1,024 to 8,192) and 176 with SwiGLU (1,024 to 25,600 x 1,024 to
// 5,120); before / after by the number of workgroups of 32, g, against the compute units:
//   plain   g <= 1/2             the other kernels (which split K over waves or workgroups) 1.02 to 1.8 times as fast, but for K of two chunks
//           up to 1              32 weight rows (0.98 to 1.55); not for 33 rows and more where g < 3/4 and K is more than 4 chunks (0.91 to 1.02).
//                                K of 5 to 8 chunks, up to 32 rows, g > 7/8: 64 weight rows (1.03; 32: 0.94)
//           more                 64 weight rows (1.04 to 2.4)
//   SwiGLU  g <= 1/2             16 gate rows (1.03 to 2.2; 32: 0.87 to 1.8)
//           up to 1              32 (1.1 to 2.0); K of 5 to 8 chunks, g > 7/8: 64 (1.01 to 1.28; 32: 0.87 to 1.15)
//           up to 2, above 3     64 (1.02 to 1.8; 32: 0.97 to 1.8)
//           above 2, up to 3     32, of which a compute unit holds three (1.03 to 1.6; 64, a nearly empty second round: 0.88 to 1.3)
static int rows_width(int M, int N, int K, int64_t lda, bool swiglu) {
  if (M <= 16 || M > 64 || K % KC != 0 || lda > (1 << 25)) return 0;       // a row's offset is of 32 bits
  const int cus = vk_device_cus(), chunks = K / KC, g = (N + 31) / 32;
  const bool middle = chunks > 4 && chunks <= 8 && 8 * g > 7 * cus && g <= cus;
  if (swiglu) {
    if (2 * g <= cus) return 16;
    if (g <= cus) return middle ? 64 : 32;
    return g <= 2 * cus || g > 3 * cus ? 64 : 32;
  }
  if (2 * g <= cus || (M > 32 && chunks > 4 && 4 * g < 3 * cus)) return 0;
  return g > cus || (middle && M <= 32) ? 64 : 32;
}
static int gemm_rows(int width, bool swiglu, elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int form, hipStream_t st) {
#define ROWS(NW, FNW, TS, S, SWIGLU)                                                                                      \
  return M <= 32 ? launch_rows<NW, FNW, 2, TS, S, SWIGLU>(out, act, w, M, N, K, lda, ldo, form, st)                       \
                 : launch_rows<NW, FNW, 4, TS, S, SWIGLU>(out, act, w, M, N, K, lda, ldo, form, st)
  if (swiglu) {
    if (width == 16) ROWS(1, 2, 4, 4, true);
    if (width == 32) ROWS(2, 2, 2, 4, true);
    ROWS(4, 2, 4, 3, true);
  }
  if (width == 32) ROWS(2, 1, 4, 4, false);
  ROWS(4, 1, 2, 4, false);
#undef ROWS
}
#endif

// ------------------------------------------------------------------ mid
// 17 to 64 rows, of 16-bit elements those that rows_width leaves (at most 4,096 weight rows, mostly) and up to 128 in blocks.  The streaming kernels
// read all activations once per 16 weight rows, which at 64 rows
// is four times the weights and binds them to the second-level cache.  Here a workgroup of eight waves
// takes 64 weight rows: wave (nt, kh) streams weight tile nt (16 rows) for the chunks kh, kh + 2, ...
// into registers with a rolling window, as the streaming kernels do, and the activations of the two
// chunks in work go into LDS once for all waves (global_load_lds, a quarter chunk at a time, two
// buffers).  After a pair of chunks the waves with kh = 1 hand their chunk sum over through LDS and the
// waves with kh = 0 add both to the total, in chunk order.  K is a multiple of 512.
//
// Waits: the barrier of a step is a bare s_barrier (a __syncthreads would wait for every weight load in
// flight); a wave waits for its part of the activation loads by count: they are followed by exactly
// MID_QS weight loads before the next step begins (MID_W at the start), kept so by scheduling barriers.
#define MID_QS 4                       // slabs per step
#define MID_W 8                        // weight slabs in flight per wave
__device__ __forceinline__ void mid_wait_vmcnt_4() { __builtin_amdgcn_s_waitcnt(0x0F74); }
__device__ __forceinline__ void mid_wait_vmcnt_w() { static_assert(MID_W == 8, "vmcnt(8)"); __builtin_amdgcn_s_waitcnt(0x0F78); }
__device__ __forceinline__ void mid_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void mid_load_to_lds16(const elem_t* src, unsigned char* dst) {
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// SWIGLU (one chunk in work, KH = 1): w holds N gate rows, then N up rows; waves 0..GT-1 take GT gate
// tiles, waves GT..2GT-1 the matching up tiles, and out[m, n] = silu(g) * u with g and u rounded to the
// element type first, as the separate kernels compute it.  With GT < 4 the other waves only help to bring
// in the activations: 12288 gate rows are 256 workgroups of three tiles, one for every compute unit,
// where four tiles a workgroup leave a quarter of them idle.
template <int MT, int KH, bool SWIGLU = false, int GT = 4>
__global__ __launch_bounds__(512) void gemm_mid_kernel(elem_t* __restrict__ out, const elem_t* __restrict__ act,
                                                       const elem_t* __restrict__ w, int M, int N, int K,
                                                       int64_t lda, int64_t ldo, int out_form) {
  static_assert(!SWIGLU || KH == 1, "the SwiGLU epilogue pairs the waves of one chunk");
  static_assert(GT == 4 || (SWIGLU && GT >= 2 && GT < 4), "fewer gate tiles only with the SwiGLU epilogue");
  constexpr int NTW = 8 / KH;                       // waves side by side along the weight rows
  constexpr int ACTIVE = SWIGLU ? 2 * GT : 8;       // waves that stream weights
  constexpr int STEPS = KC_SLABS / MID_QS;          // steps per chunk
  constexpr int ROW_B = MID_QS * 64;                // bytes of an activation row in a step: 256
  constexpr int HALF_B = 16 * MT * ROW_B;           // one chunk's part of a buffer
  constexpr int BUF_B = KH * HALF_B;
  constexpr int DMA = MT * KH / 2;                  // activation loads per wave and step (8 KH MT / 2 in all... 4 rows each)
  static_assert((MT * KH) % 2 == 0, "the activation loads divide evenly over the waves");
  extern __shared__ __attribute__((aligned(16))) unsigned char lds[];   // [2 buffers][kh][16 MT rows][256 B], then part
  f32x4* part = reinterpret_cast<f32x4*>(lds + 2 * BUF_B);              // [KH - 1][NTW tiles][MT][64 lanes]

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int nt = wave % NTW, kh = wave / NTW;
  const bool active = ACTIVE == 8 || wave < ACTIVE;
  const int row0 = blockIdx.y * 16 * MT;            // more than 16 MT rows: one block of them per blockIdx.y
  const int nchunks = K / KC, ngroups = (nchunks + KH - 1) / KH;     // group: KH chunks in work together
  const int nsteps = ngroups * STEPS;
  const int last_full = nchunks - (ngroups - 1) * KH;                // chunks of the last group: 1 .. KH

  // Weights: row of this wave's tile, chunk sequence kh, kh + KH, ...; a chunk beyond the last is read as
  // the last (and not used), so that every wave issues the same number of loads.
  const int out_col0 = SWIGLU ? (int)blockIdx.x * 16 * GT + (nt % GT) * 16 : (int)blockIdx.x * 16 * NTW + nt * 16;
  const int64_t wrow_i = SWIGLU ? (int64_t)min(nt / GT, 1) * N + min(out_col0 + r16, N - 1) : min(out_col0 + r16, N - 1);
  const elem_t* wrow = w + wrow_i * K + kg * VK_VEC;
  frag_t wbuf[MID_W];
  auto issue_w = [&](int g, int slot) {              // g: this wave's slab number; slot = g % MID_W
    const int gg = min(g, nsteps * MID_QS - 1);
    const int c = min(KH * (gg / KC_SLABS) + kh, nchunks - 1);
    wbuf[slot] = *reinterpret_cast<const frag_t*>(wrow + (int64_t)c * KC + (gg % KC_SLABS) * VK_SLAB);
  };
  // Activations of a step: KH * 16 MT rows of 256 bytes; a wave-level load fills 4 rows, lane i the
  // 16-byte column i % 16 of row i / 16, which holds the logical column (i % 16) ^ (row % 16).
  const elem_t* asrc[DMA];
  int adst[DMA], ah[DMA];
#pragma unroll
  for (int j = 0; j < DMA; ++j) {
    const int id = wave * DMA + j;                   // 0 .. 4 MT KH - 1
    const int h = id / (4 * MT), row = (id % (4 * MT)) * 4 + (lane >> 4);
    ah[j] = h;
    asrc[j] = act + (int64_t)min(row0 + row, M - 1) * lda + (((lane & 15) ^ (row & 15)) * VK_VEC);
    adst[j] = h * HALF_B + (id % (4 * MT)) * 4 * ROW_B;
  }
  auto issue_a = [&](int t) {                        // step t of the workgroup
    const int tt = min(t, nsteps - 1);
    const int group = tt / STEPS, q = tt % STEPS;
    unsigned char* base = lds + (t & 1) * BUF_B;
#pragma unroll
    for (int j = 0; j < DMA; ++j) {
      const int c = min(group * KH + ah[j], nchunks - 1);    // beyond the last chunk: the last again (not used)
      mid_load_to_lds16(asrc[j] + (int64_t)c * KC + q * MID_QS * VK_SLAB, base + adst[j]);
    }
  };

  f32x4 acc[MT], total[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = total[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  // The chunk sums of a complete group join the total in chunk order: this wave's own, then the others'.
  auto close_group = [&](int chunks_in_group) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      total[mt].x = total[mt].x + acc[mt].x; total[mt].y = total[mt].y + acc[mt].y;
      total[mt].z = total[mt].z + acc[mt].z; total[mt].w = total[mt].w + acc[mt].w;
#pragma unroll
      for (int h = 1; h < KH; ++h) {
        if (h < chunks_in_group) {
          const f32x4 p = part[(((h - 1) * NTW + nt) * MT + mt) * 64 + lane];
          total[mt].x = total[mt].x + p.x; total[mt].y = total[mt].y + p.y;
          total[mt].z = total[mt].z + p.z; total[mt].w = total[mt].w + p.w;
        }
      }
    }
  };

  constexpr int TURN = MID_W / MID_QS;      // steps in one turn of the weight window
  static_assert(STEPS % TURN == 0, "a turn of the weight window is a whole number of steps");
  issue_a(0);
  __builtin_amdgcn_sched_barrier(0);
  if (active) {
#pragma unroll
    for (int i = 0; i < MID_W; ++i) issue_w(i, i);
    __builtin_amdgcn_sched_barrier(0);
    for (int t2 = 0; t2 < nsteps; t2 += TURN) {
#pragma unroll
      for (int u = 0; u < TURN; ++u) {         // written out: the window's slots are then fixed registers
        const int t = t2 + u;
        if (t == 0) mid_wait_vmcnt_w(); else mid_wait_vmcnt_4();
        mid_barrier();          // step t's activations are in LDS; everyone is done with the other buffer
        const int group = t / STEPS, q = t % STEPS;
        if (q == 0 && group > 0) {
          if (kh == 0) close_group(KH);           // the group before is complete
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        __builtin_amdgcn_sched_barrier(0);
        issue_a(t + 1);
        __builtin_amdgcn_sched_barrier(0);
        const unsigned char* abase = lds + (t & 1) * BUF_B + kh * HALF_B;
#pragma unroll
        for (int s = 0; s < MID_QS; ++s) {
          const int g = t * MID_QS + s;
          const frag_t fw = wbuf[u * MID_QS + s];
          frag_t fa[MT];
#pragma unroll
          for (int mt = 0; mt < MT; ++mt)
            fa[mt] = *reinterpret_cast<const frag_t*>(abase + (mt * 16 + r16) * ROW_B + (((s * 4 + kg) ^ r16) << 4));
          issue_w(g + MID_W, u * MID_QS + s);
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) acc[mt] = mma_slab(fw, fa[mt], acc[mt]);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (q == STEPS - 1 && kh > 0) {
          // This wave's chunk of the group is complete: hand it over (one beyond the last chunk is not used).
#pragma unroll
          for (int mt = 0; mt < MT; ++mt) part[(((kh - 1) * NTW + nt) * MT + mt) * 64 + lane] = acc[mt];
        }
      }
    }
  } else {
    // A wave without weights only brings in its share of the activations: the same barriers, and nothing
    // in flight but those loads.
    for (int t = 0; t < nsteps; ++t) {
      __builtin_amdgcn_s_waitcnt(0x0F70);
      mid_barrier();
      issue_a(t + 1);
    }
  }
  __builtin_amdgcn_s_waitcnt(0x0F70);      // the loads issued beyond the end
  mid_barrier();
  if (kh == 0) {
    close_group(last_full);
    if (SWIGLU) {
      // Every wave is past the barrier above, so the activation buffers are free: the up waves leave
      // their sums there for the gate waves of the same columns.
      f32x4* ex = reinterpret_cast<f32x4*>(lds);       // [GT tiles][MT][64 lanes]
      if (nt >= GT && active) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) ex[((nt - GT) * MT + mt) * 64 + lane] = total[mt];
      }
      __syncthreads();
      if (nt < GT) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          const f32x4 t = total[mt], o = ex[(nt * MT + mt) * 64 + lane];
          const float g[4] = {round_to_elem(t.x), round_to_elem(t.y), round_to_elem(t.z), round_to_elem(t.w)};
          const float u[4] = {round_to_elem(o.x), round_to_elem(o.y), round_to_elem(o.z), round_to_elem(o.w)};
          f32x4 y;
          y.x = (g[0] * (1.0f / (1.0f + expf(-g[0])))) * u[0];
          y.y = (g[1] * (1.0f / (1.0f + expf(-g[1])))) * u[1];
          y.z = (g[2] * (1.0f / (1.0f + expf(-g[2])))) * u[2];
          y.w = (g[3] * (1.0f / (1.0f + expf(-g[3])))) * u[3];
          store_out4(out, ldo, row0 + mt * 16 + r16, out_col0 + 4 * kg, M, N, y, out_form);
        }
      }
      return;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      store_out4(out, ldo, row0 + mt * 16 + r16, out_col0 + 4 * kg, M, N, total[mt], out_form);
  }
}

// N: weight rows, or with SWIGLU the gate rows (and as many up rows after them).
template <int MT, int KH, bool SWIGLU = false, int GT = 4>
static int launch_mid(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo,
                      int form, hipStream_t st) {
  constexpr int NTW = 8 / KH;
  constexpr int COLS = SWIGLU ? 16 * GT : 16 * NTW; // output columns of a workgroup
  const size_t smem = (size_t)2 * KH * 16 * MT * (MID_QS * 64) + (size_t)(KH - 1) * NTW * MT * 64 * sizeof(f32x4);
  static_assert(!SWIGLU || 2 * 16 * MT * (MID_QS * 64) >= 4 * MT * 64 * (int)sizeof(f32x4), "the exchange fits the activation buffers");
  static bool configured = false;
  if (!configured) {
    (void)hipFuncSetAttribute((const void*)gemm_mid_kernel<MT, KH, SWIGLU, GT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
    configured = true;
  }
  // Blocks of 16 MT rows side by side: those of a weight tile run at about the same time, and on the same
  // chip part when the grid's width is a multiple of eight, so that all but one find it in its cache.
  const dim3 grid((N + COLS - 1) / COLS, (M + 16 * MT - 1) / (16 * MT));
  gemm_mid_kernel<MT, KH, SWIGLU, GT><<<grid, 512, smem, st>>>(out, act, w, M, N, K, lda, ldo, form);
  return vk_check_launch("gemm_mid");
}

// ---------------------------------------------------------------- split
// 17 to 64 rows and few weight rows: the kernels above give such a product a workgroup or less per compute
// unit, each walking a long stretch of K on its own with a window of loads that one latency drains.  Here
// a workgroup takes 16 NTW weight rows of ONE chunk: a wave's 16 rows x 512 elements are all in flight at
// once, the chunk of the activations goes into LDS once for its waves, and the chunk sums go to a
// workspace [chunk][weight tile][activation tile][lane]; a second kernel adds them in chunk order to a
// zero total, which is what every other kernel computes, and writes the output (with SWIGLU: of
// silu(g) * u, g and u rounded to the element type first).  16-bit elements only.
#ifdef VK_BF16
template <int MT, int NTW>
__global__ __launch_bounds__(64 * NTW) void gemm_split_kernel(f32x4* __restrict__ partial, const elem_t* __restrict__ act,
                                                              const elem_t* __restrict__ w, int M, int N, int K,
                                                              int64_t lda, int ntiles16) {
  constexpr int ROW_B = KC * (int)sizeof(elem_t);           // bytes of an activation row of a chunk: 1024
  static_assert(ROW_B == 64 * 16, "a wave-level load fills one activation row");
  __shared__ __attribute__((aligned(16))) unsigned char lds[16 * MT * ROW_B];

  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, kg = lane >> 4;
  const int c = blockIdx.y;
  const int tile = blockIdx.x * NTW + wave;                  // 16-row weight tile; beyond the last: clamped rows, nothing stored

  // Activations first: row r of the chunk lies at lds + r * 1024, its logical 16-byte column j at physical
  // column j ^ (r % 16); lane i of a wave-level load fills physical column i.
#pragma unroll
  for (int j = 0; j < 16 * MT / NTW; ++j) {
    const int r = wave + j * NTW;
    __builtin_amdgcn_global_load_lds(act + (int64_t)min(r, M - 1) * lda + (int64_t)c * KC + ((lane ^ (r & 15)) * VK_VEC),
                                     (__attribute__((address_space(3))) void*)(lds + r * ROW_B), 16, 0, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
  const elem_t* wrow = w + (int64_t)min(tile * 16 + r16, N - 1) * K + (int64_t)c * KC + kg * VK_VEC;
  frag_t wbuf[KC_SLABS];
#pragma unroll
  for (int s = 0; s < KC_SLABS; ++s) wbuf[s] = *reinterpret_cast<const frag_t*>(wrow + s * VK_SLAB);
  __builtin_amdgcn_sched_barrier(0);
  static_assert(KC_SLABS == 16, "vmcnt(16) below: the weight loads are the 16 issued last");
  __builtin_amdgcn_s_waitcnt(0x4F70);      // vmcnt(16): this wave's activation rows are in LDS; its weights still fly
  __syncthreads();

  f32x4 acc[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) acc[mt] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < KC_SLABS; ++s) {
    frag_t fa[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
      fa[mt] = *reinterpret_cast<const frag_t*>(lds + (mt * 16 + r16) * ROW_B + (((s * 4 + kg) ^ r16) << 4));
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) acc[mt] = mma_slab(wbuf[s], fa[mt], acc[mt]);
  }
  if (tile < ntiles16) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) partial[(((int64_t)c * ntiles16 + tile) * MT + mt) * 64 + lane] = acc[mt];
  }
}

// One thread per (weight tile, activation tile, lane): the chunk sums in chunk order.  up_tiles > 0: the
// tile and the one up_tiles after it are the gate and the up projection of the same output columns.
template <int MT>
__global__ __launch_bounds__(256) void gemm_split_reduce_kernel(elem_t* __restrict__ out, const f32x4* __restrict__ partial,
                                                                int M, int N, int64_t ldo, int nchunks, int ntiles16,
                                                                int up_tiles, int out_form) {
  const int64_t t = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int lane = (int)(t & 63), mt = (int)((t >> 6) % MT);
  const int tile = (int)(t / (64 * MT));
  const int out_tiles = up_tiles > 0 ? up_tiles : ntiles16;
  if (tile >= out_tiles) return;
  const int r16 = lane & 15, kg = lane >> 4;
  auto sum = [&](int tl) {
    f32x4 total = {0.f, 0.f, 0.f, 0.f};
    const f32x4* p0 = partial + ((int64_t)tl * MT + mt) * 64 + lane;
    const int64_t stride = (int64_t)ntiles16 * MT * 64;
    int c = 0;
    for (; c + 8 <= nchunks; c += 8) {         // eight loads in flight, added in chunk order
      f32x4 p[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) p[i] = p0[(c + i) * stride];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        total.x = total.x + p[i].x; total.y = total.y + p[i].y; total.z = total.z + p[i].z; total.w = total.w + p[i].w;
      }
    }
    for (; c < nchunks; ++c) {
      const f32x4 p = p0[c * stride];
      total.x = total.x + p.x; total.y = total.y + p.y; total.z = total.z + p.z; total.w = total.w + p.w;
    }
    return total;
  };
  f32x4 y = sum(tile);
  if (up_tiles > 0) {
    const f32x4 o = sum(tile + up_tiles);
    const float g[4] = {round_to_elem(y.x), round_to_elem(y.y), round_to_elem(y.z), round_to_elem(y.w)};
    const float u[4] = {round_to_elem(o.x), round_to_elem(o.y), round_to_elem(o.z), round_to_elem(o.w)};
    y.x = (g[0] * (1.0f / (1.0f + expf(-g[0])))) * u[0];
    y.y = (g[1] * (1.0f / (1.0f + expf(-g[1])))) * u[1];
    y.z = (g[2] * (1.0f / (1.0f + expf(-g[2])))) * u[2];
    y.w = (g[3] * (1.0f / (1.0f + expf(-g[3])))) * u[3];
  }
  store_out4(out, ldo, mt * 16 + r16, tile * 16 + 4 * kg, M, N, y, out_form);
}

template <int MT>
static int launch_split(elem_t* out, const elem_t* act, const elem_t* w, int M, int rows, int K, int64_t lda, int64_t ldo,
                        int swiglu, float* workspace, int form, hipStream_t st) {
  const int ntiles16 = (rows + 15) / 16, nchunks = K / KC;
  f32x4* partial = reinterpret_cast<f32x4*>(workspace);
  // Eight waves a workgroup where that still leaves two workgroups or more per compute unit, else four
  // (64 rows, 4096 x 12288: 37.3 against 35.7 us; 6144 x 4096: 19.1 against 19.9 us; sixteen waves were slower).
  if ((int64_t)((ntiles16 + 7) / 8) * nchunks >= 2 * vk_device_cus())
    gemm_split_kernel<MT, 8><<<dim3((ntiles16 + 7) / 8, nchunks), 512, 0, st>>>(partial, act, w, M, rows, K, lda, ntiles16);
  else
    gemm_split_kernel<MT, 4><<<dim3((ntiles16 + 3) / 4, nchunks), 256, 0, st>>>(partial, act, w, M, rows, K, lda, ntiles16);
  const int up_tiles = swiglu ? ntiles16 / 2 : 0;
  const int out_tiles = swiglu ? up_tiles : ntiles16;
  const int64_t threads = (int64_t)out_tiles * MT * 64;
  gemm_split_reduce_kernel<MT><<<(unsigned)((threads + 255) / 256), 256, 0, st>>>(out, partial, M, swiglu ? rows / 2 : rows, ldo,
                                                                                  nchunks, ntiles16, up_tiles, form);
  return vk_check_launch("gemm_split");
}
#endif

// ==================================================================== host
// Waves a workgroup of the streaming kernels at up to 16 rows, for K of nchunks chunks.  Wave w takes the chunks
// w, w + waves, ...: with eight waves and ten chunks two waves have a second chunk and six wait for them at every
// tile's barrier, and with two chunks six of eight waves only take up room.  One chunk a wave where a workgroup
// can be that size (16-bit elements: up to 12 waves; the registers of 32-bit activations allow 8), measured on an
// MI355X at 8 rows: 34816 gate rows x 5120: 88.6 -> 80.0 us, 7168 x 5120: 23.8 -> 20.4, 2048 x 6144: 12.5 -> 11.2,
// 151936 x 1024: 103 -> 59, 151936 x 2048: 142 -> 116, 4096 x 1024: 5.5 -> 4.2.  More chunks than that: eight waves
// (ten or twelve without resident activations: 5120 x 17408 56.8 -> 66 us).
static int stream_waves(int nchunks) {
  if (nchunks <= 2) return 2;
  if (nchunks <= 4) return 4;
  if (nchunks <= 6) return nchunks;
  if (nchunks <= 8) return 8;
#ifdef VK_BF16
  if (nchunks <= 10) return 10;
  if (nchunks <= 12) return 12;
#endif
  return 8;
}

// How many of M rows' activations a streaming kernel of `waves` waves brings in through LDS (1, 4, 8 or 16 a wave and chunk), or 0:
// straight to registers, where that does not fit beside the chunk sums (sums_bytes).  In 32-bit, 16 rows through LDS leave room
// for fewer workgroups, which only launches of one weight tile a workgroup do not miss (151,936 x 1,024: 128 -> 165 us; 1,024 x 2,048: 11.6 -> 9.5).
static constexpr int stream_lds_rows(int M, int waves, int sums_bytes) {
  const int rows = M == 1 ? 1 : M <= 4 ? 4 : M <= 8 ? 8 : 16;
  return waves * CHUNK_ROWS_BYTES(rows) + sums_bytes <= 160 * 1024 ? rows : 0;
}
// Nor do 9 to 16 rows of K = 1,024 (two chunks of 16-bit elements) on about one weight tile a compute unit: 4,096 weight rows, 9 and 16 rows take 3.89 and 3.94 us
// straight to registers, 4.14 and 4.17 through LDS; up to 3,072 and from 4,352 weight rows on the times are the same or LDS is the faster way.
static bool stream_rows_pay(int M, int weight_tiles, int64_t lda, int chunks = 0) {
  if (lda > (1 << 26)) return false;        // a row's offset is of 32 bits
  if (sizeof(elem_t) == 2 && M > 8 && chunks == 2 && weight_tiles <= vk_device_cus() && 4 * weight_tiles > 3 * vk_device_cus()) return false;
  return M <= 8 || sizeof(elem_t) == 2 || weight_tiles <= vk_device_cus();
}

// Which kernel computes a product (speed only: all give the same bits).  Every threshold is a count of
// workgroups against the device's compute units (cus), or a count of 16-row activation tiles, or whether a
// wave's share of K fits its registers; none is a model's size.  With the workgroups a kernel would start:
//   wg16  = ceil(N / 16)   the streaming kernels (one 16-row weight tile a workgroup; two with kernel 7)
//   wg32, wg64, wg128      the kernel that shares activations through LDS (32, 64 or 128 weight rows a workgroup)
//   k_resident             K <= 8 chunks: each of a workgroup's 8 waves has one chunk, whose activations stay in registers
//
//   rows     condition                                         kernel
//   1..16    where lines_rows says so                           20, 21  whole lines
//   1..16                                                      1   streaming
//   17..64   16-bit, where rows_width says so                   -   gemm_rows_kernel.  It leaves up to 4,096 weight rows (up to 6,112 of 33 rows and more of K
//                                                                  above four chunks) and rows further apart than it counts: below, 16-bit sizes reach
//                                                                  12, 9 and 1, and 10, 8 and 7 of 17 to 64 rows are for 32 bits (figures: 16-bit, from before it)
//   17..64   K whole chunks:
//              wg128 >= 0.75 cus                               10  128 weight rows a workgroup: the activations that every
//                                                                  workgroup reads are half the weight bytes (64 rows, 51200 x
//                                                                  5120: 158 -> 127 us)
//              wg64 >= 0.5 cus                                 8   64 weight rows a workgroup
//              rows > 32, wg32 <= 0.5 cus, and rows > 40 or    12  so few weight rows that workgroups of 32 leave half the units
//                not k_resident                                    idle: two blocks of 32 rows side by side (64 rows, 4096 x
//                                                                  12288: 55 -> 45 us)
//              rows > 40                                       9   32 weight rows a workgroup
//              k_resident or wg16 <= cus                       7 / 1  streaming, two weight tiles a workgroup from wg16 >= 1.5 cus
//              else                                            9   the streaming kernel would need a second pass for a few tiles
//                                                                  (32 rows, 5120 x 17408: 111 -> 65 us)
//   17..64   K not in whole chunks                             2 (rows > 32 and wg128 >= 0.5 cus), else 7 / 1 as above
//   65..256  K whole chunks, wg128 < 0.5 cus, 16-bit:              the kernel that shares activations through LDS, in blocks of 64 rows
//              16-bit, two blocks, K > 2 chunks,               9   so few weight rows that the tile kernel's workgroups of 64 leave three
//                wg32 <= 0.5 cus                                     quarters of the units idle (128 rows, 4096 x 12288: 81 us against
//                                                                  54; 1024 x 2048: 13.7 against 11.6)
//              16-bit, rows > 112, two blocks, K >= 10        8   with all of a block's rows in use and long chains the tile kernel in one round is the slower one (128 rows,
//                chunks, wg64 <= 0.5 cus                             5,120 x 5,120: 41.4 against 37.4 us; 8,192 x 6,144: 48.8, 45.4; 7 and 8 K a few sizes 1 to 4 % the other
//                                                                  way; up to 112 rows and nine chunks 0.92 to 1.33 times, 1.09 on the mean)
//              16-bit                                          2   the tile kernel in one round (pipe_fragments_in_one_round; 200 rows,
//                                                                  6144 x 4096: 40 -> 27 us)
//   more                                                       2   the pipelined tile kernel, in one round where it can be
//                                                                  (pipe_fragments_in_one_round), or the alternating one
//                                                                  (alternate_fragments)
// With a workspace the products of up to 64 rows that vk_gemm_split_preferred names go through chunk sums
// instead (the caller's choice: vk_gemm_split).
static int choose_gemm_kernel(int M, int N, int K) {
  const int cus = vk_device_cus();
  const int wg16 = (N + 15) / 16, wg32 = (N + 31) / 32, wg64 = (N + 63) / 64, wg128 = (N + 127) / 128;
  const bool whole = K % KC == 0, k_resident = K <= SK_WAVES * KC;
  const bool many16 = 2 * wg16 >= 3 * cus;
  if (M <= 16) return 1;
  if (M <= 64 && whole) {
    if (4 * wg128 >= 3 * cus) return 10;
    if (2 * wg64 >= cus) return 8;
    if (M > 32 && 2 * wg32 <= cus && (M > 40 || !k_resident)) return 12;
    if (M > 40) return 9;
    if (k_resident || wg16 <= cus) return many16 ? 7 : 1;
    return 9;
  }
  if (M <= 64) return (2 * wg128 >= cus && M > 32) ? 2 : (many16 ? 7 : 1);
  if (sizeof(elem_t) == 2 && M <= 128 && whole && 2 * wg128 < cus) {
    if (2 * wg32 <= cus && K > 2 * KC) return 9;
    return M > 112 && K >= 10 * KC && 2 * wg64 <= cus ? 8 : 2;
  }
  return 2;
}

// How many weight rows a tile of gemm_lines_kernel has for a product of these sizes (8 or 4), or 0: a streaming kernel is the faster one.
// Measured over 2,233 sizes (N of 256 to 32,768, K of 512 to 6,144, 1 to 16 rows, with and without SwiGLU): 30.9 ms with the streaming kernels, 27.4 with the
// better one everywhere.  With tiles of 16 weight rows for the streaming kernel's workgroups:
//   at most one for two compute units     whole lines from two chunks on (1.0 to 2.4 times; nine rows and more of two chunks without SwiGLU 0.94 to 1.04: from three)
//   up to one a compute unit             the streaming kernel asks for all it needs at once and has no second tile: 0.85 to 1.03 below eight chunks (five
//                                         with SwiGLU, up to seven), 0.99 to 1.11 from there on
//   more                                 the streaming kernel's last round is partly empty: 1.0 to 1.45 from four chunks on (with SwiGLU from two, up to eight
//                                         rows); only where two rounds are just filled and nine rows and more 0.94 to 0.98 below eight chunks
// Tiles of eight rows, or of four where those of eight leave more than half of the units without one, or do not fit.
static int lines_rows(int M, int N, int K, int projections) {
#ifdef VK_BF16
  if (M > 16 || K % KC != 0) return 0;
  const int cus = vk_device_cus(), chunks = K / KC, tiles16 = (N + 15) / 16;
  const bool swiglu = projections == 2;
  if (2 * tiles16 <= cus) {
    if (chunks < 2 || (!swiglu && chunks == 2 && M > 8)) return 0;
  } else if (tiles16 <= cus) {
    if (swiglu ? chunks < 5 || chunks > 7 : chunks < 8) return 0;
  } else {
    if (chunks < (swiglu && M <= 8 ? 2 : 4)) return 0;
    if (!swiglu && M > 8 && chunks < 8 && tiles16 <= 2 * cus && 16 * tiles16 > 30 * cus) return 0;
  }
  LinePlan plan;
  int lds = 0;
  if (N > 2 * cus && line_plan(M, K, 8, projections, &plan, &lds)) return 8;
  return line_plan(M, K, 4, projections, &plan, &lds) ? 4 : 0;
#else
  (void)M; (void)N; (void)K; (void)projections;
  return 0;
#endif
}

// How many 16-row weight fragments a wave of the tile kernel takes (a workgroup: 32 of them in weight rows).  The
// kernel's time goes in rounds of the workgroups that the device holds at once, two per compute unit: a last round
// that is nearly empty costs almost a whole one (0.72 of one up to half full, where every workgroup has its unit
// to itself).  A round costs 0.9, 1 and 1.25 times the square tile's with 96, 128 and 160 weight rows (measured at
// 1,024 to 8,192 rows on 4,096 to 10,240 weight rows); another width is taken when that makes the sum 3 % smaller:
// 5,120 weight rows at 2,048 rows are 1.25 rounds of 128 or one of 160 (5,120 x 5,120: 121 -> 93 us, 5,120 x
// 17,408: 452 -> 337, 5,120 x 25,600: 705 -> 481), 6,144 weight rows at 1,024 rows 0.75 rounds of 128 or one of 96
// (62 -> 53 us).
static int pipe_fragments_by_rounds(int M, int N, double* rounds_of_128 = nullptr) {
  static const double round_cost[6] = {0, 0, 0, 0.9, 1.0, 1.25};
  const double slots = 2.0 * vk_device_cus();
  const int mb = (M + 127) / 128;
  auto estimate = [&](int f) {
    const double rounds = (double)((N + 32 * f - 1) / (32 * f)) * mb / slots;
    const double whole = std::floor(rounds), part = rounds - whole;
    return round_cost[f] * (whole + (part == 0 ? 0.0 : (part <= 0.5 ? 0.72 : 1.0)));
  };
  int best = 4;
  double least = 0.97 * estimate(4);
  for (int f : {3, 5}) {
    const double e = estimate(f);
    if (e < least) {
      least = e;
      best = f;
    }
  }
  if (rounds_of_128) *rounds_of_128 = estimate(best);
  return best;
}

// How many weight fragments a wave of the tile kernel takes where that leaves no compute unit with more than one workgroup (2, 3 or 4), or 0.
// A workgroup that is alone on its unit has only its own stages to cover the way from memory, and two tiles of 32 KB do not: four stages (96 to 128
// KB of LDS, which it has to itself) keep three on their way, and of the tiles that give one round the narrowest puts most units to work.  Measured
// on MI355X in recorded launches with the weights of several layers in turn, against 64 weight rows with two stages that touch their lines four
// tiles ahead (below 257 rows: the kernels that share activations through LDS), us: 4,096 x 12,288, 130 rows 74 -> 68, 512 rows 126 -> 81, 1,000 rows
// (96 weight rows) 145 -> 114; 6,144 x 4,096, 300 rows 51 -> 33; 2,048 x 6,144, 651 rows 53 -> 36; 1,024 x 1,024, 65 to 1,024 rows 9.7 to 10.7 -> 8.6;
// with SwiGLU 9,728 x 2,560, 100 rows 47 -> 34; grouped, 2,048 x 2,048, 16 blocks 37 -> 27.  556 plain sizes of 65 to 2,048 rows (N of 1,024 to
// 16,384, K of 1,024 to 12,288) 25.8 -> 19.6 ms (three of them 3 to 5 % slower: 128 rows, 5,120 to 8,192 x 6,144), 102 with SwiGLU 3.21 -> 2.73.
// Three stages are 5 % slower with 64 weight rows and as fast with 96 and 128, five and six are slower.
static int pipe_fragments_in_one_round(int M, int N, int K) {
  const int64_t mb = (M + 127) / 128;
  if ((N + 63) / 64 * mb <= vk_device_cus()) return 2;
  if ((N + 95) / 96 * mb <= vk_device_cus()) return 3;
  // 32-bit elements (which the smaller tiles of gemm_fine_kernel leave with more workgroups than that only), K of up to two chunks and K not in whole chunks are as fast with two
  // workgroups of 64 rows a unit (two stages).
  if (sizeof(elem_t) == 2 && K % KC == 0 && K > 2 * KC && (N + 127) / 128 * mb <= vk_device_cus()) return 4;
  return 0;
}

#ifdef VK_F32
// Which products go by gemm_fine_kernel's tiles or by those of 128 rows (fine_tile says which).  Whole chunks: up to 64 rows the kernels that share activations through LDS are
// ahead where K is long (those kernels against these tiles, us: 64 rows, 1,024 x 1,024 17.4, 11.5, 3,072 x 1,536 19.1, 16.5, 2,048 x 2,048 18.3, 20.2, 4,096 x 12,288 100, 128; with SwiGLU 6,144 x 2,048 64, 52,
// 12,288 x 4,096 175, 130), up to 32 rows always (20 rows, 4,096 x 1,024 11.0, 11.2, 2,048 x 6,144 36.6, 59.3); from 65 rows on they are nowhere by more than 2 % (350 sizes of 65
// to 256 rows, 256 x 1,024 to 12,288 x 12,288: 1.45 times as fast on the mean; 65 rows, 4,096 x 12,288 147, 136, 128 rows, 8,192 x 8,192 181, 184).  K not in whole chunks, 33 to 64
// rows: the streaming kernels share K among eight waves, which few weight rows need (48 rows and fewer, K of two to three chunks: 33 rows, 1,024 x 1,504 14.1, 17.3, 4,096 x 1,504 16.4,
// 18.6, 5,840 x 1,280 29.4, 20.1; 64 rows, 2,048 x 1,280 18, 15.3), and K above three chunks up to as many as tiles of 128 fill half of the units; there it was tiles of 128
// x 64 (64 rows, 16,384 x 2,080 76.9, 48.6, 6,176 220, 138).
static bool fine_takes(int M, int N, int K, int64_t lda, bool swiglu) {
  if (K % (2 * VK_SLAB) != 0 || rows_far(lda) || M <= 32) return false;
  if (M > 64) return true;
  const int cus = vk_device_cus();
  if (K % KC == 0) return swiglu || K <= 3 * KC;
  if (K > 3 * KC) return 2 * ((N + 127) / 128) >= cus;
  return K <= 2 * KC || M > 48 || (N + 15) / 16 > cus;
}
// The tile whose launch ends first: a unit's share is ceil(tiles / units) tiles, a tile's time is its products' (FM x FN fragments), and below a share that depends
// on the tile a K tile's wait for memory.  ns for 32 elements of K and a product of fragments, fitted to 84 products of 70 to 2,048 rows, 256 x 1,024 to
// 12,288 x 2,048: {at least, in front, a tile}.  The tile so chosen against the best of the six: 2 % slower on the mean, 20 % at most (645 products of up to 20,480 x 4,096).
// false: a tile of 128 rows by gemm_pipe_kernel is the faster one (M above 64, and not where those leave units with one workgroup).  Larger tiles are ahead where they fill
// the units' rounds: 512 rows, 10,240 x 2,080, 256 tiles of 128 x 160 172 us, small ones 189; 2,048 rows, 4,096 x 544, 1,024 of 128 x 128 72.2, 86.2; with SwiGLU 512 rows,
// 8,192 x 544 73.3, 85.3.  Their time, good to 2 %: two workgroups a unit (three with 64 weight rows) at a time, a round's fixed cost, and
// {in front, a tile} as above.  The small tiles' is good to 10 %, hence the factors, by which 15 of 2,619 products (33 to 2,048 rows) take 3 to 8 % longer
// than without small tiles, all but three of them of K up to 544; with small ones alone 42 of 900 take 3 to 16 % longer.
static bool fine_tile(int M, int N, int K, bool swiglu, int& fm, int& fn) {
  static const struct { int fm, fn; double least, front, each; } kinds[6] = {{2, 4, 140, 10, 121}, {3, 2, 147, 15, 121}, {2, 2, 160, 20, 124},
                                                                               {1, 4, 175, 20, 129}, {1, 2, 250, 50, 134}, {1, 1, 320, 180, 142}};
  auto share = [](int64_t tiles) { return (tiles + vk_device_cus() - 1) / vk_device_cus(); };
  double best = 0.0;
  for (const auto& k : kinds) {
    if (swiglu && k.fn == 1) continue;
    const int columns = (swiglu ? 16 : 32) * k.fn;
    const int64_t tiles = (int64_t)((M + 32 * k.fm - 1) / (32 * k.fm)) * ((N + columns - 1) / columns);
    const double time = k.fm * k.fn * std::max(k.least, k.front + k.each * (double)share(tiles));
    if (best == 0.0 || time < best) { best = time; fm = k.fm; fn = k.fn; }
  }
  if (M <= 64) return true;
  best *= K / 32 * 1e-3;                                             // us
  const int64_t row_blocks = (M + 127) / 128;
  auto tall = [&](int products, int64_t tiles, int resident, double front, double each, double round) {
    const int64_t rounds = share(tiles) / resident, rest = share(tiles) % resident;
    return products * (K / 32) * 1e-3 * ((double)rounds * (front + each * resident) + (rest ? std::max(120.0, front + each * (double)rest) : 0.0)) +
           round * (double)(rounds + (rest > 0));
  };
  if (swiglu) {
    const int64_t tiles = row_blocks * ((N + 63) / 64);
    return tall(16, tiles, 2, 17, 109, 5.3) >= (share(tiles) == 2 ? 1.05 : 1.0) * best;
  }
  if (pipe_fragments_in_one_round(M, N, K) != 0) return true;
  if ((N + 127) / 128 * row_blocks <= vk_device_cus()) return tall(8, row_blocks * ((N + 63) / 64), 3, 3, 119, 4.3) >= 1.06 * best;
  const int f = pipe_fragments_by_rounds(M, N);
  const int64_t tiles = row_blocks * ((N + 32 * f - 1) / (32 * f));
  return tall(4 * f, tiles, 2, 17, 109, 5.3) >= (100 * tiles >= 95 * share(tiles) * vk_device_cus() ? 1.14 : 1.06) * best;
}
#endif

#ifdef VK_BF16
// How many weight fragments a wave of the alternating kernel takes (6, 5 or 4), or 0: the tile kernel is the faster one.  Both kernels' times go in
// rounds of the workgroups that run at a time, one a compute unit here; with k = K / 1,024 a round was measured at 13.1 k + 7, 15.8 k + 6 and
// 18.9 k + 8 us for 128, 160 and 192 columns, at 15 k + 4.5 for the tile kernel's round of as much as the first, and a last round at 0.64 + 0.33
// of its filled part.
static int alternate_fragments(int M, int N, int K, bool swiglu) {
  if (M < 256 || K % KC != 0 || N < (swiglu ? 96 : 192)) return 0;
  const int cus = vk_device_cus(), out_cols = swiglu ? 2 * N : N;
  // At most one workgroup a compute unit of the tile kernel's: its round is shorter then than a full one's 0.72, and has four stages (1,536 x 2,048 with SwiGLU, 256 to 512
  // rows: 22 to 23 us against 30).  The plain product's caller has asked that before.
  if (swiglu && (int64_t)((N + 63) / 64) * ((M + 127) / 128) <= cus) return 0;
  static const double slope[7] = {0, 0, 0, 0, 13.1, 15.8, 18.9}, start[7] = {0, 0, 0, 0, 7, 6, 8};
  const double k = K / 1024.0;
  double rounds = 0;
  if (swiglu) {
    const double r = (double)((N + 63) / 64) * ((M + 127) / 128) / (2.0 * cus), whole = std::floor(r), part = r - whole;
    rounds = whole + (part == 0 ? 0.0 : (part <= 0.5 ? 0.72 : 1.0));
  } else {
    pipe_fragments_by_rounds(M, N, &rounds);
  }
  double least = 0.97 * rounds * (15.0 * k + 4.5);
  int best = 0;
  for (int f = 6; f >= 4; --f) {
    if (swiglu && f == 5) continue;
    const double r = (double)((out_cols + 32 * f - 1) / (32 * f)) * ((M + 255) / 256) / cus, whole = std::floor(r), part = r - whole;
    const double e = (whole + (part == 0 ? 0.0 : 0.64 + 0.33 * part)) * (slope[f] * k + start[f]);
    if (e < least) {
      least = e;
      best = f;
    }
  }
  return best;
}
#endif

extern "C" {

// The element type's activation code in a product's entry point: 0 none, 1 the square of max(., 0) on the rounded sums (the bits
// of the plain product followed by vk_moe_relu_square).
static int out_form_of(const elem_t* out, int64_t ldo, int activation) {
  return ((ldo % 4 == 0) && ((uintptr_t)out % 16 == 0) ? OUT_VEC : 0) | (activation == 1 ? OUT_SQUARED_RELU : 0);
}

static int experts_refuse(const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, const int32_t* order, int matrices, int64_t weights_stride,
                          const int32_t* act_row, int act_rows, bool gated) {
  VK_REQUIRE(sizeof(elem_t) == 2, "experts' product: 16-bit elements");
  VK_REQUIRE(M >= 0 && M % 128 == 0 && N >= (gated ? 128 : 256) && K > 0 && K % KC == 0, "experts' product: bad sizes M=%d N=%d K=%d", M, N, K);
  VK_REQUIRE(lda >= K && lda % VK_VEC == 0 && ldo >= N, "experts' product: bad row strides");
  VK_REQUIRE(((uintptr_t)act % 16) == 0 && ((uintptr_t)w % 16) == 0 && weights_stride % VK_VEC == 0, "experts' product: operands must be 16-byte aligned");
  VK_REQUIRE(order != nullptr && (uintptr_t)order % 16 == 0 && matrices > 0, "experts' product: a plan's order is needed");
  VK_REQUIRE(act_row != nullptr ? act_rows > 0 && (int64_t)act_rows * lda * (int64_t)sizeof(elem_t) < ((int64_t)1 << 31) : !rows_far(lda, EXPERT_PART_ROWS),
             "experts' product: rows too far apart");
  return 0;
}

// A grouped product through the tile kernel: rows in blocks of 128, block b multiplied by the weight matrix
// block_weights[b] of several [N, K] matrices that lie weights_stride elements apart (negative: the block is skipped and
// its output rows are left as they are).  K in whole pairs of slabs (128 bytes of a row).  The same bits as vk_gemm gives
// for the same rows and matrix.  row_pair [M] or null: a block whose row 64 has a negative entry has no rows from there on, and its
// outputs there are left as they are.  act_row [M] or null: row r of the product is row act_row[r] of act, which has act_rows rows
// (fewer than 2^31 bytes); all entries must lie in 0 .. act_rows - 1, those of rows without a pair too.
// This spares the rows' copy in the order of the product: 32 us, of 535 with the product (2,048 tokens x 3 choices, 6,144 x 4,096 weights);
// the product itself, which then finds a token's row in the caches for each of its experts, 505 -> 472 us.
// matrices: how many w holds, or 0 where the caller does not say; it only helps to choose the kernel (grouped_wide).
int vk_gemm_grouped_experts(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo,
                            const int32_t* block_weights, int64_t weights_stride, int matrices, const int32_t* row_pair, const int32_t* act_row,
                            int act_rows, int activation, hipStream_t st) {
  VK_REQUIRE(activation == 0 || activation == 1, "grouped gemm: unknown activation %d", activation);
  VK_REQUIRE(M >= 0 && N > 0 && K > 0 && M % 128 == 0, "grouped gemm: bad sizes M=%d N=%d K=%d (rows in blocks of 128)", M, N, K);
  VK_REQUIRE(K % (2 * VK_SLAB) == 0, "grouped gemm: K=%d must be a multiple of %d", K, 2 * VK_SLAB);
  VK_REQUIRE(lda >= K && lda % VK_VEC == 0 && ldo >= N, "grouped gemm: bad row strides");
  VK_REQUIRE(((uintptr_t)act % 16) == 0 && ((uintptr_t)w % 16) == 0 && block_weights != nullptr && weights_stride % VK_VEC == 0,
             "grouped gemm: operands must be 16-byte aligned");
  VK_REQUIRE(act_row == nullptr || (act_rows > 0 && (int64_t)act_rows * lda * (int64_t)sizeof(elem_t) < ((int64_t)1 << 31)),
             "grouped gemm: %d rows to choose from", act_rows);
  if (M == 0) return 0;
  return launch_pipe<2, false, 4, true>(out, act, w, M, N, K, lda, ldo, out_form_of(out, ldo, activation), st, block_weights, weights_stride, row_pair, act_row,
                                         matrices);
}

// Whether vk_gemm_experts (gated: vk_gemm_experts_glu) takes a product of this size: rows as vk_gemm_grouped_experts counts them.
int vk_gemm_experts_takes(int M, int N, int K, int64_t lda, int matrices, int gated) {
#ifdef VK_BF16
  return experts_takes(M, N, K, lda, matrices, gated != 0);
#else
  return 0;
#endif
}

// The experts' product by a plan's order (vk_moe_route_plan_ordered) instead of its blocks: act, w, act_row and activation as in
// vk_gemm_grouped_experts, whose bits it gives.  Rows of out that no pair has are left as they are.
int vk_gemm_experts(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, const int32_t* order, int matrices,
                    int64_t weights_stride, const int32_t* act_row, int act_rows, int activation, hipStream_t st) {
  VK_REQUIRE(activation == 0 || activation == 1, "experts' product: unknown activation %d", activation);
  if (experts_refuse(act, w, M, N, K, lda, ldo, order, matrices, weights_stride, act_row, act_rows, false)) return 1;
  if (M == 0) return 0;
#ifdef VK_BF16
  return launch_experts<false>(out, act, w, M, N, K, lda, ldo, out_form_of(out, ldo, activation), order, matrices, weights_stride, act_row, GluArgs{}, st);
#else
  return 1;
#endif
}

// The same for matrices of F gate rows and then F up rows, out [., F]: the gated activation (moe_glu_kernel) of the product's elements.
// wts, row_pair (both or neither): as in vk_moe_glu_weighed.
int vk_gemm_experts_glu(elem_t* out, const elem_t* act, const elem_t* w, int M, int F, int K, int64_t lda, int64_t ldo, const int32_t* order, int matrices,
                        int64_t weights_stride, const int32_t* act_row, int act_rows, float limit, float slope, float shift, const int32_t* row_pair,
                        const float* wts, hipStream_t st) {
  VK_REQUIRE(limit > 0.f && (row_pair == nullptr) == (wts == nullptr), "experts' product: a positive limit, rows' pairs and weights or neither");
  if (experts_refuse(act, w, M, F, K, lda, ldo, order, matrices, weights_stride, act_row, act_rows, true)) return 1;
  if (M == 0) return 0;
#ifdef VK_BF16
  return launch_experts<true>(out, act, w, M, F, K, lda, ldo, out_form_of(out, ldo, 0), order, matrices, weights_stride, act_row, {limit, slope, shift, row_pair, wts}, st);
#else
  return 1;
#endif
}

int vk_gemm_grouped_rows(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo,
                         const int32_t* block_weights, int64_t weights_stride, const int32_t* row_pair, const int32_t* act_row, int act_rows,
                         int activation, hipStream_t st) {
  return vk_gemm_grouped_experts(out, act, w, M, N, K, lda, ldo, block_weights, weights_stride, 0, row_pair, act_row, act_rows, activation, st);
}

int vk_gemm_grouped_act(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo,
                        const int32_t* block_weights, int64_t weights_stride, const int32_t* row_pair, int activation, hipStream_t st) {
  return vk_gemm_grouped_rows(out, act, w, M, N, K, lda, ldo, block_weights, weights_stride, row_pair, nullptr, 0, activation, st);
}

// kernel: 0 = choose by size, 1 = skinny (M <= 64), 2 = tiled (pipelined if K allows), 3 = tiled through
// registers, 4..6 = pipelined with 2..4 stages, 7 = skinny with two weight tiles per workgroup where it has
// such a variant, 8, 9 and 10 = activations shared through LDS with 64, 32 and 128 weight rows per workgroup
// (17 to 512 rows, in blocks of 64 rows), 11 = skinny with two activation tiles resident in registers (17 to
// 32 rows of 16-bit elements, K <= 4096), 12 = as 9 in blocks of 32 rows, 13, 15 and 16 = pipelined with 64, 96
// and 160 weight rows per workgroup (14 is the callers' name for the route through chunk sums), 17, 18 and 19 = alternating
// with 192, 160 and 128 weight rows per workgroup (256 rows or more, 16-bit elements, K a multiple of 512), 20 and 21 = whole lines in
// tiles of 4 and 8 weight rows (1 to 16 rows, 16-bit elements, K a multiple of 512 up to 6,144 and as many rows as fit the LDS); for measurements and tests.  The result does not depend on the choice.
static int gemm_launch(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo,
                       int kernel, int activation, hipStream_t st) {
  VK_REQUIRE(activation == 0 || activation == 1, "gemm: unknown activation %d", activation);
  VK_REQUIRE(M >= 0 && N > 0 && K > 0, "gemm: bad sizes M=%d N=%d K=%d", M, N, K);
  VK_REQUIRE(K % VK_VEC == 0, "gemm: K=%d must be a multiple of %d for this element type", K, VK_VEC);
  VK_REQUIRE(lda >= K && lda % VK_VEC == 0, "gemm: activation row stride %lld must be >= K and a multiple of %d",
             (long long)lda, VK_VEC);
  VK_REQUIRE(ldo >= N, "gemm: output row stride %lld is smaller than N=%d", (long long)ldo, N);
  VK_REQUIRE(((uintptr_t)act % 16) == 0 && ((uintptr_t)w % 16) == 0, "gemm: operands must be 16-byte aligned");
  VK_REQUIRE(kernel >= 0 && kernel <= (sizeof(elem_t) == 2 ? 21 : 16) && kernel != 14, "gemm: unknown kernel %d", kernel);      // the alternating one takes 16-bit elements
  if (M == 0) return 0;
  const int form = out_form_of(out, ldo, activation);
  const bool by_size = kernel == 0;
#ifdef VK_F32
  if (kernel == 0 && fine_takes(M, N, K, lda, false)) {
    int fm = 0, fn = 0;
    if (fine_tile(M, N, K, false, fm, fn)) return gemm_fine(fm, fn, false, out, act, w, M, N, K, lda, ldo, form, st);
  }
#endif
  if (kernel == 0) {
#ifdef VK_BF16
    const int width = rows_width(M, N, K, lda, false);
    if (width) return gemm_rows(width, false, out, act, w, M, N, K, lda, ldo, form, st);
#endif
    const int rows = lines_rows(M, N, K, 1);
    kernel = rows ? (rows == 4 ? 20 : 21) : choose_gemm_kernel(M, N, K);
  }
#ifdef VK_BF16
  if (kernel == 17) return launch_alternate<6, 2, 3>(out, act, w, M, N, K, lda, ldo, form, st);
  if (kernel == 18) return launch_alternate<5, 3, 3>(out, act, w, M, N, K, lda, ldo, form, st);
  if (kernel == 19) return launch_alternate<4, 3, 4>(out, act, w, M, N, K, lda, ldo, form, st);
#endif
#ifdef VK_BF16
  if (kernel == 20) return launch_lines<4, 1>(out, act, w, M, N, K, lda, ldo, form, st);
  if (kernel == 21) return launch_lines<8, 1>(out, act, w, M, N, K, lda, ldo, form, st);
#endif
  if (kernel == 12) {      // 32 weight rows per workgroup, four chunks in work, blocks of 32 rows
    VK_REQUIRE(M > 16 && M <= 512 && K % KC == 0, "gemm: the mid kernel takes 17 to 512 rows and K a multiple of %d", KC);
    return launch_mid<2, 4>(out, act, w, M, N, K, lda, ldo, form, st);
  }
  if (kernel >= 8 && kernel <= 10) {
    VK_REQUIRE(M > 16 && M <= 512 && K % KC == 0, "gemm: the mid kernel takes 17 to 512 rows and K a multiple of %d", KC);
    const int mt = M > 64 ? 4 : (M + 15) / 16;       // more than 64 rows: blocks of 64
    if (kernel == 10) {     // 128 weight rows per workgroup, every wave all chunks of its tile
      if (mt == 2) return launch_mid<2, 1>(out, act, w, M, N, K, lda, ldo, form, st);
      return launch_mid<4, 1>(out, act, w, M, N, K, lda, ldo, form, st);
    }
    if (kernel == 8) {      // 64 weight rows per workgroup, two chunks in work
      if (mt == 2) return launch_mid<2, 2>(out, act, w, M, N, K, lda, ldo, form, st);
      if (mt == 3) return launch_mid<3, 2>(out, act, w, M, N, K, lda, ldo, form, st);
      return launch_mid<4, 2>(out, act, w, M, N, K, lda, ldo, form, st);
    }
    // 32 weight rows per workgroup, four chunks in work
    if (mt == 2) return launch_mid<2, 4>(out, act, w, M, N, K, lda, ldo, form, st);
    if (mt == 3) return launch_mid<3, 4>(out, act, w, M, N, K, lda, ldo, form, st);
    return launch_mid<4, 4>(out, act, w, M, N, K, lda, ldo, form, st);
  }
  if (kernel == 11)
    VK_REQUIRE(M > 16 && M <= 32 && K % KC == 0 && K <= SK_WAVES * KC && sizeof(elem_t) == 2,
               "gemm: resident activations of two tiles need 17 to 32 rows of 16-bit elements and K a multiple of %d up to %d", KC, SK_WAVES * KC);
  if (kernel == 1 || kernel == 7 || kernel == 11) {
    VK_REQUIRE(M <= 64, "gemm: the skinny kernel takes at most 64 rows, got %d", M);
    const int mt = (M + 15) / 16;
    const unsigned grid = (unsigned)((N + 15) / 16);
    if (K % KC == 0) {
#define STH(MT, W, RC, NT, NW, ROWS)                                                                    \
  do {                                                                                                    \
    constexpr size_t rows_bytes = (size_t)NW * CHUNK_ROWS_BYTES(ROWS);                                \
    static int resident = 0; /* workgroups of this kernel that the device holds at once */               \
    if (resident == 0) {                                                                                  \
      int dev = 0, cus = 0, per_cu = 0;                                                                   \
      (void)hipGetDevice(&dev);                                                                           \
      (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);                      \
      if (rows_bytes)                                                                                     \
        (void)hipFuncSetAttribute((const void*)gemm_stream_kernel<MT, W, RC, NT, NW, ROWS>,             \
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)rows_bytes);           \
      (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, gemm_stream_kernel<MT, W, RC, NT, NW, ROWS>, \
                                                         64 * NW, rows_bytes);                            \
      resident = (cus > 0 ? cus : 256) * (per_cu > 0 ? per_cu : 1);                                       \
    }                                                                                                     \
    const unsigned groups = (unsigned)((N + 16 * NT - 1) / (16 * NT));                                    \
    gemm_stream_kernel<MT, W, RC, NT, NW, ROWS><<<groups < (unsigned)resident ? groups : (unsigned)resident, \
                                             64 * NW, rows_bytes, st>>>(out, act, w, M, N, K, lda, ldo, form, NormArgs{}); \
  } while (0)
#define STW(MT, W, RC, NT, NW) STH(MT, W, RC, NT, NW, 0)
// Where as many rows do not fit beside the sums, stream_lds_rows names the kernel without them instead: nothing is compiled for a branch that is not taken.
#define STN(NW)                                                                                           \
  do {                                                                                                    \
    const int rows = stream_rows_pay(M, (N + 15) / 16, lda, K / KC) ? stream_lds_rows(M, NW, NW * 2048) : 0;   \
    if (rows == 16) STH(1, 8, 1, 1, NW, stream_lds_rows(16, NW, NW * 2048));                              \
    else if (rows == 8) STH(1, 8, 1, 1, NW, stream_lds_rows(8, NW, NW * 2048));                           \
    else if (rows == 4) STH(1, 8, 1, 1, NW, 4);                                                           \
    else if (rows == 1) STH(1, 8, 1, 1, NW, 1);                                                           \
    else STH(1, 8, 1, 1, NW, 0);                                                                          \
  } while (0)
#define ST(MT, W, RC, NT) STW(MT, W, RC, NT, SK_WAVES)
      if (mt == 1) {
        // A few weight tiles more than workgroups in flight (one per compute unit) would mean a second
        // pass of a few: two tiles a workgroup then finish sooner (16 rows, 5120 x 25600: 111 -> 86 us),
        // unless one chunk a wave keeps the activations in registers (6144 x 4096: 12.6 against 15.7 us).
        const int cus = vk_device_cus();
        const int tiles16 = (N + 15) / 16;
        // One chunk a wave, its activations in registers, wherever a workgroup can have as many waves as K has
        // chunks (stream_waves): no wave then waits at the round's barrier for one that has a second chunk.
        const int nw = kernel == 7 ? SK_WAVES : stream_waves(K / KC);
        if (nw == 2) STN(2);
        else if (nw == 4) STN(4);
        else if (nw == 5) STN(5);
        else if (nw == 6) STN(6);
#ifdef VK_BF16
        else if (nw == 10) STW(1, 8, 1, 1, 10);         // nine rows and more (lines_rows takes the others), which do not fit the LDS
        else if (nw == 12) STW(1, 8, 1, 1, 12);
#endif
        else
        if (kernel == 7 || (by_size && K > SK_WAVES * KC && tiles16 > cus && 2 * tiles16 <= 3 * cus)) ST(1, 8, 0, 2);
        else if (K <= SK_WAVES * KC) STN(SK_WAVES);
#ifdef VK_BF16
        // Two chunks a wave are 128 registers of activations (16 rows, 34816 x 5120: 118 -> 87 us);
        // three did not fit beside the rest and were slower than none (4096 x 12288: 29 -> 36 us).
        else if (K <= 2 * SK_WAVES * KC) ST(1, 8, 2, 1);
#endif
        else {
#ifdef VK_BF16
          // Not in 32-bit: the rows held are twice as many registers there (4,096 x 4,608, 8 rows 22.7 -> 29.4 us; 7,168 x 5,120, 4 rows 35.7 -> 40.2).
          const int rows = stream_rows_pay(M, tiles16, lda) ? stream_lds_rows(M, SK_WAVES, SK_WAVES * 2048) : 0;
          if (rows == 16) STH(1, 8, 0, 1, SK_WAVES, stream_lds_rows(16, SK_WAVES, SK_WAVES * 2048));
          else if (rows == 8) STH(1, 8, 0, 1, SK_WAVES, 8);
          else if (rows == 4) STH(1, 8, 0, 1, SK_WAVES, 4);
          else if (rows == 1) STH(1, 8, 0, 1, SK_WAVES, 1);
          else
#endif
          ST(1, 8, 0, 1);
        }
      }
      else if (mt == 2) {
#ifdef VK_BF16
        if (kernel == 11) ST(2, 8, 1, 1);
        else
#endif
        if (kernel == 7) ST(2, 4, 0, 2);
        else ST(2, 8, 0, 1);
      }
      else if (mt == 3) { if (kernel == 7) ST(3, 4, 0, 2); else ST(3, 4, 0, 1); }
      else { if (kernel == 7) ST(4, 4, 0, 2); else ST(4, 4, 0, 1); }
#undef ST
#undef STN
#undef STW
#undef STH
      return vk_check_launch("gemm_stream");
    }
#define SK(MT, W) gemm_skinny_kernel<MT, W><<<grid, 64 * SK_WAVES, 0, st>>>(out, act, w, M, N, K, lda, ldo, form)
    // Few weight rows leave one workgroup per compute unit: a deeper window keeps its memory pipe full.
    if (mt == 1) { if (N <= 8192) SK(1, 16); else SK(1, 8); }
    else if (mt == 2) SK(2, 8);
    else if (mt == 3) SK(3, 4);
    else SK(4, 4);
#undef SK
    return vk_check_launch("gemm_skinny");
  }
  const bool k_whole = K % (2 * VK_SLAB) == 0 && !rows_far(lda);
  if (kernel == 3) return launch_tiled<4, 4>(out, act, w, M, N, K, lda, ldo, form, st);
  if (kernel == 4 && k_whole) return launch_pipe<2>(out, act, w, M, N, K, lda, ldo, form, st);
  if (kernel == 5 && k_whole) return launch_pipe<3>(out, act, w, M, N, K, lda, ldo, form, st);
  if (kernel == 6 && k_whole) return launch_pipe<4>(out, act, w, M, N, K, lda, ldo, form, st);
  // Two stages of 32 KB leave room for two workgroups per compute unit, which hides more latency than a third stage.
  if (k_whole) {
#ifdef VK_BF16
    if (by_size) {
      const int f = pipe_fragments_in_one_round(M, N, K);
      if (f == 2) return launch_pipe<4, false, 2>(out, act, w, M, N, K, lda, ldo, form, st);
      if (f == 3) return launch_pipe<4, false, 3>(out, act, w, M, N, K, lda, ldo, form, st);
      if (f == 4) return launch_pipe<4>(out, act, w, M, N, K, lda, ldo, form, st);
    }
#endif
    // No more 128 x 128 tiles than compute units: 64 weight rows a workgroup, twice as many of them.
    const int64_t tiles = (int64_t)((N + 127) / 128) * ((M + 127) / 128);
    if (kernel == 13 || (by_size && tiles <= vk_device_cus())) return launch_pipe<2, false, 2>(out, act, w, M, N, K, lda, ldo, form, st);
#ifdef VK_BF16
    if (by_size) {
      const int f = alternate_fragments(M, N, K, false);
      if (f == 6) return launch_alternate<6, 2, 3>(out, act, w, M, N, K, lda, ldo, form, st);
      if (f == 5) return launch_alternate<5, 3, 3>(out, act, w, M, N, K, lda, ldo, form, st);
      if (f == 4) return launch_alternate<4, 3, 4>(out, act, w, M, N, K, lda, ldo, form, st);
    }
#endif
    const int fragments = kernel == 15 ? 3 : (kernel == 16 ? 5 : (by_size ? pipe_fragments_by_rounds(M, N) : 4));
    if (fragments == 3) return launch_pipe<2, false, 3>(out, act, w, M, N, K, lda, ldo, form, st);
    if (fragments == 5) return launch_pipe<2, false, 5>(out, act, w, M, N, K, lda, ldo, form, st);
    return launch_pipe<2>(out, act, w, M, N, K, lda, ldo, form, st);
  }
  return launch_tiled<4, 4>(out, act, w, M, N, K, lda, ldo, form, st);
}

// A product of 32-bit elements by tiles of 32 fm x 32 fn (0, 0: the ones chosen by size), for measurements and tests.
int vk_gemm_fine(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int fm, int fn, int swiglu, hipStream_t st) {
  VK_REQUIRE(sizeof(elem_t) == 4 && M > 0 && N > 0 && K > 0 && K % (2 * VK_SLAB) == 0 && lda >= K && lda % VK_VEC == 0 && !rows_far(lda) && ldo >= N,
             "gemm: bad sizes M=%d N=%d K=%d for tiles of 32-bit elements", M, N, K);
  VK_REQUIRE(((uintptr_t)act % 16) == 0 && ((uintptr_t)w % 16) == 0, "gemm: operands must be 16-byte aligned");
#ifdef VK_F32
  if (fm == 0) (void)fine_tile(M, N, K, swiglu != 0, fm, fn);
  return gemm_fine(fm, fn, swiglu != 0, out, act, w, M, N, K, lda, ldo, out_form_of(out, ldo, 0), st);
#else
  return 1;
#endif
}

// 1 if a product chosen by size goes by those tiles.
int vk_gemm_fine_takes(int M, int N, int K, int64_t lda, int swiglu) {
#ifdef VK_F32
  int fm = 0, fn = 0;
  return M > 0 && N > 0 && K > 0 && fine_takes(M, N, K, lda, swiglu != 0) && fine_tile(M, N, K, swiglu != 0, fm, fn);
#else
  return 0;
#endif
}

int vk_gemm(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo,
            int kernel, hipStream_t st) {
  return gemm_launch(out, act, w, M, N, K, lda, ldo, kernel, 0, st);
}

// vk_gemm (the kernel chosen by size) with an activation on the outputs.
int vk_gemm_act(elem_t* out, const elem_t* act, const elem_t* w, int M, int N, int K, int64_t lda, int64_t ldo, int activation,
                hipStream_t st) {
  return gemm_launch(out, act, w, M, N, K, lda, ldo, 0, activation, st);
}

// 1 if vk_gemm_swiglu takes these sizes (the caller otherwise runs vk_gemm and vk_swiglu, with the same result).
// 1: the streaming kernels (few rows), 2: the pipelined tile kernel (many rows), 3: the kernels for 17 to 64
// rows, 0: none.
int vk_gemm_swiglu_supported(int M, int I, int K) {
  if (M >= 1 && M <= 16 && I > 0 && K % KC == 0 && K <= SK_WAVES * KC) return 1;
#ifdef VK_BF16
  if (M >= 1 && M <= 16 && I > 0 && K % KC == 0 && K <= 2 * SK_WAVES * KC) return 1;   // two chunks a wave
#endif
  if (M > 64 && I > 0 && K % (2 * VK_SLAB) == 0) return 2;
  if (M > 16 && M <= 64 && I > 0 && K % KC == 0) return 3;      // activations shared through LDS
  return 0;
}

// out[M, I] = silu(act w_gate^T) * (act w_up^T), w = [gate rows; up rows] of shape [2I, K].
int vk_gemm_swiglu(elem_t* out, const elem_t* act, const elem_t* w, int M, int I, int K, int64_t lda, int64_t ldo,
                   hipStream_t st) {
  const int how = vk_gemm_swiglu_supported(M, I, K);
  VK_REQUIRE(how != 0, "gemm_swiglu: sizes M=%d I=%d K=%d are not supported", M, I, K);
  VK_REQUIRE(lda >= K && lda % VK_VEC == 0 && ldo >= I, "gemm_swiglu: bad row strides");
  VK_REQUIRE(((uintptr_t)act % 16) == 0 && ((uintptr_t)w % 16) == 0, "gemm_swiglu: operands must be 16-byte aligned");
#ifdef VK_BF16
  if (how == 2) {
    const int f = alternate_fragments(M, I, K, true), ok4 = (ldo % 4 == 0) && ((uintptr_t)out % 16 == 0);
    if (f == 6) return launch_alternate<6, 2, 3, true>(out, act, w, M, I, K, lda, ldo, ok4, st);
    if (f == 4) return launch_alternate<4, 3, 4, true>(out, act, w, M, I, K, lda, ldo, ok4, st);
  }
#endif
#ifdef VK_F32
  if (fine_takes(M, I, K, lda, true)) {
    int fm = 0, fn = 0;
    if (fine_tile(M, I, K, true, fm, fn))
      return gemm_fine(fm, fn, true, out, act, w, M, I, K, lda, ldo, (ldo % 4 == 0) && ((uintptr_t)out % 16 == 0), st);
  }
#endif
  if (how == 2 && rows_far(lda)) {
    VK_REQUIRE(K % KC == 0, "gemm_swiglu: rows %lld elements apart need K in whole chunks of %d", (long long)lda, KC);
    return launch_mid<4, 1, true>(out, act, w, M, I, K, lda, ldo, (ldo % 4 == 0) && ((uintptr_t)out % 16 == 0), st);
  }
  if (how == 2)
    return launch_pipe<2, true>(out, act, w, M, I, K, lda, ldo, (ldo % 4 == 0) && ((uintptr_t)out % 16 == 0), st);
#ifdef VK_BF16
  if (const int width = how == 3 ? rows_width(M, I, K, lda, true) : 0)
    return gemm_rows(width, true, out, act, w, M, I, K, lda, ldo, (ldo % 4 == 0) && ((uintptr_t)out % 16 == 0), st);
#endif
  if (how == 3) {
    const int ok4 = (ldo % 4 == 0) && ((uintptr_t)out % 16 == 0);
#ifdef VK_BF16
    // Rows too far apart for gemm_rows_kernel.
    return M <= 32 ? launch_mid<2, 1, true>(out, act, w, M, I, K, lda, ldo, ok4, st) : launch_mid<4, 1, true>(out, act, w, M, I, K, lda, ldo, ok4, st);
#else
    // Gate tiles per workgroup: of four, three and two, the number whose workgroups fill the compute units
    // best, a workgroup per unit at a time; the larger one where two fill them alike.  (Measured in 16-bit, before gemm_rows_kernel.)  64 rows, K = 4096:
    // 12288 gate rows (192, 256, 384 workgroups) 55.4, 49.7, 58.5 us; 8192 gate rows (128, 171, 256) 52.8, 47.0,
    // 41.6 us; 17408 gate rows at K = 5120 (272, 363, 544) 127.5, 108.4, 123.2 us.
    const int tiles = (I + 15) / 16, cus = vk_device_cus();
    int gt = 4;
    double best = 0.0;
    for (int g = 4; g >= 2; --g) {
      const int wgs = (tiles + g - 1) / g;
      const double filled = (double)wgs / ((double)((wgs + cus - 1) / cus) * cus);
      if (filled > best + 1e-9) { best = filled; gt = g; }
    }
    if (M <= 32) {
      if (gt == 3) return launch_mid<2, 1, true, 3>(out, act, w, M, I, K, lda, ldo, ok4, st);
      if (gt == 2) return launch_mid<2, 1, true, 2>(out, act, w, M, I, K, lda, ldo, ok4, st);
      return launch_mid<2, 1, true>(out, act, w, M, I, K, lda, ldo, ok4, st);
    }
    if (gt == 3) return launch_mid<4, 1, true, 3>(out, act, w, M, I, K, lda, ldo, ok4, st);
    if (gt == 2) return launch_mid<4, 1, true, 2>(out, act, w, M, I, K, lda, ldo, ok4, st);
    return launch_mid<4, 1, true>(out, act, w, M, I, K, lda, ldo, ok4, st);
#endif
  }
  const int ntiles = (I + 15) / 16;
  const int form = (ldo % 4 == 0) && ((uintptr_t)out % 16 == 0);
#ifdef VK_BF16
  const int lines = lines_rows(M, I, K, 2);
  if (lines == 4) return launch_lines<4, 2>(out, act, w, M, I, K, lda, ldo, form, st);
  if (lines == 8) return launch_lines<8, 2>(out, act, w, M, I, K, lda, ldo, form, st);
#endif
#define SWIGLU_STREAMH(W, RC, NW, ROWS)                                                                   \
  do {                                                                                                     \
    constexpr size_t rows_bytes = (size_t)NW * CHUNK_ROWS_BYTES(ROWS);                                \
    static int resident = 0;                                                                               \
    if (resident == 0) {                                                                                   \
      int dev = 0, cus = 0, per_cu = 0;                                                                    \
      (void)hipGetDevice(&dev);                                                                            \
      (void)hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);                       \
      if (rows_bytes)                                                                                      \
        (void)hipFuncSetAttribute((const void*)gemm_stream_swiglu_kernel<W, RC, NW, ROWS>,           \
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)rows_bytes);            \
      (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, gemm_stream_swiglu_kernel<W, RC, NW, ROWS>, \
                                                         64 * NW, rows_bytes);                             \
      resident = (cus > 0 ? cus : 256) * (per_cu > 0 ? per_cu : 1);                                        \
    }                                                                                                      \
    gemm_stream_swiglu_kernel<W, RC, NW, ROWS><<<ntiles < resident ? ntiles : resident, 64 * NW, rows_bytes, st>>>( \
        out, act, w, M, I, K, lda, ldo, form, NormArgs{});                                                \
  } while (0)
#define SWIGLU_STREAM(W, RC) SWIGLU_STREAMH(W, RC, SK_WAVES, 0)
#define SWIGLU_STREAMN(NW)                                                                                 \
  do {                                                                                                     \
    const int rows = stream_rows_pay(M, ntiles, lda) ? stream_lds_rows(M, NW, NW * 4096) : 0;                   \
    if (rows == 16) SWIGLU_STREAMH(8, 1, NW, stream_lds_rows(16, NW, NW * 4096));                       \
    else if (rows == 8) SWIGLU_STREAMH(8, 1, NW, stream_lds_rows(8, NW, NW * 4096));                    \
    else if (rows == 4) SWIGLU_STREAMH(8, 1, NW, 4);                                                    \
    else if (rows == 1) SWIGLU_STREAMH(8, 1, NW, 1);                                                    \
    else SWIGLU_STREAMH(8, 1, NW, 0);                                                                   \
  } while (0)
  const int nw = stream_waves(K / KC);       // as in vk_gemm
  if (nw == 2) SWIGLU_STREAMN(2);
  else if (nw == 4) SWIGLU_STREAMN(4);
#ifdef VK_BF16
  else if (nw == 10) SWIGLU_STREAMN(10);
  else if (nw == 12) SWIGLU_STREAMN(12);
#else
  else if (nw == 5) SWIGLU_STREAMN(5);       // 16-bit: whole lines, all of them (lines_rows)
  else if (nw == 6) SWIGLU_STREAMN(6);
#endif
  else
#ifdef VK_BF16
  if (K > SK_WAVES * KC) SWIGLU_STREAM(4, 2);
  else
#endif
    SWIGLU_STREAMN(SK_WAVES);
#undef SWIGLU_STREAMN
#undef SWIGLU_STREAMH
#undef SWIGLU_STREAM
  return vk_check_launch("gemm_swiglu");
}


// ---- products that norm their rows themselves (NormRows)
extern "C++" {
template <typename KERNEL>
static int workgroups_at_once(KERNEL kernel, int threads, int lds_bytes) {
  int n = 0;
  if (lds_bytes > 0) (void)hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds_bytes);
  (void)hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, lds_bytes);
  return (n > 0 ? n : 1) * vk_device_cus();
}
template <int ROWS, int P, int NW>
static int launch_stream_normed(elem_t* out, const elem_t* x, const elem_t* w, int M, int N, int64_t ldx, int64_t ldo, int form, const NormArgs& norm, hipStream_t st) {
  constexpr int LDS = NW * CHUNK_ROWS_BYTES(ROWS);
  const int tiles = (N + 15) / 16;
  if constexpr (P == 2) {
    static const int at_once = workgroups_at_once(gemm_stream_swiglu_kernel<8, 1, NW, ROWS, true>, 64 * NW, LDS);
    gemm_stream_swiglu_kernel<8, 1, NW, ROWS, true><<<std::min(tiles, at_once), 64 * NW, LDS, st>>>(out, x, w, M, N, NW * KC, ldx, ldo, form, norm);
  } else {
    static const int at_once = workgroups_at_once(gemm_stream_kernel<1, 8, 1, 1, NW, ROWS, true>, 64 * NW, LDS);
    gemm_stream_kernel<1, 8, 1, 1, NW, ROWS, true><<<std::min(tiles, at_once), 64 * NW, LDS, st>>>(out, x, w, M, N, NW * KC, ldx, ldo, form, norm);
  }
  return vk_check_launch("gemm_stream (normed rows)");
}
#ifdef VK_BF16
template <int R, int ROWS, int P, int NW>
static int launch_lines_normed(elem_t* out, const elem_t* x, const elem_t* w, int M, int N, int64_t ldx, int64_t ldo, int form, const NormArgs& norm, hipStream_t st) {
  LinePlan plan;
  int lds = 0;
  VK_REQUIRE(line_plan(M, NW * KC, R, P, &plan, &lds), "gemm: %d normed rows of K=%d do not fit", M, NW * KC);
  static const int at_once = workgroups_at_once(gemm_lines_kernel<R, ROWS, P, NW>, 64 * NW, lds);      // (ROWS and NW fix the LDS)
  gemm_lines_kernel<R, ROWS, P, NW><<<std::min((N + R - 1) / R, at_once), 64 * NW, lds, st>>>(out, x, w, M, N, NW * KC, ldx, ldo, form, plan, norm);
  return vk_check_launch("gemm_lines (normed rows)");
}
#endif
// How many rows, at most, are normed on their way into a product of so many chunks (0: none).  The norm is done again by every workgroup, (row, quarter) pairs a wave, so
// that it pays for few rows.  Measured as the add and norm and the product by themselves over both in one, N of 256 to 16,384, one projection and two:
//   16-bit  1 to 4 rows, K of 1 to 12 chunks        1.04 to 1.6 (a row 1.04 to 1.6, four rows 1.04 to 1.36)
//           5 and 6 rows, from 8 chunks on          0.99 to 1.24 from 1,000 weight rows on; below eight chunks 0.91 to 1.3, eight rows there 0.81 to 1.2
//           7 and 8 rows, 8 chunks (four pairs a    1.00 to 1.16; of 9 to 12 chunks 0.90 to 1.2
//             wave)
//   32-bit  1 and 2 rows                            1.00 to 1.27
//           3 and 4 rows, 4, 6 and 8 chunks         0.99 to 1.16; of 2 chunks (eight pairs a wave) 0.88 to 1.06, of 5 (four of three kilobytes) 0.93 to 1.06
//           5 and 6 rows, 8 chunks                  1.01 to 1.07
//           7 and 8 rows, 8 chunks                  with SwiGLU 0.99 to 1.07, else from a weight tile a compute unit on 1.00 to 1.02 (below 0.94 to 0.99)
// A launch is of as many waves as K has chunks, so that 32-bit products of 1, 3 and 7 chunks, which the streaming kernels take with waves to spare, have none.
static int normed_rows(int N, int chunks, int projections) {
#ifdef VK_BF16
  if (chunks < 1 || chunks > 12) return 0;
  return chunks < 8 || N <= 2 * vk_device_cus() ? 4 : chunks == 8 ? 8 : 6;
#else
  if (chunks == 2 || chunks == 5) return 2;
  if (chunks == 4 || chunks == 6) return 4;
  return chunks != 8 ? 0 : projections == 2 || (N + 15) / 16 >= vk_device_cus() ? 8 : 6;
#endif
}
// The launch.  16-bit: whole lines in tiles of eight weight rows, or of four where those do not fit the LDS (up to 512 weight rows four are as fast or, of gate and up,
// 4 to 10 % faster; otherwise up to 25 % slower), also where the streaming kernel is the faster one of a product by itself: one barrier a tile, and the norm's, cost it
// more than the lines'.  But three and four rows of two chunks and one projection are faster with it by the mean of 7 % (0.93 to 1.10 times as fast).
// Before and after, us, 1, 4 and (from eight chunks on) 8 rows, 16-bit: 4,096 x 1,024 5.8, 6.3 -> 4.0, 5.2; gate/up 3,072 x 1,024 7.8, 7.8 -> 5.2, 7.0; 4,096 x 1,536 7.0, 7.2 -> 4.5, 6.2;
// 6,144 x 3,072 10.8, 11.8 -> 8.2, 9.8; gate/up 10,240 x 2,560 21.3, 21.6 -> 18.8, 20.6; 6,144 x 4,096 12.7, 13.7, 14.5 -> 10.4, 11.3, 12.6; gate/up 10,240 x 4,096 31.8, 32.9,
// 33.3 -> 28.4, 30.7, 32.6; gate/up 10,240 x 6,144 44.2, 45.2 -> 40.9, 42.6; 32-bit, 1, 2 and 4 rows: 4,096 x 1,024 8.0, 8.1 -> 6.6, 7.7; 4,096 x 2,048 11.2, 11.2, 11.4 -> 9.7, 9.9, 10.8;
// 6,144 x 2,560 18.6, 19.0 -> 17.1, 18.3; 6,144 x 3,072 20.8, 20.9, 21.4 -> 19.1, 19.5, 20.4; gate/up 10,240 x 4,096 75.1, 75.3, 75.8 -> 68.9, 69.1, 70.2.
template <int ROWS, int P>
static int normed_product(elem_t* out, const elem_t* x, const elem_t* w, int M, int N, int K, int64_t ldx, int64_t ldo, const NormArgs& norm, hipStream_t st) {
  const int chunks = K / KC, form = ldo % 4 == 0 && (uintptr_t)out % 16 == 0;
#define STREAMED(NW) if (chunks == NW) return launch_stream_normed<ROWS, P, NW>(out, x, w, M, N, ldx, ldo, form, norm, st)
#ifdef VK_BF16
  if constexpr (ROWS == 4 && P == 1) {
    if (M > 2) STREAMED(2);
  }
#define LINED(NW) if (chunks == NW) return launch_lines_normed<P == 1 || NW <= 8 ? 8 : 4, ROWS, P, NW>(out, x, w, M, N, ldx, ldo, form, norm, st)
  if constexpr (ROWS <= 4) {
    LINED(1); LINED(2); LINED(3); LINED(4); LINED(5); LINED(6); LINED(7);
  }
  LINED(8); LINED(9); LINED(10); LINED(11); LINED(12);
#undef LINED
#else
  if constexpr (ROWS <= 4) {
    STREAMED(2); STREAMED(4); STREAMED(5); STREAMED(6);
  }
  STREAMED(8);
#endif
#undef STREAMED
  return vk_fail("gemm_normed: no launch for %d rows of K=%d", M, K);
}
}  // extern "C++"

// 1 if vk_gemm_normed takes these sizes (projections 1, or 2 with N gate rows) and is the faster way (normed_rows).
int vk_gemm_normed_takes(int M, int N, int K, int projections) {
  return M >= 1 && N >= 1 && K >= KC && K % KC == 0 && M <= normed_rows(N, K / KC, projections);
}

// out = norm(x + residual) w^T, or with two projections silu(gate) * up: vk_add_rmsnorm (sum, [M, K], takes the place of its new residual and is
// another buffer than either input) and vk_gemm or vk_gemm_swiglu in one launch, the same bits.  x, residual and sum [M, K], norm_weight [K] elements.
int vk_gemm_normed(elem_t* out, elem_t* sum, const elem_t* x, const elem_t* residual, const elem_t* norm_weight, float eps, const elem_t* w, int M, int N, int K,
                   int64_t ldo, int projections, hipStream_t st) {
  VK_REQUIRE(projections == 1 || projections == 2, "gemm_normed: one projection or two, not %d", projections);
  VK_REQUIRE(M >= 0, "gemm_normed: bad sizes M=%d N=%d K=%d", M, N, K);
  VK_REQUIRE(eps >= 0.f, "gemm_normed: eps must not be negative");
  if (M == 0) return 0;
  VK_REQUIRE(vk_gemm_normed_takes(M, N, K, projections), "gemm_normed: sizes M=%d N=%d K=%d are not supported", M, N, K);
  VK_REQUIRE(out != nullptr && ldo >= N, "gemm_normed: output row stride %lld is smaller than N=%d", (long long)ldo, N);
  VK_REQUIRE((((uintptr_t)x | (uintptr_t)residual | (uintptr_t)sum | (uintptr_t)norm_weight | (uintptr_t)w) % 16) == 0, "gemm_normed: operands must be 16-byte aligned");
  VK_REQUIRE(sum != x && sum != residual && x != nullptr && residual != nullptr && sum != nullptr && norm_weight != nullptr, "gemm_normed: the sum needs a buffer of its own");
  const NormArgs norm = {residual, sum, norm_weight, eps};
#define NORMED(ROWS) return projections == 2 ? normed_product<ROWS, 2>(out, x, w, M, N, K, K, ldo, norm, st) : normed_product<ROWS, 1>(out, x, w, M, N, K, K, ldo, norm, st)
  if (M == 1) NORMED(1);
  if (M <= 4) NORMED(4);
  NORMED(8);
#undef NORMED
}

// float32 elements of workspace that vk_gemm_split needs for these sizes, or 0 if it does not take them:
// up to 64 rows of 16-bit elements, K in whole chunks; rows: weight rows (with swiglu: gate and up rows
// together, an even number of 16-row tiles).
int64_t vk_gemm_split_floats(int M, int rows, int K, int swiglu) {
#ifdef VK_BF16
  if (M <= 0 || M > 64 || rows <= 0 || K <= 0 || K % KC != 0) return 0;
  if (swiglu && rows % 32 != 0) return 0;
  const int mt = (M + 15) / 16;
  return (int64_t)(K / KC) * ((rows + 15) / 16) * mt * 256;
#else
  (void)M; (void)rows; (void)K; (void)swiglu;
  return 0;
#endif
}

// 1 if the route through chunk sums is the faster one for these sizes (measured on an MI355X).  Not with the
// activation folded in (24576 x 4096 at 64 rows: 60 -> 62 us), not for matrices of less than 64 KB per compute
// unit (1000 x 1024 at 32 rows: 4.8 -> 6.5 us), and not where workgroups of 128 weight rows are a quarter of the
// compute units or more: the other kernels then have workgroups enough, and the chunk sums would be a large
// share of the traffic.
//   17 to 64 rows: always then (64 rows: 4096 x 12288 45 -> 32 us, 4096 x 4096 16.0 -> 13.8; 32 rows: 41 -> 27, 13.4 -> 11.7 us).  Where rows_width
//     takes such sizes, which is faster still, vk_gemm_split does so too and leaves the workspace alone.
//   Up to 16 rows the streaming kernel is the other choice.  With `fill` the share of the compute units that
//   its last round of one workgroup per 16 weight rows keeps busy:
//     K of more than 16 chunks (its waves read their activations again for every chunk): when fill < 0.9
//       (8 rows: 5120 x 17408 52.8 -> 40.3 us, 2560 x 9728 16.2 -> 14.9) or from 13 rows on
//       (4096 x 12288, fill 1: 1 row 19.4 -> 23.5 us, 8 rows 20.9 -> 23.7, 12 rows 22.6 -> 23.7, 16 rows 23.4 -> 23.7; 8192 x 12288: 8 rows 38.2 -> 42.7, 12 rows
//       42.6 -> 42.4, 16 rows 44.5 -> 42.4);
//     K of 9 to 16 chunks, where lines_rows does not take it: when fill < 0.7 (2048 x 8192, 8 rows 16.1 -> 11.4 us, 5120 x 5120, 16 rows 17.9 -> 16.7; but
//       7168 x 5120, fill 0.88, 16 rows 19.2 -> 21.0);
//     K of up to 8 chunks: never (4096 x 4096 9.1 -> 10.3 us, 2560 x 4096, fill 0.63, 8.3 -> 9.2).
int vk_gemm_split_preferred(int M, int rows, int K, int swiglu) {
  if (swiglu || vk_gemm_split_floats(M, rows, K, swiglu) == 0) return 0;
  const int cus = vk_device_cus();
  const int64_t bytes = (int64_t)rows * K * (int64_t)sizeof(elem_t);
  if (bytes < (int64_t)cus * 65536 || 4 * ((rows + 127) / 128) > cus) return 0;
  if (M > 16) return 1;
  if (lines_rows(M, rows, K, 1)) return 0;
  const int nchunks = K / KC, tiles16 = (rows + 15) / 16;
  const int rounds = (tiles16 + cus - 1) / cus;
  const bool fill_below_09 = 10 * tiles16 < 9 * rounds * cus, fill_below_07 = 10 * tiles16 < 7 * rounds * cus;
  if (nchunks > 2 * SK_WAVES) return fill_below_09 || M > 12;
  return nchunks > SK_WAVES && fill_below_07;
}

// out = act w^T (swiglu 0: w [rows, K], out [M, rows]) or silu(act w_gate^T) * (act w_up^T) (swiglu 1:
// w = [gate rows; up rows], out [M, rows / 2]), through chunk sums in a workspace: the bits of vk_gemm and
// vk_gemm_swiglu.  Calls that overlap in time need workspaces of their own.
static int gemm_split_launch(elem_t* out, const elem_t* act, const elem_t* w, int M, int rows, int K, int64_t lda, int64_t ldo,
                             int swiglu, int activation, float* workspace, int64_t workspace_floats, hipStream_t st) {
  const int64_t need = vk_gemm_split_floats(M, rows, K, swiglu);
  VK_REQUIRE(need > 0, "gemm_split: sizes M=%d rows=%d K=%d are not supported", M, rows, K);
  VK_REQUIRE(workspace != nullptr && workspace_floats >= need && ((uintptr_t)workspace % 16) == 0,
             "gemm_split: a 16-byte aligned workspace of %lld floats is needed", (long long)need);
  const int out_cols = swiglu ? rows / 2 : rows;
  VK_REQUIRE(lda >= K && lda % VK_VEC == 0 && ldo >= out_cols, "gemm_split: bad row strides");
  VK_REQUIRE(((uintptr_t)act % 16) == 0 && ((uintptr_t)w % 16) == 0, "gemm_split: operands must be 16-byte aligned");
#ifdef VK_BF16
  const int form = out_form_of(out, ldo, activation);
  const int mt = (M + 15) / 16;
  const int width = vk_gemm_split_preferred(M, rows, K, swiglu) ? rows_width(M, rows, K, lda, false) : 0;
  if (width) return gemm_rows(width, false, out, act, w, M, rows, K, lda, ldo, form, st);
  if (mt == 1) return launch_split<1>(out, act, w, M, rows, K, lda, ldo, swiglu, workspace, form, st);
  if (mt == 2) return launch_split<2>(out, act, w, M, rows, K, lda, ldo, swiglu, workspace, form, st);
  if (mt == 3) return launch_split<3>(out, act, w, M, rows, K, lda, ldo, swiglu, workspace, form, st);
  return launch_split<4>(out, act, w, M, rows, K, lda, ldo, swiglu, workspace, form, st);
#else
  (void)out; (void)st; (void)activation;
  return vk_fail("gemm_split: built for 16-bit elements only");
#endif
}

int vk_gemm_split(elem_t* out, const elem_t* act, const elem_t* w, int M, int rows, int K, int64_t lda, int64_t ldo,
                  int swiglu, float* workspace, int64_t workspace_floats, hipStream_t st) {
  return gemm_split_launch(out, act, w, M, rows, K, lda, ldo, swiglu, 0, workspace, workspace_floats, st);
}

// The plain product of vk_gemm_split with an activation on the outputs.
int vk_gemm_split_act(elem_t* out, const elem_t* act, const elem_t* w, int M, int rows, int K, int64_t lda, int64_t ldo, int activation,
                      float* workspace, int64_t workspace_floats, hipStream_t st) {
  VK_REQUIRE(activation == 0 || activation == 1, "gemm: unknown activation %d", activation);
  return gemm_split_launch(out, act, w, M, rows, K, lda, ldo, 0, activation, workspace, workspace_floats, st);
}

}  // extern "C"
