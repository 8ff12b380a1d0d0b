// What happens to the q, k and v rows between the QKV projection and attention,
// in one launch: per-head RMSNorm of q and k, rotary position encoding of q and
// k, and the write of k and v into their pages.  Each step is optional, so the
// same kernel also serves as a plain head norm, a plain rotation or a plain
// cache store.
//
// Formulas (reference):
//   head norm  kernels/triton_kernels/qk_norm.py:67-95   y = x*rsqrt(mean(x^2)+eps)*w, rounded
//   rotation   kernels/triton_kernels/rope.py:78-123     y1 = x1*cos - x2*sin; y2 = x2*cos + x1*sin,
//              halves split at rot/2, on the rounded norm output, tables indexed by position
//   store      kernels/triton_kernels/store_kv_cache.py:89-120   slot -1 writes nothing
// The reference runs them as five launches (src/exec/dense_swiglu_decoder.rs:207-272).
//
// One wave per (token, head) at a time; lane l owns elements l, l+64, l+128, l+192.
#include "common.h"
#include "vec.h"

struct QkvPostArgs {
  const elem_t* qkv;      // [T, row_stride]: nq q heads, then nkv k heads, then nkv v heads, d each
  int64_t row_stride;
  elem_t* q_out;          // [T, nq, d]
  elem_t* kc;             // [pages, nkv, P, d]
  elem_t* vc;             // [pages, nkv, d, P]
  const void* q_w;        // [d] or null
  const void* k_w;        // [d] or null
  const elem_t* bias;     // [(nq + 2 nkv) d] or null: added to the row first (the sum rounded to the element type)
  const elem_t* cos_t;    // [max_pos, rot_half] or null
  const elem_t* sin_t;
  const float* inv_freq;  // [rot_half] or null: instead of tables, the angle of pair c is position * inv_freq[c], in 32-bit,
  float mag;              // and its cosine and sine are multiplied by this
  const int32_t* positions;  // [T]
  const int32_t* slots;      // [T]: page * P + offset, or -1
  int w_is_f32, nq, nkv, d, P, rot_half;
  int norm_d;             // the head norm's own size: the mean of squares divides by it, and its weight has this many entries
  int neighbours;         // 1: pair c of a head is its elements 2c and 2c + 1 instead of c and c + rot_half
  float eps;
};

// Cosine and sine of pair c at a token: from the tables' row, or computed in 32-bit from the position and the pair's
// frequency (the product rounded once, then the library's cosine and sine, each times the magnitude).
__device__ __forceinline__ void pair_angle(const QkvPostArgs& a, int64_t trow, float posf, int c, float& cs, float& sn) {
  if (a.inv_freq != nullptr) {
    const float angle = posf * a.inv_freq[c];
    cs = cosf(angle) * a.mag;
    sn = sinf(angle) * a.mag;
  } else {
    cs = to_f32(a.cos_t[trow + c]);
    sn = to_f32(a.sin_t[trow + c]);
  }
}

// A workgroup has four waves and one token; wave w takes the heads first + w, first + w + 4, ... of the
// workgroup's `per_wave` * 4 heads, so that a long step does not start a workgroup per head.  What bounded it with
// computed angles were the cosines and sines: a token's are computed once, into LDS, not once for every head that turns by
// them, and a wave waits for its own lanes only when a head's row goes through LDS.  Measured on MI355X, heads of 128:
// 2,048 tokens of 48 heads 65 -> 47 us, 1,334 of 24 heads 33 -> 18, a step of eight tokens of 24 heads 6.8 -> 5.2.
__global__ __launch_bounds__(256) void qkv_post_kernel(QkvPostArgs a, int per_wave) {
  __shared__ float ybuf[4][256];
  __shared__ float cs[128], sn[128];       // a rotation has at most 128 pairs
  const int tok = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  float* y = ybuf[wave];
  const int d = a.d, heads = a.nq + 2 * a.nkv;
  const int rh = a.rot_half;
  // With a rotation half of 64 or 128 elements the partner of an element is held by the same lane.
  const bool in_lane = rh % 64 == 0 && !a.neighbours;
  const int shift = rh / 64;
  const bool has_rot = a.cos_t != nullptr || a.inv_freq != nullptr;
  const int slot = a.slots != nullptr ? a.slots[tok] : -1;
  if (has_rot) {
    const int pos = a.positions[tok];
    for (int c = threadIdx.x; c < rh; c += 256) pair_angle(a, (int64_t)pos * rh, (float)pos, c, cs[c], sn[c]);
    __syncthreads();
  }
  for (int j = 0; j < per_wave; ++j) {
    const int hh = (blockIdx.y * per_wave + j) * 4 + wave;
    const bool live = hh < heads;
    const int kind = hh < a.nq ? 0 : (hh < a.nq + a.nkv ? 1 : 2);   // q, k, v
    const elem_t* x = a.qkv + tok * a.row_stride + (int64_t)(live ? hh : 0) * d;
    const void* w = kind == 0 ? a.q_w : (kind == 1 ? a.k_w : nullptr);

    float xv[4];
    float part = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int c = lane + 64 * i;
      xv[i] = c < d ? to_f32(x[c]) : 0.f;
      if (a.bias != nullptr && live && c < d) xv[i] = round_to_elem(xv[i] + to_f32(a.bias[(int64_t)hh * d + c]));
      part = part + xv[i] * xv[i];
    }
    if (w != nullptr) {
      const float total = wave_sum_xor(part);
      const float rr = rsqrtf(total / (float)a.norm_d + a.eps);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = lane + 64 * i;
        if (c < d) xv[i] = c < a.norm_d ? round_to_elem((xv[i] * rr) * load_weight(w, a.w_is_f32, c)) : 0.f;
      }
    }
    const bool rotate = has_rot && kind != 2;
    if (has_rot && !in_lane) {
      if (rotate) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = lane + 64 * i;
          if (c < d) y[c] = xv[i];
        }
      }
      // The lanes of a wave read what the same wave wrote.
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
    }
    if (rotate) {
      float old[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) old[i] = xv[i];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = lane + 64 * i;
        if (a.neighbours) {
          // Element 2c is the pair's first, 2c + 1 its second; both lie in y.
          if (c < 2 * rh) {
            const float co = cs[c >> 1], si = sn[c >> 1], other = y[c ^ 1];
            xv[i] = (c & 1) ? old[i] * co + other * si : old[i] * co - other * si;
          }
        } else if (c < rh) {
          const float other = in_lane ? (i + shift < 4 ? old[(i + shift) & 3] : 0.f) : y[c + rh];
          xv[i] = old[i] * cs[c] - other * sn[c];
        } else if (c < 2 * rh) {
          const float other = in_lane ? (i >= shift ? old[(i - shift) & 3] : 0.f) : y[c - rh];
          xv[i] = old[i] * cs[c - rh] + other * sn[c - rh];
        }
      }
    }
    if (has_rot && !in_lane) {
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();       // y is free for the next head
    }
    if (!live) continue;
    if (kind == 0) {
      elem_t* o = a.q_out + ((int64_t)tok * a.nq + hh) * d;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = lane + 64 * i;
        if (c < d) o[c] = from_f32<elem_t>(xv[i]);
      }
      continue;
    }
    if (slot < 0) continue;
    const int page = slot / a.P, off = slot - page * a.P;
    if (kind == 1) {
      const int kh = hh - a.nq;
      elem_t* o = a.kc + (((int64_t)page * a.nkv + kh) * a.P + off) * d;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = lane + 64 * i;
        if (c < d) o[c] = from_f32<elem_t>(xv[i]);
      }
    } else {
      const int kh = hh - a.nq - a.nkv;
      elem_t* o = a.vc + ((int64_t)page * a.nkv + kh) * d * a.P + off;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = lane + 64 * i;
        if (c < d) o[(int64_t)c * a.P] = from_f32<elem_t>(xv[i]);
      }
    }
  }
}

// The same for head sizes 64, 128 and 256 with a full rotation (or none): a lane owns VK_VEC
// consecutive elements, so that rows are read and written 16 bytes per lane; the d / VK_VEC lanes of a
// head sit side by side, a wave holds 64 / (d / VK_VEC) heads of one token.  The sum of squares runs
// over a lane's elements in order, then as a butterfly over the head's lanes.
template <int LPH>     // lanes per head
__global__ __launch_bounds__(256) void qkv_post_vec_kernel(QkvPostArgs a, int per_wave) {
  constexpr int HPW = 64 / LPH;
  const int tok = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int d = a.d, heads = a.nq + 2 * a.nkv;
  const int j = lane % LPH, hsub = lane / LPH;
  int64_t trow = 0;
  if (a.cos_t != nullptr) trow = (int64_t)a.positions[tok] * a.rot_half;
  const int slot = a.slots != nullptr ? a.slots[tok] : -1;
  const int page = slot >= 0 ? slot / a.P : 0, off = slot >= 0 ? slot - page * a.P : 0;
  for (int it = 0; it < per_wave; ++it) {
    const int hh = ((blockIdx.y * per_wave + it) * 4 + wave) * HPW + hsub;
    const bool live = hh < heads;
    const int kind = hh < a.nq ? 0 : (hh < a.nq + a.nkv ? 1 : 2);   // q, k, v
    const elem_t* x = a.qkv + tok * a.row_stride + (int64_t)(live ? hh : 0) * d + j * VK_VEC;
    const void* w = kind == 0 ? a.q_w : (kind == 1 ? a.k_w : nullptr);
    float xv[VK_VEC];
    load_elems(x, xv);
    if (a.bias != nullptr && live) {
      float bv[VK_VEC];
      load_elems(a.bias + (int64_t)hh * d + j * VK_VEC, bv);
#pragma unroll
      for (int e = 0; e < VK_VEC; ++e) xv[e] = round_to_elem(xv[e] + bv[e]);
    }
    if (w != nullptr) {
      float part = 0.f;
#pragma unroll
      for (int e = 0; e < VK_VEC; ++e) part = part + xv[e] * xv[e];
      part = group_sum<LPH>(part);
      const float rr = rsqrtf(part / (float)d + a.eps);
      float wv[VK_VEC];
      if (a.w_is_f32) {
#pragma unroll
        for (int e = 0; e < VK_VEC; ++e) wv[e] = static_cast<const float*>(w)[j * VK_VEC + e];
      } else {
        load_elems(static_cast<const elem_t*>(w) + j * VK_VEC, wv);
      }
#pragma unroll
      for (int e = 0; e < VK_VEC; ++e) xv[e] = round_to_elem((xv[e] * rr) * wv[e]);
    }
    if (a.cos_t != nullptr) {
      // The partner of element c is c +- d/2: the same place in the lane LPH/2 away.  Every lane takes
      // part in the exchange, also those of v heads, which keep their values.
      float other[VK_VEC], cs[VK_VEC], sn[VK_VEC];
#pragma unroll
      for (int e = 0; e < VK_VEC; ++e) other[e] = __shfl_xor(xv[e], LPH / 2, VK_WAVE);
      const int tcol = (j % (LPH / 2)) * VK_VEC;
      load_elems(a.cos_t + trow + tcol, cs);
      load_elems(a.sin_t + trow + tcol, sn);
      if (kind != 2) {
        if (j < LPH / 2) {
#pragma unroll
          for (int e = 0; e < VK_VEC; ++e) xv[e] = xv[e] * cs[e] - other[e] * sn[e];
        } else {
#pragma unroll
          for (int e = 0; e < VK_VEC; ++e) xv[e] = xv[e] * cs[e] + other[e] * sn[e];
        }
      }
    }
    if (!live) continue;
    if (kind == 0) {
      store_elems(a.q_out + ((int64_t)tok * a.nq + hh) * d + j * VK_VEC, xv);
    } else if (slot >= 0) {
      if (kind == 1) {
        store_elems(a.kc + (((int64_t)page * a.nkv + (hh - a.nq)) * a.P + off) * d + j * VK_VEC, xv);
      } else {
        elem_t* o = a.vc + (((int64_t)page * a.nkv + (hh - a.nq - a.nkv)) * d + j * VK_VEC) * a.P + off;
#pragma unroll
        for (int e = 0; e < VK_VEC; ++e) o[(int64_t)e * a.P] = from_f32<elem_t>(xv[e]);
      }
    }
  }
}

extern "C" {

// Null q_w / k_w: no norm for that kind.  Null cos_t: no rotation.  nkv == 0:
// only q rows (a plain norm and/or rotation of [T, nq, d]).  nq == 0: only the
// store.  Positions must lie below the tables' row count and slots inside the
// cache; the caller checks both on the host before the upload.
static int qkv_post_launch(const elem_t* qkv, int64_t row_stride, elem_t* q_out, elem_t* kc, elem_t* vc, const void* q_w,
                           const void* k_w, int w_is_f32, const elem_t* cos_t, const elem_t* sin_t, int rot_half,
                           const int32_t* positions, const int32_t* slots, int T, int nq, int nkv, int d, int P, float eps,
                           const elem_t* bias, hipStream_t st, const float* inv_freq = nullptr, float mag = 1.f, int norm_d = 0,
                           int neighbours = 0) {
  VK_REQUIRE(T >= 0 && nq >= 0 && nkv >= 0 && nq + nkv > 0, "qkv_post: bad sizes T=%d nq=%d nkv=%d", T, nq, nkv);
  VK_REQUIRE(d > 0 && d <= 256, "qkv_post: head size %d must be in 1..256", d);
  VK_REQUIRE(row_stride >= (int64_t)(nq + 2 * nkv) * d, "qkv_post: row stride %lld too small", (long long)row_stride);
  VK_REQUIRE((cos_t == nullptr && inv_freq == nullptr) || (rot_half > 0 && 2 * rot_half <= d), "qkv_post: rotary width %d does not fit head size %d",
             2 * rot_half, d);
  VK_REQUIRE((cos_t == nullptr && inv_freq == nullptr) || positions != nullptr, "qkv_post: rotation needs positions");
  VK_REQUIRE(cos_t == nullptr || inv_freq == nullptr, "qkv_post: tables of angles or frequencies, not both");
  VK_REQUIRE(nkv == 0 || (slots != nullptr && kc != nullptr && vc != nullptr && P > 0), "qkv_post: store needs slots and caches");
  VK_REQUIRE(nq + 2 * nkv <= 65535, "qkv_post: too many heads");
  VK_REQUIRE(norm_d >= 0 && norm_d <= d, "qkv_post: a head norm over %d of %d elements", norm_d, d);
  if (norm_d == 0) norm_d = d;
  if (T == 0) return 0;
  QkvPostArgs a;
  a.qkv = qkv; a.row_stride = row_stride; a.q_out = q_out; a.kc = kc; a.vc = vc; a.q_w = q_w; a.k_w = k_w;
  a.cos_t = cos_t; a.sin_t = sin_t; a.positions = positions; a.slots = slots; a.w_is_f32 = w_is_f32; a.bias = bias;
  a.nq = nq; a.nkv = nkv; a.d = d; a.P = P; a.rot_half = rot_half; a.eps = eps; a.inv_freq = inv_freq; a.mag = mag;
  a.norm_d = norm_d;
  a.neighbours = neighbours;
  VK_REQUIRE(!neighbours || inv_freq != nullptr, "qkv_post: neighbouring pairs are built for computed angles");
  // Few tokens: four waves' worth of heads per workgroup, for many workgroups; many tokens: all heads of a token.
  const int heads = nq + 2 * nkv;
  const int lph = d / VK_VEC;          // lanes per head in the kernel with 16-byte accesses
  const bool vec = inv_freq == nullptr && norm_d == d && (d == 64 || d == 128 || d == 256) && lph <= 64 && (cos_t == nullptr || 2 * rot_half == d) &&
                   row_stride % VK_VEC == 0 && ((uintptr_t)qkv % 16) == 0 && (q_out == nullptr || (uintptr_t)q_out % 16 == 0) &&
                   (kc == nullptr || (uintptr_t)kc % 16 == 0) && (bias == nullptr || (uintptr_t)bias % 16 == 0) && (cos_t == nullptr || ((uintptr_t)cos_t % 16 == 0 && (uintptr_t)sin_t % 16 == 0));
  if (vec) {
    const int hpw = 64 / lph, per_wg = 4 * hpw;
    const int per_wave = T >= 512 ? (heads + per_wg - 1) / per_wg : 1;
    const dim3 grid(T, (heads + per_wg * per_wave - 1) / (per_wg * per_wave));
    if (lph == 8) qkv_post_vec_kernel<8><<<grid, 256, 0, st>>>(a, per_wave);
    else if (lph == 16) qkv_post_vec_kernel<16><<<grid, 256, 0, st>>>(a, per_wave);
    else if (lph == 32) qkv_post_vec_kernel<32><<<grid, 256, 0, st>>>(a, per_wave);
    else qkv_post_vec_kernel<64><<<grid, 256, 0, st>>>(a, per_wave);
    return vk_check_launch("qkv_post");
  }
  const int per_wave = T >= 512 ? (heads + 3) / 4 : 1;
  qkv_post_kernel<<<dim3(T, (heads + 4 * per_wave - 1) / (4 * per_wave)), 256, 0, st>>>(a, per_wave);
  return vk_check_launch("qkv_post");
}

int vk_qkv_post(const elem_t* qkv, int64_t row_stride, elem_t* q_out, elem_t* kc, elem_t* vc, const void* q_w,
                const void* k_w, int w_is_f32, const elem_t* cos_t, const elem_t* sin_t, int rot_half,
                const int32_t* positions, const int32_t* slots, int T, int nq, int nkv, int d, int P, float eps,
                hipStream_t st) {
  return qkv_post_launch(qkv, row_stride, q_out, kc, vc, q_w, k_w, w_is_f32, cos_t, sin_t, rot_half, positions, slots, T, nq, nkv, d, P, eps,
                         nullptr, st);
}

// The same with a bias [(nq + 2 nkv) d] that is added to every row before anything else, as a projection with a bias
// would have left it.
int vk_qkv_post_bias(const elem_t* qkv, int64_t row_stride, elem_t* q_out, elem_t* kc, elem_t* vc, const void* q_w,
                     const void* k_w, int w_is_f32, const elem_t* cos_t, const elem_t* sin_t, int rot_half,
                     const int32_t* positions, const int32_t* slots, int T, int nq, int nkv, int d, int P, float eps,
                     const elem_t* bias, hipStream_t st) {
  return qkv_post_launch(qkv, row_stride, q_out, kc, vc, q_w, k_w, w_is_f32, cos_t, sin_t, rot_half, positions, slots, T, nq, nkv, d, P, eps,
                         bias, st);
}

// The same with the angles computed instead of tabulated: pair c (elements c and c + rot_half of every q and k head)
// turns by position * inv_freq[c], the product, the cosine and the sine in 32-bit, both times `mag`.
int vk_qkv_post_angles(const elem_t* qkv, int64_t row_stride, elem_t* q_out, elem_t* kc, elem_t* vc, const float* inv_freq, float mag,
                       int rot_half, const int32_t* positions, const int32_t* slots, int T, int nq, int nkv, int d, int P, hipStream_t st) {
  VK_REQUIRE(inv_freq != nullptr, "qkv_post: the rotation's frequencies are missing");
  return qkv_post_launch(qkv, row_stride, q_out, kc, vc, nullptr, nullptr, 0, nullptr, nullptr, rot_half, positions, slots, T, nq, nkv, d, P, 0.f,
                         nullptr, st, inv_freq, mag);
}

// Head norms and computed angles together: q and k heads are normed over their first norm_d elements (weights q_w, k_w of
// that many entries, either may be null; the elements beyond, padding, come out zero), then turned as vk_qkv_post_angles
// turns them.  Rows may be longer than the heads they hold (row_stride).
int vk_qkv_post_norm_angles(const elem_t* qkv, int64_t row_stride, elem_t* q_out, elem_t* kc, elem_t* vc, const void* q_w, const void* k_w,
                            int w_is_f32, int norm_d, float eps, const float* inv_freq, float mag, int rot_half, const int32_t* positions,
                            const int32_t* slots, int T, int nq, int nkv, int d, int P, hipStream_t st) {
  VK_REQUIRE(inv_freq != nullptr, "qkv_post: the rotation's frequencies are missing");
  VK_REQUIRE(norm_d > 0 && 2 * rot_half <= norm_d, "qkv_post: a rotation of %d elements in a head norm of %d", 2 * rot_half, norm_d);
  return qkv_post_launch(qkv, row_stride, q_out, kc, vc, q_w, k_w, w_is_f32, nullptr, nullptr, rot_half, positions, slots, T, nq, nkv, d, P, eps,
                         nullptr, st, inv_freq, mag, norm_d);
}

// The same with a choice of which elements form a pair: neighbours 1 turns the elements 2c and 2c + 1 of a head by
// position * inv_freq[c] (c < rot_half), 0 is vk_qkv_post_norm_angles.  q_w and k_w may both be null (no head norms; norm_d
// is then not used).
int vk_qkv_post_norm_angles_paired(const elem_t* qkv, int64_t row_stride, elem_t* q_out, elem_t* kc, elem_t* vc, const void* q_w, const void* k_w,
                                   int w_is_f32, int norm_d, float eps, const float* inv_freq, float mag, int rot_half, int neighbours,
                                   const int32_t* positions, const int32_t* slots, int T, int nq, int nkv, int d, int P, hipStream_t st) {
  VK_REQUIRE(inv_freq != nullptr, "qkv_post: the rotation's frequencies are missing");
  VK_REQUIRE(neighbours == 0 || neighbours == 1, "qkv_post: 'neighbours' is 0 or 1");
  const bool normed = q_w != nullptr || k_w != nullptr;
  VK_REQUIRE(!normed || (norm_d > 0 && 2 * rot_half <= norm_d), "qkv_post: a rotation of %d elements in a head norm of %d", 2 * rot_half, norm_d);
  return qkv_post_launch(qkv, row_stride, q_out, kc, vc, q_w, k_w, w_is_f32, nullptr, nullptr, rot_half, positions, slots, T, nq, nkv, d, P, eps,
                         nullptr, st, inv_freq, mag, normed ? norm_d : 0, neighbours);
}

}  // extern "C"
