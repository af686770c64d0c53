// Element-wise passes of the training batch, fused (gfx950): RMSNorm, SwiGLU,
// QK-norm + RoPE and the scaled causal mask, in both directions.
//
// Reference semantics: the batch forward of RMSNorm, Qwen3MLP and
// Qwen3Attention (qwen3_naive.py:156-169, :553-590, :695-702) and its
// gradients, as torch's formulas compute them.  These kernels repeat the
// formulas: the same fp32 operations in the same grouping, the same roundings
// to bf16 in between, no contraction to FMA but the ones named (the file is
// built with -ffp-contract=off).  The norms' sums along a row (mean of squares,
// the row's gradient) and the products stay with torch; the softmax of rows of
// up to 1,024 adds in torch's order.  So values are torch's bits, except where
// a sum has another, fixed order: the norm weights' gradients, and k's and v's
// gradients summed over four or more query heads per KV head.
//
// What bounds them is memory: a norm forward moved its fp32 rows through
// memory 9 times in 9 launches and backward ~20 times, the scores took 3
// passes per direction outside the softmax.  All are one 8-element item per
// lane with 16- or 32-byte accesses.  One decoder layer forward + backward, 8 x
// 640 tokens of hidden 1024: 4,000 -> 1,985-2,100 us (850 of them fp32
// products); a two-layer training step, 2 x 389 tokens: 5,400-5,600 -> 2,890-
// 2,940 us.
#include <algorithm>

#include "qmi_common.h"

namespace {

using namespace qmi;

constexpr int kThreads = 256;
constexpr int kD = 128;   // head dim
constexpr int kTile = 64;  // tokens of a transposing tile

struct V8 {
  float v[8];
};

__device__ __forceinline__ V8 unpack8(uint4 a) {
  const uint32_t w[4] = {a.x, a.y, a.z, a.w};
  V8 r;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    r.v[2 * e] = bf16_lo(w[e]);
    r.v[2 * e + 1] = bf16_hi(w[e]);
  }
  return r;
}

__device__ __forceinline__ V8 load8(const uint16_t* p) { return unpack8(load_u4(p)); }

__device__ __forceinline__ uint4 pack8(const V8& a) {
  return make_uint4(pack_bf16x2(a.v[0], a.v[1]), pack_bf16x2(a.v[2], a.v[3]),
                    pack_bf16x2(a.v[4], a.v[5]), pack_bf16x2(a.v[6], a.v[7]));
}

__device__ __forceinline__ V8 load8f(const float* p) {
  const f32x4_t a = *reinterpret_cast<const f32x4_t*>(p);
  const f32x4_t b = *reinterpret_cast<const f32x4_t*>(p + 4);
  return V8{{a[0], a[1], a[2], a[3], b[0], b[1], b[2], b[3]}};
}

__device__ __forceinline__ void store8f(float* p, const V8& a) {
  *reinterpret_cast<f32x4_t*>(p) = f32x4_t{a.v[0], a.v[1], a.v[2], a.v[3]};
  *reinterpret_cast<f32x4_t*>(p + 4) = f32x4_t{a.v[4], a.v[5], a.v[6], a.v[7]};
}

// Correctly rounded, as torch.rsqrt's values are (the fp32 instruction's are
// off by one ulp for 11% of arguments).
__device__ __forceinline__ float inv_rms(float mean, float eps) {
  return (float)rsqrt((double)(mean + eps));
}

__device__ __forceinline__ V8 rounded(const V8& a) { return unpack8(pack8(a)); }

// Rows of n elements, `heads` of them adjacent in each bf16 row of `stride`;
// fp32 rows are contiguous.
struct Rows {
  int64_t rows, stride;
  int heads, n;
  __device__ __forceinline__ int64_t at(int64_t row, int col) const {
    if (heads == 1) return row * stride + col;
    const uint32_t r = (uint32_t)row;
    return (int64_t)(r / (uint32_t)heads) * stride + (r % (uint32_t)heads) * n + col;
  }
};

__global__ __launch_bounds__(kThreads) void square_kernel(const uint16_t* __restrict__ x, Rows d,
                                                          float* __restrict__ sq,
                                                          uint16_t* __restrict__ x_copy,
                                                          float* __restrict__ zero) {
  const int n8 = d.n / 8;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (zero && i == 0) *zero = 0.f;
  if (i >= d.rows * n8) return;
  const uint32_t row = (uint32_t)i / (uint32_t)n8;
  const int col = (int)((uint32_t)i % (uint32_t)n8) * 8;
  const uint4 raw = load_u4(x + d.at(row, col));
  if (x_copy) *reinterpret_cast<uint4*>(x_copy + 8 * i) = raw;
  V8 a = unpack8(raw);
#pragma unroll
  for (int e = 0; e < 8; ++e) a.v[e] = a.v[e] * a.v[e];
  store8f(sq + 8 * i, a);
}

__global__ __launch_bounds__(kThreads) void norm_apply_kernel(
    const uint16_t* __restrict__ x, Rows d, const float* __restrict__ mean,
    const uint16_t* __restrict__ w, float eps, uint16_t* __restrict__ y,
    uint16_t* __restrict__ w_copy) {
  const int n8 = d.n / 8;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= d.rows * n8) return;
  const uint32_t row = (uint32_t)i / (uint32_t)n8;
  const int col = (int)((uint32_t)i % (uint32_t)n8) * 8;
  const float r = inv_rms(mean[row], eps);
  V8 a = load8(x + d.at(row, col));
  const uint4 wr = load_u4(w + col);
  if (w_copy && row == 0) *reinterpret_cast<uint4*>(w_copy + col) = wr;
  const V8 ww = unpack8(wr);
#pragma unroll
  for (int e = 0; e < 8; ++e) a.v[e] = a.v[e] * r * ww.v[e];
  *reinterpret_cast<uint4*>(y + 8 * i) = pack8(a);
}

// prod = (dy * w) * x, whose row sums are the gradient of the row's rsqrt.
__global__ __launch_bounds__(kThreads) void norm_prod_kernel(
    const uint16_t* __restrict__ x, Rows d, const uint16_t* __restrict__ w,
    const uint16_t* __restrict__ dy, float* __restrict__ prod) {
  const int n8 = d.n / 8;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= d.rows * n8) return;
  const uint32_t row = (uint32_t)i / (uint32_t)n8;
  const int col = (int)((uint32_t)i % (uint32_t)n8) * 8;
  const V8 a = load8(x + d.at(row, col)), ww = load8(w + col);
  V8 g = load8(dy + 8 * i);
#pragma unroll
  for (int e = 0; e < 8; ++e) g.v[e] = g.v[e] * ww.v[e] * a.v[e];
  store8f(prod + 8 * i, g);
}

// dx of every row, and one partial dw row per workgroup: its rows of stride
// gridDim.x * groups, summed in row order per lane group, then over the groups.
__global__ __launch_bounds__(kThreads) void norm_grad_kernel(
    const uint16_t* __restrict__ x, Rows d, const float* __restrict__ mean,
    const uint16_t* __restrict__ w, float eps, const uint16_t* __restrict__ dy,
    const float* __restrict__ dr, uint16_t* __restrict__ dx, float* __restrict__ dw) {
  __shared__ float part[kThreads * 8];
  const int n8 = d.n / 8, groups = n8 >= kThreads ? 1 : kThreads / n8;
  for (int c0 = 0; c0 < n8; c0 += kThreads) {  // more than 2,048 columns: several passes
    const int grp = threadIdx.x / n8, c = c0 + (groups == 1 ? threadIdx.x : threadIdx.x % n8);
    V8 sum = {};
    if (grp < groups && c < n8) {
      const int col = 8 * c;
      const V8 ww = load8(w + col);
      for (int64_t row = (int64_t)blockIdx.x * groups + grp; row < d.rows;
           row += (int64_t)gridDim.x * groups) {
        const int64_t at = d.at(row, col);
        const float r = inv_rms(mean[row], eps);
        const float dsq = -0.5f * dr[row] * (r * r * r) / (float)d.n;
        const V8 a = load8(x + at), g = load8(dy + row * d.n + col);
        V8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          o.v[e] = g.v[e] * ww.v[e] * r + dsq * (2.0f * a.v[e]);
          sum.v[e] += g.v[e] * (a.v[e] * r);
        }
        *reinterpret_cast<uint4*>(dx + at) = pack8(o);
      }
    }
    if (groups == 1) {
      if (c < n8) store8f(dw + (int64_t)blockIdx.x * d.n + 8 * c, sum);
      continue;
    }
    store8f(part + 8 * threadIdx.x, sum);
    __syncthreads();
    if (threadIdx.x < n8) {
      V8 s = load8f(part + 8 * threadIdx.x);
      for (int q = 1; q < groups; ++q) {
        const V8 b = load8f(part + 8 * (q * n8 + threadIdx.x));
#pragma unroll
        for (int e = 0; e < 8; ++e) s.v[e] += b.v[e];
      }
      store8f(dw + (int64_t)blockIdx.x * d.n + 8 * threadIdx.x, s);
    }
  }
}

__global__ __launch_bounds__(kThreads) void silu_mul_exact_kernel(const uint16_t* __restrict__ gu,
                                                                  int64_t rows, int inter,
                                                                  uint16_t* __restrict__ y) {
  const int n8 = inter / 8;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= rows * n8) return;
  const int64_t row = i / n8;
  const int col = (int)(i % n8) * 8;
  V8 g = load8(gu + row * 2 * inter + col);
  const V8 u = load8(gu + row * 2 * inter + inter + col);
#pragma unroll
  for (int e = 0; e < 8; ++e) g.v[e] = g.v[e] / (1.0f + expf(-g.v[e]));
  g = rounded(g);
#pragma unroll
  for (int e = 0; e < 8; ++e) g.v[e] = g.v[e] * u.v[e];
  *reinterpret_cast<uint4*>(y + 8 * i) = pack8(g);
}

__global__ __launch_bounds__(kThreads) void silu_mul_grad_kernel(const uint16_t* __restrict__ gu,
                                                                 int64_t rows, int inter,
                                                                 const uint16_t* __restrict__ dy,
                                                                 uint16_t* __restrict__ dgu) {
  const int n8 = inter / 8;
  const int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x;
  if (i >= rows * n8) return;
  const int64_t row = i / n8, at = row * 2 * inter + (i % n8) * 8;
  const V8 g = load8(gu + at), u = load8(gu + at + inter), d = load8(dy + 8 * i);
  V8 silu, dsilu, dg, du;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    silu.v[e] = g.v[e] / (1.0f + expf(-g.v[e]));
    dsilu.v[e] = d.v[e] * u.v[e];
  }
  silu = rounded(silu);
  dsilu = rounded(dsilu);
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float s = 1.0f / (1.0f + expf(-g.v[e]));
    // The one contraction: torch's kernel for this expression has it too.
    dg.v[e] = dsilu.v[e] * s * fmaf(g.v[e], 1.0f - s, 1.0f);
    du.v[e] = d.v[e] * silu.v[e];
  }
  *reinterpret_cast<uint4*>(dgu + at) = pack8(dg);
  *reinterpret_cast<uint4*>(dgu + at + inter) = pack8(du);
}

// 16 lanes hold a head, 8 dims each; the RoPE partner of dim d is d ^ 64,
// lane ^ 8.  o = rope(bf16(x r w)) rounded to bf16.
__device__ __forceinline__ V8 norm_rope(const V8& x, const V8& w, float r, const float* cs,
                                        int lane16) {
  V8 n;
#pragma unroll
  for (int e = 0; e < 8; ++e) n.v[e] = x.v[e] * r * w.v[e];
  n = rounded(n);
  const V8 c = load8f(cs + 8 * (lane16 & 7)), s = load8f(cs + 64 + 8 * (lane16 & 7));
  V8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float p = shfl_xor_f32(n.v[e], 8);
    const float a = n.v[e] * c.v[e], b = p * s.v[e];
    o.v[e] = lane16 < 8 ? a - b : a + b;
  }
  return rounded(o);
}

// Gradient of the rotation, rounded to bf16 as the cast before it is.
__device__ __forceinline__ V8 rope_grad(const V8& g, const float* cs, int lane16) {
  const V8 c = load8f(cs + 8 * (lane16 & 7)), s = load8f(cs + 64 + 8 * (lane16 & 7));
  V8 o;
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float p = shfl_xor_f32(g.v[e], 8);
    const float a = g.v[e] * c.v[e], b = p * s.v[e];
    o.v[e] = lane16 < 8 ? a + b : a - b;
  }
  return rounded(o);
}

struct Heads {
  const uint16_t* qkv;
  int64_t stride;
  int batch, t, hq, hkv;
};

// q (blocks of 16 heads of a token list): qf[b][h][t][128]; v: vf[b][h][t][128]
// with each KV head repeated for its query heads.
__global__ __launch_bounds__(kThreads) void qv_forward_kernel(
    Heads p, const float* __restrict__ q_mean, const uint16_t* __restrict__ q_w, float eps,
    const float* __restrict__ cache, float* __restrict__ qf, float* __restrict__ vf,
    uint16_t* __restrict__ w_copy) {
  const int lane16 = threadIdx.x & 15;
  const int per = p.hq + p.hkv;
  const uint32_t items = (uint32_t)p.batch * p.t * per;
  const uint32_t item = min(blockIdx.x * 16u + threadIdx.x / 16, items - 1);  // whole waves shuffle
  const uint32_t tok = item / per;
  const int h = item % per, b = tok / p.t, t = tok % p.t;
  const uint16_t* row = p.qkv + (int64_t)tok * p.stride + 8 * lane16;
  if (h < p.hq) {
    const float r = inv_rms(q_mean[(int64_t)tok * p.hq + h], eps);
    const uint4 wr = load_u4(q_w + 8 * lane16);
    if (w_copy && item == 0) *reinterpret_cast<uint4*>(w_copy + 8 * lane16) = wr;
    const V8 o = norm_rope(load8(row + h * kD), unpack8(wr), r, cache + t * kD, lane16);
    store8f(qf + (((int64_t)b * p.hq + h) * p.t + t) * kD + 8 * lane16, o);
  } else {
    const int hk = h - p.hq, rep = p.hq / p.hkv;
    const V8 o = load8(row + (p.hq + p.hkv + hk) * kD);
    for (int g = 0; g < rep; ++g)
      store8f(vf + (((int64_t)b * p.hq + hk * rep + g) * p.t + t) * kD + 8 * lane16, o);
  }
}

// k: kt[b][h][128][t], repeated for the query heads.  Block: (64 tokens, KV head, sequence);
// those of the first sequence and head copy the tokens' cos/sin rows, the first one the weights.
__global__ __launch_bounds__(kThreads) void k_forward_kernel(
    Heads p, const float* __restrict__ k_mean, const uint16_t* __restrict__ k_w, float eps,
    const float* __restrict__ cache, float* __restrict__ kt, uint16_t* __restrict__ w_copy,
    float* __restrict__ cache_copy) {
  __shared__ float tile[kD][kTile + 1];
  const int lane16 = threadIdx.x & 15, t0 = blockIdx.x * kTile, hk = blockIdx.y, b = blockIdx.z;
  if (w_copy && blockIdx.x == 0 && hk == 0 && b == 0 && threadIdx.x < 16)
    *reinterpret_cast<uint4*>(w_copy + 8 * lane16) = load_u4(k_w + 8 * lane16);
  for (int i = threadIdx.x / 16; i < kTile; i += 16) {
    const int t = min(t0 + i, p.t - 1);
    const int64_t tok = (int64_t)b * p.t + t;
    const float r = inv_rms(k_mean[tok * p.hkv + hk], eps);
    if (cache_copy && hk == 0 && b == 0)
      store8f(cache_copy + t * kD + 8 * lane16, load8f(cache + t * kD + 8 * lane16));
    const V8 o = norm_rope(load8(p.qkv + tok * p.stride + (p.hq + hk) * kD + 8 * lane16),
                           load8(k_w + 8 * lane16), r, cache + t * kD, lane16);
#pragma unroll
    for (int e = 0; e < 8; ++e) tile[8 * lane16 + e][i] = o.v[e];
  }
  __syncthreads();
  const int rep = p.hq / p.hkv, i = threadIdx.x % kTile;
  if (t0 + i >= p.t) return;
  for (int g = 0; g < rep; ++g) {
    float* out = kt + ((int64_t)b * p.hq + hk * rep + g) * kD * p.t + t0 + i;
    for (int d = threadIdx.x / kTile; d < kD; d += kThreads / kTile) out[(int64_t)d * p.t] = tile[d][i];
  }
}

// Gradients of q and v: dn_q[tok][h][128] (bf16, of the norm's output), and dv
// into the packed gradient.
__global__ __launch_bounds__(kThreads) void qv_backward_kernel(
    Heads p, const float* __restrict__ dq, const float* __restrict__ dv,
    const float* __restrict__ cache, uint16_t* __restrict__ dn_q, uint16_t* __restrict__ dqkv) {
  const int lane16 = threadIdx.x & 15;
  const int per = p.hq + p.hkv;
  const uint32_t items = (uint32_t)p.batch * p.t * per;
  const uint32_t item = min(blockIdx.x * 16u + threadIdx.x / 16, items - 1);
  const uint32_t tok = item / per;
  const int h = item % per, b = tok / p.t, t = tok % p.t;
  if (h < p.hq) {
    const V8 g = rounded(load8f(dq + (((int64_t)b * p.hq + h) * p.t + t) * kD + 8 * lane16));
    const V8 o = rope_grad(g, cache + t * kD, lane16);
    *reinterpret_cast<uint4*>(dn_q + ((int64_t)tok * p.hq + h) * kD + 8 * lane16) = pack8(o);
  } else {
    const int hk = h - p.hq, rep = p.hq / p.hkv;
    const float* src = dv + (((int64_t)b * p.hq + hk * rep) * p.t + t) * kD + 8 * lane16;
    V8 s = load8f(src);
    for (int g = 1; g < rep; ++g) {
      const V8 a = load8f(src + (int64_t)g * p.t * kD);
#pragma unroll
      for (int e = 0; e < 8; ++e) s.v[e] += a.v[e];
    }
    *reinterpret_cast<uint4*>(dqkv + (int64_t)tok * p.stride + (p.hq + p.hkv + hk) * kD + 8 * lane16) =
        pack8(s);
  }
}

__global__ __launch_bounds__(kThreads) void k_backward_kernel(Heads p, const float* __restrict__ dkt,
                                                              const float* __restrict__ cache,
                                                              uint16_t* __restrict__ dn_k) {
  __shared__ float tile[kD][kTile + 1];
  const int t0 = blockIdx.x * kTile, hk = blockIdx.y, b = blockIdx.z, rep = p.hq / p.hkv;
  const int i = threadIdx.x % kTile;
  if (t0 + i < p.t) {
    const float* src = dkt + ((int64_t)b * p.hq + hk * rep) * kD * p.t + t0 + i;
    for (int d = threadIdx.x / kTile; d < kD; d += kThreads / kTile) {
      float s = src[(int64_t)d * p.t];
      for (int g = 1; g < rep; ++g) s += src[((int64_t)g * kD + d) * p.t];
      tile[d][i] = s;
    }
  }
  __syncthreads();
  const int lane16 = threadIdx.x & 15;
  for (int j = threadIdx.x / 16; j < kTile; j += 16) {
    const int t = min(t0 + j, p.t - 1), at = t - t0;
    V8 g;
#pragma unroll
    for (int e = 0; e < 8; ++e) g.v[e] = tile[8 * lane16 + e][at];
    const V8 o = rope_grad(rounded(g), cache + t * kD, lane16);
    if (t0 + j < p.t)
      *reinterpret_cast<uint4*>(dn_k + (((int64_t)b * p.t + t) * p.hkv + hk) * kD + 8 * lane16) = pack8(o);
  }
}

// [b][h][t][128] fp32 <-> [b][t][h][128] bf16.
template <bool TO_BF16>
__global__ __launch_bounds__(kThreads) void heads_kernel(float* __restrict__ f, uint16_t* __restrict__ o,
                                                         uint32_t items, int t_n, int h_n) {
  const uint32_t item = blockIdx.x * 16u + threadIdx.x / 16;
  if (item >= items) return;
  const int l = 8 * (threadIdx.x & 15);
  const uint32_t tok = item / h_n, h = item % h_n, b = tok / t_n, t = tok % t_n;
  float* src = f + (((int64_t)b * h_n + h) * t_n + t) * kD + l;
  uint16_t* dst = o + (int64_t)item * kD + l;
  if constexpr (TO_BF16)
    *reinterpret_cast<uint4*>(dst) = pack8(load8f(src));
  else
    store8f(src, load8(dst));
}

// out[row][j] = j > row % t ? masked : s * scale; row-major [rows][t].
__global__ __launch_bounds__(kThreads) void scale_mask_kernel(const float* __restrict__ s, int t, float scale,
                                                              float masked, float* __restrict__ out) {
  const uint32_t row = blockIdx.x;
  const int q = row % (uint32_t)t;
  const float* p = s + (int64_t)row * t;
  float* y = out + (int64_t)row * t;
  if (t % 4 == 0) {
    for (int j = 4 * threadIdx.x; j < t; j += 4 * kThreads) {
      f32x4_t v = {masked, masked, masked, masked};
      if (j <= q) {
        v = *reinterpret_cast<const f32x4_t*>(p + j);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = j + e > q ? masked : v[e] * scale;
      }
      *reinterpret_cast<f32x4_t*>(y + j) = v;
    }
  } else {
    for (int j = threadIdx.x; j < t; j += kThreads) y[j] = j > q ? masked : p[j] * scale;
  }
}

// Rows of causal attention, one wave each, NI x 64 columns: lane l holds
// columns l, l + 64, ..., adds its own in that order and the lanes by a
// butterfly of offsets 32 .. 1, the order of torch's softmax kernels for rows
// of at most 1,024, whose bits these are.  Columns past the diagonal hold
// exact zeros; the forward does not read them.  At 8 x 16 x 640 x 640 (210 MB)
// the forward reads half of it and writes it once, where mask and softmax moved
// four times as much; the backward reads half of w and all of dp.
__device__ __forceinline__ float butterfly_sum(float x) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) x += __shfl_xor(x, o, 64);
  return x;
}

template <int NI>
__global__ __launch_bounds__(kThreads) void causal_softmax_kernel(const float* __restrict__ s,
                                                                  uint32_t rows, int t, float scale,
                                                                  float* __restrict__ out) {
  const uint32_t row = blockIdx.x * (kThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63, q = row % (uint32_t)t;  // q, and so which chunks are skipped: uniform
  const float* p = s + (int64_t)row * t;
  float* y = out + (int64_t)row * t;
  float v[NI];
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int j = lane + 64 * i;
    v[i] = -INFINITY;
    if (64 * i > q) continue;
    if (j <= q) v[i] = p[j] * scale;
    m = v[i] > m || v[i] != v[i] ? v[i] : m;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float b = __shfl_xor(m, o, 64);
    m = m < b ? b : m;
  }
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    if (64 * i > q) continue;
    v[i] = expf(v[i] - m);
    sum += v[i];
  }
  sum = butterfly_sum(sum);
  const float past = 0.f / sum;  // a row of infinities or NaN is NaN past the diagonal too
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int j = lane + 64 * i;
    if (j < t) y[j] = j <= q ? v[i] / sum : past;
  }
}

// ds = (dp * w - w * sum(dp * w)) * scale, the difference an FMA as in torch's
// kernel.  dp past the diagonal is read for its infinities and NaN, which make
// the row's sum NaN although w is zero there.
template <int NI>
__global__ __launch_bounds__(kThreads) void causal_softmax_grad_kernel(const float* __restrict__ dp,
                                                                       const float* __restrict__ w,
                                                                       uint32_t rows, int t, float scale,
                                                                       float* __restrict__ ds) {
  const uint32_t row = blockIdx.x * (kThreads / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  if (row >= rows) return;
  const int lane = threadIdx.x & 63, q = row % (uint32_t)t;  // q, and so which chunks are skipped: uniform
  const float* p = dp + (int64_t)row * t;
  const float* pw = w + (int64_t)row * t;
  float* y = ds + (int64_t)row * t;
  // Loads without branches around them (indexes held inside the row), so that
  // all are in flight at once.
  float g[NI], o[NI];
#pragma unroll
  for (int i = 0; i < NI; ++i) g[i] = p[min(lane + 64 * i, t - 1)];
#pragma unroll
  for (int i = 0; i < NI; ++i) o[i] = 64 * i > q ? 0.f : pw[min(lane + 64 * i, q)];
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int j = lane + 64 * i;
    if (j > q) o[i] = 0.f;
    g[i] = j < t ? g[i] * o[i] : 0.f;
    sum += g[i];
  }
  sum = butterfly_sum(sum);
#pragma unroll
  for (int i = 0; i < NI; ++i) {
    const int j = lane + 64 * i;
    if (j < t) y[j] = j <= q ? fmaf(-o[i], sum, g[i]) * scale : 0.f;
  }
}

// y = bf16(sum of `parts` fp32 rows), summed in two levels of a fixed order:
// workgroup = 16 columns x 64 row groups, each with 8 loads in flight (16
// groups of one load each took 20 us for 1,024 rows).
constexpr int kSumGroups = 64;
__global__ __launch_bounds__(16 * kSumGroups) void sum_rows_kernel(const float* __restrict__ x, int parts,
                                                                   int n, uint16_t* __restrict__ y) {
  __shared__ float sm[kSumGroups][17];
  const int c = threadIdx.x % 16, grp = threadIdx.x / 16, col = blockIdx.x * 16 + c;
  float s = 0.f;
  if (col < n)
    for (int r = grp; r < parts; r += 8 * kSumGroups) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const int rr = r + k * kSumGroups;
        v[k] = rr < parts ? x[(int64_t)rr * n + col] : 0.f;
      }
#pragma unroll
      for (int k = 0; k < 8; ++k) s += v[k];
    }
  sm[grp][c] = s;
  __syncthreads();
  if (threadIdx.x < 16 && col < n) {
    s = sm[0][c];
#pragma unroll
    for (int g = 1; g < kSumGroups; ++g) s += sm[g][c];
    y[col] = f32_to_bf16(s);
  }
}

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

// A launch has fewer than 2^32 lanes in x, whole workgroups.
constexpr int64_t kMaxLanes = (1LL << 32) - kThreads;

// Items of 8 elements; 32-bit item arithmetic.
int check_rows(int64_t rows, int64_t stride, int64_t heads, int64_t n) {
  if (rows <= 0 || heads <= 0 || n <= 0 || rows % heads) return QMI_E_BAD_SHAPE;
  if (n % 8 || n > 65536 || rows > 0x7fffffffLL || rows * (n / 8) > 0x7fffff00LL) return QMI_E_UNSUPPORTED;
  if (stride < heads * n || stride % 8) return QMI_E_BAD_STRIDE;
  return QMI_OK;
}

unsigned grid_of(int64_t items) { return (unsigned)((items + kThreads - 1) / kThreads); }

int check_heads(int64_t batch, int64_t t, int64_t hq, int64_t hkv) {
  if (batch <= 0 || t <= 0 || hq <= 0 || hkv <= 0 || hq % hkv) return QMI_E_BAD_SHAPE;
  if (batch > 65535 || t > 0x7fffffffLL || hq > 65535 || hkv > 65535 ||
      batch * t * (hq + hkv) > kMaxLanes / 16)
    return QMI_E_UNSUPPORTED;
  return QMI_OK;
}

}  // namespace

#define QMI_ST reinterpret_cast<hipStream_t>(stream)

extern "C" int qmi_square_rows(const uint16_t* x, int64_t rows, int64_t stride, int64_t heads, int64_t n,
                               float* sq, uint16_t* x_copy, float* zero, void* stream) {
  const int e = check_rows(rows, stride, heads, n);
  if (e != QMI_OK) return e;
  if (!x || !sq) return QMI_E_NULL_POINTER;
  if (!al16(x) || !al16(sq) || !al16(x_copy)) return QMI_E_BAD_STRIDE;
  hipLaunchKernelGGL(square_kernel, dim3(grid_of(rows * (n / 8))), dim3(kThreads), 0, QMI_ST, x,
                     Rows{rows, stride, (int)heads, (int)n}, sq, x_copy, zero);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_norm_apply(const uint16_t* x, int64_t rows, int64_t stride, int64_t n, const float* mean,
                              const uint16_t* w, float eps, uint16_t* y, uint16_t* w_copy, void* stream) {
  const int e = check_rows(rows, stride, 1, n);
  if (e != QMI_OK) return e;
  if (!x || !mean || !w || !y) return QMI_E_NULL_POINTER;
  if (!al16(x) || !al16(w) || !al16(y) || !al16(w_copy)) return QMI_E_BAD_STRIDE;
  hipLaunchKernelGGL(norm_apply_kernel, dim3(grid_of(rows * (n / 8))), dim3(kThreads), 0, QMI_ST, x,
                     Rows{rows, stride, 1, (int)n}, mean, w, eps, y, w_copy);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_norm_prod(const uint16_t* x, int64_t rows, int64_t stride, int64_t heads, int64_t n,
                             const uint16_t* w, const uint16_t* dy, float* prod, void* stream) {
  const int e = check_rows(rows, stride, heads, n);
  if (e != QMI_OK) return e;
  if (!x || !w || !dy || !prod) return QMI_E_NULL_POINTER;
  if (!al16(x) || !al16(w) || !al16(dy) || !al16(prod)) return QMI_E_BAD_STRIDE;
  hipLaunchKernelGGL(norm_prod_kernel, dim3(grid_of(rows * (n / 8))), dim3(kThreads), 0, QMI_ST, x,
                     Rows{rows, stride, (int)heads, (int)n}, w, dy, prod);
  QMI_RETURN_LAUNCH_STATUS();
}

// Workgroups of norm_grad_kernel = rows of dw partials: four per CU at most.
extern "C" int64_t qmi_norm_grad_parts(int64_t rows, int64_t n) {
  if (rows <= 0 || n <= 0 || n % 8) return 0;
  const int64_t groups = n / 8 >= kThreads ? 1 : kThreads / (n / 8);
  return std::min<int64_t>((rows + groups - 1) / groups, 1024);
}

extern "C" int qmi_norm_grad(const uint16_t* x, int64_t rows, int64_t stride, int64_t heads, int64_t n,
                             const float* mean, const uint16_t* w, float eps, const uint16_t* dy,
                             const float* dr, uint16_t* dx, float* dw, void* stream) {
  const int e = check_rows(rows, stride, heads, n);
  if (e != QMI_OK) return e;
  if (!x || !mean || !w || !dy || !dr || !dx || !dw) return QMI_E_NULL_POINTER;
  if (!al16(x) || !al16(w) || !al16(dy) || !al16(dx) || !al16(dw)) return QMI_E_BAD_STRIDE;
  hipLaunchKernelGGL(norm_grad_kernel, dim3((unsigned)qmi_norm_grad_parts(rows, n)), dim3(kThreads), 0,
                     QMI_ST, x, Rows{rows, stride, (int)heads, (int)n}, mean, w, eps, dy, dr, dx, dw);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_silu_mul_train(const uint16_t* gate_up, int64_t rows, int64_t inter, const uint16_t* dy,
                                  uint16_t* out, void* stream) {
  const int e = check_rows(rows, 2 * inter, 1, 2 * inter);
  if (e != QMI_OK) return e;
  if (inter % 8) return QMI_E_UNSUPPORTED;
  if (!gate_up || !out) return QMI_E_NULL_POINTER;
  if (!al16(gate_up) || !al16(dy) || !al16(out)) return QMI_E_BAD_STRIDE;
  const dim3 grid(grid_of(rows * (inter / 8)));
  if (dy)
    hipLaunchKernelGGL(silu_mul_grad_kernel, grid, dim3(kThreads), 0, QMI_ST, gate_up, rows, (int)inter, dy, out);
  else
    hipLaunchKernelGGL(silu_mul_exact_kernel, grid, dim3(kThreads), 0, QMI_ST, gate_up, rows, (int)inter, out);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_train_qkv(const uint16_t* qkv, int64_t stride, int64_t batch, int64_t t, int64_t hq,
                             int64_t hkv, const float* q_mean, const float* k_mean, const uint16_t* q_w,
                             const uint16_t* k_w, float eps, const float* cache, float* qf, float* kt,
                             float* vf, uint16_t* w_copy, float* cache_copy, void* stream) {
  const int e = check_heads(batch, t, hq, hkv);
  if (e != QMI_OK) return e;
  if (!qkv || !q_mean || !k_mean || !q_w || !k_w || !cache || !qf || !kt || !vf) return QMI_E_NULL_POINTER;
  if (stride < (hq + 2 * hkv) * kD || stride % 8 || !al16(qkv) || !al16(q_w) || !al16(k_w) || !al16(cache) ||
      !al16(qf) || !al16(vf) || !al16(w_copy) || !al16(cache_copy))
    return QMI_E_BAD_STRIDE;
  const Heads p{qkv, stride, (int)batch, (int)t, (int)hq, (int)hkv};
  hipLaunchKernelGGL(qv_forward_kernel, dim3((unsigned)((batch * t * (hq + hkv) + 15) / 16)), dim3(kThreads), 0,
                     QMI_ST, p, q_mean, q_w, eps, cache, qf, vf, w_copy);
  hipLaunchKernelGGL(k_forward_kernel, dim3((unsigned)((t + kTile - 1) / kTile), (unsigned)hkv, (unsigned)batch),
                     dim3(kThreads), 0, QMI_ST, p, k_mean, k_w, eps, cache, kt, w_copy ? w_copy + kD : nullptr, cache_copy);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_train_qkv_grad(int64_t batch, int64_t t, int64_t hq, int64_t hkv, const float* dq,
                                  const float* dkt, const float* dv, const float* cache, uint16_t* dn_q,
                                  uint16_t* dn_k, uint16_t* dqkv, void* stream) {
  const int e = check_heads(batch, t, hq, hkv);
  if (e != QMI_OK) return e;
  if (!dq || !dkt || !dv || !cache || !dn_q || !dn_k || !dqkv) return QMI_E_NULL_POINTER;
  if (!al16(dq) || !al16(dv) || !al16(cache) || !al16(dn_q) || !al16(dn_k) || !al16(dqkv))
    return QMI_E_BAD_STRIDE;
  const Heads p{nullptr, (hq + 2 * hkv) * kD, (int)batch, (int)t, (int)hq, (int)hkv};
  hipLaunchKernelGGL(qv_backward_kernel, dim3((unsigned)((batch * t * (hq + hkv) + 15) / 16)), dim3(kThreads), 0,
                     QMI_ST, p, dq, dv, cache, dn_q, dqkv);
  hipLaunchKernelGGL(k_backward_kernel, dim3((unsigned)((t + kTile - 1) / kTile), (unsigned)hkv, (unsigned)batch),
                     dim3(kThreads), 0, QMI_ST, p, dkt, cache, dn_k);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_train_heads(float* f, uint16_t* o, int64_t batch, int64_t t, int64_t heads, int32_t to_bf16,
                               void* stream) {
  const int e = check_heads(batch, t, heads, heads);
  if (e != QMI_OK) return e;
  if (!f || !o) return QMI_E_NULL_POINTER;
  if (!al16(f) || !al16(o)) return QMI_E_BAD_STRIDE;
  const uint32_t items = (uint32_t)(batch * t * heads);
  const dim3 grid((items + 15) / 16);
  if (to_bf16)
    hipLaunchKernelGGL(heads_kernel<true>, grid, dim3(kThreads), 0, QMI_ST, f, o, items, (int)t, (int)heads);
  else
    hipLaunchKernelGGL(heads_kernel<false>, grid, dim3(kThreads), 0, QMI_ST, f, o, items, (int)t, (int)heads);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_scale_mask(const float* s, int64_t rows, int64_t t, float scale, float masked, float* out,
                              void* stream) {
  if (rows <= 0 || t <= 0 || rows % t) return QMI_E_BAD_SHAPE;
  if (rows > kMaxLanes / kThreads || t > 0x7fffffffLL / 4) return QMI_E_UNSUPPORTED;
  if (!s || !out) return QMI_E_NULL_POINTER;
  if (!al16(s) || !al16(out)) return QMI_E_BAD_STRIDE;
  hipLaunchKernelGGL(scale_mask_kernel, dim3((unsigned)rows), dim3(kThreads), 0, QMI_ST, s, (int)t, scale, masked,
                     out);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_sum_rows(const float* x, int64_t parts, int64_t n, uint16_t* y, void* stream) {
  if (parts <= 0 || n <= 0) return QMI_E_BAD_SHAPE;
  if (parts > (1 << 20) || n > (1 << 20)) return QMI_E_UNSUPPORTED;
  if (!x || !y) return QMI_E_NULL_POINTER;
  hipLaunchKernelGGL(sum_rows_kernel, dim3((unsigned)((n + 15) / 16)), dim3(16 * kSumGroups), 0, QMI_ST, x, (int)parts,
                     (int)n, y);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_causal_softmax(const float* s, const float* w, int64_t rows, int64_t t, float scale,
                                  float* out, void* stream) {
  if (rows <= 0 || t <= 0 || rows % t) return QMI_E_BAD_SHAPE;
  if (rows > kMaxLanes / 64 || t > 1024) return QMI_E_UNSUPPORTED;
  if (!s || !out) return QMI_E_NULL_POINTER;
  const dim3 grid((unsigned)((rows + kThreads / 64 - 1) / (kThreads / 64)));
#define QMI_CS(NI)                                                                                       \
  if (t <= 64 * NI) {                                                                                    \
    if (w)                                                                                               \
      hipLaunchKernelGGL(causal_softmax_grad_kernel<NI>, grid, dim3(kThreads), 0, QMI_ST, s, w,          \
                         (uint32_t)rows, (int)t, scale, out);                                            \
    else                                                                                                 \
      hipLaunchKernelGGL(causal_softmax_kernel<NI>, grid, dim3(kThreads), 0, QMI_ST, s, (uint32_t)rows,  \
                         (int)t, scale, out);                                                            \
    QMI_RETURN_LAUNCH_STATUS();                                                                          \
  }
  QMI_CS(1)
  QMI_CS(2)
  QMI_CS(4)
  QMI_CS(8)
  QMI_CS(12)
  QMI_CS(16)
#undef QMI_CS
  return QMI_E_UNSUPPORTED;
}
