// Causal GQA attention of a training batch, forward and backward, on bf16
// MFMA (gfx950).
//
// Reference semantics: the batch path of Qwen3Attention.forward
// (qwen3_naive.py:553-593) after QK-norm and RoPE: softmax(q k^T * scale,
// causal) v over whole sequences of T tokens, query head h reading KV head
// h / G.  That core holds scores, probabilities and their gradients in fp32;
// q, k, v and the output's gradient are bf16 there too.  So are they here:
//   * the products of two bf16 tensors (q k^T, dO v^T) are exact in fp32 and
//     accumulate in fp32;
//   * probabilities P and score gradients dS stay fp32 and enter the second
//     products (P v, P^T dO, dS k, dS^T q) as two bf16 terms, hi + lo (16
//     significant bits), both multiplied and accumulated in fp32: what is
//     left out is 2^-17 of each term, against the 2^-9 rounding of the bf16
//     results;
//   * the row dot products delta = dO . O use the fp32 output.
//
// Three kernels, all of one shape: a workgroup of 4 waves keeps 16 rows per
// wave (the forward 16 J) as MFMA B operands in registers (queries, or keys for dK / dV) and
// streams 64-row tiles of the other side through LDS, double-buffered, each
// staged once for all waves.  A tile is read two ways: rows as the A operand
// of the first products (ds_read_b128) and, transposed by ds_read_b64_tr_b16,
// as the A operand of the second.  The accumulator layout of the first
// product (lane: 4 consecutive rows of the tile, one column) is the B layout
// of the second, so P and dS never leave registers.  16-byte chunk c of row r
// sits at c ^ swz(r), a bijection on 16 rows (row reads) that also spreads
// the 8 rows a transpose read's 32 lanes touch over all 64 banks.
//
//   forward : rows = queries, tiles = K / V; online softmax; O in bf16 and,
//             for a backward, in fp32 with each row's (max, 1 / sum)
//   dQ      : rows = queries, tiles = K / V; writes delta for the next kernel
//   dK / dV : rows = keys, tiles = Q / dO of the group's G heads in turn, so
//             the sum over the group stays in the accumulators
// Separate dQ and dK / dV kernels recompute the scores once more than one
// kernel with atomic dQ would, and give the same bits on every run.
//
// What bounds them: the causal products are small beside the projections
// (8 x 640 tokens, 16 heads: 20 GFLOP with the split forward, 67 backward), so
// the chain score -> exp -> split -> product of a wave is; two waves per SIMD
// hide it, which the register budget is kept to (the forward at 296 registers
// and one wave: 64.7 us instead of 48.5).  With 32 rows per wave each LDS
// operand feeds two MFMAs; in the backward kernels that takes them to one wave
// per SIMD (8 x 640: 177 us instead of 136).  Measured at 8 x 640: forward
// 48.5 us, dQ + dK / dV 136 us, where the torch core took 2.4 ms.
#include <algorithm>

#include "qmi_common.h"

namespace {

using namespace qmi;

constexpr int kD = 128;
constexpr int kThreads = 256;
constexpr int kTile = 64;
constexpr int kTileElems = kTile * kD;
typedef __attribute__((ext_vector_type(4))) short v4s_t;

// Chunk swizzle of row r (only r % 16 matters).
__device__ __forceinline__ int swz(int r) { return ((r & 3) << 1) | ((r & 4) << 1) | ((r >> 3) & 1); }

// A 64-row tile in flight: 4 chunks of 16 bytes per thread.
struct Stage {
  uint4 v[4];
};

// Rows r0 .. r0+63 of `base` (row stride in elements); rows at or past n are zeros.
__device__ __forceinline__ Stage load_tile(const uint16_t* __restrict__ base, int64_t stride, int r0, int n) {
  Stage s;
  const int rr = threadIdx.x >> 4, ch = threadIdx.x & 15;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = r0 + rr + 16 * i;
    s.v[i] = r < n ? load_u4(base + (int64_t)r * stride + 8 * ch) : make_uint4(0, 0, 0, 0);
  }
  return s;
}

__device__ __forceinline__ void store_tile(uint16_t* lds, const Stage& s) {
  const int rr = threadIdx.x >> 4, ch = threadIdx.x & 15;
#pragma unroll
  for (int i = 0; i < 4; ++i)
    *reinterpret_cast<uint4*>(lds + (rr + 16 * i) * kD + 8 * (ch ^ swz(rr))) = s.v[i];
}

// A operand: rows 16 kb + l16, dims 32 c + 8 g4 ..+8.
__device__ __forceinline__ bf16x8_t row_operand(const uint16_t* lds, int kb, int c, int l16, int g4) {
  return *reinterpret_cast<const bf16x8_t*>(lds + (16 * kb + l16) * kD + 8 * ((4 * c + g4) ^ swz(l16)));
}

// Transposed A operand: dim 16 db + l16; rows 32 c + 4 g4 + (0..3), then 16 further.
__device__ __forceinline__ bf16x8_t col_operand(const uint16_t* lds, int c, int db, int l16, int g4) {
  const int row = 4 * g4 + (l16 >> 2);
  const uint16_t* p = lds + (32 * c + row) * kD + 8 * ((2 * db + ((l16 & 3) >> 1)) ^ swz(row)) + 4 * (l16 & 1);
  typedef __attribute__((address_space(3))) v4s_t lds_v4s;
  const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(const_cast<uint16_t*>(p)));
  const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(const_cast<uint16_t*>(p) + 16 * kD));
  typedef __attribute__((ext_vector_type(8))) short v8s_t;
  return __builtin_bit_cast(bf16x8_t, v8s_t{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
}

__device__ __forceinline__ f32x4_t mfma(bf16x8_t a, bf16x8_t b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Elements of row blocks 2c, 2c+1 as hi + lo bf16 B operands.
__device__ __forceinline__ void split_operand(const f32x4_t& a, const f32x4_t& b, bf16x8_t& hi, bf16x8_t& lo) {
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const __bf16 ha = (__bf16)a[r], hb = (__bf16)b[r];
    hi[r] = ha;
    hi[4 + r] = hb;
    lo[r] = (__bf16)(a[r] - (float)ha);
    lo[4 + r] = (__bf16)(b[r] - (float)hb);
  }
}

// The wave's 16 rows from r0 as B operands (rows at or past n are zeros).
__device__ __forceinline__ void load_rows(const uint16_t* __restrict__ base, int64_t stride, int r0, int n, int l16,
                                          int g4, bf16x8_t (&op)[4]) {
  const int r = r0 + l16;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const uint4 v = r < n ? load_u4(base + (int64_t)r * stride + 32 * c + 8 * g4) : make_uint4(0, 0, 0, 0);
    op[c] = __builtin_bit_cast(bf16x8_t, u32x4_t{v.x, v.y, v.z, v.w});
  }
}

// acc[db] holds dims 16 db + 4 g4 + (0..3) of the lane's row: 8 bytes of bf16 each.
__device__ __forceinline__ void store_row_bf16(uint16_t* __restrict__ dst, const f32x4_t (&acc)[8], float f, int g4) {
#pragma unroll
  for (int db = 0; db < 8; ++db)
    *reinterpret_cast<uint2*>(dst + 16 * db + 4 * g4) =
        make_uint2(pack_bf16x2(acc[db][0] * f, acc[db][1] * f), pack_bf16x2(acc[db][2] * f, acc[db][3] * f));
}

struct AttnArgs {
  const uint16_t *q, *k, *v;
  int64_t q_ts, k_ts, v_ts;  // token strides (elements); heads are 128 apart
  int T, Hq, Hkv;
  float scale, scale_log2;
  uint16_t* out;
  int64_t out_ts;
  float* out32;   // [B * T, Hq, 128] fp32, or null
  float2* stat;   // [B, Hq, T] (max in the log2 domain, 1 / sum), or null
  const uint16_t* dout;
  int64_t dout_ts;
  float* delta;   // [B, Hq, T]
  uint16_t *dq, *dk, *dv;
  int64_t dq_ts, dk_ts, dv_ts;
};

// Blocks: x = query head with the KV head fastest (with 8 KV heads a KV head
// stays on one XCD and its K / V in that XCD's L2), y = sequence, z = query
// block, the long late blocks first.
template <int J>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2))) void train_attn_forward(const AttnArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t sK[2][kTileElems], sV[2][kTileElems];
  const int lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.Hq / a.Hkv, kvh = blockIdx.x % a.Hkv, h = kvh * G + blockIdx.x / a.Hkv, b = blockIdx.y;
  const int q0 = (gridDim.z - 1 - blockIdx.z) * (64 * J), wq0 = q0 + wave * 16 * J;
  const int T = a.T;
  const int64_t tok0 = (int64_t)b * T;
  const uint16_t* qb = a.q + tok0 * a.q_ts + h * kD;
  const uint16_t* kb0 = a.k + tok0 * a.k_ts + kvh * kD;
  const uint16_t* vb0 = a.v + tok0 * a.v_ts + kvh * kD;
  const int kend = min(q0 + 64 * J, T), n_tiles = (kend + kTile - 1) / kTile;
  Stage ks = load_tile(kb0, a.k_ts, 0, T), vs = load_tile(vb0, a.v_ts, 0, T);
  bf16x8_t qop[J][4];
#pragma unroll
  for (int j = 0; j < J; ++j) load_rows(qb, a.q_ts, wq0 + 16 * j, T, l16, g4, qop[j]);
  float m_run[J], l_run[J];
  f32x4_t acc[J][8];
#pragma unroll
  for (int j = 0; j < J; ++j) {
    m_run[j] = -INFINITY;
    l_run[j] = 0.f;
#pragma unroll
    for (int db = 0; db < 8; ++db) acc[j][db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }
  store_tile(sK[0], ks);
  store_tile(sV[0], vs);
  __syncthreads();
  for (int t = 0; t < n_tiles; ++t) {
    const int buf = t & 1;
    const bool more = t + 1 < n_tiles;
    if (more) {
      ks = load_tile(kb0, a.k_ts, (t + 1) * kTile, T);
      vs = load_tile(vb0, a.v_ts, (t + 1) * kTile, T);
    }
    f32x4_t s[J][4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
#pragma unroll
      for (int j = 0; j < J; ++j) s[j][kb] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const bf16x8_t op = row_operand(sK[buf], kb, c, l16, g4);
#pragma unroll
        for (int j = 0; j < J; ++j) s[j][kb] = mfma(op, qop[j][c], s[j][kb]);
      }
    }
    const int key0 = t * kTile;
    const bool full = key0 + kTile - 1 <= wq0;  // every key visible to every query of the wave
    bf16x8_t hi[J][2], lo[J][2];
#pragma unroll
    for (int j = 0; j < J; ++j) {
      if (!full) {
        const int lim = wq0 + 16 * j + l16 - key0 - 4 * g4;  // key 16 kb + r visible iff <= lim
#pragma unroll
        for (int kb = 0; kb < 4; ++kb)
#pragma unroll
          for (int r = 0; r < 4; ++r) s[j][kb][r] = 16 * kb + r <= lim ? s[j][kb][r] : -INFINITY;
      }
      float mx = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) mx = fmaxf(mx, s[j][kb][r]);
      mx = rows4_max(mx) * a.scale_log2;
      // The maximum is only raised when it grows by more than 2^8: P stays
      // below 2^8 and most tiles skip the rescale.
      const bool need = mx > m_run[j] + 8.f;
      if (__ballot(need) != 0ull) {
        const float m_new = need ? mx : m_run[j];
        const float alpha = need ? fast_exp2(m_run[j] - m_new) : 1.f;
        m_run[j] = m_new;
        l_run[j] *= alpha;
#pragma unroll
        for (int db = 0; db < 8; ++db) acc[j][db] *= alpha;
      }
      float sum = 0.f;
#pragma unroll
      for (int kb = 0; kb < 4; ++kb)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          s[j][kb][r] = fast_exp2(fmaf(s[j][kb][r], a.scale_log2, -m_run[j]));
          sum += s[j][kb][r];
        }
      l_run[j] += sum;
#pragma unroll
      for (int c = 0; c < 2; ++c) split_operand(s[j][2 * c], s[j][2 * c + 1], hi[j][c], lo[j][c]);
    }
#pragma unroll
    for (int db = 0; db < 8; ++db)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const bf16x8_t op = col_operand(sV[buf], c, db, l16, g4);
#pragma unroll
        for (int j = 0; j < J; ++j) {
          acc[j][db] = mfma(op, lo[j][c], acc[j][db]);
          acc[j][db] = mfma(op, hi[j][c], acc[j][db]);
        }
      }
    if (more) {
      store_tile(sK[buf ^ 1], ks);
      store_tile(sV[buf ^ 1], vs);
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < J; ++j) {
    const int qi = wq0 + 16 * j + l16;
    const float inv = 1.0f / rows4_sum(l_run[j]);
    if (qi >= T) continue;
    store_row_bf16(a.out + (tok0 + qi) * a.out_ts + h * kD, acc[j], inv, g4);
    if (a.out32) {
      float* o = a.out32 + ((tok0 + qi) * a.Hq + h) * kD + 4 * g4;
#pragma unroll
      for (int db = 0; db < 8; ++db) *reinterpret_cast<f32x4_t*>(o + 16 * db) = acc[j][db] * inv;
      if (g4 == 0) a.stat[((int64_t)b * a.Hq + h) * T + qi] = make_float2(m_run[j], inv);
    }
  }
}

__global__ __launch_bounds__(kThreads) void train_attn_dq(const AttnArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t sK[2][kTileElems], sV[2][kTileElems];
  const int lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.Hq / a.Hkv, kvh = blockIdx.x % a.Hkv, h = kvh * G + blockIdx.x / a.Hkv, b = blockIdx.y;
  const int q0 = (gridDim.z - 1 - blockIdx.z) * 64, wq0 = q0 + wave * 16;
  const int T = a.T;
  const int64_t tok0 = (int64_t)b * T;
  const uint16_t* kb0 = a.k + tok0 * a.k_ts + kvh * kD;
  const uint16_t* vb0 = a.v + tok0 * a.v_ts + kvh * kD;
  const int kend = min(q0 + 64, T), n_tiles = (kend + kTile - 1) / kTile;
  Stage ks = load_tile(kb0, a.k_ts, 0, T), vs = load_tile(vb0, a.v_ts, 0, T);
  bf16x8_t qop[4], dop[4];
  f32x4_t acc[8];
  const int qi = wq0 + l16;
  load_rows(a.q + tok0 * a.q_ts + h * kD, a.q_ts, wq0, T, l16, g4, qop);
  load_rows(a.dout + tok0 * a.dout_ts + h * kD, a.dout_ts, wq0, T, l16, g4, dop);
  const int64_t si = ((int64_t)b * a.Hq + h) * T + qi;
  const float2 st = qi < T ? a.stat[si] : make_float2(0.f, 0.f);
  const float m = st.x, inv = st.y;
  float d = 0.f;
  if (qi < T) {
    const float* o = a.out32 + ((tok0 + qi) * a.Hq + h) * kD + 8 * g4;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const f32x4_t o0 = *reinterpret_cast<const f32x4_t*>(o + 32 * c);
      const f32x4_t o1 = *reinterpret_cast<const f32x4_t*>(o + 32 * c + 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) d += (float)dop[c][e] * o0[e] + (float)dop[c][4 + e] * o1[e];
    }
  }
  const float delta = rows4_sum(d);
  if (qi < T && g4 == 0) a.delta[si] = delta;
#pragma unroll
  for (int db = 0; db < 8; ++db) acc[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  store_tile(sK[0], ks);
  store_tile(sV[0], vs);
  __syncthreads();
  for (int t = 0; t < n_tiles; ++t) {
    const int buf = t & 1;
    const bool more = t + 1 < n_tiles;
    if (more) {
      ks = load_tile(kb0, a.k_ts, (t + 1) * kTile, T);
      vs = load_tile(vb0, a.v_ts, (t + 1) * kTile, T);
    }
    const int key0 = t * kTile;
    const bool full = key0 + kTile - 1 <= wq0;
    bf16x8_t hi[2], lo[2];
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) {  // 32 keys at a time
      f32x4_t s[2], dp[2];
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const int kb = 2 * c2 + k2;
        s[k2] = dp[k2] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const bf16x8_t ok = row_operand(sK[buf], kb, c, l16, g4);
          const bf16x8_t ov = row_operand(sV[buf], kb, c, l16, g4);
          s[k2] = mfma(ok, qop[c], s[k2]);
          dp[k2] = mfma(ov, dop[c], dp[k2]);
        }
      }
      const int lim = wq0 + l16 - key0 - 4 * g4;
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float p = fast_exp2(fmaf(s[k2][r], a.scale_log2, -m)) * inv;
          const float ds = p * (dp[k2][r] - delta);
          s[k2][r] = full || 16 * (2 * c2 + k2) + r <= lim ? ds : 0.f;
        }
      split_operand(s[0], s[1], hi[c2], lo[c2]);
    }
#pragma unroll
    for (int db = 0; db < 8; ++db)
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const bf16x8_t op = col_operand(sK[buf], c, db, l16, g4);
        acc[db] = mfma(op, lo[c], acc[db]);
        acc[db] = mfma(op, hi[c], acc[db]);
      }
    if (more) {
      store_tile(sK[buf ^ 1], ks);
      store_tile(sV[buf ^ 1], vs);
    }
    __syncthreads();
  }
  if (qi < T) store_row_bf16(a.dq + (tok0 + qi) * a.dq_ts + h * kD, acc, a.scale, g4);
}

// Blocks: x = KV head, y = sequence, z = key block (the early blocks, seen by
// the most queries, first).
__global__ __launch_bounds__(kThreads) void train_attn_dkv(const AttnArgs a) {
  __shared__ __attribute__((aligned(16))) uint16_t sQ[2][kTileElems], sO[2][kTileElems];
  __shared__ __attribute__((aligned(16))) float sStat[2][3][kTile];  // max, 1 / sum, delta
  const int lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.Hq / a.Hkv, kvh = blockIdx.x, b = blockIdx.y;
  const int k0 = blockIdx.z * 64, wk0 = k0 + wave * 16;
  const int T = a.T;
  const int64_t tok0 = (int64_t)b * T;
  const int t_first = k0 / kTile, per_head = (T + kTile - 1) / kTile - t_first, n_steps = G * per_head;
  Stage qs, os;
  float2 st;
  float de;
  auto load_step = [&](int i) {
    const int h = kvh * G + i / per_head, r0 = (t_first + i % per_head) * kTile;
    qs = load_tile(a.q + tok0 * a.q_ts + h * kD, a.q_ts, r0, T);
    os = load_tile(a.dout + tok0 * a.dout_ts + h * kD, a.dout_ts, r0, T);
    const int qi = r0 + (int)threadIdx.x;
    const bool ok = threadIdx.x < kTile && qi < T;
    const int64_t si = ((int64_t)b * a.Hq + h) * T + qi;
    st = ok ? a.stat[si] : make_float2(0.f, 0.f);
    de = ok ? a.delta[si] : 0.f;
  };
  auto store_step = [&](int buf) {
    store_tile(sQ[buf], qs);
    store_tile(sO[buf], os);
    if (threadIdx.x < kTile) {
      sStat[buf][0][threadIdx.x] = st.x;
      sStat[buf][1][threadIdx.x] = st.y;
      sStat[buf][2][threadIdx.x] = de;
    }
  };
  load_step(0);
  bf16x8_t kop[4], vop[4];
  f32x4_t acc_k[8], acc_v[8];
  load_rows(a.k + tok0 * a.k_ts + kvh * kD, a.k_ts, wk0, T, l16, g4, kop);
  load_rows(a.v + tok0 * a.v_ts + kvh * kD, a.v_ts, wk0, T, l16, g4, vop);
#pragma unroll
  for (int db = 0; db < 8; ++db) acc_k[db] = acc_v[db] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  store_step(0);
  __syncthreads();
  for (int i = 0; i < n_steps; ++i) {
    const int buf = i & 1;
    const bool more = i + 1 < n_steps;
    if (more) load_step(i + 1);
    const int r0 = (t_first + i % per_head) * kTile;
    const bool full = wk0 + 15 <= r0 && r0 + kTile <= T;
#pragma unroll
    for (int c2 = 0; c2 < 2; ++c2) {  // 32 queries at a time
      f32x4_t s[2], dp[2];
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const int qb = 2 * c2 + k2;
        s[k2] = dp[k2] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const bf16x8_t oq = row_operand(sQ[buf], qb, c, l16, g4);
          const bf16x8_t oo = row_operand(sO[buf], qb, c, l16, g4);
          s[k2] = mfma(oq, kop[c], s[k2]);
          dp[k2] = mfma(oo, vop[c], dp[k2]);
        }
      }
      bf16x8_t phi, plo, dhi, dlo;
      const int key = wk0 + l16;
#pragma unroll
      for (int k2 = 0; k2 < 2; ++k2) {
        const int row = 16 * (2 * c2 + k2) + 4 * g4;
        const f32x4_t m4 = *reinterpret_cast<const f32x4_t*>(&sStat[buf][0][row]);
        const f32x4_t i4 = *reinterpret_cast<const f32x4_t*>(&sStat[buf][1][row]);
        const f32x4_t d4 = *reinterpret_cast<const f32x4_t*>(&sStat[buf][2][row]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const bool seen = full || (key <= r0 + row + r && r0 + row + r < T);
          const float p = fast_exp2(fmaf(s[k2][r], a.scale_log2, -m4[r])) * i4[r];
          const float ds = p * (dp[k2][r] - d4[r]);
          s[k2][r] = seen ? p : 0.f;
          dp[k2][r] = seen ? ds : 0.f;
        }
      }
      split_operand(s[0], s[1], phi, plo);
      split_operand(dp[0], dp[1], dhi, dlo);
#pragma unroll
      for (int db = 0; db < 8; ++db) {
        const bf16x8_t oo = col_operand(sO[buf], c2, db, l16, g4);
        const bf16x8_t oq = col_operand(sQ[buf], c2, db, l16, g4);
        acc_v[db] = mfma(oo, plo, acc_v[db]);
        acc_k[db] = mfma(oq, dlo, acc_k[db]);
        acc_v[db] = mfma(oo, phi, acc_v[db]);
        acc_k[db] = mfma(oq, dhi, acc_k[db]);
      }
    }
    if (more) store_step(buf ^ 1);
    __syncthreads();
  }
  const int key = wk0 + l16;
  if (key >= T) return;
  store_row_bf16(a.dk + (tok0 + key) * a.dk_ts + kvh * kD, acc_k, a.scale, g4);
  store_row_bf16(a.dv + (tok0 + key) * a.dv_ts + kvh * kD, acc_v, 1.f, g4);
}

// Forward: 32 queries per wave once that still gives every CU two workgroups
// (16 heads: 8 x 640 tokens 48.5 us against 52.1 with 16, 4 x 1,152 56.4 / 65.8,
// 1 x 4,096 157 / 165); below, 16 spread the work wider (2 x 389 17.0 / 21.9,
// 1 x 1,152 34 / 46).
bool wide_forward(int64_t workgroups) { return workgroups >= 2 * device_cu_count(); }

int check_shape(int64_t batch, int64_t T, int64_t Hq, int64_t Hkv, int64_t D) {
  if (batch < 0 || T < 0 || Hq <= 0 || Hkv <= 0 || Hq % Hkv) return QMI_E_BAD_SHAPE;
  if (D != kD || batch > 65535 || T > (1 << 22) || Hq > 4096) return QMI_E_UNSUPPORTED;
  if ((T + 63) / 64 > 65535) return QMI_E_UNSUPPORTED;
  return QMI_OK;
}

inline bool al(const void* p, unsigned n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

}  // namespace

extern "C" int qmi_train_attn_forward(const uint16_t* q, int64_t q_stride, const uint16_t* k, int64_t k_stride,
                                      const uint16_t* v, int64_t v_stride, int64_t batch, int64_t seq_len,
                                      int64_t num_q_heads, int64_t num_kv_heads, int64_t head_dim, float scale,
                                      uint16_t* out, int64_t out_stride, float* out_f32, float* stats, void* stream) {
  if (int e = check_shape(batch, seq_len, num_q_heads, num_kv_heads, head_dim)) return e;
  if (batch == 0 || seq_len == 0) return QMI_OK;
  if (!q || !k || !v || !out || !out_f32 != !stats) return QMI_E_NULL_POINTER;
  if (q_stride % 8 || k_stride % 8 || v_stride % 8 || out_stride % 4 || !al(q, 16) || !al(k, 16) || !al(v, 16) ||
      !al(out, 8) || !al(out_f32, 16) || !al(stats, 8) || q_stride < num_q_heads * kD ||
      k_stride < num_kv_heads * kD || v_stride < num_kv_heads * kD || out_stride < num_q_heads * kD)
    return QMI_E_BAD_STRIDE;
  AttnArgs a{};
  a.q = q, a.k = k, a.v = v, a.q_ts = q_stride, a.k_ts = k_stride, a.v_ts = v_stride;
  a.T = (int)seq_len, a.Hq = (int)num_q_heads, a.Hkv = (int)num_kv_heads;
  a.scale = scale, a.scale_log2 = scale * kLog2e;
  a.out = out, a.out_ts = out_stride, a.out32 = out_f32, a.stat = reinterpret_cast<float2*>(stats);
  const int64_t n128 = (seq_len + 127) / 128;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (wide_forward(n128 * batch * num_q_heads))
    hipLaunchKernelGGL(train_attn_forward<2>, dim3((unsigned)num_q_heads, (unsigned)batch, (unsigned)n128),
                       dim3(kThreads), 0, st, a);
  else
    hipLaunchKernelGGL(train_attn_forward<1>,
                       dim3((unsigned)num_q_heads, (unsigned)batch, (unsigned)((seq_len + 63) / 64)), dim3(kThreads),
                       0, st, a);
  QMI_RETURN_LAUNCH_STATUS();
}

extern "C" int qmi_train_attn_backward(const uint16_t* q, int64_t q_stride, const uint16_t* k, int64_t k_stride,
                                       const uint16_t* v, int64_t v_stride, const float* out_f32, const float* stats,
                                       const uint16_t* dout, int64_t dout_stride, int64_t batch, int64_t seq_len,
                                       int64_t num_q_heads, int64_t num_kv_heads, int64_t head_dim, float scale,
                                       float* delta, uint16_t* dq, int64_t dq_stride, uint16_t* dk, int64_t dk_stride,
                                       uint16_t* dv, int64_t dv_stride, void* stream) {
  if (int e = check_shape(batch, seq_len, num_q_heads, num_kv_heads, head_dim)) return e;
  if (batch == 0 || seq_len == 0) return QMI_OK;
  if (!q || !k || !v || !out_f32 || !stats || !dout || !delta || !dq || !dk || !dv) return QMI_E_NULL_POINTER;
  if (q_stride % 8 || k_stride % 8 || v_stride % 8 || dout_stride % 8 || dq_stride % 4 || dk_stride % 4 ||
      dv_stride % 4 || !al(q, 16) || !al(k, 16) || !al(v, 16) || !al(dout, 16) || !al(out_f32, 16) || !al(stats, 8) ||
      !al(dq, 8) || !al(dk, 8) || !al(dv, 8) || !al(delta, 4))
    return QMI_E_BAD_STRIDE;
  if (q_stride < num_q_heads * kD || dout_stride < num_q_heads * kD || dq_stride < num_q_heads * kD ||
      k_stride < num_kv_heads * kD || v_stride < num_kv_heads * kD || dk_stride < num_kv_heads * kD ||
      dv_stride < num_kv_heads * kD)
    return QMI_E_BAD_STRIDE;
  AttnArgs a{};
  a.q = q, a.k = k, a.v = v, a.q_ts = q_stride, a.k_ts = k_stride, a.v_ts = v_stride;
  a.T = (int)seq_len, a.Hq = (int)num_q_heads, a.Hkv = (int)num_kv_heads;
  a.scale = scale, a.scale_log2 = scale * kLog2e;
  a.out32 = const_cast<float*>(out_f32), a.stat = reinterpret_cast<float2*>(const_cast<float*>(stats));
  a.dout = dout, a.dout_ts = dout_stride, a.delta = delta;
  a.dq = dq, a.dk = dk, a.dv = dv, a.dq_ts = dq_stride, a.dk_ts = dk_stride, a.dv_ts = dv_stride;
  const int64_t n64 = (seq_len + 63) / 64;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(train_attn_dq, dim3((unsigned)num_q_heads, (unsigned)batch, (unsigned)n64), dim3(kThreads), 0, st,
                     a);
  hipLaunchKernelGGL(train_attn_dkv, dim3((unsigned)num_kv_heads, (unsigned)batch, (unsigned)n64), dim3(kThreads), 0,
                     st, a);
  QMI_RETURN_LAUNCH_STATUS();
}
