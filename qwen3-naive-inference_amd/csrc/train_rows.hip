// Row-wise backward kernels of the training batch (gfx950).
//
// Reference semantics: the gradients of the fp32 formulas of RMSNorm, the
// per-head QK-norm and RoPE (qwen3_naive.py:44-80, :156-169, :553-570), fp32
// math from bf16 tensors with one bf16 rounding of each result.
//
// All are HBM-bound: each input is read once, each gradient written once.  A
// weight's gradient is a sum over all rows: every workgroup keeps its rows'
// sums in registers and writes one fp32 partial row; sum_columns adds the
// partial rows in a fixed order (the same bits on every run).
#include <algorithm>

#include "qmi_common.h"

namespace {

using namespace qmi;

// out[c] = bf16(sum_p parts[p][c]): 32 columns x 8 partial-row groups per
// workgroup; columns below n0 go to out0, the others to out1.
__global__ __launch_bounds__(256) void sum_columns(const float* __restrict__ parts, int n_parts, int n, int n0,
                                                   uint16_t* __restrict__ out0, uint16_t* __restrict__ out1) {
  __shared__ float sm[8][32];
  const int lane = threadIdx.x & 31, grp = threadIdx.x >> 5;
  const int c = blockIdx.x * 32 + lane;
  float s = 0.f;
  if (c < n) {
#pragma unroll 8
    for (int p = grp; p < n_parts; p += 8) s += parts[(int64_t)p * n + c];
  }
  sm[grp][lane] = s;
  __syncthreads();
  if (grp == 0 && c < n) {
#pragma unroll
    for (int i = 1; i < 8; ++i) s += sm[i][lane];
    if (c < n0)
      out0[c] = f32_to_bf16(s);
    else
      out1[c - n0] = f32_to_bf16(s);
  }
}

// ---------------------------------------------------------------------------
// Gradient of per-head RMSNorm + RoPE (qk_norm_rope_kernel with positions
// tok % seq_len): 16 lanes per (token, head), lane s owns the RoPE pairs
// (4s + i, 64 + 4s + i).  The rotation's transpose gives the normalised
// head's gradient g; with x^ = x / rms, dw += g x^ and
// dx = (g w - x^ mean(g w x^)) / rms (the norm's bf16 rounding passes the
// gradient through unchanged).
__global__ __launch_bounds__(256) void qk_norm_rope_backward_kernel(
    const uint16_t* __restrict__ dq, int64_t dq_stride, const uint16_t* __restrict__ dk, int64_t dk_stride,
    const uint16_t* __restrict__ qkv, int64_t qkv_stride, int n_q_heads, int n_kv_heads,
    const uint16_t* __restrict__ q_w, const uint16_t* __restrict__ k_w, const float* __restrict__ cos_sin,
    int seq_len, int64_t n_tok, float eps, uint16_t* __restrict__ dqkv, int64_t dqkv_stride,
    float* __restrict__ parts) {
  constexpr int D = 128, HALF = 64;
  __shared__ float sm[4][2][D];
  const int sub = threadIdx.x & 15, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int heads = n_q_heads + n_kv_heads;
  const int64_t n_items = n_tok * heads, step = (int64_t)gridDim.x * 16;
  float aw[2][8];
#pragma unroll
  for (int i = 0; i < 8; ++i) aw[0][i] = aw[1][i] = 0.f;
  for (int64_t item = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4); item < n_items; item += step) {
    const int64_t tok = item / heads;
    const int h = (int)(item - tok * heads);
    const bool is_q = h < n_q_heads;
    const uint16_t* src = qkv + tok * qkv_stride + (int64_t)h * D;
    const uint16_t* w = is_q ? q_w : k_w;
    const uint16_t* go = is_q ? dq + tok * dq_stride + (int64_t)h * D
                              : dk + tok * dk_stride + (int64_t)(h - n_q_heads) * D;
    const uint2 xa = *reinterpret_cast<const uint2*>(src + 4 * sub);
    const uint2 xb = *reinterpret_cast<const uint2*>(src + HALF + 4 * sub);
    const uint2 ga = *reinterpret_cast<const uint2*>(go + 4 * sub);
    const uint2 gb = *reinterpret_cast<const uint2*>(go + HALF + 4 * sub);
    const uint2 wa = *reinterpret_cast<const uint2*>(w + 4 * sub);
    const uint2 wb = *reinterpret_cast<const uint2*>(w + HALF + 4 * sub);
    const float* cs = cos_sin + (int64_t)((uint32_t)tok % (uint32_t)seq_len) * D;
    const float4 c = *reinterpret_cast<const float4*>(cs + 4 * sub);
    const float4 sn = *reinterpret_cast<const float4*>(cs + HALF + 4 * sub);
    const float x1[4] = {bf16_lo(xa.x), bf16_hi(xa.x), bf16_lo(xa.y), bf16_hi(xa.y)};
    const float x2[4] = {bf16_lo(xb.x), bf16_hi(xb.x), bf16_lo(xb.y), bf16_hi(xb.y)};
    const float g1[4] = {bf16_lo(ga.x), bf16_hi(ga.x), bf16_lo(ga.y), bf16_hi(ga.y)};
    const float g2[4] = {bf16_lo(gb.x), bf16_hi(gb.x), bf16_lo(gb.y), bf16_hi(gb.y)};
    const float w1[4] = {bf16_lo(wa.x), bf16_hi(wa.x), bf16_lo(wa.y), bf16_hi(wa.y)};
    const float w2[4] = {bf16_lo(wb.x), bf16_hi(wb.x), bf16_lo(wb.y), bf16_hi(wb.y)};
    const float cc[4] = {c.x, c.y, c.z, c.w}, ss4[4] = {sn.x, sn.y, sn.z, sn.w};
    float ss = 0.f, dot = 0.f, n1[4], n2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ss += x1[i] * x1[i] + x2[i] * x2[i];
      n1[i] = g1[i] * cc[i] + g2[i] * ss4[i];
      n2[i] = g2[i] * cc[i] - g1[i] * ss4[i];
      dot += n1[i] * w1[i] * x1[i] + n2[i] * w2[i] * x2[i];
    }
    ss = row16_sum(ss);
    dot = row16_sum(dot);
    const float inv = rsqrtf(ss / (float)D + eps);
    const float mean = dot * inv / (float)D;  // mean of g w x^
    float o1[4], o2[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float h1 = x1[i] * inv, h2 = x2[i] * inv;
      o1[i] = inv * (n1[i] * w1[i] - h1 * mean);
      o2[i] = inv * (n2[i] * w2[i] - h2 * mean);
      const float a = n1[i] * h1, b = n2[i] * h2;
      aw[0][i] += is_q ? a : 0.f;
      aw[0][4 + i] += is_q ? b : 0.f;
      aw[1][i] += is_q ? 0.f : a;
      aw[1][4 + i] += is_q ? 0.f : b;
    }
    uint16_t* dst = dqkv + tok * dqkv_stride + (int64_t)h * D;
    *reinterpret_cast<uint2*>(dst + 4 * sub) = make_uint2(pack_bf16x2(o1[0], o1[1]), pack_bf16x2(o1[2], o1[3]));
    *reinterpret_cast<uint2*>(dst + HALF + 4 * sub) =
        make_uint2(pack_bf16x2(o2[0], o2[1]), pack_bf16x2(o2[2], o2[3]));
  }
#pragma unroll
  for (int k = 0; k < 2; ++k)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float s = rows4_sum(aw[k][i]);  // the wave's four items
      if (lane < 16) sm[wave][k][(i < 4 ? 0 : HALF - 4) + 4 * sub + i] = s;
    }
  __syncthreads();
  const int k = threadIdx.x >> 7, d = threadIdx.x & 127;
  parts[(int64_t)blockIdx.x * 256 + threadIdx.x] = sm[0][k][d] + sm[1][k][d] + sm[2][k][d] + sm[3][k][d];
}

inline bool al(const void* p, unsigned n) { return (reinterpret_cast<uintptr_t>(p) & (n - 1)) == 0; }

// Partial rows of a launch: two workgroups per CU, fewer when the rows run out.
int64_t part_rows(int64_t units, int64_t per_workgroup) {
  return std::max<int64_t>(1, std::min<int64_t>(2 * device_cu_count(), (units + per_workgroup - 1) / per_workgroup));
}

}  // namespace

extern "C" int64_t qmi_qk_norm_rope_backward_workspace_bytes(int64_t n_tok, int64_t num_q_heads,
                                                             int64_t num_kv_heads) {
  if (n_tok <= 0 || num_q_heads <= 0 || num_kv_heads <= 0) return 0;
  return part_rows(n_tok * (num_q_heads + num_kv_heads), 16) * 256 * 4;
}

extern "C" int qmi_qk_norm_rope_backward(const uint16_t* dq, int64_t dq_stride, const uint16_t* dk, int64_t dk_stride,
                                         const uint16_t* qkv, int64_t qkv_stride, int64_t n_tok, int64_t num_q_heads,
                                         int64_t num_kv_heads, int64_t head_dim, const uint16_t* q_norm_weight,
                                         const uint16_t* k_norm_weight, const float* cos_sin_cache, int64_t seq_len,
                                         float eps, uint16_t* dqkv, int64_t dqkv_stride, uint16_t* dq_norm_weight,
                                         uint16_t* dk_norm_weight, float* workspace, int64_t workspace_bytes,
                                         void* stream) {
  if (n_tok < 0 || num_q_heads <= 0 || num_kv_heads <= 0 || seq_len <= 0) return QMI_E_BAD_SHAPE;
  if (n_tok == 0) return QMI_OK;
  if (!dq || !dk || !qkv || !q_norm_weight || !k_norm_weight || !cos_sin_cache || !dqkv || !dq_norm_weight ||
      !dk_norm_weight || !workspace)
    return QMI_E_NULL_POINTER;
  if (head_dim != 128 || n_tok > 0x7fffffffLL || seq_len > 0x7fffffffLL || num_q_heads > 4096 || num_kv_heads > 4096)
    return QMI_E_UNSUPPORTED;
  const int64_t width = (num_q_heads + num_kv_heads) * 128;
  if (dq_stride % 4 || dk_stride % 4 || qkv_stride % 4 || dqkv_stride % 4 || !al(dq, 8) || !al(dk, 8) ||
      !al(qkv, 8) || !al(dqkv, 8) || !al(q_norm_weight, 8) || !al(k_norm_weight, 8) || !al(cos_sin_cache, 16) ||
      !al(workspace, 4) || qkv_stride < width || dqkv_stride < width || dq_stride < num_q_heads * 128 ||
      dk_stride < num_kv_heads * 128)
    return QMI_E_BAD_STRIDE;
  const int64_t parts = part_rows(n_tok * (num_q_heads + num_kv_heads), 16);
  if (workspace_bytes < parts * 256 * 4) return QMI_E_WORKSPACE_TOO_SMALL;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  hipLaunchKernelGGL(qk_norm_rope_backward_kernel, dim3((unsigned)parts), dim3(256), 0, st, dq, dq_stride, dk,
                     dk_stride, qkv, qkv_stride, (int)num_q_heads, (int)num_kv_heads, q_norm_weight, k_norm_weight,
                     cos_sin_cache, (int)seq_len, n_tok, eps, dqkv, dqkv_stride, workspace);
  hipLaunchKernelGGL(sum_columns, dim3(8), dim3(256), 0, st, workspace, (int)parts, 256, 128, dq_norm_weight,
                     dk_norm_weight);
  QMI_RETURN_LAUNCH_STATUS();
}
