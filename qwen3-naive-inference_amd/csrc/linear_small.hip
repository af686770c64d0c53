// Decode projections for at most 16 rows on bf16 MFMA (gfx950), with the
// residual add + RMSNorm that precedes a projection in its prologue.
//
// Reference semantics: the decode step's input / post-attention RMSNorm
// (RMSNorm._add_rms_norm, qwen3_naive.py:156-169) followed by qkv_proj or
// gate_up_proj + silu(gate) * up (:654, :699-701), and o_proj / down_proj
// (:683, :702), with the rounding points of qmi_add_rms_norm and
// qmi_linear_rows.
//
// A few rows make a decode layer a chain of launches of 3-7 us, each bound by
// latency: the launch, one trip to HBM for the weights, the epilogue.  So:
//   * One trip.  Workgroup = 8 waves = 16 weight rows; wave w takes an eighth
//     of K and loads its whole share of the weight rows straight into the
//     MFMA A registers (32 KB per workgroup at K = 1024), right after the few
//     rows that the norm waits for: loads return in order.
//   * The norm is computed by every workgroup while the weights are in flight
//     (16 KB of rows from L2 at 4 sequences), so the separate norm launch and
//     its gap go away; its output, the B operand, stays in LDS (16-byte chunks
//     XOR-swizzled by the row).  Row r's residual sum is written by workgroup
//     r (modulo the grid).  Every workgroup reads the rows anew, which costs
//     more than the launch from some rows x depth on; the callers' rules say
//     where (hidden 1024: 14 rows of 16).
//   * The 8 partial tiles are added in wave order through LDS: no split-K
//     partials in memory, so the next norm reads bf16 rows.
//   * SwiGLU (packed [gate; up] weight): 8 gate rows and their 8 up rows.
//
// Eight layers, 4 sequences of 37-700 tokens, as a graph: 324 -> 307 us with
// the weights' loads before the rows'; 279 with the rows' first, four weight rows
// per workgroup in o_proj / down_proj and 32-bit divisions in the attention's
// schedule; 274 with the attention merge's loads four at a time.
#include "qmi_common.h"

namespace {

using namespace qmi;

constexpr int kWaves = 8;
constexpr int kThreads = 64 * kWaves;
constexpr int kMaxRows = 16;

// NS: 32-deep k-steps per wave (K = 256 NS).  RPT: weight rows per workgroup;
// with 16 / RPT > 1 the 16 A rows of an MFMA are RPT weight rows at 16 / RPT
// parts of the wave's K range, each part has products of its own with the x
// rows, of which the blocks that belong together are kept.  ROWS: rows that a
// wave normalises (0: no norm).
template <int NS, int RPT, bool SWIGLU, int ROWS>
__global__ __launch_bounds__(kThreads) void linear_small_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ res,
    int64_t res_stride, uint16_t* __restrict__ res_out, int64_t res_out_stride,
    const uint16_t* __restrict__ norm_w, float eps, const uint16_t* __restrict__ w,
    int64_t w_stride, uint16_t* __restrict__ y, int64_t y_stride, int M, int N) {
  constexpr int K = 256 * NS, KW = K / kWaves;
  constexpr int P = 16 / RPT, NP = NS / P, KP = KW / P;  // parts, steps per part, their depth
  static_assert(NS % P == 0 && (!SWIGLU || P == 1), "tile");
  __shared__ __attribute__((aligned(16))) uint16_t xs[ROWS ? kMaxRows * K : 8];
  __shared__ __attribute__((aligned(16))) float red[kWaves][16][20];  // [wave][x row][A row], padded
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int l16 = lane & 15, g4 = lane >> 4;
  const int n0 = blockIdx.x * (SWIGLU ? 8 : RPT);
  const int64_t wrow = SWIGLU ? (l16 < 8 ? n0 + l16 : N + n0 + l16 - 8) : n0 + l16 % RPT;
  const uint16_t* wp = w + wrow * w_stride + wave * KW + l16 / RPT * KP + g4 * 8;
  uint4 wf[NP], xf[NS];
  if constexpr (ROWS > 0) {
    // The rows first, then the weights: loads return in order, and the norm
    // waits for the rows alone.
    constexpr int C = NS / 2;
    uint4 xr[ROWS][C], rr[ROWS][C], nw[C];
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int64_t row = min(wave + kWaves * i, M - 1);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        xr[i][c] = load_u4(x + row * x_stride + 8 * (64 * c + lane));
        rr[i][c] = res ? load_u4(res + row * res_stride + 8 * (64 * c + lane)) : make_uint4(0, 0, 0, 0);
      }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) nw[c] = load_u4(norm_w + 8 * (64 * c + lane));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < NP; ++j) wf[j] = load_u4(wp + 32 * j);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < ROWS; ++i) {
      const int row = wave + kWaves * i;
      if (row >= M) break;
      float v[C][8];
      float ss = 0.f;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint32_t aw[4] = {xr[i][c].x, xr[i][c].y, xr[i][c].z, xr[i][c].w};
        const uint32_t bw[4] = {rr[i][c].x, rr[i][c].y, rr[i][c].z, rr[i][c].w};
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[c][2 * e] = bf16_lo(aw[e]) + bf16_lo(bw[e]);
          v[c][2 * e + 1] = bf16_hi(aw[e]) + bf16_hi(bw[e]);
          o[e] = pack_bf16x2(v[c][2 * e], v[c][2 * e + 1]);
        }
        if (res && row % gridDim.x == blockIdx.x)
          *reinterpret_cast<uint4*>(res_out + row * res_out_stride + 8 * (64 * c + lane)) =
              make_uint4(o[0], o[1], o[2], o[3]);
#pragma unroll
        for (int e = 0; e < 8; ++e) ss += v[c][e] * v[c][e];
      }
      const float inv = rsqrtf(wave_sum(ss) / (float)K + eps);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint32_t ww[4] = {nw[c].x, nw[c].y, nw[c].z, nw[c].w};
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
          o[e] = pack_bf16x2(v[c][2 * e] * inv * bf16_lo(ww[e]),
                             v[c][2 * e + 1] * inv * bf16_hi(ww[e]));
        // Logical 16-byte chunk q of the row sits at q ^ row within its 16.
        const int q = 64 * c + lane;
        *reinterpret_cast<uint4*>(xs + row * K + 8 * (q ^ row)) = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
    __syncthreads();
    // Rows past M hold whatever LDS held: they only reach output rows past M.
#pragma unroll
    for (int j = 0; j < NS; ++j)
      xf[j] = *reinterpret_cast<const uint4*>(xs + l16 * K + 8 * ((wave * (KW / 8) + 4 * j + g4) ^ l16));
  } else {
    const uint16_t* xp = x + (int64_t)min(l16, M - 1) * x_stride + wave * KW + g4 * 8;
#pragma unroll
    for (int j = 0; j < NP; ++j) wf[j] = load_u4(wp + 32 * j);
#pragma unroll
    for (int j = 0; j < NS; ++j) xf[j] = load_u4(xp + 32 * j);
  }
  f32x4_t acc[P];  // A rows 4 g4 + r, x row l16
#pragma unroll
  for (int p = 0; p < P; ++p) {
    acc[p] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < NP; ++j)
      acc[p] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(bf16x8_t, wf[j]), __builtin_bit_cast(bf16x8_t, xf[p * NP + j]), acc[p],
          0, 0, 0);
  }
  f32x4_t own = acc[0];  // of A rows 4 g4 ..: part 4 g4 / RPT
#pragma unroll
  for (int p = 1; p < P; ++p)
    if (4 * g4 / RPT == p) own = acc[p];
  *reinterpret_cast<f32x4_t*>(&red[wave][l16][4 * g4]) = own;
  __syncthreads();
  if constexpr (SWIGLU) {
    const int row = tid >> 3, c = tid & 7;
    if (row >= M) return;
    float g = red[0][row][c], u = red[0][row][c + 8];
#pragma unroll
    for (int i = 1; i < kWaves; ++i) {
      g += red[i][row][c];
      u += red[i][row][c + 8];
    }
    g = bf16_to_f32(f32_to_bf16(g));
    u = bf16_to_f32(f32_to_bf16(u));
    y[row * y_stride + n0 + c] = f32_to_bf16(g / (1.0f + __expf(-g)) * u);
  } else {
    const int row = tid / RPT, c = tid % RPT;
    if (row >= M) return;
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < kWaves; ++i)
#pragma unroll
      for (int p = 0; p < P; ++p) s += red[i][row][p * RPT + c];
    y[row * y_stride + n0 + c] = f32_to_bf16(s);
  }
}

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

extern "C" int qmi_linear_small(const uint16_t* x, int64_t x_stride, const uint16_t* residual,
                                int64_t residual_stride, uint16_t* residual_out,
                                int64_t residual_out_stride, const uint16_t* norm_weight, float eps,
                                const uint16_t* w, int64_t w_stride, int64_t m, int64_t n, int64_t k,
                                int32_t activation, uint16_t* y, int64_t y_stride, void* stream) {
  if (m < 0 || n <= 0 || k <= 0 || activation < 0 || activation > 1) return QMI_E_BAD_SHAPE;
  if (m == 0) return QMI_OK;
  if (!x || !w || !y || (residual && (!norm_weight || !residual_out))) return QMI_E_NULL_POINTER;
  if (m > kMaxRows || n % 16 || n > (1 << 20)) return QMI_E_UNSUPPORTED;
  if (x_stride < k || x_stride % 8 || !al16(x) || w_stride < k || w_stride % 8 || !al16(w) ||
      y_stride < n || !al16(norm_weight) || !al16(residual) || !al16(residual_out) ||
      (reinterpret_cast<uintptr_t>(y) & 1u))
    return QMI_E_BAD_STRIDE;
  if (residual && (residual_stride < k || residual_stride % 8 || residual_out_stride < k ||
                   residual_out_stride % 8))
    return QMI_E_BAD_STRIDE;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  // Weight rows per workgroup: the most (8 + 8 for SwiGLU) that still give a
  // workgroup per CU.
  const int64_t cus = device_cu_count();
  const int rpt = activation ? 16 : n / 16 >= cus ? 16 : n / 8 >= cus ? 8 : 4;
  const dim3 grid((unsigned)(n / (activation ? 8 : rpt)));
#define QMI_LS(NS, RPT, SG, RW)                                                                    \
  hipLaunchKernelGGL((linear_small_kernel<NS, RPT, SG, RW>), grid, dim3(kThreads), 0, st, x,       \
                     x_stride, residual, residual_stride, residual_out, residual_out_stride,       \
                     norm_weight, eps, w, w_stride, y, y_stride, (int)m, (int)n)
#define QMI_LS_R(NS, RPT, SG)    \
  do {                           \
    if (!norm_weight)            \
      QMI_LS(NS, RPT, SG, 0);    \
    else if (m <= kWaves)        \
      QMI_LS(NS, RPT, SG, 1);    \
    else                         \
      QMI_LS(NS, RPT, SG, 2);    \
  } while (0)
#define QMI_LS_K(NS)               \
  case 256 * NS:                   \
    if (activation)                \
      QMI_LS_R(NS, 16, true);      \
    else if (rpt == 16)            \
      QMI_LS_R(NS, 16, false);     \
    else if (rpt == 8)             \
      QMI_LS_R(NS, 8, false);      \
    else                           \
      QMI_LS_R(NS, 4, false);      \
    break;
  switch (k) {
    QMI_LS_K(4)
    QMI_LS_K(8)
    QMI_LS_K(12)
    QMI_LS_K(16)
    default:
      return QMI_E_UNSUPPORTED;
  }
#undef QMI_LS_K
#undef QMI_LS_R
#undef QMI_LS
  QMI_RETURN_LAUNCH_STATUS();
}
