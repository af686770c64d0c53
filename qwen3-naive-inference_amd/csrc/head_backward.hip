// Gradient of the lm_head's input on bf16 MFMA (gfx950): dX = dY W, dY [M, V]
// gradients of the logits, W [V, N] the head's weight, fp32 accumulation and one
// bf16 rounding of each element.
//
// Reference semantics: the backward of lm_head (qwen3_naive.py:840) in the
// GRPO training step (qwen3_grpo_train.py:261-286).
//
// The sum runs over the vocabulary (151,936) and the result is small: at 778
// rows x 1,024 the library's product works on 28 tiles and leaves most of the
// chip idle (594 us, 410 TFLOP/s; here 313 us; at 256 rows 447 / 109, 2,048 946 /
// 570, 5,120 1,695 / 1,381, 1.15 PFLOP/s, near the rate the operands' LDS reads
// and the barriers of two 64 KB stages allow).  Here the vocabulary is split: each of about
// one workgroup per CU sums one range of it for one 256 (n) x MT (m) tile into
// fp32 partials, and a second kernel adds a tile's partials in a fixed order.
//   * Workgroups of one range are on one XCD (8 XCDs, round robin by index), so
//     W and dY are read from HBM once and shared through its L2.
//   * 8 waves, 64-deep chunks of the vocabulary, two LDS stages filled by direct
//     global->LDS loads a chunk ahead (inline asm, one vmcnt wait and one
//     barrier per chunk).
//   * The product is taken transposed, dX^T = W^T dY^T: the A operand W^T comes
//     from the row-major W chunk by gfx950's LDS transpose read
//     (ds_read_b64_tr_b16), and the B operand reads each dY row's matching 2 x 8
//     bytes, so neither matrix is transposed in memory and a lane holds 4
//     consecutive n of one row.
//   * LDS: W rows of 512 bytes with the 16-byte chunk XORed by 2 (row % 8) (the 8
//     rows of a transpose read's 32 lanes then cover all banks), dY rows of 128
//     bytes with the chunk XORed by (row / 2) % 8.
#include <algorithm>

#include "qmi_common.h"

namespace {

using namespace qmi;

constexpr int kKC = 64;    // vocabulary entries per chunk
constexpr int kNT = 256;   // n per tile
constexpr int kWaves = 8;
constexpr int kWRowB = kNT * 2;
constexpr int kYRowB = kKC * 2;
typedef __attribute__((ext_vector_type(4))) short v4s_t;
typedef __attribute__((ext_vector_type(8))) short v8s_t;

__device__ __forceinline__ void lds_load16(const void* gbase, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               : : "s"(lds), "v"(voff), "s"(gbase) : "memory", "m0");
}

template <int MT>
__global__ __launch_bounds__(kWaves * 64) void head_dx_parts(
    const uint16_t* __restrict__ dy, int64_t dy_stride, const uint16_t* __restrict__ w, int64_t w_stride,
    float* __restrict__ part, int M, int N, int n_chunks, int n_mt, int n_nt, int S) {
  constexpr int WM = MT / 4;       // rows per wave: 4 wave columns along m, 2 wave rows along n
  constexpr int RB = WM / 16;      // 16-row blocks per wave
  constexpr int DB = kNT / 2 / 16; // 16-column blocks per wave
  constexpr int W_BYTES = kKC * kWRowB, STAGE = W_BYTES + MT * kYRowB;
  constexpr int WL = W_BYTES / 1024 / kWaves, YL = MT * kYRowB / 1024 / kWaves;
  __shared__ __attribute__((aligned(16))) unsigned char lds[2 * STAGE];
  const int lane = threadIdx.x & 63, l16 = lane & 15, g4 = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wn = wave & 1, wm = wave >> 1;
  // Range-major order within an XCD.
  const int id = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  const int tiles = n_mt * n_nt;
  if (id >= tiles * S) return;
  const int s = id / tiles, tile = id % tiles;
  const int n0 = (tile % n_nt) * kNT, m0 = (tile / n_nt) * MT;
  const int c0 = (int)((int64_t)s * n_chunks / S), c1 = (int)((int64_t)(s + 1) * n_chunks / S);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)lds;
  // Wave-load j of W: rows 2 (WL wave + j) + lane / 32, chunk lane % 32; columns
  // past N repeat the last chunk, rows past M the last row, and are never stored.
  uint32_t woff[WL], yoff[YL];
#pragma unroll
  for (int j = 0; j < WL; ++j) {
    const int r = 2 * (WL * wave + j) + (lane >> 5);
    const int c = (lane & 31) ^ ((r & 7) << 1);
    woff[j] = (uint32_t)((r * w_stride + min(n0 + 8 * c, N - 8)) * 2);
  }
#pragma unroll
  for (int j = 0; j < YL; ++j) {
    const int r = 8 * (YL * wave + j) + (lane >> 3);
    const int c = (lane & 7) ^ ((r >> 1) & 7);
    yoff[j] = (uint32_t)(8 * c * 2);
    yoff[j] += (uint32_t)((uint64_t)(min(m0 + r, M - 1) - m0) * dy_stride * 2);
  }
  const char* yb = reinterpret_cast<const char*>(dy + (int64_t)m0 * dy_stride);
  auto issue = [&](int chunk, int st) __attribute__((always_inline)) {
    const uint32_t sb = lds0 + st * STAGE;
    const char* wk = reinterpret_cast<const char*>(w + (int64_t)chunk * kKC * w_stride);
    const char* yk = yb + (int64_t)chunk * kYRowB;
#pragma unroll
    for (int j = 0; j < WL; ++j) lds_load16(wk, woff[j], sb + (WL * wave + j) * 1024);
#pragma unroll
    for (int j = 0; j < YL; ++j) lds_load16(yk, yoff[j], sb + W_BYTES + (YL * wave + j) * 1024);
  };
  f32x4_t acc[DB][RB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
#pragma unroll
    for (int r = 0; r < RB; ++r) acc[d][r] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  // Transpose reads: row 32 ks + 4 g4 + l16 / 4 (then 16 further), 8-byte piece
  // l16 % 4 of column block d; B operand: row WM wm + 16 r + l16, entries 32 ks +
  // 4 g4 (then 16 further).
  const int trow = 4 * g4 + (l16 >> 2), tx = (l16 & 3) >> 1;
  int a_off[DB];
#pragma unroll
  for (int d = 0; d < DB; ++d)
    a_off[d] = trow * kWRowB + 16 * ((2 * (DB * wn + d) + tx) ^ ((trow & 7) << 1)) + 8 * (l16 & 1);
  int b_off[4];  // 16-byte chunks 4 ks + g4 / 2 and 4 ks + 2 + g4 / 2
#pragma unroll
  for (int k = 0; k < 4; ++k)
    b_off[k] = W_BYTES + (WM * wm + l16) * kYRowB + 16 * ((2 * k + (g4 >> 1)) ^ (l16 >> 1)) + 8 * (g4 & 1);
  typedef __attribute__((address_space(3))) v4s_t lds_v4s;
  issue(c0, 0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  for (int c = c0; c < c1; ++c) {
    const int st = (c - c0) & 1;
    issue(min(c + 1, c1 - 1), st ^ 1);
    unsigned char* base = lds + st * STAGE;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      bf16x8_t b[RB];
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        const v4s_t lo = *reinterpret_cast<const v4s_t*>(base + b_off[2 * ks] + r * 16 * kYRowB);
        const v4s_t hi = *reinterpret_cast<const v4s_t*>(base + b_off[2 * ks + 1] + r * 16 * kYRowB);
        b[r] = __builtin_bit_cast(bf16x8_t, v8s_t{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
      }
#pragma unroll
      for (int d = 0; d < DB; ++d) {
        unsigned char* p = base + a_off[d] + 32 * ks * kWRowB;
        const v4s_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)p);
        const v4s_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4s*)(p + 16 * kWRowB));
        const bf16x8_t a = __builtin_bit_cast(bf16x8_t, v8s_t{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w});
#pragma unroll
        for (int r = 0; r < RB; ++r) acc[d][r] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b[r], acc[d][r], 0, 0, 0);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  }
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int row = m0 + WM * wm + 16 * r + l16;
    if (row >= M) continue;
    float* dst = part + ((int64_t)s * M + row) * N;
#pragma unroll
    for (int d = 0; d < DB; ++d) {
      const int col = n0 + 16 * (DB * wn + d) + 4 * g4;
      if (col < N) *reinterpret_cast<f32x4_t*>(dst + col) = acc[d][r];
    }
  }
}

// dx[i] = bf16(sum_s part[s][i]), 8 elements per lane.
__global__ __launch_bounds__(256) void head_dx_sum(const float* __restrict__ part, int64_t total, int S,
                                                   uint16_t* __restrict__ dx, int64_t dx_stride, int N) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8;
  if (i >= total) return;
  f32x4_t a = *reinterpret_cast<const f32x4_t*>(part + i), b = *reinterpret_cast<const f32x4_t*>(part + i + 4);
#pragma unroll 4
  for (int s = 1; s < S; ++s) {
    a += *reinterpret_cast<const f32x4_t*>(part + s * total + i);
    b += *reinterpret_cast<const f32x4_t*>(part + s * total + i + 4);
  }
  const int64_t row = i / N;
  *reinterpret_cast<uint4*>(dx + row * dx_stride + (i - row * N)) = make_uint4(
      pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]), pack_bf16x2(b[2], b[3]));
}

struct Plan {
  int mt, n_mt, n_nt, S;
};

// About one workgroup per CU, each with at least 8 chunks.  Tiles of 256 rows:
// with 128 a CU would need 47 bytes per clock from L2 for the product at full
// rate and reaches 690-730 TFLOP/s (778 rows 352 us against 313), which only
// pays up to 128 rows (85 us; 256-row tiles would multiply as much padding).
Plan plan(int64_t M, int64_t N, int64_t n_chunks) {
  Plan p;
  p.mt = M <= 128 ? 128 : 256;
  p.n_mt = (int)((M + p.mt - 1) / p.mt);
  p.n_nt = (int)((N + kNT - 1) / kNT);
  p.S = (int)std::max<int64_t>(1, std::min<int64_t>(device_cu_count() / std::max(1, p.n_mt * p.n_nt), n_chunks / 8));
  return p;
}

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

extern "C" int64_t qmi_head_backward_workspace_bytes(int64_t n_rows, int64_t hidden, int64_t vocab) {
  if (n_rows <= 0 || hidden <= 0 || vocab < kKC) return 0;
  return plan(n_rows, hidden, vocab / kKC).S * n_rows * hidden * 4;
}

extern "C" int qmi_head_backward_input(const uint16_t* dy, int64_t dy_stride, const uint16_t* w, int64_t w_stride,
                                       int64_t n_rows, int64_t hidden, int64_t vocab, uint16_t* dx, int64_t dx_stride,
                                       float* workspace, int64_t workspace_bytes, void* stream) {
  if (n_rows < 0 || hidden <= 0 || vocab <= 0) return QMI_E_BAD_SHAPE;
  if (n_rows == 0) return QMI_OK;
  if (!dy || !w || !dx || !workspace) return QMI_E_NULL_POINTER;
  // 32-bit lane offsets: 64 rows of W, 256 rows of dY.
  if (vocab % kKC || hidden % 8 || hidden > 65536 || n_rows > 65536 || vocab / kKC > 0x7fffff ||
      w_stride * 128 > 0x7fffffffLL || dy_stride * 512 > 0xffffffffLL)
    return QMI_E_UNSUPPORTED;
  if (dy_stride % 8 || w_stride % 8 || dx_stride % 8 || dy_stride < vocab || w_stride < hidden || dx_stride < hidden ||
      !al16(dy) || !al16(w) || !al16(dx) || !al16(workspace))
    return QMI_E_BAD_STRIDE;
  const int n_chunks = (int)(vocab / kKC);
  const Plan p = plan(n_rows, hidden, n_chunks);
  if (workspace_bytes < p.S * n_rows * hidden * 4) return QMI_E_WORKSPACE_TOO_SMALL;
  const int64_t grid = ((int64_t)p.n_mt * p.n_nt * p.S + 7) / 8 * 8;
  if (grid > 0x7fffffffLL) return QMI_E_UNSUPPORTED;
  const hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kWaves * 64), 0, st, dy, dy_stride, w, w_stride, workspace,
                       (int)n_rows, (int)hidden, n_chunks, p.n_mt, p.n_nt, p.S);
  };
  p.mt == 128 ? launch(head_dx_parts<128>) : launch(head_dx_parts<256>);
  const int64_t total = n_rows * hidden;
  hipLaunchKernelGGL(head_dx_sum, dim3((unsigned)((total / 8 + 255) / 256)), dim3(256), 0, st, workspace, total, p.S,
                     dx, dx_stride, (int)hidden);
  QMI_RETURN_LAUNCH_STATUS();
}
