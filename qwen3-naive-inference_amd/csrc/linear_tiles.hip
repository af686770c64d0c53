// Prefill projections on bf16 MFMA (gfx950): y = x W^T for any number of rows.
//
// Reference semantics: the bf16 nn.Linear projections of a prefill step —
// qkv_proj / o_proj (qwen3_naive.py:427-428, :616, :638) and gate_up_proj,
// silu(gate) * up, down_proj (qwen3_naive.py:692-702) — with fp32
// accumulation and one bf16 rounding of each output.
//
//   * Workgroup = WM x WN waves = a tile of BM rows x BN weight rows.  K goes
//     through an NSTAGE-deep LDS ring in 64-element chunks (128-byte rows;
//     16-byte chunk c of row r sits at c ^ (r / 2 % 8), which spreads every
//     group of lanes that a ds_read_b128 serves together over all banks),
//     filled by direct global->LDS loads (inline asm, issued NSTAGE-1 chunks
//     ahead, one explicit s_waitcnt vmcnt per chunk).  Rows past M and weight
//     rows past N load the last row and are never stored.
//   * v_mfma_f32_16x16x32_bf16 with the weight rows as the A operand and the
//     x rows as B: a lane holds 4 consecutive output columns of one row.
//   * SwiGLU (packed [gate; up] weight): staged 16-row blocks alternate
//     between gate and up, so a wave holds both for the same columns and
//     writes silu(bf16(g)) * bf16(u) (the rounding points of a bf16 GEMM
//     followed by silu_mul) without the 2 I wide intermediate.
//   * Operands of the next k-step are read while one's products run, across
//     the chunk boundary too (one barrier per chunk).
//   * Workgroup -> tile: consecutive workgroups go to different XCDs, so each
//     XCD takes a contiguous run of a tile order that walks the rows of a few
//     column tiles first; its L2 then serves the re-reads.
//
// Hidden 1024, MLP 3072, weights from HBM, us for qkv / o / gate_up with SwiGLU /
// down (the library's product, with silu_mul for gate_up): 512 rows 9 / 9 / 12 /
// 12 (11 / 10 / 19 / 13), 2,048 rows 22 / 14 / 27 / 20 (21 / 16 / 36 / 21), 4,096
// rows 39 / 25 / 56 / 35 (30 / 22 / 70 / 31).
#include "qmi_common.h"

namespace {

using namespace qmi;

constexpr int kKC = 64;         // K elements per chunk
constexpr int kRowB = kKC * 2;  // bytes per staged row
constexpr int kXcds = 8;

typedef __attribute__((ext_vector_type(4))) unsigned int u4v_t;

__device__ __forceinline__ void lds_load16(const void* gbase, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
               : : "s"(lds), "v"(voff), "s"(gbase) : "memory", "m0");
}

__device__ __forceinline__ u4v_t ds_read16(uint32_t addr) {
  u4v_t r;
  asm volatile("ds_read_b128 %0, %1" : "=v"(r) : "v"(addr) : "memory");
  return r;
}

// Makes the values of f[] depend on the waits issued so far.
template <int N>
__device__ __forceinline__ void landed(u4v_t (&f)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) asm volatile("" : "+v"(f[i])::"memory");
}

template <int BM, int BN, int WM, int WN, int NSTAGE, bool SWIGLU>
__global__ __launch_bounds__(64 * WM * WN, WM * WN > 4 ? 1 : 2) void linear_tiles_kernel(
    const uint16_t* __restrict__ x, int64_t x_stride, const uint16_t* __restrict__ w,
    int64_t w_stride, uint16_t* __restrict__ y, int64_t y_stride, int M, int N, int K, int n_mt,
    int n_nt) {
  constexpr int NW = WM * WN;
  constexpr int SB = (BM + BN) * kRowB;
  constexpr int XL = BM / 8 / NW, WL = BN / 8 / NW, LPW = XL + WL;  // 1 KB loads per wave and chunk
  constexpr int TM = BM / WM / 16, TN = BN / WN / 16;               // 16 x 16 blocks per wave
  constexpr int OUT = SWIGLU ? BN / 2 : BN;
  static_assert(BM % (8 * NW) == 0 && BN % (8 * NW) == 0 && (!SWIGLU || TN % 2 == 0), "tile");
  __shared__ __attribute__((aligned(1024))) char lds[NSTAGE * SB];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Tile of this workgroup: XCD bid % 8 takes tiles [first, first + count).
  const int tiles = n_mt * n_nt;
  const int xcd = blockIdx.x % kXcds, q = tiles / kXcds, rem = tiles % kXcds;
  const int tile = xcd * q + min(xcd, rem) + blockIdx.x / kXcds;
  const int m0 = tile % n_mt * BM, n0 = tile / n_mt * OUT;
  const int nk = K / kKC;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) char*)lds;
  // Load j (8 staged rows): lane l fetches row 8 j + l / 8, physical chunk l % 8.
  uint32_t xoff[XL], woff[WL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int r = 8 * (i * NW + wave) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    xoff[i] = (uint32_t)(((int64_t)min(m0 + r, M - 1) * x_stride + c * 8) * 2);
  }
#pragma unroll
  for (int i = 0; i < WL; ++i) {
    const int r = 8 * (i * NW + wave) + (lane >> 3), c = (lane & 7) ^ ((r >> 1) & 7);
    int row;
    if constexpr (SWIGLU)
      row = ((r >> 4) & 1 ? N : 0) + min(n0 + (r >> 5) * 16 + (r & 15), N - 1);
    else
      row = min(n0 + r, N - 1);
    woff[i] = (uint32_t)(((int64_t)row * w_stride + c * 8) * 2);
  }
  auto issue = [&](int kc, int st) {
    const uint32_t sb = lds0 + st * SB;
    const char* xb = reinterpret_cast<const char*>(x) + (int64_t)kc * kRowB;
    const char* wb = reinterpret_cast<const char*>(w) + (int64_t)kc * kRowB;
#pragma unroll
    for (int i = 0; i < XL; ++i) lds_load16(xb, xoff[i], sb + (i * NW + wave) * 1024);
#pragma unroll
    for (int i = 0; i < WL; ++i) lds_load16(wb, woff[i], sb + BM * kRowB + (i * NW + wave) * 1024);
  };
  const int l16 = lane & 15, g4 = lane >> 4;
  const int wm = wave % WM, wn = wave / WM;
  // Operand of k-step ks: logical chunk 4 ks + g4 of row l16 of a block.
  const uint32_t rd = (uint32_t)(l16 * kRowB + 16 * (g4 ^ ((l16 >> 1) & 7)));
  const uint32_t x_rd = rd + wm * (BM / WM) * kRowB, w_rd = rd + (BM + wn * (BN / WN)) * kRowB;
  f32x4_t acc[TN][TM];
#pragma unroll
  for (int n = 0; n < TN; ++n)
#pragma unroll
    for (int m = 0; m < TM; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NSTAGE; ++i) issue(min(i, nk - 1), i);
  // Operands of two k-steps in registers: while the products of one run, the
  // reads of the next are in flight, across the chunk boundary too.
  u4v_t xf[2][TM], wf[2][TN];
  auto read = [&](int st, int ks) {
    const uint32_t base = lds0 + st * SB;
#pragma unroll
    for (int m = 0; m < TM; ++m) xf[ks][m] = ds_read16(base + ((x_rd + m * 16 * kRowB) ^ (ks * 64)));
#pragma unroll
    for (int n = 0; n < TN; ++n) wf[ks][n] = ds_read16(base + ((w_rd + n * 16 * kRowB) ^ (ks * 64)));
  };
  auto products = [&](int ks) {
#pragma unroll
    for (int n = 0; n < TN; ++n)
#pragma unroll
      for (int m = 0; m < TM; ++m)
        acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
            __builtin_bit_cast(bf16x8_t, wf[ks][n]), __builtin_bit_cast(bf16x8_t, xf[ks][m]),
            acc[n][m], 0, 0, 0);
  };
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"i"((NSTAGE - 1) * LPW) : "memory");
  read(0, 0);
  int st = 0;
  for (int k = 0; k < nk; ++k) {
    read(st, 1);
    asm volatile("s_waitcnt lgkmcnt(%0)" ::"i"(TM + TN) : "memory");
    landed(xf[0]);
    landed(wf[0]);
    __builtin_amdgcn_sched_barrier(0);
    products(0);
    __builtin_amdgcn_sched_barrier(0);
    // Chunk k + 1 has landed once only the later NSTAGE - 2 chunks' loads are
    // outstanding; every wave has its operands of chunk k, whose slot the next
    // loads overwrite.
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"i"((NSTAGE - 2) * LPW) : "memory");
    landed(xf[1]);
    landed(wf[1]);
    issue(min(k + NSTAGE, nk - 1), st);
    st = st == NSTAGE - 1 ? 0 : st + 1;
    read(st, 0);
    __builtin_amdgcn_sched_barrier(0);
    products(1);
    __builtin_amdgcn_sched_barrier(0);
  }
  // Drain the last loads (re-issues of the final chunk) and reads before exit.
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  landed(xf[0]);
  landed(wf[0]);
#pragma unroll
  for (int m = 0; m < TM; ++m) {
    const int row = m0 + wm * (BM / WM) + m * 16 + l16;
    if (row >= M) continue;
    uint16_t* yr = y + (int64_t)row * y_stride;
    if constexpr (SWIGLU) {
#pragma unroll
      for (int n = 0; n < TN / 2; ++n) {
        const int col = n0 + wn * (OUT / WN) + n * 16 + 4 * g4;
        if (col >= N) continue;
        float o[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float g = bf16_to_f32(f32_to_bf16(acc[2 * n][m][r]));
          const float u = bf16_to_f32(f32_to_bf16(acc[2 * n + 1][m][r]));
          o[r] = g / (1.0f + __expf(-g)) * u;
        }
        *reinterpret_cast<uint2*>(yr + col) =
            make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
      }
    } else {
#pragma unroll
      for (int n = 0; n < TN; ++n) {
        const int col = n0 + wn * (OUT / WN) + n * 16 + 4 * g4;
        if (col >= N) continue;
        *reinterpret_cast<uint2*>(yr + col) =
            make_uint2(pack_bf16x2(acc[n][m][0], acc[n][m][1]),
                       pack_bf16x2(acc[n][m][2], acc[n][m][3]));
      }
    }
  }
}

inline bool al16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool al8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }

template <int BM, int BN, int WM, int WN, int NSTAGE, bool SWIGLU>
void launch(const uint16_t* x, int64_t x_stride, const uint16_t* w, int64_t w_stride, uint16_t* y,
            int64_t y_stride, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  const int out = SWIGLU ? BN / 2 : BN;
  const int n_mt = (int)((m + BM - 1) / BM), n_nt = (int)((n + out - 1) / out);
  hipLaunchKernelGGL((linear_tiles_kernel<BM, BN, WM, WN, NSTAGE, SWIGLU>), dim3(n_mt * n_nt),
                     dim3(64 * WM * WN), 0, st, x, x_stride, w, w_stride, y, y_stride, (int)m,
                     (int)n, (int)k, n_mt, n_nt);
}

// Tile forms with the time one 64-element K chunk takes on an MI355X (ns, all
// CUs busy; weights from HBM, qkv / gate_up / o / down of hidden 1024): here a CU
// receives 35-60 GB/s however deep the ring is (loads alone reach 80-147 GB/s
// per CU; what keeps this kernel below that is not known), so a chunk's time
// follows its (BM + BN) rows and a form's merit is the bytes per CU that its tiles and
// their last, partly filled round give.  F(BM, BN, WM, WN, NSTAGE, ns).
#define QMI_LT_FORMS(F)        \
  F(64, 64, 2, 2, 4, 360)   \
  F(128, 64, 4, 2, 4, 500)  \
  F(128, 128, 4, 2, 4, 770) \
  F(128, 192, 4, 2, 3, 1000) \
  F(256, 128, 4, 2, 3, 1350) \
  F(256, 192, 4, 2, 2, 1670)

template <bool SWIGLU>
void dispatch(const uint16_t* x, int64_t x_stride, const uint16_t* w, int64_t w_stride, uint16_t* y,
              int64_t y_stride, int64_t m, int64_t n, int64_t k, hipStream_t st) {
  // The form whose rounds of tiles take least: 256 tiles at a time, the 64 x 64
  // form (64 KB of LDS, two workgroups per CU) 512 at 1.45 times one's time.
  const int64_t cus = device_cu_count();
  int best = 0, at = 0;
  int64_t least = INT64_MAX;
#define QMI_LT_COST(BM, BN, WM, WN, NS, T)                                             \
  {                                                                                       \
    const int64_t out = SWIGLU ? BN / 2 : BN;                                             \
    const int64_t tiles = ((m + BM - 1) / BM) * ((n + out - 1) / out);                    \
    const int64_t rounds = (tiles + cus - 1) / cus;                                       \
    const int64_t c = BM * BN == 4096 ? (rounds / 2 * 145 + rounds % 2 * 100) * T / 100   \
                                      : rounds * T;                                       \
    if (c < least) {                                                                      \
      least = c;                                                                          \
      best = at;                                                                          \
    }                                                                                     \
    ++at;                                                                                 \
  }
  QMI_LT_FORMS(QMI_LT_COST)
#undef QMI_LT_COST
  at = 0;
#define QMI_LT_RUN(BM, BN, WM, WN, NS, T)                                                    \
  if (best == at++)                                                                             \
    return launch<BM, BN, WM, WN, NS, SWIGLU>(x, x_stride, w, w_stride, y, y_stride, m, n, k, st);
  QMI_LT_FORMS(QMI_LT_RUN)
#undef QMI_LT_RUN
}

}  // namespace

extern "C" int qmi_linear_tiles(const uint16_t* x, int64_t x_stride, const uint16_t* w,
                                int64_t w_stride, int64_t m, int64_t n, int64_t k,
                                int32_t activation, uint16_t* y, int64_t y_stride, void* stream) {
  if (m < 0 || n <= 0 || k <= 0 || activation < 0 || activation > 1) return QMI_E_BAD_SHAPE;
  if (!x || !w) return QMI_E_NULL_POINTER;
  if (m > (1 << 20) || k % kKC || n % 16 || n > (1 << 20) || k > (1 << 20)) return QMI_E_UNSUPPORTED;
  if (x_stride < k || w_stride < k || x_stride % 8 || w_stride % 8 || !al16(x) || !al16(w))
    return QMI_E_BAD_STRIDE;
  // Load offsets are 32-bit byte offsets from the chunk base (2 n weight rows for SwiGLU).
  if (4 * n * w_stride >= (1LL << 32) || 2 * m * x_stride >= (1LL << 32)) return QMI_E_UNSUPPORTED;
  if (m == 0) return QMI_OK;
  if (!y) return QMI_E_NULL_POINTER;
  if (y_stride < n || y_stride % 4 || !al8(y)) return QMI_E_BAD_STRIDE;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if (activation)
    dispatch<true>(x, x_stride, w, w_stride, y, y_stride, m, n, k, st);
  else
    dispatch<false>(x, x_stride, w, w_stride, y, y_stride, m, n, k, st);
  QMI_RETURN_LAUNCH_STATUS();
}
