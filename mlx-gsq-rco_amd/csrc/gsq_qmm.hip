// QMM dispatch by type; the kernels are in gsq_qmm_impl.h, instantiated per type in
// gsq_qmm_<type>.hip.
#include <cstdio>
#include <cstdlib>

#include "gsq_common.h"

namespace gsq {

// GSQ_QMM_TUNING="mf,min_cols,0,small_max_m,small_waves,small_nb,small_min_cols,order" (a prefix may
// be given; 0 keeps a field's default; the third field has no meaning) overrides the launch plans,
// read once at library load, for measuring plans without a rebuild.
static QmmTuning qmm_tuning_from_env() {
  QmmTuning t = {0, 0, 0, 0, 0, 0, 0};
  if (const char* s = std::getenv("GSQ_QMM_TUNING")) {
    int v[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    std::sscanf(s, "%d,%d,%d,%d,%d,%d,%d,%d", &v[0], &v[1], &v[2], &v[3], &v[4], &v[5], &v[6], &v[7]);
    t = {v[0], v[1], v[3], v[4], v[5], v[6], v[7]};
  }
  return t;
}
QmmTuning g_qmm_tuning = qmm_tuning_from_env();

hipError_t launch_qmm_q2_k(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_q4_k(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_q6_k(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_iq4_xs(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_iq3_s(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_iq3_xxs(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_iq2_xxs(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_iq2_xs(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_iq2_s(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_iq1_s(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);
hipError_t launch_qmm_iq1_m(const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M,
    int64_t N, int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s);

// Activations as the MFMA kernels read them: fp16, 16-byte aligned, rounded as the generic kernel
// rounds them while staging its tile. Eight values per thread, in whole 16-byte pieces when x is
// aligned to them. Bound by memory: one read and one write of x (512 x 17408 bf16, 36 MB: ~10 us
// beside a product of ~160).
template <int DT, bool VEC>
__global__ void __launch_bounds__(256) qmm_stage_x_kernel(const void* __restrict__ x, uint4* __restrict__ out,
                                                          int64_t n8) {
  typedef _Float16 half8 __attribute__((ext_vector_type(8)));
  constexpr int NV = DT == 0 ? 2 : 1;  // 16-byte pieces of eight values
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256) {
    uint32_t w[4 * NV];
    if constexpr (VEC) {
#pragma unroll
      for (int v = 0; v < NV; ++v) {
        const uint4 q = static_cast<const uint4*>(x)[NV * i + v];
        w[4 * v] = q.x; w[4 * v + 1] = q.y; w[4 * v + 2] = q.z; w[4 * v + 3] = q.w;
      }
    } else if constexpr (DT == 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) w[j] = static_cast<const uint32_t*>(x)[8 * i + j];
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint16_t* p = static_cast<const uint16_t*>(x) + 8 * i + 2 * j;
        w[j] = (uint32_t)p[0] | ((uint32_t)p[1] << 16);
      }
    }
    half8 h;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (DT == 0) h[j] = (_Float16)__builtin_bit_cast(float, w[j]);
      else if constexpr (DT == 1) h[j] = __builtin_bit_cast(_Float16, (uint16_t)(w[j >> 1] >> (16 * (j & 1))));
      else h[j] = (_Float16)__builtin_bit_cast(float, j & 1 ? w[j >> 1] & 0xFFFF0000u : w[j >> 1] << 16);
    }
    out[i] = __builtin_bit_cast(uint4, h);
  }
}

static hipError_t launch_stage_x(const void* x, int xdt, int64_t n, void* out, hipStream_t s) {
  const int64_t n8 = n / 8;  // rows are multiples of 256 values
  const dim3 grid((unsigned)(n8 + 255 < 256 * 8192 ? (n8 + 255) / 256 : 8192)), block(256);
  const bool vec = (reinterpret_cast<uintptr_t>(x) & 15) == 0;
  uint4* o = static_cast<uint4*>(out);
  if (xdt == 0 && vec) hipLaunchKernelGGL((qmm_stage_x_kernel<0, true>), grid, block, 0, s, x, o, n8);
  else if (xdt == 0) hipLaunchKernelGGL((qmm_stage_x_kernel<0, false>), grid, block, 0, s, x, o, n8);
  else if (xdt == 1) hipLaunchKernelGGL((qmm_stage_x_kernel<1, false>), grid, block, 0, s, x, o, n8);
  else if (vec) hipLaunchKernelGGL((qmm_stage_x_kernel<2, true>), grid, block, 0, s, x, o, n8);
  else hipLaunchKernelGGL((qmm_stage_x_kernel<2, false>), grid, block, 0, s, x, o, n8);
  return hipGetLastError();
}

static hipError_t launch_qmm_type(int qt, const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M, int64_t N,
                      int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s) {
  switch (qt) {
    case Q2_K: return launch_qmm_q2_k(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case Q4_K: return launch_qmm_q4_k(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case Q6_K: return launch_qmm_q6_k(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case IQ4_XS: return launch_qmm_iq4_xs(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case IQ3_S: return launch_qmm_iq3_s(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case IQ3_XXS: return launch_qmm_iq3_xxs(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case IQ2_XXS: return launch_qmm_iq2_xxs(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case IQ2_XS: return launch_qmm_iq2_xs(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case IQ2_S: return launch_qmm_iq2_s(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case IQ1_S: return launch_qmm_iq1_s(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    case IQ1_M: return launch_qmm_iq1_m(packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
    default: return hipErrorInvalidValue;
  }
}

// fp32 / bf16 activations, and fp16 ones that are not 16-byte aligned, are staged as fp16 in the
// workspace (as many rows at a time as it holds) for the MFMA kernels: 512 bf16 rows of a Q4_K
// 5120 x 17408 product 2409 -> 170 us against the generic kernel, which stays for workspaces
// without a staging area (the allocation-free entry point) and rows wider than it.
hipError_t launch_qmm(int qt, const uint8_t* packed, const void* x, int xdt, void* y, int ydt, int64_t M, int64_t N,
                      int K, const DevTables& tb, int num_cus, const QmmWorkspace& ws, hipStream_t s) {
  const int64_t cap = ws.xs ? ws.xs_bytes / (2ll * K) : 0;  // rows the staging area holds
  if (qmm_reads_x(x, xdt) || cap < 1) return launch_qmm_type(qt, packed, x, xdt, y, ydt, M, N, K, tb, num_cus, ws, s);
  // pieces of equal height, in whole 256-row tiles where they fit
  const int64_t pieces = (M + cap - 1) / cap;
  int64_t step = (M + pieces - 1) / pieces;
  if ((step + 255) / 256 * 256 <= cap) step = (step + 255) / 256 * 256;
  const int64_t xe = xdt == 0 ? 4 : 2, ye = ydt == 0 ? 4 : 2;
  for (int64_t r = 0; r < M; r += step) {
    const int64_t rows = M - r < step ? M - r : step;
    hipError_t e = launch_stage_x(static_cast<const uint8_t*>(x) + r * K * xe, xdt, rows * K, ws.xs, s);
    if (e == hipSuccess)
      e = launch_qmm_type(qt, packed, ws.xs, 1, static_cast<uint8_t*>(y) + r * N * ye, ydt, rows, N, K, tb, num_cus, ws, s);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace gsq
