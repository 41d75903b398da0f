// What spectral() does to eigenvectors before they leave the device: a sign for
// each (the entry of largest magnitude positive), the choice of columns and their
// scaling by the square roots of the eigenvalues
// (snapatac2-python/python/snapatac2/tools/_embedding.py:284-288 scales and selects;
// the signs are this package's convention).
//
// On the host these were five passes over the n x k matrix in numpy. Here they are
// one read to find the signs and one read and write, so that the matrix crosses to
// the host once, finished. With 150,000 x 30 (36 MB) spectral() over sampled cells took
// 63 ms with the numpy passes and takes 22 ms with these two kernels.
#include <algorithm>

#include "common.h"

namespace snapgpu {
namespace embed {

constexpr int kRows = 256;  // rows per block of the search, 8 at a time (3,001 x 30: 43 us with 1024, below 22 so)

// A column's leading entry so far: the magnitude as an integer (the bits of |U|, in
// the same order; every NaN above infinity and alike) and the row.
struct Best {
  uint64_t mag;
  int64_t row;
};

__device__ __forceinline__ uint64_t magnitude(double v) {
  return min((uint64_t)__double_as_longlong(v) & 0x7fffffffffffffffull, 0x7ff0000000000001ull);
}

// The order of numpy's argmax of |U|: NaN first of all, then the larger, then the first.
__device__ __forceinline__ void take(Best& best, uint64_t mag, int64_t row) {
  const bool ahead = mag > best.mag || (mag == best.mag && row < best.row);
  best.mag = ahead ? mag : best.mag;
  best.row = ahead ? row : best.row;
}

// Block (slice, column group): the leading entry of each of 32 columns over kRows rows.
__global__ void __launch_bounds__(256) lead_kernel(const double* __restrict__ U, int64_t ldu, int64_t n, int kc,
                                                   const int32_t* __restrict__ cols, Best* __restrict__ part) {
  __shared__ Best red[8][32];
  const int cl = threadIdx.x & 31, rg = threadIdx.x >> 5;
  const int c = blockIdx.y * 32 + cl;
  const int64_t r0 = (int64_t)blockIdx.x * kRows, r1 = min(n, r0 + kRows);
  Best best{0, INT64_MAX};
  if (c < kc) {
    const int col = cols[c];
    for (int64_t i = r0 + rg; i < r1; i += 8) take(best, magnitude(U[i * ldu + col]), i);
  }
  red[rg][cl] = best;
  __syncthreads();
  if (rg != 0 || c >= kc) return;
  for (int g = 1; g < 8; ++g) take(best, red[g][cl].mag, red[g][cl].row);
  part[(int64_t)blockIdx.x * kc + c] = best;
}

// sign[c] = sign of the column's leading entry (1 for zero, NaN for NaN)
__global__ void __launch_bounds__(64) sign_kernel(const Best* __restrict__ part, int64_t slices,
                                                  const double* __restrict__ U, int64_t ldu, int kc,
                                                  const int32_t* __restrict__ cols, double* __restrict__ sign) {
  __shared__ Best red[64];
  const int c = blockIdx.x;
  Best best{0, INT64_MAX};
  for (int64_t s = threadIdx.x; s < slices; s += 64) take(best, part[s * kc + c].mag, part[s * kc + c].row);
  red[threadIdx.x] = best;
  __syncthreads();
  if (threadIdx.x != 0) return;
  for (int t = 1; t < 64; ++t) take(best, red[t].mag, red[t].row);
  const double v = U[best.row * ldu + cols[c]];
  sign[c] = v > 0.0 ? 1.0 : v < 0.0 ? -1.0 : v == 0.0 ? 1.0 : v;
}

// out[i][c] = (U[i][cols[c]] * sign[c]) * scale[c]
__global__ void finish_kernel(const double* __restrict__ U, int64_t ldu, int64_t n, int kc,
                              const int32_t* __restrict__ cols, const double* __restrict__ sign,
                              const double* __restrict__ scale, double* __restrict__ out) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n * kc) return;
  const int64_t i = t / kc;
  const int c = (int)(t - i * kc);
  double v = U[i * ldu + cols[c]] * sign[c];
  if (scale) v *= scale[c];
  out[t] = v;
}

}  // namespace embed
}  // namespace snapgpu

using namespace snapgpu;
using namespace snapgpu::embed;

extern "C" {

int64_t snapgpu_embed_workspace_bytes(int64_t n, int32_t kc) {
  if (n <= 0 || kc <= 0) return 256;
  return ceil_div(n, kRows) * kc * (int64_t)sizeof(Best) + (int64_t)kc * 8 + 512;
}

int snapgpu_embed_finish(const double* d_U, int64_t ldu, int64_t n, const int32_t* d_cols, int32_t kc,
                         const double* d_scale, double* d_out, void* d_ws, int64_t ws_bytes, void* stream) {
  clear_error();
  SG_ARG(n >= 0 && kc >= 0 && ldu >= 1, "bad shape");
  if (n == 0 || kc == 0) return SNAPGPU_OK;
  SG_ARG(d_U && d_cols && d_out && d_ws, "null pointer");
  SG_ARG(ws_bytes >= snapgpu_embed_workspace_bytes(n, kc), "workspace too small");
  SG_ARG(ceil_div(n, kRows) < (1ll << 31) && ceil_div(n * kc, 256) < (1ll << 31), "too many values for one launch");
  hipStream_t st = as_stream(stream);
  char* q = (char*)(((uintptr_t)d_ws + 255) & ~(uintptr_t)255);
  const int64_t slices = ceil_div(n, kRows);
  double* sign = reinterpret_cast<double*>(q);
  Best* part = reinterpret_cast<Best*>(q + (kc * 8 + 255) / 256 * 256);
  lead_kernel<<<dim3((unsigned)slices, (unsigned)ceil_div(kc, 32)), 256, 0, st>>>(d_U, ldu, n, kc, d_cols, part);
  sign_kernel<<<(unsigned)kc, 64, 0, st>>>(part, slices, d_U, ldu, kc, d_cols, sign);
  finish_kernel<<<(unsigned)ceil_div(n * kc, 256), 256, 0, st>>>(d_U, ldu, n, kc, d_cols, sign, d_scale, d_out);
  SG_LAUNCH_CHECK();
  return SNAPGPU_OK;
}

}  // extern "C"
