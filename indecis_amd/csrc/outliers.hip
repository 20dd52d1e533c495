// outliers.hip — the LLM.int8() decomposition of linalg.MatMul8Outliers
// (linalg/int8.go:272-349) and the bias of siglip's linear.apply
// (internal/siglip/encoder.go:36-49), around the int8 GEMM:
//  * column maxima of |A| (order-free, so an atomic max of the float bits:
//    |x| is never negative);
//  * the chosen input channels zeroed in a copy of A before quantizeA;
//  * after the GEMM, per output element, the chosen channels' products
//    a[i][j] * f32(q[col][j] * sb[col]) added one by one in the chosen
//    order (product and sum rounded separately, as gc computes
//    ci[col] += x * wv for amd64 at GOAMD64 v1/v2, which has no scalar
//    FMA), then the bias (AddTo, vec_scalar.go:97-101).
// The channel choice itself (a float32 mean in channel order, a partial
// selection of the 32 largest) runs on the host over the k maxima.
#include "ixh_device.h"
#include "ixh_internal.h"

namespace ixh {

namespace {

// Rows of a workgroup of the column-max kernel, every load of a thread in
// flight at once: 784 rows of 3,072 columns 100.7 -> 5.4 us (before: 256 rows one load
// at a time, 48 workgroups).
constexpr int kColRows = 16;

__global__ __launch_bounds__(256) void colmax_kernel(const float *a, int ld, int m, int k,
                                                     unsigned *out) {
  const int j = blockIdx.x * 256 + threadIdx.x;
  if (j >= k) return;
  const int r0 = blockIdx.y * kColRows;
  float v[kColRows], mx = 0.f;
#pragma unroll
  for (int i = 0; i < kColRows; i++) v[i] = a[(size_t)min(r0 + i, m - 1) * ld + j];
#pragma unroll
  for (int i = 0; i < kColRows; i++) mx = fmax32(mx, fabsf(v[i]));
  atomicMax(out + j, __float_as_uint(mx));
}

__global__ __launch_bounds__(256) void zero_cols_kernel(float *a, int ld, int m, const int *cols,
                                                        int ncols) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long)m * ncols) return;
  const int i = (int)(e / ncols), t = (int)(e % ncols);
  a[(size_t)i * ld + cols[t]] = 0.f;
}

// w[t][col] = f32(q[col][cols[t]]) * sb[col]: the chosen channels' dequantised
// weight rows (int8.go:336-340), from the resident int8 rows.
__global__ __launch_bounds__(256) void outlier_weights_kernel(const int8_t *q, int ldq, const float *sb, const int *cols,
                                                              int n, float *w) {
  const int col = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
  if (col < n) w[(size_t)t * n + col] = (float)q[(size_t)col * ldq + cols[t]] * sb[col];
}

__global__ __launch_bounds__(256) void outlier_epilogue_kernel(float *c, int ldc, int m, int n,
                                                               const float *a, int lda,
                                                               const int *cols, int ncols,
                                                               const float *w, const float *bias) {
  const long e = (long)blockIdx.x * 256 + threadIdx.x;
  if (e >= (long)m * n) return;
  const int i = (int)(e / n), col = (int)(e % n);
  float v = c[(size_t)i * ldc + col];
  const float *ar = a + (size_t)i * lda;
  for (int t = 0; t < ncols; t++) {
    const float p = ar[cols[t]] * w[(size_t)t * n + col];
    v = v + p;
  }
  if (bias) v = v + bias[col];
  c[(size_t)i * ldc + col] = v;
}

}  // namespace

void launch_colmax(const float *a, int ld, int m, int k, unsigned *out, hipStream_t s) {
  if (m <= 0 || k <= 0) return;
  const dim3 grid((k + 255) / 256, (m + kColRows - 1) / kColRows);
  colmax_kernel<<<grid, 256, 0, s>>>(a, ld, m, k, out);
}

void launch_outlier_weights(const int8_t *q, int ldq, const float *sb, const int *cols, int ncols, int n, float *w,
                            hipStream_t s) {
  if (ncols <= 0 || n <= 0) return;
  outlier_weights_kernel<<<dim3((n + 255) / 256, ncols), 256, 0, s>>>(q, ldq, sb, cols, n, w);
}

void launch_zero_cols(float *a, int ld, int m, const int *cols, int ncols, hipStream_t s) {
  const long total = (long)m * ncols;
  if (total <= 0) return;
  zero_cols_kernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(a, ld, m, cols, ncols);
}

void launch_outlier_epilogue(float *c, int ldc, int m, int n, const float *a, int lda, const int *cols,
                             int ncols, const float *w, const float *bias, hipStream_t s) {
  const long total = (long)m * n;
  if (total <= 0) return;
  outlier_epilogue_kernel<<<(unsigned)((total + 255) / 256), 256, 0, s>>>(c, ldc, m, n, a, lda, cols,
                                                                          ncols, w, bias);
}

}  // namespace ixh
