// cnn_internal.h -- launchers of the triage-CNN kernels (cnn.hip).
#pragma once
#include <hip/hip_runtime.h>

#include "internal.h"

namespace mdsm {
namespace cnn {

// number of K slices a split-K product with `splits` requested writes
int splits_used(int64_t K, int splits);
// C (+ slice * M * N) [m][n] = sum_k a[m*asr + k*asc] * b[k*bsr + n*bsc]
int gemm_dense(const uint16_t *a, int64_t asr, int64_t asc, const uint16_t *b, int64_t bsr,
               int64_t bsc, int64_t M, int64_t N, int64_t K, int splits, float *C, hipStream_t s);
// conv layer (0, 1, 2: 2->16->32->64) + bias + ReLU + 2x2 max pool, NHWC
int conv_pool(int layer, const uint16_t *x, int64_t B, int H, int W, const uint16_t *w, const float *bias,
              uint16_t *a, uint8_t *idx, hipStream_t s);
// input gradient of layer 1 or 2 (wf: scratch of the layer's weight count)
int conv_dx(int layer, const uint16_t *dz, int64_t B, int H, int W, const uint16_t *w, uint16_t *wf, float *dx,
            hipStream_t s);
// weight gradient of layer 1 or 2 (part: conv_dw_floats())
constexpr int DW_BLOCKS = 512;
int64_t conv_dw_floats();
int conv_dw(int layer, const uint16_t *dz, const uint16_t *x, int64_t B, int H, int W, float *part, float *dw,
            hipStream_t s);
// layer 0: weight and bias gradients (adjacent in dwb) from the pooled gradient
int conv1_dw(const float *da, const uint8_t *idx, const uint16_t *x, int64_t B, int H, int W, float *part,
             float *dwb, hipStream_t s);
// offsets of the parameter segments whose device order is not the canonical one
struct CanonicalLayout {
  int64_t w[3], fw1, n;
  int ci[3], co[3], fin, hid, pix, chan;
};
int to_canonical(const float *src, const CanonicalLayout &L, float *out, hipStream_t s);
int epilogue(const float *part, int splits, int64_t M, int64_t N, const float *bias, float *out_f32,
             const float *mask, int relu, uint16_t *out_bf16, hipStream_t s);
// C = 32 or 64; db: bias gradient
int pool_backward(const float *da, const uint8_t *idx, int64_t B, int H, int W, int C, uint16_t *dz, float *part,
                  float *db, hipStream_t s);
int column_sums(const uint16_t *x, int64_t rows, int C, float *part, int max_parts, float *out,
                hipStream_t s);
int softmax_ce(const float *logits, const int32_t *y, int B, uint16_t *dl, float *loss,
               hipStream_t s);
int adam(float *p, const float *g, float *m, float *v, uint16_t *pb, int64_t n, float lr, float b1,
         float b2, float eps, int step, float wd, hipStream_t s);
int to_bf16(const float *x, uint16_t *y, int64_t n, hipStream_t s);
int nchw2_to_nhwc(const uint16_t *x, int64_t B, int64_t HW, uint16_t *y, hipStream_t s);

}  // namespace cnn
}  // namespace mdsm
