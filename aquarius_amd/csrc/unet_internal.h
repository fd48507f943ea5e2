// unet_internal.h -- kernels of the warm-start U-Net (unet_kernels.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace aqu {

struct Vol {
  int B, D, H, W;  // batch and spatial extent; voxel id ((b*D + d)*H + h)*W + w
};

void conv3_forward(int cin, int cout, const Vol& v, const __bf16* X, int xs, int xo, const __bf16* Wk,
                   const float* bias, __bf16* Y, int ys, int yo, hipStream_t s);
void conv3_dgrad(int cin, int cout, const Vol& v, const __bf16* dY, const __bf16* Wt, float* dX, hipStream_t s);
void conv3_dgrad_relu(int c, const Vol& v, const __bf16* dY, const __bf16* Wt, const __bf16* M, int ms, int mo,
                      __bf16* dYpre, hipStream_t s);
void conv3_dgrad_concat(int cin, int cout, const Vol& v, const __bf16* dY, const __bf16* Wt, float* skip,
                        const __bf16* M, __bf16* up, hipStream_t s);
void conv3_wgrad(int cin, int cout, const Vol& v, const __bf16* dY, const __bf16* X, int xs, int xo,
                 float* part, float* bpart, int nsplit, float* dW, float* db, hipStream_t s);
void skip_bwd(const Vol& v, int C, const __bf16* Y, int ys, const float* dS, const float* dP, __bf16* dYpre,
              hipStream_t s);
void avgpool(const Vol& vo, int C, const __bf16* X, int xs, int xo, __bf16* Y, hipStream_t s);
void upsample(const Vol& vi, int C, const __bf16* X, __bf16* Y, int ys, int yo, hipStream_t s);
void head_fwd(long long V, int C, const __bf16* X, const float* w, const float* b, float* y, hipStream_t s);
void head_bwd(long long V, const __bf16* X, const float* w, const float* dy, __bf16* dYpre, float* part,
              int nblk, float* dwb, hipStream_t s);
void masked_mse(long long V, const float* y, const float* t, const float* m, double* part, int nblk,
                double* out, float* dy, hipStream_t s);
void adam(long long n, float* w, const float* g, float* m, float* v, float lr_t, float b1, float b2,
          float eps, hipStream_t s);
void pack_weights(int cin, int cout, const float* W, __bf16* Wk, __bf16* Wt, hipStream_t s);
void zero_f32(float* p, long long n, hipStream_t s);
void mfma_probe(const float* A, const float* B, float* D, hipStream_t s);

}  // namespace aqu
