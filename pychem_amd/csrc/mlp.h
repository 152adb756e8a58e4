// mlp.h -- internal launchers of mlp.hip (learned-guess MLP, FP32).
#pragma once
#include <hip/hip_runtime.h>

#define MLP_MAX_LAYERS 8
#define MLP_MAX_TENSORS (2 * MLP_MAX_LAYERS)

int mlp_linear_fwd(const float* X, const float* W, const float* b, float* Z, float* A, int B, int I, int O, int act,
                   hipStream_t st);
int mlp_linear_bwd(const float* X, const float* W, const float* A, const float* dA, float* dZ, float* dX, float* dW,
                   float* db, int B, int I, int O, int act, hipStream_t st);
// whole networks (hidden layers tanh, last layer linear); mlp_forward returns
// -2 when a layer is too wide for the one-launch form and an A[l] is NULL
int mlp_forward(int nlayer, const int* dims, const float* X, const float* const* W, const float* const* b,
                float* const* A, int B, hipStream_t st);
int mlp_backward(int nlayer, const int* dims, const float* X, const float* const* A, const float* const* W,
                 const float* dY, float* const* dZ, float* const* dW, float* const* db, int B, hipStream_t st);
int mlp_mse(const float* Y, const float* T, const float* mask, float* dY, float* loss, long long n, float inv_norm,
            hipStream_t st);
int mlp_adam(int nt, float* const* p, const float* const* g, float* const* m, float* const* v, const long long* n,
             float lr, float b1, float b2, float eps, int step, hipStream_t st);
