#pragma once
#include <hip/hip_runtime.h>

namespace mhffn {

// Products of bfloat16 matrices (mhffn_product.hip), forms as MHFFN_PRODUCT_* in include/mhffn.h; N and K (TN: M and N) multiples of 8.
constexpr int PRODUCT_NT = 0, PRODUCT_NN = 1, PRODUCT_TN = 2;
int product_tile(int form, bool in_order, int M, int N, int K);      // 65536 * rows + columns of the tiles that a launch runs in
bool product_preferred(int M, int N);                                 // the result is one round of tiles or less
bool product_faster(int form, bool in_order, int M, int N, int K);    // faster than the library's product
hipError_t launch_product(int form, bool in_order, const void* A, const void* B, void* C, int M, int N, int K, hipStream_t st);
bool product_pair_faster(bool in_order, int M, int N, int K);         // ... and two launches, of which the library's may be one
// dx [M,K] = dy [M,N] w [N,K] and dw [N,K] = dy^T x [M,K] in one launch, each as launch_product in order has it
hipError_t launch_product_pair(const void* dy, const void* w, const void* x, void* dx, void* dw, int M, int N, int K, hipStream_t st);

}  // namespace mhffn
