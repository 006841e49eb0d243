// The library's own bfloat16 GEMM (gemm_mfma.hip): which shapes it takes, its plan for a
// shape, and the launch. gemm.hip runs it where it is the faster side and hipBLASLt elsewhere.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

namespace q35 {

struct MfmaPlan {
    int tile = -1;  // index of the tile form; -1: none (hipBLASLt runs the shape)
    int split = 1;  // parts of K summed in float32 by a second pass
};

// The plan for y [M, N] (rows of ldy) = x [M, K] w [N, K]^T with ws_bytes of scratch for split
// sums on a device of cus CUs. A pure function of its arguments, so a shape keeps its summation
// order from process to process. mfma_gemm_plan leaves the shapes to hipBLASLt where that measured
// faster; mfma_gemm_model does not.
MfmaPlan mfma_gemm_plan(int M, int N, int K, int ldy, size_t ws_bytes, int cus);
MfmaPlan mfma_gemm_model(int M, int N, int K, int ldy, size_t ws_bytes, int cus);

// Rows and columns of a form's tile and its ring stages; false past the last form.
bool mfma_gemm_form(int tile, int* bm, int* bn, int* stages);
// Whether the kernel can run the plan on the shape, and the scratch that its split sums need.
bool mfma_gemm_takes(const MfmaPlan& p, int M, int N, int K, int ldy, size_t ws_bytes);

// Launches the plan; scratch holds the split sums (split > 1). Queues work only.
int mfma_gemm(const MfmaPlan& p, const void* x, const void* w, void* y, void* scratch, int M, int N, int K, int ldy,
              hipStream_t st);

}  // namespace q35
