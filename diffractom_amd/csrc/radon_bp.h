// The matrix-core backprojection (radon_bp.hip), launched by dfm_radon_backward_table.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dfm {

// tbase: the 8 x 8 tiles' first bins. Sizes and offsets of orientations in quads. Returns a status as the C ABI does.
int launch_backward_mfma(const float* sino, float* img_k, const double* bgeo, const int32_t* tbase, int nx, int ny,
                         int ns, int na, int kstride4, int k4_off, int k4_n, int skstride4, float* x, float* z,
                         const float* T, float inv_p, float lam, int mode, hipStream_t st);

}  // namespace dfm
