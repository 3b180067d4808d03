// Backprojection on the FP32 matrix cores (parallel_radon.py:92-124, radon_kernels.cl radon_backward_k), with the
// solvers' primal updates in its epilogue:
//
//   img[p, k] = sum over angles a, bins s with |t_a(p) - s| < hw_a of c_a min(hw_a - |t_a(p) - s|, top_a) sino[a, s, k]
//
// A workgroup takes an 8 x 8 pixel tile and a block of 64 orientations. Per pass of 4 angles the (at most 12) bins the
// tile reaches are staged in LDS, and every pixel's two weights are computed from the angle's float64 geometry as a
// row of four over the 4 bins that its 2 x 2 pixel quad reaches. A wave sums a 4 x 4 pixel quarter of the tile for
// 64 orientations with v_mfma_f32_4x4x1_16b_f32: each of its 16 blocks is a rank-1 update (4 pixels of a quad) x (4
// orientations) by one bin, so an angle costs 16 MFMAs (4 bins x 4 orientation groups), one weight read, four 16-byte
// sinogram reads and no VALU multiply-adds. Half of the MFMA work are the zeros of the 4-bin rows; the pipe runs at
// 1.8 times the rate of unpacked v_fma_f32, and a sinogram value read from LDS serves 4 pixels instead of one (the
// VALU form reads two per pixel and is bound by those reads and their addresses). FP32 operands, products and sums as
// in the VALU form, in the same order over angles.
//
// Measured (SPDHG update; the 8 x 8 VALU form before): 99 x 99 pixels x 29760 orientations x 18 angles 1.34 -> 1.19 ms,
// 5.1 TB/s of x, z, T and sinogram traffic, what a 1 GiB copy reaches; all 180 angles of 9920 orientations, where the
// sums bound it, 3.15 -> 2.18 ms (half of the matrix pipe's rate: the rest are barriers and the staging's VALU). 95
// VGPRs, five waves per SIMD; forms held to 80 or 64 VGPRs spill and take 1.8 / 3.6 ms, passes of 8 angles (twice the
// LDS, two waves per SIMD) 1.97 ms, two orientation blocks per wave (152 VGPRs) 1.25 ms.
#include "dfm_common.h"

#include "radon_bp.h"

namespace {

using dfm::ld_stream;
using dfm::st_stream;

constexpr int N_XCD = 8;
constexpr int TBB = 12;      // bins an 8 x 8 tile reaches at one angle (7 sqrt(2) + 2, host-checked)

typedef float f4 __attribute__((ext_vector_type(4)));

// MODE: 0 writes the image, 1 the SPDHG update, 2 the EM update, 3 the PDHG primal step (as dfm_radon_backward_table)
//
// Wave wv of the four stages angle wv of every pass (its 12 bins in 3 instructions of 4 bins x 64 orientations) and
// computes that angle's 64 pixel weights, so the angle's geometry and addresses are scalar.
template <int MODE>
__global__ void __launch_bounds__(256, 4) radon_backward_mfma_kernel(
    const float4* __restrict__ sino, float4* __restrict__ out, const double* __restrict__ bgeo,
    const int* __restrict__ tbase, int nx, int ny, int ns, int na, int kstride4, int k4_off, int k4_n, int skstride4,
    float4* __restrict__ x, float4* __restrict__ z, const float4* __restrict__ T, float inv_p, float lam) {
  constexpr int ACH = 4, QW = 16;              // angles per pass, orientation quads
  __shared__ float4 sl[ACH * TBB * QW];        // staged bins: [angle][bin][orientation quad]
  __shared__ f4 wt[ACH * 64];                  // weights of a pixel on its quad's 4 bins: [angle][quarter][quad][pixel]
  __shared__ int lb[ACH * 16];                 // byte offset of a quad's first bin: [angle][quarter][quad]
  __shared__ int bad;                          // set when a staged value is infinite or NaN
  const int tnx = (nx + 7) >> 3, tny = (ny + 7) >> 3;
  const int ntiles = tnx * tny;
  const int n_grp = (k4_n + QW - 1) / QW;
  // each XCD takes one contiguous range of (orientation block, tile) pairs, so a block's sinogram slab is read by the
  // tiles of one XCD (its L2) and every XCD has work when there are few blocks
  const int total = n_grp * ntiles, per = (total + N_XCD - 1) / N_XCD;
  const int w = (int)(blockIdx.x % N_XCD) * per + (int)(blockIdx.x / N_XCD);
  if (w >= total) return;                      // uniform over the workgroup
  const int grp = w / ntiles, tile = w - grp * ntiles;
  const int tx0 = (tile % tnx) * 8, ty0 = (tile / tnx) * 8;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);   // staging: the angle; sums: the pixel quarter
  if (tid == 0) bad = 0;

  // staging: this lane's bin of the 4 of an instruction and its orientation quad
  const int sb = lane >> 4, kk = grp * QW + (lane & 15);
  const int lofs = sb * skstride4 + kk;
  const bool kok = kk < k4_n;
  // weights: this lane's pixel (quad-major within each 4 x 4 quarter)
  const int wpx = tx0 + ((lane >> 4) & 1) * 4 + ((lane >> 2) & 1) * 2 + (lane & 1);
  const int wpy = ty0 + ((lane >> 5) & 1) * 4 + ((lane >> 3) & 1) * 2 + ((lane >> 1) & 1);
  const bool wok = wpx < nx && wpy < ny;

  float4 v[3];
  f4 wr;
  int wo;
  f4 acc[4];                                   // acc[m][r]: pixel r of the lane's quad, orientation 4 (lane % 16) + m
#pragma unroll
  for (int m = 0; m < 4; ++m) acc[m] = f4{0.f, 0.f, 0.f, 0.f};

  // the tile's first bin at angle a, read one pass before its bins' addresses need it
  auto first = [&](int a) { return a < na ? tbase[(int64_t)a * ntiles + tile] : 0; };
  // the staged bins and the weights of angle a (if < na) into registers
  auto fetch = [&](int a, int b0) {
#pragma unroll
    for (int u = 0; u < 3; ++u) v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
    wr = f4{0.f, 0.f, 0.f, 0.f};
    wo = 0;
    if (a >= na) return;                       // uniform over the wave
    const float4* row = sino + ((int64_t)a * ns + b0) * skstride4;
#pragma unroll
    for (int u = 0; u < 3; ++u)
      if (kok && (unsigned)(b0 + 4 * u + sb) < (unsigned)ns) v[u] = row[lofs + 4 * u * skstride4];
    // taps s0 = floor(t - hw) + 1 and s0 + 1 with weights c clamp(hw - |t - s|, 0, top) where the bin is on the
    // detector (the host's pixel table), written on r = (t - hw) - floor(t - hw): t - s0 = r + hw - 1
    const double* g = bgeo + (int64_t)a * 6;
    const double hw = g[3], tp = g[4], sc = g[5];
    const double f = fma(g[0], (double)wpx, fma(g[1], (double)wpy, g[2])) - hw;
    const double fl = floor(f), r = f - fl;
    const int s0 = (int)fl + 1;
    const double k0 = fmin(fmin(1.0 - r, r + (2.0 * hw - 1.0)), tp), k1 = fmin(r + (2.0 * hw - 2.0), tp);
    const float w0 = (wok && (unsigned)s0 < (unsigned)ns) ? fmaxf((float)(sc * k0), 0.f) : 0.f;
    const float w1 = (wok && (unsigned)(s0 + 1) < (unsigned)ns) ? fmaxf((float)(sc * k1), 0.f) : 0.f;
    // the quad's 4 bins start at its pixels' smallest tap
    int o = wok ? min(max(s0, 0), ns - 1) - b0 : 1 << 20;
    o = min(o, __shfl_xor(o, 1, 64));
    o = min(o, __shfl_xor(o, 2, 64));
    const int rel = min(max(o, 0), TBB - 4);
    const int d = s0 - b0 - rel;               // the first tap's place on the quad's 4 bins
#pragma unroll
    for (int k = 0; k < 4; ++k) wr[k] = d == k ? w0 : d + 1 == k ? w1 : 0.f;
    wo = rel * QW * (int)sizeof(float4);
  };
  auto store = [&]() {
    float nf = 0.f;                            // NaN once a value is infinite or NaN
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      sl[wv * TBB * QW + 64 * u + lane] = v[u];
      nf = fmaf(v[u].x, 0.f, fmaf(v[u].y, 0.f, fmaf(v[u].z, 0.f, fmaf(v[u].w, 0.f, nf))));
    }
    if (nf != nf) bad = 1;
    wt[wv * 64 + lane] = wr;
    if ((lane & 3) == 0) lb[wv * 16 + (lane >> 2)] = wo;
  };
  const char* sp = reinterpret_cast<const char*>(&sl[lane & 15]);
  const f4* wp = &wt[wv * 16 + (lane >> 4) * 4];
  const int* bp = &lb[wv * 4 + (lane >> 4)];
  auto sums = [&]() {
    if (bad) {
      // an infinite or NaN bin must reach the pixels with a weight on it and no others: no products with the zeros
      // of the 4-bin rows
#pragma unroll 1
      for (int al = 0; al < ACH; ++al) {
        const char* sa = sp + al * TBB * QW * (int)sizeof(float4) + bp[al * 16];
#pragma unroll 1
        for (int k = 0; k < 4; ++k) {
          const float4 s = *reinterpret_cast<const float4*>(sa + k * QW * (int)sizeof(float4));
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float ww = wp[al * 64 + r][k];
            if (ww != 0.f) {
              acc[0][r] = fmaf(ww, s.x, acc[0][r]);
              acc[1][r] = fmaf(ww, s.y, acc[1][r]);
              acc[2][r] = fmaf(ww, s.z, acc[2][r]);
              acc[3][r] = fmaf(ww, s.w, acc[3][r]);
            }
          }
        }
      }
      return;
    }
#pragma unroll
    for (int al = 0; al < ACH; ++al) {         // angles beyond the last have zero weights and zero bins
      const f4 ww = wp[al * 64 + (lane & 3)];
      const char* sa = sp + al * TBB * QW * (int)sizeof(float4) + bp[al * 16];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float4 s = *reinterpret_cast<const float4*>(sa + k * QW * (int)sizeof(float4));
        acc[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(ww[k], s.x, acc[0], 0, 0, 0);
        acc[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(ww[k], s.y, acc[1], 0, 0, 0);
        acc[2] = __builtin_amdgcn_mfma_f32_4x4x1f32(ww[k], s.z, acc[2], 0, 0, 0);
        acc[3] = __builtin_amdgcn_mfma_f32_4x4x1f32(ww[k], s.w, acc[3], 0, 0, 0);
      }
    }
  };
  // the next pass's loads are in flight and its weights computed while this one is summed
  fetch(wv, first(wv));
  int b1 = first(ACH + wv);
  for (int a0 = 0; a0 < na; a0 += ACH) {
    __syncthreads();                           // every wave is done with the previous pass's LDS
    store();
    __syncthreads();
    if (a0 + ACH < na) {
      const int b2 = first(a0 + 2 * ACH + wv);
      fetch(a0 + ACH + wv, b1);
      b1 = b2;
    }
    sums();
  }

  if (!kok) return;
  const int qx = tx0 + (wv & 1) * 4 + ((lane >> 4) & 1) * 2, qy = ty0 + (wv >> 1) * 4 + (lane >> 5) * 2;
#pragma unroll
  for (int h = 0; h < 2; ++h) {                // two pixels at a time: their x, z, T loads in flight together
    const int py = qy + h;
    float4 zz[2], xx[2], tt[2];
    int64_t o[2];
    bool live[2];
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int px = qx + c;
      live[c] = px < nx && py < ny;
      o[c] = (int64_t)(py * nx + px) * kstride4 + kk + k4_off;
      if (MODE >= 1 && live[c]) {
        if (MODE == 1) zz[c] = ld_stream(z + o[c]);
        xx[c] = ld_stream(x + o[c]);
        tt[c] = ld_stream(T + o[c]);
      }
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      if (!live[c]) continue;
      const float4 a = make_float4(acc[0][2 * h + c], acc[1][2 * h + c], acc[2][2 * h + c], acc[3][2 * h + c]);
      if (MODE == 0) {
        st_stream(out + o[c], a);
      } else if (MODE == 1) {
        // z += dz, x = max(0, x - T (z + dz / p + lam)) where T > 0, else 0
        float4 zn, xn;
#define DFM_UPD(f)                                                                                             \
  zn.f = zz[c].f + a.f;                                                                                        \
  xn.f = tt[c].f > 0.0f ? fmaxf(0.0f, xx[c].f - tt[c].f * ((zn.f + inv_p * a.f) + lam)) : 0.0f;
        DFM_UPD(x) DFM_UPD(y) DFM_UPD(z) DFM_UPD(w)
#undef DFM_UPD
        st_stream(z + o[c], zn);
        st_stream(x + o[c], xn);
      } else if (MODE == 2) {
        // the EM update: x = x A^T r / (sens + lam) where sens > 0
        float4 xn;
#define DFM_EM(f) xn.f = tt[c].f > 0.0f ? xx[c].f * a.f / (tt[c].f + lam) : xx[c].f;
        DFM_EM(x) DFM_EM(y) DFM_EM(z) DFM_EM(w)
#undef DFM_EM
        st_stream(x + o[c], xn);
      } else {
        // the PDHG primal step and extrapolation: x' = max(0, x - T (A^T y + lam)) where T > 0, else 0; z = 2 x' - x
        float4 xn, xb;
#define DFM_PD(f)                                                                         \
  xn.f = tt[c].f > 0.0f ? fmaxf(0.0f, xx[c].f - tt[c].f * (a.f + lam)) : 0.0f;           \
  xb.f = 2.0f * xn.f - xx[c].f;
        DFM_PD(x) DFM_PD(y) DFM_PD(z) DFM_PD(w)
#undef DFM_PD
        st_stream(z + o[c], xb);
        st_stream(x + o[c], xn);
      }
    }
  }
}

}  // namespace

namespace dfm {

int launch_backward_mfma(const float* sino, float* img_k, const double* bgeo, const int32_t* tbase, int nx, int ny,
                         int ns, int na, int kstride4, int k4_off, int k4_n, int skstride4, float* x, float* z,
                         const float* T, float inv_p, float lam, int mode, hipStream_t st) {
  const int64_t total = (int64_t)((k4_n + 15) / 16) * ((nx + 7) / 8) * ((ny + 7) / 8);
  DFM_CHECK_ARG(total < ((int64_t)1 << 31) - 8, "dfm_radon_backward_table: too many tiles");
  const unsigned grid = (unsigned)((total + N_XCD - 1) / N_XCD * N_XCD);
#define DFM_BM(M)                                                                                                  \
  hipLaunchKernelGGL((radon_backward_mfma_kernel<M>), dim3(grid), dim3(256), 0, st, (const float4*)sino,           \
                     (float4*)img_k, bgeo, tbase, nx, ny, ns, na, kstride4, k4_off, k4_n, skstride4, (float4*)x,   \
                     (float4*)z, (const float4*)T, inv_p, lam)
  if (mode == 0) {
    DFM_BM(0);
  } else if (mode == 1) {
    DFM_BM(1);
  } else if (mode == 2) {
    DFM_BM(2);
  } else {
    DFM_BM(3);
  }
#undef DFM_BM
  DFM_LAUNCH_CHECK("dfm_radon_backward_table");
  return DFM_OK;
}

}  // namespace dfm
