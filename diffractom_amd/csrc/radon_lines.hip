// Forward projection by line sweep with two rays per thread, the image lines brought into LDS by the load unit
// (parallel_radon.py:92-124, radon_kernels.cl radon_forward_k); the sums are those of dfm_radon_forward_pairs_sweep, bit
// for bit when the lines are not split.
//
// A workgroup takes 32 orientations and a group of angles of one sweep class (lines: image rows for |X| >= |Y|, columns
// otherwise) and walks the lines; each thread sums two adjacent rays (bins 2 q, 2 q + 1) of one angle. On a line the two
// rays' footprints lie within 4 consecutive pixels ((2 hw + 1) / |coef| < 4, host-checked), the first ray's within the
// first three and the other's within the last three: 4 LDS reads of a quad of orientations serve 24 multiply-adds.
//
// The multiply-adds bound it (3 per ray, line and orientation, 4 cycles a wave instruction: packed FP32 stays off), so
// what counts is how much of the time the VALU runs. Line l + 1 goes from memory into one LDS buffer
// (global_load_lds, 16 bytes a lane) while line l is summed from the other: no registers hold it and no LDS stores
// follow, which leaves 126 VGPRs and two workgroups of 8 waves per CU. Against the register-staged forms (154 VGPRs and
// one workgroup, or 126 VGPRs with the loads waited for at every line's start): 99 x 99 pixels x 29760 orientations x
// 18 angles 1.03 -> 0.82 ms, 9920 x 180 angles 2.58 -> 2.02, 128 x 128 x 15040 x 18 0.98 -> 0.79, 256 x 256 x 3008 x 36
// 1.61 -> 1.20 (the table, which was the default: 1.86, 4.83, 1.82 ms; in bands 2.24).
//
// With few orientations the walk is a chain of lines on a part of the chip, so the lines may be split into nsplit
// ranges, summed by a second kernel in their order.
//
// LDS layouts of a line: pixels 8 quads (128 B) apart, or DUP: every pixel twice, in the first half of one 16-quad
// block and in the second half of the block before, lanes 8-15 of every 16 reading the second copies. A lane reads quad
// (qq + lane) % 8 at step qq, so 8 lanes hit 8 distinct 16-byte bank groups; lanes i and i + 8 meet in the plain layout
// whenever their pixels have equal parity, and never in the duplicated one.
#include "dfm_common.h"

namespace {

constexpr int N_XCD = 8;
constexpr int TH = 512;
constexpr int CQ = 8;        // orientation quads of a workgroup

struct LineGeo {
  double X, Y, T0, hw, top, scale;
};

// 16 bytes a lane from global memory to dst + 16 lane in LDS; lanes off by exec write nothing. In assembly because the
// compiler waits for every such load before the next LDS read, whatever its address. It has no register output; the
// caller waits (vmcnt) before the barrier that hands the data over. The load takes its LDS address from M0, whose scalar
// write needs one wait state before it: without the s_nop the load may still see the M0 of the load before, and the
// compiler adds none inside assembly. M0 is named as written (a reserved register: hence the warning that is off).
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_load16(const float4* p, unsigned dst) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(p), "s"(dst)
               : "memory", "m0");
}
#pragma clang diagnostic pop

template <bool DUP>
__global__ void __launch_bounds__(TH, 4) radon_forward_lines_kernel(
    const float4* __restrict__ img, float4* __restrict__ sino, const LineGeo* __restrict__ geo,
    const int* __restrict__ grp_ang, const int* __restrict__ grp_cls, int n_grp, int na_grp, int ns, int nx, int ny,
    int kstride4, int k4_off, int k4_n, int skstride4, int nsplit, int64_t part_step4) {
  extern __shared__ float4 limg[];   // 2 buffers x (len + 4) pixels x 8 float4 (DUP: (len + 5) x 16)
  constexpr int PS = DUP ? 2 * CQ : CQ;                      // float4 per pixel slot
  const int n_cb = (k4_n + CQ - 1) / CQ;
  // each XCD takes one contiguous range of (orientation block, angle group, line range): a block's image slice is read
  // by one XCD, and every XCD has work when there are few blocks
  const int per_cb = n_grp * nsplit, total = n_cb * per_cb, per = (total + N_XCD - 1) / N_XCD;
  const int wg = (int)(blockIdx.x % N_XCD) * per + (int)(blockIdx.x / N_XCD);
  if (wg >= total) return;                                    // uniform over the workgroup
  const int cb = wg / per_cb, rest = wg - cb * per_cb;
  const int split = rest / n_grp, g = rest - split * n_grp;
  const int cls = grp_cls[g];
  const int len = cls ? ny : nx, nlines = cls ? nx : ny;
  const int lper = (nlines + nsplit - 1) / nsplit;
  const int l0 = split * lper, l1 = min(nlines, l0 + lper);
  const int row = (len + 4 + (DUP ? 1 : 0)) * PS;          // float4 per buffer
  const int t = threadIdx.x, lane = t & 63;
  const int wv = __builtin_amdgcn_readfirstlane(t >> 6);
  const int npair = (ns + 1) >> 1;
  const int al = t / npair, sp = t - al * npair;
  const int a = al < na_grp ? grp_ang[g * na_grp + al] : -1;
  const bool live = a >= 0;
  const int q0 = cb * CQ;

  // ---- zero pads: pixels -2, -1, len, len + 1 of both buffers, both copies; never overwritten. Slot S (pixel S - 2)
  // lies at 8 S + q, or with DUP at 16 (S + 1) + q and 16 S + 8 + q
  if (t < 2 * 4 * CQ) {
    const int q = t % CQ, pp = (t / CQ) % 4, b = t / (4 * CQ);
    const int px = pp < 2 ? pp : len + pp;
    if (DUP) {
      limg[b * row + (px + 1) * PS + q] = make_float4(0.f, 0.f, 0.f, 0.f);
      limg[b * row + px * PS + CQ + q] = make_float4(0.f, 0.f, 0.f, 0.f);
    } else {
      limg[b * row + px * PS + q] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
  }

  // ---- a line into buffer b: 64 consecutive float4 of its LDS row per wave instruction, from slot 2 on: 8 pixels, or
  // with DUP 4 blocks of 16, the first copy of one pixel (the pad for the first block) beside the second copy of the
  // next (the pad for the last). This lane's quad and its pixel in the wave's first instruction:
  constexpr int PXC = DUP ? 4 : 8;                           // pixels per instruction
  const int q = lane & (CQ - 1);
  const int pos0 = DUP ? wv * PXC + (lane >> 4) - ((lane & CQ) ? 0 : 1) : wv * PXC + (lane >> 3);
  const bool qok = q0 + q < k4_n;
  const int64_t pstep = (int64_t)(cls ? nx : 1) * kstride4;  // along a line
  const int64_t lstep = (int64_t)(cls ? 1 : nx) * kstride4;  // from line to line
  const float4* src0 = img + k4_off + q0 + q + pos0 * pstep;
  const int64_t cstep = pstep * (PXC * (TH / 64));
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(__attribute__((address_space(3))) void*)limg) +
                        (2 * PS + wv * 64) * (unsigned)sizeof(float4);
  const int nslots = DUP ? len + 1 : len;
  auto stage = [&](int l, int b) {
    const float4* p = src0 + l * lstep;
    unsigned dst = lds0 + b * row * (unsigned)sizeof(float4);
    int pos = pos0;
    for (int c = wv * PXC; c < nslots; c += PXC * (TH / 64)) {   // uniform over the wave
      if ((unsigned)pos < (unsigned)len && qok) lds_load16(p, dst);
      pos += PXC * (TH / 64);
      p += cstep;
      dst += TH * (unsigned)sizeof(float4);
    }
  };

  // ---- ray-pair geometry: mid(l) of the left ray = m1 l + mL0 (float64), footprint hinv, float32 weight terms
  double m1 = 0.0, mL0 = 0.0, hinv = 0.0, ainv = 1.0;
  float hs = 0.f, ts = 0.f, ds = 0.f;
  int bin_l = 0, bin_r = 0;
  if (live) {
    const LineGeo gg = geo[a];
    const double coef = cls ? gg.Y : gg.X, cross = cls ? gg.X : gg.Y;
    const double inv = 1.0 / coef;
    const int s = 2 * sp;
    m1 = -cross * inv;
    mL0 = -(gg.T0 - (double)s) * inv + (inv < 0.0 ? inv : 0.0);   // the smaller of the two rays' mids
    ainv = fabs(inv);
    hinv = gg.hw * ainv;
    hs = (float)(gg.hw * gg.scale);
    ts = (float)(gg.top * gg.scale);
    ds = (float)(coef * gg.scale);
    bin_l = inv > 0.0 ? s : s + 1;
    bin_r = inv > 0.0 ? s + 1 : s;
  }
  const float c1 = ds, c2 = 2.f * ds, cr1 = (float)((1.0 - ainv) * ds), cr2 = (float)((2.0 - ainv) * ds),
              cr3 = (float)((3.0 - ainv) * ds);
  const int rot = lane & 7;                                  // this lane's quad rotation
  const int hoff = DUP ? (lane & 8) : 0;                     // DUP: lanes 8-15 of 16 read the second copies
  float4 accL[CQ], accR[CQ];
#pragma unroll
  for (int qq = 0; qq < CQ; ++qq) accL[qq] = accR[qq] = make_float4(0.f, 0.f, 0.f, 0.f);
  // the rays' first candidate pixel on line l (from pixel -2 on, so that the candidates need no bounds checks) and the
  // weights: left ray p0 .. p0 + 2, right ray p0 + 1 .. p0 + 3
  auto taps = [&](int l, float (&w)[6]) {
    const double midL = fma(m1, (double)l, mL0);
    double p0 = ceil(midL - hinv);
    p0 = fmin(fmax(p0, -2.0), (double)(len - 2));
    const float uu = (float)(p0 - midL);
    w[0] = __builtin_amdgcn_fmed3f(hs - fabsf(ds * uu), 0.f, ts);
    w[1] = __builtin_amdgcn_fmed3f(hs - fabsf(fmaf(ds, uu, c1)), 0.f, ts);
    w[2] = __builtin_amdgcn_fmed3f(hs - fabsf(fmaf(ds, uu, c2)), 0.f, ts);
    w[3] = __builtin_amdgcn_fmed3f(hs - fabsf(fmaf(ds, uu, cr1)), 0.f, ts);
    w[4] = __builtin_amdgcn_fmed3f(hs - fabsf(fmaf(ds, uu, cr2)), 0.f, ts);
    w[5] = __builtin_amdgcn_fmed3f(hs - fabsf(fmaf(ds, uu, cr3)), 0.f, ts);
    return (int)p0;
  };

  if (l0 < l1) stage(l0, 0);
  for (int l = l0, b = 0; l < l1; ++l, b ^= 1) {
    // this wave's part of line l has landed; after the barrier every wave's has, and every wave is done with the other
    // buffer
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (l + 1 < l1) stage(l + 1, b ^ 1);
    if (live) {
      float w[6];
      const int p0 = taps(l, w);
      const float4* base = limg + b * row + (p0 + 2 + (DUP ? 1 : 0)) * PS - hoff;
#pragma unroll
      for (int qq = 0; qq < CQ; ++qq) {
        const float4* px = base + ((qq + rot) & (CQ - 1));
        const float4 x0 = px[0], x1 = px[PS], x2 = px[2 * PS], x3 = px[3 * PS];
        // FMA chains into the accumulators
#define DFM_PS3(acc, c, wa, xa, wb, xb, wc, xc) acc.c = fmaf(wc, xc.c, fmaf(wb, xb.c, fmaf(wa, xa.c, acc.c)));
        DFM_PS3(accL[qq], x, w[0], x0, w[1], x1, w[2], x2) DFM_PS3(accL[qq], y, w[0], x0, w[1], x1, w[2], x2)
        DFM_PS3(accL[qq], z, w[0], x0, w[1], x1, w[2], x2) DFM_PS3(accL[qq], w, w[0], x0, w[1], x1, w[2], x2)
        DFM_PS3(accR[qq], x, w[3], x1, w[4], x2, w[5], x3) DFM_PS3(accR[qq], y, w[3], x1, w[4], x2, w[5], x3)
        DFM_PS3(accR[qq], z, w[3], x1, w[4], x2, w[5], x3) DFM_PS3(accR[qq], w, w[3], x1, w[4], x2, w[5], x3)
#undef DFM_PS3
      }
    }
  }
  // ---- an infinite or NaN pixel must reach the rays with a weight on it and no others: where a sum is not finite, it is
  // made again from memory without the products with zero weights (of quads beyond the last, whose LDS nothing wrote,
  // the sums mean nothing)
  float nf = 0.f;
#pragma unroll
  for (int qq = 0; qq < CQ; ++qq) {
    if (q0 + ((qq + rot) & (CQ - 1)) >= k4_n) continue;
    nf = fmaf(accL[qq].x, 0.f, fmaf(accL[qq].y, 0.f, fmaf(accL[qq].z, 0.f, fmaf(accL[qq].w, 0.f, nf))));
    nf = fmaf(accR[qq].x, 0.f, fmaf(accR[qq].y, 0.f, fmaf(accR[qq].z, 0.f, fmaf(accR[qq].w, 0.f, nf))));
  }
  if (nf != nf) {
#pragma unroll
    for (int qq = 0; qq < CQ; ++qq) accL[qq] = accR[qq] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 1
    for (int l = l0; l < l1; ++l) {
      float w[6];
      const int p0 = taps(l, w);
      const float wl[4] = {w[0], w[1], w[2], 0.f}, wr[4] = {0.f, w[3], w[4], w[5]};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if ((unsigned)(p0 + i) >= (unsigned)len) continue;
        const float4* px = img + l * lstep + (p0 + i) * pstep + k4_off + q0;
#pragma unroll
        for (int qq = 0; qq < CQ; ++qq) {
          const int qd = (qq + rot) & (CQ - 1);
          if (q0 + qd >= k4_n) continue;
          const float4 x = px[qd];
          if (wl[i] != 0.f) {
            accL[qq].x = fmaf(wl[i], x.x, accL[qq].x);
            accL[qq].y = fmaf(wl[i], x.y, accL[qq].y);
            accL[qq].z = fmaf(wl[i], x.z, accL[qq].z);
            accL[qq].w = fmaf(wl[i], x.w, accL[qq].w);
          }
          if (wr[i] != 0.f) {
            accR[qq].x = fmaf(wr[i], x.x, accR[qq].x);
            accR[qq].y = fmaf(wr[i], x.y, accR[qq].y);
            accR[qq].z = fmaf(wr[i], x.z, accR[qq].z);
            accR[qq].w = fmaf(wr[i], x.w, accR[qq].w);
          }
        }
      }
    }
  }
  // ---- stores through a wave-private LDS transpose: lane l holds its two rays' 8 quads (128 B of a sinogram row each);
  // after it, store instruction j has lanes 8 i .. 8 i + 7 write the 8 quads of lane 8 j + i's row, whole 128-byte lines
  __syncthreads();                                           // every wave is done with the staged lines
  float4* out = sino + split * part_step4;
  float4* wl = limg + wv * (64 * CQ);
  const int srcl = lane >> 3, qd = lane & (CQ - 1);
#pragma unroll
  for (int side = 0; side < 2; ++side) {
#pragma unroll
    for (int qq = 0; qq < CQ; ++qq) wl[lane * CQ + ((qq + rot) & (CQ - 1))] = side ? accR[qq] : accL[qq];
    __builtin_amdgcn_wave_barrier();
    const int bin = side ? bin_r : bin_l;
#pragma unroll
    for (int j = 0; j < CQ; ++j) {
      const int sl = 8 * j + srcl;                            // the lane whose row this lane stores a quad of
      const float4 val = wl[sl * CQ + qd];
      const int a_s = __shfl(a, sl, 64), bin_s = __shfl(bin, sl, 64);
      if (a_s >= 0 && bin_s < ns && q0 + qd < k4_n) out[((int64_t)a_s * ns + bin_s) * skstride4 + q0 + qd] = val;
    }
    __builtin_amdgcn_wave_barrier();
  }
}

// sino = the sum of the nsplit partial sinograms in their order
__global__ void __launch_bounds__(256) lines_sum_kernel(const float4* __restrict__ part, float4* __restrict__ sino,
                                                        int64_t n_rows, int k4_n, int skstride4, int64_t part_step4,
                                                        int nsplit) {
  const int64_t total = n_rows * k4_n;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / k4_n;
    const int64_t o = r * skstride4 + (i - r * k4_n);
    float4 acc = part[o];
    for (int s = 1; s < nsplit; ++s) {
      const float4 v = part[s * part_step4 + o];
      acc.x += v.x;
      acc.y += v.y;
      acc.z += v.z;
      acc.w += v.w;
    }
    sino[o] = acc;
  }
}

}  // namespace

extern "C" {

int dfm_radon_forward_lines(const float* img_k, float* sino, float* part, const double* geo, const int32_t* grp_ang,
                            const int32_t* grp_cls, int32_t n_grp, int32_t na_grp, int32_t n_angles, int32_t ns,
                            int32_t nx, int32_t ny, int32_t kstride, int32_t k_off, int32_t k_n, int32_t skstride,
                            int32_t nsplit, int32_t dup, dfm_stream_t stream) {
  DFM_CHECK_ARG(img_k && sino && geo && grp_ang && grp_cls && (nsplit == 1 || part),
                "dfm_radon_forward_lines: null pointer");
  const int len = nx > ny ? nx : ny;
  DFM_CHECK_ARG(n_grp >= 0 && na_grp >= 1 && n_angles >= 0 && ns >= 1 && nx >= 1 && ny >= 1 && len <= 256 &&
                    kstride % 4 == 0 && k_off % 4 == 0 && k_n % 4 == 0 && k_off >= 0 && k_n >= 0 &&
                    k_off + k_n <= kstride && skstride % 4 == 0 && skstride >= k_n && nsplit >= 1 && nsplit <= 64 &&
                    (int64_t)na_grp * ((ns + 1) / 2) <= TH,
                "dfm_radon_forward_lines: bad sizes (na_grp * ceil(ns / 2) <= 512, image <= 256 x 256, 1 to 64 line "
                "ranges)");
  if (n_grp == 0 || k_n == 0) return DFM_OK;
  // two line buffers, or the store transpose (64 lanes x 8 quads per wave), whichever is larger
  size_t lds = 2 * (size_t)(dup ? (len + 5) * 16 : (len + 4) * 8) * sizeof(float4);
  if (lds < (size_t)TH * CQ * sizeof(float4)) lds = (size_t)TH * CQ * sizeof(float4);
  const int k4n = k_n / 4;
  const int64_t total = (int64_t)((k4n + CQ - 1) / CQ) * n_grp * nsplit;
  DFM_CHECK_ARG(total < ((int64_t)1 << 31) - 8, "dfm_radon_forward_lines: too many workgroups");
  const unsigned grid = (unsigned)((total + N_XCD - 1) / N_XCD * N_XCD);
  const int64_t n_rows = (int64_t)n_angles * ns, step4 = n_rows * (skstride / 4);
  const hipStream_t st = (hipStream_t)stream;
  float4* dst = (float4*)(nsplit > 1 ? part : sino);
#define DFM_FL(D)                                                                                                    \
  hipLaunchKernelGGL((radon_forward_lines_kernel<D>), dim3(grid), dim3(TH), lds, st, (const float4*)img_k, dst,    \
                     (const LineGeo*)geo, grp_ang, grp_cls, n_grp, na_grp, ns, nx, ny, kstride / 4, k_off / 4, k4n, \
                     skstride / 4, nsplit, step4)
  if (dup) {
    DFM_FL(true);
  } else {
    DFM_FL(false);
  }
#undef DFM_FL
  DFM_LAUNCH_CHECK("dfm_radon_forward_lines");
  if (nsplit > 1) {
    hipLaunchKernelGGL(lines_sum_kernel, dim3(dfm::grid_stride_blocks(n_rows * k4n, 256, 1u << 16)), dim3(256), 0, st,
                       (const float4*)part, (float4*)sino, n_rows, k4n, skstride / 4, step4, nsplit);
    DFM_LAUNCH_CHECK("dfm_radon_forward_lines (sum)");
  }
  return DFM_OK;
}

}  // extern "C"
