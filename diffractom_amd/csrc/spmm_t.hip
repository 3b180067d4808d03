// Pole-figure CSR products on transposed operands (wavefront-segmented SpMM), both directions with one kernel:
//
//   out[s, a, row, y] = alpha * sum_{e in CSR row (r, row), col(e) in split s} val[e] * in[a, col(e), y]
//
// forward (rows = segments j, columns = orientations k):  in = sinogram transposed (a, k, y), out -> data[r, y, j]
// adjoint (rows = orientations k, columns = segments j):  in = data rows transposed (a, j, y), out -> sino[a, y, k]
// with r = omegas[a] the angle's data row (pf_kernels.cl:597-687 spmm_pf_forward_c / spmm_pf_adjoint_c;
// single_phase_forward_operator.py:38-123).
//
// A workgroup of 16 waves owns 64 R consecutive CSR rows of one angle and one column range (split s). It walks the
// range in chunks of kc columns: the chunk of `in` (kc rows of ys floats) is staged in LDS, then every wave consumes, for
// each of its R quads of rows, the rows' entries that fall in the chunk. A row belongs to 16 lanes (four rows at once in
// a wave), each holding 4 detector positions of every 64: the 16 lanes hold a window of 16 entries of their row, entry t
// reaches all of them as a DPP row broadcast (its value as an operand of the FMA, its LDS offset of the address add) and
// its operand is one contiguous 16-byte read per lane. Four entries cost 1 add, 4 NB FMAs and NB LDS reads for 64 NB
// detector positions; with an entry per wave-instruction (two v_readlane, an add and 4-byte reads each) they cost 4
// times (3 + NB), and that issue rate bounded the kernel: 9899 orientations x 180 angles x 900 segments x 103 rows, 6.2 %
// fill (9.9e7 entries), forward with its split in two and transposes 2.47 -> 1.77 ms, adjoint 2.05 -> 1.30. VALU issue
// (62 % of the time at 2.4 GHz: a third of it entries, the rest the visits, their rounding to 4 entries and the staging) and
// the waits of the visits' chains (54 % of the waves' cycles) bound it now. Rows whose
// entries run out in a chunk before the others' of their quad read a zero operand. The first two windows of a visit are
// loaded one visit ahead.
//
// Summation. Products into the transposed output (the forward: long rows of orientations) sum a row's entries of a chunk
// apart, in A interleaved sums, and add them to the row's sum, up to 192 detector positions: the FP32 chain is a chunk's
// entries / A and then the chunks, whatever the number of ranges (one chain instead: 1500 orientations in one range
// 1.4e-7 from 64 bits, so 4.8e-8, 3 % of the time). Otherwise (the adjoint: rows of segments; above 192 positions, where
// the registers leave no room for sums apart) a row is one chain in CSR order, as in the row-per-thread kernels.
#include <algorithm>
#include <type_traits>

#include "dfm_common.h"

namespace {

constexpr int SPT_WAVES = 16;
constexpr int SPT_LDS_FLOATS = 40960;   // 160 KiB

typedef float f32x4 __attribute__((ext_vector_type(4)));

// lane K of every 16 lanes, to those 16 lanes (DPP row_newbcast)
template <int K>
__device__ __forceinline__ int bcast16(int x) {
  return __builtin_amdgcn_update_dpp(0, x, 0x150 + K, 0xf, 0xf, true);
}

// An operand row in LDS is NB blocks of 16 units of 16 bytes; unit u of row c lies at u ^ swz(c) of its block. Rows of
// whole blocks: the 16-byte reads of a wave go 16 lanes at a time, 8 of one window's 16 lanes (0-3 and 12-15, or 4-11) and
// the other 8 positions of another's, so rows at one bank offset, whatever they are, never conflict (with rows of 108
// floats 42 % of the LDS cycles were conflicts); swz keeps those sets and halves the conflicts of the transposing writes.
__device__ __forceinline__ int swz(int c) { return (c >> 2 & 1) * 12; }

// entry K of the 16-lane windows: its operand row (off: byte offset in LDS, its swizzle in the unit bits; lane16: this
// lane's 16 l) and its product
template <int K, int NB>
__device__ __forceinline__ void entry_load(const char* lds, int off, int lane16, f32x4 (&x)[NB]) {
  const char* p = lds + (bcast16<K>(off) ^ lane16);
#pragma unroll
  for (int h = 0; h < NB; ++h) x[h] = *reinterpret_cast<const f32x4*>(p + 256 * h);
}
template <int K, int NB, bool FIRST>
__device__ __forceinline__ void entry_fma(int vb, const f32x4 (&x)[NB], f32x4 (&acc)[NB]) {
  const float v = __int_as_float(bcast16<K>(vb));
#pragma unroll
  for (int h = 0; h < NB; ++h)
#pragma unroll
    for (int e = 0; e < 4; ++e) acc[h][e] = FIRST ? v * x[h][e] : acc[h][e] + v * x[h][e];
}

// entries K .. 15 of the windows while fewer than `steps` are done, U operand rows in flight; entry t goes to sum t % A.
// FIRST: the sums start with the first A entries
template <int K, int U, int A, int NB, bool FIRST>
__device__ __forceinline__ void window(const char* lds, int off, int vb, int lane16, int steps, f32x4 (&acc)[A][NB]) {
  static_assert(U % A == 0, "a group of U entries starts every sum");
  if constexpr (K < 16) {
    if (steps <= K) return;                                  // uniform
    f32x4 x[U][NB];
    entry_load<K, NB>(lds, off, lane16, x[0]);
    if constexpr (U > 1) entry_load<K + 1, NB>(lds, off, lane16, x[1]);
    if constexpr (U > 2) {
      entry_load<K + 2, NB>(lds, off, lane16, x[2]);
      entry_load<K + 3, NB>(lds, off, lane16, x[3]);
    }
    __builtin_amdgcn_sched_barrier(0);
    entry_fma<K, NB, FIRST>(vb, x[0], acc[0]);
    if constexpr (U > 1) entry_fma<K + 1, NB, FIRST && (A > 1)>(vb, x[1], acc[1 % A]);
    if constexpr (U > 2) {
      entry_fma<K + 2, NB, FIRST && (A > 2)>(vb, x[2], acc[2 % A]);
      entry_fma<K + 3, NB, FIRST && (A > 2)>(vb, x[3], acc[3 % A]);
    }
    window<K + U, U, A, NB, false>(lds, off, vb, lane16, steps, acc);
  }
}

// the most entries any of the wave's four rows has in a window, from the lanes that hold one (a prefix of each 16)
__device__ __forceinline__ int window_steps(unsigned long long m) {
  const unsigned f = (unsigned)m | (unsigned)(m >> 32);
  return __popc((f | f >> 16) & 0xffffu);
}

// A > 0: a row's entries of a chunk are summed apart (A interleaved sums), then added to the row's sum; 0: one chain
template <int R, int NB, int U, int A>
__global__ void __launch_bounds__(1024) spmm_t_kernel(const float* __restrict__ inT, const int* __restrict__ row_ptr,
                                                      const uint16_t* __restrict__ col, const float* __restrict__ val,
                                                      float* __restrict__ outT, const int* __restrict__ omegas,
                                                      int my, int ys, int ncols, int nrows, int rows_out, int compact,
                                                      float alpha, int cspan, int kc, int n_angles, int64_t in_ld,
                                                      int64_t out_ld, int ys_out, int vec_out) {
  extern __shared__ __align__(16) float lin[];
  const int lane = threadIdx.x & 63, l16 = lane & 15, lane16 = 16 * l16;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int a = blockIdx.y, s = blockIdx.z;
  const int ra = omegas ? omegas[a] : a;
  const int rr = compact ? a : ra;
  const int rw0 = w * 4 * R + (lane >> 4);                   // row quad i: row rw0 + 4 i of the workgroup's 64 R
  const int row0 = blockIdx.x * SPT_WAVES * 4 * R + rw0;
  const int c_lo = s * cspan, c_hi = min(ncols, c_lo + cspan);

  // the entries of the workgroup's rows, from one before the first on (so that entry 0 is there whatever the rows hold):
  // 32-bit offsets to a scalar base
  const int* wg_ptr = row_ptr + (int64_t)rr * nrows;
  const int wr0 = blockIdx.x * SPT_WAVES * 4 * R;
  const int e0 = max(wg_ptr[min(wr0, nrows)] - 1, 0), e1 = wg_ptr[min(wr0 + SPT_WAVES * 4 * R, nrows)];
  // (no entries so far: the arrays may be empty, and the repeated entry 0 is read from row_ptr instead)
  const uint16_t* colw = e1 > 0 ? col + e0 : reinterpret_cast<const uint16_t*>(row_ptr);
  const float* valw = e1 > 0 ? val + e0 : reinterpret_cast<const float*>(row_ptr);
  // per row: the next entry (the first with column >= c_lo) and the end
  int cur[R], end[R];
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = row0 + 4 * i;
    cur[i] = end[i] = 0;
    if (row < nrows) {
      const int64_t rb = (int64_t)rr * nrows + row;
      int lo = row_ptr[rb] - e0, hi = row_ptr[rb + 1] - e0;
      end[i] = hi;
      if (c_lo > 0) {
        while (lo < hi) {
          const int mid = (lo + hi) >> 1;
          if ((int)colw[mid] < c_lo) lo = mid + 1;
          else hi = mid;
        }
      }
      cur[i] = lo;
    }
  }
  f32x4 acc[R][1][NB];
#pragma unroll
  for (int i = 0; i < R; ++i)
#pragma unroll
    for (int h = 0; h < NB; ++h) acc[i][0][h] = f32x4{0.f, 0.f, 0.f, 0.f};

  // window entry `cu + l16` of a row ending at en (past the end: a repeated entry, not counted)
  auto fetch = [&](int cu, int en, int& c, float& v) {
    const unsigned e = (unsigned)max(min(cu + l16, en - 1), 0);
    c = (int)colw[e];
    v = valw[e];
  };
  int pc0, pc1;
  float pv0, pv1;
  fetch(cur[0], end[0], pc0, pv0);
  fetch(cur[0] + 16, end[0], pc1, pv1);

  // the zero operand
  constexpr int ROW = 64 * NB;                               // floats of an operand row in LDS
  const int zoff = kc * ROW * 4;
  auto row_off = [&](int c) { return c * (ROW * 4) + (swz(c) << 4); };
  for (int i = threadIdx.x; i < 64 * NB; i += SPT_WAVES * 64) lin[kc * ROW + i] = 0.f;

  // in_ld > 0: the operand untransposed, (my, in_ld) per angle, transposed while it is staged; in_ld == 0: transposed,
  // (ncols, ys)
  const float* src = in_ld ? inT + (int64_t)a * my * in_ld : inT + (int64_t)a * ncols * ys;
  const char* lds = reinterpret_cast<const char*>(lin);
  for (int c0 = c_lo; c0 < c_hi; c0 += kc) {
    const int kn = min(kc, c_hi - c0);
    __syncthreads();
    if (in_ld) {
      // an item is 16 rows x 64 columns: a lane loads 4 rows x 4 columns (16-byte loads, 256 contiguous bytes of a row
      // for the 16 lanes of its row quad) and writes them transposed (16 bytes each). c0, in_ld and the base are
      // multiples of 4 floats, and the columns up to kn rounded up to 4 lie in the row and in the LDS chunk
      constexpr int SU = 2;                                  // items in flight per lane
      const int kq = (lane & 3) + ((lane >> 4) << 2), yq = (lane >> 2) & 3;
      const int kn4 = (kn + 3) & ~3, nj = (kn + 63) / 64, items = (my + 15) / 16 * nj;
      for (int it0 = w; it0 < items; it0 += SPT_WAVES * SU) {
        f32x4 v[SU][4];
#pragma unroll
        for (int u = 0; u < SU; ++u) {
          const int it = it0 + SPT_WAVES * u, m = it / nj;
          const int kk = min(64 * (it - m * nj) + 4 * kq, kn4 - 4), y = 16 * m + 4 * yq;
#pragma unroll
          for (int e = 0; e < 4; ++e)
            v[u][e] = *reinterpret_cast<const f32x4*>(src + (int64_t)min(y + e, my - 1) * in_ld + c0 + kk);
        }
#pragma unroll
        for (int u = 0; u < SU; ++u) {
          const int it = it0 + SPT_WAVES * u, m = it / nj;
          const int kk = 64 * (it - m * nj) + 4 * kq, y = 16 * m + 4 * yq;
          if (kk < kn && y < my) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              *reinterpret_cast<f32x4*>(lin + (kk + e) * ROW + (y ^ swz(kk) * 4)) =
                  f32x4{v[u][0][e], v[u][1][e], v[u][2][e], v[u][3][e]};
          }
        }
      }
    } else {
      constexpr int SU = 8;                                  // staging loads in flight per lane
      const float* g = src + (int64_t)c0 * ys;
      const int n4 = kn * (ROW / 4);
      for (int i0 = threadIdx.x; i0 < n4; i0 += SPT_WAVES * 64 * SU) {
        f32x4 v[SU];
#pragma unroll
        for (int u = 0; u < SU; ++u) {
          const int i = min(i0 + SPT_WAVES * 64 * u, n4 - 1), c = i / (ROW / 4), y = 4 * (i % (ROW / 4));
          v[u] = *reinterpret_cast<const f32x4*>(g + (int64_t)c * ys + min(y, ys - 4));
        }
#pragma unroll
        for (int u = 0; u < SU; ++u) {
          const int i = i0 + SPT_WAVES * 64 * u, c = i / (ROW / 4), y = 4 * (i % (ROW / 4));
          if (i < n4) *reinterpret_cast<f32x4*>(lin + c * ROW + (y ^ swz(c) * 4)) = v[u];
        }
      }
    }
    __syncthreads();
    const int c1 = c0 + kn;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      bool in0 = cur[i] + l16 < end[i] && pc0 < c1, in1 = cur[i] + 16 + l16 < end[i] && pc1 < c1;
      const int off0 = in0 ? row_off(pc0 - c0) : zoff, off1 = in1 ? row_off(pc1 - c0) : zoff;
      const int vb0 = in0 ? __float_as_int(pv0) : 0, vb1 = in1 ? __float_as_int(pv1) : 0;
      const unsigned long long m0 = __ballot(in0), m1 = __ballot(in1);
      const int shift = lane & 48;
      const int n = __popc((unsigned)(m0 >> shift) & 0xffffu) + __popc((unsigned)(m1 >> shift) & 0xffffu);
      cur[i] += n;
      // the next visit's windows (the last row quad: the first one's in the next chunk)
      fetch(cur[i + 1 < R ? i + 1 : 0], end[i + 1 < R ? i + 1 : 0], pc0, pv0);
      fetch(cur[i + 1 < R ? i + 1 : 0] + 16, end[i + 1 < R ? i + 1 : 0], pc1, pv1);
      __builtin_amdgcn_sched_barrier(0);
      // the visit's windows into p; a row with more than 32 entries in the chunk has more of them
      auto windows = [&](auto first, auto& p) {
        constexpr int NA = sizeof(p) / sizeof(p[0]);
        window<0, U, NA, NB, decltype(first)::value>(lds, off0, vb0, lane16, window_steps(m0), p);
        if (m1) window<0, U, NA, NB, false>(lds, off1, vb1, lane16, window_steps(m1), p);
        bool more = __any(n == 32);
        while (more) {
          int c;
          float v;
          fetch(cur[i], end[i], c, v);
          const bool in = cur[i] + l16 < end[i] && c < c1;
          const unsigned long long m = __ballot(in);
          window<0, U, NA, NB, false>(lds, in ? row_off(c - c0) : zoff, in ? __float_as_int(v) : 0, lane16,
                                      window_steps(m), p);
          const int nn = __popc((unsigned)(m >> shift) & 0xffffu);
          cur[i] += nn;
          more = __any(nn == 16);
          if (R == 1) {                                      // the next visit is this row's
            fetch(cur[0], end[0], pc0, pv0);
            fetch(cur[0] + 16, end[0], pc1, pv1);
          }
        }
      };
      if constexpr (A > 0) {
        if (m0) {                                            // uniform
          f32x4 p[A][NB];
          windows(std::true_type{}, p);
#pragma unroll
          for (int s = A / 2; s > 0; s /= 2)
#pragma unroll
            for (int q = 0; q < s; ++q)
#pragma unroll
              for (int h = 0; h < NB; ++h) p[q][h] += p[q + s][h];
#pragma unroll
          for (int h = 0; h < NB; ++h) acc[i][0][h] += p[0][h];
        }
      } else {
        windows(std::false_type{}, acc[i]);
      }
    }
  }

  if (out_ld) {
    // out (n_angles, my, out_ld): per group of 64 y, the workgroup's RB = 64 R rows go through LDS as (y, row) with
    // the odd row stride RB + 1 (64 (RB + 1) floats), then out one y row of RB consecutive floats at a time
    constexpr int RB = SPT_WAVES * 4 * R, RW = RB + 1;
    const int r = threadIdx.x % RB, row = blockIdx.x * RB + r;
    float* dst = outT + (int64_t)a * my * out_ld;
#pragma unroll
    for (int h = 0; h < NB; ++h) {
      __syncthreads();
#pragma unroll
      for (int i = 0; i < R; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) lin[(4 * l16 + e) * RW + rw0 + 4 * i] = alpha * acc[i][0][h][e];
      __syncthreads();
      if (row < rows_out)
        for (int yl = threadIdx.x / RB; yl < 64 && 64 * h + yl < my; yl += SPT_WAVES * 64 / RB)
          dst[(int64_t)(64 * h + yl) * out_ld + row] = lin[yl * RW + r];
    }
    return;
  }
  float* dst = outT + ((int64_t)s * n_angles + a) * rows_out * ys_out;
#pragma unroll
  for (int i = 0; i < R; ++i) {
    const int row = row0 + 4 * i;
    if (row < rows_out) {
#pragma unroll
      for (int h = 0; h < NB; ++h) {
        const int y = 64 * h + 4 * l16;
        float* d = dst + (int64_t)row * ys_out + y;
        const f32x4 v = alpha * acc[i][0][h];
        if (vec_out && y + 3 < my) {
          *reinterpret_cast<f32x4*>(d) = v;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (y + e < my) d[e] = v[e];
        }
      }
    }
  }
}

// out[ao, c, r] (+)= sum_{s < nsplit} in[s * split_stride + ai * in_mat + r * in_ld + c]: a batch of (nr x nc)
// transposes through 32 x 33 LDS tiles, ai = omegas[a] when the angle list selects input matrices (omega_out 0),
// ao = omegas[a] when it selects output matrices (omega_out 1), a otherwise.
__global__ void __launch_bounds__(256) transpose_sum_kernel(const float* __restrict__ in, float* __restrict__ out,
                                                            const int* __restrict__ omegas, int omega_out, int nr,
                                                            int nc, int64_t in_ld, int64_t in_mat, int64_t out_ld,
                                                            int64_t out_mat, int nsplit, int64_t split_stride,
                                                            int accumulate) {
  __shared__ float tile[32][33];
  const int a = blockIdx.z;
  const int ai = (omegas && !omega_out) ? omegas[a] : a;
  const int ao = (omegas && omega_out) ? omegas[a] : a;
  const int c0 = blockIdx.x * 32, r0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  const float* src = in + (int64_t)ai * in_mat;
  float* dst = out + (int64_t)ao * out_mat;
  for (int k = ty; k < 32; k += 8) {
    const int r = r0 + k, c = c0 + tx;
    float v = 0.f;
    if (r < nr && c < nc) {
      const float* p = src + (int64_t)r * in_ld + c;
      for (int q = 0; q < nsplit; ++q) v += p[(int64_t)q * split_stride];
    }
    tile[k][tx] = v;
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int c = c0 + k, r = r0 + tx;
    if (c < nc && r < nr) {
      float* p = dst + (int64_t)c * out_ld + r;
      *p = accumulate ? *p + tile[tx][k] : tile[tx][k];
    }
  }
}

template <int R, int NB>
void launch_spmm_t(dim3 grid, size_t lds, hipStream_t st, const float* inT, const int* row_ptr, const uint16_t* col,
                   const float* val, float* outT, const int* omegas, int my, int ys, int ncols, int nrows,
                   int rows_out, int compact, float alpha, int cspan, int kc, int n_angles, int64_t in_ld,
                   int64_t out_ld, int ys_out) {
  const int vec_out = ys_out % 4 == 0 && (uintptr_t)outT % 16 == 0;
  constexpr int U = NB <= 2 ? 4 : NB <= 4 ? 2 : 1, A = NB == 1 ? 4 : NB <= 3 ? 2 : 0;
#define DFM_SPT_A(AA)                                                                                               \
  hipLaunchKernelGGL((spmm_t_kernel<R, NB, U, AA>), grid, dim3(SPT_WAVES * 64), lds, st, inT, row_ptr, col, val, outT, \
                     omegas, my, ys, ncols, nrows, rows_out, compact, alpha, cspan, kc, n_angles, in_ld, out_ld,    \
                     ys_out, vec_out)
  if (out_ld) DFM_SPT_A(0);
  else DFM_SPT_A(A);
#undef DFM_SPT_A
}

// row quads per wave: 4 (256 rows a workgroup), 2 where the accumulators of more than 128 detector positions leave no
// registers for more (128 VGPRs with 16 waves on a CU)
int row_quads(int my) { return my <= 128 ? 4 : 2; }

// ... and fewer where that leaves workgroups for less than half of the 256 CUs (a workgroup's LDS fills one): the operand
// is staged again for each, the rows' serial walks shorten (us, 900 segments x 103 rows, 256 / fewer rows: adjoint, 333
// orientations x 50 angles 92 / 62, 1500 x 18 63 / 45; forward in one range, 1500 x 18 92 / 64; with 256 workgroups as
// the line 54 instead of 45, 73 instead of 64)
int row_quads(int my, int64_t rows_out, int64_t others) {
  int R = row_quads(my);
  while (R > 1 && (rows_out + 64 * R - 1) / (64 * R) * others < 128) R /= 2;
  return R;
}

// ys: the transposed input's row stride (in_ld == 0); ys_out: the transposed output's
int spmm_t_impl(const float* in, int64_t in_ld, const int32_t* row_ptr, const uint16_t* col, const float* val,
                float* out, int64_t out_ld, int32_t ys_out, const int32_t* omegas, int32_t n_angles, int32_t my,
                int32_t ys, int32_t ncols, int32_t nrows, int32_t rows_out, int32_t compact, float alpha,
                int32_t nsplit, int32_t kc, hipStream_t st) {
  const int nb = (my + 63) / 64;
  const int row = 64 * nb;           // floats of an operand row in LDS
  const int kc_max = SPT_LDS_FLOATS / row - 1;
  if (kc <= 0 || kc > kc_max) kc = kc_max;
  int cspan = (ncols + nsplit - 1) / nsplit;
  if (in_ld) {                       // 16-byte staging of the untransposed operand: chunks start at multiples of 4
    kc = std::max(kc & ~3, 4);
    cspan = (cspan + 3) & ~3;
  }
  kc = std::min(kc, in_ld ? cspan : std::min(cspan, ncols));
  if (n_angles == 0 || rows_out == 0) return DFM_OK;
  const int R = row_quads(my, rows_out, (int64_t)n_angles * nsplit);
  const dim3 grid((unsigned)((rows_out + SPT_WAVES * 4 * R - 1) / (SPT_WAVES * 4 * R)), (unsigned)n_angles,
                  (unsigned)nsplit);
  size_t lds = (size_t)(kc + 1) * row * sizeof(float);
  if (out_ld) lds = std::max(lds, (size_t)64 * (SPT_WAVES * 4 * R + 1) * sizeof(float));
#define DFM_SPT(RR, YY)                                                                                      \
  launch_spmm_t<RR, YY>(grid, lds, st, in, row_ptr, col, val, out, omegas, my, ys, ncols, nrows, rows_out,  \
                        compact, alpha, cspan, kc, n_angles, in_ld, out_ld, ys_out)
#define DFM_SPT_R(YY, RMAX)                                   \
  if (R == RMAX) DFM_SPT(RMAX, YY);                           \
  else if (R == 2) DFM_SPT(2, YY);                            \
  else DFM_SPT(1, YY)
  switch (nb) {
    case 1: DFM_SPT_R(1, 4); break;
    case 2: DFM_SPT_R(2, 4); break;
    case 3: DFM_SPT_R(3, 2); break;
    case 4: DFM_SPT_R(4, 2); break;
    case 5: DFM_SPT_R(5, 2); break;
    case 6: DFM_SPT_R(6, 2); break;
    case 7: DFM_SPT_R(7, 2); break;
    default: DFM_SPT_R(8, 2); break;
  }
#undef DFM_SPT_R
#undef DFM_SPT
  return DFM_OK;
}

}  // namespace

extern "C" {

int dfm_spmm_t_rows_per_block(int32_t my) {
  if (my <= 0 || my > 512) return 0;
  return SPT_WAVES * 4 * row_quads(my);
}

int dfm_spmm_t(const float* inT, const int32_t* row_ptr, const uint16_t* col, const float* val, float* outT,
               const int32_t* omegas, int32_t n_angles, int32_t my, int32_t ys, int32_t ncols, int32_t nrows,
               int32_t rows_out, int32_t compact, float alpha, int32_t nsplit, int32_t kc, dfm_stream_t stream) {
  DFM_CHECK_ARG(inT && row_ptr && col && val && outT, "dfm_spmm_t: null pointer");
  DFM_CHECK_ARG(n_angles >= 0 && my > 0 && my <= 512 && ys >= my && ys % 4 == 0 && ncols > 0 && ncols <= 65536 &&
                    nrows >= 0 && rows_out >= nrows && nsplit >= 1 && nsplit <= ncols && n_angles <= 65535,
                "dfm_spmm_t: bad sizes (my %d ys %d ncols %d nrows %d rows_out %d nsplit %d)", my, ys, ncols, nrows,
                rows_out, nsplit);
  if (((uintptr_t)inT) % 16) {
    dfm::set_error("dfm_spmm_t: the transposed operand must be 16-byte aligned");
    return DFM_ERR_ARG;
  }
  spmm_t_impl(inT, 0, row_ptr, col, val, outT, 0, ys, omegas, n_angles, my, ys, ncols, nrows, rows_out, compact,
              alpha, nsplit, kc, (hipStream_t)stream);
  DFM_LAUNCH_CHECK("dfm_spmm_t");
  return DFM_OK;
}

int dfm_spmm_t_direct(const float* in, int64_t in_ld, int32_t in_ys, const int32_t* row_ptr, const uint16_t* col,
                      const float* val, float* out, int64_t out_ld, int32_t out_ys, const int32_t* omegas,
                      int32_t n_angles, int32_t my, int32_t ncols, int32_t nrows, int32_t rows_out, int32_t compact,
                      float alpha, int32_t nsplit, int32_t kc, dfm_stream_t stream) {
  DFM_CHECK_ARG(in && row_ptr && col && val && out, "dfm_spmm_t_direct: null pointer");
  DFM_CHECK_ARG(n_angles >= 0 && my > 0 && my <= 512 && ncols > 0 && ncols <= 65536 && nrows >= 0 &&
                    rows_out >= nrows && nsplit >= 1 && nsplit <= ncols && n_angles <= 65535 &&
                    (in_ld ? in_ld >= ncols : (in_ys >= my && in_ys % 4 == 0)) &&
                    (out_ld ? (out_ld >= rows_out && nsplit == 1) : out_ys >= my),
                "dfm_spmm_t_direct: bad sizes (my %d ncols %d nrows %d rows_out %d nsplit %d in_ld %lld in_ys %d "
                "out_ld %lld out_ys %d)", my, ncols, nrows, rows_out, nsplit, (long long)in_ld, in_ys,
                (long long)out_ld, out_ys);
  if (((uintptr_t)in) % 16 || in_ld % 4) {
    dfm::set_error("dfm_spmm_t_direct: the input must be 16-byte aligned, in_ld a multiple of 4");
    return DFM_ERR_ARG;
  }
  spmm_t_impl(in, in_ld, row_ptr, col, val, out, out_ld, out_ys, omegas, n_angles, my, in_ys, ncols, nrows, rows_out,
              compact, alpha, nsplit, kc, (hipStream_t)stream);
  DFM_LAUNCH_CHECK("dfm_spmm_t_direct");
  return DFM_OK;
}

int dfm_transpose_sum(const float* in, float* out, const int32_t* omegas, int32_t omega_out, int32_t n_mat,
                      int32_t nr, int32_t nc, int64_t in_ld, int64_t in_mat, int64_t out_ld, int64_t out_mat,
                      int32_t nsplit, int64_t split_stride, int32_t accumulate, dfm_stream_t stream) {
  DFM_CHECK_ARG(in && out && n_mat >= 0 && n_mat <= 65535 && nr > 0 && nc > 0 && in_ld >= nc && out_ld >= nr &&
                    nsplit >= 1 && (nr + 31) / 32 <= 65535,
                "dfm_transpose_sum: bad arguments");
  if (n_mat == 0) return DFM_OK;
  const dim3 grid((unsigned)((nc + 31) / 32), (unsigned)((nr + 31) / 32), (unsigned)n_mat);
  hipLaunchKernelGGL(transpose_sum_kernel, grid, dim3(256), 0, (hipStream_t)stream, in, out, omegas, omega_out, nr,
                     nc, in_ld, in_mat, out_ld, out_mat, nsplit, split_stride, accumulate);
  DFM_LAUNCH_CHECK("dfm_transpose_sum");
  return DFM_OK;
}

}  // extern "C"
