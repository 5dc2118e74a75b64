// Split operands (sp16): fp32 matrices as two fp16 planes for the fp16 MFMA.
//
// Whoever makes the planes picks power-of-two scales (exact) so that the
// largest value of each row, column or matrix lands in 2^13 .. 2^14; the
// product's epilogue takes them out again with ldexp. The fp16 range below
// that is 2^38 wide (subnormals included: the MFMA keeps them), so what a
// value loses against its fp32 form is below 2^-39 of the largest value that
// shares its scale, or 2^-23 of itself, whichever is larger.
#pragma once

#include "aux_kernels.h"
#include "gemm_nt.h"

namespace pto {

// Exponent e with max·2^e in (2^13, 2^14] for a bound max > 0 (0 for zero,
// infinite and NaN bounds; non-finite operands never reach the products that
// read planes, or are meant to come out as NaN).
constexpr int kSplitTop = 14;
__device__ __forceinline__ int split_exp(float bound) {
  int k = 0;
  if (!(bound > 0.f) || bound > 3.0e38f * 2.f) return 0;
  (void)frexpf(bound, &k);  // bound <= 2^k
  return kSplitTop - k;
}

// Eight values as the two planes: h = fp16(v), l = fp16(v - h).
struct Split8 {
  uint4 h, l;
};
__device__ __forceinline__ Split8 split8(const float* v) {
  Split8 s;
  _Float16* h = reinterpret_cast<_Float16*>(&s.h);
  _Float16* l = reinterpret_cast<_Float16*>(&s.l);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    h[k] = static_cast<_Float16>(v[k]);
    l[k] = static_cast<_Float16>(v[k] - static_cast<float>(h[k]));
  }
  return s;
}

// p[k] and p[pl + k] = the planes of in[k] for k in [kbeg, n)
__device__ __forceinline__ void st8_split(sp16* p, int64_t pl, const float* in, int kbeg, int n) {
  const Split8 s = split8(in);
  if (full_run(kbeg, n)) {
    st16(p, s.h);
    st16(p + pl, s.l);
  } else {
    const sp16* h = reinterpret_cast<const sp16*>(&s.h);
    const sp16* l = reinterpret_cast<const sp16*>(&s.l);
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (k >= kbeg && k < n) {
        p[k] = h[k];
        p[pl + k] = l[k];
      }
  }
}

// Split planes of a fp32 matrix: out (h plane [orows][ld], l plane pl
// elements on) = planes of in(r, c)·scale_b·2^e, pads (columns to ld, rows to
// orows) zero. e = e_mat[b * e_mat_stride] (per matrix).
// Each thread takes eight consecutive output columns: 32 bytes in, 16 + 16
// out. Bound by memory: 8 bytes per element.
static __global__ void __launch_bounds__(256) split_pack_kernel(const float* __restrict__ in, int64_t rows, int64_t cols,
                                                         int64_t ld_in, int64_t s_in, const float* __restrict__ scale,
                                                         const int* __restrict__ e_mat, int e_mat_stride,
                                                         sp16* __restrict__ out, int64_t pl, int64_t orows, int64_t ld,
                                                         int64_t s_out) {
  const int b = blockIdx.y;
  const float* ib = in + (int64_t)b * s_in;
  sp16* ob = out + (int64_t)b * s_out;
  const float sc = scale ? scale[b] : 1.f;
  const int e = e_mat[(int64_t)b * e_mat_stride];
  const int64_t nch = ld / 8, total = orows * nch;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total; i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / nch, c0 = (i - r * nch) * 8;
    float v[8];
    if (r < rows && c0 + 8 <= cols) {
      const uint4 u0 = ld16(ib + r * ld_in + c0), u1 = ld16(ib + r * ld_in + c0 + 4);
      const unsigned w[8] = {u0.x, u0.y, u0.z, u0.w, u1.x, u1.y, u1.z, u1.w};
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = ldexpf(__uint_as_float(w[k]) * sc, e);
    } else {
#pragma unroll
      for (int k = 0; k < 8; ++k)
        v[k] = r < rows && c0 + k < cols ? ldexpf(ib[r * ld_in + c0 + k] * sc, e) : 0.f;
    }
    const Split8 s = split8(v);
    *reinterpret_cast<uint4*>(ob + r * ld + c0) = s.h;
    *reinterpret_cast<uint4*>(ob + pl + r * ld + c0) = s.l;
  }
}

// The planes of the transpose: out [orows][ld], out(c, r) = in(r, c)·scale_b·2^e,
// through a 64 x 64 LDS tile (65-word rows: both its accesses spread over the
// banks).
static __global__ void __launch_bounds__(256) split_pack_t_kernel(const float* __restrict__ in, int64_t rows, int64_t cols,
                                                           int64_t ld_in, int64_t s_in, const float* __restrict__ scale,
                                                           const int* __restrict__ e_mat, int e_mat_stride,
                                                           sp16* __restrict__ out, int64_t pl, int64_t orows,
                                                           int64_t ld, int64_t s_out) {
  __shared__ float tile[64][65];
  const int b = blockIdx.z;
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  const float* ib = in + (int64_t)b * s_in;
  sp16* ob = out + (int64_t)b * s_out;
  const float sc = scale ? scale[b] : 1.f;
  const int e = e_mat[(int64_t)b * e_mat_stride];
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll 8
  for (int rr = ty; rr < 64; rr += 4) {
    const int64_t r = r0 + rr, c = c0 + tx;
    tile[rr][tx] = r < rows && c < cols ? ldexpf(ib[r * ld_in + c] * sc, e) : 0.f;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < 64 * 8; q += 256) {
    const int cc = q / 8, rr = (q % 8) * 8;  // output row c0 + cc, columns r0 + rr ..
    const int64_t c = c0 + cc, r = r0 + rr;
    if (c >= orows || r >= ld) continue;
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = tile[rr + k][cc];
    const Split8 s = split8(v);
    *reinterpret_cast<uint4*>(ob + c * ld + r) = s.h;
    *reinterpret_cast<uint4*>(ob + pl + c * ld + r) = s.l;
  }
}

// Zero the pads of up to kPadBufs batched [rows][ld] buffers in one launch:
// columns [cols, ld) of rows [0, rows) and all of rows [rows, prows).
// Elements of two bytes; cols is any, ld even pitches.
constexpr int kPadBufs = 8;
struct PadList {
  struct Buf {
    uint16_t* p;
    int64_t rows, prows, cols, ld, stride;
    int batch;
  } buf[kPadBufs];
  int n = 0;
  void add(void* p, int64_t rows, int64_t prows, int64_t cols, int64_t ld, int64_t stride, int batch) {
    if (prows == rows && cols == ld) return;
    buf[n++] = Buf{static_cast<uint16_t*>(p), rows, prows, cols, ld, stride, batch};
  }
};
static __global__ void __launch_bounds__(256) zero_pads_kernel(PadList l) {
  const PadList::Buf f = l.buf[blockIdx.y];
  const int64_t w = f.ld - f.cols, side = f.rows * w, total = side + (f.prows - f.rows) * f.ld;
  for (int b = blockIdx.z; b < f.batch; b += gridDim.z) {
    uint16_t* p = f.p + (int64_t)b * f.stride;
    for (int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x; e < total; e += (int64_t)gridDim.x * 256) {
      if (e < side) {
        const int64_t r = e / w;
        p[r * f.ld + f.cols + (e - r * w)] = 0;
      } else {
        p[f.rows * f.ld + (e - side)] = 0;
      }
    }
  }
}
inline int launch_zero_pads(const PadList& l, hipStream_t stream) {
  if (l.n == 0) return 0;
  int64_t most = 1;
  int batch = 1;
  for (int i = 0; i < l.n; ++i) {
    const PadList::Buf& f = l.buf[i];
    most = std::max<int64_t>(most, f.rows * (f.ld - f.cols) + (f.prows - f.rows) * f.ld);
    batch = std::max(batch, f.batch);
  }
  const unsigned gx = (unsigned)std::min<int64_t>((most + 1023) / 1024, 256);
  hipLaunchKernelGGL(zero_pads_kernel, dim3(gx, (unsigned)l.n, (unsigned)std::min(batch, 64)), dim3(256), 0, stream, l);
  PTO_LAUNCHED("zero_pads");
  return 0;
}

}  // namespace pto
