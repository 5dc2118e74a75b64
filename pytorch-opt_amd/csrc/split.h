// Split operands (sp16): fp32 matrices as two fp16 planes for the fp16 MFMA, the
// products h·h + h·l + l·h in fp32 accumulators (Markidis, Der Chien, Laure, Peng
// and Vetter, IPDPS workshops 2018; Ootomo and Yokota, IJHPCA 2022).
//
// Whoever makes the planes picks power-of-two scales (exact); the product's
// epilogue takes them out again with ldexp. Two kinds:
//   * measured (factor updates, Grams, two-sided products): the largest value of
//     each row, or column, lands in [2^13, 2^14);
//   * from an a-priori bound (NS5): the bound does, the values lie below it by as
//     much as the bound is wide, 2^7 to 2^11 for an ordinary X.
// h has 11 significant bits and l 11 of what is left, down to fp16's smallest
// step of 2^-24 (the MFMA keeps subnormals). So a value is off by at most 2^-22 of
// itself, or by half that step, 2^-38 of a row's largest value (2^-39 of what it
// is scaled to), whichever is larger, and the product left out, l·l, is at most
// 2^-22 of h·h. What is smaller than 2^-16 of its row's largest value is held to
// fewer than 22 bits; what that means for each path:
//   * factor updates and Grams: an entry (i, j) is right to about 2^-22 of
//     |g_i|·|g_j| (the geometric mean of the two diagonal entries), not of the sum
//     of the |g_ik·g_jk|, which can be far smaller where two rows hold their large
//     values at different k;
//   * two-sided products: a row or column that is small as a whole keeps its bits
//     (apply.hip); an entry that is below 2^-16 of its row's and of its column's
//     largest value is held to 2^-38 of them;
//   * NS5: matrices with a row or column so small that this would show run the
//     fp32 chain (ns5.hip).
#pragma once

#include "aux_kernels.h"
#include "gemm_nt.h"

namespace pto {

// Exponent e with max·2^e in [2^13, 2^14) for a finite bound max > 0. Non-finite
// operands never reach the products that read these planes; an empty row or
// column has kSplitZero, which makes a zero of whatever another operand holds
// against it.
constexpr int kSplitTop = 14, kSplitZero = 1000;
__device__ __forceinline__ int split_exp(float bound) {
  int k = 0;
  if (bound == 0.f) return kSplitZero;
  if (!(bound < INFINITY)) return 0;
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
__device__ __forceinline__ void st8_planes(sp16* p, int64_t pl, const float* in, int kbeg, int n) {
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

// Elements o + k of a matrix held at m as planes, or as fp32 in their place
__device__ __forceinline__ void st8_split(sp16* m, int64_t o, int64_t pl, const float* in, int kbeg, int n, bool plain) {
  if (plain)
    st8<float, float>(reinterpret_cast<float*>(m) + o, in, kbeg, n);
  else
    st8_planes(m + o, pl, in, kbeg, n);
}

// Split planes of a fp32 matrix: out (h plane [orows][ld], l plane pl
// elements on) = planes of in(r, c)·scale_b·2^e, pads (columns to ld, rows to
// orows) zero. e = e_mat[b * e_mat_stride] (per matrix). A matrix with
// plain[b * e_mat_stride] != 0 is stored as fp32 in the place of its planes.
// Each thread takes eight consecutive output columns: 32 bytes in, 16 + 16
// out. Bound by memory: 8 bytes per element.
[[maybe_unused]] static __global__ void __launch_bounds__(256) split_pack_kernel(const float* __restrict__ in, int64_t rows, int64_t cols,
                                                         int64_t ld_in, int64_t s_in, const float* __restrict__ scale,
                                                         const int* __restrict__ e_mat, int e_mat_stride,
                                                         const int* __restrict__ plain, sp16* __restrict__ out,
                                                         int64_t pl, int64_t orows, int64_t ld, int64_t s_out) {
  const int b = blockIdx.y;
  const float* ib = in + (int64_t)b * s_in;
  sp16* ob = out + (int64_t)b * s_out;
  const float sc = scale ? scale[b] : 1.f;
  const bool as_is = plain[(int64_t)b * e_mat_stride] != 0;
  const int e = as_is ? 0 : e_mat[(int64_t)b * e_mat_stride];
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
    if (as_is) {
      st8<float, float>(reinterpret_cast<float*>(ob) + r * ld + c0, v, 0, 8);
      continue;
    }
    const Split8 s = split8(v);
    *reinterpret_cast<uint4*>(ob + r * ld + c0) = s.h;
    *reinterpret_cast<uint4*>(ob + pl + r * ld + c0) = s.l;
  }
}

// The planes of the transpose: out [orows][ld], out(c, r) = in(r, c)·scale_b·2^e,
// through a 64 x 64 LDS tile (65-word rows: both its accesses spread over the
// banks).
[[maybe_unused]] static __global__ void __launch_bounds__(256) split_pack_t_kernel(const float* __restrict__ in, int64_t rows, int64_t cols,
                                                           int64_t ld_in, int64_t s_in, const float* __restrict__ scale,
                                                           const int* __restrict__ e_mat, int e_mat_stride,
                                                           const int* __restrict__ plain, sp16* __restrict__ out,
                                                           int64_t pl, int64_t orows, int64_t ld, int64_t s_out) {
  __shared__ float tile[64][65];
  const int b = blockIdx.z;
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  const float* ib = in + (int64_t)b * s_in;
  sp16* ob = out + (int64_t)b * s_out;
  const float sc = scale ? scale[b] : 1.f;
  const bool as_is = plain[(int64_t)b * e_mat_stride] != 0;
  const int e = as_is ? 0 : e_mat[(int64_t)b * e_mat_stride];
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int rr = ty + 4 * i;
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
    if (as_is) {
      st8<float, float>(reinterpret_cast<float*>(ob) + c * ld + r, v, 0, 8);
      continue;
    }
    const Split8 s = split8(v);
    *reinterpret_cast<uint4*>(ob + c * ld + r) = s.h;
    *reinterpret_cast<uint4*>(ob + pl + c * ld + r) = s.l;
  }
}

constexpr unsigned kInfBits = 0x7f800000u;
constexpr unsigned kTinyBits = 0x0d800000u;  // 2^-100

// Planes of a fp32 matrix in either or both layouts:
//   out_s [rows][ld_s]: in(r, c)·2^(er(r) + pre), out_t [cols + ones][ld_t]:
//   in(r, c)·2^(ec(c) + pre) transposed (with `ones`, a last row of ones),
// pad columns zero, er and ec the split exponents of the maxima of
// in(r, c)·2^pre, which are stored too (batch strides mw, nw; er plus er_add's).
// pre = pre_off + pre_mul·(pre_r(r) or pre_c(c)): the scales that another
// operand's rows carry, taken out of this one. A row or column with a
// non-finite value, or whose maximum 2^pre takes to the ends of the fp32 range,
// sets bad[b].
struct SplitPack {
  const float* in;
  int64_t rows, cols, ld_in, s_in;
  unsigned* rpart;
  unsigned* cpart;
  int64_t mw, nw;
  int* er;
  int* ec;
  int* bad;
  sp16* out_s;
  int64_t pl_s, ld_s, s_s;
  sp16* out_t;
  int64_t pl_t, ld_t, s_t;
  int ones;
  const int* pre_r = nullptr;
  const int* pre_c = nullptr;
  int64_t s_pre = 0;
  int pre_mul = 0, pre_off = 0;
  const int* er_add = nullptr;  // stride mw
  int bad_stride = 1;
  __device__ __forceinline__ int pre(const int* p, int b, int64_t at, int64_t n) const {
    return p && at < n ? pre_off + pre_mul * p[(int64_t)b * s_pre + at] : 0;
  }
};

// |x|·2^e by bit patterns: what is not finite and what is not zero stay so,
// but for the rows of an empty one (|e| near kSplitZero).
__device__ __forceinline__ unsigned scaled_bits(unsigned u, int e) {
  if (u >= kInfBits || u == 0) return u;
  if (e < -kSplitZero / 2) return 0;
  return max(1u, __float_as_uint(ldexpf(__uint_as_float(u), e)));
}

// Largest |x| of the parts of a fp32 matrix's rows and columns, as bit patterns
// (which order like the values, NaN above infinity): rpart[cb][r] of columns
// 256·cb .. + 255, cpart[rb][c] of rows nr·rb .. + nr - 1; either may be null. A
// workgroup takes nr rows (a multiple of 32) x 256 columns, a wave
// eight rows at a time, 16 bytes per lane and all eight in flight (one row at a
// time waited 32 times for memory: 30 us whatever the size). Parts need neither
// zeroing nor atomics. Bound by memory: 4 bytes per element. clear: also clears
// bad[b]. SUM: also partial[b·kRedBlocks + workgroup] = the sum of its squares, in
// fp64 (a read of its own and a launch were 5 us of a 768² NS5's 195).
template <bool SUM>
__global__ void __launch_bounds__(256) absmax_kernel(SplitPack a, int nr, int clear, double* __restrict__ partial) {
  __shared__ unsigned cw[4][256];
  const int b = blockIdx.z, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t r0 = (int64_t)blockIdx.y * nr, c0 = (int64_t)blockIdx.x * 256 + lane * 4;
  const float* ib = a.in + (int64_t)b * a.s_in;
  if (clear && blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) a.bad[(int64_t)b * a.bad_stride] = 0;
  int pc[4] = {0, 0, 0, 0};
#pragma unroll
  for (int k = 0; k < 4; ++k) pc[k] = a.pre(a.pre_c, b, c0 + k, a.cols);
  unsigned cm[4] = {0, 0, 0, 0};
  double sum = 0.0;
  for (int rr = wave * 8; rr < nr; rr += 32) {
    uint4 q[8];
    unsigned rm[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int64_t r = r0 + rr + i;
      q[i] = make_uint4(0, 0, 0, 0);
      if (r < a.rows) {
        if (c0 + 4 <= a.cols) {
          q[i] = ld16(ib + r * a.ld_in + c0);
        } else {
          if (c0 < a.cols) q[i].x = __float_as_uint(ib[r * a.ld_in + c0]);
          if (c0 + 1 < a.cols) q[i].y = __float_as_uint(ib[r * a.ld_in + c0 + 1]);
          if (c0 + 2 < a.cols) q[i].z = __float_as_uint(ib[r * a.ld_in + c0 + 2]);
        }
      }
    }
    if constexpr (SUM) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const unsigned w[4] = {q[i].x, q[i].y, q[i].z, q[i].w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const double d = __uint_as_float(w[k]);
          sum += d * d;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      unsigned u[4] = {q[i].x & 0x7fffffffu, q[i].y & 0x7fffffffu, q[i].z & 0x7fffffffu, q[i].w & 0x7fffffffu};
      if (a.pre_r || a.pre_c) {
        const int pr = a.pre(a.pre_r, b, r0 + rr + i, a.rows);
#pragma unroll
        for (int k = 0; k < 4; ++k) u[k] = scaled_bits(u[k], pr + pc[k]);
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) cm[k] = max(cm[k], u[k]);
      rm[i] = max(max(u[0], u[1]), max(u[2], u[3]));
    }
    if (a.rpart) {
      // eight rows over 64 lanes: three exchanges that halve the rows a lane
      // holds, three more within its eight lanes (10 shuffles for 48)
      unsigned m4[4], m2[2];
      const bool b5 = lane & 32, b4 = lane & 16, b3 = lane & 8;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        m4[i] = max(b5 ? rm[i + 4] : rm[i], (unsigned)__shfl_xor((int)(b5 ? rm[i] : rm[i + 4]), 32, 64));
#pragma unroll
      for (int i = 0; i < 2; ++i)
        m2[i] = max(b4 ? m4[i + 2] : m4[i], (unsigned)__shfl_xor((int)(b4 ? m4[i] : m4[i + 2]), 16, 64));
      unsigned m = max(b3 ? m2[1] : m2[0], (unsigned)__shfl_xor((int)(b3 ? m2[0] : m2[1]), 8, 64));
#pragma unroll
      for (int off = 4; off > 0; off >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, off, 64));
      const int64_t r = r0 + rr + 4 * b5 + 2 * b4 + b3;
      if ((lane & 7) == 0 && r < a.rows) a.rpart[((int64_t)b * gridDim.x + blockIdx.x) * a.mw + r] = m;
    }
  }
  if constexpr (SUM) {
    __shared__ double sw[4];
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, 64);
    if (lane == 0) sw[wave] = sum;
    __syncthreads();
    if (threadIdx.x == 0)
      partial[(int64_t)b * kRedBlocks + blockIdx.y * gridDim.x + blockIdx.x] = (sw[0] + sw[1]) + (sw[2] + sw[3]);
  }
  if (!a.cpart) return;
#pragma unroll
  for (int k = 0; k < 4; ++k) cw[wave][lane * 4 + k] = cm[k];
  __syncthreads();
  const int64_t c = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (c < a.cols)
    a.cpart[((int64_t)b * gridDim.y + blockIdx.y) * a.nw + c] =
        max(max(cw[0][threadIdx.x], cw[1][threadIdx.x]), max(cw[2][threadIdx.x], cw[3][threadIdx.x]));
}
// Parts of a matrix: row parts per 256 columns; column parts per 64 rows (256
// rows a workgroup ran 4096² at 53 us for 15.5, one workgroup per CU), and at
// most 64 of them, since every tile of the packing pass reads all of its
// columns' parts.
inline int absmax_rows(int64_t rows) { return rows <= 4096 ? 64 : (int)round_up((rows + 63) / 64, 32); }
inline int64_t absmax_row_parts(int64_t cols) { return (cols + 255) / 256; }
inline int64_t absmax_col_parts(int64_t rows) { return (rows + absmax_rows(rows) - 1) / absmax_rows(rows); }

[[maybe_unused]] static __global__ void __launch_bounds__(256) split_pack_max_kernel(SplitPack a, int row_parts, int col_parts) {
  __shared__ float tile[64][65];
  __shared__ unsigned mx[4][64];
  __shared__ int xr[64], xc[64], pr[64], pc[64];
  const int b = blockIdx.z;
  const int64_t r0 = (int64_t)blockIdx.y * 64, c0 = (int64_t)blockIdx.x * 64;
  const float* ib = a.in + (int64_t)b * a.s_in;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const int rr = ty + 4 * i;
    const int64_t r = r0 + rr, c = c0 + tx;
    float x = a.ones && r < a.rows && c == a.cols ? 1.f : 0.f;
    if (r < a.rows && c < a.cols) x = ib[r * a.ld_in + c];
    tile[rr][tx] = x;
  }
  if (ty == 0) pr[tx] = a.pre(a.pre_r, b, r0 + tx, a.rows);
  if (ty == 1) pc[tx] = a.pre(a.pre_c, b, c0 + tx, a.cols);
  // the tile's exponents: waves 0, 1 its rows' parts, waves 2, 3 its columns'
  {
    const bool row = ty < 2;
    const int64_t at = row ? r0 + tx : c0 + tx, n = row ? a.rows : a.cols, w = row ? a.mw : a.nw;
    const unsigned* p = row ? a.rpart : a.cpart;
    const int parts = row ? row_parts : col_parts;
    unsigned m = 0;
    if (p && at < n)
      for (int i = ty & 1; i < parts; i += 2) m = max(m, p[((int64_t)b * parts + i) * w + at]);
    if (!row && a.ones && at == n) m = __float_as_uint(1.f);
    mx[ty][tx] = m;
  }
  __syncthreads();
  auto check = [&](unsigned u) {
    if (a.bad && (u >= kInfBits || ((a.pre_r || a.pre_c) && u != 0 && u < kTinyBits))) a.bad[(int64_t)b * a.bad_stride] = 1;
  };
  if (ty == 0 && a.out_s) {
    const unsigned u = max(mx[0][tx], mx[1][tx]);
    xr[tx] = split_exp(__uint_as_float(u));
    const int64_t at = (int64_t)b * a.mw + r0 + tx;
    if (blockIdx.x == 0 && r0 + tx < a.rows) a.er[at] = xr[tx] + (a.er_add ? a.er_add[at] : 0);
    check(u);
  } else if (ty == 1 && a.out_t) {
    const unsigned u = max(mx[2][tx], mx[3][tx]);
    xc[tx] = split_exp(__uint_as_float(u));
    if (blockIdx.y == 0 && c0 + tx < a.cols + a.ones) a.ec[(int64_t)b * a.nw + c0 + tx] = xc[tx];
    check(u);
  }
  __syncthreads();
  for (int q = threadIdx.x; q < 64 * 8; q += 256) {
    const int u = q / 8, w = (q % 8) * 8;
    float v[8];
    if (a.out_s && r0 + u < a.rows && c0 + w < a.ld_s) {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = c0 + w + k < a.cols ? ldexpf(tile[u][w + k], xr[u] + pr[u] + pc[w + k]) : 0.f;
      const Split8 s = split8(v);
      sp16* o = a.out_s + (int64_t)b * a.s_s + (r0 + u) * a.ld_s + c0 + w;
      *reinterpret_cast<uint4*>(o) = s.h;
      *reinterpret_cast<uint4*>(o + a.pl_s) = s.l;
    }
    if (a.out_t && c0 + u < a.cols + a.ones && r0 + w < a.ld_t) {
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = ldexpf(tile[w + k][u], xc[u] + pc[u] + pr[w + k]);
      const Split8 s = split8(v);
      sp16* o = a.out_t + (int64_t)b * a.s_t + (c0 + u) * a.ld_t + r0 + w;
      *reinterpret_cast<uint4*>(o) = s.h;
      *reinterpret_cast<uint4*>(o + a.pl_t) = s.l;
    }
  }
}
inline int launch_absmax(const SplitPack& a, int batch, hipStream_t stream, bool clear) {
  const dim3 gm((unsigned)absmax_row_parts(a.cols), (unsigned)absmax_col_parts(a.rows), (unsigned)batch);
  PTO_REQUIRE(gm.y < 65536 && batch < 65536, "absmax: grid too large");
  hipLaunchKernelGGL((absmax_kernel<false>), gm, dim3(256), 0, stream, a, absmax_rows(a.rows), clear ? 1 : 0,
                     (double*)nullptr);
  PTO_LAUNCHED("absmax");
  return 0;
}
inline int launch_split_pack_max(const SplitPack& a, int batch, hipStream_t stream, bool clear = true) {
  const int64_t rext = a.out_t ? std::max(a.rows, a.ld_t) : a.rows;
  const int64_t cext = std::max(a.cols + a.ones, a.out_s ? a.ld_s : 0);
  const dim3 gp((unsigned)((cext + 63) / 64), (unsigned)((rext + 63) / 64), (unsigned)batch);
  PTO_REQUIRE(gp.y < 65536, "split_pack: grid too large");
  if (launch_absmax(a, batch, stream, clear)) return -1;
  hipLaunchKernelGGL(split_pack_max_kernel, gp, dim3(256), 0, stream, a, (int)absmax_row_parts(a.cols),
                     (int)absmax_col_parts(a.rows));
  PTO_LAUNCHED("split_pack_max");
  return 0;
}

// Split exponents of the rows of a fp32 matrix: e[b·ew + r]. A wave takes a row,
// 16 bytes per lane and four runs in flight. Bound by memory: 4 bytes per
// element. Also clears bad[b].
[[maybe_unused]] static __global__ void __launch_bounds__(256) row_exp_kernel(const float* __restrict__ in, int64_t rows,
                                                                              int64_t cols, int64_t ld, int64_t s_in,
                                                                              int* __restrict__ e, int64_t ew,
                                                                              int* __restrict__ bad) {
  const int b = blockIdx.y, lane = threadIdx.x & 63;
  if (blockIdx.x == 0 && threadIdx.x == 0) bad[b] = 0;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const float* row = in + (int64_t)b * s_in + r * ld;
  unsigned m = 0;
#pragma unroll 4
  for (int64_t c = lane * 4; c + 4 <= cols; c += 256) {
    const uint4 u = ld16(row + c);
    m = max(max(m, u.x & 0x7fffffffu), max(max(u.y & 0x7fffffffu, u.z & 0x7fffffffu), u.w & 0x7fffffffu));
  }
  const int64_t t = cols / 4 * 4 + lane;
  if (t < cols) m = max(m, __float_as_uint(row[t]) & 0x7fffffffu);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, off, 64));
  if (lane == 0) e[(int64_t)b * ew + r] = split_exp(__uint_as_float(m));
}
inline int launch_row_exp(const float* in, int64_t rows, int64_t cols, int64_t ld, int64_t s_in, int batch, int* e,
                          int64_t ew, int* bad, hipStream_t stream) {
  hipLaunchKernelGGL(row_exp_kernel, dim3((unsigned)((rows + 3) / 4), (unsigned)batch), dim3(256), 0, stream, in, rows,
                     cols, ld, s_in, e, ew, bad);
  PTO_LAUNCHED("row_exp");
  return 0;
}

// Epilogue of a product of split operands: takes the rows' and columns' scales
// out (v·2^(off - er(i) - ec(j)); one ldexp, so no intermediate leaves the range of
// the result) and hands the value to In.
template <class In>
struct EpiDescale {
  typedef float S;
  In in;
  const int* er;
  const int* ec;
  int64_t s_r, s_c;
  int off = 0;  // both operands' planes together carry 2^(er + ec - off)
  typedef typename In::Pre Pre;
  typedef typename In::PreT PreT;
  static constexpr bool kVoIsV = true;  // the transposed pass takes the raw value and scales it itself
  __device__ __forceinline__ bool has_t() const { return false; }
  __device__ __forceinline__ void load(int b, int i, int j0, int kbeg, int n, Pre& p, bool) const {
    in.load(b, i, j0, kbeg, n, p);
  }
  __device__ __forceinline__ void load_t(int b, int j, int i0, int n, PreT& p, bool) const {
    in.load_t(b, j, i0, n, p);
  }
  __device__ __forceinline__ void scaled(int b, int i, int j0, const S* v, int n, S* w, bool plain) const {
    const int ei = er[(int64_t)b * s_r + i];
    const int* ej = ec + (int64_t)b * s_c + j0;
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = k < n ? (plain ? v[k] : ldexpf(v[k], off - ei - ej[k])) : 0.f;
  }
  __device__ __forceinline__ void put(int b, int i, int j0, const S* v, int kbeg, int n, const Pre& pre, S* vo,
                                      bool plain) const {
    S w[8], drop[8];
    scaled(b, i, j0, v, n, w, plain);
    in.put(b, i, j0, w, kbeg, n, pre, drop);
#pragma unroll
    for (int k = 0; k < 8; ++k) vo[k] = v[k];
  }
  // symmetric products only (er == ec)
  __device__ __forceinline__ void put_t(int b, int j, int i0, const S* v, int n, const PreT& pre, bool plain) const {
    S w[8];
    scaled(b, j, i0, v, n, w, plain);
    in.put_t(b, j, i0, w, n, pre);
  }
  __device__ __forceinline__ void finish(int) const {}
};

// Epilogue that stores the products of split operands in fp32 with their scales in.
struct EpiRaw {
  typedef float S;
  EpiStore<float, float> in;
  typedef NoPre Pre;
  typedef NoPre PreT;
  static constexpr bool kVoIsV = true;
  __device__ __forceinline__ bool has_t() const { return false; }
  __device__ __forceinline__ void load(int, int, int, int, int, Pre&, bool) const {}
  __device__ __forceinline__ void load_t(int, int, int, int, PreT&, bool) const {}
  __device__ __forceinline__ void put(int b, int i, int j0, const S* v, int kbeg, int n, const Pre& p, S* vo,
                                      bool) const {
    in.put(b, i, j0, v, kbeg, n, p, vo);
  }
  __device__ __forceinline__ void put_t(int, int, int, const S*, int, const PreT&, bool) const {}
  __device__ __forceinline__ void finish(int) const {}
};

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
[[maybe_unused]] static __global__ void __launch_bounds__(256) zero_pads_kernel(PadList l) {
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
