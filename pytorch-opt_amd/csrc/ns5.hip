// Quintic Newton–Schulz orthogonalization on gfx950.
//
// Replaces _NATIVE.newton_schulz_orthogonalize
// (pytorch_opt/ops/__init__.py:67-71, csrc/pytorch_opt_ops.cpp:65-81) with
// the same semantics as pytorch_opt/ops/reference.py:71-97:
//   X = G (work precision); if rows > cols, X = Xᵀ;  X /= (‖X‖_F + eps);
//   repeat `steps` times:  A = X·Xᵀ;  B = b·A + c·A·A;  X = a·X + B·X;
//   undo the transpose; cast back.
//
// Per iteration three MFMA launches, each with a fused epilogue:
//   1. A = X·Xᵀ                    symmetric: upper tiles only, mirrored store
//   2. B' = a·I + b·A + c·(A·A)    symmetric: upper tiles only, mirrored store
//   3. X' = B'·X  (= a·X + B·X)    full
// Folding a·X into the product as a·I on the diagonal of B' spares the
// update a read of X; the extra rounding is that of one bf16 store of
// a + B_ii, the same size as the rounding of a·X itself in a bf16 chain.
// Layouts: the gram reads X's K-contiguous rows on both sides ("NT"). In
// bf16 the square and the update read their operands from [K][·] arrays
// through transposing LDS loads (A and B' are symmetric, so each is its own
// transpose; X' = B'·X reads X as stored), so X is kept in one layout; the
// first iteration reads a caller's 128-aligned bf16 G in place, with the
// 1/(‖G‖+eps) scale applied in the gram's and update's epilogues. In fp32
// and fp64 the update reads a stored Xᵀ, which its epilogue writes beside
// X'. bf16 inputs keep X, A, B in bf16 between launches with fp32
// accumulation (short side 128 or more; smaller ones run the fp32 chain,
// see ns5_bf16); fp32 and fp64 inputs stay in their own precision
// (fp32 above the smallest sizes with its products on split operands, see
// ns5_split_run).
#include <algorithm>

#include "aux_kernels.h"
#include "gemm_nt.h"
#include "split.h"

namespace pto {

namespace {

// 1 / (sqrt(sum of partial squares) + eps), one block per matrix.
template <typename A>
__global__ void __launch_bounds__(256) ns_scale_kernel(const double* __restrict__ partial, double eps,
                                                       A* __restrict__ scale) {
  const double s = block_sum_partials(partial, blockIdx.x);
  if (threadIdx.x == 0) scale[blockIdx.x] = A(1) / (static_cast<A>(sqrt(s)) + static_cast<A>(eps));
}

// A = s²·v: the first gram reads the input itself when no pack is needed,
// so the 1/(‖G‖ + eps) scale lands here (SCALED; without it A = v). A choice at
// run time put a branch and a scalar load on every run of the epilogue, gram and
// update: bf16 4 x 768² 243.8 -> 240.0 us with kernels of their own.
template <typename T, typename A, bool SCALED = false>
struct EpiNsGram {
  typedef A S;
  T* dst;
  int64_t ld, sd;
  const A* scale;
  typedef NoPre Pre;
  typedef NoPre PreT;
  static constexpr bool kVoIsV = true;
  __device__ __forceinline__ bool has_t() const { return false; }
  __device__ __forceinline__ void load(int, int, int, int, int, Pre&) const {}
  __device__ __forceinline__ void load_t(int, int, int, int, PreT&) const {}
  __device__ __forceinline__ void store(T* p, int b, const S* v, int kbeg, int n) const {
    const S s2 = SCALED ? scale[b] * scale[b] : S(1);
    S w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = s2 * v[k];
    st8<T, S>(p, w, kbeg, n);
  }
  __device__ __forceinline__ void put(int b, int i, int j0, const S* v, int kbeg, int n, const Pre&, S* vo) const {
    store(dst + (int64_t)b * sd + (int64_t)i * ld + j0, b, v, kbeg, n);
#pragma unroll
    for (int k = 0; k < 8; ++k) vo[k] = v[k];
  }
  __device__ __forceinline__ void put_t(int b, int j, int i0, const S* v, int n, const PreT&) const {
    store(dst + (int64_t)b * sd + (int64_t)j * ld + i0, b, v, 0, n);
  }
  __device__ __forceinline__ void finish(int) const {}
};

// B' = a·I + b·A + c·v  (symmetric, so the mirror takes the same value)
template <typename T, typename A>
struct EpiNsSq {
  typedef A S;
  const T* Asrc;
  T* dst;
  int64_t ld, sd;
  A ac, bc, cc;
  typedef Raw8<T> Pre;
  typedef NoPre PreT;
  static constexpr bool kVoIsV = false;  // the mirror stores B', not the raw product
  __device__ __forceinline__ bool has_t() const { return false; }
  __device__ __forceinline__ void load(int b, int i, int j0, int kbeg, int n, Pre& p) const {
    ld8_pre<T>(Asrc + (int64_t)b * sd + (int64_t)i * ld + j0, p, kbeg, n);
  }
  __device__ __forceinline__ void load_t(int, int, int, int, PreT&) const {}
  __device__ __forceinline__ void put(int b, int i, int j0, const S* v, int kbeg, int n, const Pre& pre,
                                      S* vo) const {
    const int64_t o = (int64_t)b * sd + (int64_t)i * ld + j0;
    S a[8];
    ld8_use<T, S>(Asrc + o, pre, a, kbeg, n);
    // explicit fused multiply-adds fix the rounding, so it cannot depend on
    // how the compiler contracts this expression in a given build
#pragma unroll
    for (int k = 0; k < 8; ++k) vo[k] = fma(cc, v[k], fma(bc, a[k], i == j0 + k ? ac : A(0)));
    st8<T, S>(dst + o, vo, kbeg, n);
  }
  __device__ __forceinline__ void put_t(int b, int j, int i0, const S* v, int n, const PreT&) const {
    st8<T, S>(dst + (int64_t)b * sd + (int64_t)j * ld + i0, v, 0, n);
  }
  __device__ __forceinline__ void finish(int) const {}
};

// X' = s·v (s per matrix where SCALED: the first update of an unpacked input
// applies 1/(‖G‖ + eps) here), stored to dst (row-major)
// and/or dstT (transposed copy).
template <typename T, typename A, bool SCALED = false>
struct EpiNsUpdate {
  typedef A S;
  T* dst;
  int64_t ld_d, s_d;
  T* dstT;
  int64_t ld_t, s_t;
  const A* scale;
  typedef NoPre Pre;
  typedef NoPre PreT;
  static constexpr bool kVoIsV = true;
  __device__ __forceinline__ bool has_t() const { return dstT != nullptr; }
  __device__ __forceinline__ void load(int, int, int, int, int, Pre&) const {}
  __device__ __forceinline__ void load_t(int, int, int, int, PreT&) const {}
  __device__ __forceinline__ void store(T* p, int b, const S* v, int kbeg, int n) const {
    const S s = SCALED ? scale[b] : S(1);
    S w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = s * v[k];
    st8<T, S>(p, w, kbeg, n);
  }
  __device__ __forceinline__ void put(int b, int i, int j0, const S* v, int kbeg, int n, const Pre&, S* vo) const {
#pragma unroll
    for (int k = 0; k < 8; ++k) vo[k] = v[k];
    if (dst) store(dst + (int64_t)b * s_d + (int64_t)i * ld_d + j0, b, v, kbeg, n);
  }
  __device__ __forceinline__ void put_t(int b, int j, int i0, const S* v, int n, const PreT&) const {
    store(dstT + (int64_t)b * s_t + (int64_t)j * ld_t + i0, b, v, 0, n);
  }
  __device__ __forceinline__ void finish(int) const {}
};

template <typename T>
struct NsLayout {
  int64_t m, n, ldm, ldn;
  bool transposed;
};

// bf16 updates read X itself as the [K][N] operand of X' = B'·X (QN
// layout), ping-ponging between two X buffers with ldm rows whose pad rows
// are zero. fp32 and fp64 keep one X and a ping-pong pair of stored Xᵀ.
template <typename T>
constexpr bool ns5_qn() {
  return sizeof(T) == 2;
}

template <typename T>
size_t ns5_ws_bytes_t(int64_t batch, int64_t rows, int64_t cols) {
  int64_t m = std::min(rows, cols), n = std::max(rows, cols);
  int64_t ldm = round_up(m, kPadK), ldn = round_up(n, kPadK);
  size_t e = sizeof(T);
  size_t bytes = 0;
  auto add = [&](size_t b) { bytes = round_up(bytes, 256) + b; };
  typedef typename AccOf<T>::type A;
  add(sizeof(double) * kRedBlocks * batch);   // partial sums
  add(sizeof(A) * batch);                      // scales
  add(e * batch * ldm * ldm);                  // A (ldm rows: pad rows for the transposed read)
  add(e * batch * ldm * ldm);                  // B'
  if (ns5_qn<T>()) {
    add(e * batch * ldm * ldn);                // X ping
    add(e * batch * ldm * ldn);                // X pong
  } else {
    add(e * batch * m * ldn);                  // X
    add(e * batch * n * ldm);                  // Xᵀ ping
    add(e * batch * n * ldm);                  // Xᵀ pong
  }
  return bytes + 256;
}

// ------------------------------------------------ fp32 on split operands
//
// The fp32 chain with X, A and B' held as fp16 pairs (split.h) and its
// products on the fp16 MFMA. Their power-of-two scales come from bounds that
// need no data beyond the norm: ‖X_0‖₂ <= ‖X_0‖_F = ρ, every entry of a matrix
// is at most its spectral norm, and X' = p(X) on the singular values with
// p(s) = a·s + b·s³ + c·s⁵, so x_{t+1} = max |p| over [0, x_t] bounds X_{t+1}.
struct NsExp {
  int x, a, b, xn;  // planes hold X·2^x, A·2^a, B'·2^b; the next iterate's x
};
constexpr int kNsSplitSteps = 31;
struct NsMat {
  NsExp e[kNsSplitSteps];
  int plain;  // planes do not serve: the fp32 chain, in the same buffers
  int pad[3];
};
constexpr int kNsMatExp = sizeof(NsMat) / sizeof(NsExp), kNsMatInt = sizeof(NsMat) / sizeof(int);

// A matrix keeps the planes if the largest value of every row and column that is
// not empty is at least 2^-16 of ρ. Their scales follow ρ and the bounds x_t, so
// a value is held to about 2^-39 of ρ, and every step rounds so again. A row of a
// 1500² matrix at 2^-15.2 of ρ comes out 2.4e-6 off (3.6e-6 on the fp32 chain);
// at 2^-17 it would pass that, and one at 1e-8 of the others was 13% off. The
// rows of a random matrix lie at 2^-7 (512²) to 2^-11 (4096 x 11008). A unit that
// hardly fires makes a smaller one, and its matrix takes the fp32 chain (2048²
// 2.47 ms, against 0.70 on planes and 1.57 on the fp32 kernels; one of twelve
// 2048² 11.4 ms for all, against 5.3 and 16.4).
constexpr float kNsSpread = 1.f / 65536;

// x_{t+1}: max |p| over [0, x], with 1% for the products' rounding. |p| is largest
// at the end of the interval or where p' = a + 3b·s² + 5c·s⁴ = 0.
__host__ __device__ inline double ns_next_bound(double a, double b, double c, double x) {
  const double u = x * x;
  auto p = [&](double q) { return fabs(a + q * (b + q * c)) * sqrt(q); };  // q = s²
  double top = p(u);
  const double disc = 9.0 * b * b - 20.0 * a * c;
  if (c != 0.0 && disc >= 0.0) {
    for (int sg = -1; sg <= 1; sg += 2) {
      const double q = (-3.0 * b + sg * sqrt(disc)) / (10.0 * c);
      if (q > 0.0 && q < u) top = fmax(top, p(q));
    }
  } else if (c == 0.0 && b != 0.0) {
    const double q = -a / (3.0 * b);
    if (q > 0.0 && q < u) top = fmax(top, p(q));
  }
  return 1.01 * top;
}

// Coefficients that those bounds fit: they follow the largest singular value
// that could be there, and the planes hold what is down to 2^-39 of it, so the
// bound may not run away from the values that are. It stays at most 1.5 from
// x_0 = 1, small singular values do not shrink (a >= 1) and none shrinks below
// half in a step (q(s²) = p(s)/s >= 1/2 on [0, x_t]). The usual triple stays at
// 1.22 with q >= 0.64. With (4.1, -2.9, 0.55) the bound goes 2.0, 2.7, 30, 1e7, ...
// and five steps lost every bit of the result; such calls keep the fp32 chain.
inline bool ns_split_coeffs(int64_t steps, double a, double b, double c, double eps) {
  if (!(a >= 1.0) || !(eps >= 0.0) || steps < 1 || steps > kNsSplitSteps) return false;
  double x = 1.0;
  for (int64_t t = 0; t < steps; ++t) {
    const double u = x * x;
    auto q = [&](double v) { return a + v * (b + v * c); };
    double least = std::min(a, q(u));
    if (c != 0.0) {
      const double v = -b / (2.0 * c);
      if (v > 0.0 && v < u) least = std::min(least, q(v));
    }
    x = ns_next_bound(a, b, c, x);
    if (!(least >= 0.5) || !(x <= 1.5)) return false;
  }
  return true;
}

// Clamped to exponents that fp32 values (and so their bounds) have.
__device__ __forceinline__ int ns_exp(double bound) {
  int k = 0;
  if (!(bound > 0.0)) bound = 1.0;  // zero or NaN: any scale does
  (void)frexp(fmin(bound, 3e38), &k);
  return max(-120, min(120, kSplitTop - k));
}

// 1 / (‖G‖ + eps) as ns_scale_kernel gives it, the exponents of all steps and the
// choice of arithmetic, from the maxima of G's rows and columns (one thread each,
// over their parts).
__global__ void __launch_bounds__(256) ns_split_scale_kernel(const double* __restrict__ partial, double eps, int steps,
                                                             double a, double b, double c, SplitPack g, int row_parts,
                                                             int col_parts, int sums, float* __restrict__ scale,
                                                             NsMat* __restrict__ mat) {
  const int bm = blockIdx.y;
  const float norm = static_cast<float>(sqrt(block_sum_partials(partial, bm, sums)));
  const int64_t at = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const bool row = at < g.rows;
  if (row || at - g.rows < g.cols) {
    const int64_t i = row ? at : at - g.rows, w = row ? g.mw : g.nw;
    const int parts = row ? row_parts : col_parts;
    const unsigned* p = (row ? g.rpart : g.cpart) + (int64_t)bm * parts * w + i;
    unsigned m = 0;
#pragma unroll 8
    for (int k = 0; k < parts; ++k) m = max(m, p[k * w]);
    if (m >= kInfBits || (m != 0 && !(__uint_as_float(m) >= kNsSpread * norm))) mat[bm].plain = 1;
  }
  if (at != 0) return;
  const float sc = 1.f / (norm + static_cast<float>(eps));
  scale[bm] = sc;
  double x = (double)norm * sc;
  int ex = ns_exp(x);
  for (int t = 0; t < steps; ++t) {
    const double u = x * x;
    x = ns_next_bound(a, b, c, x);
    const int nxt = ns_exp(x);
    mat[bm].e[t] = NsExp{ex, ns_exp(u), ns_exp(fabs(a) + fabs(b) * u + fabs(c) * u * u), nxt};
    ex = nxt;
  }
}

// The exponents of matrix b in the step that ex points at
__device__ __forceinline__ NsExp ns_exps(const NsExp* ex, int b, bool plain) {
  return plain ? NsExp{0, 0, 0, 0} : ex[(int64_t)b * kNsMatExp];
}

// A = v·2^-2x, into its planes
struct EpiNsGramSplit {
  typedef float S;
  static constexpr bool kOwnPlain = true;
  sp16* dst;
  int64_t pl, ld, sd;
  const NsExp* ex;  // matrix b: ex[b * kNsMatExp]
  typedef NoPre Pre;
  typedef NoPre PreT;
  static constexpr bool kVoIsV = true;
  __device__ __forceinline__ bool has_t() const { return false; }
  __device__ __forceinline__ void load(int, int, int, int, int, Pre&, bool) const {}
  __device__ __forceinline__ void load_t(int, int, int, int, PreT&, bool) const {}
  __device__ __forceinline__ void store(int b, int64_t o, const S* v, int kbeg, int n, bool plain) const {
    const NsExp e = ns_exps(ex, b, plain);
    S w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = ldexpf(v[k], e.a - 2 * e.x);
    st8_split(dst + (int64_t)b * sd, o, pl, w, kbeg, n, plain);
  }
  __device__ __forceinline__ void put(int b, int i, int j0, const S* v, int kbeg, int n, const Pre&, S* vo,
                                      bool plain) const {
    store(b, (int64_t)i * ld + j0, v, kbeg, n, plain);
#pragma unroll
    for (int k = 0; k < 8; ++k) vo[k] = v[k];
  }
  __device__ __forceinline__ void put_t(int b, int j, int i0, const S* v, int n, const PreT&, bool plain) const {
    store(b, (int64_t)j * ld + i0, v, 0, n, plain);
  }
  __device__ __forceinline__ void finish(int) const {}
};

// B' = a·I + b·A + c·v·2^-2a
struct EpiNsSqSplit {
  typedef float S;
  static constexpr bool kOwnPlain = true;
  const sp16* Asrc;
  sp16* dst;
  int64_t pl, ld, sd;
  float ac, bc, cc;
  const NsExp* ex;
  struct Pre {
    uint4 h, l;  // plain: eight fp32 values
  };
  typedef NoPre PreT;
  static constexpr bool kVoIsV = false;  // the mirror stores B', not the raw product
  __device__ __forceinline__ bool has_t() const { return false; }
  __device__ __forceinline__ void load(int b, int i, int j0, int kbeg, int n, Pre& p, bool plain) const {
    if (full_run(kbeg, n)) {
      const int64_t o = (int64_t)i * ld + j0;
      const sp16* q = Asrc + (int64_t)b * sd + (plain ? 2 * o : o);
      p.h = ld16(q);
      p.l = ld16(q + (plain ? 8 : pl));
    }
  }
  __device__ __forceinline__ void load_t(int, int, int, int, PreT&, bool) const {}
  __device__ __forceinline__ void put(int b, int i, int j0, const S* v, int kbeg, int n, const Pre& pre, S* vo,
                                      bool plain) const {
    const NsExp e = ns_exps(ex, b, plain);
    const int64_t o = (int64_t)i * ld + j0;
    const sp16* A = Asrc + (int64_t)b * sd;
    S a[8];
    if (full_run(kbeg, n)) {
      const f16x8_t h = __builtin_bit_cast(f16x8_t, pre.h), l = __builtin_bit_cast(f16x8_t, pre.l);
      const unsigned u[8] = {pre.h.x, pre.h.y, pre.h.z, pre.h.w, pre.l.x, pre.l.y, pre.l.z, pre.l.w};
#pragma unroll
      for (int k = 0; k < 8; ++k)
        a[k] = plain ? __uint_as_float(u[k]) : static_cast<S>(h[k]) + static_cast<S>(l[k]);
    } else {
      for (int k = 0; k < 8; ++k)
        a[k] = k < kbeg || k >= n ? S(0)
               : plain            ? reinterpret_cast<const float*>(A)[o + k]
                                  : static_cast<S>(A[o + k].v) + static_cast<S>(A[o + pl + k].v);
    }
    S w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      vo[k] = fma(cc, ldexpf(v[k], -2 * e.a), fma(bc, ldexpf(a[k], -e.a), i == j0 + k ? ac : 0.f));
      w[k] = ldexpf(vo[k], e.b);
    }
    st8_split(dst + (int64_t)b * sd, o, pl, w, kbeg, n, plain);
  }
  __device__ __forceinline__ void put_t(int b, int j, int i0, const S* v, int n, const PreT&, bool plain) const {
    const NsExp e = ns_exps(ex, b, plain);
    S w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = ldexpf(v[k], e.b);
    st8_split(dst + (int64_t)b * sd, (int64_t)j * ld + i0, pl, w, 0, n, plain);
  }
  __device__ __forceinline__ void finish(int) const {}
};

// X' = v·2^-(b + x): into the next iterate's planes, or (last iteration) as
// fp32 into out, row-major (dst) or transposed (dstT).
struct EpiNsUpdateSplit {
  typedef float S;
  static constexpr bool kOwnPlain = false;
  sp16* planes;
  int64_t pl, ld, sd;
  float* dst;
  float* dstT;
  int64_t ld_o, s_o;
  const NsExp* ex;
  typedef NoPre Pre;
  typedef NoPre PreT;
  static constexpr bool kVoIsV = true;
  __device__ __forceinline__ bool has_t() const { return dstT != nullptr; }
  __device__ __forceinline__ void load(int, int, int, int, int, Pre&, bool) const {}
  __device__ __forceinline__ void load_t(int, int, int, int, PreT&, bool) const {}
  __device__ __forceinline__ void put(int b, int i, int j0, const S* v, int kbeg, int n, const Pre&, S* vo,
                                      bool plain) const {
    const NsExp e = ns_exps(ex, b, plain);
#pragma unroll
    for (int k = 0; k < 8; ++k) vo[k] = v[k];
    S w[8];
    if (planes) {
#pragma unroll
      for (int k = 0; k < 8; ++k) w[k] = ldexpf(v[k], e.xn - e.b - e.x);
      st8_split(planes + (int64_t)b * sd, (int64_t)i * ld + j0, pl, w, kbeg, n, plain);
    } else if (dst) {
#pragma unroll
      for (int k = 0; k < 8; ++k) w[k] = ldexpf(v[k], -e.b - e.x);
      st8<float, S>(dst + (int64_t)b * s_o + (int64_t)i * ld_o + j0, w, kbeg, n);
    }
  }
  __device__ __forceinline__ void put_t(int b, int j, int i0, const S* v, int n, const PreT&, bool plain) const {
    const NsExp e = ns_exps(ex, b, plain);
    S w[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) w[k] = ldexpf(v[k], -e.b - e.x);
    st8<float, S>(dstT + (int64_t)b * s_o + (int64_t)j * ld_o + i0, w, 0, n);
  }
  __device__ __forceinline__ void finish(int) const {}
};

size_t ns5_split_ws_bytes(int64_t batch, int64_t m, int64_t n) {
  const int64_t ldm = round_up(m, kPadK), ldn = round_up(n, kPadK);
  size_t bytes = 0;
  auto add = [&](size_t b) { bytes = round_up(bytes, 256) + b; };
  add(sizeof(double) * kRedBlocks * batch);
  add(sizeof(float) * batch);
  add(sizeof(NsMat) * batch);
  add(sizeof(sp16) * 2 * batch * ldm * ldm);  // A
  add(sizeof(sp16) * 2 * batch * ldm * ldm);  // B'
  add(sizeof(sp16) * 2 * batch * ldm * ldn);  // X ping
  add(sizeof(sp16) * 2 * batch * ldm * ldn);  // X pong
  return bytes + 256;
}

// Sizes that run on split operands: by one matrix alone, so that a matrix gets the
// same bits in every batch. Below a short side of 384 a single call has too few of
// the split products' 64² tiles and waits for their loads (256 x 4096 279 us
// against 229 on the fp32 MFMA's 32² tiles, 256² 116 against 106); from 512 on it
// is as fast or faster (512² the same, 768² 187 against 219, 2048² 0.70 ms against
// 1.57). Between, single calls lose (384² 132 us against 126, 384 x 1536 188
// against 165) and buckets, which is how Muon calls it, win (eight 384 x 1024 192
// against 293). Sides just above a multiple of 128, whose planes would not fit
// the workspace of the fp32 chain, keep that chain (a sum that grows with the
// batch on both sides alike).
constexpr int64_t kNsSplitMinSide = 384;
inline bool ns5_split(int64_t m, int64_t n, int64_t steps, double a, double b, double c, double eps) {
  return m >= kNsSplitMinSide && ns_split_coeffs(steps, a, b, c, eps) &&
         ns5_split_ws_bytes(1, m, n) <= ns5_ws_bytes_t<float>(1, m, n);
}

int ns5_split_run(const float* G, float* out, int64_t batch, int64_t rows, int64_t cols, int64_t steps, double a,
                  double b, double c, double eps, void* ws, size_t ws_bytes, hipStream_t stream) {
  const bool transposed = rows > cols;
  const int64_t m = std::min(rows, cols), n = std::max(rows, cols);
  const int64_t ldm = round_up(m, kPadK), ldn = round_up(n, kPadK);
  const int64_t plA = ldm * ldm, sA = 2 * plA, plX = ldm * ldn, sX = 2 * plX, sG = rows * cols;
  const int nb = (int)batch;
  Carver cv(ws, ws_bytes);
  double* partial = cv.take<double>(kRedBlocks * batch);
  float* scale = cv.take<float>(batch);
  NsMat* mat = cv.take<NsMat>(batch);
  sp16* Ab = cv.take<sp16>(batch * sA);
  sp16* Bb = cv.take<sp16>(batch * sA);
  sp16* X[2];
  for (sp16*& x : X) x = cv.take<sp16>(batch * sX);
  PTO_REQUIRE(!cv.overflow, "newton_schulz_orthogonalize: workspace too small");

  // ‖G‖ and the maxima of its rows and columns from one read, at most kRedBlocks
  // workgroups a matrix; the maxima's parts lie where the second iterate will
  const int64_t gx = absmax_row_parts(cols), gy = std::min((rows + 31) / 32, kRedBlocks / std::min<int64_t>(gx, kRedBlocks));
  const int nr = (int)round_up((rows + gy - 1) / gy, 32);
  const int64_t ny = (rows + nr - 1) / nr;
  SplitPack g{G, rows, cols, cols, sG};
  g.rpart = reinterpret_cast<unsigned*>(X[1]);
  g.cpart = g.rpart + batch * rows * gx;
  g.mw = rows;
  g.nw = cols;
  g.bad = &mat->plain;
  g.bad_stride = kNsMatInt;
  PTO_REQUIRE(4 * (rows * gx + cols * ny) <= (int64_t)sizeof(sp16) * sX, "newton_schulz_orthogonalize: workspace too small");
  const bool one_read = gx * ny <= kRedBlocks;
  const dim3 grid((unsigned)gx, (unsigned)ny, (unsigned)nb);
  if (one_read) {
    hipLaunchKernelGGL((absmax_kernel<true>), grid, dim3(256), 0, stream, g, nr, 1, partial);
  } else {
    if (launch_sumsq<float>(G, rows, cols, cols, sG, nb, partial, stream)) return -1;
    hipLaunchKernelGGL((absmax_kernel<false>), grid, dim3(256), 0, stream, g, nr, 1, partial);
  }
  PTO_LAUNCHED("absmax");
  hipLaunchKernelGGL(ns_split_scale_kernel, dim3((unsigned)((rows + cols + 255) / 256), (unsigned)nb), dim3(256), 0,
                     stream, partial, eps, (int)steps, a, b, c, g, (int)gx, (int)ny,
                     one_read ? (int)(gx * ny) : kRedBlocks, scale, mat);
  PTO_LAUNCHED("ns_split_scale");
  const int* ex0 = &mat->e[0].x;
  if (!transposed) {
    const unsigned gx = (unsigned)std::min<int64_t>((ldm * (ldn / 8) + 255) / 256, 4096);
    hipLaunchKernelGGL(split_pack_kernel, dim3(gx, (unsigned)nb), dim3(256), 0, stream, G, rows, cols, cols, sG, scale,
                       ex0, kNsMatInt, &mat->plain, X[0], plX, ldm, ldn, sX);
  } else {
    const dim3 grid((unsigned)(ldm / 64), (unsigned)(ldn / 64), (unsigned)nb);
    PTO_REQUIRE(grid.y < 65536, "newton_schulz_orthogonalize: shape too large");
    hipLaunchKernelGGL(split_pack_t_kernel, grid, dim3(256), 0, stream, G, rows, cols, cols, sG, scale, ex0, kNsMatInt,
                       &mat->plain, X[0], plX, ldm, ldn, sX);
  }
  PTO_LAUNCHED("split_pack");
  PadList pads;
  for (sp16* p : {Ab, Bb}) pads.add(p, m, ldm, m, ldm, plA, 2 * nb);
  if (steps > 1) pads.add(X[1], m, ldm, n, ldn, plX, 2 * nb);
  if (launch_zero_pads(pads, stream)) return -1;

  // the buffers of a plain matrix, as fp32 of the same extents
  auto rows_of = [](const sp16* p, int64_t ld, int64_t pl) {
    return PlainOperand{reinterpret_cast<const float*>(p), ld, 1, pl, -1};
  };
  auto args = [&](const sp16* P, int64_t ldp, int64_t plP, const sp16* Q, int64_t ldq, int64_t plQ, int64_t N, int64_t K) {
    return SplitArgs{{P, ldp, 2 * plP, Q, ldq, 2 * plQ, (int)m, (int)N, (int)round_up(K, kPadK)}, plP, plQ,
                     &mat->plain, kNsMatInt, rows_of(P, ldp, plP), rows_of(Q, ldq, plQ), (int)K};
  };
  for (int64_t t = 0; t < steps; ++t) {
    const bool last = t == steps - 1;
    const sp16* Xc = X[t & 1];
    const NsExp* ex = &mat->e[t];
    {
      EpiNsGramSplit e{Ab, plA, ldm, sA, ex};
      if (launch_gemm<sp16, true>(args(Xc, ldn, plX, Xc, ldn, plX, m, n), e, nb, stream, "ns5_gram")) return -1;
    }
    {
      const SplitArgs g = args(Ab, ldm, plA, Ab, ldm, plA, m, m);
      EpiNsSqSplit e{Ab, Bb, plA, ldm, sA, (float)a, (float)b, (float)c, ex};
      // A's rows are its columns: read K-contiguous by the 256² and 192² tiles
      // (12 x 2048²: 310 us against 325 with transposing reads), transposing
      // by the smaller ones, whose LDS reads bound them (128² 317 against 350)
      const int pick = pick_tile<sp16, true>(m, m, nb);
      if (pick == 1 || pick == 2) {
        if (launch_gemm<sp16, true>(g, e, nb, stream, "ns5_square")) return -1;
      } else if (launch_gemm_qn<EpiNsSqSplit, true, true, sp16>(g, e, nb, stream, "ns5_square", pick)) {
        return -1;
      }
    }
    {
      SplitArgs g = args(Bb, ldm, plA, Xc, ldn, plX, n, m);
      std::swap(g.fQ.row, g.fQ.k);  // X as [K][N]
      EpiNsUpdateSplit e{last ? nullptr : X[(t & 1) ^ 1], plX, ldn, sX, last && !transposed ? out : nullptr,
                         last && transposed ? out : nullptr, cols, sG, ex};
      if (launch_gemm_qn<EpiNsUpdateSplit, true, false, sp16>(g, e, nb, stream, "ns5_update")) return -1;
    }
  }
  return 0;
}

template <typename T>
int ns5_t(const T* G, T* out, int64_t batch, int64_t rows, int64_t cols, int64_t steps, double a, double b, double c,
          double eps, void* ws, size_t ws_bytes, hipStream_t stream) {
  typedef typename AccOf<T>::type A;
  const bool transposed = rows > cols;
  const int64_t m = std::min(rows, cols), n = std::max(rows, cols);
  const int64_t ldm = round_up(m, kPadK), ldn = round_up(n, kPadK);
  PTO_REQUIRE(m <= INT32_MAX && n <= INT32_MAX && batch <= 65535, "newton_schulz_orthogonalize: shape too large");
  if (batch == 0 || rows == 0 || cols == 0) return 0;

  // `out` may alias G exactly or not at all: every path below reads G only
  // in kernels that end before `out` is written, except the steps == 0
  // pack, which is tile-local (each element read before it is rewritten
  // in place) only when the two coincide.
  const int64_t sG = rows * cols;
  const uintptr_t g0 = reinterpret_cast<uintptr_t>(G), g1 = g0 + sizeof(T) * (uintptr_t)(batch * sG);
  const uintptr_t o0 = reinterpret_cast<uintptr_t>(out), o1 = o0 + sizeof(T) * (uintptr_t)(batch * sG);
  const bool aliased = g0 < o1 && o0 < g1;
  PTO_REQUIRE(!aliased || g0 == o0, "newton_schulz_orthogonalize: out partially overlaps G");

  if constexpr (std::is_same<T, float>::value) {
    if (ns5_split(m, n, steps, a, b, c, eps))
      return ns5_split_run(G, out, batch, rows, cols, steps, a, b, c, eps, ws, ws_bytes, stream);
  }

  constexpr bool QN = ns5_qn<T>();
  Carver cv(ws, ws_bytes);
  double* partial = cv.take<double>(kRedBlocks * batch);
  A* scale = cv.take<A>(batch);
  // A and B' hold ldm rows so that the bf16 update can read the symmetric
  // B' as its own transpose ([K][M], K = ldm, pad rows zero)
  const int64_t sAB = ldm * ldm;
  T* Ab = cv.take<T>(batch * sAB);
  T* Bb = cv.take<T>(batch * sAB);
  const int64_t sX = QN ? ldm * ldn : m * ldn;  // batch stride of X
  T* X[2];
  T* XT[2] = {nullptr, nullptr};
  X[0] = cv.take<T>(batch * sX);
  if (QN) {
    X[1] = cv.take<T>(batch * sX);
  } else {
    X[1] = X[0];
    XT[0] = cv.take<T>(batch * n * ldm);
    XT[1] = cv.take<T>(batch * n * ldm);
  }
  PTO_REQUIRE(!cv.overflow, "newton_schulz_orthogonalize: workspace too small");
  const int nb = (int)batch;

  // ‖X‖_F per matrix (deterministic two-stage sum), then 1/(‖X‖+eps).
  if (launch_sumsq<T>(G, rows, cols, cols, sG, nb, partial, stream)) return -1;
  hipLaunchKernelGGL(ns_scale_kernel<A>, dim3(nb), dim3(256), 0, stream, partial, eps, scale);
  PTO_LAUNCHED("ns_scale");

  if (steps == 0) {  // the normalised input, in the input's layout
    if (launch_pack<T, T, A>(G, rows, cols, cols, sG, scale, out, cols, sG, nullptr, 0, 0, false, nb, stream)) return -1;
    return 0;
  }

  // X0 = s·X (and, without the QN layout, X0ᵀ), pads zeroed. bf16 inputs
  // that need neither padding nor a transpose skip the copy: the first
  // gram and update read G itself and apply s² and s in their epilogues.
  // The MFMA operand loads are 16-byte accesses, so G must be 16-byte
  // aligned (a view at an odd element offset is packed instead), and the
  // first update reads G while its epilogue writes `out` (with one
  // iteration, the only update), so an aliased call is packed as well.
  const bool direct = QN && !transposed && m == ldm && n == ldn && (g0 & 15) == 0 && !aliased;
  // all pads are cleared by one launch (one per buffer and side were up to
  // seven, 3 us each)
  PadList pads;
  constexpr int64_t E = sizeof(T) / 2;  // its units
  if (QN && direct) {
    // no pads: X[1] is written in full by the first update
  } else if (QN) {
    if (!transposed) {
      if (launch_pack<T, T, A>(G, rows, cols, cols, sG, scale, X[0], ldn, sX, nullptr, 0, 0, false, nb, stream))
        return -1;
    } else {
      if (launch_pack<T, T, A>(G, rows, cols, cols, sG, scale, nullptr, 0, 0, X[0], ldn, sX, false, nb, stream))
        return -1;
    }
    // pad columns of the pong buffer, pad rows of both
    pads.add(X[1], m, ldm, n * E, ldn * E, sX * E, nb);
    pads.add(X[0], m, ldm, ldn * E, ldn * E, sX * E, nb);
  } else {
    if (!transposed) {
      if (launch_pack<T, T, A>(G, rows, cols, cols, sG, scale, X[0], ldn, sX, XT[0], ldm, n * ldm, false, nb, stream))
        return -1;
    } else {
      if (launch_pack<T, T, A>(G, rows, cols, cols, sG, scale, XT[0], ldm, n * ldm, X[0], ldn, sX, false, nb, stream))
        return -1;
    }
    pads.add(XT[1], n, n, m * E, ldm * E, n * ldm * E, nb);
  }
  for (T* p : {Ab, Bb}) pads.add(p, m, ldm, m * E, ldm * E, sAB * E, nb);
  if (launch_zero_pads(pads, stream)) return -1;

  int cur = 0;  // X[cur] (QN) or XT[cur] holds the current iterate
  for (int64_t t = 0; t < steps; ++t) {
    const bool last = t == steps - 1;
    // iteration 0 of an unpacked input reads G (stride sG == sX, no pads)
    const bool from_g = direct && t == 0;
    const T* Xc = from_g ? G : X[cur];
    // 1. A = X·Xᵀ
    {
      GemmArgs g{Xc, ldn, sX, Xc, ldn, sX, (int)m, (int)m, (int)ldn, 0, 0, nullptr};
      if constexpr (QN) {
        if (from_g && launch_gemm<T, true>(g, EpiNsGram<T, A, true>{Ab, ldm, sAB, scale}, nb, stream, "ns5_gram")) return -1;
      }
      if (!from_g && launch_gemm<T, true>(g, EpiNsGram<T, A>{Ab, ldm, sAB, nullptr}, nb, stream, "ns5_gram")) return -1;
    }
    // 2. B' = a·I + b·A + c·A·A
    {
      GemmArgs g{Ab, ldm, sAB, Ab, ldm, sAB, (int)m, (int)m, (int)ldm, 0, 0, nullptr};
      EpiNsSq<T, A> e{Ab, Bb, ldm, sAB, static_cast<A>(a), static_cast<A>(b), static_cast<A>(c)};
      // A is symmetric: both operands read as its own transpose (PT), on
      // any of the three symmetric tiles; without the transposing reads
      // (fp32, fp64) A's rows are its columns, so the NT launch reads A too
      if constexpr (QN) {
        if (launch_gemm_qn<EpiNsSq<T, A>, true, true>(g, e, nb, stream, "ns5_square")) return -1;
      } else {
        if (launch_gemm<T, true>(g, e, nb, stream, "ns5_square")) return -1;
      }
    }
    // 3. X' = B'·X   (QN: over X itself; else as B'·(Xᵀ)ᵀ over the stored
    //    transpose, X written in place since this product does not read it)
    {
      EpiNsUpdate<T, A> e{};
      if (!last && QN) {
        e.dst = X[cur ^ 1]; e.ld_d = ldn; e.s_d = sX;
        e.dstT = nullptr;
      } else if (!last) {
        e.dst = X[0]; e.ld_d = ldn; e.s_d = sX;
        e.dstT = XT[cur ^ 1]; e.ld_t = ldm; e.s_t = n * ldm;
      } else if (!transposed) {
        e.dst = out; e.ld_d = cols; e.s_d = sG;
        e.dstT = nullptr;
      } else {
        e.dst = nullptr;
        e.dstT = out; e.ld_t = cols; e.s_t = sG;
      }
      if constexpr (QN) {
        // B' is symmetric: read as its own transpose (PT), like X (QN)
        GemmArgs g{Bb, ldm, sAB, Xc, ldn, sX, (int)m, (int)n, (int)ldm, 0, 0, nullptr};
        if (from_g) {
          const EpiNsUpdate<T, A, true> es{e.dst, e.ld_d, e.s_d, e.dstT, e.ld_t, e.s_t, scale};
          if (launch_gemm_qn<EpiNsUpdate<T, A, true>, true>(g, es, nb, stream, "ns5_update")) return -1;
        } else if (launch_gemm_qn<EpiNsUpdate<T, A>, true>(g, e, nb, stream, "ns5_update")) {
          return -1;
        }
      } else {
        GemmArgs g{Bb, ldm, sAB, XT[cur], ldm, n * ldm, (int)m, (int)n, (int)ldm, 0, 0, nullptr};
        if (launch_gemm<T, false>(g, e, nb, stream, "ns5_update")) return -1;
      }
    }
    cur ^= 1;
  }
  return 0;
}

// bf16 inputs whose short side is below kNs5Bf16MinSide run in fp32 work
// precision, as the reference runs every bf16 input (they are small, so
// the fp32 chain costs little): G is widened to fp32, the fp32 chain runs,
// and the result is rounded to bf16 once. Keeping X, A and B' in bf16
// between launches costs few-row matrices the most accuracy (relative
// Frobenius error against the fp32 chain up to 0.057 at 3-4 rows, 0.026 at
// 32 and 0.019 at 48 on Gaussian inputs in a CPU emulation of the bf16
// chain, against <= 0.0115 from 96 rows up and ~0.01 at 4096).
constexpr int64_t kNs5Bf16MinSide = 128;

inline bool ns5_bf16_in_f32(int64_t rows, int64_t cols) { return std::min(rows, cols) < kNs5Bf16MinSide; }

size_t ns5_ws_bytes_bf16(int64_t batch, int64_t rows, int64_t cols) {
  if (!ns5_bf16_in_f32(rows, cols)) return ns5_ws_bytes_t<bf16>(batch, rows, cols);
  const size_t copy = round_up(sizeof(float) * (size_t)(batch * rows * cols), 256);
  return 2 * copy + ns5_ws_bytes_t<float>(batch, rows, cols) + 3 * 256;
}

int ns5_bf16(const bf16* G, bf16* out, int64_t batch, int64_t rows, int64_t cols, int64_t steps, double a, double b,
             double c, double eps, void* ws, size_t ws_bytes, hipStream_t stream) {
  if (!ns5_bf16_in_f32(rows, cols))
    return ns5_t<bf16>(G, out, batch, rows, cols, steps, a, b, c, eps, ws, ws_bytes, stream);
  PTO_REQUIRE(batch <= 65535, "newton_schulz_orthogonalize: shape too large");
  if (batch == 0 || rows == 0 || cols == 0) return 0;
  Carver cv(ws, ws_bytes);
  const int64_t sG = rows * cols;
  float* Gf = cv.take<float>(batch * sG);
  float* Of = cv.take<float>(batch * sG);
  const size_t rest = ns5_ws_bytes_t<float>(batch, rows, cols);
  char* wf = cv.take<char>((int64_t)rest);
  PTO_REQUIRE(!cv.overflow, "newton_schulz_orthogonalize: workspace too small");
  const int nb = (int)batch;
  // G is read in full before `out` (which may be G itself) is written
  if (launch_pack<bf16, float, float>(G, rows, cols, cols, sG, nullptr, Gf, cols, sG, nullptr, 0, 0, false, nb,
                                      stream))
    return -1;
  if (ns5_t<float>(Gf, Of, batch, rows, cols, steps, a, b, c, eps, wf, rest, stream)) return -1;
  return launch_pack<float, bf16, float>(Of, rows, cols, cols, sG, nullptr, out, cols, sG, nullptr, 0, 0, false, nb,
                                         stream);
}

}  // namespace
}  // namespace pto

extern "C" {

size_t pto_ns5_workspace_bytes(int dtype, int64_t batch, int64_t rows, int64_t cols) {
  switch (dtype) {
    case pto::kBF16: return pto::ns5_ws_bytes_bf16(batch, rows, cols);
    case pto::kF32: return pto::ns5_ws_bytes_t<float>(batch, rows, cols);
    case pto::kF64: return pto::ns5_ws_bytes_t<double>(batch, rows, cols);
    default: return 0;
  }
}

int pto_ns5(const void* G, void* out, int dtype, int64_t batch, int64_t rows, int64_t cols, int64_t steps, double a,
            double b, double c, double eps, void* workspace, size_t ws_bytes, void* stream) {
  PTO_REQUIRE(batch >= 0 && rows >= 0 && cols >= 0 && steps >= 0,
              "newton_schulz_orthogonalize: negative extent or steps");
  PTO_REQUIRE(batch * rows * cols == 0 || (G && out && workspace),
              "newton_schulz_orthogonalize: null input, output or workspace");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case pto::kBF16:
      return pto::ns5_bf16(static_cast<const pto::bf16*>(G), static_cast<pto::bf16*>(out), batch, rows, cols, steps, a,
                           b, c, eps, workspace, ws_bytes, s);
    case pto::kF32:
      return pto::ns5_t<float>(static_cast<const float*>(G), static_cast<float*>(out), batch, rows, cols, steps, a, b,
                               c, eps, workspace, ws_bytes, s);
    case pto::kF64:
      return pto::ns5_t<double>(static_cast<const double*>(G), static_cast<double*>(out), batch, rows, cols, steps, a,
                                b, c, eps, workspace, ws_bytes, s);
    default:
      PTO_REQUIRE(false, "newton_schulz_orthogonalize: unsupported dtype code");
  }
}

}  // extern "C"
