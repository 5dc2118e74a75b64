// Kronecker-factor statistics on gfx950.
//
// pto_kron_factor_update replaces _NATIVE.kron_factor_update_
// (pytorch_opt/ops/__init__.py:74-78, csrc/pytorch_opt_ops.cpp:83-94),
// following pytorch_opt/ops/reference.py:100-114:
//     L <- beta·L + (1-beta)·G·Gᵀ,   R <- beta·R + (1-beta)·Gᵀ·G
// (beta == 1 is the plain sum L += G·Gᵀ, R += Gᵀ·G), in place.
//
// pto_gram_update is the additive boundary for the K-FAC activation and
// gradient factors (pytorch_opt/curvature/kron.py:105-113 and the
// clone/EMA/running-mean step at :95-103):
//     F <- beta·F + alpha·X̃ᵀ·X̃,   X̃ = [X, 1] when append_ones is set,
// with beta == 0 meaning "overwrite".
//
// Each factor is one symmetric MFMA launch: only upper tiles are computed,
// the blend with the old factor is fused into the epilogue, and both
// (i, j) and (j, i) are written, so each factor is read and written once. Large
// fp32 products run on split operands (split.h).
#include <algorithm>

#include "aux_kernels.h"
#include "gemm_nt.h"
#include "split.h"

namespace pto {
namespace {

// ------------------------------------------------ fp32 on split operands
//
// Both factors' products on the fp16 MFMA (split.h): L from the planes of G
// with a scale per row, R from those of Gᵀ with a scale per column. The rule
// looks at one matrix only, so that a batched call gives each factor the bits
// of its single call.
// Above a short side of 1024 and this work; below, the pass for the scales and
// the two more launches cost what the products save (1536² 102 us against 92 on
// the fp32 MFMA, 4096 x 512 139 against 132; 1024 x 4096 157 against 223, 2048²
// 133 against 192, 4096² 542 against 1126: 55 in the two passes over G, 246 in
// each product, the rest in launches).
constexpr int64_t kKronSplitSide = 1024;
constexpr double kKronSplitWork = 1.2e10;  // m·n·(m + n)
inline bool kron_split(int64_t m, int64_t n) {
  return std::min(m, n) >= kKronSplitSide && (double)m * n * (m + n) >= kKronSplitWork;
}

struct KronSplitWs {
  sp16 *Gp, *GT;
  unsigned *rpart, *cpart;
  int *bad, *er, *ec;
  int64_t mw, nw;
  KronSplitWs(Carver& cv, int64_t batch, int64_t m, int64_t n) : mw(round_up(m, 8)), nw(round_up(n, 8)) {
    Gp = cv.take<sp16>(2 * batch * m * round_up(n, kPadK));
    GT = cv.take<sp16>(2 * batch * n * round_up(m, kPadK));
    rpart = cv.take<unsigned>(batch * mw * absmax_row_parts(n));
    cpart = cv.take<unsigned>(batch * nw * absmax_col_parts(m));
    bad = cv.take<int>(batch);
    er = cv.take<int>(batch * mw);
    ec = cv.take<int>(batch * nw);
  }
  static size_t bytes(int64_t batch, int64_t m, int64_t n) {
    const int64_t mw = round_up(m, 8), nw = round_up(n, 8);
    return sizeof(sp16) * 2 * (size_t)(batch * (m * round_up(n, kPadK) + n * round_up(m, kPadK))) +
           4 * (size_t)(batch * (mw * (1 + absmax_row_parts(n)) + nw * (1 + absmax_col_parts(m)) + 1)) + 8 * 256;
  }
};

template <class EpiL>
int kron_split_run(const EpiL& el, const EpiL& er, const float* G, int64_t batch, int64_t m, int64_t n, void* ws,
                   size_t ws_bytes, hipStream_t stream) {
  const int64_t ldm = round_up(m, kPadK), ldn = round_up(n, kPadK);
  const int nb = (int)batch;
  Carver cv(ws, ws_bytes);
  const KronSplitWs w(cv, batch, m, n);
  PTO_REQUIRE(!cv.overflow, "kron_factor_update_: workspace too small");
  const SplitPack p{G,    m,       n,   n,           m * n, w.rpart, w.cpart, w.mw,        w.nw, w.er, w.ec, w.bad,
                    w.Gp, m * ldn, ldn, 2 * m * ldn, w.GT,  n * ldm, ldm,     2 * n * ldm, 0};
  if (launch_split_pack_max(p, nb, stream)) return -1;
  {
    SplitArgs g{{w.Gp, ldn, 2 * m * ldn, w.Gp, ldn, 2 * m * ldn, (int)m, (int)m, (int)ldn}, m * ldn, m * ldn, w.bad, 1};
    g.fP = g.fQ = PlainOperand{G, n, 1, m * n, -1};
    g.fK = (int)n;
    const EpiDescale<EpiL> e{el, w.er, w.er, w.mw, w.mw};
    if (launch_gemm<sp16, true, EpiDescale<EpiL>, true>(g, e, nb, stream, "kron_left")) return -1;
  }
  SplitArgs g{{w.GT, ldm, 2 * n * ldm, w.GT, ldm, 2 * n * ldm, (int)n, (int)n, (int)ldm}, n * ldm, n * ldm, w.bad, 1};
  g.fP = g.fQ = PlainOperand{G, 1, n, m * n, -1};
  g.fK = (int)m;
  const EpiDescale<EpiL> e{er, w.ec, w.ec, w.nw, w.nw};
  return launch_gemm<sp16, true, EpiDescale<EpiL>, true>(g, e, nb, stream, "kron_right");
}

template <typename T>
size_t kron_ws_bytes_t(int64_t m, int64_t n) {
  if (std::is_same<T, float>::value && kron_split(m, n)) return KronSplitWs::bytes(1, m, n);
  int64_t ldm = round_up(m, kPadK), ldn = round_up(n, kPadK);
  size_t bytes = 0;
  auto add = [&](size_t b) { bytes = round_up(bytes, 256) + b; };
  add(sizeof(T) * m * ldn);  // G padded (only when n is not a pad multiple)
  add(sizeof(T) * n * ldm);  // Gᵀ
  return bytes + 256;
}

template <typename T>
int kron_t(T* L, T* R, const T* G, int64_t m, int64_t n, double beta2, void* ws, size_t ws_bytes,
           hipStream_t stream) {
  typedef typename AccOf<T>::type A;
  PTO_REQUIRE(m <= INT32_MAX && n <= INT32_MAX, "kron_factor_update_: shape too large");
  if (m == 0 || n == 0) return 0;
  const A beta = beta2 == 1.0 ? A(1) : static_cast<A>(beta2);
  const A alpha = beta2 == 1.0 ? A(1) : static_cast<A>(1.0 - beta2);
  if constexpr (std::is_same<T, float>::value) {
    if (kron_split(m, n))
      return kron_split_run(EpiBlend<T, A>{L, m, 0, beta, alpha}, EpiBlend<T, A>{R, n, 0, beta, alpha}, G, 1, m, n, ws,
                            ws_bytes, stream);
  }
  const int64_t ldm = round_up(m, kPadK), ldn = round_up(n, kPadK);
  Carver cv(ws, ws_bytes);
  T* Gp = cv.take<T>(m * ldn);
  T* GT = cv.take<T>(n * ldm);
  PTO_REQUIRE(!cv.overflow, "kron_factor_update_: workspace too small");

  const bool direct = (n % kPadK == 0) && (reinterpret_cast<uintptr_t>(G) & 15) == 0;
  const T* Grows = direct ? G : Gp;
  const int64_t ldg = direct ? n : ldn;
  if (launch_pack<T, T, A>(G, m, n, n, m * n, nullptr, direct ? nullptr : Gp, ldn, m * ldn, GT, ldm, n * ldm, false, 1,
                           stream))
    return -1;

  {
    GemmArgs g{Grows, ldg, 0, Grows, ldg, 0, (int)m, (int)m, (int)ldn, 0, 0, nullptr};
    EpiBlend<T, A> e{L, m, 0, beta, alpha};
    if (launch_gemm<T, true>(g, e, 1, stream, "kron_left")) return -1;
  }
  {
    GemmArgs g{GT, ldm, 0, GT, ldm, 0, (int)n, (int)n, (int)ldm, 0, 0, nullptr};
    EpiBlend<T, A> e{R, n, 0, beta, alpha};
    if (launch_gemm<T, true>(g, e, 1, stream, "kron_right")) return -1;
  }
  return 0;
}

// Batched form for the optimizers, which update many same-shape factors per
// step: G is one stacked tensor [batch][m][n] (the caller stacks the
// gradients), L[b] and R[b] are separate tensors reached through a pointer
// table. Each side is one launch over the whole batch; every fp32/fp64 tile
// sums a position's products in the same order, so each factor gets exactly
// the bits a single-matrix call gives.
template <typename T>
size_t kron_batched_ws_bytes_t(int64_t batch, int64_t m, int64_t n) {
  if (std::is_same<T, float>::value && kron_split(m, n)) return KronSplitWs::bytes(batch, m, n);
  int64_t ldm = round_up(m, kPadK), ldn = round_up(n, kPadK);
  size_t bytes = 0;
  auto add = [&](size_t b) { bytes = round_up(bytes, 256) + b; };
  add(sizeof(T) * batch * m * ldn);  // G padded (only when n is not a pad multiple)
  add(sizeof(T) * batch * n * ldm);  // Gᵀ
  return bytes + 256;
}

template <typename T>
int kron_batched_t(T* const* L, T* const* R, const T* G, int64_t batch, int64_t m, int64_t n, double beta2, void* ws,
                   size_t ws_bytes, hipStream_t stream) {
  typedef typename AccOf<T>::type A;
  PTO_REQUIRE(m <= INT32_MAX && n <= INT32_MAX, "kron_factor_update_batched_: shape too large");
  PTO_REQUIRE(batch >= 0 && batch <= kBlendTab, "kron_factor_update_batched_: at most 64 matrices per call");
  if (batch == 0 || m == 0 || n == 0) return 0;
  for (int64_t b = 0; b < batch; ++b) {
    PTO_REQUIRE(L[b] && R[b], "kron_factor_update_batched_: null factor");
    for (int64_t c = 0; c < batch; ++c)
      PTO_REQUIRE(L[b] != R[c] && (c == b || (L[b] != L[c] && R[b] != R[c])),
                  "kron_factor_update_batched_: factors must be distinct tensors");
  }
  const A beta = beta2 == 1.0 ? A(1) : static_cast<A>(beta2);
  const A alpha = beta2 == 1.0 ? A(1) : static_cast<A>(1.0 - beta2);
  auto table = [&](T* const* F, int64_t d) {
    EpiBlendTab<T, A> e{};
    e.ld = d;
    e.beta = beta;
    e.alpha = alpha;
    for (int64_t b = 0; b < batch; ++b) e.dst[b] = F[b];
    return e;
  };
  if constexpr (std::is_same<T, float>::value) {
    if (kron_split(m, n)) return kron_split_run(table(L, m), table(R, n), G, batch, m, n, ws, ws_bytes, stream);
  }
  const int64_t ldm = round_up(m, kPadK), ldn = round_up(n, kPadK);
  Carver cv(ws, ws_bytes);
  T* Gp = cv.take<T>(batch * m * ldn);
  T* GT = cv.take<T>(batch * n * ldm);
  PTO_REQUIRE(!cv.overflow, "kron_factor_update_batched_: workspace too small");

  const bool direct = (n % kPadK == 0) && (reinterpret_cast<uintptr_t>(G) & 15) == 0;
  const T* Grows = direct ? G : Gp;
  const int64_t ldg = direct ? n : ldn, sg = direct ? m * n : m * ldn;
  if (launch_pack<T, T, A>(G, m, n, n, m * n, nullptr, direct ? nullptr : Gp, ldn, m * ldn, GT, ldm, n * ldm, false,
                           (int)batch, stream))
    return -1;

  {
    GemmArgs g{Grows, ldg, sg, Grows, ldg, sg, (int)m, (int)m, (int)ldn, 0, 0, nullptr};
    if (launch_gemm<T, true>(g, table(L, m), (int)batch, stream, "kron_left")) return -1;
  }
  {
    GemmArgs g{GT, ldm, n * ldm, GT, ldm, n * ldm, (int)n, (int)n, (int)ldm, 0, 0, nullptr};
    if (launch_gemm<T, true>(g, table(R, n), (int)batch, stream, "kron_right")) return -1;
  }
  return 0;
}

// fp32 X on split operands: the planes of X̃ᵀ with a scale per column of X̃.
// As kron_split: 4096 x 1024 76 us against 70 on the fp32 MFMA, 16384 x 1024
// 212 against 235, 2048² 78 against 100, 8192 x 2048 217 against 360.
constexpr int64_t kGramSplitSide = 1024;
constexpr double kGramSplitWork = 8e9;  // rows·d²
template <typename TX>
bool gram_split(int64_t rows, int64_t d) {
  return std::is_same<TX, float>::value && d >= kGramSplitSide && (double)rows * d * d >= kGramSplitWork;
}
inline size_t gram_split_ws_bytes(int64_t rows, int64_t dd) {
  return sizeof(sp16) * 2 * (size_t)(dd * round_up(rows, kPadK)) +
         4 * (size_t)(round_up(dd, 8) * (1 + absmax_col_parts(rows)) + 1) + 5 * 256;
}
template <class Epi>
int gram_split_run(const Epi& epi, const float* X, int64_t rows, int64_t d, int ones, void* ws, size_t ws_bytes,
                   hipStream_t stream) {
  const int64_t dd = d + ones, ldr = round_up(rows, kPadK), dw = round_up(dd, 8);
  Carver cv(ws, ws_bytes);
  sp16* XT = cv.take<sp16>(2 * dd * ldr);
  unsigned* cpart = cv.take<unsigned>(dw * absmax_col_parts(rows));
  int* bad = cv.take<int>(1);
  int* ec = cv.take<int>(dw);
  PTO_REQUIRE(!cv.overflow, "gram_update_: workspace too small");
  const SplitPack p{X, rows, d, d, 0, nullptr, cpart, 0, dw, nullptr, ec, bad, nullptr, 0, 0, 0, XT, dd * ldr, ldr,
                    0, ones};
  if (launch_split_pack_max(p, 1, stream)) return -1;
  SplitArgs g{{XT, ldr, 0, XT, ldr, 0, (int)dd, (int)dd, (int)ldr}, dd * ldr, dd * ldr, bad, 0};
  g.fP = g.fQ = PlainOperand{X, 1, d, 0, ones ? d : -1};
  g.fK = (int)rows;
  const EpiDescale<Epi> e{epi, ec, ec, 0, 0};
  return launch_gemm<sp16, true, EpiDescale<Epi>, true>(g, e, 1, stream, "gram_update");
}

// bf16 X without the ones column is already the [K][M] operand of the
// transposing-read layout (K = tokens, M = features), for both sides of
// X̃ᵀX̃: it is read in place, with no Xᵀ pass and no workspace, when the
// token count needs no pad rows, the rows are whole 16-byte chunks and the
// tile model picks the 192² or 128² tile (the 256² tile spills with the
// fp32 blend epilogue on this layout). Returns that tile (pick_tile's code)
// or -1 for the packed path. X's 16-byte alignment is the caller's part of
// the contract (checked at launch).
template <typename TX>
int gram_direct_tile(int64_t rows, int64_t d, int append_ones) {
  if (sizeof(TX) != 2 || append_ones || rows % kPadK != 0 || d % 8 != 0 || d == 0) return -1;
  const int pick = pick_tile<TX, true>(d, d, 1);
  return pick == 0 || pick == 2 ? pick : -1;
}

template <typename TX>
size_t gram_ws_bytes_t(int64_t rows, int64_t d, int append_ones) {
  if (gram_direct_tile<TX>(rows, d, append_ones) >= 0) return 0;
  int64_t dd = d + (append_ones ? 1 : 0);
  if (gram_split<TX>(rows, d)) return gram_split_ws_bytes(rows, dd);
  return sizeof(TX) * dd * round_up(rows, kPadK) + 512;
}

// F (TF, [dd][dd]) <- beta·F + alpha·X̃ᵀX̃ with X (TX, [rows][d]).
template <typename TX, typename TF>
int gram_t(TF* F, const TX* X, int64_t rows, int64_t d, int append_ones, double beta, double alpha, void* ws,
           size_t ws_bytes, hipStream_t stream) {
  typedef typename AccOf<TX>::type A;
  const int64_t dd = d + (append_ones ? 1 : 0);
  PTO_REQUIRE(dd <= INT32_MAX && rows <= INT32_MAX, "gram_update_: shape too large");
  if (dd == 0) return 0;
  const int64_t ldr = round_up(rows, kPadK);
  if constexpr (sizeof(TX) == 2) {
    const int tile = gram_direct_tile<TX>(rows, d, append_ones);
    if (tile >= 0) {
      PTO_REQUIRE((reinterpret_cast<uintptr_t>(X) & 15) == 0,
                  "gram_update_: X must be 16-byte aligned (it is read in place)");
      GemmArgs g{X, d, 0, X, d, 0, (int)dd, (int)dd, (int)rows, 0, 0, nullptr};
      EpiBlend<TF, A> e{F, dd, 0, static_cast<A>(beta), static_cast<A>(alpha)};
      return launch_gemm_qn<EpiBlend<TF, A>, true, true>(g, e, 1, stream, "gram_update_direct", tile);
    }
  }
  if constexpr (std::is_same<TX, float>::value && std::is_same<TF, float>::value) {
    if (gram_split<TX>(rows, d))
      return gram_split_run(EpiBlend<TF, A>{F, dd, 0, static_cast<A>(beta), static_cast<A>(alpha)}, X, rows, d,
                            append_ones ? 1 : 0, ws, ws_bytes, stream);
  }
  Carver cv(ws, ws_bytes);
  TX* XT = cv.take<TX>(dd * ldr);
  PTO_REQUIRE(!cv.overflow, "gram_update_: workspace too small");
  // X̃ᵀ, [dd][ldr], with the ones row appended and the token pad zeroed.
  if (launch_pack<TX, TX, A>(X, rows, d, d, 0, nullptr, nullptr, 0, 0, XT, ldr, 0, append_ones != 0, 1, stream))
    return -1;
  GemmArgs g{XT, ldr, 0, XT, ldr, 0, (int)dd, (int)dd, (int)ldr, 0, 0, nullptr};
  EpiBlend<TF, A> e{F, dd, 0, static_cast<A>(beta), static_cast<A>(alpha)};
  return launch_gemm<TX, true>(g, e, 1, stream, "gram_update");
}

}  // namespace
}  // namespace pto

extern "C" {

size_t pto_kron_workspace_bytes(int dtype, int64_t m, int64_t n) {
  switch (dtype) {
    case pto::kBF16: return pto::kron_ws_bytes_t<pto::bf16>(m, n);
    case pto::kF32: return pto::kron_ws_bytes_t<float>(m, n);
    case pto::kF64: return pto::kron_ws_bytes_t<double>(m, n);
    default: return 0;
  }
}

int pto_kron_factor_update(void* L, void* R, const void* G, int dtype, int64_t m, int64_t n, double beta2,
                           void* workspace, size_t ws_bytes, void* stream) {
  PTO_REQUIRE(m >= 0 && n >= 0, "kron_factor_update_: negative extent");
  PTO_REQUIRE(m * n == 0 || (L && R && G && workspace), "kron_factor_update_: null factor, gradient or workspace");
  PTO_REQUIRE(L != G && R != G, "kron_factor_update_: G must not alias L or R");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case pto::kBF16:
      return pto::kron_t<pto::bf16>(static_cast<pto::bf16*>(L), static_cast<pto::bf16*>(R),
                                    static_cast<const pto::bf16*>(G), m, n, beta2, workspace, ws_bytes, s);
    case pto::kF32:
      return pto::kron_t<float>(static_cast<float*>(L), static_cast<float*>(R), static_cast<const float*>(G), m, n,
                                beta2, workspace, ws_bytes, s);
    case pto::kF64:
      return pto::kron_t<double>(static_cast<double*>(L), static_cast<double*>(R), static_cast<const double*>(G), m,
                                 n, beta2, workspace, ws_bytes, s);
    default:
      PTO_REQUIRE(false, "kron_factor_update_: unsupported dtype code");
  }
}

size_t pto_kron_batched_workspace_bytes(int dtype, int64_t batch, int64_t m, int64_t n) {
  switch (dtype) {
    case pto::kBF16: return pto::kron_batched_ws_bytes_t<pto::bf16>(batch, m, n);
    case pto::kF32: return pto::kron_batched_ws_bytes_t<float>(batch, m, n);
    case pto::kF64: return pto::kron_batched_ws_bytes_t<double>(batch, m, n);
    default: return 0;
  }
}

int pto_kron_factor_update_batched(void* const* L, void* const* R, const void* G, int dtype, int64_t batch, int64_t m,
                                   int64_t n, double beta2, void* workspace, size_t ws_bytes, void* stream) {
  PTO_REQUIRE(batch >= 0 && m >= 0 && n >= 0, "kron_factor_update_batched_: negative extent");
  PTO_REQUIRE(batch * m * n == 0 || (L && R && G && workspace),
              "kron_factor_update_batched_: null factor table, gradient stack or workspace");
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case pto::kBF16:
      return pto::kron_batched_t<pto::bf16>(reinterpret_cast<pto::bf16* const*>(L),
                                            reinterpret_cast<pto::bf16* const*>(R),
                                            static_cast<const pto::bf16*>(G), batch, m, n, beta2, workspace, ws_bytes, s);
    case pto::kF32:
      return pto::kron_batched_t<float>(reinterpret_cast<float* const*>(L), reinterpret_cast<float* const*>(R),
                                        static_cast<const float*>(G), batch, m, n, beta2, workspace, ws_bytes, s);
    case pto::kF64:
      return pto::kron_batched_t<double>(reinterpret_cast<double* const*>(L), reinterpret_cast<double* const*>(R),
                                         static_cast<const double*>(G), batch, m, n, beta2, workspace, ws_bytes, s);
    default:
      PTO_REQUIRE(false, "kron_factor_update_batched_: unsupported dtype code");
  }
}

size_t pto_gram_workspace_bytes(int x_dtype, int64_t rows, int64_t d, int append_ones) {
  switch (x_dtype) {
    case pto::kBF16: return pto::gram_ws_bytes_t<pto::bf16>(rows, d, append_ones);
    case pto::kF32: return pto::gram_ws_bytes_t<float>(rows, d, append_ones);
    case pto::kF64: return pto::gram_ws_bytes_t<double>(rows, d, append_ones);
    default: return 0;
  }
}

int pto_gram_update(void* F, int f_dtype, const void* X, int x_dtype, int64_t rows, int64_t d, int append_ones,
                    double beta, double alpha, void* workspace, size_t ws_bytes, void* stream) {
  PTO_REQUIRE(rows >= 0 && d >= 0, "gram_update_: negative extent");
  PTO_REQUIRE((d == 0 && !append_ones) || (F && (rows == 0 || X)), "gram_update_: null factor or input");
  PTO_REQUIRE(workspace || ws_bytes == 0, "gram_update_: null workspace");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (x_dtype == pto::kBF16 && f_dtype == pto::kF32)
    return pto::gram_t<pto::bf16, float>(static_cast<float*>(F), static_cast<const pto::bf16*>(X), rows, d,
                                         append_ones, beta, alpha, workspace, ws_bytes, s);
  if (x_dtype == pto::kF32 && f_dtype == pto::kF32)
    return pto::gram_t<float, float>(static_cast<float*>(F), static_cast<const float*>(X), rows, d, append_ones, beta,
                                     alpha, workspace, ws_bytes, s);
  if (x_dtype == pto::kF64 && f_dtype == pto::kF64)
    return pto::gram_t<double, double>(static_cast<double*>(F), static_cast<const double*>(X), rows, d, append_ones,
                                       beta, alpha, workspace, ws_bytes, s);
  PTO_REQUIRE(false, "gram_update_: unsupported (x dtype, factor dtype) pair");
}

}  // extern "C"
