"""fp32 operations whose products run on split (two-plane fp16) operands, against
float64: their error may not exceed that of the same computation in plain fp32
multiply-adds over k, which is how the fp32 matrix instructions sum.

Sizes sit at the edges of the 64, 128, 192 and 256 tiles, at the K padding of
128 and on both sides of the smallest sizes that take the path.
"""

import math

import pytest
import torch

from pytorch_opt import ops
from pytorch_opt.ops import reference

pytestmark = pytest.mark.gpu

NS = (3.4445, -4.7750, 2.0315)


@pytest.fixture(autouse=True)
def _native(native_backend):
    return native_backend


def _randn(seed, *shape, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(*shape, generator=g)
    x *= torch.exp(0.5 * torch.randn(*shape[:-2], 1, shape[-1], generator=g))
    return x * scale


def _rel(x, want):
    return ((x.double().cpu() - want).norm() / want.norm()).item()


def _chain(P, Q):
    """P·Qᵀ as the fp32 MFMA sums it: one accumulator, rounded after every k
    (elementwise torch on the GPU)."""
    P, Q = P.cuda(), Q.cuda()
    acc = torch.zeros(*P.shape[:-1], Q.shape[-2], device="cuda")
    for k in range(P.shape[-1]):
        acc.addcmul_(P[..., :, k, None], Q[..., None, :, k])
    return acc


def _ns_chain(G, steps, coeffs, eps=1e-7):
    a, b, c = coeffs
    X = G.cuda()
    flip = X.shape[-2] > X.shape[-1]
    X = X.mT if flip else X
    X = X / (torch.linalg.matrix_norm(X.double(), keepdim=True).float() + eps)
    for _ in range(steps):
        A = _chain(X, X)
        B = b * A + c * _chain(A, A) + a * torch.eye(A.shape[-1], device="cuda")
        X = _chain(B, X.mT)
    return X.mT if flip else X


def _no_worse(got, want, plain, roundings=2):
    """The errors of both are sums of many roundings, so their sizes are known
    to a few percent: 1.2 times, or `roundings` roundings of the result itself
    (2^-24 each) where the plain error is below that."""
    assert _rel(got, want) <= max(1.2 * _rel(plain, want), roundings * 2.0 ** -24)


def _ns64(G, steps, coeffs, eps=1e-7):
    return reference.newton_schulz_orthogonalize(G.double(), steps, coeffs, eps)


# scale: ‖G‖ far above eps, near it and far below (there X0 = G/(‖G‖ + eps) is
# tiny and its planes' exponents follow ‖X0‖)
@pytest.mark.parametrize("shape,scale", [
    ((512, 512), 1.0), ((512, 513), 1e-3), ((700, 520), 1e-3), ((4, 257, 1025), 1e-9), ((8, 192, 200), 1e3),
    ((8, 321, 185), 1e-14), ((1, 770, 2049), 1e-25), ((16, 128, 130), 1.0), ((384, 384), 1.0), ((2, 511, 700), 1e3),
    ((3000, 447), 1e-14)])
def test_ns5_split_error_is_fp32s(shape, scale):
    G = _randn(sum(shape), *shape, scale=scale)
    got = ops.newton_schulz_orthogonalize(G.cuda())
    want = torch.stack([_ns64(g, 5, NS) for g in G.reshape(-1, *shape[-2:])]).reshape(shape)
    # far below eps the iteration is five multiplications by a: X is rounded to
    # its planes each time, and a (on B's diagonal) alike each time
    _no_worse(got, want, _ns_chain(G, 5, NS), roundings=10 if scale < 1e-12 else 2)


@pytest.mark.parametrize("steps,coeffs", [(1, NS), (8, (2.0, -1.5, 0.5)), (3, (1.5, -0.5, 0.0)), (2, (9.0, 3.0, 1.0))])
def test_ns5_split_other_coefficients(steps, coeffs):
    G = _randn(5, 640, 520)
    got = ops.newton_schulz_orthogonalize(G.cuda(), steps=steps, coeffs=coeffs)
    _no_worse(got, _ns64(G, steps, coeffs), _ns_chain(G, steps, coeffs))


@pytest.mark.parametrize("bad", [math.nan, math.inf])
def test_ns5_split_non_finite_matrix_only(bad):
    G = _randn(6, 2, 520, 530)
    G[1, 7, 9] = bad
    got = ops.newton_schulz_orthogonalize(G.cuda()).cpu()
    assert torch.isnan(got[1]).all()
    _no_worse(got[0], _ns64(G[0], 5, NS), _ns_chain(G[0], 5, NS))
    Z = torch.zeros(520, 530, device="cuda")
    assert torch.equal(ops.newton_schulz_orthogonalize(Z), Z)


@pytest.mark.parametrize("steps,coeffs", [
    (5, (4.1, -2.9, 0.55)), (4, (4.1, -2.9, 0.55)), (3, (8.2872, -23.5959, 17.3004)), (5, (2.0, 0.5, 0.5)),
    (4, (2.0, 1.0, 1.0)), (3, (9.0, 3.0, 1.0)), (32, (0.6, 0.4, 0.0)), (12, (0.3, 0.0, 0.0)), (5, (0.01, 0.5, 0.0)),
    (32, (1.5, -0.5, 0.0)), (33, (1.5, -0.5, 0.0))])
def test_ns5_coefficients_off_the_usual(steps, coeffs):
    G = torch.randn(640, 576, generator=torch.Generator().manual_seed(9))
    got = ops.newton_schulz_orthogonalize(G.cuda(), steps=steps, coeffs=coeffs)
    _no_worse(got, _ns64(G, steps, coeffs), _ns_chain(G, steps, coeffs), roundings=2 * steps)


# ---------------------------------------------------------------- factor updates

KRON = [(1025, 3500), (2049, 2050), (3001, 1030)]


def _kron_plain(L, R, G, beta2, mm):
    keep, add = (1.0, 1.0) if beta2 == 1.0 else (beta2, 1.0 - beta2)
    return keep * L + add * mm(G, G), keep * R + add * mm(G.mT, G.mT)


@pytest.mark.parametrize("m,n", KRON)
@pytest.mark.parametrize("beta2", [1.0, 0.95])
def test_kron_split_error_is_fp32s(m, n, beta2):
    G, L, R = _randn(m, m, n), _randn(m + 1, m, m), _randn(n + 2, n, n)
    G[3] *= 1e-12   # a row and a column far below the others keep their own scales
    G[:, 5] *= 1e-9
    L, R = L + L.mT, R + R.mT
    L[3], L[:, 3], R[5], R[:, 5] = 0, 0, 0, 0
    Lg, Rg = L.cuda(), R.cuda()
    ops.kron_factor_update_(Lg, Rg, G.cuda(), beta2=beta2)
    want = _kron_plain(L.double(), R.double(), G.double(), beta2, lambda p, q: p @ q.mT)
    plain = _kron_plain(L.cuda(), R.cuda(), G.cuda(), beta2, _chain)
    for got, w, p in zip((Lg, Rg), want, plain):
        assert torch.equal(got, got.mT)
        _no_worse(got, w, p)
    assert _rel(Lg[3], want[0][3]) < 2e-6 and _rel(Rg[5], want[1][5]) < 2e-6


def test_kron_split_batch_gives_single_bits_and_non_finite_stays_put():
    k, m, n = 3, 1030, 3400
    Gs = [_randn(i, m, n).cuda() for i in range(k)]
    Gs[1][4, 6], Gs[1][9, 6], Gs[1][11, 8] = math.inf, -math.inf, math.nan
    Ls, Rs = [torch.zeros(m, m, device="cuda") for _ in range(k)], [torch.zeros(n, n, device="cuda") for _ in range(k)]
    ops.kron_factor_update_batched_(Ls, Rs, Gs, beta2=1.0)
    for i in range(k):
        L1, R1 = torch.zeros(m, m, device="cuda"), torch.zeros(n, n, device="cuda")
        ops.kron_factor_update_(L1, R1, Gs[i], beta2=1.0)
        assert torch.equal(Ls[i].nan_to_num(7.0), L1.nan_to_num(7.0)) and torch.equal(Rs[i].nan_to_num(7.0),
                                                                                      R1.nan_to_num(7.0))
    G = Gs[1].cpu()
    for got, plain in ((Ls[1].cpu(), G @ G.mT), (Rs[1].cpu(), G.mT @ G)):
        for kind in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(kind(got), kind(plain))
        ok = torch.isfinite(plain)
        assert _rel(got[ok], plain[ok].double()) < 2e-6


@pytest.mark.parametrize("rows,d,ones", [(2000, 2049, True), (8193, 1024, False), (1111, 2751, True), (16500, 1024, True)])
def test_gram_split_error_is_fp32s(rows, d, ones):
    X = torch.relu(_randn(rows, rows, d, scale=1e3))
    X[:, 2] = 0.0
    Xt = torch.cat([X, torch.ones(rows, 1)], 1) if ones else X
    F = torch.eye(d + ones)
    got = F.cuda()
    ops.gram_update_(got, X.cuda(), beta=0.5, alpha=1.0 / rows, append_ones=ones)
    assert torch.equal(got, got.mT)
    _no_worse(got, 0.5 * F.double() + (Xt.double().mT @ Xt.double()) / rows, 0.5 * F.cuda() + _chain(Xt.mT, Xt.mT) * (1.0 / rows))
    X[1, 3] = math.nan
    ops.gram_update_(got, X.cuda(), beta=0.5, alpha=1.0 / rows, append_ones=ones)
    hit = torch.zeros(d + ones, d + ones, dtype=torch.bool)
    hit[3], hit[:, 3] = True, True
    assert torch.equal(torch.isnan(got).cpu(), hit)


def test_gram_split_constant_column():
    # l·l, which the products leave out, is largest against h·h for a significand
    # just below 1 + 2^-11 (2^-22), and always positive on the diagonal
    X = torch.randn(8193, 1024, generator=torch.Generator().manual_seed(4))
    X[:, 0] = 1 + 2.0 ** -11 - 2.0 ** -23
    F = torch.zeros(1024, 1024, device="cuda")
    ops.gram_update_(F, X.cuda(), beta=0.0, alpha=1.0)
    want = X[:, 0].double().square().sum().item()
    assert abs(F[0, 0].item() / want - 1) <= 2.0 ** -21


# ---------------------------------------------------------------- two-sided products


def _sides(b, m, n):
    A, X, B = _randn(m, b, m, m), _randn(m + n, b, m, n, scale=1e-3), _randn(n, b, n, n)
    return A / math.sqrt(m) + 3 * torch.eye(m), X, B / math.sqrt(n) + 3 * torch.eye(n)


@pytest.mark.parametrize("m,n", [(1830, 1900), (560, 4400), (4700, 520), (2049, 1700)])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, False), (False, True), (True, True)])
def test_two_sided_split_error_is_fp32s(m, n, ta, tb):
    A, X, B = _sides(1, m, n)
    X[..., 2], X[..., 5], X[:, 3] = 0.0, X[..., 5] * 1e-12, 0.0  # empty and tiny columns, an empty row
    got = ops.two_sided_product(A[0].cuda(), X[0].cuda(), B[0].cuda(), transpose_a=ta, transpose_b=tb)
    op = lambda T, t: T.mT if t else T
    want = op(A[0], ta).double() @ X[0].double() @ op(B[0], tb).double()
    a, b = op(A[0], ta).cuda(), op(B[0], tb).cuda()
    _no_worse(got, want, _chain(_chain(a, X[0].cuda().mT), b.mT))


def test_two_sided_split_batch_shared_factors_and_non_finite():
    A, X, B = (t.cuda() for t in _sides(3, 1830, 1840))
    for a, b in ((A, B), (A[:1], B), (A, B[:1])):
        got = ops.precond_apply_two_sided(a, X, b)
        for i in range(3):
            assert torch.equal(got[i], ops.precond_apply_two_sided(a[i % len(a)], X[i], b[i % len(b)]))
    X[1, 4, 6] = math.nan
    got = ops.precond_apply_two_sided(A, X, B)
    assert torch.isnan(got[1]).all() and torch.isfinite(got[[0, 2]]).all()
    assert _rel(got[2], (A[2].double() @ X[2].double() @ B[2].double()).cpu()) < 5e-6


# Row by row and entry by entry: a row far below the others keeps the error that
# plain fp32 sums leave it.


def _err(x, want, dim=-1):
    """Relative error of every row (or column) that is not empty; an empty one
    has to come out empty."""
    x, size = x.double().cpu(), want.norm(dim=dim)
    err = (x - want).norm(dim=dim)
    assert (err[size == 0] == 0).all()
    return err / size.clamp_min(1e-300)


def _rows_no_worse(got, want, plain, dim=-1, roundings=4):
    """One row's error is a sample of a few hundred roundings or more: 1.5 times
    the plain one's, or `roundings` roundings of the result."""
    e, p = _err(got, want, dim), _err(plain, want, dim)
    over = e / torch.clamp(1.5 * p, min=roundings * 2.0 ** -24)
    worst = int(over.argmax())
    assert over[worst].item() <= 1, (worst, e[worst].item(), p[worst].item())


SMALL = {3: 1e-2, 64: 1e-4, 130: 1e-6, 131: 1e-7, 700: 1e-8, 701: 1e-12, 1100: 0.0}


@pytest.mark.parametrize("kind", ["identity", "near", "dense"])
@pytest.mark.parametrize("ta,tb", [(False, False), (True, True)])
def test_two_sided_split_keeps_small_rows_and_columns(kind, ta, tb):
    m, n = 1830, 1900
    A, X, B = (t[0] for t in _sides(1, m, n))
    X = X * 1e3
    if kind != "dense":
        A = torch.eye(m) + (1e-5 * torch.randn(m, m, generator=torch.Generator().manual_seed(1)) if kind == "near" else 0)
        B = torch.eye(n) + (1e-5 * torch.randn(n, n, generator=torch.Generator().manual_seed(2)) if kind == "near" else 0)
    for i, s in SMALL.items():
        X[i] *= s
        X[:, i + 5] *= s
    op = lambda T, t: T.mT if t else T
    got = ops.two_sided_product(A.cuda(), X.cuda(), B.cuda(), transpose_a=ta, transpose_b=tb)
    a, b = op(A, ta), op(B, tb)
    want = a.double() @ X.double() @ b.double()
    plain = _chain(_chain(a, X.mT), b.mT)
    _rows_no_worse(got, want, plain)
    _rows_no_worse(got, want, plain, dim=-2)


@pytest.mark.parametrize("scale", [1e-33, 1e-30, 1e-20, 1e18])
def test_two_sided_split_scale_of_x(scale):
    A, X, B = (t[0] for t in _sides(1, 1830, 1840))
    X = X * 1e3 * scale
    X[7] *= 1e-6
    want = A.double() @ X.double() @ B.double()
    got = ops.precond_apply_two_sided(A.cuda(), X.cuda(), B.cuda())
    _rows_no_worse(got, want, _chain(_chain(A, X.mT), B.mT))


@pytest.mark.parametrize("decades", [6, 8, 10])
def test_two_sided_split_transports_second_moments(decades):
    # SOAP: v = λ_i·μ_j (and some noise) between two bases that turned a little
    m, n = 1830, 1900
    g = torch.Generator().manual_seed(decades)

    def turn(k):
        s = torch.randn(k, k, generator=g, dtype=torch.float64) * (0.02 / math.sqrt(k))
        return torch.linalg.qr(torch.eye(k, dtype=torch.float64) + s - s.mT)[0].float().pow(2)

    A, B = turn(m), turn(n)
    lam = torch.logspace(0, -decades, m, dtype=torch.float64)[torch.randperm(m, generator=g)]
    mu = torch.logspace(0, -decades, n, dtype=torch.float64)[torch.randperm(n, generator=g)]
    v = (lam[:, None] * mu * torch.exp(torch.randn(m, n, generator=g, dtype=torch.float64))).float()
    want = A.double().mT @ v.double() @ B.double()
    got = ops.two_sided_product(A.cuda(), v.cuda(), B.cuda(), transpose_a=True)
    worst = lambda x: ((x.double().cpu() - want) / want).abs().max().item()
    plain = _chain(_chain(A.mT, v.mT), B.mT)
    assert worst(got) <= max(worst(plain), 16 * 2.0 ** -24)


def test_two_sided_split_preconditions_with_its_own_factors():
    # Shampoo: L^(-1/4)·G·R^(-1/4) of G's own factors, units that hardly fire among them
    m, n = 1830, 1900
    G = _randn(11, m, n)
    for i, s in {3: 1e-4, 64: 1e-5, 700: 1e-6}.items():
        G[i] *= s

    def root(F):
        lam, V = torch.linalg.eigh(F)
        return ((V * lam.clamp_min(1e-14 * lam[-1]).pow(-0.25)) @ V.mT).float()

    Gd = G.double()
    A, B = root(Gd @ Gd.mT), root(Gd.mT @ Gd)
    want = A.double() @ G.double() @ B.double()
    got = ops.precond_apply_two_sided(A.cuda(), G.cuda(), B.cuda())
    _rows_no_worse(got, want, _chain(_chain(A, G.mT), B.mT))


def test_two_sided_split_non_finite_lands_where_fp32_puts_it():
    A, X, B = (t[0] for t in _sides(1, 1830, 1840))
    A, B = torch.eye(1830) * 2, torch.eye(1840) * 3
    X[4, 6], X[9, 6], X[11] = math.inf, -math.inf, 0.0
    A[5, 11] = math.inf  # against an empty row of X
    plain = _chain(_chain(A, X.mT), B.mT)
    got = ops.precond_apply_two_sided(A.cuda(), X.cuda(), B.cuda())
    assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), plain.nan_to_num(7.0, 8.0, 9.0))


@pytest.mark.parametrize("b,m,n", [(8, 1024, 1024), (16, 512, 700), (3, 1500, 1501), (4, 1830, 1840)])
def test_two_sided_batch_gives_single_bits(b, m, n):
    A, X, B = (t.cuda() for t in _sides(b, m, n))
    X[1, 4, 6], B[2, 1, 7] = math.nan, math.inf
    for a, bb in ((A, B), (A[:1], B), (A, B[:1])):
        got = ops.precond_apply_two_sided(a, X, bb)
        for i in range(b):
            one = ops.precond_apply_two_sided(a[i % len(a)], X[i], bb[i % len(bb)])
            assert torch.equal(got[i].nan_to_num(7.0, 8.0, 9.0), one.nan_to_num(7.0, 8.0, 9.0))


@pytest.mark.parametrize("shape", [(576, 700), (700, 576), (1500, 1500)])
@pytest.mark.parametrize("s", [1e-1, 1e-2, 1e-3, 1e-4, 1e-6, 1e-9, 1e-12])
def test_ns5_split_keeps_small_rows_and_columns(shape, s):
    G = _randn(21, *shape)
    G[3] *= s
    G[:, 130] *= s
    G[64] = 0.0
    got = ops.newton_schulz_orthogonalize(G.cuda())
    want, plain = _ns64(G, 5, NS), _ns_chain(G, 5, NS)
    _no_worse(got, want, plain)
    # single rows' errors lie along the few smallest singular directions and so
    # spread more than independent roundings (up to 1.6 times between two fp32
    # chains); the small row and column are as near as any other
    for dim, at in ((-1, 3), (-2, 130)):
        e, p = _err(got, want, dim), _err(plain, want, dim)
        assert e.max() <= 2 * p.max() and e[at] <= 1.5 * max(p[at].item(), _rel(plain, want))


@pytest.mark.parametrize("shape", [(8, 256, 1024), (16, 128, 200), (8, 384, 512), (3, 576, 700), (4, 700, 576)])
def test_ns5_batch_gives_single_bits(shape):
    G = _randn(31, *shape).cuda()
    G[1, 5] *= 1e-8
    G[-1, 2, 3] = math.inf
    got = ops.newton_schulz_orthogonalize(G)
    for g, o in zip(G, got):
        assert torch.equal(o.nan_to_num(7.0), ops.newton_schulz_orthogonalize(g).nan_to_num(7.0))


# A matrix whose planes do not serve, over the split products' tiles: the bits of
# the fp32 kernels, which a negative eps (lost in the norm's rounding) asks for.
@pytest.mark.parametrize("shape", [(512, 640), (1000, 1100), (2048, 2048), (3100, 3000), (4, 2048, 2100), (12, 1024, 1024),
                                   (2, 3072, 768), (4096, 4096)])
def test_ns5_flagged_matrix_gets_the_fp32_kernels_bits(shape):
    G = _randn(41, *shape).cuda()
    G[..., 3, :] *= 1e-9
    got = ops.newton_schulz_orthogonalize(G, eps=0.0)
    assert torch.equal(got, ops.newton_schulz_orthogonalize(G, eps=-1e-30))


@pytest.mark.parametrize("m,n", KRON + [(1024, 6000), (4096, 4100)])
def test_kron_flagged_over_tiles(m, n):
    G = _randn(m + n, m, n)
    G[7, 9], G[m - 1, n - 1] = math.inf, math.nan
    L, R = torch.zeros(m, m, device="cuda"), torch.zeros(n, n, device="cuda")
    ops.kron_factor_update_(L, R, G.cuda(), beta2=1.0)
    for got, P in ((L, G), (R, G.mT)):
        plain = _chain(P, P)
        assert torch.equal(got.isnan(), plain.isnan()) and torch.equal(got.isposinf(), plain.isposinf())
        ok = torch.isfinite(plain)
        diff = (got[ok].double() - plain[ok].double()).norm() / plain[ok].double().norm()
        assert diff.item() <= 4e-6  # two orders of up to 6000 fp32 additions


@pytest.mark.parametrize("m,n", [(1500, 1500), (640, 4096), (2049, 1700), (3000, 3100), (4096, 4096)])
@pytest.mark.parametrize("ta,tb", [(False, True), (True, False)])
def test_two_sided_flagged_over_tiles(m, n, ta, tb):
    # a row of op(A) that meets only a row of X at 1e-34: its scale would leave fp32
    A, X, B = (t[0] for t in _sides(1, m, n))
    X, a = X * 1e3, A.mT if ta else A
    X[5] *= 1e-34
    a[5], a[5, 5] = 0.0, 2.0
    b = B.mT if tb else B
    got = ops.two_sided_product(A.cuda(), X.cuda(), B.cuda(), transpose_a=ta, transpose_b=tb)
    want = (a.double().cuda() @ X.double().cuda() @ b.double().cuda()).cpu()
    _rows_no_worse(got, want, _chain(_chain(a, X.mT), b.mT))
