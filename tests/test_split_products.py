"""fp32 operations whose products run on split (two-plane fp16) operands, against
float64: their error may not exceed that of the same computation in plain fp32
multiply-adds over k, which is how the fp32 matrix instructions sum.

Sizes sit at the edges of the 64, 128, 192 and 256 tiles, at the K padding of
128 and at the smallest sizes that take the path.
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
    ((8, 321, 185), 1e-14), ((1, 770, 2049), 1e-25), ((16, 128, 130), 1.0)])
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
