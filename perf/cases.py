"""The work that performance is measured on: public calls of pytorch_opt.

Each case is one call that a training program makes, through the entry points
such a program uses (pytorch_opt.ops and the optimizers), on tensors of the
GPU. The listed cases are the sizes of this repository's benchmark and tests
and generic ones between them; draw() gives further cases of the same ranges.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.abspath("pytorch-opt_amd"))

from pytorch_opt import Muon, ops  # noqa: E402

NS_COEFFS = (3.4445, -4.7750, 2.0315)
NS_STEPS = 5
DTYPES = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16}
BYTES = {"f32": 4, "f64": 8, "bf16": 2}

# The most floating-point work of a drawn case, below the largest listed one.
DRAW_FLOPS = {"f32": 1.2e12, "f64": 1.0e11, "bf16": 2.5e12}


def listed():
    return [
        # Muon on one small fp32 matrix: the smallest orthogonalisation of the
        # tests and the benchmark, where launches and latency count.
        {"name": "ns5_f32_512x256", "op": "ns5", "dtype": "f32", "batch": 1, "rows": 512, "cols": 256},
        # Muon's bucket of equal fp32 attention matrices of a d = 2048 model.
        {"name": "ns5_f32_12x2048x2048", "op": "ns5", "dtype": "f32", "batch": 12, "rows": 2048, "cols": 2048},
        # One bf16 MLP projection of a 7B model.
        {"name": "ns5_bf16_4096x11008", "op": "ns5", "dtype": "bf16", "batch": 1, "rows": 4096, "cols": 11008},
        # bf16 matrices whose sides are no multiple of any tile, taller than wide.
        {"name": "ns5_bf16_6x3000x1000", "op": "ns5", "dtype": "bf16", "batch": 6, "rows": 3000, "cols": 1000},
        # The factor update of one large fp32 gradient (Shampoo, SOAP).
        {"name": "kron_f32_4096x4096", "op": "kron", "dtype": "f32", "batch": 1, "rows": 4096, "cols": 4096,
         "beta2": 0.999},
        # Factor updates of several equal odd-sized gradients in one call.
        {"name": "kron_f32_8x1000x513", "op": "kron", "dtype": "f32", "batch": 8, "rows": 1000, "cols": 513,
         "beta2": 0.95},
        # K-FAC activation statistics: bf16 tokens of a d = 4096 layer.
        {"name": "gram_bf16_16384x4096", "op": "gram", "dtype": "bf16", "rows": 16384, "cols": 4096, "ones": False},
        # K-FAC statistics of an fp32 layer with a bias (a ones column).
        {"name": "gram_f32_8192x2048_ones", "op": "gram", "dtype": "f32", "rows": 8192, "cols": 2048, "ones": True},
        # Shampoo's plain step: equal fp32 gradients preconditioned on both sides.
        {"name": "apply_f32_16x2048x2048", "op": "two_sided", "dtype": "f32", "batch": 16, "rows": 2048, "cols": 2048,
         "ta": False, "tb": False},
        # Shampoo's root refresh at its default float64 root precision.
        {"name": "root_f64_8x512", "op": "root", "dtype": "f64", "batch": 8, "n": 512, "p": 4},
        # One ill-conditioned fp32 root that uses all of its 100 iterations.
        {"name": "root_f32_1024", "op": "root", "dtype": "f32", "batch": 1, "n": 1024, "p": 4},
        # A whole Muon step of a small transformer, AdamW parameters included.
        {"name": "muon_step_2x768", "op": "muon", "dtype": "f32", "layers": 2, "d": 768, "vocab": 16000},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _side(rng, lo, hi):
    """A size, log-uniform in [lo, hi]; every other one a multiple of 64."""
    n = _log(rng, lo, hi)
    return n if rng.random() < 0.5 else max(lo, n // 64 * 64)


def _drawn(rng):
    op = rng.choice(["ns5", "ns5", "ns5", "kron", "kron", "gram", "gram", "two_sided", "two_sided", "root"])
    if op == "ns5":
        dtype = rng.choice(["f32", "f32", "bf16"])
        return {"op": op, "dtype": dtype, "batch": _log(rng, 1, 12), "rows": _side(rng, 64, 4096),
                "cols": _side(rng, 64, 4096)}
    if op == "kron":
        return {"op": op, "dtype": "f32", "batch": _log(rng, 1, 8), "rows": _side(rng, 64, 4096),
                "cols": _side(rng, 64, 4096), "beta2": rng.choice([0.95, 0.999, 1.0])}
    if op == "gram":
        return {"op": op, "dtype": rng.choice(["f32", "bf16"]), "rows": _side(rng, 256, 16384),
                "cols": _side(rng, 64, 4096), "ones": rng.random() < 0.5}
    if op == "two_sided":
        ta, tb = rng.choice([(False, False), (True, False), (False, True)])
        return {"op": op, "dtype": "f32", "batch": _log(rng, 1, 16), "rows": _side(rng, 64, 4096),
                "cols": _side(rng, 64, 4096), "ta": ta, "tb": tb}
    dtype = rng.choice(["f32", "f64"])
    return {"op": op, "dtype": dtype, "batch": _log(rng, 1, 8), "n": _side(rng, 64, 768), "p": rng.choice([1, 4])}


def draw(rng):
    while True:
        case = _drawn(rng)
        w = work(case)
        if w["flops"] <= DRAW_FLOPS[case["dtype"]] and w["bytes"] <= 2e9:
            return case


# Damping by root: Shampoo's 4th roots take little, K-FAC's inverses (p = 1) more.
DAMPING = {1: 1e-3, 4: 1e-6}

# Loop iterations that the coupled Newton iteration takes on prepare()'s
# spectra: the float64 runs converge, the float32 runs end at the limit (the
# tolerance lies below float32's rounding).
ROOT_ITERS = {("f64", 4): 20, ("f64", 1): 17, ("f32", 4): 100, ("f32", 1): 100}


def work(case):
    op, e = case["op"], BYTES[case["dtype"]]
    if op == "ns5":
        m, n = sorted((case["rows"], case["cols"]))
        return {"bytes": 2 * e * case["batch"] * m * n, "flops": case["batch"] * _ns5_flops(m, n)}
    if op == "kron":
        m, n = case["rows"], case["cols"]
        return {"bytes": e * case["batch"] * (m * n + 2 * m * m + 2 * n * n),
                "flops": case["batch"] * (m * (m + 1) * n + n * (n + 1) * m)}
    if op == "gram":
        d = case["cols"] + int(case["ones"])
        return {"bytes": e * case["rows"] * case["cols"] + 8 * d * d, "flops": d * (d + 1) * case["rows"]}
    if op == "two_sided":
        m, n = case["rows"], case["cols"]
        return {"bytes": e * case["batch"] * (m * m + n * n + 2 * m * n),
                "flops": case["batch"] * (2 * m * m * n + 2 * m * n * n)}
    if op == "root":
        n = case["n"]
        products = {1: 1, 4: 3}[case["p"]]  # X·Mi and Mk's product; p = 4 adds Mi² and Mi⁴
        per = n * n * (n + 1) * (products + 1)
        return {"bytes": 8 * case["batch"] * n * n, "flops": case["batch"] * ROOT_ITERS[case["dtype"], case["p"]] * per}
    mats, flat = _muon_shapes(case)
    flops = sum(_ns5_flops(*sorted(s)) for s in mats)
    # a matrix: parameter and momentum in and out, gradient in; AdamW: two moments
    return {"bytes": 4 * (5 * sum(a * b for a, b in mats) + 7 * sum(math.prod(s) for s in flat)), "flops": flops}


def _ns5_flops(m, n):
    """Symmetric products counted once: X·Xᵀ, A·A and B·X per iteration."""
    return NS_STEPS * (m * (m + 1) * n + m * m * (m + 1) + 2 * m * m * n)


# Four times what the path differs from the same computation in 64 bits
# (bf16: its chain rounds every iterate to 8 bits), rounded up.
def tolerance(case):
    op = case["op"]
    if op == "ns5" and case["dtype"] == "bf16":
        return {"rel": 4e-2}
    if op == "root":
        # the fp32 iterate amplifies product rounding along the directions of
        # the smallest eigenvalues (condition 5e5)
        return {"rel": 2e-3} if case["dtype"] == "f32" else {"rel": 2e-7}
    if op == "ns5" or op == "muon":
        return {"rel": 2e-5}
    return {"rel": 5e-6}


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(1_000_003 * (seed % 2 ** 31) + 17)


def _grad(g, batch, rows, cols, scale=1e-3):
    """Gradients: noise whose columns and rows differ in scale, as features
    and units of a network do, plus a few strong shared directions."""
    x = torch.randn(batch, rows, cols, generator=g, device="cuda")
    x *= torch.exp(0.5 * torch.randn(batch, 1, cols, generator=g, device="cuda"))
    x *= torch.exp(0.3 * torch.randn(batch, rows, 1, generator=g, device="cuda"))
    u = torch.randn(batch, rows, 4, generator=g, device="cuda")
    v = torch.randn(batch, 4, cols, generator=g, device="cuda")
    return scale * (x + u @ v)


def _spd(g, batch, n):
    """Symmetric positive definite factors with eigenvalues log-uniform in
    [1e-6, 1]: two Householder reflections of a diagonal."""
    A = torch.diag_embed(torch.exp(torch.rand(batch, n, generator=g, device="cuda", dtype=torch.float64)
                                   * math.log(1e-6)))
    for _ in range(2):
        v = torch.randn(batch, n, 1, generator=g, device="cuda", dtype=torch.float64)
        v /= v.norm(dim=1, keepdim=True)
        w = A @ v
        A = A - 2 * v @ w.mT - 2 * w @ v.mT + 4 * (v.mT @ w) * (v @ v.mT)
    return (0.5 * (A + A.mT)).float()


def _muon_shapes(case):
    d, layers = case["d"], case["layers"]
    mats = [s for _ in range(layers) for s in [(d, d)] * 4 + [(4 * d, d), (d, 4 * d)]]
    flat = [(d,)] * (4 * layers + 2) + [(case["vocab"], d)]
    return mats, flat


def _muon_inputs(case, seed):
    g = _gen(seed)
    mats, flat = _muon_shapes(case)
    params = [0.02 * torch.randn(s, generator=g, device="cuda") for s in mats + flat]
    first = [1e-3 * torch.randn(s, generator=g, device="cuda") for s in mats + flat]
    grads = [_grad(g, 1, *s)[0] for s in mats] + [1e-3 * torch.randn(s, generator=g, device="cuda") for s in flat]
    return params, first, grads, len(mats)


def _factor_inputs(case, seed):
    g = _gen(seed)
    b, m, n = case["batch"], case["rows"], case["cols"]
    G = _grad(g, b, m, n)
    L = [(x @ x.mT) * (1.0 / 64) for x in _grad(g, b, m, 64)]
    R = [(x @ x.mT) * (1.0 / 64) for x in _grad(g, b, n, 64)]
    return L, R, list(G.unbind(0))


def _gram_inputs(case, seed):
    g = _gen(seed)
    d = case["cols"] + int(case["ones"])
    X = torch.relu(_grad(g, 1, case["rows"], case["cols"], scale=1.0)[0]).to(DTYPES[case["dtype"]])
    y = torch.randn(d, 64, generator=g, device="cuda")
    return (y @ y.mT) * (1.0 / 64), X


def _two_sided_inputs(case, seed):
    g = _gen(seed)
    b, m, n = case["batch"], case["rows"], case["cols"]

    def root(k):  # a dense symmetric preconditioner, diagonally dominated
        y = torch.randn(b, k, k, generator=g, device="cuda")
        return (0.5 / math.sqrt(k)) * (y + y.mT) + torch.diag_embed(
            torch.exp(torch.randn(b, k, generator=g, device="cuda")))

    return root(m), _grad(g, b, m, n), root(n)


def prepare(case, seed):
    ops.load_native()
    op = case["op"]
    if op == "ns5":
        G = _grad(_gen(seed), case["batch"], case["rows"], case["cols"]).to(DTYPES[case["dtype"]])
        return {"case": case, "G": G if case["batch"] > 1 else G[0]}
    if op == "kron":
        L, R, G = _factor_inputs(case, seed)
        return {"case": case, "L": L, "R": R, "G": G}
    if op == "gram":
        F, X = _gram_inputs(case, seed)
        return {"case": case, "F": F, "X": X}
    if op == "two_sided":
        A, X, B = _two_sided_inputs(case, seed)
        return {"case": case, "A": A, "X": X, "B": B}
    if op == "root":
        return {"case": case, "A": _spd(_gen(seed), case["batch"], case["n"])}
    values, first, grads, k = _muon_inputs(case, seed)
    params = [torch.nn.Parameter(v) for v in values]
    opt = Muon([{"params": params[:k]}, {"params": params[k:], "use_muon": False}], lr=0.02, weight_decay=0.01)
    for p, f in zip(params, first):  # one step of training behind it: the state exists
        p.grad = f
    opt.step()
    for p, gr in zip(params, grads):
        p.grad = gr
    return {"case": case, "opt": opt, "params": params, "k": k}


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "ns5":
        return ops.newton_schulz_orthogonalize(state["G"], steps=NS_STEPS)
    if op == "kron":
        if case["batch"] == 1:
            return ops.kron_factor_update_(state["L"][0], state["R"][0], state["G"][0], beta2=case["beta2"])
        Ls, Rs = ops.kron_factor_update_batched_(state["L"], state["R"], state["G"], beta2=case["beta2"])
        return list(Ls) + list(Rs)
    if op == "gram":
        return ops.gram_update_(state["F"], state["X"], beta=0.95, alpha=0.05 / case["rows"],
                                append_ones=case["ones"])
    if op == "two_sided":
        if not (case["ta"] or case["tb"]):
            return ops.precond_apply_two_sided(state["A"], state["X"], state["B"])
        return ops.two_sided_product(state["A"], state["X"], state["B"], transpose_a=case["ta"],
                                     transpose_b=case["tb"])
    if op == "root":
        return ops.inverse_matrix_root_each(state["A"], case["p"], damping=DAMPING[case["p"]], method="newton",
                                            root_dtype=DTYPES[case["dtype"]])
    state["opt"].step()
    st = state["opt"].state
    moments = [st[p][k] for p in state["params"] for k in ("momentum_buffer", "exp_avg", "exp_avg_sq") if k in st[p]]
    return [p.detach() for p in state["params"]] + moments


# ------------------------------------------------- the same in 64 bits


def _exact_ns5(G):
    a, b, c = NS_COEFFS
    X = G.double()
    flip = X.shape[-2] > X.shape[-1]
    X = X.mT if flip else X
    X = X / (torch.linalg.matrix_norm(X, keepdim=True) + 1e-7)
    for _ in range(NS_STEPS):
        A = X @ X.mT
        X = a * X + (b * A + c * (A @ A)) @ X
    return (X.mT if flip else X).contiguous()


def _exact_muon(case, seed):
    values, first, grads, k = _muon_inputs(case, seed)
    lr, wd, mu = 0.02, 0.01, 0.95
    a_lr, (b1, b2), a_eps = 3e-4, (0.9, 0.95), 1e-8
    params, moments = [v.double() for v in values], []
    for i, p in enumerate(params):
        if i < k:
            buf = torch.zeros_like(p)
            for gr in (first[i].double(), grads[i].double()):
                buf.mul_(mu).add_(gr)
                O = _exact_ns5(gr + mu * buf)
                p.mul_(1 - lr * wd).add_(O, alpha=-lr * max(1.0, p.shape[0] / p.shape[1]) ** 0.5)
            moments.append(buf)
            continue
        m, v = torch.zeros_like(p), torch.zeros_like(p)
        for t, gr in enumerate((first[i].double(), grads[i].double()), 1):
            m.lerp_(gr, 1 - b1)
            v.mul_(b2).addcmul_(gr, gr, value=1 - b2)
            p.add_((m / (1 - b1 ** t)) / ((v / (1 - b2 ** t)).sqrt() + a_eps), alpha=-a_lr)
        moments += [m, v]
    return params + moments


def exact(case, seed):
    op = case["op"]
    if op == "ns5":
        G = prepare(case, seed)["G"]
        if G.dim() == 2:
            return _exact_ns5(G)
        return torch.stack([_exact_ns5(x) for x in G])
    if op == "kron":
        L, R, G = _factor_inputs(case, seed)
        beta = case["beta2"]
        keep, add = (1.0, 1.0) if beta == 1.0 else (beta, 1.0 - beta)
        Ls = [keep * f.double() + add * (x.double() @ x.double().mT) for f, x in zip(L, G)]
        Rs = [keep * f.double() + add * (x.double().mT @ x.double()) for f, x in zip(R, G)]
        return (Ls[0], Rs[0]) if case["batch"] == 1 else Ls + Rs
    if op == "gram":
        F, X = _gram_inputs(case, seed)
        X = X.double()
        if case["ones"]:
            X = torch.cat([X, X.new_ones(X.shape[0], 1)], dim=1)
        return 0.95 * F.double() + (0.05 / case["rows"]) * (X.mT @ X)
    if op == "two_sided":
        A, X, B = (t.double() for t in _two_sided_inputs(case, seed))
        A = A.mT if case["ta"] else A
        B = B.mT if case["tb"] else B
        return torch.stack([a @ x @ b for a, x, b in zip(A, X, B)])
    if op == "root":
        A = _spd(_gen(seed), case["batch"], case["n"]).double()
        out = []
        for a in A:
            lam, V = torch.linalg.eigh(0.5 * (a + a.mT))
            out.append((V * (lam + DAMPING[case["p"]]).pow(-1.0 / case["p"])) @ V.mT)
        return torch.stack(out)
    return _exact_muon(case, seed)
