"""The workloads whose speed this framework is measured on.

A case is a dict of plain values.  Its ``kind`` says which public call it is:

* ``ot``     — a training step through entropic optimal transport:
  ``sinkhorn(cost)`` and the gradient of the summed transport cost, with the
  implicit or the unrolled backward, plain or with an accelerated solver or a
  regularisation schedule, uniform or given marginals;
* ``scores`` — a training step through a soft permutation / attention layer:
  ``sinkhorn_from_scores(logits)`` and the gradient of a loss on the plan;
* ``plan``   — inference: ``sinkhorn(cost, n_iters='auto')`` without gradients
  (the spectral preflight picks the iteration bound);
* ``match``  — a training step through soft sequence matching:
  ``bidirectional_softmax(sim)`` and its gradient, full or with the ragged
  lengths of a padded batch.

``listed()`` holds one case of each size and option in use, ``draw(rng)`` more
of the same ranges.
"""

import math

import torch

import dot_amd

# Element-iterations of a drawn case stay below this (the largest listed case
# takes 6.7e10, three times as many).
_MOST_WORK = 2.0e10
_MOST_ELEMS = 48 << 20


def _ot(name, B, M, N, reg, n_iters, data, tol=1e-6, marginals="uniform", mode="implicit", method="vanilla",
        omega=0.0, schedule="", reg_start=0.0, dtype="fp32", iters=0, sweeps=8):
    """``iters`` is a lower bound of the forward iterations that the input needs
    (0: all ``n_iters``), ``sweeps`` the adjoint sweeps until fp32 has converged."""
    return dict(name=name, kind="ot", B=B, M=M, N=N, reg=reg, n_iters=n_iters, data=data, tol=tol,
                marginals=marginals, mode=mode, method=method, omega=omega, schedule=schedule,
                reg_start=reg_start, dtype=dtype, iters=iters or n_iters, sweeps=sweeps)


def listed():
    return [
        # A loss term on a handful of small point sets: latency and host time.
        _ot("ot_small", 8, 64, 64, 1.0, 100, "uniform", iters=4, sweeps=4),
        # Soft permutations predicted by a network under bf16 autocast, odd
        # sizes, the default 20 iterations, a loss on the plan.
        dict(name="permutation_bf16", kind="scores", B=24, M=97, N=131, reg=0.5, n_iters=20, tol=0.0,
             dtype="bf16", iters=20, sweeps=20),
        # Point-cloud alignment: squared distances of 512-point clouds; it
        # converges in a few iterations.
        _ot("ot_clouds", 64, 512, 512, 0.1, 200, "clouds", iters=5, sweeps=4),
        # Domain adaptation with sample weights: Dirichlet marginals on both
        # sides, a sharp plan that fp32 iterates to the bound.
        _ot("ot_weighted", 16, 1024, 2048, 0.05, 500, "uniform", marginals="dirichlet"),
        # Dense feature matching at full image resolution: the largest call.
        _ot("ot_features", 4, 4096, 4096, 0.02, 1000, "features"),
        # Few sources against a long bank of targets (retrieval, codebooks):
        # rows longer than a wave holds, a fixed count.
        _ot("ot_long_rows", 4, 1024, 16384, 0.05, 100, "uniform", tol=0.0),
        # Gradients through the iterations themselves, with a learnable
        # regularisation (a scalar tensor).
        _ot("ot_unrolled", 24, 300, 260, 0.1, 50, "clouds", mode="unrolled", iters=8),
        # An accelerated solver on a sharp problem, ragged sizes.
        _ot("ot_momentum", 12, 700, 500, 0.03, 100, "clouds", method="momentum", omega=1.4, iters=20),
        # Inference on a batch beyond what the chip holds at once, with the
        # iteration bound predicted from the spectrum.
        dict(name="plan_auto", kind="plan", B=144, M=400, N=450, reg=0.1, data="clouds", tol=1e-6, iters=5),
        # Soft alignment of long sequence pairs, full length.
        dict(name="match_full", kind="match", B=32, M=1024, N=1024, tau=1.0, ragged=False, dtype="fp32"),
        # A padded batch of shorter sequence pairs of many lengths.
        dict(name="match_ragged", kind="match", B=61, M=383, N=509, tau=0.5, ragged=True, dtype="fp32"),
        # A few very long sequence pairs.
        dict(name="match_long", kind="match", B=3, M=2100, N=2900, tau=0.5, ragged=True, dtype="fp32"),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["ot", "ot", "ot", "scores", "plan", "match", "match"])
    if kind == "ot" and rng.random() < 0.15:
        M, N = _log_int(rng, 16, 2048), _log_int(rng, 4097, 16384)
    else:
        M, N = _log_int(rng, 16, 4096), _log_int(rng, 16, 4096)
    if rng.random() < 0.5:  # many programs use multiples of 8, many do not
        M, N = max(8, M // 8 * 8), max(8, N // 8 * 8)
    B = min(_log_int(rng, 1, 256), max(1, _MOST_ELEMS // (M * N)))
    E = B * M * N
    if kind == "match":
        return dict(kind="match", B=B, M=M, N=N, tau=rng.choice([0.3, 0.5, 1.0]), ragged=rng.random() < 0.5,
                    dtype=rng.choice(["fp32", "fp32", "bf16"]))
    most = max(1, int(_MOST_WORK / E))
    if kind == "scores":
        n = min(rng.choice([10, 20, 50]), most)
        return dict(kind="scores", B=B, M=M, N=N, reg=rng.choice([0.3, 0.5, 1.0]), n_iters=n, tol=0.0,
                    dtype=rng.choice(["fp32", "bf16"]), iters=n, sweeps=n)
    if kind == "plan":
        return dict(kind="plan", B=B, M=M, N=N, reg=rng.choice([0.1, 0.3, 1.0]), data="clouds", tol=1e-6,
                    iters=3)
    n = min(_log_int(rng, 20, 500), most)
    opts = rng.choice(["plain", "plain", "plain", "fixed", "weighted", "unrolled", "momentum", "annealed"])
    reg = round(math.exp(rng.uniform(math.log(0.03), math.log(1.0))), 3)
    data = rng.choice(["uniform", "clouds", "features"])
    c = _ot("", B, M, N, reg, n, data, iters=min(n, 3))
    del c["name"]
    if opts == "fixed":
        c.update(tol=0.0, iters=n)
    elif opts == "weighted":
        c.update(marginals="dirichlet")
    elif opts == "unrolled":
        c.update(mode="unrolled", n_iters=min(n, 50), iters=min(n, 3))
    elif opts == "momentum":
        c.update(method="momentum", omega=rng.choice([1.2, 1.4, 1.5]))
    elif opts == "annealed":
        c.update(schedule=rng.choice(["linear", "exponential", "cosine"]), reg_start=5.0 * reg, tol=0.0, iters=n)
    return c


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------
_DTYPES = {"fp32": torch.float32, "bf16": torch.bfloat16}


def _cost(case, g, dev):
    B, M, N = case["B"], case["M"], case["N"]
    if case["data"] == "uniform":
        return torch.rand(B, M, N, generator=g, device=dev)
    dims = 64 if case["data"] == "clouds" else 128
    x = torch.randn(B, M, dims, generator=g, device=dev)
    y = torch.randn(B, N, dims, generator=g, device=dev)
    d = torch.cdist(x, y)
    if case["data"] == "clouds":
        d = d.square_()
    return d.div_(d.amax(dim=(-2, -1), keepdim=True))


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    B, M, N = case["B"], case["M"], case["N"]
    s = {"case": case}
    if case["kind"] in ("ot", "plan"):
        s["cost"] = _cost(case, g, dev).to(_DTYPES[case.get("dtype", "fp32")])
        if case["kind"] == "ot":
            s["cost"].requires_grad_(True)
            s["a"] = s["b"] = None
            if case["marginals"] == "dirichlet":
                ea = torch.rand(B, M, generator=g, device=dev).clamp_(min=1e-6).log_().neg_()
                eb = torch.rand(B, N, generator=g, device=dev).clamp_(min=1e-6).log_().neg_()
                s["a"] = ea / ea.sum(-1, keepdim=True)
                s["b"] = eb / eb.sum(-1, keepdim=True)
            s["reg"] = case["reg"]
            if case["mode"] == "unrolled":  # the unrolled users learn the regularisation too
                s["reg"] = torch.tensor(case["reg"], device=dev, requires_grad=True)
        return s
    s["x"] = torch.randn(B, M, N, generator=g, device=dev).to(_DTYPES[case["dtype"]]).requires_grad_(True)
    s["grad"] = torch.randn(B, M, N, generator=g, device=dev)
    s["lengths"] = None
    if case["kind"] == "match" and case["ragged"]:
        f = torch.rand(B, 2, generator=g, device=dev) * 0.75 + 0.25
        full = torch.tensor([[M, N]], device=dev)
        s["lengths"] = (f * full).ceil().to(torch.int32).clamp_(min=1)
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "ot":
        res = dot_amd.sinkhorn(
            s["cost"], reg=s["reg"], n_iters=case["n_iters"], tol=case["tol"], a=s["a"], b=s["b"],
            backward_mode=case["mode"], method=case["method"], omega=case["omega"] or None,
            schedule=case["schedule"] or None, reg_start=case["reg_start"] or None)
        leaves = [s["cost"]] + ([s["reg"]] if torch.is_tensor(s["reg"]) else [])
        grads = torch.autograd.grad(res.cost.sum(), leaves)
        out = {"plan": res.transport_plan.detach(), "cost": res.cost.detach(), "grad": grads[0]}
        if len(grads) > 1:
            out["grad_reg"] = grads[1]
        return out
    if kind == "scores":
        P = dot_amd.sinkhorn_from_scores(s["x"], tau=case["reg"], n_iters=case["n_iters"], tol=case["tol"])
        return {"plan": P.detach(), "grad": torch.autograd.grad(P, s["x"], s["grad"])[0]}
    if kind == "plan":
        with torch.no_grad():
            res = dot_amd.sinkhorn(s["cost"], reg=case["reg"], n_iters="auto", tol=case["tol"])
        return {"plan": res.transport_plan, "cost": res.cost}
    P = dot_amd.bidirectional_softmax(s["x"], tau=case["tau"], lengths=s["lengths"])
    return {"match": P.detach(), "grad": torch.autograd.grad(P, s["x"], s["grad"].to(P.dtype))[0]}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    E = case["B"] * case["M"] * case["N"]
    edge = 4.0 * case["B"] * (case["M"] + case["N"])
    in_bytes = 2.0 if case.get("dtype", "fp32") == "bf16" else 4.0
    if case["kind"] == "match":
        # sim and grad_out read, out and grad written; two softmaxes, their
        # product and root, and the two-sided softmax gradient
        return {"bytes": E * (2 * in_bytes + 8.0), "flops": 30.0 * E}
    if case["kind"] == "plan":
        # cost read, plan written; per iteration a row and a column log-sum-exp
        return {"bytes": E * 8.0, "flops": 8.0 * E * case["iters"] + 20.0 * E}
    upstream = 4.0 if case["kind"] == "scores" else 0.0  # the plan's gradient
    if case.get("mode") == "unrolled":
        back = 16.0 * E * case["iters"]
    else:
        back = 4.0 * E * case["sweeps"]
    marginals = 2 * edge if case.get("marginals") == "dirichlet" else 0.0
    return {"bytes": E * (2 * in_bytes + 4.0 + upstream) + marginals,
            "flops": 8.0 * E * case["iters"] + back + 20.0 * E}


# ---------------------------------------------------------------------------
# Tolerances
# ---------------------------------------------------------------------------
def tolerance(case):
    # Errors against 64 bits, over the listed and some drawn cases: fp32 plans,
    # costs and gradients 4e-7 .. 2.2e-6, matches and their gradients 1e-7 ..
    # 3.2e-7; each bound is about four times the largest of its kind.
    if case.get("dtype") == "bf16":
        # the gradient comes back in bf16: values whose fp32 forms differ in
        # the last place now and then round to the other neighbour, 2^-8 away
        return {"rel": 5e-4}
    if case["kind"] == "match":
        return {"rel": 1.5e-6}
    # fp32 potentials of size |C| / reg: their rounding enters every entry of
    # the plan, and of the gradient through the adjoint
    return {"rel": 1e-5}


# ---------------------------------------------------------------------------
# The same results in 64 bits, by plain torch
# ---------------------------------------------------------------------------
def _lse(x, dim):
    return torch.logsumexp(x, dim)


def _scale(reg):
    """1 / reg as the operators define it: a 32-bit reciprocal of a 32-bit value."""
    return float(torch.tensor(1.0, dtype=torch.float32) / torch.tensor(float(reg), dtype=torch.float32))


def _annealed(case, step):
    n, reg = case["n_iters"], case["reg"]
    if not case.get("schedule") or n <= 1:
        return reg
    start, f = case["reg_start"], step / (n - 1)
    if case["schedule"] == "linear":
        return start * (1 - f) + reg * f
    if case["schedule"] == "cosine":
        return reg + 0.5 * (start - reg) * (1 + math.cos(math.pi * f))
    return reg * (start / reg) ** (1 - f)


def _solve(la, case, n_iters, log_a, log_b, history=None):
    """(u, v): the iteration of the plain or momentum solver with its stop test."""
    reg, tol, omega = case["reg"], case["tol"], case.get("omega", 0.0)
    B, M, N = la.shape
    u, v = la.new_zeros(B, M), la.new_zeros(B, N)
    K = la * _scale(reg)
    for t in range(n_iters):
        if case.get("schedule"):
            K = la * _scale(_annealed(case, t))
        u0, v0 = u, v
        u = log_a - _lse(K + v[:, None, :], 2)
        if omega:
            w = (1 - omega) * u0 + omega * u
            if float((w - u).abs().max()) < float((u0 - u).abs().max()):
                u = w
        v = log_b - _lse(K + u[:, :, None], 1)
        if omega:
            w = (1 - omega) * v0 + omega * v
            if float((w - v).abs().max()) < float((v0 - v).abs().max()):
                v = w
        if history is not None:
            history.append((u, v))
        if tol > 0:
            d = float((u - u0).abs().max())
            if omega:
                d = max(d, float((v - v0).abs().max()))
            if d < tol:
                break
    return u, v


def _adjoint(P, G, reg, sweeps):
    r, c = (P * G).sum(2), (P * G).sum(1)
    rs, cs = P.sum(2).clamp(min=1e-12), P.sum(1).clamp(min=1e-12)
    mu = torch.zeros_like(c)
    lam = torch.zeros_like(r)
    for _ in range(sweeps):
        lam_new = (r - (P * mu[:, None, :]).sum(2)) / rs
        mu_new = (c - (P * lam_new[:, :, None]).sum(1)) / cs
        same = torch.equal(mu_new, mu) and torch.equal(lam_new, lam)
        lam, mu = lam_new, mu_new
        if same:  # a fixed point: every later sweep repeats it
            break
    return P * (G - lam[:, :, None] - mu[:, None, :]) / reg


def _unrolled(la, P, G, reg, history):
    K = la * _scale(reg)
    X = P * G
    for t in range(len(history) - 1, -1, -1):
        u, v = history[t]
        vp = history[t - 1][1] if t > 0 else torch.zeros_like(v)
        X = X - (K + u[:, :, None] + v[:, None, :]).exp() * X.sum(1, keepdim=True)
        X = X - (K + u[:, :, None] + vp[:, None, :]).exp() * X.sum(2, keepdim=True)
    return X / reg, -(X * la).sum((1, 2)) / (reg * reg)


def _log_marginals(s, B, M, N, dev):
    if s.get("a") is not None:
        return torch.log(s["a"]).double(), torch.log(s["b"]).double()

    def uniform(n):  # a 32-bit constant of the operators
        return torch.full((B, n), float(torch.log(torch.tensor(float(n))).neg()), dtype=torch.float64, device=dev)
    return uniform(M), uniform(N)


def _auto_iters(la, case):
    """The spectral prediction: the largest over the batch."""
    B, M, N = la.shape
    P = torch.softmax(la / case["reg"], 2)
    j = torch.arange(1, N + 1, dtype=torch.float32, device=la.device)[None, :] * 12.9898
    b = torch.arange(1, B + 1, dtype=torch.float32, device=la.device)[:, None] * 78.233

    def centre(x):
        return x - x.mean(-1, keepdim=True)

    def unit(x):
        x = centre(x)
        return x / x.square().sum(-1, keepdim=True).clamp(min=1e-12).sqrt()

    v = unit(torch.sin((j + b).double()))
    for _ in range(5):
        u = centre((P * v[:, None, :]).sum(2))
        v = unit((P * u[:, :, None]).sum(1))
    est = centre((P * v[:, None, :]).sum(2)).square().sum(-1).clamp(min=1e-12).sqrt().clamp(1e-6, 0.999999)
    return int((math.log(1.0 / case["tol"]) / -est.log()).ceil().clamp(3, 1000).max())


def _match(s, case):
    x = s["x"].detach().double() * _scale(case["tau"])
    g = s["grad"].double()
    B, M, N = x.shape
    ln = s["lengths"]
    mask = torch.ones_like(x, dtype=torch.bool)
    if ln is not None:
        i = torch.arange(M, device=x.device)[None, :, None]
        j = torch.arange(N, device=x.device)[None, None, :]
        mask = (i < ln[:, 0, None, None]) & (j < ln[:, 1, None, None])
    x = x.masked_fill(~mask, -math.inf)
    r = torch.softmax(x, 2).nan_to_num_(0.0)
    c = torch.softmax(x, 1).nan_to_num_(0.0)
    out = (1e-9 + r * c).sqrt()
    d = torch.where(mask, g * 0.5 / out, torch.zeros_like(g))
    q = d * r * c
    grad = (2 * q - q.sum(2, keepdim=True) * r - q.sum(1, keepdim=True) * c) * _scale(case["tau"])
    return {"match": out * mask, "grad": grad * mask}


def exact(case, seed):
    E = case["B"] * case["M"] * case["N"]
    s = prepare(case, seed)
    if case["kind"] == "match":
        return _match(s, case)
    n = case.get("n_iters", 1000)
    if E * float(n) > 8.0e10:  # more than about 20 seconds in 64 bits
        return None
    src = s["x"] if case["kind"] == "scores" else s["cost"]
    parts = []
    B, M, N = src.shape
    log_a, log_b = _log_marginals(s, B, M, N, src.device)
    la = src.detach().double()
    if case["kind"] != "scores":
        la = -la
    history = [] if case.get("mode") == "unrolled" else None
    if case["kind"] == "plan":
        n = _auto_iters(la, case)
    u, v = _solve(la, case, n, log_a, log_b, history)
    P = (la * _scale(case["reg"]) + u[:, :, None] + v[:, None, :]).exp()
    if case["kind"] == "plan":
        return {"plan": P, "cost": -(P * la).sum((1, 2))}
    if case["kind"] == "scores":
        return {"plan": P, "grad": _adjoint(P, s["grad"].double(), case["reg"], n)}
    cost = -(P * la).sum((1, 2))
    if case["mode"] == "unrolled":
        g, greg = _unrolled(la, P, -la, case["reg"], history)
        return {"plan": P, "cost": cost, "grad": P - g, "grad_reg": greg.sum()}
    if case["method"] == "vanilla" and not case["schedule"]:
        return {"plan": P, "cost": cost, "grad": P - _adjoint(P, -la, case["reg"], n)}
    # a solver's backward is the adjoint of the plain plan at the same count
    plain = dict(case, omega=0.0, schedule="", tol=0.0)
    counted = []
    _solve(la, case, n, log_a, log_b, counted)
    u, v = _solve(la, plain, len(counted), log_a, log_b)
    Q = (la * _scale(case["reg"]) + u[:, :, None] + v[:, None, :]).exp()
    return {"plan": P, "cost": cost, "grad": P - _adjoint(Q, -la, case["reg"], n)}
