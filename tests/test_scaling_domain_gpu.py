"""The register-resident forward's scaling domain: strips of E = 2^(K log2 e - row
max) against the float64 oracle at the edges of its tiles, and elements that
leave it for the log domain (at once, after some iterations, next to elements
that stay)."""

import numpy as np
import pytest
import torch

from dot_amd import _ops
from oracle import sinkhorn as osk

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 1e-5  # plan and potentials: fp32 potentials of size |K| <= 100 round at 8e-6


def _t(x):
    return None if x is None else torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(DEV)


def _rel(a, b):
    a = np.asarray(a.cpu() if torch.is_tensor(a) else a, np.float64)
    b = np.asarray(b, np.float64)
    return float(np.abs(a - b).max() / max(np.abs(b).max(), 1e-30))


def _check(la, tau, T, lga=None, lgb=None, tol=0.0):
    """Plan, cost and u/v history of the fused forward against the oracle at its own count."""
    P, cost, counts, uh, vh = _ops.fused.sinkhorn_forward(_t(la), 1, tau, T, tol, _t(lga), _t(lgb), True, True)
    torch.cuda.synchronize()
    used = int(counts[0])
    ref = osk.dual_forward(la, tau, used, log_a=lga, log_b=lgb, keep_history=True)
    assert torch.isfinite(P).all()
    assert _rel(P, ref.P) < TOL
    if np.isfinite(la).all():  # (an infinite score times its zero plan entry makes the cost NaN)
        want = -(ref.P * la).sum((1, 2))
        assert np.abs(cost.cpu().numpy() - want).max() < TOL * np.abs(want).max()
    if used:
        # u + K + v is formed from all three, so each carries the rounding of the
        # largest potential (2^-24 of it per operation), however small itself
        scale = max(np.abs(ref.u_hist).max(), np.abs(ref.v_hist).max())
        for got, want in ((uh, ref.u_hist), (vh, ref.v_hist)):
            assert np.abs(got[:used].cpu().numpy() - want).max() < TOL * scale
    return used


@pytest.mark.parametrize("B,M,N", [
    (1, 1, 1), (3, 8, 64), (2, 9, 65), (5, 97, 131), (2, 128, 256), (2, 129, 260), (3, 513, 500), (9, 700, 500),
    (1, 64, 1024), (2, 300, 1001), (33, 40, 24),
])
def test_edges_of_the_tiles(B, M, N):
    print(f"scaling domain B={B} M={M} N={N}", flush=True)
    rng = np.random.default_rng(B + M + N)
    la = -rng.random((B, M, N)).astype(np.float32)
    lga = np.log(rng.dirichlet(np.ones(M), B)).astype(np.float32).clip(-16)
    lgb = np.log(rng.dirichlet(np.ones(N), B)).astype(np.float32).clip(-16)
    assert _check(la, 0.1, 12) == 12
    assert _check(la, 0.05, 7, lga, lgb) == 7
    _check(la, 0.5, 200, tol=1e-5)


def test_masked_entries():
    """-inf scores (K = -inf, E = 0), whole rows and columns kept feasible."""
    rng = np.random.default_rng(3)
    la = -rng.random((3, 70, 90)).astype(np.float32)
    la[rng.random(la.shape) < 0.3] = -np.inf
    idx = np.arange(90)
    la[:, idx % 70, idx] = -0.1
    assert _check(la, 0.2, 20) == 20


@pytest.mark.parametrize("far,tau", [(0.7, 0.01), (0.25, 0.004)])
def test_leaves_at_once(far, tau):
    """A far column (V past its bounds, or its sum below the floor) in one element of three."""
    rng = np.random.default_rng(9)
    la = -(0.1 * rng.random((3, 96, 120))).astype(np.float32)
    la[1, :, 7] = -far
    assert _check(la, tau, 10) == 10


@pytest.mark.parametrize("tol", [0.0, 1e-6])
def test_leaves_after_some_iterations(tol):
    """Two blocks whose masses do not match: the factors drift by a constant
    ratio per iteration until they pass the bounds in the middle of the run."""
    B, M, N = 2, 150, 140
    rng = np.random.default_rng(4)
    la = -rng.random((B, M, N)).astype(np.float32)
    la[0, : M // 2, N // 2:] -= 6.0
    la[0, M // 2:, : N // 2] -= 6.0
    a = np.full((B, M), 1.0)
    a[0, : M // 2] = 9.0
    lga = np.log(a / a.sum(1, keepdims=True)).astype(np.float32)
    _check(la, 0.1, 60, lga=lga, tol=tol)
