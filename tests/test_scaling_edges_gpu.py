"""The scaling domain's rows and marginals at their extremes, on the resident and
the tiled forward: scores masked by large finite values, by the type's lowest
value and by infinities, whole rows of them."""

import numpy as np
import pytest
import torch

import dot_amd
from dot_amd import _ops
from oracle import sinkhorn as osk

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 1e-5  # plan: fp32 potentials of size |K| <= 100 round at 8e-6

# resident, resident, tiles: several a row, one a row
SHAPES = [(2, 70, 90), (2, 200, 300), (2, 70, 1300), (2, 40, 4500), (100, 150, 600)]
LOWEST = float(torch.finfo(torch.float32).min)


def _t(x):
    return None if x is None else torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(DEV)


def _forward(la, tau, T, lga=None, lgb=None, tol=0.0):
    P, cost, counts, uh, vh = _ops.fused.sinkhorn_forward(_t(la), 1, tau, T, tol, _t(lga), _t(lgb), True, True)
    torch.cuda.synchronize()
    used = int(counts[0])
    return P.cpu().numpy(), used, uh[:used].cpu().numpy(), vh[:used].cpu().numpy()


def _rel(a, b):
    return np.abs(a - b).max() / np.abs(b).max()


@pytest.mark.parametrize("B,M,N", SHAPES)
@pytest.mark.parametrize("fill", [-1e9, -1e10, -1e12, LOWEST, -np.inf])
@pytest.mark.parametrize("T", [1, 6])
def test_masked_rows(B, M, N, fill, T):
    """Padding rows of one element.  While K is finite such a row is one of equal
    scores (and the plan that of any other value: the oracle, whose own potentials
    round at 1e-3 when K is 1e13, takes 0); otherwise it has no mass, as if it
    were not there."""
    rng = np.random.default_rng(M)
    la = -rng.random((B, M, N)).astype(np.float32)
    pad = [0, 5, M - 1]
    la[1, pad] = fill
    rows = np.delete(np.arange(M), pad)
    P, used, uh, vh = _forward(la, 0.1, T)
    assert used == T
    if fill > -1e30:
        equal = la[:2].copy()
        equal[1, pad] = 0.0
        ref = osk.dual_forward(equal, 0.1, T, keep_history=True)
        assert _rel(P[:2], ref.P) < TOL
        want = ref.u_hist[:, 1][:, rows], ref.v_hist[:, 1]
    else:
        lga = np.full((1, M - len(pad)), -np.log(M), np.float32)
        ref = osk.dual_forward(la[1:2, rows], 0.1, T, log_a=lga, keep_history=True)
        assert _rel(P[1, rows], ref.P[0]) < TOL
        assert not P[1, pad].any()
        want = ref.u_hist[:, 0], ref.v_hist[:, 0]
    scale = max(np.abs(w).max() for w in want)
    assert np.abs(uh[:, 1][:, rows] - want[0]).max() < TOL * scale
    assert np.abs(vh[:, 1] - want[1]).max() < TOL * scale


@pytest.mark.parametrize("B,M,N", SHAPES)
@pytest.mark.parametrize("far", [1e9, 1e12])
def test_masked_by_a_sum(B, M, N, far):
    """cost + 1e9 where masked: whole rows, whose differences float32 has rounded
    away, half a row, and an infinite entry."""
    rng = np.random.default_rng(N)
    C = rng.random((B, M, N)).astype(np.float32)
    C[1, [2, M - 1]] += np.float32(far)
    assert np.ptp(C[1, 2]) == 0
    C[0, 3, : N // 2] += np.float32(far)
    C[1, 4, N // 3] = np.inf
    same = C[:2].copy()
    same[1, [2, M - 1]] = 0.0
    same[0, 3, : N // 2] = 1e4
    res = dot_amd.sinkhorn(_t(C), reg=0.1, n_iters=8, tol=0.0)
    ref = osk.dual_forward(-same, 0.1, 8)
    assert _rel(res.transport_plan[:2].cpu().numpy(), ref.P) < TOL


@pytest.mark.parametrize("B,M,N", SHAPES)
def test_scores_beyond_the_range_of_k(B, M, N):
    """A score whose K overflows to +inf has no plan; the other elements are not touched by it."""
    rng = np.random.default_rng(N)
    la = -rng.random((B, M, N)).astype(np.float32)
    la[1, 3, 7] = 1e38
    P, used, _, _ = _forward(la, 0.1, 3)
    assert used == 3
    ref = osk.dual_forward(la[:1], 0.1, 3)
    assert _rel(P[:1], ref.P) < TOL
