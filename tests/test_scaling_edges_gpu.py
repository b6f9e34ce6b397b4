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
@pytest.mark.parametrize("score", [1e38, np.inf, np.nan])
def test_scores_beyond_the_range_of_k(B, M, N, score):
    """A score whose K is +inf or NaN: the other elements are not touched by it,
    and the potentials of its element stay free of NaN (one whose K overflows, or
    is infinite, has u = -inf)."""
    rng = np.random.default_rng(N)
    la = -rng.random((B, M, N)).astype(np.float32)
    la[1, 3, 7] = score
    P, used, uh, vh = _forward(la, 0.1, 3)
    assert used == 3
    ref = osk.dual_forward(la[:1], 0.1, 3)
    assert _rel(P[:1], ref.P) < TOL
    assert not np.isnan(uh[:, 1]).any() and not np.isnan(vh[:, 1]).any()
    assert np.isneginf(uh[:, 1, 3]).all() == (not np.isnan(score))


def _marginals(B, M, N, rng, zero_rows, zero_cols):
    """Log-marginals of which element 1 has -inf entries."""
    a, b = rng.dirichlet(np.ones(M), B), rng.dirichlet(np.ones(N), B)
    a[1, zero_rows] = 0.0
    b[1, zero_cols] = 0.0
    with np.errstate(divide="ignore"):
        return [np.log(x / x.sum(1, keepdims=True)).astype(np.float32).clip(-16 if not z else None)
                for x, z in ((a, len(zero_rows)), (b, len(zero_cols)))]


@pytest.mark.parametrize("B,M,N", SHAPES)
@pytest.mark.parametrize("rows,cols", [([3], []), ([0, 1, 7, 30], []), ([], [5]), ([2, 3, 4, 5], [0, 1, 60, 61, 62])])
@pytest.mark.parametrize("T", [1, 2, 7])
def test_zero_marginals(B, M, N, rows, cols, T):
    """log a or log b of -inf: u or v of -inf, a plan of zeros there, and the
    others' values those of the problem without these rows and columns."""
    rng = np.random.default_rng(B + N)
    la = -rng.random((B, M, N)).astype(np.float32)
    lga, lgb = _marginals(B, M, N, rng, rows, cols)
    P, used, uh, vh = _forward(la, 0.1, T, lga, lgb)
    assert used == T
    r, c = np.delete(np.arange(M), rows), np.delete(np.arange(N), cols)
    # the first iteration starts from v = 0 at every column, so it sees them all
    lgb1 = lgb[1:2].copy()
    ref = osk.dual_forward(la[1:2, r], 0.1, T, log_a=lga[1:2, r], log_b=lgb1, keep_history=True)
    assert not P[1, rows].any() and not P[1][:, cols].any()
    assert _rel(P[1][np.ix_(r, c)], ref.P[0][:, c]) < TOL
    scale = max(np.abs(ref.u_hist).max(), np.abs(ref.v_hist[..., c]).max())
    assert np.abs(uh[:, 1][:, r] - ref.u_hist[:, 0]).max() < TOL * scale
    assert np.abs(vh[:, 1][:, c] - ref.v_hist[:, 0][:, c]).max() < TOL * scale
    assert np.isneginf(uh[:, 1][:, rows]).all() and np.isneginf(vh[:, 1][:, cols]).all()


@pytest.mark.parametrize("B,M,N", SHAPES)
def test_zero_marginals_and_the_stop_test(B, M, N):
    """Rows of zero mass take no part in the stop test after the first iteration."""
    tol, noise = 1e-5, 5e-7
    rng = np.random.default_rng(M + 1)
    la = -rng.random((2, M, N)).astype(np.float32)
    lga, _ = _marginals(2, M, N, rng, [1, 2, M - 1], [])
    rep = -(-B // 2)
    _, used, _, _ = _forward(np.concatenate([la] * rep), 0.2, 50, np.concatenate([lga] * rep), None, tol)
    r = np.delete(np.arange(M), [1, 2, M - 1])
    deltas = np.maximum(osk.dual_forward(la[:1], 0.2, 50, log_a=lga[:1]).deltas,
                        osk.dual_forward(la[1:, r], 0.2, 50, log_a=lga[1:, r]).deltas)
    assert 1 < used < 50
    assert deltas[used - 1] < tol + noise and deltas[used - 2] > tol - noise


@pytest.mark.parametrize("B,M,N", SHAPES)
def test_small_plan_entries(B, M, N):
    """An entry below 2^-126 of its row's kernel, in a column with a large factor,
    has its own value in the plan (not 0): row 0 sees column 1 2^-131 away, the
    other rows 2^-33 away."""
    rng = np.random.default_rng(6)
    la = -(0.1 * rng.random((B, M, N))).astype(np.float32)
    la[1, 1:, 1] = -3.3 * np.log(2)
    la[1, 0, 1] = -9.1
    P, _, _, vh = _forward(la, 0.1, 12)
    ref = osk.dual_forward(la[1:2], 0.1, 12)
    want = ref.P[0, 0, 1]
    assert 1e-38 < want < 1e-30 and 20 < vh[-1, 1, 1] < 40 * np.log(2)
    assert abs(P[1, 0, 1] / want - 1) < 1e-4  # exp of a sum of terms of size 91, rounded to 91 2^-24 each
