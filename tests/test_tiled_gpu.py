"""The tiled persistent forward (row and column tiles of each element over many
workgroups) against the float64 oracle: tile edges, rows in registers and rows
streamed, one tile per row and sixteen, and elements that leave the scaling
domain."""

import numpy as np
import pytest
import torch

import dot_amd
from dot_amd import _ops, profiler
from oracle import sinkhorn as osk

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = 1e-5  # fp32 potentials of size |K| <= 100 round at 8e-6


def _t(x):
    return None if x is None else torch.from_numpy(np.ascontiguousarray(x, dtype=np.float32)).to(DEV)


def _run(la, tau, T, lga=None, lgb=None, tol=0.0, keep=True):
    out = _ops.fused.sinkhorn_forward(_t(la), 1, tau, T, tol, _t(lga), _t(lgb), True, keep)
    torch.cuda.synchronize()
    return out


def _check(la, tau, T, lga=None, lgb=None, tol=0.0, pick=slice(None)):
    """Plan, cost and potentials of the elements `pick` against the oracle at the run's own count."""
    P, cost, counts, uh, vh = _run(la, tau, T, lga, lgb, tol)
    used = int(counts[0])
    at = lambda x: None if x is None else x[pick]
    ref = osk.dual_forward(la[pick], tau, used, log_a=at(lga), log_b=at(lgb), keep_history=True)
    assert torch.isfinite(P).all()
    P = P.cpu().numpy()[pick]
    assert np.abs(P - ref.P).max() < TOL * np.abs(ref.P).max()
    want = -(ref.P * la[pick]).sum((1, 2))
    assert np.abs(cost.cpu().numpy()[pick] - want).max() < TOL * np.abs(want).max()
    scale = max(np.abs(ref.u_hist).max(), np.abs(ref.v_hist).max())  # u + K + v rounds at its largest term
    for got, w in ((uh, ref.u_hist), (vh, ref.v_hist)):
        assert np.abs(got[:used].cpu().numpy()[:, pick] - w).max() < TOL * scale
    return used


@pytest.mark.parametrize("B,M,N", [
    (1, 8, 1028), (1, 9, 2048), (2, 300, 2052), (3, 130, 4096), (1, 257, 4095), (2, 70, 5000), (1, 9, 16384),
    (1, 40, 8193), (3, 300, 1001), (64, 250, 1100), (100, 150, 600), (130, 260, 512), (200, 301, 450), (90, 180, 515),
    (256, 200, 480),
])
def test_matches_oracle(B, M, N):
    print(f"tiled B={B} M={M} N={N}", flush=True)
    rng = np.random.default_rng(B + M + N)
    la = -rng.random((B, M, N)).astype(np.float32)
    lga = np.log(rng.dirichlet(np.ones(M), B)).astype(np.float32).clip(-16)
    lgb = np.log(rng.dirichlet(np.ones(N), B)).astype(np.float32).clip(-16)
    pick = slice(None) if B * M * N < 1 << 21 else [0, B - 1]
    assert _check(la, 0.1, 7, pick=pick) == 7
    assert _check(la, 0.07, 4, lga, lgb, pick=pick) == 4
    assert _check(la, 0.5, 100, tol=1e-5, pick=pick) < 100


@pytest.mark.parametrize("B,M,N", [(3, 96, 1536), (2, 40, 4500), (40, 300, 480)])
@pytest.mark.parametrize("far,tau", [(0.7, 0.01), (0.25, 0.004)])
def test_leaves_at_once(B, M, N, far, tau):
    """A far column in one element: past the bounds of V, or its sum below the floor."""
    rng = np.random.default_rng(9)
    la = -(0.1 * rng.random((B, M, N))).astype(np.float32)
    la[1, :, N - 7] = -far
    assert _check(la, tau, 8, pick=[0, 1]) == 8


@pytest.mark.parametrize("tol", [0.0, 1e-6])
@pytest.mark.parametrize("M,N", [(150, 1400), (90, 5000)])
def test_leaves_after_some_iterations(M, N, tol):
    """Two blocks whose masses do not match: the factors drift until they pass the bounds."""
    B = 2
    rng = np.random.default_rng(4)
    la = -rng.random((B, M, N)).astype(np.float32)
    la[0, : M // 2, N // 2:] -= 6.0
    la[0, M // 2:, : N // 2] -= 6.0
    a = np.full((B, M), 1.0)
    a[0, : M // 2] = 9.0
    lga = np.log(a / a.sum(1, keepdims=True)).astype(np.float32)
    _check(la, 0.1, 45, lga=lga, tol=tol)


def test_masked_entries_and_repeat():
    """-inf scores, and the same bits from a second run."""
    rng = np.random.default_rng(3)
    la = -rng.random((2, 70, 1300)).astype(np.float32)
    la[rng.random(la.shape) < 0.3] = -np.inf
    idx = np.arange(1300)
    la[:, idx % 70, idx] = -0.1
    P, _, _, uh, vh = _run(la, 0.2, 20)
    ref = osk.dual_forward(la, 0.2, 20)
    assert np.abs(P.cpu().numpy() - ref.P).max() < TOL * ref.P.max()
    Q, _, _, uh2, vh2 = _run(la, 0.2, 20)
    assert torch.equal(P, Q) and torch.equal(uh, uh2) and torch.equal(vh, vh2)


@pytest.mark.parametrize("env", [{"DOT_AMD_TILED": "0"}, {"DOT_AMD_AGENT_SCOPE": "1"}])
def test_same_stop_count_as_the_row_tier(env, monkeypatch):
    """The stop test fires at the same iteration on the row-streaming tier; the
    exchange scope changes no bit."""
    rng = np.random.default_rng(5)
    la = -rng.random((3, 200, 2100)).astype(np.float32)
    P, _, counts, _, _ = _run(la, 0.3, 200, tol=1e-5, keep=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    Q, _, other, _, _ = _run(la, 0.3, 200, tol=1e-5, keep=False)
    assert abs(int(counts[0]) - int(other[0])) <= (1 if "DOT_AMD_TILED" in env else 0)
    if "DOT_AMD_AGENT_SCOPE" in env:
        assert torch.equal(P, Q)


@pytest.mark.parametrize("B,M,N", [(3, 2272, 80), (3, 2050, 450)])
def test_waves_without_rows(B, M, N):
    """The last strip has fewer rows than a workgroup has waves: the idle waves'
    registers, whatever ran before left there, take no part in the column sums."""
    C = torch.rand(B, M, N, generator=torch.Generator().manual_seed(M)).to(DEV)
    want = None
    for k in range(6):
        torch.full((64, 1 << 18), float("nan") if k % 2 else float("inf"), device=DEV).mul_(2.0).sum()
        res = dot_amd.sinkhorn(C, reg=0.1, n_iters=12, tol=0.0)
        if want is None:
            want = res.transport_plan
        assert torch.equal(res.transport_plan, want), k


@pytest.mark.parametrize("B,M,N", [(144, 400, 450), (100, 150, 600)])
def test_leaving_elements_touch_no_neighbour(B, M, N):
    """One tile per row: every third element leaves the scaling domain, at an
    iteration of its own.  The others keep the bits that they have beside a
    batch in which none leaves, and a second run has the same bits."""
    T = 24
    rng = np.random.default_rng(B)
    calm = -rng.random((B, M, N)).astype(np.float32)
    a = np.full((B, M), 1.0)
    la, lga0 = calm.copy(), np.log(a / M).astype(np.float32)
    for e in range(0, B, 3):
        la[e, : M // 2, N // 2:] -= 6.0
        la[e, M // 2:, : N // 2] -= 6.0
        a[e, : M // 2] = (9.0, 30.0, 100.0)[e // 3 % 3]
    lga = np.log(a / a.sum(1, keepdims=True)).astype(np.float32)
    profiler.reset()
    profiler.enable(True, ["sk_fwd_tiled"])
    try:
        got = _run(la, 0.1, T, lga)
        profiler.collect()
        assert profiler.query("sk_fwd_tiled")[0] == 1
    finally:
        profiler.enable(False)
    again, alone = _run(la, 0.1, T, lga), _run(calm, 0.1, T, lga0)
    assert int(got[2][0]) == T
    for e in range(0, B, 3):  # a potential beyond 40 ln 2 = 27.7 has left, and none starts there
        assert got[4][0, e].abs().max() < 27 < 28 < got[4][-1, e].abs().max()
    rest = [e for e in range(B) if e % 3]
    for k, dim in ((0, 0), (3, 1), (4, 1)):  # plan, u and v histories
        assert torch.equal(got[k], again[k])
        pick = torch.tensor(rest, device=DEV)
        assert torch.equal(got[k].index_select(dim, pick), alone[k].index_select(dim, pick))
    assert _check(la, 0.1, T, lga, pick=[0, 1, 3, 6, B - 1]) == T


# (2, 200, 300) is resident, the others tiled
@pytest.mark.parametrize("B,M,N", [(2, 200, 300), (2, 300, 1400), (3, 150, 5000), (160, 260, 400)])
@pytest.mark.parametrize("offset,tau", [(1.0, 0.04), (2.0, 0.04)])
def test_stops_where_64_bits_stop(B, M, N, offset, tau):
    """The stop test does not see the rounding of the potentials (2e-6 and 4e-6 at |u| of
    17 and 44, above tol): the run ends at the iteration whose change the oracle has
    below tol, up to what the ratio of two row factors resolves."""
    tol, noise = 1e-6, 5e-7
    rng = np.random.default_rng(M + N)
    la = -offset - rng.random((min(B, 3), M, N)).astype(np.float32)
    lga = np.log(rng.dirichlet(np.ones(M), len(la))).astype(np.float32).clip(-16)
    rep = -(-B // len(la))
    full = lambda x: np.concatenate([x] * rep)[:B]
    P, cost, counts, uh, vh = _run(full(la), tau, 60, full(lga), None, tol)
    used = int(counts[0])
    ref = osk.dual_forward(la, tau, 60, log_a=lga, keep_history=True)
    assert np.abs(ref.u_hist[-1]).max() > 16
    assert int(counts[1]) == 1 and 1 < used < 60
    assert ref.deltas[used - 1] < tol + noise and ref.deltas[used - 2] > tol - noise
    own = osk.dual_forward(la, tau, used, log_a=lga)
    assert np.abs(P[: len(la)].cpu().numpy() - own.P).max() < TOL * own.P.max()


@pytest.mark.parametrize("B,M,N", [(2, 200, 300), (2, 300, 1400), (3, 150, 5000), (160, 260, 400)])
def test_constant_cost_converges_at_the_second_iteration(B, M, N):
    C = torch.full((B, M, N), 50.0, device=DEV)
    res = dot_amd.sinkhorn(C, reg=1.0, n_iters=40, tol=1e-6)
    assert res.n_iters_used == 2 and bool(res.converged)
    assert torch.allclose(res.transport_plan, torch.full_like(C, 1.0 / (M * N)), rtol=TOL, atol=0.0)


@pytest.mark.parametrize("B,M,N", [(2, 200, 300), (2, 300, 1400), (3, 150, 5000)])
def test_tol_below_what_floats_resolve(B, M, N):
    """The run ends at its bound (or at an exact fixed point), with the bound's plan."""
    rng = np.random.default_rng(N)
    la = -rng.random((B, M, N)).astype(np.float32)
    P, _, counts, _, _ = _run(la, 0.05, 40, tol=1e-9, keep=False)
    assert 5 < int(counts[0]) <= 40
    ref = osk.dual_forward(la, 0.05, 40)
    assert np.abs(P.cpu().numpy() - ref.P).max() < TOL * ref.P.max()


@pytest.mark.parametrize("B,M,N", [(4, 1024, 16384), (16, 1024, 2048), (144, 400, 450)])
def test_cost_of_long_tiles(B, M, N):
    """sum(P C) of the returned plan: a lane's entries span e^20, and in one chain
    over all of them the small ones were lost (-3.3e-7 in the mean).  The fold of
    the lanes rounds ten times (wave, workgroup, tiles), either way: no more than
    10 2^-24 for an element, and less than 2^-23 in the mean."""
    C = torch.rand(B, M, N, generator=torch.Generator(device=DEV).manual_seed(N), device=DEV)
    res = dot_amd.sinkhorn(C, reg=0.05, n_iters=20, tol=0.0)
    off = res.cost.double() / (res.transport_plan.double() * C.double()).sum((1, 2)) - 1
    assert float(off.abs().max()) < 10 * 2.0 ** -24
    assert abs(float(off.mean())) < 2.0 ** -23


@pytest.mark.parametrize("B,M,N", [(2, 333, 1400), (2, 70, 5000), (160, 101, 510), (3, 2272, 80)])
@pytest.mark.parametrize("far", [1, 2, 3, 17, 0])
def test_many_columns_leave_at_once(B, M, N, far):
    """One far column of an element, some, every other one (0): the lanes that
    form their exact sums are dealt to them."""
    rng = np.random.default_rng(far + N)
    la = -(0.1 * rng.random((B, M, N))).astype(np.float32)
    cols = np.arange(0, N, 2) if far == 0 else rng.choice(N, min(far, N), replace=False)
    la[1][:, cols] -= 0.7
    assert _check(la, 0.01, 5, pick=[0, 1]) == 5
