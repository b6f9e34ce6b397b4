"""Bidirectional softmax of rows longer than 1024 columns: tiles of 1024 columns,
at the edges of the tiles and of the valid region, against the oracle."""

import numpy as np
import pytest
import torch

import dot_amd
from conftest import rel_err, sum_err
from dot_amd import _ops
from oracle import bidirectional_softmax as obs

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)

# float sums of up to L terms in another order than the oracle's: about
# sqrt(L) 2^-24 of the result, 4e-6 at 4096; the gradient subtracts two of them
FWD_TOL, GRAD_TOL = 1e-5, 1e-4


@pytest.mark.parametrize("L1,L2,lengths", [
    (9, 1024, [[9, 1024], [4, 1023]]),                     # one tile: the kernels of short rows
    (9, 1025, [[9, 1025], [9, 1024]]),                     # a second tile of one column, valid or not
    (70, 1028, [[70, 1028], [33, 1025]]),                  # ... of one float4, of which one column is valid
    (5, 2048, [[5, 2048], [5, 1]]),                        # whole tiles; a whole tile without a valid column
    (130, 2052, [[130, 2051], [129, 2047]]),
    (1, 2901, [[1, 2901], [1, 0]]),                        # one row; no valid column at all
    (17, 3100, [[0, 3100], [17, 3]]),                      # no valid row
    (300, 4096, [[300, 4096], [299, 3073]]),
    (6, 4100, [[6, 4100], [6, 2048]]),                     # beyond the longest row of one wave
])
def test_tiles(L1, L2, lengths):
    rng = np.random.default_rng(L1 + L2)
    B, tau = 2, 0.6
    s = (2.0 * rng.standard_normal((B, L1, L2))).astype(np.float32)
    g = rng.standard_normal((B, L1, L2)).astype(np.float32)
    ln = np.array(lengths, np.int32)
    out_o, r_o, c_o = obs.forward(s, tau, ln)
    gs_o, gt_o = obs.backward(s, out_o, g, r_o, c_o, tau, ln)

    def dev(x):
        return torch.as_tensor(x).to(DEV)

    # what lies past the valid region must not reach the results
    dirty = s.copy()
    for b in range(B):
        dirty[b, ln[b, 0]:, :] = np.nan
        dirty[b, :, ln[b, 1]:] = np.inf
    x = dev(dirty).requires_grad_(True)
    P = dot_amd.bidirectional_softmax(x, tau, dev(ln))
    P.backward(dev(g))
    out, r, c = _ops.bidirectional_softmax(dev(s), tau, dev(ln))
    gs, gt = _ops.bidirectional_softmax_backward(dev(s), out, dev(g), r, c, tau, dev(ln))
    for got, want in ((P.detach(), out_o), (out, out_o), (r, r_o), (c, c_o)):
        assert rel_err(got, want) < FWD_TOL
    assert rel_err(x.grad, gs_o) < GRAD_TOL and rel_err(gs, gs_o) < GRAD_TOL
    assert sum_err(gt, gt_o, gs_o * s / tau) < GRAD_TOL
    for b in range(B):
        for T in (P.detach(), x.grad, out, r, c, gs):
            assert (T[b, ln[b, 0]:, :] == 0).all() and (T[b, :, ln[b, 1]:] == 0).all()
