"""The 16-component statistics kernel of full covariance at D > 16 (every K > 8): its
column groups (every multiple of 16 up to 128 and one more), component tiles (two at
D <= 32, K > 16), short slices, and the hard and top-k responsibilities, against the oracle.

Tolerance: fp32 statistics 1e-4 of the statistic's scale, as test_hip_parity; the
top-k sums likewise (seeded problems without ties at the boundary).
"""

import pytest
import torch

from oracle import torch_ref
from tests.test_hip_parity import make_problem, to_dev

pytestmark = pytest.mark.gpu


def _close(got, exp, tol=1e-4):
    torch.testing.assert_close(got.cpu(), exp, rtol=tol, atol=tol * max(1e-30, float(exp.abs().max())))


@pytest.mark.parametrize("d,k", [(17, 9), (17, 33), (32, 12), (32, 17), (33, 16), (48, 9), (49, 31), (64, 9), (64, 32),
                                 (65, 16), (80, 12), (81, 9), (96, 16), (97, 9), (112, 16), (113, 9), (128, 16), (17, 16), (24, 32), (32, 60), (128, 17)])
@pytest.mark.parametrize("b,n", [(1, 1), (2, 33), (1, 700)])
def test_statistics_match_oracle(hip, d, k, b, n):
    print(f"[full stats] B={b} N={n} D={d} K={k}", flush=True)
    x, means, covs, w = make_problem("full", b, max(n, 8), d, k, seed=95)
    x = x[:, :n].contiguous()
    par = [to_dev(t) for t in (means, covs, w)]
    nk, sx, sq, ll = hip.estep_stats("full", to_dev(x), *par)
    e_nk, e_sx, e_sq, e_ll = torch_ref.estep_stats(x, "full", means, covs, w)
    _close(nk, e_nk)
    _close(sx, e_sx)
    _close(sq, e_sq)
    assert torch.equal(sq, sq.transpose(-1, -2))
    assert float(ll) == pytest.approx(float(e_ll), rel=1e-5, abs=1e-4)


@pytest.mark.parametrize("d,k", [(24, 20), (64, 16), (100, 9)])
@pytest.mark.parametrize("top_k", [1, 3])
def test_kept_components_only(hip, d, k, top_k):
    n = 500
    x, means, covs, w = make_problem("full", 1, n, d, k, seed=96)
    par = [to_dev(t) for t in (means, covs, w)]
    nk, sx, sq, ll = hip.estep_stats_topk("full", to_dev(x), *par, top_k)
    e_nk, e_sx, e_sq, e_ll = torch_ref.estep_stats_topk(x, "full", means, covs, w, top_k)
    _close(nk, e_nk)
    _close(sx, e_sx)
    _close(sq, e_sq)
    assert float(ll) == pytest.approx(float(e_ll), rel=1e-5, abs=1e-4)
