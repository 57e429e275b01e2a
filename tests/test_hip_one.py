"""The single-pass spherical bf16 kernels at every width: one workgroup holding all
components (K <= 256) with two, four and eight waves, the group that exchanges row
partials at D < 128, rows whose width is no multiple of a 16-byte chunk (the row's
tail shifted into place) and rows that start off a 16-byte boundary.

Tolerances as in test_hip_parity for bf16 x: statistics and parameters 2e-3 of
the statistic's scale (the responsibilities enter the M-step rounded to bf16,
half an ulp 2^-9), mean log-likelihood rtol 2e-3.
"""

import pytest
import torch

from oracle import torch_ref
from tests.test_hip_parity import assert_bf16_means, make_problem, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16

# (D, K): edges of the padded widths 32 / 64 / 96 / 128, of the wave counts
# (64 / 128 / 256 components) and of the exchanging group (2 and 4 members)
SHAPES = [(3, 70), (8, 65), (32, 128), (33, 129), (47, 256), (64, 65), (65, 1), (95, 64), (96, 65), (96, 200),
          (97, 64), (104, 128), (127, 129), (128, 17), (128, 256), (7, 300), (40, 600), (77, 257), (96, 1024),
          (121, 700)]


def _close(got, exp, tol=2e-3):
    torch.testing.assert_close(got.cpu(), exp, rtol=tol, atol=tol * max(1e-30, float(exp.abs().max())))


@pytest.mark.parametrize("b,n", [(1, 1), (2, 33), (1, 3001)])
@pytest.mark.parametrize("d,k", SHAPES, ids=[f"D{d}-K{k}" for d, k in SHAPES])
def test_single_pass_matches_oracle(hip, d, k, b, n):
    print(f"[one-pass] B={b} N={n} D={d} K={k}", flush=True)
    x, means, covs, w = make_problem("spherical", b, max(n, 8), d, k, seed=71, dtype=BF)
    x = x[:, :n].contiguous()
    xd = to_dev(x, BF)
    if d != 128 and n > 1:      # rows off a 16-byte boundary, as a view of a larger buffer has them
        buf = torch.empty(xd.numel() + 8, dtype=BF, device=DEV)
        xd = buf[3:3 + xd.numel()].copy_(xd.reshape(-1)).view(xd.shape)
    prob = hip.problem("spherical", BF, b, n, d, k)
    ws = hip.Workspace(prob, xd.device)
    nk, sx, sq, ll = hip.estep_stats("spherical", xd, to_dev(means), to_dev(covs), to_dev(w), ws=ws)
    e_nk, e_sx, e_sq, e_ll = torch_ref.estep_stats(x, "spherical", means, covs, w)
    for got, exp in ((nk, e_nk), (sx, e_sx), (sq, e_sq)):
        _close(got, exp)
    assert float(ll) == pytest.approx(float(e_ll), rel=2e-3)
    m_d, c_d, w_d = to_dev(means), to_dev(covs), to_dev(w)
    lb = torch.zeros(1, device=DEV)
    hip.em_step("spherical", xd, m_d, c_d, w_d, lb, ws=ws)
    e_m, e_c, e_w, e_lb = torch_ref.fit_one_iteration_stats(x, "spherical", means, covs, w, bf16_means=True)
    assert float(lb) == pytest.approx(e_lb, rel=2e-3)
    assert int(hip.take_status(ws).item()) == 0
    if n > 1000:                # (a few rows per component: the variances are rounding noise)
        assert_bf16_means(m_d, e_m)
        _close(c_d, e_c)
    _close(w_d, e_w)


def test_nan_row_propagates(hip):
    x, means, covs, w = make_problem("spherical", 1, 2000, 72, 100, seed=72, dtype=BF)
    x[0, 700, 71] = float("nan")
    m_d, c_d, w_d = to_dev(means), to_dev(covs), to_dev(w)
    lb = torch.zeros(1, device=DEV)
    hip.em_step("spherical", to_dev(x, BF), m_d, c_d, w_d, lb)
    assert bool(torch.isnan(lb).all()) and bool(torch.isnan(w_d).all())
    assert torch.equal(m_d.cpu(), means) and torch.equal(c_d.cpu(), covs)
