"""Sums of small problems (one row block per slice, as many partials as blocks): with one
component every responsibility is 1, so Σ x against float64 shows the summation alone.
Bar: the fp32 rounding of each total (uniform within half an ulp: at most 2^-24 / sqrt(3)
of it, rms) and a quarter of that for the fp32 sums of 32 rows, whose errors average
over the blocks."""

import pytest
import torch

from tests.test_hip_parity import to_dev

pytestmark = pytest.mark.gpu
D = 16


@pytest.mark.parametrize("cov", ["spherical", "diag", "tied", "full"])
@pytest.mark.parametrize("n", [200, 800, 1500, 4000])
def test_sums_of_one_component(hip, cov, n):
    print(f"[small sums] {cov} N={n}", flush=True)
    eye = torch.eye(D)
    covs = {"spherical": torch.ones(1, 1), "diag": torch.ones(1, 1, D), "tied": eye[None], "full": eye[None, None]}[cov]
    p = [to_dev(t) for t in (torch.full((1, 1, D), 8.0), covs, torch.ones(1, 1))]
    err = []
    for seed in range(6):
        x = 8 + torch.randn((1, n, D), generator=torch.Generator().manual_seed(seed))
        nk, sx = hip.estep_stats(cov, to_dev(x), *p)[:2]
        assert float(nk) == n
        exp = x[0].double().sum(0)
        err.append(sx[0, 0].cpu().double() / exp - 1)
    assert float(torch.cat(err).square().mean().sqrt()) <= 1.25 * 2.0 ** -24 / 3 ** 0.5
