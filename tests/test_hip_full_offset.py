"""Full-covariance scores (D <= 16) of data far from the origin: y = L⁻¹x - L⁻¹μ cancels, so
what is added to it after the cancellation must not be rounded before it.

Bar: one rounding at |L⁻¹μ| per whitened entry (2^-25 · |L⁻¹μ|, uniform: over sqrt(3) rms)
and as much again for the stored L⁻¹μ itself, through -½ y² with |y| of rms 1; a quarter for
the other roundings, and the scores' own."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,k", [(2, 2), (8, 16), (16, 9), (16, 32)])
@pytest.mark.parametrize("offset", [30.0, 300.0])
def test_scores_far_from_the_origin(hip, d, k, offset):
    print(f"[full offset] D={d} K={k} offset {offset}", flush=True)
    g = torch.Generator().manual_seed(89)
    randn = lambda *s: torch.randn(s, generator=g)                                   # noqa: E731
    n = 20000
    means = offset + 3 * randn(k, d)
    low = torch.tril((0.5 / d ** 0.5) * randn(k, d, d), -1) + torch.eye(d)
    at = torch.randint(k, (n,), generator=g)
    x = means[at] + (low[at] @ randn(n, d, 1))[..., 0]
    covs, w = low @ low.transpose(-1, -2), torch.full((k,), 1.0 / k)
    got = hip.score("full", *[t[None].contiguous().to("cuda:0") for t in (x, means, covs, w)])[0][0].cpu().double()
    chol = torch.linalg.cholesky(covs.double())
    inv = torch.linalg.inv(chol)
    maha = torch.stack([((x.double() - means[j].double()) @ inv[j].T).square().sum(-1) for j in range(k)], -1)
    exp = torch.logsumexp(-0.5 * maha - chol.diagonal(dim1=-2, dim2=-1).log().sum(-1) - 0.5 * d * 1.8378770664093453
                          - torch.log(torch.tensor(float(k), dtype=torch.double)), -1)
    white = (inv @ means.double()[..., None]).square().mean().sqrt()
    bar = 2 ** 0.5 * 2.0 ** -25 / 3 ** 0.5 * float(white) * d ** 0.5
    error = float((got - exp).square().mean().sqrt())
    print(f"error {error:.2e} bar {bar:.2e}", flush=True)
    assert error <= 1.25 * bar + 2.0 ** -23 * float(exp.abs().max())
