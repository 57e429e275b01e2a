"""Full-covariance statistics at D > 16, K > 8 against float64: relative 2-norm errors of
N_k, Σ r x and Σ r x xᵀ.

Bars: N_k and Σ r x 2^-23: each total rounded once (2^-24 at most), and as much
again for the float32 logits, whose errors (ulp 2^-17 at magnitudes of 100) average out
over the rows unless every rounding goes one way.  Σ r x xᵀ adds a running float32
sum over up to 2048 rows per slice: 1.2 · 2^-22, the four-component kernel's own
at 128 columns being 3.8e-7."""

import pytest
import torch

pytestmark = pytest.mark.gpu

CASES = [(250000, 128, 12), (60000, 80, 24), (100000, 33, 32), (250000, 17, 16), (30000, 20, 32), (30000, 48, 10)]


def _problem(n, d, k):
    g = torch.Generator(device="cuda:0").manual_seed(91)
    randn = lambda *s: torch.randn(s, generator=g, device="cuda:0")                     # noqa: E731
    means = (5 / d ** 0.5) * randn(1, k, d)
    low = torch.tril((0.5 / d ** 0.5) * randn(k, d, d), -1)
    low = low + torch.diag_embed(0.7 + 0.7 * torch.rand((k, d), generator=g, device="cuda:0"))
    at = torch.randint(k, (n,), generator=g, device="cuda:0")
    z = randn(n, d)
    x = torch.empty((1, n, d), device="cuda:0")
    for j in range(k):
        x[0, at == j] = means[0, j] + z[at == j] @ low[j].T.contiguous()
    covs = 1.3 * (low @ low.transpose(-1, -2).contiguous())[None] + 0.1 * torch.eye(d, device="cuda:0")
    return x, means + 0.2 * randn(1, k, d), covs, torch.full((1, k), 1.0 / k, device="cuda:0")


def _exact(x, means, covs, w):
    x, means, covs, w = (t[0].double() for t in (x, means, covs, w))
    k, d = means.shape
    chol = torch.linalg.cholesky(covs)
    inv = torch.linalg.solve_triangular(chol, torch.eye(d, dtype=x.dtype, device=x.device).expand(k, d, d), upper=False)
    lg = torch.stack([-0.5 * ((x - means[j]) @ inv[j].T.contiguous()).square().sum(-1) - chol[j].diagonal().log().sum()
                      + w[j].log() for j in range(k)], -1)
    r = torch.softmax(lg, -1)
    return r.sum(0), r.T.contiguous() @ x, torch.stack([(x * r[:, j:j + 1]).T.contiguous() @ x for j in range(k)])


@pytest.mark.parametrize("n,d,k", CASES, ids=[f"N{c[0]}-D{c[1]}-K{c[2]}" for c in CASES])
def test_sums_against_float64(hip, n, d, k):
    print(f"[full sums] N={n} D={d} K={k}", flush=True)
    p = _problem(n, d, k)
    errors = [float((got[0].double() - exp).norm() / exp.norm())
              for got, exp in zip(hip.estep_stats("full", *p)[:3], _exact(*p))]
    print(errors, flush=True)
    assert errors[0] <= 2.0 ** -23 and errors[1] <= 2.0 ** -23 and errors[2] <= 2.0 ** -22 * 1.2, errors
