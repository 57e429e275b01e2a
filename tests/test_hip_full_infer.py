"""Full-covariance inference at D <= 16, K <= 32: every component count (a kernel each
for ceil(K / 2)) with rows that end inside a 32-row block, against the oracle.
Scores rtol 1e-5 and responsibilities 2e-4, the bars of test_hip_parity."""

import pytest
import torch

from oracle import torch_ref
from tests.test_hip_parity import assert_labels, make_problem, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", range(1, 33))
def test_every_component_count(hip, k):
    for b, n, d in ((1, 1, 16), (2, 33, 5), (3, 321, 16), (1, 700, 1 + k % 16)):
        print(f"[full-infer] B={b} N={n} D={d} K={k}", flush=True)
        x, means, covs, w = make_problem("full", b, max(n, 8), d, k, seed=95)
        x = x[:, :n].contiguous()
        p = (to_dev(x), to_dev(means), to_dev(covs), to_dev(w))
        scores, labels = hip.score("full", *p)
        e_scores = torch_ref.score_samples(x, means, covs, w, "full")
        torch.testing.assert_close(scores.cpu(), e_scores, rtol=1e-5, atol=1e-5 * float(e_scores.abs().mean()))
        assert_labels(labels, x, means, covs, w, "full")
        assert torch.equal(hip.score("full", *p, want_scores=False)[1], labels)
        proba = hip.predict_proba("full", *p).cpu()
        torch.testing.assert_close(proba, torch_ref.predict_proba(x, means, covs, w, "full"), rtol=0, atol=2e-4)


def test_rows_that_are_not_finite_leave_the_others(hip):
    x, means, covs, w = make_problem("full", 1, 200, 16, 21, seed=96)
    p = (to_dev(means), to_dev(covs), to_dev(w))
    good = hip.predict_proba("full", to_dev(x), *p).cpu()
    bad = x.clone()
    bad[0, 70, 3], bad[0, 71, 15] = float("nan"), float("inf")
    got = hip.predict_proba("full", to_dev(bad), *p).cpu()
    keep = torch.ones(200, dtype=torch.bool)
    keep[70:72] = False
    assert torch.equal(got[:, keep], good[:, keep]) and bool(got[:, 70].isnan().all())
    labels = hip.score("full", to_dev(bad), *p, want_scores=False)[1].cpu()
    assert int(labels.min()) >= 0 and int(labels.max()) < 21
