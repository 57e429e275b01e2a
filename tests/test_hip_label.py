"""Labels of spherical bf16 rows (every component in one workgroup, K <= 1024): the
edges of the padded widths and of the component tiles, against the float64 logits
(a label may differ where its logit is within 1e-5 of the largest, relative to the
logit's terms: the fp32 accumulation), components of weight zero, equal components
and rows that are not finite."""

import pytest
import torch

from tests.test_hip_parity import assert_labels, make_problem, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16


def _labels(hip, x, means, covs, w):
    return hip.score("spherical", x, to_dev(means), to_dev(covs), to_dev(w), want_scores=False)[1]


@pytest.mark.parametrize("d", [1, 8, 31, 32, 33, 64, 65, 96, 97, 127, 128])
@pytest.mark.parametrize("k", [1, 31, 33, 64, 65, 128, 129, 256, 257, 512, 513, 1024, 1025])
def test_labels_match_the_logits(hip, d, k):
    for b, n in ((1, 1), (2, 33), (1, 2500)):
        print(f"[label] B={b} N={n} D={d} K={k}", flush=True)
        x, means, covs, w = make_problem("spherical", b, max(n, 8), d, k, seed=91, dtype=BF)
        x = x[:, :n].contiguous()
        assert_labels(_labels(hip, to_dev(x, BF), means, covs, w), x, means, covs, w, "spherical", 1e-5)


@pytest.mark.parametrize("k", [40, 100, 200, 400, 900])
def test_zero_weights_and_equal_components(hip, k):
    """A component of weight zero takes no row; of equal components the first does."""
    x, means, covs, w = make_problem("spherical", 1, 2000, 48, k, seed=92, dtype=BF)
    w[0, :k:3] = 0.0
    means[0, k // 2:2 * (k // 2)] = means[0, :k // 2]
    covs[0, k // 2:2 * (k // 2)] = covs[0, :k // 2]
    w[0, k // 2:2 * (k // 2)] = w[0, :k // 2]
    lab = _labels(hip, to_dev(x, BF), means, covs, w).cpu()
    assert bool((w[0][lab[0]] > 0).all())
    assert not bool(((lab >= k // 2) & (lab < 2 * (k // 2))).any())


def test_rows_that_are_not_finite_leave_the_others(hip):
    x, means, covs, w = make_problem("spherical", 1, 300, 100, 300, seed=93, dtype=BF)
    good = _labels(hip, to_dev(x, BF), means, covs, w)
    bad = x.clone()
    bad[0, 40, 3], bad[0, 41, 99] = float("nan"), float("inf")
    got = _labels(hip, to_dev(bad, BF), means, covs, w)
    keep = torch.ones(300, dtype=torch.bool)
    keep[40:42] = False
    assert torch.equal(got.cpu()[:, keep], good.cpu()[:, keep])
