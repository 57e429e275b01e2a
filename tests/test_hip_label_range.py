"""Labels are component indices whatever the row holds: rows that are not finite, rows
whose squared norm overflows and rows so far out that every logit is below the
padding components' constant, through every label path.  A row without a maximum
gets component 0, as torch.argmax gives for a row of NaN."""

import pytest
import torch

from tests.test_hip_parity import make_problem, to_dev

pytestmark = pytest.mark.gpu
BF = torch.bfloat16

CASES = [  # cov, D, K, dtype: one component tile, several, every padded count
    ("spherical", 20, 5, torch.float32), ("spherical", 20, 300, torch.float32), ("spherical", 128, 40, torch.float32),
    ("diag", 20, 5, torch.float32), ("diag", 64, 300, torch.float32), ("tied", 20, 5, torch.float32),
    ("tied", 20, 300, torch.float32), ("full", 10, 5, torch.float32), ("full", 10, 40, torch.float32),
    ("full", 40, 5, torch.float32), ("spherical", 20, 5, BF), ("spherical", 128, 100, BF), ("spherical", 72, 200, BF),
    ("spherical", 96, 300, BF), ("spherical", 40, 1000, BF), ("spherical", 128, 1024, BF), ("spherical", 40, 1100, BF),
    ("spherical", 128, 1500, BF),
]
VALUES = (float("nan"), float("inf"), -float("inf"), 1e30, 1e18, -3e16)


@pytest.mark.parametrize("cov,d,k,dt", CASES, ids=[f"{c[0]}-D{c[1]}-K{c[2]}-{str(c[3])[6:]}" for c in CASES])
def test_labels_are_components(hip, cov, d, k, dt):
    print(f"[label range] {cov} D={d} K={k} {dt}", flush=True)
    n = 70
    x, means, covs, w = make_problem(cov, 1, max(n, k), d, k, seed=94, dtype=dt)
    x = x[:, :n].contiguous()
    p = [to_dev(t) for t in (means, covs, w)]
    good = hip.score(cov, to_dev(x, dt), *p, want_scores=False)[1].cpu()
    bad = x.clone()
    rows = [11 * i + 1 for i in range(len(VALUES))]
    for row, v in zip(rows, VALUES):
        bad[0, row] = v if abs(v) < 1e20 else bad[0, row]
        bad[0, row, row % d] = v
    keep = torch.ones(n, dtype=torch.bool)
    keep[rows] = False
    for want_scores in (False, True):
        lab = hip.score(cov, to_dev(bad, dt), *p, want_scores=want_scores)[1].cpu()
        assert int(lab.min()) >= 0 and int(lab.max()) < k, lab[0, rows].tolist()
        assert int(lab[0, rows[0]]) == 0
        if not want_scores:
            assert torch.equal(lab[0, keep], good[0, keep])


@pytest.mark.parametrize("d,k", [(72, 50), (72, 200), (96, 300), (40, 900)])
def test_far_rows_take_the_widest_component(hip, d, k):
    """bf16 labels of finite rows at 1e16 per feature: -‖x‖²/2σ² (beyond 1e33, where the
    differences of the other terms are lost) leaves the component of largest σ²; one
    of weight zero is no candidate."""
    print(f"[label range] far rows D={d} K={k}", flush=True)
    x, means, covs, w = make_problem("spherical", 1, max(64, k), d, k, seed=93, dtype=BF)
    covs[0, k - 2], covs[0, k // 2] = 9.0, 4.0
    w[0, k - 2] = 0.0
    x = torch.full((1, 33, d), 1e16).to(BF).float()
    lab = hip.score("spherical", to_dev(x, BF), *[to_dev(t) for t in (means, covs, w)], want_scores=False)[1].cpu()
    assert lab.tolist() == [[k // 2] * 33]
