"""The reduction and the finalize in one launch (gmmxx_hip_em_step on small statistics)
against the same iteration phase by phase (gmmxx_hip_em_phase, separate launches): the
sums are added in the same order, so parameters and lower bound are bit-equal (for K
up to 256, the launch's limit)."""

import pytest
import torch

from tests.test_hip_parity import make_problem, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [  # cov, B, N, D, K, dtype: one slice, one stage, grouped slices; K = 1 and 256; bf16 single passes
    ("spherical", 1, 20, 3, 1, torch.float32), ("spherical", 2, 3000, 32, 64, torch.float32),
    ("spherical", 1, 100000, 32, 64, torch.float32), ("spherical", 1, 2000, 20, 256, torch.float32),
    ("diag", 3, 900, 50, 40, torch.float32), ("diag", 1, 60000, 64, 100, torch.float32),
    ("tied", 1, 4000, 20, 8, torch.float32), ("tied", 2, 900, 64, 256, torch.float32),
    ("full", 1, 1500, 4, 3, torch.float32), ("full", 16, 4000, 16, 32, torch.float32),
    ("spherical", 1, 5000, 24, 30, torch.bfloat16), ("spherical", 2, 5000, 96, 200, torch.bfloat16),
]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-B{c[1]}-N{c[2]}-D{c[3]}-K{c[4]}" for c in CASES])
def test_one_launch_equals_two(hip, case):
    cov, b, n, d, k, dt = case
    print(f"[finalize] {case}", flush=True)
    x, means, covs, w = make_problem(cov, b, max(n, k), d, k, seed=99, dtype=dt)
    x = x[:, :n].contiguous()
    w[0, 0] = 0.0                      # (the weight floor)
    xd = to_dev(x, dt)
    ws = hip.Workspace(hip.problem(cov, xd.dtype, b, n, d, k), xd.device)
    gram = hip.gram(xd, ws) if cov == "tied" else None
    out = []
    for phases in (False, True):
        p = [to_dev(t) for t in (means, covs, w)]
        lb = torch.zeros(2, device=DEV)
        for it in range(2):
            if phases:
                for ph in hip.EM_PHASES:
                    hip.em_phase(ph, cov, xd, *p, lb[it:it + 1], ws, gram_xx=gram)
            else:
                hip.em_step(cov, xd, *p, lb[it:it + 1], gram_xx=gram, ws=ws)
        out.append([t.cpu() for t in (*p, lb)])
    for one, two in zip(*out):
        assert torch.equal(one, two)
