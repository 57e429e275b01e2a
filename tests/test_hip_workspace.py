"""A workspace is used as allocated: every byte but the exchange's status words (cleared by
gmmxx_hip_workspace_init) is written before it is read, so results do not depend on
what the memory held (bit-equal on NaN patterns, huge values and zeros)."""

import ctypes

import pytest
import torch

from tests.test_hip_parity import make_problem, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"

CASES = [
    ("spherical", 1, 3000, 32, 64, torch.float32), ("spherical", 1, 3000, 20, 700, torch.float32),
    ("spherical", 1, 2000, 40, 1100, torch.float32), ("diag", 2, 2000, 50, 100, torch.float32),
    ("diag", 1, 2000, 64, 300, torch.float32), ("tied", 1, 3000, 20, 8, torch.float32),
    ("full", 2, 1500, 16, 20, torch.float32), ("full", 1, 1500, 40, 20, torch.float32),
    ("full", 1, 1000, 100, 3, torch.float32), ("spherical", 1, 3000, 32, 30, torch.bfloat16),
    ("spherical", 1, 3000, 96, 200, torch.bfloat16), ("spherical", 1, 3000, 96, 600, torch.bfloat16),
    ("spherical", 1, 2000, 128, 1500, torch.bfloat16),
]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-N{c[2]}-D{c[3]}-K{c[4]}" for c in CASES])
def test_results_do_not_depend_on_the_memory(hip, case):
    cov, b, n, d, k, dt = case
    print(f"[workspace] {case}", flush=True)
    x, means, covs, w = make_problem(cov, b, n, d, k, seed=98, dtype=dt)
    xd = to_dev(x, dt)
    prob = hip.problem(cov, xd.dtype, b, n, d, k)
    runs = []
    for fill in (0x00, 0xFF, 0x7E):
        ws = hip.Workspace(prob, xd.device)
        ws._buf.fill_(fill)
        if ws.exchanges:
            assert hip.load_library().gmmxx_hip_workspace_init(
                ctypes.byref(prob), ws.ptr, ws.nbytes,
                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
        gram = hip.gram(xd, ws) if cov == "tied" else None
        p = [to_dev(t) for t in (means, covs, w)]
        lb = torch.zeros(2, device=DEV)
        for it in range(2):
            hip.em_step(cov, xd, *p, lb[it:it + 1], gram_xx=gram, ws=ws)
        out = [*p, lb, *hip.score(cov, xd, *p, ws=ws), hip.score(cov, xd, *p, want_scores=False, ws=ws)[1],
               hip.predict_proba(cov, xd, *p, ws=ws), *(s for s in hip.estep_stats(cov, xd, *p, ws=ws) if s is not None)]
        assert int(hip.take_status(ws).item()) == 0
        runs.append([t.cpu() for t in out])
    for other in runs[1:]:
        for a, e in zip(other, runs[0]):
            assert torch.equal(a, e)
