"""gmmxx_hip_em_step_noalloc on problems whose usual plan needs more than the 64 MiB
scratch and whose leaner one (two passes, the per-component statistics)
does not: accepted, and the iteration agrees with the workspace entry's to the bars
of test_hip_parity (fp32 1e-4, bf16 2e-3 of the parameter's scale)."""

import pytest
import torch

from tests.test_hip_parity import make_problem, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16

CASES = [  # cov, B, N, D, K, dtype
    ("spherical", 1, 1594715, 88, 47, BF),          # one workgroup per slice: more slices than two passes
    ("spherical", 107, 725, 45, 547, BF),           # groups that exchange: their words and operands
    ("spherical", 127, 54, 108, 236, BF),           # and one-block slices
    ("spherical", 33, 4354, 128, 562, BF),          # exchanging groups, one item per problem
    ("full", 1, 10535, 75, 94, torch.float32),      # 16-component statistics
]


@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-B{c[1]}-N{c[2]}-D{c[3]}-K{c[4]}" for c in CASES])
def test_accepted_with_the_lean_plan(hip, case):
    cov, b, n, d, k, dt = case
    print(f"[scratch] {cov} B={b} N={n} D={d} K={k} {dt}", flush=True)
    prob = hip.problem(cov, dt, b, n, d, k)
    assert hip.load_library().gmmxx_hip_workspace_bytes(prob) > hip.NOALLOC_SCRATCH_BYTES
    x, means, covs, w = make_problem(cov, b, n, d, k, seed=90, dtype=dt)
    xd = to_dev(x, dt)
    out = []
    for fn in (hip.em_step, hip.em_step_noalloc):
        par = [to_dev(t) for t in (means, covs, w)]
        lb = torch.zeros(1, device=DEV)
        fn(cov, xd, *par, lb)
        out.append([t.cpu() for t in (*par, lb)])
    tol = 2e-3 if dt == BF else 1e-4
    for got, exp in zip(out[1], out[0]):
        torch.testing.assert_close(got, exp, rtol=tol, atol=tol * float(exp.abs().max()))
