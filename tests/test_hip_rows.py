"""Rows of any width through the fp32 tile kernels (16-byte loads at element-aligned
addresses, the tail of a row shifted into place) and the label pass without
exponentials: statistics against the oracle (rtol 1e-4 of the statistic's scale, as
test_hip_parity), labels alone bit-equal to the labels that come with the scores."""

import pytest
import torch

from oracle import torch_ref
from tests.test_hip_parity import assert_labels, make_problem, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _close(got, exp, tol=1e-4):
    torch.testing.assert_close(got.cpu(), exp, rtol=tol, atol=tol * max(1e-30, float(exp.abs().max())))


def _unaligned(t):
    """The same values from a buffer that starts one element past a 16-byte boundary."""
    buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
    return buf[1:].copy_(t.reshape(-1)).view(t.shape)


@pytest.mark.parametrize("cov", ["spherical", "diag", "tied", "full"])
@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 6, 7, 15, 16, 17, 31, 50, 63, 65, 100, 127])
@pytest.mark.parametrize("n,k", [(1, 2), (33, 3), (900, 40), (700, 300)])
def test_any_row_width(hip, cov, d, n, k):
    if cov == "full" and (k > 40 or (d > 65 and k > 3)):
        pytest.skip("covered by the smaller component counts")
    print(f"[rows] {cov} N={n} D={d} K={k}", flush=True)
    x, means, covs, w = make_problem(cov, 2, max(n, 8), d, k, seed=81)
    x = x[:, :n].contiguous()
    xd = to_dev(x)
    nk, sx, sq, ll = hip.estep_stats(cov, xd, to_dev(means), to_dev(covs), to_dev(w))
    e_nk, e_sx, e_sq, e_ll = torch_ref.estep_stats(x, cov, means, covs, w)
    _close(nk, e_nk)
    _close(sx, e_sx)
    if sq is not None:
        _close(sq, e_sq)
    assert float(ll) == pytest.approx(float(e_ll), rel=1e-5, abs=1e-4)
    _, both = hip.score(cov, xd, to_dev(means), to_dev(covs), to_dev(w))
    _, only = hip.score(cov, xd, to_dev(means), to_dev(covs), to_dev(w), want_scores=False)
    if cov != "tied":    # (the tied label pass leaves out the row constant xᵀPx: other roundings, same order)
        assert torch.equal(only, both)
    assert_labels(only, x, means, covs, w, cov, 1e-5)


@pytest.mark.parametrize("cov", ["spherical", "diag", "tied", "full"])
def test_rows_off_a_16_byte_boundary(hip, cov):
    """The C entry accepts rows at any element address (the Python wrapper copies such views)."""
    import ctypes
    n, d, k = 500, 16, 20
    x, means, covs, w = make_problem(cov, 1, n, d, k, seed=82)
    xd = _unaligned(to_dev(x))
    prob = hip.problem(cov, torch.float32, 1, n, d, k)
    ws = hip.Workspace(prob, xd.device)
    p = [to_dev(t) for t in (means, covs, w)]
    labels = torch.empty((1, n), dtype=torch.int64, device=DEV)
    rc = hip.load_library().gmmxx_hip_score(
        ctypes.byref(prob), ctypes.c_void_p(xd.data_ptr()), *(ctypes.c_void_p(t.data_ptr()) for t in p), None,
        ctypes.c_void_p(labels.data_ptr()), ws.ptr, ws.nbytes,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, hip.last_error()
    assert_labels(labels, x, means, covs, w, cov, 1e-5)


@pytest.mark.parametrize("cov,d,k", [("spherical", 3, 300), ("spherical", 16, 600), ("spherical", 32, 300),
                                     ("diag", 21, 300), ("tied", 32, 900), ("spherical", 64, 300)])
def test_exchange_rows_off_a_16_byte_boundary(hip, cov, d, k):
    """Several component tiles: the statistics of rows at any element address are those of
    the same rows on a boundary (which D = 16 and 32 read whole), bit for bit."""
    import ctypes
    n = 1000
    x, means, covs, w = make_problem(cov, 1, n, d, k, seed=83)
    xd = to_dev(x)
    p = [to_dev(t) for t in (means, covs, w)]
    exp = hip.estep_stats(cov, xd, *p)
    xu = _unaligned(xd)
    prob = hip.problem(cov, torch.float32, 1, n, d, k)
    ws = hip.Workspace(prob, xd.device)
    got = [None if t is None else torch.empty_like(t) for t in exp]
    ptr = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())      # noqa: E731
    rc = hip.load_library().gmmxx_hip_estep_stats(
        ctypes.byref(prob), ptr(xu), *map(ptr, p), 1e-6, 1e-8, *map(ptr, got), ws.ptr, ws.nbytes,
        ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, hip.last_error()
    for a, e in zip(got, exp):
        assert e is None or torch.equal(a, e)
