"""Fits whose workgroups exchange row partials, side by side on several streams and beside
other kernels: a group's members are then not all resident at once, and each fit
waits for its turn and returns what it returns alone (bit for bit)."""

import threading

import pytest
import torch

from gmmxx_amd import em
from tests.test_hip_parity import make_problem, to_dev

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
BF = torch.bfloat16

SHAPES = [(40000, 96, 300), (30000, 40, 700), (20000, 128, 1000)]


def _fit(x, p, k):
    labels, m, c, w, info = em.fit(x, k, "spherical", max_iters=6, tol=0.0, init_means=p[0], init_covs=p[1],
                                   init_weights=p[2])
    return labels, m, c, w, torch.tensor(info["lower_bound_history"])


def test_fits_on_several_streams(hip):
    data = []
    for n, d, k in SHAPES:
        x, *p = make_problem("spherical", 1, n, d, k, seed=92, dtype=BF)
        data.append((to_dev(x, BF), [to_dev(t) for t in p], k))
    alone = [[t.cpu() for t in _fit(*job)] for job in data]
    torch.cuda.synchronize()
    a = torch.randn((4096, 4096), device=DEV)
    stop, failed = threading.Event(), []

    def fits(job, exp):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for i in range(8):
                    got = [t.cpu() for t in _fit(*job)]
                    assert all(torch.equal(g, e) for g, e in zip(got, exp)), f"fit {i} differs"
        except BaseException as e:
            failed.append(e)

    def products():
        with torch.cuda.stream(torch.cuda.Stream()):
            while not stop.is_set():
                a @ a
                torch.cuda.current_stream().synchronize()

    busy = threading.Thread(target=products)
    threads = [threading.Thread(target=fits, args=je) for je in zip(data, alone)]
    print(f"[streams] {len(threads)} fits beside matrix products", flush=True)
    for t in (busy, *threads):
        t.start()
    for t in threads:
        t.join()
    stop.set()
    busy.join()
    if failed:
        raise failed[0]
