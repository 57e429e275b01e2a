"""Benchmark of the HIP GMM EM hot path on one MI355X.

Headline: spherical GMM, bf16 inputs with fp32
accumulation, N = 4,194,304, D = 128, K = 1024, one batch.  A "step" is one
soft-EM iteration over all N rows (prelude, E-step log-normaliser,
responsibilities, M-step statistics, finalize) with x resident in HBM;
``value`` is EM iterations per second.

The other BASELINE configs (C1, C3, C4, C5) and the supplementary small-D
large-N bf16 case (C1L) are measured the same way and reported under
``configs`` with their own roofline fractions and CPU baselines.  Data follow
the BASELINE recipes, generated on the device with seeded generators.

Reported per config:
  * iter_per_s / ms_per_iter: wall time of the timed EM iterations, each one
    ``gmmxx_hip_em_step`` call as in the estimator's fit loop;
  * roofline: the dominant kernel's algorithmic rate (FLOP/s, or bytes/s for
    the HBM-bound case) from its launch times, measured with HIP events
    recorded on the stream the kernels are launched on (a second pass over
    the same iterations, one ``gmmxx_hip_em_phase`` call per phase), against
    the MI355X peak of its bound;
  * em_iteration: the whole iteration's algorithmic rate;
  * cpu_baseline: the CPU oracle (a restatement of the reference torch
    fallback) timed on a bounded row sample, scaled linearly to full N.
``roofline.traffic`` (HBM bytes per launch of the dominant kernel) is read
from the committed rocprofv3 FETCH_SIZE/WRITE_SIZE summary when one exists
for that kernel and workload.

``--copy-calibration`` additionally runs a plain 1 GiB device copy, so that a
``rocprofv3 --pmc`` pass over this program can scale the counters by a copy
of known size.
"""

from __future__ import annotations

import argparse
import json
import math
import os
import re
import sys
import time

import torch

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

# MI355X peaks: dense bf16 and fp32 MFMA (TFLOP/s), HBM (GB/s).  "fp32x3" is the
# bound of what the fp32 configs execute: each fp32-accurate product is six
# bf16 MFMAs on three-way bf16 splits of both operands, so their algorithmic
# fp32 FLOPs top out at the bf16 peak / 6.
PEAK = {"bf16": 2516.6, "fp32": 157.3, "fp32x3": 2516.6 / 6.0, "hbm": 8000.0}
PEAK_BASIS = {"bf16": "dense bf16 MFMA peak 2516.6 TFLOP/s", "fp32": "dense fp32 MFMA peak 157.3 TFLOP/s",
              "fp32x3": "dense bf16 MFMA peak / 6 = 419.4 TFLOP/s (six bf16 MFMAs per fp32-accurate product)",
              "hbm": "HBM3E 8 TB/s"}
METRIC = "EM iter/s + % bf16 MFMA peak, spherical bf16 N=4M D=128 K=1024"
HEADLINE = "c2"

CONFIGS = {
    "c1": dict(cov="spherical", B=1, N=100_000, D=32, K=64, dtype="fp32", iters=20, seed=0, bound="fp32x3",
               desc="spherical fp32 N=100000 D=32 K=64, 20 iterations"),
    "c2": dict(cov="spherical", B=1, N=4_194_304, D=128, K=1024, dtype="bf16", iters=10, seed=1, bound="bf16",
               desc="spherical bf16 N=4194304 D=128 K=1024, 10 iterations"),
    "c3": dict(cov="diag", B=1, N=2_097_152, D=64, K=512, dtype="fp32", iters=10, seed=2, bound="fp32x3",
               desc="diag fp32 N=2097152 D=64 K=512, 10 iterations"),
    "c4": dict(cov="tied", B=1, N=1_048_576, D=64, K=256, dtype="fp32", iters=10, seed=3, bound="fp32x3",
               desc="tied fp32 N=1048576 D=64 K=256, 10 iterations"),
    "c5": dict(cov="full", B=16, N=262_144, D=16, K=32, dtype="fp32", iters=10, seed=4, bound="fp32x3",
               desc="full fp32 B=16 N=262144 D=16 K=32, 10 iterations + predict_proba + score_samples"),
    "c1l": dict(cov="spherical", B=1, N=1 << 24, D=32, K=64, dtype="bf16", iters=20, seed=0, bound="hbm",
                desc="spherical bf16 N=16777216 D=32 K=64 (C1 recipe, large N), 20 iterations"),
    # Supplementary (not in the default run, `--only c5w`): full covariance beyond
    # D = 16 on the whitening kernels (split-bf16 operands), C5's recipe at D = 64,
    # one problem.
    "c5w": dict(cov="full", B=1, N=262_144, D=64, K=32, dtype="fp32", iters=10, seed=4, bound="fp32x3",
                desc="full fp32 B=1 N=262144 D=64 K=32 (C5 recipe), 10 iterations"),
}
DEFAULT_CONFIGS = ("c1", "c2", "c3", "c4", "c5", "c1l")
# CPU-baseline samples: rows per batch and oracle iterations, about 10 s of CPU
# work for the headline (C2) and 1-4 s for the others on the GPU box's 16 cores.
CPU_SAMPLE = {"c1": (100_000, 20), "c2": (524_288, 2), "c3": (524_288, 2), "c4": (524_288, 2),
              "c5": (65_536, 2), "c1l": (4_194_304, 2), "c5w": (32_768, 2)}


def flops(cfg):
    """Algorithmic FLOPs of the minimal contractions (E-step logits and M-step
    rᵀ·[x-features | 1]) per EM iteration, split by the kernel computing them.
    Tied: the per-row xᵀPx (2·N·D² per iteration in the reference) is not
    computed by the EM iteration here -- it cancels in the responsibilities
    and the lower bound takes it back as -½·tr(P·XᵀX) -- so it is left out of
    the count rather than credited as work done."""
    b, n, d, k = cfg["B"], cfg["N"], cfg["D"], cfg["K"]
    bn = b * n
    s = d * (d + 1) // 2
    e, m = {
        "spherical": (2 * bn * k * d, 2 * bn * k * (d + 2)),
        "diag": (2 * bn * k * 2 * d, 2 * bn * k * (2 * d + 1)),
        "tied": (2 * bn * k * d, 2 * bn * k * (d + 1)),
        "full": (2 * bn * k * (s + d), 2 * bn * k * (s + d + 1)),
    }[cfg["cov"]]
    return {"lse_tile": float(e), "stats_tile": float(m), "iteration": float(e + m)}


def x_bytes(cfg):
    return cfg["B"] * cfg["N"] * cfg["D"] * (2 if cfg["dtype"] == "bf16" else 4)


# ---------------------------------------------------------------------------
# Synthetic data (BASELINE.json recipes), generated on the device
# ---------------------------------------------------------------------------

def _chunks(n, size=1 << 20):
    for s in range(0, n, size):
        yield s, min(n, s + size)


def _distinct_rows(x, k, g):
    idx = torch.randperm(x.shape[1], generator=g, device=x.device)[:k]
    return x[:, idx].to(torch.float32).contiguous()


def _global_spherical_var(x, k, reg=1e-6):
    b, n, d = x.shape
    out = []
    for bi in range(b):
        s1 = torch.zeros(d, dtype=torch.float64, device=x.device)
        s2 = torch.zeros((), dtype=torch.float64, device=x.device)
        for s, e in _chunks(n):
            xf = x[bi, s:e].to(torch.float64)
            s1 += xf.sum(0)
            s2 += xf.square().sum()
        mean = s1 / n
        out.append(max(float(((s2 / n) - mean.square().sum()).clamp_min(0.0) / d), reg))
    return torch.tensor(out, dtype=torch.float32, device=x.device)[:, None].expand(b, k).contiguous()


def _global_cov(x, reg=1e-6):
    xf = x.to(torch.float64)
    c = xf - xf.mean(dim=1, keepdim=True)
    cov = torch.bmm(c.transpose(1, 2), c) / x.shape[1]
    cov = 0.5 * (cov + cov.transpose(1, 2)) + reg * torch.eye(x.shape[2], device=x.device, dtype=torch.float64)
    return cov.to(torch.float32)


def make_data(name, device, n=None):
    """(x, initial means, covariances, weights) of a config's recipe; ``n``
    overrides the row count per problem (the parity tests run the recipes at
    sizes the CPU oracle finishes in seconds)."""
    cfg = CONFIGS[name]
    b, d, k = cfg["B"], cfg["D"], cfg["K"]
    n = cfg["N"] if n is None else int(n)
    g = torch.Generator(device=device).manual_seed(cfg["seed"])
    xdt = torch.bfloat16 if cfg["dtype"] == "bf16" else torch.float32
    x = torch.empty((b, n, d), dtype=xdt, device=device)
    w0 = torch.full((b, k), 1.0 / k, dtype=torch.float32, device=device)
    if name in ("c1", "c1l"):
        # K centres ~ U[-10, 10]^D, balanced labels (n mod K) permuted, unit noise;
        # means = first K rows, variances 1, weights 1/K.
        centers = torch.rand((k, d), generator=g, device=device) * 20.0 - 10.0
        lab = (torch.arange(n, device=device) % k)[torch.randperm(n, generator=g, device=device)]
        for s, e in _chunks(n):
            x[0, s:e] = (centers[lab[s:e]] + torch.randn((e - s, d), generator=g, device=device)).to(xdt)
        means0 = x[:, :k].to(torch.float32).contiguous()
        covs0 = torch.ones((b, k), dtype=torch.float32, device=device)
    elif name == "c2":
        # centres ~ N(0, 4I), std ~ U[0.5, 1.5], Dirichlet(1) weights, multinomial labels;
        # means = K distinct random rows, global spherical variance, weights 1/K.
        centers = 2.0 * torch.randn((k, d), generator=g, device=device)
        sigma = 0.5 + torch.rand((k,), generator=g, device=device)
        w = -torch.log(torch.rand((k,), generator=g, device=device))
        lab = torch.multinomial(w / w.sum(), n, replacement=True, generator=g)
        for s, e in _chunks(n):
            noise = torch.randn((e - s, d), generator=g, device=device)
            x[0, s:e] = (centers[lab[s:e]] + sigma[lab[s:e], None] * noise).to(xdt)
        means0 = _distinct_rows(x, k, g)
        covs0 = _global_spherical_var(x, k)
    elif name == "c3":
        # centres ~ U[-8, 8]^D, per-dimension std log-uniform in [0.5, 2], equal weights;
        # means = K distinct random rows, global per-feature variance, weights 1/K.
        centers = torch.rand((k, d), generator=g, device=device) * 16.0 - 8.0
        lo, hi = math.log(0.5), math.log(2.0)
        sigma = torch.exp(lo + (hi - lo) * torch.rand((k, d), generator=g, device=device))
        lab = torch.randint(0, k, (n,), generator=g, device=device)
        for s, e in _chunks(n):
            noise = torch.randn((e - s, d), generator=g, device=device)
            x[0, s:e] = centers[lab[s:e]] + sigma[lab[s:e]] * noise
        means0 = _distinct_rows(x, k, g)
        xf = x[0].to(torch.float64)
        gv = (xf - xf.mean(0)).square().mean(0).clamp_min(1e-6).to(torch.float32)
        covs0 = gv[None, None].expand(b, k, d).contiguous()
    elif name == "c4":
        # Σ = AAᵀ/D + 0.1I, A ~ N(0,1)^{DxD}; centres ~ N(0, 9I); equal weights;
        # x = c + chol(Σ)·z; means = K distinct random rows, global covariance, weights 1/K.
        a = torch.randn((d, d), generator=g, device=device, dtype=torch.float64)
        sig = a @ a.T / d + 0.1 * torch.eye(d, device=device, dtype=torch.float64)
        chol = torch.linalg.cholesky(sig).to(torch.float32)
        centers = 3.0 * torch.randn((k, d), generator=g, device=device)
        lab = torch.randint(0, k, (n,), generator=g, device=device)
        for s, e in _chunks(n):
            z = torch.randn((e - s, d), generator=g, device=device)
            x[0, s:e] = centers[lab[s:e]] + z @ chol.T
        means0 = _distinct_rows(x, k, g)
        covs0 = _global_cov(x)
    elif name in ("c5", "c5w"):
        # per problem and component L lower-triangular ~ N(0, 0.5²), Σ = LLᵀ + 0.05I;
        # centres ~ U[-6, 6]^D; Dirichlet(2) weights; means = K distinct rows per
        # problem, the problem's global covariance for every component, weights 1/K.
        L = torch.tril(0.5 * torch.randn((b, k, d, d), generator=g, device=device, dtype=torch.float64))
        sig = L @ L.transpose(-1, -2) + 0.05 * torch.eye(d, device=device, dtype=torch.float64)
        chol = torch.linalg.cholesky(sig).to(torch.float32)
        centers = torch.rand((b, k, d), generator=g, device=device) * 12.0 - 6.0
        u = torch.rand((b, k, 2), generator=g, device=device)
        w = -torch.log(u).sum(-1)
        means0 = torch.empty((b, k, d), dtype=torch.float32, device=device)
        for bi in range(b):
            lab = torch.multinomial(w[bi] / w[bi].sum(), n, replacement=True, generator=g)
            z = torch.randn((n, d), generator=g, device=device)
            x[bi] = centers[bi, lab] + torch.einsum("nde,ne->nd", chol[bi, lab], z)
            means0[bi] = x[bi, torch.randperm(n, generator=g, device=device)[:k]]
        covs0 = _global_cov(x)[:, None].expand(b, k, d, d).contiguous()
    else:
        raise KeyError(name)
    return x, means0, covs0, w0


# ---------------------------------------------------------------------------
# Measurement
# ---------------------------------------------------------------------------

def _traffic_from_profile(name, phase):
    """HBM bytes per launch of (config, phase) from the committed rocprofv3
    FETCH_SIZE / WRITE_SIZE summary, or None."""
    path = os.path.join(ROOT, "profiles", f"tile_{name}_hbm_traffic.txt")
    if not os.path.exists(path):
        return None
    vals = {}
    for line in open(path):
        m = re.match(r"\s*(\w+)\s*=\s*([0-9.eE+-]+)\s*$", line)
        if m:
            vals[m.group(1)] = float(m.group(2))
    key = f"{phase}_bytes_per_launch"
    return vals.get(key)


def single_pass(cfg):
    """Kernel of a one-pass EM iteration for this config, or None (two passes);
    mirrors the library's plan (gmmxx_amd/csrc/abi.hip)."""
    if cfg["cov"] == "spherical" and cfg["dtype"] == "bf16":
        if cfg["D"] <= 64 and cfg["K"] <= 64:
            return "sph_bf16_fused_kernel"
        if cfg["K"] <= 1024 and os.environ.get("GMMXX_HIP_NO_COOP") != "1":
            return "sph_bf16_coop_kernel" if cfg["K"] > 256 else "sph_bf16_one_kernel"
        return None
    if cfg["cov"] == "full" and cfg["D"] > 16:
        return None   # whitening E-step, then the statistics kernel
    # fp32 x: one tile pass when a workgroup (8 waves of CW components) holds all K;
    # with 2..4 such component tiles (spherical, tied, diag at D <= 64) the tiles
    # exchange row partials in one cooperative pass
    cw = 16 if cfg["cov"] == "full" or (cfg["cov"] == "diag" and cfg["D"] > 64) else 32
    one_tile = cfg["K"] <= 8 * cw and not (cfg["cov"] == "diag" and cfg["D"] > 64)
    if one_tile and os.environ.get("GMMXX_HIP_NO_SINGLE") != "1":
        return "em_tile_kernel"
    xch = (8 * cw < cfg["K"] <= 32 * cw and (cfg["cov"] in ("spherical", "tied") or
                                             (cfg["cov"] == "diag" and cfg["D"] <= 64)))
    if xch and os.environ.get("GMMXX_HIP_NO_XCH") != "1":
        return "em_tile_kernel (exchange)"
    return None


def kernel_label(cfg, phase):
    """Name of the kernel that runs in `phase` for this config (see gmmxx_amd/csrc)."""
    if cfg["cov"] == "full" and cfg["D"] > 16:
        if phase == "lse_tile":
            return "fw_estep_kernel"
        return "fw_stats_tile_kernel" if cfg["K"] > 8 else "fw_stats_kernel"
    one = single_pass(cfg)
    if one:
        return f"{one} (single pass)"
    if cfg["cov"] == "spherical" and cfg["dtype"] == "bf16":
        return f"sph_bf16_kernel ({phase})"
    return f"em_tile_kernel ({phase})"


def run_config(name, dev, steps=None, warmup=2, copy_calibration=False):
    from gmmxx_amd import _hip
    cfg = CONFIGS[name]
    steps = cfg["iters"] if steps is None else steps
    cov = cfg["cov"]
    print(f"[bench] {name}: generating data ({cfg['desc']})", file=sys.stderr, flush=True)
    x, means0, covs0, w0 = make_data(name, dev)
    b, n, d, k = cfg["B"], cfg["N"], cfg["D"], cfg["K"]
    prob = _hip.problem(cov, x.dtype, b, n, d, k)
    ws = _hip.Workspace(prob, dev)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    gram = _hip.gram(x, ws) if cov == "tied" else None
    torch.cuda.synchronize()
    setup_ms = 1e3 * (time.perf_counter() - t0)
    lb = torch.zeros((max(1, steps + warmup),), dtype=torch.float32, device=dev)
    phases = _hip.EM_PHASES
    means, covs, w = means0.clone(), covs0.clone(), w0.clone()

    def step(i, events=None):
        for j, ph in enumerate(phases):
            if events is not None:
                events[j].record()
            _hip.em_phase(ph, cov, x, means, covs, w, lb[i:i + 1], ws, gram_xx=gram)
        if events is not None:
            events[len(phases)].record()

    print(f"[bench] {name}: warmup {warmup}", file=sys.stderr, flush=True)
    for i in range(warmup):
        step(i)
    # The timed iterations start from the initial parameters again: one fit's EM loop.
    means.copy_(means0)
    covs.copy_(covs0)
    w.copy_(w0)
    # Timed: the product's EM loop, one gmmxx_hip_em_step call per iteration.
    print(f"[bench] {name}: timing {steps} EM iterations", file=sys.stderr, flush=True)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(steps):
        _hip.em_step(cov, x, means, covs, w, lb[warmup + i:warmup + i + 1], gram_xx=gram, ws=ws)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    ms_per_step = 1e3 * wall / steps
    lb_last = float(lb[warmup + steps - 1].item())
    # Per-phase kernel times (HIP events on the launch stream) from a second pass
    # over the same iterations, one gmmxx_hip_em_phase call per phase.
    means.copy_(means0)
    covs.copy_(covs0)
    w.copy_(w0)
    evs = [[torch.cuda.Event(enable_timing=True) for _ in range(len(phases) + 1)] for _ in range(steps)]
    for i in range(steps):
        step(warmup + i, evs[i])
    torch.cuda.synchronize()
    phase_ms = {ph: sum(e[j].elapsed_time(e[j + 1]) for e in evs) / steps for j, ph in enumerate(phases)}
    fl = flops(cfg)
    dominant = max(("lse_tile", "stats_tile"), key=lambda p: phase_ms[p])
    bound = cfg["bound"]
    if bound == "hbm":
        # Each tile pass must read x once: the algorithmic bytes of one launch.
        achieved = x_bytes(cfg) / (phase_ms[dominant] * 1e-3) / 1e9
        unit = "GB/s"
        it_rate = x_bytes(cfg) / (ms_per_step * 1e-3) / 1e9
        it_unit = "GB/s (x read once per iteration)"
    else:
        # A single-pass kernel does the E- and M-step contractions in one launch.
        work = fl["iteration"] if single_pass(cfg) else fl[dominant]
        achieved = work / (phase_ms[dominant] * 1e-3) / 1e12
        unit = "TFLOP/s"
        it_rate = fl["iteration"] / (ms_per_step * 1e-3) / 1e12
        it_unit = "TFLOP/s"
    peak = PEAK[bound]
    out = {
        "config": cfg["desc"], "covariance_type": cov, "B": b, "N": n, "D": d, "K": k, "dtype": cfg["dtype"],
        "steps": steps, "warmup": warmup, "ms_per_iter": ms_per_step, "iter_per_s": 1e3 / ms_per_step,
        "gflop_per_s": fl["iteration"] / (ms_per_step * 1e-3) / 1e9,
        "roofline": {"bound": "hbm" if bound == "hbm" else "mfma", "peak_kind": bound,
                     "peak_basis": PEAK_BASIS[bound],
                     "kernel": kernel_label(cfg, dominant), "achieved": achieved, "peak": peak, "unit": unit,
                     "frac": achieved / peak, "traffic": _traffic_from_profile(name, dominant)},
        "em_iteration": {"algorithmic_tflop": fl["iteration"] / 1e12, "achieved": it_rate, "unit": it_unit,
                         "frac": it_rate / peak, "phase_ms": phase_ms},
        "setup_ms": setup_ms,
        "lower_bound_last": lb_last,
    }
    if bound == "fp32x3":
        # the same rate against the fp32 MFMA peak, for comparison with fp32-only engines
        out["roofline"]["fp32_peak_frac"] = achieved / PEAK["fp32"]
    if name == "c5":
        # Tail of the config: predict_proba + score_samples on all points, from
        # one E-step (gmmxx_hip_predict_proba_score).
        for _ in range(2):
            _hip.predict_proba_score(cov, x, means, covs, w, ws=ws)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        reps = 5
        for _ in range(reps):
            _hip.predict_proba_score(cov, x, means, covs, w, ws=ws)
        torch.cuda.synchronize()
        tail_ms = 1e3 * (time.perf_counter() - t0) / reps
        out["tail"] = {"ms": tail_ms, "what": "predict_proba (B,N,K fp32 written) + score_samples, one E-step",
                       "proba_write_gb_per_s": b * n * k * 4 / (tail_ms * 1e-3) / 1e9,
                       "hbm_frac": (x_bytes(cfg) + b * n * (k + 1) * 4) / (tail_ms * 1e-3) / 1e9 / PEAK["hbm"]}
    if copy_calibration:
        src = torch.empty(1 << 28, dtype=torch.float32, device=dev).fill_(1.0)
        dst = torch.empty_like(src)
        for _ in range(3):
            dst.copy_(src)
        torch.cuda.synchronize()
        out["copy_calibration"] = {"bytes_read": src.numel() * 4, "bytes_written": dst.numel() * 4, "launches": 3}
    return out, (x, means0, covs0, w0)


def _cpu_facts():
    """(threads to use, description): the CPUs this process may run on, capped by
    the cgroup CPU quota when one is set; the CPU model from /proc/cpuinfo."""
    try:
        usable = len(os.sched_getaffinity(0))
    except AttributeError:
        usable = os.cpu_count() or 1
    quota = None
    try:
        q, period = open("/sys/fs/cgroup/cpu.max").read().split()[:2]
        if q != "max":
            quota = max(1, int(int(q) // int(period)))
    except (OSError, ValueError):
        pass
    threads = min(usable, quota) if quota else usable
    model = "unknown"
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return threads, {"model": model, "logical_cpus": os.cpu_count(), "affinity_cpus": usable,
                     "cgroup_cpu_quota": quota}


def cpu_baseline(name, data):
    """Oracle EM iterations on the first rows of each problem (fp32 on the
    same values; bf16 x keeps its means in bf16), scaled linearly in N to the
    full workload.  Also returns the oracle's result on that sample, which the
    parity leg compares against."""
    from oracle import torch_ref
    cfg = CONFIGS[name]
    rows, iters = CPU_SAMPLE[name]
    x, m0, c0, w0 = data
    rows = min(rows, cfg["N"])
    threads, facts = _cpu_facts()
    torch.set_num_threads(threads)
    xs = x[:, :rows].to(torch.float32).cpu()
    m, c, w = m0.cpu(), c0.cpu(), w0.cpu()
    bf = x.dtype == torch.bfloat16
    torch_ref.fit(xs[:, :min(rows, 4096)], cfg["K"], cfg["cov"], max_iters=1, tol=0.0, init_means=m,
                  init_covs=c, init_weights=w, compute_labels=False, bf16_means=bf)  # warm the thread pool
    t0 = time.perf_counter()
    ref = torch_ref.fit(xs, cfg["K"], cfg["cov"], max_iters=iters, tol=0.0, init_means=m, init_covs=c,
                        init_weights=w, compute_labels=False, bf16_means=bf)
    dt = (time.perf_counter() - t0) / iters
    full_iter_s = dt * (cfg["N"] / rows)
    sample = ("the full workload" if rows == cfg["N"] else
              f"the first {rows} of {cfg['N']} rows per problem, scaled linearly in N")
    out = {"value": 1.0 / full_iter_s, "unit": "EM iter/s", "cores": torch.get_num_threads(),
           "kind": "port", "cpu": facts,
           "sample": f"{iters} oracle EM iterations on {sample} ({dt:.3f} s per sampled iteration)"}
    return out, (rows, iters, ref)


def parity(name, data, sample):
    """Part of the CPU-baseline leg, as the checker: one GPU fit (em_step per
    iteration) on that leg's row sample from the same initial parameters,
    judged against the oracle's fit of the sample by oracle/judge.py --
    per-iteration mean log-likelihood rtol 1e-5 (fp32) / 2e-3 (bf16); fp32
    parameters element-wise rtol 1e-4 with floors 1e-5·rms(x) (means),
    1e-5·mean(x²) (covariances), 1e-7 (weights); values outside the bar count
    as explained when HIP is at least as close to a float64 fit from the same
    start as the oracle is (judge.arbiter_params_ok: largest error within 2x
    the oracle's; where the oracle itself misses the bar against float64, the
    distribution rule).  For bf16 x the bar is the log-likelihood (the means,
    bf16 on both sides, are reported against one bf16 ulp)."""
    from gmmxx_amd import em
    from oracle import f64_em, judge
    cfg = CONFIGS[name]
    rows, iters, (_, e_m, e_c, e_w, e_info) = sample
    x, m0, c0, w0 = data
    xs = x[:, :rows].contiguous()
    _, m, c, w, info = em.fit(xs, cfg["K"], cfg["cov"], max_iters=iters, tol=0.0, init_means=m0, init_covs=c0,
                              init_weights=w0, compute_labels=False, record_all_lower_bounds=True)
    bf = cfg["dtype"] == "bf16"
    xc = xs.float().cpu()
    truth = []

    def t64():
        if not truth:
            truth.extend(f64_em.trajectory(xc, cfg["cov"], m0.cpu(), c0.cpu(), w0.cpu(), iters))
        return truth

    ll = judge.judge_ll(info["lower_bound_history"], e_info["lower_bound_history"], 2e-3 if bf else 1e-5,
                        lambda: t64()[0])
    res = {"rows": rows, "iters": iters, "lower_bound_hip": info["lower_bound_history"],
           "lower_bound_oracle": e_info["lower_bound_history"], "lower_bound": ll}
    ok = ll["unexplained"] == 0
    for got, exp, kind, j in ((m, e_m, "means", 1), (c, e_c, "covs", 2), (w, e_w, "weights", 3)):
        r = judge.judge_params(got, exp, kind, xc, bf, None if bf else (lambda j=j: t64()[j]))
        res[kind] = r
        ok = ok and (bf or r["unexplained"] == 0)
    res["pass"] = bool(ok)
    return res


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20, help="timed EM iterations of the headline config")
    ap.add_argument("--warmup", type=int, default=3)
    ap.add_argument("--only", default=None, help="comma-separated configs (default: all)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--copy-calibration", action="store_true")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path; the EM iteration "
              "would shard over rows with one all-reduce of the statistics. Run with --gpus 1.",
              file=sys.stderr)
        sys.exit(2)

    from gmmxx_amd import _hip
    _hip.require_hip()
    dev = torch.device("cuda:0")
    names = args.only.split(",") if args.only else list(DEFAULT_CONFIGS)
    for nm in names:
        if nm not in CONFIGS:
            sys.exit(f"unknown config {nm!r}; choose from {sorted(CONFIGS)}")
    results = {}
    for nm in names:
        steps = args.steps if nm == HEADLINE else None
        res, data = run_config(nm, dev, steps=steps, warmup=args.warmup,
                               copy_calibration=args.copy_calibration and nm == names[-1])
        if not args.no_cpu_baseline:
            print(f"[bench] {nm}: cpu baseline", file=sys.stderr, flush=True)
            res["cpu_baseline"], sample = cpu_baseline(nm, data)
            print(f"[bench] {nm}: parity on the cpu-baseline sample", file=sys.stderr, flush=True)
            res["parity"] = parity(nm, data, sample)
        del data
        torch.cuda.empty_cache()
        results[nm] = res
        print(f"[bench] {nm}: {res['ms_per_iter']:.3f} ms/iter, {res['roofline']['kernel']} "
              f"{100 * res['roofline']['frac']:.1f}% of {res['roofline']['peak_kind']} peak",
              file=sys.stderr, flush=True)

    head = results.get(HEADLINE) or results[names[0]]
    head_name = HEADLINE if HEADLINE in results else names[0]
    cfg = CONFIGS[head_name]
    result = {
        "metric": METRIC if head_name == HEADLINE else f"EM iter/s, {cfg['desc']}",
        "value": head["iter_per_s"], "unit": "EM iter/s", "n_gpus": 1,
        "steps": head["steps"], "warmup": head["warmup"], "ms_per_step": head["ms_per_iter"],
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": cfg["dtype"],
        "data": f"synthetic (BASELINE config recipe, seed {cfg['seed']}, generated on device)",
        "config": {"workload": f"GMM soft-EM iteration: {cfg['desc'].split(',')[0]}",
                   "covariance_type": cfg["cov"], "B": cfg["B"], "N": cfg["N"], "D": cfg["D"], "K": cfg["K"],
                   "parallelism": "single GPU"},
        "roofline": {kk: v for kk, v in head["roofline"].items() if kk != "peak_kind"},
        "em_iteration": head["em_iteration"],
    }
    if "cpu_baseline" in head:
        result["cpu_baseline"] = head["cpu_baseline"]
    if "parity" in head:
        result["parity"] = head["parity"]
    result["configs"] = results
    print(json.dumps(result), flush=True)


if __name__ == "__main__":
    main()
