"""Benchmark of the KernelSwift operators on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--configs 2,1,3,4,5,mhc,fp8] [--no-cpu] [--no-dropin]

Headline (the JSON "value"): BASELINE.json configs[1] = config 2, the indexer at S_q=128, S_kv=4096,
64 heads, top-512: one step = one fused indexer call (RoPE of q and k + row statistics, exact MFMA
scores, exact top-k) on inputs already resident in HBM.  value = median device time per call
(HIP events around each call on the launch stream); the auto_bench-style wall median (perf_counter +
synchronize per call) is reported beside it.  ms_per_step = wall time of the K back-to-back timed
steps / K, bracketed by synchronize on both sides.

roofline: the dominant kernel of the step (indexer_scores_kernel), timed alone with HIP events over
K launches on the same stream: achieved = algorithmic flops per launch (2*S*H*T*D) / average launch
duration, against the published dense bf16 MFMA peak (2.5 PFLOP/s).  traffic = HBM bytes per launch
from the rocprofv3 FETCH_SIZE/WRITE_SIZE runs recorded in profiles/traffic.json (null if absent).

cpu_baseline: the torch-CPU op-for-op restatement of the reference baseline (oracle/torch_ref.py,
kind "port") timed on this host's cores over a bounded sample of the same workload.

The other configs (Sinkhorn, sparse attention prefill, indexer long, MLA decode) are measured the same
way and reported under "per_config", with two rows beyond the BASELINE.json configs: "mhc" (the mHC
residual update with the Sinkhorn fused in, HBM-bound) and "fp8" (the indexer on e4m3 rows at config 2's
shape, with the HBM-bound quantiser as its roofline).
"""
from __future__ import annotations

import argparse
import json
import os
import statistics
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

PEAK_BF16_TFLOPS = 2500.0   # MI355X dense bf16 MFMA, published
PEAK_HBM_GBS = 8000.0       # MI355X HBM3E, published


def parse():
    p = argparse.ArgumentParser()
    p.add_argument("--gpus", type=int, default=1)
    p.add_argument("--steps", type=int, default=200)
    p.add_argument("--warmup", type=int, default=20)
    p.add_argument("--configs", type=str, default="2,1,3,4,5,mhc,fp8")
    p.add_argument("--no-cpu", action="store_true", help="skip the host-CPU baseline")
    p.add_argument("--no-dropin", action="store_true", help="skip the ModelNew rows at the reference example shapes")
    p.add_argument("--cpu-seconds", type=float, default=10.0, help="budget per CPU baseline sample")
    p.add_argument("--calib-copy", action="store_true",
                   help="also run the 512 MiB calibration copy kernel (for rocprofv3 FETCH/WRITE scaling)")
    return p.parse_args()


def _events_median(fn, steps, warmup):
    """Median and mean device time (us) per call of fn, HIP events around each call on the current stream."""
    import torch
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    starts = [torch.cuda.Event(enable_timing=True) for _ in range(steps)]
    ends = [torch.cuda.Event(enable_timing=True) for _ in range(steps)]
    for i in range(steps):
        starts[i].record()
        fn()
        ends[i].record()
    torch.cuda.synchronize()
    us = [s.elapsed_time(e) * 1e3 for s, e in zip(starts, ends)]
    return statistics.median(us), statistics.fmean(us)


def _events_avg(fn, steps, warmup):
    """Average device time (us) per launch over `steps` back-to-back launches (one event pair)."""
    import torch
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    a.record()
    for _ in range(steps):
        fn()
    b.record()
    torch.cuda.synchronize()
    return a.elapsed_time(b) * 1e3 / steps


def _wall(fn, steps, warmup):
    """auto_bench semantics: per call perf_counter + synchronize, median (us); and the bracketed
    back-to-back total per step (ms)."""
    import torch
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize()
    samples = []
    for _ in range(steps):
        t0 = time.perf_counter()
        fn()
        torch.cuda.synchronize()
        samples.append((time.perf_counter() - t0) * 1e6)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        fn()
    torch.cuda.synchronize()
    total_ms = (time.perf_counter() - t0) * 1e3
    return statistics.median(samples), total_ms / steps


def _host_issue_us(fn, n=200):
    """Host time (us) to issue one call: n calls back to back, timed before the final synchronize."""
    import torch
    for _ in range(20):
        fn()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(n):
        fn()
    t1 = time.perf_counter()
    torch.cuda.synchronize()
    return (t1 - t0) * 1e6 / n


def _cpu_time(fn, budget_s, min_reps=3, max_reps=10):
    """Median wall time (ms) of fn on the CPU: 1 warmup, then reps until the budget is spent."""
    fn()
    samples = []
    t_start = time.perf_counter()
    while len(samples) < max_reps and (len(samples) < min_reps or time.perf_counter() - t_start < budget_s):
        t0 = time.perf_counter()
        fn()
        samples.append((time.perf_counter() - t0) * 1e3)
    return statistics.median(samples), len(samples)


def _traffic(*names):
    """HBM bytes per launch of the named kernels (summed), from profiles/traffic.json; None if any is absent."""
    path = os.path.join(ROOT, "profiles", "traffic.json")
    try:
        with open(path) as f:
            d = json.load(f)
        return int(sum(d[n]["fetch_bytes"] + d[n]["write_bytes"] for n in names))
    except Exception:
        return None


def _cpu_model():
    try:
        with open("/proc/cpuinfo") as f:
            for ln in f:
                if ln.startswith("model name"):
                    return ln.split(":", 1)[1].strip()
    except OSError:
        pass
    return None


def _gpu_clocks():
    """Current shader/memory/fabric clock levels from the amdgpu sysfs tables (best effort; None when absent).

    Read from sysfs rather than by running rocm-smi: under rocprofv3 a child process inherits the profiler's
    preload, initialises the GPU and would then exec its interpreter."""
    import glob
    for dev in sorted(glob.glob("/sys/class/drm/card*/device")):
        out = {}
        for clk in ("sclk", "mclk", "fclk"):
            try:
                with open(os.path.join(dev, "pp_dpm_" + clk)) as f:
                    cur = [ln.strip() for ln in f if ln.strip().endswith("*")]
            except OSError:
                continue
            if cur:
                out[clk] = cur[0].rstrip("* ").split(":", 1)[-1].strip()
        if out:
            return out
    return None


def _cpu_threads():
    try:
        return len(os.sched_getaffinity(0))
    except AttributeError:  # pragma: no cover
        return os.cpu_count() or 1


# --------------------------------------------------------------------------- per-config runners
def run_indexer(cfg, steps, warmup, do_cpu, cpu_budget):
    import torch
    from kernelswift_amd import ops, workloads
    w = workloads.CONFIGS[cfg]("cuda")
    t, p = w.tensors, w.params
    B, S, H, D = t["q"].shape
    T = t["k"].shape[1]
    ws = torch.empty(ops.indexer_workspace_size(B, S, H, D, T), dtype=torch.uint8, device="cuda")

    from kernelswift_amd import _lib
    tops = _lib.torch_ops()

    def step():  # the torch operator (TORCH_LIBRARY ks_mi355x), as a caller of the op sees it
        return tops.indexer(t["q"], t["k"], t["w"], t["freqs"], p["k_top"], p["causal"], p["start_pos"], p["ratio"],
                            p["offset"], p["rope_start"], p["rope_dim"], p["rope_k"], False, None)

    def step_ctypes():
        return ops.indexer(t["q"], t["k"], t["w"], t["freqs"], p["k_top"], p["causal"], p["start_pos"], p["ratio"],
                           p["offset"], p["rope_start"], p["rope_dim"], p["rope_k"], workspace=ws)

    dev_med, dev_mean = _events_median(step, steps, warmup)
    wall_med, ms_step = _wall(step, steps, warmup)
    host = {"torch_op": round(_host_issue_us(step), 2), "ctypes": round(_host_issue_us(step_ctypes), 2)}

    # the fused call's kernels alone, on pre-rotated inputs: the bounded score kernel (the dominant one), the
    # bounded top-k (threshold, exact recomputation of the candidates, exact selection), and for reference
    # the exact score kernel and the plain top-k of the other shapes
    qr = t["q"].clone()
    kr = t["k"].clone()
    ops.rope_inplace(qr, t["freqs"], rope_start=0, pos0=p["start_pos"])
    ops.rope_inplace(kr, t["freqs"], rope_start=0, pos0=0)
    stats = (ops.indexer_row_stats(qr), ops.indexer_row_stats(kr))
    out = torch.empty(B, S, T, dtype=torch.float32, device="cuda")
    bnd = torch.empty(B, S, T, dtype=torch.float32, device="cuda")
    kmax = torch.empty(B, (T + 255) // 256, dtype=torch.float32, device="cuda")
    idx = torch.empty(B, S, min(p["k_top"], T), dtype=torch.int32, device="cuda")
    lib = _lib.load()
    # the bounded selection's workspace: lists, bucket counts, states (the score kernel leaves the rows' histogram
    # scales in it); kmax is not read
    part = torch.zeros(lib.ks_dbg_topk_bounded_slots(B * S, T), dtype=torch.int64, device="cuda")
    (qn, qs), (kn, ks_) = stats
    stream = torch.cuda.current_stream().cuda_stream

    def scores_bounded():
        _lib.check(lib.ks_dbg_indexer_scores_bounded(qr.data_ptr(), kr.data_ptr(), t["w"].data_ptr(), qn.data_ptr(),
                                                     qs.data_ptr(), kn.data_ptr(), ks_.data_ptr(), out.data_ptr(),
                                                     bnd.data_ptr(), kmax.data_ptr(), part.data_ptr(), B, S, T, 1,
                                                     p["start_pos"], stream), "scores (bounded)")

    def topk_bounded():
        _lib.check(lib.ks_dbg_indexer_topk_bounded(out.data_ptr(), bnd.data_ptr(), kmax.data_ptr(), qr.data_ptr(),
                                                   kr.data_ptr(), t["w"].data_ptr(), qn.data_ptr(), qs.data_ptr(),
                                                   kn.data_ptr(), ks_.data_ptr(), B, S, T, p["k_top"], 1,
                                                   p["start_pos"], idx.data_ptr(), stream, part.data_ptr(),
                                                   part.numel()), "top-k (bounded)")

    def scores_exact():
        _lib.check(lib.ks_indexer_scores(qr.data_ptr(), kr.data_ptr(), t["w"].data_ptr(), 0, qn.data_ptr(),
                                         qs.data_ptr(), kn.data_ptr(), ks_.data_ptr(), out.data_ptr(), B, S, H, D, T,
                                         T, 1, p["start_pos"], 1, stream), "scores")

    score_us = _events_avg(scores_bounded, steps, warmup)
    # the bounded top-k may overwrite scores, bounds and its workspace, so every timed call starts from a fresh
    # copy of one score kernel call's output; the copies are timed alone and subtracted
    part.zero_()
    scores_bounded()
    out0, bnd0, part0 = out.clone(), bnd.clone(), part.clone()

    def restore():
        out.copy_(out0)
        bnd.copy_(bnd0)
        part.copy_(part0)

    def restore_topk():
        restore()
        topk_bounded()

    topkb_us = _events_avg(restore_topk, steps, warmup) - _events_avg(restore, steps, warmup)
    exact_us = _events_avg(scores_exact, steps, warmup)
    sc = out.clone()

    def topk():
        ops.topk_mask(sc, True, 1, T, 0, k=p["k_top"], start_pos=p["start_pos"], out_dtype=torch.int32)

    topk_us = _events_avg(topk, steps, warmup)
    flops = 2.0 * S * H * T * D
    achieved = flops / (score_us * 1e-6) / 1e12
    res = {
        "us_per_call": round(dev_med, 3), "us_per_call_mean": round(dev_mean, 3),
        "wall_us_per_call_sync": round(wall_med, 3), "ms_per_step": ms_step,
        "kernels_us": {"indexer_scores_kernel (bounded)": round(score_us, 3),
                       "bounded top-k": round(topkb_us, 3),
                       "indexer_scores_kernel (exact, other shapes)": round(exact_us, 3),
                       "topk_rows_kernel (plain, other shapes)": round(topk_us, 3)},
        "roofline": {"bound": "mfma", "kernel": "indexer_scores_kernel (bounded)", "achieved": round(achieved, 2),
                     "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s", "frac": round(achieved / PEAK_BF16_TFLOPS, 4),
                     "traffic": _traffic(f"indexer_scores_kernel<4, 128, false, true, false, false>@{cfg}")},
        # the product's bounded top-k reads a score and a bound (8 B) per column; the plain one 4 B
        "topk_bounded_GBps": round(S * T * 8 / (topkb_us * 1e-6) / 1e9, 1),
        "topk_plain_GBps": round(S * T * 4 / (topk_us * 1e-6) / 1e9, 1),
        "host_issue_us_per_call": host,
    }
    if do_cpu:
        from oracle import torch_ref
        tc = {n: v.cpu() for n, v in t.items()}
        cis = torch.view_as_complex(tc["freqs"])
        torch.set_num_threads(_cpu_threads())
        ms, reps = _cpu_time(lambda: torch_ref.indexer(tc["q"], tc["k"], tc["w"], cis, p["k_top"], True,
                                                       p["start_pos"], 1, 0, 0, 64, True), cpu_budget)
        res["cpu_baseline"] = {"value": round(ms * 1e3, 1), "unit": "us/call", "cores": torch.get_num_threads(),
                               "kind": "port",
                               "sample": f"full config-{cfg} call (torch-CPU op sequence of baseline/indexer.py), "
                                         f"median of {reps}"}
    return res


def run_sinkhorn(steps, warmup, do_cpu, cpu_budget):
    import torch
    from kernelswift_amd import ops, workloads
    w = workloads.CONFIGS[1]("cuda")
    x = w.tensors["x"]
    out = torch.empty_like(x)
    from kernelswift_amd import _lib
    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream

    def k():
        _lib.check(lib.ks_sinkhorn(x.data_ptr(), out.data_ptr(), x.shape[0], 10, 1e-6, stream), "sinkhorn")

    tops = _lib.torch_ops()

    def step():  # the torch operator (TORCH_LIBRARY ks_mi355x), as a caller of the op sees it
        return tops.sinkhorn(x, 10, 1e-6)

    dev_med, dev_mean = _events_median(step, steps, warmup)
    wall_med, ms_step = _wall(step, steps, warmup)
    ct_med, _ = _events_median(lambda: ops.sinkhorn(x, 10, 1e-6), steps, warmup)
    host = {"torch_op": round(_host_issue_us(step), 2), "ctypes": round(_host_issue_us(lambda: ops.sinkhorn(x, 10, 1e-6)), 2)}
    kus = _events_avg(k, steps, warmup)
    # the reference's other configured iteration count (hc_sinkhorn_iters = 20)
    kus20 = _events_avg(lambda: _lib.check(lib.ks_sinkhorn(x.data_ptr(), out.data_ptr(), x.shape[0], 20, 1e-6, stream),
                                           "sinkhorn"), steps, warmup)
    nbytes = 2 * x.numel() * 4
    achieved = nbytes / (kus * 1e-6) / 1e9
    # size sweep (asymptotic bandwidth; the 2 MiB config is launch/latency bound)
    sweep = {}
    for n in (1 << 20, 1 << 24):
        xx = torch.randn(n, 4, 4, device="cuda")
        oo = torch.empty_like(xx)
        # 20 warmup launches: the first few dozen on freshly allocated GiB buffers run ~15% slower
        us = _events_avg(lambda: _lib.check(lib.ks_sinkhorn(xx.data_ptr(), oo.data_ptr(), n, 10, 1e-6, stream),
                                            "sinkhorn"), 30, 20)
        gbs = 2 * n * 64 / (us * 1e-6) / 1e9
        sweep[str(n)] = {"us": round(us, 2), "GBps": round(gbs, 1), "frac": round(gbs / PEAK_HBM_GBS, 4)}
        del xx, oo
    res = {"us_per_call": round(dev_med, 3), "wall_us_per_call_sync": round(wall_med, 3), "ms_per_step": ms_step,
           "kernels_us": {"sinkhorn4x4_kernel": round(kus, 3)},
           "roofline": {"bound": "hbm", "kernel": "sinkhorn4x4_kernel", "achieved": round(achieved, 1),
                        "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": round(achieved / PEAK_HBM_GBS, 4),
                        "traffic": _traffic("sinkhorn4x4_kernel@1"), "cache": "warm (2 MiB fits in L2)"},
           "size_sweep_matrices": sweep, "repeat20_kernel_us": round(kus20, 3),
           "ctypes_us_per_call": round(ct_med, 3), "host_issue_us_per_call": host}
    if do_cpu:
        from oracle import torch_ref
        xc = x.cpu()
        torch.set_num_threads(_cpu_threads())
        ms, reps = _cpu_time(lambda: torch_ref.sinkhorn(xc, 10, 1e-6), cpu_budget)
        res["cpu_baseline"] = {"value": round(ms * 1e3, 1), "unit": "us/call", "cores": torch.get_num_threads(),
                               "kind": "port", "sample": f"full config-1 call, median of {reps}"}
    return res


def run_sparse(cfg, steps, warmup, do_cpu, cpu_budget):
    import torch
    from kernelswift_amd import ops, workloads
    w = workloads.CONFIGS[cfg]("cuda")
    t, p = w.tensors, w.params
    B, M, H, Dqk = t["q"].shape
    K = t["idx"].shape[-1]
    dv = p["dv"]
    ws_n = ops.sparse_attn_workspace_size(B, M, H, Dqk, dv, K)
    ws = torch.empty(max(ws_n, 1), dtype=torch.uint8, device="cuda")

    from kernelswift_amd import _lib
    tops = _lib.torch_ops()

    def step():  # the torch operator (TORCH_LIBRARY ks_mi355x), as a caller of the op sees it
        return tops.sparse_attn(t["q"], t["kv"], t["sink"], t["idx"], p["scale"], dv)

    def kernels():  # the kernels alone (preallocated workspace)
        return ops.sparse_attn(t["q"], t["kv"], t["sink"], t["idx"], p["scale"], dv=dv, workspace=ws)

    dev_med, dev_mean = _events_median(step, steps, warmup)
    wall_med, ms_step = _wall(step, steps, warmup)
    op_us = _events_avg(kernels, steps, warmup)
    flops = 2.0 * B * M * H * K * (Dqk + dv)
    gathered = B * M * K * Dqk * 2
    achieved = flops / (op_us * 1e-6) / 1e12
    res = {"us_per_call": round(dev_med, 3), "wall_us_per_call_sync": round(wall_med, 3), "ms_per_step": ms_step,
           "kernels_us": {"sparse_attn_kernel+combine": round(op_us, 3)},
           "roofline": {"bound": "mfma", "kernel": ("sparse_attn_kernel" if cfg == 3 else "sparse_attn_mla_kernel")
                        + " (+ combine)", "achieved": round(achieved, 2),
                        "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s", "frac": round(achieved / PEAK_BF16_TFLOPS, 4),
                        "traffic": (_traffic("sparse_attn_kernel<128, 128, 1>@3", "sparse_attn_combine_kernel<128, 2>@3")
                                    if cfg == 3 else
                                    _traffic("sparse_attn_mla_kernel<4, 3>@5", "sparse_attn_mla_combine_kernel@5")),
                        "cache": ("warm (the 2 MiB kv fits in L2)" if cfg == 3
                                  else "kv 2.25 GiB: gathered rows come from HBM")},
           "gathered_GBps": round(gathered / (op_us * 1e-6) / 1e9, 1)}
    if cfg == 3:
        # the reference's dense count-mask formulation (optimized/sparse_attention/design.md:46-69) on the MFMA at
        # this shape: every query scores every key, the top-k list as per-key counts (a diagnostic kernel; the op
        # dispatches to the gather kernel, which is faster here)
        lib = _lib.load()
        out_c = torch.empty(B, M, H, dv, dtype=torch.bfloat16, device="cuda")
        N = t["kv"].shape[1]
        strm = torch.cuda.current_stream().cuda_stream

        def dense():
            _lib.check(lib.ks_dbg_sparse_attn_count(t["q"].data_ptr(), t["kv"].data_ptr(), t["sink"].data_ptr(),
                                                    t["idx"].data_ptr(), out_c.data_ptr(), B, M, H, N, K, p["scale"],
                                                    ws.data_ptr(), ws_n, strm), "ks_dbg_sparse_attn_count")
        dense_us = _events_avg(dense, steps, warmup)
        res["dense_count_mask_us"] = round(dense_us, 3)
        res["dense_count_mask_frac_of_sparse_flops"] = round(flops / (dense_us * 1e-6) / 1e12 / PEAK_BF16_TFLOPS, 4)
    if do_cpu:
        from oracle import torch_ref
        torch.set_num_threads(_cpu_threads())
        if cfg == 3:
            tc = {n: v.cpu() for n, v in t.items()}
            ms, reps = _cpu_time(lambda: torch_ref.sparse_attn(tc["q"], tc["kv"], tc["sink"], tc["idx"], p["scale"]),
                                 cpu_budget)
            sample, scale_up = f"full config-3 call, median of {reps}", 1.0
        else:
            # bounded sample: 4 of the 32 sequences (gathered rows only); time scaled by 32/4
            nb = 4
            rows = torch.stack([t["kv"][b, t["idx"][b, 0].long()] for b in range(nb)]).cpu()
            loc = torch.arange(K, dtype=torch.int32).expand(nb, 1, K).contiguous()
            qc, sc = t["q"][:nb].cpu(), t["sink"].cpu()
            ms, reps = _cpu_time(lambda: torch_ref.sparse_attn(qc, rows, sc, loc, p["scale"], dv=dv), cpu_budget)
            scale_up = B / nb
            sample = f"{nb} of {B} sequences (per-call time scaled x{scale_up:g}), median of {reps}"
        res["cpu_baseline"] = {"value": round(ms * scale_up * 1e3, 1), "unit": "us/call",
                               "cores": torch.get_num_threads(), "kind": "port", "sample": sample}
    return res


def run_mhc(steps, warmup, do_cpu, cpu_budget, N=4096, C=4096, iters=20):
    """mHC residual connection at hc_mult = 4, hc_sinkhorn_iters = 20 (baseline/indexer.py:48-50) over N tokens of
    dim C: the residual update with the Sinkhorn fused in (ks_mhc_post) and the layer-input mix (ks_mhc_pre);
    HBM-bound streams, judged on GB/s of their algorithmic bytes."""
    import torch
    from kernelswift_amd import ops
    g = torch.Generator(device="cuda").manual_seed(42)
    x = torch.randn(N, 4, C, generator=g, device="cuda").bfloat16()
    f = torch.randn(N, C, generator=g, device="cuda").bfloat16()
    res = torch.randn(N, 4, 4, generator=g, device="cuda")
    post = torch.randn(N, 4, generator=g, device="cuda")
    pre = torch.randn(N, 4, generator=g, device="cuda")
    out = torch.empty_like(x)
    post_us = _events_avg(lambda: ops.mhc_post(x, f, res, post, iters, 1e-6, out=out), steps, warmup)
    wall_med, ms_step = _wall(lambda: ops.mhc_post(x, f, res, post, iters, 1e-6, out=out), steps, warmup)
    pre_us = _events_avg(lambda: ops.mhc_pre(x, pre), steps, warmup)
    post_bytes = N * (4 * C * 2 * 2 + C * 2 + 16 * 4 + 4 * 4)  # x read, out written, f read, logits
    pre_bytes = N * (4 * C * 2 + C * 2 + 4 * 4)
    gbs = post_bytes / (post_us * 1e-6) / 1e9
    res_d = {"us_per_call": round(post_us, 3), "wall_us_per_call_sync": round(wall_med, 3), "ms_per_step": ms_step,
             "workload": f"N={N} tokens, C={C}, hc_mult=4, sinkhorn_iters={iters}",
             "kernels_us": {"mhc_post_kernel (Sinkhorn fused)": round(post_us, 3), "mhc_pre_kernel": round(pre_us, 3)},
             "roofline": {"bound": "hbm", "kernel": "mhc_post_kernel", "achieved": round(gbs, 1),
                          "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": round(gbs / PEAK_HBM_GBS, 4),
                          "bytes_per_launch": post_bytes, "traffic": _traffic("mhc_post_kernel@mhc")},
             "pre_GBps": round(pre_bytes / (pre_us * 1e-6) / 1e9, 1)}
    if do_cpu:
        from oracle import torch_ref
        torch.set_num_threads(_cpu_threads())
        nb = 256  # bounded sample of tokens; time scaled to N
        xc, fc, rc, pc = x[:nb].cpu().float(), f[:nb].cpu().float(), res[:nb].cpu(), post[:nb].cpu()

        def cpu_post():
            S = torch_ref.sinkhorn(rc, iters, 1e-6)
            return (torch.einsum("nij,njc->nic", S, xc) + 2 * torch.sigmoid(pc)[:, :, None] * fc[:, None, :]).bfloat16()

        ms, reps = _cpu_time(cpu_post, cpu_budget)
        res_d["cpu_baseline"] = {"value": round(ms * (N / nb) * 1e3, 1), "unit": "us/call", "cores": torch.get_num_threads(),
                                 "kind": "port", "sample": f"{nb} of {N} tokens (scaled x{N // nb}), median of {reps}"}
    return res_d


def _fp8_inputs(cfg):
    """Config `cfg`'s q and k rotated, then quantised to e4m3 with one power-of-two scale per row."""
    from kernelswift_amd import ops, workloads
    w = workloads.CONFIGS[cfg]("cuda")
    t, p = w.tensors, w.params
    D = t["q"].shape[3]
    qr, kr = t["q"].clone(), t["k"].clone()
    ops.rope_inplace(qr, t["freqs"], rope_start=0, pos0=p["start_pos"])
    ops.rope_inplace(kr, t["freqs"], rope_start=0, pos0=0)
    qc, qs = ops.fp8_quant(qr, D, True)
    kc, ks_ = ops.fp8_quant(kr, D, True)
    return t, p, qr, qc, qs[..., 0].contiguous(), kc, ks_[..., 0].contiguous()


def run_fp8(steps, warmup, do_cpu, cpu_budget):
    """The indexer on FP8 rows (dtype = "fp8", scale_fmt = "ue8m0"; baseline/indexer.py:14-17) at config 2's shape
    (and config 4's beside it): q and k rotated, then quantised to e4m3 with one power-of-two scale per row (the
    cache-write side, timed as ks_fp8_quant_rows), and the indexer call on the codes (a statistics pass, then the
    bounded score and recomputation kernels reading the codes themselves, exact top-k).  The quantiser is
    HBM-bound: its roofline is GB/s of bf16 read + codes and scales written."""
    import torch
    from kernelswift_amd import _lib
    tops = _lib.torch_ops()
    t4, p4, _, qc4, qs4, kc4, ks4 = _fp8_inputs(4)
    dev4, _ = _events_median(
        lambda: tops.indexer_fp8(qc4, qs4, kc4, ks4, t4["w"], p4["k_top"], True, p4["start_pos"], 1, 0, False, None),
        steps, warmup)
    del t4, qc4, qs4, kc4, ks4
    t, p, qr, qc, qs, kc, ks_ = _fp8_inputs(2)
    B, S, H, D = qc.shape
    T = kc.shape[1]

    def step():
        return tops.indexer_fp8(qc, qs, kc, ks_, t["w"], p["k_top"], True, p["start_pos"], 1, 0, False, None)

    dev_med, dev_mean = _events_median(step, steps, warmup)
    wall_med, ms_step = _wall(step, steps, warmup)
    # the quantiser timed alone (outputs preallocated, launched through the C ABI): q rows, the larger launch
    lib = _lib.load()
    qc2, qs2 = torch.empty_like(qc), torch.empty(B * S * H, dtype=torch.float32, device="cuda")
    stream = torch.cuda.current_stream().cuda_stream

    def quant_q():
        _lib.check(lib.ks_fp8_quant_rows(qr.data_ptr(), B * S * H, D, D, 1, qc2.data_ptr(), qs2.data_ptr(), stream),
                   "fp8 quant")

    quant_us = _events_avg(quant_q, steps, warmup)
    rows = B * S * H
    qbytes = rows * D * 3 + rows * 4  # bf16 read, codes and scales written
    gbs = qbytes / (quant_us * 1e-6) / 1e9
    res = {"us_per_call": round(dev_med, 3), "us_per_call_mean": round(dev_mean, 3),
           "wall_us_per_call_sync": round(wall_med, 3), "ms_per_step": ms_step,
           "us_per_call_config4_shape": round(dev4, 3),
           "workload": f"config-2 shape on e4m3 rows (ue8m0 row scales): B={B} S_q={S} S_kv={T} H={H} D={D} "
                       f"causal top-{p['k_top']}; us_per_call_config4_shape: the same at config 4's shape",
           "kernels_us": {"fp8_quant_kernel (q rows)": round(quant_us, 3)},
           "roofline": {"bound": "hbm", "kernel": "fp8_quant_kernel", "achieved": round(gbs, 1),
                        "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": round(gbs / PEAK_HBM_GBS, 4),
                        "bytes_per_launch": qbytes,
                        "traffic": _traffic("fp8_quant_kernel<16>@fp8 (quantiser, q rows)")}}
    if do_cpu:
        from oracle import torch_ref
        torch.set_num_threads(_cpu_threads())
        qcc, kcc = qc.cpu(), kc.cpu()
        qsc, ksc, wc = qs.cpu(), ks_.cpu(), t["w"].cpu()

        def cpu_call():
            qd = (qcc.float() * qsc[..., None]).bfloat16()
            kd = (kcc.float() * ksc[..., None]).bfloat16()
            return torch_ref.indexer(qd, kd, wc, None, p["k_top"], True, p["start_pos"], 1, 0, 0, 0, False)

        ms, reps = _cpu_time(cpu_call, cpu_budget)
        res["cpu_baseline"] = {"value": round(ms * 1e3, 1), "unit": "us/call", "cores": torch.get_num_threads(),
                               "kind": "port", "sample": f"full call (dequantisation + torch-CPU op sequence of "
                                                         f"baseline/indexer.py without RoPE), median of {reps}"}
    return res


def run_dropin(steps, warmup):
    """ModelNew at the reference's own example shapes (baseline/*.py get_inputs), timed like the reference
    harness (perf_counter + synchronize per call, median): context beside BASELINE.md's published numbers,
    which were measured on other hardware."""
    import torch
    from kernelswift_amd.optimized import indexer as ix, sinkhorn as sk, sparse_attention as sa
    out = {}
    for name, mod in (("sinkhorn [1,1024,4,4]", sk),
                      ("indexer B=8 S=2600 H=16 D=64 ratio=4 k=128", ix),
                      ("sparse_attention B=8 M=2600 H=64 N=32 D=128 K=16", sa)):
        torch.manual_seed(42)
        m = mod.ModelNew(*mod.get_init_inputs()).cuda().eval()
        torch.manual_seed(42)
        inp = [v.cuda() if isinstance(v, torch.Tensor) else v for v in mod.get_inputs()]
        with torch.no_grad():
            wall, _ = _wall(lambda: m(*inp), steps, warmup)
        out[name] = {"wall_us_per_call_sync": round(wall, 2)}
        del m, inp
        torch.cuda.empty_cache()
    return out


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py: this build measures one GPU only (asked for --gpus {args.gpus}); every MI355X box "
              "here has one GPU, and the multi-GPU sharding is a design note, not a measured path.", file=sys.stderr)
        sys.exit(2)
    import torch
    assert torch.cuda.is_available(), "bench.py needs the GPU"
    torch.cuda.set_device(0)
    cfgs = [c if c in ("mhc", "fp8") else int(c) for c in args.configs.split(",") if c]
    per = {}
    for c in cfgs:
        if c in (2, 4):
            per[c] = run_indexer(c, args.steps, args.warmup, not args.no_cpu, args.cpu_seconds)
        elif c == 1:
            per[c] = run_sinkhorn(args.steps, args.warmup, not args.no_cpu, args.cpu_seconds)
        elif c in (3, 5):
            per[c] = run_sparse(c, args.steps, args.warmup, not args.no_cpu, args.cpu_seconds)
        elif c == "mhc":
            per[c] = run_mhc(args.steps, args.warmup, not args.no_cpu, args.cpu_seconds)
        elif c == "fp8":
            per[c] = run_fp8(args.steps, args.warmup, not args.no_cpu, args.cpu_seconds)
        print(f"[bench] config {c}: {json.dumps(per[c])}", file=sys.stderr, flush=True)
    dropin = None
    if not args.no_dropin:
        dropin = run_dropin(min(args.steps, 100), min(args.warmup, 20))
        print(f"[bench] drop-in ModelNew at the reference example shapes: {json.dumps(dropin)}", file=sys.stderr,
              flush=True)
    if args.calib_copy:
        from kernelswift_amd import ops
        src = torch.empty(512 << 20, dtype=torch.uint8, device="cuda").fill_(1)
        dst = torch.empty_like(src)
        for _ in range(5):
            ops.copy_bytes(src, dst)
        torch.cuda.synchronize()
        print("[bench] calibration copy: 5 x 512 MiB (copy16_kernel)", file=sys.stderr, flush=True)
    head = per.get(2) or per[cfgs[0]]
    head_cfg = 2 if 2 in per else cfgs[0]
    line = {
        "metric": "median us/call per op at 1 GPU + % of HBM/MFMA roofline vs host-CPU ref",
        "value": head["us_per_call"],
        "unit": "us/call",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(head["ms_per_step"], 5),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded N(0,1), BASELINE.json shapes)",
        "config": {"workload": ("indexer_short: B=1 S_q=128 S_kv=4096 H=64 D=128 rope64 causal top-512 "
                                "(fused rope+scores+topk)") if head_cfg == 2 else f"config {head_cfg}",
                   "config_index": head_cfg},
        "roofline": head["roofline"],
        "cpu_baseline": head.get("cpu_baseline"),
        "wall_us_per_call_sync": head["wall_us_per_call_sync"],
        "per_config": {str(k): v for k, v in per.items()},
        "dropin_example_shapes": dropin,
        "device": torch.cuda.get_device_name(0),
        "gpu_clocks": _gpu_clocks(),
        "host": {"cpu_model": _cpu_model(), "threads": _cpu_threads()},
    }
    print(json.dumps(line), flush=True)


if __name__ == "__main__":
    main()
