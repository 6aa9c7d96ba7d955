#!/usr/bin/env python3
"""Benchmark of the fused extreme-classifier training step on one MI355X.

One "step" = one call of the FP8 layer's xfc_forward_backward over all label chunks (the hot path of
src/xmc_classifiers/chunked_fp8xmc_clf.py:81-123): X[128,768] bf16 resident in HBM, W[670091(+pad),768] e4m3
resident in HBM, positives as COO int32.  Prints ONE JSON line.

  python bench.py [--gpus 1] [--steps K] [--warmup W] [--config cfg2_fp8_670k] [--round sr_fast|sr_philox|rtn]

--mode forward / forward_topk time the FP8 layer's inference instead (xfc_forward, chunked_fp8xmc_clf.py:45-60, and
the top-100 that evaluate.py:158-159 takes of it); the default mode and the headline metric is the training step.
"""
import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0
FP8_PEAK_TFLOPS = 5000.0


def padded_labels(num_labels, num_chunks):
    # src/xmc_classifiers/chunked_fp8xmc_clf.py:26
    return num_labels + 16 * num_chunks - num_labels % (16 * num_chunks)


def cpu_baseline(cfg, budget_s=12.0):
    """The reference's PyTorch CPU bf16 chunked path (oracle.torch_port) on ONE chunk of this workload,
    scaled by the number of chunks."""
    import numpy as np
    import torch
    from elmo_amd import synth
    from oracle import torch_port
    nc = cfg.num_chunks
    rows = padded_labels(cfg.num_labels, nc) // nc
    threads = min(16, os.cpu_count() or 1)
    torch.set_num_threads(threads)
    g = torch.Generator().manual_seed(cfg.seed)
    w = (torch.randn(rows, cfg.dim, generator=g) * cfg.init_std).to(torch.bfloat16)
    x = torch.from_numpy(synth.make_x(cfg.batch, cfg.dim, cfg.seed)).to(torch.bfloat16)
    lab = synth.make_labels(cfg.batch, cfg.num_labels, cfg.pos_mean, cfg.zipf_s, cfg.seed)
    lab = torch.from_numpy(lab[lab[:, 1] < rows])
    torch_port.bf16_chunked_step(w, x, lab, cfg.lr, 1)          # warm-up
    times = []
    t_start = time.perf_counter()
    while time.perf_counter() - t_start < budget_s or len(times) < 5:
        t0 = time.perf_counter()
        torch_port.bf16_chunked_step(w, x, lab, cfg.lr, 1)
        times.append(time.perf_counter() - t0)
    t_chunk = float(np.median(times))
    return {
        "value": 1.0 / (t_chunk * nc), "unit": "steps/s", "cores": threads, "kind": "port", "extrapolated": True,
        "sample": f"EXTRAPOLATED: 1 of {nc} chunks timed ({rows} labels x {cfg.dim}, batch {cfg.batch}), bf16 weights, "
                  f"round-to-nearest update, median of {len(times)} runs; value = 1 / ({nc} x seconds_per_chunk)",
        "seconds_per_chunk": t_chunk,
    }


def device_settle(dev, want_ms, nc, rows, num_labels, batch, pos_mean, zipf_s):
    """Device conditioning before the warm-up steps: about want_ms milliseconds of the fused step on a SEPARATE classifier
    of the benchmark's shape (its own weights, inputs and workspace - none of the benchmark's buffers; freed before the
    peak-memory counter is reset).  When the step kernel starts on a device that was doing something else, the first
    ~25 ms pass through a clock/power transient: over the first 40 launches of a process the same launch takes 0.47,
    then up to 0.59, then 0.45 ms, and only work with the same memory traffic gets the device past it (the same kernel
    on a classifier that stays in the caches leaves a smaller hump).  A training run is in the settled state; a 20-step
    measurement right after start-up is not.  Returns what was done, for the benchmark's output."""
    import numpy as np
    import torch
    from elmo_amd import ops, synth
    if want_ms <= 0:
        return {"ms": 0.0, "launches": 0}
    gen = torch.Generator(device=dev).manual_seed(99)
    chunks = [(torch.randn(rows, 768, generator=gen, device=dev) * 0.02).to(torch.float8_e4m3fn) for _ in range(nc)]
    x = torch.from_numpy(synth.make_x(batch, 768, 99)).to(dev).to(torch.bfloat16)
    labels = torch.from_numpy(synth.make_labels(batch, num_labels, pos_mean, zipf_s, 99)).to(dev)
    ws = ops.alloc_workspace(nc, rows, dev, batch)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    n = 0
    while (time.perf_counter() - t0) * 1e3 < want_ms:
        for _ in range(16):
            ops.fp8_step(chunks, x, labels, 0.05, seeds=np.arange(nc) + n, round_mode="sr_fast", workspace=ws)
            n += 1
        torch.cuda.synchronize()
    spent = (time.perf_counter() - t0) * 1e3
    del chunks, x, labels, ws
    torch.cuda.empty_cache()
    return {"ms": spent, "launches": n,
            "what": f"fused step on a separate classifier of the same shape ({nc} x {rows} labels, batch {batch}; not the benchmark's buffers)"}


def bench_tiled(args, cfg):
    """The secondary modes (bf16 layer, simulated FP8, true FP8 with a batch above 128) on the tiled step: one kernel over
    all chunks with 768 features, three per chunk with 1,024; timed as a whole step with HIP events on the torch stream."""
    import numpy as np
    import torch
    from elmo_amd import ops, synth
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    bf16 = cfg.weights == "bf16"
    nc = cfg.num_chunks
    gen = torch.Generator(device=dev).manual_seed(cfg.seed)
    if bf16:
        L = cfg.num_labels
        cs = -(-L // nc)
        w = (torch.randn(L, cfg.dim, generator=gen, device=dev, dtype=torch.float32) * cfg.init_std).to(torch.bfloat16)
        views = [w[c * cs:min((c + 1) * cs, L)] for c in range(nc) if c * cs < L]
        rows, wtype, wbytes = cs, "bf16", 2
    else:
        L_pad = padded_labels(cfg.num_labels, nc)
        rows = L_pad // nc
        views = [(torch.randn(rows, cfg.dim, generator=gen, device=dev, dtype=torch.float32) * cfg.init_std).to(torch.float8_e4m3fn)
                 for _ in range(nc)]
        wtype, wbytes = "e4m3", 1
    x = torch.from_numpy(synth.make_x(cfg.batch, cfg.dim, cfg.seed)).to(dev).to(torch.bfloat16)
    labels = torch.from_numpy(synth.make_labels(cfg.batch, cfg.num_labels, cfg.pos_mean, cfg.zipf_s, cfg.seed)).to(dev)
    weight_bytes = sum(v.numel() for v in views) * wbytes
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    base_alloc = torch.cuda.memory_allocated()
    ws = ops.alloc_tiled_workspace(len(views), rows, dev, cfg.batch, cfg.dim)
    grad = torch.empty(cfg.batch, cfg.dim, dtype=torch.bfloat16, device=dev)
    true_fp8 = not bf16 and "simfp8" not in cfg.name
    rng = np.random.default_rng(cfg.seed)
    # bf16 weights and simulated FP8 round with the reference's Philox recipe unless another mode is asked for by name
    # (simulated FP8 has no fast mode: its cast goes through bf16 and torch)
    mode = args.round if true_fp8 or args.round == "rtn" or (bf16 and args.round_given) else "sr_philox"

    def one_step():
        ops.tiled_step(views, rows, wtype, x, labels, cfg.lr, seeds=rng.integers(0, 1_000_000, size=len(views)),
                       round_mode=mode, workspace=ws, grad_out=grad, quantize_x=true_fp8, saturate=true_fp8)

    for _ in range(args.warmup):
        one_step()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    e0.record()
    for _ in range(args.steps):
        one_step()
    e1.record()
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    dev_ms = e0.elapsed_time(e1) / args.steps
    assert bool(torch.isfinite(grad.float()).all())
    (failed,) = ops.sticky_error_words(tiled_workspace=ws)
    assert int(failed.item()) == 0, "a step gave up waiting: its time means nothing"
    peak_bytes = torch.cuda.max_memory_allocated() - base_alloc + weight_bytes
    algo_bytes = 2.0 * cfg.num_labels * cfg.dim * wbytes
    algo_flops = 6.0 * cfg.batch * cfg.num_labels * cfg.dim
    # roofline of the step as the benchmark defines it: max(6 B L d / FP8 peak, 2 L d bytes / HBM bandwidth)
    t_mfma, t_hbm = algo_flops / (FP8_PEAK_TFLOPS * 1e12), algo_bytes / (HBM_PEAK_GBS * 1e9)
    t_roof = max(t_mfma, t_hbm)
    if t_mfma > t_hbm:
        roof = {"bound": "mfma", "achieved": algo_flops / (dev_ms * 1e-3) / 1e12, "peak": FP8_PEAK_TFLOPS, "unit": "TFLOP/s"}
    else:
        roof = {"bound": "hbm", "achieved": algo_bytes / (dev_ms * 1e-3) / 1e9, "peak": HBM_PEAK_GBS, "unit": "GB/s"}
    roof["frac"] = roof["achieved"] / roof["peak"]
    out = {
        "metric": "XMC classifier train steps/sec (%s)" % ("bf16 layer" if bf16 else "FP8, tiled step" if true_fp8 else "simulated FP8"),
        "value": args.steps / elapsed, "unit": "steps/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": elapsed / args.steps * 1e3, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16 MFMA, fp32 accumulate" + ("" if bf16 else ", e4m3 weights widened on load" + (" but in the logits (FP8 MFMA)" if true_fp8 else "")), "data": "synthetic",
        "config": {"workload": cfg.name, "labels": cfg.num_labels, "features": cfg.dim, "batch": cfg.batch,
                   "chunks": len(views), "rows_per_chunk": rows, "positives": int(labels.shape[0]), "lr": cfg.lr,
                   "rounding": mode, "seed": cfg.seed},
        "roofline": dict(roof, traffic=None, kernel="whole tiled step, HIP events",
                         kernel_ms=dev_ms, algorithmic_bytes_per_launch=algo_bytes, algorithmic_flops_per_launch=algo_flops),
        "roofline_step_frac": t_roof / (elapsed / args.steps),
        "peak_hbm_gb": peak_bytes / 1e9, "peak_hbm_over_weights": peak_bytes / weight_bytes,
    }
    print(json.dumps(out))


def bench_inference(args, cfg):
    """Inference of the FP8 layer on the workload's weights: dense logits, or the top-100 per row merged chunk by
    chunk.  Timed as whole calls with HIP events on the torch stream."""
    import torch
    from elmo_amd import ops, synth
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    nc = cfg.num_chunks
    rows = padded_labels(cfg.num_labels, nc) // nc
    gen = torch.Generator(device=dev).manual_seed(cfg.seed)
    chunks = [(torch.randn(rows, cfg.dim, generator=gen, device=dev, dtype=torch.float32) * cfg.init_std).to(torch.float8_e4m3fn)
              for _ in range(nc)]
    batch = min(cfg.batch, ops.MAX_BATCH)
    x = torch.from_numpy(synth.make_x(batch, cfg.dim, cfg.seed)).to(dev).to(torch.bfloat16)
    ws = ops.alloc_workspace(nc, rows, dev, batch)
    k = 100
    topk = args.mode == "forward_topk"
    # forward_topk: the two-pass selection (under 1 MB of scratch); --topk-path chunkwise times the general path instead
    chunkwise = topk and args.topk_path == "chunkwise"
    scratch = torch.empty(ops.topk_scratch_bytes(rows), dtype=torch.uint8, device=dev) if chunkwise else None
    fscratch = torch.empty(ops.topk_fused_scratch_bytes(), dtype=torch.uint8, device=dev) if topk and not chunkwise else None
    statuses = []
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    base_alloc = torch.cuda.memory_allocated()

    def one_call():
        if chunkwise:
            return ops.fp8_forward_topk(chunks, x, cfg.num_labels, k, workspace=ws, scratch=scratch, fused=False)
        if topk:
            # status words are looked at after the timed region, as a caller that pipelines its batches would
            v, i, st = ops.fp8_forward_topk(chunks, x, cfg.num_labels, k, workspace=ws, fused_scratch=fscratch, defer_check=True)
            statuses.append(st)
            return v, i
        return ops.fp8_forward(chunks, x, cfg.num_labels, workspace=ws)

    for _ in range(args.warmup):
        one_call()
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    t0 = time.perf_counter()
    e0.record()
    for _ in range(args.steps):
        res = one_call()
    e1.record()
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    dev_ms = e0.elapsed_time(e1) / args.steps
    extra = torch.cuda.max_memory_allocated() - base_alloc
    del res
    if statuses and int(torch.stack(statuses).abs().sum()) != 0:
        raise SystemExit("bench.py: the two-pass top-k reported an overflowing candidate list; its timing is not valid")
    weight_bytes = float(cfg.num_labels) * cfg.dim
    algo_bytes = weight_bytes + (batch * k * 6.0 if topk else 2.0 * batch * cfg.num_labels)
    achieved = algo_bytes / (dev_ms * 1e-3) / 1e9
    traffic = None
    tpath = os.path.join(ROOT, "profiles", "hbm_traffic.json")
    if os.path.exists(tpath) and not chunkwise:   # from the profile summaries, not measured in this run
        with open(tpath) as f:
            traffic = json.load(f).get(f"fp8_forward_select_kernel:{cfg.name}:forward_topk" if topk else
                                       f"fp8_forward_kernel:{cfg.name}:forward")
    print(json.dumps({
        "metric": "XMC classifier inference calls/sec, " + ("top-100 per row without the dense logits" if topk else "dense logits"),
        "value": args.steps / elapsed, "unit": "calls/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": elapsed / args.steps * 1e3, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "fp8_e4m3 MFMA, fp32 accumulate, bf16 logits", "data": "synthetic",
        "config": {"workload": cfg.name, "mode": args.mode, "labels": cfg.num_labels, "features": cfg.dim, "batch": batch,
                   "chunks": nc, "rows_per_chunk": rows, "k": k if topk else None},
        "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": traffic,
                     "kernel": ("fp8_forward_kernel + topk_chunk_kernel per segment" if chunkwise else
                                "fp8_forward_select_kernel<0> (sampled tiles) + <1> (all tiles) + bound and pick kernels" if topk
                                else "fp8_forward_kernel"),
                     "kernel_ms": dev_ms, "algorithmic_bytes_per_launch": algo_bytes},
        "memory_beyond_weights_mb": extra / 1e6,
    }))


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--config", default="cfg2_fp8_670k")
    ap.add_argument("--round", default=None, choices=["sr_fast", "sr_philox", "rtn"],
                    help="default: what the workload names - round to nearest for cfg1_bf16_131k, stochastic for the others "
                         "(sr_fast where FP8 arithmetic is used, the reference's Philox recipe for bf16 weights and simulated FP8)")
    ap.add_argument("--mode", default="step", choices=["step", "forward", "forward_topk"])
    ap.add_argument("--topk-path", default="two_pass", choices=["two_pass", "chunkwise"])
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--settle-ms", type=float, default=100.0,
                    help="milliseconds of device conditioning before the warm-up steps (the fused step on a separate classifier of the same shape); 0 = none")
    ap.add_argument("--head-kahan", default="none", choices=["none", "bf16", "e5m2"],
                    help="time the head-Kahan layer's fused step instead (fused workloads only): compensation buffer of "
                         "this type on the first min(head_ratio x padded labels, rows per chunk) rows of chunk 0")
    ap.add_argument("--head-ratio", type=float, default=0.2, help="training.FP8.head_ratio of the reference's configs")
    ap.add_argument("--scale-w", type=float, default=1.0,
                    help="per-tensor scale of the weights (weight = scale_w * code); the reference uses 1")
    ap.add_argument("--scale-x", type=float, default=1.0, help="per-tensor scale of the quantised embedding")
    ap.add_argument("--copy-calibration", type=int, default=0, metavar="MIB",
                    help="only launch the library's plain copy kernel over MIB MiB five times (counter calibration) and exit")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py: this build runs the classifier step on ONE GPU; --gpus > 1 is not supported "
              "(the path shards by label rows)", file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch
    from elmo_amd import build as _build
    _build.ensure_built()      # load what is built; compile only if there is nothing
    from elmo_amd import _lib, ops, synth

    cfg = synth.CONFIGS[args.config]
    args.round_given = args.round is not None
    if args.round is None:   # the first workload is defined with round-to-nearest, the others with stochastic rounding
        args.round = "rtn" if args.config.startswith("cfg1_bf16_131k") else "sr_fast"
    if cfg.batch > ops.MAX_BATCH_TILED:
        print(f"bench.py: config {cfg.name} is not runnable by this build (batch > {ops.MAX_BATCH_TILED})", file=sys.stderr)
        sys.exit(2)
    if args.mode != "step":
        if cfg.weights == "bf16":
            print("bench.py: the inference modes time the FP8 layer", file=sys.stderr)
            sys.exit(2)
        return bench_inference(args, cfg)
    if cfg.weights == "bf16" or "simfp8" in cfg.name or cfg.batch > ops.MAX_BATCH:
        return bench_tiled(args, cfg)
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    lib = _lib.load()
    if args.copy_calibration > 0:
        nbytes = args.copy_calibration << 20
        src = torch.full((nbytes,), 3, dtype=torch.uint8, device=dev)
        dst = torch.empty_like(src)
        stream = torch.cuda.current_stream().cuda_stream
        for _ in range(5):
            _lib.check(lib.xmc_copy_probe(dst.data_ptr(), src.data_ptr(), nbytes, stream), "xmc_copy_probe")
        torch.cuda.synchronize()
        assert bool((dst == 3).all())
        print(json.dumps({"copy_probe_kernel": {"bytes_read": nbytes, "bytes_written": nbytes, "launches": 5}}))
        return
    nc = cfg.num_chunks
    L_pad = padded_labels(cfg.num_labels, nc)
    rows = L_pad // nc

    # ---- resident inputs (synthetic, seeded)
    gen = torch.Generator(device=dev).manual_seed(cfg.seed)
    chunks = []
    for _ in range(nc):
        w = torch.randn(rows, cfg.dim, generator=gen, device=dev, dtype=torch.float32) * cfg.init_std
        chunks.append((w / args.scale_w).to(torch.float8_e4m3fn))   # code = e4m3(weight / scale_w)
        del w
    x_np = synth.make_x(cfg.batch, cfg.dim, cfg.seed)
    x = torch.from_numpy(x_np).to(dev).to(torch.bfloat16)
    labels = torch.from_numpy(synth.make_labels(cfg.batch, cfg.num_labels, cfg.pos_mean, cfg.zipf_s, cfg.seed)).to(dev)
    torch.cuda.synchronize()
    weight_bytes = sum(c.numel() for c in chunks)
    torch.cuda.empty_cache()
    torch.cuda.reset_peak_memory_stats()
    base_alloc = torch.cuda.memory_allocated()

    workspace = ops.alloc_workspace(nc, rows, dev, cfg.batch)
    grad = torch.empty(cfg.batch, cfg.dim, dtype=torch.bfloat16, device=dev)
    seed_rng = np.random.default_rng(cfg.seed)

    num_head, kahan = 0, None
    if args.head_kahan != "none":
        # the reference requires head_ratio x labels <= rows per chunk (chunked_head_kahan_fp8xmc_clf.py:48); the workload's
        # chunking is kept here and the head is cut at the first chunk's end
        assert args.scale_w == 1.0 and args.scale_x == 1.0, "the head-Kahan layer has no per-tensor scales"
        num_head = min(int(args.head_ratio * L_pad), rows)
        kahan = torch.zeros(num_head, cfg.dim, dtype=torch.bfloat16 if args.head_kahan == "bf16" else torch.float8_e5m2,
                            device=dev)

    def one_step():
        seeds = seed_rng.integers(0, 1_000_000, size=nc)
        if kahan is not None:
            ops.fp8_kahan_step(chunks, kahan, num_head, x, labels, cfg.lr, seeds=seeds, round_mode=args.round,
                               workspace=workspace, grad_out=grad)
            return
        ops.fp8_step(chunks, x, labels, cfg.lr, seeds=seeds, round_mode=args.round, scale_w=args.scale_w, scale_x=args.scale_x,
                     workspace=workspace, grad_out=grad)

    # HIP events around the fused kernel of every timed step, on the stream the kernel is launched on
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipEventCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
    hip.hipEventElapsedTime.argtypes = [ctypes.POINTER(ctypes.c_float), ctypes.c_void_p, ctypes.c_void_p]
    events = []
    for _ in range(args.steps):
        a, b = ctypes.c_void_p(), ctypes.c_void_p()
        assert hip.hipEventCreate(ctypes.byref(a)) == 0 and hip.hipEventCreate(ctypes.byref(b)) == 0
        events.append((a, b))

    def timed_run():
        """args.warmup untimed steps, then args.steps timed ones bracketed by synchronisations; the events of the fused
        kernel of every timed step are recorded on the launch stream."""
        for _ in range(args.warmup):
            one_step()
        torch.cuda.synchronize()
        t_a = time.perf_counter()
        for i in range(args.steps):
            lib.xmc_profile_events(events[i][0], events[i][1])
            one_step()
        torch.cuda.synchronize()
        return time.perf_counter() - t_a

    def kernel_times(evs):
        out_ms = []
        for a, b in evs:
            ms = ctypes.c_float()
            assert hip.hipEventElapsedTime(ctypes.byref(ms), a, b) == 0
            out_ms.append(ms.value)
        return np.asarray(out_ms, dtype=np.float64)

    # cold figure: the same measurement before any device conditioning (what a short run right after start-up sees)
    cold = None
    if args.settle_ms > 0:
        cold_elapsed = timed_run()
        cold = {"ms_per_step": cold_elapsed / args.steps * 1e3, "kernel_ms": float(np.mean(kernel_times(events)))}
    # peak memory of the benchmark's own buffers: the conditioning phase allocates (and frees) a second classifier, which
    # must not count, so the peak is read before it, reset behind it and read again after the timed run
    peak_alloc = torch.cuda.max_memory_allocated()
    settle = device_settle(dev, args.settle_ms, nc, rows, cfg.num_labels, cfg.batch, cfg.pos_mean, cfg.zipf_s)
    torch.cuda.reset_peak_memory_stats()
    elapsed = timed_run()
    (failed,) = ops.sticky_error_words(workspace)      # of every step so far
    assert int(failed.item()) == 0, "a step gave up waiting: its time means nothing"
    assert bool(torch.isfinite(grad.float()).all())
    kms = kernel_times(events)
    kernel_ms = float(np.mean(kms))

    # The other stochastic mode beside the headline's, timed the same way on a shorter run: "sr_fast" is this build's
    # own unbiased rounding (hardware converter + counter hash), "sr_philox" the reference's bit recipe
    # (fuse_kernel.py:29-36: one Philox-4x32-10 word per weight).
    def timed_mode(mode, steps):
        evs = events[:steps]
        for _ in range(3):
            ops.fp8_step(chunks, x, labels, cfg.lr, seeds=seed_rng.integers(0, 1_000_000, size=nc), round_mode=mode,
                         workspace=workspace, grad_out=grad)
        torch.cuda.synchronize()
        t_a = time.perf_counter()
        for i in range(steps):
            lib.xmc_profile_events(evs[i][0], evs[i][1])
            ops.fp8_step(chunks, x, labels, cfg.lr, seeds=seed_rng.integers(0, 1_000_000, size=nc), round_mode=mode,
                         workspace=workspace, grad_out=grad)
        torch.cuda.synchronize()
        dt = (time.perf_counter() - t_a) / steps
        k = float(np.mean(kernel_times(evs)))
        return {"steps_per_s": 1.0 / dt, "ms_per_step": dt * 1e3, "kernel_ms": k,
                "roofline_frac_kernel": 2.0 * cfg.num_labels * cfg.dim / (k * 1e-3) / 1e9 / HBM_PEAK_GBS}

    modes = {args.round: {"steps_per_s": args.steps / elapsed, "ms_per_step": elapsed / args.steps * 1e3, "kernel_ms": kernel_ms,
                          "roofline_frac_kernel": 2.0 * cfg.num_labels * cfg.dim / (kernel_ms * 1e-3) / 1e9 / HBM_PEAK_GBS}}
    other = "sr_philox" if args.round != "sr_philox" else "sr_fast"
    if kahan is None:
        modes[other] = timed_mode(other, min(args.steps, 40))
    ms_per_step = elapsed / args.steps * 1e3
    steps_per_s = args.steps / elapsed
    peak_bytes = max(peak_alloc, torch.cuda.max_memory_allocated()) - base_alloc + weight_bytes

    algo_bytes = 2.0 * cfg.num_labels * cfg.dim * 1          # each weight byte read once, written once
    algo_flops = 6.0 * cfg.batch * cfg.num_labels * cfg.dim
    t_roof = max(algo_flops / (FP8_PEAK_TFLOPS * 1e12), algo_bytes / (HBM_PEAK_GBS * 1e9))
    achieved_gbs = algo_bytes / (kernel_ms * 1e-3) / 1e9
    kernel_name = "fp8_step_role_kernel"
    traffic = None
    tpath = os.path.join(ROOT, "profiles", "hbm_traffic.json")
    if os.path.exists(tpath):
        with open(tpath) as f:
            head = "" if args.head_kahan == "none" else f":{args.head_kahan}_head_{num_head}"
            traffic = json.load(f).get(f"{kernel_name}:{cfg.name}:{args.round}{head}")

    out = {
        "metric": "XMC classifier train steps/sec at 670K labels FP8" if cfg.name == "cfg2_fp8_670k" else
                  "XMC classifier train steps/sec at %d labels FP8" % cfg.num_labels,
        "value": steps_per_s, "unit": "steps/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "warmup_effective": args.warmup + int(settle["launches"]) + (args.warmup + args.steps if cold else 0),
        "ms_per_step": ms_per_step, "cold_ms_per_step": cold["ms_per_step"] if cold else ms_per_step,
        "cold_kernel_ms": cold["kernel_ms"] if cold else kernel_ms, "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "fp8_e4m3 weights+logits MFMA, bf16 gradient MFMA, fp32 accumulate", "data": "synthetic",
        "config": {"workload": cfg.name, "labels": cfg.num_labels, "labels_padded": L_pad, "features": cfg.dim,
                   "batch": cfg.batch, "chunks": nc, "rows_per_chunk": rows, "positives": int(labels.shape[0]),
                   "lr": cfg.lr, "rounding": args.round, "seed": cfg.seed, "scale_w": args.scale_w, "scale_x": args.scale_x,
                   "head_kahan": args.head_kahan, "num_head": num_head},
        "roofline": {"bound": "hbm", "achieved": achieved_gbs, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved_gbs / HBM_PEAK_GBS, "traffic": traffic,
                     "traffic_source": "carried over, not measured in this run: profiles/hbm_traffic.json holds rocprofv3 --pmc "
                                       "FETCH_SIZE + WRITE_SIZE of this kernel from an earlier run of this command, "
                                       "scaled by the copy-kernel calibration",
                     "kernel": kernel_name,
                     "kernel_ms": kernel_ms,
                     "kernel_ms_stats": {"median": float(np.median(kms)), "p10": float(np.percentile(kms, 10)),
                                         "p90": float(np.percentile(kms, 90)), "min": float(kms.min()), "max": float(kms.max()),
                                         "first_8": [round(float(v), 4) for v in kms[:8]],
                                         "last_8": [round(float(v), 4) for v in kms[-8:]]},
                     "algorithmic_bytes_per_launch": algo_bytes, "algorithmic_flops_per_launch": algo_flops},
        "roofline_step_frac": t_roof / (ms_per_step * 1e-3),
        "roofline_steps_per_s": 1.0 / t_roof,
        "peak_hbm_gb": peak_bytes / 1e9, "peak_hbm_over_weights": peak_bytes / weight_bytes,
        "device_settle_before_warmup": settle,
        "rounding_modes": modes,
        "rounding_note": "value is measured with config.rounding; sr_fast is this build's own unbiased stochastic rounding "
                         "(not the reference's random stream), sr_philox the reference's Philox bit recipe",
    }
    if not args.no_cpu_baseline:
        out["cpu_baseline"] = cpu_baseline(cfg)
    print(json.dumps(out))


if __name__ == "__main__":
    main()
