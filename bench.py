#!/usr/bin/env python3
"""Benchmark of the quantized-MoE hot path on one MI355X.

Workload (the one the metric is quoted on): a 16-token DFlash verify block
through one Gemma-4-26B-A4B-shaped MoE layer (hidden 2816, 128 experts of intermediate 704, top-8
softmax router, MLX-affine INT4 g64 experts), synthetic seeded weights and inputs. A layer pass is one
pass of the hot path over the block: router logits + top-8, GPU-side route planning, gate/up +
GELU-tanh gating, down projection, router-weighted combine. A step takes the block through the
`--layers` distinct resident layers once (default 30 = 12.85 GB of experts), as a decode loop does, so
that no pass finds its experts in the 256 MB Infinity Cache and the timed region of even a few steps
is tens of milliseconds long.

Prints ONE JSON line. `value` = INT4 expert bytes the timed steps stream (distinct experts x
3,345,408 B per layer pass) divided by their whole time, inputs resident in HBM. `roofline` prices the dominant kernel
(gate/up) against the 8 TB/s HBM peak from HIP-event timings; `cpu_baseline` times the CPU oracle
(a C restatement of the reference's Swift test-support CPU path) on the same block.
"""
import argparse
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
for p in (ROOT, ROOT / "ane-fieldfare_amd"):
    if str(p) not in sys.path:
        sys.path.insert(0, str(p))

import numpy as np

D, F, E, K = 2816, 704, 128, 8
STRIDE = 3_358_720                       # 205 x 16 KiB per expert blob (reference layout)
EXPERT_BYTES = 3_345_408                 # gate + up + down weights, scales and biases of one expert
GATE_UP_BYTES = 2_230_272                # the share the gate/up kernel streams per expert
DOWN_BYTES = 1_115_136
HBM_PEAK_GBS = 8000.0
MFMA_BF16_PEAK_TFLOPS = 2500.0
TRAFFIC_FILE = ROOT / "profiles" / "hbm_traffic_verify16_prefill3072.txt"


def measured_traffic():
    """HBM bytes per launch measured with rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE on this same seeded workload and
    scaled by a plain 1 GiB copy: the lines `traffic <key> <bytes>` of the committed profile summary. {} when the
    file is not there."""
    out = {}
    try:
        for line in TRAFFIC_FILE.read_text().splitlines():
            parts = line.split()
            if len(parts) == 3 and parts[0] == "traffic":
                out[parts[1]] = float(parts[2])
    except OSError:
        pass
    return out


def host_cpu():
    """(logical CPUs the OS shows, model string) of the host the CPU baseline runs on."""
    model = None
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                model = line.split(":", 1)[1].strip()
                break
    except OSError:
        pass
    return os.cpu_count(), model


def clocks_under_load(burst, torch):
    """Shader / memory clock and power cap from the amdgpu driver's sysfs files (what `rocm-smi --showclocks
    --showmaxpower` prints), read while a queue of verify steps is still running. No child process is started.
    Best effort: None when the files are not there or read differently."""
    import glob

    def current(path):
        for line in open(path):
            if line.strip().endswith("*"):
                return line.split(":", 1)[1].replace("*", "").strip()
        return None

    try:
        cards = [os.path.dirname(f) for f in sorted(glob.glob("/sys/class/drm/card*/device/pp_dpm_sclk"))]
        if not cards:
            return None
        for _ in range(3):                      # let the clocks ramp, then leave a backlog on the stream
            burst()
        torch.cuda.synchronize()
        for _ in range(8):
            burst()
        seen = [(current(c + "/pp_dpm_sclk"), current(c + "/pp_dpm_mclk"), c) for c in cards]
        torch.cuda.synchronize()
        mhz = lambda v: int("".join(ch for ch in (v or "0") if ch.isdigit()) or 0)
        sclk, mclk, card = max(seen, key=lambda r: mhz(r[0]))       # the busy card, should the machine show several
        pick = {"sclk": sclk, "mclk": mclk}
        caps = glob.glob(card + "/hwmon/hwmon*/power1_cap")
        if caps:
            pick["power_cap_W"] = int(open(caps[0]).read()) / 1e6
        return pick
    except Exception:
        return None


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=8,
                    help="timed steps; a step = the verify block through every resident layer once (--layers layer passes)")
    ap.add_argument("--warmup", type=int, default=2, help="untimed steps in front of the timed ones (after the settling passes)")
    ap.add_argument("--layers", type=int, default=30)
    ap.add_argument("--tokens", type=int, default=16)
    ap.add_argument("--prefill-tokens", type=int, default=3072, help="0 skips the prefill leg")
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--no-decode", action="store_true", help="skip the secondary decode (T = 1) leg")
    ap.add_argument("--no-gemv", action="store_true", help="skip the INT4 GEMV legs (config 1 and the LM head)")
    ap.add_argument("--no-fp16", action="store_true", help="skip the FP16-activation leg (same context switched to FFMOE_FP16)")
    ap.add_argument("--no-shared", action="store_true", help="skip the shared-expert (dense INT4 FFN, width 2112) leg")
    ap.add_argument("--copy-probe", action="store_true",
                    help="also run a plain 1 GiB device-to-device copy three times: the known-size kernel that "
                         "FETCH_SIZE / WRITE_SIZE readings of a rocprofv3 --pmc run are scaled by")
    ap.add_argument("--no-sweep", action="store_true",
                    help="skip BASELINE.json config 5 (8,192-token Zipf prefill over all layers, then 256 decode steps "
                         "as 16 verify blocks with the LM head once per block)")
    ap.add_argument("--tune-dense", action="store_true",
                    help="also time the dense bf16 ceiling after the library tuned itself for the two shapes (TunableOp)")
    ap.add_argument("--no-zipf", action="store_true",
                    help="skip the Zipf(1.1) half of the prefill leg (so that a profiler's per-kernel averages of the prefill "
                         "kernels cover the router-made, near-uniform routes alone)")
    ap.add_argument("--sweep", action="store_true", help="accepted for older command lines: the sweep runs by default")
    args = ap.parse_args()
    args.sweep = not args.no_sweep and not args.no_gemv
    if args.gpus != 1:
        print("bench.py measures the one-GPU hot path only; --gpus must be 1 "
              "(the path has no collective; it would shard by expert, each GPU running its own experts' share)", file=sys.stderr)
        sys.exit(2)

    import torch
    import fieldfare_moe as ff
    from fieldfare_moe import synthetic as syn
    ff.ensure_built()                     # loads what is built in-tree; compiles only if nothing (current) is
    oracle = None
    cpu_flags = "gcc -O3 -march=x86-64-v3 -ffp-contract=off -fno-fast-math -fopenmp (the in-tree build)"
    if not args.no_cpu:                   # the CPU oracle is the checker and the cpu_baseline leg, nothing else here
        from oracle import oracle
        import tempfile
        native = oracle.use_native_build(tempfile.mkdtemp(prefix="ffmoe_oracle_"))      # this host's own instruction set
        if native:
            cpu_flags = "gcc " + native + " (compiled on this host for the baseline)"

    assert torch.cuda.is_available(), "bench.py needs a HIP device"
    torch.cuda.set_device(0)
    L, T = args.layers, args.tokens
    gen = torch.Generator(device="cuda")
    gen.manual_seed(0)
    rng = np.random.default_rng(0)
    ff_off, payload = syn.layout_offsets(D, F, align=16)
    assert payload == EXPERT_BYTES and (syn.D, syn.F, syn.E, syn.K, syn.STRIDE) == (D, F, E, K, STRIDE)
    traffic = measured_traffic()

    ctx = ff.Context(D, F, E, K, n_layers=L, max_tokens=max(8192 if args.sweep else 4096, args.prefill_tokens))
    config1 = None
    host_layer0 = None
    routers = []
    for layer in range(L):
        blob = syn.synth_layer_gpu(torch, gen, ff_off)
        ctx.upload_layer(layer, blob.view(-1), STRIDE, ff_off)
        if layer == 0 and not args.no_cpu:
            host_layer0 = blob.view(-1).cpu().numpy()
        del blob
        r = syn.router_weights(rng)
        routers.append(r)
        ctx.upload_router_bf16(layer, r)
    torch.cuda.empty_cache()

    xb = syn.bf16_bits(syn.block_tokens(rng, T))
    x = torch.from_numpy(xb.view(np.int16)).cuda().view(torch.bfloat16)
    idx = torch.empty((T, K), dtype=torch.int32, device="cuda")
    w = torch.empty((T, K), dtype=torch.bfloat16, device="cuda")
    y = torch.empty((T, D), dtype=torch.bfloat16, device="cuda")

    import ctypes as C
    Lib, h = ctx.L, ctx._h
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    px, pidx, pw, py = (C.c_void_p(t_.data_ptr()) for t_ in (x, idx, w, y))
    err = C.c_char_p()

    def step_split(layer):
        rc = Lib.ffmoe_router(h, stream, layer, px, D, T, pidx, pw, None, C.byref(err))
        rc |= Lib.ffmoe_verify(h, stream, layer, px, D, T, pidx, pw, None, py, C.byref(err))
        if rc:
            raise RuntimeError(err.value)

    def step(layer):
        # router and expert pass of the block in one call (router logits, select and gate/up share a launch)
        rc = Lib.ffmoe_route_verify(h, stream, layer, px, D, px, D, T, None, py, pidx, pw, C.byref(err))
        if rc:
            raise RuntimeError(err.value)

    if os.environ.get("FFMOE_BENCH_SPLIT"):
        step = step_split

    # distinct experts per layer for this block (decides the algorithmic bytes of each step)
    live = []
    tokens_per_expert = np.zeros(T * K + 1, np.int64)     # [n]: live experts that n of the block's routes go to
    for layer in range(L):
        step(layer)
        live.append(ctx.last_live_experts())
        per_expert = np.bincount(idx.cpu().numpy().astype(np.int64).ravel(), minlength=E)
        assert int((per_expert > 0).sum()) == live[-1], "plan and routes disagree on the live experts"
        tokens_per_expert += np.bincount(per_expert[per_expert > 0], minlength=T * K + 1)
    # A step = the block through all L resident layers, one after the other, as a decode loop runs them (L layer
    # passes; every pass streams its own layer's experts from HBM). The clocks and the address translation caches
    # settle over the first ~15 ms of back-to-back passes (with 30 passes in front the timed ones still ran 5 % below
    # the settled rate), so kSettlePasses untimed passes come first, whatever --warmup says; then the warm-up steps,
    # then exactly --steps timed steps between two device synchronisations.
    kSettlePasses = 300
    n_warm, n_timed = args.warmup * L, args.steps * L
    # What a short run without the settling passes reads (the method of this benchmark's first form: a step = one layer
    # pass, 5 warm-up passes, 20 timed ones, a timed region of about 1 ms between two synchronisations), for comparison.
    time.sleep(0.5)
    for i in range(5):
        step(i % L)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(20):
        step((5 + i) % L)
    torch.cuda.synchronize()
    cold_el = time.perf_counter() - t0
    cold_value = sum(live[(5 + i) % L] for i in range(20)) * EXPERT_BYTES / cold_el / 1e9
    for i in range(kSettlePasses + n_warm):
        step(i % L)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(n_timed):
        step(i % L)
    torch.cuda.synchronize()
    elapsed = time.perf_counter() - t0
    ms_per_step = elapsed * 1e3 / args.steps
    bytes_total = args.steps * sum(live) * EXPERT_BYTES
    value = bytes_total / elapsed / 1e9
    giveups = ctx.handover_giveups()     # waves of the one-launch routing that stopped waiting for another block: 0 on a GPU of its own

    # The ceiling of the expert stream on this box, measured in this run: ffmoe_probe_stream issues exactly the weight
    # loads of the gate/up and the down kernel for as many experts as the block touches in each layer - no routing, no
    # rows, no arithmetic, no output - as two launches per layer pass over the same cycled layers.
    def probe(layer):
        rc = Lib.ffmoe_probe_stream(h, stream, layer, live[layer], C.byref(err))
        if rc:
            raise RuntimeError(err.value)
    for i in range(2 * L):
        probe(i % L)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for i in range(n_timed):
        probe(i % L)
    torch.cuda.synchronize()
    probe_el = time.perf_counter() - t0
    ceiling_value = bytes_total / probe_el / 1e9

    # spread of the step time: one event after every step (a record costs the stream a few microseconds, so
    # these intervals sit above ms_per_step by about one record; the spread is what they are for)
    n_spread = min(n_timed, 240)
    evs = [torch.cuda.Event(enable_timing=True) for _ in range(n_spread + 1)]
    evs[0].record()
    for i in range(n_spread):
        step(i % L)
        evs[i + 1].record()
    torch.cuda.synchronize()
    per_step = np.array([evs[i].elapsed_time(evs[i + 1]) * 1e3 for i in range(n_spread)])
    step_spread = {"median": round(float(np.median(per_step)), 2), "p10": round(float(np.percentile(per_step, 10)), 2),
                   "p90": round(float(np.percentile(per_step, 90)), 2), "n": int(n_spread),
                   "note": "per-layer-pass HIP-event intervals, each including one event record"}
    props = torch.cuda.get_device_properties(0)
    device_info = {"name": props.name, "compute_units": props.multi_processor_count,
                   "hbm_GiB": round(props.total_memory / 2 ** 30, 1), "torch": torch.__version__, "hip": torch.version.hip,
                   "clocks_under_load": clocks_under_load(lambda: [step(i % L) for i in range(4 * L)], torch)}

    if args.copy_probe:
        src_c = torch.empty(1 << 28, dtype=torch.float32, device="cuda").normal_()
        dst_c = torch.empty_like(src_c)
        for _ in range(3):
            dst_c.copy_(src_c)
        torch.cuda.synchronize()
        del src_c, dst_c
        torch.cuda.empty_cache()

    # per-kernel times (HIP events on the launch stream) for the same steps
    ctx.set_profiling(True)
    ctx.profile(reset=True)
    for i in range(n_timed):
        step(i % L)
    prof = ctx.profile(reset=True)
    for i in range(n_timed):
        probe(i % L)
    probe_prof = ctx.profile(reset=True)
    ctx.set_profiling(False)
    # An event record costs the stream a few microseconds. The library measures an empty interval (two
    # records with nothing between them, once per call); a kernel's interval carries half of that - one
    # record's worth - on top of the kernel's own duration, which is what rocprofv3 --kernel-trace shows
    # (gate/up: 29.5 us raw, 5.2 us empty interval, 26.9 us corrected, 27.3 us in the trace).
    gap_ms = 0.5 * prof["event_gap"][0] / prof["event_gap"][1] if "event_gap" in prof else 0.0

    def kernel_times(pr):
        return {k_: round((v[0] / v[1] - gap_ms) * 1e3, 2) for k_, v in pr.items() if k_ != "event_gap"}
    kernel_us = kernel_times(prof)
    live_sum = args.steps * sum(live)
    if "route_gate_up" in prof:
        # router logits, select and gate/up share one launch: its bytes are the live experts' gate/up weights plus the
        # router's [E][D] bf16 matrix, its time holds the routing chain as well
        dominant = "route_gate_up_persistent (router logits + top-8 select + gate/up in one launch)"
        gu_ms = prof["route_gate_up"][0] - gap_ms * prof["route_gate_up"][1]
        achieved = (live_sum * GATE_UP_BYTES + n_timed * E * D * 2) / (gu_ms * 1e-3) / 1e9
    else:
        dominant = "skinny_gate_up_persistent"
        gu_ms = prof["gate_up"][0] - gap_ms * prof["gate_up"][1]
        achieved = live_sum * GATE_UP_BYTES / (gu_ms * 1e-3) / 1e9
    down_gbs = live_sum * DOWN_BYTES / ((prof["down"][0] - gap_ms * prof["down"][1]) * 1e-3) / 1e9
    probe_us = kernel_times(probe_prof)
    pg_ms = probe_prof["probe_gate_up"][0] - gap_ms * probe_prof["probe_gate_up"][1]
    pd_ms = probe_prof["probe_down"][0] - gap_ms * probe_prof["probe_down"][1]
    ceiling_gu = live_sum * GATE_UP_BYTES / (pg_ms * 1e-3) / 1e9
    ceiling_dn = live_sum * DOWN_BYTES / (pd_ms * 1e-3) / 1e9
    stream_ceiling = {
        "what": "ffmoe_probe_stream: the tile and scale loads of the gate/up and the down kernel for the same number of "
                "experts per layer, in those kernels' grids and order, and nothing else; two launches per layer pass, same cycled layers",
        "us_per_layer_pass": round(probe_el * 1e6 / n_timed, 2), "GBs": round(ceiling_value, 1),
        "frac_hbm_peak": round(ceiling_value / HBM_PEAK_GBS, 4),
        "value_frac_of_ceiling": round(value / ceiling_value, 4),
        "kernel_us": {"probe_gate_up": probe_us.get("probe_gate_up"), "probe_down": probe_us.get("probe_down")},
        "gate_up_stream_GBs": round(ceiling_gu, 1), "down_stream_GBs": round(ceiling_dn, 1),
        "down_kernel_frac_of_ceiling": round(down_gbs / ceiling_dn, 4)}
    # the same steps as ffmoe_router + ffmoe_verify (five launches): what the gate/up stream does as a launch of its own,
    # without the routing chain in front of it, and what the one-call form gains on the whole step
    split = None
    if "route_gate_up" in prof:
        for i in range(max(n_warm, 2 * L)):
            step_split(i % L)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for i in range(n_timed):
            step_split(i % L)
        torch.cuda.synchronize()
        split_ms = (time.perf_counter() - t0) * 1e3 / n_timed
        ctx.set_profiling(True)
        ctx.profile(reset=True)
        for i in range(n_timed):
            step_split(i % L)
        sprof = ctx.profile(reset=True)
        ctx.set_profiling(False)
        sgu_ms = sprof["gate_up"][0] - gap_ms * sprof["gate_up"][1]
        sgbs = live_sum * GATE_UP_BYTES / (sgu_ms * 1e-3) / 1e9
        split = {"calls": "ffmoe_router + ffmoe_verify (router logits, select, gate/up, down, combine: five launches)",
                 "us_per_layer_pass": round(split_ms * 1e3, 2), "kernel_us": kernel_times(sprof),
                 "gate_up_kernel": "skinny_gate_up_persistent", "gate_up_GBs": round(sgbs, 1),
                 "gate_up_frac_hbm_peak": round(sgbs / HBM_PEAK_GBS, 4)}

    # secondary figures: decode step (T = 1) and config-1 GEMV
    extra = {"event_record_us": round(gap_ms * 1e3, 2)}
    x1 = x[:1].contiguous()
    px1 = C.c_void_p(x1.data_ptr())

    def decode(layer):
        # two launches: router + select + gate/up, then down + combine
        Lib.ffmoe_route_verify(h, stream, layer, px1, D, px1, D, 1, None, py, pidx, pw, C.byref(err))

    if not args.no_decode:
        for name_, fn_ in (("decode_us_per_layer", decode),):
            for i in range(L):
                fn_(i)
            torch.cuda.synchronize()
            runs = []
            for _ in range(7):          # a run is 3 ms: the median of seven keeps a stray host hiccup out
                t0 = time.perf_counter()
                for i in range(4 * L):
                    fn_(i % L)
                torch.cuda.synchronize()
                runs.append((time.perf_counter() - t0) / (4 * L))
            dec = float(np.median(runs))
            extra[name_] = round(dec * 1e6, 2)
            extra[name_ + "_min_max"] = [round(min(runs) * 1e6, 2), round(max(runs) * 1e6, 2)]
        extra["decode_expert_GBs"] = round(K * EXPERT_BYTES / dec / 1e9, 1)

    # prefill half of the metric: 3,072 tokens through one MoE layer, router
    # included, near-uniform routing from the Gaussian router; layers cycle as above
    TP = args.prefill_tokens
    prefill = None
    if TP > 0:
        xp_bits = syn.bf16_bits(rng.normal(0, 1, (TP, D)).astype(np.float32))
        xp = torch.from_numpy(xp_bits.view(np.int16)).cuda().view(torch.bfloat16)
        pidx_t = torch.empty((TP, K), dtype=torch.int32, device="cuda")
        pw_t = torch.empty((TP, K), dtype=torch.bfloat16, device="cuda")
        py_t = torch.empty((TP, D), dtype=torch.bfloat16, device="cuda")
        pxp, ppi, ppw, ppy = (C.c_void_p(t_.data_ptr()) for t_ in (xp, pidx_t, pw_t, py_t))

        def pstep(layer):
            rc = Lib.ffmoe_router(h, stream, layer, pxp, D, TP, ppi, ppw, None, C.byref(err))
            rc |= Lib.ffmoe_prefill(h, stream, layer, pxp, D, TP, ppi, ppw, ppy, C.byref(err))
            if rc:
                raise RuntimeError(err.value)
        psteps = 2 * L                 # two passes over the layers (25 ms), whatever --steps says
        for i in range(2 * L):          # and two in front of them: clocks and address translation settled
            pstep(i % L)
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for i in range(psteps):
            pstep(i % L)
        torch.cuda.synchronize()
        pel = (time.perf_counter() - t0) / psteps
        n_pairs, n_tiles, counts = ctx.prefill_stats()
        ctx.set_profiling(True)
        ctx.profile(reset=True)
        for i in range(psteps):
            pstep(i % L)
        pprof = ctx.profile(reset=True)
        ctx.set_profiling(False)
        pk_us = kernel_times(pprof)
        flops_gu = n_pairs * 2.0 * (2 * F * D)
        flops_dn = n_pairs * 2.0 * (D * F)
        gemm_s = ((pprof["prefill_gate_up"][0] + pprof["prefill_down"][0]) / psteps - 2 * gap_ms) * 1e-3
        prefill = {"tokens": TP, "tok_per_s": round(TP / pel, 1), "ms_per_layer": round(pel * 1e3, 4),
                   "pairs": n_pairs, "m_tiles": n_tiles, "pairs_per_expert_min": int(counts.min()),
                   "pairs_per_expert_max": int(counts.max()), "kernel_us": pk_us,
                   "roofline": {"bound": "mfma", "kernel": "prefill_gemm_kernel (gate_up + down)",
                                "achieved": round((flops_gu + flops_dn) / gemm_s / 1e12, 1), "peak": MFMA_BF16_PEAK_TFLOPS,
                                "unit": "TFLOP/s", "frac": round((flops_gu + flops_dn) / gemm_s / 1e12 / MFMA_BF16_PEAK_TFLOPS, 4),
                                "traffic": traffic.get("prefill3072_gemms") if TP == 3072 else None,
                                "traffic_unit": f"HBM bytes of the two launches (rocprofv3 --pmc, profiles/{TRAFFIC_FILE.name})"}}
        # The dense bf16 GEMM ceiling of this box in the same run: the two products of the chunk's n_pairs rows as plain
        # library GEMMs (torch.matmul -> hipBLASLt / rocBLAS) on bf16 operands - no INT4 expansion, no gather, one
        # weight matrix instead of 128, a shape the library is tuned for.
        mrows = int(n_pairs)
        a_gu = torch.randn((mrows, D), device="cuda", generator=gen).to(torch.bfloat16)
        b_gu = torch.randn((D, 2 * F), device="cuda", generator=gen).to(torch.bfloat16)
        a_dn = torch.randn((mrows, F), device="cuda", generator=gen).to(torch.bfloat16)
        b_dn = torch.randn((F, D), device="cuda", generator=gen).to(torch.bfloat16)
        o_gu = torch.empty((mrows, 2 * F), dtype=torch.bfloat16, device="cuda")
        o_dn = torch.empty((mrows, D), dtype=torch.bfloat16, device="cuda")

        def dense_time(a_, b_, o_):
            for _ in range(5):
                torch.matmul(a_, b_, out=o_)
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(20):
                torch.matmul(a_, b_, out=o_)
            e1.record()
            torch.cuda.synchronize()
            return e0.elapsed_time(e1) * 1e-3 / 20
        # both operand layouts of the weight ([K x N] and the transposed view of [N x K]); the faster one counts
        bt_gu, bt_dn = b_gu.t().contiguous(), b_dn.t().contiguous()
        t_dgu = min(dense_time(a_gu, b_gu, o_gu), dense_time(a_gu, bt_gu.t(), o_gu))
        t_ddn = min(dense_time(a_dn, b_dn, o_dn), dense_time(a_dn, bt_dn.t(), o_dn))
        tuned = None
        if args.tune_dense:
            # the same products after the library searched its own solutions for them (torch's TunableOp: a few seconds
            # per shape and layout); its result file goes to the temporary directory
            try:
                torch.cuda.tunable.enable(True)
                torch.cuda.tunable.tuning_enable(True)
                import tempfile
                torch.cuda.tunable.set_filename(os.path.join(tempfile.gettempdir(), "ffmoe_bench_tunableop.csv"))
                torch.cuda.tunable.set_max_tuning_duration(30)
                t_tgu = min(dense_time(a_gu, b_gu, o_gu), dense_time(a_gu, bt_gu.t(), o_gu))
                t_tdn = min(dense_time(a_dn, b_dn, o_dn), dense_time(a_dn, bt_dn.t(), o_dn))
                tuned_tf = (flops_gu + flops_dn) / (t_tgu + t_tdn) / 1e12
                tuned = {"gate_up_us": round(t_tgu * 1e6, 1), "down_us": round(t_tdn * 1e6, 1),
                         "frac_mfma_peak": round(tuned_tf / MFMA_BF16_PEAK_TFLOPS, 4),
                         "gemm_frac_of_tuned_dense": round((flops_gu + flops_dn) / gemm_s / 1e12 / tuned_tf, 4)}
            finally:
                torch.cuda.tunable.tuning_enable(False)
                torch.cuda.tunable.enable(False)
        del bt_gu, bt_dn
        dense_tf = (flops_gu + flops_dn) / (t_dgu + t_ddn) / 1e12
        prefill["dense_bf16_ceiling_TFLOPs"] = round(dense_tf, 1)
        prefill["dense_bf16_ceiling"] = {
            "gate_up_us": round(t_dgu * 1e6, 1), "down_us": round(t_ddn * 1e6, 1),
            "shapes": f"[{mrows} x {D}] . [{D} x {2 * F}] and [{mrows} x {F}] . [{F} x {D}], bf16, torch.matmul, the faster of the weight as [K x N] and as [N x K] transposed",
            "frac_mfma_peak": round(dense_tf / MFMA_BF16_PEAK_TFLOPS, 4),
            "gemm_frac_of_dense_ceiling": round((flops_gu + flops_dn) / gemm_s / 1e12 / dense_tf, 4)}
        if tuned:
            prefill["dense_bf16_ceiling"]["tuned_by_the_library"] = tuned
        del a_gu, b_gu, a_dn, b_dn, o_gu, o_dn
        # BASELINE.json config 4 (ii): the same chunk with Zipf(1.1) routing imposed on the experts
        # (indices and weights given, no router): a few experts hold most pairs, many hold a handful
        if not args.no_zipf:
            zidx_, zw_ = syn.zipf_routes(np.random.default_rng(4), TP)
            pidx_t.copy_(torch.from_numpy(zidx_))
            pw_t.copy_(torch.from_numpy(syn.bf16_bits(zw_).view(np.int16)).view(torch.bfloat16))

            def zstep(layer):
                if Lib.ffmoe_prefill(h, stream, layer, pxp, D, TP, ppi, ppw, ppy, C.byref(err)):
                    raise RuntimeError(err.value)
            for i in range(4):
                zstep(i % L)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for i in range(psteps):
                zstep(i % L)
            torch.cuda.synchronize()
            zel = (time.perf_counter() - t0) / psteps
            _, z_tiles, zcounts = ctx.prefill_stats()
            prefill["zipf_1p1"] = {"tok_per_s": round(TP / zel, 1), "ms_per_layer": round(zel * 1e3, 4), "m_tiles": z_tiles,
                                   "pairs_per_expert_min": int(zcounts.min()), "pairs_per_expert_max": int(zcounts.max()),
                                   "pairs_per_expert_median": int(np.median(zcounts)), "router": "not run (routes imposed)"}

    def timed(fn, reps, warm=3):
        for _ in range(warm):
            fn()
        torch.cuda.synchronize()
        t0_ = time.perf_counter()
        for _ in range(reps):
            fn()
        torch.cuda.synchronize()
        return (time.perf_counter() - t0_) / reps

    # The same steps with FP16 rows (the reference's text-path type): the context is switched, run and switched back
    if not args.no_fp16:
        ctx.set_act_dtype("fp16")
        xh = x.to(torch.float16)
        wh = torch.empty((T, K), dtype=torch.float16, device="cuda")
        yh = torch.empty((T, D), dtype=torch.float16, device="cuda")
        pxh, pwh, pyh = (C.c_void_p(t_.data_ptr()) for t_ in (xh, wh, yh))

        def step16(layer, rows):
            rc = Lib.ffmoe_route_verify(h, stream, layer, pxh, D, pxh, D, rows, None, pyh, pidx, pwh, C.byref(err))
            if rc:
                raise RuntimeError(err.value)
        fp16 = {}
        for name_, rows in (("verify16_us_per_layer", T), ("decode_us_per_layer", 1)):
            for i in range(L):
                step16(i, rows)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for i in range(4 * L):
                step16(i % L, rows)
            torch.cuda.synchronize()
            fp16[name_] = round((time.perf_counter() - t0) / (4 * L) * 1e6, 2)
        if args.prefill_tokens:
            TPh = args.prefill_tokens
            xph = torch.from_numpy(rng.normal(0, 1, (TPh, D)).astype(np.float16).view(np.int16)).cuda().view(torch.float16)
            ih = torch.empty((TPh, K), dtype=torch.int32, device="cuda")
            wph = torch.empty((TPh, K), dtype=torch.float16, device="cuda")
            yph = torch.empty((TPh, D), dtype=torch.float16, device="cuda")
            pxph, pih, pwph, pyph = (C.c_void_p(t_.data_ptr()) for t_ in (xph, ih, wph, yph))

            def pstep16(layer):
                rc = Lib.ffmoe_router(h, stream, layer, pxph, D, TPh, pih, pwph, None, C.byref(err))
                rc |= Lib.ffmoe_prefill(h, stream, layer, pxph, D, TPh, pih, pwph, pyph, C.byref(err))
                if rc:
                    raise RuntimeError(err.value)
            for i in range(2 * L):          # as for the bf16 figure: two passes over the layers in front, two timed
                pstep16(i % L)
            torch.cuda.synchronize()
            t0 = time.perf_counter()
            for i in range(2 * L):
                pstep16(i % L)
            torch.cuda.synchronize()
            fp16["prefill_ms_per_layer"] = round((time.perf_counter() - t0) / (2 * L) * 1e3, 4)
            ctx.set_profiling(True)
            ctx.profile(reset=True)
            for i in range(12):
                pstep16(i % L)
            fp16["prefill_kernel_us"] = kernel_times(ctx.profile(reset=True))
            ctx.set_profiling(False)
            del xph, ih, wph, yph
        fp16["note"] = "FFMOE_FP16: router, experts and combine on FP16 rows; the prefill multiplies FP16 rows by FP16 tiles and keeps block-scaled FP16 activations (the reference's FP16 prefill arithmetic)"
        extra["fp16_mode"] = fp16
        ctx.set_act_dtype("bf16")

    # INT4 GEMV: BASELINE.json config 1 ([1408 x 2816], one input row) and the LM head of config 5
    # ([262144 x 2816]) as resident matrices; synthetic weights as in synth_layer_gpu
    head = None
    head_sample = None
    if not args.no_gemv:
        def synth_matrix(m):
            return syn.synth_matrix_gpu(torch, gen, m)
        gemv = {}
        W1, S1, B1 = synth_matrix(2 * F)
        m1 = ctx.matrix(W1, S1, B1)
        bytes1 = 2 * F * D // 2 + 2 * (2 * F) * (D // 64) * 2
        x1row = x[:1].contiguous()
        t_res = timed(lambda: m1.gemv(x1row), 200)
        t_raw = timed(lambda: ctx.gemv_int4(W1, S1, B1, x1row), 200)
        # the kernels' own durations (HIP events on the launch stream, less one event record), beside the host-timed calls
        ctx.set_profiling(True)
        ctx.profile(reset=True)
        for _ in range(50):
            m1.gemv(x1row)
        k_res = kernel_times(ctx.profile(reset=True)).get("gemv")
        for _ in range(50):
            ctx.gemv_int4(W1, S1, B1, x1row)
        k_raw = kernel_times(ctx.profile(reset=True)).get("gemv")
        ctx.set_profiling(False)
        gemv["config1_1408x2816"] = {"resident_us": round(t_res * 1e6, 2), "resident_GBs": round(bytes1 / t_res / 1e9, 1),
                                     "resident_kernel_us": k_res, "resident_kernel_GBs": round(bytes1 / (k_res * 1e-6) / 1e9, 1) if k_res else None,
                                     "reference_layout_us": round(t_raw * 1e6, 2), "reference_layout_kernel_us": k_raw, "bytes": bytes1,
                                     "note": "host-timed back-to-back calls next to the kernel's own duration: launch latency, "
                                             "not bandwidth, bounds a 2.2 MB GEMV"}
        config1 = (W1.cpu().numpy(), S1.view(torch.int16).cpu().numpy().view(np.uint16), B1.view(torch.int16).cpu().numpy().view(np.uint16))
        m1.close()
        V = 262144
        Wh, Sh, Bh = synth_matrix(V)
        if not args.no_cpu:             # the first 16,384 rows on the host, for the CPU baseline's head leg
            head_sample = (Wh[:16384].cpu().numpy(), Sh[:16384].view(torch.int16).cpu().numpy().view(np.uint16),
                           Bh[:16384].view(torch.int16).cpu().numpy().view(np.uint16))
        head = ctx.matrix(Wh, Sh, Bh, greedy=True)
        del Wh, Sh, Bh
        torch.cuda.empty_cache()
        head_bytes = V * D // 2 + 2 * V * (D // 64) * 2
        for rows in (1, 16):
            xr = x[:rows].contiguous()
            tg = timed(lambda: head.gemv(xr, f32_out=True), 40, warm=20)
            gemv[f"lm_head_262144x2816_rows{rows}"] = {"us": round(tg * 1e6, 1), "GBs": round(head_bytes / tg / 1e9, 1),
                                                        "pct_hbm_peak": round(100 * head_bytes / tg / 1e9 / HBM_PEAK_GBS, 1)}
        tg = timed(lambda: head.greedy(x), 40, warm=20)
        gemv["lm_head_greedy_rows16_us"] = round(tg * 1e6, 1)
        extra["gemv"] = gemv

    # Shared expert: the model's dense INT4 FFN (2816 -> 2112 -> 2816) that every token passes beside the
    # routed experts, as a context of one expert; 16 rows (verify block) and the prefill chunk
    if not args.no_shared:
        FS, LS = 2112, 8
        s_off, s_payload = syn.layout_offsets(D, FS, align=16)
        dense = ff.Context(D, FS, 1, 1, n_layers=LS, max_tokens=max(args.prefill_tokens, 16))
        for layer in range(LS):
            blob = torch.empty(s_payload, dtype=torch.uint8, device="cuda")
            for (w_o, s_o, b_o), (rows, cols) in (((s_off.gate_w, s_off.gate_s, s_off.gate_b), (FS, D)),
                                                  ((s_off.up_w, s_off.up_s, s_off.up_b), (FS, D)),
                                                  ((s_off.down_w, s_off.down_s, s_off.down_b), (D, FS))):
                g_ = cols // 64
                blob[w_o:w_o + rows * cols // 2] = torch.randint(0, 256, (rows * cols // 2,), dtype=torch.uint8, device="cuda", generator=gen)
                sc = (torch.randn((rows, g_), device="cuda", generator=gen) * 0.01).abs().to(torch.bfloat16)
                bi = (-8.0 * sc.float() + torch.randn((rows, g_), device="cuda", generator=gen) * 1e-3).to(torch.bfloat16)
                blob[s_o:s_o + rows * g_ * 2] = sc.view(torch.uint8).view(-1)
                blob[b_o:b_o + rows * g_ * 2] = bi.view(torch.uint8).view(-1)
            dense.upload_layer(layer, blob, s_payload, s_off)
            del blob
        state = {"i": 0}

        def dense_step(xin, yout):
            dense.dense_ffn(state["i"] % LS, xin, out=yout)
            state["i"] += 1
        shared = {"shape": f"{D} -> {FS} -> {D}, INT4 g64", "bytes_per_layer": s_payload, "layers_cycled": LS}
        y16 = torch.empty((T, D), dtype=torch.bfloat16, device="cuda")
        t16 = timed(lambda: dense_step(x, y16), 200, warm=10)
        shared["rows16"] = {"us": round(t16 * 1e6, 2), "GBs": round(s_payload / t16 / 1e9, 1)}
        x1s, y1s = x[:1].contiguous(), torch.empty((1, D), dtype=torch.bfloat16, device="cuda")
        t1 = timed(lambda: dense_step(x1s, y1s), 200, warm=10)
        shared["rows1"] = {"us": round(t1 * 1e6, 2), "GBs": round(s_payload / t1 / 1e9, 1)}
        # the same FFN in the 8-bit form the reference's packs hold by default (SharedExpertInt8.swift:56-135): two nibble
        # planes per weight on the 4-bit streaming kernels, as layers of a second dense context; gate and up are one gated
        # matrix (the activation is that pass's epilogue), then the down projection: two launches per call
        dense8 = ff.Context(D, FS, 1, 1, n_layers=LS, max_tokens=max(args.prefill_tokens, 16))
        bytes8 = 0
        for layer in range(LS):
            parts8 = []
            for rows, cols in ((FS, D), (FS, D), (D, FS)):
                g_ = cols // 64
                w8 = torch.randint(0, 256, (rows, cols), dtype=torch.uint8, device="cuda", generator=gen)
                sc = (torch.randn((rows, g_), device="cuda", generator=gen) * 0.001).abs().to(torch.bfloat16)
                bi = (-128.0 * sc.float() + torch.randn((rows, g_), device="cuda", generator=gen) * 1e-3).to(torch.bfloat16)
                parts8.append((w8, sc.contiguous(), bi.contiguous()))
                bytes8 += (rows * cols + 4 * rows * g_) if layer == 0 else 0
            dense8.upload_expert_parts(layer, 0, *parts8, int8=True)
            del parts8

        def int8_step(xin, yout):
            dense8.dense_ffn(state["i"] % LS, xin, out=yout)
            state["i"] += 1
        t8_16 = timed(lambda: int8_step(x, y16), 200, warm=10)
        t8_1 = timed(lambda: int8_step(x1s, y1s), 200, warm=10)
        shared["int8"] = {"bytes_per_layer": bytes8, "launches": 2,
                          "rows16": {"us": round(t8_16 * 1e6, 2), "GBs": round(bytes8 / t8_16 / 1e9, 1)},
                          "rows1": {"us": round(t8_1 * 1e6, 2), "GBs": round(bytes8 / t8_1 / 1e9, 1)}}
        # a short prompt / a chunk's ragged end: 64 and 256 rows, both widths (a grid row of the streaming kernels per 16 rows)
        if args.prefill_tokens >= 256:
            for rows_m in (64, 256):
                xm = torch.randn((rows_m, D), device="cuda", generator=gen).to(torch.bfloat16)
                ym = torch.empty((rows_m, D), dtype=torch.bfloat16, device="cuda")
                tm4 = timed(lambda: dense_step(xm, ym), 100, warm=20)
                tm8 = timed(lambda: int8_step(xm, ym), 100, warm=20)
                shared[f"rows{rows_m}"] = {"us": round(tm4 * 1e6, 2)}
                shared["int8"][f"rows{rows_m}"] = {"us": round(tm8 * 1e6, 2)}
                del xm, ym
        if args.prefill_tokens:
            TPs = args.prefill_tokens
            xps = torch.randn((TPs, D), device="cuda", generator=gen).to(torch.bfloat16)
            yps = torch.empty((TPs, D), dtype=torch.bfloat16, device="cuda")
            tp_ = timed(lambda: dense_step(xps, yps), 60, warm=60)      # timed like the routed prefill: after as many steps in front
            fl = 2.0 * 3 * D * FS * TPs
            shared[f"rows{TPs}"] = {"us": round(tp_ * 1e6, 1), "TFLOPs": round(fl / tp_ / 1e12, 1),
                                    "frac_mfma_peak": round(fl / tp_ / 1e12 / MFMA_BF16_PEAK_TFLOPS, 4)}
            # the 8-bit layer at many rows: a 16-bit matrix element cannot hold q * s + b of an 8-bit q; from 385 rows on (at
            # this width) the GEMMs multiply by the integers q and bring scale and bias in with the sums
            tp8 = timed(lambda: int8_step(xps, yps), 24, warm=24)
            shared["int8"][f"rows{TPs}"] = {"us": round(tp8 * 1e6, 1),
                                            "form": "GEMMs on integer weights" if TPs >= 385 else "below the integer GEMMs' row count",
                                            "TFLOPs": round(fl / tp8 / 1e12, 1)}
            del xps, yps
        extra["shared_expert"] = shared

        # One decoder layer's MoE block for a 16-token verify block, as the reference schedules it
        # (RealForwardRunner.swift:454-756): post-attention setup, then the shared expert beside router +
        # routed experts (two streams, as the reference runs them concurrently), then the layer tail.
        main_s, side_s = torch.cuda.current_stream(), torch.cuda.Stream()
        hid_b = x.clone()
        att_b = torch.randn((T, D), device="cuda", generator=gen).to(torch.bfloat16)
        wn_b = [(torch.rand((D,), device="cuda", generator=gen) + 0.5).to(torch.bfloat16) for _ in range(5)]
        outs_b = tuple(torch.empty((T, D), dtype=torch.bfloat16, device="cuda") for _ in range(3))
        h1_b = torch.empty((T, D), dtype=torch.bfloat16, device="cuda")
        ev_fork, ev_join = torch.cuda.Event(), torch.cuda.Event()
        pouts = [C.c_void_p(o.data_ptr()) for o in outs_b]

        def layer_block(i, concurrent):
            layer = i % L
            ctx.post_attn_setup(hid_b, att_b, wn_b[0], wn_b[1], wn_b[2], out=outs_b)
            if concurrent:
                ev_fork.record(main_s)
                with torch.cuda.stream(side_s):
                    side_s.wait_event(ev_fork)
                    dense.dense_ffn(i % LS, outs_b[0], out=h1_b)
                    ev_join.record(side_s)
            else:
                dense.dense_ffn(i % LS, outs_b[0], out=h1_b)
            rc = Lib.ffmoe_route_verify(h, stream, layer, pouts[2], D, pouts[1], D, T, None, py, pidx, pw, C.byref(err))
            if rc:
                raise RuntimeError(err.value)
            if concurrent:
                main_s.wait_event(ev_join)
            ctx.layer_tail(y, h1_b, hid_b, wn_b[3], wn_b[4], 1.0)
        counter = {"i": 0}

        def run_block(concurrent):
            layer_block(counter["i"], concurrent)
            counter["i"] += 1
        def layer_block_fused(i):
            # the same block with the routed experts' combine folded into the layer tail: six launches
            layer = i % L
            ctx.post_attn_setup(hid_b, att_b, wn_b[0], wn_b[1], wn_b[2], out=outs_b)
            dense.dense_ffn(i % LS, outs_b[0], out=h1_b)
            rc = Lib.ffmoe_route_verify(h, stream, layer, pouts[2], D, pouts[1], D, T, None, None, pidx, pw, C.byref(err))
            if rc:
                raise RuntimeError(err.value)
            ctx.layer_tail_routed(w, h1_b, hid_b, wn_b[3], wn_b[4], 1.0)

        def run_fused():
            layer_block_fused(counter["i"])
            counter["i"] += 1

        def layer_block_inside(i):
            # the shared expert inside the routed experts' two launches as well: three launches
            ctx.post_attn_setup(hid_b, att_b, wn_b[0], wn_b[1], wn_b[2], out=outs_b)
            rc = Lib.ffmoe_route_verify_shared(h, dense._h, stream, i % L, i % LS, pouts[2], D, pouts[1], D, pouts[0], D, T,
                                               pidx, pw, C.byref(err))
            if rc:
                raise RuntimeError(err.value)
            ctx.layer_tail_routed_shared(dense, w, hid_b, wn_b[3], wn_b[4], 1.0)

        def run_inside():
            layer_block_inside(counter["i"])
            counter["i"] += 1
        def layer_block_int8(i, inside):
            # the block with the shared expert in the packs' default 8-bit form: separate calls with the combine in the
            # tail (six launches), or inside the routed experts' launches like the 4-bit one (four)
            ctx.post_attn_setup(hid_b, att_b, wn_b[0], wn_b[1], wn_b[2], out=outs_b)
            if inside:
                rc = Lib.ffmoe_route_verify_shared(h, dense8._h, stream, i % L, i % LS, pouts[2], D, pouts[1], D, pouts[0], D, T,
                                                   pidx, pw, C.byref(err))
                if rc:
                    raise RuntimeError(err.value)
                ctx.layer_tail_routed_shared(dense8, w, hid_b, wn_b[3], wn_b[4], 1.0)
                return
            dense8.dense_ffn(i % LS, outs_b[0], out=h1_b)
            rc = Lib.ffmoe_route_verify(h, stream, i % L, pouts[2], D, pouts[1], D, T, None, None, pidx, pw, C.byref(err))
            if rc:
                raise RuntimeError(err.value)
            ctx.layer_tail_routed(w, h1_b, hid_b, wn_b[3], wn_b[4], 1.0)

        def run_int8(inside):
            layer_block_int8(counter["i"], inside)
            counter["i"] += 1
        t_seq = timed(lambda: run_block(False), 120, warm=30)
        t_con = timed(lambda: run_block(True), 120, warm=30)
        t_i8 = timed(lambda: run_int8(False), 120, warm=30)
        t_i8c = timed(lambda: run_int8(True), 120, warm=30)
        t_fus = timed(run_fused, 120, warm=30)
        t_ins = timed(run_inside, 120, warm=30)
        # the same chain of L layers as a HIP graph: nine launches per layer from Python are host-bound,
        # a replay shows the device time (the library only enqueues kernels, so the chain captures as it is)
        graph_us = {}
        for label, conc in (("one_stream", False), ("shared_expert_on_second_stream", True), ("combine_in_layer_tail", None),
                            ("shared_expert_inside_routed_launches", "inside"), ("shared_expert_int8", "int8"),
                            ("shared_expert_int8_inside_routed_launches", "int8i")):
            gph = torch.cuda.CUDAGraph()
            cap = torch.cuda.Stream()
            cap.wait_stream(main_s)
            with torch.cuda.graph(gph, stream=cap):
                main_s = torch.cuda.current_stream()
                stream = C.c_void_p(main_s.cuda_stream)
                for i in range(L):
                    if conc == "inside":
                        layer_block_inside(i)
                    elif conc in ("int8", "int8i"):
                        layer_block_int8(i, conc == "int8i")
                    elif conc is None:
                        layer_block_fused(i)
                    else:
                        layer_block(i, conc)
            main_s = torch.cuda.current_stream()
            stream = C.c_void_p(main_s.cuda_stream)
            graph_us[label] = round(timed(gph.replay, 8, warm=2) / L * 1e6, 2)
            del gph
        extra["layer_block_rows16"] = {"one_stream_us": round(t_seq * 1e6, 2), "shared_expert_on_second_stream_us": round(t_con * 1e6, 2),
                                       "combine_in_layer_tail_us": round(t_fus * 1e6, 2),
                                       "shared_expert_inside_routed_launches_us": round(t_ins * 1e6, 2),
                                       "best_one_stream_us": round(min(t_seq, t_fus, t_ins) * 1e6, 2),
                                       "shared_expert_int8_us": round(t_i8 * 1e6, 2),
                                       "shared_expert_int8_inside_routed_launches_us": round(t_i8c * 1e6, 2),
                                       "launches": {"one_stream": 7, "combine_in_layer_tail": 6, "shared_expert_inside_routed_launches": 4,
                                                    "shared_expert_int8": 6, "shared_expert_int8_inside_routed_launches": 4},
                                       "hip_graph_replay_us": graph_us,
                                       "steps": "post-attention setup, shared expert, router, routed experts, layer tail"}
        # the same block for a decode step (one row), separate calls against the shared expert inside the routed launches
        hid1, att1 = hid_b[:1].contiguous(), att_b[:1].contiguous()
        outs1 = tuple(torch.empty((1, D), dtype=torch.bfloat16, device="cuda") for _ in range(3))
        h11 = torch.empty((1, D), dtype=torch.bfloat16, device="cuda")

        def block1_separate():
            i = counter["i"]
            counter["i"] += 1
            ctx.post_attn_setup(hid1, att1, wn_b[0], wn_b[1], wn_b[2], out=outs1)
            dense.dense_ffn(i % LS, outs1[0], out=h11)
            _, _, w1 = ctx.route_verify(i % L, outs1[2], outs1[1], combine=False)
            ctx.layer_tail_routed(w1, h11, hid1, wn_b[3], wn_b[4], 1.0)

        def block1_inside():
            i = counter["i"]
            counter["i"] += 1
            ctx.post_attn_setup(hid1, att1, wn_b[0], wn_b[1], wn_b[2], out=outs1)
            _, w1 = ctx.route_verify_shared(dense, i % L, i % LS, outs1[2], outs1[1], outs1[0])
            ctx.layer_tail_routed_shared(dense, w1, hid1, wn_b[3], wn_b[4], 1.0)
        def block1_int8(inside):
            i = counter["i"]
            counter["i"] += 1
            ctx.post_attn_setup(hid1, att1, wn_b[0], wn_b[1], wn_b[2], out=outs1)
            if inside:
                _, w1 = ctx.route_verify_shared(dense8, i % L, i % LS, outs1[2], outs1[1], outs1[0])
                ctx.layer_tail_routed_shared(dense8, w1, hid1, wn_b[3], wn_b[4], 1.0)
                return
            dense8.dense_ffn(i % LS, outs1[0], out=h11)
            _, _, w1 = ctx.route_verify(i % L, outs1[2], outs1[1], combine=False)
            ctx.layer_tail_routed(w1, h11, hid1, wn_b[3], wn_b[4], 1.0)
        t1_sep = timed(block1_separate, 120, warm=30)
        t1_ins = timed(block1_inside, 120, warm=30)
        t1_i8 = timed(lambda: block1_int8(False), 120, warm=30)
        t1_i8c = timed(lambda: block1_int8(True), 120, warm=30)
        # a serving loop replays the decode step as a HIP graph: L layers' blocks, shared expert inside, either width
        graph1_us = {}
        for label, fn in (("shared_expert_inside_routed_launches", block1_inside),
                          ("shared_expert_int8_inside_routed_launches", lambda: block1_int8(True))):
            gph = torch.cuda.CUDAGraph()
            cap = torch.cuda.Stream()
            cap.wait_stream(torch.cuda.current_stream())
            with torch.cuda.graph(gph, stream=cap):
                for _ in range(L):
                    fn()
            graph1_us[label] = round(timed(gph.replay, 8, warm=2) / L * 1e6, 2)
            del gph
        extra["layer_block_rows1"] = {"separate_calls_us": round(t1_sep * 1e6, 2),
                                      "hip_graph_replay_us": graph1_us,
                                      "shared_expert_inside_routed_launches_us": round(t1_ins * 1e6, 2),
                                      "shared_expert_int8_us": round(t1_i8 * 1e6, 2),
                                      "shared_expert_int8_inside_routed_launches_us": round(t1_i8c * 1e6, 2),
                                      "launches": {"separate_calls": 6, "shared_expert_inside_routed_launches": 4, "shared_expert_int8": 6,
                                                   "shared_expert_int8_inside_routed_launches": 4},
                                      "moe_blocks_of_30_layers_ms": round(30 * t1_ins * 1e3, 3),
                                      "steps": "post-attention setup, shared expert, router, routed experts, layer tail (combine in the tail)"}
        # the same block at the prefill chunk: setup, shared expert (4-bit grouped GEMMs / 8-bit GEMM form), router + routed
        # experts + combine, layer tail - one layer's MoE block for the chunk's tokens, shared expert in either width
        if args.prefill_tokens:
            TPb = args.prefill_tokens
            hid_p = torch.randn((TPb, D), device="cuda", generator=gen).to(torch.bfloat16)
            att_p = torch.randn((TPb, D), device="cuda", generator=gen).to(torch.bfloat16)
            outs_p = tuple(torch.empty((TPb, D), dtype=torch.bfloat16, device="cuda") for _ in range(3))
            h1_p = torch.empty((TPb, D), dtype=torch.bfloat16, device="cuda")
            h2_p = torch.empty((TPb, D), dtype=torch.bfloat16, device="cuda")

            def block_prefill(shared_ctx, concurrent=False):
                i = counter["i"]
                counter["i"] += 1
                ctx.post_attn_setup(hid_p, att_p, wn_b[0], wn_b[1], wn_b[2], out=outs_p)
                if concurrent:
                    # the shared expert beside router + sort + routed experts, as the reference schedules the two branches
                    ev_fork.record(main_s)
                    with torch.cuda.stream(side_s):
                        side_s.wait_event(ev_fork)
                        shared_ctx.dense_ffn(i % LS, outs_p[0], out=h1_p)
                        ev_join.record(side_s)
                else:
                    shared_ctx.dense_ffn(i % LS, outs_p[0], out=h1_p)
                idx_p, w_p = ctx.router(i % L, outs_p[2])
                ctx.prefill(i % L, outs_p[1], idx_p, w_p, out=h2_p)
                if concurrent:
                    main_s.wait_event(ev_join)
                ctx.layer_tail(h2_p, h1_p, hid_p, wn_b[3], wn_b[4], 1.0)
            tb4 = timed(lambda: block_prefill(dense), 2 * L, warm=2 * L)
            tb8 = timed(lambda: block_prefill(dense8), 2 * L, warm=2 * L)
            tb4c = timed(lambda: block_prefill(dense, True), 2 * L, warm=2 * L)
            tb8c = timed(lambda: block_prefill(dense8, True), 2 * L, warm=2 * L)
            extra[f"layer_block_rows{TPb}"] = {"shared_expert_4bit_ms": round(tb4 * 1e3, 4), "shared_expert_8bit_ms": round(tb8 * 1e3, 4),
                                               "shared_expert_4bit_on_second_stream_ms": round(tb4c * 1e3, 4),
                                               "shared_expert_8bit_on_second_stream_ms": round(tb8c * 1e3, 4),
                                               "tok_per_s_4bit": round(TPb / min(tb4, tb4c), 1), "tok_per_s_8bit": round(TPb / min(tb8, tb8c), 1),
                                               "steps": "post-attention setup, shared expert, router, routed experts + combine, layer tail"}
            del hid_p, att_p, outs_p, h1_p, h2_p
        dense.close()
        dense8.close()

    # The row-wise steps either side of the MoE stage at the prefill chunk and at a verify block:
    # 2 row reads + 4 row writes (setup), 3 reads + 1 write (tail); weights stay in cache
    if not args.no_shared:
        rowk = {}
        for rows_ in sorted({T, args.prefill_tokens} - {0}):
            hid = torch.randn((rows_, D), device="cuda", generator=gen).to(torch.bfloat16)
            att = torch.randn((rows_, D), device="cuda", generator=gen).to(torch.bfloat16)
            h1_ = torch.randn((rows_, D), device="cuda", generator=gen).to(torch.bfloat16)
            wn = [(torch.rand((D,), device="cuda", generator=gen) + 0.5).to(torch.bfloat16) for _ in range(5)]
            outs_ = tuple(torch.empty((rows_, D), dtype=torch.bfloat16, device="cuda") for _ in range(3))
            ts = timed(lambda: ctx.post_attn_setup(hid, att, wn[0], wn[1], wn[2], out=outs_), 50)
            tt = timed(lambda: ctx.layer_tail(att, h1_, hid, wn[3], wn[4], 1.0), 50)
            row_bytes = rows_ * D * 2
            rowk[f"rows{rows_}"] = {"post_attn_setup_us": round(ts * 1e6, 2), "post_attn_setup_GBs": round(6 * row_bytes / ts / 1e9, 1),
                                    "layer_tail_us": round(tt * 1e6, 2), "layer_tail_GBs": round(4 * row_bytes / tt / 1e9, 1)}
            del hid, att, h1_, outs_
        extra["row_kernels"] = rowk

    # all layers resident, one 8,192-token prefill with Zipf(1.1) routing imposed on
    # the experts, then 256 decode steps as 16 verify blocks of 16 tokens, the LM head once per block
    sweep = None
    if args.sweep:
        TS = 8192
        zr = np.random.default_rng(5)
        zidx, zw = syn.zipf_routes(zr, TS)
        xs_ = syn.bf16_cuda(torch, zr.normal(0, 1, (TS, D)).astype(np.float32))
        zi = torch.from_numpy(zidx).cuda()
        zwt = syn.bf16_cuda(torch, zw)
        ys_ = torch.empty((TS, D), dtype=torch.bfloat16, device="cuda")
        pzx, pzi, pzw, pzy = (C.c_void_p(t_.data_ptr()) for t_ in (xs_, zi, zwt, ys_))

        def prefill_all():
            for layer in range(L):
                rc = Lib.ffmoe_prefill(h, stream, layer, pzx, D, TS, pzi, pzw, pzy, C.byref(err))
                if rc:
                    raise RuntimeError(err.value)
        t_pf = timed(prefill_all, 2, warm=1)
        counts_z = np.bincount(zidx.ravel(), minlength=E)
        ctx.set_profiling(True)
        ctx.profile(reset=True)
        prefill_all()
        zprof = ctx.profile(reset=True)
        ctx.set_profiling(False)

        def decode_blocks():
            for _ in range(16):
                for layer in range(L):
                    step(layer)
                if head is not None:
                    head.greedy(x)
        t_dec = timed(decode_blocks, 2, warm=1)
        ctx.set_profiling(True)
        ctx.profile(reset=True)
        decode_blocks()
        dprof = ctx.profile(reset=True)
        ctx.set_profiling(False)
        flops_pf = L * TS * K * 2.0 * (3 * F * D)
        sweep = {
            "layers": L, "prefill_tokens": TS, "routing": "Zipf s=1.1 over a permuted expert order, 8 distinct experts per token",
            "pairs_per_expert_min": int(counts_z.min()), "pairs_per_expert_max": int(counts_z.max()),
            "prefill_ms_all_layers": round(t_pf * 1e3, 2), "prefill_tok_per_s_per_layer": round(TS * L / t_pf, 1),
            "prefill_expert_TFLOPs": round(flops_pf / t_pf / 1e12, 1),
            "prefill_kernel_ms": {k_: round(v[0], 3) for k_, v in zprof.items()},
            "decode_steps": 256, "decode_ms_256_steps": round(t_dec * 1e3, 2),
            "decode_us_per_block_layer": round(t_dec * 1e6 / (16 * L), 2),
            "decode_kernel_ms": {k_: round(v[0], 3) for k_, v in dprof.items()},
            "lm_head_included": head is not None,
            "note": "router of the prefill is imposed (not run); decode blocks run router + experts per layer and the "
                    "LM-head greedy choice once per block; times are host-timed whole phases, kernel_ms are HIP-event sums",
        }
    if head is not None:
        head.close()

    cpu = None
    if not args.no_cpu:
        # The CPU oracle (a C restatement of the reference's Swift test-support CPU path: dequantise, then multiply)
        # on the host's cores, bounded samples of the same workloads. Threads: what one GPU has of its host (16 for
        # it; OMP_NUM_THREADS says so), whatever the OS shows.
        from concurrent.futures import ThreadPoolExecutor
        o_off, _ = oracle.layout_offsets(D, F, align=16)
        pool = oracle.ExpertPool(host_layer0, o_off, STRIDE, D, F)
        threads = min(16, oracle.max_threads())
        nproc, cpu_model = host_cpu()

        def best_of(fn, budget_s, min_reps=2):
            reps, t_best, t_start = 0, float("inf"), time.perf_counter()
            while reps < min_reps or time.perf_counter() - t_start < budget_s:
                t0_ = time.perf_counter()
                fn()
                t_best = min(t_best, time.perf_counter() - t0_)
                reps += 1
            return t_best, reps

        # config 3 (the headline): layer 0 of the same 16-token block
        t0 = time.perf_counter()
        ridx, rw, ry = oracle.moe_layer(pool, routers[0], xb, K, threads=1)
        single = time.perf_counter() - t0
        multi, reps = best_of(lambda: oracle.moe_layer(pool, routers[0], xb, K, threads=threads), 1.5, 3)
        cpu_bytes = len(np.unique(ridx)) * EXPERT_BYTES
        legs = {"config3_verify16": {"GBs_1_thread": round(cpu_bytes / single / 1e9, 3), f"GBs_{threads}_threads": round(cpu_bytes / multi / 1e9, 3),
                                     "ms_1_thread": round(single * 1e3, 1), f"ms_{threads}_threads": round(multi * 1e3, 2)}}
        # config 2: one token through the same layer (8 experts)
        d1, _ = best_of(lambda: oracle.moe_layer(pool, routers[0], xb[:1], K, threads=1), 0.5)
        dm, _ = best_of(lambda: oracle.moe_layer(pool, routers[0], xb[:1], K, threads=min(threads, K)), 0.5)
        legs["config2_decode"] = {"ms_1_thread": round(d1 * 1e3, 2), f"ms_{min(threads, K)}_threads": round(dm * 1e3, 2),
                                  "GBs_1_thread": round(K * EXPERT_BYTES / d1 / 1e9, 3),
                                  f"GBs_{min(threads, K)}_threads": round(K * EXPERT_BYTES / dm / 1e9, 3),
                                  "note": "8 routes: at most 8 threads have work"}
        # config 1: the [1408 x 2816] GEMV (dequantise the row, then dot), one thread and rows split over the threads
        if config1 is not None:
            W1h, S1h, B1h = config1
            x1f = oracle.bf16_to_float(xb[0])
            g1, _ = best_of(lambda: oracle.gemv_int4_ref(W1h, S1h, B1h, x1f), 0.5, 5)
            cuts = np.linspace(0, W1h.shape[0], threads + 1).astype(int)
            with ThreadPoolExecutor(threads) as ex:
                def split_gemv():
                    list(ex.map(lambda i: oracle.gemv_int4_ref(W1h[cuts[i]:cuts[i + 1]], S1h[cuts[i]:cuts[i + 1]], B1h[cuts[i]:cuts[i + 1]], x1f),
                                range(threads)))
                gm, _ = best_of(split_gemv, 0.5, 5)
            b1 = W1h.size + 2 * S1h.size * 2
            legs["config1_gemv_1408x2816"] = {"us_1_thread": round(g1 * 1e6, 1), f"us_{threads}_threads": round(gm * 1e6, 1),
                                              "GBs_1_thread": round(b1 / g1 / 1e9, 3), f"GBs_{threads}_threads": round(b1 / gm / 1e9, 3)}
        # config 4: a sample of the 3,072-token chunk (the oracle's per-pair FFN is independent per token), extrapolated
        if prefill is not None:
            n_s = 4 * threads
            ps, _ = best_of(lambda: oracle.moe_layer(pool, routers[0], xp_bits[:n_s], K, threads=threads), 2.0, 1)
            legs["config4_prefill"] = {"sample_tokens": n_s, "sample_ms": round(ps * 1e3, 1), f"tok_per_s_{threads}_threads": round(n_s / ps, 1),
                                       "ms_per_layer_extrapolated": round(ps / n_s * prefill["tokens"] * 1e3, 1),
                                       "note": f"first {n_s} of the chunk's {prefill['tokens']} tokens; time scales with the token count"}
        # config 5: the LM head GEMV [262144 x 2816] (dequantise the row, then dot), on a sample of its rows split over
        # the threads, extrapolated to the whole head (the rows are independent)
        if head_sample is not None:
            Wq, Sq, Bq = head_sample
            xh = oracle.bf16_to_float(xb[0])
            cuts_h = np.linspace(0, Wq.shape[0], threads + 1).astype(int)
            with ThreadPoolExecutor(threads) as ex:
                def split_head():
                    list(ex.map(lambda i: oracle.gemv_int4_ref(Wq[cuts_h[i]:cuts_h[i + 1]], Sq[cuts_h[i]:cuts_h[i + 1]],
                                                               Bq[cuts_h[i]:cuts_h[i + 1]], xh), range(threads)))
                hm, _ = best_of(split_head, 1.0, 2)
            hb = Wq.size + 2 * Sq.size * 2
            legs["config5_lm_head_262144x2816"] = {
                "sample_rows": int(Wq.shape[0]), "sample_ms": round(hm * 1e3, 2), f"GBs_{threads}_threads": round(hb / hm / 1e9, 3),
                "ms_per_row_of_x_extrapolated": round(hm * 262144 / Wq.shape[0] * 1e3, 1),
                "note": f"first {Wq.shape[0]} of the head's 262,144 rows, one input row; time scales with the row count"}
        cpu = {"value": round(cpu_bytes / multi / 1e9, 3), "unit": "GB/s", "cores": threads, "kind": "port",
               "nproc": nproc, "cpu_model": cpu_model, "omp_num_threads_env": os.environ.get("OMP_NUM_THREADS"),
               "compiler": cpu_flags,
               "sample": f"config 3: layer 0 of the same 16-token block, best of {reps} reps on {threads} threads "
                         f"({multi * 1e3:.1f} ms); 1 thread: {single * 1e3:.0f} ms = {cpu_bytes / single / 1e9:.3f} GB/s; "
                         f"C restatement of the reference's Swift CPU dequant+matmul path; the other configurations' samples are in legs",
               "legs": legs}
        # the GPU result of layer 0 against that CPU result: the bench measures a correct path
        step(0)
        torch.cuda.synchronize()
        got = oracle.bf16_to_float(y.view(torch.int16).cpu().numpy().view(np.uint16))
        assert np.array_equal(idx.cpu().numpy().astype(np.uint32), ridx), "top-k indices differ from the oracle"
        rel = float(np.abs(got - ry).max() / np.abs(ry).max())
        assert rel <= 1e-2, f"layer output differs from the oracle: rel err {rel}"
        extra["parity_rel_err_layer0"] = round(rel, 5)

    out = {
        "metric": "MoE-layer INT4 weight GB/s (% HBM peak) @16-tok verify; prefill MoE tok/s",
        "value": round(value, 1), "unit": "GB/s", "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 5), "us_per_layer_pass": round(ms_per_step * 1e3 / L, 2), "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"workload": f"config 3: {T}-token DFlash verify block through the MoE layer, hidden {D}, "
                               f"{E} experts x intermediate {F}, top-{K}, INT4 g64; a step takes the block through "
                               f"the {L} resident layers once ({L} layer passes, each streaming its own layer's experts)",
                   "tokens": T, "layers_resident": L, "layer_passes_per_step": L,
                   "settle_layer_passes_before_warmup": kSettlePasses,
                   "distinct_experts_mean": round(float(np.mean(live)), 1),
                   "distinct_experts_min": int(min(live)), "distinct_experts_max": int(max(live)),
                   "expert_bytes_per_step": int(sum(live) * EXPERT_BYTES),
                   "expert_bytes_per_layer_pass_mean": int(np.mean(live) * EXPERT_BYTES),
                   "routes_per_live_expert_hist": {str(n): int(c) for n, c in enumerate(tokens_per_expert) if c},
                   "routes_per_live_expert_note": f"over the {L} layers: how many live experts receive n of the block's {T * K} routes"},
        "pct_hbm_peak": round(100 * value / HBM_PEAK_GBS, 2),
        "stream_ceiling": stream_ceiling,
        "handover_giveups_in_timed_region": giveups,
        "value_first_20_passes_after_5": {"GBs": round(cold_value, 1), "us_per_layer_pass": round(cold_el * 1e6 / 20, 2),
                                          "note": "25 layer passes straight after a pause, no settling passes: a 1 ms timed region "
                                                  "between two synchronisations, which the launch latency in front and the "
                                                  "wake-up behind it weigh on"},
        "layer_pass_us": step_spread,
        "device": device_info,
        "roofline": {"bound": "hbm", "kernel": dominant, "achieved": round(achieved, 1),
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": round(achieved / HBM_PEAK_GBS, 4),
                     "traffic": traffic.get("verify16_route_gate_up" if "route_gate_up" in prof else "verify16_gate_up") if (T == 16 and L == 30) else None,
                     "traffic_unit": f"bytes per launch (rocprofv3 --pmc, profiles/{TRAFFIC_FILE.name})",
                     "algorithmic_bytes_per_launch": int(achieved * 1e9 * gu_ms * 1e-3 / n_timed),
                     "avg_kernel_us": round(gu_ms * 1e3 / n_timed, 2),
                     "measured_ceiling_GBs": round(ceiling_gu, 1), "frac_of_ceiling": round(achieved / ceiling_gu, 4),
                     "ceiling_note": "measured_ceiling_GBs: the same launch's weight loads alone (stream_ceiling.kernel_us.probe_gate_up), this run, this box",
                     "note": ("the launch also holds the routing chain (logits, select, routes: about 6 us before the first weight is "
                              "requested); five_launch_form.gate_up_* is the same stream as a launch of its own") if split else None},
        "five_launch_form": split,
        "kernel_us": kernel_us,
        "down_kernel_GBs": None if down_gbs is None else round(down_gbs, 1),
        "prefill_tok_s": prefill["tok_per_s"] if prefill else None,
        "prefill": prefill,
        "cpu_baseline": cpu,
        "extra": extra,
        "sweep": sweep,
    }
    print(json.dumps(out))
    ctx.close()


if __name__ == "__main__":
    main()
