#!/usr/bin/env python3
"""Benchmark of the ictc_o3 hot path on one MI355X.

Headline (``value``): channelwise CG tensor product forward + VJP (grads to
features, harmonics and gates), C=128, lmax=3 (23 paths), 131,072 instances,
fp32 -- BASELINE.json configs[1].  One "step" = one TP forward + one fused VJP
over the batch; inputs are resident in HBM before the timed region.

Also reported on the same JSON line:
* ``roofline`` of the dominant kernel (the fused VJP kernel): algorithmic bytes
  per launch / its mean duration from HIP events around each launch on the
  launch stream, against the 8 TB/s HBM3E peak;
* ``cpu_baseline``: the CPU oracle (a PyTorch restatement of the reference's CPU
  path, ``_forward_index_add`` + autograd) on a bounded sample on the host cores;
* ``extra``: forward-only throughput at 262,144 instances and its roofline, and the
  other configurations of BASELINE.json, each with its own roofline and a bounded
  CPU-oracle sample:
    - cfg 0, the TP forward at C=64, lmax 2 (11 paths), 65,536 instances (14,116 algorithmic
      bytes per instance), beside the CPU reference path (the oracle's _forward_index_add);
    - cfg 2, graph message (C=64, lmax 2, 16,384 atoms at 0.1 A^-3, r_c 5 A, gates from
      a random-init 8-Bessel radial MLP): fused gather -> TP -> receiver sum forward, and
      its VJP (edge + node kernels);
    - cfg 3, symmetric contraction (C=128, lmax 3 -> 0e+1o, correlation 3, 65,536 nodes,
      10 species): forward and VJP to the node features (VALU-bound: FLOPs counted on the
      generated code as useful FLOPs, and from the committed VALU counters as executed FLOPs,
      against the published fp32 vector peak and the measured rate of a non-packed FMA probe);
    - cfg 4, MACE-style energy + forces (C=128, lmax 3, 2 interactions, correlation 3,
      2,048 atoms at 0.1 A^-3 with 1.5 A minimum separation, r_c 5 A, 10 species):
      inference and one force-loss training step (fused AdamW), atom-steps/s, reference timing
      protocol (>= 2 s and 3 warmup calls, median of 5 synchronised calls), run eager (as
      the reference does) and as HIP-graph replays of the captured steps;
    - the HIP periodic radius graph build for the cfg-2 and cfg-4 structures (outside every
      timed hot-path region).

``--kernels-only`` runs a 1 GiB device-to-device copy (the counter calibration
reference) and three launches of each TP kernel at the benchmark sizes, for
rocprofv3 --pmc passes.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu] [--kernels-only]
                      [--only tp|tp0|message|sc|mace|mace_steps|graph|linear|radial|l4|valu]
"""
from __future__ import annotations

import argparse
import itertools
import json
import math
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "ictc-o3-hp-ascend_amd"))

import torch  # noqa: E402

HBM_PEAK_GBS = 8000.0                       # MI355X HBM3E, GB/s
PUBLISHED_FWD_VJP_INST_S = 0.729e6          # the reference HP path on an Ascend 910B3 (its published figure)
C, L, ROWS_VJP, ROWS_FWD = 128, 3, 131072, 262144
P = 23
X_W, Y_W, G_W, O_W = C * (L + 1) ** 2, (L + 1) ** 2, P * C, 99 * C
BYTES_FWD = 4 * (X_W + Y_W + G_W + O_W)                   # 70,720 B/inst
BYTES_VJP = 4 * (O_W + 2 * (X_W + Y_W + G_W))             # 90,752 B/inst


def _harmonics(n: torch.Tensor) -> torch.Tensor:
    from ictc_o3.backends.hip.harmonics import direction_harmonics_packed
    return direction_harmonics_packed(n, L)


def _inputs(rows: int, device, seed: int = 0):
    gen = torch.Generator(device="cpu").manual_seed(seed)
    x = torch.randn(rows, X_W, generator=gen)
    n = torch.nn.functional.normalize(torch.randn(rows, 3, generator=gen), dim=-1)
    g = torch.randn(rows, G_W, generator=gen) / math.sqrt(P)
    o = torch.randn(rows, O_W, generator=gen)
    x, n, g, o = (t.to(device) for t in (x, n, g, o))
    return x, _harmonics(n).contiguous(), g, o


def _time_gpu(args, plan, device):
    from ictc_o3.backends.hip.tensor_product import _backward_raw, _forward_raw
    x, y, g, o = _inputs(ROWS_VJP, device)
    need = (True, True, True)
    stream = torch.cuda.current_stream(device)

    def step(ev=None):
        out = _forward_raw(plan, x, y, g)
        if ev is not None:
            ev[0].record(stream)
        dx, dy, dg = _backward_raw(plan, need, x, y, g, o)
        if ev is not None:
            ev[1].record(stream)
        return out, dx, dy, dg

    t_end = time.time() + 2.0                 # reference protocol: >= 2 s warmup
    for _ in range(max(args.warmup, 1)):
        step()
    while time.time() < t_end:
        step()
    torch.cuda.synchronize(device)
    events = [(torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True))
              for _ in range(args.steps)]
    torch.cuda.synchronize(device)
    t0 = time.perf_counter()
    for k in range(args.steps):
        step(events[k])
    torch.cuda.synchronize(device)
    elapsed = time.perf_counter() - t0
    vjp_ms = sum(a.elapsed_time(b) for a, b in events) / args.steps
    del x, y, g, o

    # forward-only at 262,144 instances
    x, y, g, _ = _inputs(ROWS_FWD, device, seed=1)
    for _ in range(3):
        _forward_raw(plan, x, y, g)
    torch.cuda.synchronize(device)
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    reps = max(args.steps, 5)
    s.record(stream)
    for _ in range(reps):
        _forward_raw(plan, x, y, g)
    e.record(stream)
    torch.cuda.synchronize(device)
    fwd_ms = s.elapsed_time(e) / reps
    return elapsed, vjp_ms, fwd_ms


def _copy_gbs(device, nbytes: int = 1 << 30, reps: int = 5) -> float:
    """Device-to-device copy bandwidth (read + write bytes / time)."""
    src = torch.empty(nbytes // 4, device=device)
    dst = torch.empty_like(src)
    src.fill_(1.0)
    dst.copy_(src)
    torch.cuda.synchronize(device)
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record()
    for _ in range(reps):
        dst.copy_(src)
    e.record()
    torch.cuda.synchronize(device)
    return 2 * nbytes * reps / (s.elapsed_time(e) * 1e-3) / 1e9


def _stream_mix_gbs(device, reads: int, writes: int, total_bytes: int, reps: int = 5):
    """Best bandwidth of an ideal grid-stride float4 streaming kernel (stream_probe.hip)
    moving total_bytes in the given read:write mix, over three grid sizes and both load cache
    policies (default, non-temporal); None if the probe library is absent."""
    import ctypes
    path = os.path.join(ROOT, "libictc_stream_probe.so")
    if not os.path.exists(path):
        return None
    lib = ctypes.CDLL(path)
    lib.ictc_probe_stream_mix.restype = ctypes.c_int
    lib.ictc_probe_stream_mix.argtypes = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p,
                                          ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_void_p]
    units = total_bytes // (16 * (reads + writes))
    a = torch.ones(reads * units * 4, device=device)
    b = torch.empty(writes * units * 4, device=device)
    stream = torch.cuda.current_stream(device)
    best = 0.0
    for nt, grid in itertools.product((0, 1), (8192, 65536, min((units + 255) // 256, 2 ** 31 - 1))):
        def launch():
            if lib.ictc_probe_stream_mix(reads, writes, nt, a.data_ptr(), b.data_ptr(), units, grid,
                                         ctypes.c_void_p(stream.cuda_stream)) != 0:
                raise RuntimeError("stream probe launch failed")
        for _ in range(2):
            launch()
        s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        s.record(stream)
        for _ in range(reps):
            launch()
        e.record(stream)
        torch.cuda.synchronize(device)
        best = max(best, 16 * (reads + writes) * units * reps / (s.elapsed_time(e) * 1e-3) / 1e9)
    del a, b
    torch.cuda.empty_cache()
    return best


def _kernels_only(plan, device) -> None:
    from ictc_o3.backends.hip.tensor_product import _backward_raw, _forward_raw
    src = torch.ones((1 << 30) // 4, device=device)
    torch.empty_like(src).copy_(src)          # calibration copy: 1 GiB read + 1 GiB written
    torch.cuda.synchronize(device)
    del src
    x, y, g, o = _inputs(ROWS_VJP, device)
    for _ in range(3):
        _forward_raw(plan, x, y, g)
        _backward_raw(plan, (True, True, True), x, y, g, o)
    torch.cuda.synchronize(device)
    print("kernels-only pass done", flush=True)


def _profile_value(name: str, key: str):
    """A `key: value` line of a committed profiles/ summary (None if absent)."""
    try:
        for line in open(os.path.join(ROOT, "profiles", name)):
            if line.startswith(key + ":"):
                return float(line.split(":", 1)[1])
    except OSError:
        pass
    return None


def _measured_traffic():
    """HBM bytes per VJP launch from the committed rocprofv3 FETCH_SIZE/WRITE_SIZE summary
    (calibrated against a 1 GiB copy); None if the summary is absent."""
    path = os.path.join(ROOT, "profiles", "tp_c128_l3_hbm_traffic.md")
    try:
        for line in open(path):
            if line.startswith("traffic_bytes_per_vjp_launch:"):
                return float(line.split(":", 1)[1])
    except OSError:
        pass
    return None


def _cpu_model() -> str:
    """The host CPU's model name (reported beside every CPU baseline)."""
    try:
        for line in open("/proc/cpuinfo"):
            if line.startswith("model name"):
                return line.split(":", 1)[1].strip()
    except OSError:
        pass
    return "unknown"


def _cpu_baseline(budget_s: float = 12.0):
    """Oracle fwd+VJP (reference CPU path restated) on a bounded C128/L3 sample."""
    sys.path.insert(0, ROOT)
    from oracle import ictc_basis as B
    from oracle.tensor_product import TensorProductOracle
    threads = os.cpu_count() or 1
    torch.set_num_threads(threads)
    op = TensorProductOracle(C, L, L, L, dtype=torch.float32)
    rows = 2048
    gen = torch.Generator().manual_seed(0)
    x = torch.randn(rows, X_W, generator=gen)
    n = torch.nn.functional.normalize(torch.randn(rows, 3, generator=gen, dtype=torch.float64), dim=-1)
    y = B.direction_harmonics_packed(n, L).float()
    g = torch.randn(rows, G_W, generator=gen) / math.sqrt(P)
    o = torch.randn(rows, O_W, generator=gen)

    def step():
        leaves = [t.clone().requires_grad_() for t in (x, y, g)]
        torch.autograd.grad(op.forward(*leaves), leaves, o)

    step()
    done, t0 = 0, time.perf_counter()
    while time.perf_counter() - t0 < budget_s:
        step()
        done += 1
    dt = time.perf_counter() - t0
    return {"value": rows * done / dt, "unit": "instances/s", "cores": threads, "cpu_model": _cpu_model(), "kind": "port",
            "sample": f"oracle fwd+VJP (PyTorch CPU fp32, reference _forward_index_add + autograd), "
                      f"C128/lmax3, {rows} instances x {done} steps in {dt:.1f}s"}


VALU_PEAK_TFLOPS = 157.3                    # MI355X fp32 vector (published)


def _median_call_ms(fn, device, *, warmup_s: float = 2.0, warmup_calls: int = 3, calls: int = 5):
    """Reference protocol: >= 2 s and 3 warmup calls, then the median of synchronised calls."""
    t_end = time.time() + warmup_s
    for _ in range(warmup_calls):
        fn()
    while time.time() < t_end:
        fn()
    torch.cuda.synchronize(device)
    times = []
    for _ in range(calls):
        t0 = time.perf_counter()
        fn()
        torch.cuda.synchronize(device)
        times.append((time.perf_counter() - t0) * 1e3)
    return sorted(times)[len(times) // 2]


def _event_ms(fn, device, reps: int = 10, warmup: int = 3, warm_s: float = 0.05) -> float:
    """Mean duration of fn's launches between HIP events on the current stream, after `warmup`
    calls and at least `warm_s` seconds of back-to-back calls (the GPU clocks ramp up over the
    first milliseconds of work: a few warm-up calls alone time a short leg partly at lower
    clocks)."""
    for _ in range(warmup):
        fn()
    torch.cuda.synchronize(device)
    t0 = time.perf_counter()
    while time.perf_counter() - t0 < warm_s:
        for _ in range(4):
            fn()
        torch.cuda.synchronize(device)
    stream = torch.cuda.current_stream(device)
    s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    s.record(stream)
    for _ in range(reps):
        fn()
    e.record(stream)
    torch.cuda.synchronize(device)
    return s.elapsed_time(e) / reps


def _probe_lib():
    import ctypes
    path = os.path.join(ROOT, "libictc_stream_probe.so")
    if not os.path.exists(path):
        return None
    lib = ctypes.CDLL(path)
    lib.ictc_probe_valu_fma.restype = ctypes.c_int
    lib.ictc_probe_valu_fma.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    lib.ictc_probe_valu_form.restype = ctypes.c_int
    lib.ictc_probe_valu_form.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_void_p]
    lib.ictc_probe_valu_chains.restype = ctypes.c_int
    lib.ictc_probe_valu_chains.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_int,
                                           ctypes.c_void_p]
    return lib


VALU_FORMS = ("v_fmac_f32_e32 v,v,v", "v_fmac_f32_e32 v,literal,v", "v_fma_f32 v,v,v,v (VOP3)",
              "v_fmac_f32_e32 v,s,v (SGPR operand)", "v_fmac_f32_e64 v,v,v (VOP3 encoding)", "v_fmac_f32_dpp",
              "v_cndmask_b32_e64 (SGPR-pair mask)", "v_readlane_b32")


def _valu_form_cycles(device, grid: int = 16384, iters: int = 2048, clock_ghz: float = 2.4):
    """Issue cost of VALU instruction forms (stream_probe.hip valu_form_kernel): nanoseconds per
    wave instruction per SIMD at full occupancy, and the same in cycles of the 2.4 GHz peak
    clock; None if the probe library is absent."""
    import ctypes
    lib = _probe_lib()
    if lib is None:
        return None
    out = torch.empty(grid * 256, device=device)
    stream = torch.cuda.current_stream(device)
    simds = torch.cuda.get_device_properties(device).multi_processor_count * 4
    res = {}
    for form, name in enumerate(VALU_FORMS):
        def launch():
            if lib.ictc_probe_valu_form(out.data_ptr(), form, iters, grid, ctypes.c_void_p(stream.cuda_stream)) != 0:
                raise RuntimeError("VALU form probe launch failed")
        ms = _event_ms(launch, device, reps=5, warmup=2)
        wave_insts = grid * 4 * iters * 16
        ns = ms * 1e6 / (wave_insts / simds)
        res[name] = {"ns_per_wave_instruction_per_simd": ns, "cycles_at_2.4GHz": ns * clock_ghz}
    # one wave's issue rate: independent FMA chains at 1, 2 and 4 resident waves per SIMD
    cus, chain_iters = simds // 4, 20000
    out = torch.empty(cus * 4 * 256, device=device)
    chains = {}
    for waves in (1, 2, 4):
        for k in (1, 2, 4, 8):
            def launch():
                if lib.ictc_probe_valu_chains(out.data_ptr(), k, waves, cus, chain_iters,
                                              ctypes.c_void_p(stream.cuda_stream)) != 0:
                    raise RuntimeError("VALU chain probe launch failed")
            ms = _event_ms(launch, device, reps=2, warmup=1)
            cycles = ms * 1e-3 * clock_ghz * 1e9
            chains[f"{waves}_waves_per_simd_{k}_chains"] = {
                "cycles_per_wave_instruction_per_wave": cycles / (chain_iters * 16),
                "cycles_per_wave_instruction_per_simd": cycles / (chain_iters * 16 * waves)}
    res["fma_chains_by_occupancy"] = chains
    return res


def _valu_fma_tflops(device, grid: int = 16384, iters: int = 2048, reps: int = 5):
    """fp32 FMA rate of register-only kernels of scalar (non-packed) fma chains
    (stream_probe.hip) in both instruction forms the compiler emits: v_fma_f32 with SGPR
    operands (VOP3) and v_fmac_f32 with every operand in a VGPR (VOP2); None if the probe
    library is absent."""
    import ctypes
    lib = _probe_lib()
    if lib is None:
        return None
    out = torch.empty(grid * 256, device=device)
    stream = torch.cuda.current_stream(device)
    rates = {}
    for name, vgpr in (("v_fma_f32_sgpr_operands", 0), ("v_fmac_f32_vgpr_operands", 1)):
        def launch():
            if lib.ictc_probe_valu_fma(out.data_ptr(), iters, grid, vgpr, ctypes.c_void_p(stream.cuda_stream)) != 0:
                raise RuntimeError("VALU probe launch failed")
        ms = _event_ms(launch, device, reps=reps, warmup=2)
        rates[name] = 32.0 * iters * grid * 256 / (ms * 1e-3) / 1e12
    return rates


TP0_C, TP0_L, TP0_P, TP0_ROWS = 64, 2, 11, 65536
TP0_X, TP0_Y, TP0_O = TP0_C * (TP0_L + 1) ** 2, (TP0_L + 1) ** 2, 35 * TP0_C
BYTES_TP0 = 4 * (TP0_X + TP0_Y + TP0_P * TP0_C + TP0_O)          # 14,116 B/inst


def _tp0_inputs(rows: int, device):
    """cfg 0: x ~ N(0,1) packed ir_mul [E, 576]; unit directions -> ICTC Y [E, 9]; gates in the
    API layout [E, P, C] ~ N(0,1)/sqrt(P) (the config's w[N,C,P] transposed to the operator's
    path-major order); tp.weight = 1."""
    gen = torch.Generator(device="cpu").manual_seed(0)
    x = torch.randn(rows, TP0_X, generator=gen)
    n = torch.nn.functional.normalize(torch.randn(rows, 3, generator=gen), dim=-1)
    g = torch.randn(rows, TP0_P, TP0_C, generator=gen) / math.sqrt(TP0_P)
    return x, n, g


def _bench_tp_cfg0(device):
    from ictc_o3 import EdgeTensorProduct
    from ictc_o3.backends.hip.harmonics import direction_harmonics_packed
    from ictc_o3.backends.hip.tensor_product import _forward_raw
    op = EdgeTensorProduct.create(channels=TP0_C, input_lmax=TP0_L, edge_lmax=TP0_L, device=device)
    assert op.tp.num_paths == TP0_P and op.output_width == TP0_O
    x, n, g = _tp0_inputs(TP0_ROWS, device)
    x, g = x.to(device), g.to(device).reshape(TP0_ROWS, -1)
    y = direction_harmonics_packed(n.to(device), TP0_L).contiguous()
    ms = _event_ms(lambda: _forward_raw(op.plan, x, y, g), device, reps=20)
    gbs = BYTES_TP0 * TP0_ROWS / (ms * 1e-3) / 1e9
    traffic = _profile_value("tp_c64_l2_cfg0_kernel_trace_and_traffic.md", "traffic_bytes_per_launch")
    return {"workload": "cfg0 channelwise TP forward C64/lmax2 (11 paths), 65,536 instances, ir_mul",
            "kernel": "tp_forward_kernel<2,2,2,1,false>", "mean_launch_ms": ms,
            "instances_per_s": TP0_ROWS / (ms * 1e-3), "vs_published_11.57M": TP0_ROWS / (ms * 1e-3) / 11.57e6,
            "roofline": {"bound": "hbm", "algorithmic_bytes_per_instance": BYTES_TP0,
                         "algorithmic_bytes_per_launch": BYTES_TP0 * TP0_ROWS, "achieved": gbs,
                         "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": gbs / HBM_PEAK_GBS,
                         "traffic": traffic, "traffic_unit": "bytes/launch"}}


GEN_C, GEN_L, GEN_ROWS = 64, 4, 65536


def _tp_degree_leg(device, lin: int, le: int, lout: int):
    """Forward and VJP of the TP at C = 64 over GEN_ROWS instances of degrees (lin, le, lout),
    against both bounds: algorithmic HBM bytes (x, Y, g read and out written; the VJP also reads
    dout and writes dx, dY, dg) and the FMA work the kernels execute (forward 2·NB·C per instance
    plus 2·Σ_p n1 n2 n3 for the bond rows; the VJP 2·2·NB·C for dg and dx, 2·Σ_p n1 n2 n3·C for
    the per-channel dY contraction, and the bond rows)."""
    from ictc_o3 import EdgeTensorProduct
    from ictc_o3.backends.hip.harmonics import direction_harmonics_packed
    from ictc_o3.backends.hip.tensor_product import _backward_raw, _forward_raw
    op = EdgeTensorProduct.create(channels=GEN_C, input_lmax=lin, edge_lmax=le, output_lmax=lout, device=device)
    plan = op.plan
    gen = torch.Generator(device=device).manual_seed(5)
    x = torch.randn(GEN_ROWS, plan.x_width, device=device, generator=gen)
    n = torch.nn.functional.normalize(torch.randn(GEN_ROWS, 3, device=device, generator=gen), dim=-1)
    y = direction_harmonics_packed(n, le).contiguous()
    g = torch.randn(GEN_ROWS, plan.full_gate_width, device=device, generator=gen)
    go = torch.randn(GEN_ROWS, plan.full_out_width, device=device, generator=gen)
    fwd_ms = _event_ms(lambda: _forward_raw(plan, x, y, g), device, reps=10)
    vjp_ms = _event_ms(lambda: _backward_raw(plan, (True, True, True), x, y, g, go), device, reps=10)
    paths = plan.full_paths
    nb = sum((2 * a + 1) * (2 * c + 1) for a, _, c in paths)
    dense = sum((2 * a + 1) * (2 * b + 1) * (2 * c + 1) for a, b, c in paths)
    xw, yw, gw, ow = plan.x_width, plan.y_width, plan.full_gate_width, plan.full_out_width
    fwd_bytes, vjp_bytes = 4 * (xw + yw + gw + ow), 4 * (ow + 2 * (xw + yw + gw))
    fwd_flops = 2 * nb * GEN_C + 2 * dense
    vjp_flops = 2 * 2 * nb * GEN_C + 2 * dense * GEN_C + 2 * dense

    def leg(ms, nbytes, flops):
        gbs = nbytes * GEN_ROWS / (ms * 1e-3) / 1e9
        tf = flops * GEN_ROWS / (ms * 1e-3) / 1e12
        return {"mean_launch_ms": ms, "instances_per_s": GEN_ROWS / (ms * 1e-3),
                "hbm": {"algorithmic_bytes_per_instance": nbytes, "achieved": gbs, "peak": HBM_PEAK_GBS,
                        "unit": "GB/s", "frac": gbs / HBM_PEAK_GBS},
                "valu": {"fma_flops_per_instance": flops, "achieved": tf, "peak": VALU_PEAK_TFLOPS,
                         "unit": "TFLOP/s", "frac": tf / VALU_PEAK_TFLOPS}}

    return {"workload": f"TP C{GEN_C}, degrees ({lin},{le},{lout}), {len(paths)} paths, {GEN_ROWS:,} instances, "
                        f"ir_mul",
            "forward": leg(fwd_ms, fwd_bytes, fwd_flops), "vjp": leg(vjp_ms, vjp_bytes, vjp_flops)}


def _bench_tp_l4(device):
    """Degree-4 tensor products: the symmetric (4, 4, 4) set (42 paths) on its compiled kernels,
    and the (4, 4, 3) set on the degree-generic ones (run-time path tables: every set with a degree
    above 3 other than the compiled ones)."""
    out = _tp_degree_leg(device, GEN_L, GEN_L, GEN_L)
    out["kernels"] = "tp_forward_kernel<4,4,4,1,false>, tp_backward_wide_kernel<4,4,4,false>"
    gen = _tp_degree_leg(device, GEN_L, GEN_L, GEN_L - 1)
    gen["kernels"] = "gen_tp_forward_kernel, gen_tp_backward_kernel"
    out["generic_443"] = gen
    return out


def _cpu_tp_cfg0(budget_s: float = 10.0, rows: int = 8192):
    """cfg 0 on the CPU reference path: the oracle's _forward_index_add restatement, fp32, all host
    threads, on the first `rows` instances of the same seeded inputs."""
    sys.path.insert(0, ROOT)
    from oracle import ictc_basis as B
    from oracle.tensor_product import TensorProductOracle
    threads = os.cpu_count() or 1
    torch.set_num_threads(threads)
    op = TensorProductOracle(TP0_C, TP0_L, TP0_L, TP0_L, dtype=torch.float32)
    x, n, g = _tp0_inputs(TP0_ROWS, "cpu")
    x, n, g = x[:rows], n[:rows], g[:rows].reshape(rows, -1)
    y = B.direction_harmonics_packed(n.double(), TP0_L).float()
    with torch.no_grad():
        done, dt = _cpu_time(lambda: op.forward(x, y, g), budget_s)
    return {"value": rows * done / dt, "unit": "instances/s", "cores": threads, "cpu_model": _cpu_model(),
            "kind": "port", "sample": f"oracle TP forward (reference _forward_index_add restated, PyTorch CPU "
                                      f"fp32), C64/lmax2, {rows} of the 65,536 instances x {done} calls in {dt:.1f}s"}


MSG_C, MSG_L, MSG_P, MSG_ATOMS = 64, 2, 11, 16384


def _message_inputs(device):
    """cfg 2 structure, features, harmonics and radial-MLP gates (all resident on the GPU)."""
    from mace_hip.radial import bessel_embedding
    from mace_hip import radius_graph_pbc_gpu, uniform_box
    st = uniform_box(MSG_ATOMS, 0.1, seed=4)
    pos, cell = st.positions.to(device), st.cell.to(device)
    src, dst, shifts = radius_graph_pbc_gpu(pos, 5.0, cell)
    vec = pos[dst] - pos[src] + shifts.to(pos.dtype) @ cell
    r = vec.norm(dim=1)
    from ictc_o3.backends.hip.harmonics import direction_harmonics_packed
    y = direction_harmonics_packed((vec / r[:, None]).contiguous(), MSG_L).contiguous()
    gen = torch.Generator(device="cpu").manual_seed(0)
    x = torch.randn(MSG_ATOMS, MSG_C * (MSG_L + 1) ** 2, generator=gen).to(device)
    gen_w = torch.Generator(device="cpu").manual_seed(2)
    w = [torch.randn(o, i, generator=gen_w) / math.sqrt(i) for i, o in ((8, 64), (64, 64), (64, MSG_P * MSG_C))]
    with torch.no_grad():
        h = bessel_embedding(r, r_max=5.0, num_basis=8, cutoff_p=5)
        for k, wk in enumerate(w):
            h = h @ wk.to(device).t()
            if k < len(w) - 1:
                h = torch.nn.functional.silu(h) * 1.6791767923989418
    go = torch.randn(MSG_ATOMS, 35 * MSG_C, generator=gen).to(device)
    return src, dst, x, y, h.contiguous(), go


def _message_traffic():
    """HBM bytes per dispatch of the cfg-2 message kernels from the committed rocprofv3
    FETCH_SIZE/WRITE_SIZE summary (2.0 x FETCH + 1.0 x WRITE, calibrated on a 1 GiB copy):
    (forward, VJP passes summed), or None if the summary is absent."""
    path = os.path.join(ROOT, "profiles", "msg_c64_l2_cfg2_kernel_trace_and_traffic.md")
    found = {}
    try:
        for line in open(path):
            if line.startswith("| `ictc::msg_") and line.rstrip().endswith("GB |"):
                cells = [c.strip() for c in line.strip().strip("|").split("|")]
                found[cells[0].strip("`")] = float(cells[-1].split()[0]) * 1e9
    except OSError:
        return None
    fwd = [v for k, v in found.items() if k.startswith("ictc::msg_forward_kernel")]
    vjp = [v for k, v in found.items() if not k.startswith("ictc::msg_forward_kernel")]
    if len(fwd) != 1 or len(vjp) < 2:
        return None
    return fwd[0], sum(vjp)


def _bench_message(device):
    from ictc_o3 import EdgeTensorProduct
    from ictc_o3.backends.hip.graph_message import _backward_raw, _forward_raw, message_graph
    op = EdgeTensorProduct.create(channels=MSG_C, input_lmax=MSG_L, edge_lmax=MSG_L, device=device)
    plan = op.plan
    src, dst, x, y, g, go = _message_inputs(device)
    edges = src.numel()
    graph = message_graph(src, dst, MSG_ATOMS, MSG_ATOMS)
    fwd_ms = _event_ms(lambda: _forward_raw(plan, graph, x, y, g), device)
    need = (True, True, True)
    bwd_ms = _event_ms(lambda: _backward_raw(plan, graph, need, x, y, g, go), device)
    # unique-byte model: per edge Y, gates, src index; per node x read once, out written once
    fwd_bytes = edges * (4 * (9 + MSG_P * MSG_C) + 8) + MSG_ATOMS * 4 * (576 + 35 * MSG_C)
    # VJP: per edge Y, gates, index read + dY, dgates written; per node x, go, dx
    bwd_bytes = edges * (4 * 2 * (9 + MSG_P * MSG_C) + 8) + MSG_ATOMS * 4 * (2 * 576 + 35 * MSG_C)
    fwd_gbs, bwd_gbs = fwd_bytes / (fwd_ms * 1e-3) / 1e9, bwd_bytes / (bwd_ms * 1e-3) / 1e9
    traffic = _message_traffic()     # measured HBM bytes per call (L2-miss gathers, bond/dxe rows included)
    real = {} if traffic is None else {
        "forward": {"traffic_bytes": traffic[0], "traffic_gbs": traffic[0] / (fwd_ms * 1e-3) / 1e9},
        "vjp": {"traffic_bytes": traffic[1], "traffic_gbs": traffic[1] / (bwd_ms * 1e-3) / 1e9}}
    return {"workload": "cfg2 graph message C64/lmax2, 16,384 atoms, r_c 5 A", "edges": edges,
            "edges_per_atom": edges / MSG_ATOMS,
            "forward": {"mean_ms": fwd_ms, "edges_per_s": edges / (fwd_ms * 1e-3),
                        "algorithmic_bytes": fwd_bytes, "achieved_gbs": fwd_gbs,
                        "frac": fwd_gbs / HBM_PEAK_GBS, "kernel": "msg_forward_kernel<2,2,2> (in-kernel bond rows)",
                        **real.get("forward", {})},
            "vjp": {"mean_ms": bwd_ms, "edges_per_s": edges / (bwd_ms * 1e-3), "algorithmic_bytes": bwd_bytes,
                    "achieved_gbs": bwd_gbs, "frac": bwd_gbs / HBM_PEAK_GBS,
                    "kernels": "msg_edge_grad_degree_kernel (dg, dY and dxe; one launch per input degree) + "
                               "msg_node_grad_kernel",
                    **real.get("vjp", {})}}


def _bench_message3(device):
    """The MACE layer-1 message at lmax 3 on the cfg-4 graph (C = 128, 2,048 atoms): forward, VJP,
    and the tangent forward and tangent VJP of the force-loss double backward, each one call of
    the raw launchers on HBM-resident inputs.  Unique-byte models: per edge the harmonics, gates
    and source index read once and the per-edge outputs (dg, dY) written once; per node the
    features and cotangent read once and the node outputs written once; the tangent passes also
    read the tangent harmonics, gates and features.  Bond rows and x[src] gathers beyond the
    first are design traffic outside the models."""
    from ictc_o3 import EdgeTensorProduct
    from ictc_o3.backends.hip.graph_message import _backward_raw, _bonds, _forward_raw, _second_order_raw, message_graph
    c, l = 128, 3
    op = EdgeTensorProduct.create(channels=c, input_lmax=l, edge_lmax=l, device=device)
    plan = op.plan
    _, graph_in = _mace_graph(device)
    src, dst = graph_in["edge_src"], graph_in["edge_dst"]
    n, e = MACE_ATOMS, src.numel()
    pos = graph_in["positions"]
    vec = pos[dst] - pos[src] + graph_in["edge_shifts"].to(pos.dtype) @ graph_in["cell"][0]
    from ictc_o3.backends.hip.harmonics import direction_harmonics_packed
    y = direction_harmonics_packed((vec / vec.norm(dim=1, keepdim=True)).contiguous(), l).contiguous()
    gen = torch.Generator(device="cpu").manual_seed(3)
    nx, ny, ng, no = 16 * c, 16, 23 * c, 99 * c
    x, tx = (torch.randn(n, nx, generator=gen).to(device) for _ in range(2))
    g, tg = (torch.randn(e, ng, generator=gen).to(device) / math.sqrt(23) for _ in range(2))
    ty = torch.randn(e, ny, generator=gen).to(device)
    go = torch.randn(n, no, generator=gen).to(device)
    graph = message_graph(src, dst, n, n)
    bonds = _bonds(plan, graph, y)
    need3, need4 = (True, True, True), (True, True, True, True)
    calls = {
        "forward": (lambda: _forward_raw(plan, graph, x, y, g, bonds),
                    e * (4 * (ny + ng) + 8) + n * 4 * (nx + no)),
        "vjp": (lambda: _backward_raw(plan, graph, need3, x, y, g, go),
                e * (4 * 2 * (ny + ng) + 8) + n * 4 * (2 * nx + no)),
        "tangent_forward": (lambda: _second_order_raw(plan, graph, (False, False, False, True), x, y, g, go, tx, ty,
                                                      tg, bonds),
                            e * (4 * 2 * (ny + ng) + 8) + n * 4 * (2 * nx + no)),
        "tangent_vjp": (lambda: _second_order_raw(plan, graph, (True, True, True, False), x, y, g, go, tx, ty, tg,
                                                  bonds),
                        e * (4 * (2 * (ny + ng) + ny + ng) + 8) + n * 4 * (3 * nx + no)),
    }
    out = {"workload": "cfg4 graph, MACE layer-1 message C128/lmax3, 2,048 atoms, r_c 5 A", "edges": e}
    for name, (fn, nbytes) in calls.items():
        ms = _event_ms(fn, device)
        gbs = nbytes / (ms * 1e-3) / 1e9
        out[name] = {"mean_ms": ms, "algorithmic_bytes": nbytes, "achieved_gbs": gbs, "frac": gbs / HBM_PEAK_GBS}
    return out


SC_C, SC_L, SC_T, SC_K, SC_NODES, SC_S = 128, 3, 1, 3, 65536, 10


def _sc_inputs(device, nodes=SC_NODES):
    gen = torch.Generator(device="cpu").manual_seed(0)
    x = torch.randn(nodes, SC_C * (SC_L + 1) ** 2, generator=gen)
    species = torch.randint(0, SC_S, (nodes,), generator=torch.Generator().manual_seed(5))
    go = torch.randn(nodes, SC_C * (SC_T + 1) ** 2, generator=torch.Generator().manual_seed(3))
    return x.to(device), species.to(device), go.to(device)


def _bench_sc(device):
    import sc_flops
    from ictc_o3.backends.hip.symmetric_contraction import ContractionPlan, _forward_raw, _vjp_raw
    plan = ContractionPlan(SC_L, SC_T, SC_K, SC_C, SC_S)
    x, species, go = _sc_inputs(device)
    # per-element weights ~ N(0,1)/sqrt(n_paths) per (degree, order) block (BASELINE.json cfg 3)
    gen = torch.Generator(device="cpu").manual_seed(6)
    from ictc_o3.basis.symmetric_u import chains
    blocks = []
    for lo in range(SC_T + 1):
        for nu in range(SC_K, 0, -1):
            k = len(chains(SC_L, lo, nu))
            blocks.append(torch.randn(SC_S, k, SC_C, generator=gen) / math.sqrt(k))
    w = torch.cat(blocks, 1).to(device).contiguous()
    fwd_ms = _event_ms(lambda: _forward_raw(plan, x, species, w), device)
    vjp_ms = _event_ms(lambda: _vjp_raw(plan, x, species, w, go), device)
    flops = sc_flops.flop_counts(SC_L, SC_T, SC_K)        # useful FLOPs per (node, channel)
    executed = _sc_executed_flops()                        # per lane, from the committed VALU counters
    probe = _valu_fma_tflops(device)
    d, o = (SC_L + 1) ** 2, (SC_T + 1) ** 2
    fwd_bytes = SC_NODES * (4 * SC_C * (d + o) + 8)
    vjp_bytes = SC_NODES * (4 * SC_C * (o + 2 * d) + 8)

    def leg(ms, nbytes, nflops, kernel, mode):
        lanes = SC_C * SC_NODES
        tflops = nflops * lanes / (ms * 1e-3) / 1e12
        gbs = nbytes / (ms * 1e-3) / 1e9
        out = {"mean_ms": ms, "nodes_per_s": SC_NODES / (ms * 1e-3), "kernel": kernel,
               "bound": "valu", "useful_flops_per_node": nflops * SC_C, "achieved_tflops": tflops,
               "peak_tflops": VALU_PEAK_TFLOPS, "frac": tflops / VALU_PEAK_TFLOPS,
               "algorithmic_bytes": nbytes, "achieved_gbs": gbs, "hbm_frac": gbs / HBM_PEAK_GBS}
        if probe:
            out["frac_of_measured_fma_rate"] = tflops / max(probe.values())
        if executed and mode in executed:
            ex = executed[mode] * lanes / (ms * 1e-3) / 1e12
            out.update({"executed_flops_per_node": executed[mode] * SC_C, "executed_tflops": ex,
                        "executed_frac": ex / VALU_PEAK_TFLOPS})
        return out
    return {"workload": "cfg3 symmetric contraction C128, lmax 3 -> 0e+1o, correlation 3, 65,536 nodes",
            "weight_columns": plan.ktot, "measured_valu_fma_tflops": probe,
            "forward": leg(fwd_ms, fwd_bytes, flops["forward"], "sc_kernel<3,1,3,0>", "forward"),
            "vjp": leg(vjp_ms, vjp_bytes, flops["vjp"], "sc_kernel<3,1,3,1>", "vjp")}


def _sc_executed_flops():
    """Executed fp32 FLOPs per (node, channel) lane of the cfg-3 contraction kernels from the
    committed rocprofv3 VALU-counter summary (64 lanes x (2 FMA + MUL + ADD) per wave
    instruction, divided by the lanes); None if the summary is absent."""
    path = os.path.join(ROOT, "profiles", "sc_c128_l3_cfg3_valu_counters.md")
    out = {}
    try:
        for line in open(path):
            if line.startswith("executed_flops_per_lane_"):
                key, value = line.split(":", 1)
                out[key[len("executed_flops_per_lane_"):]] = float(value)
    except OSError:
        return None
    return out or None


MACE_ATOMS, MACE_ZS, MACE_CPU_ATOMS = 2048, tuple(range(1, 11)), 128


def _mace_graph(device, atoms=MACE_ATOMS):
    from mace_hip import radius_graph, radius_graph_pbc_gpu, sequential_insertion
    st = sequential_insertion(atoms, 0.1, min_separation=1.5, num_species=10, seed=4)
    pos, cell = st.positions.to(device), st.cell.to(device)
    if pos.device.type == "cuda":
        src, dst, shifts = radius_graph_pbc_gpu(pos, 5.0, cell)
        shifts = shifts.to(pos.dtype)
    else:                                  # the CPU-oracle sample builds its graph on the host
        src, dst, shifts = radius_graph(pos, cell, 5.0)
    return st, dict(positions=pos, atomic_numbers=torch.tensor(MACE_ZS, device=device)[st.species.to(device)],
                    batch=torch.zeros(atoms, dtype=torch.int64, device=device), edge_src=src, edge_dst=dst,
                    edge_shifts=shifts, cell=cell[None])


def _bench_mace(device):
    """Eager steps (the reference's execution mode) and the same steps captured into HIP graphs
    and replayed on the same inputs (positions re-copied into the graph's buffer every call)."""
    from mace_hip import (CapturedEnergyAndForces, CapturedTrainingStep, create_model, energy_and_forces,
                          training_step)
    _, graph = _mace_graph(device)

    def fresh():
        model = create_model(channels=128, lmax=3, num_interactions=2, correlation=3, atomic_numbers=MACE_ZS,
                             cutoff=5.0, device=device, seed=0)
        return model, model.species_index(graph["atomic_numbers"])
    model, species = fresh()
    opt = torch.optim.AdamW(model.parameters(), lr=1e-3, fused=True)     # one kernel per update, same AdamW
    train_ms = _median_call_ms(lambda: training_step(model, opt, graph, species=species), device)
    model.eval().requires_grad_(False)
    infer_ms = _median_call_ms(lambda: energy_and_forces(model, **graph, species=species), device)
    infer_peak = _peak_bytes(lambda: energy_and_forces(model, **graph, species=species), device)
    streaming = {}
    for size in (16384, 24576):                # radial streaming: no [E, P*C] gate tensor
        model.set_message_streaming(size)
        eager_ms = _median_call_ms(lambda: energy_and_forces(model, **graph, species=species), device)
        peak = _peak_bytes(lambda: energy_and_forces(model, **graph, species=species), device)
        captured = CapturedEnergyAndForces(model, **graph, species=species)
        streaming[size] = (eager_ms, _median_call_ms(lambda: captured(graph["positions"]), device), peak)
        del captured
    model.set_message_streaming(None)
    captured = CapturedEnergyAndForces(model, **graph, species=species)
    infer_graph_ms = _median_call_ms(lambda: captured(graph["positions"]), device)
    del captured
    model, species = fresh()
    opt = torch.optim.AdamW(model.parameters(), lr=1e-3, capturable=True, fused=True)
    step = CapturedTrainingStep(model, opt, graph, species=species)
    train_graph_ms = _median_call_ms(lambda: step(graph["positions"]), device)
    del step

    def leg(ms, published, mode):
        rate = MACE_ATOMS / (ms * 1e-3)
        return {"median_ms": ms, "atom_steps_per_s": rate, f"vs_published_{published / 1e3:.2f}k": rate / published,
                "execution": mode}
    floor = {}
    for name, train, ms in (("inference", False, infer_graph_ms), ("training", True, train_graph_ms)):
        f = _mace_floor(graph["edge_src"].numel(), MACE_ATOMS, train)
        floor[name] = {**f, "replay_ms": ms, "frac": f["t_min_ms"] / ms}
    return {"workload": "cfg4 MACE C128/lmax3, 2 interactions, correlation 3, 2,048 atoms, r_c 5 A",
            "edges": graph["edge_src"].numel(),
            "step_roofline": {"what": "sum of the modelled work at its own roofline (unique bytes at 8 TB/s, "
                                      "useful FLOPs at 157.3 TFLOP/s, split-bf16 products at 417) over the HIP-graph "
                                      "replay time",
                              **floor},
            "inference": leg(infer_ms, 11.0e3, "eager"),
            "training": leg(train_ms, 3.81e3, "eager"),
            "inference_hip_graph": leg(infer_graph_ms, 11.0e3, "HIP graph replay"),
            "training_hip_graph": leg(train_graph_ms, 3.81e3, "HIP graph replay"),
            "inference_radial_streaming": {
                **leg(streaming[16384][0], 11.0e3, "eager, radial streaming over 16,384-edge receiver ranges"),
                "peak_bytes": streaming[16384][2], "peak_bytes_whole_gates": infer_peak,
                "gate_tensor_bytes": graph["edge_src"].numel() * 23 * 128 * 4,
                "ratio_to_whole_gates_eager": streaming[16384][0] / infer_ms,
                "ranges": {str(size): {"eager_ms": e, "replay_ms": r, "peak_bytes": pk,
                                       "ratio_eager": e / infer_ms, "ratio_replay": r / infer_graph_ms}
                           for size, (e, r, pk) in streaming.items()}}}


def _bench_mace_steps(device, modes=("inference", "training"), replays: int = 20):
    """The captured inference and/or training step alone, replayed a fixed number of times after
    its capture (3 eager warm-up calls inside the capture helper, then 3 replays): a kernel trace
    of a one-mode run divides into per-step figures (calls / (replays + 6))."""
    from mace_hip import CapturedEnergyAndForces, CapturedTrainingStep, create_model
    _, graph = _mace_graph(device)
    out = {"replays_after_warmup": replays, "executions_per_mode": replays + 6}
    for mode in modes:
        model = create_model(channels=128, lmax=3, num_interactions=2, correlation=3, atomic_numbers=MACE_ZS,
                             cutoff=5.0, device=device, seed=0)
        species = model.species_index(graph["atomic_numbers"])
        if mode == "inference":
            model.eval().requires_grad_(False)
            step = CapturedEnergyAndForces(model, **graph, species=species)
        else:
            opt = torch.optim.AdamW(model.parameters(), lr=1e-3, capturable=True, fused=True)
            step = CapturedTrainingStep(model, opt, graph, species=species)
        for _ in range(3):
            step(graph["positions"])
        torch.cuda.synchronize(device)
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(replays):
            step(graph["positions"])
        end.record()
        torch.cuda.synchronize(device)
        out[mode] = {"mean_replay_ms": start.elapsed_time(end) / replays}
        del step
    return out


LIN_COUNTS, LIN_C = (4, 6, 7, 6), 128
MFMA_F32_PEAK_TFLOPS = 157.3                    # fp32 MFMA, dense (published)
MFMA_SPLIT_PEAK_TFLOPS = 2500.0 / 6             # fp32 product as six bf16 part products (bf16 MFMA, dense, published)


def _bench_linear(device):
    """The second interaction's message linear of the cfg-4 MACE step (per degree 4 / 6 / 7 / 6
    path blocks of C = 128 channels into 128, 2,048 atoms, alpha = 1/avg_num_neighbors) on the
    split-bf16 MFMA kernels, forward, input adjoint and weight adjoint, beside the dense-GEMM
    routes they replaced (per-degree rearranged copies, library products, concatenation)."""
    from ictc_o3.backends.hip.degree_linear import DegreeLinearPlan, _forward_raw, _input_grad_raw, _weight_grad_raw
    from ictc_o3.backends.hip.linear import mm
    n, c, alpha = MACE_ATOMS, LIN_C, 1.0 / 50.0
    plan = DegreeLinearPlan(LIN_COUNTS, c, c)
    gen = torch.Generator().manual_seed(0)
    x = torch.randn(n, plan.in_width, generator=gen).to(device)
    gy = torch.randn(n, plan.out_width, generator=gen).to(device)
    ws = [(torch.randn(c, k * c, generator=gen) / math.sqrt(k * c)).to(device) for k in LIN_COUNTS]

    def dense_forward():
        return torch.cat([mm(plan.x_rows(x, l), ws[l].t()).reshape(n, 2 * l + 1, c).transpose(1, 2)
                          .reshape(n, -1) for l in range(len(LIN_COUNTS))], 1) * alpha

    def dense_input_grad():
        return torch.cat([mm(plan.y_rows(gy, l), ws[l]).reshape(n, 2 * l + 1, k, c).transpose(1, 2)
                          .reshape(n, -1) for l, k in enumerate(LIN_COUNTS)], 1) * alpha

    def dense_weight_grad():   # the rearranged-rows route: copies of both operands, one product per degree
        return [mm(plan.y_rows(gy, l).t(), plan.x_rows(x, l)) * alpha for l in range(len(LIN_COUNTS))]
    need = [True] * len(LIN_COUNTS)
    # 30 warm-up launches (about 3 ms of work) first: the clocks ramp up over the first launches
    fwd_ms = _event_ms(lambda: _forward_raw(plan, x, ws, alpha), device, reps=100, warmup=30)
    grad_ms = _event_ms(lambda: _input_grad_raw(plan, gy, ws, alpha), device, reps=100, warmup=30)
    wgrad_ms = _event_ms(lambda: _weight_grad_raw(plan, 0, gy, x, alpha, need), device, reps=100, warmup=30)
    dense = (_event_ms(dense_forward, device, reps=20), _event_ms(dense_input_grad, device, reps=20),
             _event_ms(dense_weight_grad, device, reps=20))
    flops = 2 * n * c * sum((2 * l + 1) * k * c for l, k in enumerate(LIN_COUNTS))
    nbytes = 4 * (n * (plan.in_width + plan.out_width) + sum(w.numel() for w in ws))

    def leg(ms, dense_ms, kernel):
        tf = flops / (ms * 1e-3) / 1e12
        return {"kernel": kernel, "mean_launch_ms": ms, "dense_gemm_route_ms": dense_ms,
                "roofline": {"bound": "mfma", "achieved": tf, "peak": MFMA_SPLIT_PEAK_TFLOPS, "unit": "TFLOP/s",
                             "frac": tf / MFMA_SPLIT_PEAK_TFLOPS, "flops_per_launch": flops},
                "algorithmic_bytes": nbytes, "hbm_frac": nbytes / (ms * 1e-3) / 1e9 / HBM_PEAK_GBS}
    return {"workload": "cfg4 MACE message linear (interaction 2): per-degree path blocks 4/6/7/6 x C128 -> C128, "
                        "2,048 atoms, fp32",
            "forward": leg(fwd_ms, dense[0], "degree_linear_split_kernel<0, 128>"),
            "input_grad": leg(grad_ms, dense[1], "degree_linear_input_grad_kernel<8>"),
            "weight_grad": leg(wgrad_ms, dense[2], "degree_linear_wgrad_kernel<0> + degree_linear_wgrad_sum_kernel")}


RADIAL_EDGES = 105_634     # edges of the cfg-4 MACE graph (2,048 atoms, r_c 5 A)


def _bench_radial(device):
    """The interaction's radial MLP up to its last Linear (8 Bessel features -> 64 -> 64 -> 64,
    normalised SiLU) at the cfg-4 edge count, per derivative mode on the MFMA kernel
    (ictc_hip_radial_mlp), beside the composed route it replaced (one GEMM per layer and
    direction plus the elementwise activation passes, under autograd)."""
    from mace_hip.radial_mlp import VALUE, VJP, VJP_VJP, _launch, hidden_formula
    e, b, s = RADIAL_EDGES, 8, 1.6791767923989418
    gen = torch.Generator().manual_seed(0)
    f = torch.randn(e, b, generator=gen).to(device)
    w1 = (torch.randn(64, b, generator=gen) / math.sqrt(b)).to(device)
    w2 = (torch.randn(64, 64, generator=gen) / 8).to(device)
    w3 = (torch.randn(64, 64, generator=gen) / 8).to(device)
    gh = torch.randn(e, 64, generator=gen).to(device)
    u = torch.randn(e, b, generator=gen).to(device)
    fwd, adj, wg = b * 64 + 2 * 64 * 64, 2 * 64 * 64 + 64 * b, b * 64 + 2 * 64 * 64
    modes = {   # (call, useful FLOPs per edge, kernel)
        "value": (lambda: _launch(VALUE, f, w1, w2, w3, s, hidden=True), 2 * fwd,
                  "radial_mlp_kernel<0, false>"),
        "vjp_features": (lambda: _launch(VJP, f, w1, w2, w3, s, gh, grad_feats=True), 2 * (fwd + adj),
                         "radial_mlp_kernel<1, false>"),
        "vjp_weights": (lambda: _launch(VJP, f, w1, w2, w3, s, gh, grad_weights=(True, True, True)),
                        2 * (fwd + adj - 64 * b + wg), "radial_mlp_kernel<1, true> + radial_wsum_kernel"),
        "vjp_vjp": (lambda: _launch(VJP_VJP, f, w1, w2, w3, s, gh, u, grad_grad=True,
                                    grad_weights=(True, True, True)),
                    2 * (2 * fwd + 2 * (adj - 64 * b) + 2 * wg), "radial_mlp_kernel<2, true> + radial_wsum_kernel"),
    }
    fr, w1r, w2r, w3r = (t.clone().requires_grad_() for t in (f, w1, w2, w3))

    def composed(mode):
        h = hidden_formula(fr, w1r, w2r, w3r, s)
        if mode == "value":
            return h
        if mode == "vjp_features":
            return torch.autograd.grad(h, fr, gh)
        if mode == "vjp_weights":
            return torch.autograd.grad(h, (w1r, w2r, w3r), gh)
        ghr = gh.clone().requires_grad_()
        gf, = torch.autograd.grad(h, fr, ghr, create_graph=True)
        return torch.autograd.grad(gf, (w1r, w2r, w3r, ghr), u)
    out = {"workload": f"cfg4 MACE radial MLP hidden layers: {e:,} edges, 8 -> 64 -> 64 -> 64, fp32"}
    for name, (fn, per_edge, kernel) in modes.items():
        ms = _event_ms(fn, device, reps=50, warmup=10)
        comp = _event_ms(lambda: composed(name), device, reps=10)
        tf = per_edge * e / (ms * 1e-3) / 1e12
        out[name] = {"kernel": kernel, "mean_launch_ms": ms, "composed_route_ms": comp,
                     "roofline": {"bound": "mfma", "achieved": tf, "peak": MFMA_F32_PEAK_TFLOPS, "unit": "TFLOP/s",
                                  "frac": tf / MFMA_F32_PEAK_TFLOPS, "flops_per_launch": per_edge * e}}
    return out


def _mace_floor(edges: int, atoms: int, training: bool):
    """Lower bound on the device time of one cfg-4 step: each modelled piece of work at its own
    roofline (unique bytes at 8 TB/s for the HBM-bound message kernels, useful FLOPs at
    157.3 TFLOP/s for the fp32 GEMMs, the radial hidden layers and the VALU contraction, at 417 for
    the split-bf16 products: the radial network's last layer and the message linear), summed; the
    elementwise glue and the design traffic (bond rows, dxe, gathers beyond the first) count zero.
    Per interaction (input degree 0 then 3; 4 / 23 paths, 16 / 99 message output rows):
    inference = forward + force backward (message VJP, radial-MLP and linear input adjoints, the
    contraction's VJP); training adds the loss backward: the energy path's message VJP, the force
    path's tangent forward and tangent VJP, four more GEMMs per radial layer (the weight gradient
    and the two adjoints of each force-pass product), four more message-linear and channel-linear
    products and twice more contraction work (VJP and its directional derivative)."""
    import sc_flops
    e, n, c, s = edges, atoms, 128, 10
    terms = {}

    def add(name, nbytes=0.0, flops=0.0, peak=MFMA_F32_PEAK_TFLOPS):
        terms[name] = terms.get(name, 0.0) + max(nbytes / (HBM_PEAK_GBS * 1e9), flops / (peak * 1e12)) * 1e3
    for lin, npath, noc, target in ((0, 4, 16, 3), (3, 23, 99, 0)):
        nx = (lin + 1) ** 2
        hidden = 2 * e * (8 * 64 + 2 * 64 * 64)                          # radial MLP forward
        last = 2 * e * 64 * npath * c                                     # its last layer: the gates
        fwd_b = e * (4 * npath * c + 64 + 8) + n * 4 * c * (nx + noc)
        vjp_b = e * (8 * npath * c + 64 + 64 + 8) + n * 4 * c * (2 * nx + noc)
        lin_f = 2 * n * c * c * noc                                       # message linear
        chan_f = 2 * n * c * c * (nx + (target + 1) ** 2 + s)             # linear_up, product, self
        sc = sc_flops.flop_counts(3, target, 3)
        sc_f = (sc["forward"] + sc["vjp"]) * n * c
        add("message kernels", nbytes=fwd_b + vjp_b)
        add("radial MLP", flops=2 * hidden)
        add("radial MLP", flops=2 * last, peak=MFMA_SPLIT_PEAK_TFLOPS)
        add("message linear", flops=2 * lin_f, peak=MFMA_SPLIT_PEAK_TFLOPS)
        add("channel linears", flops=2 * chan_f)
        add("symmetric contraction", flops=sc_f)
        if training:
            tfwd_b = e * (8 * npath * c + 128 + 8) + n * 4 * c * (2 * nx + noc)
            tvjp_b = e * (12 * npath * c + 128 + 64 + 8) + n * 4 * c * (3 * nx + noc)
            add("message kernels", nbytes=vjp_b + tfwd_b + tvjp_b)
            add("radial MLP", flops=4 * hidden)
            add("radial MLP", flops=4 * last, peak=MFMA_SPLIT_PEAK_TFLOPS)
            add("message linear", flops=4 * lin_f, peak=MFMA_SPLIT_PEAK_TFLOPS)
            add("channel linears", flops=4 * chan_f)
            add("symmetric contraction", flops=2 * sc_f)
    return {"terms_ms": terms, "t_min_ms": sum(terms.values())}


def _peak_bytes(fn, device) -> int:
    """Device memory a call allocates at its peak beyond what was allocated before it."""
    fn()
    torch.cuda.synchronize(device)
    torch.cuda.reset_peak_memory_stats(device)
    base = torch.cuda.memory_allocated(device)
    fn()
    torch.cuda.synchronize(device)
    return int(torch.cuda.max_memory_allocated(device) - base)


def _bench_graph(device):
    """Periodic radius graph on HIP (cell list) for the cfg-2 and cfg-4 structures: median of
    synchronised calls (the builder returns edge counts to the host, so calls are synchronous)."""
    from mace_hip import radius_graph_pbc_gpu, sequential_insertion, uniform_box
    out = {}
    for name, st in (("cfg2_16384_atoms", uniform_box(MSG_ATOMS, 0.1, seed=4)),
                     ("cfg4_2048_atoms", sequential_insertion(MACE_ATOMS, 0.1, min_separation=1.5, num_species=10,
                                                              seed=4))):
        pos, cell = st.positions.to(device), st.cell.to(device)
        edges = radius_graph_pbc_gpu(pos, 5.0, cell)[0].numel()
        ms = _median_call_ms(lambda: radius_graph_pbc_gpu(pos, 5.0, cell), device, warmup_s=0.5)
        out[name] = {"atoms": pos.shape[0], "edges": edges, "median_ms": ms, "edges_per_s": edges / (ms * 1e-3)}
    return out


def _cpu_time(fn, budget_s: float, warmup: bool = True):
    if warmup:
        fn()
    done, t0 = 0, time.perf_counter()
    while time.perf_counter() - t0 < budget_s or done == 0:
        fn()
        done += 1
    return done, time.perf_counter() - t0


def _cpu_message(budget_s: float = 8.0):
    """Oracle gather -> TP -> index_add on the edges of the first 512 receivers of cfg 2."""
    sys.path.insert(0, ROOT)
    from oracle.tensor_product import TensorProductOracle
    from mace_hip.structures import radius_graph, uniform_box
    threads = os.cpu_count() or 1
    torch.set_num_threads(threads)
    st = uniform_box(MSG_ATOMS, 0.1, seed=4)
    src, dst, shifts = radius_graph(st.positions, st.cell, 5.0, rows_per_chunk=512)
    keep = dst < 512
    src, dst, shifts = src[keep], dst[keep], shifts[keep]
    from oracle import ictc_basis as B
    vec = (st.positions[dst] - st.positions[src] + shifts @ st.cell).double()
    y = B.direction_harmonics_packed(vec / vec.norm(dim=1, keepdim=True), MSG_L).float()
    gen = torch.Generator().manual_seed(0)
    x = torch.randn(MSG_ATOMS, 576, generator=gen)
    g = torch.randn(src.numel(), MSG_P * MSG_C, generator=gen) / math.sqrt(MSG_P)
    op = TensorProductOracle(MSG_C, MSG_L, MSG_L, MSG_L, dtype=torch.float32)
    done, dt = _cpu_time(lambda: op.graph_message(x, y, g, src, dst, nodes=MSG_ATOMS), budget_s)
    return {"value": src.numel() * done / dt, "unit": "edges/s", "cores": threads, "cpu_model": _cpu_model(), "kind": "port",
            "sample": f"oracle message forward (gather -> _forward_index_add -> index_add, fp32), "
                      f"{src.numel()} edges of 512 receivers x {done} calls in {dt:.1f}s"}


def _cpu_sc(budget_s: float = 8.0):
    """Oracle _forward_selected_elements recursion + autograd VJP on 256 nodes of cfg 3."""
    sys.path.insert(0, ROOT)
    from oracle.symmetric_contraction import SymmetricContractionOracle
    threads = os.cpu_count() or 1
    torch.set_num_threads(threads)
    ref = SymmetricContractionOracle(SC_S, SC_C, SC_L, SC_T, SC_K, seed=1, dtype=torch.float32)
    x, species, go = (t.cpu() for t in _sc_inputs("cpu", 256))

    def step():
        xx = x.clone().requires_grad_()
        torch.autograd.grad(ref.forward(xx, species), xx, go)
    done, dt = _cpu_time(step, budget_s)
    return {"value": 256 * done / dt, "unit": "nodes/s (fwd+VJP)", "cores": threads, "cpu_model": _cpu_model(), "kind": "port",
            "sample": f"oracle contraction recursion + autograd VJP (fp32), 256 nodes x {done} calls in {dt:.1f}s"}


def _cpu_mace(budget_s: float = 10.0, training: bool = False):
    """Float32 oracle model on a smaller cell (same density and cutoff as cfg 4): E + F
    (inference), or the force-loss training step (E + F with create_graph, loss
    mean((E/N)^2) + mean(F^2), backward to every parameter, AdamW)."""
    sys.path.insert(0, ROOT)
    from oracle.mace import MaceOracle
    from mace_hip.model import MaceICTC
    threads = os.cpu_count() or 1
    torch.set_num_threads(threads)
    torch.manual_seed(0)
    model = MaceICTC(channels=128, lmax=3, num_interactions=2, correlation=3, atomic_numbers=MACE_ZS, cutoff=5.0)
    params = {k: v.detach().clone().requires_grad_(training) for k, v in model.named_parameters()}
    oracle = MaceOracle({**dict(model.named_buffers()), **params}, channels=128, lmax=3, num_interactions=2, correlation=3, num_elements=10,
                        cutoff=5.0, avg_num_neighbors=50.0)
    st, g = _mace_graph("cpu", atoms=MACE_CPU_ATOMS)
    args = dict(pos=g["positions"], species=st.species, src=g["edge_src"], dst=g["edge_dst"],
                shifts=g["edge_shifts"], cell=g["cell"], batch=g["batch"])
    if training:
        opt = torch.optim.AdamW(list(params.values()), lr=1e-3)

        def step():
            energy, forces, _ = oracle.energy_and_forces(**args, create_graph=True)
            loss = (energy / MACE_CPU_ATOMS).square().mean() + forces.square().mean()
            loss.backward()
            opt.step()
            opt.zero_grad(set_to_none=True)
        what, unit = "force-loss training step", "atom-steps/s (force-loss training)"
    else:
        def step():
            oracle.energy_and_forces(**args)
        what, unit = "E+F", "atom-steps/s (E+F inference)"
    # a training step takes seconds on the host: it is timed without a warmup call
    done, dt = _cpu_time(step, budget_s, warmup=not training)
    return {"value": MACE_CPU_ATOMS * done / dt, "unit": unit, "cores": threads, "cpu_model": _cpu_model(),
            "kind": "port",
            "sample": f"oracle MACE restatement fp32 {what}, {MACE_CPU_ATOMS} atoms ({g['edge_src'].numel()} edges) "
                      f"x {done} calls in {dt:.1f}s"}


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=50)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--kernels-only", action="store_true")
    ap.add_argument("--only", choices=("tp", "tp0", "message", "message3", "sc", "mace", "mace_steps",
                                       "mace_steps_inference", "mace_steps_training", "graph", "linear", "radial",
                                       "l4", "valu"),
                    default=None,
                    help="run one section and print its JSON (for profiling)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py: this build measures one GPU only (got --gpus {args.gpus}); the hot "
              "path is embarrassingly parallel over instances and is not run multi-GPU here.",
              file=sys.stderr)
        return 2
    device = torch.device("cuda", 0)
    from ictc_o3 import EdgeTensorProduct
    op = EdgeTensorProduct.create(channels=C, input_lmax=L, edge_lmax=L, device=device)
    if args.kernels_only:
        _kernels_only(op.plan, device)
        return 0
    if args.only in ("tp0", "message", "message3", "sc", "mace", "mace_steps", "mace_steps_inference",
                     "mace_steps_training", "graph", "linear", "radial", "l4", "valu"):
        fn = {"tp0": _bench_tp_cfg0, "message": _bench_message, "message3": _bench_message3, "sc": _bench_sc,
              "mace": _bench_mace, "mace_steps": _bench_mace_steps,
              "mace_steps_inference": lambda d: _bench_mace_steps(d, ("inference",)),
              "mace_steps_training": lambda d: _bench_mace_steps(d, ("training",)),
              "graph": _bench_graph, "linear": _bench_linear, "radial": _bench_radial,
              "l4": _bench_tp_l4, "valu": _valu_form_cycles}[args.only]
        print(json.dumps({args.only: fn(device)}), flush=True)
        return 0
    elapsed, vjp_ms, fwd_ms = _time_gpu(args, op.plan, device)
    copy_gbs = _copy_gbs(device)
    mix_vjp = _stream_mix_gbs(device, 7, 2, BYTES_VJP * ROWS_VJP)
    mix_fwd = _stream_mix_gbs(device, 2, 5, BYTES_FWD * ROWS_FWD)
    value = ROWS_VJP * args.steps / elapsed
    achieved = BYTES_VJP * ROWS_VJP / (vjp_ms * 1e-3) / 1e9
    fwd_achieved = BYTES_FWD * ROWS_FWD / (fwd_ms * 1e-3) / 1e9
    cpu = None if args.no_cpu else _cpu_baseline()
    others = {}
    if args.only is None:
        others = {"tp_cfg0": _bench_tp_cfg0(device), "message_cfg2": _bench_message(device),
                  "message_cfg4_lmax3": _bench_message3(device), "sc_cfg3": _bench_sc(device),
                  "mace_cfg4": _bench_mace(device), "message_linear_cfg4": _bench_linear(device),
                  "radial_mlp_cfg4": _bench_radial(device),
                  "radius_graph": _bench_graph(device), "tp_l4": _bench_tp_l4(device)}
        if not args.no_cpu:
            others["tp_cfg0"]["cpu_baseline"] = _cpu_tp_cfg0()
            others["message_cfg2"]["cpu_baseline"] = _cpu_message()
            others["sc_cfg3"]["cpu_baseline"] = _cpu_sc()
            others["mace_cfg4"]["cpu_baseline"] = _cpu_mace()
            others["mace_cfg4"]["cpu_baseline_training"] = _cpu_mace(training=True)
    line = {
        "metric": "TP instances/s fwd+VJP C128/lmax3; MACE E+F atom-steps/s; % HBM peak",
        "value": value, "unit": "instances/s", "n_gpus": 1, "steps": args.steps,
        "warmup": args.warmup, "ms_per_step": elapsed * 1e3 / args.steps, "higher_is_better": True,
        "scaling": "weak", "vs_baseline": value / PUBLISHED_FWD_VJP_INST_S, "dtype": "fp32",
        "data": "synthetic (seeded N(0,1) features, unit-sphere directions -> ICTC Y, N(0,1)/sqrt(P) gates)",
        "config": {"workload": "channelwise CG TP forward + VJP (grads x, Y, gates)", "channels": C,
                   "lmax": L, "paths": P, "instances": ROWS_VJP, "layout": "ir_mul"},
        "roofline": {"bound": "hbm", "kernel": "tp_backward_kernel<3,3,3,2>", "achieved": achieved,
                     "peak": HBM_PEAK_GBS, "unit": "GB/s", "frac": achieved / HBM_PEAK_GBS,
                     "traffic": _measured_traffic(), "traffic_unit": "bytes/launch",
                     "algorithmic_bytes_per_launch": BYTES_VJP * ROWS_VJP,
                     "mean_launch_ms": vjp_ms},
        "cpu_baseline": cpu,
        "extra": {"copy_gbs_measured": copy_gbs,
                  "vjp_frac_of_copy": achieved / copy_gbs,
                  "stream_mix_reference": {
                      "what": "ideal grid-stride float4 streaming kernel moving the same bytes per launch in "
                              "a matching read:write mix (7:2 for the VJP's 3.53:1, 2:5 for the forward's "
                              "0.395:1), best of three grid sizes and both load cache policies",
                      "vjp_mix_gbs": mix_vjp, "fwd_mix_gbs": mix_fwd,
                      "vjp_frac_of_mix": achieved / mix_vjp if mix_vjp else None,
                      "fwd_frac_of_mix": fwd_achieved / mix_fwd if mix_fwd else None},
                  "step_hbm_gbs": (BYTES_FWD + BYTES_VJP) * value / 1e9,
                  "step_hbm_frac": (BYTES_FWD + BYTES_VJP) * value / 1e9 / HBM_PEAK_GBS,
                  "forward_only": {"instances": ROWS_FWD, "instances_per_s": ROWS_FWD / (fwd_ms * 1e-3),
                                   "mean_launch_ms": fwd_ms, "achieved_gbs": fwd_achieved,
                                   "frac": fwd_achieved / HBM_PEAK_GBS,
                                   "vs_published_2.70M": ROWS_FWD / (fwd_ms * 1e-3) / 2.70e6},
                  **others},
    }
    print(json.dumps(line), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
