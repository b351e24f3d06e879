#!/usr/bin/env python3
"""Throughput of the gate-application hot path on one MI355X.

Workload: the 30-qubit random-layer circuit (20 layers; each layer U3(theta,
phi, lambda) on every qubit, emitted as U1, plus CZ on a seeded perfect
matching, emitted as CP pi; 900 gates, seed 2) applied as a plain gate list
(sq_apply_gates, the MEM_Runner::run(vector<Gate*>&) interface) to a
complex128 state in HBM (16 GiB) from |0...0>.  One step = the whole 900-gate
circuit: its op records encoded and uploaded, every pass run.  The pass
schedule is planned on the first call and reused from the engine's schedule
cache (keyed by the gates' qubits and classes) on later calls; that first
call, planning included, is reported as cold_first_call_ms.  The engine runs the list as register passes (a
run of one-qubit and diagonal gates per read and write of the state, each gate
with its own 2x2 or diagonal arithmetic); the same list one launch per gate is
reported beside it.  The fused planner blocks (complex64 and complex128) and
a complex64 state are reported against the complex128 result.

Prints one JSON line (rank 0).  value = complex128 gates/s over the K timed
steps; roofline = the kernel with the most time in those steps, timed with HIP
events on the engine's stream; cpu_baseline = the reference's own MEM gate
code (oracle/_ref) or the oracle port, on this host, on a bounded sample of
the same circuit (its first layer, 45 gates at 30 qubits).
"""
import argparse
import json
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

METRIC = "30q random circuit: gates/s, HBM GB/s; fused c64 vs plain c128 @1e-6 infid"
HBM_PEAK_GBS = 8000.0
FP64_VALU_PEAK_TFLOPS = 78.6   # MI355X vector FP64 (no packed FP32 in these kernels)
N_QUBITS, LAYERS, SEED = 30, 20, 2


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=2)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--qubits", type=int, default=N_QUBITS)
    ap.add_argument("--layers", type=int, default=LAYERS)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-c64", action="store_true")
    ap.add_argument("--cpu-sample-gates", type=int, default=45)
    ap.add_argument("--no-fused", action="store_true")
    ap.add_argument("--fused-k", type=int, default=5)
    ap.add_argument("--fused-dtypes", default="c64,c128")
    ap.add_argument("--no-adjoint", action="store_true")
    ap.add_argument("--workload", default="random30",
                    choices=["random30", "fused32", "stream", "qft20", "blocks30", "traffic"],
                    help="random30: the headline line (default).  fused32: 32 qubits, 24 layers, "
                         "fused complex64 vs plain complex128.  stream: out-of-core runner "
                         "(state in pinned host memory) vs the same circuit in HBM.  qft20: "
                         "20-qubit QFT on a seeded state.  blocks30: the 30-qubit circuit as a "
                         "chunk-12 subcircuit file.  traffic: a short fixed kernel "
                         "sequence for rocprofv3 --pmc HBM-byte counts")
    ap.add_argument("--stream-dtype", default="c128")
    ap.add_argument("--resident-qbit", type=int, default=30)
    ap.add_argument("--stream-layers", type=int, default=12)
    return ap.parse_args()


def traffic_from_profiles(kernel):
    """HBM bytes per launch measured by rocprofv3 --pmc (FETCH_SIZE + WRITE_SIZE),
    committed under profiles/; None when no measurement exists."""
    p = os.path.join(ROOT, "profiles", "traffic.json")
    if not os.path.exists(p):
        return None
    try:
        return json.load(open(p)).get(kernel, {}).get("bytes_per_launch")
    except Exception:
        return None


def cpu_baseline(text, n, sample_gates):
    """Times the first sample_gates gates of the circuit on this host's cores."""
    import ctypes
    import numpy as np
    threads = int(os.environ.get("OMP_NUM_THREADS", "0")) or os.cpu_count()
    lines = [l for l in text.splitlines() if l.strip()][:sample_gates]
    sample = "\n".join(lines) + "\n"
    state = np.zeros(1 << n, dtype=np.complex128)
    state[0] = 1
    ref = os.path.join(ROOT, "oracle", "_ref", "libsqref.so")
    secs = ctypes.c_double(0)
    if os.path.exists(ref):
        L = ctypes.CDLL(ref)
        L.sqref_set_threads.argtypes = [ctypes.c_int]
        L.sqref_time_plain_text.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_char_p,
                                            ctypes.POINTER(ctypes.c_double)]
        L.sqref_set_threads(threads)
        rc = L.sqref_time_plain_text(state.ctypes.data, n, 12, sample.encode(), ctypes.byref(secs))
        kind = "reference"
    else:
        L = ctypes.CDLL(os.path.join(ROOT, "oracle", "libsq_oracle.so"))
        L.sqo_set_threads.argtypes = [ctypes.c_int]
        L.sqo_run_plain_text.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_char_p, ctypes.c_void_p]
        L.sqo_set_threads(threads)
        t0 = time.perf_counter()
        rc = L.sqo_run_plain_text(state.ctypes.data, n, 12, sample.encode(), None)
        secs.value = time.perf_counter() - t0
        kind = "port"
    if rc != 0:
        return None
    del state
    return {"value": len(lines) / secs.value, "unit": "gates/s", "cores": threads, "kind": kind,
            "sample": f"first {len(lines)} gates (one layer) of the {n}-qubit circuit, complex128, "
                      f"chunk_qbit=12, {threads} OpenMP threads, {secs.value:.2f} s",
            "seconds": secs.value}


def copy_ceiling(eng, n):
    """Device-to-device copy bandwidth (HIP's own copy kernel) inside the
    engine's state buffer: the first half copied onto the second half, 5 times.
    Bytes = read + write.  Measured before the timed steps; the state is reset
    afterwards by init_zero."""
    import ctypes
    hip = ctypes.CDLL("libamdhip64.so")
    hip.hipMemcpyDtoD.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    hip.hipDeviceSynchronize.argtypes = []
    ptr, _ = eng.device_state()
    half = (16 << n) // 2
    eng.sync()
    if hip.hipMemcpyDtoD(ptr + half, ptr, half) != 0 or hip.hipDeviceSynchronize() != 0:
        return None
    t0 = time.perf_counter()
    for _ in range(5):
        hip.hipMemcpyDtoD(ptr + half, ptr, half)
    if hip.hipDeviceSynchronize() != 0:
        return None
    return 5 * 2 * half / (time.perf_counter() - t0) / 1e9


def log(msg):
    print(f"[bench] {msg}", file=sys.stderr, flush=True)


def line(metric, value, unit, steps, warmup, ms, dtype, config, **extra):
    out = {"metric": metric, "value": round(value, 3), "unit": unit, "n_gpus": 1, "steps": steps,
           "warmup": warmup, "ms_per_step": round(ms, 2), "higher_is_better": True, "scaling": "weak",
           "vs_baseline": None, "dtype": dtype, "data": "synthetic (seeded generator)", "config": config}
    out.update(extra)
    return out


def fused_kernel_figures(st, dtype, n):
    """The kernel that applied the blocks: k_fused5 (one 32x32 product per
    block), or the register passes that carry complex128 blocks."""
    name = f"fused5_{dtype}" if f"fused5_{dtype}" in st else max(st, key=lambda k: st[k]["total_ms"])
    k = st[name]
    avg_ms = k["total_ms"] / k["launches"]
    gbs = k["alg_bytes"] / k["launches"] / (avg_ms * 1e-3) / 1e9
    out = {"name": name, "launches": k["launches"], "avg_launch_ms": round(avg_ms, 4), "hbm_gbs": round(gbs, 1),
           "hbm_frac": round(gbs / HBM_PEAK_GBS, 4)}
    if name.startswith("fused5"):
        tflops = 8.0 * 32 * 2 ** n / (avg_ms * 1e-3) / 1e12   # complex 32x32 per 32-amplitude column
        peak_tf = 157.3 if dtype == "c64" else 78.6
        out.update(mfma_tflops=round(tflops, 1), mfma_frac=round(tflops / peak_tf, 4), mfma_peak_tflops=peak_tf)
    return out


def fused_passes_leg(sq, gates, ng, n, args, ref, plain_c128_s):
    """sq_apply_gates_fused on a complex64 state: the gate list in LDS-resident
    tile passes, four-qubit blocks on MFMA (split bf16 products, FP32
    accumulation).  The first call plans (cold_first_call_ms); the timed calls
    reuse the plan from the engine's cache and compose and apply every block."""
    eng = sq.Engine(n, dtype="c64")
    eng.init_zero()
    eng.sync()
    t0 = time.perf_counter()
    eng.apply_gates_fused(gates, ng)
    eng.sync()
    cold = time.perf_counter() - t0
    for _ in range(max(0, args.warmup - 1)):
        eng.init_zero()
        eng.apply_gates_fused(gates, ng)
    eng.sync()
    eng.stats_reset()
    eng.stats_enable(True)
    times = []
    for _ in range(args.steps):
        eng.init_zero()
        eng.sync()
        t0 = time.perf_counter()
        eng.apply_gates_fused(gates, ng)
        eng.sync()
        times.append(time.perf_counter() - t0)
        log(f"fused passes c64 step {len(times)}: {times[-1]*1e3:.1f} ms")
    st = eng.stats()
    eng.stats_enable(False)
    k = st["fpass_c64"]
    avg_ms = k["total_ms"] / k["launches"]
    bpl = k["alg_bytes"] / k["launches"]
    # MFMA work as executed: three split products per block (bf16, dense peak 2.5 PFLOP/s)
    mfma_tf = 3.0 * k["alg_flops"] / (k["total_ms"] * 1e-3) / 1e12
    ov = ref.inner(eng)
    infid = 1.0 - abs(ov) ** 2 / (ref.norm2() * eng.norm2())
    err = ref.max_abs_diff(eng)
    eng.close()
    tt = sum(times) / len(times)
    return {"gates_s": round(ng / tt, 2), "ms_per_step": round(tt * 1e3, 2), "cold_first_call_ms": round(cold * 1e3, 2),
            "passes": k["launches"] // args.steps, "speedup_vs_plain_c128": round(plain_c128_s / tt, 2),
            "infidelity_vs_plain_c128": infid, "max_abs_err_vs_plain_c128": err,
            "kernel": {"name": "k_fpass<13>", "avg_launch_ms": round(avg_ms, 4),
                       "hbm_gbs": round(bpl / (avg_ms * 1e-3) / 1e9, 1),
                       "hbm_frac": round(bpl / (avg_ms * 1e-3) / 1e9 / HBM_PEAK_GBS, 4),
                       "mfma_bf16_tflops_executed": round(mfma_tf, 1),
                       "mfma_frac": round(mfma_tf / 2500.0, 4), "mfma_peak_tflops": 2500.0},
            "what": "sq_apply_gates_fused: tile passes of 13 qubits, four-qubit blocks composed in FP64, "
                    "split-bf16 MFMA products accumulated in FP32"}


def workload_fused32(args):
    """32 qubits, 24 layers of the random-layer generator (1152 gates, seed 3):
    planner -> 5-qubit blocks composed in FP64 and applied on MFMA to a
    complex64 state (32 GiB), against the plain complex128 sweep (64 GiB) as
    register passes (schedule planned on a warm-up call) and one launch per
    gate (the reference's plain sweep shape); the same gate list as fused
    passes (fused_passes_c64) beside it."""
    import subquokka_dev_amd as sq
    n, layers, seed = 32, 24, 3
    text = sq.gen_circuit("random", n, layers, seed=seed)
    gates, _, ng, _ = sq.parse_circuit(text, n)
    log(f"fused32: {ng} gates")
    ref = sq.Engine(n, dtype="c128")
    ref.init_zero()
    ref.apply_gates(gates, ng)   # warm-up: plans the register passes, caches the schedule
    ref.init_zero()
    ref.sync()
    t0 = time.perf_counter()
    ref.apply_gates(gates, ng)
    ref.sync()
    t_plain = time.perf_counter() - t0
    log(f"plain c128 (register passes): {t_plain:.3f} s")
    g1 = sq.Engine(n, dtype="c128", sweep_mode=1)
    g1.init_zero()
    g1.sync()
    t0 = time.perf_counter()
    g1.apply_gates(gates, ng)
    g1.sync()
    t_gate = time.perf_counter() - t0
    gate_diff = ref.max_abs_diff(g1)
    g1.close()
    log(f"plain c128 (one launch per gate): {t_gate:.2f} s")
    t0 = time.perf_counter()
    plan = sq.plan(text, n, 1, args.fused_k)
    plan_s = time.perf_counter() - t0
    fg, fb, _, fnb = sq.parse_circuit(plan, n, is_subcircuit=True)
    eng = sq.Engine(n, dtype="c64")
    for _ in range(args.warmup):
        eng.init_zero()
        eng.run_fused(fg, fb, fnb)
    eng.sync()
    eng.stats_reset()
    eng.stats_enable(True)
    times = []
    for _ in range(args.steps):
        eng.init_zero()
        eng.sync()
        t0 = time.perf_counter()
        eng.run_fused(fg, fb, fnb)
        eng.sync()
        times.append(time.perf_counter() - t0)
        log(f"fused c64 step {len(times)}: {times[-1]*1e3:.1f} ms")
    st = eng.stats()
    eng.stats_enable(False)
    ov = ref.inner(eng)
    infid = 1.0 - abs(ov) ** 2 / (ref.norm2() * eng.norm2())
    tt = sum(times) / len(times)
    out = line("32q random circuit: fused c64 gates/s (planner blocks, MFMA) vs plain c128",
               ng / tt, "gates/s", args.steps, args.warmup, tt * 1e3, "f32",
               {"workload": f"random_layers_{n}q_{layers}l_seed{seed}_fused{args.fused_k}_c64", "n_qubits": n,
                "layers": layers, "gates": ng, "blocks": fnb, "state": "complex64 in HBM (32 GiB)"},
               plain_c128={"gates_s": round(ng / t_plain, 2), "seconds": round(t_plain, 3),
                           "what": "register passes, schedule from a warm-up call"},
               plain_c128_one_launch_per_gate={"gates_s": round(ng / t_gate, 2), "seconds": round(t_gate, 3),
                                               "max_abs_diff_vs_register_passes": gate_diff},
               speedup_vs_plain_c128=round(t_plain / tt, 2),
               speedup_vs_plain_c128_one_launch_per_gate=round(t_gate / tt, 2), infidelity_vs_plain_c128=infid,
               max_abs_err_vs_plain_c128=ref.max_abs_diff(eng), plan_s=round(plan_s, 3),
               kernel=fused_kernel_figures(st, "c64", n),
               compose_ms_per_step=round(st.get("compose_f64", {"total_ms": 0})["total_ms"] / args.steps, 3))
    eng.close()
    out["fused_passes_c64"] = fused_passes_leg(sq, gates, ng, n, args, ref, t_plain)
    fp = out["fused_passes_c64"]
    fp["speedup_vs_plain_c128_one_launch_per_gate"] = round(t_gate / (fp["ms_per_step"] * 1e-3), 2)
    ref.close()
    return out


def workload_stream(args):
    """Out-of-core runner (DIO_Runner role, host RAM tier): the state lives in
    pinned host memory and is streamed through two HBM buffers of
    2^resident_qbit amplitudes, pass by pass; the same circuit then runs with
    the state resident in HBM.  --stream-layers layers (default 12) of the
    random-layer generator, seed 5."""
    import subquokka_dev_amd as sq
    n, layers, seed, dtype = args.qubits, args.stream_layers, 5, args.stream_dtype
    text = sq.gen_circuit("random", n, layers, seed=seed)
    per_layer = [l for l in text.splitlines() if l.strip()]
    ng = len(per_layer)
    chunks = 4
    step = (ng + chunks - 1) // chunks
    parts = ["\n".join(per_layer[i:i + step]) + "\n" for i in range(0, ng, step)]
    B = 16 if dtype == "c128" else 8
    log(f"stream: {n} qubits {dtype}, {ng} gates, host state {B * 2 ** n / 2 ** 30:.0f} GiB, "
        f"HBM groups of 2^{args.resident_qbit}")
    eng = sq.Engine(n, dtype=dtype, resident_qbit=args.resident_qbit)
    t0 = time.perf_counter()
    eng.init_zero()
    eng.sync()
    log(f"host init {time.perf_counter() - t0:.1f} s")
    eng.stats_reset()
    t0 = time.perf_counter()
    for i, p in enumerate(parts):
        eng.apply_text(p)
        eng.sync()
        log(f"stream part {i + 1}/{len(parts)}: {time.perf_counter() - t0:.1f} s")
    t_stream = time.perf_counter() - t0
    passes, link_bytes, tier = eng.stream_info()
    zz_s, nrm_s = eng.expect_zz_ring(), eng.norm2()
    eng.close()
    hbm = sq.Engine(n, dtype=dtype)
    hbm.init_zero()
    hbm.sync()
    t0 = time.perf_counter()
    hbm.apply_text(text)
    hbm.sync()
    t_hbm = time.perf_counter() - t0
    zz_h, nrm_h = hbm.expect_zz_ring(), hbm.norm2()
    hbm.close()
    log(f"in HBM: {t_hbm:.2f} s; <ZZ> {zz_s:.12f} vs {zz_h:.12f}")
    return line(f"{n}q random circuit, state outside HBM ({tier} host tier) streamed through HBM: gates/s",
                ng / t_stream, "gates/s", 1, 0, t_stream * 1e3, "f64" if dtype == "c128" else "f32",
                {"workload": f"random_layers_{n}q_{layers}l_seed{seed}_stream_{dtype}_w{args.resident_qbit}",
                 "n_qubits": n, "layers": layers, "gates": ng, "state": f"{dtype} in {tier} host memory"},
                passes=passes, host_tier=tier, host_link_gbs=round(link_bytes / t_stream / 1e9, 1),
                host_link_bytes=link_bytes, in_hbm={"seconds": round(t_hbm, 3), "gates_s": round(ng / t_hbm, 2)},
                stream_over_hbm_time=round(t_stream / t_hbm, 2),
                zz_ring={"stream": zz_s, "hbm": zz_h, "abs_diff": abs(zz_s - zz_h)},
                norm2={"stream": nrm_s, "hbm": nrm_h})


def workload_qft20(args):
    """20-qubit QFT (cir_qft.py order, 220 gates) on a seeded Gaussian state,
    complex128, whole state in HBM (16 MiB: cache-resident, launch-bound)."""
    import subquokka_dev_amd as sq
    n = 20
    text = sq.gen_circuit("qft", n)
    gates, _, ng, _ = sq.parse_circuit(text, n)
    s0 = sq.gen_state(n, 1)
    eng = sq.Engine(n, dtype="c128")
    for _ in range(args.warmup):
        eng.set_state(s0)
        eng.apply_gates(gates, ng)
    times = []
    for _ in range(args.steps):
        eng.set_state(s0)
        eng.sync()
        t0 = time.perf_counter()
        eng.apply_gates(gates, ng)
        eng.sync()
        times.append(time.perf_counter() - t0)
    eng.close()
    tt = sum(times) / len(times)
    return line("20q QFT on a seeded state: gates/s", ng / tt, "gates/s", args.steps, args.warmup, tt * 1e3,
                "f64", {"workload": "qft_20q_seed1_plain_c128", "n_qubits": n, "gates": ng,
                        "state": "complex128 in HBM (16 MiB)"})


def workload_blocks30(args):
    """The 30-qubit random-layer circuit as a subcircuit file (finder format,
    chunk_qbit 12: gate blocks and VSWAP blocks, no order restore) through
    sq_apply_blocks, complex128 in HBM.  The default sweep relabels the VSWAPs
    on the host and applies one set of qubit swaps at the end; the
    reference-shaped sweep (physical VSWAP passes and one LDS tile pass per
    gate block) is timed beside it, and the two final states compared."""
    import subquokka_dev_amd as sq
    n, layers, chunk = 30, 20, 12
    text = sq.gen_circuit("random", n, layers, seed=SEED)
    plan = sq.plan(text, n, 0, chunk)
    gates, blocks, ng, nb = sq.parse_circuit(plan, n, is_subcircuit=True)
    n_vswap = sum(1 for l in plan.splitlines() if l.startswith("VSWAP"))

    def timed(sweep_mode, steps, warmup):
        eng = sq.Engine(n, dtype="c128", chunk=chunk, sweep_mode=sweep_mode)
        for _ in range(warmup):
            eng.init_zero()
            eng.apply_blocks(gates, blocks, nb)
        eng.sync()
        times, st = [], None
        for _ in range(steps):
            eng.init_zero()
            eng.sync()
            eng.stats_reset()
            eng.stats_enable(True)
            t0 = time.perf_counter()
            eng.apply_blocks(gates, blocks, nb)
            eng.sync()
            times.append(time.perf_counter() - t0)
            st = eng.stats()
        return eng, sum(times) / len(times), st

    def kstats(st):
        return {k: {"launches": v["launches"], "avg_ms": round(v["total_ms"] / v["launches"], 3),
                    "gbs": round(v["alg_bytes"] / (v["total_ms"] * 1e-3) / 1e9, 1)} for k, v in st.items()}

    e0, t0, st0 = timed(0, args.steps, args.warmup)
    e1, t1, st1 = timed(1, 1, 1)
    diff = e0.max_abs_diff(e1)
    e0.close()
    e1.close()
    out = line("30q random circuit as a chunk-12 subcircuit file: gates/s", (ng - n_vswap) / t0, "gates/s",
               args.steps, args.warmup, t0 * 1e3, "f64",
               {"workload": f"random_layers_{n}q_{layers}l_seed{SEED}_blocks_chunk{chunk}_c128", "n_qubits": n,
                "gates": ng - n_vswap, "vswap_blocks": n_vswap, "blocks": nb, "state": "complex128 in HBM",
                "mode": "MEM_Runner::run(vector<vector<Gate*>>&) form: VSWAPs relabelled, register passes"})
    out["kernels"] = kstats(st0)
    out["reference_shaped_sweep"] = {"ms_per_step": round(t1 * 1e3, 1), "kernels": kstats(st1),
                                     "what": "physical VSWAP sweeps + one LDS tile pass per gate block",
                                     "max_abs_diff_vs_default": diff}
    return out


def workload_traffic(args):
    """A short fixed kernel sequence whose HBM bytes per dispatch rocprofv3
    --pmc reads (FETCH_SIZE, WRITE_SIZE): a 4 GiB device copy of known size
    (the scale factor), then on a 30-qubit complex128 state, one launch per
    gate, 3 dense one-qubit gates with the target at or above bit 6, 3 with
    the target in bits 0-5 and 3 CP gates; the 30-qubit random circuit
    (900 gates) as register passes in complex128 and in complex64; the same
    circuit as a chunk-12 subcircuit file (register passes, then the one
    bit-permutation pass to the final qubit order); one fused 5-qubit block
    in complex128 and in complex64."""
    import torch
    import subquokka_dev_amd as sq
    n = 30
    a = torch.ones(2 ** 30, dtype=torch.float32, device="cuda")
    b = torch.empty_like(a)
    ev0, ev1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    b.copy_(a)
    torch.cuda.synchronize()
    ev0.record()
    for _ in range(5):
        b.copy_(a)
    ev1.record()
    torch.cuda.synchronize()
    copy_gbs = 5 * 2 * 4 * 2 ** 30 / (ev0.elapsed_time(ev1) * 1e-3) / 1e9
    del a, b
    torch.cuda.empty_cache()
    u = "0.6 0.0 0.0 0.8 0.8 0.0 0.0 -0.6"
    text = "".join(f"U1 {q} {u}\n" for q in (20, 25, 29)) + "".join(f"U1 {q} {u}\n" for q in (0, 2, 5)) + \
        "".join(f"CP {a} {b} 3.141592653589793\n" for a, b in ((3, 17), (8, 22), (11, 28)))
    eng = sq.Engine(n, dtype="c128", sweep_mode=1)
    eng.init_zero()
    eng.apply_text(text)
    eng.sync()
    eng.close()
    # register passes: the whole 30-qubit random circuit
    circ = sq.gen_circuit("random", n, LAYERS, seed=SEED)
    for dtype in ("c128", "c64"):
        eng = sq.Engine(n, dtype=dtype)
        eng.init_zero()
        eng.apply_text(circ)
        eng.sync()
        eng.close()
    # the same circuit as a chunk-12 subcircuit file (ends with k_bitperm)
    gates, blocks, _, nb = sq.parse_circuit(sq.plan(circ, n, 0, 12), n, is_subcircuit=True)
    eng = sq.Engine(n, dtype="c128", chunk=12)
    eng.init_zero()
    eng.apply_blocks(gates, blocks, nb)
    eng.sync()
    eng.close()
    blk = "".join(f"U1 {q} {u}\n" for q in (6, 12, 18, 24, 29)) + "CP 6 29 0.5\n"
    import ctypes
    g, _, ng_, _ = sq.parse_circuit(blk, n)
    for dtype in ("c128", "c64"):
        eng = sq.Engine(n, dtype=dtype)
        eng.init_zero()
        eng.run_fused(g, (ctypes.c_uint32 * 1)(ng_), 1)
        eng.sync()
        eng.close()
    return {"workload": "traffic_probe", "copy_gbs_torch": round(copy_gbs, 1)}


def main():
    args = parse()
    if args.gpus != 1:
        print(json.dumps({"error": "this build runs on one GPU only; --gpus must be 1 "
                          "(multi-GPU sharding is a design note, not an implemented path)"}))
        return 2
    import numpy as np
    if args.workload != "random30":
        fn = {"fused32": workload_fused32, "stream": workload_stream, "qft20": workload_qft20,
              "blocks30": workload_blocks30, "traffic": workload_traffic}[args.workload]
        if args.workload == "stream" and args.qubits == N_QUBITS:
            args.qubits = 33
        print(json.dumps(fn(args)), flush=True)
        return 0
    import subquokka_dev_amd as sq

    n, layers = args.qubits, args.layers
    text = sq.gen_circuit("random", n, layers, seed=SEED)
    gates, _, ng, _ = sq.parse_circuit(text, n)
    print(f"[bench] {n} qubits, {layers} layers, {ng} gates", file=sys.stderr, flush=True)

    def run_steps(dtype, steps, warmup, stats, sweep_mode=0):
        eng = sq.Engine(n, dtype=dtype, sweep_mode=sweep_mode)
        if dtype == "c128":
            out_extra["hbm_copy_gbs"] = copy_ceiling(eng, n)
        for w in range(warmup):
            eng.init_zero()
            eng.sync()
            t0 = time.perf_counter()
            eng.apply_gates(gates, ng)
            eng.sync()
            if w == 0:
                out_extra[f"cold_first_call_ms_{dtype}_{sweep_mode}"] = round((time.perf_counter() - t0) * 1e3, 2)
        eng.sync()
        eng.stats_reset()
        eng.stats_enable(stats)
        times = []
        for _ in range(steps):
            eng.init_zero()
            eng.sync()
            t0 = time.perf_counter()
            eng.apply_gates(gates, ng)
            eng.sync()
            times.append(time.perf_counter() - t0)
            print(f"[bench] {dtype} sweep_mode {sweep_mode} step {len(times)}: {times[-1]*1e3:.1f} ms",
                  file=sys.stderr, flush=True)
        st = eng.stats() if stats else {}
        eng.stats_enable(False)
        return eng, times, st

    out_extra = {}
    eng128, t128, st128 = run_steps("c128", args.steps, args.warmup, True)
    total_t = sum(t128)
    gates_s = args.steps * ng / total_t
    alg_bytes = sum(v["alg_bytes"] for v in st128.values()) / args.steps
    hbm_gbs = alg_bytes / (total_t / args.steps) / 1e9

    # dominant kernel: most total time
    dom_name, dom = max(st128.items(), key=lambda kv: kv[1]["total_ms"])
    avg_ms = dom["total_ms"] / dom["launches"]
    bytes_per_launch = dom["alg_bytes"] / dom["launches"]
    achieved = bytes_per_launch / (avg_ms * 1e-3) / 1e9
    roofline = {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBS, "unit": "GB/s",
                "frac": round(achieved / HBM_PEAK_GBS, 4), "traffic": traffic_from_profiles(dom_name),
                "kernel": dom_name, "avg_launch_ms": round(avg_ms, 4),
                "alg_bytes_per_launch": bytes_per_launch}
    if dom.get("alg_flops"):
        tf = dom["alg_flops"] / dom["launches"] / (avg_ms * 1e-3) / 1e12
        roofline["valu_fp64"] = {"achieved_tflops": round(tf, 2), "peak_tflops": FP64_VALU_PEAK_TFLOPS,
                                 "frac": round(tf / FP64_VALU_PEAK_TFLOPS, 4),
                                 "alg_flops_per_launch": dom["alg_flops"] / dom["launches"]}
    kernels = {k: {"launches": v["launches"], "avg_ms": round(v["total_ms"] / v["launches"], 4),
                   "gbs": round(v["alg_bytes"] / (v["total_ms"] * 1e-3) / 1e9, 1)} for k, v in st128.items()}

    out = {"metric": METRIC, "value": round(gates_s, 2), "unit": "gates/s", "n_gpus": 1,
           "steps": args.steps, "warmup": args.warmup, "ms_per_step": round(total_t / args.steps * 1e3, 2),
           "higher_is_better": True, "scaling": "weak", "vs_baseline": None, "dtype": "f64",
           "data": "synthetic (seeded random-layer circuit, |0...0> initial state)",
           "config": {"workload": f"random_layers_{n}q_{layers}l_seed{SEED}_plain_c128", "n_qubits": n,
                      "layers": layers, "gates": ng, "state": "complex128 in HBM",
                      "mode": "plain gate list (MEM_Runner::run(vector<Gate*>&) form) as register passes, "
                              "5 register qubits + 6 lane qubits per pass (3 lane positions chosen per pass); "
                              "each U3 as its phases (applied together per pass) and a real rotation (three "
                              "in-place shears, or one FMA per part on lane bits 0-3), CZ as sign flips",
                      "schedule": "planned on the first (warm-up) call, reused from the engine's schedule cache "
                                  "in the timed steps; op records encoded and uploaded every step"},
           "hbm_gbs": round(hbm_gbs, 1), "roofline": roofline, "kernels_c128": kernels}
    if "cold_first_call_ms_c128_0" in out_extra:
        out["cold_first_call_ms"] = out_extra["cold_first_call_ms_c128_0"]
    if out_extra.get("hbm_copy_gbs"):
        out["hbm_copy_ceiling"] = {"gbs": round(out_extra["hbm_copy_gbs"], 1),
                                   "what": "hipMemcpyDtoD of 8 GiB inside the state buffer (read + write bytes)",
                                   "dominant_kernel_over_copy": round(achieved / out_extra["hbm_copy_gbs"], 4)}

    # the same gate list, one launch per gate (the reference's one pass per gate)
    engpg, tpg, stpg = run_steps("c128", 1, 0, True, sweep_mode=1)
    dpg = max(stpg.items(), key=lambda kv: kv[1]["total_ms"])
    out["plain_one_launch_per_gate_c128"] = {
        "gates_s": round(ng / sum(tpg), 2), "ms_per_step": round(sum(tpg) * 1e3, 2),
        "register_pass_speedup": round(sum(tpg) / (total_t / args.steps), 2),
        "max_abs_diff_vs_register_passes": eng128.max_abs_diff(engpg),
        "dominant_kernel": {"name": dpg[0], "avg_ms": round(dpg[1]["total_ms"] / dpg[1]["launches"], 4),
                            "gbs": round(dpg[1]["alg_bytes"] / (dpg[1]["total_ms"] * 1e-3) / 1e9, 1),
                            "hbm_frac": round(dpg[1]["alg_bytes"] / (dpg[1]["total_ms"] * 1e-3) / 1e9 / HBM_PEAK_GBS, 4)},
        "kernels": {k: {"launches": v["launches"], "avg_ms": round(v["total_ms"] / v["launches"], 4),
                        "gbs": round(v["alg_bytes"] / (v["total_ms"] * 1e-3) / 1e9, 1)} for k, v in stpg.items()}}
    engpg.close()

    if not args.no_fused:
        # Planner (host, once per circuit, outside the timed region -- the
        # reference runs its finder offline too), then per step: FP64
        # composition of every block on the GPU + MFMA application.
        t0 = time.perf_counter()
        plan = sq.plan(text, n, 1, args.fused_k)
        plan_s = time.perf_counter() - t0
        fg, fb, fng, fnb = sq.parse_circuit(plan, n, is_subcircuit=True)
        print(f"[bench] fused plan: {fnb} blocks of <= {args.fused_k} qubits ({plan_s:.2f} s)", file=sys.stderr, flush=True)
        fused = {}
        for dtype in args.fused_dtypes.split(","):
            eng = sq.Engine(n, dtype=dtype)
            for _ in range(args.warmup):
                eng.init_zero()
                eng.run_fused(fg, fb, fnb)
            eng.sync()
            eng.stats_reset()
            eng.stats_enable(True)
            times = []
            for _ in range(args.steps):
                eng.init_zero()
                eng.sync()
                t0 = time.perf_counter()
                eng.run_fused(fg, fb, fnb)
                eng.sync()
                times.append(time.perf_counter() - t0)
                print(f"[bench] fused {dtype} step {len(times)}: {times[-1]*1e3:.1f} ms", file=sys.stderr, flush=True)
            st = eng.stats()
            eng.stats_enable(False)
            ov = eng128.inner(eng)
            infid = 1.0 - abs(ov) ** 2 / (eng128.norm2() * eng.norm2())
            tt = sum(times)
            fused[dtype] = {
                "gates_s": round(args.steps * ng / tt, 2), "ms_per_step": round(tt / args.steps * 1e3, 2),
                "blocks": fnb, "speedup_vs_plain_c128": round((total_t / args.steps) / (tt / args.steps), 2),
                "infidelity_vs_plain_c128": infid, "max_abs_err_vs_plain_c128": eng128.max_abs_diff(eng),
                "kernel": fused_kernel_figures(st, dtype, n),
                "compose_ms_per_step": round(st.get("compose_f64", {"total_ms": 0})["total_ms"] / args.steps, 3),
                "plan_s": round(plan_s, 3)}
            eng.close()
        out["fused"] = fused
        out["fused_passes_c64"] = fused_passes_leg(sq, gates, ng, n, args, eng128, total_t / args.steps)
        fp = out["fused_passes_c64"]
        fp["speedup_vs_plain_c128_one_launch_per_gate"] = round(sum(tpg) / (fp["ms_per_step"] * 1e-3), 2)

    if not args.no_c64:
        eng64, t64, st64 = run_steps("c64", args.steps, args.warmup, False)
        ov = eng128.inner(eng64)
        infid = 1.0 - abs(ov) ** 2 / (eng128.norm2() * eng64.norm2())
        out["c64_plain"] = {"gates_s": round(args.steps * ng / sum(t64), 2),
                            "ms_per_step": round(sum(t64) / args.steps * 1e3, 2),
                            "infidelity_vs_c128": infid, "max_abs_err_vs_c128": eng128.max_abs_diff(eng64)}
        eng64.close()
    # measurement sampler on the final 30-qubit state: one pass over the state
    # (block sums), then one wave per shot reading its 16 KiB block
    shots = 1 << 20
    eng128.sample(1000, 7)
    eng128.sync()
    ts = []
    for _ in range(3):
        t0s = time.perf_counter()
        eng128.sample(shots, 7)
        ts.append(time.perf_counter() - t0s)
    out["sampler"] = {"shots": shots, "ms": round(min(ts) * 1e3, 2), "shots_per_s": round(shots / min(ts), 1),
                      "state": "the circuit's final complex128 state, 2^30 amplitudes",
                      "what": "sq_sample: exact seeded shots (FP64 sums), shots copied to the host"}
    eng128.close()

    if not args.no_adjoint:
        # Adjoint gradient of the 24-qubit hardware-efficient ansatz (8 layers,
        # 384 parameters), complex64 with FP64 checkpoints every 3 layers:
        # cost of energy + full gradient against one forward pass.
        an, al = 24, 8
        theta = np.random.default_rng(4).uniform(-np.pi, np.pi, 2 * an * al)
        ea = sq.Engine(an, dtype="c64")
        ea.hea_energy(al, theta)
        ea.adjoint_grad_hea(al, theta, 3)
        ea.sync()
        fwd, grd = [], []
        for _ in range(3):
            t0 = time.perf_counter()
            ea.hea_energy(al, theta)
            fwd.append(time.perf_counter() - t0)
            t0 = time.perf_counter()
            _, g = ea.adjoint_grad_hea(al, theta, 3)
            grd.append(time.perf_counter() - t0)
        ea.close()
        f, gtime = min(fwd), min(grd)
        out["adjoint_24q_384p_c64"] = {"forward_ms": round(f * 1e3, 3), "energy_and_gradient_ms": round(gtime * 1e3, 3),
                                       "gradient_over_forward": round(gtime / f, 3), "checkpoint_every_layers": 3,
                                       "entry": "sq_adjoint_grad_hea (the ansatz's own kernels)"}
        print(f"[bench] adjoint 24q: forward {f*1e3:.2f} ms, energy+gradient {gtime*1e3:.2f} ms",
              file=sys.stderr, flush=True)
        # The same ansatz as circuit text through the general entry point
        # (sq_adjoint_grad; CNOT as U2): its forward is the plain sweep's
        # register passes, against which the gradient is timed.
        atext = sq.gen_circuit("hea", an, al, theta=theta)
        alines = atext.strip().splitlines()
        aparam, k = [], 0
        for line in alines:
            if line.startswith(("RY", "RZ")):
                aparam.append(k)
                k += 1
            else:
                aparam.append(-1)
        aterms = [(1.0, [q, (q + 1) % an]) for q in range(an)]
        ea = sq.Engine(an, dtype="c64")
        agates, _, ang, _ = sq.parse_circuit(atext, an)
        ea.init_zero()
        ea.apply_gates(agates, ang)
        ea.adjoint_grad(atext, aparam, theta, aterms, 144)
        ea.sync()
        fwd, grd = [], []
        for _ in range(3):
            ea.init_zero()
            ea.sync()
            t0 = time.perf_counter()
            ea.apply_gates(agates, ang)
            e_fwd = ea.expect_z(aterms)
            fwd.append(time.perf_counter() - t0)
            ea.init_zero()
            ea.sync()
            t0 = time.perf_counter()
            e_g, g2 = ea.adjoint_grad(atext, aparam, theta, aterms, 144)
            grd.append(time.perf_counter() - t0)
        ea.close()
        f2, gt2 = min(fwd), min(grd)
        out["adjoint_general_24q_384p_c64"] = {
            "forward_ms": round(f2 * 1e3, 3), "energy_and_gradient_ms": round(gt2 * 1e3, 3),
            "gradient_over_forward": round(gt2 / f2, 3), "checkpoint_every_params": 144,
            "energy_diff_vs_forward": abs(e_g - e_fwd),
            "max_grad_diff_vs_hea_entry": float(np.max(np.abs(g2 - g))),
            "entry": "sq_adjoint_grad (circuit text, Z-string observable); forward = register passes"}
        print(f"[bench] adjoint (general) 24q: forward {f2*1e3:.2f} ms, energy+gradient {gt2*1e3:.2f} ms",
              file=sys.stderr, flush=True)

    if not args.no_cpu_baseline:
        print("[bench] cpu baseline", file=sys.stderr, flush=True)
        cb = cpu_baseline(text, n, args.cpu_sample_gates)
        out["cpu_baseline"] = cb
    else:
        out["cpu_baseline"] = None
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
