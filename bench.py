#!/usr/bin/env python3
"""Benchmark of the fp32 linear hot path on one MI355X.

Workload (the configuration the headline metric "linear
GEMM TFLOP/s" is quoted on): Y = X W^T + b, dX = dY W, dW = dY^T X, db for
M in {1, 64, 512, 4096} x (K -> N) in {768->2304, 768->3072, 3072->768,
896->4864, 4864->896}; X ~ N(0,1), W ~ N(0,1/K), b ~ N(0,0.02), dY ~ N(0,1).
One step = all 20 shapes x {forward, dX, dW with db} (60 library calls: dW
and db are requested by one linear_bwd call, as a layer's backward asks for
them, and for batches above 8 one GEMM launch computes both).  Every
(shape, M) owns its own buffers (~1.3 GB in total, far above the 256 MB
Infinity Cache), so each call starts cold, as the M=1 GEMV rule requires.

value = total GEMM FLOPs (2MNK per forward, dX and dW) / time of the K
timed steps, inputs resident in HBM; the timed region holds the K steps
between two HIP events on the library stream and nothing else.  A second
pass over the same K steps records an event after every call (each record
costs ~3.6 us of GPU time, ~0.3 ms per step, which is why it is kept out of
the headline region); it gives every call's and kernel's duration and the
roofline entry: the dominant kernel's average is taken over its launches
without a split-tile fixup, so the event-bracketed time is that kernel's own
duration plus one event record -- and, for the split_* kernels (operands as
fp16 pairs), plus the launch that packs both operands, which belongs to the
call.  The roofline kernel is the one with the most time in such launches; its
peak is the FP32 MFMA's, or for a split_* kernel a third of the FP16 MFMA's
(three products per FP32 product).  "dtype" is that of the operands, results
and sums; "operands" in the config says what the split_* kernels multiply.

The CPU baseline runs the reference's own CPU code (oracle/_ref/libref.so,
compiled from the reference sources) in a child process on a bounded sample
of the same workload.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--no-cpu]
"""
import argparse
import json
import os
import subprocess
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, os.path.join(ROOT, "saphira-cncm_amd"))

METRIC = "linear GEMM TFLOP/s (% FP32 MFMA peak); NCP fwd tokens/s; Qwen2-0.5B tok/s"
PEAK_TFLOPS = 157.3   # MI355X dense FP32 MFMA
PEAK_SPLIT_TFLOPS = 2500.0 / 3   # dense FP16 MFMA, three products per FP32 product (the split_* kernels)
PEAK_HBM_GBS = 8000.0
SHAPES = [(768, 2304), (768, 3072), (3072, 768), (896, 4864), (4864, 896)]  # (K, N)
MS = [1, 64, 512, 4096]
CPU_MS = [1, 64, 512]
# HBM bytes per launch of the roofline kernel are measured in each run by two
# rocprofv3 counter passes (FETCH_SIZE, then WRITE_SIZE) over a child process
# that repeats the roofline kernel's own launches (measure_traffic below).
TRAFFIC_REPS = 3


def build_workload(ncmhip, seed=0, only=None):
    """The sweep's 80 calls (or those whose label is in `only`), with their
    operands on the device: (kernel, flops, label, call, no fixup launch?)."""
    D = ncmhip.DeviceBuffer
    rng = np.random.default_rng(seed)
    calls = []
    keep = []
    for M in MS:
        for K, N in SHAPES:
            if only is not None and not any(l.endswith(f" M={M} {K}->{N}") for l in only):
                continue
            x = D.from_numpy(rng.standard_normal((M, K), dtype=np.float32))
            W = D.from_numpy((rng.standard_normal((N, K), dtype=np.float32) / np.float32(np.sqrt(K))))
            b = D.from_numpy((rng.standard_normal(N, dtype=np.float32) * np.float32(0.02)))
            dy = D.from_numpy(rng.standard_normal((M, N), dtype=np.float32))
            y, dx, dW, db = D.empty((M, N)), D.empty((M, K)), D.empty((N, K)), D.empty(N)
            for buf in (dx, dW, db):
                buf.upload(np.zeros(buf.shape, np.float32))
            keep += [x, W, b, dy, y, dx, dW, db]
            flops = 2.0 * M * N * K
            fwd_k, fwd_s = ncmhip.linear_route("fwd", M, N, K)
            dx_k, dx_s = ncmhip.linear_route("dx", M, N, K)
            dw_k, dw_s = ncmhip.linear_route("dwdb", M, N, K)
            # (kernel, flops, label, call, no fixup launch?)
            calls.append((fwd_k, flops, f"fwd M={M} {K}->{N}",
                          lambda x=x, W=W, b=b, y=y, M=M, N=N, K=K: ncmhip.linear_fwd(x, W, b, y, M, N, K),
                          fwd_s == 1))
            calls.append((dx_k, flops, f"dX M={M} {K}->{N}",
                          lambda x=x, W=W, dy=dy, dx=dx, M=M, N=N, K=K:
                          ncmhip.linear_bwd(x, W, dy, dx, None, None, M, N, K), dx_s == 1 and M > 8))
            # dW and db from one linear_bwd call (for batches above 8 one GEMM
            # launch sums both); a batch of at most 8 adds the column-sum launch
            calls.append((dw_k, flops, f"dW+db M={M} {K}->{N}",
                          lambda x=x, W=W, dy=dy, dW=dW, db=db, M=M, N=N, K=K:
                          ncmhip.linear_bwd(x, W, dy, None, dW, db, M, N, K), dw_s == 1 and M > 8))
    if only is not None:
        calls = [c for c in calls if c[2] in only]
    return calls, keep


def algo_bytes(labels):
    """Mean algorithmic HBM bytes per call over sweep labels ("fwd|dX|dW+db
    M=m k->n"): each operand read once, each output written once, and the
    accumulated gradients (dX, or dW and db) also read once."""
    tot = 0.0
    for lab in labels:
        op, m, kn = lab.split()
        M = int(m[2:])
        K, N = (int(v) for v in kn.split("->"))
        if op == "fwd":
            b = M * K + N * K + N + M * N
        elif op == "dX":
            b = M * N + N * K + 2 * M * K
        else:
            b = M * N + M * K + 2 * N * K + 2 * N
        tot += 4.0 * b
    return tot / len(labels)


def traffic_child(labels, reps):
    """Counter-pass child: three 256 MiB device copies (the known-size
    calibration) and `reps` rounds of the given sweep calls."""
    import ncmhip
    ncmhip.init(0)
    src, dst = ncmhip.DeviceBuffer(256 << 20), ncmhip.DeviceBuffer(256 << 20)
    for _ in range(3):
        ncmhip.load().mem_d2d(dst.ptr, src.ptr, 256 << 20)
    ncmhip.check()
    del src, dst
    calls, keep = build_workload(ncmhip, only=set(labels))
    for _ in range(reps):
        for c in calls:
            c[3]()
    ncmhip.sync()
    ncmhip.check()


def measure_traffic(kernel, labels, reps=TRAFFIC_REPS):
    """HBM bytes per launch of `kernel` over the sweep calls `labels`: one
    rocprofv3 --pmc pass per counter (FETCH_SIZE, WRITE_SIZE) of a child that
    repeats those calls, each counter scaled by what it reads for the child's
    256 MiB copies.  Returns (bytes or None, note)."""
    import csv
    import glob
    import shutil
    import tempfile
    prof = shutil.which("rocprofv3") or "/opt/rocm/bin/rocprofv3"
    if not os.path.exists(prof):
        return None, "rocprofv3 not found"
    total, parts = 0.0, []
    for ctr in ("FETCH_SIZE", "WRITE_SIZE"):
        d = tempfile.mkdtemp(prefix="ncm_traffic_", dir="/tmp")
        cmd = ["timeout", "-s", "KILL", "120", prof, "--pmc", ctr, "--output-format", "csv", "-d", d, "-o", "t",
               "--", sys.executable, os.path.abspath(__file__), "--traffic-child", ";".join(labels),
               "--traffic-reps", str(reps)]
        try:
            subprocess.run(cmd, check=True, capture_output=True, text=True, timeout=180, cwd="/tmp",
                           env=dict(os.environ, TMPDIR="/tmp"))
            files = glob.glob(os.path.join(d, "**", "*counter_collection.csv"), recursive=True)
            rows = [r for f in files for r in csv.DictReader(open(f))]
        except Exception as e:  # reported, never fatal for the GPU number
            return None, f"{ctr} pass failed: {e}"
        finally:
            shutil.rmtree(d, ignore_errors=True)
        cal = [float(r["Counter_Value"]) for r in rows
               if r["Kernel_Name"].startswith("__amd_rocclr_copyBuffer") and float(r["Counter_Value"]) > 1e5]
        vals = [float(r["Counter_Value"]) for r in rows if r["Kernel_Name"].split("(")[0].strip() == kernel]
        if not cal or not vals:
            return None, f"{ctr} pass: no calibration copies or no {kernel} dispatches in the counters"
        factor = (sum(cal) / len(cal)) / 262144.0          # counter KiB per KiB copied
        per = sum(vals) / len(vals) * 1024.0 / factor
        total += per
        parts.append(f"{ctr} {per / 1e6:.1f} MB (x{1 / factor:.3f}, {len(vals)} dispatches)")
    return total, "measured in this run: " + "; ".join(parts)


def timed(ncmhip, fn, reps, warm=1):
    """Runs fn warm times, then reps times between two HIP events on the
    library stream; returns ms per call."""
    for _ in range(warm):
        fn()
    ncmhip.sync()
    e0, e1 = ncmhip.Event(), ncmhip.Event()
    e0.record()
    for _ in range(reps):
        fn()
    e1.record()
    e1.synchronize()
    return e0.elapsed_ms(e1) / reps


EXTRAS = ("ncp_fwd", "vq_multiscale", "vq_full", "qwen", "gpt2_train")
QWEN_STEPS = 256   # greedy steps after the 2048-token prefill (config 4); --qwen-steps for profiling runs


def extras(ncmhip, only=EXTRAS):
    """The other BASELINE configurations, each at its full size, reported
    beside the headline (synthetic data, random-init weights); `only` picks
    a subset by name."""
    import ctypes
    D = ncmhip.DeviceBuffer
    lib = ncmhip.load()
    lib.arena_init(24 << 30)
    ncmhip.check()
    rng = np.random.default_rng(7)
    out = {}

    def normal(shape, std=0.02, mean=0.0):
        return D.from_numpy(rng.standard_normal(shape, dtype=np.float32) * np.float32(std) + np.float32(mean))

    def _ncp_fwd():
        # -- config 1: NCP forward, 64 boards x 81 tokens
        n_layer, C, H, Kv, I, V, B, S = 4, 256, 4, 2, 1024, 16, 64, 81
        cfg = ncmhip.NcpConfig(n_layer, C, H, Kv, I, V, 10000)
        shapes = [ncmhip_shape(lib.ncm_ncp_param_shape, cfg, i) for i in range(lib.ncm_ncp_param_count(ctypes.byref(cfg)))]
        bufs = [normal(sh, mean=1.0 if is_gain(i, len(shapes), 14, (0, 6), 4) else 0.0) for i, sh in enumerate(shapes)]
        ids = rng.integers(0, V, (B, S)).astype(np.int32)
        ptrs = ncmhip.ptr_array(bufs)
        ms = timed(ncmhip, lambda: lib.ncm_ncp_forward(ctypes.byref(cfg), ptrs, ids.ctypes.data, B, S), 20, 3)
        ncmhip.check()
        R, hd = B * S, C // H
        fl = n_layer * (2 * R * C * (C + 2 * Kv * hd) + 2 * R * C * C + 3 * 2 * R * C * I + 4 * B * H * S * S * hd) \
            + 2 * R * C * V
        out["ncp_fwd"] = {"config": "C1: 4 layers, d 256, 4/2 heads, SwiGLU 1024, vocab 16, 64 x 81 tokens; "
                                    "pre-LayerNorm eps 1e-6 as the reference's ncp_block (ncp.c:199, 277), which "
                                    "has no RMSNorm variant",
                          "tokens_per_s": round(R / (ms / 1e3), 1), "ms_per_forward": round(ms, 4),
                          "tflops": round(fl / (ms / 1e3) / 1e12, 3), "gflop": round(fl / 1e9, 3)}
        del bufs

    if "ncp_fwd" in only:
        _ncp_fwd()

    def _vq_multiscale():
        # -- config 3: VQ multiscale, 65536 x 256, 4 scales of 4096 codewords
        R3, D3, V3 = 65536, 256, 4096
        z = normal((R3, D3), std=1.0)
        Es = [normal((V3, D3), std=1.0 / 16) for _ in range(4)]
        idx, zh, zr = D.empty((1, 4 * R3), np.int32), D.empty((R3, D3)), D.empty((R3, D3))
        ms = timed(ncmhip, lambda: ncmhip.vq_quantize_multiscale(z, Es, [V3] * 4, 1, R3, D3, idx, zh, zr), 5, 1)
        fl = 4 * 2.0 * R3 * V3 * D3
        out["vq_multiscale"] = {"config": "C3: 65536 x 256, 4 scales x 4096 codewords",
                                "vectors_scales_per_s": round(4 * R3 / (ms / 1e3), 1), "ms": round(ms, 3),
                                "tflops": round(fl / (ms / 1e3) / 1e12, 3),
                                "frac_fp32_mfma_peak": round(fl / (ms / 1e3) / 1e12 / PEAK_TFLOPS, 4)}
        del z, Es, idx, zh, zr

    if "vq_multiscale" in only:
        _vq_multiscale()

    def _vq_full():
        # -- config 3 with the full quantizer of vq.c: the same 65536 x 256 vectors as
        # 4096 sequences over levels 1, 2, 4, 8, 16, 4096 codes per level, Phi
        # partially shared (4 convs, ratio 0.5); vq_load + vq_z_to_idx on the device
        Bq, levs, Vq, Dq = 4096, [1, 2, 4, 8, 16], 4096, 256
        wq = {}
        for i in range(5):
            wq[f"embeddings.{i}.weight"] = normal((Vq, Dq), std=1.0 / 16.0)
        for i in range(4):
            wq[f"quant_resi.{i}.weight"] = normal((Dq, Dq, 3), std=0.5 / np.sqrt(3 * Dq))
            wq[f"quant_resi.{i}.bias"] = normal((Dq,))
        items = (ncmhip.NamedTensor * len(wq))()
        tens = []
        for j, (k, buf) in enumerate(wq.items()):
            t = ncmhip.TensorS()
            t.data = buf.ptr
            for a, sdim in enumerate(buf.shape):
                t.shape[a] = sdim
            t.ndim, t.n = len(buf.shape), int(np.prod(buf.shape))
            tens.append(t)
            items[j].name = k.encode()
            items[j].t = ctypes.pointer(t)
        wsq = ncmhip.WeightStore(items, len(wq))
        cq = ncmhip.NCMConfig()
        cq.n_qlevels, cq.vq_embed_dim = 5, Dq
        for i, lv in enumerate(levs):
            cq.levels[i], cq.vq_vocab[i] = lv, Vq
        cq.quant_resi_enabled, cq.quant_resi_ratio, cq.quant_resi_share_mode = 1, 0.5, 4
        vq = lib.vq_load(ctypes.byref(cq), ctypes.byref(wsq), b"")
        ncmhip.check()
        zq = normal((Bq, 16, Dq), std=1.0)
        idxq = D.empty((Bq, sum(levs)), np.int32)
        ms_q = timed(ncmhip, lambda: lib.vq_z_to_idx_dev(vq, zq.ptr, Bq, idxq.ptr, None, None), 3, 1)
        ncmhip.check()
        lib.vq_free(vq)
        rows_q = Bq * sum(levs)
        fl_q = 2.0 * rows_q * Vq * Dq
        conv_fl = 5 * 2.0 * Bq * 16 * Dq * Dq * 3
        out["vq_full"] = {"config": "C3 vectors through the full quantizer: 4096 x 16 x 256, levels 1/2/4/8/16 (area "
                                    "down, linear up), 4096 codes per level, Phi 4 partially shared convs (fp64, "
                                    "ratio 0.5)",
                          "ms": round(ms_q, 3), "code_rows_per_s": round(rows_q / (ms_q / 1e3), 1),
                          "argmin_gflop": round(fl_q / 1e9, 1), "phi_conv_gflop_fp64": round(conv_fl / 1e9, 1)}
        del wq, items, tens, zq, idxq

    if "vq_full" in only:
        _vq_full()

    def _qwen():
        # -- config 4: Qwen2-0.5B shape, prefill 2048 then 256 greedy steps
        qc = ncmhip.QwenConfig(24, 896, 14, 2, 4864, 151936, 2304, 1e6)
        nq = lib.ncm_qwen_param_count(ctypes.byref(qc))
        shapes = [ncmhip_shape(lib.ncm_qwen_param_shape, qc, i) for i in range(nq)]
        bufs = [normal(sh, mean=1.0 if is_gain(i, nq, 12, (0, 8), 1, base=1) else 0.0) for i, sh in enumerate(shapes)]
        nparam = sum(int(np.prod(sh)) for sh in shapes)
        m = lib.ncm_qwen_new(ctypes.byref(qc), ncmhip.ptr_array(bufs))
        ncmhip.check()
        prompt = rng.integers(0, qc.vocab, 2048).astype(np.int32)
        n_new = QWEN_STEPS
        gen = np.zeros(n_new, np.int32)
        ms_pre = timed(ncmhip, lambda: lib.ncm_qwen_forward(m, prompt.ctypes.data, 2048, 1), 3, 1)
        ms_gen = timed(ncmhip, lambda: lib.ncm_qwen_generate(m, prompt.ctypes.data, 2048, n_new, -1, gen.ctypes.data),
                       2, 1)
        ncmhip.check()
        # the same 256 steps drawing from sample_topkp (temp 0.8, top-k 0, top-p 0.9) on the device
        st, nflag = ctypes.c_uint64(0x5EED), ctypes.c_int(0)
        ms_samp = timed(ncmhip, lambda: lib.ncm_qwen_generate_sample(m, prompt.ctypes.data, 2048, n_new, -1, 0.8, 0, 0.9,
                                                                     ctypes.byref(st), gen.ctypes.data,
                                                                     ctypes.byref(nflag)), 2, 1)
        ncmhip.check()
        # one draw of the sampler alone on a 151936-entry row
        row = D.from_numpy(rng.standard_normal(qc.vocab).astype(np.float32) * np.float32(3.0))
        srng, sout, sflag = D.from_numpy(np.array([7], np.uint64)), D.empty(1, np.int32), D.empty(1, np.int32)
        ms_draw = timed(ncmhip, lambda: lib.sample_topkp_dev(row.ptr, qc.vocab, 0.8, 0, 0.9, srng.ptr, sout.ptr,
                                                             sflag.ptr), 20, 2)
        ncmhip.check()
        del row, srng, sout, sflag
        ms_tok = (ms_gen - ms_pre) / (n_new - 1)
        kv_bytes = 2 * 24 * 2 * 64 * 4 * (2048 + 128)          # mean KV cache read per step
        dec_bytes = 4 * nparam + kv_bytes
        pre_fl = 2 * 2048 * (nparam - qc.vocab * 896) + 24 * 4 * 14 * 2048 * 2048 * 64 / 2 + 2 * 896 * qc.vocab
        lib.ncm_qwen_free(m)
        out["qwen"] = {"config": "C4: 24 layers, d 896, 14/2 heads, FFN 4864, vocab 151936; prefill 2048, "
                                 f"{n_new} greedy steps (KV cache, device argmax, no eos stop)",
                       "prefill_tok_per_s": round(2048 / (ms_pre / 1e3), 1), "prefill_ms": round(ms_pre, 3),
                       "prefill_tflops": round(pre_fl / (ms_pre / 1e3) / 1e12, 3),
                       "decode_tok_per_s": round(1e3 / ms_tok, 1), "decode_ms_per_tok": round(ms_tok, 4),
                       "decode_gbs": round(dec_bytes / (ms_tok / 1e3) / 1e9, 1),
                       "decode_frac_hbm": round(dec_bytes / (ms_tok / 1e3) / 1e9 / PEAK_HBM_GBS, 4),
                       "generate_ms": round(ms_gen, 2),
                       "sampled_decode_tok_per_s": round((n_new - 1) / ((ms_samp - ms_pre) / 1e3), 1),
                       "sampled_flagged_draws": nflag.value,
                       "sample_draw_us": round(ms_draw * 1e3, 2)}
        del bufs

    if "qwen" in only:
        _qwen()

    def _gpt2_train():
        # -- config 5: GPT-style training step, 12 layers, d 768, 32 x 512 tokens
        gc = ncmhip.Gpt2Config(12, 768, 12, 4096, 512)
        ng = lib.ncm_gpt2_param_count(ctypes.byref(gc))
        shapes = [ncmhip_shape(lib.ncm_gpt2_param_shape, gc, i) for i in range(ng)]
        P = [normal(sh, mean=1.0 if is_gain(i, ng, 12, (0, 6), 2, base=2) else 0.0) for i, sh in enumerate(shapes)]
        G, M, Vm = ([D.from_numpy(np.zeros(sh, np.float32)) for sh in shapes] for _ in range(3))
        xin = rng.integers(0, 4096, (32, 512)).astype(np.int32)
        xout = rng.integers(0, 4096, (32, 512)).astype(np.int32)
        tape = lib.ncm_tape_new()
        gn = ctypes.c_double()
        pp, gp, mp, vp_ = (ncmhip.ptr_array(x) for x in (P, G, M, Vm))
        step = [0]

        def train_step():
            step[0] += 1
            lib.ncm_gpt2_train_step(tape, ctypes.byref(gc), pp, gp, mp, vp_, xin.ctypes.data, xout.ctypes.data, 32, 512,
                                    step[0], 3e-4, 100.0, 1000.0, 0.1, ctypes.byref(gn))

        ms = timed(ncmhip, train_step, 3, 1)
        ncmhip.check()
        lib.ncm_tape_free(tape)
        R5, C5 = 32 * 512, 768
        nblock = sum(int(np.prod(sh)) for sh in shapes[2:-2] if len(sh) == 2)
        fl = 3 * (2 * R5 * nblock + 2 * R5 * C5 * 4096) + 12 * 12 * 32 * (4 + 8) * 512 * 512 * 64
        out["gpt2_train"] = {"config": "C5: 12 layers, d 768, 12 heads, GELU 3072, LayerNorm, vocab 4096, "
                                       "32 x 512 tokens; forward + CE + tape backward + clip + AdamW",
                             "ms_per_step": round(ms, 2), "tokens_per_s": round(R5 / (ms / 1e3), 1),
                             "tflops": round(fl / (ms / 1e3) / 1e12, 3), "tflop_per_step": round(fl / 1e12, 3)}

    if "gpt2_train" in only:
        _gpt2_train()

    return out


def ncmhip_shape(fn, cfg, i):
    import ctypes
    r, c = ctypes.c_int64(), ctypes.c_int64()
    fn(ctypes.byref(cfg), i, ctypes.byref(r), ctypes.byref(c))
    return (r.value, c.value) if c.value > 1 else (r.value,)


def is_gain(i, n, per, slots, tail, base=1):
    """True for the norm gains of a flat parameter list (per-layer slots, or
    the final norm weight `tail` entries from the end)."""
    if i == n - tail:
        return True
    return base <= i < n - tail and (i - base) % per in slots


def cpu_baseline_child():
    """Runs in a child process: the reference CPU path on bounded samples of
    the headline workload (config 2) and of configs 1, 3, 4 and 5."""
    sys.path.insert(0, os.path.join(ROOT, "oracle"))
    import oracle as O
    rng = np.random.default_rng(1)
    kind = "reference" if O.ref_available() else "port"
    threads = int(os.environ.get("OMP_NUM_THREADS", os.cpu_count() or 1))
    flops, secs = 0.0, 0.0
    for M in CPU_MS:
        for K, N in SHAPES:
            x = rng.standard_normal((M, K), dtype=np.float32)
            W = rng.standard_normal((N, K), dtype=np.float32) / np.float32(np.sqrt(K))
            b = rng.standard_normal(N, dtype=np.float32) * np.float32(0.02)
            dy = rng.standard_normal((M, N), dtype=np.float32)
            t0 = time.perf_counter()
            if kind == "reference":
                # t_linear forward + tape host backward (dX, dW, db)
                O.ref_linear_bwd(x, W, b, dy)
            else:
                O.linear_fwd(x, W, b)
                O.linear_bwd(x, W, dy)
            secs += time.perf_counter() - t0
            flops += 3 * 2.0 * M * N * K
    res = {"value": flops / secs / 1e12, "unit": "TFLOP/s", "cores": threads, "kind": kind,
           "seconds": round(secs, 3),
           "threads": f"OMP_NUM_THREADS={threads}, OMP_PROC_BIND={os.environ.get('OMP_PROC_BIND')}, "
                      f"OMP_PLACES={os.environ.get('OMP_PLACES')}",
           "sample": "linear sweep fwd+dX+dW+db at M in {1,64,512} x the 5 (K->N) shapes "
                     "(the M=4096 rows are left out to bound CPU time); "
                     + ("reference src/kernels.c linear_fwd + train_tape.c TOP_LINEAR host "
                        "backward, gcc -O2 -fopenmp" if kind == "reference"
                        else "oracle C restatement")}
    if kind == "reference":
        res["configs"] = cpu_configs(O, threads)
    print(json.dumps(res))


def cpu_configs(O, threads):
    """The reference's own CPU code (oracle/_ref/libref.so) on bounded samples
    of configs 1, 3, 4 and 5; each entry says what was timed."""
    import tempfile
    rng = np.random.default_rng(2)
    out = {}

    def normal(shape, std=0.02, mean=0.0):
        return (rng.standard_normal(shape, dtype=np.float32) * np.float32(std) + np.float32(mean)).astype(np.float32)

    # config 1: the reference's ncp_load + ncp_forward (ncp.c:94-175, 480-640) at full size
    n_layer, C, H, Kv, I, V, B, S = 4, 256, 4, 2, 1024, 16, 64, 81
    shapes = O.ncp_shapes(n_layer, C, H, Kv, I, V)
    params = [normal(sh, mean=1.0 if is_gain(i, len(shapes), 14, (0, 6), 4) else 0.0) for i, sh in enumerate(shapes)]
    ids = rng.integers(0, V, (B, S)).astype(np.int32)
    x = np.eye(V, dtype=np.float32)[ids]
    named = O.ncp_named(params, n_layer, C)
    cfg = O.ncp_single_level_cfg(n_layer, C, H, Kv, V, S)
    reps = 3
    t0 = time.perf_counter()
    for _ in range(reps):
        O.ref_ncp_forward(cfg, named, x)
    t = (time.perf_counter() - t0) / reps
    out["C1_ncp_fwd"] = {"value": round(B * S / t, 1), "unit": "tokens/s", "cores": threads, "kind": "reference",
                         "seconds": round(t * reps, 3),
                         "sample": "full config 1 (64 x 81 tokens, 4 layers, d 256), 3 forwards through the "
                                   "reference's ncp_load + ncp_forward on one-hot inputs (one level, no prefix)"}

    # config 3: one of the 4 scales of vq_z_to_idx (rowwise_l2sq + host argmin + residual,
    # vq.c:388-500) on all 65536 rows
    rows, D3, V3 = 65536, 256, 4096
    z = normal((rows, D3), std=1.0)
    E = normal((V3, D3), std=1.0 / 16)
    t0 = time.perf_counter()
    O.ref_vq_multiscale(z, [E], 1, rows)
    t = time.perf_counter() - t0
    out["C3_vq"] = {"value": round(rows / t, 1), "unit": "vectors*scales/s", "cores": threads, "kind": "reference",
                    "seconds": round(t, 3), "tflops": round(2.0 * rows * V3 * D3 / t / 1e12, 5),
                    "sample": "one of the 4 scales on all 65536 rows x 4096 codewords x 256: the reference's "
                              "vq_z_to_idx with the materialised 1 GiB distance matrix and host argmin"}

    # config 4: the reference's qwen_forward (qwen.c:121-190) at full model size on a 128-token prompt,
    # and one full-recompute greedy step at that context (qwen_generate, qwen.c:204-228)
    qcfg = dict(n_layer=24, C=896, H=14, K=2, I=4864, V=151936)
    qshapes = O.qwen_shapes(**qcfg)
    qp = [normal(sh, mean=1.0 if is_gain(i, len(qshapes), 12, (0, 8), 1, base=1) else 0.0)
          for i, sh in enumerate(qshapes)]
    T4 = 128
    prompt = rng.integers(0, qcfg["V"], T4).astype(np.int32)
    with tempfile.TemporaryDirectory() as td:
        m = O.RefQwen(qp, qcfg["n_layer"], qcfg["C"], qcfg["H"], qcfg["K"], T4 + 8, 1e6, os.path.join(td, "q.ncm"))
        try:
            t0 = time.perf_counter()
            m.forward(prompt, last_only=True)
            t_pre = time.perf_counter() - t0
            t0 = time.perf_counter()
            m.generate(prompt, 2)
            t_gen = time.perf_counter() - t0
        finally:
            m.close()
    out["C4_qwen"] = {"value": round(T4 / t_pre, 2), "unit": "prefill tokens/s", "cores": threads,
                      "kind": "reference", "seconds": round(t_pre + t_gen, 3),
                      "decode_tok_per_s_at_context_128": round(2 / t_gen, 3),
                      "sample": "full config-4 model (24 layers, d 896, vocab 151936) through the reference's "
                                "qwen_forward on a 128-token prompt (not 2048), then 2 greedy steps of its "
                                "qwen_generate, which recomputes the whole context every step (no KV cache)"}
    del qp

    # config 5: the reference's taped GPT-2 step (train_gpt2.c:42-147 + t_ce + tape_backward_host)
    # for 1 of the 12 layers and 2 of the 32 sequences of 512
    L5, C5, H5, V5, T5, B5 = 1, 768, 12, 4096, 512, 2
    gshapes = O.gpt2_shapes(L5, C5, V5, T5)
    gp = [normal(sh) for sh in gshapes]
    for i, sh in enumerate(gshapes):
        if len(sh) == 1 and sh[0] == C5 and (i >= len(gp) - 2 or (i - 2) % 12 in (0, 6)):
            gp[i] += np.float32(1.0)
    gi = rng.integers(0, V5, (B5, T5)).astype(np.int32)
    go = rng.integers(0, V5, (B5, T5)).astype(np.int32)
    t0 = time.perf_counter()
    O.ref_gpt2_grads(gp, L5, C5, H5, V5, T5, gi, go)
    t = time.perf_counter() - t0
    R5 = B5 * T5
    fl = 3 * (2 * R5 * 12 * C5 * C5 + 2 * R5 * C5 * V5) + 12 * B5 * (4 + 8) * T5 * T5 * 64
    out["C5_train"] = {"value": round(R5 / t, 1), "unit": "tokens/s", "cores": threads, "kind": "reference",
                       "seconds": round(t, 3), "tflops": round(fl / t / 1e12, 5),
                       "est_full_step_s": round(t * 12 * 16, 1),
                       "sample": "forward + CE + host tape backward of 1 layer (of 12) on 2 x 512 tokens "
                                 "(of 32 x 512) through the reference's train_gpt2_forward, t_ce and "
                                 "tape_backward_host; est_full_step_s scales by 12 layers x 16 batches"}
    return out


def run_cpu_baseline():
    try:
        env = dict(os.environ, OMP_PROC_BIND="close", OMP_PLACES="cores")
        out = subprocess.run([sys.executable, os.path.abspath(__file__), "--cpu-baseline-child"],
                             check=True, capture_output=True, text=True, timeout=900, env=env).stdout
        return json.loads(out.strip().splitlines()[-1])
    except Exception as e:  # reported, never fatal for the GPU number
        return {"value": None, "unit": "TFLOP/s", "cores": None, "kind": None, "sample": f"failed: {e}"}


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=30)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--no-cpu", action="store_true")
    ap.add_argument("--no-extras", action="store_true", help="skip configs 1, 3, 4, 5")
    ap.add_argument("--extras", default=",".join(EXTRAS),
                    help="comma-separated subset of the extra configurations to run (default: all of "
                         + ", ".join(EXTRAS) + ")")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="also run 3 device-to-device copies of 256 MiB (the known-size kernel the HBM "
                         "counters of a rocprofv3 --pmc run are scaled by)")
    ap.add_argument("--qwen-steps", type=int, default=256,
                    help="decode steps of config 4 (256; fewer only to keep profiler runs short)")
    ap.add_argument("--cpu-baseline-child", action="store_true")
    ap.add_argument("--no-traffic", action="store_true",
                    help="skip the two rocprofv3 counter passes that measure roofline.traffic")
    ap.add_argument("--traffic-child", default=None, help=argparse.SUPPRESS)
    ap.add_argument("--traffic-reps", type=int, default=TRAFFIC_REPS, help=argparse.SUPPRESS)
    args = ap.parse_args()
    if args.cpu_baseline_child:
        cpu_baseline_child()
        return
    if args.traffic_child is not None:
        traffic_child(args.traffic_child.split(";"), args.traffic_reps)
        return
    global QWEN_STEPS
    QWEN_STEPS = max(2, args.qwen_steps)
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(f"bench.py: this build measures one MI355X only (asked for --gpus {args.gpus}, "
              f"WORLD_SIZE {world}); the multi-GPU sharding is a design note, not a measured path",
              file=sys.stderr)
        sys.exit(2)

    import ncmhip
    ncmhip.init(0)
    if args.copy_calibration:
        src, dst = ncmhip.DeviceBuffer(256 << 20), ncmhip.DeviceBuffer(256 << 20)
        for _ in range(3):
            ncmhip.load().mem_d2d(dst.ptr, src.ptr, 256 << 20)
        ncmhip.check()
        del src, dst
    calls, keep = build_workload(ncmhip)
    ncmhip.sync()
    for _ in range(args.warmup):
        for c in calls:
            c[3]()
    ncmhip.sync()

    n = len(calls)
    # timed region: the K steps between two events, nothing else on the stream
    h0, h1 = ncmhip.Event(), ncmhip.Event()
    ncmhip.sync()
    t0 = time.perf_counter()
    h0.record()
    for _ in range(args.steps):
        for c in calls:
            c[3]()
    h1.record()
    h1.synchronize()
    ncmhip.sync()
    wall = time.perf_counter() - t0
    gpu_ms = h0.elapsed_ms(h1)

    # instrumented pass: the same K steps with an event after every call
    evs = [ncmhip.Event() for _ in range(n * args.steps + 1)]
    ncmhip.sync()
    evs[0].record()
    e = 1
    for _ in range(args.steps):
        for c in calls:
            c[3]()
            evs[e].record()
            e += 1
    evs[-1].synchronize()
    ncmhip.sync()
    inst_ms = evs[0].elapsed_ms(evs[-1])

    per_kernel = {}
    solo = {}
    per_call = {}
    for s in range(args.steps):
        for i, (kname, flops, label, _, alone) in enumerate(calls):
            j = s * n + i
            ms = evs[j].elapsed_ms(evs[j + 1])
            k = per_kernel.setdefault(kname, [0.0, 0.0, 0])
            k[0] += ms
            k[1] += flops
            k[2] += 1
            if alone:
                k = solo.setdefault(kname, [0.0, 0.0, 0, set()])
                k[0] += ms
                k[1] += flops
                k[2] += 1
                k[3].add(label)
            pc = per_call.setdefault(label, [0.0, flops, kname])
            pc[0] += ms / args.steps
    total_flops = sum(c[1] for c in calls) * args.steps
    t = max(gpu_ms / 1e3, 1e-12)
    value = total_flops / t / 1e12
    # roofline kernel: the one with the most time in calls without a fixup
    # launch in the event bracket (a split_* call's bracket holds its packing)
    dom = max((k for k in solo if solo[k][1] > 0), key=lambda k: solo[k][0])
    dms, dfl, dn, dlabels = solo[dom]
    achieved = dfl / (dms / 1e3) / 1e12
    # the kernel with the most time over every call whose main launch it is
    # (fixup launches included)
    top = max((k for k in per_kernel if per_kernel[k][1] > 0), key=lambda k: per_kernel[k][0])
    tms, tfl, tn = per_kernel[top]
    peak = PEAK_SPLIT_TFLOPS if dom.startswith("split_") else PEAK_TFLOPS
    tpeak = PEAK_SPLIT_TFLOPS if top.startswith("split_") else PEAK_TFLOPS
    traffic, traffic_note = (None, "skipped (--no-traffic)") if args.no_traffic else \
        measure_traffic(dom, sorted(dlabels))

    result = {
        "metric": METRIC,
        "value": round(value, 3),
        "unit": "TFLOP/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(gpu_ms / args.steps, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic",
        "config": {"workload": "BASELINE config 2: fp32 linear sweep, fwd + dX + dW + db, "
                               "M in {1,64,512,4096} x 5 (K->N) shapes",
                   "operands": "fp32; split_* kernels hold each value as two fp16 numbers (23 of its 24 bits) and "
                               "sum three fp16 products in fp32",
                   "calls_per_step": n, "gflop_per_step": round(total_flops / args.steps / 1e9, 3),
                   "frac_fp32_mfma_peak": round(value / PEAK_TFLOPS, 4),
                   "wall_s": round(wall, 4),
                   "ms_per_step_instrumented": round(inst_ms / args.steps, 4)},
        "roofline": {"bound": "mfma", "kernel": dom, "achieved": round(achieved, 3),
                     "peak": round(peak, 1), "unit": "TFLOP/s", "frac": round(achieved / peak, 4),
                     "avg_launch_us": round(dms / dn * 1e3, 3), "launches_per_step": dn // args.steps,
                     "launches": sorted(dlabels),
                     "traffic": None if traffic is None else round(traffic), "traffic_note": traffic_note,
                     "traffic_over_algorithmic": None if traffic is None else
                     round(traffic / algo_bytes(dlabels), 3),
                     "all_launches": {"kernel": top, "achieved": round(tfl / (tms / 1e3) / 1e12, 3),
                                      "frac": round(tfl / (tms / 1e3) / 1e12 / tpeak, 4),
                                      "calls_per_step": tn // args.steps}},
        "kernels": {k: {"ms_per_step": round(v[0] / args.steps, 4),
                        "tflops": round(v[1] / (v[0] / 1e3) / 1e12, 3) if v[1] else None}
                    for k, v in sorted(per_kernel.items(), key=lambda kv: -kv[1][0])},
        "calls_us": {k: [round(v[0] * 1e3, 2), round(v[1] / (v[0] / 1e3) / 1e12, 2) if v[1] else None, v[2]]
                     for k, v in per_call.items()},
    }
    if not args.no_extras:
        result["extras"] = extras(ncmhip, tuple(e for e in args.extras.split(",") if e))
    if not args.no_cpu:
        result["cpu_baseline"] = run_cpu_baseline()
    print(json.dumps(result))


if __name__ == "__main__":
    main()
