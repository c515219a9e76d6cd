#!/usr/bin/env python3
"""Benchmark of the XAttention prefill path on one MI355X.

    python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload 2]

A step is one pass of the hot path - antidiagonal estimate, block selection,
block-sparse attention - over one synthetic single-layer workload whose q/k/v
already sit in HBM.  The default workload is the headline one (L=131072,
32 query / 8 KV heads, d=128, stride 16, tau 0.9, chunk 16384, causal, bf16).
Prints ONE JSON line: the per-layer time (estimate + select + sparse attention;
mean, median and minimum over the timed steps), the speedup over this
library's own dense FlashAttention, the roofline of the longer of the two MFMA
kernels (the estimator's GEMM at the headline) and of the other one, the same
measurements for the other GPU workloads, two library yardsticks (a bf16 GEMM
of the estimator's shape, a causal flash attention) and a CPU baseline (the
torch restatement of the reference path on workload 0).

Timing protocol (the reference's eval/efficiency/attention_speedup.py:82-132
uses 30 warm-ups and 50 timed runs): W untimed warm-up steps, then K timed steps
with HIP events on the launch stream between the stages of every step; the dense
baseline gets its own warm-ups and timed launches.
"""
import argparse
import hashlib
import json
import os
import statistics
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
for _p in (ROOT, os.path.join(ROOT, "x-attention_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

PEAK_BF16_TFLOPS = 2500.0   # MI355X dense bf16 MFMA
PEAK_HBM_GBS = 8000.0
# HBM-side bytes per launch come from the FETCH_SIZE / WRITE_SIZE counter runs (counters cannot be read from inside
# this process): the summary of those runs for the headline workload is kept as a table under profiles/ and read here.
TRAFFIC_SUMMARY = os.path.join(ROOT, "profiles", "bench_headline_hbm_traffic.md")
HEADLINE = "cfg2_llama8b_L131072_gqa32x8_S16"
KERNEL_SOURCES = ("attn_plan.h", "attn_rows32.h", "attn_rows64.h", "attn_tiles.h", "attn_unit.h", "block_sparse_attn.hip", "estimate.h",
                  "estimate.hip", "estimate_params.h", "estimate_small.h", "select_row.h", "select_blocks.hip", "xattn_common.h")


def kernel_source_hash():
    """sha256 (16 hex digits) over the sources of the measured kernels.  The counter summary under profiles/
    names the hash it was taken at; a summary taken at other sources is not quoted."""
    h = hashlib.sha256()
    for name in KERNEL_SOURCES:
        with open(os.path.join(ROOT, "x-attention_amd", "csrc", name), "rb") as f:
            h.update(f.read())
    return h.hexdigest()[:16]


def measured_traffic_bytes(*kernel_prefixes):
    """Scaled total bytes of the traffic summary's rows for these kernels, added up: of each the first row whose
    kernel name starts with the prefix (last column, in GB).  None when the summary or a row is missing, or when
    the summary was taken at other kernel sources than the ones in the tree."""
    try:
        with open(TRAFFIC_SUMMARY) as f:
            text = f.read()
    except OSError:
        return None
    if ("kernel sources sha256/16: " + kernel_source_hash()) not in text:
        return None
    rows = [[c.strip().strip("`") for c in line.strip().strip("|").split("|")] for line in text.splitlines()]
    total = 0.0
    for prefix in kernel_prefixes:
        row = next((cells for cells in rows if len(cells) >= 6 and cells[0].startswith(prefix)), None)
        try:
            total += float(row[-1]) * 1e9
        except (TypeError, ValueError):
            return None
    return total


def _ms(a, b):
    return a.elapsed_time(b)


def _stats(xs):
    return {"mean": round(statistics.mean(xs), 4), "median": round(statistics.median(xs), 4), "min": round(min(xs), 4)}


def cpu_baseline(reps=5, warmup=2):
    """Times the oracle (torch restatement of the reference's torch path) on the
    host cores: workload 0 exactly (fp32, L=4096, 32 heads, stride 8, chunk 2048)."""
    import torch

    from oracle import xattn_oracle as O
    from xattn.synthetic import WORKLOADS, make_inputs

    w = WORKLOADS[0]
    cores = os.cpu_count() or 1
    threads = min(cores, int(os.environ.get("OMP_NUM_THREADS", cores)))
    torch.set_num_threads(threads)
    q, k, v = make_inputs(w, device="cpu", seed=0)
    t_est, t_att = [], []
    mask = None
    with torch.no_grad():
        for i in range(warmup + reps):
            t0 = time.perf_counter()
            _, mask = O.xattn_estimate(q, k, 128, w.stride, threshold=w.threshold, chunk_size=w.chunk_size, causal=True)
            t1 = time.perf_counter()
            O.block_sparse_attention(q, k, v, mask, causal=True)
            t2 = time.perf_counter()
            if i >= warmup:
                t_est.append((t1 - t0) * 1e3)
                t_att.append((t2 - t1) * 1e3)
    est, att = statistics.median(t_est), statistics.median(t_att)
    with torch.no_grad():
        # the other setting of the torch-branch slice quirk (keys of earlier chunks visible), for the record
        _, mask_all_keys = O.xattn_estimate(q, k, 128, w.stride, threshold=w.threshold, chunk_size=w.chunk_size,
                                            causal=True, pad0_quirk=False)
        torch.set_num_threads(1)
        t0 = time.perf_counter()
        _, m1 = O.xattn_estimate(q, k, 128, w.stride, threshold=w.threshold, chunk_size=w.chunk_size, causal=True)
        O.block_sparse_attention(q, k, v, m1, causal=True)
        single = (time.perf_counter() - t0) * 1e3
        torch.set_num_threads(threads)
    with torch.no_grad():
        # for the GPU-vs-oracle mask comparison below: the oracle on the very bf16 values the GPU path reads
        qb, kb = q.bfloat16().float(), k.bfloat16().float()
        bf16_sums, bf16_mask = O.xattn_estimate(qb, kb, 128, w.stride, threshold=w.threshold, chunk_size=w.chunk_size,
                                                causal=True)
    return {
        "value": round(est + att, 3),
        "unit": "ms per layer",
        "cores": threads,
        "kind": "port",
        "sample": (
            "workload 0 (fp32, L=4096, 32 heads, stride 8, tau 0.9, chunk 2048, causal): oracle xattn_estimate "
            f"+ dense masked softmax attention, median of {reps} after {warmup} warm-ups; the headline L=131072 "
            "does not finish on a CPU in bounded time"
        ),
        "estimate_ms": round(est, 3),
        "attention_ms": round(att, 3),
        "torch_threads": torch.get_num_threads(),
        "os_cpu_count": cores,
        "torch": torch.__version__,
        "single_thread_ms": round(single, 1),
        "mask_density": round(float(mask.float().mean()), 4),
        "mask_density_all_earlier_keys_visible": round(float(mask_all_keys.float().mean()), 4),
    }, (q, k, v, bf16_sums, bf16_mask)


def decode_leg(q, k, v, reps=50):
    """One decode step (the token after the prefill) over the workload's KV cache.

    Not part of the headline value: its own object on the line, with the HBM
    roofline that bounds it (the step reads K and V once: 2 * H_kv * L * 256 bytes).
    """
    import torch
    from xattn.src import hip_backend
    from xattn.src.decode import single_decode_with_kv_cache

    lib = hip_backend.lib()
    heads, kv_heads, L = q.shape[1], k.shape[1], k.shape[2]
    q1 = q[0, :, -1].contiguous()
    ws = torch.empty(lib.xattn_decode_workspace_bytes(heads, kv_heads, L), dtype=torch.uint8, device=q.device)
    out = torch.empty(heads, 128, dtype=q.dtype, device=q.device)
    for _ in range(5):
        single_decode_with_kv_cache(q1, k[0], v[0], kv_layout="HND", out=out, workspace=ws)
    torch.cuda.synchronize()
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record()
    for _ in range(reps):
        single_decode_with_kv_cache(q1, k[0], v[0], kv_layout="HND", out=out, workspace=ws)
    e1.record()
    torch.cuda.synchronize()
    us = _ms(e0, e1) * 1e3 / reps
    nbytes = 2.0 * kv_heads * L * 256
    tbs = nbytes / (us * 1e-6) / 1e12
    return {
        "kernels": "decode_partial_kernel + decode_merge_kernel",
        "kv_len": L, "us_per_step": round(us, 1), "bytes": nbytes,
        "roofline": {"bound": "hbm", "achieved": round(tbs * 1e3, 1), "peak": PEAK_HBM_GBS, "unit": "GB/s",
                     "frac": round(tbs * 1e3 / PEAK_HBM_GBS, 4)},
    }


def mfma_probe(dev):
    """What a stream of bf16 MFMAs sustains on this part: alone, and with the vector-ALU load of an attention
    tile (one exponential and three fmas per MFMA, no dependences, no memory) issued beside it; each with constant
    operand bits and with random ones (the clock the part holds depends on the switching activity of the operands)."""
    import ctypes

    import torch
    from xattn.src import hip_backend

    lib = hip_backend.lib()
    sink = torch.zeros(1, dtype=torch.float32, device=dev)
    res = {}
    gen = torch.Generator(device="cpu").manual_seed(0)
    tables = {
        "constant_operands": torch.full((4096 * 8,), 0.5, dtype=torch.bfloat16),
        "random_operands": torch.randn(4096 * 8, generator=gen).bfloat16(),
    }
    for name, host in tables.items():
        bits = host.to(dev)
        for mix, suffix in ((0, ""), (1, "_with_softmax_valu_mix")):
            flops = ctypes.c_double(0.0)
            stream = torch.cuda.current_stream().cuda_stream
            hip_backend.check(lib.xattn_mfma_rate_probe(bits.data_ptr(), 20000, mix, sink.data_ptr(), ctypes.byref(flops), stream), "probe")
            torch.cuda.synchronize()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            hip_backend.check(lib.xattn_mfma_rate_probe(bits.data_ptr(), 100000, mix, sink.data_ptr(), ctypes.byref(flops), stream), "probe")
            e1.record()
            torch.cuda.synchronize()
            res[name + suffix + "_tflops"] = round(flops.value / (_ms(e0, e1) * 1e-3) / 1e12, 1)
    return res


def flops_and_bytes(w, L, chunk, n_sel):
    """Algorithmic work of the three stages for a workload of length L."""
    H = w.heads
    nb = (L + 127) // 128
    Lp = (L + chunk - 1) // chunk * chunk
    n_r = Lp // w.stride
    nkb_p = Lp // 128
    rbs = 128 // w.stride
    causal = w.causal
    full_blocks = H * nb * (nb + 1) // 2 if causal else H * nb * nb
    f_est = (2.0 * w.stride * 128 * H * n_r * (n_r + 1) / 2) if causal else (2.0 * w.stride * 128 * H * n_r * n_r)
    f_dense = (4.0 * 128 * H * L * (L + 1) / 2) if causal else (4.0 * 128 * H * L * L)
    f_sparse = 4.0 * 128 ** 3 * n_sel
    # what the normalise-and-select pass moves: the visible part of the partial block sums (fp32 [H][Nk_p][n_r])
    # and of the tile statistics (two fp32 [H][n_r/128][n_r]) in, the column lists and counts out
    vis = 0.5 if causal else 1.0
    pass_bytes = 4.0 * H * n_r * nkb_p * vis + 2 * 4.0 * H * n_r * (n_r / 128.0) * vis + 4.0 * (n_sel + H * nkb_p)
    # the selection as the reference stages it: the full block-sum matrix in, a byte mask and the lists out
    staging_bytes = H * nkb_p * nkb_p * 5 + 4.0 * (n_sel + H * nkb_p)
    return dict(full_blocks=full_blocks, f_est=f_est, f_dense=f_dense, f_sparse=f_sparse, pass_bytes=pass_bytes,
                staging_bytes=staging_bytes, rbs=rbs)


def measure(w, q, k, v, L, tau, chunk, steps, warmup, dense_steps, dense_warmup):
    """Times `steps` passes of estimate -> select -> sparse attention (what the operator runs: column lists only,
    block sums kept in LDS) after `warmup` untimed ones, and the dense baseline.  Returns per-stage statistics."""
    import torch
    from xattn.src.Xattention import block_sparse_attention, estimate_and_select

    def step(marks):
        r = estimate_and_select(q, k, w.stride, tau, chunk, causal=w.causal, marks=marks, want_mask=False,
                                want_sums=False)
        out = block_sparse_attention(q, k, v, r["col_idx"], r["col_cnt"], causal=w.causal)
        if marks is not None:
            ev = torch.cuda.Event(enable_timing=True)
            ev.record()
            marks.append(("sparse_end", ev))
        return r, out

    with torch.no_grad():
        for _ in range(warmup):
            r, out = step(None)
        torch.cuda.synchronize()
        all_marks = []
        t0 = time.perf_counter()
        for _ in range(steps):
            m = []
            r, out = step(m)
            all_marks.append(dict(m))
        torch.cuda.synchronize()
        wall_ms = (time.perf_counter() - t0) * 1e3 / steps
        est = [_ms(m["estimate_begin"], m["select_begin"]) for m in all_marks]
        sel = [_ms(m["select_begin"], m["select_end"]) for m in all_marks]
        att = [_ms(m["select_end"], m["sparse_end"]) for m in all_marks]
        tot = [_ms(m["estimate_begin"], m["sparse_end"]) for m in all_marks]
        del out
        # dense FlashAttention written the same way (same kernel, every visible block)
        for _ in range(dense_warmup):
            block_sparse_attention(q, k, v, causal=w.causal)
        torch.cuda.synchronize()
        dense = []
        for _ in range(dense_steps):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            block_sparse_attention(q, k, v, causal=w.causal)
            e1.record()
            torch.cuda.synchronize()
            dense.append(_ms(e0, e1))
    nb = (L + 127) // 128
    n_sel = int(r["col_cnt"][:, :nb].sum().item())
    return dict(est=est, sel=sel, att=att, tot=tot, dense=dense, wall_ms=wall_ms, n_sel=n_sel, col_cnt=r["col_cnt"])


def mask_parity(w, q, k, tau, chunk, col_cnt):
    """Block-mask parity with the oracle (fp32, on the same bf16 values) for the query heads with the fewest and
    the most kept blocks: mismatches, and how many of them the contract allows (within 1e-5 of tau, or runs of
    equal sums cut by the crossing).  The mask compared is the product path's (normalise-and-select pass)."""
    from oracle.parity import head_mask_parity
    from xattn.src.Xattention import estimate_and_select

    kept = col_cnt.long().sum(-1)
    heads = sorted({int(kept.argmin()), int(kept.argmax())})
    r = estimate_and_select(q, k, w.stride, tau, chunk, causal=w.causal, want_lists=False, want_sums=False)
    tot = {"blocks": 0, "mismatches": 0, "in_band": 0, "ties": 0, "outside_band": 0}
    for h in heads:
        rep = head_mask_parity(q, k, h, r["mask"][h], w.stride, tau, chunk, w.causal, pad0_quirk=False)
        for key in tot:
            tot[key] += rep[key]
    tot["heads"] = heads
    return tot


def summarize(w, L, tau, chunk, m, headline_traffic=False):
    """The per-workload numbers of the JSON line from measure()'s samples."""
    fb = flops_and_bytes(w, L, chunk, m["n_sel"])
    t_est, t_sel, t_att = statistics.mean(m["est"]), statistics.mean(m["sel"]), statistics.mean(m["att"])
    t_tot, t_dense = statistics.mean(m["tot"]), statistics.median(m["dense"])
    est_tf = fb["f_est"] / (t_est * 1e-3) / 1e12
    att_tf = fb["f_sparse"] / (t_att * 1e-3) / 1e12
    rl_est = {
        "kernel": "estimate_gemm_kernel", "bound": "mfma", "achieved": round(est_tf, 1), "peak": PEAK_BF16_TFLOPS,
        "unit": "TFLOP/s", "frac": round(est_tf / PEAK_BF16_TFLOPS, 4), "ms": round(t_est, 3), "flop": fb["f_est"],
        "traffic": measured_traffic_bytes("xattn::estimate_gemm_kernel") if headline_traffic else None,
    }
    rl_att = {
        "kernel": "block_sparse_fwd64_kernel<true>, block_sparse_fwd_kernel<true>", "bound": "mfma", "achieved": round(att_tf, 1),
        "peak": PEAK_BF16_TFLOPS, "unit": "TFLOP/s", "frac": round(att_tf / PEAK_BF16_TFLOPS, 4), "ms": round(t_att, 3),
        "flop": fb["f_sparse"],
        "traffic": measured_traffic_bytes("xattn::block_sparse_fwd64_kernel<true", "xattn::block_sparse_fwd_kernel<true") if headline_traffic else None,
    }
    sel_gbs = fb["pass_bytes"] / (t_sel * 1e-3) / 1e9
    rl_sel = {
        "kernel": "estimate_select_kernel (normalisation + selection, block sums in LDS)", "bound": "hbm",
        "achieved": round(sel_gbs, 1), "peak": PEAK_HBM_GBS, "unit": "GB/s", "frac": round(sel_gbs / PEAK_HBM_GBS, 4),
        "ms": round(t_sel, 3), "bytes": fb["pass_bytes"],
        "reference_staging_bytes": fb["staging_bytes"],     # full block-sum matrix in, byte mask + lists out
        "traffic": measured_traffic_bytes("xattn::estimate_select_kernel") if headline_traffic else None,
    }
    return {
        "estimate_ms": round(t_est, 3), "select_ms": round(t_sel, 3), "sparse_attn_ms": round(t_att, 3),
        "total_ms": round(t_tot, 3), "total_ms_stats": _stats(m["tot"]),
        "estimate_ms_stats": _stats(m["est"]), "select_ms_stats": _stats(m["sel"]), "sparse_attn_ms_stats": _stats(m["att"]),
        "dense_fa_ms": round(t_dense, 3), "dense_fa_ms_stats": _stats(m["dense"]),
        "speedup_vs_dense_fa": round(t_dense / t_tot, 3),
        "estimate_fraction_of_total": round((t_est + t_sel) / t_tot, 4),
        "sparsity": round(1.0 - m["n_sel"] / fb["full_blocks"], 4), "selected_blocks": m["n_sel"],
        "estimate_tflops": round(est_tf, 1), "sparse_tflops": round(att_tf, 1),
        "dense_fa_tflops": round(fb["f_dense"] / (t_dense * 1e-3) / 1e12, 1),
        "select_gbs": round(sel_gbs, 1),
        "roofline_estimator": rl_est, "roofline_sparse_attention": rl_att, "roofline_select": rl_sel,
    }


def workload_config(w, L, tau, chunk, rank8="head"):
    return {
        "workload": (w.name if L == w.L else f"{w.name}@L={L}") + ("" if rank8 == "head" else "@rank8=token"),
        "seq_len": L, "q_heads": w.heads, "kv_heads": w.kv_heads, "head_dim": 128, "stride": w.stride,
        "threshold": tau, "chunk_size": chunk, "block_size": 128, "causal": w.causal,
        "estimator_semantics": "all earlier keys visible (reference Triton branch)",
    }


def density_sweep(w, L, chunk, dev, t_dense, qkv, steps=3):
    """The headline shape at other operating points, so that estimate share and speedup are read against a range
    of densities: thresholds 0.9 / 0.95 / 0.99 on the workload's inputs, and the per-token reading of the rank-8
    term (diffuse attention) at 0.9.  Same stages as the headline, fewer steps."""
    import torch
    from xattn.synthetic import make_inputs

    rows = []
    for rank8, taus in (("head", (0.9, 0.95, 0.99)), ("token", (0.9,))):
        q, k, v = qkv if rank8 == "head" else make_inputs(w, device=dev, seed=0, L=L, dtype=torch.bfloat16, rank8=rank8)
        for tau in taus:
            m = measure(w, q, k, v, L, tau, chunk, steps, 1, 0, 0)
            fb = flops_and_bytes(w, L, chunk, m["n_sel"])
            t_est, t_sel, t_att = statistics.mean(m["est"]), statistics.mean(m["sel"]), statistics.mean(m["att"])
            total = t_est + t_sel + t_att
            rows.append({
                "rank8": rank8, "threshold": tau, "density": round(m["n_sel"] / fb["full_blocks"], 4),
                "estimate_ms": round(t_est, 3), "select_ms": round(t_sel, 3), "sparse_attn_ms": round(t_att, 3),
                "total_ms": round(total, 3), "estimate_share": round((t_est + t_sel) / total, 4),
                "estimate_pflops": round(fb["f_est"] / (t_est * 1e-3) / 1e15, 3),
                "sparse_pflops": round(fb["f_sparse"] / (t_att * 1e-3) / 1e15, 3),
                "speedup_vs_dense_fa": round(t_dense / total, 2),
            })
        del q, k, v
    return rows


def yardsticks(dev):
    """Two library kernels of known provenance on the same box, measurement only (nothing in the package uses
    them): torch.matmul (hipBLASLt) on a bf16 GEMM of the estimator's per-head shape - reshaped length 8192,
    depth stride * 128 = 2048, the full square, i.e. twice the causal estimator's flops per head - called 32
    times back to back like the 32 heads; and torch's flash scaled_dot_product_attention, causal, 32 heads,
    L = 32768 (workload 1's shape with K/V repeated to 32 heads).  The batched form of the GEMM
    ([32, 8192, 2048] x [32, 2048, 8192], a 4 GiB result) is not used: that call ended in an illegal memory
    access inside the library on this image."""
    import torch
    import torch.nn.functional as F
    from torch.nn.attention import SDPBackend, sdpa_kernel

    def timed(fn, warm, reps):
        for _ in range(warm):
            fn()
        torch.cuda.synchronize()
        ts = []
        for _ in range(reps):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            fn()
            e1.record()
            torch.cuda.synchronize()
            ts.append(_ms(e0, e1))
        return ts

    res = {}
    with torch.no_grad():
        a = torch.randn(8192, 2048, device=dev).bfloat16()
        b = torch.randn(8192, 2048, device=dev).bfloat16()

        def gemm32():
            for _ in range(32):
                torch.matmul(a, b.t())

        ts = timed(gemm32, 2, 5)
        fl = 32 * 2.0 * 8192 * 8192 * 2048
        res["gemm_bf16_8192x8192x2048_x32"] = {
            "library": "torch.matmul (hipBLASLt)", "ms": _stats(ts), "tflops": round(fl / (statistics.median(ts) * 1e-3) / 1e12, 1)}
        del a, b
        L = 32768
        try:
            q = torch.randn(1, 32, L, 128, device=dev).bfloat16()
            k = torch.randn(1, 32, L, 128, device=dev).bfloat16()
            v = torch.randn(1, 32, L, 128, device=dev).bfloat16()
            with sdpa_kernel(SDPBackend.FLASH_ATTENTION):
                ts = timed(lambda: F.scaled_dot_product_attention(q, k, v, is_causal=True), 1, 3)
            fl = 4.0 * 128 * 32 * L * (L + 1) / 2
            res["sdpa_flash_causal_L32768_h32"] = {
                "library": "torch scaled_dot_product_attention, FLASH_ATTENTION backend", "ms": _stats(ts),
                "tflops": round(fl / (statistics.median(ts) * 1e-3) / 1e12, 1)}
            del q, k, v
        except Exception as e:      # the backend may refuse the call on another build; the GEMM figure stands alone then
            res["sdpa_flash_causal_L32768_h32"] = {"error": f"{type(e).__name__}: {str(e)[:200]}"}
    return res


def main():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=30)
    ap.add_argument("--warmup", type=int, default=10)
    ap.add_argument("--workload", type=int, default=2, help="index into the synthetic workloads (default: headline)")
    ap.add_argument("--dense-steps", type=int, default=5)
    ap.add_argument("--dense-warmup", type=int, default=2)
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-decode", action="store_true", help="skip the decode-step measurement")
    ap.add_argument("--no-mfma-probe", action="store_true", help="skip the MFMA-only rate probe")
    ap.add_argument("--no-workloads", action="store_true", help="skip the measurements of the other GPU workloads")
    ap.add_argument("--no-yardsticks", action="store_true", help="skip the library GEMM / flash attention yardsticks")
    ap.add_argument("--compare-pipelined", action="store_true",
                    help="also time Xattention_prefill with and without chunk-by-chunk stream pipelining")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="also run one plain 1 GiB device copy (reads 1 GiB, writes 1 GiB) so that HBM byte "
                         "counters collected over this command can be scaled by a kernel of known traffic")
    ap.add_argument("--seq-len", type=int, default=None, help="override L (debug only; invalidates the metric)")
    ap.add_argument("--threshold", type=float, default=None,
                    help="override the workload's tau (a point of the density sweep; the headline value uses the workload's own)")
    ap.add_argument("--rank8", choices=("head", "token"), default="head",
                    help="reading of the text workloads' shared rank-8 component (see xattn/synthetic.py)")
    ap.add_argument("--no-density-sweep", action="store_true",
                    help="skip the extra timings of the headline shape at other thresholds / the per-token generator")
    ap.add_argument("--no-mask-parity", action="store_true", help="skip the oracle runs on two heads of each workload")
    args = ap.parse_args()
    if args.gpus != 1 or int(os.environ.get("WORLD_SIZE", "1")) != 1:
        print("bench.py measures one GPU: the prefill path uses no collectives; run with --gpus 1", file=sys.stderr)
        sys.exit(2)

    import torch

    from xattn.src import hip_backend
    from xattn.src.Xattention import block_sparse_attention, default_chunk_size, estimate_and_select
    from xattn.synthetic import WORKLOADS, make_inputs

    hip_backend.lib()   # fail loudly if the HIP library has not been built
    if not torch.cuda.is_available():
        raise SystemExit("no GPU visible")
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    w = WORKLOADS[args.workload]
    L = args.seq_len or w.L
    tau = w.threshold if args.threshold is None else args.threshold
    q, k, v = make_inputs(w, device=dev, seed=0, L=L, dtype=torch.bfloat16, rank8=args.rank8)
    chunk = w.chunk_size or default_chunk_size(L)
    torch.cuda.synchronize()

    m = measure(w, q, k, v, L, tau, chunk, args.steps, args.warmup, args.dense_steps, args.dense_warmup)
    as_configured = L == w.L and args.threshold is None and args.rank8 == "head"
    is_headline = as_configured and w.name == HEADLINE
    head = summarize(w, L, tau, chunk, m, headline_traffic=is_headline)
    rl_est, rl_att = head["roofline_estimator"], head["roofline_sparse_attention"]
    dominant = rl_est if rl_est["ms"] >= rl_att["ms"] else rl_att

    result = {
        "metric": "per-layer prefill attn ms (estimate+sparse) at 128k; speedup vs dense FA",
        "value": head["total_ms"],
        "unit": "ms",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(m["wall_ms"], 3),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic",
        "config": workload_config(w, L, tau, chunk, args.rank8),
        "timing": {"warmup_steps": args.warmup, "timed_steps": args.steps, "value_is": "mean of the timed steps",
                   "dense_warmup": args.dense_warmup, "dense_timed": args.dense_steps, "dense_fa_ms_is": "median",
                   "stages": "estimate_ms = the estimator's MFMA pass (estimate_gemm_kernel), select_ms = its normalisation "
                             "fused with the block selection (estimate_select_kernel), sparse_attn_ms = block_sparse_fwd64_kernel and block_sparse_fwd_kernel"},
        "kernel_sources_sha256_16": kernel_source_hash(),
    }
    result.update({key: val for key, val in head.items() if not key.startswith("roofline_")})
    # the launch that takes longest of the two MFMA stages; both are listed after it, and the selection pass
    result["roofline"] = dict(dominant)
    result["roofline_estimator"] = rl_est
    result["roofline_sparse_attention"] = rl_att
    result["roofline_select"] = head["roofline_select"]
    if not args.no_mask_parity:
        result["mask_parity"] = mask_parity(w, q, k, tau, chunk, m["col_cnt"])
    if (not args.no_density_sweep) and is_headline:
        result["density_sweep"] = density_sweep(w, L, chunk, dev, head["dense_fa_ms"], (q, k, v))
    if args.compare_pipelined:
        from xattn.src.Xattention import Xattention_prefill

        for flag in (False, True):
            for _ in range(2):
                Xattention_prefill(q, k, v, w.stride, threshold=w.threshold, chunk_size=chunk, causal=w.causal,
                                   pipeline_chunks=flag)
            torch.cuda.synchronize()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(args.steps):
                Xattention_prefill(q, k, v, w.stride, threshold=w.threshold, chunk_size=chunk, causal=w.causal,
                                   pipeline_chunks=flag)
            e1.record()
            torch.cuda.synchronize()
            result["operator_ms_pipelined" if flag else "operator_ms_single_launch"] = round(_ms(e0, e1) / args.steps, 3)
    if args.copy_calibration:
        src = torch.empty(1 << 28, dtype=torch.float32, device=dev).normal_()
        dst = torch.empty_like(src)
        hip_backend.check(
            hip_backend.lib().xattn_calibration_copy(
                dst.data_ptr(), src.data_ptr(), src.numel() * 4, torch.cuda.current_stream().cuda_stream
            ),
            "xattn_calibration_copy",
        )
        torch.cuda.synchronize()
        del src, dst
    if not args.no_decode:
        result["decode_step"] = decode_leg(q, k, v)
    del q, k, v, m
    torch.cuda.empty_cache()
    if (not args.no_workloads) and is_headline:
        # the other GPU workloads, same protocol with fewer steps (their launches are up to 20x longer)
        others = []
        for idx in (1, 3, 4):
            w2 = WORKLOADS[idx]
            c2 = w2.chunk_size or default_chunk_size(w2.L)
            q2, k2, v2 = make_inputs(w2, device=dev, seed=0, L=w2.L, dtype=torch.bfloat16)
            steps2 = 30 if idx == 1 else 10
            m2 = measure(w2, q2, k2, v2, w2.L, w2.threshold, c2, steps2, 10 if idx == 1 else 3, 5 if idx == 1 else 3, 1)
            row = {"config": workload_config(w2, w2.L, w2.threshold, c2), "steps": steps2}
            s2 = summarize(w2, w2.L, w2.threshold, c2, m2)
            for key in ("roofline_estimator", "roofline_sparse_attention", "roofline_select"):
                s2[key] = {kk: vv for kk, vv in s2[key].items() if kk in ("kernel", "achieved", "unit", "frac", "ms")}
            row.update(s2)
            if not args.no_mask_parity:
                row["mask_parity"] = mask_parity(w2, q2, k2, w2.threshold, c2, m2["col_cnt"])
            others.append(row)
            del q2, k2, v2, m2
            torch.cuda.empty_cache()
        result["workloads"] = others
    if not args.no_yardsticks:
        result["yardsticks"] = yardsticks(dev)
    if not args.no_mfma_probe:
        result["mfma_alone"] = mfma_probe(dev)
    if not args.no_cpu_baseline:
        base, (cq, ck, cv, csums, cmask) = cpu_baseline()
        # the same sample on the GPU path (bf16), for scale
        gq, gk, gv = cq.to(dev).bfloat16(), ck.to(dev).bfloat16(), cv.to(dev).bfloat16()
        w0 = WORKLOADS[0]
        for _ in range(3):
            rr = estimate_and_select(gq, gk, w0.stride, w0.threshold, w0.chunk_size, causal=True, use_triton=False)
            block_sparse_attention(gq, gk, gv, rr["col_idx"], rr["col_cnt"], causal=True)
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(10):
            rr = estimate_and_select(gq, gk, w0.stride, w0.threshold, w0.chunk_size, causal=True, use_triton=False)
            block_sparse_attention(gq, gk, gv, rr["col_idx"], rr["col_cnt"], causal=True)
        e1.record()
        torch.cuda.synchronize()
        base["gpu_same_sample_ms"] = round(_ms(e0, e1) / 10, 3)
        # GPU mask against the oracle's on identical values (the sample rounded to bf16, oracle in fp32)
        from oracle.parity import mask_mismatch_detail

        d = mask_mismatch_detail(csums[0], rr["mask"], cmask[0], w0.threshold, True, 0, w0.chunk_size // 128)
        base["gpu_mask_vs_oracle_same_inputs"] = {"blocks": int(cmask[0].numel()), **d}
        result["cpu_baseline"] = base
    print(json.dumps(result))


if __name__ == "__main__":
    main()
