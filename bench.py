#!/usr/bin/env python3
"""Benchmark of the KV compression hot path on one MI355X.

A step is one round trip of the hot path over one request: compress (K-statistics
pass + fused gather/FWHT/quantize/bitpack pass) and decompress (fused
unpack/dequantize/inverse-FWHT/scatter pass) of the BASELINE config-2 request:
Llama-3-8B-shaped, 32 layers x 8 KV heads x D=128 x 8192 tokens of bf16 KV in
16-token paged blocks scattered over a 65536-block pool per layer (128 GiB of
pools), K/V ~ N(0,1) with 4 outlier K channels per head, head split with the
Llama-3.1-8B mask at hybrid 0.3, 16/16 levels, bitpack 4 bits, 4 streams of 8 layers.

value = raw bf16 KV bytes of the request / (compress + decompress time), GB/s.
Inputs are resident in HBM before the timed region; plans (device descriptors) are
built before it too.  After the W warmup steps the K steps are timed once ("unsettled"),
then untimed steps run back to back for --settle-ms (default 150 ms; reported as
settle_steps) and the K steps are timed again: that second timing is the headline, the
sustained-load rate (from idle the step time falls over the first ~40 ms of load,
--settle-curve).  Per-direction throughput and the fraction of HBM peak are printed
alongside.  Prints ONE JSON line.

    python bench.py [--gpus 1] [--steps 20] [--warmup 5]
                    [--workload config2|config3|config4|config5|config2_ans|connector]

The other BASELINE configurations can be timed with --workload (the metric is quoted
on config2, the default; multi-request workloads run as one batched plan per
direction, and the CPU baseline is measured for config2 only).  --workload connector
times the config-2 request through the vLLM connector (save + load, host-timed) and
the reference connector's extract/stack/compress procedure beside it; --workload
config2_ans times the same request with the reference's nvCOMP-ANS profile served by
the GPU rANS codec.  --workload config2_v3 times the request's layers through the fused
Hadamard quantizer (impl "tilelang_fused", kvmi_v3_*).
"""

from __future__ import annotations

import argparse
import ctypes
import json
import os
import platform
import re
import subprocess
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

HBM_PEAK_GBPS = 8000.0  # MI355X HBM3E
METRIC = "compress/decompress GB/s of raw bf16 KV on 1 MI355X; % of HBM peak"


WORKLOADS = {
    "config2": "config2: Llama-3-8B-shaped request, 32 layers x 8 KV heads x D=128 x 8192 tokens, "
               "16-token blocks at seeded random ids of a 65536-block pool per layer, "
               "Hadamard seed 0xC0FEBABE, head split (Llama-3.1-8B mask, hybrid 0.3), "
               "16/16 levels, bitpack 4 bits, 4 streams of 8 layers; step = compress + decompress",
    "config3": "config3: 16 requests of U[1024,16384] tokens, 32 layers x 8 heads x D=128, per-(layer, head) "
               "levels in {6,12} for K and V, bitpack 4, seeded random blocks of a 32768-block pool per "
               "layer (32 distinct pools: the 262144-block pool of the configuration needs 512 GiB for 32 "
               "layers), one batched plan per direction; "
               "step = compress + decompress",
    "config4": "config4: Qwen2.5-72B-shaped request, 80 layers x 8 heads x D=128 x 32768 tokens, 2% "
               "Student-t(3) outliers, layer split levels 12/6 alternating, bitpack 4, contiguous caches, "
               "10 streams of 8 layers; step = compress + decompress",
    "config5": "config5: 256 requests x 256 tokens, 16 layers x 8 heads x D=64, 6/6 levels, bitpack 3, seeded "
               "random blocks, one batched plan per direction; step = compress + decompress",
    "config2_ans": "config2_ans: the config2 request with the reference's shipped nvCOMP-ANS profile "
                   "(configs/compression/original_top_nvcomp.json: Hadamard seed 0xC0FEBABE, Llama-3.1-8B head "
                   "split hybrid 0.9, levels 6/6/6/4) served by the GPU rANS codec over 3-bit symbols, 4 streams of "
                   "8 layers; decompress scatters to a disjoint set of 512 block ids; step = compress (kstats, "
                   "encode, one batched rANS encode + scan + compact for the 4 streams) + decompress (one batched "
                   "rANS decode, decode)",
    "connector": "connector: the config2 request through CompressedKVConnector (save_kv_layer x 32 + wait_for_save "
                 "-> LoopbackTransport -> start_load_kv into the same caches and block ids), Hadamard seed "
                 "0xC0FEBABE, Llama-3.1-8B head split hybrid 0.3, 16/16 levels, bitpack 4; step = save + load, "
                 "host-timed with device synchronization; the reference connector's procedure (extract, stack, "
                 "compress, build_wire / restore, decompress, inject) on the same kernels timed beside it",
    "config2_v3": "config2_v3: the config2 request's 32 layers, gathered dense [2, 512, 16, 8, 128] outside the "
                  "timed region, through impl 'tilelang_fused' (kvmi_v3_compress / kvmi_v3_decompress: fp32 FWHT and "
                  "statistics, uint8 symbols, fp32 metadata out, float16 metadata in), Hadamard seed 0xC0FEBABE, "
                  "Llama-3.1-8B head split hybrid 0.3, 16/16 levels; step = compress + decompress of every layer",
    "bitpack": "bitpack: the operator-path BitPackCodec alone (kvmi_bitpack_encode / kvmi_bitpack_decode), "
               "the config-2 request's 2^29 uint8 symbols (32 layers x 2 x 8192 tokens x 8 heads x 128) of "
               "seeded values < 16 at 4 bits, all buffers allocated outside the timed region; step = encode + "
               "decode",
    "runtime": "runtime: fixed-profile runtime (create_runtime backend 'fused'), token view (block_size 1) 1024 "
               "tokens x 28 layers x 4 KV "
               "heads x D=128, default profile (Hadamard, layer split, K channel / V token, levels 12/8 high "
               "6/4 low, ANS codec = GPU rANS over bytes), slot_count 2, one 1024-block chunk per part, seeded "
               "N(0,1) caches; step = encode K then V with completion waits, decode K then V into disjoint "
               "blocks (the reference's scripts/bench_runtime_dispatch.py procedure)",
}

RUNTIME_REFERENCE = {"encode_gbps": 84.11, "decode_gbps": 88.92, "hardware": "H200 NVL, fused C++ + nvCOMP ANS",
                     "source": "docs/benchmarks/h200-runtime-dispatch-20261105/README.md:23-25"}

CONNECTOR_PROFILE = {
    "pipeline": ["transformer", "quantizer", "codec"],
    "transformer_config": {"transform_type": "hadamard", "seed": 0xC0FEBABE},
    "quantizer_config": {"model_name": "Llama-3.1-8B-Instruct", "hybrid_ratio": 0.3, "high_key_max_value": 16,
                         "high_value_max_value": 16, "low_key_max_value": 16, "low_value_max_value": 16,
                         "axis_key": "channel", "axis_value": "token", "split_type": "head"},
    "codec_config": {"codec_type": "bitpack", "bitpack_bits": 4},
}


def hip_kernel_names(codec, S: int, H: int, D: int, bits: int, cplan=None) -> dict:
    """Name of the HIP kernel each entry point runs for this geometry: MFMA, or what
    kvmi_paged_kernels says (wave tiles, quad-per-row or generic rows)."""
    default_axes = tuple(getattr(codec, "axes", ("channel", "token"))) == ("channel", "token")
    pow2 = D in (64, 128) and default_axes
    if D == 256 and H <= 16 and default_axes and codec.fwht == "mfma" and codec.transform:
        Hv = 2 * H  # paired virtual heads of 128 (kvmi_common.hpp paired_view)
        ok = 8 % Hv == 0 or (Hv in (16, 32) and S & (S - 1) == 0 and ((32 // Hv) * 128 * bits // 8) % 16 == 0)
        if ok and (S * Hv) % 32 == 0:
            hm = 8 if Hv <= 8 else 32
            return {"kvmi_encode_paged": f"encode_mfma_pair_kernel<{bits}, false, {hm}>",
                    "kvmi_decode_paged": f"decode_mfma_pair_kernel<{bits}, 8, {hm}>",
                    "kvmi_kstats_paged": "kstats_mfma_pair_kernel" if Hv <= 8 else "kstats_wide_pair_kernel",
                    "finalize": "kstats_finalize_kernel"}
    wide = H in (16, 32) and S & (S - 1) == 0 and ((32 // H) * D * bits // 8) % 16 == 0  # wide-head MFMA
    mfma = pow2 and codec.fwht == "mfma" and codec.transform and (8 % H == 0 or wide) and (S * H) % 32 == 0
    if mfma and wide:
        return {"kvmi_encode_paged": f"encode_mfma_wide_kernel<{D // 32}, {bits}, false>",
                "kvmi_decode_paged": f"decode_mfma_wide_kernel<{D // 32}, {bits}, 8>",
                "kvmi_kstats_paged": f"kstats_wide_kernel<{D // 32}>", "finalize": "kstats_finalize_kernel"}
    if mfma:
        names = {"kvmi_encode_paged": f"encode_mfma_kernel<{D // 32}, {bits}, false>",
                 "kvmi_decode_paged": ("decode_kt_kernel<8>" if (D, bits) == (128, 4)
                                       else f"decode_mfma_kernel<{D // 32}, {bits}, 8>"),
                 "kvmi_kstats_paged": f"kstats_mfma_kernel<{D // 32}>", "finalize": "kstats_finalize_kernel"}
        if cplan is not None and getattr(cplan, "workspace", None) is not None:  # the one-pass kernel runs
            names["kvmi_compress_paged"] = f"onepass_kernel<{D // 32}, {bits}, false>"
        return names
    from kvserve_amd import _lib

    geo = _lib.Geometry(block_size=S, num_heads=H, head_dim=D, bits=bits, max_groups=1)
    geo.flags = {"valu": _lib.F_VALU_FWHT, "rows": _lib.F_ROW_FWHT}.get(codec.fwht, 0)
    geo.flags |= 0 if codec.transform else _lib.F_NO_TRANSFORM
    geo.flags |= _lib.F_NATIVE_LAYOUT if getattr(codec, "layout", "permuted") == "native" else 0
    geo.flags |= {"channel": 0, "token": _lib.F_K_TOKEN, "tensor": _lib.F_K_TENSOR}[codec.axes[0]]
    geo.flags |= {"token": 0, "channel": _lib.F_V_CHANNEL, "tensor": _lib.F_V_TENSOR}[codec.axes[1]]
    blocks = max(1, getattr(cplan, "max_blocks", 1))
    lpr = 1 << max(0, (D // 16 - 1).bit_length())  # generic rows: next_pow2(D / 16) lanes per row
    tile = f"{D}, {'true' if codec.transform else 'false'}, {4 if bits == 4 else 0}"
    names = {}
    for call, decode in (("kvmi_encode_paged", 0), ("kvmi_decode_paged", 1)):
        family = _lib.load().kvmi_paged_kernels(ctypes.byref(geo), 1, blocks, decode, None)
        kind = "decode" if decode else "encode"
        names[call] = {_lib.KERNELS_TILE: f"tile_{kind}_kernel<{tile}>", _lib.KERNELS_QUAD: f"{kind}_kernel<{D}, {bits}>",
                       _lib.KERNELS_ROWS: f"rows_{kind}_kernel<{lpr}, {bits}>"}[family]
        if not decode:
            stats = f"tile_stats_kernel<{D}>" if codec.transform else "tile_plain_stats_kernel"
            names["kvmi_kstats_paged"] = {_lib.KERNELS_TILE: stats, _lib.KERNELS_QUAD: f"kstats_kernel<{D}>",
                                          _lib.KERNELS_ROWS: f"rows_stats_kernel<{lpr}>"}[family]
            names["finalize"] = "kstats_finalize_kernel" if family == _lib.KERNELS_QUAD else "rows_finalize_kernel"
    return names


def compress_kernels(names: dict, cplan) -> list:
    """HIP kernels of one compress of `cplan`, in launch order."""
    if "kvmi_compress_paged" in names:
        return [names["kvmi_compress_paged"]]
    return [names["kvmi_kstats_paged"], names["finalize"], names["kvmi_encode_paged"]]


def traffic_frac(kernels, seconds: float, workload: str):
    """Fraction of HBM peak moved by `kernels` (profiled bytes per dispatch, summed)
    in `seconds`, or None when a kernel has no committed profile."""
    total = 0
    for k in kernels:
        t = profiled_traffic(k, workload)
        if t is None:
            return None
        total += t
    return round(total / seconds / 1e9 / HBM_PEAK_GBPS, 4)


def profiled_traffic(kernel: str, workload: str = "config2", root: Path = None):
    """HBM bytes per dispatch of `kernel` on this workload from the committed rocprofv3
    --pmc FETCH_SIZE / WRITE_SIZE summaries (copy-calibrated read + write MiB), or None
    when no summary covers this kernel.  A row is used only if its scaled MiB follow
    from its KiB columns and the summary's stated calibration factors."""
    cal = re.compile(r"FETCH_SIZE is scaled by ([0-9]+\.[0-9]+) and WRITE_SIZE by ([0-9]+\.[0-9]+)")
    root = Path(__file__).resolve().parent / "profiles" if root is None else Path(root)
    for md in sorted(root.glob(f"*{workload}*.md")):
        text = md.read_text()
        m = cal.search(text)
        if not m:
            continue
        fs, ws = float(m.group(1)), float(m.group(2))
        in_table = False
        for line in text.splitlines():
            cells = [c.strip() for c in line.strip().strip("|").split("|")]
            if not line.startswith("|"):
                in_table = False
            elif cells[-2:] == ["scaled read MiB", "scaled write MiB"]:
                in_table = True
            elif in_table and cells[0] == kernel:
                fk, wk, rm, wm = (float(c) for c in cells[1:5])
                if abs(fk * fs / 1024 - rm) > 0.1 or abs(wk * ws / 1024 - wm) > 0.1:
                    return None  # inconsistent row: not evidence
                return int(round((rm + wm) * 2**20))
    return None


def cpu_model() -> str:
    try:
        out = subprocess.run(["lscpu"], capture_output=True, text=True).stdout
        for line in out.splitlines():
            if line.startswith("Model name:"):
                return line.split(":", 1)[1].strip()
    except Exception:
        pass
    return platform.processor() or "unknown"


def _oracle_worker_init():
    """Imports of an oracle worker process, done before anything is timed."""
    import oracle.kvpipe  # noqa: F401
    import torch  # noqa: F401  (the sign recipe's generator)


def _oracle_worker_ready(_):
    time.sleep(0.05)  # long enough that every worker takes one of these


def _oracle_round_trip(task):
    """One layer through the CPU oracle (compress then decompress); seconds spent."""
    import numpy as np

    from oracle import kvpipe as kp

    blocks, prof, seed, bits, layer_id = task
    B = blocks.shape[1]
    t0 = time.perf_counter()
    chunks = kp.compress_request([blocks], list(range(B)), [prof], seed, bits, layer_ids=[layer_id])
    kp.decompress_request(chunks, [np.zeros_like(blocks)], list(range(B)), [prof], seed, bits, layer_ids=[layer_id])
    return time.perf_counter() - t0


def cpu_baseline(wl, budget_s: float, workers: int = 16):
    """Time the CPU oracle (numpy restatement of the reference pipeline) on whole
    layers of the same request: one thread for about half of `budget_s`, then every
    layer of the request spread over `workers` processes (the box's CPU share, at most
    os.cpu_count()); GB/s of raw KV for a round trip (compress + decompress)."""
    import multiprocessing as mp

    import numpy as np
    import torch

    from oracle import kvpipe as kp

    req = wl.requests[0]
    ids = req.block_ids.long()
    tasks = []
    for l in range(len(req.pools)):
        blocks = req.pools[l][:, ids].contiguous().cpu().view(torch.int16).numpy().view(np.uint16)
        p = req.profiles[l]
        prof = kp.LayerProfile(kp.PartProfile(p.k_order, p.k_levels, p.k_groups()),
                               kp.PartProfile(p.v_order, p.v_levels, p.v_group))
        tasks.append((blocks, prof, wl.seed, wl.bits, req.layer_ids[l]))
    one_bytes, one_s, one_layers = 0, 0.0, 0
    for task in tasks:
        one_s += _oracle_round_trip(task)
        one_bytes += task[0].nbytes
        one_layers += 1
        if one_s >= budget_s / 2:
            break
    single = one_bytes / one_s / 1e9
    n = max(1, min(workers, os.cpu_count() or 1))
    # worker processes are started fresh (spawn), and never touch the GPU
    with mp.get_context("spawn").Pool(n, initializer=_oracle_worker_init) as pool:
        pool.map(_oracle_worker_ready, range(4 * n), chunksize=1)  # start-up and imports, untimed
        t0 = time.perf_counter()
        pool.map(_oracle_round_trip, tasks, chunksize=1)
        wall = time.perf_counter() - t0
    total = sum(t[0].nbytes for t in tasks)
    return {
        "value": round(total / wall / 1e9, 4),
        "unit": "GB/s (round trip, raw bf16 KV)",
        "cores": n,
        "kind": "port",
        "value_1_core": round(single, 4),
        "sample": f"all {len(tasks)} layers of the config-2 request ({total / 2**20:.0f} MiB raw) over {n} processes "
                  f"in {wall:.1f} s, and {one_layers} layers on one thread in {one_s:.1f} s; numpy oracle "
                  f"compress+decompress on {cpu_model()} (os.cpu_count()={os.cpu_count()})",
    }


NVCOMP_QUANTIZER = {"model_name": "Llama-3.1-8B-Instruct", "hybrid_ratio": 0.9, "high_key_max_value": 6,
                    "high_value_max_value": 6, "low_key_max_value": 6, "low_value_max_value": 4,
                    "axis_key": "channel", "axis_value": "token", "split_type": "head"}


def bench_entropy(args) -> dict:
    """The config-2 request with the entropy-coded profile: fused kernels plus the
    rANS codec stage, every buffer allocated before the timed region."""
    import ctypes
    import dataclasses

    import torch

    from kvserve_amd import _lib, workloads
    from kvserve_amd.compression.codec.rans_codec import unpack_target
    from kvserve_amd.engine import FusedKVCodec
    from kvserve_amd.profiles import profiles_from_quantizer_config

    dev = torch.device("cuda", 0)
    wl = workloads.make_config2(device=dev, num_layers=args.layers)
    req = wl.requests[0]
    L, S, H, D, B = len(req.pools), wl.block_size, wl.num_heads, wl.head_dim, req.block_ids.numel()
    bits = max(NVCOMP_QUANTIZER[k] for k in NVCOMP_QUANTIZER if k.endswith("max_value")).bit_length()
    profiles = profiles_from_quantizer_config(NVCOMP_QUANTIZER, L, H)
    codec = FusedKVCodec(H, D, S, bits, wl.seed)
    cplan = codec.plan_compress(req.pools, req.block_ids, profiles, req.layer_ids)
    packet = cplan.packet
    perm = torch.randperm(65536, generator=torch.Generator().manual_seed(77))
    used = set(req.block_ids.tolist())
    dst_ids = torch.tensor([i for i in perm.tolist() if i not in used][:B], dtype=torch.int32, device=dev)

    lib = _lib.load()
    stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream)
    per = 2 * H * B * S * D
    chunks = []
    for (s0, e0), st in zip(packet.chunks, packet.streams):
        n = (e0 - s0) * per
        cap, scr = lib.kvmi_rans_max_bytes(n, bits), lib.kvmi_rans_scratch_bytes(n, bits)
        chunks.append({"n": n, "packed": st, "out": torch.empty((cap + 7) // 8 * 8, dtype=torch.uint8, device=dev),
                       "scratch": torch.empty(scr, dtype=torch.uint8, device=dev),
                       "len": torch.zeros(1, dtype=torch.int64, device=dev),
                       "target": unpack_target(n, bits, dev)})
    err = torch.zeros(1, dtype=torch.int32, device=dev)

    enc_jobs = (_lib.RansEncJob * len(chunks))(*[
        _lib.RansEncJob(c["packed"].data_ptr() + 16, c["n"], c["out"].data_ptr(), c["out"].numel(),
                        c["scratch"].data_ptr(), c["scratch"].numel(), c["len"].data_ptr()) for c in chunks])

    def rans_encode_all():  # every stream of the request in one launch per kernel
        _lib.check(lib.kvmi_rans_encode_batch(enc_jobs, len(chunks), bits, sp), "kvmi_rans_encode_batch")

    def rans_decode_all():
        _lib.check(lib.kvmi_rans_decode_batch(dec_jobs, len(chunks), bits, err.data_ptr(), sp),
                   "kvmi_rans_decode_batch")

    def compress():
        for name in cplan.launches():
            cplan.launch(name)
        rans_encode_all()

    compress()
    torch.cuda.synchronize()
    cplan.check_errors()
    for c in chunks:
        c["nbytes"] = int(c["len"].item())
    dec_jobs = (_lib.RansDecJob * len(chunks))(*[
        _lib.RansDecJob(c["out"].data_ptr(), c["nbytes"], c["n"], c["target"].data_ptr() + 16) for c in chunks])
    dpacket = dataclasses.replace(packet, streams=[c["target"] for c in chunks])
    dplan = codec.plan_decompress(dpacket, req.pools, dst_ids)

    def decompress():
        rans_decode_all()
        for name in dplan.launches():
            dplan.launch(name)

    print(f"bench: config2_ans: warmup {args.warmup} steps", file=sys.stderr, flush=True)
    for _ in range(args.warmup):
        compress()
        decompress()
    torch.cuda.synchronize()
    ev = [[torch.cuda.Event(enable_timing=True) for _ in range(3)] for _ in range(args.steps)]
    print(f"bench: config2_ans: timing {args.steps} steps", file=sys.stderr, flush=True)
    t0 = time.perf_counter()
    for k in range(args.steps):
        ev[k][0].record(stream)
        compress()
        ev[k][1].record(stream)
        decompress()
        ev[k][2].record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    cplan.check_errors()
    dplan.check_errors()
    if int(err.item()):
        raise RuntimeError(f"rANS decode reported error {int(err.item())}")
    for c in chunks:
        if not torch.equal(c["target"][16:], c["packed"][16:]):
            raise RuntimeError("rANS round trip differs from the packed symbols")
        if int(c["len"].item()) != c["nbytes"]:
            raise RuntimeError("stream length changed between steps")
    t_c = sum(e[0].elapsed_time(e[1]) for e in ev) / args.steps
    t_d = sum(e[1].elapsed_time(e[2]) for e in ev) / args.steps
    R = L * 2 * B * S * H * D * 2
    nsym = L * per
    wire = sum(c["nbytes"] for c in chunks)
    meta = (packet.kmeta.numel() + packet.vmeta.numel()) * 2
    return {
        "metric": "compress/decompress GB/s of raw bf16 KV on 1 MI355X, entropy-coded profile",
        "value": round(R / ((t_c + t_d) / 1e3) / 1e9, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(wall / args.steps * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded N(0,1) KV, 4 outlier K channels/head x10)",
        "config": {"workload": WORKLOADS["config2_ans"], "requests": 1, "layers": L, "tokens": B * S,
                   "raw_bytes": R, "symbols": nsym, "symbol_bits": bits, "packed_bytes": nsym * bits // 8,
                   "wire_bytes": wire, "meta_bytes": meta},
        "compress_ms": round(t_c, 4),
        "decompress_ms": round(t_d, 4),
        "compress_gbps": round(R / t_c / 1e6, 2),
        "decompress_gbps": round(R / t_d / 1e6, 2),
        "ratio_vs_uint8_symbols": round(nsym / wire, 3),
        "ratio_vs_raw_bf16": round(R / (wire + meta), 3),
        "bits_per_symbol": round(wire * 8 / nsym, 4),
        "roofline": None,
        "cpu_baseline": None,
    }


def bench_connector(args) -> dict:
    """Time one request through the connector's worker path and, beside it, the
    reference connector's procedure on the same operators."""
    from types import SimpleNamespace

    import torch

    from kvserve_amd import workloads
    from kvserve_amd.compression import KVCompressionAdapter
    from kvserve_amd.compression.wire import CompressedWire, build_wire, restore_from_wire
    from kvserve_amd.connector import (CompressedKVConnector, CompressedKVConnectorMetadata, KVConnectorRole,
                                       LoopbackTransport, extract_kv_from_layer_by_blocks,
                                       inject_kv_into_layer_by_blocks)

    dev = torch.device("cuda", 0)
    wl = workloads.make_config2(device=dev, num_layers=args.layers)
    req = wl.requests[0]
    L, S, H, D = len(req.pools), wl.block_size, wl.num_heads, wl.head_dim
    names = [f"model.layers.{i}.self_attn.attn" for i in range(L)]
    caches = dict(zip(names, req.pools))
    ids = [int(b) for b in req.block_ids.tolist()]
    tokens = list(range(len(ids) * S))

    def cfg(producer: bool, port: int):
        extra = {"compression": CONNECTOR_PROFILE, "transport_class": "loopback"}
        return SimpleNamespace(
            kv_transfer_config=SimpleNamespace(is_kv_producer=producer, kv_buffer_size=1 << 36, kv_ip="127.0.0.1",
                                               kv_port=port, kv_connector_extra_config=extra),
            cache_config=SimpleNamespace(block_size=S),
            model_config=SimpleNamespace(get_num_kv_heads=lambda pc: H, get_head_size=lambda: D,
                                         model="Llama-3.1-8B-Instruct", use_mla=False),
            parallel_config=SimpleNamespace())

    class Layer:
        def __init__(self, cache):
            self.kv_cache = [cache]

    prod = CompressedKVConnector(cfg(True, 31000), KVConnectorRole.WORKER)
    cons = CompressedKVConnector(cfg(False, 31000), KVConnectorRole.WORKER)
    pm, dm = CompressedKVConnectorMetadata(), CompressedKVConnectorMetadata()
    pm.add_request("req", "T", tokens, ids, S)
    dm.add_request("req", "T", tokens, ids, S)
    prod.bind_connector_metadata(pm)
    cons.bind_connector_metadata(dm)
    fctx = SimpleNamespace(no_compile_layers={n: Layer(c) for n, c in caches.items()}, virtual_engine=0)

    def connector_step():
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for n in names:
            prod.save_kv_layer(n, caches[n], None)
        prod.wait_for_save()
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        cons.start_load_kv(fctx)
        torch.cuda.synchronize()
        return t1 - t0, time.perf_counter() - t1

    ad = KVCompressionAdapter(CONNECTOR_PROFILE, num_kv_heads=H, head_size=D, model_name="Llama-3.1-8B-Instruct")
    tx = LoopbackTransport(True, port=31001)
    rx = LoopbackTransport(False, port=31001, recv_buffer_size=1 << 36)
    order = sorted(names)

    def reference_step():
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        stacked = torch.stack([extract_kv_from_layer_by_blocks(caches[n], ids) for n in order])
        wire = build_wire(ad.compress(stacked, "req"), 512 << 20)
        tx.send_bundle("T", ["__compressed__"] + order, wire.meta, wire.body_chunks, wire.aux_tensors)
        tx.wait_for_sent()
        del stacked, wire
        torch.cuda.synchronize()
        t1 = time.perf_counter()
        ((_, payload),) = rx.drain_received()["T"]
        out = ad.decompress(restore_from_wire(CompressedWire(payload["meta"], payload["body_chunks"],
                                                             payload["aux_tensors"])))
        for i, n in enumerate(order):
            inject_kv_into_layer_by_blocks(caches[n], out[i], ids)
        torch.cuda.synchronize()
        rx.release_received("T", rx.payload_nbytes(payload))
        return t1 - t0, time.perf_counter() - t1

    def timed(step, label):
        print(f"bench: {label}: warmup {args.warmup} steps", file=sys.stderr, flush=True)
        for _ in range(args.warmup):
            step()
        print(f"bench: {label}: timing {args.steps} steps", file=sys.stderr, flush=True)
        ts = [step() for _ in range(args.steps)]
        return sum(t[0] for t in ts) / len(ts), sum(t[1] for t in ts) / len(ts)

    save_s, load_s = timed(connector_step, "connector")
    wire_bytes = next(r["payload_bytes"] for r in reversed(prod._transport.stats) if r["direction"] == "send")

    # the kernels alone on the same request: the producer's codec, plans built outside
    # the timed region, HIP events on the launch stream
    mgr = prod._get_compressor()._manager
    codec = mgr._codec(H, D, S)
    profs = mgr.profiles(list(range(L)), H)
    cplan = codec.plan_compress([caches[n] for n in order], ids, profs)
    dplan = codec.plan_decompress(cplan.packet, [caches[n] for n in order], ids)
    for _ in range(args.warmup):
        cplan.run()
        dplan.run()
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(3)]
    kc = kd = 0.0
    for _ in range(args.steps):
        ev[0].record()
        cplan.run()
        ev[1].record()
        dplan.run()
        ev[2].record()
        ev[2].synchronize()
        kc += ev[0].elapsed_time(ev[1])
        kd += ev[1].elapsed_time(ev[2])
    kernel_ms = (kc + kd) / args.steps
    ref_save_s, ref_load_s = timed(reference_step, "reference procedure")
    R = L * 2 * len(ids) * S * H * D * 2
    return {
        "metric": "connector save + load GB/s of raw bf16 KV on 1 MI355X (wait_for_save + start_load_kv)",
        "value": round(R / (save_s + load_s) / 1e9, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round((save_s + load_s) * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded N(0,1) KV, 4 outlier K channels/head x10)",
        "config": {"workload": WORKLOADS["connector"], "requests": 1, "layers": L, "tokens": len(tokens),
                   "raw_bytes": R, "wire_bytes": wire_bytes},
        "save_ms": round(save_s * 1e3, 4),
        "load_ms": round(load_s * 1e3, 4),
        "kernel_ms": {"compress": round(kc / args.steps, 4), "decompress": round(kd / args.steps, 4)},
        "connector_over_kernels": round((save_s + load_s) * 1e3 / kernel_ms, 3),
        # the in-process LoopbackTransport hands the producer's tensors and metadata over
        # as they are; a network transport adds serialization and staging copies
        "transport": "LoopbackTransport (in-process hand-off: no serialization, no staging copy)",
        "save_gbps": round(R / save_s / 1e9, 2),
        "load_gbps": round(R / load_s / 1e9, 2),
        "reference_procedure": {"save_ms": round(ref_save_s * 1e3, 4), "load_ms": round(ref_load_s * 1e3, 4),
                                "gbps": round(R / (ref_save_s + ref_load_s) / 1e9, 2)},
        "roofline": None,
        "cpu_baseline": None,
    }


def bench_fused_v3(args) -> dict:
    """impl "tilelang_fused" (kvmi_v3_* through the C-ABI) on the config-2 request's
    layers.  The operator takes the dense layer [2, B, 16, H, D] that the reference's
    connector gathers before calling it, so the layers are gathered once outside the
    timed region; every output buffer is allocated before it."""
    import ctypes

    import numpy as np
    import torch

    from kvserve_amd import _lib, workloads
    from kvserve_amd.compression.quantizer import FusedHadamardQuantizer

    dev = torch.device("cuda", 0)
    wl = workloads.make_config2(device=dev, num_layers=args.layers)
    req = wl.requests[0]
    L, S, H, D, B = len(req.pools), wl.block_size, wl.num_heads, wl.head_dim, req.block_ids.numel()
    rows = B * S
    idx = req.block_ids.long()
    x = torch.stack([p[:, idx].reshape(2, rows, H, D) for p in req.pools])  # [L, 2, rows, H, D]
    del idx
    qz = FusedHadamardQuantizer(base_seed=wl.seed, **CONNECTOR_PROFILE["quantizer_config"])
    tables = [qz._device_tables(l, H, D, dev) for l in range(L)]
    lib = _lib.load()
    q = torch.empty((L, 2, rows, H, D), dtype=torch.uint8, device=dev)
    kmeta = torch.empty((L, 2, H, D), dtype=torch.float32, device=dev)
    vmeta = torch.empty((L, 2, rows, H), dtype=torch.float32, device=dev)
    scratch = torch.empty(int(lib.kvmi_v3_scratch_bytes(rows, H, D)), dtype=torch.uint8, device=dev)
    out = torch.empty_like(x)
    stream = torch.cuda.current_stream()
    sp = ctypes.c_void_p(stream.cuda_stream)

    def compress():
        for l in range(L):
            lv, grp, sg = tables[l]
            _lib.check(lib.kvmi_v3_compress(x[l].data_ptr(), rows, H, D, sg.data_ptr(), lv.data_ptr(),
                                            grp.data_ptr(), q[l].data_ptr(), kmeta[l].data_ptr(),
                                            vmeta[l].data_ptr(), scratch.data_ptr(), sp), "kvmi_v3_compress")

    compress()
    km16, vm16 = kmeta.to(torch.float16), vmeta.to(torch.float16)  # the wire form of the metadata

    def decompress():
        for l in range(L):
            _lib.check(lib.kvmi_v3_decompress(q[l].data_ptr(), rows, H, D, tables[l][2].data_ptr(),
                                              km16[l].data_ptr(), vm16[l].data_ptr(), out[l].data_ptr(), sp),
                       "kvmi_v3_decompress")

    print(f"bench: warmup {args.warmup} steps", file=sys.stderr, flush=True)
    for _ in range(args.warmup):
        compress()
        decompress()
    torch.cuda.synchronize()
    print(f"bench: timing {args.steps} steps", file=sys.stderr, flush=True)
    ev = [[torch.cuda.Event(enable_timing=True) for _ in range(3)] for _ in range(args.steps)]
    t0 = time.perf_counter()
    for e in ev:
        e[0].record(stream)
        compress()
        e[1].record(stream)
        decompress()
        e[2].record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    t_c = sum(e[0].elapsed_time(e[1]) for e in ev) / args.steps
    t_d = sum(e[1].elapsed_time(e[2]) for e in ev) / args.steps
    R = x.numel() * 2
    Q = q.numel()
    M32, M16 = (kmeta.numel() + vmeta.numel()) * 4, (km16.numel() + vm16.numel()) * 2
    alg_c, alg_d = R + Q + M32, Q + M16 + R  # read KV, write symbols + meta (or the reverse)
    # profiled HBM bytes per dispatch (committed rocprofv3 --pmc summary), per layer
    dk = f"v3_dequant_kernel<{D}>"
    ct = [profiled_traffic(k, "config2_v3") for k in (f"v3_kstats_kernel<{D}>", "v3_kfinal_kernel",
                                                     f"v3_quant_kernel<{D}>")]
    dt = profiled_traffic(dk, "config2_v3")
    res = {
        "metric": "compress/decompress GB/s of raw bf16 KV on 1 MI355X, impl tilelang_fused",
        "value": round(R / ((t_c + t_d) / 1e3) / 1e9, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(wall / args.steps * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "f32",
        "data": "synthetic (seeded N(0,1) KV, 4 outlier K channels/head x10)",
        "config": {"workload": WORKLOADS["config2_v3"], "requests": 1, "layers": L, "tokens": rows,
                   "raw_bytes": R, "symbol_bytes": Q, "meta_bytes_fp32": M32, "meta_bytes_fp16": M16},
        "compress_ms": round(t_c, 4),
        "decompress_ms": round(t_d, 4),
        "compress_gbps": round(R / t_c / 1e6, 2),
        "decompress_gbps": round(R / t_d / 1e6, 2),
        "compress_hbm_frac": round(alg_c / t_c / 1e6 / HBM_PEAK_GBPS, 4),
        "decompress_hbm_frac": round(alg_d / t_d / 1e6 / HBM_PEAK_GBPS, 4),
        "compress_traffic_hbm_frac": (round(L * sum(ct) / (t_c / 1e3) / 1e9 / HBM_PEAK_GBPS, 4)
                                      if None not in ct else None),
        "decompress_traffic_hbm_frac": (round(L * dt / (t_d / 1e3) / 1e9 / HBM_PEAK_GBPS, 4)
                                        if dt is not None else None),
        "roofline": {"bound": "hbm", "kernel": f"{dk} (one launch per layer)",
                     "achieved": round(alg_d / L / (t_d / L / 1e3) / 1e9, 1), "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                     "frac": round(alg_d / t_d / 1e6 / HBM_PEAK_GBPS, 4), "traffic": dt,
                     "algorithmic_bytes_per_launch": alg_d // L},
        "cpu_baseline": None,
    }
    if not args.no_cpu_baseline:
        from oracle import fused_v3 as fv
        from oracle import kvpipe as kp

        print("bench: CPU oracle baseline", file=sys.stderr, flush=True)
        xb = x[0].cpu().view(torch.int16).numpy().view(np.uint16)
        k_lv, v_lv = qz.levels(0, H)
        signs = kp.rademacher_signs(wl.seed, 0, H, D)
        n, t_cpu = 0, 0.0
        while t_cpu < args.cpu_budget / 2 and n < L:
            t1 = time.perf_counter()
            rq, rm = fv.compress_layer(xb, signs, k_lv, v_lv)
            fv.decompress_layer(rq, rm["kmin"].astype(np.float16), rm["kscale"].astype(np.float16),
                                rm["vmin"].astype(np.float16), rm["vscale"].astype(np.float16), signs)
            t_cpu += time.perf_counter() - t1
            n += 1
        res["cpu_baseline"] = {"value": round(n * (R // L) / t_cpu / 1e9, 4), "unit": "GB/s (round trip, raw bf16 KV)",
                               "cores": 1, "kind": "port",
                               "sample": f"{n} x layer 0 of the request ({R // L >> 20} MiB raw) in {t_cpu:.1f} s; "
                                         f"numpy oracle (oracle/fused_v3.py) compress+decompress, one thread, on "
                                         f"{cpu_model()}"}
    return res


def bench_bitpack(args) -> dict:
    """BitPackCodec of the operator path (bitpack_codec.py:100-135) through the C-ABI on
    the config-2 symbol count; every buffer is allocated before the timed region."""
    import ctypes

    import numpy as np
    import torch

    from kvserve_amd import _lib

    dev = torch.device("cuda", 0)
    bits, n = 4, 1 << 29
    g = torch.Generator(device=dev).manual_seed(7)
    sym = torch.randint(0, 1 << bits, (n,), dtype=torch.uint8, device=dev, generator=g)
    nbytes = 16 + (n * bits + 7) // 8
    stream_buf = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    back = torch.empty(n, dtype=torch.uint8, device=dev)
    err = torch.zeros(1, dtype=torch.int32, device=dev)
    lib = _lib.load()
    st = torch.cuda.current_stream()
    sp = ctypes.c_void_p(st.cuda_stream)

    def encode():
        _lib.check(lib.kvmi_bitpack_encode(sym.data_ptr(), n, bits, stream_buf.data_ptr(), err.data_ptr(), sp),
                   "kvmi_bitpack_encode")

    def decode():
        _lib.check(lib.kvmi_bitpack_decode(stream_buf.data_ptr(), nbytes, n, bits, back.data_ptr(), err.data_ptr(),
                                           sp), "kvmi_bitpack_decode")

    print(f"bench: warmup {args.warmup} steps", file=sys.stderr, flush=True)
    for _ in range(args.warmup):
        encode()
        decode()
    torch.cuda.synchronize()
    if err.item() != 0 or not torch.equal(back, sym):
        raise RuntimeError("bitpack round trip failed")
    print(f"bench: timing {args.steps} steps", file=sys.stderr, flush=True)
    ev = [[torch.cuda.Event(enable_timing=True) for _ in range(3)] for _ in range(args.steps)]
    t0 = time.perf_counter()
    for e in ev:
        e[0].record(st)
        encode()
        e[1].record(st)
        decode()
        e[2].record(st)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    t_e = sum(e[0].elapsed_time(e[1]) for e in ev) / args.steps
    t_d = sum(e[1].elapsed_time(e[2]) for e in ev) / args.steps
    alg = n + nbytes  # read the symbols, write the stream (or the reverse)
    k_e, k_d = f"bitpack_encode_kernel<{bits}, true>", f"bitpack_decode_kernel<{bits}, true>"
    te, td = profiled_traffic(k_e, "bitpack"), profiled_traffic(k_d, "bitpack")
    dom, t_dom, tr_dom = (k_e, t_e, te) if t_e >= t_d else (k_d, t_d, td)
    res = {
        "metric": "bitpack encode/decode GB/s of uint8 symbols on 1 MI355X",
        "value": round(n / ((t_e + t_d) / 1e3) / 1e9, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(wall / args.steps * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u8",
        "data": "synthetic (seeded uniform symbols < 16)",
        "config": {"workload": WORKLOADS["bitpack"], "symbols": n, "bits": bits, "stream_bytes": nbytes},
        "encode_ms": round(t_e, 4),
        "decode_ms": round(t_d, 4),
        "encode_hbm_frac": round(alg / t_e / 1e6 / HBM_PEAK_GBPS, 4),
        "decode_hbm_frac": round(alg / t_d / 1e6 / HBM_PEAK_GBPS, 4),
        "roofline": {"bound": "hbm", "kernel": dom, "achieved": round(alg / t_dom / 1e6, 1), "peak": HBM_PEAK_GBPS,
                     "unit": "GB/s", "frac": round(alg / t_dom / 1e6 / HBM_PEAK_GBPS, 4), "traffic": tr_dom,
                     "algorithmic_bytes_per_launch": alg},
        "cpu_baseline": None,
    }
    if not args.no_cpu_baseline:
        from oracle import cbitpack

        print("bench: CPU oracle baseline", file=sys.stderr, flush=True)
        m = 1 << 26
        host = sym[:m].cpu().numpy()
        k, t_cpu = 0, 0.0
        while t_cpu < args.cpu_budget and k < 64:
            t1 = time.perf_counter()
            body = cbitpack.encode(host, bits)
            cbitpack.decode(body, m, bits)
            t_cpu += time.perf_counter() - t1
            k += 1
        res["cpu_baseline"] = {"value": round(k * m / t_cpu / 1e9, 4), "unit": "GB/s (encode + decode, symbols)",
                               "cores": 1, "kind": "port",
                               "sample": f"{k} x {m >> 20} Mi symbols in {t_cpu:.1f} s; the C oracle "
                                         f"(oracle/cbitpack.py) encode + decode, one thread, on {cpu_model()}"}
    return res


def bench_runtime(args) -> dict:
    """The reference's runtime dispatch benchmark on the HIP runtime: wall time of
    K then V encode (each fenced), then K then V decode, plus device time of each
    stage from events on the slot streams."""
    import ctypes

    import torch

    from kvserve_amd import _lib
    from kvserve_amd.runtime import CacheSpec, CompressionConfig, build_memory_plan, create_runtime

    dev = torch.device("cuda", 0)
    block, blocks, layers, heads, dim = args.rt_block_size, args.rt_blocks, args.rt_layers, 4, 128
    torch.manual_seed(3817)
    config = CompressionConfig.from_extra_config({"compression": {
        "enable-compression-pipeline": True, "logical_blocks_per_chunk": blocks, "slot_count": 2}})
    specs = {f"layer.{i}": CacheSpec(i, block, heads, dim, torch.bfloat16) for i in range(layers)}
    caches = {n: torch.randn((2 * blocks, heads, block, 2 * dim), device=dev, dtype=torch.bfloat16) for n in specs}
    plan = build_memory_plan(config, specs, blocks_per_logical=1, num_layers=layers, device=dev)
    # the reference's number is its fused backend (scripts/bench_runtime_dispatch.py:92-93)
    runtime = create_runtime(plan, "HND", 1, dev, backend="fused")
    runtime.bind_kv_caches(caches, dict.fromkeys(specs, 0))
    tokens = blocks * block
    source, destination = list(range(blocks)), list(range(blocks, 2 * blocks))
    raw = layers * tokens * heads * dim * 2 * 2

    def encode():
        chunks = []
        for part in (0, 1):
            chunk = runtime.encode(part, [source], part, valid_tokens_by_group={0: tokens})
            chunk.event.synchronize()
            chunks.append(chunk)
        return chunks

    def decode(chunks):
        for part, chunk in enumerate(chunks):
            runtime.decode(part, [destination], part, chunk.codec_bytes, chunk.u8_bytes,
                           valid_tokens_by_group={0: tokens}).synchronize()

    print(f"bench: runtime: warmup {args.warmup} steps", file=sys.stderr, flush=True)
    for _ in range(args.warmup):
        decode(encode())
    print(f"bench: runtime: timing {args.steps} steps", file=sys.stderr, flush=True)
    enc_s, dec_s = [], []
    for _ in range(args.steps):
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        chunks = encode()
        t1 = time.perf_counter()
        decode(chunks)
        t2 = time.perf_counter()
        enc_s.append(t1 - t0)
        dec_s.append(t2 - t1)
    med = lambda v: sorted(v)[len(v) // 2]  # noqa: E731
    enc, dec = med(enc_s), med(dec_s)
    coded = [c.codec_bytes for c in chunks]

    # device time per stage: the body launch set (kvmi_rt_encode / kvmi_rt_decode) and
    # the rANS codec, each called through the C-ABI on the slot stream with events
    lib = _lib.load()
    stages = {}
    for part in (0, 1):
        pipe, slot = runtime.pipelines[part], runtime.slots[part]
        stream = runtime.streams[part]
        sp = ctypes.c_void_p(stream.cuda_stream)
        launch = pipe._launches[part][0]
        ids = slot.block_indices[0, :blocks]
        with torch.cuda.stream(stream):
            ids.copy_(torch.tensor(source, dtype=torch.int64))
        packed = slot.arena_b[runtime.layout.u8_base:]
        u8 = chunks[part].u8_bytes

        def body_enc():
            _lib.check(lib.kvmi_rt_encode(ctypes.byref(launch.geometry), launch.table.data_ptr(), launch.num_layers,
                                          ids.data_ptr(), blocks, slot.canonical.data_ptr(), packed.data_ptr(),
                                          slot.aux.data_ptr(), runtime.layout.aux_arena_bytes // 2, sp), "encode")

        def body_dec():
            _lib.check(lib.kvmi_rt_decode(ctypes.byref(launch.geometry), launch.table.data_ptr(), launch.num_layers,
                                          ids.data_ptr(), blocks, packed.data_ptr(), slot.aux.data_ptr(), sp),
                       "decode")

        codec = pipe.codec

        def rans_enc():
            codec.encode(packed, slot.arena_a, u8, torch.cuda.Event())

        def rans_dec():
            codec.decode(slot.arena_a, packed, coded[part], u8, torch.cuda.Event())

        for name, fn in (("body_encode", body_enc), ("rans_encode", rans_enc), ("rans_decode", rans_dec),
                         ("body_decode", body_dec)):
            for _ in range(3):
                fn()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record(stream)
            for _ in range(args.steps):
                fn()
            e1.record(stream)
            e1.synchronize()
            stages[f"{name}_{'kv'[part]}_us"] = round(e0.elapsed_time(e1) * 1e3 / args.steps, 2)
    runtime.shutdown()
    part_raw = raw // 2
    # dominant launch set: the K part's rANS encode (encode + compaction kernels);
    # algorithmic bytes = the u8 symbols read once + the stream written once
    rans_k = stages["rans_encode_k_us"]
    rans_bytes = chunks[0].u8_bytes + coded[0]
    achieved = rans_bytes / (rans_k * 1e-6) / 1e9
    traffic = [profiled_traffic(k, "runtime") for k in ("rans_encode_kernel<8>", "rans_compact_kernel<8, true>")]
    cpu = None if args.no_cpu_baseline else runtime_cpu_baseline(plan, caches, source, args.cpu_budget)
    return {
        "metric": "fixed-profile runtime encode GB/s of raw bf16 K+V on 1 MI355X (K then V, fenced)",
        "value": round(raw / enc / 1e9, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round((enc + dec) * 1e3, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": round(raw / enc / 1e9 / RUNTIME_REFERENCE["encode_gbps"], 3),
        "dtype": "bf16",
        "data": "synthetic (seeded N(0,1) KV)",
        "config": {"workload": WORKLOADS["runtime"], "layers": layers, "tokens": tokens, "block_size": block,
                   "raw_bytes": raw, "encoded_bytes": coded},
        "encode_ms": round(enc * 1e3, 4),
        "decode_ms": round(dec * 1e3, 4),
        "decode_gbps": round(raw / dec / 1e9, 2),
        "decode_vs_baseline": round(raw / dec / 1e9 / RUNTIME_REFERENCE["decode_gbps"], 3),
        "reference": RUNTIME_REFERENCE,
        "stages": stages,
        "roofline": {"bound": "hbm", "achieved": round(achieved, 1), "peak": HBM_PEAK_GBPS, "unit": "GB/s",
                     "frac": round(achieved / HBM_PEAK_GBPS, 4),
                     "traffic": None if None in traffic else sum(traffic),
                     "kernel": "rANS encode launch set of the K part (rans_encode_kernel<8> + "
                               "rans_compact_kernel<8, true>); latency-bound, not HBM-bound"},
        "cpu_baseline": cpu,
    }


def runtime_cpu_baseline(plan, caches, source, budget_s: float):
    """The runtime oracle (numpy, one thread) encoding and decoding whole layers of the
    same chunk, with the rANS oracle as the codec, until `budget_s` is spent."""
    import numpy as np
    import torch

    from kvserve_amd.runtime import build_signs
    from oracle import crans
    from oracle import runtime_ref as R

    cfg, layout = plan.config, plan.layout
    orders = plan.head_selection.local_orders
    done, t_total, layers = 0, 0.0, 0
    for name in caches:
        cache = caches[name].cpu().view(torch.int16).numpy().view(np.uint16)
        target = np.zeros_like(cache)
        for kv in (0, 1):
            part = next(p for p in layout.parts(kv) if p.layer_name == name)
            sections = [R.Section(s.head_start, s.head_count, s.num_levels, s.axis, s.aux_min_offset,
                                  s.aux_scale_offset) for s in part.sections]
            signs = build_signs(part, orders[part.layer_index], cfg.seed).reshape(part.num_heads, -1)
            mk = lambda c: R.LayerPart(cache=c, channel_offset=kv * part.head_size, head_size=part.head_size,  # noqa
                                       order=orders[part.layer_index], u8_offset=0,
                                       signs=signs.to(torch.int8).numpy(), sections=sections)
            tokens = len(source) * part.block_size
            n = part.raw_bytes // 2
            t0 = time.perf_counter()
            payload, aux, tail = R.encode_part([mk(cache)], source, tokens, part.block_size, 1, True, True, n,
                                               layout.aux_bytes_by_part[kv])
            stream = crans.encode(payload, 8)
            back = crans.decode(stream, n, 8)
            R.decode_part([mk(target)], source, tokens, part.block_size, 1, True, True, back, aux, tail)
            t_total += time.perf_counter() - t0
            done += part.raw_bytes
        layers += 1
        if t_total >= budget_s:
            break
    return {
        "value": round(done / t_total / 1e9, 5),
        "unit": "GB/s (encode + decode, raw bf16 K+V)",
        "cores": 1,
        "kind": "port",
        "sample": f"{layers} of {len(caches)} layers, K and V parts of the 1024-token chunk "
                  f"({done / 2**20:.0f} MiB raw), numpy runtime oracle + C rANS oracle encode and decode on "
                  f"{cpu_model()} (os.cpu_count()={os.cpu_count()}), {t_total:.1f} s",
    }


def timed_steps(launches, nc: int, steps: int, stream):
    """Time `steps` steps with a HIP event after every launch (on the launch stream).
    Returns (compress ms, decompress ms, per-launch ms, wall seconds); the first `nc`
    launches are the compress direction."""
    import torch

    ev = [[torch.cuda.Event(enable_timing=True) for _ in range(len(launches) + 1)] for _ in range(steps)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for k in range(steps):
        ev[k][0].record(stream)
        for i, (plan, name) in enumerate(launches):
            plan.launch(name)
            ev[k][i + 1].record(stream)
    torch.cuda.synchronize()
    wall = time.perf_counter() - t0
    per_i = [sum(ev[k][i].elapsed_time(ev[k][i + 1]) for k in range(steps)) / steps for i in range(len(launches))]
    return sum(per_i[:nc]), sum(per_i[nc:]), per_i, wall


def _sysfs_clocks() -> dict:
    """Current shader / memory clock levels from the amdgpu sysfs tables, where readable."""
    out = {}
    for card in sorted(Path("/sys/class/drm").glob("card*/device")):
        for key in ("pp_dpm_sclk", "pp_dpm_mclk", "pp_dpm_fclk"):
            try:
                rows = (card / key).read_text().splitlines()
            except OSError:
                continue
            cur = [r.split(":", 1)[1].strip().rstrip("*").strip() for r in rows if r.rstrip().endswith("*")]
            if cur:
                out[key[7:]] = cur[0]
        if out:
            break
    return out


def settle_curve(step, launches, nc: int, args) -> dict:
    """Step time against time under load from an idle device: after a 0.5 s pause, run
    windows of 8 steps back to back for about 300 ms and report each window's mean
    compress / decompress time (HIP events) and its start time since the load began,
    with the amdgpu sysfs clock levels read after the window where the box exposes them."""
    import torch

    stream = torch.cuda.current_stream()
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    time.sleep(0.5)
    rows, t_start = [], time.perf_counter()
    while time.perf_counter() - t_start < 0.3:
        t_w = (time.perf_counter() - t_start) * 1e3
        t_c, t_d, _, _ = timed_steps(launches, nc, 8, stream)
        rows.append({"t_ms": round(t_w, 2), "compress_ms": round(t_c, 4), "decompress_ms": round(t_d, 4),
                     **_sysfs_clocks()})
    return {"settle_curve": rows, "window_steps": 8, "workload": args.workload}


def settle_device(step, settle_ms: float) -> int:
    """Run untimed steps back to back for `settle_ms` of wall time before the warmup and
    return how many ran.  From an idle device the step time falls over the first ~40 ms
    of load and is flat afterwards (config 2: compress 0.49 -> 0.41 ms, decompress 0.30
    -> 0.28 ms) while the shader clock keeps falling (2.36 -> 2.07 GHz over 300 ms) and
    the memory clock stays at 2.0 GHz: a memory / fabric-side transient, which a few
    warmup steps alone would time instead of the sustained rate a serving loop sees
    (bench.py --settle-curve prints the curve).  The same timed steps are also run
    before this phase and reported as "unsettled"."""
    import torch

    n = 0
    if settle_ms <= 0:
        return n
    t_end = time.perf_counter() + settle_ms / 1e3
    while True:
        step()
        n += 1
        if n % 8 == 0:
            torch.cuda.synchronize()
            if time.perf_counter() >= t_end:
                return n


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=20)
    ap.add_argument("--warmup", type=int, default=5)
    ap.add_argument("--settle-ms", type=float, default=150.0,
                    help="untimed back-to-back steps for this long before the warmup (device clocks settle)")
    ap.add_argument("--cpu-budget", type=float, default=12.0, help="seconds of CPU-oracle work")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--layers", type=int, default=32, help="(debug) layers of the config-2 request")
    ap.add_argument("--heads", type=int, default=8,
                    help="KV heads of the config-2 request (other than 8: a wide-head variant, not the metric's config)")
    ap.add_argument("--head-dim", type=int, default=128,
                    help="head_dim of the config-2 request (other than 128: a variant, not the metric's config)")
    ap.add_argument("--layout", default="permuted", choices=["permuted", "native"],
                    help="(config2) symbol order of the stream, KVSERVE_CODEC_LAYOUT (native: a variant, "
                         "not the metric's config)")
    ap.add_argument("--axes", default="channel,token",
                    help="(config2) axis_key,axis_value of the quantizer (other than channel,token: the "
                         "generic row kernels, a variant, not the metric's config)")
    ap.add_argument("--config3-pools", default="distinct", choices=["distinct", "aliased"],
                    help="(config3) distinct: one 32768-block pool per layer (64 GiB), every layer its own "
                         "memory; aliased: 32 logical 262144-block layer pools over 2 physical ones, so 16 "
                         "layers read the same blocks and some compress reads hit the caches (a variant)")
    ap.add_argument("--workload", default="config2", choices=sorted(WORKLOADS),
                    help="BASELINE.json configuration to time (the metric is quoted on config2)")
    ap.add_argument("--rt-block-size", type=int, default=1, help="(runtime) tokens per block; 1 = token view")
    ap.add_argument("--rt-blocks", type=int, default=1024, help="(runtime) blocks per chunk")
    ap.add_argument("--rt-layers", type=int, default=28, help="(runtime) layers")
    ap.add_argument("--compress-path", default=None, choices=["two_pass", "one_pass"],
                    help="compress kernels: two_pass (the engine's default) or one_pass "
                         "(kvmi_compress_paged, K read once)")
    ap.add_argument("--settle-curve", action="store_true",
                    help="only print the per-window step times over the first ~300 ms of load after idle")
    ap.add_argument("--copy-calibration", action="store_true",
                    help="only run a 1 GiB device-to-device copy --steps times (scales rocprof byte counters)")
    args = ap.parse_args()
    if args.gpus != 1:
        print(f"bench.py measures one GPU only (this build has no multi-GPU path); got --gpus {args.gpus}",
              file=sys.stderr)
        return 2

    import torch

    if args.workload in ("connector", "config2_ans", "runtime", "config2_v3", "bitpack"):
        torch.cuda.set_device(0)
        fn = {"connector": bench_connector, "config2_ans": bench_entropy, "runtime": bench_runtime,
              "config2_v3": bench_fused_v3, "bitpack": bench_bitpack}[args.workload]
        print(json.dumps(fn(args)), flush=True)
        return 0

    if args.copy_calibration:
        src = torch.empty(1 << 30, dtype=torch.uint8, device="cuda").fill_(1)
        dst = torch.empty_like(src)
        for _ in range(args.steps):
            dst.copy_(src)
        torch.cuda.synchronize()
        print(json.dumps({"copy_bytes": src.numel(), "steps": args.steps}))
        return 0

    from kvserve_amd import workloads
    from kvserve_amd.engine import FusedKVCodec

    dev = torch.device("cuda", 0)
    torch.cuda.set_device(dev)
    print(f"bench: building {args.workload} workload", file=sys.stderr, flush=True)
    if args.workload == "config2":
        wl = workloads.make_config2(device=dev, num_layers=args.layers, num_heads=args.heads, head_dim=args.head_dim)
    elif args.workload == "config3":
        wl = (workloads.make_config3(device=dev, pool_blocks=32768, physical_pools=32)
              if args.config3_pools == "distinct" else workloads.make_config3(device=dev))
    else:
        wl = getattr(workloads, "make_" + args.workload)(device=dev)
    reqs = wl.requests
    S, H, D, bits = wl.block_size, wl.num_heads, wl.head_dim, wl.bits
    axes = tuple(a.strip() for a in args.axes.split(","))
    if args.config3_pools != "distinct" and args.workload != "config3":
        raise SystemExit("--config3-pools applies to the config3 workload only")
    if (axes != ("channel", "token") or args.layout != "permuted") and args.workload != "config2":
        raise SystemExit("--axes and --layout apply to the config2 workload only")
    codec = FusedKVCodec(H, D, S, bits, wl.seed, compress_path=args.compress_path, axes=axes, layout=args.layout)
    if len(reqs) == 1:
        req = reqs[0]
        cplan = codec.plan_compress(req.pools, req.block_ids, req.profiles, req.layer_ids)
        packets = [cplan.packet]
        dplan = codec.plan_decompress(cplan.packet, req.pools, req.block_ids)
    else:
        # one launch per kernel for all requests; decompress writes back in place
        cplan = codec.plan_compress_batch([(r.pools, r.block_ids, r.profiles, r.layer_ids) for r in reqs])
        packets = cplan.packets
        dplan = codec.plan_decompress_batch([(pk, r.pools, r.block_ids) for pk, r in zip(packets, reqs)])
    # first run of each plan: a device block table is checked by it (kvmi_check_block_ids
    # runs on a plan's first run only), so the timed steps enqueue the kernels alone
    cplan.run()
    dplan.run()
    torch.cuda.synchronize()
    cplan.check_errors()

    stream = torch.cuda.current_stream()
    launches = [(cplan, n) for n in cplan.launches()] + [(dplan, n) for n in dplan.launches()]
    nc = len(cplan.launches())
    step = lambda: [plan.launch(name) for plan, name in launches]
    if args.settle_curve:
        print(json.dumps(settle_curve(step, launches, nc, args)), flush=True)
        return 0
    print(f"bench: warmup {args.warmup} steps", file=sys.stderr, flush=True)
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    # the same timing before the settle phase (clocks still ramping under the new load)
    t_c_cold, t_d_cold, _, _ = timed_steps(launches, nc, args.steps, stream)
    settle = settle_device(step, args.settle_ms)
    torch.cuda.synchronize()

    print(f"bench: timing {args.steps} steps", file=sys.stderr, flush=True)
    t_c, t_d, per_i, wall = timed_steps(launches, nc, args.steps, stream)
    cplan.check_errors()
    dplan.check_errors()
    per = {}
    for i, (_, name) in enumerate(launches):
        per[name] = per.get(name, 0.0) + per_i[i]

    R = sum(len(r.pools) * 2 * r.block_ids.numel() * S * H * D * 2 for r in reqs)
    P = sum(pk.compressed_bytes() for pk in packets)
    M = sum((pk.kmeta.numel() + pk.vmeta.numel()) * 2 for pk in packets)
    idx = sum(len(r.pools) * r.block_ids.numel() * 4 for r in reqs)
    alg = R + P + M + idx  # one direction: read KV + write stream/meta (or the reverse)
    comp_gbps, dec_gbps = R / t_c / 1e6, R / t_d / 1e6
    comp_frac, dec_frac = alg / t_c / 1e6 / HBM_PEAK_GBPS, alg / t_d / 1e6 / HBM_PEAK_GBPS
    dom = max(per, key=per.get)
    names = hip_kernel_names(codec, S, H, D, bits, cplan)
    dom_kernel = names.get(dom, dom)
    achieved = alg / per[dom] / 1e6
    ms_step = wall / args.steps * 1e3

    out = {
        "metric": METRIC,
        "value": round(R / ((t_c + t_d) / 1e3) / 1e9, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "settle_steps": settle,
        "ms_per_step": round(ms_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic (seeded N(0,1) KV, 4 outlier K channels/head x10)",
        "config": {
            "workload": WORKLOADS[args.workload] + (f" [variant: {H} KV heads, head_dim {D}]"
                                                    if args.workload == "config2" and (H, D) != (8, 128) else "")
                        + (f" [variant: axis_key {axes[0]}, axis_value {axes[1]}]"
                           if axes != ("channel", "token") else "")
                        + (f" [variant: {args.layout} symbol order]" if args.layout != "permuted" else "")
                        + (" [variant: 262144-block layer pools aliasing 2 physical pools]"
                           if args.workload == "config3" and args.config3_pools == "aliased" else ""),
            "requests": len(reqs), "layers": len(reqs[0].pools),
            "tokens": sum(r.block_ids.numel() for r in reqs) * S, "raw_bytes": R, "packed_bytes": P,
            "meta_bytes": M,
        },
        "compress_gbps": round(comp_gbps, 2),
        "decompress_gbps": round(dec_gbps, 2),
        "compress_hbm_frac": round(comp_frac, 4),
        "decompress_hbm_frac": round(dec_frac, 4),
        # the same steps timed right after the warmup, before the settle phase
        "unsettled": {"compress_hbm_frac": round(alg / t_c_cold / 1e6 / HBM_PEAK_GBPS, 4),
                      "decompress_hbm_frac": round(alg / t_d_cold / 1e6 / HBM_PEAK_GBPS, 4),
                      "compress_ms": round(t_c_cold, 4), "decompress_ms": round(t_d_cold, 4)},
        # the same times over the bytes the kernels actually move (rocprofv3 FETCH_SIZE /
        # WRITE_SIZE per dispatch, copy-calibrated): compress reads K twice
        "compress_traffic_hbm_frac": traffic_frac(compress_kernels(names, cplan), t_c / 1e3, args.workload),
        "decompress_traffic_hbm_frac": traffic_frac([names["kvmi_decode_paged"]], t_d / 1e3, args.workload),
        "kernel_ms": {k: round(v, 4) for k, v in per.items()},
        "roofline": {
            "bound": "hbm",
            "kernel": dom_kernel,
            "achieved": round(achieved, 1),
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": round(achieved / HBM_PEAK_GBPS, 4),
            "traffic": profiled_traffic(dom_kernel, args.workload),
            "algorithmic_bytes_per_launch": alg,
        },
        "cpu_baseline": None,
    }
    if not args.no_cpu_baseline and args.workload == "config2":
        print("bench: CPU oracle baseline", file=sys.stderr, flush=True)
        out["cpu_baseline"] = cpu_baseline(wl, args.cpu_budget)
    print(json.dumps(out), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
