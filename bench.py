"""Throughput benchmark of the LCT codec hot path on one MI355X.

Workload (the north-star configuration): randn(16384, 8192) with CPU seed 0,
cast to BF16 (256 MiB), Distribution(GAUSSIAN), CLEAN layout.  A step is one
decompression of the whole tensor through the public API; compression is
timed the same way.  Inputs stay resident in HBM; two input/compressed sets
alternate and three output blocks are written in turn, so the 256 MB Infinity
Cache can neither serve repeated reads nor absorb repeated writes.

Prints one JSON line: ``value`` is decompression throughput in GB/s of
uncompressed BF16 (2n bytes / time), with compression throughput, the
compression ratio, the decoder kernel's roofline fraction (``roofline``), the
one-launch compress kernel's (``encode_roofline``: center sampling, encoder
and overflow bookkeeping), config C2 (an 8192x8192 weight-like tensor, MEDIUM
layout: ``config2``), config C3 (a sparse activation-like tensor with forced
overflow in a shared 64 MiB buffer: ``config3``), the fused momentum update of
config C4 with its single-pass kernel's roofline (``update``), the weight step of
compressed SGD-momentum with its single-pass kernel's roofline
(``weight_update``), config 5 (a GPT-2-small training step with weights,
activations and Muon momentum compressed, against the same step uncompressed:
``config5``) and a host-core CPU baseline (the C oracle, OpenMP over codec
blocks) beside them.

Usage: python bench.py [--gpus 1] [--steps K] [--warmup W] [--skip-cpu] [--skip-train]
"""
from __future__ import annotations

import argparse
import json
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))

METRIC = "decompress/compress GB/s (BF16 bytes) & % HBM peak; compression ratio"
HBM_PEAK_GBPS = 8000.0   # MI355X HBM3E, 8 TB/s
SHAPE = (16384, 8192)


def _log(message: str) -> None:
    print(f"[bench] {message}", file=sys.stderr, flush=True)


def decode_bytes(ct) -> int:
    """Algorithmic bytes of one decode: payload + side + tails + 2/entry +
    block metadata read, 2n written."""
    B, L, S, W = ct.codec_geometry
    nb = ct.size // B
    count = int(ct.fallback_count.item())
    tails = int(ct.fallback_used.item())
    return nb * L * W * 4 + ct.size + tails + 2 * count + 12 * nb + 2 * ct.logical_numel


def encode_bytes(ct) -> int:
    """Algorithmic bytes of one encode: 2n read; side, payload, extra starts,
    tails, 2/entry and block metadata written."""
    B, L, S, W = ct.codec_geometry
    nb = ct.size // B
    count = int(ct.fallback_count.item())
    tails = int(ct.fallback_used.item())
    return 2 * ct.logical_numel + ct.size + nb * L * W * 4 + nb * L + tails + 2 * count + 12 * nb


TRAFFIC_PROFILE = ROOT / "profiles" / "codec_kernels_NS_C4_traffic.md"


def measured_traffic(kernel: str, workgroups: int):
    """HBM bytes per launch of ``kernel`` at ``workgroups`` workgroups from the
    committed rocprofv3 FETCH_SIZE/WRITE_SIZE summary (calibrated on a 256 MiB
    copy), or None."""
    try:
        for line in TRAFFIC_PROFILE.read_text().splitlines():
            fields = line.split()
            if (len(fields) == 4 and fields[0] == "traffic_bytes_per_launch"
                    and fields[1] == kernel and int(fields[2]) == workgroups):
                return int(fields[3])
    except (OSError, ValueError):
        pass
    return None


def _time_events(fn, steps: int, warmup: int, torch) -> float:
    """Average milliseconds per call over ``steps`` calls (after warm-up)."""
    for i in range(warmup):
        fn(i)
    torch.cuda.synchronize()
    start = torch.cuda.Event(enable_timing=True)
    end = torch.cuda.Event(enable_timing=True)
    start.record()
    for i in range(steps):
        fn(i)
    end.record()
    torch.cuda.synchronize()
    return start.elapsed_time(end) / steps


# Output sets used in turn by every timed loop: a step never writes the block
# the previous step wrote, so the 256 MB Infinity Cache cannot absorb a
# step's writes (with one output block, reused by the caching allocator after
# each step, it does: the public-API step came out faster than the kernel it
# launches).
ROTATION = 3


def _keeping(make, release=None):
    """A timed-loop body that keeps the last ``ROTATION - 1`` results alive, so
    every call's outputs come from a block that none of the previous
    ``ROTATION - 1`` calls wrote; ``release`` runs on each result as it drops
    out (after its successor exists)."""
    kept = [None] * (ROTATION - 1)

    def step(i):
        slot = i % len(kept)
        old = kept[slot]
        kept[slot] = make(i)
        if old is not None and release is not None:
            release(old)

    def drain():
        """Release and drop the results still kept."""
        for slot, old in enumerate(kept):
            if old is not None and release is not None:
                release(old)
            kept[slot] = None

    step.drain = drain
    return step


def _kernel_ms(launch, steps: int, torch, rounds: int = 3) -> float:
    """Average duration of back-to-back launches, bracketed by one event pair
    recorded on the stream the kernel is launched on (torch's current stream,
    which dispatch passes to the library); the median of ``rounds`` rounds of
    ``steps`` launches."""
    stream = torch.cuda.current_stream()
    results = []
    for _ in range(rounds):
        torch.cuda.synchronize()
        start = torch.cuda.Event(enable_timing=True)
        end = torch.cuda.Event(enable_timing=True)
        start.record(stream)
        for i in range(steps):
            launch(i)
        end.record(stream)
        end.synchronize()
        results.append(start.elapsed_time(end) / steps)
    return sorted(results)[len(results) // 2]


# Wall time of the warm-up before each workload's timed loops.
WARM_UP_S = 0.3


def _warm_up(work, seconds: float, torch) -> None:
    """Keep the GPU busy with ``work`` for ``seconds`` of wall time, so that
    clocks and memory mappings have settled before anything is timed (the
    first timed loop on a fresh box otherwise runs up to 12% slow)."""
    deadline = time.perf_counter() + seconds
    i = 0
    while time.perf_counter() < deadline:
        for _ in range(8):
            work(i)
            i += 1
        torch.cuda.synchronize()


def cpu_baseline(x_cpu, dist, min_seconds: float):
    """Time the C oracle (OpenMP over blocks) compress + decompress on host cores."""
    import numpy as np

    import oracle
    from losslessly_compressed_tensors_amd.compression.huffman_tables import distribution_codebook

    book = distribution_codebook(dist)
    geometry = oracle.geometry_of("gaussian", "clean")
    bits = x_cpu.view(-1).view(__import__("torch").int16).numpy()
    nbytes = 2 * bits.size

    def timed(seconds):
        reps = 0
        enc_s = dec_s = 0.0
        restored = None
        while reps < 2 or enc_s + dec_s < seconds:
            t0 = time.perf_counter()
            compressed = oracle.compress(bits, geometry, book.encode, book.decode,
                                         book.rare_length)
            t1 = time.perf_counter()
            restored = oracle.decompress(compressed)
            t2 = time.perf_counter()
            enc_s += t1 - t0
            dec_s += t2 - t1
            reps += 1
        assert np.array_equal(restored, bits.view(np.uint16))
        return reps, enc_s, dec_s

    cores = oracle.num_threads()
    reps, enc_s, dec_s = timed(min_seconds)
    # The same on one thread, over a shorter window.
    oracle.set_num_threads(1)
    try:
        reps1, enc1, dec1 = timed(min_seconds / 4)
    finally:
        oracle.set_num_threads(cores)
    return {
        "value": round(nbytes * reps / dec_s / 1e9, 3),
        "unit": "GB/s",
        "cores": cores,
        "kind": "port",
        "sample": f"full workload tensor ({bits.size} BF16), {reps} decompressions "
                  f"({dec_s:.1f} s) and compressions ({enc_s:.1f} s) on {cores} threads; "
                  f"{reps1} of each ({dec1:.1f} s, {enc1:.1f} s) on 1 thread",
        "compress_value": round(nbytes * reps / enc_s / 1e9, 3),
        "one_thread_value": round(nbytes * reps1 / dec1 / 1e9, 3),
        "one_thread_compress_value": round(nbytes * reps1 / enc1 / 1e9, 3),
    }


def time_update(args, torch, device):
    """Config C4: m <- 0.95*m + g on a compressed 4096x11008 momentum
    (EMPIRICAL CLEAN, buffer-backed so no step syncs), m0 ~ N(0, 1e-3^2) seed 4,
    g ~ N(0, 1e-2^2) seeds 100, 101, 102 in turn.  Reports the step time, the
    BF16 throughput 2n/t and the fraction of HBM peak that the single-pass
    minimum traffic (payload + side + 2n read, side + payload written) would
    need at that time."""
    from losslessly_compressed_tensors_amd.comp_format import DistType, Distribution
    from losslessly_compressed_tensors_amd.LCTensor import LCTTensor
    from losslessly_compressed_tensors_amd.operations import decompress
    from losslessly_compressed_tensors_amd.tensor_buffer import TensorBuffer

    shape = (4096, 11008)
    gen = torch.Generator().manual_seed(4)
    m0 = (torch.randn(*shape, generator=gen) * 1e-3).to(torch.bfloat16).to(device)
    # Three gradients in turn: a gradient's 90 MB come back after three steps
    # (about 650 MB of traffic), past the 256 MB Infinity Cache.
    grads = []
    for seed in (100, 101, 102):
        gen = torch.Generator().manual_seed(seed)
        grads.append((torch.randn(*shape, generator=gen) * 1e-2).to(torch.bfloat16).to(device))
    dist = Distribution(DistType.EMPIRICAL)
    buffer = TensorBuffer(64 << 20, device=device)
    # Three copies of the momentum are updated in turn, so consecutive steps
    # touch different device blocks.
    momenta = [LCTTensor(m0, buffer, dist) for _ in range(ROTATION)]
    alpha = torch.tensor([0.95], dtype=torch.float32, device=device)
    steps = max(10, args.steps // 2)
    # The host-side set-up above leaves the GPU idle for seconds; decompressing
    # the momenta (which leaves them unchanged) settles the clocks first.
    _warm_up(lambda i: decompress(momenta[i % ROTATION].x), WARM_UP_S, torch)
    ms = _time_events(lambda i: momenta[i % ROTATION].mul_add_(alpha, grads[i % len(grads)]),
                      steps,
                      args.warmup, torch)
    ct = momenta[0].x
    B, L, S, W = ct.codec_geometry
    nb = ct.size // B
    n = ct.logical_numel
    minimum = 2 * (nb * L * W * 4 + ct.size) + 2 * n

    # The single-pass kernel alone, launched back to back on the final
    # momentum with outputs preallocated: reads A's payload and side bytes and
    # B, writes the result's side bytes, payload, extra starts and summaries.
    from losslessly_compressed_tensors_amd.codec.decode import overlay_of, shifted_decode_table
    from losslessly_compressed_tensors_amd.compression.huffman_tables import (
        get_distribution_tables,
    )
    from losslessly_compressed_tensors_amd.kernels import dispatch

    base_encode, base_decode, rare = get_distribution_tables(dist, device)
    sample_size = min(n, 4096)
    launch = dict(rare_length=rare, logical_numel=n, block_symbols=B, lanes=L, steps=S,
                  fixed_words=W, op=2, alpha_is_one=False, beta_is_one=True,
                  sample_size=sample_size, overflow=overlay_of(ct))
    sets = []
    for momentum in momenta:
        a = momentum.x
        table = shifted_decode_table(a)
        partials = torch.empty(2 * -(-sample_size // 64), dtype=torch.int32, device=device)
        dispatch.pointwise_sample(a.data, a.sign_mantissa, table, a.center, grads[0], alpha,
                                  None, partials, a.size, a_samples=a.sample_values,
                                  **{**launch, "overflow": overlay_of(a)})
        sets.append(dict(
            a=a, table=table, partials=partials, overflow=overlay_of(a),
            center=torch.empty(1, dtype=torch.int32, device=device),
            shifted=torch.empty(1024, dtype=torch.int32, device=device),
            side=torch.empty(a.size, dtype=torch.uint8, device=device),
            encoded=torch.empty(nb * L * W + 4, dtype=torch.int32, device=device),
            extra=torch.empty(nb * L, dtype=torch.uint8, device=device),
            summaries=torch.empty(5 * nb + 1, dtype=torch.int32, device=device),
            exponents=torch.empty(n, dtype=torch.uint8, device=device)))

    def launch_fused(i):
        o = sets[i % ROTATION]
        a = o["a"]
        dispatch.pointwise_encode(a.data, a.sign_mantissa, o["table"], a.center,
                                  grads[i % len(grads)],
                                  alpha, None, o["partials"], base_encode, base_decode,
                                  o["center"], o["shifted"], o["side"], o["encoded"], o["extra"],
                                  o["summaries"], o["exponents"], a.size,
                                  **{**launch, "overflow": o["overflow"]})

    _warm_up(launch_fused, WARM_UP_S, torch)
    fused_ms = _kernel_ms(launch_fused, steps, torch)
    fused_alg = minimum + nb * L + 8 * nb
    return {
        "workload": "C4: 4096x11008, EMPIRICAL CLEAN, LCTTensor.mul_add_(0.95, g), buffered",
        "steps": steps,
        "ms_per_step": round(ms, 5),
        "gbps": round(2 * n / (ms * 1e-3) / 1e9, 2),
        "single_pass_bytes": minimum,
        "single_pass_hbm_frac": round(minimum / (ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
        "kernel_roofline": {
            "kernel": "pointwise_encode_kernel",
            "kernel_us": round(fused_ms * 1e3, 2),
            "algorithmic_bytes": fused_alg,
            "achieved": round(fused_alg / (fused_ms * 1e-3) / 1e9, 1),
            "frac": round(fused_alg / (fused_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
            "traffic": measured_traffic("pointwise_encode_kernel<false>", nb),
        },
    }


def time_weight_update(args, torch, device):
    """The weight half of the compressed SGD-momentum step
    (LCT/components/sparse_utils.py:52-54): p <- p + (-lr) * m with both the
    weight p and the momentum m compressed, at config C4's shape 4096x11008.
    p ~ N(0, 0.02^2) seed 5 under the reference's weight distribution (LAPLACE
    CLEAN), m ~ N(0, 1e-2^2) seed 100 under its momentum distribution
    (EMPIRICAL CLEAN, zero_prob 0.02), both buffer-backed; lr = 0.01.  Reports
    the step time and the single-pass kernel's roofline (reads both operands'
    payload and side bytes, writes the result's)."""
    from losslessly_compressed_tensors_amd.codec.decode import overlay_of, shifted_decode_table
    from losslessly_compressed_tensors_amd.comp_format import DistType, Distribution
    from losslessly_compressed_tensors_amd.compression.huffman_tables import (
        get_distribution_tables,
    )
    from losslessly_compressed_tensors_amd.kernels import dispatch
    from losslessly_compressed_tensors_amd.LCTensor import LCTTensor
    from losslessly_compressed_tensors_amd.operations import decompress
    from losslessly_compressed_tensors_amd.tensor_buffer import TensorBuffer

    shape = (4096, 11008)
    gen = torch.Generator().manual_seed(5)
    p0 = (torch.randn(*shape, generator=gen) * 0.02).to(torch.bfloat16).to(device)
    gen = torch.Generator().manual_seed(100)
    m0 = (torch.randn(*shape, generator=gen) * 1e-2).to(torch.bfloat16).to(device)
    weight_dist = Distribution(DistType.LAPLACE)
    momentum_dist = Distribution(DistType.EMPIRICAL, zero_prob=0.02)
    buffer = TensorBuffer(96 << 20, device=device)
    # Three weight/momentum pairs are stepped in turn, so consecutive steps
    # touch different device blocks.
    pairs = [(LCTTensor(p0, buffer, weight_dist), LCTTensor(m0, buffer, momentum_dist))
             for _ in range(ROTATION)]
    neg_lr = torch.tensor([-0.01], dtype=torch.float32, device=device)
    steps = max(10, args.steps // 2)

    def weight_step(i):
        weight, momentum = pairs[i % ROTATION]
        weight.add_comp_(momentum, neg_lr)

    _warm_up(lambda i: decompress(pairs[i % ROTATION][i % 2].x), WARM_UP_S, torch)
    ms = _time_events(weight_step, steps, args.warmup, torch)

    b = pairs[0][0].x
    B, L, S, W = b.codec_geometry
    nb = b.size // B
    n = b.logical_numel
    base_encode, base_decode, rare = get_distribution_tables(weight_dist, device)
    sample_size = min(n, 4096)
    launch = dict(rare_length=rare, logical_numel=n, block_symbols=B, lanes=L, steps=S,
                  fixed_words=W, sample_size=sample_size)
    sets = []
    for weight, momentum in pairs:
        a, b = momentum.x, weight.x
        tables = shifted_decode_table(a), shifted_decode_table(b)
        storages = overlay_of(a), overlay_of(b)
        partials = torch.empty(2 * -(-sample_size // 64), dtype=torch.int32, device=device)
        dispatch.dual_sample(a.data, a.sign_mantissa, tables[0], a.center, storages[0], b.data,
                             b.sign_mantissa, tables[1], b.center, storages[1], neg_lr,
                             partials, b.size, a_samples=a.sample_values,
                             b_samples=b.sample_values, **launch)
        sets.append(dict(
            a=a, b=b, tables=tables, storages=storages, partials=partials,
            center=torch.empty(1, dtype=torch.int32, device=device),
            shifted=torch.empty(1024, dtype=torch.int32, device=device),
            side=torch.empty(b.size, dtype=torch.uint8, device=device),
            encoded=torch.empty(nb * L * W + 4, dtype=torch.int32, device=device),
            extra=torch.empty(nb * L, dtype=torch.uint8, device=device),
            summaries=torch.empty(5 * nb + 1, dtype=torch.int32, device=device),
            exponents=torch.empty(n, dtype=torch.uint8, device=device)))

    def launch_fused(i):
        o = sets[i % ROTATION]
        a, b, tables, storages = o["a"], o["b"], o["tables"], o["storages"]
        dispatch.dual_encode(a.data, a.sign_mantissa, tables[0], a.center, storages[0], b.data,
                             b.sign_mantissa, tables[1], b.center, storages[1], neg_lr,
                             o["partials"], base_encode, base_decode, o["center"], o["shifted"],
                             o["side"], o["encoded"], o["extra"], o["summaries"],
                             o["exponents"], b.size, **launch)

    _warm_up(launch_fused, WARM_UP_S, torch)
    fused_ms = _kernel_ms(launch_fused, steps, torch)
    stream_bytes = nb * L * W * 4 + b.size
    fused_alg = 3 * stream_bytes + nb * L + 8 * nb
    return {
        "workload": "SGD-momentum weight step at C4's shape: 4096x11008, weight LAPLACE CLEAN, "
                    "momentum EMPIRICAL CLEAN, LCTTensor.add_comp_(m, -0.01), buffered",
        "steps": steps,
        "ms_per_step": round(ms, 5),
        "gbps": round(2 * n / (ms * 1e-3) / 1e9, 2),
        "kernel_roofline": {
            "kernel": "dual_encode_kernel",
            "kernel_us": round(fused_ms * 1e3, 2),
            "algorithmic_bytes": fused_alg,
            "achieved": round(fused_alg / (fused_ms * 1e-3) / 1e9, 1),
            "frac": round(fused_alg / (fused_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
            "traffic": measured_traffic("dual_encode_kernel<false>", nb),
        },
    }


def time_bandwidth(args, torch, device, read_bytes: int, write_bytes: int):
    """Attainable HBM bandwidth with the codec kernels' access shape
    (``lct_bandwidth_probe``: 16-byte non-temporal buffer accesses, 16 KiB per
    workgroup pass): a 256 MiB copy, read-only and write-only passes, and a
    pass that reads ``read_bytes`` while it writes ``write_bytes`` (the NS
    decoder's mix).  Two sources and three destinations are used in turn, so
    the Infinity Cache serves nothing; each figure is the best over 1024, 2048
    and 4096 workgroups (the median of three rounds each)."""
    from losslessly_compressed_tensors_amd.kernels import hip

    size = 256 << 20
    mix_read = read_bytes // 16 * 16
    mix_write = write_bytes // 16 * 16
    srcs = [torch.empty(size, dtype=torch.uint8, device=device).random_(0, 256)
            for _ in range(2)]
    dsts = [torch.empty(max(size, mix_write), dtype=torch.uint8, device=device)
            for _ in range(ROTATION)]
    stream = torch.cuda.current_stream().cuda_stream
    cases = {
        "copy_gbps": (0, size, size, 2 * size),
        "read_gbps": (1, size, 4096, size),
        "write_gbps": (2, 0, size, size),
        "decoder_mix_gbps": (3, mix_read, mix_write, mix_read + mix_write),
    }
    out = {"workload": f"256 MiB copy, read and write passes; mix: {mix_read} B read with "
                       f"{mix_write} B written (the NS decode's bytes)"}
    for name, (kind, src_bytes, dst_bytes, moved) in cases.items():
        best = None
        for workgroups in (1024, 2048, 4096):
            def launch(i):
                src = srcs[i % 2].data_ptr() if kind != 2 else None
                hip.call("lct_bandwidth_probe", kind, src, src_bytes,
                         dsts[i % ROTATION].data_ptr(), dst_bytes, workgroups, stream)

            _warm_up(launch, 0.05, torch)
            ms = _kernel_ms(launch, max(10, args.steps), torch)
            best = ms if best is None else min(best, ms)
        out[name] = round(moved / (best * 1e-3) / 1e9, 1)
    return out


def time_config2(args, torch, device):
    """a weight-like 8192x8192 BF16 tensor,
    randn * 0.02 with CPU seed 1, Distribution(GAUSSIAN) MEDIUM layout (the
    family's unit shape: the sampled center absorbs the 0.02 scale); compress
    (buffered, the previous result freed) and decompress timed separately
    through the public API.  Two sets alternate."""
    from losslessly_compressed_tensors_amd.comp_format import DistType, Distribution, NoiseLevel
    from losslessly_compressed_tensors_amd.operations import compress, decompress
    from losslessly_compressed_tensors_amd.tensor_buffer import TensorBuffer

    dist = Distribution(DistType.GAUSSIAN, noise_level=NoiseLevel.MEDIUM)
    xs = []
    for seed in (1, 2):
        gen = torch.Generator().manual_seed(seed)
        xs.append((torch.randn(8192, 8192, generator=gen) * 0.02).to(torch.bfloat16).to(device))
    buffer = TensorBuffer(64 << 20, device=device)
    cts = [compress(x, dist, buffer=buffer) for x in xs]
    for ct, x in zip(cts, xs):
        if not torch.equal(decompress(ct).view(torch.int16), x.view(torch.int16)):
            raise AssertionError("config C2 round trip is not bit-exact")
    nbytes = 2 * xs[0].numel()
    # The reference times 100 iterations after warm-up
    # (examples/benchmarks/benchmark_lct.py:17-18).
    steps, warmup = max(100, args.steps), max(10, args.warmup)
    _warm_up(_keeping(lambda i: decompress(cts[i % 2])), WARM_UP_S, torch)
    dec_ms = _time_events(_keeping(lambda i: decompress(cts[i % 2])), steps, warmup, torch)
    enc_ms = _time_events(_keeping(lambda i: compress(xs[i % 2], dist, buffer=buffer),
                                   release=lambda ct: ct.free()),
                          steps, warmup, torch)
    dec_alg, enc_alg = decode_bytes(cts[0]), encode_bytes(cts[0])
    return {
        "workload": "C2: randn(8192, 8192) * 0.02, CPU seed 1, BF16 (128 MiB); "
                    "Distribution(GAUSSIAN) MEDIUM; public API, buffered",
        "steps": steps,
        "warmup": warmup,
        "geometry": list(cts[0].codec_geometry),
        "compression_ratio": round(nbytes / cts[0].memory_size(), 5),
        "decompress_gbps": round(nbytes / (dec_ms * 1e-3) / 1e9, 2),
        "decompress_hbm_frac": round(dec_alg / (dec_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
        "compress_gbps": round(nbytes / (enc_ms * 1e-3) / 1e9, 2),
        "compress_hbm_frac": round(enc_alg / (enc_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
    }


def time_config3(args, torch, device):
    """an activation-like 8x2048x4096 BF16 tensor,
    relu(randn) with CPU seed 2 (about half exact zeros), 0.1% of its entries
    (randperm with CPU seed 3) scaled by 1e4 in FP32 to force escapes and
    stream overflow; Distribution(LAPLACE, 1.0, zero_prob=0.5) SPARSE in a
    64 MiB TensorBuffer.  A step is the config's compress, decompress, free
    sequence through the public API; compress+free and decompress are also
    timed on their own.  Two sets alternate (the second from seeds 4 and 5)."""
    from losslessly_compressed_tensors_amd.comp_format import (
        DistType, Distribution, NoiseLevel,
    )
    from losslessly_compressed_tensors_amd.operations import compress, decompress
    from losslessly_compressed_tensors_amd.tensor_buffer import (
        TensorBuffer, _free_regions_snapshot, verify_buffer,
    )

    dist = Distribution(DistType.LAPLACE, 1.0, zero_prob=0.5, noise_level=NoiseLevel.SPARSE)
    xs = []
    for seed, perm_seed in ((2, 3), (4, 5)):
        z = torch.relu(torch.randn(8, 2048, 4096, generator=torch.Generator().manual_seed(seed)))
        n = z.numel()
        idx = torch.randperm(n, generator=torch.Generator().manual_seed(perm_seed))[: n // 1000]
        z.view(-1)[idx] *= 1e4
        xs.append(z.to(torch.bfloat16).to(device))
    buffer = TensorBuffer(64 << 20, device=device)
    cts = [compress(x, dist, buffer=buffer) for x in xs]
    for ct, x in zip(cts, xs):
        if not torch.equal(decompress(ct).view(torch.int16), x.view(torch.int16)):
            raise AssertionError("config C3 round trip is not bit-exact")
    nbytes = 2 * xs[0].numel()
    overflow_streams = int(cts[0].fallback_count.item())
    tail_bytes = int(cts[0].fallback_used.item())
    ratio = nbytes / cts[0].memory_size()
    dec_alg, enc_alg = decode_bytes(cts[0]), encode_bytes(cts[0])
    _warm_up(_keeping(lambda i: decompress(cts[i % 2])), WARM_UP_S, torch)
    dec_ms = _time_events(_keeping(lambda i: decompress(cts[i % 2])), args.steps, args.warmup,
                          torch)
    for ct in cts:
        ct.free()

    def sequence(i):
        ct = compress(xs[i % 2], dist, buffer=buffer)
        out = decompress(ct)
        ct.free()
        return ct, out

    compress_step = _keeping(lambda i: compress(xs[i % 2], dist, buffer=buffer),
                             release=lambda ct: ct.free())
    enc_ms = _time_events(compress_step, args.steps, args.warmup, torch)
    compress_step.drain()
    # The sequence frees each tensor's tails itself; the results are kept
    # only so their device blocks rotate.
    seq_ms = _time_events(_keeping(sequence), args.steps, args.warmup, torch)
    torch.cuda.synchronize()
    verify_buffer(buffer)
    regions = _free_regions_snapshot(buffer)
    if len(regions) != 1:
        raise AssertionError(f"config C3 left {len(regions)} free regions, expected 1")
    return {
        "workload": "C3: relu(randn(8, 2048, 4096)), CPU seed 2, 0.1% of entries x 1e4 "
                    "(randperm seed 3), BF16 (128 MiB); Distribution(LAPLACE, 1.0, "
                    "zero_prob=0.5) SPARSE; 64 MiB TensorBuffer; public API",
        "geometry": list(cts[0].codec_geometry),
        "compression_ratio": round(ratio, 5),
        "overflow_streams": overflow_streams,
        "tail_bytes": tail_bytes,
        "decompress_gbps": round(nbytes / (dec_ms * 1e-3) / 1e9, 2),
        "decompress_hbm_frac": round(dec_alg / (dec_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
        "compress_gbps": round(nbytes / (enc_ms * 1e-3) / 1e9, 2),
        "compress_hbm_frac": round(enc_alg / (enc_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
        "sequence_ms": round(seq_ms, 5),
        "sequence_gbps": round(2 * nbytes / (seq_ms * 1e-3) / 1e9, 2),
    }


def time_config5(torch, device, steps: int = 5, warmup: int = 2):
    """one GPT-2-small-shaped training step (12
    layers, width 768, 12 heads, sequence 1024, batch 8, random init, uniform
    random token ids), with weights, activations and Muon momentum compressed
    and without; tokens per second and peak allocated device memory of each
    (examples/nanogpt/train_gpt_lct.py)."""
    from examples.nanogpt import train_gpt_lct as gpt

    runs = {mode: gpt.measure(device, compressed=mode == "lct", steps=steps, warmup=warmup)
            for mode in ("dense", "lct")}
    return {
        "workload": "GPT-2-small step: 12 layers, d_model 768, 12 heads, seq 1024, batch 8 "
                    "(8192 tokens), vocab 50304 (ids < 50257), AdamW + Muon; synthetic tokens",
        "steps": steps,
        "warmup": warmup,
        **runs,
        "tokens_per_s_ratio": round(runs["lct"]["tokens_per_s"] / runs["dense"]["tokens_per_s"], 4),
        "peak_hbm_ratio": round(runs["lct"]["peak_allocated_mib"]
                                / runs["dense"]["peak_allocated_mib"], 4),
        "resident_state_ratio": round(runs["lct"]["resident_state_mib"]
                                      / runs["dense"]["resident_state_mib"], 4),
    }


def main() -> int:
    parser = argparse.ArgumentParser(description=__doc__)
    parser.add_argument("--gpus", type=int, default=1)
    parser.add_argument("--steps", type=int, default=50)
    parser.add_argument("--warmup", type=int, default=5)
    parser.add_argument("--cpu-seconds", type=float, default=12.0)
    parser.add_argument("--skip-cpu", action="store_true")
    parser.add_argument("--skip-train", action="store_true",
                        help="leave out the config-5 training step")
    args = parser.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU only: the codec path has no multi-GPU form here "
              "(codec blocks are independent; a sharded tensor would need only its center "
              "and its overflow totals exchanged). Run with --gpus 1.", file=sys.stderr)
        return 2

    import torch

    from losslessly_compressed_tensors_amd.codec.decode import overlay_of, shifted_decode_table
    from losslessly_compressed_tensors_amd.comp_format import DistType, Distribution
    from losslessly_compressed_tensors_amd.compression.huffman_tables import (
        get_distribution_tables,
    )
    from losslessly_compressed_tensors_amd.kernels import dispatch
    from losslessly_compressed_tensors_amd.operations import compress, decompress
    from losslessly_compressed_tensors_amd.tensor_buffer import TensorBuffer

    if not torch.cuda.is_available():
        print("bench.py needs a GPU", file=sys.stderr)
        return 1
    device = torch.device("cuda", 0)
    dist = Distribution(DistType.GAUSSIAN)
    _log("generating inputs")
    host_inputs = []
    for seed in (0, 1):
        gen = torch.Generator().manual_seed(seed)
        host_inputs.append(torch.randn(*SHAPE, generator=gen).to(torch.bfloat16))
    xs = [h.to(device) for h in host_inputs]
    n = xs[0].numel()
    nbytes = 2 * n

    _log("correctness pass")
    private = compress(xs[0], dist)
    restored = decompress(private)
    if not torch.equal(restored.view(torch.int16), xs[0].view(torch.int16)):
        raise AssertionError("round trip is not bit-exact")
    ratio = nbytes / private.memory_size()

    buffer = TensorBuffer(64 << 20, device=device)
    cts = [compress(x, dist, buffer=buffer) for x in xs]
    for ct, x in zip(cts, xs):
        if not torch.equal(decompress(ct).view(torch.int16), x.view(torch.int16)):
            raise AssertionError("buffered round trip is not bit-exact")

    _log("warming up")
    warm_outputs = _keeping(lambda i: decompress(cts[i % 2]))
    _warm_up(lambda i: (warm_outputs(i), compress(xs[i % 2], dist)), 1.0, torch)
    warm_outputs.drain()

    _log("timing decompress")
    dec_ms = _time_events(_keeping(lambda i: decompress(cts[i % 2])), args.steps, args.warmup,
                          torch)

    # Decoder kernel alone: three preallocated outputs in turn, launches back
    # to back.
    _, _, rare = get_distribution_tables(dist, device)
    B, L, S, W = cts[0].codec_geometry
    outs = [torch.empty(n, dtype=torch.int16, device=device) for _ in range(ROTATION)]

    def launch_decode(i):
        ct = cts[i % 2]
        dispatch.decode_kernel(ct.data, ct.sign_mantissa, outs[i % ROTATION],
                               shifted_decode_table(ct),
                               ct.center, ct.size, logical_numel=n, block_symbols=B, lanes=L,
                               steps=S, fixed_words=W, rare_length=rare, overflow=overlay_of(ct))

    for i in range(args.warmup):
        launch_decode(i)
    back_to_back_ms = _kernel_ms(launch_decode, args.steps, torch)
    # Each headline step is exactly one decode launch and the host issues a
    # step in about 12 us against the kernel's ~80 us, so the GPU never waits
    # for the host: the step time bounds the kernel's duration from above and
    # the roofline below is taken from it.  The back-to-back launches measure
    # the same kernel directly (equal within noise).
    kernel_ms = dec_ms
    dec_alg = decode_bytes(cts[0])

    _log("timing compress")

    enc_ms = _time_events(_keeping(lambda i: compress(xs[i % 2], dist, buffer=buffer),
                                   release=lambda ct: ct.free()),
                          args.steps, args.warmup, torch)
    enc_private_ms = _time_events(_keeping(lambda i: compress(xs[i % 2], dist)),
                                  max(20, args.steps), 2, torch)
    enc_alg = encode_bytes(cts[0])

    # The fused compress kernel alone (center sampling, encoder and overflow
    # bookkeeping in one launch, private form: no arena), launched back to back
    # into preallocated outputs; each launch's words carry a fresh epoch.
    encode_table, decode_table, _ = get_distribution_tables(dist, device)
    nb = n // B
    enc_sets = [dict(side=torch.empty(n, dtype=torch.uint8, device=device),
                     encoded=torch.empty(nb * L * W + 4, dtype=torch.int32, device=device),
                     center=torch.empty(1, dtype=torch.int32, device=device),
                     shifted=torch.empty(1024, dtype=torch.int32, device=device),
                     samples=torch.empty(4096, dtype=torch.int16, device=device),
                     extra=torch.empty(nb * L, dtype=torch.uint8, device=device),
                     summaries=torch.empty(dispatch.summaries_length(nb), dtype=torch.int32,
                                           device=device),
                     counts=torch.empty(4, dtype=torch.int32, device=device),
                     blocks=torch.empty(3 * nb, dtype=torch.int32, device=device))
                for _ in range(ROTATION)]

    def launch_encode(i):
        o = enc_sets[i % ROTATION]
        dispatch.encode_fused(xs[i % 2].view(-1).view(torch.int16), o["side"], o["encoded"],
                              4096, encode_table, decode_table, o["center"], o["shifted"],
                              o["samples"], o["extra"], o["summaries"], o["blocks"], o["counts"],
                              n, precomputed=False, logical_numel=n, block_symbols=B, lanes=L,
                              steps=S, fixed_words=W)

    for i in range(args.warmup):
        launch_encode(i)
    encode_kernel_ms = _kernel_ms(launch_encode, args.steps, torch)

    _log("timing config C2")
    config2 = time_config2(args, torch, device)
    _log("timing config C3")
    config3 = time_config3(args, torch, device)
    _log("timing fused update (C4)")
    update = time_update(args, torch, device)
    _log("timing fused weight update")
    weight_update = time_weight_update(args, torch, device)

    # Reference traffic for counter calibration: a plain 256 MiB device copy
    # (reads and writes exactly 2n bytes each).
    copy_out = torch.empty_like(xs[0])
    copy_ms = _time_events(lambda i: copy_out.copy_(xs[i % 2]), 5, 2, torch)

    _log("timing attainable-bandwidth probes")
    bandwidth = time_bandwidth(args, torch, device, read_bytes=dec_alg - nbytes,
                               write_bytes=nbytes)

    result = {
        "metric": METRIC,
        "value": round(nbytes / (dec_ms * 1e-3) / 1e9, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(dec_ms, 5),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "u32",
        "data": "synthetic",
        "config": {
            "workload": "NS: randn(16384, 8192), CPU seed 0, cast to BF16 (256 MiB); "
                        "Distribution(GAUSSIAN) CLEAN; step = one public-API decompress",
            "elements": n,
            "geometry": [B, L, S, W],
            "sets_rotated": 2,
            "output_sets_rotated": ROTATION,
        },
        "decompress_gbps": round(nbytes / (dec_ms * 1e-3) / 1e9, 2),
        "decompress_hbm_frac": round(dec_alg / (dec_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
        "compress_gbps": round(nbytes / (enc_ms * 1e-3) / 1e9, 2),
        "compress_hbm_frac": round(enc_alg / (enc_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
        "compress_private_gbps": round(nbytes / (enc_private_ms * 1e-3) / 1e9, 2),
        "compress_private_hbm_frac": round(enc_alg / (enc_private_ms * 1e-3) / 1e9
                                           / HBM_PEAK_GBPS, 4),
        "compress_private_ms": round(enc_private_ms, 5),
        "compress_ms": round(enc_ms, 5),
        "compression_ratio": round(ratio, 5),
        "copy_gbps": round(2 * nbytes / (copy_ms * 1e-3) / 1e9, 1),
        "roofline": {
            "bound": "hbm",
            "kernel": "decode_kernel_grouped",
            "achieved": round(dec_alg / (kernel_ms * 1e-3) / 1e9, 1),
            "peak": HBM_PEAK_GBPS,
            "unit": "GB/s",
            "frac": round(dec_alg / (kernel_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
            "traffic": measured_traffic("decode_kernel_grouped", nb),
            "traffic_source": TRAFFIC_PROFILE.relative_to(ROOT).as_posix(),
            "algorithmic_bytes": dec_alg,
            "kernel_us": round(kernel_ms * 1e3, 2),
            "kernel_timing": "headline loop (one decode launch per public-API step)",
            "kernel_us_back_to_back": round(back_to_back_ms * 1e3, 2),
            "frac_back_to_back": round(dec_alg / (back_to_back_ms * 1e-3) / 1e9
                                       / HBM_PEAK_GBPS, 4),
            # The same bytes against the streaming probe with the decoder's
            # read/write mix (an attainable ceiling, not the peak).
            "frac_of_attainable_mix": round(dec_alg / (kernel_ms * 1e-3) / 1e9
                                            / bandwidth["decoder_mix_gbps"], 4),
        },
        "encode_roofline": {
            "kernel": "compress_kernel",
            "kernel_us": round(encode_kernel_ms * 1e3, 2),
            "algorithmic_bytes": enc_alg,
            "achieved": round(enc_alg / (encode_kernel_ms * 1e-3) / 1e9, 1),
            "frac": round(enc_alg / (encode_kernel_ms * 1e-3) / 1e9 / HBM_PEAK_GBPS, 4),
            "traffic": measured_traffic("compress_kernel<2,false>", nb),
        },
    }
    result["bandwidth"] = bandwidth
    result["config2"] = config2
    result["config3"] = config3
    result["update"] = update
    result["weight_update"] = weight_update
    if not args.skip_train:
        _log("timing config 5 (GPT-2-small training step)")
        del copy_out
        torch.cuda.empty_cache()
        result["config5"] = time_config5(torch, device)
    if not args.skip_cpu:
        _log("cpu baseline")
        result["cpu_baseline"] = cpu_baseline(host_inputs[0], dist, args.cpu_seconds)
    print(json.dumps(result), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
