"""Benchmark: effective quantized-payload GB/s of the MatVec hot path on one MI355X.

Headline workload: Ternary2 MatVec 4096x4096, block 128, batch 1 (FP32 weights ~N(0,1) from seed 1729,
quantized by Ternary2Matrix.Quantize; x ~ U(-1, 1)). One 4096x4096 matrix is 4.72 MB, far below the
256 MB Infinity Cache and below launch latency, so a step is one pass over G distinct resident copies
of it (G * 4.72 MB >= 1 GiB), issued as ONE grouped launch (satori_hip_group_execute): every step streams
>= 1 GiB of payload from HBM. GB/s = G * payload bytes / step time (the reference's method: payload
bytes including scales and padding, activations and outputs excluded). Inputs are resident in HBM
before the timed region; no host transfer is timed.

The same line carries, labelled:
  formats:   the same measurement for Q8_0 4096^2, Q4_0 11008x4096 and 4096x11008, Q4_K and Q6_K at the
             Qwen-1.5B shapes (K formats on the Q8_K integer path: quantize + product per step),
             and Ternary2 at the other block sizes;
  single:    one launch per matrix (rotating copies), which includes launch gaps;
  cache:     the grouped launch over G references to ONE copy (cache resident, not an HBM figure);
  decode_step: the 197 projections of one decode token of a Qwen-1.5B-shaped model (Q4_K/Q6_K on the Q8_K
             integer path, 1.03 GB per token), replayed as one graph; tokens/s and GB/s;
  decode_token: a whole token of that model on the device (operators, attention over a 511-token KV prefix,
             projections; the residual adds and RmsNorms folded into the projection launches),
             captured once and replayed, with the fused and unfused operator sequences beside it;
  prefill:   the same model's projections over 512 positions (ExecuteBatch in 256-position chunks);
             tokens/s and int8 TOP/s;
  loading:   upload rates of a GGUF tensor (device scale check), an STQ2 file and an STB1 bitplane file;
  host_call: the drop-in host-buffer call on one matrix (copies, scan, launch, synchronisation), per format;
  parity:    before anything of a workload is timed, the launches it times are checked against the oracle
             (every copy of a grouped case, every launch of the decode step, sampled prefill positions); a
             mismatch stops the benchmark with a non-zero exit before timing;
  roofline:  for the headline kernel, from HIP events on the launch stream;
  cpu_baseline: the restated reference AVX2 kernel (Ternary2Avx2Kernel) on one host core; each format's
             entry also carries its own restated reference AVX2 path timed on one core (cpu_gbs).

Usage: python bench.py [--steps K] [--warmup W] [--gpus 1] [--quick]
"""
from __future__ import annotations

import argparse
import ctypes
import json
import math
import os
import sys
import time

import numpy as np

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

import satori_amd as S  # noqa: E402

HBM_PEAK_GBS = 8000.0
ROTATION_BYTES = 1 << 30
CALIBRATION_BYTES = 1 << 30
BQ = S.BlockQuantization
METRIC = "effective quantized-payload GB/s (% of MI355X HBM peak) per format, 4096² batch 1"
PUBLISHED_AVX2_T2_4096_B128 = 1.31  # GB/s, Ternary2 AVX2 4096^2 B128, docs/benchmarks/avx2-2026-10-12 run 1
# The same run's scalar figure for that shape (ExecuteScalarCore): 114.150 ms, 4,718,592 B (run 1).
PUBLISHED_SCALAR_T2_4096_B128_MS = 114.150
# The same run's AVX2 figures for the whole size x block grid (docs/benchmarks/avx2-2026-10-12/README.md:5-17,
# run 1, EffectiveWeightGBPerSecond), GB/s by (size, block).
PUBLISHED_AVX2_T2 = {(1024, 64): 1.33, (1024, 128): 1.23, (1024, 256): 1.15,
                     (2048, 64): 1.29, (2048, 128): 1.32, (2048, 256): 1.22,
                     (4096, 64): 1.37, (4096, 128): 1.31, (4096, 256): 1.22}


class HipEvents:
    """hipEvent timing on a given stream, through the HIP runtime the library already loaded."""

    def __init__(self):
        S._ffi.lib()
        self.rt = ctypes.CDLL("libamdhip64.so.7")
        self.rt.hipEventCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
        self.rt.hipEventRecord.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
        self.rt.hipEventSynchronize.argtypes = [ctypes.c_void_p]
        self.rt.hipEventElapsedTime.argtypes = [ctypes.POINTER(ctypes.c_float), ctypes.c_void_p, ctypes.c_void_p]
        self.rt.hipEventDestroy.argtypes = [ctypes.c_void_p]

        self.created = []

    def event(self):
        e = ctypes.c_void_p()
        assert self.rt.hipEventCreate(ctypes.byref(e)) == 0
        self.created.append(e)
        return e

    def close(self):
        for e in self.created:
            self.rt.hipEventDestroy(e)
        self.created = []

    def record(self, event, stream):
        assert self.rt.hipEventRecord(event, ctypes.c_void_p(stream)) == 0

    def elapsed_ms(self, start, stop) -> float:
        assert self.rt.hipEventSynchronize(stop) == 0
        ms = ctypes.c_float()
        assert self.rt.hipEventElapsedTime(ctypes.byref(ms), start, stop) == 0
        return ms.value


def rng(seed: int) -> np.random.Generator:
    return np.random.Generator(np.random.PCG64(seed))


def make_ternary2(rows, columns, block, seed=1729):
    g = rng(seed)
    w = g.standard_normal((rows, columns), dtype=np.float32)
    x = g.uniform(-1, 1, columns).astype(np.float32)
    return S.Ternary2Matrix.quantize(w, rows, columns, block).data, x


def make_gguf(fmt, rows, columns, seed=20261014):
    g = rng(seed + rows + columns)
    w = (g.standard_normal((rows, columns), dtype=np.float32) * np.float32(0.02)).astype(np.float32)
    x = g.standard_normal(columns, dtype=np.float32)
    return S.quantize_weights(w, rows, columns, fmt), x


class Case:
    """G resident copies of one matrix plus device input/outputs, and the launches to time."""

    def __init__(self, ctx, name, create, payload_bytes, rows, columns, x, quantized, copies=None):
        self.ctx, self.name, self.payload_bytes, self.rows, self.columns = ctx, name, payload_bytes, rows, columns
        self.quantized = quantized
        self.expected = self.bound = None  # set by check_case
        self.copies = copies or max(1, math.ceil(ROTATION_BYTES / payload_bytes))
        first = create()
        self.mats = [first] + [first.clone() for _ in range(self.copies - 1)]
        self.x = x
        self.dx = ctx.alloc(x.nbytes)
        ctx.upload(self.dx, x)
        self.dy = [ctx.alloc(4 * rows) for _ in range(self.copies)]
        self.group = S.HipGroup(ctx, self.mats, [self.dx] * self.copies, self.dy, quantized)
        self.cache_group = S.HipGroup(ctx, [first] * self.copies, [self.dx] * self.copies, self.dy, quantized)

    def run_group(self):
        self.group.execute()

    def run_cache(self):
        self.cache_group.execute()

    def run_single(self):
        for m, y in zip(self.mats, self.dy):
            if self.quantized:
                m.execute_batch_device(self.dx, 1, y)
            else:
                m.execute_device(self.dx, y)

    def close(self):
        self.group.dispose()
        self.cache_group.dispose()
        for m in self.mats:
            m.dispose()
        for y in self.dy:
            self.ctx.free(y)
        self.ctx.free(self.dx)


def time_launches(ctx, events, fn, steps, warmup) -> float:
    """Milliseconds per call of fn() over `steps` timed calls on the context stream."""
    for _ in range(warmup):
        fn()
    ctx.synchronize()
    start, stop = events.event(), events.event()
    events.record(start, ctx.stream)
    for _ in range(steps):
        fn()
    events.record(stop, ctx.stream)
    ms = events.elapsed_ms(start, stop)
    ctx.synchronize()
    return ms / steps


def warm_up(ctx, fn, seconds: float) -> None:
    """Run fn() back to back for `seconds` of wall time, so the timed region starts at steady-state clocks
    (the first ~0.1 s of work on an idle GPU runs at lower clocks)."""
    t0 = time.perf_counter()
    while time.perf_counter() - t0 < seconds:
        for _ in range(20):
            fn()
        ctx.synchronize()


def progress(message: str) -> None:
    print(f"[bench] {message}", file=sys.stderr, flush=True)


class ParityError(RuntimeError):
    """A timed launch's outputs disagree with the oracle: the benchmark stops before timing."""


def fp32_bound(data, rows, columns, fmt, x, block=None) -> np.ndarray:
    """1e-5 * sum_i |w_i x_i| per row (FP64) on the decoded weights (the oracle decodes them)."""
    from oracle import oracle as O

    ax = np.abs(x.astype(np.float64))
    if fmt is None:
        return 1e-5 * (np.abs(O.t2_dequantize(data, rows, columns, block).astype(np.float64)) @ ax)
    row_bytes = data.size // rows
    return 1e-5 * np.array([np.abs(O.q_decode_row(data[r * row_bytes:(r + 1) * row_bytes], columns, int(fmt))) @ ax
                            for r in range(rows)])


def check_case(ctx, case: Case, data, rows, columns, fmt, x, quantized) -> dict:
    """Parity of the launch that is timed, before it is timed (the reference benchmark validates before it
    measures, benchmarks/Satori.Benchmarks/Program.cs:38-61): one grouped launch, then every copy's output
    against the oracle, which only checks: Ternary2, Q8_0 and Q4_0 within 1e-5 * sum|w x| per row of the scalar
    restatement, K formats on the Q8_K path identical to the ExecuteQuantizedTiled composition."""
    from oracle import oracle as O

    if fmt is None:
        expected, bound = O.t2_matvec_scalar(data, rows, columns, quantized, x), fp32_bound(data, rows, columns,
                                                                                            None, x, quantized)
    elif quantized:
        expected, bound = O.qk_matvec_quantized_avx2(data, rows, columns, int(fmt), O.q8k_quantize_row(x)), None
    else:
        expected, bound = O.q_matvec_scalar(data, rows, columns, int(fmt), x), fp32_bound(data, rows, columns, fmt, x)
    case.expected, case.bound = expected, bound
    case.run_group()
    worst = check_outputs(ctx, case, "grouped launch")
    return {"parity_checked": True, "parity_copies": case.copies,
            "parity": "bit-exact" if bound is None else f"max |err| / (1e-5 sum|w x|) = {worst:.3g}"}


def check_outputs(ctx, case: Case, what: str) -> float:
    """Every copy's output against the expected values check_case stored (raises ParityError); returns the
    worst error as a fraction of the bound (0 for bit-exact comparisons)."""
    ctx.synchronize()
    worst = 0.0
    for i, dy in enumerate(case.dy):
        y = ctx.download(np.zeros(case.rows, np.float32), dy)
        ctx.upload(dy, np.full(case.rows, np.nan, np.float32))  # the next launch checked must write it again
        if case.bound is None:
            if not np.array_equal(y.view(np.uint32), case.expected.view(np.uint32)):
                raise ParityError(f"{case.name} ({what}): copy {i} differs from the oracle")
        else:
            ratio = np.abs(y.astype(np.float64) - case.expected) / np.maximum(case.bound, 1e-300)
            if not np.all(np.isfinite(y)) or not np.all(ratio <= 1.0):
                raise ParityError(f"{case.name} ({what}): copy {i} outside 1e-5 * sum|w x| (worst ratio {ratio.max()})")
            worst = max(worst, float(ratio.max()))
    return worst


def measure(ctx, events, case: Case, steps, warmup, single=True) -> dict:
    progress(f"{case.name}: {case.copies} copies x {case.payload_bytes} B")
    warm_up(ctx, case.run_group, 0.25)
    group_ms = time_launches(ctx, events, case.run_group, steps, warmup)
    step_bytes = case.copies * case.payload_bytes
    out = {
        "shape": [case.rows, case.columns],
        "payload_bytes": case.payload_bytes,
        "copies": case.copies,
        "gbs": step_bytes / (group_ms * 1e-3) / 1e9,
        "launch_us": group_ms * 1e3,
        "rows_per_s": case.copies * case.rows / (group_ms * 1e-3),
    }
    out["pct_hbm"] = 100.0 * out["gbs"] / HBM_PEAK_GBS
    cache_ms = time_launches(ctx, events, case.run_cache, max(2, steps // 2), 1)
    out["cache_resident_gbs"] = step_bytes / (cache_ms * 1e-3) / 1e9
    if single:
        # One launch per matrix, issued back to back from Python (the ctypes call and the library's host
        # work included), then the same launches captured once and replayed (the device time per launch).
        if case.expected is not None:  # single matrices may take another plan than the group
            case.run_single()
            check_outputs(ctx, case, "single launches")
            out["single_launch_parity_checked"] = True
        single_ms = time_launches(ctx, events, case.run_single, max(2, steps // 4), 1)
        out["single_launch_us"] = single_ms * 1e3 / case.copies
        out["single_launch_gbs"] = step_bytes / (single_ms * 1e-3) / 1e9
        ctx.capture_begin()
        case.run_single()
        replay = ctx.capture_end()
        try:
            graph_ms = time_launches(ctx, events, replay.execute, max(2, steps // 4), 1)
        finally:
            replay.dispose()
        out["single_launch_graph_us"] = graph_ms * 1e3 / case.copies
    return out


def host_call_latency(case: Case, calls: int = 200) -> dict:
    """The drop-in host call on one resident matrix, host buffers in and out (satori_hip_matvec: input copy,
    finiteness scan where the surface has one, launch, output copy, stream synchronisation): median and
    minimum wall time per call. K formats also through ExecuteBatch at one position (the Q8_K integer product,
    the decode path)."""
    m, x = case.mats[0], case.x
    y = np.zeros(case.rows, np.float32)

    def timed(fn):
        fn()
        samples = []
        for _ in range(calls):
            t0 = time.perf_counter()
            fn()
            samples.append(time.perf_counter() - t0)
        samples.sort()
        return samples[len(samples) // 2] * 1e6, samples[0] * 1e6

    out = {}
    out["host_call_us_median"], out["host_call_us_min"] = timed(lambda: m.execute(x, y))
    if case.quantized:
        out["host_call_batch1_us_median"], out["host_call_batch1_us_min"] = timed(lambda: m.execute_batch(x, 1, y))
    return out


class DecodeModel:
    """A Qwen-1.5B-shaped model's projections: 28 layers of q 1536x1536, k and v 256x1536, o 1536x1536, gate and
    up 8960x1536 in Q4_K, down 1536x8960 in Q6_K, then the output projection 151936x1536 in Q6_K (197
    projections, 1,027,772,928 payload bytes). Random-init weights, every matrix a distinct resident copy."""

    D, KV, FFN, VOCAB, LAYERS = 1536, 256, 8960, 151936, 28

    def __init__(self, ctx):
        self.ctx = ctx
        d, kv, ffn, vocab = self.D, self.KV, self.FFN, self.VOCAB
        self.roles = {"q": (d, d, BQ.Q4_K), "k": (kv, d, BQ.Q4_K), "v": (kv, d, BQ.Q4_K), "o": (d, d, BQ.Q4_K),
                      "gate": (ffn, d, BQ.Q4_K), "up": (ffn, d, BQ.Q4_K), "down": (d, ffn, BQ.Q6_K)}
        self.shapes = dict(self.roles, output=(vocab, d, BQ.Q6_K))
        first = {}
        self.host = {}  # the payloads, for the parity check
        for name, (r, c, fmt) in self.roles.items():
            data, _ = make_gguf(fmt, r, c)
            self.host[name] = data
            first[name] = ctx.create(data, S.QuantizedMatrixShape(r, c, fmt))
        # Output projection: rows of a 4096-row random Q6_K matrix repeated to 151,936 rows (rows are
        # independent byte ranges, so the payload is a valid matrix of that shape).
        base, _ = make_gguf(BQ.Q6_K, 4096, d)
        row_bytes = base.size // 4096
        tiled = np.tile(base.reshape(4096, row_bytes), (-(-vocab // 4096), 1))[:vocab].reshape(-1)
        self.output = ctx.create(tiled, S.QuantizedMatrixShape(vocab, d, BQ.Q6_K))
        self.host["output"] = tiled
        self.layers = [{name: (first[name] if layer == 0 else first[name].clone()) for name in self.roles}
                       for layer in range(self.LAYERS)]
        payload = sum(r * (c // 256) * (144 if fmt == BQ.Q4_K else 210) for r, c, fmt in self.roles.values())
        self.token_bytes = self.LAYERS * payload + vocab * (d // 256) * 210
        self.buffers = []

    def device(self, values):
        p = self.ctx.alloc(values.nbytes)
        self.ctx.upload(p, values)
        self.buffers.append(p)
        return p

    def close(self):
        for layer in self.layers:
            for m in layer.values():
                m.dispose()
        self.output.dispose()
        for p in self.buffers:
            self.ctx.free(p)


# The input each projection of a layer reads (q/k/v the normed residual, o the attention output, gate/up the
# second normed residual, down the SwiGLU output), and the output projection's.
FEEDS = {"q": "h", "k": "h", "v": "h", "o": "attn", "gate": "h2", "up": "h2", "down": "act", "output": "h"}


def decode_inputs(model: "DecodeModel") -> dict:
    """The decode step's fixed FP32 projection inputs (seeded)."""
    g = rng(2026)
    return {"h": g.standard_normal(model.D).astype(np.float32), "attn": g.standard_normal(model.D).astype(np.float32),
            "h2": g.standard_normal(model.D).astype(np.float32), "act": g.standard_normal(model.FFN).astype(np.float32)}


def prefill_inputs(model: "DecodeModel", positions: int) -> dict:
    """The prefill's fixed FP32 projection inputs, [positions][columns] flattened (seeded)."""
    g = rng(2027)
    return {"h": g.standard_normal(positions * model.D).astype(np.float32),
            "attn": g.standard_normal(positions * model.D).astype(np.float32),
            "h2": g.standard_normal(positions * model.D).astype(np.float32),
            "act": g.standard_normal(positions * model.FFN).astype(np.float32)}


def decode_step(ctx, events, model: DecodeModel, steps: int, warmup: int, eager_only: bool = False) -> dict:
    """The projection sequence of one decode token (197 projections, batch 1) on the Q8_K integer path, launched
    as the whole token launches them. Projections that share an input form one group (q/k/v, gate/up); the
    113 groups of a token are captured once as a graph (satori_hip_step) and replayed. Attention and the norms
    are not part of the path: their outputs are fixed random vectors. q/k/v, o and gate/up quantize their FP32
    input inside their launch; the gate/up launch also writes SwiGLU of its outputs, which down reads and
    quantizes in its own launch, so every projection's Q8_K input is produced inside the timed step (the
    reference's ExecuteBatch quantizes each input per call, QuantizedMatVec.cs:144-149). Also timed: the same
    groups launched eagerly."""
    d, ffn, vocab = model.D, model.FFN, model.VOCAB
    host_in = decode_inputs(model)
    h, attn, h2, act = (model.device(host_in[k]) for k in ("h", "attn", "h2", "act"))
    out = {name: model.device(np.zeros(r, np.float32)) for name, (r, _, _) in model.roles.items()}
    logits = model.device(np.zeros(vocab, np.float32))
    out["output"] = logits
    groups, members = [], []
    for m in model.layers:
        groups.append(S.HipGroup(ctx, [m["q"], m["k"], m["v"]], [h] * 3, [out["q"], out["k"], out["v"]], True))
        groups.append(S.HipGroup(ctx, [m["o"]], [attn], [out["o"]], True))
        groups.append(S.HipGroup(ctx, [m["gate"], m["up"]], [h2] * 2, [out["gate"], out["up"]], True))
        groups.append(S.HipGroup(ctx, [m["down"]], [act], [out["down"]], True))
        members += [("q", "k", "v"), ("o",), ("gate", "up"), ("down",)]
    groups.append(S.HipGroup(ctx, [model.output], [h], [logits], True))
    members.append(("output",))
    for grp, names in zip(groups, members):
        if names == ("gate", "up"):
            grp.set_output_swiglu(act)  # SwiGLU of the gate/up outputs, in the same launch; down quantizes it
    # Parity before timing: every launch of the step, one at a time, against the oracle (not timed).
    from oracle import oracle as O
    expected = {}
    for name, (r, c, fmt) in model.shapes.items():
        if name == "down":
            continue
        expected[name] = O.qk_matvec_quantized_avx2(model.host[name], r, c, int(fmt),
                                                    O.q8k_quantize_row(host_in[FEEDS[name]]))
    activated = O.swiglu(expected["gate"], expected["up"])  # down's input: SwiGLU of the gate/up outputs
    expected["down"] = O.qk_matvec_quantized_avx2(model.host["down"], d, ffn, int(BQ.Q6_K), O.q8k_quantize_row(activated))
    for grp, names in zip(groups, members):
        for name in names:
            ctx.upload(out[name], np.full(model.shapes[name][0], np.nan, np.float32))
        grp.execute()
        for name in names:
            y = ctx.download(np.zeros(model.shapes[name][0], np.float32), out[name])
            if not np.array_equal(y.view(np.uint32), expected[name].view(np.uint32)):
                raise ParityError(f"decode step: {name} differs from the oracle")

    def eager():
        for grp in groups:
            grp.execute()

    if eager_only:  # for kernel statistics: the same launches without the graph
        warm_up(ctx, eager, 0.5)
        graph_ms = eager_ms = time_launches(ctx, events, eager, steps, warmup)
    else:
        step = S.HipStep(ctx, groups)
        warm_up(ctx, step.execute, 0.5)
        graph_ms = time_launches(ctx, events, step.execute, steps, warmup)
        eager_ms = time_launches(ctx, events, eager, max(5, steps // 4), 2)
        step.dispose()
    for grp in groups:
        grp.dispose()
    return {
        "model": "Qwen-1.5B-shaped decode step, random-init Q4_K/Q6_K weights, batch 1",
        "parity_checked": True,
        "parity": f"each of the {len(groups)} launches of one step bit-exact against the oracle before timing",
        "projections_per_token": 28 * 7 + 1,
        "kernel_launches_per_token": len(groups),
        "bytes_per_token": model.token_bytes,
        "us_per_token": graph_ms * 1e3,
        "tokens_per_s": 1e3 / graph_ms,
        "gbs": model.token_bytes / (graph_ms * 1e-3) / 1e9,
        "pct_hbm": 100.0 * model.token_bytes / (graph_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
        "eager_us_per_token": eager_ms * 1e3,
    }


def decode_token(ctx, events, model: DecodeModel, steps: int, warmup: int, position: int = 511) -> dict:
    """A whole decode token on the device (satori_amd.decode.DeviceDecoder): embedding-row decode, per layer
    RmsNorm, q/k/v, bias adds, RoPE, grouped attention over a `position`-token key/value prefix (random),
    o, residual, RmsNorm, gate/up, SwiGLU, down, residual; then the final norm and the output projection
    (tied to the embedding, as Qwen2.5-1.5B). Captured once as one step and replayed; also timed eagerly,
    and replayed once more at the end of a 4096-token context."""
    from satori_amd.decode import DecoderConfig, DeviceDecoder
    g = rng(2029)
    cfg = DecoderConfig(hidden=model.D, heads=12, kv_heads=2, head_dim=128, ffn=model.FFN, epsilon=1e-6,
                        rope_base=1e6, max_tokens=position + 1)
    vectors = []
    for _ in model.layers:
        vectors.append({
            "attn_norm": model.device(g.uniform(0.5, 1.5, model.D).astype(np.float32)),
            "ffn_norm": model.device(g.uniform(0.5, 1.5, model.D).astype(np.float32)),
            "q_bias": model.device((g.standard_normal(model.D) * 0.1).astype(np.float32)),
            "k_bias": model.device((g.standard_normal(model.KV) * 0.1).astype(np.float32)),
            "v_bias": model.device((g.standard_normal(model.KV) * 0.1).astype(np.float32)),
        })
    out_norm = model.device(g.uniform(0.5, 1.5, model.D).astype(np.float32))
    dec = DeviceDecoder(ctx, cfg, model.layers, vectors, out_norm, model.output, model.output)
    for layer in range(len(model.layers)):
        prefix = (g.standard_normal((cfg.max_tokens, model.KV)) * 0.5).astype(np.float32)
        ctx.upload(dec.keys[layer], prefix)
        ctx.upload(dec.values[layer], prefix[::-1].copy())
    # Folded (add + RmsNorm inside the projection launches), the default; fused and unfused for comparison.
    step = dec.capture(151, position, folded=True)
    warm_up(ctx, step.execute, 0.5)
    graph_ms = time_launches(ctx, events, step.execute, steps, warmup)
    eager_ms = time_launches(ctx, events, lambda: dec.enqueue(151, position, folded=True), max(5, steps // 4), 2)
    folded_logits = dec.read_logits()
    timed = {}
    for name, fused in (("fused", True), ("unfused", False)):
        other = dec.capture(151, position, fused=fused)
        timed[name] = time_launches(ctx, events, other.execute, max(5, steps // 2), 2)
        other.dispose()
    same = bool(np.array_equal(dec.read_logits().view(np.uint32), folded_logits.view(np.uint32)))
    finite = bool(np.all(np.isfinite(folded_logits)))
    step.dispose()
    dec.dispose()
    # The same token at the end of a 4096-token context (FP32 key/value cache of 4096 positions).
    long_position = 4095
    long_cfg = DecoderConfig(hidden=model.D, heads=12, kv_heads=2, head_dim=128, ffn=model.FFN, epsilon=1e-6,
                             rope_base=1e6, max_tokens=long_position + 1)
    long_dec = DeviceDecoder(ctx, long_cfg, model.layers, vectors, out_norm, model.output, model.output)
    for layer in range(len(model.layers)):
        prefix = (g.standard_normal((long_cfg.max_tokens, model.KV)) * 0.5).astype(np.float32)
        ctx.upload(long_dec.keys[layer], prefix)
        ctx.upload(long_dec.values[layer], prefix[::-1].copy())
    long_step = long_dec.capture(151, long_position, folded=True)
    warm_up(ctx, long_step.execute, 0.3)
    long_ms = time_launches(ctx, events, long_step.execute, steps, warmup)
    long_finite = bool(np.all(np.isfinite(long_dec.read_logits())))
    long_launches = long_dec.launches_per_token(folded=True, position=long_position)
    long_step.dispose()
    long_dec.dispose()
    return {
        "model": "Qwen-1.5B-shaped whole decode token on the device (random-init weights and KV prefix)",
        "position": position,
        "kernel_launches_per_token": dec.launches_per_token(folded=True, position=position),
        "us_per_token": graph_ms * 1e3,
        "tokens_per_s": 1e3 / graph_ms,
        "eager_us_per_token": eager_ms * 1e3,
        "fused_us_per_token": timed["fused"] * 1e3,
        "fused_launches_per_token": dec.launches_per_token(position=position),
        "unfused_us_per_token": timed["unfused"] * 1e3,
        "unfused_launches_per_token": dec.launches_per_token(fused=False, position=position),
        "same_logits_all_modes": same,
        "finite_logits": finite,
        "context_4096": {"position": long_position, "us_per_token": long_ms * 1e3, "tokens_per_s": 1e3 / long_ms,
                         "kernel_launches_per_token": long_launches, "finite_logits": long_finite},
    }


def token_eager(ctx, events, model: DecodeModel, steps: int, warmup: int, positions=(511, 4095)) -> dict:
    """The whole decode token (folded operator sequence, as decode_token captures it) launched eagerly at the
    given positions, for kernel statistics under a profiler (no graph)."""
    from satori_amd.decode import DecoderConfig, DeviceDecoder
    g = rng(2029)
    out = {}
    vectors = [{"attn_norm": model.device(g.uniform(0.5, 1.5, model.D).astype(np.float32)),
                "ffn_norm": model.device(g.uniform(0.5, 1.5, model.D).astype(np.float32)),
                "q_bias": model.device((g.standard_normal(model.D) * 0.1).astype(np.float32)),
                "k_bias": model.device((g.standard_normal(model.KV) * 0.1).astype(np.float32)),
                "v_bias": model.device((g.standard_normal(model.KV) * 0.1).astype(np.float32))}
               for _ in model.layers]
    out_norm = model.device(g.uniform(0.5, 1.5, model.D).astype(np.float32))
    for position in positions:
        cfg = DecoderConfig(hidden=model.D, heads=12, kv_heads=2, head_dim=128, ffn=model.FFN, epsilon=1e-6,
                            rope_base=1e6, max_tokens=position + 1)
        dec = DeviceDecoder(ctx, cfg, model.layers, vectors, out_norm, model.output, model.output)
        for layer in range(len(model.layers)):
            prefix = (g.standard_normal((cfg.max_tokens, model.KV)) * 0.5).astype(np.float32)
            ctx.upload(dec.keys[layer], prefix)
            ctx.upload(dec.values[layer], prefix[::-1].copy())
        ms = time_launches(ctx, events, lambda: dec.enqueue(151, position, folded=True), steps, warmup)
        out[f"position_{position}"] = {"eager_us_per_token": ms * 1e3,
                                       "kernel_launches_per_token": dec.launches_per_token(folded=True,
                                                                                           position=position)}
        dec.dispose()
    return out


def batch_fp32(ctx, events, steps: int = 20, warmup: int = 3, positions: int = 256) -> dict:
    """ExecuteBatch of the FP32-activation formats (QuantizedMatVec.ExecuteBatchFloat / ExecuteBatchRows) at
    256 positions on the Q8_0 4096 x 4096 and Q4_0 11008 x 4096 / 4096 x 11008 shapes, through the device
    entry point: the activations are split into exact bf16 parts once per call and the matrix-core product
    reads each matrix once per 64 positions. Parity first (sampled positions within 1e-5 * sum|w x| of the oracle's scalar
    product), then timed. `per_position_gbs` is the payload bytes times positions over the time, the rate a
    per-position MatVec would have to stream at to match."""
    from oracle import oracle as O

    out = {}
    for label, fmt, rows, columns in (("q8_0-4096x4096", BQ.Q8_0, 4096, 4096),
                                      ("q4_0-11008x4096", BQ.Q4_0, 11008, 4096),
                                      ("q4_0-4096x11008", BQ.Q4_0, 4096, 11008)):
        data, _ = make_gguf(fmt, rows, columns)
        g = rng(99 + rows)
        x = g.standard_normal((positions, columns), dtype=np.float32)
        m = ctx.create(data, S.QuantizedMatrixShape(rows, columns, fmt))
        dx, dy = ctx.alloc(x.nbytes), ctx.alloc(4 * rows * positions)
        ctx.upload(dx, x)
        m.execute_batch_device(dx, positions, dy)
        ctx.synchronize()
        y = ctx.download(np.zeros(positions * rows, np.float32), dy).reshape(positions, rows)
        wq = np.abs(O.decode_matrix(data, rows, columns, int(fmt)).astype(np.float64))
        for p in (0, 1, 31, 32, positions // 2, positions - 1):
            want = O.q_matvec_scalar(data, rows, columns, int(fmt), x[p])
            bound = 1e-5 * (wq @ np.abs(x[p].astype(np.float64)))
            if not np.all(np.abs(y[p].astype(np.float64) - want) <= bound):
                raise ParityError(f"batch {label}: position {p} outside 1e-5 * sum|w x| of the oracle")
        ms = time_launches(ctx, events, lambda: m.execute_batch_device(dx, positions, dy), steps, warmup)
        out[label] = {"positions": positions, "parity_checked": True, "us_per_call": ms * 1e3,
                      "gflops": 2.0 * rows * columns * positions / (ms * 1e-3) / 1e9,
                      "per_position_gbs": data.size * positions / (ms * 1e-3) / 1e9}
        ctx.free(dx)
        ctx.free(dy)
        m.dispose()
    return out


def prefill(ctx, events, model: DecodeModel, steps: int, warmup: int, positions: int = 512) -> dict:
    """The projections of a 512-token prefill: every layer projection over all positions in chunks of 256
    positions (the reference's chunk, and the ABI's limit for K formats), q/k/v and gate/up each as one
    grouped product over their shared input (DenseForward.LayerBatch), o and down through ExecuteBatch,
    and the output projection for the last position only (DenseSession.cs:156-159). The FLOP-based rate
    counts 2 int8 operations per weight per position."""
    d, ffn = model.D, model.FFN
    host_in = prefill_inputs(model, positions)
    h, attn, h2, act = (model.device(host_in[k]) for k in ("h", "attn", "h2", "act"))
    out = {name: model.device(np.zeros(positions * r, np.float32)) for name, (r, _, _) in model.roles.items()}
    logits = model.device(np.zeros(model.VOCAB, np.float32))
    inputs = {"q": h, "k": h, "v": h, "o": attn, "gate": h2, "up": h2, "down": act}
    chunk = 256
    chunks = [(p0, min(chunk, positions - p0)) for p0 in range(0, positions, chunk)]

    def group(m, names, p0):
        # Projections of one chunk that read one input (q/k/v, gate/up): one grouped many-position product.
        return S.HipGroup(ctx, [m[n] for n in names],
                          [inputs[n] + 4 * p0 * model.roles[n][1] for n in names],
                          [out[n] + 4 * p0 * model.roles[n][0] for n in names], True)

    plan = []  # per layer and chunk: the q/k/v group, o, the gate/up group, down
    for m in model.layers:
        for p0, n in chunks:
            plan.append((group(m, ("q", "k", "v"), p0), group(m, ("gate", "up"), p0), m, p0, n))

    def single(m, name, p0, n):
        r, c, _ = model.roles[name]
        m[name].execute_batch_device(inputs[name] + 4 * p0 * c, n, out[name] + 4 * p0 * r)

    def run():
        for qkv, gateup, m, p0, n in plan:
            qkv.execute_batch(n)
            single(m, "o", p0, n)
            gateup.execute_batch(n)
            single(m, "down", p0, n)
        model.output.execute_batch_device(h + 4 * (positions - 1) * d, 1, logits)

    # The first run allocates the workspaces and builds each Q6_K matrix's weight planes (once per matrix, kept
    # until it is destroyed): setup, reported apart from the timed runs.
    t0 = time.perf_counter()
    run()
    ctx.synchronize()
    first_ms = (time.perf_counter() - t0) * 1e3
    # Parity before timing (the oracle is not timed): the last layer's outputs at sampled positions of both chunks
    # (tile edges 0/31/32, chunk edges 255/256, the last position) and the output projection, bit-exact.
    from oracle import oracle as O
    sampled = [p for p in (0, 1, 31, 32, 100, 255, 256, 257, 300, 400, 511) if p < positions]
    ctx.synchronize()
    for name, (r, c, fmt) in model.roles.items():
        y = ctx.download(np.zeros(positions * r, np.float32), out[name]).reshape(positions, r)
        for p in sampled:
            x = host_in[FEEDS[name]][p * c:(p + 1) * c]
            want = O.qk_matvec_quantized_avx2(model.host[name], r, c, int(fmt), O.q8k_quantize_row(x))
            if not np.array_equal(y[p].view(np.uint32), want.view(np.uint32)):
                raise ParityError(f"prefill: {name} at position {p} differs from the oracle")
    want = O.qk_matvec_quantized_avx2(model.host["output"], model.VOCAB, d, int(BQ.Q6_K),
                                      O.q8k_quantize_row(host_in["h"][(positions - 1) * d:positions * d]))
    if not np.array_equal(ctx.download(np.zeros(model.VOCAB, np.float32), logits).view(np.uint32), want.view(np.uint32)):
        raise ParityError("prefill: output projection differs from the oracle")
    ms = time_launches(ctx, events, run, steps, warmup)
    for qkv, gateup, *_ in plan:
        qkv.dispose()
        gateup.dispose()
    weights = sum(r * c for r, c, _ in model.roles.values()) * model.LAYERS
    ops = 2.0 * weights * positions + 2.0 * model.VOCAB * d
    plane_bytes = model.LAYERS * sum(-(-r // 32) * (c // 256) * 16512 for r, c, f in model.roles.values() if f == BQ.Q6_K)
    return {
        "positions": positions,
        "first_run_ms": first_ms,
        "weight_plane_bytes": plane_bytes,
        "parity_checked": True,
        "parity": f"last layer at positions {sampled} and the output projection bit-exact against the oracle",
        "ms": ms,
        "tokens_per_s": positions / (ms * 1e-3),
        "int8_tops": ops / (ms * 1e-3) / 1e12,
        "pct_int8_peak": 100.0 * ops / (ms * 1e-3) / 5.0e15,
    }


def write_gguf(path: str, tensors) -> None:
    """A GGUF v3 file (the subset the reader accepts, docs/gguf-subset-v1.md) holding `tensors`:
    (name, rows, columns, ggml type, payload bytes), 32-byte aligned."""
    import struct

    def string(v: str) -> bytes:
        raw = v.encode()
        return struct.pack("<Q", len(raw)) + raw

    out = bytearray(b"GGUF" + struct.pack("<IQQ", 3, len(tensors), 3))
    out += string("general.architecture") + struct.pack("<I", 8) + string("llama")
    out += string("general.alignment") + struct.pack("<II", 4, 32)
    out += string("general.quantization_version") + struct.pack("<II", 4, 2)
    offset, blobs = 0, []
    for name, rows, columns, type_, payload in tensors:
        out += string(name) + struct.pack("<I", 2) + struct.pack("<QQ", columns, rows) + struct.pack("<IQ", type_, offset)
        blobs.append((offset, payload))
        offset += (payload.size + 31) // 32 * 32
    while len(out) % 32:
        out += b"\0"
    data = bytearray(offset)
    for off, payload in blobs:
        data[off:off + payload.size] = payload.tobytes()
    with open(path, "wb") as f:
        f.write(bytes(out) + bytes(data))


def loading(ctx, seconds: float = 0.5) -> dict:
    """Resident upload rates of the on-disk formats (payload bytes / time, files in the page cache):
    a GGUF tensor bound and uploaded straight from the mapping with its block scales checked on the device
    (satori_hip_gguf_matrix_create), an STQ2 file opened, validated and uploaded (MappedTernary2Matrix), and
    the same matrix as an STB1 bitplane file (satori_hip_bitplane_open, converted on upload); beside them the
    upload of the same payloads from host memory."""
    import shutil
    import tempfile

    d = tempfile.mkdtemp(prefix="satori_bench_")
    out = {}

    def rate(fn, nbytes):
        fn()
        n, t0 = 0, time.perf_counter()
        while time.perf_counter() - t0 < seconds or n < 3:
            fn()
            n += 1
        return nbytes * n / (time.perf_counter() - t0) / 1e9

    try:
        q4, _ = make_gguf(BQ.Q4_K, 8960, 1536)
        q6, _ = make_gguf(BQ.Q6_K, 1536, 8960)
        path = os.path.join(d, "model.gguf")
        write_gguf(path, [("blk.0.ffn_gate.weight", 8960, 1536, 12, q4), ("blk.0.ffn_down.weight", 1536, 8960, 14, q6)])
        with S.GgufFile(path) as f:
            for name, data, fmt, rows, cols in (("blk.0.ffn_gate.weight", q4, BQ.Q4_K, 8960, 1536),
                                                ("blk.0.ffn_down.weight", q6, BQ.Q6_K, 1536, 8960)):
                gm = S.GgufQuantizedMatrix(f, name)
                label = f"gguf_{fmt.name.lower()}_{rows}x{cols}"
                out[label + "_gbs"] = rate(lambda: gm.create_execution(ctx).dispose(), data.size)
                out[label + "_host_gbs"] = rate(lambda: ctx.create(data, S.QuantizedMatrixShape(rows, cols, fmt)).dispose(),
                                                data.size)
        payload, _ = make_ternary2(4096, 4096, 128)
        t2 = S.Ternary2Matrix.from_packed(4096, 4096, 128, payload)
        stq2 = os.path.join(d, "matrix.stq2")
        t2.save(stq2)
        out["stq2_4096_b128_gbs"] = rate(lambda: S.MappedTernary2Matrix(stq2, ctx).dispose(), payload.size)
        out["ternary2_4096_b128_host_gbs"] = rate(lambda: ctx.create_ternary2(4096, 4096, 128, payload).dispose(),
                                                  payload.size)
        bp = S.TernaryBitplaneMatrix.from_ternary2(t2)
        stb1 = os.path.join(d, "matrix.stb1")
        bp.save(stb1)
        out["stb1_bitplane_4096_b128_gbs"] = rate(lambda: ctx.open_bitplane(stb1).dispose(), payload.size)
    finally:
        shutil.rmtree(d, ignore_errors=True)
    return out


def profiled_traffic(name: str):
    """HBM bytes per launch of the headline kernel, from the committed rocprofv3 FETCH_SIZE / WRITE_SIZE
    summary (calibrated against a copy of known size); None when the summary is absent."""
    path = os.path.join(ROOT, "profiles", name)
    try:
        with open(path) as f:
            for line in f:
                if line.startswith("traffic_bytes_per_launch:"):
                    return int(line.split(":", 1)[1]), "profiles/" + name
    except OSError:
        pass
    return None, None


def pin_one_core():
    """Pins this process to its first allowed core (the CPU baselines run on one thread, as the reference's
    own measurements do); returns the core, or None where affinity cannot be set."""
    try:
        core = sorted(os.sched_getaffinity(0))[0]
        os.sched_setaffinity(0, {core})
        return core
    except (AttributeError, OSError):
        return None


def cpu_format(data, rows, columns, fmt, x, quantized, seconds) -> dict:
    """Restated reference AVX2 path of one format (oracle) on one host core, warm payload, bounded sample:
    Ternary2Avx2Kernel for Ternary2, QuantizedAvx2Kernel for Q8_0 / Q4_0, and for the K formats the decode
    path (Q8KCodec.QuantizeRow of x, then QuantizedKAvx2Kernel.ExecuteQuantizedTiled at one position); and the
    scalar reference of the format (`cpu_scalar_*`)."""
    from oracle import oracle as O

    y = np.zeros(rows, np.float32)
    if fmt is None:  # Ternary2, block size in `quantized`
        run = lambda: O.t2_matvec_avx2(data, rows, columns, quantized, x, y)
    elif quantized:
        run = lambda: O.qk_matvec_quantized_avx2(data, rows, columns, int(fmt), O.q8k_quantize_row(x), y)
    else:
        run = lambda: O.q_matvec_avx2(data, rows, columns, int(fmt), x, y)
    run()  # warm
    samples, start = [], time.perf_counter()
    while time.perf_counter() - start < seconds or len(samples) < 3:
        t0 = time.perf_counter()
        run()
        samples.append(time.perf_counter() - t0)
    best = min(samples)
    # The scalar reference beside it (Ternary2MatVec.ExecuteScalarCore / QuantizedMatVec.ExecuteScalar,
    # restated in oracle/satori_oracle.c), a short bounded sample: at least three runs, min reported.
    if fmt is None:
        scalar_run = lambda: O.t2_matvec_scalar(data, rows, columns, quantized, x)
    else:
        scalar_run = lambda: O.q_matvec_scalar(data, rows, columns, int(fmt), x)
    scalar_samples, s0 = [], time.perf_counter()
    while time.perf_counter() - s0 < 0.5 or len(scalar_samples) < 3:
        t0 = time.perf_counter()
        scalar_run()
        scalar_samples.append(time.perf_counter() - t0)
    return {"cpu_gbs": data.size / best / 1e9, "cpu_ms_min": best * 1e3,
            "cpu_ms_median": sorted(samples)[len(samples) // 2] * 1e3, "cpu_runs": len(samples),
            "cpu_scalar_gbs": data.size / min(scalar_samples) / 1e9, "cpu_scalar_ms_min": min(scalar_samples) * 1e3,
            "cpu_scalar_runs": len(scalar_samples)}


def cpu_decode_step(host, shapes, host_in, seconds) -> dict:
    """The decode step's 197 projections on one host core through the restated reference path (oracle):
    per projection Q8KCodec.QuantizeRow of its FP32 input, then QuantizedKAvx2Kernel.ExecuteQuantizedTiled at
    one position -- what QuantizedMatVec.ExecuteBatch runs for each projection of DenseForward.Step
    (DenseForward.cs:119; QuantizedMatVec.cs:136-219), quantization included. Each of the 28 layers has its
    own copy of the payloads, as on the GPU (no layer finds another's weights in the caches)."""
    from oracle import oracle as O

    layers = [{name: host[name].copy() for name in shapes if name != "output"} for _ in range(28)]
    ys = {name: np.zeros(r, np.float32) for name, (r, _, _) in shapes.items()}

    def token():
        for layer in layers:
            for name, data in layer.items():
                r, c, fmt = shapes[name]
                O.qk_matvec_quantized_avx2(data, r, c, int(fmt), O.q8k_quantize_row(host_in[FEEDS[name]]), ys[name])
        r, c, fmt = shapes["output"]
        O.qk_matvec_quantized_avx2(host["output"], r, c, int(fmt), O.q8k_quantize_row(host_in["h"]), ys["output"])

    token()  # warm
    samples, start = [], time.perf_counter()
    while time.perf_counter() - start < seconds or len(samples) < 3:
        t0 = time.perf_counter()
        token()
        samples.append(time.perf_counter() - t0)
    best, median = min(samples), sorted(samples)[len(samples) // 2]
    return {"cpu_ms_per_token": best * 1e3, "cpu_ms_per_token_median": median * 1e3, "cpu_tokens": len(samples),
            "cpu_sample": ("restated reference Q8KCodec.QuantizeRow + ExecuteQuantizedTiled at one position "
                           "(oracle/satori_oracle_avx2.c), per projection, 197 projections of 28 distinct layer "
                           f"copies; {len(samples)} tokens, 1 thread pinned; min reported")}


def cpu_prefill_chunk(host, shapes, host_in, positions: int, repeats: int) -> dict:
    """One 256-position layer-chunk of the prefill on one host core through the restated reference path: per
    projection Q8KCodec.QuantizeRow of its 256 input rows, then ExecuteQuantizedTiled over the 256 positions
    (QuantizedKAvx2Kernel.cs:47-99, the reference's tile), as DenseForward.LayerBatch calls ExecuteBatch per
    projection. The whole prefill is that times 28 layers times the chunks, plus the output projection of the
    last position (extrapolated, labelled)."""
    from oracle import oracle as O

    def chunk():
        for name, data in host.items():
            if name == "output":
                continue
            r, c, fmt = shapes[name]
            x = host_in[FEEDS[name]][:positions * c]
            acts = np.concatenate([O.q8k_quantize_row(x[p * c:(p + 1) * c]) for p in range(positions)])
            O.qk_matvec_quantized_tiled_avx2(data, r, c, int(fmt), acts, positions, ys[name])

    ys = {name: np.zeros(positions * r, np.float32) for name, (r, _, _) in shapes.items() if name != "output"}
    samples = []
    for _ in range(repeats):
        t0 = time.perf_counter()
        chunk()
        samples.append(time.perf_counter() - t0)
    r, c, fmt = shapes["output"]
    t0 = time.perf_counter()
    O.qk_matvec_quantized_avx2(host["output"], r, c, int(fmt), O.q8k_quantize_row(host_in["h"][:c]))
    output_ms = (time.perf_counter() - t0) * 1e3
    best = min(samples) * 1e3
    return {"cpu_ms_per_layer_chunk": best, "cpu_chunk_positions": positions,
            "cpu_ms_extrapolated": best * 28 * 2 + output_ms,
            "cpu_sample": (f"restated reference QuantizeRow + ExecuteQuantizedTiled over {positions} positions "
                           f"(oracle/satori_oracle_avx2.c) for the 7 projections of one layer, {repeats} runs, "
                           "1 thread pinned, min reported; cpu_ms_extrapolated = 56 layer-chunks + the output "
                           "projection of the last position")}


def cpu_baseline(payload, rows, columns, block, x, seconds, scalar_seconds: float = 3.0) -> dict:
    """Restated reference AVX2 Ternary2 kernel (oracle), one host core, warm payload, bounded sample; and the
    scalar reference beside it (`scalar`)."""
    from oracle import oracle as O

    host = host_cpu()  # before pinning: the CPUs available to the process
    core = pin_one_core()
    y = np.zeros(rows, np.float32)
    O.t2_matvec_avx2(payload, rows, columns, block, x, y)  # warm
    iterations, start = 0, time.perf_counter()
    samples = []
    while time.perf_counter() - start < seconds:
        t0 = time.perf_counter()
        O.t2_matvec_avx2(payload, rows, columns, block, x, y)
        samples.append(time.perf_counter() - t0)
        iterations += 1
    elapsed = time.perf_counter() - start
    # The scalar reference (Ternary2MatVec.ExecuteScalarCore, restated in oracle/satori_oracle.c: sequential
    # FP32 adds, no fast-math), a bounded sample on the same pinned core.
    scalar_samples, s0 = [], time.perf_counter()
    while time.perf_counter() - s0 < scalar_seconds or len(scalar_samples) < 3:
        t0 = time.perf_counter()
        O.t2_matvec_scalar(payload, rows, columns, block, x)
        scalar_samples.append(time.perf_counter() - t0)
    scalar_best = min(scalar_samples)
    scalar = {
        "gbs": payload.size / scalar_best / 1e9,
        "ms_min": scalar_best * 1e3,
        "ms_median": sorted(scalar_samples)[len(scalar_samples) // 2] * 1e3,
        "runs": len(scalar_samples),
        "kind": "port",
        "sample": (f"restated reference scalar Ternary2MatVec.ExecuteScalarCore (oracle/satori_oracle.c) on the "
                   f"same payload and x, {len(scalar_samples)} MatVecs, 1 thread pinned to core {core}, min reported"),
        "published_ms": PUBLISHED_SCALAR_T2_4096_B128_MS,
        "published_gbs": payload.size / (PUBLISHED_SCALAR_T2_4096_B128_MS * 1e-3) / 1e9,
        "published_reference": "docs/benchmarks/avx2-2026-10-12 run 1, one thread of a Core Ultra 7 155H",
    }
    return {
        "value": payload.size * iterations / elapsed / 1e9,
        "unit": "GB/s",
        "cores": 1,
        "kind": "port",
        "host_model": host["model"],
        "host_logical_cpus": host["logical_cpus"],
        "host_cpus_available": host["available"],
        "sample": (f"restated reference AVX2 Ternary2Avx2Kernel (oracle/satori_oracle_avx2.c, -O3 -mavx2 -mfma) "
                   f"on the same 4096x4096 B128 payload and x, {iterations} MatVecs over {elapsed:.1f} s, "
                   f"1 thread pinned to core {core}; min {min(samples) * 1e3:.3f} ms, "
                   f"median {sorted(samples)[len(samples) // 2] * 1e3:.3f} ms; host: {host['model']}, "
                   f"{host['logical_cpus']} logical CPUs ({host['available']} available to this process)"),
        "scalar": scalar,
    }


def host_cpu() -> dict:
    """The host CPU's model name (as lscpu prints it) and logical CPU counts."""
    model = ""
    try:
        with open("/proc/cpuinfo") as f:
            model = next((l.split(":", 1)[1].strip() for l in f if l.startswith("model name")), "")
    except OSError:
        pass
    try:
        available = len(os.sched_getaffinity(0))
    except (AttributeError, OSError):
        available = None
    return {"model": model, "logical_cpus": os.cpu_count(), "available": available}


def ternary2_sweep(ctx, events, formats: dict) -> dict:
    """The Ternary2 size x block grid of the reference's own CPU benchmark (1024^2, 2048^2, 4096^2 x B64 / B128 /
    B256): for the two smaller sizes, a grouped launch over >= 1 GiB of distinct copies (HBM-streaming, every
    copy's output checked against the oracle first) and the single-matrix launch replayed from a graph; the
    4096^2 rows repeat the format entries measured above. The CPU column is filled in later."""
    out = {}
    for size in (1024, 2048, 4096):
        for b in (64, 128, 256):
            label = f"ternary2-{size}-b{b}"
            if size == 4096:
                f = formats.get(label)
                if f is None:
                    continue
                out[label] = {k: f[k] for k in ("payload_bytes", "copies", "gbs", "pct_hbm", "single_launch_graph_us",
                                                "parity_checked") if k in f}
            else:
                p, xb = make_ternary2(size, size, b)
                c = Case(ctx, label, lambda p=p, b=b, size=size: ctx.create_ternary2(size, size, b, p), p.size, size,
                         size, xb, False)
                parity = check_case(ctx, c, p, size, size, None, xb, b)
                m = measure(ctx, events, c, 50, 10)
                c.close()
                out[label] = {k: m[k] for k in ("payload_bytes", "copies", "gbs", "pct_hbm", "single_launch_graph_us")}
                out[label].update(parity)
            out[label]["published_avx2_gbs"] = PUBLISHED_AVX2_T2[(size, b)]
            out[label]["vs_published_avx2"] = out[label]["gbs"] / PUBLISHED_AVX2_T2[(size, b)]
    return out


def other_formats(ctx):
    """(label, make) for the Ternary2 block sizes besides 128 and the GGUF formats at their configurations;
    make() returns the grouped Case and the CPU baseline's arguments (payload, rows, columns, format or None
    for Ternary2, x, block size or quantized flag)."""
    rows = columns = 4096
    out = []
    for b in (64, 256):
        def make(b=b):
            p, xb = make_ternary2(rows, columns, b)
            c = Case(ctx, f"ternary2-4096-b{b}", lambda: ctx.create_ternary2(rows, columns, b, p), p.size, rows,
                     columns, xb, False)
            return c, (p, rows, columns, None, xb, b)
        out.append((f"ternary2-4096-b{b}", make))

    # The like-for-like input of the reference's own benchmark: NumericalCorpus.RandomMatrix (xorshift32
    # weights and x, as the oracle restates it), quantized to B128 (the payload bytes do not depend on values).
    def make_corpus():
        from oracle import oracle as O
        wc, xc = O.corpus_random_matrix(rows, columns)
        p = S.Ternary2Matrix.quantize(wc, rows, columns, 128).data
        c = Case(ctx, "ternary2-4096-b128-corpus", lambda: ctx.create_ternary2(rows, columns, 128, p), p.size, rows,
                 columns, xc, False)
        return c, (p, rows, columns, None, xc, 128)
    out.append(("ternary2-4096-b128-corpus", make_corpus))
    # Ternary2 beyond 4096 x 4096 (B = 128): FFN shapes of a 7B-class model and an 8192 x 8192 matrix.
    for r, cc in ((11008, 4096), (4096, 11008), (8192, 8192)):
        def make_large(r=r, cc=cc):
            label = f"ternary2-{r}x{cc}-b128"
            p, xb = make_ternary2(r, cc, 128)
            c = Case(ctx, label, lambda: ctx.create_ternary2(r, cc, 128, p), p.size, r, cc, xb, False)
            return c, (p, r, cc, None, xb, 128)
        out.append((f"ternary2-{r}x{cc}-b128", make_large))
    for fmt, r, cc, quantized, label in (
            (BQ.Q8_0, 4096, 4096, False, "q8_0-4096x4096"),
            (BQ.Q4_0, 11008, 4096, False, "q4_0-11008x4096"),
            (BQ.Q4_0, 4096, 11008, False, "q4_0-4096x11008"),
            (BQ.Q4_K, 8960, 1536, True, "q4_k-8960x1536-q8k"),
            (BQ.Q4_K, 1536, 8960, True, "q4_k-1536x8960-q8k"),
            (BQ.Q6_K, 8960, 1536, True, "q6_k-8960x1536-q8k"),
            (BQ.Q6_K, 1536, 8960, True, "q6_k-1536x8960-q8k"),
            # Q4_K at 4096 x 4096 and at larger FFN shapes (an 8B-class model's gate/up and down).
            (BQ.Q4_K, 4096, 4096, True, "q4_k-4096x4096-q8k"),
            (BQ.Q4_K, 14336, 4096, True, "q4_k-14336x4096-q8k"),
            (BQ.Q4_K, 4096, 14336, True, "q4_k-4096x14336-q8k"),
            # The K formats' FP32-activation MatVec (IQuantizedMatrix.Execute / ExecuteScalar's DotBlock; CPU:
            # QuantizedKAvx2Kernel.ExecuteQ4K / ExecuteQ6K).
            (BQ.Q4_K, 8960, 1536, False, "q4_k-8960x1536-f32"),
            (BQ.Q4_K, 1536, 8960, False, "q4_k-1536x8960-f32"),
            (BQ.Q4_K, 4096, 4096, False, "q4_k-4096x4096-f32"),
            (BQ.Q6_K, 8960, 1536, False, "q6_k-8960x1536-f32"),
            (BQ.Q6_K, 1536, 8960, False, "q6_k-1536x8960-f32")):
        def make(fmt=fmt, r=r, cc=cc, quantized=quantized, label=label):
            data, xf = make_gguf(fmt, r, cc)
            shape = S.QuantizedMatrixShape(r, cc, fmt)
            c = Case(ctx, label, lambda: ctx.create(data, shape), data.size, r, cc, xf, quantized)
            return c, (data, r, cc, fmt, xf, quantized)
        out.append((label, make))
    return out


def main() -> int:
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=200)
    ap.add_argument("--warmup", type=int, default=20)
    ap.add_argument("--cpu-seconds", type=float, default=10.0)
    ap.add_argument("--cpu-format-seconds", type=float, default=1.0,
                    help="CPU sample per format (restated reference AVX2 path, one core)")
    ap.add_argument("--cpu-decode-seconds", type=float, default=4.0,
                    help="CPU sample of the decode step's 197 projections (restated reference path, one core)")
    ap.add_argument("--warmup-seconds", type=float, default=1.5,
                    help="untimed headline launches before the first timed region (steady-state clocks)")
    ap.add_argument("--quick", action="store_true", help="headline workload only, no other formats")
    ap.add_argument("--profile", action="store_true",
                    help="only the headline grouped launches (for rocprofv3 kernel statistics), no other timing")
    ap.add_argument("--profile-prefill", action="store_true",
                    help="only the 512-position prefill (steps and warmup as given), for rocprofv3")
    ap.add_argument("--profile-decode", action="store_true",
                    help="only the decode step, launched eagerly (steps and warmup as given), for rocprofv3")
    ap.add_argument("--profile-token", action="store_true",
                    help="only the whole decode token at positions 511 and 4095, launched eagerly (steps and "
                         "warmup as given), for rocprofv3")
    ap.add_argument("--profile-single", action="store_true",
                    help="only the headline matrix's single launches (one per resident copy, checked against the "
                         "oracle first), steps and warmup as given, for rocprofv3")
    ap.add_argument("--profile-formats", action="store_true",
                    help="only the grouped launches of every format (steps and warmup as given), for rocprofv3")
    ap.add_argument("--profile-batch", action="store_true",
                    help="only the FP32-activation batches at 256 positions (checked against the oracle first; "
                         "steps and warmup as given), for rocprofv3")
    args = ap.parse_args()
    if args.gpus != 1:
        print("bench.py measures one GPU: the library runs the MatVec on a single MI355X "
              "(multi-GPU row sharding is design-only); run with --gpus 1", file=sys.stderr)
        return 2

    # The context and the events are released before the process exits: the stream and the device work are
    # torn down by the library, not by the runtime's exit path (a profiler attached to the process flushes
    # its buffers at exit).
    ctx = S.HipContext(0)
    events = HipEvents()
    try:
        return run(args, ctx, events)
    finally:
        events.close()
        try:
            ctx.dispose()
        except S.SatoriError as e:
            print(f"bench.py: context not released: {e}", file=sys.stderr)


def run(args, ctx, events) -> int:
    if args.profile_prefill or args.profile_decode or args.profile_token:
        model = DecodeModel(ctx)
        if args.profile_prefill:
            result = {"profile": "prefill", **prefill(ctx, events, model, args.steps, args.warmup)}
        elif args.profile_token:
            result = {"profile": "whole token (eager)", **token_eager(ctx, events, model, args.steps, args.warmup)}
        else:
            result = {"profile": "decode step (eager)",
                      **decode_step(ctx, events, model, args.steps, args.warmup, eager_only=True)}
        model.close()
        print(json.dumps(result))
        return 0

    if args.profile_batch:
        print(json.dumps({"profile": "FP32-activation batches", **batch_fp32(ctx, events, args.steps, args.warmup)}))
        return 0

    if args.profile_formats:
        lines = {}
        for label, make in other_formats(ctx):
            c, _ = make()
            warm_up(ctx, c.run_group, 0.25)
            ms = time_launches(ctx, events, c.run_group, args.steps, args.warmup)
            lines[label] = {"copies": c.copies, "launch_us": round(ms * 1e3, 2),
                            "gbs": round(c.copies * c.payload_bytes / (ms * 1e-3) / 1e9, 1),
                            "algorithmic_bytes_per_launch": c.copies * c.payload_bytes}
            progress(f"{label}: {lines[label]}")
            c.close()
        src, dst = ctx.alloc(CALIBRATION_BYTES), ctx.alloc(CALIBRATION_BYTES)
        ctx.copy_device(dst, src, CALIBRATION_BYTES)
        ctx.free(src)
        ctx.free(dst)
        print(json.dumps({"profile": "formats grouped", "launches": args.steps + args.warmup, "formats": lines,
                          "calibration_copy_bytes": CALIBRATION_BYTES}))
        return 0

    rows = columns = 4096
    block = 128
    payload, x = make_ternary2(rows, columns, block)
    head = Case(ctx, "ternary2-4096-b128", lambda: ctx.create_ternary2(rows, columns, block, payload),
                payload.size, rows, columns, x, False)
    try:
        head_parity = check_case(ctx, head, payload, rows, columns, None, x, block)
    except ParityError as e:
        print(f"bench.py: parity check failed, nothing timed: {e}", file=sys.stderr)
        return 1
    warm_up(ctx, head.run_group, args.warmup_seconds)
    if args.profile_single:
        head.run_single()
        check_outputs(ctx, head, "single launches")
        ms = time_launches(ctx, events, head.run_single, args.steps, args.warmup)
        print(json.dumps({"profile": "ternary2-4096-b128 single launches", "copies": head.copies,
                          "launches": (args.steps + args.warmup + 1) * head.copies,
                          "launch_us": round(ms * 1e3 / head.copies, 3)}))
        head.close()
        return 0
    if args.profile:
        ms = time_launches(ctx, events, head.run_group, args.steps, args.warmup)
        gbs = head.copies * payload.size / (ms * 1e-3) / 1e9
        # Calibration for the HBM byte counters: one device-to-device copy of a known size (the runtime's
        # copy kernel reads and writes CALIBRATION_BYTES each).
        src, dst = ctx.alloc(CALIBRATION_BYTES), ctx.alloc(CALIBRATION_BYTES)
        ctx.copy_device(dst, src, CALIBRATION_BYTES)
        ctx.free(src)
        ctx.free(dst)
        print(json.dumps({"profile": "ternary2-4096-b128 grouped", "launches": args.steps + args.warmup,
                          "launch_us": round(ms * 1e3, 2), "gbs": round(gbs, 1), "copies": head.copies,
                          "algorithmic_bytes_per_launch": head.copies * int(payload.size),
                          "calibration_copy_bytes": CALIBRATION_BYTES}))
        head.close()
        return 0
    headline = measure(ctx, events, head, args.steps, args.warmup)
    headline.update(head_parity)
    # The reference's measurement rule (several repetitions, never one run): five further timed repetitions,
    # their minimum, median, maximum and spread. The contract's value is the timed region above.
    rep_launches = 50
    warm_up(ctx, head.run_group, 0.25)  # the single-launch timings above ran last
    reps = sorted(head.copies * payload.size / (time_launches(ctx, events, head.run_group, rep_launches, 2) * 1e-3)
                  / 1e9 for _ in range(5))
    headline["repetitions"] = {"count": 5, "launches_each": rep_launches, "gbs_min": round(reps[0], 1),
                               "gbs_median": round(reps[2], 1), "gbs_max": round(reps[-1], 1),
                               "spread_pct": round(100.0 * (reps[-1] - reps[0]) / reps[2], 2)}
    # Timed region of the headline itself, for the contract fields.
    ms_per_step = headline["launch_us"] * 1e-3
    headline.update(host_call_latency(head))
    head.close()

    formats = {"ternary2-4096-b128": headline}
    cpu_cases = {"ternary2-4096-b128": (payload, rows, columns, None, x, block)}
    decode = pre = token = load = fbatch = sweep = None
    try:
        if not args.quick:
            for label, make in other_formats(ctx):
                c, cpu_case = make()
                parity = check_case(ctx, c, *cpu_case)
                formats[label] = measure(ctx, events, c, max(50, args.steps // 2), 10)
                formats[label].update(parity)
                formats[label].update(host_call_latency(c))
                cpu_cases[label] = cpu_case
                c.close()
            progress("Ternary2 size x block sweep (1024^2, 2048^2)")
            sweep = ternary2_sweep(ctx, events, formats)

        if not args.quick:
            progress("decode step (197 projections per token)")
            model = DecodeModel(ctx)
            model_host, model_shapes = model.host, model.shapes
            decode = decode_step(ctx, events, model, 50, 5)
            progress("whole decode token (operators + projections, position 511)")
            token = decode_token(ctx, events, model, 30, 3)
            progress("prefill (512 positions)")
            pre = prefill(ctx, events, model, 3, 1)
            model.close()
            progress("FP32-activation batches (256 positions)")
            fbatch = batch_fp32(ctx, events)
            progress("loading (GGUF, STQ2, STB1 uploads)")
            load = loading(ctx)
    except ParityError as e:
        print(f"bench.py: parity check failed: {e}", file=sys.stderr)
        return 1

    progress("cpu baseline")
    cpu = cpu_baseline(payload, rows, columns, block, x, args.cpu_seconds)
    if not args.quick:
        progress("cpu baseline per format")
        for label, case in cpu_cases.items():
            formats[label].update(cpu_format(*case, args.cpu_format_seconds))
            formats[label]["gpu_over_cpu"] = formats[label]["gbs"] / formats[label]["cpu_gbs"]
        progress("cpu baseline: Ternary2 sweep")
        for label, entry in sweep.items():
            if label in formats:
                entry["cpu_gbs"] = formats[label]["cpu_gbs"]
            else:
                size, b = int(label.split("-")[1]), int(label.split("-b")[1])
                p, xb = make_ternary2(size, size, b)
                entry["cpu_gbs"] = cpu_format(p, size, size, None, xb, b, 0.5)["cpu_gbs"]
            entry["gpu_over_cpu"] = entry["gbs"] / entry["cpu_gbs"]
        progress("cpu baseline: decode step and one prefill layer-chunk")
        decode.update(cpu_decode_step(model_host, model_shapes, decode_inputs(model), args.cpu_decode_seconds))
        decode["gpu_over_cpu"] = decode["cpu_ms_per_token"] * 1e3 / decode["us_per_token"]
        pre.update(cpu_prefill_chunk(model_host, model_shapes, prefill_inputs(model, 512), 256, 2))
        pre["gpu_over_cpu"] = pre["cpu_ms_extrapolated"] / pre["ms"]
    value = headline["gbs"]
    traffic, traffic_source = profiled_traffic("ternary2_4096_b128_grouped.md")
    line = {
        "metric": METRIC,
        "value": round(value, 2),
        "unit": "GB/s",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(ms_per_step, 4),
        "higher_is_better": True,
        "scaling": "weak",
        "vs_baseline": round(value / PUBLISHED_AVX2_T2_4096_B128, 1),
        "vs_baseline_reference": (f"published AVX2 Ternary2 4096x4096 B128, one thread of a Core Ultra 7 155H: "
                                  f"{PUBLISHED_AVX2_T2_4096_B128} GB/s (docs/benchmarks/avx2-2026-10-12)"),
        "vs_same_run_cpu": round(value / cpu["value"], 1),
        "dtype": "f32",
        "data": "synthetic",
        "config": {
            "workload": (f"Ternary2 MatVec 4096x4096 block 128, batch 1, FP32 x; one step = one grouped launch "
                         f"over {headline['copies']} resident copies ({headline['copies'] * payload.size / 1e9:.2f} GB "
                         f"of payload) so every step streams from HBM"),
            "payload_bytes_per_matvec": int(payload.size),
            "seed": 1729,
            "pct_of_hbm_peak": round(headline["pct_hbm"], 1),
        },
        "roofline": {
            "bound": "hbm",
            "achieved": round(value, 1),
            "peak": HBM_PEAK_GBS,
            "unit": "GB/s",
            "frac": round(value / HBM_PEAK_GBS, 4),
            "traffic": traffic,
            "traffic_source": traffic_source,
            "kernel": "t2_kernel<128, 16> + t2_fixup_kernel<16> (one grouped launch)",
            "launch_us": round(headline["launch_us"], 2),
            "algorithmic_bytes_per_launch": headline["copies"] * int(payload.size),
        },
        "repetitions": headline["repetitions"],
        "cpu_baseline": cpu,
        "decode_step": ({k: (round(v, 3) if isinstance(v, float) else v) for k, v in decode.items()}
                        if decode else None),
        "decode_token": ({k: (round(v, 3) if isinstance(v, float) else v) for k, v in token.items()}
                         if token else None),
        "prefill": ({k: (round(v, 3) if isinstance(v, float) else v) for k, v in pre.items()} if pre else None),
        "batch_fp32": ({label: {k: (round(v, 3) if isinstance(v, float) else v) for k, v in r.items()}
                        for label, r in fbatch.items()} if fbatch else None),
        "loading": ({k: round(v, 2) for k, v in load.items()} if load else None),
        "ternary2_sweep": ({label: {k: (round(v, 3) if isinstance(v, float) else v) for k, v in r.items()}
                            for label, r in sweep.items()} if sweep else None),
        "formats": {k: {kk: (round(vv, 3) if isinstance(vv, float) else vv) for kk, vv in v.items()}
                    for k, v in formats.items()},
    }
    print(json.dumps(line))
    return 0


if __name__ == "__main__":
    sys.exit(main())
