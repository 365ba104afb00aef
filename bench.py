"""Benchmark of the MI355X activation-offload engine on MOSS-Image DiT training.

Default run (one GPU): BASELINE config 3, a 5B-shaped DiT LoRA training step at 1024^2
(40 joint blocks, hidden 3072, 24x128 heads, MLP 12288, bf16 frozen weights N(0, 0.02), LoRA
rank 32 on q/k/v/o/ffn_up_gate/ffn_down, batch 1, 4096 latent + 512 text tokens, autocast bf16,
AdamW on the adapters), with every block's saved activations offloaded. Each regime is timed
three ways in the same process on the same seeds:

  none       hooks off (reference point for the hidden-copy fraction)
  engine     moss_offload.activation_cpu_offload (this project)
  reference  the reference's hook algorithm restated for the GPU (pinned tensor + copy_ on the
             compute stream + event per save; restore with empty_strided + copy_)

Regime A: every block under non-reentrant checkpointing (the reference default), so the hook
sees each block's inputs. Regime B: no checkpointing, so the hook sees every activation.

Prints ONE JSON line (stdout) with every leg's step times and rates; the whole record, 30 KB of
counters, goes to --detail. Progress goes to stderr.

Leg Q: the config-5 int8 weight-only GEMMs on the HIP MFMA kernels against the eager path.
Leg BR: regime B on the first 16 blocks, where the reference hooks' pinned copies fit the host.
Legs A4, C5U and C5P: config 4 (2048^2 + 4096 text tokens, regime A) and config 5 (int8 bases,
LoRA r16, four buckets, regime A) unpacked (four graphs before one backward) and packed (one
varlen traversal), 3 timed steps after 1 warm-up.
Leg AH: regime A with 100 ms of host work after every step, on both host-link transports (the
SDMA link's unpack waits on the host for its H2D; the HIP-stream link's never does).
Parity: loss and LoRA gradients against hooks off in regimes A, B and B at 16 blocks.

  python bench.py [--steps K] [--warmup W] [--regimes M,Q,A,B] [--micro-iters N]
"""

from __future__ import annotations

import argparse
import copy
import gc
import json
import os
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
# legs whose steps take seconds: timed over --steps-big steps
BIG_LEGS = ("A4", "B4", "B4R", "C5U", "C5P", "S5", "F3", "F3S")
# legs whose hooks-off and engine modes are timed in alternating rounds (--rounds-big), so that
# drift over the run falls on both alike; their exposed time is reported per round
INTERLEAVED = ("A4", "B4", "B4R", "C5U", "C5P")
# torch's pinned host allocator (the reference hooks' pin_memory) fails after about 55.6 GiB on
# the MI355X box (raw hipHostMalloc after about 65 GiB); a reference mode whose per-save pins
# would pass this is not attempted
PINNED_CAP_BYTES = 55 << 30
for _p in (ROOT / "moss-image_amd", ROOT):
    if str(_p) not in sys.path:
        sys.path.insert(0, str(_p))

HBM_PEAK_GBPS = 8000.0  # MI355X HBM3E
LINK_SPEC_GBPS = 64.0  # PCIe Gen5 x16, per direction

CONFIG3 = dict(dim=3072, ffn_dim=12288, num_heads=24, num_layers=40, text_dim=4096, freq_dim=256, latent_channels=16)
GRID = (64, 64)
TEXT_TOKENS = 512
LORA_RANK = 32
# 2048^2 (128 x 128 latent grid) + 4096 text tokens
C4_GRID = (128, 128)
C4_TEXT = 4096
# int8 weight-only bases, LoRA r16, batch of 4 aspect buckets (1024^2,
# 768x1344, 1344x768, 896x1152 -> latent grids /16) with fixed text lengths
C5_BUCKETS = ((64, 64), (48, 84), (84, 48), (56, 72))
C5_TEXT = (512, 384, 448, 256)
C5_RANK = 16


def log(msg: str) -> None:
    print(f"[bench {time.strftime('%H:%M:%S')}] {msg}", file=sys.stderr, flush=True)


# ---------------------------------------------------------------------------------------------
# reference hooks, restated for the GPU (baseline only; never the product path)


def reference_offload_context(model, enabled, device):
    """The reference algorithm (training/activation_offload.py:80-149) on PyTorch-ROCm."""

    import torch
    from contextlib import nullcontext

    if not enabled or device.type != "cuda" or not torch.is_grad_enabled():
        return nullcontext()

    def key(t):
        return t.device.type, t.device.index, t.untyped_storage().data_ptr()

    resident = {key(t) for t in (*model.parameters(), *model.buffers()) if t.device.type == "cuda"}

    def view_of(t):
        shape = list(t.shape)
        source = t
        for d, (size, stride) in enumerate(zip(t.shape, t.stride())):
            if stride < 0:
                return None
            if stride == 0 and size > 1:
                source = source.narrow(d, 0, 1)
                shape[d] = 1
        extent = 1
        for stride, size in sorted((st, sz) for sz, st in zip(shape, t.stride()) if sz > 1):
            if stride < extent:
                return None
            extent += (size - 1) * stride
        return source, tuple(shape)

    def pack(t):
        if t.device.type != "cuda" or key(t) in resident:
            return t
        view = view_of(t)
        if view is None:
            return t
        source, payload_shape = view
        cpu = torch.empty(payload_shape, dtype=t.dtype, device="cpu", pin_memory=True)
        cpu.copy_(source, non_blocking=True)
        ready = torch.cuda.Event()
        ready.record(torch.cuda.current_stream(t.device))
        return (cpu, t.device, ready, tuple(t.shape), tuple(t.stride()), payload_shape)

    def unpack(saved):
        if isinstance(saved, torch.Tensor):
            return saved
        cpu, device, ready, shape, stride, payload_shape = saved
        torch.cuda.current_stream(device).wait_event(ready)
        restored = torch.empty_strided(payload_shape, stride, dtype=cpu.dtype, device=device)
        restored.copy_(cpu, non_blocking=True)
        return restored.as_strided(shape, stride)

    return torch.autograd.graph.saved_tensors_hooks(pack, unpack)


# ---------------------------------------------------------------------------------------------
# workload


def build_model(device, layers: int):
    import torch
    from moss_offload import dit

    torch.manual_seed(0)
    cfg = dict(CONFIG3, num_layers=layers)
    with torch.device(device):
        model = dit.MOSSImageTransformer(**cfg)
    model = model.to(torch.bfloat16)
    dit.init_weights(model, std=0.02)
    dit.inject_lora(model, rank=LORA_RANK, alpha=float(LORA_RANK), b_std=0.03)
    return model.train()


def make_inputs(device, grid=GRID, text=TEXT_TOKENS, seed=0):
    import torch

    g = torch.Generator(device="cpu").manual_seed(seed)
    clean = torch.randn(1, CONFIG3["latent_channels"], *grid, generator=g).to(device)
    noise = torch.randn(clean.shape, generator=g).to(device)
    context = torch.randn(1, text, CONFIG3["text_dim"], generator=g).to(device)
    sigma = torch.rand(1, generator=g).to(device)
    return clean, noise, sigma, context


def build_c5_model(device, layers: int, int8_backend: str = "auto"):
    """Config 5: config-3 dims with int8 weight-only joint-block bases and LoRA r16; the bases
    run on ``int8_backend`` (auto: the HIP MFMA kernels, eager: decode + hipBLASLt)."""

    import torch
    from moss_offload import dit

    torch.manual_seed(0)
    cfg = dict(CONFIG3, num_layers=layers)
    with torch.device(device):
        model = dit.MOSSImageTransformer(**cfg)
    model = model.to(torch.bfloat16)
    dit.init_weights(model, std=0.02)
    dit.quantize_joint_linears(model, torch.Generator(device=device).manual_seed(5))
    dit.inject_lora(model, rank=C5_RANK, alpha=float(C5_RANK), b_std=0.03)
    dit.configure_quantized_backend(model, int8_backend)
    return model.train()


class InBackwardSGD:
    """Full-parameter SGD applied inside backward by post-accumulate-grad hooks: the shape of a
    fused optimizer such as the reference's FusedAdafactor (fused_adafactor.py:478-515), which the
    trainable block ring requires. Each hook updates its parameter in place and reports it."""

    def __init__(self, model, lr: float, streamer=None) -> None:
        self.lr = lr
        self.streamer = streamer
        for p in model.parameters():
            if p.requires_grad:
                p.register_post_accumulate_grad_hook(self._hook)

    def _hook(self, p) -> None:
        import torch

        grad = p.grad
        p.grad = None
        with torch.no_grad():
            p.add_(grad, alpha=-self.lr)
        if self.streamer is not None:
            self.streamer.mark_updated(p)

    def zero_grad(self, set_to_none: bool = True) -> None:
        pass

    def step(self) -> None:
        if self.streamer is not None:
            self.streamer.finish_backward()


def build_full_model(device, layers: int):
    """Config-3 dims, bf16, every parameter trainable (full fine-tuning)."""

    import torch
    from moss_offload import dit

    torch.manual_seed(0)
    with torch.device(device):
        model = dit.MOSSImageTransformer(**dict(CONFIG3, num_layers=layers))
    model = model.to(torch.bfloat16)
    dit.init_weights(model, std=0.02)
    return model.train()


def make_c5_batch(device):
    return [make_inputs(device, grid, text, seed=50 + i) for i, (grid, text) in enumerate(zip(C5_BUCKETS, C5_TEXT))]


def config3_forward(model, inputs):
    """One shape group: the squared velocity error and its element count (train.py:102-157)."""

    from moss_offload import dit

    clean, noise, sigma, context = inputs
    return dit.squared_error(model, clean, noise, sigma, context)


def grouped_forward(model, batch):
    """Config 5 unpacked: one forward per shape group, so four live graphs before one backward."""

    error, count = None, 0
    for inputs in batch:
        e, c = config3_forward(model, inputs)
        error = e if error is None else error + e
        count += c
    return error, count


def packed_forward(model, batch):
    """Config 5 packed: one varlen traversal over the four samples (model.py:502-626)."""

    import torch
    from moss_offload import dit

    noisy, velocity, contexts, sigmas = [], [], [], []
    for clean, noise, sigma, context in batch:
        n, v = dit.noisy_latent(clean, sigma, noise)
        noisy.append(n[0].to(model.compute_dtype))
        velocity.append(v[0])
        contexts.append(context[0].to(model.compute_dtype))
        sigmas.append(sigma)
    outputs = model.forward_packed(noisy, torch.cat(sigmas).float() * 1000.0, contexts)
    error = sum((o.float() - v.float()).square().sum() for o, v in zip(outputs, velocity))
    return error, sum(v.numel() for v in velocity)


def loss_and_backward(model, inputs, forward=config3_forward):
    import torch

    with torch.autocast("cuda", dtype=torch.bfloat16):
        error, count = forward(model, inputs)
    loss = error / count
    loss.backward()
    return loss.detach()


_SECOND_ENGINES: dict = {}


def hipdma_offload_context(model, enabled, device):
    """The engine's hooks on a second engine that moves its copies on HIP streams (link
    "hipdma": ordered by hipStreamWaitEvent, so an unpack never blocks the host)."""

    import torch
    import moss_offload
    from moss_offload.activation_offload import _ActivationOffload

    if not enabled or device.type != "cuda" or not torch.is_grad_enabled():
        return moss_offload.activation_cpu_offload(model, enabled, device)
    return _ActivationOffload(model, device, engine=hipdma_engine(device))


def hipdma_engine(device):
    import dataclasses

    from moss_offload.engine import OffloadEngine, get_engine

    engine = _SECOND_ENGINES.get("hipdma")
    if engine is None:
        engine = OffloadEngine(device, dataclasses.replace(get_engine(device).config, link="hipdma"))
        _SECOND_ENGINES["hipdma"] = engine
    return engine


def configure_mode(model, mode: str, regime: str):
    import moss_offload

    model.gradient_checkpointing = regime == "A"
    model.checkpoint_fraction = 1.0
    model.activation_offload = mode != "none"
    model.offload_context = {"reference": reference_offload_context,
                             "engine_hipdma": hipdma_offload_context}.get(mode, moss_offload.activation_cpu_offload)


def mode_engine(device, mode: str):
    """The engine a mode's hooks use (None for modes without one)."""

    from moss_offload.engine import get_engine

    if mode == "engine":
        return get_engine(device)
    if mode == "engine_hipdma":
        return hipdma_engine(device)
    return None


def host_work(seconds: float) -> None:
    """Busy the calling thread for ``seconds``: a trainer's per-step host work (data loading,
    logging), which overlaps the GPU only if the host thread is ahead of it."""

    end = time.perf_counter() + seconds
    while time.perf_counter() < end:
        pass


# engine statistics that are levels at the time of reading, not counts: summed over a mode's
# rounds they would mean nothing, so the last reading stands
ENGINE_LEVELS = ("groups_live", "entries_live", "host_bytes_in_use", "host_bytes_reserved", "device_ring_bytes",
                 "py_groups_live", "restore_slots_big", "restore_slots_small")


def add_counts(total: dict, reading: dict, latest=(), peak=()) -> None:
    """Add one reading of counters to ``total``: sums, except the ``latest`` keys (the last
    reading) and the ``peak`` keys (the largest)."""

    for key, value in reading.items():
        if key in latest or key not in total:
            total[key] = value
        elif key in peak:
            total[key] = max(total[key], value)
        else:
            total[key] += value


def time_steps(model, opt, inputs, steps: int, warmup: int, label: str, forward=config3_forward,
               host_work_s: float = 0.0):
    import torch

    for i in range(warmup):
        t0 = time.perf_counter()
        opt.zero_grad(set_to_none=True)
        loss_and_backward(model, inputs, forward)
        opt.step()
        host_work(host_work_s)
        torch.cuda.synchronize()
        log(f"{label}: warmup {i + 1}/{warmup} {time.perf_counter() - t0:.3f} s")
    torch.cuda.synchronize()
    gc.collect()
    torch.cuda.reset_peak_memory_stats()
    start = time.perf_counter()
    for i in range(steps):
        opt.zero_grad(set_to_none=True)
        loss_and_backward(model, inputs, forward)
        opt.step()
        host_work(host_work_s)
    torch.cuda.synchronize()
    elapsed = (time.perf_counter() - start) / steps
    peak = torch.cuda.max_memory_allocated()
    log(f"{label}: {elapsed:.4f} s/it over {steps} steps, peak device {peak / 2**30:.1f} GiB")
    return elapsed, peak


def _mode_step(model, inputs, mode: str, regime: str):
    import torch

    configure_mode(model, mode, regime)
    model.zero_grad(set_to_none=True)
    loss = loss_and_backward(model, inputs)
    grads = [p.grad.detach().float().clone() for p in model.parameters() if p.grad is not None]
    model.zero_grad(set_to_none=True)
    if mode == "reference":
        torch.cuda.synchronize()
        torch._C._host_emptyCache()
    return loss.float(), grads


def _compare_to_none(results: dict) -> dict:
    import torch

    base_loss, base_grads = results["none"]
    out = {}
    for mode, (loss, grads) in results.items():
        if mode == "none":
            continue
        num = sum(float((g - b).norm() ** 2) for g, b in zip(grads, base_grads)) ** 0.5
        den = sum(float(b.norm() ** 2) for b in base_grads) ** 0.5
        worst = max(float((g - b).norm() / b.norm().clamp_min(1e-30)) for g, b in zip(grads, base_grads))
        out[mode] = {"loss_rel": abs((loss - base_loss) / base_loss).item(), "grad_rel": num / den,
                     "worst_tensor_grad_rel": worst, "loss_bitwise": bool(torch.equal(loss, base_loss)),
                     "grads_bitwise": all(torch.equal(g, b) for g, b in zip(grads, base_grads)),
                     "lora_tensors": len(grads)}
    return out


def parity(model, inputs, ref_layers: int):
    """Loss and adapter gradients of one step per mode from the same state (no optimizer step),
    against hooks off: regime A (engine and reference hooks, 40 blocks), regime B (engine; the
    reference's per-save pinned copies exceed the host's pinned-memory cap at 40 blocks), and
    regime B at ``ref_layers`` blocks, where the reference hooks fit (engine and reference)."""

    from torch import nn

    out = {"A": _compare_to_none({m: _mode_step(model, inputs, m, "A") for m in ("none", "engine", "reference")}),
           "B": _compare_to_none({m: _mode_step(model, inputs, m, "B") for m in ("none", "engine")})}
    layers = model.layers
    model.layers = nn.ModuleList(list(layers)[:ref_layers])
    try:
        out[f"B{ref_layers}"] = _compare_to_none(
            {m: _mode_step(model, inputs, m, "B") for m in ("none", "engine", "reference")})
    finally:
        model.layers = layers
    return out


def link_peaks(device, nbytes: int = 256 << 20, iters: int = 10):
    """Measured pinned-host <-> device bandwidth (hipMemcpyAsync via torch, and the copy kernel)."""

    import ctypes

    import torch
    from moss_offload import _native

    dev = torch.empty(nbytes, dtype=torch.uint8, device=device)
    host = torch.empty(nbytes, dtype=torch.uint8, pin_memory=True)
    out = {}
    stream = torch.cuda.current_stream(device)
    for name, fn in (
        ("dma_d2h", lambda: host.copy_(dev, non_blocking=True)),
        ("dma_h2d", lambda: dev.copy_(host, non_blocking=True)),
    ):
        fn()
        torch.cuda.synchronize()
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record(stream)
        for _ in range(iters):
            fn()
        end.record(stream)
        end.synchronize()
        out[name] = nbytes * iters / (start.elapsed_time(end) / 1e3) / 1e9
    lib = _native.load()
    for name, dst, src in (("kernel_d2h", host, dev), ("kernel_h2d", dev, host)):
        for blocks in (64,):
            call = lambda: lib.mo_link_copy(dst.data_ptr(), src.data_ptr(), nbytes, 0, blocks, stream.cuda_stream)
            _native.check("mo_link_copy", call())
            torch.cuda.synchronize()
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record(stream)
            for _ in range(iters):
                _native.check("mo_link_copy", call())
            end.record(stream)
            end.synchronize()
            out[name] = nbytes * iters / (start.elapsed_time(end) / 1e3) / 1e9
    del dev, host
    return {k: round(v, 2) for k, v in out.items()}


def record_manifest(model, inputs, regime: str, forward=config3_forward):
    """Saved-tensor manifest of one step's forward in the given regime (bytes the hooks see)."""

    import torch
    from moss_offload.manifest import ManifestRecorder

    configure_mode(model, "none", regime)
    recorder = ManifestRecorder(model)
    marks = []
    layer = model.layers[len(model.layers) // 2]
    handles = [
        layer.register_forward_pre_hook(lambda m, a: marks.append(len(recorder.records))),
        layer.register_forward_hook(lambda m, a, o: marks.append(len(recorder.records))),
    ]
    try:
        with recorder, torch.autocast("cuda", dtype=torch.bfloat16):
            error, _ = forward(model, inputs)
    finally:
        for h in handles:
            h.remove()
    del error
    # the saves of one joint block (regime B: its activations; regime A: none inside, the
    # checkpoint saves the block inputs just before the pre-hook)
    recorder.block = recorder.records[marks[0] : marks[1]] if len(marks) >= 2 else []
    return recorder


def capture_block_saves(model, inputs):
    """The offloadable saved tensors of one joint block in regime B, in the order the hook sees them.

    One forward of the whole model without checkpointing; a pack hook keeps the tensors saved
    between the middle block's forward pre- and post-hooks, minus parameter/buffer-backed saves
    and layouts the reference keeps resident (training/activation_offload.py:101-121). Repeated
    saves of the same view are kept once (the engine deduplicates them).
    """

    import torch
    from moss_offload import dit
    from moss_offload.activation_offload import _bf16_exact, _offload_view, _storage_key

    configure_mode(model, "none", "B")
    resident = {_storage_key(t) for t in (*model.parameters(), *model.buffers())}
    layer = model.layers[len(model.layers) // 2]
    state = {"on": False}
    saved, seen, narrow = [], set(), []

    def pack(t):
        if state["on"] and t.device.type == "cuda" and _storage_key(t) not in resident and _offload_view(t) is not None:
            key = (t.data_ptr(), tuple(t.shape), tuple(t.stride()), t.dtype)
            if key not in seen:
                seen.add(key)
                # detached: a saved tensor's grad_fn would keep the whole graph (and every
                # activation up to this block) alive after the forward is dropped; whether the
                # hook would narrow it is decided now, while the graph is there
                saved.append(t.detach())
                narrow.append(_bf16_exact(t, _offload_view(t)[0]))
        # detached alias: returning `t` itself would tie outputs saved by their own node into
        # a reference cycle through the graph that the collector cannot break
        return t.detach()

    handles = [
        layer.register_forward_pre_hook(lambda m, a: state.__setitem__("on", True)),
        layer.register_forward_hook(lambda m, a, o: state.__setitem__("on", False)),
    ]
    clean, noise, sigma, context = inputs
    try:
        with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t), torch.autocast("cuda", dtype=torch.bfloat16):
            error, _ = dit.squared_error(model, clean, noise, sigma, context)
    finally:
        for h in handles:
            h.remove()
    del error
    return saved, narrow


def _same_bits(a, b) -> bool:
    import torch

    ints = {1: torch.uint8, 2: torch.int16, 4: torch.int32, 8: torch.int64}
    if a.shape != b.shape or a.stride() != b.stride() or a.dtype != b.dtype:
        return False
    dt = ints[a.element_size()]
    return bool(torch.equal(a.view(dt), b.view(dt)))


PACK_PROFILE = ROOT / "profiles" / "mo_pack_kernel_block_microbench.md"


def profiled_traffic():
    """HBM bytes per mo_pack_kernel launch on the microbench workload, from the committed
    rocprofv3 --pmc FETCH_SIZE / WRITE_SIZE summary (counters scaled by a calibration copy).
    None when the summary is not there."""

    import re

    try:
        text = PACK_PROFILE.read_text()
    except OSError:
        return None
    m = re.search(r"^traffic_bytes_per_launch:\s*(\d+)\s*$", text, re.M)
    return int(m.group(1)) if m else None


CAL_BYTES = 256 << 20
CAL_BLOCKS = 1024


def calibration_copy(device, stream: int, repeats: int = 3) -> None:
    """A plain device-to-device copy of CAL_BYTES with the engine's link-copy kernel.

    Under ``rocprofv3 --pmc FETCH_SIZE`` / ``WRITE_SIZE`` its dispatches (grid CAL_BLOCKS x 256)
    read and write exactly CAL_BYTES each, which scales the counters to bytes.
    """

    import torch
    from moss_offload import _native

    lib = _native.load()
    buf = torch.empty(2, CAL_BYTES, dtype=torch.uint8, device=device)
    for _ in range(repeats):
        _native.check("mo_link_copy", lib.mo_link_copy(buf[1].data_ptr(), buf[0].data_ptr(), CAL_BYTES, 0,
                                                       CAL_BLOCKS, stream))
    torch.cuda.synchronize()
    del buf


def kernel_context_leg(device, nbytes: int = 28 << 20, reps: int = 24):
    """Leg K: one-piece gathers and scatters of a regime-A checkpoint input's size (28 MiB),
    timed per dispatch with HIP events on the launch stream, back to back and right after other
    work: a GEMM with a 128 MiB output (what precedes an unpack in a checkpointed backward), a
    GEMM of the same power draw with a 128 KiB output, a 128 MiB fill and a 1 GiB read. Shows
    how much of a copy's in-step duration the state the previous kernel leaves behind sets."""

    import ctypes
    import statistics

    import torch
    from moss_offload import _native

    lib = _native.load()
    stream = torch.cuda.current_stream(device)
    pool = 6
    src = [torch.full((nbytes,), i + 1, dtype=torch.uint8, device=device) for i in range(pool)]
    dst = [torch.zeros(nbytes, dtype=torch.uint8, device=device) for _ in range(pool)]
    a = torch.randn(8192, 8192, device=device, dtype=torch.bfloat16)
    out_big = torch.empty(8192, 8192, device=device, dtype=torch.bfloat16)
    k1 = torch.randn(256, 1 << 20, device=device, dtype=torch.bfloat16)
    k2 = torch.randn(1 << 20, 256, device=device, dtype=torch.bfloat16)
    out_small = torch.empty(256, 256, device=device, dtype=torch.bfloat16)
    fill_buf = torch.empty(128 << 20, dtype=torch.uint8, device=device)
    read_buf = torch.randn(256 << 20, device=device)
    sink = torch.empty((), device=device)
    zero = (ctypes.c_uint64 * 1)(0)

    def described(t):
        arr = (_native.MoTensor * 1)()
        _native.describe(t, arr[0])
        return arr

    def gather(r):
        _native.check("mo_gather", lib.mo_gather(described(src[(r + 3) % pool]), 1, dst[r % pool].data_ptr(), zero,
                                                 stream.cuda_stream))

    def scatter(r):
        _native.check("mo_scatter", lib.mo_scatter(described(dst[r % pool]), 1, src[(r + 3) % pool].data_ptr(), zero,
                                                   stream.cuda_stream))

    before = {
        "back_to_back": None,
        "gemm_128MiB_output": lambda: torch.mm(a, a, out=out_big),
        "gemm_128KiB_output": lambda: torch.mm(k1, k2, out=out_small),
        "fill_128MiB": lambda: fill_buf.fill_(7),
        "read_1GiB": lambda: torch.sum(read_buf, dim=0, out=sink),
    }
    out = {"bytes_per_dispatch": nbytes, "dispatches": reps}
    for name, fn in before.items():
        row = {}
        for kind, op in (("gather", gather), ("scatter", scatter)):
            times = []
            for r in range(reps + 3):
                if fn is not None:
                    fn()
                start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                start.record(stream)
                op(r)
                end.record(stream)
                times.append((start, end))
            torch.cuda.synchronize()
            us = statistics.median(s.elapsed_time(e) * 1e3 for s, e in times[3:])
            row[kind] = {"median_us": round(us, 2), "tb_s": round(2 * nbytes / us / 1e6, 3)}
        out[name] = row
        log(f"kernel context {name}: gather {row['gather']['median_us']} us, scatter {row['scatter']['median_us']} us")
    return out


def micro(device, tensors, iters: int, warmup: int, slot_mib: int, stage_slots: int, restore_slots: int,
          batch_packs: bool = True, d2h_engine: int = 0, h2d_engine: int = 0, narrow=None, link: str = "sdma",
          cache: dict | None = None):
    """one regime-B block's saved set through pack -> D2H -> H2D -> unpack.

    Every iteration packs the block's tensors into one group (staging ring + SDMA D2H), commits
    it, restores every entry (SDMA H2D + unpack kernel, staged restore off so each byte crosses
    the link both ways) and releases the group. The sources are refilled with fresh random bits
    before the first and the last iteration, and those iterations' restored tensors are checked
    bitwise against them (shape, strides, dtype, bits).
    """

    import torch
    from moss_offload.engine import EngineConfig, OffloadEngine

    engine = OffloadEngine(device, EngineConfig(
        stage_slot_bytes=slot_mib << 20, stage_slots=stage_slots, restore_slots=restore_slots,
        stage_slots_max=0, restore_slots_max=0, restore_small_slots=0,  # the microbench's rings as given
        timing=True, kernel_timing=True, staged_restore=False, prefetch=False, batch_packs=batch_packs,
        d2h_engine=d2h_engine, h2d_engine=h2d_engine, link=link, **(cache or {})))
    stream = torch.cuda.current_stream(device).cuda_stream
    payload = sum(t.numel() * t.element_size() for t in tensors)
    storages = {}
    for t in tensors:
        storages.setdefault(t.untyped_storage().data_ptr(), t)

    narrow = list(narrow) if narrow is not None else [False] * len(tensors)

    def refill():
        for t in storages.values():
            torch.empty(0, dtype=torch.uint8, device=device).set_(t.untyped_storage()).random_(0, 256)
        for t, nr in zip(tensors, narrow):
            if nr:  # keep the float32 casts of bfloat16 values exact bfloat16, as the hook found them
                t.view(torch.int32).bitwise_and_(-65536)

    def one(keep: bool):
        refs = [engine.pack(t, stream, narrow=nr) for t, nr in zip(tensors, narrow)]
        engine.commit(stream)
        outs = [engine.restore(g, i, stream) for g, i in refs]
        for g, i in refs:
            engine.drop(g, i)
        return outs if keep else None

    def check(outs) -> bool:
        torch.cuda.synchronize()
        return all(_same_bits(o.as_strided(t.shape, t.stride()), t) for o, t in zip(outs, tensors))

    try:
        refill()
        first_ok = check(one(keep=True))
        for _ in range(max(0, warmup - 1)):
            one(keep=False)
        torch.cuda.synchronize()
        engine.synchronize()
        engine.reset_stats()
        start = time.perf_counter()
        for _ in range(iters):
            one(keep=False)
        torch.cuda.synchronize()
        engine.synchronize()
        seconds = (time.perf_counter() - start) / iters
        st = engine.stats()
        # after the timed region: fresh bits, one more iteration, checked
        refill()
        last_ok = check(one(keep=True))
        calibration_copy(device, stream)
    finally:
        engine.close()
    out = {
        "tensors": len(tensors),
        "payload_bytes": payload,
        "iters": iters,
        "s_per_iter": seconds,
        "bitwise_first": first_ok,
        "bitwise_last": last_ok,
        "d2h_gbps": st["timed_d2h_bytes"] / max(st["d2h_ms"], 1e-9) / 1e6,
        "h2d_gbps": st["timed_h2d_bytes"] / max(st["h2d_ms"], 1e-9) / 1e6,
        "pipeline_gbps": 2 * payload / seconds / 1e9,
        "pack_hbm_gbps": st["timed_pack_hbm_bytes"] / max(st["pack_ms"], 1e-9) / 1e6,
        "unpack_hbm_gbps": st["timed_unpack_hbm_bytes"] / max(st["unpack_ms"], 1e-9) / 1e6,
        "pack_avg_launch_us": st["pack_ms"] * 1e3 / max(st["timed_pack_launches"], 1),
        "unpack_avg_launch_us": st["unpack_ms"] * 1e3 / max(st["timed_unpack_launches"], 1),
        "pack_bytes_per_launch": st["timed_pack_bytes"] / max(st["timed_pack_launches"], 1),
        "unpack_bytes_per_launch": st["timed_unpack_bytes"] / max(st["timed_unpack_launches"], 1),
        "pack_hbm_bytes_per_launch": st["timed_pack_hbm_bytes"] / max(st["timed_pack_launches"], 1),
        "pack_launches_per_iter": st["timed_pack_launches"] / iters,
        "wire_segments": st["wire_segments"],
        "wire_ratio": (st["wire_bytes"] / st["wire_raw_bytes"]) if st["wire_raw_bytes"] else None,
        "unpack_launches_per_iter": st["timed_unpack_launches"] / iters,
        "host_blocks_per_iter": st["host_blocks"] / iters,
        "host_block_ms_per_iter": st["host_block_ms"] / iters,
        "copy_failures": st["copy_failures"],
    }
    return out


MFMA_BF16_PEAK_TFLOPS = 2500.0  # MI355X dense bf16 MFMA
# config-5 joint-block linears (out_features, in_features) and their count per block
C5_GEMMS = {"qkvo": ((3072, 3072), 4), "ffn_up_gate": ((2 * 12288, 3072), 1), "ffn_down": ((3072, 12288), 1)}


def int8_gemm_leg(device, iters: int = 20, warmup: int = 3, rounds: int = 3) -> dict:
    """Config-5 int8 weight-only GEMMs (moss_offload.quant_kernels) on the packed token count of
    one config-5 batch, forward and input gradient, by path:

      hip        the default dispatch (``auto``): the fused kernels for reductions at least four
                 times the output width whose plan splits a reduction, else one HIP decode and
                 the library GEMM
      fused      the fused MFMA kernels alone (weight decoded in registers)
      fused_lds  the same with the large tile decoding the weight into LDS
      library    one HIP decode, then the eager path's GEMM call
      eager      the reference's eager path: decode (cast, scale), then F.linear / matmul

    Timed with HIP events on the stream the kernels run on, ``rounds`` interleaved rounds of
    ``iters`` calls per path (after ``warmup`` calls), median of the rounds; TFLOP/s = 2 rows in
    out / call time."""

    import statistics

    import torch
    import torch.nn.functional as F

    from moss_offload import quant_kernels as qk

    rows = sum(h * w + t for (h, w), t in zip(C5_BUCKETS, C5_TEXT))
    g = torch.Generator(device=device).manual_seed(5)
    stream = torch.cuda.current_stream(device)
    calibration_copy(device, stream.cuda_stream)  # scales rocprofv3 FETCH_SIZE / WRITE_SIZE to bytes

    def timed(fn):
        for _ in range(warmup):
            fn()
        start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record(stream)
        for _ in range(iters):
            fn()
        stop.record(stream)
        stop.synchronize()
        return start.elapsed_time(stop) / 1e3 / iters

    def with_kernel(kernel, fn):
        def run():
            qk.set_kernel(kernel)
            try:
                fn()
            finally:
                qk.set_kernel("registers")
        return run

    paths = ("hip", "fused", "fused_lds", "library", "eager")
    shapes = {}
    block = dict.fromkeys(paths, 0.0)
    block_flop = 0.0
    ramped = False
    for name, ((out_f, in_f), count) in C5_GEMMS.items():
        x = torch.randn(rows, in_f, device=device, generator=g).to(torch.bfloat16)
        dy = torch.randn(rows, out_f, device=device, generator=g).to(torch.bfloat16)
        w = torch.randint(-127, 128, (out_f, in_f), dtype=torch.int8, device=device, generator=g)
        s = torch.empty(out_f, device=device).uniform_(1e-3, 2e-2, generator=g)
        assert qk.resolve_backend("auto", x, w, s, torch.bfloat16) == "hip"
        flop = 2.0 * rows * in_f * out_f
        calls = {
            "hip_fwd": lambda: qk.int8_linear_forward(x, w, s),
            "hip_bwd": lambda: qk.int8_linear_backward(dy, w, s, x.shape),
            "fused_fwd": lambda: qk.int8_linear_forward(x, w, s, path="fused"),
            "fused_bwd": lambda: qk.int8_linear_backward(dy, w, s, x.shape, path="fused"),
            "fused_lds_fwd": with_kernel("lds", lambda: qk.int8_linear_forward(x, w, s, path="fused")),
            "fused_lds_bwd": with_kernel("lds", lambda: qk.int8_linear_backward(dy, w, s, x.shape, path="fused")),
            "library_fwd": lambda: qk.int8_linear_forward(x, w, s, path="library"),
            "library_bwd": lambda: qk.int8_linear_backward(dy, w, s, x.shape, path="library"),
            "eager_fwd": lambda: F.linear(x, qk.decode(w, s, torch.bfloat16)),
            "eager_bwd": lambda: dy.matmul(qk.decode(w, s, torch.bfloat16)),
        }
        if not ramped:  # about a second of GEMMs first, so the clocks have settled
            for _ in range(8):
                timed(calls["eager_fwd"])
            ramped = True
        samples = {k: [] for k in calls}
        for _ in range(rounds):
            for k, fn in calls.items():
                samples[k].append(timed(fn))
        t = {k: statistics.median(v) for k, v in samples.items()}
        with torch.no_grad():
            wd = qk.decode(w, s, torch.bfloat16)
            yh, ye = qk.int8_linear_forward(x, w, s).float(), F.linear(x, wd).float()
            gh, ge = qk.int8_linear_backward(dy, w, s, x.shape).float(), dy.matmul(wd).float()
        rec = {"rows": rows, "in_features": in_f, "out_features": out_f, "per_block": count,
               "hip_fwd_path": "fused" if not torch.equal(yh, ye) else "library",
               "hip_bwd_path": "fused" if not torch.equal(gh, ge) else "library"}
        for k, sec in t.items():
            rec[k + "_ms"] = round(sec * 1e3, 4)
            rec[k + "_ms_range"] = [round(min(samples[k]) * 1e3, 4), round(max(samples[k]) * 1e3, 4)]
            rec[k + "_tflops"] = round(flop / sec / 1e12, 1)
        rec["fwd_vs_eager_max_rel_diff"] = ((yh - ye).abs().max() / ye.abs().max()).item()
        rec["bwd_vs_eager_max_rel_diff"] = ((gh - ge).abs().max() / ge.abs().max()).item()
        shapes[name] = rec
        for p_ in paths:
            block[p_] += count * (t[p_ + "_fwd"] + t[p_ + "_bwd"])
        block_flop += count * 2 * flop
        log(f"int8 GEMM {name} ({out_f}x{in_f}, {rows} rows), TFLOP/s fwd/bwd: "
            + " | ".join(f"{p_} {rec[p_ + '_fwd_tflops']}/{rec[p_ + '_bwd_tflops']}" for p_ in paths)
            + f" (hip: {rec['hip_fwd_path']}/{rec['hip_bwd_path']})")
        del x, dy, w, s, wd, yh, ye, gh, ge
    achieved = block_flop / block["hip"] / 1e12
    return {
        "shapes": shapes,
        "block_ms": {k: round(v * 1e3, 3) for k, v in block.items()},
        "block_speedup_vs_eager": round(block["eager"] / block["hip"], 4),
        "fused_block_speedup_vs_eager": round(block["eager"] / block["fused"], 4),
        "fused_lds_block_speedup_vs_eager": round(block["eager"] / block["fused_lds"], 4),
        "library_block_speedup_vs_eager": round(block["eager"] / block["library"], 4),
        "library_rows": qk.LIBRARY_ROWS,
        "library_weight_elements": qk.LIBRARY_WEIGHT,
        "long_reduction_ratio": qk.LONG_REDUCTION,
        "timing": f"median of {rounds} interleaved rounds of {iters} calls per path",
        "roofline": {"bound": "mfma",
                     "kernels": ("auto dispatch at these rows: mo_int8_ws_{fwd,kscale} (+ _split, mo_int8_split_reduce) "
                                 f"where the reduction is >= {qk.LONG_REDUCTION}x the output width and the plan splits "
                                 "it, else the library GEMM on the weight as mo_int8_decode_kernel, or for input "
                                 f"gradients from {qk.TRANSPOSED_REDUCTION[0]} to {qk.TRANSPOSED_REDUCTION[1]} features "
                                 "mo_int8_decode_transposed_kernel, gives it"),
                     "workload": "one config-5 joint block: 4 x qkvo + ffn_up_gate + ffn_down, forward and "
                                 f"input gradient, {rows} rows",
                     "achieved": round(achieved, 1), "peak": MFMA_BF16_PEAK_TFLOPS, "unit": "TFLOP/s",
                     "frac": round(achieved / MFMA_BF16_PEAK_TFLOPS, 4)},
    }


def host_grad_leg(device, layers: int, steps: int, warmup: int, threads: int) -> dict:
    """Host fp32 gradient accumulation (FusedAdafactor's CPU accumulation mode) on full-parameter
    training at config-3 dims (regime A): each logical step is two micro-batches; the first
    runs with the step disabled, so every gradient is stashed on the host, and the second
    applies an in-backward SGD update from the current gradient plus the host sum.

      device     early gradients stay on the device (the reference's default mode)
      engine     moss_offload.host_gradients.HostGradientAccumulator (16 x 64 MiB staging slots +
                 SDMA + background fp32 adds; the take through pop_to_device, prefetched by SDMA)
      reference  the reference's stash restated: fp32 pinned tensor, blocking copy_, host add_
    """

    import torch

    from moss_offload.harness_optim import HostModeSGD
    from moss_offload.host_gradients import HostGradientAccumulator

    model = build_full_model(device, layers)
    model.gradient_checkpointing = True
    model.checkpoint_fraction = 1.0
    model.activation_offload = False
    micro = [make_inputs(device, seed=0), make_inputs(device, seed=1)]
    trainable = [p for p in model.parameters() if p.requires_grad]
    grad_bytes = sum(p.numel() * p.element_size() for p in trainable)
    out = {"layers": layers, "micro_batches": 2, "parameters": sum(p.numel() for p in trainable),
           "gradient_bytes_per_micro_batch": grad_bytes, "host_threads": threads}
    gc.collect()
    gc.freeze()

    def logical_step(opt):
        opt.set_step_enabled(False)
        loss_and_backward(model, micro[0])
        opt.set_step_enabled(True)
        loss_and_backward(model, micro[1])
        opt.finish_backward()

    for mode in ("device", "engine", "reference"):
        acc = HostGradientAccumulator(device, slots=16, host_threads=threads) if mode == "engine" else None
        opt = HostModeSGD(trainable, 1e-6, stash=mode, accumulator=acc)
        for i in range(warmup):
            t0 = time.perf_counter()
            logical_step(opt)
            torch.cuda.synchronize()
            log(f"G/{mode}: warmup {i + 1}/{warmup} {time.perf_counter() - t0:.3f} s")
        if acc is not None:
            acc.synchronize()
            acc.reset_stats()
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        start = time.perf_counter()
        for _ in range(steps):
            logical_step(opt)
        torch.cuda.synchronize()
        elapsed = (time.perf_counter() - start) / steps
        rec = {"s_per_step": elapsed, "peak_device_bytes": torch.cuda.max_memory_allocated()}
        if acc is not None:
            st = acc.stats()
            rec.update(
                link_bytes_per_step=st["bytes"] / steps,
                d2h_gbps=st["d2h_done_bytes"] / max(st["d2h_ms"], 1e-9) / 1e6,
                d2h_busy_s_per_step=st["d2h_ms"] / 1e3 / steps,
                host_accumulate_s_per_step=st["accumulate_ms"] / 1e3 / steps,
                host_accumulate_gelems_per_s=st["elements"] / max(st["accumulate_ms"], 1e-9) / 1e6,
                host_blocks_per_step=st["host_blocks"] / steps,
                host_block_s_per_step=st["host_block_ms"] / 1e3 / steps,
                copy_failures=st["copy_failures"],
            )
        log(f"G/{mode}: {elapsed:.4f} s per logical step (2 micro-batches), peak device "
            f"{rec['peak_device_bytes'] / 2**30:.1f} GiB")
        opt.close()
        del opt, acc
        gc.collect()
        torch.cuda.synchronize()
        torch._C._host_emptyCache()
        out[mode] = rec
    base = out["device"]["s_per_step"]
    for mode in ("engine", "reference"):
        out[mode]["exposed_s"] = out[mode]["s_per_step"] - base
    return out


def cpu_baseline(recorder, threads: int, budget_s: float = 15.0):
    """The oracle's restatement of the reference hooks with CPU payloads, on the host cores.

    Sample: the saved-tensor set of ONE 1024^2 joint block in regime B (shapes, strides and
    dtypes from the recorded manifest, data N(0, 1)), packed (dense copy) and unpacked
    (empty_strided + copy_ + as_strided) repeatedly within ``budget_s``.
    """

    import torch
    from oracle import reference_hooks

    torch.set_num_threads(threads)
    block = [r for r in recorder.block if not r.resident and r.dup_of is None]
    if not block:  # regime A: nothing is saved inside a checkpointed block; use the whole step
        block = [r for r in recorder.offloaded() if r.dup_of is None]
    tensors = []
    for r in block:
        span = 1 + sum((s - 1) * st for s, st in zip(r.shape, r.stride) if s > 0)
        backing = torch.randn(span, dtype=torch.float32).to(r.dtype) if r.dtype.is_floating_point else torch.zeros(span, dtype=r.dtype)
        tensors.append(backing.as_strided(r.shape, r.stride))
    payload = sum(r.payload_bytes for r in block)
    start = time.perf_counter()
    iters = 0
    while True:
        for t in tensors:
            source, payload_shape = reference_hooks.offload_view(t)
            cpu = torch.empty(payload_shape, dtype=t.dtype)
            cpu.copy_(source)
            reference_hooks.restore_layout(cpu, t.device, tuple(t.shape), tuple(t.stride()), payload_shape, non_blocking=False)
        iters += 1
        if time.perf_counter() - start > budget_s:
            break
    elapsed = time.perf_counter() - start
    gbps = 2 * payload * iters / elapsed / 1e9  # pack + unpack each move P
    return {"gbps": gbps, "iters": iters, "payload_bytes": payload, "seconds": elapsed}


def run(args) -> dict:
    import torch

    import moss_offload
    from moss_offload.engine import configure, get_engine

    device = torch.device("cuda", 0)
    props = torch.cuda.get_device_properties(device)
    log(f"device {props.name}, {props.total_memory / 2**30:.0f} GiB, host cores {os.cpu_count()}")
    configure(
        timing=True,
        kernel_timing=True,
        stage_slots=args.stage_slots,
        restore_slots=args.restore_slots,
        stage_slots_max=args.stage_slots_max,
        restore_slots_max=args.restore_slots_max,
        restore_small_slots=args.restore_small_slots,
        prefetch_depth=args.prefetch_depth,
        stage_slot_bytes=args.slot_mib << 20,
        **({} if args.restore_ahead_mib is None else {"restore_ahead_bytes": args.restore_ahead_mib << 20}),
        staged_restore=not args.no_staged_restore,
        kernel_copy=args.kernel_copy,
        link=args.link,
        pack_nt_load=not args.pack_cached_load,
        unpack_nt_load=not args.unpack_cached_load,
        unpack_nt_store=not args.unpack_cached_store,
        batch_packs=not args.eager_pack,
        d2h_engine=args.d2h_engine,
        h2d_engine=args.h2d_engine,
        narrow_bf16_casts=not args.no_narrow,
        wire_coding=args.wire_coding,
    )
    model = build_model(device, args.layers)
    inputs = make_inputs(device)
    params = [p for p in model.parameters() if p.requires_grad]
    opt = torch.optim.AdamW(params, lr=1e-4, foreach=True)
    log(f"model built: {sum(p.numel() for p in model.parameters()) / 1e9:.2f} B params, {len(params)} adapter tensors")
    # Long-lived objects (model, optimizer, modules) leave the cyclic collector's scope, as in a
    # production training loop: a full collection over them stalls the host for ~100 ms at
    # random steps, in every mode alike, which would otherwise dominate the step-time noise.
    gc.collect()
    gc.freeze()

    peaks = link_peaks(device)
    log(f"host link: {peaks}")
    # 256 MiB device-to-device copies with the engine's copy kernel: under rocprofv3 --pmc they
    # scale FETCH_SIZE / WRITE_SIZE to bytes for any leg of this run
    calibration_copy(device, torch.cuda.current_stream(device).cuda_stream)

    result = {"regimes": {}, "link": peaks, "hook_features": moss_offload.hook_features()}
    if not args.no_parity:
        result["parity"] = parity(model, inputs, args.ref_layers)
        log(f"parity: {result['parity']}")

    if "M" in args.regimes:
        tensors, narrow = capture_block_saves(model, inputs)
        if args.no_narrow:
            narrow = [False] * len(tensors)
        torch.cuda.synchronize()
        payload = sum(t.numel() * t.element_size() for t in tensors)
        moved = sum(t.numel() * (2 if nr else t.element_size()) for t, nr in zip(tensors, narrow))
        log(f"micro: one regime-B block, {len(tensors)} unique saves, {payload / 1e6:.1f} MB "
            f"({sum(narrow)} bf16 casts narrowed: {moved / 1e6:.1f} MB over the link)")
        result["micro"] = micro(device, tensors, args.micro_iters, args.micro_warmup, args.slot_mib,
                                args.stage_slots, args.restore_slots, batch_packs=not args.eager_pack,
                                d2h_engine=args.d2h_engine, h2d_engine=args.h2d_engine, narrow=narrow,
                                link=args.link,
                                cache=dict(wire_coding=args.micro_wire_coding,
                                           pack_nt_load=not args.pack_cached_load,
                                           unpack_nt_load=not args.unpack_cached_load,
                                           unpack_nt_store=not args.unpack_cached_store))
        result["micro"].update(narrowed_tensors=sum(narrow), link_bytes_per_iter=moved)
        m = result["micro"]
        log(f"micro: {m['s_per_iter'] * 1e3:.2f} ms/iter, D2H {m['d2h_gbps']:.1f} GB/s, H2D {m['h2d_gbps']:.1f} GB/s, "
            f"pack {m['pack_hbm_gbps']:.0f} GB/s ({m['pack_avg_launch_us']:.1f} us/launch), unpack "
            f"{m['unpack_hbm_gbps']:.0f} GB/s, bitwise {m['bitwise_first'] and m['bitwise_last']}")
        del tensors

    if "K" in args.regimes:
        result["kernel_context"] = kernel_context_leg(device)
        torch.cuda.empty_cache()
    if "Q" in args.regimes:
        result["int8_gemm"] = int8_gemm_leg(device)
        torch.cuda.empty_cache()
    if "G" in args.regimes:
        result["host_gradients"] = host_grad_leg(device, args.layers, max(1, args.steps_b), max(1, args.warmup_b),
                                                 args.gradacc_threads)
        torch.cuda.empty_cache()

    c4 = {}
    c5 = {}
    full = {}

    def workload(name):
        """(model, optimizer, inputs, forward, checkpoint regime) of a bench leg."""

        if name in ("A", "B"):
            return model, opt, inputs, config3_forward, name
        if name == "AH":  # regime A with host work after every step (the transports' host blocking)
            return model, opt, inputs, config3_forward, "A"
        if name == "BR":  # regime B on the first --ref-layers blocks, where the reference hooks fit
            layers = model.layers
            model.layers = torch.nn.ModuleList(list(layers)[: args.ref_layers])
            cleanups.append(lambda: setattr(model, "layers", layers))
            return model, opt, inputs, config3_forward, "B"
        if name == "BK":  # regime B with the engine keeping the last --keep-last-blocks blocks resident
            return model, opt, inputs, config3_forward, "B"
        if name == "A4":
            return model, opt, make_inputs(device, C4_GRID, C4_TEXT, seed=4), config3_forward, "A"
        if name in ("B4", "B4R"):
            # config 4 (2048^2 + 4096 text) not checkpointed, so the host link sets the pace: on
            # --b4-layers blocks, whose coded saves fit the pinned-memory cap, and on
            # --b4-ref-layers, where the reference hooks' per-save pins fit it too
            layers = model.layers
            count = args.b4_layers if name == "B4" else args.b4_ref_layers
            model.layers = torch.nn.ModuleList(list(layers)[:count])
            cleanups.append(lambda: setattr(model, "layers", layers))
            if "c4" not in c4:
                c4["c4"] = make_inputs(device, C4_GRID, C4_TEXT, seed=4)
            return model, opt, c4["c4"], config3_forward, "B"
        if name in ("C5U", "C5P"):
            if not c5:
                c5["model"] = build_c5_model(device, args.layers, args.int8_backend)
                c5["opt"] = torch.optim.AdamW([p for p in c5["model"].parameters() if p.requires_grad], lr=1e-4,
                                              foreach=True)
                c5["batch"] = make_c5_batch(device)
                gc.collect()
                gc.freeze()
            forward = grouped_forward if name == "C5U" else packed_forward
            return c5["model"], c5["opt"], c5["batch"], forward, "A"
        if name == "S5":
            # config 5's low-VRAM path: every joint block streamed from pinned host masters
            # (frozen int8 bases; adapters stay on the device), packed batch
            if "streamed" not in c5:
                workload("C5P")
                from moss_offload.memory import place_model

                streamed = copy.deepcopy(c5["model"])
                place_model(streamed, device, len(streamed.layers), block_swap_mode="async")
                c5["streamed"] = streamed
                c5["streamed_opt"] = torch.optim.AdamW([p for p in streamed.parameters() if p.requires_grad],
                                                       lr=1e-4, foreach=True)

                def loss_and_grads(m):
                    configure_mode(m, "none", "A")
                    m.zero_grad(set_to_none=True)
                    loss = loss_and_backward(m, c5["batch"], packed_forward)
                    grads = [p.grad.detach().float().clone() for p in m.parameters() if p.grad is not None]
                    m.zero_grad(set_to_none=True)
                    return loss.float(), grads

                base_loss, base_grads = loss_and_grads(c5["model"])
                loss, grads = loss_and_grads(streamed)
                num = sum(float((g - b).norm() ** 2) for g, b in zip(grads, base_grads)) ** 0.5
                den = sum(float(b.norm() ** 2) for b in base_grads) ** 0.5
                def device_bytes(m):
                    tensors = {t.untyped_storage().data_ptr(): t.untyped_storage().nbytes()
                               for t in (*m.parameters(), *m.buffers()) if t.is_cuda}
                    manager = getattr(m, "block_swap_manager", None)
                    if manager is not None:
                        tensors.update({b.data_ptr(): b.numel() for b in manager.owned_cuda_buffers()})
                    return sum(tensors.values())

                result["stream_parity"] = {"loss_bitwise": bool(torch.equal(loss, base_loss)),
                                           "loss_rel": abs(float((loss - base_loss) / base_loss)),
                                           "grad_rel": num / den, "grads": len(grads),
                                           "resident_model_device_bytes": device_bytes(c5["model"]),
                                           "streamed_model_device_bytes": device_bytes(streamed)}
                log(f"stream parity: {result['stream_parity']}")
                del base_grads, grads
                torch.cuda.empty_cache()
                gc.collect()
                gc.freeze()
            return c5["streamed"], c5["streamed_opt"], c5["batch"], packed_forward, "A"
        if name in ("F3", "F3S"):
            # full-parameter training with an in-backward optimizer; F3S streams every block
            # through the trainable two-slot ring (async_full)
            if name not in full:
                if "F3" not in full:
                    resident = build_full_model(device, args.layers)
                    full["F3"] = (resident, InBackwardSGD(resident, 1e-6))
                if name == "F3S":
                    from moss_offload.memory import place_model

                    streamed = build_full_model(device, args.layers)
                    place_model(streamed, device, len(streamed.layers), block_swap_mode="async_full")
                    full["F3S"] = (streamed, InBackwardSGD(streamed, 1e-6, streamed.block_swap_manager))
                torch.cuda.empty_cache()
                gc.collect()
                gc.freeze()
            model_f, opt_f = full[name]
            return model_f, opt_f, inputs, config3_forward, "A"
        raise ValueError(f"unknown regime {name}")

    def run_leg(regime_name):
        wl_model, wl_opt, wl_inputs, forward, regime = workload(regime_name)
        manifest = record_manifest(wl_model, wl_inputs, regime, forward)
        payload_unique = manifest.payload_bytes(unique=True)
        payload_copied = manifest.payload_bytes(unique=False)
        torch.cuda.synchronize()
        log(f"regime {regime_name}: hooks see {len(manifest.records)} saves, payload {payload_unique / 1e9:.2f} GB "
            f"unique ({payload_copied / 1e9:.2f} GB as the reference copies it)")
        if regime_name == "A":
            steps, warmup = args.steps, args.warmup
        elif regime_name in BIG_LEGS:
            steps, warmup = max(1, args.steps_big), max(1, args.warmup_big)
        else:
            steps, warmup = max(1, args.steps_b), max(1, args.warmup_b)
        host_work_s = args.host_work_ms / 1e3 if regime_name == "AH" else 0.0
        if regime_name == "BK":
            entry_extra = {"keep_last_blocks": args.keep_last_blocks}
        elif regime_name == "AH":
            entry_extra = {"host_work_ms_per_step": args.host_work_ms}
        elif regime_name == "BR":
            entry_extra = {"layers": len(wl_model.layers)}
        else:
            entry_extra = {}
        block = [r for r in manifest.block if not r.resident]
        entry = {"payload_unique_bytes": payload_unique, "payload_copied_bytes": payload_copied,
                 "saves": len(manifest.records),
                 "block_payload_unique_bytes": sum(r.payload_bytes for r in block if r.dup_of is None),
                 "block_payload_copied_bytes": sum(r.payload_bytes for r in block), **entry_extra}
        if regime_name == "B":
            entry["cpu_sample"] = manifest
        streamer = getattr(wl_model, "block_swap_manager", None)
        modes = list(args.modes)
        if regime_name == "AH" and "engine" in modes:
            modes.insert(modes.index("engine") + 1, "engine_hipdma")
        if regime_name == "BK" and "reference" in modes:
            modes.remove("reference")  # the reference offloads every block
        if "reference" in modes:
            # the reference pins one host tensor per save, dups included, each rounded up to a
            # power of two by torch's caching host allocator
            pins = sum(1 << max(0, (r.payload_bytes - 1).bit_length()) for r in manifest.records
                       if not r.resident and r.payload_bytes)
            if pins > PINNED_CAP_BYTES:
                modes.remove("reference")
                entry["reference"] = {"skipped": f"needs {pins / 2**30:.1f} GiB of pinned host memory per step "
                                      f"(one pin per save), over the {PINNED_CAP_BYTES / 2**30:.0f} GiB a process "
                                      f"can pin on this box", "pinned_bytes_needed": pins}
                log(f"{regime_name}/reference skipped: {entry['reference']['skipped']}")
        rounds = max(1, args.rounds_big) if regime_name in INTERLEAVED else 1
        times = {mode: [] for mode in modes}
        peaks = {mode: 0 for mode in modes}
        counted = {mode: 0 for mode in modes}  # steps (warmup included) the statistics below cover
        engine_stats, hook_stats, stream_stats = {}, {}, {}
        failed = {}

        def enter(mode, first):
            configure_mode(wl_model, mode, regime)
            engine = mode_engine(device, mode) or get_engine(device)
            engine.config.keep_last_blocks = args.keep_last_blocks if regime_name == "BK" else 0
            if first:
                # wire buffers a previous leg allocated (coding ran there) are freed, so each
                # leg's ring bytes are its own
                engine.trim()
                # marks the start of each leg and mode in a kernel trace, and scales rocprofv3
                # FETCH_SIZE / WRITE_SIZE to bytes in a counter run
                calibration_copy(device, torch.cuda.current_stream(device).cuda_stream)
            # every mode and round starts from zero (the modes share the engine), and what it
            # counted is added to its own totals right after it ran
            engine.reset_stats()
            if first:
                free, total = torch.cuda.mem_get_info(device)
                st0 = engine.stats()
                log(f"{regime_name}/{mode}: device free {free / 2**30:.1f} of {total / 2**30:.1f} GiB, torch reserved "
                    f"{torch.cuda.memory_reserved(device) / 2**30:.1f} GiB, engine rings {st0['device_ring_bytes'] / 2**30:.1f} "
                    f"GiB, pinned pool {st0['host_bytes_reserved'] / 2**30:.1f} GiB")
            moss_offload.reset_hook_counters()
            if streamer is not None:
                streamer.reset_stats()
            return engine

        def collect(mode, engine, nsteps):
            counted[mode] += nsteps
            add_counts(hook_stats.setdefault(mode, {}), moss_offload.hook_counters())
            if streamer is not None:
                torch.cuda.synchronize()
                add_counts(stream_stats.setdefault(mode, {}), streamer.stats())
            if mode in ("engine", "engine_hipdma"):
                engine.synchronize()
                add_counts(engine_stats.setdefault(mode, {}), engine.stats(), latest=ENGINE_LEVELS,
                           peak=("host_bytes_peak",))

        for rnd in range(rounds):
            for mode in modes:
                if mode in failed or (mode == "reference" and rnd > 0):  # one round of the baseline
                    continue
                engine = enter(mode, rnd == 0)
                try:
                    seconds, peak = time_steps(wl_model, wl_opt, wl_inputs, steps, warmup if rnd == 0 else 0,
                                               f"{regime_name}/{mode}" + (f" round {rnd + 1}/{rounds}" if rounds > 1 else ""),
                                               forward, host_work_s)
                except RuntimeError as exc:  # e.g. the reference hooks exhausting pinned host memory
                    import traceback

                    log(f"{regime_name}/{mode} failed: {exc}\n{traceback.format_exc(limit=-4)}")
                    failed[mode] = str(exc).splitlines()[0]
                    # the traceback held the failed step's graph, and with it every pinned copy it
                    # made; they are freed now, and the cached pinned blocks go back to the host
                    wl_opt.zero_grad(set_to_none=True)
                    gc.collect()
                    torch.cuda.synchronize()
                    torch._C._host_emptyCache()
                    continue
                times[mode].append(seconds)
                peaks[mode] = max(peaks[mode], peak)
                collect(mode, engine, steps + (warmup if rnd == 0 else 0))
                if mode == "reference":
                    torch._C._host_emptyCache()

        for mode in modes:
            if mode in failed:
                entry[mode] = {"error": failed[mode]}
                continue
            engine = mode_engine(device, mode) or get_engine(device)
            timed = times[mode]
            record = {"s_per_it": sum(timed) / len(timed), "peak_device_bytes": peaks[mode]}
            if len(timed) > 1:
                record["s_per_it_rounds"] = timed
            n = counted[mode]
            if streamer is not None:
                ss = stream_stats[mode]
                record["stream"] = {
                    "fills_per_step": ss["fills"] / n,
                    "bytes_per_step": ss["bytes"] / n,
                    "busy_s_per_step": ss["busy_ms"] / 1e3 / n,
                    "h2d_gbps": ss["timed_bytes"] / max(ss["busy_ms"], 1e-9) / 1e6,
                    "host_block_ms_per_step": ss["host_block_ms"] / n,
                    "copy_failures": ss["copy_failures"],
                    "writebacks_per_step": ss["writebacks"] / n,
                    "writeback_bytes_per_step": ss["writeback_bytes"] / n,
                    "writeback_busy_s_per_step": ss["writeback_busy_ms"] / 1e3 / n,
                    "writeback_gbps": ss["timed_writeback_bytes"] / max(ss["writeback_busy_ms"], 1e-9) / 1e6,
                }
            if mode in ("engine", "engine_hipdma"):
                engine.synchronize()
                st = engine_stats[mode]
                record["link"] = engine.link_name()
                record["hook_counters_per_step"] = {k: v / n for k, v in hook_stats[mode].items()}
                # the staging and restore rings (and their wire buffers once coding ran) are the
                # engine's own hipMalloc, outside torch's allocator and so outside peak_device_bytes
                rings = st["device_ring_bytes"]
                record.update(
                    engine_ring_bytes=rings,
                    peak_device_bytes_with_rings=peaks[mode] + rings,
                    d2h_bytes_per_step=st["bytes_d2h"] / n,
                    h2d_bytes_per_step=st["bytes_h2d"] / n,
                    d2h_copies_per_step=st["d2h_copies"] / n,
                    h2d_copies_per_step=st["h2d_copies"] / n,
                    d2h_s_per_step=st["d2h_ms"] / 1e3 / n,
                    h2d_s_per_step=st["h2d_ms"] / 1e3 / n,
                    d2h_gbps=st["timed_d2h_bytes"] / max(st["d2h_ms"], 1e-9) / 1e6,
                    h2d_gbps=st["timed_h2d_bytes"] / max(st["h2d_ms"], 1e-9) / 1e6,
                    pack_hbm_gbps=st["timed_pack_hbm_bytes"] / max(st["pack_ms"], 1e-9) / 1e6,
                    unpack_hbm_gbps=st["timed_unpack_hbm_bytes"] / max(st["unpack_ms"], 1e-9) / 1e6,
                    pack_avg_launch_us=st["pack_ms"] * 1e3 / max(st["timed_pack_launches"], 1),
                    unpack_avg_launch_us=st["unpack_ms"] * 1e3 / max(st["timed_unpack_launches"], 1),
                    pack_bytes_per_launch=st["timed_pack_bytes"] / max(st["timed_pack_launches"], 1),
                    pack_hbm_bytes_per_launch=st["timed_pack_hbm_bytes"] / max(st["timed_pack_launches"], 1),
                    unpack_bytes_per_launch=st["timed_unpack_bytes"] / max(st["timed_unpack_launches"], 1),
                    wire_segments_per_step=st["wire_segments"] / n,
                    wire_ratio=(st["wire_bytes"] / st["wire_raw_bytes"]) if st["wire_raw_bytes"] else None,
                    wire_fallbacks=st["wire_fallbacks"],
                    pack_launches_per_step=st["timed_pack_launches"] / n,
                    unpack_launches_per_step=st["timed_unpack_launches"] / n,
                    pack_hbm_bytes_per_step=st["timed_pack_hbm_bytes"] / n,
                    unpack_hbm_bytes_per_step=st["timed_unpack_hbm_bytes"] / n,
                    host_blocks=st["host_blocks"],
                    host_block_ms=st["host_block_ms"],
                    staged_hits=st["staged_hits"],
                    bytes_staged=st["bytes_staged"],
                    prefetch_hits=st["prefetch_hits"],
                    restore_fetches=st["restore_fetches"],
                    host_pinned_peak_bytes=st["host_bytes_peak"],
                    host_pinned_reserved_bytes=st["host_bytes_reserved"],  # the pool only grows within a mode
                    restores_per_step=st["py_ahead_restores"] / n,
                    groups_restored_ahead_per_step=st["py_ahead_restored"] / n,
                    groups_offered_ahead_per_step=st["py_ahead_offered"] / n,
                    ahead_not_resident_per_step=st["ahead_not_resident"] / n,
                    ahead_in_flight_per_step=st["ahead_in_flight"] / n,
                )
                engine.trim()
                left = engine.stats()
                # what the engine still holds once the mode is over: no live group, and the
                # pinned pool given back to the driver but for chunks a live payload still uses
                record.update(groups_live_after=left["groups_live"], py_groups_live_after=left["py_groups_live"],
                              pinned_reserved_after_trim=left["host_bytes_reserved"])
            entry[mode] = record
        none = entry.get("none", {}).get("s_per_it")
        for name in ("engine", "engine_hipdma"):
            eng = entry.get(name)
            if none is None or eng is None or "s_per_it" not in eng:
                continue
            copy_s = eng["d2h_s_per_step"] + eng["h2d_s_per_step"]

            def hidden(exposed):
                return min(1.0, max(0.0, 1.0 - exposed / copy_s)) if copy_s > 0 else None

            eng["exposed_s"] = eng["s_per_it"] - none
            eng["hidden_fraction"] = hidden(eng["exposed_s"])
            pairs = list(zip(times.get(name, []), times.get("none", [])))
            if len(pairs) > 1:
                # per round: the engine's steps against the hooks-off steps timed just before them
                per_round = sorted(e - o for e, o in pairs)
                mid = len(per_round) // 2
                median = per_round[mid] if len(per_round) % 2 else (per_round[mid - 1] + per_round[mid]) / 2
                eng["exposed_s_rounds"] = [e - o for e, o in pairs]
                eng["exposed_s_median"] = median
                eng["exposed_s_range"] = [per_round[0], per_round[-1]]
                eng["hidden_fraction_median"] = hidden(median)
                eng["hidden_fraction_range"] = [hidden(per_round[-1]), hidden(per_round[0])]
        ref = entry.get("reference")
        if none is not None and ref is not None and "s_per_it" in ref:
            ref["exposed_s"] = ref["s_per_it"] - none
        return entry

    cleanups = []
    for regime_name in (r for r in args.regimes if r not in ("M", "K", "Q", "G")):
        try:
            result["regimes"][regime_name] = run_leg(regime_name)
        finally:
            while cleanups:
                cleanups.pop()()
            # a leg's second engines (the HIP-stream transport) go with the leg: their rings and
            # pinned pool are not the next leg's
            while _SECOND_ENGINES:
                _SECOND_ENGINES.popitem()[1].close()
    return result


# what the printed line keeps of a leg's mode and of the microbench; the rest is in --detail
BRIEF_LEG = ("s_per_it", "exposed_s", "exposed_s_median", "hidden_fraction", "hidden_fraction_median", "d2h_gbps",
             "h2d_gbps", "peak_device_bytes", "skipped")
BRIEF_MICRO = ("s_per_iter", "d2h_gbps", "h2d_gbps", "pack_hbm_gbps", "unpack_hbm_gbps", "bitwise_first", "bitwise_last")


def brief(result: dict) -> dict:
    """The part of the record that the printed line carries: readers that keep only the last 8 KB of
    the output must still find the line whole."""

    def pick(figures: dict, keys: tuple[str, ...]) -> dict:
        kept = {k: figures[k] for k in keys if figures.get(k) is not None}
        return {k: float(f"{v:.5g}") if isinstance(v, float) else v for k, v in kept.items()}

    out = {k: result[k] for k in ("link", "parity") if k in result}
    out["regimes"] = {name: {mode: pick(figures, BRIEF_LEG) for mode, figures in leg.items() if isinstance(figures, dict)}
                      for name, leg in result["regimes"].items()}
    if "micro" in result:
        out["micro"] = pick(result["micro"], BRIEF_MICRO)
    if "int8_gemm" in result:
        out["int8_gemm"] = {k: v for k, v in result["int8_gemm"].items() if k.startswith("block_")}
    return out


def write_detail(path: str, record: dict) -> None:
    try:
        os.makedirs(os.path.dirname(path) or ".", exist_ok=True)
        with open(path, "w") as f:
            json.dump(record, f, default=float, indent=1)
    except OSError as e:  # the measurements are printed all the same
        log(f"whole record not written: {e}")


def main() -> int:
    parser = argparse.ArgumentParser(description=__doc__, formatter_class=argparse.RawDescriptionHelpFormatter)
    parser.add_argument("--gpus", type=int, default=1)
    parser.add_argument("--steps", type=int, default=6)
    parser.add_argument("--warmup", type=int, default=2)
    parser.add_argument("--steps-b", type=int, default=5, help="timed steps of the legs other than A")
    parser.add_argument("--warmup-b", type=int, default=2)
    parser.add_argument("--steps-big", type=int, default=2,
                        help="timed steps per round of the config-4/5 and full-parameter legs (2.1-4.7 s steps)")
    parser.add_argument("--rounds-big", type=int, default=4,
                        help="rounds of the interleaved legs (A4, B4, B4R, C5U, C5P): hooks off and engine take "
                             "turns, --steps-big steps each; the reference hooks time one round")
    parser.add_argument("--warmup-big", type=int, default=1)
    parser.add_argument("--b4-layers", type=int, default=24,
                        help="blocks of the B4 leg (config 4 not checkpointed): its coded saves fit the pinned cap")
    parser.add_argument("--b4-ref-layers", type=int, default=6,
                        help="blocks of the B4R leg, where the reference hooks' per-save pins fit the cap too")
    parser.add_argument("--regimes", default="M,K,Q,A,B,BR,AH,A4,B4,B4R,C5U,C5P",
                        help="M = config-2 block microbench, K = 28 MiB gathers/scatters back to back and after "
                        "other kernels (a GEMM with a large output, a fill, a read), Q = config-5 int8 GEMMs "
                        "(HIP vs eager), "
                        "A/B = config-3 steps (checkpointed / not), BR = regime B on --ref-layers blocks (none, "
                        "engine and the reference hooks, which fit the pinned-memory cap there), AH = regime A "
                        "with --host-work-ms of host work per step (none, engine on SDMA, engine on HIP "
                        "streams), BK = regime B keeping the last "
                        "--keep-last-blocks blocks' saves resident, G = host gradient accumulation "
                        "(full-parameter config-3 dims, 2 micro-batches: device / engine / reference stash), "
                        "A4 = config 4 (2048^2, regime A), B4/B4R = config 4 not checkpointed on --b4-layers / "
                        "--b4-ref-layers blocks (the host link sets the pace), "
                        "C5U/C5P = config 5 unpacked / packed (regime A), "
                        "S5 = config 5 packed with every block streamed from pinned host masters, "
                        "F3/F3S = full-parameter training at config-3 dims, resident / every block on the trainable ring")
    parser.add_argument("--micro-iters", type=int, default=1000)
    parser.add_argument("--ref-layers", type=int, default=16,
                        help="blocks of the BR leg and of regime B's reference parity: the reference hooks pin one "
                             "tensor per save, and 40 blocks of regime B exceed the host's pinned-memory cap")
    parser.add_argument("--host-work-ms", type=float, default=100.0,
                        help="AH leg: host work after every step, which overlaps the GPU only when the host is ahead")
    parser.add_argument("--micro-warmup", type=int, default=3)
    parser.add_argument("--modes", default="none,engine,reference")
    parser.add_argument("--layers", type=int, default=CONFIG3["num_layers"])
    parser.add_argument("--no-parity", action="store_true")
    parser.add_argument("--stage-slots", type=int, default=4)
    parser.add_argument("--restore-slots", type=int, default=16)
    parser.add_argument("--stage-slots-max", type=int, default=8,
                        help="staging ring growth cap (0: fixed ring)")
    parser.add_argument("--restore-slots-max", type=int, default=32,
                        help="restore ring growth cap (0: fixed ring)")
    parser.add_argument("--restore-small-slots", type=int, default=24,
                        help="quarter-size restore slots for checkpointed blocks' inputs (0: none, and every "
                             "restore slot allocated up front)")
    parser.add_argument("--prefetch-depth", type=int, default=16,
                        help="groups the engine prefetches ahead of backward after each restored group")
    parser.add_argument("--slot-mib", type=int, default=128)
    parser.add_argument("--restore-ahead-mib", type=int, default=None,
                        help="payload MiB of further groups one unpack may restore (default: the engine's)")
    parser.add_argument("--no-staged-restore", action="store_true")
    parser.add_argument("--d2h-engine", type=lambda v: int(v, 0), default=0,
                        help="SDMA engine bits for D2H (0: two engines, copies split in halves)")
    parser.add_argument("--h2d-engine", type=lambda v: int(v, 0), default=0,
                        help="SDMA engine bits for H2D (0: one engine, the lowest not used by D2H)")
    parser.add_argument("--no-narrow", action="store_true",
                        help="offload float32 casts of bfloat16 tensors whole instead of as their high halves")
    parser.add_argument("--eager-pack", action="store_true",
                        help="one gather launch per save instead of one per staging segment")
    parser.add_argument("--kernel-copy", action="store_true", help="copy kernel on HIP streams instead of SDMA")
    parser.add_argument("--pack-cached-load", action="store_true",
                        help="pack reads saves with ordinary loads instead of non-temporal ones")
    parser.add_argument("--unpack-cached-load", action="store_true",
                        help="unpack reads payloads with ordinary loads instead of non-temporal ones")
    parser.add_argument("--unpack-cached-store", action="store_true",
                        help="unpack writes restored tensors with ordinary stores instead of streaming ones")
    parser.add_argument("--wire-coding", default="auto", choices=("off", "on", "auto"),
                        help="lossless coding of staging segments before D2H (SDMA link) in the step legs: off, on, "
                             "or auto (only while two staging slots of D2H bytes are queued)")
    parser.add_argument("--micro-wire-coding", default="off", choices=("off", "on", "auto"),
                        help="wire coding in the block microbench, which measures the pack and unpack kernels "
                             "(off by default: it refills its sources with random bits, which do not code)")
    parser.add_argument("--link", default="sdma", choices=("sdma", "hipdma"),
                        help="host-link transport: SDMA through HSA with host-side ordering, or the same DMA "
                             "copies on HIP streams ordered by hipStreamWaitEvent")
    parser.add_argument("--cpu-threads", type=int, default=16)
    parser.add_argument("--gradacc-threads", type=int, default=12, help="host threads of the G leg's accumulator")
    parser.add_argument("--keep-last-blocks", type=int, default=16,
                        help="BK leg: the engine keeps the saves of the last N blocks on the device")
    parser.add_argument("--int8-backend", default="auto", choices=("auto", "eager", "hip"),
                        help="backend of config 5's int8 bases (auto = the HIP MFMA kernels when supported)")
    parser.add_argument("--cpu-budget", type=float, default=15.0)
    parser.add_argument("--detail", default=str(ROOT / "build" / "bench_detail.json"),
                        help="file for the whole record, every counter of every leg ('': not written)")
    args = parser.parse_args()
    world = int(os.environ.get("WORLD_SIZE", "1"))
    if args.gpus != 1 or world != 1:
        print(
            "bench.py measures one GPU: activation offload is per-GPU host-link traffic with no "
            "cross-GPU exchange, and this build runs on a single MI355X. Use --gpus 1.",
            file=sys.stderr,
        )
        return 2
    args.regimes = [r.strip().upper() for r in args.regimes.split(",") if r.strip()]
    args.modes = [m.strip() for m in args.modes.split(",") if m.strip()]

    import torch

    if not torch.cuda.is_available():
        print("bench.py needs a HIP device", file=sys.stderr)
        return 2
    result = run(args)
    regimes = result["regimes"]
    headline = regimes.get("A") or next(iter(regimes.values()), {})
    eng = headline.get("engine", {})
    # cpu baseline: oracle restatement, bounded sample (one regime-B block's saves if recorded)
    sample = None
    for r in ("B", "A"):
        if r in regimes and "cpu_sample" in regimes[r]:
            sample = regimes[r].pop("cpu_sample")
            break
    cpu = None
    if sample is not None:
        log("cpu baseline (oracle reference hooks, host memory)")
        threads = min(args.cpu_threads, os.cpu_count() or 1)
        base = cpu_baseline(sample, threads, args.cpu_budget)
        cpu = {
            "value": round(base["gbps"], 3),
            "unit": "GB/s",
            "cores": threads,
            "kind": "port",
            "sample": f"reference hook pack+unpack (dense copy_, empty_strided+copy_) of the regime-B saves of one "
            f"40-block 1024^2 step forward ({base['payload_bytes'] / 1e9:.2f} GB unique), {base['iters']} iteration(s) "
            f"in {base['seconds']:.1f} s on host memory",
            "host_cores": os.cpu_count(),
        }
    for r in regimes.values():
        r.pop("cpu_sample", None)
    # dominant engine kernel of the headline regime
    # Dominant engine kernel: the pack kernel (mo_pack_kernel). Measured on the config-2 block
    # microbench when it ran (one regime-B block's saves, the bulk of all offload traffic),
    # else on the headline regime's steps. achieved = device-memory bytes per launch (read the
    # source, write the staging slot: 2 x payload, or 3 x for a narrowed float32 piece, which
    # reads 4 bytes per 2 it writes) / average dispatch duration (HIP events of the launch).
    src = result.get("micro") or eng
    pack_bound = {
        "bound": "hbm",
        "kernel": "mo_pack_kernel",
        "workload": "config-2 block microbench" if "micro" in result else "headline regime steps",
        "achieved": round(src.get("pack_hbm_gbps", 0.0), 1),
        "peak": HBM_PEAK_GBPS,
        "unit": "GB/s",
        "frac": round(src.get("pack_hbm_gbps", 0.0) / HBM_PEAK_GBPS, 4),
        "traffic": profiled_traffic() if "micro" in result else None,
        "traffic_source": PACK_PROFILE.name if "micro" in result else None,
        "algorithmic_bytes_per_launch": src.get("pack_hbm_bytes_per_launch", 0.0),
        "avg_launch_us": src.get("pack_avg_launch_us"),
    }
    line = {
        "metric": "DiT step s/it @1024² w/ act-offload; D2H/H2D GB/s; % copy hidden",
        "value": round(eng.get("s_per_it", float("nan")), 5),
        "unit": "s/it",
        "n_gpus": 1,
        "steps": args.steps,
        "warmup": args.warmup,
        "ms_per_step": round(eng.get("s_per_it", float("nan")) * 1e3, 3),
        "higher_is_better": False,
        "scaling": "weak",
        "vs_baseline": None,
        "dtype": "bf16",
        "data": "synthetic: random-init weights N(0,0.02), LoRA B~N(0,0.03), latents/text N(0,1)",
        "config": {
            "workload": "BASELINE config 3: 5B-shaped MOSS DiT LoRA step, 1024^2, all blocks offloaded, "
            "regime A (every block checkpointed, reference default) as value; regime B reported alongside",
            "layers": args.layers, "hidden": 3072, "heads": "24x128", "mlp": 12288, "lora_rank": LORA_RANK,
            "batch": 1, "image_tokens": 4096, "text_tokens": TEXT_TOKENS, "parallelism": "none (1 GPU)",
        },
        "d2h_gbps": round(eng.get("d2h_gbps", 0.0), 2),
        "h2d_gbps": round(eng.get("h2d_gbps", 0.0), 2),
        "copy_hidden_fraction": eng.get("hidden_fraction"),
        "link_frac_of_spec": round(min(eng.get("d2h_gbps", 0.0), eng.get("h2d_gbps", 0.0)) / LINK_SPEC_GBPS, 4),
        "roofline": pack_bound,
        "int8_gemm_roofline": result.get("int8_gemm", {}).get("roofline"),
        "cpu_baseline": cpu,
        "detail": brief(result),
    }
    if args.detail:
        write_detail(args.detail, {**line, "detail": result})
    print(json.dumps(line, default=float), flush=True)
    return 0


if __name__ == "__main__":
    sys.exit(main())
