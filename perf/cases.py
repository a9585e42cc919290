"""The workloads whose speed this framework is judged by, as plain cases.

A pass is one session, the way a program uses the framework: the streams start from reset, a run
of events goes through the public calls one step at a time (or, for a replay, as one preloaded
trace), and the scores (for a replay the carried state) come back. A session is longer than the
window, so the ring fills, wraps and evicts within every pass, and a pass repeats exactly.

Kinds:
  step      Runtime (FUSED backend, one workgroup per compute unit), Runtime.step per event
  replay    the same runtime rebuilding a stream's state from its history: Runtime.device_trace
            over the whole history, then Runtime.snapshot
  batch     BatchRuntime, independent streams in phase kernels, BatchRuntime.step per event
  resident  BatchRuntime(resident=True), the small-batch form
With `save`, the session ends with a snapshot of its last stream, as when a stream is closed and
kept; the state comes back with the scores.

Weights are random with standard deviation 1 / sqrt(inputs), so that logits, gates and residuals
have the size they have in a trained network; events are N(0, 1).
"""
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path('streaming-transformer_amd').resolve()))

from streamtx import Backend, BatchRuntime, ModelConfig, Runtime, RuntimeOptions, WeightStorage  # noqa: E402
from streamtx.model import round_bf16, tensor_names  # noqa: E402

DEVICE = 'cuda' if torch.cuda.is_available() else 'cpu'


def _case(name, kind, weights, config, streams, steps, save=False):
    layers, width, heads, ffn, window, features = config
    return dict(name=name, kind=kind, weights=weights, layers=layers, width=width, heads=heads, ffn=ffn,
                window=window, features=features, streams=streams, steps=steps, save=save)


SMALL = (4, 256, 4, 1024, 64, 256)
MAIN = (8, 512, 8, 2048, 128, 512)
LARGE = (12, 1024, 16, 4096, 512, 1024)


def listed():
    return [
        # The smallest published checkpoint, one event at a time: launch and exchange latency only.
        _case('step-tiny-fp32', 'step', 'fp32', (1, 64, 4, 128, 64, 32), 1, 80, True),
        # The ordinary single stream: a per-event scoring service on 16-bit weights and K/V.
        _case('step-main-mixed', 'step', 'mixed', MAIN, 1, 160),
        # The large single stream, bound by streaming its FP32 weights.
        _case('step-large-fp32', 'step', 'fp32', LARGE, 1, 576),
        # Recovery of a stream after a restart: its history replayed on the device, state read back.
        _case('replay-main-fp32', 'replay', 'fp32', MAIN, 1, 512),
        # A few low-latency streams sharing one GPU, one launch per step.
        _case('resident-main-bf16w-4', 'resident', 'bf16w', MAIN, 4, 160),
        # A small batch of streams: one MFMA tile, a chain of short kernels.
        _case('batch-main-bf16w-16', 'batch', 'bf16w', MAIN, 16, 160),
        # A few streams with a long history each: attention over the ring dominates.
        _case('batch-longwindow-bf16w-4', 'batch', 'bf16w', (8, 512, 8, 2048, 1024, 512), 4, 1088),
        # An odd batch of an odd model: padded events, rows and batch tiles.
        _case('batch-odd-fp32-37', 'batch', 'fp32', (3, 384, 8, 1000, 200, 29), 37, 232, True),
        # A small FP32 model serving many streams.
        _case('batch-small-fp32-100', 'batch', 'fp32', SMALL, 100, 96, True),
        # The reference's FP16 mode at a medium batch.
        _case('batch-main-mixed-64', 'batch', 'mixed', MAIN, 64, 160),
        # The fullest batch: throughput serving.
        _case('batch-main-bf16w-256', 'batch', 'bf16w', MAIN, 256, 160),
        # The large model serving a batch with its long window.
        _case('batch-large-bf16w-32', 'batch', 'bf16w', LARGE, 32, 544),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(['step', 'step', 'replay', 'resident', 'batch', 'batch', 'batch', 'batch'])
    weights = rng.choice(['fp32', 'mixed', 'bf16w'])
    dim = rng.choice([16, 32, 48, 64, 64, 128])
    heads = max(1, min(1024 // dim, _log_int(rng, 64, 1024) // dim))
    width = dim * heads
    ffn = min(4096, 8 * max(8, int(width * rng.uniform(1.5, 4.0)) // 8))
    streams = {'step': 1, 'replay': 1, 'resident': _log_int(rng, 1, 16), 'batch': _log_int(rng, 1, 256)}[kind]
    case = _case('', kind, weights, (_log_int(rng, 1, 12), width, heads, ffn, _log_int(rng, 16, 1024),
                                     _log_int(rng, 16, 1024)), streams, 0,
                 kind != 'replay' and rng.random() < 0.3)
    del case['name']
    # A session a little longer than the window, shortened (then with fewer streams) where it
    # would cost more than the largest listed case.
    case['steps'] = max(48, case['window'] + case['window'] // 8 + rng.randrange(8))
    most = max(_cost(c) for c in listed())
    while _cost(case) > most:
        if case['steps'] > 64:
            case['steps'] = max(64, case['steps'] * 3 // 4)
        elif case['streams'] > 1:
            case['streams'] = max(1, case['streams'] * 3 // 4)
        else:
            case['layers'] -= 1
    return case


def _cost(case):
    w = work(case)
    return w['bytes'] + w['flops'] / 50


def _config(case):
    return ModelConfig(case['layers'], case['width'], case['heads'], case['ffn'], case['window'], case['features'])


def _inputs(case, seed):
    """(tensors, events): the checkpoint's tensors as float32 arrays (FP16 values in mixed mode)
    and the session's events [steps, streams, features], made from the seed alone."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(1000003 * (seed + 1))
    tensors = {}
    for name, shape in tensor_names(_config(case)):
        t = torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32)
        # Matrices as the reference initialises them; norm gains around one.
        t = t / math.sqrt(shape[1]) if len(shape) == 2 else 1.0 + 0.1 * t
        if case['weights'] == 'mixed':
            t = t.half().float()
        tensors[name] = t.cpu().numpy()
    events = torch.randn((case['steps'], case['streams'], case['features']), generator=gen, device=DEVICE,
                         dtype=torch.float32).cpu().numpy()
    return tensors, events


class _State:
    """A user's handle and events. The handle closes with the state."""

    def __init__(self, case, seed):
        tensors, self.events = _inputs(case, seed)
        self.kind, self.save, self.last = case['kind'], case['save'], case['streams'] - 1
        model = (_config(case), tensors, case['weights'] == 'mixed')
        storage = WeightStorage.BF16 if case['weights'] == 'bf16w' else WeightStorage.AS_MODEL
        if self.kind in ('step', 'replay'):
            self.runtime = Runtime(model, RuntimeOptions(backend=Backend.FUSED, blocks=0, weight_dtype=storage))
            self.events = self.events[:, 0]
        else:
            self.runtime = BatchRuntime(model, case['streams'], storage, resident=self.kind == 'resident')


def prepare(case, seed):
    return _State(case, seed)


def run(state):
    rt = state.runtime
    if state.kind == 'replay':
        rt.device_trace(state.events)  # resets the stream, then runs the whole history
        return _kept(rt.snapshot())
    rt.reset()
    out = {'scores': np.array([rt.step(event) for event in state.events], dtype=np.float32)}
    if state.save:
        out.update(_kept(rt.snapshot() if state.kind == 'step' else rt.snapshot(state.last)))
    return out


def _kept(snapshot):
    return dict(zip(('position', 'keys', 'values', 'hidden'), snapshot))


def work(case):
    """Per step: the weights once, each stream's valid K/V rows read and one row written, the
    events in and the scores out; with a saved state also that. Multiply-adds of the
    projections and of attention."""
    c = case
    d, f, n = c['width'], c['ffn'], c['layers']
    wb = 4 if c['weights'] == 'fp32' else 2
    kvb = 2 if c['weights'] == 'mixed' else 4
    params = c['features'] * d + n * (4 * d * d + 3 * d * f + 2 * d) + 2 * d
    rows = sum(min(t + 1, c['window']) for t in range(c['steps']))
    read = c['steps'] * wb * params + c['streams'] * rows * 2 * n * d * kvb
    write = c['steps'] * c['streams'] * (2 * n * d * kvb + 4)
    if c['kind'] == 'replay' or c['save']:
        write += 2 * n * d * c['window'] * 4 + n * d * 4
    events = c['steps'] * c['streams'] * c['features'] * 4
    flops = c['streams'] * (2 * params * c['steps'] + 4 * n * d * rows)
    return {'bytes': read + write + events, 'flops': flops}


def tolerance(case):
    # About four times the measured distance from float64: up to 2.8e-6 in FP32 arithmetic
    # (through 12 layers), 1.7e-3 in mixed mode, which rounds every layer's values to FP16.
    if case['weights'] == 'mixed':
        return {'rel': 6e-3}
    return {'rel': 1e-5}


def exact(case, seed):
    """The session as one causal windowed pass in float64 (no FP16 rounding inside the step)."""
    c = _config(case)
    tensors, events = _inputs(case, seed)
    if case['weights'] == 'bf16w':
        tensors = {k: round_bf16(v) for k, v in tensors.items()}
    w = {k: torch.from_numpy(v).to(DEVICE, torch.float64) for k, v in tensors.items()}
    steps, streams = events.shape[:2]
    ev = torch.from_numpy(events).to(DEVICE, torch.float64).transpose(0, 1).contiguous()  # [B, T, f]
    t = torch.arange(steps, device=DEVICE)
    seen = (t[None, :] <= t[:, None]) & (t[None, :] > t[:, None] - c.window)
    freq = 10000.0 ** (-torch.arange(0, c.dim, 2, device=DEVICE, dtype=torch.float64) / c.dim)
    angle = t.to(torch.float64)[:, None] * freq[None, :]
    co, si = torch.cos(angle), torch.sin(angle)

    def norm(x, g):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + c.epsilon) * g

    def heads(x):
        return x.reshape(streams, steps, c.heads, c.dim).transpose(1, 2)  # [B, H, T, dh]

    def rotate(x):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack((a * co - b * si, a * si + b * co), -1).flatten(-2)

    x = ev @ w['input'].T
    state_k, state_v, state_h = [], [], []
    for n in range(c.layers):
        p = f'layers.{n}.'
        z = norm(x, w[p + 'norm1'])
        q, k, v = rotate(heads(z @ w[p + 'q'].T)), rotate(heads(z @ w[p + 'k'].T)), heads(z @ w[p + 'v'].T)
        attn = torch.empty_like(q)
        for b in range(streams):  # one stream's logits at a time
            for h in range(c.heads):
                logits = (q[b, h] @ k[b, h].T) / math.sqrt(c.dim)
                attn[b, h] = torch.softmax(logits.masked_fill(~seen, -math.inf), -1) @ v[b, h]
        x = x + attn.transpose(1, 2).reshape(streams, steps, c.width) @ w[p + 'out'].T
        z = norm(x, w[p + 'norm2'])
        x = x + (torch.nn.functional.silu(z @ w[p + 'gate'].T) * (z @ w[p + 'up'].T)) @ w[p + 'down'].T
        state_k.append(k[-1])
        state_v.append(v[-1])
        state_h.append(x[-1, -1])
    out = {}
    if case['kind'] != 'replay':
        scores = (norm(x, w['final_norm']) @ w['score'][0]).T.contiguous().cpu().numpy()  # [T, B]
        out['scores'] = scores[:, 0] if case['kind'] == 'step' else scores
    if case['kind'] == 'replay' or case['save']:
        def ring(rows):  # position t lives in slot t mod window
            out = torch.zeros((c.layers, c.heads, c.window, c.dim), dtype=torch.float64, device=DEVICE)
            kept = t[max(0, steps - c.window):]
            out[:, :, kept % c.window] = torch.stack(rows)[:, :, kept]
            return out.cpu().numpy()
        out.update(_kept((None, ring(state_k), ring(state_v), torch.stack(state_h).cpu().numpy())))
    return out
