"""What is timed: the work a program has this codec do, through its public entry points.

Each case is a dict of plain values; ``kind`` picks the path:

* ``forward``        encode -> decode round trip of a batch of clips (``MimiModel.forward``);
* ``decode``         codes -> waveform (``MimiModel.decode``);
* ``stream_encode``  a live capture: chunks of whole code frames through ``MimiModel.encode`` with its
                     padding and key/value caches;
* ``stream_decode``  live playback: code frames through ``MimiModel.decode`` with its key/value cache;
* ``transformer``    one eight-layer transformer (``MimiRuntime.transformer``), captured in a hipGraph
                     as the model captures it;
* ``conv_down``      one strided encoder convolution (``torch.ops.fast_mimi_amd.conv1d``);
* ``conv_up``        one transposed decoder convolution (``...conv_transpose1d``);
* ``resblock``       one SEANet residual block (``...resblock``);
* ``quantize``       the residual vector quantizer on encoder outputs (``MimiRuntime.quantize``).

The model is the package's default configuration with its seeded weights (LayerScale and LayerNorm
moved away from their initial constants); a process builds it once, as a server does, and the seed of
a case makes the inputs only.
"""

from __future__ import annotations

import functools
import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "fast-mimi_amd"))

from fast_mimi_amd import MimiKVCache, MimiModel  # noqa: E402
from fast_mimi_amd import _native as nat  # noqa: E402
from fast_mimi_amd.flops import layer_table, roundtrip_flops  # noqa: E402

DEV = "cuda:0"
RATIOS = (8, 6, 5, 4)  # decoder strides; the encoder walks them backwards
FRAME = 1920           # samples per code frame
DIM, ENTRIES, VQ = 512, 2048, 256


# ----------------------------------------------------------------- the cases
def listed():
    return [
        # Live microphone to codes in 80 ms steps, the smallest unit the codec can send.
        {"name": "stream_encode_b1_80ms", "kind": "stream_encode", "batch": 1, "frames": 1, "chunks": 4, "nq": 8},
        # Live playback of the same stream.
        {"name": "stream_decode_b1_80ms", "kind": "stream_decode", "batch": 1, "frames": 1, "chunks": 4, "nq": 8},
        # A short spoken reply (13 frames, about a second) from a speech model's codes.
        {"name": "decode_b1_1s", "kind": "decode", "batch": 1, "frames": 13, "nq": 8},
        # The round trip of one 10 s clip, the benchmark's workload.
        {"name": "forward_b1_10s", "kind": "forward", "batch": 1, "samples": 240_000, "nq": 8},
        # The same for a batch of 16 clips, a quarter of them padded: throughput of a data pipeline.
        {"name": "forward_b16_10s", "kind": "forward", "batch": 16, "samples": 240_000, "nq": 8},
        # The transformer of one 10 s clip (250 rows), where each kernel is short.
        {"name": "transformer_enc_b1_10s", "kind": "transformer", "side": "enc", "batch": 1, "frames": 250},
        # The transformer of one 100 s clip (2500 rows), ten attention windows long.
        {"name": "transformer_dec_b1_100s", "kind": "transformer", "side": "dec", "batch": 1, "frames": 2500},
        # Encoder convolution 128 -> 256, stride 5, on a clip whose length is not a multiple of the stride.
        {"name": "conv_down5_b1_10s", "kind": "conv_down", "stage": 1, "batch": 1, "length": 59_997},
        # Decoder upsampling 1024 -> 512, stride 8, of one clip: few rows, the widest weights.
        {"name": "conv_up8_b1_10s", "kind": "conv_up", "stage": 0, "batch": 1, "length": 250},
        # Decoder upsampling 128 -> 64, stride 4, of 16 clips: the largest layer of a batch.
        {"name": "conv_up4_b16_10s", "kind": "conv_up", "stage": 3, "batch": 16, "length": 60_000},
        # Decoder residual block at 128 channels of one clip.
        {"name": "resblock128_dec_b1_10s", "kind": "resblock", "side": "dec", "stage": 2, "batch": 1,
         "length": 60_000},
        # All 32 codebooks for 64 clips of 10 s: dataset tokenisation at the highest bitrate.
        {"name": "quantize_b64_10s_nq32", "kind": "quantize", "batch": 64, "frames": 125, "nq": 32},
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choice(["stream_encode", "stream_decode", "decode", "forward", "forward", "transformer",
                       "conv_down", "conv_up", "resblock", "quantize"])
    nq = rng.choice([1, 4, 8, 8, 16, 32])
    case = {"kind": kind, "batch": _log(rng, 1, 16)}
    if kind in ("stream_encode", "stream_decode"):
        case.update(batch=_log(rng, 1, 8), frames=rng.randint(1, 4), chunks=rng.randint(2, 5), nq=max(nq, 2))
    elif kind == "decode":
        case.update(frames=_log(rng, 2, 2000 // case["batch"]), nq=nq)
    elif kind == "forward":
        case.update(samples=_log(rng, 4_000, 3_600_000 // case["batch"]), nq=nq)
    elif kind == "transformer":
        case.update(side=rng.choice(["enc", "dec"]), frames=_log(rng, 8, 4000 // case["batch"]))
    elif kind == "conv_down":
        stage = rng.randrange(4)
        case.update(stage=stage, length=_log(rng, 60, 3_600_000 // case["batch"] // (1, 4, 20, 120)[stage]))
    elif kind == "conv_up":
        stage = rng.randrange(4)
        case.update(stage=stage, length=_log(rng, 10, 3_600_000 // case["batch"] // (960, 120, 20, 4)[stage]))
    elif kind == "resblock":
        stage = rng.randrange(1, 3)
        case.update(side=rng.choice(["enc", "dec"]), stage=stage,
                    length=_log(rng, 100, 3_600_000 // case["batch"] // (120, 20, 4)[stage]))
    else:
        case.update(batch=_log(rng, 1, 64), nq=max(nq, 2))
        case.update(frames=_log(rng, 1, 8000 // case["batch"]))
    return case


# ------------------------------------------------------- the model and inputs
@functools.lru_cache(maxsize=None)
def _model():
    model = MimiModel()
    g = torch.Generator().manual_seed(20)
    state = model.state_dict()
    for name, t in state.items():
        # A trained checkpoint's LayerScale and LayerNorm are not their initial constants.
        if name.endswith("layer_scale.scale"):
            state[name] = 0.05 + 0.35 * torch.rand(t.shape, generator=g)
        elif name.endswith("layernorm.weight"):
            state[name] = 1.0 + 0.1 * torch.randn(t.shape, generator=g)
        elif name.endswith("layernorm.bias"):
            state[name] = 0.1 * torch.randn(t.shape, generator=g)
    model.load_state_dict(state)
    return model.to(DEV)


def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _audio(batch, samples, seed):
    """Three tones and noise per clip, peaks 0.1-0.9; in a batch the last quarter of the clips is padded
    with zeros from 60% on."""
    g = _generator(seed)
    t = torch.arange(samples, device=DEV, dtype=torch.float64) / 24_000
    u = torch.rand((batch, 7), generator=g, device=DEV, dtype=torch.float64)
    freq = 80.0 * 50.0 ** u[:, :3]
    wave = torch.sin(2 * math.pi * (freq[:, :, None] * t + u[:, 3:6, None])).sum(1)
    wave = wave + 0.12 * torch.randn((batch, samples), generator=g, device=DEV, dtype=torch.float64)
    wave = wave / wave.abs().amax(1, keepdim=True) * (0.1 + 0.8 * u[:, 6:])
    if batch >= 4:
        wave[batch - batch // 4:, int(0.6 * samples):] = 0
    return wave.float()[:, None].contiguous()


def _codes(batch, nq, frames, seed):
    return torch.randint(0, ENTRIES, (batch, nq, frames), generator=_generator(seed), device=DEV)


def _rows(batch, length, channels, seed, elu=False):
    x = torch.randn((batch, length, channels), generator=_generator(seed), device=DEV)
    return F.elu(x) if elu else x


def _inputs(case, seed):
    kind, b = case["kind"], case["batch"]
    if kind == "forward":
        return _audio(b, case["samples"], seed)
    if kind == "stream_encode":
        return _audio(b, case["frames"] * case["chunks"] * FRAME, seed)
    if kind == "decode":
        return _codes(b, case["nq"], case["frames"], seed)
    if kind == "stream_decode":
        return _codes(b, case["nq"], case["frames"] * case["chunks"], seed)
    if kind == "transformer":
        return _rows(b, case["frames"], DIM, seed)
    if kind == "quantize":
        return _rows(b, case["frames"], DIM, seed)
    # Convolutions read what an ELU left; a residual block reads a convolution's output.
    return _rows(b, case["length"], _channels(case), seed, elu=kind != "resblock")


def _channels(case):
    """Input channels of a conv_down / conv_up / resblock case."""
    stage = case["stage"]
    if case["kind"] == "conv_down":
        return 64 << stage
    if case["kind"] == "conv_up":
        return 1024 >> stage
    return 64 << stage if case["side"] == "enc" else 512 >> stage


def prepare(case, seed):
    model = _model()
    rt = model.runtime()
    x = _inputs(case, seed)
    kind, b = case["kind"], case["batch"]
    state = {"case": case, "model": model, "rt": rt, "x": x}
    if kind == "forward":
        state["mask"] = torch.ones_like(x, dtype=torch.bool)
    elif kind in ("stream_encode", "stream_decode"):
        step = case["frames"] * (FRAME if kind == "stream_encode" else 1)
        state["x"] = [c.contiguous() for c in x.split(step, dim=-1)]
    elif kind == "transformer":
        layers = rt.enc_tf if case["side"] == "enc" else rt.dec_tf
        rt.prepare(case["frames"])

        # The transformer works in place, so the call gets a copy of its input.
        def call():
            return rt.transformer(x.clone(), b, case["frames"], layers)

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.inference_mode():
            with torch.cuda.stream(side):
                call()
            torch.cuda.current_stream().wait_stream(side)
            state["graph"] = torch.cuda.CUDAGraph()
            with torch.cuda.graph(state["graph"]):
                state["out"] = call()
    elif kind == "conv_down":
        state["layer"] = rt.enc_stages[case["stage"]][1]
    elif kind == "conv_up":
        state["layer"] = rt.dec_stages[case["stage"]][0]
    elif kind == "resblock":
        stage = case["stage"]
        state["layer"] = rt.enc_stages[stage][0] if case["side"] == "enc" else rt.dec_stages[stage][1]
    return state


@torch.inference_mode()
def run(state):
    case, model, rt, x = state["case"], state["model"], state["rt"], state["x"]
    kind, b = case["kind"], case["batch"]
    if kind == "forward":
        out = model(x, state["mask"], num_quantizers=case["nq"])
        return {"codes": out.audio_codes, "audio": out.audio_values}
    if kind == "decode":
        return {"audio": model.decode(x).audio_values}
    if kind == "stream_encode":
        kv = pad = None
        codes = []
        for chunk in x:
            out = model.encode(chunk, num_quantizers=case["nq"], encoder_past_key_values=kv,
                               padding_cache=pad, use_streaming=True)
            kv, pad = out.encoder_past_key_values, out.padding_cache
            codes.append(out.audio_codes)
        return {"codes": codes, "keys": list(kv.key_cache), "values": list(kv.value_cache)}
    if kind == "stream_decode":
        kv = MimiKVCache(model.config.num_hidden_layers, model.config.sliding_window)
        audio = [model.decode(chunk, decoder_past_key_values=kv).audio_values for chunk in x]
        return {"audio": audio, "keys": list(kv.key_cache), "values": list(kv.value_cache)}
    if kind == "transformer":
        state["graph"].replay()
        return {"h": state["out"]}
    if kind == "quantize":
        return {"codes": rt.quantize(x, b, case["frames"], case["nq"])}
    ops, length = torch.ops.fast_mimi_amd, case["length"]
    ws = rt.workspace
    if kind == "conv_down":
        lay = state["layer"]
        rows = -(-length // lay.stride)
        y = torch.empty((b, rows, lay.c_out), device=x.device)
        ops.conv1d(x, b, length, lay.c_in, lay.w, lay.b, lay.c_out, lay.k, lay.stride, 0, lay.flags, None,
                   y, rows, ws, ws.numel() * 4)
        return {"y": y}
    if kind == "conv_up":
        lay = state["layer"]
        y = torch.empty((b, length * lay.stride, lay.c_out), device=x.device)
        ops.conv_transpose1d(x, b, length, lay.c_in, lay.w, lay.b, lay.c_out, lay.k, lay.stride, lay.flags,
                             None, y, ws, ws.numel() * 4)
        return {"y": y}
    c1, c2 = state["layer"]
    y = torch.empty_like(x)
    flags = 1 | (c1.flags & c2.flags) | (nat.ACT_EXP if case["side"] == "dec" else 0)
    ops.resblock(x, b, length, c2.c_out, c1.w, c1.b, c2.w, c2.b, flags, y)
    return {"y": y}


# --------------------------------------------------- what cannot be done without
def _tf_work(batch, frames, layers=8):
    rows = batch * frames
    window = sum(min(t + 1, 250) for t in range(frames)) * batch
    weights = DIM * (3 * DIM + DIM + 2 * 2048)
    return {"bytes": 4 * (layers * weights + 2 * rows * DIM),
            "flops": layers * (2 * rows * weights + 4 * DIM * window)}


def work(case):
    kind, b = case["kind"], case["batch"]
    config = _model().config
    if kind in ("forward", "decode", "stream_encode", "stream_decode"):
        samples = case["samples"] if kind == "forward" else FRAME * case["frames"] * case.get("chunks", 1)
        nq = case["nq"]
        frames = -(-samples // FRAME)
        rows = layer_table(config, b, samples, nq)
        cut = next(i for i, r in enumerate(rows) if r[0] == "rvq.out")
        encode, decode = sum(r[2] for r in rows[:cut]), sum(r[2] for r in rows[cut:])
        params = 4 * sum(p.numel() for p in _model().parameters()) // 2  # about half on either side
        codes, audio, books = 8 * b * nq * frames, 4 * b * samples, 4 * nq * ENTRIES * VQ
        params *= case.get("chunks", 1)  # each chunk is a call that reads the weights
        if kind == "forward":
            return {"bytes": 2 * params + books + 2 * audio + codes,
                    "flops": roundtrip_flops(config, b, samples, nq)}
        if kind == "stream_encode":
            return {"bytes": params + books + audio + codes, "flops": encode}
        gathered = 4 * VQ * b * nq * frames
        return {"bytes": params + min(books, gathered) + audio + codes, "flops": decode}
    if kind == "transformer":
        return _tf_work(b, case["frames"])
    if kind == "quantize":
        rows, nq = b * case["frames"], case["nq"]
        return {"bytes": 4 * (rows * DIM + DIM * DIM + nq * ENTRIES * VQ) + 8 * rows * nq,
                "flops": 2 * rows * (DIM * DIM + nq * ENTRIES * VQ)}
    c, length = _channels(case), case["length"]
    if kind == "conv_down":
        stride = (4, 5, 6, 8)[case["stage"]]
        rows = -(-length // stride)
        return {"bytes": 4 * (b * length * c + b * rows * 2 * c + 4 * c * c * stride),
                "flops": 2 * b * rows * 2 * c * c * 2 * stride}
    if kind == "conv_up":
        stride = RATIOS[case["stage"]]
        return {"bytes": 4 * (b * length * c + b * length * stride * c // 2 + c * c * stride),
                "flops": 2 * b * length * c * c * stride}
    return {"bytes": 4 * (2 * b * length * c + 2 * c * c), "flops": 2 * b * length * 2 * c * c}


def tolerance(case):
    """About four times what the 32-bit kernels differ from 64 bits by; codes may differ where two entries
    are equally near within that (measured: 1 in 10,000)."""
    kind = case["kind"]
    if kind == "quantize":
        return {"rel": 0.0, "differ": 0.001}
    if kind == "forward":
        # A code at a tie moves its frame's waveform (measured: 0.0126 where one code in 16,000 differs).
        return {"rel": 0.03, "max": 0.99, "differ": 0.001}
    if kind in ("stream_encode", "stream_decode", "decode"):
        return {"rel": 4e-6, "max": 2e-5, "differ": 0.001}
    if kind == "transformer":
        return {"rel": 1e-6, "max": 4e-6}
    return {"rel": 2.4e-6, "max": 2.4e-5}


# ------------------------------------------------------- the same in 64 bits
def _w(name):
    return _model().state_dict()[name].to(DEV).double()


def _conv64(x, prefix, stride=1, replicate=False):
    """Causal convolution of [B, L, C]: one product per tap."""
    w = _w(f"{prefix}.conv.weight")
    co, ci, k = w.shape
    b, length, _ = x.shape
    rows = -(-length // stride)
    left, total = k - stride, (rows - 1) * stride + k
    first, last = x[:, :1], x[:, -1:]
    if not replicate:
        first, last = torch.zeros_like(first), torch.zeros_like(last)
    x = torch.cat([first.expand(-1, left, -1), x, last.expand(-1, max(0, total - left - length), -1)], 1)
    y = 0
    for j in range(k):
        tap = x[:, j:j + (rows - 1) * stride + 1:stride].reshape(b * rows, ci)
        y = y + tap @ w[:, :, j].t().contiguous()
    if f"{prefix}.conv.bias" in _model().state_dict():
        y = y + _w(f"{prefix}.conv.bias")
    return y.view(b, rows, co)


def _convt64(x, prefix, stride):
    w = _w(f"{prefix}.conv.weight")
    ci, co, k = w.shape
    b, length, _ = x.shape
    full = x.new_zeros((b, (length - 1) * stride + k, co))
    for j in range(k):
        tap = x.reshape(-1, ci) @ w[:, :, j].contiguous()
        full[:, j:j + (length - 1) * stride + 1:stride] += tap.view(b, length, co)
    return full[:, :length * stride] + _w(f"{prefix}.conv.bias")


def _upsample64(x):
    """Depthwise transposed convolution, kernel 4, stride 2."""
    w = _w("upsample.conv.weight")[:, 0]  # [C, 4]
    b, length, c = x.shape
    full = x.new_zeros((b, 2 * length + 2, c))
    for j in range(4):
        full[:, j:j + 2 * length - 1:2] += x * w[:, j]
    return full[:, :2 * length]


def _res64(x, prefix):
    return x + _conv64(F.elu(_conv64(F.elu(x), f"{prefix}.block.1")), f"{prefix}.block.3")


def _rope64(x, frames):
    """Rotation by the model's float32 angles; x [B, H, T, 64]."""
    inv = 1.0 / (10_000.0 ** (torch.arange(0, 64, 2, dtype=torch.int64).float() / 64))
    angle = torch.arange(frames).float()[:, None] * inv[None]
    angle = torch.cat((angle, angle), -1).double().to(DEV)
    half = torch.cat((-x[..., 32:], x[..., :32]), -1)
    return x * angle.cos() + half * angle.sin()


def _transformer64(h, prefix, state=None):
    """Eight pre-norm layers on [B, T, 512]; ``state`` collects each layer's last 249 keys and values."""
    b, t, _ = h.shape
    pos = torch.arange(t, device=DEV)
    hidden = (pos[None] > pos[:, None]) | (pos[None] <= pos[:, None] - 250)
    for i in range(8):
        p = f"{prefix}.layers.{i}"

        def norm(x, name):
            return F.layer_norm(x, (DIM,), _w(f"{p}.{name}.weight"), _w(f"{p}.{name}.bias"), 1e-5)

        def lin(x, name):
            return x @ _w(f"{p}.{name}.weight").t().contiguous()

        x = norm(h, "input_layernorm")
        q, k, v = (lin(x, f"self_attn.{n}_proj").view(b, t, 8, 64).transpose(1, 2) for n in "qkv")
        q, k = _rope64(q, t), _rope64(k, t)
        if state is not None:
            for key, x in (("keys", k), ("values", v)):
                state[key].append(x.transpose(1, 2).reshape(b, t, DIM)[:, -249:])
        out = []
        for j in range(b):  # one clip's scores at a time
            s = (q[j] @ k[j].transpose(1, 2).contiguous() / 8.0).masked_fill(hidden, -math.inf)
            out.append((s.softmax(-1) @ v[j].contiguous()).transpose(0, 1).reshape(t, DIM))
        h = h + _w(f"{p}.self_attn_layer_scale.scale") * lin(torch.stack(out), "self_attn.o_proj")
        x = F.gelu(lin(norm(h, "post_attention_layernorm"), "mlp.fc1"))
        h = h + _w(f"{p}.mlp_layer_scale.scale") * lin(x, "mlp.fc2")
    return h


def _codebook(j):
    branch, i = ("semantic", j) if j < 1 else ("acoustic", j - 1)
    p = f"quantizer.{branch}_residual_vector_quantizer.layers.{i}.codebook"
    return _w(f"{p}.embed_sum") / _w(f"{p}.cluster_usage").clamp(min=1e-5)[:, None]


def _branch_proj(branch, which):
    return _w(f"quantizer.{branch}_residual_vector_quantizer.{which}_proj.weight")[:, :, 0].t().contiguous()


def _quantize64(h, nq):
    b, t, _ = h.shape
    rows, codes = h.reshape(b * t, DIM), []
    for branch, books in (("semantic", range(1)), ("acoustic", range(1, nq))):
        r = rows @ _branch_proj(branch, "input")
        for j in books:
            e = _codebook(j)
            codes.append(((e * e).sum(1) - 2 * (r @ e.t().contiguous())).argmin(1))
            r = r - e[codes[-1]]
    return torch.stack(codes, 1).view(b, t, nq).transpose(1, 2).contiguous()


def _encoder64(audio, state=None):
    x = _conv64(audio.double().transpose(1, 2), "encoder.layers.0")
    for i, stride in enumerate(reversed(RATIOS)):
        x = _conv64(F.elu(_res64(x, f"encoder.layers.{1 + 3 * i}")), f"encoder.layers.{3 + 3 * i}", stride)
    x = _conv64(F.elu(x), "encoder.layers.14")
    return _conv64(_transformer64(x, "encoder_transformer", state), "downsample", 2, replicate=True)


def _decoder64(codes, chunk=None, state=None):
    """Chunks share the transformer only: the convolutions see each chunk alone."""
    b, nq, t = codes.shape
    chunk = t if chunk is None else chunk
    q = [sum(_codebook(j)[codes[:, j]] for j in js) if len(js) else None for js in (range(1), range(1, nq))]
    x = sum(v @ _branch_proj(n, "output") for n, v in zip(("semantic", "acoustic"), q) if v is not None)
    x = torch.cat([_upsample64(c) for c in x.split(chunk, 1)], 1)
    x = _transformer64(x, "decoder_transformer", state)
    audio = []
    for x in x.split(2 * chunk, 1):
        x = _conv64(x, "decoder.layers.0")
        for i, stride in enumerate(RATIOS):
            x = _res64(_convt64(F.elu(x), f"decoder.layers.{2 + 3 * i}", stride), f"decoder.layers.{3 + 3 * i}")
        audio.append(_conv64(F.elu(x), "decoder.layers.14").transpose(1, 2).contiguous())
    return audio


@torch.inference_mode()
def exact(case, seed):
    kind = case["kind"]
    x = _inputs(case, seed)
    if kind == "forward":
        codes, audio = [], []
        for clip in x.split(1):
            codes.append(_quantize64(_encoder64(clip), case["nq"]))
            audio.append(_decoder64(codes[-1])[0][..., :case["samples"]])
        return {"codes": torch.cat(codes), "audio": torch.cat(audio)}
    if kind == "decode":
        return {"audio": torch.cat([_decoder64(c)[0] for c in x.split(1)])}
    if kind == "stream_encode":
        state = {"keys": [], "values": []}
        codes = _quantize64(_encoder64(x, state), case["nq"])
        return {"codes": [c.contiguous() for c in codes.split(case["frames"], 2)], **state}
    if kind == "stream_decode":
        state = {"keys": [], "values": []}
        return {"audio": _decoder64(x, case["frames"], state), **state}
    x = x.double()
    if kind == "transformer":
        return {"h": _transformer64(x, "encoder_transformer" if case["side"] == "enc" else "decoder_transformer")}
    if kind == "quantize":
        return {"codes": _quantize64(x, case["nq"])}
    stage = case["stage"]
    if kind == "conv_down":
        return {"y": torch.cat([_conv64(c, f"encoder.layers.{3 + 3 * stage}", (4, 5, 6, 8)[stage])
                                for c in x.split(1)])}
    if kind == "conv_up":
        return {"y": torch.cat([_convt64(c, f"decoder.layers.{2 + 3 * stage}", RATIOS[stage])
                                for c in x.split(1)])}
    prefix = f"encoder.layers.{1 + 3 * stage}" if case["side"] == "enc" else f"decoder.layers.{3 + 3 * stage}"
    return {"y": torch.cat([F.elu(_res64(c, prefix)) for c in x.split(1)])}
