"""The work a program has this library do, as cases that can be timed and compared.

A text-to-speech program holds three engines: the unmasking generator, the
audio tokenizer's decoder (codes to audio) and its encoder (a reference
recording to codes). It generates codes for utterances of half a second to
fifteen seconds, alone, with a cloned voice or as a batch of long text's
chunks; it decodes them, a second at a time while streaming or a minute at
once; and it encodes reference recordings of a few to some twenty seconds.

The generator runs the released dimensions with the library's seeded
synthetic weights. The tokenizer's two halves load a checkpoint of seeded
random float32 weights, as a program loads its own. The engines are built
once per process and kept, as a server keeps them.
"""
import functools
import json
import math
import os
import struct
import tempfile

import numpy as np
import torch

import omnivoice_amd as ov

CODEBOOKS, VOCAB, MASK = 8, 1025, 1024
GENERATOR_SEED = 1234
MOST_ROWS = 3440  # packed rows of the largest listed batch
MOST_FRAMES = 1500


def listed():
    return [
        # An interjection ("Yes, sure."): half a second, launches and latency count.
        dict(name="generate 0.5 s", kind="generate", text=6, reference=0, frames=12, items=1),
        # A short sentence: 2 s of speech.
        dict(name="generate 2 s", kind="generate", text=20, reference=0, frames=50, items=1),
        # An ordinary sentence, the benchmark's headline workload: 10 s of speech.
        dict(name="generate 10 s", kind="generate", text=80, reference=0, frames=250, items=1),
        # 15 s of speech in the voice of a 5 s reference.
        dict(name="generate clone", kind="generate", text=180, reference=125, frames=375,
             items=1),
        # Long text: four 15 s chunks as one batch.
        dict(name="generate chunks", kind="generate", text=110, reference=0, frames=375,
             items=4),
        # One pass of the backbone whose logits the program itself reads.
        dict(name="forward 10 s", kind="forward", text=80, reference=0, frames=250, items=1),
        # Streaming: a second of codes that are on the device, audio that stays there.
        dict(name="decode 1 s", kind="decode", frames=25, device=True),
        # An utterance of 10 s, codes and audio on the host.
        dict(name="decode 10 s", kind="decode", frames=250, device=False),
        # The long text's minute as one signal, on the device.
        dict(name="decode 60 s", kind="decode", frames=1500, device=True),
        # The reference recordings of a cloned voice: the shortest that is of use, an
        # ordinary one, and a long one of a ragged length.
        dict(name="encode 3 s", kind="encode", frames=75),
        dict(name="encode 10 s", kind="encode", frames=250),
        dict(name="encode 21 s", kind="encode", frames=523),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["generate", "generate", "generate", "forward", "decode", "decode",
                       "encode", "encode"])
    if kind == "decode":
        return dict(kind=kind, frames=_log(rng, 10, MOST_FRAMES), device=rng.random() < 0.5)
    if kind == "encode":
        return dict(kind=kind, frames=_log(rng, 25, 523))
    while True:
        case = dict(kind=kind, text=_log(rng, 4, 200),
                    reference=_log(rng, 50, 250) if rng.random() < 0.4 else 0,
                    frames=_log(rng, 12, 400),
                    items=rng.choice([1, 1, 2, 3, 4]) if kind == "generate" else 1)
        if _rows(case) <= MOST_ROWS:
            return case


# ------------------------------------------------------------------ what a pass cannot do without

def _rows(case):
    """Rows of the packed guidance batch: every item's conditional sequence
    (text, reference, target) and its unconditional one (target)."""
    return case["items"] * (case["text"] + case["reference"] + 2 * case["frames"])


def _step_work(case):
    """One pass of the backbone and the heads."""
    c = ov.released_config()
    h, inter, qd, kvd = c["hidden_size"], c["intermediate_size"], 2048, 1024
    layer = h * (qd + 2 * kvd) + qd * h + 3 * h * inter
    rows, targets = _rows(case), 2 * case["items"] * case["frames"]
    cond = case["text"] + case["reference"] + case["frames"]
    pairs = case["items"] * (cond * cond + case["frames"] ** 2)
    heads = CODEBOOKS * VOCAB * h
    flops = 2.0 * c["layers"] * (rows * layer + 2 * pairs * qd) + 2.0 * targets * heads
    return flops, 2.0 * (c["layers"] * layer + heads) + 4.0 * rows * h


def work(case):
    if case["kind"] == "generate":
        flops, bytes_ = _step_work(case)
        steps = sum(1 for n in _schedule(case["frames"]) if n > 0)
        # and the pass that rates the finished utterances
        return dict(flops=flops * (steps + 1), bytes=bytes_ * (steps + 1))
    if case["kind"] == "forward":
        flops, bytes_ = _step_work(case)
        return dict(flops=flops, bytes=bytes_ + 8.0 * case["frames"] * CODEBOOKS * VOCAB)
    if case["kind"] == "decode":
        flops, weights, length = 0.0, 8 * 1024 * 64, case["frames"]
        for _, cin, cout, taps, scale in _decoder_convs():
            length *= scale
            # a transposed convolution has two taps for every output
            flops += 2.0 * cin * cout * (2 if scale > 1 else taps) * length
            weights += cin * cout * (2 * scale if scale > 1 else taps)
        return dict(flops=flops, bytes=4.0 * (weights + 8 * case["frames"] + length))
    flops, weights = _encoder_work(case["frames"])
    outputs = case["frames"] * (CODEBOOKS + 768 + 256 + 1024)
    return dict(flops=flops, bytes=4.0 * (weights + 960 * case["frames"] + outputs))


def _schedule(frames):
    d = ov.DecodingConfig()
    return ov.unmask_schedule(CODEBOOKS * frames, d.steps, d.t_shift)


def tolerance(case):
    if case["kind"] == "generate":
        # 32 steps, each fed the codes the one before it chose: a pass that rounds a
        # logit otherwise chooses other codes further on, so only the same ones agree.
        return "exact"
    if case["kind"] == "forward":
        # 28 layers with 16-bit activations: 7e-4 from the same pass in 64 bits.
        return dict(rel=3e-3)
    if case["kind"] == "decode":
        # 37 convolutions of 32-bit sums in a row: up to 4.6e-6 from 64 bits.
        return dict(rel=2e-5, max=1e-3)
    # 32-bit sums throughout, up to 1.7e-6 from 64 bits; a code differs where two
    # entries are as near.
    return dict(rel=1e-5, max=1e-3, differ=5e-3)


# ------------------------------------------------------------------ the tokenizer's checkpoint

def _decoder_convs():
    """(name, input channels, output channels, taps, upsampling) of the decoder in order."""
    c = ov.codec_released_config()
    ch = c["channels"]
    convs = [("acoustic_decoder.conv1", c["latent"], ch, 7, 1)]
    for i, ratio in enumerate(c["ratios"]):
        p = f"acoustic_decoder.block.{i}"
        convs.append((p + ".conv_t1", ch, ch // 2, 2 * ratio, ratio))
        ch //= 2
        for u in (1, 2, 3):
            convs += [(f"{p}.res_unit{u}.conv1", ch, ch, 7, 1),
                      (f"{p}.res_unit{u}.conv2", ch, ch, 1, 1)]
    return convs + [("acoustic_decoder.conv2", ch, 1, 7, 1)]


class _Weights:
    """Seeded random tensors by checkpoint name."""

    def __init__(self, seed):
        self.rng, self.tensors = torch.Generator().manual_seed(seed), {}

    def normal(self, name, shape, scale, offset=0.0):
        t = torch.empty(shape, dtype=torch.float32)
        t.normal_(offset, scale, generator=self.rng)
        self.tensors[name] = t

    def conv(self, name, out, cin, taps, gain=1.0, bias=True, transposed=False):
        fan = 2 * cin if transposed else cin * taps
        shape = (cin, out, taps) if transposed else (out, cin, taps)
        self.normal(name + ".weight", shape, gain / math.sqrt(fan))
        if bias:
            self.normal(name + ".bias", (out,), 0.01)

    def linear(self, name, out, cin, gain=1.0):
        self.normal(name + ".weight", (out, cin), gain / math.sqrt(cin))
        self.normal(name + ".bias", (out,), 0.01)

    def norm(self, name, width):
        self.normal(name + ".weight", (width,), 0.1, 1.0)
        self.normal(name + ".bias", (width,), 0.1)

    def alpha(self, name, channels):
        t = torch.empty((1, channels, 1), dtype=torch.float32)
        self.tensors[name + ".alpha"] = t.normal_(0.0, 0.1, generator=self.rng).exp_()

    def units(self, prefix, channels):
        for u in (1, 2, 3):
            p = f"{prefix}.res_unit{u}"
            self.alpha(p + ".snake1", channels)
            self.conv(p + ".conv1", channels, channels, 7)
            self.alpha(p + ".snake2", channels)
            self.conv(p + ".conv2", channels, channels, 1, gain=0.3)

    def write(self, path):
        """The safetensors format: header length, JSON header, the tensors' bytes."""
        header, at = {}, 0
        for name, t in self.tensors.items():
            n = 4 * t.numel()
            header[name] = dict(dtype="F32", shape=list(t.shape), data_offsets=[at, at + n])
            at += n
        text = json.dumps(header).encode()
        text += b" " * (-len(text) % 8)
        with open(path, "wb") as f:
            f.write(struct.pack("<Q", len(text)) + text)
            for t in self.tensors.values():
                f.write(t.numpy().tobytes())

    def load(self, engine, cfg):
        with tempfile.TemporaryDirectory() as root:
            os.mkdir(os.path.join(root, "audio_tokenizer"))
            self.write(os.path.join(root, "audio_tokenizer", "model.safetensors"))
            return engine.load(cfg, root)


def _quantizer(w):
    for q in range(CODEBOOKS):
        p = f"quantizer.quantizers.{q}"
        w.normal(p + ".codebook.embed", (1024, 64), 0.35)
        w.linear(p + ".project_in", 64, 1024)
        w.linear(p + ".project_out", 1024, 64)


@functools.lru_cache(maxsize=1)
def _decoder_weights():
    w, cfg = _Weights(71), ov.codec_released_config()
    _quantizer(w)
    w.linear("fc2", cfg["latent"], cfg["hidden"])
    ch = cfg["channels"]
    w.conv("acoustic_decoder.conv1", ch, cfg["latent"], 7)
    for i, ratio in enumerate(cfg["ratios"]):
        p = f"acoustic_decoder.block.{i}"
        w.alpha(p + ".snake1", ch)
        w.conv(p + ".conv_t1", ch // 2, ch, 2 * ratio, transposed=True)
        ch //= 2
        w.units(p, ch)
    w.alpha("acoustic_decoder.snake1", ch)
    w.conv("acoustic_decoder.conv2", 1, ch, 7, gain=0.1)
    return w


@functools.lru_cache(maxsize=1)
def _encoder_weights():
    w, cfg = _Weights(72), ov.encoder_released_config()
    W, inter = cfg["width"], cfg["intermediate"]
    p, cin = "semantic_model.feature_extractor.conv_layers", 1
    for i, (out, k) in enumerate(zip(cfg["conv_dim"], cfg["conv_kernel"])):
        w.conv(f"{p}.{i}.conv", out, cin, k, bias=False)
        cin = out
    w.norm(f"{p}.0.layer_norm", cfg["conv_dim"][0])
    w.norm("semantic_model.feature_projection.layer_norm", cin)
    w.linear("semantic_model.feature_projection.projection", W, cin)
    p = "semantic_model.encoder.pos_conv_embed.conv"
    w.normal(p + ".parametrizations.weight.original0", (1, 1, cfg["pos_kernel"]), 0.1, 1.0)
    w.normal(p + ".parametrizations.weight.original1",
             (W, W // cfg["pos_groups"], cfg["pos_kernel"]), 1.0)
    w.normal(p + ".bias", (W,), 0.01)
    w.norm("semantic_model.encoder.layer_norm", W)
    for i in range(cfg["layers"]):
        p = f"semantic_model.encoder.layers.{i}"
        for name in ("q_proj", "k_proj", "v_proj", "out_proj"):
            w.linear(f"{p}.attention.{name}", W, W)
        w.norm(p + ".layer_norm", W)
        w.linear(p + ".feed_forward.intermediate_dense", inter, W)
        w.linear(p + ".feed_forward.output_dense", W, inter, gain=0.5)
        w.norm(p + ".final_layer_norm", W)
    w.conv("encoder_semantic.conv", W, W, 3, bias=False)
    for b in range(2):
        p = f"encoder_semantic.conv_blocks.{b}"
        for u in range(2):
            w.conv(f"{p}.res_units.{u}.conv1", W, W, 3, bias=False)
            w.conv(f"{p}.res_units.{u}.conv2", W, W, 1, gain=0.3, bias=False)
        w.conv(p + ".conv", W, W, 3)
    ch = cfg["enc_channels"]
    w.conv("acoustic_encoder.conv1", ch, 1, 7)
    for i, ratio in enumerate(cfg["ratios"]):
        p = f"acoustic_encoder.block.{i}"
        w.units(p, ch)
        w.alpha(p + ".snake1", ch)
        w.conv(p + ".conv1", 2 * ch, ch, 2 * ratio)
        ch *= 2
    w.alpha("acoustic_encoder.snake1", ch)
    w.conv("acoustic_encoder.conv2", cfg["latent"], ch, 3)
    w.linear("fc", W + cfg["latent"], W + cfg["latent"])
    _quantizer(w)
    return w


def _encoder_work(frames):
    """(operations, weights) of one encode."""
    cfg, flops, weights = ov.encoder_released_config(), 0.0, 0
    W, inter = cfg["width"], cfg["intermediate"]

    def layer(positions, cin, cout, taps=1, times=1):
        nonlocal flops, weights
        flops += 2.0 * positions * cin * cout * taps * times
        weights += cin * cout * taps * times

    length, cin = 640 * frames + 320, 1
    for out, k, s in zip(cfg["conv_dim"], cfg["conv_kernel"], cfg["conv_stride"]):
        length = (length - k) // s + 1
        layer(length, cin, out, k)
        cin = out
    layer(length, cin, W)
    layer(length, W // cfg["pos_groups"], W, cfg["pos_kernel"])
    layer(length, W, 4 * W + 2 * inter, times=cfg["layers"])
    flops += 4.0 * cfg["layers"] * length * length * W
    layer(frames, W, W, 3, times=7)
    layer(frames, W, W, 1, times=4)
    length, ch = 960 * frames, cfg["enc_channels"]
    layer(length, 1, ch, 7)
    for ratio in cfg["ratios"]:
        layer(length, ch, ch, 8, times=3)
        length //= ratio
        layer(length, ch, 2 * ch, 2 * ratio)
        ch *= 2
    layer(length, ch, cfg["latent"], 3)
    layer(frames, W + cfg["latent"], W + cfg["latent"])
    layer(frames, W + cfg["latent"], 64, times=CODEBOOKS)
    flops += 2.0 * frames * 1024 * 64 * CODEBOOKS
    return flops, weights + CODEBOOKS * 1024 * 64 * 2


# ------------------------------------------------------------------ the engines and the calls

@functools.lru_cache(maxsize=1)
def _generator():
    return ov.Generator.synthetic(ov.released_config(), GENERATOR_SEED)


@functools.lru_cache(maxsize=1)
def _decoder():
    return _decoder_weights().load(ov.Codec, ov.codec_released_config())


@functools.lru_cache(maxsize=1)
def _encoder():
    return _encoder_weights().load(ov.Encoder, ov.encoder_released_config())


def _inputs(case, seed):
    """Text tokens, the reference's codes and masked target frames of each item."""
    rng = np.random.default_rng(seed)
    vocab = ov.released_config()["vocab_size"]
    inputs = []
    for _ in range(case["items"]):
        ref = (rng.integers(0, MASK, size=(CODEBOOKS, case["reference"]), dtype=np.int32)
               if case["reference"] else None)
        inputs.append(ov.ConditionalInput.build(rng.integers(0, vocab, size=case["text"]), ref,
                                                case["reference"], case["frames"]))
    return inputs


def _codes(case, seed):
    return np.random.default_rng(seed).integers(0, 1024, size=(CODEBOOKS, case["frames"]),
                                                dtype=np.int32)


def _speech(case, seed):
    """A voice-like recording: harmonics of a wandering pitch under a syllable-rate
    envelope with pauses, and breath noise, 24 kHz."""
    rng = np.random.default_rng(seed)
    n = 960 * case["frames"]
    t = np.arange(n) / 24000.0
    pitch = rng.uniform(90, 220) * (1.0 + 0.1 * np.sin(2 * np.pi * rng.uniform(0.3, 0.9) * t))
    phase = 2 * np.pi * np.cumsum(pitch) / 24000.0
    voice = sum(rng.uniform(0.3, 1.0) / k * np.sin(k * phase + rng.uniform(0, 6.28))
                for k in range(1, 13))
    envelope = np.clip(np.sin(2 * np.pi * rng.uniform(2.5, 4.5) * t + rng.uniform(0, 6.28)) + 0.6,
                       0.0, None)
    return (0.12 * envelope * voice + 0.004 * rng.standard_normal(n)).astype(np.float32)


def prepare(case, seed):
    if case["kind"] in ("generate", "forward"):
        return dict(case=case, engine=_generator(), inputs=_inputs(case, seed),
                    seeds=[seed + i for i in range(case["items"])])
    if case["kind"] == "decode":
        codes = _codes(case, seed)
        if not case["device"]:
            return dict(case=case, engine=_decoder(), codes=codes)
        return dict(case=case, engine=_decoder(), codes=torch.from_numpy(codes).cuda(),
                    audio=torch.zeros(960 * case["frames"], device="cuda"))
    return dict(case=case, engine=_encoder(), samples=_speech(case, seed))


def run(state):
    case, engine = state["case"], state["engine"]
    if case["kind"] == "generate":
        results = engine.generate_batch(state["inputs"], ov.DecodingConfig(), state["seeds"])
        # The program rates what it got by the model's own confidence in the finished
        # utterance, the first one's where it made several.
        first, codes = state["inputs"][0], results[0].codes
        ids = first.ids.copy()
        ids[:, first.length - first.target_frames:] = codes
        prediction, confidence = engine.score(
            ov.ConditionalInput(first.codebooks, first.length, first.audio_start,
                                first.target_frames, ids))
        return dict(codes=[r.codes for r in results],
                    unmasked_at=[r.unmasked_at for r in results],
                    prediction=prediction, confidence=confidence)
    if case["kind"] == "forward":
        return engine.forward(state["inputs"][0])
    if case["kind"] == "decode":
        if not case["device"]:
            return engine.decode(state["codes"])
        engine.decode_device(state["codes"], state["audio"])
        return state["audio"]
    return engine.encode(state["samples"], intermediates=True)


# ------------------------------------------------------------------ the same in 64 bits

def exact(case, seed):
    if case["kind"] == "generate":
        return None  # 32 passes, each on codes that the one before it chose
    if case["kind"] == "forward":
        return _exact_forward(_inputs(case, seed)[0])
    if case["kind"] == "decode":
        audio = _exact_decode(torch.from_numpy(_codes(case, seed)).cuda())
        return audio if case["device"] else audio.cpu().numpy()
    return _exact_encode(_speech(case, seed))


def _double(weights):
    return lambda name: weights.tensors[name].cuda().double()


def _conv(x, w, b=None, dilation=1, stride=1, pad=None):
    """Conv1d of x [in][T] with w [out][in][taps], tap by tap."""
    taps = w.shape[2]
    pad = (taps - 1) * dilation // 2 if pad is None else pad
    x = torch.nn.functional.pad(x, (pad, pad))
    n = (x.shape[1] - (taps - 1) * dilation - 1) // stride + 1
    y = 0
    for k in range(taps):
        at = k * dilation
        y = y + w[:, :, k].contiguous() @ x[:, at:at + (n - 1) * stride + 1:stride].contiguous()
    return y if b is None else y + b[:, None]


def _conv_transpose(x, w, b, stride):
    """ConvTranspose1d of kernel 2 stride, cropped to T stride samples."""
    n, pad = x.shape[1], (stride + 1) // 2
    y = torch.zeros(w.shape[1], (n + 2) * stride, dtype=x.dtype, device=x.device)
    for k in range(2 * stride):
        y[:, k:k + (n - 1) * stride + 1:stride] += w[:, :, k].t().contiguous() @ x
    return y[:, pad:pad + n * stride] + b[:, None]


def _snake(x, alpha):
    a = alpha.reshape(-1, 1)
    return x + torch.sin(a * x) ** 2 / (a + 1e-9)


def _units(x, get, prefix):
    for u, dilation in ((1, 1), (2, 3), (3, 9)):
        p = f"{prefix}.res_unit{u}"
        y = _conv(_snake(x, get(p + ".snake1.alpha")), get(p + ".conv1.weight"),
                  get(p + ".conv1.bias"), dilation)
        x = x + _conv(_snake(y, get(p + ".snake2.alpha")), get(p + ".conv2.weight"),
                      get(p + ".conv2.bias"))
    return x


def _exact_decode(codes):
    get = _double(_decoder_weights())
    z = 0
    for q in range(CODEBOOKS):
        p = f"quantizer.quantizers.{q}"
        rows = get(p + ".codebook.embed")[codes[q].long()]
        z = z + rows @ get(p + ".project_out.weight").t() + get(p + ".project_out.bias")
    x = (z @ get("fc2.weight").t() + get("fc2.bias")).t().contiguous()
    x = _conv(x, get("acoustic_decoder.conv1.weight"), get("acoustic_decoder.conv1.bias"))
    for i, ratio in enumerate(ov.codec_released_config()["ratios"]):
        p = f"acoustic_decoder.block.{i}"
        x = _conv_transpose(_snake(x, get(p + ".snake1.alpha")), get(p + ".conv_t1.weight"),
                            get(p + ".conv_t1.bias"), ratio)
        x = _units(x, get, p)
    x = _snake(x, get("acoustic_decoder.snake1.alpha"))
    return _conv(x, get("acoustic_decoder.conv2.weight"),
                 get("acoustic_decoder.conv2.bias")).reshape(-1)


def _resample(samples):
    """24 kHz to 16 kHz by the windowed sinc of 6 zero crossings and rolloff 0.99,
    its bank in 32 bits as the tokenizer defines it, and 160 zeros on each side."""
    base, width, f = 2 * 0.99, 10, np.float32
    t = (-np.arange(2, dtype=f)[:, None] / f(2) +
         np.arange(-width, width + 3, dtype=f)[None, :] / f(3))
    t = np.clip(t * f(base), f(-6), f(6))
    window = np.cos(t * f(math.pi) / f(6) / f(2)) ** 2 * f(base / 3)
    t = t * f(math.pi)
    bank = np.where(t == 0, f(1), np.sin(t) / np.where(t == 0, f(1), t)) * window
    n = (2 * len(samples) + 2) // 3
    x = torch.from_numpy(samples).cuda().double()
    x = torch.nn.functional.pad(x, (width, width + 3))[None]
    w = torch.from_numpy(bank.astype(np.float64)).cuda()[:, None, :]
    y = _conv(x, w, stride=3, pad=0).t().reshape(-1)[:n]
    return torch.nn.functional.pad(y, (160, 160))[None]


def _layer_norm(x, get, name, eps):
    """Over the channels of x [channels][positions]."""
    d = x - x.mean(0)
    return (d / torch.sqrt((d * d).mean(0) + eps) * get(name + ".weight")[:, None] +
            get(name + ".bias")[:, None])


def _exact_encode(samples):
    cfg, get = ov.encoder_released_config(), _double(_encoder_weights())
    gelu, elu = torch.nn.functional.gelu, torch.nn.functional.elu
    W, heads, eps = cfg["width"], cfg["heads"], cfg["eps"]
    frames = len(samples) // cfg["frame_samples"]
    # HuBERT
    x = _resample(samples)
    p = "semantic_model.feature_extractor.conv_layers"
    for i, stride in enumerate(cfg["conv_stride"]):
        x = _conv(x, get(f"{p}.{i}.conv.weight"), stride=stride, pad=0)
        if i == 0:
            d = x - x.mean(1, keepdim=True)
            x = (d / torch.sqrt((d * d).mean(1, keepdim=True) + 1e-5) *
                 get(p + ".0.layer_norm.weight")[:, None] +
                 get(p + ".0.layer_norm.bias")[:, None])
        x = gelu(x)

    def linear(name, x):
        return get(name + ".weight") @ x + get(name + ".bias")[:, None]

    h = linear("semantic_model.feature_projection.projection",
               _layer_norm(x, get, "semantic_model.feature_projection.layer_norm", eps))
    p, K, G = "semantic_model.encoder.pos_conv_embed.conv", cfg["pos_kernel"], cfg["pos_groups"]
    v = get(p + ".parametrizations.weight.original1")
    v = v / torch.sqrt((v * v).sum((0, 1), keepdim=True))
    v = v * get(p + ".parametrizations.weight.original0")
    n = W // G
    pos = torch.cat([_conv(h[g * n:(g + 1) * n], v[g * n:(g + 1) * n], pad=K // 2)
                     for g in range(G)])[:, :h.shape[1]]
    h = _layer_norm(h + gelu(pos + get(p + ".bias")[:, None]), get,
                    "semantic_model.encoder.layer_norm", eps)
    mean = h
    for i in range(cfg["layers"]):
        p = f"semantic_model.encoder.layers.{i}"
        q, k, v = (linear(f"{p}.attention.{c}_proj", h).reshape(heads, W // heads, -1)
                   for c in "qkv")
        scores = q.transpose(1, 2).contiguous() @ k / math.sqrt(W // heads)
        a = v @ torch.softmax(scores, -1).transpose(1, 2).contiguous()
        h = _layer_norm(h + linear(p + ".attention.out_proj", a.reshape(W, -1)), get,
                        p + ".layer_norm", eps)
        y = linear(p + ".feed_forward.output_dense",
                   gelu(linear(p + ".feed_forward.intermediate_dense", h)))
        h = _layer_norm(h + y, get, p + ".final_layer_norm", eps)
        mean = mean + h
    semantic = (mean / (cfg["layers"] + 1))[:, ::cfg["semantic_stride"]][:, :frames].contiguous()
    # the semantic encoder
    s = _conv(semantic, get("encoder_semantic.conv.weight"))
    for b in range(2):
        p = f"encoder_semantic.conv_blocks.{b}"
        for u in range(2):
            y = _conv(elu(s), get(f"{p}.res_units.{u}.conv1.weight"))
            s = s + _conv(elu(y), get(f"{p}.res_units.{u}.conv2.weight"))
        s = _conv(s, get(p + ".conv.weight"), get(p + ".conv.bias"))
    # the acoustic encoder
    x = torch.from_numpy(samples).cuda().double()[None]
    x = _conv(x, get("acoustic_encoder.conv1.weight"), get("acoustic_encoder.conv1.bias"))
    for i, stride in enumerate(cfg["ratios"]):
        p = f"acoustic_encoder.block.{i}"
        x = _snake(_units(x, get, p), get(p + ".snake1.alpha"))
        x = _conv(x, get(p + ".conv1.weight"), get(p + ".conv1.bias"), stride=stride,
                  pad=(stride + 1) // 2)
    x = _snake(x, get("acoustic_encoder.snake1.alpha"))
    acoustic = _conv(x, get("acoustic_encoder.conv2.weight"), get("acoustic_encoder.conv2.bias"))
    embeddings = linear("fc", torch.cat([acoustic, s]))
    return dict(codes=None, **{name: v.t().contiguous().cpu().numpy() for name, v in (
        ("semantic", semantic), ("acoustic", acoustic), ("embeddings", embeddings))})


def _exact_forward(inp):
    """Logits of the conditional then the unconditional target rows."""
    c = ov.released_config()
    h, hd, heads, kv = c["hidden_size"], c["head_dim"], c["heads"], c["kv_heads"]
    inter, eps = c["intermediate_size"], c["rms_norm_eps"]

    def values(tensor, rows, cols, first=0):
        v = ov.synthetic_values(GENERATOR_SEED, tensor, first * cols, rows * cols)
        return torch.from_numpy(v).cuda().double().reshape(rows, cols)

    def norm(x):  # the synthetic model's norm weights are one
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)

    audio = values(2, CODEBOOKS * VOCAB, h)
    ids = torch.from_numpy(inp.ids).long()
    length, frames = inp.length, inp.target_frames

    def embed(columns):
        rows = []
        for t in columns:
            if t < inp.audio_start:
                rows.append(values(1, 1, h, int(ids[0, t]))[0])
            else:
                at = (ids[:, t] + VOCAB * torch.arange(CODEBOOKS)).cuda()
                rows.append(audio[at].sum(0))
        return torch.stack(rows)

    inv = np.float32(1) / np.power(np.float32(c["rope_theta"]),
                                   np.arange(0, hd, 2, dtype=np.float32) / np.float32(hd))
    inv = torch.from_numpy(inv).cuda().double()

    def rope(x):  # [rows][heads][head_dim]
        angle = torch.arange(x.shape[0], device="cuda").double()[:, None, None] * inv
        a, b = x[..., :hd // 2], x[..., hd // 2:]
        return torch.cat([a * angle.cos() - b * angle.sin(),
                          b * angle.cos() + a * angle.sin()], -1)

    sequences = [embed(range(length)), embed(range(length - frames, length))]
    for l in range(c["layers"]):
        t = 100 + 16 * l
        wq, wk, wv = (values(t + j, n * hd, h) for j, n in enumerate((heads, kv, kv)))
        wo, wg, wu = values(t + 3, h, heads * hd), values(t + 4, inter, h), values(t + 5, inter, h)
        wd = values(t + 6, h, inter)
        for s, x in enumerate(sequences):
            y = norm(x)
            q = rope(norm((y @ wq.t()).reshape(-1, heads, hd))).transpose(0, 1)
            k = rope(norm((y @ wk.t()).reshape(-1, kv, hd))).transpose(0, 1)
            v = (y @ wv.t()).reshape(-1, kv, hd).transpose(0, 1)
            k, v = (z.repeat_interleave(heads // kv, 0).contiguous() for z in (k, v))
            scores = q.contiguous() @ k.transpose(1, 2).contiguous() / math.sqrt(hd)
            a = (torch.softmax(scores, -1) @ v).transpose(0, 1).reshape(-1, heads * hd)
            x = x + a @ wo.t()
            y = norm(x)
            sequences[s] = x + (torch.nn.functional.silu(y @ wg.t()) * (y @ wu.t())) @ wd.t()
    rows = torch.cat([x[-frames:] for x in sequences])
    return (norm(rows) @ values(3, CODEBOOKS * VOCAB, h).t()).cpu().numpy()
