"""What the framework's speed is measured on.

Three kinds of call, each through the public bindings (qllm_provider.Provider
and qllm_provider.Model):

* "verify": one speculative decode step of a dense FP4 decoder - 1 guaranteed
  token and a few drafts over a cache that a prompt has filled;
* "prompt": a prompt, or the next turn of a conversation, through the same
  decoder up to the logits of the token after it;
* "turn": a request on a model folder (mixed-layer or latent-attention
  decoder): its prompt, then single tokens, then its end.

Layer widths are those of the repository's own benchmark and tests; a model has
a few layers of each kind instead of all of them, with weights of its own per
layer, so that a pass reads more than the caches hold.  All weights, prompts
and drafts come from the seed.
"""
import json
import math
import os
import random
import shutil
import struct
import sys
import tempfile

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "quantum-llm_amd", "python"))

import qllm_provider as qp  # noqa: E402

VOCABULARY = 32000
DEVICE = "cuda:0"

# The dense decoders: the benchmark's 27B widths, the smaller decoder it sets
# beside the mixed-layer one, and the head layout of the reference's own 27B
# model (head_dim 256, gated attention, head norms, a quarter of a head turned).
DENSE = {
    "small": dict(hidden=2048, intermediate=5632, query_heads=16, kv_heads=4, head_dim=128,
                  rotary_dim=128, output_gated=0, qk_norm=0, zero_centered_norm=0),
    "wide": dict(hidden=5120, intermediate=17408, query_heads=64, kv_heads=8, head_dim=128,
                 rotary_dim=128, output_gated=0, qk_norm=0, zero_centered_norm=0),
    "gated": dict(hidden=5120, intermediate=17408, query_heads=24, kv_heads=4, head_dim=256,
                  rotary_dim=64, output_gated=1, qk_norm=1, zero_centered_norm=1),
}
DENSE_LAYERS = 4
EPSILON, THETA = 1.0e-6, 1.0e6

FOLDER = {
    2048: dict(ff=5632, heads=16, kv_heads=4, recurrent=32, query_rank=768),
    4096: dict(ff=14336, heads=32, kv_heads=8, recurrent=64, query_rank=1536),
}
WINDOW, KEPT, DECAY_RANK = 1024, 4, 64


def listed():
    return [
        # the smallest step: a small decoder early in a conversation, where the
        # launches count and not the bytes
        dict(name="verify-small", kind="verify", model="small", scales="f16", contract="bf16",
             cache="q4h", context=500, rows=5, sampled=False),
        # the headline: the verify step of the 27B widths at 32K context
        dict(name="verify-wide-32k", kind="verify", model="wide", scales="f16",
             contract="bf16", cache="q4h", context=32768, rows=5, sampled=False),
        # the artifact's default contract (per-row Q8 activations, block-32
        # scales) at the reference's head layout, sampled as its figures are
        dict(name="verify-gated-q8-sampled", kind="verify", model="gated", scales="ue8m0",
             contract="q8", cache="q4h", context=4001, rows=5, sampled=True),
        # the exact cache, two drafts, a ragged context
        dict(name="verify-wide-exact-12k", kind="verify", model="wide", scales="f16",
             contract="bf16", cache="f16", context=12345, rows=3, sampled=False),
        # a user's next message in a running conversation
        dict(name="prompt-wide-turn-48", kind="prompt", model="wide", scales="f16",
             cache="q4h", start=2048, rows=48),
        # a short first prompt
        dict(name="prompt-wide-300", kind="prompt", model="wide", scales="f16", cache="q4h",
             start=0, rows=300),
        # a long document, the largest case
        dict(name="prompt-wide-16k", kind="prompt", model="wide", scales="f16", cache="q4h",
             start=0, rows=16384),
        # an ordinary prompt at the reference's head layout, block-32 scales
        dict(name="prompt-gated-3001", kind="prompt", model="gated", scales="ue8m0",
             cache="q4h", start=0, rows=3001),
        # a chat turn on the mixed-layer decoder, mostly single-token decode
        dict(name="mixed-turn", kind="turn", design="mixed", width=2048, layers=4,
             mode="bf16", prompt=100, decoded=32),
        # an ordinary prompt on the wider mixed-layer decoder
        dict(name="mixed-prompt-3000", kind="turn", design="mixed", width=4096, layers=3,
             mode="bf16", prompt=3000, decoded=1),
        # a long prompt and an answer on the latent-attention decoder
        dict(name="latent-turn-6000", kind="turn", design="latent", width=2048, layers=4,
             mode="bf16", prompt=6000, decoded=24),
        # the 32-bit mode, which a user runs to check a model against its source
        dict(name="mixed-turn-32bit", kind="turn", design="mixed", width=2048, layers=4,
             mode="fp32", prompt=333, decoded=8),
    ]


def _between(rng, low, high):
    """An integer spread over the logarithm of the range."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["verify", "verify", "prompt", "prompt", "turn", "turn"])
    if kind == "verify":
        model = rng.choice(["small", "wide", "gated"])
        contract = rng.choice(["bf16", "bf16", "q8"])
        scales = "ue8m0" if contract == "q8" else rng.choice(["f16", "f16", "ue8m0"])
        # (a Q8 prompt takes five rows a pass: a shorter context for those)
        cache = "q4h" if contract == "q8" else rng.choice(["q4h", "q4h", "f16"])
        most = {"q4h": 32768, "f16": 16384}[cache] if contract == "bf16" else 4096
        return dict(kind=kind, model=model, scales=scales, contract=contract, cache=cache,
                    context=_between(rng, 64, most), rows=rng.randint(2, 5),
                    sampled=rng.random() < 0.3)
    if kind == "prompt":
        model = rng.choice(["small", "wide", "wide", "gated"])
        cache = rng.choice(["q4h", "q4h", "q4h", "f16"])
        return dict(kind=kind, model=model, scales=rng.choice(["f16", "f16", "ue8m0"]),
                    cache=cache, start=rng.choice([0, 0, _between(rng, 16, 4096)]),
                    rows=_between(rng, 8, {("q4h", True): 12000, ("q4h", False): 6000}.get(
                        (cache, model != "gated"), 4000)))
    mode = rng.choice(["bf16", "bf16", "bf16", "fp32"])
    width = 2048 if mode == "fp32" else rng.choice([2048, 2048, 4096])
    return dict(kind=kind, design=rng.choice(["mixed", "latent"]), width=width,
                layers=4 if width == 2048 else 3, mode=mode,
                prompt=_between(rng, 8, 500 if mode == "fp32" else 6000),
                decoded=rng.randint(1, 32 if mode == "bf16" else 8))


# ---- random numbers --------------------------------------------------------------

class Pool:
    """Random blocks on the GPU and in host memory; a matrix is a stretch of one
    at a place of its own."""

    def __init__(self, seed):
        self.generator = torch.Generator(device=DEVICE).manual_seed(seed)
        self.places = random.Random(seed)
        self.blocks = {}

    def stretch(self, key, make, count):
        """`count` values of the block `key`, which make(generator) fills once."""
        if key not in self.blocks:
            self.blocks[key] = make(self.generator).cpu().numpy()
        block = self.blocks[key]
        if count > block.size:
            block = self.blocks[key] = np.resize(block, count + 4096)
        start = self.places.randrange((block.size - count) // 64 + 1) * 64
        return block[start:start + count]

    def normal(self, shape):
        return torch.randn(shape, generator=self.generator, device=DEVICE).cpu().numpy()

    def integers(self, high, count):
        return torch.randint(0, high, (count,), generator=self.generator,
                             device=DEVICE).cpu().numpy()


# ---- the dense decoder -------------------------------------------------------------

def _dense_shapes(model):
    g = DENSE[model]
    H, I, Q, KV, d = (g["hidden"], g["intermediate"], g["query_heads"], g["kv_heads"],
                      g["head_dim"])
    return dict(query_projection=(Q * d * (1 + g["output_gated"]), H),
                key_projection=(KV * d, H), value_projection=(KV * d, H),
                output_projection=(H, Q * d), gate_projection=(I, H), up_projection=(I, H),
                down_projection=(H, I))


def _dense_weights(case, seed):
    """FP4 matrices (codes, scales) and F32 norm weights under their roles: the
    model's own, and a dict per layer."""
    g, pool = DENSE[case["model"]], Pool(seed)
    H = g["hidden"]

    def matrix(shape, gain=1.0):
        rows, columns = shape
        codes = pool.stretch("codes", lambda r: torch.randint(
            0, 256, (96 << 20,), generator=r, device=DEVICE, dtype=torch.uint8),
            rows * columns // 2).reshape(rows, columns // 2)
        # E2M1 codes have a root mean square of 2.93
        target = gain / (2.93 * math.sqrt(columns))
        if case["scales"] == "f16":
            scales = pool.stretch(("f16", target), lambda r: (target * torch.exp(
                0.5 * torch.randn(12 << 20, generator=r, device=DEVICE))).half(),
                rows * columns // 16).view(np.uint16).reshape(rows, columns // 16)
        else:
            base = 127 + round(math.log2(target))
            scales = pool.stretch(("ue8m0", base), lambda r: torch.randint(
                base - 1, base + 2, (6 << 20,), generator=r, device=DEVICE,
                dtype=torch.uint8), rows * columns // 32).reshape(rows, columns // 32)
        return codes, scales

    def norm(size):
        return ((0.0 if g["zero_centered_norm"] else 1.0)
                + 0.1 * pool.normal((size,))).astype(np.float32)

    # as in a trained decoder, a layer changes the stream by less than it holds:
    # a code of the 4-bit cache that falls to the other side of an edge then
    # moves the logits by about what bf16 activations do
    gains = dict(output_projection=0.25, down_projection=0.5)
    top = dict(token_embedding=matrix((VOCABULARY, H), math.sqrt(H)), hidden_norm=norm(H),
               output_head=matrix((VOCABULARY, H)))
    layers = []
    for _ in range(DENSE_LAYERS):
        layer = {role: matrix(shape, gains.get(role, 1.0))
                 for role, shape in _dense_shapes(case["model"]).items()}
        layer["input_norm"], layer["post_attention_norm"] = norm(H), norm(H)
        if g["qk_norm"]:
            layer["query_norm"] = 0.1 * pool.normal((g["head_dim"],))
            layer["key_norm"] = 0.1 * pool.normal((g["head_dim"],))
        layers.append(layer)
    return top, layers, pool


def _dense_provider(case, top, layers, positions):
    g = DENSE[case["model"]]
    f16 = case["scales"] == "f16"
    provider = qp.Provider(
        layers=DENSE_LAYERS, vocabulary=VOCABULARY, rope_theta=THETA, norm_epsilon=EPSILON,
        scale_scheme=1 if f16 else 0, kv_encoding=1 if case["cache"] == "f16" else 0,
        kv_page_tokens=256, max_context=(positions + 511) // 256 * 256,
        draft_depth=4, activation_q8=int(case.get("contract") == "q8"), **g)
    abi, tag = (16, "fp4-f16-block16") if f16 else (3, "fp4-block32")

    def stage(source, *roles):
        for role in roles:
            value = source[role]
            if isinstance(value, tuple):
                codes, scales = value
                provider.stage_fp4(role, codes, scales, codes.shape[0], 2 * codes.shape[1],
                                   abi)
            else:
                provider.stage_f32(role, value)

    stage(top, "token_embedding")
    provider.prepare(f"embedding.lookup.{tag}.v1")
    for layer in layers:
        stage(layer, "input_norm", "query_projection", "key_projection", "value_projection",
              "output_projection")
        if g["qk_norm"]:
            stage(layer, "query_norm", "key_norm")
        provider.prepare("block.full-attention.output-gated.v1" if g["output_gated"]
                         else "block.full-attention.standard-gqa.v1")
        stage(layer, "post_attention_norm", "gate_projection", "up_projection",
              "down_projection")
        provider.prepare(f"ffn.swiglu.dense.{tag}.v1")
    stage(top, "hidden_norm", "output_head")
    provider.prepare(f"head.rmsnorm.token-select.{tag}.v1")
    provider.prepare_exact_decode(f"decode.mtp.dense-full-attention.{tag}.exact.v2")
    return provider


def _dense_tokens(case, pool):
    """(context, the call's own tokens): drafts after a guaranteed token, or a
    prompt."""
    before = case["context"] if case["kind"] == "verify" else case["start"]
    tokens = pool.integers(VOCABULARY, before + case["rows"]).astype(np.uint32)
    return tokens[:before], tokens[before:]


class DeviceRows:
    """Rows of a provider's device buffer for torch.as_tensor; holds the
    provider, whose memory it is."""

    def __init__(self, provider, pointer, rows, columns):
        self.provider = provider
        self.__cuda_array_interface__ = {"data": (pointer, False), "shape": (rows, columns),
                                         "typestr": "<f4", "version": 2}


class Dense:
    def __init__(self, case, seed):
        self.case = case
        top, layers, pool = _dense_weights(case, seed)
        self.before, self.tokens = _dense_tokens(case, pool)
        self.position = len(self.before)
        self.provider = provider = _dense_provider(case, top, layers,
                                                   self.position + case["rows"])
        if case.get("sampled"):
            provider.begin_request(temperature_ppm=1000000, top_p_ppm=950000, top_k=20,
                                   seed=seed)
        else:
            provider.begin_request()
        if case.get("contract") == "q8":
            following = np.append(self.before[1:], self.tokens[:1])
            for first in range(0, self.position, 5):
                provider.execute_program(self.before[first:first + 5], first)
                provider.synchronize_batch(following[first:first + 5], first, False)
        elif self.position:
            provider.prefill(self.before, 0)
        rows = case["rows"] if case["kind"] == "verify" else 1
        self.logits = torch.as_tensor(DeviceRows(
            provider, provider.lib.qllm_provider_logits(provider.handle), rows, VOCABULARY),
            device=DEVICE)
        self.hidden = torch.as_tensor(DeviceRows(
            provider, provider.lib.qllm_provider_hidden(provider.handle), rows,
            DENSE[case["model"]]["hidden"]), device=DEVICE)

    def run(self):
        provider = self.provider
        if self.case["kind"] == "prompt":
            provider.prefill(self.tokens, self.position)
            return {"logits": self.logits, "hidden": self.hidden}
        guaranteed = int(self.tokens[0])
        provider.synchronize(guaranteed, self.position)
        provider.set_drafts(self.tokens[1:])
        provider.verify(guaranteed, self.position, provider.geometry.max_context)
        return {"logits": self.logits, "hidden": self.hidden}


# ---- model folders ---------------------------------------------------------------

def _folder_config(case):
    width = case["width"]
    s = FOLDER[width]
    if case["design"] == "mixed":
        attention = {"type": "attention",
                     "mixer": {"heads": s["heads"], "kv_heads": s["kv_heads"], "dim": 128,
                               "vdim": 128, "mask": {"size": WINDOW, "keep_first": KEPT},
                               "rot": {"dims": 128, "base": 10000.0}, "scale": 128 ** -0.5,
                               "v_mix": True}}
        recurrent = {"heads": s["recurrent"], "dim": 64}
        layers = [attention, {"type": "general_delta", "mixer": recurrent},
                  {"type": "wkv", "mixer": recurrent}, attention]
        config = {"architecture": "Zatupel"}
    else:
        windowed = {"type": "latent_attention_2",
                    "mixer": {"heads": s["heads"], "dim": 128, "rot_dim": 64, "vdim": 128,
                              "kv_rank": 512, "q_rank": s["query_rank"],
                              "mask": {"size": WINDOW},
                              "rot": {"dims": 64, "base": 10000.0,
                                      "scaling": {"factor": 8.0, "original": 4096,
                                                  "fast": 32.0, "slow": 1.0}},
                              "scale": 192 ** -0.5}}
        everything = {"type": "latent_attention",
                      "mixer": {"heads": s["heads"], "dim": 128, "vdim": 128, "kv_rank": 512,
                                "scale": 128 ** -0.5}}
        gated = {"type": "gla", "mixer": {"heads": s["recurrent"] // 2, "dim": 64,
                                          "vdim": 128, "tau": 16.0}}
        layers = [gated, windowed, everything, windowed]
        config = {"architecture": "Nametar", "residual_mult": 0.8}
    layers = [dict(layer, mlp={"kind": "dense", "ff": s["ff"]})
              for layer in layers[:case["layers"]]]
    return dict(config, vocab=VOCABULARY, width=width, norm={"eps": 1e-5},
                embedding={"scale": 1.0}, layers=layers)


def _folder_shapes(config):
    vocab, width = config["vocab"], config["width"]
    out = {"embed": (vocab, width), "final.norm": (width,), "head": (vocab, width)}
    latent = config["architecture"] == "Nametar"
    for index, layer in enumerate(config["layers"]):
        p, m, kind = f"l{index}.mix.", layer["mixer"], layer["type"]
        heads, dim = m["heads"], m["dim"]
        vdim = m.get("vdim", dim)
        inner = heads * vdim
        names = ["norm1", "norm2"] + (["norm1b", "norm2b"] if latent else [])
        out.update({f"l{index}.{name}": (width,) for name in names})
        if kind == "attention":
            out.update({p + "q": (heads * dim, width), p + "k": (m["kv_heads"] * dim, width),
                        p + "v": (m["kv_heads"] * vdim, width), p + "g": (heads, width),
                        p + "talk": (heads, heads), p + "vmix": ()})
        elif kind in ("general_delta", "wkv"):
            out.update({p + name: (inner, width) for name in "rkvg"})
            out.update({p + "w1": (DECAY_RANK, width), p + "w2": (inner, DECAY_RANK),
                        p + "w0": (inner,), p + "norm": (inner,)})
            if kind == "general_delta":
                out.update({p + "a": (inner, width), p + "a.b": (inner,)})
            else:
                out.update({p + "mu." + name: (width,) for name in "rkvgw"})
                out[p + "u"] = (heads, dim)
        elif kind == "gla":
            out.update({p + "q": (heads * dim, width), p + "k": (heads * dim, width),
                        p + "v": (inner, width), p + "g": (inner, width),
                        p + "a1": (DECAY_RANK, width), p + "a2": (heads * dim, DECAY_RANK),
                        p + "a2.b": (heads * dim,), p + "norm": (vdim,)})
        else:
            turned = m.get("rot_dim", 0)
            if kind == "latent_attention":
                out.update({p + "q": (heads * dim, width), p + "g": (inner, width)})
            else:
                out.update({p + "dq": (m["q_rank"], width), p + "dq.norm": (m["q_rank"],),
                            p + "uq": (heads * (dim + turned), m["q_rank"])})
            out.update({p + "dkv": (m["kv_rank"] + turned, width),
                        p + "dkv.norm": (m["kv_rank"],),
                        p + "uk": (heads * dim, m["kv_rank"]), p + "uv": (inner, m["kv_rank"])})
        out[p + "o"] = (width, inner)
        ff = layer["mlp"]["ff"]
        out.update({f"l{index}.mlp.gate": (ff, width), f"l{index}.mlp.up": (ff, width),
                    f"l{index}.mlp.down": (width, ff)})
    return out


def _bf16(array):
    return torch.from_numpy(np.ascontiguousarray(array, dtype=np.float32)).bfloat16().view(
        torch.int16).numpy()


def _folder_weights(config, pool):
    """Tensor name -> bf16 bits, scaled so that activations stay O(1) and scores
    spread."""
    weights = {}
    for name, shape in _folder_shapes(config).items():
        last = name.rsplit(".", 1)[-1]
        if len(shape) == 2 and last not in ("talk", "u"):
            gain = 1.0 if last == "embed" else shape[1] ** -0.5 * (
                1.5 if last in ("q", "k", "uq", "uk") else 1.0)
            weights[name] = pool.stretch(("bf16", gain), lambda r: (gain * torch.randn(
                16 << 20, generator=r, device=DEVICE)).bfloat16().view(torch.int16),
                shape[0] * shape[1]).reshape(shape)
            continue
        value = pool.normal(shape)
        if last.startswith("norm"):
            value = 1.0 + 0.2 * value
        elif last == "w0":
            value = value - 3.0
        elif last == "b":
            value = value + (1.0 if name.endswith("a2.b") else 0.0)
        elif last == "vmix":
            value = np.full((), 0.4, np.float32)
        elif ".mu." in name:
            value = 1.0 / (1.0 + np.exp(-value))
        elif last == "u":
            value = 0.5 * value
        elif last == "talk":
            value = np.eye(shape[0]) + 0.2 * value
        weights[name] = _bf16(value).reshape(shape)
    return weights


def _folder_tokens(case, pool):
    tokens = pool.integers(VOCABULARY, case["prompt"] + case["decoded"]).astype(np.uint32)
    return tokens[:case["prompt"]], tokens[case["prompt"]:]


class Folder:
    def __init__(self, case, seed):
        config, pool = _folder_config(case), Pool(seed)
        weights = _folder_weights(config, pool)
        self.prompt, self.answer = _folder_tokens(case, pool)
        header, offset = {}, 0
        for name, bits in weights.items():
            header[name] = {"dtype": "BF16", "shape": list(bits.shape),
                            "data_offsets": [offset, offset + 2 * bits.size]}
            offset += 2 * bits.size
        text = json.dumps(header).encode()
        text += b" " * (-len(text) % 8)
        path = tempfile.mkdtemp()
        try:
            with open(os.path.join(path, "config.json"), "w", encoding="utf-8") as out:
                json.dump(config, out)
            with open(os.path.join(path, "model.safetensors"), "wb") as out:
                out.write(struct.pack("<Q", len(text)) + text)
                for bits in weights.values():
                    out.write(np.ascontiguousarray(bits).data)
            self.model = qp.Model(path, case["prompt"] + case["decoded"] + 8,
                                  kv_page_tokens=256, kv_cache_dtype=case["mode"])
        finally:
            shutil.rmtree(path, ignore_errors=True)

    def run(self):
        """Logits after the prompt and after the last token of an answer that is
        already known, token by token."""
        model = self.model
        request = model.begin()
        first, _ = model.step(request, self.prompt, [len(self.prompt) - 1])
        last = len(self.answer) - 1
        for index, token in enumerate(self.answer):
            logits, _ = model.step(request, [token], [0] if index == last else ())
        model.end(request)
        return {"first": first, "last": logits}

    def __del__(self):
        if hasattr(self, "model"):
            self.model.close()


def prepare(case, seed):
    return (Folder if case["kind"] == "turn" else Dense)(case, seed)


def run(state):
    return state.run()


# ---- what a pass cannot do without --------------------------------------------------

def work(case):
    if case["kind"] == "turn":
        return _folder_work(case)
    g = DENSE[case["model"]]
    H, Q, KV, d = g["hidden"], g["query_heads"], g["kv_heads"], g["head_dim"]
    rows = case["rows"]
    before = case["context"] if case["kind"] == "verify" else case["start"]
    per_weight = 0.5 + (2 / 16 if case["scales"] == "f16" else 1 / 32)
    weights = DENSE_LAYERS * sum(a * b for a, b in _dense_shapes(case["model"]).values())
    head = VOCABULARY * H
    head_rows = rows if case["kind"] == "verify" else 1
    record = KV * 2 * (d // 2 + 2 if case["cache"] == "q4h" else 2 * d)
    seen = rows * before + rows * (rows + 1) // 2
    return {"bytes": ((weights + head) * per_weight + rows * H * per_weight
                      + DENSE_LAYERS * (before + 2 * rows) * record
                      + head_rows * (VOCABULARY + H) * 4),
            "flops": (2 * weights * rows + 2 * head * head_rows
                      + 4 * DENSE_LAYERS * Q * d * seen)}


def _folder_work(case):
    config = _folder_config(case)
    shapes = _folder_shapes(config)
    matrices = sum(s[0] * s[1] for n, s in shapes.items()
                   if len(s) == 2 and n not in ("embed", "head"))
    head = VOCABULARY * case["width"]
    tokens, passes = case["prompt"] + case["decoded"], 1 + case["decoded"]
    size = 4 if case["mode"] == "fp32" else 2
    moved = passes * (2 * (matrices + head) + 4 * VOCABULARY)
    flops = 2 * matrices * tokens + 2 * head * passes
    for layer in config["layers"]:
        m = layer["mixer"]
        heads, dim, vdim = m["heads"], m["dim"], m.get("vdim", m["dim"])
        if layer["type"] in ("general_delta", "wkv", "gla"):
            moved += passes * 2 * heads * dim * vdim * 4
            flops += 6 * tokens * heads * dim * vdim
            continue
        window = m.get("mask", {}).get("size", tokens)
        seen = [min(i + 1, window) for i in range(tokens)]
        pair = 2 * heads * (dim + m.get("rot_dim", 0) + vdim)
        if layer["type"] == "attention":
            record, pair = m["kv_heads"] * (dim + vdim), pair + 2 * heads * heads
        else:
            record = m["kv_rank"] + m.get("rot_dim", 0)
        moved += size * record * (tokens + sum(seen[case["prompt"]:]))
        flops += pair * sum(seen)
    return {"bytes": moved, "flops": flops}


def tolerance(case):
    """Up to four times what the path shows against exact().  Activations are
    bf16 (or Q8) between the matrices, and 4-bit or 8-bit codes of the cache and
    of Q8 rows move by one where a value lies near an edge."""
    return {"rel": 1.2e-5 if case.get("mode") == "fp32" else 3e-2}


# ---- the same in 64 bits --------------------------------------------------------------

FP4 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _dequantise(matrix, scheme):
    codes, scales = (torch.from_numpy(np.ascontiguousarray(m)).to(DEVICE) for m in (
        matrix[0], matrix[1].view(np.int16) if scheme == "f16" else matrix[1]))
    table = torch.tensor(FP4 + [-v for v in FP4], dtype=torch.float64, device=DEVICE)
    values = table[torch.stack([codes & 15, codes >> 4], dim=-1).reshape(
        codes.shape[0], -1).int()]
    if scheme == "f16":
        factor, block = scales.view(torch.float16).double(), 16
    else:
        factor, block = torch.exp2(scales.double() - 127), 32
    values.view(codes.shape[0], -1, block).mul_(factor[:, :, None])
    return values


def _row_norm(x, weight, epsilon, zero_centred):
    x = x / torch.sqrt(x.square().mean(-1, keepdim=True) + epsilon)
    return x * (1.0 + weight if zero_centred else weight)


def _q4h(x):
    """What the 4-bit cache holds of rows of a head: codes -7..7 times a binary16
    scale."""
    scale = (x.abs().amax(-1, keepdim=True) / 7.0).clamp_min(2.0 ** -24).half().double()
    return torch.clamp(torch.round(x / scale), -7, 7) * scale


def _q8_rows(x):
    scale = x.abs().amax(-1, keepdim=True) / 127.0
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    return torch.clamp(torch.round(x / scale), -127, 127) * scale


def _device64(array):
    return torch.from_numpy(np.ascontiguousarray(array)).to(DEVICE).double()


def _turn_halves(x, dims, positions):
    """x [tokens, heads, d]: dimension i turns with i + dims / 2."""
    half = dims // 2
    per = THETA ** (-2.0 * torch.arange(half, dtype=torch.float64, device=DEVICE) / dims)
    angle = positions[:, None, None] * per
    c, s = torch.cos(angle), torch.sin(angle)
    u, v = x[..., :half], x[..., half:dims]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., dims:]], dim=-1)


def _causal(q, k, v, scale, first, gate=None, step=256):
    """q [rows, heads, d] at positions first .., k / v [keys, kv heads, d]."""
    rows, heads, d = q.shape
    group = heads // k.shape[1]
    k, v = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    out = torch.empty_like(q)
    for at in range(0, rows, step):
        n = min(step, rows - at)
        keys = first + at + n
        for h in range(k.shape[0]):
            part = q[at:at + n, h * group:(h + 1) * group].permute(1, 0, 2).reshape(-1, d)
            scores = (part @ k[h, :, :keys]).view(group, n, keys).mul_(scale)
            late = (torch.arange(keys, device=DEVICE)[None, :]
                    > first + at + torch.arange(n, device=DEVICE)[:, None])
            scores.masked_fill_(late, -math.inf)
            o = torch.softmax(scores, dim=-1).view(-1, keys) @ v[h, :keys]
            out[at:at + n, h * group:(h + 1) * group] = o.view(group, n, d).permute(1, 0, 2)
    return out


def _dense_exact(case, seed):
    g, (top, layers, pool) = DENSE[case["model"]], _dense_weights(case, seed)
    before, tokens = _dense_tokens(case, pool)
    tokens = torch.from_numpy(np.concatenate([before, tokens]).astype(np.int64)).to(DEVICE)
    KV, Q, d = g["kv_heads"], g["query_heads"], g["head_dim"]
    zero, gated = g["zero_centered_norm"], g["output_gated"]
    q8 = case.get("contract") == "q8"
    positions = torch.arange(len(tokens), dtype=torch.float64, device=DEVICE)
    last = case["rows"] if case["kind"] == "verify" else 1

    def linear(x, matrix):
        return (_q8_rows(x) if q8 else x) @ _dequantise(matrix, case["scales"]).T

    embedding = _dequantise(top["token_embedding"], case["scales"])
    x = embedding[tokens]
    del embedding
    for index, layer in enumerate(layers):
        h = _row_norm(x, _device64(layer["input_norm"]), EPSILON, zero)
        q = linear(h, layer["query_projection"]).view(len(tokens), Q, -1)
        k = linear(h, layer["key_projection"]).view(len(tokens), KV, d)
        v = linear(h, layer["value_projection"]).view(len(tokens), KV, d)
        gate = q[..., d:] if gated else None
        q = q[..., :d]
        if g["qk_norm"]:
            q = _row_norm(q, _device64(layer["query_norm"]), EPSILON, True)
            k = _row_norm(k, _device64(layer["key_norm"]), EPSILON, True)
        q = _turn_halves(q, g["rotary_dim"], positions)
        k = _turn_halves(k, g["rotary_dim"], positions)
        k, v = (_q4h(k), _q4h(v)) if case["cache"] == "q4h" else (
            k.half().double(), v.half().double())
        if index == len(layers) - 1:       # only the last rows are looked at
            q, x = q[-last:], x[-last:]
            gate = gate[-last:] if gated else None
        o = _causal(q.contiguous(), k, v, d ** -0.5, len(tokens) - len(q))
        if gated:
            o = o * torch.sigmoid(gate)
        x = x + linear(o.reshape(len(q), Q * d), layer["output_projection"])
        del q, k, v, o, gate
        h = _row_norm(x, _device64(layer["post_attention_norm"]), EPSILON, zero)
        for at in range(0, len(x), 4096):
            act = linear(h[at:at + 4096], layer["gate_projection"])
            act = torch.nn.functional.silu(act) * linear(h[at:at + 4096],
                                                         layer["up_projection"])
            x[at:at + 4096] += linear(act, layer["down_projection"])
    logits = linear(_row_norm(x, _device64(top["hidden_norm"]), EPSILON, zero),
                    top["output_head"])
    return {"logits": logits, "hidden": x}


def _sharpened(scores, seen):
    return torch.softmax(scores.masked_fill(~seen, -math.inf), dim=-1)


def _norm64(x, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps)


def _turn_pairs(x, dims, base):
    """x [tokens, heads, d]: dimension 2i turns with 2i + 1."""
    per = base ** (-2.0 * torch.arange(dims // 2, dtype=torch.float64, device=DEVICE) / dims)
    angle = torch.arange(x.shape[0], dtype=torch.float64, device=DEVICE)[:, None, None] * per
    c, s = torch.cos(angle), torch.sin(angle)
    u, v = x[..., 0:dims:2], x[..., 1:dims:2]
    turned = torch.stack([u * c - v * s, v * c + u * s], dim=-1).flatten(-2)
    return torch.cat([turned, x[..., dims:]], dim=-1)


def _mixed_attention(h, w, p, m, first_values):
    n, heads, group = len(h), m["heads"], m["heads"] // m["kv_heads"]
    q = _turn_pairs((h @ w[p + "q"].T).view(n, heads, -1), 128, m["rot"]["base"])
    k = _turn_pairs((h @ w[p + "k"].T).view(n, m["kv_heads"], -1), 128, m["rot"]["base"])
    own = v = (h @ w[p + "v"].T).view(n, m["kv_heads"], -1)
    if first_values is not None:
        v = (1.0 - w[p + "vmix"]) * v + w[p + "vmix"] * first_values
    out = torch.empty(n, heads, v.shape[-1], dtype=torch.float64, device=DEVICE)
    j = torch.arange(n, device=DEVICE)
    for at in range(0, n, 512):
        i = torch.arange(at, min(at + 512, n), device=DEVICE)[:, None]
        low = 0 if at < WINDOW else at - WINDOW + 1
        cols = torch.cat([j[:min(KEPT, low)], j[low:int(i[-1]) + 1]])
        seen = (cols <= i) & ((i - cols < WINDOW) | (cols < KEPT))
        weights = torch.stack([_sharpened(q[i[:, 0], a] @ k[cols, a // group].T * m["scale"],
                                          seen) for a in range(heads)])
        weights = (w[p + "talk"] @ weights.view(heads, -1)).view_as(weights)
        for a in range(heads):
            out[i[:, 0], a] = weights[a] @ v[cols, a // group]
    out = out * torch.sigmoid(h @ w[p + "g"].T)[:, :, None]
    return out.reshape(n, -1) @ w[p + "o"].T, own


def _recurrence(h, w, p, m, kind, eps):
    """The three recurrences, one token after the other, all heads at once."""
    n, heads, dim, vdim = len(h), m["heads"], m["dim"], m.get("vdim", m["dim"])
    before = torch.cat([torch.zeros_like(h[:1]), h[:-1]])
    inputs = {c: h + (before - h) * w[p + "mu." + c] if kind == "wkv" else h for c in "rkvgw"}
    first = "q" if kind == "gla" else "r"
    r = (inputs["r"] @ w[p + first].T).view(n, heads, dim)
    k = (inputs["k"] @ w[p + "k"].T).view(n, heads, dim)
    v = (inputs["v"] @ w[p + "v"].T).view(n, heads, vdim)
    gate = inputs["g"] @ w[p + "g"].T
    if kind == "gla":
        r = r / math.sqrt(dim)
        z = h @ w[p + "a1"].T @ w[p + "a2"].T + w[p + "a2.b"]
        decay = torch.exp(torch.nn.functional.logsigmoid(z) / m["tau"])
    else:
        z = torch.tanh(inputs["w"] @ w[p + "w1"].T) @ w[p + "w2"].T + w[p + "w0"]
        decay = torch.exp(-torch.exp(z)) if kind == "wkv" else torch.exp(
            -math.exp(-0.5) * torch.sigmoid(z))
    decay = decay.view(n, heads, dim)
    state = torch.zeros(heads, dim, vdim, dtype=torch.float64, device=DEVICE)
    out = torch.empty(n, heads, 1, vdim, dtype=torch.float64, device=DEVICE)
    if kind == "general_delta":
        rate = torch.sigmoid(h @ w[p + "a"].T + w[p + "a.b"]).view(n, heads, dim)
        unit = k / torch.sqrt(k.square().sum(-1, keepdim=True) + 1e-6)
        left, row = torch.stack([-rate * unit, k], dim=-1), unit[:, :, None, :]
        for t in range(n):
            right = torch.cat([row[t] @ state, v[t][:, None, :]], dim=1)
            state = torch.baddbmm(decay[t][:, :, None] * state, left[t], right)
            out[t] = r[t][:, None, :] @ state
    else:
        for t in range(n):
            fresh = k[t][:, :, None] * v[t][:, None, :]
            if kind == "wkv":
                out[t] = r[t][:, None, :] @ (state + w[p + "u"][:, :, None] * fresh)
            state = torch.addcmul(fresh, decay[t][:, :, None], state)
            if kind == "gla":
                out[t] = r[t][:, None, :] @ state
    out = _norm64(out[:, :, 0], eps)
    out = (out * w[p + "norm"]).reshape(n, -1) if kind == "gla" else (
        out.reshape(n, -1) * w[p + "norm"])
    out = out * (torch.sigmoid(gate) if kind == "general_delta"
                 else torch.nn.functional.silu(gate))
    return out @ w[p + "o"].T


def _yarn(rot):
    dims, base, s = rot["dims"], rot["base"], rot["scaling"]

    def turning(turns):
        return dims * math.log(s["original"] / (2 * math.pi * turns)) / (2 * math.log(base))

    low, high = max(math.floor(turning(s["fast"])), 0), min(math.ceil(turning(s["slow"])),
                                                            dims - 1)
    per = []
    for i in range(dims // 2):
        plain = base ** (-2.0 * i / dims)
        ramp = min(max((i - low) / max(high - low, 0.001), 0.0), 1.0)
        per.append(plain / s["factor"] * ramp + plain * (1.0 - ramp))
    return torch.tensor(per, dtype=torch.float64, device=DEVICE), (
        0.1 * math.log(s["factor"]) + 1.0)


def _turn_yarn(x, rot):
    """x [tokens, heads, dims]: dimension i turns with i + dims / 2."""
    per, magnitude = _yarn(rot)
    angle = torch.arange(x.shape[0], dtype=torch.float64, device=DEVICE)[:, None, None] * per
    c, s = torch.cos(angle) * magnitude, torch.sin(angle) * magnitude
    u, v = x.chunk(2, dim=-1)
    return torch.cat([u * c - v * s, v * c + u * s], dim=-1)


def _latent_attention(h, w, p, m, eps):
    n, heads, dim, rank = len(h), m["heads"], m["dim"], m["kv_rank"]
    turned = m.get("rot_dim", 0)
    if turned:
        q = _norm64(h @ w[p + "dq"].T, eps) * w[p + "dq.norm"] @ w[p + "uq"].T
    else:
        q = h @ w[p + "q"].T
    q = q.view(n, heads, dim + turned)
    down = h @ w[p + "dkv"].T
    c = _norm64(down[:, :rank], eps) * w[p + "dkv.norm"]
    if turned:
        shared = _turn_yarn(down[:, None, rank:], m["rot"])[:, 0]
        q = torch.cat([q[..., :dim], _turn_yarn(q[..., dim:], m["rot"])], dim=-1)
    window = m.get("mask", {}).get("size", n)
    out = torch.empty(n, heads, m["vdim"], dtype=torch.float64, device=DEVICE)
    j = torch.arange(n, device=DEVICE)
    for a in range(heads):
        k = c @ w[p + "uk"][a * dim:(a + 1) * dim].T
        v = c @ w[p + "uv"][a * m["vdim"]:(a + 1) * m["vdim"]].T
        k = torch.cat([k, shared], dim=1) if turned else k
        for at in range(0, n, 2048):
            i = torch.arange(at, min(at + 2048, n), device=DEVICE)[:, None]
            low = max(0, at - window + 1)
            cols = j[low:int(i[-1]) + 1]
            weights = _sharpened(q[i[:, 0], a] @ k[cols].T * m["scale"],
                                 (cols <= i) & (i - cols < window))
            out[i[:, 0], a] = weights @ v[cols]
    out = out.reshape(n, -1)
    if not turned:
        out = out * torch.sigmoid(h @ w[p + "g"].T)
    return out @ w[p + "o"].T


def _folder_exact(case, seed):
    config, pool = _folder_config(case), Pool(seed)
    weights = _folder_weights(config, pool)
    prompt, answer = _folder_tokens(case, pool)
    tokens = torch.from_numpy(np.concatenate([prompt, answer]).astype(np.int64)).to(DEVICE)
    w = {name: torch.from_numpy(np.ascontiguousarray(bits)).to(DEVICE).view(
        torch.bfloat16).double() for name, bits in weights.items()}
    eps = config["norm"]["eps"]
    latent = config["architecture"] == "Nametar"
    x, first_values = w["embed"][tokens], None

    def mlp(h, p):
        act = h @ w[p + "gate"].T
        act = (torch.nn.functional.silu(act) if latent
               else torch.nn.functional.gelu(act, approximate="tanh"))
        return (act * (h @ w[p + "up"].T)) @ w[p + "down"].T

    for index, layer in enumerate(config["layers"]):
        l, m, kind = f"l{index}.", layer["mixer"], layer["type"]
        h = _norm64(x, eps) * w[l + "norm1"]
        if kind == "attention":
            change, own = _mixed_attention(h, w, l + "mix.", m, first_values)
            first_values = own if first_values is None else first_values
        elif kind.startswith("latent"):
            change = _latent_attention(h, w, l + "mix.", m, eps)
        else:
            change = _recurrence(h, w, l + "mix.", m, kind, eps)
        if latent:
            x = x + config["residual_mult"] * _norm64(change, eps) * w[l + "norm1b"]
            change = mlp(_norm64(x, eps) * w[l + "norm2"], l + "mlp.")
            x = x + config["residual_mult"] * _norm64(change, eps) * w[l + "norm2b"]
        else:
            x = x + change + mlp(_norm64(x, eps) * w[l + "norm2"], l + "mlp.")
    x = x[[len(prompt) - 1, len(tokens) - 1]]
    logits = (_norm64(x, eps) * w["final.norm"]) @ w["head"].T
    return {"first": logits[:1], "last": logits[1:]}


def exact(case, seed):
    with torch.no_grad():
        return (_folder_exact if case["kind"] == "turn" else _dense_exact)(case, seed)
