"""The calls that a speech synthesis makes on this library, as cases to measure.

One utterance is: a text prefix through both language models (`text_prefix`,
`prefill`), then for each 160 ms patch a BaseLM step (`decode`), a ResidualLM step
(`residual`) and a flow-matching solve (`cfm`), and the AudioVAE over the latents,
patch by patch or for the whole utterance (`vae`).

The models are synthetic ones of the VoxCPM2 geometry with trained-like scales
(projections of unit rows stay near unit variance). They are made once per
process, as a program loads its model once; everything that a request brings
(tokens, hidden states, latents, caches, noise seeds) comes from the case's seed.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch

from voxgen_amd import abi, synth
from voxgen_amd.audiovae import AudioVaeEngine
from voxgen_amd.baselm import BaseLmEngine
from voxgen_amd.locdit import CfmOptions, LocDit
from voxgen_amd.residual import ResidualFsqEngine, prefill_text_cross_engine
from voxgen_amd.runtime import Context, Model

GPU = "cuda"
HEADS, KV_HEADS, HEAD = 16, 2, 128
KV = KV_HEADS * HEAD


# --------------------------------------------------------------------- the cases
def listed():
    return [
        # One BaseLM step of an ordinary utterance with the LM head and the top logits:
        # the whole model, as the benchmark and the token-by-token CLI call it.
        dict(name="decode_token_q8", kind="decode", weights="q8_0", context=512, position=300, tokens=1, head=True),
        # Steps late in a long context with F16 weights, enqueued without host waits.
        dict(name="decode_run_f16_long", kind="decode", weights="f16", context=8192, position=5003, tokens=8,
             head=False),
        # A short, an ordinary and a long prompt through four decoder layers.
        dict(name="prefill_q8_37", kind="prefill", weights="q8_0", context=512, position=0, tokens=37),
        dict(name="prefill_q8_384", kind="prefill", weights="q8_0", context=512, position=0, tokens=384),
        dict(name="prefill_q8_1900", kind="prefill", weights="q8_0", context=2048, position=0, tokens=1900),
        # The text run ahead of a synthesis through both language models.
        dict(name="text_prefix_200", kind="text_prefix", weights="q8_0", context=512, tokens=200),
        # Acoustic positions: FSQ, fusion and the eight F16 layers of the ResidualLM.
        dict(name="residual_steps_8", kind="residual", context=512, tokens=8),
        # A flow-matching solve per patch: the 11-token contract from the language
        # models' buffers, and the wider 37-token conditioning.
        dict(name="cfm_contract", kind="cfm", geometry="contract", cond=4, steps=10),
        dict(name="cfm_cond32", kind="cfm", geometry="wide", cond=32, steps=10),
        # Audio of one patch (streaming), of two seconds through the host call, and of
        # a ten-second utterance between device buffers.
        dict(name="vae_patch", kind="vae", frames=4, host=False),
        dict(name="vae_48_host", kind="vae", frames=48, host=True),
        dict(name="vae_252", kind="vae", frames=252, host=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "prefill", "prefill", "text_prefix", "residual", "cfm", "cfm", "vae", "vae"])
    if kind == "decode":
        context = rng.choice([512, 1024, 4096, 8192])
        head = rng.random() < 0.4
        tokens = 1 if head else rng.randint(1, 8)
        return dict(kind=kind, weights=rng.choice(["q8_0", "f16"]), context=context,
                    position=min(_log(rng, 2, context), context - tokens), tokens=tokens, head=head)
    if kind == "prefill":
        tokens = _log(rng, 2, 1900)
        position = 0 if rng.random() < 0.7 else rng.randint(1, 1000)
        return dict(kind=kind, weights=rng.choice(["q8_0", "q8_0", "f16"]),
                    context=512 if position + tokens <= 512 else 4096, position=position, tokens=tokens)
    if kind == "text_prefix":
        return dict(kind=kind, weights=rng.choice(["q8_0", "f16"]), context=512, tokens=_log(rng, 5, 500))
    if kind == "residual":
        return dict(kind=kind, context=512, tokens=rng.randint(1, 12))
    if kind == "cfm":
        wide = rng.random() < 0.5
        return dict(kind=kind, geometry="wide" if wide else "contract", cond=_log(rng, 4, 60) if wide else 4,
                    steps=rng.randint(4, 12))
    return dict(kind=kind, frames=4 * _log(rng, 1, 63), host=rng.random() < 0.3)


# -------------------------------------------------------------- models and buffers
class _View:
    """Device memory of the library as a torch tensor; keeps its owner alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr, data=(ptr, False), version=2)


def view(buf, shape, dtype=torch.float32, owner=None):
    typestr = {torch.float32: "<f4", torch.float16: "<f2"}[dtype]
    return torch.as_tensor(_View((buf, owner), buf.device_ptr, shape, typestr), device=GPU)


@functools.lru_cache(maxsize=1)
def context():
    torch.zeros(1, device=GPU)   # torch's device context first
    return Context(torch.cuda.current_device())


def _rng(seed):
    return torch.Generator(device=GPU).manual_seed(int(seed) & 0x7FFFFFFFFFFF)


def normal(seed, *shape, dtype=torch.float32):
    return torch.randn(*shape, generator=_rng(seed), device=GPU, dtype=torch.float32).to(dtype)


def _spread(t):
    """(mean, deviation) of a tensor's values; projections 0.02 as the models' initialisers."""
    n = t.name
    if not n.startswith("audio_vae."):
        return (1.0, 0.02) if n.endswith("norm.weight") else (0.0, 0.02)
    if n.endswith("alpha"):
        return 1.0, 0.1
    if n.endswith("scale_embed"):
        return 1.0, 0.05
    if n.endswith((".bias", "bias_embed")):
        return 0.0, 0.02
    gain = 0.1 if ".model.9" in n else 0.3 if n.endswith(".block.3") and n.count(".block.") == 2 else 1.0
    up = n.endswith(".block.1") and n.count(".block.") == 1        # transposed: 2 taps reach an output
    return 0.0, gain / math.sqrt(2 * t.dims[2] if up else t.dims[0] * t.dims[1])


def fill(tensors, seed):
    """The data region of a tensor table, on the GPU."""
    size = max(t.offset + t.nbytes for t in tensors)
    data = torch.zeros((size + 255) // 256 * 256, dtype=torch.uint8, device=GPU)
    for i, t in enumerate(tensors):
        n, g = math.prod(t.dims), _rng(seed * 65537 + i)
        to = data[t.offset:t.offset + t.nbytes]
        if t.name.startswith("rope_factors"):
            to.view(torch.float32).fill_(1.0)
        elif t.ggml_type == abi.DTYPE_Q8_0:       # blocks of an f16 scale and 32 int8 quants
            blocks = to.view(n // 32, 34)
            d = 0.02 / 32 * (1 + 0.1 * torch.randn(n // 32, 1, generator=g, device=GPU))
            blocks[:, :2] = d.half().view(torch.uint8).view(n // 32, 2)
            q = (32 * torch.randn(n // 32, 32, generator=g, device=GPU)).round_().clamp_(-127, 127)
            blocks[:, 2:] = q.to(torch.int8).view(torch.uint8)
        else:
            mean, std = _spread(t)
            x = mean + std * torch.randn(n, generator=g, device=GPU)
            to.copy_(x.to(torch.float16 if t.ggml_type == abi.DTYPE_F16 else torch.float32).view(torch.uint8))
    return data


def _config(name):
    """(configuration, tensor table, seed of the weights)."""
    if name.startswith("base"):
        _, weights, layers = name.split()
        cfg = synth.baselm_config(layers=int(layers), vocab=73448 if layers == "28" else 8192, active_context=512,
                                  embedding_scale=12.0)
        return cfg, synth.build_baselm(cfg, weight_type=weights, with_data=False).tensors, 11
    if name == "acoustic":
        cfg = synth.acoustic_config(active_context=512)
        return cfg, synth.build_acoustic(cfg, with_data=False).tensors, 12
    if name == "vae":
        cfg = synth.audiovae_config()
        return cfg, synth.build_audiovae(cfg, with_data=False).tensors, 13
    # the flow-matching estimator: its generator has no table without data, so a
    # one-layer one gives the tensors and the data is replaced
    wide = name.startswith("wide")
    if wide:
        cfg = synth.locdit_config(layers=8, q_heads=16, kv_heads=16, head_dim=64, n_mu=0, n_cond=int(name.split()[1]),
                                  cond_raw=1, uncond_zero_cond=1)
    else:
        cfg = synth.locdit_config()
    return cfg, _locdit_tensors(wide), 14


@functools.lru_cache(maxsize=2)
def _locdit_tensors(wide):
    cfg = (synth.locdit_config(layers=8, q_heads=16, kv_heads=16, head_dim=64, n_mu=0, n_cond=32, cond_raw=1,
                               uncond_zero_cond=1) if wide else synth.locdit_config())
    return synth.build_locdit(cfg).tensors


@functools.lru_cache(maxsize=8)
def model(name):
    """An uploaded model: made once, as a program loads its file once."""
    _, tensors, seed = _config(name)
    return Model(context(), fill(tensors, seed).cpu().numpy(), tensors)


def _model_name(case):
    kind = case["kind"]
    if kind == "decode":
        return f"base {case['weights']} 28"
    if kind in ("prefill", "text_prefix"):
        return f"base {case['weights']} 4"
    if kind == "residual":
        return "acoustic"
    if kind == "cfm":
        return f"wide {case['cond']}" if case["geometry"] == "wide" else "contract"
    return "vae"


def _loaded(name):
    return model("wide 32" if name.startswith("wide") else name)


# ------------------------------------------------------------------------- inputs
def inputs(case, seed):
    """The request: tensors on the GPU (and plain numbers)."""
    kind = case["kind"]
    if kind in ("decode", "prefill", "text_prefix"):
        cfg = _config(_model_name(case))[0]
        n, layers = case["tokens"], cfg["block_count"]
        r = dict(tokens=torch.randint(0, cfg["vocab_size"], (n,), generator=_rng(seed), device=GPU).cpu().numpy()
                 .astype(np.uint32))
        p = case.get("position", 0)
        if p:   # what earlier steps left in the cache
            r["k"] = normal(seed + 1, layers, p, KV, dtype=torch.float16)
            r["v"] = normal(seed + 2, layers, p, KV, dtype=torch.float16)
        return r
    if kind == "residual":
        n = case["tokens"]
        return dict(base=normal(seed, n, 2048), embedding=normal(seed + 1, n, 2048))
    if kind == "cfm":
        if case["geometry"] == "wide":
            return dict(cond=normal(seed, case["cond"] * 1024).cpu().numpy(), noise=int(seed) & 0xFFFFFFFFFF)
        return dict(cond=normal(seed, 4 * 64).cpu().numpy(), noise=int(seed) & 0xFFFFFFFFFF,
                    lm=normal(seed + 1, 2048), residual=normal(seed + 2, 2048))
    return dict(latents=normal(seed, case["frames"], 64))


def _base_engine(case):
    name = _model_name(case)
    cfg = dict(_config(name)[0], active_context_length=case["context"])
    return BaseLmEngine(context(), _loaded(name), cfg, strict_geometry=False)


def _cache(eng, layers, context_length):
    return [view(eng.buffer(b), (layers, context_length, KV), torch.float16, eng) for b in ("kv_k", "kv_v")]


def _residual_engine(case):
    cfg = dict(_config("acoustic")[0], active_context_length=case["context"])
    return ResidualFsqEngine(context(), model("acoustic"), cfg)


def _device(x):
    """A buffer of the library with x's values."""
    b = context().alloc(x.numel() * x.element_size())
    view(b, x.shape, x.dtype).copy_(x)
    return b


def prepare(case, seed):
    kind, r = case["kind"], inputs(case, seed)
    s = dict(case=case)
    if kind in ("decode", "prefill", "text_prefix"):
        eng = s["eng"] = _base_engine(case)
        layers, n, p = eng.config["block_count"], case["tokens"], case.get("position", 0)
        k, v = _cache(eng, layers, case["context"])
        if p:
            k[:, :p], v[:, :p] = r["k"], r["v"]
        s["tokens"] = r["tokens"]
        s["out"] = dict(hidden=view(eng.buffer("norm"), (2048,), owner=eng), k=k[:, p:p + n], v=v[:, p:p + n])
        if case.get("head"):
            s["out"]["logits"] = view(eng.buffer("logits"), (eng.config["vocab_size"],), owner=eng)
        if kind == "text_prefix":
            s["out"].pop("hidden")   # its place after a run over rows is not specified
    if kind in ("residual", "text_prefix"):
        res = s["res"] = _residual_engine(case)
        k, v = _cache(res, 8, case["context"])
        n = case["tokens"]
        s.setdefault("out", {}).update(res_out=view(res.output_buffer(), (2048,), owner=res),
                                       res_k=k[:, :n], res_v=v[:, :n])
        if kind == "residual":
            s["rows"], s["emb_rows"] = _device(r["base"]), _device(r["embedding"])
            s["base"], s["emb"] = context().alloc(8192), context().alloc(8192)
    if kind == "cfm":
        name = _model_name(case)
        s["loc"] = LocDit(context(), _loaded(name), _config(name)[0], strict_geometry=case["geometry"] == "contract")
        s["cond"] = r["cond"]
        s["options"] = CfmOptions(n_timesteps=case["steps"], seed=r["noise"])
        if "lm" in r:
            s["lm"], s["residual"] = _device(r["lm"]), _device(r["residual"])
    if kind == "vae":
        s["vae"] = AudioVaeEngine(context(), _loaded("vae"), _config("vae")[0])
        if case["host"]:
            s["latents"] = r["latents"].cpu().numpy()
        else:
            s["latents"], s["wave"] = _device(r["latents"]), context().alloc(case["frames"] * 1920 * 4)
            s["out"] = view(s["wave"], (case["frames"] * 1920,))
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------------ one pass
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        eng = s["eng"]
        eng.set_position(case["position"])
        if case["head"]:
            r = eng.decode_token(int(s["tokens"][0]), top_k=8)
            return dict(s["out"], top=np.array([v for _, v in r.top_logits], np.float32))
        eng.decode_tokens_gpu_only(s["tokens"])
        return s["out"]
    if kind == "prefill":
        s["eng"].set_position(case["position"])
        s["eng"].prefill_tokens_batched_gpu_only(s["tokens"])
        return s["out"]
    if kind == "text_prefix":
        s["eng"].reset()
        s["res"].reset()
        prefill_text_cross_engine(s["eng"], s["res"], s["tokens"])
        return s["out"]
    if kind == "residual":
        res, ctx = s["res"], context()
        res.reset()
        for i in range(case["tokens"]):   # the language model leaves its row in one buffer, the encoder in another
            abi.call("vx_copy", ctx.handle, s["base"].handle, 0, s["rows"].handle, 8192 * i, 8192)
            abi.call("vx_copy", ctx.handle, s["emb"].handle, 0, s["emb_rows"].handle, 8192 * i, 8192)
            res.step_from_gpu_base_and_embedding_gpu_only(s["base"], s["emb"])
        return s["out"]
    if kind == "cfm":
        if "lm" in s:
            return s["loc"].cfm_from_model_hiddens(s["lm"], s["residual"], s["cond"], s["options"])[0]
        return s["loc"].cfm_solve(s["cond"], None, s["options"])[0]
    if case["host"]:
        return s["vae"].decode_latents(s["latents"])[1]
    s["vae"].decode_latents_gpu(s["latents"], case["frames"], s["wave"])
    return s["out"]


# ---------------------------------------------------------------- what it must cost
def _layer_macs(hidden=2048, ffn=6144, q=2048, kv=256):
    return hidden * (q + 2 * kv) + q * hidden + 3 * hidden * ffn


def work(case):
    kind, n = case["kind"], case.get("tokens", 1)
    per_weight = 34 / 32 if case.get("weights") == "q8_0" else 2
    if kind in ("decode", "prefill", "text_prefix"):
        layers = 28 if kind == "decode" else 4
        p = case.get("position", 0)
        passes = n if kind == "decode" else 1      # a decoded token needs every weight again
        cached = sum(p + i + 1 for i in range(n)) if kind == "decode" else p + n
        by = layers * (passes * (_layer_macs() * per_weight + 2 * 2048 * 4) + 2 * 2 * KV * (cached + n)) + n * 4096
        keys = n * p + n * (n + 1) // 2
        fl = layers * (2 * n * _layer_macs() + 4 * keys * HEADS * HEAD)
        if case.get("head"):
            by, fl = by + 73448 * 2048 * 2 + 73448 * 4, fl + 2 * 73448 * 2048
        if kind == "text_prefix":
            by += 2 * (8 * _layer_macs() + 2048 * 4096) + 8 * 2 * 2 * KV * n
            fl += 2 * n * (8 * _layer_macs() + 2048 * 2048) + 8 * 4 * keys * HEADS * HEAD
        return dict(bytes=by, flops=fl)
    if kind == "residual":
        macs = 8 * _layer_macs() + 4096 * 2048 + 2 * 2048 * 512
        keys = n * (n + 1) // 2
        return dict(bytes=n * (2 * macs + 2 * 8192) + 8 * 2 * 2 * KV * (keys + n),
                    flops=2 * n * macs + 8 * 4 * keys * HEADS * HEAD)
    if kind == "cfm":
        wide = case["geometry"] == "wide"
        tokens = case["cond"] + 5 if wide else 11
        macs = (8 if wide else 12) * _layer_macs(1024, 4096, 1024 if wide else 2048, 1024 if wide else 256)
        steps = case["steps"] - 1                  # CFG-Zero* skips the first
        return dict(bytes=steps * 2 * macs + 2 * 4 * 1024 * 1024, flops=steps * 2 * 2 * tokens * macs)
    frames = case["frames"]
    macs, weights, c, length = 64 * 2048 * frames, 64 * 2048, 2048, frames
    for s in (8, 6, 5, 2, 2, 2):
        macs += length * s * (c // 2) * 2 * c
        weights += 2 * s * c * (c // 2)
        c, length = c // 2, length * s
        macs += 3 * length * c * (c + 7)
        weights += 3 * c * c
    return dict(bytes=2 * weights + frames * (64 + 1920) * 4, flops=2 * (macs + length * c * 7))


def tolerance(case):
    # About four times the distance measured from the values in 64 bits: sums in 32 bits
    # (4.6e-6 through the AudioVAE, 8e-6 through a solve), and cache rows that are kept
    # as f16, where another order of the sums moves a few values by one unit in the last
    # place (up to 2.4e-4, single values by 1e-3).
    if case["kind"] == "vae":
        return dict(rel=2e-5, max=2e-4)
    if case["kind"] == "cfm":
        return dict(rel=4e-5, max=4e-4)
    return dict(rel=1e-3, max=5e-3)


# ------------------------------------------------------- the same values in 64 bits
class _Weights:
    def __init__(self, name):
        self.cfg, tensors, seed = _config(name)
        self.data, self.t = fill(tensors, seed), {t.name: t for t in tensors}

    def raw(self, name):
        t = self.t[name]
        b = self.data[t.offset:t.offset + t.nbytes]
        if t.ggml_type == abi.DTYPE_Q8_0:
            b = b.view(-1, 34)
            return (b[:, :2].contiguous().view(torch.float16).double() * b[:, 2:].contiguous().view(torch.int8)
                    .double()).view(-1)
        return b.view(torch.float16 if t.ggml_type == abi.DTYPE_F16 else torch.float32).double()

    def mat(self, name):
        return self.raw(name).view(self.t[name].dims[1], self.t[name].dims[0])

    def lin(self, name, x):
        return x @ self.mat(name + ".weight").T + self.raw(name + ".bias")


def _rms(x, w, eps=1e-6):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _rope(x, heads, head, positions):
    half = head // 2
    angle = positions.double()[:, None] / 10000.0 ** (torch.arange(half, device=GPU).double() * 2 / head)
    c, s = angle.cos()[:, None], angle.sin()[:, None]
    x = x.view(-1, heads, head)
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, k, v, mask):
    """q [n, heads, d] over k, v [m, kv heads, d]; mask [n, m] of the keys a row may not see."""
    g = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(g, 1), v.repeat_interleave(g, 1)
    out = []
    for h in range(q.shape[1]):
        s = q[:, h] @ k[:, h].T.contiguous() / math.sqrt(q.shape[2])
        out.append(torch.softmax(s.masked_fill(mask, -math.inf), -1) @ v[:, h].contiguous())
    return torch.stack(out, 1).reshape(q.shape[0], -1)


def _decoder(w, prefix, layers, h, p, kc, vc, rope):
    """Layers over rows h at positions p..; returns (h, new K rows, new V rows), cached as f16."""
    n = h.shape[0]
    pos = torch.arange(p, p + n, device=GPU)
    mask = torch.arange(p + n, device=GPU)[None, :] > pos[:, None]
    ks, vs = [], []
    for layer in range(layers):
        m = lambda x: w.mat(f"{prefix}blk.{layer}.{x}.weight")  # noqa: E731
        x = _rms(h, w.raw(f"{prefix}blk.{layer}.attn_norm.weight"))
        q, k, v = x @ m("attn_q").T, x @ m("attn_k").T, x @ m("attn_v").T
        q = _rope(q, HEADS, HEAD, pos) if rope else q.view(n, HEADS, HEAD)
        k = _rope(k, KV_HEADS, HEAD, pos).reshape(n, KV) if rope else k
        k, v = k.half().double(), v.half().double()
        ks.append(k)
        vs.append(v)
        if p:
            k, v = torch.cat([kc[layer].double(), k]), torch.cat([vc[layer].double(), v])
        a = _attend(q, k.view(-1, KV_HEADS, HEAD), v.view(-1, KV_HEADS, HEAD), mask)
        h = h + a @ m("attn_output").T
        x = _rms(h, w.raw(f"{prefix}blk.{layer}.ffn_norm.weight"))
        h = h + (torch.nn.functional.silu(x @ m("ffn_gate").T) * (x @ m("ffn_up").T)) @ m("ffn_down").T
    return h, torch.stack(ks), torch.stack(vs)


def _exact_base(case, r):
    w = _Weights(_model_name(case))
    tokens = torch.from_numpy(r["tokens"].astype(np.int64)).to(GPU)
    h = 12.0 * w.mat("token_embd.weight")[tokens]
    h, k, v = _decoder(w, "", w.cfg["block_count"], h, case.get("position", 0), r.get("k"), r.get("v"), True)
    rows = _rms(h, w.raw("output_norm.weight"))
    out = dict(hidden=rows[-1], k=k, v=v)
    if case.get("head"):
        out["logits"] = w.mat("token_embd.weight") @ rows[-1]
        out["top"] = out["logits"].topk(8).values
    return rows, out


def _exact_residual(fused, w):
    h, k, v = _decoder(w, "residual_lm.", 8, fused, 0, None, None, False)
    return dict(res_out=_rms(h, w.raw("residual_lm.output_norm.weight"))[-1], res_k=k, res_v=v)


def _noise(n, seed):
    """cfm_noise.comp: Box-Muller pairs from an integer hash."""
    def mix(v):
        v = v.astype(np.uint64)
        for shift, by in ((16, 0x7FEB352D), (15, 0x846CA68B)):
            v = ((v ^ (v >> np.uint64(shift))) * np.uint64(by)) & np.uint64(0xFFFFFFFF)
        return v ^ (v >> np.uint64(16))
    i = np.arange(n, dtype=np.uint64)
    a = mix((i >> np.uint64(1)) ^ np.uint64((seed & 0xFFFFFFFF) ^ 0x9E3779B9))
    b = mix((i >> np.uint64(1)) ^ np.uint64((seed >> 32 & 0xFFFFFFFF) ^ 0x85EBCA6B))
    unit = lambda v: ((v.astype(np.float32) + np.float32(0.5)) * np.float32(2.0 ** -32)).astype(np.float64)  # noqa: E731
    radius = np.sqrt(-2 * np.log(np.maximum(unit(a), 1e-7)))
    turn = 2 * math.pi * unit(b)
    return torch.from_numpy(radius * np.where(i & np.uint64(1), np.sin(turn), np.cos(turn))).to(GPU)


def _exact_cfm(case, r):
    w = _Weights(_model_name(case))
    c, wide = w.cfg, case["geometry"] == "wide"
    hd, heads, kv_heads = c["head_dim"], c["q_heads"], c["kv_heads"]
    silu, mats = torch.nn.functional.silu, {}

    def m(name):
        if name not in mats:
            mats[name] = w.mat(name).T.contiguous()
        return mats[name]

    def time_row(t):
        j = torch.arange(512, device=GPU).double()
        out = 0
        for p, v in (("locdit.time_mlp", t), ("locdit.delta_time_mlp", 0.0)):
            a = 1000.0 * v * torch.exp(j * (-math.log(10000.0) / 511))
            x = torch.cat([a.sin(), a.cos()])[None]
            out = out + w.lin(p + ".linear_2", silu(w.lin(p + ".linear_1", x)))
        return out

    def estimate(x, mu, time, cond):
        h = torch.cat([mu, time, cond, w.lin("locdit.in_proj", x.view(4, 64))])
        n = h.shape[0]
        pos, mask = torch.arange(n, device=GPU), torch.zeros(n, n, dtype=torch.bool, device=GPU)
        for layer in range(c["layers"]):
            p = f"locdit.blk.{layer}."
            y = _rms(h, w.raw(p + "attn_norm.weight"))
            q = _rope(y @ m(p + "attn_q.weight"), heads, hd, pos)
            k = _rope(y @ m(p + "attn_k.weight"), kv_heads, hd, pos)
            v = (y @ m(p + "attn_v.weight")).view(n, kv_heads, hd)
            h = h + _attend(q, k, v, mask) @ m(p + "attn_output.weight")
            y = _rms(h, w.raw(p + "ffn_norm.weight"))
            h = h + (silu(y @ m(p + "ffn_gate.weight")) * (y @ m(p + "ffn_up.weight"))) @ m(p + "ffn_down.weight")
        return w.lin("locdit.out_proj", _rms(h[-4:], w.raw("locdit.norm.weight"))).view(-1)

    cond = torch.from_numpy(r["cond"]).to(GPU).double()
    if wide:
        cond = cond.view(-1, 1024)
        mu = torch.zeros(0, 1024, device=GPU, dtype=torch.float64)
    else:
        cond = w.lin("locdit.cond_proj", cond.view(4, 64))
        mu = torch.cat([w.lin("projections.lm_to_dit_proj", r["lm"].double()[None]),
                        w.lin("projections.res_to_dit_proj", r["residual"].double()[None])])
    x = _noise(256, r["noise"])
    f32 = lambda v: float(np.float32(v))  # noqa: E731  (the time grid is a table of 32-bit numbers)
    grid = [1.0 - i / case["steps"] for i in range(case["steps"] + 1)]
    grid = [f32(t + (math.cos(math.pi / 2 * t) - 1.0 + t)) for t in grid]
    skipped = max(1, int(len(grid) * 0.04))
    for i in range(1 + skipped, len(grid)):
        t, dt = grid[i - 1], grid[i - 1] - grid[i]
        row = time_row(t)
        pos = estimate(x, mu, row, cond)
        neg = estimate(x, torch.zeros_like(mu), row, torch.zeros_like(cond) if wide else cond)
        neg = neg * ((pos @ neg) / (neg @ neg + 1e-8))
        x = x - dt * (neg + 2.0 * (pos - neg))
    return x


def _exact_vae(case, r):
    w = _Weights("vae")
    p = "audio_vae.decoder."

    def snake(x, alpha):
        a = w.raw(alpha)
        return x + torch.sin(a * x) ** 2 / (a + 1e-9)

    def causal(x, name, dilation):     # depthwise, 7 taps, [length, channels]
        taps, n = w.raw(name).view(x.shape[1], 7), x.shape[0]
        padded = torch.cat([x.new_zeros(6 * dilation, x.shape[1]), x])
        out = w.raw(name + ".bias").expand_as(x).clone()
        for k in range(7):
            out += padded[k * dilation:k * dilation + n] * taps[:, k]
        return out

    x = causal(r["latents"].double(), p + "model.0", 1)
    x = x @ w.raw(p + "model.1").view(2048, 64).T + w.raw(p + "model.1.bias")
    c = 2048
    for i, s in enumerate((8, 6, 5, 2, 2, 2)):
        b, row = f"{p}model.{i + 2}", slice(3 * c, 4 * c)      # the 48 kHz bucket
        x = x * w.raw(f"{p}sr_cond_model.{i + 2}.scale_embed")[row] + w.raw(f"{p}sr_cond_model.{i + 2}.bias_embed")[row]
        x = snake(x, b + ".block.0.alpha")
        up = w.raw(b + ".block.1").view(c, c // 2, 2, s).permute(0, 2, 3, 1)      # [in, tap, phase, out]
        now = x @ up[:, 0].reshape(c, -1)
        now[1:] += x[:-1] @ up[:, 1].reshape(c, -1)
        c //= 2
        x = now.view(-1, c) + w.raw(b + ".block.1.bias")
        for j, dilation in enumerate((1, 3, 9)):
            q = f"{b}.block.{j + 2}.block"
            y = snake(causal(snake(x, q + ".0.alpha"), q + ".1", dilation), q + ".2.alpha")
            x = x + y @ w.raw(q + ".3").view(c, c).T + w.raw(q + ".3.bias")
    y = snake(x, p + "model.8.alpha")
    taps, n = w.raw(p + "model.9").view(c, 7), y.shape[0]
    y = torch.cat([y.new_zeros(6, c), y])
    out = w.raw(p + "model.9.bias").expand(n).clone()
    for k in range(7):
        out += y[k:k + n] @ taps[:, k]
    return torch.tanh(out)


def exact(case, seed):
    r, kind = inputs(case, seed), case["kind"]
    if kind in ("decode", "prefill"):
        return _exact_base(case, r)[1]
    if kind == "text_prefix":
        rows, out = _exact_base(case, r)
        w = _Weights("acoustic")
        out.pop("hidden")
        fusion = w.mat("projections.res_fusion_proj.weight")[:, :2048].T
        return dict(out, **_exact_residual(rows @ fusion + w.raw("projections.res_fusion_proj.bias"), w))
    if kind == "residual":
        w = _Weights("acoustic")
        latent = torch.tanh(w.lin("fsq.in_proj", r["base"].double())) * 9.0
        latent = torch.sign(latent) * torch.floor(latent.abs() + 0.5) / 9.0
        lm = w.lin("fsq.out_proj", latent)
        return _exact_residual(w.lin("projections.res_fusion_proj", torch.cat([lm, r["embedding"].double()], 1)), w)
    if kind == "cfm":
        return _exact_cfm(case, r)
    return _exact_vae(case, r)
