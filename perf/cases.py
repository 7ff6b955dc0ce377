"""Timed cases of the framework: the work a speech program has it do, through the public
entry points of the `mingtts` package.

Kinds of case (each dict's "kind"):

  linear  one mt_linear / mt_linear_rmsnorm call: any call site of the engine on its own.
  stack   the four linears of one backbone layer with 16-bit activations (the prefill GEMM
          configuration of the benchmark).
  layer   one Qwen2-0.5B layer over M rows of one sequence: rmsnorm + qkv, RoPE + cache append,
          causal (or sliding-window) attention, o +=, rmsnorm + gate|up, down +=.  The prompt's
          prefill, a long context, and the audio encoder's frames (window 65).
  attn    the attention half of a batched decode step by separate calls: rmsnorm + qkv, RoPE +
          append, attention over B caches of their own lengths.
  dit     one DiT block over P sequences of two rows: the reference latents of a voice prompt
          through the aggregator.
  decode  one decode step as one plan: 24 layers with attention over B sequences, then the
          final norm and the stop head.
  vae     one latent of the streaming audio decoder: upsampling, the 24-layer window-65 stack at
          four rows as one plan, the spectrum head, inverse STFT and emission.
  flow    the flow-matching stage of one generation step: the cond embedder and the ODE steps of
          the eight DiT blocks at six rows (one plan), final layer, Euler update.

Sizes are the model's own (hidden 896, 14 query and 2 key heads of 64, MLP 4864, 24 layers; DiT
hidden 1024, 16 heads, MLP 4096; caches of 512 positions and up to the 4096 the entry points
take).  Weights are N(0, 0.02^2), activations N(0, 1), all from the seed.
"""
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ming-tts_amd"))
import mingtts as mt  # noqa: E402

H, QKV, INTER, LAYERS, HQ, HKV = 896, 1152, 4864, 24, 14, 2
HID, HEADS, LATENT, BLOCKS = 1024, 16, 64, 8
NFFT, HOP, RING = 3528, 882, 8
EPS = 1e-6
F = mt.GemvFlags
TYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def listed():
    return [
        # One GEMV of the repository's single-linear configuration: the smallest call, a row
        # through one projection (what latency and the host's share of a call come to).
        dict(name="gemv_row", kind="linear", M=1, N=4864, K=896, x="f16", w="f16", gated=False, norm=False, bias=False,
             act=""),
        # The prefill GEMM configuration: 16-bit activations at the full 512-position cache.
        dict(name="prefill_gemm_512", kind="stack", M=512, w="f16"),
        # The benchmark's text prompt, 174 tokens, one layer, in the types of the fp16 model.
        dict(name="layer_prompt_174", kind="layer", M=174, pos0=0, window=0, cap=512, w="f16", cache="f16"),
        # A long context in one pass: half the longest cache the attention takes.
        dict(name="layer_context_2048", kind="layer", M=2048, pos0=0, window=0, cap=4096, w="f16", cache="f16"),
        # The clone path's audio encoder: 1600 frames, window 65, the checkpoint's bf16 weights
        # and the fp32 cache.
        dict(name="layer_encoder_1600", kind="layer", M=1600, pos0=0, window=65, cap=1600, w="bf16", cache="f32"),
        # Batched serving's decode attention by separate calls: eight sequences, ragged lengths.
        dict(name="attn_decode_8", kind="attn", B=8, cap=2048, window=0, w="f16", cache="f16"),
        # The reference latents of a long voice prompt (400 latents) through an aggregator block.
        dict(name="dit_clone_400", kind="dit", P=400, w="bf16"),
        # The generation step's language-model token, bf16 weights and the fp32 cache.
        dict(name="decode_token", kind="decode", B=1, cap=512, w="bf16", cache="f32"),
        # The guided pair (conditional and unconditional row): the headline decode step.
        dict(name="decode_pair", kind="decode", B=2, cap=512, w="f16", cache="f16"),
        # Two guided pairs at once.
        dict(name="decode_two_pairs", kind="decode", B=4, cap=512, w="f16", cache="f16"),
        # 80 ms of audio from one latent.
        dict(name="vae_latent", kind="vae", at=50, w="f16", cache="f16"),
        # The flow stage of one generation step, ten ODE steps.
        dict(name="flow_stage", kind="flow", steps=10, w="bf16"),
    ]


# (N, K, gated) of the engine's linears.
SHAPES = ((1152, 896, False), (896, 896, False), (4864, 896, True), (896, 4864, False), (3072, 1024, False),
          (1024, 1024, False), (4096, 1024, False), (1024, 4096, False), (3530, 896, False), (64, 1024, False),
          (896, 64, False), (896, 192, False))


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("linear", "linear", "linear", "stack", "layer", "layer", "layer", "attn", "dit", "dit", "decode",
                       "decode", "vae", "flow"))
    w = rng.choice(("f16", "bf16"))
    cache = rng.choice(("f16", "f32"))
    if kind == "linear":
        N, K, gated = rng.choice(SHAPES)
        x = rng.choice(("f32", "f32", w))
        norm = x == "f32" and rng.random() < 0.5
        return dict(kind=kind, M=_log(rng, 1, 2048), N=N, K=K, x=x, w=w, gated=gated, norm=norm, bias=rng.random() < 0.5,
                    act="" if gated else rng.choice(("", "", "gelu", "silu")))
    if kind == "stack":
        return dict(kind=kind, M=_log(rng, 24, 2048), w=w)
    if kind == "layer":
        if rng.random() < 0.4:  # the encoder's frames
            M = _log(rng, 16, 1600)
            return dict(kind=kind, M=M, pos0=0, window=65, cap=M, w=w, cache=cache)
        M = _log(rng, 9, 2048)
        pos0 = 0 if rng.random() < 0.6 else _log(rng, 1, 1024)
        return dict(kind=kind, M=M, pos0=pos0, window=0, cap=max(512, 4 * ((M + pos0 + 3) // 4)), w=w, cache=cache)
    if kind == "attn":
        return dict(kind=kind, B=rng.randint(1, 8), cap=_log(rng, 256, 4096), window=0 if rng.random() < 0.8 else 65, w=w,
                    cache=cache)
    if kind == "dit":
        return dict(kind=kind, P=_log(rng, 1, 400), w=w)
    if kind == "decode":
        return dict(kind=kind, B=rng.choice((1, 2, 4)), cap=_log(rng, 128, 1024), w=w, cache=cache)
    if kind == "vae":
        return dict(kind=kind, at=rng.randint(0, 120), w=w, cache=cache)
    return dict(kind=kind, steps=rng.choice((5, 6, 7, 8, 9, 10)), w=w)


# ------------------------------------------------------------------ inputs --

class Values:
    """Seeded device tensors."""

    def __init__(self, case, seed):
        self.dev = torch.device("cuda", 0)
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(0x5EED + int(seed))
        self.wt = TYPES[case["w"]]

    def act(self, *shape, scale=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=self.dev) * scale).to(dtype)

    def weight(self, *shape, scale=0.02):
        return self.act(*shape, scale=scale, dtype=self.wt)

    def gain(self, *shape):
        return (1.0 + 0.1 * torch.randn(*shape, generator=self.g, device=self.dev)).to(self.wt)

    def zeros(self, *shape):
        return torch.zeros(*shape, device=self.dev)

    def ints(self, lo, hi, n):
        return torch.randint(lo, hi, (n,), generator=self.g, device=self.dev, dtype=torch.int32)

    def inv_freq(self, base):
        i = torch.arange(32, device=self.dev, dtype=torch.float64)
        return torch.pow(torch.tensor(base, device=self.dev, dtype=torch.float64), -2.0 * i / 64.0).float()


def _backbone(v, layers):
    return dict(qkv=v.weight(layers, QKV, H), qkv_b=v.weight(layers, QKV), o=v.weight(layers, H, H),
                gate=v.weight(layers, INTER, H), up=v.weight(layers, INTER, H), down=v.weight(layers, H, INTER),
                n1=v.gain(layers, H), n2=v.gain(layers, H))


def _dit(v, blocks):
    return dict(qkv=v.weight(blocks, 3 * HID, HID), qkv_b=v.weight(blocks, 3 * HID), out=v.weight(blocks, HID, HID),
                out_b=v.weight(blocks, HID), ff1=v.weight(blocks, 4 * HID, HID), ff1_b=v.weight(blocks, 4 * HID),
                ff2=v.weight(blocks, HID, 4 * HID), ff2_b=v.weight(blocks, HID), n1=v.gain(blocks, HID),
                n2=v.gain(blocks, HID))


def _buffers(v, s, rows):
    s.update(resid=v.zeros(rows, H), qkv=v.zeros(rows, QKV), att=v.zeros(rows, HQ * 64), mlp=v.zeros(rows, INTER))


def _caches(v, s, case, *lead):
    shape = (*lead, HKV, case["cap"], 64)
    s["kc"], s["vc"] = v.act(*shape, dtype=TYPES[case["cache"]]), v.act(*shape, dtype=TYPES[case["cache"]])


def _inputs(case, seed):
    """The case's input tensors (no handle, no plan): what `exact` recomputes from too."""
    v, kind = Values(case, seed), case["kind"]
    s = dict(case=case)
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        s.update(x=v.act(M, K, dtype=TYPES[case["x"]]), W=v.weight(N, K), W2=v.weight(N, K) if case["gated"] else None,
                 b=v.weight(N) if case["bias"] else None, g=v.gain(K) if case["norm"] else None, y=v.zeros(M, N))
    elif kind == "stack":
        M = case["M"]
        s.update(p=_backbone(v, 1), x=v.act(M, H, dtype=v.wt), xi=v.act(M, INTER, dtype=v.wt), h=v.act(M, H),
                 yq=v.zeros(M, QKV), yh=v.zeros(M, H), ym=v.zeros(M, INTER))
    elif kind == "layer":
        s.update(p=_backbone(v, 1), h=v.act(case["M"], H), invf=v.inv_freq(1e6))
        _buffers(v, s, case["M"])
        _caches(v, s, case)
    elif kind == "attn":
        B = case["B"]
        s.update(p=_backbone(v, 1), h=v.act(B, H), invf=v.inv_freq(1e6), pos=v.ints(case["cap"] // 4, case["cap"], B))
        s["lens"] = s["pos"] + 1
        _buffers(v, s, B)
        _caches(v, s, case, B)
    elif kind == "dit":
        M = 2 * case["P"]
        s.update(p=_dit(v, 1), h=v.act(M, HID), invf=v.inv_freq(1e4), x=v.zeros(M, HID), qkv=v.zeros(M, 3 * HID),
                 att=v.zeros(M, HID), ff=v.zeros(M, 4 * HID))
    elif kind == "decode":
        B = case["B"]
        s.update(p=_backbone(v, LAYERS), h=v.act(B, H), invf=v.inv_freq(1e6), pos=v.ints(32, case["cap"], B),
                 fin=v.gain(H), stop_w=v.weight(2, H), stop_b=v.weight(2), z=v.zeros(B, H), logits=v.zeros(B, 2))
        _buffers(v, s, B)
        _caches(v, s, case, LAYERS, B)
    elif kind == "vae":
        case = dict(case, cap=512)
        s.update(p=_backbone(v, LAYERS), h=v.act(3, H), invf=v.inv_freq(1e6), head=v.weight(NFFT + 2, H),
                 head_b=v.weight(NFFT + 2), spec=v.zeros(4, NFFT + 2), ring=v.act(RING, NFFT, scale=0.1),
                 pcm=v.zeros(4 * HOP), pos=torch.arange(4 * s["case"]["at"], 4 * s["case"]["at"] + 4, device=v.dev,
                                                        dtype=torch.int32))
        t = torch.arange(NFFT, device=v.dev, dtype=torch.float64)
        s["win"] = (0.5 - 0.5 * torch.cos(2 * torch.pi * (t + 0.5) / NFFT)).float()
        s["cos"] = torch.cos(2 * torch.pi * t / NFFT).float()
        _buffers(v, s, 4)
        _caches(v, s, case, LAYERS)
    else:
        s.update(p=_dit(v, BLOCKS), invf=v.inv_freq(1e4), noise=v.act(LATENT), hist=v.act(LATENT), z=v.act(1, H),
                 cond=v.weight(HID, H), cond_b=v.weight(HID), xw=v.weight(HID, LATENT, scale=0.05),
                 xb=v.weight(HID, scale=0.05), null=v.weight(HID, scale=1.0), fin=v.gain(HID), fin_w=v.weight(LATENT, HID),
                 fin_b=v.weight(LATENT), t1=v.weight(HID, 256), t1_b=v.weight(HID), t2=v.weight(HID, HID),
                 t2_b=v.weight(HID), y=v.zeros(LATENT), cemb=v.zeros(1, HID), x=v.zeros(6, HID), qkv=v.zeros(6, 3 * HID),
                 att=v.zeros(6, HID), ff=v.zeros(6, 4 * HID), pred=v.zeros(6, LATENT))
    return s


def _backbone_plan(s, rows, attn):
    p, items = s["p"], []
    for i in range(LAYERS):
        items += [mt.op(s["resid"], p["qkv"][i], s["qkv"], rows, bias=p["qkv_b"][i], norm=p["n1"][i], eps=EPS), attn(i),
                  mt.op(s["att"], p["o"][i], s["resid"], rows, flags=F.accumulate),
                  mt.op(s["resid"], p["gate"][i], s["mlp"], rows, flags=F.siluGate, w2=p["up"][i], norm=p["n2"][i],
                        eps=EPS),
                  mt.op(s["mlp"], p["down"][i], s["resid"], rows, flags=F.accumulate)]
    return mt.Seq(items)


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "decode":
        B, cap = case["B"], case["cap"]
        s["plan"] = _backbone_plan(s, B, lambda i: mt.attn_op(s["qkv"], B, HQ, HKV, s["pos"], s["kc"][i], s["vc"][i], cap,
                                                              HKV * cap * 64, s["invf"], s["att"]))
    elif kind == "vae":
        s["plan"] = _backbone_plan(s, 4, lambda i: mt.attn_op(s["qkv"], 4, HQ, HKV, s["pos"], s["kc"][i], s["vc"][i], 512,
                                                              0, s["invf"], s["att"], window=65))
    elif kind == "flow":
        p, items = s["p"], []
        for i in range(BLOCKS):
            items += [mt.op(s["x"], p["qkv"][i], s["qkv"], 6, bias=p["qkv_b"][i], norm=p["n1"][i], eps=EPS),
                      mt.dit_attn_op(s["qkv"], 2, 3, HEADS, s["invf"], s["att"]),
                      mt.op(s["att"], p["out"][i], s["x"], 6, flags=F.accumulate, bias=p["out_b"][i]),
                      mt.op(s["x"], p["ff1"][i], s["ff"], 6, flags=F.gelu, bias=p["ff1_b"][i], norm=p["n2"][i], eps=EPS),
                      mt.op(s["ff"], p["ff2"][i], s["x"], 6, flags=F.accumulate, bias=p["ff2_b"][i])]
        s["plan"] = mt.Seq(items)
        s["times"] = mt.FlowSchedule.timesteps(case["steps"])
        s["temb"] = mt.time_embeddings((s["t1"], s["t1_b"]), (s["t2"], s["t2_b"]), s["times"])
    return s


# -------------------------------------------------------------------- runs --

def _run_linear(s):
    c = s["case"]
    flags = (F.siluGate if c["gated"] else 0) | {"": 0, "gelu": F.gelu, "silu": F.silu}[c["act"]]
    mt.linear(s["x"], s["W"], s["y"], flags=flags, w2=s["W2"], bias=s["b"], norm=s["g"], eps=EPS)
    return s["y"]


def _run_stack(s):
    p = s["p"]
    s["yh"].copy_(s["h"])  # the residual rows
    mt.linear(s["x"], p["qkv"][0], s["yq"], bias=p["qkv_b"][0])
    mt.linear(s["x"], p["o"][0], s["yh"], flags=F.accumulate)
    mt.linear(s["x"], p["gate"][0], s["ym"], flags=F.siluGate, w2=p["up"][0])
    mt.linear(s["xi"], p["down"][0], s["yh"], flags=F.accumulate)
    return s["yq"], s["ym"], s["yh"]


def _run_layer(s):
    c, p, M = s["case"], s["p"], s["case"]["M"]
    s["resid"].copy_(s["h"])  # the rows' embeddings
    mt.linear(s["resid"], p["qkv"][0], s["qkv"], bias=p["qkv_b"][0], norm=p["n1"][0], eps=EPS)
    if M <= 64:
        mt.rope_attention(s["qkv"], QKV, M, HQ, HKV, c["pos0"], c["window"], s["kc"], s["vc"], c["cap"], s["invf"], s["att"],
                          H)
    else:
        mt.rope_cache(s["qkv"], QKV, M, HQ, HKV, c["pos0"], s["kc"], s["vc"], c["cap"], s["invf"])
        mt.attention(s["qkv"], QKV, M, HQ, HKV, c["pos0"], c["window"], s["kc"], s["vc"], c["cap"], s["att"], H)
    mt.linear(s["att"], p["o"][0], s["resid"], flags=F.accumulate)
    mt.linear(s["resid"], p["gate"][0], s["mlp"], flags=F.siluGate, w2=p["up"][0], norm=p["n2"][0], eps=EPS)
    mt.linear(s["mlp"], p["down"][0], s["resid"], flags=F.accumulate)
    return s["resid"], s["att"], s["kc"], s["vc"]


def _run_attn(s):
    c, p, B = s["case"], s["p"], s["case"]["B"]
    stride = HKV * c["cap"] * 64
    mt.linear(s["h"], p["qkv"][0], s["qkv"], bias=p["qkv_b"][0], norm=p["n1"][0], eps=EPS)
    mt.rope_cache_decode(s["qkv"], QKV, B, HQ, HKV, s["pos"], s["kc"], s["vc"], c["cap"], stride, s["invf"])
    mt.attention_decode(s["qkv"], QKV, B, HQ, HKV, s["lens"], c["window"], s["kc"], s["vc"], c["cap"], stride, s["att"], H)
    return s["att"], s["kc"], s["vc"]


def _run_dit(s):
    p, P = s["p"], s["case"]["P"]
    s["x"].copy_(s["h"])  # the cls and embedded rows
    mt.linear(s["x"], p["qkv"][0], s["qkv"], bias=p["qkv_b"][0], norm=p["n1"][0], eps=EPS)
    if 2 * P <= 32:
        mt.dit_attention_linear(s["qkv"], P, 2, HEADS, s["invf"], p["out"][0], s["x"], flags=F.accumulate, bias=p["out_b"][0])
    else:
        mt.dit_attention(s["qkv"], P, 2, HEADS, s["invf"], s["att"])
        mt.linear(s["att"], p["out"][0], s["x"], flags=F.accumulate, bias=p["out_b"][0])
    mt.linear(s["x"], p["ff1"][0], s["ff"], flags=F.gelu, bias=p["ff1_b"][0], norm=p["n2"][0], eps=EPS)
    mt.linear(s["ff"], p["ff2"][0], s["x"], flags=F.accumulate, bias=p["ff2_b"][0])
    return s["x"]


def _run_decode(s):
    s["resid"].copy_(s["h"])  # the token's embedding
    s["plan"].run()
    mt.rmsnorm(s["resid"], s["fin"], s["z"], eps=EPS)
    mt.linear(s["z"], s["stop_w"], s["logits"], bias=s["stop_b"])
    return s["resid"], s["z"], s["logits"], s["kc"], s["vc"]


def _run_vae(s):
    at, h = s["case"]["at"], s["h"]
    mt.upsample4(h[0] if at else None, h[1], h[2], s["resid"])
    s["plan"].run()
    mt.linear(s["resid"], s["head"], s["spec"], bias=s["head_b"])
    mt.istft_frames(s["spec"], 4, NFFT, s["cos"], s["win"], s["ring"], 4 * at, RING)
    mt.istft_emit(s["ring"], s["win"], NFFT, HOP, 4 * at * HOP, 4 * HOP, 4 * at + 3, RING, s["pcm"])
    return s["pcm"], s["ring"], s["spec"], s["kc"], s["vc"]


def _run_flow(s):
    steps, t, temb = s["case"]["steps"], s["times"], s["temb"]
    s["y"].copy_(s["noise"])
    mt.linear(s["z"], s["cond"], s["cemb"], bias=s["cond_b"])
    mt.flow_assemble(s["y"], s["hist"], s["cemb"][0], s["null"], temb[0], s["xw"], s["xb"], s["x"])
    for k in range(steps):
        s["plan"].run()
        mt.linear(s["x"], s["fin_w"], s["pred"], bias=s["fin_b"], norm=s["fin"], eps=EPS)
        dt = float(t[k + 1] - t[k])
        if k + 1 < steps:
            mt.flow_euler_assemble(s["y"], s["pred"], 2, 5, 2.0, dt, s["hist"], s["cemb"][0], s["null"], temb[k + 1],
                                   s["xw"], s["xb"], s["x"])
        else:
            mt.flow_euler(s["y"], s["pred"], 2, 5, 2.0, dt)
    return s["y"], s["pred"], s["x"]


_RUN = dict(linear=_run_linear, stack=_run_stack, layer=_run_layer, attn=_run_attn, dit=_run_dit, decode=_run_decode,
            vae=_run_vae, flow=_run_flow)


def run(state):
    return _RUN[state["case"]["kind"]](state)


# -------------------------------------------------------------------- work --

def _size(t):
    return 4 if t == "f32" else 2


_LAYER_MACS = QKV * H + H * H + 2 * INTER * H + H * INTER
_LAYER_BYTES = 2 * (_LAYER_MACS + QKV + 2 * H)
_DIT_MACS = 12 * HID * HID
_DIT_BYTES = 2 * (_DIT_MACS + 11 * HID)


def _keys(M, pos0, window):
    """(row, key) pairs of M causal rows, and the distinct keys they read."""
    pairs = sum(min(pos0 + m + 1, window or 1 << 30) for m in range(M))
    first = max(0, pos0 + 1 - window) if window else 0
    return pairs, pos0 + M - first


def work(case):
    k = case["kind"]
    if k == "linear":
        M, N, K, g = case["M"], case["N"], case["K"], 2 if case["gated"] else 1
        return dict(bytes=2 * N * K * g + _size(case["x"]) * M * K + 4 * M * N + (2 * N if case["bias"] else 0) +
                    (2 * K if case["norm"] else 0), flops=2 * M * N * K * g)
    if k == "stack":
        M = case["M"]
        return dict(bytes=2 * _LAYER_MACS + 2 * QKV + M * (2 * (H + INTER) + 4 * (QKV + INTER + 2 * H)),
                    flops=2 * M * _LAYER_MACS)
    if k == "layer":
        M, cs = case["M"], _size(case["cache"])
        pairs, keys = _keys(M, case["pos0"], case["window"])
        return dict(bytes=_LAYER_BYTES + M * 4 * 2 * H + 2 * HKV * 64 * cs * (keys + M) + 4 * M * H,
                    flops=2 * M * _LAYER_MACS + 4 * 64 * HQ * pairs)
    if k == "attn":
        B, cs = case["B"], _size(case["cache"])
        keys = B * (min(case["window"], case["cap"]) if case["window"] else (5 * case["cap"]) // 8)  # on the mean
        return dict(bytes=2 * QKV * H + B * 4 * (H + HQ * 64) + 2 * HKV * 64 * cs * keys,
                    flops=2 * B * QKV * H + 4 * 64 * HQ * keys)
    if k == "dit":
        M = 2 * case["P"]
        return dict(bytes=_DIT_BYTES + M * 4 * 2 * HID, flops=2 * M * _DIT_MACS + 4 * 64 * HEADS * M * 2)
    if k == "decode":
        B, cs = case["B"], _size(case["cache"])
        keys = B * (32 + case["cap"]) // 2  # on the mean
        return dict(bytes=LAYERS * (_LAYER_BYTES + 2 * HKV * 64 * cs * (keys + B)) + B * 4 * 3 * H,
                    flops=LAYERS * (2 * B * _LAYER_MACS + 4 * 64 * HQ * keys))
    if k == "vae":
        cs = _size(case["cache"])
        pairs, keys = _keys(4, 4 * case["at"], 65)
        return dict(bytes=LAYERS * (_LAYER_BYTES + 2 * HKV * 64 * cs * (keys + 4)) + 2 * (NFFT + 2) * H +
                    4 * (4 * (NFFT + 2) + 2 * RING * NFFT + 4 * HOP),
                    flops=LAYERS * (8 * _LAYER_MACS + 4 * 64 * HQ * pairs) + 8 * (NFFT + 2) * H)
    # Each ODE step reads the blocks' weights once (201 MB, more than the chip's L2 holds).
    return dict(bytes=case["steps"] * (BLOCKS * _DIT_BYTES + 4 * HID * LATENT), flops=case["steps"] * 12 * BLOCKS * _DIT_MACS)


# About four times the largest relative error seen against `exact` (fp32 sums; fp32 activations
# meet 16-bit weights as hi + lo halves, 2^-17 with bf16; a K / V value that rounds the other way
# in an fp16 cache differs by 2^-10 of itself, which `max` allows).
_TOL = dict(linear=(1e-5, 1e-3), stack=(1e-6, 1e-4), layer=(1.5e-4, 4e-3), attn=(1.5e-4, 4e-3), dit=(1e-5, 1e-3),
            decode=(1e-4, 4e-3), vae=(1e-4, 4e-3), flow=(3e-5, 3e-3))


def tolerance(case):
    rel, most = _TOL[case["kind"]]
    return dict(rel=rel, max=most)


# ------------------------------------------------------ the same in 64 bits --

def _d(t):
    return None if t is None else t.double()


def _mm(x, w, b=None):
    y = x @ w.double().t().contiguous()
    return y if b is None else y + b.double()


def _norm(x, g):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS) * g.double()


def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _gelu(v):
    return 0.5 * v * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (v + 0.044715 * v ** 3)))


def _neox(x, pos, invf):
    """Pairs (i, i + 32) of [rows, heads, 64] at the fp32 angles pos * inv_freq (the operation's
    own definition of the angle)."""
    a = (pos.float()[:, None] * invf[None, :]).double()[:, None, :]
    x0, x1, c, s = x[..., :32], x[..., 32:], torch.cos(a), torch.sin(a)
    return torch.cat([x0 * c - x1 * s, x1 * c + x0 * s], -1)


def _softmax_av(q, k, v, lo, hi):
    """q [rows, 64], k / v [keys, 64]; row m attends over keys lo[m] .. hi[m] - 1."""
    j = torch.arange(k.shape[0], device=q.device)
    s = (q @ k.t().contiguous()) * 0.125
    s = s.masked_fill((j[None, :] < lo[:, None]) | (j[None, :] >= hi[:, None]), -math.inf)
    return torch.softmax(s, -1) @ v


def _attend(qkv, rows, pos, kc, vc, window, invf, shared):
    """Appends the rows' k and v to the caches (given and returned as fp64 holding the stored
    values) and attends.  shared: the rows are consecutive positions of one cache [hkv, cap,
    64]; otherwise row b has cache [b]."""
    q = _neox(qkv[:, : HQ * 64].reshape(rows, HQ, 64), pos, invf)
    k = _neox(qkv[:, HQ * 64 : (HQ + HKV) * 64].reshape(rows, HKV, 64), pos, invf)
    v = qkv[:, (HQ + HKV) * 64 :].reshape(rows, HKV, 64)
    kd, vd = kc.double(), vc.double()
    for m in range(rows) if not shared else ():
        kd[m, :, pos[m]] = k[m].to(kc.dtype).double()
        vd[m, :, pos[m]] = v[m].to(vc.dtype).double()
    if shared:
        p0 = int(pos[0])
        kd[:, p0 : p0 + rows] = k.transpose(0, 1).to(kc.dtype).double()
        vd[:, p0 : p0 + rows] = v.transpose(0, 1).to(vc.dtype).double()
    out = torch.empty(rows, HQ, 64, dtype=torch.float64, device=qkv.device)
    hi = pos.long() + 1
    lo = (hi - window).clamp(min=0) if window else torch.zeros_like(hi)
    for h in range(HQ):
        g = h // (HQ // HKV)
        if shared:
            n = int(hi[-1])
            out[:, h] = _softmax_av(q[:, h], kd[g, :n], vd[g, :n], lo, hi)
        else:
            for m in range(rows):
                out[m, h] = _softmax_av(q[m : m + 1, h], kd[m, g], vd[m, g], lo[m : m + 1], hi[m : m + 1])[0]
    return out.reshape(rows, HQ * 64), kd, vd


def _backbone_layer(x, p, i, pos, kc, vc, window, invf, shared):
    rows = x.shape[0]
    qkv = _mm(_norm(x, p["n1"][i]), p["qkv"][i], p["qkv_b"][i])
    att, kd, vd = _attend(qkv, rows, pos, kc, vc, window, invf, shared)
    x = x + _mm(att, p["o"][i])
    n = _norm(x, p["n2"][i])
    x = x + _mm(_silu(_mm(n, p["gate"][i])) * _mm(n, p["up"][i]), p["down"][i])
    return x, att, kd, vd


def _dit_block(x, p, i, S, invf):
    rows = x.shape[0]
    qkv = _mm(_norm(x, p["n1"][i]), p["qkv"][i], p["qkv_b"][i]).reshape(rows // S, S, 3, HEADS, 64)
    a = (torch.arange(S, device=x.device).float()[:, None] * invf[None, :]).double()[None, :, None, :]
    c, s = torch.cos(a), torch.sin(a)

    def rot(t):
        e, o = t[..., 0::2], t[..., 1::2]
        return torch.stack([e * c - o * s, o * c + e * s], -1).flatten(-2)

    q, k, v = (t.permute(0, 2, 1, 3).contiguous() for t in (rot(qkv[:, :, 0]), rot(qkv[:, :, 1]), qkv[:, :, 2]))
    w = torch.softmax((q[:, :, :, None] * k[:, :, None]).sum(-1) * 0.125, -1)
    att = (w[..., None] * v[:, :, None]).sum(3).permute(0, 2, 1, 3).reshape(rows, HID)
    x = x + _mm(att, p["out"][i], p["out_b"][i])
    ff = _gelu(_mm(_norm(x, p["n2"][i]), p["ff1"][i], p["ff1_b"][i]))
    return x + _mm(ff, p["ff2"][i], p["ff2_b"][i])


def exact(case, seed):
    """What `run` returns, in 64 bits.  None for an fp16 cache and for the attention read straight
    from it: which way a stored value rounds is no matter of 64-bit arithmetic, and one that
    rounds the other way outweighs every other error there."""
    v = _exact(case, seed)
    if case.get("cache") == "f16":
        cached = dict(layer=(1, 2, 3), attn=(0, 1, 2), decode=(3, 4), vae=(3, 4))[case["kind"]]
        v = tuple(None if i in cached else x for i, x in enumerate(v))
        v = None if all(x is None for x in v) else v
    return v


def _exact(case, seed):
    s, k = _inputs(case, seed), case["kind"]
    if k == "linear":
        x = _d(s["x"])
        if case["norm"]:
            x = _norm(x, s["g"])
        y = _mm(x, s["W"], s["b"])
        if case["gated"]:
            y = _silu(y) * _mm(x, s["W2"])
        return _gelu(y) if case["act"] == "gelu" else _silu(y) if case["act"] == "silu" else y
    p = s["p"]
    if k == "stack":
        x, xi = _d(s["x"]), _d(s["xi"])
        ym = _silu(_mm(x, p["gate"][0])) * _mm(x, p["up"][0])
        return _mm(x, p["qkv"][0], p["qkv_b"][0]), ym, _d(s["h"]) + _mm(x, p["o"][0]) + _mm(xi, p["down"][0])
    if k == "layer":
        pos = torch.arange(case["pos0"], case["pos0"] + case["M"], device=s["h"].device)
        return _backbone_layer(_d(s["h"]), p, 0, pos, s["kc"], s["vc"], case["window"], s["invf"], True)
    if k == "attn":
        qkv = _mm(_norm(_d(s["h"]), p["n1"][0]), p["qkv"][0], p["qkv_b"][0])
        return _attend(qkv, case["B"], s["pos"], s["kc"], s["vc"], case["window"], s["invf"], False)
    if k == "dit":
        return _dit_block(_d(s["h"]), p, 0, 2, s["invf"])
    if k in ("decode", "vae"):
        if k == "decode":
            x = _d(s["h"])
        else:
            a, h, n = _d(s["h"])
            if not case["at"]:
                a = h
            x = torch.stack([0.625 * h + 0.375 * a, 0.875 * h + 0.125 * a, 0.875 * h + 0.125 * n, 0.625 * h + 0.375 * n])
        ks, vs = [], []
        for i in range(LAYERS):
            x, _, kd, vd = _backbone_layer(x, p, i, s["pos"], s["kc"][i], s["vc"][i], 65 if k == "vae" else 0, s["invf"],
                                           k == "vae")
            ks.append(kd)
            vs.append(vd)
        if k == "decode":
            z = _norm(x, s["fin"])
            return x, z, _mm(z, s["stop_w"], s["stop_b"]), torch.stack(ks), torch.stack(vs)
        spec = _mm(x, s["head"], s["head_b"])
        bins = NFFT // 2 + 1
        full = torch.polar(torch.exp(spec[:, :bins]).clamp(max=100.0), spec[:, bins:])
        full.imag[:, 0] = 0.0
        full.imag[:, -1] = 0.0
        ring, win, f0 = _d(s["ring"]), _d(s["win"]), 4 * case["at"]
        for f in range(4):
            t = torch.arange(NFFT, device=x.device)
            b = torch.arange(1, bins - 1, device=x.device)
            ang = ((b[:, None] * t[None, :]) % NFFT).double() * (2.0 * math.pi / NFFT)
            y = full[f, 0].real + full[f, -1].real * (1.0 - 2.0 * (t % 2).double())
            y = y + 2.0 * (full[f, 1:-1].real @ torch.cos(ang) - full[f, 1:-1].imag @ torch.sin(ang))
            ring[(f0 + f) % RING] = y / NFFT * win
        at = f0 * HOP + torch.arange(4 * HOP, device=x.device) + (NFFT - HOP) // 2
        acc, env = torch.zeros(4 * HOP, dtype=torch.float64, device=x.device), torch.zeros(4 * HOP, dtype=torch.float64,
                                                                                          device=x.device)
        for f in range(max(0, f0 - 4), f0 + 4):
            t = at - f * HOP
            ok = (t >= 0) & (t < NFFT)
            t = t.clamp(0, NFFT - 1)
            acc += torch.where(ok, ring[f % RING][t], 0.0)
            env += torch.where(ok, win[t] ** 2, 0.0)
        return acc / env, ring, spec, torch.stack(ks), torch.stack(vs)
    # flow: the schedule and the sinusoids are the sampler's fp32 host arithmetic, given.
    steps, dev = case["steps"], s["noise"].device
    times = mt.FlowSchedule.timesteps(steps)
    sinus = torch.from_numpy(mt.FlowSchedule.sinusoids(times[:steps])).to(dev).double()
    temb = _mm(_silu(_mm(sinus, s["t1"], s["t1_b"])), s["t2"], s["t2_b"])
    cemb = _mm(_d(s["z"]), s["cond"], s["cond_b"])[0]
    y, pred, x = _d(s["noise"]), None, None
    emb = lambda v: _mm(v[None], s["xw"], s["xb"])[0]  # noqa: E731
    for i in range(steps):
        x = torch.stack([temb[i] + cemb, emb(_d(s["hist"])), emb(y), temb[i] + _d(s["null"]), emb(_d(s["hist"])), emb(y)])
        for b in range(BLOCKS):
            x = _dit_block(x, p, b, 3, s["invf"])
        pred = _mm(_norm(x, s["fin"]), s["fin_w"], s["fin_b"])
        y = y + (pred[2] + (pred[2] - pred[5]) * 2.0) * float(times[i + 1] - times[i])
    return y, pred, x
