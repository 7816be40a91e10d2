"""Performance cases: the calls that programs on this framework spend their time in, over the sizes they meet.

Whole calls: GPT-2 124M decode steps and prompt chunks (f32), the Qwen3 language model's decode steps and prompt
chunks (f16, 4 of its 28 identical layers, full vocabulary) and the MNIST MLP. Blocks of the Kokoro-82M speech model
(f32), each through the model's own method: the ALBERT text encoder, a BiLSTM, a decoder block, a generator resblock.
The whole Kokoro forward is no case: the phase of its harmonic source is a running sum over all frames, which turns
last-bit differences of the pitch curve into different audio, so no two correct implementations agree on it.

Model blocks run as stream-captured graphs (lk.capture) that read their activations in place, as inside the forward.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import lokinfer_amd as lk
from lokinfer_amd import gpt2 as G
from lokinfer_amd import kokoro_weights as KW
from lokinfer_amd.kokoro import KokoroGpu
from lokinfer_amd.qwen3 import Qwen3Config, Qwen3Lm

QWEN = Qwen3Config(layers=4)
STYLE = 128


def listed() -> list[dict]:
    return [
        # the smallest call: one image through the MNIST MLP (784 -> 128 -> 10), where launches and host time count
        {"name": "mlp_b1", "kind": "mlp", "batch": 1},
        # Kokoro at the benchmark's short (59 tokens, 287 frames) and long (487 tokens, 2444 frames) utterances
        {"name": "albert_t59", "kind": "albert", "tokens": 59},
        {"name": "albert_t487", "kind": "albert", "tokens": 487},
        # the frame-level BiLSTM of the long utterance: the longest serial recurrence of a forward
        {"name": "lstm_t2444", "kind": "lstm", "steps": 2444},
        # a decoder AdainResBlk1d (1090 -> 1024 channels) at frame rate
        {"name": "decoder_f287", "kind": "decoder", "frames": 287, "up": False},
        # generator Snake resblocks: the short utterance's stage 0, and the long one's stage 1, the widest of a forward
        {"name": "resblock_s0_f287_k7", "kind": "resblock", "frames": 287, "stage": 0, "k": 7},
        {"name": "resblock_s1_f2444_k11", "kind": "resblock", "frames": 2444, "stage": 1, "k": 11},
        # GPT-2 serving: one token at a 512-token cache, and the 512-token prompt that filled it
        {"name": "gpt2_decode_p512", "kind": "gpt2", "tokens": 1, "pos": 512},
        {"name": "gpt2_prefill_t512", "kind": "gpt2", "tokens": 512, "pos": 0},
        # Qwen3 serving: a decode step after a 10 s clip's prompt, that prompt (400 audio rows + 16 ids), and the
        # largest prefill chunk of the transcribe loop
        {"name": "qwen3_decode_p416", "kind": "qwen3", "tokens": 1, "pos": 416},
        {"name": "qwen3_prefill_t416", "kind": "qwen3", "tokens": 416, "pos": 0},
        {"name": "qwen3_prefill_t2048", "kind": "qwen3", "tokens": 2048, "pos": 0},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng) -> dict:
    kind = rng.choice(["mlp", "albert", "lstm", "decoder", "resblock", "resblock", "gpt2", "gpt2", "qwen3", "qwen3"])
    if kind == "mlp":
        return {"kind": kind, "batch": _log(rng, 1, 512)}
    if kind == "albert":
        return {"kind": kind, "tokens": rng.randint(8, 510)}
    if kind == "lstm":
        return {"kind": kind, "steps": _log(rng, 12, 2444)}
    if kind == "decoder":
        return {"kind": kind, "frames": _log(rng, 40, 2444), "up": rng.random() < 0.3}
    if kind == "resblock":
        return {"kind": kind, "frames": _log(rng, 40, 2444), "stage": rng.randint(0, 1), "k": rng.choice([3, 7, 11])}
    if kind == "gpt2":
        if rng.random() < 0.4:
            return {"kind": kind, "tokens": 1, "pos": rng.randint(1, 1023)}
        t = _log(rng, 2, 1024)
        return {"kind": kind, "tokens": t, "pos": rng.choice([0, rng.randint(0, 1024 - t)])}
    if rng.random() < 0.4:
        return {"kind": kind, "tokens": 1, "pos": _log(rng, 16, 4096)}
    return {"kind": kind, "tokens": _log(rng, 2, 2048), "pos": rng.choice([0, rng.randint(0, 2048)])}


# ---- inputs and weights (made on the GPU from the seed alone) ---------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(g, *shape) -> torch.Tensor:
    return torch.randn(*shape, device="cuda", generator=g)


def _host(g, shape, scale=1.0, shift=0.0) -> np.ndarray:
    return (_randn(g, *shape) * scale + shift).cpu().numpy()


def _kokoro_sd(g, prefixes: tuple) -> dict:
    """Random weights, distributed as kokoro_weights.random_weights', of the modules named by `prefixes`, and of the
    two that give the style banks of both model roots their first column block."""
    keep = prefixes + ("predictor.text_encoder.lstms.1.fc", "decoder.encode.norm1.fc")
    shapes = KW.param_shapes()
    sd = {}
    for k in sorted(shapes):
        if not k.startswith(keep):
            continue
        shape = shapes[k]
        z = _host(g, shape)
        if k.endswith(("LayerNorm.weight", "layer_norm.weight", ".gamma")):
            z = 1 + 0.1 * z
        elif k.endswith(("LayerNorm.bias", "layer_norm.bias", ".beta")):
            z = 0.1 * z
        elif ".alpha" in k:
            z = np.exp(0.1 * z)
        elif "embeddings" not in k:
            if k.endswith(".bias"):
                shape = shapes[k[:-5] + ".weight"]
            elif "bias_ih" in k or "bias_hh" in k:
                shape = shapes[k.replace("bias_", "weight_")]
            fan = shape[2] if ".pool." in k else int(np.prod(shape[1:]))
            z = z / math.sqrt(fan)
        sd[k] = z.astype(np.float32)
    return sd


def _resblock_name(case) -> str:
    return "decoder.generator.resblocks.%d" % (3 * case["stage"] + (3, 7, 11).index(case["k"]))


def _kokoro_inputs(case, seed):
    """(state dict, input of the block as a float32 device tensor or ids, style vector) of a Kokoro block."""
    g = _gen(seed)
    kind = case["kind"]
    if kind == "albert":
        sd = _kokoro_sd(g, ("bert.",))
        ids = torch.randint(0, KW.N_TOKENS, (case["tokens"],), device="cuda", generator=g)
        ids[0] = ids[-1] = 0
        return sd, ids, None
    if kind == "lstm":
        sd = _kokoro_sd(g, ("predictor.shared",))
        return sd, _randn(g, case["steps"], 640), None
    style = _randn(g, 1, STYLE)
    if kind == "decoder":
        sd = _kokoro_sd(g, ("decoder.decode.%d." % (3 if case["up"] else 0),))
        x = torch.zeros(case["frames"], 1104, device="cuda")  # 1090 channels, padded to a multiple of 16
        x[:, :1090] = _randn(g, case["frames"], 1090)
        return sd, x, style
    sd = _kokoro_sd(g, (_resblock_name(case) + ".",))
    length, ch = (20 * case["frames"], 256) if case["stage"] == 0 else (120 * case["frames"] + 1, 128)
    return sd, _randn(g, length, ch), style


def _gpt2_sd(g) -> dict:
    sd = {}
    for k, shape in sorted(G.param_shapes().items()):
        norm = k.endswith(("ln_1.weight", "ln_2.weight", "ln_f.weight"))
        sd[k] = _host(g, shape, 0.02, 1.0 if norm else 0.0)
    return sd


def _gpt2_inputs(case, seed):
    """(state dict, ids, K and V rows 0 .. pos-1 of every layer): the rows as an earlier prompt left them."""
    g = _gen(seed)
    sd = _gpt2_sd(g)
    ids = torch.randint(0, G.VOCAB, (case["tokens"],), device="cuda", generator=g)
    past = [(0.5 * _randn(g, case["pos"], G.D), 0.5 * _randn(g, case["pos"], G.D)) for _ in range(G.N_LAYER)]
    return sd, ids, past


def _qwen_inputs(case, seed):
    """(state dict as float16 device tensors, ids, audio rows, K / V cache [layers, 2, P, kvh * 128])."""
    c, g = QWEN, _gen(seed)
    from lokinfer_amd import f16_gpu as F
    from lokinfer_amd import qwen3 as Q

    sd = {}
    for k, shape in sorted(Q.param_shapes(c).items()):
        sd[k] = (_randn(g, *shape) * 0.02 + (1.0 if k.endswith(".g") else 0.0)).half()
    t, pos = case["tokens"], case["pos"]
    ids = torch.randint(0, F.PAD_ID, (t,), device="cuda", generator=g)
    n_audio = max(0, t - 16) if t > 1 and pos == 0 else 0  # the prompt layout: 9 prefix ids, the audio run, the rest
    if n_audio:
        ids[Q.AUDIO_START:Q.AUDIO_START + n_audio] = F.PAD_ID
    audio = _randn(g, max(1, n_audio), c.d).half()
    kv = torch.zeros(c.layers, 2, pos + t, c.dk, dtype=torch.float16, device="cuda")
    kv[:, :, :pos] = _randn(g, c.layers, 2, pos, c.dk).half()
    return sd, ids, audio, kv


def prepare(case: dict, seed: int) -> dict:
    kind = case["kind"]
    if kind == "mlp":
        x, w1, b1, w2, b2 = (lk.Tensor(t) for t in _mlp_inputs(case, seed))
        model = lk.compile(lambda a: lk.ops.gemm_bias_f32_gpu(lk.ops.gemm_bias_relu_f32_gpu(a, w1, b1), w2, b2),
                           inputs=[x])
        model.run_inplace(x)
        return {"model": model, "args": (x,)}
    if kind == "gpt2":
        sd, ids, past = _gpt2_inputs(case, seed)
        m = G.Gpt2Generator(sd, chunk_graph=True)
        for (kc, vc), (k, v) in zip(m.caches, past):
            kc.t[:case["pos"]] = k
            vc.t[:case["pos"]] = v
        ids = lk.Tensor(ids)
        m.run(ids, case["pos"])
        return {"gpt2": m, "ids": ids, "pos": case["pos"]}
    if kind == "qwen3":
        sd, ids, audio, kv = _qwen_inputs(case, seed)
        m = Qwen3Lm({k: v.cpu().numpy() for k, v in sd.items()}, QWEN)
        st = {"qwen3": m, "ids": lk.Tensor(ids), "audio": lk.Tensor(audio), "kv": lk.Tensor(kv), "pos": case["pos"]}
        m.run(st["ids"], st["audio"], st["pos"], st["kv"])
        return st
    sd, x, style = _kokoro_inputs(case, seed)
    m = KokoroGpu(sd)
    x = lk.Tensor(x)
    if kind == "albert":
        fn = m.albert
    elif kind == "lstm":
        fn = lambda a: m.lstm(a, "predictor.shared")  # noqa: E731
    else:
        w, b, offs = m.banks["decoder"]
        bank = (lk.ops.gemv4_f32_gpu(lk.Tensor(style), w, b), offs)  # once per style vector
        if kind == "decoder":
            p, co = ("decoder.decode.3", 512) if case["up"] else ("decoder.decode.0", 1024)
            fn = lambda a: m.resblk(a, bank, p, 1090, co, case["up"])  # noqa: E731
        else:
            fn = lambda a: m.resblock1(a, bank, _resblock_name(case), case["k"])  # noqa: E731
    return {"model": lk.capture(fn, inputs=[x], by_ref=(0,)), "args": (x,)}


def run(state: dict):
    if "model" in state:
        return state["model"].run_inplace(*state["args"]).t
    if "gpt2" in state:
        m = state["gpt2"]
        logits, _ = m.run(state["ids"], state["pos"])
        return {"logits": logits.t, "k": [k.t for k, _ in m.caches], "v": [v.t for _, v in m.caches]}
    logits, _ = state["qwen3"].run(state["ids"], state["audio"], state["pos"], state["kv"])
    return {"logits": logits.t, "kv": state["kv"].t}


def _mlp_inputs(case, seed):
    g = _gen(seed)
    return (_randn(g, case["batch"], 784), _randn(g, 784, 128) / 28, _randn(g, 128) / 28,
            _randn(g, 128, 10) / math.sqrt(128), _randn(g, 10) / math.sqrt(128))


# ---- what a pass cannot do without --------------------------------------------------------------------------------

def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "mlp":
        b, w = case["batch"], 784 * 128 + 128 * 10
        return {"bytes": 4 * (w + 138 + b * 794), "flops": 2 * b * w}
    if kind == "albert":
        t, w = case["tokens"], 768 * 2304 + 768 * 768 + 2 * 768 * 2048
        return {"bytes": 4 * (w + 128 * 768 + t * (2 * 128 + 768)), "flops": 12 * (2 * t * w + 4 * t * t * 768)
                + 2 * t * 128 * 768}
    if kind == "lstm":
        t, w = case["steps"], 640 * 2048 + 256 * 2048
        return {"bytes": 4 * (w + t * (640 + 512)), "flops": 2 * t * w}
    if kind == "decoder":
        f, co = case["frames"], 512 if case["up"] else 1024
        lo = 2 * f if case["up"] else f
        w = 1090 * co * 3 + co * co * 3 + 1090 * co
        return {"bytes": 4 * (w + f * 1090 + lo * co), "flops": 2 * lo * w}
    if kind == "resblock":
        n, ch = (20 * case["frames"], 256) if case["stage"] == 0 else (120 * case["frames"] + 1, 128)
        w = 6 * ch * ch * case["k"]
        return {"bytes": 4 * (w + 2 * n * ch), "flops": 2 * n * w}
    t, pos = case["tokens"], case["pos"]
    pairs = t * pos + t * (t + 1) // 2  # (query, key) pairs of causal attention
    if kind == "gpt2":
        w = G.N_LAYER * (G.D * 3 * G.D + G.D * G.D + 2 * G.D * G.FFN)
        head = G.VOCAB * G.D
        return {"bytes": 4 * (w + head + 2 * G.N_LAYER * (pos + t) * G.D + G.VOCAB + 2 * t * G.D),
                "flops": 2 * t * w + 2 * head + 4 * G.N_LAYER * pairs * G.D}
    c = QWEN
    w = c.layers * (c.d * (c.dq + 2 * c.dk) + c.dq * c.d + 3 * c.d * c.ffn)
    head = c.vocab * c.d
    return {"bytes": 2 * (w + head + 2 * c.layers * (pos + t) * c.dk + t * c.d) + 4 * c.vocab,
            "flops": 2 * t * w + 2 * head + 4 * c.layers * pairs * c.dq}


# Largest relative differences (2-norm) between correct implementations at the same precision: four to five times the
# largest measured against float64 (mlp 4e-7, albert 2.6e-7, lstm 3.2e-7, decoder 9.6e-7, resblock 2.5e-6, gpt2 6.3e-7;
# qwen3, whose float64 run has no f16 roundings, 2.4e-3).
TOLERANCE = {"mlp": 2e-6, "albert": 1.5e-6, "lstm": 1.5e-6, "decoder": 4e-6, "resblock": 1e-5, "gpt2": 3e-6,
             "qwen3": 1e-2}


def tolerance(case: dict):
    return {"rel": TOLERANCE[case["kind"]]}


# ---- the same results in float64 (plain torch) --------------------------------------------------------------------

def _ln(x, w, b, eps):
    return torch.nn.functional.layer_norm(x, (x.shape[-1],), w, b, eps)


def _attend(q, k, v, pos):
    """Causal attention of q [H, T, d] at positions pos.. over k, v [H, pos + T, d], in blocks of queries."""
    t, out = q.shape[1], []
    keys = torch.arange(k.shape[1], device=q.device)
    for i in range(0, t, 256):
        s = q[:, i:i + 256] @ k.transpose(1, 2).contiguous() / math.sqrt(q.shape[2])
        rows = pos + i + torch.arange(s.shape[1], device=q.device)
        s = s.masked_fill(keys[None, None] > rows[None, :, None], -math.inf)
        out.append(torch.softmax(s, -1) @ v.contiguous())
    return torch.cat(out, 1)


def _conv(x, w, b, dilation=1):
    """Same-length conv1d of x [L, Ci] with w [Co, Ci, K]."""
    k = w.shape[2]
    pad = dilation * (k - 1) // 2
    xp = torch.nn.functional.pad(x, (0, 0, pad, pad))
    y = sum(xp[j * dilation:j * dilation + x.shape[0]] @ w[:, :, j].T.contiguous() for j in range(k))
    return y if b is None else y + b


def _adain(x, w, p, style):
    h = w[p + ".weight"] @ style + w[p + ".bias"]
    c = x.shape[1]
    return (1 + h[:c]) * (x - x.mean(0)) / torch.sqrt(x.var(0, unbiased=False) + 1e-5) + h[c:]


@torch.no_grad()
def exact(case: dict, seed: int):
    kind = case["kind"]
    f = torch.nn.functional
    if kind == "mlp":
        x, w1, b1, w2, b2 = (t.double() for t in _mlp_inputs(case, seed))
        return torch.relu(x @ w1 + b1) @ w2 + b2
    if kind == "gpt2":
        return _exact_gpt2(case, seed)
    if kind == "qwen3":
        return _exact_qwen3(case, seed)
    sd, x, style = _kokoro_inputs(case, seed)
    w = {k: torch.from_numpy(v).cuda().double() for k, v in sd.items()}
    if kind == "albert":
        e, t = "bert.embeddings.", case["tokens"]
        h = w[e + "word_embeddings.weight"][x] + w[e + "position_embeddings.weight"][:t]
        h = _ln(h + w[e + "token_type_embeddings.weight"][0], w[e + "LayerNorm.weight"], w[e + "LayerNorm.bias"], 1e-12)
        lin = lambda a, p: a @ w[p + ".weight"].T + w[p + ".bias"]  # noqa: E731
        h = lin(h, "bert.encoder.embedding_hidden_mapping_in")
        p = "bert.encoder.albert_layer_groups.0.albert_layers.0."
        for _ in range(12):
            q, k, v = (lin(h, p + "attention." + n).view(t, 12, 64).transpose(0, 1).contiguous()
                       for n in ("query", "key", "value"))
            a = (torch.softmax(q @ k.transpose(1, 2).contiguous() / 8, -1) @ v).transpose(0, 1).reshape(t, 768)
            h = _ln(h + lin(a, p + "attention.dense"), w[p + "attention.LayerNorm.weight"],
                    w[p + "attention.LayerNorm.bias"], 1e-12)
            m = lin(f.gelu(lin(h, p + "ffn"), approximate="tanh"), p + "ffn_output")
            h = _ln(m + h, w[p + "full_layer_layer_norm.weight"], w[p + "full_layer_layer_norm.bias"], 1e-12)
        return h
    if kind == "lstm":
        net = torch.nn.LSTM(640, 256, bidirectional=True).double()
        net.load_state_dict({k[len("predictor.shared."):]: v.cpu() for k, v in w.items()
                             if k.startswith("predictor.shared.")})
        return net(x.cpu().double()[:, None])[0][:, 0]
    style = style[0].double()
    if kind == "decoder":
        p = "decoder.decode.3" if case["up"] else "decoder.decode.0"
        x = x[:, :1090].double()
        r = f.leaky_relu(_adain(x, w, p + ".norm1.fc", style), 0.2)
        if case["up"]:
            r = f.conv_transpose1d(r.T[None].cpu(), w[p + ".pool.weight"].cpu(), w[p + ".pool.bias"].cpu(), stride=2,
                                   padding=1, output_padding=1, groups=1090)[0].T.cuda().contiguous()
            x = x.repeat_interleave(2, 0)
        r = _conv(r, w[p + ".conv1.weight"], w[p + ".conv1.bias"])
        r = f.leaky_relu(_adain(r, w, p + ".norm2.fc", style), 0.2)
        r = _conv(r, w[p + ".conv2.weight"], w[p + ".conv2.bias"])
        return (r + _conv(x, w[p + ".conv1x1.weight"], None)) / math.sqrt(2)
    p, x = _resblock_name(case), x.double()
    for j, d in enumerate((1, 3, 5)):
        h = x
        for a, c, dil in (("1", "convs1", d), ("2", "convs2", 1)):
            al = w[f"{p}.alpha{a}.{j}"].reshape(-1)
            h = _adain(h, w, f"{p}.adain{a}.{j}.fc", style)
            h = _conv(h + torch.sin(al * h) ** 2 / al, w[f"{p}.{c}.{j}.weight"], w[f"{p}.{c}.{j}.bias"], dil)
        x = h + x
    return x


def _exact_gpt2(case, seed):
    sd, ids, past = _gpt2_inputs(case, seed)
    w = {k[len("transformer."):]: torch.from_numpy(v).cuda().double() for k, v in sd.items()}
    t, pos = case["tokens"], case["pos"]
    h = w["wte.weight"][ids] + w["wpe.weight"][pos:pos + t]
    ks, vs = [], []
    heads = lambda a: a.view(-1, G.HEADS, 64).transpose(0, 1).contiguous()  # noqa: E731
    for i, (kp, vp) in enumerate(past):
        p = "h.%d." % i
        lin = lambda a, n: a @ w[p + n + ".weight"] + w[p + n + ".bias"]  # noqa: E731, B023
        q, k, v = lin(_ln(h, w[p + "ln_1.weight"], w[p + "ln_1.bias"], G.LN_EPS), "attn.c_attn").split(G.D, 1)
        k, v = torch.cat([kp.double(), k]), torch.cat([vp.double(), v])
        a = _attend(heads(q), heads(k), heads(v), pos).transpose(0, 1).reshape(t, G.D)
        h = h + lin(a, "attn.c_proj")
        m = lin(_ln(h, w[p + "ln_2.weight"], w[p + "ln_2.bias"], G.LN_EPS), "mlp.c_fc")
        h = h + lin(torch.nn.functional.gelu(m, approximate="tanh"), "mlp.c_proj")
        rest = (0, 0, 0, G.N_POS - pos - t)
        ks.append(torch.nn.functional.pad(k, rest))
        vs.append(torch.nn.functional.pad(v, rest))
    logits = _ln(h[-1:], w["ln_f.weight"], w["ln_f.bias"], G.LN_EPS) @ w["wte.weight"].T
    return {"logits": logits, "k": ks, "v": vs}


def _exact_qwen3(case, seed):
    from lokinfer_amd import f16_gpu as F

    c = QWEN
    sd, ids, audio, kv = _qwen_inputs(case, seed)
    t, pos = case["tokens"], case["pos"]
    kv = kv.double()
    h = sd["embed"][ids].double()
    pads = ids == F.PAD_ID
    h[pads] = audio[:int(pads.sum())].double()
    invf = (1.0 / c.theta ** (torch.arange(64, device="cuda").double() / 64)).float()
    ang = ((pos + torch.arange(t, device="cuda")).float()[:, None] * invf[None]).double()
    cos, sin = torch.cos(ang)[:, None], torch.sin(ang)[:, None]
    rms = lambda x, g: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + c.eps) * g.double()  # noqa: E731

    def rope(x):  # [T, heads, 128]
        lo, hi = x[..., :64], x[..., 64:]
        return torch.cat([lo * cos - hi * sin, hi * cos + lo * sin], -1)

    for i in range(c.layers):
        w = {k[len("lm.%d." % i):]: v for k, v in sd.items() if k.startswith("lm.%d." % i)}
        lin = lambda a, n: a @ w[n + ".w"].double()  # noqa: E731, B023
        a = rms(h, w["ln1.g"])
        q = rope(rms(lin(a, "q").view(t, c.qh, c.hd), w["qn.g"]))
        kv[i, 0, pos:] = rope(rms(lin(a, "k").view(t, c.kvh, c.hd), w["kn.g"])).reshape(t, c.dk)
        kv[i, 1, pos:] = lin(a, "v")
        k, v = (kv[i, j].view(-1, c.kvh, c.hd).transpose(0, 1).repeat_interleave(c.qh // c.kvh, 0) for j in (0, 1))
        att = _attend(q.transpose(0, 1).contiguous(), k, v, pos).transpose(0, 1).reshape(t, c.dq)
        h = h + lin(att, "o")
        a = rms(h, w["ln2.g"])
        h = h + lin(torch.nn.functional.silu(lin(a, "gate")) * lin(a, "up"), "down")
    return {"logits": rms(h[-1:], sd["lm.norm.g"]) @ sd["embed"].double().T, "kv": kv}
