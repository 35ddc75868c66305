"""The workloads this framework's speed is measured on, through its public entry points.

The framework decodes speech tokens: a text (phones, with BERT features) and a prompt (codes of a
reference recording) go through a 24-layer decoder (prefill, then one token per step), and a BERT
encoder makes the features. So the cases are: generation for one caller, for a full batch and for
a large batch stepped by a scheduler; the prefill of one sentence and of the longest batch; the
bit-exact mode; the BERT encoder on one sentence, on a ragged batch of paragraphs and with F32
weights; and single kernels of the decoder at the shapes in which they carry most of the work.
The weights are synthetic, in files of the exporter's format written once to the temporary
folder; a program keeps its loaded models, so they are loaded once per process.

`listed` names the cases, `draw` makes more of the same ranges, `prepare` makes what a program
holds before a call, `run` is one call, `work` counts the bytes and operations it cannot do
without, `tolerance` is what another correct implementation may differ by, and `exact` computes
the result in 64 bits.
"""
import math
import os
import struct
import sys
import tempfile

import numpy as np
import torch

PACKAGE = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gsv.cpp_amd")
if PACKAGE not in sys.path:
    sys.path.insert(0, PACKAGE)

import gsvk  # noqa: E402
import synth_model  # noqa: E402

D, NH, HD, FFN, NL, V, EOS = 512, 16, 32, 2048, 24, 1025, 1024
PHONES, BERT_DIM = 732, 1024
BD, BH, BF, BL, BV = 1024, 16, 4096, 22, 21128   # the BERT encoder: width, heads, FFN, layers, vocabulary
PROJ = {"qkv": (3 * D, D), "out": (D, D), "ffn1": (FFN, D), "ffn2": (D, FFN)}
SCALE = 1.0 / math.sqrt(HD)


# ---- the cases ----------------------------------------------------------------------------

def listed():
    return [
        # one caller, one sentence, decoded token by token: the latency that a listener waits for
        {"name": "generate_b1", "kind": "generate", "B": 1, "lo": 128, "hi": 128, "prompt": 64, "steps": 48,
         "bert": True, "exact": False},
        # a server's batch of requests of mixed length: the benchmark's headline shape
        {"name": "generate_b16", "kind": "generate", "B": 16, "lo": 36, "hi": 336, "prompt": 64, "steps": 64,
         "bert": True, "exact": False},
        # a scheduler that drives a large batch step by step and reads every step's logits
        {"name": "steps_b64", "kind": "steps", "B": 64, "lo": 36, "hi": 336, "prompt": 64, "steps": 32,
         "bert": True},
        # the first token of one short sentence: a prefill of about 100 rows
        {"name": "prefill_b1", "kind": "prefill", "B": 1, "lo": 45, "hi": 45, "prompt": 64, "bert": True},
        # the longest prefill of the benchmark: 16 requests padded to 1024 rows, 256 prompt codes
        {"name": "prefill_b16_s1024", "kind": "prefill", "B": 16, "lo": 256, "hi": 768, "prompt": 256, "bert": True},
        # callers that need the CPU reference's tokens bit for bit
        {"name": "generate_exact_b2", "kind": "generate", "B": 2, "lo": 60, "hi": 130, "prompt": 64, "steps": 12,
         "bert": True, "exact": True},
        # text features of one sentence, F16 weights (the file that the engine loads)
        {"name": "bert_f16_b1", "kind": "bert", "type": "f16", "B": 1, "lo": 64, "hi": 64},
        # text features of a batch of ragged paragraphs
        {"name": "bert_f16_b16", "kind": "bert", "type": "f16", "B": 16, "lo": 5, "hi": 301},
        # the exporter's default F32 weights
        {"name": "bert_f32_b8", "kind": "bert", "type": "f32", "B": 8, "lo": 33, "hi": 97},
        # decode attention of one layer at batch 64 over unequal rows
        {"name": "attn_decode_b64", "kind": "attn_decode", "B": 64, "lo": 256, "hi": 2048},
        # prefill attention of one layer at the mixed-length batch's 16 x 400 rows
        {"name": "attn_prefill_b16", "kind": "attn_prefill", "B": 16, "lo": 36, "hi": 336, "prompt": 64},
        # one projection of a layer over the rows of such a prefill
        {"name": "proj_ffn2_6411", "kind": "proj", "proj": "ffn2", "rows": 6411},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["generate", "generate", "steps", "prefill", "prefill", "exact", "bert", "bert",
                       "attn_decode", "attn_prefill", "proj"])
    if kind in ("generate", "exact"):
        ex = kind == "exact"
        B = _log(rng, 1, 3 if ex else 32)
        hi = _log(rng, 20, 130 if ex else 336)
        return {"kind": "generate", "B": B, "lo": rng.randint(5, hi), "hi": hi, "prompt": rng.randint(16, 64 if ex else 100),
                "steps": rng.randint(4, 12) if ex else rng.randint(16, 64), "bert": rng.random() < 0.7, "exact": ex}
    if kind == "steps":
        hi = _log(rng, 20, 336)
        return {"kind": "steps", "B": rng.randint(33, 64), "lo": rng.randint(5, hi), "hi": hi,
                "prompt": rng.randint(16, 64), "steps": rng.randint(8, 32), "bert": rng.random() < 0.7}
    if kind == "prefill":
        hi = _log(rng, 10, 768)
        return {"kind": "prefill", "B": _log(rng, 1, 16), "lo": rng.randint(5, hi), "hi": hi,
                "prompt": rng.randint(8, 256), "bert": rng.random() < 0.7}
    if kind == "bert":
        f32 = rng.random() < 0.3
        hi = _log(rng, 8, 128 if f32 else 512)
        return {"kind": "bert", "type": "f32" if f32 else "f16", "B": _log(rng, 1, 8 if f32 else 16),
                "lo": rng.randint(3, hi), "hi": hi}
    if kind == "attn_decode":
        hi = _log(rng, 100, 2048)
        return {"kind": "attn_decode", "B": _log(rng, 1, 64), "lo": rng.randint(30, hi), "hi": hi}
    if kind == "attn_prefill":
        hi = _log(rng, 30, 600)
        return {"kind": "attn_prefill", "B": _log(rng, 2, 16), "lo": rng.randint(5, hi), "hi": hi,
                "prompt": rng.randint(16, 256)}
    return {"kind": "proj", "proj": rng.choice(sorted(PROJ)), "rows": _log(rng, 64, 16384)}


# ---- what a program holds ------------------------------------------------------------------

_models = {}


def _model_path(key):
    """The synthetic weights' file, written on first use."""
    if key == "ar":
        d = os.path.join(tempfile.gettempdir(), "gsv_perf_models_%d" % os.getuid())
        return synth_model.cached_model(d, n_layer=NL)
    d = os.path.join(tempfile.gettempdir(), "gsv_perf_models_%d" % os.getuid())
    os.makedirs(d, exist_ok=True)
    path = os.path.join(d, "bert_%s.gguf" % key)
    if not os.path.exists(path):
        synth_model.write_bert_model(path, n_layer=BL, layers_used=BL, vocab=BV, wtype=key)
    return path


def _model(key):
    if key not in _models:
        _models[key] = gsvk.Model(_model_path("ar")) if key == "ar" else gsvk.Bert(_model_path(key))
    return _models[key]


def _lens(case):
    """Lengths of the case's sequences, uniform over its range; the first is the longest allowed."""
    n = np.random.Generator(np.random.PCG64(case["lo"])).integers(case["lo"], case["hi"] + 1, case["B"])
    n[0] = case["hi"]
    return n


def _requests(case, seed):
    rng = np.random.Generator(np.random.PCG64([seed, 1]))
    reqs = synth_model.synth_requests(seed, case["B"], case["prompt"], _lens(case), bert=case["bert"])
    return reqs, rng.integers(0, EOS, (case.get("steps", 1), case["B"])).astype(np.int32)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _q8(x):
    """Q8_0 of rows [m][k], by the rule of the x86 quantiser: quants int8, scales that fp16 holds."""
    b = x.reshape(x.shape[0], -1, 32)
    amax = b.abs().amax(-1)
    inv = torch.where(amax > 0, 127.0 / amax.clamp(min=1e-30), torch.zeros_like(amax))
    q = torch.round(b * inv[..., None]).clamp(-127, 127).to(torch.int8)
    return q.reshape(x.shape).contiguous(), (amax / 127.0).half()


def _attn_decode_inputs(case, seed):
    lens = _lens(case)
    g, B, ls = _gen(seed), case["B"], case["hi"] + 1
    q = torch.randn(B, NH, HD, generator=g, device="cuda")
    k = torch.randn(B, NH, ls, HD, generator=g, device="cuda", dtype=torch.float16)
    v = torch.randn(B, NH, ls, HD, generator=g, device="cuda", dtype=torch.float16)
    end = torch.full((B,), case["hi"], device="cuda", dtype=torch.int32)
    begin = end - torch.from_numpy(lens.astype(np.int32)).cuda()   # left padding, as the decoder's cache has it
    return q, k, v, begin, end


def _attn_prefill_inputs(case, seed):
    lens = _lens(case)
    S = case["hi"] + case["prompt"]
    qkv = torch.randn(case["B"], S, 3 * D, generator=_gen(seed), device="cuda")
    return qkv, torch.from_numpy((case["hi"] - lens).astype(np.int32)).cuda()


def _proj_inputs(case, seed):
    n, k = PROJ[case["proj"]]
    g = _gen(seed)
    wq, wd = _q8(0.02 * torch.randn(n, k, generator=g, device="cuda"))
    x = torch.randn(case["rows"], k, generator=g, device="cuda")
    xq, xd = _q8(x.relu() if case["proj"] == "ffn2" else x)
    return wq, wd, xq, xd.float(), 0.02 * torch.randn(n, generator=g, device="cuda")


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("generate", "steps", "prefill"):
        reqs, toks = _requests(case, seed)
        return {"case": case, "model": _model("ar"), "reqs": reqs, "toks": toks, "seed": seed}
    if kind == "bert":
        rng = np.random.Generator(np.random.PCG64([seed, 4]))
        seqs = [rng.integers(0, BV, n).astype(np.int32) for n in _lens(case)]
        return {"case": case, "model": _model(case["type"]), "seqs": seqs}
    s = {"case": case}
    if kind == "attn_decode":
        s["in"] = _attn_decode_inputs(case, seed)
        ws = gsvk.attn_workspace_bytes(case["B"], NH, case["hi"])
        s["ws"] = torch.zeros(max(ws, 16), dtype=torch.uint8, device="cuda")
        s["out"] = torch.empty(case["B"], D, device="cuda")
    elif kind == "attn_prefill":
        s["in"] = _attn_prefill_inputs(case, seed)
        m = s["in"][0].shape[:2]
        s["out"] = torch.empty(*m, D, device="cuda")
        s["oq"] = torch.empty(*m, D, device="cuda", dtype=torch.int8)
        s["od"] = torch.empty(*m, D // 32, device="cuda")
    else:
        s["in"] = _proj_inputs(case, seed)
        s["out"] = torch.empty(case["rows"], PROJ[case["proj"]][0], device="cuda")
    return s


# ---- one call ------------------------------------------------------------------------------

def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "generate":
        # sequence 0 follows given tokens, so that its probabilities can be compared; the others
        # sample. (The whole vocabulary is kept: a top-k cut flips at ties.)
        m = s["model"]
        if case["exact"]:
            m.set_exact(True)
        try:
            r = m.generate(s["reqs"], sampler=(0, 1.0, 1.0, 1.35), max_steps=case["steps"], oracle=s["toks"][:, 0],
                           seeds=[s["seed"] + b + 1 for b in range(case["B"])], flags=gsvk.GSVK_GEN_EOS_MASK_ALL,
                           want_probs0=True)
        finally:
            if case["exact"]:
                m.set_exact(False)
        return {"probs": r["probs0"], "tokens": r["tokens"]} if case["exact"] else {"probs": r["probs0"]}
    if kind == "steps":
        m = s["model"]
        gsvk.check(gsvk.lib().gsvk_kv_alloc(m.h, case["B"], case["hi"] + case["prompt"] + case["steps"] + 8), "kv_alloc")
        out = [m.prefill(s["reqs"])[0]]
        out += [m.decode_step(t) for t in s["toks"]]
        return {"logits": np.stack(out)}
    if kind == "prefill":
        return {"logits": s["model"].first_logits(s["reqs"])}
    if kind == "bert":
        return {"features": s["model"].encode(s["seqs"])}
    if kind == "attn_decode":
        q, k, v, begin, end = s["in"]
        gsvk.op_attn_decode(q, k, v, begin, end, case["hi"], SCALE, s["out"], ws=s["ws"])
        return {"out": s["out"]}
    if kind == "attn_prefill":
        qkv, pad = s["in"]
        gsvk.op_attn_prefill(qkv, case["hi"], pad, NH, SCALE, s["out"], s["oq"], s["od"])
        return {"out": s["out"], "oq": s["oq"], "od": s["od"]}
    wq, wd, xq, xd, bias = s["in"]
    n, k = PROJ[case["proj"]]
    gsvk.op_q8_gemm(wq, wd.view(torch.int16), n, k, xq, xd, case["rows"], bias, 1 if case["proj"] == "ffn1" else 0,
                    s["out"])
    return {"out": s["out"]}


# ---- what a call cannot do without ---------------------------------------------------------

W_LAYER = sum(n * k for n, k in PROJ.values())          # weights of a layer
W_BYTES = NL * (W_LAYER // 32 * 34 + (3 * D + D + FFN + D + 4 * D) * 4) + V * D * 2


def work(case):
    kind, B = case["kind"], case.get("B", 1)
    n = _lens(case).astype(float) if "lo" in case else np.zeros(1)
    T, TT = float(n.mean()), float((n * n).mean())   # of the lengths and of their squares
    if kind in ("generate", "steps", "prefill"):
        P, n = case["prompt"], case.get("steps", 0)
        rows = B * (T + P)
        pairs = B * (TT + P * T + P * (P + 1) / 2)
        flops = NL * (2 * W_LAYER * rows + 4 * D * pairs) + 2 * B * V * D
        flops += 2 * D * BERT_DIM * B * T if case["bert"] else 0
        read = W_BYTES + (B * T * BERT_DIM * 4 if case["bert"] else 0) + NL * rows * 4 * D
        keys = B * (T + P + n / 2)   # of a step, on average
        return {"bytes": read + n * (W_BYTES + NL * (keys + B) * 4 * D),
                "flops": flops + n * (NL * (2 * W_LAYER * B + 4 * D * keys) + 2 * B * V * D)}
    if kind == "bert":
        w = BL * (4 * BD * BD + 2 * BD * BF)
        rows, pairs = B * T, BL * B * TT
        return {"bytes": w * (2 if case["type"] == "f16" else 4) + 2 * rows * BD * 4,
                "flops": 2 * w * rows + 4 * BD * pairs}
    if kind == "attn_decode":
        return {"bytes": B * T * NH * HD * 4 + B * D * 8, "flops": 4 * D * B * T}
    if kind == "attn_prefill":
        S, P = case["hi"] + case["prompt"], case["prompt"]
        return {"bytes": B * S * D * (12 + 4 + 1 + 0.125), "flops": 4 * D * B * (TT + P * T + P * (P + 1) / 2)}
    n, k = PROJ[case["proj"]]
    m = case["rows"]
    return {"bytes": n * (k // 32) * 34 + m * (k // 32) * 36 + n * m * 4, "flops": 2 * n * k * m}


# ---- how far another correct implementation may be off -------------------------------------

def tolerance(case):
    kind = case["kind"]
    if kind == "generate":
        # bit-exact mode: the same bits. Otherwise a last-bit difference in one layer flips a
        # quantised activation by a whole step (1/127), which the layers after it spread: the
        # decode paths, which differ in the order of their sums, are up to 0.0051 apart
        return "exact" if case["exact"] else {"rel": 0.02, "max": 0.09}
    if kind in ("steps", "prefill"):
        # logits of the default and of the exact mode are 0.011 (at most 0.05) apart
        return {"rel": 0.03, "max": 0.2}
    if kind == "bert":
        # activations rounded to fp16 between the layers (F16 weights: 7.7e-4 from 64 bits),
        # 32-bit sums otherwise (8.3e-7)
        return {"rel": 2e-3 if case["type"] == "f16" else 4e-6}
    if kind == "attn_prefill":
        return {"rel": 2e-6, "max": 0.01, "differ": 1e-3}   # (oq, od: a quant or scale moves by one step at a tie)
    return {"rel": 2e-6}


# ---- the results in 64 bits ----------------------------------------------------------------

def _gguf(path):
    """The tensors of a GGUF file as float64 on the GPU, by name, read on demand."""
    size = {0: (1, 4), 1: (1, 2), 8: (32, 34)}
    with open(path, "rb") as f:
        head = f.read(1 << 20)
    at = 4 + 4
    nt, nkv = struct.unpack_from("<QQ", head, at)
    at += 16

    def text():
        nonlocal at
        n = struct.unpack_from("<Q", head, at)[0]
        at += 8 + n
        return head[at - n:at].decode()

    for _ in range(nkv):
        text()
        t = struct.unpack_from("<I", head, at)[0]
        at += 4
        if t == 8:
            text()
        else:
            at += 4
    infos = {}
    for _ in range(nt):
        name = text()
        nd = struct.unpack_from("<I", head, at)[0]
        ne = struct.unpack_from("<%dQ" % nd, head, at + 4)
        t, off = struct.unpack_from("<IQ", head, at + 4 + 8 * nd)
        at += 4 + 8 * nd + 12
        infos[name] = (tuple(reversed(ne)), t, off)
    base = (at + 31) // 32 * 32
    data = np.memmap(path, np.uint8, "r")

    def get(name):
        shape, t, off = infos[name]
        per, nb = size[t]
        n = int(np.prod(shape))
        raw = torch.from_numpy(np.array(data[base + off:base + off + n // per * nb])).cuda()
        if t == 0:
            return raw.view(torch.float32).double().reshape(shape)
        if t == 1:
            return raw.view(torch.float16).double().reshape(shape)
        b = raw.reshape(-1, 34)
        return (b[:, :2].contiguous().view(torch.float16).double() * b[:, 2:].contiguous().view(torch.int8).double()).reshape(shape)

    return get


def _ln(x, w, b, eps):
    return (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + eps) * w + b


def _heads_attention(q, k, v, mask):
    """q, k, v [T][heads][dim] of one sequence; mask [T][T] (true: seen) or None."""
    q, k, v = (t.transpose(0, 1).contiguous() for t in (q, k, v))
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
    if mask is not None:
        s = s.masked_fill(~mask, -math.inf)
    return torch.matmul(torch.softmax(s, -1), v).transpose(0, 1).reshape(q.shape[1], -1)


def _pe(n):
    pos = torch.arange(n, dtype=torch.float64, device="cuda")[:, None]
    div = torch.exp(torch.arange(0, D, 2, dtype=torch.float64, device="cuda") * (-math.log(10000.0) / D))
    pe = torch.zeros(n, D, dtype=torch.float64, device="cuda")
    pe[:, 0::2], pe[:, 1::2] = torch.sin(pos * div), torch.cos(pos * div)
    return pe


def _decoder(reqs, extra, keep):
    """Logits in 64 bits of each request's last 1 + len(extra[b]) positions, its prompt followed by extra[b]."""
    get = _gguf(_model_path("ar"))
    xs, masks = [], []
    te, ae, pw, pb = (get("ar." + n) for n in ("text_emb", "audio_emb", "bert_proj", "bert_proj_b"))
    for r, more in zip(reqs, extra):
        T = len(r["phones"])
        text = te[torch.from_numpy(r["phones"]).long().cuda()] + pb
        if r["bert"] is not None:
            text = text + torch.from_numpy(r["bert"]).cuda().double().T.contiguous() @ pw.T.contiguous()
        codes = np.concatenate([r["prompt"], more]).astype(np.int64)
        sem = ae[torch.from_numpy(codes).cuda()]
        text, sem = text + _pe(T) * get("ar.text_pe_alpha"), sem + _pe(len(codes)) * get("ar.audio_pe_alpha")
        xs.append(torch.cat([text, sem]))
        n = T + len(codes)
        at = torch.arange(n, device="cuda")
        seen = at[None] <= torch.where(at < T, T - 1, at)[:, None]
        masks.append(seen)
    for li in range(NL):
        g = lambda n: get("transformer.block%d.%s" % (li, n))  # noqa: E731
        w = {n: g(n) for n in ("qkv_w", "qkv_b", "out_w", "out_b", "norm1_w", "norm1_b", "ffn1_w", "ffn1_b", "ffn2_w",
                               "ffn2_b", "norm2_w", "norm2_b")}
        for b, x in enumerate(xs):
            qkv = (x @ w["qkv_w"].T + w["qkv_b"]).reshape(-1, 3, NH, HD)
            a = _heads_attention(qkv[:, 0], qkv[:, 1], qkv[:, 2], masks[b])
            x = _ln(x + a @ w["out_w"].T + w["out_b"], w["norm1_w"], w["norm1_b"], 1e-5)
            h = torch.relu(x @ w["ffn1_w"].T + w["ffn1_b"])
            xs[b] = _ln(x + h @ w["ffn2_w"].T + w["ffn2_b"], w["norm2_w"], w["norm2_b"], 1e-5)
    head = get("ar.predict")
    return [x[-keep:] @ head.T for x in xs]


def exact(case, seed):
    kind = case["kind"]
    if kind == "prefill":
        reqs, _ = _requests(case, seed)
        return {"logits": torch.cat(_decoder(reqs, [[]] * len(reqs), 1))}
    if kind == "steps":
        reqs, toks = _requests(case, seed)
        n = len(toks)
        return {"logits": torch.stack(_decoder(reqs, list(toks.T), n + 1), 1)}
    if kind == "generate":
        reqs, toks = _requests(case, seed)
        n, forced = len(toks), toks[:, 0]
        z = _decoder(reqs[:1], [forced[:-1]], n)[0]
        hist = torch.zeros(V, device="cuda", dtype=torch.float64)
        hist += torch.bincount(torch.from_numpy(reqs[0]["prompt"]).cuda().long(), minlength=V)
        rows = []
        for i in range(n):
            p = torch.where(z[i] < 0, z[i] * 1.35 ** hist, z[i] / 1.35 ** hist)
            p[EOS] = -math.inf
            rows.append(torch.softmax(p, -1))
            hist[int(forced[i])] += 1
        out = {"probs": torch.stack(rows)}
        return dict(out, tokens=[None] * case["B"]) if case["exact"] else out
    if kind == "bert":
        rng = np.random.Generator(np.random.PCG64([seed, 4]))
        seqs = [torch.from_numpy(rng.integers(0, BV, n)).cuda() for n in _lens(case)]
        get = _gguf(_model_path(case["type"]))
        word, pos, typ = get("bert.word_emb"), get("bert.pos_emb"), get("bert.type_emb")[0]
        lens = [len(q) for q in seqs]
        x = torch.cat([word[q] + pos[:len(q)] + typ for q in seqs])
        x = _ln(x, get("bert.emb_ln_w"), get("bert.emb_ln_b"), 1e-12)
        for li in range(BL):
            g = lambda n: get("bert.l%d.%s" % (li, n))  # noqa: E731
            qkv = (x @ g("qkv_w").T + g("qkv_b")).reshape(-1, 3, BH, BD // BH)
            a = torch.cat([_heads_attention(*t.unbind(1), None) for t in qkv.split(lens)])
            x = _ln(x + a @ g("attn_out_w").T + g("attn_out_b"), g("attn_ln_w"), g("attn_ln_b"), 1e-12)
            h = x @ g("ff1_w").T + g("ff1_b")
            h = 0.5 * h * (1 + torch.erf(h / math.sqrt(2.0)))
            x = _ln(x + h @ g("ff2_w").T + g("ff2_b"), g("out_ln_w"), g("out_ln_b"), 1e-12)
        return {"features": [t.T.contiguous() for t in x.split(lens)]}
    if kind == "attn_decode":
        q, k, v, begin, end = _attn_decode_inputs(case, seed)
        at = torch.arange(k.shape[2], device="cuda")
        out = []
        for b in range(case["B"]):
            s = torch.matmul(k[b].double(), q[b].double()[..., None])[..., 0] * SCALE
            s = s.masked_fill(~((at >= begin[b]) & (at < end[b])), -math.inf)
            out.append((torch.softmax(s, -1)[..., None] * v[b].double()).sum(1).reshape(-1))
        return {"out": torch.stack(out)}
    if kind == "attn_prefill":
        qkv, pad = _attn_prefill_inputs(case, seed)
        B, S, _ = qkv.shape
        at = torch.arange(S, device="cuda")
        out = []
        for b in range(B):
            x = qkv[b].double().reshape(S, 3, NH, HD)
            seen = (at[None] >= pad[b]) & (at[None] < torch.where(at < case["hi"], case["hi"], at + 1)[:, None])
            out.append(_heads_attention(x[:, 0], x[:, 1], x[:, 2], seen))
        return {"out": torch.stack(out), "oq": None, "od": None}
    wq, wd, xq, xd, bias = _proj_inputs(case, seed)
    w = wq.double().reshape(wq.shape[0], -1, 32) * wd.double()[..., None]
    x = xq.double().reshape(xq.shape[0], -1, 32) * xd.double()[..., None]
    y = x.reshape(xq.shape) @ w.reshape(wq.shape).T.contiguous() + bias.double()
    return {"out": y.relu() if case["proj"] == "ffn1" else y}
