"""What the speed of this framework is measured on: passes through its public entry points at the sizes people run.

Six kinds of pass:

  decode    one greedy step of the quantised engine: the program holds the step's tokens, positions and block table on the device, hands them to
            ``DecoderEngine.set_inputs`` and replays the captured step;
  prefill   prompts through ``DecoderEngine.prefill`` and the greedy first token of each;
  sample    the sampler behind the output head: temperature, penalties, top-k / top-p filter and draw (``sampler.sample_greedy``);
  score     a hybrid model reads whole prompts in one ragged step (``ServingEngine.run_step``), the logits of some rows come back;
  serve     a hybrid model takes a batch of prompts and then decodes forced tokens, one ragged step each, graphs on; everything is released.

Weights, caches and prompts are random, made on the device from the seed.  The embedding and the output head of the quantised models are
correlated (as in a trained model, the next token is not a coin toss), so greedy tokens have a margin that rounding does not cross."""
import math

import torch

from rtp_llm_amd import model, ops, sampler
from rtp_llm_amd.hybrid import HybridConfig, HybridModel
from rtp_llm_amd.kvcache import CacheManager
from rtp_llm_amd.scheduler import ServingEngine

DEV = "cuda"
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one user in front of a small unquantised model: launches and latency
        dict(name="decode-0.5b-fp16-b1", kind="decode", model="qwen2-0.5b", weights="fp16", kv="16", dtype="fp16", batch=1, ctx=128, ragged=False, page=16),
        # one user, 4-bit 7B: the weights' stream
        dict(name="decode-7b-w4-b1", kind="decode", model="qwen2-7b", weights="w4", kv="16", dtype="fp16", batch=1, ctx=1024, ragged=False, page=16),
        # the benchmark's headline: a full batch over 4-bit weights and a 16-bit cache
        dict(name="decode-7b-w4-b64", kind="decode", model="qwen2-7b", weights="w4", kv="16", dtype="fp16", batch=64, ctx=1024, ragged=False, page=16),
        # a full batch with long contexts over an 8-bit cache
        dict(name="decode-7b-w4-kv8-b64", kind="decode", model="qwen2-7b", weights="w4", kv="int8", dtype="fp16", batch=64, ctx=4096, ragged=False, page=16),
        # 8-bit weights in bf16, an odd number of sequences of unequal length, large pages
        dict(name="decode-7b-w8-bf16-b13", kind="decode", model="qwen2-7b", weights="int8", kv="16", dtype="bf16", batch=13, ctx=1024, ragged=True, page=64),
        # a batch of prompts into the 4-bit model
        dict(name="prefill-7b-w4-8x512", kind="prefill", model="qwen2-7b", weights="w4", kv="16", dtype="fp16", prompts=8, length=512, ragged=False, page=16),
        # three prompts of unequal, odd length into the 8-bit-weight model
        dict(name="prefill-7b-w8-ragged", kind="prefill", model="qwen2-7b", weights="int8", kv="16", dtype="fp16", prompts=3, length=389, ragged=True, page=16),
        # one prompt into the small unquantised model, in bf16
        dict(name="prefill-0.5b-bf16", kind="prefill", model="qwen2-0.5b", weights="fp16", kv="16", dtype="bf16", prompts=1, length=777, ragged=False, page=64),
        # the sampler behind a full decode batch
        dict(name="sample-b64", kind="sample", rows=64, vocab=152064, history=256, penalties=True),
        # recurrent hybrid: a batch of long prompts
        dict(name="score-recurrent-4x2048", kind="score", design="recurrent", width=2048, layers=16, prompts=4, length=2048, ragged=False, every=512),
        # hybrid of experts and latent attention: one long prompt scored
        dict(name="score-experts-1537", kind="score", design="experts", width=1024, layers=8, prompts=1, length=1537, ragged=False, every=4),
        # recurrent hybrid in service: eight short prompts, then decoding
        dict(name="serve-recurrent-b8", kind="serve", design="recurrent", width=2048, layers=16, prompts=8, length=96, ragged=True, steps=8),
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "sample", "score", "score", "serve"])
    if kind in ("decode", "prefill"):
        m, w = rng.choice([("qwen2-7b", "w4"), ("qwen2-7b", "w4"), ("qwen2-7b", "int8"), ("qwen2-0.5b", "fp16"), ("qwen2-0.5b", "w4")])
        c = dict(kind=kind, model=m, weights=w, kv=rng.choice(["16", "16", "int8"]) if kind == "decode" else "16",
                 dtype=rng.choice(["fp16", "fp16", "bf16"]), ragged=rng.random() < 0.6, page=rng.choice([16, 64]))
        if kind == "decode":
            c["batch"] = _log(rng, 1, 64)
            c["ctx"] = _log(rng, 32, min(4096, (262144 if c["kv"] == "int8" else 131072) // c["batch"]))
        else:
            c["prompts"] = _log(rng, 1, 8)
            c["length"] = _log(rng, 16, 512 if c["prompts"] > 1 else 1500)
        return c
    if kind == "sample":
        return dict(kind=kind, rows=_log(rng, 1, 64), vocab=rng.choice([32000, 128256, 151936, 152064]), history=_log(rng, 16, 512), penalties=rng.random() < 0.5)
    design = rng.choice(["recurrent", "experts"])
    width, layers = rng.choice([(1024, 8), (2048, 16)]) if design == "recurrent" else (1024, 8)
    c = dict(kind=kind, design=design, width=width, layers=layers, ragged=rng.random() < 0.6)
    if kind == "score":
        c.update(prompts=_log(rng, 1, 4), length=_log(rng, 64, 2048), every=rng.choice([4, 7] if design == "experts" else [32, 100]))
    else:
        c.update(prompts=_log(rng, 1, 16), length=_log(rng, 16, 512), steps=rng.randint(4, 12))
    return c


# ------------------------------------------------------------------------------------------------ the quantised models
class Canon:
    """The model's tensors in the loader's conventions (linears [in, out]; 4-bit codes with their effective zeros; int8 codes with a scale per column)."""

    def __init__(self, case, seed):
        cfg = self.cfg = model.MODELS[case["model"]]
        g = self.g = torch.Generator(device=DEV).manual_seed(int(seed))
        self.kind, self.dt = case["weights"], DTYPES[case["dtype"]]
        self.embedding = (torch.randn(cfg.vocab, cfg.hidden, device=DEV, generator=g) * 0.5).to(self.dt)
        self.final_norm = self._norm()
        after = torch.randperm(cfg.vocab, device=DEV, generator=g)                       # the token that tends to follow each token
        head = torch.randn(cfg.hidden, cfg.vocab, device=DEV, generator=g, dtype=torch.float16) * cfg.hidden ** -0.5
        head[:, after] += (self.embedding.t() * (43.0 / cfg.hidden)).half()
        self.head = head.to(self.dt)
        n = (cfg.nh + 2 * cfg.nkv) * cfg.hd
        self.shapes = {"qkv": (cfg.hidden, n), "o": (cfg.nh * cfg.hd, cfg.hidden), "gate_up": (cfg.hidden, 2 * cfg.inter), "down": (cfg.inter, cfg.hidden)}

    def _norm(self):
        return (1.0 + 0.1 * torch.randn(self.cfg.hidden, device=DEV, generator=self.g)).to(self.dt)

    def layers(self):
        """One layer's tensors at a time, in order."""
        g = self.g
        for _ in range(self.cfg.num_layers):
            L = {}
            for name, (K, N) in self.shapes.items():
                a = math.sqrt(6.0 / (K + N))
                if self.kind == "w4":
                    q = torch.randint(0, 16, (K, N), device=DEV, generator=g, dtype=torch.uint8)
                    z = torch.randint(7, 9, (K // 128, N), device=DEV, generator=g, dtype=torch.uint8)
                    s = ((torch.rand(K // 128, N, device=DEV, generator=g) + 0.5) * (2 * a / 15)).half()
                    L[name] = (q, s, z)
                elif self.kind == "int8":
                    q = torch.randint(-127, 128, (K, N), device=DEV, generator=g, dtype=torch.int8)
                    L[name] = (q, ((torch.rand(N, device=DEV, generator=g) + 0.5) * (a / 127)).half(), None)
                else:
                    L[name] = (((torch.rand(K, N, device=DEV, generator=g) * 2 - 1) * a).to(self.dt), None, None)
            L["bias"] = ((torch.rand(self.shapes["qkv"][1], device=DEV, generator=g) - 0.5) * 0.2).to(self.dt)
            L["norms"] = (self._norm(), self._norm())
            yield L

    def linear(self, t):
        q, s, z = t
        K, N = q.shape
        if self.kind == "w4":
            return model.CanonLinear("w4", K, N, q=q, scales=s, z_eff=z, group_size=128)
        return model.CanonLinear("int8", K, N, q=q, scales=s) if self.kind == "int8" else model.CanonLinear("fp16", K, N, w=q)

    def dense(self, t):
        """The linear's weights in 64 bits."""
        q, s, z = t
        if self.kind == "w4":
            return ((q.double().view(-1, 128, q.shape[1]) - z.double()[:, None]) * s.double()[:, None]).view(q.shape)
        return q.double() * s.double() if self.kind == "int8" else q.double()


def _lengths(n, top, ragged):
    """Lengths of n sequences, the last of them the longest: a case's own, whatever the seed."""
    if not ragged:
        return [top] * n
    g = torch.Generator().manual_seed(n * 10007 + top)
    return [int(v) for v in torch.randint(max(1, top // 4), top + 1, (n - 1,), generator=g)] + [top]


def _plan(case, seed):
    """(tokens per sequence, cached tokens per sequence, block table) on the host."""
    g = torch.Generator().manual_seed(int(seed) * 7 + 1)
    vocab, page = model.MODELS[case["model"]].vocab, case["page"]
    if case["kind"] == "decode":
        B, top = case["batch"], case["ctx"]
        old = [n - 1 for n in _lengths(B, top, case["ragged"])]
        toks = [[int(t)] for t in torch.randint(0, vocab, (B,), generator=g)]
    else:
        B, top = case["prompts"], case["length"]
        old, toks = [0] * B, [torch.randint(0, vocab, (k,), generator=g).tolist() for k in _lengths(B, top, case["ragged"])]
    per = -(-(top + 1) // page)
    return toks, old, torch.randperm(B * per, generator=g).reshape(B, per).to(torch.int32)


def _fill_cache(kv, scales, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed) + 77)
    for i, t in enumerate(kv):
        if t.dtype == torch.int8:
            t.copy_(torch.randint(-127, 128, t.shape, device=DEV, generator=g, dtype=torch.int8))
            scales[i].copy_(torch.rand(scales[i].shape, device=DEV, generator=g) * 0.02 + 0.005)
        else:
            t.copy_(torch.randn(t.shape, device=DEV, generator=g, dtype=torch.float16))


def _prepare_engine(case, seed):
    c = Canon(case, seed)
    toks, old, table = _plan(case, seed)
    layers = [{"qkv_bias": L["bias"], "input_norm": L["norms"][0], "post_norm": L["norms"][1], **{k: c.linear(L[k]) for k in c.shapes}} for L in c.layers()]
    weights = {"layers": layers, "embedding": c.embedding, "final_norm": c.final_norm, "lm_head": model.CanonLinear("fp16", *c.head.shape, w=c.head)}
    B = len(toks)
    eng = model.DecoderEngine(c.cfg, weights, kv_int8=case["kv"] == "int8", page=case["page"], num_blocks=table.numel(), max_batch=B,
                              max_seq_len=table.shape[1] * case["page"], device=DEV, dtype=c.dt)
    if case["kind"] == "prefill":
        return dict(eng=eng, prompts=toks, table=table)
    _fill_cache(eng.kv, eng.kv_scale, seed)
    i32 = dict(dtype=torch.int32, device=DEV)
    state = dict(eng=eng, ids=torch.tensor([t[0] for t in toks], **i32), pos=torch.tensor(old, **i32), table=table.to(DEV), batch=B)
    eng.set_inputs(state["ids"], state["pos"], state["table"])
    eng.capture(B)
    return state


def _engine_out(eng, logits, tokens):
    return {"logits": logits, "tokens": tokens, "kv": list(eng.kv), "kv_scale": [s for s in eng.kv_scale if s is not None]}


def _run_decode(s):
    eng, B = s["eng"], s["batch"]
    eng.set_inputs(s["ids"], s["pos"], s["table"])
    eng.replay(B, 1)
    return _engine_out(eng, eng.logits[:B], eng.token_ids[:B])


def _run_prefill(s):
    logits = s["eng"].prefill(s["prompts"], s["table"])
    return _engine_out(s["eng"], logits, ops.argmax(logits))


def _exact_engine(case, seed):
    c = Canon(case, seed)
    cfg, f64 = c.cfg, torch.float64
    toks, old, table = _plan(case, seed)
    B, page, int8 = len(toks), case["page"], case["kv"] == "int8"
    H, G, D = cfg.nh, cfg.nkv, cfg.hd
    n = [len(t) for t in toks]
    starts = [sum(n[:b]) for b in range(B + 1)]
    flat = torch.tensor([t for seq in toks for t in seq], device=DEV)
    pos = torch.cat([torch.arange(o, o + k, device=DEV) for o, k in zip(old, n)])
    seq = torch.cat([torch.full((k,), b, device=DEV) for b, k in enumerate(n)])
    tab = table.to(DEV).long()
    block, off = tab[seq, pos // page], pos % page
    shape = (table.numel(), 2, G, page, D)
    # the cache as the program finds it
    kv = [torch.zeros(shape, dtype=torch.int8 if int8 else c.dt, device=DEV) for _ in range(cfg.num_layers)]
    scales = [torch.ones(shape[:-1], device=DEV) if int8 else None for _ in kv]
    if case["kind"] == "decode":
        _fill_cache(kv, scales, seed)
    step = (torch.tensor(float(cfg.rope_theta), dtype=f64, device=DEV) ** (-torch.arange(0, D, 2, dtype=f64, device=DEV) / D))
    ang = pos.double()[:, None] * step
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]

    def rot(t):
        a, b = t[..., :D // 2], t[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    def norm(t, w):
        return t / torch.sqrt((t * t).mean(-1, keepdim=True) + cfg.rms_eps) * w.double()

    x = c.embedding[flat].double()
    out_kv, out_scale = [], []
    for i, L in enumerate(c.layers()):
        qkv = norm(x, L["norms"][0]) @ c.dense(L["qkv"]) + L["bias"].double()
        q, k, v = qkv[:, :H * D].view(-1, H, D), qkv[:, H * D:(H + G) * D].view(-1, G, D), qkv[:, (H + G) * D:].view(-1, G, D)
        q, k = rot(q), rot(k)
        # keys lie [token][channel] in a block, values [channel][token]
        full = kv[i].bitwise_xor(torch.tensor(-128, dtype=torch.int8, device=DEV)).double() if int8 else kv[i].double()
        ks, vs = full[:, 0], full[:, 1].reshape(-1, G, D, page)
        if int8:
            sc = scales[i].double()
            new = [torch.where((t != 0).any(-1), t.abs().amax(-1) / 127, torch.ones_like(t[..., 0])) for t in (k, v)]
            kq, vq = ((t / s[..., None]).round().clamp(-128, 127) for t, s in zip((k, v), new))
            ks[block, :, off], vs[block, :, :, off] = kq, vq
            sc[block, 0, :, off], sc[block, 1, :, off] = new
            out_scale.append(sc)
            out_kv.append(None)
            ks, vs = ks * sc[:, 0, :, :, None], vs * sc[:, 1, :, None, :]
        else:
            ks[block, :, off], vs[block, :, :, off] = k, v
            out_kv.append(full)
        o = torch.empty_like(q)
        for b in range(B):
            last = old[b] + n[b]
            use = tab[b, : -(-last // page)]
            kb = ks[use].transpose(0, 1).reshape(G, -1, D)[:, :last]
            vb = vs[use].permute(1, 0, 3, 2).reshape(G, -1, D)[:, :last]
            qb = q[starts[b]:starts[b + 1]].view(n[b], G, H // G, D).permute(1, 2, 0, 3).reshape(G, -1, D)
            sco = (qb @ kb.transpose(1, 2).contiguous()).view(G, H // G, n[b], last) * D ** -0.5
            ok = torch.arange(last, device=DEV)[None] <= pos[starts[b]:starts[b + 1], None]
            p = sco.masked_fill(~ok, float("-inf")).softmax(-1).view(G, -1, last)
            o[starts[b]:starts[b + 1]] = (p @ vb).view(G, H // G, n[b], D).permute(2, 0, 1, 3).reshape(n[b], H, D)
        x = x + o.reshape(-1, H * D) @ c.dense(L["o"])
        gu = norm(x, L["norms"][1]) @ c.dense(L["gate_up"])
        gate, up = gu[:, :cfg.inter], gu[:, cfg.inter:]
        x = x + (gate * torch.sigmoid(gate) * up) @ c.dense(L["down"])
        del full, ks, vs, qkv, gu
    rows = torch.tensor([s - 1 for s in starts[1:]], device=DEV)
    logits = norm(x[rows], c.final_norm) @ c.head.double()
    return {"logits": logits, "tokens": None, "kv": out_kv, "kv_scale": out_scale}


def _engine_work(case):
    cfg = model.MODELS[case["model"]]
    params = cfg.num_layers * (cfg.hidden * (cfg.nh + 2 * cfg.nkv) * cfg.hd + cfg.nh * cfg.hd * cfg.hidden + 3 * cfg.hidden * cfg.inter)
    per = {"w4": 0.5 + 4 / 128, "int8": 1.0, "fp16": 2.0}[case["weights"]]
    kv_tok = cfg.num_layers * 2 * cfg.nkv * (cfg.hd + 4 if case["kv"] == "int8" else 2 * cfg.hd)
    toks, old, _ = _plan(case, 0)
    rows, seqs = sum(len(t) for t in toks), len(toks)
    seen = sum(o + (len(t) + 1) / 2 for t, o in zip(toks, old) for _ in t)
    last = sum(o + len(t) for t, o in zip(toks, old))
    return {"bytes": params * per + 2 * cfg.hidden * cfg.vocab + last * kv_tok + seqs * 4 * cfg.vocab + 2 * rows * cfg.hidden,
            "flops": 2 * rows * params + 2 * seqs * cfg.hidden * cfg.vocab + 4 * cfg.num_layers * cfg.nh * cfg.hd * seen}


# ------------------------------------------------------------------------------------------------ the sampler
def _sample_inputs(case, seed):
    B, V, n = case["rows"], case["vocab"], case["history"]
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    h = torch.Generator().manual_seed(int(seed) * 7 + 1)
    # a bulk of unlikely tokens and a few dozen candidates above it
    logits = torch.randn(B, V, device=DEV, generator=g) * 2.0
    cand = torch.rand(B, V, device=DEV, generator=g).topk(48).indices
    logits.scatter_(1, cand, 8.0 + 2.5 * torch.randn(B, 48, device=DEV, generator=g))
    hist = torch.randint(0, V, (B, n + 1), generator=h, dtype=torch.int32)
    hist[:, : min(n, 24)] = cand[:, : min(n, 24)].cpu().int()
    pick = lambda values: torch.tensor(values)[torch.randint(0, len(values), (B,), generator=h)]
    p = dict(top_k=pick([0, 20, 50, 100]).int(), top_p=pick([0.8, 0.9, 0.95]).float(), temperature=pick([0.6, 0.8, 1.0]).float(),
             uniform=torch.rand(B, generator=h) * 0.998 + 0.001)
    if case["penalties"]:
        p.update(repetition_penalty=pick([1.0, 1.05, 1.1]).float(), presence_penalty=pick([0.0, 0.5]).float(), frequency_penalty=pick([0.0, 0.2]).float())
    return logits, hist, torch.full((B,), n, dtype=torch.int32), p


def _run_sample(s):
    logits = s["logits"].clone()                       # the head writes new logits for every step; the sampler works on them in place
    tokens = s["hist"]
    ids = sampler.sample_greedy(sampler.GreedyParams(logits=logits, input_lengths=s["lens"], sequence_lengths=s["lens"], token_ids=tokens,
                                                     step=tokens.shape[1] - 1, **s["params"]))
    return {"ids": ids, "probs": logits}


def _exact_sample(case, seed):
    logits, hist, lens, p = _sample_inputs(case, seed)
    x = logits.double()
    if bool((p["temperature"] != 1.0).any()):
        x = x / (p["temperature"].double() + 1e-6).to(DEV)[:, None]
    if case["penalties"]:
        count = torch.zeros_like(x).scatter_add_(1, hist[:, :-1].long().to(DEV), torch.ones(hist.shape[0], hist.shape[1] - 1, dtype=x.dtype, device=DEV))
        rep, pres, freq = (p[k + "_penalty"].double().to(DEV)[:, None] for k in ("repetition", "presence", "frequency"))
        x = torch.where(count > 0, torch.where(x < 0, x * rep, x / rep) - pres - freq * count, x)
    return {"ids": None, "probs": x.softmax(-1)}


# ------------------------------------------------------------------------------------------------ the hybrid models
def _hybrid_config(case):
    W, n = case["width"], case["layers"]
    H, G, ff, hd = W // 128, max(1, W // 512), {1024: 2816, 2048: 5632}[W], 128
    layers, owner = [], None
    for i in range(n):
        if case["design"] == "recurrent":
            t = ["gla", "attention", "hgrn2", "gla", "gla", "shared", "hgrn2", "gla"][i % 8]
            mlp = {"kind": "dense", "ff": ff}
            if t in ("attention", "shared"):
                mx = {"heads": H, "kv_heads": G, "dim": hd, "vdim": hd, "scale": hd ** -0.5, "mask": {"size": 1024}, "rot": {"base": 1e6, "dims": hd}}
                if t == "shared":
                    mx["kv_from"] = owner
                else:
                    owner = i
                layers.append({"type": "attention", "mixer": mx, "mlp": mlp})
            else:
                mx = {"heads": H, "dim": hd // 2, "vdim": hd}
                if t == "gla":
                    mx["tau"] = 16.0
                layers.append({"type": t, "mixer": mx, "mlp": mlp})
        else:
            t = ["retention", "latent", "latent", "retention", "latent", "latent", "retention", "latent"][i % 8]
            fe = ff // 4 // 32 * 32
            mlp = {"kind": "dense", "ff": ff} if i == 0 else {"kind": "moe", "expert": {"ff": fe}, "shared": {"ff": fe},
                                                               "router": {"experts": 16, "top": 4, "groups": {"count": 4, "keep": 2}}}
            if t == "latent":
                mx = {"heads": H, "dim": hd, "rot_dim": hd // 2, "vdim": hd, "kv_rank": 3 * hd // 2, "scale": (hd + hd // 2) ** -0.5,
                      "rot": {"base": 1e6, "dims": hd // 2, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
                layers.append({"type": "latent_attention", "mixer": mx, "mlp": mlp})
            else:
                mx = {"heads": H, "dim": hd // 2, "vdim": hd, "decay": [1.0 - 2.0 ** -(5 + h % 8) for h in range(H)], "rot": {"base": 1e6, "dims": hd // 2}}
                layers.append({"type": "retention", "mixer": mx, "mlp": mlp})
    cfg = {"architecture": "Nufalorn" if case["design"] == "recurrent" else "Pokepel", "layers": layers, "vocab": 32000, "width": W}
    if case["design"] == "recurrent":
        return {**cfg, "norm": {"eps": 1e-5}, "residual_mult": 0.3, "logit_softcap": 30.0}
    return {**cfg, "norm": {"eps": 1e-6}}


def _hybrid_weights(cfg, seed):
    g = torch.Generator(device=DEV).manual_seed(int(seed))
    W = cfg["width"]
    lin = lambda o, i, k=1.0: (torch.randn(o, i, device=DEV, generator=g) * (k * i ** -0.5)).bfloat16()
    vec = lambda n, k=0.1, off=0.0: (torch.randn(n, device=DEV, generator=g) * k + off).bfloat16()
    experts = cfg["architecture"] == "Pokepel"
    one = 1.0 if experts else 0.0                       # norm weights: plain, or offsets from one
    w = {"embed": torch.randn(cfg["vocab"], W, device=DEV, generator=g).bfloat16(), "head": lin(cfg["vocab"], W), "final.norm": vec(W, 0.1, one)}
    for i, L in enumerate(cfg["layers"]):
        p, mx, mlp, t = f"l{i}.", L["mixer"], L["mlp"], L["type"]
        H, d, dv = mx["heads"], mx["dim"], mx["vdim"]
        q = p + "mix."
        w[p + "norm1"] = vec(W, 0.1, one)
        if not experts:
            w[p + "norm2"] = vec(W)
        if t == "attention":
            w[q + "q"], w[q + "o"] = lin(H * d, W), lin(W, H * dv)
            if "kv_from" not in mx:
                w[q + "k"], w[q + "v"] = lin(mx["kv_heads"] * d, W), lin(mx["kv_heads"] * dv, W)
        elif t == "hgrn2":
            w[q + "q"], w[q + "f"], w[q + "v"], w[q + "o"] = lin(H * d, W), lin(H * d, W), lin(H * dv, W), lin(W, H * dv)
            w[q + "f.b"], w[q + "lower"], w[q + "norm"] = vec(H * d, 0.5), torch.sigmoid(vec(H * d, 1.0).float()).bfloat16(), vec(dv, 0.1, 1.0)
        elif t == "gla":
            w[q + "q"], w[q + "k"], w[q + "v"], w[q + "g"], w[q + "a1"] = lin(H * d, W), lin(H * d, W), lin(H * dv, W), lin(H * dv, W), lin(16, W)
            w[q + "a2"], w[q + "a2.b"], w[q + "norm"], w[q + "o"] = lin(H * d, 16), vec(H * d, 1.0, 2.0), vec(dv, 0.1, 1.0), lin(W, H * dv)
        elif t == "latent_attention":
            dr, R = mx["rot_dim"], mx["kv_rank"]
            for n, (o, k) in {"q": (H * (d + dr), W), "dkv": (R + dr, W), "uk": (H * d, R), "uv": (H * dv, R), "g": (H * dv, W), "o": (W, H * dv)}.items():
                w[q + n] = lin(o, k)
            w[q + "dkv.norm"], w[q + "sink"] = vec(R, 0.1, 1.0), vec(H, 1.0)
        else:
            for n, (o, k) in {"q": (H * d, W), "k": (H * d, W), "v": (H * dv, W), "g": (H * dv, W), "o": (W, H * dv)}.items():
                w[q + n] = lin(o, k)
        if experts:
            for n in ("rg1", "rg2"):
                w[p + n], w[p + n + ".b"] = lin(W, W), vec(W, 0.5)
        m = p + "mlp."
        if not experts:
            w[m + "gate"], w[m + "up"], w[m + "down"] = lin(mlp["ff"], W), lin(mlp["ff"], W), lin(W, mlp["ff"])
        elif mlp["kind"] == "dense":
            w[m + "up"], w[m + "down"], w[m + "act"] = lin(mlp["ff"], W), lin(W, mlp["ff"]), torch.tensor([0.6, 0.3, 0.1, 0.0]).bfloat16()
        else:
            w[m + "router"] = lin(mlp["router"]["experts"], W, 2.5)      # a trained router is decided: a few experts carry most of the weight
            f = mlp["expert"]["ff"]
            for n in [f"e{j}" for j in range(mlp["router"]["experts"])] + ["shared"]:
                w[m + n + ".gate"], w[m + n + ".up"], w[m + n + ".down"] = lin(f, W), lin(f, W), lin(W, f)
    return w


PAGE = 64


def _hybrid_plan(case, seed):
    """(prompts, forced continuation per step, rows wanted per prompt) on the host."""
    g = torch.Generator().manual_seed(int(seed) * 7 + 1)
    B = case["prompts"]
    n = _lengths(B, case["length"], case["ragged"])
    prompts = [torch.randint(0, 32000, (k,), generator=g).tolist() for k in n]
    forced = [torch.randint(0, 32000, (B,), generator=g).tolist() for _ in range(case.get("steps", 0))]
    if case["kind"] == "serve":
        wants = [[k - 1] for k in n]
    else:
        wants = [sorted(set(range(case["every"] - 1, k, case["every"])) | {k - 1}) for k in n]
    return prompts, forced, wants


def _prepare_hybrid(case, seed):
    cfg = _hybrid_config(case)
    mdl = HybridModel(HybridConfig.from_json(cfg), _hybrid_weights(cfg, seed), torch.bfloat16, torch.device(DEV), PAGE)
    prompts, forced, wants = _hybrid_plan(case, seed)
    tokens = sum(-(-(len(p) + len(forced)) // PAGE) * PAGE for p in prompts)
    eng = ServingEngine(mdl, max_tokens=tokens, max_seqs=len(prompts))
    s = dict(eng=eng, prompts=prompts, forced=forced, wants=wants)
    if case["kind"] == "serve":
        eng.use_graphs = True
        _run_hybrid(s)                                 # a server decodes once before it takes requests: its step graphs are kept
        for t in _cache_tensors(eng):
            t.zero_()
        eng.cache = CacheManager(eng.cache.pages.num_pages, PAGE, len(prompts))      # hands out its pages in order again
    return s


def _cache_tensors(eng):
    out, seen = [], set()
    for entry in eng.tensors:
        for t in entry if isinstance(entry, tuple) else (entry,):
            if t is not None and t.data_ptr() not in seen:
                seen.add(t.data_ptr())
                out.append(t)
    return out


def _run_hybrid(s):
    eng = s["eng"]
    ids = range(len(s["prompts"]))
    logits = [eng.run_step([(i, s["prompts"][i], s["wants"][i]) for i in ids])]
    for forced in s["forced"]:
        logits.append(eng.run_step([(i, [forced[i]], [0]) for i in ids]))
    for i in ids:
        eng.release(i)
    return {"logits": logits, "cache": _cache_tensors(eng)}


def _steps_of(rot, dims):
    i = torch.arange(dims // 2, dtype=torch.float64, device=DEV)
    f = float(rot["base"]) ** (-2.0 * i / dims)
    sc = rot.get("scaling")
    if not sc:
        return f, 1.0
    at = lambda turns: dims * math.log(sc["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(rot["base"]))
    lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


def _turn(t, steps, mag=1.0, sign=1.0, halves=False):
    """t [T, heads, d] (all d channels turned) by sign * position * step; pairs (2i, 2i + 1), or half a span apart."""
    a = sign * torch.arange(t.shape[0], dtype=torch.float64, device=DEV)[:, None] * steps
    c, s = (a.cos() * mag)[:, None], (a.sin() * mag)[:, None]
    h = t.shape[-1] // 2
    u, v = (t[..., :h], t[..., h:]) if halves else (t[..., 0::2], t[..., 1::2])
    x, y = u * c - v * s, v * c + u * s
    return torch.cat([x, y], -1) if halves else torch.stack([x, y], -1).flatten(-2)


def _softmax_rows(q, k, v, scale, ok, sink):
    """q [T, H, d], k / v [T, H, .], ok [T, T], sink [H]: one more logit per head that carries no value."""
    s = (q.transpose(0, 1) @ k.permute(1, 2, 0).contiguous()) * scale
    s = torch.cat([s.masked_fill(~ok, float("-inf")), sink.view(-1, 1, 1).expand(-1, s.shape[1], 1)], -1).softmax(-1)
    return (s[..., :-1].contiguous() @ v.transpose(0, 1).contiguous()).transpose(0, 1)


def _walk(q, k, v, a):
    """S <- diag(a_t) S + k_t v_t^T, o_t = S^T q_t over all heads.  q, k, a [T, H, d], v [T, H, dv] -> (o, last S)."""
    S = torch.zeros(q.shape[1], q.shape[2], v.shape[2], dtype=q.dtype, device=DEV)
    o = torch.empty(q.shape[0], q.shape[1], v.shape[2], dtype=q.dtype, device=DEV)
    for t in range(q.shape[0]):
        S = S * a[t][:, :, None] + k[t][:, :, None] * v[t][:, None, :]
        o[t] = (S * q[t][:, :, None]).sum(1)
    return o, S


def _exact_sequence(cfg, w, tokens):
    """(logits of every row, cached tensors per layer) of one sequence run whole, in 64 bits."""
    experts, eps = cfg["architecture"] == "Pokepel", cfg["norm"]["eps"]
    wt = lambda n: w[n].to(DEV).double()
    unit = lambda t: t / torch.sqrt((t * t).mean(-1, keepdim=True) + eps)
    norm = lambda t, n: unit(t) * (wt(n) if experts else 1.0 + wt(n))
    silu = torch.nn.functional.silu
    x = wt("embed")[torch.tensor(tokens, device=DEV)]
    T = x.shape[0]
    at = torch.arange(T, device=DEV)
    cached = []
    for i, L in enumerate(cfg["layers"]):
        p, mx, mlp, t = f"l{i}.", L["mixer"], L["mlp"], L["type"]
        q_, H, d, dv = p + "mix.", mx["heads"], mx["dim"], mx["vdim"]
        h = norm(x, p + "norm1")
        lin = lambda n: h @ wt(q_ + n).t()
        if t == "attention":
            G, steps = mx["kv_heads"], _steps_of(mx["rot"], d)[0]
            if "kv_from" in mx:
                k, v = cached[mx["kv_from"]]
                cached.append(None)
            else:
                k, v = _turn(lin("k").view(T, G, d), steps), _turn(unit(lin("v").view(T, G, dv)), steps)
                cached.append((k, v))
            size = mx["mask"]["size"]
            ok = (at[None] <= at[:, None]) & (at[None] >= at[:, None] // size * size)
            rep = lambda u: u.repeat_interleave(H // G, 1)
            o = _softmax_rows(_turn(lin("q").view(T, H, d), steps), rep(k), rep(v), mx["scale"], ok, torch.zeros(H, dtype=x.dtype, device=DEV))
            y = _turn(o, steps, sign=-1.0).reshape(T, -1) @ wt(q_ + "o").t()
        elif t == "latent_attention":
            dr, R = mx["rot_dim"], mx["kv_rank"]
            steps, mag = _steps_of(mx["rot"], dr)
            q, down = lin("q").view(T, H, d + dr), lin("dkv")
            c = unit(down[:, :R]) * wt(q_ + "dkv.norm")
            kr = _turn(down[:, None, R:], steps, mag)
            cached.append(torch.cat([c, kr[:, 0]], -1))
            k = torch.cat([(c @ wt(q_ + "uk").t()).view(T, H, d), kr.expand(-1, H, -1)], -1)
            q = torch.cat([q[..., :d], _turn(q[..., d:], steps, mag)], -1)
            o = _softmax_rows(q, k, (c @ wt(q_ + "uv").t()).view(T, H, dv), mx["scale"], at[None] <= at[:, None], wt(q_ + "sink"))
            y = (o.reshape(T, -1) * torch.sigmoid(lin("g"))) @ wt(q_ + "o").t()
        else:
            v = lin("v").view(T, H, dv)
            if t == "hgrn2":
                low = wt(q_ + "lower").view(H, d)
                a = low + (1.0 - low) * torch.sigmoid(lin("f") + wt(q_ + "f.b")).view(T, H, d)
                q, k = silu(lin("q")).view(T, H, d), 1.0 - a
            elif t == "gla":
                a = torch.exp(torch.nn.functional.logsigmoid(lin("a1") @ wt(q_ + "a2").t() + wt(q_ + "a2.b")) / mx["tau"]).view(T, H, d)
                q, k = lin("q").view(T, H, d) * d ** -0.5, lin("k").view(T, H, d)
            else:
                steps = _steps_of(mx["rot"], d)[0]
                a = torch.tensor(mx["decay"], dtype=x.dtype, device=DEV).view(1, H, 1).expand(T, H, d)
                q, k = _turn(lin("q").view(T, H, d), steps, halves=True), _turn(lin("k").view(T, H, d), steps, halves=True) * d ** -0.5
            o, S = _walk(q, k, v, a)
            cached.append(S)
            o = unit(o) if t == "retention" else unit(o) * wt(q_ + "norm")
            o = o.reshape(T, -1)
            y = (o if t == "hgrn2" else o * silu(lin("g"))) @ wt(q_ + "o").t()
        m = p + "mlp."
        if not experts:
            h2 = norm(x, p + "norm2")
            f = (torch.relu(h2 @ wt(m + "gate").t()) * (h2 @ wt(m + "up").t())) @ wt(m + "down").t()
            x = x + cfg["residual_mult"] * (y + f)
            continue
        if mlp["kind"] == "dense":
            z = h @ wt(m + "up").t()
            a, b, c3, e = [float(u) for u in w[m + "act"]]
            f = (a * unit(z) + b * unit(z * z) + c3 * unit(z * z * z) + e) @ wt(m + "down").t()
        else:
            expert = lambda rows, n: (silu(rows @ wt(m + n + ".gate").t()) * (rows @ wt(m + n + ".up").t())) @ wt(m + n + ".down").t()
            r = mlp["router"]
            s = torch.softmax(h @ wt(m + "router").t(), -1)
            grp = s.view(T, r["groups"]["count"], -1)
            keep = torch.zeros(T, grp.shape[1], dtype=torch.bool, device=DEV).scatter_(1, grp.amax(-1).topk(r["groups"]["keep"], -1).indices, True)
            ids = grp.masked_fill(~keep[..., None], -1.0).view(T, -1).topk(r["top"], -1).indices
            f = expert(h, "shared")
            for j in range(r["experts"]):
                rows = (ids == j).any(-1).nonzero()[:, 0]
                if rows.numel():
                    f[rows] += s[rows, j, None] * expert(h[rows], f"e{j}")
        gate = lambda n: torch.sigmoid(h @ wt(p + n).t() + wt(p + n + ".b"))
        x = x + y * gate("rg1") + f * gate("rg2")
    logits = norm(x, "final.norm") @ wt("head").t()
    cap = cfg.get("logit_softcap")
    return (cap * torch.tanh(logits / cap) if cap else logits), cached


def _exact_hybrid(case, seed):
    cfg = _hybrid_config(case)
    w = _hybrid_weights(cfg, seed)
    prompts, forced, wants = _hybrid_plan(case, seed)
    B, n = len(prompts), len(forced)
    got = [_exact_sequence(cfg, w, p + [f[b] for f in forced]) for b, p in enumerate(prompts)]
    logits = [torch.cat([got[b][0][wants[b]] for b in range(B)])]
    logits += [torch.stack([got[b][0][len(prompts[b]) + j] for b in range(B)]) for j in range(n)]
    # pages in the order in which a fresh pool hands them out: the prompts' first, then one at a time as sequences outgrow theirs
    total = sum(-(-(len(p) + n) // PAGE) for p in prompts)
    free, pages = iter(range(total)), []
    for p in prompts:
        pages.append([next(free) for _ in range(-(-len(p) // PAGE))])
    for j in range(n):
        for b, p in enumerate(prompts):
            if len(pages[b]) * PAGE < len(p) + j + 1:
                pages[b].append(next(free))
    cache = []
    for i, L in enumerate(cfg["layers"]):
        if "kv_from" in L["mixer"]:
            continue
        if L["type"] not in ("attention", "latent_attention"):
            cache.append(torch.stack([got[b][1][i] for b in range(B)]))
            continue
        parts = [got[b][1][i] if isinstance(got[b][1][i], tuple) else (got[b][1][i][:, None],) for b in range(B)]
        for which in range(len(parts[0])):
            heads, width = parts[0][which].shape[1:]
            pool = torch.zeros(total, heads, PAGE, -(-width // 32) * 32, dtype=torch.float64, device=DEV)
            for b in range(B):
                t = parts[b][which]
                at = torch.arange(t.shape[0], device=DEV)
                pool[torch.tensor(pages[b], device=DEV)[at // PAGE], :, at % PAGE, :width] = t
            cache.append(pool if L["type"] == "attention" else pool[:, 0])
    return {"logits": logits, "cache": cache}


def _hybrid_work(case):
    cfg = _hybrid_config(case)
    prompts, forced, wants = _hybrid_plan(case, 0)
    W, V, B, steps = cfg["width"], cfg["vocab"], len(prompts), 1 + len(forced)
    rows = [len(p) + len(forced) for p in prompts]
    T = sum(rows)
    heads = sum(len(x) for x in wants) + B * len(forced)
    weights, active, other_flops, state = 0, 0, 0, 0
    for L in cfg["layers"]:
        mx, mlp = L["mixer"], L["mlp"]
        H, d, dv = mx["heads"], mx["dim"], mx["vdim"]
        if L["type"] == "attention":
            own = 0 if "kv_from" in mx else mx["kv_heads"] * (d + dv)
            n = W * (H * d + own + H * dv)
            size = mx["mask"]["size"]
            other_flops += sum(2 * H * (d + dv) * sum(t % size + 1 for t in range(r)) for r in rows)
            state += T * mx["kv_heads"] * (d + dv) * 2
        elif L["type"] == "latent_attention":
            R, dr = mx["kv_rank"], mx["rot_dim"]
            n = W * (H * (d + dr) + R + dr + 2 * H * dv) + H * R * (d + dv)
            other_flops += sum(H * (d + dr + dv) * r * (r + 1) for r in rows)
            state += T * (R + dr) * 2
        else:
            n = W * H * (2 * d + (2 if L["type"] == "hgrn2" else 3) * dv) + (16 * (W + H * d) if L["type"] == "gla" else 0)
            other_flops += 5 * T * H * d * dv
            state += B * H * d * dv * 4 * (2 * steps - 1)
        if cfg["architecture"] == "Pokepel":
            n += 2 * W * W
        weights, active = weights + n, active + n
        if mlp["kind"] == "moe":
            f, r = mlp["expert"]["ff"], mlp["router"]
            active += 3 * W * f * (r["top"] + 1) + W * r["experts"]
            weights += 3 * W * f * (min(r["experts"], r["top"] * T) + 1) + W * r["experts"]
        else:
            k = 2 if cfg["architecture"] == "Pokepel" else 3
            weights, active = weights + k * W * mlp["ff"], active + k * W * mlp["ff"]
    return {"bytes": steps * 2 * (weights + V * W) + state + 2 * T * W + heads * V * 4, "flops": 2 * T * active + 2 * heads * V * W + other_flops}


# ------------------------------------------------------------------------------------------------ what the measurement calls
def prepare(case, seed):
    if case["kind"] in ("decode", "prefill"):
        return {"kind": case["kind"], **_prepare_engine(case, seed)}
    if case["kind"] == "sample":
        logits, hist, lens, params = _sample_inputs(case, seed)
        return dict(kind="sample", logits=logits, hist=hist, lens=lens, params=params)
    return {"kind": case["kind"], **_prepare_hybrid(case, seed)}


def run(state):
    return {"decode": _run_decode, "prefill": _run_prefill, "sample": _run_sample, "score": _run_hybrid, "serve": _run_hybrid}[state["kind"]](state)


def work(case):
    if case["kind"] in ("decode", "prefill"):
        return _engine_work(case)
    if case["kind"] == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": 8 * n + 4 * case["rows"] * case["history"], "flops": 6 * n}   # logits read, probabilities written
    return _hybrid_work(case)


def tolerance(case):
    """About four times what the path is off its 64-bit result: 32-bit sums and exponentials in the sampler (4.5e-7 measured), a whole stack in fp16
    (2e-3) or bf16 (1e-2), a hybrid stack in bf16 over an fp32 residual (4e-3; with experts 1.4e-2, some rows then take another last expert).  An 8-bit
    cache may round a new code the other way."""
    if case["kind"] == "sample":
        return {"rel": 5e-6, "max": 1e-4, "differ": 0.0}
    if case["kind"] in ("decode", "prefill"):
        return {"rel": 3e-2 if case["dtype"] == "bf16" else 8e-3, "max": 0.6, "differ": 1e-2 if case["kv"] == "int8" else 0.0}
    return {"rel": 3e-2, "max": 0.9, "differ": 0.0} if case["design"] == "experts" else {"rel": 2e-2, "max": 0.6, "differ": 0.0}


def exact(case, seed):
    if case["kind"] in ("decode", "prefill"):
        return _exact_engine(case, seed)
    if case["kind"] == "sample":
        return _exact_sample(case, seed)
    return _exact_hybrid(case, seed)
