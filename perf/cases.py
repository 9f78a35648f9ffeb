"""What this framework is timed on: the calls a serving process makes.

* ``embed``: token ids of a request's documents through ``EmbeddingEngine.embed_sync``, host
  arrays of vectors back (what ``/v1/embeddings`` and embed jobs run).
* ``prefill``: one step over whole prompts through ``LLMEngine.feed``, the logits of each
  prompt's last token back (a request's time to first token).
* ``decode``: one token for every running stream: the model's forward on the engine's cache and
  state slots and the greedy sampler, captured once in a graph, as the serving loop does.  A pass
  replays it.  Models with recurrent states advance them with every pass.

Models and widths are presets of ``llm_mcp_amd.models.config``; weights are random.  Sequence
lengths inside a batch are ragged: a case's ``tokens`` / ``context`` is the longest.
"""
import math
import random

import numpy as np
import torch

PAGE = 32
F64 = torch.float64


def listed():
    return [
        # a search query to embed: the smallest call, launches and host work count
        dict(name="embed-query", path="embed", model="nomic-embed-text", docs=1, tokens=16),
        # one API request of 16 documents
        dict(name="embed-request", path="embed", model="nomic-embed-text", docs=16, tokens=1024),
        # a batch of passages of an indexing job
        dict(name="embed-passages", path="embed", model="mxbai-embed-large", docs=48, tokens=512),
        # a short chat turn of one user
        dict(name="prefill-turn", path="prefill", model="llama-3-8b", prompts=1, tokens=160),
        # part of a wave of chat requests
        dict(name="prefill-wave", path="prefill", model="llama-3-8b", prompts=16, tokens=512),
        # one long document
        dict(name="prefill-long", path="prefill", model="llama-3-8b", prompts=1, tokens=7680),
        # a prompt of a decoder with linear attention, state-space layers and attention
        dict(name="prefill-hybrid", path="prefill", model="zegopel-8b", prompts=1, tokens=2048),
        # a small model answering one user: latency
        dict(name="decode-small", path="decode", model="llama-3.2-1b", streams=1, context=200),
        # one user of the flagship
        dict(name="decode-one", path="decode", model="llama-3-8b", streams=1, context=1024),
        # a lightly loaded server
        dict(name="decode-16", path="decode", model="llama-3-8b", streams=16, context=1024),
        # a full one
        dict(name="decode-256", path="decode", model="llama-3-8b", streams=256, context=768),
        # the decoder with recurrent states, moderately loaded
        dict(name="decode-hybrid", path="decode", model="zegopel-8b", streams=64, context=1024),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    path = rng.choice(("embed", "embed", "prefill", "decode", "decode"))
    if path == "embed":
        model = rng.choice(("nomic-embed-text", "mxbai-embed-large"))
        longest = _log_int(rng, 8, 1024 if model == "nomic-embed-text" else 512)
        return dict(path=path, model=model, tokens=longest,
                    docs=_log_int(rng, 1, min(64, 24576 // longest)))
    model = rng.choice(("llama-3.2-1b", "llama-3-8b", "zegopel-8b"))
    if path == "prefill":
        longest = _log_int(rng, 16, 7680 if model != "zegopel-8b" else 2048)
        return dict(path=path, model=model, tokens=longest,
                    prompts=_log_int(rng, 1, max(1, min(32, 7680 // longest))))
    most = 64 if model == "zegopel-8b" else 256
    context = _log_int(rng, 32, 4096)
    return dict(path=path, model=model, context=context,
                streams=_log_int(rng, 1, min(most, 196608 // context)))


def _lengths(case):
    """Ragged lengths; the first sequence is the longest."""
    n = case.get("docs") or case.get("prompts") or case.get("streams")
    longest = case.get("tokens") or case["context"]
    r = random.Random(n * 10007 + longest)
    return [longest] + [r.randint(max(1, longest // 2), longest) for _ in range(n - 1)]


def _config(case):
    from llm_mcp_amd.models.config import resolve
    return resolve(case["model"])


# ---------------------------------------------------------------- weights ----
def _maker(seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(seed)

    def rnd(*shape, std=0.02, mean=0.0, dtype=torch.bfloat16):
        return torch.empty(shape, dtype=dtype, device=device).normal_(mean, std, generator=g)
    return rnd


def _nomic_weights(cfg, rnd):
    d, ff = cfg.hidden_size, cfg.intermediate_size
    s, t = d ** -0.5, ff ** -0.5
    layers = [dict(wqkv=rnd(3 * d, d, std=s), wo=rnd(d, d, std=s), w_gate_up=rnd(2 * ff, d, std=s),
                   w_down=rnd(d, ff, std=t), ln1_w=rnd(d, mean=1.0, std=0.1), ln1_b=rnd(d),
                   ln2_w=rnd(d, mean=1.0, std=0.1), ln2_b=rnd(d)) for _ in range(cfg.num_layers)]
    return dict(word=rnd(cfg.vocab_size, d, std=1.0), type=rnd(cfg.type_vocab_size, d),
                emb_ln_w=rnd(d, mean=1.0, std=0.1), emb_ln_b=rnd(d), layers=layers)


def _bert_weights(cfg, rnd):
    d, ff = cfg.hidden_size, cfg.intermediate_size
    s, t = d ** -0.5, ff ** -0.5
    layers = [dict(wqkv=rnd(3 * d, d, std=s), bqkv=rnd(3 * d), wo=rnd(d, d, std=s), bo=rnd(d),
                   ln1_w=rnd(d, mean=1.0, std=0.1), ln1_b=rnd(d), w1=rnd(ff, d, std=s), b1=rnd(ff),
                   w2=rnd(d, ff, std=t), b2=rnd(d), ln2_w=rnd(d, mean=1.0, std=0.1), ln2_b=rnd(d))
              for _ in range(cfg.num_layers)]
    return dict(word=rnd(cfg.vocab_size, d, std=1.0), pos=rnd(cfg.max_position, d),
                type=rnd(cfg.type_vocab_size, d), emb_ln_w=rnd(d, mean=1.0, std=0.1),
                emb_ln_b=rnd(d), layers=layers)


def _llama_weights(cfg, rnd):
    d, ff, D = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    deep = 0.02 / math.sqrt(2 * cfg.num_layers)
    layers = [dict(ln1=rnd(d, mean=1.0, std=0.1), ln2=rnd(d, mean=1.0, std=0.1),
                   wqkv=rnd((cfg.num_heads + 2 * cfg.num_kv_heads) * D, d),
                   wo=rnd(d, cfg.num_heads * D, std=deep), w_gate_up=rnd(2 * ff, d),
                   w_down=rnd(d, ff, std=deep)) for _ in range(cfg.num_layers)]
    embed = rnd(cfg.vocab_size, d, std=1.0)
    return dict(embed=embed, norm=rnd(d, mean=1.0, std=0.1),
                lm_head=embed if cfg.tie_embeddings else rnd(cfg.vocab_size, d), layers=layers)


def _zegopel_weights(cfg, rnd):
    d, W = cfg.hidden_size, dict(embed=rnd(cfg.vocab_size, cfg.hidden_size, std=1.0))
    deep = 0.02 / math.sqrt(2 * len(cfg.layers))
    for i, L in enumerate(cfg.layers):
        m, p = L["mixer"], "l%d." % i
        x = p + "mix."
        if L["type"] == "lightning":
            qk, vg = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            for n, r in (("q", qk), ("k", qk), ("v", vg), ("g", vg)):
                W[x + n] = rnd(r, d)
            W[x + "norm"] = rnd(vg, mean=1.0, std=0.1)
            W[x + "o"] = rnd(d, vg, std=deep)
        elif L["type"] == "mamba2":
            inner, H = m["heads"] * m["vdim"], m["heads"]
            c = inner + 2 * m["groups"] * m["state"]
            W.update({x + "in": rnd(inner + c + H, d), x + "o": rnd(d, inner, std=deep),
                      x + "conv": rnd(c, m["conv"], mean=1.0 / m["conv"], std=0.2),
                      x + "conv.b": rnd(c), x + "dt_bias": rnd(H, mean=-3.0, std=1.0),
                      x + "A_log": rnd(H, mean=0.5, std=0.5), x + "D": rnd(H, mean=1.0, std=0.1),
                      x + "norm": rnd(inner, mean=1.0, std=0.1)})
        else:
            for n, h, s in (("q", "heads", "dim"), ("k", "kv_heads", "dim"),
                            ("v", "kv_heads", "vdim")):
                r = m[h] * m[s]
                W.update({x + n: rnd(r, d), x + n + ".b": rnd(r),
                          x + n + ".conv": rnd(r, m["conv"], mean=1.0 / m["conv"], std=0.2)})
            W[x + "g"] = rnd(m["heads"] * m["vdim"], d)
            W[x + "o"] = rnd(d, m["heads"] * m["vdim"], std=deep)
        for n in ("norm1", "norm1b") + (("norm2", "norm2b") if L["mlp"] else ()):
            W[p + n] = rnd(d, std=0.1)
        if L["mlp"]:
            f = L["mlp"]["ff"]
            W.update({p + "mlp.gate": rnd(f, d), p + "mlp.up": rnd(f, d),
                      p + "mlp.down": rnd(d, f, std=deep)})
    W["final.norm"] = rnd(d, std=0.1)
    W["head"] = rnd(cfg.vocab_size, d)
    return W


_WEIGHTS = {"nomic-bert": _nomic_weights, "bert": _bert_weights, "llama": _llama_weights,
            "zegopel": _zegopel_weights}


def _weights(cfg, seed, device="cuda"):
    return _WEIGHTS[cfg.family](cfg, _maker(seed, device))


def _sequences(case, cfg, seed):
    r = np.random.RandomState(seed % (1 << 31))
    return [r.randint(1000, cfg.vocab_size, n).tolist() for n in _lengths(case)]


# --------------------------------------------------- a decode step's inputs ----
def _pages(case, seed):
    """Pages of every stream in a pool that has been in use: [streams, most] page ids, the
    pool's size, the places of the streams' new tokens."""
    lens = _lengths(case)
    need = [-(-n // PAGE) for n in lens]
    ids = np.random.RandomState((seed + 1) % (1 << 31)).permutation(sum(need)).astype(np.int32)
    table = np.zeros((len(lens), max(need)), np.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = ids[at:at + n]
        at += n
    slots = [int(table[i, (n - 1) // PAGE]) * PAGE + (n - 1) % PAGE for i, n in enumerate(lens)]
    return table, sum(need), slots


def _cache(case, cfg, seed, pages, device="cuda"):
    """Yields each attention layer's cached keys [pages, heads, PAGE, D] and values [pages, heads,
    PAGE / 4, D, 4] (four neighbouring tokens of a channel side by side)."""
    rnd = _maker(seed + 2, device)
    for H, D in _cached_heads(cfg):
        yield rnd(pages, H, PAGE, D, std=1.0), rnd(pages, H, PAGE // 4, D, 4, std=1.0)


def _cached_heads(cfg):
    if cfg.family == "zegopel":
        return [(L["mixer"]["kv_heads"], L["mixer"]["dim"]) for L in cfg.layers
                if L["type"] == "attention"]
    return [(cfg.num_kv_heads, cfg.head_dim)] * cfg.num_layers


def _states(case, cfg, seed, device="cuda"):
    """What the streams of a hybrid decoder keep beside the cache, layer by layer: recurrent
    states [streams, heads, keys, values] and the last inputs of convolutions."""
    rnd, n = _maker(seed + 3, device), case["streams"]
    if cfg.family != "zegopel":
        return
    for L in cfg.layers:
        m = L["mixer"]
        if L["type"] == "lightning":
            yield rnd(n, m["heads"], m["dim"], m["vdim"], std=1.0, dtype=torch.float32)
        elif L["type"] == "mamba2":
            yield rnd(n, m["heads"], m["state"], m["vdim"], std=1.0, dtype=torch.float32)
            yield rnd(n, m["conv"] - 1, m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"],
                      std=1.0)
        else:
            r = m["heads"] * m["dim"] + m["kv_heads"] * (m["dim"] + m["vdim"])
            yield rnd(n, m["conv"] - 1, r, std=1.0)


# ------------------------------------------------------------ prepare, run ----
def prepare(case, seed):
    return dict(case=case, **{"embed": _prepare_embed, "prefill": _prepare_prefill,
                              "decode": _prepare_decode}[case["path"]](case, seed))


def _prepare_embed(case, seed):
    from llm_mcp_amd.engine.embed_engine import EmbeddingEngine
    cfg = _config(case)
    return dict(engine=EmbeddingEngine(cfg, device="cuda", weights=_weights(cfg, seed)),
                seqs=_sequences(case, cfg, seed))


def _engine(cfg, case, seed, seqs, tokens, longest):
    from llm_mcp_amd.engine.engine import EngineConfig, LLMEngine
    ecfg = EngineConfig(model=case["model"], max_num_seqs=seqs, max_batched_tokens=max(64, tokens),
                        mixed_prefill_tokens=0, max_model_len=longest, kv_cache_tokens=tokens,
                        prefix_cache=False, use_graphs=False)
    return LLMEngine(ecfg, device="cuda", model_cfg=cfg, weights=_weights(cfg, seed))


def _prepare_prefill(case, seed):
    cfg = _config(case)
    seqs = _sequences(case, cfg, seed)
    pool = sum(-(-len(s) // PAGE) + 1 for s in seqs) * PAGE
    engine = _engine(cfg, case, seed, len(seqs), pool, max(map(len, seqs)) + PAGE)
    return dict(engine=engine, entries=[(i + 1, s, [len(s) - 1]) for i, s in enumerate(seqs)],
                end=[i + 1 for i in range(len(seqs))])


def _prepare_decode(case, seed):
    from llm_mcp_amd import ops
    from llm_mcp_amd.models.llama import StepInputs
    cfg, n, lens = _config(case), case["streams"], _lengths(case)
    table, pages, slots = _pages(case, seed)
    engine = _engine(cfg, case, seed, n, pages * PAGE, max(lens))

    def dev(x, dtype=torch.int32):
        return torch.as_tensor(np.asarray(x)).to(dtype).cuda()

    rows = StepInputs(
        dev([s[-1] for s in _sequences(case, cfg, seed)]), dev(lens) - 1, dev(slots), n, dev(table),
        dev(lens), dev(np.arange(n + 1)), dev([0, 0]), dev(np.arange(n), torch.int64), n, n,
        decode_order=dev(ops.decode_order(lens)), state_slots=dev(np.arange(n)),
        states=engine.states)
    # as the serving loop: key partitions while there are fewer workgroups than compute units
    parts = max(1, min(16, -(-256 // (n * engine.Hkv))))
    scratch = ops.DecodeWorkspace(n, engine.Hq, engine.D, parts, engine.device)
    greedy = (torch.zeros(n, device="cuda"), dev(np.zeros(n)), torch.ones(n, device="cuda"),
              dev(np.zeros(n), torch.int64), dev(np.zeros(n)))
    out = {}

    def step():
        out["logits"] = engine.model.forward(rows, engine.k_caches, engine.v_caches, scratch)
        out["token"], out["logprob"] = ops.sample(out["logits"], *greedy)

    with torch.no_grad():
        stream = torch.cuda.Stream()
        stream.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(stream):
            step()
        torch.cuda.current_stream().wait_stream(stream)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            step()
    for i, (k, v) in enumerate(_cache(case, cfg, seed, pages)):
        engine.k_caches[i].copy_(k)
        engine.v_caches[i].copy_(v)
    for t, s in zip(engine.states, _states(case, cfg, seed)):
        t.copy_(s)
    return dict(engine=engine, rows=rows, scratch=scratch, greedy=greedy, graph=graph, out=out)


def run(state):
    path = state["case"]["path"]
    if path == "embed":
        return state["engine"].embed_sync(state["seqs"])
    if path == "prefill":
        with torch.inference_mode():
            return state["engine"].feed(state["entries"], state["end"])
    state["graph"].replay()
    # the sampled token is the place of the largest logit: the logits say where that is a tie
    return dict(logits=state["out"]["logits"], logprob=state["out"]["logprob"])


# --------------------------------------------------------- work, tolerance ----
def _products(cfg):
    """Weights that every token is multiplied with, the output layer apart."""
    d = cfg.hidden_size
    if cfg.family == "nomic-bert":
        return cfg.num_layers * (4 * d * d + 3 * d * cfg.intermediate_size)
    if cfg.family == "bert":
        return cfg.num_layers * (4 * d * d + 2 * d * cfg.intermediate_size)
    if cfg.family == "llama":
        D = cfg.head_dim
        return cfg.num_layers * (d * D * (2 * cfg.num_heads + 2 * cfg.num_kv_heads)
                                 + 3 * d * cfg.intermediate_size)
    n = 0
    for L in cfg.layers:
        m = L["mixer"]
        if L["type"] == "lightning":
            n += d * m["heads"] * (2 * m["dim"] + 3 * m["vdim"])
        elif L["type"] == "mamba2":
            n += d * (3 * m["heads"] * m["vdim"] + 2 * m["groups"] * m["state"] + m["heads"])
        else:
            n += d * (m["heads"] * (m["dim"] + 2 * m["vdim"])
                      + m["kv_heads"] * (m["dim"] + m["vdim"]))
        n += 3 * d * L["mlp"]["ff"] if L["mlp"] else 0
    return n


def _mixing(cfg, pairs, tokens):
    """Operations of attention over so many (query, key) pairs and of recurrences over tokens."""
    if cfg.family != "zegopel":
        return 4 * pairs * cfg.num_heads * cfg.head_dim * cfg.num_layers
    n = 0
    for L in cfg.layers:
        m = L["mixer"]
        if L["type"] == "attention":
            n += 2 * pairs * m["heads"] * (m["dim"] + m["vdim"])
        else:
            n += 4 * tokens * m["heads"] * m["vdim"] * m.get("dim", m.get("state"))
    return n


def work(case):
    cfg, lens, path = _config(case), _lengths(case), case["path"]
    products, head = _products(cfg), cfg.vocab_size * cfg.hidden_size
    n, T = len(lens), sum(lens)
    if path == "embed":
        return dict(bytes=2 * products + T * (4 + 2 * cfg.hidden_size) + 4 * n * cfg.embed_dim,
                    flops=2 * products * T + _mixing(cfg, sum(x * x for x in lens), 0))
    cache = sum(4 * H * D for H, D in _cached_heads(cfg))       # bytes of a token's keys and values
    if path == "prefill":
        return dict(bytes=2 * (products + head) + T * (4 + 2 * cfg.hidden_size + cache)
                    + 4 * n * cfg.vocab_size,
                    flops=2 * products * T + 2 * head * n
                    + _mixing(cfg, sum(x * (x + 1) // 2 for x in lens), T))
    states = 0
    for L in cfg.layers if cfg.family == "zegopel" else []:
        m = L["mixer"]
        if L["type"] != "attention":
            states += 8 * m["heads"] * m["vdim"] * m.get("dim", m.get("state"))
    return dict(bytes=2 * (products + head) + T * cache + n * (states + 2 * cfg.vocab_size),
                flops=2 * (products + head) * n + _mixing(cfg, T, n))


def tolerance(case):
    # bf16 activations through 12 to 48 layers: 0.007 to 0.024 off the 64-bit results
    return {"rel": 0.03, "max": 0.3}


# ------------------------------------------------- the same in 64 bits, plainly ----
def exact(case, seed):
    cfg, dev = _config(case), "cuda"
    with torch.no_grad():
        W, seqs = _weights(cfg, seed, dev), _sequences(case, cfg, seed)
        if case["path"] == "embed":
            return _exact_embed(cfg, W, seqs)
        if case["path"] == "prefill":
            one = _exact_zegopel if cfg.family == "zegopel" else _exact_llama
            return torch.stack([one(cfg, W, torch.tensor(s, device=dev)) for s in seqs]).cpu()
        table, pages, _ = _pages(case, seed)
        lens = torch.tensor(_lengths(case), device=dev)
        ids = torch.tensor([s[-1] for s in seqs], device=dev)
        cache, states = _cache(case, cfg, seed, pages, dev), _states(case, cfg, seed, dev)
        step = _exact_zegopel_step if cfg.family == "zegopel" else _exact_llama_step
        logits = step(cfg, W, ids, lens, torch.tensor(table, device=dev).long(), cache, states)
        return dict(logits=logits, logprob=torch.log_softmax(logits, -1).max(-1).values)


def _mul(x, w):
    return x @ w.to(F64).T


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, w, b, eps):
    x = x - x.mean(-1, keepdim=True)
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w.to(F64) + b.to(F64)


def _frequencies(cfg, device):
    f = cfg.rope_theta ** (-torch.arange(0, cfg.head_dim, 2, dtype=F64, device=device) / cfg.head_dim)
    s = getattr(cfg, "rope_scaling", None)
    if s:
        wave, old = 2 * math.pi / f, s["original_max_position_embeddings"]
        lo, hi = s["low_freq_factor"], s["high_freq_factor"]
        mix = ((old / wave - lo) / (hi - lo)).clamp(0, 1)
        f = (1 - mix) * f / s["factor"] + mix * f
    return f


def _rotate(x, pos, freq):
    """x [T, heads, D]: channels i and i + D / 2 are a pair."""
    a = (pos.to(F64)[:, None] * freq)[:, None]
    u, v = x.chunk(2, -1)
    return torch.cat([u * a.cos() - v * a.sin(), v * a.cos() + u * a.sin()], -1)


def _attend(q, k, v, scale, causal):
    """q [T, H, D], k and v [T, G, D]; query head h reads head h // (H / G)."""
    T, H, _ = q.shape
    out = torch.empty((T, H, v.shape[2]), dtype=F64, device=q.device)
    for h in range(H):
        g = h // (H // k.shape[1])
        s = (q[:, h] @ k[:, g].T) * scale
        if causal:
            s.masked_fill_(torch.ones(T, T, dtype=torch.bool, device=q.device).triu(1), -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, g]
    return out.reshape(T, -1)


def _exact_embed(cfg, W, seqs):
    H, D, eps, dev = cfg.num_heads, cfg.head_dim, cfg.ln_eps, W["word"].device
    nomic = cfg.family == "nomic-bert"
    lens = [len(s) for s in seqs]
    pos = torch.cat([torch.arange(n, device=dev) for n in lens])
    x = W["word"][torch.tensor([t for s in seqs for t in s], device=dev)].to(F64) + W["type"][0].to(F64)
    x = _layer_norm(x if nomic else x + W["pos"][pos].to(F64), W["emb_ln_w"], W["emb_ln_b"], eps)
    for L in W["layers"]:
        qkv = _mul(x, L["wqkv"]) + (0 if nomic else L["bqkv"].to(F64))
        q, k, v = (t.reshape(-1, H, D) for t in qkv.chunk(3, -1))
        if nomic:
            freq = _frequencies(cfg, dev)
            q, k = _rotate(q, pos, freq), _rotate(k, pos, freq)
        a = torch.cat([_attend(*t, D ** -0.5, False)
                       for t in zip(q.split(lens), k.split(lens), v.split(lens))])
        x = _layer_norm(x + _mul(a, L["wo"]) + (0 if nomic else L["bo"].to(F64)),
                        L["ln1_w"], L["ln1_b"], eps)
        if nomic:
            g, u = _mul(x, L["w_gate_up"]).chunk(2, -1)
            y = _mul(torch.nn.functional.silu(g) * u, L["w_down"])
        else:
            y = torch.nn.functional.gelu(_mul(x, L["w1"]) + L["b1"].to(F64))
            y = _mul(y, L["w2"]) + L["b2"].to(F64)
        x = _layer_norm(x + y, L["ln2_w"], L["ln2_b"], eps)
    e = torch.stack([t[0] if getattr(cfg, "pooling", "mean") == "cls" else t.mean(0)
                     for t in x.split(lens)])
    return (e / e.norm(dim=-1, keepdim=True)).cpu()


def _llama_layers(cfg, W, x, pos, attend):
    """attend(layer, q, k, v) on rotated heads."""
    H, G, D, freq = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, _frequencies(cfg, x.device)
    for i, L in enumerate(W["layers"]):
        qkv = _mul(_rms(x, cfg.rms_eps) * L["ln1"].to(F64), L["wqkv"]).reshape(len(x), -1, D)
        q, k, v = qkv.split((H, G, G), 1)
        x = x + _mul(attend(_rotate(q, pos, freq), _rotate(k, pos, freq), v), L["wo"])
        g, u = _mul(_rms(x, cfg.rms_eps) * L["ln2"].to(F64), L["w_gate_up"]).chunk(2, -1)
        x = x + _mul(torch.nn.functional.silu(g) * u, L["w_down"])
    return x


def _exact_llama(cfg, W, ids):
    pos = torch.arange(len(ids), device=ids.device)
    x = _llama_layers(cfg, W, W["embed"][ids].to(F64), pos,
                      lambda q, k, v: _attend(q, k, v, cfg.head_dim ** -0.5, True))
    return _mul(_rms(x[-1:], cfg.rms_eps) * W["norm"].to(F64), W["lm_head"])[0]


def _attend_cached(q, k, v, scale, lens, table, cache):
    """q [B, H, D] of each stream's last token, its k and v [B, G, D] beside the cached ones."""
    kc, vc = next(cache)
    B, H, _ = q.shape
    out = torch.empty((B, H, v.shape[2]), dtype=F64, device=q.device)
    for b in range(B):
        n = int(lens[b])
        at = table[b, :-(-n // PAGE)]
        ks = kc[at].transpose(0, 1).flatten(1, 2)[:, :n].to(F64)           # [G, n, D]
        vs = vc[at].transpose(-1, -2).flatten(2, 3).transpose(0, 1).flatten(1, 2)[:, :n].to(F64)
        ks[:, -1], vs[:, -1] = k[b], v[b]
        s = (q[b].reshape(ks.shape[0], -1, ks.shape[2]) @ ks.transpose(1, 2)) * scale
        out[b] = (torch.softmax(s, -1) @ vs).reshape(H, -1)
    return out.reshape(B, -1)


def _exact_llama_step(cfg, W, ids, lens, table, cache, _):
    x = _llama_layers(cfg, W, W["embed"][ids].to(F64), lens - 1,
                      lambda q, k, v: _attend_cached(q, k, v, cfg.head_dim ** -0.5, lens, table,
                                                     cache))
    return _mul(_rms(x, cfg.rms_eps) * W["norm"].to(F64), W["lm_head"])


def _conv(u, w, tail=None):
    """u [T, C], w [C, taps], zeros before the first row; with a tail [B, taps - 1, C] every row
    is the next input of its own sequence."""
    w = w.to(F64)
    taps = w.shape[1]
    if tail is not None:
        return (torch.cat([tail.to(F64), u[:, None]], 1) * w.T).sum(1)
    pad = torch.cat([u.new_zeros(taps - 1, u.shape[1]), u])
    return sum(pad[j:j + len(u)] * w[:, j] for j in range(taps))


def _recur(q, k, v, logdecay, state):
    """S <- decay S + k v^T, o = S^T q per head: a whole sequence q, k [T, H, N], v [T, H, P],
    logdecay [T, H] from zero (every token's weight of every earlier one), or one token of each
    sequence from its state [T, H, N, P]."""
    if state is not None:
        S = logdecay.exp()[:, :, None, None] * state.to(F64) + k[..., None] * v[:, :, None]
        return (S * q[..., None]).sum(2)
    total, out = logdecay.cumsum(0), torch.empty_like(v)
    later = torch.ones(len(q), len(q), dtype=torch.bool, device=q.device).triu(1)
    for h in range(q.shape[1]):
        w = (total[:, None, h] - total[None, :, h]).masked_fill_(later, -math.inf).exp_()
        out[:, h] = (w * (q[:, h] @ k[:, h].T)) @ v[:, h]
    return out


def _zegopel_layers(cfg, W, x, pos, attend, states):
    silu, sigmoid, eps = torch.nn.functional.silu, torch.sigmoid, cfg.rms_eps

    def norm(y, name):
        return _rms(y, eps) * (1.0 + W[name].to(F64))

    for i, L in enumerate(cfg.layers):
        m, p = L["mixer"], "l%d.mix." % i
        h, T = norm(x, "l%d.norm1" % i), len(x)
        if L["type"] == "lightning":
            H, N, P = m["heads"], m["dim"], m["vdim"]
            q, k, v = (silu(_mul(h, W[p + n])).reshape(T, H, -1) for n in "qkv")
            decay = torch.tensor(m["decay"], dtype=F64, device=x.device).log().expand(T, H)
            o = _recur(q, k, v, decay, next(states) if states else None).reshape(T, -1)
            y = _rms(o, eps) * W[p + "norm"].to(F64) * sigmoid(_mul(h, W[p + "g"]))
        elif L["type"] == "mamba2":
            H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            z, u, dt = _mul(h, W[p + "in"]).split((H * P, H * P + 2 * G * N, H), -1)
            S, tail = (next(states), next(states)) if states else (None, None)
            u = silu(_conv(u, W[p + "conv"], tail) + W[p + "conv.b"].to(F64))
            v, B, C = u.split((H * P, G * N, G * N), -1)
            v = v.reshape(T, H, P)
            B, C = (t.reshape(T, G, N).repeat_interleave(H // G, 1) for t in (B, C))
            dt = torch.nn.functional.softplus(dt + W[p + "dt_bias"].to(F64))
            o = _recur(C, B * dt[..., None], v, -W[p + "A_log"].to(F64).exp() * dt, S)
            o = (o + W[p + "D"].to(F64)[:, None] * v).reshape(T, -1) * silu(z)
            y = _rms(o.reshape(T, m["norm_groups"], -1), eps).reshape(T, -1) * W[p + "norm"].to(F64)
        else:
            H, G, e = m["heads"], m["kv_heads"], m["vdim"]
            sizes = (H * m["dim"], G * m["dim"], G * e)
            tails = next(states).split(sizes, -1) if states else (None,) * 3
            q, k, v = (_conv(_mul(h, W[p + n]) + W[p + n + ".b"].to(F64), W[p + n + ".conv"], t)
                       for n, t in zip("qkv", tails))
            t = m["q_temp"]
            hot = 1 + t["coef"] * torch.log(torch.floor((pos.to(F64) + 1) / t["every"]) + 1)
            q = _rms(q.reshape(T, H, -1), eps) * hot[:, None, None]
            k = _rms(k.reshape(T, G, -1), eps)
            y = attend(q, k, v.reshape(T, G, -1), m["scale"]) * sigmoid(_mul(h, W[p + "g"]))
        x = x + norm(_mul(y, W[p + "o"]), "l%d.norm1b" % i)
        if L["mlp"]:
            f, h = "l%d.mlp." % i, norm(x, "l%d.norm2" % i)
            y = _mul(torch.relu(_mul(h, W[f + "gate"])) * _mul(h, W[f + "up"]), W[f + "down"])
            x = x + norm(y, "l%d.norm2b" % i)
    return x


def _exact_zegopel(cfg, W, ids):
    x = _zegopel_layers(cfg, W, W["embed"][ids].to(F64), torch.arange(len(ids), device=ids.device),
                        lambda q, k, v, scale: _attend(q, k, v, scale, True), None)
    return _mul(_rms(x[-1:], cfg.rms_eps) * (1 + W["final.norm"].to(F64)), W["head"])[0]


def _exact_zegopel_step(cfg, W, ids, lens, table, cache, states):
    x = _zegopel_layers(cfg, W, W["embed"][ids].to(F64), lens - 1,
                        lambda q, k, v, scale: _attend_cached(q, k, v, scale, lens, table, cache),
                        states)
    return _mul(_rms(x, cfg.rms_eps) * (1 + W["final.norm"].to(F64)), W["head"])
