"""The work that is timed: steps of the engine as its users issue them.

A case is one model and one pass of its engine.  Two kinds of pass:

  step      one call of ``Engine.step`` and the sampling of its tokens, what the scheduler does once per step: ``held``
            requests bring one token each (decoding), ``portions`` requests bring a part of a prompt (prefill); either may be
            none.  The MiniCPM shapes run so.  Afterwards every request is back where it was (a decoding request is
            cut down to its cached prefix, a prompt is dropped), so that a pass can be repeated.
  lifetime  requests from their prompts to their last token: one step over all prompts, then ``steps`` steps of one token
            each, then they are freed.  The designs with recurrent state run so (such a state does not go backwards).

Weights are random with the spread of a trained model's (unit gain per product), tokens are uniform, the cached tokens are what
the model itself computed for them.  Requests that hold a context hold prefixes of one document (a system prompt or a chat's
history, copied with ``Engine.fork``): every copy has pages of its own.
"""
import math

import torch

PAGE = 64
MAX_BATCH = 64

# MiniCPM-shaped models: benchmark and tests of this repository use these three sizes.
MINICPM = {
    "1b": dict(vocab_size=73440, hidden_size=1536, num_hidden_layers=52, num_attention_heads=24, num_key_value_heads=8,
               intermediate_size=3840, rms_norm_eps=1e-5, max_position_embeddings=4096, tie_word_embeddings=True),
    "2b": dict(vocab_size=122753, hidden_size=2304, num_hidden_layers=40, num_attention_heads=36, num_key_value_heads=36,
               intermediate_size=5760, rms_norm_eps=1e-5, max_position_embeddings=4096, tie_word_embeddings=True),
    "8b": dict(vocab_size=73448, hidden_size=4096, num_hidden_layers=32, num_attention_heads=32, num_key_value_heads=2,
               intermediate_size=16384, rms_norm_eps=1e-6, max_position_embeddings=32768, tie_word_embeddings=False),
}
SCALE_EMB, DIM_MODEL_BASE, SCALE_DEPTH, ROPE_THETA = 12, 256, 1.4, 10000.0

# Layer sizes of the benchmark's list of designs (four layers each).
SIZES = {
    "1b": dict(width=1536, heads=24, kv=8, dim=64, ff=3840, vocab=32000, window=512),
    "2b": dict(width=2304, heads=36, kv=36, dim=64, ff=5760, vocab=32000, window=1024),
    "8b": dict(width=4096, heads=32, kv=8, dim=128, ff=14336, vocab=32000, window=2048),
}
EPS = 1e-5


# ---- the cases ------------------------------------------------------------------------------------------------------------
def _step(name, model, dtype="bf16", held=0, past=(0, 0), portions=0, new=(0, 0), portion_past=0, sampled=False):
    return dict(name=name, kind="step", model=model, dtype=dtype, held=held, past_min=past[0], past_max=past[1], portions=portions,
                new_min=new[0], new_max=new[1], portion_past=portion_past, sampled=sampled)


def _life(name, model, size, prompts, new, steps):
    return dict(name=name, kind="lifetime", model=model, size=size, dtype="bf16", portions=prompts, new_min=new[0], new_max=new[1],
                steps=steps)


def listed():
    return [
        # one user in a short chat: every token waits for the whole step, launches count
        _step("reply_1b_batch1", "1b", held=1, past=(257, 257)),
        # one user, a full page of history: weights and one cache are read once per token
        _step("reply_2b_batch1", "2b", held=1, past=(2063, 2063)),
        # the benchmark's headline: eight users decode together
        _step("decode_2b_batch8", "2b", held=8, past=(1900, 2100)),
        # a busy server: 64 users with histories of all lengths, sampled with temperature, top-k and top-p
        _step("decode_2b_batch64", "2b", held=64, past=(300, 2100), sampled=True),
        # four users over long documents
        _step("decode_8b_long", "8b", held=4, past=(16301, 16384)),
        # a whole prompt in one step: time to the first token
        _step("prompt_2b_2048", "2b", portions=1, new=(2048, 2048)),
        # several short questions arrive together
        _step("prompts_1b_short", "1b", portions=7, new=(19, 301)),
        # continuous batching: prompts in portions beside the users that decode, a budget of about a thousand tokens
        _step("mixed_1b", "1b", held=40, past=(100, 2048), portions=2, new=(463, 512), portion_past=512),
        # a long document in one step, the largest call
        _step("prompt_8b_16384", "8b", portions=1, new=(16384, 16384)),
        # true 32-bit: a portion beside eight users
        _step("mixed_1b_float32", "1b", dtype="fp32", held=8, past=(100, 900), portions=1, new=(509, 509), portion_past=130),
        # designs with recurrent and latent mixers, requests from prompt to last token
        _life("life_mezinex_8b", "mezinex", "8b", 4, (400, 1100), 8),
        _life("life_fokinex_2b", "fokinex", "2b", 2, (1500, 2500), 8),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    what = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "mixed", "mixed", "fp32", "life", "life"])
    if what == "decode":
        model = rng.choice(["1b", "2b", "8b"])
        held = _log_int(rng, 1, 64)
        longest = _log_int(rng, 64, min(16384 if model == "8b" else 4000, 140000 // held))
        return _drawn(_step("", model, held=held, past=(_log_int(rng, 16, longest), longest), sampled=rng.random() < 0.4))
    if what == "prompt":
        model = rng.choice(["1b", "2b", "8b"])
        portions = _log_int(rng, 1, 8)
        longest = _log_int(rng, 17, 4000 // portions)
        return _drawn(_step("", model, portions=portions, new=(_log_int(rng, 2, longest), longest),
                            portion_past=rng.choice([0, 0, _log_int(rng, 1, 2000) if longest < 2000 else 0])))
    if what == "mixed":
        longest = _log_int(rng, 100, 3500)
        return _drawn(_step("", rng.choice(["1b", "2b", "8b"]), held=_log_int(rng, 1, 60), past=(_log_int(rng, 16, longest), longest),
                            portions=rng.randint(1, 3), new=(_log_int(rng, 2, 100), _log_int(rng, 100, 700)),
                            portion_past=rng.choice([0, _log_int(rng, 1, 3000)]), sampled=rng.random() < 0.4))
    if what == "fp32":
        longest = _log_int(rng, 32, 2000)
        portions = rng.randint(0, 2)
        return _drawn(_step("", "1b", dtype="fp32", held=_log_int(rng, 1, 32), past=(_log_int(rng, 16, longest), longest),
                            portions=portions, new=(_log_int(rng, 2, 50), _log_int(rng, 50, 600)) if portions else (0, 0),
                            portion_past=rng.choice([0, _log_int(rng, 1, 1500)]) if portions else 0))
    prompts = _log_int(rng, 1, 8)
    longest = _log_int(rng, 20, 3000 // prompts)
    return _drawn(_life("", rng.choice(["mezinex", "fokinex"]), rng.choice(["1b", "2b", "8b"]), prompts,
                        (_log_int(rng, 2, longest), longest), rng.randint(2, 10)))


def _drawn(case):
    del case["name"]
    return case


def _spread(n, lo, hi):
    """n lengths between lo and hi, spread evenly over their logarithm in a shuffled order, the longest among them."""
    if n == 0:
        return []
    at = [1.0] + [(i * 0.6180339887498949) % 1.0 for i in range(1, n)]
    return [int(round(lo * (hi / lo) ** a)) for a in at]


def _held(case):
    return _spread(case.get("held", 0), case.get("past_min", 0), case.get("past_max", 0))


def _portions(case):
    return _spread(case["portions"], case["new_min"], case["new_max"])


def _dtype(case):
    return torch.bfloat16 if case["dtype"] == "bf16" else torch.float32


# ---- inputs: weights and tokens, from the seed alone --------------------------------------------------------------------------
class _Draw:
    """Tensors from one seeded generator on the GPU, in the order in which they are asked for."""

    def __init__(self, seed, dtype):
        self.g = torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + 17)
        self.dtype = dtype

    def matrix(self, rows, cols, gain=1.0):
        t = torch.empty(rows, cols, dtype=self.dtype, device="cuda")
        return t.normal_(0.0, gain / math.sqrt(cols), generator=self.g)

    def table(self, rows, cols, std):
        return torch.empty(rows, cols, dtype=self.dtype, device="cuda").normal_(0.0, std, generator=self.g)

    def vector(self, n, mean=1.0, std=0.1):
        return torch.empty(n, dtype=torch.float32, device="cuda").normal_(mean, std, generator=self.g).bfloat16().float()


def _minicpm_config(model):
    return dict(MINICPM[model], model_type="minicpm", scale_emb=SCALE_EMB, dim_model_base=DIM_MODEL_BASE, scale_depth=SCALE_DEPTH,
                rope_theta=ROPE_THETA, eos_token_id=2)


def _minicpm_weights(model, seed, dtype):
    c, w = MINICPM[model], _Draw(seed, dtype)
    d, di, nh, nkv = c["hidden_size"], c["intermediate_size"], c["num_attention_heads"], c["num_key_value_heads"]
    dh = d // nh
    W = {"model.embed_tokens.weight": w.table(c["vocab_size"], d, 1.0 / SCALE_EMB if not c["tie_word_embeddings"] else 0.05)}
    W["lm_head.weight"] = W["model.embed_tokens.weight"] if c["tie_word_embeddings"] else w.table(c["vocab_size"], d, 0.02)
    W["model.norm.weight"] = w.vector(d)
    for i in range(c["num_hidden_layers"]):
        p = "model.layers.%d." % i
        W[p + "input_layernorm.weight"], W[p + "post_attention_layernorm.weight"] = w.vector(d), w.vector(d)
        W[p + "self_attn.q_proj.weight"], W[p + "self_attn.k_proj.weight"] = w.matrix(nh * dh, d, 1.2), w.matrix(nkv * dh, d, 1.2)
        W[p + "self_attn.v_proj.weight"], W[p + "self_attn.o_proj.weight"] = w.matrix(nkv * dh, d), w.matrix(d, nh * dh)
        W[p + "mlp.gate_proj.weight"], W[p + "mlp.up_proj.weight"] = w.matrix(di, d), w.matrix(di, d)
        W[p + "mlp.down_proj.weight"] = w.matrix(d, di, 1.5)
    return W


def _design_config(model, size):
    """The benchmark's configurations of the two designs: four layers, every mixer of the design among them."""
    z = SIZES[size]
    big = z["dim"] >= 128
    latent = dict(heads=z["heads"], dim=z["dim"], rot_dim=64 if big else 32, vdim=z["dim"], q_rank=z["width"] // 3 // 64 * 64,
                  kv_rank=512 if big else 256, scale=(z["dim"] + (64 if big else 32)) ** -0.5,
                  rot=dict(base=1000000.0, dims=64 if big else 32))
    ff = dict(kind="dense", ff=z["ff"])
    if model == "mezinex":
        rglru = dict(width=z["width"], blocks=z["heads"], conv=4)
        ssm = dict(heads=2 * z["width"] // 64, vdim=64, state=128, groups=8, norm_groups=8, conv=4)
        kinds = [("latent_attention", latent), ("rglru", rglru), ("mamba2", ssm), ("latent_attention", latent)]
        return dict(architecture="Mezinex", vocab=z["vocab"], width=z["width"], norm=dict(eps=EPS), logit_scale=1.0, streams=2,
                    embedding=dict(bigram=dict(buckets=65521, mul_prev=127, mul_cur=17)),
                    layers=[dict(type=k, mixer=m, mlp=ff) for k, m in kinds])
    latent = dict(latent, mask=dict(size=z["window"]),
                  rot=dict(latent["rot"], scaling=dict(factor=16.0, original=1024, fast=32.0, slow=1.0)))
    both = dict(left=dict(heads=z["heads"], kv_heads=z["kv"], dim=z["dim"], vdim=z["dim"], scale=z["dim"] ** -0.5, softcap=50.0,
                          mask=dict(size=z["window"])),
                right=dict(heads=z["heads"], kv_heads=z["heads"] // 4, dim=z["dim"], vdim=z["dim"], conv=4),
                left_scale=0.7, right_scale=0.7)
    return dict(architecture="Fokinex", vocab=z["vocab"], width=z["width"], norm=dict(eps=EPS), embedding=dict(scale=1.0),
                layers=[dict(type="latent_attention", mixer=latent, mlp=ff), dict(type="parallel", mixer=both, mlp=ff),
                        dict(type="latent_attention", mixer=dict(latent, kv_from=0), mlp=ff),
                        dict(type="latent_attention", mixer=latent, mlp=ff)])


def _design_weights(model, size, seed):
    cfg, w = _design_config(model, size), _Draw(seed, torch.bfloat16)
    d, V = cfg["width"], cfg["vocab"]
    W = {"embed": w.table(V, d, 1.0), "head": w.matrix(V, d), "final.norm": w.vector(d)}
    if model == "mezinex":
        W["bigram"] = w.table(cfg["embedding"]["bigram"]["buckets"] + 1, d, 0.5)

    def latent(p, m, gated):
        H, R, E, q = m["heads"], m["kv_rank"], m["rot_dim"], m["q_rank"]
        W[p + "dq"], W[p + "dq.norm"], W[p + "uq"] = w.matrix(q, d), w.vector(q), w.matrix(H * (m["dim"] + E), q)
        if m.get("kv_from") is None:
            W[p + "dkv"], W[p + "dkv.norm"] = w.matrix(R + E, d), w.vector(R)
        W[p + "uk"], W[p + "uv"] = w.matrix(H * m["dim"], R), w.matrix(H * m["vdim"], R)
        if gated:
            W[p + "g"] = w.matrix(H * m["vdim"], d)
        else:
            W[p + "sink"] = w.vector(H, 0.5, 1.0)
        W[p + "o"] = w.matrix(d, H * m["vdim"])

    def conv(p, channels, taps):
        W[p] = w.vector(channels * taps, 0.0, 0.5).view(channels, taps)

    for i, l in enumerate(cfg["layers"]):
        p, m = "l%d." % i, l["mixer"]
        W[p + "norm1"] = w.vector(d)
        if l["type"] == "latent_attention":
            latent(p + "mix.", m, model == "mezinex")
        elif l["type"] == "rglru":
            n, b = m["width"], m["blocks"]
            for k in ("y", "x"):
                W[p + "mix." + k], W[p + "mix." + k + ".b"] = w.matrix(n, d), w.vector(n, 0.0)
            conv(p + "mix.conv", n, m["conv"])
            W[p + "mix.conv.b"], W[p + "mix.lam"], W[p + "mix.o"] = w.vector(n, 0.0), w.vector(n, -3.0, 1.0), w.matrix(d, n)
            for k in ("ra", "ri"):
                W[p + "mix." + k] = w.matrix(b * (n // b), n // b).view(b, n // b, n // b)
                W[p + "mix." + k + ".b"] = w.vector(n, 0.0).view(b, n // b)
        elif l["type"] == "mamba2":
            inner, gn = m["heads"] * m["vdim"], m["groups"] * m["state"]
            W[p + "mix.in"] = w.matrix(2 * inner + 2 * gn + m["heads"], d)
            conv(p + "mix.conv", inner + 2 * gn, m["conv"])
            W[p + "mix.conv.b"], W[p + "mix.dt_bias"] = w.vector(inner + 2 * gn, 0.0), w.vector(m["heads"], -2.0, 0.5)
            W[p + "mix.A_log"], W[p + "mix.D"] = w.vector(m["heads"], 0.5, 0.5), w.vector(m["heads"])
            W[p + "mix.norm"], W[p + "mix.o"] = w.vector(inner), w.matrix(d, inner)
        else:
            a, b = m["left"], m["right"]
            L, R = p + "mix.left.", p + "mix.right."
            H, G, n = a["heads"], a["kv_heads"], a["dim"]
            W[L + "q"], W[L + "k"], W[L + "g"], W[L + "o"] = w.matrix(H * n, d), w.matrix(G * n, d), w.matrix(H * n, d), w.matrix(d, H * n)
            W[L + "q.norm"], W[L + "k.norm"] = w.vector(H * n), w.vector(G * n)
            H, G, dk, dv = b["heads"], b["kv_heads"], b["dim"], b["vdim"]
            for k, c in (("q", G * dk), ("k", G * dk), ("v", H * dv)):
                W[R + k] = w.matrix(c, d)
                conv(R + k + ".conv", c, b["conv"])
            W[R + "b"], W[R + "a"] = w.matrix(H, d), w.matrix(H, d)
            W[R + "A_log"], W[R + "dt_bias"] = w.vector(H, -1.0, 0.7), w.vector(H, -2.0, 0.7)
            W[R + "norm"], W[R + "g"], W[R + "o"] = w.vector(dv), w.matrix(H * dv, d), w.matrix(d, H * dv)
        f = l["mlp"]["ff"]
        W[p + "norm2"], W[p + "mlp.gate"], W[p + "mlp.up"], W[p + "mlp.down"] = w.vector(d), w.matrix(f, d), w.matrix(f, d), w.matrix(d, f)
        if model == "mezinex":
            for q in ("1", "2"):
                W[p + "hc" + q + ".in"], W[p + "hc" + q + ".out"] = w.vector(2, 0.5, 0.1), w.vector(2, 0.7, 0.1)
                W[p + "hc" + q + ".mix"] = (torch.eye(2, device="cuda") + w.vector(4, 0.0, 0.1).view(2, 2)).bfloat16().float()
        else:
            del W[p + "norm2"]
    return W


def _tokens(case, seed):
    """(the document, one new token per holding request, the portions' tokens, per later step one token per request), as lists."""
    g = torch.Generator().manual_seed(7919 * int(seed) + 3)
    vocab = MINICPM[case["model"]]["vocab_size"] if case["kind"] == "step" else SIZES[case["size"]]["vocab"]
    some = lambda n: torch.randint(0, vocab, (n,), generator=g).tolist()
    held, portions = _held(case), _portions(case)
    doc = some(max(held + [case.get("portion_past", 0) if portions else 0, 1]))
    later = [some(len(portions)) for _ in range(case.get("steps", 0))]
    return doc, some(len(held)), [some(n) for n in portions], later


def _uniforms(n):
    return [(0.5 + i * 0.7548776662466927) % 1.0 for i in range(n)]


def prepare(case, seed):
    """The engine with its weights, the requests that are in flight with their caches, the step's tokens as lists.  The step has been
    issued before (as every step but the first of a server's life)."""
    from infinicore_infer_amd.config import config_from_dict
    from infinicore_infer_amd.engine import Engine, StepEntry
    from infinicore_infer_amd.parts import Runtime, build_model
    minicpm = case["kind"] == "step"
    conf = config_from_dict(_minicpm_config(case["model"]) if minicpm else _design_config(case["model"], case["size"]))
    model = build_model(conf.model_spec(), Runtime(dtype=_dtype(case), device="cuda:0"))
    model.load_weights(_minicpm_weights(case["model"], seed, _dtype(case)) if minicpm
                       else _design_weights(case["model"], case["size"], seed))
    held, portions = _held(case), _portions(case)
    doc, fresh, parts, later = _tokens(case, seed)
    past = case.get("portion_past", 0)
    pages = lambda n: (n + PAGE - 1) // PAGE
    total = pages(len(doc)) + sum(pages(n + 1) for n in held) + sum(pages(past + n + len(later)) for n in portions)
    engine = Engine(model, max_tokens=total * PAGE, page_size=PAGE, max_requests=len(held) + len(portions) + 1, graph_max_batch=MAX_BATCH)
    ids = ["h%d" % i for i in range(len(held))]
    if held or past:
        engine.step([StepEntry("doc", doc, [])])
        for rid, n in zip(ids, held):
            engine.fork("doc", rid, n)
        for i in range(len(portions) if past else 0):
            engine.fork("doc", "p%d" % i, past)
        engine.free("doc")
    state = dict(engine=engine, entry=StepEntry, ids=ids, held=held, fresh=fresh, parts=parts, past=past, later=later, turn=0,
                 sampling=None)
    if case.get("sampled"):
        n = len(held) + len(portions)
        state["sampling"] = ([0.8] * n, [50] * n, [0.9] * n, _uniforms(n))
    state["tokens_too"] = minicpm and len(held) + len(portions) >= 32
    run(state)
    run(state)
    return state


def run(state):
    engine, entry = state["engine"], state["entry"]
    prompt = lambda i, toks: entry("p%d" % i, toks, [len(toks) - 1])
    if state["later"]:
        # lifetimes: all prompts in one step, then token by token
        n = len(state["parts"])
        logits = [engine.step([prompt(i, toks) for i, toks in enumerate(state["parts"])]).clone()]
        for toks in state["later"]:
            logits.append(engine.step([entry("p%d" % i, [toks[i]], [0]) for i in range(n)]).clone())
            engine.sample_ahead(logits[-1])
        for i in range(n):
            engine.free("p%d" % i)
        return logits
    entries = [entry(rid, [t], [0]) for rid, t in zip(state["ids"], state["fresh"])]
    ends = ("", "'")
    was, now = ends[state["turn"]], ends[state["turn"] ^ 1]
    if state["past"]:
        entries += [entry("p%d%s" % (i, was), toks, [len(toks) - 1]) for i, toks in enumerate(state["parts"])]
    else:
        entries += [prompt(i, toks) for i, toks in enumerate(state["parts"])]
    logits = engine.step(entries)
    if state["sampling"] is None:
        tokens, _ = engine.sample_ahead(logits)
    else:
        tokens, _ = engine.sample_ahead(logits, *state["sampling"])
    # back to the cached prefixes: the same request goes on from them under its other name
    ids = state["ids"]
    for k, n in enumerate(state["held"]):
        ids[k] = "h%d%s" % (k, now)
        engine.adopt("h%d%s" % (k, was), ids[k], n)
    for i in range(len(state["parts"])):
        if state["past"]:
            engine.adopt("p%d%s" % (i, was), "p%d%s" % (i, now), state["past"])
        else:
            engine.free("p%d" % i)
    state["turn"] ^= 1
    # (a token drawn from near-equal logits may differ between correct implementations: returned where many are drawn)
    return [logits, tokens] if state["tokens_too"] else [logits]


# ---- what a pass cannot do without ------------------------------------------------------------------------------------------------
def work(case):
    eb = 2 if case["dtype"] == "bf16" else 4
    held, portions = _held(case), _portions(case)
    if case["kind"] == "step":
        c, past = MINICPM[case["model"]], case["portion_past"]
        d, L, di, V = c["hidden_size"], c["num_hidden_layers"], c["intermediate_size"], c["vocab_size"]
        nh, nkv = c["num_attention_heads"], c["num_key_value_heads"]
        dh = d // nh
        layer = (nh + 2 * nkv) * dh * d + nh * dh * d + 3 * d * di
        rows, wanted = len(held) + sum(portions), len(held) + len(portions)
        pairs = sum(n + 1 for n in held) + sum(past * n + n * (n + 1) // 2 for n in portions)
        tokens = sum(n + 1 for n in held) + sum(past + n for n in portions)
        return {"bytes": eb * (L * layer + V * d) + 2 * L * nkv * dh * eb * tokens + 4 * wanted * V,
                "flops": 2.0 * rows * L * layer + 4.0 * L * nh * dh * pairs + 2.0 * wanted * V * d}
    cfg, steps, B = _design_config(case["model"], case["size"]), case["steps"], len(portions)
    d, V = cfg["width"], cfg["vocab"]
    total = sum(portions)
    weights, flops, cache = V * d, 2.0 * V * d * B * (1 + steps), 0.0

    def pairs(n, window):            # (query, key) pairs of a prompt of n tokens
        w = min(n, window) if window else n
        return w * (w + 1) / 2.0 + (n - w) * w

    def decode_keys(window):         # keys seen by all later tokens together
        return sum(min(n + s + 1, window or 1 << 30) for n in portions for s in range(steps))

    def attention(qk, pv, row, window):
        nonlocal flops, cache
        flops += 2.0 * (qk + pv) * sum(pairs(n, window) for n in portions) + 2.0 * (qk + pv) * decode_keys(window)
        cache += row * (total + decode_keys(window))

    def recurrence(state):
        nonlocal flops, cache
        flops += 6.0 * state * (total + B * steps)
        cache += 4 * state * B * (1 + 2 * steps)

    for l in cfg["layers"]:
        m, n = l["mixer"], 3 * d * l["mlp"]["ff"]
        if l["type"] == "latent_attention":
            H, R, E, q = m["heads"], m["kv_rank"], m["rot_dim"], m["q_rank"]
            n += q * d + H * (m["dim"] + E) * q + H * (m["dim"] + m["vdim"]) * R + H * m["vdim"] * d
            n += H * m["vdim"] * d if case["model"] == "mezinex" else 0
            n += (R + E) * d if m.get("kv_from") is None else 0
            attention(H * (m["dim"] + E), H * m["vdim"], eb * (R + E), (m.get("mask") or {}).get("size"))
        elif l["type"] == "rglru":
            n += 3 * m["width"] * d + 2 * m["width"] * (m["width"] // m["blocks"])
            recurrence(m["width"])
        elif l["type"] == "mamba2":
            inner = m["heads"] * m["vdim"]
            n += (2 * inner + 2 * m["groups"] * m["state"] + m["heads"]) * d + d * inner
            recurrence(inner * m["state"])
        else:
            a, b = m["left"], m["right"]
            n += (2 * a["heads"] + a["kv_heads"]) * a["dim"] * d + d * a["heads"] * a["dim"]
            n += (2 * b["kv_heads"] * b["dim"] + 2 * b["heads"] * b["vdim"] + 2 * b["heads"]) * d + d * b["heads"] * b["vdim"]
            attention(a["heads"] * a["dim"], a["heads"] * a["dim"], 2 * eb * a["kv_heads"] * a["dim"], a["mask"]["size"])
            recurrence(b["heads"] * b["dim"] * b["vdim"])
        weights += n
        flops += 2.0 * n * (total + B * steps)
    return {"bytes": eb * weights * (1 + steps) + cache + 4.0 * V * B * (1 + steps), "flops": flops}


def tolerance(case):
    """Four times what the listed cases show against ``exact``: 1e-2 in bfloat16 (activations rounded between the products of 32 to
    52 layers), 3.4e-6 in float32; the largest of some 100,000 logits is about five times the mean error away.  Tokens are
    sampled: a draw next to a boundary between two tokens falls on the other side."""
    if case["dtype"] == "fp32":
        return {"rel": 1.4e-5, "max": 8e-5}
    return {"rel": 4e-2, "max": 0.2, "differ": 0.2}


# ---- the same results in 64 bits ----------------------------------------------------------------------------------------------------
def _rms(x, w=None, eps=EPS):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _silu(z):
    return z * torch.sigmoid(z)


def _softplus(z):
    return torch.log1p(torch.exp(-z.abs())) + z.clamp(min=0.0)


def _product(x, w):
    return x @ w.double().t()


def _attend(q, k, v, scale, first, window=None, sink=None, cap=None, slope=None):
    """q [n, H, a] of positions first.., k [t, G, a], v [t, G, b] of positions 0..: causal, pieces of queries, head by head."""
    n, H, _ = q.shape
    per = H // k.shape[1]
    out = torch.empty(n, H, v.shape[2], dtype=q.dtype, device=q.device)
    for lo in range(0, n, 4096):
        hi = min(n, lo + 4096)
        t = first + hi
        back = (first + torch.arange(lo, hi, device=q.device))[:, None] - torch.arange(t, device=q.device)[None, :]
        hidden = back < 0 if window is None else (back < 0) | (back >= window)
        for h in range(H):
            s = (q[lo:hi, h] @ k[:t, h // per].t()) * scale
            if cap:
                s = cap * torch.tanh(s / cap)
            if slope is not None:
                s -= slope[h] * back
            s.masked_fill_(hidden, float("-inf"))
            if sink is not None:
                s = torch.cat([s, sink[h].expand(hi - lo, 1)], 1)
            p = torch.softmax(s, -1)
            out[lo:hi, h] = p[:, :t] @ v[:t, h // per]
    return out


def _rotate_halves(x, pos, theta):
    half = x.shape[-1] // 2
    a = pos.double()[:, None] * theta ** (-torch.arange(half, device=x.device, dtype=torch.float64) / half)
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * c - v * s, v * c + u * s], -1)


def _exact_step(case, seed):
    c, W = MINICPM[case["model"]], _minicpm_weights(case["model"], seed, _dtype(case))
    d, L, eps = c["hidden_size"], c["num_hidden_layers"], c["rms_norm_eps"]
    nh, nkv = c["num_attention_heads"], c["num_key_value_heads"]
    dh = d // nh
    held, portions, past = _held(case), _portions(case), case["portion_past"]
    doc, fresh, parts, _ = _tokens(case, seed)
    if not held and not past:
        doc = []
    requests = [(n, [t]) for n, t in zip(held, fresh)] + [(past, toks) for toks in parts]       # (cached prefix, new tokens)
    dev = "cuda"
    toks = torch.tensor(doc + [t for _, new in requests for t in new], device=dev)
    pos = torch.cat([torch.arange(len(doc))] + [n + torch.arange(len(new)) for n, new in requests]).to(dev)
    D = len(doc)
    bounds, at = [], D
    for n, new in requests:
        bounds.append((n, at, at + len(new)))
        at += len(new)
    x = W["model.embed_tokens.weight"][toks].double() * SCALE_EMB
    res = SCALE_DEPTH / math.sqrt(L)
    for i in range(L):
        p = "model.layers.%d." % i
        h = _rms(x, W[p + "input_layernorm.weight"].double(), eps)
        q = _rotate_halves(_product(h, W[p + "self_attn.q_proj.weight"]).view(-1, nh, dh), pos, ROPE_THETA)
        k = _rotate_halves(_product(h, W[p + "self_attn.k_proj.weight"]).view(-1, nkv, dh), pos, ROPE_THETA)
        v = _product(h, W[p + "self_attn.v_proj.weight"]).view(-1, nkv, dh)
        a = torch.empty_like(q)
        if D:
            a[:D] = _attend(q[:D], k[:D], v[:D], dh ** -0.5, 0)
        for n, lo, hi in bounds:
            if hi - lo == 1:         # a single token: all heads at once
                kk, vv = torch.cat([k[:n], k[lo:hi]]), torch.cat([v[:n], v[lo:hi]])
                s = torch.matmul(q[lo].view(nkv, nh // nkv, dh), kk.permute(1, 2, 0).contiguous()) * dh ** -0.5
                a[lo] = torch.matmul(torch.softmax(s, -1), vv.permute(1, 0, 2).contiguous()).reshape(nh, dh)
            else:
                a[lo:hi] = _attend(q[lo:hi], torch.cat([k[:n], k[lo:hi]]), torch.cat([v[:n], v[lo:hi]]), dh ** -0.5, n)
        x = x + res * _product(a.reshape(-1, nh * dh), W[p + "self_attn.o_proj.weight"])
        h = _rms(x, W[p + "post_attention_layernorm.weight"].double(), eps)
        for lo in range(0, h.shape[0], 4096):
            g = h[lo:lo + 4096]
            x[lo:lo + 4096] += res * _product(_silu(_product(g, W[p + "mlp.gate_proj.weight"])) * _product(g, W[p + "mlp.up_proj.weight"]),
                                              W[p + "mlp.down_proj.weight"])
    last = torch.tensor([hi - 1 for _, _, hi in bounds], device=dev)
    h = _rms(x[last], W["model.norm.weight"].double(), eps) * float(d // DIM_MODEL_BASE)
    logits = _product(h, W["lm_head.weight"])
    return [logits, None] if len(requests) >= 32 else [logits]


def _frequencies(rot):
    dims, base, scaling = rot["dims"], rot["base"], rot.get("scaling")
    f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    if not scaling:
        return f, 1.0
    index = lambda turns: dims * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
    lo, hi = max(math.floor(index(scaling["fast"])), 0), min(math.ceil(index(scaling["slow"])), dims - 1)
    ramp = [min(max((i - lo) / max(hi - lo, 0.001), 0.0), 1.0) for i in range(dims // 2)]
    return [v / scaling["factor"] * r + v * (1.0 - r) for v, r in zip(f, ramp)], 0.1 * math.log(scaling["factor"]) + 1.0


def _rotate_pairs(x, rot):
    f, mult = _frequencies(rot)
    a = torch.arange(x.shape[0], device=x.device, dtype=torch.float64)[:, None] * torch.tensor(f, device=x.device, dtype=torch.float64)
    shape = [x.shape[0]] + [1] * (x.dim() - 2) + [len(f)]
    c, s = (torch.cos(a) * mult).view(shape), (torch.sin(a) * mult).view(shape)
    out, n = x.clone(), 2 * len(f)
    u, v = x[..., 0:n:2], x[..., 1:n:2]
    out[..., 0:n:2], out[..., 1:n:2] = u * c - v * s, v * c + u * s
    return out


def _conv(x, w, b=None):
    taps = w.shape[1]
    padded = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
    out = sum(w[:, j].double() * padded[j:j + x.shape[0]] for j in range(taps))
    return out if b is None else out + b.double()


def _latent(h, W, p, m, rows, gated):
    T, H, n, E = h.shape[0], m["heads"], m["dim"], m["rot_dim"]
    latent, k_rot = rows
    q = _product(_rms(_product(h, W[p + "dq"]), W[p + "dq.norm"].double()), W[p + "uq"]).view(T, H, n + E)
    q = torch.cat([q[..., :n], _rotate_pairs(q[..., n:], m["rot"])], -1)
    k = torch.cat([_product(latent, W[p + "uk"]).view(T, H, n), k_rot[:, None].expand(T, H, E)], -1)
    v = _product(latent, W[p + "uv"]).view(T, H, m["vdim"])
    o = _attend(q, k, v, m["scale"], 0, (m.get("mask") or {}).get("size"), None if gated else W[p + "sink"].double()).reshape(T, -1)
    if gated:
        o = o * torch.sigmoid(_product(h, W[p + "g"]))
    return _product(o, W[p + "o"])


def _rglru(h, W, p, m):
    T, n, b = h.shape[0], m["width"], m["blocks"]
    y = _product(h, W[p + "y"]) + W[p + "y.b"].double()
    y = 0.5 * y * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (y + 0.044715 * y ** 3)))
    u = _conv(_product(h, W[p + "x"]) + W[p + "x.b"].double(), W[p + "conv"], W[p + "conv.b"])
    ub = u.view(T, b, n // b).transpose(0, 1).contiguous()
    gate = lambda k: torch.sigmoid(torch.matmul(ub, W[p + k].double().transpose(1, 2).contiguous()).transpose(0, 1)
                                   + W[p + k + ".b"].double()).reshape(T, n)
    a = torch.exp(-8.0 * gate("ra") * _softplus(W[p + "lam"].double()))
    add = torch.sqrt(1.0 - a * a) * gate("ri") * u
    S, out = torch.zeros_like(u[0]), torch.empty_like(u)
    for t in range(T):
        S = a[t] * S + add[t]
        out[t] = S
    return _product(out * y, W[p + "o"])


def _mamba2(h, W, p, m):
    T, H, dv, N, G = h.shape[0], m["heads"], m["vdim"], m["state"], m["groups"]
    inner = H * dv
    proj = _product(h, W[p + "in"])
    xbc = _silu(_conv(proj[:, inner:2 * inner + 2 * G * N], W[p + "conv"], W[p + "conv.b"]))
    dt = _softplus(proj[:, 2 * inner + 2 * G * N:] + W[p + "dt_bias"].double())
    x = xbc[:, :inner].reshape(T, H, dv)
    B = xbc[:, inner:inner + G * N].reshape(T, G, N).repeat_interleave(H // G, 1)
    C = xbc[:, inner + G * N:].reshape(T, G, N).repeat_interleave(H // G, 1)
    decay = torch.exp(-torch.exp(W[p + "A_log"].double()) * dt)
    S, y = h.new_zeros(H, N, dv), torch.empty_like(x)
    dx = dt[..., None] * x
    for t in range(T):
        S = decay[t][:, None, None] * S + B[t][:, :, None] * dx[t][:, None, :]
        y[t] = (S * C[t][:, :, None]).sum(1)
    y = (y + W[p + "D"].double()[:, None] * x).reshape(T, inner) * _silu(proj[:, :inner])
    y = _rms(y.view(T, m["norm_groups"], -1)).reshape(T, inner) * W[p + "norm"].double()
    return _product(y, W[p + "o"])


def _tied(h, W, p, m):
    T, H, G, n = h.shape[0], m["heads"], m["kv_heads"], m["dim"]
    raw = _product(h, W[p + "k"])
    q = _rms(_product(h, W[p + "q"]), W[p + "q.norm"].double()).view(T, H, n)
    k = _rms(raw, W[p + "k.norm"].double()).view(T, G, n)
    o = _attend(q, k, raw.view(T, G, n), m["scale"], 0, m["mask"]["size"], None, m["softcap"], [2.0 ** (-8.0 * (i + 1) / H) for i in range(H)])
    return _product(o.reshape(T, -1) * torch.sigmoid(_product(h, W[p + "g"])), W[p + "o"])


def _delta(h, W, p, m):
    T, H, G, dk, dv = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (_silu(_conv(_product(h, W[p + n]), W[p + n + ".conv"])) for n in ("q", "k", "v"))
    unit = lambda z: z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6)
    q = unit(q.view(T, G, dk)).repeat_interleave(H // G, 1) * dk ** -0.5
    k = unit(k.view(T, G, dk)).repeat_interleave(H // G, 1)
    v = v.view(T, H, dv)
    beta = torch.sigmoid(_product(h, W[p + "b"]))
    decay = torch.exp(-torch.exp(W[p + "A_log"].double()) * _softplus(_product(h, W[p + "a"]) + W[p + "dt_bias"].double()))
    S, o = h.new_zeros(H, dk, dv), torch.empty_like(v)
    for t in range(T):
        S = decay[t][:, None, None] * S
        u = beta[t][:, None] * (v[t] - (S * k[t][:, :, None]).sum(1))
        S = S + k[t][:, :, None] * u[:, None, :]
        o[t] = (S * q[t][:, :, None]).sum(1)
    o = (_rms(o) * W[p + "norm"].double()).reshape(T, -1) * _silu(_product(h, W[p + "g"]))
    return _product(o, W[p + "o"])


def _design_forward(model, cfg, W, tokens, n_last):
    """Logits of the last n_last places of one whole sequence."""
    t = torch.tensor(tokens, device="cuda")
    x = W["embed"][t].double()
    if model == "mezinex":
        big = cfg["embedding"]["bigram"]
        rows = [big["buckets"]] + [(a * big["mul_prev"] + b * big["mul_cur"]) % big["buckets"] for a, b in zip(tokens, tokens[1:])]
        x = x + W["bigram"][torch.tensor(rows, device="cuda")].double()
        xs = torch.stack([x, x])
    mlp = lambda h, p: _product(_silu(_product(h, W[p + "mlp.gate"])) * _product(h, W[p + "mlp.up"]), W[p + "mlp.down"])
    kept = {}
    for i, l in enumerate(cfg["layers"]):
        p, m = "l%d." % i, l["mixer"]
        rot_rows = lambda h: (lambda r: (_rms(r[:, :m["kv_rank"]], W[p + "mix.dkv.norm"].double()),
                                         _rotate_pairs(r[:, m["kv_rank"]:], m["rot"])))(_product(h, W[p + "mix.dkv"]))
        if model == "mezinex":
            for q in ("1", "2"):
                mix, win, wout = W[p + "hc" + q + ".mix"].double(), W[p + "hc" + q + ".in"].double(), W[p + "hc" + q + ".out"].double()
                h = _rms((win[:, None, None] * xs).sum(0), W[p + "norm" + q].double())
                if q == "2":
                    y = mlp(h, p)
                elif l["type"] == "latent_attention":
                    y = _latent(h, W, p + "mix.", m, rot_rows(h), True)
                else:
                    y = (_rglru if l["type"] == "rglru" else _mamba2)(h, W, p + "mix.", m)
                xs = torch.stack([mix[0, s] * xs[0] + mix[1, s] * xs[1] + wout[s] * y for s in (0, 1)])
            continue
        h = _rms(x, W[p + "norm1"].double())
        if l["type"] == "latent_attention":
            if m.get("kv_from") is None:
                kept[i] = rot_rows(h)
            y = _latent(h, W, p + "mix.", m, kept[i if m.get("kv_from") is None else m["kv_from"]], False)
        else:
            y = m["left_scale"] * _tied(h, W, p + "mix.left.", m["left"]) + m["right_scale"] * _delta(h, W, p + "mix.right.", m["right"])
        x = x + y + mlp(h, p)
    if model == "mezinex":
        x = xs.sum(0)
    return _product(_rms(x[-n_last:], W["final.norm"].double()), W["head"])




def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "step":
            return _exact_step(case, seed)
        _, _, parts, later = _tokens(case, seed)
        cfg, W = _design_config(case["model"], case["size"]), _design_weights(case["model"], case["size"], seed)
        rows = [_design_forward(case["model"], cfg, W, toks + [l[i] for l in later], 1 + len(later)) for i, toks in enumerate(parts)]
        return [torch.stack([r[s] for r in rows]) for s in range(1 + len(later))]
