"""The work that a user of this engine has it do, as cases that can be timed and compared.

A case is one pass through ``LLM`` and its ``Engine.step``: a model with random weights (drawn on the
GPU from the seed, as the ``random_weights_seed`` launch option does), requests whose earlier tokens are
already in the cache, and the step or steps that a serving loop would run next.  ``kind`` says which:

``decode``    ``rows`` requests with ``context`` cached tokens each bring one token a step, ``steps`` times
              (tokens are given, so that the logits of every step can be compared); the requests are then
              set back to where they were
``prefill``   ``prompts`` prompts of ``tokens`` tokens each start in one step, or continue behind
              ``behind`` cached tokens; the logits of each prompt's last token
``mixed``     one step with ``rows`` decoding requests and a prompt's portion of ``tokens`` tokens beside them
``whole``     ``prompts`` short requests from their first token on: one step with the prompts, then ``steps``
              tokens each, then released
``generate``  ``LLM.generate``: scheduler, sampler and steps, until every request has ``steps`` new tokens

``ragged`` spreads contexts and prompt lengths between a sixteenth of the stated number and the number
itself, instead of all being equal.  The model sizes are those of the repository's benchmark; the models of
3B and 8B layer sizes have half and three eighths of the layers, so that several fit beside each other.
"""
import hashlib
import json
import math
import os
import random
import tempfile

import torch

VOCAB = 128256
EPS = 1e-5
PAGE = 16
STD = 0.02
ROPE_THETA = 500000.0
SCALING = dict(rope_type="llama3", low_freq_factor=1.0, high_freq_factor=4.0, original_max_position_embeddings=8192)
SIZES = {
    "1b": dict(width=2048, ff=8192, layers=16, heads=32, kv_heads=8, dim=64, tied=True, factor=32.0),
    "3b": dict(width=3072, ff=8192, layers=14, heads=24, kv_heads=8, dim=128, tied=True, factor=32.0),
    "8b": dict(width=4096, ff=14336, layers=12, heads=32, kv_heads=8, dim=128, tied=False, factor=8.0),
}
TEDELIX_TURNS = ("general_delta", "attention", "lightning")
TEDELIX_RANK = 16          # the rank of the decay's input where no checkpoint says another
TEDELIX_WINDOW = 1024


# --------------------------------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------------------------------
def _case(name=None, design="llama", sizes="1b", dtype="bfloat16", kind="decode", rows=0, context=0, prompts=0,
          tokens=0, behind=0, steps=1, ragged=False):
    c = dict(design=design, sizes=sizes, dtype=dtype, kind=kind, rows=rows, context=context, prompts=prompts,
             tokens=tokens, behind=behind, steps=steps, ragged=ragged)
    return dict(c, name=name) if name is not None else c


def listed():
    return [
        # one user, one token after another, soon after a short prompt: the launches count as much as the weights
        _case("decode 1 row 1b", kind="decode", rows=1, context=90, steps=4),
        # the repository's headline: eight requests behind prompts of 2,048 tokens
        _case("decode 8 rows 8b", sizes="8b", kind="decode", rows=8, context=2048, steps=4),
        # a busy server: many requests of very different lengths, their number no multiple of anything
        _case("decode 43 ragged rows 3b", sizes="3b", kind="decode", rows=43, context=3000, steps=4, ragged=True),
        # the repository's prompt benchmark: one prompt of 2,048 tokens in one step
        _case("prefill 2048 8b", sizes="8b", kind="prefill", prompts=1, tokens=2048),
        # a chat turn of a few words
        _case("prefill 37 1b", kind="prefill", prompts=1, tokens=37),
        # several waiting prompts of different lengths in one step
        _case("prefill 5 ragged 3b", sizes="3b", kind="prefill", prompts=5, tokens=1700, ragged=True),
        # the next portion of a long document
        _case("prefill 2048 behind 14336 1b", kind="prefill", prompts=1, tokens=2048, behind=14336),
        # continuous batching: a portion of an arriving prompt beside the requests that decode
        _case("mixed 248 + 8 rows 8b", sizes="8b", kind="mixed", rows=8, context=700, tokens=248, behind=256),
        # the true 32-bit path through the Python entry point, its tokens sampled (temperature, top-k, top-p)
        _case("generate float32 1b", dtype="float32", kind="generate", prompts=6, tokens=100, steps=12, ragged=True),
        # the true 32-bit path on a prompt
        _case("prefill 600 float32 1b", dtype="float32", kind="prefill", prompts=1, tokens=600),
        # the hybrid design (windowed attention, lightning attention, delta rule): a prompt, and short requests served whole
        _case("prefill 2048 tedelix 1b", design="tedelix", kind="prefill", prompts=1, tokens=2048),
        _case("whole 8 x 30 + 12 tedelix 1b", design="tedelix", kind="whole", prompts=8, tokens=30, steps=12),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def _cost(case):
    w = work(case)
    rate = 20e12 if case["dtype"] == "float32" else 6e14
    return max(w["bytes"] / 4e12, w["flops"] / rate)


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "mixed", "mixed", "whole", "generate"])
        sizes = rng.choice(["1b", "3b", "8b"])
        if kind == "decode":
            c = _case(sizes=sizes, kind=kind, rows=_log_int(rng, 1, 64), context=_log_int(rng, 16, 4000), steps=4, ragged=rng.random() < 0.5)
        elif kind == "prefill":
            form = rng.random()
            if form < 0.25:
                c = _case(dtype="float32", kind=kind, prompts=1, tokens=_log_int(rng, 3, 600))
            elif form < 0.45:
                c = _case(design="tedelix", kind=kind, prompts=1, tokens=_log_int(rng, 10, 2048))
            elif form < 0.6:
                c = _case(sizes=sizes, kind=kind, prompts=1, tokens=_log_int(rng, 20, 2048), behind=rng.randint(100, 14336))
            else:
                prompts = _log_int(rng, 1, 8)
                c = _case(sizes=sizes, kind=kind, prompts=prompts, tokens=_log_int(rng, 5, 4096 // prompts), ragged=prompts > 1)
        elif kind == "mixed":
            c = _case(sizes=sizes, kind=kind, rows=_log_int(rng, 1, 48), context=_log_int(rng, 16, 3000), tokens=_log_int(rng, 8, 768),
                      behind=rng.choice([0, rng.randint(1, 2048)]), ragged=rng.random() < 0.5)
        elif kind == "whole":
            c = _case(design="tedelix", kind=kind, prompts=_log_int(rng, 1, 24), tokens=_log_int(rng, 4, 80), steps=rng.randint(4, 16))
        else:
            c = _case(dtype="float32", kind=kind, prompts=_log_int(rng, 1, 8), tokens=_log_int(rng, 5, 100), steps=rng.randint(4, 12), ragged=True)
        if _cost(c) <= most:
            return c


def _spread(case, count, most, salt):
    """``count`` lengths of at most ``most``: all ``most``, or spread over a factor of sixteen (the longest is ``most``)."""
    if not case["ragged"] or count < 2:
        return [most] * count
    rng = random.Random(f"{salt} {count} {most}")
    out = [max(1, int(most * 16.0 ** -rng.random())) for _ in range(count)]
    out[rng.randrange(count)] = most
    return out


def _lengths(case):
    """(contexts of the decoding requests, [(cached, new)] of the prompts)"""
    contexts = _spread(case, case["rows"], case["context"], "context")
    if case["kind"] == "mixed":
        return contexts, [(case["behind"], case["tokens"])]
    return contexts, [(case["behind"], n) for n in _spread(case, case["prompts"], case["tokens"], "prompt")]


# --------------------------------------------------------------------------------------------------
# what a user's program has before the call
# --------------------------------------------------------------------------------------------------
def _config(case):
    s = SIZES[case["sizes"]]
    if case["design"] == "llama":
        return dict(architectures=["LlamaForCausalLM"], hidden_size=s["width"], intermediate_size=s["ff"], num_hidden_layers=s["layers"],
                    num_attention_heads=s["heads"], num_key_value_heads=s["kv_heads"], head_dim=s["dim"], vocab_size=VOCAB,
                    tie_word_embeddings=s["tied"], rms_norm_eps=EPS, rope_theta=ROPE_THETA, rope_scaling=dict(SCALING, factor=s["factor"]),
                    max_position_embeddings=131072)
    layers = []
    for i in range(s["layers"]):
        kind = TEDELIX_TURNS[i % len(TEDELIX_TURNS)]
        if kind == "attention":
            mixer = dict(heads=s["heads"], kv_heads=s["kv_heads"], dim=s["dim"], vdim=s["dim"], mask=dict(size=TEDELIX_WINDOW),
                         scale=s["dim"] ** -0.5, rot=dict(base=10000.0, dims=s["dim"]))
        elif kind == "lightning":
            mixer = dict(heads=s["heads"], dim=s["dim"], vdim=s["dim"],
                         decay=[1.0 - 2.0 ** (-5 - 3 * h / (s["heads"] - 1)) for h in range(s["heads"])])
        else:
            mixer = dict(heads=s["heads"], dim=s["dim"])
        layers.append(dict(type=kind, mixer=mixer, mlp=dict(kind="dense", ff=s["ff"])))
    return dict(architecture="Tedelix", vocab=VOCAB, width=s["width"], norm=dict(eps=EPS), logit_scale=1.0, logit_softcap=30.0, layers=layers)


def _tokens(case, seed):
    """({request: its cached tokens}, {request: the tokens it brings}) of the decoding requests and of the prompts"""
    g = torch.Generator().manual_seed(int(seed) * 7919 + 17)
    ids = lambda n: torch.randint(0, VOCAB, (n,), generator=g).tolist()  # noqa: E731
    contexts, prompts = _lengths(case)
    cached, new = {}, {}
    for i, n in enumerate(contexts):
        cached[f"d{i}"], new[f"d{i}"] = ids(n), ids(case["steps"])
    for i, (before, n) in enumerate(prompts):
        cached[f"p{i}"], new[f"p{i}"] = ids(before), ids(n + (case["steps"] if case["kind"] == "whole" else 0))
    return cached, new


def prepare(case, seed):
    from rustinfer_amd import LLM, SamplingParams
    from rustinfer_amd.engine import StepEntry
    cached, new = _tokens(case, seed)
    requests = len(cached)
    spare = case["steps"] + 1
    longest = max(len(cached[r]) + len(new[r]) for r in cached) + spare
    pages = sum(-(-(len(cached[r]) + len(new[r]) + spare) // PAGE) for r in cached) + 8
    with tempfile.TemporaryDirectory() as folder:
        with open(os.path.join(folder, "config.json"), "w") as f:
            json.dump(_config(case), f)
        llm = LLM(model=folder, random_weights_seed=int(seed), dtype=case["dtype"], num_blocks=pages, max_batch_seqs=max(requests, 1),
                  max_model_len=max(4096, longest), max_batch_tokens=8192)
    engine, state = llm.engine, dict(llm=llm, cached=cached, new=new, kind=case["kind"], steps=case["steps"])
    if case["kind"] == "generate":
        state["params"] = [SamplingParams(temperature=0.8, top_k=50, top_p=0.95, seed=int(seed) + i, max_tokens=case["steps"], ignore_eos=True)
                           for i in range(len(new))]
        return state
    waiting = {r: list(t) for r, t in cached.items() if t}
    while waiting:                                   # what the requests hold already, in steps as large as the engine takes
        entries, room = [], 8192
        for r in list(waiting):
            part = waiting[r][:room]
            if not part:
                break
            waiting[r] = waiting[r][len(part):]
            room -= len(part)
            if not waiting[r]:
                del waiting[r]
            entries.append(StepEntry(r, part, []))
        engine.step(entries)
    decoding = [r for r in new if r[0] == "d" or case["kind"] == "whole"]
    if case["kind"] in ("decode", "whole"):
        llm.capture_graphs(len(decoding), max(len(cached[r]) + len(new[r]) for r in decoding))
    state["out"] = torch.empty(case["steps"] + (case["kind"] == "whole"), len(decoding), VOCAB, dtype=torch.float32, device="cuda") \
        if case["kind"] in ("decode", "whole") else None
    torch.cuda.synchronize()
    return state


def run(state):
    """One pass; see the head of this file."""
    from rustinfer_amd.engine import StepEntry
    llm, kind, new, cached = state["llm"], state["kind"], state["new"], state["cached"]
    engine = llm.engine
    if kind == "generate":
        return torch.tensor([r.token_ids for r in llm.generate(list(new.values()), state["params"])], dtype=torch.int64)
    if kind == "decode":
        for i in range(state["steps"]):
            state["out"][i].copy_(engine.step([StepEntry(r, [t[i]], [0]) for r, t in new.items()]))
        out = state["out"]
    elif kind == "whole":
        n = {r: len(t) - state["steps"] for r, t in new.items()}
        state["out"][0].copy_(engine.step([StepEntry(r, t[:n[r]], [n[r] - 1]) for r, t in new.items()]))
        for i in range(state["steps"]):
            state["out"][i + 1].copy_(engine.step([StepEntry(r, [t[n[r] + i]], [0]) for r, t in new.items()]))
        out = state["out"]
    else:                                            # each entry's last token is what its request samples from next
        out = engine.step([StepEntry(r, t, [len(t) - 1]) for r, t in new.items()])
    for r in new:
        if cached[r]:
            engine.cache.truncate(r, len(cached[r]))
        else:
            engine.release(r)
    return out


# --------------------------------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------------------------------
def _layer_numbers(case, i):
    """(weights, key/value elements a token, state elements a request, attention flops a key, recurrence flops a token) of layer i"""
    s = SIZES[case["sizes"]]
    d, ff, q, kv = s["width"], s["ff"], s["heads"] * s["dim"], s["kv_heads"] * s["dim"]
    if case["design"] == "llama":
        return d * (q + 2 * kv) + q * d + 3 * d * ff, 2 * kv, 0, 4.0 * q, 0.0
    kind = TEDELIX_TURNS[i % 3]
    if kind == "attention":
        return d * (q + 2 * kv) + q * d + 2 * d * ff, 2 * kv, 0, 4.0 * q, 0.0
    state = s["heads"] * s["dim"] * s["dim"]
    if kind == "lightning":
        return 5 * d * q + 2 * d * ff, 0, state, 0.0, 4.0 * state
    return 6 * d * q + 2 * TEDELIX_RANK * d + 2 * d * ff, 0, state, 0.0, 10.0 * state


def work(case):
    s, el = SIZES[case["sizes"]], 4 if case["dtype"] == "float32" else 2
    contexts, prompts = _lengths(case)
    # the steps of a pass: [(tokens cached before, new tokens, logits wanted)] a step
    if case["kind"] == "decode":
        steps = [[(n + i, 1) for n in contexts] for i in range(case["steps"])]
    elif case["kind"] == "mixed":
        steps = [[(n, 1) for n in contexts] + prompts]
    elif case["kind"] == "prefill":
        steps = [prompts]
    else:
        more = case["steps"] - (case["kind"] == "generate")         # a generated token's own step is the next one's
        steps = [prompts] + [[(n + i, 1) for _, n in prompts] for i in range(more)]
    window = TEDELIX_WINDOW if case["design"] == "tedelix" else 1 << 40
    bytes_ = flops = 0.0
    for step in steps:
        T, rows = sum(n for _, n in step), len(step)
        head = VOCAB * s["width"]
        bytes_ += head * el + T * s["width"] * el + rows * VOCAB * 4
        flops += 2.0 * rows * head
        for i in range(s["layers"]):
            weights, kv, state, per_key, per_token = _layer_numbers(case, i)
            keys_read = sum(min(before, window) for before, _ in step)
            keys_seen = sum(sum(min(j + 1, window) for j in range(before, before + n)) for before, n in step)
            bytes_ += el * (weights + 2 * s["width"] + kv * (keys_read + T)) + 2 * 4 * state * rows
            flops += 2.0 * T * weights + per_key * keys_seen + per_token * T
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    if case["kind"] == "generate":                    # tokens; a draw falls within 1e-6 of a boundary hardly ever
        return {"rel": 0.0, "differ": 0.01}
    if case["dtype"] == "float32":                    # 1.0e-6 from ``exact`` over 16 layers
        return {"rel": 1e-5}
    # bfloat16 rows between the products: 0.010 to 0.036 from ``exact`` over 12 to 16 layers; implementations that
    # round in the same places are closer to each other than to it
    return {"rel": 0.03, "max": 0.3}


# --------------------------------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# --------------------------------------------------------------------------------------------------
class _Weights:
    """The tensors that the random-weights launch option draws: a generator a tensor, seeded by the seed and the
    tensor's name; deviation 0.02 (1 + that for norms) unless the tensor has its own."""

    def __init__(self, case, seed):
        self.seed, self.dtype = int(seed), getattr(torch, case["dtype"])

    def __call__(self, name, *shape, mean=0.0, std=STD):
        h = hashlib.blake2b(f"{self.seed}:{name}".encode(), digest_size=8).digest()
        g = torch.Generator(device="cuda").manual_seed(int.from_bytes(h, "little") & ((1 << 63) - 1))
        t = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std + mean
        return t.to(self.dtype).double()


def _norm(x, w=None):
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return y if w is None else y * w


def _turn(x, pos, freqs, sign=1.0):
    """x [T, heads, size] with feature i and i + size / 2 turned by ``sign * pos * freqs[i]``"""
    ang = sign * pos[:, None].double() * freqs
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _llama_freqs(s):
    out = []
    low, high = SCALING["original_max_position_embeddings"] / SCALING["low_freq_factor"], SCALING["original_max_position_embeddings"] / SCALING["high_freq_factor"]
    for i in range(s["dim"] // 2):
        f = ROPE_THETA ** (-2.0 * i / s["dim"])
        length = 2.0 * math.pi / f
        if length > low:
            f /= s["factor"]
        elif length >= high:
            t = (SCALING["original_max_position_embeddings"] / length - SCALING["low_freq_factor"]) / (SCALING["high_freq_factor"] - SCALING["low_freq_factor"])
            f = (1.0 - t) * f / s["factor"] + t * f
        out.append(f)
    return torch.tensor(out, dtype=torch.float64, device="cuda")


def _attend(q, k, v, scale, window=0, first=0):
    """Causal softmax attention of queries at positions ``first``.. ; q [T, H, d], k and v [L, G, d]"""
    T, H, _ = q.shape
    L, G, dv = v.shape
    kt, vt = k.permute(1, 2, 0).contiguous(), v.permute(1, 0, 2).contiguous()
    out = torch.empty(T, H, dv, dtype=q.dtype, device=q.device)
    for lo in range(0, T, 512):
        hi = min(T, lo + 512)
        end = first + hi
        beg = max(0, first + lo - window + 1) if window else 0
        i = torch.arange(first + lo, end, device=q.device)[:, None]
        j = torch.arange(beg, end, device=q.device)[None]
        hidden = j > i
        if window:
            hidden |= j <= i - window
        for g in range(G):
            part = q[lo:hi, g * (H // G):(g + 1) * (H // G)].permute(1, 0, 2)
            s = torch.matmul(part, kt[g, :, beg:end]) * scale
            p = torch.softmax(s.masked_fill_(hidden, -math.inf), -1)
            out[lo:hi, g * (H // G):(g + 1) * (H // G)] = torch.matmul(p, vt[g, beg:end]).permute(1, 0, 2)
    return out


def _walk_lightning(q, k, v, decay):
    S = torch.zeros(q.shape[1], q.shape[2], v.shape[2], dtype=q.dtype, device=q.device)
    out = torch.empty_like(v)
    for t in range(q.shape[0]):
        S = decay[:, None, None] * S + k[t][:, :, None] * v[t][:, None]
        out[t] = (S * q[t][:, :, None]).sum(1)
    return out


def _walk_delta(r, k, v, w, a):
    S = torch.zeros(r.shape[1], r.shape[2], v.shape[2], dtype=r.dtype, device=r.device)
    out = torch.empty_like(v)
    u = k * torch.rsqrt(k.square().sum(-1, keepdim=True) + 1e-6)
    for t in range(r.shape[0]):
        S = w[t][:, :, None] * S - (a[t] * u[t])[:, :, None] * (S * u[t][:, :, None]).sum(1, keepdim=True) + k[t][:, :, None] * v[t][:, None]
        out[t] = (S * r[t][:, :, None]).sum(1)
    return out


def _llama_layer(W, s, i, xs, freqs):
    p, d, q, kv = f"model.layers.{i}.", s["width"], s["heads"] * s["dim"], s["kv_heads"] * s["dim"]
    n1, n2 = W(p + "input_layernorm.weight", d, mean=1.0), W(p + "post_attention_layernorm.weight", d, mean=1.0)
    wq, wk, wv, wo = W(p + "self_attn.q_proj.weight", q, d), W(p + "self_attn.k_proj.weight", kv, d), W(p + "self_attn.v_proj.weight", kv, d), W(p + "self_attn.o_proj.weight", d, q)
    gate, up, down = W(p + "mlp.gate_proj.weight", s["ff"], d), W(p + "mlp.up_proj.weight", s["ff"], d), W(p + "mlp.down_proj.weight", d, s["ff"])
    out = []
    for x in xs:
        T = x.shape[0]
        pos = torch.arange(T, device=x.device)
        n = _norm(x, n1)
        heads = lambda w, h: (n @ w.T).view(T, h, s["dim"])  # noqa: E731
        y = _attend(_turn(heads(wq, s["heads"]), pos, freqs), _turn(heads(wk, s["kv_heads"]), pos, freqs), heads(wv, s["kv_heads"]), s["dim"] ** -0.5)
        x = x + y.reshape(T, q) @ wo.T
        parts = [(torch.nn.functional.silu(m @ gate.T) * (m @ up.T)) @ down.T for m in _norm(x, n2).split(4096)]
        out.append(x + torch.cat(parts))
    return out


def _tedelix_layer(W, s, i, xs):
    p, d, H, size = f"l{i}.", s["width"], s["heads"], s["dim"]
    q, kv, kind = H * size, s["kv_heads"] * size, TEDELIX_TURNS[i % 3]
    norm, up, down, wo = W(p + "norm1", d, mean=1.0), W(p + "mlp.up", s["ff"], d), W(p + "mlp.down", d, s["ff"]), W(p + "mix.o", d, q)
    out = []
    for x in xs:
        T = x.shape[0]
        n = _norm(x, norm)
        pos = torch.arange(T, device=x.device)
        proj = lambda name, rows=q: n @ W(p + "mix." + name, rows, d).T  # noqa: E731
        heads = lambda t: t.view(T, -1, size)  # noqa: E731
        if kind == "attention":
            f = 10000.0 ** (-2.0 * torch.arange(size // 2, dtype=torch.float64, device=x.device) / size)
            y = _attend(_turn(heads(proj("q")), pos, f), _turn(heads(proj("k", kv)), pos, f), _turn(heads(proj("v", kv)), pos, f), size ** -0.5, TEDELIX_WINDOW)
            y = _turn(y, pos, f, -1.0).reshape(T, q)
        elif kind == "lightning":
            decay = torch.tensor([1.0 - 2.0 ** (-5 - 3 * h / (H - 1)) for h in range(H)], dtype=torch.float64, device=x.device)
            act = torch.nn.functional.silu
            y = _walk_lightning(heads(act(proj("q"))), heads(act(proj("k"))), heads(act(proj("v"))), decay).reshape(T, q)
            y = _norm(y, W(p + "mix.norm", q, mean=1.0)) * torch.sigmoid(proj("g"))
        else:
            w = torch.tanh(proj("w1", TEDELIX_RANK)) @ W(p + "mix.w2", q, TEDELIX_RANK).T + W(p + "mix.w0", q, std=1.0)
            w = torch.exp(-math.exp(-0.5) * torch.sigmoid(w))
            a = torch.sigmoid(proj("a") + W(p + "mix.a.b", q, std=1.0))
            y = _walk_delta(heads(proj("r")), heads(proj("k")), heads(proj("v")), heads(w), heads(a))
            y = _norm(y).reshape(T, q) * W(p + "mix.norm", q, mean=1.0) * torch.sigmoid(proj("g"))
        out.append(x + y @ wo.T + torch.relu(n @ up.T).square() @ down.T)
    return out


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "generate":
        return None                                   # tokens: whole values
    cached, new = _tokens(case, seed)
    s, W = SIZES[case["sizes"]], _Weights(case, seed)
    total = sum(len(cached[r]) + len(new[r]) for r in new)
    weights = sum(_layer_numbers(case, i)[0] for i in range(s["layers"]))
    if 2.0 * total * weights > 4e14:
        return None                                   # over about 20 seconds in 64 bits
    names = ("model.embed_tokens.weight", "model.norm.weight", "lm_head.weight") if case["design"] == "llama" else ("embed", "final.norm", "")
    table = W(names[0], VOCAB, s["width"])
    xs = [table[torch.tensor(cached[r] + new[r], device="cuda")] for r in new]
    if case["design"] == "llama" and not s["tied"]:
        del table
        table = W(names[2], VOCAB, s["width"])
    freqs = _llama_freqs(s)
    for i in range(s["layers"]):
        xs = _llama_layer(W, s, i, xs, freqs) if case["design"] == "llama" else _tedelix_layer(W, s, i, xs)
    final = W(names[1], s["width"], mean=1.0)

    def logits(x):
        z = _norm(x, final) @ table.T
        return z if case["design"] == "llama" else 30.0 * torch.tanh(z / 30.0)

    if case["kind"] in ("decode", "whole"):
        more = case["steps"] if case["kind"] == "decode" else case["steps"] + 1
        return torch.stack([logits(torch.stack([x[x.shape[0] - more + i] for x in xs])) for i in range(more)])
    return logits(torch.stack([x[-1] for x in xs]))
