"""The work this framework is measured on, through its public entry points.

Training: a step of a Llama decoder and the flash attention that every decoder
trains on.  Serving: short requests through the engine, and the mechanisms of a
serving layer one by one - paged attention, latent attention, experts, matrix
memories - for prompts and for single tokens.  Sizes are those of the
configurations in ``models/`` and of the serving benchmark.

``exact`` computes the same with plain torch in 64 bits.
"""

import math

import torch
import torch.nn.functional as F
from torch.utils.checkpoint import checkpoint

from neuronx_distributed_amd import inference
from neuronx_distributed_amd.inference.engine import TILE_ROWS, RaggedBatch
from neuronx_distributed_amd.kernels.flash_attn import flash_attn_func
from neuronx_distributed_amd.models import build_model, get_config
from neuronx_distributed_amd.ops import serving as sv

BF16 = torch.bfloat16
PAGE = sv.PAGE_SIZE
EPS = 1e-5
HEAD = 128                   # elements of an attention head
NEW = 16                     # tokens a served request asks for
ROPE_BASE = 10000.0
# of a latent attention, of the experts' activation
RANK, SHARED, ROT_BASE = 512, 64, 1e4
ALPHA, LIMIT, SHIFT = 1.702, 7.0, 1.0

TRAIN = dict(path="train", batch=2, seq=4096, layers=2, width=4096, ff=11008,
             heads=32, kv_heads=32, vocab=32000)
ATTENTION = dict(path="attention", batch=1, seq=8192, heads=32, kv_heads=8,
                 window=0)
GENERATE = dict(path="generate", requests=32, prompt=4800, layers=4,
                width=4096, ff=14336, heads=32, kv_heads=8, vocab=32000)
PAGED = dict(path="paged", portions=3, tokens=6000, singles=5, context=4096,
             heads=32, kv_heads=8, window=4096, keep=64)
LATENT = dict(path="latent", portions=2, tokens=4096, singles=0, context=1024,
              heads=32, dim=128, vdim=128, window=4096)
EXPERTS = dict(path="experts", tokens=4096, experts=8, top=2, width=4096,
               ff=14336)
MEMORY = dict(path="memory", gate="time", requests=2, tokens=4096, single=False,
              heads=128, dim=128, vdim=64, groups=8)


def _like(base, name=None, **changes):
    return dict(base, **changes) if name is None else \
        dict(base, name=name, **changes)


def listed():
    return [
        # a pretraining step at the widths of a 7B decoder
        _like(TRAIN, "train"),
        # its attention with grouped heads at a long sequence
        _like(ATTENTION, "attention_8k"),
        # documents of an odd length under a sliding window
        _like(ATTENTION, "attention_window", batch=2, seq=3001, window=1024),
        # one user waits for a short answer: latency
        _like(GENERATE, "generate_1", requests=1, prompt=100),
        # 32 users at once, prompts of all lengths
        _like(GENERATE, "generate_32"),
        # portions of long prompts beside decoding rows, in one step
        _like(PAGED, "paged_prompt"),
        # decoding at full context, batch 32
        _like(PAGED, "paged_decode", portions=0, tokens=0, singles=32,
              window=0, keep=0),
        # the same two for a latent cache
        _like(LATENT, "latent_prompt"),
        _like(LATENT, "latent_decode", portions=0, tokens=0, singles=32,
              context=4096),
        # a prompt through 8 large experts, a decode batch through 64 small
        _like(EXPERTS, "experts_prompt"),
        _like(EXPERTS, "experts_decode", tokens=32, experts=64, top=6,
              width=2048, ff=1408),
        # two prompts through a state-space memory
        _like(MEMORY, "memory_prompt"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["train", "attention", "attention", "generate", "paged",
                       "paged", "latent", "latent", "experts", "experts",
                       "memory", "memory"])
    if path == "train":
        width, ff, heads, kv = rng.choice([(4096, 11008, 32, 32),
                                           (4096, 14336, 32, 8),
                                           (3584, 18944, 28, 4),
                                           (2048, 5632, 16, 16)])
        return _like(TRAIN, batch=rng.randint(1, 2), seq=_log(rng, 200, 4096),
                     layers=rng.randint(1, 2), width=width, ff=ff, heads=heads,
                     kv_heads=kv)
    if path == "attention":
        heads, kv = rng.choice([(32, 8), (32, 32), (28, 4), (40, 40)])
        seq = _log(rng, 130, 8192)
        return _like(ATTENTION, batch=rng.randint(1, 2 if seq > 2000 else 8),
                     seq=seq, heads=heads, kv_heads=kv,
                     window=rng.choice([0, 0, 1024, 4096, seq // 3]))
    if path == "generate":
        n = _log(rng, 1, 64)
        return _like(GENERATE, requests=n,
                     prompt=n * _log(rng, 20, 300) + rng.randint(0, n),
                     layers=rng.randint(2, 4))
    if path in ("paged", "latent"):
        base = PAGED if path == "paged" else LATENT
        kind = rng.choice(["prompt", "decode", "mixed"])
        portions = 0 if kind == "decode" else rng.randint(1, 4)
        singles = 0 if kind == "prompt" else _log(rng, 1, 128)
        c = _like(base, portions=portions, singles=singles,
                  tokens=portions * _log(rng, 40, 2048) + portions // 2,
                  context=_log(rng, 64, 6000),
                  heads=rng.choice([16, 32]),
                  window=rng.choice([0, 1024, 4096]))
        if path == "paged":
            c["keep"] = rng.choice([0, 64]) if c["window"] else 0
        return c
    if path == "experts":
        experts, top, width, ff = rng.choice([(8, 2, 4096, 14336),
                                              (64, 6, 2048, 1408)])
        return _like(EXPERTS, experts=experts, top=top, width=width, ff=ff,
                     tokens=_log(rng, 1, 4096))
    kind = rng.choice(["time", "decay", "exp"])
    sizes = {"time": rng.choice([dict(heads=128, groups=8),
                                 dict(heads=64, groups=4)]),
             "decay": dict(heads=32, vdim=128, groups=32),
             "exp": dict(heads=16, vdim=256, groups=16)}[kind]
    single = rng.random() < 0.5
    n = _log(rng, 1, 128) if single else rng.randint(1, 4)
    return _like(MEMORY, gate=kind, requests=n, single=single,
                 tokens=n if single else n * _log(rng, 50, 1500) + n // 2,
                 **sizes)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------

class _Source:
    """Random tensors from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator("cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0, dtype=BF16, mean=0.0):
        t = torch.empty(shape, dtype=dtype, device="cuda")
        return t.normal_(mean, std, generator=self.g)

    def uniform(self, *shape, lo=0.0, hi=1.0, dtype=torch.float32):
        t = torch.empty(shape, dtype=torch.float32, device="cuda")
        return t.uniform_(lo, hi, generator=self.g).to(dtype)

    def integers(self, hi, *shape):
        return torch.randint(hi, shape, generator=self.g, device="cuda")

    def permutation(self, n):
        return torch.randperm(n, generator=self.g, device="cuda").int()


def _split(total, n):
    """``total`` in ``n`` unequal parts, the first the smallest."""
    cut = [total * i * (i + 1) // (n * (n + 1)) for i in range(n + 1)]
    return [b - a for a, b in zip(cut, cut[1:])]


def _i32(x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


def _llama_weights(case, r):
    """Name -> tensor, as the model names them."""
    W, kv = case["width"], case["kv_heads"] * HEAD
    q = case["heads"] * HEAD

    def matrix(out, inp):
        return r.normal(out, inp, std=0.02)

    def vector():
        return r.normal(W, std=0.1, mean=1.0)

    w = {"model.embed_tokens.weight": r.normal(case["vocab"], W, std=0.02)}
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        w[p + "self_attn.qkv_proj.weight_q"] = matrix(q, W)
        w[p + "self_attn.qkv_proj.weight_k"] = matrix(kv, W)
        w[p + "self_attn.qkv_proj.weight_v"] = matrix(kv, W)
        w[p + "self_attn.o_proj.weight"] = matrix(W, q)
        w[p + "mlp.gate_up_proj.weight"] = matrix(2 * case["ff"], W)
        w[p + "mlp.down_proj.weight"] = matrix(W, case["ff"])
        w[p + "input_layernorm.weight"] = vector()
        w[p + "post_attention_layernorm.weight"] = vector()
    w["model.norm.weight"] = vector()
    w["lm_head.weight"] = matrix(case["vocab"], W)
    return w


def _llama(case, weights, positions):
    inference.single_process_groups()
    cfg = get_config("llama2-7b", hidden_size=case["width"],
                     intermediate_size=case["ff"],
                     num_hidden_layers=case["layers"],
                     num_attention_heads=case["heads"],
                     num_key_value_heads=case["kv_heads"],
                     vocab_size=case["vocab"], rope_theta=ROPE_BASE,
                     rms_norm_eps=EPS, max_position_embeddings=positions)
    model = build_model("LlamaForCausalLM", cfg, BF16, "cuda")
    model.load_state_dict(weights)
    return model


def _tokens(case, r):
    return r.integers(case["vocab"], case["batch"], case["seq"])


def _heads(case, r):
    """Queries, keys, values and the gradient of the output, as a decoder
    makes them: (batch, sequence, heads, 128)."""
    B, S = case["batch"], case["seq"]
    return [r.normal(B, S, n, HEAD) for n in
            (case["heads"], case["kv_heads"], case["kv_heads"],
             case["heads"])]


def _requests(case, r):
    """Prompts, and the tokens that follow them."""
    lens = _split(case["prompt"], case["requests"])
    prompts = [r.integers(case["vocab"], max(2, n)).tolist() for n in lens]
    return prompts, [r.integers(case["vocab"], NEW).tolist() for _ in lens]


def _rows(case):
    """(context, new tokens) of every request of a step: portions of prompts
    first, then single tokens."""
    n, s, c = case["portions"], case["singles"], case["context"]
    out = [(c * i // max(1, n - 1), t) for i, t in
           enumerate(_split(case["tokens"], n) if n else [])]
    return out + [(c - c * 7 * i // (8 * s), 1) for i in range(s)]


def _batch(case, r):
    """The step as the kernels see it, over randomly placed pages."""
    rows, n = _rows(case), case["portions"]
    need = [-(-(c + t) // PAGE) for c, t in rows]
    place = r.permutation(sum(need))
    table = torch.zeros(len(rows), max(need), dtype=torch.int32,
                        device="cuda")
    at = 0
    for i, k in enumerate(need):
        table[i, :k] = place[at:at + k]
        at += k
    pos, seq, tiles, segs = [], [], [], []
    for i, (c, t) in enumerate(rows):
        r0 = len(pos)
        pos += range(c, c + t)
        seq += [i] * t
        segs.append((i, r0, t, c))
        if i < n:
            tiles += [(i, r0 + q, min(TILE_ROWS, t - q), c + q)
                      for q in range(0, t, TILE_ROWS)]
    chunks, first = sv.chunk_table(segs[:n])
    spans = {}
    if case["path"] == "latent" and \
            max((t for _, t in rows[:n]), default=0) >= sv.EXPAND_MIN_TOKENS:
        pages, places = sv.key_spans(segs[:n], table[:n].tolist(),
                                     case["window"])
        spans[case["window"]] = sv.KeySpans(_i32(pages), _i32(places))
    return RaggedBatch(
        tokens=_i32([0] * len(pos)), pos=_i32(pos), seq=_i32(seq),
        block_table=table, tiles=_i32(tiles).reshape(-1, 4),
        portions=_i32(segs[:n]).reshape(-1, 4),
        chunks=_i32(chunks).reshape(-1, 4), chunk_first=_i32(first),
        singles=_i32(segs[n:]).reshape(-1, 4), want=_i32([]),
        portion_tokens=sum(t for _, t in rows[:n]),
        max_keys=max(c + t for c, t in rows), spans=spans), sum(need)


def _paged_inputs(case, r):
    H, G = case["heads"], case["kv_heads"]
    batch, pages = _batch(case, r)
    proj = r.normal(batch.pos.shape[0], (H + 2 * G) * HEAD)
    cache = [r.normal(pages, G, PAGE, HEAD) for _ in "kv"]
    return batch, proj, cache


def _latent_inputs(case, r):
    H, D, E = case["heads"], case["dim"], case["vdim"]
    batch, pages = _batch(case, r)
    T = batch.pos.shape[0]
    return dict(batch=batch, q=r.normal(T, H * (D + SHARED)),
                kv=r.normal(T, RANK + SHARED), gate=r.normal(T, H * E),
                cache=r.normal(pages, PAGE, RANK + SHARED),
                norm=r.normal(RANK, std=0.1, mean=1.0),
                uk=r.normal(H * D, RANK, std=RANK ** -0.5),
                uv=r.normal(H * E, RANK, std=RANK ** -0.5))


def _experts_inputs(case, r):
    T, E, W, ff = (case[k] for k in ("tokens", "experts", "width", "ff"))
    h = r.normal(T, W)
    router = r.normal(E, W, std=W ** -0.5)
    return dict(h=h, z=torch.mm(h.float(), router.float().t()),
                bias=r.normal(E, std=0.1),
                gate_up=r.normal(E, 2 * ff, W, std=W ** -0.5),
                down=r.normal(E, W, ff, std=ff ** -0.5),
                x=r.normal(T, W, dtype=torch.float32),
                weight=r.normal(W, std=0.1, mean=1.0))


def _memory_inputs(case, r):
    H, D, E, G = (case[k] for k in ("heads", "dim", "vdim", "groups"))
    B, T, f32 = case["requests"], case["tokens"], torch.float32
    lens = [1] * B if case["single"] else _split(T, B)
    ctx = PAGE if case["single"] else 0
    segs, at = [], 0
    for b, n in enumerate(lens):
        segs.append((b, at, n, ctx))
        at += n
    proj = r.normal(T, 2 * G * D + 2 * H * E)
    s = dict(segs=segs, proj=proj, S=r.normal(B, H, D, E, dtype=f32), n=None,
             m=None)
    if case["gate"] == "decay":
        s["decay"] = [math.exp(-2.0 ** (-8.0 * (h + 1) / H))
                      for h in range(H)]
    elif case["gate"] == "exp":
        nt = -(-E // 32)
        n = r.normal(B, H, 1, D, dtype=f32)
        m = r.normal(B, H, 1, dtype=f32)
        s.update(n=n.expand(B, H, nt, D).contiguous(),
                 m=m.expand(B, H, nt).contiguous(),
                 raw=r.normal(T, 2 * H, dtype=f32),
                 i_bias=r.normal(H, std=0.1),
                 f_bias=r.normal(H, std=0.1, mean=3.0))
    else:
        # time steps of 0.001 to 0.1, decays of 1 to 16 a unit of time
        dt = r.uniform(H, lo=math.log(1e-3), hi=math.log(0.1)).exp()
        s.update(raw=r.normal(T, H, std=0.5, dtype=f32),
                 bias=torch.expm1(dt).log().to(BF16),
                 A_log=r.uniform(H, lo=1.0, hi=16.0).log().to(BF16),
                 skip=r.normal(H, std=0.1, mean=1.0))
    return s


# ---------------------------------------------------------------------------
# what a program has in hand, and one pass
# ---------------------------------------------------------------------------

def prepare(case, seed):
    r, path = _Source(seed), case["path"]
    if path == "train":
        model = _llama(case, _llama_weights(case, r), max(4096, case["seq"]))
        return dict(case=case, model=model.train(), ids=_tokens(case, r))
    if path == "attention":
        q, k, v, grad = _heads(case, r)
        return dict(case=case, grad=grad.transpose(1, 2),
                    qkv=[t.requires_grad_() for t in (q, k, v)])
    if path == "generate":
        weights = _llama_weights(case, r)
        prompts, new = _requests(case, r)
        pages = sum(-(-(len(p) + NEW) // PAGE) for p in prompts)
        longest = max(len(p) for p in prompts) + NEW
        engine = inference.InferenceEngine(
            _llama(case, weights, 4096), max_tokens=pages * PAGE,
            max_seqs=len(prompts), max_context=longest)
        state = dict(case=case, engine=engine, prompts=prompts, new=new)
        run(state)               # a server captures its graphs before it serves
        return state
    if path == "paged":
        batch, proj, cache = _paged_inputs(case, r)
        return dict(case=case, batch=batch, proj=proj, cache=cache)
    if path == "latent":
        s = _latent_inputs(case, r)
        H, D = case["heads"], case["dim"]
        w = sv.LatentWeights(
            s["norm"],
            s["uk"].view(H, D, RANK).transpose(1, 2).contiguous(),
            torch.cat([s["uk"], s["uv"]]),
            sv.rotary_frequencies(ROT_BASE, SHARED, "cuda"))
        return dict(s, case=case, weights=w)
    if path == "experts":
        return dict(_experts_inputs(case, r), case=case)
    s = dict(_memory_inputs(case, r), case=case)
    H, D = case["heads"], case["dim"]
    if case["gate"] == "decay":
        s["gating"] = sv.decay_gate(s["decay"], "cuda")
    elif case["gate"] == "exp":
        s["gating"] = sv.ExpGate(s["raw"], s["i_bias"], s["f_bias"], 15.0,
                                 D ** -0.5)
    s["seg"] = _i32(s["segs"])
    s["chunks"] = ()
    if not case["single"]:
        rows, first = sv.chunk_table(s["segs"])
        s["chunks"] = _i32(rows), _i32(first)
    return s


def _memory_parts(case, proj):
    """q, k, v and the skip's gate: slices of one projection."""
    H, D, E, G = (case[k] for k in ("heads", "dim", "vdim", "groups"))
    return proj.split((G * D, G * D, H * E, H * E), dim=1)


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "train":
        model, ids = state["model"], state["ids"]
        for p in model.parameters():
            p.grad = None
        loss = model(ids, labels=ids)
        loss.backward()
        return {"loss": loss.detach(),
                "grad": {n: p.grad for n, p in model.named_parameters()}}
    if path == "attention":
        q, k, v = state["qkv"]
        out = flash_attn_func(q.transpose(1, 2), k.transpose(1, 2),
                              v.transpose(1, 2), causal=True,
                              window=case["window"] or None)
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["grad"])
        return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}
    if path == "generate":
        engine, prompts, new = (state[k] for k in ("engine", "prompts",
                                                   "new"))
        step = inference.StepEntry
        logits = [engine.step([step(i, p, [len(p) - 1])
                               for i, p in enumerate(prompts)])]
        for t in range(NEW - 1):
            logits.append(engine.step([step(i, [n[t]], [0])
                                       for i, n in enumerate(new)]))
        for i in range(len(prompts)):
            engine.finish(i)
        return logits
    if path == "paged":
        H, G = case["heads"] * HEAD, case["kv_heads"] * HEAD
        q, k, v = state["proj"].split((H, G, G), dim=1)
        out = sv.ragged_attention(q, k, v, state["batch"], state["cache"],
                                  case["heads"], HEAD ** -0.5, case["window"],
                                  case["keep"])
        return {"out": out, "k": state["cache"][0], "v": state["cache"][1]}
    if path == "latent":
        H, D, E = case["heads"], case["dim"], case["vdim"]
        # the call turns the queries in place: a pass starts from fresh ones,
        # as a projection makes them
        out = sv.latent_attention(
            state["q"].clone(), state["kv"], state["gate"], state["batch"],
            state["cache"], state["weights"], H, D, E, (D + SHARED) ** -0.5,
            EPS, case["window"])
        return {"out": out, "cache": state["cache"]}
    if path == "experts":
        pending = sv.moe_mlp(state["h"], state["z"], state["bias"],
                             state["gate_up"], state["down"], case["top"],
                             ALPHA, LIMIT, SHIFT)
        x, h, _ = sv.residual_norm(state["x"], pending, EPS, state["weight"])
        return {"x": x, "h": h}
    q, k, v, z = _memory_parts(case, state["proj"])
    gate = state.get("gating") or sv.TimeGate(
        state["raw"], state["bias"], state["A_log"], state["skip"], z)
    out = sv.memory_mix(q, k, v, gate, state["S"], state["n"], state["m"],
                        state["seg"], case["heads"], *state["chunks"])
    return {"out": out, "S": state["S"], "n": state["n"], "m": state["m"]}


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _pairs(context, tokens, window=0, keep=0):
    """Visible (query, key) pairs of new tokens behind a context."""
    total = 0
    if window <= 0:
        return tokens * context + tokens * (tokens + 1) // 2
    for i in range(context, context + tokens):
        lo = max(0, i - window + 1)
        total += i + 1 - lo + min(keep, lo)
    return total


def _seen(context, tokens, window=0, keep=0):
    """Keys that any of the new tokens sees."""
    lo = max(0, context - window + 1) if window > 0 else 0
    return context + tokens - lo + min(keep, lo)


def _llama_size(case):
    """Weights that are multiplied: of the layers, of the head."""
    W, h, g = case["width"], case["heads"] * HEAD, case["kv_heads"] * HEAD
    return case["layers"] * (W * (2 * h + 2 * g) + 3 * W * case["ff"]), \
        W * case["vocab"]


def work(case):
    path = case["path"]
    if path == "train":
        B, S = case["batch"], case["seq"]
        n, head = _llama_size(case)
        pairs = B * _pairs(0, S) * case["layers"] * case["heads"] * HEAD
        return {"flops": 6.0 * (n + head) * B * S + 12.0 * pairs,
                "bytes": 4.0 * (n + 2 * head)}
    if path == "attention":
        B, S, H, G = (case[k] for k in ("batch", "seq", "heads", "kv_heads"))
        pairs = B * _pairs(0, S, case["window"]) * H * HEAD
        return {"flops": 12.0 * pairs,
                "bytes": 2.0 * B * S * HEAD * (4 * H + 4 * G)}
    if path == "generate":
        n, head = _llama_size(case)
        B, P = case["requests"], case["prompt"]
        lens = [max(2, x) for x in _split(P, B)]
        pairs = sum(_pairs(0, x + NEW - 1) for x in lens) * \
            case["layers"] * case["heads"] * HEAD
        # every step reads the weights, a decoding one its requests' keys
        keys = sum(x + t for x in lens for t in range(1, NEW))
        return {"flops": 2.0 * n * (sum(lens) + B * (NEW - 1)) +
                2.0 * head * B * NEW + 4.0 * pairs,
                "bytes": 2.0 * NEW * (n + head) + 4.0 * keys *
                case["layers"] * case["kv_heads"] * HEAD +
                4.0 * B * NEW * case["vocab"]}
    if path in ("paged", "latent"):
        rows, W = _rows(case), case["window"]
        keep, H = case.get("keep", 0), case["heads"]
        T = sum(t for _, t in rows)
        pairs = sum(_pairs(c, t, W, keep) for c, t in rows) * H
        seen = sum(_seen(c, t, W, keep) for c, t in rows)
        if path == "paged":
            G = case["kv_heads"]
            return {"flops": 4.0 * pairs * HEAD,
                    "bytes": 4.0 * G * HEAD * (seen + T) +
                    4.0 * T * H * HEAD}
        D, E = case["dim"], case["vdim"]
        n = case["portions"]
        singles = sum(_pairs(c, t, W) for c, t in rows[n:]) * H
        # portions attend to expanded keys and values, single tokens in the
        # latent space
        expand = sum(_seen(c, t, W) for c, t in rows[:n])
        return {"flops": 2.0 * (pairs - singles) * (D + SHARED + E) +
                2.0 * singles * (2 * RANK + SHARED) +
                2.0 * (expand + case["singles"]) * H * (D + E) * RANK,
                "bytes": 2.0 * (RANK + SHARED) * (seen + T) +
                2.0 * T * H * (D + SHARED + 2 * E) +
                2.0 * H * (D + E) * RANK}
    if path == "experts":
        T, E, top, W, ff = (case[k] for k in ("tokens", "experts", "top",
                                              "width", "ff"))
        used = E * (1 - (1 - top / E) ** T)      # expected
        return {"flops": 6.0 * T * top * W * ff,
                "bytes": 6.0 * used * W * ff + 2.0 * T * W * (1 + 2 + 2 + 1)}
    H, D, E, G = (case[k] for k in ("heads", "dim", "vdim", "groups"))
    B, T = case["requests"], case["tokens"]
    chunk = 1 if case["single"] else 64
    return {"flops": 2.0 * T * H * (chunk / 2 * (D + E) + 2 * D * E),
            "bytes": 2.0 * T * (2 * G * D + 3 * H * E) +
            (8.0 if case["single"] else 4.0) * B * H * D * E}


def tolerance(case):
    """About four times what these paths differ by from ``exact``: 0.003 for the
    gradients of an attention and the latent form, 0.0016 to 0.002 for what is
    rounded once, 0.02 for gradients and logits behind several layers in bf16
    (the most that is allowed, 0.03, stands there)."""
    return {"rel": {"train": 0.03, "attention": 0.012, "generate": 0.03,
                    "paged": 0.007, "latent": 0.013, "experts": 0.008,
                    "memory": 0.007}[case["path"]]}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------

def _rms(x, w=None):
    x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + EPS)
    return x if w is None else x * w


def _rotate(x, pos, base):
    """Element i of the last size turns with element i + half."""
    half = x.shape[-1] // 2
    f = base ** (-torch.arange(half, dtype=torch.float64, device="cuda") /
                 half)
    a = (pos.double()[:, None] * f).reshape(
        pos.shape[0], *[1] * (x.dim() - 2), half)
    u, v = x[..., :half], x[..., half:]
    return torch.cat([u * a.cos() - v * a.sin(),
                      v * a.cos() + u * a.sin()], -1)


def _attend(q, k, v, pos, kpos, scale, window=0, keep=0):
    """q (T, H, D) at positions ``pos`` over k (N, G, D), v (N, G, E) at
    ``kpos``, some rows at a time."""
    T, H = q.shape[:2]
    rep = H // k.shape[1]
    k, v = k.permute(1, 2, 0), v.transpose(0, 1)
    out, rows = [], max(1, (1 << 28) // (H * kpos.shape[0]))
    for a in range(0, T, rows):
        p = pos[a:a + rows, None]
        gone = kpos > p
        if window > 0:
            gone = gone | ((p - kpos >= window) & (kpos >= keep))
        x = q[a:a + rows].reshape(-1, H // rep, rep, q.shape[2])
        x = x.permute(1, 2, 0, 3)                       # (G, rep, t, D)
        s = torch.matmul(x, k[:, None]) * scale
        s = s.masked_fill(gone, -math.inf).softmax(-1)
        out.append(torch.matmul(s, v[:, None]).permute(2, 0, 1, 3).reshape(
            -1, H, v.shape[2]))
    return torch.cat(out)


def _llama64(case, w, ids):
    """The decoder's last rows (batch, sequence, width)."""
    B, S = ids.shape
    H, G = case["heads"], case["kv_heads"]
    pos = torch.arange(S, device="cuda")

    def attend(q, k, v):
        return torch.stack([_attend(
            _rotate(q[b].view(S, H, HEAD), pos, ROPE_BASE),
            _rotate(k[b].view(S, G, HEAD), pos, ROPE_BASE),
            v[b].view(S, G, HEAD), pos, pos, HEAD ** -0.5).reshape(S, -1)
            for b in range(B)])

    def layer(x, p):
        h = _rms(x, w[p + "input_layernorm.weight"])
        q, k, v = (h @ w[p + "self_attn.qkv_proj.weight_" + n].t()
                   for n in "qkv")
        x = x + attend(q, k, v) @ w[p + "self_attn.o_proj.weight"].t()
        h = _rms(x, w[p + "post_attention_layernorm.weight"])
        g, u = (h @ w[p + "mlp.gate_up_proj.weight"].t()).chunk(2, -1)
        return x + (F.silu(g) * u) @ w[p + "mlp.down_proj.weight"].t()

    x = w["model.embed_tokens.weight"][ids]
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        x = checkpoint(layer, x, p, use_reentrant=False) \
            if torch.is_grad_enabled() else layer(x, p)
    return _rms(x, w["model.norm.weight"])


def _exact_train(case, r):
    w = {n: t.double().requires_grad_()
         for n, t in _llama_weights(case, r).items()}
    ids = _tokens(case, r)

    def loss_of(h):
        z = h[:-1] @ w["lm_head.weight"].t()
        return lambda t: F.cross_entropy(z, t, reduction="sum")

    with torch.enable_grad():
        h = _llama64(case, w, ids)
        loss = sum(checkpoint(lambda x, t: loss_of(x)(t), h[b], ids[b, 1:],
                              use_reentrant=False)
                   for b in range(ids.shape[0]))
        loss = loss / (ids.shape[0] * (ids.shape[1] - 1))
        loss.backward()
    return {"loss": loss.detach(), "grad": {n: t.grad for n, t in w.items()}}


def _exact_attention(case, r):
    q, k, v, grad = (t.double() for t in _heads(case, r))
    B, S, H, _ = q.shape
    G = case["kv_heads"]
    rep, W = H // G, case["window"]
    out, dq = torch.empty_like(q), torch.empty_like(q)
    dk, dv = torch.zeros_like(k), torch.zeros_like(v)
    pos = torch.arange(S, device="cuda")
    gone = pos > pos[:, None]
    if W:
        gone |= pos[:, None] - pos >= W
    for b in range(B):
        for h in range(H):
            g = h // rep
            a, c, d = q[b, :, h] * HEAD ** -0.5, k[b, :, g], v[b, :, g]
            p = (a @ c.t()).masked_fill_(gone, -math.inf).softmax(-1)
            o = p @ d
            y = grad[b, :, h]
            ds = p * (y @ d.t() - (y * o).sum(-1, keepdim=True))
            out[b, :, h] = o
            dq[b, :, h] = ds @ c * HEAD ** -0.5
            dk[b, :, g] += ds.t() @ a
            dv[b, :, g] += p.t() @ y
    return {"out": out.transpose(1, 2), "dq": dq, "dk": dk, "dv": dv}


def _exact_generate(case, r):
    w = {n: t.double() for n, t in _llama_weights(case, r).items()}
    prompts, new = _requests(case, r)
    lens = [len(p) for p in prompts]
    L = max(lens) + NEW
    ids = torch.tensor([(p + n + [0] * L)[:L] for p, n in zip(prompts, new)],
                       device="cuda")
    at = torch.tensor(lens, device="cuda")[:, None] - 1 + \
        torch.arange(NEW, device="cuda")
    h = torch.cat([_llama64(case, w, ids[b:b + 8])
                   for b in range(0, len(lens), 8)])
    h = h.gather(1, at[..., None].expand(-1, -1, h.shape[2]))
    z = h @ w["lm_head.weight"].t()
    return [z[:, t] for t in range(NEW)]


def _cached(cache, table, n):
    """The first n rows of a request."""
    return cache[table[:-(-n // PAGE)].long()], n


def _exact_paged(case, r):
    batch, proj, cache = _paged_inputs(case, r)
    H, G = case["heads"], case["kv_heads"]
    x = proj.double()
    q, k, v = x.split((H * HEAD, G * HEAD, G * HEAD), dim=1)
    out, at = torch.empty(x.shape[0], H * HEAD, dtype=torch.float64,
                          device="cuda"), 0
    for i, (c, t) in enumerate(_rows(case)):
        kv = []
        for pages, row in zip(cache, (k, v)):
            old, _ = _cached(pages, batch.block_table[i], c + t)
            old = old.transpose(1, 2).reshape(-1, G, HEAD)[:c].double()
            kv.append(torch.cat([old, row[at:at + t].view(t, G, HEAD)]))
        kpos = torch.arange(c + t, device="cuda")
        out[at:at + t] = _attend(
            q[at:at + t].view(t, H, HEAD), *kv, kpos[c:], kpos, HEAD ** -0.5,
            case["window"], case["keep"]).reshape(t, -1)
        at += t
    return {"out": out, "k": None, "v": None}


def _exact_latent(case, r):
    s = _latent_inputs(case, r)
    H, D, E = case["heads"], case["dim"], case["vdim"]
    w = {n: s[n].double() for n in ("q", "kv", "gate", "norm", "uk", "uv")}
    T = w["q"].shape[0]
    out, at = torch.empty(T, H * E, dtype=torch.float64, device="cuda"), 0
    for i, (c, t) in enumerate(_rows(case)):
        kpos = torch.arange(c + t, device="cuda")
        old, _ = _cached(s["cache"], s["batch"].block_table[i], c + t)
        old = old.reshape(-1, RANK + SHARED)[:c].double()
        new = w["kv"][at:at + t]
        lat = torch.cat([old[:, :RANK], _rms(new[:, :RANK], w["norm"])])
        rot = torch.cat([old[:, RANK:],
                         _rotate(new[:, RANK:], kpos[c:], ROT_BASE)])
        k = torch.cat([(lat @ w["uk"].t()).view(-1, H, D),
                       rot[:, None].expand(-1, H, -1)], -1)
        v = (lat @ w["uv"].t()).view(-1, H, E)
        q = w["q"][at:at + t].view(t, H, D + SHARED)
        q = torch.cat([q[..., :D], _rotate(q[..., D:], kpos[c:], ROT_BASE)],
                      -1)
        o = _attend(q, k, v, kpos[c:], kpos, (D + SHARED) ** -0.5,
                    case["window"])
        out[at:at + t] = o.reshape(t, -1) * w["gate"][at:at + t].sigmoid()
        at += t
    return {"out": out, "cache": None}


def _exact_experts(case, r):
    s = _experts_inputs(case, r)
    val, idx = (s["z"] + s["bias"].float()).topk(case["top"])
    coef = val.double().softmax(-1)
    h, y = s["h"].double(), torch.zeros_like(s["x"], dtype=torch.float64)
    for e in range(case["experts"]):
        row, k = (idx == e).nonzero(as_tuple=True)
        g, u = (h[row] @ s["gate_up"][e].double().t()).chunk(2, -1)
        g, u = g.clamp(max=LIMIT), u.clamp(-LIMIT, LIMIT)
        a = g * torch.sigmoid(ALPHA * g) * (u + SHIFT)
        y.index_add_(0, row, coef[row, k, None] *
                     (a @ s["down"][e].double().t()))
    x = s["x"].double() + y
    return {"x": x, "h": _rms(x, s["weight"].double())}


def _exact_memory(case, r):
    s = _memory_inputs(case, r)
    H, D, E, G = (case[k] for k in ("heads", "dim", "vdim", "groups"))
    T, kind = case["tokens"], case["gate"]
    q, k, v, z = (t.double() for t in _memory_parts(case, s["proj"]))
    if kind == "decay":
        q, k, v = F.silu(q), F.silu(k), F.silu(v)
    q, k = (t.reshape(T, G, D).repeat_interleave(H // G, 1) for t in (q, k))
    v = v.reshape(T, H, E)
    keep = torch.ones(T, H, dtype=torch.float64, device="cuda")
    take = keep.clone()
    if kind == "decay":
        keep *= torch.tensor(s["decay"], dtype=torch.float64, device="cuda")
    elif kind == "time":
        take = F.softplus(s["raw"].double() + s["bias"].double())
        keep = torch.exp(-s["A_log"].double().exp() * take)
    else:
        i, f = (15.0 * torch.tanh((x.double() + b.double()) / 15.0) for x, b
                in zip(s["raw"].chunk(2, -1), (s["i_bias"], s["f_bias"])))
        f = F.logsigmoid(f)
        q = q * D ** -0.5
    out = torch.empty(T, H, E, dtype=torch.float64, device="cuda")
    S_all, n_all, m_all = s["S"].double(), s["n"], s["m"]
    if kind == "exp":
        n_all, m_all = n_all.double(), m_all.double()
    for b, at, rows, ctx in s["segs"]:
        S = S_all[b] if ctx else torch.zeros_like(S_all[b])
        if kind == "exp":
            n = n_all[b, :, 0] if ctx else torch.zeros_like(n_all[b, :, 0])
            m = m_all[b, :, 0] if ctx else torch.zeros_like(m_all[b, :, 0])
        for t in range(at, at + rows):
            a, c = keep[t], take[t]
            if kind == "exp":
                top = torch.maximum(f[t] + m, i[t])
                a, c = torch.exp(f[t] + m - top), torch.exp(i[t] - top)
                m = top
                n = a[:, None] * n + c[:, None] * k[t]
            S = a[:, None, None] * S + \
                (c[:, None] * k[t])[..., None] * v[t][:, None]
            o = (q[t][:, None] @ S)[:, 0]
            if kind == "exp":
                o = o / (torch.maximum((n * q[t]).sum(-1).abs(),
                                       torch.exp(-m)) + 1e-6)[:, None]
            out[t] = o
        S_all[b] = S
        if kind == "exp":
            n_all[b], m_all[b] = n[:, None], m[:, None]
    if kind == "time":
        out = (out + s["skip"].double()[:, None] * v) * \
            F.silu(z.reshape(T, H, E))
    return {"out": out.reshape(T, H * E), "S": S_all, "n": n_all, "m": m_all}


_EXACT = {"train": _exact_train, "attention": _exact_attention,
          "generate": _exact_generate, "paged": _exact_paged,
          "latent": _exact_latent, "experts": _exact_experts,
          "memory": _exact_memory}


def exact(case, seed):
    with torch.no_grad():
        return _EXACT[case["path"]](case, _Source(seed))
