"""Engine steps that stand for what a user of the framework runs: one step is one pass of the model over the
tokens that the scheduler put together (decoded tokens, prompt portions, or both), as the serving loop runs it -
metadata built and uploaded, the step's hipGraph replayed, the samplers run, the step before it collected.

The models are slices of the repository's presets: their layer sizes as they are, a few layers of each and a smaller
vocabulary, so that a step's layers weigh as much against its output matrix as they do at full depth. A case:

  model    preset; quant "awq" for int4 weights (transformers), "" for bf16
  decode   sequences that decode one token each, after about `context` tokens of their own
  prompts  sequences whose prompt of about `tokens` tokens is read in this step, from its start

Lengths within a step are unequal, as they are in real batches (see `spread`).
"""
import math
import shutil
import tempfile
import zlib

import torch

from vgate.models.config import resolve_arch
from vgate.models.hybrid import save_checkpoint
from vgate.runtime.engine import EngineConfig, LLMEngine
from vgate.runtime.model_runner import DEFAULT_T_BUCKETS
from vgate.runtime.sampling_params import SamplingParams
from vgate.runtime.scheduler import ScheduledBatch
from vgate.runtime.sequence import Sequence

BLOCK = 16          # tokens in a page of the paged caches
STEP_TOKENS = 2048  # most tokens of one step (the engine's default)

# transformers: hidden, heads, key/value heads, feed-forward, base of the rotation, eps, bias on q / k / v, tied output matrix
TRANSFORMERS = {
    "qwen2.5-1.5b": dict(W=1536, H=12, G=2, F=8960, base=1e6, eps=1e-6, bias=True, tied=True, layers=6, vocab=32000),
    "llama-3-8b": dict(W=4096, H=32, G=8, F=14336, base=5e5, eps=1e-5, bias=False, tied=False, layers=4, vocab=32000),
}
# layered hybrid designs: width, heads of 128, feed-forward, ...; low-rank pairs inside a mixer are RANK wide
RANK = 16
HYBRIDS = {
    # latent attention with routed experts, then the generalized delta rule with a dense feed-forward. The layer with the
    # router comes first: its choice of experts then rests on the embedding alone and does not turn on rounding.
    "zadirax-bench-1024": dict(kind="zadirax", W=1024, H=8, F=4096, KR=256, QR=512, R=64, E=8, top=2, EF=2048, vocab=8192),
    # gated linear attention, window attention over pooled blocks, window attention beside lightning attention
    "pozalorn-bench-1024": dict(kind="pozalorn", W=1024, H=8, G=2, F=4096, window=1024, pool=64, vocab=8192),
    # latent attention, window attention beside the gated delta rule, selective scan
    "vugudra-bench-1536": dict(kind="vugudra", W=1536, H=12, G=2, F=8960, KR=512, QR=768, R=64, window=1024, keep=64,
                               C=3072, N=16, DT=96, taps=4, vocab=8192),
}
D = 128  # head size of every one of them


def listed():
    c = lambda name, model, quant="", decode=0, context=0, prompts=0, tokens=0: dict(  # noqa: E731
        name=name, model=model, quant=quant, decode=decode, context=context, prompts=prompts, tokens=tokens)
    return [
        # one user at the keyboard: the smallest step there is, all latency
        c("chat of one", "qwen2.5-1.5b", decode=1, context=96),
        # the headline load: eight clients, answers of 64 tokens
        c("eight clients decode", "qwen2.5-1.5b", decode=8, context=96),
        # a busy server: many sequences of some hundred tokens
        c("64 clients decode", "qwen2.5-1.5b", decode=64, context=600),
        # the headline load's waves: eight new prompts at once
        c("eight clients arrive", "qwen2.5-1.5b", prompts=8, tokens=48),
        # int4 weights under continuous batching: a prompt read beside the running sequences
        c("int4, prompt among decodes", "qwen2.5-1.5b", quant="awq", decode=23, context=300, prompts=1, tokens=210),
        # time to first token of a long prompt: the largest step
        c("8B long prompt", "llama-3-8b", prompts=1, tokens=2048),
        # the layered designs: a long prompt, and a batch of decoding sequences, of each
        c("zadirax prompt", "zadirax-bench-1024", prompts=1, tokens=1999),
        c("zadirax decode", "zadirax-bench-1024", decode=32, context=512),
        c("pozalorn prompt", "pozalorn-bench-1024", prompts=1, tokens=1801),
        c("pozalorn decode", "pozalorn-bench-1024", decode=16, context=1500),
        c("vugudra prompts among decodes", "vugudra-bench-1536", decode=5, context=200, prompts=3, tokens=601),
        c("vugudra decode", "vugudra-bench-1536", decode=32, context=700),
    ]


def draw(rng):
    log = lambda lo, hi: int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))  # noqa: E731
    model, quant = rng.choice([("qwen2.5-1.5b", ""), ("qwen2.5-1.5b", "awq"), ("llama-3-8b", ""), ("zadirax-bench-1024", ""),
                               ("pozalorn-bench-1024", ""), ("vugudra-bench-1536", "")])
    kind = rng.choice(["decode", "prompts", "both"])
    case = dict(model=model, quant=quant, decode=0, context=0, prompts=0, tokens=0)
    if kind != "prompts":
        case["decode"] = log(1, 64)
        case["context"] = log(16, min(1600, 40000 // case["decode"]))
    if kind != "decode":
        case["prompts"] = log(1, 8)
        most = (1000 if kind == "both" or model == "llama-3-8b" else 1900) // case["prompts"]
        case["tokens"] = log(9, most)
    return case


def spread(mean, count):
    """`count` unequal lengths around `mean`, the same for every seed."""
    return [max(2, round(mean * (0.75 + 0.5 * ((i + 1) * 0.618 % 1.0)))) for i in range(count)] if count > 1 else [mean] * count


def lengths(case):
    """(tokens before the step, tokens in the step) of every sequence."""
    return [(n, 1) for n in spread(case["context"], case["decode"])] + [(0, n) for n in spread(case["tokens"], case["prompts"])]


def token_ids(case, seed):
    sizes = TRANSFORMERS.get(case["model"]) or HYBRIDS[case["model"]]
    g = torch.Generator().manual_seed(seed * 7919 + 5)
    return [torch.randint(0, sizes["vocab"], (a + n,), generator=g).tolist() for a, n in lengths(case)]


# ------------------------------------------------------------------------------------------------------- the step
def prepare(case, seed):
    todo, ids = lengths(case), token_ids(case, seed)
    S = 1 << max(0, (len(todo) - 1).bit_length())
    nt = sum(n for _, n in todo)
    T = min(b for b in DEFAULT_T_BUCKETS if b >= (max(nt, S + 1) if case["prompts"] else nt))
    longest = max(a + n for a, n in todo)
    cfg = dict(model=case["model"], quantization=case["quant"] or None, device="cuda", seed=seed, max_num_seqs=S,
               max_model_len=(longest + 64) // 64 * 64, max_num_batched_tokens=max(T, STEP_TOKENS), graph_token_buckets=[T],
               num_kv_blocks=sum(-(-(a + n) // BLOCK) for a, n in todo) + 1, enable_prefix_caching=False)
    if case["model"] in TRANSFORMERS:
        m = TRANSFORMERS[case["model"]]
        engine = LLMEngine(EngineConfig(arch_overrides=dict(num_layers=m["layers"], vocab_size=m["vocab"]), **cfg))
    else:
        m = HYBRIDS[case["model"]]
        arch = resolve_arch(case["model"])
        order = (1, 0) if m["kind"] == "zadirax" else range(3)
        over = dict(vocab_size=m["vocab"], layers=tuple(arch.layers[i] for i in order))
        where = tempfile.mkdtemp(prefix="perf_weights_")
        try:
            save_checkpoint(arch, {k: v.cpu() for k, v in tensors(case["model"], seed).items()}, where, {})
            engine = LLMEngine(EngineConfig(weights_path=where, arch_overrides=over, **cfg))
        finally:
            shutil.rmtree(where)
    runner, seqs = engine.runner, []
    for i, (t, (a, n)) in enumerate(zip(ids, todo)):  # every other sequence samples, the rest take the likeliest token
        s = Sequence("r%d" % i, t, SamplingParams(temperature=0.8, top_p=0.95) if i % 2 else SamplingParams(temperature=0.0), seed=seed + i)
        if not engine.kvm.ensure(s, a + n):
            raise RuntimeError("too few cache pages")
        seqs.append(s)
    while True:  # the tokens before the step, in portions, as the scheduler would send them
        items, room = [], STEP_TOKENS
        for s, (a, _) in zip(seqs, todo):
            n = min(a - s.num_computed, room)
            if n > 0:
                items.append((s, n))
                room -= n
        if not items:
            break
        runner.collect(runner.launch(ScheduledBatch(items, STEP_TOKENS - room, STEP_TOKENS - room, 0, [])))
        for s, n in items:
            s.num_computed += n
    runner.warmup([T], [S])
    batch = ScheduledBatch([(s, n) for s, (_, n) in zip(seqs, todo)], nt, nt - case["decode"], case["decode"], [])
    return {"engine": engine, "batch": batch, "seqs": len(seqs), "last": None}


def run(state):
    """Launch the step, then collect the one before it: the serving loop's order. Returns the step's logits with what else
    it wrote: the last layer's keys and values, or the recurrent states."""
    runner = state["engine"].runner
    handle = runner.launch(state["batch"])
    if state["last"] is not None:
        runner.collect(state["last"])
    state["last"] = handle
    out = {"logits": runner.graphs[handle.bucket].vg_out[1][: state["seqs"]]}
    if hasattr(runner.model, "allocate_caches"):
        out["state"] = recurrent(runner.kv)
    else:
        out["keys"], out["values"] = runner.kv[-1]
    return out


def recurrent(caches):
    """The fp32 tensors among the layers' caches, in order."""
    if isinstance(caches, torch.Tensor):
        return [caches] if caches.dtype == torch.float32 else []
    return [t for c in caches if c is not None for t in recurrent(c)]


# --------------------------------------------------------------------------------------------------- what it costs
def work(case):
    todo, T = lengths(case), sum(n for _, n in lengths(case))
    S = len(todo)
    # query-key pairs that causal attention has to look at, and keys that have to be read
    pairs = sum(n * a + n * (n + 1) // 2 for a, n in todo)
    keys = sum(a + n for a, n in todo)
    if case["model"] in TRANSFORMERS:
        m = TRANSFORMERS[case["model"]]
        per = m["W"] * (m["H"] + 2 * m["G"]) * D + m["H"] * D * m["W"] + 3 * m["W"] * m["F"]
        weights = m["layers"] * per * (0.5 + 4 / 128 if case["quant"] else 2) + m["W"] * m["vocab"] * 2
        flops = 2 * T * m["layers"] * per + 4 * pairs * m["H"] * D * m["layers"] + 2 * S * m["W"] * m["vocab"]
        cache = m["layers"] * 2 * m["G"] * D * 2 * (keys + T)
        return {"bytes": weights + cache + T * m["W"] * 2 + S * m["vocab"] * 4, "flops": flops}
    m = HYBRIDS[case["model"]]
    shapes = {k: math.prod(v) for k, v in tensor_shapes(case["model"]).items()}
    matrices = sum(v for k, v in shapes.items() if v > 4 * m["W"] and k not in ("embed", "head") and ".e" not in k)
    flops, bytes_ = 2 * T * matrices + 2 * S * m["W"] * m["vocab"], 2 * (matrices + m["W"] * m["vocab"])
    state = lambda per: 8 * S * per  # noqa: E731  (read and written, fp32)
    seen = sum(min(a + i + 1, m.get("window", 1 << 30)) for a, n in todo for i in range(n))
    near = sum(min(a + n, m.get("window", 1 << 30) + n) for a, n in todo)
    latent = lambda: (2 * pairs * m["H"] * (2 * m["KR"] + m["R"]), 2 * (keys + T) * (m["KR"] + m["R"]))  # noqa: E731
    if m["kind"] == "zadirax":
        expert = 3 * m["W"] * m["EF"]
        f, b = latent()
        flops += f + 2 * T * m["top"] * expert + 8 * T * m["H"] * D * D
        bytes_ += b + 2 * min(m["E"], T * m["top"]) * expert + state(m["H"] * D * D)
    elif m["kind"] == "pozalorn":
        flops += 2 * 4 * T * m["H"] * D * D + 2 * 4 * seen * m["H"] * D
        bytes_ += 2 * state(m["H"] * D * D) + 2 * 2 * 2 * m["G"] * D * (near + T)
    else:
        f, b = latent()
        flops += f + 4 * seen * m["H"] * D + 8 * T * m["H"] * D * D + 6 * T * m["C"] * m["N"]
        bytes_ += b + 2 * 2 * m["G"] * D * (near + T) + state(m["H"] * D * D + m["C"] * m["N"])
    return {"bytes": bytes_ + T * m["W"] * 2 + S * m["vocab"] * 4, "flops": flops}


def tolerance(case):
    """bf16 activations through a few layers, fp32 sums. Against 64 bits: bf16 transformers 0.9e-2 to 1.1e-2, int4 ones 3e-3 (their
    short and long steps round the weights in different places), layered designs 4e-3 to 7e-3 (states 2e-3 to 7e-3)."""
    if case["model"] in TRANSFORMERS:
        return {"rel": 0.013 if case["quant"] else 0.03}
    return {"rel": 0.025}


# ------------------------------------------------------------------------------------------------------ the weights
def tensor_shapes(model):
    """name -> shape of a layered design's checkpoint."""
    m = HYBRIDS[model]
    W, H, F, V = m["W"], m["H"], m["F"], m["vocab"]
    n = H * D
    out = {"embed": (V, W), "head": (V, W), "final.norm": () if m["kind"] == "zadirax" else (W,)}
    put = lambda pre, **t: out.update({pre + k.replace("__", "."): v for k, v in t.items()})  # noqa: E731
    dense = lambda i: put("l%d.mlp." % i, gate=(F, W), up=(F, W), down=(W, F))  # noqa: E731

    def latent(pre, gate):
        put(pre, dq=(m["QR"], W), dq__norm=(m["QR"],), uq=(H * (D + m["R"]), m["QR"]), dkv=(m["KR"] + m["R"], W),
            dkv__norm=(m["KR"],), uk=(n, m["KR"]), uv=(n, m["KR"]), g=(gate, W), o=(W, n))

    def window(pre, norm):
        g = m["G"] * D
        put(pre, q=(n, W), k=(g, W), v=(g, W), o=(W, n), q__b=(n,), k__b=(g,), v__b=(g,),
            q__norm=(n,) if norm == "all" else (D,), k__norm=(g,) if norm == "all" else (D,))

    linear = lambda pre, norm: put(pre, q=(n, W), k=(n, W), v=(n, W), g=(n, W), o=(W, n), norm=(norm,))  # noqa: E731
    if m["kind"] == "zadirax":
        latent("l0.mix.", n)
        put("l0.mlp.", router=(m["E"], W), correction=(m["E"],))
        for e in range(m["E"]):
            put("l0.mlp.e%d." % e, gate=(m["EF"], W), up=(m["EF"], W), down=(W, m["EF"]))
        put("l1.mix.", **{k: (n, W) for k in "rkvga"}, a__b=(n,), w1=(RANK, W), w2=(n, RANK), w0=(n,), norm=(n,), o=(W, n))
        dense(1)
        for i in (0, 1):
            put("l%d." % i, norm1=(), rg1=(W, W), rg1__b=(W,), rg2=(W, W), rg2__b=(W,))
        return out
    if m["kind"] == "pozalorn":
        linear("l0.mix.", D)
        put("l0.mix.", a1=(RANK, W), a2=(n, RANK), a2__b=(n,))
        window("l1.mix.", "all")
        window("l2.mix.left.", "head")
        put("l2.mix.left.", sink=(H,), o__b=(W,))
        linear("l2.mix.right.", n)
        for i in range(3):
            put("l%d." % i, dwa=(i + 2,))
    else:
        latent("l0.mix.", H)
        put("l0.mix.", sink=(H,))
        put("l1.mix.left.", q=(n, W), k=(m["G"] * D, W), o=(W, n), q__norm=(D,), k__norm=(D,), out=(W,))
        put("l1.mix.right.", **{k: (n, W) for k in "qkv"}, **{k + "__conv": (n, m["taps"]) for k in "qkv"}, b=(H, W), A_log=(H,),
            norm=(D,), a1=(RANK, W), a2=(n, RANK), dt_bias=(n,), g1=(RANK, W), g2=(n, RANK), o=(W, n), out=(W,))
        C, N = m["C"], m["N"]
        put("l2.mix.", **{"in": (2 * C, W)}, conv=(C, m["taps"]), conv__b=(C,), x=(m["DT"] + 2 * N, C), dt=(C, m["DT"]), dt__b=(C,),
            A_log=(C, N), D=(C,), o=(W, C))
    for i in range(3):
        dense(i)
        put("l%d." % i, norm1=(W,), norm2=(W,))
    return out


def tensors(model, seed, device="cuda"):
    """Random bf16 weights that keep activations near 1: matrices ~ N(0, 1 / fan in), norms near 1 (those of the third
    design are stored around 0), small biases. Every tensor has a stream of its own."""
    out = {}
    around_zero = HYBRIDS[model]["kind"] == "vugudra"
    for name, shape in tensor_shapes(model).items():
        g = torch.Generator(device).manual_seed((seed * 1000003 + zlib.crc32(name.encode())) & 0x7FFFFFFF)
        leaf = name.rsplit(".", 1)[-1]
        w = torch.randn(shape, generator=g, device=device)
        if leaf == "dwa":  # close to "hand on the newest result"
            w = 0.1 * w / shape[0]
            w[-1] += 1.0
        elif leaf.startswith("norm") or leaf == "out":
            w = 0.1 * w + (0.0 if around_zero and (leaf in ("norm1", "norm2") or name == "final.norm") else 1.0)
        elif len(shape) == 2 and leaf != "A_log":
            w = w * (0.5 if name == "embed" else shape[1] ** -0.5)
        else:
            w = 0.3 * w
        out[name] = w.to(torch.bfloat16)
    return out


# ---------------------------------------------------------------------------------- the same step in 64 bits, in torch
def rms(x, eps, w=None):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def angles(dims, base, scaling=None, device="cuda"):
    f = base ** (-torch.arange(0, dims, 2, dtype=torch.float64, device=device) / dims)
    if scaling == "stretched":  # long wavelengths of a context of 8192 stretched eightfold, blended between 2048 and 8192
        turns = 8192 * f / (2 * math.pi)
        blend = ((turns - 1.0) / 3.0).clamp(0.0, 1.0)
        f = (1.0 - blend) * f / 8.0 + blend * f
    elif scaling == "yarn":     # fourfold, of a context of 4096: by the index between 32 turns and one
        index = lambda turns: dims * math.log(4096 / (2.0 * math.pi * turns)) / (2.0 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(index(32)), 0), min(math.ceil(index(1)), dims - 1)
        ramp = ((torch.arange(dims // 2, device=device) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0).double()
        f = f / 4.0 * ramp + f * (1.0 - ramp)
    return f


def turn(x, pos, f, halves, amp=1.0):
    """x [n, heads, d], all of d in pairs: (i, i + d / 2) if `halves`, else (2i, 2i + 1)."""
    a = pos.double()[:, None, None] * f
    c, s = torch.cos(a) * amp, torch.sin(a) * amp
    d = x.shape[-1]
    u, v = (x[..., : d // 2], x[..., d // 2:]) if halves else (x[..., 0::2], x[..., 1::2])
    a, b = u * c - v * s, v * c + u * s
    return torch.cat([a, b], -1) if halves else torch.stack([a, b], -1).flatten(-2)


def attend(q, k, v, scale, seen=None, sink=None):
    """q [n, H, d], k / v [m, G, .] with H a multiple of G; `seen` [n, m] (default: every earlier token)."""
    n, H, G = q.shape[0], q.shape[1], k.shape[1]
    if seen is None:
        seen = torch.ones(n, k.shape[0], dtype=torch.bool, device=q.device).tril()
    out = torch.empty(n, H, v.shape[-1], dtype=q.dtype, device=q.device)
    for h in range(H):
        s = (q[:, h] @ k[:, h * G // H].t() * scale).masked_fill(~seen, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].expand(n, 1)], -1)
        out[:, h] = torch.softmax(s, -1)[:, : k.shape[0]] @ v[:, h * G // H]
    return out


def per_sequence(spans, fn, *xs):
    """fn(tokens' positions, rows of every x) of each sequence alone, put together again."""
    return torch.cat([fn(torch.arange(b - a, device=xs[0].device), *(x[a:b] for x in xs)) for a, b in spans])


def recur(spans, step, state, *xs):
    """Token by token through all sequences side by side: state, o = step(state, rows of xs at this token)."""
    n = [b - a for a, b in spans]
    order = sorted(range(len(n)), key=lambda i: -n[i])   # the longest first: those still running are a prefix
    pad = [torch.nn.utils.rnn.pad_sequence([x[spans[i][0]: spans[i][1]] for i in order], True) for x in xs]
    out = None
    for t in range(max(n)):
        live = sum(1 for v in n if v > t)
        state[:live], o = step(state[:live], *(p[:live, t] for p in pad))
        if out is None:
            out = torch.zeros(len(n), max(n), *o.shape[1:], dtype=o.dtype, device=o.device)
        out[:live, t] = o
    back = sorted(range(len(n)), key=lambda i: order[i])
    return state[back], torch.cat([out[back[i], : n[i]] for i in range(len(n))])


def exact(case, seed):
    ids = token_ids(case, seed)
    ends, spans = 0, []
    for t in ids:
        spans.append((ends, ends + len(t)))
        ends += len(t)
    flat = torch.tensor([t for s in ids for t in s], device="cuda")
    last = torch.tensor([b - 1 for _, b in spans], device="cuda")
    if case["model"] in TRANSFORMERS:
        return {"logits": exact_transformer(case, seed, flat, spans, last), "keys": None, "values": None}
    x, state = HYBRID_EXACT[HYBRIDS[case["model"]]["kind"]](case["model"], seed, flat, spans, last)
    slots = 1 << max(0, (len(ids) - 1).bit_length())   # one for every sequence that the engine may hold
    whole = [torch.cat([s, s.new_zeros(slots - s.shape[0], *s.shape[1:])]) for s in state]
    return {"logits": x, "state": whole}


def exact_transformer(case, seed, ids, spans, last):
    m = TRANSFORMERS[case["model"]]
    g = torch.Generator("cuda").manual_seed(seed * 1000003)   # the weights that the model draws for this seed, in its order
    normal = lambda shape, std: (torch.randn(shape, generator=g, device="cuda") * std).bfloat16().double()  # noqa: E731
    W, H, G, F = m["W"], m["H"], m["G"], m["F"]

    def matrix(rows, cols):
        if not case["quant"]:
            return normal((rows, cols), cols ** -0.5)
        q = torch.randint(0, 16, (rows, cols), generator=g, device="cuda", dtype=torch.int32)
        return (q.double() - 8.0) * torch.tensor(cols ** -0.5 / 4.61).bfloat16().double().item()

    embed = normal((m["vocab"], W), 0.02)
    f = angles(D, m["base"])
    x = embed[ids]
    for _ in range(m["layers"]):
        b = normal(((H + 2 * G) * D,), 0.02) if m["bias"] else 0.0
        wqkv, wo, wgu, wd = matrix((H + 2 * G) * D, W), matrix(W, H * D), matrix(2 * F, W), matrix(W, F)
        q, k, v = (t.unflatten(1, (-1, D)) for t in (rms(x, m["eps"]) @ wqkv.t() + b).split([H * D, G * D, G * D], 1))
        one = lambda p, q, k, v: attend(turn(q, p, f, True), turn(k, p, f, True), v, D ** -0.5)  # noqa: E731
        x = x + per_sequence(spans, one, q, k, v).flatten(1) @ wo.t()
        gate, up = (rms(x, m["eps"]) @ wgu.t()).split(F, 1)
        x = x + (torch.nn.functional.silu(gate) * up) @ wd.t()
    head = embed if m["tied"] else normal((m["vocab"], W), W ** -0.5)
    return rms(x[last], m["eps"]) @ head.t()


class Tensors:
    """A design's weights in 64 bits, by name below a prefix."""

    def __init__(self, all_, prefix=""):
        self.all, self.prefix = all_, prefix

    def __getitem__(self, name):
        return self.all[self.prefix + name].double()

    def sub(self, name):
        return Tensors(self.all, self.prefix + name + ".")

    def lin(self, x, name):
        return x @ self[name].t()

    def heads(self, x, name):
        return self.lin(x, name).unflatten(1, (-1, D))


def exact_latent(m, t, h, spans, halves, scaling, amp, sink):
    q = t.lin(rms(t.lin(h, "dq"), 1e-6, t["dq.norm"]), "uq").unflatten(1, (m["H"], -1))
    kv = t.lin(h, "dkv")
    c = rms(kv[:, : m["KR"]], 1e-6, t["dkv.norm"])
    f = angles(m["R"], 10000.0, scaling)

    def one(p, q, k, v, kr):
        kr = turn(kr[:, None], p, f, halves, amp).expand(-1, m["H"], -1)
        q = torch.cat([q[..., :D], turn(q[..., D:], p, f, halves, amp)], -1)
        return attend(q, torch.cat([k, kr], -1), v, (D + m["R"]) ** -0.5, sink=sink)

    o = per_sequence(spans, one, q, t.heads(c, "uk"), t.heads(c, "uv"), kv[:, m["KR"]:])
    gate = torch.sigmoid(t.lin(h, "g"))
    return t.lin((o * (gate.unflatten(1, (m["H"], -1)))).flatten(1), "o")


def exact_dense(t, h, act):
    return t.lin(act(t.lin(h, "gate")) * t.lin(h, "up"), "down")


def exact_zadirax(model, seed, ids, spans, last):
    m, eps = HYBRIDS[model], 1e-6
    all_ = tensors(model, seed)
    t = Tensors(all_)
    x, sig = t["embed"][ids], torch.sigmoid

    def add(i, h, y, ff):
        L = t.sub("l%d" % i)
        return x + y * sig(L.lin(h, "rg1") + L["rg1.b"]) + ff * sig(L.lin(h, "rg2") + L["rg2.b"])

    h = rms(x, eps) * t["l0.norm1"]
    y = exact_latent(m, t.sub("l0.mix"), h, spans, False, None, 1.0, None)
    moe = t.sub("l0.mlp")
    s = sig(moe.lin(h, "router"))
    pick = torch.topk(s + moe["correction"], m["top"], -1).indices
    w = s.gather(1, pick)
    w = w / w.sum(-1, keepdim=True)
    ff = torch.zeros_like(x)
    for e in range(m["E"]):
        tok, slot = torch.where(pick == e)
        E = moe.sub("e%d" % e)
        a, u = E.lin(h[tok], "gate").clamp(max=7.0), E.lin(h[tok], "up").clamp(-7.0, 7.0)
        ff.index_add_(0, tok, E.lin(a * sig(1.702 * a) * (u + 1.0), "down") * w[tok, slot, None])
    x = add(0, h, y, ff)

    h = rms(x, eps) * t["l1.norm1"]
    d = t.sub("l1.mix")
    r, k, v, g, a = (d.heads(h, n) for n in "rkvga")
    decay = torch.exp(-math.exp(-0.5) * sig(d.lin(torch.tanh(d.lin(h, "w1")), "w2") + d["w0"])).unflatten(1, (-1, D))
    u = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    au = sig(a + d["a.b"].view(-1, D)) * u

    def step(S, w, au, u, k, v, r):
        S = w[..., None] * S - au[..., None] * (u[..., None, :] @ S) + k[..., None] * v[..., None, :]
        return S, (r[..., None, :] @ S)[..., 0, :]

    state, o = recur(spans, step, x.new_zeros(len(spans), m["H"], D, D), decay, au, u, k, v, r)
    o = rms(o, eps) * d["norm"].view(-1, D) * sig(g)
    x = add(1, h, d.lin(o.flatten(1), "o"), exact_dense(t.sub("l1.mlp"), h, torch.nn.functional.silu))
    return t.lin(rms(x[last], eps) * t["final.norm"], "head"), [state]


def exact_linear(t, h, spans, decay, act, q_scale):
    """S <- diag(decay) S + k v^T, o = S^T q (fp64), of all heads."""
    q, k, v = (act(t.heads(h, n)) for n in "qkv")

    def step(S, a, q, k, v):
        S = a[..., None] * S + k[..., None] * v[..., None, :]
        return S, (q[..., None, :] @ S)[..., 0, :]

    return recur(spans, step, h.new_zeros(len(spans), q.shape[1], D, D), decay, q * q_scale, k, v)


def exact_pozalorn(model, seed, ids, spans, last):
    m, eps = HYBRIDS[model], 1e-6
    t = Tensors(tensors(model, seed))
    H, P, window = m["H"], m["pool"], m["window"]
    f, fv = angles(D, 5e5, "stretched"), angles(D, 5e5)
    silu, sig = torch.nn.functional.silu, torch.sigmoid

    def windowed(w, h, whole, sink):
        q, k, v = (w.lin(h, n) + w[n + ".b"] for n in "qkv")
        if whole:
            q, k = rms(q, eps, w["q.norm"]), rms(k, eps, w["k.norm"])
        q, k, v = (y.unflatten(1, (-1, D)) for y in (q, k, v))
        if not whole:
            q, k = rms(q, eps, w["q.norm"]), rms(k, eps, w["k.norm"])

        def one(p, q, k, v):
            q, k = turn(q, p, f, False), turn(k, p, f, False)
            far = p[:, None] - p[None]
            seen = (far >= 0) & (far < window)
            if not whole:   # (the layer with the sink has no pooled blocks, and its values do not turn)
                return attend(q, k, v, D ** -0.5, seen, sink)
            v = turn(v, p, fv, False)
            nb = len(p) // P
            mean = lambda y: y[: nb * P].unflatten(0, (nb, P)).mean(1)  # noqa: E731
            end = torch.arange(nb, device=p.device) * P + P - 1
            seen = torch.cat([end[None] <= p[:, None] - window, seen], 1)
            o = attend(q, torch.cat([mean(k), k]), torch.cat([mean(v), v]), D ** -0.5, seen)
            return turn(o, -p, fv, False)

        return per_sequence(spans, one, q, k, v).flatten(1)

    x = t["embed"][ids]
    seen, states = [x], []
    for i in range(3):
        L = t.sub("l%d" % i)
        mix = L.sub("mix")
        if i == 0:
            z = mix.lin(mix.lin(x, "a1"), "a2") + mix["a2.b"]
            S, o = exact_linear(mix, x, spans, torch.exp(torch.nn.functional.logsigmoid(z) / 16.0).unflatten(1, (-1, D)),
                                lambda y: y, D ** -0.5)
            y = mix.lin((rms(o, eps, mix["norm"]) * silu(mix.heads(x, "g"))).flatten(1), "o")
        elif i == 1:
            y = mix.lin(windowed(mix, x, True, None), "o")
        else:
            a, b = mix.sub("left"), mix.sub("right")
            y = a.lin(windowed(a, x, False, a["sink"]), "o") + a["o.b"]
            fade = torch.tensor([math.exp(-(2.0 ** (-8.0 * (j + 1) / H))) for j in range(H)], device=x.device).double()
            S, o = exact_linear(b, x, spans, fade[None, :, None].expand(len(x), -1, D), silu, 1.0)
            y = y + b.lin(rms(o.flatten(1), eps, b["norm"]) * sig(b.lin(x, "g")), "o")
        if i != 1:
            states.append(S)
        x = x + rms(y, eps, L["norm1"])
        x = x + rms(exact_dense(L.sub("mlp"), x, lambda y: torch.nn.functional.gelu(y, approximate="tanh")), eps, L["norm2"])
        seen.append(x)
        x = sum(c * y for c, y in zip(L["dwa"], seen))
    return t.lin(rms(x[last], eps, t["final.norm"]), "head"), states


def exact_vugudra(model, seed, ids, spans, last):
    m, eps = HYBRIDS[model], 1e-6
    t = Tensors(tensors(model, seed))
    silu, sig, soft = torch.nn.functional.silu, torch.sigmoid, torch.nn.functional.softplus
    taps = m["taps"]

    def conv(x, w, b=0.0):
        return per_sequence(spans, lambda p, x: sum(w[:, i] * torch.nn.functional.pad(x, (0, 0, taps - 1 - i, 0))[: len(p)]
                                                    for i in range(taps)) + b, x)

    def kept(x):   # a sequence's last inputs of the convolution
        return torch.stack([torch.nn.functional.pad(x[a:b], (0, 0, taps - 1, 0))[-(taps - 1):] for a, b in spans])

    def beside(mix, h):
        w, r = mix.sub("left"), mix.sub("right")
        q, kp = w.heads(h, "q"), w.heads(h, "k")
        f = angles(D, 10000.0)

        def one(p, q, k, v):
            far = p[:, None] - p[None]
            seen = (far >= 0) & ((far < m["window"]) | (p[None] < m["keep"]))
            return attend(turn(q, p, f, False), turn(k, p, f, False), v, D ** -0.5, seen)

        a = w.lin(per_sequence(spans, one, rms(q, eps, w["q.norm"]), rms(kp, eps, w["k.norm"]), kp).flatten(1), "o")
        raw = [r.lin(h, n) for n in "qkv"]
        q, k, v = (silu(conv(y, r[n + ".conv"])).unflatten(1, (-1, D)) for y, n in zip(raw, "qkv"))
        unit = lambda y: y / torch.sqrt((y * y).sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        z = r.lin(r.lin(h, "a1"), "a2") + r["dt_bias"]
        g = torch.exp(-torch.exp(r["A_log"])[:, None] * soft(z).unflatten(1, (-1, D)))

        def step(S, g, beta, q, k, v):
            S = g[..., None] * S
            u = beta[..., None] * (v - (k[..., None, :] @ S)[..., 0, :])
            S = S + k[..., None] * u[..., None, :]
            return S, (q[..., None, :] @ S)[..., 0, :]

        S, o = recur(spans, step, h.new_zeros(len(spans), m["H"], D, D), g, sig(r.lin(h, "b")), unit(q) * D ** -0.5, unit(k), v)
        b = r.lin((rms(o, eps, r["norm"]) * sig(r.lin(r.lin(h, "g1"), "g2")).unflatten(1, (-1, D))).flatten(1), "o")
        return 0.5 * (rms(a, eps, w["out"]) + rms(b, eps, r["out"])), [S, kept(torch.cat(raw, 1))]

    def scan(mix, h):
        C, N, R = m["C"], m["N"], m["DT"]
        xin, z = mix.lin(h, "in").split(C, 1)
        x = silu(conv(xin, mix["conv"], mix["conv.b"]))
        r, B, Cc = mix.lin(x, "x").split([R, N, N], 1)
        d = soft(mix.lin(r, "dt") + mix["dt.b"])
        A = -torch.exp(mix["A_log"])

        def step(S, d, x, B, Cc):
            S = torch.exp(d[..., None] * A) * S + (d * x)[..., None] * B[:, None]
            return S, (S @ Cc[..., None])[..., 0]

        S, y = recur(spans, step, h.new_zeros(len(spans), C, N), d, x, B, Cc)
        return mix.lin((y + mix["D"] * x) * silu(z), "o"), [S, kept(xin)]

    x, states = t["embed"][ids], []
    for i in range(3):
        L = t.sub("l%d" % i)
        h, mix = rms(x, eps, 1.0 + L["norm1"]), L.sub("mix")
        if i == 0:
            y, S = exact_latent(m, mix, h, spans, True, "yarn", 0.1 * math.log(4.0) + 1.0, mix["sink"]), []
        else:
            y, S = (beside if i == 1 else scan)(mix, h)
        states += S
        x = x + y + exact_dense(L.sub("mlp"), rms(x, eps, 1.0 + L["norm2"]), silu)
    return t.lin(rms(x[last], eps, 1.0 + t["final.norm"]), "head"), states


HYBRID_EXACT = {"zadirax": exact_zadirax, "pozalorn": exact_pozalorn, "vugudra": exact_vugudra}
