"""The cases whose speed is measured: the Qwen3 token loop as a host program
drives it through the binding `rlh` (load a model once, keep a KV cache per
conversation, prefill prompts, decode greedily or with the sampler).

Shapes are those of rlh.SPECS. The 0.6B models are whole; of the larger ones
a slice of a few layers is taken, with the vocabulary cut so that the logits
product keeps the share of a step that it has in the whole model. A slice's
weights exceed the 256 MB last-level cache where the whole model's do, so a
decode step streams them from HBM as in the whole model.

Weights are random blocks drawn from a pool that `_pool` encodes, the same
for every seed: a program loads its model once. The token ids (the prompt,
the earlier conversation, the token that decoding starts from), the sampler's
logits and its window come from the seed.
"""
import ctypes
import math
import os
import sys
import weakref

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "llama.rs_amd"))
import rlh  # noqa: E402

# layers and vocabulary of the slice of each shape
SLICES = {"0.6b": (28, 151936), "4b": (6, 25344), "8b": (4, 16896), "32b": (2, 4864)}
SHAPE_SPEC = {"0.6b": "qwen3-0.6b-q4km", "4b": "qwen3-4b-q4km", "8b": "qwen3-8b-q4km", "32b": "qwen3-32b-q4km"}


# ---- cases ------------------------------------------------------------------

def listed():
    """op prefill: `tokens` prompt tokens after `ctx` earlier ones, logits out.
    op decode: after `ctx` tokens, one step, then `tokens` greedy tokens, then
    the last one's logits. op sampled: the same loop with the device sampler.
    op sampler: softmax and one sampled token over `vocab` device logits."""
    cli = {"temperature": 0.7, "top_k": 40, "top_p": 0.95}
    return [
        # one token chosen from logits a program already holds on the device,
        # with the command line's sampling defaults; its probabilities beside it
        {"name": "sampler 151936", "op": "sampler", "vocab": 151936, **cli},
        # a short chat prompt and its reply on the smallest model
        {"name": "prefill 0.6b q8_0 48", "op": "prefill", "shape": "0.6b", "mix": "q8_0", "ctx": 0, "tokens": 48},
        {"name": "decode 0.6b q4km 48+32", "op": "decode", "shape": "0.6b", "mix": "q4km", "ctx": 48, "tokens": 32},
        # a sampled reply (command line defaults): one host round trip per token
        {"name": "sampled 0.6b q8_0 112+24", "op": "sampled", "shape": "0.6b", "mix": "q8_0", "ctx": 112,
         "tokens": 24, **cli},
        # a paragraph-sized prompt of odd length, and greedy decoding after it
        {"name": "prefill 4b q4km 237", "op": "prefill", "shape": "4b", "mix": "q4km", "ctx": 0, "tokens": 237},
        {"name": "decode 4b q4km 384+32", "op": "decode", "shape": "4b", "mix": "q4km", "ctx": 384, "tokens": 32},
        # the headline model: its 512-token prompt, and its decode window's middle
        {"name": "prefill 8b q4km 512", "op": "prefill", "shape": "8b", "mix": "q4km", "ctx": 0, "tokens": 512},
        {"name": "decode 8b q4km 768+32", "op": "decode", "shape": "8b", "mix": "q4km", "ctx": 768, "tokens": 32},
        # the next user turn of a conversation that is already in the cache
        {"name": "turn 8b q4km 700+61", "op": "prefill", "shape": "8b", "mix": "q4km", "ctx": 700, "tokens": 61},
        # the other common mix of block types (five-bit blocks multiply f32
        # activations in prefill): a prompt of odd length
        {"name": "prefill 4b q5km 131", "op": "prefill", "shape": "4b", "mix": "q5km", "ctx": 0, "tokens": 131},
        # the largest model on a long document: reading it, and answering
        {"name": "prefill 32b q4km 4096", "op": "prefill", "shape": "32b", "mix": "q4km", "ctx": 0, "tokens": 4096},
        {"name": "decode 32b q4km 4100+24", "op": "decode", "shape": "32b", "mix": "q4km", "ctx": 4100, "tokens": 24},
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Prompt lengths 2 to 4096 and contexts up to 4200 over their logarithm,
    every shape, the common block mixes and (for the small shapes) float
    weights, vocabularies 1000 to 200000 and the sampler's option sets."""
    op = rng.choice(["prefill", "prefill", "prefill", "decode", "decode", "sampled", "sampler"])
    options = rng.choice([{"temperature": 0.7, "top_k": 40, "top_p": 0.95},
                          {"temperature": 1.0, "top_k": 0, "top_p": 0.9},
                          {"temperature": 0.8, "top_k": 100, "top_p": 1.0},
                          {"temperature": 0.0, "top_k": 0, "top_p": 1.0}])
    if op == "sampler":
        return {"op": op, "vocab": _log_uniform(rng, 1000, 200000), **options}
    mix = rng.choice(["q4km", "q4km", "q4km", "q8_0", "q8_0", "q5km", "f16", "bf16"])
    shape = rng.choice(["0.6b", "4b", "8b", "32b"] if mix in ("q4km", "q8_0") else ["0.6b", "4b"])
    if op == "prefill":
        most = 4096 if mix in ("q4km", "q8_0") else 256
        tokens = _log_uniform(rng, 2, most if shape != "0.6b" else most // 4)
        ctx = rng.choice([0, 0, _log_uniform(rng, 16, 2048)])
        if shape == "32b":
            ctx = min(ctx, 4096 - tokens)
        return {"op": op, "shape": shape, "mix": mix, "ctx": ctx, "tokens": tokens}
    most = {"0.6b": 1024, "4b": 2048, "8b": 4200, "32b": 4200}[shape]
    case = {"op": op, "shape": shape, "mix": mix, "ctx": _log_uniform(rng, 16, most),
            "tokens": _log_uniform(rng, 4, 24)}
    return {**case, **options} if op == "sampled" else case


# ---- weights ----------------------------------------------------------------

def _scale_bytes(sc, mn):
    """The 12 bytes of eight 6-bit scales and mins of a Q4_K / Q5_K block."""
    out = np.zeros((len(sc), 12), np.uint8)
    out[:, 0:4] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    out[:, 4:8] = mn[:, :4] | ((mn[:, 4:] >> 4) << 6)
    out[:, 8:12] = (sc[:, 4:] & 15) | ((mn[:, 4:] & 15) << 4)
    return out


_POOL = 4096
_pools = {}


def _pool(ty):
    """_POOL runs of 256 N(0, 0.02) weights encoded in the block format of
    `ty`: (bytes of each run, the values they stand for in 64 bits)."""
    if ty in _pools:
        return _pools[ty]
    w = np.random.RandomState(1000 + ty).normal(0.0, 0.02, (_POOL, 256)).astype(np.float32)
    if ty == rlh.Q8_0:
        b = w.reshape(_POOL, 8, 32)
        d = (np.abs(b).max(2) / 127).astype(np.float16)
        q = np.clip(np.rint(b / d[:, :, None].astype(np.float64)), -127, 127).astype(np.int8)
        by = np.concatenate([d[:, :, None].view(np.uint8).reshape(_POOL, 8, 2), q.view(np.uint8)], 2)
        val = q * d[:, :, None].astype(np.float64)
    elif ty in (rlh.Q4_K, rlh.Q5_K):
        top = 15 if ty == rlh.Q4_K else 31
        b = w.reshape(_POOL, 8, 32).astype(np.float64)
        lo = np.maximum(-b.min(2), 0)
        step = (b.max(2) + lo) / top
        d = (step.max(1) / 63).astype(np.float16)
        dm = (lo.max(1) / 63).astype(np.float16)
        sc = np.clip(np.rint(step / d[:, None].astype(np.float64)), 1, 63).astype(np.uint8)
        mn = np.clip(np.rint(lo / dm[:, None].astype(np.float64)), 0, 63).astype(np.uint8)
        s, m = sc * d[:, None].astype(np.float64), mn * dm[:, None].astype(np.float64)
        q = np.clip(np.rint((b + m[:, :, None]) / s[:, :, None]), 0, top).astype(np.uint8)
        val = q * s[:, :, None] - m[:, :, None]
        lo4 = (q & 15).reshape(_POOL, 4, 2, 32)
        qs = (lo4[:, :, 0] | (lo4[:, :, 1] << 4)).reshape(_POOL, 128)
        parts = [d[:, None].view(np.uint8), dm[:, None].view(np.uint8), _scale_bytes(sc, mn)]
        if ty == rlh.Q5_K:
            parts.append(((q >> 4) << np.arange(8, dtype=np.uint8)[None, :, None]).sum(1).astype(np.uint8))
        by = np.concatenate(parts + [qs], 1)
    elif ty == rlh.Q6_K:
        b = w.reshape(_POOL, 16, 16).astype(np.float64)
        step = np.abs(b).max(2) / 31
        d = (step.max(1) / 127).astype(np.float16)
        sc = np.clip(np.rint(step / d[:, None].astype(np.float64)), 1, 127).astype(np.int8)
        s = sc * d[:, None].astype(np.float64)
        q = np.clip(np.rint(b / s[:, :, None]), -32, 31)
        val = q * s[:, :, None]
        u = (q + 32).astype(np.uint8).reshape(_POOL, 2, 4, 32)  # half, quarter, position
        ql = np.concatenate([(u[:, :, 0] & 15) | ((u[:, :, 2] & 15) << 4), (u[:, :, 1] & 15) | ((u[:, :, 3] & 15) << 4)], 2)
        qh = (u[:, :, 0] >> 4) | ((u[:, :, 1] >> 4) << 2) | ((u[:, :, 2] >> 4) << 4) | ((u[:, :, 3] >> 4) << 6)
        by = np.concatenate([ql.reshape(_POOL, 128), qh.reshape(_POOL, 64), sc.view(np.uint8), d[:, None].view(np.uint8)], 1)
    elif ty == rlh.F16:
        h = w.astype(np.float16)
        by, val = h.view(np.uint8), h.astype(np.float64)
    elif ty == rlh.BF16:
        bits = (w.view(np.uint32) + 0x8000) >> 16
        by, val = bits.astype(np.uint16).view(np.uint8), (bits << 16).astype(np.uint32).view(np.float32).astype(np.float64)
    else:
        raise ValueError(f"no encoder for type {ty}")
    _pools[ty] = np.ascontiguousarray(by.reshape(_POOL, -1)), np.ascontiguousarray(val.reshape(_POOL, 256))
    return _pools[ty]


def _mix(mix, tied):
    """Tensor types of a block mix: the _M mixes keep attn_v, ffn_down and the
    logits matrix in Q6_K; the others hold one type."""
    base = {"q4km": rlh.Q4_K, "q5km": rlh.Q5_K, "q8_0": rlh.Q8_0, "f16": rlh.F16, "bf16": rlh.BF16}[mix]
    six = rlh.Q6_K if mix in ("q4km", "q5km") else base
    t = {k: base for k in (rlh.T_ATTN_Q, rlh.T_ATTN_K, rlh.T_ATTN_OUTPUT, rlh.T_FFN_GATE, rlh.T_FFN_UP)}
    t.update({rlh.T_ATTN_V: six, rlh.T_FFN_DOWN: six, rlh.T_TOKEN_EMBD: six if tied else base, rlh.T_OUTPUT: six})
    return t


def _spec(case):
    s = rlh.SPECS[SHAPE_SPEC[case["shape"]]]
    layers, vocab = SLICES[case["shape"]]
    return rlh.ModelSpec(f"{case['shape']}-{case['mix']}", layers, s.n_embd, s.n_ff, s.n_head, s.n_head_kv, vocab,
                         s.tied, _mix(case["mix"], s.tied), n_ctx=8192)


def _runs(kind, layer, rows, cols):
    """The pool runs that make up a matrix, in row order."""
    r = np.random.RandomState((kind * 131 + layer) & 0x7FFFFFFF)
    return r.randint(0, _POOL, rows * cols // 256)


def _matrices(spec):
    """(kind, layer, rows, cols) of every matrix."""
    yield rlh.T_TOKEN_EMBD, 0, spec.vocab, spec.n_embd
    if not spec.tied:
        yield rlh.T_OUTPUT, 0, spec.vocab, spec.n_embd
    for layer in range(spec.n_layer):
        for kind, rows, cols in spec.shapes():
            yield kind, layer, rows, cols


def _vector(kind, layer, n):
    return np.random.RandomState((kind * 131 + layer + 7) & 0x7FFFFFFF).normal(1.0, 0.02, n).astype(np.float32)


def _vectors(spec):
    yield rlh.T_OUTPUT_NORM, 0, spec.n_embd
    for layer in range(spec.n_layer):
        yield rlh.T_ATTN_NORM, layer, spec.n_embd
        yield rlh.T_FFN_NORM, layer, spec.n_embd
        yield rlh.T_ATTN_Q_NORM, layer, spec.head_dim
        yield rlh.T_ATTN_K_NORM, layer, spec.head_dim


class _Loaded:
    """A model on the device, released with the last program state that uses it."""

    def __init__(self, spec):
        self.spec = spec

        def tensors():
            for kind, layer, rows, cols in _matrices(spec):
                yield kind, layer, spec.types[kind], cols, rows, _pool(spec.types[kind])[0][_runs(kind, layer, rows, cols)]
            for kind, layer, n in _vectors(spec):
                yield kind, layer, rlh.F32, n, 1, _vector(kind, layer, n).view(np.uint8)

        self.model = rlh.Model(spec, tensors())
        weakref.finalize(self, self.model.close)


_latest = {}


def _load(spec):
    if spec.name not in _latest:
        _latest.clear()
        _latest[spec.name] = _Loaded(spec)
    return _latest[spec.name]


# ---- program states ---------------------------------------------------------

class _Conversation:
    """A cache that already holds `ctx` tokens, and what comes next."""

    def __init__(self, case, seed):
        rng = np.random.RandomState(seed & 0x7FFFFFFF)
        self.case, self.ctx = case, case["ctx"]
        self.loaded = _load(_spec(case))
        room = self.ctx + case["tokens"] + 8
        self.cache = self.loaded.model.new_cache(room)
        weakref.finalize(self, self.cache.close)
        self.earlier, self.ids = _ids(case, rng)
        if self.ctx:
            self.cache.forward_into(self.earlier, 0, copy=False)
        self.one = np.empty(1, np.uint32)
        if case["op"] == "sampled":
            self.params = _params(case)


def _ids(case, rng):
    """The earlier tokens and the new ones (one for the decode loops)."""
    vocab = SLICES[case["shape"]][1]
    n = case["tokens"] if case["op"] == "prefill" else 1
    ids = rng.randint(0, vocab, case["ctx"] + n).astype(np.uint32)
    return ids[: case["ctx"]], ids[case["ctx"]:]


def _params(case):
    return rlh.sampling_params(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"])


class _Choice:
    """Device logits shaped like a language model's (a wide bulk, a few tall
    tokens), a sampler and the window of recent tokens."""

    def __init__(self, case, seed):
        self.case = case
        self.logits = _logits(case, seed).to("cuda", torch.float32)
        self.recent = np.random.RandomState((seed + 1) & 0x7FFFFFFF).randint(0, case["vocab"], 64).astype(np.uint32)
        self.sampler = rlh.DeviceSampler(seed, case["vocab"])
        weakref.finalize(self, self.sampler.close)
        self.seeded = self.sampler.state.value
        self.params = _params(case)


def _logits(case, seed):
    rng = np.random.RandomState(seed & 0x7FFFFFFF)
    x = rng.normal(0.0, 2.0, case["vocab"])
    tall = rng.randint(0, case["vocab"], 30)
    x[tall] += rng.exponential(4.0, 30) + 6.0
    return torch.from_numpy(x.astype(np.float32))


def prepare(case, seed):
    return _Choice(case, seed) if case["op"] == "sampler" else _Conversation(case, seed)


def run(state):
    case = state.case
    if case["op"] == "sampler":
        n, ds = case["vocab"], state.sampler
        ds.state.value = state.seeded  # the reply's own seed
        probs = state.logits.clone()
        ds.softmax(probs.data_ptr(), n)
        token = ds.sample(state.logits.data_ptr(), n, state.params, state.recent)
        return {"probs": probs, "token": token}
    cache, ctx = state.cache, state.ctx
    if case["op"] == "prefill":
        return {"logits": cache.forward_into(state.ids, ctx)}
    first = cache.forward_into(state.ids, ctx)
    if case["op"] == "decode":
        tokens = cache.generate_greedy(cache.greedy_next(), case["tokens"])
        return {"first": first, "tokens": tokens, "last": cache.forward_into(tokens[-1:], cache.len)}
    rng_state = ctypes.c_uint64(rlh.load().rlh_sampler_init(state.params.seed))
    recent = np.empty(ctx + 1 + case["tokens"], np.uint32)
    recent[:ctx] = state.earlier
    recent[ctx] = state.ids[0]
    last = None
    for i in range(ctx + 1, ctx + 1 + case["tokens"]):
        recent[i] = state.one[0] = cache.sample_next(state.params, recent[:i], rng_state)
        last = cache.forward_into(state.one, i, copy=i == ctx + case["tokens"])
    return {"first": first, "tokens": recent[ctx + 1:], "last": last}


# ---- what a pass cannot do without ------------------------------------------

def work(case):
    if case["op"] == "sampler":
        return {"bytes": 2 * 4 * case["vocab"], "flops": 20 * case["vocab"]}  # logits in, probabilities out
    spec = _spec(case)
    qd, kvd = spec.n_head * spec.head_dim, spec.n_head_kv * spec.head_dim
    layer_values = sum(r * c for _, r, c in spec.shapes())
    head_values = spec.vocab * spec.n_embd
    weights = spec.weight_bytes_per_token()
    ctx, n = case["ctx"], case["tokens"]
    if case["op"] == "prefill":
        pairs = n * ctx + n * (n + 1) // 2  # causal (token, position) pairs
        flops = spec.n_layer * (2 * layer_values * n + 4 * qd * pairs) + 2 * head_values
        kv = 4 * 2 * kvd * spec.n_layer * (ctx + n)  # earlier rows in, new rows out
        return {"bytes": weights + kv + 4 * spec.vocab, "flops": flops}
    steps = n + (2 if case["op"] == "decode" else 1)
    seen = sum(ctx + 1 + i for i in range(steps))
    flops = steps * 2 * (spec.n_layer * layer_values + head_values) + spec.n_layer * 4 * qd * seen
    return {"bytes": steps * weights + 4 * 2 * kvd * spec.n_layer * (seen + steps) + 8 * spec.vocab, "flops": flops}


def tolerance(case):
    """The path promises the reference's bits (include/rlh.h): every sum runs
    in the reference's order, so another correct implementation shows none."""
    return "exact"


# ---- the same in 64 bits ----------------------------------------------------

def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _forward64(spec, ids):
    """Logits of the last of `ids` in float64 (no activation is quantized)."""
    dev = "cuda"
    pools = {t: torch.from_numpy(_pool(t)[1]).to(dev) for t in set(spec.types.values())}

    def mat(kind, layer, rows, cols):
        return pools[spec.types[kind]][torch.from_numpy(_runs(kind, layer, rows, cols)).to(dev)].view(rows, cols)

    def vec(kind, layer, n):
        return torch.from_numpy(_vector(kind, layer, n)).to(dev, torch.float64)

    n, hd, heads, kvh = len(ids), spec.head_dim, spec.n_head, spec.n_head_kv
    at = torch.from_numpy(ids.astype(np.int64)).to(dev)
    runs = torch.from_numpy(_runs(rlh.T_TOKEN_EMBD, 0, spec.vocab, spec.n_embd)).to(dev).view(spec.vocab, -1)
    x = pools[spec.types[rlh.T_TOKEN_EMBD]][runs[at]].view(n, spec.n_embd)
    freq = spec.rope_theta ** (-2.0 * torch.arange(hd // 2, device=dev, dtype=torch.float64) / hd)
    angle = torch.arange(n, device=dev, dtype=torch.float64)[:, None] * freq
    cos, sin = torch.cos(angle)[:, None], torch.sin(angle)[:, None]

    def rope(t):
        a, b = t[..., : hd // 2], t[..., hd // 2:]
        return torch.cat([a * cos - b * sin, a * sin + b * cos], -1)

    for layer in range(spec.n_layer):
        w = {k: (r, c) for k, r, c in spec.shapes()}
        h = _rms(x, vec(rlh.T_ATTN_NORM, layer, spec.n_embd), spec.rms_eps)
        q, k, v = (h @ mat(kind, layer, *w[kind]).T for kind in (rlh.T_ATTN_Q, rlh.T_ATTN_K, rlh.T_ATTN_V))
        q = rope(_rms(q.view(n, heads, hd), vec(rlh.T_ATTN_Q_NORM, layer, hd), spec.rms_eps))
        k = rope(_rms(k.view(n, kvh, hd), vec(rlh.T_ATTN_K_NORM, layer, hd), spec.rms_eps))
        v = v.view(n, kvh, hd)
        out = torch.empty_like(q)
        hidden = torch.ones(n, n, device=dev, dtype=torch.bool).triu(1)
        for head in range(heads):
            g = head // (heads // kvh)
            p = (q[:, head] @ k[:, g].T / math.sqrt(hd)).masked_fill_(hidden, float("-inf"))
            out[:, head] = torch.softmax(p, -1) @ v[:, g]
        x = x + out.reshape(n, -1) @ mat(rlh.T_ATTN_OUTPUT, layer, *w[rlh.T_ATTN_OUTPUT]).T
        h = _rms(x, vec(rlh.T_FFN_NORM, layer, spec.n_embd), spec.rms_eps)
        gate, up = (h @ mat(kind, layer, *w[kind]).T for kind in (rlh.T_FFN_GATE, rlh.T_FFN_UP))
        x = x + (torch.nn.functional.silu(gate) * up) @ mat(rlh.T_FFN_DOWN, layer, *w[rlh.T_FFN_DOWN]).T
    h = _rms(x[-1:], vec(rlh.T_OUTPUT_NORM, 0, spec.n_embd), spec.rms_eps)
    kind = rlh.T_TOKEN_EMBD if spec.tied else rlh.T_OUTPUT
    return (h @ mat(kind, 0, spec.vocab, spec.n_embd).T).view(-1).cpu().numpy()


def exact(case, seed):
    if case["op"] == "sampler":
        return {"probs": torch.softmax(_logits(case, seed).double(), 0).numpy(), "token": None}
    earlier, ids = _ids(case, np.random.RandomState(seed & 0x7FFFFFFF))
    logits = _forward64(_spec(case), np.concatenate([earlier, ids]))
    # later steps follow the tokens that the path itself chose
    return {"logits": logits} if case["op"] == "prefill" else {"first": logits, "tokens": None, "last": None}
