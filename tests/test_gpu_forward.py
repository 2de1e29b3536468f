"""End-to-end parity of the device token loop against the CPU oracle.

Reference modes: decode = the AVX2 integer path (ops.rs:93-128); prefill =
RUST_LLAMA_BATCH_INT=1 (ops.rs:192-236). Required bars:
per-layer hidden states within 1e-3 relative L2, logits within 2e-3,
identical greedy tokens. The device path is built to match bit for bit, and
these tests assert that stronger property (the L2 numbers are printed).
"""
import ctypes

import numpy as np
import pytest

import oracle
import rlh
from helpers import bits, rel_l2

pytestmark = pytest.mark.gpu

_models = {}


def _get(name, seed=1234):
    key = (name, seed)
    if key not in _models:
        spec = rlh.SPECS[name]
        tensors = rlh.synth_model(spec, seed)
        _models[key] = (spec, tensors, rlh.Model(spec, tensors), oracle.OracleModel(spec, tensors))
    return _models[key]


def _greedy_ref(oc, prompt, n_gen):
    """main.rs:500-516 loop on the oracle: argmax after every step."""
    lib = oracle.load()
    logits = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
    toks = [lib.orc_argmax(logits.ctypes.data, len(logits))]
    per_step = []
    for i in range(n_gen):
        lg = oc.forward_into(np.array([toks[-1]], np.uint32), len(prompt) + i, oracle.MODE_DEFAULT)
        per_step.append(lg)
        toks.append(lib.orc_argmax(lg.ctypes.data, len(lg)))
    return logits, toks, per_step


@pytest.mark.parametrize("name", ["tiny-q4km", "tiny-q8_0", "tiny-q4_0", "tiny-q4km-untied", "small-q4km",
                                  "tiny-smallvocab"])
def test_prefill_and_decode_bit_exact(name):
    print(f"forward parity {name}", flush=True)
    spec, tensors, m, om = _get(name)
    n_prompt, n_gen = 12, 10
    prompt = rlh.synth_tokens(99, n_prompt, spec.vocab)
    c = m.new_cache(64)
    oc = om.new_cache(64)
    c.set_debug(True)
    oc.enable_dump(n_prompt)
    logits = c.forward_into(prompt, 0)
    ref_logits = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
    print(f"  prefill logits rel L2 {rel_l2(logits, ref_logits):.3e}")
    for l in range(spec.n_layer):
        h = c.layer_hidden(l, n_prompt)
        r = oc.hidden(l, n_prompt)
        assert rel_l2(h, r) <= 1e-3
        assert np.array_equal(bits(h), bits(r)), f"layer {l} hidden differs"
    for l in range(spec.n_layer):
        for which in (0, 1):
            assert np.array_equal(bits(c.read_kv(l, which, n_prompt)), bits(oc.read_kv(l, which, n_prompt)))
    assert rel_l2(logits, ref_logits) <= 2e-3
    assert np.array_equal(bits(logits), bits(ref_logits))
    assert c.len == n_prompt and oc.len == n_prompt

    # decode: one step at a time through forward_into (n == 1 -> forward_one)
    lib = oracle.load()
    tok = lib.orc_argmax(ref_logits.ctypes.data, len(ref_logits))
    assert c.greedy_next() == tok
    for i in range(n_gen):
        lg = c.forward_into(np.array([tok], np.uint32), n_prompt + i)
        rg = oc.forward_into(np.array([tok], np.uint32), n_prompt + i, oracle.MODE_DEFAULT)
        assert np.array_equal(bits(lg), bits(rg)), f"decode step {i} logits differ (rel {rel_l2(lg, rg):.2e})"
        tok = lib.orc_argmax(rg.ctypes.data, len(rg))
        assert c.greedy_next() == tok
    c.close()
    oc.close()


@pytest.mark.parametrize("name", ["tiny-q4km", "small-q4km"])
def test_decode_ring_plans_bit_exact(name, monkeypatch):
    """Decode with ring plans forced (RLH_MV_RING=1 when the cache, and with
    it the captured step, is made): ffn_down's row chains are added round by
    round while the producers stream the next tiles."""
    print(f"ring decode parity {name}", flush=True)
    monkeypatch.setenv("RLH_MV_RING", "1")
    spec, tensors, m, om = _get(name)
    n_prompt = 8
    prompt = rlh.synth_tokens(98, n_prompt, spec.vocab)
    c = m.new_cache(64)
    oc = om.new_cache(64)
    c.forward_into(prompt, 0)
    ref = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
    lib = oracle.load()
    tok = lib.orc_argmax(ref.ctypes.data, len(ref))
    for i in range(6):
        lg = c.forward_into(np.array([tok], np.uint32), n_prompt + i)
        rg = oc.forward_into(np.array([tok], np.uint32), n_prompt + i, oracle.MODE_DEFAULT)
        assert np.array_equal(bits(lg), bits(rg)), f"decode step {i} logits differ (rel {rel_l2(lg, rg):.2e})"
        tok = lib.orc_argmax(rg.ctypes.data, len(rg))
    c.close()
    oc.close()


@pytest.mark.parametrize("max_ctx,n_prompt", [(64, 40), (6000, 40), (1600, 700), (4400, 4100)])
def test_decode_attention_paths(max_ctx, n_prompt):
    """Decode attention with 8 query heads per KV head (the 32B grouping):
    the softmax kernel and the PV kernel that streams p and V through an
    8-slot LDS ring. 40 positions fit one 64-position chunk; 700 and 4100
    positions wrap the ring many times, hand chunks two ahead from the
    producers to the ordered adds and end on a clamped ragged tail (4100 is
    the 32B workload's context). The 700- and 4100-token prompts also run
    the prefill in several 512-token chunks with 8 heads per KV head.
    Logits bit-exact in every step."""
    print(f"decode attention g8 max_ctx {max_ctx} prompt {n_prompt}", flush=True)
    spec, tensors, m, om = _get("tiny-g8-q4km")
    prompt = rlh.synth_tokens(77, n_prompt, spec.vocab)
    c = m.new_cache(max_ctx)
    oc = om.new_cache(max_ctx)
    lg = c.forward_into(prompt, 0)
    rg = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
    assert np.array_equal(bits(lg), bits(rg))
    lib = oracle.load()
    tok = lib.orc_argmax(rg.ctypes.data, len(rg))
    for i in range(6):
        lg = c.forward_into(np.array([tok], np.uint32), len(prompt) + i)
        rg = oc.forward_into(np.array([tok], np.uint32), len(prompt) + i, oracle.MODE_DEFAULT)
        assert np.array_equal(bits(lg), bits(rg)), f"decode step {i} logits differ (rel {rel_l2(lg, rg):.2e})"
        tok = lib.orc_argmax(rg.ctypes.data, len(rg))
    c.close()
    oc.close()


@pytest.mark.parametrize("max_ctx,n_prompt", [(300, 62), (1200, 250), (1200, 600), (1200, 1100), (4096, 130),
                                              (8000, 70)])
def test_decode_attention_g4_paths(max_ctx, n_prompt):
    """Decode attention with 4 query heads per KV head. Caches up to about
    1200 positions take the kernel that keeps its V slices in LDS (the
    products run two 64-position chunks ahead of the ordered adds, the
    exponentials 256-position chunks ahead of the softmax sums: the steps
    cross chunk boundaries, end on ragged chunks and, at 600 and 1100
    positions, use three and five exponential chunks), 4096 and 8000
    positions the softmax kernel and the PV kernel that streams p and V
    through LDS rings. Logits bit-exact in every step."""
    print(f"decode attention g4 max_ctx {max_ctx} prompt {n_prompt}", flush=True)
    spec, tensors, m, om = _get("tiny-g4-q4km")
    prompt = rlh.synth_tokens(55, n_prompt, spec.vocab)
    c = m.new_cache(max_ctx)
    oc = om.new_cache(max_ctx)
    lg = c.forward_into(prompt, 0)
    rg = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
    assert np.array_equal(bits(lg), bits(rg))
    lib = oracle.load()
    tok = lib.orc_argmax(rg.ctypes.data, len(rg))
    for i in range(6):
        lg = c.forward_into(np.array([tok], np.uint32), n_prompt + i)
        rg = oc.forward_into(np.array([tok], np.uint32), n_prompt + i, oracle.MODE_DEFAULT)
        assert np.array_equal(bits(lg), bits(rg)), f"decode step {i} logits differ (rel {rel_l2(lg, rg):.2e})"
        tok = lib.orc_argmax(rg.ctypes.data, len(rg))
    c.close()
    oc.close()


@pytest.mark.parametrize("name,max_ctx,n_prompt", [("tiny-g1-q4km", 64, 30), ("tiny-g1-q4km", 2000, 200),
                                                   ("tiny-g2-q4km", 64, 30), ("tiny-g2-q4km", 2000, 130),
                                                   ("tiny-g3-q4km", 64, 30), ("tiny-g3-q4km", 1200, 1100),
                                                   ("tiny-g3-q4km", 3000, 1300),
                                                   ("tiny-g5-q4km", 64, 30), ("tiny-g5-q4km", 3000, 1300),
                                                   ("tiny-g6-q4km", 64, 30), ("tiny-g6-q4km", 3000, 700),
                                                   ("tiny-g7-q4km", 64, 30), ("tiny-g7-q4km", 3000, 1300),
                                                   ("tiny-wide-q4km", 64, 20), ("tiny-wide-q4km", 3000, 100)])
def test_decode_attention_groupings(name, max_ctx, n_prompt):
    """Decode attention with 1, 2 and 3 query heads per KV head (the
    resident-V kernel for short caches, the softmax + streamed-ring PV
    kernels past ~1200-1500 positions), with 5, 6 and 7 (groups that do not
    divide the prefill kernels' 64 (token, head) pairs or the decode
    kernels' 64-lane chains: ragged pair tiles, 8-wide ring slices) and with
    13312-wide attention rows, where attn_output reads the Q8 blocks the
    attention kernels write (the fused streamed kernel for 64 positions, the
    softmax kernel + the streamed PV kernel for 3000). Prompts of 700-1300
    tokens run the prefill in two or three 512-token chunks, and decode rows
    of 1024 positions or more take the softmax sum by monosum run pairs.
    Logits bit-exact."""
    print(f"decode attention {name} max_ctx {max_ctx} prompt {n_prompt}", flush=True)
    spec, tensors, m, om = _get(name)
    prompt = rlh.synth_tokens(66, n_prompt, spec.vocab)
    c = m.new_cache(max_ctx)
    oc = om.new_cache(max_ctx)
    lg = c.forward_into(prompt, 0)
    rg = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
    assert np.array_equal(bits(lg), bits(rg))
    lib = oracle.load()
    tok = lib.orc_argmax(rg.ctypes.data, len(rg))
    for i in range(5):
        lg = c.forward_into(np.array([tok], np.uint32), n_prompt + i)
        rg = oc.forward_into(np.array([tok], np.uint32), n_prompt + i, oracle.MODE_DEFAULT)
        assert np.array_equal(bits(lg), bits(rg)), f"decode step {i} logits differ (rel {rel_l2(lg, rg):.2e})"
        tok = lib.orc_argmax(rg.ctypes.data, len(rg))
    c.close()
    oc.close()


@pytest.mark.parametrize("name", ["tiny-q4km", "small-q4km"])
def test_generate_greedy_matches_cpu_tokens(name):
    spec, tensors, m, om = _get(name)
    prompt = rlh.synth_tokens(5, 9, spec.vocab)
    n_gen = 24
    c = m.new_cache(64)
    oc = om.new_cache(64)
    logits = c.forward_into(prompt, 0)
    first = c.greedy_next()
    toks = c.generate_greedy(first, n_gen)
    _, ref_toks, _ = _greedy_ref(oc, prompt, n_gen)
    assert list(map(int, toks)) == ref_toks
    assert c.len == len(prompt) + n_gen
    c.close()
    oc.close()


@pytest.mark.parametrize("name", ["tiny-q4km", "small-q4km"])
def test_generate_sampled_matches_cpu(name):
    """Model::generate with temperature / top-k / top-p / repetition penalty
    (the SamplingParams defaults, sampler.rs:15-26): same tokens as the oracle,
    and generation stops at EOS."""
    print(f"sampled generate {name}", flush=True)
    spec, tensors, m, om = _get(name)
    prompt = rlh.synth_tokens(31, 10, spec.vocab)
    c = m.new_cache(64)
    oc = om.new_cache(64)
    params = rlh.sampling_params(seed=0xC0FFEE)
    oparams = oracle.SamplingParams(0.7, 40, 0.95, 1.1, 64, 0xC0FFEE)
    eos = spec.vocab + 7  # never sampled: full length
    toks = c.generate(prompt, 24, params, eos)
    ref = oc.generate(prompt, 24, oparams, eos)
    assert list(map(int, toks)) == list(map(int, ref))
    assert len(toks) == 24 and c.len == len(prompt) + 24
    eos = int(toks[5])
    first = int(np.flatnonzero(toks == eos)[0])
    toks2 = c.generate(prompt, 24, params, eos)
    assert list(map(int, toks2)) == list(map(int, toks[:first]))
    c.close()
    oc.close()


def test_forward_errors():
    spec, tensors, m, om = _get("tiny-q4km")
    c = m.new_cache(16)
    with pytest.raises(rlh.RlhError) as e:
        c.forward_into(np.array([spec.vocab], np.uint32), 0)
    assert e.value.code == rlh.RLH_EINVAL
    with pytest.raises(rlh.RlhError) as e:
        c.forward_into(np.array([1], np.uint32), 16)
    assert e.value.code == rlh.RLH_ECTX
    # batch truncation to max_ctx - start_pos (model.rs:392)
    c.forward_into(np.arange(20, dtype=np.uint32), 0)
    assert c.len == 16
    with pytest.raises(rlh.RlhError) as e:
        c.generate_greedy(1, 4)
    assert e.value.code == rlh.RLH_ECTX
    c.reset()
    assert c.len == 0
    c.close()


def test_cache_max_ctx_clamped_to_n_ctx():
    spec, tensors, m, om = _get("tiny-q4km")
    c = m.new_cache(10 ** 6)
    assert c.max_ctx == spec.n_ctx
    c.close()


def test_long_prefill_chunks_and_continuation():
    """A prompt longer than one prefill chunk (512 tokens), then a second
    batch continuing at start_pos > 0: logits and every K/V row bit-exact
    against the oracle's single forward_batch calls."""
    spec, tensors, m, om = _get("small-q4km")
    prompt = rlh.synth_tokens(123, 600, spec.vocab)
    more = rlh.synth_tokens(321, 30, spec.vocab)
    c = m.new_cache(700)
    oc = om.new_cache(700)
    lg = c.forward_into(prompt, 0)
    rg = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
    print(f"  600-token prefill logits rel L2 {rel_l2(lg, rg):.3e}", flush=True)
    assert np.array_equal(bits(lg), bits(rg))
    lg2 = c.forward_into(more, 600)
    rg2 = oc.forward_into(more, 600, oracle.MODE_BATCH_INT)
    assert np.array_equal(bits(lg2), bits(rg2))
    for l in (0, spec.n_layer - 1):
        for which in (0, 1):
            assert np.array_equal(bits(c.read_kv(l, which, 630)), bits(oc.read_kv(l, which, 630)))
    assert c.len == 630
    c.close()
    oc.close()


def test_prefill_softmax_row_kernels():
    """Prefill rows of up to 4988 positions take the softmax kernel with one
    wave per row (16, 8 or 4 rows per block by row length), longer rows the
    kernel with one block per row: a 5200-token prompt in 512-token chunks
    uses the first for the chunks that end at or below position 4988
    (among them the chunk ending at 4608, whose 4 rows exceed 64 KB of LDS)
    and the second for the last two chunks (ending at 5120 and 5200). Logits and the last layer's K/V rows
    bit-exact against the oracle."""
    spec, tensors, m, om = _get("tiny-g4-q4km")
    prompt = rlh.synth_tokens(77, 5200, spec.vocab)
    c = m.new_cache(5300)
    oc = om.new_cache(5300)
    lg = c.forward_into(prompt, 0)
    rg = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
    assert np.array_equal(bits(lg), bits(rg)), f"logits differ (rel {rel_l2(lg, rg):.2e})"
    for which in (0, 1):
        l = spec.n_layer - 1
        assert np.array_equal(bits(c.read_kv(l, which, 5200)), bits(oc.read_kv(l, which, 5200)))
    c.close()
    oc.close()


def _chunks(start, n):
    return [(start + c, min(512, n - c)) for c in range(0, n, 512)]


def _score_tiles(spec, pos, n):
    """Position tiles per block of the prefill scores kernel for a chunk of n
    tokens at pos: the most of 8, 4, 2, 1 that leave 512 blocks with work."""
    per = 64 // (spec.n_head // spec.n_head_kv)
    for tiles in (8, 4, 2):
        blocks = sum((pos + min(n, y + per) - 1) // 32 // tiles + 1 for y in range(0, n, per))
        if blocks * spec.n_head_kv >= 512:
            return tiles
    return 1


def _pv_waves(spec, n):
    """Waves per block of the prefill PV kernel."""
    per = 16 // (spec.n_head // spec.n_head_kv)
    return 8 if spec.n_head_kv * -(-n // per) >= 1024 else 4


def _close_all(*objs):
    for o in objs:
        o.close()


def _same(got, ref):
    nan = np.isnan(ref)
    return np.array_equal(np.isnan(got), nan) and np.array_equal(bits(got[~nan]), bits(ref[~nan]))


def _check_prefill(spec, tensors, tokens, parts):
    """Prefills the parts one after the other on the device and on the oracle:
    logits after each and every layer's K/V rows bit for bit, NaN exactly
    where the oracle has NaN. Returns the oracle's K/V rows [layer][k, v] and
    its last logits."""
    m, om = rlh.Model(spec, tensors), oracle.OracleModel(spec, tensors)
    c, oc = m.new_cache(len(tokens) + 8), om.new_cache(len(tokens) + 8)
    try:
        at = 0
        for n in parts:
            lg = c.forward_into(tokens[at:at + n], at)
            with np.errstate(all="ignore"):
                rg = oc.forward_into(tokens[at:at + n], at, oracle.MODE_BATCH_INT)
            assert _same(lg, rg), f"logits after {at} + {n} tokens differ"
            at += n
        rows = []
        for l in range(spec.n_layer):
            rows.append([oc.read_kv(l, which, at) for which in (0, 1)])
            for which in (0, 1):
                assert _same(c.read_kv(l, which, at), rows[l][which]), f"layer {l} {'kv'[which]} rows differ"
        return rows, rg
    finally:
        _close_all(c, oc, m, om)


# Qwen3-14B's 40 / 8 heads: 5 per KV head leave one of 16 combinations of a
# block empty, and the last block of 509 or 1021 tokens most of them
_G5_WIDE = rlh.ModelSpec("g5-wide", 2, 256, 512, 40, 8, 1000, True, rlh._q4km(True, rlh.Q4_K, None), n_ctx=4096)


@pytest.mark.parametrize("spec,parts,tiles,waves", [
    (rlh.SPECS["tiny-g4-q4km"], [4300], {1, 2, 4, 8}, {4}),
    (rlh.SPECS["small-q4km"], [600, 30], {1, 2}, {4}),
    (_G5_WIDE, [509, 70], {1, 8}, {4, 8}),
    (_G5_WIDE, [1021], {8}, {8}),
], ids=["g4-4300", "small-600-30", "g5-509-70", "g5-1021"])
def test_prefill_scores_kernels(spec, parts, tiles, waves):
    """The prefill scores kernel with every number of position tiles per block
    and the PV kernel with both widths, as the chunk lengths and contexts
    select them (restated above): a 4300-token prompt (9 chunks of up to 512
    tokens, 4 query heads per KV head), a prompt continued at an odd
    position, and blocks whose combinations are partly empty. Logits and all
    K/V rows bit-exact against the oracle."""
    chunks, at = [], 0
    for n in parts:
        chunks += _chunks(at, n)
        at += n
    assert {_score_tiles(spec, *c) for c in chunks} == tiles
    assert {_pv_waves(spec, n) for _, n in chunks} == waves
    print(f"prefill scores {spec.name} {parts}", flush=True)
    _check_prefill(spec, rlh.synth_model(spec, 1234), rlh.synth_tokens(91, sum(parts), spec.vocab), parts)


def test_nan_logits_argmax_semantics():
    """NaN logits: every 8th row of the untied output matrix has a NaN Q6_K
    scale, so every logits block starts with a NaN row and logits[0] is NaN.
    The device greedy argmax follows main.rs:453-463 (NaN never wins) in the
    standalone argmax and in the fused greedy loop, and rlh_sample_next's
    greedy fast path follows sampler.rs:62-70 (index 0 kept when logits[0]
    is NaN), both as the oracle."""
    spec = rlh.SPECS["tiny-q4km-untied"]
    tensors = rlh.synth_model(spec, 4321)
    for kind, layer, ty, cols, rows, buf in tensors:
        if kind == rlh.T_OUTPUT:
            assert ty == rlh.Q6_K
            rb = rlh.row_bytes(ty, cols)
            for r in range(0, rows, 8):
                buf[r * rb + 208] = 0x00  # f16 NaN 0x7e00 in d of the first super-block
                buf[r * rb + 209] = 0x7E
    m = rlh.Model(spec, tensors)
    om = oracle.OracleModel(spec, tensors)
    lib = oracle.load()
    prompt = rlh.synth_tokens(8, 9, spec.vocab)
    c = m.new_cache(64)
    oc = om.new_cache(64)
    try:
        lg = c.forward_into(prompt, 0)
        rg = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
        nan = np.isnan(rg)
        assert nan[0] and nan.sum() == spec.vocab // 8
        assert np.array_equal(np.isnan(lg), nan)
        assert np.array_equal(bits(lg[~nan]), bits(rg[~nan]))
        tok = c.greedy_next()
        assert tok == lib.orc_argmax(rg.ctypes.data, len(rg)) and tok % 8 != 0
        greedy = rlh.sampling_params(temperature=0.0, repetition_penalty=1.0)
        ogreedy = oracle.SamplingParams(0.0, 40, 0.95, 1.0, 64, 1)
        s = lib.orc_sampler_create(1)
        assert c.sample_next(greedy, prompt, ctypes.c_uint64(1)) == 0
        assert lib.orc_sampler_sample(s, rg.ctypes.data, len(rg), ogreedy, prompt.ctypes.data, len(prompt)) == 0
        lib.orc_sampler_destroy(s)
        toks = c.generate_greedy(tok, 6)
        ref = [tok]
        for i in range(6):
            r = oc.forward_into(np.array([ref[-1]], np.uint32), len(prompt) + i, oracle.MODE_DEFAULT)
            ref.append(lib.orc_argmax(r.ctypes.data, len(r)))
        assert list(map(int, toks)) == ref
    finally:
        c.close()
        oc.close()
        m.close()
        om.close()


def test_qwen2_biases_bit_exact():
    """q/k/v biases (Qwen2, model.rs:444-464 prefill and 626-640 decode): added
    after the products, before QK-norm and RoPE; prefill and decode logits
    bit-exact against the oracle."""
    spec = rlh.SPECS["tiny-q4km"]
    tensors = rlh.synth_model(spec, 606)
    lib = rlh.load()
    qd, kvd = spec.n_head * spec.head_dim, spec.n_head_kv * spec.head_dim
    for layer in range(spec.n_layer):
        for kind, n in ((rlh.T_ATTN_Q_BIAS, qd), (rlh.T_ATTN_K_BIAS, kvd), (rlh.T_ATTN_V_BIAS, kvd)):
            v = np.empty(n, np.float32)
            lib.rlh_synth_normal(606, rlh.tensor_id(kind, layer), 0, n, 0.0, 0.5, v.ctypes.data)
            tensors.append((kind, layer, rlh.F32, n, 1, v.view(np.uint8)))
    m = rlh.Model(spec, tensors)
    om = oracle.OracleModel(spec, tensors)
    olib = oracle.load()
    prompt = rlh.synth_tokens(607, 13, spec.vocab)
    c = m.new_cache(32)
    oc = om.new_cache(32)
    try:
        lg = c.forward_into(prompt, 0)
        rg = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
        assert np.array_equal(bits(lg), bits(rg))
        # without the biases the logits differ (the biases are applied)
        m0 = rlh.Model(spec, [t for t in tensors if t[0] < rlh.T_ATTN_Q_BIAS])
        c0 = m0.new_cache(32)
        assert not np.array_equal(bits(c0.forward_into(prompt, 0)), bits(lg))
        c0.close()
        m0.close()
        tok = olib.orc_argmax(rg.ctypes.data, len(rg))
        for i in range(5):
            lg = c.forward_into(np.array([tok], np.uint32), len(prompt) + i)
            rg = oc.forward_into(np.array([tok], np.uint32), len(prompt) + i, oracle.MODE_DEFAULT)
            assert np.array_equal(bits(lg), bits(rg)), f"decode step {i} logits differ"
            tok = olib.orc_argmax(rg.ctypes.data, len(rg))
    finally:
        c.close()
        oc.close()
        m.close()
        om.close()


@pytest.mark.parametrize("n_prompt", [1100, 4100])
def test_softmax_walk_replays_bit_exact(n_prompt, monkeypatch):
    """The decode softmax's exact parallel sum (rows of 1024 positions or
    more; 8 query heads per KV head take k_attn_softmax) with its replay
    paths forced by RLH_SOFTMAX_WALK_SHIFT, which moves the runs' predicted
    binades: 1 every run's one up, 2 one down (every run is replayed from
    its exact start, a walk pass per run, stops at every lane of a 64-run
    group including the last), 3 every third run's one up (scans that pass
    two runs, then stop). The sum, and so every logit, must not change:
    bit-exact against the oracle's sequential loop in every mode, six decode
    steps each, and equal to the unforced run."""
    print(f"softmax walk replays, prompt {n_prompt}", flush=True)
    spec, tensors, m, om = _get("tiny-g8-q4km")
    prompt = rlh.synth_tokens(78, n_prompt, spec.vocab)
    max_ctx = n_prompt + 16
    lib = oracle.load()
    oc = om.new_cache(max_ctx)
    rg = oc.forward_into(prompt, 0, oracle.MODE_BATCH_INT)
    toks, refs = [lib.orc_argmax(rg.ctypes.data, len(rg))], []
    for i in range(6):
        rg = oc.forward_into(np.array([toks[-1]], np.uint32), n_prompt + i, oracle.MODE_DEFAULT)
        refs.append(rg)
        toks.append(lib.orc_argmax(rg.ctypes.data, len(rg)))
    oc.close()
    for mode in ("0", "1", "2", "3"):
        print(f"  walk shift mode {mode}", flush=True)
        monkeypatch.setenv("RLH_SOFTMAX_WALK_SHIFT", mode)
        c = m.new_cache(max_ctx)
        try:
            c.forward_into(prompt, 0)
            for i in range(6):
                lg = c.forward_into(np.array([toks[i]], np.uint32), n_prompt + i)
                assert np.array_equal(bits(lg), bits(refs[i])), \
                    f"mode {mode} step {i}: logits differ (rel {rel_l2(lg, refs[i]):.2e})"
        finally:
            c.close()


def _add_biases(spec, tensors, seed):
    qd, kvd = spec.n_head * spec.head_dim, spec.n_head_kv * spec.head_dim
    lib = rlh.load()
    for layer in range(spec.n_layer):
        for kind, n in ((rlh.T_ATTN_Q_BIAS, qd), (rlh.T_ATTN_K_BIAS, kvd), (rlh.T_ATTN_V_BIAS, kvd)):
            v = np.empty(n, np.float32)
            lib.rlh_synth_normal(seed, rlh.tensor_id(kind, layer), 0, n, 0.0, 0.5, v.ctypes.data)
            tensors.append((kind, layer, rlh.F32, n, 1, v.view(np.uint8)))


@pytest.mark.parametrize("ty,biases", [(rlh.Q4_K, False), (rlh.Q6_K, True), (rlh.Q8_0, False), (rlh.Q8_0, True),
                                       (rlh.Q4_0, True), (rlh.Q5_K, True), (rlh.F16, False), (rlh.F32, True)])
def test_prefill_one_type_wide(ty, biases):
    """q, k and v of one type in one launch, and gate and up in one, at sizes
    that take the large tiles: 499 tokens x 2560 rows are 1280 tiles of 32 x
    32 (16 x 16 ones below 1024), for the f32 types 8 x 80 blocks of 32 rows
    (the 16-row ones would put five on a CU against three). With a v bias the
    third segment goes to a buffer, without one straight into the cache's
    rows."""
    print(f"prefill one type {ty} biases={biases}", flush=True)
    spec = rlh.ModelSpec("one-type-wide", 2, 512, 1024, 12, 4, 300, True, rlh._all(ty), n_ctx=1024)
    tensors = rlh.synth_model(spec, 71 + ty)
    if biases:
        _add_biases(spec, tensors, 72)
    _check_prefill(spec, tensors, rlh.synth_tokens(73, 530, spec.vocab), [499, 31])


@pytest.mark.parametrize("kind", ["subnormal", "nan", "overflow"])
def test_prefill_attention_special_values(kind):
    """K, V, scores and probabilities outside the normal range through the
    attention products, over rows of several 32-position chunks.
    subnormal: every K and V value and every p * V product is subnormal or
    just above (large q and attn_output values bring scores and outputs back).
    nan: one token's K and V rows are NaN; the tokens before it, whose blocks
    and chunks hold those rows too, must not see them.
    overflow: K so large that some scores are infinite: -inf ones take no
    weight, rows with a +inf one become NaN."""
    print(f"attention special values: {kind}", flush=True)
    types = {**rlh._all(rlh.F16), rlh.T_ATTN_V: rlh.F32, rlh.T_ATTN_OUTPUT: rlh.F32, rlh.T_TOKEN_EMBD: rlh.F32}
    spec = rlh.ModelSpec("special", 2, 256, 512, 8, 2, 500, True, types, n_ctx=512)
    tensors = rlh.synth_model(spec, 81)
    tokens = rlh.synth_tokens(82, 171, spec.vocab)
    first = {k: buf.view(np.float32) for k, l, ty, _, _, buf in tensors if l == 0 and ty == rlh.F32}
    if kind == "subnormal":
        first[rlh.T_ATTN_K_NORM][:] *= np.float32(3e-39)
        first[rlh.T_ATTN_Q_NORM][:] *= np.float32(3e37)
        first[rlh.T_ATTN_V][:] *= np.float32(1e-38)
        first[rlh.T_ATTN_OUTPUT][:] *= np.float32(1e38)
    elif kind == "nan":
        bad = int(tokens[101])
        tokens[tokens == bad] = (bad + 1) % spec.vocab
        tokens[101] = bad
        first[rlh.T_TOKEN_EMBD].reshape(spec.vocab, -1)[bad, 7] = np.nan
    else:
        first[rlh.T_ATTN_K_NORM][:] = 0  # one value per KV head: a score is two products
        first[rlh.T_ATTN_K_NORM][5] = 6e37
    rows, logits = _check_prefill(spec, tensors, tokens, [150, 21])
    v1 = rows[1][1]
    if kind == "subnormal":
        tiny = np.finfo(np.float32).tiny
        assert (np.abs(rows[0][0]) < tiny).mean() > 0.9 and (np.abs(rows[0][1]) < tiny).mean() > 0.9
        assert np.isfinite(logits).all() and np.abs(v1).max() > 0
    elif kind == "nan":
        assert np.isfinite(v1[:101]).all() and np.isnan(v1[101:]).all()
    else:
        assert np.isfinite(rows[0][0]).all() and np.isfinite(v1[0]).all() and np.isnan(v1[-1]).any()
