"""Ragged multi-sequence decode (soc_decode_batch / soc_decode_batch_steps) on an MI355X.

A batch row has the reference's one-sequence decode semantics for its own KV slot (GenerationContext::
DecodeNextToken, Mac/gpu/src/runtime/generation_context.cpp:68-172). Checks:
  (1) each row vs soc_decode of the same slot on an identical cache: logits within the model tolerance
      (max |diff| <= 2e-2 and <= 1e-2 * max |logit|), identical greedy tokens;
  (2) permuting the rows permutes the results bit for bit (rows are independent);
  (3) each row vs the CPU oracle's cached forward of that sequence, with KV lengths that mix short prefixes and
      several 256-key attention chunks;
  (4) soc_decode_batch_steps equals a loop of soc_decode_batch, bit for bit;
  (5) bad batches are rejected without touching any slot.
"""
import numpy as np
import pytest

import soc_amd as S
from tests.parity import assert_logits_close

pytestmark = pytest.mark.gpu

def small_cfg(nq=4, nkv=2):
    return S.QwenConfig(vocab_size=2048, hidden_size=256, num_hidden_layers=2, num_attention_heads=nq,
                        num_key_value_heads=nkv, intermediate_size=512, tie_word_embeddings=False)


PROMPT_LENS = [5, 17, 33, 2, 64]


def _prefilled_caches(m, cfg, count, cap=128):
    """`count` caches holding the same five prompts (GPU prefill) in slots 0..4; returns caches and last tokens."""
    caches, last = [], None
    for _ in range(count):
        kv = S.KVCache(m, len(PROMPT_LENS), cap)
        toks = []
        for slot, n in enumerate(PROMPT_LENS):
            ids = S.synth_tokens(20 + slot, "batch.prompt", cfg.vocab_size, n)
            _, t = S.prefill(m, kv, slot, ids, 0, logit_rows=0)
            toks.append(t)
        caches.append(kv)
        last = toks
    return caches, np.array(last, np.int32)


@pytest.mark.parametrize("nq,nkv", [(4, 2), (8, 2)])
def test_batch_rows_equal_single_sequence_decode(gpu_ctx, nq, nkv):
    cfg = small_cfg(nq, nkv)
    m = S.Model(gpu_ctx, cfg).load(S.synth_weights(cfg, 31))
    (a, b), last = _prefilled_caches(m, cfg, 2)
    try:
        order = np.array([3, 0, 4, 1, 2], np.int32)
        lg, nxt = S.decode_batch(m, a, order, last[order])
        for i, slot in enumerate(order):
            ref, t = S.decode(m, b, int(slot), int(last[slot]))
            assert_logits_close(lg[i], ref, f"row {i} (slot {slot})")
            assert int(nxt[i]) == t
            assert a.length(int(slot)) == b.length(int(slot)) == PROMPT_LENS[slot] + 1
    finally:
        a.close()
        b.close()
        m.close()


def test_batch_many_rows_slabs_and_tiled_path(gpu_ctx):
    """20 and 70 rows, beyond the 16 of the skinny projections (split-K row GEMMs on 64- and 128-row tiles): every row
    agrees with single-sequence decode of its slot within the model tolerance, with the same greedy token."""
    cfg = small_cfg()
    m = S.Model(gpu_ctx, cfg).load(S.synth_weights(cfg, 33))
    nslots = 70
    kvs = [S.KVCache(m, nslots, 32) for _ in range(2)]
    try:
        last = np.zeros(nslots, np.int32)
        for kv in kvs:
            for slot in range(nslots):
                ids = S.synth_tokens(40 + slot, "batch.many", cfg.vocab_size, 1 + slot % 7)
                _, last[slot] = S.prefill(m, kv, slot, ids, 0, logit_rows=0)
        for n in (20, 70):
            slots = np.arange(n, dtype=np.int32)[::-1].copy()
            lg, nxt = S.decode_batch(m, kvs[0], slots, last[slots])
            for i, slot in enumerate(slots):
                ref, t = S.decode(m, kvs[1], int(slot), int(last[slot]))
                assert_logits_close(lg[i], ref, f"{n} rows, row {i} (slot {slot})")
                assert int(nxt[i]) == t
            last[slots] = nxt
    finally:
        for kv in kvs:
            kv.close()
        m.close()


def test_batch_permutation_invariance_and_steps(gpu_ctx):
    cfg = small_cfg()
    m = S.Model(gpu_ctx, cfg).load(S.synth_weights(cfg, 32))
    (a, b), last = _prefilled_caches(m, cfg, 2)
    try:
        p1 = np.array([0, 1, 2, 3, 4], np.int32)
        p2 = np.array([4, 2, 0, 3, 1], np.int32)
        l1, n1 = S.decode_batch(m, a, p1, last[p1])
        l2, n2 = S.decode_batch(m, b, p2, last[p2])
        inv = np.argsort(p2)
        assert np.array_equal(l1, l2[inv]) and np.array_equal(n1, n2[inv])
        for slot in range(5):  # the appended keys/values agree too
            ka, va = a.read(slot, 1)
            kb, vb = b.read(slot, 1)
            assert np.array_equal(ka, kb) and np.array_equal(va, vb)
        # 4 graph-replayed steps == 4 single steps
        steps = S.decode_batch_steps(m, a, p1, n1, 4)
        tok, loop = n1.copy(), []
        for _ in range(4):
            _, tok = S.decode_batch(m, b, p1, tok)
            loop.append(tok.copy())
        assert np.array_equal(steps, np.stack(loop))
        for slot in range(5):
            assert a.length(slot) == b.length(slot) == PROMPT_LENS[slot] + 5
    finally:
        a.close()
        b.close()
        m.close()


def test_batch_matches_oracle_mixed_lengths(gpu_ctx, oracle_mod):
    """KV prefixes of 300, 5, 520 and 64 positions (seeded N(0,1) fp16 contents) in one batch: each row's logits
    and greedy token against the oracle's cached forward over the same (fp16-valued) prefix."""
    cfg = small_cfg()
    w = S.synth_weights(cfg, 33)
    m = S.Model(gpu_ctx, cfg).load(w)
    lens = [300, 5, 520, 64]
    kv = S.KVCache(m, len(lens), 544)
    try:
        for slot, n in enumerate(lens):
            kv.fill_synthetic(slot, n, 900 + slot)
        prefixes = {slot: [kv.read(slot, layer) for layer in range(cfg.num_hidden_layers)] for slot in range(4)}
        tokens = S.synth_tokens(34, "batch.tok", cfg.vocab_size, 4)
        slots = np.array([2, 0, 3, 1], np.int32)
        lg, nxt = S.decode_batch(m, kv, slots, tokens[slots])
        om = oracle_mod.OracleModel(cfg, w)
        for i, slot in enumerate(slots):
            n = lens[slot]
            cache = oracle_mod.OracleCache(om, n + 1)
            for layer, (k, v) in enumerate(prefixes[int(slot)]):
                for pos in range(n):
                    cache.write(layer, pos, k[:, pos, :].astype(np.float32), v[:, pos, :].astype(np.float32))
            ref = cache.forward(np.array([tokens[slot]], np.int32), n)
            assert_logits_close(lg[i], ref[0], f"row {i} (slot {slot}, {n} cached positions)")
            assert int(nxt[i]) == oracle_mod.sample(ref[0])
            assert kv.length(int(slot)) == n + 1
    finally:
        kv.close()
        m.close()


def test_ragged_qwen3_4b_matches_reference(gpu_ctx, golden):
    """The benchmarked ragged step at its own workload: Qwen3-4B (seed-1 weights), 16 sequences with KV lengths
    U[64, 4096] (seed 5) of seeded N(0, 1) fp16 contents, one token each (seed 6). The rows of the longest and
    shortest sequences and of slots 0 and 1 against the compiled reference's cached forward over the same caches;
    then a second step of all 16 rows, whose checked rows equal single-sequence decode of those slots."""
    g = golden("ragged4b.npz")
    cfg = S.QWEN3_4B
    m = S.Model(gpu_ctx, cfg).synthesize(int(g["weight_seed"]), 0.02)
    lens = g["kv_lens"].astype(np.int64)
    n = len(lens)
    kv = S.KVCache(m, n, int(lens.max()) + 4)
    try:
        for slot, ln in enumerate(lens):
            kv.fill_synthetic(slot, int(ln), 7)
        slots = np.arange(n, dtype=np.int32)
        toks = g["tokens"]
        lg, nxt = S.decode_batch(m, kv, slots, toks)
        for r, slot in enumerate(g["slots"]):
            what = f"4B ragged slot {int(slot)} (kv {int(lens[slot])})"
            assert int(nxt[slot]) == int(g["argmax"][r]), what
            assert_logits_close(lg[slot][g["top_ids"][r]], g["top_vals"][r], what + " top-64")
            assert_logits_close(lg[slot][g["sample_idx"]], g["sample_vals"][r], what + " sampled")
        # a second batch step vs one-sequence decode of the same slots (a second cache with the same contents in
        # those slots)
        lg2, nxt2 = S.decode_batch(m, kv, slots, nxt)
        one = S.KVCache(m, n, int(lens.max()) + 4)
        try:
            for slot in g["slots"]:
                slot = int(slot)
                one.fill_synthetic(slot, int(lens[slot]), 7)
                _, t0 = S.decode(m, one, slot, int(toks[slot]))
                assert t0 == int(nxt[slot])
                lg1, t1 = S.decode(m, one, slot, t0)
                assert t1 == int(nxt2[slot])
                assert_logits_close(lg2[slot], lg1, f"4B ragged slot {slot} batch step 2 vs decode")
        finally:
            one.close()
    finally:
        kv.close()
        m.close()


@pytest.mark.parametrize("pattern", ["repeated_rows", "all_zero"])
def test_batch_greedy_ties_across_chunks(gpu_ctx, pattern):
    """Exact ties in the greedy choice: a 65536-token LM head whose rows from 40000 on repeat 8 seeded rows (every
    maximum recurs ~3000 times, across all the blocks that scan a row), or an all-zero LM head (every logit 0).
    Each row's token must be the lowest index of its maximum logit: the reference's greedy pick
    (Mac/cpu/src/sampler.cpp:41-58, a top-1 partial sort, which replaces its candidate only on a strictly greater
    score)."""
    cfg = S.QwenConfig(vocab_size=65536, hidden_size=256, num_hidden_layers=2, num_attention_heads=4,
                       num_key_value_heads=2, intermediate_size=512, tie_word_embeddings=False)
    w = S.synth_weights(cfg, 36)
    head = np.zeros((cfg.vocab_size, cfg.hidden_size), np.float16)
    if pattern == "repeated_rows":
        rows = w["lm_head.weight"][:8]
        head[40000:] = rows[np.arange(cfg.vocab_size - 40000) % 8]
    w["lm_head.weight"] = head
    m = S.Model(gpu_ctx, cfg).load(w)
    (kv,), last = _prefilled_caches(m, cfg, 1)
    try:
        for n in (5, 1, 3):  # 64 blocks per row for each n
            slots = np.arange(n, dtype=np.int32)
            lg, nxt = S.decode_batch(m, kv, slots, last[slots])
            for i in range(n):
                want = int(np.argmax(lg[i]))  # numpy: first index of the maximum
                assert int(nxt[i]) == want, (pattern, n, i)
                if pattern == "all_zero":
                    assert want == 0
                else:
                    assert want >= 40000 or lg[i].max() == 0.0
            last[slots] = nxt
    finally:
        kv.close()
        m.close()


def test_batch_error_paths(gpu_ctx):
    cfg = small_cfg()
    m = S.Model(gpu_ctx, cfg).load(S.synth_weights(cfg, 35))
    kv = S.KVCache(m, 3, 8)
    try:
        for slot in range(3):
            S.prefill(m, kv, slot, np.array([1, 2, 3], np.int32), 0, logit_rows=0)
        with pytest.raises(S.SocError) as e:
            S.decode_batch(m, kv, [0, 0], [1, 2])  # duplicate slot
        assert e.value.code == S.capi.SOC_ERR_INVALID
        with pytest.raises(S.SocError) as e:
            S.decode_batch(m, kv, [0, 5], [1, 2])  # slot out of range
        assert e.value.code == S.capi.SOC_ERR_INVALID
        with pytest.raises(S.SocError) as e:
            S.decode_batch(m, kv, [0, 1], [1, cfg.vocab_size])  # token out of range
        assert e.value.code == S.capi.SOC_ERR_INVALID
        with pytest.raises(S.SocError) as e:
            S.decode_batch_steps(m, kv, [0, 1], [1, 2], 6)  # 3 + 6 > capacity 8
        assert e.value.code == S.capi.SOC_ERR_CAPACITY
        assert [kv.length(s) for s in range(3)] == [3, 3, 3]
        S.decode_batch_steps(m, kv, [2, 0], [1, 2], 5)
        assert [kv.length(s) for s in range(3)] == [8, 3, 8]
    finally:
        kv.close()
        m.close()


def test_batch_rows_staged_through_pinned_memory(gpu_ctx):
    """Calls of growing and shrinking row counts (the staging area is regrown, then used in part; counts around the
    256 rows of a staging block): the returned tokens are the argmax of the returned logits, slots advance by one, and
    a graph step run on a second cache from the same rows gives the same tokens."""
    cfg = small_cfg()
    m = S.Model(gpu_ctx, cfg).load(S.synth_weights(cfg, 71))
    a, b = S.KVCache(m, 300, 16), S.KVCache(m, 300, 16)
    rng = np.random.default_rng(72)
    try:
        for n in (2, 256, 257, 300, 3, 1):
            slots = rng.permutation(300)[:n].astype(np.int32)
            toks = rng.integers(0, cfg.vocab_size, n).astype(np.int32)
            for i in range(300):
                a.reset(i)
                b.reset(i)
            for step in range(2):
                lg, nxt = S.decode_batch(m, a, slots, toks)
                np.testing.assert_array_equal(nxt, np.argmax(lg, axis=1), err_msg=f"{n} rows")
                assert all(a.length(int(i)) == step + 1 for i in slots)
                np.testing.assert_array_equal(S.decode_batch_steps(m, b, slots, toks, 1)[0], nxt)
                toks = nxt
    finally:
        a.close()
        b.close()
        m.close()


@pytest.mark.parametrize("n", [17, 64, 65, 128, 130])
def test_batch_row_gemm_edges(gpu_ctx, n):
    """The split-K row GEMMs of more than 16 rows at the edges of their 64- and 128-row tiles, widths off the 128-column
    tiles (hidden 352, intermediate 480): rows agree with single-sequence decode within the model tolerance, permuting
    them permutes the results bit for bit, and the captured steps equal the eager ones."""
    cfg = S.QwenConfig(vocab_size=1000, hidden_size=352, num_hidden_layers=2, num_attention_heads=4,
                       num_key_value_heads=2, intermediate_size=480, tie_word_embeddings=False)
    m = S.Model(gpu_ctx, cfg).load(S.synth_weights(cfg, 51))
    kvs = [S.KVCache(m, n, 300) for _ in range(2)]
    try:
        last = np.zeros(n, np.int32)
        for kv in kvs:
            for slot in range(n):
                plen = 270 if slot == 3 else 1 + slot % 5  # one row over two attention chunks
                _, last[slot] = S.prefill(m, kv, slot, S.synth_tokens(60 + slot, "rows", cfg.vocab_size, plen), 0,
                                          logit_rows=0)
        order = np.random.RandomState(n).permutation(n).astype(np.int32)
        lg, nxt = S.decode_batch(m, kvs[0], order, last[order])
        ident = np.arange(n, dtype=np.int32)
        lg2, nxt2 = S.decode_batch(m, kvs[1], ident, last)
        assert np.array_equal(lg2[order], lg) and np.array_equal(nxt2[order], nxt)
        for kv in kvs:
            for slot in range(n):
                kv_len = 270 if slot == 3 else 1 + slot % 5
                S.capi.check(S.lib().soc_kv_set_length(kv.h, slot, kv_len))
        for slot in (0, 3, n - 1):
            ref, t = S.decode(m, kvs[1], slot, int(last[slot]))
            assert_logits_close(lg2[slot], ref, f"{n} rows, slot {slot}")
            assert int(nxt2[slot]) == t
            S.capi.check(S.lib().soc_kv_set_length(kvs[1].h, slot, 270 if slot == 3 else 1 + slot % 5))
        steps = S.decode_batch_steps(m, kvs[0], ident, last, 3)
        tok, loop = last.copy(), []
        for _ in range(3):
            _, tok = S.decode_batch(m, kvs[1], ident, tok)
            loop.append(tok.copy())
        assert np.array_equal(steps, np.stack(loop))
    finally:
        for kv in kvs:
            kv.close()
        m.close()


def test_batch_rows_of_models_that_share_a_context(gpu_ctx):
    """Two models of one context take turns with growing and shrinking batches (their rows are staged in the same pinned
    words): each call's logits and tokens are bit for bit those of the model stepping alone."""
    cfgs = [small_cfg(), S.QwenConfig(vocab_size=64, hidden_size=128, num_hidden_layers=1, num_attention_heads=2,
                                      num_key_value_heads=1, intermediate_size=128, tie_word_embeddings=True)]
    models = [S.Model(gpu_ctx, c).load(S.synth_weights(c, 90 + i)) for i, c in enumerate(cfgs)]
    counts = (3, 1, 40, 17, 1024, 2)
    kvs = [S.KVCache(m, max(counts), 8) for m in models for _ in range(2)]

    def step(which, turn, copy):
        n, kv = counts[turn], kvs[2 * which + copy]
        rng = np.random.default_rng(10 * turn + which)
        slots = rng.permutation(max(counts))[:n].astype(np.int32)
        return S.decode_batch(models[which], kv, slots, rng.integers(0, cfgs[which].vocab_size, n).astype(np.int32))

    try:
        alone = [[step(i, t, 0) for t in range(len(counts))] for i in range(2)]
        for t in range(len(counts)):
            for i in range(2):
                lg, nxt = step(i, t, 1)
                assert np.array_equal(lg, alone[i][t][0]) and np.array_equal(nxt, alone[i][t][1]), (t, i)
                assert np.array_equal(nxt, np.argmax(lg, axis=1))
    finally:
        for kv in kvs:
            kv.close()
        for m in models:
            m.close()


@pytest.mark.parametrize("hidden,inter,nq", [(1024, 3072, 16), (2560, 9728, 32)])
def test_batch_rows_keep_their_bits_as_others_join(gpu_ctx, hidden, inter, nq):
    """A sequence's logits and appended keys are bit for bit the same at every row count that takes as many row tiles: 1 ..
    16 rows, 17 .. 64, 65 .. 128, 129 .. 256 (Qwen3-0.6B and 4B widths, where K is split)."""
    cfg = S.QwenConfig(vocab_size=512, hidden_size=hidden, num_hidden_layers=1, num_attention_heads=nq,
                       num_key_value_heads=8, intermediate_size=inter, tie_word_embeddings=True)
    m = S.Model(gpu_ctx, cfg).synthesize(7)
    kv = S.KVCache(m, 256, 48)
    toks = np.random.default_rng(8).integers(0, cfg.vocab_size, 256).astype(np.int32)
    try:
        for slot in range(256):
            kv.fill_synthetic(slot, 1 + slot % 40, 9)
        for counts in ((1, 2, 9, 16), (17, 18, 33, 64), (65, 100, 128), (129, 200, 256)):
            first = None
            for n in counts:
                for slot in range(n):
                    S.capi.check(S.lib().soc_kv_set_length(kv.h, slot, 1 + slot % 40))
                rows = np.arange(n, dtype=np.int32)
                lg, _ = S.decode_batch(m, kv, rows, toks[:n])
                got = lg[: counts[0]], kv.read(0, 0)[0]
                first = first or got
                assert np.array_equal(got[0], first[0]) and np.array_equal(got[1], first[1]), n
    finally:
        kv.close()
        m.close()


def _first_token_logits(cfg, w, toks, cached, round_head=False):
    """Logits of sequences of one token in float64; the attention, over one key, returns its value, for which the cached
    fp16 values [layers][n][kv heads * 128] stand. round_head: the head's input rounded to fp16, as it would be without
    its low half. Also the values before their rounding."""
    f = {k: v.view(np.float16).astype(np.float64) for k, v in w.items()}

    def norm(x, gain):
        return x / np.sqrt(np.mean(x * x, -1, keepdims=True) + cfg.rms_norm_eps) * gain

    x, values = f["model.embed_tokens.weight"][toks], []
    for l in range(cfg.num_hidden_layers):
        p = f"model.layers.{l}."
        values.append(norm(x, f[p + "input_layernorm.weight"]) @ f[p + "self_attn.v_proj.weight"].T)
        v = cached[l].astype(np.float64).reshape(len(toks), -1, 128)
        attn = np.repeat(v, cfg.num_attention_heads // cfg.num_key_value_heads, axis=1).reshape(len(toks), -1)
        x = x + attn @ f[p + "self_attn.o_proj.weight"].T
        h = norm(x, f[p + "post_attention_layernorm.weight"])
        g = h @ f[p + "mlp.gate_proj.weight"].T
        x = x + (g / (1 + np.exp(-g)) * (h @ f[p + "mlp.up_proj.weight"].T)) @ f[p + "mlp.down_proj.weight"].T
    h = norm(x, f["model.norm.weight"])
    if round_head:
        h = h.astype(np.float16).astype(np.float64)
    return h @ f["model.embed_tokens.weight"].T, np.stack(values)


@pytest.mark.parametrize("n,hidden,vocab", [
    (65, 256, 65537), (130, 256, 65537),             # the head's 128 x 128 tiles (512 of them), one and two high
    (17, 1024, 512), (65, 2048, 512), (17, 2560, 512), (130, 4160, 512),  # each width of the residual and norm step
])
def test_batch_row_gemms_in_full_precision(gpu_ctx, n, hidden, vocab):
    """Rows beyond 16 against a float64 forward, tightly enough to see the low halves of the activation pairs: fp32 sums
    and 22-bit activations are good for some 1e-6 of a row's norm (2e-7 to 7e-7 seen), the head's input without its low
    half is off by 2^-11 / sqrt(12) = 1.4e-4 (checked on the reference). The cached values are the reference's to within
    one fp16 rounding."""
    cfg = S.QwenConfig(vocab_size=vocab, hidden_size=hidden, num_hidden_layers=2, num_attention_heads=4,
                       num_key_value_heads=2, intermediate_size=512, tie_word_embeddings=True)
    w = S.synth_weights(cfg, 61, 0.05)
    m = S.Model(gpu_ctx, cfg).load(w)
    kv = S.KVCache(m, n, 4)
    try:
        toks = np.random.default_rng(62).integers(0, vocab, n).astype(np.int32)
        lg, _ = S.decode_batch(m, kv, np.arange(n, dtype=np.int32), toks)
        cached = np.stack([[kv.read(slot, l)[1][:, 0].reshape(-1) for slot in range(n)]
                           for l in range(cfg.num_hidden_layers)])
    finally:
        kv.close()
        m.close()
    ref, values = _first_token_logits(cfg, w, toks, cached)
    # half an fp16 step, and 3e-6 of a value's spread over the row (0.05 sqrt(hidden) <= 3.3) for its fp32 sum
    assert np.all(np.abs(cached - values) <= 2.0 ** -11 * np.abs(values) + 1e-5)
    scale = np.linalg.norm(ref, axis=1)
    err = np.max(np.linalg.norm(lg - ref, axis=1) / scale)
    rounded = np.min(np.linalg.norm(_first_token_logits(cfg, w, toks, cached, True)[0] - ref, axis=1) / scale)
    print(f"[rows] {n} x {hidden}, {vocab} words: {err:.2e}, head input in fp16 alone {rounded:.2e}", flush=True)
    assert err <= 1e-5 < rounded / 2, (err, rounded)
