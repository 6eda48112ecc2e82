"""Group-quantized models (soc_model_quantize) on the GPU against the oracle run on the same weights: the projections
packed by the library's packer and dequantized (w = code * scale, exact in fp32), everything else as the fp16 model.
Prefill logits of every row, greedy decode steps, and the device-fed decode loop; int8 and int4. A prompt of up to 8
rows runs the group-quantized kernels (exact products); a longer one the fp16 prefill kernels on each layer's
projections dequantized to fp16 (rounded to nearest). The GPU rounds the projections' input activations to fp16;
the tolerance is the model tolerance."""
import numpy as np
import pytest

import soc_amd as S
from tests.parity import assert_logits_close

pytestmark = pytest.mark.gpu

CFG = S.QwenConfig(vocab_size=1024, hidden_size=256, num_hidden_layers=2, num_attention_heads=4,
                   num_key_value_heads=2, intermediate_size=512, tie_word_embeddings=False)


def _dequantized(oracle_mod, w, bits):
    """The model's weights with every projection replaced by its dequantized group-quantized copy (fp32)."""
    out = dict(w)
    for name, arr in w.items():
        if any(p in name for p in ("q_proj", "k_proj", "v_proj", "o_proj", "gate_proj", "up_proj", "down_proj")):
            n, k = arr.shape
            codes, scales = S.quantize_group(arr, bits)
            out[name] = oracle_mod.dequant_group(codes, bits, scales, n, k)
    return out


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("n", [5, 13, 100])
def test_quantized_model_matches_oracle(gpu_ctx, oracle_mod, bits, n):
    w = S.synth_weights(CFG, 41, 0.05)
    m = S.Model(gpu_ctx, CFG).load(w).quantize(bits)
    om = oracle_mod.OracleModel(CFG, _dequantized(oracle_mod, w, bits))
    cap = n + 16
    kv = S.KVCache(m, 1, cap)
    try:
        assert m.decode_path() == "graph"
        ids = S.synth_tokens(42, "quant", CFG.vocab_size, n)
        lg, tok = S.prefill(m, kv, 0, ids, 0, logit_rows=n)
        cache = oracle_mod.OracleCache(om, cap)
        ref = cache.forward(ids, 0, logit_rows=n)
        assert_logits_close(lg, ref, f"int{bits} prefill rows, {n} tokens")
        assert tok == oracle_mod.sample(ref[-1])
        toks = [tok]
        for i in range(6):
            lg, t = S.decode(m, kv, 0, toks[-1])
            r = cache.forward(np.array([toks[-1]], np.int32), n + i)
            assert_logits_close(lg, r[0], f"int{bits} decode {i}")
            assert t == oracle_mod.sample(r[0])
            toks.append(t)
        # the device-fed loop (captured decode graph) from the same state
        kv2 = S.KVCache(m, 1, cap)
        try:
            _, t0 = S.prefill(m, kv2, 0, ids, 0, logit_rows=0)
            assert [t0] + S.decode_steps(m, kv2, 0, t0, 6).tolist() == toks
        finally:
            kv2.close()
        with pytest.raises(S.SocError):
            S.decode_batch(m, kv, [0], [toks[-1]])
        with pytest.raises(S.SocError):
            m.quantize(bits)  # already quantized
    finally:
        kv.close()
        m.close()


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("hidden,inter,n", [(64, 64, 3), (320, 704, 8), (1088, 3136, 2), (2112, 1088, 1)])
def test_quantized_layer_widths(gpu_ctx, oracle_mod, bits, hidden, inter, n):
    """The fused quantized projections (RMSNorm, residual and SwiGLU folded in) at widths off their tiles: one scale
    group, odd numbers of groups, and rows past one and two code loads per wave; a prompt of n <= 8 rows (row kernel),
    then three decode steps (one-row kernel), against the oracle on the dequantized weights."""
    cfg = S.QwenConfig(vocab_size=512, hidden_size=hidden, num_hidden_layers=2, num_attention_heads=4,
                       num_key_value_heads=2, intermediate_size=inter, tie_word_embeddings=False)
    w = S.synth_weights(cfg, 43, 0.05)
    m = S.Model(gpu_ctx, cfg).load(w).quantize(bits)
    om = oracle_mod.OracleModel(cfg, _dequantized(oracle_mod, w, bits))
    kv = S.KVCache(m, 1, 32)
    try:
        ids = S.synth_tokens(44, "widths", cfg.vocab_size, n)
        lg, tok = S.prefill(m, kv, 0, ids, 0, logit_rows=n)
        cache = oracle_mod.OracleCache(om, 32)
        assert_logits_close(lg, cache.forward(ids, 0, logit_rows=n), f"int{bits} {hidden}/{inter}, {n} rows")
        for i in range(3):
            lg, t = S.decode(m, kv, 0, tok)
            r = cache.forward(np.array([tok], np.int32), n + i)
            assert_logits_close(lg, r[0], f"int{bits} {hidden}/{inter}, decode {i}")
            tok = t
    finally:
        kv.close()
        m.close()


@pytest.mark.parametrize("length", [97, 300])
@pytest.mark.parametrize("bits", [8, 4])
def test_quantized_decode_keeps_its_bits(gpu_ctx, golden, bits, length):
    """One decode row of a quantized model in the summation order of separate norm, projection, SwiGLU and residual
    kernels, bit for bit: tests/golden/qdecode_rows.npz holds the logits of four steps that those kernels gave
    (Qwen3-0.6B widths, two layers, 97 and 300 cached keys: one attention chunk and five). Every projection rounds its
    input to fp16, so any other order shows as a few 1e-4."""
    cfg = S.QwenConfig(vocab_size=256, hidden_size=1024, num_hidden_layers=2, num_attention_heads=16,
                       num_key_value_heads=8, intermediate_size=3072)
    m = S.Model(gpu_ctx, cfg).load(S.synth_weights(cfg, 81)).quantize(bits)
    kv = S.KVCache(m, 1, 320)
    try:
        kv.fill_synthetic(0, length, 82)
        got = np.stack([S.decode(m, kv, 0, t)[0] for t in (11, 200, 77, 5)])
    finally:
        kv.close()
        m.close()
    want = golden("qdecode_rows.npz")[f"int{bits}_{length}"]
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), float(np.max(np.abs(got - want)))


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("n", [2, 3, 5, 8])
@pytest.mark.parametrize("hidden,inter", [(1088, 6144), (4160, 1088)])
def test_quantized_long_rows(gpu_ctx, oracle_mod, bits, n, hidden, inter):
    """Prompts of 2 to 8 rows where a projection's rows outgrow the registers of the row kernel (K > 4096 int4, 3072
    int8), so that each tile takes several passes over K: the residual form (inter 6144, the down projection of
    Qwen3-1.7B), the RMSNorm and SwiGLU forms (hidden 4160), against the oracle on the dequantized weights."""
    cfg = S.QwenConfig(vocab_size=512, hidden_size=hidden, num_hidden_layers=1, num_attention_heads=4,
                       num_key_value_heads=2, intermediate_size=inter, tie_word_embeddings=True)
    w = S.synth_weights(cfg, 47, 0.05)
    m = S.Model(gpu_ctx, cfg).load(w).quantize(bits)
    om = oracle_mod.OracleModel(cfg, _dequantized(oracle_mod, w, bits))
    kv = S.KVCache(m, 1, 16)
    try:
        ids = S.synth_tokens(48, "long rows", cfg.vocab_size, n)
        lg, _ = S.prefill(m, kv, 0, ids, 0, logit_rows=n)
        ref = oracle_mod.OracleCache(om, 16).forward(ids, 0, logit_rows=n)
        assert_logits_close(lg, ref, f"int{bits} {hidden}/{inter}, {n} rows")
    finally:
        kv.close()
        m.close()
