"""GPU parity of the batched prefill (fllm_prefill with a prompt that continues the cache).

The contract is that of n consecutive Forward calls (LlamaLanguageModel.cs:133-137): the K/V rows
of every position, the last position's logits and its greedy token. The batched path runs the
projections as matrix-core GEMMs over all tokens and a causal attention over the cache, so its
results are compared with the oracle and with the per-token path within the f32 bar (normwise
relative error 1e-3), and the greedy tokens that follow must be the oracle's.
"""
import numpy as np
import pytest

import dotnetfoundryllm_amd as F
import dotnetfoundryllm_amd._native as N
import oracle_bind as O
from dotnetfoundryllm_amd.configs import CONFIGS, desc_of, synth_bytes, tensor_plan
from fixtures import f32_of, synthetic, upload

pytestmark = pytest.mark.gpu
TOL = 1e-3


def device_model(ctx, desc, tensors):
    m = F.Model(ctx, desc)
    upload(m, tensors)
    return m


def _oracle_prefill(orc, prompt):
    for pos, t in enumerate(prompt):
        assert orc.forward(int(t), pos) == 0


def _oracle_continue(orc, first, pos, n):
    nxt, out = int(first), []
    for _ in range(n):
        assert orc.forward(nxt, pos) == 0
        pos += 1
        lg = orc.logits()
        nxt = int(O.lib.orc_argmax(O.fp(lg), lg.size))
        out.append(nxt)
    return out


SMALL = ["test-llama", "test-llama-straddle", "test-mistral", "test-qwen2", "test-gemma2", "test-gemma2-hd256",
         "test-mixed", "test-ragged", "test-wide-ffn"]


@pytest.mark.parametrize("name", SMALL)
def test_batched_prefill_matches_oracle_and_stepwise(ctx, name):
    cfg, desc, tensors = synthetic(name)
    m = device_model(ctx, desc, tensors)
    kv_b, kv_s = F.HipKvCache(m), F.HipKvCache(m)
    fb, fs = F.HipForwardPass(m), F.HipForwardPass(m)
    orc = O.OracleModel(desc, tensors)
    n = min(40, desc.max_ctx - 10)
    prompt = F.synth_tokens(cfg["seed"], 5, desc.vocab, n)
    try:
        fb.prefill(prompt, 0, kv_b)  # batched
        for pos, t in enumerate(prompt):
            fs.forward(int(t), pos, kv_s)  # one step per token
        _oracle_prefill(orc, prompt)
        assert kv_b.current_length == n == kv_s.current_length
        want = orc.logits()
        assert O.normwise_rel_err(fb.logits, want) <= TOL
        assert O.normwise_rel_err(fb.logits, fs.logits) <= TOL
        for l in range(desc.n_layers):
            for kind, get in ((0, kv_b.get_keys), (1, kv_b.get_values)):
                got = get(l)
                assert O.normwise_rel_err(got, orc.kv(l, kind)) <= TOL, (l, kind)
        assert fb.sample_greedy() == int(O.lib.orc_argmax(O.fp(want), want.size))
        # decoding after the batched prefill gives the oracle's greedy tokens
        steps = min(8, desc.max_ctx - n - 1)
        toks = fb.decode_greedy(int(prompt[-1]), n, steps, kv_b)
        assert list(toks) == _oracle_continue(orc, prompt[-1], n, steps)
    finally:
        orc.close()
        kv_b.close()
        kv_s.close()
        m.close()


@pytest.mark.parametrize("name,cap,n", [("test-llama", 256, 200), ("test-qwen2", 256, 200), ("test-gemma2", 256, 200),
                                        ("test-gemma2", 1280, 1100), ("test-gemma2-hd256", 256, 200),
                                        ("test-mistral", 256, 200)])
def test_batched_prefill_split_attention(ctx, name, cap, n):
    """A prompt of several query blocks with a partial last one (200 tokens: blocks of 64, 64, 64,
    8; 1100: 17 blocks and 12) into a 256- (1280-) position cache: the prefill attention runs every
    block but the first as two halves of its key range plus a merge when all halves fit the
    resident workgroups, as here. Head dim 64 (Llama; Qwen2 with its q/k/v bias; Mistral with its
    window) on the f32 kernel, 128 (Gemma-2: softcaps, window on the even layer; also over 1100
    keys) and 256 on the fp16 kernel over the K / V planes. Logits and every K/V row against the
    oracle, then greedy decode."""
    cfg, desc, tensors = synthetic(name)
    m = device_model(ctx, desc, tensors)
    kv = F.HipKvCache(m, cap)
    fwd = F.HipForwardPass(m)
    orc = O.OracleModel(desc, tensors, cap)
    prompt = F.synth_tokens(cfg["seed"], 7, desc.vocab, n)
    try:
        fwd.prefill(prompt, 0, kv)
        _oracle_prefill(orc, prompt)
        want = orc.logits()
        err = O.normwise_rel_err(fwd.logits, want)
        print(f"{name}: {n} tokens, logits normwise rel err {err:.2e}")
        assert err <= TOL
        for l in range(desc.n_layers):
            assert O.normwise_rel_err(kv.get_keys(l), orc.kv(l, 0)) <= TOL, l
            assert O.normwise_rel_err(kv.get_values(l), orc.kv(l, 1)) <= TOL, l
        toks = fwd.decode_greedy(int(prompt[-1]), n, 4, kv)
        assert list(toks) == _oracle_continue(orc, prompt[-1], n, 4)
    finally:
        orc.close()
        kv.close()
        m.close()


def test_prefill_chunk_contract(ctx):
    """fllm_seq_set_prefill_chunk: tokens < 1 is out of range; a chunk of 24 tokens takes a 61-token
    prompt in passes of 24, 24 and 13 (logits, K/V and the greedy token against the oracle); after
    it, a chunk of 40 makes the next prefill replace the 24-row scratch with a 40-row one, and a
    30-token prompt in one pass stores the same K/V rows as the oracle's first 30 positions."""
    cfg, desc, tensors = synthetic("test-llama")
    m = device_model(ctx, desc, tensors)
    kv = F.HipKvCache(m)
    fwd = F.HipForwardPass(m)
    orc = O.OracleModel(desc, tensors)
    prompt = F.synth_tokens(cfg["seed"], 5, desc.vocab, 61)
    try:
        for bad in (0, -5):
            with pytest.raises(F.ArgumentOutOfRangeException):
                F.set_prefill_chunk(kv, bad)
        F.set_prefill_chunk(kv, 100)
        F.set_prefill_chunk(kv, 24)  # another value before the first prefill
        fwd.prefill(prompt, 0, kv)
        _oracle_prefill(orc, prompt)
        want = orc.logits()
        assert O.normwise_rel_err(fwd.logits, want) <= TOL
        for l in range(desc.n_layers):
            assert O.normwise_rel_err(kv.get_keys(l), orc.kv(l, 0)) <= TOL
            assert O.normwise_rel_err(kv.get_values(l), orc.kv(l, 1)) <= TOL
        assert fwd.sample_greedy() == int(O.lib.orc_argmax(O.fp(want), want.size))
        F.set_prefill_chunk(kv, 40)
        kv.clear()
        fwd.prefill(prompt[:30], 0, kv)
        assert kv.current_length == 30
        kvdim = desc.n_kv_heads * desc.head_dim
        for l in range(desc.n_layers):
            for got, kind in ((kv.get_keys(l), 0), (kv.get_values(l), 1)):
                assert O.normwise_rel_err(got, orc.kv(l, kind)[: 30 * kvdim]) <= TOL, (l, kind)
    finally:
        orc.close()
        kv.close()
        m.close()


@pytest.mark.parametrize("chunk", [512, None], ids=["chunk-512", "chunk-default"])
def test_batched_prefill_several_chunks(ctx, chunk):
    """1100 tokens go through the layers in chunks of 512, 512 and 76: every chunk attends to the
    rows the earlier chunks stored (and, with the default chunk, in one pass). No window; K/V of the
    first, a middle and the last position and the logits against the oracle."""
    from dotnetfoundryllm_amd.configs import _cfg, _types
    cfg = _cfg("chunks-llama", N.ARCH_LLAMA, 2, 256, 4, 2, 512, 512, 1200, 10000.0,
               _types(N.Q4_K, N.Q4_K, N.Q6_K, N.Q4_K, N.Q4_K, N.Q4_K, N.Q6_K, N.Q6_K), norm_std=0.1, seed=23)
    desc = desc_of(cfg)
    tensors = {e[0]: (e, synth_bytes(cfg, e)) for e in tensor_plan(cfg)}
    m = device_model(ctx, desc, tensors)
    kv = F.HipKvCache(m)
    fwd = F.HipForwardPass(m)
    orc = O.OracleModel(desc, tensors)
    prompt = F.synth_tokens(cfg["seed"], 3, desc.vocab, 1100)
    try:
        if chunk:
            F.set_prefill_chunk(kv, chunk)
        fwd.prefill(prompt, 0, kv)
        _oracle_prefill(orc, prompt)
        assert kv.current_length == 1100
        assert O.normwise_rel_err(fwd.logits, orc.logits()) <= TOL
        for l in range(desc.n_layers):
            k, v = kv.get_keys(l), kv.get_values(l)
            kr, vr = orc.kv(l, 0), orc.kv(l, 1)
            assert O.normwise_rel_err(k, kr) <= TOL and O.normwise_rel_err(v, vr) <= TOL
            kvdim = desc.n_kv_heads * desc.head_dim
            for pos in (0, 600, 1099):
                row = slice(pos * kvdim, (pos + 1) * kvdim)
                assert O.normwise_rel_err(k[row], kr[row]) <= TOL, (l, pos)
        toks = fwd.decode_greedy(int(prompt[-1]), 1100, 6, kv)
        assert list(toks) == _oracle_continue(orc, prompt[-1], 1100, 6)
    finally:
        orc.close()
        kv.close()
        m.close()


@pytest.mark.parametrize("chunk", [512, None], ids=["chunk-512", "chunk-default"])
@pytest.mark.parametrize("arch", [N.ARCH_MISTRAL, N.ARCH_GEMMA2])
def test_batched_prefill_window_across_chunks(ctx, arch, chunk):
    """A sliding window of 700 over a 1100-token prompt (chunks of 512, 512, 76, or one pass with the
    default chunk): from position 700 on, the first keys a row may attend are in an earlier chunk, so
    the window start of the batched attention is checked against keys other chunks stored (Mistral:
    every layer windowed; Gemma-2: the even layer, with softcaps). Logits, K/V rows on both sides of
    the edge and the greedy tokens after it against the oracle."""
    from dotnetfoundryllm_amd.configs import _cfg, _types
    if arch == N.ARCH_MISTRAL:
        cfg = _cfg("window-mistral", arch, 2, 256, 4, 2, 512, 512, 1200, 10000.0, _types(*([N.Q8_0] * 8)),
                   window=700, norm_std=0.1, seed=24)
    else:
        cfg = _cfg("window-gemma2", arch, 2, 256, 4, 2, 512, 512, 1200, 10000.0, _types(*([N.Q8_0] * 8)),
                   head_dim=128, emb_type=N.BF16, window=700, attn_softcap=50.0, final_softcap=30.0,
                   norm_std=0.1, seed=25)
    desc = desc_of(cfg)
    tensors = {e[0]: (e, synth_bytes(cfg, e)) for e in tensor_plan(cfg)}
    m = device_model(ctx, desc, tensors)
    kv = F.HipKvCache(m)
    fwd = F.HipForwardPass(m)
    orc = O.OracleModel(desc, tensors)
    prompt = F.synth_tokens(cfg["seed"], 3, desc.vocab, 1100)
    try:
        if chunk:
            F.set_prefill_chunk(kv, chunk)
        fwd.prefill(prompt, 0, kv)
        _oracle_prefill(orc, prompt)
        assert kv.current_length == 1100
        assert O.normwise_rel_err(fwd.logits, orc.logits()) <= TOL
        kvdim = desc.n_kv_heads * desc.head_dim
        for l in range(desc.n_layers):
            k, v = kv.get_keys(l), kv.get_values(l)
            kr, vr = orc.kv(l, 0), orc.kv(l, 1)
            assert O.normwise_rel_err(k, kr) <= TOL and O.normwise_rel_err(v, vr) <= TOL
            for pos in (0, 511, 512, 699, 700, 701, 1023, 1024, 1099):
                row = slice(pos * kvdim, (pos + 1) * kvdim)
                assert O.normwise_rel_err(k[row], kr[row]) <= TOL, (l, pos)
                assert O.normwise_rel_err(v[row], vr[row]) <= TOL, (l, pos)
        toks = fwd.decode_greedy(int(prompt[-1]), 1100, 6, kv)
        assert list(toks) == _oracle_continue(orc, prompt[-1], 1100, 6)
    finally:
        orc.close()
        kv.close()
        m.close()


def test_batched_prefill_llama3_8b_shape(ctx):
    """Full Llama-3-8B shapes (Q4_K + Q6_K, tile-interleaved weights), two layers, a 24-token
    prompt: logits, K/V and the next greedy tokens against the oracle."""
    cfg, desc, tensors = synthetic("llama3-8b-q4km", n_layers=2)
    m = device_model(ctx, desc, tensors)
    kv = F.HipKvCache(m, 64)
    fwd = F.HipForwardPass(m)
    orc = O.OracleModel(desc, tensors, 64)
    prompt = F.synth_tokens(cfg["seed"], 4, desc.vocab, 24)
    try:
        fwd.prefill(prompt, 0, kv)
        _oracle_prefill(orc, prompt)
        err = O.normwise_rel_err(fwd.logits, orc.logits())
        print(f"logits normwise rel err {err:.2e}")
        assert err <= TOL
        for l in range(desc.n_layers):
            assert O.normwise_rel_err(kv.get_keys(l), orc.kv(l, 0)) <= TOL
            assert O.normwise_rel_err(kv.get_values(l), orc.kv(l, 1)) <= TOL
        toks = fwd.decode_greedy(int(prompt[-1]), 24, 3, kv)
        assert list(toks) == _oracle_continue(orc, prompt[-1], 24, 3)
    finally:
        orc.close()
        kv.close()
        m.close()


def test_prefill_argument_contract(ctx):
    """Out-of-range tokens and a prompt beyond the cache fail before anything runs; a prompt that
    does not continue the cache takes the per-token path with the Forward checks."""
    cfg, desc, tensors = synthetic("test-llama")
    m = device_model(ctx, desc, tensors)
    kv = F.HipKvCache(m, 16)
    fwd = F.HipForwardPass(m)
    try:
        with pytest.raises(F.ArgumentOutOfRangeException):
            fwd.prefill(np.array([1, desc.vocab, 2], dtype=np.int32), 0, kv)
        assert kv.current_length == 0
        with pytest.raises(F.ArgumentOutOfRangeException):
            fwd.prefill(np.arange(17, dtype=np.int32), 0, kv)
        assert kv.current_length == 0
        fwd.prefill(np.arange(16, dtype=np.int32), 0, kv)
        assert kv.current_length == 16
        with pytest.raises(F.ArgumentOutOfRangeException):
            fwd.prefill(np.array([1, 2], dtype=np.int32), 16, kv)  # cache full
    finally:
        kv.close()
        m.close()


@pytest.mark.parametrize("types,hidden", [
    ("q4_k", 512), ("q5_k", 512), ("q6_k", 512), ("q8_0", 512), ("q5_k q8_0 q6_k q4_k q4_k q6_k q5_k", 512),
    ("q4_k", 2304), ("q5_k", 2304), ("q6_k", 2304), ("q8_0", 2304), ("q4_0", 512), ("f16", 512), ("q4_0", 352)],
    ids=["q4_k", "q5_k", "q6_k", "q8_0", "mixed", "q4_k-rows", "q5_k-rows", "q6_k-rows", "q8_0-rows", "q4_0", "f16",
         "q4_0-352"])
def test_prefill_gemm_tile_edges(ctx, types, hidden):
    """The large-tile GEMMs at the edges of the tiles of 64 tokens x 256 weight rows: 2 to
    200 tokens on 128-, 512- and 768-row matrices (at most 24 such tiles: never the ones of 128 tokens), every tile-interleaved type alone, launches that mix
    them, and GGUF rows (2304 = 9 blocks has no tile layout, Q4_0 and F16 none at all; 352 is no whole
    number of blocks and stays on the general row kernel). K / V rows of both layers (the second
    layer's carry every GEMM of the first) against the oracle. Bound: operands of 22 bits or more and
    f32 sums of at most 2304 products, 2^-22 + sqrt(2304) 2^-24 (3e-6) for a projection, five of them
    in a row: 1.5e-5; a third more. The softmax multiplies a score's relative error by the score, and
    these seeded weights make scores q k of about 5e4 (|q|, |k| about 27 over 64 elements): Gemma-2's
    own attention scale, here 1e-5, keeps the scores below 1 and the bound that of the GEMMs. It is
    the median row's; a row whose sums nearly cancel (the seeded weights are not zero-mean) has the
    file's bar."""
    name_of = {"q4_k": N.Q4_K, "q5_k": N.Q5_K, "q6_k": N.Q6_K, "q8_0": N.Q8_0, "q4_0": N.Q4_0, "f16": N.F16}
    t = [name_of[x] for x in types.split()]
    t = t * 7 if len(t) == 1 else t
    cfg = dict(CONFIGS["test-gemma2"], n_layers=2, hidden=hidden, n_heads=8, n_kv_heads=2, head_dim=64, ffn=768, max_ctx=256,
               window=0x7FFFFFFF,
               types=dict(zip(("q", "k", "v", "o", "gate", "up", "down", "out"), t + [t[0]])))
    desc = desc_of(cfg)
    desc.attn_scale = 1e-5
    tensors = {e[0]: (e, synth_bytes(cfg, e)) for e in tensor_plan(cfg)}
    m = device_model(ctx, desc, tensors)
    kv, fwd = F.HipKvCache(m), F.HipForwardPass(m)
    orc = O.OracleModel(desc, tensors)
    prompt = F.synth_tokens(cfg["seed"], 9, desc.vocab, 200)
    try:
        _oracle_prefill(orc, prompt)
        for n in (2, 33, 64, 65, 128, 129, 200):
            kv.clear()
            fwd.prefill(prompt[:n], 0, kv)
            for l in range(desc.n_layers):
                for kind, get in ((0, kv.get_keys), (1, kv.get_values)):
                    got, want = get(l), orc.kv(l, kind)
                    got = np.asarray(got, dtype=np.float64).reshape(n, -1)
                    want = np.asarray(want, dtype=np.float64).reshape(-1)[:got.size].reshape(n, -1)
                    err = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
                    assert np.median(err) <= 2e-5 and err.max() <= TOL, (n, l, kind, err.max())
        assert O.normwise_rel_err(fwd.logits, orc.logits()) <= TOL
    finally:
        orc.close()
        kv.close()
        m.close()


@pytest.mark.parametrize("top", [1e-5, 1.0, 4e3, 4e6])
@pytest.mark.parametrize("q,v,hidden", [(N.Q4_K, N.Q4_K, 512), (N.Q5_K, N.Q5_K, 512), (N.Q8_0, N.Q5_K, 512),
                                        (N.Q4_K, N.Q4_K, 2304), (N.Q5_K, N.Q5_K, 2304)],
                         ids=["q4_k", "q5_k", "mixed", "q4_k-rows", "q5_k-rows"])
def test_prefill_kquant_offset_magnitudes(ctx, q, v, hidden, top):
    """V of a Q4_K / Q5_K matrix whose largest offset dmin m is `top`: from near the smallest half to near
    the largest (the offsets enter the matrix cores as two halves). Bound against float64: operands of 22
    bits and f32 sums of `hidden` products, 2^-22 + sqrt(hidden) 2^-24."""
    cfg = dict(CONFIGS["test-llama"], n_layers=1, hidden=hidden, n_heads=8, n_kv_heads=2, head_dim=64, ffn=256, max_ctx=128,
               types=dict(zip(("q", "k", "v", "o", "gate", "up", "down", "out"), [q, q, v] + [N.Q4_K] * 5)))
    desc = desc_of(cfg)
    tensors = {e[0]: (e, synth_bytes(cfg, e)) for e in tensor_plan(cfg)}
    entry, data = tensors["blk.0.attn_v.weight"]
    blocks = data.copy().reshape(-1, N.BLOCK[v][0])
    mid = 7.5 if v == N.Q4_K else 15.5
    d, dmin = np.float16(top / 63 / mid), np.float16(top / 63)  # at 1e-5 d is 0: the offsets alone
    blocks[:, :4] = np.array([d, dmin]).view(np.uint8)
    tensors["blk.0.attn_v.weight"] = (entry, blocks.reshape(-1))
    m = device_model(ctx, desc, tensors)
    kv, fwd = F.HipKvCache(m), F.HipForwardPass(m)
    prompt = F.synth_tokens(cfg["seed"], 11, desc.vocab, 70)
    try:
        fwd.prefill(prompt, 0, kv)
        x = f32_of(tensors, "token_embd.weight").astype(np.float64).reshape(-1, hidden)[prompt]
        x = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-5) * f32_of(tensors, "blk.0.attn_norm.weight")
        want = x @ f32_of(tensors, "blk.0.attn_v.weight").astype(np.float64).reshape(-1, hidden).T
        got = np.asarray(kv.get_values(0), dtype=np.float64).reshape(want.shape)
        assert np.linalg.norm(got - want) / np.linalg.norm(want) <= 2.0**-22 + np.sqrt(hidden) * 2.0**-24
    finally:
        kv.close()
        m.close()


@pytest.mark.parametrize("t,hidden", [(N.Q4_K, 2048), (N.Q5_K, 2048), (N.Q6_K, 2048), (N.Q8_0, 2048), (N.Q4_K, 2304),
                                      (N.Q5_K, 2304), (N.Q6_K, 2304), (N.Q8_0, 2304), (N.Q4_0, 2048)],
                         ids=["q4_k", "q5_k", "q6_k", "q8_0", "q4_k-rows", "q5_k-rows", "q6_k-rows", "q8_0-rows", "q4_0"])
def test_prefill_gemm_rounds_without_bias(ctx, t, hidden):
    """The mean signed error of V over 200 tokens x 512 rows, against float64. The matrix cores round sums down,
    which blocks of alternating sign cancel (an odd ninth of 2304 columns is left): -4e-8 of the result's root
    mean square without that (Q8_0). The rest is the mean of 102400 roundings of about 3e-7
    (1e-9), and each token's rounded norm (6e-8 of the tokens' common mean, at most 2e-2 of the root mean
    square): 6e-9 allowed."""
    cfg = dict(CONFIGS["test-llama"], n_layers=1, hidden=hidden, n_heads=8, n_kv_heads=8, head_dim=64, ffn=256, max_ctx=256,
               vocab=512, types={k: t for k in ("q", "k", "v", "o", "gate", "up", "down", "out")})
    desc = desc_of(cfg)
    tensors = {e[0]: (e, synth_bytes(cfg, e)) for e in tensor_plan(cfg)}
    m = device_model(ctx, desc, tensors)
    kv, fwd = F.HipKvCache(m), F.HipForwardPass(m)
    prompt = F.synth_tokens(3, 11, desc.vocab, 200)
    try:
        fwd.prefill(prompt, 0, kv)
        x = f32_of(tensors, "token_embd.weight").astype(np.float64).reshape(-1, hidden)[prompt]
        x = x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-5) * f32_of(tensors, "blk.0.attn_norm.weight")
        want = x @ f32_of(tensors, "blk.0.attn_v.weight").astype(np.float64).reshape(-1, hidden).T
        got = np.asarray(kv.get_values(0), dtype=np.float64).reshape(want.shape)
        assert abs(np.mean(got - want)) <= 6e-9 * np.sqrt(np.mean(want * want))
    finally:
        kv.close()
        m.close()


@pytest.mark.parametrize("gate,up,hidden,ffn,lengths", [
    ("q4_k", "q4_k", 512, 8480, (193, 256, 257, 300)), ("q5_k", "q5_k", 512, 8480, (193, 257)),
    ("q6_k", "q6_k", 512, 8480, (193, 257)), ("q8_0", "q8_0", 512, 8480, (193, 257)),
    ("q5_k", "q8_0", 512, 8480, (193, 257)), ("q8_0", "q4_k", 512, 8480, (193, 257)), ("q6_k", "q5_k", 512, 8480, (193, 257)),
    ("q4_k", "q4_k", 2304, 8480, (193, 257)), ("q5_k", "q5_k", 2304, 8480, (193, 257)),
    ("q6_k", "q6_k", 2304, 8480, (193, 257)), ("q8_0", "q8_0", 2304, 8480, (193, 257)),
    ("q4_0", "q4_0", 512, 8480, (193, 256, 257, 300)), ("f16", "f16", 512, 8480, (193, 257)),
    ("q4_k", "q4_k", 8192, 8192, (256,)), ("q4_0", "q4_0", 5632, 8192, (256,))],
    ids=["q4_k", "q5_k", "q6_k", "q8_0", "q5_k+q8_0", "q8_0+q4_k", "q6_k+q5_k", "q4_k-rows", "q5_k-rows", "q6_k-rows",
         "q8_0-rows", "q4_0", "f16", "q4_k-split", "q4_0-split"])
def test_prefill_gemm_tiles_of_128_tokens(ctx, gate, up, hidden, ffn, lengths):
    """Gate / up launches that take the tiles of 128 tokens x 256 rows by the modelled time: 2 x 8480 rows are
    68 column tiles, 193 to 256 tokens then 272 tiles of 64 tokens (two waves of 256) or 136 of 128 (one), 257
    to 300 tokens 340 or 204; a last tile of one token, of 65, of 44 and a full one, 32 rows in each segment's
    last tile. 2 x 8192 rows of 22 or 32 blocks over 256 tokens run in two parts of K. Each form alone and mixed.
    The output projection is zero, so V of the second layer is a function of the first layer's FFN. Bound
    against float64: three projections of operands of 22 bits and f32 sums of at most 8480 products,
    3 (2^-22 + sqrt(8480) 2^-24)."""
    name_of = {"q4_k": N.Q4_K, "q5_k": N.Q5_K, "q6_k": N.Q6_K, "q8_0": N.Q8_0, "q4_0": N.Q4_0, "f16": N.F16}
    cfg = dict(CONFIGS["test-llama"], n_layers=2, hidden=hidden, n_heads=4, n_kv_heads=2, head_dim=64, ffn=ffn, max_ctx=320,
               vocab=512, types=dict(zip(("q", "k", "v", "o", "gate", "up", "down", "out"),
                                         [N.Q8_0] * 4 + [name_of[gate], name_of[up]] + [N.Q8_0] * 2)))
    desc = desc_of(cfg)
    tensors = {e[0]: (e, synth_bytes(cfg, e)) for e in tensor_plan(cfg)}
    for l in range(2):
        e, data = tensors[f"blk.{l}.attn_output.weight"]
        tensors[f"blk.{l}.attn_output.weight"] = (e, np.zeros_like(data))

    def mul(x, name):
        return x @ f32_of(tensors, name).astype(np.float64).reshape(-1, x.shape[1]).T

    def norm(x, name):
        return x / np.sqrt(np.mean(x * x, axis=1, keepdims=True) + 1e-5) * f32_of(tensors, name)

    m = device_model(ctx, desc, tensors)
    kv, fwd = F.HipKvCache(m), F.HipForwardPass(m)
    prompt = F.synth_tokens(cfg["seed"], 7, desc.vocab, max(lengths))
    try:
        x = f32_of(tensors, "token_embd.weight").astype(np.float64).reshape(-1, hidden)[prompt]
        xn = norm(x, "blk.0.ffn_norm.weight")
        g = mul(xn, "blk.0.ffn_gate.weight")
        x = x + mul(g / (1.0 + np.exp(-np.clip(g, -700, 700))) * mul(xn, "blk.0.ffn_up.weight"), "blk.0.ffn_down.weight")
        want = mul(norm(x, "blk.1.attn_norm.weight"), "blk.1.attn_v.weight")
        for n in lengths:
            kv.clear()
            fwd.prefill(prompt[:n], 0, kv)
            got = np.asarray(kv.get_values(1), dtype=np.float64).reshape(n, -1)
            err = np.linalg.norm(got - want[:n], axis=1) / np.linalg.norm(want[:n], axis=1)
            assert err.max() <= 3 * (2.0**-22 + np.sqrt(8480) * 2.0**-24), (n, int(err.argmax()), err.max())
    finally:
        kv.close()
        m.close()
