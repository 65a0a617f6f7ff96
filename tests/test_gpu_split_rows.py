"""GPU parity of the prompt products that run on f16 pairs (prompts of more than 32 rows, 47 with bf16-stored weights, and of few rows, three to
32 with bf16-stored weights and 17 to 32 with f32 ones; inner sizes that are multiples of 64): row and column counts around the tiles' edges, one piece of K and many, rows of very different
magnitudes, rows of zeros and rows that are not finite, against the CPU oracle.

Tolerance: the suite's 1e-4 of the largest logit for f32 weights, and the same for bf16-stored ones, whose values the oracle
holds too (the pairs carry 2^-22 of a product; sums of up to 3000 f32 terms 3e-7)."""
import numpy as np
import pytest

from lumen_amd import synth
from lumen_amd.layers import KVCacheInner, RotaryEmbedding
from lumen_amd.models import LlamaModel
from oracle import lumen_oracle as lo
from tests import hybrid_util, nufapel_util
from tests.gpu_util import max_rel
from tests.test_gpu_attention import gpu_prefill

pytestmark = pytest.mark.gpu


def config(hidden, inter, heads, kv_heads, layers=2, vocab=301, max_seq=320):
    return dict(vocab_size=vocab, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=layers, num_attention_heads=heads,
                num_key_value_heads=kv_heads, rms_norm_eps=1e-5, max_seq_len=max_seq, rope_theta=10000.0)


def build(cfg, bf16, change=None):
    params = synth.make_params(cfg, seed=3, std=0.1, gains_one=False)
    if change:
        change(params, np.random.default_rng(7))
    gcfg, bits = dict(cfg), {}
    if bf16:
        gcfg["weight_dtype"] = "bf16"
        bits = {n: synth.bf16_round(a).reshape(a.shape) for n, a in params.items() if a.ndim == 2}
        params = {n: synth.bf16_widen(bits[n]) if n in bits else a for n, a in params.items()}
    gpu = LlamaModel(gcfg)
    for n, a in params.items():
        gpu.set_param(n, bits.get(n, a))
    return gpu, lo.Llama(cfg, params)


def magnitudes(params, rng):
    """Tokens, and rows of the matrices that write the residual stream, spread over many powers of two; a row of zeros."""
    for n, a in params.items():
        if "embed" in n:
            a *= np.exp2(rng.integers(-20, 20, (len(a), 1))).astype(np.float32)
        elif "o_proj" in n or "down_proj" in n:
            a *= np.exp2(rng.integers(-30, 6, (len(a), 1))).astype(np.float32)
            a[5] = 0


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("cfg,rows", [
    (config(64, 64, 4, 2), (3, 17, 32)),                       # two blocks of K: half a chunk
    (config(128, 192, 4, 1, vocab=257), (4, 16, 19)),          # columns that fill no tile
    (config(320, 704, 5, 5), (3, 16, 17, 31)),                 # chunks of K that end early, K splits
    (config(1024, 2824, 16, 4, layers=1), (3, 15, 18, 32)),    # (f32 weights: from 5 Mi of them on)
    (config(64, 64, 4, 2, layers=1, vocab=81925), (17, 32)),
], ids=["64", "128", "320", "1024", "vocab"])
def test_prompts_of_few_rows(cfg, rows, bf16):
    gpu, ora = build(cfg, bf16, magnitudes)
    for s in rows:
        ids = synth.make_tokens(s, cfg["vocab_size"], seed=s)
        gpu.reset_kv_caches()
        ora.reset()
        got = gpu.forward(ids, all_rows=True)
        rc, ref = ora.forward(ids)
        assert rc == lo.LO_OK
        for t in range(s):
            assert max_rel(got[t], ref[t]) <= 1e-4, (s, t)


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
@pytest.mark.parametrize("cfg,rows", [
    (config(64, 64, 4, 2), (33, 64)),                  # one piece of K
    (config(128, 192, 4, 1, vocab=257), (127, 128, 129)),
    (config(320, 704, 5, 5), (255, 257, 300)),         # columns that fill no tile, several pieces, K splits
    (config(256, 320, 2, 1), (96, 161)),               # heads of 128
    (config(1024, 2816, 16, 4, layers=1, max_seq=1152), (1101,)),  # many tiles of 128
    # 256 x 256 tiles: gate|up (32000 columns) and head (32001), whole K, four rows of tiles of which the last holds 132
    (config(128, 16000, 2, 1, layers=1, vocab=32001, max_seq=1024), (900,)),
    (config(1024, 16384, 16, 4, layers=1, max_seq=1024), (897,)),  # ... and K in 16: down (16384 inner values)
], ids=["64", "128", "320", "256", "1024", "wide", "deep"])
def test_prompts_at_the_edges_of_tiles(cfg, rows, bf16):
    gpu, ora = build(cfg, bf16)
    for s in rows:
        ids = synth.make_tokens(s, cfg["vocab_size"], seed=s)
        gpu.reset_kv_caches()
        ora.reset()
        got = gpu.forward(ids, all_rows=True)
        rc, ref = ora.forward(ids)
        assert rc == lo.LO_OK
        assert max_rel(got, ref) <= 1e-4
        gpu.reset_kv_caches()
        last = gpu.forward(ids, all_rows=False)
        assert max_rel(last, ref[-1]) <= 1e-4


@pytest.mark.parametrize("bf16", [False, True], ids=["f32", "bf16"])
def test_rows_of_very_different_magnitudes(bf16):
    cfg = config(192, 320, 6, 3)
    gpu, ora = build(cfg, bf16, magnitudes)
    ids = synth.make_tokens(150, cfg["vocab_size"], seed=1)
    got = gpu.forward(ids, all_rows=True)
    rc, ref = ora.forward(ids)
    assert rc == lo.LO_OK
    for t in range(len(ids)):  # every row by itself: rows of small logits have to be right too
        assert max_rel(got[t], ref[t]) <= 1e-4, t


def test_a_token_that_is_not_finite_stays_in_its_row():
    cfg = config(128, 192, 4, 2)
    for bad in (np.inf, np.nan):
        def change(params, rng):
            params["model.embed_tokens.weight"][7, 3] = bad
        gpu, ora = build(cfg, False, change)
        ids = synth.make_tokens(90, cfg["vocab_size"], seed=2)
        ids[ids == 7] = 8
        ids[-1] = 7  # (the last: no other token sees it)
        got = gpu.forward(ids, all_rows=True)
        _, ref = ora.forward(ids[:-1])
        assert not np.isfinite(got[-1]).any()
        assert max_rel(got[:-1], ref) <= 1e-4


@pytest.mark.parametrize("d,h,h_kv,s,past", [(64, 8, 1, 96, 0), (64, 6, 2, 129, 70), (128, 4, 4, 97, 0), (128, 4, 2, 200, 33), (64, 2, 2, 127, 1),
                                                (128, 4, 2, 40, 461), (64, 8, 1, 97, 300), (128, 3, 1, 2, 510),  # keys in parts
                                                (128, 4, 4, 97, 403), (128, 4, 2, 200, 300), (128, 6, 2, 129, 371), (128, 8, 1, 64, 440)])
@pytest.mark.parametrize("q_exp,k_exp,v_exp", [(0, 0, 0), (-90, 88, -100), (60, -61, 90)])
def test_prompt_attention_over_magnitudes(d, h, h_kv, s, past, q_exp, k_exp, v_exp):
    """Queries, keys and values far from 1, and keys and values spread over 2^8 within a head (2e-5 of the largest output, the suite's bound for
    attention: scores of a few units, so that a relative error of 2^-22 of the terms of a score moves a weight by 1e-6)."""
    rng = np.random.default_rng(s + d)

    def draw(n, heads, e):
        spread = np.exp2(rng.uniform(-8, 0, (1, n, heads, 1)))
        return (rng.normal(0, 1, (1, n, heads, d)) * spread * 2.0 ** e).astype(np.float32)
    rope, scale = RotaryEmbedding(d, 512, 10000.0), d ** -0.5 * 4.0
    cos, sin = lo.rope_table(d, 512, 10000.0)
    gpu, ora = KVCacheInner(1, h_kv, 512, d), lo.KVCache(1, h_kv, 512, d)
    for n in (past, s):
        if not n:
            continue
        q, k, v = draw(n, h, q_exp), draw(n, h_kv, k_exp), draw(n, h_kv, v_exp)
        got = gpu_prefill(gpu, rope, q, k, v, scale)
        rc, ref = lo.attn_prefill(ora, q, k, v, cos, sin, scale)
        assert rc == lo.LO_OK
    assert max_rel(got * 2.0 ** -v_exp, ref * 2.0 ** -v_exp) <= 2e-5


HYBRIDS = {
    "pinavik": lambda: (hybrid_util, hybrid_util.config(1024, 307, [
        hybrid_util.attention(4, 2, 32, 32, 50, ff=320), hybrid_util.wkv(4, 32, ff=100), hybrid_util.delta(2, 1, 64, 32, ff=192),
        hybrid_util.wkv(2, 64)], loop=(1, 3, 2))),
    "nufapel": lambda: (nufapel_util, nufapel_util.config(1024, 307, [
        nufapel_util.parallel((4, 2, 32, 32), (2, 64, 64), nufapel_util.dense(320)), nufapel_util.general(4, 32, nufapel_util.dense(100))], loop=(0, 2, 2))),
}


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("name,tokens", [("pinavik", 193), ("pinavik", 320), ("nufapel", 449)])
def test_hybrid_prompt_at_once_and_in_portions(tmp_path, name, tokens, dtype):
    """Portions of 60 tokens run on f32 rows (their rows times the width are below what split rows are taken for), the prompt at once on split
    ones; sums of up to 1024 terms in another order, over a few layers: 2e-5 of the largest logit, as for other cuts of a prompt."""
    util, cfg = HYBRIDS[name]()
    model = hybrid_util.load(tmp_path, cfg, util.make_params(cfg, seed=4), dtype)
    ids = synth.make_tokens(tokens, 307, seed=tokens)
    at_once, portions = (hybrid_util.run(model, ids, cuts) for cuts in ([tokens], [60]))
    assert max_rel(at_once, portions) <= 2e-5
    assert not np.array_equal(at_once, portions)  # (else both ran on the same kernels)
