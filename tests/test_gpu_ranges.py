"""Operands of very different magnitudes beside each other, which pairs of f16 values cannot hold with one exponent: what a row does not
see must not cost it bits, and small values count where the large ones are multiplied by nothing.

Tolerance: 2e-5 of the largest output of the row (attention; the suite's bound) and of the row of logits (products), each row
by itself, at any factor."""
import numpy as np
import pytest

from lumen_amd._lib import check, lib
from lumen_amd.autograd import Tensor
from lumen_amd.layers import KVCacheInner, RotaryEmbedding
from oracle import lumen_oracle as lo
from tests.gpu_util import dev

pytestmark = pytest.mark.gpu


def attention_rows(d, h, h_kv, past, s, change, causal=True, batch=1):
    """(rows of this call from the GPU, from the oracle) after change(q, k, v) of the values of all past + s positions"""
    rng = np.random.default_rng(d + s)
    n = past + s
    q = rng.normal(0, 1, (batch, n, h, d)).astype(np.float32)
    k, v = (rng.normal(0, 1, (batch, n, h_kv, d)).astype(np.float32) for _ in range(2))
    change(q, k, v)
    rope, scale = RotaryEmbedding(d, 512, 10000.0), d ** -0.5
    cos, sin = lo.rope_table(d, 512, 10000.0)
    gpu, ora = KVCacheInner(batch, h_kv, 512, d), lo.KVCache(batch, h_kv, 512, d)
    for at, m in ((0, past), (past, s)):
        if not m:
            continue
        part = [np.ascontiguousarray(x[:, at:at + m]) for x in (q, k, v)]
        dev_part, out = [dev(x) for x in part], Tensor.empty(part[0].shape)
        check(lib.lumen_attn_prefill_f32(gpu.handle, rope.handle, *(x.ptr for x in dev_part), out.ptr, m, h, scale, int(causal)))
        got = out.data()
        rc, ref = lo.attn_prefill(ora, *part, cos, sin, scale, causal=causal)
        assert rc == lo.LO_OK
    return got, ref


def row_error(got, ref):
    return (np.abs(got - ref).max(-1) / np.maximum(np.abs(ref).max(-1), 1e-30)).max()


def later(what, first, e):
    def change(q, k, v):
        (k if what == "k" else v)[:, first:] *= np.float32(2.0 ** e)
    return change


@pytest.mark.parametrize("e", [12, 16, 18, 20, 24, 30, 40, 100])
@pytest.mark.parametrize("what", ["k", "v"])
@pytest.mark.parametrize("d,h,h_kv,past,s", [(64, 4, 1, 0, 96), (128, 2, 2, 0, 97), (64, 8, 1, 301, 99)])
def test_attention_rows_before_a_large_key_or_value(d, h, h_kv, past, s, what, e):
    """The last position only, and all from one inside a tile on."""
    for first in (past + s - 1, past + 37):
        got, ref = attention_rows(d, h, h_kv, past, s, later(what, first, e))
        assert row_error(got[:, :first - past], ref[:, :first - past]) <= 2e-5, first


@pytest.mark.parametrize("e", [-40, -24, -18, 24, 40])
@pytest.mark.parametrize("d,h,h_kv,past,s", [(64, 4, 2, 0, 130), (128, 4, 1, 400, 20)])
def test_attention_channels_of_other_magnitudes(d, h, h_kv, past, s, e):
    """Half of the value channels, each held to its own largest output; a rotated pair of channels of the queries, to which the keys are zero;
    one head's values beside the others'."""
    f = np.float32(2.0 ** e)

    def values(q, k, v):
        v[..., ::2] *= f
    got, ref = attention_rows(d, h, h_kv, past, s, values)
    for part in (slice(0, None, 2), slice(1, None, 2)):
        assert row_error(got[..., part], ref[..., part]) <= 2e-5

    def queries(q, k, v):
        for c in (5, 5 + d // 2):
            q[..., c] *= f
            k[..., c] = 0
    assert row_error(*attention_rows(d, h, h_kv, past, s, queries)) <= 2e-5

    def head(q, k, v):
        v[:, :, 0] *= f
    assert row_error(*attention_rows(d, h, h_kv, past, s, head)) <= 2e-5


@pytest.mark.parametrize("d,h,h_kv,past,s,batch", [(64, 4, 2, 0, 96, 2), (128, 3, 1, 300, 5, 1), (64, 2, 2, 130, 140, 1), (64, 8, 2, 448, 3, 2)])
def test_attention_without_a_mask(d, h, h_kv, past, s, batch):
    """All keys for every position, keys in parts and in one, also with tiles that lie far apart in magnitude."""
    for change in (lambda q, k, v: None, later("v", past + s - 20, -30), later("v", past + s - 20, 30)):
        assert row_error(*attention_rows(d, h, h_kv, past, s, change, causal=False, batch=batch)) <= 2e-5
