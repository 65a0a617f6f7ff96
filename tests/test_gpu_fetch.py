"""GPU check of the results a model call brings to the host: around the size up to which they travel through pinned memory (2^18 - 1 words),
with and without logits, ids of one and several steps, and the position a prompt leaves for the next token."""
import pytest

from lumen_amd import synth
from lumen_amd.models import LlamaModel
from oracle import lumen_oracle as lo
from tests.gpu_util import max_rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab,rows", [(87381, 3), (65536, 4), (131072, 2), (257, 2)])
def test_logits_and_ids_around_the_pinned_size(vocab, rows):
    cfg = dict(vocab_size=vocab, hidden_size=64, intermediate_size=64, num_hidden_layers=1, num_attention_heads=4, num_key_value_heads=2,
               rms_norm_eps=1e-5, max_seq_len=32, rope_theta=10000.0)
    params = synth.make_params(cfg, seed=3, std=0.1, gains_one=False)
    gpu, ora = LlamaModel(cfg), lo.Llama(cfg, params)
    for n, a in params.items():
        gpu.set_param(n, a)
    ids = synth.make_tokens(rows, vocab, seed=1)
    rc, ref = ora.forward(ids)
    assert rc == lo.LO_OK
    assert max_rel(gpu.forward(ids, all_rows=True), ref) <= 1e-4
    first = int(ref[-1].argmax())
    one = gpu.forward([first], all_rows=True)  # one token, at the position the prompt left
    rc, ref = ora.forward([first])
    assert rc == lo.LO_OK and max_rel(one, ref) <= 1e-4
    tok = int(ref[-1].argmax())
    got = [int(t) for t in gpu.decode_greedy(tok, 1)] + [int(t) for t in gpu.decode_greedy(tok, 3)]
    want = []
    for n in (1, 3):
        t = tok
        for _ in range(n):
            rc, ref = ora.forward([t])
            assert rc == lo.LO_OK
            t = int(ref[-1].argmax())
            want.append(t)
    assert got == want
