"""Prompts read without logits (logits_out NULL: no LM head) leave the same
cache as prompts read with them: the K/V rows are equal bit for bit and the
next token's logits too. Both the multi-row forward (up to 32 rows) and the
prefill kernels, f32 and bf16, and generation, whose prefill computes the last
rows' logits only, against the argmax of every row's."""
import numpy as np
import pytest

from rusttorch_amd import synth
from rusttorch_amd.gpt2 import Gpt2Config, Gpt2Model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("batch,chunks", [(1, (5, 27)), (4, (8, 1)), (1, (33, 2, 140)), (3, (70,)), (20, (19,))])
def test_cache_is_the_same(storage, batch, chunks):
    sh = synth.ModelShape(515, 256, 768, 2, 12)
    cfg = Gpt2Config(sh.vocab_size, sh.n_positions, sh.n_embd, sh.n_layer, sh.n_head, sh.layer_norm_epsilon)
    m = Gpt2Model.from_state_dict(synth.make_weights(sh, bf16=storage == "bf16"), cfg, storage=storage)
    total = sum(chunks)
    ids = np.stack([synth.make_tokens(total + 1, sh.vocab_size, stream=70 + b) for b in range(batch)])
    a, b = m.new_cache(batch), m.new_cache(batch)
    print(f"[gpu] no logits {storage} batch {batch} chunks {chunks}", flush=True)
    at = 0
    for n in chunks:
        last = m.forward_cached_batched(ids[:, at:at + n], a)[:, -1]
        assert m.forward_cached_batched(ids[:, at:at + n], b, want_logits=False) is None
        at += n
        assert a.len() == b.len() == at
    for layer in range(sh.n_layer):
        for seq in {0, batch - 1}:
            for values in (False, True):
                assert np.array_equal(a.read(layer, 3, seq, values), b.read(layer, 3, seq, values))
    nxt = ids[:, total:total + 1]
    assert np.array_equal(m.forward_cached_batched(nxt, a), m.forward_cached_batched(nxt, b))
    if len(chunks) == 1:
        first = m.generate_cached_batched(ids[:, :total], 1)[:, -1]
        top = np.sort(last, axis=-1)
        clear = top[:, -1] - top[:, -2] > 1e-4  # (rows without a near tie; the two runs' sums differ in order)
        assert np.array_equal(first[clear], np.argmax(last, axis=-1)[clear])
    a.close()
    b.close()
    m.close()
