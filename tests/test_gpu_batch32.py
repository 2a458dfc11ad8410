"""The batched decode step with 17 to 32 sequences (two blocks of 16 rows per
GEMV), through forward_cached with one token per sequence, against the CPU
oracle sequence by sequence at the logits bar, and greedy generation of the
batch against the sequences run alone."""
import os

import numpy as np
import pytest

from rusttorch_amd import synth
from rusttorch_amd.gpt2 import Gpt2Config, Gpt2Model

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


def build(sh, storage):
    sd = synth.make_weights(sh, bf16=storage == "bf16")
    cfg = Gpt2Config(sh.vocab_size, sh.n_positions, sh.n_embd, sh.n_layer, sh.n_head, sh.layer_norm_epsilon)
    return sd, Gpt2Model.from_state_dict(sd, cfg, storage=storage)


@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("d,heads,V,batch", [(128, 2, 301, 17), (768, 12, 515, 24), (768, 12, 50257, 31),
                                             (1600, 25, 258, 32)])
def test_decode_logits(oracle_lib, storage, d, heads, V, batch):
    sh = synth.ModelShape(V, 64, d, 2, heads)
    sd, m = build(sh, storage)
    om = oracle_lib.OracleModel.from_shape(sd, sh, threads=THREADS)
    ids = np.stack([synth.make_tokens(7 + 3, V, stream=300 + b) for b in range(batch)])
    print(f"[gpu] batch {batch} {sh} {storage}", flush=True)
    c = m.new_cache(batch)
    m.forward_cached_batched(ids[:, :7], c, want_logits=False)
    got = np.stack([m.forward_cached_batched(ids[:, t:t + 1], c)[:, 0] for t in range(7, 10)], axis=1)
    for b in (0, 15, 16, batch - 1):
        ref = om.forward(ids[b])[7:]
        worst = np.max(np.abs(got[b] - ref) - (1e-3 + 1e-4 * np.abs(ref)))
        assert worst <= 0, (b, worst)
        assert np.max(np.abs(got[b] - ref)) < 5e-5  # what f32 sums of this depth give, as the steps up to 16 do
    c.close()
    m.close()


def test_generation_equals_single_sequences():
    sh = synth.ModelShape(515, 64, 768, 2, 12)
    _, m = build(sh, "f32")
    prompts = np.stack([synth.make_tokens(9, 515, stream=500 + b) for b in range(27)])
    out = m.generate_cached_batched(prompts, 20)
    for b in range(0, 27, 2):
        assert out[b].tolist() == m.generate_cached(prompts[b], 20, 0.0), b
    m.close()
