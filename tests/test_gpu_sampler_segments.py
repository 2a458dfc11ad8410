"""The sampler over segments (sampling.hip: vocabularies above 2048 with top-k
up to 128, no filter, or greedy with a penalty), replayed against the
restatement as tests/test_gpu_parity.py does: vocabularies around a multiple
of the segment and just above the limit, k from 1 to beyond the number of
segments and beyond 128 (the whole-row sampler), ties at the cut-off and
vocabularies of equal logits (more candidates than are ranked: the whole-row
passes inside the same launch)."""
import numpy as np
import pytest

from rusttorch_amd import synth
from rusttorch_amd.gpt2 import Gpt2Model
from tests.test_gpu_parity import _sampler_replay, cfg_of

pytestmark = pytest.mark.gpu


def model(vocab, change=None):
    sh = synth.ModelShape(vocab, 64, 128, 1, 2)
    sd = synth.make_weights(sh)
    if change:
        change(sd)
    return sh, Gpt2Model.from_state_dict(sd, cfg_of(sh))


@pytest.mark.parametrize("vocab", [2049, 4160, 50257, 65536])
def test_vocabularies_and_k(vocab):
    sh, m = model(vocab)
    print(f"[gpu] sampler segments vocab {vocab}", flush=True)
    for k in (1, 2, 50, 128, 129):
        for top_p, penalty in ((1.0, 1.0), (0.7, 1.3)):
            _sampler_replay(m, sh, dict(temperature=0.7, top_k=k, top_p=top_p, repetition_penalty=penalty), steps=5,
                            stream=k)
    _sampler_replay(m, sh, dict(temperature=1.2, top_k=0, top_p=1.0, repetition_penalty=1.1), steps=8, stream=3)
    _sampler_replay(m, sh, dict(temperature=0.0, top_k=0, top_p=1.0, repetition_penalty=1.7), steps=8, stream=4)
    m.close()


@pytest.mark.parametrize("distinct", [700, 90, 3, 1])
def test_ties(distinct):
    """Rows of wte repeat, so every logit value is shared by vocab / distinct
    tokens: ties at the cut-off, then more candidates than fit."""
    def change(sd):
        sd["wte.weight"] = np.ascontiguousarray(sd["wte.weight"][np.arange(6400) % distinct])
    sh, m = model(6400, change)
    print(f"[gpu] sampler ties {distinct}", flush=True)
    for kw in (dict(temperature=0.8, top_k=40, top_p=1.0, repetition_penalty=1.0),
               dict(temperature=0.8, top_k=40, top_p=0.5, repetition_penalty=1.2),
               dict(temperature=0.8, top_k=0, top_p=1.0, repetition_penalty=1.0),
               dict(temperature=0.0, top_k=0, top_p=1.0, repetition_penalty=1.2)):
        _sampler_replay(m, sh, kw, steps=5, stream=7)
    m.close()
