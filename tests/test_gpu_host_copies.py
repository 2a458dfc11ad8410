"""Logits on their way to the host: one staging chunk (4 MiB) or less, just over
one, several with a short last one, through forward_cached, against
rtg_forward_cached_noalloc (the same kernels, copied by the runtime), bit for
bit; several threads at once on caches of their own; and a program's own batched
token loop, whose steps become graph replays, against the same tokens behind a
fresh cache."""
import threading

import numpy as np
import pytest

from rusttorch_amd import _lib, synth
from rusttorch_amd.gpt2 import Gpt2Config, Gpt2Model
from tests.test_zz_no_alloc import call

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def model():
    sh = synth.ModelShape(50257, 256, 768, 2, 12)
    cfg = Gpt2Config(sh.vocab_size, sh.n_positions, sh.n_embd, sh.n_layer, sh.n_head, sh.layer_norm_epsilon)
    m = Gpt2Model.from_state_dict(synth.make_weights(sh), cfg)
    yield sh, m
    m.close()


@pytest.mark.parametrize("n", [2, 20, 21, 33, 50])
def test_every_chunk_arrives(model, n):
    sh, m = model
    ids = synth.make_tokens(n, sh.vocab_size, stream=900 + n)
    print(f"[gpu] host copy of {n} rows", flush=True)
    a, b = m.new_cache(), m.new_cache()
    assert np.array_equal(m.forward_cached(ids, a), call("rtg_forward_cached_noalloc", m, b, ids, sh.vocab_size))
    a.close()
    b.close()


def test_no_page_locked_memory(model, monkeypatch):
    """Results still arrive, through the runtime's own staging: one token (the
    persistent step and its error word), the multi-row forward, several chunks."""
    sh, m = model
    texts = [synth.make_tokens(n, sh.vocab_size, stream=930 + n) for n in (1, 9, 50)]
    want = [m.forward(t) for t in texts]
    print("[gpu] host copies without page-locked memory", flush=True)
    _lib.load().rtg_cleanup()  # the stages that calls so far left behind
    monkeypatch.setenv("RTG_TEST_PINNED_FAIL", "1")
    for t, w in zip(texts, want):
        assert np.array_equal(m.forward(t), w)


def test_threads_have_their_own_stages(model):
    sh, m = model
    texts = [synth.make_tokens(n, sh.vocab_size, stream=950 + n) for n in (1, 37, 64, 150, 90, 40)]
    want = [m.forward(t) for t in texts]
    got = [[None] * 3 for _ in texts]

    def work(i):
        for k in range(3):
            got[i][k] = m.forward(texts[i])

    print("[gpu] host copies from six threads", flush=True)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(texts))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(len(texts)):
        for k in range(3):
            assert np.array_equal(got[i][k], want[i])


@pytest.mark.parametrize("batch", [2, 32, 33])
def test_batched_token_loop(model, batch):
    sh, m = model
    ids = np.stack([synth.make_tokens(14, sh.vocab_size, stream=980 + b) for b in range(batch)])
    print(f"[gpu] batched token loop {batch}", flush=True)
    c = m.new_cache(batch)
    m.forward_cached_batched(ids[:, :6], c, want_logits=False)
    steps = [m.forward_cached_batched(ids[:, t:t + 1], c) for t in range(6, 14)]
    for t in (2, 5, 7):  # the step as a graph replay, and the same step launched kernel by kernel
        d = m.new_cache(batch)
        m.forward_cached_batched(ids[:, :6 + t], d, want_logits=False)
        one = m.forward_cached_batched(ids[:, 6 + t:7 + t], d)
        assert np.max(np.abs(one - steps[t])) < 2e-5  # the prefix's K/V came from other kernels
        d.close()
    c.close()
