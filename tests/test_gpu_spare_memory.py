"""The prefill's second copy of the weights is memory that the library can do
without: an allocation that fails takes it back and succeeds, and the model's
prompts run the f32-MFMA kernels from then on. RTG_TEST_MALLOC_FAIL=1 makes the
first try of every allocation count as failed, so nothing has to fill the
device."""
import threading
import time

import numpy as np
import pytest

from rusttorch_amd import synth
from rusttorch_amd.gpt2 import Gpt2Config, Gpt2Model
from tests import ref64

pytestmark = pytest.mark.gpu

SH = synth.ModelShape(515, 256, 192, 2, 3)
CFG = Gpt2Config(SH.vocab_size, SH.n_positions, SH.n_embd, SH.n_layer, SH.n_head, SH.layer_norm_epsilon)


def off(a, ref):
    return float(np.linalg.norm(a.astype(np.float64) - ref) / np.linalg.norm(ref))


@pytest.mark.parametrize("n", [40, 200])
def test_a_failed_allocation_takes_the_copy_back(monkeypatch, n):
    sd = synth.make_weights(SH)
    models = [Gpt2Model.from_state_dict(sd, CFG) for _ in range(2)]
    ids = synth.make_tokens(n, SH.vocab_size, stream=70 + n)
    before = [m.forward(ids) for m in models]
    print(f"[gpu] spare memory, prompt of {n}", flush=True)
    monkeypatch.setenv("RTG_TEST_MALLOC_FAIL", "1")
    cache = models[0].new_cache(3)  # (needs memory: every model's copy goes)
    monkeypatch.delenv("RTG_TEST_MALLOC_FAIL")
    cache.close()
    ref = ref64.forward(sd, ids, SH.n_layer, SH.n_head, SH.layer_norm_epsilon)
    for m, a in zip(models, before):
        b = m.forward(ids)
        assert not np.array_equal(a, b)  # other kernels, the same product to f32's accuracy
        assert off(a, ref) < 2e-6 and off(b, ref) < 2e-6, (off(a, ref), off(b, ref))
        m.close()
    late = Gpt2Model.from_state_dict(sd, CFG)  # a model loaded afterwards has its copy
    assert np.array_equal(late.forward(ids), before[0])
    late.close()


def test_while_other_threads_read_prompts(monkeypatch):
    """Passes under way keep the copy until they are enqueued: every result is
    one of the two forms' whole. (100 rows: neither form splits k there, so a
    form's results do not depend on its cache's workspace.)"""
    sd = synth.make_weights(SH)
    m = Gpt2Model.from_state_dict(sd, CFG)
    ids = synth.make_tokens(100, SH.vocab_size, stream=77)
    first = m.forward(ids)
    results, stop = [[] for _ in range(4)], threading.Event()

    def work(out):
        while not stop.is_set() and len(out) < 2000:
            out.append(m.forward(ids))

    def more(than):
        while any(t.is_alive() and len(r) < n + 5 for t, r, n in zip(threads, results, than)):
            time.sleep(0.001)

    monkeypatch.setenv("RTG_TEST_MALLOC_FAIL", "0")  # (set before the threads read the environment)
    print("[gpu] spare memory, threads", flush=True)
    threads = [threading.Thread(target=work, args=(r,)) for r in results]
    for t in threads:
        t.start()
    more([0] * 4)
    monkeypatch.setenv("RTG_TEST_MALLOC_FAIL", "1")
    cache = m.new_cache(2)
    monkeypatch.setenv("RTG_TEST_MALLOC_FAIL", "0")
    more([len(r) for r in results])
    stop.set()
    for t in threads:
        t.join()
    cache.close()
    last = m.forward(ids)
    assert not np.array_equal(first, last)
    for r in results:
        assert len(r) >= 10 and all(np.array_equal(x, first) or np.array_equal(x, last) for x in r)
    m.close()
