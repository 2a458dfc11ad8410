"""The sampler over segments (sampling.hip: vocabularies above 2048 with top-k
up to 128, no filter, or greedy with a penalty), replayed against the
restatement as tests/test_gpu_parity.py does: vocabularies around a multiple
of the segment and just above the limit, k from 1 to beyond the number of
segments and beyond 128 (the whole-row sampler), ties at the cut-off and
vocabularies of equal logits (more candidates than are ranked: the whole-row
passes inside the same launch)."""
import ctypes as C

import numpy as np
import pytest

from rusttorch_amd import _lib, synth
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


class Params(C.Structure):
    """SampleParams (kernels.h)."""
    _fields_ = [("temperature", C.c_float), ("top_k", C.c_int), ("top_p", C.c_float), ("penalty", C.c_float),
                ("seed", C.c_uint64), ("draw0", C.c_uint32)]


class Device:
    """Device buffers through the library's own HIP runtime."""

    def __init__(self):
        self.lib = _lib.load()  # (its handle finds the runtime's functions too)
        self.ptrs = []
        self.sample = self.lib["_ZN3rtg13launch_sampleEP12ihipStream_tPKfiPKjiPjPKiRKNS_12SampleParamsES6_Pv"]
        self.sample.restype = C.c_bool
        self.work_bytes = self.lib["_ZN3rtg17sample_work_bytesEi"]
        self.work_bytes.restype = C.c_size_t

    def alloc(self, n):
        p = C.c_void_p()
        assert self.lib.hipMalloc(C.byref(p), C.c_size_t(n)) == 0
        self.ptrs.append(p)
        return p

    def put(self, a, p=None):
        p = p or self.alloc(a.nbytes)
        assert self.lib.hipMemcpy(p, a.ctypes.data_as(C.c_void_p), C.c_size_t(a.nbytes), 1) == 0
        return p

    def get(self, p, n):
        a = np.empty(n, np.uint32)
        assert self.lib.hipMemcpy(a.ctypes.data_as(C.c_void_p), p, C.c_size_t(a.nbytes), 2) == 0
        return a

    def close(self):
        for p in self.ptrs:
            self.lib.hipFree(p)


DRAWS = 24
FORMS = [(0.9, 50, 0.95, 1.2), (0.7, 128, 1.0, 1.0), (1.3, 40, 0.3, 1.0), (1.0, 1, 0.9, 1.0), (1.0, 0, 1.0, 1.0),
         (0.8, 0, 1.0, 1.3), (0.0, 0, 1.0, 1.5)]


@pytest.mark.parametrize("vocab", [2049, 4160, 20001, 50257, 65536])
def test_same_bits_as_the_whole_row(vocab):
    """The launch with segments and the one without choose the same token of
    every draw: their sums are the same bits, so no draw can fall between them.
    Flat, peaked and coarse rows (ties everywhere), rows with -inf, with one NaN
    and with one +inf."""
    rng = np.random.default_rng(vocab)
    flat = (rng.standard_normal(vocab) * 0.5).astype(np.float32)
    rows = {"flat": flat, "peaked": flat * 16, "ties": np.round(flat * 16) / 16,
            "-inf": np.where(rng.random(vocab) < 0.9, np.float32(-np.inf), flat), "nan": flat.copy(),
            "inf": flat.copy()}
    rows["nan"][vocab // 3] = np.nan
    rows["inf"][vocab - 2] = np.inf
    d = Device()
    prompt = d.put(rng.integers(0, vocab, 9).astype(np.uint32))
    steps = d.put(np.arange(1, DRAWS + 1, dtype=np.int32))
    logits, token = d.alloc(vocab * 4), d.alloc(256)
    ids = [d.alloc(DRAWS * 4) for _ in range(2)]
    work = d.alloc(d.work_bytes(C.c_int(vocab)))
    for kind, row in rows.items():
        d.put(row.astype(np.float32), logits)
        for f, (temperature, top_k, top_p, penalty) in enumerate(FORMS):
            print(f"[gpu] sampler bits vocab {vocab} {kind} form {f}", flush=True)
            sp = Params(temperature, top_k, top_p, penalty, 1000 * f + vocab, 0)
            for out, w in zip(ids, (None, work)):
                for g in range(DRAWS):
                    assert d.sample(None, logits, C.c_int(vocab), prompt, C.c_int(9), out,
                                    C.c_void_p(steps.value + 4 * g), C.byref(sp), token, w)
            assert d.lib.hipDeviceSynchronize() == 0
            assert np.array_equal(d.get(ids[0], DRAWS), d.get(ids[1], DRAWS)), (kind, f)
    d.close()
