"""The prefill on f16-pair GEMMs and attention (gemm_pair.hip, attn_pair.hip)
through forward_cached, against float64 (tests/ref64.py).

The bar is the CPU oracle's own distance from float64 on the same model and
ids (f32 throughout, sums in k order): the library may be at most twice as far
in the 2-norm, plus 2e-7 (3 ulp of f32) where the oracle happens to be closer.
bf16 storage is compared on weights that are bf16 values already.

Shapes: one layer, chosen so that every tile of the dispatch occurs with and
without a k split for both kinds of weights (tests/test_pair_choice.py checks
that on the CPU), with ragged M and V and head dims 64 and 32; a second chunk behind cached rows; widths above 2048
(the block-per-row LayerNorm); weights and gains whose magnitudes spread over
many powers of two; and weights for which the path is not taken at all.
"""
import numpy as np
import pytest

from rusttorch_amd import synth
from rusttorch_amd.gpt2 import Gpt2Config, Gpt2Model
from tests import ref64

pytestmark = pytest.mark.gpu


def build(sh, storage="f32", change=None):
    sd = synth.make_weights(sh, bf16=storage == "bf16")
    if change:
        change(sd)
    cfg = Gpt2Config(sh.vocab_size, sh.n_positions, sh.n_embd, sh.n_layer, sh.n_head, sh.layer_norm_epsilon)
    return sd, Gpt2Model.from_state_dict(sd, cfg, storage=storage)


def off(a, ref):
    return float(np.linalg.norm(np.asarray(a, np.float64) - ref) / np.linalg.norm(ref))


def check(oracle_lib, sh, sd, m, chunks, batch=1):
    print(f"[gpu] pair gemm {sh} {m.storage} chunks {chunks} batch {batch}", flush=True)
    total = sum(chunks)
    ids = np.stack([synth.make_tokens(total, sh.vocab_size, stream=40 + b) for b in range(batch)])
    c = m.new_cache(batch)
    got, at = [], 0
    for n in chunks:
        got.append(m.forward_cached_batched(ids[:, at:at + n], c))
        at += n
    got = np.concatenate(got, axis=1)
    om = oracle_lib.OracleModel.from_shape(sd, sh, threads=8)
    for b in sorted({0, batch - 1}):
        ref = ref64.forward(sd, ids[b], sh.n_layer, sh.n_head, sh.layer_norm_epsilon)
        mine, plain = off(got[b], ref), off(om.forward(ids[b]), ref)
        print(f"  sequence {b}: {mine:.2e} from float64, oracle {plain:.2e}", flush=True)
        assert mine <= 2 * plain + 2e-7, (mine, plain)
    c.close()


# width, heads, vocabulary, batch, chunks
SHAPES = [
    (192, 3, 301, 1, (33,)),          # 32 x 64 tiles, split
    (192, 6, 301, 3, (17,)),          # head_dim 32, 51 rows
    (192, 3, 301, 5, (131, 7)),       # 655 rows, then 35 behind 131 cached
    (192, 3, 301, 1, (520, 40)),      # attention's keys over 8 waves, then behind 520 cached
    (192, 3, 301, 90, (33, 34)),      # 64 and 32 queries per attention workgroup
    (768, 12, 515, 1, (65,)),
    (768, 12, 515, 2, (161,)),
    (768, 12, 515, 9, (129,)),        # 64 x 64 and 64 x 128 tiles
    (768, 12, 515, 10, (65,)),        # 128 x 128 tiles of 8 waves
    (1024, 16, 258, 1, (40,)),        # 64 x 64 tiles, split
    (1024, 16, 258, 16, (65,)),       # 128 x 128 tiles, split
    (1280, 20, 258, 1, (40,)),        # 64 x 128 tiles, split
    (1600, 25, 258, 1, (40,)),
    (1600, 25, 258, 3, (65,)),        # 128 x 128 tiles of 8 waves, split
    (1600, 25, 258, 16, (65,)),       # K = 6400 split
    (1600, 25, 258, 22, (65,)),       # 256 x 256 tiles, split
    (128, 2, 50257, 1, (40,)),        # a wide LM head: 64 x 128 tiles,
    (128, 2, 50257, 1, (70,)),        #   128 x 128 tiles of 4 waves,
    (128, 2, 50257, 1, (200,)),       #   256 x 256 tiles,
    (128, 2, 50257, 1, (999,)),       #   and over many rows
]
MANY_ROWS = (640, 10, 130, 32, (403,))


@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("d,heads,V,batch,chunks", SHAPES)
def test_shapes(oracle_lib, storage, d, heads, V, batch, chunks):
    sh = synth.ModelShape(V, 1024, d, 1, heads)
    sd, m = build(sh, storage)
    check(oracle_lib, sh, sd, m, chunks, batch)
    m.close()


@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_many_rows(oracle_lib, storage):
    """Enough rows that the layer GEMMs take the 256 x 256 and 128 x 128 tiles."""
    d, heads, V, batch, chunks = MANY_ROWS
    sh = synth.ModelShape(V, 512, d, 1, heads)
    sd, m = build(sh, storage)
    check(oracle_lib, sh, sd, m, chunks, batch=batch)
    m.close()


def test_wide_rows(oracle_lib):
    sh = synth.ModelShape(70, 64, 2112, 1, 33)
    sd, m = build(sh)
    check(oracle_lib, sh, sd, m, (35,))
    m.close()


def test_spread_magnitudes(oracle_lib):
    """Gains, weight rows and columns of very different sizes: the input and
    row scales keep every pair as good as f32."""
    def change(sd):
        for k in ("h.0.ln_1.weight", "h.0.ln_2.weight", "ln_f.weight"):
            sd[k][5] *= 3000.0
            sd[k][7:40] *= 2.0 ** -14
        for k, n in (("h.0.attn.c_attn.weight", 192), ("h.0.mlp.c_fc.weight", 192), ("h.0.mlp.c_proj.weight", 768)):
            sd[k][:, 3::7] *= 2.0 ** -20
            sd[k][n // 2:n // 2 + 9] *= 2.0 ** 9
        sd["h.0.mlp.c_fc.bias"][::5] = 40.0
        sd["wte.weight"][17] *= 2.0 ** 12
    sh = synth.ModelShape(301, 256, 192, 1, 3)
    sd, m = build(sh, change=change)
    check(oracle_lib, sh, sd, m, (77, 120))
    m.close()


@pytest.mark.parametrize("storage", ["f32", "bf16"])
@pytest.mark.parametrize("d,heads,batch,chunks", [
    (192, 3, 1, (40, 30)),       # at most 64 rows, split; 30 behind 40 cached
    (192, 6, 3, (27,)),          # head_dim 32, 81 rows
    (192, 3, 1, (520, 90)),      # 64 x 128 tiles, keys over 8 waves
    (768, 12, 9, (129,)),        # 128 x 128 tiles, split
    (192, 3, 90, (33, 34)),      # more than 1024 rows; 64 and 32 queries per attention workgroup
    (640, 10, 32, (403,)),       # 128 queries per attention workgroup
])
def test_f32_kernels(oracle_lib, storage, d, heads, batch, chunks):
    """The f32-MFMA prefill, which drawn prompts and models without the pair
    copy run: a negative epsilon keeps a model off the pair GEMMs."""
    sh = synth.ModelShape(301, 1024, d, 1, heads, -1e-9)
    sd, m = build(sh, storage)
    check(oracle_lib, sh, sd, m, chunks, batch)
    m.close()


@pytest.mark.parametrize("chunks", [(77,), (200,)])  # a wave of keys per workgroup, and the keys split over waves
@pytest.mark.parametrize("what", ["collapsed head", "collapsed keys", "large value", "uneven columns"])
def test_score_range(oracle_lib, what, chunks):
    """A head whose queries and keys are 1e-20 (its scores are 0: uniform
    attention), one whose keys alone are, a value column of 1e29 that c_proj
    brings back to 1 (past the bounds: the f32 kernels run), and a head with a
    query column 2^24 times the others whose keys are that much smaller, and the
    other way round."""
    def change(sd):
        w, b = sd["h.0.attn.c_attn.weight"], sd["h.0.attn.c_attn.bias"]
        if what == "uneven columns":
            for c, f in ((64, 2.0 ** 24), (70, 2.0 ** -24)):
                for col, g in ((c, f), (192 + c, 1 / f)):
                    w[:, col] *= g
                    b[col] *= g
            return
        if what == "large value":
            b[2 * 192 + 64] = 1e29
            sd["h.0.attn.c_proj.weight"][64] *= 1e-29
            return
        for first in (64, 192 + 64) if what == "collapsed head" else (192 + 64,):
            w[:, first:first + 64] *= 1e-20
            b[first:first + 64] *= 1e-20
    sh = synth.ModelShape(301, 256, 192, 1, 3)
    sd, m = build(sh, change=change)
    check(oracle_lib, sh, sd, m, chunks)
    m.close()


@pytest.mark.parametrize("what", ["nan bias", "inf weight", "negative epsilon"])
def test_models_outside_the_bounds(oracle_lib, what):
    """No finite bound, or an epsilon for which it does not hold: the f32 GEMMs
    run, with the oracle's pattern of finite values."""
    def change(sd):
        if what == "nan bias":
            sd["h.0.mlp.c_fc.bias"][3] = np.nan
        if what == "inf weight":
            sd["wte.weight"][9, 4] = np.inf  # one logit column
    eps = -1e-9 if what == "negative epsilon" else 1e-5
    sh = synth.ModelShape(301, 64, 192, 1, 3, eps)
    sd, m = build(sh, change=change)
    ids = synth.make_tokens(40, 300, stream=3)
    ids[ids == 9] = 8
    got = m.forward(ids)
    ref = oracle_lib.OracleModel.from_shape(sd, sh, threads=8).forward(ids)
    assert np.array_equal(np.isfinite(got), np.isfinite(ref))
    fine = np.isfinite(ref)
    assert np.all(np.abs(got[fine] - ref[fine]) <= 1e-3 + 1e-4 * np.abs(ref[fine]))
    m.close()


@pytest.mark.parametrize("storage", ["f32", "bf16"])
def test_no_bias(storage):
    """The largest tiles' rounding errors have no common part (small terms are
    rounded towards minus infinity when an MFMA adds them to a large sum): the
    mean error of the first layer's keys and values, in units of the errors'
    deviation, is what the mean of as many independent errors shows, 6 standard
    deviations of it, plus 0.01 (without the weights' signs: -0.042 and -0.059)."""
    d, heads, V, batch, (n,) = MANY_ROWS
    sh = synth.ModelShape(V, 512, d, 1, heads)
    sd, m = build(sh, storage)
    ids = np.stack([synth.make_tokens(n, V, stream=40 + b) for b in range(batch)])
    c = m.new_cache(batch)
    print(f"[gpu] pair gemm bias {storage}", flush=True)
    m.forward_cached_batched(ids, c, want_logits=False)
    errors = []
    for b in (0, batch // 2, batch - 1):
        x = sd["wte.weight"].astype(np.float64)[ids[b]] + sd["wpe.weight"].astype(np.float64)[:n]
        x = ref64.layer_norm(x, sd["h.0.ln_1.weight"].astype(np.float64), sd["h.0.ln_1.bias"].astype(np.float64),
                             sh.layer_norm_epsilon)
        kv = x @ sd["h.0.attn.c_attn.weight"].astype(np.float64) + sd["h.0.attn.c_attn.bias"].astype(np.float64)
        for h in range(heads):
            for values in (False, True):
                col = d * (1 + values) + 64 * h
                errors.append(c.read(0, h, b, values=values) - kv[:, col:col + 64])
    e = np.stack(errors)
    print(f"  mean {e.mean() / e.std():.4f} of the deviation, {e.size} errors", flush=True)
    assert abs(e.mean()) / e.std() <= 6 / np.sqrt(e.size) + 0.01
    c.close()
    m.close()
