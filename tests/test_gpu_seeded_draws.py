"""A seed gives the text it gave before the f16-pair prefill and the sampler
over segments came in: ids recorded from the build that ran f32-MFMA prefills
and the whole-row sampler for every model.

The models' distributions are nearly flat (random weights: tens of thousands of
kept tokens of 2e-5 each), where a change of the logits or of the running sums
by 1e-6 moves about one draw in a few hundred to the next token. The recorded
cases are ones that came out differently: "topp" and "uncached" with the prompt
on the f16-pair GEMMs, one for every kind of GEMM that a prompt meets (up to 32
and 64 rows, more, f32 and bf16 weights, the uncached loop); "temp" with segment
sums in another order than the whole row's. Ids are whole numbers: equal."""
import pytest

from rusttorch_amd import synth
from rusttorch_amd.gpt2 import GenerationConfig, Gpt2Config, Gpt2Model

pytestmark = pytest.mark.gpu

# vocabulary, positions, width, layers, heads
SHAPES = {
    "small": (50257, 256, 768, 2, 12),
    "wide": (50257, 256, 1600, 1, 25),
    "thin": (50257, 256, 192, 2, 3),
}
FILTERS = {
    "topp": dict(temperature=0.8, top_k=0, top_p=0.9, repetition_penalty=1.0),
    "temp": dict(temperature=1.0, top_k=0, top_p=1.0, repetition_penalty=1.1),
}
# (shape, storage, prompt length, filters, seed): the ids drawn
IDS = {
    ("small", "f32", 100, "topp", 16): [
        18334, 4033, 42627, 29638, 32296, 11620, 18851, 2, 27916, 44025, 33834, 31937,
        1442, 42322, 12185, 31553, 33310, 6574, 37855, 3303, 4049, 32372, 45364, 43033,
        10418, 23673, 8429, 3579, 27853, 22408, 30579, 37190],
    ("small", "f32", 140, "topp", 15): [
        26435, 39164, 27964, 10798, 8965, 45789, 39612, 38568, 17396, 25306, 8729, 29823,
        8552, 6009, 17754, 28894, 19663, 38725, 34862, 11406, 21146, 32205, 8369, 25154,
        28135, 20922, 17951, 20688, 1120, 6476, 9563, 1671],
    ("small", "bf16", 20, "topp", 29): [
        36775, 36439, 44193, 16240, 3984, 26292, 38894, 16097, 45938, 9962, 42438, 37749,
        37881, 29113, 7835, 4272, 29067, 50240, 20753, 26657, 45882, 3308, 14387, 25853,
        33463, 15601, 32727, 39829, 30485, 18329, 5623, 33543],
    ("small", "bf16", 45, "topp", 3): [
        5620, 35266, 30756, 3662, 10990, 31990, 6745, 44627, 24627, 44657, 35057, 35681,
        24117, 16803, 36069, 40143, 15300, 5290, 8760, 29475, 41141, 47050, 33608, 9604,
        31189, 44747, 10954, 6065, 32103, 43791, 34847, 36364],
    ("small", "bf16", 45, "uncached", 8): [
        31058, 30752, 34589, 26864, 3206, 18892, 47956, 17953, 4032, 21900, 31459, 37098],
    ("wide", "bf16", 20, "topp", 19): [
        36962, 6071, 18379, 4191, 39356, 48203, 24289, 28879, 12680, 26330, 45353, 46404,
        40984, 43793, 39032, 37349, 27569, 28605, 22243, 29320, 28637, 17669, 27401, 1585,
        29716, 18369, 6239, 21168, 35730, 5234, 21280, 37077],
    ("thin", "f32", 40, "topp", 19): [
        36916, 5871, 18238, 4188, 39400, 48142, 23945, 28681, 12518, 26470, 45479, 46562,
        40780, 43876, 39174, 37608, 27750, 28550, 22122, 29018, 28629, 17568, 27265, 1522,
        29727, 18656, 6210, 21173, 35697, 5110, 21307, 37133],
    ("small", "f32", 45, "temp", 20): [
        10638, 961, 12674, 18128, 5136, 8648, 41604, 15630, 4011, 17558, 6226, 38943,
        18533, 26529, 33253, 33690, 1486, 22114, 38017, 40084, 2379, 10593, 26949, 13096,
        48074, 26700, 35747, 400, 37502, 23136, 12985, 11538],
    ("small", "bf16", 45, "temp", 31): [
        42266, 37071, 25295, 27165, 29937, 16461, 19855, 30785, 13810, 38021, 39756, 15159,
        32775, 8863, 17261, 10060, 7633, 17290, 47044, 9713, 8506, 42861, 7061, 38799,
        22561, 17018, 26119, 795, 47672, 5540, 12150, 12771],
    ("small", "bf16", 100, "temp", 18): [
        3355, 35866, 21592, 35294, 6024, 46137, 49253, 6607, 35695, 26125, 19523, 43338,
        41650, 1323, 43295, 13206, 2731, 9708, 50237, 22400, 30768, 35837, 23408, 26335,
        4891, 11517, 4929, 29602, 22809, 33105, 41395, 6059],
    ("wide", "bf16", 20, "temp", 38): [
        46123, 410, 4021, 11210, 16475, 46531, 16519, 40052, 23112, 1670, 21127, 46281,
        29316, 10920, 34562, 11729, 39491, 24780, 22625, 24052, 43012, 2052, 49071, 3666,
        22267, 5004, 3875, 23808, 26848, 43249, 16256, 14703],
}


@pytest.mark.parametrize("shape,storage", sorted({k[:2] for k in IDS}))
def test_seeded_text(shape, storage):
    sh = synth.ModelShape(*SHAPES[shape])
    m = Gpt2Model.from_state_dict(synth.make_weights(sh, bf16=storage == "bf16"), Gpt2Config(*SHAPES[shape], 1e-5),
                                  storage=storage)
    for (name, kind, n, how, seed), want in IDS.items():
        if (name, kind) != (shape, storage):
            continue
        prompt = synth.make_tokens(n, sh.vocab_size, stream=60 + n)
        print(f"[gpu] seeded draws {shape} {storage} prompt {n} {how} seed {seed}", flush=True)
        if how == "uncached":
            got = m.generate(prompt, len(want), 0.9, seed)
        else:
            got = m.generate_with_config(prompt, GenerationConfig(max_new_tokens=len(want), seed=seed, **FILTERS[how]))
        assert got[n:] == want, (n, how, seed)
    m.close()
