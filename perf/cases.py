"""Performance cases of the GPT-2 token loop: what programs do with a `Gpt2Model`.

A case names a call pattern, a model width and its sizes:

  call     loop     a program's own token loop: the prompt through `forward_cached` with every
                    row's logits, then one token at a time
           fill     a prompt read into a session's cache without its logits, then one token at a
                    time per sequence
           greedy   `generate_cached_batched`, then the generated text read into a session's cache
                    and the logits of what follows it (the next turn of a session)
           sample   `forward_cached` over the prompt (its logits score it), then
                    `generate_with_config`
           forward  `forward` over a text, all logits to the host (scoring)
  model    a GPT-2 width; layers: how many of its layers are stacked (each costs the same, so the
           wide models are measured on a shorter stack)
  storage  f32, or bf16 weights (activations, cache and sums stay f32)
  batch, prompt, new: sequences, tokens per prompt, tokens generated or fed one by one

Weights follow GPT-2's initialisation with LayerNorm gains and biases off their
neutral values, ids are uniform; everything is made from the seed.
"""
import math

import numpy as np
import torch

from rusttorch_amd.gpt2 import GenerationConfig, Gpt2Config, Gpt2Model

_WIDTHS = {
    "small": Gpt2Config.gpt2_small,
    "medium": Gpt2Config.gpt2_medium,
    "large": Gpt2Config.gpt2_large,
    "xl": Gpt2Config.gpt2_xl,
}

_LISTED = [
    # the smallest call: the first tokens of an interactive session, each with its logits
    dict(name="loop_small_b1_p1", call="loop", model="small", layers=12, storage="f32", batch=1, prompt=1, new=3),
    # batch-1 greedy completion of a short prompt: GPT-2 small as it is, 64 tokens
    dict(name="greedy_small_b1_p32", call="greedy", model="small", layers=12, storage="f32", batch=1, prompt=32,
         new=64),
    # a completion behind a long document: long-KV attention, a prompt of odd length
    dict(name="greedy_medium_b1_p701", call="greedy", model="medium", layers=12, storage="f32", batch=1, prompt=701,
         new=96),
    # eight requests served together
    dict(name="greedy_small_b8_p128", call="greedy", model="small", layers=12, storage="f32", batch=8, prompt=128,
         new=64),
    # documents of nearly the whole context read in one batch: the prefill at its largest
    dict(name="fill_large_b16_p1023", call="fill", model="large", layers=8, storage="f32", batch=16, prompt=1023,
         new=1),
    # the widest model with bf16 weights, sixteen requests
    dict(name="greedy_xl_bf16_b16_p64", call="greedy", model="xl", layers=8, storage="bf16", batch=16, prompt=64,
         new=64),
    # sampled completion with every filter on (GenerationConfig.creative)
    dict(name="sample_small_creative_p45", call="sample", model="small", layers=12, storage="f32", batch=1, prompt=45,
         new=64, temperature=0.9, top_k=50, top_p=0.95, penalty=1.2),
    # scoring a text: all logits to the host
    dict(name="forward_small_p333", call="forward", model="small", layers=12, storage="f32", batch=1, prompt=333,
         new=0),
    # a paragraph read and continued on a bf16 model, batch 1
    dict(name="fill_medium_bf16_b1_p100", call="fill", model="medium", layers=12, storage="bf16", batch=1, prompt=100,
         new=4),
    # more requests than one matrix tile has rows
    dict(name="greedy_small_b24_p50", call="greedy", model="small", layers=12, storage="f32", batch=24, prompt=50,
         new=24),
    # a question to a wide f32 model, its answer fed token by token
    dict(name="fill_large_b1_p77", call="fill", model="large", layers=8, storage="f32", batch=1, prompt=77, new=8),
    # a short question to the widest model, nucleus sampling
    dict(name="sample_xl_bf16_top_p_p20", call="sample", model="xl", layers=8, storage="bf16", batch=1, prompt=20,
         new=32, temperature=0.8, top_k=0, top_p=0.9, penalty=1.0),
]


def listed():
    return [dict(c) for c in _LISTED]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    most = [max(work(c)[k] for c in _LISTED) for k in ("bytes", "flops")]
    while True:
        call = rng.choice(["loop", "fill", "greedy", "greedy", "sample", "forward"])
        model, storage = rng.choice([("small", "f32"), ("small", "f32"), ("small", "bf16"), ("medium", "f32"),
                                     ("medium", "bf16"), ("large", "f32"), ("xl", "bf16")])
        c = dict(call=call, model=model, layers=rng.randint(4, 12 if model in ("small", "medium") else 8),
                 storage=storage, batch=1, prompt=1, new=0)
        if call == "loop":
            c.update(prompt=_log_int(rng, 1, 64), new=rng.randint(1, 16))
        elif call == "fill":
            c.update(batch=_log_int(rng, 1, 32), prompt=_log_int(rng, 2, 1016), new=rng.randint(1, 8))
        elif call == "greedy":
            c.update(batch=_log_int(rng, 1, 32), prompt=_log_int(rng, 1, 900), new=_log_int(rng, 4, 96))
        elif call == "sample":
            c.update(prompt=_log_int(rng, 2, 96), new=_log_int(rng, 4, 96),
                     temperature=rng.choice([0.7, 0.8, 0.9, 1.0]), top_k=rng.choice([0, 40, 50]),
                     top_p=rng.choice([1.0, 0.9, 0.95]), penalty=rng.choice([1.0, 1.0, 1.2]))
        else:
            c.update(prompt=_log_int(rng, 2, 500))
        # (the logits of a pass stay below a gigabyte, and no pass costs more than the largest listed one)
        if c["batch"] * max(1, c["new"] if call == "fill" else 1) > 64 or c["prompt"] + c["new"] > 1023:
            continue
        w = work(c)
        if w["bytes"] <= most[0] and w["flops"] <= most[1]:
            return c


# -- inputs --


def _config(case):
    cfg = _WIDTHS[case["model"]]()
    cfg.n_layer = case["layers"]
    return cfg


def _weights(case, seed):
    """The state dict on the GPU, f32, in Conv1D layout [in, out]."""
    cfg = _config(case)
    g = torch.Generator(device="cuda").manual_seed(seed)
    d, out = cfg.n_embd, {}

    def normal(name, shape, std, mean=0.0):
        out[name] = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).add_(mean)

    resid = 0.02 / math.sqrt(2 * cfg.n_layer)
    normal("wte.weight", (cfg.vocab_size, d), 0.02)
    normal("wpe.weight", (cfg.n_positions, d), 0.01)
    for i in range(cfg.n_layer):
        p = f"h.{i}."
        for ln in ("ln_1", "ln_2"):
            normal(p + ln + ".weight", (d,), 0.1, 1.0)
            normal(p + ln + ".bias", (d,), 0.02)
        for name, n_in, n_out, std in (("attn.c_attn", d, 3 * d, 0.02), ("attn.c_proj", d, d, resid),
                                       ("mlp.c_fc", d, 4 * d, 0.02), ("mlp.c_proj", 4 * d, d, resid)):
            normal(p + name + ".weight", (n_in, n_out), std)
            normal(p + name + ".bias", (n_out,), 0.02)
    normal("ln_f.weight", (d,), 0.1, 1.0)
    normal("ln_f.bias", (d,), 0.02)
    return out


def _ids(case, seed):
    """[batch, prompt] ids, and the [batch, new] ids that loop and fill feed one by one."""
    rng = np.random.default_rng(seed)
    ids = rng.integers(0, _config(case).vocab_size, (case["batch"], case["prompt"] + case["new"]))
    return ids[:, :case["prompt"]], ids[:, case["prompt"]:]


def _sampling(case, seed):
    return GenerationConfig(max_new_tokens=case["new"], temperature=case["temperature"], top_k=case["top_k"],
                            top_p=case["top_p"], repetition_penalty=case["penalty"], seed=seed)


def prepare(case, seed):
    sd = {k: v.cpu().numpy() for k, v in _weights(case, seed).items()}
    model = Gpt2Model.from_state_dict(sd, _config(case), storage=case["storage"])
    prompt, fed = _ids(case, seed)
    state = {"call": case["call"], "new": case["new"], "model": model, "prompt": prompt, "fed": fed}
    if case["call"] != "forward":
        state["cache"] = model.new_cache(case["batch"])
    if case["call"] == "sample":
        state["config"] = _sampling(case, seed)
    return state


def run(state):
    model, prompt, fed, call = state["model"], state["prompt"], state["fed"], state["call"]
    if call == "forward":
        return {"logits": model.forward(prompt[0])}
    cache = state["cache"]
    cache.clear()
    if call == "loop":
        logits = [model.forward_cached(prompt[0], cache)]
        for t in range(fed.shape[1]):
            logits.append(model.forward_cached(fed[0, t:t + 1], cache))
        return {"logits": logits}
    if call == "fill":
        model.forward_cached_batched(prompt, cache, want_logits=False)
        return {"logits": [model.forward_cached_batched(fed[:, t:t + 1], cache) for t in range(fed.shape[1])]}
    if call == "greedy":
        ids = model.generate_cached_batched(prompt, state["new"])
        model.forward_cached_batched(ids[:, :-1], cache, want_logits=False)
        return {"ids": ids, "logits": model.forward_cached_batched(ids[:, -1:], cache)}
    logits = model.forward_cached(prompt[0], cache)
    return {"ids": np.array(model.generate_with_config(prompt[0], state["config"])), "logits": logits}


# -- what a pass cannot do without --


def work(case):
    cfg = _config(case)
    d, L, V, B = cfg.n_embd, cfg.n_layer, cfg.vocab_size, case["batch"]
    wbytes = 2 if case["storage"] == "bf16" else 4
    layers, head, small = L * 12 * d * d * wbytes, V * d * wbytes, (L * 13 * d + 2 * d) * 4

    def forward(n, past, rows, out):
        """n new tokens per sequence behind `past`; the logits of `rows` rows, out of them to the host."""
        kv = L * 2 * d * 4
        b = layers + small + (head if rows else 0)
        b += B * (kv * (past + n) + (kv + 8 * d) * n) + out * V * 4
        f = B * n * L * (24 * d * d + 4 * d * (past + (n + 1) / 2)) + rows * 2 * d * V
        return b, f

    P, N, passes = case["prompt"], case["new"], []
    if case["call"] == "forward":
        passes.append(forward(P, 0, P, P))
    elif case["call"] == "loop":
        passes += [forward(P, 0, P, P)] + [forward(1, P + t, 1, 1) for t in range(N)]
    elif case["call"] == "fill":
        passes += [forward(P, 0, 0, 0)] + [forward(1, P + t, B, B) for t in range(N)]
    else:
        passes += [forward(P, 0, B, 0)] + [forward(1, P + t, B, 0) for t in range(N - 1)]
        if case["call"] == "greedy":
            passes += [forward(P + N - 1, 0, 0, 0), forward(1, P + N - 1, B, B)]
        else:
            passes.append(forward(P, 0, P, P))
    return {"bytes": float(sum(p[0] for p in passes)), "flops": float(sum(p[1] for p in passes))}


def tolerance(case):
    # f32 sums in every storage type: up to 9e-7 off 64 bits over the ranges, so two implementations
    # are up to 1.3e-6 apart; ids follow the logits, whose near ties are far apart
    return {"rel": 5e-6, "max": 1e-4, "differ": 0.01}


# -- the same in 64 bits --


class _Exact:
    """GPT-2's forward in float64 with a growing cache."""

    def __init__(self, case, seed):
        self.cfg = _config(case)
        self.w = {}
        for k, v in _weights(case, seed).items():
            matrix = v.dim() == 2 and k != "wpe.weight"
            self.w[k] = (v.bfloat16() if matrix and case["storage"] == "bf16" else v).double()
        self.kv = [None] * self.cfg.n_layer
        self.past = 0

    def _norm(self, x, name):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], self.w[name + ".weight"], self.w[name + ".bias"],
                                              self.cfg.layer_norm_epsilon)

    def _linear(self, x, name):
        return x @ self.w[name + ".weight"] + self.w[name + ".bias"]

    def _attend(self, q, k, v):
        """q [H, n, hd] of one sequence over k, v [H, past + n, hd]."""
        n, total = q.shape[1], k.shape[1]
        s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
        hidden = torch.ones(n, total, dtype=torch.bool, device=q.device).triu(total - n + 1)
        return torch.matmul(torch.softmax(s.masked_fill_(hidden, float("-inf")), -1), v)

    def forward(self, ids, rows="all"):
        """Logits [B, n, V] of ids [B, n] behind the cache: of all rows, the last one, or none."""
        ids = torch.as_tensor(np.ascontiguousarray(ids).astype(np.int64), device="cuda")
        B, n = ids.shape
        H, d = self.cfg.n_head, self.cfg.n_embd
        at = torch.arange(self.past, self.past + n, device="cuda")
        x = self.w["wte.weight"][ids] + self.w["wpe.weight"][at]
        for i in range(self.cfg.n_layer):
            p = f"h.{i}."
            qkv = self._linear(self._norm(x, p + "ln_1"), p + "attn.c_attn")
            q, k, v = (t.reshape(B, n, H, d // H).transpose(1, 2).contiguous() for t in qkv.split(d, -1))
            if self.kv[i] is not None:
                k, v = torch.cat([self.kv[i][0], k], 2), torch.cat([self.kv[i][1], v], 2)
            self.kv[i] = (k, v)
            a = torch.stack([self._attend(q[b], k[b], v[b]) for b in range(B)])
            x = x + self._linear(a.transpose(1, 2).reshape(B, n, d), p + "attn.c_proj")
            h = self._linear(self._norm(x, p + "ln_2"), p + "mlp.c_fc")
            h = 0.5 * h * (1 + torch.tanh(math.sqrt(2 / math.pi) * (h + 0.044715 * h ** 3)))
            x = x + self._linear(h, p + "mlp.c_proj")
        self.past += n
        if rows == "none":
            return None
        x = x if rows == "all" else x[:, -1:]
        return self._norm(x, "ln_f") @ self.w["wte.weight"].t()


def exact(case, seed):
    m, (prompt, fed) = _Exact(case, seed), _ids(case, seed)
    if case["call"] == "forward":
        return {"logits": m.forward(prompt)[0]}
    if case["call"] == "loop":
        return {"logits": [m.forward(prompt)[0]] + [m.forward(fed[:, t:t + 1])[0] for t in range(fed.shape[1])]}
    if case["call"] == "fill":
        m.forward(prompt, "none")
        return {"logits": [m.forward(fed[:, t:t + 1]) for t in range(fed.shape[1])]}
    if case["call"] == "greedy":
        # the token fed last is the last one chosen: its step's logits are what run() returns
        logits = m.forward(prompt, "last")
        for _ in range(case["new"]):
            token = logits.argmax(-1)
            logits = m.forward(token.cpu().numpy())
        return {"ids": None, "logits": logits}
    return {"ids": None, "logits": m.forward(prompt)[0]}
