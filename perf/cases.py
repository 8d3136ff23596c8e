"""What users of this library have it do, as cases to be timed.

A case is one request or one batch of requests: prompts of given lengths run through `Engine.step` ("prompt": the
logits at every prompt's last place, as a scoring program or a scheduler of its own asks for them) or prompts and
decoding steps through `EngineBackend` ("chat": replayed decoding steps, sampled on the device, tokens read back every
step, as the generation loop runs them; the last step's logits are kept).  The models are the benchmark's: the Llama
shapes, and the six hybrid designs at their layer sizes of a real model with fewer layers.

The weights are drawn from the seed, with the properties of trained ones that matter here: residual branches that are
small beside the stream, step sizes and decays over the ranges such layers are initialised to, routers that are sure of
their experts, and a head whose logits have a clear maximum (by some nats), so that a token does not hang on the
rounding of a sum.  The token after t is `follower(t)` for that reason, which `exact` relies on and checks.
"""
from __future__ import annotations

import hashlib
import math

import torch

import longbow_quarrel_amd as lq
from longbow_quarrel_amd.engine import EngineBackend, StepEntry
from longbow_quarrel_amd.kernels.hip import HipKernels
from longbow_quarrel_amd.model import DecoderModel
from longbow_quarrel_amd.parts.base import BuildEnv
from longbow_quarrel_amd.registry import spec_from_config

DEVICE = "cuda:0"
F64 = torch.float64
NAMES = {"vafodra": lq.VafodraConfig, "vupelorn": lq.VupelornConfig, "mifidra": lq.MifidraConfig,
         "sofinex": lq.SofinexConfig, "puzonex": lq.PuzonexConfig, "tukedra": lq.TukedraConfig}


# ---- the cases --------------------------------------------------------------------------------------------------
def _case(name, design, width, layers, kind, batch, shortest, longest, new=0, portions=1, dtype="bfloat16",
          sampled=False):
    """`portions`: a prompt comes in that many steps, one after the other; `sampled`: temperature, top-k, top-p and
    repetition penalty instead of the arg-max."""
    return {"name": name, "design": design, "width": width, "layers": layers, "kind": kind, "batch": batch,
            "shortest": shortest, "longest": longest, "new": new, "portions": portions, "dtype": dtype,
            "sampled": sampled}


def listed():
    return [
        # a few words to the small model: nothing but latency
        _case("llama_1b_short", "llama", 2048, 16, "prompt", 1, 17, 17),
        # one user's chat with the 8B shape: weights streamed for a single row
        _case("llama_8b_chat", "llama", 4096, 32, "chat", 1, 96, 96, new=33),
        # the benchmark's own batch: eight prompts of 512 tokens and decoding behind them
        _case("llama_8b_batch_8", "llama", 4096, 32, "chat", 8, 512, 512, new=33),
        # a long document and a short answer: the largest
        _case("llama_8b_document", "llama", 4096, 32, "chat", 1, 7003, 7003, new=17),
        # a service's batch of unequal prompts, sampled with all options
        _case("llama_1b_service", "llama", 2048, 16, "chat", 16, 64, 1500, new=33, sampled=True),
        # the true 32-bit path, as a check of a model's numbers uses it
        _case("llama_float32", "llama", 4096, 4, "chat", 4, 100, 333, new=9, dtype="float32"),
        # the hybrid designs: one long prompt, unequal prompts together, a prompt in portions, and batches that decode
        _case("vafodra_prompt", "vafodra", 2048, 8, "prompt", 1, 2048, 2048),
        _case("vupelorn_batch", "vupelorn", 2048, 8, "chat", 8, 200, 700, new=33),
        _case("mifidra_prompts", "mifidra", 2048, 8, "prompt", 3, 257, 1500),
        _case("sofinex_batch", "sofinex", 2048, 8, "chat", 8, 512, 512, new=17),
        _case("puzonex_chat", "puzonex", 2048, 8, "chat", 2, 900, 1100, new=33),
        _case("tukedra_portions", "tukedra", 2048, 8, "prompt", 1, 4001, 4001, portions=2),
    ]


def _spread(rng, low, high):
    """A whole number, uniform in its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """The same models and kinds of requests at other sizes, none of them larger than the largest above."""
    design = rng.choice(["llama"] * 6 + sorted(NAMES))
    dtype = "float32" if design == "llama" and rng.random() < 0.15 else "bfloat16"
    if design == "llama":
        width, layers = rng.choice([(2048, 16), (4096, 32)]) if dtype == "bfloat16" else (4096, 4)
    else:
        width, layers = rng.choice([1024, 1536, 2048, 3072, 4096]), rng.choice([4, 8])
    kind = rng.choice(["prompt", "chat"])
    batch = _spread(rng, 1, 24)
    most = 4096 if design == "llama" and dtype == "bfloat16" else 3000 if dtype == "bfloat16" else 1200
    longest = min(_spread(rng, 5, most), most // batch + 5)
    shortest = rng.randint(max(1, longest // 4), longest)
    return {"design": design, "width": width, "layers": layers, "kind": kind, "batch": batch, "shortest": shortest,
            "longest": longest, "new": rng.randint(5, 24) if kind == "chat" else 0,
            "portions": rng.choice([1, 1, 2]) if kind == "prompt" and shortest >= 8 else 1, "dtype": dtype,
            "sampled": kind == "chat" and rng.random() < 0.4}


# ---- models: layer sizes ----------------------------------------------------------------------------------------
def _llama(width, layers):
    config = {"architectures": ["LlamaForCausalLM"], "hidden_size": width, "intermediate_size": width * 7 // 2,
              "num_hidden_layers": layers, "num_attention_heads": width // 128, "num_key_value_heads": 8,
              "head_dim": 128, "vocab_size": 128256, "max_position_embeddings": 8192, "rms_norm_eps": 1e-5,
              "rope_theta": 500000.0, "rope_scaling": None, "tie_word_embeddings": False, "torch_dtype": "bfloat16",
              "bos_token_id": 128000, "eos_token_id": 128001}
    if width == 2048:  # the 1B shape
        config.update(intermediate_size=8192, head_dim=64, num_attention_heads=32, tie_word_embeddings=True,
                      rope_scaling={"rope_type": "llama3", "factor": 32.0, "low_freq_factor": 1.0,
                                    "high_freq_factor": 4.0, "original_max_position_embeddings": 8192})
    return config


YARN = {"base": 10000.0, "dims": 64, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}


def _config(case):
    """The configuration as its config.json holds it; the hybrid designs at the benchmark's layer sizes."""
    design, width, layers, vocab = case["design"], case["width"], case["layers"], 32000
    heads = width // 128
    half, kv = max(1, heads // 2), max(1, heads // 4)
    dense = {"kind": "dense", "ff": width * 7 // 2}
    if design == "llama":
        return _llama(width, layers)
    if design == "vafodra":
        left = {"dim": 128, "vdim": 128, "heads": heads, "kv_heads": kv, "mask": {"size": 1024, "keep_first": 4},
                "scale": 128 ** -0.5}
        right = {"conv": 4, "groups": 8, "heads": width // 64, "norm_groups": 8, "state": 128, "vdim": 64}
        delta = {"conv": 4, "dim": 128, "heads": heads, "kv_heads": half, "vdim": 128}
        kinds = [{"type": "parallel", "mixer": {"left": left, "right": right}, "mlp": dense}] * 3 \
            + [{"type": "delta", "mixer": delta, "mlp": dense}]
        more = {"architecture": "Vafodra", "embedding": {"scale": 1.0}, "norm": {"eps": 1e-5}, "residual_mult": 0.5}
    elif design == "vupelorn":
        latent = {"heads": heads, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "q_rank": width * 3 // 8,
                  "scale": 192 ** -0.5, "rot": {"base": 10000.0, "dims": 64}}
        gla = {"heads": width // 256, "dim": 128, "vdim": 256, "tau": 16.0, "decay_rank": 16}
        moe = {"kind": "moe", "expert": {"ff": width * 7 // 4, "limit": 7.0}, "router": {"experts": 8, "top": 2}}
        kinds = [{"type": "gla", "mixer": gla, "mlp": moe},
                 {"type": "latent_attention", "mixer": dict(latent, rot=YARN), "mlp": moe},
                 {"type": "latent_attention_2", "mixer": latent, "mlp": moe},
                 {"type": "latent_attention_2", "mixer": latent, "mlp": moe}]
        more = {"architecture": "Vupelorn", "norm": {"eps": 1e-6},
                "embedding": {"bigram": {"buckets": 65521, "mul_prev": 31, "mul_cur": 7}}}
    elif design in ("mifidra", "sofinex"):
        left = {"dim": 128, "vdim": 128, "heads": heads, "kv_heads": kv, "scale": 128 ** -0.5, "rot": YARN}
        right = {"conv": 4, "dim": 128, "vdim": 128, "heads": heads, "kv_heads": half, "decay_rank": 64,
                 "gate_rank": 64}
        moe = {"kind": "moe", "expert": {"ff": width * 5 // 4}, "shared": {"ff": width},
               "router": {"experts": 8, "top": 2, "groups": {"count": 4, "keep": 2}}}
        if design == "mifidra":
            mixer = {"left": left, "right": right, "left_scale": 1.0, "right_scale": 1.0}
            kinds = [{"type": "parallel", "mixer": mixer, "mlp": m} for m in (dense, moe)]
            more = {"architecture": "Mifidra", "logit_scale": 0.02, "norm": {"eps": 1e-5}}
        else:
            blend = {"base": 500000.0, "dims": 64,
                     "scaling": {"factor": 8.0, "original": 8192, "low": 1.0, "high": 4.0}}
            diff = {"dim": 128, "vdim": 256, "heads": half, "kv_heads": max(1, heads // 8), "scale": 128 ** -0.5,
                    "mask": {"size": 2048}, "rot": blend, "diff": 0.5}
            moe["router"] = dict(moe["router"], experts=6, identity=2)
            kinds = [{"type": "parallel", "mixer": {"left": dict(left, mask={"size": 1024}), "right": right},
                      "mlp": dict(dense, ff=width * 21 // 4)},
                     {"type": "attention", "mixer": diff, "mlp": moe}]
            more = {"architecture": "Sofinex", "embedding": {"scale": 1.0}, "norm": {"eps": 1e-5}}
    elif design == "puzonex":
        shaped = {"dim": 128, "vdim": 128, "heads": heads, "kv_heads": kv, "scale": 128 ** -0.5, "softcap": 30.0,
                  "mask": {"size": 1024}}
        memory = {"heads": max(1, width // 512), "dim": 256, "vdim": 512, "gate_cap": 15.0}
        scan = {"type": "mamba1", "mlp": dense,
                "mixer": {"inner": 2 * width, "state": 16, "dt_rank": width // 16, "conv": 4}}
        kinds = [scan, {"type": "parallel", "mlp": dense,
                        "mixer": {"left": {**shaped, "bias_max": 512, "bias_rows": 32}, "right": memory}},
                 {"type": "attention", "mlp": dense, "mixer": shaped}, scan]
        more = {"architecture": "Puzonex", "norm": {"eps": 1e-5}}
    else:
        def fading(n):
            return [1.0 - 2.0 ** (-5.0 - 3.0 * i / max(1, n - 1)) for i in range(n)]
        lightning = {"type": "lightning", "mixer": {"heads": heads, "dim": 128, "vdim": 128, "decay": fading(heads)}}
        retention = {"type": "retention", "mixer": {"heads": half, "dim": 256, "vdim": 256, "decay": fading(half),
                                                    "rot": {"base": 10000.0, "dims": 256}}}
        chunked = {"type": "attention", "mixer": {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128,
                                                  "scale": 128 ** -0.5, "mask": {"size": 1024}, "rot": YARN}}
        moe = {"kind": "moe", "expert": {"ff": width * 7 // 4}, "shared": {"ff": width * 7 // 4},
               "router": {"experts": 8, "top": 2}}
        kinds = [dict(k, mlp=moe) for k in (lightning, retention, chunked, lightning)]
        more = {"architecture": "Tukedra", "embedding": {"scale": 1.0}, "logit_scale": 1.0, "logit_softcap": 30.0,
                "norm": {"eps": 1e-5}, "streams": 4}
    made = [kinds[i % len(kinds)] for i in range(layers)]
    if design == "vupelorn":  # every fourth layer reads the latent of the layer before it
        made = [dict(m, mixer=dict(m["mixer"], kv_from=i - 1)) if i % 4 == 3 else m for i, m in enumerate(made)]
    if design == "tukedra":
        made[0] = dict(made[0], mlp=dense)
    return {**more, "layers": made, "vocab": vocab, "width": width}


def _typed_config(case):
    config = _config(case)
    return (lq.LlamaConfig if case["design"] == "llama" else NAMES[case["design"]]).from_dict(config)


# ---- weights ----------------------------------------------------------------------------------------------------
TIED = ("vupelorn", "mifidra")


class Weights:
    """A model's tensors by name, each from a generator of its own, rounded to the run's type."""

    def __init__(self, case, seed):
        self.case, self.seed = case, seed
        self.dtype = {"bfloat16": torch.bfloat16, "float32": torch.float32}[case["dtype"]]
        self.tied = case["design"] in TIED or (case["design"] == "llama" and case["width"] == 2048)
        self.vocab = 128256 if case["design"] == "llama" else 32000
        # the stream's size: small where the head is the embedding's table, as such tables are
        self.size = 0.02 if case["design"] == "llama" and self.tied else 1.0

    def _generator(self, name):
        digest = hashlib.sha256(f"{self.seed}/{name}".encode()).digest()
        return torch.Generator(device=DEVICE).manual_seed(int.from_bytes(digest[:7], "little"))

    def _normal(self, name, shape, mean=0.0, std=1.0):
        return torch.empty(shape, device=DEVICE).normal_(mean, std, generator=self._generator(name))

    def _uniform(self, name, shape, low, high):
        return torch.empty(shape, device=DEVICE).uniform_(low, high, generator=self._generator(name))

    def follower(self, t):
        """The token that is to follow t: t itself where head and embedding are one table."""
        return t if self.tied else (t * 7919 + 12345) % self.vocab

    def _before(self):
        """[vocab]: the token that is followed by each token."""
        t = torch.arange(self.vocab, device=DEVICE)
        out = torch.empty_like(t)
        out[self.follower(t)] = t
        return out

    def _directions(self):
        """[experts, width], of length 1: what the routers of all layers look for."""
        d = self._normal("directions", (8, self.case["width"]))
        return d / d.norm(dim=1, keepdim=True)

    def _embedding(self, shape):
        e = self._normal("embed", shape, 0.0, self.size)
        if self.case["design"] in ("vupelorn", "mifidra", "sofinex", "tukedra"):  # which two experts a token goes to
            t, d = torch.arange(shape[0], device=DEVICE), self._directions()
            e += 14.0 * (d[t % 8] + d[(t + 3 + t // 8 % 3) % 8])
        return e

    def __call__(self, name, shape):
        return self._drawn(name, tuple(shape)).to(self.dtype)

    def _drawn(self, name, shape):
        last = name.rsplit(".", 1)[-1]
        branches = math.sqrt(2 * self.case["layers"])  # as many sublayers add to the stream
        if self.case["design"] == "llama":
            last = {"embed_tokens": "embed", "lm_head": "head", "o_proj": "o", "down_proj": "down"}.get(
                name.split(".")[-2], "norm" if "norm" in name else last)
        if last == "embed":
            return self._embedding(shape)
        if last == "head":
            return 0.02 * self._embedding(shape)[self._before()]
        if last == "bigram":
            return self._normal(name, shape, 0.0, 0.3)
        if last == "router":
            return self._normal(name, shape, 0.0, 0.001) + 0.8 * self._directions()
        if name.split(".")[-1] in ("norm1", "norm2", "norm1b", "norm2b"):
            if self.case["design"] == "sofinex":  # stored around zero
                return self._normal(name, shape, 0.0, 0.1)
            after = self.case["design"] in ("vupelorn", "puzonex") or last in ("norm1b", "norm2b")
            return self._normal(name, shape, 0.3 if after else 1.0, 0.03 if after else 0.1)
        if last == "norm":  # (Sofinex's gain on the way to the head is stored around zero too)
            return self._normal(name, shape, 0.0 if name == "final.norm" and self.case["design"] == "sofinex" else 1.0, 0.1)
        if last in ("out", "D", "alpha", "temp", "r1", "r2", "in") and (len(shape) < 2):
            return self._normal(name, shape, 1.0, 0.1)
        if last == "mix":
            return self._normal(name, shape, 0.0, 0.1) + torch.eye(*shape, device=DEVICE)
        if last == "conv":
            return self._normal(name, shape, 0.0, 0.35)
        if last == "A_log":  # decay rates of 1 to 16 a unit of step size, step sizes of 0.001 to 0.1
            return torch.log(self._uniform(name, shape, 1.0, 16.0))
        if last == "dt_bias" or name.endswith(".dt.b"):
            return torch.log(torch.expm1(torch.exp(self._uniform(name, shape, math.log(0.001), math.log(0.1)))))
        if name.endswith(".f.b"):  # forget gates that keep
            return self._uniform(name, shape, 3.0, 6.0)
        if last in ("sink", "rel"):
            return self._normal(name, shape, 0.0, 0.5)
        if last in ("lq1", "lk1", "lq2", "lk2", "correction"):
            return self._normal(name, shape, 0.0, 0.05 if last != "correction" else 0.01)
        if len(shape) < 2:  # biases
            return self._normal(name, shape, 0.0, 0.02)
        std = 0.02 if shape[1] >= 1024 else shape[1] ** -0.5
        if last in ("o", "down"):
            std *= self.size / branches
        if last in ("dt", "a2") and self.case["design"] != "vupelorn":  # steps stay near their biases
            std *= 0.3
        return self._normal(name, shape, 0.0, std)


# ---- what a program has in hand ---------------------------------------------------------------------------------
def _lengths(case):
    n = case["batch"]
    return [case["shortest"] + (case["longest"] - case["shortest"]) * (i * 7 % n if n % 7 else i) // max(1, n - 1)
            for i in range(n)]


def _prompts(case, seed, vocab):
    gen = torch.Generator().manual_seed(seed * 1000003 + 17)
    return [torch.randint(0, vocab, (n,), generator=gen).tolist() for n in _lengths(case)]


def _sampling(case, seed):
    if not case["sampled"]:
        return lq.SamplingParams(temperature=0.0)
    return lq.SamplingParams(temperature=0.5, top_k=40, top_p=0.95, repetition_penalty=1.05, seed=seed)


def prepare(case, seed):
    """An engine with its weights and an empty cache, the requests, and the backend that drives it."""
    weights = Weights(case, seed)
    config = _typed_config(case)
    model = DecoderModel(spec_from_config(config))
    tensors = {}
    for s in model.tensor_specs():
        if not s.optional:
            t = weights(s.name, s.shape)
            tensors[s.name] = t.float() if s.kind == "vector32" else t
    model.bind(tensors, BuildEnv(dtype=weights.dtype, device=torch.device(DEVICE), kernels=HipKernels()), consume=True)
    lengths = _lengths(case)
    room = sum(-(-(n + case["new"]) // 64) * 64 for n in lengths)
    engine = lq.Engine(model, model.env, max_tokens=room, max_slots=case["batch"], max_sequence_tokens=8192)
    prompts = _prompts(case, seed, weights.vocab)
    backend = EngineBackend(engine, _sampling(case, seed)) if case["kind"] == "chat" else None
    return {"case": case, "engine": engine, "backend": backend, "prompts": prompts}


def _run_prompt(engine, prompts, portions):
    slots = [engine.new_sequence() for _ in prompts]
    for k in range(portions):
        cuts = [(len(p) * k // portions, len(p) * (k + 1) // portions) for p in prompts]
        logits = engine.step([StepEntry(s, p[a:b], [b - a - 1] if k == portions - 1 else [])
                              for s, p, (a, b) in zip(slots, prompts, cuts)])
    for s in slots:
        engine.release(s)
    return {"logits": logits}


def _run_chat(backend, prompts, new):
    """What the generation loop does for one batch without stop ids; the last step is not queued ahead, because its
    logits are kept."""
    slots = [backend.new_sequence(r, p) for r, p in enumerate(prompts)]
    tokens = [backend.prefill(slots, prompts)]
    for i in range(1, new):
        backend.keep_logits = i == new - 1
        backend.expect_more(i < new - 2)
        tokens.append(backend.decode(slots, tokens[-1], i == 1))
    backend.keep_logits = False
    for s in slots:
        backend.release(s)
    return {"tokens": torch.tensor(tokens, dtype=torch.int32), "logits": backend.last_logits}


def run(state):
    case = state["case"]
    if case["kind"] == "prompt":
        return _run_prompt(state["engine"], state["prompts"], case["portions"])
    return _run_chat(state["backend"], state["prompts"], case["new"])


# ---- bytes and operations ---------------------------------------------------------------------------------------
def work(case):
    """Every weight once a step (of the experts as many as its tokens can choose), two operations a weight and token,
    causal attention's scores and values within their windows, the cached keys and values of a step's sequences."""
    config = _config(case)
    element = 2 if case["dtype"] == "bfloat16" else 4
    lengths = _lengths(case)
    experts = max([m["router"]["experts"] + m["router"].get("identity", 0) for m in
                   (l.get("mlp") or {} for l in config.get("layers", ())) if "router" in m], default=1)
    top = 2 if experts > 1 else 1
    fixed = chosen = head = 0
    for s in DecoderModel(spec_from_config(_typed_config(case))).tensor_specs():
        n = math.prod(s.shape)
        if s.optional or len(s.shape) < 2 or s.name == "bigram":
            continue
        if s.name in ("head", "lm_head.weight"):
            head = n
        elif s.name in ("embed", "model.embed_tokens.weight"):
            head = max(head, n) if case["design"] in TIED or case["design"] == "llama" and case["width"] == 2048 else head
        elif ".e" in s.name and s.name.split(".e")[-1].split(".")[0].isdigit():
            chosen += n
        else:
            fixed += n
    # attention: (score and value entries a pair of tokens, cached entries a token, window) of every layer
    pairs = []
    if case["design"] == "llama":
        hd, h, g = (64, 32, 8) if case["width"] == 2048 else (128, 32, 8)
        pairs = [(2 * h * hd, 2 * g * hd, None)] * case["layers"]
    for layer in config.get("layers", ()):
        m = layer["mixer"].get("left", layer["mixer"])
        if layer["type"].startswith("latent"):
            pairs.append((m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"]), m["kv_rank"] + m["rot_dim"], None))
        elif "scale" in m:
            maps = 2 if "diff" in m else 1
            pairs.append((maps * m["heads"] * (m["dim"] + m["vdim"]), m["kv_heads"] * (maps * m["dim"] + m["vdim"]),
                          (m.get("mask") or {}).get("size")))

    def seen(n, w):  # pairs of a prompt of n tokens
        return n * (n + 1) / 2 if w is None or n <= w else w * (w + 1) / 2 + (n - w) * w

    rows = sum(lengths)
    flops = 2.0 * rows * (fixed + chosen * top / experts) + 2.0 * case["batch"] * head
    flops += sum(2.0 * e * seen(n, w) for e, _, w in pairs for n in lengths)
    bytes_ = element * (case["portions"] * (fixed + chosen) + head) + 4.0 * case["batch"] * 128256
    steps = max(0, case["new"] - 1)
    flops += steps * 2.0 * case["batch"] * (fixed + chosen * top / experts + head)
    bytes_ += steps * element * (fixed + chosen * min(1.0, case["batch"] * top / experts) + head)
    for i in range(steps):
        for e, cached, w in pairs:
            n = sum(min(m + i + 1, w or m + i + 1) for m in lengths)
            flops, bytes_ = flops + 2.0 * e * n, bytes_ + element * cached * n
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    """About four times the distances from `exact` that were measured: 8e-7 in 32 bits; in bfloat16 5.6e-3 over the 32
    layers of the 8B shape, 1e-3 to 3.3e-3 over the others.  A vocabulary's largest error lies at 5 to 6 of these."""
    if case["dtype"] == "float32":
        return {"rel": 4e-6, "max": 4e-5, "differ": 0.0}
    if case["layers"] == 32:
        return {"rel": 0.022, "max": 0.13, "differ": 0.0}
    return {"rel": 0.013, "max": 0.08, "differ": 0.0}


# ---- the same in 64 bits ----------------------------------------------------------------------------------------
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _softplus(z):
    return torch.nn.functional.softplus(z, threshold=1e9)


def _gelu_tanh(z):
    return 0.5 * z * (1 + torch.tanh(math.sqrt(2 / math.pi) * (z + 0.044715 * z ** 3)))


def _frequencies(rot):
    """(frequencies of the rotated pairs, what cosine and sine are multiplied by)"""
    dims, base, sc = rot["dims"], rot["base"], rot.get("scaling")
    f = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=F64, device=DEVICE)
    if not sc:
        return f, 1.0
    if "low" in sc:  # blended by wavelength
        s = ((sc["original"] * f / (2 * math.pi) - sc["low"]) / (sc["high"] - sc["low"])).clamp(0, 1)
        return (1 - s) * f / sc["factor"] + s * f, 1.0

    def pair(turns):
        return dims * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(base))

    lo, hi = max(math.floor(pair(sc["fast"])), 0), min(math.ceil(pair(sc["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=F64, device=DEVICE) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


def _rotate(x, rot, interleaved):
    """x [batch, T, ..., dim], the first `dims` entries of every head turned by the token's position"""
    f, mag = _frequencies(rot)
    dims, half = rot["dims"], rot["dims"] // 2
    angle = torch.arange(x.shape[1], dtype=F64, device=DEVICE)[:, None] * f
    angle = angle.view([1, x.shape[1]] + [1] * (x.dim() - 3) + [half])
    c, s = torch.cos(angle) * mag, torch.sin(angle) * mag
    a, b = (slice(0, dims, 2), slice(1, dims, 2)) if interleaved else (slice(0, half), slice(half, dims))
    out = x.clone()
    out[..., a], out[..., b] = x[..., a] * c - x[..., b] * s, x[..., b] * c + x[..., a] * s
    return out


def _seen(T, mask=None, by_chunk=False):
    i = torch.arange(T, device=DEVICE)
    n = i[:, None] - i[None, :]
    seen = n >= 0
    if mask and by_chunk:
        seen &= (i // mask["size"])[:, None] == (i // mask["size"])[None, :]
    elif mask:
        seen &= (n < mask["size"]) | (i < mask.get("keep_first", 0))[None, :]
    return seen


def _attend(q, k, v, scale, seen, sink=None, shape_scores=None):
    """q [batch, T, H, d], k and v [batch, T, G, .] -> [batch, T, H, vdim]; `sink` [H]: one more term in the
    denominator; `shape_scores(h, scores)`: what a head does to its scores ahead of the softmax."""
    out = torch.empty(*q.shape[:3], v.shape[3], dtype=F64, device=DEVICE)
    hidden, per = ~seen, q.shape[2] // k.shape[2]
    for b in range(q.shape[0]):
        for h in range(q.shape[2]):
            score = (q[b, :, h] @ k[b, :, h // per].T).mul_(scale)
            if shape_scores is not None:
                score = shape_scores(h, score)
            score.masked_fill_(hidden, -math.inf)
            peak = score.amax(-1, keepdim=True)
            if sink is not None:
                peak = torch.maximum(peak, sink[h])
            total = score.sub_(peak).exp_().sum(-1, keepdim=True)
            if sink is not None:
                total = total + torch.exp(sink[h] - peak)
            out[b, :, h] = (score @ v[b, :, h // per]) / total
    return out


def _conv(x, taps, bias=None):
    n, T = taps.shape[1], x.shape[1]
    padded = torch.nn.functional.pad(x, (0, 0, n - 1, 0))
    y = sum(padded[:, j: j + T] * taps[:, j] for j in range(n))
    return _silu(y if bias is None else y + bias)


def _memory(q, k, v, decay, erase=None):
    """S <- decay S + k v^T, o = S^T q along the sequence; q and k [batch, T, H, d], v [batch, T, H, e], decay
    [batch, T, H, d or 1].  With `erase` [batch, T, H] (the delta rule) v is first made what S lacks of it."""
    S = torch.zeros(v.shape[0], v.shape[2], q.shape[3], v.shape[3], dtype=F64, device=DEVICE)
    out = torch.empty_like(v)
    for t in range(v.shape[1]):
        S.mul_(decay[:, t, :, :, None])
        new = v[:, t]
        if erase is not None:
            new = erase[:, t, :, None] * (new - (S * k[:, t, :, :, None]).sum(2))
        S.addcmul_(k[:, t, :, :, None], new[:, :, None, :])
        out[:, t] = (S * q[:, t, :, :, None]).sum(2)
    return out


def _over(x, heads):
    """The heads of groups repeated for every head that reads them."""
    return x.repeat_interleave(heads // x.shape[2], dim=2)


class Exact:
    """A design over whole sequences, all positions at once where that can be, step by step where not."""

    def __init__(self, case, seed):
        self.case, self.weights, self.config = case, Weights(case, seed), _config(case)
        self.eps = self.config["norm"]["eps"] if case["design"] != "llama" else self.config["rms_norm_eps"]
        self.kept = {}

    def w(self, name, *shape):
        return self.weights(name, shape).to(F64)

    def lin(self, x, name, out):
        return x @ self.w(name, out, x.shape[-1]).T

    def heads(self, x, name, heads, dim):
        return self.lin(x, name, heads * dim).view(*x.shape[:2], heads, dim)

    def flat(self, x):
        return x.reshape(*x.shape[:2], -1)

    # -- mixers: h [batch, T, width], p the tensors' prefix, m the mixer's configuration
    def vafodra_left(self, h, p, m):
        q, k, v = (self.heads(h, f"{p}.{n}", c, 128) for n, c in
                   (("q", m["heads"]), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
        zero = torch.zeros(m["heads"], dtype=F64, device=DEVICE)
        o = _attend(q, k, v, m["scale"], _seen(h.shape[1], m["mask"]), zero)
        return self.flat(o * torch.sigmoid(self.lin(h, p + ".g", m["heads"]))[..., None])

    def vafodra_right(self, h, p, m):
        H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
        inner, cut = H * P, [H * P, H * P + 2 * G * N, H]
        z, xbc, dt = self.lin(h, p + ".in", sum(cut)).split(cut, -1)
        xbc = _conv(xbc, self.w(p + ".conv", cut[1], m["conv"]), self.w(p + ".conv.b", cut[1]))
        x = xbc[..., :inner].reshape(*h.shape[:2], H, P)
        B, C = (_over(t.reshape(*h.shape[:2], G, N), H) for t in xbc[..., inner:].split(G * N, -1))
        dt = _softplus(dt + self.w(p + ".dt_bias", H))[..., None]
        y = _memory(C, B, dt * x, torch.exp(-torch.exp(self.w(p + ".A_log", H))[:, None] * dt))
        y = self.flat(y + self.w(p + ".D", H)[:, None] * x) * _silu(z)
        return _rms(y.view(*h.shape[:2], m["norm_groups"], -1), self.eps).reshape(y.shape) * self.w(p + ".norm", inner)

    def delta(self, h, p, m):
        """The gated delta rule: one decay a head (Vafodra) or one a key channel (Mifidra, Sofinex)."""
        H, G, d, e = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (_conv(self.lin(h, f"{p}.{n}", c), self.w(f"{p}.{n}.conv", c, m["conv"])).view(*h.shape[:2], -1, d)
                   for n, c in (("q", G * d), ("k", G * d), ("v", H * e)))
        q = _over(q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * d ** -0.5, H)
        k = _over(k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6), H)
        rate = torch.exp(self.w(p + ".A_log", H))[:, None]
        if "decay_rank" in m:
            low = self.lin(h, p + ".a1", m["decay_rank"])
            step = _softplus(self.lin(low, p + ".a2", H * d) + self.w(p + ".dt_bias", H * d)).view(*h.shape[:2], H, d)
            gate = torch.sigmoid(self.lin(self.lin(h, p + ".g1", m["gate_rank"]), p + ".g2", H * e))
        else:
            step = _softplus(self.lin(h, p + ".a", H) + self.w(p + ".dt_bias", H))[..., None]
            gate = _silu(self.lin(h, p + ".g", H * e))
        o = _memory(q, k, v, torch.exp(-rate * step), torch.sigmoid(self.lin(h, p + ".b", H)))
        return self.flat(_rms(o, self.eps) * self.w(p + ".norm", e)) * gate

    def gla(self, h, p, m):
        H, d, e = m["heads"], m["dim"], m["vdim"]
        q, k, v = (self.heads(h, f"{p}.{n}", H, c) for n, c in (("q", d), ("k", d), ("v", e)))
        z = self.lin(self.lin(h, p + ".a1", m["decay_rank"]), p + ".a2", H * d) + self.w(p + ".a2.b", H * d)
        decay = (torch.nn.functional.logsigmoid(z) / m["tau"]).exp().view(q.shape)
        o = _rms(_memory(q * d ** -0.5, k, v, decay), self.eps) * self.w(p + ".norm", e)
        return self.flat(o) * _silu(self.lin(h, p + ".g", H * e))

    def latent(self, h, p, m, i, interleaved):
        H, dn, dr, dv, r = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        if "kv_from" in m:
            c, kr = self.kept[m["kv_from"]]
        else:
            low = self.lin(h, p + ".dkv", r + dr)
            c = _rms(low[..., :r], self.eps) * self.w(p + ".dkv.norm", r)
            kr = _rotate(low[..., r:][:, :, None], m["rot"], interleaved)
            self.kept[i] = c, kr
        cq = _rms(self.lin(h, p + ".dq", m["q_rank"]), self.eps) * self.w(p + ".dq.norm", m["q_rank"])
        q = self.heads(cq, p + ".uq", H, dn + dr)
        q = torch.cat([q[..., :dn], _rotate(q[..., dn:], m["rot"], interleaved)], -1)
        k = torch.cat([self.heads(c, p + ".uk", H, dn), kr.expand(-1, -1, H, -1)], -1)
        return self.flat(_attend(q, k, self.heads(c, p + ".uv", H, dv), m["scale"], _seen(h.shape[1])))

    def normed_attention(self, h, p, m, interleaved, sink=None):
        """Mifidra's and Sofinex's: rotated, then q and k of unit mean square"""
        q, k, v = (self.heads(h, f"{p}.{n}", c, 128) for n, c in
                   (("q", m["heads"]), ("k", m["kv_heads"]), ("v", m["kv_heads"])))
        q, k = (_rms(_rotate(t, m["rot"], interleaved), self.eps) for t in (q, k))
        return self.flat(_attend(q, k, v, m["scale"], _seen(h.shape[1], m.get("mask")), sink))

    def differential(self, h, p, m):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        q, k = (_rotate(self.heads(h, f"{p}.{n}", 2 * c, d), m["rot"], False) for n, c in (("q", H), ("k", G)))
        v, seen = self.heads(h, p + ".v", G, m["vdim"]), _seen(h.shape[1], m["mask"])
        a, b = (_attend(q[:, :, j::2], k[:, :, j::2], v, m["scale"], seen) for j in (0, 1))
        lam = m["diff"]
        for sign, j in ((1, 1), (-1, 2)):
            lam = lam + sign * torch.exp((self.w(f"{p}.lq{j}", d) * self.w(f"{p}.lk{j}", d)).sum())
        return self.flat(_rms(a - lam * b, self.eps) * (1 - m["diff"]))

    def mamba(self, h, p, m):
        c, n, r = m["inner"], m["state"], m["dt_rank"]
        x, z = self.lin(h, p + ".in", 2 * c).split(c, -1)
        x = _conv(x, self.w(p + ".conv", c, m["conv"]), self.w(p + ".conv.b", c))
        low, B, C = self.lin(x, p + ".x", r + 2 * n).split([r, n, n], -1)
        dt = _softplus(self.lin(low, p + ".dt", c) + self.w(p + ".dt.b", c))
        A, S = -torch.exp(self.w(p + ".A_log", c, n)), torch.zeros(h.shape[0], c, n, dtype=F64, device=DEVICE)
        y = torch.empty_like(x)
        for t in range(h.shape[1]):
            S = torch.exp(dt[:, t, :, None] * A) * S + (dt[:, t] * x[:, t])[..., None] * B[:, t, None]
            y[:, t] = (S * C[:, t, None]).sum(-1)
        return (y + self.w(p + ".D", c) * x) * _silu(z)

    def puzonex_qk(self, h, p, m):
        H, G = m["heads"], m["kv_heads"]
        return (self.lin(h, f"{p}.{n}", c * 128) + self.w(f"{p}.{n}.b", c * 128)
                for n, c in (("q", H), ("k", G), ("v", G))[: 2 if "bias_rows" in m else 3])

    def puzonex_attention(self, h, p, m):
        shape, cap, H = (*h.shape[:2], -1, 128), m["softcap"], m["heads"]
        q, k, v = (_rms(t.view(shape), self.eps) for t in self.puzonex_qk(h, p, m))
        q, k = q * self.w(p + ".q.norm", 128), k * self.w(p + ".k.norm", 128)
        i = torch.arange(h.shape[1], dtype=F64, device=DEVICE)
        n = (i[:, None] - i[None, :]).clamp(min=0)
        r1, r2 = self.w(p + ".r1", H), self.w(p + ".r2", H)
        return self.flat(_attend(q, k, v, m["scale"], _seen(h.shape[1], m["mask"]), self.w(p + ".sink", H),
                                 lambda g, s: cap * torch.tanh(s / cap) - r1[g] * torch.log(1 + r2[g] * n)))

    def puzonex_left(self, h, p, m):
        T, H, shape, cap = h.shape[1], m["heads"], (*h.shape[:2], -1, 128), m["softcap"]
        q, k = self.puzonex_qk(h, p, m)
        v = k.view(shape)
        q, k = (_rms(t, self.eps) * self.w(f"{p}.{n}.norm", t.shape[-1]) for t, n in ((q, "q"), (k, "k")))
        rows, half = m["bias_rows"], m["bias_rows"] // 2
        bucket = [n if n < half else min(rows - 1, half + math.floor(
            math.log(n / half) / math.log(m["bias_max"] / half) * (rows - half) + 1e-9)) for n in range(T)]
        i = torch.arange(T, device=DEVICE)
        row = torch.tensor(bucket, device=DEVICE)[(i[:, None] - i[None, :]).clamp(min=0)]
        rel, temp = self.w(p + ".rel", rows, H), self.w(p + ".temp", H)
        o = _attend(q.view(shape), k.view(shape), v, m["scale"], _seen(T, m["mask"]), None,
                    lambda g, s: cap * torch.tanh(s * temp[g] / cap) + rel[:, g][row])
        o = self.flat(o) * torch.sigmoid(self.lin(h, p + ".g", H * 128))
        return self.lin(o, p + ".o", h.shape[-1]) + self.w(p + ".o.b", h.shape[-1])

    def mlstm(self, h, p, m):
        H, d, e, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k, v = (self.heads(h, f"{p}.{n}", H, c) for n, c in (("q", d), ("k", d), ("v", e)))
        take, keep = (cap * torch.tanh((self.lin(h, f"{p}.{n}", H) + self.w(f"{p}.{n}.b", H)) / cap) for n in "if")
        keep = torch.nn.functional.logsigmoid(keep)
        # the running maximum of the logarithms of the gates, by which both are divided
        top, m0 = [], torch.zeros_like(keep[:, 0])
        for t in range(h.shape[1]):
            m0 = torch.maximum(keep[:, t] + m0, take[:, t])
            top.append(m0)
        top = torch.stack(top, 1)
        before = torch.cat([torch.zeros_like(top[:, :1]), top[:, :-1]], 1)
        decay, take = torch.exp(keep + before - top)[..., None], torch.exp(take - top)[..., None]
        one = torch.ones_like(v[..., :1])
        o = _memory(q * d ** -0.5, k * take, torch.cat([v, one], -1), decay)  # (a column of ones: the normaliser)
        o = o[..., :-1] / (torch.maximum(o[..., -1:].abs(), torch.exp(-top)[..., None]) + 1e-6)
        o = self.flat(_rms(o, self.eps)) * self.w(p + ".norm", H * e)
        return o * torch.sigmoid(self.lin(h, p + ".g", H * e))

    def fixed_decay(self, h, p, m, rotated):
        H, d = m["heads"], m["dim"]
        q, k, v = (self.heads(h, f"{p}.{n}", H, d) for n in "qkv")
        gate = self.lin(h, p + ".g", H * d)
        decay = torch.tensor(m["decay"], dtype=F64, device=DEVICE)[:, None].expand(*h.shape[:2], H, 1)
        if rotated:
            q, k = _rotate(q, m["rot"], False), _rotate(k, m["rot"], False) * d ** -0.5
            return self.flat(_rms(_memory(q, k, v, decay), self.eps)) * _silu(gate)
        o = self.flat(_memory(_silu(q), _silu(k), _silu(v), decay))
        return _rms(o, self.eps) * self.w(p + ".norm", H * d) * torch.sigmoid(gate)

    def key_attention(self, h, p, m):
        q, k = (self.heads(h, f"{p}.{n}", c, 128) + self.w(f"{p}.{n}.b", c * 128).view(c, 128)
                for n, c in (("q", m["heads"]), ("k", m["kv_heads"])))
        qr, kr = (_rms(_rotate(t, m["rot"], True), self.eps) for t in (q, k))
        return self.flat(_attend(qr, kr, k, m["scale"], _seen(h.shape[1], m["mask"], by_chunk=True)))

    def mixer(self, h, i):
        layer, p, D = self.config["layers"][i], f"l{i}.mix", self.case["design"]
        m, kind, width = layer["mixer"], layer["type"], h.shape[-1]

        def out(x, q):
            return self.lin(x, q + ".o", width)

        if kind == "parallel" and D == "mifidra":
            return m["left_scale"] * out(self.normed_attention(h, p + ".left", m["left"], True), p + ".left") \
                + m["right_scale"] * out(self.delta(h, p + ".right", m["right"]), p + ".right")
        if kind == "parallel":
            if D == "vafodra":
                a = out(self.vafodra_left(h, p + ".left", m["left"]), p + ".left")
                b = out(self.vafodra_right(h, p + ".right", m["right"]), p + ".right")
            elif D == "sofinex":
                sink = self.w(p + ".left.sink", m["left"]["heads"])
                a = out(self.normed_attention(h, p + ".left", m["left"], False, sink), p + ".left")
                b = out(self.delta(h, p + ".right", m["right"]), p + ".right")
            else:
                a = self.puzonex_left(h, p + ".left", m["left"])
                b = out(self.mlstm(h, p + ".right", m["right"]), p + ".right")
            return 0.5 * (_rms(a, self.eps) * self.w(p + ".left.out", width)
                          + _rms(b, self.eps) * self.w(p + ".right.out", width))
        if kind.startswith("latent"):
            return out(self.latent(h, p, m, i, kind == "latent_attention_2"), p)
        if kind == "attention":
            return out({"sofinex": self.differential, "puzonex": self.puzonex_attention,
                        "tukedra": self.key_attention}[D](h, p, m), p)
        if kind in ("lightning", "retention"):
            return out(self.fixed_decay(h, p, m, kind == "retention"), p)
        return out({"delta": self.delta, "gla": self.gla, "mamba1": self.mamba}[kind](h, p, m), p)

    # -- feed-forwards
    def dense(self, h, p, m):
        D, ff, width = self.case["design"], m["ff"], h.shape[-1]
        up = self.lin(h, p + ".up", ff)
        if D == "sofinex":
            return self.lin(0.5 * up * (1 + torch.erf(up / math.sqrt(2.0))), p + ".down", width)
        gate = self.lin(h, p + ".gate", ff)
        if D == "mifidra":
            y = _silu(gate + self.w(p + ".gate.b", ff)) * (up + self.w(p + ".up.b", ff))
            return self.lin(y, p + ".down", width) + self.w(p + ".down.b", width)
        act = {"vafodra": torch.relu, "puzonex": _gelu_tanh, "tukedra": _silu}[D]
        return self.lin(act(gate) * up, p + ".down", width)

    def expert(self, h, p, m, weight):
        up, width = self.lin(h, p + ".up", m["ff"]), h.shape[-1]
        if self.case["design"] == "tukedra":
            return self.lin(torch.relu(up) ** 2 * weight, p + ".down", width)
        gate = self.lin(h, p + ".gate", m["ff"])
        return self.lin(_silu(gate) * up * weight, p + ".down", width)

    def limited_expert(self, h, p, m, weight):
        h, limit = weight * h, m["limit"]
        gate = self.lin(h, p + ".gate", m["ff"]).clamp(max=limit)
        up = self.lin(h, p + ".up", m["ff"]).clamp(-limit, limit)
        return self.lin(gate * torch.sigmoid(1.702 * gate) * (up + 1), p + ".down", h.shape[-1])

    def experts(self, h, p, m):
        D, shape = self.case["design"], h.shape
        h = h.reshape(-1, shape[-1])
        r = m["router"]
        n = r["experts"] + r.get("identity", 0)
        z = self.lin(h, p + ".router", n)
        score = {"vupelorn": torch.sigmoid, "mifidra": torch.sigmoid, "tukedra": lambda t: t,
                 "sofinex": lambda t: torch.softmax(t, -1)}[D](z)
        choice = score + self.w(p + ".correction", n) if D in ("mifidra", "sofinex") else score
        if "groups" in r:
            of_group = choice.view(len(h), r["groups"]["count"], -1)
            marks = of_group.topk(2, -1).values.sum(-1) if D == "mifidra" else of_group.amax(-1)
            kept = torch.zeros_like(marks).scatter_(1, marks.topk(r["groups"]["keep"], -1).indices, 1.0)
            choice = choice.masked_fill(kept.repeat_interleave(of_group.shape[2], 1) == 0, -math.inf)
        chosen = choice.topk(r["top"], -1).indices
        share = score.gather(1, chosen)
        share = torch.softmax(share, -1) if D == "tukedra" else share
        if D == "sofinex":
            share = share / (share.sum(-1, keepdim=True) + 1e-20)
        y = torch.zeros_like(h)
        run_expert = self.limited_expert if D == "vupelorn" else self.expert
        for e in range(n):
            at, place = (chosen == e).nonzero(as_tuple=True)
            if len(at):
                weight = share[at, place][:, None]
                y[at] += weight * h[at] if e >= r["experts"] else run_expert(h[at], f"{p}.e{e}", m["expert"], weight)
        if "shared" in m:
            open_ = torch.sigmoid(self.lin(h, p + ".shared.sg", 1)) if D == "sofinex" else 1.0
            y = y + self.expert(h, p + ".shared", m["shared"], open_)
        return y.view(shape)

    def feed_forward(self, h, i):
        m = self.config["layers"][i]["mlp"]
        return (self.dense if m["kind"] == "dense" else self.experts)(h, f"l{i}.mlp", m)

    # -- whole models: tokens [batch, T] -> what the final norm gives
    def llama(self, tokens):
        c, eps = self.config, self.eps
        width, H, G, d = c["hidden_size"], c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        rot, sc = {"base": c["rope_theta"], "dims": d}, c["rope_scaling"]
        if sc:
            rot["scaling"] = {"factor": sc["factor"], "low": sc["low_freq_factor"], "high": sc["high_freq_factor"],
                              "original": sc["original_max_position_embeddings"]}
        x = self.weights("model.embed_tokens.weight", (c["vocab_size"], width))[tokens].to(F64)
        seen = _seen(tokens.shape[1])
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = _rms(x, eps) * self.w(p + "input_layernorm.weight", width)
            q, k, v = (self.heads(h, f"{p}self_attn.{n}_proj.weight", k_, d) for n, k_ in (("q", H), ("k", G), ("v", G)))
            o = _attend(_rotate(q, rot, False), _rotate(k, rot, False), v, d ** -0.5, seen)
            x = x + self.lin(self.flat(o), p + "self_attn.o_proj.weight", width)
            h = _rms(x, eps) * self.w(p + "post_attention_layernorm.weight", width)
            gate, up = (self.lin(h, f"{p}mlp.{n}_proj.weight", c["intermediate_size"]) for n in ("gate", "up"))
            x = x + self.lin(_silu(gate) * up, p + "mlp.down_proj.weight", width)
        return _rms(x, eps) * self.w("model.norm.weight", width)

    def hybrid(self, tokens):
        c, D, eps, width = self.config, self.case["design"], self.eps, self.case["width"]
        x = self.weights("embed", (c["vocab"], width))[tokens].to(F64)
        if D == "vupelorn":
            bg = c["embedding"]["bigram"]
            row = (tokens[:, :-1] * bg["mul_prev"] + tokens[:, 1:] * bg["mul_cur"]) % bg["buckets"]
            row = torch.cat([torch.full_like(row[:, :1], bg["buckets"]) if row.shape[1] else
                             torch.full_like(tokens[:, :1], bg["buckets"]), row], 1)
            x = x + self.weights("bigram", (bg["buckets"] + 1, width))[row].to(F64)
        if D == "puzonex":  # sinusoids of the positions
            i = torch.arange(width, device=DEVICE)
            angle = torch.arange(tokens.shape[1], dtype=F64, device=DEVICE)[:, None] \
                * 10000.0 ** (-(i - i % 2).to(F64) / width)
            x = x + torch.where(i % 2 == 0, torch.sin(angle), torch.cos(angle))
        if D == "tukedra":
            return self.over_streams(x)
        for i in range(len(c["layers"])):
            if D == "vafodra":
                h = torch.tanh(self.w(f"l{i}.norm1.alpha") * x) * self.w(f"l{i}.norm1", width) \
                    + self.w(f"l{i}.norm1.b", width)
                x = x + c["residual_mult"] * (self.mixer(h, i) + self.feed_forward(h, i))
                continue
            for q, fn in (("1", self.mixer), ("2", self.feed_forward)):
                gain = self.w(f"l{i}.norm{q}", width)
                if D == "sofinex":
                    x = x + fn(_rms(x, eps) * (1 + gain), i)
                elif D == "mifidra":
                    x = x + _rms(fn(_rms(x, eps) * gain, i), eps) * self.w(f"l{i}.norm{q}b", width)
                else:
                    x = x + _rms(fn(x, i), eps) * gain
        gain = self.w("final.norm", width)
        if D == "vafodra":
            return torch.tanh(self.w("final.norm.alpha") * x) * gain + self.w("final.norm.b", width)
        return _rms(x, eps) * (1 + gain if D == "sofinex" else gain)

    def over_streams(self, x):
        width, n = self.case["width"], self.config["streams"]
        X = torch.stack([x] * n)
        for i in range(len(self.config["layers"])):
            for q, fn in (("1", self.mixer), ("2", self.feed_forward)):
                p = f"l{i}.hc{q}"
                read = torch.tensordot(self.w(p + ".in", n), X, 1)
                y = fn(_rms(read, self.eps) * self.w(f"l{i}.norm{q}", width), i)
                X = torch.tensordot(self.w(p + ".mix", n, n).T, X, 1) + self.w(p + ".out", n).view(n, 1, 1, 1) * y
        return _rms(X.sum(0), self.eps) * self.w("final.norm", width)

    def logits(self, tokens, rows):
        """`rows`: (sequence, position) of the wanted logits"""
        n = (self.llama if self.case["design"] == "llama" else self.hybrid)(tokens)
        n = torch.stack([n[b, t] for b, t in rows])
        names = ("model.embed_tokens.weight", "lm_head.weight") if self.case["design"] == "llama" else ("embed", "head")
        head = self.weights(names[0 if self.weights.tied else 1], (self.weights.vocab, self.case["width"]))
        out = torch.cat([n @ part.to(F64).T for part in head.split(16384)], 1) * self.config.get("logit_scale", 1.0)
        cap = self.config.get("logit_softcap")
        return cap * torch.tanh(out / cap) if cap else out


def exact(case, seed):
    ex = Exact(case, seed)
    prompts, new = _prompts(case, seed, ex.weights.vocab), case["new"]
    rows = [p + [0] * max(0, new - 1) for p in prompts]
    for b, p in enumerate(prompts):  # the tokens that are to follow
        for i in range(len(p), len(rows[b])):
            rows[b][i] = int(ex.weights.follower(rows[b][i - 1]))
    T = max(map(len, rows))
    tokens = torch.tensor([r + [0] * (T - len(r)) for r in rows], device=DEVICE)
    if case["kind"] == "prompt":
        return {"logits": ex.logits(tokens, [(b, len(p) - 1) for b, p in enumerate(prompts)])}
    asked = [(b, len(p) - 1 + i) for i in range(new) for b, p in enumerate(prompts)]
    logits = ex.logits(tokens, asked).view(new, len(prompts), -1)
    found = logits.argmax(-1).cpu()
    wanted = torch.tensor([[int(ex.weights.follower(rows[b][len(p) - 1 + i])) for b, p in enumerate(prompts)]
                           for i in range(new)])
    if not torch.equal(found, wanted):
        raise ValueError("a token that does not follow: the head's maximum is not clear")
    last = logits[-1]
    if case["sampled"]:  # the repetition penalty, on the last 64 tokens
        for b, p in enumerate(prompts):
            recent = torch.tensor(sorted(set(rows[b][: len(p) + new - 1][-64:])), device=DEVICE)
            z = last[b, recent]
            last[b, recent] = torch.where(z > 0, z / 1.05, z * 1.05)
    return {"tokens": found.to(torch.int32), "logits": last}
