"""The work that is timed when the speed of this package is judged: what its users have it do, through the
public entry points (`Castle`, `ops.castle_attention_hip`, `CastleLM`), from calls of a few hundred rows,
where launches and host work are all there is, to the longest sequences.

Kinds of case
  layer     one `Castle` module over whole sequences: mode "train" is a forward and a backward pass with every
            gradient, "forward" an evaluation under no_grad
  operator  the attention operator on six (B, H, L, d) tensors, for callers with projections of their own; mode
            "forward" also asks for the lookahead keys
  generate  one `Castle` module serving a request: a prompt through the parallel pass, then single-token steps
            on its cache
  lm_train  a `CastleLM`: loss of a batch of token sequences and every gradient
  lm_sample a `CastleLM`: a prompt extended by sampled tokens
"""
import math

import torch

from lookahead_keys_attention_amd import Castle, CastleLM
from lookahead_keys_attention_amd.ops import castle_attention_hip

DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
VOCABULARY = 256   # bytes: the language model is a character-level one
DEVICE = "cuda"


def _layer(name, mode, B, L, dim, heads, d, dtype, rotary=False, prenorm=False):
    return {"name": name, "kind": "layer", "mode": mode, "B": B, "L": L, "dim": dim, "heads": heads, "d": d,
            "dtype": dtype, "rotary": rotary, "prenorm": prenorm}


def _operator(name, mode, B, H, L, d, dtype, rotary=False):
    return {"name": name, "kind": "operator", "mode": mode, "B": B, "heads": H, "L": L, "d": d, "dtype": dtype, "rotary": rotary}


def _generate(name, B, prompt, steps, dim, heads, d, dtype, rotary=False, prenorm=False):
    return {"name": name, "kind": "generate", "B": B, "L": prompt, "steps": steps, "dim": dim, "heads": heads, "d": d,
            "dtype": dtype, "rotary": rotary, "prenorm": prenorm}


def _lm(name, kind, B, L, depth, dim, heads, d, steps=0):
    return {"name": name, "kind": kind, "B": B, "L": L, "steps": steps, "depth": depth, "dim": dim, "heads": heads, "d": d,
            "dtype": "bfloat16"}


def listed():
    return [
        # evaluating one short sequence with a small layer: latency of the host path and of the launches
        _layer("layer forward short", "forward", 1, 96, 128, 2, 64, "bfloat16", prenorm=True),
        # the default type of the module at the size of its smallest benchmark configuration
        _layer("layer train fp32 128", "train", 2, 128, 512, 8, 64, "float32"),
        # a batch of documents of no round length, rotary embedding and norm on
        _layer("layer train ragged 1000", "train", 3, 1000, 256, 4, 64, "bfloat16", rotary=True, prenorm=True),
        # the headline configuration
        _layer("layer train 4096", "train", 4, 4096, 512, 8, 64, "bfloat16"),
        # the long-context configuration
        _layer("layer train 16384 d128", "train", 1, 16384, 2048, 16, 128, "bfloat16"),
        # small heads in half precision, odd length, through the operator
        _operator("operator train d32 777", "train", 8, 4, 777, 32, "float16"),
        # wide heads at an ordinary training length
        _operator("operator train d128 2048", "train", 2, 16, 2048, 128, "bfloat16"),
        # full precision at an ordinary length
        _operator("operator train fp32 1024", "train", 2, 8, 1024, 64, "float32"),
        # batch serving: the decode configuration, prefill and the first 64 steps
        _generate("generate batch 32", 32, 2048, 64, 512, 8, 64, "bfloat16"),
        # one interactive stream
        _generate("generate single stream", 1, 300, 64, 512, 8, 64, "bfloat16", rotary=True, prenorm=True),
        # training a language model of the layer sizes of the language-model configuration
        _lm("lm train 16x1024", "lm_train", 16, 1024, 8, 512, 8, 64),
        # sampling from the 12-layer model of the language-model configuration
        _lm("lm sample 16x512", "lm_sample", 16, 512, 12, 512, 8, 64, steps=48),
    ]


# A drawn case costs at most about what the longest listed one does.  The rates are rough throughputs of an
# MI355X on this work (flop/s), only there to bound the draw.
_ROUGH_RATE = {"float32": 3e13, "bfloat16": 2e14, "float16": 2e14}
_LONGEST_S = 0.012


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(["layer"] * 4 + ["operator"] * 3 + ["generate"] * 3 + ["lm_train", "lm_sample"])
        dtype = rng.choice(["bfloat16", "bfloat16", "float32", "float16"])
        d = rng.choice([32, 64, 64, 128]) if dtype != "float32" else rng.choice([32, 64])
        heads = rng.choice([1, 2, 4, 6, 8, 12, 16])
        dim = heads * d if rng.random() < 0.6 else rng.choice([128, 256, 384, 512, 768, 1024])
        rotary, prenorm = rng.random() < 0.5, rng.random() < 0.5
        if kind == "layer":
            case = _layer("", rng.choice(["train", "train", "forward"]), _log_int(rng, 1, 32), _log_int(rng, 20, 12000), dim, heads, d, dtype, rotary, prenorm)
        elif kind == "operator":
            case = _operator("", rng.choice(["train", "train", "forward"]), _log_int(rng, 1, 32), heads, _log_int(rng, 20, 12000), d, dtype, rotary)
        elif kind == "generate":
            case = _generate("", _log_int(rng, 1, 48), _log_int(rng, 16, 4000), rng.randint(24, 96), dim, heads, d, dtype, rotary, prenorm)
        else:
            d, heads = rng.choice([32, 64]), rng.choice([4, 6, 8])
            B, L = _log_int(rng, 1, 24), _log_int(rng, 64, 1500)
            case = _lm("", kind, B, L, rng.randint(2, 8), d * heads, heads, d, steps=rng.randint(16, 64) if kind == "lm_sample" else 0)
        tokens = case["B"] * (case["L"] + case.get("steps", 0))
        w = work({**case, "name": "drawn"})
        if tokens <= 70000 and w["flops"] / _ROUGH_RATE[case["dtype"]] + w["bytes"] / 4e12 <= _LONGEST_S:
            del case["name"]
            return case


def _module(case):
    with torch.device(DEVICE):
        return Castle(case["dim"], heads=case["heads"], dim_head=case["d"], rotary_emb=case["rotary"],
                      prenorm=case["prenorm"]).to(DTYPES[case["dtype"]])


def prepare(case, seed):
    torch.manual_seed(seed)   # the modules draw their default initialisation from it
    g = torch.Generator(device=DEVICE).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    B, L = case["B"], case["L"]

    def normal(*shape, std=1.0):
        return (torch.randn(*shape, generator=g, device=DEVICE) * std).to(dtype)

    state = {"case": case}
    kind = case["kind"]
    if kind == "layer":
        train = case["mode"] == "train"
        state["model"] = _module(case).train(train)
        state["x"] = normal(B, L, case["dim"]).requires_grad_(train)
        state["gy"] = normal(B, L, case["dim"]) if train else None
    elif kind == "operator":
        train = case["mode"] == "train"
        shape = (B, case["heads"], L, case["d"])
        # a projection of unit-normal rows by default-initialised weights has a standard deviation of 0.58
        state["six"] = [normal(*shape, std=0.6).requires_grad_(train) for _ in range(6)]
        state["gy"] = normal(*shape) if train else None
    elif kind == "generate":
        state["model"] = _module(case).eval()
        state["prompt"] = normal(B, L, case["dim"])
        state["tokens"] = normal(B, case["steps"], case["dim"])
    else:
        # The embedding is shared with the logits, as in the language-model configuration.
        with torch.device(DEVICE):
            model = CastleLM(num_tokens=VOCABULARY, dim=case["dim"], depth=case["depth"], heads=case["heads"], dim_head=case["d"],
                             tie_embedding=True).to(dtype)
        state["model"] = model.train(kind == "lm_train")
        n = L + 1 if kind == "lm_train" else L
        state["ids"] = torch.randint(0, VOCABULARY, (B, n), generator=g, device=DEVICE)
        state["seed"], state["generator"] = seed, torch.Generator(device=DEVICE)
    return state


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "layer":
        model, x = state["model"], state["x"]
        if case["mode"] == "forward":
            with torch.no_grad():
                return model(x)
        model.zero_grad(set_to_none=True)
        x.grad = None
        y = model(x)
        y.backward(state["gy"])
        return [y, x.grad] + [p.grad for p in model.parameters() if p.requires_grad]
    if kind == "operator":
        six, scale = state["six"], case["d"] ** -0.5
        if case["mode"] == "forward":
            with torch.no_grad():
                return castle_attention_hip(*six, scale, True, rotary=case["rotary"])
        for t in six:
            t.grad = None
        out = castle_attention_hip(*six, scale, rotary=case["rotary"])
        out.backward(state["gy"])
        return [out] + [t.grad for t in six]
    if kind == "generate":
        model, tokens = state["model"], state["tokens"]
        with torch.no_grad():
            y, cache = model(state["prompt"], return_next_cache=True)
            outs = [y]
            for i in range(case["steps"]):
                y, cache = model(tokens[:, i:i + 1], cache=cache)
                outs.append(y)
            return [outs[0], torch.cat(outs[1:], dim=1), cache]
    if kind == "lm_train":
        model = state["model"]
        model.zero_grad(set_to_none=True)
        loss = model(state["ids"], return_loss=True)
        loss.backward()
        return [loss] + [p.grad for p in model.parameters() if p.requires_grad]
    generator = state["generator"].manual_seed(state["seed"])
    return state["model"].sample(state["ids"], case["L"] + case["steps"], generator=generator)


def _core_flops(B, H, L, d, contractions):
    """Contractions of the attention core: B H L^2 d flop each (2 d per causal pair): 5 forward, 14 backward."""
    return contractions * float(B) * H * L * L * d


def work(case):
    es = DTYPES[case["dtype"]].itemsize
    B, L, H, d = case["B"], case["L"], case["heads"], case["d"]
    kind, inner = case["kind"], case["heads"] * case["d"]
    rows = float(B) * L
    if kind == "operator":
        n = rows * inner * es
        if case["mode"] == "forward":
            return {"bytes": 8 * n, "flops": _core_flops(B, H, L, d, 5)}          # six operands, out, lookahead keys
        return {"bytes": 14 * n, "flops": _core_flops(B, H, L, d, 19)}            # six operands, out, dout, six gradients
    dim = case["dim"]
    weights = 7.0 * inner * dim * es
    gemm = 2.0 * rows * dim * 7 * inner
    if kind == "layer":
        if case["mode"] == "forward":
            return {"bytes": 2 * rows * dim * es + weights, "flops": _core_flops(B, H, L, d, 5) + gemm}
        return {"bytes": 4 * rows * dim * es + 2 * weights, "flops": _core_flops(B, H, L, d, 19) + 3 * gemm}
    steps = case["steps"]
    # one step reads the four cached tensors and the weights; B rows in and out, one row appended to each tensor
    cached = sum(4.0 * B * H * (L + i) * d * es for i in range(steps))
    if kind == "generate":
        step = weights + 2.0 * B * dim * es + 4.0 * B * inner * es
        return {"bytes": 2 * rows * dim * es + weights + 4 * rows * inner * es + cached + steps * step,
                "flops": _core_flops(B, H, L, d, 5) + gemm + steps * 2.0 * B * dim * 7 * inner + 2.0 * cached / es}
    depth = case["depth"]
    weights = depth * (weights + 8.0 * dim * dim * es) + VOCABULARY * dim * es
    gemm = depth * (gemm + 2.0 * rows * dim * 8 * dim) + 2.0 * rows * dim * VOCABULARY
    if kind == "lm_train":
        return {"bytes": 8 * rows + 2 * weights, "flops": depth * _core_flops(B, H, L, d, 19) + 3 * gemm}
    return {"bytes": 8 * rows + weights + depth * (4 * rows * inner * es + cached) + steps * weights,
            "flops": depth * (_core_flops(B, H, L, d, 5) + 2.0 * cached / es) + gemm * (1 + steps / L)}


def tolerance(case):
    if case["kind"] == "lm_sample":
        return "exact"   # token numbers; the shared embedding leaves no near ties
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 1e-2}   # 32-bit sums behind exponentials of scores of several tens
    if case["kind"] == "lm_train":
        return {"rel": 2e-2, "max": 0.8}    # 16-bit roundings through all layers and back
    return {"rel": 1e-2, "max": 0.4}        # 16-bit operands and results, 32-bit accumulation
