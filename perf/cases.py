"""The work that a program on this framework has it do, as timed cases: a decoder's prompt, its incremental
steps, its beam-search steps, and the packing of weights that are already on the GPU.

Every decoder case runs through Int8Decoder (LlamaMmha / BaichuanMmha, GatedFeedForwardNetworkInt8, LayerNorm
and the fp16 head) at the widths of the two configurations the repository is built for -- 4096 / 32 heads /
11008 with rotary positions and 5120 / 40 heads / 13696 with ALiBi -- or at smaller generic widths with the
other head sizes.  A case takes a few layers of such a decoder: enough distinct weights and cache rows that
every pass streams them from HBM as the whole decoder would.
"""
import math

import torch

from eet_amd import decoder as D
from eet_amd import ops

# name -> hidden, heads, d_ff, vocab, ALiBi instead of rotary positions
WIDTHS = {
    "4096": (4096, 32, 11008, 32000, False),      # LLaMA-7B
    "5120": (5120, 40, 13696, 64000, True),       # Baichuan-13B
    "3072": (3072, 32, 8192, 32000, False),       # head size 96
    "2048": (2048, 32, 5632, 32000, False),       # head size 64
    "1024": (1024, 16, 2816, 8000, False),        # head size 64, a small decoder
}


def listed():
    return [
        # one user of a small decoder, a few dozen tokens in: launches and host work are all there is
        dict(name="decode_small_b1", kind="decode", width="1024", layers=6, batch=1, context=75, new=4, padded=False),
        # one chat user deep into a long context: few heads to spread over the chip
        dict(name="decode_4096_b1_long", kind="decode", width="4096", layers=6, batch=1, context=3001, new=4, padded=False),
        # the serving batch of the 7B configuration, 1024 prompt tokens
        dict(name="decode_4096_b8", kind="decode", width="4096", layers=8, batch=8, context=1024, new=4, padded=False),
        # a loaded server: more sequences than the decode kernels' 32 rows, left-padded to one length
        dict(name="decode_4096_b56", kind="decode", width="4096", layers=4, batch=56, context=513, new=4, padded=True),
        # the serving batch of the 13B configuration: ALiBi, 2048 prompt tokens
        dict(name="decode_5120_b32", kind="decode", width="5120", layers=3, batch=32, context=2048, new=4, padded=False),
        # beam search: 4 prompts x 4 beams, the cache follows the surviving beams on every step
        dict(name="beam_4096_4x4", kind="beam", width="4096", layers=4, batch=4, beams=4, context=400, new=6),
        # a short question
        dict(name="prompt_4096_1x45", kind="prompt", width="4096", layers=6, batch=1, context=45, padded=False),
        # two users' prompts of different lengths, left-padded
        dict(name="prompt_4096_2x203", kind="prompt", width="4096", layers=6, batch=2, context=203, padded=True),
        # head size 64, four prompts of an ordinary length
        dict(name="prompt_2048_4x500", kind="prompt", width="2048", layers=6, batch=4, context=500, padded=False),
        # one long ALiBi prompt: the 2048-token GEMMs of the 13B configuration
        dict(name="prompt_5120_1x2048", kind="prompt", width="5120", layers=3, batch=1, context=2048, padded=False),
        # the prompt batch of the 7B configuration
        dict(name="prompt_4096_8x1024", kind="prompt", width="4096", layers=3, batch=8, context=1024, padded=False),
        # packing a checkpoint's matrix on the GPU
        dict(name="quantize_11008x4096", kind="quantize", rows=11008, cols=4096, dtype="float16", unprocessed=False),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / 1e15


def draw(rng):
    """One more case of the same ranges: batch 1 .. 64 and context 16 .. 4096 in decode, up to 16 beam rows,
    prompts of 16 .. 2048 tokens and up to 8192 tokens in a call, matrices of 1024 .. 16384 rows and columns."""
    most = max(_cost(c) for c in listed())
    while True:
        kind = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "prompt", "beam", "quantize"])
        if kind == "quantize":
            case = dict(kind=kind, rows=64 * _log_int(rng, 16, 256), cols=16 * _log_int(rng, 64, 1024),
                        dtype=rng.choice(["float16", "float16", "float32"]), unprocessed=rng.random() < 0.25)
        else:
            case = dict(kind=kind, width=rng.choice(["4096", "4096", "5120", "3072", "2048", "1024"]),
                        layers=rng.randint(2, 6))
            if kind == "decode":
                case.update(batch=_log_int(rng, 1, 64), context=_log_int(rng, 16, 4096), new=rng.randint(2, 4),
                            padded=rng.random() < 0.3)
            elif kind == "beam":
                beams = rng.randint(2, 5)
                case.update(beams=beams, batch=rng.randint(1, 16 // beams), context=_log_int(rng, 16, 1024),
                            new=rng.randint(3, 6))
            else:
                case.update(batch=_log_int(rng, 1, 8), context=_log_int(rng, 16, 2048), padded=rng.random() < 0.3)
                if case["batch"] * case["context"] > 8192:
                    continue
        if _cost(case) <= most:
            return case


def _pads(case):
    """Left padding of a padded batch: sequence b lacks b * 37 mod half the context (the first is whole)."""
    half = max(1, case["context"] // 2)
    return [(b * 37) % half for b in range(case["batch"])]


def _decoder(case, rows, gen):
    hidden, heads, d_ff, vocab, alibi = WIDTHS[case["width"]]
    new = case.get("new", 0)
    cfg = D.DecoderConfig(num_layers=case["layers"], hidden=hidden, heads=heads, d_ff=d_ff, vocab=vocab, alibi=alibi,
                          max_batch=rows, max_prompt=case["context"], max_full_seq=case["context"] + max(new, 1))

    def normal(*shape, std=0.02):
        return torch.randn(*shape, generator=gen, device="cuda:0", dtype=torch.float16) * std
    sd = {}
    for i in range(cfg.num_layers):
        pre = f"layer.{i}."
        for name, k, n in (("self_attn.qkv_proj", hidden, 3 * hidden), ("self_attn.out_proj", hidden, hidden),
                           ("ffn.intermediate_0", hidden, d_ff), ("ffn.intermediate_1", hidden, d_ff),
                           ("ffn.output", d_ff, hidden)):
            sd[pre + name + ".weight"], sd[pre + name + ".scale"] = ops.quant_weights_device(normal(k, n))
        for name in ("self_attn.layernorm.weight", "ffn.layernorm.weight"):
            sd[pre + name] = 1 + normal(hidden, std=0.1)
    sd["embed_tokens.weight"] = normal(vocab, hidden)
    sd["norm.weight"] = 1 + normal(hidden, std=0.1)
    sd["lm_head.weight"] = normal(vocab, hidden)
    return D.Int8Decoder(cfg, sd, device="cuda:0")


@torch.no_grad()
def prepare(case, seed):
    gen = torch.Generator(device="cuda:0").manual_seed(seed)
    if case["kind"] == "quantize":
        w = torch.randn(case["rows"], case["cols"], generator=gen, device="cuda:0") * 0.02
        return {"kind": "quantize", "weight": w.to(getattr(torch, case["dtype"])), "unprocessed": case["unprocessed"]}
    rows = case["batch"] * case.get("beams", 1)
    model = _decoder(case, rows, gen)
    vocab, context, new = model.cfg.vocab, case["context"], case.get("new", 0)

    def tokens(*shape):
        return torch.randint(0, vocab, shape, generator=gen, device="cuda:0")
    state = {"kind": case["kind"], "model": model, "context": context, "mask": None}
    if case.get("padded"):
        pads = torch.tensor(_pads(case), device="cuda:0")
        state["mask"] = (torch.arange(context, device="cuda:0")[None, :] >= pads[:, None]).long()
    if case["kind"] == "prompt":
        state["ids"] = tokens(rows, context)
        return state
    state["ids"] = [tokens(rows, 1) for _ in range(new)]
    if case["kind"] == "beam":
        first = torch.arange(rows, device="cuda:0") // case["beams"] * case["beams"]
        state["order"] = [first + torch.randint(0, case["beams"], (rows,), generator=gen, device="cuda:0")
                          for _ in range(new)]
    model(tokens(rows, context), True, state["mask"])      # the prompt fills the caches
    return state


@torch.no_grad()
def run(state):
    if state["kind"] == "quantize":
        return ops.quant_weights_device(state["weight"], state["unprocessed"])
    model = state["model"]
    if state["kind"] == "prompt":
        return model(state["ids"], True, state["mask"])    # hidden states of every position
    # the sequence goes on from the end of its prompt, with tokens given
    for attn, _ in model.layers:
        attn.step = state["context"]
    if model.cfg.alibi:
        model.past = state["context"]
    out = []
    for i, ids in enumerate(state["ids"]):
        if state["kind"] == "beam":
            model.reorder_state = state["order"][i]
        out.append(model.logits(ids, False, state["mask"]))
    return out


def work(case):
    if case["kind"] == "quantize":
        size = 2 if case["dtype"] == "float16" else 4
        n = case["rows"] * case["cols"]
        return {"bytes": n * (size + (2 if case["unprocessed"] else 1)) + size * case["cols"], "flops": 2 * n}
    hidden, heads, d_ff, vocab, _ = WIDTHS[case["width"]]
    layers, rows, context = case["layers"], case["batch"] * case.get("beams", 1), case["context"]
    params = 4 * hidden * hidden + 3 * hidden * d_ff
    weights = layers * (params + 2 * (7 * hidden + 2 * d_ff))            # int8 weights, fp16 scales and norms
    pads = sum(_pads(case)) if case.get("padded") else 0
    if case["kind"] == "prompt":
        seen = sum((context - p) * (context - p + 1) / 2 for p in (_pads(case) if pads else [0] * rows))
        tokens = rows * context
        return {"bytes": weights + layers * 2 * tokens * hidden * 2 + 2 * tokens * hidden * 2 + tokens * 8,
                "flops": layers * (2 * tokens * params + 4 * seen * hidden)}
    total_bytes = total_flops = 0
    for i in range(case["new"]):
        cached = rows * (context + i + 1) - pads
        total_bytes += weights + layers * 2 * cached * hidden * 2 + 2 * vocab * hidden + 2 * rows * (vocab + hidden)
        total_flops += layers * (2 * rows * params + 4 * cached * hidden) + 2 * rows * vocab * hidden
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    if case["kind"] == "quantize":
        return "exact"
    # Two correct evaluations at this precision -- every launch's sums taken in another order (other tiles, another
    # split of the cached rows, the other prompt-attention kernel) -- differ by up to 2.3e-3 in the 2-norm and
    # 1.3e-2 at one element: the fp16 buffers between the launches round at different points.
    return {"rel": 1e-2, "max": 6e-2}
