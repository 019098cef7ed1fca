"""Attention work as a user's program calls it, for timing: forward calls of the variants, decoding steps over a cache,
training steps (forward and gradients), and the Evoformer's row attention, inference and training.

`listed()` names fixed sizes, `draw(rng)` gives further ones of the same ranges; `prepare` makes what a program has in
hand before the call (operands on the GPU), `run` is one pass through the public entry points.
"""
import math

import torch

from flashlight_amd import attention_variants as A
from flashlight_amd import workloads as W

TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
# no drawn case asks for more than the largest listed one
MAX_FLOPS, MAX_BYTES = 1.1e12, 6.0e8


def listed():
    return [
        # one short causal call (the smallest configuration of the test suite): launch latency, a part that is not full
        _fwd("causal_512", "causal", 2, 8, 8, 512, 64),
        # unmasked attention at the headline shape of the benchmark
        _fwd("vanilla_4096", "vanilla", 4, 16, 16, 4096, 128),
        # a language model's prefill: grouped heads, ALiBi and soft-cap under the causal mask
        _fwd("alibi_softcap_8192", "alibi_softcap", 2, 32, 8, 8192, 128, softcap=50.0),
        # local attention: few keys per query, bound by memory rather than by the products
        _fwd("sliding_4096", "sliding", 4, 16, 16, 4096, 128, window=256),
        # packed documents in one long row; the ids are new with every call, as in a data loader's batches
        _fwd("document_16384", "document", 1, 16, 16, 16384, 64),
        # differential attention: two softmax branches over values twice as wide
        _fwd("diff_4096", "diff", 2, 16, 16, 4096, 64),
        # one decoding step of one sequence with a long cache
        _decode("decode_1x32768", 1, 32, 8, 1, 32768, 128),
        # one decoding step of a batch whose caches lie in longer buffers and have an odd length
        _decode("decode_8x3001", 8, 32, 8, 1, 3001, 128, buffer=4096),
        # a pre-training step's attention, forward and gradients
        _train("train_causal_4096", "causal", 4, 16, 16, 4096, 128),
        # fine-tuning on short ragged batches in fp16: grouped heads, operands as a projection leaves them ([B, S, H, D])
        _train("train_prefix_1000", "prefix", 3, 16, 4, 1000, 64, dtype="fp16", prefix=200, layout="bshd"),
        # MSA row attention with pair bias and gate, inference
        _evo("evoformer_256x384", False, 1, 256, 384, 8, 32, gate=True, mask=False),
        # the same module in training, with a padding mask: gradients of every operand, the pair bias and the gate included
        _evo("evoformer_train_128x256", True, 1, 128, 256, 8, 32, gate=True, mask=True),
    ]


def _fwd(name, variant, B, Hq, Hkv, S, D, dtype="bf16", layout="bhsd", softcap=0.0, window=0, prefix=0):
    return {"name": name, "kind": "forward", "variant": variant, "B": B, "Hq": Hq, "Hkv": Hkv, "S": S, "D": D, "dtype": dtype,
            "layout": layout, "softcap": softcap, "window": window, "prefix": prefix}


def _train(name, variant, B, Hq, Hkv, S, D, **kw):
    return dict(_fwd(name, variant, B, Hq, Hkv, S, D, **kw), kind="train")


def _decode(name, B, Hq, Hkv, Lq, Lk, D, dtype="bf16", buffer=0):
    return {"name": name, "kind": "decode", "B": B, "Hq": Hq, "Hkv": Hkv, "Lq": Lq, "Lk": Lk, "D": D, "dtype": dtype,
            "buffer": buffer}  # buffer: allocated length of the caches (0: exactly Lk)


def _evo(name, train, B, N, S, H, D, dtype="bf16", gate=True, mask=False):
    return {"name": name, "kind": "evoformer", "train": train, "B": B, "N": N, "S": S, "H": H, "D": D, "dtype": dtype,
            "gate": gate, "mask": mask}


# ---- drawn cases ---------------------------------------------------------------------------------------------------------

def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            del c["name"]
            return c


def _draw(rng):
    kind = rng.choice(("forward", "forward", "forward", "train", "train", "decode", "decode", "evoformer"))
    dtype = "fp16" if rng.random() < 0.2 else "bf16"
    if kind == "decode":
        Hkv = rng.choice((4, 8, 16, 32))
        group = rng.choice((1, 4, 8))
        Lk = _log(rng, 128, 65536)
        return _decode("", _log(rng, 1, 128), Hkv * group, Hkv, rng.choice((1, 1, 1, 2, 4)), Lk, rng.choice((64, 128)), dtype,
                       buffer=rng.choice((0, 1)) * (1 << (Lk - 1).bit_length()))
    if kind == "evoformer":
        S = _log(rng, 64, 512)
        return _evo("", rng.random() < 0.5, rng.choice((1, 1, 2)), _log(rng, 16, 256), S if rng.random() < 0.5 else (S + 31) // 32 * 32,
                    rng.choice((4, 8)), rng.choice((32, 32, 64)), dtype, gate=rng.random() < 0.7, mask=rng.random() < 0.5)
    variants = ["vanilla", "causal", "sliding", "prefix", "document", "alibi_softcap"] + (["diff"] if kind == "forward" else [])
    variant = rng.choice(variants)
    S = _log(rng, 96, 16384 if kind == "forward" else 8192)
    D = 64 if variant == "diff" else rng.choice((64, 128))
    Hq = rng.choice((8, 16, 32))
    Hkv = Hq if variant == "diff" else Hq // rng.choice((1, 4, 8))
    make = _fwd if kind == "forward" else _train
    return make("", variant, _log(rng, 1, 16), Hq, Hkv, S, D, dtype=dtype, layout=rng.choice(("bhsd", "bshd")),
                softcap=rng.choice((30.0, 50.0)) if variant == "alibi_softcap" else 0.0,
                window=rng.randint(64, 1024) if variant == "sliding" else 0,
                prefix=rng.randint(1, S) if variant == "prefix" else 0)


# ---- operands ------------------------------------------------------------------------------------------------------------

def _doc_lengths(c, seed):
    S = c["S"]
    return W.document_lengths(S, seed, max(1, min(512, S // 8)), max(2, min(4096, S // 2)))


def prepare(case, seed):
    c, g, dtype = case, torch.Generator(device="cuda").manual_seed(int(seed)), TYPES[case["dtype"]]

    def randn(*shape):
        return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).to(dtype)

    if c["kind"] == "decode":
        rows = max(c["buffer"], c["Lk"])
        k, v = (randn(c["B"], c["Hkv"], rows, c["D"])[:, :, :c["Lk"]] for _ in range(2))
        return {"case": c, "q": randn(c["B"], c["Hq"], c["Lq"], c["D"]), "k": k, "v": v}
    if c["kind"] == "evoformer":
        B, N, S, H, D = c["B"], c["N"], c["S"], c["H"], c["D"]
        s = {"case": c, "q": randn(B, N, S, H, D), "k": randn(B, N, S, H, D), "v": randn(B, N, S, H, D),
             "pair": randn(B, 1, H, S, S), "mask": None, "gate": randn(B, N, S, H, D) if c["gate"] else None}
        if c["mask"]:  # a tenth of the residues is padding, another tenth missing here and there
            hidden = torch.rand(B, N, 1, 1, S, generator=g, device="cuda") < 0.1
            hidden[..., S - S // 10:] = True
            hidden[..., 0] = False
            s["mask"] = torch.zeros(B, N, 1, 1, S, device="cuda", dtype=dtype).masked_fill_(hidden, -1e9 if dtype == torch.bfloat16 else -6e4)
        if c["train"]:
            s["leaves"] = [s[n].requires_grad_(True) for n in ("q", "k", "v", "pair", "gate") if s[n] is not None]
            s["dout"] = randn(B, N, S, H, D)
        return s
    B, Hq, Hkv, S, D = c["B"], c["Hq"], c["Hkv"], c["S"], c["D"]

    def operand(heads, width):
        if c["layout"] == "bshd":
            return randn(B, S, heads, width).transpose(1, 2)
        return randn(B, heads, S, width)

    two = 2 if c["variant"] == "diff" else 1
    s = {"case": c, "q": operand(two * Hq, D), "k": operand(two * Hkv, D), "v": operand(Hkv, two * D)}
    if c["variant"] == "document":
        s["ids"] = W.document_ids(_doc_lengths(c, int(seed)), B, "cuda")
    if c["variant"] == "alibi_softcap":
        s["alibi"] = A.generate_alibi_bias_pytorch(Hq)
    if c["kind"] == "train":
        s["leaves"] = [s[n].requires_grad_(True) for n in ("q", "k", "v")]
        s["dout"] = operand(Hq, D)
    return s


def _attend(s):
    c, q, k, v = s["case"], s["q"], s["k"], s["v"]
    gqa, variant = c["Hq"] != c["Hkv"], c["variant"]
    if variant == "vanilla":
        out = A.attention_pytorch(q, k, v, enable_gqa=gqa)
    elif variant == "causal":
        out = A.attention_pytorch_causal(q, k, v, enable_gqa=gqa)
    elif variant == "sliding":
        out = A.attention_pytorch_sliding_window(q, k, v, window_size=c["window"], enable_gqa=gqa)
    elif variant == "prefix":
        out = A.attention_pytorch_prefix_lm(q, k, v, prefix_lengths=c["prefix"], enable_gqa=gqa)
    elif variant == "document":
        out = A.attention_pytorch_document_mask(q, k, v, s["ids"], enable_gqa=gqa, is_causal=True)
    elif variant == "alibi_softcap":
        out = A.attention_pytorch_alibi(q, k, v, score_mod=s["alibi"], is_causal=True, enable_gqa=gqa, softcap=c["softcap"])
    else:
        out = A.diffattn(q, k, v, lambda_full=0.8, is_causal=True)
    return out


def run(state):
    c = state["case"]
    if c["kind"] == "decode":
        return A.attention_pytorch(state["q"], state["k"], state["v"], enable_gqa=c["Hq"] != c["Hkv"])
    if c["kind"] == "evoformer":
        biases = [b for b in (state["mask"], state["pair"]) if b is not None]
        kw = {} if state["gate"] is None else {"gate": state["gate"]}
        out = A.attention_reference(state["q"], state["k"], state["v"], biases, **kw)
        if not c["train"]:
            return out
        return [out.detach(), *torch.autograd.grad(out, state["leaves"], state["dout"])]
    out = _attend(state)
    if c["kind"] == "forward":
        return out
    return [out.detach(), *torch.autograd.grad(out, state["leaves"], state["dout"].view(out.shape) if out.dim() == 4
                                               else state["dout"].unflatten(1, out.shape[1:3]))]


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------

def work(case):
    """Operands and results once; 2 FLOPs per multiply-add of the two products over attended pairs, and 5 products
    instead of 2 for the gradients besides (scores again, and one for each of dP, dQ, dK, dV)."""
    c = case
    if c["kind"] == "decode":
        q, kv = c["B"] * c["Hq"] * c["Lq"] * c["D"], c["B"] * c["Hkv"] * c["Lk"] * c["D"]
        return {"bytes": 2 * (2 * q + 2 * kv), "flops": 4 * q * c["Lk"]}
    if c["kind"] == "evoformer":
        rows = c["B"] * c["N"]
        t, pair = rows * c["S"] * c["H"] * c["D"], c["B"] * c["H"] * c["S"] ** 2
        n = t * (4 + c["gate"]) + pair + (rows * c["S"] if c["mask"] else 0)
        if c["train"]:  # dout in; dq, dk, dv, the pair bias's and the gate's gradient out
            n += t * (4 + c["gate"]) + pair
        return {"bytes": 2 * n, "flops": (14 if c["train"] else 4) * c["D"] * rows * c["H"] * c["S"] ** 2}
    B, Hq, Hkv, S, D, variant = c["B"], c["Hq"], c["Hkv"], c["S"], c["D"], c["variant"]
    pairs = {"vanilla": lambda: W.pairs_none(S), "sliding": lambda: W.pairs_sliding(S, c["window"]),
             "prefix": lambda: W.pairs_prefix(S, c["prefix"]),
             "document": lambda: W.pairs_documents(_doc_lengths(c, 1), True)}.get(variant, lambda: W.pairs_causal(S))()
    if variant == "diff":
        return {"bytes": 2 * B * S * (2 * (Hq + Hkv) * D + 2 * (Hq + Hkv) * D), "flops": 12 * D * pairs * B * Hq}
    n = B * S * D * (2 * Hq + 2 * Hkv)
    if c["kind"] == "train":
        n += B * S * D * (2 * Hq + 2 * Hkv)  # dout in, dq, dk, dv out
    return {"bytes": 2 * n + (8 * B * S if variant == "document" else 0),
            "flops": (14 if c["kind"] == "train" else 4) * D * pairs * B * Hq}


def tolerance(case):
    # 16-bit results of 16-bit operands: weights, score gradients and results are rounded to that type
    return {"rel": 1e-2} if case["dtype"] == "bf16" else {"rel": 3e-3}
