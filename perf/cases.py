"""Workloads by which the speed of this package is judged: what a user's program asks of flash_forward and
flash_forward_splitkv, from a call that is over in a few microseconds to launches that fill the GPU for half a
millisecond.

listed() names twelve of them, draw() gives more of the same ranges.  prepare() makes what the program has in hand before
the call (fp16 Q, K and V on the GPU, and the slope table where ALiBi is on), run() is one call as such a program writes
it, with every other argument left at its default.
"""
import math

import torch

import flash_attn_amd as fa

# Fields of a case.  entry: "forward" (whole key range in one kernel) or "splitkv" (the library chooses how many pieces
# the key range is cut into, as it does for decode and for long caches); B, H, Hk: batch, query heads, K/V heads;
# Nq, Nk, d: query rows, keys, head dimension; left, right: window in keys, -1 for none; p: dropout probability.
_DEFAULTS = {"entry": "forward", "causal": False, "left": -1, "right": -1, "alibi": False, "p": 0.0}


def _case(name, B, H, Nq, Nk, d, Hk=None, **options):
    c = dict(_DEFAULTS, B=B, H=H, Hk=H if Hk is None else Hk, Nq=Nq, Nk=Nk, d=d)
    c.update(options)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # one short sequence through a small layer: what counts is the way to the GPU
        _case("tiny plain", 1, 2, 128, 128, 64),
        # a single sequence of odd length with narrow heads, the sizes that the command-line driver runs by default
        _case("single odd d31", 1, 8, 1021, 1021, 31, entry="splitkv"),
        # a batch of short documents through an encoder: no mask, many heads, few keys
        _case("encoder batch d64", 32, 32, 512, 512, 64),
        # prompt processing of a decoder, one K/V head per query head
        _case("causal prefill d128", 4, 16, 2048, 2048, 128, causal=True),
        # prompt processing with eight query heads per K/V head, the largest number of operations here
        _case("grouped prefill d128", 4, 32, 4096, 4096, 128, Hk=4, causal=True),
        # prompts of odd length with a head dimension between the powers of two
        _case("ragged causal d80", 3, 12, 1777, 1777, 80, causal=True),
        # sliding-window layer with position biases
        _case("window alibi d64", 2, 16, 4096, 4096, 64, left=256, right=0, alibi=True),
        # a training step's forward with dropout, the length no multiple of a tile
        _case("causal dropout d96", 8, 32, 1000, 1000, 96, causal=True, p=0.1),
        # generation, one user: one token against a cache of moderate length
        _case("decode one d128", 1, 32, 1, 4096, 128, entry="splitkv"),
        # generation, a full batch with long caches: the largest number of bytes here
        _case("decode batch d128", 16, 32, 1, 16384, 128, entry="splitkv"),
        # generation with four query heads per K/V head, the cache in the middle of a block
        _case("decode grouped d128", 8, 32, 1, 5003, 128, Hk=8, entry="splitkv"),
        # a chunk of a prompt against the cache of what came before
        _case("chunk on cache d128", 1, 32, 128, 16384, 128, causal=True, entry="splitkv"),
    ]


def _size(rng, lo, hi):
    """An integer spread over the logarithm of the range, every other time a multiple of 64 where it is large enough."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if n >= 128 and rng.random() < 0.5:
        n = n // 64 * 64
    return max(lo, min(hi, n))


# dimensions that the tests and the benchmark use, by how common they are
_DIMS = (64, 64, 128, 128, 128, 32, 96, 80, 31, 40, 72, 100, 112)
_MOST_FLOPS = 1.5e11  # of a drawn case, counted at 64 columns where the heads are narrower
_MOST_BYTES = 2.0e9


def draw(rng):
    while True:
        kind = rng.choice(("plain", "causal", "causal", "window", "dropout", "decode", "decode", "chunk"))
        d = rng.choice(_DIMS)
        group = rng.choice((1, 1, 1, 2, 4, 8))
        hk = rng.choice((1, 2, 3, 4, 8, 8, 12, 16, 32)) if group == 1 else rng.choice((1, 2, 4, 8))
        B = _size(rng, 1, 32)
        options = {}
        if kind == "decode":
            nq, nk = 1, _size(rng, 256, 32768)
            options["entry"] = "splitkv"
        elif kind == "chunk":
            nq, nk = _size(rng, 2, 512), _size(rng, 1024, 32768)
            options.update(entry="splitkv", causal=True)
        else:
            nq = nk = _size(rng, 64, 8192)
            options["causal"] = kind in ("causal", "dropout")
            if kind == "window":
                options.update(left=_size(rng, 64, 2048), right=0, alibi=rng.random() < 0.5)
            if kind == "dropout":
                options["p"] = rng.choice((0.05, 0.1, 0.2))
        c = _case(None, B, hk * group, nq, nk, d, Hk=hk, **options)
        w = work(c)
        if w["flops"] * max(d, 64) / d <= _MOST_FLOPS and w["bytes"] <= _MOST_BYTES:
            return c


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    B, H, Hk, Nq, Nk, d = (case[x] for x in ("B", "H", "Hk", "Nq", "Nk", "d"))

    def normal(*shape):
        return torch.randn(shape, generator=g, dtype=torch.float16, device="cuda")

    q, k, v = normal(B, H, Nq, d), normal(B, Hk, Nk, d), normal(B, Hk, Nk, d)
    options = {}
    if case["causal"]:
        options["causal"] = True
    if case["left"] >= 0 or case["right"] >= 0:
        options["window"] = (case["left"], case["right"])
    if case["alibi"]:
        options["alibi_slopes"] = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)], dtype=torch.float32, device="cuda")
    if case["p"] > 0:
        options.update(dropout_p=case["p"], seed=seed + 1)
    return {"call": fa.flash_forward if case["entry"] == "forward" else fa.flash_forward_splitkv, "qkv": (q, k, v), "options": options}


def run(state):
    return state["call"](*state["qkv"], **state["options"])


def _visible_pairs(case):
    """(row, key) pairs of one head that the masks leave; row i stands at key position i + Nk - Nq."""
    Nq, Nk = case["Nq"], case["Nk"]
    pairs = 0
    for i in range(Nk - Nq, Nk):
        first = max(0, i - case["left"]) if case["left"] >= 0 else 0
        last = Nk - 1
        if case["causal"]:
            last = min(last, i)
        if case["right"] >= 0:
            last = min(last, i + case["right"])
        pairs += max(0, last - first + 1)
    return pairs


def work(case):
    """Q, K and V read once, O (fp16) and the log-sum-exp (fp32) written once; two products over the visible pairs."""
    B, H, Hk, Nq, Nk, d = (case[x] for x in ("B", "H", "Hk", "Nq", "Nk", "d"))
    return {"bytes": 2 * d * (2 * B * H * Nq + 2 * B * Hk * Nk) + 4 * B * H * Nq, "flops": 4 * d * B * H * _visible_pairs(case)}


def tolerance(case):
    """Probabilities enter the second product in fp16 and O leaves in fp16: a relative rounding of 2^-12 on average and
    2^-11 at most each, in either implementation, and single outputs in which large terms cancel are off by several
    times that of the typical output.  (The log-sum-exp in fp32 is far inside.)"""
    return {"rel": 1e-3, "max": 1e-2}
