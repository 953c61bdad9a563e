"""The performance cases of the quantised linear layers: what a program that runs a GPTQ model has them do.

A case is one of three kinds of work, through ``QuantLinear`` and ``fuse_shared_input_layers``:

* ``forward``: one layer applied to the tokens of a decoding step (``tokens`` = 1, ``batch`` sequences) or of a prompt;
* ``block``: the seven linear layers of a decoder block in a decoding step, called one after the other as the model's
  code calls them, with or without the fusion of the layers that read one input;
* ``train``: forward and backward (gradient of the input) of a frozen layer, as adapters on top of it need them.

``layers`` says what the module holds: ``tiled`` is what ``from_quantized`` leaves (the tiled copy as the only one),
``kept`` a module with its checkpoint tensors, which builds the copies that it wants on its first calls.
"""
import math

import torch
import torch.nn as nn

from autogptq.tvm_amd import QuantLinear
from autogptq.tvm_amd.fused import fuse_shared_input_layers

LARGEST = 4096 * 8192 * 28672    # rows x K x N of the largest product; drawn ones stay within it


def _forward(name, bits, K, N, group, act, batch, tokens, layers="tiled", bias=False):
    return {"name": name, "kind": "forward", "bits": bits, "K": K, "N": N, "group": group, "act": act, "batch": batch,
            "tokens": tokens, "layers": layers, "bias": bias}


def listed():
    return [
        # decoding, one sequence: a layer of a small model
        _forward("decode-int4-1024x1024", 4, 1024, 1024, 128, False, 1, 1),
        # the same for an attention projection and a feed-forward projection of common width (4 and 3 bits; the second
        # with the activation order that GPTQ quantisers write by default)
        _forward("decode-int4-4096x4096", 4, 4096, 4096, 128, False, 1, 1),
        _forward("decode-int3-4096x11008-act", 3, 4096, 11008, 128, True, 1, 1),
        # a feed-forward layer of a large model, one group per column: the decoding call that is bound by memory
        _forward("decode-int3-9216x36864-g1", 3, 9216, 36864, -1, True, 1, 1),
        # a decoding step of one sequence through the linear layers of a decoder block
        {"name": "block-int4-4096-11008-act", "kind": "block", "bits": 4, "K": 4096, "N": 11008, "kv": 4096, "group": 128,
         "act": True, "batch": 1, "fused": False},
        # small and middling batches of sequences
        _forward("decode8-int4-11008x4096-act", 4, 11008, 4096, 128, True, 8, 1, layers="kept"),
        _forward("decode32-int4-4096x11008-act", 4, 4096, 11008, 128, True, 32, 1),
        # prompts: short, of ragged sizes (8 bits, groups of 64, a bias), long on a module that kept its checkpoint
        # tensors, and a batch of long ones on a layer of a large model
        _forward("prompt128-int4-4096x11008-act", 4, 4096, 11008, 128, True, 1, 128),
        _forward("prompt333-int8-5120x3424", 8, 5120, 3424, 64, False, 1, 333, bias=True),
        _forward("prompt2000-int3-9216x9216-g1", 3, 9216, 9216, -1, True, 1, 2000, layers="kept"),
        _forward("prompt4096-int4-8192x28672", 4, 8192, 28672, 128, False, 2, 2048),
        # a training step's share of one frozen layer
        {"name": "train2048-int4-4096x4096-act", "kind": "train", "bits": 4, "K": 4096, "N": 4096, "group": 128, "act": True,
         "batch": 4, "tokens": 512, "layers": "kept", "bias": False},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    bits = rng.choice((4, 4, 4, 4, 3, 3, 8, 2))
    group = rng.choice((128, 128, 128, 64, 32, -1))
    unit = max(group, 32)
    K = max(1, round(_log(rng, 1024, 20480) / unit)) * unit
    N = max(1, round(_log(rng, 1024, 32768) / 32)) * 32
    act = rng.random() < 0.5
    kind = rng.choice(("decode", "decode", "decode", "prompt", "prompt", "prompt", "block", "train"))
    if kind == "block":
        K = min(K, 8192)
        N = max(unit, round(min(N, 4 * K) / unit) * unit)      # the last layer's channels come in whole groups too
        kv = max(32, round(K / rng.choice((1, 1, 4)) / 32) * 32)
        return {"kind": "block", "bits": bits, "K": K, "N": N, "kv": kv, "group": group, "act": act,
                "batch": rng.choice((1, 1, 2, 4, 7)), "fused": rng.random() < 0.5}
    layers = rng.choice(("tiled", "kept")) if kind != "train" else "kept"
    bias = rng.random() < 0.25
    if kind == "decode":
        batch, tokens = _log(rng, 1, 64), 1
    elif kind == "prompt":
        batch, tokens = 1, _log(rng, 17, 4096)
    else:
        batch, tokens = rng.choice((1, 2, 4)), _log(rng, 32, 1024)
    most = LARGEST // (2 if kind == "train" else 1) // (K * N)
    tokens = max(1, min(tokens, most // batch))
    c = _forward("", bits, K, N, group, act, batch, tokens, layers, bias)
    del c["name"]
    c["kind"] = "train" if kind == "train" else "forward"
    return c


# ------------------------------------------------------------------ inputs
def _pack(codes, bits):
    """[32 B, C] codes as the little-endian bit stream of the format along the first axis: int32 [bits B, C]."""
    blocks = codes.view(-1, 32, codes.shape[1])
    words = torch.zeros((blocks.shape[0], bits, codes.shape[1]), dtype=torch.int32, device=codes.device)
    for j in range(32):
        w, off = divmod(bits * j, 32)
        words[:, w] |= blocks[:, j] << off
        if off + bits > 32:
            words[:, w + 1] |= blocks[:, j] >> (32 - off)
    return words.view(-1, codes.shape[1])


def _codes(shape, bits, gen):
    """Codes as a quantiser leaves them: bell-shaped around the middle of the range."""
    top = 2 ** bits - 1
    c = torch.randn(shape, device="cuda", generator=gen)
    return c.mul_(top / 6).add_(top / 2).round_().clamp_(0, top).to(torch.int32)


def _order(K, group, act, gen):
    """g_idx: the group of every input channel, in the order the quantiser met the channels."""
    where = torch.randperm(K, device="cuda", generator=gen) if act else torch.arange(K, device="cuda")
    return (where // (K if group == -1 else group)).to(torch.int32)


def _layer(bits, K, N, group, g_idx, bias, gen):
    layer = QuantLinear(bits, group, K, N, bias)
    groups = layer.scales.shape[0]
    layer.qweight = _pack(_codes((K, N), bits, gen), bits)
    mid = 2 ** (bits - 1) - 1                                   # the format stores the zero point less one
    zeros = torch.randint(max(0, mid - 1), mid + 1, (N, groups), device="cuda", generator=gen, dtype=torch.int32)
    layer.qzeros = _pack(zeros, bits).t().contiguous()
    spread = torch.rand((groups, N), device="cuda", generator=gen) + 0.5
    layer.scales = (spread * (6 / (2 ** bits - 1) / math.sqrt(K))).half()
    layer.g_idx = g_idx
    if bias:
        layer.bias = torch.randn(N, device="cuda", generator=gen).half()
    return layer


def _tensor(shape, gen):
    return torch.randn(shape, device="cuda", generator=gen, dtype=torch.float16)


class Block(nn.Module):
    """The linear layers of a decoder block, under the names that the fusion looks for."""

    def __init__(self, case, gen):
        super().__init__()
        K, N, kv, bits, group = (case[k] for k in ("K", "N", "kv", "bits", "group"))
        for names, k, widths in ((("q_proj", "k_proj", "v_proj"), K, (K, kv, kv)), (("o_proj",), K, (K,)),
                                 (("gate_proj", "up_proj"), K, (N, N)), (("down_proj",), N, (K,))):
            g_idx = _order(k, group, case["act"], gen)          # layers that read one input share their order
            for name, n in zip(names, widths):
                setattr(self, name, _layer(bits, k, n, group, g_idx, False, gen))

    def forward(self, h, attended, h2, gated):
        return [self.q_proj(h), self.k_proj(h), self.v_proj(h), self.o_proj(attended), self.gate_proj(h2),
                self.up_proj(h2), self.down_proj(gated)]


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    K, N = case["K"], case["N"]
    if case["kind"] == "block":
        block = Block(case, gen)
        if case["fused"]:
            fuse_shared_input_layers(block)
        for m in block.modules():
            if isinstance(m, QuantLinear):
                m.compact()
        return {"kind": "block", "model": block.eval(), "x": [_tensor((case["batch"], 1, k), gen) for k in (K, K, K, N)]}
    g_idx = _order(K, case["group"], case["act"], gen)
    layer = _layer(case["bits"], K, N, case["group"], g_idx, case["bias"], gen).eval()
    if case["layers"] == "tiled":
        layer.compact()
    state = {"kind": case["kind"], "model": layer, "x": _tensor((case["batch"], case["tokens"], K), gen)}
    if case["kind"] == "train":
        state["x"].requires_grad_(True)
        state["gy"] = _tensor((case["batch"], case["tokens"], N), gen)
    return state


def run(state):
    if state["kind"] == "train":
        y = state["model"](state["x"])
        gx, = torch.autograd.grad(y, state["x"], state["gy"])
        return [y.detach(), gx]
    with torch.no_grad():
        if state["kind"] == "block":
            return state["model"](*state["x"])
        return state["model"](state["x"])


# ------------------------------------------------------------------ what a pass cannot do without
def _need(case, K, N, rows):
    groups = 1 if case["group"] == -1 else -(-K // case["group"])
    weights = K * N * case["bits"] // 8 + groups * N * (2 + case["bits"] / 8)
    if case["act"] and groups > 1:
        weights += 4 * K
    return weights + 2 * N * bool(case.get("bias")), 2 * rows * (K + N), 2 * rows * K * N


def work(case):
    K, N = case["K"], case["N"]
    if case["kind"] == "block":
        shapes = [(K, K), (K, case["kv"]), (K, case["kv"]), (K, K), (K, N), (K, N), (N, K)]
        parts = [_need(case, k, n, case["batch"]) for k, n in shapes]
        shared_x = 2 * case["batch"] * 3 * K                    # q, k, v read one input, gate and up another
        return {"bytes": sum(w + a for w, a, _ in parts) - shared_x, "flops": sum(f for _, _, f in parts)}
    weights, ends, flops = _need(case, K, N, case["batch"] * case["tokens"])
    times = 2 if case["kind"] == "train" else 1                 # the gradient reads one end and writes the other again
    return {"bytes": weights + times * ends, "flops": times * flops}


def tolerance(case):
    # fp16 weights (rounded or not) and results, 32-bit sums: two roundings of 2^-11
    return {"rel": 1e-3}
