"""What a program that uses this package has it do, as cases that can be timed.

Four kinds of work, each through the public entry points:

``linear``   one eager call of a compressed linear layer (:class:`CompressedLinear`, i.e. ``F.linear``
             with a compressed weight), from one row of activations (a decode step outside a graph)
             over a handful (batched decoding, speculative tokens, a short prompt) to a long prompt;
``layer``    a decoder layer's decode step recorded into one graph and replayed, as serving runs it:
             RMSNorm + q/k/v in one grouped launch, the one-launch attention step over the key/value
             cache (one row; with more rows the layer's linears alone, since attention over several
             sequences is the model's own code), o_proj + residual, RMSNorm, gate/up, SwiGLU + down_proj
             + residual;
``decode``   the BF16 weight back from its compressed form (``get_weight``), bit for bit;
``convert``  compressing a BF16 ``nn.Linear`` that lies in host memory (what ``convert_all_linear`` does
             per layer when a checkpoint has been loaded).

Sizes: the linears of a Qwen2.5-7B and a Qwen3-8B decoder layer and of smaller layers of the same
build; weights iid N(0, 0.02) or Student-t with three degrees of freedom of the same spread.
"""
import math

import torch

from bf16_huffman_infer_amd.cudagraph_utils import GraphedCallable
from bf16_huffman_infer_amd.functional import (ANSWeight, CompressedLinear, HuffmanWeight, NibbleWeight, convert,
                                               linear_grouped)
from bf16_huffman_infer_amd.ops import decode_attention, rms_norm
from bf16_huffman_infer_amd.utils import get_block_size_n

CODECS = {"huffman": HuffmanWeight, "ans": ANSWeight, "nibble": NibbleWeight}
HEAD = 128                      # head dimension of both decoders
EPS = 1e-6
# bytes of a compressed weight over those of its BF16 form
RATIO = {("huffman", "normal"): 0.69, ("huffman", "student"): 0.71, ("ans", "normal"): 0.70, ("ans", "student"): 0.72,
         ("nibble", "normal"): 0.751, ("nibble", "student"): 0.751, ("smallest", "normal"): 0.69, ("smallest", "student"): 0.71}

HALF_STREAM = 0.09              # words of the exponent stream per weight: always more than this and less than twice this


def _linear(name, codec, dist, M, K, rows, bias=False):
    return {"name": name, "kind": "linear", "codec": codec, "dist": dist, "M": M, "K": K, "rows": rows, "bias": bias}


def _layer(name, codec, hidden, inter, kv_heads, rows, context):
    return {"name": name, "kind": "layer", "codec": codec, "dist": "normal", "hidden": hidden, "inter": inter,
            "kv_heads": kv_heads, "rows": rows, "context": context}


def listed():
    return [
        # k_proj / v_proj of Qwen3-8B for one token outside a graph: the smallest call of a decode step
        _linear("kv_proj_1row", "huffman", "normal", 1024, 4096, 1),
        # q/k/v of Qwen2.5-7B as one matrix, which has a bias, for five sequences; the rANS codec
        _linear("qkv_bias_5rows", "ans", "normal", 4608, 3584, 5, bias=True),
        # batched decoding, sixteen sequences, gate or up projection of Qwen3-8B; heavy-tailed weights
        _linear("up_proj_16rows", "huffman", "student", 12288, 4096, 16),
        # a short prompt of an odd length through the down projection of Qwen3-8B
        _linear("down_proj_77rows", "huffman", "student", 4096, 12288, 77),
        # a prompt of a few hundred tokens, rANS
        _linear("gate_proj_300rows", "ans", "normal", 11008, 4096, 300),
        # a long prompt through the largest linear of a Qwen2.5-7B layer
        _linear("prefill_2048rows", "huffman", "normal", 18944, 3584, 2048),
        # one token of Qwen3-8B early in a conversation: a layer of the recorded step
        _layer("token_qwen3_early", "huffman", 4096, 12288, 8, 1, 300),
        # one token of Qwen2.5-7B late in a long one
        _layer("token_qwen25_late", "huffman", 3584, 18944, 4, 1, 6000),
        # eight sequences decoded together, Qwen2.5-7B
        _layer("step_qwen25_8rows", "huffman", 3584, 18944, 4, 8, 0),
        # two sequences, Qwen3-8B, rANS
        _layer("step_qwen3_ans_2rows", "ans", 4096, 12288, 8, 2, 0),
        # the BF16 weight of a down projection back from its compressed form
        {"name": "get_weight", "kind": "decode", "codec": "huffman", "dist": "student", "M": 4096, "K": 12288},
        # conversion of a loaded checkpoint, one gate or up projection of Qwen3-8B
        {"name": "convert_up_proj", "kind": "convert", "codec": "huffman", "dist": "normal", "M": 12288, "K": 4096},
    ]


LARGEST = 18944 * 3584          # weights of the largest listed matrix
LARGEST_CONVERT = 12288 * 4096


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _units(rng, lo, hi):
    """A multiple of 128, spread over the logarithm of the range."""
    return 128 * max(1, round(_log_uniform(rng, lo, hi) / 128))


def _columns(rng, lo, hi):
    """A number of in_features that can be cut into column blocks."""
    while True:
        K = _units(rng, lo, hi)
        try:
            get_block_size_n(torch.empty(1, K, device="meta"))
            return K
        except RuntimeError:
            pass


def draw(rng):
    kind = rng.choices(("linear", "layer", "decode", "convert"), (6, 4, 1, 1))[0]
    codec = rng.choices(("huffman", "ans", "nibble"), (6, 3, 1))[0]
    dist = rng.choice(("normal", "student"))
    if kind == "layer":
        heads = rng.randint(8, 32)
        kv_heads = rng.choice([h for h in (1, 2, 4, 8) if heads % h == 0])
        hidden = heads * HEAD
        try:
            get_block_size_n(torch.empty(1, hidden, device="meta"))
        except RuntimeError:
            heads, kv_heads, hidden = 28, 4, 3584
        inter = _columns(rng, 2 * hidden, 5 * hidden)
        rows = rng.choice((1, 1, 1, 2, 3, 4, 5, 6, 7, 8))
        context = int(_log_uniform(rng, 16, 8191)) if rows == 1 else 0
        case = _layer("", "huffman" if codec == "nibble" else codec, hidden, inter, kv_heads, rows, context)
        del case["name"]
        return case
    most = LARGEST_CONVERT if kind == "convert" else LARGEST
    K = _columns(rng, 1024, 18944)
    M = _units(rng, 512, min(32768, most // K))
    M = min(M, most // K // 128 * 128)
    case = {"kind": kind, "codec": codec, "dist": dist, "M": M, "K": K}
    if kind == "linear":
        case.update(rows=int(_log_uniform(rng, 1, 2049)), bias=rng.random() < 0.3)
    if kind == "convert":
        case["codec"] = rng.choices(("huffman", "ans", "smallest"), (4, 2, 2))[0]
        if case["codec"] == "smallest":
            case["M"] = max(128, M // 2 // 128 * 128)
    return case


# ------------------------------------------------------------------ preparation
def _weight(gen, dist, M, K):
    z = torch.randn(M, K, generator=gen, device="cuda")
    if dist == "student":
        chi2 = sum(torch.randn(M, K, generator=gen, device="cuda") ** 2 for _ in range(3))
        z = z * torch.rsqrt(chi2)              # Student-t with 3 degrees of freedom over sqrt(3): unit spread
    return (z * 0.02).bfloat16()


def _compressed(gen, codec, dist, M, K):
    return CODECS[codec].compress(_weight(gen, dist, M, K)).cuda()


def _rope_tables(length, theta=1e6):
    inv = 1.0 / (theta ** (torch.arange(0, HEAD, 2, device="cuda").float() / HEAD))
    angle = torch.arange(length, device="cuda").float()[:, None] * inv[None, :]
    return torch.cat((angle.cos(), angle.cos()), -1), torch.cat((-angle.sin(), angle.sin()), -1)


class _Layer:
    """A decoder layer with compressed projections and its recorded decode step."""

    def __init__(self, case, gen):
        self.rows, self.kv_heads = case["rows"], case["kv_heads"]
        hidden, inter = case["hidden"], case["inter"]
        self.heads = hidden // HEAD
        kv = self.kv_heads * HEAD

        def proj(M, K):
            return _compressed(gen, case["codec"], case["dist"], M, K)
        self.q, self.k, self.v, self.o = proj(hidden, hidden), proj(kv, hidden), proj(kv, hidden), proj(hidden, hidden)
        self.gate, self.up, self.down = proj(inter, hidden), proj(inter, hidden), proj(hidden, inter)

        def norm(*shape):
            return (1 + 0.1 * torch.randn(*shape, generator=gen, device="cuda")).bfloat16()
        self.input_norm, self.post_norm = norm(hidden), norm(hidden)
        self.x = torch.randn(self.rows, hidden, generator=gen, device="cuda").bfloat16()
        if self.rows == 1:
            self.head_norm = norm(self.heads + self.kv_heads, HEAD)
            slots = 1024 if case["context"] < 1024 else 8192
            self.cos, self.sin = _rope_tables(slots)
            self.k_cache = torch.randn(self.kv_heads, slots, HEAD, generator=gen, device="cuda").bfloat16()
            self.v_cache = torch.randn(self.kv_heads, slots, HEAD, generator=gen, device="cuda").bfloat16()
            self.pos = torch.tensor([case["context"]], device="cuda")
        self.recorded = GraphedCallable(self.step, (self.x,))

    def step(self, x):
        if self.rows == 1:
            nq, nk = self.heads * HEAD, self.kv_heads * HEAD
            qk, v = x.new_empty(1, nq + nk), x.new_empty(1, nk)
            linear_grouped(x, [self.q, self.k, self.v], input_norm=(self.input_norm, EPS), outs=[qk[:, :nq], qk[:, nq:], v])
            a = decode_attention(qk.view(-1, HEAD), v.view(-1, HEAD), self.head_norm, self.cos, self.sin, self.pos,
                                 self.k_cache, self.v_cache, eps=EPS).view(1, nq)
            k = qk[:, nq:]
        else:
            a, k, v = linear_grouped(x, [self.q, self.k, self.v], input_norm=(self.input_norm, EPS))
        x, = linear_grouped(a, [self.o], residuals=[x])
        gate, up = linear_grouped(rms_norm(x, self.post_norm, EPS), [self.gate, self.up])
        x, = linear_grouped(up, [self.down], input_gate=gate, residuals=[x])
        return x, a, k, v


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    kind = case["kind"]
    if kind == "layer":
        return "layer", _Layer(case, gen)
    M, K = case["M"], case["K"]
    if kind == "convert":
        linear = torch.nn.Linear(K, M, bias=False, dtype=torch.bfloat16, device="meta")
        linear.weight = torch.nn.Parameter(_weight(gen, case["dist"], M, K).cpu(), requires_grad=False)
        return "convert", linear, case["codec"]
    weight = _compressed(gen, case["codec"], case["dist"], M, K)
    if kind == "decode":
        return "decode", weight
    bias = None
    if case["bias"]:
        bias = torch.nn.Parameter((0.1 * torch.randn(M, generator=gen, device="cuda")).bfloat16(), requires_grad=False)
    x = torch.randn(case["rows"], K, generator=gen, device="cuda").bfloat16()
    return "linear", CompressedLinear(weight, bias), x


# ------------------------------------------------------------------ one pass
@torch.no_grad()
def run(state):
    kind = state[0]
    if kind == "linear":
        return state[1](state[2])
    if kind == "layer":
        layer = state[1]
        out = layer.recorded(layer.x)
        return out + (layer.k_cache, layer.v_cache) if layer.rows == 1 else out
    if kind == "decode":
        return state[1].get_weight()
    buffers = dict(convert(state[1], "proj", algo=state[2]).weight.named_buffers())
    # the length of the exponent stream depends on the weights: it is handed out as two
    # overlapping views of a size that depends on the layer only, which together hold all of it
    exp = buffers.pop("exp")
    half = int(HALF_STREAM * buffers["rem"].numel())
    assert half <= exp.numel() <= 2 * half
    return {**buffers, "exp_words": exp.numel(), "exp_front": exp[:half], "exp_back": exp[-half:]}


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    ratio = RATIO[case["codec"], case["dist"]]
    if case["kind"] == "layer":
        hidden, inter, rows = case["hidden"], case["inter"], case["rows"]
        kv = case["kv_heads"] * HEAD
        weights = 2 * hidden * hidden + 2 * kv * hidden + 3 * inter * hidden
        attended = (case["context"] + 1) * hidden * 4 if rows == 1 else 0            # q k^T and the weighted sum
        cache = (case["context"] + 1) * kv * 4 if rows == 1 else 0
        return {"bytes": 2 * ratio * weights + cache + 2 * rows * (3 * hidden + 2 * kv), "flops": 2 * weights * rows + attended}
    M, K = case["M"], case["K"]
    if case["kind"] == "linear":
        rows = case["rows"]
        return {"bytes": 2 * ratio * M * K + 2 * rows * (M + K), "flops": 2 * M * K * rows}
    return {"bytes": 2 * (1 + ratio) * M * K, "flops": 0}


def tolerance(case):
    """About four times the distance to the same path in 64-bit floats without its BF16 roundings
    (linear: 2-norm 0.0017 without and 0.0023 with a bias, largest difference 0.0075; layer: 0.0056 and
    0.023; with the roundings kept and the sums in 64 bits 0.00005 and 0.0078, 0.0019 and 0.012)."""
    if case["kind"] in ("decode", "convert"):
        return "exact"
    if case["kind"] == "layer":
        return {"rel": 0.02, "max": 0.09}
    return {"rel": 0.007, "max": 0.03}
