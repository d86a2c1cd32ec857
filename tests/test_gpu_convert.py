"""The conversion passes around the encoders (needs a GPU) against tensor operations on the CPU."""
import pytest
import torch

from helpers import gaussian_weight, random_bits_weight, student_t_weight

pytestmark = pytest.mark.gpu


def _lane_order(plane, n):
    """[M, K] bytes -> [split, group, step, lane, column]."""
    M, K = plane.shape
    x = plane.view(M // 4, 4, n, K // n // 128, 16, 8)
    return x.permute(2, 0, 3, 4, 1, 5).reshape(n, M // 4, K // n // 128, 512)


@pytest.mark.parametrize("make", [gaussian_weight, random_bits_weight])
@pytest.mark.parametrize("offset", [0, 1])
@pytest.mark.parametrize("M,K,n", [(128, 128, 1), (128, 1152, 1), (256, 2176, 1), (128, 3456, 3), (640, 1024, 2), (28672, 384, 3)])
def test_split_planes_and_histogram(cuda, make, offset, M, K, n):
    """Whole weights and, one element on, weights that are aligned to two bytes only; one to four chunks of
    steps that do not divide evenly; a workgroup that is not full."""
    from bf16_huffman_infer_amd import _lib, ops
    from bf16_huffman_infer_amd.utils import split_bf16
    w = make(M, K, seed=M + K)
    held = torch.empty(M * K + 1, dtype=torch.bfloat16, device="cuda")[offset:offset + M * K].view(M, K)
    held.copy_(w)
    rem, exp = ops.split_planes(held, n)
    wrem, wexp = split_bf16(w)
    assert torch.equal(rem.cpu().view(-1), _lane_order(wrem, n).reshape(-1))
    order, S = _lane_order(wexp, n), K // n // 128
    nc = _lib.load().bhi_chunks_per_group(M, K // n, n)
    want = torch.cat([order[:, :, S * c // nc:S * (c + 1) // nc].reshape(-1) for c in range(nc)])
    assert torch.equal(exp.cpu(), want)
    pairs = wexp[:, 0::2].to(torch.int64) | wexp[:, 1::2].to(torch.int64) << 8
    assert torch.equal(ops.pair_histogram(exp).cpu(), torch.bincount(pairs.flatten(), minlength=65536))


@pytest.mark.parametrize("algo", ["huffman", "ans", "smallest", "nibble"])
def test_convert_leaves_the_layer_alone_and_returns_host_buffers(cuda, algo):
    from bf16_huffman_infer_amd.functional import convert
    w = gaussian_weight(4096, 1024, seed=5)
    linear = torch.nn.Linear(1024, 4096, dtype=torch.bfloat16)
    linear.weight.data.copy_(w)
    module = convert(linear, "layer", algo=algo)
    assert torch.equal(linear.weight.data, w) and not linear.weight.is_cuda
    assert all(not b.is_cuda for b in module.buffers()) and module.bias is linear.bias
    assert torch.equal(module.cuda().weight.get_weight().cpu().view(torch.int16), w.view(torch.int16))


@pytest.mark.parametrize("algo", ["huffman", "ans", "nibble"])
@pytest.mark.parametrize("M,K", [(128, 384), (3, 6), (7, 10), (1, 2)])
def test_get_codec_takes_any_even_width(cuda, algo, M, K):
    """A code for a matrix of any even width, from host or GPU memory, equal to the one of a histogram on the CPU."""
    from bf16_huffman_infer_amd.functional import (ANS_PRECISION, ANSWeight, HuffmanWeight, LUTHuffmanEncoder, NibbleCodec,
                                                   NibbleWeight, RANSEncoder)
    from bf16_huffman_infer_amd.utils import split_bf16
    w = gaussian_weight(M, K, seed=K)
    exp = split_bf16(w)[1].to(torch.int64)
    counts = torch.bincount(exp.flatten(), minlength=256)
    for a in (w, w.cuda(), w.cuda().T.contiguous().T):
        if algo == "huffman":
            want = LUTHuffmanEncoder()
            want.build_lut(torch.bincount((exp[:, 0::2] | exp[:, 1::2] << 8).flatten(), minlength=65536))
            got = HuffmanWeight.get_codec(a)
            assert (got.enc_table == want.enc_table).all() and (got.LUT1 == want.LUT1).all()
        elif algo == "ans":
            want = RANSEncoder(counts.tolist(), precision=ANS_PRECISION)
            got = ANSWeight.get_codec(a)
            assert list(got.freq) == list(want.freq) and list(got.cum) == list(want.cum)
        else:
            want, got = NibbleCodec(counts), NibbleWeight.get_codec(a)
            assert (got.base, got.has_escapes) == (want.base, want.has_escapes)


@pytest.mark.parametrize("algo", ["huffman", "ans", "nibble"])
def test_compress_uses_the_class_own_codec(cuda, algo):
    """``get_codec`` is where a subclass chooses the code: here one built from another matrix."""
    from bf16_huffman_infer_amd import functional
    base = {"huffman": functional.HuffmanWeight, "ans": functional.ANSWeight, "nibble": functional.NibbleWeight}[algo]
    other = gaussian_weight(128, 1024, seed=9, std=0.1)
    asked = []

    class Own(base):
        @classmethod
        def get_codec(cls, a):
            asked.append(a.shape)
            # every exponent of `a` occurs in the code as well
            return base.get_codec(torch.cat([other, a.detach().cpu()]))
    w = gaussian_weight(256, 1024, seed=4)
    mod = Own.compress(w)
    want = base.get_lut_kwargs(base.get_codec(torch.cat([other, w])))
    assert asked == [w.shape] and type(mod) is Own
    assert all(torch.equal(getattr(mod, name), t) for name, t in want.items())
    assert torch.equal(mod.cuda().get_weight().cpu().view(torch.int16), w.view(torch.int16))


def test_convert_compares_with_the_layer_itself(cuda):
    """The precision check runs the layer that would be replaced, a subclass's forward, its further parameters and
    hooks included; the layer keeps its storage."""
    from bf16_huffman_infer_amd.functional import CompressedLinear, convert

    class Adapted(torch.nn.Linear):
        def __init__(self, *args, **kwargs):
            super().__init__(*args, **kwargs)
            self.gain = torch.nn.Parameter(torch.ones(self.out_features, dtype=torch.bfloat16))
            self.register_buffer("shift", torch.zeros(self.out_features, dtype=torch.bfloat16))

        def forward(self, x):
            return super().forward(x) * self.gain + self.shift
    w = gaussian_weight(4096, 1024, seed=6)
    for change, accepted in ((None, True), ("gain", False), ("shift", False), ("hook", False)):
        linear = Adapted(1024, 4096, dtype=torch.bfloat16)
        linear.weight.data.copy_(w)
        linear.bias.data.fill_(10)               # outputs around 10: their BF16 steps are 0.6 %, the check's bound is 2 %
        if change == "hook":
            linear.register_forward_hook(lambda module, args, out: out + 1)
        elif change:
            getattr(linear, change).data.add_(1)
        held = {name: p.data_ptr() for name, p in linear.named_parameters()}
        module = convert(linear, "layer", disable_precision_check=False)
        assert (type(module) is CompressedLinear) == accepted, change
        assert module.bias is linear.bias
        assert {name: p.data_ptr() for name, p in linear.named_parameters()} == held
        assert not linear.shift.is_cuda and torch.equal(linear.weight.data, w)
    on_gpu = torch.nn.Linear(1024, 4096, dtype=torch.bfloat16).cuda()
    on_gpu.weight.data.copy_(w)
    module = convert(on_gpu, "layer")
    assert type(module) is CompressedLinear and not on_gpu.weight.is_cuda and torch.equal(on_gpu.weight.data, w)


def _count_sets():
    g = torch.Generator().manual_seed(11)
    at = torch.randperm(65536, generator=g)
    spread = (torch.rand(65536, generator=g).double() ** -3).clamp(max=1e9).long()
    yield "one pair", torch.zeros(65536).long().index_fill(0, at[:1], 5)
    yield "one pair, once", torch.zeros(65536).long().index_fill(0, at[:1], 1)
    yield "two pairs of one count", torch.zeros(65536).long().index_fill(0, at[:2], 7)
    for n in (3, 64, 65, 1000, 1535, 1536, 1537, 1538, 4000, 65536):
        counts = torch.zeros(65536).long()
        counts[at[:n]] = spread[at[:n]]
        yield f"{n} pairs", counts
        counts = counts.clone()
        counts[at[:n]] = 1 + spread[at[:n]] % 3
        yield f"{n} pairs of three counts", counts
    yield "all once", torch.ones(65536).long()
    steep = torch.zeros(65536).long()
    steep[at[:40]] = 1 << torch.arange(40)                       # beyond 32 bits, far beyond eleven levels
    yield "powers of two", steep
    steep = steep.clone()
    steep[at[40:3000]] = 1
    yield "powers of two and a tail", steep


def test_pair_code_on_the_gpu_is_the_host_one(cuda):
    from bf16_huffman_infer_amd.huffman import LUTHuffmanEncoder
    weights = [student_t_weight(256, 1024, seed=5), gaussian_weight(1024, 1024, seed=6)]
    sets = list(_count_sets())
    for w in weights:
        e = ((w.view(torch.int16).int() >> 7) & 0xFF)
        sets.append(("a weight", torch.bincount((e[:, 0::2] | e[:, 1::2] << 8).flatten(), minlength=65536)))
    for name, counts in sets:
        here, there = LUTHuffmanEncoder(), LUTHuffmanEncoder()
        here.build_lut(counts)
        there.build_lut(counts.cuda())
        assert (here.enc_table == there.enc_table).all() and (here.dec_table == there.dec_table).all(), name
        assert (here.code_lengths == there.code_lengths).all() and here.expected_bits == there.expected_bits, name
    for refused in (torch.zeros(65536).long(), -torch.ones(65536).long(), torch.ones(100).long()):
        with pytest.raises(AssertionError):
            LUTHuffmanEncoder().build_lut(refused.cuda())


@pytest.mark.parametrize("negative", [1, 3, 2000])
def test_pair_code_of_counts_that_are_partly_negative(cuda, negative):
    """Sorted, they are not in order for the kernel's unsigned searches: it looks at them first and builds nothing."""
    from bf16_huffman_infer_amd import ops
    from bf16_huffman_infer_amd.huffman import LUTHuffmanEncoder
    counts = torch.zeros(65536).long()
    counts[:3000] = torch.arange(3000, 0, -1)
    counts[40000:40000 + negative] = -torch.arange(1, negative + 1)
    for here in (counts, counts.cuda()):
        with pytest.raises(AssertionError):
            LUTHuffmanEncoder().build_lut(here)
    assert ops.pair_code(counts.cuda())[2].tolist() == [-1, 0, 0]
