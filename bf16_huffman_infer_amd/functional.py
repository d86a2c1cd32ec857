"""Compressed-weight modules, conversion and the ``F.linear`` dispatch.

Public surface of the reference's ``bf16_huffman_infer/functional.py``:
``HuffmanWeight``, ``ANSWeight``, ``CompressedLinear``, ``convert``,
``convert_all_linear``, ``linear_huffman`` (plus ``linear_ans``, ``mv_huffman``,
``mv_ans``).  Module buffers keep the reference's names and dtypes
(``rem, exp, offsets, LUT1..LUT4, code_lengths`` / ``rem, exp, offsets, LUT``), the
bytes inside ``rem``/``exp``/``offsets``/``LUT1`` follow the wave64 layout of this
package's HIP kernels.
"""
import contextlib
import functools
from typing import Optional

import torch
from torch import Tensor, nn
import torch.nn.functional as F
from tqdm import tqdm

from . import _lib
from .ans import RANSEncoder
from .huffman import LUTHuffmanEncoder
from . import ops as _ops
from .ops import (GEMM_MAX_ROWS, ans_decode, ans_encode, ans_encode_capacity, encode_capacity, gemm_bf16,
                  gemm_bf16_grouped,
                  gemv_bf16_ans, gemv_bf16_grouped, gemv_bf16_huffman, gemv_bf16_nibble, huffman_decode, huffman_encode,
                  nibble_decode, nibble_encode, nibble_encode_capacity)
from .utils import get_block_size_n
from .workspace import recorded

ANS_PRECISION = 8
MAX_FUSED_BATCH = 8
GROUP_ROWS = 4
STEP_COLS = 128
LANES = 64
LANE_COLS = 8
ENCODE_PART_BYTES = 256 << 20       # scratch bound per encode call

__all__ = [
    "linear_huffman",
    "linear_ans",
    "linear_nibble",
    "linear_grouped",
    "LinearGroup",
    "HuffmanWeight",
    "ANSWeight",
    "NibbleWeight",
    "CompressedLinear",
    "convert_all_linear",
    "convert",
    "load_compressed_state_dict",
    "check_layout",
]


def _exponents(a: Tensor) -> Tensor:
    """The exponent bytes of BF16 ``a`` on the GPU (:func:`.utils.split_bf16`'s, without the other plane and the
    32-bit integers)."""
    assert a.dtype == torch.bfloat16
    return (a.detach().to(torch.device('cuda', 0)).contiguous().view(torch.int16) >> 7).to(torch.uint8)


def _kernel_counts(exp: Tensor) -> bool:
    """Whether the histogram kernel takes ``exp``: eight-byte loads of GPU memory."""
    return exp.is_cuda and exp.numel() > 0 and exp.numel() % 8 == 0 and exp.data_ptr() % 8 == 0


def _single_counts(pairs: Tensor) -> Tensor:
    """int64 ``[256]`` occurrences of every exponent from those of the pairs."""
    pairs = pairs.view(256, 256)                 # [second, first]
    return pairs.sum(0) + pairs.sum(1)


def _exponent_counts(exp: Tensor) -> Tensor:
    """int64 ``[256]`` occurrences of every exponent."""
    exp = exp.flatten()
    if _kernel_counts(exp):
        return _single_counts(_ops.pair_histogram(exp))
    return torch.bincount(exp.to(torch.int32), minlength=256)


def _to_host(t: Tensor) -> Tensor:
    """``t`` in host memory.  Copying into memory that was never touched runs at the pace of its page faults,
    taken one by one (50 MB: 11.6 ms); a fill takes them on all threads first."""
    if not t.is_cuda:
        return t.cpu()
    host = torch.empty(t.shape, dtype=t.dtype)
    host.zero_()
    return host.copy_(t)


def _promote_single_split(A_rem: Tensor, offsets: Tensor):
    """A weight stored without the leading split dimension (``rem`` ``[M, N]``, ``offsets`` one
    rank lower as well) is a single split: the reference's ``mv_*`` accept that older form
    (``functional.py:33-36, 421-424``)."""
    if A_rem.dim() == 2:
        A_rem = A_rem[None, :, :]
        if offsets.dim() == 1:
            offsets = offsets[None, :]
    return A_rem, offsets


def _check_weight_call(A_rem: Tensor, A_exp: Tensor, X: Tensor):
    split_k, M, N = A_rem.shape
    assert M % 128 == 0
    assert N % 128 == 0
    assert X.dim() == 3 and X.size(-1) == N
    assert X.dtype == torch.bfloat16
    assert A_rem.is_cuda and A_exp.is_cuda and X.is_cuda
    assert A_rem.get_device() == A_exp.get_device() == X.get_device()


def mv_huffman(
    A_rem: Tensor, A_exp: Tensor, X: Tensor,
    offsets: Tensor,
    LUT1: Tensor, LUT2: Tensor, LUT3: Tensor, LUT4: Tensor,
    code_lengths: Tensor,
) -> Tensor:
    """Y[b, :] = W @ X[b, :] for b < 8 with W held compressed (reference ``functional.py:28-63``)."""
    A_rem, offsets = _promote_single_split(A_rem, offsets)
    split_k, M, N = A_rem.shape
    X = X.view(-1, split_k, N)
    _check_weight_call(A_rem, A_exp, X)
    Y = torch.empty((X.size(0), M), dtype=torch.bfloat16, device=A_rem.device)
    gemv_bf16_huffman(A_rem.contiguous(), A_exp.contiguous(), X.contiguous(), Y, offsets.contiguous(),
                      LUT1.contiguous(), LUT2.contiguous(), LUT3.contiguous(), LUT4.contiguous(),
                      code_lengths.contiguous())
    return Y


def mv_ans(A_rem: Tensor, A_exp: Tensor, X: Tensor, offsets: Tensor, LUT: Tensor) -> Tensor:
    """rANS counterpart of :func:`mv_huffman` (reference ``functional.py:414-444``)."""
    A_rem, offsets = _promote_single_split(A_rem, offsets)
    split_k, M, N = A_rem.shape
    X = X.view(-1, split_k, N)
    _check_weight_call(A_rem, A_exp, X)
    Y = torch.empty((X.size(0), M), dtype=torch.bfloat16, device=A_rem.device)
    gemv_bf16_ans(A_rem.contiguous(), A_exp.contiguous(), X.contiguous(), Y, offsets.contiguous(), LUT.contiguous())
    return Y


# what the names of these functions mean while nobody has put a wrapper in their place
_MV_HUFFMAN, _MV_ANS, _GEMV_HUFFMAN, _GEMV_ANS, _GEMV_GROUPED = (
    mv_huffman, mv_ans, gemv_bf16_huffman, gemv_bf16_ans, gemv_bf16_grouped)


class HuffmanWeight(nn.Module):
    """A BF16 weight ``[M, K]`` stored as a raw sign/mantissa plane plus a Huffman-coded
    exponent stream.  Passing the module as the weight of ``F.linear`` runs the fused
    kernels (reference ``functional.py:66-242``)."""

    def __init__(
        self,
        rem: Tensor,
        exp: Tensor,
        offsets: Tensor,
        LUT1: Tensor,
        LUT2: Tensor,
        LUT3: Tensor,
        LUT4: Tensor,
        code_lengths: Tensor,
    ):
        super().__init__()
        self.rem = nn.Buffer(rem)
        self.exp = nn.Buffer(exp)
        self.offsets = nn.Buffer(offsets)
        self.LUT1 = nn.Buffer(LUT1)
        self.LUT2 = nn.Buffer(LUT2)
        self.LUT3 = nn.Buffer(LUT3)
        self.LUT4 = nn.Buffer(LUT4)
        self.code_lengths = nn.Buffer(code_lengths)

    def kwargs(self) -> dict[str, Tensor]:
        return dict(self.named_buffers())

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        if func is not F.linear:
            return NotImplemented
        return linear_huffman(*args, **(kwargs or {}))

    def _empty_weight(self) -> Tensor:
        split_k, M, Ks = self.rem.shape
        assert self.rem.device.type == 'cuda'
        return torch.empty((M, split_k * Ks), dtype=torch.bfloat16, device=self.rem.device)

    def get_weight(self) -> Tensor:
        """The original BF16 weight, bit for bit."""
        if (weight := _eager_weight(self, True)) is not None:
            return weight
        weight = self._empty_weight()
        huffman_decode(self.rem, self.exp, weight, self.offsets,
                       self.LUT1, self.LUT2, self.LUT3, self.LUT4, self.code_lengths)
        return weight

    # ------------------------------------------------------------------ compression
    @classmethod
    def get_codec(cls, a: Tensor) -> LUTHuffmanEncoder:
        """One code per weight matrix, built from the histogram of exponent pairs."""
        return cls._codec_of(cls._pair_counts(_exponents(a)))

    @classmethod
    def _codec_of(cls, counts: Tensor) -> LUTHuffmanEncoder:
        """The code for int64 ``[65536]`` pair counts."""
        codec = LUTHuffmanEncoder()
        codec.build_lut(counts)
        return codec

    @staticmethod
    def _pair_counts(exp: Tensor) -> Tensor:
        """int64 [65536]: occurrences of every exponent pair ``a | b << 8`` (a = even column) of ``[M, K]``
        exponents, K even."""
        exp = exp.contiguous()
        if exp.size(1) % 2 == 0 and _kernel_counts(exp):
            return _ops.pair_histogram(exp)
        pairs = exp[:, 0::2].to(torch.int32) | (exp[:, 1::2].to(torch.int32) << 8)
        return torch.bincount(pairs.flatten(), minlength=65536)

    @classmethod
    def get_lut_kwargs(cls, codec: LUTHuffmanEncoder) -> dict[str, Tensor]:
        return {
            'LUT1': torch.from_numpy(codec.LUT1.copy()),
            'LUT2': torch.from_numpy(codec.LUT2.copy()),
            'LUT3': torch.from_numpy(codec.LUT3.copy()),
            'LUT4': torch.from_numpy(codec.LUT4.copy()),
            'code_lengths': torch.from_numpy(codec.code_lengths.copy()),
        }

    @classmethod
    def capacity(cls, n_steps: int) -> int:
        return encode_capacity(n_steps)

    @classmethod
    def compress_groups(cls, x: Tensor, codec) -> tuple[Tensor, Tensor]:
        """x: uint8 ``[tasks, steps*512]`` lane-ordered exponents of equally long tasks ->
        (streams int32 ``[tasks, capacity]``, words used per task)."""
        device = x.device
        n_steps = x.size(1) // (LANES * LANE_COLS)
        out = torch.zeros(x.size(0), cls.capacity(n_steps), dtype=torch.int32, device=device)
        lengths = torch.zeros(x.size(0), dtype=torch.int32, device=device)
        table = torch.from_numpy(codec.enc_table.view('int32').copy()).to(device)
        huffman_encode(x, table, out, lengths)
        return out, lengths

    @classmethod
    def compress_split_n(cls, a: Tensor, n: int = 2):
        """Compress ``a`` with ``n`` column splits (the reference's ``compress_split_n``,
        ``functional.py:195-238``)."""
        assert a.dim() == 2 and a.dtype == torch.bfloat16
        return cls(**{name: _to_host(t) for name, t in cls._compress_on_device(a, n).items()})

    @classmethod
    def _compress_on_device(cls, a: Tensor, n: int) -> dict[str, Tensor]:
        """The buffers of the compressed ``a``, on the GPU."""
        M, K = a.shape
        assert M % 128 == 0 and K % n == 0 and (K // n) % STEP_COLS == 0, a.shape
        Ks = K // n
        S, G = Ks // STEP_COLS, M // GROUP_ROWS
        device = torch.device('cuda', 0)
        lib = _lib.load()
        consts = _lib.constants()
        nc = lib.bhi_chunks_per_group(M, Ks, n)

        a = a.detach().to(device).contiguous()
        rem, sym = _ops.split_planes(a, n)
        if getattr(cls.get_codec, '__func__', None) in _COUNTING_CODECS:
            # what get_codec(a) gives, from the exponents at hand: another pass over `a` and its memory are 0.9 ms
            codec = cls._codec_of(_ops.pair_histogram(sym))
        else:
            codec = cls.get_codec(a)                                         # a subclass chooses its own
        del a

        lengths = torch.zeros(n, G, nc, dtype=torch.int64, device=device)
        pieces = []                                                          # (chunk, first task, streams, lengths)
        done = 0
        for c in range(nc):
            t0, t1 = (S * c) // nc, (S * (c + 1)) // nc
            size = (t1 - t0) * LANES * LANE_COLS
            tasks = sym[done:done + n * G * size].view(n * G, size)
            done += tasks.numel()
            per_call = max(1, ENCODE_PART_BYTES // (4 * cls.capacity(t1 - t0)))
            for first in range(0, n * G, per_call):
                out, ln = cls.compress_groups(tasks[first:first + per_call], codec)
                used = int(ln.max().item())
                pieces.append((c, first, out[:, :used].clone(), ln))
                lengths.view(n * G, nc)[first:first + ln.numel(), c] = ln
        del sym

        total = int(lengths.sum().item())
        assert total + consts['tail_pad_words'] < 2 ** 31, "exponent stream too large for int32 offsets"
        starts = (torch.cumsum(lengths.flatten(), 0) - lengths.flatten()).view(n * G, nc)
        words = torch.zeros(total + consts['tail_pad_words'], dtype=torch.int32, device=device)
        for c, first, out, ln in pieces:
            _ops.place_streams(out, ln, starts[first:first + ln.numel(), c], words)
        offsets = torch.zeros(n, G, GROUP_ROWS, dtype=torch.int32, device=device)
        offsets[:, :, :nc] = starts.view(n, G, nc).to(torch.int32)
        return dict(rem=rem, exp=words, offsets=offsets.view(n, M), **cls.get_lut_kwargs(codec))

    @classmethod
    def compress(cls, a: Tensor):
        return cls.compress_split_n(a, n=get_block_size_n(a)[0])


class ANSWeight(HuffmanWeight):
    """Same planes and stream layout with an interleaved rANS exponent stream
    (reference ``functional.py:245-310``)."""

    def __init__(self, rem: Tensor, exp: Tensor, offsets: Tensor, LUT: Tensor):
        nn.Module.__init__(self)
        self.rem = nn.Buffer(rem)
        self.exp = nn.Buffer(exp)
        self.offsets = nn.Buffer(offsets)
        self.LUT = nn.Buffer(torch.as_tensor(LUT))

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        if func is not F.linear:
            return NotImplemented
        return linear_ans(*args, **(kwargs or {}))

    def get_weight(self) -> Tensor:
        if (weight := _eager_weight(self, False)) is not None:
            return weight
        weight = self._empty_weight()
        ans_decode(self.rem, self.exp, weight, self.offsets, self.LUT)
        return weight

    @classmethod
    def get_codec(cls, a: Tensor) -> RANSEncoder:
        return RANSEncoder(_exponent_counts(_exponents(a)).tolist(), precision=ANS_PRECISION)

    @classmethod
    def _codec_of(cls, counts: Tensor) -> RANSEncoder:
        return RANSEncoder(_single_counts(counts).tolist(), precision=ANS_PRECISION)

    @classmethod
    def get_lut_kwargs(cls, codec: RANSEncoder) -> dict[str, Tensor]:
        lut = torch.tensor(codec.decode_lut, dtype=torch.int32)
        return {'LUT': (lut[:, 0] << 24) | (lut[:, 1] << 12) | lut[:, 2]}

    @classmethod
    def capacity(cls, n_steps: int) -> int:
        return ans_encode_capacity(n_steps)

    @classmethod
    def compress_groups(cls, x: Tensor, codec: RANSEncoder) -> tuple[Tensor, Tensor]:
        device = x.device
        n_steps = x.size(1) // (LANES * LANE_COLS)
        out = torch.zeros(x.size(0), cls.capacity(n_steps), dtype=torch.int32, device=device)
        lengths = torch.zeros(x.size(0), dtype=torch.int32, device=device)
        freq = torch.tensor(codec.freq, dtype=torch.int32, device=device)
        cum = torch.tensor(codec.cum, dtype=torch.int32, device=device)
        ans_encode(x, freq, cum, out, lengths)
        return out, lengths


class NibbleCodec:
    """Per-matrix parameters of the fixed-width code: the start of the 15-wide exponent
    window that covers the most weights, and whether anything falls outside it."""

    WINDOW = 15

    def __init__(self, counts: Tensor):
        counts = counts.to(torch.int64).cpu()
        assert counts.numel() == 256
        cover = counts.unfold(0, self.WINDOW, 1).sum(-1)          # cover[b] = counts[b : b + 15]
        # base + 15 (the escape nibble) must stay below 256: the decoder adds the base to four
        # nibbles with one 32-bit add, and a carry would spill into the neighbouring exponent
        cover = cover[:256 - self.WINDOW]
        self.base = int(torch.argmax(cover).item())               # first best window
        self.has_escapes = int(cover[self.base].item()) != int(counts.sum().item())


class NibbleWeight(ANSWeight):
    """Same planes and task layout with a fixed-width exponent code: 4 bits per exponent
    (offset from a per-matrix base, escape list for outliers).  Not one of the reference's
    codecs: about nine percent larger than the Huffman form and noticeably faster to
    multiply with, because its decoder has no tables, cursors or serial dependencies."""

    MAGIC = 0x4E494242          # LUT[2]: tells this module's LUT from a rANS slot table (whose frequency field is <= 256)

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        if func is not F.linear:
            return NotImplemented
        return linear_nibble(*args, **(kwargs or {}))

    def get_weight(self) -> Tensor:
        weight = self._empty_weight()
        nibble_decode(self.rem, self.exp, weight, self.offsets, self.LUT)
        return weight

    @classmethod
    def get_codec(cls, a: Tensor) -> NibbleCodec:
        return NibbleCodec(_exponent_counts(_exponents(a)))

    @classmethod
    def _codec_of(cls, counts: Tensor) -> NibbleCodec:
        return NibbleCodec(_single_counts(counts))

    @classmethod
    def get_lut_kwargs(cls, codec: NibbleCodec) -> dict[str, Tensor]:
        lut = torch.zeros(256, dtype=torch.int32)
        lut[0], lut[1], lut[2] = codec.base, int(codec.has_escapes), cls.MAGIC
        return {'LUT': lut}

    @classmethod
    def capacity(cls, n_steps: int) -> int:
        return nibble_encode_capacity(n_steps)

    @classmethod
    def compress_groups(cls, x: Tensor, codec: NibbleCodec) -> tuple[Tensor, Tensor]:
        device = x.device
        n_steps = x.size(1) // (LANES * LANE_COLS)
        out = torch.zeros(x.size(0), cls.capacity(n_steps), dtype=torch.int32, device=device)
        lengths = torch.zeros(x.size(0), dtype=torch.int32, device=device)
        nibble_encode(x, cls.get_lut_kwargs(codec)['LUT'].to(device), out, lengths)
        return out, lengths


_COUNTING_CODECS = [c.get_codec.__func__ for c in (HuffmanWeight, ANSWeight, NibbleWeight)]


class CompressedLinear(nn.Module):
    def __init__(self, weight: HuffmanWeight, bias: Optional[Tensor]) -> None:
        super().__init__()
        self.weight = weight
        self.bias = bias
        self._group = None          # a LinearGroup when this module shares launches with siblings

    def forward(self, input: Tensor) -> Tensor:
        group = getattr(self, '_group', None)
        if group is not None:
            return group.forward(self, input)
        return F.linear(input, self.weight, self.bias)


def fuses_input(rows: int, n_weights: int, norm: bool, huffman: bool, in_graph: bool = True) -> bool:
    """Whether the RMSNorm (``norm``) or the SwiGLU product in front of a GEMV of ``n_weights`` weights
    in all happens inside its launch or in a launch of its own.

    A launch of its own costs 2.4 us.  Inside, every wavefront transforms the X of every step and row
    it multiplies, in a kernel whose steps are short of issue slots as it is: the cost grows with rows
    times weights.  Measured on MI355X in recorded graphs (us, inside / of its own):

    ==================================  ===========  ===========  ===========  ===========
    launch                              1 row        2 rows       3 rows       4 rows
    ==================================  ===========  ===========  ===========  ===========
    Huffman, norm, 1536x1024            5.9 / 7.0    6.2 / 7.6    6.6 / 7.5    6.9 / 7.7
    Huffman, norm, 3072x2048            8.1 / 8.6    8.7 / 9.3    9.6 / 9.5    10.3 / 9.7
    Huffman, norm, 4608x3584            11.3 / 11.4  12.5 / 12.1  14.3 / 12.9  16.2 / 13.6
    Huffman, norm, 6144x4096            12.7 / 13.0  14.6 / 13.9  18.8 / 14.4  20.8 / 15.2
    Huffman, norm, 24576x4096           34.4 / 32.6  38.8 / 34.9  46.9 / 36.6  50.8 / 34.2
    Huffman, SwiGLU, 1024x3072          6.4 / 8.0    6.7 / 8.4    7.1 / 8.4    7.7 / 8.6
    Huffman, SwiGLU, 2048x8192          11.3 / 12.6  13.2 / 12.9  14.9 / 13.2  16.7 / 13.5
    Huffman, SwiGLU, 4096x12288         20.8 / 21.0  26.0 / 21.7  31.9 / 21.7  36.1 / 22.8
    Huffman, SwiGLU, 3584x18944         28.8 / 26.3  34.9 / 28.0  42.6 / 29.5  49.6 / 30.3
    rANS, norm, 6144x4096               16.0 / 16.1  18.4 / 17.2  21.7 / 17.6  24.6 / 18.2
    rANS, norm, 24576x4096              44.0 / 40.7  49.7 / 43.5  57.6 / 46.0  65.2 / 43.7
    rANS, SwiGLU, 1024x3072             7.1 / 8.8    7.6 / 9.0    8.1 / 9.2    8.6 / 9.4
    rANS, SwiGLU, 2048x8192             14.6 / 15.0  16.1 / 15.2  17.7 / 15.4  19.2 / 15.8
    rANS, SwiGLU, 4096x12288            28.8 / 26.1  34.1 / 27.0  38.9 / 27.4  42.4 / 28.2
    ==================================  ===========  ===========  ===========  ===========

    Outside a graph (``in_graph=False``) another launch is 8 to 11 us of host time, and most of these calls are bound by
    the host (us per call):

    ==================================  ===========  ===========  ===========
    eager call                          1 row        2 rows       4 rows
    ==================================  ===========  ===========  ===========
    Huffman, norm, 4608x3584            20.7 / 31.6  20.8 / 31.0  22.3 / 31.2
    Huffman, norm, 24576x4096           30.8 / 38.9  34.7 / 39.2  45.2 / 45.7
    Huffman, SwiGLU, 4096x12288         20.9 / 28.8  22.4 / 28.9  33.7 / 28.9
    Huffman, SwiGLU, 3584x18944         23.7 / 28.9  29.7 / 28.9  46.3 / 33.6
    rANS, norm, 24576x4096              38.5 / 41.1  42.5 / 42.1  58.4 / 46.2
    rANS, SwiGLU, 4096x12288            24.2 / 30.9  29.7 / 30.0  40.7 / 30.3
    rANS, SwiGLU, 3584x18944            33.2 / 30.5  42.1 / 30.9  57.8 / 34.4
    ==================================  ===========  ===========  ===========
    """
    if rows > _ops.X_TRANSFORM_MAX_ROWS:
        return False
    if not in_graph:
        return rows * n_weights <= ((210e6 if norm else 110e6) if huffman else (150e6 if norm else 60e6))
    if rows == 1:
        return n_weights <= (28e6 if norm else 51e6 if huffman else 20e6)
    return rows * n_weights <= (18e6 if norm else 22e6)


def linear_grouped(input: Tensor, weights, biases=None, *, residuals=None, input_norm=None, input_gate=None,
                   outs=None) -> list:
    """``[F.linear(h, w, b) (+ r) for w, b, r in zip(weights, biases, residuals)]`` in ONE launch, where
    ``h`` is ``input``, or -- so that the layer in front of the linears needs no kernel of its own --

    * ``input_norm=(gamma, eps)``: ``h = rms_norm(input) * gamma`` (RMSNorm in front of q/k/v or gate/up),
    * ``input_gate=gate``: ``h = silu(gate) * input`` (the SwiGLU product in front of down_proj).

    ``weights`` are up to four compressed weights of one class with the same
    ``in_features`` split (``rem.shape[0]`` and ``rem.shape[2]``); ``input`` has at most
    8 rows after flattening.  ``residuals[i]`` (shaped like output ``i``) is added last, as a
    separate BF16 addition would; ``outs[i]`` (bf16 ``[rows, M_i]``, contiguous -- a column slice of a
    one-row buffer qualifies) receives output ``i`` instead of a new tensor.  This is what the q/k/v (or gate/up) projections of a
    decoder layer need: the reference overlaps them on parallel streams
    (``cudastream_utils.py:8-47``), here they are one grid.  Where it pays (:func:`fuses_input`) the
    norm / gate product happens inside the kernel; otherwise it runs as this package's own
    elementwise kernel first -- the same arithmetic, the same bits.
    """
    assert input.dim() >= 2, input
    assert input_norm is None or input_gate is None, "one transform of the input at a time"
    shape = input.shape
    x = input.flatten(0, -2)
    if x.size(0) > MAX_FUSED_BATCH:
        raise RuntimeError(f'linear_grouped takes at most {MAX_FUSED_BATCH} rows, got {x.size(0)}')
    first = weights[0]
    split_k, _, N = first.rem.shape
    mode, aux, eps = _ops.X_PLAIN, None, 0.0
    if input_norm is not None or input_gate is not None:
        fusable = not isinstance(first, NibbleWeight) and fuses_input(
            x.size(0), sum(w.rem.numel() for w in weights), input_norm is not None, hasattr(first, 'LUT1'), recorded())
        if input_norm is not None:
            gamma, eps = input_norm
            gamma = gamma.detach()
            if fusable:
                mode, aux = _ops.X_RMS, gamma.contiguous()
            else:
                x = _ops.rms_norm(x, gamma, eps)
        else:
            gate = input_gate.flatten(0, -2)
            assert gate.shape == x.shape, (gate.shape, x.shape)
            if fusable:
                mode, aux = _ops.X_SILU_MUL, gate.contiguous()
            else:
                x = _ops.silu_mul(gate, x)
    x = x.view(-1, split_k, N)
    _check_weight_call(first.rem, first.exp, x)
    if outs is not None:
        ys = [o.view(x.size(0), w.rem.shape[1]) for o, w in zip(outs, weights)]
    else:
        ys = [torch.empty((x.size(0), w.rem.shape[1]), dtype=torch.bfloat16, device=x.device) for w in weights]
    if biases is not None:
        biases = [None if b is None else b.detach().contiguous() for b in biases]
    if residuals is not None:
        residuals = [None if r is None else r.detach().reshape(x.size(0), -1).contiguous() for r in residuals]
    total = sum(w.rem.shape[1] for w in weights)
    if (mode == _ops.X_PLAIN and not isinstance(first, NibbleWeight)
            and (all(prefers_matrix_cores(x.size(0), w.rem.shape[1], split_k * N) for w in weights)
                 or prefers_matrix_cores(x.size(0), total, split_k * N))):
        # layers this large -- or this large together -- are faster through the matrix-core kernel
        gemm_bf16_grouped(weights, x.contiguous(), ys, biases, residuals)
    else:
        gemv_bf16_grouped(weights, x.contiguous(), ys, biases, residuals, mode, aux, float(eps))
    return [y.unflatten(0, shape[:-1]) for y in ys]


class LinearGroup:
    """Sibling :class:`CompressedLinear` modules that a model always calls one after the
    other on the same input tensor (q/k/v of an attention block, gate/up of an MLP).

    The call of the first member computes every member's output in one grouped launch
    and keeps the others until their own call collects them.  Whatever does not fit that
    pattern -- more than 8 rows, a member called alone or on another tensor, weights of
    different codecs or splits -- runs each member's ordinary path.  Grouping changes the
    number of launches and, where members that are large only together move to the matrix-core
    kernel (:func:`prefers_matrix_cores`), the order of the fp32 sums: a last bit of BF16 here
    and there, nothing else.
    """

    def __init__(self, members):
        self.members = list(members)
        for m in self.members:
            if not isinstance(m, CompressedLinear):
                raise TypeError('LinearGroup takes CompressedLinear modules')
        if not 2 <= len(self.members) <= 4:
            raise ValueError('a group has 2 to 4 members')
        first = self.members[0].weight
        self.uniform = all(type(m.weight) is type(first) and m.weight.rem.shape[0] == first.rem.shape[0]
                           and m.weight.rem.shape[2] == first.rem.shape[2] for m in self.members)
        self._input = None
        self._outputs = None
        for m in self.members:
            m._group = self

    def _biases_fit(self, input: Tensor) -> bool:
        """The grouped launch adds BF16 biases on the input's device; anything else takes the
        members' own path (``output += bias``), as an ungrouped module would."""
        return all(m.bias is None or (m.bias.dtype == torch.bfloat16 and m.bias.device == input.device)
                   for m in self.members)

    def dissolve(self) -> None:
        for m in self.members:
            m._group = None

    def forward(self, module: CompressedLinear, input: Tensor) -> Tensor:
        index = next(i for i, m in enumerate(self.members) if m is module)
        if index == 0:
            self._input = self._outputs = None
            rows = input.numel() // input.shape[-1] if input.dim() >= 2 else MAX_FUSED_BATCH + 1
            if self.uniform and input.is_cuda and rows <= MAX_FUSED_BATCH and self._biases_fit(input):
                self._outputs = linear_grouped(input, [m.weight for m in self.members],
                                               [m.bias for m in self.members])
                self._input = input
                return self._outputs[0]
        elif self._input is input and self._outputs is not None:
            out = self._outputs[index]
            self._outputs[index] = None
            if index == len(self.members) - 1:
                self._input = self._outputs = None
            if out is not None:
                return out
        return F.linear(input, module.weight, module.bias)


def _weight_bytes(w: nn.Module) -> int:
    return sum(b.nelement() * b.element_size() for b in w.buffers())


@contextlib.contextmanager
def _visiting_gpu(module: nn.Module):
    """``module`` on the current GPU for a while, then in host memory.  Parameters that lay there get their
    own storage back: nothing is copied, and the pages of a copy (:func:`_to_host`) need not be touched."""
    at_home = [(p, p.data) for p in module.parameters() if not p.is_cuda]
    try:
        yield module.cuda()
    finally:
        for p, data in at_home:
            p.data = data
        module.cpu()


def convert(linear: nn.Linear, name, disable_precision_check=True, algo='huffman') -> nn.Module:
    """Compress one ``nn.Linear`` (reference ``functional.py:323-375``).

    Returns the original module when compression does not shrink it or when the decoded
    weight is not bit-identical; with ``disable_precision_check=False`` also when one
    random GEMV deviates by 2 % or more from the dense layer.
    """
    assert algo in ('huffman', 'ans', 'smallest', 'nibble')
    n = get_block_size_n(linear.weight)[0]
    assert linear.weight.dim() == 2 and linear.weight.dtype == torch.bfloat16
    classes = {'huffman': [HuffmanWeight], 'ans': [ANSWeight], 'nibble': [NibbleWeight],
               'smallest': [HuffmanWeight, ANSWeight]}[algo]
    with _visiting_gpu(linear):
        dense = linear.weight.detach()
        compressed = min([cls(**cls._compress_on_device(dense, n)) for cls in classes], key=_weight_bytes)
        ratio = _weight_bytes(compressed) / (dense.nelement() * dense.element_size())
        module = CompressedLinear(weight=compressed.cuda(), bias=linear.bias)
        x = torch.randn(1, linear.in_features, dtype=torch.bfloat16, device='cuda')
        with torch.no_grad():
            # the layer itself: a subclass's forward and whatever hooks it has are part of the comparison
            y1 = linear(x)
            y2 = module(x)
            lossless = torch.equal(compressed.get_weight().view(torch.int16), dense.view(torch.int16))
        max_rtol = ((y2 - y1).abs() / y1.abs().clamp(min=1e-4)).max().item()
        del dense
    module.bias = linear.bias

    fallback = False
    if ratio >= 1:
        print(f'\nWarning! {name} ratio = {ratio:.2%}')
        fallback = True
    if not lossless:
        print(f'\nWarning! {name} does not decode to the original weight')
        fallback = True
    if not disable_precision_check and max_rtol >= 0.02:
        print(f'\nWarning! {name} output mismatch: max rtol = {max_rtol:.2f}')
        fallback = True
    if fallback:
        print('Fallback to regular nn.Linear')
        return linear
    compressed._apply(_to_host)
    return module


def convert_all_linear(model: nn.Module, min_out_features=4096, progress=True, algo='huffman') -> None:
    """Replace every ``nn.Linear`` with at least ``min_out_features`` outputs in place."""
    targets = [name for name, m in model.named_modules()
               if isinstance(m, nn.Linear) and m.out_features >= min_out_features]
    for name in tqdm(targets, disable=not progress):
        model.set_submodule(name, convert(model.get_submodule(name), name, algo=algo))


def linear_nibble(input: Tensor, weight: NibbleWeight, bias: Optional[Tensor] = None) -> Tensor:
    """``F.linear`` with a :class:`NibbleWeight` (fused up to 8 rows, else decode + GEMM)."""
    def fused(x):
        split_k, M, N = weight.rem.shape
        x = x.view(-1, split_k, N)
        _check_weight_call(weight.rem, weight.exp, x)
        y = torch.empty((x.size(0), M), dtype=torch.bfloat16, device=x.device)
        gemv_bf16_nibble(weight.rem, weight.exp, x.contiguous(), y, weight.offsets, weight.LUT)
        return y
    return _linear_compressed(input, weight, bias, fused)


def check_layout(weight: "HuffmanWeight") -> None:
    """Raises unless ``weight``'s buffers are in THIS package's task layout.

    A weight saved by the reference package has the same buffer names, dtypes and (for rANS)
    shapes, but its ``offsets`` are per row and its stream has no zero tail: the kernels would
    read it as garbage, past the end of ``exp``.  Checked: the format header (Huffman), unused
    chunk slots of ``offsets`` are 0, offsets are aligned and ascending in task order, the last
    task ends in front of the tail pad, and the tail pad is zero."""
    consts = _lib.constants()
    lib = _lib.load()
    hint = ('; a weight compressed by the reference package must be converted with '
            'bf16_huffman_infer_amd.reference_format.transcode_reference_weight')
    rem, exp, offsets = weight.rem, weight.exp, weight.offsets
    if rem.dim() != 3 or offsets.dim() != 2 or tuple(offsets.shape) != tuple(rem.shape[:2]):
        raise RuntimeError(f'compressed weight: rem {tuple(rem.shape)} / offsets {tuple(offsets.shape)} do not fit' + hint)
    split_k, M, Ks = rem.shape
    if isinstance(weight, HuffmanWeight) and hasattr(weight, 'LUT1'):
        header = weight.code_lengths.flatten()[:2].tolist()
        if weight.LUT1.numel() != 4 << consts['table_bits'] or header != [consts['format_version'], consts['table_bits']]:
            raise RuntimeError('compressed weight: Huffman tables are not in this package\'s format' + hint)
    if M % GROUP_ROWS or Ks % STEP_COLS:
        raise RuntimeError(f'compressed weight: {M}x{split_k * Ks} does not fit the task layout' + hint)
    nc = lib.bhi_chunks_per_group(M, Ks, split_k)
    pad, align = consts['tail_pad_words'], consts['align_words']
    off = offsets.reshape(split_k, M // GROUP_ROWS, GROUP_ROWS).to(torch.int64)
    used = off[:, :, :nc].flatten()
    ok = (exp.numel() >= pad and not bool(off[:, :, nc:].any()) and not bool((used % align).any())
          and bool((used[1:] > used[:-1]).all()) and int(used[0]) == 0 and int(used[-1]) < exp.numel() - pad
          and not bool(exp[exp.numel() - pad:].any()))
    if not ok:
        raise RuntimeError('compressed weight: offsets / exp are not in this package\'s task layout' + hint)


def load_compressed_state_dict(model: nn.Module, state_dict: dict, strict: bool = True):
    """Load the ``state_dict()`` of a converted model into a freshly built, unconverted one.

    The reference leaves this to the user (its converted modules only exist after
    ``convert_all_linear`` has run on real weights).  Here every ``nn.Linear`` of ``model``
    whose compressed buffers are in ``state_dict`` (``<name>.weight.rem`` ...) is replaced
    by a :class:`CompressedLinear` around those tensors -- ``LUT1`` present means Huffman,
    ``LUT`` means rANS or (by its marker word) the nibble code -- and the remaining entries go through ``load_state_dict``.  The
    skeleton's linears may live on the meta device; nothing is decoded or re-encoded.
    """
    huffman_keys = ('rem', 'exp', 'offsets', 'LUT1', 'LUT2', 'LUT3', 'LUT4', 'code_lengths')
    ans_keys = ('rem', 'exp', 'offsets', 'LUT')
    for name, module in list(model.named_modules()):
        if not isinstance(module, nn.Linear) or f'{name}.weight.rem' not in state_dict:
            continue
        keys = huffman_keys if f'{name}.weight.LUT1' in state_dict else ans_keys
        if keys is huffman_keys:
            cls = HuffmanWeight
        else:
            nibble = int(state_dict[f'{name}.weight.LUT'][2]) == NibbleWeight.MAGIC
            cls = NibbleWeight if nibble else ANSWeight
        weight = cls(**{k: state_dict[f'{name}.weight.{k}'] for k in keys})
        check_layout(weight)
        split_k, M, Ks = weight.rem.shape
        if (M, split_k * Ks) != (module.out_features, module.in_features):
            raise RuntimeError(f'{name}: compressed weight is {M}x{split_k * Ks}, '
                               f'the module expects {module.out_features}x{module.in_features}')
        bias = state_dict.get(f'{name}.bias')
        if bias is not None:
            bias = nn.Parameter(bias, requires_grad=False)
        model.set_submodule(name, CompressedLinear(weight=weight, bias=bias))
    return model.load_state_dict(state_dict, strict=strict, assign=True)


def prefers_matrix_cores(rows: int, M: int, K: int) -> bool:
    """Whether ``rows`` <= 8 rows of activations go through the matrix-core kernel rather than the
    GEMV.  The GEMV spends four dot products per row and step and one load of X per row; the
    matrix-core kernel shares X among the wavefronts of a block through LDS and costs the same for
    5..8 rows, but starts slower and keeps fewer wavefronts on a compute unit.  Measured on MI355X
    (us, GEMV / matrix cores):

    ===========  ===========  ===========  ===========  ===========
    M x K        4 rows       5 rows       6 rows       8 rows
    ===========  ===========  ===========  ===========  ===========
    3584x18944   26.4 / 25.9  29.3 / 28.4  31.5 / 28.7  36.8 / 29.3
    14336x4096   21.8 / 20.5  23.6 / 22.5  25.2 / 22.5  28.4 / 22.5
    18944x3584   23.4 / 23.9  25.3 / 26.1  27.0 / 26.1  30.8 / 26.2
    12288x4096   19.0 / 19.4  20.6 / 21.2  23.9 / 21.2  26.4 / 21.2
    11008x4096   18.6 / 19.0  20.3 / 20.7  23.2 / 20.8  25.3 / 20.8
    4096x14336   21.9 / 22.8  24.1 / 24.4  26.0 / 24.8  29.5 / 25.5
    4096x12288   22.1 / 26.1  24.6 / 27.7  25.7 / 27.8  28.6 / 28.0
    4096x11008   18.6 / 20.7  20.5 / 22.7  21.7 / 23.1  24.7 / 23.8
    8192x8192    23.1 / 27.7  25.1 / 30.0  27.1 / 30.2  30.8 / 30.3
    ===========  ===========  ===========  ===========  ===========

    and the layers of 6144x4096 and below are 0.4-4 us faster on the GEMV at every row count; output
    layers the size of a vocabulary -- or a group of layers that large together -- are faster on the
    matrix cores from 3 rows (152064x3584: 138 / 147, 157 / 148, 180 / 148, 225 / 185 us at 2, 3, 4, 8
    rows; 37888x3584: 39.1 / 39.6, 41.9 / 39.7, 44.4 / 39.8, 58.7 / 48.9).  The rANS kernels cross over
    at the same places (18944x3584 at 6 rows 37.7 / 36.0, 3584x18944 at 4 rows 34.7 / 33.9,
    37888x3584 at 3 rows 53.6 / 51.2)."""
    return bool(_lib.load().bhi_prefers_matrix_cores(rows, M, K))


@functools.lru_cache(maxsize=1024)        # an eager call asks every time
def prefers_tiles(rows: int, M: int, K: int, split_k: int = 1, huffman: bool = True) -> bool:
    """Whether ``rows`` > 16 rows of activations go through the tiled product (``bhi_tile.h``) rather than
    the matrix-core kernel (up to 32 rows) or decoding and a dense GEMM (above).  Measured on MI355X in
    recorded graphs, 37 shapes of 13 row counts and both codecs (us, the other path / tiled; four copies of
    a weight in turn):

    =======================  ===========  ===========  ===========  ===========  ===========
    M x K                    17 rows      24 rows      32 rows      64 rows      96 rows
    =======================  ===========  ===========  ===========  ===========  ===========
    640x1024 Huffman         12.9 / 9.8   14.2 / 9.8   16.6 / 10.0  12.3 / 12.1  11.8 / 14.4
    640x1024 rANS            13.8 / 11.3  15.1 / 11.2  17.3 / 11.4  12.6 / 13.6  12.4 / 15.9
    4096x4096 Huffman        22.2 / 16.9  24.5 / 16.6  28.6 / 16.7  27.4 / 20.2  32.6 / 24.5
    12288x4096 Huffman       28.3 / 27.7  29.7 / 27.1  33.7 / 27.5  56.4 / 33.6  57.3 / 40.7
    12288x4096 rANS          35.6 / 37.3  36.5 / 36.7  40.0 / 37.0  59.0 / 41.5  59.0 / 51.7
    4096x11008 rANS          37.5 / 40.7  40.0 / 40.4  44.8 / 40.4  58.2 / 44.8  69.0 / 51.4
    4096x12288 rANS          42.4 / 37.6  44.6 / 37.2  50.4 / 37.2  62.0 / 44.1  76.6 / 53.1
    1024x18944 rANS          31.7 / 35.2  34.5 / 35.3  37.9 / 35.3  67.8 / 39.7  68.9 / 46.1
    3584x18944 Huffman       41.2 / 47.7  44.8 / 47.6  50.7 / 48.1  102 / 58.3   108 / 63.9
    3584x18944 rANS          50.7 / 70.5  53.6 / 70.3  60.1 / 70.7  104 / 76.3   109 / 75.7
    16384x3584 Huffman       29.7 / 38.9  31.1 / 38.7  35.1 / 39.0  56.1 / 45.8  58.0 / 46.9
    18944x3584 Huffman       44.5 / 36.2  47.5 / 36.2  55.2 / 36.5  65.1 / 43.9  67.6 / 59.6
    18944x3584 rANS          56.4 / 53.1  59.7 / 53.2  66.5 / 53.5  66.4 / 57.9  69.2 / 80.6
    =======================  ===========  ===========  ===========  ===========  ===========
    """
    tasks = split_k * _lib.load().bhi_chunks_per_group(M, K // split_k, split_k)      # of a row group
    steps = K / (STEP_COLS * tasks)                                                   # of a task
    if rows <= 32:
        # The other kernel is at its best with 12 to 16 wavefronts for every compute unit (it is cut along K
        # below 8192 rows only) and pays for each four rows of X; this one lags on long tasks, whose lanes
        # drift out of the ring, and its rANS steps cost more.
        waves = (M if M >= 8192 else M * tasks) / (4 * 256)
        if 12 < waves <= 16 and steps > 24:
            return huffman and rows > 28 and tasks > 1
        if huffman or rows > 20:
            return True
        return waves > 16 or (M >= 8192 and waves > 12) or (steps < 13 and K < 16384)
    if rows <= 64:
        # a small layer's weight stays in the caches between the decoder and the GEMM
        return huffman or rows <= 48 or M * K >= 7 << 18
    # Above, the library's kernel gains on this one with every row.  With one task per row group and four to
    # five wavefronts for a unit, blocks of six or eight leave a quarter of the units idle (F.linear asks prefers_wide
    # first, which takes all of these).
    if M * K < 16 << 20:
        return False
    return huffman or rows <= 80 or not (tasks == 1 and 4 * 4096 < M < 5 * 4096)


@functools.lru_cache(maxsize=1024)
def prefers_wide(rows: int, M: int, K: int, split_k: int = 1, huffman: bool = True) -> bool:
    """Whether 17 to 640 rows of activations go through the wide product (``bhi_wide.h``) rather than what
    :func:`prefers_tiles` and the paths behind it choose.  Its blocks of 64 weight rows, cut along K as long as
    every block has a compute unit of its own, cover the units in rounds; what counts is how full the
    last one is.  Measured on MI355X in recorded graphs, twelve shapes of 17 row counts and both codecs (us, the
    other path / wide; more in ``bhi_wide.h``):

    ================================  ===========  ===========  ===========  ===========  ===========
    M x K (filled units)              32 rows      64 rows      96 rows      256 rows     640 rows
    ================================  ===========  ===========  ===========  ===========  ===========
    512x1024 (6 %) Huffman            10.0 / 10.4  12.1 / 11.1  12.3 / 12.2  12.7 / 15.9  13.1 / 27.1
    1024x4096 (25 %) Huffman          15.0 / 14.6  18.2 / 16.0  17.3 / 17.6  21.7 / 25.2  27.3 / 45.4
    2048x2048 (50 %) rANS             13.4 / 13.6  16.1 / 14.4  17.0 / 16.6  20.6 / 23.4  24.3 / 38.3
    4608x3584 (56 %) Huffman          18.1 / 19.4  22.5 / 21.5  32.4 / 23.2  46.4 / 31.7  44.8 / 55.0
    12288x4096 (75 %) Huffman         29.9 / 32.2  35.6 / 35.6  42.7 / 37.0  79.3 / 50.3  97.4 / 92.0
    3584x3584 (88 %) rANS             18.9 / 18.1  21.8 / 18.8  30.3 / 21.8  29.8 / 29.9  42.0 / 48.0
    4096x12288 (100 %) rANS           39.7 / 38.2  46.2 / 40.5  55.0 / 43.5  81.5 / 58.8   123 / 96.6
    8192x8192 (100 %) Huffman         44.2 / 35.4  52.8 / 40.4  57.8 / 42.8   105 / 61.7   121 / 116
    18944x3584 (two rounds, 58 %) H   38.2 / 49.8  45.2 / 54.8  61.4 / 57.1  86.0 / 79.3   122 / 145
    18944x3584 (two rounds, 58 %) r   55.5 / 63.0  59.5 / 67.6  71.0 / 69.2  90.5 / 90.9   130 / 149
    32768x2048 (two rounds, full) r   36.4 / 42.7  42.8 / 45.6  47.1 / 47.0  86.2 / 67.1   128 / 113
    ================================  ===========  ===========  ===========  ===========  ===========

    The limits lie between neighbouring measured shapes and row counts and have no other reason.  Of the entries here and
    in ``bhi_wide.h`` four are left to the slower path: 512x1024 at 64 rows, 1024x4096 at 32, rANS 3584x3584 at 32
    (by 0.4 to 1.0 us) and 4096x4096 at 300 (by 2.4).
    """
    slices = _lib.load().bhi_wide_slices(split_k, M, K // split_k)
    if slices < 1 or M < 128 or M % 128 != 0:     # refused by the library, or by the operand check of every fused call
        return False
    blocks = M // 64 * slices
    rounds = -(-blocks // 256)
    filled = blocks / (256 * rounds)
    weights = M * K
    useful = filled * weights              # a layer that leaves units idle needs more work per block to win
    if rows > 128:
        if rounds > 1 and filled < 0.75:
            return rows <= (320 if huffman else 192)
        return useful >= 8 << 20 and rows <= (256 if useful < 24 << 20 else _ops.WIDE_MAX_ROWS)
    if rounds > 1:
        return rows > 80
    if rows <= 32:
        return filled >= 0.85 and weights >= 32 << 20
    if filled >= 0.85 and weights >= 8 << 20:
        return True
    if weights < 4 << 20:
        return False
    if useful < 8 << 20:
        return 48 < rows <= (96 if filled >= 0.5 else 64)
    return rows > (64 if slices == 1 else 48)


def _fuses_above_32_rows(input: Tensor, bias: Optional[Tensor]) -> bool:
    """Decoding and ``F.linear`` pass gradients, forward-mode tangents, function transforms, autocast, dispatch
    modes and tracing on to the input (and the bias); a fused product does not, and takes over only where
    none of them is in play."""
    if torch.is_grad_enabled() and (input.requires_grad or (bias is not None and bias.requires_grad)):
        return False
    if torch.autograd.forward_ad._current_level >= 0 or torch._C._functorch.peek_interpreter_stack() is not None:
        return False
    if torch.is_autocast_enabled('cuda') or torch._C._len_torch_dispatch_stack():
        return False
    if torch.compiler.is_compiling() or torch._C._get_tracing_state() is not None:       # torch.compile / export; torch.jit.trace
        return False
    return type(input) in (Tensor, nn.Parameter)


def _takes(input: Tensor, weight: HuffmanWeight, bias: Optional[Tensor], first: int, last: int, rule) -> bool:
    """Whether a fused product for ``first`` to ``last`` rows takes the place of what runs else: its operands fit
    it, ``rule`` wants it, and above 32 rows nothing is asked for but the value."""
    rows = input.size(0)
    if not first <= rows <= last or isinstance(weight, NibbleWeight):
        return False
    split_k, M, N = _ops._buffer(weight, 'rem').shape
    if input.dtype != torch.bfloat16 or (bias is not None and bias.dtype != torch.bfloat16) or not input.is_cuda:
        return False
    if split_k < 1 or input.size(1) != split_k * N or input.numel() >= 2 ** 31:
        return False
    # whole numbers: under torch.jit.trace these are tensors, which the rules would keep
    if not rule(int(rows), int(M), int(split_k * N), int(split_k), not isinstance(weight, ANSWeight)):
        return False
    return rows <= GEMM_MAX_ROWS or ((bias is None or tuple(bias.shape) == (M,)) and _fuses_above_32_rows(input, bias))


def _tiled(input: Tensor, weight: HuffmanWeight, bias: Optional[Tensor]) -> bool:
    return _takes(input, weight, bias, _ops.TILE_MIN_ROWS, _ops.TILE_MAX_ROWS, prefers_tiles)


def _wide(input: Tensor, weight: HuffmanWeight, bias: Optional[Tensor]) -> bool:
    return (_takes(input, weight, bias, _ops.WIDE_MIN_ROWS, _ops.WIDE_MAX_ROWS, prefers_wide)
            and (input.size(0) + 15) * input.size(1) < 2 ** 31)


def _linear_compressed(input: Tensor, weight: HuffmanWeight, bias: Optional[Tensor], fused) -> Tensor:
    assert input.dim() >= 2, input
    shape = input.shape
    if len(shape) > 2:
        input = input.flatten(0, -2)
    rows = input.size(0)
    split_k, M, N = _ops._buffer(weight, 'rem').shape
    if rows == 0:                       # no rows: nothing to launch
        return input.new_empty((*shape[:-1], M))
    matrix_cores = (not isinstance(weight, NibbleWeight) and input.dtype == torch.bfloat16
                    and (bias is None or bias.dtype == torch.bfloat16))
    wide = rows <= MAX_FUSED_BATCH and matrix_cores and prefers_matrix_cores(rows, M, split_k * N)
    if rows <= MAX_FUSED_BATCH and not wide:
        if bias is not None and bias.dtype == torch.bfloat16:
            # the grouped entry point adds the bias in the kernel's last store (same bits, one launch less)
            x = input.view(-1, split_k, N)
            _check_weight_call(weight.rem, weight.exp, x)
            output = torch.empty((rows, M), dtype=torch.bfloat16, device=x.device)
            gemv_bf16_grouped([weight], x.contiguous(), [output], [bias.detach().contiguous()])
        else:
            output = fused(input)
            if bias is not None:
                output += bias[None, :]
    elif matrix_cores and rows > MAX_FUSED_BATCH and (
            product := _ops.wide_bf16 if _wide(input, weight, bias) else _ops.tile_bf16 if _tiled(input, weight, bias) else None):
        # 17..640 rows where the rules say so: as below, but the matrix instructions take sixteen weight rows, in the
        # wide product out of LDS, where a block has decoded 64
        x = (input if rows <= GEMM_MAX_ROWS else input.contiguous()).view(-1, split_k, N).contiguous()
        if x.data_ptr() % 16:
            x = x.clone()
        _check_weight_call(weight.rem, weight.exp, x)
        output = torch.empty((rows, M), dtype=torch.bfloat16, device=x.device)
        product(weight, x, output, None if bias is None else bias.detach().contiguous())
    elif wide or (rows <= GEMM_MAX_ROWS and matrix_cores):
        # up to 32 rows that neither the GEMV nor the tiled product takes: decode inside the matrix-core kernel,
        # no BF16 weight in memory
        x = input.view(-1, split_k, N)
        _check_weight_call(weight.rem, weight.exp, x)
        output = torch.empty((rows, M), dtype=torch.bfloat16, device=x.device)
        gemm_bf16(weight, x.contiguous(), output, None if bias is None else bias.detach().contiguous())
    else:
        output = F.linear(input, weight.get_weight(), bias)
    return output if len(shape) == 2 else output.unflatten(0, shape[:-1])


def _eager(input: Tensor, weight: HuffmanWeight, bias: Optional[Tensor], huffman: bool) -> Optional[Tensor]:
    """A call of the GEMV that nothing watches, in one native step (``bhi_torch.cpp``); None where the path through the
    custom ops has to take it or to refuse it.  Whoever has put a wrapper in the place of this module's
    ``mv_huffman`` / ``mv_ans`` or of the ops that they and a call with a bias run, ``gemv_bf16_huffman`` /
    ``gemv_bf16_ans`` and ``gemv_bf16_grouped`` (to count or to log calls), watches too."""
    if torch.compiler.is_compiling() or gemv_bf16_grouped is not _GEMV_GROUPED or not (
            mv_huffman is _MV_HUFFMAN and gemv_bf16_huffman is _GEMV_HUFFMAN if huffman
            else mv_ans is _MV_ANS and gemv_bf16_ans is _GEMV_ANS):
        return None
    step = _lib.eager()
    return None if step is None else step.linear(input, getattr(weight, '_buffers', None), bias, huffman)


def _eager_weight(weight: HuffmanWeight, huffman: bool) -> Optional[Tensor]:
    """The same for a weight that is decoded, by ``huffman_decode`` / ``ans_decode``."""
    if torch.compiler.is_compiling() or not (
            huffman_decode is _ops.huffman_decode if huffman else ans_decode is _ops.ans_decode):
        return None
    step = _lib.eager()
    return None if step is None else step.weight(getattr(weight, '_buffers', None), huffman)


def linear_huffman(input: Tensor, weight: HuffmanWeight, bias: Optional[Tensor] = None) -> Tensor:
    """``F.linear`` with a :class:`HuffmanWeight`: fused kernels up to 32 rows and, where they are faster,
    up to 640, else decode + dense GEMM (reference ``functional.py:390-411``)."""
    if (output := _eager(input, weight, bias, True)) is not None:
        return output

    def fused(x):
        b = weight._buffers          # without nn.Module's attribute lookups, a microsecond of the call
        try:
            args = (b['rem'], b['exp'], x, b['offsets'], b['LUT1'], b['LUT2'], b['LUT3'], b['LUT4'], b['code_lengths'])
        except KeyError:             # a parametrization takes a buffer out and puts a property in its place
            w = weight
            args = (w.rem, w.exp, x, w.offsets, w.LUT1, w.LUT2, w.LUT3, w.LUT4, w.code_lengths)
        return mv_huffman(*args)
    return _linear_compressed(input, weight, bias, fused)


def linear_ans(input: Tensor, weight: ANSWeight, bias: Optional[Tensor] = None) -> Tensor:
    """rANS counterpart of :func:`linear_huffman` (reference ``functional.py:447-466``)."""
    if (output := _eager(input, weight, bias, False)) is not None:
        return output

    def fused(x):
        b = weight._buffers          # as above
        try:
            args = (b['rem'], b['exp'], x, b['offsets'], b['LUT'])
        except KeyError:
            args = (weight.rem, weight.exp, x, weight.offsets, weight.LUT)
        return mv_ans(*args)
    return _linear_compressed(input, weight, bias, fused)
