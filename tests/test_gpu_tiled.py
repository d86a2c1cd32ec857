"""The tiled product (17 to 128 rows of X, needs a GPU) against 64-bit sums of the same BF16 operands."""
import pytest
import torch

from helpers import gaussian_weight, random_bits_weight, student_t_weight

pytestmark = pytest.mark.gpu


def _cls(algo):
    from bf16_huffman_infer_amd.functional import ANSWeight, HuffmanWeight
    return {"huffman": HuffmanWeight, "ans": ANSWeight}[algo]


def escaping_weight(M, K, seed=0):
    """Exponents uniform over 64 values: more pairs than get codes, most steps escape on some lane, and the
    streams are long (a lane reads more than a row per step)."""
    bits = random_bits_weight(M, K, seed).view(torch.int16).to(torch.int32) & 0xFFFF
    exp = 64 + ((bits >> 7) & 0x3F)
    return ((bits & 0x807F) | (exp << 7)).to(torch.int16).view(torch.bfloat16)


def _check(y, x, w, bias=None):
    """One BF16 rounding of the result (2^-9 relative; with a bias and up to 32 rows, one of the product
    as well), and fp32 sums in any order: each of K additions is off by 2^-24 of a partial sum."""
    x, w = x.cuda().double(), w.cuda().double()
    ref, mag = x @ w.T, x.abs() @ w.abs().T
    bound = (x.shape[1] + 1) * 2.0 ** -24 * mag
    if bias is not None:
        if x.shape[0] <= 32:
            bound = bound + 2.0 ** -8 * ref.abs()
        ref = ref + bias.double()
    bound = bound + 2.0 ** -8 * ref.abs()
    assert bool(((y.double() - ref).abs() <= bound).all())


# (M, K, splits): four wavefronts and two K slices; four wavefronts (sixteen ring rows from 65 rows of X
# on), whole; six wavefronts and a last block that is not full; from 65 rows on eight wavefronts; six or
# four wavefronts, four slices, tasks of 32 steps; three splits, tasks of one step, odd counts
SHAPES = [(640, 1024, 1), (16384, 256, 1), (16640, 128, 1), (24704, 128, 1), (128, 16384, 1), (128, 384, 3), (256, 1664, 1)]


@pytest.mark.parametrize("algo", ["huffman", "ans"])
@pytest.mark.parametrize("make", [gaussian_weight, student_t_weight, escaping_weight])
@pytest.mark.parametrize("M,K,n", SHAPES)
def test_tiled_product(cuda, algo, make, M, K, n):
    from bf16_huffman_infer_amd import ops
    w = make(M, K, seed=M + K)
    mod = _cls(algo).compress_split_n(w, n=n).cuda()
    for rows in (17, 32, 33, 48, 49, 64, 65, 80, 81, 96, 97, 112, 113, 128):
        x = torch.randn(rows, K, generator=torch.Generator().manual_seed(rows)).bfloat16().cuda()
        held = torch.full((rows * M + 8192,), 7.0, dtype=torch.bfloat16, device="cuda")      # Y in the middle
        y = held[4096:-4096].view(rows, M)
        y.fill_(float("nan"))
        bias = (0.1 * torch.randn(M, device="cuda")).bfloat16() if rows % 2 else None
        for _ in range(2):                     # the second launch finds the first one's counters
            ops.tile_bf16(mod, x.view(rows, n, K // n), y, bias)
            _check(y, x, w, bias)
        assert bool((held[:4096] == 7.0).all()) and bool((held[-4096:] == 7.0).all())


@pytest.mark.parametrize("rows", [24, 40, 100])
def test_linear_takes_the_tiled_product(cuda, rows):
    """Through ``F.linear``: contiguous, strided and misaligned inputs, and inputs that want gradients."""
    from bf16_huffman_infer_amd.functional import CompressedLinear, _tiled
    M, K = 8192, 2048
    w = gaussian_weight(M, K, seed=rows)
    lin = CompressedLinear(_cls("huffman").compress(w), None).cuda()
    x = torch.randn(rows, K, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    assert _tiled(x, lin.weight, None)
    _check(lin(x), x, w)
    odd = torch.empty(rows * K + 1, dtype=torch.bfloat16, device="cuda")[1:].view(rows, K)
    odd.copy_(x)
    assert torch.equal(lin(odd), lin(x))
    if rows > 32:
        assert torch.equal(lin(x.T.contiguous().T), lin(x))
        g = x.clone().requires_grad_()
        assert not _tiled(g, lin.weight, None)
        lin(g).float().sum().backward()
        want = w.cuda().double().sum(0)
        assert bool(((g.grad.double() - want).abs() <= 2.0 ** -7 * want.abs() + M * 2.0 ** -24 * w.cuda().double().abs().sum(0)).all())


@pytest.mark.parametrize("algo", ["huffman", "ans"])
def test_tiled_product_recorded_and_replayed(cuda, algo):
    M, K = 1024, 4096                          # cut along K: counters and partial sums in a workspace
    mod = _cls(algo).compress(gaussian_weight(M, K, seed=3)).cuda()
    x = torch.randn(48, K, generator=torch.Generator().manual_seed(2)).bfloat16().cuda()
    eager = torch.nn.functional.linear(x, mod)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = torch.nn.functional.linear(x, mod)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        assert torch.equal(torch.nn.functional.linear(x, mod), eager)


def test_tiled_product_rejections(cuda):
    from bf16_huffman_infer_amd import _lib, ops
    mod = _cls("huffman").compress(gaussian_weight(1024, 1024, seed=1)).cuda()
    for rows in (16, 129):
        x = torch.zeros(rows, 1, 1024, dtype=torch.bfloat16, device="cuda")
        with pytest.raises(RuntimeError, match="17 to 128"):
            ops.tile_bf16(mod, x, torch.empty(rows, 1024, dtype=torch.bfloat16, device="cuda"))
    x = torch.zeros(40, 1024, dtype=torch.bfloat16, device="cuda")
    y = torch.empty(40, 1024, dtype=torch.bfloat16, device="cuda")
    member = (_lib.GemvMember * 1)()
    ops._fill_member(member[0], mod, y, None, mod.rem)
    rc = _lib.load().bhi_tile_bf16_huffman(member, x.data_ptr(), 1, 1024, 40, None, 0, None)
    assert rc != 0 and b"workspace" in _lib.load().bhi_last_error_string()


@pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning")
def test_traced_call_records_the_product(cuda):
    """``torch.jit.trace`` at a row count of the tiled product: the module it returns computes."""
    from bf16_huffman_infer_amd.functional import CompressedLinear
    M, K, rows = 1024, 1024, 40
    w = gaussian_weight(M, K, seed=8)
    lin = CompressedLinear(_cls("huffman").compress(w), None).cuda().eval()
    a, b = (torch.randn(rows, K, generator=torch.Generator().manual_seed(i)).bfloat16().cuda() for i in range(2))
    with torch.no_grad():
        traced = torch.jit.trace(lambda x: torch.nn.functional.linear(x, lin.weight), (a,), check_trace=False)
        assert "linear" in str(traced.graph)
        _check(traced(b), b, w)
