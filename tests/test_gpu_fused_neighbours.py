"""RMSNorm and SiLU*mul in front of the grouped GEMV, and the residual behind it (needs a GPU):
fused == this package's unfused kernels + plain GEMV, bit for bit; both close to PyTorch's ops."""
import pytest
import torch
import torch.nn.functional as F

from helpers import gaussian_weight, student_t_weight

pytestmark = pytest.mark.gpu

RTOL, ATOL = 1e-2, 1e-3


def _cls(algo):
    from bf16_huffman_infer_amd.functional import ANSWeight, HuffmanWeight, NibbleWeight
    return {"huffman": HuffmanWeight, "ans": ANSWeight, "nibble": NibbleWeight}[algo]


def _bits(t):
    return t.contiguous().view(torch.int16)


@pytest.mark.parametrize("rows", [1, 2, 3, 4, 7])
def test_rms_norm_kernel_against_torch(cuda, rows):
    from bf16_huffman_infer_amd import ops
    g = torch.Generator().manual_seed(rows)
    x = (torch.randn(rows, 4096, generator=g) * 3).bfloat16().cuda()
    gamma = (1 + 0.1 * torch.randn(4096, generator=g)).bfloat16().cuda()
    got = ops.rms_norm(x, gamma, 1e-6)
    want = (x.float() * torch.rsqrt(x.float().pow(2).mean(-1, keepdim=True) + 1e-6) * gamma.float())
    # one BF16 rounding of the fp32 result: half a step of relative error
    torch.testing.assert_close(got.float(), want, rtol=2.0 ** -8, atol=1e-6)
    torch.testing.assert_close(got.float(), F.rms_norm(x, (4096,), gamma, 1e-6).float(), rtol=2.0 ** -6, atol=1e-5)


def test_silu_mul_kernel_against_torch(cuda):
    from bf16_huffman_infer_amd import ops
    g = torch.Generator().manual_seed(3)
    gate = (torch.randn(3, 12288, generator=g) * 2).bfloat16().cuda()
    up = torch.randn(3, 12288, generator=g).bfloat16().cuda()
    got = ops.silu_mul(gate, up)
    want = F.silu(gate) * up
    same = (_bits(got) == _bits(want)).float().mean().item()
    assert same > 0.999                                    # exp is evaluated differently: a rare last-place flip of the BF16 silu
    torch.testing.assert_close(got.float(), want.float(), rtol=2.0 ** -6, atol=1e-6)


@pytest.mark.parametrize("rows", [1, 5])
@pytest.mark.parametrize("K", [2, 126, 2046, 2048, 2050, 4096, 4098, 5120, 8192, 8194, 18944, 20480, 20482, 24576])
def test_rms_norm_kernel_row_lengths(cuda, rows, K):
    """Rows that a block holds in registers (up to 2048, 4096, 8192 and 20480 elements) and longer ones, which it reads
    twice; each row on its own scale, and nothing written past the last."""
    from bf16_huffman_infer_amd import _lib
    g = torch.Generator().manual_seed(K + rows)
    x = (torch.randn(rows, K, generator=g) * torch.arange(1, rows + 1)[:, None]).bfloat16().cuda()
    gamma = (1 + 0.1 * torch.randn(K, generator=g)).bfloat16().cuda()
    held = torch.full((rows * K + 512,), 7.0, dtype=torch.bfloat16, device="cuda")
    got = held[256:-256].view(rows, K)
    _lib.check(_lib.load().bhi_rms_norm(x.data_ptr(), gamma.data_ptr(), got.data_ptr(), rows, K, 1e-6,
                                        torch.cuda.current_stream().cuda_stream), "rms_norm")
    want = x.double() * torch.rsqrt(x.double().pow(2).mean(-1, keepdim=True) + 1e-6) * gamma.double()
    # one rounding to BF16's eight significant bits (half a step of 2^-7 at 1: 2^-8), and fp32 sums of up to 24576
    # squares, each thread's at most 96 in a row, 14 more to join them, a handful of roundings after: 128 * 2^-24
    assert bool(((got.double() - want).abs() <= (2.0 ** -8 + 2.0 ** -17) * want.abs()).all())
    assert bool((held[:256] == 7.0).all()) and bool((held[-256:] == 7.0).all())


def _fused(mods, x, mode, aux, residuals=None, eps=0.0):
    """The launch with the transform inside, whatever :func:`fuses_input` would choose."""
    from bf16_huffman_infer_amd import ops
    rows = x.shape[0]
    ys = [torch.full((rows, m.rem.shape[1]), float("nan"), dtype=torch.bfloat16, device="cuda") for m in mods]
    ops.gemv_bf16_grouped(mods, x.view(rows, *mods[0].rem.shape[::2]), ys, None, residuals, mode, aux, eps)
    return ys


@pytest.mark.parametrize("algo", ["huffman", "ans"])
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
@pytest.mark.parametrize("K", [1024, 4096, 5120, 12288, 22528])
def test_transforms_inside_the_launch(cuda, algo, rows, K):
    """Both transforms inside the GEMV at every row count, on short and long tasks and rows of every kind that
    the RMSNorm kernel tells apart: the bits of the kernels of their own."""
    from bf16_huffman_infer_amd import ops
    from bf16_huffman_infer_amd.functional import linear_grouped
    mods = [_cls(algo).compress(gaussian_weight(M, K, seed=M + K)).cuda() for M in (256, 128)]
    g = torch.Generator().manual_seed(rows + K)
    x = (torch.randn(rows, K, generator=g) * 2).bfloat16().cuda()
    gamma = (1 + 0.1 * torch.randn(K, generator=g)).bfloat16().cuda()
    gate = (torch.randn(rows, K, generator=g) * 1.5).bfloat16().cuda()
    res = [torch.randn(rows, m.rem.shape[1], generator=g).bfloat16().cuda() for m in mods]
    for inside, own in ((_fused(mods, x, ops.X_RMS, gamma, eps=1e-6), linear_grouped(ops.rms_norm(x, gamma, 1e-6), mods)),
                        (_fused(mods, x, ops.X_SILU_MUL, gate, res),
                         linear_grouped(ops.silu_mul(gate, x), mods, residuals=res))):
        for a, b in zip(inside, own):
            assert torch.equal(_bits(a), _bits(b))


@pytest.mark.parametrize("algo", ["huffman", "ans"])
@pytest.mark.parametrize("rows", [1, 2, 3, 4])
def test_norm_in_front_of_grouped_gemv(cuda, algo, rows):
    """q/k/v of a decoder layer: RMSNorm(x) * gamma, then three products -- one launch."""
    from bf16_huffman_infer_amd import ops
    from bf16_huffman_infer_amd.functional import linear_grouped
    K, Ms = 2048, (512, 128, 128)
    ws = [(gaussian_weight if i % 2 == 0 else student_t_weight)(M, K, seed=40 + i) for i, M in enumerate(Ms)]
    mods = [_cls(algo).compress(w).cuda() for w in ws]
    g = torch.Generator().manual_seed(rows)
    x = (torch.randn(rows, K, generator=g) * 2).bfloat16().cuda()
    gamma = (1 + 0.1 * torch.randn(K, generator=g)).bfloat16().cuda()
    fused = _fused(mods, x, ops.X_RMS, gamma, eps=1e-6)
    for a, b in zip(fused, linear_grouped(x, mods, input_norm=(gamma, 1e-6))):
        assert torch.equal(_bits(a), _bits(b))                  # wherever the rule puts the norm
    h = ops.rms_norm(x, gamma, 1e-6)
    unfused = linear_grouped(h, mods)
    for w, a, b in zip(ws, fused, unfused):
        assert torch.equal(_bits(a), _bits(b))
        ref = h.float() @ w.cuda().float().T
        torch.testing.assert_close(a.float(), ref, rtol=RTOL, atol=ATOL)


@pytest.mark.parametrize("algo", ["huffman", "ans"])
@pytest.mark.parametrize("rows", [1, 4])
@pytest.mark.parametrize("M,K", [(512, 3072), (4096, 12288)])
def test_gate_product_in_front_and_residual_behind(cuda, algo, rows, M, K):
    """down_proj of a decoder layer: x + W (silu(gate) * up) -- one launch."""
    from bf16_huffman_infer_amd import ops
    from bf16_huffman_infer_amd.functional import linear_grouped
    w = gaussian_weight(M, K, seed=M)
    mod = _cls(algo).compress(w).cuda()
    g = torch.Generator().manual_seed(rows + M)
    gate = (torch.randn(rows, K, generator=g) * 1.5).bfloat16().cuda()
    up = torch.randn(rows, K, generator=g).bfloat16().cuda()
    res = torch.randn(rows, M, generator=g).bfloat16().cuda()
    fused, = _fused([mod], up, ops.X_SILU_MUL, gate, [res])
    chosen, = linear_grouped(up, [mod], input_gate=gate, residuals=[res])
    h = ops.silu_mul(gate, up)
    plain, = linear_grouped(h, [mod])
    assert torch.equal(_bits(fused), _bits(chosen))             # wherever the rule puts the product
    assert torch.equal(_bits(fused), _bits(plain + res))        # a separate BF16 addition gives the same bits
    prod = h.float() @ w.cuda().float().T
    bound = ATOL + RTOL * (prod + res.float()).abs() + 2.0 ** -8 * prod.abs()
    assert ((fused.float() - (prod + res.float())).abs() <= bound).all()


@pytest.mark.parametrize("algo", ["huffman", "nibble"])
def test_more_rows_or_other_codecs_run_the_unfused_kernels(cuda, algo):
    from bf16_huffman_infer_amd import ops
    from bf16_huffman_infer_amd.functional import linear_grouped
    K, M, rows = 1024, 256, 6
    mod = _cls(algo).compress(gaussian_weight(M, K, seed=5)).cuda()
    g = torch.Generator().manual_seed(1)
    x = torch.randn(rows, K, generator=g).bfloat16().cuda()
    gamma = (1 + 0.1 * torch.randn(K, generator=g)).bfloat16().cuda()
    a, = linear_grouped(x, [mod], input_norm=(gamma, 1e-5))
    b, = linear_grouped(ops.rms_norm(x, gamma, 1e-5), [mod])
    assert torch.equal(_bits(a), _bits(b))
    gate = torch.randn(rows, K, generator=g).bfloat16().cuda()
    a, = linear_grouped(x, [mod], input_gate=gate)
    b, = linear_grouped(ops.silu_mul(gate, x), [mod])
    assert torch.equal(_bits(a), _bits(b))


@pytest.mark.parametrize("recorder", ["torch", "package"])
@pytest.mark.parametrize("rows,Ms,K", [(2, (4608,), 3584), (4, (1024, 512), 8192)])
def test_eager_and_recorded_calls_give_the_same_bits(cuda, recorder, rows, Ms, K):
    """Eager calls keep the transform inside where a graph gives it a launch of its own."""
    from bf16_huffman_infer_amd.cudagraph_utils import GraphedCallable
    from bf16_huffman_infer_amd.functional import fuses_input, linear_grouped
    mods = [_cls("huffman").compress(gaussian_weight(M, K, seed=M)).cuda() for M in Ms]
    g = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, K, generator=g).bfloat16().cuda()
    gate = torch.randn(rows, K, generator=g).bfloat16().cuda()
    gamma = (1 + 0.1 * torch.randn(K, generator=g)).bfloat16().cuda()
    n = sum(Ms) * K
    for norm in (True, False):
        assert fuses_input(rows, n, norm, True, False) and not fuses_input(rows, n, norm, True, True)
    outs = [torch.empty(rows, 2 * sum(Ms), dtype=torch.bfloat16, device="cuda") for _ in range(2)]

    def step(out):
        out.copy_(torch.cat(linear_grouped(x, mods, input_norm=(gamma, 1e-6)) + linear_grouped(x, mods, input_gate=gate), -1))
        return out
    step(outs[0])
    if recorder == "package":
        graph = GraphedCallable(lambda: step(outs[1]), ())
    else:
        step(outs[1])
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            step(outs[1])
    for _ in range(3):
        outs[1].zero_()
        graph.replay()
        assert torch.equal(_bits(outs[0]), _bits(outs[1]))
