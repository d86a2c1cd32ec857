"""The wide product (17 to 640 rows of X, needs a GPU) against 64-bit sums of the same BF16 operands."""
import pytest
import torch

from helpers import gaussian_weight, student_t_weight
from test_gpu_tiled import _check, _cls, escaping_weight

pytestmark = pytest.mark.gpu

# (M, K, splits): one task of one step; two and four slices; tasks of one step, three slices; odd counts of
# steps; more blocks than units; one slice out of five tasks per row group and a last task that is shorter
SHAPES = [(128, 128, 1), (640, 1024, 1), (128, 16384, 1), (128, 384, 3), (256, 1664, 1), (16640, 128, 1), (3328, 6400, 5)]


@pytest.mark.parametrize("algo", ["huffman", "ans"])
@pytest.mark.parametrize("make", [gaussian_weight, student_t_weight, escaping_weight])
@pytest.mark.parametrize("M,K,n", SHAPES)
def test_wide_product(cuda, algo, make, M, K, n):
    from bf16_huffman_infer_amd import ops
    w = make(M, K, seed=M + K)
    mod = _cls(algo).compress_split_n(w, n=n).cuda()
    # both ends of every number of tiles per wavefront, and of both splits of the weight rows
    for rows in (17, 32, 33, 64, 65, 128, 129, 144, 145, 192, 193, 256, 257, 384, 385, 512, 513, 639, 640):
        x = torch.randn(rows, K, generator=torch.Generator().manual_seed(rows)).bfloat16().cuda()
        held = torch.full((rows * M + 8192,), 7.0, dtype=torch.bfloat16, device="cuda")      # Y in the middle
        y = held[4096:-4096].view(rows, M)
        y.fill_(float("nan"))
        bias = (0.1 * torch.randn(M, device="cuda")).bfloat16() if rows % 2 else None
        for _ in range(2):                     # the second launch finds the first one's counters
            ops.wide_bf16(mod, x.view(rows, n, K // n), y, bias)
            _check(y, x, w, bias)
        assert bool((held[:4096] == 7.0).all()) and bool((held[-4096:] == 7.0).all())


def test_a_row_of_x_stays_its_own(cuda):
    """Infinities and NaN in one row of X (the last, which fills the last tile as well) reach no other row."""
    from bf16_huffman_infer_amd import ops
    w = gaussian_weight(256, 512, seed=4)
    mod = _cls("huffman").compress(w).cuda()
    x = torch.randn(150, 512, generator=torch.Generator().manual_seed(5)).bfloat16().cuda()
    x[149, 3], x[149, 200] = float("inf"), float("nan")
    y = torch.empty(150, 256, dtype=torch.bfloat16, device="cuda")
    ops.wide_bf16(mod, x.view(150, 1, 512), y)
    _check(y[:149], x[:149], w)
    assert bool(y[149].isnan().all())


@pytest.mark.parametrize("rows", [40, 200, 600])
def test_linear_takes_the_wide_product(cuda, rows):
    """Through ``F.linear``: contiguous, strided and misaligned inputs, and inputs that want gradients."""
    from bf16_huffman_infer_amd.functional import CompressedLinear, _wide
    M, K = 8192, 4096
    w = gaussian_weight(M, K, seed=rows)
    bias = torch.nn.Parameter((0.1 * torch.randn(M)).bfloat16(), requires_grad=False)
    lin = CompressedLinear(_cls("huffman").compress(w), bias).cuda()
    x = torch.randn(rows, K, generator=torch.Generator().manual_seed(1)).bfloat16().cuda()
    assert _wide(x, lin.weight, lin.bias)
    y = lin(x)
    _check(y, x, w, lin.bias)
    odd = torch.empty(rows * K + 1, dtype=torch.bfloat16, device="cuda")[1:].view(rows, K)
    odd.copy_(x)
    assert torch.equal(lin(odd), y) and torch.equal(lin(x.T.contiguous().T), y)
    assert torch.equal(lin(x.view(2, rows // 2, K)), y.view(2, rows // 2, M))
    g = x.clone().requires_grad_()
    assert not _wide(g, lin.weight, lin.bias)
    lin(g).float().sum().backward()
    assert g.grad is not None


@pytest.mark.parametrize("algo", ["huffman", "ans"])
def test_wide_product_recorded_and_replayed(cuda, algo):
    M, K = 4096, 4096                          # cut along K: counters and partial sums in a workspace
    mod = _cls(algo).compress(gaussian_weight(M, K, seed=3)).cuda()
    x = torch.randn(150, K, generator=torch.Generator().manual_seed(2)).bfloat16().cuda()
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


def test_wide_product_rejections(cuda):
    from bf16_huffman_infer_amd import _lib, ops
    lib = _lib.load()
    mod = _cls("huffman").compress(gaussian_weight(1024, 1024, seed=1)).cuda()
    for rows in (16, 641):
        x = torch.zeros(rows, 1, 1024, dtype=torch.bfloat16, device="cuda")
        with pytest.raises(RuntimeError, match="17 to 640"):
            ops.wide_bf16(mod, x, torch.empty(rows, 1024, dtype=torch.bfloat16, device="cuda"))
    x = torch.zeros(41, 1024, dtype=torch.bfloat16, device="cuda")
    y = torch.empty(41, 1024, dtype=torch.bfloat16, device="cuda")
    member = (_lib.GemvMember * 1)()
    ops._fill_member(member[0], mod, y[:40], None, mod.rem)
    need = lib.bhi_wide_workspace_bytes(1, 1024, 1024, 40)
    ws = torch.zeros(need, dtype=torch.uint8, device="cuda")
    for x_ptr, ws_ptr, nbytes, text in ((x.data_ptr(), None, 0, b"workspace"), (x.data_ptr(), ws.data_ptr(), need - 1, b"workspace"),
                                        (x.data_ptr() + 2, ws.data_ptr(), need, b"aligned")):
        assert lib.bhi_wide_bf16_huffman(member, x_ptr, 1, 1024, 40, ws_ptr, nbytes, None) != 0
        assert text in lib.bhi_last_error_string()


def test_two_threads_on_one_stream_keep_their_own_x(cuda):
    """Both use the workspace of the stream that they share; every result is compared."""
    import threading
    from bf16_huffman_infer_amd import ops
    mods = [_cls(algo).compress(gaussian_weight(512, 1024, seed=i)).cuda() for i, algo in enumerate(("huffman", "ans"))]
    g = torch.Generator().manual_seed(9)
    xs = [[torch.randn(rows, 1, 1024, generator=g).bfloat16().cuda() for rows in sizes] for sizes in ((40, 150, 40), (40, 600, 65))]

    def product(mod, x):
        y = torch.empty(x.shape[0], 512, dtype=torch.bfloat16, device="cuda")
        ops.wide_bf16(mod, x, y)
        return y
    want = [[product(mod, x) for x in mine] for mod, mine in zip(mods, xs)]
    got, stream, start = [[], []], torch.cuda.current_stream(), threading.Barrier(2)

    def calls(i):
        with torch.cuda.stream(stream):
            start.wait()
            for _ in range(50):
                got[i].append([product(mods[i], x) for x in xs[i]])
    threads = [threading.Thread(target=calls, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(2):
        assert len(got[i]) == 50
        assert all(torch.equal(y, w) for ys in got[i] for y, w in zip(ys, want[i]))


@pytest.mark.parametrize("algo", ["huffman", "ans"])
@pytest.mark.parametrize("M", [4, 32, 64, 96])
def test_heights_that_fused_calls_refuse_are_decoded(cuda, algo, M):
    """Weights that the package's conversion does not make, but the library takes: the first rows of one that it makes."""
    from bf16_huffman_infer_amd.functional import CompressedLinear, check_layout
    whole = gaussian_weight(128, 256, seed=M)
    kwargs = {n: t.cpu() for n, t in _cls(algo).compress_split_n(whole, n=1).kwargs().items()}
    assert not kwargs["offsets"][0].view(-1, 4)[:, 1:].any()                    # one task per row group, in their order
    words = int(kwargs["offsets"][0, M])
    kwargs.update(rem=kwargs["rem"][:, :M].contiguous(), offsets=kwargs["offsets"][:, :M].contiguous(),
                  exp=torch.cat((kwargs["exp"][:words], torch.zeros(2048, dtype=torch.int32))))
    weight = _cls(algo)(**kwargs)
    check_layout(weight)
    lin = CompressedLinear(weight, None).cuda()
    assert torch.equal(lin.weight.get_weight().cpu(), whole[:M])
    for rows in (129, 200, 640):
        x = torch.randn(rows, 256, generator=torch.Generator().manual_seed(rows)).bfloat16().cuda()
        _check(lin(x), x, whole[:M])
