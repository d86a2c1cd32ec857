"""Eager calls of the GEMV in one native step (needs a GPU): the bits of the custom ops, and the calls it leaves to them."""
import pytest
import torch
import torch.nn.functional as F

from helpers import gaussian_weight

pytestmark = pytest.mark.gpu


def _layer(algo, M=384, K=1024, bias=False):
    from bf16_huffman_infer_amd.functional import ANSWeight, CompressedLinear, HuffmanWeight
    weight = {"huffman": HuffmanWeight, "ans": ANSWeight}[algo].compress_split_n(gaussian_weight(M, K, seed=M), n=2)
    b = torch.nn.Parameter((0.1 * torch.randn(M)).bfloat16(), requires_grad=False) if bias else None
    return CompressedLinear(weight, b).cuda()


def _step(lin, x):
    from bf16_huffman_infer_amd.functional import _eager
    return _eager(x, lin.weight, lin.bias, hasattr(lin.weight, "LUT1"))


def _through_ops(lin, x):
    from bf16_huffman_infer_amd.functional import mv_ans, mv_huffman
    y = (mv_huffman if hasattr(lin.weight, "LUT1") else mv_ans)(X=x.reshape(-1, x.shape[-1]), **{
        {"rem": "A_rem", "exp": "A_exp"}.get(k, k): v for k, v in lin.weight.kwargs().items()})
    if lin.bias is not None:
        y += lin.bias.detach()
    return y.view(*x.shape[:-1], -1)


@pytest.mark.parametrize("algo", ["huffman", "ans"])
@pytest.mark.parametrize("bias", [False, True])
def test_same_bits_as_the_custom_ops(cuda, algo, bias):
    lin = _layer(algo, bias=bias)
    gen = torch.Generator().manual_seed(1)
    with torch.no_grad():
        for shape in ((1, 1024), (2, 1024), (7, 1024), (8, 1024), (1, 1, 1024), (2, 3, 1024), (1, 2, 1, 1024)):
            x = torch.randn(shape, generator=gen).bfloat16().cuda()
            want = _through_ops(lin, x)                   # (and with it the library's first use of the device)
            y = _step(lin, x)
            assert y is not None and y.shape == want.shape and y.stride() == want.stride() and torch.equal(y, want)
            assert torch.equal(lin(x), want)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            y = lin(x)
        side.synchronize()
        assert torch.equal(y, want)


def test_calls_that_the_custom_ops_keep(cuda):
    lin = _layer("huffman")
    x = torch.randn(2, 1024).bfloat16().cuda()
    want = _through_ops(lin, x)
    assert _step(lin, x) is not None
    wants_grad = x.clone().requires_grad_()
    assert _step(lin, wants_grad) is None
    with torch.no_grad():
        assert _step(lin, wants_grad) is not None
    assert _step(lin, x.T.contiguous().T) is None and torch.equal(lin(x.T.contiguous().T), want)
    for other in (x.float(), x.cpu(), x[0], x[:, :512].contiguous(), x[:0], torch.randn(9, 1024).bfloat16().cuda()):
        assert _step(lin, other) is None

    class Sub(torch.Tensor):
        pass
    assert _step(lin, x.as_subclass(Sub)) is None
    seen = []

    class Mode(torch.utils._python_dispatch.TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            seen.append(str(func))
            return func(*args, **(kwargs or {}))
    with Mode():
        assert _step(lin, x) is None and torch.equal(lin(x), want)
    assert any("gemv_bf16_huffman" in name for name in seen)
    with torch.profiler.profile() as prof:
        lin(x)
    assert any("gemv_bf16_huffman" in e.name for e in prof.events())
    taken = []
    torch.func.vmap(lambda v: (taken.append(_step(lin, x)), v)[1])(x)
    assert taken == [None]
    with torch.device("cuda"):                            # a function mode
        assert _step(lin, x) is None
    del lin.weight._buffers["offsets"]
    assert _step(lin, x) is None


def test_recorded_and_replayed(cuda):
    lin = _layer("ans", bias=True)
    x = torch.randn(3, 1024).bfloat16().cuda()
    with torch.no_grad():
        want = _through_ops(lin, x)
        lin(x)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = lin(x)
        for _ in range(3):
            y.zero_()
            graph.replay()
            assert torch.equal(y, want) and torch.equal(lin(x), want)


@pytest.mark.parametrize("algo", ["huffman", "ans"])
def test_weight_back_in_one_step(cuda, algo):
    from bf16_huffman_infer_amd.functional import _eager_weight
    weight, huffman = _layer(algo).weight, algo == "huffman"
    weight.get_weight()                                    # the library's first use of the device
    want = gaussian_weight(384, 1024, seed=384)
    y = _eager_weight(weight, huffman)
    assert torch.equal(y.cpu().view(torch.int16), want.view(torch.int16)) and not y.requires_grad
    with torch.device("cuda"):                             # a function mode: the custom op
        assert _eager_weight(weight, huffman) is None and torch.equal(weight.get_weight(), y)
    taken = []
    torch.func.vmap(lambda v: (taken.append(_eager_weight(weight, huffman)), v)[1])(y)
    assert taken == [None]
    assert _eager_weight(_layer(algo).weight.cpu(), huffman) is None
    del weight._buffers["exp"]
    assert _eager_weight(weight, huffman) is None


def test_short_of_memory_raises_torchs_own_error(cuda):
    lin = _layer("huffman", M=131072, K=256)               # 2 MB of output, 67 MB of weight
    x = torch.randn(8, 256).bfloat16().cuda()
    with torch.no_grad():
        want = lin(x)
        torch.cuda.empty_cache()
        limit = torch.cuda.memory_reserved() + (1 << 20)
        torch.cuda.set_per_process_memory_fraction(limit / torch.cuda.get_device_properties(0).total_memory)
        held = []
        try:
            with pytest.raises(torch.OutOfMemoryError):    # what the allocator still holds
                for _ in range(64):
                    held.append(torch.empty(1 << 21, dtype=torch.uint8, device="cuda"))
            for call in (lambda: lin(x), lin.weight.get_weight):
                with pytest.raises(torch.OutOfMemoryError):
                    call()
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        held.clear()
        assert torch.equal(lin(x), want)


@pytest.mark.parametrize("algo", ["huffman", "ans"])
def test_launches_without_the_interpreter_lock(cuda, algo):
    """In the place of the library's entry points stands the interpreter's own question whether this thread holds the
    lock: 0, which the step takes for a launch, where it does not."""
    import ctypes
    from bf16_huffman_infer_amd import _lib
    lin, huffman = _layer(algo), algo == "huffman"
    x = torch.randn(1, 1024).bfloat16().cuda()
    with torch.no_grad():
        want = lin(x)
        asked = ctypes.cast(ctypes.pythonapi.PyGILState_Check, ctypes.c_void_p).value
        lib, step = _lib.load(), _lib.eager()
        prefers = ctypes.cast(lib.bhi_prefers_matrix_cores, ctypes.c_void_p).value
        step.bind(asked, asked, asked, asked, prefers)
        try:
            taken = [step.linear(x, lin.weight._buffers, None, huffman), step.weight(lin.weight._buffers, huffman)]
        finally:
            step.bind(*(ctypes.cast(f, ctypes.c_void_p).value for f in (
                lib.bhi_gemv_bf16_huffman_grouped, lib.bhi_gemv_bf16_ans_grouped, lib.bhi_huffman_decode, lib.bhi_ans_decode)), prefers)
        assert taken[0] is not None and taken[1] is not None
        assert torch.equal(lin(x), want)
