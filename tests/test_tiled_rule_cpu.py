"""Where the tiled product may take the place of decoding and ``F.linear``, and the workspace it asks for."""
import pytest
import torch
import torch.autograd.forward_ad as forward_ad


def test_only_where_nothing_but_the_value_is_asked_for():
    from bf16_huffman_infer_amd.functional import _fuses_above_32_rows as fuses
    x, bias = torch.zeros(40, 128), torch.zeros(64)
    assert fuses(x, None) and fuses(x, bias) and fuses(torch.nn.Parameter(x, requires_grad=False), bias)
    wants = x.clone().requires_grad_()
    assert not fuses(wants, None) and not fuses(x, bias.clone().requires_grad_())
    with torch.no_grad():
        assert fuses(wants, None)
    with forward_ad.dual_level():
        assert not fuses(x, None)
    seen = []
    torch.func.vmap(lambda v: (seen.append(fuses(x, None)), v)[1])(x)
    assert seen == [False]
    with torch.utils._python_dispatch.TorchDispatchMode():
        assert not fuses(x, None)

    class Sub(torch.Tensor):
        pass
    assert not fuses(x.as_subclass(Sub), None)


def test_workspace_follows_the_slice_choice():
    """Counters, then whole blocks of sixteen-row tiles per slice; nothing where K is not cut; never more
    row blocks than there are counters."""
    from bf16_huffman_infer_amd import _lib
    lib = _lib.load()
    for split_k, M, Ks in [(1, 128, 128), (1, 1024, 4096), (3, 4096, 4096), (4, 3584, 4736), (1, 18944, 3584), (1, 12288, 4096),
                           (2, 65536, 2048), (1, 132, 512)]:
        per_group = split_k * lib.bhi_chunks_per_group(M, Ks, split_k)
        for rows in (17, 32, 33, 64, 65, 80, 81, 96, 97, 112, 128):
            need = lib.bhi_tile_workspace_bytes(split_k, M, Ks, rows)
            assert need >= 0
            if need:
                tiles = (rows + 15) // 16
                choices = [(nw, d) for nw in (4, 6, 8) for d in range(2, 9) if per_group % d == 0
                           and -(-M // (16 * nw)) <= 256 and 1024 + -(-M // (16 * nw)) * 16 * nw * tiles * 64 * d == need]
                assert choices, (split_k, M, Ks, rows, need)
        assert lib.bhi_tile_workspace_bytes(split_k, M, Ks, 16) < 0 and lib.bhi_tile_workspace_bytes(split_k, M, Ks, 129) < 0


def test_not_while_the_call_is_traced(monkeypatch):
    """A tracer records what goes through the dispatcher: of the tiled product that is the empty output alone."""
    from bf16_huffman_infer_amd.functional import _fuses_above_32_rows as fuses
    x, seen = torch.zeros(40, 8), []

    def step(v):
        seen.append((torch.jit.is_tracing(), fuses(v, None)))
        return v + 1
    torch.jit.trace(step, (x,), check_trace=False)
    assert seen == [(True, False)]
    assert fuses(x, None)
    monkeypatch.setattr(torch.compiler, "is_compiling", lambda: True)
    assert not fuses(x, None)


# (M, K, rows, Huffman, rANS): whether the tiled product was the faster one by more than 2 % (None: about equal)
MEASURED = [
    (640, 1024, 17, True, True), (640, 1024, 48, True, None), (640, 1024, 64, None, False), (640, 1024, 65, False, False),
    (1024, 4096, 17, True, None), (4096, 4096, 17, True, True), (4096, 4096, 96, True, True),
    (12288, 4096, 17, None, False), (12288, 4096, 32, True, True), (12288, 4096, 128, True, True),
    (11008, 4096, 20, None, False), (13824, 5120, 20, True, True), (4096, 11008, 17, None, False), (4096, 11008, 32, True, True),
    (4096, 12288, 17, True, True), (2048, 11008, 17, True, True), (1024, 18944, 17, None, False), (1024, 18944, 32, True, True),
    (3584, 18944, 17, False, False), (3584, 18944, 24, False, False), (3584, 18944, 32, True, False), (3584, 18944, 33, True, True),
    (4096, 14336, 24, False, False), (16384, 3584, 17, False, False), (16384, 3584, 32, False, False), (16384, 3584, 33, True, True),
    (16384, 4096, 24, False, False), (18944, 3584, 17, True, True), (18944, 3584, 80, True, True), (18944, 3584, 96, True, False),
    (24576, 4096, 17, True, True), (24576, 4096, 96, True, True), (8192, 8192, 17, True, False), (8192, 8192, 24, True, None),
    (1536, 6784, 17, True, False), (9216, 5504, 20, True, False), (5120, 13824, 17, True, True), (16384, 1024, 112, True, True),
]


@pytest.mark.parametrize("M,K,rows,huffman,rans", MEASURED)
def test_tiled_product_is_chosen_where_it_was_faster(M, K, rows, huffman, rans):
    from bf16_huffman_infer_amd.functional import prefers_tiles
    from bf16_huffman_infer_amd.utils import get_block_size_n
    split_k, = get_block_size_n(torch.empty(1, K, device="meta"))
    assert huffman is None or prefers_tiles(rows, M, K, split_k, True) == huffman
    assert rans is None or prefers_tiles(rows, M, K, split_k, False) == rans


def test_wide_product_is_cut_while_every_block_has_a_unit():
    """Slices divide the tasks of a row group and leave at most 256 blocks; the workspace holds counters, whole
    tiles of X and, where K is cut, whole rounds of eight tiles per slice."""
    from bf16_huffman_infer_amd import _lib
    lib = _lib.load()
    for split_k, M, Ks in [(1, 128, 128), (1, 1024, 4096), (3, 4096, 4096), (4, 3584, 4736), (1, 18944, 3584), (1, 12288, 4096),
                           (2, 65536, 2048), (5, 3328, 1280), (12, 128, 1024)]:
        per_group = split_k * lib.bhi_chunks_per_group(M, Ks, split_k)
        slices = lib.bhi_wide_slices(split_k, M, Ks)
        assert slices == max([1] + [d for d in range(2, 9) if per_group % d == 0 and M // 64 * d <= 256])
        for rows in (17, 128, 129, 144, 145, 320, 321, 640):
            tiles = -(-rows // 16)
            want = 1024 + tiles * 16 * split_k * Ks * 2 + (-(-tiles // 8) * 8 * 16 * M * 4 * slices if slices > 1 else 0)
            assert lib.bhi_wide_workspace_bytes(split_k, M, Ks, rows) == want
        assert lib.bhi_wide_workspace_bytes(split_k, M, Ks, 16) < 0 and lib.bhi_wide_workspace_bytes(split_k, M, Ks, 641) < 0


def test_wide_rule():
    """Sides of the measured table: small layers and long prompts on half-empty units stay where they were."""
    from bf16_huffman_infer_amd.functional import prefers_wide
    assert [r for r in (32, 33, 64, 96, 256, 640) if prefers_wide(r, 12288, 4096)] == [96, 256, 640]
    assert [r for r in (32, 33, 96, 256, 640) if prefers_wide(r, 4096, 12288, 3)] == [32, 33, 96, 256, 640]
    assert [r for r in (33, 80, 81, 192, 193, 320, 321) if prefers_wide(r, 18944, 3584)] == [81, 192, 193, 320]
    assert [r for r in (33, 80, 81, 192, 193, 320) if prefers_wide(r, 18944, 3584, 1, False)] == [81, 192]
    assert not any(prefers_wide(r, 512, 1024) for r in (17, 33, 64, 128, 300, 640))


# (M, K, Huffman, rows where the wide product was faster by more than 2 %, rows where the other path was): every such entry of the
# tables in prefers_wide and bhi_wide.h but the four that prefers_wide names as left to the slower side
WIDE_MEASURED = [
    (512, 1024, True, [], [32, 256, 640]),
    (1024, 4096, True, [64], [256, 640]),
    (2048, 2048, False, [64, 96], [256, 640]),
    (4608, 3584, True, [64, 96, 256], [32, 640]),
    (12288, 4096, True, [96, 128, 192, 256, 300, 512, 640], [32, 33]),
    (3584, 3584, False, [64, 96], [640]),
    (4096, 12288, False, [32, 64, 96, 256, 640], []),
    (8192, 8192, True, [32, 64, 96, 256, 640], []),
    (18944, 3584, True, [96, 128, 192, 256, 300], [32, 33, 64, 512, 640]),
    (18944, 3584, False, [96], [32, 64, 640]),
    (32768, 2048, False, [256, 640], [32, 64]),
    (4096, 4096, True, [33, 64, 96, 128, 192], [512]),
    (12288, 4096, False, [96, 128, 192, 300, 512], [33]),
    (4096, 12288, True, [33, 64, 96, 128, 192, 300, 512], []),
    (3584, 18944, True, [33, 64, 96, 128, 192, 300, 512], []),
    (8192, 8192, False, [33, 64, 96, 128, 192, 300, 512], []),
]


@pytest.mark.parametrize("M,K,huffman,wide,other", WIDE_MEASURED)
def test_wide_product_is_chosen_where_it_was_faster(M, K, huffman, wide, other):
    from bf16_huffman_infer_amd.functional import prefers_wide
    from bf16_huffman_infer_amd.utils import get_block_size_n
    split_k, = get_block_size_n(torch.empty(1, K, device="meta"))
    assert [r for r in wide if not prefers_wide(r, M, K, split_k, huffman)] == []
    assert [r for r in other if prefers_wide(r, M, K, split_k, huffman)] == []


# in front of the rules: what the package's own conversion does not make (it wants M % 128 == 0), but check_layout and the library take
@pytest.mark.parametrize("M", [4, 32, 60, 96, 192, 8256, 12224])
@pytest.mark.parametrize("rows", [17, 40, 128, 200, 640])
def test_wide_rule_leaves_heights_that_fused_calls_refuse(M, rows):
    from bf16_huffman_infer_amd.functional import prefers_wide
    for K, split_k in ((1024, 1), (4096, 1), (12288, 3)):
        assert not prefers_wide(rows, M, K, split_k, True) and not prefers_wide(rows, M, K, split_k, False)


def test_wide_rule_leaves_widths_that_the_library_refuses():
    from bf16_huffman_infer_amd.functional import prefers_wide
    for M, K, split_k in ((128, 100, 1), (128, 64, 1), (16384, 4000, 1), (16384, 8192, 3), (128, 1 << 20, 1)):
        assert not any(prefers_wide(rows, M, K, split_k) for rows in (17, 40, 200, 640)), (M, K, split_k)


def test_rules_are_asked_with_whole_numbers():
    """Under torch.jit.trace sizes are tensors, and the rules remember what they were asked."""
    import types
    from bf16_huffman_infer_amd.functional import _takes
    asked, x = [], torch.zeros(24, 512, dtype=torch.bfloat16)
    weight = types.SimpleNamespace(rem=torch.zeros(2, 128, 256, dtype=torch.uint8))

    def rule(*args):
        asked.append(args)
        return True

    def step(v, rem):
        of_gpu = types.SimpleNamespace(size=v.size, numel=v.numel, dtype=v.dtype, is_cuda=True)
        assert type(v.size(0)) is torch.Tensor
        assert _takes(of_gpu, types.SimpleNamespace(rem=rem), None, 17, 32, rule)
        return v + 1
    torch.jit.trace(step, (x, weight.rem), check_trace=False)
    assert asked and all(type(a) in (int, bool) for args in asked for a in args) and asked[0][:4] == (24, 128, 512, 2)
