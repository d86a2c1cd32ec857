"""The one-token attention launch (needs a GPU): against the same step written with torch
operations -- fp32 RMSNorm and rotation, BF16 q/k/cache, fp32 scores and softmax, BF16 weights."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def tables(max_len, d, theta=1e6, device="cuda"):
    inv = 1.0 / (theta ** (torch.arange(0, d, 2, device=device).float() / d))
    ang = torch.arange(max_len, device=device).float()[:, None] * inv[None, :]
    return torch.cat((ang.cos(), ang.cos()), -1).contiguous(), torch.cat((-ang.sin(), ang.sin()), -1).contiguous()


def torch_step(qk, v, w, cos, sin, pos, k_cache, v_cache, q_heads, kv_heads, eps):
    d = qk.shape[-1]
    p = int(pos.item())
    x = F.rms_norm(qk.float(), (d,), None, eps)
    if w is not None:
        x = x * w
    turned = x.view(-1, 2, d // 2).flip(1).reshape(-1, d)
    x = x * cos[p] + turned * sin[p]
    x[:q_heads] *= d ** -0.5
    x = x.bfloat16()
    k_cache[:, p] = x[q_heads:]
    v_cache[:, p] = v
    q = x[:q_heads].view(kv_heads, q_heads // kv_heads, d).float()
    scores = q @ k_cache[:, :p + 1].float().transpose(1, 2)
    weights = torch.softmax(scores, -1).bfloat16().float()
    return (weights @ v_cache[:, :p + 1].float()).view(q_heads, d)


@pytest.mark.parametrize("q_heads,kv_heads", [(32, 8), (4, 2), (8, 8)])
@pytest.mark.parametrize("max_len,positions", [(1024, (0, 1, 5, 255, 256, 257, 700, 1023)), (300, (0, 299)), (4096, (3000,))])
@pytest.mark.parametrize("with_weight", [True, False])
def test_matches_the_torch_formulation(cuda, q_heads, kv_heads, max_len, positions, with_weight):
    from bf16_huffman_infer_amd import ops
    d = 128
    g = torch.Generator(device="cuda").manual_seed(q_heads * 1000 + max_len)
    cos, sin = tables(max_len, d)
    w = (1 + 0.1 * torch.randn(q_heads + kv_heads, d, generator=g, device="cuda")).bfloat16() if with_weight else None
    for p in positions:
        kc = torch.randn(kv_heads, max_len, d, generator=g, device="cuda").bfloat16()
        vc = torch.randn(kv_heads, max_len, d, generator=g, device="cuda").bfloat16()
        qk = (torch.randn(q_heads + kv_heads, d, generator=g, device="cuda") * 3).bfloat16()
        v = torch.randn(kv_heads, d, generator=g, device="cuda").bfloat16()
        pos = torch.tensor([p], device="cuda")
        kc_ref, vc_ref = kc.clone(), vc.clone()
        want = torch_step(qk, v, w, cos, sin, pos, kc_ref, vc_ref, q_heads, kv_heads, 1e-6)
        got = ops.decode_attention(qk, v, w, cos, sin, pos, kc, vc, eps=1e-6)
        # the caches: only slot p changed; v bit for bit, k within one BF16 step (fp32 rounding order of the rotation)
        assert torch.equal(vc.view(torch.int16), vc_ref.view(torch.int16)), p
        untouched = torch.ones(max_len, dtype=torch.bool, device="cuda")
        untouched[p] = False
        assert torch.equal(kc[:, untouched].view(torch.int16), kc_ref[:, untouched].view(torch.int16)), p
        torch.testing.assert_close(kc[:, p].float(), kc_ref[:, p].float(), rtol=2 ** -7, atol=1e-3)
        torch.testing.assert_close(got.float(), want, rtol=2e-2, atol=2e-2, msg=lambda m: f"pos {p}: {m}")


def test_follows_the_position_inside_a_recorded_graph(cuda):
    from bf16_huffman_infer_amd import ops
    q_heads, kv_heads, d, max_len = 8, 2, 128, 512
    g = torch.Generator(device="cuda").manual_seed(5)
    cos, sin = tables(max_len, d)
    kc = torch.zeros(kv_heads, max_len, d, dtype=torch.bfloat16, device="cuda")
    vc = torch.zeros_like(kc)
    qk = torch.zeros(q_heads + kv_heads, d, dtype=torch.bfloat16, device="cuda")
    v = torch.zeros(kv_heads, d, dtype=torch.bfloat16, device="cuda")
    pos = torch.zeros(1, dtype=torch.int64, device="cuda")
    out = torch.empty(q_heads, d, dtype=torch.bfloat16, device="cuda")
    ops.decode_attention(qk, v, None, cos, sin, pos, kc, vc, out=out)
    torch.cuda.synchronize()
    kc.zero_(); vc.zero_()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        ops.decode_attention(qk, v, None, cos, sin, pos, kc, vc, out=out)
        pos.add_(1)
    kc.zero_(); vc.zero_(); pos.zero_()
    kc_ref, vc_ref = kc.clone(), vc.clone()
    for step in range(40):
        qk.copy_((torch.randn(qk.shape, generator=g, device="cuda") * 2).bfloat16())
        v.copy_(torch.randn(v.shape, generator=g, device="cuda").bfloat16())
        want = torch_step(qk, v, None, cos, sin, torch.tensor([step]), kc_ref, vc_ref, q_heads, kv_heads, 1e-6)
        graph.replay()
        torch.cuda.synchronize()
        assert int(pos.item()) == step + 1
        torch.testing.assert_close(out.float(), want, rtol=2e-2, atol=2e-2, msg=lambda m: f"step {step}: {m}")
        kc_ref.copy_(kc)            # keep the reference cache on the kernel's (BF16-step close) k values


def test_rejections(cuda):
    from bf16_huffman_infer_amd import ops
    cos, sin = tables(64, 128)
    kc = torch.zeros(2, 64, 128, dtype=torch.bfloat16, device="cuda")
    qk = torch.zeros(6, 128, dtype=torch.bfloat16, device="cuda")
    v = torch.zeros(2, 128, dtype=torch.bfloat16, device="cuda")
    with pytest.raises(RuntimeError, match="pos"):
        ops.decode_attention(qk, v, None, cos, sin, torch.zeros(1, dtype=torch.int64), kc, kc.clone())
    with pytest.raises(RuntimeError, match="cos and sin"):
        ops.decode_attention(qk, v, None, cos[:32], sin, torch.zeros(1, dtype=torch.int64, device="cuda"), kc, kc.clone())
    with pytest.raises(RuntimeError, match="head dimension"):
        c64, s64 = tables(64, 64)
        ops.decode_attention(qk[:, :64].contiguous(), v[:, :64].contiguous(), None, c64, s64,
                             torch.zeros(1, dtype=torch.int64, device="cuda"), kc[..., :64].contiguous(), kc[..., :64].contiguous())


def _case(q_heads, kv_heads, max_len, seed):
    d = 128
    g = torch.Generator(device="cuda").manual_seed(seed)

    def rand(*shape, scale=1.0):
        return (torch.randn(*shape, generator=g, device="cuda") * scale).bfloat16()
    return (rand(q_heads + kv_heads, d, scale=3), rand(kv_heads, d), rand(kv_heads, max_len, d), rand(kv_heads, max_len, d),
            *tables(max_len, d))


def _step_error(qk, v, cos, sin, p, kc, vc, q_heads, kv_heads, call):
    """Largest difference of ``call``'s output to the torch formulation, in units of its bound: half a
    BF16 step for the output, and 2**-6 of the largest |v| for what last-place flips of q (2**-8 of
    scores of a few tens at most, through the softmax) and the BF16 weights of the torch formulation can do."""
    kc_ref, vc_ref = kc.clone(), vc.clone()
    pos = torch.tensor([p], device="cuda")
    want = torch_step(qk, v, None, cos, sin, pos, kc_ref, vc_ref, q_heads, kv_heads, 1e-6)
    got = call(pos).float()
    assert torch.equal(vc, vc_ref)
    torch.testing.assert_close(kc.float(), kc_ref.float(), rtol=2 ** -7, atol=1e-3)
    return ((got - want).abs() / (want.abs() * 2 ** -8 + 2 ** -6 * vc_ref.float().abs().max())).max().item()


@pytest.mark.parametrize("q_heads,kv_heads", [(28, 4), (31, 1), (32, 1), (6, 2), (20, 1), (16, 16), (128, 64)])
@pytest.mark.parametrize("max_len,positions", [(64, (0, 63)), (1000, (14, 15, 16, 47, 62, 63, 64, 65, 127, 128, 190, 999)),
                                               (8192, (255, 256, 3967, 3968, 6000, 8191))])
def test_split_edges(cuda, q_heads, kv_heads, max_len, positions):
    """Slots at the edges of matrix tiles (16), of a wavefront's share, of splits (64 and its
    multiples) and of the cache; groups of q heads that fill no tile, and more than one tile."""
    from bf16_huffman_infer_amd import ops
    qk, v, kc, vc, cos, sin = _case(q_heads, kv_heads, max_len, q_heads + max_len)
    for p in positions:
        err = _step_error(qk, v, cos, sin, p, kc, vc, q_heads, kv_heads,
                          lambda pos: ops.decode_attention(qk, v, None, cos, sin, pos, kc, vc, eps=1e-6))
        assert err <= 1.0, (p, err)


@pytest.mark.parametrize("q_heads,kv_heads", [(28, 4), (16, 16)])
@pytest.mark.parametrize("positions", [(128, 129, 143, 144, 191), (4095, 4096, 4143, 4144, 5999, 6143, 6144)])
def test_shares_of_three_tiles(cuda, q_heads, kv_heads, positions):
    """Splits of 129 to 192 slots: a wavefront has three matrix tiles, the last block's fewer or a part of one."""
    from bf16_huffman_infer_amd import ops
    qk, v, kc, vc, cos, sin = _case(q_heads, kv_heads, 8192, q_heads)
    for p in positions:
        err = _step_error(qk, v, cos, sin, p, kc, vc, q_heads, kv_heads,
                          lambda pos: ops.decode_attention(qk, v, None, cos, sin, pos, kc, vc, eps=1e-6))
        assert err <= 1.0, (p, err)


@pytest.mark.parametrize("q_heads,kv_heads,max_len,positions", [(28, 4, 8192, (0, 63, 64, 255, 256, 257, 5000)), (3, 3, 300, (299,))])
def test_entry_without_workspace(cuda, q_heads, kv_heads, max_len, positions):
    """The C entry that takes no workspace walks all slots in one block per q head."""
    from bf16_huffman_infer_amd import _lib
    qk, v, kc, vc, cos, sin = _case(q_heads, kv_heads, max_len, 5)
    out = torch.empty(q_heads, 128, dtype=torch.bfloat16, device="cuda")

    def call(pos):
        _lib.check(_lib.load().bhi_decode_attention(
            qk.data_ptr(), v.data_ptr(), None, cos.data_ptr(), sin.data_ptr(), pos.data_ptr(), kc.data_ptr(), vc.data_ptr(),
            out.data_ptr(), q_heads, kv_heads, 128, max_len, 1e-6, 128 ** -0.5, torch.cuda.current_stream().cuda_stream), "attention")
        return out
    for p in positions:
        assert _step_error(qk, v, cos, sin, p, kc, vc, q_heads, kv_heads, call) <= 1.0, p


@pytest.mark.parametrize("recorder", ["torch", "package"])
def test_second_graph_does_not_depend_on_the_first(cuda, recorder):
    """Two graphs recorded one after the other (torch records both on one stream): the second is
    replayed alone, then both in turn, against the eager bits."""
    from bf16_huffman_infer_amd import ops
    from bf16_huffman_infer_amd.cudagraph_utils import GraphedCallable
    qk, v, kc, vc, cos, sin = _case(32, 8, 4096, 9)
    pos = torch.tensor([3000], device="cuda")
    want = ops.decode_attention(qk, v, None, cos, sin, pos, kc, vc).clone()
    graphs, outs = [], []
    for _ in range(2):
        out = torch.zeros_like(want)

        def step(out=out):
            return ops.decode_attention(qk, v, None, cos, sin, pos, kc, vc, out=out)
        if recorder == "package":
            graph = GraphedCallable(step, ())
        else:
            graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(graph):
                step()
        graphs.append(graph)
        outs.append(out)
    for i in (1, 1, 0, 1, 0, 0):
        outs[i].zero_()
        graphs[i].replay()
        assert torch.equal(outs[i], want), i
        assert torch.equal(ops.decode_attention(qk, v, None, cos, sin, pos, kc, vc), want)


def _without_workspace(qk, v, cos, sin, pos, kc, vc, q_heads, kv_heads, out):
    from bf16_huffman_infer_amd import _lib
    _lib.check(_lib.load().bhi_decode_attention(
        qk.data_ptr(), v.data_ptr(), None, cos.data_ptr(), sin.data_ptr(), pos.data_ptr(), kc.data_ptr(), vc.data_ptr(),
        out.data_ptr(), q_heads, kv_heads, 128, kc.shape[1], 1e-6, 128 ** -0.5, torch.cuda.current_stream().cuda_stream), "attention")


@pytest.mark.parametrize("q_heads,kv_heads", [(8, 2), (31, 1), (3, 3)])
@pytest.mark.parametrize("max_len,positions", [(1, (0,)), (64, (0, 1, 15, 63)), (1000, (0, 16, 130, 700)), (4096, (0, 4000))])
@pytest.mark.parametrize("split", [True, False])
def test_slots_from_the_position_on_are_not_read(cuda, q_heads, kv_heads, max_len, positions, split):
    """A cache is allocated once and filled token by token: whatever lies in the slots from the token's
    own on (here NaN, Inf) has no part in the result, which is that of a cache of zeros there, bit for bit."""
    from bf16_huffman_infer_amd import ops
    qk, v, kc, vc, cos, sin = _case(q_heads, kv_heads, max_len, 3 + max_len)
    for p in positions:
        pos = torch.tensor([p], device="cuda")
        results = []
        for filler in (0.0, float("nan"), float("inf")):
            k, w = kc.clone(), vc.clone()
            k[:, p:], w[:, p:] = filler, filler
            out = torch.full((q_heads, 128), 7.0, dtype=torch.bfloat16, device="cuda")
            if split:
                ops.decode_attention(qk, v, None, cos, sin, pos, k, w, out=out)
            else:
                _without_workspace(qk, v, cos, sin, pos, k, w, q_heads, kv_heads, out)
            assert torch.equal(w[:, p], v) and bool(k[:, p].isfinite().all())
            results.append(out)
        assert bool(results[0].isfinite().all())
        assert torch.equal(results[1], results[0]) and torch.equal(results[2], results[0]), p


@pytest.mark.parametrize("split", [True, False])
def test_infinite_values_in_the_last_cached_row_stay_infinite(cuda, split):
    """Slots that fill up a matrix tile read the last cached row again; Inf there is Inf in the output
    (as of any softmax with a weight above 0), not the NaN of 0 * Inf."""
    from bf16_huffman_infer_amd import ops
    q_heads, kv_heads, max_len, p = 8, 2, 512, 70
    qk, v, kc, vc, cos, sin = _case(q_heads, kv_heads, max_len, 11)
    pos = torch.tensor([p], device="cuda")
    want = torch.empty(q_heads, 128, dtype=torch.bfloat16, device="cuda")
    got = torch.empty_like(want)

    def call(out):
        if split:
            ops.decode_attention(qk, v, None, cos, sin, pos, kc, vc, out=out)
        else:
            _without_workspace(qk, v, cos, sin, pos, kc, vc, q_heads, kv_heads, out)
    call(want)
    vc[:, p - 1, 5] = float("inf")
    call(got)
    assert bool((got[:, 5] == float("inf")).all())
    others = torch.arange(128, device="cuda") != 5
    assert torch.equal(got[:, others], want[:, others])
