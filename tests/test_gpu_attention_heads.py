"""GPU parity of the fused self-attention past 128 keys, at most 80, and at head sizes other than
64, through the graph executor: against float64 within 1e-5, with the padding mask, both scale
positions, partial chunks, key tiles and query tiles, and the range it leaves for a
DynamicQuantizeLinear.
"""
import threading

import numpy as np
import pytest
import torch

import oracle
from iconnx_amd import graphs, ops
from iconnx_amd.executor import GpuGraphExecutor

pytestmark = pytest.mark.gpu


def reference(q, k, v, heads, mask=None):
    B, S, HD = q.shape
    split = lambda t: t.astype(np.float64).reshape(B, S, heads, HD // heads).transpose(0, 2, 1, 3)  # noqa: E731
    s = split(q) @ split(k).transpose(0, 1, 3, 2) / np.sqrt(HD // heads)
    if mask is not None:
        s = np.where(mask[:, None, None, :] == 0, float(graphs.F32_MIN), s)
    e = np.exp(s - s.max(-1, keepdims=True))
    return ((e / e.sum(-1, keepdims=True)) @ split(v)).transpose(0, 2, 1, 3).reshape(B, S, HD)


def inputs(B, S, HD, seed):
    rng = np.random.default_rng(seed)
    return {n: rng.normal(size=(B, S, HD)).astype(np.float32) * (1.0 + i) for i, n in enumerate("qkv")}


def close(got, want):
    # sums of <= 128 products and <= 8192 weights in float32; outputs of the values' magnitude
    assert np.abs(got - want).max() <= 1e-5 * max(1.0, np.abs(want).max())


# every padded head size (16, 32, 48, 64, 80, 96, 128), one and several chunks of 128 keys, one
# key, one past a key tile; the last two take 128 queries a block
@pytest.mark.parametrize("B,S,H,D", [(1, 1, 1, 4), (2, 17, 3, 16), (3, 128, 2, 20), (2, 130, 3, 32), (2, 37, 4, 40),
                                     (1, 257, 2, 48), (2, 129, 3, 64), (1, 100, 2, 72), (1, 300, 2, 80),
                                     (2, 65, 2, 96), (1, 200, 2, 100), (1, 385, 2, 128), (64, 129, 16, 32),
                                     (40, 200, 16, 64)])
def test_head_sizes(B, S, H, D):
    feeds = inputs(B, S, H * D, S + D)
    ex = GpuGraphExecutor()
    for n in "qkv":
        ex.add_input(n, [None, None, H * D])
    ctx = graphs.add_self_attention(ex, "q", "k", "v", H, D, "a")
    quant = graphs.add_dynamic_quantize(ex, ctx, "d")
    out = ex.run(feeds, [ctx] + list(quant))
    close(out[ctx], reference(*feeds.values(), H))
    for name, w in zip(quant, oracle.dynamic_quantize_linear(out[ctx])):
        assert np.array_equal(out[name], w), name


@pytest.mark.parametrize("B,S,H,D", [(3, 50, 2, 32), (2, 256, 2, 48), (2, 300, 3, 64), (2, 140, 2, 128)])
def test_padding_mask(B, S, H, D):
    feeds = inputs(B, S, H * D, 7)
    mask = np.ones((B, S), np.int64)
    for b in range(B):
        mask[b, S - 1 - 13 * b:] = 0
    mask[0, ::3] = 0
    ex = GpuGraphExecutor()
    for n in "qkv":
        ex.add_input(n, [None, None, H * D])
    ex.add_input("m", [None, None], 7)
    ctx = graphs.add_self_attention_export(ex, "q", "q", "k", "v", "m", H, D, "a")
    close(ex.run(dict(feeds, m=mask), [ctx])[ctx], reference(*feeds.values(), H, mask))


# heads of 64 about the 80 keys up to which the f32 context comes from this kernel: against
# float64, and with the context not requested, where the one-tile kernel quantizes its own
# output, that output is the quantization of the same bits
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("B,S,H", [(2, 1, 1), (2, 16, 3), (3, 17, 2), (2, 63, 3), (4, 64, 2), (3, 65, 4), (2, 80, 3), (2, 81, 3)])
def test_heads_of_64_both_kernels(B, S, H, masked):
    feeds = inputs(B, S, H * 64, S)
    mask = np.ones((B, S), np.int64)
    if masked:
        mask[0, ::3] = 0
        mask[B - 1, S // 2 + 1:] = 0
        feeds = dict(feeds, m=mask)

    def build(requested):
        ex = GpuGraphExecutor()
        for n in "qkv":
            ex.add_input(n, [None, None, H * 64])
        if masked:
            ex.add_input("m", [None, None], 7)
            ctx = graphs.add_self_attention_export(ex, "q", "q", "k", "v", "m", H, 64, "a")
        else:
            ctx = graphs.add_self_attention(ex, "q", "k", "v", H, 64, "a")
        quant = list(graphs.add_dynamic_quantize(ex, ctx, "d"))
        out = ex.run(feeds, quant + [ctx] * requested)
        return out, ctx, quant, ex.quantized_outputs()[1]

    out, ctx, quant, launches = build(True)
    assert launches == 0
    # a row whose every key is masked: equal weights
    close(out[ctx], reference(feeds["q"], feeds["k"], feeds["v"], H, mask if masked else None))
    want = oracle.dynamic_quantize_linear(out[ctx])
    own, _, _, launches = build(False)
    assert launches == 1
    for name, w in zip(quant, want):
        assert np.array_equal(out[name], w), name
        assert np.array_equal(own[name], w), name


@pytest.mark.parametrize("scale,div", [(8.0, True), (3.0, True), (0.125, False)])
def test_score_scales(scale, div):
    f = inputs(2, 259, 128, 9)
    q, k, v = (torch.from_numpy(f[n]).cuda() for n in "qkv")
    want = reference(f["q"] * (8.0 / scale if div else 8.0 * scale), f["k"], f["v"], 2)
    close(ops.gpu_attention(q, k, v, 2, scale, scale_div=div).cpu().numpy(), want)


def test_unaligned_inputs_run_node_by_node():
    f = inputs(1, 40, 96, 11)
    ex = GpuGraphExecutor()
    bound = {}
    for n in "qkv":
        ex.add_input(n, [None, None, 96])
        buf = torch.empty(40 * 96 + 1, device="cuda")
        bound[n] = buf[1:].view(1, 40, 96)
        bound[n].copy_(torch.from_numpy(f[n]))
    ctx = graphs.add_self_attention(ex, "q", "k", "v", 3, 32, "a")
    close(ex.run_device(bound, [ctx])[ctx].cpu().numpy(), reference(*f.values(), 3))


# no less exact than the nodes that it stands for (the same random inputs: a fixed outcome)
@pytest.mark.parametrize("B,S,H,D", [(32, 128, 12, 32), (16, 384, 12, 32), (8, 200, 12, 40), (8, 128, 16, 80),
                                     (4, 512, 8, 128), (8, 256, 8, 56)])
def test_error_of_the_separate_nodes(B, S, H, D):
    g = torch.Generator(device="cuda").manual_seed(S + D)
    feeds = {n: torch.randn((B, S, H * D), generator=g, device="cuda") for n in "qkv"}
    ex = GpuGraphExecutor()
    for n in "qkv":
        ex.add_input(n, [None, None, H * D])
    ctx = graphs.add_self_attention(ex, "q", "k", "v", H, D, "a")
    got = ex.run_device(feeds, [ctx])[ctx]
    q, k, v = (ops.gpu_transpose(feeds[n].view(B, S, H, D), (0, 2, 1, 3)) for n in "qkv")
    scale = torch.full((1,), float(np.float32(np.sqrt(D))), device="cuda")
    s = ops.gpu_matmul_f32(ops.gpu_fused_chain(q, [("Div", scale, False)]), ops.gpu_transpose(k, (0, 1, 3, 2)))
    nodes = ops.gpu_transpose(ops.gpu_matmul_f32(ops.gpu_softmax(s), v), (0, 2, 1, 3)).reshape(B, S, H * D)
    s = torch.matmul(q.double(), k.double().transpose(2, 3).contiguous()) / D ** 0.5
    want = torch.matmul(torch.softmax(s, -1), v.double()).transpose(1, 2).reshape(B, S, H * D)
    err = lambda t: float((t.double() - want).norm())  # noqa: E731
    assert err(got) <= err(nodes)


# scores of -25 to -80 below one of 0, all exact, over values that pick one weight each: the sum
# rounds to 1, so a context is the exponential itself, within 1 ulp (2^-23) and the division's
# half one; an exponential whose argument, the product with log2 e, is rounded to float is off by
# up to 2^-18 ln 2 = 2.6e-6
@pytest.mark.parametrize("D,S", [(16, 16), (32, 32), (96, 96)])
def test_weights_of_distant_scores(D, S):
    rng = np.random.default_rng(D)
    q, k, v = (np.zeros((1, S, D), np.float32) for _ in range(3))
    q[0, :, 0] = np.float32(np.sqrt(D))  # divided by the scale: 1
    k[0, 1:, 0] = -rng.uniform(25.0, 80.0, S - 1).astype(np.float32)
    v[0, np.arange(S), np.arange(S)] = 1.0
    ex = GpuGraphExecutor()
    for n in "qkv":
        ex.add_input(n, [None, None, D])
    ctx = graphs.add_self_attention(ex, "q", "k", "v", 1, D, "a")
    got = ex.run(dict(q=q, k=k, v=v), [ctx])[ctx].astype(np.float64)
    want = np.exp(k[0, :, 0].astype(np.float64))
    assert (np.abs(got[0] / want - 1.0) <= 1.5 * 2.0 ** -23).all()


def test_threads_with_streams_of_their_own():
    """First launches of the kernels with more than 64 KB of LDS from several threads at once."""
    def work(i, results):
        D, S = [80, 96, 128, 64][i % 4], 40 + 70 * (i // 4)
        f = inputs(1, S, 2 * D, 50 + i)
        with torch.cuda.stream(torch.cuda.Stream()):
            ex = GpuGraphExecutor()
            for n in "qkv":
                ex.add_input(n, [None, None, 2 * D])
            ctx = graphs.add_self_attention(ex, "q", "k", "v", 2, D, "a")
            results[i] = [ex.run(f, [ctx])[ctx] for _ in range(3)], reference(*f.values(), 2)

    torch.cuda.synchronize()
    results = {}
    threads = [threading.Thread(target=work, args=(i, results)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(results) == 8
    for got, want in results.values():
        for g in got:
            close(g, want)
