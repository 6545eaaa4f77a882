"""GPU parity of an encoder over few tokens, where the linears quantize the f32 they read from
the range its producer left: bit-identical, layer by layer, to the same graph with every
DynamicQuantizeLinear a launch of its own.
"""
import numpy as np
import pytest
import torch

from iconnx_amd import graphs
from iconnx_amd.executor import GpuGraphExecutor

pytestmark = pytest.mark.gpu


def build(hidden, heads, ffn, fused):
    ex = GpuGraphExecutor()
    out, names, _ = graphs.encoder_graph(ex, layers=2, heads=heads, hidden=hidden, ffn=ffn)
    if not fused:
        ex.set_option("quantized_outputs", False)
    return ex, out, names


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


# launches per run that quantize their input: layer 0's Q/K/V input comes from the caller, so
# a layer has o, ff1 and (after the first) Q/K/V, and ff2 too where its K is at most 1024
@pytest.mark.parametrize("hidden,heads,ffn,B,S,launches", [
    (768, 12, 3072, 1, 1, 5), (768, 12, 3072, 1, 16, 5), (768, 12, 3072, 1, 37, 5), (768, 12, 3072, 3, 17, 3),
    (768, 12, 3072, 2, 96, 2), (768, 12, 3072, 5, 100, 0), (256, 4, 1024, 1, 9, 7), (256, 4, 1024, 1, 129, 7),
    (768, 12, 3072, 9, 128, 0)])
def test_equals_separate_launches(hidden, heads, ffn, B, S, launches):
    x = graphs.encoder_input(B, S, hidden, seed=B * S)
    ref, out, names = build(hidden, heads, ffn, False)
    want = ref.run({"x": x}, [out] + [t[k] for t in names for k in ("q", "v", "o", "x1", "f", "out")])
    ex, _, _ = build(hidden, heads, ffn, True)
    for rep in range(2):
        got = ex.run({"x": x}, [out])[out]
        assert np.array_equal(bits(got), bits(want[out])), rep
    assert ex.range_quantized_inputs() == 2 * launches
    # the same with intermediates requested (not the DQLs'), and recorded and replayed
    keep = [t[k] for t in names for k in ("q", "v", "o", "x1", "f", "out")]
    more, _, _ = build(hidden, heads, ffn, True)
    xin = torch.from_numpy(x).cuda()
    more.capture({"x": xin}, [out] + keep)
    for rep in range(2):
        more.replay()
        got = {k: v.cpu().numpy() for k, v in more.outputs(keep).items()}
        more.check_status()
        for k in keep:
            assert np.array_equal(bits(got[k]), bits(want[k])), (rep, k)


@pytest.mark.parametrize("case", ["nan", "zero", "huge", "one_sided"])
def test_special_values(case):
    """LayerNorm(x) -> DQL -> linear, with the LayerNorm's gain and shift making the DQL's edge
    cases: NaN, an all-zero input (empty range), magnitudes near the f32 limit, one side."""
    M, K, N = 21, 768, 96
    rng = np.random.default_rng(3)
    sc, bi = np.ones(K, np.float32), np.zeros(K, np.float32)
    if case == "nan":
        bi[5::7] = np.nan
        bi[1::9] = -0.0
    elif case == "zero":
        sc[:] = 0.0
    elif case == "huge":
        sc[:] = 5e37
    else:
        bi[:] = 100.0
    x, w = rng.normal(size=(1, M, K)).astype(np.float32), rng.integers(-127, 128, (K, N)).astype(np.int8)

    def make(fused):
        ex = GpuGraphExecutor()
        for name in ("x", "r"):
            ex.add_input(name, [None, None, K])
        n = graphs.add_layer_norm(ex, "x", "r", sc, bi, 1e-5, "ln")
        y = graphs.add_quantized_linear(ex, n, w, None, np.float32(0.01), np.ones(N, np.float32))
        if not fused:
            ex.set_option("quantized_outputs", False)
        return ex.run({"x": x, "r": x[:, ::-1].copy()}, [y])[y], ex

    want, _ = make(False)
    got, ex = make(True)
    assert ex.range_quantized_inputs() == 1
    assert np.array_equal(bits(got), bits(want))
