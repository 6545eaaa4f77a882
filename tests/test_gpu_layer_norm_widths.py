"""GPU parity of the LayerNorm at any width: bit-exact against the oracle's summation order at
the edges of its row blocks, load widths and leftovers, with row-periodic residuals and the
range it leaves for a DynamicQuantizeLinear.
"""
import numpy as np
import pytest
import torch

import oracle
from iconnx_amd import graphs, ops
from iconnx_amd.executor import GpuGraphExecutor

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def bits(a):
    return np.ascontiguousarray(a).view(np.uint32)


def params(rng, cols):
    return rng.uniform(0.9, 1.1, cols).astype(np.float32), rng.normal(size=cols).astype(np.float32)


@pytest.mark.parametrize("rows,cols", [(1, 1), (33, 1), (5, 7), (65, 9), (1025, 64), (4099, 96), (1200, 127),
                                       (513, 384), (12288, 384), (515, 1028), (3, 4095), (600, 4096), (2, 12288),
                                       (2, 12289)])
@pytest.mark.parametrize("residual", [False, True])
def test_bit_exact_at_any_width(rows, cols, residual):
    rng = np.random.default_rng(rows * 13 + cols)
    x, r = (rng.normal(size=(rows, cols)).astype(np.float32) for _ in range(2))
    sc, bi = params(rng, cols)
    got = ops.gpu_layer_norm(dev(x), dev(sc), dev(bi), 1e-5, dev(r) if residual else None).cpu().numpy()
    want = oracle.layer_norm(oracle.add(x, r) if residual else x, sc, bi, eps=1e-5)
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("cols", [384, 768])
def test_unaligned_input_and_no_affine(cols):
    rng = np.random.default_rng(cols)
    x = rng.normal(size=(70, cols)).astype(np.float32)
    buf = torch.empty(x.size + 1, device="cuda")
    buf[1:] = dev(x).reshape(-1)
    got = ops.gpu_layer_norm(buf[1:].view(70, cols), None, None, 1e-5).cpu().numpy()
    want = oracle.layer_norm(x, np.ones(cols, np.float32), np.full(cols, -0.0, np.float32), eps=1e-5)
    assert np.array_equal(bits(got), bits(want))


@pytest.mark.parametrize("B,S,cols", [(3, 37, 384), (2, 50, 90), (40, 128, 320)])
def test_periodic_residual_then_dynamic_quantize(B, S, cols):
    """[1, S, C] added over [B, S, C], the node-by-node LayerNorm, its DynamicQuantizeLinear."""
    rng = np.random.default_rng(B * S)
    x, pos = rng.normal(size=(B, S, cols)).astype(np.float32), rng.normal(size=(1, S, cols)).astype(np.float32)
    sc, bi = params(rng, cols)
    ex = GpuGraphExecutor()
    ex.add_input("x", [None, None, cols])
    ex.add_initializer("pos", pos)
    y = graphs.add_layer_norm_decomposed(ex, "x", "pos", sc, bi, 1e-12, "ln")
    q = graphs.add_dynamic_quantize(ex, y, "q")
    out = ex.run({"x": x}, list(q) + [y])
    want = oracle.layer_norm_decomposed(oracle.add(x, pos), sc, bi, np.float32(1e-12), square=True)
    assert np.array_equal(bits(out[y]), bits(want))
    for name, w in zip(q, oracle.dynamic_quantize_linear(want)):
        assert np.array_equal(out[name], w), name
