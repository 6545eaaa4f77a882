"""GPU parity of the one-block DynamicQuantizeLinear: equal to the oracle at the edges of its
sizes, with and without row sums, ties, NaN, infinities, an empty range and unaligned inputs.
"""
import numpy as np
import pytest
import torch

import oracle
from iconnx_amd import ops

pytestmark = pytest.mark.gpu


def check(x, row_len=None, offset=0):
    buf = torch.empty(x.size + 4, device="cuda")
    xd = buf[offset:offset + x.size].view(x.shape)
    xd.copy_(torch.from_numpy(x))
    got = ops.gpu_dynamic_quantize_linear(xd, row_len)
    y, s, z = oracle.dynamic_quantize_linear(x)
    np.testing.assert_array_equal(got[0].cpu().numpy(), y)
    assert np.float32(s).tobytes() == got[1].cpu().numpy().tobytes() and int(z) == int(got[2])
    if row_len:
        np.testing.assert_array_equal(got[3].cpu().numpy(), y.reshape(-1, row_len).astype(np.int32).sum(1))


@pytest.mark.parametrize("n", [1, 3, 4, 5, 767, 4095, 4096, 16383, 16384, 16387, 32767, 32768, 32771, 32772])
def test_sizes(n):
    x = np.random.default_rng(n).normal(size=n).astype(np.float32) * 3
    check(x)
    check(x, offset=1)


@pytest.mark.parametrize("rows,row_len", [(1, 4), (2048, 4), (2049, 4), (16, 768), (4, 4096), (5, 4096), (7, 36), (9, 7)])
def test_row_sums(rows, row_len):
    check(np.random.default_rng(rows).normal(size=(rows, row_len)).astype(np.float32) + 0.5, row_len)


@pytest.mark.parametrize("case", ["ties", "nan", "zeros", "inf", "tiny"])
def test_special_values(case):
    x = np.random.default_rng(1).normal(size=5001).astype(np.float32)
    if case == "ties":  # scale exactly 1: halves lie on ties
        x = (np.arange(5001) % 511).astype(np.float32) / 2
        x[0] = 255.0
    elif case == "nan":
        x[::3] = np.nan
    elif case == "zeros":
        x[:] = 0.0
    elif case == "inf":
        x[7] = np.inf
    else:
        x *= np.float32(1e-41)
    check(x)
