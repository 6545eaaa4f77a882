"""GPU parity of products whose K is no multiple of 16 (or whose rows are unaligned) past the
small-product sizes, with the weight packed on the call: exact against a float64 product.
"""
import numpy as np
import pytest
import torch

from iconnx_amd import ops

pytestmark = pytest.mark.gpu


def ints(g, dt, shape):
    lo, hi = (-128, 128) if dt == torch.int8 else (0, 256)
    return torch.randint(lo, hi, shape, generator=g, device="cuda", dtype=torch.int32).to(dt)


def shifted(t, by):
    buf = torch.empty(t.numel() + 32, dtype=t.dtype, device="cuda")
    v = buf[by:by + t.numel()].view(t.shape)
    v.copy_(t)
    return v


# 64x64 tiles up to 384 tiles of 128x128, 128x128 past that; K < 16, one short of / one past a
# 64-wide step, whole steps on unaligned rows, K % 16 == 0 with a partial step
@pytest.mark.parametrize("M,N", [(1530, 1500), (4097, 130), (2200, 4100)])
@pytest.mark.parametrize("K", [3, 15, 17, 63, 65, 128, 200, 1000, 1040])
def test_exact(M, N, K):
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    adt, bdt = [(torch.uint8, torch.uint8), (torch.int8, torch.int8), (torch.uint8, torch.int8)][K % 3]
    a, b = ints(g, adt, (M, K)), ints(g, bdt, (K, N))
    azp, bzp = ints(g, adt, ()), ints(g, bdt, ())
    want = (a.double() - azp.double()) @ (b.double() - bzp.double())  # below 2^53: exact
    for ad, bd in ((a, b), (shifted(a, 1), shifted(b, 3))):
        got = ops.gpu_matmul_integer(ad, bd, azp, bzp)
        assert torch.equal(got.double(), want)
    w = ops.PackedWeight(shifted(b, 5))
    assert torch.equal(w.packed.t().int(), b.int() - (128 if bdt == torch.uint8 else 0))
    assert torch.equal(w.colsum, w.packed.sum(1, dtype=torch.int32))
    y = ops.gpu_qlinear(a, w, azp, bzp, epilogue=[("Mul", torch.tensor(0.5, device="cuda"), False)])
    assert torch.equal(y, want.float() * 0.5)  # |acc| < 2^24 * 255: the Cast rounds as .float()


def test_full_operand_epilogue():
    g = torch.Generator(device="cuda").manual_seed(5)
    M, K, N = 1100, 333, 900
    a, b, full = ints(g, torch.uint8, (M, K)), ints(g, torch.int8, (K, N)), torch.randn(M, N, generator=g, device="cuda")
    y = ops.gpu_qlinear(a, ops.PackedWeight(b), epilogue=[("Add", full, False)])
    assert torch.equal(y, (a.double() @ b.double()).float() + full)


def test_unpacked_row_sums_of_long_rows():
    g = torch.Generator(device="cuda").manual_seed(6)
    a, b = ints(g, torch.uint8, (700, 4099)), ints(g, torch.uint8, (4099, 1111))
    azp, bzp = ints(g, torch.uint8, ()), ints(g, torch.uint8, (1111,))
    want = (a.double() - azp.double()) @ (b.double() - bzp.double())
    assert torch.equal(ops.gpu_matmul_integer(a, b, azp, bzp).double(), want)


def test_rows_up_to_the_launch_limit():
    """2^26 - 4 rows of one byte and 8 weight columns: the sums of either fit a launch of one wave
    a row (2^32 - 1 threads), the two together do not."""
    M, N = (1 << 26) - 4, 8
    a = torch.randint(0, 256, (M, 1), device="cuda", dtype=torch.uint8)
    b = torch.randint(0, 256, (1, N), device="cuda", dtype=torch.uint8)
    azp, bzp = (torch.tensor(z, dtype=torch.uint8, device="cuda") for z in (7, 131))
    got = ops.gpu_matmul_integer(a, b, azp, bzp)
    assert torch.equal(got, (a.int() - 7) * (b.int() - 131))
