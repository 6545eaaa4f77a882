"""GPU parity of the products with few output tiles (the kernel that splits K over a block's
waves): exact int32 at the edges of its 16 / 32 / 64-row tiles, 64-wide K steps, partial last
steps and unaligned rows, in all sign combinations, and its epilogue against the oracle's ops.
"""
import ctypes

import numpy as np
import pytest
import torch

import oracle
from iconnx_amd import _lib, ops

pytestmark = pytest.mark.gpu


def dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def off_by_one(a):
    """The same matrix on the device, its first byte one past a 16-byte boundary."""
    buf = torch.empty(a.size + 17, dtype=torch.from_numpy(a).dtype, device="cuda")
    v = buf[1:1 + a.size].view(a.shape)
    v.copy_(torch.from_numpy(a))
    return v


def draw(rng, dt, shape):
    return rng.integers(np.iinfo(dt).min, np.iinfo(dt).max + 1, shape).astype(dt)


def want_i32(a, b, azp, bzp):
    acc = (a.astype(np.int64) - np.int64(azp)) @ (b.astype(np.int64) - np.asarray(bzp, np.int64))
    return acc.astype(np.int32)


# 16x16 tiles (up to 384 of them), 32x32, and 64x32 with K >= 2048 (64x256x... and the last two)
@pytest.mark.parametrize("M,N", [(1, 1), (15, 17), (16, 16), (17, 33), (33, 3000), (300, 601), (31, 4096)])
@pytest.mark.parametrize("K", [1, 15, 16, 17, 63, 64, 65, 100, 256, 783, 1040])
def test_edges_of_tiles_and_steps(M, N, K):
    rng = np.random.default_rng(M * 7919 + N * 31 + K)
    adt, bdt = [(np.uint8, np.int8), (np.int8, np.int8), (np.int8, np.uint8), (np.uint8, np.uint8)][(M + K) % 4]
    a, b = draw(rng, adt, (M, K)), draw(rng, bdt, (K, N))
    azp, bzp, bcol = draw(rng, adt, ()), draw(rng, bdt, ()), draw(rng, bdt, (N,))
    w = ops.PackedWeight(dev(b))
    for bz in (bzp, bcol):
        want = want_i32(a, b, azp, bz)
        for ad in (dev(a), off_by_one(a)):
            np.testing.assert_array_equal(ops.gpu_matmul_integer(ad, w, dev(azp), dev(bz)).cpu().numpy(), want)
    rs = dev(a.astype(np.int64).sum(1).astype(np.int32))  # row sums given rather than formed
    np.testing.assert_array_equal(ops.gpu_matmul_integer(dev(a), w, dev(azp), dev(bzp), a_rowsum=rs).cpu().numpy(),
                                  want_i32(a, b, azp, bzp))


@pytest.mark.parametrize("M,K,N", [(1, 3072, 768), (100, 3072, 768), (129, 4096, 4090), (1000, 2050, 512),
                                   (128, 4096, 4096)])
def test_long_rows(M, K, N):
    rng = np.random.default_rng(M + K + N)
    a, b = draw(rng, np.uint8, (M, K)), draw(rng, np.int8, (K, N))
    azp, bzp = draw(rng, np.uint8, ()), draw(rng, np.int8, ())
    w = ops.PackedWeight(dev(b))
    got = ops.gpu_matmul_integer(dev(a), w, dev(azp), dev(bzp)).cpu().numpy()
    exact = (dev(a).double() - float(azp)) @ (dev(b).double() - float(bzp))  # below 2^53: exact
    np.testing.assert_array_equal(got, exact.cpu().numpy().astype(np.int64).astype(np.int32))


@pytest.mark.parametrize("M,K,N", [(5, 100, 31), (37, 768, 768), (70, 2064, 130)])
def test_epilogue_forms(M, K, N):
    """Column chains, a Div, the erf-GELU's operand-free steps and a full-tensor operand, each
    equal to the oracle's separate ops (the erf within its stated 2e-7 of the formula)."""
    rng = np.random.default_rng(M + K)
    a, b = draw(rng, np.uint8, (M, K)), draw(rng, np.int8, (K, N))
    azp = draw(rng, np.uint8, ())
    s, col = np.float32(1e-3), rng.uniform(0.5, 2, N).astype(np.float32)
    bias, full = rng.normal(size=N).astype(np.float32), rng.normal(size=(M, N)).astype(np.float32)
    w = ops.PackedWeight(dev(b))
    y = want_i32(a, b, azp, 0).astype(np.float32)  # Cast: |acc| < 2^31, rounded to nearest even
    y = oracle.add(oracle.mul(y, oracle.mul(s, col)), bias)
    epi = [("Mul", (dev(np.array(s)), dev(col)), False), ("Add", dev(bias), False)]
    got = ops.gpu_qlinear(dev(a), w, dev(azp), epilogue=epi + [("Div", dev(col), True)]).cpu().numpy()
    np.testing.assert_array_equal(got, oracle.div(np.broadcast_to(col, y.shape), y))
    got = ops.gpu_qlinear(dev(a), w, dev(azp), epilogue=epi + [("Sub", dev(full), False)]).cpu().numpy()
    np.testing.assert_array_equal(got, (y - full).astype(np.float32))
    one, half, rt2 = (dev(np.array(v, np.float32)) for v in (1.0, 0.5, 1.4142135381698608))
    gelu = [("Save", None, False), ("Div", rt2, False), ("Erf", None, False), ("Add", one, False),
            ("MulSaved", None, False), ("Mul", half, False)]
    got = ops.gpu_qlinear(dev(a), w, dev(azp), epilogue=epi + gelu).cpu().numpy()
    e = oracle.erf(oracle.div(y, np.float32(1.4142135381698608)))
    want = oracle.mul(oracle.mul(y, oracle.add(e, np.float32(1.0))), np.float32(0.5))
    # erf differs by at most 1e-6 (the GELU form's bound), times |y| / 2, plus the roundings
    np.testing.assert_allclose(got, want, rtol=4e-7, atol=float(np.abs(y).max()) * 6e-7)


@pytest.mark.parametrize("N", [512, 8192])  # one of few tiles, one of many
@pytest.mark.parametrize("kind,form", [("full", "div"), ("row", "div"), ("full", "gelu"), ("full", "gelu_mul")])
def test_one_row_with_erf_keeps_its_steps(kind, form, N):
    """A full-tensor (or row) operand over a single row: an epilogue with an Erf gives the bits
    that each row of two gives, the division ahead of the Erf and the Erf itself included."""
    K = 128
    rng = np.random.default_rng(5)
    a, w = dev(draw(rng, np.uint8, (1, K))), ops.PackedWeight(dev(draw(rng, np.int8, (K, N))))
    shape = (1, N) if kind == "full" else (1, 1)
    d, scale = dev(rng.uniform(1.0, 2.0, shape).astype(np.float32)), dev(np.full(N, 1 / 5e3, np.float32))
    rt2, inv, one, half = (dev(np.array(v, np.float32)) for v in (1.4142135, 0.70710677, 1.0, 0.5))

    def rows(m):
        am, dm = a.repeat(m, 1), d.repeat(m, 1)
        if form == "div":
            chain = [("Mul", scale, False), ("Div", dm, False), ("Erf", None, False)]
        else:
            chain = [("Mul", scale, False), ("Add", dm, False), ("Save", None, False),
                     ("Div", rt2, False) if form == "gelu" else ("Mul", inv, False), ("Erf", None, False),
                     ("Add", one, False), ("MulSaved", None, False), ("Mul", half, False)]
        ch, keep = ops.build_chain(chain, m, N)
        ch.ops[1].kind0 = _lib.BCAST_FULL if kind == "full" else _lib.BCAST_ROW
        y = torch.empty((m, N), device="cuda")
        ws = torch.empty(1 << 16, dtype=torch.uint8, device="cuda")
        _lib.check(_lib.lib().icx_qlinear_f32(torch.cuda.current_stream().cuda_stream, am.data_ptr(), _lib.ICX_U8,
                                              w.packed.data_ptr(), _lib.ICX_I8, 1, w.colsum.data_ptr(), m, K, N, None,
                                              None, 1, None, ctypes.byref(ch), y.data_ptr(), ws.data_ptr(), ws.numel()))
        torch.cuda.synchronize()
        return y.cpu().numpy()

    one_row, two = rows(1), rows(2)
    assert np.array_equal(one_row[0].view(np.uint32), two[0].view(np.uint32))
    assert np.array_equal(two[0].view(np.uint32), two[1].view(np.uint32))
    assert 0.1 < np.abs(one_row).mean()  # the erf's range is met
