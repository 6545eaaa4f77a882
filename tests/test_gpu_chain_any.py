"""GPU parity of the fused chain with row and full-tensor operands and at any width: bit-exact
against the oracle's separate ops, every op on either side, factor pairs, and the erf steps.
"""
import numpy as np
import pytest
import torch

import oracle
from iconnx_amd import ops

pytestmark = pytest.mark.gpu
OPS = {"Add": oracle.add, "Sub": oracle.sub, "Mul": oracle.mul, "Div": oracle.div}


def dev(a, off=0):
    buf = torch.empty(a.size + 4, device="cuda")
    v = buf[off:off + a.size].view(a.shape)
    v.copy_(torch.from_numpy(np.ascontiguousarray(a)).reshape(a.shape))
    return v


def want(x, chain):
    for op, f, lhs in chain:
        f = oracle.mul(*f) if isinstance(f, tuple) else f
        f = np.broadcast_to(f, x.shape).astype(np.float32)
        x = OPS[op](f, x) if lhs else OPS[op](x, f)
    return x


# one chunk a lane and several, widths of 4 and odd ones, one row, one column
@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 4), (3, 7), (37, 64), (500, 205), (3000, 456), (4097, 1023), (5, 4095),
                                       (70000, 1), (40000, 100)])
@pytest.mark.parametrize("off", [0, 1])
def test_every_operand_kind(rows, cols, off):
    rng = np.random.default_rng(rows + cols)
    u = lambda *s: rng.uniform(0.5, 2.0, s).astype(np.float32)  # noqa: E731
    x, full, row, col, one = u(rows, cols), u(rows, cols), u(rows, 1), u(cols), u()
    chain = [("Mul", (one, col), False), ("Add", full, False), ("Div", row, True), ("Sub", (full, row), True),
             ("Div", col, False), ("Sub", full, False), ("Mul", (col, full), True), ("Add", one, False)]
    on = lambda f: tuple(dev(t, off) for t in f) if isinstance(f, tuple) else dev(f, off)  # noqa: E731
    got = ops.gpu_fused_chain(dev(x, off), [(op, on(f), lhs) for op, f, lhs in chain]).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), want(x, chain).view(np.uint32))


@pytest.mark.parametrize("rows,cols", [(33, 30), (33, 64)])
def test_erf_steps_and_special_values(rows, cols):
    rng = np.random.default_rng(rows * cols)
    x, full = (rng.normal(size=(rows, cols)).astype(np.float32) for _ in range(2))
    x[0, :4] = [np.nan, np.inf, -np.inf, -0.0]
    full[0, :4] = 1.0
    got = ops.gpu_fused_chain(dev(x), [("Save", None, False), ("Erf", None, False), ("Add", dev(full), False),
                                       ("MulSaved", None, False)]).cpu().numpy()
    ref = oracle.mul(x, oracle.add(oracle.erf(x), full))
    # the device erf is within 2e-7 of the oracle's, times |x|
    np.testing.assert_allclose(got, ref, rtol=3e-7, atol=1e-6)


# rows whose grid of whole rows would pass 2^21 blocks (where a 32-bit step of the index wraps), and
# narrower ones past one chunk a lane; a column factor, alone and beside a full tensor
@pytest.mark.parametrize("rows,cols", [(1, 2096131), (1, 2097153), (3, 2097155), (3, 300001), (40, 30522), (100, 4095)])
@pytest.mark.parametrize("inplace", [False, True])
def test_wide_rows(rows, cols, inplace):
    rng = np.random.default_rng(cols)
    u = lambda *s: rng.uniform(0.5, 2.0, s).astype(np.float32)  # noqa: E731
    x, full, row, col, col2 = u(rows, cols), u(rows, cols), u(rows, 1), u(cols), u(cols)
    for chain in ([("Mul", col, False)], [("Sub", col, True), ("Mul", (col, col2), False), ("Add", full, False), ("Div", row, False)]):
        xd = dev(x)
        got = ops.gpu_fused_chain(xd, [(op, tuple(map(dev, f)) if isinstance(f, tuple) else dev(f), lhs)
                                       for op, f, lhs in chain], out=xd if inplace else None).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), want(x, chain).view(np.uint32))
    if rows == 1:  # the same through a 1-D tensor
        got = ops.gpu_fused_chain(dev(x[0]), [("Add", dev(col), False)]).cpu().numpy()
        assert np.array_equal(got.view(np.uint32), oracle.add(x[0], col).view(np.uint32))
