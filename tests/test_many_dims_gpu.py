"""Layouts of more dims than the 32-bit kernels' arguments have room for: they run in the kernels with 64-bit offsets, which go
through the dims in 32 bits where the offsets fit."""
import numpy as np
import pytest

from tests.util import assert_bit_equal

pytestmark = pytest.mark.gpu


def _window(thc, kind, x, cut):
    """A window of x on the device, some elements narrower in every dim: no two dims merge."""
    dev = thc.Tensor.from_numpy(x)
    host = x
    for d in range(x.ndim):
        dev = dev.narrow(d, cut[d], x.shape[d] - 1)
        host = np.take(host, range(cut[d], cut[d] + x.shape[d] - 1), axis=d)
    return dev, host


@pytest.mark.parametrize("force64", [False, True])
@pytest.mark.parametrize("kind", ["float", "half", "int", "byte"])
@pytest.mark.parametrize("sizes", [(3, 4, 3, 4, 3, 5), (3, 4, 3, 4, 3, 4, 18), (2, 3, 4, 3, 2, 4, 3, 9), (2, 3, 2, 3, 2, 3, 2, 3, 2, 4, 2, 3, 5)])
def test_more_dims_than_the_32_bit_kernels_hold(thc, kind, sizes, force64):
    dtype = {"float": np.float32, "half": np.float16, "int": np.int32, "byte": np.uint8}[kind]
    rng = np.random.default_rng(len(sizes))
    shape = tuple(s + 1 for s in sizes)
    x, y = (rng.integers(0, 5, shape).astype(dtype) for _ in range(2))
    a, ha = _window(thc, kind, x, [int(rng.integers(0, 2)) for _ in shape])
    b, hb = _window(thc, kind, y, [int(rng.integers(0, 2)) for _ in shape])
    order = tuple(reversed(range(len(sizes))))
    strides = [1]
    for s in reversed(sizes[1:]):
        strides.append(strides[-1] * s)
    rev = thc.Tensor.from_storage(np.ascontiguousarray(ha.transpose(order)).reshape(-1), 0, sizes,
                                  tuple(int(np.prod(sizes[:d], dtype=np.int64)) for d in range(len(sizes))), kind=kind)
    thc.force_64bit_index(force64)
    try:
        assert_bit_equal(thc.Tensor(kind).resize(sizes).copy(a).numpy(), ha, "copy")
        assert_bit_equal(thc.Tensor(kind).resize(sizes).cadd(a, 1, b).numpy(), ha + hb, "add")
        assert_bit_equal(thc.Tensor(kind).resize(sizes).cmul(rev, b).numpy(), ha * hb, "reversed")
        # (one scalar a row, gathered beside dense operands)
        row = thc.Tensor.from_numpy(np.ascontiguousarray(ha[..., :1]))
        wide = row.view_as_strided(0, sizes, tuple(s // sizes[-1] for s in reversed(strides))[:-1] + (0,))
        dense = thc.Tensor.from_numpy(np.ascontiguousarray(hb))
        assert_bit_equal(thc.Tensor(kind).resize(sizes).cadd(wide, 1, dense).numpy(), np.broadcast_to(ha[..., :1], sizes) + hb, "row scalar")
        # (operands of different shapes are paired by their linear index)
        flat = thc.Tensor(kind).resize((int(np.prod(sizes)),))
        assert_bit_equal(flat.copy(a).numpy(), ha.reshape(-1), "other shape")
        for dim in (0, len(sizes) // 2, len(sizes) - 1):
            assert_bit_equal(thc.Tensor(kind).sum(a, dim).numpy(), ha.astype(np.int64).sum(axis=dim, keepdims=True).astype(dtype), "sum %d" % dim)
            vals, idx = thc.Tensor(kind), thc.Tensor("long")
            vals.max(idx, a, dim)
            assert_bit_equal(vals.numpy(), ha.max(axis=dim, keepdims=True), "max %d" % dim)
            assert np.array_equal(idx.numpy(), np.expand_dims(ha.argmax(axis=dim), dim) + 1), dim
        assert int(a.sumall()) == int(ha.astype(np.int64).sum())
    finally:
        thc.force_64bit_index(False)


@pytest.mark.parametrize("reach", [(1 << 31) - 1, 1 << 31, (1 << 31) + 77])
def test_many_dims_on_both_sides_of_32_bit_offsets(thc, reach):
    """Eight dims of two whose last element lies `reach` elements in: the largest offset that 32 bits are used for, and past it."""
    sizes = (2,) * 8
    steps = [3 ** k for k in range(7)]                          # any sum of some of them is another offset
    steps.append(reach - sum(steps))
    store = thc.Tensor("byte").resize((reach + 1,)).zero()
    offsets = [sum(s for s, bit in zip(steps, range(8)) if i >> (7 - bit) & 1) for i in range(256)]
    for i, o in enumerate(offsets):
        store.narrow(0, o, 1).fill(1 + i % 255)
    view = store.view_as_strided(0, sizes, tuple(steps))
    want = (1 + np.arange(256) % 255).astype(np.uint8).reshape(sizes)
    assert_bit_equal(thc.Tensor("byte").resize(sizes).copy(view).numpy(), want, "copy")
    assert_bit_equal(thc.Tensor("byte").sum(view, 3).numpy(), want.sum(axis=3, keepdims=True, dtype=np.int64).astype(np.uint8), "sum")
    vals, idx = thc.Tensor("byte"), thc.Tensor("long")
    vals.max(idx, view, 0)
    assert_bit_equal(vals.numpy(), want.max(axis=0, keepdims=True), "max")
    assert np.array_equal(idx.numpy(), np.expand_dims(want.argmax(axis=0), 0) + 1)
    view.mul(view, 3)
    assert_bit_equal(thc.Tensor("byte").resize(sizes).copy(view).numpy(), (want.astype(np.int64) * 3).astype(np.uint8), "in place")
