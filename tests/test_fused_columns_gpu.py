"""c = a + b with all dims of a reversed and sizes that leave no row on the 16-byte grid: the inner dims of the
dense operands run as one column dim, and a tile's columns cross the inner dim's boundaries. Every size around
the tile extents (64 x 128 of 4-byte elements, 32 x 64 of 8-byte ones, 56 x 248 of halves); the whole
storages are compared, so nothing outside the output is written."""
import numpy as np
import pytest

from tests.util import assert_bit_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,dtype", [("float", np.float32), ("double", np.float64), ("half", np.float16), ("int", np.int32)])
@pytest.mark.parametrize("x,y,z", [(65, 3, 43), (63, 129, 9), (9, 7, 8), (127, 5, 51), (33, 65, 17), (130, 31, 11), (61, 2, 249)])
def test_reversed_operand_over_odd_sizes(thc, kind, dtype, x, y, z):
    rng = np.random.default_rng(x * 1000 + z)
    n = x * y * z
    for off in (0, 1):
        a = rng.integers(-8, 9, n + 2).astype(dtype)
        b = rng.integers(-8, 9, n + 2).astype(dtype)
        c = np.full(n + 4, 5, dtype)
        ta = thc.Tensor.from_storage(a, off, (x, y, z), (1, x, x * y), kind=kind)
        tb = thc.Tensor.from_storage(b, off, (x, y, z), (y * z, z, 1), kind=kind)
        tc = thc.Tensor.from_storage(c, off, (x, y, z), (y * z, z, 1), kind=kind)
        tc.cadd(ta, 1, tb)
        assert thc.last_kernel() == ("tiled-shift" if kind == "half" else "tiled-ragged-fused"), thc.last_kernel()
        want = c.copy()
        want[off:off + n] = (a[off:off + n].reshape(z, y, x).transpose(2, 1, 0).reshape(-1).astype(np.float64)
                             + b[off:off + n]).astype(dtype)
        assert_bit_equal(tc.storage_numpy(), want, "%s %s +%d" % (kind, (x, y, z), off))


def _strides(sizes, order):
    """Dense strides of `sizes` with the dims laid out in `order`, slowest first."""
    st, run = [0] * len(sizes), 1
    for d in reversed(order):
        st[d], run = run, run * sizes[d]
    return tuple(st)


def _check(thc, kind, dtype, sizes, a_order, b_order, off, expect, seed):
    """c = a + b over whole storages: a (and b) laid out in the given dim orders, c dense."""
    rng = np.random.default_rng(seed)
    n = int(np.prod(sizes))
    nd = len(sizes)
    views, stores = [], []
    for order in (a_order, b_order):
        x = rng.integers(-8, 9, n + 3).astype(dtype)
        views.append(thc.Tensor.from_storage(x, off, sizes, _strides(sizes, order), kind=kind))
        stores.append(x[off:off + n].reshape([sizes[d] for d in order]).transpose(np.argsort(order)).astype(np.float64))
    c = np.full(n + 5, 5, dtype)
    out = thc.Tensor.from_storage(c, off, sizes, _strides(sizes, range(nd)), kind=kind)
    out.cadd(views[0], 1, views[1])
    assert thc.last_kernel() == expect, (sizes, kind, thc.last_kernel())
    want = c.copy()
    want[off:off + n] = (stores[0] + stores[1]).astype(dtype).reshape(-1)
    assert_bit_equal(out.storage_numpy(), want, "%s %s +%d" % (kind, sizes, off))


@pytest.fixture(params=["as planned", "64-bit offsets", "three workgroups"])
def engine(request, thc):
    """The tile loop as launched, with 64-bit offsets, and with a grid that makes a workgroup take many tiles."""
    thc.set_tuning("apply.tiled.fuse_q", 2)      # (wherever the layout allows it)
    if request.param == "64-bit offsets":
        thc.force_64bit_index(True)
    if request.param == "three workgroups":
        thc.set_tuning("apply.tiled.max_grid", 3)
    yield request.param
    thc.force_64bit_index(False)
    thc.set_tuning("apply.tiled.max_grid", 1 << 22)
    thc.set_tuning("apply.tiled.fuse_q", 1)


@pytest.mark.parametrize("kind,dtype", [("float", np.float32), ("double", np.float64), ("long", np.int64)])
def test_three_and_four_fused_dims_and_a_batch(thc, engine, kind, dtype):
    for sizes, order in (((13, 5, 7, 11), (3, 2, 1, 0)), ((67, 3, 5, 9), (3, 2, 1, 0)), ((9, 3, 5, 2, 11), (4, 3, 2, 1, 0)),
                         ((9, 3, 2, 5, 3, 13), (5, 4, 3, 2, 1, 0)),            # a fifth column dim: batches
                         ((3, 65, 4, 43), (0, 3, 2, 1)),                       # the slowest dim in place: batches
                         ((200, 35, 77), (2, 1, 0)), ((131, 129, 9), (2, 1, 0))):   # 64 tiles and more: dealt to the XCDs
        dense = tuple(range(len(sizes)))
        for off in (0, 1):
            _check(thc, kind, dtype, sizes, order, dense, off, "tiled-ragged-fused", len(sizes) * 100 + off)


@pytest.mark.parametrize("kind,dtype", [("double", np.float64), ("long", np.int64)])
def test_two_reversed_operands(thc, engine, kind, dtype):
    """Two staged operands of 8 bytes, whose column offsets differ."""
    for sizes, a, b in (((33, 5, 19), (2, 1, 0), (2, 1, 0)), ((35, 4, 21), (2, 1, 0), (1, 2, 0)),
                        ((97, 31, 45), (1, 2, 0), (2, 1, 0)), ((13, 5, 7, 11), (3, 2, 1, 0), (2, 3, 1, 0))):
        for off in (0, 1):
            _check(thc, kind, dtype, sizes, a, b, off, "tiled-ragged-fused", sum(sizes) + off)


def test_a_gap_behind_the_rows_keeps_the_dims_apart(thc):
    """Columns of a wider output: its inner dims are no run."""
    x, y, z = 33, 5, 19
    rng = np.random.default_rng(7)
    a, b = (rng.integers(-8, 9, x * y * z).astype(np.float32) for _ in range(2))
    c = np.full(x * y * (z + 2), 5, np.float32)
    ta = thc.Tensor.from_storage(a, 0, (x, y, z), (1, x, x * y))
    tb = thc.Tensor.from_storage(np.pad(b.reshape(x, y, z), ((0, 0), (0, 0), (0, 2))).reshape(-1), 0, (x, y, z), (y * (z + 2), z + 2, 1))
    tc = thc.Tensor.from_storage(c, 0, (x, y, z), (y * (z + 2), z + 2, 1))
    tc.cadd(ta, 1, tb)
    assert thc.last_kernel() == "tiled-ragged", thc.last_kernel()
    want = c.reshape(x, y, z + 2).copy()
    want[:, :, :z] = a.reshape(z, y, x).transpose(2, 1, 0) + b.reshape(x, y, z)
    assert_bit_equal(tc.storage_numpy(), want.reshape(-1))


@pytest.mark.parametrize("forced64", [False, True])
def test_halves_fuse_their_columns_where_one_dim_leaves_tiles_empty(thc, forced64):
    """Halves take the line-cut tiles (64 x 256, whose columns start up to 63 early) over fused columns only: sizes around those
    extents, one staged operand in either place and copies, offsets off the grid, and larger tensors without the knob."""
    thc.force_64bit_index(forced64)
    thc.set_tuning("apply.tiled.fuse_half_min", 0)
    try:
        for seed, sizes in enumerate(((65, 3, 43), (63, 129, 9), (9, 7, 8), (127, 5, 51), (33, 65, 17), (130, 31, 11), (16, 257, 101))):
            for off in (0, 1, 3):
                for a_order, b_order in (((2, 1, 0), (0, 1, 2)), ((0, 1, 2), (2, 1, 0))):
                    _check(thc, "half", np.float16, sizes, a_order, b_order, off, "tiled-ragged-fused", seed)
    finally:
        thc.set_tuning("apply.tiled.fuse_half_min", 1 << 17)
        thc.force_64bit_index(False)
    _check(thc, "half", np.float16, (301, 67, 47), (2, 1, 0), (0, 1, 2), 1, "tiled-ragged-fused", 77)
    _check(thc, "half", np.float16, (301, 17, 241), (2, 1, 0), (0, 1, 2), 1, "tiled-shift", 78)      # (rows that fill their tiles)
    x = np.random.default_rng(5).integers(0, 9, 201 * 33 * 47).astype(np.float16)
    src = thc.Tensor.from_numpy(x).view_as_strided(0, (201, 33, 47), (1, 201, 201 * 33))
    got = thc.Tensor("half").resize((201, 33, 47)).copy(src)
    assert thc.last_kernel() == "tiled-ragged-fused"
    assert_bit_equal(got.numpy(), np.ascontiguousarray(x.reshape(47, 33, 201).transpose(2, 1, 0)))
