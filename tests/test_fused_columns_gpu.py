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
        assert thc.last_kernel().startswith("tiled"), thc.last_kernel()
        want = c.copy()
        want[off:off + n] = (a[off:off + n].reshape(z, y, x).transpose(2, 1, 0).reshape(-1).astype(np.float64)
                             + b[off:off + n]).astype(dtype)
        assert_bit_equal(tc.storage_numpy(), want, "%s %s +%d" % (kind, (x, y, z), off))
