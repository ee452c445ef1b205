"""Whole-tensor reductions whose last workgroup folds the partials of the others: one workgroup, which hands nothing
over, two, as many as there are, and some between; every accumulator width, repeated so that an
older launch's partials would show."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,dtype", [("float", np.float32), ("half", np.float16), ("double", np.float64),
                                        ("int", np.int32), ("byte", np.uint8), ("long", np.int64)])
def test_sums_and_extremes_around_the_workgroup_counts(thc, kind, dtype):
    batch = 256 * 8 * (16 // np.dtype(dtype).itemsize)      # elements of one workgroup's full batch
    rng = np.random.default_rng(41)
    for blocks in (1, 2, 15, 16, 17, 33, 512):
        for n in (blocks * batch - 1, blocks * batch, blocks * batch + 1):
            x = rng.integers(0, 3, n).astype(dtype)
            x[n // 2] = 7
            t = thc.Tensor.from_numpy(x)
            for _ in range(2):
                assert t.sumall() == float(x.astype(np.int64).sum()), (kind, n)
                assert t.maxall() == 7, (kind, n)


@pytest.mark.parametrize("kind,dtype", [("float", np.float32), ("double", np.float64)])
def test_moments_around_the_workgroup_counts(thc, kind, dtype):
    batch = 256 * 8 * (16 // np.dtype(dtype).itemsize)
    rng = np.random.default_rng(43)
    # Welford's recurrence per lane (at most a few hundred steps here) and pairwise merges: a few dozen roundings
    tol = 64 * np.finfo(dtype).eps
    for n in (2, 255, batch - 1, batch + 1, 16 * batch + 5, 17 * batch, 300 * batch + 3):
        x = (rng.standard_normal(n) + 3).astype(dtype)
        t = thc.Tensor.from_numpy(x)
        want = x.astype(np.float64).var(ddof=1)
        for _ in range(2):
            assert abs(t.varall() - want) <= tol * want, (kind, n)


@pytest.mark.parametrize("rows,cols", [(67001, 10), (33000, 33), (200003, 3), (150000, 18)])
def test_var_of_tall_matrices_folds_in_one_workgroup_per_column_tile(thc, rows, cols):
    x = (np.random.default_rng(47).standard_normal((rows, cols)) + 2).astype(np.float32)
    got = thc.Tensor("float").var(thc.Tensor.from_numpy(x), 0).numpy().reshape(-1)
    assert thc.last_kernel() == "var-tall", thc.last_kernel()
    want = x.astype(np.float64).var(axis=0, ddof=1)
    assert np.all(np.abs(got - want) <= 64 * np.finfo(np.float32).eps * want)


@pytest.mark.parametrize("kind,dtype", [("float", np.float32), ("double", np.float64)])
def test_more_workgroups_than_the_handed_over_values_have_room_for(thc, kind, dtype):
    """Variances publish three values a workgroup, of two words each for doubles: their workgroups are held to the room there is,
    behind which the words of one-read scans lie (a scan afterwards meets none of theirs)."""
    cus = thc.lib().THCAmd_getNumComputeUnits(thc.state())
    n = 9 * cus * 256 * 8 * (16 // np.dtype(dtype).itemsize) + 5
    x = (np.arange(n) % 3 == 0).astype(dtype)
    t = thc.Tensor.from_numpy(x)
    want, sums = x.astype(np.float64).var(ddof=1), np.cumsum(x, dtype=np.float64)
    for per_cu in (2, 3, 4, 5, 8):
        thc.set_tuning("reduce.all.blocks_per_cu", per_cu)
        try:
            for _ in range(2):
                assert abs(t.varall() - want) <= 64 * np.finfo(dtype).eps * want, per_cu
                assert t.sumall() == x.sum(dtype=np.float64), per_cu
                if sums[-1] < 2 ** 24 or kind == "double":
                    assert np.array_equal(thc.Tensor(kind).cumsum(t, 0).numpy(), sums.astype(dtype)), per_cu
        finally:
            thc.set_tuning("reduce.all.blocks_per_cu", 2)
