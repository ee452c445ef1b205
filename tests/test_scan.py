"""cumsum / cumprod (lib/THC/generic/THCTensorMathScan.cu:76-126). Oracle
pinned against numpy.cumsum/cumprod in float64 (and bit-exactly on
integer-valued data); HIP path against the oracle: integer-valued data
bit-exact, random data within 1e-5 of the running mass."""
import ctypes
import os
import subprocess
import threading

import numpy as np
import pytest

from tests.util import assert_bit_equal, contiguous_geometry, fill_storage, random_geometry


@pytest.mark.parametrize("seed", range(6))
def test_oracle_scan_matches_numpy(oracle, seed):
    rng = np.random.default_rng(seed)
    nd = int(rng.integers(1, 4))
    shape = tuple(int(x) for x in rng.integers(1, 9, nd))
    dim = int(rng.integers(0, nd))
    n, off, size, stride = random_geometry(rng, shape)
    st = fill_storage(rng, n, dist="uniform")
    src = oracle.View(st, off, size, stride)
    x = src.numpy().astype(np.float64)
    np.testing.assert_allclose(oracle.scan_dim(src, dim).numpy(), np.cumsum(x, axis=dim), rtol=1e-6, atol=1e-6)
    np.testing.assert_allclose(oracle.scan_dim(src, dim, product=True).numpy(), np.cumprod(x, axis=dim),
                               rtol=1e-6, atol=1e-30)
    xi = rng.integers(-9, 10, shape).astype(np.float32)
    assert_bit_equal(oracle.scan_dim(oracle.View.of(xi), dim).numpy(), np.cumsum(xi.astype(np.int64), axis=dim).astype(np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half"])
def test_gpu_scan_of_small_slices_goes_through_lds(thc, oracle, kind):
    """Short rows and small R x inner slices are scanned in LDS by a thread per
    column; input and output runs may sit at different misalignments."""
    rng = np.random.default_rng(18)
    dtype = np.float32 if kind == "float" else np.float16
    for shape, dim in (((5000, 10), 1), ((777, 33), 1), ((300, 8, 16), 1), ((1000, 33, 2), 1), ((41, 7), 0),
                       ((2, 3, 5, 7), 2), ((3, 500), 1), ((9, 1, 4), 1), ((1, 60, 60), 1)):
        n = int(np.prod(shape))
        for off in (0, 1, 3):
            st = [1] * len(shape)
            for d in range(len(shape) - 2, -1, -1):
                st[d] = st[d + 1] * shape[d + 1]
            x = rng.integers(-4, 5, n + off).astype(dtype)
            dev = thc.Tensor.from_storage(x, off, shape, tuple(st), kind=kind)
            got = thc.Tensor(kind).cumsum(dev, dim)
            assert thc.last_kernel() == "scan-slab", (shape, dim, thc.last_kernel())
            want = np.cumsum(x[off:].reshape(shape).astype(np.int64), axis=dim).astype(dtype)   # exact: small integers
            assert_bit_equal(got.numpy(), want, "%s %d off %d" % (shape, dim, off))
            dev.cumsum(dev, dim)                                         # in place, misaligned output
            assert_bit_equal(dev.numpy(), want)
            assert_bit_equal(dev.storage_numpy()[:off], x[:off])       # nothing written before the run
    thc.set_tuning("scan.slab", 0)
    try:
        x = rng.integers(-4, 5, (777, 33)).astype(dtype)
        got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), 1)
        assert thc.last_kernel() == "scan-rows"
        assert_bit_equal(got.numpy(), np.cumsum(x.astype(np.int64), axis=1).astype(dtype))
    finally:
        thc.set_tuning("scan.slab", 1)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half", "int", "double"])
def test_gpu_long_scans_with_few_columns_run_in_chunks(thc, oracle, kind):
    """A scan that would occupy a handful of workgroups is cut into chunks of
    rows: chunk totals, their scan (recursively, here down to three levels with
    small chunks), then every chunk scans from its carry. Exact on small integers."""
    rng = np.random.default_rng(19)
    dtype = {"float": np.float32, "half": np.float16, "int": np.int32, "double": np.float64}[kind]
    for shape, dim, chunk in (((200000, 10), 0, 32768), ((3, 70001), 1, 32768), ((2, 50000, 7), 1, 32768),
                              ((1, 5000, 136), 1, 32768), ((100003, 3), 0, 512), ((2, 40000), 1, 256)):
        sparse = (rng.integers(0, 50, shape) == 0) * rng.integers(-2, 3, shape)     # running sums fit half
        x = sparse.astype(dtype)
        thc.set_tuning("scan.chunk_bytes", chunk)
        thc.set_tuning("scan.cols.split", 0)     # (wide rows would take the split column kernel,
        thc.set_tuning("scan.rows.split", 0)     #  long rows a wave per piece)
        try:
            got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), dim)
            assert thc.last_kernel() == "scan-chunked", (shape, thc.last_kernel())
            results = [got]
            if kind in ("float", "half"):
                # the one-read form with look-back (off by default: slower), as it is and with readers
                # that never wait (a word that is still empty is computed by the reader itself)
                thc.set_tuning("scan.lookback", 1)
                for spin in (4096, 0):
                    thc.set_tuning("scan.lookback_spin", spin)
                    results.append(thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), dim))
                    assert thc.last_kernel() == "scan-lookback", (shape, thc.last_kernel())
                # in place: the two-read form (a reader that gives up waiting would need another chunk's input)
                same = thc.Tensor.from_numpy(x)
                same.cumsum(same, dim)
                assert thc.last_kernel() == "scan-chunked"
                results.append(same)
        finally:
            thc.set_tuning("scan.chunk_bytes", 32768)
            thc.set_tuning("scan.cols.split", 1)
            thc.set_tuning("scan.rows.split", 1)
            thc.set_tuning("scan.lookback", 0)
            thc.set_tuning("scan.lookback_spin", 4096)
        want = np.cumsum(sparse, axis=dim)
        assert np.abs(want).max() < 2048
        for r in results:
            assert_bit_equal(r.numpy(), want.astype(dtype), "%s %s" % (kind, shape))
    rows, every = (150000, 1000) if kind == "double" else (40000, 2000)
    ones = np.ones((rows, 2), dtype)
    ones[::every] = 2
    thc.set_tuning("scan.strided", 0)        # (products of integers would be read once)
    got = thc.Tensor(kind).cumprod(thc.Tensor.from_numpy(ones), 0)
    thc.set_tuning("scan.strided", -1)
    assert thc.last_kernel() == "scan-chunked"
    want = np.cumprod(ones, axis=0, dtype=np.int64 if kind == "int" else np.float64)
    if kind == "half":
        assert_bit_equal(got.numpy()[:30000], want[:30000].astype(dtype))   # 2^15 still is a half
    else:
        assert_bit_equal(got.numpy(), want.astype(dtype))
    thc.set_tuning("scan.chunked", 0)
    thc.set_tuning("scan.rows.split", 0)
    try:
        x = rng.integers(-2, 3, (3, 70001)).astype(dtype)
        got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), 1)
        assert thc.last_kernel() == "scan-rows"
    finally:
        thc.set_tuning("scan.chunked", 1)
        thc.set_tuning("scan.rows.split", 1)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half", "int", "double", "byte", "long"])
def test_gpu_few_long_rows_scan_in_pieces(thc, oracle, kind):
    """A 1-D cumprod of floating elements (or a few long rows), and any scan of more chunks than the one-read form has
    room for (`scan.onepass` = 0 here), is cut into pieces that scan side by side, a wave per piece:
    totals of the pieces, their scan, then every piece from its carry. Exact on small integers and on products
    of -1, 2 and 0.5; row lengths that are and are not whole packs, storage offsets off the 16-byte grid, in place."""
    thc.set_tuning("scan.onepass", 0)
    try:
        _few_long_rows_in_pieces(thc, kind)
    finally:
        thc.set_tuning("scan.onepass", 1)


def _few_long_rows_in_pieces(thc, kind):
    rng = np.random.default_rng(29)
    dtype = {"float": np.float32, "half": np.float16, "int": np.int32, "double": np.float64, "byte": np.uint8,
             "long": np.int64}[kind]
    for shape, dim, off, iters in (((1 << 20,), 0, 0, 8), ((1000003,), 0, 0, 8), ((3, 300000), 1, 0, 8),
                                   ((2, 1, 70001), 2, 1, 2), ((5, 40960), 1, 3, 1), ((1, 123457), 1, 0, 1)):
        n = int(np.prod(shape))
        if kind == "byte":
            sparse = (rng.integers(0, 6000, n + off) == 0) * rng.integers(0, 2, n + off)
        else:
            sparse = (rng.integers(0, 600, n + off) == 0) * rng.integers(-2, 3, n + off)     # running sums fit half
        x = sparse.astype(dtype)
        strides = [1] * len(shape)
        for d in range(len(shape) - 2, -1, -1):
            strides[d] = strides[d + 1] * shape[d + 1]
        thc.set_tuning("scan.rows.split_min_iters", iters)
        try:
            dev = thc.Tensor.from_storage(x, off, shape, tuple(strides), kind=kind)
            got = thc.Tensor(kind).cumsum(dev, dim)
            assert thc.last_kernel() == "scan-rows-split", (shape, thc.last_kernel())
            dev.cumsum(dev, dim)
            assert thc.last_kernel() == "scan-rows-split"
        finally:
            thc.set_tuning("scan.rows.split_min_iters", 8)
        want = np.cumsum(sparse[off:].reshape(shape), axis=dim)
        assert np.abs(want).max() < (256 if kind == "byte" else 2048)
        assert_bit_equal(got.numpy(), want.astype(dtype), "%s %s" % (kind, shape))
        assert_bit_equal(dev.numpy(), want.astype(dtype), "%s %s in place" % (kind, shape))
        assert_bit_equal(dev.storage_numpy()[:off], x[:off])       # nothing written before the rows
        # products: every few hundred elements a factor 2, 0.5, 2, ... (floating types) or -1, so that all are exact
        at = np.flatnonzero(rng.integers(0, 300, n + off) == 0)
        f = np.ones(n + off, np.float64)
        f[at] = -1
        if kind in ("float", "half", "double"):
            for r in range(n // shape[dim]):           # (per row: each begins with a 2)
                mine = at[(at >= off + r * shape[dim]) & (at < off + (r + 1) * shape[dim])]
                f[mine[0::3]] = np.where(np.arange(len(mine[0::3])) % 2 == 0, 2, 0.5)
        x = f.astype(np.int64).astype(dtype) if kind not in ("float", "half", "double") else f.astype(dtype)
        want = np.cumprod(f[off:].reshape(shape), axis=dim)
        want = want.astype(np.int64).astype(dtype) if kind not in ("float", "half", "double") else want.astype(dtype)
        thc.set_tuning("scan.rows.split_min_iters", iters)
        try:
            dev = thc.Tensor.from_storage(x, off, shape, tuple(strides), kind=kind)
            got = thc.Tensor(kind).cumprod(dev, dim)
            assert thc.last_kernel() == "scan-rows-split", (shape, thc.last_kernel())
            dev.cumprod(dev, dim)
            assert thc.last_kernel() == "scan-rows-split"
        finally:
            thc.set_tuning("scan.rows.split_min_iters", 8)
        assert_bit_equal(got.numpy(), want, "%s %s product" % (kind, shape))
        assert_bit_equal(dev.numpy(), want, "%s %s product in place" % (kind, shape))
        assert_bit_equal(dev.storage_numpy()[:off], x[:off])
    if kind != "byte":
        ones = np.ones((2, 100000), dtype)
        ones[:, ::9000] = 2
        ones[1, 5::17000] = -1
        got = thc.Tensor(kind).cumprod(thc.Tensor.from_numpy(ones), 1)
        assert thc.last_kernel() == "scan-rows-split"
        assert_bit_equal(got.numpy(), np.cumprod(ones.astype(np.float64), axis=1).astype(dtype))
    if kind in ("float", "double"):
        x = rng.standard_normal(3000001).astype(dtype)
        got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), 0).numpy().astype(np.float64)
        assert thc.last_kernel() == "scan-rows-split"
        want = np.cumsum(x.astype(np.float64))
        mass = np.cumsum(np.abs(x.astype(np.float64)))
        assert np.all(np.abs(got - want) <= 1e-5 * np.maximum(np.abs(want), mass / 64))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half", "int", "double", "byte", "long"])
def test_gpu_long_scans_over_wide_rows_split_the_rows(thc, oracle, kind):
    """A long scan over rows wide enough for the column kernel's lanes, but with too few column tiles
    for the chip, cuts the rows into parts that scan side by side: totals of the parts, their scan,
    then every part from its carry. Exact on small integers; row counts that leave a short last
    part, widths that are and are not whole packs, several slices, in place."""
    rng = np.random.default_rng(23)
    dtype = {"float": np.float32, "half": np.float16, "int": np.int32, "double": np.float64, "byte": np.uint8,
             "long": np.int64}[kind]
    for shape, dim, min_rows in (((20000, 1000), 0, 256), ((3, 9001, 136), 1, 256), ((1, 30011, 257), 1, 256),
                                 ((2, 4099, 64), 1, 64), ((1500, 2000), 0, 64), ((70001, 100), 0, 256)):
        if kind == "byte":
            sparse = (rng.integers(0, 400, shape) == 0) * rng.integers(0, 2, shape)
        else:
            sparse = (rng.integers(0, 50, shape) == 0) * rng.integers(-2, 3, shape)     # running sums fit half
        x = sparse.astype(dtype)
        thc.set_tuning("scan.cols.split_min_rows", min_rows)
        thc.set_tuning("scan.cols.split_min_row_bytes", 1)      # (narrower rows are scanned in chunks by default,
        thc.set_tuning("scan.chunked", 0)                       #  and so are rows that are not whole packs)
        try:
            got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), dim)
            assert thc.last_kernel() == "scan-cols-split", (shape, thc.last_kernel())
            same = thc.Tensor.from_numpy(x)
            same.cumsum(same, dim)
            assert thc.last_kernel() == "scan-cols-split"
        finally:
            thc.set_tuning("scan.cols.split_min_rows", 256)
            thc.set_tuning("scan.cols.split_min_row_bytes", 256)
            thc.set_tuning("scan.chunked", 1)
        want = np.cumsum(sparse, axis=dim)
        assert np.abs(want).max() < (256 if kind == "byte" else 2048)
        assert_bit_equal(got.numpy(), want.astype(dtype), "%s %s" % (kind, shape))
        assert_bit_equal(same.numpy(), want.astype(dtype), "%s %s in place" % (kind, shape))
    if kind != "byte":
        ones = np.ones((9000, 320), dtype)
        ones[::700] = 2
        ones[1::1300, ::7] = -1
        thc.set_tuning("scan.strided", 0)    # (products of integers would be read once)
        got = thc.Tensor(kind).cumprod(thc.Tensor.from_numpy(ones), 0)
        thc.set_tuning("scan.strided", -1)
        assert thc.last_kernel() == "scan-cols-split"
        assert_bit_equal(got.numpy(), np.cumprod(ones.astype(np.float64), axis=0).astype(dtype))
    if kind in ("float", "double"):
        x = rng.standard_normal((50000, 520)).astype(dtype)
        dev, ref = thc.Tensor.from_numpy(x), oracle.View.of(x)
        thc.set_tuning("scan.strided", 0)
        got = thc.Tensor(kind).cumsum(dev, 0).numpy().astype(np.float64)
        thc.set_tuning("scan.strided", -1)
        assert thc.last_kernel() == "scan-cols-split"
        want = oracle.scan_dim(ref, 0).numpy().astype(np.float64) if kind == "float" else np.cumsum(x, axis=0)
        mass = np.cumsum(np.abs(x.astype(np.float64)), axis=0)
        assert np.all(np.abs(got - want) <= 1e-5 * np.maximum(np.abs(want), mass / 64))
    thc.set_tuning("scan.cols.split", 0)
    try:
        x = ((rng.integers(0, 50, (20000, 1000)) == 0) * 1).astype(dtype)
        got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), 0)
        assert thc.last_kernel() in ("scan-cols", "scan-chunked")
        assert_bit_equal(got.numpy(), np.cumsum(x.astype(np.int64), axis=0).astype(dtype))
    finally:
        thc.set_tuning("scan.cols.split", 1)


@pytest.mark.gpu
@pytest.mark.parametrize("slab", [1, 0])
@pytest.mark.parametrize("kind", ["float", "half"])
def test_gpu_scan(thc, oracle, kind, slab):
    thc.set_tuning("scan.slab", slab)
    try:
        _gpu_scan_cases(thc, oracle, kind)
    finally:
        thc.set_tuning("scan.slab", 1)


def _gpu_scan_cases(thc, oracle, kind):
    rng = np.random.default_rng(17)
    dtype = np.float32 if kind == "float" else np.float16
    tol = 1e-5 if kind == "float" else 2e-3
    for shape, dim in (((7, 1000), 1), ((3, 257), 1), ((300, 5), 1), ((50, 64), 0), ((4, 33, 20), 1),
                       ((2, 3, 4, 130), 3), ((1,), 0), ((9000,), 0), ((6, 5, 1), 1), ((2, 1000, 24), 1),
                       ((3, 300, 7), 1), ((1, 5000, 136), 1), ((700, 2), 0), ((5, 2049), 1), ((2, 130, 8, 16), 1)):
        geom = random_geometry(rng, shape) if len(shape) == 3 else contiguous_geometry(shape)
        st = rng.uniform(-1, 1, geom[0]).astype(dtype)
        dev = thc.Tensor.from_storage(st, *geom[1:], kind=kind)
        ref = oracle.View(st.copy(), *geom[1:])
        got = thc.Tensor(kind).cumsum(dev, dim)
        assert got.shape == tuple(shape)
        want = oracle.scan_dim(ref, dim).numpy().astype(np.float64)
        mass = np.cumsum(np.abs(ref.numpy().astype(np.float64)), axis=dim)
        err = np.abs(got.numpy().astype(np.float64) - want) / np.maximum(np.abs(want), mass * 2.0 ** -6 + 1e-30)
        assert err.max() <= tol, (shape, dim, err.max())
        stp = rng.uniform(0.9, 1.1, geom[0]).astype(dtype)
        devp = thc.Tensor.from_storage(stp, *geom[1:], kind=kind)
        gotp = thc.Tensor(kind).cumprod(devp, dim).numpy().astype(np.float64)
        wantp = oracle.scan_dim(oracle.View(stp.copy(), *geom[1:]), dim, product=True).numpy().astype(np.float64)
        # (one step of half's subnormal grid where a product has decayed that far)
        np.testing.assert_allclose(gotp, wantp, rtol=max(tol, 2e-5) * 4, atol=6e-8 if kind == "half" else 0)
    xi = rng.integers(-9, 10, (37, 700)).astype(np.float32)
    for dim in (0, 1):
        got = thc.Tensor("float").cumsum(thc.Tensor.from_numpy(xi), dim)
        assert_bit_equal(got.numpy(), np.cumsum(xi.astype(np.int64), axis=dim).astype(np.float32))
    t = thc.Tensor.from_numpy(xi)
    t.cumsum(t, 1)                                               # in place
    assert_bit_equal(t.numpy(), np.cumsum(xi.astype(np.int64), axis=1).astype(np.float32))
    with pytest.raises(thc.THCError, match="out of range"):
        thc.Tensor("float").cumsum(thc.Tensor.from_numpy(xi), 2)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half", "int", "double"])
def test_gpu_scan_over_a_strided_dim_in_every_strip_width(thc, oracle, kind):
    """The scan over a non-innermost dim picks a strip width (8-64 lanes) and whether the next
    segment's packs are requested ahead from the shape and the chip; here each is forced in turn.
    Small integers: exact whatever the split; row counts off the segment size; an odd inner size
    takes the element-wise variant."""
    rng = np.random.default_rng(23)
    dtype = {"float": np.float32, "half": np.float16, "int": np.int32, "double": np.float64}[kind]
    thc.set_tuning("scan.chunked", 0)       # (few long slices would otherwise be cut into chunks of rows,
    thc.set_tuning("scan.slab", 0)          #  small ones scanned in LDS,
    thc.set_tuning("scan.cols.split", 0)    #  long ones over wide rows cut into parts of rows)
    try:
        for shape in ((3, 300, 520), (2, 129, 1024), (1, 64, 96), (2, 1000, 136), (1, 77, 515), (5, 1, 8192), (4, 9, 4100)):
            sparse = (rng.integers(0, 12, shape) == 0) * rng.integers(-2, 3, shape)
            x = thc.Tensor.from_numpy(sparse.astype(dtype))
            want = np.cumsum(sparse, axis=1)
            assert np.abs(want).max() < 2048
            for pf in (0, 1):
                for tx in (8, 16, 32, 64):
                    thc.set_tuning("scan.cols.prefetch", pf)
                    thc.set_tuning("scan.cols.min_tx", tx)
                    thc.set_tuning("scan.cols.max_tx", tx)
                    got = thc.Tensor(kind).cumsum(x, 1)
                    assert thc.last_kernel() == "scan-cols", (shape, thc.last_kernel())
                    assert_bit_equal(got.numpy(), want.astype(dtype), "%s %s pf=%d tx=%d" % (kind, shape, pf, tx))
    finally:
        thc.set_tuning("scan.chunked", 1)
        thc.set_tuning("scan.slab", 1)
        thc.set_tuning("scan.cols.split", 1)
        thc.set_tuning("scan.cols.prefetch", -1)
        thc.set_tuning("scan.cols.min_tx", 8)
        thc.set_tuning("scan.cols.max_tx", 64)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half", "int", "double", "byte", "long"])
def test_gpu_one_read_scans_at_the_edges_of_their_chunks(thc, kind):
    """Rows of 4096 elements and more are cut into chunks of 256, 512 or 1024 threads x 8 packs: lengths one
    below, at and one above every chunk and every group of 64 chunks, rows and offsets off the 16-byte
    grid. Exact on small integers; a NaN reaches everything behind it and nothing before."""
    dtype = {"float": np.float32, "half": np.float16, "int": np.int32, "double": np.float64, "byte": np.uint8,
             "long": np.int64}[kind]
    unit = 16 // np.dtype(dtype).itemsize * 8
    rng = np.random.default_rng(31)
    sizes = [4096, 4097] + [n + d for n in (256 * unit, 512 * unit, 1024 * unit, 64 * 512 * unit) for d in (-1, 0, 1) if n + d >= 4096]
    for n in sizes:
        for rows, off in ((1, 0), (3, 1)):
            every = 6000 if kind == "byte" else 600
            x = ((rng.integers(0, every, rows * n + off) == 0) * rng.integers(0 if kind == "byte" else -2, 3, rows * n + off)).astype(dtype)
            dev = thc.Tensor.from_storage(x, off, (rows, n), (n, 1), kind=kind)
            got = thc.Tensor(kind).cumsum(dev, 1)
            assert thc.last_kernel() == "scan-onepass", (n, thc.last_kernel())
            want = np.cumsum(x[off:].reshape(rows, n).astype(np.int64), axis=1)
            assert kind not in ("half", "float") or np.abs(want).max() < 2048
            assert_bit_equal(got.numpy(), want.astype(dtype), "%s %d x %d" % (kind, rows, n))
    if kind in ("float", "half", "double"):
        n = 64 * 512 * unit + 5
        for at in (0, 4097, 512 * unit, n - 1):
            x = np.zeros(n, dtype)
            x[::5000] = 1
            want = np.cumsum(x.astype(np.float64)).astype(dtype)
            x[at] = want[at:] = np.nan
            assert_bit_equal(thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), 0).numpy(), want, "%s NaN at %d" % (kind, at))
    if kind in ("float", "double"):
        x = rng.standard_normal(3000001).astype(dtype)
        got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), 0).numpy().astype(np.float64)
        assert thc.last_kernel() == "scan-onepass"
        want, mass = np.cumsum(x.astype(np.float64)), np.cumsum(np.abs(x.astype(np.float64)))
        assert np.all(np.abs(got - want) <= 1e-5 * np.maximum(np.abs(want), mass / 64))


@pytest.mark.gpu
def test_gpu_one_read_scan_beyond_4096_chunks(thc):
    """More than 64 x 64 chunks in a row: the third level of published totals."""
    n = 4097 * 1024 * 32 + 3
    x = (np.arange(n, dtype=np.int32) % 7) - 2
    got = thc.Tensor("int").cumsum(thc.Tensor.from_numpy(x), 0)
    assert thc.last_kernel() == "scan-onepass"
    assert_bit_equal(got.numpy(), np.cumsum(x, dtype=np.int32))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["byte", "char", "half", "short"])
def test_gpu_rows_that_end_early_in_a_chunk(thc, kind):
    """Rows of 1- and 2-byte elements that fill a part of a chunk's waves: the segments (64 packs) behind a
    row's end are left alone. Row ends at, around and between segments, in the first wave and in a later one, rows on
    and off the 16-byte grid; whole storages are compared. Many short aligned rows of bytes stay a wave per row."""
    dtype = {"byte": np.uint8, "char": np.int8, "half": np.float16, "short": np.int16}[kind]
    seg = 64 * 16 // np.dtype(dtype).itemsize
    rng = np.random.default_rng(43)
    for n in (4096, 4096 + seg - 1, 4096 + seg, 4096 + seg + 1, 8 * seg - 1, 8 * seg + 1, 13 * seg + 5, 24 * seg, 31 * seg + 3):
        for rows, off in ((1, 0), (5, 3)):
            x = ((rng.integers(0, 200, rows * n + off) == 0) * 1).astype(dtype)
            dev = thc.Tensor.from_storage(x, off, (rows, n), (n, 1), kind=kind)
            out = thc.Tensor.from_storage(np.full(rows * n + off + 40, 7, dtype), off, (rows, n), (n, 1), kind=kind)
            out.cumsum(dev, 1)
            got, want = out.storage_numpy(), np.full(rows * n + off + 40, 7, dtype)
            want[off:off + rows * n] = np.cumsum(x[off:].reshape(rows, n).astype(np.int64), axis=1).astype(dtype).reshape(-1)
            assert_bit_equal(got, want, "%s %d x %d" % (kind, rows, n))
    cus = thc.lib().THCAmd_getNumComputeUnits(thc.state())
    for rows, n in ((4 * cus + 1, 4096), (4 * cus, 4096), (4 * cus + 1, 4100), (4 * cus + 1, 8192)):
        x = (rng.integers(0, 400, (rows, n)) == 0).astype(dtype)
        got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), 1)
        assert (thc.last_kernel() == "scan-rows") == (np.dtype(dtype).itemsize == 1 and rows > 4 * cus and n == 4096), (rows, n)
        assert_bit_equal(got.numpy(), np.cumsum(x, axis=1, dtype=np.int64).astype(dtype))


@pytest.mark.gpu
def test_gpu_one_read_scans_of_two_threads_on_one_stream_stay_in_their_tensors(thc):
    """Two host threads on the default stream: their launches interleave, and each scan is one launch whose words and ticket belong
    to scans alone. Both threads' calls end, nothing outside the outputs is written, and the next scans are right."""
    rng = np.random.default_rng(37)
    guard, jobs = 64, []
    for kind, dtype, rows, n in (("float", np.float32, 3, 70001), ("long", np.int64, 2, 40003), ("byte", np.uint8, 1, 900001),
                                 ("double", np.float64, 1, 300007)):
        x = (rng.integers(0, 600, (rows, n)) == 0).astype(dtype)
        out = thc.Tensor.from_storage(np.full(rows * n + 2 * guard, 5, dtype), guard, (rows, n), (n, 1), kind=kind)
        jobs.append((thc.Tensor.from_numpy(x), out, x, dtype))
    failed = []

    def work(mine):
        try:
            for i in range(100):
                for src, out, _, _ in mine:
                    out.cumsum(src, 1)
        except Exception as e:                        # reported by the main thread
            failed.append(e)

    threads = [threading.Thread(target=work, args=(jobs[i::2],)) for i in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed, failed
    for src, out, x, dtype in jobs:
        out.cumsum(src, 1)
        got = out.storage_numpy()
        assert np.all(got[:guard] == 5) and np.all(got[-guard:] == 5)
        assert_bit_equal(got[guard:-guard].reshape(x.shape), np.cumsum(x, axis=1, dtype=np.int64).astype(dtype))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half", "int", "double", "byte", "long"])
def test_gpu_one_read_scans_along_a_strided_dim(thc, kind):
    """Strips of columns (1) and runs of whole narrow rows (2), each forced on shapes at their edges: rows one below, at
    and one above a chunk and a group of chunks, more than two levels of groups, widths of one pack, one element
    more, and of packs that leave a strip one pack; offsets off the 16-byte grid, in place; whole storages
    are compared. Exact on small integers."""
    dtype = {"float": np.float32, "half": np.float16, "int": np.int32, "double": np.float64, "byte": np.uint8, "long": np.int64}[kind]
    vec = 16 // np.dtype(dtype).itemsize
    rng = np.random.default_rng(47)
    lanes = 128 // vec if vec < 16 else 8
    lanes = min(max(lanes, 8), 32)
    shapes = [(1, 512 // lanes * 8 * n + d, lanes * vec) for n in (1, 4) for d in (-1, 0, 1)]          # chunks and groups of four
    shapes += [(2, 70, vec), (1, 4099, vec + 1), (3, 200, 33 * vec - 1), (2, 515, 97 * vec + 1), (2, 33, 1000), (7, 1, 40),
               (1, 160000, vec), (1, 20011, 3), (40, 33, 7), (1, 300001, 2)]
    for shape in shapes:
        outer, n, inner = shape
        off = int(rng.integers(0, 4))
        every = max(24, n // 100)
        x = ((rng.integers(0, every, outer * n * inner + off + 9) == 0) * rng.integers(0 if kind == "byte" else -2, 3, outer * n * inner + off + 9)).astype(dtype)
        size = outer * n * inner
        want = np.cumsum(x[off:off + size].reshape(shape).astype(np.int64), axis=1)
        assert kind != "half" or np.abs(want).max() < 2048
        whole = x.copy()
        whole[off:off + size] = want.astype(dtype).reshape(-1)
        for form, name in ((1, "scan-cols-split"), (2, "scan-chunked")):
            if form == 1 and inner < vec or form == 2 and inner * np.dtype(dtype).itemsize > 8192:
                continue
            thc.set_tuning("scan.strided", form)
            thc.set_tuning("scan.strided_two_reads", 0)      # (the forms of two reads have the same names)
            thc.set_tuning("scan.slab", 0)
            try:
                strides = (n * inner, inner, 1)
                dev = thc.Tensor.from_storage(x, off, shape, strides, kind=kind)
                out = thc.Tensor.from_storage(x, off, shape, strides, kind=kind)
                out.cumsum(dev, 1)
                if n > 1:
                    assert thc.last_kernel() == name, (shape, form, thc.last_kernel())
                dev.cumsum(dev, 1)
            finally:
                thc.set_tuning("scan.strided", -1)
                thc.set_tuning("scan.strided_two_reads", 1)
                thc.set_tuning("scan.slab", 1)
            assert_bit_equal(out.storage_numpy(), whole, "%s %s form %d" % (kind, shape, form))
            assert_bit_equal(dev.storage_numpy(), whole, "%s %s form %d in place" % (kind, shape, form))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half", "double"])
def test_gpu_strided_one_read_scans_of_random_values_and_of_nans(thc, kind):
    """Against float64 sums, with a NaN that reaches what lies behind it in its column and nothing else; the same bits on
    every run."""
    dtype = {"float": np.float32, "half": np.float16, "double": np.float64}[kind]
    rng = np.random.default_rng(53)
    for shape in ((1, 3001, 257), (3, 1000, 130), (1, 40001, 5), (2, 9001, 11)):
        x = rng.uniform(-1, 1, shape).astype(dtype)
        dev = thc.Tensor.from_numpy(x)
        first = thc.Tensor(kind).cumsum(dev, 1).numpy()
        want, mass = np.cumsum(x.astype(np.float64), axis=1), np.cumsum(np.abs(x.astype(np.float64)), axis=1)
        # (half: one rounding of the result beside the float sums')
        tol = {"float": 1e-5, "half": 2e-3, "double": 1e-12}[kind]
        assert np.all(np.abs(first.astype(np.float64) - want) <= tol * np.maximum(np.abs(want), mass / 64)), shape
        assert_bit_equal(thc.Tensor(kind).cumsum(dev, 1).numpy(), first)
        at, col = shape[1] // 2 + 3, shape[2] - 2
        x[0, at, col] = np.nan
        got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), 1).numpy()
        assert np.all(np.isnan(got[0, at:, col]))
        got[0, at:, col] = first[0, at:, col]
        assert_bit_equal(got, first, "%s %s" % (kind, shape))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "half", "double", "byte", "int"])
def test_gpu_rows_below_4096_elements_in_one_chunk(thc, kind):
    """Rows that are not whole packs from 2 KiB on, and few rows that are: a workgroup per row; row ends at and around the
    64-pack segments and the widths of a workgroup, and row counts on both sides of where a wave per row takes over."""
    dtype = {"float": np.float32, "half": np.float16, "double": np.float64, "byte": np.uint8, "int": np.int32}[kind]
    item = np.dtype(dtype).itemsize
    seg = 64 * 16 // item
    cus = thc.lib().THCAmd_getNumComputeUnits(thc.state())
    rng = np.random.default_rng(59)
    for n in [m for m in (2048 // item, 2048 // item + 1, 3 * seg + 1, 2047, 2048, 2049, 3 * seg - 1, 4095) if m * item >= 2048]:
        for rows, off in ((1, 1), (5, 0), (cus, 0), (12 * cus + 1, 0)):
            if rows > cus and n > 2100:
                continue
            x = (rng.integers(0, 300, rows * n + off) == 0).astype(dtype)
            dev = thc.Tensor.from_storage(x, off, (rows, n), (n, 1), kind=kind)
            got = thc.Tensor(kind).cumsum(dev, 1)
            if rows <= cus and (off or n % (16 // item)):
                assert thc.last_kernel() == "scan-onepass", (n, rows, thc.last_kernel())
            assert_bit_equal(got.numpy(), np.cumsum(x[off:].reshape(rows, n), axis=1, dtype=np.int64).astype(dtype), "%s %d x %d" % (kind, rows, n))


@pytest.mark.gpu
def test_gpu_one_read_scans_in_a_graph(thc):
    """A captured scan is replayed with other scans and a change of its input between the replays: tickets, tags and words
    are the device's own, so no replay meets an older one's totals."""
    hip = ctypes.CDLL("libamdhip64.so")
    ptr = ctypes.c_void_p
    rng = np.random.default_rng(61)
    jobs = []
    for shape in ((300001,), (3001, 257), (40001, 5)):
        jobs.append((thc.Tensor("float").resize(shape), thc.Tensor("float").resize(shape)))

    def refill():
        values = [(rng.integers(0, 30, x.shape) == 0).astype(np.float32) for x, _ in jobs]
        for (x, _), v in zip(jobs, values):
            x._fn("copyFromHost")(x._st, x.h, v.ctypes.data_as(ptr))
        return [np.cumsum(v, axis=0, dtype=np.float64).astype(np.float32) for v in values]

    refill()
    lib, st, stream, graph, ready = thc.lib(), thc.state(), ptr(), ptr(), ptr()
    assert hip.hipStreamCreate(ctypes.byref(stream)) == 0
    lib.THCState_setCurrentStream(st, stream)
    try:
        for x, y in jobs:
            y.cumsum(x, 0)                # (the stream's scratch is there before the capture)
        assert hip.hipStreamSynchronize(stream) == 0
        assert hip.hipStreamBeginCapture(stream, 2) == 0
        for x, y in jobs:
            y.cumsum(x, 0)
        assert hip.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(ready), graph, None, None, ctypes.c_size_t(0)) == 0
        for i in range(5):
            want = refill()
            assert hip.hipGraphLaunch(ready, stream) == 0
            for x, y in jobs[i % 4:]:
                thc.Tensor("float").cumsum(x, 0)
            assert hip.hipStreamSynchronize(stream) == 0
            for (x, y), w in zip(jobs, want):
                assert_bit_equal(y.numpy(), w, "replay %d" % i)
        assert hip.hipGraphExecDestroy(ready) == 0 and hip.hipGraphDestroy(graph) == 0
    finally:
        hip.hipStreamSynchronize(stream)
        lib.THCState_setCurrentStream(st, None)


def test_the_counter_of_one_read_scans_starts_its_tags_again(tmp_path):
    """On the host (tests/scan_ticket_test.cpp): no scan accepts what the scan before it published, also where the tags start again."""
    root, exe = os.path.dirname(os.path.dirname(os.path.abspath(__file__))), str(tmp_path / "scan_ticket_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-I", os.path.join(root, "cutorch_amd", "csrc"),
                    os.path.join(root, "tests", "scan_ticket_test.cpp"), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip() == "ok", res.stdout + res.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("first", [1, 0xfffffffd])
def test_gpu_one_read_scans_where_the_tags_start_again(thc, first):
    """Scans of several chunks on a new stream whose counter starts a few tags before the last one: rows, strips and runs."""
    hip = ctypes.CDLL("libamdhip64.so")
    rng = np.random.default_rng(67)
    inputs = [(rng.integers(0, 30, shape) == 0).astype(np.float32) for shape in ((300001,), (3001, 257), (40001, 5))]
    dev = [thc.Tensor.from_numpy(x) for x in inputs]
    want = [np.cumsum(x, axis=0, dtype=np.float64).astype(np.float32) for x in inputs]
    stream = ctypes.c_void_p()
    assert hip.hipDeviceSynchronize() == 0 and hip.hipStreamCreate(ctypes.byref(stream)) == 0
    thc.set_tuning("scan.first_tag", first)
    thc.lib().THCState_setCurrentStream(thc.state(), stream)
    try:
        for i in range(6):
            for k in range(3):
                got = thc.Tensor("float").cumsum(dev[k], 0)
                assert hip.hipStreamSynchronize(stream) == 0
                assert_bit_equal(got.numpy(), want[k], "scan %d of input %d" % (i, k))
    finally:
        thc.set_tuning("scan.first_tag", 1)
        hip.hipStreamSynchronize(stream)
        thc.lib().THCState_setCurrentStream(thc.state(), None)


@pytest.mark.gpu
def test_gpu_scans_of_many_slices_of_one_chunk_each_need_no_words(thc):
    """Slices that fit one chunk publish nothing, so their number is not held to the room for published totals: on both sides of that
    room, strips and runs (the element-wise column kernel, which they went to, walks such rows alone)."""
    rng = np.random.default_rng(79)
    for shape, name in (((1010, 33, 1025), "scan-cols-split"), ((1030, 33, 1025), "scan-cols-split"),
                        ((140000, 5, 7), "scan-chunked"), ((155000, 5, 7), "scan-chunked")):
        x = rng.integers(-9, 10, shape).astype(np.float64)      # (two words a total)
        thc.set_tuning("scan.slab", 0)
        thc.set_tuning("scan.strided_two_reads", 0)
        try:
            got = thc.Tensor("double").cumsum(thc.Tensor.from_numpy(x), 1)
            assert thc.last_kernel() == name, (shape, thc.last_kernel())
        finally:
            thc.set_tuning("scan.slab", 1)
            thc.set_tuning("scan.strided_two_reads", 1)
        assert_bit_equal(got.numpy(), np.cumsum(x, axis=1), "%s" % (shape,))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "byte", "double"])
def test_gpu_strips_of_any_knob_value(thc, kind):
    """Widths and threads of the strips that the kernel has no room for or is not built for are held to those that it is: every
    row is written, in place as well, and nothing else."""
    dtype = {"float": np.float32, "byte": np.uint8, "double": np.float64}[kind]
    vec = 16 // np.dtype(dtype).itemsize
    rng = np.random.default_rng(83)
    thc.set_tuning("scan.strided", 1)
    thc.set_tuning("scan.strided_two_reads", 0)
    thc.set_tuning("scan.slab", 0)
    try:
        for inner in (vec, 3 * vec + 1, 40 * vec, 65 * vec - 1):
            shape = (2, 1200, inner)
            x = ((rng.integers(0, 60, 2 * 1200 * inner + 3) == 0) * 1).astype(dtype)
            size = x.size - 3
            want = x.copy()
            want[1:1 + size] = np.cumsum(x[1:1 + size].reshape(shape), axis=1, dtype=np.int64).astype(dtype).reshape(-1)
            for lanes in (-3, 0, 1, 2, 7, 32, 33, 1000):
                for threads in (1, 256, 300, 512, 1024, 5000):
                    thc.set_tuning("scan.strips.lanes", lanes)
                    thc.set_tuning("scan.strips.threads", threads)
                    dev = thc.Tensor.from_storage(x, 1, shape, (1200 * inner, inner, 1), kind=kind)
                    dev.cumsum(dev, 1)
                    assert thc.last_kernel() == "scan-cols-split", (inner, lanes, threads)
                    assert_bit_equal(dev.storage_numpy(), want, "%s %d lanes %d threads %d" % (kind, inner, lanes, threads))
    finally:
        thc.set_tuning("scan.strided", -1)
        thc.set_tuning("scan.strided_two_reads", 1)
        thc.set_tuning("scan.slab", 1)
        thc.set_tuning("scan.strips.lanes", 0)
        thc.set_tuning("scan.strips.threads", 0)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,name", [((1, 200, 257), "scan-cols"), ((39, 128, 515), "scan-cols"), ((40, 128, 515), "scan-cols-split"), ((1, 65, 1001), "scan-cols"), ((6, 400, 131), "scan-cols"),
                                        ((1, 600, 257), "scan-cols-split"), ((1, 300, 515), "scan-cols-split"), ((6, 65, 9001), "scan-cols-split")])
def test_gpu_small_scans_of_bytes_along_a_strided_dim_are_not_chunked(thc, shape, name):
    """Tensors of a few hundred rows of bytes stay with the column kernel, which is the faster one there."""
    x = np.random.default_rng(101).integers(0, 9, shape).astype(np.uint8)
    got = thc.Tensor("byte").cumsum(thc.Tensor.from_numpy(x), 1)
    assert thc.last_kernel() == name, thc.last_kernel()
    assert_bit_equal(got.numpy(), np.cumsum(x, axis=1, dtype=np.int64).astype(np.uint8), "%s" % (shape,))


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["float", "double"])
@pytest.mark.parametrize("rows", [256, 257, 300, 512, 513])
def test_gpu_strips_of_a_few_hundred_rows(thc, kind, rows):
    """On both sides of 20 MiB, from which on strips of 4- and 8-byte elements are cut along the rows instead of being made 128 bytes wide."""
    dtype = {"float": np.float32, "double": np.float64}[kind]
    for mb in (19.5, 20.5):
        inner = int(mb * 2 ** 20 / (6 * rows * np.dtype(dtype).itemsize)) | 1
        x = np.random.default_rng(rows).integers(-9, 10, (6, rows, inner)).astype(dtype)
        got = thc.Tensor(kind).cumsum(thc.Tensor.from_numpy(x), 1)
        assert thc.last_kernel() == "scan-cols-split", (inner, thc.last_kernel())
        assert_bit_equal(got.numpy(), np.cumsum(x, axis=1, dtype=np.float64).astype(dtype), "%s %d x %d" % (kind, rows, inner))
