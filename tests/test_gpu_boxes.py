"""Boxes of points between dats and host arrays (fetch, set, slabs,
declarations with data): bytes, so equal to numpy's slices exactly.  Sizes
around the copy's pieces (4 MiB) and units (1 to 16 bytes)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [
    # size (x first), halo, components, structure of arrays, type
    ([524288], 1, 1, False, np.float64),         # one row: a piece and two halo points
    ([3], 1, 1, False, np.float32),
    ([1031, 700], 2, 1, False, np.float64),      # odd rows, two pieces
    ([1500, 1400], 1, 1, False, np.float32),     # three pieces, 16-byte units inside a row
    ([33, 17, 9], 1, 1, False, np.float64),
    ([130, 64, 70], 3, 1, False, np.float32),
    ([37, 20, 11], 1, 3, False, np.float64),
    ([37, 20, 11], 1, 3, True, np.float64),
    ([600, 300, 9], 1, 3, True, np.float32),     # components together, two pieces
    ([257, 190], 1, 2, True, np.int32),
]


@pytest.mark.parametrize("size,halo,dim,soa,dtype", CASES)
def test_boxes_equal_numpy_slices(gpu_ops, size, halo, dim, soa, dtype):
    ops = gpu_ops
    nd = len(size)
    ops.ops_set_soa(soa)
    try:
        blk = ops.ops_decl_block(nd, "boxes")
        d = ops.ops_decl_dat(blk, size, [-halo] * nd, [halo] * nd, dtype, "d", dim=dim)
    finally:
        ops.ops_set_soa(False)
    # the dat's x padding belongs to its upper halo (d_p as declared here)
    shape = tuple(n + 2 * halo for n in reversed(size)) + ((dim,) if dim > 1 else ())
    rng = np.random.RandomState(7)
    ref = (rng.randint(-2 ** 30, 2 ** 30, shape)).astype(dtype)
    ops.set_whole(d, ref)
    assert np.array_equal(ops.get_whole(d), ref)
    inner = tuple(slice(halo, -halo) for _ in size)
    if dim == 1:
        assert np.array_equal(ops.ops_dat_fetch_data(d), ref[inner])
        new = (rng.randint(-2 ** 30, 2 ** 30, ref[inner].shape)).astype(dtype)
        ops.ops_dat_set_data(d, new)
        ref[inner] = new
        assert np.array_equal(ops.get_whole(d), ref)
    # a slab off every alignment: [1, n - 1) in each dimension
    slab = [v for n in size for v in (1, n - 1)]
    at = tuple(slice(halo + 1, halo + n - 1) for n in reversed(size))
    assert np.array_equal(ops.ops_dat_fetch_data_slab(d, slab), ref[at])
    new = (rng.randint(-2 ** 30, 2 ** 30, ref[at].shape)).astype(dtype)
    ops.ops_dat_set_data_slab(d, slab, new)
    ref[at] = new
    assert np.array_equal(ops.get_whole(d), ref)
    ops.ops_free_dat(d)


@pytest.mark.parametrize("size", [[5], [700, 300], [1031, 700], [40, 30, 20]])
def test_declaration_with_data(gpu_ops, size):
    ops = gpu_ops
    nd = len(size)
    shape = tuple(n + 2 for n in reversed(size))
    data = np.random.RandomState(3).rand(*shape)
    d = ops.ops_decl_dat(ops.ops_decl_block(nd, "withdata"), size, data=data, name="d")
    assert np.array_equal(ops.get_whole(d), data)
    ops.ops_free_dat(d)


def test_declared_data_is_not_cleared_afterwards(gpu_ops):
    """Clearing a new array is ordered before the upload into it, also while
    the GPU is still clearing a large array declared just before (6 GiB, about
    a millisecond).  The shell of zeros past the uploaded rows stays."""
    ops = gpu_ops
    blk = ops.ops_decl_block(2, "clearing")
    data = np.arange(302 * 202, dtype=np.float64).reshape(202, 302) + 1
    for _ in range(3):
        big = ops.ops_decl_dat(blk, [16384, 49152], name="big")
        d = ops.ops_decl_dat(blk, [300, 200], data=data, name="d")
        assert np.array_equal(ops.get_whole(d), data)
        corner = ops.ops_dat_fetch_data_slab(big, [16000, 16384, 49151, 49152])
        assert not corner.any()
        ops.ops_free_dat(d)
        ops.ops_free_dat(big)


@pytest.mark.parametrize("size", [[0], [5, 0], [0, 5], [4, 0, 3], [4, 3, 0]])
def test_declaration_with_data_and_no_points(gpu_ops, size):
    """an empty array (a dimension of no points and no halo) with a data
    pointer: nothing to upload"""
    ops = gpu_ops
    nd = len(size)
    blk = ops.ops_decl_block(nd, "empty")
    d = ops.ops_decl_dat(blk, size, [0] * nd, [0] * nd, data=np.zeros(size[::-1]), name="d")
    ops.ops_free_dat(d)


@pytest.mark.parametrize("size,halo", [([256], 1), ([257], 1), ([3], 1), ([65536, 3], 1), ([65537, 3], 1),
                                       ([70000, 2, 2], 1), ([200000], 2)])
def test_boxes_on_both_sides_of_the_copy_rules(gpu_ops, size, halo):
    """rows around the widths (2 KiB single, 512 KiB) that go by a copy call"""
    test_boxes_equal_numpy_slices(gpu_ops, size, halo, 1, False, np.float64)


def test_declaration_with_data_in_device_memory(gpu_ops):
    """the data pointer may be device memory (here another dat's, rows without
    padding, 512 MiB): copied when the call returns, whichever stream the
    library works on"""
    import ctypes as C
    ops = gpu_ops
    nx, ny = 4094, 16382
    blk = ops.ops_decl_block(2, "ondevice")
    a = ops.ops_decl_dat(blk, [nx, ny], name="a")
    for y in (0, 1, ny // 2, ny - 1):
        ops.ops_dat_set_data_slab(a, [0, nx, y, y + 1], np.arange(nx, dtype=np.float64).reshape(1, nx) + 1000.5 * y)
    space = C.c_int(ops.OPS_DEVICE)
    addr = ops._call("ops_dat_get_raw_pointer", a.ptr, 0, None, C.byref(space)) - 8 * (1 + (nx + 2))  # point (-1, -1)
    p = ops._call("ops_decl_dat_char", blk.ptr, 1, ops._ints([nx, ny]), ops._ints([0, 0]), ops._ints([-1, -1]),
                  ops._ints([1, 1]), ops._ints([1, 1]), addr, 8, b"double", b"b")
    b = ops.Dat(p, blk, [nx, ny], [-1, -1], [1, 1], np.dtype(np.float64), "b", 1)
    last = ops.ops_dat_fetch_data_slab(b, [0, nx, ny - 1, ny])
    ops._call("ops_dat_release_raw_data", a.ptr, 0, ops.OPS_READ)
    assert np.array_equal(last, ops.ops_dat_fetch_data_slab(a, [0, nx, ny - 1, ny])) and last[0, 1] != 0
    assert np.array_equal(ops.get_whole(b), ops.get_whole(a))
    ops.ops_free_dat(a)
    ops.ops_free_dat(b)
