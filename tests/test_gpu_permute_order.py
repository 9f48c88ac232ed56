"""Permutes over every tile order: launch order (rows of whole cache lines,
few tiles), patches dealt to the XCDs, blocks too large for the cache, and
batches that mix them, with block addresses on and off cache lines.  Data
movement: bit for bit numpy's transpose.
"""
import numpy as np
import pytest

from aces4_amd import sipgpu as sg
from aces4_amd.workloads import uniform

pytestmark = pytest.mark.gpu


def transposed(x, dims, perm):
    y = x.reshape(dims, order="F").transpose([perm.index(i + 1) for i in range(len(dims))])
    return y.ravel(order="F")


# (dims, perm): one tile; one tile and one element more; a matrix of whole
# lines and its odd neighbours; up to 63 and 64 tiles; enough for patches, with
# both counts of tiles no multiple of a patch; several U dims; row mode;
# identity; input and output of 512 MB and more.
SHAPES = [([2, 3], [2, 1]), ([32, 64], [2, 1]), ([33, 65], [2, 1]), ([512, 1024], [2, 1]),
          ([511, 1025], [2, 1]), ([512, 1040], [2, 1]), ([31, 7, 29, 21], [3, 4, 1, 2]),
          ([97, 5, 89, 23], [3, 2, 4, 1]), ([40, 39, 38, 37], [4, 3, 2, 1]),
          ([16, 32, 48, 16], [3, 4, 1, 2]), ([5, 6, 7, 8, 9, 10], [6, 4, 2, 1, 3, 5]),
          ([41, 30, 29, 7], [1, 3, 2, 4]), ([13, 11, 17], [1, 2, 3]), ([331, 317, 321], [3, 1, 2])]


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("dims, perm", SHAPES, ids=lambda v: "x".join(map(str, v)))
def test_permute_tile_orders(dims, perm, off):
    sg.init(0)
    print("permute order", dims, perm, off, flush=True)
    n = int(np.prod(dims))
    x = uniform(7, n)
    src, dst = sg.DeviceArray(n + 2), sg.DeviceArray(n + 2)
    dst.fill_bytes(0xAB)
    src.upload_range(off, x)
    sg.permute(dims, [1] + perm, src.at(off), dst.at(1 - off))
    sg.synchronize()
    got = dst.download()
    assert np.array_equal(got[1 - off:1 - off + n], transposed(x, dims, perm))
    guard = np.full(16, 0xAB, dtype=np.uint8).view(np.float64)[0]  # nothing written beside it
    rest = np.concatenate([got[:1 - off], got[1 - off + n:]])
    assert np.array_equal(rest.view(np.uint64), np.full(2, guard).view(np.uint64))
    src.free()
    dst.free()


@pytest.mark.parametrize("copies", [1, 5])
def test_permute_batch_tile_orders(copies):
    sg.init(0)
    shapes = SHAPES[:-1] * copies
    sizes = [int(np.prod(d)) for d, _ in shapes]
    at = np.concatenate([[0], np.cumsum(sizes)])
    x = uniform(9, int(at[-1]))
    src, dst = sg.DeviceArray.from_host(x), sg.DeviceArray(x.size)
    print("permute batch order", len(shapes), flush=True)
    b = sg.PermuteBatch([sg.permutation(d, [1] + p, src.at(int(o)), dst.at(int(o)))
                         for (d, p), o in zip(shapes, at)])
    b.execute()
    sg.synchronize()
    got = dst.download()
    for (d, p), o, n in zip(shapes, at, sizes):
        assert np.array_equal(got[o:o + n], transposed(x[o:o + n], d, p)), (d, p)
    b.destroy()
    src.free()
    dst.free()


def test_permute_batch_beyond_the_cache():
    """2^25 elements and more: entries that store through the cache (ragged runs)
    beside those that stream (whole lines, whole rows, identity, one tile) in one
    launch."""
    sg.init(0)
    shapes = SHAPES + [([36, 14, 18, 18, 20, 16], [6, 2, 4, 3, 5, 1])] + SHAPES[:4]
    sizes = [int(np.prod(d)) for d, _ in shapes]
    at = np.concatenate([[0], np.cumsum([(s + 15) // 16 * 16 for s in sizes])])
    assert sum(sizes) >= 1 << 25
    x = uniform(10, int(at[-1]))
    src, dst = sg.DeviceArray.from_host(x), sg.DeviceArray(x.size)
    print("permute batch beyond the cache", len(shapes), flush=True)
    b = sg.PermuteBatch([sg.permutation(d, [1] + p, src.at(int(o)), dst.at(int(o)))
                         for (d, p), o in zip(shapes, at)])
    b.execute()
    sg.synchronize()
    got = dst.download()
    for (d, p), o, n in zip(shapes, at, sizes):
        assert np.array_equal(got[o:o + n], transposed(x[o:o + n], d, p)), (d, p)
    b.destroy()
    src.free()
    dst.free()
