"""Denominators and energies of every rank, with the energies in LDS (2048 at
most) and read from memory (more), and with fewer elements than threads.

D is added in a fixed order (occupied energies in index order, then virtual
ones subtracted in index order) and the division is correctly rounded, so x / D
must equal the host's value bit for bit.  The energy is a sum of n terms in
another order than the host's: within n 2^-53 of the sum of their magnitudes,
at most 1e-12 of it here.
"""
import numpy as np
import pytest

from aces4_amd import sipgpu as sg

pytestmark = pytest.mark.gpu
CASES = [([1], [1]), ([2048], [-1]), ([2049], [1]), ([1025, 1024], [1, -1]), ([1024, 1024], [-1, 1]),
         ([7, 3, 5], [-1, -1, -1]), ([300, 2, 1747], [1, -1, 1]), ([11, 13, 9, 17], [-1, 1, -1, 1]),
         ([3, 1, 4, 1, 5], [1, 1, -1, -1, 1]), ([5, 4, 6, 3, 7, 8], [-1, 1, -1, 1, -1, 1])]


@pytest.mark.parametrize("dims, signs", CASES, ids=lambda v: str(v))
def test_denominator_and_energy(dims, signs):
    sg.init(0)
    rng = np.random.default_rng(dims)
    n = int(np.prod(dims))
    print("energy", dims, signs, flush=True)
    eps = [rng.uniform(0.5, 2.0, d) * s * (1 if s > 0 else 3) for d, s in zip(dims, signs)]
    x, y = rng.standard_normal(n), rng.standard_normal(n)
    grid = [e[i] for e, i in zip(eps, np.unravel_index(np.arange(n), dims, order="F"))]
    D = None
    for want in (1, -1):
        for e, s in zip(grid, signs):
            if s == want:
                D = s * e if D is None else (D + e if s > 0 else D - e)
    xd, yd, out = (sg.DeviceArray.from_host(v) for v in (x, y, np.zeros(1)))
    ed = [sg.DeviceArray.from_host(e) for e in eps]
    ep = [e.ptr for e in ed]
    for left, right in ((xd, yd), (xd, xd)):
        out.upload(np.zeros(1))
        sg.energy_sum(dims, left.ptr, right.ptr, ep, signs, 0.5, out.ptr)
        sg.synchronize()
        terms = 0.5 * (x / D) * (y if right is yd else x)
        assert abs(out.download()[0] - np.sum(terms)) <= 1e-12 * np.sum(np.abs(terms))
    sg.energy_denominator(dims, xd.ptr, ep, signs)
    sg.synchronize()
    assert np.array_equal(xd.download(), x / D)
    for v in [xd, yd, out] + ed:
        v.free()


# over 4 x 4096 x 256 elements: every thread's queue of loads is refilled, and its
# digits advance more than four times
LARGE = [([67, 63, 37, 29], [-1, 1, -1, 1]), ([2101, 23, 9, 11], [-1, -1, 1, 1])]


@pytest.mark.parametrize("dims, signs", LARGE, ids=lambda v: str(v))
def test_blocks_longer_than_the_loads_ahead(dims, signs):
    assert np.prod(dims) > 4 * 4096 * 256
    test_denominator_and_energy(dims, signs)
