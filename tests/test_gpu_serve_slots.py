"""Server batches whose descriptors outgrow the slots' first size of 32 MiB:
16 contractions with K = N = 1 and about 2^20 rows, no two alike, so that each
brings offset tables of 4 MiB of its own.  A product of one term is rounded
once in FP64: bit for bit numpy's; 14 moduli hold each operand to 51 bits
relative to its row: within 1e-14."""
import numpy as np
import pytest

from aces4_amd import sipgpu as sg

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("moduli", [0, 14])
def test_descriptors_beyond_the_first_slot_size(moduli):
    sg.init(0)
    print("server slots", moduli, flush=True)
    ptrn, e = sg.get_contraction_ptrn(2, 2, 2, [1, 2, 3, 1, 3, 2])
    assert e == 0
    rng = np.random.default_rng(4)
    cache = sg.Cache(1 << 30)
    server = sg.Server(cache, max_batch=64)
    work = []
    for i in range(16):
        M = (1 << 20) + i
        l, r = rng.standard_normal(M), rng.standard_normal(1)
        for key, x in ((3 * i, l), (3 * i + 1, r)):
            cache.insert(key + 1, x.size, host=x)
        cache.insert(3 * i + 3, M, init="zero")
        work.append((M, l, r, sg.make_request(ptrn, 3 * i + 1, [1, M], 3 * i + 2, [1, 1],
                                              3 * i + 3, [M, 1], moduli=moduli)))
    tickets = [server.submit(w[3]) for w in work]
    for t in tickets:
        server.wait(t)
    for i, (M, l, r, _) in enumerate(work):
        got = cache.read(3 * i + 3, M)
        if moduli:
            assert np.all(np.abs(got - l * r[0]) <= 1e-14 * np.abs(l * r[0]))
        else:
            assert np.array_equal(got, l * r[0])
    server.destroy()
    cache.destroy()
