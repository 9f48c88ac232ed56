"""The split path on whole numbers is exact.

Operands of at most 10 bits fit the scaled integers of every number of moduli
(the smallest, 6, keeps 19 bits at these K), so the product, recovered from
its residues, must equal the integer product, and a destination of whole
numbers added to it must too: no tolerance.  Sizes at the edges of the
reconstruction (four elements to a thread, 1024 to a workgroup, rows shorter
than four) and of the conversion (32 rows, 128 k), with destinations whose
elements follow each other in memory and ones whose do not.
"""
import numpy as np
import pytest

from aces4_amd import sipgpu as sg

pytestmark = pytest.mark.gpu
SHAPES = [(1, 1, 1), (3, 1, 17), (5, 3, 16), (33, 31, 129), (1, 1030, 8), (1025, 1, 127),
          (34, 61, 40), (2, 513, 300)]
# D(i,n) = sum_k L(i,k) R(k,n), D(n,i), and D(i,j,n) = sum_k L(i,j,k) R(k,n) stored (i,n,j)
FORMS = ["mn", "nm", "inj"]


@pytest.mark.parametrize("moduli", [6, 7, 8, 11, 12, 13, 14])
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("M, N, K", SHAPES)
def test_whole_numbers_are_exact(M, N, K, form, moduli):
    sg.init(0)
    rng = np.random.default_rng([M, N, K, moduli])
    print("split exact", M, N, K, form, moduli, flush=True)
    J = 3 if form == "inj" else 1
    A = rng.integers(-1023, 1024, (M, J, K))
    B = rng.integers(-1023, 1024, (K, N))
    A[M // 2] = 0  # a row without a scale
    D0 = rng.integers(-1000, 1000, (M, J, N))
    order = {"mn": (0, 1, 2), "nm": (2, 1, 0), "inj": (0, 2, 1)}[form]
    labels = {"mn": [1, 2, 1, 3, 3, 2], "nm": [2, 1, 1, 3, 3, 2],
              "inj": [1, 2, 4, 1, 4, 3, 3, 2]}[form]
    ranks = (3, 3, 2) if form == "inj" else (2, 2, 2)
    ptrn, e = sg.get_contraction_ptrn(*ranks, labels)
    assert e == 0
    drop = lambda s: [x for i, x in enumerate(s) if form == "inj" or i != 1]
    flat = lambda x: x.astype(np.float64).ravel(order="F")
    ldims = drop([M, J, K])
    ddims = [M, N, J] if form == "inj" else ([M, N] if form == "mn" else [N, M])
    for accumulate in (False, True):
        l, r, d = (sg.DeviceArray.from_host(x)
                   for x in (flat(A), flat(B), flat(D0.transpose(order))))
        c = sg.make_contraction(ptrn, l.ptr, ldims, r.ptr, [K, N], d.ptr, ddims,
                                accumulate=accumulate)
        b = sg.Batch([c], moduli=moduli)
        assert b.kind == "split"
        b.execute()
        sg.synchronize()
        want = np.einsum("ijk,kn->ijn", A, B) + (D0 if accumulate else 0)
        assert np.array_equal(d.download(), flat(want.transpose(order)))
        b.destroy()
        for x in (l, r, d):
            x.free()
