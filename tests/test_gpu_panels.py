"""GPU parity of the panel layout (units of 16 rows) on the FP64 panels and on
each GEMM tile of the split path.

Against the oracle's contractions added in list order.  FP64 panels: 1e-13
relative Frobenius error (sums of at most a few thousand products).  Split
path, 14 moduli: 1e-12, the bound of operands rounded once to P bits a row.
Sizes at the edges: rows around 16 and around a tile of 128 or 256, K around
the 8 or 16 of a unit and the stages of 64 and 128, result blocks merged into
grids whose stacked operands have odd row counts, pairs of unequal K.
"""
import numpy as np
import pytest

from cases import rel_fro
from checker import Oracle

from aces4_amd import sipgpu as sg

pytestmark = pytest.mark.gpu
o = Oracle()
WAYS = [("packed", None, -1, 1e-13), ("packed", None, 64, 1e-13), ("split", 14, 128, 1e-12),
        ("split", 14, 256, 1e-12), ("split", 14, 257, 1e-12)]
# rows of the left blocks, of the right blocks, K of the pairs
GRIDS = [([1], [1], [1]), ([16], [17], [8]), ([15], [31], [9]), ([17, 1, 16], [33, 15], [16, 7]),
         ([128], [127], [64, 65]), ([129, 3], [255, 2], [63, 129, 1]), ([256], [257], [128]),
         ([100, 100, 57], [100, 31, 100], [100, 3, 40]), ([5], [300], [1000, 24]),
         ([40, 260], [270], [17] * 30)]


@pytest.mark.parametrize("nfast", [False, True])
@pytest.mark.parametrize("path, moduli, tile, tol", WAYS, ids=lambda v: str(v))
@pytest.mark.parametrize("rows, cols, ks", GRIDS, ids=lambda v: str(v)[:16])
def test_panels_vs_oracle(rows, cols, ks, path, moduli, tile, tol, nfast):
    """Every block of a grid of result blocks, D(i,j) += sum_p L(i,p) R(p,j)."""
    sg.init(0)
    rng = np.random.default_rng([sum(rows), sum(cols), sum(ks), nfast])
    print("panels", path, tile, rows, cols, ks[:4], nfast, flush=True)
    # D(m,n) or D(n,m) = L(m,k) R(k,n)
    ptrn, e = sg.get_contraction_ptrn(2, 2, 2, ([2, 1] if nfast else [1, 2]) + [1, 3, 3, 2])
    assert e == 0
    L = [[rng.standard_normal(m * k) for k in ks] for m in rows]
    R = [[rng.standard_normal(k * n) for k in ks] for n in cols]
    D0 = [[rng.standard_normal(m * n) for n in cols] for m in rows]
    up = lambda t: [[sg.DeviceArray.from_host(x) for x in r] for r in t]
    Ld, Rd, Dd = up(L), up(R), up(D0)
    dims = lambda m, n: [m, n] if not nfast else [n, m]
    cs = [sg.make_contraction(ptrn, Ld[i][p].ptr, [m, k], Rd[j][p].ptr, [k, n], Dd[i][j].ptr,
                              dims(m, n), accumulate=True)
          for i, m in enumerate(rows) for j, n in enumerate(cols) for p, k in enumerate(ks)]
    b = sg.plan_choice(cs, path, moduli=moduli, tile=tile)
    b.execute()
    sg.synchronize()
    assert b.kind == path
    for i, m in enumerate(rows):
        for j, n in enumerate(cols):
            want = D0[i][j].copy()
            for p, k in enumerate(ks):
                tmp, e = o.contract(ptrn, L[i][p], [m, k], R[j][p], [k, n], dims(m, n))
                assert e == 0
                want = want + tmp
            assert rel_fro(Dd[i][j].download(), want) <= tol
    b.destroy()
    for t in (Ld, Rd, Dd):
        for r in t:
            for x in r:
                x.free()
