"""GPU parity of the 32 x 32 tiles whose K is split over a workgroup's waves.

Against the oracle's contractions added in list order, within 1e-13 relative
Frobenius error (sums of at most a few thousand FP64 products).  Sizes at the
edges: one element, one below and above a 16 or 32 block, fewer k-steps than
waves, K that leaves part of a k-step, more pairs than one look-up covers,
pairs of one k between long ones.
"""
import numpy as np
import pytest

from cases import rel_fro
from checker import Oracle

from aces4_amd import sipgpu as sg

pytestmark = pytest.mark.gpu
o = Oracle()
SPLIT_K = 18  # tile configuration
# (pattern, left extents, right extents): k first, k last, one of each
FORMS = [([-1, 1, -1, 2], lambda m, n, k: ([k, m], [k, n])),
         ([1, -2, 2, -2], lambda m, n, k: ([m, k], [n, k])),
         ([1, -1, -2, 2], lambda m, n, k: ([m, k], [k, n]))]


def pairs_of(rng, form, M, N, ks):
    ptrn, dims = form
    out = []
    for k in ks:
        ld, rd = dims(M, N, k)
        out.append((ld, rd, rng.standard_normal(M * k), rng.standard_normal(N * k)))
    return ptrn, out


def run(ptrn, pairs, M, N, D0, accumulate, config):
    dev = [(sg.DeviceArray.from_host(l), sg.DeviceArray.from_host(r)) for _, _, l, r in pairs]
    d = sg.DeviceArray.from_host(D0)
    cs = [sg.make_contraction(ptrn, l.ptr, ld, r.ptr, rd, d.ptr, [M, N],
                              accumulate=accumulate or i > 0)
          for i, ((ld, rd, _, _), (l, r)) in enumerate(zip(pairs, dev))]
    b = sg.plan_choice(cs, "tables", config=config)
    b.execute()
    sg.synchronize()
    got = d.download()
    b.destroy()
    for a in [d] + [x for p in dev for x in p]:
        a.free()
    return got


def expected(ptrn, pairs, M, N, D0, accumulate):
    want = D0.copy() if accumulate else np.zeros(M * N)
    for ld, rd, l, r in pairs:
        tmp, e = o.contract(ptrn, l, ld, r, rd, [M, N])
        assert e == 0
        want = want + tmp
    return want


CASES = [(1, 1, [1]), (16, 16, [4]), (17, 15, [3]), (32, 33, [5]), (31, 65, [33, 31]),
         (33, 47, [64]), (48, 16, [65, 1, 129]), (100, 100, [100] * 16), (20, 37, [257]),
         (5, 70, [1, 300, 2, 2, 7]), (40, 9, [1] * 150), (18, 34, [3, 8, 5] * 45)]


@pytest.mark.parametrize("form", range(3))
@pytest.mark.parametrize("M, N, ks", CASES, ids=lambda v: str(v)[:24])
def test_splitk_tiles_vs_oracle(M, N, ks, form):
    sg.init(0)
    rng = np.random.default_rng([M, N, len(ks), form])
    print("split K", M, N, ks[:5], len(ks), form, flush=True)
    ptrn, pairs = pairs_of(rng, FORMS[form], M, N, ks)
    D0 = rng.standard_normal(M * N)
    for accumulate in (False, True):
        got = run(ptrn, pairs, M, N, D0, accumulate, SPLIT_K)
        want = expected(ptrn, pairs, M, N, D0, accumulate)
        assert rel_fro(got, want) <= 1e-13


def test_blocks_of_both_configurations_in_one_batch():
    """A block large enough for 64 x 64 tiles (2000 x 1100) beside small ones:
    each within 1e-13 of the oracle and bitwise what a batch of its own gives."""
    sg.init(0)
    rng = np.random.default_rng(3)
    shapes = [(2000, 1100, 6), (40, 50, 70), (64, 33, 20)]
    cs, parts = [], []
    for M, N, K in shapes:
        ptrn, pairs = pairs_of(rng, FORMS[2], M, N, [K])
        ld, rd, l, r = pairs[0]
        dl, dr, d = (sg.DeviceArray.from_host(x) for x in (l, r, np.zeros(M * N)))
        cs.append(sg.make_contraction(ptrn, dl.ptr, ld, dr.ptr, rd, d.ptr, [M, N]))
        parts.append((ptrn, pairs, M, N, d, (dl, dr)))
    print("both configurations", flush=True)
    b = sg.Batch(cs)
    assert b.kind == "tables"
    b.execute()
    sg.synchronize()
    got = [p[4].download() for p in parts]
    b.destroy()
    for c, (ptrn, pairs, M, N, d, _), g in zip(cs, parts, got):
        assert rel_fro(g, expected(ptrn, pairs, M, N, np.zeros(M * N), False)) <= 1e-13
        d.zero()
        alone = sg.Batch([c])
        alone.execute()
        sg.synchronize()
        assert np.array_equal(d.download().view(np.uint64), g.view(np.uint64))
        alone.destroy()


# single contractions in K segments: of 32 x 32 tiles (fewer and more tiles
# than CUs), of 64 x 64 tiles, and of neither (K one below the shortest)
SINGLES = [(320, 320, 1025), (600, 600, 770), (450, 320, 1030), (850, 296, 515), (500, 500, 255),
           (33, 31, 2500), (1, 1, 5000)]


@pytest.mark.parametrize("form", range(3))
@pytest.mark.parametrize("M, N, K", SINGLES)
def test_single_contraction_segments(M, N, K, form):
    sg.init(0)
    rng = np.random.default_rng([M, N, K, form])
    print("segments", M, N, K, form, flush=True)
    ptrn, pairs = pairs_of(rng, FORMS[form], M, N, [K])
    ld, rd, l, r = pairs[0]
    D0 = rng.standard_normal(M * N)
    dl, dr = sg.DeviceArray.from_host(l), sg.DeviceArray.from_host(r)
    for accumulate in (False, True):
        d = sg.DeviceArray.from_host(D0)
        sg.contract(ptrn, dl.ptr, ld, dr.ptr, rd, d.ptr, [M, N], accumulate=accumulate)
        sg.synchronize()
        assert rel_fro(d.download(), expected(ptrn, pairs, M, N, D0, accumulate)) <= 1e-13
        d.free()
    dl.free()
    dr.free()


def test_more_tiles_than_one_launch_holds():
    """8193 rows of 32768 as 32 x 32 tiles: over 2^23 workgroups of 512."""
    sg.init(0)
    print("split K, two launches", flush=True)
    n, N = 8193, 32768
    rng = np.random.default_rng(8)
    l, r = rng.standard_normal(n), rng.standard_normal(N)
    dl, dr, d = sg.DeviceArray.from_host(l), sg.DeviceArray.from_host(r), sg.DeviceArray(n * N)
    ptrn, _ = FORMS[0]
    cs = [sg.make_contraction(ptrn, dl.at(i), [1, 1], dr.ptr, [1, N], d.at(i * N), [1, N])
          for i in range(n)]
    b = sg.plan_choice(cs, "tables", config=SPLIT_K)
    b.execute()
    sg.synchronize()
    b.destroy()
    for i in range(0, n, 64):
        m = min(64, n - i)
        got = d.download_range(i * N, m * N).reshape(m, N)
        assert np.array_equal(got, l[i:i + m, None] * r)  # one product, rounded once
    for a in (dl, dr, d):
        a.free()
