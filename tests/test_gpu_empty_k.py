"""Products whose contracted index is empty: D (+)= 0, on every tile
configuration of the table kernels, the packed and split paths and a single
contraction, beside products that are not empty.  Zeros and untouched values
bit for bit."""
import numpy as np
import pytest

from aces4_amd import sipgpu as sg

pytestmark = pytest.mark.gpu
PTRN = [-1, 1, -1, 2]


def entries(M, N, ks, D, L, R, accumulate):
    return [sg.make_contraction(PTRN, L.ptr, [k, M], R.ptr, [k, N], D.at(i * M * N), [M, N],
                                accumulate=accumulate) for i, k in enumerate(ks)]


def check(plan, ks, tol):
    M, N = 150, 130
    rng = np.random.default_rng(6)
    l, r = rng.standard_normal(40 * M), rng.standard_normal(40 * N)
    L, R = sg.DeviceArray.from_host(l), sg.DeviceArray.from_host(r)
    prod = (l.reshape(M, 40) @ r.reshape(N, 40).T).ravel(order="F")
    D0 = rng.standard_normal(len(ks) * M * N)
    for accumulate in (False, True):
        D = sg.DeviceArray.from_host(D0)
        b = plan(entries(M, N, ks, D, L, R, accumulate))
        b.execute()
        sg.synchronize()
        got = D.download().reshape(len(ks), M * N)
        for k, g, d0 in zip(ks, got, D0.reshape(len(ks), M * N)):
            was = d0 if accumulate else np.zeros(M * N)
            if k == 0:
                assert np.array_equal(g, was)
            else:
                assert np.linalg.norm(g - was - prod) <= tol * np.linalg.norm(was + prod)
        b.destroy()
        D.free()


@pytest.mark.parametrize("ks", [[0], [40, 0], [0, 40, 0, 0, 40, 0]], ids=str)
@pytest.mark.parametrize("config", range(19))
def test_table_configurations(config, ks):
    sg.init(0)
    print("empty K", config, ks, flush=True)
    check(lambda cs: sg.plan_choice(cs, "tables", config=config), ks, 1e-13)


@pytest.mark.parametrize("ks", [[0], [40, 0], [0, 40, 0, 0, 40, 0]], ids=str)
def test_panel_paths(ks):
    sg.init(0)
    print("empty K, packed", ks, flush=True)
    check(lambda cs: sg.plan_choice(cs, "packed"), ks, 1e-13)
    for tile in (128, 256, 257):
        print("empty K, split", tile, ks, flush=True)
        check(lambda cs: sg.plan_choice(cs, "split", moduli=14, tile=tile), ks, 1e-12)


@pytest.mark.parametrize("M, N", [(150, 130), (1700, 1500)])
def test_single_contraction(M, N):
    sg.init(0)
    print("empty K, single", M, N, flush=True)
    D0 = np.random.default_rng(7).standard_normal(M * N)
    L, R = sg.DeviceArray(1), sg.DeviceArray(1)
    for accumulate in (True, False):
        D = sg.DeviceArray.from_host(D0)
        sg.contract(PTRN, L.ptr, [0, M], R.ptr, [0, N], D.ptr, [M, N], accumulate=accumulate)
        sg.synchronize()
        assert np.array_equal(D.download(), D0 if accumulate else np.zeros(M * N))
        D.free()
