"""Host <-> device copies of fields (gd_set_state, gd_get_state): every value
arrives unchanged, for dense rows and rows with a leading dimension, odd
num_lon, single fields, and grids whose fields take several turns through the
32 MiB staging buffer."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,M,ld", [(8, 5, 8), (45, 23, 45), (72, 37, 76), (361, 90, 361), (1440, 721, 1440),
                                   (2050, 1001, 2061)])
def test_state_round_trip(gd, N, M, ld):
    rng = np.random.default_rng(N)
    u, v, g, hs = (rng.standard_normal((r, ld)) for r in (M, M - 1, M, M))
    g = 1.0e4 + np.abs(g)
    u[0] = u[-1] = 0.0
    lib = gd.lib()
    with gd.Dycore(N, M, 60.0, use_zonal_tend_filter=False, members=2) as d:
        gd._check(lib.gd_set_state(d.h, 1, *[gd._dp(x) for x in (u, v, g, hs)], ld), d.h)
        out = [np.full((r, ld), -7.0) for r in (M, M - 1, M)]
        gd._check(lib.gd_get_state(d.h, 1, *[gd._dp(x) for x in out], ld), d.h)
        for x, y in zip(out, (u, v, g)):
            np.testing.assert_array_equal(x[:, :N], y[:, :N])
            assert np.all(x[:, N:] == -7.0)  # nothing past num_lon is written
        one = np.full((M - 1, ld), -7.0)
        gd._check(lib.gd_get_state(d.h, 1, None, gd._dp(one), None, ld), d.h)
        np.testing.assert_array_equal(one[:, :N], v[:, :N])
        gd._check(lib.gd_get_state(d.h, 1, None, None, None, C.c_int64(ld)), d.h)


def test_step_series_of_many_members(gd):
    """The per-step mass, energy and beta of every member, in one call of more
    steps than the device ring holds and in single steps."""
    N, M = 72, 37
    kw = dict(split_scheme="none", members=5, zonal_tend_filter_cutoff_wavenumber=[6, 5, 4])
    out = []
    for chunks in ([520], [1] * 3 + [517]):
        with gd.Dycore(N, M, 100.0, **kw) as d:
            for m in range(5):
                d.set_state(*gd.ic_balanced(N, M, seed=m, nmax=6), member=m)
            out.append([np.concatenate(x) for x in zip(*[d.step(n)[:3] for n in chunks])])
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
        assert np.all(x[1:] != 0.0)
