"""The rows away from the polar filter in the fast and slow passes of an
integrator call as strip tiles (GD_STRIP = rows per tile when the handle is
created, 0: the row tiles), beside every form of the phase launches
(GD_FUSED: 0 separate, 1 k_phase, 2 k_wphase, 3 k_rphase, one workgroup per
filtered row with a wave per component).  All form every value by the same
expressions and add every sum in the same order, so states, per-step mass,
energy and beta must agree bit for bit; and with the oracle to the tolerance
of the other whole-step comparisons (1e-11 after a few steps)."""
import os
from contextlib import contextmanager

import numpy as np
import pytest

from conftest import rel_err

pytestmark = pytest.mark.gpu


@contextmanager
def env(**kw):
    old = {k: os.environ.get(k) for k in kw}
    os.environ.update({k: str(v) for k, v in kw.items()})
    try:
        yield
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v


def run(gd, rows, form, N, M, dt, steps, members=1, active=None, **kw):
    with env(GD_STRIP=rows, GD_FUSED=form), gd.Dycore(N, M, dt, members=members, **kw) as d:
        for m in range(members):
            d.set_state(*gd.ic_balanced(N, M, seed=19, nmax=8, n_mountains=2, mountain_seed=7,
                                        pert_seed=50 + m, pert_nmax=6, pert_rms=5.0), member=m)
        if active is not None:
            d.set_active_members(active)
        fam = set(d.profile_kernels(1))
        n = members if active is None else active
        out = [x[:, :n] for x in d.step(steps)[:3]]
        for m in range(n):
            out += d.get_state(member=m)
    return fam, out


# one segment that ends inside a wave, on its first and its last lane; two and
# three segments with a last one of 1, 2, 64, 65 longitudes; the smallest
# num_lon; odd rows; rows of 8, 12 and 16 longitudes per lane of a wave
CASES = [(8, 41, {}), (64, 42, {}), (65, 43, dict(uv_adv_scheme="upwind")), (128, 44, {}), (254, 61, {}),
         (255, 43, {}), (256, 45, dict(uv_adv_scheme="upwind", uv_adv_upwind_lon_beta=0.3)), (318, 43, {}),
         (319, 42, {}), (360, 181, dict(subcycles=6)), (405, 61, dict(uv_adv_scheme="upwind")), (720, 121, {}),
         (768, 61, {}), (1000, 41, {}), (1440, 91, {})]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_strip_tiles_bitwise(gd, case, prec):
    N, M, opts = CASES[case]
    dt = 240.0 * 180 / max(N, 2 * M)
    kw = dict(dict(split_scheme="csp2", subcycles=3), **opts, precision=prec,
              zonal_tend_filter_cutoff_wavenumber=gd.cutoff_from_lat0(N, M, 75.0))
    print(f"strip N={N} M={M} {opts} {prec}", flush=True)
    ref = run(gd, 0, 1, N, M, dt, 3, **kw)[1]
    for rows, form in ((4, 1), (1, 0), (7, 2), (4, 2), (2, 3), (0, 2), (32, 1)):
        for x, y in zip(run(gd, rows, form, N, M, dt, 3, **kw)[1], ref):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("form", [1, 3])
def test_strip_active_subset_and_diffusion(gd, form):
    N, M = 180, 91
    kw = dict(split_scheme="csp2", subcycles=4, use_diffusion=True, diffusion_coef=1e5, precision="mixed",
              zonal_tend_filter_cutoff_wavenumber=gd.cutoff_from_lat0(N, M, 75.0))
    ref = run(gd, 0, 1, N, M, 480.0, 5, members=5, active=3, **kw)[1]
    for x, y in zip(run(gd, 4, form, N, M, 480.0, 5, members=5, active=3, **kw)[1], ref):
        np.testing.assert_array_equal(x, y)


def test_default_forms_by_members(gd):
    """The forms the handle picks by itself for one, a few and many runs."""
    N, M = 180, 91
    kw = dict(split_scheme="csp2", subcycles=2, zonal_tend_filter_cutoff_wavenumber=gd.cutoff_from_lat0(N, M, 75.0))
    ics = [gd.ic_balanced(N, M, seed=4, nmax=8, pert_seed=60 + m, pert_nmax=6, pert_rms=5.0) for m in range(3)]
    out = []
    for members in (1, 4, 24):
        with gd.Dycore(N, M, 480.0, members=members, **kw) as d:
            for m in range(members):
                d.set_state(*ics[m % 3], member=m)
            mass, energy, beta, _ = d.step(4)
            out.append([mass[:, 0], energy[:, 0], beta[:, 0], *d.get_state(member=0)])
    for o in out[1:]:
        for x, y in zip(o, out[0]):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("rows", [0, 4])
@pytest.mark.parametrize("N,M,cut", [(90, 46, None), (100, 51, []), (96, 49, [5, 4, 3])])
def test_strip_against_oracle(gd, oracle_mod, N, M, cut, rows):
    """With a lat0 table, without a filter, and with a short table; mountains."""
    cut = gd.cutoff_from_lat0(N, M, 75.0) if cut is None else cut
    dt = 300.0 if cut else 20.0  # unfiltered pole rows need the small step
    kw = dict(split_scheme="csp2", subcycles=4)
    ic = gd.ic_balanced(N, M, seed=19, nmax=8, n_mountains=2, mountain_seed=7)
    o = oracle_mod.Oracle(N, M, dt, cutoff=cut, **kw)
    o.set_initial_state(*ic)
    o.start()
    mass, energy, beta, _ = o.run(4)
    with env(GD_STRIP=rows), gd.Dycore(N, M, dt, zonal_tend_filter_cutoff_wavenumber=cut, **kw) as d:
        d.set_state(*ic)
        m, e, b, _ = d.step(4)
        state = d.get_state()
    for k, x in enumerate(state):
        assert rel_err(x, o.state(o.old, k)) < 1e-11
    assert np.all(np.abs(m[:, 0] / mass - 1) < 1e-13) and np.all(np.abs(e[:, 0] / energy - 1) < 1e-12)
    assert np.all(np.abs(b[:, 0] - beta) < 1e-11)
