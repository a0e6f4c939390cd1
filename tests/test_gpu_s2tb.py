"""Strip tiles that form the second predictor S0 + hdt Tb in the corrector
phase (GD_S2TB = 1 when the handle is created) beside those that load the one
phase B stored (GD_S2TB = 0).  One expression forms both, so states, per-step
mass, energy and beta must agree bit for bit."""
import numpy as np
import pytest

from test_gpu_fold import env

pytestmark = pytest.mark.gpu


def run(gd, s2, form, rows, N, M, steps, members=1, look=None, **kw):
    e = dict(GD_S2TB=s2)
    if form is not None:
        e["GD_FUSED"] = form
    if rows is not None:
        e["GD_STRIP"] = rows
    with env(**e), gd.Dycore(N, M, 240.0 * 180 / max(N, 2 * M), members=members, split_scheme="csp2",
                             zonal_tend_filter_cutoff_wavenumber=gd.cutoff_from_lat0(N, M, 75.0), **kw) as d:
        for m in range(members):
            d.set_state(*gd.ic_balanced(N, M, seed=19, nmax=8, n_mountains=2, mountain_seed=7,
                                        pert_seed=50 + m % 3, pert_nmax=6, pert_rms=5.0), member=m)
        out = list(d.step(steps)[:3])
        for m in range(members) if look is None else look:
            out += d.get_state(member=m)
    return out


# few and many rows of strips (the rows next to their ends keep the stored
# predictor), groups of one row, of a few and of more rows than there are;
# segments that end on a wave's edge; rows of 8, 12, 16 longitudes per lane of
# k_rphase and of 4 and 8 per thread of k_phase
CASES = [(8, 41, 4), (64, 42, 1), (65, 43, 7), (255, 43, 32), (254, 61, 2), (405, 61, None), (720, 121, 4),
         (1000, 41, 3), (1440, 91, None)]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("N,M,rows", CASES)
def test_second_predictor_bitwise(gd, N, M, rows, prec):
    kw = dict(precision=prec, subcycles=3, uv_adv_scheme="upwind" if N % 2 else "center_diff")
    print(f"s2tb N={N} M={M} rows={rows} {prec}", flush=True)
    for form in (1, 3):
        ref = run(gd, 0, form, rows, N, M, 3, members=2, **kw)
        for x, y in zip(run(gd, 1, form, rows, N, M, 3, members=2, **kw), ref):
            np.testing.assert_array_equal(x, y)


def test_rule_takes_a_large_batch(gd):
    """100 members of 180x91 (223 MB of a call's fields), eight-step graph and
    one step more, by the rule and without."""
    kw = dict(precision="mixed", subcycles=2, use_diffusion=True, diffusion_coef=1e5)
    ref = run(gd, 0, None, None, 180, 91, 9, members=100, look=(0, 57, 99), **kw)
    for x, y in zip(run(gd, "", None, None, 180, 91, 9, members=100, look=(0, 57, 99), **kw), ref):
        np.testing.assert_array_equal(x, y)
