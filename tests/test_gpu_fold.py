"""csp2 calls that leave their update to the next call's phase A (GD_FOLD = 1
when the handle is created) beside the k_update launches (GD_FOLD = 0).  Both
form S + dt beta Tc by one expression and add the beta partials in one order,
so states, per-step mass, energy and beta must agree bit for bit."""
import os
from contextlib import contextmanager

import numpy as np
import pytest

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


def run(gd, fold, form, N, M, steps, members=1, active=None, nograph=False, **kw):
    e = dict(GD_FOLD=fold)
    if form is not None:
        e["GD_FUSED"] = form
    if nograph:
        e["GD_NO_GRAPH"] = 1
    with env(**e), gd.Dycore(N, M, 240.0 * 180 / max(N, 2 * M), members=members, split_scheme="csp2", **kw) as d:
        for m in range(members):
            d.set_state(*gd.ic_balanced(N, M, seed=19, nmax=8, n_mountains=2, mountain_seed=7,
                                        pert_seed=50 + m, pert_nmax=6, pert_rms=5.0), member=m)
        n = members
        if active is not None:
            d.set_active_members(active)
            n = active
        out = [x[:, :n] for x in d.step(steps)[:3]]
        for m in range(n):
            out += d.get_state(member=m)
    return out


# the partials of fewer rows than one round of loads, of exactly one round and
# of one entry more (768 entries a round), of several rounds; segments that end
# on a wave's edge; unequal cutoffs; no polar filter; one subcycle; rows of 1,
# 2, 4 and 8 longitudes per filter thread
CASES = [(8, 41, {}), (64, 42, {}), (65, 43, dict(uv_adv_scheme="upwind")), (255, 43, dict(qcon_modified=False)),
         (254, 61, dict(subcycles=1)), (300, 91, dict(cut=[])), (360, 181, dict(subcycles=6)),
         (508, 384, dict(subcycles=2)), (509, 257, dict(subcycles=2)), (405, 61, dict(cut=[5, 4, 3])),
         (720, 121, dict(uv_adv_scheme="upwind")), (1440, 181, dict(subcycles=2))]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_folded_update_bitwise(gd, case, prec):
    N, M, opts = CASES[case]
    kw = dict(dict(subcycles=3, precision=prec), **opts)
    cut = kw.pop("cut", None)
    kw["zonal_tend_filter_cutoff_wavenumber"] = gd.cutoff_from_lat0(N, M, 75.0) if cut is None else cut
    print(f"fold N={N} M={M} {opts} {prec}", flush=True)
    ref = run(gd, 0, 1, N, M, 3, **kw)
    for form in (1, 2, None):
        for x, y in zip(run(gd, 1, form, N, M, 3, **kw), ref):
            np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("diff", [False, True])
def test_folded_update_members_and_graphs(gd, diff):
    """Five members with three active; graphs of eight steps and one, and none;
    the rule's own choice."""
    N, M = 180, 91
    kw = dict(subcycles=4, use_diffusion=diff, diffusion_coef=1e5, precision="mixed",
              zonal_tend_filter_cutoff_wavenumber=gd.cutoff_from_lat0(N, M, 75.0))
    ref = run(gd, 0, None, N, M, 9, members=5, active=3, **kw)
    for fold, nograph in ((1, False), (1, True), ("", False)):
        for x, y in zip(run(gd, fold, None, N, M, 9, members=5, active=3, nograph=nograph, **kw), ref):
            np.testing.assert_array_equal(x, y)
