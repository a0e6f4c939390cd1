"""The launches behind the bitwise comparisons of the strip, folded-update and
second-predictor tests: the settings those tests force, and the handle's own
rules, must make the launches they are meant to, or a path would be compared
with itself.  gd_profile_kernels names the launches: tend and filter
(separate), phase (k_phase), wphase (k_wphase), rphase (k_rphase), *_s2tb for a
corrector phase that forms the second predictor again; a folded update has no
update launch."""
import pytest

import test_gpu_fold
import test_gpu_s2tb
import test_gpu_strip
from test_gpu_fold import env

pytestmark = pytest.mark.gpu

PHASES = {"tend", "phase", "wphase", "rphase", "phase_s2tb", "rphase_s2tb"}


def launches(gd, N, M, members=1, active=None, subcycles=3, cut=None, lat0=75.0, split="csp2", env_=(), **kw):
    """{family: launches} of one step."""
    cut = gd.cutoff_from_lat0(N, M, lat0) if cut is None else cut
    with env(**dict(env_)), gd.Dycore(N, M, 240.0 * 180 / max(N, 2 * M), members=members, split_scheme=split,
                                      subcycles=subcycles, zonal_tend_filter_cutoff_wavenumber=cut, **kw) as d:
        ic = gd.ic_balanced(N, M, seed=19, nmax=6)
        for m in range(members):
            d.set_state(*ic, member=m)
        if active is not None:
            d.set_active_members(active)
        return {k: v[0] for k, v in d.profile_kernels(1).items()}


def forced(N, form, strips):
    """The phase launches of a forced form at N longitudes."""
    wide = 255 <= N <= 762
    return {0: "tend", 1: "phase", 2: "wphase" if wide else "phase",
            3: "rphase" if strips and N <= 1024 else "phase"}[form]


@pytest.mark.parametrize("case", range(len(test_gpu_strip.CASES)))
def test_forms_of_the_strip_cases(gd, case):
    N, M, opts = test_gpu_strip.CASES[case]
    for rows, form in ((0, 1), (4, 1), (1, 0), (7, 2), (4, 2), (2, 3), (0, 2), (32, 1)):
        got = launches(gd, N, M, env_=dict(GD_STRIP=rows, GD_FUSED=form, GD_S2TB=0), **opts)
        assert set(got) & PHASES == {forced(N, form, rows)}, (rows, form)
        # the fold follows its rule: never without strip tiles or in forms 0, 3
        calls = opts.get("subcycles", 3) + 2
        assert got["update"] in (1, calls)
        if rows == 0 or forced(N, form, rows) in ("tend", "rphase"):
            assert got["update"] == calls


@pytest.mark.parametrize("case", range(len(test_gpu_fold.CASES)))
def test_updates_of_the_fold_cases(gd, case):
    N, M, opts = test_gpu_fold.CASES[case]
    opts = dict(dict(subcycles=3), **opts)
    calls = opts["subcycles"] + 2
    for fold in (0, 1):
        for form in (1, 2, None):
            e = dict(GD_FOLD=fold) if form is None else dict(GD_FOLD=fold, GD_FUSED=form)
            got = launches(gd, N, M, env_=e, **opts)
            # without filtered rows nothing is fused, and no update is folded
            fused = opts.get("cut") != []
            assert got["update"] == (1 if fold and fused and "rphase" not in got else calls), (fold, form)
            assert ("tend" in got) != fused and "rphase" not in got


@pytest.mark.parametrize("N,M,rows", test_gpu_s2tb.CASES)
def test_correctors_of_the_second_predictor_cases(gd, N, M, rows):
    for form in (1, 3):
        fam = "rphase" if form == 3 and N <= 1024 else "phase"
        for s2 in (0, 1):
            e = dict(GD_S2TB=s2, GD_FUSED=form, GD_FOLD=0)
            if rows is not None:
                e["GD_STRIP"] = rows
            got = launches(gd, N, M, members=2, env_=e)
            want = {fam: 15} if not s2 else {fam: 10, fam + "_s2tb": 5}
            assert {k: v for k, v in got.items() if k in PHASES} == want


def test_second_predictor_is_not_formed_again_in_other_forms(gd):
    for form, fam in ((0, "tend"), (2, "wphase")):
        got = launches(gd, 360, 91, env_=dict(GD_S2TB=1, GD_FUSED=form))
        assert set(got) & PHASES == {fam}


# the handle's own choice: by members (180x91), by the grid, and past the limits
# of the launches without strip tiles (24576 row tiles, 6144 past 1024
# longitudes), where csp2 stays fused and unsplit steps do not
RULES = [(180, 91, 1, {}, {"phase"}, True), (180, 91, 8, {}, {"phase"}, True), (180, 91, 24, {}, {"rphase"}, False),
         (180, 91, 100, {}, {"rphase", "rphase_s2tb"}, False), (360, 181, 1, {}, {"wphase"}, True),
         (360, 181, 16, {}, {"rphase"}, False), (720, 361, 1, {}, {"wphase"}, True),
         (720, 361, 2, {}, {"phase"}, True), (1440, 181, 1, {}, {"phase"}, True),
         (1440, 361, 1, {}, {"phase"}, False), (1440, 37, 30, {}, {"phase", "phase_s2tb"}, False),
         (1440, 37, 30, dict(split="none"), {"tend"}, False), (180, 91, 272, {}, {"rphase", "rphase_s2tb"}, False),
         (180, 91, 272, dict(split="none"), {"tend"}, False), (180, 91, 1, dict(cut=[]), {"tend"}, False),
         (2050, 37, 1, {}, {"tend"}, False), (1000, 41, 64, {}, {"phase", "phase_s2tb"}, False)]


@pytest.mark.parametrize("N,M,members,more,phases,folded", RULES)
def test_rules(gd, N, M, members, more, phases, folded):
    got = launches(gd, N, M, members=members, precision="mixed", **more)
    assert set(got) & PHASES == phases
    calls = 1 if more.get("split") == "none" else 5
    assert got["update"] == (1 if folded else calls)


def test_active_members_decide(gd):
    """100 members in the handle, 8 of them stepped: the forms of 8."""
    got = launches(gd, 180, 91, members=100, active=8, precision="mixed")
    assert set(got) & PHASES == {"phase"} and got["update"] == 1
