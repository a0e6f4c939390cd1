"""What gd_autotune writes to its cache and takes from it: the form that a step
really runs under a forced setting, entries of the same settings and launch
rules only, and no form that the handle's calls cannot take."""
import re

import numpy as np
import pytest

from test_gpu_fold import env

pytestmark = pytest.mark.gpu

FAMILY = {0: "tend", 1: "phase", 2: "wphase", 3: "rphase"}
N, M = 180, 91


def tuned(gd, cache, **e):
    """autotune() and the phase launches of a step after it."""
    kw = dict(split_scheme="csp2", subcycles=2, members=2,
              zonal_tend_filter_cutoff_wavenumber=gd.cutoff_from_lat0(N, M, 75.0))
    with env(**e), gd.Dycore(N, M, 480.0, **kw) as d:
        for m in range(2):
            d.set_state(*gd.ic_balanced(N, M, seed=4 + m, nmax=8), member=m)
        choice = d.autotune(steps=2, cache=cache)
        fam = set(d.profile_kernels(1)) & set(FAMILY.values())
    assert fam == {FAMILY[choice["form"]]}
    return choice


@pytest.mark.parametrize("form", [0, 1, 3])
def test_forced_form_has_its_own_entry(gd, tmp_path, form):
    cache = tmp_path / "tune.txt"
    first = tuned(gd, cache, GD_FUSED=form)
    assert first["form"] == form
    assert tuned(gd, cache, GD_FUSED=form) == first  # from the cache
    assert len(cache.read_text().splitlines()) == 1
    tuned(gd, cache)  # another handle, not forced: timed for itself
    assert len(cache.read_text().splitlines()) == 2


@pytest.mark.parametrize("name", ["GD_STRIP", "GD_FOLD", "GD_S2TB"])
def test_forced_rules_have_their_own_entry(gd, tmp_path, name):
    cache = tmp_path / "tune.txt"
    tuned(gd, cache, **{name: 0})
    tuned(gd, cache)
    assert len(cache.read_text().splitlines()) == 2


def test_rows_form_needs_strip_tiles(gd, tmp_path):
    """Without strip tiles no call takes form 3: an entry that says so is timed
    again."""
    cache = tmp_path / "tune.txt"
    assert tuned(gd, cache, GD_STRIP=0)["form"] != 3
    line = cache.read_text().splitlines()[0]
    cache.write_text(re.sub(r"fused=\d.*", "fused=3 wpm=4 ms=1e-9", line) + "\n")
    again = tuned(gd, cache, GD_STRIP=0)
    assert again["form"] != 3 and again["ms_per_step"] > 1e-6


def test_entry_of_earlier_rules_is_timed_again(gd, tmp_path):
    """Lines without the version of the launch rules, or with another."""
    cache = tmp_path / "tune.txt"
    tuned(gd, cache)
    line = cache.read_text().splitlines()[0]
    key = line.split(" | ")[0]
    for old in (re.sub(r" v=.*", "", key), re.sub(r" v=\d+", " v=1", key)):
        cache.write_text(old + " | fused=0 wpm=4 ms=1e-9\n")
        assert tuned(gd, cache)["ms_per_step"] > 1e-6
        assert len(cache.read_text().splitlines()) == 2


def test_taken_entry_gives_the_default_bits(gd, tmp_path):
    """An entry of this library is applied without timing, and a run under each
    form gives the bits of the default run."""
    cache = tmp_path / "tune.txt"
    tuned(gd, cache)
    key = cache.read_text().splitlines()[0].split(" | ")[0]
    kw = dict(split_scheme="csp2", subcycles=2, members=2,
              zonal_tend_filter_cutoff_wavenumber=gd.cutoff_from_lat0(N, M, 75.0))
    out = []
    for form in (None, 0, 1, 3):
        with gd.Dycore(N, M, 480.0, **kw) as d:
            for m in range(2):
                d.set_state(*gd.ic_balanced(N, M, seed=4 + m, nmax=8), member=m)
            if form is not None:
                cache.write_text(f"{key} | fused={form} wpm=4 ms=1e-9\n")
                assert d.autotune(steps=2, cache=cache) == dict(fused=form != 0, form=form, upd_wpm=4,
                                                                ms_per_step=1e-9, cache=cache)
            out.append(list(d.step(3)[:3]) + [x for m in range(2) for x in d.get_state(member=m)])
    for o in out[1:]:
        for x, y in zip(o, out[0]):
            np.testing.assert_array_equal(x, y)
