"""A cache entry that gd_autotune cannot apply (workgroups or a form out of
range) is not used in any part: the shapes are timed, and a step runs."""
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["fused=1 wpm=0", "fused=1 wpm=100000", "fused=7 wpm=4", "fused=-1 wpm=4"])
def test_refused_entry_is_timed_again(gd, tmp_path, entry):
    cache = tmp_path / "tune.txt"
    N, M = 72, 37
    kw = dict(split_scheme="csp2", subcycles=2, zonal_tend_filter_cutoff_wavenumber=[6, 5, 4])
    ic = gd.ic_balanced(N, M, seed=4, nmax=8)
    out = []
    for plant in (False, True):
        with gd.Dycore(N, M, 600.0, **kw) as d:
            d.set_state(*ic)
            if plant:
                cache.write_text(re.sub(r"fused=.*", f"{entry} ms=1e-9", cache.read_text()))
            got = d.autotune(steps=2, cache=cache)
            assert got["ms_per_step"] > 1e-6 and 1 <= got["upd_wpm"] <= M and 0 <= got["form"] <= 3
            out.append(list(d.step(3)[:3]) + list(d.get_state()))
    assert len(cache.read_text().splitlines()) == 2
    for x, y in zip(*out):
        np.testing.assert_array_equal(x, y)
