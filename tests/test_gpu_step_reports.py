"""What reports on a step follows the launches the step makes: the timing hook
of the phase launch, and the benchmark's kernel names and bytes, also where
the launches without strip tiles take another form (past 6144 row tiles of
more than 1024 longitudes)."""
import pytest

from test_gpu_fold import env

pytestmark = pytest.mark.gpu

N, M, MEMBERS = 1440, 37, 30  # 6660 row tiles


def make(gd, split, **e):
    kw = dict(split_scheme=split, subcycles=2, members=MEMBERS,
              zonal_tend_filter_cutoff_wavenumber=gd.cutoff_from_lat0(N, M, 60.0))
    with env(**e):
        d = gd.Dycore(N, M, 30.0 if split == "csp2" else 5.0, **kw)
    ic = gd.ic_balanced(N, M, seed=3, nmax=6)
    for m in range(MEMBERS):
        d.set_state(*ic, member=m)
    return d


@pytest.mark.parametrize("split,e,kernel", [("csp2", {}, "k_phase"), ("csp2", dict(GD_FUSED=0), "k_tend"),
                                            ("csp2", dict(GD_STRIP=0), "k_tend"), ("none", {}, "k_tend")])
def test_timed_launch_is_the_steps(gd, split, e, kernel):
    import bench
    with make(gd, split, **e) as d:
        prof = d.profile_kernels(1)
        assert bench.phase_kernel(prof) == kernel
        if kernel == "k_tend":
            with pytest.raises(gd.DycoreError, match="fused") as err:
                d.time_kernel("phase", 2)
            assert err.value.code == 4  # GD_ERR_NOT_SUPPORTED
        else:
            assert d.time_kernel("phase", 2) > 0.0
        asked, time_kernel = [], d.time_kernel
        d.time_kernel = lambda k, reps: (asked.append(k), time_kernel(k, reps))[1]
        us, name, _ = bench._kernel_us(d, 2)
        assert us > 0.0 and name == kernel and asked == ["tend" if kernel == "k_tend" else "phase"]


@pytest.mark.parametrize("s2", [0, 1])
def test_bytes_follow_the_predictor_store(gd, s2):
    import bench
    with make(gd, "csp2", GD_S2TB=s2) as d:
        prof = d.profile_kernels(1)
        assert ("phase_s2tb" in prof) == bool(s2)
        calls = 4  # of three phases
        assert prof["phase"][0] == 3 * calls - (calls if s2 else 0)
        full, half, _, _ = d.filter_table()
        clear = [j for j in range(2, M - 3) if not full[j] and not half[j]]
        assert clear == list(range(clear[0], clear[-1] + 1))
        rows = len(clear) - 4 if s2 else 0
        assert bench.unstored_rows(d, prof) == rows
        assert (bench.tend_launch_bytes(N, M, "mixed", rows)
                == bench.tend_launch_bytes(N, M, "mixed") - 24 * N * rows)
        before = d.get_state(member=3)
        assert d.time_kernel("phase", 3) > 0.0
        for x, y in zip(d.get_state(member=3), before):
            assert (x == y).all()
