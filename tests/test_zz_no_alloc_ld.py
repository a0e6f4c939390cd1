"""gd_filter_rows_noalloc refuses a leading dimension whose row offsets do not
fit 63 bits, before it looks at the memory.  Taken modulo 2^64 the span of such
calls can be one row (the last flagged full row is row 32 of 34, and 32 * 2^56 *
8 = 2^64), which would pass for rows inside the allocation while the rows
between lie anywhere."""
import numpy as np
import pytest

from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ld", [2**56, 2**60, 2**61, 2**63 - 1])
def test_wrapping_ld_is_refused(gd, ld):
    hip = Hip()
    N, M = 64, 34
    x = np.random.default_rng(3).standard_normal((M, N))
    with gd.Dycore(N, M, 60.0, zonal_tend_filter_cutoff_wavenumber=[5, 4, 3]) as d:
        p = hip.alloc(x.nbytes)
        for half in (False, True):
            hip.put(p, x)
            with pytest.raises(gd.DycoreError, match="ld too large") as e:
                d.filter_rows_noalloc(p.value, half=half, ld=ld)
            assert e.value.code == gd.GD_ERR_INVALID_ARG
            np.testing.assert_array_equal(hip.get(p, x.shape), x)
        # (the handle still filters)
        d.filter_rows_noalloc(p.value)
        np.testing.assert_array_equal(hip.get(p, x.shape), d.filter_rows(x.copy()))
        hip.free(p)
