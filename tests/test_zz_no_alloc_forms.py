"""gd_filter_rows_noalloc filters rows of the device's own allocations in place
and copies all others (here: pinned host memory) through the scratch array;
both must give the rows of gd_filter_rows bit for bit, and leave everything
around them alone: unflagged rows, the padding of a row, and what lies before
an offset start that is aligned to one double only."""
import ctypes as C

import numpy as np
import pytest

from test_zz_no_alloc import Hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("N,M,ld,off", [(8, 41, 8, 0), (65, 43, 67, 1), (360, 181, 360, 3), (1440, 61, 1601, 1),
                                        (2050, 31, 2050, 0)])
def test_forms_match_filter_rows(gd, N, M, ld, off, pinned):
    hip = Hip()
    cut = gd.cutoff_from_lat0(N, M, 60.0)
    x = np.random.default_rng(N).standard_normal((M, N))
    print(f"no-alloc forms N={N} M={M} ld={ld} off={off} pinned={pinned}", flush=True)
    with gd.Dycore(N, M, 60.0, zonal_tend_filter_cutoff_wavenumber=cut) as d:
        for half, rows in ((False, M), (True, M - 1)):
            ref = d.filter_rows(x[:rows].copy(), half=half)
            # the last row ends the allocation: no padding behind it
            buf = np.full(off + (rows - 1) * ld + N, -7.25)
            view = np.lib.stride_tricks.as_strided(buf[off:], (rows, N), (ld * 8, 8))
            view[:] = x[:rows]
            want = buf.copy()
            np.lib.stride_tricks.as_strided(want[off:], (rows, N), (ld * 8, 8))[:] = ref
            if pinned:
                p = C.c_void_p()
                hip.ok(hip.L.hipHostMalloc(C.byref(p), C.c_size_t(buf.nbytes), C.c_uint(0)), "hipHostMalloc")
            else:
                p = hip.alloc(buf.nbytes)
            try:
                hip.put(p, buf)
                d.filter_rows_noalloc(p.value + off * 8, half=half, ld=ld)
                got = hip.get(p, buf.shape)
            finally:
                hip.ok(hip.L.hipHostFree(p) if pinned else hip.L.hipFree(p), "free")
            np.testing.assert_array_equal(got, want)


def test_in_place_under_capture(gd):
    """Captured in a graph and replayed on new rows, beside eager calls."""
    hip = Hip()
    N, M = 180, 91
    cut = gd.cutoff_from_lat0(N, M, 60.0)
    rng = np.random.default_rng(5)
    with gd.Dycore(N, M, 60.0, zonal_tend_filter_cutoff_wavenumber=cut) as d:
        s, p = hip.stream(), hip.alloc(M * N * 8)
        graph, run = C.c_void_p(), C.c_void_p()
        hip.ok(hip.L.hipStreamBeginCapture(s, 0), "hipStreamBeginCapture")
        d.filter_rows_noalloc(p.value, stream=s.value)
        hip.ok(hip.L.hipStreamEndCapture(s, C.byref(graph)), "hipStreamEndCapture")
        hip.ok(hip.L.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)), "hipGraphInstantiate")
        for _ in range(3):
            x = rng.standard_normal((M, N))
            hip.put(p, x)
            hip.ok(hip.L.hipGraphLaunch(run, s), "hipGraphLaunch")
            hip.sync(s)
            got = hip.get(p, (M, N))
            np.testing.assert_array_equal(got, d.filter_rows(x.copy()))
            hip.put(p, x)
            d.filter_rows_noalloc(p.value)
            np.testing.assert_array_equal(hip.get(p, (M, N)), got)
        hip.ok(hip.L.hipGraphExecDestroy(run), "hipGraphExecDestroy")
        hip.ok(hip.L.hipGraphDestroy(graph), "hipGraphDestroy")
        hip.free(p)
        hip.destroy(s)
