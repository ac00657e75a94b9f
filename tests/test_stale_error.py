"""An error that an earlier, unrelated HIP call of the thread left behind is not
this library's: transfers, steps and the routines that wait for the device
succeed and give the same state, bit for bit, as without it."""
import numpy as np
import pytest

from common import STATE_KEYS, bitwise_mismatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["sp", "dp"])
def test_calls_succeed_after_an_unrelated_error(prec, gpu_available):
    import fwcases
    import fwgpu
    import fwsetup
    print(f"\n[stale error] {prec}", flush=True)
    c = fwcases.beach_1d(mglob=60, nglob=40, xslp=24.0, xc_wk=12.0, sponge_west=6.0)
    c.params["PERIODIC"] = False
    st = fwsetup.build_state(c, prec)
    g, r = fwgpu.Solver(st, prec), fwgpu.Solver(st, prec)
    eta = (st["Eta"] + 0.01 * st["MASK"]).astype(st["Eta"].dtype)

    def leave_error():
        # no such device: refused on the host (hipErrorInvalidDevice), and the
        # device in use stays the current one
        assert g.lib.hipSetDevice(1 << 20) != 0

    for stale in (leave_error, None):
        s = g if stale else r
        for call in (lambda: s.upload("Eta", eta), lambda: s.download("Eta"), s.estimate_dt, s.check_blowup, s.breaking,
                     lambda: s.step(1), lambda: s.time_steps(1)):
            if stale:
                stale()
            call()
    g.lib.hipGetLastError()
    bad = {k: bitwise_mismatch(g.download(k), r.download(k)) for k in STATE_KEYS}
    assert not any(bad.values()), bad
    assert np.count_nonzero(g.download("U")) > 0
    g.close()
    r.close()
