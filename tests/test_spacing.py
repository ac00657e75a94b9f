"""Grid spacings that are not powers of two, where FP32 forms the quotients by
the spacing from FP64 sums instead of dividing: values of every magnitude,
subnormal numbers and zeros of both signs among them, against the oracle.
The quotients are the division's, so every array agrees bit for bit (with the
Froude cap's per-cell ATAN2, COS and SIN left to the host)."""
import numpy as np
import pytest

from common import bitwise_mismatch

pytestmark = pytest.mark.gpu

KEYS = ["U4", "V4", "ETAT", "ETAx", "ETAy", "P", "Q", "Fx", "Gy", "Eta", "U", "V", "HU", "HV", "Ubar", "Vbar", "H"]


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("dx,dy", [(1.5, 1.5), (0.7, 2.0), (2.0, 3.1), (1.0 / 3.0, 1e3), (2.0, 0.25)])
def test_matches_oracle(dx, dy, prec, gpu_available):
    import fwcases
    import fwgpu
    import fwsetup
    import oracle
    print(f"\n[spacing] {dx} x {dy} {prec}", flush=True)
    m, n = 70, 37
    c = fwcases.beach_1d(mglob=m, nglob=n, xslp=0.4 * m, xc_wk=0.2 * m, sponge_west=7.0)
    c.params.update({"PERIODIC": False, "WAVEMAKER": "NONE", "DIRECT_SPONGE": False, "DX": dx, "DY": dy,
                     "DEPTH_TYPE": "DATA"})
    c.depth = np.full((n, m), 5.0)
    st = fwsetup.build_state(c, prec)
    rng = np.random.default_rng(int(100 * dx + dy))
    rdt = st["Depth"].dtype
    shape = st["Depth"].shape
    least = -45.0 if prec == "sp" else -322.0
    for k in ("Eta", "U", "V"):
        mag = 10.0 ** np.where(rng.random(shape) < 0.5, rng.uniform(-6.0, -2.0, shape),
                               rng.uniform(least, -2.0, shape))
        # whole regions of tiny values, so that differences are tiny as well
        mag[:, : m // 3] = 10.0 ** rng.uniform(least, least + 8.0, mag[:, : m // 3].shape)
        v = mag * np.where(rng.random(mag.shape) < 0.5, -1.0, 1.0)
        st[k] = np.where(rng.random(mag.shape) < 0.1, np.copysign(0.0, v), v).astype(rdt)
    st["H"] = (st["Eta"] + st["Depth"]).astype(rdt)
    st["HU"], st["HV"] = (st["H"] * st["U"]).astype(rdt), (st["H"] * st["V"]).astype(rdt)
    st["Ubar"], st["Vbar"] = st["HU"].copy(), st["HV"].copy()
    g, o = fwgpu.Solver(st, prec, host_math=True), oracle.OracleSolver(st)
    for steps in (1, 2):
        assert g.step(steps) == (o.run(steps), (o.dt.value, o.time.value))[1]
        bad = {k: bitwise_mismatch(g.download(k), o[k]) for k in KEYS}
        assert not any(bad.values()), bad
    g.close()
    # and the production kernels against the routine-by-routine path
    g, r = fwgpu.Solver(st, prec), fwgpu.Solver(st, prec, full_state=True)
    assert g.step(3) == r.step(3)
    bad = {k: bitwise_mismatch(g.download(k), r.download(k)) for k in ("Eta", "U", "V", "Ubar", "Vbar", "H")}
    assert not any(bad.values()), bad
    g.close()
    r.close()
