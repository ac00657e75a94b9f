"""fw_step's breaking tail: the fixed point and ghost fill of one stage done by
a workgroup of the next launch (the dispersion's, or without dispersion the
fluxes' of a small and of a large grid), the last stage's by launches of
their own (boundaries of up to and beyond 4096 ghost cells), against the
routine-by-routine path (every intermediate kept).  The same operations in
both: bit for bit."""
import numpy as np
import pytest

from common import bitwise_mismatch

pytestmark = pytest.mark.gpu

KEYS = ["Eta", "U", "V", "HU", "HV", "Ubar", "Vbar", "H", "MASK", "MASK9", "AGE_BREAKING", "nu_break"]


# 2100 x 1430 cells take the fluxes as two launches in FP32
@pytest.mark.parametrize("m,n,prec", [(40, 30, "sp"), (340, 342, "sp"), (340, 343, "sp"), (1540, 1000, "sp"), (2100, 1430, "sp"),
                                      (40, 30, "dp"), (900, 700, "dp")])
@pytest.mark.parametrize("dispersion", [False, True])
def test_step_matches_routines(m, n, prec, dispersion, gpu_available):
    import fwcases
    import fwgpu
    import fwsetup
    print(f"\n[step breaking] {m} x {n} {prec} dispersion={dispersion}", flush=True)
    c = fwcases.beach_1d(mglob=m, nglob=n, xslp=0.4 * m, xc_wk=0.2 * m, sponge_west=min(10.0, 0.1 * m))
    x = np.arange(m) + 0.5
    c.depth = np.tile(np.where(x > 0.4 * m, 4.0 - 8.0 * (x / m - 0.4), 4.0), (n, 1))
    c.params.update({"DEPTH_TYPE": "DATA", "PERIODIC": False, "VISCOSITY_BREAKING": True, "SHOW_BREAKING": True,
                     "DISPERSION": dispersion, "WAVEMAKER": "NONE", "DIRECT_SPONGE": False, "Cbrk1": 0.02, "Cbrk2": 0.01})
    st = fwsetup.build_state(c, prec)
    rng = np.random.default_rng(m + n)
    on = st["MASK"] * (st["Depth"] > 0.5)
    rdt = st["Depth"].dtype
    # steep waves and strong currents across the whole grid, the boundary cells
    # among them, and a fast rising surface (ETAT is kept as it is without
    # dispersion): ages grow at once
    wave = 0.4 * np.sin(np.arange(m + 6) / 2.5)[None, :] + 0.02 * rng.standard_normal(on.shape)
    st["Eta"] = np.where(on > 0, wave, st["Eta"]).astype(rdt)
    st["H"] = np.where(on > 0, st["Eta"] + st["Depth"], st["H"]).astype(rdt)
    st["U"] = np.where(on > 0, 3.0 * wave, 0).astype(rdt)
    st["HU"] = (st["H"] * st["U"]).astype(rdt)
    st["Ubar"] = st["HU"].copy()
    st["ETAT"] = np.where(on > 0, 6.0 * rng.random(on.shape), 0).astype(rdt)
    st["ETAx"], st["ETAy"] = (rng.standard_normal(on.shape).astype(rdt) for _ in range(2))
    g, r = fwgpu.Solver(st, prec), fwgpu.Solver(st, prec, full_state=True)
    for steps in (1, 2):
        assert g.step(steps) == r.step(steps)
        bad = {k: bitwise_mismatch(g.download(k), r.download(k)) for k in KEYS}
        assert not any(bad.values()), bad
    assert np.count_nonzero(g.download("nu_break")) > 0
    g.close()
    r.close()


# ghost cells included, 6 (Mloc + Nloc) = 4092 of them go with the fixed point, 4098
# by a launch of their own
@pytest.mark.parametrize("m,n", [(330, 340), (330, 341), (9, 661), (662, 9)])
@pytest.mark.parametrize("dispersion", [False, True])
def test_step_on_both_sides_of_the_fill_limit(m, n, dispersion, gpu_available):
    for prec in ("sp", "dp"):
        test_step_matches_routines(m, n, prec, dispersion, gpu_available)
