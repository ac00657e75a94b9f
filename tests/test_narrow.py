"""Domains of one and two interior cells across, where ghost cells mirror other
ghost cells: EXCHANGE against the oracle, whose fills run in the reference's
order (bc.F:631-1272).  Copies and sign changes only, so the tolerance is
none: every array bit for bit, ghost cells included."""
import numpy as np
import pytest

from common import bitwise_mismatch

pytestmark = pytest.mark.gpu

# walls on both sides; (m, n) interior cells
WALLED = [(1, 1), (1, 2), (2, 1), (2, 2), (1, 7), (7, 1), (2, 9), (9, 2), (1, 900), (900, 1), (2, 300), (300, 2)]
# periodic in y: narrow in x only
PERIODIC = [(1, 3), (2, 4), (2, 70), (1, 400)]


def narrow_state(m, n, prec, periodic=False, **params):
    """Shallow water of random depth over m x n cells, some cells dry on the
    longer domains, with random surface and velocities in the wet ones."""
    import fwcases
    import fwsetup
    rng = np.random.default_rng(100 * m + n)
    c = fwcases.beach_1d(mglob=m, nglob=n, xslp=0.4 * m, xc_wk=0.3 * m, sponge_west=min(10.0, 0.2 * m))
    dep = 2.0 + 0.2 * rng.standard_normal((n, m))
    if m * n > 6:
        dep.reshape(-1)[:: 5] = -0.3
    c.depth = dep
    c.params.update({"DEPTH_TYPE": "DATA", "PERIODIC": periodic, "WAVEMAKER": "NONE", "DIRECT_SPONGE": False,
                     "Cbrk1": 0.05, "Cbrk2": 0.02, **params})
    st = fwsetup.build_state(c, prec)
    rdt = st["Depth"].dtype
    wet = st["MASK"] > 0
    for k, a in (("Eta", 0.05), ("U", 0.1), ("V", 0.1)):
        st[k] = np.where(wet, a * rng.standard_normal(wet.shape), st.get(k, 0)).astype(rdt)
    st["H"] = np.where(wet, st["Eta"] + st["Depth"], st["H"]).astype(rdt)
    st["HU"], st["HV"] = (st["H"] * st["U"]).astype(rdt), (st["H"] * st["V"]).astype(rdt)
    st["Ubar"], st["Vbar"] = st["HU"].copy(), st["HV"].copy()
    return st


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("periodic,m,n", [(False, *s) for s in WALLED] + [(True, *s) for s in PERIODIC])
def test_exchange_matches_oracle(periodic, m, n, prec, gpu_available):
    import fwgpu
    import oracle
    print(f"\n[narrow exchange] {m} x {n} {prec} periodic={periodic}", flush=True)
    st = narrow_state(m, n, prec, periodic)
    rng = np.random.default_rng(m + 7 * n)
    rdt = st["Depth"].dtype
    M, N = st["Mloc"], st["Nloc"]
    # every array the exchange fills starts with values of its own in all ghost cells
    for k, shape in (("Eta", (N, M)), ("U", (N, M)), ("V", (N, M)), ("HU", (N, M)), ("HV", (N, M)), ("P", (N, M + 1)),
                     ("Q", (N + 1, M)), ("AGE_BREAKING", (N, M)), ("nu_break", (N, M))):
        st[k] = rng.standard_normal(shape).astype(rdt)
    st["MASK"] = rng.integers(0, 2, (N, M)).astype(np.int32)
    g, o = fwgpu.Solver(st, prec), oracle.OracleSolver(st)
    for rep in range(3):
        g.exchange()
        o.exchange()
        bad = {k: bitwise_mismatch(g.download(k), o[k])
               for k in ("Eta", "U", "V", "HU", "HV", "P", "Q", "MASK", "AGE_BREAKING", "nu_break")}
        assert not any(bad.values()), (rep, bad)
    g.close()
