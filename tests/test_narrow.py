"""Domains of one and two interior cells across, where ghost cells mirror other
ghost cells: EXCHANGE against the oracle, whose fills run in the reference's
order (bc.F:631-1272); whole steps of the production path and of batches
against the routine-by-routine path, and that against the oracle.  The same
operations everywhere, so the tolerance is none: every array bit for bit,
ghost cells included (against the oracle with the Froude cap's ATAN2, COS and
SIN left to the host)."""
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


STEP_KEYS = ["Eta", "Eta0", "U", "V", "U0", "V0", "HU", "HV", "Ubar", "Vbar", "Ubar0", "Vbar0", "H", "MASK", "MASK9",
             "AGE_BREAKING", "nu_break", "DepthX", "DepthY", "P", "Q"]
OPTIONS = [{}, {"DISPERSION": False}, {"VISCOSITY_BREAKING": False}, {"DIRECT_SPONGE": True},
           {"SHOW_BREAKING": False, "DX": 1.5, "DY": 1.5},
           {"VISCOSITY_BREAKING": False, "DIFFUSION_SPONGE": True, "FRICTION_SPONGE": True}]


# (three cells are the least that take the merged passes, whose threads write
# only the ghost cells that mirror an interior cell)
@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("m,n", [(1, 1), (1, 2), (2, 1), (2, 2), (7, 1), (2, 9), (1, 130), (150, 2), (3, 3), (3, 8), (4, 5)])
def test_steps_match_routines_and_oracle(m, n, prec, gpu_available):
    import fwgpu
    import oracle
    for opt in OPTIONS:
        print(f"\n[narrow step] {m} x {n} {prec} {opt}", flush=True)
        st = narrow_state(m, n, prec, **opt)
        g, r = fwgpu.Solver(st, prec), fwgpu.Solver(st, prec, full_state=True)
        h, o = fwgpu.Solver(st, prec, host_math=True), oracle.OracleSolver(st)
        for steps in (1, 2):
            assert g.step(steps) == r.step(steps)
            bad = {k: bitwise_mismatch(g.download(k), r.download(k)) for k in STEP_KEYS}
            assert not any(bad.values()), bad
            assert h.step(steps) == (o.run(steps), (o.dt.value, o.time.value))[1]
            bad = {k: bitwise_mismatch(h.download(k), o[k]) for k in STEP_KEYS}
            assert not any(bad.values()), bad
        for s in (g, r, h):
            s.close()


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("opt", OPTIONS[:4])
def test_batch_matches_members_alone(opt, prec, gpu_available):
    import fwgpu
    print(f"\n[narrow batch] {prec} {opt}", flush=True)
    sts = [narrow_state(m, n, prec, DT_fixed=0.02, **opt) for m, n in ((40, 30), (1, 7), (2, 2), (9, 2), (3, 3))]
    alone, gs = ([fwgpu.Solver(st, prec) for st in sts] for _ in range(2))
    b = fwgpu.Batch(gs)
    for steps in (1, 2, 4):
        b.step(steps)
        for g, a in zip(gs, alone):
            a.step(steps)
            assert g.clock == a.clock
            bad = {k: bitwise_mismatch(g.download(k), a.download(k)) for k in STEP_KEYS}
            assert not any(bad.values()), (g.M, g.N, bad)
    b.close()
    for s in gs + alone:
        s.close()
