"""The line solves (k_trid_fac, k_trid_solve) at the sizes where their
chunking can go wrong, against the oracle: lines shorter than one check
group, of whole and partial chunks (32 and 64 rows) and groups (8 and 16),
longer than what fits into LDS (FP32 beyond 2112 rows, FP64 beyond 1024),
partial blocks of 16 lines, rows that are kept (MASK9 = 0) and numerators
that decay to zero.  Every quantity is the same correctly rounded operation
as the oracle's, so the tolerance is none: every array bit for bit (with the
Froude cap's per-cell ATAN2, COS and SIN left to the host, as there)."""
import numpy as np
import pytest

from common import bitwise_mismatch

pytestmark = pytest.mark.gpu

KEYS = ["Eta", "U", "V", "HU", "HV", "Ubar", "Vbar", "H", "MASK", "MASK9", "U4", "V4", "P", "Q", "nu_break"]


def _state(m, n, prec, visc, quiet, periodic=False):
    """A sloping beach that dries at its east end, with random small waves in
    its western part only when quiet is set (still water elsewhere)."""
    import fwcases
    import fwsetup
    c = fwcases.beach_1d(mglob=m, nglob=n, xslp=0.4 * m, xc_wk=0.2 * m, sponge_west=min(10.0, 0.1 * m))
    x = np.arange(m) + 0.5
    c.depth = np.tile(np.where(x > 0.4 * m, 4.0 - 8.0 * (x / m - 0.4), 4.0), (n, 1))
    c.params.update({"DEPTH_TYPE": "DATA", "PERIODIC": periodic, "VISCOSITY_BREAKING": visc, "WAVEMAKER": "NONE",
                     "DIRECT_SPONGE": False})
    st = fwsetup.build_state(c, prec)
    rng = np.random.default_rng(m * 1000 + n)
    on = st["MASK"] * (st["Depth"] > 1.0)
    if quiet:
        on = on * (np.arange(m + 6) < 0.3 * (m + 6))[None, :]
    rdt = st["Depth"].dtype
    for k, a in (("Eta", 0.05), ("U", 0.1), ("V", 0.1)):
        st[k] = np.where(on > 0, (a * rng.standard_normal(on.shape)), st.get(k, 0)).astype(rdt)
    st["H"] = np.where(on > 0, st["Eta"] + st["Depth"], st["H"]).astype(rdt)
    st["HU"], st["HV"] = (st["H"] * st["U"]).astype(rdt), (st["H"] * st["V"]).astype(rdt)
    st["Ubar"], st["Vbar"] = st["HU"].copy(), st["HV"].copy()
    return st


SIZES = [(3, 3), (9, 17), (16, 15), (31, 33), (64, 16), (65, 129), (127, 48), (200, 3), (1023, 5), (1025, 7),
         (2048, 3), (2113, 4), (5, 2300)]


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("m,n", SIZES)
def test_lines_match_oracle(m, n, prec, gpu_available):
    import fwgpu
    import oracle
    for visc, quiet in ((True, True), (False, False)):
        print(f"\n[line solves] {m} x {n} {prec} viscosity={visc} quiet={quiet}", flush=True)
        st = _state(m, n, prec, visc, quiet)
        g, o = fwgpu.Solver(st, prec, host_math=True), oracle.OracleSolver(st)
        for steps in (1, 2):
            assert g.step(steps) == (o.run(steps), (o.dt.value, o.time.value))[1]
            bad = {k: bitwise_mismatch(g.download(k), o[k]) for k in KEYS}
            assert not any(bad.values()), bad
        # and routine by routine: c' beside ESTIMATE_HUV's own kernel
        g.dispersion(); o.dispersion()
        g.fluxes(); o.fluxes()
        g.sources(); o.sources()
        g.estimate_huv(2); o.estimate_huv(2)
        bad = {k: bitwise_mismatch(g.download(k), o[k]) for k in ("Eta", "U", "V", "HU", "HV")}
        assert not any(bad.values()), bad
        g.close()


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("m,n", [(40, 3), (333, 4), (64, 21)])
def test_periodic_lines_match_oracle(m, n, prec, gpu_available):
    import fwgpu
    import oracle
    print(f"\n[line solves] periodic {m} x {n} {prec}", flush=True)
    st = _state(m, n, prec, True, False, periodic=True)
    g, o = fwgpu.Solver(st, prec, host_math=True), oracle.OracleSolver(st)
    assert g.step(3) == (o.run(3), (o.dt.value, o.time.value))[1]
    bad = {k: bitwise_mismatch(g.download(k), o[k]) for k in KEYS}
    assert not any(bad.values()), bad
    g.close()


# periodic y lines: all in one workgroup (up to 320 columns in fw_step, 256 by
# routine, 128 KB of a plane), one more column, one more row, a remainder of a
# wavefront, and many
@pytest.mark.parametrize("m,n,prec", [(64, 16, "sp"), (256, 20, "sp"), (257, 20, "sp"), (320, 102, "sp"), (320, 103, "sp"),
                                      (321, 20, "sp"), (130, 252, "sp"), (130, 253, "sp"), (700, 33, "sp"),
                                      (320, 51, "dp"), (320, 52, "dp"), (321, 17, "dp"), (129, 130, "dp")])
def test_periodic_y_lines_match_oracle(m, n, prec, gpu_available):
    import fwgpu
    import oracle
    print(f"\n[line solves] periodic y {m} x {n} {prec}", flush=True)
    st = _state(m, n, prec, True, False, periodic=True)
    g, o = fwgpu.Solver(st, prec, host_math=True), oracle.OracleSolver(st)
    assert g.step(2) == (o.run(2), (o.dt.value, o.time.value))[1]
    bad = {k: bitwise_mismatch(g.download(k), o[k]) for k in KEYS}
    assert not any(bad.values()), bad
    g.dispersion(); o.dispersion()
    g.fluxes(); o.fluxes()
    g.sources(); o.sources()
    g.estimate_huv(2); o.estimate_huv(2)
    bad = {k: bitwise_mismatch(g.download(k), o[k]) for k in ("Eta", "U", "V", "HU", "HV")}
    assert not any(bad.values()), bad
    g.close()


# x lines too long for LDS (FP32 beyond 2112 rows, FP64 beyond 1024): their d'
# goes through memory, periodic domains and batches included
@pytest.mark.parametrize("m,n,prec", [(2112, 4, "sp"), (2113, 4, "sp"), (3000, 5, "sp"), (1024, 4, "dp"), (1025, 4, "dp"),
                                      (2300, 5, "dp")])
def test_long_periodic_lines_match_oracle(m, n, prec, gpu_available):
    import fwgpu
    import oracle
    print(f"\n[line solves] long periodic {m} x {n} {prec}", flush=True)
    for visc in (True, False):
        st = _state(m, n, prec, visc, False, periodic=True)
        g, o = fwgpu.Solver(st, prec, host_math=True), oracle.OracleSolver(st)
        assert g.step(2) == (o.run(2), (o.dt.value, o.time.value))[1]
        bad = {k: bitwise_mismatch(g.download(k), o[k]) for k in KEYS}
        assert not any(bad.values()), bad
        g.close()
        # and the production kernels against the routine-by-routine path
        g, r = fwgpu.Solver(st, prec), fwgpu.Solver(st, prec, full_state=True)
        assert g.step(3) == r.step(3)
        bad = {k: bitwise_mismatch(g.download(k), r.download(k)) for k in KEYS}
        assert not any(bad.values()), bad
        g.close()
        r.close()


@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("periodic", [False, True])
def test_batch_with_a_long_member(periodic, prec, gpu_available):
    """One member past the LDS limit puts every member's lines on the path
    through memory: each as alone, where the short ones stay in LDS."""
    import fwgpu
    long = 2113 if prec == "sp" else 1025
    sizes = [(long, 4), (65, 7), (130, 20), (16, 5)] if periodic else [(long, 4), (65, 7), (7, 130), (5, long)]
    print(f"\n[line solves] batch {sizes} {prec}", flush=True)
    sts = [dict(_state(m, n, prec, True, False, periodic=periodic), FIXED_DT=1, DT_fixed=0.03125) for m, n in sizes]
    gs, alone = ([fwgpu.Solver(st, prec) for st in sts] for _ in range(2))
    b = fwgpu.Batch(gs)
    b.step(3)
    for g, a in zip(gs, alone):
        a.step(3)
        assert g.clock == a.clock
        bad = {k: bitwise_mismatch(g.download(k), a.download(k)) for k in KEYS}
        assert not any(bad.values()), (g.M, g.N, bad)
    b.close()
    for s in gs + alone:
        s.close()


# whole steps of the production path at the sizes whose edge cells mirror across
# several walls, against the routine-by-routine path; wet everywhere (MASK9
# stays 1, and the second stage forms no c') or drying
@pytest.mark.parametrize("prec", ["sp", "dp"])
@pytest.mark.parametrize("m,n", [(3, 3), (3, 8), (8, 3), (4, 5), (6, 6), (7, 31), (33, 5), (64, 16), (65, 129)])
@pytest.mark.parametrize("dry", [False, True])
def test_small_production_steps_match_routines(dry, m, n, prec, gpu_available):
    import fwgpu
    for visc, sponge in ((True, True), (False, True), (True, False), (False, False)):
        print(f"\n[line solves] production {m} x {n} {prec} dry={dry} viscosity={visc} sponge={sponge}", flush=True)
        st = _state(m, n, prec, visc, False)
        if not dry:
            st.update(_wet(st))
        st = dict(st, DIRECT_SPONGE=int(sponge))
        st["SPONGE"] = 1.0 + 0.5 * np.random.default_rng(m).random(st["SPONGE"].shape).astype(st["SPONGE"].dtype)
        g, r = fwgpu.Solver(st, prec), fwgpu.Solver(st, prec, full_state=True)
        for steps in (1, 2, 3):
            assert g.step(steps) == r.step(steps)
            bad = {k: bitwise_mismatch(g.download(k), r.download(k)) for k in KEYS}
            assert not any(bad.values()), bad
        g.close()
        r.close()


def _wet(st):
    """The state's waves over a flat bottom."""
    N, M = st["Depth"].shape
    d = {k: np.full_like(st[k], 3.0) for k in ("Depth", "DepthX", "DepthY")}
    d.update(MASK=np.ones((N, M), np.int32), MASK9=np.ones((N, M), np.int32))
    d["Eta"] = np.where(st["MASK"] > 0, st["Eta"], 0).astype(st["Eta"].dtype)
    d["H"] = (d["Eta"] + d["Depth"]).astype(st["H"].dtype)
    return d
