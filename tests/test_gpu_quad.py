"""The four-cells-per-wavefront integrator against the FP64 oracle: call sizes
that leave groups or wavefronts without a cell, both reactor types, both entry
points, and calls on the two sides of each dispatch limit (one integrator runs
one cell per lane or per wavefront, the other four per wavefront).  Bounds: the
oracle's, |dT|/T <= 1e-6 and |dY| <= 1e-6 max(Y, 1e-3); between two kernels that
take the same steps an implicit solve damps the rounding differences (a few
1e-15 per evaluation), 1e-9 leaves six digits."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]


def _opts(**kw):
    from openhurricane_amd import _lib

    return _lib.default_opts(**dict(dict(atol=1e-10, rtol=1e-6, atol_inc=1e-10, rtol_inc=1e-6), **kw))


def _states(mech, n, seed):
    from openhurricane_amd.sampler import h2air_states

    st = h2air_states(mech.species, mech.tables()["W"], n, seed=seed)
    return {k: np.ascontiguousarray(st[k]) for k in ("T", "p", "rho", "Y")}


@pytest.mark.parametrize("n", [1, 3, 5, 66])
@pytest.mark.parametrize("flow,exact", [(0, 0), (1, 1)])
def test_small_compiled_calls_match_oracle(h2mech, h2oracle, n, flow, exact):
    from openhurricane_amd.chemistry import ChemistrySource

    o = _opts(flow_type=flow, jacobian=exact)
    cs = ChemistrySource(h2mech, opts=o)
    assert cs.kernel_name.startswith("lane:")
    print(f"{n} cells, flow {flow}", flush=True)
    st = _states(h2mech, n, 3 + n)
    dt = np.full(n, 1e-6)
    To, Yo, sub_o, s_o = h2oracle.solve_update(o, st["T"], st["p"], st["rho"], st["Y"], dt, 1.0)
    T, Y = st["T"].copy(), st["Y"].copy()
    sub, s = cs.solve_update(T, st["p"], st["rho"], Y, dt, 1.0)
    assert (np.abs(T - To) / To).max() <= 1e-6
    assert (np.abs(Y - Yo) / np.maximum(Yo, 1e-3)).max() <= 1e-6
    np.testing.assert_allclose(sub, sub_o, rtol=1e-3)
    assert s["cells"] == s_o["cells"] and abs(s["steps"] - s_o["steps"]) <= 0.01 * s_o["steps"] + 1
    R, _, _ = cs.solve(st["T"], st["p"], st["rho"], st["Y"], dt, 1.0)
    Ro = h2oracle.solve(o, st["T"], st["p"], st["rho"], st["Y"], dt, 1.0)[0]
    assert (np.abs(R - Ro) / np.abs(Ro).max(0)).max() <= 1e-6


@pytest.mark.parametrize("kernel,limit", [(0, 1 << 17), (2, 4096)])
@pytest.mark.parametrize("flow", [0, 1])
def test_both_sides_of_the_dispatch_limit_agree(h2mech, kernel, limit, flow):
    from openhurricane_amd.chemistry import ChemistrySource

    cs = ChemistrySource(h2mech, opts=_opts(flow_type=flow, kernel=kernel))
    m = 512
    st = _states(h2mech, m, 21)
    res = []
    for n in (limit - 1, limit, limit + 1):
        print(f"kernel {kernel}: {n} cells", flush=True)
        idx = np.arange(n) % m
        T, Y = st["T"][idx], np.ascontiguousarray(st["Y"][:, idx])
        sub, s = cs.solve_update(T, np.ascontiguousarray(st["p"][idx]),
                                 np.ascontiguousarray(st["rho"][idx]), Y, np.full(n, 1e-7), 1.0)
        # a cell's result does not depend on its place
        np.testing.assert_array_equal(T, T[:m][idx])
        np.testing.assert_array_equal(Y, Y[:, :m][:, idx])
        assert s["cells"] == n
        res.append((T[:m], Y[:, :m], sub[:m]))
    for T, Y, sub in res[1:]:
        np.testing.assert_allclose(T, res[0][0], rtol=1e-9)
        np.testing.assert_allclose(Y, res[0][1], rtol=1e-9, atol=1e-12)
        np.testing.assert_allclose(sub, res[0][2], rtol=1e-9)


def test_cells_without_a_number_fail_and_leave_the_others(h2mech):
    """A cell with a NaN composition ends as failed; its neighbours in the
    wavefront keep their results bit for bit."""
    from openhurricane_amd import _lib
    from openhurricane_amd.chemistry import ChemistrySource

    cs = ChemistrySource(h2mech, opts=_opts())
    n = 9
    st = _states(h2mech, n, 5)
    dt = np.full(n, 1e-6)
    T, Y = st["T"].copy(), st["Y"].copy()
    cs.solve_update(T, st["p"], st["rho"], Y, dt, 1.0)
    Tb, Yb = st["T"].copy(), st["Y"].copy()
    Yb[0, 2] = np.nan
    with pytest.raises(_lib.OhcError):
        cs.solve_update(Tb, st["p"], st["rho"], Yb, dt, 1.0)
    keep = np.arange(n) != 2
    if np.isfinite(Tb[keep]).all() and not np.array_equal(Tb, st["T"]):
        np.testing.assert_array_equal(Tb[keep], T[keep])
        np.testing.assert_array_equal(Yb[:, keep], Y[:, keep])


@pytest.mark.parametrize("integrator,n", [(2, 67), (0, (1 << 17) + 5)])
@pytest.mark.parametrize("flow", [0, 1])
def test_lane_kernel_outside_the_fits(h2mech, h2oracle, integrator, n, flow):
    """One cell per lane at temperatures below, inside and above the thermo fits
    (clamped there), in one wavefront; cells inside keep their bits whatever
    their neighbours are."""
    from openhurricane_amd.chemistry import ChemistrySource

    o = _opts(flow_type=flow, integrator=integrator, T_threshold=100.0)
    cs = ChemistrySource(h2mech, opts=o)
    m = 67
    st = _states(h2mech, m, 33)
    lo, hi = h2mech.tables()["Tlow"].max(), h2mech.tables()["Thigh"].min()
    Tx = st["T"].copy()
    Tx[::5] = lo - 40.0
    Tx[3::11] = hi + 60.0
    out = (Tx < lo) | (Tx > hi)
    assert 0 < out.sum() < m
    idx = np.arange(n) % m
    res = {}
    for name, T0 in (("mixed", Tx), ("inside", st["T"])):
        print(f"integrator {integrator}, {n} cells, {name}", flush=True)
        T, Y = T0[idx].copy(), np.ascontiguousarray(st["Y"][:, idx])
        rho = np.ascontiguousarray((st["rho"] * st["T"] / T0)[idx])
        cs.solve_update(T, np.ascontiguousarray(st["p"][idx]), rho, Y, np.full(n, 1e-8), 1.0)
        res[name] = (T, Y)
    np.testing.assert_array_equal(res["mixed"][0][~out[idx]], res["inside"][0][~out[idx]])
    np.testing.assert_array_equal(res["mixed"][1][:, ~out[idx]], res["inside"][1][:, ~out[idx]])
    To, Yo, _, _ = h2oracle.solve_update(o, Tx, st["p"], st["rho"] * st["T"] / Tx, st["Y"],
                                         np.full(m, 1e-8), 1.0)
    T, Y = res["mixed"][0][:m], res["mixed"][1][:, :m]
    assert (np.abs(T - To) / To).max() <= 1e-6
    assert (np.abs(Y - Yo) / np.maximum(Yo, 1e-3)).max() <= 1e-6


@pytest.mark.parametrize("flow", [0, 1])
def test_compiled_limit_agrees(h2mech, flow):
    """98,304 and 98,305 cells: four cells per wavefront and one cell per lane."""
    from openhurricane_amd.chemistry import ChemistrySource

    cs = ChemistrySource(h2mech, opts=_opts(flow_type=flow))
    m, res = 500, []
    st = _states(h2mech, m, 22)
    for n in (3 << 15, (3 << 15) + 1):
        print(f"{n} cells", flush=True)
        idx = np.arange(n) % m
        T, Y = st["T"][idx], np.ascontiguousarray(st["Y"][:, idx])
        sub, s = cs.solve_update(T, np.ascontiguousarray(st["p"][idx]),
                                 np.ascontiguousarray(st["rho"][idx]), Y, np.full(n, 1e-7), 1.0)
        np.testing.assert_array_equal(T, T[:m][idx])
        res.append((T[:m], Y[:, :m], sub[:m], s["steps"] / n))
    np.testing.assert_allclose(res[1][0], res[0][0], rtol=1e-9)
    np.testing.assert_allclose(res[1][1], res[0][1], rtol=1e-9, atol=1e-12)
    np.testing.assert_allclose(res[1][2], res[0][2], rtol=1e-9)
    assert abs(res[1][3] - res[0][3]) <= 0.01 * res[0][3]


def test_cold_neighbours_take_the_guarded_pass(h2mech):
    """A wavefront in which one cell's equilibrium constants pass 1e100 (150 K)
    evaluates the reactions with all limits; the other cells keep their bits."""
    from openhurricane_amd.chemistry import ChemistrySource

    cs = ChemistrySource(h2mech, opts=_opts(T_threshold=100.0))
    n, m = (1 << 17) + 64, 64
    st = _states(h2mech, m, 41)
    idx = np.arange(n) % m
    res = []
    for cold in (False, True):
        T0 = st["T"].copy()
        if cold:
            T0[7] = 150.0
        T, Y = T0[idx], np.ascontiguousarray(st["Y"][:, idx])
        print("cold", cold, flush=True)
        cs.solve_update(T, np.ascontiguousarray(st["p"][idx]),
                        np.ascontiguousarray((st["rho"] * st["T"] / T0)[idx]), Y,
                        np.full(n, 1e-8), 1.0)
        assert np.isfinite(T).all() and np.isfinite(Y).all()
        res.append((T, Y))
    keep = idx != 7
    np.testing.assert_array_equal(res[1][0][keep], res[0][0][keep])
    np.testing.assert_array_equal(res[1][1][:, keep], res[0][1][:, keep])
