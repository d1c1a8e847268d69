"""The lane-per-cell kernels for run-time mechanism tables (transport,
temperature recovery, source terms) against the FP64 oracle, at sizes off their
64-cell blocks and on both sides of the dispatch limits, and at temperatures
outside the fits.  Bounds: the sums involved have at most 54 + 270 terms of
either sign, each good to a few 1e-16; 1e-12 of a cell's largest value leaves
cancellation of three digits (1e-11 for the rates, whose products chain three
of them)."""
import numpy as np
import pytest

from conftest import gpu_available

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a HIP GPU")]

PATM = 1.01325e5


def _mech(name):
    from openhurricane_amd.chemistry import Mechanism

    if name == "h2air":
        return Mechanism.h2air()
    ns, nr, seed = {"syn16": (16, 60, 3), "syn24": (24, 110, 3), "syn32": (32, 150, 1),
                    "syn44": (44, 200, 3), "syn54": (54, 270, 2)}[name]
    return Mechanism.synthetic(ns, nr, seed=seed)


def _states(mech, n, seed):
    """Random compositions, one in four with absent species; T beyond both ends of the fits."""
    rng = np.random.default_rng(seed)
    t = mech.tables()
    Y = rng.uniform(0.0, 1.0, (mech.ns, n)) ** 4
    Y[:, ::4] *= rng.uniform(size=(mech.ns, len(Y[0, ::4]))) > 0.5
    Y[-1] += 1e-3
    Y /= Y.sum(0)
    T = rng.uniform(310.0, 3500.0, n)
    T[:4] = [250.0, 299.0, 5200.0, 1000.0]
    p = rng.uniform(0.5, 5.0, n) * PATM
    rho = p / (8314.46261815324 * T * (Y / t["W"][:, None]).sum(0))
    return {"T": T, "p": p, "rho": rho, "Y": np.ascontiguousarray(Y)}


def _close(a, b, tol):
    a, b = np.atleast_2d(a), np.atleast_2d(b)
    scale = np.abs(b).max(0) + 1e-300
    assert np.isfinite(a).all()
    assert (np.abs(a - b) / scale).max() <= tol


@pytest.mark.parametrize("name", ["h2air", "syn16", "syn24", "syn32", "syn44", "syn54"])
@pytest.mark.parametrize("n", [1, 63, 65])
def test_props_and_T_from_h(name, n):
    from openhurricane_amd import _lib
    from openhurricane_amd.chemistry import ChemistrySource
    from oracle import Oracle

    mech = _mech(name)
    print(f"props {name}: {n} cells", flush=True)
    st = _states(mech, max(n, 4), 7)
    st = {k: np.ascontiguousarray(v[..., :n]) for k, v in st.items()}
    opts = _lib.default_opts(kernel=2)
    cs = ChemistrySource(mech, opts=opts)
    got = cs.mix_props(st["T"], st["p"], st["Y"], hk=True)
    want = Oracle(mech).mix_props(st["T"], st["p"], st["Y"])
    for k in ("mu", "kappa", "cp", "ha"):
        np.testing.assert_allclose(got[k], want[k], rtol=1e-12, err_msg=k)
    np.testing.assert_allclose(got["Dk"], want["Dk"], rtol=1e-11)
    T0 = st["T"] * 1.03
    T = cs.T_from_h(got["ha"], st["p"], st["Y"], T0)
    # the result is held to [T_low, T_high]; else within the Newton stop (1e-4 T0)
    # squared, over a cp that varies by its own size
    np.testing.assert_allclose(T, np.clip(st["T"], opts.T_low, opts.T_high), rtol=1e-6)


@pytest.mark.parametrize("name", ["h2air", "syn24", "syn32", "syn54"])
@pytest.mark.parametrize("exact", [0, 1])
def test_source_terms_both_kernels(name, exact):
    from openhurricane_amd import _lib
    from openhurricane_amd.chemistry import ChemistrySource

    mech = _mech(name)
    n = 8193  # one cell past a block, past the dispatch limit
    print(f"source {name}: {n} cells", flush=True)
    st = _states(mech, n, 11)
    cs = ChemistrySource(mech, opts=_lib.default_opts(kernel=2, jacobian=exact))
    a = (st["T"], st["p"], st["rho"], st["Y"])
    head = tuple(np.ascontiguousarray(v[..., :300]) for v in a)  # wavefront-per-cell kernel
    for kw in ({"diag": True}, {"diag": True, "without_last": True}):
        R, D = cs.source_terms(*a, **kw)
        Rh, Dh = cs.source_terms(*head, **kw)
        _close(R[:, :300], Rh, 1e-11)
        _close(D[:, :300], Dh, 1e-11)
        Rs = cs.source_terms(*a)
        _close(Rs, R, 1e-13)
        assert np.isfinite(R).all() and np.isfinite(D).all()
    sliced = ChemistrySource(mech, opts=_lib.default_opts(kernel=2, jacobian=exact,
                                                          max_slice_cells=4000))
    Rq, Dq = sliced.source_terms(*a, diag=True, without_last=True)
    assert np.array_equal(Rq, R) and np.array_equal(Dq, D)
