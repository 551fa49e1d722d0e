"""Host transfers of fields large enough for several copying threads (pieces
that the sizes do not divide) and tables kept from one geometry to the next."""
import ctypes

import numpy as np
import pytest

from turbins_amd import Solver, abi, workload as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims", [(4, 4, 4), (131, 67, 35), (259, 131, 67)])
def test_round_trip(dims):
    nx, ny, nz = dims
    c = W.case("lock64", nx=nx, ny=ny, nz=nz)
    g = Solver(W.config_for(c))
    rng = np.random.default_rng(nx)
    a, b = rng.standard_normal(g.NT), rng.standard_normal(g.NT)
    for _ in range(2):   # the staging is kept for the second pass
        g.upload("U", a)
        g.upload("C", b)
        assert np.array_equal(g.download("U").ravel(), a) and np.array_equal(g.download("C").ravel(), b)
        a, b = b, a
    g.close()


@pytest.mark.parametrize("heights", [(0.3, 0.6, 0.1, 0.6), (0.5, 0.0, 0.5)])
def test_repeated_geometry(heights):
    """Each set-up gives what a new solver's does (0: no bump)."""
    dims = dict(nx=67, ny=30, nz=18)

    def state(g):
        return [g.flags(q) for q in range(4)] + [g.download(f) for f in ("SDF_C",)]

    g = Solver(W.config_for(W.case("bump_small", **dims)))
    rng = np.random.default_rng(1)
    x, b = rng.standard_normal(g.NT), rng.standard_normal(g.NT)
    for h in heights:
        c = W.case("bump_small", bump_height=h, **dims) if h else W.case("bump_small", bump="none", **dims)
        new = Solver(W.config_for(c))
        for s in (g, new):
            s.setup_geometry(W.topography(c))
        for p, q in zip(state(g), state(new)):
            assert np.array_equal(p, q)
        for q in range(4):   # the rows of the IMMERSED nodes
            assert np.array_equal(g.helmholtz_apply(q, c["dt"], x), new.helmholtz_apply(q, c["dt"], x))
            assert np.array_equal(g.helmholtz_gs_sweeps(q, c["dt"], b, x, 3),
                                  new.helmholtz_gs_sweeps(q, c["dt"], b, x, 3))
        new.close()
    g.close()


@pytest.mark.parametrize("ny", [30, 31, 32, 33])
def test_geometry_clears_transfer_scratch(ny):
    """What a transfer left in the scratch vector (a field of NaN) stays out
    of the row padding of the signed distance, which a Poisson guess takes
    over whole: the guesses of the steps that follow are accepted.  The last
    of the reinitialisation's two buffers is the scratch vector or not, with
    the parity of its step count."""
    c = W.case("bump_small", nx=67, ny=ny, nz=18)
    g = Solver(W.config_for(c, pois_mode=abi.POIS_LEARNED_IR))
    g.upload("SCRATCH0", np.full(g.NT, np.nan))
    g.setup_geometry(W.topography(c))
    print("reinitialisation steps", g.reinit_iterations(), flush=True)
    for k, v in W.initial_fields(c, [g.flags(q) for q in range(4)]).items():
        g.upload(k, v)
    g.step(c["dt"])
    # a right-hand side whose solution the signed distance is, up to a constant
    b = g.poisson_apply(g.download("SDF_C")).reshape(19, ny + 1, 68)
    b[:-1, :-1, :-1] -= b[:-1, :-1, :-1].mean()
    b[-1], b[:, -1], b[:, :, -1] = 0.0, 0.0, 0.0
    g.upload("PRHS", b)
    st = abi.SolveStats()
    g._ok(g.L.tb_poisson_solve_guess(g.h, abi.F["SDF_C"], ctypes.byref(st)), "tb_poisson_solve_guess")
    print("guess", st.iterations, st.fallback, st.res0, flush=True)
    pois = [p for _ in range(4) for p in g.step(c["dt"]).pois]
    print([(p.iterations, p.fallback) for p in pois], flush=True)
    assert all(p.converged and not p.fallback & 2 for p in pois)
    assert np.isfinite(g.download("PHI")).all()
    g.close()
