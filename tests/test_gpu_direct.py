"""The direct solver of the shifted stencil behind the Newton corrections."""
import numpy as np
import pytest

from helpers import L, axes_for, grain_radius

pytestmark = pytest.mark.gpu


def _axes(kind, dims):
    return [axes_for(kind, n)[0][0] for n in dims]


# extents around the 16- and 32-point tiles and the 8- and 16-deep products of
# the matrix-core transforms, below a tile, and with factors of 3; enough
# points for the 32-point tiles in the last two
SIZES = [(3, 2, 4), (6, 12, 24), (16, 8, 32), (24, 48, 16), (32, 12, 96), (64, 64, 64), (96, 128, 192)]


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["eqst", "sist", "hyst"])
@pytest.mark.parametrize("dims", SIZES)
def test_one_correction_solves_a_nearly_uniform_box(ctx, kind, dims, prec):
    """rho = 1 + d, |d| <= 1e-4, from phi = 0: e = exp(phi) = 1 = c, so the first correction x solves
    J x = -F exactly and |x| <= max|d| (maximum principle, c = 1).  What is left is the nonlinear term
    exp(x) - 1 - x <= 0.51 |x|^2 <= 5.1e-9 (an FP32 correction adds its rounding, 1e-4 of max|d| times the
    condition of the transforms at most: a few 1e-9).  A V-cycle leaves more than 1e-6."""
    import kielflow_amd as kf
    print("direct", kind, dims, prec, flush=True)
    g = kf.Grid(ctx, _axes(kind, dims))
    d = np.random.default_rng(5).uniform(-1e-4, 1e-4, dims)
    p = kf.Poisson(g, kf.KF_FP64 if prec == "fp64" else kf.KF_MIXED, tol=6e-9 if prec == "fp64" else 3e-8, max_it=1)
    phi, rho = g.rfield(), ctx.to_device(1.0 + d)
    it, res, code = p.solve(phi, rho, raise_on_error=False)
    assert code == kf.api.KF_OK and it <= 1, (it, res)
    assert np.abs(phi.get()).max() <= 1.01e-4
    p.close()
    g.close()


@pytest.mark.parametrize("kind,dims", [("eqst", (48, 32, 96)), ("sist", (32, 48, 24)), ("hyst", (24, 64, 32))])
def test_direct_and_multigrid_corrections_agree(ctx, monkeypatch, kind, dims):
    """Both stop at the same residual of the same equation: the solutions differ by at most the two
    residuals, 2 tol max|rho| / min e, where exp(phi) > 0.5."""
    import kielflow_amd as kf
    axes = _axes(kind, dims)
    ln_n, nd, _ = kf.setup_host(axes, seed=2, amp=1e-3, Q=-0.2, a=2.0 * grain_radius(kind, dims[0]))
    rho = np.exp(ln_n) + nd
    tol, out = 1e-11, []
    for direct in ("1", "0"):
        monkeypatch.setenv("KF_DIRECT", direct)
        g = kf.Grid(ctx, axes)
        p = kf.Poisson(g, kf.KF_FP64, tol=tol, max_it=60)
        phi = g.rfield()
        it, res, _ = p.solve(phi, ctx.to_device(rho))
        assert res <= tol
        out.append(phi.get())
        p.close()
        g.close()
    assert np.exp(out[0]).min() > 0.5
    assert np.abs(out[0] - out[1]).max() <= 4 * tol * np.abs(rho).max()


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["eqst", "sist"])
def test_strongly_varying_coefficient_falls_back_to_multigrid(ctx, kind, prec):
    """A half box at rho = 60 beside one at 0.02: exp(phi) spans three decades, one shift contracts slowly,
    and multigrid takes the solve to its tolerance, in this solve and in later ones."""
    import kielflow_amd as kf
    n = 32
    axes = _axes(kind, (n, n, n))
    rho = np.full((n, n, n), 0.02)
    rho[: n // 2] = 60.0
    g = kf.Grid(ctx, axes)
    p = kf.Poisson(g, kf.KF_FP64 if prec == "fp64" else kf.KF_MIXED, tol=1e-9, max_it=100)
    drho = ctx.to_device(rho)
    for _ in range(4):
        phi = ctx.to_device(np.log(rho))
        it, res, code = p.solve(phi, drho)
        assert code == kf.api.KF_OK and res <= 1e-9
        # the equation holds: the solver's residual is its own kernel's, this one an independent call
        assert p.residual(phi, drho) <= 2e-9
    p.close()
    g.close()


def test_axis_without_mirror_symmetry_takes_multigrid(ctx):
    """A hyperbolic axis that does not start at -L/2 has no even and odd modes: the solve still converges."""
    import kielflow_amd as kf
    n = 24
    axes = [kf.axis(kf.HYST, n, -0.5 * L + 0.3, L, 3.0), kf.axis(kf.EQST, n, -0.5 * L, L),
            kf.axis(kf.EQST, n, -0.5 * L, L)]
    g = kf.Grid(ctx, axes)
    p = kf.Poisson(g, kf.KF_FP64, tol=1e-10, max_it=100)
    rho = 1.0 + 0.1 * np.random.default_rng(1).uniform(-1, 1, (n, n, n))
    phi = g.rfield()
    it, res, code = p.solve(phi, ctx.to_device(rho))
    assert code == kf.api.KF_OK and res <= 1e-10


@pytest.mark.parametrize("kind,dims,prec,peak,mean", [
    ("eqst", (96, 64, 96), "fp64", 1 / 512, 1 / 128), ("eqst", (64, 96, 128), "mixed", 1 / 512, 1 / 128),
    ("eqst", (24, 24, 24), "fp64", 1 / 512, 1 / 128), ("sist", (64, 48, 64), "fp64", 1 / 128, 1 / 64),
    ("hyst", (64, 64, 64), "mixed", 1 / 128, 1 / 64)])
def test_direct_solve_error_is_a_multigrid_solves(ctx, kind, dims, prec, peak, mean):
    """A direct correction leaves a smooth residual F, whose error is F / e where a V-cycle's rough one is far
    less: direct solves stop at max|F| <= tol max(peak max|rho|, mean c), c = max(mean e, 0.55 max e), so the
    error is at most that over min e (maximum principle), and the reference's own, 2e-13 max|rho| / min e."""
    import kielflow_amd as kf
    axes = _axes(kind, dims)
    a = grain_radius(kind, dims[0])
    for seed in (1, 2, 3):
        ln_n, nd, _ = kf.setup_host(axes, seed=seed, amp=1e-3, Q=-0.3, a=a)
        rho = np.exp(ln_n + 0.1 * np.sin(np.arange(dims[1]) * 2 * np.pi / dims[1] + seed)[None, :, None]) + nd
        out = []
        for tol in (1e-10, 2e-13):
            g = kf.Grid(ctx, axes)
            p = kf.Poisson(g, kf.KF_FP64 if prec == "fp64" or tol < 1e-10 else kf.KF_MIXED, tol=tol, max_it=60)
            phi = g.rfield()
            p.solve(phi, ctx.to_device(rho))
            out.append(phi.get())
            p.close()
            g.close()
        e, top = np.exp(out[1]), np.abs(rho).max()
        c = max(e.mean(), 0.55 * e.max())
        bound = (1e-10 * max(peak * top, mean * min(c, top)) + 2e-13 * top) / e.min()
        err = np.abs(out[0] - out[1]).max()
        print("direct error", kind, dims, prec, seed, err, "bound", bound, flush=True)
        assert err <= bound


def test_other_switches_leave_the_corrections_direct(ctx, monkeypatch):
    """Only KF_DIRECT selects the corrector: a switch of the V-cycle or of the right-hand side, set to any value,
    changes neither the corrections of a direct solve nor its result."""
    import kielflow_amd as kf
    axes = _axes("eqst", (24, 32, 16))
    ln_n, nd, _ = kf.setup_host(axes, seed=2, amp=1e-3, Q=-0.2, a=2.0)
    rho, out = ctx.to_device(np.exp(ln_n) + nd), {}
    for name in ("none", "KF_COARSE_N", "KF_COARSE_WAVE", "KF_PRECOND_COPY", "KF_RHO_STATE", "KF_DIRECT"):
        if name != "none":
            monkeypatch.setenv(name, "0" if name == "KF_DIRECT" else "1")
        g = kf.Grid(ctx, axes)
        p = kf.Poisson(g, kf.KF_FP64, tol=1e-10, max_it=60)
        phi = g.rfield()
        it, _, _ = p.solve(phi, rho)
        out[name] = (it, phi.get())
        p.close()
        g.close()
        monkeypatch.delenv(name, raising=False)
    for name in ("KF_COARSE_N", "KF_COARSE_WAVE", "KF_PRECOND_COPY", "KF_RHO_STATE"):
        assert out[name][0] == out["none"][0] and np.array_equal(out[name][1], out["none"][1]), name
    assert not np.array_equal(out["KF_DIRECT"][1], out["none"][1])


def _two_halves(kind, n):
    rho = np.full((n, n, n), 0.02)
    rho[: n // 2] = 60.0
    return _axes(kind, (n, n, n)), rho


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["eqst", "sist"])
def test_a_budget_that_multigrid_meets_is_met(ctx, monkeypatch, kind, prec):
    """Corrections that stall do not count against the budget of the multigrid that takes over."""
    import kielflow_amd as kf
    axes, rho = _two_halves(kind, 32)
    budget = 100
    for direct in ("0", "1"):
        monkeypatch.setenv("KF_DIRECT", direct)
        g = kf.Grid(ctx, axes)
        p = kf.Poisson(g, kf.KF_FP64 if prec == "fp64" else kf.KF_MIXED, tol=1e-9, max_it=budget)
        phi = ctx.to_device(np.log(rho))
        it, res, code = p.solve(phi, ctx.to_device(rho))
        assert code == kf.api.KF_OK and res <= 1e-9
        if direct == "0":
            budget = it + 2
        p.close()
        g.close()


def test_residual_leaves_the_solver_alone(ctx):
    """kf_poisson_residual between solves does not change which corrector the next ones take."""
    import kielflow_amd as kf
    axes, rho = _two_halves("eqst", 32)
    drho, counts = ctx.to_device(rho), []
    for between in (False, True):
        g = kf.Grid(ctx, axes)
        p = kf.Poisson(g, kf.KF_FP64, tol=1e-9, max_it=100)
        its = []
        for _ in range(4):
            phi = ctx.to_device(np.log(rho))
            its.append(p.solve(phi, drho)[0])
            if between:
                p.residual(phi, drho)
        counts.append(its)
        p.close()
        g.close()
    assert counts[0] == counts[1] and counts[0][2] < counts[0][0], counts
