"""The y and z passes of a transform on x planes in LDS against the separate passes (KF_PLANES=0)."""
import numpy as np
import pytest

from helpers import axes_for

pytestmark = pytest.mark.gpu

# y and z extents at the ends of the plane passes' range, factors of 3 in
# either, planes whose columns take two shares of the threads (128 x 128 in
# FP64), and x extents below, at and off the other two; planes of 10 waves and
# more than 512 workgroups of four fields (the penalization pass without its
# early loads)
DIMS = [(16, 16, 16), (12, 24, 32), (6, 16, 192), (24, 128, 16), (16, 48, 96), (8, 64, 192), (12, 96, 48),
        (8, 128, 128), (6, 96, 96), (192, 16, 16)]


def _eval(ctx, monkeypatch, kind, dims, prec, planes, steps=0):
    import kielflow_amd as kf
    if planes is None:
        monkeypatch.delenv("KF_PLANES", raising=False)
    else:
        monkeypatch.setenv("KF_PLANES", planes)
    rng = np.random.default_rng(7)
    axes = [axes_for(kind, n)[0][0] for n in dims]
    g = kf.Grid(ctx, axes)
    P = kf.KF_FP64 if prec == "fp64" else kf.KF_MIXED
    ps = kf.Poisson(g, P, tol=1e-11 if prec == "fp64" else 1e-10, max_it=80)
    rhs = kf.Rhs(g, ps, M=1.2, tau=0.1, theta=100.0, sv_on=True, pen_on=True, precision=P)
    x = [np.linspace(-8, 8, n, endpoint=False) for n in dims]
    r2 = x[0][:, None, None] ** 2 + x[1][None, :, None] ** 2 + x[2][None, None, :] ** 2
    mask = np.exp(-r2 / 4.0)
    phi = g.rfield()
    rhs.set_fields(phi, ctx.to_device(-0.05 * mask), ctx.to_device(mask))
    F = [ctx.to_device(np.fft.rfftn(1e-2 * rng.standard_normal(dims))) for _ in range(4)]
    if steps:
        rk = kf.Rk4(rhs, 1e-3)
        rk.step(F, steps)
    else:
        rhs.solve(0.0, F)
    assert rhs.poisson_failures() == 0
    out = [f.get() for f in F] + [phi.get()]
    monkeypatch.delenv("KF_PLANES", raising=False)
    return out


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["eqst", "sist"])
@pytest.mark.parametrize("dims", DIMS)
def test_plane_passes_give_identical_results(ctx, monkeypatch, kind, dims, prec):
    """Same butterflies, radices, twiddles and functors: an RHS evaluation is the same bit for bit."""
    print("planes", kind, dims, prec, flush=True)
    a = _eval(ctx, monkeypatch, kind, dims, prec, "1")
    b = _eval(ctx, monkeypatch, kind, dims, prec, "0")
    for name, x, y in zip(["FUx", "FUy", "FUz", "Fn", "phi"], a, b):
        assert np.isfinite(x).all() and np.array_equal(x, y), (name, float(np.abs(x - y).max()))


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("kind", ["eqst", "sist"])
@pytest.mark.parametrize("dims", [(8, 128, 128), (64, 96, 96), (96, 96, 96), (128, 128, 64)])
def test_the_rule_for_one_field_gives_identical_results(ctx, monkeypatch, kind, dims, prec):
    """Without the switch a field's own forward and inverse passes take planes or not by Nx and the plane's bytes,
    each for itself, beside the launches of several fields: the same bits as planes throughout."""
    print("plane rule", kind, dims, prec, flush=True)
    a = _eval(ctx, monkeypatch, kind, dims, prec, None)
    b = _eval(ctx, monkeypatch, kind, dims, prec, "1")
    for name, x, y in zip(["FUx", "FUy", "FUz", "Fn", "phi"], a, b):
        assert np.isfinite(x).all() and np.array_equal(x, y), (name, float(np.abs(x - y).max()))


@pytest.mark.parametrize("kind,prec", [("eqst", "fp64"), ("eqst", "mixed"), ("hyst", "fp64"), ("hyst", "mixed")])
def test_plane_passes_give_identical_steps(ctx, monkeypatch, kind, prec):
    """The RK4 update in the last store of the batched x passes, over several steps."""
    dims = (24, 32, 48)
    a = _eval(ctx, monkeypatch, kind, dims, prec, "1", steps=4)
    b = _eval(ctx, monkeypatch, kind, dims, prec, "0", steps=4)
    for name, x, y in zip(["FUx", "FUy", "FUz", "Fn", "phi"], a, b):
        assert np.array_equal(x, y), (name, float(np.abs(x - y).max()))


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("dims", DIMS)
def test_plane_transforms_give_identical_results(ctx, monkeypatch, dims, prec):
    import kielflow_amd as kf
    real, cplx = (np.float64, np.complex128) if prec == "fp64" else (np.float32, np.complex64)
    x = np.random.default_rng(3).standard_normal(dims).astype(real)
    out = []
    for planes in ("1", "0"):
        monkeypatch.setenv("KF_PLANES", planes)
        g = kf.Grid(ctx, [axes_for("eqst", n)[0][0] for n in dims])
        f = kf.FFT(g, kf.KF_FP64 if prec == "fp64" else kf.KF_FP32)
        X, y = ctx.zeros(g.cshape, cplx), ctx.zeros(g.rshape, real)
        f.r2c(ctx.to_device(x), X)
        f.c2r(X, y)
        out.append((X.get(), y.get()))
        f.close()
        g.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])


def _adjoint(ctx, monkeypatch, kind, dims, planes, sv, M):
    import kielflow_amd as kf
    monkeypatch.setenv("KF_PLANES", planes)
    monkeypatch.setenv("KF_XY_UNSHARED", "1")  # forward derivatives one by one on both sides
    rng = np.random.default_rng(11)
    g = kf.Grid(ctx, [axes_for(kind, n)[0][0] for n in dims])
    ps = kf.Poisson(g, kf.KF_FP64, tol=1e-12, max_it=80)
    rhs = kf.Rhs(g, ps, M=M, tau=0.1, theta=100.0, sv_on=sv, pen_on=True)
    x = [np.linspace(-8, 8, n, endpoint=False) for n in dims]
    mask = np.exp(-(x[0][:, None, None] ** 2 + x[1][None, :, None] ** 2 + x[2][None, None, :] ** 2) / 4.0)
    rhs.set_fields(g.rfield(), ctx.to_device(-0.05 * mask), ctx.to_device(mask))
    S = [ctx.to_device(np.fft.rfftn(1e-2 * rng.standard_normal(dims))) for _ in range(4)]
    w = [ctx.to_device(rng.standard_normal(g.cshape) + 1j * rng.standard_normal(g.cshape)) for _ in range(4)]
    adj = kf.Adjoint(rhs, 1e-3)
    adj.reset()
    Fb, ndbar = [g.cfield() for _ in range(4)], g.rfield()
    adj.rhs_adjoint(S, w, Fb)
    Mbar = adj.accumulators(ndbar)
    adj.step_adjoint(S, w)
    return [f.get() for f in Fb] + [ndbar.get()] + [f.get() for f in w], Mbar


@pytest.mark.parametrize("kind,sv,M", [("sist", True, 1.2), ("hyst", False, 0.0)])
@pytest.mark.parametrize("dims", [(16, 16, 16), (12, 24, 32), (6, 16, 192), (24, 128, 16), (16, 48, 96)])
def test_batched_adjoint_gives_identical_results(ctx, monkeypatch, kind, sv, M, dims):
    """The adjoint evaluation with a launch for several fields against one field at a time, and a step of it."""
    print("batched adjoint", kind, sv, M, dims, flush=True)
    a, ma = _adjoint(ctx, monkeypatch, kind, dims, "1", sv, M)
    b, mb = _adjoint(ctx, monkeypatch, kind, dims, "0", sv, M)
    assert ma == mb
    for i, (x, y) in enumerate(zip(a, b)):
        assert np.isfinite(x).all() and np.array_equal(x, y), (i, float(np.abs(x - y).max()))
