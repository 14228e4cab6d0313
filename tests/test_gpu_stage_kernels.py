"""The x pass with a thread group per field and the y pass that fuses one stage's K3 with the next
stage's K1, at the edges of the sizes, radices and layouts they are built for.

Tolerances: the fused y pass evaluates the expressions of K3 and K1, so it gives their bits (per-kernel
timing steps with those two kernels).  The grouped x pass packs and transforms as the plain one and
rounds differently at most: calcN agrees to the 1e-13 (FP64) and 2e-6 (FP32) that it is held to
against the oracle.
"""
import numpy as np
import pytest

from oracle import fourierflows as off
from oracle import singlelayerqg as osl
from tests.conftest import rel

pytestmark = pytest.mark.gpu


def state(ny, nx, dtype, seed=3):
    rng = np.random.default_rng(seed)
    sh = np.fft.rfft2(0.1 * rng.standard_normal((ny, nx)))
    sh[0, 0] = 0
    return sh.astype(np.complex128 if dtype == np.float64 else np.complex64)


@pytest.mark.parametrize("nx,ny,p2", [(16, 32, 4), (32, 16, 8), (64, 18, 4), (128, 32, 8), (256, 64, 4), (512, 32, 4),
                                      (512, 34, 8), (1024, 32, 16), (1024, 32, 4), (2048, 32, 8), (2048, 16, 16), (4096, 16, 16)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_a_group_per_field_gives_the_plain_x_pass(gf, nx, ny, p2, dtype):
    tol = 1e-13 if dtype == np.float64 else 2e-6
    eta = 0.1 * np.random.default_rng(1).standard_normal((ny, nx))
    s = state(ny, nx, dtype)
    for kw in (dict(eta=eta, U=0.3), dict(eta=eta, U=0.2 * np.cos(2 * np.pi * np.arange(ny) / ny))):
        out = []
        for k2 in (0, 1):
            p = gf.SingleLayerQG.Problem(gf.GPU(), nx=nx, ny=ny, β=2.0, μ=0.1, T=dtype, **kw)
            if ny & (ny - 1) == 0:
                gf.set_schedule(p, 0, p2, 0)
                gf.set_splits(p, 0, k2, 0)
            out.append(p.calcN(s)[0])
        assert rel(out[1], out[0]) < tol


# (nx, ny, P of K3, K1 split, K3 split): the smallest and largest columns of each form (three groups of one
# and of several waves, one group, pairs and single columns) and rectangles
FORMS = [(32, 32, 4, 1, 0), (32, 32, 8, 1, 0), (64, 64, 4, 1, 0), (128, 64, 8, 1, 0), (64, 128, 4, 1, 0), (32, 256, 4, 1, 1),
         (256, 256, 8, 1, 0), (64, 512, 8, 1, 1), (64, 512, 4, 1, 0), (32, 1024, 4, 1, 1), (32, 1024, 8, 1, 0), (64, 1024, 8, 0, 1),
         (32, 2048, 4, 1, 0), (64, 2048, 8, 0, 1), (32, 4096, 8, 0, 0), (32, 4096, 8, 0, 1), (32, 4096, 16, 0, 0)]


@pytest.mark.parametrize("nx,ny,p3,k1,k3", FORMS)
@pytest.mark.parametrize("stepper", ["ETDRK4", "FilteredRK4", "AB3", "FilteredForwardEuler"])
def test_fused_stages_give_the_bits_of_the_separate_kernels(gf, nx, ny, p3, k1, k3, stepper):
    lib = gf._lib.lib
    kw = dict(nx=nx, ny=ny, Ly=2 * np.pi * ny / nx, dt=1e-4, stepper=stepper)
    made = [lambda T: gf.TwoDNavierStokes.Problem(gf.GPU(), ν=1e-6, calcF=gf.RingForcing(5.0, 1.5, 0.1, seed=7), T=T, **kw),
            lambda T: gf.SingleLayerQG.Problem(gf.GPU(), β=2.0, μ=0.1, U=0.2, deformation_radius=0.7, T=T,
                                               eta=lambda x, y: 0.1 * np.cos(x), **kw)]
    for make, T in ((made[0], np.float64), (made[1], np.float64), (made[1], np.float32)):
        sols = []
        for timed in (0, 1):
            p = make(T)
            gf.set_schedule(p, 0, 0, p3)
            gf.set_splits(p, k1, 0, k3)
            p.sol = state(ny, nx, T)
            assert lib.gf_timing(p._ctx, timed) == 0
            gf.stepforward(p, 4)
            gf.stepforward(p, 1)
            sols.append(p.sol)
        assert np.isfinite(sols[0]).all() and np.array_equal(sols[0], sols[1])


@pytest.mark.parametrize("nx,ny,p3,k1,k3", [(32, 32, 4, 1, 0), (64, 256, 4, 1, 1), (64, 1024, 8, 1, 1), (128, 2048, 8, 0, 1)])
def test_fused_stages_match_the_oracle(gf, nx, ny, p3, k1, k3):
    kw = dict(nx=nx, ny=ny, Ly=2 * np.pi * ny / nx, dt=1e-3, stepper="FilteredETDRK4")
    p = gf.SingleLayerQG.Problem(gf.GPU(), β=2.0, μ=0.1, ν=1e-5, **kw)
    gf.set_schedule(p, 0, 0, p3)
    gf.set_splits(p, k1, 1, k3)
    r = osl.Problem(beta=2.0, mu=0.1, nu=1e-5, **kw)
    p.sol = state(ny, nx, np.float64)
    r.sol[...] = p.sol
    gf.stepforward(p, 5)
    off.stepforward(r, 5)
    assert rel(p.sol, r.sol) < 1e-12


@pytest.mark.parametrize("counts,stepper,dtype", [((1, 1, 1, 1, 1), "ETDRK4", np.float64), ((2, 1, 1, 1, 1), "FilteredRK4", np.float32),
                                                  ((60, 60, 60, 60, 0), "RK4", np.float64), ((700, 0, 0, 20, 8), "AB3", np.float64)])
def test_both_ensemble_forms_match_members_stepped_alone(gf, counts, stepper, dtype):
    # few entries run with three thread groups each, many with one; every size, the last step of a
    # call in full; to the rounding of a few steps (a member alone has another radix schedule)
    tol = 1e-13 if dtype == np.float64 else 2e-5
    sizes = [n for n, c in zip((32, 64, 128, 256, 512), counts) for _ in range(c)]
    made = []
    for i, n in enumerate(sizes):
        kw = dict(nx=n, dt=1e-3, stepper=stepper, μ=0.1, T=dtype)
        if i % 2:
            made.append((gf.TwoDNavierStokes.Problem, dict(ν=1e-5, calcF=gf.RingForcing(5.0, 1.5, 0.1, seed=i), **kw)))
        else:
            made.append((gf.SingleLayerQG.Problem, dict(β=2.0, U=0.2 * np.cos(2 * np.pi * np.arange(n) / n) if i % 4 else 0.1, **kw)))
    ens = gf.Ensemble(made)
    look = sorted({0, 1, 2, 3, len(sizes) - 1, len(sizes) - 2} | {sizes.index(n) for n in set(sizes)})
    starts = {}
    for i, p in enumerate(ens.problems):
        s = state(sizes[i], sizes[i], dtype, seed=sizes[i] + i % 3)
        p.sol = s
        starts[i] = s
    gf.stepforward(ens, 4)
    gf.stepforward(ens, 1)
    for i in look:
        ctor, kw = made[i]
        single = ctor(gf.GPU(), **kw)
        single.sol = starts[i]
        gf.stepforward(single, 5)
        assert rel(ens[i].sol, single.sol) < tol, (i, sizes[i])


@pytest.mark.parametrize("nl,nx,ny", [(2, 32, 32), (3, 64, 64), (2, 32, 128), (4, 32, 256), (5, 32, 512), (3, 64, 512), (2, 18, 30), (5, 32, 34),
                                      (3, 66, 62), (2, 128, 126), (4, 30, 254), (6, 32, 32), (2, 32, 16), (1, 64, 18), (1, 66, 250), (1, 22, 126)])
@pytest.mark.parametrize("stepper,linear", [("ETDRK4", False), ("FilteredRK4", False), ("AB3", False), ("ETDRK4", True)])
def test_fused_layers_and_ragged_columns_give_the_bits_of_the_separate_kernels(gf, nl, nx, ny, stepper, linear):
    # multi-layer problems (2 to 5 layers are fused, 6 are not) with drag, ring forcing and topography, and
    # TwoDNS / SingleLayerQG with columns that are not a power of two long
    lib = gf._lib.lib
    ring = gf.RingForcing(4.0, 1.5, 0.1, seed=7)
    kw = dict(nx=nx, ny=ny, Ly=2 * np.pi * ny / nx, dt=1e-4, stepper=stepper)
    eta = 0.1 * np.random.default_rng(1).standard_normal((ny, nx))
    if nl > 1:
        H = np.ones(nl) / nl
        make = [lambda T: gf.MultiLayerQG.Problem(nl, gf.GPU(), f0=1.0, β=1.0, μ=0.2, ν=1e-6, U=0.1 * np.arange(nl), H=H,
                                                  b=-1.0 - np.arange(nl) / nl, eta=eta, calcFq=ring, linear=linear, T=T, **kw)]
    elif linear:
        pytest.skip("one layer here is TwoDNS or SingleLayerQG")
    else:
        make = [lambda T: gf.TwoDNavierStokes.Problem(gf.GPU(), ν=1e-6, calcF=ring, T=T, **kw),
                lambda T: gf.SingleLayerQG.Problem(gf.GPU(), β=2.0, μ=0.1, eta=eta, deformation_radius=0.7, T=T, **kw)]
    for mk in make:
        for T in (np.float64, np.float32):
            sols = []
            for timed in (0, 1):
                p = mk(T)
                s = state(ny, nx, T)
                p.sol = s if nl == 1 else np.stack([s * (1 - 0.1 * j) for j in range(nl)])
                assert lib.gf_timing(p._ctx, timed) == 0
                gf.stepforward(p, 4)
                gf.stepforward(p, 1)
                sols.append(p.sol)
            assert np.isfinite(sols[0]).all() and np.array_equal(sols[0], sols[1])


@pytest.mark.parametrize("n", [32, 64, 128, 256, 512, 1024])
def test_two_launch_adjoint_matches_the_separate_kernels(gf, n):
    # per-kernel timing runs KA1, KA2 and KA3 one by one (1024^2 always does); the two forms sum the same
    # terms of 5 steps in other orders: 1e-12 relative
    z = 0.3 * np.random.default_rng(n).standard_normal((n, n))
    target = 0.1 * np.random.default_rng(n + 1).standard_normal((n, n))
    got = []
    for timed in (0, 1):
        p = gf.TwoDNavierStokes.Problem(gf.GPU(), nx=n, ν=1e-3, nν=1, dt=1e-3, stepper="ETDRK4")
        gf.TwoDNavierStokes.set_ζ(p, z)
        assert gf._lib.lib.gf_timing(p._ctx, timed) == 0
        got.append(gf.TwoDNavierStokes.adjoint_gradient(p, target, 5, 2))
    (J0, g0, nu0), (J1, g1, nu1) = got
    assert abs(J0 - J1) <= 1e-13 * abs(J1) and abs(nu0 - nu1) <= 1e-11 * abs(nu1)
    assert rel(g0, g1) < 1e-12


# gradients that depend on y only: the x pass multiplies v's spectrum by Qy; with a topography (here one
# of height 1e-200) it transforms u Qx + v Qy.  Both round each of at most 2 log2(nx ny) butterfly levels and a handful of
# products once; the sum of the three terms cancels to no less than a tenth of its largest one.
@pytest.mark.parametrize("nl,nx,ny", [(1, 32, 32), (1, 64, 32), (1, 512, 64), (1, 1024, 32), (1, 2048, 32), (1, 4096, 16), (1, 34, 62),
                                      (1, 126, 32), (1, 64, 30), (2, 32, 64), (3, 512, 32), (2, 1024, 32), (2, 2048, 32), (2, 18, 30),
                                      (5, 128, 126), (8, 64, 32)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
def test_gradients_in_y_only_match_transformed_ones(gf, nl, nx, ny, dtype):
    eps = np.finfo(dtype).eps
    tol = 10 * (2 * np.log2(nx * ny) + 10) * eps
    y = 2 * np.pi * np.arange(ny) / ny
    kw = dict(nx=nx, ny=ny, β=1.5, μ=0.05, T=dtype)
    s = np.stack([state(ny, nx, dtype, seed=k) for k in range(nl)])
    for aliased, U in ((1 / 3, 0.2), (0.0, 0.3)):
        out = []
        for eta in (np.full((ny, nx), 1e-200), None):
            more = dict(kw, aliased_fraction=aliased)
            if nl == 1:
                p = gf.SingleLayerQG.Problem(gf.GPU(), U=U * np.cos(y), eta=eta, **more)
            else:
                prof = U * np.cos(y)[None, :] * np.arange(1, nl + 1)[:, None] / nl
                p = gf.MultiLayerQG.Problem(nl, gf.GPU(), f0=1.0, U=prof, H=[1.0 / nl] * nl, b=list(-0.2 * np.arange(nl)),
                                            eta=eta, **more)
            splits = [(0, 0, 0), (0, 1, 0)] if nl == 1 and (nx & (nx - 1)) == 0 and (ny & (ny - 1)) == 0 else [None]
            for sp in splits:
                if sp is not None:
                    gf.set_splits(p, *sp)
                out.append(p.calcN(s if nl > 1 else s[0])[0])
        for o in out[1:]:
            assert rel(o, out[0]) < tol
