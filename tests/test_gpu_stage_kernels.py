"""The x pass with a thread group per field, at the edges of the sizes, radices and layouts it is built for.

Tolerances: the grouped x pass packs and transforms as the plain one and
rounds differently at most: calcN agrees to the 1e-13 (FP64) and 2e-6 (FP32) that it is held to
against the oracle.
"""
import numpy as np
import pytest

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
