"""The transform of grid lengths that are not powers of two, at the lengths where it can go wrong: the
shortest and longest of each power of two's range, twice a prime, and each paired with a power of
two; every model's x-pass mode, both precisions.

Tolerances (relative L2 of calcN against the oracle): a transform adds up at most 64 folded terms, so
about 8 roundings in the root mean square, 1e-15 in FP64 and 5e-7 in FP32, for each of the two
directions; 1e-13 and 2e-6 as the other checks of calcN.
"""
import numpy as np
import pytest

from oracle import multilayerqg as oml
from oracle import singlelayerqg as osl
from tests.conftest import rel

pytestmark = pytest.mark.gpu


def spec(shape, dtype):
    rng = np.random.default_rng(shape[-1])
    s = 0.05 * (rng.standard_normal(shape) + 1j * rng.standard_normal(shape))
    s[..., 0, 0] = 0
    return s.astype(np.complex64 if dtype == np.float32 else np.complex128).astype(np.complex128)


@pytest.mark.parametrize("nx,ny,dtype", [(18, 30, np.float64), (30, 18, np.float64), (34, 62, np.float64), (62, 34, np.float64),
                                         (66, 254, np.float64), (254, 66, np.float64), (130, 122, np.float64), (256, 254, np.float64),
                                         (254, 256, np.float64), (16, 22, np.float64), (22, 16, np.float64), (254, 254, np.float32)])
def test_calcN_of_every_mode_matches_the_oracle(gf, nx, ny, dtype):
    tol = 1e-13 if dtype == np.float64 else 2e-6
    eta = 0.1 * np.random.default_rng(1).standard_normal((ny, nx)).astype(dtype).astype(np.float64)
    Uy = 0.2 * np.cos(2 * np.pi * np.arange(ny) / ny)
    s = spec((ny, nx // 2 + 1), dtype)
    for kw in (dict(eta=eta), dict(eta=eta, U=Uy)):
        p = gf.SingleLayerQG.Problem(gf.GPU(), nx=nx, ny=ny, β=2.0, μ=0.1, T=dtype, **kw)
        r = osl.Problem(nx=nx, ny=ny, beta=2.0, mu=0.1, **kw)
        N, _ = p.calcN(s)
        Nr, sr = np.zeros_like(s), s.copy()
        osl.calcN(Nr, sr, 0.0, r.clock, r.vars, r.params, r.grid)
        assert rel(N, Nr) < tol
    for n in (1, 2):
        kw = dict(nx=nx, ny=ny, f0=1.0, U=[0.3, 0.1][:n], H=[0.4, 0.6][:n], b=[-1.0, -1.5][:n], eta=eta)
        p = gf.MultiLayerQG.Problem(n, gf.GPU(), β=1.0, μ=0.05, T=dtype, **kw)
        r = oml.Problem(n, beta=1.0, mu=0.05, **kw)
        sn = s if n == 1 else np.stack([s, 0.5 * s])
        N, _ = p.calcN(sn)
        sr = sn.reshape(n, ny, nx // 2 + 1).copy()
        Nr = np.zeros_like(sr)
        oml.calcN(Nr, sr, 0.0, r.clock, r.vars, r.params, r.grid)
        assert rel(N.reshape(Nr.shape), Nr) < tol
