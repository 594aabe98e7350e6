"""Lengths that the mixed-radix lines do not take, on the GPU: the generic
transform kernel against numpy, and the jobs that run the unfused reference
order on it (1D periodic, infinite wall, 2D, Born) against the FP64 oracle.
Every length of REFUSED is checked on the host to have no mixed-radix plan
(test_mix_refused.py)."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_born import opts, pot2d, pot3d
from test_gpu_split import gauss2d, run_1d, run_2d

pytestmark = pytest.mark.gpu

# the primes of a single pass, lengths with a large prime whose line does not
# fit LDS twice (the first and the last of them, a wall's 2n), and beyond 5120
REFUSED = [2, 3, 7, 11, 13, 3153, 3163, 3202, 3407, 3994, 4001, 4006, 4999, 5119, 8192]

SHAPES = [(3153,), (3202,), (4001,), (4999,), (5119,), (7, 3407), (3163, 12), (13,)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("precision", [64, 32])
def test_fft_beside_mixed_radix(shape, precision):
    """The generic kernel adds the P terms of a factor one by one: each sum
    rounds to about sqrt(P / 6) units, at most sqrt(P) of them are allowed
    here and twice that for the twiddles and the other factors."""
    from qusim_amd import fftn
    rng = np.random.default_rng(len(shape) * 1000 + shape[0])
    x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    if precision == 32:
        x = x.astype(np.complex64)
    tol = 3 * np.sqrt(max(shape)) * 2.0 ** (-53 if precision == 64 else -24)
    xd = x.astype(np.complex128)
    assert rel_l2(fftn(x, precision=precision), np.fft.fftn(xd)) < tol
    assert rel_l2(fftn(x, inverse=True, precision=precision), np.fft.ifftn(xd) * x.size) < tol


@pytest.mark.parametrize("n", [13, 3163, 4001, 4999])
@pytest.mark.parametrize("method", [2, 4])
def test_1d_unfused_order_matches_oracle(n, method, oracle):
    x = -25.0 + 50.0 / n * np.arange(n)
    psi = np.exp(0.7j * x - (x + 6) ** 2 / 9.0)
    V = 0.4 * np.exp(-x ** 2 / 6) - 0.02j * np.exp(-(x - 8) ** 2 / 20)
    got = run_1d(psi, V, -25.0, 25.0, 0.04, 5, method, complex_v=True).GetPsi()
    ref = oracle.split1d(psi, V, -25.0, 25.0, 0.04, 5, method=method, complex_v=True)
    assert rel_l2(got, ref) < 1e-12


@pytest.mark.parametrize("n", [1601, 1997, 2003, 4096])
@pytest.mark.parametrize("method", [2, 4])
def test_wall_unfused_order_matches_oracle(n, method, oracle):
    """2n points with a large prime, and 8192 points (a four-step transform);
    psi(0) is not zero at the start"""
    x = -25.0 + 50.0 / n * np.arange(n)
    psi = np.exp(0.7j * x - (x + 6) ** 2 / 40.0)
    V = 0.4 * np.exp(-x ** 2 / 6)
    got = run_1d(psi, V, -25.0, 25.0, 0.04, 5, method, boundary=1).GetPsi()
    ref = oracle.split1d(psi, V, -25.0, 25.0, 0.04, 5, method=method, boundary=1)
    assert rel_l2(got, ref) < 1e-12


@pytest.mark.parametrize("shape", [(7, 100), (100, 11), (4001, 16), (12, 3163)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("method", [2, 4])
def test_2d_unfused_order_matches_oracle(shape, method, oracle):
    psi, V, L0, L1 = gauss2d(*shape)
    got = run_2d(psi, V, L0, L1, 0.05, 4, method, complex_v=True).GetPsi()
    ref = oracle.split2d(psi, V, L0[0], L0[1], L1[0], L1[1], 0.05, 4, method=method,
                         complex_v=True, threads=8)
    assert rel_l2(got, ref) < 1e-12


@pytest.mark.parametrize("shape", [(13, 300), (40, 3163), (26, 11, 30)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("pre", [0, 1, 2, 3, 4])
def test_born_unfused_order_matches_oracle(shape, pre, oracle):
    """every preconditioner (4: none)"""
    from qusim_amd.api import QuPerturbation2D, QuPerturbation3D, SolverMethod
    lo, hi = (-60.0, -50.0, -40.0)[:len(shape)], (60.0, 50.0, 40.0)[:len(shape)]
    d = (0.3, -0.5, 0.8)[:len(shape)]
    box = [v for s, a, b in zip(shape, lo, hi) for v in (a, b, s)]
    V = (pot2d if len(shape) == 2 else pot3d)(shape, lo, hi)
    cls = QuPerturbation2D if len(shape) == 2 else QuPerturbation3D
    s = cls().init(V, *box, 2.0, 0.01, *d, SolverMethod.BornSerise, 1.0, 1.0,
                   opts(pre != 4, min(pre, 3), 0.7, 3))
    s.Compute()
    ref, _, _, _ = oracle.born(V, lo, hi, 2.0, d, order=3, preconditional=int(pre != 4),
                               preconditioner=min(pre, 3), slow=0.7, epsilon=0.01, threads=8)
    assert rel_l2(s.GetPsi(), ref) < 1e-12
