"""Mixed-radix lines on the GPU: the transform plan against numpy, the
split-operator jobs against the FP64 oracle, at the edges of their ranges
(the shortest and longest lengths, one and several lines per workgroup, every
radix, more butterflies than threads, tiles that the last lines do not fill)."""
import numpy as np
import pytest

from conftest import rel_l2
from test_gpu_split import gauss2d, run_1d, run_2d

pytestmark = pytest.mark.gpu

SHAPES = [(4,), (6,), (9,), (15,), (1000,), (3003,), (5000,), (5103,), (5120,), (4900,),
          (4, 6), (6, 1000), (1000, 6), (100, 169), (143, 77), (1500, 1100), (1, 60), (60, 1),
          (9, 10, 12), (14, 15, 98), (100, 120, 90), (17, 60, 50),
          # a prime above 13 alone, with others, twice, beside one line per workgroup
          (17,), (34,), (323,), (850,), (1369,), (2003,), (3109,), (3150,), (59, 118), (1009, 20),
          (23, 38, 62)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("precision", [64, 32])
def test_fft_mixed_radix(shape, precision):
    """Each axis of at most 6 passes rounds to a few units per pass: 32 units
    of 2^-53 (FP64) or, with every pass stored in FP32, 2^-24 per pass and
    axis."""
    from qusim_amd import fftn
    rng = np.random.default_rng(len(shape) * 1000 + shape[0])
    x = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    if precision == 32:
        x = x.astype(np.complex64)
    tol = len(shape) * (32 * 2.0 ** -53 if precision == 64 else 6 * 2.0 ** -24)
    xd = x.astype(np.complex128)
    assert rel_l2(fftn(x, precision=precision), np.fft.fftn(xd)) < tol
    assert rel_l2(fftn(x, inverse=True, precision=precision), np.fft.ifftn(xd) * x.size) < tol


@pytest.mark.parametrize("n", [4, 12, 60, 1000, 1300, 3003, 5082, 5103, 5120,
                               17, 850, 1009, 3109])
@pytest.mark.parametrize("method", [2, 4])
def test_1d_mixed_radix_matches_oracle(n, method, oracle):
    x = -25.0 + 50.0 / n * np.arange(n)
    psi = np.exp(0.7j * x - (x + 6) ** 2 / 9.0)
    V = 0.4 * np.exp(-x ** 2 / 6) - 0.02j * np.exp(-(x - 8) ** 2 / 20)
    e = run_1d(psi, V, -25.0, 25.0, 0.04, 31, method, complex_v=True)
    ref = oracle.split1d(psi, V, -25.0, 25.0, 0.04, 31, method=method, complex_v=True)
    assert rel_l2(e.GetPsi(), ref) < 1e-12
    # steps split over several calls
    f = run_1d(psi, V, -25.0, 25.0, 0.04, 30, method, complex_v=True, batch=5)
    f.steps(0)
    g = oracle.split1d(psi, V, -25.0, 25.0, 0.04, 30, method=method, complex_v=True)
    assert rel_l2(f.GetPsi(), g) < 1e-12


@pytest.mark.parametrize("n", [2, 15, 500, 1024, 1500, 2560, 17, 517, 1549])
@pytest.mark.parametrize("method", [2, 4])
def test_wall_mixed_radix_matches_oracle(n, method, oracle):
    """the odd extension to 2n points; psi(0) is not zero at the start"""
    x = -25.0 + 50.0 / n * np.arange(n)
    psi = np.exp(0.7j * x - (x + 6) ** 2 / 40.0)
    V = 0.4 * np.exp(-x ** 2 / 6)
    e = run_1d(psi, V, -25.0, 25.0, 0.04, 23, method, boundary=1)
    ref = oracle.split1d(psi, V, -25.0, 25.0, 0.04, 23, method=method, boundary=1)
    assert rel_l2(e.GetPsi(), ref) < 1e-12


@pytest.mark.parametrize("shape", [(4, 4), (6, 1000), (1000, 6), (65, 130), (750, 600),
                                   (1024, 250), (98, 2048), (5120, 12), (32, 32),
                                   (34, 59), (850, 101), (64, 1009), (3109, 17)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("method", [2, 4])
def test_2d_mixed_radix_matches_oracle(shape, method, oracle):
    psi, V, L0, L1 = gauss2d(*shape)
    got = run_2d(psi, V, L0, L1, 0.05, 6, method, complex_v=True).GetPsi()
    ref = oracle.split2d(psi, V, L0[0], L0[1], L1[0], L1[1], 0.05, 6, method=method,
                         complex_v=True)
    assert rel_l2(got, ref) < 1e-12


def _born(shape, E, pre, precision="fp64", order=5):
    from test_gpu_born import opts, pot2d, pot3d
    from qusim_amd.api import QuPerturbation2D, QuPerturbation3D, SolverMethod
    lo = tuple(-s / 2.0 for s in shape)
    hi = tuple(s / 2.0 for s in shape)
    d = (0.3, -0.5, 0.8)[:len(shape)]
    box = [v for s, a, b in zip(shape, lo, hi) for v in (a, b, s)]
    V = (pot2d if len(shape) == 2 else pot3d)(shape, lo, hi)
    cls = QuPerturbation2D if len(shape) == 2 else QuPerturbation3D
    s = cls().init(V, *box, E, 0.01, *d, SolverMethod.BornSerise, 1.0, 1.0,
                   opts(pre != 4, min(pre, 3), 0.7, order, precision=precision))
    return s, V, lo, hi, d


# shortest axes, one that needs several radices, a power of two among them, a
# plane that the last workgroup does not fill; every preconditioner (4: none)
@pytest.mark.parametrize("shape", [(4, 300), (300, 6), (250, 350), (4, 6, 250), (26, 64, 33),
                                   (34, 251), (23, 38, 51),
                                   (32, 32, 32)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("pre", [0, 1, 2, 3, 4])
def test_born_mixed_radix_matches_oracle(shape, pre, oracle):
    if pre != 4 and min(shape) < 20:
        pytest.skip("the preconditioned solver refuses boxes this small")
    E = 6.0 if len(shape) == 2 else 2.0
    if len(shape) == 2 and pre != 4:
        E = (1.1 * 24 * 2 * np.pi / min(shape)) ** 2 / 2
    s, V, lo, hi, d = _born(shape, E, pre)
    s.Compute()
    ref, _, _, _ = oracle.born(V, lo, hi, E, d, order=5, preconditional=int(pre != 4),
                               preconditioner=min(pre, 3), slow=0.7, epsilon=0.01, threads=8)
    assert rel_l2(s.GetPsi(), ref) < 1e-12


def test_born_mixed_radix_stops_at_the_first_update_below_the_tolerance():
    shape, E = (24, 20, 28), [2.0, 2.6]
    one, _, _, _, _ = _born(shape, E, 1, order=1)
    res = []
    for _ in range(7):
        one.Compute()
        res.append(list(one.residual))
    many, _, _, _, _ = _born(shape, E, 1)
    tol = 0.5 * (res[3][0] + res[4][0])
    many.Compute(max_iter=7, tol=tol)
    want = [next((k + 1 for k in range(7) if res[k][e] < tol), 7) for e in range(2)]
    assert many.iters == want and want[0] == 5
    for e in range(2):
        assert abs(many.residual[e] / res[want[e] - 1][e] - 1) < 1e-13
