"""Reductions on both sides of the one-workgroup limit (4096 elements) and of
a workgroup's 256 threads, against long double sums.  Every term is rounded a
few times and the compensated total once: a unit of 2^-53 for each."""
import numpy as np
import pytest

from test_gpu_ops import N, fold, up  # noqa: F401

pytestmark = pytest.mark.gpu

U = 2.0 ** -53


@pytest.mark.parametrize("n", [1, 255, 256, 257, 4095, 4096, 4097, 8193])
def test_reductions_at_the_workgroup_limits(N, n):  # noqa: F811
    rng = np.random.default_rng(n)
    a = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    b = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    da, db = up(N, a), up(N, b)
    x, y = a.astype(np.clongdouble), b.astype(np.clongdouble)

    def near(got, want, units):
        assert abs(got - want) <= units * U * abs(want), (got, want)

    near(N.reduce1("qsim_hip_norm2", da.ptr, n), (x.real ** 2 + x.imag ** 2).sum(), 3)
    d = x - y
    near(N.reduce1("qsim_hip_minus_norm2", da.ptr, db.ptr, n), (d.real ** 2 + d.imag ** 2).sum(),
         5)
    i = np.arange(n)
    near(N.reduce1("qsim_hip_abs2_idx", da.ptr, n), ((x.real ** 2 + x.imag ** 2) * i).sum(), 4)
    assert N.reduce1("qsim_hip_max_abs", da.ptr, n) == pytest.approx(np.max(abs(a)), rel=1e-15)
    assert N.reduce1("qsim_hip_min_abs", da.ptr, n) == pytest.approx(np.min(abs(a)), rel=1e-15)
    # the extreme at each end of the array
    for at in (0, n - 1):
        c = a.copy()
        c[at] = 100.0
        assert N.reduce1("qsim_hip_max_abs", up(N, c).ptr, n) == 100.0
        c[at] = 1e-3 * np.min(abs(a))
        assert N.reduce1("qsim_hip_min_abs", up(N, c).ptr, n) == c[at].real
