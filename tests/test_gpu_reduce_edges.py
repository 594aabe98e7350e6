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


@pytest.mark.parametrize("shape", [(1, 7, 1), (16, 16, 6), (29, 53, 1), (16, 16, 10), (13, 197, 1),
                                   (16, 16, 16), (17, 241, 1)], ids=lambda s: "x".join(map(str, s)))
def test_index_and_phase_reductions_at_the_workgroup_limits(N, shape):  # noqa: F811
    """1536 and 1537 elements (cross sections), 2560 and 2561 (kinetic
    energies), 4096 and 4097; terms of both signs: the absolute sum scales the
    bound, a dozen units for the rounding of the phase (below 4)."""
    nx, ny, nz = shape
    n = nx * ny * nz
    rng = np.random.default_rng(n)
    p0, p, V = (rng.standard_normal(n) + 1j * rng.standard_normal(n) for _ in range(3))
    I, J, K = (g.ravel().astype(np.longdouble) for g in
               np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz), indexing="ij"))
    d0, d1, dv = up(N, p0), up(N, p), up(N, V)
    k = (0.3, -0.02, 0.5)
    lo, d = (-1.0, -0.5, -2.0), (0.25, 0.5, 0.125)
    kx, ky, kz = map(np.longdouble, k)
    ph = (lo[0] + I * d[0]) * kx + (lo[1] + J * d[1]) * ky + (lo[2] + K * d[2]) * kz
    t = (p0.astype(np.clongdouble) + p) * V.real * np.exp(-1j * ph)
    got = N.reduce_c("qsim_hip_xsection3d", d0.ptr, d1.ptr, dv.ptr, *k, *lo, *d, nx, ny, nz)
    assert abs(got - t.sum()) <= 20 * U * abs(t).sum()
    # the 2D forms
    if nz == 1:
        ph = (lo[0] + I * d[0]) * kx + (lo[1] + J * d[1]) * ky
        t = (p0.astype(np.clongdouble) + p) * V.real * np.exp(-1j * ph)
        got = N.reduce_c("qsim_hip_xsection2d", d0.ptr, d1.ptr, dv.ptr, *k[:2], *lo[:2], *d[:2],
                         nx, ny)
        assert abs(got - t.sum()) <= 20 * U * abs(t).sum()
    w = abs(p0.astype(np.clongdouble)) ** 2
    fi, fj, fk = fold(I, nx), fold(J, ny), fold(K, nz)
    want = (w * (fi ** 2 * 0.25 + fj ** 2 * 0.5 + fk ** 2 * 2)).sum()
    got = N.reduce1("qsim_hip_abs2_k3d", d0.ptr, 0.25, nx, 0.5, ny, 2.0, nz)
    assert abs(got - want) <= 8 * U * want
    if nz == 1:
        want = (w * (fi ** 2 * 0.25 + fj ** 2 * 0.5)).sum()
        got = N.reduce1("qsim_hip_abs2_k2d", d0.ptr, 0.25, nx, 0.5, ny)
        assert abs(got - want) <= 8 * U * want
