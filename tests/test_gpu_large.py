"""GPU: a layer whose planes exceed 2^31 bytes, against a small layer.

A Cartesian linear layer of 24576 x 24576 cells (2.4 GB per plane) and one
of 512 x 512 share depth, spacing and time step, and carry the same
Gaussian hump at the same offsets from a cell, placed near the far corner
of the large layer (plane offsets beyond 2^31 bytes).  The scheme reaches
at most two cells per step, so after n steps every cell within 256 - 2n of
the hump sees neither layer's edges, and holds the same bits in both:
indexing, tiling and launch shapes at the largest sizes change nothing.
"""
import ctypes

import numpy as np
import pytest

from gcomcot import DeviceRun
from gcomcot import scenarios as S
from gcomcot import lib

pytestmark = pytest.mark.gpu

STEPS = 60
FILL = 40          # hump radius in cells; zero beyond
SIGMA = 8.0


def _layer(n, ci, cj, depth, dx, dt):
    h = np.full((n, n), depth, np.float32)
    z0 = np.zeros((n, n), np.float32)
    d = np.arange(-FILL, FILL + 1)
    dj, di = np.meshgrid(d, d, indexing="ij")
    hump = (np.float32(1.5) * np.exp(-(di * di + dj * dj) / (2.0 * SIGMA * SIGMA))).astype(np.float32)
    z0[cj - 1 - FILL:cj + FILL, ci - 1 - FILL:ci + FILL] = hump
    spec = S.LayerSpec(id=1, parent=-1, level=1, laycord=1, laygov=0, nx=n, ny=n, dx=dx, dy=dx,
                       dt=dt, h=h, z0=z0, fric_switch=1, fric_coef=0.0)
    return S.Scenario(f"cartesian-linear-{n}x{n}", [spec], STEPS)


def _planes(n):
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    z = np.empty((n, n), np.float32)
    m = np.empty((n, n), np.float32)
    q = np.empty((n, n), np.float32)
    one = ctypes.byref(ctypes.c_int(1))
    lib().cuda_getz1_(p(z), one)
    lib().cuda_getmn1_(p(m), p(q), one)
    return z, m, q


def test_large_layer_equals_a_small_one_inside_the_domain_of_dependence():
    depth, dx = np.float32(4000.0), 1000.0
    dt = S.cr_dt(1, 0, np.full((4, 4), depth, np.float32), dx, dx, 0.0, 0.0)
    big_n, small_n = 24576, 512
    bi, bj = big_n - 400, big_n - 400          # hump cell of the large layer
    si, sj = small_n // 2, small_n // 2        # and of the small one
    print(f"[gpu] large layer {big_n}x{big_n}, {STEPS} steps", flush=True)
    dev = DeviceRun(_layer(small_n, si, sj, depth, dx, dt))
    dev.run(STEPS)
    small = _planes(small_n)
    dev.close()
    dev = DeviceRun(_layer(big_n, bi, bj, depth, dx, dt))
    dev.run(STEPS)
    big = _planes(big_n)
    dev.close()
    r = small_n // 2 - 2 * STEPS - 8
    for name, a, b in zip(("z", "m", "n"), small, big):
        wa = a[sj - 1 - r:sj + r, si - 1 - r:si + r]
        wb = b[bj - 1 - r:bj + r, bi - 1 - r:bi + r]
        assert np.abs(wa).max() > 1e-3, name
        assert np.array_equal(wa.view(np.int32), wb.view(np.int32)), \
            f"{name}: {np.count_nonzero(wa.view(np.int32) != wb.view(np.int32))} cells differ"


def _wide_layer(laygov, nx, ny):
    """A spherical layer of nx x ny cells from a small pattern of depths, shoals
    and land, its elevation from another, so that every part has waves."""
    j, i = np.mgrid[0:509, 0:511].astype(np.float32)
    h = 1500.0 + 1400.0 * np.sin(i / 37.0) * np.cos(j / 29.0)
    h[200:230, 100:160] = 12.0 - 0.5 * i[200:230, 0:60]
    z = 0.8 * np.sin(i / 11.0) * np.sin(j / 13.0)
    reps = (-(-ny // 509), -(-nx // 511))
    grid = lambda a: np.ascontiguousarray(np.tile(a.astype(np.float32), reps)[:ny, :nx])  # noqa: E731
    h, z0 = grid(h), grid(np.where(h > 0, z, 0.0))
    dx = 0.25
    y = (-20.0 + np.arange(ny) * dx / 60.0).astype(np.float32)
    fric = dict(fric_switch=0, fric_coef=0.013) if laygov else dict(fric_switch=1, fric_coef=0.0)
    dt = S.cr_dt(0, laygov, h, dx, dx, float(y[0]), float(y[-1]))
    spec = S.LayerSpec(id=1, parent=-1, level=1, laycord=0, laygov=laygov, nx=nx, ny=ny, dx=dx, dy=dx, dt=dt,
                       h=h, z0=z0, y=y, dely=np.full(ny, dx, np.float32), **fric)
    return S.Scenario(f"wide-{laygov}-{nx}x{ny}", [spec], 8)


@pytest.mark.parametrize("laygov,nx,ny", [(0, 9001, 11801), (1, 9001, 10801)], ids=["linear", "nonlinear"])
def test_marched_layer_of_almost_4_gb_equals_tiles(laygov, nx, ny):
    """The marching kernels reach a layer's planes by 32-bit offsets into one
    block: layers whose block ends just below 4 GB (40 and 44 bytes a cell),
    so that most planes lie beyond 2 GB, against the tiles."""
    from gcomcot._lib import ip
    sc = _wide_layer(laygov, nx, ny)
    assert 2 ** 32 - 5e7 < nx * ny * (44 if laygov else 40) < 2 ** 32 - 1e7
    got = []
    try:
        for march in (True, False):
            print(f"[gpu] {sc.name} march {march}", flush=True)
            assert lib().gcomcot_set_temporal_blocking_(ip(1 if march else 0)) == 0
            assert lib().gcomcot_set_tile_variant_(ip(0 if march else 1)) == 0
            dev = DeviceRun(sc)
            dev.run(3 if laygov else 7)
            z, m, n = (np.empty((ny, nx), np.float32) for _ in range(3))
            p = lambda a: a.ctypes.data_as(ctypes.c_void_p)  # noqa: E731
            lib().cuda_getz1_(p(z), ip(1))
            lib().cuda_getmn1_(p(m), p(n), ip(1))
            mx = dev.maxima(1)
            got.append(dict(z=z, m=m, n=n, zmax=mx["zmax_wet"], arrival=mx["arrival"]))
            dev.close()
    finally:
        lib().gcomcot_set_temporal_blocking_(ip(1))
        lib().gcomcot_set_tile_variant_(ip(0))
    assert np.abs(got[0]["m"][-600:]).max() > 1.0
    for k in got[0]:
        a, b = got[0][k].view(np.int32), got[1][k].view(np.int32)
        assert np.array_equal(a, b), f"{k}: {np.count_nonzero(a != b)} cells differ"
