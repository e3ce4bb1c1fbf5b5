"""Ray lists at the sizes where their launch changes (FP64: the lone-ray walk
with four wavefronts a ray up to 1,024, with one up to 20,000, bundles beyond;
FP32C: shot in FP64 up to 16,000), on coarse leaves and with big particles,
against the oracle and, to the bit, against the grid launch.

Tolerance: the same algorithm in the same precision, sums in another order:
relative |d alpha| <= 1e-9, |d A| <= 1e-8 (the bounds of the FP64 walk's tests).
"""
import numpy as np
import pytest

import oracle as O
import slsimlib_amd as S
from slsimlib_amd import workloads as W

pytestmark = pytest.mark.gpu

LIMIT64, LIMIT32, FOUR_WAVES = 20000, 16000, 1024


def _check(lens, L, x, y, A, zs=None):
    sub = np.unique(np.concatenate([np.arange(0, len(x), max(1, len(x) // 400)), [len(x) - 1]]))
    yr, Ar = L.shoot(x[sub], zs=None if zs is None else zs[sub])
    a = np.linalg.norm(x[sub] - yr, axis=1)
    scale = np.maximum(a, 1e-3 * np.sqrt(np.mean(a ** 2)))
    assert (np.linalg.norm(y[sub] - yr, axis=1) / np.maximum(scale, 1e-300)).max() <= 1e-9
    assert np.abs(A[sub] - Ar).max() <= 1e-8 * max(1.0, np.abs(Ar).max())


@pytest.fixture(scope="module")
def field(ctx):
    lens, parts, _ = W.build_field_lens(ctx, config=7, nplanes=3, n=1 << 14, mass_scale=1 / 64,
                                        keep_particles=True)
    L = O.Lens(3.0)
    for (x, y, m, h, z) in parts:
        L.moveinMainHalo(O.Tree(x, y, m, h), z)
    return lens, L


@pytest.mark.parametrize("n", [1, 63, 64, 65, FOUR_WAVES, FOUR_WAVES + 1, 2048, 2049, LIMIT32,
                               LIMIT32 + 1, LIMIT64, LIMIT64 + 1, 49152, 49153])
def test_list_sizes_match_oracle(field, n):
    lens, L = field
    rng = np.random.default_rng(n)
    x = (rng.random((n, 2)) - 0.5) * W.grid_range(300.0)
    zs = rng.uniform(0.05, 4.0, n) if n % 2 else None
    y, A = lens.rayshooterInternal(x, zs)
    _check(lens, L, x, y, A, zs)
    st = {}
    y32, A32 = lens.rayshooterInternal(x, zs, S.SLSIM_FP32C, stats=st)
    if n <= LIMIT32:                      # FP64 results: nothing to guard
        assert np.array_equal(y32, y) and np.array_equal(A32, A) and st["n_guarded"] == 0
    # the precision form within its bound of the FP64 path at every ray
    a = np.linalg.norm(x - y, axis=1)
    scale = np.maximum(a, 1e-3 * np.sqrt(np.mean(a ** 2)))
    assert (np.linalg.norm(y32 - y, axis=1) <= 1e-5 * scale).all()
    assert np.abs(A32 - A).max() <= 1e-3


@pytest.mark.parametrize("bucket,max_range", [(1, -1.0), (20, -1.0), (700, -1.0), (20, 0.02)])
def test_leaves_and_big_particles_match_oracle(ctx, bucket, max_range):
    rng = np.random.default_rng(bucket)
    n = 5000
    x = np.concatenate([0.05 * rng.normal(size=n), 1.0 + 0.01 * rng.random(n // 2)])
    y = np.concatenate([0.05 * rng.normal(size=n), 0.01 * rng.random(n // 2)])
    m = (1e9 * (0.5 + rng.random(x.size))).astype(np.float32)
    h = (10.0 ** rng.uniform(-6, -0.5, x.size)).astype(np.float32)
    lens, L = S.Lens(ctx, 2.0), O.Lens(2.0)
    for z, ia in ((0.5, 0.0), (0.5, 30.0), (1.0, 0.0)):
        lens.moveinMainHalo(S.LensHaloParticles(ctx, x, y, m, h, z, bucket=bucket, inv_area=ia,
                                                max_range=max_range))
        L.moveinMainHalo(O.Tree(x, y, m, h, bucket=bucket, inv_area=ia, max_range=max_range), z)
    for k in (30, 2500):
        pos = (rng.random((k, 2)) - 0.5) * W.grid_range(60.0)
        yy, A = lens.rayshooterInternal(pos)
        _check(lens, L, pos, yy, A)


def _same(r, y, A):
    return np.array_equal(r[0], y) and np.array_equal(r[1], A)


@pytest.mark.parametrize("N", [1, 6, 8, 32, 33, 45, 46, 90, 127, 141, 142, 222])
def test_list_is_its_gridmap_to_the_bit(ctx, field, N):
    """A ray's FP64 result does not depend on the rays beside it: the rays of
    a GridMap as a list in another order, as two lists, and as a served list
    (sizes on both sides of every limit of the list's walk)."""
    lens, _ = field
    rg = W.grid_range(300.0)
    g = S.GridMap(lens, N, (0.0, 0.0), rg, S.SLSIM_FP64)
    x, n = g.positions(), N * N
    perm = np.random.default_rng(N).permutation(n)
    y, A = g.y()[perm], g.A()[perm]
    assert _same(lens.rayshooterInternal(x[perm]), y, A)
    for part in (slice(0, n // 3), slice(n // 3, n)):
        if len(x[perm][part]):
            assert _same(lens.rayshooterInternal(x[perm][part]), y[part], A[part])
    srv = S.Server(ctx, hbm_budget=1 << 30)
    r = srv.wait_rays(srv.submit_rays(lens, x[perm], precision=S.SLSIM_FP64), n)
    srv.close()
    assert _same(r, y, A)


@pytest.mark.parametrize("bucket,max_range,theta", [(1, -1.0, 0.1), (20, -1.0, 0.1),
                                                    (700, -1.0, 0.1), (20, 0.02, 0.1),
                                                    (5, -1.0, 0.004), (1, -1.0, 0.004),
                                                    (1, -1.0, 0.5)])
def test_trees_of_any_form_give_the_grid_bits(ctx, bucket, max_range, theta):
    """As above on coarse leaves, big particles, a mass sheet and, at the
    smallest opening angle, more opened cells than the walk lists at a time."""
    rng = np.random.default_rng(bucket)
    n = 6000
    x = np.concatenate([0.05 * rng.normal(size=n), 1.0 + 0.01 * rng.random(n // 2)])
    y = np.concatenate([0.05 * rng.normal(size=n), 0.01 * rng.random(n // 2)])
    m = (1e9 * (0.5 + rng.random(x.size))).astype(np.float32)
    h = (10.0 ** rng.uniform(-6, -0.5, x.size)).astype(np.float32)
    lens = S.Lens(ctx, 2.0)
    for z, ia in ((0.5, 0.0), (0.5, 30.0), (1.0, 0.0)):
        lens.moveinMainHalo(S.LensHaloParticles(ctx, x, y, m, h, z, bucket=bucket, theta=theta,
                                                inv_area=ia, max_range=max_range))
    for N in (30, 40):                    # four wavefronts a ray, and one
        g = S.GridMap(lens, N, (0.0, 0.0), W.grid_range(60.0), S.SLSIM_FP64)
        assert _same(lens.rayshooterInternal(g.positions()), g.y(), g.A())
    lens.close()


@pytest.mark.parametrize("N", [2, 8, 32, 33, 64, 126, 127, 128, 222])
def test_fp32c_list_is_a_gridmap_to_the_bit(ctx, field, N):
    """The precision form: a GridMap's rays as a list in another order and as a
    served list.  Up to 16,000 rays they are shot in FP64, so they are the FP64
    GridMap's results and within the form's bound of the FP32C GridMap's; beyond,
    they are the FP32C GridMap's with the rays its guard shot again."""
    lens, _ = field
    rg = W.grid_range(300.0)
    n = N * N
    g = S.GridMap(lens, N, (0.0, 0.0), rg, S.SLSIM_FP64 if n <= LIMIT32 else S.SLSIM_FP32C)
    x = g.positions()
    perm = np.random.default_rng(N).permutation(n)
    y, A = g.y()[perm], g.A()[perm]
    st = {}
    assert _same(lens.rayshooterInternal(x[perm], precision=S.SLSIM_FP32C, stats=st), y, A)
    srv = S.Server(ctx, hbm_budget=1 << 30)
    r = srv.wait_rays(srv.submit_rays(lens, x[perm], precision=S.SLSIM_FP32C), n)
    srv.close()
    assert _same(r, y, A)
    g32 = S.GridMap(lens, N, (0.0, 0.0), rg, S.SLSIM_FP32C)
    if n > LIMIT32:
        assert st["n_guarded"] == g32.stats["n_guarded"]
    else:
        a = np.linalg.norm(x - g.y(), axis=1)
        scale = np.maximum(a, 1e-3 * np.sqrt(np.mean(a ** 2)))
        assert st["n_guarded"] == 0
        assert (np.linalg.norm(g32.y() - g.y(), axis=1) <= 1e-5 * scale).all()


def test_server_counts_the_rays_of_its_lists(ctx, field):
    """A scheduler iteration takes up to 32,768 bundles' worth of work, eight
    rays of a short FP64 list counting as one (it takes a wavefront per ray):
    40 lists of 16,000 rays through three planes are more than seven
    iterations' worth.  Their results are the lone call's to the bit, split over
    iterations as they are."""
    lens, _ = field
    rng = np.random.default_rng(40)
    n, lists, planes = 16000, 40, 3
    x = (rng.random((n, 2)) - 0.5) * W.grid_range(300.0)
    ref = lens.rayshooterInternal(x)
    srv = S.Server(ctx, hbm_budget=1 << 30)
    ids = [srv.submit_rays(lens, x, precision=S.SLSIM_FP64) for _ in range(lists)]
    out = [srv.wait_rays(i, n) for i in ids]
    iterations = srv.stats()["iterations"]
    srv.close()
    assert all(_same(ref, y, A) for y, A, _ in out)
    assert iterations * 32768 >= lists * planes * (n // 8)


@pytest.mark.parametrize("N", [65, 129, 257])
@pytest.mark.parametrize("precision", [S.SLSIM_FP64, S.SLSIM_FP32C])
def test_rectangular_grid_is_the_grid_to_the_bit(field, N, precision):
    """A rectangular GridMap's points go as a list.  Over a power of two of
    radians with 2^k + 1 points a side they are the square GridMap's to the bit,
    and so are its results (FP32C up to 16,000 rays: the FP64 one's)."""
    lens, _ = field
    rg = 2.0 ** -10
    a = S.GridMap.rect(lens, N, (0.0, 0.0), rg, rg, precision)
    b = S.GridMap(lens, N, (0.0, 0.0), rg, S.SLSIM_FP64 if N * N <= LIMIT32 else precision)
    assert np.array_equal(a.positions(), b.positions())
    assert _same((a.y(), a.A()), b.y(), b.A())
