"""Ray lists on the lone-ray FP64 walk: the sizes where its launch changes
(four wavefronts a ray, one, the bundle walk beyond), coarse leaves whose
particles outgrow its list, and big particles, against the oracle.

Tolerance: the same algorithm in the same precision, sums in another order:
relative |d alpha| <= 1e-9, |d A| <= 1e-8 (the bounds of the FP64 walk's tests).
"""
import numpy as np
import pytest

import oracle as O
import slsimlib_amd as S
from slsimlib_amd import workloads as W

pytestmark = pytest.mark.gpu

LIMIT64, LIMIT32, FOUR_WAVES = 49152, 16000, 2048


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


@pytest.mark.parametrize("n", [1, 63, 64, 65, FOUR_WAVES, FOUR_WAVES + 1, LIMIT32, LIMIT32 + 1,
                               LIMIT64, LIMIT64 + 1])
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
