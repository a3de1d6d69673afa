"""GPU tests of the paths that are chosen by the particle count, at the sizes
where they change over: tile edges, remainders, the smallest and largest."""
from __future__ import annotations

import numpy as np
import pytest

import ics

pytestmark = pytest.mark.gpu

sphgpu = pytest.importorskip("sphgpu")


def _random_state(n, dim, seed=0):
    """n random particles in the periodic unit box, some of them coincident."""
    p = ics.default_params(dim)
    p.update(periodic=1, leaf_particle_num=8, range_min=[0.0] * 3,
             range_max=[1.0 if k < dim else 0.0 for k in range(3)])
    rng = np.random.default_rng([seed, n, dim])
    f = ics.empty_fields(n)
    f[ics.F_POS:ics.F_POS + dim] = rng.random((dim, n))
    # coincident particles: their keys are equal, a stable sort keeps their order
    twin = rng.permutation(n)[: n // 16]
    f[ics.F_POS:ics.F_POS + dim, twin] = f[ics.F_POS:ics.F_POS + dim, :1]
    f[ics.F_MASS] = 1.0 / n
    f[ics.F_DENS] = 1.0
    f[ics.F_ENE] = 1.0
    f[ics.F_SML] = 0.1
    return p, f


def _key_order(p, x):
    """Stable order of the octant keys (src/bhtree.cpp:211-239: one digit per
    level from pos > centre, centres by the same FP64 recursion)."""
    d = x.shape[0]
    c = np.full_like(x, 0.5)
    e, key = 1.0, np.zeros(x.shape[1], dtype=np.uint64)
    for _ in range(p["max_tree_level"]):
        up = x > c
        c = c + np.where(up, 1.0, -1.0) * (e * 0.25)
        e *= 0.5
        key = (key << np.uint64(d)) | sum((up[k].astype(np.uint64) << np.uint64(k)) for k in range(d))
    return np.argsort(key, kind="stable")


@pytest.mark.parametrize("dim", [1, 2, 3])
@pytest.mark.parametrize("n", [1, 63, 1023, 1025, 3071, 4095, 4096, 4097, 8191, 8193, 20481])
def test_key_sort_order(n, dim):
    """The particle order of a tree build is the stable key order, for sorts in
    one workgroup (up to 4096 particles) and in tiles of 4096."""
    p, f = _random_state(n, dim)
    c = sphgpu.Context(p, n)
    c.upload(f)
    c.build_tree()
    np.testing.assert_array_equal(c.tree_dump()["members"], _key_order(p, f[ics.F_POS:ics.F_POS + dim]))
    c.close()
