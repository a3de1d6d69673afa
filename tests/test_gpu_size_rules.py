"""GPU tests of the rules that choose a path by size: what a rule costs on both
of its sides, and the results over the ranges that it splits."""
from __future__ import annotations

import numpy as np
import pytest

import ics

pytestmark = pytest.mark.gpu

sphgpu = pytest.importorskip("sphgpu")


def _box(dim, n, seed=0):
    """n random particles of equal mass in the periodic unit box."""
    p = ics.default_params(dim)
    p.update(periodic=1, leaf_particle_num=32, range_min=[0.0] * 3, range_max=[1.0 if k < dim else 0.0 for k in range(3)])
    f = ics.empty_fields(n)
    f[ics.F_POS:ics.F_POS + dim] = np.random.default_rng([seed, n, dim]).random((dim, n))
    f[ics.F_MASS] = 1.0 / n
    f[ics.F_DENS] = f[ics.F_ENE] = 1.0
    f[ics.F_SML] = (50.0 / n) ** (1.0 / dim)
    return p, f


def test_periodic_fp32_walk_cost():
    """The FP32 gravity walk in a periodic 3D box does the FP64 walk's
    interactions with half-width registers and terms: it takes clearly less time
    (0.5 of it at 205k particles; 1.2 of it with 37 registers spilled into the
    pair loop)."""
    t = {}
    for prec in (ics.PAIR_FP32, ics.PAIR_FP64):
        p, f = _box(3, 205000)
        p.update(use_gravity=1, pair_precision=prec)
        c = sphgpu.Context(p, f.shape[1])
        c.upload(f)
        c.build_tree()
        c.gravity()
        c.enable_timing(1)
        for _ in range(5):
            c.gravity()
        t[prec] = c.kernel_times()["gravity"][0]
        c.close()
    assert t[ics.PAIR_FP32] < 0.8 * t[ics.PAIR_FP64], t
