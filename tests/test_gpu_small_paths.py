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


def _hk_sum(x, m, h, g):
    """Direct softened sum (src/bhtree.cpp:319-345, 362-378), FP64."""
    d = x[:, :, None] - x[:, None, :]
    r = np.sqrt((d * d).sum(axis=0))
    np.fill_diagonal(r, 1.0)

    def fg(e):
        u = r / e
        f1 = (-0.5 * u * u * (1 / 3 - 3 / 20 * u * u + u ** 3 / 20) + 1.4) / e
        f2 = -1 / (15 * r) + (-u * u * (4 / 3 - u + 0.3 * u * u - u ** 3 / 30) + 1.6) / e
        g1 = (4 / 3 - 1.2 * u * u + 0.5 * u ** 3) / e ** 3
        g2 = (-1 / 15 + 8 / 3 * u ** 3 - 3 * u ** 4 + 1.2 * u ** 5 - u ** 6 / 6) / r ** 3
        return np.where(u < 1, f1, np.where(u < 2, f2, 1 / r)), np.where(u < 1, g1, np.where(u < 2, g2, 1 / r ** 3))

    fi, gi = fg(np.broadcast_to(0.5 * h[:, None], r.shape))
    fj, gj = fg(np.broadcast_to(0.5 * h[None, :], r.shape))
    w = g * np.broadcast_to(m[None, :], r.shape).copy()
    np.fill_diagonal(w, 0.0)
    return -(0.5 * w * (fi + fj)).sum(axis=1), -(d * (0.5 * w * (gi + gj))).sum(axis=2)


@pytest.mark.parametrize("prec,tol", [(ics.PAIR_FP64, 1e-12), (ics.PAIR_FP32, 2e-6)])
@pytest.mark.parametrize("n,leaf", [(2, 1), (9, 1), (63, 4), (64, 64), (65, 1), (300, 8), (1500, 32)])
def test_gravity_pieces_direct_sum(n, leaf, prec, tol):
    """With theta = 0 every node is opened, so the walk's pieces (as many as the
    nodes, at the smallest sizes) must add up to the direct sum.  FP32: 20 u of
    the summed magnitudes (positions rounded to FP32 move a term by a few u;
    the sums are compensated), FP64 far below."""
    rng = np.random.default_rng([n, leaf])
    p = ics.default_params(3)
    p.update(use_gravity=1, theta=0.0, leaf_particle_num=leaf, pair_precision=prec, gravity_constant=0.7)
    f = ics.empty_fields(n)
    f[ics.F_POS:ics.F_POS + 3] = rng.uniform(-1, 1, (3, n))
    f[ics.F_MASS] = rng.uniform(0.5, 1.5, n) / n
    f[ics.F_DENS] = f[ics.F_ENE] = 1.0
    f[ics.F_SML] = rng.uniform(0.1, 0.5, n)
    c = sphgpu.Context(p, n)
    c.upload(f)
    c.build_tree()
    c.gravity()
    out = c.download()
    c.close()
    phi, acc = _hk_sum(f[ics.F_POS:ics.F_POS + 3], f[ics.F_MASS], f[ics.F_SML], 0.7)
    np.testing.assert_allclose(out[ics.F_PHI], phi, rtol=tol)
    # acceleration on the scale of the terms' magnitudes, not of their sum
    x = f[ics.F_POS:ics.F_POS + 3]
    d = x[:, :, None] - x[:, None, :]
    r2 = (d * d).sum(axis=0) + np.eye(n)
    scale = (0.7 * f[ics.F_MASS][None, :] / r2 * (1 - np.eye(n))).sum(axis=1)
    assert (np.abs(out[ics.F_ACC:ics.F_ACC + 3] - acc) / scale).max() < tol


@pytest.mark.parametrize("dim,periodic", [(3, 1), (3, 0), (2, 1), (1, 0)])
@pytest.mark.parametrize("n", [7, 64, 65, 32768, 32769, 98304, 98305, 262143, 262144])
def test_search_sets_by_size(n, dim, periodic):
    """Neighbour sets at the sizes where the search changes its lanes per
    particle, both predicates, exact against FP64 distances from a sample of
    particles (the first, the last and random ones).  Small and large leaves."""
    rng = np.random.default_rng([n, dim])
    p = ics.default_params(dim)
    p.update(periodic=periodic, leaf_particle_num=1 if n % 2 else 20, range_min=[0.0] * 3,
             range_max=[1.0 if k < dim else 0.0 for k in range(3)])
    f = ics.empty_fields(n)
    x = rng.random((dim, n))
    f[ics.F_POS:ics.F_POS + dim] = x
    f[ics.F_MASS] = 1.0 / n
    f[ics.F_DENS] = f[ics.F_ENE] = 1.0
    # about 20 neighbours, radii within a factor of 1.5
    h = {1: 10.0 / n, 2: (20 / np.pi / n) ** 0.5, 3: (15 / np.pi / n) ** (1 / 3)}[dim] * rng.uniform(0.8, 1.2, n)
    h = np.minimum(h, 0.4)
    c = sphgpu.Context(p, n)
    c.upload(f)
    c.build_tree()
    pick = np.unique(np.concatenate([[0, n - 1], rng.integers(0, n, 60)]))
    for is_ij in (0, 1):
        cnt, lists = c.neighbor_sets(h, is_ij, cap=160)
        for i in pick:
            d = x[:, i:i + 1] - x
            if periodic:
                d = np.where(np.abs(d) <= np.abs(np.abs(d) - 1.0), d, d - np.sign(d))
            r2 = d[0] * d[0]
            for k in range(1, dim):
                r2 = r2 + d[k] * d[k]
            want = (np.sqrt(r2) < np.maximum(h[i], h)) & (r2 != 0.0) if is_ij else r2 < h[i] * h[i]
            np.testing.assert_array_equal(np.sort(lists[i, :cnt[i]]), np.flatnonzero(want))
    c.close()


@pytest.mark.parametrize("n", [1, 63, 65, 4096, 4097, 8192, 12353])
def test_mlp_gradient_by_rows(n):
    """Loss and gradient over n rows, at the edges of the 64-row tiles and of
    the 64 tiles whose partial gradients one chain sums, against the FP64
    reference: bf16 operands (2^-9 relative rounding each, three layers deep)
    leave the gradient's direction within 1e-3 and its norm within 5e-2."""
    import sys
    from pathlib import Path
    sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "oracle"))
    import mlp_oracle as M
    rng = np.random.default_rng(n)
    rows = np.stack([rng.normal(0, 0.5, n), rng.uniform(0.3, 3, n), 10 ** rng.uniform(-1, 0.5, n),
                     rng.normal(0, 0.5, n), rng.uniform(0.3, 3, n), 10 ** rng.uniform(-1, 0.5, n),
                     10 ** rng.uniform(-1, 0.5, n)], 1).astype(np.float32)
    p, f = ics.sedov_3d(4)
    c = sphgpu.Context(p, f.shape[1])
    c.mlp_init(seed=3)
    loss, grad = c.mlp_loss_grad(rows)
    want_loss, want = M.loss_grad(c.mlp_get_params(), rows, p["gamma"])
    assert abs(loss - want_loss) < 2e-2 * want_loss
    assert grad @ want > 0.999 * np.linalg.norm(grad) * np.linalg.norm(want)
    assert abs(np.linalg.norm(grad) / np.linalg.norm(want) - 1) < 5e-2
    # the evaluation after training is the loss of the same rows (a rate of 0
    # leaves the weights): the same tiles' losses, summed in FP64
    assert abs(c.mlp_train(rows, 1, 1000, 0.0) - loss) <= 1e-6 * loss
    c.close()


def _slab_with_cluster(total, side, seed=1):
    """A jittered lattice in the lower half of the unit box and a small dense
    cluster of side^3 particles at its upper corner (which fixes the root cell),
    out of reach of the rest: `total` lattice particles come first in key order
    and neither their tree cells nor their neighbours depend on the cluster."""
    rng = np.random.default_rng(seed)
    nz = int((total / 4) ** (1 / 3))
    nx = int(np.ceil((total / nz) ** 0.5))
    g = np.stack(np.meshgrid(*[(np.arange(k) + 0.5) / nx for k in (nx, nx, nz)], indexing="ij")).reshape(3, -1)
    g = (g + rng.uniform(-0.2, 0.2, g.shape) / nx)[:, :total]
    assert g.shape[1] == total and g[2].max() < 0.5
    g[:, 0] = 0.0  # the lower corner of the root cell
    c = np.stack(np.meshgrid(*[1.0 - 0.001 * np.arange(side)] * 3, indexing="ij")).reshape(3, -1)
    n = total + side ** 3
    f = ics.empty_fields(n)
    f[ics.F_POS:ics.F_POS + 3] = np.concatenate([g, c], axis=1)
    f[ics.F_VEL:ics.F_VEL + 3, :total] = 0.3 * np.sin(7.0 * g)
    f[ics.F_MASS] = 1.0 / nx ** 3
    f[ics.F_DENS, :total] = 1.0
    f[ics.F_DENS, total:] = 1e9 / nx ** 3
    f[ics.F_ENE, :total] = 1.0 + 0.3 * np.sin(9.0 * g[0]) + 0.05 * rng.random(total)
    f[ics.F_ENE, total:] = 1.0
    f[ics.F_SOUND] = np.sqrt(10.0 / 9.0 * f[ics.F_ENE])
    f[ics.F_ALPHA] = f[ics.F_BALSARA] = 1.0
    return f


@pytest.mark.parametrize("limit,prec,over", [
    (131072, ics.PAIR_FP32, dict(sph_type=ics.GSPH, riemann_solver=ics.RIEMANN_ITERATIVE)),
    (131072, ics.PAIR_FP32, dict(sph_type=ics.GDISPH, gsph_2nd_order=1)),
    (131072, ics.PAIR_FP32, dict(sph_type=ics.DISPH, kernel=ics.WENDLAND, use_time_dependent_av=1)),
    (131072, ics.PAIR_FP32, dict(sph_type=ics.SSPH, use_ac=1)),
    (196608, ics.PAIR_FP32, dict(sph_type=ics.GSPH, riemann_solver=ics.RIEMANN_ITERATIVE)),
    (196608, ics.PAIR_FP32, dict(sph_type=ics.GSPH, riemann_solver=ics.RIEMANN_HLL, gsph_2nd_order=0)),
    (524288, ics.PAIR_FP64, dict(sph_type=ics.GSPH, riemann_solver=ics.RIEMANN_ITERATIVE)),
])
def test_quad_and_single_lane_forms_agree(limit, prec, over):
    """PreInteraction and the GSPH force run with a quad of lanes per particle up
    to a size and with one lane beyond; both add every sum in the same order, so
    the particles that the two sizes share must come out bit for bit equal."""
    out = []
    total = limit - 150
    for side in (5, 6):  # total + 125 <= limit < total + 216
        f = _slab_with_cluster(total, side)
        p = ics.default_params(3)
        p.update(neighbor_number=40, leaf_particle_num=32, pair_precision=prec, gamma=5.0 / 3.0, **over)
        c = sphgpu.Context(p, f.shape[1])
        c.upload(f)
        c.dt = 1e-4
        c.build_tree()
        # the first rounds settle h at the free surfaces, where the guess from
        # the given densities is too small for the derived force lists
        for _ in range(4):
            c.pre_interaction()
        c.fluid_force()
        g = c.download()[:, :total]
        assert c.stats()["flist_searches"] == 0
        c.close()
        out.append(g)
    assert np.isfinite(out[0]).all() and np.abs(out[0][ics.F_ACC]).max() > 0
    for row in range(out[0].shape[0]):
        np.testing.assert_array_equal(out[0][row], out[1][row], err_msg=f"field row {row}")


@pytest.mark.parametrize("nn,reach", [(20, 0.0), (20, 0.15), (60, 0.35), (60, 0.6), (200, 0.9)])
def test_force_list_runs_sorted(nn, reach):
    """Force lists whose appended part (particles j with h_j > r >= h_i) is
    short, of tens, of up to a few hundred entries (each sorted its own way): the
    lists hold the exact pair sets, and two contexts agree bit for bit in the
    forces whatever order the appends came in.  A sparse half with large h beside
    a dense half gives the long runs; `reach` widens the sparse spacing."""
    n_dense, n_sparse = 3000, 300
    p = ics.default_params(1)
    p.update(neighbor_number=nn, leaf_particle_num=4, gamma=1.4, pair_precision=ics.PAIR_FP32)
    n = n_dense + n_sparse
    f = ics.empty_fields(n)
    rng = np.random.default_rng([nn, int(100 * reach)])
    dx = 1.0 / n_dense
    f[ics.F_POS] = np.concatenate([-(np.arange(n_dense) + 0.5) * dx, (np.arange(n_sparse) + 0.5) * dx * (1 + 20 * reach)])
    f[ics.F_POS] += 0.1 * dx * rng.uniform(-1, 1, n)
    f[ics.F_MASS] = dx
    f[ics.F_DENS] = f[ics.F_ENE] = 1.0
    f[ics.F_DENS, n_dense:] = 1.0 / (1 + 20 * reach)
    f[ics.F_SOUND] = 1.0
    runs = []
    for _ in range(2):
        c = sphgpu.Context(p, n)
        c.upload(f)
        c.build_tree()
        for _ in range(4):
            c.pre_interaction()
        cnt, lists = c.neighbor_sets(None, 2, cap=4096)
        c.fluid_force()
        out = c.download()
        c.close()
        runs.append(out)
    x, h = out[ics.F_POS], out[ics.F_SML]
    tail = 0
    for i in range(n_dense - 200, n, 3):
        r = np.sqrt((x[i] - x) ** 2)
        want = np.flatnonzero((r < np.maximum(h[i], h)) & (r != 0.0))
        np.testing.assert_array_equal(np.sort(lists[i, :cnt[i]]), want)
        tail = max(tail, int((r[want] >= h[i]).sum()))
    print("longest appended run", tail)
    np.testing.assert_array_equal(runs[0], runs[1])


@pytest.mark.parametrize("dim,leaf", [(1, 1), (2, 1), (3, 1), (3, 8), (2, 70)])
@pytest.mark.parametrize("n", [1, 2, 9, 64, 65, 513, 4097, 70001])
def test_tree_ranges_and_children(n, dim, leaf):
    """Node ranges (found eight probes at a time), pre-order and the partition of
    every node's members by its children, for random and coincident particles,
    and for a second build after the particles moved (its launches are sized by
    the first one's nodes, here far fewer)."""
    p, f = _random_state(n, dim, seed=leaf)
    p["leaf_particle_num"] = leaf
    c = sphgpu.Context(p, n)
    packed = f.copy()
    packed[ics.F_POS:ics.F_POS + dim] = 0.5  # one cell to the last level
    # (a chain of 21 nodes exceeds the pool of 5 n + 1 below five particles)
    for state in (packed, f) if n > 4 else (f, f):
        c.upload(state)
        c.build_tree()
        d = c.tree_dump()
        members, first, count, level = d["members"], d["first"], d["count"], d["level"]
        x = state[ics.F_POS:ics.F_POS + dim][:, members]
        assert first[0] == 0 and count[0] == n and level[0] == 1
        parents, used = [], np.zeros(len(level), dtype=int)
        for k in range(len(level)):
            while parents and level[parents[-1]] >= level[k]:
                parents.pop()
            if parents:
                q = parents[-1]
                assert level[k] == level[q] + 1 and first[k] == first[q] + used[q]
                used[q] += count[k]
            parents.append(k)
            inside = x[:, first[k]:first[k] + count[k]]
            assert (np.abs(inside - d["center"][k, :dim, None]) <= 0.5 * d["edge"][k]).all()
        leafs = d["is_leaf"] == 1
        assert (used[~leafs] == count[~leafs]).all() and (used[leafs] == 0).all()
        assert ((count[leafs] <= leaf) | (level[leafs] == p["max_tree_level"] + 1)).all()
        assert (count[~leafs][1:] > leaf).all()
    c.close()


@pytest.mark.parametrize("dim,leaf", [(1, 1), (3, 8)])
@pytest.mark.parametrize("n", [5, 63, 64, 65, 4095, 4096, 4097, 8193, 300001])
def test_node_kernel_sizes(n, dim, leaf):
    """Largest smoothing length below every node (maxima over blocks of 64 and
    of 4096 particles, both levels in one launch), exactly."""
    p, f = _random_state(n, dim, seed=3)
    p["leaf_particle_num"] = leaf
    f[ics.F_SML] = 0.01 + 0.1 * np.random.default_rng(n).random(n)
    c = sphgpu.Context(p, n)
    c.upload(f)
    c.build_tree()
    c.set_kernel()
    d = c.tree_dump()
    h = f[ics.F_SML][d["members"]]
    top = [h[a:a + k].max() for a, k in zip(d["first"], d["count"])]
    np.testing.assert_array_equal(d["kernel_size"], top)
    c.close()


def _hk_pair(r, h):
    """Softened f and g of one particle against several, by their own lengths."""
    e = 0.5 * h
    u = r / e
    f1 = (-0.5 * u * u * (1 / 3 - 3 / 20 * u * u + u ** 3 / 20) + 1.4) / e
    f2 = -1 / (15 * r) + (-u * u * (4 / 3 - u + 0.3 * u * u - u ** 3 / 30) + 1.6) / e
    g1 = (4 / 3 - 1.2 * u * u + 0.5 * u ** 3) / e ** 3
    g2 = (-1 / 15 + 8 / 3 * u ** 3 - 3 * u ** 4 + 1.2 * u ** 5 - u ** 6 / 6) / r ** 3
    return np.where(u < 1, f1, np.where(u < 2, f2, 1 / r)), np.where(u < 1, g1, np.where(u < 2, g2, 1 / r ** 3))


@pytest.mark.parametrize("prec,tol", [(ics.PAIR_FP64, 1e-12), (ics.PAIR_FP32, 2e-6)])
@pytest.mark.parametrize("n,leaf,theta", [(40, 4, 0.5), (65, 1, 1.5), (700, 8, 0.5), (700, 33, 0.8), (900, 65, 0.5),
                                          (1500, 140, 1.0), (3000, 32, 0.7)])
def test_gravity_opened_leaves(n, leaf, theta, prec, tol):
    """Leaves opened by any number of a wavefront's lanes (1, 2, 4, 8 or 16
    lanes take one particle's members, 32 or 64 of them at a time) against the
    walk of every particle by itself.  Tolerances as for the direct sum above:
    20 u of the summed magnitudes in FP32."""
    rng = np.random.default_rng([n, leaf, 5])
    p = ics.default_params(3)
    p.update(use_gravity=1, theta=theta, leaf_particle_num=leaf, pair_precision=prec, gravity_constant=0.7)
    f = ics.empty_fields(n)
    x = rng.normal(0, 1, (3, n))
    f[ics.F_POS:ics.F_POS + 3] = x
    m = f[ics.F_MASS] = rng.uniform(0.5, 1.5, n) / n
    f[ics.F_DENS] = f[ics.F_ENE] = 1.0
    h = f[ics.F_SML] = rng.uniform(0.1, 0.9, n)
    c = sphgpu.Context(p, n)
    c.upload(f)
    c.build_tree()
    d = c.tree_dump()
    c.gravity()
    out = c.download()
    c.close()
    level, e2, members = d["level"], d["edge"] ** 2, d["members"]
    skip = [next((j for j in range(k + 1, len(level)) if level[j] <= level[k]), len(level)) for k in range(len(level))]
    worst = 0.0
    for i in range(0, n, max(1, n // 300)):
        phi, acc, s_phi, s_acc, k = 0.0, np.zeros(3), 0.0, 0.0, 0
        while k < len(level):
            v = x[:, i] - d["com"][k]
            r2 = (v * v).sum()
            if e2[k] > theta * theta * r2 or r2 < e2[k]:
                if d["is_leaf"][k]:
                    j = members[d["first"][k]:d["first"][k] + d["count"][k]]
                    j = j[j != i]
                    dx = x[:, [i]] - x[:, j]
                    r = np.sqrt((dx * dx).sum(axis=0))
                    (fi, gi), (fj, gj) = _hk_pair(r, h[i]), _hk_pair(r, h[j])
                    t = 0.35 * m[j] * (fi + fj)
                    q = dx * (0.35 * m[j] * (gi + gj))
                    phi, acc = phi - t.sum(), acc - q.sum(axis=1)
                    s_phi, s_acc = s_phi + t.sum(), s_acc + (0.7 * m[j] / (r * r)).sum()
                k += 1
                continue
            phi, acc = phi - 0.7 * d["mass"][k] / np.sqrt(r2), acc - 0.7 * d["mass"][k] / r2 ** 1.5 * v
            s_phi, s_acc = s_phi + 0.7 * d["mass"][k] / np.sqrt(r2), s_acc + 0.7 * d["mass"][k] / r2
            k = skip[k]
        worst = max(worst, abs(out[ics.F_PHI, i] - phi) / s_phi,
                    np.abs(out[ics.F_ACC:ics.F_ACC + 3, i] - acc).max() / s_acc)
    assert worst < tol


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("n", [1, 511, 4097, 13107, 26215, 52429, 131072, 1000003])
def test_exchange_rows(n, pinned):
    """Uploads and downloads of many and of few rows, in one or several rounds
    through the pinned halves, and directly from pinned
    memory: every masked row exactly, the others untouched."""
    torch = pytest.importorskip("torch")
    p = ics.default_params(3)
    c = sphgpu.Context(p, n)
    rows = [r for a in (ics.F_POS, ics.F_VEL, ics.F_ACC) for r in (a, a + 1, a + 2)]
    rows += [ics.F_MASS, ics.F_DENS, ics.F_ENE, ics.F_SML]
    rng = np.random.default_rng(n)
    block = torch.empty((ics.NFIELDS if hasattr(ics, "NFIELDS") else sphgpu.NFIELDS, n), dtype=torch.float64,
                        pin_memory=pinned)
    f = block.numpy()
    want = np.zeros_like(f)
    f[:] = -7.0
    for some in (rows, rows[2:6] + rows[11:], rows[:1]):
        for r in some:
            want[r] = f[r] = rng.random(n)
        c.upload(f, sum(1 << r for r in some))
        f[some] = -7.0  # the upload is complete when it returns
        for part in (rows, rows[5:7], rows[-1:]):
            got = c.download(sum(1 << r for r in part))
            assert (got[part] == want[part]).all()
            rest = np.setdiff1d(np.arange(f.shape[0]), part)
            assert (got[rest] == 0).all()
    f[:] = -7.0
    c._check(c.lib.sphgpu_download(c.h, sphgpu._dp(f), sum(1 << r for r in rows)), "download")
    assert (f[rows] == want[rows]).all()
    assert (f[np.setdiff1d(np.arange(f.shape[0]), rows)] == -7.0).all()
    c.close()


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("n", [3, 65, 500, 4096, 4097, 16384, 16385, 65535])
def test_key_sort_order_clustered(n, dim):
    """The sort by the top bits and the ordering within their cells against the
    stable order of the whole keys: particles alone, in cells of a few, in cells
    of hundreds (later builds then take more passes), and coincident."""
    p, f = _random_state(n, dim, seed=9)
    rng = np.random.default_rng([n, dim])
    x = f[ics.F_POS:ics.F_POS + dim]
    k = n // 3
    x[:, :k] = 0.3 + 1e-4 * rng.random((dim, k))
    x[:, k:2 * k] = 0.7 + 0.02 * rng.random((dim, k))
    x[:, 2 * k:2 * k + n // 9] = x[:, :1]
    x[:] = x[:, rng.permutation(n)]
    want = _key_order(p, x)
    c = sphgpu.Context(p, n)
    for _ in range(4):
        c.upload(f)
        c.build_tree()
        order = c.tree_dump()["members"]
        # coincident particles keep the order of the build before: compare by key
        rank = np.empty(n, dtype=int)
        rank[want] = np.arange(n)
        moved = order != want
        assert (x[:, order[moved]] == x[:, want[moved]]).all()
    c.close()


@pytest.mark.parametrize("dim,n,levels", [(2, 20000, 2), (3, 70000, 2), (1, 5000, 2), (3, 6000, 1)])
def test_wide_leaves(dim, n, levels):
    """Leaves of more than 512 particles (a shallow tree; more of them in one
    workgroup than it notes, too): the search through their boxes finds the same
    neighbours as through the leaves of the deep tree."""
    p, f = _random_state(n, dim, seed=4)
    f[ics.F_POS:ics.F_POS + dim] = np.random.default_rng(n).random((dim, n))
    h = np.full(n, {1: 10 / n, 2: (10 / n) ** 0.5 / 2, 3: (10 / n) ** (1 / 3) / 2}[dim])
    found = []
    for ml in (levels, 20):
        q = dict(p)
        q["max_tree_level"] = ml
        c = sphgpu.Context(q, n)
        c.upload(f)
        c.build_tree()
        if ml == levels:
            assert (c.tree_dump()["count"][c.tree_dump()["is_leaf"] == 1] > 512).any()
        count, lists = c.neighbor_sets(h, 0, cap=128)
        found.append((count, np.sort(np.where(np.arange(128) < count[:, None], lists, n), axis=1)))
        c.close()
    np.testing.assert_array_equal(found[0][0], found[1][0])
    np.testing.assert_array_equal(found[0][1], found[1][1])
