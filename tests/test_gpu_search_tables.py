"""Neighbor search: the staged search against the search without sets (every
list form has to give the same lists in the same order) and against all pairs,
at the edges of its tables: few particles, block remainders, spray with
many cells a block, rows of more than 32 candidates, sets beyond the stage, a
string of particles too long for the row masks, dense walls and truncated lists."""
import numpy as np
import pytest

import splishsplash_for_cuda_amd as S
from splishsplash_for_cuda_amd.scene import box_surface, fluid_block

pytestmark = pytest.mark.gpu
R = 0.025
H = 4.0 * R


def _jitter(x, rng, j):
    return x + rng.uniform(-j * R, j * R, x.shape)


def _scene(name, rng):
    """fluid, walls, max_neighbors"""
    box = (2.0, 2.0, 2.0)
    walls = box_surface((0, 0, 0), box, 2 * R)
    maxn = 128
    if name.startswith("n="):
        n = int(name[2:])
        x = _jitter(fluid_block((0.05, 0.05, 0.05), (9, 9, 9), 2 * R), rng, 0.2)[:n]
    elif name == "spray":
        x = rng.uniform(0.05, 1.95, (3000, 3))
    elif name == "thin spray":
        x = rng.uniform(0.05, 1.95, (700, 3))
    elif name == "rows over 32":
        x = _jitter(fluid_block((0.4, 0.4, 0.4), (16, 16, 16), 1.25 * R), rng, 0.2)
        maxn = 255
    elif name == "sets over the stage":
        x = _jitter(fluid_block((0.4, 0.4, 0.4), (22, 20, 21), 1.02 * R), rng, 0.2)
        maxn = 255
    elif name == "string":
        walls = box_surface((0, 0, 0), (12.0, 0.4, 0.4), 2 * R)
        x = _jitter(np.stack([np.linspace(0.1, 11.9, 900), np.full(900, 0.2), np.full(900, 0.2)], 1), rng, 0.5)
    elif name == "dense walls":
        walls = box_surface((0, 0, 0), (0.8, 0.8, 0.8), 0.6 * R)
        x = _jitter(fluid_block((0.04, 0.04, 0.04), (15, 14, 13), 2 * R), rng, 0.2)
        maxn = 255
    else:                                       # "truncated"
        x = _jitter(fluid_block((0.05, 0.05, 0.05), (14, 13, 12), 2 * R), rng, 0.2)
        maxn = 21
    return x.astype(np.float32), walls.astype(np.float32), maxn


def _search(x, walls, maxn, mode):
    s = S.Solver(S.default_params(particle_radius=R, max_neighbors=maxn, list_mode=mode))
    s.upload_boundary(walls)
    s.upload_fluid(x)
    s.neighbor_search()
    nf, nb, L = s.neighbors()
    out = (s.download(S.FIELD_POS), s.download(S.FIELD_BOUNDARY_POS), nf, nb, L, s.neighbor_stats())
    s.close()
    return out


@pytest.mark.parametrize("name", ["n=1", "n=2", "n=63", "n=511", "n=512", "n=513", "spray", "thin spray", "rows over 32",
                                  "sets over the stage", "string", "dense walls", "truncated"])
def test_search_tables(name):
    x, walls, maxn = _scene(name, np.random.default_rng(11))
    pos, bpos, nf, nb, L, stats = _search(x, walls, maxn, S.LISTS_AUTO)
    _, _, gf, gb, G, gstats = _search(x, walls, maxn, S.LISTS_GLOBAL)
    assert stats == gstats
    assert np.array_equal(nf, gf) and np.array_equal(nb, gb) and np.array_equal(L, G)
    # all pairs in 64 bits: equal except within rounding of the support's edge
    p, q = pos.astype(np.float64), bpos.astype(np.float64)
    h2 = float(np.float32(H)) ** 2
    over = 0
    for i in range(len(p)):
        d, db = ((p - p[i]) ** 2).sum(1), ((q - p[i]) ** 2).sum(1)
        d[i] = np.inf
        edge = (np.abs(d - h2) < 1e-5 * h2).any() or (np.abs(db - h2) < 1e-5 * h2).any()
        wf, wb = np.flatnonzero(d < h2), np.flatnonzero(db < h2)
        over += len(wf) + len(wb) > maxn
        if edge:
            continue
        got_f, got_b = L[i, :nf[i]], L[i, nf[i]:nf[i] + nb[i]]
        if len(wf) + len(wb) <= maxn:
            assert np.array_equal(np.sort(got_f), wf) and np.array_equal(np.sort(got_b), wb)
        else:
            assert len(got_f) == min(len(wf), maxn) and len(got_f) + len(got_b) == maxn
            assert np.isin(got_f, wf).all() and np.isin(got_b, wb).all()
    assert over > 0 or name != "truncated"


@pytest.mark.parametrize("crowd", [0, 700])
@pytest.mark.parametrize("n", [1, 513, 4000])
def test_cell_order_is_stable(n, crowd):
    """Inside a cell the sorted particles keep the order they had (here their ids),
    also in a cell of hundreds and with ids scattered over the cells."""
    rng = np.random.default_rng(n + crowd)
    x = rng.uniform(0.1, 1.9, (n, 3))
    if crowd:
        x = np.concatenate([x, 1.0 + rng.uniform(0.0, 0.2 * H, (crowd, 3))])
        x = x[rng.permutation(len(x))]
    s = S.Solver(S.default_params(particle_radius=R, max_neighbors=20))
    s.upload_boundary(box_surface((0, 0, 0), (2.0, 2.0, 2.0), 2 * R).astype(np.float32))
    x = x.astype(np.float32)
    s.upload_fluid(x)
    s.neighbor_search()
    ids, pos, inf = s.download(S.FIELD_ID), s.download(S.FIELD_POS), s.info()
    s.close()
    assert np.array_equal(np.sort(ids), np.arange(len(x))) and np.array_equal(pos, x[ids])
    inv = np.float32(1.0 / inf.cell_size)
    cell = np.floor((pos - np.array(inf.grid_origin[:], np.float32)) * inv).astype(np.int64)
    same = (cell[1:] == cell[:-1]).all(1)
    assert (ids[1:][same] > ids[:-1][same]).all()
    # each cell is one run
    assert (~same).sum() + 1 == len(np.unique(cell, axis=0))


@pytest.mark.parametrize("name", ["n=1", "n=63", "n=513", "spray", "thin spray", "rows over 32", "dense walls", "truncated"])
def test_sweeps_agree_between_list_forms(name):
    """Both solvers on lists of every remainder (full and half batches, walls): the
    staged sweeps equal the ones over 32-bit global lists to the last bit."""
    x, walls, maxn = _scene(name, np.random.default_rng(12))
    v = np.random.default_rng(13).normal(scale=0.3, size=x.shape).astype(np.float32)
    out = []
    for mode in (S.LISTS_AUTO, S.LISTS_NO_LDS, S.LISTS_GLOBAL):
        s = S.Solver(S.default_params(particle_radius=R, max_neighbors=maxn, list_mode=mode))
        s.upload_boundary(walls)
        s.upload_fluid(x, v)
        for _ in range(2):
            s.neighbor_search()
            s.divergence_solve(4, 0.0)
            s.external_forces()
            s.update_vel()
            s.pressure_solve(3, 0.0)
        out.append([s.download(f) for f in (S.FIELD_ID, S.FIELD_VEL, S.FIELD_DENSITY, S.FIELD_FACTOR, S.FIELD_KAPPA,
                                            S.FIELD_KAPPAV, S.FIELD_ACC)])
        s.close()
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("blocks", [32, 33, 65, 129])
def test_search_shares(blocks):
    """Blocks that share a set (8, 4, 2 and 1 of them): one particle in the last one,
    lists as the search without sets has them, neighbors as a k-d tree counts them."""
    from scipy.spatial import cKDTree
    n = 512 * (blocks - 1) + 1
    rng = np.random.default_rng(blocks)
    x = _jitter(fluid_block((0.05, 0.05, 0.05), (38, 38, -(-n // 1444)), 2 * R), rng, 0.2)[:n].astype(np.float32)
    walls = box_surface((0, 0, 0), (2.0, 2.0, 0.2 + 2 * R * -(-n // 1444)), 2 * R).astype(np.float32)
    pos, bpos, nf, nb, L, stats = _search(x, walls, 96, S.LISTS_AUTO)
    _, _, gf, gb, G, gstats = _search(x, walls, 96, S.LISTS_GLOBAL)
    assert len(pos) == n and stats == gstats
    assert np.array_equal(nf, gf) and np.array_equal(nb, gb) and np.array_equal(L, G)
    p = cKDTree(pos.astype(np.float64))
    for r, low in ((H * (1 - 1e-5), True), (H * (1 + 1e-5), False)):
        wf = p.query_ball_point(pos.astype(np.float64), r, return_length=True) - 1
        wb = cKDTree(bpos.astype(np.float64)).query_ball_point(pos.astype(np.float64), r, return_length=True)
        assert ((wf <= nf) & (wb <= nb)).all() if low else ((wf >= nf) & (wb >= nb)).all()


@pytest.mark.parametrize("n", [(1 << 21) - 1, 1 << 21, 1 << 22])
def test_streamed_lists(n):
    """Sweeps on both sides of the sizes from which the lists, then the sets' ids, are
    read past the caches: the same bits as over the 32-bit lists, which never are."""
    rng = np.random.default_rng(n)
    x = fluid_block((0.05, 0.05, 0.05), (128, 128, -(-n // 16384)), 2 * R)[:n].astype(np.float32)
    x += rng.uniform(-0.2 * R, 0.2 * R, x.shape).astype(np.float32)
    v = rng.normal(scale=0.3, size=x.shape).astype(np.float32)
    walls = box_surface((0, 0, 0), (6.6, 6.6, 0.2 + 2 * R * -(-n // 16384)), 2 * R).astype(np.float32)
    out = []
    for mode in (S.LISTS_AUTO, S.LISTS_GLOBAL):
        s = S.Solver(S.default_params(particle_radius=R, max_neighbors=60, list_mode=mode))
        s.upload_boundary(walls)
        s.upload_fluid(x, v)
        s.neighbor_search()
        s.divergence_solve(2, 0.0)
        s.external_forces()
        s.update_vel()
        s.pressure_solve(2, 0.0)
        out.append([s.download(f) for f in (S.FIELD_VEL, S.FIELD_DENSITY, S.FIELD_FACTOR, S.FIELD_KAPPA, S.FIELD_ACC)])
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("fluid, wall", [(1.2, 2.0), (1.2, 0.7), (2.0, 0.6)])
def test_search_windows(fluid, wall):
    """Sets and walls that pass through the stage in windows (spacings in radii: two
    windows of the set, then of the walls too, then of the walls alone): each list's members by a k-d
    tree, in the order of the cells, with and without LDS-staged sweeps."""
    from scipy.spatial import cKDTree
    rng = np.random.default_rng(int(100 * fluid + wall))
    x = _jitter(fluid_block((0.05, 0.05, 0.05), (13, 14, 15), fluid * R), rng, 0.2).astype(np.float32)
    walls = box_surface((0, 0, 0), (0.8, 0.8, 0.8), wall * R).astype(np.float32)
    pos, bpos, nf, nb, L, stats = _search(x, walls, 255, S.LISTS_AUTO)
    for mode in (S.LISTS_NO_LDS, S.LISTS_GLOBAL):
        other = _search(x, walls, 255, mode)
        assert np.array_equal(nf, other[2]) and np.array_equal(nb, other[3]) and np.array_equal(L, other[4])
    p, q = pos.astype(np.float64), bpos.astype(np.float64)
    lo_f, hi_f = (cKDTree(p).query_ball_point(p, H * (1 + e)) for e in (-1e-5, 1e-5))
    lo_b, hi_b = (cKDTree(q).query_ball_point(p, H * (1 + e)) for e in (-1e-5, 1e-5))
    assert (nf + nb).max() < 255                # no list is truncated
    for i in range(len(p)):
        f, b = L[i, :nf[i]], L[i, nf[i]:nf[i] + nb[i]]
        assert set(lo_f[i]) - {i} <= set(f) <= set(hi_f[i]) - {i} and len(set(f)) == len(f)
        assert set(lo_b[i]) <= set(b) <= set(hi_b[i]) and len(set(b)) == len(b)


@pytest.mark.parametrize("at", [0.05, 0.2])
def test_search_across_octants(at):
    """Blocks that run from one octant of a 32-cell cube to the next, whose set's box has
    34 x 34 rows: neighbors as a k-d tree counts them, few particles around."""
    from scipy.spatial import cKDTree
    rng = np.random.default_rng(int(100 * at))
    edge = 16 * 1.001 * H                         # between the cube's octants
    corner = np.stack(np.meshgrid(*[[0.0, edge - 6 * R, edge + 4 * R, 2 * edge - 6 * R]] * 3, indexing="ij"), -1).reshape(-1, 3)
    x = np.concatenate([_jitter(fluid_block(c, (3, 3, 3), 2 * R), rng, 0.2) for c in corner + at]).astype(np.float32)
    walls = box_surface((0, 0, 0), (4.0, 4.0, 4.0), 2 * R).astype(np.float32)
    pos, bpos, nf, nb, L, stats = _search(x, walls, 96, S.LISTS_AUTO)
    trees = cKDTree(pos.astype(np.float64)), cKDTree(bpos.astype(np.float64))
    p = pos.astype(np.float64)
    for r, low in ((H * (1 - 1e-5), True), (H * (1 + 1e-5), False)):
        wf = trees[0].query_ball_point(p, r, return_length=True) - 1
        wb = trees[1].query_ball_point(p, r, return_length=True)
        assert ((wf <= nf) & (wb <= nb)).all() if low else ((wf >= nf) & (wb >= nb)).all()


@pytest.mark.parametrize("name", ["n=513", "spray", "dense walls"])
def test_sweeps_between_sorted_and_unsorted_searches(name):
    """Solves on the lists of an unsorted search (no block has a set) between solves on
    sorted ones: the same bits as with 32-bit lists throughout."""
    x, walls, maxn = _scene(name, np.random.default_rng(14))
    v = np.random.default_rng(15).normal(scale=0.3, size=x.shape).astype(np.float32)
    out = []
    for mode in (S.LISTS_AUTO, S.LISTS_GLOBAL):
        s = S.Solver(S.default_params(particle_radius=R, max_neighbors=maxn, list_mode=mode))
        s.upload_boundary(walls)
        s.upload_fluid(x, v)
        fields = []
        for sort in (True, False, False, True):
            s.neighbor_search(sort)
            s.divergence_solve(3, 0.0)
            s.external_forces()
            s.update_vel()
            s.pressure_solve(2, 0.0)
            fields += [s.download(f) for f in (S.FIELD_ID, S.FIELD_VEL, S.FIELD_DENSITY, S.FIELD_FACTOR, S.FIELD_KAPPA,
                                               S.FIELD_KAPPAV, S.FIELD_ACC)]
        out.append(fields)
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b, equal_nan=True)


@pytest.mark.parametrize("name", ["n=1", "n=2", "n=513", "spray", "rows over 32", "dense walls", "truncated"])
def test_unsorted_search(name):
    """The search of fluid left in its order, here a shuffled one, cells of every size: the
    lists of the sorted search, as ids and in the same order."""
    x, walls, maxn = _scene(name, np.random.default_rng(16))
    x = x[np.random.default_rng(17).permutation(len(x))]
    s = S.Solver(S.default_params(particle_radius=R, max_neighbors=maxn))
    s.upload_boundary(walls)
    s.upload_fluid(x)
    s.neighbor_search(False)
    assert np.array_equal(s.download(S.FIELD_POS), x)
    nf, nb, L = s.neighbors()
    s.neighbor_search()
    ids = s.download(S.FIELD_ID)
    sf, sb, G = s.neighbors()
    s.close()
    assert np.array_equal(nf[ids], sf) and np.array_equal(nb[ids], sb) and sf.max() >= (len(x) > 2)
    for k, i in enumerate(ids):
        f = int(sf[k])
        assert np.array_equal(ids[G[k, :f]], L[i, :f])
        assert np.array_equal(G[k, f:f + int(sb[k])], L[i, f:f + int(sb[k])])


@pytest.mark.parametrize("n", [(1 << 28) // 85 - 1, (1 << 28) // 85])
def test_streamed_ids(n):
    """The same on both sides of the size from which the ids are streamed too."""
    test_streamed_lists(n)
