"""Group neighbor walk (64 particles and 64 candidates at a time on the matrix
cores): the lists it writes hold the oracle's pairs, each once, where its
windows, passes and remainders can go wrong — grids of 2 to 9 cells per axis,
boxes of unequal edges, groups that straddle replicas and grid rows, 1 to 64
particles, more candidates than one segment, several list radii.
"""

import numpy as np
import pytest

import oracle
from azplugins_amd import _azp
from azplugins_amd.batch import ReplicaBatch
from gpu_util import say

torch = _azp.torch
pytestmark = pytest.mark.gpu

RC, BUFF = 1.1, 0.4
RL = RC + BUFF


def _batch_lists(boxes, pos4, r_cut):
    """Directed pairs (i << 32 | j) of every replica, by replica-local index."""
    nt = r_cut.shape[0]
    b = ReplicaBatch([p.shape[0] for p in pos4], boxes, ntypes=nt, r_cut=RC, r_buff=BUFF, precision="fp64")
    for i in range(nt):
        for j in range(i, nt):
            b.set_params(i, j, M_d=1.0, M_r=0.2, r_eq=1.0, omega=20.0, alpha=0.4, repulsion=True)
            _azp.call("azp_batch_set_r_cut", b._h, i, j, float(r_cut[i, j]))
    b.load(np.concatenate(pos4))
    b.compute(force_rebuild=True)
    nn, lst = b.nlist()
    out = []
    for r in range(len(pos4)):
        lo, hi = int(b.offsets[r]), int(b.offsets[r + 1])
        n = nn[lo:hi].astype(np.int64)
        k = np.arange(lst.shape[0])[:, None] < n[None, :]
        j = lst[:, lo:hi].astype(np.int64) - lo
        i = np.broadcast_to(np.arange(hi - lo)[None, :], j.shape)
        assert np.all((j[k] >= 0) & (j[k] < hi - lo)), "neighbor outside its replica"
        out.append(np.sort((i[k] << 32) | j[k]))
    return out


def _oracle_pairs(box, pos4, r_cut):
    nt = r_cut.shape[0]
    a, b = (x.astype(np.int64) for x in oracle.nlist(pos4, np.asarray(box), nt,
                                                     oracle.r_listsq_matrix(r_cut.ravel(), BUFF), "brute"))
    return np.sort(np.concatenate([(a << 32) | b, (b << 32) | a]))


def _check(boxes, sizes, r_cut, seed):
    rng = np.random.default_rng(seed)
    pos4 = []
    for box, n in zip(boxes, sizes):
        p = np.zeros((n, 4))
        p[:, :3] = rng.uniform(-0.5, 0.5, (n, 3)) * np.asarray(box)
        p[:, 3] = rng.integers(0, r_cut.shape[0], n)
        pos4.append(p)
    say(f"[group walk] sizes {sizes} types {r_cut.shape[0]}")
    got = _batch_lists(boxes, pos4, r_cut)
    for r, (box, p) in enumerate(zip(boxes, pos4)):
        assert np.array_equal(got[r], _oracle_pairs(box, p, r_cut)), f"replica {r}"


@pytest.mark.parametrize("cells", [2, 3, 4, 5, 6, 7, 9])
def test_group_walk_grids(cells):
    """Cubic and unequal boxes of `cells` cells on the shortest axis."""
    L = cells * RL * (1.0 + 1e-8)
    boxes = [(L, L, L), (L, 1.7 * L, 1.1 * L), (1.3 * L, L, 2.4 * L), (cells * RL,) * 3, (L, L, L)]
    _check(boxes, [31, 700, 333, 64, 1], np.array([[RC]]), cells)


def test_group_walk_straddling_replicas():
    """Replicas of a few particles share groups."""
    rng = np.random.default_rng(3)
    sizes = [1, 2, 3, 5, 8, 13, 21, 32, 33, 7, 1, 64]
    boxes = [tuple(rng.uniform(2.0, 7.0, 3) * RL) for _ in sizes]
    _check(boxes, sizes, np.array([[RC]]), 4)


def test_group_walk_more_candidates_than_a_segment():
    """Three cells per axis hold 8,700 candidates for every particle."""
    L = 3.1 * RL
    _check([(L, L, L), (L, L, L)], [8700, 40], np.array([[RC]]), 5)


@pytest.mark.parametrize("types", [2, 3, 8, 11])
def test_group_walk_list_radii(types):
    """Several list radii, excluded type pairs among them."""
    rng = np.random.default_rng(types)
    rc = rng.uniform(0.5 * RC, RC, (types, types))
    rc = np.minimum(rc, rc.T)
    rc[0, 0] = RC
    rc[1, 1] = 0.0
    rc[0, types - 1] = rc[types - 1, 0] = 0.0
    L = 4.2 * RL
    _check([(L, L, L), (2.1 * RL, 1.5 * L, L), (2.5 * L, L, L)], [500, 200, 900], rc, 6)


@pytest.mark.parametrize("types", [1, 11])
@pytest.mark.parametrize("edge", [2.2, 3.3])
def test_group_walk_elongated_boxes(edge, types):
    """Boxes 10,000 to 1,000,000 list radii long hold pairs at the list radius
    give or take 1e-7 to 1e-3: a fixed-point step is up to 2e-4 list radii."""
    rng = np.random.default_rng(17 + types)
    rc = np.full((types, types), RC)
    if types > 1:
        rc[1, 1] = 0.7 * RC  # several radii among more than eight types: direct tests
    boxes, pos4 = [], []
    for length in (1e4, 1e5, 1e6):
        box = np.array([edge * RL, edge * RL, length * RL])
        n = 400
        a = (rng.random((n, 3)) - 0.5) * box
        a[:, 2] = (np.arange(n) + 0.5 - n / 2) * box[2] / n
        d = rng.normal(size=(n, 3)) * [0.3, 0.3, 1.0]
        d /= np.linalg.norm(d, axis=1)[:, None]
        far = 1.0 + rng.choice([-1.0, 1.0], n) * 10.0 ** rng.uniform(-7, -3, n)
        p = np.concatenate([a, a + d * (RL * far)[:, None]])
        p -= box * np.floor(p / box + 0.5)
        q = np.zeros((2 * n, 4))
        q[:, :3] = p
        q[:, 3] = rng.integers(0, types, 2 * n)
        boxes.append(tuple(box))
        pos4.append(q)
    got = _batch_lists(boxes, pos4, rc)
    for r, (box, p) in enumerate(zip(boxes, pos4)):
        assert np.array_equal(got[r], _oracle_pairs(box, p, rc)), f"replica {r}"


def test_group_walk_reach_of_half_a_box():
    """Six cells that fit the box to 1e-9: a particle on the far face of its
    pass's cells and a neighbor at the list radius lie half a box from the
    pass's middle to within one fixed-point step."""
    L = 6.0 * RL * (1.0 + 1e-9) * (1.0 + 1e-12)
    assert int(L / (RL * (1.0 + 1e-9))) == 6
    rng = np.random.default_rng(1)
    pos4 = []
    for axis in range(3):
        for flip in (1.0, -1.0):
            # cells 2, 3, 4 and 5 of one row; the middle particle lies in cell 4
            x = [0.5 * L * (1.0 - 1e-13)]
            x.append(x[0] + RL * (1.0 - 1e-12) - L)
            for cell, n in ((2, 10), (3, 10), (4, 30), (5, 9)):
                x.extend(((cell + rng.uniform(0.1, 0.9, n)) / 6.0 - 0.5) * L)
            p = np.zeros((len(x), 4))
            p[:, :3] = L * 0.25 / 6.0
            p[:, axis] = flip * np.array(x)
            pos4.append(p)
    rc = np.array([[RC]])
    got = _batch_lists([(L, L, L)] * len(pos4), pos4, rc)
    for r, p in enumerate(pos4):
        assert np.array_equal(got[r], _oracle_pairs((L, L, L), p, rc)), f"replica {r}"
