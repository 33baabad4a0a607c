"""Edges of the tiled list built from matrix-core group walks.

Two to eight types with unequal radii (the type pairs' radii as a one-hot
contraction), nine (left to the plain walk), boxes from two to nine cells an
axis (reach of the group's span), and clusters in a wide box (whose tiles span
too many cells: left to the plain walk).  Each list must equal the plain
walk's, and the plain walk's pairs the oracle's.
"""

import numpy as np
import pytest

import oracle
from azplugins_amd import _azp
from azplugins_amd import _azplugins
from gpu_util import GpuSystem, jittered_lattice, nlist_pairs, say

torch = _azp.torch
pytestmark = pytest.mark.gpu


def _lists(sysm, nt, rc, tiled, r_buff=0.4):
    nl = _azplugins.NeighborListGPU(r_buff)
    nl.set_r_cut(nt, [float(x) for x in rc])
    if tiled:
        nl.set_tiled(True)
    nl.update(sysm.particles())
    torch.cuda.synchronize()
    return nl


def _check(pos4, Lv, nt, rc, kind=1):
    sysm = GpuSystem(pos4, Lv)
    plain, tiled = _lists(sysm, nt, rc, False), _lists(sysm, nt, rc, True)
    size = tiled.get_tiles()[3]
    say(f"[edges] N={sysm.N} types={nt} L={Lv[0]:.1f}: tile size {size}, walk {tiled.walk_kind()}")
    assert plain.walk_kind() == 0 and tiled.walk_kind() == kind
    assert size in (256, 512)
    got = nlist_pairs(tiled, sysm.N)
    assert got == nlist_pairs(plain, sysm.N)
    pairs = oracle.nlist(pos4, Lv, nt, oracle.r_listsq_matrix(rc, 0.4), "cell")
    assert got == set(zip(pairs[0].tolist(), pairs[1].tolist()))


@pytest.mark.parametrize("nt", [2, 3, 8, 9])
def test_unequal_radii(nt):
    pos4, rng = jittered_lattice(15, 16.0, 0.2, nt, seed=nt)
    rc = rng.uniform(0.8, 2.6, size=(nt, nt))
    rc = np.maximum(rc, rc.T)
    _check(pos4, np.full(3, 16.0), nt, rc.ravel(), 1 if nt <= 8 else 0)


@pytest.mark.parametrize("cells", [2, 3, 4, 5, 6, 7, 9])
def test_small_grids(cells):
    L = cells * 1.9 + 0.2
    n = int(L / 1.05)
    pos4, _ = jittered_lattice(n, L, 0.2, 1, seed=cells)
    _check(pos4, np.full(3, L), 1, [1.5])


@pytest.mark.parametrize("per", [40, 120])
def test_dense_clusters(per):
    rng = np.random.default_rng(per)
    L = 24.0
    centres = rng.uniform(-L / 2, L / 2, size=(60, 3))
    p = (centres[:, None, :] + rng.normal(scale=0.45, size=(60, per, 3))).reshape(-1, 3)
    p -= L * np.floor(p / L + 0.5)
    pos4 = np.zeros((p.shape[0], 4))
    pos4[:, :3] = p
    _check(pos4, np.full(3, L), 1, [1.2], kind=0)
