"""Rooms of the per-tile walk: a first build of an ordinary system has enough of
them and runs once; a build that needs more is repeated with more, and its list
equals the plain walk's entry for entry.
"""

import numpy as np
import pytest

from azplugins_amd import _azp
from azplugins_amd import _azplugins
from gpu_util import GpuSystem, say

torch = _azp.torch
pytestmark = pytest.mark.gpu


def _new(r_cut, tiled):
    nl = _azplugins.NeighborListGPU(0.4)
    nl.set_r_cut(1, [r_cut])
    nl.set_tiled(tiled)
    return nl


def _update(nl, sysm):
    nl.update(sysm.particles())
    torch.cuda.synchronize()


def _same_as_plain(nl, sysm, r_cut):
    plain = _new(r_cut, False)
    _update(plain, sysm)
    (nn, lst), (nn0, lst0) = nl.download(sysm.N), plain.download(sysm.N)
    assert np.array_equal(nn, nn0)
    top = int(nn.max())
    mine = np.arange(top)[:, None] < nn[None, :]
    assert np.array_equal(lst[:top, :sysm.N][mine], lst0[:top, :sysm.N][mine])


def _fluid(N, density, seed):
    rng = np.random.default_rng(seed)
    L = (N / density) ** (1.0 / 3.0)
    pos4 = np.zeros((N, 4))
    pos4[:, :3] = (rng.random((N, 3)) - 0.5) * L
    return GpuSystem(pos4, np.full(3, L))


@pytest.mark.parametrize("density, r_cut, N", [(0.85, 3.0, 900), (0.85, 3.0, 1760), (0.85, 3.0, 30011),
                                               (0.5, 4.0, 1500), (0.5, 4.0, 9000), (3.0, 1.0, 900),
                                               (3.0, 1.0, 5000), (3.0, 1.0, 60000)])
def test_first_build_runs_once(density, r_cut, N):
    sysm = _fluid(N, density, N)
    nl = _new(r_cut, 256 if r_cut > 3.5 else 512)
    _update(nl, sysm)
    assert nl.walk_kind() == 1
    assert nl.walk_runs()[0] == 1


def test_rooms_grow():
    """A cluster of 3,800 particles all within reach of each other, alone in
    a box of 9 x 9 x 9 cells: 60 batches a group and 30,720 rank-table entries
    a tile, more than the first rooms have."""
    rng = np.random.default_rng(7)
    r_cut, L = 1.2, 9.1 * 1.6
    ball = rng.normal(size=(3800, 3))
    ball *= (0.75 * rng.random(3800) ** (1.0 / 3.0) / np.linalg.norm(ball, axis=1))[:, None]
    pos4 = np.zeros((3800, 4))
    pos4[:, :3] = ball
    sysm = GpuSystem(pos4, np.full(3, L))
    nl = _new(r_cut, 512)
    _update(nl, sysm)
    rows, compactions = nl.walk_runs()
    say(f"[rooms] rows {rows} compactions {compactions}")
    assert nl.walk_kind() == 1
    assert rows > 1 and compactions > 1
    _same_as_plain(nl, sysm, r_cut)
    nl.update(sysm.particles(), force_rebuild=True)
    torch.cuda.synchronize()
    assert nl.walk_runs() == (rows + 1, compactions + 1)


def test_rows_serve_both_tile_sizes():
    """At less than three particles a cell 512 slots span more than 128 cells: the rows are
    made once and the second size compacts them; later builds go to it at once.
    A list that served a dense system before has fewer rooms for cells and
    grows them."""
    dense, sparse = _fluid(6000, 0.416, 1), _fluid(12000, 1.0, 2)
    nl = _new(1.0, True)
    _update(nl, sparse)
    assert nl.walk_kind() == 1 and nl.get_tiles()[3] == 256
    assert nl.walk_runs() == (1, 2)
    _same_as_plain(nl, sparse, 1.0)
    for n in range(1, 12):
        nl.update(sparse.particles(), force_rebuild=True)
        assert nl.walk_kind() == 1 and nl.walk_runs() == (1 + n, 2 + n)
    nl = _new(5.5, True)
    _update(nl, dense)
    assert nl.walk_kind() == 1
    rows = nl.walk_runs()[0]
    nl.set_r_cut(1, [1.0])
    _update(nl, sparse)
    assert nl.walk_kind() == 1 and nl.walk_runs()[0] == rows + 2
    _same_as_plain(nl, sparse, 1.0)


def test_sparse_cells_leave_the_walk_alone():
    """Below two particles a cell no tile size fits: found before the rows, once."""
    sysm = _fluid(20000, 0.5, 3)
    nl = _new(1.0, True)
    for n in range(12):
        nl.update(sysm.particles(), force_rebuild=True)
        assert nl.walk_kind() == 0 and nl.walk_runs() == (1, 1)
    _same_as_plain(nl, sysm, 1.0)
