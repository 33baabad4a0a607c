"""Small dense boxes keep the per-tile walk.

On grids of three or four cells an axis a group of 64 particles is served in
two or three passes that each read nearly the whole box, so at 50 to 100
particles a cell it needs 65 to about 110 batches of 64 candidates.  Its tiles'
rank tables hold 272 a group: the walk serves these systems, and its lists
equal the plain walk's.
"""

import numpy as np
import pytest

from azplugins_amd import _azp
from azplugins_amd import _azplugins
from gpu_util import GpuSystem, say

torch = _azp.torch
pytestmark = pytest.mark.gpu


def _list(sysm, r_cut, tiled):
    nl = _azplugins.NeighborListGPU(0.4)
    nl.set_r_cut(1, [r_cut])
    nl.set_tiled(tiled)
    nl.update(sysm.particles())
    torch.cuda.synchronize()
    return nl


def _lattice(density, N):
    rng = np.random.default_rng(N)
    k = int(np.ceil(N ** (1.0 / 3.0) - 1e-9))
    L = (k**3 / density) ** (1.0 / 3.0)
    g = (np.arange(k) + 0.5) * (L / k) - 0.5 * L
    sites = np.stack(np.meshgrid(g, g, g, indexing="ij"), -1).reshape(-1, 3)
    pos4 = np.zeros((N, 4))
    pos4[:, :3] = sites[rng.permutation(k**3)[:N]] + rng.uniform(-0.1, 0.1, (N, 3))
    pos4[:, :3] -= L * np.floor(pos4[:, :3] / L + 0.5)
    return GpuSystem(pos4, np.full(3, L)), L


def _same(walk, plain, N):
    (nn, lst), (nn0, lst0) = walk.download(N), plain.download(N)
    assert np.array_equal(nn, nn0)
    top = int(nn.max())
    mine = np.arange(top)[:, None] < nn[None, :N]
    assert np.array_equal(lst[:top, :N][mine], lst0[:top, :N][mine])


@pytest.mark.parametrize("tile", [True, 256])
@pytest.mark.parametrize("density, r_cut, N", [(0.85, 3.0, 1350), (0.85, 3.0, 1650), (0.85, 3.0, 3750),
                                               (0.5, 4.0, 1760), (0.5, 4.0, 4800), (0.5, 4.0, 6100),
                                               (0.416, 5.5, 1400), (0.416, 5.5, 2900), (0.416, 5.5, 6144)])
def test_small_dense_boxes(density, r_cut, N, tile):
    sysm, L = _lattice(density, N)
    walk, plain = _list(sysm, r_cut, tile), _list(sysm, r_cut, False)
    say(f"[dense] N={N} cells an axis {int(L / (r_cut + 0.4))}")
    assert plain.walk_kind() == 0 and walk.walk_kind() == 1
    assert walk.get_tiles()[3] in ((256,) if tile == 256 else (256, 512))
    _same(walk, plain, N)


@pytest.mark.parametrize("density, r_cut, N", [(0.5, 4.0, 50000), (0.5, 4.0, 100000), (0.5, 4.0, 160000)])
def test_candidates_of_wide_tiles(density, r_cut, N):
    """512-column tiles of 6,145 to 6,656 candidates."""
    sysm, _ = _lattice(density, N)
    walk, plain = _list(sysm, r_cut, True), _list(sysm, r_cut, False)
    assert walk.walk_kind() == 1 and walk.get_tiles()[3] == 512
    _same(walk, plain, N)
