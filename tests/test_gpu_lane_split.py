"""Several lanes per particle (csrc/lane_split.h).

Up to 65,536 particles, systems of at most 2^18 / 2^s get 2^s lanes each
(s <= 4); above, the pair term decides about two.  The sizes lie on both sides
of lines of that rule, with lists shorter than one lane's batch, ragged last
tiles and columns without entries.  The split does not depend on the list's
layout, so the plain and the tiled list give the same bits at every size; the
oracle bounds the sums (FP64: a few hundred terms of 2^-53 each, 1e-12; mixed
form: its FP32 terms, 1e-5).
"""

import numpy as np
import pytest

import oracle
from azplugins_amd import _azp
from gpu_util import GpuSystem, gpu_pair, jittered_lattice, rel_err, say

torch = _azp.torch
pytestmark = pytest.mark.gpu

SIZES = [700, 16384, 16385, 50001, 131072, 131073]
YK = {(0, 0): {"epsilon": 1.0, "kappa": 2.0, "delta": 0.2}, (0, 1): {"epsilon": 0.7, "kappa": 1.5, "delta": 0.3},
      (1, 1): {"epsilon": 1.3, "kappa": 2.5, "delta": 0.1}}
TPM = {(0, 0): {"M_d": 1.0, "M_r": 0.2, "r_eq": 1.0, "omega": 20.0, "alpha": 0.4, "repulsion": True}}
DPD = {(0, 0): {"A": 25.0, "gamma": 4.5, "s": 0.5}, (0, 1): {"A": 40.0, "gamma": 4.5, "s": 1.0},
       (1, 1): {"A": 25.0, "gamma": 3.5, "s": 2.0}}


def _slab(N, ntypes, seed):
    """The first N sites of a jittered lattice: a slab with two free faces."""
    n = 51 if N > 1000 else 10
    L = float(n)
    pos4, rng = jittered_lattice(n, L, 0.15, ntypes, seed=seed)
    return pos4[:N], np.array([L, L, L]), rng


@pytest.mark.parametrize("rc", [1.05, 2.2])
@pytest.mark.parametrize("N", SIZES)
def test_pair_sums(N, rc):
    pos4, Lv, _ = _slab(N, 2, seed=N)
    sysm = GpuSystem(pos4, Lv)
    pairs = oracle.nlist(pos4, Lv, 2, oracle.r_listsq_matrix([rc] * 4, 0.3), "cell")
    fo, vo = oracle.pair_forces(oracle.EXPANDED_YUKAWA, pos4, Lv, pairs, 2,
                                oracle.pack_matrix(oracle.EXPANDED_YUKAWA, YK, 2), np.full(4, rc * rc))
    for precision, tol in (("fp64", 1e-12), ("mixed", 1e-5), ("mixed_acc64", 1e-5)):
        plain = gpu_pair("PotentialPairExpandedYukawa", sysm, 2, YK, rc, r_buff=0.3, precision=precision)
        say(f"[split] N={N} rc={rc} {precision}")
        assert rel_err(plain.force, fo) < tol
        assert rel_err(plain.virial, vo) < tol
        for tile in (256, 512):
            tiled = gpu_pair("PotentialPairExpandedYukawa", sysm, 2, YK, rc, r_buff=0.3, precision=precision,
                             tiled=tile)
            assert tiled.nl.get_tiles()[3] == tile
            assert np.array_equal(plain.force, tiled.force)
            assert np.array_equal(plain.virial, tiled.virial)


@pytest.mark.parametrize("N", SIZES)
def test_dpd_sums(N):
    rng = np.random.default_rng(N)
    L = (N / 3.0) ** (1.0 / 3.0)
    Lv = np.array([L, L, L])
    pos4 = np.zeros((N, 4))
    pos4[:, :3] = rng.uniform(-0.5, 0.5, size=(N, 3)) * Lv
    pos4[:, 3] = rng.integers(0, 2, size=N)
    vel4 = np.ones((N, 4))
    vel4[:, :3] = rng.normal(size=(N, 3))
    seed, t, dt, kT = 3, 1000, 0.02, 1.0
    sysm = GpuSystem(pos4, Lv, vel4)
    pairs = oracle.nlist(pos4, Lv, 2, oracle.r_listsq_matrix([1.0] * 4, 0.4), "cell")
    fo, vo = oracle.dpd_forces(pos4, vel4, np.arange(N), Lv, pairs, 2, oracle.pack_matrix(4, DPD, 2), np.ones(4),
                               seed, t, dt, kT)
    plain = gpu_pair("PotentialPairDPDThermoGeneralWeight", sysm, 2, DPD, 1.0, thermostat=(seed, dt, kT), timestep=t)
    say(f"[split] dpd N={N}")
    assert rel_err(plain.force, fo) < 1e-12
    assert rel_err(plain.virial, vo) < 1e-12
    for tile in (256, 512):
        tiled = gpu_pair("PotentialPairDPDThermoGeneralWeight", sysm, 2, DPD, 1.0, thermostat=(seed, dt, kT),
                         timestep=t, tiled=tile)
        assert tiled.nl.get_tiles()[3] == tile
        assert np.array_equal(plain.force, tiled.force)
        assert np.array_equal(plain.virial, tiled.virial)


@pytest.mark.parametrize("N", SIZES)
def test_aniso_sums(N):
    pos4, Lv, rng = _slab(N, 1, seed=N + 1)
    q = rng.normal(size=(N, 4))
    q /= np.linalg.norm(q, axis=1)[:, None]
    rc = 1.7
    sysm = GpuSystem(pos4, Lv, quat=q)
    pairs = oracle.nlist(pos4, Lv, 1, oracle.r_listsq_matrix([rc], 0.3), "cell")
    fo, to, vo = oracle.aniso_forces(pos4, q, Lv, pairs, 1, oracle.pack_matrix(5, TPM, 1), np.array([rc * rc]), "none")
    for precision, tol in (("fp64", 1e-12), ("mixed", 1e-5)):
        say(f"[split] aniso N={N} {precision}")
        r = gpu_pair("AnisoPotentialPairTwoPatchMorse", sysm, 1, TPM, rc, r_buff=0.3, precision=precision)
        assert rel_err(r.force, fo) < tol
        assert rel_err(r.torque[:, :3], to[:, :3]) < tol
        assert rel_err(r.virial, vo) < tol
