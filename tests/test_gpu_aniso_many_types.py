"""TwoPatchMorse with parameter tables near the largest: 24 and 27 types, whose
FP64 launches take different amounts of dynamic LDS above 64 KiB, from two
threads at once.  Every launch succeeds and gives the oracle's sums.
"""

import threading

import numpy as np
import pytest

import oracle
from azplugins_amd import _azp
from gpu_util import GpuSystem, gpu_pair, jittered_lattice, rel_err, say

torch = _azp.torch
pytestmark = pytest.mark.gpu


def _case(nt):
    rng = np.random.default_rng(nt)
    pos4, _ = jittered_lattice(9, 10.0, 0.15, nt, seed=nt)
    q = rng.normal(size=(pos4.shape[0], 4))
    q /= np.linalg.norm(q, axis=1)[:, None]
    params = {(a, b): {"M_d": float(rng.uniform(0.5, 1.5)), "M_r": 0.2, "r_eq": 1.0, "omega": 20.0,
                       "alpha": float(rng.uniform(0.2, 0.6)), "repulsion": bool(rng.integers(0, 2))}
              for a in range(nt) for b in range(a, nt)}
    Lv, rc = np.full(3, 10.0), 2.0
    pairs = oracle.nlist(pos4, Lv, nt, oracle.r_listsq_matrix([rc] * nt * nt, 0.3), "cell")
    want = oracle.aniso_forces(pos4, q, Lv, pairs, nt, oracle.pack_matrix(5, params, nt), np.full(nt * nt, rc * rc),
                               "none")
    return pos4, q, Lv, params, rc, want


def test_many_types_from_two_threads():
    cases = {nt: _case(nt) for nt in (24, 27)}
    errors = []

    def work(nt):
        try:
            pos4, q, Lv, params, rc, (fo, to, vo) = cases[nt]
            for _ in range(8):
                with torch.cuda.stream(torch.cuda.Stream()):
                    r = gpu_pair("AnisoPotentialPairTwoPatchMorse", GpuSystem(pos4, Lv, quat=q), nt, params, rc,
                                 r_buff=0.3)
                assert rel_err(r.force, fo) < 1e-12
                assert rel_err(r.torque[:, :3], to[:, :3]) < 1e-12
                assert rel_err(r.virial, vo) < 1e-12
        except Exception as e:  # noqa: BLE001 - reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(nt,)) for nt in cases]
    say("[aniso] 24 and 27 types from two threads")
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors[0]
