"""Both sides of the lines at which a particle gets more lanes (csrc/lane_split.h)
above the sizes of test_gpu_lane_split.py, with several types and every shift
mode, over the plain, the tiled (256 and 512) and the head list: the same bits
in every layout, and the oracle's sums (FP64: a few dozen terms of 2^-53 each,
1e-12; mixed form: its FP32 terms, 1e-5).
"""

import ctypes

import numpy as np
import pytest

import oracle
from azplugins_amd import _azp
from gpu_util import GpuSystem, gpu_pair, jittered_lattice, raw_args, rel_err, say

torch = _azp.torch
pytestmark = pytest.mark.gpu

PARAMS = {
    1: {(0, 0): {"epsilon": 1.0, "kappa": 2.0, "delta": 0.2}, (0, 1): {"epsilon": 0.7, "kappa": 1.5, "delta": 0.3},
        (1, 1): {"epsilon": 1.3, "kappa": 2.5, "delta": 0.1}},
    0: {(0, 0): {"epsilon": 1.0}, (0, 1): {"epsilon": 1.5}, (1, 1): {"epsilon": 2.0}},
    3: {(0, 0): {"A": 144.0, "a_1": 0.0, "a_2": 0.0, "sigma": 1.0},
        (0, 1): {"A": 100.0, "a_1": 0.0, "a_2": 0.5, "sigma": 1.0},
        (1, 1): {"A": 40.0, "a_1": 0.5, "a_2": 0.5, "sigma": 1.0}},
}
MODES = {"none": 0, "shift": 1, "xplor": 2}
CLASSES = {0: "PotentialPairHertz", 1: "PotentialPairExpandedYukawa", 3: "PotentialPairColloid"}
TPM = {(0, 0): {"M_d": 1.0, "M_r": 0.2, "r_eq": 1.0, "omega": 20.0, "alpha": 0.4, "repulsion": True}}


def _slab(N, spacing, ntypes):
    """The first N sites of a jittered 65 x 65 x 65 lattice: a slab with two free faces."""
    L = 65.0 * spacing
    pos4, rng = jittered_lattice(65, L, 0.15 * spacing, ntypes, seed=N)
    return np.ascontiguousarray(pos4[:N]), np.full(3, L), rng


def _head_force(sysm, ref, ev, nt, rc, ro, mode, precision, pitch):
    """The head-list launch over the column list's entries, rows end to end."""
    nn, lst = ref.nl.download(sysm.N)
    top = int(nn.max())
    mine = (np.arange(top)[:, None] < nn[None, :]).T
    flat = np.concatenate([lst[:top, :sysm.N].T[mine], np.zeros(1, dtype=np.uint32)])
    d_flat = torch.tensor(flat.astype(np.int64).astype(np.int32), device="cuda")
    d_head = torch.tensor(np.concatenate([[0], np.cumsum(nn.astype(np.int64))[:-1]]), device="cuda")
    keys = {0: ("epsilon",), 1: ("epsilon", "kappa", "delta"), 3: ("A", "a_1", "a_2", "sigma")}[ev]
    size = _azp.lib().azp_param_size(ev)
    pods = []
    for a in range(nt):
        for b in range(nt):
            pod = (ctypes.c_char * size)()
            v = PARAMS[ev][(min(a, b), max(a, b))]
            _azp.call("azp_param_pack", ev, _azp.dbl_array([float(v[k]) for k in keys]), pod)
            pods.append(np.frombuffer(bytes(pod), dtype=np.uint8).copy())
    d_params = torch.tensor(np.concatenate(pods), device="cuda")
    rcsq = torch.full((nt * nt,), rc * rc, dtype=torch.float64, device="cuda")
    ronsq = torch.full((nt * nt,), ro * ro, dtype=torch.float64, device="cuda")
    vp = (sysm.N + 63) // 64 * 64
    f = torch.full((sysm.N, 4), np.nan, dtype=torch.float64, device="cuda")
    v = torch.full((6, vp), np.nan, dtype=torch.float64, device="cuda")
    a = raw_args(sysm, ref.nl, rcsq, ronsq, nt, f, v, vp, mode=MODES[mode], precision=_azp.PRECISIONS[precision])
    a.d_nlist, a.d_head_list, a.nlist_pitch = d_flat.data_ptr(), d_head.data_ptr(), pitch
    _azp.call("azp_gpu_compute_pair_forces", ctypes.byref(a), ev, _azp.dptr(d_params))
    torch.cuda.synchronize()
    return f.cpu().numpy(), v[:, :sysm.N].cpu().numpy()


def _check(N, ev, spacing, rc, mode, precisions):
    nt = 2
    ro = 0.9 * rc if mode == "xplor" else 0.0
    pos4, Lv, _ = _slab(N, spacing, nt)
    sysm = GpuSystem(pos4, Lv)
    pairs = oracle.nlist(pos4, Lv, nt, oracle.r_listsq_matrix([rc] * 4, 0.2), "cell")
    fo, vo = oracle.pair_forces(ev, pos4, Lv, pairs, nt, oracle.pack_matrix(ev, PARAMS[ev], nt), np.full(4, rc * rc),
                                np.full(4, ro * ro), mode)
    for precision in precisions:
        kw = dict(r_buff=0.2, mode=mode, precision=precision, r_on=ro)
        plain = gpu_pair(CLASSES[ev], sysm, nt, PARAMS[ev], rc, **kw)
        say(f"[lines] evaluator {ev} N={N} {mode} {precision}")
        tol = 1e-12 if precision == "fp64" else 1e-5
        assert rel_err(plain.force, fo) < tol
        assert rel_err(plain.virial, vo) < tol
        for tile in (256, 512):
            tiled = gpu_pair(CLASSES[ev], sysm, nt, PARAMS[ev], rc, tiled=tile, **kw)
            assert tiled.nl.get_tiles()[3] == tile
            assert np.array_equal(plain.force, tiled.force)
            assert np.array_equal(plain.virial, tiled.virial)
        f, v = _head_force(sysm, plain, ev, nt, rc, ro, mode, precision, 0)
        assert np.array_equal(plain.force, f)
        assert np.array_equal(plain.virial, v)


@pytest.mark.parametrize("mode", ["none", "shift", "xplor"])
@pytest.mark.parametrize("N", [65536, 65537, 131073, 196608, 196609, 262145])
def test_pair_lines(N, mode):
    _check(N, 1, 1.0, 1.15, mode, ("fp64", "mixed", "mixed_acc64"))


@pytest.mark.parametrize("N", [32768, 32769, 65536, 65537])
def test_short_list_lines(N):
    _check(N, 0, 1.0, 1.15, "shift", ("fp64", "mixed"))


@pytest.mark.parametrize("N", [131072, 131073, 262144, 262145])
def test_colloid_lines(N):
    _check(N, 3, 2.0, 2.3, "shift", ("fp64",))


@pytest.mark.parametrize("N", [65537, 98304, 98305, 131073, 163841, 262145])
def test_aniso_lines(N):
    pos4, Lv, rng = _slab(N, 1.0, 1)
    q = rng.normal(size=(N, 4))
    q /= np.linalg.norm(q, axis=1)[:, None]
    rc = 1.15
    sysm = GpuSystem(pos4, Lv, quat=q)
    pairs = oracle.nlist(pos4, Lv, 1, oracle.r_listsq_matrix([rc], 0.2), "cell")
    fo, to, vo = oracle.aniso_forces(pos4, q, Lv, pairs, 1, oracle.pack_matrix(5, TPM, 1), np.array([rc * rc]), "none")
    for precision, tol in (("fp64", 1e-12), ("mixed", 1e-5)):
        say(f"[lines] aniso N={N} {precision}")
        r = gpu_pair("AnisoPotentialPairTwoPatchMorse", sysm, 1, TPM, rc, r_buff=0.2, precision=precision)
        assert rel_err(r.force, fo) < tol
        assert rel_err(r.torque[:, :3], to[:, :3]) < tol
        assert rel_err(r.virial, vo) < tol


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_head_list_pitch_is_not_read(precision):
    """The head-list launch gives the same bits whatever nlist_pitch holds."""
    pos4, Lv, _ = _slab(4097, 1.0, 2)
    sysm = GpuSystem(pos4, Lv)
    ref = gpu_pair(CLASSES[1], sysm, 2, PARAMS[1], 2.2, r_buff=0.2, precision=precision, r_on=0.0)
    for pitch in (0, 1, 0xffffffff):
        f, v = _head_force(sysm, ref, 1, 2, 2.2, 0.0, "none", precision, pitch)
        assert np.array_equal(ref.force, f)
        assert np.array_equal(ref.virial, v)
