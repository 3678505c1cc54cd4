"""Which adjoint contractions of one triple share a launch in the split-BF16x3 walks
(host-only), and the projected adjoint whose triples (l, j, k) come in any order of
l: contractions of one launch run concurrently, so no two of them may write the
same address."""
import ctypes

import numpy as np
import pytest
import torch

from pyscfad_amd import _lib
from pyscfad_amd.cc import _ops
from pyscfad_amd.gen import make_problem
from tests.gemm_emulator import GemmDesc, _decomp


def _launches(o, v, i, j, k):
    f = _lib.load().pamd_debug_adjoint_launches
    f.argtypes = [ctypes.c_int] * 5 + [ctypes.c_void_p] * 3 + [ctypes.c_int] + \
        [ctypes.POINTER(ctypes.c_int)] * 2
    bases = (ctypes.c_ulonglong * 10)(*[(n + 1) << 40 for n in range(10)])
    buf, at, n, nb = (GemmDesc * 64)(), (ctypes.c_int * 64)(), ctypes.c_int(), ctypes.c_int()
    assert f(o, v, i, j, k, bases, buf, at, 64, ctypes.byref(n), ctypes.byref(nb)) == 0
    assert nb.value == ctypes.sizeof(GemmDesc)
    return [(at[q], buf[q]) for q in range(n.value)]


def _written(d):
    if d.mode >= 2:   # split-K parts (of 8 bytes at most)
        return int(d.partial) + 8 * np.arange(d.splits * d.M * d.N)
    m, n = np.arange(d.M), np.arange(d.N)
    return (int(d.C.p) + 8 * (_decomp(m, d.C.mdiv, d.C.mx, d.C.my)[:, None] +
                              _decomp(n, d.C.ndiv, d.C.nx, d.C.ny)[None, :])).reshape(-1)


@pytest.mark.parametrize('o,v,i,j,k', [(3, 8, 0, 1, 2), (3, 8, 2, 0, 1), (3, 8, 1, 0, 1), (3, 8, 2, 1, 2),
                                       (3, 8, 0, 0, 2), (3, 8, 0, 2, 2), (2, 8, 1, 1, 1), (8, 16, 5, 2, 5)])
def test_contractions_of_a_launch_write_disjoint_addresses(o, v, i, j, k):
    seen = {}
    for launch, d in _launches(o, v, i, j, k):
        seen.setdefault(launch, []).append(_written(d))
    assert sum(len(w) for w in seen.values()) == 18
    for launch, w in seen.items():
        every = np.concatenate(w)
        assert np.unique(every).size == every.size, (launch, len(w))


def test_distinct_triples_still_share_launches():
    """Particle t2 and hole ovoo parts always, the two families of three slabs when the
    occupied indices differ."""
    count = lambda *t: len({q for q, _ in _launches(3, 8, *t)})  # noqa: E731
    assert count(0, 1, 2) == count(2, 0, 1) == 4
    assert count(1, 0, 1) == count(0, 0, 2) == 8


# (v % 8 == 0: the ovvv adjoints run on the direct engine; o % 8 == 0: the hole-term ones too)
@pytest.mark.gpu
@pytest.mark.parametrize('o,v,nfrag', [(3, 16, 1), (5, 24, 2), (8, 16, 2)])
def test_split_projected_adjoint_matches_fp64(o, v, nfrag, cuda):
    """The split form's bound on every cotangent block is 1e-6 of its norm."""
    p = make_problem(o, v, 3 * v, seed=o + v, fvo_scale=1e-3)
    u = np.random.default_rng(3).normal(size=(nfrag, o))
    out = [_ops.projected_energy_vjp(_ops.Inputs(p.mo_energy, p.t1, p.t2, p.ovvv_packed(), p.ovoo, p.ovov, p.fvo,
                                                 precision=prec, device=cuda), u, et_bar=0.7)
           for prec in ('fp64', 'bf16x3')]
    (e0, g0), (e1, g1) = out
    assert abs(float(e1 - e0)) <= 1e-9
    for k in g0:
        assert float(torch.linalg.norm(g1[k] - g0[k])) <= 1e-6 * float(torch.linalg.norm(g0[k])), k
