"""Split-BF16x3 calls around the sizes (nvir <= 16) whose products leave the direct
engine for the register-staged one, against FP64: nvir and nocc at, below and above
multiples of 8."""
import pytest
import torch

from pyscfad_amd.cc import _ops
from pyscfad_amd.gen import make_problem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('o,v,fvo', [(2, 2, 0.0), (3, 7, 1e-3), (2, 8, 0.0), (8, 8, 1e-3), (3, 9, 1e-3),
                                     (8, 16, 0.0), (5, 16, 1e-3), (4, 17, 1e-3), (8, 24, 0.0)])
def test_small_split_gradient_matches_fp64(o, v, fvo, cuda):
    """1e-9 Eh in E(T) and 1e-6 of each block's norm, the split form's bounds."""
    p = make_problem(o, v, 3 * v, seed=o * 10 + v, fvo_scale=fvo)
    e, g = {}, {}
    for prec in ('fp64', 'bf16x3'):
        inp = _ops.Inputs(p.mo_energy, p.t1, p.t2, p.ovvv_packed(), p.ovoo, p.ovov, p.fvo, precision=prec,
                          device=cuda)
        e[prec], g[prec] = _ops.energy_vjp(inp, et_bar=0.7)
        assert abs(float(_ops.energy(inp) - e['fp64'])) <= 1e-9
    assert abs(float(e['bf16x3'] - e['fp64'])) <= 1e-9
    for k, ref in g['fp64'].items():
        assert float(torch.linalg.norm(g['bf16x3'][k] - ref)) <= 1e-6 * float(torch.linalg.norm(ref)), k
