"""The batched FP64 walk against the one-triple walk, which a call falls back to
when its workspace holds no batch: the smallest workspace the entry point takes
against the one pamd_ccsdt_workspace_size asks for.  Sizes at the edges of the
padding (v = 8 n, 8 n +- 1), of a run of 8 triples and of the tiles (16, 48, 80);
each sum is the same terms in another order, so the blocks agree to a few times
the rounding of sums of at most o^2 v^2 terms (1e-12 relative)."""
import ctypes

import pytest
import torch

from pyscfad_amd import _lib
from pyscfad_amd.cc import _ops
from pyscfad_amd.gen import make_problem

pytestmark = pytest.mark.gpu


def _least(call, full):
    """The least byte count (a multiple of 256) that ``call(nbytes)`` accepts."""
    lo, hi = 0, full
    while hi - lo > 256:
        mid = (lo + hi) // 512 * 256
        if call(mid) == _lib.PAMD_OK:
            hi = mid
        else:
            lo = mid
    return hi


def _smallest_workspace(inp):
    lib = _lib.load()
    full = _lib.workspace_size(inp.cfg, True)
    ws = torch.empty(full, dtype=torch.uint8, device=inp.device)
    out = _ops._cotangent_outputs(inp)
    e = torch.zeros((), dtype=torch.float64, device=inp.device)

    def call(n):
        return lib.pamd_ccsdt_energy_vjp(ctypes.byref(inp.cfg), *inp.args(), ctypes.c_double(0.7),
                                         _ops._ptr(ws), n, _ops._ptr(e), *_ops._cotangent_ptrs(out),
                                         _ops._stream(inp.device))

    return ws, _least(call, full)


@pytest.mark.parametrize('o,v,fvo,packed', [(2, 7, 1e-3, True), (3, 9, 0.0, False), (4, 16, 1e-3, True),
                                            (5, 47, 1e-3, False), (3, 81, 0.0, True),
                                            (6, 49, 1e-3, True), (1, 12, 1e-3, False), (2, 33, 1e-3, True),
                                            (2, 131, 1e-3, True), (2, 263, 0.0, True)])
def test_batched_walk_matches_the_one_triple_walk(o, v, fvo, packed, cuda):
    p = make_problem(o, v, 3 * v, seed=o * 100 + v, fvo_scale=fvo)
    inp = _ops.Inputs(p.mo_energy, p.t1, p.t2, p.ovvv_packed() if packed else p.ovvv, p.ovoo, p.ovov,
                      p.fvo, device=cuda)
    e, g = _ops.energy_vjp(inp, et_bar=0.7)
    ws, least = _smallest_workspace(inp)
    e1, g1 = _ops.energy_vjp(inp, et_bar=0.7, workspace=(ws, least))
    assert torch.allclose(e, e1, rtol=1e-12, atol=1e-18)
    for k in g:
        ref = float(g1[k].norm())
        assert float((g[k] - g1[k]).norm()) <= 1e-12 * ref + 1e-18, k
    assert torch.allclose(_ops.energy(inp), e1, rtol=1e-12, atol=1e-18)


@pytest.mark.parametrize('o,v,nfrag,fvo', [(2, 9, 1, 1e-3), (5, 31, 2, 0.0), (3, 48, 3, 1e-3),
                                           (4, 17, 8, 1e-3), (17, 8, 2, 0.0)])
def test_batched_projected_walk_matches_the_one_triple_walk(o, v, nfrag, fvo, cuda):
    p = make_problem(o, v, 3 * v, seed=o * 10 + v, fvo_scale=fvo)
    inp = _ops.Inputs(p.mo_energy, p.t1, p.t2, p.ovvv_packed(), p.ovoo, p.ovov, p.fvo, device=cuda)
    u = torch.randn((nfrag, o), generator=torch.Generator().manual_seed(o), dtype=torch.float64)
    e, g = _ops.projected_energy_vjp(inp, u, et_bar=0.7)
    lib = _lib.load()
    un = u.numpy()
    ws, full = _ops._projected_ws(inp, nfrag, True)
    out = _ops._cotangent_outputs(inp)
    out['ulo_bar'] = torch.empty((nfrag, o), dtype=torch.float64, device=cuda)
    e1 = torch.zeros((), dtype=torch.float64, device=cuda)

    def call(n):
        return lib.pamd_ccsdt_projected_energy_vjp(
            ctypes.byref(inp.cfg), *inp.args(), un.ctypes.data_as(ctypes.c_void_p), nfrag,
            ctypes.c_double(0.7), _ops._ptr(ws), n, _ops._ptr(e1), *_ops._cotangent_ptrs(out),
            _ops._ptr(out['ulo_bar']), _ops._stream(inp.device))

    assert call(_least(call, full)) == _lib.PAMD_OK
    torch.cuda.synchronize()
    assert torch.allclose(e, e1, rtol=1e-12, atol=1e-18)
    for k in out:
        assert float((g[k] - out[k]).norm()) <= 1e-12 * float(out[k].norm()) + 1e-18, k
    assert torch.allclose(_ops.projected_energy(inp, u), e1, rtol=1e-12, atol=1e-18)


# (v < 24: the 32x32-MFMA tiles, which sum in FP64; o = 6, 12 with v a multiple of
# 8; one virtual below and above a multiple; nothing but padding changes at (8, 40);
# v = 239: the direct engine's 240-wide tiles against the register-staged engine)
@pytest.mark.parametrize('o,v,fvo,packed', [(2, 7, 1e-3, True), (3, 17, 0.0, False), (6, 48, 1e-3, True),
                                            (12, 40, 0.0, False), (8, 40, 1e-3, True), (5, 63, 1e-3, False),
                                            (9, 81, 0.0, True), (1, 24, 1e-3, True), (3, 239, 0.0, True)])
def test_padded_walk_matches_the_unpadded_one(o, v, fvo, packed, cuda):
    """The split-BF16x3 walk on operands padded to multiples of 8 against the same walk
    on unpadded ones, which a call falls back to when its workspace does not hold
    the padded arrays: the smallest workspace the entry point takes against the one
    pamd_ccsdt_workspace_size asks for.  Padding keeps every FP32 sum (the same
    products in the same order), so gradients differ by FP64 roundings (1e-12
    relative) and by the few elements of Wbar whose last bf16 piece rounds the other
    way: 2^-24 of one term of a sum each, below 1e-9 of a block's norm."""
    p = make_problem(o, v, 3 * v, seed=o * 100 + v, fvo_scale=fvo)
    inp = _ops.Inputs(p.mo_energy, p.t1, p.t2, p.ovvv_packed() if packed else p.ovvv, p.ovoo, p.ovov,
                      p.fvo, precision='bf16x3', device=cuda)
    e, g = _ops.energy_vjp(inp, et_bar=0.7)
    ws, least = _smallest_workspace(inp)
    assert least < ws.numel()
    e1, g1 = _ops.energy_vjp(inp, et_bar=0.7, workspace=(ws, least))
    assert torch.allclose(e, e1, rtol=1e-12, atol=1e-18)
    for k in g:
        assert float((g[k] - g1[k]).norm()) <= 1e-9 * float(g1[k].norm()) + 1e-18, k
    assert torch.allclose(_ops.energy(inp), e1, rtol=1e-12, atol=1e-18)
