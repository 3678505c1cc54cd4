"""The FP64 walks against each other, each forced: batches of many triples, one triple
at a time, and that on one stream or two.  (With the least workspace an entry point
takes, a batch of 8 is often still there, so the workspace alone does not say which
walk runs; pamd_debug_walk_batch does.)"""
import ctypes

import pytest
import torch

from pyscfad_amd import _lib
from pyscfad_amd.cc import _ops
from pyscfad_amd.gen import make_problem


def _batch(o, v, nbytes, nfrag=0, vjp=True):
    n = ctypes.c_int(-1)
    assert _lib.load().pamd_debug_walk_batch(o, v, nfrag, int(vjp), nbytes, ctypes.byref(n)) == _lib.PAMD_OK
    return n.value


def _triples(o):
    return o * (o + 1) * (o + 2) // 6 - o


# (with the preferred workspace, with the needed one)
@pytest.mark.parametrize('o,v,batches', [(5, 47, (8, 8)), (6, 49, (8, 8)), (7, 64, (32, 16)), (4, 16, (16, 0)),
                                         (12, 100, (176, 8)), (40, 400, (16, 0))])
def test_walk_batch_by_workspace(o, v, batches):
    cfg = _lib.make_config(o, v)
    assert tuple(_batch(o, v, _lib.workspace_size(cfg, True, least=q)) for q in (False, True)) == batches


def _inputs(o, v, fvo, packed, cuda):
    p = make_problem(o, v, 3 * v, seed=o * 100 + v, fvo_scale=fvo)
    return _ops.Inputs(p.mo_energy, p.t1, p.t2, p.ovvv_packed() if packed else p.ovvv, p.ovoo, p.ovov, p.fvo,
                       device=cuda)


def _one_triple(inp, two_streams):
    n = _lib.workspace_size(inp.cfg, True, least=True)
    ws = torch.empty(n, dtype=torch.uint8, device=inp.device)
    out = _ops._cotangent_outputs(inp)
    e = torch.zeros((), dtype=torch.float64, device=inp.device)
    st = _lib.load().pamd_debug_one_triple_vjp(
        ctypes.byref(inp.cfg), *inp.args(), ctypes.c_double(0.7), int(two_streams), _ops._ptr(ws), n, _ops._ptr(e),
        *_ops._cotangent_ptrs(out), _ops._stream(inp.device))
    assert st == _lib.PAMD_OK
    torch.cuda.synchronize()
    return e, out


def _same(e, g, e1, g1):
    """Sums of the same terms, at most o^2 v^2 of them, in another order."""
    assert torch.allclose(e, e1, rtol=1e-12, atol=1e-18)
    for k, ref in g1.items():
        assert float((g[k] - ref).norm()) <= 1e-12 * float(ref.norm()) + 1e-18, k


# (o >= 5: several batches at either workspace)
@pytest.mark.gpu
@pytest.mark.parametrize('o,v,fvo,packed', [(5, 47, 1e-3, False), (6, 49, 1e-3, True), (3, 81, 0.0, True),
                                            (7, 64, 0.0, True), (4, 16, 1e-3, True), (2, 7, 0.0, False)])
def test_batches_match_one_triple_at_a_time(o, v, fvo, packed, cuda):
    inp = _inputs(o, v, fvo, packed, cuda)
    e1, g1 = _one_triple(inp, False)
    for least in (False, True):
        n = _lib.workspace_size(inp.cfg, True, least=least)
        nb = _batch(o, v, n)
        print(f'o{o} v{v}: {_triples(o)} triples, batches of {nb}', flush=True)
        ws = torch.empty(n, dtype=torch.uint8, device=cuda)
        _same(*_ops.energy_vjp(inp, et_bar=0.7, workspace=(ws, n)), e1, g1)
        if o >= 5:
            assert 0 < nb < _triples(o)


@pytest.mark.gpu
@pytest.mark.parametrize('o,v,fvo', [(8, 40, 1e-3), (5, 24, 0.0), (3, 9, 1e-3)])
def test_two_streams_match_one_in_fp64(o, v, fvo, cuda):
    """Every sum is written by one stream in walk order: the same bits."""
    inp = _inputs(o, v, fvo, True, cuda)
    (e, g), (e1, g1) = _one_triple(inp, True), _one_triple(inp, False)
    assert torch.equal(e, e1)
    for k in g:
        assert torch.equal(g[k], g1[k]), k


@pytest.mark.gpu
@pytest.mark.parametrize('o,v,nfrag,fvo', [(3, 48, 3, 1e-3), (5, 31, 2, 0.0), (4, 17, 8, 1e-3), (9, 24, 1, 1e-3)])
def test_projected_batches_match_one_triple_at_a_time(o, v, nfrag, fvo, cuda):
    inp = _inputs(o, v, fvo, True, cuda)
    u = torch.randn((nfrag, o), generator=torch.Generator().manual_seed(o), dtype=torch.float64)
    ws, n = _ops._projected_ws(inp, nfrag, True)
    assert _batch(o, v, n, nfrag) >= o
    out = _ops._cotangent_outputs(inp)
    out['ulo_bar'] = torch.empty((nfrag, o), dtype=torch.float64, device=cuda)
    e1 = torch.zeros((), dtype=torch.float64, device=cuda)
    un = u.numpy()
    st = _lib.load().pamd_debug_one_triple_projected_vjp(
        ctypes.byref(inp.cfg), *inp.args(), un.ctypes.data_as(ctypes.c_void_p), nfrag, ctypes.c_double(0.7),
        _ops._ptr(ws), n, _ops._ptr(e1), *_ops._cotangent_ptrs(out), _ops._ptr(out['ulo_bar']),
        _ops._stream(inp.device))
    assert st == _lib.PAMD_OK
    torch.cuda.synchronize()
    _same(*_ops.projected_energy_vjp(inp, u, et_bar=0.7), e1, out)
