"""Device workspaces: what a call needs against what it uses when that is there.

The needed sizes are those of one occupied triple (a pair's, in the projected walk)
at a time, and must not grow with the batches that a larger workspace allows; where
the device does not hold the preferred size the calls run with less."""
import ctypes

import numpy as np
import pytest
import torch

from pyscfad_amd import _lib
from pyscfad_amd.cc import _ops, df
from pyscfad_amd.gen import make_problem


# (energy, energy + VJP) bytes of one triple at a time
@pytest.mark.parametrize('o,v,precision,fwd,vjp', [(16, 160, 'fp64', 883479040, 1752310272),
                                                   (6, 400, 'fp64', 3723118336, 8353746688),
                                                   (40, 400, 'fp64', 27341497600, 51549441280),
                                                   (6, 400, 'bf16x3', 3769198336, 9423826688),
                                                   (2, 7, 'fp64', 26112, 157696)])
def test_needed_workspace_is_one_triples(o, v, precision, fwd, vjp):
    cfg = _lib.make_config(o, v, precision=precision)
    assert [_lib.workspace_size(cfg, w, least=True) for w in (False, True)] == [fwd, vjp]
    for w, n in ((False, fwd), (True, vjp)):
        assert _lib.workspace_size(cfg, w) >= n


# (nvir = 100 and 112: where eight blocks of v^3 pass the library's 128 MiB, with and
# without an adjoint)
@pytest.mark.parametrize('v', [1, 40, 99, 100, 112, 300])
def test_one_occupied_orbital_has_workspace_sizes(v):
    cfg = _lib.make_config(1, v)
    for w in (False, True):
        assert 0 < _lib.workspace_size(cfg, w, least=True) <= _lib.workspace_size(cfg, w)


@pytest.mark.gpu
@pytest.mark.parametrize('v', [40, 112])
def test_one_occupied_orbital_gives_zeros(v, cuda):
    """There is no triple: E(T) and every cotangent are zero."""
    p = make_problem(1, v, 2 * v, seed=v, fvo_scale=1e-3)
    inp = _ops.Inputs(p.mo_energy, p.t1, p.t2, p.ovvv_packed(), p.ovoo, p.ovov, p.fvo, device=cuda)
    assert float(_ops.energy(inp)) == 0.0
    e, g = _ops.energy_vjp(inp, et_bar=0.7)
    assert float(e) == 0.0
    for k, x in g.items():
        assert not bool(x.any()), k


def _projected(cfg, nfrag, name):
    n = ctypes.c_size_t(0)
    assert getattr(_lib.load(), name)(ctypes.byref(cfg), nfrag, 1, ctypes.byref(n)) == _lib.PAMD_OK
    return n.value


def test_needed_projected_workspace_is_one_triples():
    cfg = _lib.make_config(12, 96)
    assert _projected(cfg, 4, 'pamd_ccsdt_projected_workspace_size') == 429056000
    assert _projected(cfg, 4, 'pamd_ccsdt_projected_preferred_workspace_size') > 429056000


def _walk_bytes(o, v, vjp, limit, nfrag=0):
    n = ctypes.c_size_t(0)
    assert _lib.load().pamd_debug_walk_bytes(o, v, nfrag, vjp, limit, ctypes.byref(n)) == _lib.PAMD_OK
    return n.value


# (batches are cut to equal sizes, and a smaller batch can take more parts of an adjoint:
# o13/v47 at 537679616 bytes, o15/v24 at 97909504)
@pytest.mark.parametrize('o', [2, 5, 8, 13, 15, 17, 24, 33, 61, 100])
def test_batches_stay_within_any_workspace(o):
    lib = _lib.load()
    for v in list(range(2, 60)) + [64, 72, 77, 96, 120, 160]:
        for vjp in (0, 1):
            top = _walk_bytes(o, v, vjp, 1 << 62)
            limits = [lib.pamd_ccsdt_noalloc_scratch_bytes(), 537679616, 97909504, top // 2, top // 4]
            for _ in range(20):   # every layout the rule can end at: just what the next smaller one takes
                limits.append(top)
                top = _walk_bytes(o, v, vjp, max(top - 1, 1))
            for n in limits:
                assert _walk_bytes(o, v, vjp, n) <= n, (v, vjp, n)
                if o <= 17 and v % 8 == 0:
                    assert _walk_bytes(o, v, vjp, n, nfrag=2) <= n, (v, vjp, n)


def test_noalloc_size_says_which_problems_fit():
    lib = _lib.load()
    n = ctypes.c_size_t(0)
    for o, v, fits in ((10, 64, True), (8, 56, True), (16, 64, False), (11, 77, False)):
        cfg = _lib.make_config(o, v)
        assert lib.pamd_ccsdt_noalloc_workspace_size(ctypes.byref(cfg), ctypes.byref(n)) == _lib.PAMD_OK
        assert (n.value <= lib.pamd_ccsdt_noalloc_scratch_bytes()) == fits, (o, v)


def test_scratch_takes_what_fits(monkeypatch):
    asked, real = [], torch.empty

    def empty(n, **kw):
        asked.append(n)
        if n > 1000:
            raise torch.OutOfMemoryError('no')
        return real(n, **kw)

    monkeypatch.setattr(torch, 'empty', empty)
    ws, n = _ops._scratch(8192, lambda: 700, 'cpu', 'test')
    assert (ws.numel(), n) == (700, 700) and asked == [8192, 4096, 2048, 1024, 700]
    assert _ops._scratch(512, lambda: 700, 'cpu', 'test')[1] == 512   # the preferred one fits
    with pytest.raises(torch.OutOfMemoryError, match='needed'):
        _ops._scratch(4096, lambda: 1001, 'cpu', 'test')


@pytest.mark.gpu
def test_calls_run_where_only_the_needed_workspace_fits(cuda):
    """With as much memory left as the needed workspace (and the outputs) takes: the same
    terms in other batches, 1e-12 relative."""
    o, v, naux = 10, 64, 192
    p = make_problem(o, v, naux, seed=9, fvo_scale=1e-3)
    u = np.random.default_rng(2).normal(size=(2, o))
    inp = _ops.Inputs(p.mo_energy, p.t1, p.t2, p.ovvv_packed(), p.ovoo, p.ovov, p.fvo, device=cuda)
    g = torch.Generator(device='cuda').manual_seed(1)
    L = torch.randn((naux, o + v, o + v), generator=g, dtype=torch.float64, device='cuda')
    bars = [torch.randn(s, generator=g, dtype=torch.float64, device='cuda')
            for s in ((o, v, v * (v + 1) // 2), (o, v, o, o), (o, v, o, v))]
    n = ctypes.c_size_t(0)
    _lib.check(_lib.load().pamd_df_eris_workspace_size(o, o + v, naux, 0, ctypes.byref(n)), 'size')
    calls = [(lambda: _ops.energy_vjp(inp, et_bar=0.7), _lib.workspace_size(inp.cfg, True, least=True)),
             (lambda: _ops.energy_vjp(inp, et_bar=0.7, workspace=inp.workspace(True)),
              _lib.workspace_size(inp.cfg, True, least=True)),
             (lambda: (_ops.pair_energy(inp), {}), _lib.workspace_size(inp.cfg, False, least=True)),
             (lambda: _ops.projected_energy_vjp(inp, u, et_bar=0.7),
              _projected(inp.cfg, 2, 'pamd_ccsdt_projected_workspace_size')),
             (lambda: (df.df_eris_vjp(L, o, *bars), {}), 2 * n.value)]
    total = torch.cuda.get_device_properties(0).total_memory
    for call, least in calls:
        torch.cuda.empty_cache()
        e, g = call()
        torch.cuda.synchronize()
        torch.cuda.empty_cache()
        # 64 MB for the outputs and the allocator's rounding
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + least + (64 << 20)) / total)
        try:
            e1, g1 = call()
            torch.cuda.synchronize()
        finally:
            torch.cuda.set_per_process_memory_fraction(1.0)
        assert float((e - e1).abs().max()) <= 1e-12 * float(e.abs().max())
        for k in g:
            assert float((g[k] - g1[k]).norm()) <= 1e-12 * float(g[k].norm()) + 1e-18, k
