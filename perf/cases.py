"""Performance cases of the framework: what its users run, through its public entry points.

Kinds of case:

* ``energy``    -- E(T) of one molecule (``cc.ccsd_t.kernel``);
* ``gradient``  -- E(T) and every cotangent (``kernel`` under torch autograd);
* ``fragment``  -- the local-orbital projected (T) and its cotangents
  (``lno.ccsd_t.kernel``);
* ``pairs``     -- one labelled instance of the learned screen: exact
  pair-resolved (T) and the MP2 pair features;
* ``df``        -- the (T) integrals from density-fitting factors and the
  cotangent of the factors (``cc.df.make_df_eris``);
* ``train``     -- one training step of one member of the screen's ensemble;
* ``predict``   -- the ensemble's answer for a set of instances.

The inputs are the seeded density-fitting-like problems of the benchmark
(symmetric factors N(0, 0.1/sqrt(naux)), MP2 amplitudes, t1 ~ N(0, 1e-3),
sorted orbital energies with a gap of at least 0.4 Eh), drawn on the GPU.
"""
import math

import torch

from pyscfad_amd import gen
from pyscfad_amd.cc import ccsd_t, df
from pyscfad_amd.cc.eris import ChemistsERIs, SimpleCCSD
from pyscfad_amd.lno import ccsd_t as lno_ccsd_t
from pyscfad_amd.screen import data as screen_data
from pyscfad_amd.screen import features as screen_features
from pyscfad_amd.screen.ensemble import Screen
from pyscfad_amd.screen.mlp import MLP, to_bf16

GRAD_LEAVES = ('mo_energy', 'fock', 't1', 't2', 'ovvv', 'ovoo', 'ovov')


def _t(name, kind, nocc, nvir, precision='fp64', packed=True, fvo=False, nfrag=0):
    return dict(name=name, kind=kind, nocc=nocc, nvir=nvir, precision=precision, packed=packed,
                fvo=fvo, nfrag=nfrag)


def listed():
    return [
        # a small molecule in an odd-sized basis, full ovvv (conventional
        # integrals): one energy inside a scan, where launches are all that counts
        _t('energy_o5v19', 'energy', 5, 19, packed=False),
        # the smallest gradient in use (the smoke problem): an optimisation step of a
        # small molecule with density-fitted integrals
        _t('gradient_o4v16', 'gradient', 4, 16),
        # the small benchmark configuration, the default precision
        _t('gradient_o8v40', 'gradient', 8, 40),
        # odd sizes and a non-canonical reference (fvo != 0), full ovvv
        _t('gradient_o11v77_fvo', 'gradient', 11, 77, packed=False, fvo=True),
        # the screen's molecule size as an ordinary gradient, in both precisions
        _t('gradient_o16v160', 'gradient', 16, 160),
        _t('gradient_o16v160_bf16x3', 'gradient', 16, 160, precision='bf16x3'),
        # the benchmark's virtual space with few occupied orbitals
        _t('gradient_o6v400_bf16x3', 'gradient', 6, 400, precision='bf16x3'),
        # the largest single-call energy: the mid-size benchmark configuration
        _t('energy_o24v240_bf16x3', 'energy', 24, 240, precision='bf16x3'),
        # one local-orbital fragment of an LNO-CCSD(T) gradient
        _t('fragment_o10v64', 'fragment', 10, 64, nfrag=2),
        # one label and feature row of the screen's data set
        _t('pairs_o16v160', 'pairs', 16, 160, packed=False),
        # integrals and their adjoint on the device
        dict(name='df_o16v160', kind='df', nocc=16, nvir=160, naux=640),
        # one step of the screen's training loop at its batch size and widths
        dict(name='train_b128', kind='train', nocc=16, rows=128),
    ]


def _seconds(kind, o, v, precision):
    """Rough cost of a (T) case, to keep drawn ones below the largest listed."""
    f = 2.0 * o ** 3 * v ** 3 * (o + v)
    rate = 30e12 if precision == 'fp64' else 60e12
    ntrip = o ** 3 / 6
    if kind == 'fragment':
        builds = o * o * (o + 1) / 2
        return 8 * f / rate * builds / ntrip / 2 + 4 * builds * 60e-6
    if kind == 'gradient':
        return 4 * f / rate + ntrip * 100e-6
    return f / rate + ntrip * 30e-6


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(('energy', 'energy', 'gradient', 'gradient', 'gradient', 'fragment', 'pairs',
                       'df', 'train', 'predict'))
    if kind in ('train', 'predict'):
        rows = 8 * rng.randint(4, 64) if kind == 'train' else _log(rng, 8, 2000)
        return dict(kind=kind, nocc=rng.randint(6, 24), rows=rows)
    if kind == 'df':
        o, v = _log(rng, 3, 20), _log(rng, 16, 200)
        return dict(kind=kind, nocc=o, nvir=v, naux=rng.randint(2 * (o + v), 4 * (o + v)))
    while True:
        precision = rng.choice(('fp64', 'fp64', 'bf16x3'))
        o, v = _log(rng, 3, 24), _log(rng, 8, 400)
        nfrag = 0
        if kind == 'fragment':
            o, v, nfrag = _log(rng, 3, 12), _log(rng, 12, 96), rng.randint(1, 4)
        if kind == 'pairs':
            o, v, precision = _log(rng, 6, 20), _log(rng, 40, 180), 'fp64'
        if v < o or _seconds(kind, o, v, precision) > 0.9 or \
                6.0 * o ** 3 * v ** 3 * (o + v) > 9e13:
            continue
        return dict(kind=kind, nocc=o, nvir=v, precision=precision,
                    packed=kind != 'pairs' and rng.random() < 0.6,
                    fvo=kind != 'pairs' and rng.random() < 0.4, nfrag=nfrag)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device='cuda').manual_seed(seed)


def _factors(o, v, naux, g):
    n = o + v
    L = torch.randn((naux, n, n), generator=g, dtype=torch.float64, device='cuda')
    L *= 0.1 / math.sqrt(naux)
    L = torch.tril(L)
    return L + torch.tril(L, -1).transpose(1, 2)


def _energies(o, v, g):
    e = torch.rand(o + v, generator=g, dtype=torch.float64, device='cuda')
    return torch.cat([(-1.5 + 1.2 * e[:o]).sort().values, (0.1 + 2.9 * e[o:]).sort().values])


def _problem(case, seed):
    """The (T) inputs of a case, as a dict of float64 device tensors."""
    o, v = case['nocc'], case['nvir']
    naux = 4 * v
    g = _gen(seed)
    L = _factors(o, v, naux, g)
    mo = _energies(o, v, g)
    Lov = L[:, :o, o:].reshape(naux, o * v)
    Lvv = L[:, o:, o:].reshape(naux, v * v).contiguous()
    il, jl = torch.tril_indices(v, v, device='cuda')
    if case['packed']:
        Lvv = Lvv.view(naux, v, v)[:, il, jl].contiguous()
    ovvv = torch.stack([L[:, i, o:].T @ Lvv for i in range(o)])
    if not case['packed']:
        ovvv = ovvv.view(o, v, v, v)
    ovoo = (Lov.T @ L[:, :o, :o].reshape(naux, o * o)).view(o, v, o, o)
    ovov = (Lov.T @ Lov).view(o, v, o, v)
    eia = mo[:o, None] - mo[None, o:]
    t2 = (ovov.permute(0, 2, 1, 3) / (eia[:, None, :, None] + eia[None, :, None, :])).contiguous()
    t1 = 1e-3 * torch.randn((o, v), generator=g, dtype=torch.float64, device='cuda')
    fock = torch.diag(mo)
    if case['fvo']:
        f = 1e-3 * torch.randn((v, o), generator=g, dtype=torch.float64, device='cuda')
        fock[o:, :o] = f
        fock[:o, o:] = f.T
    p = dict(mo_energy=mo, fock=fock, t1=t1, t2=t2, ovvv=ovvv, ovoo=ovoo, ovov=ovov)
    if case['nfrag']:
        u = torch.randn((case['nfrag'], o), generator=g, dtype=torch.float64, device='cuda')
        p['ulo'] = u / torch.linalg.norm(u, dim=1, keepdim=True)
    return p


def _widths(nocc):
    pad = lambda n: (n + 7) // 8 * 8  # noqa: E731
    return (pad(screen_features.n_features(nocc)), 256, 256, pad(screen_features.n_labels(nocc)))


def _weights(sizes, g):
    """Trained-looking layers: (w, b, first moments, second moments) of each."""
    out = []
    for fan_in, fan_out in zip(sizes[:-1], sizes[1:]):
        r = lambda *s: torch.randn(s, generator=g, device='cuda')  # noqa: E731
        out.append(dict(w=r(fan_out, fan_in) * math.sqrt(2.0 / fan_in), b=0.1 * r(fan_out),
                        m_w=1e-3 * r(fan_out, fan_in), m_b=1e-3 * r(fan_out),
                        v_w=1e-5 + 1e-5 * r(fan_out, fan_in) ** 2, v_b=1e-5 + 1e-5 * r(fan_out) ** 2))
    return out


def _load(net, weights, step):
    for layer, w in zip(net.layers, weights):
        for k in w:
            layer[k].copy_(w[k])
        layer['wb'], layer['wt'] = to_bf16(layer['w'], with_t=True)
    net.step_count = step


def _train_inputs(case, seed):
    g = _gen(seed)
    sizes = _widths(case['nocc'])
    weights = _weights(sizes, g)
    x = torch.randn((case['rows'], sizes[0]), generator=g, device='cuda')
    y = torch.randn((case['rows'], sizes[-1]), generator=g, device='cuda')
    return sizes, weights, x, y


def _predict_inputs(case, seed):
    g = _gen(seed)
    n_in = screen_features.n_features(case['nocc'])
    n_out = screen_features.n_labels(case['nocc'])
    r = lambda *s: torch.randn(s, generator=g, dtype=torch.float64, device='cuda')  # noqa: E731
    sizes = _widths(case['nocc'])
    members = [_weights(sizes, g) for _ in range(4)]
    # pair energies of about 1e-3 Eh, spread over the instances by some per cent
    x_mean, x_std = 1e-3 * r(n_in), 1e-5 * (0.5 + r(n_in).abs())
    y_mean, y_std = 1e-5 * r(n_out), 1e-7 * (0.5 + r(n_out).abs())
    X = x_mean + x_std * r(case['rows'], n_in)
    return n_in, n_out, members, (x_mean, x_std, y_mean, y_std), X


def prepare(case, seed):
    kind = case['kind']
    if kind == 'train':
        sizes, weights, x, y = _train_inputs(case, seed)
        net = MLP(sizes, 'cuda')
        _load(net, weights, 200)
        x16, x16_t = to_bf16(x, with_t=True)
        return dict(kind=kind, net=net, x=x16, xt=x16_t, y=y)
    if kind == 'predict':
        n_in, n_out, members, stats, X = _predict_inputs(case, seed)
        sc = Screen(n_in, n_out, 'cuda', members=len(members))
        for net, w in zip(sc.members, members):
            _load(net, w, 200)
        sc.x_mean, sc.x_std, sc.y_mean, sc.y_std = stats
        return dict(kind=kind, screen=sc, X=X)
    if kind == 'df':
        o, v, naux = case['nocc'], case['nvir'], case['naux']
        L, mo, bars = _df_inputs(case, seed)
        return dict(kind=kind, L=L.requires_grad_(), mo=mo, nocc=o, bars=bars)
    p = _problem(case, seed)
    if kind == 'pairs':
        prob = gen.Problem(case['nocc'], case['nvir'], 4 * case['nvir'], **p)
        return dict(kind=kind, p=prob, precision=case['precision'])
    if kind != 'energy':
        for x in p.values():
            x.requires_grad_()
    cc = SimpleCCSD(t1=p['t1'], t2=p['t2'], verbose=0, ccsd_t_precision=case['precision'])
    eris = ChemistsERIs(**{k: p[k] for k in GRAD_LEAVES if k not in ('t1', 't2')})
    return dict(kind=kind, cc=cc, eris=eris, p=p)


def _df_inputs(case, seed):
    o, v, naux = case['nocc'], case['nvir'], case['naux']
    g = _gen(seed)
    L = _factors(o, v, naux, g)
    mo = _energies(o, v, g)
    r = lambda *s: 1e-3 * torch.randn(s, generator=g, dtype=torch.float64, device='cuda')  # noqa: E731
    return L, mo, [r(o, v, v * (v + 1) // 2), r(o, v, o, o), r(o, v, o, v)]


def run(state):
    kind = state['kind']
    if kind == 'energy':
        return ccsd_t.kernel(state['cc'], state['eris'])
    if kind == 'gradient':
        e = ccsd_t.kernel(state['cc'], state['eris'])
        return (e,) + torch.autograd.grad(e, [state['p'][k] for k in GRAD_LEAVES])
    if kind == 'fragment':
        e = lno_ccsd_t.kernel(state['cc'], state['eris'], state['p']['ulo'], verbose=0)
        return (e,) + torch.autograd.grad(e, [state['p'][k] for k in GRAD_LEAVES + ('ulo',)])
    if kind == 'pairs':
        p = state['p']
        ep = screen_data.exact_pairs(p, precision=state['precision'])
        return (screen_features.features(p.mo_energy, p.ovov, p.nocc),
                screen_features.fold_pairs(ep), ep.sum())
    if kind == 'df':
        e = df.make_df_eris(state['L'], state['nocc'], state['mo'])
        blocks = [e.ovvv, e.ovoo, e.ovov]
        (g,) = torch.autograd.grad(blocks, [state['L']], state['bars'])
        return [b.detach() for b in blocks], g
    if kind == 'train':
        net = state['net']
        loss = net.train_step(state['x'], state['xt'], state['y'], 1e-3, 1e-5)
        return loss, [[L[k] for k in ('w', 'b', 'm_w', 'm_b', 'v_w', 'v_b')] for L in net.layers]
    return state['screen'].predict(state['X'])


def work(case):
    kind = case['kind']
    if kind in ('train', 'predict'):
        s, n = _widths(case['nocc']), case['rows']
        macs = sum(a * b for a, b in zip(s[:-1], s[1:]))
        if kind == 'predict':
            return dict(flops=4 * 2.0 * n * macs,
                        bytes=4 * 2.0 * macs + 8.0 * n * (screen_features.n_features(case['nocc']) + 2))
        # w, both moments read and written; both bf16 copies written, one read
        return dict(flops=(6.0 * macs - 2.0 * s[0] * s[1]) * n,
                    bytes=(6 * 4 + 3 * 2) * macs + n * (2.0 * s[0] + 4.0 * s[-1]))
    o, v = case['nocc'], case['nvir']
    if kind == 'df':
        naux, n = case['naux'], o + v
        cols = v * (v + 1) / 2 + o * o + o * v
        return dict(flops=2.0 * naux * o * v * cols * 3,
                    bytes=8.0 * (2 * naux * n * n + 2 * o * v * cols))
    f = 2.0 * o ** 3 * v ** 3 * (o + v)
    nvvv = o * v * (v * (v + 1) / 2 if case['packed'] else v * v)
    inputs = 8.0 * (nvvv + 2.0 * o * o * v * v + o ** 3 * v + (o + v))
    if kind == 'fragment':  # one W build per occupied pair and orbital; twice that for the adjoint
        return dict(flops=3 * f * (o * o * (o + 1) / 2) / (o ** 3 / 6), bytes=2 * inputs)
    if kind == 'gradient':
        return dict(flops=3 * f, bytes=2 * inputs)
    return dict(flops=f, bytes=inputs)


# ---------------------------------------------------------------------------
# 64-bit values by plain torch
# ---------------------------------------------------------------------------
def _w_block(q, i, j, ks):
    """W_ijk[a, b, c] for the occupied indices k in ``ks``: [n, v, v, v]."""
    t2, vv, oo = q['t2'], q['full'], q['ovoo']
    e = torch.einsum
    w = e('afb,ncf->nabc', vv[i], t2[ks, j]) + e('afc,nbf->nabc', vv[i], t2[j, ks])
    w = w + e('bfa,ncf->nabc', vv[j], t2[ks, i]) + e('bfc,naf->nabc', vv[j], t2[i, ks])
    w = w + e('ncfa,bf->nabc', vv[ks], t2[j, i]) + e('ncfb,af->nabc', vv[ks], t2[i, j])
    w = w - e('am,nmcb->nabc', oo[i, :, :, j], t2[ks]) - e('amn,mbc->nabc', oo[i][:, :, ks], t2[j])
    w = w - e('bm,nmca->nabc', oo[j, :, :, i], t2[ks]) - e('bmn,mac->nabc', oo[j][:, :, ks], t2[i])
    return w - e('ncm,mba->nabc', oo[ks][..., i], t2[j]) - e('ncm,mab->nabc', oo[ks][..., j], t2[i])


def _z_and_d(q, i, j, ks, w):
    """Z = r3(W + V) and the denominators, laid out like ``w``."""
    o = q['t1'].shape[0]
    t1, t2, ov, fvo = q['t1'], q['t2'], q['ovov'], q['fock'][o:, :o]
    sym = lambda x, y: ov[x, :, y, :] + ov[y, :, x, :].T  # noqa: E731
    amp = lambda x, y: t2[x, y] + t2[y, x].T  # noqa: E731
    stack = lambda f, x: torch.stack([f(x, k) for k in ks.tolist()])  # noqa: E731
    e = torch.einsum
    x = w + 0.5 * (e('ab,nc->nabc', sym(i, j), t1[ks]) + e('nac,b->nabc', stack(sym, i), t1[j]) +
                   e('nbc,a->nabc', stack(sym, j), t1[i]))
    x = x + 0.5 * (e('ab,cn->nabc', amp(i, j), fvo[:, ks]) +
                   e('nac,b->nabc', stack(amp, i), fvo[:, j]) +
                   e('nbc,a->nabc', stack(amp, j), fvo[:, i]))
    z = 4 * x + x.permute(0, 2, 3, 1) + x.permute(0, 3, 1, 2)
    z = z - 2 * (x.permute(0, 3, 2, 1) + x.permute(0, 1, 3, 2) + x.permute(0, 2, 1, 3))
    eo, ev = q['mo_energy'][:o], q['mo_energy'][o:]
    d = (eo[i] + eo[j] + eo[ks])[:, None, None, None] - ev[:, None, None] - ev[:, None] - ev
    return z, d


def _unpacked(p):
    v = p['t1'].shape[1]
    ovvv = p['ovvv']
    if ovvv.dim() == 3:
        il, jl = torch.tril_indices(v, v, device='cuda')
        at = torch.zeros((v, v), dtype=torch.int64, device='cuda')
        at[il, jl] = torch.arange(il.numel(), device='cuda')
        at[jl, il] = torch.arange(il.numel(), device='cuda')
        ovvv = ovvv[:, :, at]
    return dict(p, full=ovvv)


def _triples(case, p, grad):
    """(E, triple energies [o, o, o] over i <= j <= k); gradients go to p's leaves."""
    o, v = case['nocc'], case['nvir']
    q = _unpacked(p)
    if grad:  # each block's backward stops at q and is passed on at the end
        full = q['full']
        q['full'] = full.detach().requires_grad_()
    total = torch.zeros((), dtype=torch.float64, device='cuda')
    tri = torch.zeros((o, o, o), dtype=torch.float64, device='cuda')
    most = max(1, int(20e9 / (8 * 40 * v ** 3)))
    for i in range(o):
        for j in range(i, o):
            for k0 in range(j, o, most):
                ks = torch.arange(k0, min(o, k0 + most), device='cuda')
                w = _w_block(q, i, j, ks)
                z, d = _z_and_d(q, i, j, ks, w)
                e = (w * z / d).sum((1, 2, 3))
                same = (ks == j).double() + float(i == j)
                weight = torch.where(same == 2, 0.0, torch.where(same == 1, 1.0, 2.0))
                if grad:
                    (weight * e).sum().backward()
                total += (weight * e.detach()).sum()
                tri[i, j, k0:k0 + len(ks)] = e.detach()
    if grad:
        if full.requires_grad and full is not p['ovvv']:
            full.backward(q['full'].grad)
        else:
            p['ovvv'].grad = q['full'].grad
    return total, tri


def _fragment(case, p):
    o, v = case['nocc'], case['nvir']
    q = _unpacked(p)
    full = q['full']
    q['full'] = full.detach().requires_grad_()
    total = torch.zeros((), dtype=torch.float64, device='cuda')
    ls = torch.arange(o, device='cuda')
    for j in range(o):
        for k in range(j, o):
            w = _w_block(q, j, k, ls)
            z, d = _z_and_d(q, j, k, ls, w)
            a = torch.einsum('fn,nbca->fbca', p['ulo'], w)
            b = torch.einsum('fn,nbca->fbca', p['ulo'], z / d)
            e = (a * b).sum() * ((1.0 if j == k else 2.0) / 3.0)
            e.backward()
            total += e.detach()
    if full is not p['ovvv']:
        full.backward(q['full'].grad)
    else:
        p['ovvv'].grad = q['full'].grad
    return total


def _mlp64(weights, x):
    h = x
    for n, (w, b) in enumerate(weights):
        h = h @ w.T + b
        if n < len(weights) - 1:
            h = h * torch.sigmoid(h)
    return h


def _bf(x):
    return x.to(torch.bfloat16).double()


def exact(case, seed):
    kind = case['kind']
    if kind == 'train':
        sizes, layers, x, y = _train_inputs(case, seed)
        weights = [(_bf(L['w']).requires_grad_(), L['b'].double().requires_grad_()) for L in layers]
        loss = ((_mlp64(weights, _bf(x)) - y.double()) ** 2).mean()
        loss.backward()
        step, out = 201, []
        for L, (w, b) in zip(layers, weights):
            new = {}
            for k, g, wd in (('w', w.grad, 1e-5), ('b', b.grad, 0.0)):
                m = 0.9 * L['m_' + k].double() + 0.1 * g
                s = 0.999 * L['v_' + k].double() + 0.001 * g * g
                x0 = L[k].double()
                up = (m / (1 - 0.9 ** step)) / ((s / (1 - 0.999 ** step)).sqrt() + 1e-8)
                new.update({k: x0 - 1e-3 * (up + wd * x0), 'm_' + k: m, 'v_' + k: s})
            out.append([new[k] for k in ('w', 'b', 'm_w', 'm_b', 'v_w', 'v_b')])
        return loss.detach(), out
    if kind == 'predict':
        n_in, n_out, members, (x_mean, x_std, y_mean, y_std), X = _predict_inputs(case, seed)
        pad = _widths(case['nocc'])[0] - n_in
        x = torch.nn.functional.pad((X - x_mean) / x_std, (0, pad))
        e = torch.stack([
            (_mlp64([(_bf(L['w']), L['b'].double()) for L in net], x)[:, :n_out] * y_std + y_mean).sum(-1)
            for net in members])
        return e.mean(0), e.std(0)
    if kind == 'df':
        o, v = case['nocc'], case['nvir']
        L, _, bars = _df_inputs(case, seed)
        L.requires_grad_()
        il, jl = torch.tril_indices(v, v, device='cuda')
        Lov = L[:, :o, o:].reshape(L.shape[0], -1)
        blocks = [(Lov.T @ L[:, o:, o:][:, il, jl]).view(o, v, -1),
                  (Lov.T @ L[:, :o, :o].reshape(L.shape[0], -1)).view(o, v, o, o),
                  (Lov.T @ Lov).view(o, v, o, v)]
        (g,) = torch.autograd.grad(blocks, [L], bars)
        return [b.detach() for b in blocks], g
    o, v = case['nocc'], case['nvir']
    # v^3-sized passes of a block, its launches and its contractions
    blocks = o * (o + 1) / 2
    passes = (o if kind == 'fragment' else o / 3) * blocks
    grad = kind in ('gradient', 'fragment')
    cost = (3 if grad else 1) * (passes * (60 * 8 * v ** 3 / 3e12 + 12 * 2.0 * v ** 4 / 3e13) + blocks * 5e-3)
    if cost > 15:
        return None
    p = _problem(case, seed)
    if grad:
        for x in p.values():
            x.requires_grad_()
    if kind == 'energy':
        return _triples(case, p, False)[0]
    if kind == 'gradient':
        e, _ = _triples(case, p, True)
    elif kind == 'fragment':
        e = _fragment(case, p)
    else:
        e, tri = _triples(case, p, False)
        full = torch.zeros_like(tri)
        for perm in ((0, 1, 2), (0, 2, 1), (1, 0, 2), (1, 2, 0), (2, 0, 1), (2, 1, 0)):
            t = tri.permute(perm)
            full = torch.where(t != 0, t, full)
        n = torch.arange(o, device='cuda')
        full[n, n, n] = 0
        ep = full.sum(2) / 3
        g = p['ovov'].permute(0, 2, 1, 3)
        mp2 = (p['t2'] * (2 * g - g.transpose(2, 3))).sum((2, 3))
        mo = p['mo_energy']
        iu, ju = torch.triu_indices(o, o, offset=1, device='cuda')
        x = torch.cat([(mp2 + mp2.T)[iu, ju], torch.stack(
            [mo[o:].min() - mo[:o].max(), mo[:o].mean(), mo[:o].std(), mo[:o].min(), mo[o:].mean(),
             mo[o:].std(), mo[o:].max(), mp2.sum()])])
        iu, ju = torch.triu_indices(o, o, device='cuda')
        y = torch.where(iu == ju, ep[iu, iu], (ep + ep.T)[iu, ju])
        return x, y, e
    names = GRAD_LEAVES + (('ulo',) if kind == 'fragment' else ())
    return (e,) + tuple(p[k].grad if p[k].grad is not None else torch.zeros_like(p[k]) for k in names)
