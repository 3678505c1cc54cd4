"""The whole-network MLP launches against the layer-by-layer kernels they stand for:
the same MFMAs, roundings and expressions per element, so predictions are bitwise
equal; a training step differs only where FP32 expressions are contracted or summed
in another order (a few ulp: 1e-5 relative to the largest entry).  Sizes: the
screen's, one row block with a remainder, one tile of 8 columns, widths that are no
multiple of 16; and the forms that must go the layer-by-layer way."""
import copy

import pytest
import torch

from tests import mlp_reference as REF

pytestmark = pytest.mark.gpu

KEYS = ('w', 'b', 'm_w', 'v_w', 'm_b', 'v_b')


def _net(M, sizes, rows, dev, seed=1):
    g = torch.Generator().manual_seed(seed)
    net = M.MLP(sizes, dev, seed=seed)
    for L in net.layers:
        L['b'].copy_(0.1 * torch.randn(L['b'].shape, generator=g))
        for k in ('w', 'b'):
            L['m_' + k].copy_(1e-3 * torch.randn(L[k].shape, generator=g))
            L['v_' + k].copy_(1e-5 + 1e-5 * torch.rand(L[k].shape, generator=g))
    net.step_count = 20
    x = torch.randn(rows, sizes[0], generator=g).to(dev)
    y = torch.randn(rows, sizes[-1], generator=g).to(dev)
    return (net,) + tuple(M.to_bf16(x, with_t=True)) + (y,)


@pytest.mark.parametrize('sizes,rows', [((128, 256, 256, 136), 128), ((40, 64, 24), 72), ((8, 8), 8),
                                        ((24, 40, 8, 56, 16), 16)])
def test_train_step_matches_the_layerwise_step(cuda, sizes, rows):
    from pyscfad_amd.screen import mlp as M
    net, x, xt, y = _net(M, sizes, rows, cuda)
    ref = copy.deepcopy(net)
    for _ in range(2):
        loss = net._fused_step(x, xt, y, 1e-3, 1e-4)
        assert loss is not None
        _, loss_r, g = ref.grads(x, xt, y)
        ref.adam(g, lr=1e-3, wd=1e-4)
        assert abs(float(loss) - float(loss_r)) <= 1e-5 * float(loss_r)
        for L, R in zip(net.layers, ref.layers):
            for k in KEYS:
                assert float((L[k] - R[k]).abs().max()) <= 1e-5 * float(R[k].abs().max()), k
            assert torch.equal(L['wb'].T, L['wt'])
            assert torch.equal(M.bf16_to_f32(L['wb']).cpu(), REF.bf16_round(L['w'].cpu()))
    assert net.step_count == ref.step_count


@pytest.mark.parametrize('sizes,rows', [((128, 256, 256, 136), 248), ((40, 64, 24), 1), ((8, 8), 17)])
def test_member_forward_is_bitwise_the_layerwise_one(cuda, sizes, rows):
    from pyscfad_amd.screen import mlp as M
    nets = [_net(M, sizes, 8, cuda, seed=s)[0] for s in (1, 2, 3)]
    x = M.to_bf16(torch.randn(rows, sizes[0], device=cuda))
    out = M.forward_members(nets, x)
    for net, z in zip(nets, out):
        assert torch.equal(net.forward(x), z)


def test_other_forms_go_layer_by_layer(cuda):
    from pyscfad_amd.screen import mlp as M
    net, x, xt, y = _net(M, (64, 1024, 1024, 16), 16, cuda)      # activations beyond LDS
    assert net._fused_step(x, xt, y, 1e-3, 0.0) is None and net.step_count == 20
    float(net.train_step(x, xt, y, 1e-3))
    assert net.step_count == 21
    net, x, xt, y = _net(M, (16, 24, 8), 16, cuda)
    wide = torch.zeros((16, 32), dtype=torch.int16, device=cuda)
    wide[:, :16] = x                                             # strided rows
    assert M.forward_members([net], wide[:, :16]) is None
    assert torch.equal(net.forward(wide[:, :16]), M.forward_members([net], x)[0])


def test_standardise_is_the_torch_expression(cuda):
    from pyscfad_amd.screen import mlp as M
    g = torch.Generator().manual_seed(3)
    X = torch.randn(37, 29, generator=g, dtype=torch.float64).to(cuda)
    mean, std = X.mean(0), X.std(0)
    ref = M.to_bf16(torch.nn.functional.pad(((X - mean) / std).float(), (0, 3)))
    assert torch.equal(M.standardise(X, mean, std, 32), ref)
