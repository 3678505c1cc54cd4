"""Training steps that the whole-network kernels do not take look at nothing but the
widths and the row count before they go the per-layer way."""
import types

import pytest
import torch

from pyscfad_amd.screen.mlp import MLP


class _Layers(list):
    """Layers that may not be looked at."""

    def __iter__(self):
        raise AssertionError('layers were walked')


# activations beyond LDS; too many layers; rows or a width that is no multiple of 8
@pytest.mark.parametrize('sizes,rows', [([64, 512, 512, 64], 64), ([8, 1024, 1024, 8], 64),
                                        ([16, 32, 32, 32, 32, 8], 64), ([16, 32, 8], 12), ([16, 36, 8], 16)])
def test_unsupported_steps_are_refused_by_their_widths(sizes, rows):
    net = types.SimpleNamespace(sizes=sizes, layers=_Layers(), step_count=0)
    x = torch.zeros((rows, sizes[0]), dtype=torch.int16)
    assert MLP._fused_step(net, x, x.t().contiguous(), torch.zeros((rows, sizes[-1])), 1e-3, 0.0) is None
    assert net.step_count == 0
