"""GPU parity of dx over two-valued inputs at the lines between passes of 256 and of 512 frames: 512, 1024, 1350 and 1600 nodes, 2000 and 10000 groups, long and short lists, a second pass of one frame."""
import pytest
import torch

from test_gpu_few_inputs import layer, reference

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n, I, O, F", [(6, 800, 1350, 2049), (6, 800, 1350, 2048), (4, 800, 1351, 2049), (5, 1400, 1600, 1025), (2, 1333, 1025, 1281), (3, 40, 24, 51201),
                                        (6, 892, 1350, 2049), (6, 1000, 1350, 2048), (6, 996, 1350, 2048), (5, 480, 1600, 4097), (5, 480, 1601, 4097), (4, 1600, 700, 1025), (4, 3000, 1030, 3585), (4, 3000, 1030, 3300),
                                        (6, 1333, 1000, 1281), (6, 1333, 999, 1281), (2, 900, 512, 2049), (2, 900, 513, 2049)])
def test_dx_in_two_passes(n, I, O, F):
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    idx, W, x, dy = layer(n, I, O, F, 10 * n + O)
    rev = ops.reverse_table(idx, I)
    mean, rstd = W.mean(dim=1).contiguous(), (0.5 / W.std(dim=1)).contiguous()
    for norm in (None, (mean, rstd, 0.7, 0.5)):
        dW = torch.zeros_like(W)
        if norm is None:
            dx = ops.bit_stochastic_lut_backward(n, x, dy, idx, W, dW, F, rev, bias=0.25)
        else:
            dx = ops.bit_differentiable_lut_backward(n, x, dy, idx, W, dW, F, mean, rstd, rev, gamma=0.7, beta=0.5, bias=0.25)
        want = reference(n, idx, W, x, dy, F, 0.25, norm)
        # a sum over an input's connections, in fp32: their number times half a unit of rounding, relative to the largest sum, and as much for each factor;
        # the difference of two corner values of up to 1 is off by a unit for each of the n steps that form them, and batch-norm multiplies by 0.7 rstd
        links, gain = int(rev[:, 0].max()), 1.0 if norm is None else 0.7 * float(rstd.max())
        bound = 2 * links * 2.0 ** -24 * (float(want.abs().max()) + n * gain * float(dy[:, :F].abs().max())) + 1e-6
        assert float((dx[:, :F] - want).abs().max()) <= bound, norm is None
