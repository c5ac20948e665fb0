"""GPU parity of the table gradient and dx of few nodes over 2049 to 16384 frames (two-valued inputs; a workgroup sums a node's frames): every width, the smallest and
largest ranges, shares that end within a pass or hold nothing, rows of any pitch, gradients added to what is there."""
import pytest
import torch

from test_gpu_few_inputs import layer, reference

pytestmark = pytest.mark.gpu


def table_gradient(n, idx, W, x, dy, F, bias, norm=None):
    """dW in 64 bits, by the sums of g over the frames at each corner, and the sum of |g| over the frames of each node"""
    hi, lo = 0.5 + bias, 0.5 - bias
    p = torch.arange(1 << n, device="cuda")
    factors = torch.ones((1 << n, 1 << n), dtype=torch.float64, device="cuda")              # [entry][corner]
    for k in range(n):
        at = torch.where((p >> k) & 1 == 1, hi, lo).double()
        factors *= torch.where(((p >> k) & 1 == 1)[:, None], at[None, :], 1 - at[None, :])
    V = W.double() @ factors
    shift = torch.arange(32, device="cuda", dtype=torch.int32)
    bits = ((x[:, :(F + 31) // 32, None] >> shift) & 1).reshape(x.shape[0], -1)[:, :F]
    dW, size = torch.zeros_like(V), torch.zeros((W.shape[0], 1), dtype=torch.float64, device="cuda")
    for o in range(W.shape[0]):
        corner = sum(bits[idx[o, k].long()].long() << k for k in range(n))
        g = dy[o, :F].double()
        size[o] = g.abs().sum()
        if norm is not None:
            mean, rstd, gamma, beta = norm[0][o].double(), norm[1][o].double(), norm[2], norm[3]
            t = (V[o] - mean) * rstd * gamma + beta
            g = torch.where(((t > 0) & (t < 1))[corner], g, torch.zeros_like(g))
            v = V[o][corner] - mean
            size[o] = gamma * rstd * (g.abs().sum() + g.sum().abs() + (v * rstd).abs().mean() * (g * v * rstd).abs().sum())
            g = gamma * rstd * (g - g.sum() / F - v * rstd * rstd * (g * v).sum() / F)
        D = torch.zeros(1 << n, dtype=torch.float64, device="cuda").index_add_(0, corner, g)
        dW[o] = factors @ D
    return dW, size


@pytest.mark.parametrize("n, I, O, F, pitch", [(6, 40, 256, 2049, 0), (6, 9, 24, 16384, 0), (6, 7, 3, 4097, 4097), (6, 300, 72, 9001, 9003), (5, 40, 130, 2304, 0), (5, 11, 256, 16383, 0),
                                               (4, 60, 512, 3000, 0), (4, 9, 10, 16129, 16131), (3, 33, 300, 8193, 0), (2, 5, 50, 5000, 0), (6, 30, 257, 5000, 0), (6, 30, 20, 16385, 0)])
def test_sums_of_few_nodes(n, I, O, F, pitch):
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    idx, W, x, dy = layer(n, I, O, F, 10 * n + O)
    if pitch: dy = torch.nn.functional.pad(dy[:, :F], (0, pitch - F), value=float("nan")).contiguous()
    rev = ops.reverse_table(idx, I)
    mean, rstd = W.mean(dim=1).contiguous(), (0.5 / W.std(dim=1)).contiguous()
    for norm in (None, (mean, rstd, 0.7, 0.5)):
        before = torch.rand_like(W)
        dW = before.clone()
        if norm is None:
            dx = ops.bit_stochastic_lut_backward(n, x, dy, idx, W, dW, F, rev, bias=0.25)
        else:
            dx = ops.bit_differentiable_lut_backward(n, x, dy, idx, W, dW, F, mean, rstd, rev, gamma=0.7, beta=0.5, bias=0.25)
        want, size = table_gradient(n, idx, W, x, dy, F, 0.25, norm)
        # fp32 sums of at most 32 frames of a lane, 18 groups of columns, 8 wavefronts, and some 20 operations to fold them, each half a unit of rounding of sums of |g|
        assert bool(((dW - before.double() - want).abs() <= 80 * 2.0 ** -24 * (size + 2)).all()), norm is None
        want = reference(n, idx, W, x, dy, F, 0.25, norm)
        assert float((dx[:, :F] - want).abs().max()) <= 2 * int(rev[:, 0].max()) * 2.0 ** -24 * float(want.abs().max()) + 1e-6, norm is None
