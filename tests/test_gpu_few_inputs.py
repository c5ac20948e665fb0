"""GPU parity of dx formed node by node (layers of few inputs over many frames, two-valued inputs): widths, one to 28 inputs, up to 4096 nodes, last words, last pairs
of frames, last rounds of nodes, more workgroups than are resident, gradients that are not finite behind a closed window, reverse tables of the caller's own, fp32 frames."""
import numpy as np
import pytest
import torch

from binarybrain_amd import synth
from util import host

pytestmark = pytest.mark.gpu
LEAST = 191 * 512 + 1           # frames


def layer(n, I, O, F, seed):
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda"); gen.manual_seed(seed)
    idx = torch.from_numpy(synth.wiring(rng, I, O, n) if I >= n else rng.integers(0, I, (O, n)).astype(np.int32)).cuda()
    W = torch.rand((O, 1 << n), device="cuda", generator=gen)
    x = torch.randint(-(1 << 31), 1 << 31, (I, synth.frame_stride_bit(F)), device="cuda", generator=gen).to(torch.int32)
    dy = torch.full((O, synth.frame_stride_fp32(F)), float("nan"), device="cuda")            # what lies behind the frames enters nothing
    dy[:, :F] = torch.randn((O, F), device="cuda", generator=gen)
    return idx, W, x, dy


def reference(n, idx, W, x, dy, F, bias, norm=None, rev=None):
    """dx in 64 bits, by the corner values and their differences; norm: (mean, rstd, gamma, beta) of a batch-norm layer; rev: the reverse table where it is not the
    one of the wiring (a connection's gradient goes to the inputs whose rows list it, as often as they do)"""
    O, I, dev = idx.shape[0], x.shape[0], "cuda"
    rows = [[[int(idx[o, k])] for k in range(n)] for o in range(O)] if rev is None else [[[] for _ in range(n)] for _ in range(O)]
    if rev is not None:
        for i, row in enumerate(host(rev)):
            for e in row[1:1 + row[0]]:
                rows[e // n][e % n].append(i)
    hi, lo = 0.5 + bias, 0.5 - bias
    p = torch.arange(1 << n, device=dev)
    V = torch.zeros((O, 1 << n), dtype=torch.float64, device=dev)
    for i in range(1 << n):
        f = torch.ones(1 << n, dtype=torch.float64, device=dev)
        for k in range(n):
            v = torch.where((p >> k) & 1 == 1, hi, lo).double()
            f *= v if (i >> k) & 1 else 1 - v
        V += W[:, i:i + 1].double() * f
    words, shift = x[:, :(F + 31) // 32], torch.arange(32, device=dev, dtype=torch.int32)
    bits = ((words[:, :, None] >> shift) & 1).reshape(I, -1)[:, :F]
    dx = torch.zeros((I, F), dtype=torch.float64, device=dev)
    for o in range(O):
        corner = sum(bits[idx[o, k].long()].long() << k for k in range(n))
        g = dy[o, :F].double()
        if norm is not None:
            mean, rstd, gamma, beta = norm[0][o].double(), norm[1][o].double(), norm[2], norm[3]
            t = (V[o] - mean) * rstd * gamma + beta
            g = torch.where(((t > 0) & (t < 1))[corner], g, torch.zeros_like(g))
            v = V[o][corner] - mean
            g = gamma * rstd * (g - g.sum() / F - v * rstd * rstd * (g * v).sum() / F)
        for k in range(n):
            slope = (V[o][p | (1 << k)] - V[o][p & ~(1 << k)]) / (hi - lo)
            for i in rows[o][k]:
                dx[i] += slope[corner] * g
    return dx


# (from 513 nodes on the threads of a workgroup fill the wiring in several rounds; 4096 nodes are the most, with the most LDS; 262144 frames fill the device once)
@pytest.mark.parametrize("n, I, O, F", [(6, 28, 38, LEAST), (6, 27, 216, LEAST + 30), (5, 9, 41, LEAST + 1), (4, 1, 50, LEAST + 127), (3, 13, 67, LEAST + 129), (2, 25, 121, LEAST + 510),
                                        (6, 27, 513, LEAST + 3), (6, 28, 4096, LEAST), (2, 3, 4096, LEAST + 2), (4, 9, 50, 262144), (6, 6, 37, 262146)])
def test_dx_node_by_node(n, I, O, F):
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
        # a sum over an input's connections, in fp32: their number times half a unit of rounding, relative to the largest sum, and as much for each factor
        links = int(rev[:, 0].max())
        assert float((dx[:, :F] - want).abs().max()) <= 2 * links * 2.0 ** -24 * float(want.abs().max()) + 1e-6, norm is None


def test_a_discarded_gradient_may_hold_anything():
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    n, I, O, F = 6, 27, 40, LEAST + 3
    idx, W, x, dy = layer(n, I, O, F, 4)
    rev = ops.reverse_table(idx, I)
    mean, rstd = W.mean(dim=1).contiguous(), (2.0 / W.std(dim=1)).contiguous()
    y = ops.bit_stochastic_lut_forward(n, x, idx, W, F, dy.shape[1], bias=0.25)[:, :F].double()
    t = (y - mean[:, None].double()) * rstd[:, None].double() + 0.5
    closed = (t < -1e-3) | (t > 1.001)
    assert 0.2 < float(closed.double().mean()) < 0.95
    zeros, poisoned = dy.clone(), dy.clone()
    zeros[:, :F][closed] = 0.0
    poisoned[:, :F][closed] = torch.tensor([np.inf, -np.inf, np.nan, 3.0e38], device="cuda")[torch.arange(int(closed.sum()), device="cuda") % 4]
    got = [host(ops.bit_differentiable_lut_backward(n, x, g, idx, W, torch.zeros_like(W), F, mean, rstd, rev, gamma=1.0, beta=0.5, bias=0.25))[:, :F] for g in (zeros, poisoned)]
    assert np.isfinite(got[1]).all() and np.array_equal(*got)


@pytest.mark.parametrize("n, I, O, F", [(6, 27, 40, LEAST + 1), (4, 9, 600, LEAST), (2, 5, 130, LEAST + 257)])
@pytest.mark.parametrize("how", ["left out", "twice", "descending", "elsewhere"])
def test_dx_goes_by_the_reverse_table(n, I, O, F, how):
    """A caller's reverse table need not be the wiring's own: the deterministic dx walks its lists, in layers of this size as in others."""
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    idx, W, x, dy = layer(n, I, O, F, 7 * n + O)
    rows = [list(r[1:1 + r[0]]) for r in host(ops.reverse_table(idx, I))]
    if how == "left out":     del rows[1][2]; rows[3] = []                           # a connection, and all of an input
    if how == "twice":        rows[0].append(rows[0][-1]); rows[2].pop(0)           # (as many entries as connections)
    if how == "descending":   rows = [r[::-1] for r in rows]
    if how == "elsewhere":    rows[4].append(rows[0].pop(0))
    rev = np.zeros((I, 1 + max(len(r) for r in rows)), np.int32)
    for i, r in enumerate(rows):
        rev[i, 0], rev[i, 1:1 + len(r)] = len(r), r
    rev = torch.from_numpy(rev).cuda()
    mean, rstd = W.mean(dim=1).contiguous(), (0.5 / W.std(dim=1)).contiguous()
    for norm in (None, (mean, rstd, 0.7, 0.5)):
        dW = torch.zeros_like(W)
        if norm is None:
            dx = ops.bit_stochastic_lut_backward(n, x, dy, idx, W, dW, F, rev, bias=0.25)
        else:
            dx = ops.bit_differentiable_lut_backward(n, x, dy, idx, W, dW, F, mean, rstd, rev, gamma=0.7, beta=0.5, bias=0.25)
        want = reference(n, idx, W, x, dy, F, 0.25, norm, rev)
        assert float((dx[:, :F] - want).abs().max()) <= 2 * int(rev[:, 0].max()) * 2.0 ** -24 * float(want.abs().max()) + 1e-6, (how, norm is None)


@pytest.mark.parametrize("n, I, O, F", [(6, 27, 40, LEAST + 1), (4, 9, 60, LEAST)])
def test_fp32_frames_of_binary_mode(n, I, O, F):
    """fp32 frames are packed to bits by the call itself, behind the tables that dx is formed from in the same scratch memory: the bits of the packed call"""
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    idx, W, xb, dy = layer(n, I, O, F, n + O)
    shift = torch.arange(32, device="cuda", dtype=torch.int32)
    x = torch.full((I, dy.shape[1]), float("nan"), device="cuda")
    x[:, :F] = ((xb[:, :(F + 31) // 32, None] >> shift) & 1).reshape(I, -1)[:, :F].float()
    rev = ops.reverse_table(idx, I)
    mean, rstd = W.mean(dim=1).contiguous(), (0.5 / W.std(dim=1)).contiguous()
    for bn in (False, True):
        got = []
        for call, inputs in (("bit_", xb), ("", x)):
            dW = torch.zeros_like(W)
            if bn: dx = getattr(ops, call + "differentiable_lut_backward")(n, inputs, dy, idx, W, dW, F, mean, rstd, rev, gamma=0.7, beta=0.5, bias=0.25)
            else:  dx = getattr(ops, call + "stochastic_lut_backward")(n, inputs, dy, idx, W, dW, F, rev, bias=0.25, **({} if call else {"input_binary": True}))
            got.append((dx[:, :F], dW))
        assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1]), bn
