"""GPU parity of the backward pass over two-valued inputs (per-corner sums, fold, dx from kept corner indices) at the sizes where its kernels
have edges: last words and last groups of four frames, passes of 256 and blocks of 2048 frames, several slabs per node, shared work lists."""
import numpy as np
import pytest

import oracle
from binarybrain_amd import synth
from util import assert_bwd, dev, host

pytestmark = pytest.mark.gpu


# inputs, nodes, frames, row pitch of the fp32 buffers (0: the frame buffer's)
SHAPES = [(7, 3, 1, 0), (7, 3, 5, 0), (9, 5, 31, 31), (16, 9, 33, 35), (40, 70, 255, 255), (6, 130, 257, 0), (24, 4, 2047, 2047), (12, 6, 2049, 2052),
          (27, 36, 6001, 6001), (8, 40, 20001, 0), (600, 520, 300, 0), (1030, 1100, 65, 0)]


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("shape", SHAPES)
def test_corner_backward(n, shape):
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    I, O, F, stride = shape
    stride = stride or synth.frame_stride_fp32(F)
    rng = np.random.default_rng(100 * n + F)
    idx = synth.wiring(rng, I, O, n); W = synth.lut_tables(rng, O, n)
    x = synth.uniform_frames(rng, I, F, stride); dy = synth.normal_frames(rng, O, F, stride)
    xb = synth.pack_bits((x[:, :F] > 0.5).astype(np.uint8), (F + 31) // 32)
    _, mean, rstd, _, _ = oracle.differentiable_lut_forward_training(n, x, idx, W, F, np.zeros(O, np.float32), np.ones(O, np.float32))
    want = {True: oracle.differentiable_lut_backward(n, x, dy, idx, W, F, mean, rstd),
            False: oracle.stochastic_lut_backward(n, x, dy, idx, W, F, input_binary=True, simd=False)}
    dy[:, F:] = np.nan                              # what lies behind the frames enters nothing
    d_x, d_xb, d_dy, d_idx, d_W = dev(x), dev(xb), dev(dy), dev(idx), dev(W)
    rev = ops.reverse_table(d_idx, I)
    start = dev(np.full_like(W, 0.25))
    for bn in ((True, False) if F > 4 else (False,)):            # (the gradient through the statistics of a frame or two is rounding alone)
        dx_ref, dW_ref = want[bn]
        got = []
        for packed in (False, True):
            dW = start.clone()
            if bn:
                args = (n, d_xb if packed else d_x, d_dy, d_idx, d_W, dW, F, dev(mean), dev(rstd), rev)
                dx = (ops.bit_differentiable_lut_backward if packed else ops.differentiable_lut_backward)(*args)
            else:
                args = (n, d_xb if packed else d_x, d_dy, d_idx, d_W, dW, F, rev)
                dx = ops.bit_stochastic_lut_backward(*args) if packed else ops.stochastic_lut_backward(*args, input_binary=True)
            assert_bwd(host(dx)[:, :F], dx_ref[:, :F], "dx bn=%d packed=%d" % (bn, packed))
            assert_bwd(host(dW) - 0.25, dW_ref, "dW bn=%d packed=%d" % (bn, packed))
            got.append((host(dx)[:, :F], host(dW)))
        assert all(np.array_equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("bias", [0.0, 0.01, 0.0625])
def test_input_values_that_nearly_meet(bias):
    """slopes are not taken from differences of corner values where those lose digits"""
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    rng = np.random.default_rng(3)
    I, O, F = 20, 30, 200
    stride = synth.frame_stride_fp32(F)
    idx = synth.wiring(rng, I, O, 6); W = synth.lut_tables(rng, O, 6)
    x = synth.uniform_frames(rng, I, F, stride); dy = synth.normal_frames(rng, O, F, stride)
    dx_ref, dW_ref = oracle.stochastic_lut_backward(6, x, dy, idx, W, F, input_binary=True, bias=bias, simd=False)
    dW = dev(np.zeros_like(W))
    d_idx = dev(idx)
    dx = ops.stochastic_lut_backward(6, dev(x), dev(dy), d_idx, dev(W), dW, F, ops.reverse_table(d_idx, I), input_binary=True, bias=bias)
    assert_bwd(host(dx)[:, :F], dx_ref[:, :F], "dx"); assert_bwd(host(dW), dW_ref, "dW")


@pytest.mark.parametrize("n", [2, 4, 6])
@pytest.mark.parametrize("shape", [(7, 3, 33, 0), (40, 70, 255, 255), (24, 40, 1300, 0), (12, 600, 3000, 0), (1030, 1100, 65, 0), (27, 36, 20001, 0)])
def test_a_discarded_gradient_may_hold_anything(n, shape):
    """dy counts as 0 where the batch-norm output lies outside the hard-tanh window, also where it is infinite or no number: the same bits as with
    zeros there.  One frame of values per lane and of every kind of dx launch: single words, shared lists, one to four groups of 256 frames."""
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    I, O, F, stride = shape
    stride = stride or synth.frame_stride_fp32(F)
    rng = np.random.default_rng(n + F)
    idx = synth.wiring(rng, I, O, n); W = synth.lut_tables(rng, O, n)
    x = synth.uniform_frames(rng, I, F, stride); dy = synth.normal_frames(rng, O, F, stride)
    v = oracle.stochastic_lut_forward(n, x, idx, W, F, input_binary=True, simd=False)[:, :F].astype(np.float64)
    mean, rstd = v.mean(axis=1), 1.0 / np.sqrt(v.var(axis=1) + 1e-5)
    t = (v - mean[:, None]) * rstd[:, None] + 0.5                  # gamma 1: about two frames in three lie outside
    closed = (t < -1e-3) | (t > 1.001)
    assert 0.2 < closed.mean() < 0.95
    poisoned = dy.copy()
    poisoned[:, :F][closed] = rng.choice(np.array([np.inf, -np.inf, np.nan, 3.0e38], np.float32), int(closed.sum()))
    dy[:, :F][closed] = 0.0
    d_x, d_idx, d_W = dev(x), dev(idx), dev(W)
    rev = ops.reverse_table(d_idx, I)
    got = []
    for g in (dy, poisoned):
        dW = dev(np.zeros_like(W))
        dx = ops.differentiable_lut_backward(n, d_x, dev(g), d_idx, d_W, dW, F, dev(mean.astype(np.float32)), dev(rstd.astype(np.float32)), rev, gamma=1.0)
        got.append((host(dx)[:, :F], host(dW)))
    assert np.isfinite(got[1][0]).all() and all(np.array_equal(a, b) for a, b in zip(*got))


def test_corner_values_beyond_4_gib():
    """2^24 + 64 nodes of six inputs: their corner values do not fit one buffer of 32-bit offsets, while dy and the indices do"""
    import torch
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    n, I, O, F = 6, 1 << 16, (1 << 24) + 64, 32
    gen = torch.Generator(device="cuda"); gen.manual_seed(4)
    idx = (torch.arange(n * O, dtype=torch.int32, device="cuda") % I).reshape(O, n)
    link = torch.arange(I, dtype=torch.int32, device="cuda")[:, None] + I * torch.arange((n * O + I - 1) // I, dtype=torch.int32, device="cuda")[None, :]
    rev = torch.cat([(link < n * O).sum(dim=1, dtype=torch.int32)[:, None], torch.where(link < n * O, link, 0)], dim=1).contiguous()
    x = torch.randint(-(1 << 31), 1 << 31, (I, 1), device="cuda", generator=gen).to(torch.int32)
    W = torch.rand((O, 1 << n), device="cuda", generator=gen)
    dy = torch.randn((O, F), device="cuda", generator=gen)
    dW = torch.zeros_like(W)
    # input values 0 and 1: a corner value is a table entry, and entry p of the table gradient the sum at corner p alone
    dx = ops.bit_stochastic_lut_backward(n, x, dy, idx, W, dW, F, rev, bias=0.5)
    base = torch.arange(O, device="cuda") << n
    for f in (0, 17, 31):
        bit = ((x[:, 0] >> f) & 1).long()
        corner = sum(bit[idx[:, k].long()] << k for k in range(n))
        want = torch.zeros(I, dtype=torch.float64, device="cuda")
        for k in range(n):
            slope = W.view(-1)[base + (corner | (1 << k))] - W.view(-1)[base + (corner & ~(1 << k))]
            want.index_add_(0, idx[:, k].long(), slope.double() * dy[:, f].double())
        assert_bwd(host(dx[:, f]), host(want), "dx of frame %d" % f)
    for first in (0, O - 1000):
        bits = (x[idx[first:first + 1000].long(), 0][:, :, None] >> torch.arange(F, device="cuda")) & 1
        corner = sum(bits[:, k].long() << k for k in range(n))
        want = torch.zeros((1000, 1 << n), dtype=torch.float64, device="cuda").scatter_add_(1, corner, dy[first:first + 1000].double())
        assert_bwd(host(dW[first:first + 1000]), host(want), "dW")


def test_corner_sums_of_long_skewed_rows():
    """Rows of 65536 frames whose inputs are nearly always set, in one slab (2000 nodes): a lane adds most of its 1024 frames into one bin.  rms error
    against 64 bits relative to a node's largest entry, by a model in fp32: 6.4e-8 in slabs of at most 4096 frames, 1.6e-7 as one chain."""
    import torch
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    I, O, F, n = 8, 2000, 65536, 6
    rng = np.random.default_rng(8)
    gen = torch.Generator(device="cuda"); gen.manual_seed(8)
    idx = synth.wiring(rng, I, O, n)
    set_ = rng.random((I, F)) < 0.98
    d_idx, d_W = dev(idx), dev(synth.lut_tables(rng, O, n))
    dy = torch.randn((O, F), device="cuda", generator=gen)
    dW = torch.zeros_like(d_W)
    # input values 0 and 1: entry p of the gradient is the sum at corner p alone
    ops.bit_stochastic_lut_backward(n, dev(synth.pack_bits(set_.astype(np.uint8), F // 32)), dy, d_idx, d_W, dW, F, ops.reverse_table(d_idx, I), bias=0.5)
    some = torch.arange(0, O, 20, device="cuda")
    bits, rows = dev(set_.astype(np.int64)), d_idx[some].long()
    corner = sum(bits[rows[:, k]] << k for k in range(n))
    want = torch.stack([torch.where(corner == p, dy[some].double(), 0.0).sum(dim=1) for p in range(1 << n)], dim=1)
    e = (dW[some].double() - want) / want.abs().amax(dim=1, keepdim=True)
    rms = float((e * e).mean().sqrt())
    print("rms %.2e" % rms)
    assert rms <= 9e-8


@pytest.mark.parametrize("n", [5, 6])
@pytest.mark.parametrize("frames", [20485, 40965])
def test_a_discarded_gradient_in_long_passes(n, frames):
    """the same where a wavefront of the dx kernel takes two (20485) and four (40965) groups of 256 frames: the launch has workgroups enough"""
    test_a_discarded_gradient_may_hold_anything(n, (216, 36, frames, 0))


# a list of exactly as many items as wavefronts share it, one more, one less; sixteen and four wavefronts; a short list among long ones; two groups of
# 256 frames per wavefront
@pytest.mark.parametrize("shape", [(7, 17, 2000), (7, 19, 1100), (12, 31, 1500), (12, 67, 1300), (40, 700, 6200), (9, 40, 90000)])
def test_shared_lists(shape):
    test_corner_backward(6, shape + (0,))


@pytest.mark.parametrize("n, shape", [(6, (7, 17, 5000)), (6, (12, 67, 4500)), (4, (9, 150, 4200)), (6, (40, 700, 4100))])
def test_shared_lists_of_real_valued_inputs(n, shape):
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    I, O, F = shape
    stride = synth.frame_stride_fp32(F)
    rng = np.random.default_rng(O)
    idx = synth.wiring(rng, I, O, n); W = synth.lut_tables(rng, O, n)
    x = synth.uniform_frames(rng, I, F, stride); dy = synth.normal_frames(rng, O, F, stride)
    dx_ref, dW_ref = oracle.stochastic_lut_backward(n, x, dy, idx, W, F)
    d_idx, dW = dev(idx), dev(np.zeros_like(W))
    dx = ops.stochastic_lut_backward(n, dev(x), dev(dy), d_idx, dev(W), dW, F, ops.reverse_table(d_idx, I))
    assert_bwd(host(dx)[:, :F], dx_ref[:, :F], "dx"); assert_bwd(host(dW), dW_ref, "dW")


# lists of 400 items and more in fewer workgroups than compute units, whose wavefronts take consecutive items: plain layers, and (the last two) batch-norm
@pytest.mark.parametrize("n, shape", [(6, (8, 560, 300)), (3, (7, 1000, 70)), (6, (40, 4750, 300)), (5, (64, 9100, 33))])
def test_long_lists_in_few_workgroups(n, shape):
    test_corner_backward(n, shape + (0,))


# the largest frame counts of the forms that request all frames at once, one more, rows that hold no whole groups of four; enough nodes for every wavefront
@pytest.mark.parametrize("n", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("shape", [(30, 33, 1024, 0), (30, 33, 1023, 1023), (30, 33, 1025, 1025), (30, 33, 2048, 0), (9, 700, 60, 0), (1600, 41, 700, 703)])
def test_sums_of_one_slab(n, shape):
    test_corner_backward(n, shape)
