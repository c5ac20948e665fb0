"""GPU parity of StochasticLut training steps whose backward pass is one launch, at its edges: wavefront steps and units, work lists shared by four and
by sixteen wavefronts, the largest call that it serves and the first that goes to the kernels beyond."""
import numpy as np
import pytest

import oracle
from binarybrain_amd import synth
from util import assert_bwd, assert_fwd, dev, host

pytestmark = pytest.mark.gpu

SHAPES = [(9, 5, 1), (16, 9, 64), (7, 33, 65), (40, 6, 256), (12, 13, 257), (1100, 30, 300), (260, 11, 2047), (70, 1200, 130), (40, 3000, 20),
          (300, 640, 2048), (300, 641, 2048), (27, 16, 2049), (216, 36, 3900), (27, 4, 4096), (27, 4, 4097), (27, 36, 30000), (7, 1, 70000)]


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("shape", SHAPES)
def test_small_plain_training(n, shape):
    import torch
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    I, O, F = shape
    rng = np.random.default_rng(10 * n + F)
    stride = synth.frame_stride_fp32(F)
    idx = synth.wiring(rng, I, O, n); W = synth.lut_tables(rng, O, n)
    x = synth.uniform_frames(rng, I, F, stride, -0.1, 1.1); dy = synth.normal_frames(rng, O, F, stride)
    binarize = bool(n & 1)
    y_ref = oracle.stochastic_lut_forward(n, x, idx, W, F, input_binary=False, lut_binarize=binarize)
    dx_ref, dW_ref = oracle.stochastic_lut_backward(n, x, dy, idx, W, F, input_binary=False, lut_binarize=binarize)
    x[:, F:] = np.nan; dy[:, F:] = np.nan           # what lies behind the frames enters nothing
    d_x, d_dy, d_idx, d_W = dev(x), dev(dy), dev(idx), dev(W)
    rev = ops.reverse_table(d_idx, I)
    y = ops.stochastic_lut_forward(n, d_x, d_idx, d_W, F, input_binary=False, lut_binarize=binarize)
    assert_fwd(host(y)[:, :F], y_ref[:, :F])
    got = []
    for overwrite in (False, True, True):
        dW = torch.full((O, 1 << n), 0.0 if not overwrite else np.nan, device="cuda")
        dx = ops.stochastic_lut_backward(n, d_x, d_dy, d_idx, d_W, dW, F, rev, input_binary=False, lut_binarize=binarize, overwrite_dw=overwrite)
        assert_bwd(host(dx)[:, :F], dx_ref[:, :F])
        assert_bwd(host(dW), dW_ref)
        got.append((host(dx)[:, :F], host(dW)))
    assert all(np.array_equal(a, b) for g in got[1:] for a, b in zip(got[0], g))        # the same bits each time


@pytest.mark.parametrize("n, bound", [(4, 7.0e-8), (5, 6.5e-8), (6, 6.0e-8)])
@pytest.mark.parametrize("frames", [1000, 2048, 4000])
def test_table_gradient_rounding(n, bound, frames):
    """The sums over frames round no worse than multiply-adds per lane in slabs do.  rms error against 64 bits relative to a node's largest entry,
    of those multiply-adds by a model of their order in fp32: 6.9e-8, 5.9e-8, 5.1e-8 for four, five, six inputs; what rounds every term to
    the size of sums without a factor 1 - x, or adds a wavefront's share in one chain, is at 1.0e-7 and above for six."""
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    I, O = 64, 200
    rng = np.random.default_rng(n + frames)
    stride = synth.frame_stride_fp32(frames)
    idx = synth.wiring(rng, I, O, n); W = synth.lut_tables(rng, O, n)
    x = synth.uniform_frames(rng, I, frames, stride); dy = synth.normal_frames(rng, O, frames, stride)
    d_idx = dev(idx)
    dW = dev(np.zeros_like(W))
    ops.stochastic_lut_backward(n, dev(x), dev(dy), d_idx, dev(W), dW, frames, ops.reverse_table(d_idx, I))
    x64, want = x[:, :frames].astype(np.float64), np.zeros((O, 1 << n))
    for o in range(O):
        p = dy[o:o + 1, :frames].astype(np.float64)
        for k in range(n):
            p = np.concatenate([p * (1.0 - x64[idx[o, k]]), p * x64[idx[o, k]]])
        want[o] = p.sum(axis=1)
    e = (host(dW) - want) / np.abs(want).max(axis=1, keepdims=True)
    rms = float(np.sqrt((e * e).mean()))
    print("n=%d frames=%d rms %.2e" % (n, frames, rms))
    assert rms <= bound


# four wavefront-steps per unit as four consecutive frames per lane: last groups of one to four frames, pitches that put dx rows off 16 bytes, and rows too
# short for whole groups (pitch = frames); own lists and shared ones
@pytest.mark.parametrize("n", [2, 4, 6])
@pytest.mark.parametrize("shape", [(1030, 300, 257, 0), (1030, 300, 510, 513), (700, 200, 511, 511), (520, 160, 768, 768), (300, 700, 1021, 0), (300, 700, 1023, 1025)])
def test_four_frames_per_lane(n, shape):
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    I, O, F, stride = shape
    stride = stride or synth.frame_stride_fp32(F)
    rng = np.random.default_rng(F + n)
    idx = synth.wiring(rng, I, O, n); W = synth.lut_tables(rng, O, n)
    x = synth.uniform_frames(rng, I, F, stride, -0.1, 1.1); dy = synth.normal_frames(rng, O, F, stride)
    dx_ref, dW_ref = oracle.stochastic_lut_backward(n, x, dy, idx, W, F)
    x[:, F:] = np.nan; dy[:, F:] = np.nan           # what lies behind the frames enters nothing
    d_idx, dW = dev(idx), dev(np.zeros_like(W))
    dx = ops.stochastic_lut_backward(n, dev(x), dev(dy), d_idx, dev(W), dW, F, ops.reverse_table(d_idx, I))
    assert_bwd(host(dx)[:, :F], dx_ref[:, :F], "dx"); assert_bwd(host(dW), dW_ref, "dW")
