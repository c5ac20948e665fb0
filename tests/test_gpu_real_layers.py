"""GPU parity of batch-norm training over real-valued inputs where one launch takes all frames of a node, at its edges: wavefront steps, wavefronts
per node, the largest calls that it serves and the first that go to the kernels beyond."""
import numpy as np
import pytest

import oracle
from binarybrain_amd import synth
from util import assert_bwd, assert_fwd, dev, host

pytestmark = pytest.mark.gpu

SHAPES = [(9, 5, 3), (16, 9, 64), (7, 33, 65), (40, 6, 256), (12, 13, 257), (30, 3, 511), (8, 70, 513), (10, 7, 1025), (50, 21, 2048), (6, 5, 2049), (9, 4, 4096),
          (11, 3, 4097)]


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("shape", SHAPES)
def test_real_valued_training(n, shape):
    import torch
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    I, O, F = shape
    rng = np.random.default_rng(100 * n + F)
    stride = synth.frame_stride_fp32(F)
    idx = synth.wiring(rng, I, O, n); W = synth.lut_tables(rng, O, n)
    x = synth.uniform_frames(rng, I, F, stride, -0.1, 1.1); dy = synth.normal_frames(rng, O, F, stride)
    y_ref, mean, rstd, rm_ref, rv_ref = oracle.differentiable_lut_forward_training(n, x, idx, W, F, np.zeros(O, np.float32), np.ones(O, np.float32), binary_mode=False)
    x[:, F:] = np.nan; dy[:, F:] = np.nan           # what lies behind the frames enters nothing
    d_x, d_dy, d_idx, d_W = dev(x), dev(dy), dev(idx), dev(W)
    rev = ops.reverse_table(d_idx, I)
    got = []
    for tables in (None, ops.prepared_tables_buffer(n, O)):
        rm, rv = torch.zeros(O, device="cuda"), torch.ones(O, device="cuda")
        y, m, r = ops.differentiable_lut_forward_training(n, d_x, d_idx, d_W, F, rm, rv, binary_mode=False, clamp_w=(-9.0, 9.0), tables=tables)
        assert np.allclose(host(m), mean, rtol=1e-4, atol=1e-6) and np.allclose(host(r), rstd, rtol=1e-3)
        assert np.allclose(host(rm), rm_ref, rtol=1e-4, atol=1e-6) and np.allclose(host(rv), rv_ref, rtol=1e-3)
        assert np.abs(host(y)[:, :F] - y_ref[:, :F]).max() <= 2e-4
        dx_ref, dW_ref = oracle.differentiable_lut_backward(n, x, dy, idx, W, F, mean, rstd, binary_mode=False)
        dW = torch.full((O, 1 << n), 0.25, device="cuda")
        dx = ops.differentiable_lut_backward(n, d_x, d_dy, d_idx, d_W, dW, F, dev(mean), dev(rstd), rev, binary_mode=False, tables=tables)
        if F > 4:                                   # (the gradient through the statistics of a frame or two is rounding alone)
            assert_bwd(host(dx)[:, :F], dx_ref[:, :F], "dx"); assert_bwd(host(dW) - 0.25, dW_ref, "dW")
        got.append((host(y)[:, :F], host(m), host(dx)[:, :F], host(dW)))
    assert all(np.array_equal(a, b) for a, b in zip(*got))


def test_scratch_arguments_of_the_backward_call_are_not_used():
    """66000 frames: more units than a wavefront adds up itself, so that dmean and dvar are formed by a launch of their own, in the library's scratch"""
    import torch
    from binarybrain_amd import ops
    from binarybrain_amd.capi import check, lib, ptr, stream_ptr
    ops.set_dx_mode(0)
    n, I, O, F = 6, 12, 5, 66000
    rng = np.random.default_rng(66)
    stride = synth.frame_stride_fp32(F)
    idx = synth.wiring(rng, I, O, n); W = synth.lut_tables(rng, O, n)
    x = synth.uniform_frames(rng, I, F, stride); dy = synth.normal_frames(rng, O, F, stride)
    _, mean, rstd, _, _ = oracle.differentiable_lut_forward_training(n, x, idx, W, F, np.zeros(O, np.float32), np.ones(O, np.float32), binary_mode=False)
    dx_ref, dW_ref = oracle.differentiable_lut_backward(n, x, dy, idx, W, F, mean, rstd, binary_mode=False)
    d_x, d_dy, d_idx, d_W, d_mean, d_rstd, dW = dev(x), dev(dy), dev(idx), dev(W), dev(mean), dev(rstd), dev(np.zeros_like(W))
    rev = ops.reverse_table(d_idx, I)
    dx = torch.empty((I, stride), device="cuda")
    tmp = torch.full((2, O), 7.0, device="cuda")
    check(lib().bbhip_fp32_DifferentiableLutN_Backward(n, ptr(d_x), ptr(d_dy), ptr(dx), None, ptr(d_idx), ptr(rev), ptr(d_W), ptr(dW), ptr(d_mean), ptr(d_rstd),
                                                      ptr(tmp[0]), ptr(tmp[1]), 0.3, 0.5, 0.25, rev.shape[1], I, O, F, stride, 0, 0, 0, 0, stream_ptr()))
    assert_bwd(host(dx)[:, :F], dx_ref[:, :F]); assert_bwd(host(dW), dW_ref)
    assert bool((tmp == 7.0).all())
    again = torch.zeros_like(dW)
    got = ops.differentiable_lut_backward(n, d_x, d_dy, d_idx, d_W, again, F, d_mean, d_rstd, rev, binary_mode=False)
    assert torch.equal(got[:, :F], dx[:, :F]) and torch.equal(again, dW)


# passes of four consecutive frames per lane: last groups of one to four frames, one lane and 64 lanes in the last pass, shared and own lists, rows of dx on 16
# bytes and not (pitch 8197, 4101), rows too short for whole groups (pitch = frames)
@pytest.mark.parametrize("n", [2, 4, 6])
@pytest.mark.parametrize("shape", [(600, 500, 8191, 0), (520, 400, 8193, 8197), (90, 700, 4100, 4101), (80, 300, 4354, 0), (520, 400, 8193, 8193), (530, 400, 7936, 7936)])
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
