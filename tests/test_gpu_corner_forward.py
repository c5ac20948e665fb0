"""GPU parity of the forward pass over two-valued inputs that forms the corner indices of 32 frames per lane, at the sizes where it has edges:
last words, blocks of 2048 frames, one to sixteen wavefronts per node, the largest one-launch training pass, row pitches of any kind."""
import numpy as np
import pytest

import oracle
from binarybrain_amd import synth
from util import assert_fwd, dev, host

pytestmark = pytest.mark.gpu

# inputs, nodes, frames, row pitch of the fp32 output (0: the frame buffer's), row pitch of the packed input (0: the frame buffer's)
SHAPES = [(9, 5, 1025, 0, 0), (16, 9, 2047, 2047, 67), (12, 70, 2048, 0, 0), (7, 3, 2049, 2051, 65), (40, 33, 4097, 0, 131), (8, 6, 8193, 8193, 0),
          (11, 2, 32769, 0, 0), (6, 3, 49152, 0, 0), (6, 5, 49153, 49153, 1537), (30, 40, 55000, 0, 0)]


# few nodes, whose output several workgroups share: two blocks and more, remainders of the shares, one to sixteen wavefronts per node
SHAPES += [(9, 130, 2049, 0, 0), (7, 60, 6145, 6145, 0), (12, 100, 10241, 0, 0), (6, 24, 33800, 0, 0), (8, 90, 40961, 40963, 0)]


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("shape", SHAPES)
def test_corner_forward(n, shape):
    import torch
    from binarybrain_amd import ops
    I, O, F, stride, words = shape
    stride, words = stride or synth.frame_stride_fp32(F), words or synth.frame_stride_bit(F)
    rng = np.random.default_rng(10 * n + F)
    idx = synth.wiring(rng, I, O, n); W = rng.random((O, 1 << n), dtype=np.float32)
    x = synth.uniform_frames(rng, I, F)
    bits = (x[:, :F] > 0.5).astype(np.uint8)
    xb = np.full((I, words), -1, np.int32)                        # what lies behind the frames enters nothing
    nw = (F + 31) // 32
    xb[:, :nw] = synth.pack_bits(bits, nw)
    if F & 31: xb[:, nw - 1] |= np.int32(-1) << np.int32(F & 31)
    v = oracle.bit_stochastic_lut_forward(n, xb, idx, W, F, stride, 0)[:, :F]
    d_xb, d_idx, d_W = dev(xb), dev(idx), dev(W)
    assert_fwd(host(ops.bit_stochastic_lut_forward(n, d_xb, d_idx, d_W, F, stride, 0))[:, :F], v, "fp32 output")
    gamma, beta = 0.3, 0.45

    def check(y, mean, rstd):
        m, r = host(mean).astype(np.float64), host(rstd).astype(np.float64)
        assert np.allclose(m, v.mean(axis=1, dtype=np.float64), rtol=1e-5)
        assert np.allclose(r, 1 / np.sqrt(np.maximum(v.var(axis=1, dtype=np.float64), 1e-5)), rtol=2e-4)
        t = (v - m[:, None]) * r[:, None] * gamma + beta
        assert not np.any((y != (t > 0.5)) & (np.abs(t - 0.5) > 1e-5))

    stats = lambda: (torch.zeros(O, device="cuda"), torch.ones(O, device="cuda"))          # noqa: E731
    rm, rv = stats()
    y, mean, rstd = ops.bit_differentiable_lut_forward_training(n, d_xb, d_idx, d_W, F, rm, rv, gamma=gamma, beta=beta, momentum=0.5)
    check(synth.unpack_bits(host(y), y.shape[1] * 32)[:, :F], mean, rstd)
    assert np.allclose(host(rm), 0.5 * host(mean), rtol=1e-6) and np.allclose(host(rv), 0.5 + 0.5 / host(rstd) ** 2, rtol=1e-4)
    for kw in ({}, {"packed": ops.packed_input_buffer(I, F)}):
        copy = ops.packed_input_buffer(O, F); copy.fill_(-1)
        y, mean, rstd = ops.differentiable_lut_forward_training(n, dev(x), d_idx, d_W, F, *stats(), gamma=gamma, beta=beta, packed_out=copy, **kw)
        check(host(y)[:, :F], mean, rstd)
        assert np.array_equal(synth.unpack_bits(host(copy), copy.shape[1] * 32)[:, :F], host(y)[:, :F].astype(np.uint8)) and not host(copy)[:, nw:].any()


@pytest.mark.parametrize("nodes,frames", [(24, 33800), (100, 2049), (130, 33800)])
def test_running_statistics_of_shared_nodes_move_once(nodes, frames):
    """However many workgroups share a node's fp32 output, its running statistics take one step per call."""
    import torch
    from binarybrain_amd import ops
    rng = np.random.default_rng(frames)
    idx = synth.wiring(rng, 12, nodes, 6); W = rng.random((nodes, 64), dtype=np.float32)
    d_x, d_idx, d_W = dev(synth.uniform_frames(rng, 12, frames)), dev(idx), dev(W)
    rm, rv = torch.full((nodes,), 0.25, device="cuda"), torch.ones(nodes, device="cuda")
    want_m, want_v = host(rm), host(rv)
    for _ in range(3):
        _, mean, rstd = ops.differentiable_lut_forward_training(6, d_x, d_idx, d_W, frames, rm, rv, gamma=0.3, beta=0.5, momentum=0.75)
        want_m, want_v = 0.75 * want_m + 0.25 * host(mean), 0.75 * want_v + 0.25 / host(rstd) ** 2
    assert np.allclose(host(rm), want_m, rtol=1e-5) and np.allclose(host(rv), want_v, rtol=1e-4)
