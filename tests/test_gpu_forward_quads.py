"""GPU parity of the forward pass over two-valued inputs of up to 1024 frames (four frames per lane), at the sizes where it has edges: passes of 256 frames, one
to four wavefronts per node or one that makes all passes, last words, rows that hold no whole groups of four, packed copies and padding."""
import numpy as np
import pytest

import oracle
from binarybrain_amd import synth
from util import assert_fwd, dev, host

pytestmark = pytest.mark.gpu

# inputs, nodes, frames, row pitch of the fp32 rows (0: the frame buffer's), row pitch of packed rows (0: the frame buffer's)
SHAPES = [(9, 5, 1, 1, 1), (7, 3, 3, 0, 0), (40, 65, 33, 33, 2), (12, 70, 255, 255, 0), (16, 9, 256, 0, 9), (8, 6, 257, 259, 0), (30, 33, 512, 512, 0),
          (11, 1023, 513, 0, 17), (20, 1024, 1001, 1001, 0), (24, 1025, 511, 0, 16), (33, 1030, 769, 771, 0), (10, 1031, 1024, 0, 33)]


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("shape", SHAPES)
def test_forward_quads(n, shape):
    import torch
    from binarybrain_amd import ops
    I, O, F, stride, words = shape
    stride, words = stride or synth.frame_stride_fp32(F), words or synth.frame_stride_bit(F)
    rng = np.random.default_rng(10 * n + F)
    idx = synth.wiring(rng, I, O, n); W = rng.random((O, 1 << n), dtype=np.float32)
    x = synth.uniform_frames(rng, I, F, stride)
    x[:, F:] = np.nan                                             # what lies behind the frames enters nothing
    bits = (x[:, :F] > 0.5).astype(np.uint8)
    nw = (F + 31) // 32
    xb = np.full((I, words), -1, np.int32)
    xb[:, :nw] = synth.pack_bits(bits, nw)
    if F & 31: xb[:, nw - 1] |= np.int32(-1) << np.int32(F & 31)
    v = oracle.bit_stochastic_lut_forward(n, xb, idx, W, F, stride, 0)[:, :F]
    d_x, d_xb, d_idx, d_W = dev(x), dev(xb), dev(idx), dev(W)
    assert_fwd(host(ops.bit_stochastic_lut_forward(n, d_xb, d_idx, d_W, F, stride))[:, :F], v, "packed, plain")
    assert_fwd(host(ops.stochastic_lut_forward(n, d_x, d_idx, d_W, F, input_binary=True))[:, :F], v, "fp32, plain")
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
    assert not synth.unpack_bits(host(y), y.shape[1] * 32)[:, F:].any()
    assert np.allclose(host(rm), 0.5 * host(mean), rtol=1e-6) and np.allclose(host(rv), 0.5 + 0.5 / host(rstd) ** 2, rtol=1e-4)
    first = None
    for kw in ({}, {"packed": ops.packed_input_buffer(I, F)}):
        copy = ops.packed_input_buffer(O, F); copy.fill_(-1)
        W2 = d_W * 1.5 - 0.25
        tables = ops.prepared_tables_buffer(n, O).zero_()
        clamped = W2.clamp(0, 1)
        y, mean, rstd = ops.differentiable_lut_forward_training(n, d_x, d_idx, W2, F, *stats(), gamma=gamma, beta=beta, packed_out=copy, clamp_w=(0.0, 1.0), tables=tables, **kw)
        assert torch.equal(W2, clamped)
        assert np.array_equal(synth.unpack_bits(host(copy), copy.shape[1] * 32)[:, :F], host(y)[:, :F].astype(np.uint8)) and not host(copy)[:, nw:].any()
        got = (host(y)[:, :F], host(mean), host(rstd), host(tables))
        first = first or got
        assert all(np.array_equal(a, b) for a, b in zip(got, first))                       # the same bits with the hints and without
        if kw:
            assert np.array_equal(synth.unpack_bits(host(kw["packed"]), kw["packed"].shape[1] * 32)[:, :F], bits)
            y, mean, rstd = ops.differentiable_lut_forward_training(n, d_x, d_idx, W2, F, *stats(), gamma=gamma, beta=beta, packed_holds=True, **kw)
            assert np.array_equal(host(y)[:, :F], first[0]) and np.array_equal(host(mean), first[1])
    y, mean, rstd = ops.differentiable_lut_forward_training(n, d_x, d_idx, d_W, F, *stats(), gamma=gamma, beta=beta)
    check(host(y)[:, :F], mean, rstd)
    rm, rv = mean.clone(), (1 / rstd ** 2).contiguous()
    t = (v - host(rm)[:, None]) / np.sqrt(host(rv))[:, None] * gamma + beta
    y = host(ops.bit_differentiable_lut_forward_inference(n, d_xb, d_idx, d_W, F, rm, rv, gamma=gamma, beta=beta))
    y = synth.unpack_bits(y, y.shape[1] * 32)
    assert not np.any((y[:, :F] != (t > 0.5)) & (np.abs(t - 0.5) > 1e-4)) and not y[:, F:].any()
