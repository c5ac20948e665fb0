"""The one-launch backward pass of small layers over two-valued inputs against the oracle, where it can go wrong: last frames of words, of groups of
four and of its forms of 256, 512 and 1024 frames; rows that hold no whole groups of four; lists shared by a workgroup and not; empty lists and lists
of a share of one to twenty; with the prepared tables of the forward call and without."""
import numpy as np
import pytest

import oracle
from binarybrain_amd import capi, synth
from util import assert_bwd, dev, host

pytestmark = pytest.mark.gpu

# inputs, nodes, frames, row pitch of dy and dx (0: the frame buffer's)
SHAPES = [(9, 5, 5, 0), (40, 70, 31, 31), (40, 70, 255, 255), (40, 70, 256, 0), (40, 70, 257, 259), (300, 200, 511, 511), (300, 200, 512, 0),
          (90, 60, 513, 513), (90, 60, 1023, 1023), (90, 60, 1024, 0), (2100, 300, 64, 0), (2100, 300, 251, 251), (30, 300, 200, 0), (16, 40, 33, 0)]


@pytest.mark.parametrize("n", [2, 3, 5, 6])
@pytest.mark.parametrize("shape", SHAPES)
def test_small_backward(n, shape):
    import ctypes as C
    import torch
    from binarybrain_amd import ops
    ops.set_dx_mode(0)
    I, O, F, stride = shape
    stride = stride or synth.frame_stride_fp32(F)
    rng = np.random.default_rng(10 * n + F)
    idx = synth.wiring(rng, I, O, n); W = synth.lut_tables(rng, O, n)
    x = synth.uniform_frames(rng, I, F, synth.frame_stride_fp32(F)); dy = synth.normal_frames(rng, O, F, stride)
    xb = np.zeros((I, synth.frame_stride_bit(F)), np.int32)
    xb[:, :(F + 31) // 32] = synth.pack_bits((x[:, :F] > 0.5).astype(np.uint8), (F + 31) // 32)
    _, mean, rstd, _, _ = oracle.differentiable_lut_forward_training(n, x, idx, W, F, np.zeros(O, np.float32), np.ones(O, np.float32))
    xs = np.ascontiguousarray(x[:, :stride]) if stride <= x.shape[1] else np.pad(x, ((0, 0), (0, stride - x.shape[1])))
    want_bn = oracle.differentiable_lut_backward(n, xs, dy, idx, W, F, mean, rstd)
    want_plain = oracle.stochastic_lut_backward(n, xs, dy, idx, W, F, input_binary=True, simd=False)
    dy[:, F:] = np.nan                              # what lies behind the frames enters nothing
    d_xb, d_dy, d_idx, d_W = dev(xb), dev(dy), dev(idx), dev(W)
    rev = ops.reverse_table(d_idx, I)
    lib = capi.lib()
    got = []
    for tables in (ops.prepared_tables_buffer(n, O), None):
        if tables is not None:
            ops.bit_differentiable_lut_forward_training(n, d_xb, d_idx, d_W, F, dev(np.zeros(O, np.float32)), dev(np.ones(O, np.float32)), tables=tables)
        dW = torch.full_like(d_W, 0.25)
        lib.bbhip_KernelTimer_Enable(1)
        dx = ops.bit_differentiable_lut_backward(n, d_xb, d_dy, d_idx, d_W, dW, F, dev(mean), dev(rstd), rev, tables=tables)
        lib.bbhip_KernelTimer_Enable(0)
        ms, dx_launches = C.c_float(), C.c_int()
        capi.check(lib.bbhip_KernelTimer_Read(3, C.byref(ms), C.byref(dx_launches)))
        assert dx_launches.value == 0               # no dx launch of its own
        assert_bwd(host(dx)[:, :F], want_bn[0][:, :F], "dx"); assert_bwd(host(dW) - 0.25, want_bn[1], "dW")
        got.append((host(dx)[:, :F], host(dW)))
    assert all(np.array_equal(a, b) for a, b in zip(*got))
    dW = torch.zeros_like(d_W)
    dx = ops.bit_stochastic_lut_backward(n, d_xb, d_dy, d_idx, d_W, dW, F, rev)
    assert_bwd(host(dx)[:, :F], want_plain[0][:, :F], "plain dx"); assert_bwd(host(dW), want_plain[1], "plain dW")


@pytest.mark.parametrize("frames,pitch", [(1, 1), (63, 63), (64, 0), (255, 255), (256, 0)])
def test_lists_shared_by_sixteen_wavefronts(frames, pitch):
    """few inputs with long lists: 0, 1, 15, 16, 17, 77, 78 and 80 consumers, so that wavefronts of one list have none, one or five items"""
    import torch
    from binarybrain_amd import ops
    n, counts = 6, [0, 1, 15, 16, 17, 80, 77, 80, 78, 80, 0, 80, 80, 80]
    I, O, F = len(counts), sum(counts) // n, frames
    assert sum(counts) == O * n
    S, rng = pitch or synth.frame_stride_fp32(F), np.random.default_rng(frames)
    slots = np.repeat(np.arange(I, dtype=np.int32), counts)
    idx = np.ascontiguousarray(rng.permutation(slots).reshape(O, n)); W = synth.lut_tables(rng, O, n)
    x = np.zeros((I, S), np.float32); x[:, :F] = rng.random((I, F)) > 0.5
    xb = np.zeros((I, synth.frame_stride_bit(F)), np.int32)
    xb[:, :(F + 31) // 32] = synth.pack_bits(x[:, :F].astype(np.uint8), (F + 31) // 32)
    dy = synth.normal_frames(rng, O, F, S)
    _, mean, rstd, _, _ = oracle.differentiable_lut_forward_training(n, x, idx, W, F, np.zeros(O, np.float32), np.ones(O, np.float32))
    want_bn = oracle.differentiable_lut_backward(n, x, dy, idx, W, F, mean, rstd)
    want_plain = oracle.stochastic_lut_backward(n, x, dy, idx, W, F, input_binary=True, simd=False)
    d_xb, d_dy, d_idx, d_W = dev(xb), dev(dy), dev(idx), dev(W)
    rev = ops.reverse_table(d_idx, I)
    dW = torch.zeros_like(d_W)
    dx = ops.bit_stochastic_lut_backward(n, d_xb, d_dy, d_idx, d_W, dW, F, rev)
    assert_bwd(host(dx)[:, :F], want_plain[0][:, :F], "plain dx"); assert_bwd(host(dW), want_plain[1], "plain dW")
    tables = ops.prepared_tables_buffer(n, O)
    ops.bit_differentiable_lut_forward_training(n, d_xb, d_idx, d_W, F, dev(np.zeros(O, np.float32)), dev(np.ones(O, np.float32)), tables=tables)
    for t in (tables, None):
        dW = torch.zeros_like(d_W)
        dx = ops.bit_differentiable_lut_backward(n, d_xb, d_dy, d_idx, d_W, dW, F, dev(mean), dev(rstd), rev, tables=t)
        assert not host(dx)[[0, 10], :F].any()
        if F > 1:                       # (a single frame is its own mean: rstd is that of rounding, and the gradient through it has no digits)
            assert_bwd(host(dx)[:, :F], want_bn[0][:, :F], "dx"); assert_bwd(host(dW), want_bn[1], "dW")
