"""GPU parity of BinaryLutN<N> packed inference for N = 2 .. 6 (bbhip_bit_BinaryLutN_Forward): bit-exact against the CPU oracle and
against vectors written by the reference's own class; equal to StochasticLut<N> with a 0 / 1 table on the same bits."""
import os

import numpy as np
import pytest

import oracle
from binarybrain_amd import synth
from util import dev, host

pytestmark = pytest.mark.gpu
GOLD = np.load(os.path.join(os.path.dirname(os.path.abspath(__file__)), "golden", "binary_lutn.npz"))


@pytest.fixture(scope="module")
def ops():
    from binarybrain_amd import ops as o
    return o


def tables(rng, O, n):
    if n == 6:
        return synth.truth_tables(rng, O)
    return rng.integers(0, 1 << (1 << n), (O, 1), dtype=np.int64).astype(np.uint32).view(np.int32)


@pytest.mark.parametrize("n", [2, 3, 4, 5, 6])
@pytest.mark.parametrize("shape", [(16, 16, 32), (70, 33, 1000), (8, 5, 7), (6, 1, 1), (300, 1000, 64 * 32 * 3 + 5), (64, 130, 131072 + 37)])
def test_bit_exact(ops, n, shape):
    I, O, F = shape
    rng = np.random.default_rng(I + O + F + n)
    stride = synth.frame_stride_bit(F)
    idx = synth.wiring(rng, I, O, n); T = tables(rng, O, n)
    xb = synth.bernoulli_bits(rng, I, F, stride)
    y = ops.binary_lutn_forward(n, dev(xb), dev(idx), dev(T), F)
    assert np.array_equal(host(y), oracle.binary_lutn_forward(n, xb, idx, T, F))        # padding bits and words are zero on both sides


@pytest.mark.parametrize("n", [2, 3, 4, 5])
@pytest.mark.parametrize("nodes", [85, 175, 176])
def test_several_nodes_per_wavefront(ops, n, nodes):
    """201 units of 128 words: enough workgroups for two (85) and four (175, 176) nodes per wavefront, the last ones with nodes to skip or none"""
    I, F = 37, 200 * 4096 + 33
    rng = np.random.default_rng(nodes + n)
    idx = synth.wiring(rng, I, nodes, n); T = tables(rng, nodes, n)
    xb = synth.bernoulli_bits(rng, I, F, synth.frame_stride_bit(F))
    y = ops.binary_lutn_forward(n, dev(xb), dev(idx), dev(T), F)
    assert np.array_equal(host(y), oracle.binary_lutn_forward(n, xb, idx, T, F))


@pytest.mark.parametrize("n", [2, 5])
def test_rows_too_far_apart_for_one_extent(ops, n):
    """a pitch of 2^27 words and more takes one node per wavefront, with 64-bit row offsets"""
    import torch
    I, O, F, pitch = 6, 5, 5000, (1 << 27) + 64
    rng = np.random.default_rng(n)
    idx = dev(synth.wiring(rng, I, O, n)); T = dev(tables(rng, O, n))
    xb = dev(synth.bernoulli_bits(rng, I, F, synth.frame_stride_bit(F)))
    far = torch.zeros((I, pitch), dtype=torch.int32, device="cuda")
    far[:, :xb.shape[1]] = xb
    words = (F + 31) // 32
    y = ops.binary_lutn_forward(n, far, idx, T, F)
    assert torch.equal(y[:, :words], ops.binary_lutn_forward(n, xb, idx, T, F)[:, :words])


def _wide_rows(bits, pitch):
    """the rows of `bits` at another pitch, and memory of that shape that holds anything for the call's output"""
    import torch
    wide = torch.zeros((bits.shape[0], pitch), dtype=torch.int32, device="cuda")
    wide[:, :bits.shape[1]] = bits
    return wide


# padding that the wavefront of a row's end writes (up to 4096 words), one word more, and far more; nodes to skip in the last wavefront, and none
@pytest.mark.parametrize("n", [2, 5, 6])
@pytest.mark.parametrize("nodes", [5, 64])
@pytest.mark.parametrize("frames, padding", [(70, 1), (70, 4096), (70, 4097), (4096 * 3, 5000), (4096 * 3 + 1, 100003)])
def test_padding_of_far_rows_is_zero(ops, n, nodes, frames, padding):
    import torch
    I, words = 9, (frames + 31) // 32
    rng = np.random.default_rng(frames + n)
    idx = dev(synth.wiring(rng, I, nodes, n)); T = dev(tables(rng, nodes, n))
    xb = dev(synth.bernoulli_bits(rng, I, frames, words))
    far = _wide_rows(xb, words + padding)
    dirty = torch.full((nodes, words + padding), -1, dtype=torch.int32, device="cuda")
    del dirty                                       # (its memory is what the call's output is made of)
    y = ops.binary_lutn_forward(n, far, idx, T, frames)
    assert torch.equal(y[:, :words], ops.binary_lutn_forward(n, xb, idx, T, frames)) and not y[:, words:].any()
    W = torch.rand((nodes, 1 << n), device="cuda")
    dirty = torch.full((nodes, words + padding), -1, dtype=torch.int32, device="cuda")
    del dirty
    y = ops.bit_bit_stochastic_lut_forward(n, far, idx, W, frames)
    assert torch.equal(y[:, :words], ops.bit_bit_stochastic_lut_forward(n, xb, idx, W, frames)) and not y[:, words:].any()


def test_padding_of_the_farthest_rows(ops):
    """a pitch of 2^31 - 1 words: no word number that leaves the range of an int"""
    import torch
    frames, pitch = 70, (1 << 31) - 1
    x = torch.zeros((1, pitch), dtype=torch.int32, device="cuda")
    x[0, :3] = torch.tensor([0x12345678, -3, 63], dtype=torch.int32)
    idx = torch.zeros((1, 2), dtype=torch.int32, device="cuda")
    dirty = torch.full((1, pitch), -1, dtype=torch.int32, device="cuda")
    del dirty
    y = ops.binary_lutn_forward(2, x, idx, torch.full((1, 1), 8, dtype=torch.int32, device="cuda"), frames)      # x AND x
    assert torch.equal(y[0, :3], x[0, :3])
    assert all(not part.any() for part in y[0, 3:].split(1 << 28))
    del x, y
    torch.cuda.empty_cache()


def test_reference_vectors_on_gpu(ops):
    for k in range(int(GOLD["count"][0])):
        p = "c%d_" % k
        n, I, O, F = [int(v) for v in GOLD[p + "meta"]]
        y = ops.binary_lutn_forward(n, dev(GOLD[p + "xbits"]), dev(GOLD[p + "idx"]), dev(GOLD[p + "table"]), F)
        assert np.array_equal(host(y), GOLD[p + "y"]), (k, n)


@pytest.mark.parametrize("n", [2, 3, 4, 5])
def test_equals_the_stochastic_lut_on_bits(ops, n):
    """the same layer as a StochasticLut<n> with W in {0, 1} and bit inputs mapped to 0 / 1 (bias 0.5): y > 0.5 reproduces the table"""
    rng = np.random.default_rng(60 + n)
    I, O, F = 40, 24, 4096 + 70
    idx = synth.wiring(rng, I, O, n); T = tables(rng, O, n)
    xb = synth.bernoulli_bits(rng, I, F, synth.frame_stride_bit(F))
    W = np.array([[(int(np.uint32(T[o, 0])) >> b) & 1 for b in range(1 << n)] for o in range(O)], np.float32)
    y = ops.binary_lutn_forward(n, dev(xb), dev(idx), dev(T), F)
    yb = ops.bit_bit_stochastic_lut_forward(n, dev(xb), dev(idx), dev(W), F, bias=0.5)
    assert np.array_equal(synth.unpack_bits(host(yb), F), synth.unpack_bits(host(y), F))


def test_rejected_arguments(ops):
    import torch
    x = torch.zeros((8, 8), dtype=torch.int32, device="cuda")
    idx = torch.zeros((4, 7), dtype=torch.int32, device="cuda")
    with pytest.raises(RuntimeError):
        from binarybrain_amd.capi import lib, check
        from binarybrain_amd.ops import ptr
        check(lib().bbhip_bit_BinaryLutN_Forward(7, ptr(x), ptr(x), ptr(idx), ptr(idx), 4, 64, 8, None))
