"""Functional layer over the C ABI: torch device tensors in, torch device tensors out.

Every function is a direct call of one entry point of include/bbhip.h on the current torch stream.  Buffers follow
the FrameBuffer layout: ``[nodes, stride]`` float32 rows (stride >= frames) or ``[nodes, stride_words]`` int32 rows of
packed bits.  Nothing here has a CPU fallback: without the built library, or off a GPU, calls raise.

The calls go through the extension module built from csrc/ops_native.cpp (`native` below), which checks every tensor argument (device,
contiguous), allocates outputs and takes the current stream: what a call costs on the host bounds every pass over small layers.
"""
import numpy as np
import torch

from . import capi, synth
from .capi import check, lib, native, ptr, stream_ptr       # noqa: F401  (check, ptr, stream_ptr: for callers of the ctypes binding)


def set_dx_mode(mode):
    """0: deterministic dx, input-centric re-evaluation through the reverse table (default); 1: fp32 atomics;
    2: the reference's scheme (per-connection gradients in dx_tmp, summed through the reverse table)."""
    lib().bbhip_SetDxMode(int(mode))


def vector_clamp_(t, lo=0.0, hi=1.0):
    native.fp32_Vector_clamp(t, t, lo, hi, t.numel())
    return t


def vector_set_(t, value):
    native.fp32_Vector_set(t, value, t.numel())
    return t


def _out(dst, like):
    return torch.empty_like(like) if dst is None else dst


def vector_add_ex(src0, src1, a=1.0, b=1.0, c=0.0, out=None):
    """a * src0 + b * src1 + c"""
    dst = _out(out, src0)
    native.fp32_Vector_add_ex(dst, src0, src1, a, b, c, src0.numel())
    return dst


def vector_mul_ex(src0, src1, a=1.0, b=0.0, out=None):
    """a * src0 * src1 + b"""
    dst = _out(out, src0)
    native.fp32_Vector_mul_ex(dst, src0, src1, a, b, src0.numel())
    return dst


def vector_div_ex(src0, src1, a=1.0, b=0.0, c=1.0, d=0.0, out=None):
    """(a * src0 + b) / (c * src1 + d)"""
    dst = _out(out, src0)
    native.fp32_Vector_div_ex(dst, src0, src1, a, b, c, d, src0.numel())
    return dst


def vector_unary(name, src, out=None):
    """name in {"sqrt", "exp"}"""
    dst = _out(out, src)
    getattr(native, "fp32_Vector_" + name)(dst, src, src.numel())
    return dst


def vector_minmax(name, src0, src1, out=None):
    """name in {"min", "max"}; src1 is a tensor or a Python float (the *_v entry points)"""
    dst = _out(out, src0)
    if isinstance(src1, torch.Tensor):
        getattr(native, "fp32_Vector_" + name)(dst, src0, src1, src0.numel())
    else:
        getattr(native, "fp32_Vector_%s_v" % name)(dst, src0, float(src1), src0.numel())
    return dst


class AdamState:
    """Device-side tables of one parameter list for bbhip_fp32_OptimizerAdam, with the bias-correction products kept
    on the host as the reference does (include/bb/OptimizerAdam.h:104-110, 166-180)."""

    def __init__(self, params, grads, learning_rate=0.001, beta1=0.9, beta2=0.999):
        for tensor in (*params, *grads):
            if not tensor.is_cuda or not tensor.is_contiguous():
                raise capi.BbhipError("bbhip ops need contiguous device tensors")
        self.params, self.grads = list(params), list(grads)
        self.m = [torch.zeros_like(p) for p in params]
        self.v = [torch.zeros_like(p) for p in params]
        dev = params[0].device
        table = lambda ts: torch.tensor([t.data_ptr() for t in ts], dtype=torch.int64, device=dev)
        self.t_params, self.t_grads, self.t_m, self.t_v = table(self.params), table(self.grads), table(self.m), table(self.v)
        self.t_size = torch.tensor([p.numel() for p in params], dtype=torch.int32, device=dev)
        f32 = np.float32
        self.lr, self.beta1, self.beta2 = f32(learning_rate), f32(beta1), f32(beta2)
        self.b1, self.b2 = f32(beta1), f32(beta2)

    def lr_t(self):
        """the bias-corrected rate of the next step: lr * sqrt(1 - b2) / (1 - b1), every operation rounded to float"""
        return np.float32(native.adam_rate(self.lr, self.b1, self.b2))

    def step(self):
        native.fp32_OptimizerAdam(len(self.params), self.t_size, self.t_params, self.t_grads, self.t_m, self.t_v,
                                  self.lr_t(), self.beta1, self.beta2)
        self.b1 = self.b1 * self.beta1
        self.b2 = self.b2 * self.beta2

    def update(self):
        """Optimizer::Update of the reference = step, then the gradients set to zero (include/bb/Optimizer.h:31-35), in one launch."""
        native.fp32_OptimizerAdam_Update(len(self.params), self.t_size, self.t_params, self.t_grads, self.t_m, self.t_v,
                                         self.lr_t(), self.beta1, self.beta2)
        self.b1 = self.b1 * self.beta1
        self.b2 = self.b2 * self.beta2


BORDER_MODES = {"constant": 0, "reflect": 1, "reflect_101": 2, "replicate": 3, "wrap": 4}


def im2col_geometry(h, w, fh, fw, ys=1, xs=1, padding="valid"):
    """(oh, ow, y_offset, x_offset) of a filter fh x fw stepping by (ys, xs) (reference: include/bb/ConvolutionIm2Col.h:183-198)"""
    if padding == "valid":
        return ((h - fh + 1) + (ys - 1)) // ys, ((w - fw + 1) + (xs - 1)) // xs, 0, 0
    if padding != "same":
        raise capi.BbhipError("padding must be 'valid' or 'same'")
    return (h + ys - 1) // ys, (w + xs - 1) // xs, (fh - 1) // 2, (fw - 1) // 2


def _stride_for(frames, bit):
    return synth.frame_stride_bit(frames) if bit else synth.frame_stride_fp32(frames)


def im2col_forward(x, c, h, w, frames, fh, fw, ys=1, xs=1, padding="valid", border="reflect_101", border_value=0.0):
    """x [c*h*w, stride] float32 or packed int32 -> y [c*fh*fw, stride'] holding frames*oh*ow frames"""
    bit = x.dtype == torch.int32
    oh, ow, yo, xo = im2col_geometry(h, w, fh, fw, ys, xs, padding)
    of = frames * oh * ow
    y = (native.new_zero_bits if bit else native.new_rows)(x, c * fh * fw, _stride_for(of, bit))
    if bit:
        native.bit_Im2Col_Forward(x, y, xs, ys, xo, yo, frames, x.shape[1], w, h, c, ow, oh, y.shape[1], fw, fh, BORDER_MODES[border])
    else:
        native.fp32_Im2Col_Forward(x, y, xs, ys, xo, yo, frames, x.shape[1], w, h, c, ow, oh, y.shape[1], fw, fh, BORDER_MODES[border], border_value)
    return y


def im2col_backward(dy, c, h, w, frames, fh, fw, ys=1, xs=1, padding="valid"):
    oh, ow, yo, xo = im2col_geometry(h, w, fh, fw, ys, xs, padding)
    dx = native.new_rows(dy, c * h * w, _stride_for(frames, False))
    native.fp32_Im2Col_Backward(dy, dx, xs, ys, xo, yo, frames, dx.shape[1], w, h, c, ow, oh, dy.shape[1], fw, fh)
    return dx


def col2im_forward(x, c, h, w, frames):
    """x [c, stride] over frames*h*w frames -> y [c*h*w, stride'] over frames frames"""
    bit = x.dtype == torch.int32
    y = (native.new_zero_bits if bit else native.new_rows)(x, c * h * w, _stride_for(frames, bit))
    fn = native.bit_Col2Im_Forward if bit else native.fp32_Col2Im_Forward
    fn(x, y, w, h, c, x.shape[1], frames, y.shape[1])
    return y


def col2im_backward(dy, c, h, w, frames):
    dx = native.new_rows(dy, c, _stride_for(frames * h * w, False))
    native.fp32_Col2Im_Backward(dy, dx, w, h, c, dx.shape[1], frames, dy.shape[1])
    return dx


def stochastic_maxpool2x2_forward(x, c, h, w, frames):
    oh, ow = (h + 1) // 2, (w + 1) // 2
    y = native.new_rows(x, c * oh * ow, x.shape[1])
    native.fp32_StochasticMaxPooling2x2_Forward(x, y, w, h, ow, oh, c, frames, x.shape[1])
    return y


def stochastic_maxpool2x2_backward(x, dy, c, h, w, frames):
    oh, ow = (h + 1) // 2, (w + 1) // 2
    dx = torch.empty_like(x)
    native.fp32_StochasticMaxPooling2x2_Backward(x, dy, dx, w, h, ow, oh, c, frames, x.shape[1])
    return dx


def stochastic_bn_forward_training(x, running_mean, running_var, frame_size, gamma=0.2, beta=0.5, momentum=0.9):
    """Per-node batch normalisation with scalar gamma / beta, training pass: x [nodes, stride] -> (y, mean, rstd); the running
    statistics are updated in place."""
    nodes = x.shape[0]
    y = torch.empty_like(x)
    mean = native.new_line(x, nodes)
    rstd = native.new_line(x, nodes)
    native.fp32_StochasticBatchNormalization_ForwardTraining(x, y, mean, rstd, running_mean, running_var, gamma, beta, momentum, nodes, frame_size, x.shape[1])
    return y, mean, rstd


def stochastic_bn_reforward(x, mean, rstd, frame_size, gamma=0.2, beta=0.5):
    y = torch.empty_like(x)
    native.fp32_StochasticBatchNormalization_ReForward(x, y, mean, rstd, gamma, beta, x.shape[0], frame_size, x.shape[1])
    return y


def stochastic_bn_forward_inference(x, running_mean, running_var, frame_size, gamma=0.2, beta=0.5):
    y = torch.empty_like(x)
    native.fp32_StochasticBatchNormalization_ForwardInference(x, y, running_mean, running_var, gamma, beta, x.shape[0], frame_size, x.shape[1])
    return y


def stochastic_bn_backward(x, dy, mean, rstd, frame_size, gamma=0.2):
    dx = torch.empty_like(dy)
    native.fp32_StochasticBatchNormalization_Backward(x, dy, dx, mean, rstd, gamma, 1.0 / frame_size, dy.shape[0], frame_size, dy.shape[1], x.shape[1])
    return dx


def average_lut_forward(x, idx, frame_size, binarize_input=False, binarize_output=True, mean=True):
    """fp32 x [I, stride] -> y [O, stride]: the sign of the sum of the n wired inputs (their votes when binarize_input) or, without
    binarize_output, sum * (1 / n) as the reference's CUDA kernel writes it; mean=False: the plain sum of the reference's host loop."""
    O, n = idx.shape
    y = native.new_rows(x, O, x.shape[1])
    entry = native.fp32_AverageLut_Forward if mean else native.fp32_AverageLut_ForwardSum
    entry(x, y, idx, n, O, frame_size, x.shape[1], int(binarize_input), int(binarize_output))
    return y


def bit_average_lut_forward(xbits, idx, frame_size):
    """packed x [I, words] -> packed y [O, words]: strict majority of the n wired inputs."""
    O, n = idx.shape
    y = native.new_zero_bits(xbits, O, xbits.shape[1])
    native.bit_AverageLut_Forward(xbits, y, idx, n, O, frame_size, xbits.shape[1])
    return y


def average_lut_backward(dy, idx, input_nodes, frame_size):
    O, n = idx.shape
    dx = native.new_rows(dy, input_nodes, dy.shape[1])
    native.fp32_AverageLut_Backward(dy, dx, idx, n, input_nodes, O, frame_size, dy.shape[1])
    return dx


def max_lut_forward(x, idx, frame_size, binarize_input=False, binarize_output=True):
    """fp32 x [I, stride] -> y [O, stride]: the largest of the n wired inputs (not below -1), or its sign."""
    O, n = idx.shape
    y = native.new_rows(x, O, x.shape[1])
    native.fp32_MaxLut_Forward(x, y, idx, n, O, frame_size, x.shape[1], int(binarize_input), int(binarize_output))
    return y


def bit_max_lut_forward(xbits, idx, frame_size):
    """packed x [I, words] -> packed y [O, words]: the OR of the n wired inputs."""
    O, n = idx.shape
    y = native.new_bits(xbits, O, xbits.shape[1])
    native.bit_MaxLut_Forward(xbits, y, idx, n, O, frame_size, xbits.shape[1])
    return y


def max_lut_backward(x, dy, idx, frame_size, binarize_input=False):
    """dx [I, stride]: each node's dy goes to its first largest input."""
    O, n = idx.shape
    if x.shape[1] != dy.shape[1]:
        raise capi.BbhipError("max_lut_backward: x and dy must have the same row pitch")
    dx = native.new_rows(dy, x.shape[0], dy.shape[1])
    native.fp32_MaxLut_Backward(x, dy, dx, idx, n, x.shape[0], O, frame_size, dy.shape[1], int(binarize_input))
    return dx


def bit_max_lut_backward(xbits, dy, idx, frame_size):
    O, n = idx.shape
    dx = native.new_rows(dy, xbits.shape[0], dy.shape[1])
    native.bit_fp32_MaxLut_Backward(xbits, dy, dx, idx, n, xbits.shape[0], O, frame_size, xbits.shape[1], dy.shape[1])
    return dx


def reduce_forward(x, output_nodes, frame_size):
    """fp32 x [I, stride] -> y [O, stride]: node o is the mean of the inputs o, O + o, 2 O + o, ..."""
    y = native.new_rows(x, output_nodes, x.shape[1])
    native.fp32_Reduce_Forward(x, y, x.shape[0], output_nodes, frame_size, x.shape[1])
    return y


def bit_reduce_forward(xbits, output_nodes, frame_size, y_stride):
    """packed x [I, words] (bits read as +1 / -1) -> fp32 y [O, y_stride]"""
    y = native.new_rows(xbits, output_nodes, y_stride)
    native.bit_fp32_Reduce_Forward(xbits, y, xbits.shape[0], output_nodes, frame_size, xbits.shape[1], y_stride)
    return y


def reduce_backward(dy, input_nodes, frame_size):
    dx = native.new_rows(dy, input_nodes, dy.shape[1])
    native.fp32_Reduce_Backward(dy, dx, input_nodes, dy.shape[0], frame_size, dy.shape[1])
    return dx


def real_to_binary_forward(x, depth, points, frame_size, frame_mod=1, depth_mod=1, lo=0.0, hi=1.0, binarize=True, bit=False, y_stride=None):
    """fp32 x [depth * points, stride] -> y [depth * depth_mod * points, y_stride]: fp32, or rows of packed words with `bit`
    (padding words of a packed row beyond the last frame's word are left as allocated: zero)."""
    out_frames = frame_size * frame_mod
    if y_stride is None:
        y_stride = (out_frames + 31) // 32 if bit else out_frames
    nodes = depth * depth_mod * points
    if bit:
        y = native.new_padded_bits(x, nodes, y_stride)
        f = native.fp32_bit_RealToBinary_Forward
    else:
        y = native.new_rows(x, nodes, y_stride)
        f = native.fp32_RealToBinary_Forward
    f(x, y, depth_mod, frame_mod, lo, hi, points, depth, frame_size, x.shape[1], y_stride, int(binarize))
    return y


def binary_to_real_forward(x, output_nodes, y_frame_size, frame_mux=1, y_stride=None):
    """x [I, stride] fp32 (counted where > 0) or int32 packed bits, y_frame_size * frame_mux frames -> fp32 y [O, y_stride]"""
    y_stride = y_frame_size if y_stride is None else y_stride
    y = native.new_rows(x, output_nodes, y_stride)
    f = native.bit_fp32_BinaryToReal_Forward if x.dtype == torch.int32 else native.fp32_BinaryToReal_Forward
    f(x, y, x.shape[0] // output_nodes, frame_mux, output_nodes, x.shape[1], y_frame_size, y_stride)
    return y


def binary_to_real_backward(dy, input_nodes, y_frame_size, frame_mux=1, x_stride=None):
    x_stride = y_frame_size * frame_mux if x_stride is None else x_stride
    dx = native.new_rows(dy, input_nodes, x_stride)
    native.fp32_BinaryToReal_Backward(dy, dx, input_nodes // dy.shape[0], frame_mux, dy.shape[0], x_stride, y_frame_size, dy.shape[1])
    return dx


def binarize_forward(x, frame_size, th=0.0, low=-1.0, high=1.0, bit=False, y_stride=None):
    """y = x > th ? high : low, or with `bit` the packed bits of x > th"""
    if bit:
        y_stride = (frame_size + 31) // 32 if y_stride is None else y_stride
        y = native.new_zero_bits(x, x.shape[0], y_stride)
        native.fp32_bit_Binarize_Forward(x, y, th, x.shape[0], frame_size, x.shape[1], y_stride)
        return y
    y = torch.empty_like(x)
    native.fp32_Binarize_Forward(x, y, th, low, high, x.shape[0], frame_size, x.shape[1])
    return y


def hard_tanh_forward(x, frame_size, lo=-1.0, hi=1.0):
    y = torch.empty_like(x)
    native.fp32_HardTanh_Forward(x, y, lo, hi, x.shape[0], frame_size, x.shape[1])
    return y


def hard_tanh_backward(x, dy, frame_size, lo=-1.0, hi=1.0):
    """dx = dy inside the open window (lo, hi), 0 elsewhere; also the backward of Binarize"""
    dx = torch.empty_like(dy)
    native.fp32_HardTanh_Backward(x, dy, dx, lo, hi, x.shape[0], frame_size, x.shape[1])
    return dx


def _pool_out(h, w, fh, fw):
    return (h + fh - 1) // fh, (w + fw - 1) // fw


def max_pooling_forward(x, c, h, w, fh, fw, frame_size):
    """fp32 x [c * h * w, stride] -> (y, argmax) [c * oh * ow, stride]"""
    oh, ow = _pool_out(h, w, fh, fw)
    y = native.new_rows(x, c * oh * ow, x.shape[1])
    arg = native.new_bits(x, c * oh * ow, x.shape[1])
    native.fp32_MaxPooling_Forward(x, y, arg, fh, fw, w, h, ow, oh, c, frame_size, x.shape[1])
    return y, arg


def max_pooling_backward(argmax, dy, c, h, w, fh, fw, frame_size):
    oh, ow = _pool_out(h, w, fh, fw)
    dx = native.new_rows(dy, c * h * w, dy.shape[1])
    native.fp32_MaxPooling_Backward(argmax, dy, dx, fh, fw, w, h, ow, oh, c, frame_size, dy.shape[1])
    return dx


def bit_max_pooling_forward(xbits, c, h, w, fh, fw, frame_size):
    oh, ow = _pool_out(h, w, fh, fw)
    y = native.new_zero_bits(xbits, c * oh * ow, xbits.shape[1])
    native.bit_MaxPooling_Forward(xbits, y, fh, fw, w, h, ow, oh, c, frame_size, xbits.shape[1])
    return y


def bit_max_pooling_backward(xbits, dy, c, h, w, fh, fw, frame_size):
    oh, ow = _pool_out(h, w, fh, fw)
    dx = native.new_rows(dy, c * h * w, dy.shape[1])
    native.bit_fp32_MaxPooling_Backward(xbits, dy, dx, fh, fw, w, h, ow, oh, c, frame_size, xbits.shape[1], dy.shape[1])
    return dx


def up_sampling_forward(x, c, h, w, fh, fw, frame_size, fill=True):
    """x [c * h * w, stride], fp32 or int32 packed words -> y [c * h fh * w fw, stride] of the same type"""
    if x.dtype == torch.int32:
        y = native.new_zero_bits(x, c * h * fh * w * fw, x.shape[1])
        f = native.bit_UpSampling_Forward
    else:
        y = native.new_rows(x, c * h * fh * w * fw, x.shape[1])
        f = native.fp32_UpSampling_Forward
    f(x, y, w, h, c, fw, fh, int(fill), frame_size, x.shape[1])
    return y


def up_sampling_backward(dy, c, h, w, fh, fw, frame_size, fill=True):
    dx = native.new_rows(dy, c * h * w, dy.shape[1])
    native.fp32_UpSampling_Backward(dy, dx, w, h, c, fw, fh, int(fill), frame_size, dy.shape[1])
    return dx


def shuffle_forward(x, shuffle_unit, frame_size):
    """x [nodes, stride], fp32 or int32 packed words: row i * shuffle_unit + j of the result is row j * (nodes / shuffle_unit) + i"""
    y = torch.empty_like(x)
    native.Shuffle_Forward(x, y, shuffle_unit, x.shape[0], frame_size, x.shape[1])
    return y


def shuffle_backward(dy, shuffle_unit, frame_size):
    dx = torch.empty_like(dy)
    native.Shuffle_Backward(dy, dx, shuffle_unit, dy.shape[0], frame_size, dy.shape[1])
    return dx


def loss_mean_squared_error(y, t, frame_size, loss_buf, batch_size=None, reduction_sum=False):
    """-> dy; loss_buf (float64, device, any length >= 1) receives the batch's partial sums ON TOP of what it holds.  The layer's loss is
    loss_buf.sum() / frames seen (the sum itself with reduction "sum")."""
    nodes = y.shape[0]
    batch_size = frame_size if batch_size is None else batch_size
    grad_reduction = np.float32(1.0) if reduction_sum else np.float32(1.0) / np.float32(nodes * batch_size)
    loss_reduction = 1.0 if reduction_sum else 1.0 / nodes
    dy = torch.empty_like(y)
    native.fp32_LossMeanSquaredError(y, t, dy, loss_buf, loss_buf.numel(), nodes, frame_size, y.shape[1], float(np.float32(2) * grad_reduction), loss_reduction)
    return dy


def metrics_mean_squared_error(y, t, frame_size, accuracy_buf):
    """accuracy_buf (float64, device) += the batch's partial sums of (t - y)^2 / nodes; the metric is accuracy_buf.sum() / frames seen."""
    native.fp32_MetricsMeanSquaredError(y, t, accuracy_buf, accuracy_buf.numel(), y.shape[0], frame_size, y.shape[1])


def loss_softmax_cross_entropy(y, t, ch_size, pix_size, frame_size, t_sum=None):
    """y, t [ch*pix, stride] -> (dy, loss_buf [frames] float64, t_sum).  t_sum defaults to the sum of the targets of the
    frames in use, taken in float64 as the reference's device path does; the loss of the batch is -loss_buf.sum() / t_sum."""
    if t_sum is None:
        t_sum = float(t[:, :frame_size].sum(dtype=torch.float64).item())
    dy = torch.empty_like(y)
    loss_buf = torch.empty((frame_size,), dtype=torch.float64, device=y.device)
    native.fp32_LossSoftmaxCrossEntropy(y, t, dy, loss_buf, t_sum, pix_size, ch_size, frame_size, y.shape[1])
    return dy, loss_buf, t_sum


def metrics_categorical_accuracy(y, t, ch_size, pix_size, frame_size):
    """-> (accuracy_buf, category_buf) int32 [frames]; the metric of the batch is the ratio of their sums."""
    acc = torch.empty((frame_size,), dtype=torch.int32, device=y.device)
    cat = torch.empty((frame_size,), dtype=torch.int32, device=y.device)
    native.fp32_MetricsCategoricalAccuracy(y, t, acc, cat, pix_size, ch_size, frame_size, y.shape[1])
    return acc, cat


def classifier_tail(x, idx, t, frame_size, t_sum=None, binarize_input=False, mean=True, want_y=True, want_dy=False, want_accuracy=True):
    """AverageLut forward (un-binarized) + softmax cross entropy + categorical accuracy + AverageLut backward in one launch; the same
    bits as `average_lut_forward`, `loss_softmax_cross_entropy`, `metrics_categorical_accuracy` and `average_lut_backward` called one
    after the other.  returns (y or None, dx, loss_buf, accuracy or None, category or None, dy or None)."""
    if t_sum is None:
        t_sum = float(t[:, :frame_size].sum(dtype=torch.float64).item())
    return native.classifier_tail(x, idx, t, frame_size, t_sum, binarize_input, mean, want_y, want_dy, want_accuracy)


def conv_bit_to_real(xbits, frame_size, y_stride, value0=0.0, value1=1.0):
    y = native.new_rows(xbits, xbits.shape[0], y_stride)
    native.fp32_ConvBitToReal(xbits, y, value0, value1, xbits.shape[0], frame_size, xbits.shape[1], y_stride)
    return y


def packed_input_buffer(rows, frame_size, device="cuda"):
    """A place for the packed copy of a binarized fp32 input of `rows` node rows (see `packed=` of the LUT forward / backward wrappers):
    the forward call fills it, the backward call on the same input reads it instead of packing the input again."""
    return torch.empty((rows, lib().bbhip_PackedRowWords(frame_size)), dtype=torch.int32, device=device)


def prepared_tables_buffer(n, node_size, device="cuda"):
    """A buffer for bbhip_HintPreparedTables: the tables that a LUT call derives from W, kept from a step's forward call for its
    backward call (`tables=` of the DifferentiableLut wrappers)."""
    return torch.empty(lib().bbhip_PreparedTablesBytes(n, node_size) // 4, dtype=torch.float32, device=device)


HINTS = True          # False: the wrappers pass no bbhip_Hint* at all (what a caller of the reference's plain signatures gets)


def stochastic_lut_forward(n, x, idx, W, frame_size, input_binary=False, lut_binarize=False, bias=0.25, out=None, clamp_w=None, packed=None,
                           packed_holds=False):
    """clamp_w = (lo, hi): W is clamped in place first, as StochasticLutN::Forward does (include/bb/StochasticLutN.h:451),
    by the same launch that prepares the tables."""
    return native.stochastic_lut_forward(n, x, idx, W, frame_size, input_binary, lut_binarize, bias, out, clamp_w, packed, packed_holds, HINTS)


def bit_stochastic_lut_forward(n, xbits, idx, W, frame_size, y_stride, lut_binarize=False, bias=0.25):
    O = idx.shape[0]
    y = native.new_rows(xbits, O, y_stride)
    native.bit_fp32_StochasticLut_Forward(n, xbits, y, idx, W, O, frame_size, y_stride, xbits.shape[1], int(lut_binarize), bias)
    return y


def bit_bit_stochastic_lut_forward(n, xbits, idx, W, frame_size, lut_binarize=False, bias=0.25):
    O = idx.shape[0]
    y = native.new_padded_bits(xbits, O, xbits.shape[1])
    native.bit_bit_fp32_StochasticLut_Forward(n, xbits, y, idx, W, O, frame_size, xbits.shape[1], int(lut_binarize), bias)
    return y


def _tmp_frames(output_nodes, n, frame_size, max_tmp_bytes=256 * 1024 * 1024):
    """Frames per dx_tmp pass, as the reference sizes its scratch (include/bb/StochasticLutN.h:584-587)."""
    t = max_tmp_bytes // (4 * output_nodes * n)
    t = max(t, 32)
    t = (t + 31) & ~0x1f
    return min(t, frame_size)


def stochastic_lut_backward(n, x, dy, idx, W, dW, frame_size, rev=None, input_binary=False, lut_binarize=False, bias=0.25,
                            dx_tmp=None, tmp_frame_size=None, max_tmp_bytes=256 * 1024 * 1024, out=None, packed=None, overwrite_dw=False):
    """dW is accumulated in place; returns dx [I, stride]. ``rev`` (reverse table) is needed by dx modes 0 and 2,
    dx_tmp by mode 2 only (allocated here when not given)."""
    return native.stochastic_lut_backward(n, x, dy, idx, W, dW, frame_size, rev, input_binary, lut_binarize, bias, dx_tmp,
                                          -1 if tmp_frame_size is None else tmp_frame_size, max_tmp_bytes, out, packed, overwrite_dw, HINTS)


def bit_stochastic_lut_backward(n, xbits, dy, idx, W, dW, frame_size, rev=None, lut_binarize=False, bias=0.25,
                                max_tmp_bytes=256 * 1024 * 1024):
    return native.bit_stochastic_lut_backward(n, xbits, dy, idx, W, dW, frame_size, rev, lut_binarize, bias, max_tmp_bytes)


def differentiable_lut_forward_training(n, x, idx, W, frame_size, running_mean, running_var, gamma=0.3, beta=0.5,
                                        momentum=0.9, bias=0.25, lut_binarize=False, binary_mode=True, clamp_w=None, packed=None, tables=None,
                                        packed_holds=False, packed_out=None):
    """fp32 frames. running_mean / running_var are updated in place. returns (y, mean, rstd).
    packed_holds: `packed` already holds the packed copy of x (it was the `packed_out` of the layer before): nothing is packed.
    packed_out: a `packed_input_buffer(O, frame_size)` that receives the binarized output as packed bits, for the next layer.
    tables: a `prepared_tables_buffer` that receives the tables derived from W, for the backward call of the same step.
    packed: a `packed_input_buffer` that receives the packed copy of the binarized input (binary mode), for the backward call.
    clamp_w = (lo, hi): W is clamped in place first, by the launch that prepares the tables (the model class's clamp before the
    first forward pass after a backward pass, include/bb/DifferentiableLutN.h:605-608)."""
    return native.differentiable_lut_forward_training(n, x, idx, W, frame_size, running_mean, running_var, gamma, beta, momentum, bias, lut_binarize,
                                                      binary_mode, clamp_w, packed, tables, packed_holds, packed_out, HINTS)


def bit_differentiable_lut_forward_training(n, xbits, idx, W, frame_size, running_mean, running_var, gamma=0.3, beta=0.5,
                                            momentum=0.9, bias=0.25, lut_binarize=False, clamp_w=None, tables=None, out=None):
    """out: a packed output buffer [O, words] to write into (a layer keeps one); None: a new zero-filled one."""
    if out is not None and (out.shape != (idx.shape[0], xbits.shape[1]) or out.dtype != torch.int32):
        raise ValueError("out must be int32 [%d, %d]" % (idx.shape[0], xbits.shape[1]))
    return native.bit_differentiable_lut_forward_training(n, xbits, idx, W, frame_size, running_mean, running_var, gamma, beta, momentum, bias,
                                                          lut_binarize, clamp_w, tables, out, HINTS)


def differentiable_lut_forward_inference(n, x, idx, W, frame_size, running_mean, running_var, gamma=0.3, beta=0.5,
                                         bias=0.25, lut_binarize=False, binary_mode=True, packed=None, packed_holds=False, packed_out=None):
    return native.differentiable_lut_forward_inference(n, x, idx, W, frame_size, running_mean, running_var, gamma, beta, bias, lut_binarize,
                                                       binary_mode, packed, packed_holds, packed_out, HINTS)


def bit_differentiable_lut_forward_inference(n, xbits, idx, W, frame_size, running_mean, running_var, gamma=0.3,
                                             beta=0.5, bias=0.25, lut_binarize=False):
    return native.bit_differentiable_lut_forward_inference(n, xbits, idx, W, frame_size, running_mean, running_var, gamma, beta, bias, lut_binarize)


def differentiable_lut_forward_nobn(n, x, idx, W, frame_size, bias=0.25, lut_binarize=False, binary_mode=True, packed=None, packed_holds=False,
                                    packed_out=None):
    return native.differentiable_lut_forward_nobn(n, x, idx, W, frame_size, bias, lut_binarize, binary_mode, packed, packed_holds, packed_out, HINTS)


def differentiable_lut_backward(n, x, dy, idx, W, dW, frame_size, mean, rstd, rev=None, gamma=0.3, beta=0.5, bias=0.25,
                                lut_binarize=False, binary_mode=True, max_tmp_bytes=256 * 1024 * 1024, packed=None, tables=None, overwrite_dw=False):
    """tables: the buffer that this step's forward call with the same W filled (`prepared_tables_buffer`): no preparation launch.
    packed: the buffer that the forward call on the same x filled (`packed_input_buffer`): the call reads it instead of packing x."""
    return native.differentiable_lut_backward(n, x, dy, idx, W, dW, frame_size, mean, rstd, rev, gamma, beta, bias, lut_binarize, binary_mode,
                                              max_tmp_bytes, packed, tables, overwrite_dw, HINTS)


def bit_differentiable_lut_backward(n, xbits, dy, idx, W, dW, frame_size, mean, rstd, rev=None, gamma=0.3, beta=0.5,
                                    bias=0.25, lut_binarize=False, max_tmp_bytes=256 * 1024 * 1024, tables=None):
    return native.bit_differentiable_lut_backward(n, xbits, dy, idx, W, dW, frame_size, mean, rstd, rev, gamma, beta, bias, lut_binarize,
                                                  max_tmp_bytes, tables, HINTS)


def binary_lut6_forward(xbits, idx, table, frame_size, out=None):
    return native.binary_lut_forward(6, xbits, idx, table, frame_size, out)


def binary_lutn_forward(n, xbits, idx, table, frame_size, out=None):
    """BinaryLutN<n> on packed bits, n = 2 .. 6: table [O, 1] words for n <= 5 (entry i = bit i), [O, 2] for n = 6"""
    assert idx.shape[1] == n and table.shape == (idx.shape[0], 2 if n == 6 else 1)
    return native.binary_lut_forward(n, xbits, idx, table, frame_size, out)


def reverse_table(idx, input_nodes):
    """Reverse connection table as the reference builds it (include/bb/FixedSizeConnectionTable.h:180-215):
    ``[input_nodes, 1 + max fan-out]`` int32, row r = [count, node*n + input ... ascending, zero tail].
    Built on the host with numpy (index bookkeeping, not on the timed path); returned on idx's device."""
    h = idx.detach().cpu().numpy().astype(np.int64)
    O, n = h.shape
    flat = h.reshape(-1)
    counts = np.bincount(flat, minlength=input_nodes)
    stride = int(counts.max()) + 1 if flat.size else 1
    order = np.argsort(flat, kind="stable")                      # ascending (node, input) within each input row
    starts = np.concatenate([[0], np.cumsum(counts)[:-1]])
    rev = np.zeros((input_nodes, stride), np.int32)
    rev[:, 0] = counts
    pos = np.arange(flat.size) - np.repeat(starts, counts)
    rev[flat[order], 1 + pos] = order.astype(np.int32)
    return torch.from_numpy(rev).to(idx.device)
