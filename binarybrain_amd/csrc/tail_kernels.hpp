// The tail of a LUT classifier: AverageLut (sum / vote over n wired inputs), softmax cross entropy and categorical accuracy.
//
// All of it is streaming work over node-major, frame-minor buffers: one lane per frame (or per 32-frame word), rows read
// as contiguous runs.  Results follow the reference's host loops (include/bb/AverageLut.h:320-345, 386-406;
// LossSoftmaxCrossEntropy.h:159-211; MetricsCategoricalAccuracy.h:144-173): AverageLut writes the SUM when the output is
// not binarized, gradients are dy / n added node ascending then input ascending, each product that the host code rounds
// on its own is rounded on its own here.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "corner_index.hpp"
#include "vector_kernels.hpp"

namespace bbhip {

constexpr int kTailBlock = 256;

// one thread per (output node, frame)
// scale: what an un-binarized sum is multiplied by — 1 (the host loop of the reference writes the sum) or the fp32
// reciprocal of n (its CUDA kernel writes sum * (1 / n), cuda/AverageLut.cu:46-54)
__global__ __launch_bounds__(kTailBlock) void average_lut_forward_kernel(float const *x, float *y, int const *idx, int n, int frame_size,
                                                                         int frame_stride, int binarize_input, int binarize_output, int f_blocks,
                                                                         float scale)
{
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const node = blockIdx.x / f_blocks;
    if (f >= frame_size) { return; }
    int const *row = idx + (size_t)node * n;
    float sum = 0.0f;
    for (int i = 0; i < n; ++i) {
        float v = x[(size_t)row[i] * frame_stride + f];
        if (binarize_input) { v = (v > 0.0f) ? 1.0f : -1.0f; }
        sum += v;
    }
    if (binarize_output) { sum = (sum > 0.0f) ? 1.0f : -1.0f; }
    else                 { sum = rounded_mul(sum, scale); }
    y[(size_t)node * frame_stride + f] = sum;
}

// Packed bits, one thread per (output node, 32-frame word): the n input words are added into P bit planes (plane p holds
// bit p of each frame's count of ones) and the count is compared with floor(n / 2): ones > n / 2 is the strict majority
// that the host loop computes as (ones - zeros) > 0.
template <int P>
__global__ __launch_bounds__(kTailBlock) void average_lut_forward_bit_kernel(int const *x, int *y, int const *idx, int n, int words,
                                                                             int frame_stride, int w_blocks)
{
    int const w = (int)(blockIdx.x % w_blocks) * kTailBlock + threadIdx.x;
    int const node = blockIdx.x / w_blocks;
    if (w >= words) { return; }
    int const *row = idx + (size_t)node * n;
    uint32_t plane[P];
#pragma unroll
    for (int p = 0; p < P; ++p) { plane[p] = 0u; }
    for (int i = 0; i < n; ++i) {
        uint32_t carry = (uint32_t)x[(size_t)row[i] * frame_stride + w];
#pragma unroll
        for (int p = 0; p < P; ++p) {
            uint32_t const t = plane[p] & carry;
            plane[p] ^= carry;
            carry = t;
        }
    }
    uint32_t const threshold = (uint32_t)n >> 1;
    uint32_t gt = 0u, eq = ~0u;
#pragma unroll
    for (int p = P - 1; p >= 0; --p) {
        uint32_t const tb = ((threshold >> p) & 1u) ? ~0u : 0u;
        gt |= eq & plane[p] & ~tb;
        eq &= ~(plane[p] ^ tb);
    }
    y[(size_t)node * frame_stride + w] = (int)gt;
}

// any n: per frame bit, count the ones directly
__global__ __launch_bounds__(kTailBlock) void average_lut_forward_bit_wide_kernel(int const *x, int *y, int const *idx, int n, int words,
                                                                                  int frame_stride, int w_blocks)
{
    int const w = (int)(blockIdx.x % w_blocks) * kTailBlock + threadIdx.x;
    int const node = blockIdx.x / w_blocks;
    if (w >= words) { return; }
    int const *row = idx + (size_t)node * n;
    uint32_t out = 0u;
    for (int base = 0; base < 32; base += 4) {               // four frame bits per sweep over the inputs
        int ones[4] = {0, 0, 0, 0};
        for (int i = 0; i < n; ++i) {
            uint32_t const v = (uint32_t)x[(size_t)row[i] * frame_stride + w] >> base;
#pragma unroll
            for (int b = 0; b < 4; ++b) { ones[b] += (int)((v >> b) & 1u); }
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) { out |= (2 * ones[b] > n) ? (1u << (base + b)) : 0u; }
    }
    y[(size_t)node * frame_stride + w] = (int)out;
}

// Reverse wiring for the backward pass, built on the device: for input node i, offsets[i] = number of table entries that
// name a smaller input, and list[offsets[i] ...] = the output nodes wired to i in table order (node ascending, input
// position ascending).  One thread per input node (plus one for the end offset) sweeps the whole table twice; the block
// stages the table through LDS in pieces, so a sweep is one coalesced load per piece and broadcast LDS reads.
// Entries outside [0, input_node_size) match no thread.
constexpr int kReversePiece = 2048;

// copy `count` table entries into LDS and fill up to the next multiple of four with -1, which matches no input node
__device__ __forceinline__ void stage_piece(int *piece, int const *__restrict__ src, int count)
{
    int const padded = (count + 3) & ~3;
    for (int k = threadIdx.x; k < padded; k += kTailBlock) { piece[k] = (k < count) ? src[k] : -1; }
}

// entry_ids: the list holds table positions (node * n + input position) instead of output nodes
__global__ __launch_bounds__(kTailBlock) void average_lut_reverse_kernel(int const *__restrict__ idx, int total, int n, int input_node_size,
                                                                         int *__restrict__ offsets, int *__restrict__ list, int entry_ids)
{
    __shared__ __attribute__((aligned(16))) int piece[kReversePiece];
    int const i = blockIdx.x * kTailBlock + threadIdx.x;
    bool const live = (i <= input_node_size);
    int below = 0;
    for (int base = 0; base < total; base += kReversePiece) {
        int const count = min(kReversePiece, total - base);
        __syncthreads();
        stage_piece(piece, idx + base, count);
        __syncthreads();
#pragma unroll 2
        for (int k = 0; k < count; k += 4) {
            int4 const e = *reinterpret_cast<int4 const *>(&piece[k]);
            below += ((uint32_t)e.x < (uint32_t)i) + ((uint32_t)e.y < (uint32_t)i) + ((uint32_t)e.z < (uint32_t)i) + ((uint32_t)e.w < (uint32_t)i);
        }
    }
    if (live) { offsets[i] = below; }
    int at = below;
    for (int base = 0; base < total; base += kReversePiece) {
        int const count = min(kReversePiece, total - base);
        __syncthreads();
        stage_piece(piece, idx + base, count);
        __syncthreads();
        if (live && i < input_node_size) {
#pragma unroll 2
            for (int k = 0; k < count; k += 4) {
                int4 const e = *reinterpret_cast<int4 const *>(&piece[k]);
                if (e.x == i) { list[at++] = entry_ids ? (base + k)     : (base + k) / n; }
                if (e.y == i) { list[at++] = entry_ids ? (base + k + 1) : (base + k + 1) / n; }
                if (e.z == i) { list[at++] = entry_ids ? (base + k + 2) : (base + k + 2) / n; }
                if (e.w == i) { list[at++] = entry_ids ? (base + k + 3) : (base + k + 3) / n; }
            }
        }
    }
}

// one thread per (input node, column of the row pitch): dx = sum over the wired output nodes, in table order, of dy / n
__global__ __launch_bounds__(kTailBlock) void average_lut_backward_kernel(float const *dy, float *dx, int const *offsets, int const *list,
                                                                          int n, int frame_size, int frame_stride, int f_blocks)
{
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const in = blockIdx.x / f_blocks;
    if (f >= frame_stride) { return; }
    if (f >= frame_size) { dx[(size_t)in * frame_stride + f] = 0.0f; return; }      // the row's padding reads as zero, as after the host's FillZero
    int const begin = offsets[in], end = offsets[in + 1];
    float const fn = (float)n;
    float acc = 0.0f;
    for (int k = begin; k < end; ++k) { acc += dy[(size_t)list[k] * frame_stride + f] / fn; }
    dx[(size_t)in * frame_stride + f] = acc;
}

// The same for a table of at most kReversePiece entries, without the reverse wiring: every workgroup (one input node, kTailBlock
// columns) stages the whole table in LDS and walks it in table order; the comparison is the same for all its threads.  For the
// tails of classifiers (tens of entries) this saves the launch that builds the reverse wiring, which costs more than the walk.
__global__ __launch_bounds__(kTailBlock) void average_lut_backward_small_kernel(float const *dy, float *dx, int const *__restrict__ idx, int total,
                                                                                int n, int frame_size, int frame_stride, int f_blocks)
{
    __shared__ __attribute__((aligned(16))) int piece[kReversePiece];
    stage_piece(piece, idx, total);
    __syncthreads();
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const in = blockIdx.x / f_blocks;
    if (f >= frame_stride) { return; }
    if (f >= frame_size) { dx[(size_t)in * frame_stride + f] = 0.0f; return; }
    float const fn = (float)n;
    float acc = 0.0f;
    for (int k = 0; k < total; ++k) {
        if (piece[k] == in) { acc += dy[(size_t)(k / n) * frame_stride + f] / fn; }
    }
    dx[(size_t)in * frame_stride + f] = acc;
}

// MaxLut: the largest of the n wired inputs, starting from -1 and replaced by strictly larger values only (reference host
// loop: include/bb/MaxLut.h:293-318); binarize_input as in the reference's device kernel (cuda/MaxLut.cu:33-36).
// One thread per (output node, frame).
__global__ __launch_bounds__(kTailBlock) void max_lut_forward_kernel(float const *x, float *y, int const *idx, int n, int frame_size,
                                                                     int frame_stride, int binarize_input, int binarize_output, int f_blocks)
{
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const node = blockIdx.x / f_blocks;
    if (f >= frame_size) { return; }
    int const *row = idx + (size_t)node * n;
    float max_val = -1.0f;
    for (int i = 0; i < n; ++i) {
        float v = x[(size_t)row[i] * frame_stride + f];
        if (binarize_input) { v = (v > 0.0f) ? 1.0f : -1.0f; }
        if (v > max_val) { max_val = v; }
    }
    if (binarize_output) { max_val = (max_val > 0.0f) ? 1.0f : -1.0f; }
    y[(size_t)node * frame_stride + f] = max_val;
}

// packed bits, one thread per (output node, 32-frame word): the OR of the n input words
__global__ __launch_bounds__(kTailBlock) void max_lut_forward_bit_kernel(int const *x, int *y, int const *idx, int n, int words,
                                                                         int frame_stride, int w_blocks)
{
    int const w = (int)(blockIdx.x % w_blocks) * kTailBlock + threadIdx.x;
    int const node = blockIdx.x / w_blocks;
    if (w >= words) { return; }
    int const *row = idx + (size_t)node * n;
    uint32_t any = 0u;
    for (int i = 0; i < n; ++i) { any |= (uint32_t)x[(size_t)row[i] * frame_stride + w]; }
    y[(size_t)node * frame_stride + w] = (int)any;
}

// One thread per (input node, column of the dx row pitch): over the table positions that name this input, in table order, add
// the node's dy where this position holds the node's first largest input (include/bb/MaxLut.h:394-424).  BITS: x is packed, the
// first largest input is the first one that is set (position 0 when none is).
// the position of a node's first largest input at frame f (BITS: the first input that is set; position 0 when none is)
template <bool BITS>
__device__ __forceinline__ int max_lut_winner(void const *x_buf, int const *row, int n, int f, int x_stride, int binarize_input)
{
    int first = 0;
    if (BITS) {
        uint32_t const *xb = static_cast<uint32_t const *>(x_buf);
        for (int i = 0; i < n; ++i) {
            if ((xb[(size_t)row[i] * x_stride + (f >> 5)] >> (f & 31)) & 1u) { first = i; break; }
        }
    }
    else {
        float const *xf = static_cast<float const *>(x_buf);
        float max_val = -1.0f;
        for (int i = 0; i < n; ++i) {
            float v = xf[(size_t)row[i] * x_stride + f];
            if (binarize_input) { v = (v > 0.0f) ? 1.0f : -1.0f; }
            if (v > max_val) { max_val = v; first = i; }
        }
    }
    return first;
}

// One thread per (input node, column of the dx row pitch): over the table positions that name this input, in table order, add
// the node's dy where this position holds the node's first largest input (include/bb/MaxLut.h:394-424).
template <bool BITS>
__global__ __launch_bounds__(kTailBlock) void max_lut_backward_kernel(void const *x_buf, float const *dy, float *dx, int const *idx,
                                                                      int const *offsets, int const *list, int n, int frame_size,
                                                                      int x_stride, int dy_stride, int binarize_input, int f_blocks)
{
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const in = blockIdx.x / f_blocks;
    if (f >= dy_stride) { return; }
    if (f >= frame_size) { dx[(size_t)in * dy_stride + f] = 0.0f; return; }         // the row's padding reads as zero, as after the host's FillZero
    int const begin = offsets[in], end = offsets[in + 1];
    float acc = 0.0f;
    for (int k = begin; k < end; ++k) {
        int const entry = list[k], node = entry / n, pos = entry - node * n;
        if (max_lut_winner<BITS>(x_buf, idx + (size_t)node * n, n, f, x_stride, binarize_input) == pos) { acc += dy[(size_t)node * dy_stride + f]; }
    }
    dx[(size_t)in * dy_stride + f] = acc;
}

// the same for a table of at most kReversePiece entries, walked from LDS without the reverse wiring (see average_lut_backward_small_kernel)
template <bool BITS>
__global__ __launch_bounds__(kTailBlock) void max_lut_backward_small_kernel(void const *x_buf, float const *dy, float *dx, int const *__restrict__ idx,
                                                                            int total, int n, int frame_size, int x_stride, int dy_stride,
                                                                            int binarize_input, int f_blocks)
{
    __shared__ __attribute__((aligned(16))) int piece[kReversePiece];
    stage_piece(piece, idx, total);
    __syncthreads();
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const in = blockIdx.x / f_blocks;
    if (f >= dy_stride) { return; }
    if (f >= frame_size) { dx[(size_t)in * dy_stride + f] = 0.0f; return; }
    float acc = 0.0f;
    for (int k = 0; k < total; ++k) {
        if (piece[k] != in) { continue; }
        int const node = k / n, pos = k - node * n;
        if (max_lut_winner<BITS>(x_buf, piece + node * n, n, f, x_stride, binarize_input) == pos) { acc += dy[(size_t)node * dy_stride + f]; }
    }
    dx[(size_t)in * dy_stride + f] = acc;
}

// Reduce: output node o is the mean of the input nodes o, O + o, 2 O + o, ... (reference host loop: include/bb/Reduce.h:172-190;
// the reference has no device code for this layer).  One thread per (output node, frame); BITS: packed input read as +1 / -1.
template <bool BITS>
__global__ __launch_bounds__(kTailBlock) void reduce_forward_kernel(void const *x_buf, float *y, int mux, int output_node_size, int frame_size,
                                                                    int x_stride, int y_stride, int f_blocks)
{
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const o = blockIdx.x / f_blocks;
    if (f >= frame_size) { return; }
    float sum = 0.0f;
    for (int i = 0; i < mux; ++i) {
        size_t const row = (size_t)output_node_size * i + o;
        if (BITS) { sum += ((static_cast<uint32_t const *>(x_buf)[row * x_stride + (f >> 5)] >> (f & 31)) & 1u) ? 1.0f : -1.0f; }
        else      { sum += static_cast<float const *>(x_buf)[row * x_stride + f]; }
    }
    y[(size_t)o * y_stride + f] = sum / (float)mux;
}

// dx[input node] = dy[input node mod O] / mux (include/bb/Reduce.h:229-247); one thread per (input node, frame)
__global__ __launch_bounds__(kTailBlock) void reduce_backward_kernel(float const *dy, float *dx, int mux, int output_node_size, int frame_size,
                                                                     int frame_stride, int f_blocks)
{
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const in = blockIdx.x / f_blocks;
    if (f >= frame_size) { return; }
    dx[(size_t)in * frame_stride + f] = dy[(size_t)(in % output_node_size) * frame_stride + f] / (float)mux;
}

// Mean squared error.  One thread per (group of kMseNodes nodes, frame): dy = (y - t) * grad_scale, and the group's share of the
// frame's loss, node ascending, in double: partial[group][frame] = sum of (float)(y - t)^2 * loss_scale (LOSS: NaN squares left
// out, as the reference's loss does, include/bb/LossMeanSquaredError.h:150-169; else sum of (float)(t - y)^2 / node_size, as its
// metric, MetricsMeanSquaredError.h:66-85).
constexpr int kMseNodes = 64;

template <bool LOSS>
__global__ __launch_bounds__(kTailBlock) void mean_squared_error_kernel(float const *y, float const *t, float *dy, double *partial,
                                                                        float grad_scale, double loss_scale, int node_size, int frame_size,
                                                                        int frame_stride, int f_blocks)
{
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const group = blockIdx.x / f_blocks;
    if (f >= frame_size) { return; }
    int const first = group * kMseNodes, last = min(first + kMseNodes, node_size);
    double acc = 0.0;
    for (int node = first; node < last; ++node) {
        size_t const at = (size_t)node * frame_stride + f;
        if (LOSS) {
            float const grad = y[at] - t[at];
            float const error = rounded_mul(grad, grad);
            dy[at] = rounded_mul(grad, grad_scale);
            if (error == error) { acc += (double)error * loss_scale; }
        }
        else {
            float const grad = t[at] - y[at];
            acc += (double)rounded_mul(grad, grad) / loss_scale;
        }
    }
    partial[(size_t)group * frame_size + f] = acc;
}

// buf[s] += the partial sums of the frames s, s + buf_size, s + 2 buf_size, ...: frames ascending, groups ascending within a frame
__global__ __launch_bounds__(kTailBlock) void mean_squared_error_sum_kernel(double const *partial, double *buf, int buf_size, int groups,
                                                                            int frame_size)
{
    int const s = blockIdx.x * kTailBlock + threadIdx.x;
    if (s >= buf_size || s >= frame_size) { return; }
    double acc = 0.0;
    for (int f = s; f < frame_size; f += buf_size) {
        for (int g = 0; g < groups; ++g) { acc += partial[(size_t)g * frame_size + f]; }
    }
    buf[s] += acc;
}

// Softmax cross entropy, one thread per (pixel, frame); node = ch * pix_size + pix.  partial[pix * frame_size + frame]
// receives sum over the channels with t > 0 of log(softmax + eps) * t_max in double; with one pixel that is loss_buf itself.
__global__ __launch_bounds__(kTailBlock) void softmax_cross_entropy_kernel(float const *y, float const *t, float *dy, double *partial,
                                                                           float t_sum, int pix_size, int ch_size, int frame_size,
                                                                           int frame_stride, int f_blocks)
{
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const pix = blockIdx.x / f_blocks;
    if (f >= frame_size) { return; }
    float const eps = 1.0e-7f;
    size_t const node_step = (size_t)pix_size * frame_stride;
    size_t const first = (size_t)pix * frame_stride + f;
    float c = -3.402823466e+38f;
    for (int ch = 0; ch < ch_size; ++ch) {
        float const v = y[first + ch * node_step];
        c = (c < v) ? v : c;
    }
    float y_sum = 0.0f, t_max = 0.0f;
    for (int ch = 0; ch < ch_size; ++ch) {
        y_sum += expf(y[first + ch * node_step] - c);
        t_max += t[first + ch * node_step];
    }
    if (y_sum <= eps) { y_sum = eps; }
    double loss = 0.0;
    for (int ch = 0; ch < ch_size; ++ch) {
        size_t const at = first + ch * node_step;
        float const tv = t[at];
        float const softmax = expf(y[at] - c) / y_sum;
        if (tv > 0.0f) { loss += (double)rounded_mul(logf(softmax + eps), t_max); }
        dy[at] = (rounded_mul(t_max, softmax) - tv) / t_sum;
    }
    partial[(size_t)pix * frame_size + f] = loss;
}

// The same arithmetic for at most CH channels with every y and t of the (pixel, frame) loaded first: the loads of the three passes
// above depend on nothing, but issued one pass after the other their latencies add up, which is what a small batch pays for.
template <int CH>
__global__ __launch_bounds__(kTailBlock) void softmax_cross_entropy_few_kernel(float const *y, float const *t, float *dy, double *partial,
                                                                               float t_sum, int pix_size, int ch_size, int frame_size,
                                                                               int frame_stride, int f_blocks)
{
    int const f = (int)(blockIdx.x % f_blocks) * kTailBlock + threadIdx.x;
    int const pix = blockIdx.x / f_blocks;
    if (f >= frame_size) { return; }
    float const eps = 1.0e-7f;
    size_t const node_step = (size_t)pix_size * frame_stride;
    size_t const first = (size_t)pix * frame_stride + f;
    float yv[CH], tv[CH];
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) {
        yv[ch] = (ch < ch_size) ? y[first + ch * node_step] : 0.0f;
        tv[ch] = (ch < ch_size) ? t[first + ch * node_step] : 0.0f;
    }
    float c = -3.402823466e+38f;
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) { if (ch < ch_size) { c = (c < yv[ch]) ? yv[ch] : c; } }
    float y_sum = 0.0f, t_max = 0.0f;
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) {
        if (ch < ch_size) {
            yv[ch] = expf(yv[ch] - c);
            y_sum += yv[ch];
            t_max += tv[ch];
        }
    }
    if (y_sum <= eps) { y_sum = eps; }
    double loss = 0.0;
#pragma unroll
    for (int ch = 0; ch < CH; ++ch) {
        if (ch < ch_size) {
            float const softmax = yv[ch] / y_sum;
            if (tv[ch] > 0.0f) { loss += (double)rounded_mul(logf(softmax + eps), t_max); }
            dy[first + ch * node_step] = (rounded_mul(t_max, softmax) - tv[ch]) / t_sum;
        }
    }
    partial[(size_t)pix * frame_size + f] = loss;
}

// The whole tail of a LUT classifier in one launch: AverageLut forward over the last layer's output (un-binarized: the logits), softmax
// cross entropy against t, categorical accuracy, and the AverageLut backward pass of the loss gradient — four launches of a few
// microseconds each when called one by one, which at training batch sizes cost their launch latencies rather than their work.
// A workgroup of CH wavefronts owns 64 frames of ALL nodes, one frame per lane and one channel per wavefront, so that the chain of dependent
// steps is that of ONE channel: at training batches the launch is latency, not work (70 -> 10 nodes: 64 frames 13.7 -> 7.1 us, 1024 frames
// 14.6 -> 8.1 us against four wavefronts that each took every channel's loss terms and walked the whole table).
//   1. wavefront ch loads its n inputs (eight in flight at a time), sums them in table order, times `scale` (as average_lut_forward_kernel);
//   2. the logits meet in LDS; wavefront ch takes their maximum and its own exponential;
//   3. the exponentials meet in LDS; wavefront ch adds them up in channel order and takes its own softmax, gradient and loss term (as
//      softmax_cross_entropy_few_kernel, pix_size 1), wavefront 0 also the accuracy (as categorical_accuracy_kernel);
//   4. the gradients dy / n and loss terms meet in LDS; wavefront 0 adds the loss terms in channel order, and wavefront w takes the inputs
//      w, w + CH, ...: the lanes compare 64 table entries at a time with the input, and the matches, ascending, add their node's gradient (the
//      order of the host loop, include/bb/AverageLut.h:395-404, and of average_lut_backward_kernel).
// Columns between frame_size and frame_stride of dx are written as 0, as the backward kernels do.  Same bits as the four entries called
// one after the other.  LDS: 5 CH x 64 floats + the table.
template <int CH>
__global__ __launch_bounds__(64 * CH) void classifier_tail_kernel(float const *__restrict__ x, float *__restrict__ y, float *__restrict__ dx,
                                                             int const *__restrict__ idx, float const *__restrict__ t,
                                                             float *__restrict__ dy_out, double *__restrict__ loss_buf,
                                                             int *__restrict__ accuracy_buf, int *__restrict__ category_buf,
                                                             float t_sum, float scale, int n, int input_node_size, int ch_size,
                                                             int frame_size, int frame_stride, int binarize_input)
{
    extern __shared__ __attribute__((aligned(16))) float tail_lds[];
    int const lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    int const total = ch_size * n;
    double *term = reinterpret_cast<double *>(tail_lds);                        // [CH][64]: loss terms
    float *logit = tail_lds + 2 * CH * 64;                                      // [CH][64]
    float *expo  = logit + CH * 64;                                             // [CH][64]: exp(logit - max), then dy / n of the lane's frame
    float *target = expo + CH * 64;                                             // [CH][64]
    int *piece   = reinterpret_cast<int *>(target + CH * 64);                   // [total]: the table
    int const f = blockIdx.x * 64 + lane;
    bool const in_row = f < frame_stride, live = f < frame_size;
    int const fc = live ? f : 0;                                                // (a lane without a frame loads frame 0 and stores nothing)
    bool const mine = wave < ch_size;                                           // wave-uniform: the wavefront has a channel
    float tv = 0.0f, yv = 0.0f;
    for (int k = threadIdx.x; k < total; k += 64 * CH) { piece[k] = idx[k]; }
    if (mine) {
        tv = t[(size_t)wave * frame_stride + fc];
        int const *row = idx + wave * n;
        float sum = 0.0f;
        for (int i0 = 0; i0 < n; i0 += 8) {
            float v[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) { v[j] = x[(size_t)row[(i0 + j < n) ? i0 + j : 0] * frame_stride + fc]; }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                if (i0 + j < n) {
                    float u = v[j];
                    if (binarize_input) { u = (u > 0.0f) ? 1.0f : -1.0f; }
                    sum += u;
                }
            }
        }
        yv = rounded_mul(sum, scale);
        logit[wave * 64 + lane]  = yv;
        target[wave * 64 + lane] = tv;
        if (live && y != nullptr) { y[(size_t)wave * frame_stride + f] = yv; }
    }
    __syncthreads();
    float const eps = 1.0e-7f;
    float ev = 0.0f;
    if (mine) {
        float c = -3.402823466e+38f;
#pragma unroll
        for (int ch = 0; ch < CH; ++ch) { if (ch < ch_size) { float const o = logit[ch * 64 + lane]; c = (c < o) ? o : c; } }
        ev = expf(yv - c);
        expo[wave * 64 + lane] = ev;
    }
    __syncthreads();
    float dyn = 0.0f;
    if (mine) {
        float y_sum = 0.0f, t_max = 0.0f;
#pragma unroll
        for (int ch = 0; ch < CH; ++ch) {
            if (ch < ch_size) {
                y_sum += expo[ch * 64 + lane];
                t_max += target[ch * 64 + lane];
            }
        }
        if (y_sum <= eps) { y_sum = eps; }
        float const softmax = ev / y_sum;
        term[wave * 64 + lane] = (tv > 0.0f) ? (double)rounded_mul(logf(softmax + eps), t_max) : 0.0;
        float const g = (rounded_mul(t_max, softmax) - tv) / t_sum;
        if (live && dy_out != nullptr) { dy_out[(size_t)wave * frame_stride + f] = g; }
        dyn = g / (float)n;
    }
    if (wave == 0 && live) {
        // accuracy: the first largest logit sits on a channel with a positive target (one pixel per frame)
        float max_y = -3.402823466e+38f, max_t = -3.402823466e+38f;
        bool valid = false;
#pragma unroll
        for (int ch = 0; ch < CH; ++ch) {
            if (ch < ch_size) {
                float const o = logit[ch * 64 + lane], tc = target[ch * 64 + lane];
                valid = valid || (tc > 0.0f);
                if (o > max_y) { max_y = o; max_t = tc; }
            }
        }
        if (accuracy_buf != nullptr) { accuracy_buf[f] = (valid && max_t > 0.0f) ? 1 : 0; }
        if (category_buf != nullptr) { category_buf[f] = valid ? 1 : 0; }
    }
    __syncthreads();                                                            // the exponentials have been read
    if (mine) { expo[wave * 64 + lane] = dyn; }
    __syncthreads();
    if (wave == 0 && live) {
        double loss = 0.0;
#pragma unroll
        for (int ch = 0; ch < CH; ++ch) {
            if (ch < ch_size && target[ch * 64 + lane] > 0.0f) { loss += term[ch * 64 + lane]; }
        }
        loss_buf[f] = loss;
    }
    for (int in = wave; in < input_node_size; in += CH) {
        float sum = 0.0f;
        for (int k0 = 0; k0 < total; k0 += 64) {
            uint64_t hits = __ballot(k0 + lane < total && piece[(k0 + lane < total) ? k0 + lane : 0] == in);
            while (hits != 0) {                                                 // wave-uniform
                int const k = k0 + (int)__builtin_ctzll(hits);
                hits &= hits - 1;
                sum += expo[(k / n) * 64 + lane];
            }
        }
        if (in_row) { dx[(size_t)in * frame_stride + f] = live ? sum : 0.0f; }
    }
}

// The same for a small batch of as many inputs as connections (each its own, as a rule): a wavefront owns four frames and all nodes, lane 16 i + ch is
// channel ch of frame i (a row of 16 lanes: what the channels exchange goes by data-parallel moves, without LDS and barriers), and every
// wavefront is a workgroup, with a compute unit of its own.
//   1. a lane loads its n inputs and sums them; while they are on the way, the wavefront counts in LDS how many connections take each input;
//   2. the row takes its maximum, every lane its exponential, the sum of the row's in channel order, its softmax, gradient and loss term; the loss terms are added
//      up in channel order, masks of the wavefront give the accuracy;
//   3. where every input is one connection's, a lane writes its gradient dy / n to those of its node; else a lane takes every 16th input and adds up what its
//      connections give it, ascending, by counts per input and node.
// The same bits.  Latency: above, a SIMD issues for four wavefronts that each go through all channels, and meet four times.  70 -> 10 nodes, 64 frames 6.35 -> 3.66 us,
// 1024 frames 6.64 -> 3.99; nodes that share inputs, 1024 frames, 6.40 -> 5.51 (11.4 where such inputs were gone through one by one), 208 -> 16 nodes 14.3 -> 9.7
// (25.2).  tail_small has both sides of its lines.
constexpr int kTailChannels = 16, kTailFrames = kWave / kTailChannels;
// the value of lane CH of the lane's row of 16
template <int CH> __device__ __forceinline__ float of_channel(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + CH, 0xf, 0xf, true));           // row_newbcast
}
template <int CH> __device__ __forceinline__ double of_channel(double v)
{
    uint64_t const b = (uint64_t)__double_as_longlong(v);
    uint32_t const lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0x150 + CH, 0xf, 0xf, true);
    uint32_t const hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), 0x150 + CH, 0xf, 0xf, true);
    return __longlong_as_double((long long)(((uint64_t)hi << 32) | lo));
}
// 0 + the values of channels 0 .. ch_size - 1 of the lane's row, in that order
template <class V, int CH = 0> __device__ __forceinline__ V sum_of_channels(V v, int ch_size, V sum = V(0))
{
    if constexpr (CH < kTailChannels) {
        if (CH < ch_size) { sum += of_channel<CH>(v); }                         // wave-uniform
        return sum_of_channels<V, CH + 1>(v, ch_size, sum);
    }
    else { return sum; }
}

// s[g] += the gradients `v` of channels 0 .. ch_size - 1 of the lane's row, in that order, each as often as its byte of count[g] says, ONCE: not more than once (adding 0 for those that have none
// leaves a sum that began as +0 as it is)
template <bool ONCE, int G, int CH = 0> __device__ __forceinline__ void add_of_takers(float (&s)[G], unsigned const (&count)[G][kTailChannels / 4], float v, int ch_size)
{
    if constexpr (CH < kTailChannels) {
        if (CH < ch_size) {                                                     // wave-uniform
            float const b = of_channel<CH>(v);
            unsigned c[G], most = 0;
#pragma unroll
            for (int g = 0; g < G; ++g) {
                c[g] = (count[g][CH / 4] >> (8 * (CH % 4))) & 0xffu;
                s[g] += c[g] != 0 ? b : 0.0f;
                most = max(most, c[g]);
            }
            if constexpr (!ONCE) {
                for (unsigned r = 1; __ballot(most > r) != 0; ++r) {
#pragma unroll
                    for (int g = 0; g < G; ++g) { s[g] += c[g] > r ? b : 0.0f; }
                }
            }
        }
        add_of_takers<ONCE, G, CH + 1>(s, count, v, ch_size);
    }
}

__global__ __launch_bounds__(kWave) void classifier_tail_small_kernel(float const *__restrict__ x, float *__restrict__ y, float *__restrict__ dx,
                                                             int const *__restrict__ idx, float const *__restrict__ t,
                                                             float *__restrict__ dy_out, double *__restrict__ loss_buf,
                                                             int *__restrict__ accuracy_buf, int *__restrict__ category_buf,
                                                             float t_sum, float scale, int n, int input_node_size, int ch_size,
                                                             int frame_size, int frame_stride, int binarize_input)
{
    __shared__ unsigned taken[kTailChannels * kTailInputs];                     // [input]: connections that take it
    __shared__ __align__(16) unsigned takers[kTailChannels * kTailInputs][kTailChannels / 4];      // [input]: a byte per node, its connections that do
    int const lane = threadIdx.x, ch = lane % kTailChannels, f = blockIdx.x * kTailFrames + lane / kTailChannels;
    int const total = ch_size * n;
    bool const in_row = f < frame_stride, live = f < frame_size, mine = ch < ch_size;
    int const fc = live ? f : 0;                                                // (a lane without a frame or channel loads another's and stores nothing)
    int const *const row = idx + (mine ? ch : 0) * n;

    for (int in = lane; in < input_node_size; in += kWave) { taken[in] = 0; }
    constexpr int kPieces = kTailChannels * kTailInputs / kWave;                // the table, 64 entries to a register
    int piece[kPieces];
#pragma unroll
    for (int q = 0; q < kPieces; ++q) { piece[q] = (q * kWave + lane < total) ? idx[q * kWave + lane] : -1; }
    float const tv = t[(size_t)(mine ? ch : 0) * frame_stride + fc];
    constexpr int kAhead = 8;
    int in[kAhead];
    float v[kAhead];
    auto request = [&](int i0) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j) { in[j] = row[(i0 + j < n) ? i0 + j : 0]; }
#pragma unroll
        for (int j = 0; j < kAhead; ++j) { v[j] = x[(size_t)in[j] * frame_stride + fc]; }
    };
    request(0);
    wave_fence();
    // (as many connections as inputs, each within them and the first to take its input: each takes one of its own)
    bool second = false;
#pragma unroll
    for (int q = 0; q < kPieces; ++q) {
        if (q * kWave + lane < total) { second |= (unsigned)piece[q] >= (unsigned)input_node_size || atomicAdd(&taken[piece[q]], 1u) != 0; }
    }
    bool const apart = total == input_node_size && __ballot(second) == 0;       // wave-uniform
    if (!apart) {
        for (int in_at = lane; in_at < input_node_size; in_at += kWave) { *reinterpret_cast<uint4 *>(takers[in_at]) = make_uint4(0, 0, 0, 0); }
        wave_fence();
#pragma unroll
        for (int q = 0; q < kPieces; ++q) {
            if ((unsigned)piece[q] < (unsigned)input_node_size) {
                int const node = (q * kWave + lane) / n;
                atomicAdd(&takers[piece[q]][node / 4], 1u << (8 * (node % 4)));
            }
        }
        wave_fence();
    }
    float sum = 0.0f;
    for (int i0 = 0; i0 < n; i0 += kAhead) {
        if (i0 > 0) { request(i0); }
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            if (i0 + j < n) {
                float u = v[j];
                if (binarize_input) { u = (u > 0.0f) ? 1.0f : -1.0f; }
                sum += u;
            }
        }
    }
    float const yv = rounded_mul(sum, scale), eps = 1.0e-7f, lowest = -3.402823466e+38f;
    float const over = (mine && lowest < yv) ? yv : lowest;                     // (never NaN)
    float c = over;
#pragma unroll
    for (int o = 1; o < kTailChannels; o <<= 1) { float const other = lane_xor(c, o); c = (c < other) ? other : c; }
    float const ev = expf(yv - c);
    float y_sum = sum_of_channels(ev, ch_size);
    float const t_max = sum_of_channels(tv, ch_size);
    if (y_sum <= eps) { y_sum = eps; }
    float const softmax = ev / y_sum;
    float const g = (rounded_mul(t_max, softmax) - tv) / t_sum;
    float const slope = g / (float)n;

    if (apart) {
        for (int i0 = 0; i0 < n; i0 += kAhead) {
            if (n > kAhead) {
#pragma unroll
                for (int j = 0; j < kAhead; ++j) { in[j] = row[(i0 + j < n) ? i0 + j : 0]; }
            }
#pragma unroll
            for (int j = 0; j < kAhead; ++j) {
                if (i0 + j < n && mine && in_row) { dx[(size_t)in[j] * frame_stride + f] = live ? 0.0f + slope : 0.0f; }
            }
        }
    }
    else {
        constexpr int kTogether = 4;                                            // inputs of a lane
        for (int i0 = 0; i0 < input_node_size; i0 += kTogether * kTailChannels) {
            unsigned count[kTogether][kTailChannels / 4], most = 0;
            float s[kTogether];
#pragma unroll
            for (int g = 0; g < kTogether; ++g) {
                int const input = i0 + g * kTailChannels + ch;
                uint4 const c = *reinterpret_cast<uint4 const *>(takers[min(input, input_node_size - 1)]);
                count[g][0] = c.x; count[g][1] = c.y; count[g][2] = c.z; count[g][3] = c.w;
                most |= c.x | c.y | c.z | c.w;
                s[g] = 0.0f;
            }
            if (__ballot((most & 0xfefefefeu) != 0) == 0) { add_of_takers<true>(s, count, slope, ch_size); }      // wave-uniform
            else                                          { add_of_takers<false>(s, count, slope, ch_size); }
#pragma unroll
            for (int g = 0; g < kTogether; ++g) {
                int const input = i0 + g * kTailChannels + ch;
                if (input < input_node_size && in_row) { dx[(size_t)input * frame_stride + f] = live ? s[g] : 0.0f; }
            }
        }
    }

    if (live && mine) {
        if (y != nullptr)      { y[(size_t)ch * frame_stride + f] = yv; }
        if (dy_out != nullptr) { dy_out[(size_t)ch * frame_stride + f] = g; }
    }
    double const term = (tv > 0.0f) ? (double)rounded_mul(logf(softmax + eps), t_max) : 0.0;
    double const loss = sum_of_channels(term, ch_size);
    // accuracy: the first largest logit sits on a channel with a positive target (one pixel per frame)
    int const shift = lane & ~(kTailChannels - 1);
    unsigned const largest = (unsigned)(__ballot(mine && over == c && yv > lowest) >> shift) & 0xffffu, wanted = (unsigned)(__ballot(mine && tv > 0.0f) >> shift) & 0xffffu;
    if (live && ch == 0) {
        loss_buf[f] = loss;
        if (accuracy_buf != nullptr) { accuracy_buf[f] = (largest & (0u - largest) & wanted) ? 1 : 0; }
        if (category_buf != nullptr) { category_buf[f] = wanted ? 1 : 0; }
    }
}

// loss_buf[frame] = sum over the pixels, ascending, of the per-pixel terms
__global__ __launch_bounds__(kTailBlock) void loss_pixel_sum_kernel(double const *partial, double *loss_buf, int pix_size, int frame_size)
{
    int const f = blockIdx.x * kTailBlock + threadIdx.x;
    if (f >= frame_size) { return; }
    double loss = 0.0;
    for (int pix = 0; pix < pix_size; ++pix) { loss += partial[(size_t)pix * frame_size + f]; }
    loss_buf[f] = loss;
}

// Per frame: pixels with a positive target (category) and, of those, pixels whose first largest y sits on a channel with
// a positive target (accuracy).  One thread per frame.
__global__ __launch_bounds__(kTailBlock) void categorical_accuracy_kernel(float const *y, float const *t, int *accuracy_buf, int *category_buf,
                                                                          int pix_size, int ch_size, int frame_size, int frame_stride)
{
    int const f = blockIdx.x * kTailBlock + threadIdx.x;
    if (f >= frame_size) { return; }
    size_t const node_step = (size_t)pix_size * frame_stride;
    int accuracy = 0, category = 0;
    for (int pix = 0; pix < pix_size; ++pix) {
        size_t const first = (size_t)pix * frame_stride + f;
        float max_y = -3.402823466e+38f, max_t = -3.402823466e+38f;
        bool valid = false;
        for (int ch = 0; ch < ch_size; ++ch) {
            float const yv = y[first + ch * node_step], tv = t[first + ch * node_step];
            valid = valid || (tv > 0.0f);
            if (yv > max_y) { max_y = yv; max_t = tv; }
        }
        if (valid) { category += 1; accuracy += (max_t > 0.0f) ? 1 : 0; }
    }
    accuracy_buf[f] = accuracy;
    category_buf[f] = category;
}

}  // namespace bbhip
