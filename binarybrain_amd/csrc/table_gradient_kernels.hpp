// Batch-norm training of small LUT layers on real-valued inputs, node by node: forward pass, and backward pass up to the dx kernel, one launch each.
#pragma once

#include "lut_kernels.hpp"

namespace bbhip {

// dW[e] = sum over frames of  d prod_j (bit_j(e) ? x_j : 1 - x_j)  is for each node a sum of outer products: with the corner products of inputs
// 0, 1 as a column and those of inputs 2, 3 as a row, one v_mfma_f32_4x4x1_16b_f32 adds the 4 x 4 products of sixteen frames, a quad of lanes
// each, in the time of two vector instructions where 16 fused multiply-adds per lane and four frames would take four.  Inputs 4 and 5 double the
// columns and the rows: four products per frame, sixteen accumulator registers per lane and set instead of 64, and the sum over the quads at the
// end takes 30 instructions instead of a transposition of 64 registers through LDS.  That end is what pays in a small layer; over long slabs of
// frames the operands (44 instructions per 64 frames and the 16 products) take longer than the 64 multiply-adds.
//
// Lane 4 b + r of quad b supplies entry r of column and row.  The four frames of a quad take turns (t): entry r of frame 4 b + t needs that frame's
// inputs in all four lanes, which a data-parallel move brings as an operand of the instruction that uses it.  A corner factor is one addition: x
// where the lane's corner has the bit set, x - 1 = -(1 - x) where it has not; the sign is applied to the sum.
//
// Rounding: every term is formed with its own factors before it is added (a sum of the terms with 1 - x taken as the difference of two sums without
// that factor rounds to the size of those: 1.0e-7 of the largest entry for six inputs and 1000 frames where this gives 4.3e-8 and multiply-adds
// per lane in slabs 4.9e-8, rms against 64 bits).  A register is one chain of four additions per 64 frames, or of two where the turns go to two SETS of
// accumulators.  The callers add at most 256 frames between two totals, or 512 with two sets, which keeps the error of every width at or below that
// of the multiply-adds.
template <int N, int SETS>
struct TableGradient {
    static constexpr int CQ = (N > 4) ? 2 : 1, RQ = (N > 5) ? 2 : 1, R = 4 * CQ * RQ;
    mfma_f4 acc[SETS][RQ][CQ];
    float c0, c1;                   // 0 or -1: what the lane adds to inputs 0 / 2 and 1 / 3

    __device__ __forceinline__ void clear(int lane)
    {
#pragma unroll
        for (int i = 0; i < SETS * RQ * CQ; ++i) { acc[i / (RQ * CQ)][i / CQ % RQ][i % CQ] = mfma_f4{0.0f, 0.0f, 0.0f, 0.0f}; }
        c0 = (lane & 1) ? 0.0f : -1.0f;
        c1 = (lane & 2) ? 0.0f : -1.0f;
    }

    template <int T>
    __device__ __forceinline__ static float quad_lane(float v)
    {
        return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), T * 0x55, 0xf, 0xf, true));
    }

    template <int T>
    __device__ __forceinline__ void add_turn(float const (&x)[N], float d)
    {
        float col[CQ], row[RQ];
        col[0] = quad_lane<T>(d) * ((quad_lane<T>(x[0]) + c0) * (quad_lane<T>(x[1]) + c1));
        if constexpr (N >= 4)      { row[0] = (quad_lane<T>(x[2]) + c0) * (quad_lane<T>(x[3]) + c1); }
        else if constexpr (N == 3) { row[0] = quad_lane<T>(x[2]) + c0; }
        else                       { row[0] = 1.0f; }
        if constexpr (CQ == 2) { col[1] = quad_lane<T>(x[N > 4 ? 4 : 0]) * col[0]; col[0] = col[1] - col[0]; }
        if constexpr (RQ == 2) { row[1] = quad_lane<T>(x[N > 5 ? 5 : 0]) * row[0]; row[0] = row[1] - row[0]; }
#pragma unroll
        for (int q = 0; q < RQ; ++q) {
#pragma unroll
            for (int p = 0; p < CQ; ++p) { acc[T % SETS][q][p] = __builtin_amdgcn_mfma_f32_4x4x1f32(col[p], row[q], acc[T % SETS][q][p], 0, 0, 0); }
        }
    }
    // 64 frames, one per lane: inputs in [0, 1] and the gradient of the LUT output (0 where the frame does not count)
    __device__ __forceinline__ void add(float const (&x)[N], float d)
    {
        add_turn<0>(x, d); add_turn<1>(x, d); add_turn<2>(x, d); add_turn<3>(x, d);
    }

    // what of (a, b) a lane keeps and adds up over lane and lane ^ M: lanes without bit M keep a, the others b
    template <int M>
    __device__ __forceinline__ static float fold_pair(float a, float b, int lane)
    {
        if constexpr (M == 32) {
            auto const s = __builtin_amdgcn_permlane32_swap(__float_as_int(a), __float_as_int(b), false, false);
            return __int_as_float(s[0]) + __int_as_float(s[1]);
        }
        else if constexpr (M == 16) {
            auto const s = __builtin_amdgcn_permlane16_swap(__float_as_int(a), __float_as_int(b), false, false);
            return __int_as_float(s[0]) + __int_as_float(s[1]);
        }
        else {
            float const mine = (lane & M) ? b : a, other = (lane & M) ? a : b;
            return mine + lane_xor(other, M);
        }
    }
    template <int M, int COUNT>
    __device__ __forceinline__ static float fold(float const (&v)[COUNT], int lane)
    {
        // the register index goes to the lane bits from the top that hold it: lane bits 5 .. 2 are the quads
        if constexpr (M == 2) { return v[0]; }
        else if constexpr (COUNT * 4 > M) {
            float h[COUNT / 2];
#pragma unroll
            for (int r = 0; r < COUNT / 2; ++r) { h[r] = fold_pair<M>(v[r], v[r + COUNT / 2], lane); }
            return fold<M / 2, COUNT / 2>(h, lane);
        }
        else {
            float h[COUNT];
#pragma unroll
            for (int r = 0; r < COUNT; ++r) { h[r] = v[r] + lane_xor(v[r], M); }
            return fold<M / 2, COUNT>(h, lane);
        }
    }

    // the sums over the wavefront: in lane L the entry table_entry(L) of the node's table (narrow tables: several lanes hold the same entry)
    __device__ __forceinline__ float total(int lane) const
    {
        float v[R];
#pragma unroll
        for (int q = 0; q < RQ; ++q) {
#pragma unroll
            for (int p = 0; p < CQ; ++p) {
#pragma unroll
                for (int r = 0; r < 4; ++r) { v[(q * CQ + p) * 4 + r] = SETS == 2 ? acc[0][q][p][r] + acc[SETS - 1][q][p][r] : acc[0][q][p][r]; }
            }
        }
        float s = fold<32, R>(v, lane);
        // register index = ((bit of input 5) (bit of input 4) (bit of input 1) (bit of input 0)); a sign for each factor 1 - x
        int zeros = 2 - ((lane >> 2) & 1) - ((lane >> 3) & 1);
        if (N >= 3) { zeros += 1 - (lane & 1); }
        if (N >= 4) { zeros += 1 - ((lane >> 1) & 1); }
        if (N >= 5) { zeros += 1 - ((lane >> 4) & 1); }
        if (N >= 6) { zeros += 1 - ((lane >> 5) & 1); }
        return (zeros & 1) ? -s : s;
    }
    __device__ __forceinline__ static int table_entry(int lane)
    {
        int e = ((lane >> 2) & 1) | (((lane >> 3) & 1) << 1);
        if (N >= 3) { e |= (lane & 1) << 2; }
        if (N >= 4) { e |= ((lane >> 1) & 1) << 3; }
        if (N >= 5) { e |= ((lane >> 4) & 1) << 4; }
        if (N >= 6) { e |= ((lane >> 5) & 1) << 5; }
        return e;
    }
    // one lane per entry writes it
    __device__ __forceinline__ static bool owns_entry(int lane)
    {
        if (N == 2) { return (lane & ~0xc) == 0; }
        if (N == 3) { return (lane & ~0xd) == 0; }
        return lane < (1 << N);
    }
};

// inputs of a wavefront step as the LUT sees them (reference: include/bb/StochasticLutN.h:542)
template <int N>
__device__ __forceinline__ void input_values(uint32_t const (&raw)[N], float (&x)[N])
{
#pragma unroll
    for (int k = 0; k < N; ++k) { x[k] = __builtin_amdgcn_fmed3f(__uint_as_float(raw[k]), 0.0f, 1.0f); }
}

// The LUT output of a frame from its inputs, where the batch-norm kinds need it: the node's table on the matrix unit where its width allows
template <int N>
struct LutOutput {
    using D = LutDims<N>;
    static constexpr bool kMatrix = LutMatrixQ<N>::kUsable;
    LutMatrixQ<N> mq;
    float C[kMatrix ? 1 : D::NN], cv[kMatrix ? 1 : D::H];
    // the centred table, one entry per lane
    __device__ __forceinline__ void take(float c, int lane)
    {
        if constexpr (kMatrix) { mq.take(c, lane); }
        else {
#pragma unroll
            for (int i = 0; i < D::NN; ++i) { C[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(c), i)); }
            LutEval<N>::pin_constants(C, cv);
        }
    }
    __device__ __forceinline__ float operator()(float const (&x)[N]) const
    {
        float z[N];
#pragma unroll
        for (int k = 0; k < N; ++k) { z[k] = x[k] - 0.5f; }
        if constexpr (kMatrix) { return mq.forward(z); }
        else                   { return LutEval<N>::forward(C, cv, z); }
    }
};

// Batch-norm training pass over real-valued inputs in one launch: a.node_waves wavefronts take a node and all its frames, keep the LUT outputs of
// their up to kNodeSteps steps in registers, exchange the sums of the statistics and write the batch-norm output.  The node's table is derived in
// the wavefront (as in lut_forward_kernel), so that the pass has neither a table launch nor a statistics launch nor a second gather.
constexpr int kNodeSteps = 4, kNodeWaves = 16;

template <int N>
__global__ __launch_bounds__(kNodeWaves * kWave) void lut_forward_node_kernel(FwdArgs a)
{
    constexpr int NN = 1 << N, U = 2;
    int const wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave)), waves = blockDim.x / kWave;
    int const lane = threadIdx.x & (kWave - 1);
    int const nw = a.node_waves, sub = wave % nw, slot = wave / nw;
    int node = xcd_remap(blockIdx.x, a.tiles.count) * (waves / nw) + slot;
    bool const live = node < a.node_size;
    if (!live) { node = a.node_size - 1; }                              // (barriers ahead: repeats the last node and stores nothing)

    void const *rows[N];
#pragma unroll
    for (int k = 0; k < N; ++k) { rows[k] = reinterpret_cast<float const *>(a.x) + (size_t)a.idx[node * N + k] * a.x_stride; }
    int const i = lane & (NN - 1);
    float w = a.W_inline[(size_t)node * NN + i];
    bool clamp_store = false;
    if (a.clamp_W != nullptr) {
        float const wc = fminf(a.clamp_hi, fmaxf(a.clamp_lo, w));
        clamp_store = (wc != w);
        w = wc;
    }
    float const table_w = w;
    if (a.lut_binarize) { w = (w > 0.5f) ? 1.0f : 0.0f; }
    float const c = centred_butterfly<N>(w, i);
    float const c0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(c)));
    LutOutput<N> output;
    output.take(c, lane);

    int const f_begin = sub * kNodeSteps * kWave, f_end = min(f_begin + kNodeSteps * kWave, a.frame_size), f_last = a.frame_size - 1;
    float v[kNodeSteps], s1 = 0.0f, s2 = 0.0f;
    uint32_t raw[2][U][N];                                              // the next steps' operands are requested before the present ones are used
    auto request = [&](int fb, uint32_t (&r)[U][N]) {
#pragma unroll
        for (int u = 0; u < U; ++u) { Gather<N, kXClamp>::load_raw(rows, fb + u * kWave, lane, f_last, r[u]); }
    };
    request(f_begin, raw[0]);
#pragma unroll
    for (int s = 0; s < kNodeSteps; s += U) {
        int const fb = f_begin + s * kWave;
        if (fb >= f_end) { break; }                                     // wave-uniform
        if (s + U < kNodeSteps && fb + U * kWave < f_end) { request(fb + U * kWave, raw[(s / U + 1) & 1]); }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float x[N];
            input_values<N>(raw[(s / U) & 1][u], x);
            v[s + u] = output(x);
            float const d = (fb + u * kWave + lane < f_end) ? v[s + u] - c0 : 0.0f;
            s1 += d;
            s2 = __builtin_fmaf(d, d, s2);
        }
    }
    // (as the statistics launch and the output launch of larger layers add them: the same bits)
    s1 = wave_sum(s1);
    s2 = wave_sum(s2);
    __shared__ float sums[kNodeWaves][2];
    if (lane == 0) { sums[wave][0] = s1; sums[wave][1] = s2; }
    __syncthreads();
    s1 = wave_sum(lane < nw ? sums[slot * nw + (lane < nw ? lane : 0)][0] : 0.0f);
    s2 = wave_sum(lane < nw ? sums[slot * nw + (lane < nw ? lane : 0)][1] : 0.0f);
    if (!live) { return; }
    float mean, var, rstd;
    batch_statistics(s1, s2, c0, a.frame_size, mean, var, rstd);
    float *const row = reinterpret_cast<float *>(a.y) + (size_t)node * a.y_stride;
#pragma unroll
    for (int s = 0; s < kNodeSteps; ++s) {
        int const f = f_begin + s * kWave + lane;
        if (f < f_end) { __builtin_nontemporal_store(__builtin_amdgcn_fmed3f(batch_norm_output(v[s], mean, rstd, a.gamma, a.beta), 0.0f, 1.0f), row + f); }
    }
    if (sub != 0) { return; }
    if (lane == 0) { store_statistics(a.mean_out, a.rstd_out, a.running_mean, a.running_var, node, mean, var, rstd, a.momentum); }
    if (lane < NN) {
        if (clamp_store)        { a.clamp_W[(size_t)node * NN + lane] = table_w; }
        if (a.C_out != nullptr) { a.C_out[(size_t)node * NN + lane] = c; }
    }
}

struct NodeGradientArgs {
    void const  *x;
    float const *dy;
    int const   *idx;
    int   node_size, frame_size, x_stride, dy_stride;
    int   node_tiles;               // workgroups of nodes
    int   node_waves;               // wavefronts per node, of kNodeSteps steps each
    float *dW;
    int   overwrite;                // dW = instead of +=
    float const *W, *C;             // the table, or the centred one of the forward call (C not null)
    int   lut_binarize;
    float const *mean, *rstd;
    float gamma, beta, inv_frames;
    float *dyh;  int dyh_stride;    // dL/d(LUT output), for the dx kernel
    TermArgs tt;                    // the last tt.blocks workgroups build the dx kernel's term table
};

// Backward pass through batch-norm in one launch ahead of the dx kernel: a.node_waves wavefronts take a node and all its frames, as in
// lut_forward_node_kernel.  A first pass leaves the LUT output and the gated dy of each frame in registers and its sums in LDS, a second one adds
// the table gradient and writes dL/d(LUT output).
// Bound by its chain: wiring, rows, table, sums, rows again, reduction.  Measured, training step (with the forward pass above: three launches
// instead of six): 1024 x 1024 x 1000 46.7 -> 34.6 us, 64 x 64 x 100 25.7 -> 16.4 us.
template <int N>
__global__ __launch_bounds__(kNodeWaves * kWave) void lut_node_gradient_kernel(NodeGradientArgs a)
{
    constexpr int NN = 1 << N, U = 2;
    int const bid = blockIdx.x;
    if (bid >= a.node_tiles) {
        // the term table of the dx kernel depends on nothing this launch computes: its workgroups ride at the end
        if (threadIdx.x < kBlock) { term_table_node_block<N>(a.tt, bid - a.node_tiles); }
        return;
    }
    int const wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave)), waves = blockDim.x / kWave;
    int const lane = threadIdx.x & (kWave - 1);
    int const nw = a.node_waves, sub = wave % nw, slot = wave / nw;
    int node = xcd_remap(bid, a.node_tiles) * (waves / nw) + slot;
    bool const live = node < a.node_size;
    if (!live) { node = a.node_size - 1; }                              // (barriers ahead: repeats the last node and stores nothing)

    void const *rows[N];
#pragma unroll
    for (int k = 0; k < N; ++k) { rows[k] = reinterpret_cast<float const *>(a.x) + (size_t)a.idx[node * N + k] * a.x_stride; }
    float const *dyr = a.dy + (size_t)node * a.dy_stride;
    int const f_begin = sub * kNodeSteps * kWave, f_end = min(f_begin + kNodeSteps * kWave, a.frame_size), f_last = a.frame_size - 1;

    uint32_t raw[2][U][N];                                              // the next steps' operands are requested before the present ones are used
    float dy[kNodeSteps];
    auto request = [&](int fb, uint32_t (&r)[U][N]) {
#pragma unroll
        for (int u = 0; u < U; ++u) { Gather<N, kXClamp>::load_raw(rows, fb + u * kWave, lane, f_last, r[u]); }
    };
    request(f_begin, raw[0]);
#pragma unroll
    for (int s = 0; s < kNodeSteps; ++s) {
        dy[s] = __builtin_nontemporal_load(reinterpret_cast<float const *>(reinterpret_cast<char const *>(dyr) + (uint32_t)min(f_begin + s * kWave + lane, f_last) * 4u));
    }

    float const mean = a.mean[node], rstd = a.rstd[node], gain = a.gamma * rstd;
    int const i = lane & (NN - 1);
    float c;
    if (a.C != nullptr) { c = a.C[(size_t)node * NN + i]; }
    else {
        c = a.W[(size_t)node * NN + i];
        if (a.lut_binarize) { c = (c > 0.5f) ? 1.0f : 0.0f; }
        c = centred_butterfly<N>(c, i);
    }
    LutOutput<N> output;
    output.take(c, lane);

    // dL/d(LUT output) of a frame is  g gain + shift + (v - mean) scale, g = dy behind the hard-tanh window (reference: DifferentiableLutN.h:1206-1250)
    float v[kNodeSteps], g[kNodeSteps], s0 = 0.0f, s1 = 0.0f;
#pragma unroll
    for (int s = 0; s < kNodeSteps; s += U) {
        int const fb = f_begin + s * kWave;
        if (fb >= f_end) { break; }                                     // wave-uniform
        if (s + U < kNodeSteps && fb + U * kWave < f_end) { request(fb + U * kWave, raw[(s / U + 1) & 1]); }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float x[N];
            input_values<N>(raw[(s / U) & 1][u], x);
            float const y = output(x), t = batch_norm_output(y, mean, rstd, a.gamma, a.beta);
            v[s + u] = y - mean;
            g[s + u] = (fb + u * kWave + lane < f_end && t > 0.0f && t < 1.0f) ? dy[s + u] : 0.0f;
            s0 += g[s + u];
            s1 = __builtin_fmaf(g[s + u], v[s + u], s1);
        }
    }
    request(f_begin, raw[0]);                                           // (on the way while the sums are formed)
    s0 = wave_sum(s0);
    s1 = wave_sum(s1);
    __shared__ float sums[kNodeWaves][2], part[kNodeWaves][kWave];
    if (nw > 1) {
        if (lane == 0) { sums[wave][0] = s0; sums[wave][1] = s1; }
        __syncthreads();
        s0 = 0.0f; s1 = 0.0f;
        for (int k = 0; k < nw; ++k) { s0 += sums[slot * nw + k][0]; s1 += sums[slot * nw + k][1]; }
    }
    float const shift = -(a.gamma * s0) * rstd * a.inv_frames;
    float const scale = -(a.gamma * s1) * (rstd * rstd) * rstd * a.inv_frames;

    using Gradient = TableGradient<N, N <= 4 ? 2 : 1>;
    Gradient grad;
    grad.clear(lane);
#pragma unroll
    for (int s = 0; s < kNodeSteps; s += U) {
        int const fb = f_begin + s * kWave;
        if (fb >= f_end) { break; }
        if (s + U < kNodeSteps && fb + U * kWave < f_end) { request(fb + U * kWave, raw[(s / U + 1) & 1]); }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            int const f = fb + u * kWave + lane;
            float x[N];
            input_values<N>(raw[(s / U) & 1][u], x);
            float const d = (f < f_end) ? __builtin_fmaf(g[s + u], gain, __builtin_fmaf(v[s + u], scale, shift)) : 0.0f;
            if (live && f < f_end) { a.dyh[(size_t)node * a.dyh_stride + f] = d; }
            grad.add(x, d);
        }
    }
    float sum = grad.total(lane);
    if (nw > 1) {
        part[wave][lane] = sum;
        __syncthreads();
        if (sub != 0) { return; }
        for (int k = 1; k < nw; ++k) { sum += part[wave + k][lane]; }
    }
    if (live && Gradient::owns_entry(lane)) {
        float *out = a.dW + (size_t)node * NN + Gradient::table_entry(lane);
        *out = a.overwrite ? sum : *out + sum;
    }
}

}  // namespace bbhip
