// Backward pass of a small StochasticLut layer on real-valued inputs in one launch: table gradient and dx.
#pragma once

#include "table_gradient_kernels.hpp"

namespace bbhip {

// dV/dx_k of a node, a polynomial of the other M inputs, from the node's table held one entry per lane
template <int N>
struct LutSlope {
    static constexpr int M = N - 1, HN = 1 << M;
    static constexpr bool kMatrix = M >= 3;
    static constexpr int ML = kMatrix ? M / 2 : 0, MH = M - ML, L = 1 << ML, H = 1 << MH;
    static_assert(!kMatrix || (H % 4 == 0 && (H / 4) * L <= 16), "the coefficients fill at most one register");
    float t;
    float c[kMatrix ? 1 : HN];

    // w: W' (lane e: entry e, repeated over the wavefront); k is the same in every lane
    __device__ __forceinline__ void take(float w, int k, int lane)
    {
        // coefficients of the plain basis, (a, b) -> (a, b - a) per index bit; those of the slope are the entries with bit k set
#pragma unroll
        for (int j = 0; j < N; ++j) {
            float const o = lane_xor(w, 1 << j);
            w = ((lane >> j) & 1) ? (w - o) : w;
        }
        int s = lane & (HN - 1);
        if constexpr (kMatrix) {                            // lane 4 u + r: the coefficient of result r in update u (LutMatrixQ)
            int const u = lane >> 2, e = (4 * (u / L) + (lane & 3)) * L + u % L;
            s = e & (HN - 1);
        }
        int const entry = (s & ((1 << k) - 1)) | (1 << k) | ((s >> k) << (k + 1));
        t = __int_as_float(__builtin_amdgcn_ds_bpermute(entry << 2, __float_as_int(w)));
        if constexpr (!kMatrix) {
#pragma unroll
            for (int i = 0; i < HN; ++i) { c[i] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(t), i)); }
        }
    }
    __device__ __forceinline__ float operator()(float const (&x)[M]) const
    {
        float q[H];
        if constexpr (kMatrix) {
            float xl[ML > 0 ? ML : 1], l[L];
#pragma unroll
            for (int j = 0; j < ML; ++j) { xl[j] = x[j]; }
            monomials<ML>(xl, l);
            mfma_broadcast_matvec<H / 4, L>(t, l, q);
        }
        else {
#pragma unroll
            for (int i = 0; i < H; ++i) { q[i] = c[i]; }
        }
#pragma unroll
        for (int v = 0; v < MH; ++v) {                      // Horner over the high variables
#pragma unroll
            for (int i = 0; i < (H >> (v + 1)); ++i) { q[i] = __builtin_fmaf(x[ML + v], q[2 * i + 1], q[2 * i]); }
        }
        return q[0];
    }
};

struct SmallBackwardArgs {
    DxArgs dx;                      // rows, work lists, units and split mode as in lut_dx_kernel (no term table, no rider)
    int const   *idx;
    float const *W;
    int   lut_binarize, node_size;
    float *dW;
    int   overwrite;                // dW = instead of +=
    int   node_waves, node_tiles;   // table gradient: wavefronts that share a node, and workgroups
};

// A small layer's launches wait for one another, not for the device: here the workgroups of the table gradient and those of dx share one, which the
// dx kernel of larger layers cannot because its terms' coefficients come from a table that a launch ahead of it builds.  The first node_tiles
// workgroups take nodes, node_waves wavefronts for the frames of each (as lut_node_gradient_kernel; dW is written directly, there are no partial
// sums to fold).  The others take an input and U x 64 frames each and walk the input's consumers; a term's coefficients are derived in the
// wavefront (one load of the table, N lane exchanges, one permutation), and the matrix unit, whose operand a lane quad can hand to all the
// others, spares the 2^(N-1) moves to scalar registers.  That is 40 vector instructions per term more than lut_dx_kernel has.
// Training step (with the forward pass that derives its tables, two launches instead of four): 100 inputs x 100 nodes x 300 frames 18.2 -> 11.5 us,
// 300 x 1000 x 500 20.7 -> 16.6, 4000 x 400 x 2000 32.8 -> 24.9.
// WIDE: the four steps of a lane are four consecutive frames of rows that hold whole groups of four, one load each (lut_dx_kernel): 1001 inputs x 1531
// nodes x 1999 frames, four inputs per node, 26.6 us a training step instead of 30.6.
// (waves_per_eu: results of the matrix unit in ordinary registers, without a move for each)
template <int N, int U, int WAVES, bool WIDE = false>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(2))) void lut_small_backward_kernel(SmallBackwardArgs s)
{
    static_assert(!WIDE || U == 4, "four frames per lane");
    constexpr int NN = 1 << N, M = N - 1;
    DxArgs const &a = s.dx;
    int const lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    __shared__ float part[WAVES][U][kWave];

    if ((int)blockIdx.x < s.node_tiles) {
        int const nw = s.node_waves, sub = wave % nw, slot = wave / nw;
        int node = xcd_remap(blockIdx.x, s.node_tiles) * (WAVES / nw) + slot;
        bool const live = node < s.node_size;
        if (!live) { node = s.node_size - 1; }                          // (a barrier ahead: repeats the last node and stores nothing)
        void const *rows[N];
#pragma unroll
        for (int k = 0; k < N; ++k) { rows[k] = reinterpret_cast<float const *>(a.x) + (size_t)s.idx[node * N + k] * a.x_stride; }
        float const *dyr = a.dy + (size_t)node * a.dy_stride;
        int const steps = (a.frame_size + kWave - 1) / kWave, f_last = a.frame_size - 1;
        int const f_begin = (steps * sub / nw) * kWave, f_end = min((steps * (sub + 1) / nw) * kWave, a.frame_size);

        constexpr int S = 2;                                            // wavefront-steps whose loads are issued together
        struct Operands { uint32_t x[S][N]; float dy[S]; };
        auto request = [&](int fb, Operands &o) {
#pragma unroll
            for (int u = 0; u < S; ++u) {
                Gather<N, kXClamp>::load_raw(rows, fb + u * kWave, lane, f_last, o.x[u]);
                o.dy[u] = *reinterpret_cast<float const *>(reinterpret_cast<char const *>(dyr) + (uint32_t)min(fb + u * kWave + lane, f_last) * 4u);
            }
        };
        using Gradient = TableGradient<N, 2>;
        Gradient grad;
        grad.clear(lane);
        auto add = [&](int fb, Operands const &o) {
#pragma unroll
            for (int u = 0; u < S; ++u) {
                float x[N];
                input_values<N>(o.x[u], x);
                grad.add(x, (fb + u * kWave + lane < f_end) ? o.dy[u] : 0.0f);
            }
        };
        float sum = 0.0f;
        Operands o0, o1;
        if (f_begin < f_end) { request(f_begin, o0); }
        for (int fb = f_begin; fb < f_end; fb += 2 * S * kWave) {
            if (fb + S * kWave < f_end) { request(fb + S * kWave, o1); }
            add(fb, o0);
            if (fb + 2 * S * kWave < f_end) { request(fb + 2 * S * kWave, o0); }
            if (fb + S * kWave < f_end) { add(fb + S * kWave, o1); }
            // chains of at most 512 frames (TableGradient)
            if (((fb - f_begin) & 511) == 512 - 2 * S * kWave && fb + 2 * S * kWave < f_end) { sum += grad.total(lane); grad.clear(lane); }
        }
        sum += grad.total(lane);
        if (nw > 1) {
            part[wave][0][lane] = sum;
            __syncthreads();
            if (sub != 0) { return; }
            for (int k = 1; k < nw; ++k) { sum += part[wave + k][0][lane]; }
        }
        if (live && Gradient::owns_entry(lane)) {
            float *out = s.dW + (size_t)node * NN + Gradient::table_entry(lane);
            *out = s.overwrite ? sum : *out + sum;
        }
        return;
    }

    int const lid = xcd_remap((int)blockIdx.x - s.node_tiles, a.chunk_count * a.tiles.count);
    int ck, tile;
    split_tile(lid, a.tiles, ck, tile);
    int in, share;
    dx_list_share(a, tile, wave, in, share);
    if (in >= a.input_node_size) { return; }                            // (workgroup-uniform in split mode)

    typedef __attribute__((address_space(4))) int const const_int;
    const_int *list = (const_int *)(a.rev + (size_t)in * a.rev_stride);
    const_int *idx = (const_int *)s.idx;
    int t_begin, t_end;
    dx_list_range<WAVES>(list[0], share, t_begin, t_end);
    list += 1;
    // whole buffers of less than 4 GiB: rows are 32-bit offsets into them, and a lane past the last frame reads what lies there (its sum is not stored)
    uint32_t const x_pitch = (uint32_t)a.x_stride * 4u, y_pitch = (uint32_t)a.dy_stride * 4u;
    uint32_t const row_bytes = (uint32_t)(WIDE ? (a.frame_size + 3) & ~3 : a.frame_size) * 4u;
    __amdgpu_buffer_rsrc_t const xr = row_descriptor(a.x, 0, 0, (uint32_t)(a.input_node_size - 1) * x_pitch + row_bytes);
    __amdgpu_buffer_rsrc_t const yr = row_descriptor(a.dy, 0, 0, (uint32_t)(s.node_size - 1) * y_pitch + row_bytes);
    __amdgpu_buffer_rsrc_t const wr = row_descriptor(s.W, 0, 0, (uint32_t)s.node_size * (NN * 4u));
    int const f_begin = ck * U * kWave;
    uint32_t const off = (uint32_t)(f_begin + (WIDE ? U : 1) * lane) * 4u;

    // a term's wiring and table are requested while the term before it is evaluated (and not looked at before), its list entry another term ahead
    struct Head { int ins[N]; float w; int node, k; };
    auto head = [&](int e, Head &h) {
        uint32_t const node = (uint32_t)e / (uint32_t)N;
        h.node = (int)node;
        h.k = e - (int)node * N;
        h.w = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(wr, (lane & (NN - 1)) * 4, node * (NN * 4u), 0));
#pragma unroll
        for (int j = 0; j < N; ++j) { h.ins[j] = idx[node * N + j]; }
    };
    float acc[U];
#pragma unroll
    for (int u = 0; u < U; ++u) { acc[u] = 0.0f; }
    Head next;
    int e_ahead = 0;
    if (t_begin < t_end) {
        head(list[t_begin], next);
        e_ahead = list[min(t_begin + 1, t_end - 1)];
    }
    for (int t = t_begin; t < t_end; ++t) {
        Head const h = next;
        uint32_t raw[U][M];
        float dy[U];
#pragma unroll
        for (int j = 0; j < M; ++j) {
            uint32_t const row = (uint32_t)(j < h.k ? h.ins[j] : h.ins[j + 1]) * x_pitch;
            if constexpr (WIDE) {
                auto const q = __builtin_amdgcn_raw_buffer_load_b128(xr, off, row, 0);
#pragma unroll
                for (int u = 0; u < U; ++u) { raw[u][j] = q[u]; }
                continue;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) { raw[u][j] = __builtin_amdgcn_raw_buffer_load_b32(xr, off + u * (kWave * 4u), row, 0); }
        }
        if constexpr (WIDE) {
            auto const q = __builtin_amdgcn_raw_buffer_load_b128(yr, off, (uint32_t)h.node * y_pitch, 0);
#pragma unroll
            for (int u = 0; u < U; ++u) { dy[u] = __uint_as_float(q[u]); }
        }
        else {
#pragma unroll
        for (int u = 0; u < U; ++u) { dy[u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(yr, off + u * (kWave * 4u), (uint32_t)h.node * y_pitch, 0)); }
        }
        LutSlope<N> slope;
        slope.take(s.lut_binarize ? (h.w > 0.5f ? 1.0f : 0.0f) : h.w, h.k, lane);
        __builtin_amdgcn_sched_barrier(0);              // (the permutation is waited for with the scalar loads issued ahead of it: none of the next term's)
        if (t + 1 < t_end) {
            head(e_ahead, next);
            e_ahead = list[min(t + 2, t_end - 1)];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            float x[M];
            input_values<M>(raw[u], x);
            acc[u] = __builtin_fmaf(dy[u], slope(x), acc[u]);
        }
    }
    dx_store_pass<U, WAVES, WIDE>(a, part, in, wave, lane, f_begin, acc);
}

}  // namespace bbhip
