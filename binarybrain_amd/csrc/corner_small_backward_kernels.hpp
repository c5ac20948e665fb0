// Backward pass of a small layer on two-valued inputs in one launch: table gradient and dx.
#pragma once

#include "corner_backward_kernels.hpp"

namespace bbhip {

struct CornerSmallArgs {
    CornerSumsArgs sums;        // one slab, no indices kept, no node constants
    DxArgs dx;                  // work lists, split mode and rows
    int   dx_blocks;            // the first workgroups: dx; the others: a node per wavefront
    float inv_step;             // 1 / (hi - lo)
};

// The corner indices of a wavefront's frames, four consecutive ones per lane and pass of 256 frames, from the words that request_corner_words loaded
template <int N, int PASSES>
struct CornerQuads {
    // one pass: the lane loads the word that holds its frames; more: a lane loads 32 frames, and the indices change lanes through LDS
    static constexpr bool kExchange = PASSES > 1;
    __device__ __forceinline__ static uint32_t offset(int lane) { return (uint32_t)(kExchange ? lane : lane >> 3) * 4u; }
    __device__ __forceinline__ static void form(uint32_t const (&w)[N], int lane, uint32_t *shared, uint32_t (&at)[PASSES])
    {
        if constexpr (kExchange) {
            uint32_t quad[8];
            corner_bytes<N>(w, quad);
            wave_fence();
            if (lane < PASSES * 8) {
                uint4 *ex = reinterpret_cast<uint4 *>(shared + 8 * lane);
                ex[0] = make_uint4(quad[0], quad[1], quad[2], quad[3]);
                ex[1] = make_uint4(quad[4], quad[5], quad[6], quad[7]);
            }
            wave_fence();
#pragma unroll
            for (int p = 0; p < PASSES; ++p) { at[p] = shared[p * kWave + lane]; }
        }
        else {
            at[0] = 0;
#pragma unroll
            for (int k = 0; k < N; ++k) {           // bits 0 .. 3 to bits 0, 8, 16, 24 (the four copies that the product adds up do not meet)
                uint32_t const nibble = __builtin_amdgcn_ubfe(w[k], (uint32_t)(4 * (lane & 7)), 4u);
                at[0] |= (__umul24(nibble, 0x00204081u) & 0x01010101u) << k;
            }
        }
    }
};

constexpr int kCornerSmallItems = kWave;        // items of a work list that a wavefront walks: one per lane

// Batch-norm: what a frame takes from its corner: V - mean, dV/dx_k, and all bits set where the corner lies inside the hard-tanh window
struct __align__(16) CornerSlope { float above_mean, slope; uint32_t open, unused; };

// both sums over the wavefront: the halves of it add up one each
__device__ __forceinline__ void wave_sum_pair(float &s0, float &s1)
{
    auto const h = __builtin_amdgcn_permlane32_swap(__float_as_int(s0), __float_as_int(s1), false, false);
    float s = __int_as_float(h[0]) + __int_as_float(h[1]);              // lanes 0 .. 31: of s0, 32 .. 63: of s1
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) { s += lane_xor(s, o); }
    s0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 0));
    s1 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(s), 32));
}

template <int N, bool BN, int PASSES>
struct CornerSmallDxShared {            // a wavefront's LDS
    __align__(16) std::conditional_t<BN, CornerSlope, float> table[1 << N];
    __align__(16) uint32_t quads[PASSES > 1 ? PASSES * kWave : 4];
    float4 part[PASSES][kWave];
};

// dx[input][all frames] by one wavefront (or, in split mode, the WAVES wavefronts of a workgroup), consumer by consumer in the reverse table's order.  A
// wavefront sees all frames of a consumer, so it forms the two sums that the gradient through the statistics needs (s0, s1 of
// corner_backward_kernels.hpp) itself instead of waiting for a launch that does: as many times as the node has inputs, but side by side.
// The lists are in registers (lane l: an item, its node's wiring and statistics), and the next item's rows are requested while one is evaluated, on
// every path alike: an item past the end reads from buffers of no length.
// Bound by latency: an item takes 0.45 us of a wavefront's time (256 frames; 0.75 and 1.1 with 512 and 1024), about 160 instructions that wait for one
// another, a launch 4.5 to 5 us.  Backward call of 1024 inputs x 360 nodes x 256 frames 9.0 -> 5.8 us, 784 x 1024 9.4 -> 6.2, 360 x 70 x 1024
// 8.8 -> 5.9 (the rule with both sides of the line: corner_small_waves).
template <int N, bool BN, int PASSES, bool QUADS, int WAVES>
__device__ __forceinline__ void corner_small_dx_unit(CornerSmallArgs const &t, CornerSmallDxShared<N, BN, PASSES> *shared, int tile, int wave, int lane)
{
    constexpr int NN = 1 << N;
    using Quads = CornerQuads<N, PASSES>;
    DxArgs const &a = t.dx;
    CornerSumsArgs const &s = t.sums;
    int in, share;
    dx_list_share(a, tile, wave, in, share);
    if (in >= a.input_node_size) { return; }                            // (workgroup-uniform in split mode)
    int const *const list = a.rev + (size_t)in * a.rev_stride;
    int t_begin, t_end;
    dx_list_range<WAVES>(list[0], share, t_begin, t_end);

    // (byte offsets into the whole buffers, which the host keeps below 4 GiB here)
    struct Slots { int e; uint32_t row[N], dy; float mean, rstd; };
    struct Stage { int e; uint32_t w[N]; float4 dy[PASSES]; float v; };
    uint32_t const x_bytes  = (uint32_t)(a.input_node_size - 1) * (uint32_t)s.x_stride * 4u + (uint32_t)((a.frame_size + 31) >> 5) * 4u;
    uint32_t const dy_bytes = (uint32_t)(s.node_size - 1) * (uint32_t)s.dy_stride * 4u + quad_row_bytes(a.frame_size, QUADS);
    float const *const tables = s.V != nullptr ? s.V : s.W_inline;
    auto request = [&](Slots const &slots, int slot, bool live, Stage &g) {
        auto const item = [&](uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)v, slot); };
        g.e = (int)item((uint32_t)slots.e);
        __amdgpu_buffer_rsrc_t const xr  = row_descriptor(s.x, 0, 0, live ? x_bytes : 0u);
        __amdgpu_buffer_rsrc_t const dyr = row_descriptor(s.dy, 0, 0, live ? dy_bytes : 0u);
        __amdgpu_buffer_rsrc_t const vr  = row_descriptor(tables, 0, 0, live ? (uint32_t)s.node_size * (NN * 4u) : 0u);
#pragma unroll
        for (int k = 0; k < N; ++k) { g.w[k] = __builtin_amdgcn_raw_buffer_load_b32(xr, Quads::offset(lane), item(slots.row[k]), 0); }
        g.v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(vr, (uint32_t)(lane & (NN - 1)) * 4u, ((uint32_t)g.e / (uint32_t)N) * (NN * 4u), 0));
        uint32_t const dy_row = item(slots.dy);
#pragma unroll
        for (int p = 0; p < PASSES; ++p) { g.dy[p] = load_quad<QUADS>(dyr, (uint32_t)(p * 4 * kWave + 4 * lane) * 4u, dy_row); }
    };

    float4 acc[PASSES];
#pragma unroll
    for (int p = 0; p < PASSES; ++p) { acc[p] = make_float4(0.0f, 0.0f, 0.0f, 0.0f); }
    auto &mine = shared[wave];
    int const left = a.frame_size - 4 * lane;                           // frame 4 lane + i of pass p exists: 256 p + i < left
    auto add = [&](Stage const &g, float mean, float rstd) {
        int const k = g.e - (int)((uint32_t)g.e / (uint32_t)N) * N;
        uint32_t at[PASSES];
        Quads::form(g.w, lane, mine.quads, at);
        float v = g.v;
        if (s.V == nullptr) {
            if (s.lut_binarize) { v = (v > 0.5f) ? 1.0f : 0.0f; }
            v = corner_butterfly<N>(centred_butterfly<N>(v, lane & (NN - 1)), lane & (NN - 1), s.bias);
        }
        float const other = __int_as_float(__builtin_amdgcn_ds_bpermute((lane * 4) ^ (4 << k), __float_as_int(v)));
        // V[k at hi] - V[k at lo]: the lane's own value minus the other's, negated where the lane holds the lower corner
        float const slope = __uint_as_float(__float_as_uint(v - other) ^ (((uint32_t)~lane << (31 - k)) & 0x80000000u)) * t.inv_step;
        wave_fence();
        if constexpr (BN) {
            float const bn = batch_norm_output(v, mean, rstd, s.fold.gamma, s.fold.beta);
            if (NN == kWave || lane < NN) { mine.table[lane] = CornerSlope{v - mean, slope, (bn <= 0.0f || bn >= 1.0f) ? 0u : 0xffffffffu, 0u}; }
        }
        else { if (NN == kWave || lane < NN) { mine.table[lane] = slope; } }
        wave_fence();
        if constexpr (BN) {
            float s0 = 0.0f, s1 = 0.0f, above[PASSES][4], slopes[PASSES][4], grad[PASSES][4];
#pragma unroll
            for (int p = 0; p < PASSES; ++p) {
                float const dy[4] = {g.dy[p].x, g.dy[p].y, g.dy[p].z, g.dy[p].w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    CornerSlope const q = mine.table[(at[p] >> (8 * i)) & 0xffu];
                    above[p][i] = q.above_mean; slopes[p][i] = q.slope;
                    // (behind a closed window dy counts as 0, whatever it is; so does what lies behind the frames)
                    grad[p][i] = __uint_as_float(__float_as_uint(dy[i]) & (p * 4 * kWave + i < left ? q.open : 0u));
                    s0 += grad[p][i];
                    s1 = __builtin_fmaf(grad[p][i], q.above_mean, s1);
                }
            }
            wave_sum_pair(s0, s1);
            float const gain = s.fold.gamma * rstd;
            float const shift = -(s.fold.gamma * s0) * rstd * s.fold.inv_frames;
            float const scale = -(s.fold.gamma * s1) * (rstd * rstd) * rstd * s.fold.inv_frames;
#pragma unroll
            for (int p = 0; p < PASSES; ++p) {
                float *const sum[4] = {&acc[p].x, &acc[p].y, &acc[p].z, &acc[p].w};
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    *sum[i] = __builtin_fmaf(slopes[p][i], __builtin_fmaf(grad[p][i], gain, __builtin_fmaf(above[p][i], scale, shift)), *sum[i]);
                }
            }
        }
        else {
#pragma unroll
            for (int p = 0; p < PASSES; ++p) {
                acc[p].x = __builtin_fmaf(g.dy[p].x, mine.table[at[p] & 0xffu], acc[p].x);
                acc[p].y = __builtin_fmaf(g.dy[p].y, mine.table[(at[p] >> 8) & 0xffu], acc[p].y);
                acc[p].z = __builtin_fmaf(g.dy[p].z, mine.table[(at[p] >> 16) & 0xffu], acc[p].z);
                acc[p].w = __builtin_fmaf(g.dy[p].w, mine.table[at[p] >> 24], acc[p].w);
            }
        }
    };

    int const count = t_end - t_begin;                                  // at most kCornerSmallItems (the host)
    if (count > 0) {
        Slots slots{};
        if (lane < count) {
            slots.e = list[1 + t_begin + lane];
            int const node = (int)((uint32_t)slots.e / (uint32_t)N);
#pragma unroll
            for (int k = 0; k < N; ++k) { slots.row[k] = (uint32_t)s.idx[(size_t)node * N + k] * (uint32_t)s.x_stride * 4u; }
            slots.dy = (uint32_t)node * (uint32_t)s.dy_stride * 4u;
            if (BN) { slots.mean = s.fold.mean[node]; slots.rstd = s.fold.rstd[node]; }
        }
        auto statistic = [&](float v, int slot) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), slot)); };
        Stage even, odd;
        request(slots, 0, true, even);
        for (int i = 0; i < count; i += 2) {
            request(slots, min(i + 1, kWave - 1), i + 1 < count, odd);
            add(even, statistic(slots.mean, i), statistic(slots.rstd, i));
            request(slots, min(i + 2, kWave - 1), i + 2 < count, even);
            if (i + 1 < count) { add(odd, statistic(slots.mean, i + 1), statistic(slots.rstd, i + 1)); }
        }
    }

    if (a.split) {                              // the shares of the list, added in wavefront order (dx_store_pass)
#pragma unroll
        for (int p = 0; p < PASSES; ++p) { mine.part[p][lane] = acc[p]; }
        __syncthreads();
        if (wave != 0) { return; }
#pragma unroll
        for (int p = 0; p < PASSES; ++p) {
#pragma unroll
            for (int w = 1; w < WAVES; ++w) {
                float4 const o = shared[w].part[p][lane];
                acc[p].x += o.x; acc[p].y += o.y; acc[p].z += o.z; acc[p].w += o.w;
            }
        }
    }
    float *const row = a.dx + (size_t)in * a.dx_stride;
#pragma unroll
    for (int p = 0; p < PASSES; ++p) {
        int const f = p * 4 * kWave + 4 * lane;
        if (f     < a.frame_size) { row[f]     = acc[p].x; }
        if (f + 1 < a.frame_size) { row[f + 1] = acc[p].y; }
        if (f + 2 < a.frame_size) { row[f + 2] = acc[p].z; }
        if (f + 3 < a.frame_size) { row[f + 3] = acc[p].w; }
    }
}

// WAVES: wavefronts of a workgroup, that is nodes of one, or wavefronts that share an input's list
template <int N, bool BN, int PASSES, bool QUADS, int WAVES>
__global__ __launch_bounds__(WAVES * kWave) void lut_corner_small_backward_kernel(CornerSmallArgs t)
{
    constexpr int FORM = PASSES;                // (kSums256, kSums512, kSumsShort)
    using Sums = SumsShared<N, BN, FORM>;
    using Dx = CornerSmallDxShared<N, BN, PASSES>;
    __shared__ __align__(16) unsigned char shared[WAVES * (sizeof(Sums) > sizeof(Dx) ? sizeof(Sums) : sizeof(Dx))];
    int const wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave)), lane = threadIdx.x & (kWave - 1);
    int const bid = blockIdx.x;
    if (bid < t.dx_blocks) { corner_small_dx_unit<N, BN, PASSES, QUADS, WAVES>(t, reinterpret_cast<Dx *>(shared), bid, wave, lane); return; }
    int const node = (bid - t.dx_blocks) * WAVES + wave;
    if (node >= t.sums.node_size) { return; }
    corner_sums_unit<N, BN, FORM, QUADS>(t.sums, reinterpret_cast<Sums *>(shared)[wave], node, 0, lane);
}

}  // namespace bbhip
