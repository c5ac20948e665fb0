// Backward pass of the LUT layers on two-valued inputs (packed bits; fp32 frames binarized at 0.5 are packed first).
//
// Over two-valued inputs a node's frames fall into 2^N corners, and everything that the backward pass needs of them is, per corner,
//     D[p] = the sum of dy over the frames at corner p,     n[p] = the number of those frames.
// With batch-norm, dL/d(LUT output) of a frame at corner p is  open[p] gamma rstd dy + E[p]  (reference: DifferentiableLutN.h:1206-1250), where
// open[p] says whether the batch-norm output of the corner lies inside the hard-tanh window and E[p] is the gradient through the statistics, so
//     sum of g              s0 = sum_p open[p] D[p],        sum of g (v - mean)   s1 = sum_p open[p] D[p] (V[p] - mean),
//     E[p] = shift + (V[p] - mean) scale,   shift = -gamma rstd s0 / F,   scale = -gamma rstd^3 s1 / F
//            (the reference's dmean + V dvar / F with mean dvar / F left out of both: where V is hundreds of times its own spread that
//            difference costs two digits),
//     gradient at corner p  G[p] = open[p] gamma rstd D[p] + n[p] E[p],
//     dW[i]                 = sum_p G[p] prod_j (bit_j(i) ? x_j(p) : 1 - x_j(p)).
// One pass over the inputs and dy gives D and n (lut_corner_sums_kernel), the rest is arithmetic on 2^N values per node (corner_fold): no
// statistics pass of its own, no polynomial, no 2^N multiply-adds per frame, and no row of dL/d(LUT output) is written.  The dx kernel
// (lut_dx_table_kernel) applies the same two terms per corner:  dx = sum over consumers of  A[p] dy + B[p].
#pragma once

#include "corner_index.hpp"
#include "lut_kernels.hpp"

namespace bbhip {

// quads of a node's table for lut_dx_few_inputs_kernel: (gain, E, d0, d1) of every corner, then (d2 .. d5)
constexpr int few_entry_quads(int n) { return (n > 2 ? 2 : 1) << n; }

// A look through the reverse table for lut_dx_few_inputs_kernel, which goes by the index table: listed[i] = the entries of row i if each is a connection of input i
// and they ascend, else a number below any sum of others.  The sum over the rows is the number of connections if the table lists each of them once.
struct ReverseRows {
    int const *rev, *idx;
    int   rev_stride, links;            // links: connections, node_size N
    int   inputs;                       // rows to look through (0: none)
    int  *listed;
};

// row `in`, by a workgroup
__device__ __forceinline__ void look_through_reverse_row(ReverseRows const &a, int in)
{
    __shared__ int astray[kWavesPerBlk];
    int const *const row = a.rev + (size_t)in * a.rev_stride;
    int const count = row[0], entries = min(count, a.rev_stride - 1);
    bool wrong = false;
#pragma unroll 4
    for (int j = threadIdx.x; j < entries; j += kBlock) {
        int const e = row[1 + j], before = j > 0 ? row[j] : -1;
        bool const known = (unsigned)e < (unsigned)a.links && e > before;
        wrong |= !known || a.idx[known ? e : 0] != in;
    }
    bool const any = __ballot(wrong) != 0;
    if (threadIdx.x % kWave == 0) { astray[threadIdx.x / kWave] = any; }
    __syncthreads();
    if (threadIdx.x != 0) { return; }
    int n = count;
#pragma unroll
    for (int w = 0; w < kWavesPerBlk; ++w) { n = astray[w] ? -(1 << 24) : n; }
    a.listed[in] = n;
}
__global__ __launch_bounds__(kBlock) void reverse_rows_kernel(ReverseRows a) { look_through_reverse_row(a, blockIdx.x); }

struct CornerFoldArgs {
    float const *mean, *rstd;           // batch-norm
    float gamma, beta, inv_frames;
    int   frame_size;
    float lo, hi;                       // the two input values, 1/2 -+ bias
    float *dW;
    int   overwrite;                    // dW = instead of dW +=
    struct NodeConsts *node_consts;     // batch-norm: what lut_dx_table_kernel needs of each node beside its corner values (null: nothing)
    // batch-norm: *discard = call where a discarded dy (one at a corner outside the hard-tanh window) may not be finite.  `call` is another number for
    // each call, so that nothing has to be cleared ahead; a stale equal value only sends the dx kernel to its slower walk
    uint32_t *discard;
    uint32_t call;
    float4 *entries;                    // the node's table for lut_dx_few_inputs_kernel (null: none)
};

// A[p] and B[p] of the dx kernel are, for a connection with difference d[p] = V[input at hi] - V[input at lo],
//     A[p] = open[p] ? d[p] gain : 0,     B[p] = d[p] (shift + (V[p] - mean) scale)            (gain, shift, scale divided by hi - lo)
struct __align__(32) NodeConsts { float mean, gain, shift, scale; uint64_t open; uint64_t unused; };

// Lane p (of every group of 2^N lanes) holds the node's V[p], D[p], n[p]: the node's table gradient and, with batch-norm, its constants
// (mean, rstd and the entry of dW that the gradient adds to: loaded by the caller, long before)
struct CornerFoldInputs { float mean, rstd, dW; };
template <int N, bool BN>
__device__ __forceinline__ CornerFoldInputs corner_fold_inputs(CornerFoldArgs const &a, int node, int lane)
{
    CornerFoldInputs q{0.0f, 1.0f, 0.0f};
    if (BN) { q.mean = a.mean[node]; q.rstd = a.rstd[node]; }
    if (!a.overwrite) { q.dW = a.dW[((size_t)node << N) + (lane & ((1 << N) - 1))]; }
    return q;
}
template <int N, bool BN>
__device__ __forceinline__ void corner_fold(CornerFoldArgs const &a, CornerFoldInputs const &q, int node, int lane, float v, float D, float n)
{
    constexpr int NN = 1 << N;
    float G = D;
    float const inv_step = 1.0f / (a.hi - a.lo);
    float gain = inv_step, e = 0.0f;                                    // of the lane's corner, for a.entries
    if (BN) {
        float const mean = q.mean, rstd = q.rstd;
        float const t = batch_norm_output(v, mean, rstd, a.gamma, a.beta);
        float const g = (t <= 0.0f || t >= 1.0f) ? 0.0f : D;
        float const counted = (lane < NN) ? g : 0.0f;                   // narrow tables repeat over the wavefront
        float const s0 = wave_sum(counted), s1 = wave_sum(counted * (v - mean));
        float const shift = -(a.gamma * s0) * rstd * a.inv_frames;
        float const scale = -(a.gamma * s1) * (rstd * rstd) * rstd * a.inv_frames;
        G = __builtin_fmaf(g, a.gamma * rstd, n * __builtin_fmaf(v - mean, scale, shift));
        uint64_t const open = __ballot(!(t <= 0.0f || t >= 1.0f));
        gain = __builtin_amdgcn_inverse_ballot_w64(open) ? a.gamma * rstd * inv_step : 0.0f;
        e = __builtin_fmaf(v - mean, scale * inv_step, shift * inv_step);
        // (one value that is not finite makes its corner's sum such)
        bool const discard = __ballot((t <= 0.0f || t >= 1.0f) && !(fabsf(D) < __builtin_inff())) != 0;
        if (lane == 0 && discard && a.node_consts != nullptr) { *a.discard = a.call; }
        if (lane == 0 && a.node_consts != nullptr) { a.node_consts[node] = NodeConsts{mean, a.gamma * rstd * inv_step, shift * inv_step, scale * inv_step, open, 0}; }
    }
    if (a.entries != nullptr) {
        float d[6] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 0; k < N; ++k) {                                   // V[k at hi] - V[k at lo]
            float const o = lane_xor(v, 1 << k);
            d[k] = ((lane >> k) & 1) ? v - o : o - v;
        }
        if (lane < NN) {
            float4 *const to = a.entries + (size_t)node * few_entry_quads(N) + lane;
            to[0] = make_float4(gain, e, d[0], d[1]);
            if (N > 2) { to[NN] = make_float4(d[2], d[3], d[4], d[5]); }
        }
    }
    // per input: (G0, G1) -> ((1 - lo) G0 + (1 - hi) G1, lo G0 + hi G1), and 1 - lo = hi: either lane keeps hi of its own and takes lo of the other's
#pragma unroll
    for (int j = 0; j < N; ++j) { G = __builtin_fmaf(a.hi, G, a.lo * lane_xor(G, 1 << j)); }
    if (lane < NN) { a.dW[(size_t)node * NN + lane] = a.overwrite ? G : q.dW + G; }
}

// How a wavefront adds up the frames of a node (SumsForm, see lut_corner_sums_kernel)
template <int N, bool BN, int FORM>
struct SumsTraits {
    static constexpr int  NN = 1 << N;
    static constexpr bool kLoop = FORM == kSumsLong;
    // (with few corners the atomics that count them collide, and the plain form has little to keep anyway; over 2048 frames the chains of columns that
    // two lanes share would be longer: rms error of dW, inputs set in 98 of 100 frames, 9.4e-8 instead of 7.0e-8)
    static constexpr bool kAtomics = !kLoop && N >= 5 && FORM != kSumsBlock, kCountSets = BN && !kAtomics, kCountFrames = BN && kAtomics;
    static constexpr int  kPasses = kLoop ? 8 : FORM;
    static constexpr int  kColumns = !kAtomics ? kWave : FORM == kSums256 ? 16 : 32;
};
template <int N, bool BN, int FORM>
struct SumsShared {                     // a wavefront's LDS
    using T = SumsTraits<N, BN, FORM>;
    __align__(16) float    bins[T::NN * T::kColumns];
    __align__(16) uint32_t quads[T::kPasses * kWave];
    uint32_t counts[T::kCountFrames ? T::NN : 1];
};
constexpr int kSkewedChain = 4096, kFairChain = 16384;          // frames, see there

struct CornerSumsArgs {
    uint32_t const *x;
    float const *dy;
    int const   *idx;
    float const *V;             // [O][2^N] corner values, or null:
    float const *W_inline;      // the wavefront derives them from the table; the wavefront of a node's first slab stores them to V_out
    float       *V_out;
    int   lut_binarize;
    float bias;
    int   node_size, frame_size, x_stride, dy_stride;
    int   slab, slab_count;     // frames per unit, a multiple of 256
    TileDivisor tiles;
    uint32_t *own;              // the corner index of every (node, frame), a byte each in frame order, for the dx kernel: rows of own_stride words
    int   own_stride;
    float *partial;             // several slabs: [slab][O][BN ? 2 : 1][2^N], D and then n
    CornerFoldArgs fold;        // one slab: the wavefront folds its sums itself
};

// sums over the COLS columns of row (lane mod ROWS) of a wavefront's [ROWS][COLS] block in LDS.  A lane takes four columns at a time, in an order
// of its own, so that the lanes that are served together read different banks; with fewer than 64 rows several lanes share one.
template <int ROWS, int COLS, typename V4>
__device__ __forceinline__ auto row_sum(V4 const *block, int lane)
{
    constexpr int LANES = kWave / ROWS, EACH = COLS / 4 / LANES;        // lanes per row, groups of four columns for each
    static_assert(EACH >= 1, "a group of columns for every lane");
    int const p = lane & (ROWS - 1), part = lane / ROWS;
    decltype(block[0].x + block[0].x) s = 0;
#pragma unroll
    for (int g = 0; g < EACH; ++g) {
        V4 const q = block[p * (COLS / 4) + part * EACH + (g ^ (p & (EACH - 1)))];
        s += (q.x + q.y) + (q.z + q.w);
    }
#pragma unroll
    for (int o = ROWS; o < kWave; o <<= 1) { s += lane_xor(s, o); }
    return s;
}

// One wavefront = one node x one slab of frames, in blocks of 2048 frames.  A lane loads the words of 32 frames of each input and turns them
// into corner indices (corner_bytes), which go to memory for the dx kernel and through LDS to the lanes that hold the frames' dy: a pass is 256
// frames, four consecutive ones per lane.  Each lane keeps bins of its own in LDS ([corner][lane]: no two lanes share an address, and the 64 lanes
// of a step always touch 64 different banks) and adds its dy by a plain read-add-write: 12 clocks per step of 64 frames and CU, where the 64
// multiply-adds of a polynomial form take 64 vector instructions per step and an LDS float atomic (ds_add_f32) 193 clocks.  n: a lane counts,
// for each set of inputs, the frames of its words where all of them are set (2 instructions per set and 32 frames); the lanes' counts
// are added at the end and differences over the sets give the corners' counts.
// A bin is a chain of additions, and where the inputs are skewed nearly all frames of a lane go to one: after kFairChain frames, or kSkewedChain where
// in some block a quarter of the lanes had more than half of their words' frames at the corner of the first one, the bins are added up and
// cleared (256 clocks of LDS).  rms error of dW against 64 bits relative to a node's largest entry, by a model of the order of operations, 65536
// frames, against multiply-adds in slabs of 4096 frames: inputs set in half of the frames 4e-8 (multiply-adds 8e-8), in 85 of 100 4e-8 (5e-8),
// in 98 of 100 5e-8 (6e-8; 1.5e-7 as one chain).  4096 x 8192 and 216 x 230400 take 1 and 5 us longer where the bins are closed every 4096 frames.
// The bins leave two workgroups per compute unit, so what the wavefronts wait for shows: words and dy are requested a block ahead, on every path (a
// load that a path may leave out makes the compiler wait for all that are under way), as vector loads (scalar loads would be waited for with the LDS
// accesses: 101 us for the first shape below), and four frames' bins are read together.  4096 nodes x 8192 frames 40.0 -> 36.4 us, 3003 x 5005
// 27.8 -> 23.0, 216 x 230400 65 -> 57 (4.4 TB/s of dy and indices).
// QUADS: rows of dy hold whole groups of four frames.
// The statistics and table-gradient launches that it replaces took 53 + 141 us for 216 nodes x 230400 frames, 31 + 106 for 4096 x 8192.
// kSumsShort: up to kShortSlab frames in one slab.  Such a launch is a chain of latencies, so what counts is how many wavefronts share a compute unit: for five
// and six inputs two lanes share a column of bins (they add in turn), and the corners are counted by integer atomics (one instruction per step, and nothing
// to add up).  6144 nodes x 1024 frames 20.5 -> 13.6 us, 6000 x 100 17.4 -> 9.6 us; four lanes per column measured the same or slower.
// kSumsBlock: up to 2048 frames, a column for each lane (corner_sums_form has both sides of the lines).
struct CornerSums { float v, D, n; CornerFoldInputs in; };          // lane p (of every group of 2^N lanes): of corner p
template <int N, bool BN, int FORM, bool QUADS>
__device__ __forceinline__ CornerSums corner_sums(CornerSumsArgs const &a, SumsShared<N, BN, FORM> &sh, int node, int sl, int lane, bool fold)
{
    using T = SumsTraits<N, BN, FORM>;
    constexpr int NN = 1 << N, kPasses = T::kPasses, COLS = T::kColumns;
    constexpr bool kLoop = T::kLoop, kCountSets = T::kCountSets, kCountFrames = T::kCountFrames;
    int const f_begin = sl * a.slab;
    int const f_end   = min(f_begin + a.slab, a.frame_size);
    __amdgpu_buffer_rsrc_t const dyr = row_descriptor(a.dy, node, a.dy_stride, quad_row_bytes(f_end, QUADS));      // (past the slab: no access, zeros)
    uint32_t const x_row_bytes = (uint32_t)((a.frame_size + 31) >> 5) * 4u;
    __amdgpu_buffer_rsrc_t xr[N];
#pragma unroll
    for (int k = 0; k < N; ++k) { xr[k] = row_descriptor(a.x, a.idx[node * N + k], a.x_stride, x_row_bytes); }

    uint32_t w_next[N];
    auto request_words = [&](int base) {
#pragma unroll
        for (int k = 0; k < N; ++k) { w_next[k] = __builtin_amdgcn_raw_buffer_load_b32(xr[k], (uint32_t)((base >> 5) + lane) * 4u, 0, 0); }
    };
    float4 dy[kPasses];
    request_words(f_begin);
#pragma unroll
    for (int i = 0; i < kPasses; ++i) { dy[i] = load_quad<QUADS>(dyr, (uint32_t)(f_begin + i * 4 * kWave + 4 * lane) * 4u); }

    CornerFoldInputs fold_in{};
    if (fold) { fold_in = corner_fold_inputs<N, BN>(a.fold, node, lane); }
    float v;                                                            // lane p: V[p]
    if (a.V != nullptr) { v = a.V[(size_t)node * NN + (lane & (NN - 1))]; }
    else {
        int const i = lane & (NN - 1);
        float w = a.W_inline[(size_t)node * NN + i];
        if (a.lut_binarize) { w = (w > 0.5f) ? 1.0f : 0.0f; }
        v = corner_butterfly<N>(centred_butterfly<N>(w, i), i, a.bias);
    }

    float *const mine = sh.bins;
    auto clear_bins = [&]() {
#pragma unroll
        for (int i = 0; i < NN * COLS / (4 * kWave); ++i) { *reinterpret_cast<float4 *>(mine + (i * kWave + lane) * 4) = make_float4(0.0f, 0.0f, 0.0f, 0.0f); }
    };
    // Four frames into bins that may be the same: all four bins are read before any is written, a later frame takes an earlier one's sum.  (One
    // after another, each waits for the bin that the one before it wrote.)
    auto add_quad = [&](uint32_t corners, float4 const &d) {
        uint32_t const p0 = corners & 0xffu, p1 = (corners >> 8) & 0xffu, p2 = (corners >> 16) & 0xffu, p3 = corners >> 24;
        float *const col = mine + (lane & (COLS - 1));
        float r0 = col[p0 * COLS], r1 = col[p1 * COLS], r2 = col[p2 * COLS], r3 = col[p3 * COLS];
        asm("" : "+v"(r0), "+v"(r1), "+v"(r2), "+v"(r3));               // (no branch around a read whose value a lane does not need)
        float const v0 = r0 + d.x;
        float const v1 = (p1 == p0 ? v0 : r1) + d.y;
        float const v2 = (p2 == p1 ? v1 : p2 == p0 ? v0 : r2) + d.z;
        float const v3 = (p3 == p2 ? v2 : p3 == p1 ? v1 : p3 == p0 ? v0 : r3) + d.w;
        col[p0 * COLS] = v0; col[p1 * COLS] = v1; col[p2 * COLS] = v2; col[p3 * COLS] = v3;
    };
    clear_bins();
    if (kCountFrames && lane < NN) { sh.counts[lane] = 0; }
    wave_fence();

    float D = 0.0f;                                                     // lane p: sums of the bins that were closed
    int  opened = f_begin;
    bool skewed = false;
    uint32_t count[kCountSets ? NN : 1];                                // [S]: frames of the lane's words where every input of S is set
#pragma unroll
    for (int i = 0; i < (kCountSets ? NN : 1); ++i) { count[i] = 0; }

    for (int base = f_begin; base < f_end; base += kPasses * 4 * kWave) {
        uint32_t quad[8];
        {
            uint32_t w[N];
#pragma unroll
            for (int k = 0; k < N; ++k) { w[k] = w_next[k]; }
            if (kLoop) { request_words(base + kPasses * 4 * kWave); }  // (past the row: zeros)
            corner_bytes<N>(w, quad);
            if (kLoop) {
                uint32_t elsewhere = 0;                                 // frames at another corner than the lane's first
#pragma unroll
                for (int k = 0; k < N; ++k) { elsewhere |= w[k] ^ (uint32_t)((int32_t)(w[k] << 31) >> 31); }
                skewed |= __popcll(__ballot(__popc(elsewhere) < 16)) >= kWave / 4;
            }
            int const live = f_end - (base + 32 * lane);                // frames of the lane's words that belong to the slab
            if (live > 0 && a.own != nullptr) {
                uint4 *out = reinterpret_cast<uint4 *>(a.own + (size_t)node * a.own_stride + ((base >> 2) + 8 * lane));
                out[0] = make_uint4(quad[0], quad[1], quad[2], quad[3]);
                out[1] = make_uint4(quad[4], quad[5], quad[6], quad[7]);
            }
            if (kLoop || lane < kPasses * 8) {                         // (the lanes whose words hold frames of the slab)
                uint4 *ex = reinterpret_cast<uint4 *>(sh.quads + 8 * lane);
                ex[0] = make_uint4(quad[0], quad[1], quad[2], quad[3]);
                ex[1] = make_uint4(quad[4], quad[5], quad[6], quad[7]);
            }
            if constexpr (kCountSets) {
                uint32_t all[NN];
                all[0] = (live >= 32) ? 0xffffffffu : (live <= 0) ? 0u : ((1u << live) - 1u);
                count[0] += __popc(all[0]);
#pragma unroll
                for (int s = 1; s < NN; ++s) {
                    all[s] = all[s & (s - 1)] & w[__builtin_ctz(s)];
                    count[s] += __popc(all[s]);
                    asm volatile("" : "+v"(count[s]));                  // (here, not moved behind the passes with all 2^N sets alive)
                }
            }
        }
        wave_fence();
        uint32_t at[kPasses];
#pragma unroll
        for (int i = 0; i < kPasses; ++i) { at[i] = sh.quads[i * kWave + lane]; }
#pragma unroll
        for (int i = 0; i < kPasses; ++i) {
            int const fb = base + i * 4 * kWave;
            if (fb < f_end) {                                           // wave-uniform
                float4 d = dy[i];
                if (fb + 4 * kWave > a.frame_size) {                    // the row's padding may hold anything
                    int const f = fb + 4 * lane;
                    if (f     >= a.frame_size) { d.x = 0.0f; }
                    if (f + 1 >= a.frame_size) { d.y = 0.0f; }
                    if (f + 2 >= a.frame_size) { d.z = 0.0f; }
                    if (f + 3 >= a.frame_size) { d.w = 0.0f; }
                }
                if constexpr (kCountFrames) {
                    int const f = fb + 4 * lane;
                    if (f     < f_end) { atomicAdd(&sh.counts[at[i] & 0xffu], 1u); }
                    if (f + 1 < f_end) { atomicAdd(&sh.counts[(at[i] >> 8) & 0xffu], 1u); }
                    if (f + 2 < f_end) { atomicAdd(&sh.counts[(at[i] >> 16) & 0xffu], 1u); }
                    if (f + 3 < f_end) { atomicAdd(&sh.counts[at[i] >> 24], 1u); }
                }
                if constexpr (COLS == kWave) { add_quad(at[i], d); }
                else {
#pragma unroll
                    for (int turn = 0; turn < kWave / COLS; ++turn) {
                        if (lane / COLS == turn) { add_quad(at[i], d); }
                        wave_fence();
                    }
                }
            }
            // (outside of the condition: loads that a path may leave out make the compiler wait for all that are under way)
            __builtin_amdgcn_sched_barrier(0);                          // (into the registers that are free now)
            if (kLoop) { dy[i] = load_quad<QUADS>(dyr, (uint32_t)(fb + kPasses * 4 * kWave + 4 * lane) * 4u); }
        }
        wave_fence();
        int const next = base + kPasses * 4 * kWave;
        if (next >= f_end || next - opened >= (skewed ? kSkewedChain : kFairChain)) {           // (else: one block)
            D += row_sum<NN, COLS>(reinterpret_cast<float4 const *>(mine), lane);
            if (next < f_end) {
                opened = next;
                skewed = false;
                wave_fence();
                clear_bins();
                wave_fence();
            }
        }
    }

    uint32_t n = 0;
    if constexpr (kCountFrames) { n = sh.counts[lane & (NN - 1)]; }
    if constexpr (kCountSets) {
        wave_fence();
        uint32_t *const cells = reinterpret_cast<uint32_t *>(mine);
#pragma unroll
        for (int s = 0; s < NN; ++s) { cells[s * kWave + lane] = count[s]; }
        wave_fence();
        n = row_sum<NN, kWave>(reinterpret_cast<uint4 const *>(cells), lane);  // lane S: frames where every input of S is set (the others either way)
#pragma unroll
        for (int k = 0; k < N; ++k) {
            uint32_t const o = lane_xor(n, 1 << k);
            if (!((lane >> k) & 1)) { n -= o; }                         // ... minus those where input k is set too
        }
    }

    if (a.V_out != nullptr && sl == 0 && lane < NN) { a.V_out[(size_t)node * NN + lane] = v; }
    return CornerSums{v, D, (float)n, fold_in};
}
template <int N, bool BN, int FORM, bool QUADS>
__device__ __forceinline__ void corner_sums_unit(CornerSumsArgs const &a, SumsShared<N, BN, FORM> &sh, int node, int sl, int lane)
{
    constexpr int NN = 1 << N;
    CornerSums const q = corner_sums<N, BN, FORM, QUADS>(a, sh, node, sl, lane, a.slab_count == 1);
    if (a.slab_count == 1) { corner_fold<N, BN>(a.fold, q.in, node, lane, q.v, q.D, q.n); }
    else if (lane < NN) {
        float *out = a.partial + ((size_t)sl * a.node_size + node) * (BN ? 2 * NN : NN) + lane;
        out[0] = q.D;
        if (BN) { out[NN] = q.n; }
    }
}

template <int N, bool BN, int FORM, bool QUADS>
__global__ __launch_bounds__(kBlock, 2) void lut_corner_sums_kernel(CornerSumsArgs a)
{
    __shared__ SumsShared<N, BN, FORM> shared[kWavesPerBlk];
    int const lid = xcd_remap(blockIdx.x, a.slab_count * a.tiles.count);
    int sl, tile;
    split_tile(lid, a.tiles, sl, tile);
    int const wv   = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    int const node = tile * kWavesPerBlk + wv;
    if (node >= a.node_size) { return; }
    corner_sums_unit<N, BN, FORM, QUADS>(a, shared[wv], node, sl, threadIdx.x & (kWave - 1));
}

// Few nodes (node_sums): a workgroup per node, whose wavefronts take a part of up to kBlockSlab frames each (a.slab) and leave their sums in LDS to the first,
// which folds them.  A chain of latencies like the forms of one slab, but without partial sums in memory and the launch that folds them.  Backward call of 40 inputs, six per node: 100 nodes x 4000 frames 12.6 -> 10.9 us, 130 x 10000 16.6 -> 13.9, 256 x 4500 16.5 -> 13.6.
template <int N, bool BN, bool QUADS>
__global__ __launch_bounds__(kNodeSumsWaves * kWave) void lut_corner_sums_node_kernel(CornerSumsArgs a)
{
    __shared__ SumsShared<N, BN, kSumsBlock> shared[kNodeSumsWaves];
    static_assert((1 << N) * kWave >= 2 * kWave, "room for both sums");
    int const wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave)), lane = threadIdx.x & (kWave - 1), node = blockIdx.x;
    CornerSums q = corner_sums<N, BN, kSumsBlock, QUADS>(a, shared[wave], node, wave, lane, wave == 0);   // (past the last frame: zeros)
    wave_fence();
    float *const mine = shared[wave].bins;                              // (the bins are added up)
    mine[lane] = q.D;
    mine[kWave + lane] = q.n;
    __syncthreads();
    if (wave != 0) { return; }
#pragma unroll
    for (int w = 1; w < kNodeSumsWaves; ++w) { q.D += shared[w].bins[lane]; q.n += shared[w].bins[kWave + lane]; }
    corner_fold<N, BN>(a.fold, q.in, node, lane, q.v, q.D, q.n);
}

// Several slabs per node: a workgroup per node adds them up, each wavefront every fourth slab, and folds.  (The last `rows.inputs` workgroups look through the
// reverse table, for nothing beside the others: 27 inputs x 72 nodes x 230400 frames 41.4 us for the backward call with and without, 42.5 where each
// workgroup of the dx launch looked for itself.)
template <int N, bool BN>
__global__ __launch_bounds__(kBlock) void lut_corner_fold_kernel(CornerFoldArgs a, ReverseRows rows, float const *__restrict__ partial, float const *__restrict__ V,
                                                                 int node_size, int slab_count)
{
    constexpr int NN = 1 << N, REC = BN ? 2 * NN : NN;
    if ((int)blockIdx.x >= node_size) { look_through_reverse_row(rows, blockIdx.x - node_size); return; }
    __shared__ float red[2][kWavesPerBlk][kWave];
    int const node = blockIdx.x;
    int const wv = threadIdx.x / kWave, lane = threadIdx.x & (kWave - 1);
    float const *in = partial + (size_t)node * REC + (lane & (NN - 1));
    CornerFoldInputs const fold_in = corner_fold_inputs<N, BN>(a, node, lane);
    float const v = V[(size_t)node * NN + (lane & (NN - 1))];
    float D = 0.0f, n = 0.0f;
#pragma unroll 4
    for (int s = wv; s < slab_count; s += kWavesPerBlk) {
        float const *q = in + (size_t)s * node_size * REC;
        D += q[0];
        if (BN) { n += q[NN]; }
    }
    red[0][wv][lane] = D;
    red[1][wv][lane] = n;
    __syncthreads();
    if (wv != 0) { return; }
#pragma unroll
    for (int w = 1; w < kWavesPerBlk; ++w) { D += red[0][w][lane]; n += red[1][w][lane]; }
    corner_fold<N, BN>(a, fold_in, node, lane, v, D, n);
}

struct DxTableArgs {
    DxArgs dx;                          // units, work lists, split mode and rows as in lut_dx_kernel (no term table, no rider)
    uint32_t const *own;                // kept corner indices, a byte per frame, rows of own_stride words
    int   own_stride;
    int   node_size;
    int   far;                          // see lut_dx_table_kernel
    int   dx_quads;                     // rows of dx start on 16 bytes
    float const *V;                     // [O][2^N]
    NodeConsts const *node_consts;      // batch-norm
    float inv_step;                     // 1 / (hi - lo)
    uint32_t const *discard;            // batch-norm: see CornerFoldArgs
    uint32_t call;
};

// Input-centric dx over kept corner indices.  One wavefront owns dx[input][256 Q frames], four consecutive frames per lane and quad, and walks the
// input's consumers in the reverse table's order (split mode: a part of them).  A consumer's term of a frame at corner p is  A[p] dy + B[p]  with
//     A[p] = dV/dx_k[p] open[p] gamma rstd,   B[p] = dV/dx_k[p] E[p]           (plain layers: A = dV/dx_k, B = 0),
// and y is linear in input k, so dV/dx_k[p] = (V[k at hi] - V[k at lo]) / (hi - lo): lane p computes entry p from the node's 2^N corner values
// and its constants (288 bytes per node that all its consumers share), the wavefront puts the table into LDS, and the frames fetch their
// entry from there: a random 8-byte LDS read takes 4.5 clocks per CU and step where two ds_bpermute take 14.  Per term and pass one vector load
// of V, Q of indices and Q of dy; the next term's are in flight while a term is evaluated.
// The kernel is bound by vector instructions (4 per element and about 20 per term) and by what its L2 delivers: rows are addressed by a 32-bit
// offset into the whole buffer, dy by one 16-byte load per lane and quad, and a lane past the last frame reads whatever lies there.
// FAR: buffers (dy, indices, V) of 4 GiB and more, and rows of dy that do not hold whole groups of four: a descriptor per row, single words.
// Behind a closed hard-tanh window dy counts as 0, whatever it is.  A = 0 gives that for finite values; where the per-corner sums say that there are
// others (*discard), a walk of its own sets the values of closed corners to 0 first (three instructions per element more).  A
// training step of 3003 nodes x 5005 frames takes 0.6 us longer for that than without, of 76; with a test per term in one walk 1.4.
// Measured against the kernel that formed the indices from the packed rows: 27 inputs x 216 nodes x 230400 frames (Q = 2) 85 us instead of 117;
// 4096 x 4096 x 8192 (Q = 1) 108 us instead of 138: 745 MB of L2 misses at 6.9 TB/s.  Half as many frames per wavefront miss 479 MB, but the walk's
// scalar instructions and loads per term then take 144 us; four terms in flight and constants by vector loads were slower at every Q.
template <int N, bool BN, int Q, int WAVES, bool FAR = false>
__global__ __launch_bounds__(WAVES * kWave) void lut_dx_table_kernel(DxTableArgs t)
{
    constexpr int NN = 1 << N, kPass = 4 * kWave * Q;
    using Entry = std::conditional_t<BN, float2, float>;
    DxArgs const &a = t.dx;
    int const lid = xcd_remap(blockIdx.x, a.chunk_count * a.tiles.count);
    int ck, tile;
    split_tile(lid, a.tiles, ck, tile);
    __shared__ __align__(16) float4 part[WAVES][Q][kWave];
    __shared__ Entry table[WAVES][2][NN];
    int const wave = threadIdx.x / kWave;
    int in, share;
    dx_list_share(a, tile, wave, in, share);
    if (in >= a.input_node_size) { return; }                            // (workgroup-uniform in split mode)
    int const lane = threadIdx.x & (kWave - 1);

    typedef __attribute__((address_space(4))) int const const_int;
    typedef __attribute__((address_space(4))) NodeConsts const const_consts;
    const_int *list = (const_int *)(a.rev + (size_t)in * a.rev_stride);
    const_consts *consts = (const_consts *)t.node_consts;
    typedef __attribute__((address_space(4))) uint32_t const const_word;
    int const fan = list[0];
    uint32_t const discard_word = BN ? *(const_word *)t.discard : 0u;   // (on the way with the list's length)
    int first, step, items;
    dx_list_steps<WAVES>(a.in_turn != 0, fan, share, first, step, items);
    list += 1 + first;
    int const f_lane = ck * kPass + 4 * lane;
    uint32_t const dy_bytes = (uint32_t)(t.node_size - 1) * (uint32_t)a.dy_stride * 4u + quad_row_bytes(a.frame_size, true);
    __amdgpu_buffer_rsrc_t const dyr = row_descriptor(a.dy, 0, 0, FAR ? 0u : dy_bytes);
    __amdgpu_buffer_rsrc_t const ir  = row_descriptor(t.own, 0, 0, FAR ? 0u : (uint32_t)t.node_size * (uint32_t)t.own_stride * 4u);
    __amdgpu_buffer_rsrc_t const vr  = row_descriptor(t.V, 0, 0, FAR ? 0u : (uint32_t)t.node_size * (NN * 4u));

    float4 acc[Q];
#pragma unroll
    for (int q = 0; q < Q; ++q) { acc[q] = make_float4(0.0f, 0.0f, 0.0f, 0.0f); }

    struct Stage { uint32_t iw[Q]; float4 dy[Q]; float v; float mean, gain, shift, scale; uint64_t open; int k; };
    auto request = [&](int e, Stage &s) {
        uint32_t const node = (uint32_t)e / (uint32_t)N;
        s.k = e - (int)node * N;
        __amdgpu_buffer_rsrc_t const v_row = FAR ? row_descriptor(t.V, (int)node, NN, NN * 4u) : vr;
        s.v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(v_row, (lane & (NN - 1)) * 4, FAR ? 0u : node * (NN * 4u), 0));
        if (BN) {
            const_consts &c = consts[node];
            s.mean = c.mean; s.gain = c.gain; s.shift = c.shift; s.scale = c.scale; s.open = c.open;
        }
        __amdgpu_buffer_rsrc_t const i_row = FAR ? row_descriptor(t.own, (int)node, t.own_stride, (uint32_t)t.own_stride * 4u) : ir;
        __amdgpu_buffer_rsrc_t const d_row = FAR ? row_descriptor(a.dy, (int)node, a.dy_stride, (uint32_t)a.frame_size * 4u) : dyr;
        uint32_t const i_off = FAR ? 0u : node * (uint32_t)t.own_stride * 4u, d_off = FAR ? 0u : node * (uint32_t)a.dy_stride * 4u;
#pragma unroll
        for (int q = 0; q < Q; ++q) { s.iw[q] = __builtin_amdgcn_raw_buffer_load_b32(i_row, (uint32_t)(f_lane + q * 4 * kWave), i_off, 0); }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            if constexpr (FAR) { s.dy[q] = load_quad<false>(d_row, (uint32_t)(f_lane + q * 4 * kWave) * 4u); continue; }
            auto const d = __builtin_amdgcn_raw_buffer_load_b128(d_row, (uint32_t)(f_lane + q * 4 * kWave) * 4u, d_off, 0);
            s.dy[q] = make_float4(__uint_as_float(d[0]), __uint_as_float(d[1]), __uint_as_float(d[2]), __uint_as_float(d[3]));
        }
    };
    auto add = [&](Stage const &s, Entry *tab, auto gated) {
        float const other = __int_as_float(__builtin_amdgcn_ds_bpermute((lane * 4) ^ (4 << s.k), __float_as_int(s.v)));
        // V[k at hi] - V[k at lo]: the lane's own value minus the other's, negated where the lane holds the lower corner
        float const d = __uint_as_float(__float_as_uint(s.v - other) ^ (((uint32_t)~lane << (31 - s.k)) & 0x80000000u));
        if constexpr (BN) {
            float const A = __builtin_amdgcn_inverse_ballot_w64(s.open) ? d * s.gain : 0.0f;
            if (NN == kWave || lane < NN) { tab[lane] = make_float2(A, d * __builtin_fmaf(s.v - s.mean, s.scale, s.shift)); }
        }
        else { if (NN == kWave || lane < NN) { tab[lane] = d * t.inv_step; } }
        wave_fence();
        auto one = [&](float &sum, float y, uint32_t corner) {
            Entry const e = tab[corner];
            if constexpr (decltype(gated)::value) {
                // (no 64-bit shift by a register: where that is the last one that the wavefront has, this GPU shifts by another)
                uint32_t const half = (corner & 32u) ? (uint32_t)(s.open >> 32) : (uint32_t)s.open;
                y = ((half >> (corner & 31u)) & 1u) ? y : 0.0f;
            }
            if constexpr (BN) { sum = __builtin_fmaf(y, e.x, sum + e.y); }
            else              { sum = __builtin_fmaf(y, e, sum); }
        };
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            one(acc[q].x, s.dy[q].x, s.iw[q] & 0xffu);
            one(acc[q].y, s.dy[q].y, (s.iw[q] >> 8) & 0xffu);
            one(acc[q].z, s.dy[q].z, (s.iw[q] >> 16) & 0xffu);
            one(acc[q].w, s.dy[q].w, s.iw[q] >> 24);
        }
    };
    // two stages in turn; the list is read a term ahead of the requests
    auto walk = [&](auto gated) {
        Stage s0, s1;
        int e_ahead = 0;
        if (items > 0) {
            request(list[0], s0);
            e_ahead = list[min(1, items - 1) * step];
        }
        for (int i = 0; i < items; i += 2) {
            if (i + 1 < items) {
                request(e_ahead, s1);
                e_ahead = list[min(i + 2, items - 1) * step];
            }
            add(s0, table[wave][0], gated);
            if (i + 1 < items) {
                if (i + 2 < items) {
                    request(e_ahead, s0);
                    e_ahead = list[min(i + 3, items - 1) * step];
                }
                add(s1, table[wave][1], gated);
            }
        }
    };
    if constexpr (BN) {
        if (discard_word == t.call) { walk(std::true_type{}); }
        else                        { walk(std::false_type{}); }
    }
    else { walk(std::false_type{}); }

    if (a.split) {                              // the shares of the list, added in wavefront order (dx_store_pass)
#pragma unroll
        for (int q = 0; q < Q; ++q) { part[wave][q][lane] = acc[q]; }
        __syncthreads();
        if (wave != 0) { return; }
#pragma unroll
        for (int q = 0; q < Q; ++q) {
#pragma unroll
            for (int w = 1; w < WAVES; ++w) {
                float4 const o = part[w][q][lane];
                acc[q].x += o.x; acc[q].y += o.y; acc[q].z += o.z; acc[q].w += o.w;
            }
        }
    }
    float *const row = a.dx + (size_t)in * a.dx_stride;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
        int const f = f_lane + q * 4 * kWave;
        if (t.dx_quads && f + 3 < a.frame_size) {
            typedef float f32x4 __attribute__((ext_vector_type(4)));
            f32x4 const o = {acc[q].x, acc[q].y, acc[q].z, acc[q].w};
            __builtin_nontemporal_store(o, reinterpret_cast<f32x4 *>(row + f));
        }
        else {
            if (f     < a.frame_size) { row[f]     = acc[q].x; }
            if (f + 1 < a.frame_size) { row[f + 1] = acc[q].y; }
            if (f + 2 < a.frame_size) { row[f + 2] = acc[q].z; }
            if (f + 3 < a.frame_size) { row[f + 3] = acc[q].w; }
        }
    }
}

}  // namespace bbhip
