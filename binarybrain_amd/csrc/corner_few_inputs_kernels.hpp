// dx of layers of few inputs on two-valued inputs: a wavefront keeps the gradients of ALL inputs for its frames in vector registers and walks the nodes.
#pragma once

#include "corner_backward_kernels.hpp"

namespace bbhip {

typedef uint32_t few_u32x4  __attribute__((ext_vector_type(4)));
typedef uint32_t few_u32x8  __attribute__((ext_vector_type(8)));
typedef uint32_t few_u32x16 __attribute__((ext_vector_type(16)));
typedef float    few_f32x2  __attribute__((ext_vector_type(2)));
typedef float    few_f32x4  __attribute__((ext_vector_type(4)));
typedef float    few_f32x8  __attribute__((ext_vector_type(8)));
typedef float    few_f32x16 __attribute__((ext_vector_type(16)));
typedef float    few_f32x32 __attribute__((ext_vector_type(32)));

constexpr int kFewWaves = 8, kFewUnits = 4;        // a workgroup: wavefronts, and groups of frames; the wavefronts of a group share the nodes
constexpr int kFewBatch = 6;            // nodes whose tables a wavefront takes between two barriers, and whose rows of dy are on the way: pairs of nodes
constexpr int kFewFrames = 2;           // consecutive frames per lane
constexpr int kFewMost = 28;            // most inputs: 56 registers of sums

struct FewInputsArgs {
    uint32_t const *x;                  // packed input rows
    int const   *idx;                   // [O][N]
    int const   *rev;                   // reverse table [I][rev_stride]
    float const *dy;
    float       *dx;
    few_f32x4 const *entries;           // [O][few_entry_quads]
    NodeConsts const *node_consts;      // batch-norm
    int const   *listed;                // [I]: see ReverseRows
    uint32_t const *discard;            // batch-norm: see CornerFoldArgs
    uint32_t call;
    int   input_node_size, node_size, frame_size;
    int   x_stride, dy_stride, dx_stride, rev_stride;
};

// quads of a round's tables, whole instructions of 64 (the entries' buffer has room for that much behind the last node)
constexpr int few_round_quads(int n) { return (kFewWaves / kFewUnits * kFewBatch * few_entry_quads(n) + kWave - 1) / kWave * kWave; }
inline size_t few_entry_bytes(int n, int node_size) { return ((size_t)node_size * few_entry_quads(n) + few_round_quads(n)) * 16; }
// LDS: the tables of two rounds and the rows of dy, later four inputs' sums of every wavefront; a word per node
constexpr int few_inputs_lds(int n, int node_size)
{
    int const tables = 2 * few_round_quads(n) * 16, rows = kFewWaves * kFewBatch * kFewFrames * kWave * 4, sums = 4 * kFewWaves * kWave * 8;
    return (tables + rows > sums ? tables + rows : sums) + node_size * 4;
}

// The sums of a lane's frames for every input, in v72 .. v127, and the frames' input bits, in v44 .. v71, where the blocks of assembly below
// pick an input's registers by the vector-register index mode.
struct FewSums {
    few_f32x32 s0; few_f32x16 s1; few_f32x8 s2;
    __device__ __forceinline__ float at(int r) const { return r < 32 ? s0[r & 31] : r < 48 ? s1[r & 15] : s2[r & 7]; }
};
struct FewBits {
    few_u32x16 b0; few_u32x8 b1; few_u32x4 b2;
    __device__ __forceinline__ void set(int i, uint32_t v) { if (i < 16) { b0[i & 15] = v; } else if (i < 24) { b1[i & 7] = v; } else { b2[i & 3] = v; } }
};

// The corner indices of a lane's frames of one node: sum over k of  bits[in_k] << k, the input's register picked by the index mode (on for source 0).
#define BBHIP_FEW_BITS "{v[44:59]}"(bits.b0), "{v[60:67]}"(bits.b1), "{v[68:71]}"(bits.b2)
template <int N>
__device__ __forceinline__ uint32_t few_inputs_index(FewBits const &bits, int const (&in)[N])
{
    uint32_t q;
    if constexpr (N == 6) {
        asm volatile("s_set_gpr_idx_on %[i0], gpr_idx(SRC0)\n\tv_mov_b32 %[q], v44\n\t"
                     "s_set_gpr_idx_idx %[i1]\n\tv_lshl_or_b32 %[q], v44, 1, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i2]\n\tv_lshl_or_b32 %[q], v44, 2, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i3]\n\tv_lshl_or_b32 %[q], v44, 3, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i4]\n\tv_lshl_or_b32 %[q], v44, 4, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i5]\n\tv_lshl_or_b32 %[q], v44, 5, %[q]\n\t"
                     "s_set_gpr_idx_off"
                     : [q] "=&v"(q) : [i0] "s"(in[0]), [i1] "s"(in[1]), [i2] "s"(in[2]), [i3] "s"(in[3]), [i4] "s"(in[4]), [i5] "s"(in[5]), BBHIP_FEW_BITS);
    }
    else if constexpr (N == 5) {
        asm volatile("s_set_gpr_idx_on %[i0], gpr_idx(SRC0)\n\tv_mov_b32 %[q], v44\n\t"
                     "s_set_gpr_idx_idx %[i1]\n\tv_lshl_or_b32 %[q], v44, 1, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i2]\n\tv_lshl_or_b32 %[q], v44, 2, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i3]\n\tv_lshl_or_b32 %[q], v44, 3, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i4]\n\tv_lshl_or_b32 %[q], v44, 4, %[q]\n\t"
                     "s_set_gpr_idx_off"
                     : [q] "=&v"(q) : [i0] "s"(in[0]), [i1] "s"(in[1]), [i2] "s"(in[2]), [i3] "s"(in[3]), [i4] "s"(in[4]), BBHIP_FEW_BITS);
    }
    else if constexpr (N == 4) {
        asm volatile("s_set_gpr_idx_on %[i0], gpr_idx(SRC0)\n\tv_mov_b32 %[q], v44\n\t"
                     "s_set_gpr_idx_idx %[i1]\n\tv_lshl_or_b32 %[q], v44, 1, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i2]\n\tv_lshl_or_b32 %[q], v44, 2, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i3]\n\tv_lshl_or_b32 %[q], v44, 3, %[q]\n\t"
                     "s_set_gpr_idx_off"
                     : [q] "=&v"(q) : [i0] "s"(in[0]), [i1] "s"(in[1]), [i2] "s"(in[2]), [i3] "s"(in[3]), BBHIP_FEW_BITS);
    }
    else if constexpr (N == 3) {
        asm volatile("s_set_gpr_idx_on %[i0], gpr_idx(SRC0)\n\tv_mov_b32 %[q], v44\n\t"
                     "s_set_gpr_idx_idx %[i1]\n\tv_lshl_or_b32 %[q], v44, 1, %[q]\n\t"
                     "s_set_gpr_idx_idx %[i2]\n\tv_lshl_or_b32 %[q], v44, 2, %[q]\n\t"
                     "s_set_gpr_idx_off"
                     : [q] "=&v"(q) : [i0] "s"(in[0]), [i1] "s"(in[1]), [i2] "s"(in[2]), BBHIP_FEW_BITS);
    }
    else {
        asm volatile("s_set_gpr_idx_on %[i0], gpr_idx(SRC0)\n\tv_mov_b32 %[q], v44\n\t"
                     "s_set_gpr_idx_idx %[i1]\n\tv_lshl_or_b32 %[q], v44, 1, %[q]\n\t"
                     "s_set_gpr_idx_off"
                     : [q] "=&v"(q) : [i0] "s"(in[0]), [i1] "s"(in[1]), BBHIP_FEW_BITS);
    }
    return q;
}
#undef BBHIP_FEW_BITS

// sums[in Q + j] += slope[j] g[j], j < Q: register v72 + in Q + j, picked by the index mode (on for source 2 and the destination); two inputs of a node per block
__device__ __forceinline__ void few_inputs_add(FewSums &s, int at0, int at1, float const (&g)[2], few_f32x2 a, few_f32x2 b)
{
    asm volatile("s_set_gpr_idx_on %[at0], gpr_idx(SRC2,DST)\n\t"
                 "v_fma_f32 v72, %[a0], %[g0], v72\n\tv_fma_f32 v73, %[a1], %[g1], v73\n\t"
                 "s_set_gpr_idx_idx %[at1]\n\t"
                 "v_fma_f32 v72, %[b0], %[g0], v72\n\tv_fma_f32 v73, %[b1], %[g1], v73\n\t"
                 "s_set_gpr_idx_off"
                 : "+{v[72:103]}"(s.s0), "+{v[104:119]}"(s.s1), "+{v[120:127]}"(s.s2)
                 : [at0] "s"(at0), [at1] "s"(at1), [g0] "v"(g[0]), [g1] "v"(g[1]), [a0] "v"(a[0]), [a1] "v"(a[1]), [b0] "v"(b[0]), [b1] "v"(b[1]));
}
__device__ __forceinline__ void few_inputs_add(FewSums &s, int at0, float const (&g)[2], few_f32x2 a)
{
    asm volatile("s_set_gpr_idx_on %[at0], gpr_idx(SRC2,DST)\n\t"
                 "v_fma_f32 v72, %[a0], %[g0], v72\n\tv_fma_f32 v73, %[a1], %[g1], v73\n\t"
                 "s_set_gpr_idx_off"
                 : "+{v[72:103]}"(s.s0), "+{v[104:119]}"(s.s1), "+{v[120:127]}"(s.s2)
                 : [at0] "s"(at0), [g0] "v"(g[0]), [g1] "v"(g[1]), [a0] "v"(a[0]), [a1] "v"(a[1]));
}

// dx of a lane's frames from the lists of the reverse table, for inputs `first`, first + kShares, ...: whatever the lists say, the tables of lut_dx_few_inputs_kernel
// and its arithmetic.  (An entry that is no connection adds nothing.)
template <int N, bool BN>
__device__ __forceinline__ void few_inputs_by_lists(FewInputsArgs const &a, int first, int f_lane, bool gated)
{
    constexpr int NN = 1 << N, kQuads = few_entry_quads(N);
    typedef __attribute__((address_space(4))) int const const_int;
    typedef __attribute__((address_space(4))) NodeConsts const const_consts;
    const_consts *consts = (const_consts *)a.node_consts;
#pragma nounroll
    for (int i = first; i < a.input_node_size; i += kFewWaves / kFewUnits) {
        const_int *list = (const_int *)(a.rev + (size_t)i * a.rev_stride);
        int const fan = list[0];
        few_f32x2 sum = 0.0f;
#pragma nounroll
        for (int t = 1; t <= fan; ++t) {
            uint32_t const e = (uint32_t)list[t], node = e / (uint32_t)N;
            int const k = (int)(e - node * N);
            if (node >= (uint32_t)a.node_size) { continue; }             // wave-uniform
            const_int *in = (const_int *)(a.idx + (size_t)node * N);
#pragma unroll
            for (int q = 0; q < kFewFrames; ++q) {
                int const f = min(f_lane + q, a.frame_size - 1);
                uint32_t corner = 0;
#pragma unroll
                for (int j = 0; j < N; ++j) { corner |= ((a.x[(size_t)min((uint32_t)in[j], (uint32_t)a.input_node_size - 1) * a.x_stride + (f >> 5)] >> (f & 31)) & 1u) << j; }
                float d = a.dy[(size_t)node * a.dy_stride + f];
                if (BN && gated) {
                    uint64_t const open = consts[node].open;
                    uint32_t const half = (corner & 32u) ? (uint32_t)(open >> 32) : (uint32_t)open;
                    d = ((half >> (corner & 31u)) & 1u) ? d : 0.0f;
                }
                float const *entry = reinterpret_cast<float const *>(a.entries + (size_t)node * kQuads + corner);
                float const g = BN ? __builtin_fmaf(d, entry[0], entry[1]) : d * entry[0];
                sum[q] = __builtin_fmaf(k < 2 ? entry[2 + k] : entry[NN * 4 + k - 2], g, sum[q]);
            }
        }
#pragma unroll
        for (int q = 0; q < kFewFrames; ++q) { if (f_lane + q < a.frame_size) { a.dx[(size_t)i * a.dx_stride + f_lane + q] = sum[q]; } }
    }
}

// A wavefront owns 128 frames, two consecutive ones per lane, and the sums dx[input][frame] of all (up to 28) inputs for them.  It walks the nodes; a frame's
// corner index p comes from the input bits in registers, the frame's entry of the node's table from LDS, and each of the node's inputs k gets
//     dx[in_k] += d_k[p] g,      g = gain[p] dy + E[p]        (A[p] = d_k[p] gain[p] and B[p] = d_k[p] E[p] of lut_dx_table_kernel; E = 0 in plain layers),
// so that dy is read once, where a walk over every input's consumers reads it once per connection, and no corner indices are kept by the launch before.
// The node's tables are formed by corner_fold, once per call.
// The wiring is that of the index table where the launch before has found the same in the reverse table (ReverseRows); else (a caller's own table that
// leaves connections out, say) the workgroup goes by the lists, an input after another, without hurry.
// Bound by LDS (two random 16-byte reads per frame and node: 20 clocks per 64 frames, 22 with the row of dy by the counters, 12 of them for bank conflicts, LDS
// busy for 68 % of the time; four 8-byte reads take 18 if the compiler leaves them apart, 40 if it pairs them) and by what the four wavefronts of a SIMD leave idle around it.  27 inputs x 216 nodes x 230400 frames, six per node: 80 -> 52 us (dy at 3.9 TB/s), and
// the sums launch, which has no indices to keep, 50 -> 38; with tables formed by the workgroups themselves 59 us, with dy through registers 53.
// (230400 frames are 450 workgroups of 512 frames, of which the device holds 512 at once.)
template <int N, bool BN>
__global__ __launch_bounds__(kFewWaves * kWave) __attribute__((amdgpu_waves_per_eu(4, 4))) void lut_dx_few_inputs_kernel(FewInputsArgs a)
{
    constexpr int NN = 1 << N, Q = kFewFrames, kFrames = kWave * Q, kShares = kFewWaves / kFewUnits, kPairs = kFewBatch / 2, kQuads = few_entry_quads(N);
    constexpr int kRound = kShares * kFewBatch, kTable = few_round_quads(N);      // nodes of the workgroup between two barriers
    extern __shared__ __align__(16) few_f32x4 tables[];                 // [2][kTable]: [share][kFewBatch][kQuads]
    few_f32x2 *const rows = reinterpret_cast<few_f32x2 *>(tables + 2 * kTable);        // [wavefront][kFewBatch][lane]: dy
    uint32_t *const wiring = reinterpret_cast<uint32_t *>(tables + few_inputs_lds(N, 0) / 16);           // a node's inputs, five bits each
    int const wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave)), lane = threadIdx.x & (kWave - 1);
    int const unit = wave % kFewUnits, share = wave / kFewUnits, begin = share * kFewBatch;
    int const f_unit = (xcd_remap(blockIdx.x, gridDim.x) * kFewUnits + unit) * kFrames, f_lane = f_unit + Q * lane;
    int const last = a.node_size - 1;
    uint32_t const last_input = (uint32_t)a.input_node_size - 1;

    typedef __attribute__((address_space(4))) uint32_t const const_word;
    typedef __attribute__((address_space(4))) NodeConsts const const_consts;
    const_consts *consts = (const_consts *)a.node_consts;
    uint32_t const discard_word = BN ? *(const_word *)a.discard : 0u;
    int listed = lane < a.input_node_size ? a.listed[lane] : 0;

    // Tables and rows of dy go from memory to LDS without a stop in registers, 1 KB per instruction: 16 bytes per lane, to the address in M0 and up.  A round's
    // tables are consecutive, a part of them for every wavefront; dy comes in pairs of nodes, half a wavefront for each.  Loads return in order, so that what
    // is waited for is told by how many younger ones there are: a round asks for the tables of the next, then for a pair of rows after each pair it has used.
    // Every address lies within the buffers: what there is no node or frame for repeats the last one's.
    constexpr int kPieces = kTable / kWave, kEach = (kPieces + kFewWaves - 1) / kFewWaves;
    uint32_t const lds_tables = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void *)tables;
    uint32_t const lds_rows = lds_tables + 2 * kTable * 16 + (uint32_t)wave * (kFewBatch * kFrames * 4);
    // (M0 must be written a wait state before such a load reads it; the compiler, which does not look into the asm, would put the s_nop there too)
    auto load_to_lds = [](uint32_t lds, uint32_t off, __amdgpu_buffer_rsrc_t from, uint32_t base) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" :: "s"(lds), "v"(off), "s"(from), "s"(base) : "memory");
    };
    __amdgpu_buffer_rsrc_t const er = row_descriptor(a.entries, 0, 0, (uint32_t)a.node_size * (kQuads * 16u) + kTable * 16u);
    int const last_round = last / kRound;
    auto request_tables = [&](int round) {
#pragma unroll
        for (int p = 0; p < kEach; ++p) {        // (every wavefront issues the same number: a piece too many is loaded twice)
            uint32_t const piece = (uint32_t)min(wave * kEach + p, kPieces - 1) * 1024u;
            load_to_lds(lds_tables + (uint32_t)(round & 1) * (kTable * 16u) + piece, (uint32_t)lane * 16u, er,
                        (uint32_t)min(round, last_round) * (kRound * kQuads * 16u) + piece);
        }
    };
    uint32_t const dy_pitch = (uint32_t)a.dy_stride * 4u;
    __amdgpu_buffer_rsrc_t const dyr = row_descriptor(a.dy, 0, 0, (uint32_t)last * dy_pitch + (uint32_t)((a.frame_size + 3) & ~3) * 4u);
    uint32_t const dy_one = (uint32_t)min(f_unit + (lane & 31) * 4, ((a.frame_size + 3) & ~3) - 4) * 4u, dy_two = dy_one + (lane & 32 ? dy_pitch : 0u);
    auto request_rows = [&](int node, int pair) {
        load_to_lds(lds_rows + (uint32_t)pair * (2 * kFrames * 4), node < last ? dy_two : dy_one, dyr, (uint32_t)min(node, last) * dy_pitch);
    };
    request_tables(0);
    for (int node = threadIdx.x; node < a.node_size; node += kFewWaves * kWave) {
        uint32_t w = 0;
#pragma unroll
        for (int k = 0; k < N; ++k) { w |= min((uint32_t)a.idx[(size_t)node * N + k], last_input) << (5 * k); }
        wiring[node] = w;
    }

    // the lane's frames of every input: bit j of the input at bit 16 j + 4 (an index is an offset into entries of 16 bytes)
    FewBits bits;
    {
        uint32_t const x_bytes = (uint32_t)((a.frame_size + 31) >> 5) * 4u, x_pitch = (uint32_t)a.x_stride * 4u;
        __amdgpu_buffer_rsrc_t const xr = row_descriptor(a.x, 0, 0, last_input * x_pitch + x_bytes);
#pragma unroll
        for (int i = 0; i < kFewMost; ++i) {
            uint32_t const w = __builtin_amdgcn_raw_buffer_load_b32(xr, min((uint32_t)(f_lane >> 5) * 4u, x_bytes - 4u), min((uint32_t)i, last_input) * x_pitch, 0) >> (f_lane & 31);
            bits.set(i, ((w & 3u) * 0x00080010u) & 0x00100010u);
        }
    }
    FewSums sums;
    sums.s0 = 0.0f; sums.s1 = 0.0f; sums.s2 = 0.0f;

#pragma unroll
    for (int p = 0; p < kPairs; ++p) { request_rows(begin + 2 * p, p); }

    // a node's corner indices are formed while the node before it waits for its entries
    int in[N];
    auto take_index = [&](uint32_t of_lane, int j) {
        uint32_t const w = (uint32_t)__builtin_amdgcn_readlane((int)of_lane, j);
#pragma unroll
        for (int k = 0; k < N; ++k) { in[k] = (int)((w >> (5 * k)) & 31u); }
        return few_inputs_index<N>(bits, in);
    };
    auto wiring_of = [&](int base) { return wiring[min(base + (lane < kFewBatch ? lane : 0), last)]; };        // lane j: of node j of the share's round
    __syncthreads();
#pragma unroll
    for (int o = 1; o < 32; o <<= 1) { listed += lane_xor(listed, o); }
    static_assert(kFewMost <= 32, "half a wavefront's lanes");
    if (__builtin_amdgcn_readfirstlane(listed) != a.node_size * N) {     // the same for all wavefronts
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                 // (nothing is on its way to LDS when the workgroup ends)
        few_inputs_by_lists<N, BN>(a, share, f_lane, discard_word == a.call);
        return;
    }
    uint32_t words = wiring_of(begin), quad = take_index(words, 0);
    few_f32x2 const *const my_rows = rows + wave * (kFewBatch * kWave) + lane;

    auto walk = [&](auto gated) {
        for (int round = 0; round * kRound < a.node_size; ++round) {
            int const base = begin + round * kRound;
            asm volatile("s_waitcnt vmcnt(%0)" :: "i"(kPairs) : "memory");              // younger than the round's tables: kPairs pairs of rows
            __syncthreads();
            request_tables(round + 1);
            few_f32x4 const *const mine = tables + (round & 1) * kTable + begin * kQuads;
            uint32_t const words_next = wiring_of(base + kRound);
#pragma unroll
            for (int j = 0; j < kFewBatch; ++j) {
                int const node = base + j;
                if (j % 2 == 0) { asm volatile("s_waitcnt vmcnt(%0)" :: "i"(kPairs - 1 + kEach) : "memory"); }
                few_f32x2 const dy = my_rows[j * kWave];
                few_f32x4 const *tab = mine + j * kQuads;
                few_f32x4 e0[Q], e1[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    uint32_t const off = q ? quad >> 16 : quad & 0xffffu;
                    e0[q] = *reinterpret_cast<few_f32x4 const *>(reinterpret_cast<char const *>(tab) + off);
                    if (N > 2) { e1[q] = *reinterpret_cast<few_f32x4 const *>(reinterpret_cast<char const *>(tab + NN) + off); }
                }
                uint32_t const corners = quad;
                int at[N];
#pragma unroll
                for (int k = 0; k < N; ++k) { at[k] = in[k] * Q; }
                quad = j + 1 < kFewBatch ? take_index(words, j + 1) : take_index(words_next, 0);      // of the next node
                float g[Q];
#pragma unroll
                for (int q = 0; q < Q; ++q) {
                    float d = dy[q];
                    if constexpr (decltype(gated)::value) {              // behind a closed window dy counts as 0 whatever it is
                        uint64_t const open = consts[min(node, last)].open;
                        uint32_t const corner = (q ? corners >> 16 : corners & 0xffffu) >> 4;
                        uint32_t const half = (corner & 32u) ? (uint32_t)(open >> 32) : (uint32_t)open;
                        d = ((half >> (corner & 31u)) & 1u) ? d : 0.0f;
                    }
                    g[q] = BN ? __builtin_fmaf(d, e0[q][0], e0[q][1]) : d * e0[q][0];
                }
                auto slopes = [&](int k) {
                    few_f32x2 s;
#pragma unroll
                    for (int q = 0; q < Q; ++q) { s[q] = k < 2 ? e0[q][2 + k] : e1[q][k - 2]; }
                    return s;
                };
                if (node <= last) {                                      // wave-uniform
#pragma unroll
                    for (int k = 0; k + 1 < N; k += 2) { few_inputs_add(sums, at[k], at[k + 1], g, slopes(k), slopes(k + 1)); }
                    if constexpr (N % 2) { few_inputs_add(sums, at[N - 1], g, slopes(N - 1)); }
                }
                __builtin_amdgcn_sched_barrier(0);
                if (j % 2) { request_rows(node - 1 + kRound, j / 2); }
            }
            words = words_next;
        }
    };
    if constexpr (BN) {
        if (discard_word == a.call) { walk(std::true_type{}); }
        else                        { walk(std::false_type{}); }
    }
    else { walk(std::false_type{}); }

    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                     // (LDS is used for something else from here on)
    __syncthreads();
    // the shares' sums, four inputs of every unit at a time: share s adds up and stores input s mod 4 in share order
    few_f32x2 *const part = reinterpret_cast<few_f32x2 *>(tables);                 // [4][share][unit][lane]
#pragma unroll
    for (int i0 = 0; i0 < kFewMost; i0 += 4) {
        if (i0 >= a.input_node_size) { break; }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (i0 + i < kFewMost) {
                few_f32x2 v;
#pragma unroll
                for (int q = 0; q < Q; ++q) { v[q] = sums.at((i0 + i) * Q + q); }
                part[(i * kFewWaves + wave) * kWave + lane] = v;
            }
        }
        __syncthreads();
        for (int i = share; i < 4; i += kShares) {
            if (i0 + i >= a.input_node_size) { break; }
            few_f32x2 sum = part[(i * kFewWaves + unit) * kWave + lane];
#pragma unroll
            for (int s = 1; s < kShares; ++s) { sum += part[(i * kFewWaves + s * kFewUnits + unit) * kWave + lane]; }
            float *const row = a.dx + (size_t)(i0 + i) * a.dx_stride + f_lane;
            if (f_lane + Q <= a.frame_size) { __builtin_nontemporal_store(sum, reinterpret_cast<few_f32x2 *>(row)); }
            else {
#pragma unroll
                for (int q = 0; q < Q; ++q) { if (f_lane + q < a.frame_size) { row[q] = sum[q]; } }
            }
        }
        __syncthreads();
    }
}

}  // namespace bbhip
