// Forward pass of the LUT layers on two-valued inputs, 32 frames per lane and step of index forming.
#pragma once

#include "corner_index.hpp"
#include "lut_kernels.hpp"

namespace bbhip {

constexpr int kByteBlock = 32 * kWave;               // frames whose corner indices a wavefront forms in one step: 32 per lane
constexpr int kByteWaves = 16;                       // most wavefronts of a workgroup
constexpr int kByteFusedFrames = 49152;              // most frames of a one-launch training pass: a byte of LDS per frame

// LDS of lut_forward_bytes_kernel: per wavefront two tables and two sums, and the indices
inline int forward_bytes_lds(int waves, int index_blocks) { return waves * (2 * kWave + 2) * 4 + index_blocks * kByteBlock; }

// The words of a lane's 32 frames from frame base + 32 lane (base a multiple of 64)
template <int N, int XMODE>
struct WordLoad {
    __amdgpu_buffer_rsrc_t row[N];
    __device__ __forceinline__ void open(FwdArgs const &a, int const (&in)[N])
    {
        uint32_t const bytes = (XMODE == kXBit) ? (uint32_t)((a.frame_size + 31) >> 5) * 4u : (uint32_t)a.frame_size * 4u;
#pragma unroll
        for (int k = 0; k < N; ++k) { row[k] = row_descriptor(a.x, in[k], a.x_stride, bytes); }
    }
    __device__ __forceinline__ void load(int base, int lane, int f_end, uint32_t (&w)[N]) const
    {
        if constexpr (XMODE == kXBit) {
#pragma unroll
            for (int k = 0; k < N; ++k) { w[k] = __builtin_amdgcn_raw_buffer_load_b32(row[k], (uint32_t)((base >> 5) + lane) * 4u, 0, 0); }
        }
        else {                                       // fp32 frames: 64 of them are one ballot, two lanes' words
#pragma unroll
            for (int k = 0; k < N; ++k) { w[k] = 0; }
            int const steps = min(kByteBlock / kWave, (f_end - base + kWave - 1) / kWave);
            constexpr int U = 4;                     // steps whose loads are issued together (past the row: zeros)
            for (int u0 = 0; u0 < steps; u0 += U) {
                float v[U][N];
#pragma unroll
                for (int u = 0; u < U; ++u) {
#pragma unroll
                    for (int k = 0; k < N; ++k) { v[u][k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(row[k], (uint32_t)(base + (u0 + u) * kWave + lane) * 4u, 0, 0)); }
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
#pragma unroll
                    for (int k = 0; k < N; ++k) {
                        uint64_t const m = __ballot(v[u][k] > 0.5f);
                        uint32_t const half = (lane & 1) ? (uint32_t)(m >> 32) : (uint32_t)m;
                        w[k] = ((lane >> 1) == u0 + u) ? half : w[k];
                    }
                }
            }
        }
    }
};

// the word of eight lanes of four frames each, from the lanes' four bits
__device__ __forceinline__ uint32_t quad_word(uint32_t m, int lane)
{
    m <<= 4 * (lane & 7);
    m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1, 0xf, 0xf, true);                  // quad_perm [1, 0, 3, 2]
    m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xf, 0xf, true);                  // quad_perm [2, 3, 0, 1]
    m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xf, 0xf, true);                 // row_half_mirror
    return m;
}

// One wavefront = one node x one unit of frames in blocks of 2048 (kinds 0, 1, 2 as in lut_forward_kernel), or, for a batch-norm training pass
// in one launch (kStatInline), a.node_waves wavefronts = one node and all its frames.  A lane loads the words of 32 frames of each input and turns
// them into corner indices (corner_bytes: two instructions per frame and lane where the scalar lane masks of lut_forward_corner_kernel take
// N + 2), times 4, so that a byte is an offset into a table in LDS: a wavefront's 64 random reads of it take 4 clocks, a ds_bpermute 7.
//   statistics  every lane sums V - C0 and its square over its own 32 frames;
//   output      the index bytes go through LDS to the lanes that hold four consecutive frames each (16-byte stores of y; the packed copy collects
//               its words over a block and leaves by one store), packed output is assembled by the lane that formed the indices.
// In one launch the indices of all frames stay in LDS between the two, so nothing is gathered or formed twice, and the wavefronts of a node
// exchange their two sums there; where nodes are few, several workgroups hold the indices of a part of a node's frames each and write its output
// (forward_out_blocks), and all of them sum the statistics of all frames.  The kernel is bound by the fp32 output where there is one, else by its chain of latencies (wiring, words, tables).
// Measured against lut_forward_corner_kernel's statistics and output launches: 4096 x 4096 x 8192 fp32 output 36 us (3.8 TB/s written) instead of
// 25 + 31; 2001 x 3003 x 5005 packed 14 us instead of 15 + 13; 216 nodes x 230400 frames (two launches) 14 + 46 us instead of 22 + 46; packed
// inference of 2048 nodes x 3500 frames 6.2 us instead of 11.5.
template <int N, int XMODE, int YMODE, int KIND>
__global__ __launch_bounds__(kByteWaves * kWave) void lut_forward_bytes_kernel(FwdArgs a)
{
    constexpr int NN = 1 << N, kPasses = kByteBlock / (4 * kWave), kBlockWords = kByteBlock / 4;
    extern __shared__ __align__(16) uint32_t lds[];
    int const waves = blockDim.x / kWave, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave));
    int const lane = threadIdx.x & (kWave - 1);
    bool const fused = (KIND == 1) && a.stat_mode == kStatInline;
    float *const stat_tab = reinterpret_cast<float *>(lds) + wave * 2 * kWave, *const out_tab = stat_tab + kWave;
    float *const sums = reinterpret_cast<float *>(lds) + waves * 2 * kWave;

    int const nw = fused ? a.node_waves : 1, sub = wave % nw;
    int ck = 0, tile;
    int const lid = xcd_remap(blockIdx.x, a.chunk_count * a.tiles.count);
    split_tile(lid, a.tiles, ck, tile);
    int const slot = wave / nw;
    int node = tile * (waves / nw) + slot;
    bool const live = node < a.node_size;
    if (!live) {
        if (nw == 1) { return; }
        node = a.node_size - 1;                      // (with barriers ahead: repeats the last node and stores nothing)
    }
    int const f_begin = (YMODE != kYBit && fused) ? 0 : ck * a.chunk, f_end = min(f_begin + a.chunk, a.frame_size);
    int const blocks = (f_end - f_begin + kByteBlock - 1) / kByteBlock;
    // in one launch with fp32 output: the blocks whose output is this workgroup's
    bool const parted = YMODE != kYBit && fused && a.out_blocks < blocks;
    int const out_first = parted ? ck * a.out_blocks : 0, out_end = parted ? min(out_first + a.out_blocks, blocks) : blocks;
    uint32_t *const bytes = lds + waves * (2 * kWave + 2) + (fused ? slot * (parted ? a.out_blocks : blocks) : wave) * kBlockWords;

    int in[N];
#pragma unroll
    for (int k = 0; k < N; ++k) { in[k] = a.idx[node * N + k]; }
    WordLoad<N, XMODE> words;
    words.open(a, in);
    uint32_t w[N];
    if (XMODE == kXBit && sub < blocks) { words.load(f_begin + sub * kByteBlock, lane, f_end, w); }

    // the node's tables (as in lut_forward_corner_kernel)
    int const i = lane & (NN - 1);
    float corner, c0 = 0.0f, table_c = 0.0f, table_w = 0.0f;
    bool clamp_store = false;
    if (a.W_inline != nullptr) {
        float t = a.W_inline[(size_t)node * NN + i];
        if (a.clamp_W != nullptr) {
            float const tc = fminf(a.clamp_hi, fmaxf(a.clamp_lo, t));
            clamp_store = (tc != t);
            t = tc;
        }
        table_w = t;
        if (a.lut_binarize) { t = (t > 0.5f) ? 1.0f : 0.0f; }
        table_c = centred_butterfly<N>(t, i);
        corner = corner_butterfly<N>(table_c, i, a.bias);
        c0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(table_c)));
    }
    else {
        corner = a.V[(size_t)node * NN + i];
        if (KIND == 2 || (KIND == 1 && (a.stat_mode == kStatPartial || a.stat_mode == kStatInline))) { c0 = a.C[(size_t)node * NN]; }
    }

    auto lookup = [](float const *tab, uint32_t quad, int j) {
        return *reinterpret_cast<float const *>(reinterpret_cast<char const *>(tab) + ((quad >> (8 * j)) & 0xffu));
    };
    float s1 = 0.0f, s2 = 0.0f;
    auto statistics = [&](uint32_t const (&quad)[8], int frames) {          // frames: how many of the lane's 32 belong to the unit
        if (__builtin_amdgcn_ballot_w64(frames < 32) == 0) {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float const d = lookup(stat_tab, quad[q], j);
                    s1 += d;
                    s2 = __builtin_fmaf(d, d, s2);
                }
            }
        }
        else {
#pragma unroll
            for (int q = 0; q < 8; ++q) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float const d = (4 * q + j < frames) ? lookup(stat_tab, quad[q], j) : 0.0f;
                    s1 += d;
                    s2 = __builtin_fmaf(d, d, s2);
                }
            }
        }
    };
    auto keep = [&](uint32_t const (&quad)[8], uint32_t *block) {
        uint4 *out = reinterpret_cast<uint4 *>(block + 8 * lane);
        out[0] = make_uint4(quad[0], quad[1], quad[2], quad[3]);
        out[1] = make_uint4(quad[4], quad[5], quad[6], quad[7]);
    };
    // packed output of the lane's 32 frames
    auto output_word = [&](uint32_t const (&quad)[8], int base) {
        int const f = base + 32 * lane, frames = f_end - f;
        uint32_t word = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
#pragma unroll
            for (int j = 0; j < 4; ++j) { word |= __float_as_uint(lookup(out_tab, quad[q], j)) << (4 * q + j); }
        }
        if (frames < 32) { word &= (frames > 0) ? (1u << frames) - 1u : 0u; }
        if (live && frames > 0) { reinterpret_cast<uint32_t *>(a.y)[(size_t)node * a.y_stride + (f >> 5)] = word; }
    };
    // fp32 output of one pass of 256 frames whose index bytes are in LDS
    auto output_pass = [&](uint32_t const *pass, int fb) {
        float *const row = reinterpret_cast<float *>(a.y) + (size_t)node * a.y_stride;
        int const f = fb + 4 * lane;
        uint32_t const at = pass[lane];
        typedef float f32x4 __attribute__((ext_vector_type(4)));
        f32x4 v;
#pragma unroll
        for (int j = 0; j < 4; ++j) { v[j] = lookup(out_tab, at, j); }
        if (YMODE == kYBinarize && a.y_bits != nullptr) {
            uint32_t m = 0;
#pragma unroll
            for (int j = 0; j < 4; ++j) { m |= (v[j] != 0.0f && f + j < f_end) ? 1u << j : 0u; }
            m = quad_word(m, lane);
            if (live && f < f_end && (lane & 7) == 0) { a.y_bits[(size_t)node * a.y_bits_stride + (f >> 5)] = m; }
        }
        if (!live) { return; }
        if (a.y_quads && f + 3 < f_end) { __builtin_nontemporal_store(v, reinterpret_cast<f32x4 *>(row + f)); }
        else {
#pragma unroll
            for (int j = 0; j < 4; ++j) { if (f + j < f_end) { row[f + j] = v[j]; } }
        }
    };
    // fp32 output of a block whose index bytes are in LDS
    auto output_rows = [&](uint32_t const *block, int base) {
        float *const row = reinterpret_cast<float *>(a.y) + (size_t)node * a.y_stride;
        uint32_t mine = 0;                           // word (lane & 7) * 8 + (lane >> 3) of the block's packed copy
#pragma unroll
        for (int p = 0; p < kPasses; ++p) {
            int const fb = base + p * 4 * kWave, f = fb + 4 * lane;
            if (fb >= f_end) { break; }              // wave-uniform
            uint32_t const at = block[p * kWave + lane];
            typedef float f32x4 __attribute__((ext_vector_type(4)));
            f32x4 v;
#pragma unroll
            for (int j = 0; j < 4; ++j) { v[j] = lookup(out_tab, at, j); }
            if (YMODE == kYBinarize && a.y_bits != nullptr) {
                uint32_t m = 0;
#pragma unroll
                for (int j = 0; j < 4; ++j) { m |= (v[j] != 0.0f && f + j < f_end) ? 1u << j : 0u; }
                m = quad_word(m, lane);
                mine = ((lane & 7) == p) ? m : mine;
            }
            if (!live) { continue; }
            if (a.y_quads && f + 3 < f_end) { __builtin_nontemporal_store(v, reinterpret_cast<f32x4 *>(row + f)); }
            else {
#pragma unroll
                for (int j = 0; j < 4; ++j) { if (f + j < f_end) { row[f + j] = v[j]; } }
            }
        }
        if (YMODE == kYBinarize && a.y_bits != nullptr && live) {
            int const f = base + 32 * ((lane & 7) * 8 + (lane >> 3));
            if (f < f_end) { a.y_bits[(size_t)node * a.y_bits_stride + (f >> 5)] = mine; }
        }
    };
    // what a frame fetches: the finished output, for packed output as a bit
    auto write_out_table = [&](float mean, float rstd) {
        float y = (KIND == 1) ? batch_norm_output(corner, mean, rstd, a.gamma, a.beta) : corner;
        if (YMODE == kYClamp)         { y = __builtin_amdgcn_fmed3f(y, 0.0f, 1.0f); }
        else if (YMODE == kYBinarize) { y = (y > 0.5f) ? 1.0f : 0.0f; }
        else                          { y = __uint_as_float((y > 0.5f) ? 1u : 0u); }
        out_tab[lane] = y;
        wave_fence();
    };

    float mean = 0.0f, var = 0.0f, rstd = 1.0f;
    uint32_t quad[8];
    if (fused || KIND == 2) {
        stat_tab[lane] = corner - c0;
        wave_fence();
        for (int b = sub; b < blocks; b += nw) {
            int const base = f_begin + b * kByteBlock;
            if (XMODE != kXBit) { words.load(base, lane, f_end, w); }
            corner_bytes<N, 2>(w, quad);
            if (XMODE == kXBit && b + nw < blocks) { words.load(base + nw * kByteBlock, lane, f_end, w); }
            if (fused && (YMODE == kYBit || (b >= out_first && b < out_end))) { keep(quad, bytes + (b - out_first) * kBlockWords); }
            statistics(quad, f_end - (base + 32 * lane));
        }
        if (KIND == 2) { forward_store_stats(a, ck, node, live, lane, s1, s2); }
        else {
            s1 = wave_sum(s1);
            s2 = wave_sum(s2);
            if (nw > 1) {
                if (lane == 0) { sums[2 * wave] = s1; sums[2 * wave + 1] = s2; }
                __syncthreads();
                s1 = 0.0f; s2 = 0.0f;
                for (int k = 0; k < nw; ++k) { s1 += sums[2 * (slot * nw + k)]; s2 += sums[2 * (slot * nw + k) + 1]; }
            }
            batch_statistics(s1, s2, c0, a.frame_size, mean, var, rstd);
            write_out_table(mean, rstd);
            if (parted) {
                // a few blocks for all wavefronts of the node: pass by pass, whoever formed the bytes (a barrier lies between)
                int const passes = (out_end - out_first) * kPasses;
                for (int q = sub; q < passes; q += nw) {
                    int const fb = out_first * kByteBlock + q * 4 * kWave;
                    if (fb < f_end) { output_pass(bytes + q * kWave, fb); }
                }
            }
            else {
                // the blocks that this wavefront formed
                for (int b = sub; b < blocks; b += nw) {
                    int const base = f_begin + b * kByteBlock;
                    uint32_t const *block = bytes + b * kBlockWords;
                    if (YMODE == kYBit) {
                        uint4 const *own = reinterpret_cast<uint4 const *>(block + 8 * lane);
                        uint4 const lo = own[0], hi = own[1];
                        uint32_t const q[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
                        output_word(q, base);
                    }
                    else { output_rows(block, base); }
                }
            }
        }
    }
    else {
        if (KIND == 1) { forward_statistics(a, node, lane, c0, mean, var, rstd); }
        write_out_table(mean, rstd);
        for (int b = 0; b < blocks; ++b) {
            int const base = f_begin + b * kByteBlock;
            if (XMODE != kXBit) { words.load(base, lane, f_end, w); }
            corner_bytes<N, 2>(w, quad);
            if (XMODE == kXBit && b + 1 < blocks) { words.load(base + kByteBlock, lane, f_end, w); }
            if (YMODE == kYBit) { output_word(quad, base); }
            else {
                keep(quad, bytes);
                wave_fence();
                output_rows(bytes, base);
                wave_fence();                        // the next block overwrites the bytes
            }
        }
    }

    // (stores of the set-up's results at the end: ahead of the loads they would be waited for with them)
    if (sub == 0) {
        if (KIND == 1) { forward_store_statistics(a, node, live, ck, lane, mean, var, rstd); }
        if (YMODE == kYBinarize && KIND != 2) { zero_packed_tail(a, ck, node, live, lane); }
        if (YMODE == kYBit && KIND != 2)      { zero_output_padding(a, ck, node, live, lane); }
        if (a.W_inline != nullptr && ck == 0 && live && lane < NN) {
            if (clamp_store)         { a.clamp_W[(size_t)node * NN + lane] = table_w; }
            if (a.C_out != nullptr)  { a.C_out[(size_t)node * NN + lane] = table_c; }
            if (a.V_out != nullptr)  { a.V_out[(size_t)node * NN + lane] = corner; }
        }
    }
}

static_assert(FwdArgs{}.quad_passes < 0, "a call that says nothing takes another kernel than lut_forward_quads_kernel");
static_assert(kQuadFrames == 4 * kWave && kQuadMost == kWavesPerBlk * kQuadFrames, "four frames per lane, a workgroup per node");
// Up to kQuadMost frames: a.node_waves wavefronts (1, 2 or 4) = one node, PASSES x 256 frames each, four consecutive ones per lane and pass (PASSES 0: up to 64 frames, one per lane).  All kinds that need the node's frames
// in one place: plain (0), batch-norm (1) with running statistics or those of the call (kStatInline), which the node's wavefronts add up and exchange in LDS.
// A frame's corner index is formed from the input words' four bits (spread to bytes by a multiplication) or from the fp32 frames, its corner value fetched once from the
// lane that holds it, and what follows is arithmetic on the value.  The fp32 frames of a small training pass may also be packed, by extra workgroups.
// Such a launch is a chain (wiring, inputs, index, value, sums, output), and the less a wavefront does in turn the shorter; with thousands of nodes its scalar
// instructions count (169 per wavefront with a division by the wavefronts of a node and products of signed numbers, 7372 plain nodes x 31 frames 4.80 us; 3.89 without).  Against a
// wavefront per node in steps of 64 frames, whose input masks were scalar loads, training calls on packed bits: 70 nodes x 1024 frames 5.0 -> 3.4 us, 1024 x 1024 5.0 -> 4.3, 6144 x 1024
// 7.8 -> 7.6, 700 x 1000 5.3 -> 3.9, 210 x 236 3.9 -> 3.1, 360 x 64 3.6 -> 3.0; inference 4000 x 1024 9.3 -> 5.3, 8000 x 1000 10.7 -> 7.6, 120 x 8 3.0 -> 2.5; plain 7372 x 31 4.5 -> 3.9.
template <int N, int XMODE, int YMODE, int KIND, int PASSES>
__global__ __launch_bounds__(kBlock) void lut_forward_quads_kernel(FwdArgs a)
{
    static_assert((XMODE == kXBit || XMODE == kXBinary) && (KIND == 0 || KIND == 1), "two-valued inputs, all frames of a node");
    // LANE: consecutive frames of a lane; PASSES 0: one pass of one frame per lane, up to 64 frames
    constexpr int NN = 1 << N, LANE = PASSES == 0 ? 1 : 4, P = PASSES == 0 ? 1 : PASSES;
    __shared__ float sums[kWavesPerBlk][2];
    int const B = a.tiles.count;
    if constexpr (XMODE == kXBinary && YMODE == kYBinarize && KIND == 1) {
        if ((int)blockIdx.x >= B) {
            int row, block;
            split_tile(blockIdx.x - B, a.pack.row_blocks, row, block);
            binarize_pack4_block(a.pack.x, a.pack.bits, a.frame_size, a.pack.x_stride, a.pack.y_stride, row, block);
            return;
        }
    }
    int const wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / kWave)), lane = threadIdx.x & (kWave - 1);
    // (a power of two: no division, which would head the chain; one wavefront in the forms that make several passes)
    int const nw = PASSES == 1 ? a.node_waves : 1, shift = PASSES == 1 ? __builtin_ctz((unsigned)nw) : 0, sub = wave & (nw - 1), slot = wave >> shift;
    int node = xcd_remap(blockIdx.x, B) * (kWavesPerBlk >> shift) + slot;
    bool const live = node < a.node_size;
    if (!live) {
        if (nw == 1) { return; }
        node = a.node_size - 1;                      // (with a barrier ahead: repeats the last node and stores nothing)
    }
    int const f0 = sub * kQuadFrames + LANE * lane;              // (PASSES != 1: one wavefront per node)

    int in[N];
#pragma unroll
    for (int k = 0; k < N; ++k) { in[k] = a.idx[node * N + k]; }
    int const i = lane & (NN - 1);
    float t = 0.0f, corner = 0.0f, c0 = 0.0f, table_c = 0.0f;
    bool const own_tables = a.W_inline != nullptr;
    if (own_tables) { t = a.W_inline[(size_t)node * NN + i]; }
    else {
        corner = a.V[(size_t)node * NN + i];
        if (KIND == 1) { c0 = a.C[(size_t)node * NN]; }
    }
    uint32_t const x_bytes = XMODE == kXBit ? (uint32_t)((a.frame_size + 31) >> 5) * 4u : quad_row_bytes(a.frame_size, a.x_stride >= ((a.frame_size + 3) & ~3));
    __amdgpu_buffer_rsrc_t rows[N];
#pragma unroll
    for (int k = 0; k < N; ++k) {                    // (row_descriptor takes the product of signed 64-bit numbers: twice the scalar instructions)
        rows[k] = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(reinterpret_cast<char const *>(a.x)) + (uint64_t)(uint32_t)in[k] * (uint32_t)a.x_stride * 4u,
                                                    0, (int)x_bytes, 0x00020000);
    }
    uint32_t w[XMODE == kXBit ? P : 1][N];
    std::conditional_t<LANE == 4, float4, float> x[XMODE == kXBit ? 1 : N];
    auto fetch = [&](int p) {                        // (past the row: zeros)
        int const f = f0 + p * kQuadFrames;
#pragma unroll
        for (int k = 0; k < N; ++k) {
            if constexpr (XMODE == kXBit) { w[p][k] = __builtin_amdgcn_raw_buffer_load_b32(rows[k], (uint32_t)(f >> 5) * 4u, 0, 0); }
            else if constexpr (LANE == 1) { x[k] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rows[k], (uint32_t)f * 4u, 0, 0)); }
            else if (a.x_stride >= ((a.frame_size + 3) & ~3)) { x[k] = load_quad<true>(rows[k], (uint32_t)f * 4u); }
            else { x[k] = load_quad<false>(rows[k], (uint32_t)f * 4u); }
        }
    };
    if constexpr (XMODE == kXBit) {
#pragma unroll
        for (int p = 0; p < P; ++p) { fetch(p); }
    }
    else { fetch(0); }

    // the node's tables (as in lut_forward_corner_kernel)
    bool clamp_store = false;
    float table_w = 0.0f;
    if (own_tables) {
        if (a.clamp_W != nullptr) {
            float const tc = fminf(a.clamp_hi, fmaxf(a.clamp_lo, t));
            clamp_store = (tc != t);
            t = tc;
        }
        table_w = t;
        if (a.lut_binarize) { t = (t > 0.5f) ? 1.0f : 0.0f; }
        table_c = centred_butterfly<N>(t, i);
        corner = corner_butterfly<N>(table_c, i, a.bias);
        c0 = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(table_c)));
    }

    float v[P][LANE];                                // the frames' corner values
    float s1 = 0.0f, s2 = 0.0f;
#pragma unroll
    for (int p = 0; p < P; ++p) {
        if (PASSES > 1 && p * kQuadFrames >= a.frame_size) { break; }              // wave-uniform
        uint32_t at[LANE];                           // corner indices, times 4
        if constexpr (LANE == 1) {
            uint32_t c = 0;
#pragma unroll
            for (int k = 0; k < N; ++k) {
                uint32_t bit;
                if constexpr (XMODE == kXBit) { bit = (w[0][k] >> (f0 & 31)) & 1u; }
                else                          { bit = x[k] > 0.5f ? 1u : 0u; }
                c |= bit << k;
            }
            at[0] = c << 2;
        }
        else if constexpr (XMODE == kXBit) {
            uint32_t quad = 0;
#pragma unroll
            for (int k = 0; k < N; ++k) { quad |= ((((w[p][k] >> (f0 & 31)) & 15u) * 0x00204081u) & 0x01010101u) << (k + 2); }
#pragma unroll
            for (int j = 0; j < 4; ++j) { at[j] = (quad >> (8 * j)) & 0xffu; }
        }
        else {
            if (p > 0) { fetch(p); }
#pragma unroll
            for (int j = 0; j < 4; ++j) { at[j] = 0; }
#pragma unroll
            for (int k = N - 1; k >= 0; --k) {
                at[0] = 2 * at[0] + (x[k].x > 0.5f ? 1 : 0); at[1] = 2 * at[1] + (x[k].y > 0.5f ? 1 : 0);
                at[2] = 2 * at[2] + (x[k].z > 0.5f ? 1 : 0); at[3] = 2 * at[3] + (x[k].w > 0.5f ? 1 : 0);
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) { at[j] <<= 2; }
        }
#pragma unroll
        for (int j = 0; j < LANE; ++j) { v[p][j] = __int_as_float(__builtin_amdgcn_ds_bpermute((int)at[j], __float_as_int(corner))); }
        if (KIND == 1 && a.stat_mode == kStatInline) {
#pragma unroll
            for (int j = 0; j < LANE; ++j) {
                float const d = (f0 + p * kQuadFrames + j < a.frame_size) ? v[p][j] - c0 : 0.0f;
                s1 += d;
                s2 = __builtin_fmaf(d, d, s2);
            }
        }
    }

    float mean = 0.0f, var = 0.0f, rstd = 1.0f;
    if (KIND == 1) {
        if (a.stat_mode == kStatInline) {
            s1 = wave_sum(s1);
            s2 = wave_sum(s2);
            if (nw > 1) {
                if (lane == 0) { sums[wave][0] = s1; sums[wave][1] = s2; }
                __syncthreads();
                s1 = 0.0f; s2 = 0.0f;
                for (int k = 0; k < nw; ++k) { s1 += sums[slot * nw + k][0]; s2 += sums[slot * nw + k][1]; }
            }
            batch_statistics(s1, s2, c0, a.frame_size, mean, var, rstd);
        }
        else { forward_statistics(a, node, lane, c0, mean, var, rstd); }
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
        int const f = f0 + p * kQuadFrames, frames = a.frame_size - f;              // frames: how many of the lane's four there are, and more
        if (PASSES > 1 && p * kQuadFrames >= a.frame_size) { break; }
        uint32_t m = 0;                              // the lane's bits of the packed output
#pragma unroll
        for (int j = 0; j < LANE; ++j) {
            float y = (KIND == 1) ? batch_norm_output(v[p][j], mean, rstd, a.gamma, a.beta) : v[p][j];
            if (YMODE == kYClamp) { v[p][j] = __builtin_amdgcn_fmed3f(y, 0.0f, 1.0f); }
            else {
                m |= (y > 0.5f && j < frames) ? 1u << j : 0u;
                v[p][j] = (y > 0.5f) ? 1.0f : 0.0f;
            }
        }
        if (live && frames > 0 && YMODE != kYBit) {
            float *const row = reinterpret_cast<float *>(a.y) + (size_t)node * a.y_stride + f;
            if constexpr (LANE == 1) { __builtin_nontemporal_store(v[p][0], row); }
            else if (a.y_quads && frames >= 4) {
                typedef float f32x4 __attribute__((ext_vector_type(4)));
                f32x4 const q = {v[p][0], v[p][1], v[p][2], v[p][3]};
                __builtin_nontemporal_store(q, reinterpret_cast<f32x4 *>(row));
            }
            else {
#pragma unroll
                for (int j = 0; j < 4; ++j) { if (j < frames) { row[j] = v[p][j]; } }
            }
        }
        if (YMODE == kYBit || (YMODE == kYBinarize && a.y_bits != nullptr)) {       // a word of 32 / LANE lanes
            constexpr int kWordLanes = 32 / LANE;
            if constexpr (LANE == 1) {
                uint64_t const all = __ballot(m != 0);
                m = (lane & 32) ? (uint32_t)(all >> 32) : (uint32_t)all;
            }
            else {
                m = quad_word(m, lane);
            }
            if (live && frames > 0 && (lane & (kWordLanes - 1)) == 0) {
                if (YMODE == kYBit) { reinterpret_cast<uint32_t *>(a.y)[(size_t)node * a.y_stride + (f >> 5)] = m; }
                else                { a.y_bits[(size_t)node * a.y_bits_stride + (f >> 5)] = m; }
            }
        }
    }

    if (sub != 0) { return; }
    if (KIND == 1) { forward_store_statistics(a, node, live, 0, lane, mean, var, rstd); }
    if (YMODE == kYBinarize) { zero_packed_tail(a, 0, node, live, lane); }
    if (YMODE == kYBit)      { zero_output_padding(a, 0, node, live, lane); }
    if (own_tables && live && lane < NN) {
        if (clamp_store)         { a.clamp_W[(size_t)node * NN + lane] = table_w; }
        if (a.C_out != nullptr)  { a.C_out[(size_t)node * NN + lane] = table_c; }
        if (a.V_out != nullptr)  { a.V_out[(size_t)node * NN + lane] = corner; }
    }
}

}  // namespace bbhip
