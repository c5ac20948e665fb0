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

// One wavefront = one node x one unit of frames in blocks of 2048 (kinds 0, 1, 2 as in lut_forward_kernel), or, for a batch-norm training pass
// in one launch (kStatInline), a.node_waves wavefronts = one node and all its frames.  A lane loads the words of 32 frames of each input and turns
// them into corner indices (corner_bytes: two instructions per frame and lane where the scalar lane masks of lut_forward_corner_kernel take
// N + 2), times 4, so that a byte is an offset into a table in LDS: a wavefront's 64 random reads of it take 4 clocks, a ds_bpermute 7.
//   statistics  every lane sums V - C0 and its square over its own 32 frames;
//   output      the index bytes go through LDS to the lanes that hold four consecutive frames each (16-byte stores of y; the packed copy collects
//               its words over a block and leaves by one store), packed output is assembled by the lane that formed the indices.
// In one launch the indices of all frames stay in LDS between the two, so nothing is gathered or formed twice, and the wavefronts of a node
// exchange their two sums there.  The kernel is bound by the fp32 output where there is one, else by its chain of latencies (wiring, words, tables).
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
    int const f_begin = ck * a.chunk, f_end = min(f_begin + a.chunk, a.frame_size);
    int const blocks = (f_end - f_begin + kByteBlock - 1) / kByteBlock;
    uint32_t *const bytes = lds + waves * (2 * kWave + 2) + (fused ? slot * blocks : wave) * kBlockWords;

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
                m <<= 4 * (lane & 7);
                m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0xB1, 0xf, 0xf, true);          // quad_perm [1, 0, 3, 2]
                m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x4E, 0xf, 0xf, true);          // quad_perm [2, 3, 0, 1]
                m |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, 0x141, 0xf, 0xf, true);         // row_half_mirror
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
            if (fused) { keep(quad, bytes + b * kBlockWords); }
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

}  // namespace bbhip
