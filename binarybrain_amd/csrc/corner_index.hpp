// Corner indices of two-valued inputs, 32 frames per lane at a time, and rows read four frames per lane: shared by the forward and the backward kernels.
#pragma once

#include "lut_math.hpp"

namespace bbhip {

// Words of N inputs (32 frames) -> the 32 corner indices, times 2^SHIFT, a byte each in frame order: quad[i] holds the frames 4 i .. 4 i + 3.
// Eight rows of four bytes are transposed bit by bit (rows a power of two apart exchange bit fields: three rounds), which leaves frame
// 8 c + j in byte c of row j, then byte by byte: about two instructions per frame and lane where building an index bit by bit takes N.
template <int N, int SHIFT = 0>
__device__ __forceinline__ void corner_bytes(uint32_t const (&w)[N], uint32_t (&quad)[8])
{
    static_assert(N + SHIFT <= 8, "an index is a byte");
    uint32_t r[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) { r[k] = (k >= SHIFT && k - SHIFT < N) ? w[(k >= SHIFT && k - SHIFT < N) ? k - SHIFT : 0] : 0u; }
    auto exchange = [&](int i, int j, int s, uint32_t low) {
        uint32_t const a = r[i], b = r[j];
        r[i] = (a & low) | ((b << s) & ~low);
        r[j] = ((a >> s) & low) | (b & ~low);
    };
#pragma unroll
    for (int k = 0; k < 4; ++k) { exchange(k, k + 4, 4, 0x0f0f0f0fu); }
#pragma unroll
    for (int k = 0; k < 8; k += 4) { exchange(k, k + 2, 2, 0x33333333u); exchange(k + 1, k + 3, 2, 0x33333333u); }
#pragma unroll
    for (int k = 0; k < 8; k += 2) { exchange(k, k + 1, 1, 0x55555555u); }
#pragma unroll
    for (int h = 0; h < 2; ++h) {           // rows 4 h .. 4 h + 3: byte c of row j -> byte j of quad 2 c + h
        uint32_t const *q = r + 4 * h;
        uint32_t const p0 = __builtin_amdgcn_perm(q[1], q[0], 0x05010400u), p1 = __builtin_amdgcn_perm(q[3], q[2], 0x05010400u);      // bytes 0, 1 of row pairs
        uint32_t const p2 = __builtin_amdgcn_perm(q[1], q[0], 0x07030602u), p3 = __builtin_amdgcn_perm(q[3], q[2], 0x07030602u);      // bytes 2, 3
        quad[0 + h] = __builtin_amdgcn_perm(p1, p0, 0x05040100u);
        quad[2 + h] = __builtin_amdgcn_perm(p1, p0, 0x07060302u);
        quad[4 + h] = __builtin_amdgcn_perm(p3, p2, 0x05040100u);
        quad[6 + h] = __builtin_amdgcn_perm(p3, p2, 0x07060302u);
    }
}

// orders a wavefront's own accesses to LDS
__device__ __forceinline__ void wave_fence(void)
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// four consecutive frames of a row from byte offset off; QUADS: the row holds whole groups of four
template <bool QUADS>
__device__ __forceinline__ float4 load_quad(__amdgpu_buffer_rsrc_t r, uint32_t off, uint32_t row_off = 0)
{
    if constexpr (QUADS) {
        auto const q = __builtin_amdgcn_raw_buffer_load_b128(r, off, row_off, 0);
        return make_float4(__uint_as_float(q[0]), __uint_as_float(q[1]), __uint_as_float(q[2]), __uint_as_float(q[3]));
    }
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) { v[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off + 4 * j, row_off, 0)); }
    return make_float4(v[0], v[1], v[2], v[3]);
}

// valid bytes of a row for load_quad: whole groups of four where the row holds them (frames past the last read 0 or the row's padding)
__device__ __forceinline__ uint32_t quad_row_bytes(int frame_size, bool quads)
{
    return (uint32_t)(quads ? (frame_size + 3) & ~3 : frame_size) * 4u;
}

}  // namespace bbhip
