// Rules by which the host side divides work into launches, apart from the code that launches: plain C++, checked on the CPU by tests/cpp/test_host.cpp.
#pragma once

namespace bbhip {

inline int ceil_div(int a, int b) { return a / b + (a % b != 0); }      // (no sum that could leave the range)

// What a launch of the per-corner sums costs in slabs of `frames` frames, in frames' worth of a workgroup: ceil(workgroups / 512) rounds of resident workgroups
// (two per compute unit: 64 KB of bins each), a unit costs its frames plus about 1024 frames' worth of set-up and closing sums, and more than one slab per
// node needs the fold launch (about 3072 frames' worth on top).
inline long long corner_slab_cost(int frame_size, int tile_count, long long frames)
{
    long long const slabs = (frame_size + frames - 1) / frames, rounds = (slabs * tile_count + 511) / 512;
    return rounds * ((frames < frame_size ? frames : frame_size) + 1024) + (slabs > 1 ? 3072 : 0);
}

// Frames per unit of the per-corner sums, in at most max_slabs slabs: the cheapest of one slab, the equal slabs that fill one to four rounds, and
// powers of two.  Equal slabs serve few nodes, where a power of two leaves a round short or a slab nearly empty (216 nodes x 230400 frames in 9 slabs
// instead of 8, convolutional block 345.8 -> 340.6 us; 87 x 94500 in 22 instead of 93, 120.4 -> 114.3).  Layers of many nodes have few
// such slabs (2100 nodes two or three, 4200 nodes none), and over many frames more rounds of shorter slabs leave less of the device idle in the last one:
// backward call of 512 inputs x 4200 nodes x 65536 frames 1061 us in one slab and 1012 in eight, 4200 x 4200 x 32768 711 and 693, 512 x 4200 x 230400
// 3789 and 3668; 512 x 2100 x 230400 1651 in three slabs, 1628 in 29.
inline int corner_slab_frames(int frame_size, int tile_count, long long max_slabs)
{
    long long const whole = (long long)ceil_div(frame_size, 256) * 256;
    long long best = whole;
    auto consider = [&](long long frames) {
        if (frames >= whole || (frame_size + frames - 1) / frames > max_slabs) { return; }
        if (corner_slab_cost(frame_size, tile_count, frames) < corner_slab_cost(frame_size, tile_count, best)) { best = frames; }
    };
    for (int rounds = 1; rounds <= 4; ++rounds) {
        int const slabs = rounds * 512 / tile_count;
        if (slabs < 2) { continue; }
        int const frames = ceil_div(ceil_div(frame_size, slabs), 256) * 256;
        consider(frames < 1024 ? 1024 : frames);
    }
    for (long long frames = 1024; frames < frame_size; frames *= 2) { consider(frames); }
    return (int)best;
}

}  // namespace bbhip
