// Rules by which the host side divides work into launches, apart from the code that launches: plain C++, checked on the CPU by tests/cpp/test_host.cpp.
#pragma once

namespace bbhip {

inline int ceil_div(int a, int b) { return a / b + (a % b != 0); }      // (no sum that could leave the range)

// What a launch of the per-corner sums costs in slabs of `frames` frames, in frames' worth of a workgroup: ceil(workgroups / 512) rounds of resident workgroups
// (two per compute unit: 64 KB of bins each), a unit costs its frames plus about 1024 frames' worth of set-up and closing sums, and more than one slab per
// node needs the fold launch (about 2700 frames' worth on top, and 2.5 for each node: a workgroup each).  1000 frames' worth is about 1.25 us.  Several slabs
// against one, promised with 3072 on top for any node count and measured: 64 inputs x 2666 nodes x 8646 frames, five per node, 0.2 us less and 4.2 more (58.3 us in
// one slab), 2795 x 10066 0.8 less and 4.5 more (79.3), 1420 x 31338 3.0 less and 3.6 more (117.7); 24 x 4223 0.2 and 0.6 less (14.7).
inline long long corner_slab_cost(int frame_size, int tile_count, long long frames)
{
    long long const slabs = (frame_size + frames - 1) / frames, rounds = (slabs * tile_count + 511) / 512;
    return rounds * ((frames < frame_size ? frames : frame_size) + 1024) + (slabs > 1 ? 2700 + 10LL * tile_count : 0);
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

// Wavefronts that walk an input's list in the one-launch backward pass of a small layer on two-valued inputs: 1, or 4 or 16 that share it, or 0: two
// launches.  What its wavefronts walk one after another must be short: an item costs 0.45 us, 0.65 where the wavefront also derives the node's corner
// values (no prepared tables); and what they do for every connection (the sums through the statistics) little in all.  The rule does not ask for prepared
// tables: a hint changes no bit of a result, and these forms add in different orders.  Device time of the backward call of a batch-norm layer of six
// inputs per node, with prepared tables / without, in microseconds; fan: the longest list.
//   up to 256 frames                         4 wavefronts    16              two launches
//   784 inputs x 1024 nodes (fan 19)         5.8 /  6.9       -              7.8 /  8.4
//   26 x 104 (fan 35)                        6.7 /  8.2      5.3 /  6.2      7.4 /  7.8
//   347 x 1643 (fan 44)                      8.3 / 10.5      9.2 / 11.3      9.1 /  9.7
//   207 x 1495 (fan 63)                     10.3 / 13.1      8.9 / 10.3      8.7 /  9.5
//   645 x 4947 (fan 69)                     14.0 / 18.4     18.0 / 22.3     13.9 / 15.9
//   650 x 4818, four inputs (fan 49)        10.1 / 11.8     13.9 / 15.8     13.4 / 14.3
//   784 x 6144, plain (fan 71)              12.1 / 17.2     14.0 / 16.9     15.9 / 18.3
//   149 x 2247, three inputs (fan 66)        9.8 / 11.2      6.5 /  7.4      9.4 /  9.7
//   47 x 469 (fan 76)                       11.7 / 14.9      7.7 /  9.7      8.6 /  9.0 (one launch less for the host)
//   34 x 598 (fan 129)                      18.4 / 23.9     10.3 / 13.7      9.7 / 10.3
//   512 frames: 300 x 300 (fan 15) 6.2 / 6.9 with four, 10.3 / 10.8 in two; 784 x 1024 (fan 19) 8.5 / 9.6 and 9.1 / 9.7
//   1024 frames: 360 x 70 (fan 6) 4.5 / 4.8 and 7.3 / 7.6, 500 x 500 (fan 16) 8.7 / 9.3 and 9.6 / 10.0
// Many inputs with little to walk: a wavefront each.  6144 x 1024 (256 frames, fan 6) 7.1 / 8.8, shared 9.2 / 10.0, two launches 8.4 / 8.9.
constexpr int kCornerSmallShare = 20;           // items of a list that a wavefront takes at most
inline int corner_small_waves(int n, bool batch_norm, int frame_size, int input_node_size, int node_size, int max_fan)
{
    int const items = ceil_div(max_fan, 4);
    long long const links = (long long)node_size * n;
    if (frame_size > 256) {
        int const passes = frame_size <= 512 ? 2 : 4;
        return (input_node_size <= 1536 && items <= 16 / passes && links * passes <= 12000) ? 4 : 0;
    }
    if (input_node_size > 2048) { return max_fan <= 8 ? 1 : 0; }
    if (items > kCornerSmallShare || links > 40000) { return 0; }
    // (two launches take longer as there is more to do in all)
    if (input_node_size <= (batch_norm && n >= 5 ? 128 : 256)) { return items <= 8 + links / 6000 ? 4 : 16; }
    return items <= (!batch_norm ? 13 : n >= 5 ? 9 : 12) + links / 6000 ? 4 : 0;
}

// Passes of 256 frames, 1, 2 or 4, of a wavefront of lut_dx_table_kernel.  A term's table and its loads are shared by the passes, so more of them where the rows of
// dy and of indices that they gather from (5 bytes per node and frame) stay in an XCD's L2, and where the launch does not fall short of workgroups: a
// workgroup is four inputs, or one whose list its wavefronts share (27 inputs x 87 nodes x 94500 frames in passes of 256 / 512 / 1024 frames, convolutional
// block with 10000 / 5000 / 2500 workgroups: 125 / 117 / 122 us; 27 x 216 x 230400 371 / 348 / 346).
// Two passes, training call whose inputs and buffers are other ones than those of the call before (four sets in turn; from one set, which the L2s hold in part, two passes look up to 12 % better), with
// one and with two: from 2000 groups of four inputs in passes of 256 frames, which leaves out what the last frames do not fill, lists of 4.5 items on average up to 1350 nodes, 1024 of two and three
// inputs: six inputs 605 x 1347 x 3349 32.5 and 30.7 us, 585 x 772 x 5509 34.3 and 30.1, 168 x 959 x 17363 78.7 and 73.2; five, 632 x 1175 x 5013 36.5 and 31.7, 750 x 1231 x 2879 29.1 and 26.2; four,
// 701 x 1067 x 3501 27.2 and 25.6, 910 x 1232 x 2723 26.7 and 25.3; three, 408 x 943 x 7051 31.0 and 28.6.  Shorter lists gain only where workgroups abound: six, 1336 x 804 x 1505 20.1 and 20.6, 2740 x
// 921 x 734 16.6 and 17.6, 1023 x 695 x 1921 20.1 and 20.8; four, 1341 x 902 x 1385 18.1 and 19.1, 1764 x 1151 x 1263 19.1 and 20.5, 3845 x 1301 x 687 17.0 and 17.9, 2328 x 1331 x 3232 (7566
// groups) 28.8 and 29.6; but six, 6144 x 1024 x 1024 (3072 groups in passes of 512) 19.3 and 18.6, 3664 x 1195 x 7782 (28396 in passes of 256) 57.9 and 52.8, five, 6653 x 1291 x 1828 (13312) 28.5 and 27.0.  Up
// to 512 nodes any list: 1391 x 128 x 1469, six, 16.8 and 16.5, 337 x 445 x 6515 30.0 and 27.3, 511 x 128 x 9917, two, 17.7 and 17.1, but 111 x 237 x 38759 31.3 and 32.2.  Fewer groups: six, 1418 x 705 x 1150 18.5 and 19.9, 1348 x 896 x
// 1164 19.7 and 21.0, 2754 x 1341 x 498 16.7 and 17.6; three inputs, 1708 x 1259 x 14639 74.2 and 73.1, two, 527 x 1189 x 15747 58.8 and 61.0.
// Tables of five and six inputs also up to 1600 nodes where wavefronts share the lists and two passes end in one round of the 2048 workgroups that fit: six, 457 x 1398 x 5546 41.6 and 39.0, 1206 x
// 1382 x 1813 27.9 and 25.4, 1000 x 1500 x 3000 34.1 and 30.8; five, 773 x 1482 x 3855 34.2 and 30.1; but lists of up to 15, six, 2354 x 1398 x 1030 23.6 and 24.6, five, 1529 x 1382 x 1275 21.2
// and 22.6, and 2048 workgroups and more, 1762 x 1542 x 2740, 32.7 and 35.1, five, 1833 x 1530 x 6448 47.2 and 48.9.
inline int dx_table_quads(int n, int input_node_size, int output_node_size, int frame_size, bool long_lists)
{
    auto const groups = [&](int q) { return (long long)ceil_div(frame_size, q * 256) * ceil_div(input_node_size, 4); };
    auto const shared = [&](int q) { return long_lists && (long long)ceil_div(frame_size, q * 256) * input_node_size >= 3072; };
    if (output_node_size <= 512 && (groups(4) >= 2048 || shared(4))) { return 4; }
    bool const many = output_node_size <= 512 ? groups(1) >= 2000 : output_node_size <= 1024 ? groups(2) >= 2048 : groups(1) >= 10000;
    bool const listed = groups(1) >= 2000 && 2LL * output_node_size * n >= 9LL * input_node_size;
    if (output_node_size <= (n >= 4 ? 1350 : 1024) && (many || listed || shared(2))) { return 2; }
    return (n >= 5 && output_node_size <= 1600 && frame_size > 1024 && long_lists && groups(2) >= 1000 && groups(2) <= 2048) ? 2 : 1;
}

// Whether the sixteen wavefronts that share an input's list in lut_dx_table_kernel take its items in turn (they then walk the nodes together, and rows that
// outgrow an L2 come from behind it once) or consecutive ones.  A launch of fewer workgroups than compute units leaves the L2s room; what counts there is that
// an item's list entry, row and index are requested one item ahead only, and consecutive entries of a long list share a cache line.  Backward call, plain,
// in turn and consecutive: 12 inputs x 3623 nodes x 297 frames (24 workgroups, lists of 1840) 57.2 and 48.1 us, 17 x 2078 x 1839 (136, 653) 28.1 and 24.2,
// 22 x 5774 x 1449 (132, 1645) 63.7 and 55.1; 12 x 707 x 108
// (12, 388) 13.9 and 14.4, 60 x 5776 x 3633 (900, 621) 77.9 and 103.0.  The longer items of
// batch-norm layers hide more: 14 x 2990 x 1129 (70, 1361) 57.8 and 53.2, 11 x 2343 x 127 (11, 897) 31.5 and 33.8, 35 x 5912 x 5652 (805) 103.7 and 151.3.
inline bool dx_items_in_turn(bool batch_norm, long long workgroups, int max_fan)
{
    if (workgroups >= 256) { return true; }
    return batch_norm ? workgroups < 64 || max_fan < 700 : max_fan < 400;
}

// How a wavefront of lut_corner_sums_kernel adds up a node's frames (see there): in blocks of 2048 whose next one is requested ahead, or all frames of one slab
// requested at once: 256, 512, 1024 (kSumsShort) or 2048 (kSumsBlock) of them.  Where a slab ends with its first block, the requests ahead and the
// registers that they take are for nothing.  Sums launch, in blocks and at once: 2932 inputs x 3358 nodes x 489 frames, three inputs, rows of 489:
// 11.2 and 8.2 us; 296 x 6754 x 747, two inputs, rows of 747: 15.6 and 11.1; 141 x 5121 x 82, two: 8.7 and 8.0; 126 x 4657 x 1981, four: 16.1 and
// 15.2; 307 x 3081 x 1140, five: 13.7 and 13.3; 67 x 5667 x 1696, five: 20.3 and 18.4; six inputs, 1638 x 5110 x 1045: 21.7 and 21.0, 111 x 5234 x 1928: 25.3
// and 24.8.
enum SumsForm : int { kSumsLong = 0, kSums256 = 1, kSums512 = 2, kSumsShort = 4, kSumsBlock = 8 };
constexpr int kShortSlab = 1024, kBlockSlab = 2048;
constexpr SumsForm corner_sums_form(int frame_size, int slab_count)
{
    return (slab_count > 1 || frame_size > kBlockSlab) ? kSumsLong : frame_size <= kShortSlab ? kSumsShort : kSumsBlock;
}

// Whether a workgroup of eight wavefronts sums a node's frames (lut_corner_sums_node_kernel) instead of slabs and a launch that folds them.  Up to 2048 frames
// for each wavefront, in one block, and up to a node per compute unit with five and six inputs, whose bins leave room for one workgroup, two with fewer.
// Backward call of 40 inputs in slabs and by workgroups: six per node, 12 nodes x 2300 frames 10.8 and 9.5 us, 80 x 14000 15.9 and 13.4, 256 x 4500 16.6 and 13.6,
// 256 x 16384 22.4 and 21.6; four, 30 x 10000 11.6 and 9.2, 512 x 6000 17.2 and 15.9.  Beyond: six, 80 x 24000 18.6 and 17.7, but 40 x 24000 14.9 and 15.1, 30 x
// 100000 20.5 and 29.4; 300 x 4500 17.0 and 18.7; five, 300 x 4000 14.4 and 16.0; up to 2048 frames, one slab, 100 x 1500 9.9 and 10.2.
constexpr int kNodeSumsWaves = 8;
inline bool node_sums(int n, int node_size, int frame_size)
{
    return frame_size > kBlockSlab && frame_size <= kNodeSumsWaves * kBlockSlab && node_size <= (n > 4 ? 256 : 512);
}

// Whether dx over two-valued inputs is formed node by node, with the sums of all inputs in registers (lut_dx_few_inputs_kernel), instead of input by input from
// kept corner indices.  It reads dy once where the other reads it once per connection, and asks for frames for every compute unit (a workgroup
// takes 512) and for nodes enough to pay for its set-up and closing sums.  Backward call, input by input and node by node, batch-norm unless said otherwise:
// 27 inputs x 216 nodes x 230400 frames 117 and 90 us, x 115200 64.7 and 53.6, x 80000 50.2 and 49.1, x 50000 40.2 and 44.5; 9 x 72 x 230400 48.6 and 38.5;
// 6 x 216 x 262144 142 and 88; four inputs per node, 9 x 100 x 230400 48.8 and 40.2; two, 9 x 216 x 100000 41.7 and 35.6.  Few connections in all, or for each
// input: 27 x 24 x 230400 25.2 and 25.7, 18 x 24 x 400000 34.6 and 35.2, 12 x 16 x 180000, two per node, plain, 13.9 and 16.4; but 27 x 36 x 700000 68.6 and 63.9.
// 512 workgroups are resident, so that 262145 frames begin a second round that is nearly empty: 27 x 216 x 262144 141 and 90, x 262656 141 and 109; with few connections
// the two are even there, 27 x 44 x 263000 39.6 and 39.7, 27 x 52 x 263000 43.3 and 44.1, 27 x 36 x 180000 28.7 and 29.2, the widest of 85 shapes on that side.  More nodes: 27 x 1000 x 97793 307 and
// 192, 27 x 1600 x 150000 777 and 467; from about 2000 nodes on, whose wiring leaves a compute unit's LDS room for one workgroup, 27 x 2100 x 150000 1098 and 735, 27 x 4000 x 97793
// 1484 and 711; four inputs, 9 x 4000 x 120000, 1409 and 699.
constexpr int kFewInputs = 28, kFewInputNodes = 4096;
inline bool few_inputs_dx(int n, int input_node_size, int node_size, int frame_size)
{
    long long const links = (long long)node_size * n;
    return input_node_size <= kFewInputs && node_size <= kFewInputNodes && frame_size > 191 * 512 && links >= 200 && links >= 8LL * input_node_size;
}

// The shortest list that the wavefronts of a workgroup share in lut_dx_kernel (real-valued inputs), in a launch that would otherwise have `groups` workgroups of
// four inputs each.  Its terms take long enough for lists from eight items where the launch falls short of wavefronts: training call of batch-norm
// layers, six inputs per node, shared and not, 69 inputs x 66 nodes x 906 frames (list of 13) 10.4 and 15.0 us, 1500 x 800 x 700 (14) 20.6 and 23.0, 1024 x 1024 x
// 1000 (14) 23.8 and 26.1.  Many frames of few inputs have wavefronts enough, whose rows all lie close: 16 x 26 x 29705 (14) 20.1 and 16.8, 40 x 63 x
// 15921 (9) 11.2 and 9.8, 116 x 321 x 8625 (12) 25.8 and 23.3, but 16 x 26 x 14420 (13) 12.7 and 14.4.  Nor do layers of more than 5000 rows gain, which
// have passes of 128 frames: 3383 x 3689 x 235 (14) 19.6 and 18.4, 3817 x 6000 x 253 (15) 21.3 and 19.9.
constexpr int kDxWideRows = 5000;       // (dx_wide_passes)
inline int dx_shortest_shared_list(int input_node_size, int output_node_size, int frame_size, long long groups)
{
    if (groups >= 2048 || (long long)input_node_size + output_node_size > kDxWideRows) { return 16; }
    long long const passes = ceil_div(frame_size, 256);
    return (passes <= 32 || passes * input_node_size < 1000) ? 8 : 16;
}

// Real-valued inputs: passes of 256 frames, four consecutive ones per lane (lut_dx_kernel, WIDE), where a term's coefficients and addresses serve twice the
// frames of the usual 128 and its rows come by a quarter of the loads.  All rows of x and dy that a window touches, 1 KB each, should be what an
// L2 holds (training steps with and without: 1024 inputs + 2000 nodes x 4000 frames 106 and 112 us, 300 + 4000 x 4000 179 and 186, 500 + 1000 x 4000
// with batch-norm 67 and 72.5, 1024 + 1024 x 1000 31.8 and 35.0; 3000 + 3000 x 6000 239 either way, 4096 + 4096 x 8192 498 and 457), and the launch should
// have workgroups enough.  Over 400 shapes of two to six inputs, drawn: where lists are shared (a workgroup per input and pass) passes of 256 frames take 1.04
// times as long below 700 workgroups, 0.95 to 1.00 from 700 to 1400, 0.95 to 2000, 0.93 to 4000 and 0.84 to 0.90 above; else (a workgroup per four inputs)
// 1.03 below 512 workgroups, 1.02 to 1024, 0.97 to 2048 and 0.92 to 0.98 above; few items make it worse (1500 + 800 x 700, lists of three, 29.8 and 29.2).
inline bool dx_wide_passes(int input_node_size, int output_node_size, int frame_size, int max_fan, long long links)
{
    if ((long long)input_node_size + output_node_size > kDxWideRows) { return false; }
    long long const passes = ceil_div(frame_size, 256), groups = passes * ceil_div(input_node_size, 4);
    if (max_fan >= dx_shortest_shared_list(input_node_size, output_node_size, frame_size, groups)) { return passes * input_node_size >= 1400; }
    return groups >= 1024 && passes * links >= 20480;
}

// Order of the workgroups of the Im2Col kernels.  Neighbouring pieces of a row share cache lines and belong in one L2: either the workgroups of an XCD are
// consecutive ones, pieces first, or, where the tiles of 64 frames are a multiple of the eight XCDs, frames come first and every XCD has frames of its own, with
// all pieces and all rows, so that its L2 also keeps the input for the next tap of the window.  Forward, pieces and frames first: 3 x 32 x 32 x 1024 frames, 3 x 3,
// 31.5 and 27.5 us, 6 x 23 x 36 x 1024 48.7 and 42.0, 43 x 39 x 23 x 1521, 1 x 1, 108.8 and 92.5; 32 x 32 x 32 x 64 20.4 and 23.0 (one tile), 216 x 30 x 30 x 256, 1 x 1,
// 78 and 97 (four).
inline bool im2col_frames_first(int f_tiles, int tile_frames) { return tile_frames == 64 && f_tiles % 8 == 0; }

// Passes of 256 frames that a wavefront of lut_forward_quads_kernel makes: one, the node's passes side by side (they wait for each other where they exchange sums), or
// all, one after another, where nodes alone fill the device.  Side by side and one after another, 784 inputs: batch-norm training call on fp32 frames 700 nodes x 1000 frames
// 4.89 and 5.93 us, 1024 x 1024 5.18 and 5.73, 1200 x 1024 6.99 and 7.11; 1500 x 600 6.46 and 5.60, 3000 x 400 7.57 and 7.13, 4000 x 300 8.81 and 7.98, 6144 x 1024 15.0 and 10.9 (packed
// frames 700 x 1000 4.03 and 4.12, 1024 x 1024 4.21 and 3.96, 1500 x 600 5.19 and 4.34, packed inference 1024 x 1024 3.41 and 3.56).  0: up to 64 frames, one per lane.
// Each count has a form of its own, whose inputs are all requested at once: two passes in the form for two and in that for four, packed training call 1100 x 512 3.81 and 3.93 us,
// 3000 x 300 4.35 and 4.68, inference 1500 x 512 3.27 and 3.42, four inputs per node, 6144 x 400, training call 5.19 and 5.23; up to 64 frames in the form for one frame per lane and
// in that for one pass, 360 x 64 2.89 and 3.06, fp32 frames 2.93 and 3.39, 7372 x 31 5.68 and 6.22, fp32 5.75 and 6.99.
constexpr int kQuadFrames = 256, kQuadMost = 1024;               // frames of a pass, most frames of a node there
inline int forward_quad_passes(int node_size, int frame_size) { return frame_size <= 64 ? 0 : (node_size <= 1024 || frame_size <= kQuadFrames) ? 1 : frame_size <= 2 * kQuadFrames ? 2 : 4; }

// Blocks of 2048 frames whose fp32 output a workgroup of lut_forward_bytes_kernel writes in a one-launch training pass: all of its nodes', or, where nodes are few, a part,
// with the statistics of all frames in each of the workgroups that share a node (they cost a third of the output, and an exchange would be a launch).  Up to 256
// workgroups, a node each, 1024 threads where rows are long: 512 of those are two rounds.  Training call, whole nodes and parts: 72 nodes x 33800 frames 10.1 and 8.2 us
// (13.2 in parts for 512 workgroups), 24 x 33800 9.4 and 6.9, 12 x 49000 10.4 and 7.1, 24 x 12000 7.1 and 5.5, 36 x 4000 6.9 and 6.0, 5 x 20000 7.7 and 5.9.  Packed
// output is too little to share: 24 x 33800 6.75 and 6.6, 70 x 3500 5.0 and 5.2.
inline int forward_out_blocks(int tile_count, int node_waves, int blocks)
{
    int const parts = 256 / tile_count;
    return (node_waves < 2 || parts < 2) ? blocks : parts < blocks ? ceil_div(blocks, parts) : 1;
}

// Packed rows whose padding the caller wants as 0: the wavefront of a row's last unit writes that much of it, an iteration per 64 words, and what a longer pitch
// leaves is a launch of its own (zero_row_ends_kernel).  BinaryLut5, rows of 1000 frames, by the wavefronts and by the launch: 1000 rows of 2080 words 3.8 and
// 5.7 us, 10000 words 8.7 and 11.3; 4 rows of 100000 words 42.1 and 5.8, 64 of 1000000 397 and 36.
constexpr int kPaddingWords = 4096;
inline int packed_padding_end(int words, int stride) { return (long long)words + kPaddingWords < stride ? words + kPaddingWords : stride; }

// Words per unit of the BinaryLut kernels: 128 (see there), or 64 where the launch still has fewer than 512 workgroups then, that is compute units to spare, and a
// unit's second step only takes time.  3 inputs per node, 30 nodes x 93 words 2.24 -> 2.00 us, 239 nodes x 261 words, five, 2.26 -> 2.13, 183 x 688, three, 2.21 -> 2.09
// (506 workgroups); 29 x 6663, two, 2.19 and 2.29 (840), 4708 x 69, three, 3.19 and 3.84 (2354).
inline int binary_unit_words(int words, int node_size)
{
    return (long long)ceil_div(words, 64) * ceil_div(node_size, 4) < 512 ? 64 : 128;
}

// Whether a thread of the pooling kernels takes four frames (rows start on 16 bytes): not for rows of less than 16 frames that are no whole groups of four, where
// every wavefront would do the last group's frames one by one beside the whole groups.  One frame and four per thread, forward / backward: 2280 rows of 3 frames
// 2.3 / 2.9 and 3.5 / 4.8 us, 840 of 11 2.2 / 2.7 and 2.7 / 3.5, 31995 of 11 3.6 / 6.0 and 3.9 / 7.1; many rows of more frames gain from four, 27183 of 18
// 4.0 / 6.9 and 3.6 / 6.9, the more so the longer they are.
inline bool pool_four_frames(int frame_size) { return frame_size >= 16 || frame_size % 4 == 0; }

// Whether the classifier tail runs with a row of 16 lanes per frame (classifier_tail_small_kernel): where there are as many inputs as connections (the wiring policies then
// give every input to one node, which that form writes at once), channels fill half a row or more, and frames are few, of which it has four to a wavefront and
// 16 bytes of a row to a cache line.  70 -> 10 nodes, by a wavefront per channel and by a row of lanes: 64 frames 6.35 and 3.66 us, 1024 6.64 and 3.99, 2048 6.66 and 4.41, 4000
// 6.75 and 5.44, 6000 6.89 and 6.90, 16384 8.37 and 13.7, 65536 20.6 and 44.8; 192 -> 16 nodes, 1024 frames, 12.4 and 6.15.  A table of the caller's own whose nodes
// share inputs: 70 -> 10 nodes, 64 frames 6.16 and 5.19, 1024 6.40 and 5.51, 2000 6.47 and 5.95, 4000 6.56 and 6.74, and where a node takes an input twice 6.10 and 5.41, 6.32
// and 5.89, 6.38 and 6.27, 6.48 and 7.21; 208 -> 16, 4000 frames, 14.7 and 12.8.  Other counts of inputs and fewer channels stay with the wider
// form, though this one would serve them too (60 inputs, 1024 frames, 6.35 and 4.98, 80 -> 5 nodes x 2000 frames 6.39 and 5.79, 40 -> 4 x 1000 4.88 and 4.65).
constexpr int kTailInputs = 16;                 // most inputs of a node there
inline bool tail_small(int n, int input_node_size, int ch_size, int frame_stride)
{
    return n <= kTailInputs && ch_size >= 8 && input_node_size == ch_size * n && frame_stride <= 4096;
}

// Rows that share a workgroup of 256 threads in the pooling kernels, `lanes` threads each.  A row has a workgroup of its own where sharing saves no more than
// one or two idle wavefronts of it and there are workgroups for every compute unit either way: up to 256 rows (120 rows x 203 frames, backward, 3.31 us shared and
// 3.08 not), and where whole wavefronts stream through memory (48600 x 256 forward 35.4 and 33.3, backward 82.1 and 79.7; 46740 x 512 backward 151.8 and
// 146.4).  7056 x 256 4.8 and 5.8, backward 10.3 and 11.5; 90000 x 128 32.4 and 40.8, 29070 x 280 backward 49.8 and 61.3.
inline int pool_shared_rows(int lanes, long long nodes)
{
    bool const full = lanes % 64 == 0 || lanes % 64 >= 48;              // the last wavefront of a row
    return (lanes > 32 && (nodes <= 256 || (nodes > 16384 && full))) ? 1 : 256 / lanes;
}

}  // namespace bbhip
