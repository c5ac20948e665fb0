// CPU test of the host-side plumbing (no device needed): frame-buffer layout and bit packing, tensors, the connection
// table and its reverse table against the oracle, command handling, and the refusal to run without a device.
#include <algorithm>
#include <cstdio>
#include <map>
#include <set>
#include <sstream>
#include <vector>

#include "bb/StochasticLutN.h"
#include "bb/DifferentiableLutN.h"
#include "bb/BinaryLutN.h"
#include "bb/ObjectLoader.h"
#include "bb/BinaryModulation.h"
#include "bb/DifferentiableLutDiscreteN.h"
#include "bb/MaxPooling.h"
#include "bb/UpSampling.h"
#include "bb/Shuffle.h"
#include "../../binarybrain_amd/csrc/launch_rules.hpp"
#include "../../binarybrain_amd/csrc/tile_divisor.hpp"

extern "C" int oracle_ReverseTable(int n, std::int32_t const *idx, int input_node_size, int output_node_size, std::int32_t *rev, int rev_cap);

static int g_fail = 0;
#define CHECK(cond) do { if (!(cond)) { ++g_fail; std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond); } } while (0)

int main(void)
{
    bb::Manager::SetHostOnly(true);
    CHECK(!bb::Manager::IsDeviceAvailable());

    // frame buffer: node-major rows, stride a 256-byte multiple and never a 2 KiB multiple
    {
        bb::FrameBuffer buf(100, {3, 5}, BB_TYPE_FP32, true);
        CHECK(buf.GetNodeSize() == 15 && buf.GetFrameSize() == 100 && buf.GetFrameStride() == 512);
        CHECK(bb::FrameBuffer::CalcFrameStride(BB_TYPE_FP32, 8192) == 32768 + 512);
        CHECK(bb::FrameBuffer::CalcFrameStride(BB_TYPE_BIT, 262144) == 32768 + 384);
        CHECK(bb::FrameBuffer::CalcFrameStride(BB_TYPE_BIT, 1) == 256);
        buf.SetFP32(99, 14, 3.5f);
        buf.SetFP32(0, 0, -1.0f);
        CHECK(buf.GetFP32(99, 14) == 3.5f && buf.GetFP32(0, 0) == -1.0f);
        auto p = buf.LockConst<float>();
        CHECK(p.GetAddr(14)[99] == 3.5f);
        CHECK((char const *)p.GetAddr(1) - (char const *)p.GetAddr(0) == 512);
        bb::FrameBuffer alias = buf;                       // copies share storage, as in the reference
        alias.SetFP32(1, 1, 7.0f);
        CHECK(buf.GetFP32(1, 1) == 7.0f);
    }
    // packed bits: frame f is bit f & 7 of byte f >> 3 (bit f & 31 of little-endian word f >> 5)
    {
        bb::FrameBuffer buf(70, {4}, BB_TYPE_BIT, true);
        buf.FillZero();
        buf.SetBit(0, 2, true); buf.SetBit(33, 2, true); buf.SetBit(69, 2, true);
        auto p = buf.LockConst<bb::Bit>();
        std::uint32_t const *w = reinterpret_cast<std::uint32_t const *>(p.GetAddr(2));
        CHECK(w[0] == 1u && w[1] == 2u && w[2] == (1u << 5));
        CHECK(buf.GetBit(33, 2) && !buf.GetBit(34, 2) && !buf.GetBit(33, 1));
        buf.SetBit(33, 2, false);
        CHECK(!buf.GetBit(33, 2));
        bool threw = false;
        try { buf.Lock<float>(); } catch (bb::Exception const &) { threw = true; }
        CHECK(threw);                                      // typed access checks the element type
    }
    // tensors
    {
        bb::Tensor_<float> t(bb::indices_t({4, 8}), true);
        t = 0.25f;
        auto p = t.Lock();
        p(3, 7) = 1.0f;
        CHECK(p[31] == 1.0f && p(0, 0) == 0.25f && t.GetSize() == 32);
        bb::Tensor w({16, 64}, BB_TYPE_FP32, true);
        w.InitNormalDistribution(0.5, 0.01, 1);
        double s = 0; { auto q = w.LockConst<float>(); for (int i = 0; i < 1024; ++i) { s += q[i]; } }
        CHECK(std::abs(s / 1024 - 0.5) < 0.01);
    }
    // connection table: distinct inputs per node, balanced use of inputs, reverse table equal to the oracle's
    for (std::string policy : {"", "random", "serial"}) {
        int const I = 50, O = 37;
        bb::FixedSizeConnectionTable<6> tbl;
        tbl.SetShape({I}, {O});
        tbl.InitializeConnection(3, policy);
        std::vector<std::int32_t> idx((size_t)O * 6);
        std::map<int, int> use;
        for (int o = 0; o < O; ++o) {
            std::set<int> seen;
            for (int i = 0; i < 6; ++i) { int v = (int)tbl.GetInputConnection(o, i); CHECK(v >= 0 && v < I); seen.insert(v); use[v]++; idx[(size_t)o * 6 + i] = v; }
            CHECK(seen.size() == 6);
        }
        int lo = 1 << 30, hi = 0;
        for (int v = 0; v < I; ++v) { lo = std::min(lo, use[v]); hi = std::max(hi, use[v]); }
        CHECK(hi - lo <= 2);                               // every input used about equally often
        int const stride = oracle_ReverseTable(6, idx.data(), I, O, nullptr, 0);
        std::vector<std::int32_t> rev((size_t)I * stride);
        oracle_ReverseTable(6, idx.data(), I, O, rev.data(), (int)rev.size());
        CHECK(tbl.GetReverseTableStride() == stride);
        auto p = tbl.LockConst_ReverseTable();
        bool same = true;
        for (int r = 0; r < I; ++r) for (int c = 0; c < stride; ++c) { same = same && (p(r, c) == rev[(size_t)r * stride + c]); }
        CHECK(same);
        tbl.SetInputConnection(0, 0, (tbl.GetInputConnection(0, 0) + 1) % I);     // editing the wiring rebuilds the reverse table
        idx[0] = (std::int32_t)tbl.GetInputConnection(0, 0);
        int const stride2 = oracle_ReverseTable(6, idx.data(), I, O, nullptr, 0);
        std::vector<std::int32_t> rev2((size_t)I * stride2);
        oracle_ReverseTable(6, idx.data(), I, O, rev2.data(), (int)rev2.size());
        auto p2 = tbl.LockConst_ReverseTable();
        same = (tbl.GetReverseTableStride() == stride2);
        for (int r = 0; same && r < I; ++r) for (int c = 0; c < stride2; ++c) { same = same && (p2(r, c) == rev2[(size_t)r * stride2 + c]); }
        CHECK(same);
    }
    // models: shapes, parameters, commands, ForwardNode, and no silent host execution
    {
        auto lut = bb::StochasticLutN<6, float>::Create(10);
        CHECK(lut->GetModelName() == "StochasticLut6");
        CHECK(lut->SetInputShape({4, 5}) == bb::indices_t({10}));
        CHECK(lut->GetInputNodeSize() == 20 && lut->GetOutputNodeSize() == 10);
        CHECK(lut->GetParameters().GetSize() == 1 && lut->GetGradients().GetSize() == 1);
        CHECK(lut->W().GetShape() == bb::indices_t({10, 64}));
        { auto W = lut->lock_W(); for (int i = 0; i < 64; ++i) { W(3, i) = (i == 37) ? 0.9f : 0.1f; } }
        std::vector<double> in(6);
        for (int b = 0; b < 6; ++b) { in[(size_t)b] = (37 >> b) & 1; }
        CHECK(lut->ForwardNode(3, in)[0] == 1.0);                                // lut_binarize is on by default
        lut->SendCommand("lut_binarize false");
        CHECK(std::abs(lut->ForwardNode(3, in)[0] - 0.9) < 1e-6);
        in[0] = 1.0 - in[0];
        CHECK(std::abs(lut->ForwardNode(3, in)[0] - 0.1) < 1e-6);
        bool threw = false;
        try { lut->Forward(bb::FrameBuffer(8, {4, 5}, BB_TYPE_FP32, true)); } catch (bb::Exception const &) { threw = true; }
        CHECK(threw);
        auto dl = bb::DifferentiableLutN<6, bb::Bit>::Create(12);
        CHECK(dl->GetModelName() == "DifferentiableLut6");
        dl->SetInputShape({30});
        CHECK(dl->GetParameters().GetSize() == 1);
        dl->SendCommand("parameter_lock true");
        CHECK(dl->GetParameters().GetSize() == 0);
        { auto v = dl->lock_var_const(); auto m = dl->lock_mean_const(); CHECK(v[0] == 1.0f && m[11] == 0.0f); }
        auto bl = bb::BinaryLutN<6, bb::Bit>::Create(5);
        bl->SetInputShape({9});
        bl->SetLutTable(2, 40, true);  CHECK(bl->GetLutTable(2, 40));
        bl->SetLutTable(2, 40, false); CHECK(!bl->GetLutTable(2, 40));
        std::set<bb::index_t> seen;
        for (int i = 0; i < 6; ++i) { seen.insert(bl->GetNodeConnectionIndex(4, i)); }
        CHECK(seen.size() == 6);
        CHECK(bl->Backward(bb::FrameBuffer(8, {5}, BB_TYPE_FP32, true)).GetNodeSize() == 9);
    }
    // serialization, in the shape of the reference's tests (tests/gtest/DifferentiableLutTest.cpp:10-53: dump, load into a
    // fresh layer, compare; tests/gtest/ObjectTest.cpp:191-216: reconstruct by the recorded name)
    {
        auto lut0 = bb::DifferentiableLutN<6, float>::Create(16);
        lut0->SetInputShape({16});
        { auto W = lut0->lock_W(); W(5, 9) = 0.125f; }
        { auto v = lut0->lock_var(); v[3] = 2.5f; }
        std::stringstream ss(std::ios::in | std::ios::out | std::ios::binary);
        lut0->DumpObject(ss);
        auto lut1 = bb::DifferentiableLutN<6, float>::Create(16);
        lut1->LoadObject(ss);
        CHECK(lut0->GetGamma() == lut1->GetGamma() && lut0->GetBeta() == lut1->GetBeta());
        CHECK(lut0->GetOutputShape() == lut1->GetOutputShape() && lut0->GetInputShape() == lut1->GetInputShape());
        bool same = true;
        for (bb::index_t o = 0; o < lut0->GetOutputNodeSize(); ++o) {
            for (bb::index_t i = 0; i < lut0->GetNodeConnectionSize(o); ++i) { same = same && (lut0->GetNodeConnectionIndex(o, i) == lut1->GetNodeConnectionIndex(o, i)); }
        }
        CHECK(same);
        { auto a = lut0->lock_W_const(); auto b = lut1->lock_W_const(); for (int k = 0; k < 16 * 64; ++k) { same = same && (a[k] == b[k]); } }
        { auto v = lut1->lock_var_const(); same = same && (v[3] == 2.5f) && (v[4] == 1.0f); }
        CHECK(same);
        CHECK(lut1->GetGradients().GetSize() == 1 && lut1->dW().GetShape() == bb::indices_t({16, 64}));

        auto model = bb::DifferentiableLutN<6, bb::Bit, float>::Create(bb::indices_t({1, 2, 3}));
        model->SetInputShape({32, 8});
        CHECK(model->GetObjectName() == "DifferentiableLut6_bit_fp32");
        std::stringstream s2(std::ios::in | std::ios::out | std::ios::binary);
        model->DumpObject(s2);
        auto obj = std::dynamic_pointer_cast<bb::DifferentiableLutN<6, bb::Bit, float>>(bb::Object_Load(s2));
        CHECK((bool)obj);
        if (obj) {
            CHECK(obj->GetObjectName() == model->GetObjectName());
            CHECK(obj->GetInputShape() == bb::indices_t({32, 8}) && obj->GetOutputShape() == bb::indices_t({1, 2, 3}));
        }
        // a layer of another class or width does not load into this one, and a name nobody knows reconstructs to nothing
        std::stringstream s3(std::ios::in | std::ios::out | std::ios::binary);
        model->DumpObject(s3);
        bool threw = false;
        try { bb::StochasticLutN<6, bb::Bit>::Create(6)->LoadObject(s3); } catch (bb::Exception const &) { threw = true; }
        CHECK(threw);
        std::stringstream s4(std::ios::in | std::ios::out | std::ios::binary);
        s4.write("BB_OBJ", 6); bb::SaveValue(s4, (std::int64_t)1); bb::SaveValue(s4, std::string("NoSuchLayer"));
        CHECK(!bb::Object_Load(s4));
        // tensors on their own
        bb::Tensor_<std::int32_t> t(bb::indices_t({2, 3}), true);
        { auto p = t.Lock(); for (int k = 0; k < 6; ++k) { p[k] = k + 1; } }
        std::stringstream s5(std::ios::in | std::ios::out | std::ios::binary);
        t.DumpObject(s5);
        auto t2 = std::dynamic_pointer_cast<bb::Tensor_<std::int32_t>>(bb::Object_Load(s5));
        CHECK(t2 && t2->GetShape() == bb::indices_t({2, 3}));
        if (t2) { auto p = t2->LockConst(); CHECK(p(1, 1) == 5 && p(1, 2) == 6); }          // ObjectTest.cpp:185-186
    }
    // the layers around the LUT layers: shapes, commands, refusals, and the device path's refusal without a device
    {
        auto r2b = bb::RealToBinary<bb::Bit>::Create(7, 3);
        CHECK(r2b->SetInputShape({2, 4, 5}) == bb::indices_t({6, 4, 5}) && r2b->GetInputNodeSize() == 40 && r2b->GetOutputNodeSize() == 120);
        CHECK(r2b->GetObjectName() == "RealToBinary_bit_fp32" && r2b->GetModulationSize() == 7);
        bool threw = false;
        try { bb::RealToBinary<float>::Create(2, std::make_shared<bb::Tensor>()); } catch (bb::Exception const &) { threw = true; }
        CHECK(threw);                                                   // thresholds from a value generator are not provided
        auto b2r = bb::BinaryToReal<bb::Bit>::Create(7, bb::indices_t({10}));
        CHECK(b2r->SetInputShape({70}) == bb::indices_t({10}));
        auto by_depth = bb::BinaryToReal<float>::Create(1, 7);
        CHECK(by_depth->SetInputShape({70, 2}) == bb::indices_t({10, 2}));
        threw = false;
        try { bb::BinaryToReal<float>::Create(1, bb::indices_t({9}))->SetInputShape({70}); } catch (bb::Exception const &) { threw = true; }
        CHECK(threw);                                                   // 70 inputs do not fold into 9 outputs
        auto pool = bb::MaxPooling<bb::Bit>::Create(2, 3);
        CHECK(pool->SetInputShape({4, 5, 7}) == bb::indices_t({4, 3, 3}) && pool->GetFilterHeight() == 2 && pool->GetFilterWidth() == 3);
        auto up = bb::UpSampling<>::Create(2, 3, false);
        CHECK(up->SetInputShape({4, 5, 7}) == bb::indices_t({4, 10, 21}) && up->GetOutputNodeSize() == 840);
        auto shuffle = bb::Shuffle::Create(3, bb::indices_t({2, 6}));
        CHECK(shuffle->SetInputShape({12}) == bb::indices_t({2, 6}) && shuffle->SetInputShape({6}) == bb::indices_t({6}));
        {
            std::stringstream ss(std::ios::in | std::ios::out | std::ios::binary);
            shuffle->DumpObject(ss);
            auto back = std::dynamic_pointer_cast<bb::Model>(bb::Object_Load(ss));
            CHECK((bool)back && back->GetObjectName() == "Shuffle" && back->GetOutputShape() == bb::indices_t({6}));
        }
        threw = false;
        try { bb::Shuffle::Create(4)->SetInputShape({6}); } catch (bb::Exception const &) { threw = true; }
        CHECK(threw);                                                   // 6 nodes do not split into units of 4
        {   // the stamp that says whether a tensor could have been written to since it was last looked at
            bb::Tensor_<float> t(bb::indices_t({4}));
            { auto w = t.Lock(true); w[0] = 1.0f; }
            auto const s0 = t.WriteStamp();
            { auto r = t.LockConst(); CHECK(r[0] == 1.0f); }
            CHECK(t.WriteStamp() == s0);                                // reading does not move it
            { auto w = t.Lock(); w[1] = 2.0f; }
            CHECK(t.WriteStamp() != s0);                                // a writable lock does
            auto const s1 = t.WriteStamp();
            t.Resize(bb::indices_t({8}));
            CHECK(t.WriteStamp() != s1);                                // and so does a new block
        }
        auto tanh = bb::HardTanh<>::Create(0.0f, 1.0f);
        CHECK(tanh->ForwardNode(0, {-0.5, 0.25, 2.0}) == std::vector<double>({0.0, 0.25, 1.0}));
        tanh->SendCommand("binary true");
        CHECK(tanh->ForwardNode(0, {0.4, 0.6}) == std::vector<double>({0.0, 1.0}));
        auto body = bb::Sequential::Create();
        body->Add(bb::DifferentiableLutN<6, bb::Bit>::Create((bb::index_t)36));
        body->Add(bb::DifferentiableLutDiscreteN<6, bb::Bit>::Create((bb::index_t)12));
        auto net = bb::BinaryModulation<bb::Bit>::Create(body, 7, 15);
        CHECK(net->SetInputShape({20}) == bb::indices_t({12}) && net->GetInputNodeSize() == 20 && net->GetLayer() == body);
        CHECK(net->GetParameters().GetSize() == 2 && net->GetGradients().GetSize() == 2);
        std::stringstream ss(std::ios::in | std::ios::out | std::ios::binary);
        net->DumpObject(ss);
        auto again = std::dynamic_pointer_cast<bb::Model>(bb::Object_Load(ss));
        CHECK((bool)again && again->GetObjectName() == "BinaryModulation_bit_fp32" && again->GetOutputNodeSize() == 12);
        std::stringstream s1(std::ios::in | std::ios::out | std::ios::binary), s2(std::ios::in | std::ios::out | std::ios::binary);
        net->DumpObject(s1);
        if (again) { again->DumpObject(s2); CHECK(s1.str() == s2.str()); }
        bb::FrameBuffer x(8, {20}, BB_TYPE_FP32, true);
        threw = false;
        try { net->Forward(x); } catch (bb::Exception const &) { threw = true; }
        CHECK(threw);                                                   // no device: the layers refuse instead of computing on the host
    }
    // workgroup index -> (frame chunk, node tile) without an integer division: exact for every index below 2^31
    {
        int const divisors[] = {1, 2, 3, 5, 7, 64, 255, 256, 257, 1000, 1024, 1536, 4096, 65535, 1 << 20, (1 << 20) + 1, 0x3fffffff, 0x7fffffff};
        std::uint64_t state = 0x9e3779b97f4a7c15ull;
        for (int d : divisors) {
            bbhip::TileDivisor const t = bbhip::make_tile_divisor(d);
            auto check = [&](std::uint32_t n) {
                int outer, tile;
                bbhip::split_tile((int)n, t, outer, tile);
                if (outer != (int)(n / (std::uint32_t)d) || tile != (int)(n % (std::uint32_t)d)) { CHECK(!"split_tile"); }
            };
            for (std::uint32_t n = 0; n < 70000; ++n) { check(n); }
            for (std::uint32_t k = 1; k < 200; ++k) {                 // around multiples of d and at the top of the range
                std::uint64_t const m = (std::uint64_t)k * (std::uint64_t)d;
                if (m < 0x7fffffffull) { check((std::uint32_t)m); check((std::uint32_t)m - 1); check((std::uint32_t)m + 1 < 0x80000000u ? (std::uint32_t)m + 1 : 0); }
                check(0x7fffffffu - k);
            }
            for (int i = 0; i < 200000; ++i) {
                state ^= state << 13; state ^= state >> 7; state ^= state << 17;
                check((std::uint32_t)(state >> 33));
            }
            check(0x7fffffffu);
        }
    }
    // slabs of the per-corner sums: never dearer than the best power of two, or than equal slabs that fill whole rounds of 512 workgroups, whatever the
    // node count; within the number of slabs that the scratch memory holds
    {
        std::uint64_t state = 0x2545f4914f6cdd1dull;
        auto draw = [&](int lo, int hi) { state ^= state << 13; state ^= state >> 7; state ^= state << 17; return lo + (int)((state >> 20) % (std::uint64_t)(hi - lo + 1)); };
        auto check = [&](int nodes, int frames, long long max_slabs) {
            int const tiles = bbhip::ceil_div(nodes, 4), slab = bbhip::corner_slab_frames(frames, tiles, max_slabs);
            long long const cost = bbhip::corner_slab_cost(frames, tiles, slab);
            bool ok = slab > 0 && slab % 256 == 0 && bbhip::ceil_div(frames, slab) <= max_slabs && (frames > 1024 || slab >= frames);
            auto not_dearer = [&](long long than) { if ((frames + than - 1) / than <= max_slabs) { ok = ok && cost <= bbhip::corner_slab_cost(frames, tiles, than); } };
            not_dearer(bbhip::ceil_div(frames, 256) * 256);
            for (int power = 1024; power < frames && power <= 65536; power *= 2) { not_dearer(power); }
            for (int rounds = 1; rounds <= 4; ++rounds) {
                int const slabs = rounds * 512 / tiles, equal = slabs < 1 ? 0 : bbhip::ceil_div(bbhip::ceil_div(frames, slabs), 256) * 256;
                if (equal >= 1024) { not_dearer(equal); }
            }
            if (!ok) { std::printf("%d nodes x %d frames, at most %lld slabs: %d\n", nodes, frames, max_slabs, slab); CHECK(!"corner_slab_frames"); }
        };
        int const sizes[][2] = {{4200, 65536}, {4200, 230400}, {4500, 65536}, {4200, 32768}, {2100, 230400}, {4200, 1 << 20}, {216, 230400}, {87, 94500}, {4096, 8192}, {1, 1}};
        for (auto const &s : sizes) { check(s[0], s[1], 1 << 20); }
        // one slab or several, as measured (several 7 and 6 % slower; 4, 5 and 10 % faster)
        for (auto const &s : {std::make_pair(2666, 8646), {2795, 10066}}) { CHECK(bbhip::corner_slab_frames(s.second, bbhip::ceil_div(s.first, 4), 1 << 20) >= s.second); }
        for (auto const &s : {std::make_pair(24, 4223), {4200, 32768}, {300, 7756}}) { CHECK(bbhip::corner_slab_frames(s.second, bbhip::ceil_div(s.first, 4), 1 << 20) < s.second); }
        for (int i = 0; i < 20000; ++i) { check(draw(1, 1 << draw(0, 14)), draw(1, 1 << draw(0, 20)), 1 + draw(0, 1 << draw(0, 12))); }
    }

    // one-launch backward pass of small layers on two-valued inputs, where its forms and two launches were measured (device time in microseconds, with
    // prepared tables and without; 0: not measured): within a tenth of two launches, and of the fastest on the mean of the two
    {
        struct { int n; bool batch_norm; int inputs, nodes, frames, fan; double four[2], sixteen[2], two[2]; } const rows[] = {
            {6, true, 784, 1024, 256, 19, {5.8, 6.9}, {9, 9}, {7.8, 8.4}},          {6, true, 26, 104, 64, 35, {6.7, 8.2}, {5.3, 6.2}, {7.4, 7.8}},
            {6, true, 347, 1643, 64, 44, {8.3, 10.5}, {9.2, 11.3}, {9.1, 9.7}},     {6, true, 95, 579, 256, 51, {9.0, 11.2}, {6.5, 7.9}, {8.0, 8.3}},
            {6, true, 207, 1495, 64, 63, {10.3, 13.1}, {8.9, 10.3}, {8.7, 9.5}},    {6, true, 784, 6144, 64, 69, {15.1, 20.5}, {21.0, 25.8}, {16.0, 18.2}},
            {6, true, 645, 4947, 64, 69, {14.0, 18.4}, {18.0, 22.3}, {13.9, 15.9}}, {6, true, 47, 469, 34, 76, {11.7, 14.9}, {7.7, 9.7}, {8.6, 9.0}},
            {6, true, 50, 522, 116, 79, {12.1, 15.5}, {8.0, 9.9}, {8.8, 9.2}},      {6, true, 34, 598, 64, 129, {18.4, 23.9}, {10.3, 13.7}, {9.7, 10.3}},
            {3, true, 149, 2247, 64, 66, {9.8, 11.2}, {6.5, 7.4}, {9.4, 9.7}},      {2, true, 362, 3324, 64, 34, {6.6, 7.1}, {6.6, 6.9}, {9.5, 9.7}},
            {4, true, 650, 4818, 64, 49, {10.1, 11.8}, {13.9, 15.8}, {13.4, 14.3}}, {6, true, 915, 2624, 256, 33, {9.1, 11.3}, {15.9, 18.1}, {11.5, 12.7}},
            {6, false, 210, 1841, 44, 74, {8.7, 12.1}, {6.7, 8.2}, {7.9, 8.7}},     {6, false, 784, 6144, 256, 71, {12.1, 17.2}, {14.0, 16.9}, {15.9, 18.3}},
            {4, false, 482, 5161, 64, 62, {7.6, 9.4}, {8.6, 9.7}, {10.7, 11.5}},    {6, true, 300, 300, 512, 15, {6.2, 6.9}, {9, 9}, {10.3, 10.8}},
            {6, true, 360, 70, 1024, 6, {4.5, 4.8}, {9, 9}, {7.3, 7.6}}};
        for (auto const &r : rows) {
            int const waves = bbhip::corner_small_waves(r.n, r.batch_norm, r.frames, r.inputs, r.nodes, r.fan);
            double const *const taken = waves == 16 ? r.sixteen : waves == 4 ? r.four : r.two;
            auto mean = [](double const *t) { return 0.5 * (t[0] + t[1]); };
            bool ok = mean(taken) <= 1.1 * std::min(mean(r.four), std::min(mean(r.sixteen), mean(r.two)));
            for (int plain = 0; plain < 2; ++plain) { ok = ok && taken[plain] <= 1.1 * r.two[plain]; }
            if (!ok) { std::printf("%d inputs x %d nodes x %d frames: %d wavefronts\n", r.inputs, r.nodes, r.frames, waves); CHECK(!"corner_small_waves"); }
        }
        // no list is longer than what the kernel holds, whatever the layer
        for (int fan = 0; fan <= 4096; ++fan) {
            for (int inputs : {1, 256, 257, 1536, 1537, 2048, 2049, 100000}) {
                for (int frames : {1, 256, 257, 512, 513, 1024}) {
                    int const waves = bbhip::corner_small_waves(6, fan % 2 == 0, frames, inputs, 1, fan);
                    CHECK(waves == 0 || bbhip::ceil_div(fan, waves) <= bbhip::kCornerSmallShare);
                }
            }
        }
    }

    // items of shared lists in turn or one after another, where both were measured (backward calls, microseconds): at most a twentieth slower than the faster
    {
        struct { bool batch_norm; int workgroups, fan; double in_turn, consecutive; } const rows[] = {
            {false, 24, 1840, 57.2, 48.1}, {false, 34, 1128, 39.1, 34.6}, {false, 54, 973, 33.4, 29.6},  {false, 58, 1031, 36.9, 32.7},  {false, 70, 948, 36.1, 31.7},
            {false, 132, 1645, 63.7, 55.1}, {false, 136, 653, 28.1, 24.2}, {false, 12, 388, 13.9, 14.4}, {false, 900, 621, 77.9, 103.0}, {false, 286, 447, 27.2, 29.9},
            {true, 70, 1361, 57.8, 53.2},  {true, 11, 897, 31.5, 33.8},   {true, 805, 889, 103.7, 151.3}, {true, 640, 1280, 126.6, 173.2}, {true, 42, 524, 21.6, 23.0}};
        for (auto const &r : rows) {
            double const taken = bbhip::dx_items_in_turn(r.batch_norm, r.workgroups, r.fan) ? r.in_turn : r.consecutive;
            if (taken > 1.05 * std::min(r.in_turn, r.consecutive)) { std::printf("%d workgroups, lists of %d\n", r.workgroups, r.fan); CHECK(!"dx_items_in_turn"); }
        }
    }

    // passes of a wavefront in the forward pass of up to 1024 frames, where both were measured (microseconds)
    {
        struct { int nodes, frames; double side_by_side, in_turn; } const rows[] = {{700, 1000, 4.89, 5.93}, {1024, 1024, 5.18, 5.73}, {1500, 600, 6.46, 5.60}, {3000, 400, 7.57, 7.13}, {4000, 300, 8.81, 7.98}, {6144, 1024, 15.0, 10.9}};
        for (auto const &r : rows) { CHECK((bbhip::forward_quad_passes(r.nodes, r.frames) == 1) == (r.side_by_side < r.in_turn)); }
        CHECK(bbhip::forward_quad_passes(8000, 64) == 0 && bbhip::forward_quad_passes(8000, 65) == 1 && bbhip::forward_quad_passes(8000, 256) == 1 &&
              bbhip::forward_quad_passes(8000, 512) == 2 && bbhip::forward_quad_passes(8000, 513) == 4);
    }

    {
        // workgroups that share a node's fp32 output: at most 256 of them altogether, every block in one share, no share empty, none for a single wavefront or block
        for (int tiles : {1, 2, 3, 24, 72, 85, 100, 127, 128, 129, 255, 256, 257, 4096}) {
            for (int blocks = 1; blocks <= 24; ++blocks) {
                int const share = bbhip::forward_out_blocks(tiles, 4, blocks), parts = (blocks + share - 1) / share;
                CHECK(share >= 1 && share <= blocks && (parts == 1 || tiles * parts <= 256) && (parts - 1) * share < blocks);
                CHECK(bbhip::forward_out_blocks(tiles, 1, blocks) == blocks && (tiles <= 128 || parts == 1));
            }
        }
    }

    // per-corner sums in slabs or a node by a workgroup, where both were measured (backward call, microseconds): at most 5 % slower than the faster
    {
        struct { int n, nodes, frames; double slabs, workgroups; } const rows[] = {
            {6, 12, 2300, 10.8, 9.5}, {6, 80, 14000, 15.9, 13.4}, {6, 256, 4500, 16.6, 13.6}, {6, 256, 16384, 22.4, 21.6}, {6, 40, 24000, 14.9, 15.1}, {6, 30, 100000, 20.5, 29.4},
            {6, 300, 4500, 17.0, 18.7}, {5, 300, 4000, 14.4, 16.0}, {5, 256, 6000, 16.1, 13.6}, {4, 30, 10000, 11.6, 9.2}, {4, 512, 6000, 17.2, 15.9}, {2, 400, 10000, 13.8, 12.3}, {6, 100, 1500, 9.9, 10.2}};
        for (auto const &r : rows) {
            double const taken = bbhip::node_sums(r.n, r.nodes, r.frames) ? r.workgroups : r.slabs;
            if (taken > 1.05 * std::min(r.slabs, r.workgroups)) { std::printf("%d x %d\n", r.nodes, r.frames); CHECK(!"node_sums"); }
        }
        CHECK(!bbhip::node_sums(6, 256, 2048) && bbhip::node_sums(6, 256, 2049) && bbhip::node_sums(6, 256, 16384) && !bbhip::node_sums(6, 256, 16385) && !bbhip::node_sums(2, 513, 4000));
    }

    // dx of few inputs input by input or node by node, where both were measured (backward call, microseconds): at most 5 % slower than the faster
    {
        struct { int n, inputs, nodes, frames; double by_input, by_node; } const rows[] = {
            {6, 27, 216, 230400, 117.5, 90.8}, {6, 27, 216, 115200, 64.7, 53.6}, {6, 27, 216, 50000, 40.2, 44.5}, {6, 27, 87, 94500, 31.4, 31.7}, {6, 28, 300, 60000, 53.5, 58.4},
            {6, 9, 150, 100000, 49.0, 39.1}, {2, 9, 216, 100000, 41.7, 35.6}, {4, 9, 100, 230400, 48.8, 40.2}, {6, 27, 36, 700000, 68.6, 63.9}, {6, 27, 24, 230400, 25.2, 25.7},
            {4, 9, 16, 400000, 21.6, 25.9}, {2, 18, 16, 180000, 14.4, 17.5}, {3, 28, 16, 262144, 19.3, 21.4}, {6, 20, 500, 30000, 54.2, 77.1}, {4, 27, 216, 80000, 40.7, 43.2},
            {6, 27, 216, 262144, 140.9, 90.4}, {6, 27, 216, 262656, 140.8, 109.3}, {6, 27, 52, 263000, 43.3, 44.1}, {6, 27, 36, 180000, 28.7, 29.2}, {6, 27, 72, 530000, 92.9, 80.8},
            {6, 27, 1000, 97793, 307, 192}, {6, 27, 2100, 150000, 1098, 735}, {6, 27, 4000, 97793, 1484, 711}, {4, 9, 4000, 120000, 1409, 699}, {2, 9, 130, 263000, 63.1, 56.9}};
        for (auto const &r : rows) {
            double const taken = bbhip::few_inputs_dx(r.n, r.inputs, r.nodes, r.frames) ? r.by_node : r.by_input;
            if (taken > 1.05 * std::min(r.by_input, r.by_node)) { std::printf("%d x %d x %d\n", r.inputs, r.nodes, r.frames); CHECK(!"few_inputs_dx"); }
        }
        CHECK(!bbhip::few_inputs_dx(6, 29, 216, 230400) && !bbhip::few_inputs_dx(6, 27, 4097, 230400));
    }

    // dx from kept indices in passes of 256 or 512 frames, where both were measured (training call, microseconds): at most 5 % slower than the faster
    {
        struct { int n, inputs, nodes, frames, max_fan; double one, two; } const rows[] = {
            {6, 560, 1055, 3778, 22, 32.9, 29.4}, {5, 632, 1175, 5013, 21, 37.2, 32.8}, {6, 3664, 1195, 7782, 8, 60.8, 55.0}, {6, 807, 1033, 12218, 18, 62.8, 59.4},
            {6, 877, 1425, 3698, 21, 36.5, 33.0}, {6, 1727, 1444, 9479, 14, 67.0, 68.6}, {6, 3987, 1569, 514, 9, 19.0, 19.9}, {5, 1833, 1530, 6448, 12, 46.9, 48.9},
            {4, 2909, 1145, 1358, 8, 20.6, 20.0}, {2, 825, 468, 4363, 5, 18.7, 17.4}, {5, 333, 469, 5793, 14, 25.4, 24.5}, {6, 2754, 1341, 498, 11, 16.2, 17.8},
            {6, 2046, 2018, 1150, 15, 25.6, 27.1}, {6, 98, 1550, 1284, 117, 24.2, 28.6}, {6, 585, 772, 5509, 16, 35.0, 30.2},
            // (with other inputs and buffers than the call before)
            {6, 1418, 705, 1150, 12, 18.5, 19.9}, {6, 1348, 896, 1164, 13, 19.7, 21.0}, {6, 3418, 753, 988, 8, 17.2, 17.0}, {3, 1775, 945, 1869, 7, 18.9, 19.3}, {5, 1529, 1382, 1275, 14, 21.2, 22.6},
            {6, 1206, 1382, 1813, 19, 27.9, 25.4}, {6, 1511, 1428, 2118, 16, 31.3, 30.4}, {5, 773, 1482, 3855, 20, 34.2, 30.1}, {6, 168, 959, 17363, 50, 78.7, 73.2}, {6, 2919, 482, 519, 6, 15.9, 15.9},
            {3, 1708, 1259, 14639, 9, 74.2, 73.1}, {2, 527, 1189, 15747, 11, 58.8, 61.0}, {2, 2386, 762, 12598, 5, 47.1, 46.6}, {6, 1336, 804, 1505, 12, 20.1, 20.6}, {6, 2740, 921, 734, 9, 16.6, 17.6},
            {4, 1341, 902, 1385, 10, 18.1, 19.1}, {4, 1764, 1151, 1263, 10, 19.1, 20.5}, {4, 1016, 898, 1816, 12, 18.5, 19.4}, {4, 3845, 1301, 687, 7, 17.0, 17.9}, {5, 3141, 1142, 568, 8, 16.9, 17.8},
            {5, 6653, 1291, 1828, 6, 28.5, 27.0}, {5, 440, 623, 8009, 15, 34.9, 30.8}, {5, 968, 1345, 3056, 17, 30.8, 27.6}, {4, 910, 1232, 2723, 14, 26.7, 25.3}, {4, 5773, 1346, 3968, 6, 38.0, 34.8},
            {6, 2316, 1272, 1222, 11, 23.0, 24.2}, {6, 605, 1347, 3349, 26, 32.5, 30.7}, {6, 851, 1206, 2832, 19, 32.1, 28.9}};
        for (auto const &r : rows) {
            double const taken = bbhip::dx_table_quads(r.n, r.inputs, r.nodes, r.frames, r.max_fan > 15) == 1 ? r.one : r.two;
            if (taken > 1.05 * std::min(r.one, r.two)) { std::printf("%d x %d x %d\n", r.inputs, r.nodes, r.frames); CHECK(!"dx_table_quads"); }
        }
        CHECK(bbhip::dx_table_quads(6, 27, 216, 230400, true) == 4 && bbhip::dx_table_quads(6, 6144, 1024, 1024, true) == 2 && bbhip::dx_table_quads(6, 4096, 4096, 8192, false) == 1);
    }

    // per-corner sums of one slab: in blocks requested ahead, or all frames at once, where both were measured (sums launch, microseconds)
    {
        struct { int frames; double blocks, at_once; } const rows[] = {
            {489, 11.2, 8.2}, {747, 15.6, 11.1}, {82, 8.7, 8.0}, {150, 10.7, 8.7}, {1981, 16.1, 15.2}, {1140, 13.7, 13.3}, {1696, 20.3, 18.4}, {102, 23.9, 13.3},
            {1008, 25.3, 16.9}, {911, 13.8, 11.8}, {1045, 21.7, 21.0}};
        for (auto const &r : rows) {
            bool const blocks = bbhip::corner_sums_form(r.frames, 1) == bbhip::kSumsLong;
            if ((blocks ? r.blocks : r.at_once) > std::min(r.blocks, r.at_once)) { std::printf("%d frames\n", r.frames); CHECK(!"corner_sums_form"); }
        }
        for (int frames = 1; frames <= 5000; ++frames) {        // (what does not fit the form that is taken would be left out of the sums)
            int const form = bbhip::corner_sums_form(frames, 1);
            CHECK(form == bbhip::kSumsLong || frames <= form * 256);
            CHECK(bbhip::corner_sums_form(frames, 2) == bbhip::kSumsLong);
        }
    }

    // real-valued inputs: lists of 8 to 15 items shared or not, in passes of 128 or 256 frames as the rules take them, where both were measured (training
    // calls, microseconds): at most a twentieth slower than the other
    {
        struct { int inputs, nodes, frames, fan, links; double shared, own; } const rows[] = {
            {69, 66, 906, 13, 396, 10.4, 15.0},     {1500, 800, 700, 14, 4800, 20.6, 22.9},  {1024, 1024, 1000, 14, 6144, 23.7, 25.9}, {16, 26, 14420, 13, 156, 12.7, 14.4},
            {268, 181, 1715, 11, 1086, 13.8, 16.0}, {1192, 1047, 163, 15, 6282, 13.4, 16.7}, {16, 26, 29705, 14, 156, 20.1, 16.8},     {40, 63, 15921, 9, 189, 11.2, 9.8},
            {116, 321, 8625, 12, 642, 25.8, 23.3},  {26, 25, 15518, 9, 150, 13.7, 12.5},     {73, 89, 19508, 9, 267, 22.2, 21.1},      {3383, 3689, 235, 14, 14756, 19.6, 18.4},
            {3817, 6000, 253, 15, 18000, 21.3, 19.9}};
        for (auto const &r : rows) {
            bool const wide = bbhip::dx_wide_passes(r.inputs, r.nodes, r.frames, r.fan, r.links);
            long long const groups = (long long)bbhip::ceil_div(r.frames, wide ? 256 : 128) * bbhip::ceil_div(r.inputs, 4);
            bool const shared = r.fan >= bbhip::dx_shortest_shared_list(r.inputs, r.nodes, r.frames, groups);
            if ((shared ? r.shared : r.own) > 1.05 * std::min(r.shared, r.own)) {
                std::printf("%d inputs x %d nodes x %d frames: shared %d\n", r.inputs, r.nodes, r.frames, shared); CHECK(!"dx_shortest_shared_list");
            }
        }
    }

    // order of the Im2Col kernels' workgroups, where both were measured (forward, microseconds, pieces of a row first and frames first)
    {
        struct { int frames; double pieces, frames_first; } const rows[] = {
            {1024, 31.5, 27.5}, {1024, 48.7, 42.0}, {1521, 108.8, 92.5}, {1991, 31.1, 29.3}, {64, 20.4, 23.0}, {256, 78.0, 97.0}, {370, 114.1, 146.1}, {620, 89.8, 97.0}};
        for (auto const &r : rows) {
            bool const first = bbhip::im2col_frames_first(bbhip::ceil_div(r.frames, 64), 64);
            if ((first ? r.frames_first : r.pieces) > std::min(r.pieces, r.frames_first)) { std::printf("%d frames\n", r.frames); CHECK(!"im2col_frames_first"); }
        }
    }

    // padding that the kernel of a packed output writes: no word number near the end of the range, and a bounded number of iterations
    for (int words : {1, 3, 1 << 24}) {
        for (int stride : {words, words + 1, words + 4095, words + 4096, words + 4097, 0x7fffffff}) {
            int const end = bbhip::packed_padding_end(words, stride);
            CHECK(end <= stride && end - words <= 4096 && (end == stride || end - words == 4096));
        }
    }

    // units of the BinaryLut kernels, where both were measured (microseconds, units of 64 and of 128 words)
    {
        struct { int nodes, words; double short_units, long_units; } const rows[] = {{30, 93, 2.00, 2.24}, {40, 256, 2.01, 2.24}, {239, 261, 2.13, 2.26}, {183, 688, 2.09, 2.21},
            {154, 69, 2.01, 2.18}, {354, 394, 2.43, 2.38}, {29, 6663, 2.29, 2.19}, {4708, 69, 3.84, 3.19}, {5405, 5653, 59.97, 41.02}};
        for (auto const &r : rows) { CHECK((bbhip::binary_unit_words(r.words, r.nodes) == 64) == (r.short_units < r.long_units)); }
    }

    // the classifier tail by a wavefront per channel or by a row of lanes, where both were measured (microseconds)
    {
        struct { int n, inputs, channels, stride; double wavefront, row; } const rows[] = {{7, 70, 10, 64, 6.35, 3.66}, {7, 70, 10, 1152, 6.64, 3.99}, {7, 70, 10, 2176, 6.66, 4.41},
            {7, 70, 10, 4096, 6.75, 5.44}, {12, 192, 16, 1152, 12.4, 6.15}, {13, 208, 16, 4096, 14.7, 11.8}, {7, 70, 10, 6144, 6.89, 6.90}, {7, 70, 10, 16512, 8.37, 13.7}, {7, 70, 10, 65664, 20.6, 44.8}};
        for (auto const &r : rows) { CHECK(bbhip::tail_small(r.n, r.inputs, r.channels, r.stride) == (r.row < r.wavefront)); }
        // other counts of inputs, fewer channels, and more inputs per node than that form has room for
        CHECK(!bbhip::tail_small(7, 60, 10, 1152) && !bbhip::tail_small(16, 80, 5, 2176) && !bbhip::tail_small(15, 45, 3, 640) && !bbhip::tail_small(30, 240, 8, 640) && !bbhip::tail_small(30, 90, 3, 640));
    }

    // rows that share a workgroup in the pooling kernels, where both were measured (microseconds): at most 3 % slower than the faster
    {
        struct { int nodes, lanes; double shared, own; } const rows[] = {{120, 51, 3.31, 3.08}, {180, 64, 3.12, 2.93}, {48600, 64, 82.1, 79.7}, {50445, 64, 35.0, 32.9},
            {46740, 128, 151.8, 146.4}, {73872, 61, 133.5, 129.9}, {7056, 64, 10.3, 11.5}, {90000, 32, 32.4, 40.8}, {29070, 70, 49.8, 61.3}, {4056, 13, 2.6, 4.1}, {16, 1, 2.16, 2.30},
            {12936, 45, 14.1, 16.3}, {4482, 83, 8.9, 10.2}, {60, 15, 2.30, 2.47}};
        for (auto const &r : rows) {
            int const count = bbhip::pool_shared_rows(r.lanes, r.nodes);
            CHECK(count >= 1 && count * r.lanes <= 256);
            if ((count > 1 ? r.shared : r.own) > 1.03 * std::min(r.shared, r.own)) { std::printf("%d rows, %d threads\n", r.nodes, r.lanes); CHECK(!"pool_shared_rows"); }
        }
    }

    // frames per thread of the pooling kernels, as measured (share of the time of four frames that one frame per thread takes, few rows, backward)
    {
        struct { int frames; double one; } const rows[] = {{2, 0.79}, {3, 0.65}, {5, 0.81}, {6, 0.74}, {7, 0.71}, {9, 0.83}, {11, 0.78}, {13, 0.83}, {15, 0.79}, {4, 1.1}, {8, 1.1}, {50, 1.22}, {99, 1.39}};
        for (auto const &r : rows) { CHECK(bbhip::pool_four_frames(r.frames) == (r.one > 1.0)); }
    }

    std::printf("%s (%d failed checks)\n", g_fail ? "FAILED" : "OK", g_fail);
    return g_fail ? 1 : 0;
}
