// All layers of a decode step of one to eight rows in one launch.
//
// As launches a layer of so few rows is five of 3.6 to 7 us for 1 us of work each: start, kernel arguments, the first loads' round trip, the end and 1.4 us to the next.
// Here 256 workgroups, one to a CU, walk through the layers together.  What a phase leaves for the next goes through memory at device scope without flags: a place of a
// hand-off buffer is empty (kResidentEmpty) until its value is there, and whoever needs the values reads them until none is empty.  A layer of Qwen3-0.6B with one row of 137 tokens
// takes 16.3 us, 27 as launches: five hand-offs of 1.8 to 2.4, four products of 0.4, their sums 0.4, the attention 3.5; the weights (31.5 MB) are 6.2 of memory behind them.
//
// What a hand-off costs with 256 workgroups that all read what all wrote, measured alone: 1.44 us; with a flag a workgroup, waited for before the values are read, 3.4.  And:
//  - a wave's loads return behind its own earlier stores, which take 2 us to be there: one wave hands on and empties, others read (22 -> 20.5 us a layer);
//  - with 8 or 32 workgroups' words to a line 2.8 to 4 us: each has lines of its own (45 -> 34 us a layer of 8 rows with its places side by side, 32 in lines of their own);
//  - 8 MB of weights asked for at once meanwhile: 2.9 us.  They come a few at a time, and not before the hand-on is on its way (20.5 -> 16.7);
//  - many values a reader: one of them until it is there, then all (8 rows 31.5 -> 27.5 us a layer, 4 rows 24 -> 21);
//  - what a reader does with a value: a place within a block for each reader, of every B-th block, so that the steps from one to the next are constants of the loads and LDS
//    writes (a step of 8 rows 983 -> 880 us, of 4 737 -> 696, of 2 635 -> 608; with the steps in registers 8 rows took 998).  That goes for every width of the feed-forward: with steps in registers where
//    it is not 3072, four layers of 1024 features took 8 rows 121 us, 110 as launches, and now 109; 28 layers of 8 heads on 8 681, 661 and 605.
//
// A workgroup is four row waves and four weight waves.  Weight waves hold what the workgroup needs of the weights in registers (30 KB a wave), asked for one or two phases ahead,
// because a wave's loads return in order: a value asked for behind weights would wait for them.  Row waves wait for values, lay them into LDS as bf16 planes, run the attention, add up
// the products' partial sums, and hand on.
//
// Products: a workgroup has four features of the 1024 of the stream ("a quad"), NQ / 1024 quads of q, k and v and I / 1024 of gate and of up.  One matrix instruction takes a quad at
// four places of K: operand row i is feature i & 3 at K's part i >> 2, operand column c row c & 3 of the batch at part c >> 2; the 16 of 256 results whose parts agree
// count.  The work left out costs no time: 0.3 us a phase is the chain of LDS reads, 8 products and LDS writes.
//
// Buffers are emptied while the step goes on.  A workgroup that has read all of phase p's values knows that everybody has handed on phase p, so nobody reads phase
// p - 1's values any more: it empties its own places of those, and its next hand-on but one comes after (stores_there), so that whoever has seen that finds them empty.  What the last
// layer leaves is emptied by the next launch, which uses the other set.
//
// Waits are bounded: a launch whose workgroups do not all get onto the chip (other processes with such launches on it) ends, says so, and the caller runs the step as launches.
#include "resident.h"

#include "attn_wave.h"

namespace nvllm {
namespace {

constexpr int H = 1024;                       // the stream: a quad to a workgroup
constexpr int kMaxQ = 4, kMaxO = 2, kMaxI = 3;  // NQ, KO, I in 1024ths: 8 + 4 + 12 + 6 fragments of 4 registers a lane are a layer's weights
// Turns of 64 cycles between two weight fragments, and before the first behind a hand-on.  One and eight rows of 137 tokens, us a step: 8 and 8 542, 855; 5 and 12 554, 876; 8 and 12
// 556, 860; 8 and 5 550, 859; 8 and 2 551, 843; 5 and 5 561, 847; 11 and 5 565, 863; without a pause 640 (one row)
constexpr int kPace = 8, kBehind = 8;
constexpr int kSlot = 20;                     // float4 from one (quad, row)'s partial sums to the next's: 16 and 4 to be on other banks

// What a workgroup hands on is a block of lines of its own: with 8 or 32 workgroups to a line a hand-on took 2 us longer.
__host__ __device__ constexpr int lines(int words) { return (words + 31) / 32 * 32; }
// hand-off buffers, in words
struct Places {
    size_t qkv, ctx, part, mid, act, out, words;  // act, out: of set 0; set 1's behind them
    size_t act_words, out_words;
};
__host__ __device__ inline Places places(const ResidentSizes& z) {
    Places p{};
    size_t at = 0;
    auto take = [&](size_t n) { const size_t a = at; at += n; return a; };
    p.qkv = take((size_t)kResidentGroups * lines(kResidentRows * (z.NQ / 256)));
    p.ctx = take((size_t)kResidentRows * z.KO);
    p.part = take((size_t)kResidentRows * z.nh * kResidentParts * kResidentPart);
    p.mid = take((size_t)kResidentGroups * lines(kResidentRows * 5));
    p.act_words = (size_t)kResidentGroups * lines(kResidentRows * (z.I / 256));
    p.out_words = (size_t)kResidentGroups * lines(kResidentRows * 5);
    p.act = take(2 * p.act_words);
    p.out = take(2 * p.out_words);
    p.words = at;
    return p;
}

__device__ __forceinline__ uint32_t filled(uint32_t v) { return v == kResidentEmpty ? 0x7FC00000u : v; }  // (a NaN either way)
__device__ __forceinline__ uint32_t word_of(float v) { return filled(__builtin_bit_cast(uint32_t, v)); }
__device__ __forceinline__ uint32_t planes_word(float v) {
    uint16_t h, l;
    split_bf16(v, h, l);
    return filled((uint32_t)h << 16 | l);
}
__device__ __forceinline__ uint32_t load_shared4(__amdgpu_buffer_rsrc_t r, int offset) { return __builtin_amdgcn_raw_buffer_load_b32(r, offset, 0, 16); }
__device__ __forceinline__ uint32_t most(const uint4& v) { return max(max(v.x, v.y), max(v.z, v.w)); }
__device__ __forceinline__ uint32_t most(const uint2& v) { return max(v.x, v.y); }
// every wave of the workgroup; loads and stores to memory stay in flight
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void stores_there() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }
// sum over the four lanes of a quad
__device__ __forceinline__ float lanes4_sum(float v) {
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xf, 0xf, false));
    v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xf, 0xf, false));
    return v;
}

// A wave's waits.  read(): asks for its values, then says whether none of this lane's is empty.  Once a wait has run out, here or elsewhere, the wave waits no more and walks on with
// whatever it finds (a way out of the layers' loop would have the compiler wait for weights that are not needed yet).
struct Waiting {
    int* gave_up;
    int* host_gave_up;
    int spins;
    bool over = false;
    template <class F>
    __device__ __forceinline__ bool until(F read) {
        for (int n = 0;; ++n) {
            if (__builtin_amdgcn_ballot_w64(!read()) == 0) return !over;
            asm volatile("" ::: "memory");
            if (over) return false;
            if (n < spins && ((n & 63) != 63 || __builtin_amdgcn_readfirstlane(__hip_atomic_load(gave_up, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) == 0)) continue;
            over = true;
            if ((threadIdx.x & 63) == 0) {
                __hip_atomic_store(gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                __hip_atomic_store(host_gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            return false;
        }
    }
};

// RP: rows the launch is made for (1, 2, 4, 8), R of them there
template <int RP>
struct Lds {
    static constexpr int RS = (RP + 3) / 4, SR = RS * 4;          // sets of four rows: a matrix instruction's
    static constexpr int x_bytes(int K) { return K * 2 + 16; }    // a row of a plane: four rows' fragments on different banks
    int lo, part, ssq, ml, obuf, q, fresh, bytes;  // offsets
    __host__ __device__ Lds(int widest, int gqa) {
        int at = 0;
        auto take = [&](int n) { const int a = at; at += (n + 15) / 16 * 16; return a; };
        lo = take(RP * x_bytes(widest)); take(RP * x_bytes(widest));
        part = take(2 * kMaxI * SR * kSlot * 16);
        ssq = take(kResidentRows * 16);
        ml = take(4 * 2 * 16 * 4);
        obuf = take(4 * gqa * 33 * 16);
        q = take(2 * gqa * 136 * 2);
        fresh = take(2 * 128 * 2);
        lo = RP * x_bytes(widest);
        bytes = at;
    }
};

// a layer's pointers by scalar loads, as uniform values
typedef const __attribute__((address_space(4))) ResidentLayer* layers_t;

template <int RP>
__global__ void __launch_bounds__(512, 2) resident_step_kernel(ResidentArgs a) {
    using L = Lds<RP>;
    constexpr int RS = L::RS, SR = L::SR;
    extern __shared__ __attribute__((aligned(16))) char smem[];
    const layers_t layers = (layers_t)(uintptr_t)a.layers;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nq = a.z.NQ >> 10, ko = a.z.KO >> 10, ni = a.z.I >> 10, R = a.R, gqa = a.z.nh / a.z.kv;
    const L lds(max(a.z.KO, max(a.z.I, H)), gqa);
    const Places at = places(a.z);
    // quads of a weight tile's 16 features to workgroups of one XCD, whose L2 reads their lines once
    const int wg = blockIdx.x, quad = (wg & 7) * (kResidentGroups / 8) + (wg >> 3);
    // attention: workgroup = key head, row and part of the context; a wave = one head of a row in parts
    const int units = R * a.z.kv * a.parts;
    const int u_head = wg % a.z.kv, u_row = min(wg / a.z.kv % R, R - 1), u_part = wg / (a.z.kv * R);
    const uniform_ints_t rec = uniform_ints(reinterpret_cast<const int*>(a.rows + u_row));
    const int pos = rec[2], n_tiles = (pos >> 5) + 1, t_begin = u_part * a.part_tiles, t_end = min(n_tiles, t_begin + a.part_tiles);
    const bool unit = wg < units && t_begin < n_tiles;

    uint32_t* const b_qkv = a.buffer + at.qkv;
    uint32_t* const b_ctx = a.buffer + at.ctx;
    uint32_t* const b_part = a.buffer + at.part;
    uint32_t* const b_mid = a.buffer + at.mid;
    uint32_t* const b_act = a.buffer + at.act + a.set * at.act_words;
    uint32_t* const b_out = a.buffer + at.out + a.set * at.out_words;
    float* const ssq = reinterpret_cast<float*>(smem + lds.ssq);  // [row][4]
    using std::integral_constant;
    using std::true_type;
    using std::false_type;

    if (wave >= 4) {
        // ---- weight waves ----------------------------------------------------------------------------------------------------
        const int ww = wave - 4, l15 = lane & 15, kk = lane >> 4, g = l15 >> 2, c4 = l15 & 3;
        // this lane's 16 bytes of a fragment: feature c4 of the quad, K's part g of four tiles
        auto lane_at = [&](int q) { return (g * 64 + kk * 16 + (q & 3) * 4 + c4) * 16; };
        bool live = true;  // behind the last layer the loads are from buffers of no bytes: they return zeros and cost no access
        auto load = [&](const uint4* w, int K, int tile, int q, int i) {  // fragment ww + 4 i of K of quad q of the weight tile
            const auto r = buffer_of(reinterpret_cast<const char*>(w) + (size_t)tile * K * 32, live && i < K >> 9 ? K * 32 : 0);
            return buffer_load16(r, lane_at(q), min(i, (K >> 9) - 1) * 16384 + ww * 4096);
        };
        uint4 wq[kMaxQ * 2], wo[4], wu[2 * kMaxI * 2], wd[6];
        // fragments [FROM, TO) of a product's, one after the other: all at once they would hold up what is handed on meanwhile (8 MB in a hand-off of 1.4 us: 2.9)
        auto pace = [&](int turns) __attribute__((always_inline)) {
            __builtin_amdgcn_sched_barrier(0);
            for (int i = 0; i < turns; ++i) __builtin_amdgcn_s_sleep(1);
            __builtin_amdgcn_sched_barrier(0);
        };
        auto load_qkv = [&](auto from, auto to, const uint4* w) __attribute__((always_inline)) {
#pragma unroll
            for (int j = decltype(from)::value; j < decltype(to)::value; ++j) {
                const int id = quad * nq + min(j >> 1, nq - 1);
                wq[j] = load(w, H, id >> 2, id, j & 1);
                pace(kPace);
            }
        };
        auto load_o = [&](const uint4* w) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                wo[i] = load(w, a.z.KO, quad >> 2, quad, i);
                pace(kPace);
            }
        };
        auto load_gu = [&](auto from, auto to, const uint4* w) __attribute__((always_inline)) {
#pragma unroll
            for (int j = decltype(from)::value; j < decltype(to)::value; ++j) {
                const int id = quad * ni + min(j >> 2, ni - 1);
                wu[j] = load(w, H, 2 * (id >> 2) + ((j >> 1) & 1), id, j & 1);
                pace(kPace);
            }
        };
        auto load_down = [&](const uint4* w) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < 6; ++i) {
                wd[i] = load(w, a.z.I, quad >> 2, quad, i);
                pace(kPace);
            }
        };
        // NQD quads' sums over this wave's fragments, KF of them at most
        auto multiply = [&](auto quads, auto frags, const auto& w, int K) __attribute__((always_inline)) {
            constexpr int NQD = decltype(quads)::value, KF = decltype(frags)::value;
            const int S = L::x_bytes(K);
            f32x4 acc[NQD][RS];
#pragma unroll
            for (int q = 0; q < NQD; ++q)
#pragma unroll
                for (int s = 0; s < RS; ++s) acc[q][s] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < KF; ++i) {
                const int kf = min(ww + 4 * i, (K >> 7) - 1);  // (the weights of a fragment past the end are zeros)
                bf16x8 xh[RS], xl[RS];
#pragma unroll
                for (int s = 0; s < RS; ++s) {
                    const char* p = smem + min(s * 4 + c4, R - 1) * S + g * 64 + kk * 16 + kf * 256;
                    xh[s] = *reinterpret_cast<const bf16x8*>(p);
                    xl[s] = *reinterpret_cast<const bf16x8*>(p + lds.lo);
                }
#pragma unroll
                for (int q = 0; q < NQD; ++q)
#pragma unroll
                    for (int s = 0; s < RS; ++s) {
                        const bf16x8 f = __builtin_bit_cast(bf16x8, w[q * KF + i]);
                        acc[q][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f, xh[s], acc[q][s], 0, 0, 0);
                        acc[q][s] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f, xl[s], acc[q][s], 0, 0, 0);
                    }
            }
            if (g == kk) {
                float4* part = reinterpret_cast<float4*>(smem + lds.part);
#pragma unroll
                for (int q = 0; q < NQD; ++q)
#pragma unroll
                    for (int s = 0; s < RS; ++s) part[(q * SR + s * 4 + c4) * kSlot + ww * 4 + g] = make_float4(acc[q][s][0], acc[q][s][1], acc[q][s][2], acc[q][s][3]);
            }
        };
        constexpr integral_constant<int, 0> c0;
        constexpr integral_constant<int, 2> c2;
        constexpr integral_constant<int, 4> c4_;
        constexpr integral_constant<int, 8> c8;
        constexpr integral_constant<int, 2 * kMaxI * 2> call;
        load_qkv(c0, c8, layers->qkv);
        load_o(layers->o);
        load_gu(c0, c2, layers->gu);
        for (int l = 0; l < a.L; ++l) {
            const layers_t w = layers + l, next = layers + min(l + 1, a.L - 1);
            live = true;
            meet();
            multiply(integral_constant<int, kMaxQ>(), c2, wq, H);
            meet();
            pace(kBehind);
            load_gu(c2, c8, w->gu);
            if (unit) meet();
            load_gu(c8, call, w->gu);
            load_down(w->down);
            if (unit) meet();
            meet();
            multiply(integral_constant<int, 1>(), c4_, wo, a.z.KO);
            meet();
            live = l + 1 < a.L;
            pace(kBehind);
            load_qkv(c0, c4_, next->qkv);
            meet();
            multiply(integral_constant<int, 2 * kMaxI>(), c2, wu, H);
            meet();
            pace(kBehind);
            load_qkv(c4_, c8, next->qkv);
            meet();
            multiply(integral_constant<int, 1>(), integral_constant<int, 6>(), wd, a.z.I);
            meet();
            pace(kBehind);
            load_o(next->o);
            load_gu(c0, c2, next->gu);
        }
        return;
    }

    // ---- row waves -----------------------------------------------------------------------------------------------------------
    // Wave 0 hands on and empties, waves 1 to 3 read: a wave's loads return behind its stores, and a store takes 2 us to be there.
    Waiting waiting{a.gave_up, a.host_gave_up, a.spins};
    const int t0 = threadIdx.x;
    // what the launch before left of its last layer
    {
        const int n_act = (int)(at.act_words / kResidentGroups), n_out = (int)(at.out_words / kResidentGroups);
        if (t0 < n_act) hand_on(a.buffer + at.act + (1 - a.set) * at.act_words + wg * n_act + t0, kResidentEmpty);
        if (t0 < n_out) hand_on(a.buffer + at.out + (1 - a.set) * at.out_words + wg * n_out + t0, kResidentEmpty);
    }
    float stream = 0.f;                     // wave 0, this lane's element of the residual stream in the first RP * 4 lanes
    if (t0 >> 2 < RP) stream = bf16_to_f32(a.embed[(size_t)a.ids[min(t0 >> 2, R - 1)] * H + quad * 4 + (t0 & 3)]);
    // ---- the attention's own state
    constexpr int HD = 128, half = 64, DC = 4, DT = 8, OS = HD / 4 + 1, QS = HD + 8;
    const auto b2 = [](const float* p) { return *reinterpret_cast<const float2*>(p); };
    const float2 cs = b2(a.cos + (size_t)pos * half + (lane & 31) * 2), sn = b2(a.sin + (size_t)pos * half + (lane & 31) * 2);
    const int new_block = rec[3];
    const uniform_ints_t table = uniform_ints(a.block_tables + (size_t)rec[1] * a.max_blocks);
    auto block_of = [&](int kt) { return table[min(kt, t_end - 1) >> 3]; };
    const int block0 = unit ? block_of(t_begin + wave) : 0;
    const int u_parts = (n_tiles + a.part_tiles - 1) / a.part_tiles;
    // ... and a row's head whose context is in parts: two dims a lane of wave 3
    const int c_row = min(wg / a.z.nh, R - 1), c_head = wg % a.z.nh;
    const int c_parts = ((uniform_ints(reinterpret_cast<const int*>(a.rows + c_row))[2] >> 5) + a.part_tiles) / a.part_tiles;
    const bool combines = a.parts > 1 && wg < R * a.z.nh && c_parts > 1;
    struct Tile { uint4 k[2 * DC], v[DT]; };
    constexpr int SQ = (RP + 3) / 4;        // a block of the stream ends with so many times four sums of squares
    constexpr int kStream = lines(RP * 4 + SQ * 4);
    const int qkv_words = RP * nq * 4, act_words = RP * ni * 4;

    // wave 0: this lane's words of what the workgroup hands on, (row, quad, feature) each: rows and places of their partial sums
    constexpr int IQ = (RP * kMaxQ * 4 + 63) / 64, IA = (RP * kMaxI * 4 + 63) / 64;
    int q_row[IQ], q_at[IQ], a_row[IA], a_at[IA];
#pragma unroll
    for (int i = 0; i < IQ; ++i) {
        const int slot = (lane + 64 * i) >> 2;
        q_row[i] = min(slot / nq, RP - 1);
        q_at[i] = (slot % nq * SR + q_row[i]) * kSlot + (lane & 3);
    }
#pragma unroll
    for (int i = 0; i < IA; ++i) {
        const int slot = (lane + 64 * i) >> 2;
        a_row[i] = min(slot / ni, RP - 1);
        a_at[i] = (2 * (slot % ni) * SR + a_row[i]) * kSlot + (lane & 3);
    }
    for (int l = 0; l < a.L; ++l) {
        const layers_t w = layers + l;
        // every layer works its addresses out again: kept from layer to layer they are more than the registers hold
        int t = t0, lane = t0 & 63;
        asm volatile("" : "+v"(t), "+v"(lane));
        const int reader = t - 64;          // of 192
        // four words of planes into LDS
        auto lay = [&](const uint4& v, char* p) __attribute__((always_inline)) {
            *reinterpret_cast<uint2*>(p) = make_uint2(__builtin_amdgcn_perm(v.y, v.x, 0x07060302), __builtin_amdgcn_perm(v.w, v.z, 0x07060302));
            *reinterpret_cast<uint2*>(p + lds.lo) = make_uint2(__builtin_amdgcn_perm(v.y, v.x, 0x05040100), __builtin_amdgcn_perm(v.w, v.z, 0x05040100));
        };
        // units of 16 bytes, v[i] at `at` + i * step of `r`, but the last one at `at_last`; past its end they are zeros.  Many: one of them until it is there, then all
        auto read = [&](auto& v, __amdgpu_buffer_rsrc_t r, int at, int step, int at_last) __attribute__((always_inline)) {
            constexpr int NU = sizeof(v) / 16;
            if constexpr (NU > 4)
                waiting.until([&]() __attribute__((always_inline)) { return most(load_shared16(r, at, NU / 2 * step)) != kResidentEmpty; });
            waiting.until([&]() __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < NU - 1; ++i) v[i] = load_shared16(r, at, i * step);
                v[NU - 1] = load_shared16(r, at_last);
                uint32_t m = 0;
#pragma unroll
                for (int i = 0; i < NU; ++i) m = max(m, most(v[i]));
                return m != kResidentEmpty;
            });
        };
        constexpr int kNowhere = 0x7ffffff0;
        // A reader has one unit of a block, of every B-th block: what is left of the readers has none.  The stream and its rows' sums of squares: blocks of RP + SQ units
        auto read_stream = [&](const uint32_t* from) __attribute__((always_inline)) {
            constexpr int U = RP + SQ, B = 192 / U, NU = (kResidentGroups + B - 1) / B;
            const int g0 = reader / U, in = reader % U, at = (g0 * kStream + in * 4) * 4, S = L::x_bytes(H);
            const bool any = g0 < B, last = any && g0 + (NU - 1) * B < kResidentGroups;
            uint4 v[NU];
            read(v, buffer_of(from, kStream * kResidentGroups * 4), any ? at : 0, B * kStream * 4, last ? at + (NU - 1) * B * kStream * 4 : kNowhere);
            float4 sq = make_float4(0.f, 0.f, 0.f, 0.f);
            if (in < RP && any) {
                char* const p = smem + in * S + g0 * 8;
#pragma unroll
                for (int i = 0; i < NU - 1; ++i) lay(v[i], p + i * B * 8);
                if (last) lay(v[NU - 1], p + (NU - 1) * B * 8);
            } else if (any) {
#pragma unroll
                for (int i = 0; i < NU; ++i) {  // (a last one that is not there is zeros)
                    const float4 f = __builtin_bit_cast(float4, v[i]);
                    sq.x += f.x; sq.y += f.y; sq.z += f.z; sq.w += f.w;
                }
            }
#pragma unroll
            for (int r = 0; r < RP; ++r) {
                const float own = (r & 3) == 0 ? sq.x : (r & 3) == 1 ? sq.y : (r & 3) == 2 ? sq.z : sq.w;
                const float sum = wave_sum_uniform(SQ == 1 || in == RP + r / 4 ? own : 0.f);
                if (lane == 0) ssq[r * 4 + wave] = sum;
            }
        };
        // the activations: blocks of RP x NI units
        auto read_act = [&](auto wide) __attribute__((always_inline)) {
            constexpr int NI = decltype(wide)::value, U = RP * NI, B = 192 / U, NU = (kResidentGroups + B - 1) / B, block = lines(U * 4), step = B * block * 4;
            const int g0 = reader / U, in = reader % U, row = in / NI, at = (g0 * block + in * 4) * 4, S = L::x_bytes(NI << 10);
            const bool last = kResidentGroups % B == 0 || g0 + (NU - 1) * B < kResidentGroups;
            uint4 v[NU];
            read(v, buffer_of(b_act, block * kResidentGroups * 4), at, step, last ? at + (NU - 1) * step : kNowhere);
            char* const p = smem + row * S + (g0 * NI + in - row * NI) * 8;
#pragma unroll
            for (int i = 0; i < NU - 1; ++i) lay(v[i], p + i * B * NI * 8);
            if (last) lay(v[NU - 1], p + (NU - 1) * B * NI * 8);
        };
        // the attention's output: R rows of ko * 256 units, 16 bytes of LDS between two rows
        auto read_ctx = [&]() __attribute__((always_inline)) {
            constexpr int NU = (kMaxO * RP * kResidentGroups + 191) / 192;
            const auto r = buffer_of(b_ctx, R * ko * 4096);
            uint4 v[NU];
            auto all = [&]() __attribute__((always_inline)) {
                uint32_t m = 0;
#pragma unroll
                for (int i = 0; i < NU; ++i) v[i] = load_shared16(r, (reader + 192 * i) * 16);  // (past the last row: zeros)
#pragma unroll
                for (int i = 0; i < NU; ++i) m = max(m, most(v[i]));
                return m != kResidentEmpty;
            };
            if constexpr (NU > 4) waiting.until([&]() __attribute__((always_inline)) { return most(load_shared16(r, (reader + 192 * (NU / 2)) * 16)) != kResidentEmpty; });
            waiting.until(all);
#pragma unroll
            for (int i = 0; i < NU; ++i) {
                const int u = reader + 192 * i, row = u >> (7 + ko);
                if (u < R * ko * 256) lay(v[i], smem + u * 8 + row * 16);
            }
        };
        // wave 0: this lane's feature of (quad q, row), a lane of the four that add up the weight waves' partial sums and then own a feature each
        const float4* const part = reinterpret_cast<const float4*>(smem + lds.part);
        auto sum_of = [&](int at) __attribute__((always_inline)) {
            float4 s = part[at];
#pragma unroll
            for (int i = 1; i < 4; ++i) {
                const float4 u = part[at + i * 4];
                s.x += u.x; s.y += u.y; s.z += u.z; s.w += u.w;
            }
            s.x = lanes4_sum(s.x); s.y = lanes4_sum(s.y); s.z = lanes4_sum(s.z); s.w = lanes4_sum(s.w);
            const float u = lane & 1 ? s.y : s.x, v = lane & 1 ? s.w : s.z;
            return lane & 2 ? v : u;
        };
        auto rinv_of = [&](int row) {
            const float4 s = *reinterpret_cast<const float4*>(ssq + row * 4);
            return 1.0f / sqrtf(((s.x + s.y) + (s.z + s.w)) * (1.0f / H) + a.eps);
        };
        // the stream on, times the next norm's weight
        auto hand_stream = [&](uint32_t* to, float weight) __attribute__((always_inline)) {
            stream += sum_of((lane >> 2) % SR * kSlot + (lane & 3));
            const float own = lanes4_sum(stream * stream), sq = __shfl(own, (lane - RP * 4) * 4);
            if (lane < RP * 4 + SQ * 4) hand_on(to + quad * kStream + lane, lane < RP * 4 ? planes_word(stream * weight) : word_of(lane < RP * 5 ? sq : 0.f));
        };
        auto empty = [&](uint32_t* from, int words) __attribute__((always_inline)) {
            for (int i = lane; i < words; i += 64) hand_on(from + i, kResidentEmpty);
        };
        const int feature = quad * 4 + (lane & 3);
        const float ln2 = w->ln2[feature], next = (l + 1 < a.L ? w[1].ln1 : a.norm)[feature];

        // ---- q, k, v
        if (l == 0) {
#pragma unroll
            for (int r = 0; r < RP; ++r) {
                const int row = min(r, R - 1);
                const uint2 e = *reinterpret_cast<const uint2*>(a.embed + (size_t)a.ids[row] * H + t * 4);
                const float4 n = *reinterpret_cast<const float4*>(w->ln1 + t * 4);
                const float x[4] = {__builtin_bit_cast(float, e.x << 16), __builtin_bit_cast(float, e.x & 0xffff0000u), __builtin_bit_cast(float, e.y << 16), __builtin_bit_cast(float, e.y & 0xffff0000u)};
                uint4 v;
                v.x = planes_word(x[0] * n.x); v.y = planes_word(x[1] * n.y); v.z = planes_word(x[2] * n.z); v.w = planes_word(x[3] * n.w);
                const float s = wave_sum_uniform((x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]));
                lay(v, smem + r * L::x_bytes(H) + t * 8);
                if (lane == 0) ssq[r * 4 + wave] = s;
            }
        } else if (wave) read_stream(b_out);
        if (wave == 0) stores_there();  // what is emptied, before anything else is handed on
        // the attention's first tile comes while the products are made
        const char* const kc = reinterpret_cast<const char*>(w->k);
        const char* const vc = reinterpret_cast<const char*>(w->v);
        // a 32-token tile, past the end of the part from a buffer of no bytes
        auto place = [&](const char* c, int kt, int block) { return buffer_of(c + (size_t)(block * a.z.kv + u_head) * (kBlockTokens * HD * 2), unit && kt < t_end ? kBlockTokens * HD * 2 : 0); };
        auto load_k = [&](int kt, int block, Tile& to) __attribute__((always_inline)) {
            const auto rk = place(kc, kt, block);
            const int k_at = (min(kt, t_end - 1) & 7) * (2 * DC * 1024);
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                to.k[2 * c] = buffer_stream16(rk, lane * 16 + c * 1024, k_at);
                to.k[2 * c + 1] = buffer_stream16(rk, lane * 16 + c * 1024, k_at + DC * 1024);
            }
        };
        auto load_v = [&](int kt, int block, Tile& to) __attribute__((always_inline)) {
            const auto rv = place(vc, kt, block);
            const int v_at = (min(kt, t_end - 1) & 7) * (DT * 1024);
#pragma unroll
            for (int d = 0; d < DT; ++d) to.v[d] = buffer_stream16(rv, lane * 16 + (d % 4) * 1024, v_at + d / 4 * 4096);
        };
        Tile tile;
        load_k(t_begin + wave, block0, tile);
        load_v(t_begin + wave, block0, tile);
        meet();
        if (wave == 0) {
            float rinv[IQ];
#pragma unroll
            for (int i = 0; i < IQ; ++i) rinv[i] = rinv_of(q_row[i]);  // while the products are made
            meet();
            uint32_t* const to = b_qkv + quad * lines(qkv_words);
#pragma unroll
            for (int i = 0; i < IQ; ++i) {
                const uint32_t v = word_of(sum_of(q_at[i]) * rinv[i]);
                if (lane + 64 * i < qkv_words) hand_on(to + lane + 64 * i, v);
            }
            empty(b_act + quad * lines(act_words), act_words);
            if (l == 0 && lane < RP) ssq[lane * 4] = 0.f;  // (from here on waves 1 to 3 have sums of squares)
        } else meet();

        // ---- attention
        if (unit) {
            const int l15 = lane & 15, grp = lane >> 4, hl = lane >> 5, hd2 = (lane & 31) * 2;
            const int items = gqa + 2, item = wave * 2 - 2 + hl;  // q heads, k head, v head: 32 lanes of a reader each
            AttnWave<HD, 1, 0> aw;
            const int last = pos >> 5;
            const bool has_new = last < t_end;  // (t_end - 1 is the row's last tile in one part only)
            // offsets, not pointers to choose between: every access stays one to LDS
            auto lds16 = [&](int byte) { return reinterpret_cast<_Float16*>(smem + byte); };
            if (wave && wave * 2 - 2 < items) {
                const int it = min(item, items - 1);
                const float2 wa = b2((item < gqa ? w->qn : w->kn) + hd2), wb = b2((item < gqa ? w->qn : w->kn) + half + hd2);
                const auto r = buffer_of(b_qkv, lines(qkv_words) * kResidentGroups * 4);
                const int head = it < gqa ? u_head * gqa + it : it == gqa ? a.z.nh + u_head : a.z.nh + a.z.kv + u_head;
                const int by_nq = nq == 1 ? 65536 : nq == 2 ? 32768 : nq == 3 ? 21846 : 16384;
                auto place_of = [&](int dim) {  // in bytes
                    const int qd = (head * HD + dim) >> 2, block = qd * by_nq >> 16;
                    return (block * lines(qkv_words) + (u_row * nq + qd - block * nq) * 4 + (dim & 3)) * 4;
                };
                const int from = place_of(hd2), from_half = place_of(half + hd2);
                uint2 xa, xb;
                const bool there = waiting.until([&]() __attribute__((always_inline)) {
                    xa = load_shared8(r, from);
                    xb = load_shared8(r, from_half);
                    return max(most(xa), most(xb)) != kResidentEmpty;
                });
                const float y[4] = {__builtin_bit_cast(float, xa.x), __builtin_bit_cast(float, xa.y), __builtin_bit_cast(float, xb.x), __builtin_bit_cast(float, xb.y)};
                float ss = row16_sum((y[0] * y[0] + y[1] * y[1]) + (y[2] * y[2] + y[3] * y[3]));
                ss += __shfl_xor(ss, 16);
                const float rinv = 1.0f / sqrtf(ss / (float)HD + a.eps);
                const float n[4] = {wa.x, wa.y, wb.x, wb.y}, c[2] = {cs.x, cs.y}, s[2] = {sn.x, sn.y};
                float z[4];  // dims hd2, hd2 + 1, half + hd2, half + hd2 + 1
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float n1 = (y[e] * rinv) * n[e], n2 = (y[2 + e] * rinv) * n[2 + e];
                    z[e] = n1 * c[e] - n2 * s[e];
                    z[2 + e] = n2 * c[e] + n1 * s[e];
                }
                if (item < gqa) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float v = z[e] * a.q_scale;
                        const _Float16 h = (_Float16)v;
                        const int to = lds.q + (item * QS + (e >> 1) * half + hd2 + (e & 1)) * 2;
                        *lds16(to) = h;
                        *lds16(to + gqa * QS * 2) = (_Float16)(v - (float)h);
                    }
                } else if (has_new && item < items && there) {
                    const bool isv = item > gqa;
                    _Float16* const to = reinterpret_cast<_Float16*>(isv ? w->v : w->k) + (size_t)(new_block * a.z.kv + u_head) * kBlockTokens * HD;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int dim = (e >> 1) * half + hd2 + (e & 1);
                        const _Float16 h = f16_sat(isv ? y[e] : z[e]);
                        to[isv ? v_packed_offset(pos & 255, dim, HD) : k_packed_offset(pos & 255, dim, HD)] = h;
                        *lds16(lds.fresh + (isv ? HD * 2 : 0) + dim * 2) = h;
                    }
                }
            }
            meet();
            const int new_tile = has_new && ((last - t_begin) & 3) == wave ? last : -1;
#pragma unroll
            for (int c = 0; c < DC; ++c) {
                const int from = lds.q + ((l15 % gqa) * QS + grp * 8) * 2 + c * 64;  // columns of no row repeat one: nothing of theirs is handed on
                aw.qh[0][c] = *reinterpret_cast<const f16x8*>(smem + from);
                aw.ql[0][c] = *reinterpret_cast<const f16x8*>(smem + from + gqa * QS * 2);
            }
            aw.my_row[0] = l15 < gqa ? u_row : -1;
            aw.my_pos[0] = pos;
            aw.start();
            // the new token into its place of a tile: K's lanes l15 == token % 16 of the token half, V's lane group and halfword
            auto patch = [&](Tile& x) __attribute__((always_inline)) {
                const int tt = pos & 31, e = (tt >> 4) * 4 + (tt & 3);
                const bool kl = l15 == (tt & 15), ka_lane = kl && tt < 16, kb_lane = kl && tt >= 16, v_lane = grp == ((tt & 15) >> 2);
#pragma unroll
                for (int c = 0; c < DC; ++c) {
                    const uint4 n = *reinterpret_cast<const uint4*>(lds16(lds.fresh) + c * 32 + grp * 8);
                    uint4 &ka = x.k[2 * c], &kb = x.k[2 * c + 1];
                    ka.x = ka_lane ? n.x : ka.x; ka.y = ka_lane ? n.y : ka.y; ka.z = ka_lane ? n.z : ka.z; ka.w = ka_lane ? n.w : ka.w;
                    kb.x = kb_lane ? n.x : kb.x; kb.y = kb_lane ? n.y : kb.y; kb.z = kb_lane ? n.z : kb.z; kb.w = kb_lane ? n.w : kb.w;
                }
                uint32_t mask[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) mask[i] = v_lane && (e >> 1) == i ? ((e & 1) ? 0xffff0000u : 0x0000ffffu) : 0u;
                const uint16_t* nv = reinterpret_cast<const uint16_t*>(smem + lds.fresh + HD * 2);
#pragma unroll
                for (int d = 0; d < DT; ++d) {
                    const uint32_t n = nv[d * 16 + l15] * 0x10001u;
                    uint4& v = x.v[d];
                    v.x = (v.x & ~mask[0]) | (n & mask[0]); v.y = (v.y & ~mask[1]) | (n & mask[1]);
                    v.z = (v.z & ~mask[2]) | (n & mask[2]); v.w = (v.w & ~mask[3]) | (n & mask[3]);
                }
            };
            const uint4 none[1] = {};
            for (int kt = t_begin + wave; kt < t_end; kt += 4) {
                if (kt == new_tile) patch(tile);
                aw.tile(kt << 5, grp, pos, tile.k, none, tile.v, none, [&] { load_k(kt + 4, block_of(kt + 4), tile); });
                load_v(kt + 4, block_of(kt + 4), tile);
            }
            float* const ml = reinterpret_cast<float*>(smem + lds.ml);  // [wave][2][16]
            f32x4* const obuf = reinterpret_cast<f32x4*>(smem + lds.obuf);
            float lsum = aw.lsum[0];
            lsum += __shfl_xor(lsum, 16);
            lsum += __shfl_xor(lsum, 32);
            if (l15 < gqa) {
                if (grp == 0) {
                    ml[(wave * 2 + 0) * 16 + l15] = lsum != 0.f ? aw.m[0] : -1e30f;  // a wave without a tile has no reference
                    ml[(wave * 2 + 1) * 16 + l15] = lsum;
                }
#pragma unroll
                for (int d = 0; d < DT; ++d) obuf[(wave * gqa + l15) * OS + d * 4 + grp] = aw.o[0][d];
            }
            meet();
            if (wave == 0)
                for (int i = lane; i < gqa * (HD / 4); i += 64) {
                    const int col = i / (HD / 4), d4 = i % (HD / 4), head = u_head * gqa + col;
                    float ms = -1e30f;
#pragma unroll
                    for (int q = 0; q < 4; ++q) ms = fmaxf(ms, ml[(q * 2 + 0) * 16 + col]);
                    float ltot = 0.f;
                    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        const float f = exp2f(ml[(q * 2 + 0) * 16 + col] - ms);
                        const f32x4 v = obuf[(q * gqa + col) * OS + d4];
                        ltot += ml[(q * 2 + 1) * 16 + col] * f;
                        acc[0] += v[0] * f; acc[1] += v[1] * f; acc[2] += v[2] * f; acc[3] += v[3] * f;
                    }
                    if (u_parts > 1) {
                        uint32_t* to = b_part + ((size_t)(u_row * a.z.nh + head) * kResidentParts + u_part) * kResidentPart;
                        hand_on16(to + d4 * 4, word_of(acc[0]), word_of(acc[1]), word_of(acc[2]), word_of(acc[3]));
                        if (d4 == 0) { hand_on(to + HD, word_of(ms)); hand_on(to + HD + 1, word_of(ltot)); }
                    } else {
                        const float inv = 1.0f / ltot;
                        hand_on16(b_ctx + (size_t)u_row * a.z.KO + head * HD + d4 * 4, planes_word(acc[0] * inv), planes_word(acc[1] * inv), planes_word(acc[2] * inv), planes_word(acc[3] * inv));
                    }
                }
        }
        if (combines && wave == 3) {
            const auto r = buffer_of(b_part + (size_t)(c_row * a.z.nh + c_head) * kResidentParts * kResidentPart, c_parts * kResidentPart * 4);
            uint2 v[kResidentParts], ml[kResidentParts];
            waiting.until([&]() __attribute__((always_inline)) {
                uint32_t m = 0;
#pragma unroll
                for (int i = 0; i < kResidentParts; ++i) {
                    v[i] = load_shared8(r, (i * kResidentPart + lane * 2) * 4);
                    ml[i] = load_shared8(r, (i * kResidentPart + HD) * 4);
                }
#pragma unroll
                for (int i = 0; i < kResidentParts; ++i) m = max(m, max(most(v[i]), most(ml[i])));
                return m != kResidentEmpty;
            });
            float ms = -1e30f, ltot = 0.f, y0 = 0.f, y1 = 0.f;
#pragma unroll
            for (int i = 0; i < kResidentParts; ++i) ms = i < c_parts ? fmaxf(ms, __builtin_bit_cast(float, ml[i].x)) : ms;
#pragma unroll
            for (int i = 0; i < kResidentParts; ++i) {  // (parts past the end are zeros)
                const float f = exp2f(fminf(__builtin_bit_cast(float, ml[i].x) - ms, 0.f));
                ltot += __builtin_bit_cast(float, ml[i].y) * f;
                y0 += __builtin_bit_cast(float, v[i].x) * f;
                y1 += __builtin_bit_cast(float, v[i].y) * f;
            }
            const float inv = 1.0f / ltot;
            hand_on8(b_ctx + (size_t)c_row * a.z.KO + c_head * HD + lane * 2, planes_word(y0 * inv), planes_word(y1 * inv));
        }

        // ---- o
        if (wave) read_ctx();
        else stores_there();
        meet();
        meet();
        if (wave == 0) {
            hand_stream(b_mid, ln2);
            empty(b_qkv + quad * lines(qkv_words), qkv_words);
            empty(b_out + quad * kStream, RP * 4 + SQ * 4);
        }

        // ---- gate, up
        if (wave) read_stream(b_mid);
        else stores_there();
        meet();
        if (wave) meet();
        else {
            float rinv[IA];
#pragma unroll
            for (int i = 0; i < IA; ++i) rinv[i] = rinv_of(a_row[i]);
            meet();
            uint32_t* const to = b_act + quad * lines(act_words);
#pragma unroll
            for (int i = 0; i < IA; ++i) {
                const float gate = sum_of(a_at[i]) * rinv[i], up = sum_of(a_at[i] + SR * kSlot) * rinv[i];
                const uint32_t v = planes_word(silu_mul(gate, up));
                if (lane + 64 * i < act_words) hand_on(to + lane + 64 * i, v);
            }
            if (unit && u_parts == 1) empty(b_ctx + (size_t)u_row * a.z.KO + u_head * gqa * HD, gqa * HD);
            if (unit && u_parts > 1)
                for (int c = 0; c < gqa; ++c) empty(b_part + ((size_t)(u_row * a.z.nh + u_head * gqa + c) * kResidentParts + u_part) * kResidentPart, HD + 2);
            if (combines) empty(b_ctx + (size_t)c_row * a.z.KO + c_head * HD, HD);
        }

        // ---- down
        if (wave) {
            if (ni == 3) read_act(integral_constant<int, 3>());
            else if (ni == 2) read_act(integral_constant<int, 2>());
            else read_act(integral_constant<int, 1>());
        }
        else stores_there();
        meet();
        meet();
        if (wave == 0) {
            hand_stream(b_out, next);
            empty(b_mid + quad * kStream, RP * 4 + SQ * 4);
        }
    }
    // the rows for the head, a workgroup each
    if (wg >= R) return;
    const auto r = buffer_of(b_out, kStream * kResidentGroups * 4);
    uint4 v;
    uint32_t sq;
    const bool there = waiting.until([&]() __attribute__((always_inline)) {
        v = load_shared16(r, (t0 * kStream + wg * 4) * 4);
        sq = load_shared4(r, (t0 * kStream + RP * 4 + wg) * 4);
        return max(most(v), sq) != kResidentEmpty;
    });
    const float sum = wave_sum_uniform(__builtin_bit_cast(float, sq));
    if (lane == 0) ssq[wave] = sum;
    meet();  // (the weight waves have ended)
    if (!there) return;
    *reinterpret_cast<uint2*>(a.xh + (size_t)wg * H + t0 * 4) = make_uint2(__builtin_amdgcn_perm(v.y, v.x, 0x07060302), __builtin_amdgcn_perm(v.w, v.z, 0x07060302));
    *reinterpret_cast<uint2*>(a.xl + (size_t)wg * H + t0 * 4) = make_uint2(__builtin_amdgcn_perm(v.y, v.x, 0x05040100), __builtin_amdgcn_perm(v.w, v.z, 0x05040100));
    if (t0 == 0) a.ssq[wg] = (ssq[0] + ssq[1]) + (ssq[2] + ssq[3]);
}

template <int RP>
hipError_t launch(const ResidentArgs& a, hipStream_t s) {
    const int bytes = Lds<RP>(std::max(std::max(a.z.KO, a.z.I), H), a.z.nh / a.z.kv).bytes;
    static std::atomic<uint64_t> done{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(resident_step_kernel<RP>), 160 * 1024, done);
    resident_step_kernel<RP><<<kResidentGroups, 512, bytes, s>>>(a);
    return hipGetLastError();
}

}  // namespace

bool resident_sizes_ok(int hidden, const ResidentSizes& z) {
    if (hidden != H || z.hd != 128 || z.kv < 1 || z.nh % z.kv || z.nh / z.kv > 4) return false;
    if (z.NQ % 1024 || z.KO % 1024 || z.I % 1024 || z.NQ < 1024 || z.KO < 1024 || z.I < 1024) return false;
    return z.NQ <= kMaxQ * 1024 && z.KO <= kMaxO * 1024 && z.I <= kMaxI * 1024 && kResidentRows * z.nh <= kResidentGroups && kResidentRows * z.kv <= kResidentGroups;
}
size_t resident_buffer_words(const ResidentSizes& z) { return places(z).words; }
hipError_t launch_resident(const ResidentArgs& a, hipStream_t s) {
    if (!resident_sizes_ok(H, a.z) || a.R < 1 || a.R > kResidentRows || a.L < 1 || a.parts < 1 || a.parts > kResidentParts || a.R * a.z.kv * a.parts > kResidentGroups || a.part_tiles < 1)
        return hipErrorInvalidValue;
    if (a.R == 1) return launch<1>(a, s);
    if (a.R == 2) return launch<2>(a, s);
    if (a.R <= 4) return launch<4>(a, s);
    return launch<8>(a, s);
}

}  // namespace nvllm
