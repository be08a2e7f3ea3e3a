// Prefill GEMM for gfx950: out[M][N] = x[M][K] . W[N][K]^T with x as bf16 hi + lo planes
// (replaces candle_nn::Linear::forward on prompt chunks: src/layers/linear.rs:35-36,72-77,184-198 via
//  src/models/qwen3.rs:205 (QKV), :278 (o_proj), :324-326 (gate/up + SiluAndMul, down)).
//
// MFMA-bound shape (hundreds to thousands of rows), so the design is about operand reuse and keeping the matrix
// pipe fed, not about HBM:
//   * one workgroup = 256 rows x 32*NTW features, 8 waves as 4 (rows) x 2 (features): a wave owns 64 rows x 16*NTW
//     features = 4 x NTW accumulator tiles (128 registers at NTW = 8), two waves per SIMD;
//   * BOTH operands are already in MFMA fragment order in HBM (W: PackedW; x: xpack_off planes written by the
//     producing kernel), so every stage is plain 1 KiB LDS-DMA wave-copies into a lane-linear image: no swizzle,
//     no ds_write, no bank conflicts, and each W fragment read from LDS feeds 8 MFMAs (4 row tiles x hi/lo), each
//     x fragment NTW;
//   * K advances one 32-deep k-tile per stage through a ring of three LDS stages: the DMA of stage s+2 is issued
//     right after the barrier that opens stage s, so it has a whole stage of MFMAs (64 per wave) to land; ONE
//     barrier per stage.  Inside a stage the fragments of the next sub-step (and, in the last one, the first
//     fragments of stage s+1, which the opening barrier already published) are read while the current MFMAs run.
//   * the blocks of an XCD (blockIdx % 8) are a run of an order that goes through groups of `band` row blocks feature block by feature
//     block: an eighth of the blocks to each XCD, rounded up, the last ones what is left; a run is about as many bytes of x as of W, for
//     the operand re-reads to hit that XCD's L2.  Dealing whole row blocks to XCDs instead gave two of them twice the work wherever the row blocks are not a
//     multiple of 8: 2391 rows, 10 x 24 blocks of gate/up, 91 -> 51 us; 4096 rows, where the runs are only squarer, 79 -> 75.
// MODE 0: f32 [M][N].  MODE 2: W is the gate/up matrix interleaved in 16-row tiles; the epilogue writes
// silu(gate)*up as hi/lo planes [M][N/2] (row-major or xpack_off order) -- SiluAndMul, activation.rs:13-18.
// MODE 4, 8: squared ReLU, exact GELU of every feature as hi/lo planes [M][N].
// MODE 5, 7, 6: every row block belongs to a group with weights of its own (routed experts): post relu2(pre x.W^T) as planes, post silu(g) u
// of interleaved gate / up features as planes, plain f32.
// MODE 3 (NTW = 8, head_dim 128): W is the fused QKV matrix, so a wave's 64 rows x 128 features are 64 tokens of ONE
// head and the epilogue is the whole of qwen3.rs:208-234 on registers: RMS norm over the head (q_norm / k_norm BEFORE
// RoPE), half-split RoPE (rotary_embedding.rs:82-107: features d and d+64 sit in the same lane, accumulators j and j+4),
// then q (scaled) to the f32 q buffer, K and V as f16 into the paged cache in their fragment orders.  No f32 QKV
// round trip through HBM and no separate row kernel.
// RT 3, 2: blocks of 192 and 128 rows of it (tile_qkv_rows).  MODE 9: the same into a 24-bit cache, the residual bytes beside the f16 values: 4096 rows of a 0.6B layer, the f32 product 60 us and the row
// kernel 31, now 75 in one.
#include <algorithm>
#include <cmath>

#include "device_common.h"
#include "kernels.h"

namespace nvllm {

struct TileArgs {
    const uint4* xh = nullptr;  // packed planes [ceil(M/16)][KT][64] uint4
    const uint4* xl = nullptr;
    const uint4* wp = nullptr;  // [N/16][KT][64] uint4
    float* out = nullptr;       // MODE 0
    uint16_t* act_hi = nullptr; // MODE 2, 4
    uint16_t* act_lo = nullptr;
    int act_packed = 0;
    GluSpec glu;                // MODE 2
    RowNorm rn;                 // MODE 2: deferred input norm (MODE 3, 9: q.rn)
    int M = 0, N = 0, KT = 0;
    int kts = 0;                // k-tiles per K split (blockIdx.y); split y writes slab out + y*M*N (MODE 0 only)
    int MB = 0, NB = 0;         // row blocks, feature blocks
    int map = 0;                // GROUPS: 0: id -> (nb fastest); 1: blocks of one XCD share rows; 2: share features
    int band = 1;               // else: row blocks of a group
    QkvArgs q;                  // MODE 3
    TileGroups g;               // MODE 5, 6
#ifdef NVLLM_STAMPS
    unsigned long long* stamps = nullptr;  // diagnostic build: [workgroup][16 waves][8 points] of s_memrealtime
#endif
};

#ifdef NVLLM_STAMPS
// diagnostic build only: the next tile launches record their stamps here, one kStride block per launch (tools/stamp_tile_gemm.py)
static unsigned long long* g_tile_stamps = nullptr;
static int g_tile_stamp_launch = 0, g_tile_stamp_max = 0;
void tile_gemm_stamps_arm(unsigned long long* base, int max_launches) { g_tile_stamps = base; g_tile_stamp_launch = 0; g_tile_stamp_max = max_launches; }
int tile_gemm_stamps_count() { return g_tile_stamp_launch; }
#endif

// WN = waves along the features (2: 256 rows x 32*NTW features; 4: 128 rows x 64*NTW features -- the narrow-output shape,
// N = hidden size, where 256-row tiles cannot fill the chip)
// RT = row tiles (16 rows) of a wave: 4, or 3 and 2 where blocks of 192 or 128 rows fill the chip better (gemm_tile_rows_kernel)
template <int NTW, int WN, int MODE, int RT>
__device__ __forceinline__ void tile_body(const TileArgs& a) {
    constexpr bool GROUPS = MODE == 5 || MODE == 6 || MODE == 7, GATHER = MODE == 5 || MODE == 7;
    constexpr bool QKV = MODE == 3 || MODE == 9, LO = MODE == 9;  // LO: a 24-bit cache
    constexpr int WM = 8 / WN;             // waves along the rows, RT row tiles each
    constexpr int WR = 16 * RT, XT = WM * RT;  // rows per wave; row tiles per workgroup
    constexpr int FRW = WN * NTW;          // 1 KiB fragments per stage: W ...
    constexpr int FR = FRW + 2 * XT;       // ... then [plane][row tile] of x
    constexpr int NI = (FR + 7) / 8;       // DMA wave-copies per wave per stage
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    uint4* lds = reinterpret_cast<uint4*>(smem_raw);
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // uniform: DMA sources / LDS targets stay scalar
    const int l15 = lane & 15, grp = lane >> 4;
    const int wm = wave / WN, wn = wave % WN;
    const int KT = a.kts;                  // stages of this workgroup
    const int kt0 = blockIdx.y * a.kts;

    // workgroup -> (row block, feature block); blockIdx % 8 labels the workgroups that land on one XCD
    int mb, nb;
    {
        const int id = blockIdx.x, xcd = id & 7, slot = id >> 3;
        if constexpr (!GROUPS) {
            const int b = xcd * ((int)gridDim.x >> 3) + slot;
            if (b >= a.MB * a.NB) return;  // whole workgroup, before any barrier
            const int group = b / (a.band * a.NB), r = b - group * a.band * a.NB, high = min(a.band, a.MB - group * a.band);
            nb = r / high;
            mb = group * a.band + r - nb * high;
        } else if (a.map == 1) { nb = slot % a.NB; mb = (slot / a.NB) * 8 + xcd; }
        else if (a.map == 2) { mb = slot % a.MB; nb = (slot / a.MB) * 8 + xcd; }
        else { nb = id % a.NB; mb = id / a.NB; }
        if (mb >= a.MB || nb >= a.NB) return;  // whole workgroup, before any barrier
    }
    const int mtiles = (a.M + 15) >> 4;
    const uint4* wbase = a.wp;
    if constexpr (GROUPS) {
        const int g = a.g.tile_group[mb * (WM * WR) / a.g.align];
        if (g < 0) return;  // whole workgroup, before any barrier
        wbase += (size_t)g * a.g.w_group;
    }
    NVLLM_STAMP(a, 0);
    // deferred input norm: 1 / rms of the block's rows, behind the ring (the K loop's barriers publish it)
    [[maybe_unused]] float* rinv = reinterpret_cast<float*>(smem_raw + 3 * FR * 1024);
    [[maybe_unused]] const RowNorm& rn = QKV ? a.q.rn : a.rn;
    if constexpr (QKV || MODE == 2) {
        if (rn.ssq && (int)threadIdx.x < WM * WR) {
            const int row = min(mb * (WM * WR) + (int)threadIdx.x, a.M - 1);
            float t = 0.f;
            for (int g = 0; g < rn.groups; g += 8) {
                float v[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] = rn.ssq[(size_t)min(g + i, rn.groups - 1) * rn.stride + row];
#pragma unroll
                for (int i = 0; i < 8; ++i) t += g + i < rn.groups ? v[i] : 0.f;
            }
            rinv[threadIdx.x] = 1.0f / sqrtf(t * rn.inv_h + rn.eps);
        }
    }
    [[maybe_unused]] auto rinv_of = [&](int local) { return rn.ssq ? rinv[local] : 1.0f; };
    // MODE 3: position and cache block of this lane's four tokens, fetched NOW (two dependent loads each) so that they
    // land under the K loop; in the epilogue they were 8 us of latency chain per workgroup (stamps)
    [[maybe_unused]] int e_pos[RT], e_blk[RT], e_slot0 = 0;
    [[maybe_unused]] bool e_one_seq = true;  // this lane's four tokens belong to one sequence
    if constexpr (QKV) {
#pragma unroll
        for (int b = 0; b < RT; ++b) {
            const int rowc = min(mb * (WM * WR) + wm * WR + b * 16 + l15, a.M - 1);
            const int sl = a.q.slot[rowc];
            if (b == 0) e_slot0 = sl;
            e_one_seq = e_one_seq && sl == e_slot0;
            e_pos[b] = a.q.pos[rowc];
            e_blk[b] = a.q.block_tables[(size_t)sl * a.q.max_blocks + (e_pos[b] >> 8)];
        }
    }

    // DMA sources of this wave's copies at k-tile 0, without the lane part (advance: 64 uint4 per k-tile).  Row tiles
    // past the end are clamped to the last one: their products land in columns of D that are never stored.
    const uint4* src[NI];
    [[maybe_unused]] uint32_t voff[NI], kstep[NI];  // GATHER: x is row-major and its rows are gathered: lane part, uint4 per k-tile
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int f = min(wave + 8 * i, FR - 1);
        if constexpr (GATHER) {
            voff[i] = lane;
            kstep[i] = 64;
            if (f >= FRW) {
                const int g = f - FRW, row = a.g.src[mb * (WM * WR) + (g % XT) * 16 + l15];
                src[i] = g >= XT ? a.xl : a.xh;
                voff[i] = (uint32_t)min(max(row, 0), a.g.x_rows - 1) * (uint32_t)(a.KT * 4) + grp;  // padding: any row, its factors are 0
                kstep[i] = 4;
                continue;
            }
        }
        if (f < FRW) {
            // MODE 3: the block's two heads are nb and NB + nb, not neighbours: a V head (whose epilogue is scattered
            // 2-byte cache stores) then always shares its workgroup with a q head, and the V tail spreads over twice the CUs
            const int ntile = QKV ? (f < NTW ? nb : a.NB + nb) * NTW + f % NTW : nb * FRW + f;
            src[i] = wbase + ((size_t)ntile * a.KT + kt0) * 64;
        } else {
            const int g = f - FRW, plane = g / XT, mt = min(mb * XT + (g % XT), mtiles - 1);
            src[i] = (plane ? a.xl : a.xh) + ((size_t)mt * a.KT + kt0) * 64;
        }
    }
    // k-tile s (clamped: the two issues past the end re-fetch the last k-tile into a stage nobody reads, so the
    // stage body has no branch) -> LDS stage `buf`
    auto issue_part = [&](int s, int buf, int i0, int i1) {  // copies i0 .. i1 - 1 of the stage
        const size_t koff = (size_t)min(s, KT - 1) * 64;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            if (i < i0 || i >= i1) continue;
            const int f = wave + 8 * i;
            if constexpr (GATHER) {
                if (FR % 8 == 0 || f < FR)
                    __builtin_amdgcn_global_load_lds((gptr_t)(src[i] + (size_t)min(s, KT - 1) * kstep[i] + voff[i]), (lptr_t)(lds + (size_t)(buf * FR + f) * 64), 16, 0, 0);
            } else if (FR % 8 == 0 || f < FR)
                __builtin_amdgcn_global_load_lds((gptr_t)(src[i] + koff + lane), (lptr_t)(lds + (size_t)(buf * FR + f) * 64), 16, 0, 0);
        }
    };
    auto issue = [&](int s, int buf) { issue_part(s, buf, 0, NI); };
    // LDS byte addresses this lane reads in the three stages: W fragments of this wave's features, x fragments of its
    // rows.  The fragment reads are inline asm with hand-counted lgkmcnt waits: left to hipcc (ROCm 7.2) every wait in
    // this loop came out as lgkmcnt(0), i.e. each sub-step also waited for the reads it had just issued for the next one.
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lptr_t)smem_raw;
    uint32_t w_cur = lds0 + (uint32_t)((wn * NTW) * 64 + lane) * 16;
    uint32_t x_cur = lds0 + (uint32_t)((FRW + wm * RT) * 64 + lane) * 16;
    uint32_t w_nxt = w_cur + FR * 1024, x_nxt = x_cur + FR * 1024, w_fre = w_cur + 2 * FR * 1024, x_fre = x_cur + 2 * FR * 1024;
    int fre = 2, cur_i = 0, nxt_i = 1;  // stage indices (scalar) for the DMA targets
#define NVLLM_LDSR(DST_, ADDR_, OFF_) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(DST_) : "v"(ADDR_), "n"(OFF_))
#define NVLLM_WF(DST_, P_, J_) NVLLM_LDSR(DST_, P_, (J_) * 1024)
#define NVLLM_XF(DST_, P_, PL_, MT_) NVLLM_LDSR(DST_, P_, ((PL_) * XT + (MT_)) * 1024)
#define NVLLM_LGKM(N_) asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N_) : "memory")

    f32x4 acc[NTW][RT];
#pragma unroll
    for (int j = 0; j < NTW; ++j)
#pragma unroll
        for (int b = 0; b < RT; ++b) acc[j][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    // every wave waits for its own DMA, then the barrier publishes all of them (and says: the stage read two
    // barriers ago is free).  One asm statement: the compiler can neither split it nor move LDS reads across it.
    auto publish = [&]() { asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); };

    if constexpr (NTW == 4) {
        // 128 x 256 blocks are bound by LDS (1024 cycles a stage, as many as their products), and their sub-steps of eight products are too
        // short to hide its reads: their accumulators leave registers for two whole sets of fragments, so the next stage's are read under
        // this stage's products and a stage waits once, at its barrier; its slot is free from the start, and copies go two stages ahead
        // (slot s % 3 takes stage s + 3).  6.9 k tokens of a 1024-wide decoder, o and down 39.8 -> 35.2 us, 800 of 0.6B, gate/up 30.9 -> 28.0.
        // 256 x 192 blocks, bound by their products, lost (gate/up of 4096 rows 76.6 -> 80.4, 8B q/k/v 312 -> 322).
        static_assert(NTW != 4 || RT == 4, "");
        constexpr int VM = FR / 8;  // copies of a wave in a stage, at least: those of the stage after next stay in flight
        bf16x8 WA[NTW], HA[4], LA[4], WB[NTW], HB[4], LB[4];
#define NVLLM_RD_SET(W_, H_, L_, WP_, XP_)                                                                   \
    do {                                                                                                     \
        _Pragma("unroll") for (int j = 0; j < NTW; ++j) NVLLM_WF(W_[j], WP_, j);                             \
        _Pragma("unroll") for (int b = 0; b < RT; ++b) { NVLLM_XF(H_[b], XP_, 0, b); NVLLM_XF(L_[b], XP_, 1, b); } \
    } while (0)
// the set's reads have arrived and the next stage's copies of every wave; the empty statements tie the registers to the wait
#define NVLLM_SET_READY(W_, H_, L_, VM_)                                                                     \
    do {                                                                                                     \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(VM_) : "memory");                  \
        _Pragma("unroll") for (int j = 0; j < NTW; ++j) asm volatile("" : "+v"(W_[j]));                      \
        _Pragma("unroll") for (int b = 0; b < RT; ++b) { asm volatile("" : "+v"(H_[b])); asm volatile("" : "+v"(L_[b])); } \
    } while (0)
#define NVLLM_MM(W_, X_, B_)                                                                                 \
    do {                                                                                                     \
        _Pragma("unroll") for (int j = 0; j < NTW; ++j)                                                      \
            acc[j][B_] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W_[j], X_, acc[j][B_], 0, 0, 0);            \
    } while (0)
#define NVLLM_TILE_STAGE(W_, H_, L_, WN_, HN_, LN_, S_)                                                      \
    do {                                                                                                     \
        NVLLM_SET_READY(W_, H_, L_, VM);                                                                     \
        NVLLM_RD_SET(WN_, HN_, LN_, w_nxt, x_nxt);                                                           \
        __builtin_amdgcn_sched_barrier(0);                                                                   \
        _Pragma("unroll") for (int b = 0; b < RT; ++b) {                                                      \
            NVLLM_MM(W_, H_[b], b);                                                                          \
            NVLLM_MM(W_, L_[b], b);                                                                          \
            __builtin_amdgcn_sched_barrier(0);                                                               \
            issue_part((S_) + 3, cur_i, b * NI / RT, (b + 1) * NI / RT);                                       \
            __builtin_amdgcn_sched_barrier(0);                                                               \
        }                                                                                                    \
        { const uint32_t t_ = w_cur; w_cur = w_nxt; w_nxt = w_fre; w_fre = t_; }                             \
        { const uint32_t t_ = x_cur; x_cur = x_nxt; x_nxt = x_fre; x_fre = t_; }                             \
        { const int t_ = cur_i; cur_i = nxt_i; nxt_i = fre; fre = t_; }                                      \
    } while (0)
        issue(0, 0);
        issue(1, 1);
        issue(2, 2);
        asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * VM) : "memory");
        NVLLM_STAMP(a, 1);
        NVLLM_RD_SET(WA, HA, LA, w_cur, x_cur);
        for (int s = 0; s < KT; s += 2) {  // KT is even (host)
            NVLLM_TILE_STAGE(WA, HA, LA, WB, HB, LB, s);
            NVLLM_TILE_STAGE(WB, HB, LB, WA, HA, LA, s + 1);
        }
        NVLLM_SET_READY(WA, HA, LA, 0);  // the reads and copies past the end
#undef NVLLM_TILE_STAGE
#undef NVLLM_MM
#undef NVLLM_SET_READY
#undef NVLLM_RD_SET
    } else {
    issue(0, 0);
    issue(1, 1);
    publish();
    NVLLM_STAMP(a, 1);
    bf16x8 WA[NTW], WB[NTW], xh0, xl0, xh1, xl1;
#pragma unroll
    for (int j = 0; j < NTW; ++j) NVLLM_WF(WA[j], w_cur, j);
    NVLLM_XF(xh0, x_cur, 0, 0);
    NVLLM_XF(xl0, x_cur, 1, 0);

#define NVLLM_SB __builtin_amdgcn_sched_barrier(0)
#define NVLLM_TILE_MFMA_HALF(W_, X_, MT_)                                                                    \
    do {                                                                                                     \
        _Pragma("unroll") for (int j = 0; j < NTW; ++j)                                                      \
            acc[j][MT_] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W_[j], X_, acc[j][MT_], 0, 0, 0);          \
    } while (0)
    // One stage = k-tile s: Wc (registers) x the four row tiles of this wave; Wn <- W fragments of stage s+1.
    // Each sub-step: issue the reads of the NEXT sub-step, wait until only those are outstanding (LDS returns in
    // order), run this sub-step's 2*NTW MFMAs; the sched_barriers keep the MFMAs on their side of the waits.
    // The DMA of stage s+2 is issued between the hi and lo MFMA groups of the first sub-step (its scalar address
    // arithmetic issues in the shadow of the MFMAs instead of between the barrier and the first MFMA).
    constexpr int W1 = NTW / 3, W2 = 2 * NTW / 3;
#define NVLLM_TILE_STAGE(Wc_, Wn_, S_)                                                                       \
    do {                                                                                                     \
        publish();                                                                                           \
        NVLLM_XF(xh1, x_cur, 0, 1); NVLLM_XF(xl1, x_cur, 1, 1);                                              \
        _Pragma("unroll") for (int j = 0; j < W1; ++j) NVLLM_WF(Wn_[j], w_nxt, j);                           \
        NVLLM_LGKM(2 + W1);                                                                                  \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_MFMA_HALF(Wc_, xh0, 0);                                                                   \
        issue((S_) + 2, fre);                                                                                \
        NVLLM_TILE_MFMA_HALF(Wc_, xl0, 0);                                                                   \
        NVLLM_SB;                                                                                            \
        NVLLM_XF(xh0, x_cur, 0, 2); NVLLM_XF(xl0, x_cur, 1, 2);                                              \
        _Pragma("unroll") for (int j = W1; j < W2; ++j) NVLLM_WF(Wn_[j], w_nxt, j);                          \
        NVLLM_LGKM(2 + W2 - W1);                                                                             \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_MFMA_HALF(Wc_, xh1, 1); NVLLM_TILE_MFMA_HALF(Wc_, xl1, 1);                                \
        NVLLM_SB;                                                                                            \
        NVLLM_XF(xh1, x_cur, 0, 3); NVLLM_XF(xl1, x_cur, 1, 3);                                              \
        _Pragma("unroll") for (int j = W2; j < NTW; ++j) NVLLM_WF(Wn_[j], w_nxt, j);                         \
        NVLLM_LGKM(2 + NTW - W2);                                                                            \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_MFMA_HALF(Wc_, xh0, 2); NVLLM_TILE_MFMA_HALF(Wc_, xl0, 2);                                \
        NVLLM_SB;                                                                                            \
        NVLLM_XF(xh0, x_nxt, 0, 0); NVLLM_XF(xl0, x_nxt, 1, 0);                                              \
        NVLLM_LGKM(2);                                                                                       \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_MFMA_HALF(Wc_, xh1, 3); NVLLM_TILE_MFMA_HALF(Wc_, xl1, 3);                                \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_NEXT;                                                                                     \
    } while (0)
#define NVLLM_TILE_NEXT                                                                                      \
    do {                                                                                                     \
        { const uint32_t t_ = w_cur; w_cur = w_nxt; w_nxt = w_fre; w_fre = t_; }                             \
        { const uint32_t t_ = x_cur; x_cur = x_nxt; x_nxt = x_fre; x_fre = t_; }                             \
        { const int t_ = cur_i; cur_i = nxt_i; nxt_i = fre; fre = t_; }                                      \
    } while (0)

// Three or two row tiles: the registers of the first change from stage to stage
#define NVLLM_TILE_STAGE3(Wc_, Wn_, HA_, LA_, HB_, LB_, S_)                                                  \
    do {                                                                                                     \
        publish();                                                                                           \
        NVLLM_XF(HB_, x_cur, 0, 1); NVLLM_XF(LB_, x_cur, 1, 1);                                              \
        _Pragma("unroll") for (int j = 0; j < W1; ++j) NVLLM_WF(Wn_[j], w_nxt, j);                           \
        NVLLM_LGKM(2 + W1);                                                                                  \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_MFMA_HALF(Wc_, HA_, 0);                                                                   \
        issue((S_) + 2, fre);                                                                                \
        NVLLM_TILE_MFMA_HALF(Wc_, LA_, 0);                                                                   \
        NVLLM_SB;                                                                                            \
        NVLLM_XF(HA_, x_cur, 0, 2); NVLLM_XF(LA_, x_cur, 1, 2);                                              \
        _Pragma("unroll") for (int j = W1; j < W2; ++j) NVLLM_WF(Wn_[j], w_nxt, j);                          \
        NVLLM_LGKM(2 + W2 - W1);                                                                             \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_MFMA_HALF(Wc_, HB_, 1); NVLLM_TILE_MFMA_HALF(Wc_, LB_, 1);                                \
        NVLLM_SB;                                                                                            \
        NVLLM_XF(HB_, x_nxt, 0, 0); NVLLM_XF(LB_, x_nxt, 1, 0);                                              \
        _Pragma("unroll") for (int j = W2; j < NTW; ++j) NVLLM_WF(Wn_[j], w_nxt, j);                         \
        NVLLM_LGKM(2 + NTW - W2);                                                                            \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_MFMA_HALF(Wc_, HA_, RT - 1); NVLLM_TILE_MFMA_HALF(Wc_, LA_, RT - 1);                      \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_NEXT;                                                                                     \
    } while (0)
#define NVLLM_TILE_STAGE2(Wc_, Wn_, S_)                                                                      \
    do {                                                                                                     \
        publish();                                                                                           \
        NVLLM_XF(xh1, x_cur, 0, 1); NVLLM_XF(xl1, x_cur, 1, 1);                                              \
        _Pragma("unroll") for (int j = 0; j < NTW / 2; ++j) NVLLM_WF(Wn_[j], w_nxt, j);                      \
        NVLLM_LGKM(2 + NTW / 2);                                                                             \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_MFMA_HALF(Wc_, xh0, 0);                                                                   \
        issue((S_) + 2, fre);                                                                                \
        NVLLM_TILE_MFMA_HALF(Wc_, xl0, 0);                                                                   \
        NVLLM_SB;                                                                                            \
        NVLLM_XF(xh0, x_nxt, 0, 0); NVLLM_XF(xl0, x_nxt, 1, 0);                                              \
        _Pragma("unroll") for (int j = NTW / 2; j < NTW; ++j) NVLLM_WF(Wn_[j], w_nxt, j);                    \
        NVLLM_LGKM(2 + NTW - NTW / 2);                                                                       \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_MFMA_HALF(Wc_, xh1, RT - 1); NVLLM_TILE_MFMA_HALF(Wc_, xl1, RT - 1);                      \
        NVLLM_SB;                                                                                            \
        NVLLM_TILE_NEXT;                                                                                     \
    } while (0)

    for (int s = 0; s < KT; s += 2) {  // KT is even (host)
        if constexpr (RT == 4) {
            NVLLM_TILE_STAGE(WA, WB, s);
            NVLLM_TILE_STAGE(WB, WA, s + 1);
        } else if constexpr (RT == 3) {
            NVLLM_TILE_STAGE3(WA, WB, xh0, xl0, xh1, xl1, s);
            NVLLM_TILE_STAGE3(WB, WA, xh1, xl1, xh0, xl0, s + 1);
        } else {
            NVLLM_TILE_STAGE2(WA, WB, s);
            NVLLM_TILE_STAGE2(WB, WA, s + 1);
        }
    }
#undef NVLLM_TILE_STAGE
#undef NVLLM_TILE_STAGE3
#undef NVLLM_TILE_STAGE2
#undef NVLLM_TILE_NEXT
#undef NVLLM_TILE_MFMA_HALF
#undef NVLLM_SB
    }
#undef NVLLM_WF
#undef NVLLM_XF
#undef NVLLM_LDSR
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // the two issues past the end, the last prefetch reads
#undef NVLLM_LGKM
    NVLLM_STAMP(a, 2);

    // D[feature 4*grp + r][token l15]
    const int nt0 = nb * FRW + wn * NTW;
    const int row0 = mb * (WM * WR) + wm * WR;
    if constexpr (MODE == 0 || MODE == 6) {
#pragma unroll
        for (int b = 0; b < RT; ++b) {
            const int row = row0 + b * 16 + l15;
            if (row < a.M) {
                float* o = a.out + (size_t)blockIdx.y * a.M * a.N + (size_t)row * a.N + (size_t)nt0 * 16 + grp * 4;
#pragma unroll
                for (int j = 0; j < NTW; ++j) {
                    const f32x4 v = acc[j][b];
                    *reinterpret_cast<float4*>(o + j * 16) = make_float4(v[0], v[1], v[2], v[3]);
                }
            }
        }
    } else if constexpr (QKV) {
        static_assert(!QKV || (NTW == 8 && WN == 2), "one wave tile = one 128-wide head");
        const QkvArgs& q = a.q;
        const int hh = wn == 0 ? nb : a.NB + nb;  // this wave's head: [q heads | k heads | v heads]
        const int nh = q.nh_l, kvl = q.kv.kv_l;
        // V heads: in the cache's PV fragment order TOKENS are the fast index (8 per 16-byte slot), while a lane here
        // holds 4 features of ONE token -- stored directly that is 128 two-byte stores per lane, and the V workgroups set
        // the kernel's end (stamps: epilogue 20 us against 13).  When the wave's 64 rows are consecutive positions of one
        // sequence (the usual case) the tile goes through LDS instead -- the ring is free now -- as Vt[feature][token +
        // pos % 4], so that every aligned group of four positions is one 8-byte word: 34 eight-byte stores per lane.
        asm volatile("s_barrier" ::: "memory");  // every wave has finished reading the ring (uniform: all modes-3 waves)
        bool v_done = false;
        if (hh >= nh + kvl) {
            const int nvalid = min(WR, a.M - row0);
            const int P0 = __builtin_amdgcn_readfirstlane(e_pos[0]);
            bool okl = e_one_seq && e_slot0 == __builtin_amdgcn_readfirstlane(e_slot0);
#pragma unroll
            for (int b = 0; b < RT; ++b) okl = okl && (b * 16 + l15 >= nvalid || e_pos[b] == P0 + b * 16 + l15);
            if (nvalid > 0 && __builtin_amdgcn_ballot_w64(!okl) == 0) {
                constexpr int LDV = WR + 8;  // halves per feature row: the tokens + 3 shift, padded to a multiple of 4
                _Float16* vt = reinterpret_cast<_Float16*>(smem_raw) + (size_t)wm * (128 * LDV);
                [[maybe_unused]] uint8_t* vtl = reinterpret_cast<uint8_t*>(smem_raw) + (size_t)WM * (128 * LDV) * 2 + (size_t)wm * (128 * LDV);  // residual bytes
                const int sh = P0 & 3;
#pragma unroll
                for (int b = 0; b < RT; ++b) {
                    const float ri = rinv_of(wm * WR + b * 16 + l15);
#pragma unroll
                    for (int j = 0; j < 8; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            const float y = acc[j][b][r] * ri;
                            const int at = (j * 16 + grp * 4 + r) * LDV + b * 16 + l15 + sh;
                            vt[at] = f16_sat(y);
                            if constexpr (LO) vtl[at] = residual24(y, f16_sat(y));
                        }
                }
                const int blkA = __builtin_amdgcn_readfirstlane(e_blk[0]);                       // block of position P0
                const int blkB = __builtin_amdgcn_readlane(e_blk[(nvalid - 1) >> 4], (nvalid - 1) & 15);  // ... of the last valid token
                const int kvh = hh - nh - kvl;
                for (int cq = 0; cq < WR / 4 + 1; ++cq) {
                    const int tfirst = 4 * cq - sh;  // token of the word's first column
                    if (tfirst + 3 < 0 || tfirst >= nvalid) continue;
                    const int p = P0 + tfirst;       // multiple of 4
                    const int blk = (p >> 8) == (P0 >> 8) ? blkA : blkB;
                    _Float16* vdst = reinterpret_cast<_Float16*>(q.kv.v) + (size_t)(blk * kvl + kvh) * kBlockTokens * 128;
                    [[maybe_unused]] uint8_t* vldst = LO ? q.kv.vlo + (size_t)(blk * kvl + kvh) * kBlockTokens * 128 : nullptr;
                    const int tib = p & 255, tile32 = tib >> 5, tt = tib & 31;
                    const bool full = tfirst >= 0 && tfirst + 3 < nvalid;
#pragma unroll
                    for (int e = 0; e < 2; ++e) {
                        const int d = lane * 2 + e;
                        const uint2 w = *reinterpret_cast<const uint2*>(vt + d * LDV + 4 * cq);
                        const size_t off = ((size_t)(tile32 * 8 + (d >> 4)) * 64 + ((tt & 15) >> 2) * 16 + (d & 15)) * 8 + (tt >> 4) * 4;
                        if constexpr (LO) {
                            const uint32_t wl = *reinterpret_cast<const uint32_t*>(vtl + d * LDV + 4 * cq);
                            uint8_t* to = vldst + vlo_packed_offset(tib, d, 128);  // the word's four bytes are neighbours there too
                            if (full) *reinterpret_cast<uint32_t*>(to) = wl;
                            else
#pragma unroll
                                for (int i = 0; i < 4; ++i)
                                    if (tfirst + i >= 0 && tfirst + i < nvalid) to[i] = (uint8_t)(wl >> (8 * i));
                        }
                        if (full) {
                            *reinterpret_cast<uint2*>(vdst + off) = w;
                        } else {
                            const uint16_t hv[4] = {(uint16_t)(w.x & 0xffff), (uint16_t)(w.x >> 16), (uint16_t)(w.y & 0xffff), (uint16_t)(w.y >> 16)};
#pragma unroll
                            for (int i = 0; i < 4; ++i)
                                if (tfirst + i >= 0 && tfirst + i < nvalid) reinterpret_cast<uint16_t*>(vdst)[off + i] = hv[i];
                        }
                    }
                }
                v_done = true;
            }
        }
        if (hh < nh + kvl) {
            // q / k head.  cos / sin rows of the NEXT 16 tokens are fetched while the current 16 are rotated (two register
            // sets, static indices); hoisting the norm weights as well spilled (256 registers + scratch)
            const float* w = hh < nh ? q.qn : q.kn;
            auto load_cs = [&](int pos, float4 (&cs)[4], float4 (&sn)[4]) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    cs[j] = *reinterpret_cast<const float4*>(q.cos + (size_t)pos * 64 + j * 16 + grp * 4);
                    sn[j] = *reinterpret_cast<const float4*>(q.sin + (size_t)pos * 64 + j * 16 + grp * 4);
                }
            };
            auto tokens16 = [&](auto bc, const float4 (&cs)[4], const float4 (&sn)[4]) {
                constexpr int b = decltype(bc)::value;
                const int row = row0 + b * 16 + l15;
                const int pos = e_pos[b];
                const float ri = rinv_of(wm * WR + b * 16 + l15);  // deferred input norm (1 when the planes were normalised)
                // whole-vector arithmetic on the f32x4 accumulators: hipcc pairs it into v_pk_mul / v_pk_fma (two lanes' worth
                // of flops per instruction) -- this epilogue is VALU-bound (every wave of the chip is in it at once)
                f32x4 ss4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const f32x4 x = acc[j][b] * ri;
                    acc[j][b] = x;
                    ss4 += x * x;
                }
                float ss = (ss4[0] + ss4[1]) + (ss4[2] + ss4[3]);
                ss += __shfl_xor(ss, 16);  // the four lane groups hold the other 96 features of this token
                ss += __shfl_xor(ss, 32);
                const float rinv = 1.0f / sqrtf(ss / 128.0f + q.eps);
                const float osc = hh < nh ? q.q_scale : 1.0f;  // q leaves scaled; folded into the norm weight
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const f32x4 w1 = __builtin_bit_cast(f32x4, *reinterpret_cast<const float4*>(w + j * 16 + grp * 4)) * (rinv * osc);
                    const f32x4 w2 = __builtin_bit_cast(f32x4, *reinterpret_cast<const float4*>(w + 64 + j * 16 + grp * 4)) * (rinv * osc);
                    const f32x4 c = __builtin_bit_cast(f32x4, cs[j]), sn_ = __builtin_bit_cast(f32x4, sn[j]);
                    const f32x4 n1 = acc[j][b] * w1, n2 = acc[j + 4][b] * w2;
                    acc[j][b] = n1 * c - n2 * sn_;
                    acc[j + 4][b] = n2 * c + n1 * sn_;
                }
                if (row < a.M) {
                    if (hh < nh) {
                        float* qo = q.q_out + (size_t)row * (nh * 128) + (size_t)hh * 128 + grp * 4;
#pragma unroll
                        for (int j = 0; j < 8; ++j)
                            *reinterpret_cast<float4*>(qo + j * 16) = make_float4(acc[j][b][0], acc[j][b][1], acc[j][b][2], acc[j][b][3]);
                    } else {
                        _Float16* k = reinterpret_cast<_Float16*>(q.kv.k) + (size_t)(e_blk[b] * kvl + (hh - nh)) * kBlockTokens * 128;
#pragma unroll
                        for (int j = 0; j < 8; ++j) {
                            typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
                            const f16x4 v = {f16_sat(acc[j][b][0]), f16_sat(acc[j][b][1]), f16_sat(acc[j][b][2]), f16_sat(acc[j][b][3])};
                            *reinterpret_cast<f16x4*>(k + k_packed_offset(pos & 255, j * 16 + grp * 4, 128)) = v;
                        }
                        if constexpr (LO) {
                            if (q.kv.klo) {  // four neighbouring bytes as well
                                uint8_t* kl = q.kv.klo + (size_t)(e_blk[b] * kvl + (hh - nh)) * kBlockTokens * 128;
#pragma unroll
                                for (int j = 0; j < 8; ++j) {
                                    uint32_t w4 = 0;
#pragma unroll
                                    for (int r = 0; r < 4; ++r) w4 |= (uint32_t)residual24(acc[j][b][r], f16_sat(acc[j][b][r])) << (8 * r);
                                    *reinterpret_cast<uint32_t*>(kl + klo_packed_offset(pos & 255, j * 16 + grp * 4, 128)) = w4;
                                }
                            }
                        }
                    }
                }
            };
            float4 csA[4], snA[4], csB[4], snB[4];
            load_cs(e_pos[0], csA, snA);
            load_cs(e_pos[1], csB, snB);
            tokens16(std::integral_constant<int, 0>{}, csA, snA);
            if constexpr (RT > 2) load_cs(e_pos[2], csA, snA);
            tokens16(std::integral_constant<int, 1>{}, csB, snB);
            if constexpr (RT > 3) load_cs(e_pos[3], csB, snB);
            if constexpr (RT > 2) tokens16(std::integral_constant<int, 2>{}, csA, snA);
            if constexpr (RT > 3) tokens16(std::integral_constant<int, 3>{}, csB, snB);
        } else if (!v_done) {  // V head, rows of several sequences in this wave: element-wise copy into the PV fragment order
#pragma unroll
            for (int b = 0; b < RT; ++b) {
                const int row = row0 + b * 16 + l15;
                if (row < a.M) {
                    const float ri = rinv_of(wm * WR + b * 16 + l15);
                    const int pos = e_pos[b];
                    _Float16* v = reinterpret_cast<_Float16*>(q.kv.v) + (size_t)(e_blk[b] * kvl + (hh - nh - kvl)) * kBlockTokens * 128;
#pragma unroll
                    for (int j = 0; j < 8; ++j)
#pragma unroll
                        for (int r = 0; r < 4; ++r)
                            store_v24(v, LO ? q.kv.vlo + (size_t)(e_blk[b] * kvl + (hh - nh - kvl)) * kBlockTokens * 128 : nullptr, pos & 255, j * 16 + grp * 4 + r, 128,
                                      acc[j][b][r] * ri);
                }
            }
        }
    } else if constexpr (MODE == 4 || MODE == 5 || MODE == 8) {
#pragma unroll
        for (int b = 0; b < RT; ++b) {
            const int row = row0 + b * 16 + l15;
            if (row < a.M) {
                [[maybe_unused]] float pre = 1.f, post = 1.f;
                if constexpr (MODE == 5) { pre = a.g.pre[row]; post = a.g.post[row]; }
#pragma unroll
                for (int j = 0; j < NTW; ++j) {
                    const int f0 = (nt0 + j) * 16 + grp * 4;
                    uint16_t h[4], l[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) split_bf16(MODE == 5 ? relu2(acc[j][b][r] * pre) * post : act_of<MODE == 8 ? ACT_GELU : ACT_RELU2>(acc[j][b][r]), h[r], l[r]);
                    const size_t xo = a.act_packed ? xpack_off(row, f0, a.N >> 5) : (size_t)row * a.N + f0;
                    *reinterpret_cast<uint2*>(a.act_hi + xo) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                    *reinterpret_cast<uint2*>(a.act_lo + xo) = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
                }
            }
        }
    } else {
        static_assert((MODE != 2 && MODE != 7) || NTW % 2 == 0, "gate and up tiles of a feature live in one wave");
        const int I = a.N >> 1;
#pragma unroll
        for (int b = 0; b < RT; ++b) {
            const int row = row0 + b * 16 + l15;
            if (row < a.M) {
                [[maybe_unused]] float post = 1.f;
                if constexpr (MODE == 7) post = a.g.post[row];
                [[maybe_unused]] const float ri = MODE == 2 ? rinv_of(wm * WR + b * 16 + l15) : 1.f;
#pragma unroll
                for (int pr = 0; pr < NTW / 2; ++pr) {
                    const int f0 = ((nt0 >> 1) + pr) * 16 + grp * 4;
                    uint16_t h[4], l[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float g = acc[2 * pr][b][r], u = acc[2 * pr + 1][b][r];
                        split_bf16(MODE == 7 ? silu_mul(g, u) * post : glu_mul(g * ri, u * ri, a.glu), h[r], l[r]);
                    }
                    const size_t xo = a.act_packed ? xpack_off(row, f0, I >> 5) : (size_t)row * I + f0;
                    *reinterpret_cast<uint2*>(a.act_hi + xo) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                    *reinterpret_cast<uint2*>(a.act_lo + xo) = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
                }
            }
        }
    }
    NVLLM_STAMP(a, 3);
}
template <int NTW, int WN, int MODE>
__global__ void __launch_bounds__(512) gemm_tile_kernel(TileArgs a) {
    tile_body<NTW, WN, MODE, 4>(a);
}
template <int MODE, int RT>
__global__ void __launch_bounds__(512) gemm_tile_rows_kernel(TileArgs a) {
    tile_body<8, 2, MODE, RT>(a);
}

// ---- narrow output, residual add and the next norm's preparation in the epilogue --------------------------------------------
struct TileResidArgs {
    const uint4 *xh = nullptr, *xl = nullptr, *wp = nullptr;
    const float *resid_in = nullptr, *next_w = nullptr;
    float *resid_out = nullptr, *ssq = nullptr;
    uint16_t *oh = nullptr, *ol = nullptr;
    int ssq_stride = 0, M = 0, N = 0, KT = 0, MB = 0, NB = 0, band = 1;
};
// One workgroup = 32 RT rows x 128 features x the whole K, for outputs so narrow that wider blocks would have to split K over workgroups, whose
// slabs then go to memory and back before the residual and the norm can be added.  Here the K split is inside the workgroup: waves 0 to 3 take
// the even k-tiles, 4 to 7 the odd ones, 16 RT x 64 each (at RT 4, 12 fragments read from LDS for 32 products; eight waves of 64 x 32 over the
// same block need 10 for 16 and are bound by those reads).  A stage is two k-tiles; three stages in the ring, copies two stages ahead; all
// fragments of the next stage are read under this stage's products, so a stage waits once, at its barrier.  At the end the halves of the split
// exchange row tiles, add the residual and leave the stream, the next norm's planes (weight times stream) and the rows' sums of squares.
// What it spends, by stamps at 4096 rows, K 2048 / 3072: first copies 4.3 us, loop 25.5 / 38.3, exchange 0.5, sums and stores (33 MB from every CU at once) 3.8; at 2391 rows (RT 3) 3.4, 19.1 /
// 30.2, 0.5, 3.1; at 1280 (RT 2) 2.2, 16.0 / 24.5, 0.3, 2.0.  The loop's stage of 0.80 us at RT 4 is not the LDS's 1152 cycles nor the products' 1024, both under 0.5 us; a workgroup takes in
// 48 KiB a stage, more per product than the other tile kernels' blocks.  That this is what bounds it has not been shown.
// RT: the smallest whose blocks are one round of the CUs, 4 above.  0.6B, o and down, us each at RT 1, 2, 3, 4: 1000 rows 22 / 26 / 30 / 36, 1280
// 28 / 27 / 31 / 37, 2020 34 / 29 / 32 / 39, 2391 45 / 45 / 35 / 40, 3000 48 / 47 / 36 / 40, 4000 65 / 57 / 62 / 45; with K splits over
// workgroups and a norm launch 22 + 9, 26 + 16, 26 + 17, 37 + 15 (2391) and 39 + 17 (4096).
template <int RT>
__global__ void __launch_bounds__(512) tile_resid_kernel(TileResidArgs a) {
    constexpr int XT = 2 * RT, FR1 = 8 + 2 * XT, FR = 2 * FR1;  // row tiles; 1 KiB fragments of a k-tile (8 of W, XT of each plane of x) and of a stage
    constexpr int NI = FR / 8, OWN = (RT + 1) / 2;              // copies of a wave in a stage; row tiles of a half of the K split at the end
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    uint4* lds = reinterpret_cast<uint4*>(smem_raw);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l15 = lane & 15, grp = lane >> 4;
    const int kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
    int mb, nb;
    {
        const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, b = xcd * ((int)gridDim.x >> 3) + slot;
        if (b >= a.MB * a.NB) return;  // whole workgroup, before any barrier
        const int group = b / (a.band * a.NB), r = b - group * a.band * a.NB, high = min(a.band, a.MB - group * a.band);
        nb = r / high;
        mb = group * a.band + r - nb * high;
    }
    const int NS = a.KT >> 1, mtiles = (a.M + 15) >> 4;
    // the residual of this wave's own two row tiles comes before the streams
    const int tile0 = kg * OWN, row0 = mb * (32 * RT) + wm * (16 * RT) + tile0 * 16 + l15, f0 = nb * 128 + wn * 64 + grp * 4;
    float4 r4[OWN][4];
#pragma unroll
    for (int b = 0; b < OWN; ++b)
#pragma unroll
        for (int j = 0; j < 4; ++j) r4[b][j] = *reinterpret_cast<const float4*>(a.resid_in + (size_t)min(row0 + b * 16, a.M - 1) * a.N + f0 + j * 16);
    __builtin_amdgcn_sched_barrier(0);
    const uint4* src[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) {
        const int f = wave + 8 * i, h = f / FR1, g = f % FR1;  // k-tile of the stage; W's n-tiles, then [plane][row tile] of x
        const int mt = min(mb * XT + (g - 8) % XT, mtiles - 1);  // past the end: the last row tile again, not stored
        src[i] = (g < 8 ? a.wp + (size_t)(nb * 8 + g) * a.KT * 64 : (g - 8 >= XT ? a.xl : a.xh) + (size_t)mt * a.KT * 64) + h * 64 + lane;
    }
    auto issue = [&](int s, int buf, int i0, int i1) {  // copies i0 .. i1 - 1 of stage s (past the end: the last stage again)
        const size_t koff = (size_t)min(s, NS - 1) * 128;
#pragma unroll
        for (int i = 0; i < NI; ++i)
            if (i >= i0 && i < i1) __builtin_amdgcn_global_load_lds((gptr_t)(src[i] + koff), (lptr_t)(lds + (size_t)(buf * FR + wave + 8 * i) * 64), 16, 0, 0);
    };
    const uint32_t lds0 = (uint32_t)(uintptr_t)(lptr_t)smem_raw;
    uint32_t w_at[3], x_at[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        w_at[i] = lds0 + (uint32_t)((i * FR + kg * FR1 + wn * 4) * 64 + lane) * 16;
        x_at[i] = lds0 + (uint32_t)((i * FR + kg * FR1 + 8 + wm * RT) * 64 + lane) * 16;
    }
    f32x4 acc[4][RT];
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int b = 0; b < RT; ++b) acc[j][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 WA[4], HA[RT], LA[RT], WB[4], HB[RT], LB[RT];
#define NVLLM_RD(DST_, ADDR_, OFF_) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(DST_) : "v"(ADDR_), "n"(OFF_))
#define NVLLM_RD_SET(W_, H_, L_, WP_, XP_)                                                                                   \
    do {                                                                                                                      \
        _Pragma("unroll") for (int j = 0; j < 4; ++j) NVLLM_RD(W_[j], WP_, j * 1024);                                         \
        _Pragma("unroll") for (int b = 0; b < RT; ++b) { NVLLM_RD(H_[b], XP_, b * 1024); NVLLM_RD(L_[b], XP_, (XT + b) * 1024); } \
    } while (0)
// the set's reads have arrived, this wave's copies of the stage after it too, then every wave's; the empty statements tie the registers to the wait
#define NVLLM_SET_READY(W_, H_, L_, VM_)                                                                                     \
    do {                                                                                                                      \
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(VM_) : "memory");                                   \
        _Pragma("unroll") for (int j = 0; j < 4; ++j) asm volatile("" : "+v"(W_[j]));                                         \
        _Pragma("unroll") for (int b = 0; b < RT; ++b) { asm volatile("" : "+v"(H_[b])); asm volatile("" : "+v"(L_[b])); }    \
    } while (0)
#define NVLLM_MM(W_, H_, L_, B_)                                                                                             \
    do {                                                                                                                      \
        _Pragma("unroll") for (int j = 0; j < 4; ++j) acc[j][B_] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W_[j], H_[B_], acc[j][B_], 0, 0, 0); \
        _Pragma("unroll") for (int j = 0; j < 4; ++j) acc[j][B_] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(W_[j], L_[B_], acc[j][B_], 0, 0, 0); \
        __builtin_amdgcn_sched_barrier(0);                                                                                    \
    } while (0)
#define NVLLM_STAGE(W_, H_, L_, WN_, HN_, LN_, S_)                                                                           \
    do {                                                                                                                      \
        NVLLM_SET_READY(W_, H_, L_, NI);                                                                                      \
        NVLLM_RD_SET(WN_, HN_, LN_, w_at[1], x_at[1]);                                                                        \
        __builtin_amdgcn_sched_barrier(0);                                                                                    \
        _Pragma("unroll") for (int b = 0; b < RT; ++b) {                                                                      \
            NVLLM_MM(W_, H_, L_, b);                                                                                          \
            issue((S_) + 3, cur, b * NI / RT, (b + 1) * NI / RT);                                                             \
            __builtin_amdgcn_sched_barrier(0);                                                                                \
        }                                                                                                                     \
        cur = cur == 2 ? 0 : cur + 1;                                                                                         \
        { const uint32_t t_ = w_at[0]; w_at[0] = w_at[1]; w_at[1] = w_at[2]; w_at[2] = t_; }                                  \
        { const uint32_t t_ = x_at[0]; x_at[0] = x_at[1]; x_at[1] = x_at[2]; x_at[2] = t_; }                                  \
    } while (0)
#pragma unroll
    for (int i = 0; i < 3; ++i) issue(i, i, 0, NI);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * NI) : "memory");
    NVLLM_RD_SET(WA, HA, LA, w_at[0], x_at[0]);
    int cur = 0;
    for (int s = 0; s < NS; s += 2) {  // NS is even (host)
        NVLLM_STAGE(WA, HA, LA, WB, HB, LB, s);
        NVLLM_STAGE(WB, HB, LB, WA, HA, LA, s + 1);
    }
    NVLLM_SET_READY(WA, HA, LA, 0);  // the reads and copies past the end; the ring is free
#undef NVLLM_STAGE
#undef NVLLM_MM
#undef NVLLM_SET_READY
#undef NVLLM_RD_SET
#undef NVLLM_RD
    // each half of the K split keeps its own row tiles and hands the others to its partner
    f32x4* xch = reinterpret_cast<f32x4*>(smem_raw);                             // [8 waves][OWN][4][64]
    float* red = reinterpret_cast<float*>(smem_raw + 8 * OWN * 4 * 1024);        // [wm][RT][16]
#pragma unroll
    for (int b = 0; b < OWN; ++b)
#pragma unroll
        for (int j = 0; j < 4; ++j) xch[((wave * OWN + b) * 4 + j) * 64 + lane] = kg ? acc[j][b] : acc[j][min(OWN + b, RT - 1)];
    __syncthreads();
    float ss[OWN];
#pragma unroll
    for (int b = 0; b < OWN; ++b) {
        const int row = row0 + b * 16;
        const bool mine = tile0 + b < RT;  // an odd RT: the second half has one less
        ss[b] = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const f32x4 other = xch[(((wave ^ 4) * OWN + b) * 4 + j) * 64 + lane], own = kg ? acc[j][min(OWN + b, RT - 1)] : acc[j][b];
            const f32x4 v = kg ? other + own : own + other;
            const float s0 = v[0] + r4[b][j].x, s1 = v[1] + r4[b][j].y, s2 = v[2] + r4[b][j].z, s3 = v[3] + r4[b][j].w;
            if (mine && row < a.M) {
                const float4 w4 = *reinterpret_cast<const float4*>(a.next_w + f0 + j * 16);
                *reinterpret_cast<float4*>(a.resid_out + (size_t)row * a.N + f0 + j * 16) = make_float4(s0, s1, s2, s3);
                uint16_t h[4], l[4];
                split_bf16(s0 * w4.x, h[0], l[0]); split_bf16(s1 * w4.y, h[1], l[1]); split_bf16(s2 * w4.z, h[2], l[2]); split_bf16(s3 * w4.w, h[3], l[3]);
                const size_t o = xpack_off(row, f0 + j * 16, a.N >> 5);
                *reinterpret_cast<uint2*>(a.oh + o) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                *reinterpret_cast<uint2*>(a.ol + o) = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
            }
            ss[b] += (s0 * s0 + s1 * s1) + (s2 * s2 + s3 * s3);
        }
        ss[b] += __shfl_xor(ss[b], 16);
        ss[b] += __shfl_xor(ss[b], 32);
        if (mine && wn == 1 && grp == 0) red[(wm * RT + tile0 + b) * 16 + l15] = ss[b];
    }
    __syncthreads();
    if (wn == 0 && grp == 0)
#pragma unroll
        for (int b = 0; b < OWN; ++b)
            if (tile0 + b < RT && row0 + b * 16 < a.M) a.ssq[(size_t)nb * a.ssq_stride + row0 + b * 16] = ss[b] + red[(wm * RT + tile0 + b) * 16 + l15];
}

// ---- host side -------------------------------------------------------------------------------------
// Shape of the launch for an [M][N] output: block geometry (NTW, WN) and K splits.  Candidates: 256 x 256 and 256 x 192 (WN 2), and 128 x 256
// and 128 x 128 (WN 4, NTW 4 and 2) for outputs too narrow or too short to fill the chip with bigger blocks; mode 0 may split K (f32 slabs,
// summed by the consumer like the chunked kernel's).  Cost in microseconds = chip rounds x one block's MFMA time (hi + lo planes, half the
// dense peak as the sustained rate, the narrow blocks charged for their LDS reads per MFMA: 25 %, and 100 % for 128 x 128) + the slabs'
// write and re-read when K is split.  Without 128 x 128 blocks and with them, ms: 0.6B prompts of 257 tokens 3.41 -> 3.01, 512 3.73 -> 3.39,
// 1024 5.09 -> 4.98, from 1300 on the same; four prompts of 64 to 200 tokens of a 1024-wide decoder 0.929 -> 0.858.  Charged 60 % instead
// they take over where they lose: 2391 tokens 7.62 -> 7.94, 18.7 k tokens 41.9 -> 44.8.
// ntw == 0: not covered, or fewer than min_wgs workgroups.
struct TileShape { int ntw = 0, wn = 0, ks = 1; double cost = 0; };
static TileShape tile_shape(int M, int N, int K, int mode, int min_wgs, int max_split) {
    TileShape best;
    if (M < 1 || K % 64 != 0 || K < 128 || N % 32 != 0) return best;
    const int KT = K / 32;
    const int cand[4][2] = {{8, 2}, {6, 2}, {4, 4}, {2, 4}};
    for (const auto& c : cand) {
        const int ntw = c[0], wn = c[1], cols = wn * ntw * 16, rows = (8 / wn) * 64;
        if (N % cols != 0 || (mode == 2 && ntw % 2)) continue;
        const int64_t blocks = (int64_t)((M + rows - 1) / rows) * (N / cols);
        for (int ks = 1; ks <= (mode == 0 ? max_split : 1); ks *= 2) {
            if (KT % (2 * ks) != 0 || (ks > 1 && KT / ks < 8)) continue;
            const int64_t wgs = blocks * ks;
            if (wgs < min_wgs) continue;
            const double block_us = 4.0 * rows * cols * (double)(K / ks) / (2.5e15 * 0.5 / 256) * 1e6 * (ntw == 2 ? 2.0 : wn == 4 ? 1.25 : 1.0);
            const double slab_us = ks > 1 ? 2.0 * ks * (double)M * N * 4 / 4e12 * 1e6 : 0.0;
            const double cost = (double)((wgs + 255) / 256) * block_us + slab_us;
            if (!best.ntw || cost < best.cost) best = TileShape{ntw, wn, ks, cost};
        }
    }
    return best;
}

bool tile_resid_ok(int M, int N, int K) { return M > 0 && N % 128 == 0 && N / 128 <= 64 && K % 128 == 0; }
template <int RT>
static hipError_t tile_resid_launch(TileResidArgs& a, hipStream_t s) {
    a.MB = (a.M + 32 * RT - 1) / (32 * RT);
    const int per = (a.MB * a.NB + 7) / 8;
    a.band = std::min(a.MB, std::max(1, (int)std::lround(std::sqrt(per * 128.0 / (2.0 * 32 * RT)))));
    const size_t lds = (size_t)3 * 2 * (8 + 4 * RT) * 1024;
    static std::atomic<uint64_t> lds_set{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(tile_resid_kernel<RT>), lds, lds_set);
    tile_resid_kernel<RT><<<8 * per, 512, lds, s>>>(a);
    return hipGetLastError();
}
hipError_t launch_tile_resid(const bf16_bits* xh, const bf16_bits* xl, const PackedW& w, int M, float* resid, const float* next_w, bf16_bits* oh, bf16_bits* ol, float* ssq, int ssq_stride,
                             hipStream_t s) {
    if (!tile_resid_ok(M, w.N, w.K)) return hipErrorNotSupported;
    TileResidArgs a;
    a.xh = reinterpret_cast<const uint4*>(xh); a.xl = reinterpret_cast<const uint4*>(xl); a.wp = w.data;
    a.resid_in = resid; a.resid_out = resid; a.next_w = next_w; a.oh = oh; a.ol = ol; a.ssq = ssq; a.ssq_stride = ssq_stride;
    a.M = M; a.N = w.N; a.KT = w.K / 32; a.NB = w.N / 128;
    // the shortest blocks that are one round of the CUs
    auto one_round = [&](int rt) { return (M + 32 * rt - 1) / (32 * rt) * a.NB <= 256; };
    if (one_round(1)) return tile_resid_launch<1>(a, s);
    if (one_round(2)) return tile_resid_launch<2>(a, s);
    if (one_round(3)) return tile_resid_launch<3>(a, s);
    return tile_resid_launch<4>(a, s);
}

bool gemm_tile_ok(int M, int N, int K, int mode, int min_wgs) { return tile_shape(M, N, K, mode, min_wgs, 1).ntw != 0; }
// An activation in the epilogue wants the whole K in one workgroup.  Where splitting K would fill the chip instead, the product of f32 slabs
// and a launch that sums them and applies the activation, about 5 us, can be the faster pair; by the cost above.  129 rows, N 4608, K 1024:
// 72 workgroups, 27 us; N 9216, K 2048: 50.  Decode steps of decoders with these, always the epilogue and by this rule: 129 rows 0.891 ->
// 0.870 and 0.761 -> 0.713 ms, 200 rows 1.095 -> 1.091 and 0.876 -> 0.839, 256 rows 1.275 -> 1.268 and 0.937 -> 0.905, 400 rows the same.
// min_wgs 1 (whenever the shape fits) takes the epilogue.
bool gemm_tile_act_ok(int M, int N, int K, int act, int min_wgs, int max_split) {
    const TileShape one = tile_shape(M, N, K, 4 + act, min_wgs, 1);
    if (!one.ntw || min_wgs == 1) return one.ntw != 0;
    const TileShape split = tile_shape(M, N, K, 0, min_wgs, max_split);
    return split.ks == 1 || one.cost <= split.cost + 5.0;
}
int gemm_tile_splits(int M, int N, int K, int min_wgs, int max_split) { return tile_shape(M, N, K, 0, min_wgs, max_split).ntw ? tile_shape(M, N, K, 0, min_wgs, max_split).ks : 0; }

template <int NTW, int WN, int MODE, int RT = 4>
static hipError_t tile_launch_t(TileArgs& a, int ks, hipStream_t s) {
    constexpr int rows = (8 / WN) * 16 * RT, FR = WN * NTW + 2 * (8 / WN) * RT;
    a.NB = a.N / (WN * NTW * 16);
    a.MB = (a.M + rows - 1) / rows;
    a.kts = a.KT / ks;
    int grid;
    if (!(MODE == 5 || MODE == 6 || MODE == 7)) {
        const int per = (a.MB * a.NB + 7) / 8, cols = WN * NTW * 16;
        a.band = std::min(a.MB, std::max(1, (int)std::lround(std::sqrt((double)per * cols / (2.0 * rows)))));
        grid = 8 * per;
    } else if (a.MB >= 8) { a.map = 1; grid = ((a.MB + 7) / 8) * 8 * a.NB; }
    else if (a.NB >= 8) { a.map = 2; grid = ((a.NB + 7) / 8) * 8 * a.MB; }
    else { a.map = 0; grid = a.MB * a.NB; }
    const size_t lds = (size_t)3 * FR * 1024 + (MODE == 2 || MODE == 3 || MODE == 9 ? (size_t)rows * 4 : 0);
    static std::atomic<uint64_t> lds_set{0};
    void (*kernel)(TileArgs) = nullptr;
    if constexpr (RT == 4) kernel = gemm_tile_kernel<NTW, WN, MODE>;
    else kernel = gemm_tile_rows_kernel<MODE, RT>;
    ensure_dyn_lds(reinterpret_cast<const void*>(kernel), lds, lds_set);
#ifdef NVLLM_STAMPS
    if (g_tile_stamps && g_tile_stamp_launch < g_tile_stamp_max && (size_t)grid * ks <= 1024)
        a.stamps = g_tile_stamps + (size_t)(g_tile_stamp_launch++) * ((size_t)1024 * 16 * 8);
#endif
    kernel<<<dim3(grid, ks), 512, lds, s>>>(a);
    return hipGetLastError();
}

// n_slabs (nullable): K splits the launch wrote (out = [n_slabs][M][N]); nullptr -> never split
hipError_t launch_gemm_tile(const bf16_bits* xh, const bf16_bits* xl, const PackedW& w, int M, int mode, float* out,
                            bf16_bits* act_hi, bf16_bits* act_lo, int act_packed, int min_wgs, int max_split, int* n_slabs,
                            hipStream_t s, const GluSpec& glu, const RowNorm& rn) {
    const TileShape t = tile_shape(M, w.N, w.K, mode, min_wgs, n_slabs ? max_split : 1);
    if (!t.ntw) return hipErrorNotSupported;
    if (mode == 2 && act_packed && (w.N / 2) % 32 != 0) return hipErrorNotSupported;
    if (mode >= 4 && act_packed && w.N % 32 != 0) return hipErrorNotSupported;
    TileArgs a;
    a.xh = reinterpret_cast<const uint4*>(xh); a.xl = reinterpret_cast<const uint4*>(xl); a.wp = w.data;
    if (rn.ssq && (mode != 2 || rn.row_idx)) return hipErrorNotSupported;
    a.out = out; a.act_hi = act_hi; a.act_lo = act_lo; a.act_packed = act_packed; a.glu = glu; a.rn = rn;
    a.M = M; a.N = w.N; a.KT = w.K / 32;
    if (n_slabs) *n_slabs = t.ks;
    if (mode == 0) {
        if (t.ntw == 2) return tile_launch_t<2, 4, 0>(a, t.ks, s);
        if (t.wn == 4) return tile_launch_t<4, 4, 0>(a, t.ks, s);
        return t.ntw == 8 ? tile_launch_t<8, 2, 0>(a, t.ks, s) : tile_launch_t<6, 2, 0>(a, t.ks, s);
    }
    if (mode == 2) {
        if (t.ntw == 2) return tile_launch_t<2, 4, 2>(a, 1, s);
        if (t.wn == 4) return tile_launch_t<4, 4, 2>(a, 1, s);
        return t.ntw == 8 ? tile_launch_t<8, 2, 2>(a, 1, s) : tile_launch_t<6, 2, 2>(a, 1, s);
    }
    if (mode == 4) {
        if (t.ntw == 2) return tile_launch_t<2, 4, 4>(a, 1, s);
        if (t.wn == 4) return tile_launch_t<4, 4, 4>(a, 1, s);
        return t.ntw == 8 ? tile_launch_t<8, 2, 4>(a, 1, s) : tile_launch_t<6, 2, 4>(a, 1, s);
    }
    if (mode == 4 + ACT_GELU) {
        if (t.ntw == 2) return tile_launch_t<2, 4, 8>(a, 1, s);
        if (t.wn == 4) return tile_launch_t<4, 4, 8>(a, 1, s);
        return t.ntw == 8 ? tile_launch_t<8, 2, 8>(a, 1, s) : tile_launch_t<6, 2, 8>(a, 1, s);
    }
    return hipErrorInvalidValue;
}

// Row tiles of a wave for the QKV product with its epilogue: blocks of 256 rows, or of 192 or 128 where their rounds of the chip are the cheaper ones
// (a block costs about RT + 2: what does not grow with its rows is the W it reads, its start and its epilogue); 0: no such block, f32 sums and the row kernel.
// Those may split K, and 128 rows by 256 features are short of LDS, so where blocks of 256 rows were not the best, the lower ones take over only from the workgroups
// below on.  K 1024 has no such line: tests/test_qk_rows_gpu.py has the row kernel run at up to 2040 rows, where blocks of 128 would be the better ones (83.1 -> 79.4 at 1024
// rows, 115 -> 96.3 at 2048).  With 4096 features blocks of 256 rows take over at 2049 rows; with 2048, at 4097, nothing was measured in between.
// us a layer of all products and the row kernel, one prompt of so many tokens, by the rule before (256 rows, or f32 sums) and this one:
//   0.6B (H 1024)  2391 127 / 115, 2600 130 / 119, 3072 139 / 128, 4096 the same; 24 bits 2391 132 / 120
//   H 2048         1200 144 / 133, 2048 171 / 149, 2391 200 / 185, 3000 206 / 199, 4096 the same; 1024 by blocks of 128 118 / 125
//   H 4096, 32 heads on 8  1400 345 / 323, 1800 378 / 348, 3400 609 / 555, 4096 the same; 1200 by blocks of 128 310 / 314
static int tile_qkv_rows(int M, int N, int K, int min_wgs) {
    const TileShape t = tile_shape(M, N, K, 0, min_wgs, 1);
    if (!t.ntw || N % 256) return 0;
    auto blocks = [&](int rt) { return (int64_t)((M + 64 * rt - 1) / (64 * rt)) * (N / 256); };
    auto cost = [&](int rt) { return (blocks(rt) + 255) / 256 * (rt + 2); };
    int rt = 4;
    for (int r : {3, 2}) if (cost(r) < cost(rt)) rt = r;
    if (t.ntw == 8 && t.wn == 2) return rt;
    return K <= 1024 ? 0 : K <= 2048 ? (blocks(rt) >= 160 ? rt : 0) : rt >= 3 && blocks(rt) >= 192 ? rt : 0;
}
bool gemm_tile_qkv_ok(int M, int N, int K, int hd, int min_wgs) { return hd == 128 && tile_qkv_rows(M, N, K, min_wgs) != 0; }

hipError_t launch_gemm_tile_qkv(const bf16_bits* xh, const bf16_bits* xl, const PackedW& w, int M, const QkvArgs& qa, int min_wgs,
                                hipStream_t s) {
    if (!gemm_tile_qkv_ok(M, w.N, w.K, qa.kv.hd, min_wgs) || w.N != (qa.nh_l + 2 * qa.kv.kv_l) * 128) return hipErrorNotSupported;
    if (qa.kv.klo && !qa.kv.vlo) return hipErrorInvalidValue;  // 24-bit K comes with 24-bit V only
    TileArgs a;
    a.xh = reinterpret_cast<const uint4*>(xh); a.xl = reinterpret_cast<const uint4*>(xl); a.wp = w.data;
    a.M = M; a.N = w.N; a.KT = w.K / 32; a.q = qa;
    const int rt = tile_qkv_rows(M, w.N, w.K, min_wgs);
    if (rt == 2) return qa.kv.vlo ? tile_launch_t<8, 2, 9, 2>(a, 1, s) : tile_launch_t<8, 2, 3, 2>(a, 1, s);
    if (rt == 3) return qa.kv.vlo ? tile_launch_t<8, 2, 9, 3>(a, 1, s) : tile_launch_t<8, 2, 3, 3>(a, 1, s);
    return qa.kv.vlo ? tile_launch_t<8, 2, 9>(a, 1, s) : tile_launch_t<8, 2, 3>(a, 1, s);
}

// rows of a block, features of a block: 256 x 256, 256 x 192 or 128 x 256 (few rows per group)
static TileShape group_shape(int N, int K, int align) {
    TileShape t;
    if (K % 64 || K < 128) return t;
    if (align == 128) { if (N % 256 == 0) { t.ntw = 4; t.wn = 4; } }
    else if (align == 256) { t.ntw = N % 256 == 0 ? 8 : N % 192 == 0 ? 6 : 0; t.wn = 2; }
    return t;
}
bool gemm_tile_group_ok(int N, int K, int align) { return group_shape(N, K, align).ntw != 0; }
hipError_t launch_gemm_tile_group(const bf16_bits* xh, const bf16_bits* xl, const PackedW& w, int positions, const TileGroups& g, float* out, bf16_bits* act_hi,
                                  bf16_bits* act_lo, hipStream_t s) {
    const TileShape t = group_shape(w.N, w.K, g.align);
    if (!t.ntw || positions % g.align || !g.tile_group || (act_hi && ((!g.gated && !g.pre) || !g.post || !g.src || g.x_rows < 1 || (int64_t)g.x_rows * w.K / 8 > INT32_MAX))) return hipErrorNotSupported;
    if (positions <= 0) return hipSuccess;
    TileArgs a;
    a.xh = reinterpret_cast<const uint4*>(xh); a.xl = reinterpret_cast<const uint4*>(xl); a.wp = w.data;
    a.out = out; a.act_hi = act_hi; a.act_lo = act_lo; a.act_packed = 1; a.M = positions; a.N = w.N; a.KT = w.K / 32; a.g = g;
    if (act_hi && g.gated) {
        if (t.wn == 4) return tile_launch_t<4, 4, 7>(a, 1, s);
        return t.ntw == 8 ? tile_launch_t<8, 2, 7>(a, 1, s) : tile_launch_t<6, 2, 7>(a, 1, s);
    }
    if (act_hi) {
        if (t.wn == 4) return tile_launch_t<4, 4, 5>(a, 1, s);
        return t.ntw == 8 ? tile_launch_t<8, 2, 5>(a, 1, s) : tile_launch_t<6, 2, 5>(a, 1, s);
    }
    if (t.wn == 4) return tile_launch_t<4, 4, 6>(a, 1, s);
    return t.ntw == 8 ? tile_launch_t<8, 2, 6>(a, 1, s) : tile_launch_t<6, 2, 6>(a, 1, s);
}

// row-major plane [M][K] -> xpack_off order (tests and the tuning bench; the product's producers write the order directly)
__global__ void __launch_bounds__(256) xpack_plane_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, int M, int K) {
    const int KT = K >> 5;
    const int64_t n = (int64_t)((M + 15) >> 4) * KT * 64;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) {
        const int lane = (int)(i & 63);
        const int64_t t = i >> 6;
        const int kt = (int)(t % KT), mt = (int)(t / KT);
        const int row = min(mt * 16 + (lane & 15), M - 1);
        dst[i] = src[((size_t)row * K + (size_t)kt * 32 + (lane >> 4) * 8) >> 3];
    }
}
hipError_t launch_xpack_plane(const bf16_bits* src, bf16_bits* dst, int M, int K, hipStream_t s) {
    if (K % 32 != 0 || M < 1) return hipErrorInvalidValue;
    const int64_t n = (int64_t)((M + 15) / 16) * (K / 32) * 64;
    xpack_plane_kernel<<<(int)std::min<int64_t>((n + 255) / 256, 8192), 256, 0, s>>>(reinterpret_cast<const uint4*>(src),
                                                                                      reinterpret_cast<uint4*>(dst), M, K);
    return hipGetLastError();
}

}  // namespace nvllm
