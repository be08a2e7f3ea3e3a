// Internal host-side state shared by the translation units behind the C ABI: context, sequence / block bookkeeping, model.
#pragma once
#include <hip/hip_runtime.h>
#include <rccl/rccl.h>

#include <condition_variable>
#include <memory>
#include <mutex>
#include <string>
#include <unordered_map>
#include <vector>

#include "../../include/nvllm_amd.h"
#include "../../include/nvllm_amd_debug.h"
#include "kernels.h"
#include "latent.h"

namespace nvllm { struct ResidentLayer; }
using namespace nvllm;

// In-process loopback communicator (tests only): contexts created with the same group name by different
// host threads of ONE process exchange through host memory.  It exercises every tensor-parallel code path
// (sharded load, per-rank kernels, all-reduce placement, vocab-parallel arg-max) on a single GPU; production
// uses RCCL.
struct LoopGroup {
    std::mutex mu;
    std::condition_variable cv;
    int size = 0, arrived = 0;
    uint64_t generation = 0;
    std::vector<float> acc;
    std::vector<unsigned char> gather;
    std::vector<float*> os_data;      // one-shot all-reduce buffers of the ranks (same process, same device: plain pointers)
    std::vector<uint32_t*> os_flag;
};
struct nvllm_ctx {
    std::shared_ptr<LoopGroup> loop;
    bool null_comm = false;  // projection mode: tp_size > 1 shard shapes, every collective skipped (results meaningless)
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    int tp_rank = 0, tp_size = 1;
    ncclComm_t comm = nullptr;
    std::string err;
    // one-shot all-reduce (oneshot.hip), opt-in; empty when not set up
    bool oneshot = false;
    float* os_data = nullptr;     // [2 generations][tp][os_slot] f32, uncached device memory
    uint32_t* os_flag = nullptr;  // [2][tp]
    unsigned* os_done = nullptr;  // push kernel's workgroup counter
    int* os_err = nullptr;        // set by a wait that timed out
    int* os_agree = nullptr;      // [tp] error words gathered at the end of a step: every rank takes the same decision
    size_t os_slot = 0, os_data_bytes = 0, os_flag_bytes = 0;
    uint64_t os_calls = 0;
    OneShotPeers os_peers;
    hipEvent_t resident_ev = nullptr;  // see resident_turn: behind this context's last resident step, if recorded
    bool resident_recorded = false;
    std::vector<void*> os_ipc;    // peer mappings opened with hipIpcOpenMemHandle
};

int fail(nvllm_ctx* ctx, int code, const char* fmt, ...);
int model_fail(nvllm_model* m, int code, const char* fmt, ...);

#define HIPCHK(ctx, expr)                                                                              \
    do {                                                                                               \
        hipError_t e_ = (expr);                                                                        \
        if (e_ != hipSuccess) return fail(ctx, NVLLM_EHIP, "%s -> %s", #expr, hipGetErrorString(e_)); \
    } while (0)
#define NCCLCHK(ctx, expr)                                                                               \
    do {                                                                                                 \
        ncclResult_t r_ = (expr);                                                                        \
        if (r_ != ncclSuccess) return fail(ctx, NVLLM_ERCCL, "%s -> %s", #expr, ncclGetErrorString(r_)); \
    } while (0)

// sum over the tensor-parallel group, in place (no-op for one rank)
int comm_allreduce_sum(nvllm_ctx* ctx, float* buf, size_t n);

template <typename T>
static int dmalloc(nvllm_ctx* c, T** p, size_t count) {
    HIPCHK(c, hipMalloc((void**)p, std::max<size_t>(count * sizeof(T), 16)));
    return NVLLM_OK;
}

// activation planes in fragment order (padded to 16 rows) from this many rows on: a row-major fragment is 16 places of memory, one of them a row.
// Steps of 0.6B, row-major and packed, ms: 1 row 0.885 / 0.930, 2 0.936 / 0.965, 3 0.957 / 0.967, 4 0.974 / 0.969, 8 1.044 / 0.980,
// 15 1.166 / 0.992; a 1024-wide decoder of another design 4 rows 0.239 / 0.233, 15 0.265 / 0.232; a prompt of 15 tokens 1.323 / 1.196.
constexpr int kPackedMinRows = 4;
constexpr int kFusedMaxRows = 480;  // the fused decode path (deferred norms, row-parallel epilogues) handles up to this many rows ...
constexpr int kRowMaxRows = 128;    // ... and so many where a projection of the layer has no register-direct form; row-parallel products elsewhere
// one-shot all-reduce: messages of up to this many rows; its slots are sized for them (uncached memory on every peer).  Longer ones go
// through the communicator, in decode steps of more rows too: what the one-shot form does for those was never measured
constexpr int kOneshotMaxRows = 128;
constexpr int kMaxPending = 4;   // decode steps that may be enqueued before one is collected
constexpr int kAttnMaxParts = 64;  // split-KV partitions per sequence (partition grows with context beyond 8K)

struct LayerW {
    PackedW qkv, o, gu, down;
    float *ln1 = nullptr, *ln2 = nullptr, *qn = nullptr, *kn = nullptr;
};

struct SeqState {
    int slot = -1;
    int cached = 0;  // tokens whose K/V are in the cache
    std::vector<int> blocks;
    int released = 0;  // leading blocks given back because no window reaches them (blocks[i] = -1)
};

// Pinned blocks for the metadata of chunks (stage_kernel): the host fills the next one while the device may still read the others.
struct Staging {
    static constexpr int kSlots = 4;
    int *host = nullptr, *dev = nullptr;  // kSlots blocks of `ints`
    size_t ints = 0, used = 0;
    int slot = 0, n_runs = 0, longest = 0;
    bool busy[kSlots] = {}, recorded[kSlots] = {};
    hipEvent_t ev[kSlots] = {};
    StageArgs args;
};
int stage_alloc(nvllm_model* m, size_t ints);
void stage_release(nvllm_model* m);
int stage_begin(nvllm_model* m);                    // a block the device no longer reads
int* stage_put(nvllm_model* m, int* dst, size_t n); // room for n ints bound for dst; nullptr: the block is full
int stage_flush(nvllm_model* m, bool more);         // launches; more: the stream is not waited for before the next block is filled

struct DecoderImpl;  // decoder.h

struct nvllm_model {
    nvllm_model();
    ~nvllm_model();
    nvllm_ctx* ctx = nullptr;
    std::unique_ptr<DecoderImpl> dec;  // a decoder built from layer descriptions; nullptr: Qwen3
    nvllm_qwen3_config cfg{};
    int H = 0, hd = 0, L = 0, nh_l = 0, kv_l = 0, I_l = 0, V_l = 0, gqa = 1;
    bf16_bits* embed = nullptr;  // [V][H] row-major bf16 (gather table, replicated)
    PackedW lm_head;             // [V_l][H]
    float* norm = nullptr;
    std::vector<LayerW> layers;
    std::unordered_map<std::string, bool> loaded;
    bool finalized = false;
    float *cosv = nullptr, *sinv = nullptr;
    int rope_len = 0;

    // KV pool
    int widest_window = 0;  // > 0: no layer sees further back than this
    int num_blocks = 0, max_seqs = 0, max_blocks = 0, max_rows = 0;
    std::vector<f16_bits*> kcache, vcache;
    std::vector<uint8_t*> vlocache;  // 24-bit V (opt_kv_v_bits == 24): one residual byte per V element, else empty
    std::vector<uint8_t*> klocache;  // 24-bit K (opt_kv_k_bits == 24, only with 24-bit V): the same for K
    std::vector<int> free_blocks, free_slots;
    std::unordered_map<int64_t, SeqState> seqs;
    int* d_block_tables = nullptr;
    std::vector<int> h_block_tables;

    // step buffers
    uint32_t* d_ids = nullptr;
    int *d_pos = nullptr, *d_slot = nullptr, *d_tile_row0 = nullptr, *d_tile_nrows = nullptr, *d_tile_slot = nullptr,
        *d_last_rows = nullptr, *d_tile_order = nullptr;
    nvllm::DecodeRow* d_decode_rows = nullptr;  // Qwen3 only
    bool decode_in_order = false;               // record i is row i
    PrefillTile* d_prefill_tiles = nullptr;  // Qwen3 designs
    float *resid = nullptr, *slabs = nullptr, *qbuf = nullptr, *logits = nullptr, *d_maxval = nullptr, *red = nullptr;
    float* last_resid = nullptr;  // the residual stream of the rows the head wants, in the last layer (last_rows_alone)
    bf16_bits *xh = nullptr, *xl = nullptr, *xh2 = nullptr, *xl2 = nullptr, *ctxh = nullptr, *ctxl = nullptr;
    float *ssqA = nullptr, *ssqB = nullptr;  // deferred-norm partial sums of squares [groups][kFusedMaxRows]
    float* ssqT = nullptr;                   // the same of a prompt chunk [H / 128][max_rows]
    uint64_t* d_keys = nullptr;              // device sampling: per-row RNG keys and temperatures
    float* d_temps = nullptr;
    // The streaming GEMM's in-launch split-K combine (epilogues 1-3) is OFF by default: measured slower than slabs + a
    // consumer launch on MI355X (Qwen3-8B batch 64: 8.6 vs 6.4 ms/step; 32B TP=8 shard: 8.9 vs 6.5 ms) -- one workgroup
    // per n-group reads every slab behind an agent-scope release of all the others.  nvllm_debug_set_option turns it on.
    int opt_stream_combine = 0;
    int opt_oneshot_allreduce = 0;  // TP decode: one-shot all-reduce instead of the communicator's (set before kv_alloc; opt-in)
    int opt_kv_v_bits = 16;            // 24: V as f16 + e5m2 residual (13..14 significant bits, V bytes x1.5); read at kv_alloc
    int opt_kv_k_bits = 16;            // 24: K likewise (needs kv_v_bits = 24: K/V bytes x1.5 together); read at kv_alloc
    int opt_stage_fail = 0;            // test hook: the next N metadata launches fail before they are made
    int opt_leave_fail = 0;            // test hook: the next N steps fail when their results are to leave
    int opt_oneshot_skip_push = 0;     // test hook: this rank "forgets" its next N pushes (the give-up path of its peers' waits)
    int opt_oneshot_spins = 20000000;  // bound of the one-shot wait kernel's poll (~ seconds): a missing peer is an error code
    int opt_no_fused = 0, opt_no_xpack = 0, opt_no_rowpar = 0;  // A/B switches (nvllm_debug_set_option): force the generic paths
    int opt_no_attn_prologue = 0;  // A/B: decode q/k-norm + RoPE + KV write in their own row kernel, not in the attention prologue
    int opt_tile_fuse_qk = 1;    // QKV tile GEMM with the q/k-norm + RoPE + KV-write epilogue (head_dim 128, 256-wide blocks)
    int opt_last_rows = -1;      // last_rows_alone
    int opt_prefill_deal = -1;   // AttnArgs::deal
    int opt_latent_absorb = 0;   // prompt chunks of latent attention: 1 always absorbed, -1 expanded whenever possible, 0 by cost
    int opt_latent_wgs = 0;      // decode: workgroups the split of the visible context aims at (0: by latent size)
    int64_t latent_expanded = 0; // layer runs served by the expanded form so far
    int opt_latent_plain = 0;    // latent attention: the plain kernel instead of the matrix-core one (A/B, tests)
    // prompt tile product: smallest grid it is used for.  Its blocks beat the chunked kernel's long before they fill the 256 CUs: prompt of
    // one sequence on Qwen3-0.6B, smallest grid 192 / 128 / 64: 300 rows 3.97 / 3.93 / 3.43 ms, 512 rows 4.42 / 4.32 / 3.76, 1300 rows
    // 6.89 / 5.79 / 5.78, 2391 rows 8.65 / 7.65 / 7.65 (800 rows 4.73 / 4.35 / 4.44); four 8B layers, 257 rows 1.74 / 1.65 / 1.65
    int opt_tile_min_wgs = 64;
    // the resident decode step (resident.hip); empty where sizes, device or cache are not its own
    nvllm::ResidentLayer* d_resident_layers = nullptr;
    uint32_t* resident_buffer = nullptr;
    int* resident_gave_up = nullptr;       // device: a wait of the last launch ran out ...
    int *h_resident = nullptr, *dev_resident = nullptr;  // ... and the same in pinned memory
    int resident_set = 0;
    int resident_rest = 0;                 // after a launch that gave up: steps that stay launches
    int64_t resident_give_ups = 0;         // since kv_alloc
    bool resident_waited = false;          // the step's results are waited for before the next one is enqueued
    bool resident_ran = false;             // this step is such a launch
    int opt_resident = 1;                  // 0: never
    int opt_resident_spins = 1000000;      // turns of a wait, about a second
    int64_t resident_launches = 0;
    unsigned* tickets = nullptr;             // arrival counters of the streaming GEMM's in-launch combine (zero between launches)
    float* qkv_out = nullptr;                // complete QKV sums of the streaming GEMM (its combine reads the slabs in m->slabs)
    uint32_t* d_next = nullptr;
    float *attn_po = nullptr, *attn_pml = nullptr;  // split-KV partials [max_seqs][nh_l][kAttnMaxParts][hd] / [..][2]
    int* attn_done = nullptr;                       // [max_seqs][kv_l]: their parts that have ended, 0 between launches
    int attn_part_tiles = 4, attn_parts_max = 1, attn_waves = 4;   // this step's split geometry and waves of a workgroup (decode only)
    bool attn_ahead = false;  // ... and AttnArgs::ahead
    float* part_val = nullptr;  // fused LM-head arg-max partials [V_l/16][max_seqs]
    int* part_idx = nullptr;
    unsigned long long* argmax_scratch = nullptr;  // ticket + per-row keys of argmax_parts_kernel
    bool want_logits = false;   // this step stores the last-row logits
    bool want_ids = true;       // ... and its greedy ids are read (not where positions are scored or the device samples)
    int cur_n = 0;              // sequences of the step in flight
    struct PrefillList { int tiles = 0; bool deal = false; };
    PrefillList prefill_all, prefill_last;  // the chunk's q-tiles in d_prefill_tiles, and behind room for all of them those of the groups with a row the head wants
    int cur_max_len = 0;        // longest of them (tokens, the new ones included)
    size_t slab_floats = 0;
    static constexpr size_t kOutSlot = 1 << 20;
    static constexpr int kOutSlots = 16;
    char* pin_out = nullptr;                  // pinned: up to kOutSlots slots for logits on their way to the caller, then ids: a step's, and those of kMaxPending enqueued ones
    size_t out_ids = 0;                       // bytes of a step's ids
    int out_slots = 0;
    char* dev_out = nullptr;                  // the same for the device
    struct OutFlag { uint32_t seq; uint32_t pad[15]; };
    OutFlag *out_flag = nullptr, *dev_out_flag = nullptr;  // pinned, per slot and per ids: the last copy into it that is whole, by number
    static constexpr int kOutFlags = kOutSlots + 1 + kMaxPending;
    uint32_t out_seq[kOutFlags] = {};                    // ... the last one asked for
    unsigned* out_done = nullptr;                          // device, per slot: workgroups of a copy that have finished, 0 between copies
    Staging stage;
    std::vector<int> table_news;  // entries of h_block_tables the device does not have yet
    int64_t table_copies = 0;     // whole tables sent because the pinned block had no room for them
    float *tap_h = nullptr, *tap_res = nullptr;
    bool taps = false;
    int tap_rows = 0;

    // last step (for nvllm_decode_next / byte accounting)
    std::vector<int64_t> last_ids;
    std::vector<int> last_lens;
    int64_t last_bytes = 0;
    bool decode_resident = false;  // device metadata describes a pure-decode batch == last_ids
    // pipelined decode (nvllm_decode_enqueue / _collect)
    std::vector<int> pending;
    int pend_next = 0;

    // diagnostic build (-DNVLLM_STAMPS): in-kernel time stamps of every launch of the fused decode path
    unsigned long long* stamps = nullptr;
    bool stamps_on = false;
    int stamp_launch = 0;
    int64_t tile_launches = 0;  // projections run by the tile GEMM so far (tests assert the path they force was taken)
    int64_t qk_rows16_launches = 0;  // likewise: q/k norm, rotation and cache writes by 16 rows and a head
    int64_t prefill_dealt_launches = 0; // ... prompt attention with a q-tile to a workgroup
    int64_t prefill_dealt_tiles = 0;    // ... q-tiles of those
    int64_t row_sum_launches = 0;       // ... products that add up the slabs of the one before (launch_gemm_rowsum)
    int64_t eight_wave_launches = 0; // ... decode attention on eight waves
    int64_t merged_parts_launches = 0; // ... decode attention in parts that are merged in the launch
    int64_t tiles_ahead_launches = 0; // ... with both tile sets asked for before the prologue
    int64_t scan_gate_launches = 0;  // ... step sizes of a decode step's scan by their own launch
    int64_t two_launches = 0;        // ... two products in one launch
    int64_t tile_resid_launches = 0; // ... prompt products with residual and norm preparation in their epilogue

    // per-kernel-class HIP-event timing (bench roofline leg); 0 = off
    int prof_kind = 0;
    std::vector<hipEvent_t> prof_ev;
    size_t prof_used = 0;
};

#ifdef NVLLM_STAMPS
constexpr int kStampLaunches = 160;               // launches recorded per step (fused decode path: 5 per layer)
constexpr size_t kStampStride = (size_t)1024 * 16 * 8;  // u64 per launch: [<= 1024 workgroups][16 waves][8 points]
#define STAMPS(args_, m_)                                                                                        \
    do {                                                                                                         \
        if ((m_)->stamps_on && (m_)->stamp_launch < kStampLaunches) (args_).stamps = (m_)->stamps + (size_t)((m_)->stamp_launch++) * kStampStride; \
    } while (0)
#else
#define STAMPS(args_, m_) do { } while (0)
#endif

enum { PROF_ATTN = 1, PROF_GEMM = 2, PROF_NORM = 3, PROF_QK = 4, PROF_SILU = 5, PROF_LMHEAD = 6, PROF_EMPTY = 7, PROF_RECUR = 8 };

// bracket one launch with HIP events on the library stream when its class is being profiled
#define PROF(m_, kind_, expr_)                                                           \
    do {                                                                                  \
        if ((m_)->prof_kind == (kind_)) {                                                 \
            if ((m_)->prof_used + 2 > (m_)->prof_ev.size()) {                             \
                for (int i_ = 0; i_ < 256; ++i_) {                                        \
                    hipEvent_t evn_;                                                      \
                    HIPCHK((m_)->ctx, hipEventCreate(&evn_));                              \
                    (m_)->prof_ev.push_back(evn_);                                        \
                }                                                                         \
            }                                                                             \
            HIPCHK((m_)->ctx, hipEventRecord((m_)->prof_ev[(m_)->prof_used], (m_)->ctx->stream));     \
            HIPCHK((m_)->ctx, expr_);                                                     \
            HIPCHK((m_)->ctx, hipEventRecord((m_)->prof_ev[(m_)->prof_used + 1], (m_)->ctx->stream)); \
            (m_)->prof_used += 2;                                                         \
        } else {                                                                          \
            HIPCHK((m_)->ctx, expr_);                                                     \
        }                                                                                 \
    } while (0)

// Past the last layer's mixer only the rows the head wants go on: the stream of the others is read by nothing.  Taken for prompt chunks
// (more rows than the products of few rows, whose time is their weights', handle) of which at most half is wanted; layer taps want all rows.
// Option "last_rows": 1 by this rule, 0 never, -1 (default) by this rule unless "tile_min_wgs" 1 forces the prompt product on every projection.
inline bool last_rows_alone(const nvllm_model* m, int R, int n_last) {
    const bool on = m->opt_last_rows < 0 ? m->opt_tile_min_wgs != 1 : m->opt_last_rows != 0;
    return on && R > kRowMaxRows && 2 * n_last <= R && !m->taps;
}
inline size_t last_rows_cap(const nvllm_model* m) { return std::min((size_t)m->max_seqs, (size_t)m->max_rows / 2 + 1); }

// y (f32 slabs) = x.W^T with the kernel that fits the row count (api.cpp)
bool gemm_streams(const nvllm_model* m, const PackedW& w, int R);
int gemm_slabs(nvllm_model* m, const bf16_bits* xh, const bf16_bits* xl, int ldx, const PackedW& w, float* out, int R,
               int max_split, int* n_slabs, int x_packed = 0);
uint16_t host_f32_to_bf16(float f);
