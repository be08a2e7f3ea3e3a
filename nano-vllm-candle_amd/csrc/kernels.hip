// Hand-written gfx950 (CDNA4, wave64) kernels of the Qwen3 forward path.
//
// Reference behaviour each kernel replaces is cited at the kernel.
// MFMA: v_mfma_f32_16x16x32_{bf16,f16}.  Lane l of a wave: l15 = l & 15, grp = l >> 4.
//   A frag: A[row l15][k = 8*grp + j]      B frag: B[k = 8*grp + j][col l15]      (j = 0..7)
//   C/D   : D[row 4*grp + reg][col l15]    (reg = 0..3)
#include "kernels.h"

#include <algorithm>
#include <atomic>
#include <cstdlib>

#include "attn_wave.h"
#include "device_common.h"
#include "synth_device.h"

namespace nvllm {

// ---------------------------------------------------------------------------------------------------
// weight packing / synthetic fill
// ---------------------------------------------------------------------------------------------------
// one thread per 16-byte lane slot of the destination: (dest row r, k-chunk of 8)
// ileave >= 0: destination rows are interleaved in 16-row tiles, source row r -> ((r/16)*2 + ileave)*16 + r%16
// (gate_up: tile 2t = gate features 16t.., tile 2t+1 = up features 16t.. so one wave holds both of a feature)
__device__ __forceinline__ int dest_row(int row0, int rl, int ileave) {
    return row0 + (ileave < 0 ? rl : (((rl >> 4) * 2 + ileave) << 4) + (rl & 15));
}

__global__ void __launch_bounds__(256) pack_rows_kernel(uint4* __restrict__ dst, int KT, int row0, int rows,
                                                        const uint16_t* __restrict__ src, int64_t ld, int ileave) {
    const int64_t chunks_per_row = (int64_t)KT * 4;
    const int64_t total = (int64_t)rows * chunks_per_row;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int rl = (int)(i / chunks_per_row);
        const int kc8 = (int)(i % chunks_per_row);
        const int r = dest_row(row0, rl, ileave);
        const uint4 v = *reinterpret_cast<const uint4*>(src + (int64_t)rl * ld + (int64_t)kc8 * 8);
        const int nt = r >> 4, kt = kc8 >> 2, lane = ((kc8 & 3) << 4) | (r & 15);
        dst[((int64_t)nt * KT + kt) * 64 + lane] = v;
    }
}

__global__ void __launch_bounds__(256) synth_packed_kernel(uint4* __restrict__ dst, int KT, int row0, int rows,
                                                           SynthSpec spec, int64_t src_row0, int64_t src_col0,
                                                           int64_t src_ld, int ileave) {
    const int64_t chunks_per_row = (int64_t)KT * 4;
    const int64_t total = (int64_t)rows * chunks_per_row;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int rl = (int)(i / chunks_per_row);
        const int kc8 = (int)(i % chunks_per_row);
        const int r = dest_row(row0, rl, ileave);
        const uint64_t base = (uint64_t)(src_row0 + rl) * (uint64_t)src_ld + (uint64_t)(src_col0 + (int64_t)kc8 * 8);
        // the element's hidden channel without a division: src_ld is the full tensor's row length (== spec.cols)
        const uint32_t crow = (uint32_t)(src_row0 + rl), ccol = (uint32_t)(src_col0 + (int64_t)kc8 * 8);
        const bool by_row = spec.axis == kSynthAxisRow;
        uint32_t w[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t a = synth_bits_chan(spec, base + 2 * j, by_row ? crow : ccol + 2 * j);
            const uint32_t b = synth_bits_chan(spec, base + 2 * j + 1, by_row ? crow : ccol + 2 * j + 1);
            w[j] = a | (b << 16);
        }
        const int nt = r >> 4, kt = kc8 >> 2, lane = ((kc8 & 3) << 4) | (r & 15);
        dst[((int64_t)nt * KT + kt) * 64 + lane] = make_uint4(w[0], w[1], w[2], w[3]);
    }
}

__global__ void __launch_bounds__(256) synth_rowmajor_bf16_kernel(uint16_t* __restrict__ dst, SynthSpec spec, int64_t first,
                                                                  int64_t count) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = synth_bits(spec, (uint64_t)(first + i));
}
__global__ void __launch_bounds__(256) synth_rowmajor_f32_kernel(float* __restrict__ dst, SynthSpec spec, int64_t first,
                                                                 int64_t count) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = bf16_to_f32(synth_bits(spec, (uint64_t)(first + i)));
}

static inline int grid_for(int64_t n, int per_block = 256, int cap = 8192) {
    int64_t g = (n + per_block - 1) / per_block;
    if (g < 1) g = 1;
    if (g > cap) g = cap;
    return (int)g;
}

hipError_t launch_pack_rows(const PackedW& dst, int row0, int rows, const bf16_bits* src, int64_t ld, int ileave,
                            hipStream_t s) {
    const int KT = dst.K / 32;
    pack_rows_kernel<<<grid_for((int64_t)rows * KT * 4), 256, 0, s>>>(dst.data, KT, row0, rows, src, ld, ileave);
    return hipGetLastError();
}
hipError_t launch_synth_packed(const PackedW& dst, int row0, int rows, const SynthSpec& spec, int64_t src_row0,
                               int64_t src_col0, int64_t src_ld, int ileave, hipStream_t s) {
    const int KT = dst.K / 32;
    if (spec.profile != 0 && spec.axis != kSynthAxisNone && spec.cols != src_ld) return hipErrorInvalidValue;
    synth_packed_kernel<<<grid_for((int64_t)rows * KT * 4), 256, 0, s>>>(dst.data, KT, row0, rows, spec, src_row0,
                                                                        src_col0, src_ld, ileave);
    return hipGetLastError();
}
hipError_t launch_synth_rowmajor_bf16(bf16_bits* dst, const SynthSpec& spec, int64_t first, int64_t count, hipStream_t s) {
    synth_rowmajor_bf16_kernel<<<grid_for(count), 256, 0, s>>>(dst, spec, first, count);
    return hipGetLastError();
}
hipError_t launch_synth_rowmajor_f32(float* dst, const SynthSpec& spec, int64_t first, int64_t count, hipStream_t s) {
    synth_rowmajor_f32_kernel<<<grid_for(count), 256, 0, s>>>(dst, spec, first, count);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// debug: scan an f16 buffer (K / V cache) for saturated elements.  Every cache write goes through f16_sat(), which clamps
// to +-65504 (0x7BFF): an element AT that magnitude was (with probability ~1) clamped.  Off the hot path: the kernels that
// write the cache carry no counter.
// ---------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) f16_scan_kernel(const uint4* __restrict__ data, int64_t n16, unsigned long long* sat,
                                                       unsigned* absmax_bits) {
    unsigned long long cnt = 0;
    unsigned mx = 0;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (int64_t)gridDim.x * blockDim.x) {
        const uint4 v = data[i];
        const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const unsigned a = w[j] & 0x7FFFu, b = (w[j] >> 16) & 0x7FFFu;
            cnt += (a >= 0x7BFFu) + (b >= 0x7BFFu);  // 0x7BFF = 65504; above it: inf / NaN (never written by f16_sat of a finite value)
            mx = max(mx, max(a, b));
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) { cnt += __shfl_xor(cnt, o); mx = max(mx, (unsigned)__shfl_xor((int)mx, o)); }
    if ((threadIdx.x & 63) == 0) {
        if (cnt) atomicAdd(sat, cnt);
        atomicMax(absmax_bits, mx);
    }
}
hipError_t launch_f16_scan(const f16_bits* data, int64_t n, unsigned long long* sat, unsigned* absmax_bits, hipStream_t s) {
    f16_scan_kernel<<<grid_for(n / 8, 256, 2048), 256, 0, s>>>(reinterpret_cast<const uint4*>(data), n / 8, sat, absmax_bits);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// conversions
// ---------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) f32_to_bf16_kernel(const float* __restrict__ src, uint16_t* __restrict__ dst,
                                                          int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = bf16_bits_of(src[i]);
}
__global__ void __launch_bounds__(256) bf16_to_f32_kernel(const uint16_t* __restrict__ src, float* __restrict__ dst,
                                                          int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
        dst[i] = bf16_to_f32(src[i]);
}
__global__ void __launch_bounds__(256) split_hilo_kernel(const float* __restrict__ x, uint16_t* __restrict__ hi,
                                                         uint16_t* __restrict__ lo, int64_t n) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        uint16_t h, l;
        split_bf16(x[i], h, l);
        hi[i] = h;
        lo[i] = l;
    }
}
hipError_t launch_f32_to_bf16(const float* src, bf16_bits* dst, int64_t n, hipStream_t s) {
    f32_to_bf16_kernel<<<grid_for(n), 256, 0, s>>>(src, dst, n);
    return hipGetLastError();
}
hipError_t launch_bf16_to_f32(const bf16_bits* src, float* dst, int64_t n, hipStream_t s) {
    bf16_to_f32_kernel<<<grid_for(n), 256, 0, s>>>(src, dst, n);
    return hipGetLastError();
}
hipError_t launch_split_hilo(const float* x, bf16_bits* hi, bf16_bits* lo, int64_t n, hipStream_t s) {
    split_hilo_kernel<<<grid_for(n), 256, 0, s>>>(x, hi, lo, n);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// GEMM  out[ks][M][N] = x[M][Kslice] . W[N][Kslice]^T        (replaces candle_nn::Linear::forward,
// src/layers/linear.rs:35-36,72-77,184-198; src/models/qwen3.rs:205,278,324,326,548)
//
// Weight-streaming design: every wave owns NT n-tiles (16 output features each) and streams their
// packed A-fragments straight from HBM into VGPRs, one contiguous 1 KiB wave-load per (n-tile, k-tile);
// the activation slice (B operand) is staged once per workgroup through LDS in fragment order and
// shared by the NW waves.  Activations are bf16 hi + bf16 lo (x = hi + lo to 2^-17), two MFMAs per
// fragment pair, f32 accumulate: this keeps logits within 1e-3 of the f32 reference.
// grid = (n-groups, k-splits, m-blocks); k-splits write separate f32 slabs, summed by the consumer.
// ---------------------------------------------------------------------------------------------------
// MODE 0: f32 slabs.  MODE 1: + per-wave partial arg-max (LM head).  MODE 2: SwiGLU epilogue -- the weight is
// the gate/up matrix interleaved in 16-row tiles (NT == 2: tile 0 = gate, tile 1 = up of the same 16 features),
// the wave writes silu(gate)*up as bf16 hi/lo planes act[M][N/2] (SiluAndMul, activation.rs:13-18); no split-K.
template <int MT, int NT, int NW, int KC, int MODE>
__global__ void __launch_bounds__(NW * 64)
gemm_kernel(const uint16_t* __restrict__ xh, const uint16_t* __restrict__ xl, int ldx, const uint4* __restrict__ wp,
            float* __restrict__ out, int M, int N, int KT, int kt_per_split, float* __restrict__ part_val,
            int* __restrict__ part_idx, uint16_t* __restrict__ act_hi, uint16_t* __restrict__ act_lo, RowNorm rn, GluSpec glu) {
    // LDS: two buffers of [2 planes][MT][KC][64 lanes] 16-byte slots, filled by LDS-DMA (global_load_lds):
    // the image is lane-linear per fragment, so every wave-DMA writes one contiguous 1 KiB and every
    // ds_read_b128 of a fragment is conflict-free.
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    uint4* lds = reinterpret_cast<uint4*>(smem_raw);
    constexpr int FRAGS = 2 * MT * KC;  // per buffer
    float* lds_rn = reinterpret_cast<float*>(smem_raw + (size_t)2 * FRAGS * 1024);  // [4][MT*16] deferred-norm partials
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l15 = lane & 15, grp = lane >> 4;
    const int ntiles = N >> 4;
    const int nt0 = (blockIdx.x * NW + wave) * NT;
    const int kt_begin = blockIdx.y * kt_per_split;
    const int kt_end = min(KT, kt_begin + kt_per_split);
    const int m0 = blockIdx.z * (MT * 16);
    const int nchunks = (kt_end - kt_begin + KC - 1) / KC;

    f32x4 acc[NT][MT];
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    // Two named register sets / LDS buffers (static indices only: a runtime-selected set would make
    // every MFMA depend on the loads still in flight for the other one).
    uint4 wf0[NT][KC], wf1[NT][KC];
    int xrows[MT];  // staged row of each m-tile for this lane (gathered once: LM head on last tokens only)
#pragma unroll
    for (int b = 0; b < MT; ++b) {
        xrows[b] = min(m0 + b * 16 + l15, M - 1);
        if (rn.row_idx) xrows[b] = rn.row_idx[xrows[b]];
    }
    // issue the loads of one chunk: weight fragments -> VGPRs, activation fragments -> LDS by DMA.
    // Rows >= M and k-tiles past the split are clamped to valid addresses: their products are never
    // stored (rows) or meet zeroed weight fragments (k), so only finiteness matters.
    auto issue = [&](int c, int buf, uint4 (&w)[NT][KC]) {
        const int kc = kt_begin + c * KC;
        // unconditional loads from clamped (always valid) n-tiles: a branch around a load makes hipcc wait
        // vmcnt(0) after each one (serialised HBM round trips), and so does any immediate use of the data.
        // The host guarantees every split is a whole number of chunks (K % (32*KC) == 0), so no k masking.
#pragma unroll
        for (int a = 0; a < NT; ++a) {
            const int ntc = min(nt0 + a, ntiles - 1);
#pragma unroll
            for (int k = 0; k < KC; ++k) w[a][k] = wp[((size_t)ntc * KT + kc + k) * 64 + lane];
        }
#pragma unroll
        for (int i = 0; i < (FRAGS + NW - 1) / NW; ++i) {
            const int f = wave + i * NW;
            if (FRAGS % NW == 0 || f < FRAGS) {
                const int plane = f / (MT * KC);
                const int rem = f - plane * (MT * KC);
                const int mt = rem / KC, k = rem - mt * KC;
                const int row = xrows[mt];
                const uint16_t* src = (plane ? xl : xh) + (size_t)row * ldx + (size_t)(kc + k) * 32 + grp * 8;
                __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(lds + (size_t)(buf * FRAGS + f) * 64), 16, 0, 0);
            }
        }
    };
    auto compute = [&](int buf, const uint4 (&w)[NT][KC]) {
#pragma unroll
        for (int k = 0; k < KC; ++k) {
            bf16x8 bh[MT], bl[MT];
#pragma unroll
            for (int b = 0; b < MT; ++b) {  // all LDS reads of this k-step first, then the MFMAs
                bh[b] = __builtin_bit_cast(bf16x8, lds[(size_t)(buf * FRAGS + (0 * MT + b) * KC + k) * 64 + lane]);
                bl[b] = __builtin_bit_cast(bf16x8, lds[(size_t)(buf * FRAGS + (1 * MT + b) * KC + k) * 64 + lane]);
            }
#pragma unroll
            for (int a = 0; a < NT; ++a) {
                const bf16x8 wv = __builtin_bit_cast(bf16x8, w[a][k]);
#pragma unroll
                for (int b = 0; b < MT; ++b) {
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, bh[b], acc[a][b], 0, 0, 0);
                    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, bl[b], acc[a][b], 0, 0, 0);
                }
            }
        }
    };

    if (nchunks <= 2) {
        // Both chunks are issued up front (both LDS buffers, both register sets): a K-slice of <= 2 chunks --
        // every decode-shape split -- costs ONE memory round trip instead of two dependent ones.
        if (nchunks > 0) issue(0, 0, wf0);
        if (nchunks > 1) issue(1, 1, wf1);
        // deferred-norm partials: loaded AFTER the main loads were issued (vmcnt is in order), parked in LDS
        if constexpr (MODE != 0) rownorm_partials<MT * 16>(rn, m0, M, lds_rn);
        dma_publish_barrier();  // vmcnt(0) + barrier: everything has landed
        if (nchunks > 0) compute(0, wf0);
        if (nchunks > 1) compute(1, wf1);
    } else {
        // long K (LM head, prefill): one chunk ahead, one barrier per chunk
        issue(0, 0, wf0);
        if constexpr (MODE != 0) rownorm_partials<MT * 16>(rn, m0, M, lds_rn);
        for (int c = 0; c < nchunks; c += 2) {
            dma_publish_barrier();  // chunk c has landed; buffer 1 is free again
            if (c + 1 < nchunks) issue(c + 1, 1, wf1);
            compute(0, wf0);
            if (c + 1 >= nchunks) break;
            dma_publish_barrier();
            if (c + 2 < nchunks) issue(c + 2, 0, wf0);
            compute(1, wf1);
        }
    }
    if constexpr (MODE == 1) {  // LM head on a deferred final norm: logits = rinv[row] * acc
        if (rn.ssq) {
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const float ri = rownorm_rinv_lds<MT * 16>(rn, lds_rn, b * 16 + l15);
#pragma unroll
                for (int a = 0; a < NT; ++a) {
                    acc[a][b][0] *= ri; acc[a][b][1] *= ri; acc[a][b][2] *= ri; acc[a][b][3] *= ri;
                }
            }
        }
    }
    if constexpr (MODE == 1) {
        if (rn.softcap > 0.f) {
#pragma unroll
            for (int a = 0; a < NT; ++a)
#pragma unroll
                for (int b = 0; b < MT; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[a][b][r] = soft_cap(acc[a][b][r], rn.softcap);
        }
    }
    // D[feature 4*grp+reg][token l15] -> out[token][feature..feature+3]
    if (MODE != 2 && out) {
        float* o = out + (size_t)blockIdx.y * (size_t)M * N;
#pragma unroll
        for (int a = 0; a < NT; ++a) {
            if (nt0 + a >= ntiles) continue;
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const int row = m0 + b * 16 + l15;
                if (row < M) {
                    const f32x4 v = acc[a][b];
                    *reinterpret_cast<float4*>(o + (size_t)row * N + (size_t)(nt0 + a) * 16 + grp * 4) =
                        make_float4(v[0], v[1], v[2], v[3]);
                }
            }
        }
    }
    if constexpr (MODE == 2) {
        static_assert(MODE != 2 || NT % 2 == 0, "SwiGLU epilogue needs gate and up tiles of a feature in one wave");
        const int I = N >> 1;
#pragma unroll
        for (int pr = 0; pr < NT / 2; ++pr) {
            if (nt0 + 2 * pr + 1 >= ntiles) continue;
            const int f0 = ((nt0 >> 1) + pr) * 16 + grp * 4;  // activation feature of acc[.][.][0]
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const int row = m0 + b * 16 + l15;
                if (row < M) {
                    const float ri = rownorm_rinv_lds<MT * 16>(rn, lds_rn, b * 16 + l15);
                    uint16_t h[4], l[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float g = acc[2 * pr][b][r] * ri, u = acc[2 * pr + 1][b][r] * ri;
                        split_bf16(glu_mul(g, u, glu), h[r], l[r]);
                    }
                    *reinterpret_cast<uint2*>(act_hi + (size_t)row * I + f0) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                    *reinterpret_cast<uint2*>(act_lo + (size_t)row * I + f0) = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
                }
            }
        }
    }
    if constexpr (MODE == 1) {
        // per-wave partial argmax over its NT*16 features (greedy LM head): LAST max wins
        // (llm_engine.rs:135-142).  part_*[wave_global][row]; finished by argmax_parts_kernel.
        const int wg = blockIdx.x * NW + wave;
#pragma unroll
        for (int b = 0; b < MT; ++b) {
            float bv = -INFINITY;
            int bi = -1;
#pragma unroll
            for (int a = 0; a < NT; ++a) {
                if (nt0 + a >= ntiles) continue;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float v = acc[a][b][r];
                    const int idx = (nt0 + a) * 16 + grp * 4 + r;
                    if (bi < 0 || v > bv || (v == bv && idx > bi)) { bv = v; bi = idx; }
                }
            }
#pragma unroll
            for (int o = 16; o <= 32; o <<= 1) {
                const float ov = __shfl_xor(bv, o);
                const int oi = __shfl_xor(bi, o);
                if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi > bi))) { bv = ov; bi = oi; }
            }
            const int row = m0 + b * 16 + l15;
            if (grp == 0 && row < M) {
                part_val[(size_t)wg * M + row] = bv;
                part_idx[(size_t)wg * M + row] = bi;
            }
        }
    }
}

// finish the fused LM-head arg-max.  part_*[p][row] (row fastest): thread = (row%64, plane); a block scans one
// slice of the partials with coalesced loads, reduces its 4 planes in LDS and folds its result into a per-row
// 64-bit key {order-preserving float bits, index} with one atomicMax per row; the last block to finish decodes
// the keys into ids / max values and re-arms the scratch words (keys and ticket are zero between launches).
__device__ __forceinline__ unsigned long long argmax_key(float v, int idx) {
    unsigned u = __builtin_bit_cast(unsigned, v);
    u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
    return ((unsigned long long)u << 32) | (unsigned)idx;
}
__global__ void __launch_bounds__(256) argmax_parts_kernel(const float* __restrict__ part_val,
                                                           const int* __restrict__ part_idx, int n_parts, int M,
                                                           unsigned long long* __restrict__ keys,
                                                           unsigned* __restrict__ ticket, uint32_t* __restrict__ ids,
                                                           float* __restrict__ maxval) {
    __shared__ unsigned long long sk[256];
    __shared__ unsigned last;
    const int r = threadIdx.x & 63, plane = threadIdx.x >> 6;
    const int row = blockIdx.y * 64 + r;
    const int per = (n_parts + gridDim.x - 1) / gridDim.x;
    const int p0 = blockIdx.x * per, p1 = min(n_parts, p0 + per);
    unsigned long long best = 0;
    if (row < M)
        for (int p = p0 + plane; p < p1; p += 4) {
            const int i = part_idx[(size_t)p * M + row];
            if (i >= 0) {
                const unsigned long long k = argmax_key(part_val[(size_t)p * M + row], i);
                best = k > best ? k : best;
            }
        }
    sk[threadIdx.x] = best;
    __syncthreads();
    if (plane == 0 && row < M) {
        for (int q = 1; q < 4; ++q) best = sk[q * 64 + r] > best ? sk[q * 64 + r] : best;
        if (best) atomicMax(&keys[row], best);
    }
    __threadfence();
    __syncthreads();
    if (threadIdx.x == 0) last = atomicAdd(ticket, 1u) == gridDim.x * gridDim.y - 1 ? 1u : 0u;
    __syncthreads();
    if (last) {
        __threadfence();
        for (int i = threadIdx.x; i < M; i += blockDim.x) {
            const unsigned long long k = __hip_atomic_load(&keys[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            ids[i] = (uint32_t)(k & 0xffffffffu);
            if (maxval) {
                unsigned u = (unsigned)(k >> 32);
                u = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
                maxval[i] = __builtin_bit_cast(float, u);
            }
            keys[i] = 0;
        }
        if (threadIdx.x == 0) *ticket = 0;
    }
}

// every split covers a whole number of KC-chunks
void set_split(GemmPlan& p, int KT, int want) {
    int per = (KT + want - 1) / want;
    per = (per + p.kc - 1) / p.kc * p.kc;
    p.kt_per_split = per;
    p.n_split = (KT + per - 1) / per;
}

GemmPlan plan_gemm(int M, int N, int K, int max_split) {
    GemmPlan p;
    p.mt = M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : 8;
    p.kc = p.mt == 8 ? 2 : 4;
    const int rowblocks = (M + 16 * p.mt - 1) / (16 * p.mt);
    const int ntiles = N / 16;
    p.nw = 4;
    p.nt = ((int64_t)ntiles * rowblocks >= 2048) ? 2 : 1;
    // prefill (MFMA-bound): 128 x 256 output tile per workgroup, 128 MFMAs per wave between barriers so the
    // next chunk's LDS-DMA hides behind the matrix pipe; 64 KiB of LDS -> two workgroups per CU
    if (M >= 256 && ntiles % 4 == 0) p.nt = 4;
    const int KT = K / 32;
    const int64_t groups = (int64_t)((ntiles + p.nt * p.nw - 1) / (p.nt * p.nw)) * rowblocks;
    int ns = 1;
    while (groups * ns < 256 && ns * 2 <= max_split && KT / (ns * 2) >= 8) ns *= 2;
    set_split(p, KT, ns);
    return p;
}

struct GemmExtra {
    float* part_val = nullptr;   // MODE 1
    int* part_idx = nullptr;
    bf16_bits* act_hi = nullptr; // MODE 2
    bf16_bits* act_lo = nullptr;
    RowNorm rn;
    GluSpec glu;
};

template <int MT, int NT, int NW, int KC, int MODE>
static hipError_t gemm_launch_t(const GemmPlan& p, const bf16_bits* xh, const bf16_bits* xl, int ldx, const PackedW& w,
                                float* out, int M, const GemmExtra& x, hipStream_t s) {
    const int ntiles = w.N / 16;
    dim3 grid((ntiles + NT * NW - 1) / (NT * NW), p.n_split, (M + MT * 16 - 1) / (MT * 16));
    const size_t lds = (size_t)2 * 2 * MT * KC * 1024 + (size_t)4 * MT * 16 * 4;
    static std::atomic<uint64_t> lds_set{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(gemm_kernel<MT, NT, NW, KC, MODE>), lds, lds_set);
    gemm_kernel<MT, NT, NW, KC, MODE><<<grid, NW * 64, lds, s>>>(xh, xl, ldx, w.data, out, M, w.N, w.K / 32, p.kt_per_split,
                                                                x.part_val, x.part_idx, x.act_hi, x.act_lo, x.rn, x.glu);
    return hipGetLastError();
}

template <int NW, int MODE>
static hipError_t gemm_dispatch_nw(const GemmPlan& p, const bf16_bits* xh, const bf16_bits* xl, int ldx, const PackedW& w,
                                   float* out, int M, const GemmExtra& x, hipStream_t s) {
#define NVLLM_GEMM_CASE(MT_, NT_, KC_) \
    if (p.mt == MT_ && p.nt == NT_ && p.kc == KC_) return gemm_launch_t<MT_, NT_, NW, KC_, MODE>(p, xh, xl, ldx, w, out, M, x, s);
    if constexpr (MODE != 2) {
        NVLLM_GEMM_CASE(1, 1, 4)
        NVLLM_GEMM_CASE(2, 1, 4)
        NVLLM_GEMM_CASE(4, 1, 4)
        NVLLM_GEMM_CASE(8, 1, 2)
    }
    NVLLM_GEMM_CASE(1, 2, 4)
    NVLLM_GEMM_CASE(2, 2, 4)
    NVLLM_GEMM_CASE(4, 2, 4)
    NVLLM_GEMM_CASE(8, 2, 2)
    if constexpr (NW == 4) { NVLLM_GEMM_CASE(8, 4, 2) }  // prefill tile: 128 rows x 256 features per workgroup
    if constexpr (NW == 8 && MODE != 2) { NVLLM_GEMM_CASE(4, 1, 8) }  // big-K streaming: 256-deep chunks
    if constexpr (NW == 8) { NVLLM_GEMM_CASE(4, 2, 8) }
#undef NVLLM_GEMM_CASE
    return hipErrorInvalidValue;
}

template <int MODE>
static hipError_t gemm_dispatch(const GemmPlan& p, const bf16_bits* xh, const bf16_bits* xl, int ldx, const PackedW& w,
                                float* out, int M, const GemmExtra& x, hipStream_t s) {
    if ((w.K / 32) % p.kc != 0 || p.kt_per_split % p.kc != 0) return hipErrorInvalidValue;
    if (p.nw == 2) return gemm_dispatch_nw<2, MODE>(p, xh, xl, ldx, w, out, M, x, s);
    if (p.nw == 4) return gemm_dispatch_nw<4, MODE>(p, xh, xl, ldx, w, out, M, x, s);
    if (p.nw == 8) return gemm_dispatch_nw<8, MODE>(p, xh, xl, ldx, w, out, M, x, s);
    return hipErrorInvalidValue;
}

hipError_t launch_gemm(const GemmPlan& p, const bf16_bits* xh, const bf16_bits* xl, int ldx, const PackedW& w,
                       float* out, int M, hipStream_t s) {
    return gemm_dispatch<0>(p, xh, xl, ldx, w, out, M, GemmExtra{}, s);
}

// ---------------------------------------------------------------------------------------------------
// LM head for decode: logits = x.W^T (Qwen3ForCausalLM::compute_logits, qwen3.rs:542-550) with
// the greedy arg-max (llm_engine.rs:135-142, LAST max wins) in the epilogue.  The vocabulary matrix is the
// largest stream of a step (311 MB for Qwen3-0.6B), read exactly once: one workgroup per CU, 8 waves, each wave
// owns NT n-tiles for the WHOLE K and keeps two 2-k-tile weight sets (2*NT KiB each) in flight while all 64 rows
// of x ride through LDS in 8-k-tile chunks (double buffered, every wave stages one k-tile of a chunk).
// More rows: slices of 64, the workgroups of one group of columns beside each other on an XCD, so that the matrix comes from memory once
// and from that XCD's L2 for the other slices; bound by the matrix cores from about 100 rows on.  0.6B steps: 65 rows 1.715 -> 1.63 ms,
// 100 rows 1.919 -> 1.83, 129 rows 2.452 -> 2.24, 200 rows (head 377 -> 176 us) 3.082 -> 2.85, each against the chunked kernel.
// ---------------------------------------------------------------------------------------------------
template <int MT, int NT, int NCH>
__global__ void __launch_bounds__(512) lmhead_kernel(const uint16_t* __restrict__ xh, const uint16_t* __restrict__ xl, int ldx,
                                                     const uint4* __restrict__ wp, float* __restrict__ out, int M, int N, int KT,
                                                     float* __restrict__ part_val, int* __restrict__ part_idx, RowNorm rn) {
    // Sets of SC k-tiles: 64 rows of five n-tiles, 80 accumulator registers leave room for one only; with one or two n-tiles a wave what is in flight comes from depth.
    // Sets of 1 or 2 / these, us at 1, 32, 64, 200 rows: 32768 x 1024 21.5 22.0 28.3 82 / 17.8 19.7 25.4 67, 32768 x 2048 (in a loop / unrolled) 33.0 36.0 50 155 / 32.4 34.8 45
    // 121, 65536 x 1024 34 35.5 40.5 102 / 30.8 31.2 40.8 96, 65536 x 2048 50.6 54 62.4 190 / 50.3 51.4 59 172 (sets of 4 at 33 rows and more of two n-tiles: 64 rows 1 us more)
    constexpr int NW = 8, KC = 8, SC = NT <= 2 && NCH > 0 ? (NT == 2 && MT == 4 ? 2 : 4) : MT == 4 ? 1 : 2;
    // Both x buffers asked for ahead of the weights, and the first barrier waits for x alone: 151936 x 1024, one row 52.9 -> 51.0 us; 64 rows the same, in slices (200 rows) 170 -> 174
    constexpr bool EARLY = MT < 4;
    constexpr int FRAGS = 2 * MT * KC;  // 1 KiB fragments per x chunk: [2 planes][MT][KC]
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    uint4* lds = reinterpret_cast<uint4*>(smem_raw);                                    // [2][FRAGS][64]
    float* lds_rn = reinterpret_cast<float*>(smem_raw + (size_t)2 * FRAGS * 1024);      // [4][MT*16]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l15 = lane & 15, grp = lane >> 4;
    const int ntiles = N >> 4;
    const int n_groups = (ntiles + NW * NT - 1) / (NW * NT), slices = (M + MT * 16 - 1) / (MT * 16);
    int group = blockIdx.x, row0 = 0;
    if (slices > 1) {  // more than 64 rows
        const int slot = (int)blockIdx.x >> 3;
        row0 = (slot % slices) * MT * 16;
        group = (slot / slices) * 8 + ((int)blockIdx.x & 7);
        if (group >= n_groups) return;  // whole workgroup, before any barrier
    }
    const int nt0 = (group * NW + wave) * NT;
    // deferred-norm partials first, while no other registers are live: 16 independent loads, parked in LDS
    rownorm_partials<MT * 16>(rn, row0, M, lds_rn);
    __builtin_amdgcn_sched_barrier(0);
    unsigned xoff[MT];  // element offset of this lane's 16-byte piece in row block b (k-tile 0), < 2^32 elements
#pragma unroll
    for (int b = 0; b < MT; ++b) {
        int r = min(row0 + b * 16 + l15, M - 1);
        if (rn.row_idx) r = rn.row_idx[r];
        xoff[b] = (unsigned)r * (unsigned)ldx + (unsigned)(wave * 32 + grp * 8);
    }
    f32x4 acc[NT][MT];
#pragma unroll
    for (int a = 0; a < NT; ++a)
#pragma unroll
        for (int b = 0; b < MT; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    // wave w stages k-tile w of the chunk for both planes and every row block (2*MT LDS-DMA loads)
    auto stage = [&](int c, int buf) {
#pragma unroll
        for (int plane = 0; plane < 2; ++plane)
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const uint16_t* src = (plane ? xl : xh) + (size_t)(xoff[b] + (unsigned)(c * KC * 32));
                __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(lds + (size_t)(buf * FRAGS + (plane * MT + b) * KC + wave) * 64), 16, 0, 0);
            }
    };
    uint4 wA[NT][SC], wB[NT][SC];
    auto issue_w = [&](int kt0, uint4 (&w)[NT][SC]) {
        const int kt = min(kt0, KT - SC);  // past the end: a harmless re-read of the last set
#pragma unroll
        for (int a = 0; a < NT; ++a) {
            const int ntc = min(nt0 + a, ntiles - 1);
#pragma unroll
            for (int j = 0; j < SC; ++j) w[a][j] = ld_stream16(wp + ((size_t)ntc * KT + kt + j) * 64 + lane);  // read once per step, by this CU only
        }
    };
    auto compute = [&](int k0, int buf, const uint4 (&w)[NT][SC]) {
#pragma unroll
        for (int j = 0; j < SC; ++j)
#pragma unroll
            for (int plane = 0; plane < 2; ++plane) {  // hi plane, then lo plane: MT x-fragments live at a time
                bf16x8 bx[MT];
                if constexpr (MT == 4) {  // by asm that waits for itself, see gemm_stream_kernel (64 rows 1.326 -> 1.314 ms a step; fewer rows lose)
                    lds_read_fragments<KC * 1024>(bx, lds_address(lds) + (uint32_t)(buf * FRAGS * 1024 + lane * 16), (plane * MT * KC + k0 + j) * 1024);
                } else {
#pragma unroll
                    for (int b = 0; b < MT; ++b)
                        bx[b] = __builtin_bit_cast(bf16x8, lds[(size_t)(buf * FRAGS + (plane * MT + b) * KC + k0 + j) * 64 + lane]);
                }
#pragma unroll
                for (int a = 0; a < NT; ++a) {
                    const bf16x8 wv = __builtin_bit_cast(bf16x8, w[a][j]);
#pragma unroll
                    for (int b = 0; b < MT; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, bx[b], acc[a][b], 0, 0, 0);
                }
            }
    };
    // NCH > 0: the chunk loop is fully unrolled (the compiler then tracks every load in flight exactly; with a
    // back-edge it falls back to vmcnt(0) after each refill)
    const int nchunks = NCH > 0 ? NCH : KT / KC;
    stage(0, 0);
    if constexpr (EARLY) {
        if (nchunks > 1) stage(1, 1);
        __builtin_amdgcn_sched_barrier(0);
    }
    issue_w(0, wA);
    issue_w(SC, wB);
    if constexpr (EARLY) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < nchunks; ++c) {
        // chunk c is in LDS and every wave is done with the other buffer.  After the first chunk the wait covers
        // only this wave's x stage: the KC/SC weight sets issued after it (vmcnt retires in order) stay in flight
        // across the barrier instead of draining the stream four times per launch.
        if (EARLY && c == 0) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * NT * SC) : "memory");
        else if (c == 0) dma_publish_barrier();
        else asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"((KC / SC) * NT * SC) : "memory");
        if ((c > 0 || !EARLY) && c + 1 < nchunks) stage(c + 1, (c + 1) & 1);
        __builtin_amdgcn_sched_barrier(0);  // the weight loads below are issued AFTER the stage (the count above relies on it)
        const int base = c * KC, buf = c & 1;
        // scheduling fences: a refill is issued exactly where it is written (the compiler otherwise sinks it to its
        // first use to save registers, which serialises every 1 KiB load behind a vmcnt(0))
#define NVLLM_LM_STEP(k0_, set_, next_)            \
    compute(k0_, buf, set_);                       \
    __builtin_amdgcn_sched_barrier(0);             \
    issue_w(next_, set_);                          \
    __builtin_amdgcn_sched_barrier(0);
        if constexpr (SC == 4) {
            NVLLM_LM_STEP(0, wA, base + 8)
            NVLLM_LM_STEP(4, wB, base + 12)
        } else if constexpr (SC == 2) {
            NVLLM_LM_STEP(0, wA, base + 4)
            NVLLM_LM_STEP(2, wB, base + 6)
            NVLLM_LM_STEP(4, wA, base + 8)
            NVLLM_LM_STEP(6, wB, base + 10)
        } else {
            NVLLM_LM_STEP(0, wA, base + 2)
            NVLLM_LM_STEP(1, wB, base + 3)
            NVLLM_LM_STEP(2, wA, base + 4)
            NVLLM_LM_STEP(3, wB, base + 5)
            NVLLM_LM_STEP(4, wA, base + 6)
            NVLLM_LM_STEP(5, wB, base + 7)
            NVLLM_LM_STEP(6, wA, base + 8)
            NVLLM_LM_STEP(7, wB, base + 9)
        }
#undef NVLLM_LM_STEP
    }
    if (rn.ssq) {  // deferred final norm: logits = rinv[row] * acc
#pragma unroll
        for (int b = 0; b < MT; ++b) {
            const float ri = rownorm_rinv_lds<MT * 16>(rn, lds_rn, b * 16 + l15);
#pragma unroll
            for (int a = 0; a < NT; ++a) {
                acc[a][b][0] *= ri; acc[a][b][1] *= ri; acc[a][b][2] *= ri; acc[a][b][3] *= ri;
            }
        }
    }
    if (rn.softcap > 0.f) {
#pragma unroll
        for (int a = 0; a < NT; ++a)
#pragma unroll
            for (int b = 0; b < MT; ++b)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[a][b][r] = soft_cap(acc[a][b][r], rn.softcap);
    }
    const int wg = group * NW + wave;
#pragma unroll
    for (int b = 0; b < MT; ++b) {
        const int row = row0 + b * 16 + l15;
        float bv = -INFINITY;
        int bi = -1;
#pragma unroll
        for (int a = 0; a < NT; ++a) {
            if (nt0 + a >= ntiles) continue;
            const f32x4 v = acc[a][b];
            if (out && row < M) *reinterpret_cast<float4*>(out + (size_t)row * N + (size_t)(nt0 + a) * 16 + grp * 4) = make_float4(v[0], v[1], v[2], v[3]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int idx = (nt0 + a) * 16 + grp * 4 + r;
                if (bi < 0 || v[r] > bv || (v[r] == bv && idx > bi)) { bv = v[r]; bi = idx; }
            }
        }
#pragma unroll
        for (int o = 16; o <= 32; o <<= 1) {
            const float ov = __shfl_xor(bv, o);
            const int oi = __shfl_xor(bi, o);
            if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi > bi))) { bv = ov; bi = oi; }
        }
        if (grp == 0 && row < M) {  // part_*[row][wave]: one workgroup per row finishes (argmax_rows_kernel)
            const size_t n_parts = (size_t)n_groups * NW;
            part_val[(size_t)row * n_parts + wg] = bv;
            part_idx[(size_t)row * n_parts + wg] = bi;
        }
    }
}

// finish the streaming LM head's arg-max: part_*[row][n_parts], one workgroup per row, no atomics
__global__ void __launch_bounds__(256) argmax_rows_kernel(const float* __restrict__ part_val, const int* __restrict__ part_idx,
                                                          int n_parts, uint32_t* __restrict__ ids, float* __restrict__ maxval) {
    __shared__ unsigned long long sk[4];
    const int row = blockIdx.x;
    const float* pv = part_val + (size_t)row * n_parts;
    const int* pi = part_idx + (size_t)row * n_parts;
    unsigned long long best = 0;
    for (int p0 = 0; p0 < n_parts; p0 += 256 * 4) {
        int i4[4]; float v4[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {  // unconditional loads (clamped), validity applied afterwards
            const int p = min(p0 + u * 256 + (int)threadIdx.x, n_parts - 1);
            i4[u] = pi[p]; v4[u] = pv[p];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool ok = (p0 + u * 256 + (int)threadIdx.x) < n_parts && i4[u] >= 0;
            const unsigned long long k = ok ? argmax_key(v4[u], i4[u]) : 0ull;
            best = k > best ? k : best;
        }
    }
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned lo = __shfl_xor((unsigned)best, o), hi = __shfl_xor((unsigned)(best >> 32), o);
        const unsigned long long k = ((unsigned long long)hi << 32) | lo;
        best = k > best ? k : best;
    }
    if ((threadIdx.x & 63) == 0) sk[threadIdx.x >> 6] = best;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int q = 1; q < 4; ++q) best = sk[q] > best ? sk[q] : best;
        ids[row] = (uint32_t)(best & 0xffffffffu);
        if (maxval) {
            unsigned u = (unsigned)(best >> 32);
            u = (u & 0x80000000u) ? (u & 0x7fffffffu) : ~u;
            maxval[row] = __builtin_bit_cast(float, u);
        }
    }
}
hipError_t launch_argmax_rows(const float* part_val, const int* part_idx, int n_parts, int M, uint32_t* ids, float* maxval, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    argmax_rows_kernel<<<M, 256, 0, s>>>(part_val, part_idx, n_parts, ids, maxval);
    return hipGetLastError();
}

template <int MT, int NT, int NCH>
static hipError_t lmhead_launch_t(const bf16_bits* xh, const bf16_bits* xl, int ldx, const PackedW& w, float* out, int M,
                                  float* part_val, int* part_idx, const RowNorm& rn, hipStream_t s) {
    const size_t lds = (size_t)2 * (2 * MT * 8) * 1024 + (size_t)4 * MT * 16 * 4;
    static std::atomic<uint64_t> lds_set{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(lmhead_kernel<MT, NT, NCH>), lds, lds_set);
    const int waves = (w.N / 16 + NT - 1) / NT;
    const int groups = (waves + 7) / 8, slices = (M + MT * 16 - 1) / (MT * 16);
    lmhead_kernel<MT, NT, NCH><<<slices > 1 ? (groups + 7) / 8 * 8 * slices : groups, 512, lds, s>>>(xh, xl, ldx, w.data, out, M, w.N, w.K / 32, part_val, part_idx, rn);
    return hipGetLastError();
}

GemmPlan plan_lmhead(int M, int N, int K) {
    GemmPlan p = plan_gemm(M, N, K, 1);
    if (K % 256 || N % 16) return p;
    // one workgroup (8 waves) per CU: n-tiles per wave so that the grid fits the 256 CUs in one round
    const int ntiles = N / 16;
    int nt = (ntiles + 2047) / 2048;
    if (nt > 6) nt = 6;  // bigger vocabularies run several rounds
    p.lm_nt = nt;
    return p;
}

hipError_t launch_gemm_argmax(const GemmPlan& p, const bf16_bits* xh, const bf16_bits* xl, int ldx, const PackedW& w,
                              float* out, int M, float* part_val, int* part_idx, const RowNorm* rn, hipStream_t s) {
    if (!part_val || !part_idx || p.n_split != 1) return hipErrorInvalidValue;
    GemmExtra x;
    x.part_val = part_val; x.part_idx = part_idx;
    if (rn) x.rn = *rn;
    if (p.lm_nt > 0) {
        if (M < 1 || w.K % 256) return hipErrorInvalidValue;
        const int mt = M <= 16 ? 1 : M <= 32 ? 2 : 4;
#define NVLLM_LM(MT_, NT_)                                                                                                   \
    if (mt == MT_ && p.lm_nt == NT_)                                                                                       \
        return w.K == 1024 ? lmhead_launch_t<MT_, NT_, 4>(xh, xl, ldx, w, out, M, part_val, part_idx, x.rn, s)             \
               : w.K == 2048 && NT_ <= 2 ? lmhead_launch_t<MT_, NT_, NT_ <= 2 ? 8 : 0>(xh, xl, ldx, w, out, M, part_val, part_idx, x.rn, s) \
                           : lmhead_launch_t<MT_, NT_, 0>(xh, xl, ldx, w, out, M, part_val, part_idx, x.rn, s);
#define NVLLM_LM_MT(MT_) NVLLM_LM(MT_, 1) NVLLM_LM(MT_, 2) NVLLM_LM(MT_, 3) NVLLM_LM(MT_, 4) NVLLM_LM(MT_, 5) NVLLM_LM(MT_, 6)
        NVLLM_LM_MT(1) NVLLM_LM_MT(2) NVLLM_LM_MT(4)
#undef NVLLM_LM_MT
#undef NVLLM_LM
        return hipErrorNotSupported;
    }
    return gemm_dispatch<1>(p, xh, xl, ldx, w, out, M, x, s);
}

// gate/up GEMM with the SwiGLU epilogue; w = interleaved gate_up [2I][K]; act planes [M][I]
hipError_t launch_gemm_swiglu(const GemmPlan& p, const bf16_bits* xh, const bf16_bits* xl, int ldx, const PackedW& w,
                              int M, bf16_bits* act_hi, bf16_bits* act_lo, const RowNorm* rn, hipStream_t s, const GluSpec& glu) {
    if (p.nt % 2 || p.n_split != 1 || !act_hi || !act_lo) return hipErrorInvalidValue;
    GemmExtra x;
    x.act_hi = act_hi; x.act_lo = act_lo; x.glu = glu;
    if (rn) x.rn = *rn;
    return gemm_dispatch<2>(p, xh, xl, ldx, w, nullptr, M, x, s);
}
GemmPlan plan_gemm_swiglu(int M, int N2, int K) {
    GemmPlan p = plan_gemm(M, N2, K, 1);
    p.nt = 2;
    if (M <= 128) {
        // decode: no K-split is possible (the epilogue needs whole sums), so parallelism comes from splitting
        // the ROWS over workgroups (16 rows each); the weight tiles are re-read through L2 by the row blocks.
        // Measured cold, M=64 0.6B gate_up: mt=1/nw=2 9.8 us vs mt=4/nw=2 15.8 us (tools/tune_gemm2.py)
        p.mt = 1; p.kc = 4; p.nw = 2;
    } else {
        p.nw = 4;
        if (M >= 256 && (N2 / 16) % 4 == 0) p.nt = 4;
    }
    set_split(p, K / 32, 1);
    return p;
}

int gemm_argmax_parts(const GemmPlan& p, int N) {
    if (p.lm_nt > 0) return (((N / 16 + p.lm_nt - 1) / p.lm_nt + 7) / 8) * 8;  // one partial per wave, 8 waves per workgroup
    return ((N / 16 + p.nt * p.nw - 1) / (p.nt * p.nw)) * p.nw;
}

hipError_t launch_argmax_parts(const float* part_val, const int* part_idx, int n_parts, int M, void* scratch,
                               uint32_t* ids, float* maxval, hipStream_t s) {
    if (M <= 0) return hipSuccess;
    // scratch: [0] ticket (u32, padded to 8 B), then M u64 keys; zeroed once at allocation, re-armed by the kernel
    unsigned* ticket = reinterpret_cast<unsigned*>(scratch);
    unsigned long long* keys = reinterpret_cast<unsigned long long*>(scratch) + 1;
    dim3 grid(std::max(1, std::min(64, n_parts / 64)), (M + 63) / 64);
    argmax_parts_kernel<<<grid, 256, 0, s>>>(part_val, part_idx, n_parts, M, keys, ticket, ids, maxval);
    return hipGetLastError();
}


// ---------------------------------------------------------------------------------------------------
// Row-parallel projection (o_proj, down_proj) for decode with a residual + next-norm epilogue.
// Replaces: RowParallelLinear::forward (linear.rs:184-198) + the following RMSNorm::forward(x, residual)
// (layernorm.rs:44-60; qwen3.rs:393 / :378 of the next layer): resid += x.W^T ; x' = w_next (.) resid ;
// ssq[group][row] = partial sum of squares (the consumer applies 1/rms, see RowNorm).
//
// One workgroup = 16 rows x NWN n-tiles; its NWN*NWK waves split K NWK ways.  EVERY load of the workgroup
// is issued before the first wait: each wave's PH*TPW weight fragments (HBM -> VGPR) and the x fragments of
// phase 0 (LDS-DMA, shared by all waves).  K ranges too large for LDS run in PH = 2 phases (the second x
// image comes from L2 while the weights are already in registers).  Partial sums meet in LDS, the k-slice-0
// waves run the epilogue.  Rows are split over blockIdx.z (weights re-read through L2 by the row blocks).
// ---------------------------------------------------------------------------------------------------
template <int MT, int NWN, int NWK, int TPW, int PH, int EPI>
__global__ void __launch_bounds__(NWN * NWK * 64) gemm_rowpar_kernel(RowParArgs a, const uint4* __restrict__ wp, int N, int KT) {
    constexpr int NW = NWN * NWK;
    constexpr int KTP = NWK * TPW;            // k-tiles per phase (MT*KTP <= 32: one x image <= 64 KiB)
    constexpr int NBUF = PH > 1 ? 2 : 1;      // x images resident at once
    constexpr int IMG = 2 * MT * KTP;         // 1 KiB fragments per x image: [2 planes][MT][KTP]
    constexpr int NR = 16 * MT;               // rows per workgroup
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    uint4* lds_x = reinterpret_cast<uint4*>(smem_raw);                                  // [NBUF][IMG][64]
    // the cross-wave reduction buffer aliases the x image (dead after the last compute; one extra barrier)
    f32x4* red = reinterpret_cast<f32x4*>(smem_raw);                                    // [NW][MT][64]
    constexpr size_t kMainBytes = (size_t)NBUF * IMG * 1024 > (size_t)NW * MT * 1024 ? (size_t)NBUF * IMG * 1024 : (size_t)NW * MT * 1024;
    float* sred = reinterpret_cast<float*>(smem_raw + kMainBytes);                      // [NWN][NR] / rinv partials [4][NR]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l15 = lane & 15, grp = lane >> 4;
    const int wn = wave / NWK, wk = wave % NWK;
    const int ntiles = N >> 4;
    const int ntile = min((int)blockIdx.x * NWN + wn, ntiles - 1);
    const int m0 = blockIdx.z * NR;
    const int kb = blockIdx.y * (PH * KTP);   // first k-tile of this workgroup's K slice (split-K over blockIdx.y)
    const int M = a.M;

    // every weight fragment of this wave, all phases, issued before anything else (HBM -> VGPR)
    uint4 w[PH][TPW];
#pragma unroll
    for (int p = 0; p < PH; ++p)
#pragma unroll
        for (int t = 0; t < TPW; ++t) w[p][t] = wp[((size_t)ntile * KT + kb + p * KTP + wk * TPW + t) * 64 + lane];

    int xrows[MT];
#pragma unroll
    for (int b = 0; b < MT; ++b) xrows[b] = min(m0 + b * 16 + l15, M - 1);
    auto stage = [&](int p, int buf) {
#pragma unroll
        for (int i = 0; i < IMG / NW; ++i) {
            const int f = wave + i * NW;
            const int plane = f / (MT * KTP);
            const int rem = f - plane * (MT * KTP);
            const int mt = rem / KTP, k = rem - mt * KTP;
            const uint16_t* src = (plane ? a.xl : a.xh) + (size_t)xrows[mt] * a.ldx + (size_t)(kb + p * KTP + k) * 32 + grp * 8;
            __builtin_amdgcn_global_load_lds((gptr_t)src, (lptr_t)(lds_x + (size_t)(buf * IMG + f) * 64), 16, 0, 0);
        }
    };
    f32x4 acc[MT];
#pragma unroll
    for (int b = 0; b < MT; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](const uint4 (&wf)[TPW], int buf) {
#pragma unroll
        for (int t = 0; t < TPW; ++t) {
            const int kl = wk * TPW + t;
            const bf16x8 wv = __builtin_bit_cast(bf16x8, wf[t]);
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const bf16x8 bh = __builtin_bit_cast(bf16x8, lds_x[(size_t)(buf * IMG + (0 * MT + b) * KTP + kl) * 64 + lane]);
                const bf16x8 bl = __builtin_bit_cast(bf16x8, lds_x[(size_t)(buf * IMG + (1 * MT + b) * KTP + kl) * 64 + lane]);
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, bh, acc[b], 0, 0, 0);
                acc[b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, bl, acc[b], 0, 0, 0);
            }
        }
    };
    // x images: the first two phases are in flight together with the weights (one memory round trip for short K);
    // later phases are staged into the buffer that was just consumed
    stage(0, 0);
    if constexpr (PH > 1) stage(1, 1);
    // epilogue operands are independent of the product: fetch them now, behind the streaming loads
    const bool tile_ok = ((int)blockIdx.x * NWN + wn) < ntiles;
    float4 r4[MT], nw4 = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int b = 0; b < MT; ++b) r4[b] = make_float4(0.f, 0.f, 0.f, 0.f);
    if constexpr (EPI == 0) {
        if (wk == 0 && tile_ok) {
            nw4 = *reinterpret_cast<const float4*>(a.next_w + (size_t)ntile * 16 + grp * 4);
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const int row = m0 + b * 16 + l15;
                if (row < M) r4[b] = *reinterpret_cast<const float4*>(a.resid_in + (size_t)row * N + (size_t)ntile * 16 + grp * 4);
            }
        }
    }
    if constexpr (EPI == 1) rownorm_partials<NR>(a.rn, m0, M, sred);
    dma_publish_barrier();
#pragma unroll
    for (int p = 0; p < PH; ++p) {
        compute(w[p], p & 1);
        if (p + 2 < PH) {
            __syncthreads();  // WAR: all waves are done with buffer p&1
            stage(p + 2, p & 1);
        }
        if (p + 1 < PH && p >= 1) dma_publish_barrier();  // phase p+1 (staged after the first barrier) landed
    }
    __syncthreads();  // every wave is done reading the x image: it becomes the reduction buffer
#pragma unroll
    for (int b = 0; b < MT; ++b) red[(size_t)(wave * MT + b) * 64 + lane] = acc[b];
    __syncthreads();
    if (wk == 0) {
#pragma unroll
        for (int k = 1; k < NWK; ++k)
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const f32x4 v = red[(size_t)((wn * NWK + k) * MT + b) * 64 + lane];
                acc[b][0] += v[0]; acc[b][1] += v[1]; acc[b][2] += v[2]; acc[b][3] += v[3];
            }
    }
    if constexpr (EPI == 0) {
        if (wk == 0) {
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const int row = m0 + b * 16 + l15;
                float ssq_part = 0.f;
                if (tile_ok && row < M) {
                    const size_t o = (size_t)row * N + (size_t)ntile * 16 + grp * 4;
                    const float s0 = acc[b][0] + r4[b].x, s1 = acc[b][1] + r4[b].y, s2 = acc[b][2] + r4[b].z, s3 = acc[b][3] + r4[b].w;
                    *reinterpret_cast<float4*>(a.resid_out + o) = make_float4(s0, s1, s2, s3);
                    uint16_t h0, h1, h2, h3, l0, l1, l2, l3;
                    split_bf16(s0 * nw4.x, h0, l0); split_bf16(s1 * nw4.y, h1, l1); split_bf16(s2 * nw4.z, h2, l2); split_bf16(s3 * nw4.w, h3, l3);
                    *reinterpret_cast<uint2*>(a.oh + o) = make_uint2(h0 | ((uint32_t)h1 << 16), h2 | ((uint32_t)h3 << 16));
                    *reinterpret_cast<uint2*>(a.ol + o) = make_uint2(l0 | ((uint32_t)l1 << 16), l2 | ((uint32_t)l3 << 16));
                    ssq_part = s0 * s0 + s1 * s1 + s2 * s2 + s3 * s3;
                }
                ssq_part += __shfl_xor(ssq_part, 16);
                ssq_part += __shfl_xor(ssq_part, 32);
                if (grp == 0) sred[wn * NR + b * 16 + l15] = ssq_part;
            }
        }
        __syncthreads();
        if (wave == 0) {
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const int row = m0 + b * 16 + l15;
                if (grp == 0 && row < M) {
                    float t = 0.f;
#pragma unroll
                    for (int k = 0; k < NWN; ++k) t += sred[k * NR + b * 16 + l15];
                    a.ssq[(size_t)blockIdx.x * a.ssq_stride + row] = t;
                }
            }
        }
    } else if constexpr (EPI == 1) {
        // SwiGLU: even n-tile of a pair = gate, odd = up of the same 16 features (interleaved weight)
        static_assert(EPI != 1 || (NWN % 2 == 0), "SwiGLU epilogue pairs two n-tiles");
        // odd n-tile waves (up) park their sums in their own slots; the even (gate) wave of the pair finishes
        if (wk == 0 && (wn & 1)) {
#pragma unroll
            for (int b = 0; b < MT; ++b) red[(size_t)((wn * NWK) * MT + b) * 64 + lane] = acc[b];
        }
        __syncthreads();
        const int pair = (int)blockIdx.x * (NWN / 2) + (wn >> 1);  // activation feature tile
        if (wk == 0 && !(wn & 1) && (pair * 2 + 1) < ntiles) {
            const int I = N >> 1;
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const int row = m0 + b * 16 + l15;
                if (row >= M) continue;
                const f32x4 up = red[(size_t)(((wn + 1) * NWK) * MT + b) * 64 + lane];
                const float ri = rownorm_rinv_lds<NR>(a.rn, sred, b * 16 + l15);
                uint16_t h[4], l[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float g = acc[b][r] * ri, u = up[r] * ri;
                    split_bf16(glu_mul(g, u, a.glu), h[r], l[r]);
                }
                const size_t o = (size_t)row * I + (size_t)pair * 16 + grp * 4;
                *reinterpret_cast<uint2*>(a.oh + o) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                *reinterpret_cast<uint2*>(a.ol + o) = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
            }
        }
    } else {
        if (wk == 0 && tile_ok) {
            float* o = a.out + (size_t)blockIdx.y * (size_t)M * N;  // split-K partial slab
#pragma unroll
            for (int b = 0; b < MT; ++b) {
                const int row = m0 + b * 16 + l15;
                if (row < M)
                    *reinterpret_cast<float4*>(o + (size_t)row * N + (size_t)ntile * 16 + grp * 4) = make_float4(acc[b][0], acc[b][1], acc[b][2], acc[b][3]);
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------
// Row-parallel projection, register-direct form (decode, K <= 4096): one workgroup = 16 rows x NT n-tiles for
// the WHOLE K, its NWK waves each own TK k-tiles of every n-tile.  No x image in LDS and no phases: a wave's
// weight fragments (NT*TK KiB) and its own x fragments (2*TK KiB, read by no other wave of the workgroup) all
// go HBM/L2 -> VGPR in one round trip, the K slices meet in LDS once, wave t finishes n-tile t.
// Measured on MI355X (tools/probe_l2.py, weights L2-warm): every LDS phase of the staged kernel above costs
// 1.5-2 us of dependent latency; this form has none.  Epilogues as gemm_rowpar_kernel.
// With more (row block, n-group) pairs than CUs a workgroup keeps its weight fragments and walks row blocks blockIdx.z,
// + gridDim.z, ...; the next block's rows are on their way while the K slices of the current one meet.  A second round of workgroups
// would fetch its weights again behind the first one's tail.  Qwen3-0.6B, the four products of a layer: 117 rows 38.6 -> 35.9 us (gate/up
// 13.1 -> 11.5), 200 rows 83 (chunked kernel) -> 50 us.
// ---------------------------------------------------------------------------------------------------
constexpr int kRowDirBlocks = 4;  // most row blocks of a workgroup
constexpr int kSumIn = 3, kSumRows = 4;  // most partial sums and rows of launch_gemm_rowsum
// SUM: its rows (at most), the residual stream plus the partial sums a.in, are made here (launch_gemm_rowsum).  k_base: the workgroup's first k-tile, slab: where its sums go
template <int NT, int NWK, int TK, int EPI, bool LOOP, int SUM = 0>
__device__ __forceinline__ void rowdir_body(const RowParArgs& a, const uint4* __restrict__ wp, int N, int KT, int group, int k_base = 0, size_t slab = 0) {
    constexpr int UNROLL = LOOP ? 4 : NWK;  // LDS reads at once where the K slices meet: beside the kept weights all of them would spill
    static_assert(NT <= NWK, "wave t finishes n-tile t");
    constexpr int NR = 16;
    // sred: [NT][16] ssq partials (epilogue 0) or [4][16] rinv partials of every row block (epilogue 1)
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    f32x4* red = reinterpret_cast<f32x4*>(smem_raw);                                // [NWK][NT][64]
    float* sred = reinterpret_cast<float*>(smem_raw + (size_t)NWK * NT * 1024);     // [NS][16]
    [[maybe_unused]] float* head_ss = sred + 4 * NR;   // epilogue 5: [NT][16]
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l15 = lane & 15, grp = lane >> 4;
    const int ntiles = N >> 4;
    const int tile0 = group * NT;
    int m0 = blockIdx.z * NR;
    const int M = a.M, m_step = LOOP ? gridDim.z * NR : 1 << 30;
    const int k0 = k_base + wave * TK;
    NVLLM_STAMP(a, 0);

    uint4 w[NT][TK];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int nt = min(tile0 + t, ntiles - 1);
#pragma unroll
        for (int j = 0; j < TK; ++j) w[t][j] = wp[((size_t)nt * KT + k0 + j) * 64 + lane];
    }
    uint4 xh[TK], xl[TK];
    auto load_x = [&](int m) {
        // row-major: 16 rows x 64 B per wave-load; packed: one contiguous 1 KiB fragment (rows >= M of the last
        // block hold stale finite-or-not values whose products are never stored)
        const size_t xo = a.x_packed ? (((size_t)(m >> 4) * KT + k0) << 9) + (size_t)lane * 8
                                     : (size_t)min(m + l15, M - 1) * a.ldx + (size_t)k0 * 32 + grp * 8;
        const int xs = a.x_packed ? 512 : 32;
#pragma unroll
        for (int j = 0; j < TK; ++j) {
            xh[j] = *reinterpret_cast<const uint4*>(a.xh + xo + j * xs);
            xl[j] = *reinterpret_cast<const uint4*>(a.xl + xo + j * xs);
        }
    };
    // SUM: a lane is a column of the wave's 64
    [[maybe_unused]] float part[kSumIn][SUM ? SUM : 1], stream[SUM ? SUM : 1], weight = 0.f;
    if constexpr (SUM) {
        static_assert(SUM == 0 || (TK == 2 && SUM <= 4 * NT), "a wave's columns are its lanes, its rows' planes fit its place of red");
        const size_t col = (size_t)k0 * 32 + lane;
        weight = a.next_w[col];
#pragma unroll
        for (int r = 0; r < SUM; ++r) {
            const size_t at = (size_t)min(r, M - 1) * a.ldx + col;
            stream[r] = a.resid_in[at];
#pragma unroll
            for (int p = 0; p < kSumIn; ++p) part[p][r] = a.in[(size_t)min(p, a.n_in - 1) * a.in_stride + at];
        }
    } else load_x(m0);
    // epilogue operands of the finishing waves (independent of the product): behind the streaming loads
    const int ntile = min(tile0 + wave, ntiles - 1);
    const bool fin = wave < NT && (tile0 + wave) < ntiles;
    float4 r4 = make_float4(0.f, 0.f, 0.f, 0.f), nw4 = make_float4(0.f, 0.f, 0.f, 0.f);
    auto load_resid = [&](int m) { return *reinterpret_cast<const float4*>(a.resid_in + (size_t)min(m + l15, M - 1) * N + (size_t)ntile * 16 + grp * 4); };
    if constexpr (EPI == 0) {
        if (fin) {
            nw4 = *reinterpret_cast<const float4*>(a.next_w + (size_t)ntile * 16 + grp * 4);
            r4 = load_resid(m0);
        }
    }
    // epilogue 5: this row's position and cache block
    [[maybe_unused]] int pos = 0, blk = 0;
    if constexpr (EPI == 5) {
        static_assert(EPI != 5 || (NT == 8 && !LOOP), "a workgroup's features are one head of 128");
        if (wave < NT) {
            const int r = min(m0 + l15, M - 1);
            pos = a.q.pos[r];
            blk = a.q.block_tables[(size_t)a.q.slot[r] * a.q.max_blocks + (pos >> 8)];
        }
    }
    if constexpr (EPI == 1 && LOOP) rownorm_partials_blocks<NR>(a.rn, m0, m_step, M, sred);
    if constexpr ((EPI == 1 || EPI == 5) && !LOOP && !SUM) rownorm_partials<NR>(a.rn, m0, M, sred);
    __builtin_amdgcn_sched_barrier(0);  // every load above is issued before the first use below (one round trip)
    NVLLM_STAMP(a, 1);
    if constexpr (SUM) {
        uint16_t* planes = reinterpret_cast<uint16_t*>(smem_raw + wave * (NT * 1024));  // the wave's [hi, lo][SUM][64], where its sums go later
#pragma unroll
        for (int r = 0; r < SUM; ++r) {
            float v = part[0][r];
#pragma unroll
            for (int p = 1; p < kSumIn; ++p) v += p < a.n_in ? part[p][r] : 0.f;
            v += stream[r];
            if (group == 0 && r < M) a.resid_out[(size_t)r * a.ldx + (size_t)k0 * 32 + lane] = v;
            stream[r] = v;
            uint16_t h, l;
            split_bf16(v * weight, h, l);
            planes[r * 64 + lane] = h;
            planes[(SUM + r) * 64 + lane] = l;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the lanes read what others of the wave wrote
        const int at = min(l15, SUM - 1) * 64 + grp * 8;
#pragma unroll
        for (int j = 0; j < TK; ++j) {
            xh[j] = *reinterpret_cast<const uint4*>(planes + at + j * 32);
            xl[j] = *reinterpret_cast<const uint4*>(planes + SUM * 64 + at + j * 32);
        }
        asm volatile("" ::: "memory");
    }
    [[maybe_unused]] auto sum_rinv = [&]() {  // of row l15, behind the barrier
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < NWK; ++k) t += sred[k * NR + min(l15, SUM - 1)];
        return 1.0f / sqrtf(t * a.rn.inv_h + a.rn.eps);
    };

    for (;;) {
    const int row = m0 + l15, m_next = LOOP ? m0 + m_step : M;
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < TK; ++j) {
        const bf16x8 bh = __builtin_bit_cast(bf16x8, xh[j]);
        const bf16x8 bl = __builtin_bit_cast(bf16x8, xl[j]);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const bf16x8 wv = __builtin_bit_cast(bf16x8, w[t][j]);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, bh, acc[t], 0, 0, 0);
            acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, bl, acc[t], 0, 0, 0);
        }
    }
#ifdef NVLLM_STAMPS
    asm volatile("" ::"v"(acc[0][0]));  // the stamp below is taken after the last MFMA's result exists
#endif
    NVLLM_STAMP(a, 2);
    if constexpr (SUM)
#pragma unroll
        for (int r = 0; r < SUM; ++r) {
            const float ss = wave_sum_uniform(stream[r] * stream[r]);
            if (lane == 0) sred[wave * NR + r] = ss;
        }
#pragma unroll
    for (int t = 0; t < NT; ++t) red[(size_t)(wave * NT + t) * 64 + lane] = acc[t];
    float4 r4_next = r4;
    if (m_next < M) {  // the same for the whole workgroup
        load_x(m_next);
        if constexpr (EPI == 0)
            if (fin) r4_next = load_resid(m_next);
        __builtin_amdgcn_sched_barrier(0);
    }
    // epilogue 5: what the rotation and the norm of this wave's 16 features and of those it is paired with need
    [[maybe_unused]] f32x4 cs, sn, w_own, w_other;
    if constexpr (EPI == 5) {
        if (wave < NT && group < a.q.nh_l + a.q.kv.kv_l) {
            const float* w8 = group < a.q.nh_l ? a.q.qn : a.q.kn;
            const size_t at = (size_t)pos * 64 + (wave & 3) * 16 + grp * 4;
            cs = *reinterpret_cast<const f32x4*>(a.q.cos + at);
            sn = *reinterpret_cast<const f32x4*>(a.q.sin + at);
            w_own = *reinterpret_cast<const f32x4*>(w8 + wave * 16 + grp * 4);
            w_other = *reinterpret_cast<const f32x4*>(w8 + (wave ^ 4) * 16 + grp * 4);
        }
    }
    __syncthreads();
    NVLLM_STAMP(a, 3);
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    if (wave < NT) {
#pragma unroll UNROLL
        for (int k = 0; k < NWK; ++k) {
            const f32x4 v = red[(size_t)(k * NT + wave) * 64 + lane];
            sum[0] += v[0]; sum[1] += v[1]; sum[2] += v[2]; sum[3] += v[3];
        }
    }
    if constexpr (EPI == 0) {
        if (wave < NT) {
            float ssq_part = 0.f;
            if (fin && row < M) {
                const size_t o = (size_t)row * N + (size_t)ntile * 16 + grp * 4;
                const float s0 = sum[0] + r4.x, s1 = sum[1] + r4.y, s2 = sum[2] + r4.z, s3 = sum[3] + r4.w;
                *reinterpret_cast<float4*>(a.resid_out + o) = make_float4(s0, s1, s2, s3);
                uint16_t h0, h1, h2, h3, l0, l1, l2, l3;
                split_bf16(s0 * nw4.x, h0, l0); split_bf16(s1 * nw4.y, h1, l1); split_bf16(s2 * nw4.z, h2, l2); split_bf16(s3 * nw4.w, h3, l3);
                const size_t ob = a.o_packed ? xpack_off(row, ntile * 16 + grp * 4, N >> 5) : o;
                *reinterpret_cast<uint2*>(a.oh + ob) = make_uint2(h0 | ((uint32_t)h1 << 16), h2 | ((uint32_t)h3 << 16));
                *reinterpret_cast<uint2*>(a.ol + ob) = make_uint2(l0 | ((uint32_t)l1 << 16), l2 | ((uint32_t)l3 << 16));
                ssq_part = s0 * s0 + s1 * s1 + s2 * s2 + s3 * s3;
            }
            ssq_part += __shfl_xor(ssq_part, 16);
            ssq_part += __shfl_xor(ssq_part, 32);
            if constexpr (NT == 1) {
                if (grp == 0 && row < M) a.ssq[(size_t)group * a.ssq_stride + row] = ssq_part;
            } else {
                if (grp == 0) sred[wave * NR + l15] = ssq_part;
            }
        }
        if constexpr (NT > 1) {
            __syncthreads();
            if (wave == 0 && grp == 0 && row < M) {
                float t = 0.f;
#pragma unroll
                for (int k = 0; k < NT; ++k) t += sred[k * NR + l15];
                a.ssq[(size_t)group * a.ssq_stride + row] = t;
            }
        }
    } else if constexpr (EPI == 1) {
        static_assert(EPI != 1 || (NT % 2 == 0), "SwiGLU epilogue pairs two n-tiles");
        // odd tiles (up) park their sums in slot [0][t]; the even (gate) wave of the pair finishes
        __syncthreads();  // every finishing wave is done reading red
        if (wave < NT && (wave & 1)) red[(size_t)wave * 64 + lane] = sum;
        __syncthreads();
        const int pair = (tile0 + wave) >> 1;  // activation feature tile
        if (wave < NT && !(wave & 1) && (tile0 + wave + 1) < ntiles && row < M) {
            const int I = N >> 1;
            const f32x4 up = red[(size_t)(wave + 1) * 64 + lane];
            const float ri = SUM ? sum_rinv() : rownorm_rinv_lds<NR>(a.rn, sred, l15);
            uint16_t h[4], l[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float g = sum[r] * ri, u = up[r] * ri;
                split_bf16(glu_mul(g, u, a.glu), h[r], l[r]);
            }
            const size_t o = a.o_packed ? xpack_off(row, pair * 16 + grp * 4, I >> 5) : (size_t)row * I + (size_t)pair * 16 + grp * 4;
            *reinterpret_cast<uint2*>(a.oh + o) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
            *reinterpret_cast<uint2*>(a.ol + o) = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
        }
    } else if constexpr (EPI == 5) {
        // qwen3.rs:208-234 on the head: norm over its 128 features (q, k), half-split rotation (features d and d + 64: tiles t and t + 4),
        // then q to the f32 buffer and k, v into the cache.  The f32 sums' way through memory and the row kernel's launch (4.5 us and the gap
        // before it) for a longer epilogue: rule and figures at gemm_rowdir_qkv_ok
        const QkvArgs& q = a.q;
        const int head = group;
        const float ri = rownorm_rinv_lds<NR>(a.rn, sred, l15);
        __syncthreads();  // every finishing wave is done reading red
        if (wave < NT) {
#pragma unroll
            for (int r = 0; r < 4; ++r) sum[r] *= ri;
            red[(size_t)wave * 64 + lane] = sum;
            float ss = (sum[0] * sum[0] + sum[1] * sum[1]) + (sum[2] * sum[2] + sum[3] * sum[3]);
            ss += __shfl_xor(ss, 16);
            ss += __shfl_xor(ss, 32);
            if (grp == 0) head_ss[wave * NR + l15] = ss;
        }
        __syncthreads();
        if (wave < NT && row < M) {
            const int kv_l = q.kv.kv_l, f0 = wave * 16 + grp * 4;
            if (head < q.nh_l + kv_l) {
                float ss = 0.f;
#pragma unroll
                for (int k = 0; k < NT; ++k) ss += head_ss[k * NR + l15];
                const float rinv = 1.0f / sqrtf(ss / 128.0f + q.eps), turn = wave < 4 ? -1.0f : 1.0f;
                const f32x4 other = red[(size_t)(wave ^ 4) * 64 + lane];
#pragma unroll
                for (int r = 0; r < 4; ++r) sum[r] = (sum[r] * rinv) * w_own[r] * cs[r] + turn * ((other[r] * rinv) * w_other[r] * sn[r]);
            }
            if (head < q.nh_l) {
                *reinterpret_cast<float4*>(q.q_out + (size_t)row * (q.nh_l * 128) + (size_t)head * 128 + f0) =
                    make_float4(sum[0] * q.q_scale, sum[1] * q.q_scale, sum[2] * q.q_scale, sum[3] * q.q_scale);
            } else {
                const bool is_k = head < q.nh_l + kv_l;
                const size_t slab = (size_t)(blk * kv_l + head - q.nh_l - (is_k ? 0 : kv_l)) * kBlockTokens * 128;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    if (is_k) store_k24(reinterpret_cast<_Float16*>(q.kv.k) + slab, q.kv.klo ? q.kv.klo + slab : nullptr, pos & 255, f0 + r, 128, sum[r]);
                    else store_v24(reinterpret_cast<_Float16*>(q.kv.v) + slab, q.kv.vlo ? q.kv.vlo + slab : nullptr, pos & 255, f0 + r, 128, sum[r]);
                }
            }
        }
    } else if constexpr (EPI >= 3) {
        if (fin && row < M) {
            uint16_t h[4], l[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) split_bf16(act_of<EPI - 3>(sum[r]), h[r], l[r]);
            const int f0 = ntile * 16 + grp * 4;
            const size_t o = a.o_packed ? xpack_off(row, f0, N >> 5) : (size_t)row * N + f0;
            *reinterpret_cast<uint2*>(a.oh + o) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
            *reinterpret_cast<uint2*>(a.ol + o) = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
        }
    } else {
        if (fin && row < M) {
            const float f = SUM ? sum_rinv() : 1.f;
            *reinterpret_cast<float4*>(a.out + slab + (size_t)row * N + (size_t)ntile * 16 + grp * 4) = make_float4(sum[0] * f, sum[1] * f, sum[2] * f, sum[3] * f);
        }
    }
    NVLLM_STAMP(a, 4);
    if (m_next >= M) break;
    __syncthreads();  // red and sred are read
    m0 = m_next;
    if constexpr (EPI == 1) sred += 4 * NR;
    r4 = r4_next;
    }
}
template <int NT, int NWK, int TK, int EPI>
__global__ void __launch_bounds__(NWK * 64) gemm_rowdir_kernel(RowParArgs a, const uint4* __restrict__ wp, int N, int KT) {
    rowdir_body<NT, NWK, TK, EPI, false>(a, wp, N, KT, blockIdx.x);
}
template <int NT, int NWK, int TK, int EPI>
__global__ void __launch_bounds__(NWK * 64) gemm_rowdir_loop_kernel(RowParArgs a, const uint4* __restrict__ wp, int N, int KT) {
    rowdir_body<NT, NWK, TK, EPI, true>(a, wp, N, KT, blockIdx.x);
}

// One to a few rows (launch_gemm_rowslab, launch_gemm_rowsum).  The residual and norm epilogue wants a whole K in a workgroup, so o_proj and down_proj of one row block are
// 64 workgroups of 64 and 96 KB of weights, whose intake is what sets them apart from the 256 workgroups of 32 KB of the QKV product.  Cut into slices of 1024
// they are 128 and 192 workgroups, and their consumers add up the slabs: two or three more rows of f32 to read, a column a lane (as B fragments, 16 bytes
// a lane with fifteen rows of none, they were 320 loads a workgroup and 3 us).  One row, us by trace: o 4.6 -> 3.7, down 6.0 -> 4.1, gate/up 5.8 the same, q/k/v 3.9 -> 4.7.
template <int TK>
__global__ void __launch_bounds__(1024) gemm_rowslab_kernel(RowParArgs a, const uint4* __restrict__ wp, int N, int KT) {
    rowdir_body<1, 16, TK, 2, false>(a, wp, N, KT, blockIdx.x, blockIdx.y * 16 * TK, (size_t)blockIdx.y * a.M * N);
}
template <int NT, int EPI, int ROWS>
__global__ void __launch_bounds__(1024) gemm_rowsum_kernel(RowParArgs a, const uint4* __restrict__ wp, int N, int KT) {
    rowdir_body<NT, 16, 2, EPI, false, ROWS>(a, wp, N, KT, blockIdx.x);
}

// Two plain products of the same rows in one launch, where neither needs the other (the projections of a layer's two branches, whose outputs
// the next norm adds up): workgroups below groups_a make the first.  Each alone is a launch's latency on a quarter of the chip: 24 rows, 1024
// features of K 2048 and of K 3072, 5.2 and 6.5 us and the boundary between them, together 7.1.  A step of six layers with each of the nine pairs of
// K that gemm_rowdir_two_ok takes, 256 to 2048 features, 1 to 64 rows: 2.1 to 7.6 us a layer less, 1024 features 2.4 (K 1024 + 2048, 4
// rows) to 7.5 (K 3072 + 2048, 64).
template <int NTA, int TKA, int NTB, int TKB>
__global__ void __launch_bounds__(1024) gemm_rowdir_two_kernel(RowParArgs a, const uint4* __restrict__ wa, int NA, int groups_a, RowParArgs b, const uint4* __restrict__ wb, int NB) {
    if ((int)blockIdx.x < groups_a) rowdir_body<NTA, 16, TKA, 2, false>(a, wa, NA, 16 * TKA, blockIdx.x);
    else rowdir_body<NTB, 16, TKB, 2, false>(b, wb, NB, 16 * TKB, (int)blockIdx.x - groups_a);
}

// Register-direct products of 65 to 896 rows: RB row blocks at a time (blocks z, z + gz, ... of blockIdx.z = z), K split over NWK waves, the
// weights kept.  Bound by what a CU takes in (x and W of its workgroup, 0.4 to 0.6 MB) and by the phases of a round: products, K slices to
// LDS, their sums, the epilogue.  Eight waves instead of sixteen halve the slices and have registers for two blocks, so that a round's phases
// serve 32 rows; gate and up of a feature meet in one wave; two n-tiles of o and down halve the rows a workgroup takes in.  0.6B, us a launch,
// the 16-wave loop / this: 200 rows q/k/v 10.0 / 8.8, gate/up 15.0 / 12.4, o and down 12.5 / 9.6 each; 117 rows gate/up 11.6 / 9.8, o and down
// 8.6 / 7.6; 250 rows 10.4 / 9.2, 15.5 / 12.7, 12.9 / 10.1.
// Past 256 rows a round more to every 128 rows, against tile products with K slices, whose slabs are launches more, and which fill and drain a CU for a few stages: up to where o and down are one
// launch each as tiles too (tile_resid_kernel).  A prompt of 0.6B, ms, tile products / these: 257 tokens 2.63 / 1.94, 300 2.67 / 1.98, 384 2.84 / 2.04, 480 2.88 / 2.34; a step of 257 rows 3.30 / 2.49.
// Past 480 q/k/v and gate/up alone: 481 tokens 2.91 / 2.60, 512 2.93 / 2.62, 640 3.25 / 2.88, 768 3.36 / 3.10, 896 3.45 / 3.30, 897 3.45 / 3.43, 1024 3.53 / 3.52.
// But only while the CUs hold all of their workgroups at once: 16 blocks each at most makes it more than that of wide layers.  A prompt of 12 layers, ms, tile products / these, the last row count in one round and
// the first in two: gate/up of 9216 features 512 rows 1.36 / 1.35 and 528 1.40 / 1.54, of 6912 768 1.45 / 1.40 and 832 1.47 / 1.65; q/k/v of 5120 768 1.58 / 1.51 and 832 1.64 / 1.72, of 6144 512 1.45 / 1.32 and
// 528 1.46 / 1.44 (640 1.49 / 1.53, 896 1.68 / 1.77), of 9216, never in one, 512 1.52 / 1.56 and 896 1.80 / 2.02.
template <int NT, int NWK, int TK, int RB, int EPI>
__global__ void __launch_bounds__(NWK * 64) gemm_rowpair_kernel(RowParArgs a, const uint4* __restrict__ wp, int N, int KT) {
    constexpr int NR = 16, PER = EPI == 1 ? 2 : 1, UNITS = RB * NT / PER, UPW = (UNITS + NWK - 1) / NWK;  // a unit: a row block's n-tile, or its gate and up
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    f32x4* red = reinterpret_cast<f32x4*>(smem_raw);                                     // [NWK][RB][NT][64]
    float* sred = reinterpret_cast<float*>(smem_raw + (size_t)NWK * RB * NT * 1024);     // [row block][4][16] rinv partials (epilogue 1)
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l15 = lane & 15, grp = lane >> 4;
    const int tile0 = (int)blockIdx.x * NT, k0 = wave * TK, M = a.M;
    const int blocks = (M + NR - 1) / NR, gz = gridDim.z;
    uint4 w[NT][TK];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < TK; ++j) w[t][j] = wp[((size_t)(tile0 + t) * KT + k0 + j) * 64 + lane];
    uint4 xh[RB][TK], xl[RB][TK];
    auto load_x = [&](int blk) {  // a block past the end: the last one again, its products are not stored
#pragma unroll
        for (int b = 0; b < RB; ++b) {
            const size_t xo = (((size_t)min(blk + b * gz, blocks - 1) * KT + k0) << 9) + (size_t)lane * 8;
#pragma unroll
            for (int j = 0; j < TK; ++j) {
                xh[b][j] = *reinterpret_cast<const uint4*>(a.xh + xo + j * 512);
                xl[b][j] = *reinterpret_cast<const uint4*>(a.xl + xo + j * 512);
            }
        }
    };
    int blk = blockIdx.z;
    load_x(blk);
    // a unit's residual rows (epilogue 0) come behind the streams
    float4 r4[UPW], nw4[UPW];
    auto load_resid = [&](int blk_) {
#pragma unroll
        for (int i = 0; i < UPW; ++i) {
            const int u = min(wave + i * NWK, UNITS - 1), b = u / NT, t = u - b * NT;
            const int row = min((blk_ + b * gz) * NR + l15, M - 1);
            r4[i] = *reinterpret_cast<const float4*>(a.resid_in + (size_t)row * N + (size_t)(tile0 + t) * 16 + grp * 4);
            nw4[i] = *reinterpret_cast<const float4*>(a.next_w + (size_t)(tile0 + t) * 16 + grp * 4);
        }
    };
    if constexpr (EPI == 0) load_resid(blk);
    if constexpr (EPI == 1) {
        rownorm_partials_blocks<NR>(a.rn, blk * NR, gz * NR, M, sred);
        if (blk + NWK * gz < blocks) rownorm_partials_blocks<NR>(a.rn, (blk + NWK * gz) * NR, gz * NR, M, sred + NWK * 4 * NR);
    }
    __builtin_amdgcn_sched_barrier(0);
    for (;;) {
        const int next = blk + RB * gz;
        f32x4 acc[RB][NT];
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int t = 0; t < NT; ++t) acc[b][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int j = 0; j < TK; ++j) {
                const bf16x8 bh = __builtin_bit_cast(bf16x8, xh[b][j]), bl = __builtin_bit_cast(bf16x8, xl[b][j]);
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const bf16x8 wv = __builtin_bit_cast(bf16x8, w[t][j]);
                    acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, bh, acc[b][t], 0, 0, 0);
                    acc[b][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv, bl, acc[b][t], 0, 0, 0);
                }
            }
#pragma unroll
        for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int t = 0; t < NT; ++t) red[(size_t)((wave * RB + b) * NT + t) * 64 + lane] = acc[b][t];
        const bool more = next < blocks;  // the same for the whole workgroup
        if (more) {
            load_x(next);
            __builtin_amdgcn_sched_barrier(0);
        }
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (not a wait for the loads in flight)
#pragma unroll
        for (int i = 0; i < UPW; ++i) {
            const int u = wave + i * NWK;
            if (UNITS % NWK && u >= UNITS) break;
            const int b = u / (NT / PER), t = (u - b * (NT / PER)) * PER, ntile = tile0 + t;
            const int row = (blk + b * gz) * NR + l15;
            f32x4 sum[PER];
#pragma unroll
            for (int q = 0; q < PER; ++q) {
                sum[q] = red[(size_t)(b * NT + t + q) * 64 + lane];
#pragma unroll
                for (int k = 1; k < NWK; ++k) sum[q] += red[(size_t)((k * RB + b) * NT + t + q) * 64 + lane];
            }
            if constexpr (EPI == 0) {
                float ssq_part = 0.f;
                if (row < M) {
                    const size_t o = (size_t)row * N + (size_t)ntile * 16 + grp * 4;
                    const float s0 = sum[0][0] + r4[i].x, s1 = sum[0][1] + r4[i].y, s2 = sum[0][2] + r4[i].z, s3 = sum[0][3] + r4[i].w;
                    *reinterpret_cast<float4*>(a.resid_out + o) = make_float4(s0, s1, s2, s3);
                    uint16_t h[4], l[4];
                    split_bf16(s0 * nw4[i].x, h[0], l[0]); split_bf16(s1 * nw4[i].y, h[1], l[1]); split_bf16(s2 * nw4[i].z, h[2], l[2]); split_bf16(s3 * nw4[i].w, h[3], l[3]);
                    const size_t ob = a.o_packed ? xpack_off(row, ntile * 16 + grp * 4, N >> 5) : o;
                    *reinterpret_cast<uint2*>(a.oh + ob) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                    *reinterpret_cast<uint2*>(a.ol + ob) = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
                    ssq_part = s0 * s0 + s1 * s1 + s2 * s2 + s3 * s3;
                }
                ssq_part += __shfl_xor(ssq_part, 16);
                ssq_part += __shfl_xor(ssq_part, 32);
                if (grp == 0 && row < M) a.ssq[(size_t)ntile * a.ssq_stride + row] = ssq_part;  // a group of the norm's sum to a tile
            } else if constexpr (EPI == 1) {
                if (row < M) {
                    const int I = N >> 1, pair = ntile >> 1;
                    const float ri = rownorm_rinv_lds<NR>(a.rn, sred + b * 4 * NR, l15);
                    uint16_t h[4], l[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) split_bf16(glu_mul(sum[0][r] * ri, sum[PER - 1][r] * ri, a.glu), h[r], l[r]);
                    const size_t o = a.o_packed ? xpack_off(row, pair * 16 + grp * 4, I >> 5) : (size_t)row * I + (size_t)pair * 16 + grp * 4;
                    *reinterpret_cast<uint2*>(a.oh + o) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                    *reinterpret_cast<uint2*>(a.ol + o) = make_uint2(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16));
                }
            } else {
                if (row < M)
                    *reinterpret_cast<float4*>(a.out + (size_t)row * N + (size_t)ntile * 16 + grp * 4) = make_float4(sum[0][0], sum[0][1], sum[0][2], sum[0][3]);
            }
        }
        if (!more) break;
        if constexpr (EPI == 0) load_resid(next);
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // red is read
        blk = next;
        if constexpr (EPI == 1) sred += RB * 4 * NR;
    }
}
static std::atomic<int64_t> g_rowpair_launches{0};
int64_t rowpair_launches() { return g_rowpair_launches.load(std::memory_order_relaxed); }
// workgroups that share a product's row blocks: one round of the CUs, 16 blocks each at most, for epilogue 1 holds the norms of two blocks a wave
static int rowpair_groups(int groups, int blocks) { return std::min(blocks, std::max(256 / groups, (blocks + 15) / 16)); }
template <int NT, int NWK, int TK, int RB, int EPI>
static hipError_t rowpair_launch(const RowParArgs& a, const PackedW& w, hipStream_t s) {
    const int groups = w.N / 16 / NT, blocks = (a.M + 15) / 16;
    const size_t lds = (size_t)NWK * RB * NT * 1024 + (EPI == 1 ? (size_t)16 * 64 * 4 : 0);
    static std::atomic<uint64_t> lds_set{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(gemm_rowpair_kernel<NT, NWK, TK, RB, EPI>), lds, lds_set);
    const int gz = rowpair_groups(groups, blocks);
    gemm_rowpair_kernel<NT, NWK, TK, RB, EPI><<<dim3(groups, 1, gz), NWK * 64, lds, s>>>(a, w.data, w.N, w.K / 32);
    g_rowpair_launches.fetch_add(1, std::memory_order_relaxed);
    return hipGetLastError();
}
// Products of 65 to kRowPairRows rows of packed planes whose shape has an instance (else hipErrorNotReady); whether such a product is register-direct at all says rowdir_shape.  Up to 64 rows every workgroup has one block: the
// 16-wave forms below are as fast or faster there (64 rows, gate/up 8.1 us against 10.6, o 4.8 against 5.6).  So they are, for q/k/v and gate/up,
// while the grid gives every block its own workgroup, whose second block would be nothing, and for 5 blocks on two workgroups.  A product's time by
// this less the 16-wave form's, us, at 5 to 16 blocks of 1024-wide rows:
//   q/k/v    1536 features +0.5 to +0.9 up to 10 blocks, -0.3 to -0.7 above; 2048 +0.4 to +0.8 up to 8, -0.3 to -0.9; 2560 +0.9 +0.4 up to 6, -0.9 to
//            +0.1; 3072 +0.5 at 5, -1.9 to +0.3; 4096 -1.3 to 0.0; 5120 -4.7 to +0.1; 6144 +0.9 at 5, -4.8 to +0.1
//   gate/up  1536 +0.8 to +1.2, 3072 +0.8 to +1.5 (both up to 8); 4608 +1.4 at 5, -0.8 to -1.1; 6144 -2.5 to -0.4; 9216 +0.9 at 5, -0.6 to -3.9
static bool rowpair_ok(int N, int K, int epi, int M) {
    if (M <= 64 || M > kRowPairRows) return false;
    auto pairs = [&](int nt) {  // row blocks for two at a time
        const int blocks = (M + 15) / 16, room = 256 / (N / 16 / nt);
        return blocks > room && !(room <= 2 && blocks <= 5);
    };
    // epilogue 0, up to 64 tiles: each leaves its own group of the next norm's sum, as the 16-wave form's workgroups do
    if (epi == 0) return N % 32 == 0 && N <= 1024 && (K == 1024 || K == 2048 || K == 3072);
    if (epi == 1) return K == 1024 && N % 96 == 0 && pairs(6);
    return epi == 2 && K == 1024 && N % 64 == 0 && pairs(4);
}
template <int EPI>
static hipError_t rowpair_dispatch(const RowParArgs& a, const PackedW& w, hipStream_t s) {
    if (!a.x_packed || !rowpair_ok(w.N, w.K, EPI, a.M)) return hipErrorNotReady;
    if constexpr (EPI == 0) {
        const bool one = (a.M + 15) / 16 <= 256 / (w.N / 32);  // a block to a workgroup
        if (w.K == 1024) return one ? rowpair_launch<2, 8, 4, 1, 0>(a, w, s) : rowpair_launch<2, 8, 4, 2, 0>(a, w, s);
        if (w.K == 2048) return one ? rowpair_launch<2, 8, 8, 1, 0>(a, w, s) : rowpair_launch<2, 8, 8, 2, 0>(a, w, s);
        return rowpair_launch<2, 8, 12, 1, 0>(a, w, s);
    } else if constexpr (EPI == 1) {
        return rowpair_launch<6, 8, 4, 2, 1>(a, w, s);
    } else {
        return rowpair_launch<4, 8, 4, 2, 2>(a, w, s);
    }
}

// shape of the register-direct kernel for (N, K, epi, M): nt == 0 -> not applicable
struct RowDirShape { int nt, nwk, tk; };
static RowDirShape rowdir_shape(int N, int K, int epi, int M) {
    RowDirShape none{0, 0, 0};
    if (N % 16 || K % 32 || (M > 256 && !rowpair_ok(N, K, epi, M))) return none;
    const int KT = K / 32, ntiles = N / 16;
    if (KT % 16 || KT / 16 < 2 || KT / 16 > 8 || (KT / 16) % 2) return none;  // K in {1024, 2048, 3072, 4096}
    const int tk = KT / 16;
    int nt;
    if (epi == 0) {
        nt = 1;
        while ((ntiles + nt - 1) / nt > 64) nt *= 2;  // deferred-norm consumers sum <= 64 ssq groups
        if (nt > 4 || nt * tk > 16 || (nt == 2 && tk == 8)) return none;
    } else if (epi == 1) {
        nt = (ntiles % 6 == 0 && tk == 2) ? 6 : 4;
        if (ntiles % 2 || nt * tk > 16) return none;
        // one row block (<= 16 rows, e.g. batch 1): the grid is the n-groups alone, so fewer tiles per workgroup put the
        // matrix on more CUs (0.6B gate/up: 64 -> 192 workgroups)
        if (M <= 16 && ntiles / 2 <= 512) nt = 2;
        else if (M <= 32 && nt == 6 && 2 * ((ntiles + 5) / 6) < 256) nt = 4;  // two row blocks: below
    } else {
        nt = 4;
        if (nt * tk > 16) nt = 2;
        if (nt * tk > 16) return none;
        // two row blocks whose workgroups do not fill the chip: fewer tiles each (0.6B QKV 128 -> 256 workgroups, gate/up 128 -> 192).  Steps
        // of 17, 24, 32 rows, 100 to 300 tokens: 1.090 -> 1.041, 1.117 -> 1.064, 1.147 -> 1.091 ms; QKV alone 1.067, 1.087, 1.118, gate/up alone
        // 1.070, 1.092, 1.127, gate/up with two tiles 1.088, 1.109, 1.138; two decoders of other designs 3 to 5 %
        if (M > 16 && M <= 32 && nt == 4 && 2 * ((ntiles + 3) / 4) < 256) nt = 2;
        if (M <= 16 && ntiles <= 512) nt = 1;  // as above (0.6B QKV: 64 -> 256 workgroups)
    }
    // weights are streamed once per row block: big matrices belong to the 64-row kernel
    if ((size_t)N * K * 2 >= ((size_t)24 << 20) && M > 16) return none;
    return RowDirShape{nt, 16, tk};
}

struct RowParShape { int mt, nwn, nwk, tpw, ph, ns; };
// Decomposition of y[M,N] = x.W^T for the row-parallel kernel (false: use the generic kernel).
//   small matrices: 16 rows per workgroup (row blocks re-read the weights through L2), whole K in one workgroup;
//   big matrices (>= 24 MB): all rows (up to 64) in one workgroup so every weight byte crosses L2 once, K sliced
//   into <= 1024-deep pieces over blockIdx.y (plain epilogue only: the slices leave f32 slabs).
static bool rowpar_shape(int N, int K, int epi, int M, RowParShape& sh) {
    if (N % 16 || K % 32 || epi >= 3) return false;
    const int KT = K / 32, ntiles = N / 16;
    const bool big = (size_t)N * K * 2 >= (size_t)24 << 20 && M > 16;
    static const int tpws[] = {8, 12, 16};
    if (big) {
        if (epi != 2) return false;
        const int mt = 4;  // 64 rows: x image 2*4*8 KiB per phase
        for (int ph = 4; ph >= 1; --ph) {
            if (KT % (ph * 8)) continue;
            sh = {mt, (ntiles % 8 == 0) ? 8 : (ntiles % 4 == 0 ? 4 : (ntiles % 2 == 0 ? 2 : 1)), 1, 8, ph, KT / (ph * 8)};
            if ((2 * mt * 8) % sh.nwn) continue;
            return true;
        }
        return false;
    }
    const int mblocks = (std::max(M, 1) + 15) / 16;
    // fewest phases whose x image fits 64 KiB (KTP <= 32 k-tiles), most k-slices per workgroup first
    for (int ph = 1; ph <= 4; ++ph)
        for (int nwk : {4, 2, 1})
            for (int tpw : tpws) {
                if (ph * nwk * tpw != KT || nwk * tpw > 32) continue;
                int nwn = ntiles % 2 == 0 ? 2 : 1;
                // wide projections (QKV, gate/up): 4 n-tiles per workgroup halves the x re-staging and keeps the
                // whole grid resident in one round -- only where it still leaves >= 192 workgroups
                if (epi != 0 && ph == 1 && nwk == 4 && tpw == 8 && ntiles % 4 == 0 && (ntiles / 4) * mblocks >= 192) nwn = 4;
                if ((2 * tpw) % nwn) continue;
                sh = {1, nwn, nwk, tpw, ph, 1};
                return true;
            }
    return false;
}
bool gemm_rowpar_supported(int N, int K) {
    RowParShape sh;
    return (rowdir_shape(N, K, 0, 64).nt || rowpar_shape(N, K, 0, 64, sh)) && gemm_rowpar_groups(N, K) <= 64;
}
bool gemm_rowpar_ok(int N, int K, int epi, int M) {
    if (rowdir_shape(N, K, epi, M).nt) return true;
    RowParShape sh;
    return rowpar_shape(N, K, epi, M, sh) && !(epi == 1 && sh.nwn % 2);
}
// ssq groups the epilogue-0 kernel leaves: its tiles per workgroup follow from N and K alone, for any row count of the fused path
int gemm_rowpar_groups(int N, int K) {
    const RowDirShape d = rowdir_shape(N, K, 0, 64);
    if (d.nt) return (N / 16 + d.nt - 1) / d.nt;
    RowParShape sh;
    if (!rowpar_shape(N, K, 0, 64, sh)) return 0;
    return (N / 16 + sh.nwn - 1) / sh.nwn;
}
bool gemm_rowdir_ok(int N, int K, int epi, int M) { return rowdir_shape(N, K, epi, M).nt != 0; }
bool gemm_rowpair_at_once(int N, int K, int epi, int M) {
    if (!rowpair_ok(N, K, epi, M) || !rowdir_shape(N, K, epi, M).nt) return false;
    const int groups = N / 16 / (epi == 0 ? 2 : epi == 1 ? 6 : 4);
    return groups * rowpair_groups(groups, (M + 15) / 16) <= 256;
}
int gemm_rowpar_splits(int N, int K, int epi, int M) {
    if (rowdir_shape(N, K, epi, M).nt) return 1;
    RowParShape sh;
    return rowpar_shape(N, K, epi, M, sh) ? sh.ns : 0;
}

template <int NT, int NWK, int TK, int EPI>
static hipError_t rowdir_launch_t(const RowParArgs& a, const PackedW& w, hipStream_t s) {
    constexpr size_t red = (size_t)NWK * NT * 1024;
    const int groups = (w.N / 16 + NT - 1) / NT, blocks = (a.M + 15) / 16;
    // one round of the 256 CUs where a few row blocks per workgroup make it one, and where the 128 registers of a 1024-thread workgroup
    // hold the weights beside the next block's rows
    if constexpr (EPI != 5 && NT * TK + 2 * TK <= (EPI == 1 || EPI == 2 ? 24 : 18)) {
        if (groups * blocks > 256) {
            const size_t lds = red + (size_t)std::max(NT, 4 * kRowDirBlocks) * 16 * 4;
            static std::atomic<uint64_t> lds_set{0};
            ensure_dyn_lds(reinterpret_cast<const void*>(gemm_rowdir_loop_kernel<NT, NWK, TK, EPI>), lds, lds_set);
            const int each = std::min(kRowDirBlocks, (groups * blocks + 255) / 256);
            gemm_rowdir_loop_kernel<NT, NWK, TK, EPI><<<dim3(groups, 1, (blocks + each - 1) / each), NWK * 64, lds, s>>>(a, w.data, w.N, w.K / 32);
            return hipGetLastError();
        }
    }
    const size_t lds = red + (size_t)(EPI == 5 ? NT + 4 : NT > 4 ? NT : 4) * 16 * 4;
    static std::atomic<uint64_t> lds_set{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(gemm_rowdir_kernel<NT, NWK, TK, EPI>), lds, lds_set);
    gemm_rowdir_kernel<NT, NWK, TK, EPI><<<dim3(groups, 1, blocks), NWK * 64, lds, s>>>(a, w.data, w.N, w.K / 32);
    return hipGetLastError();
}
template <int EPI>
static hipError_t rowdir_dispatch(const RowDirShape& d, const RowParArgs& a, const PackedW& w, hipStream_t s) {
#define NVLLM_RD(NT_, TK_) if (d.nt == NT_ && d.tk == TK_) return rowdir_launch_t<NT_, 16, TK_, EPI>(a, w, s);
    if constexpr (EPI == 0) { NVLLM_RD(1, 2) NVLLM_RD(1, 4) NVLLM_RD(1, 6) NVLLM_RD(1, 8) NVLLM_RD(2, 2) NVLLM_RD(2, 4) NVLLM_RD(2, 6) NVLLM_RD(4, 2) NVLLM_RD(4, 4) }
    if constexpr (EPI == 1) { NVLLM_RD(6, 2) NVLLM_RD(4, 2) NVLLM_RD(4, 4) NVLLM_RD(2, 2) NVLLM_RD(2, 4) NVLLM_RD(2, 6) NVLLM_RD(2, 8) }
    if constexpr (EPI >= 2) { NVLLM_RD(4, 2) NVLLM_RD(4, 4) NVLLM_RD(2, 2) NVLLM_RD(2, 4) NVLLM_RD(2, 6) NVLLM_RD(2, 8) NVLLM_RD(1, 2) NVLLM_RD(1, 4) NVLLM_RD(1, 6) NVLLM_RD(1, 8) }
#undef NVLLM_RD
    return hipErrorNotSupported;
}

// One round of workgroups (a head x 16 rows) that fills more than half the chip: 0.6B prompts of 90, 117 and 128 tokens 1.576 -> 1.521, 1.625 ->
// 1.547 and 1.656 -> 1.563 ms; fewer rows gain nothing (64: 1.321 -> 1.312; 16, where the plain product spreads a head over 8 workgroups, 1.135
// -> 1.199), a second round neither (129: 1.840 -> 1.863, 200: 2.112 -> 2.105).
bool gemm_rowdir_qkv_ok(int N, int K, int hd, int M) {
    const int wgs = N / 128 * ((M + 15) / 16);
    return hd == 128 && K == 1024 && N % 128 == 0 && wgs > 128 && wgs <= 256 && rowdir_shape(N, K, 2, M).nt != 0;
}
hipError_t launch_gemm_rowdir_qkv(const RowParArgs& a, const PackedW& w, hipStream_t s) {
    if (!gemm_rowdir_qkv_ok(w.N, w.K, a.q.kv.hd, a.M) || w.N != (a.q.nh_l + 2 * a.q.kv.kv_l) * 128) return hipErrorNotSupported;
    if (a.q.kv.klo && !a.q.kv.vlo) return hipErrorInvalidValue;  // 24-bit K comes with 24-bit V only
    if (a.M <= 0) return hipSuccess;
    // eight waves halve the K slices that meet in LDS: 117 rows 10.0 -> 9.3 us; row-major fragments, which cost a wave more each, stay with sixteen
    return a.x_packed ? rowdir_launch_t<8, 8, 4, 5>(a, w, s) : rowdir_launch_t<8, 16, 2, 5>(a, w, s);
}

template <int MT, int NWN, int NWK, int TPW, int PH, int EPI>
static hipError_t rowpar_launch_t(const RowParShape& sh, const RowParArgs& a, const PackedW& w, hipStream_t s) {
    constexpr int NW = NWN * NWK, KTP = NWK * TPW, NBUF = PH > 1 ? 2 : 1, IMG = 2 * MT * KTP;
    const size_t lds = std::max((size_t)NBUF * IMG * 1024, (size_t)NW * MT * 1024) + (size_t)4 * 16 * MT * 4;
    static std::atomic<uint64_t> lds_set{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(gemm_rowpar_kernel<MT, NWN, NWK, TPW, PH, EPI>), lds, lds_set);
    dim3 grid((w.N / 16 + NWN - 1) / NWN, sh.ns, (a.M + 16 * MT - 1) / (16 * MT));
    gemm_rowpar_kernel<MT, NWN, NWK, TPW, PH, EPI><<<grid, NW * 64, lds, s>>>(a, w.data, w.N, w.K / 32);
    return hipGetLastError();
}

template <int EPI>
static hipError_t rowpar_dispatch(const RowParShape& sh, const RowParArgs& a, const PackedW& w, hipStream_t s) {
#define NVLLM_RP(MT_, NWN_, NWK_, TPW_, PH_) \
    if (sh.mt == MT_ && sh.nwn == NWN_ && sh.nwk == NWK_ && sh.tpw == TPW_ && sh.ph == PH_) return rowpar_launch_t<MT_, NWN_, NWK_, TPW_, PH_, EPI>(sh, a, w, s);
#define NVLLM_RP_PH(NWN_, PH_)                                                                        \
    NVLLM_RP(1, NWN_, 4, 8, PH_) NVLLM_RP(1, NWN_, 2, 8, PH_) NVLLM_RP(1, NWN_, 2, 12, PH_) NVLLM_RP(1, NWN_, 2, 16, PH_) \
    NVLLM_RP(1, NWN_, 1, 8, PH_) NVLLM_RP(1, NWN_, 1, 12, PH_) NVLLM_RP(1, NWN_, 1, 16, PH_)
    NVLLM_RP_PH(2, 1) NVLLM_RP_PH(2, 2) NVLLM_RP_PH(2, 3) NVLLM_RP_PH(2, 4)
    if constexpr (EPI != 1) { NVLLM_RP_PH(1, 1) NVLLM_RP_PH(1, 2) NVLLM_RP_PH(1, 3) NVLLM_RP_PH(1, 4) }
    if constexpr (EPI != 0) { NVLLM_RP(1, 4, 4, 8, 1) }
    if constexpr (EPI == 2) {  // big matrices: 64 rows per workgroup, K slices over blockIdx.y
        NVLLM_RP(4, 8, 1, 8, 1) NVLLM_RP(4, 8, 1, 8, 2) NVLLM_RP(4, 8, 1, 8, 3) NVLLM_RP(4, 8, 1, 8, 4)
        NVLLM_RP(4, 4, 1, 8, 1) NVLLM_RP(4, 4, 1, 8, 2) NVLLM_RP(4, 4, 1, 8, 3) NVLLM_RP(4, 4, 1, 8, 4)
    }
#undef NVLLM_RP_PH
#undef NVLLM_RP
    return hipErrorNotSupported;
}

template <int NTA, int TKA, int NTB, int TKB>
static hipError_t rowdir_two_launch(const RowParArgs& a, const PackedW& wa, const RowParArgs& b, const PackedW& wb, hipStream_t s) {
    const int ga = (wa.N / 16 + NTA - 1) / NTA, gb = (wb.N / 16 + NTB - 1) / NTB;
    const size_t lds = (size_t)16 * std::max(NTA, NTB) * 1024 + 4 * 16 * 4;
    static std::atomic<uint64_t> lds_set{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(gemm_rowdir_two_kernel<NTA, TKA, NTB, TKB>), lds, lds_set);
    gemm_rowdir_two_kernel<NTA, TKA, NTB, TKB><<<dim3(ga + gb, 1, (a.M + 15) / 16), 1024, lds, s>>>(a, wa.data, wa.N, ga, b, wb.data, wb.N);
    return hipGetLastError();
}
// K of 1024, 2048 or 3072 each, one round of workgroups together (up to 64 rows)
bool gemm_rowdir_two_ok(const PackedW& wa, const PackedW& wb, int M) {
    if (M > 64 || M < 1) return false;
    const RowDirShape da = rowdir_shape(wa.N, wa.K, 2, M), db = rowdir_shape(wb.N, wb.K, 2, M);
    if (!da.nt || !db.nt || da.tk > 6 || db.tk > 6) return false;
    auto most = [](const RowDirShape& d) { return d.nt == (d.tk == 6 ? 2 : 4); };  // n-tiles of a workgroup
    if (!(da.nt == db.nt && da.nt <= 2) && !(most(da) && most(db))) return false;
    return ((wa.N / 16 + da.nt - 1) / da.nt + (wb.N / 16 + db.nt - 1) / db.nt) * ((M + 15) / 16) <= 256;
}
hipError_t launch_gemm_rowdir_two(const RowParArgs& a, const PackedW& wa, const RowParArgs& b, const PackedW& wb, hipStream_t s) {
    if (a.M != b.M || !gemm_rowdir_two_ok(wa, wb, a.M)) return hipErrorNotSupported;
    const RowDirShape da = rowdir_shape(wa.N, wa.K, 2, a.M), db = rowdir_shape(wb.N, wb.K, 2, b.M);
#define NVLLM_TWO(NTA_, TKA_, NTB_, TKB_) if (da.nt == NTA_ && da.tk == TKA_ && db.nt == NTB_ && db.tk == TKB_) return rowdir_two_launch<NTA_, TKA_, NTB_, TKB_>(a, wa, b, wb, s);
#define NVLLM_TWO_N(TKA_, TKB_) NVLLM_TWO(1, TKA_, 1, TKB_) NVLLM_TWO(2, TKA_, 2, TKB_) NVLLM_TWO((TKA_ == 6 ? 2 : 4), TKA_, (TKB_ == 6 ? 2 : 4), TKB_)
    NVLLM_TWO_N(2, 2) NVLLM_TWO_N(2, 4) NVLLM_TWO_N(2, 6) NVLLM_TWO_N(4, 2) NVLLM_TWO_N(4, 4) NVLLM_TWO_N(4, 6) NVLLM_TWO_N(6, 2) NVLLM_TWO_N(6, 4) NVLLM_TWO_N(6, 6)
#undef NVLLM_TWO_N
#undef NVLLM_TWO
    return hipErrorNotSupported;
}

// A stream of 1024 features (a wave's share of it is a column a lane), K of whole slices.  Rows: a consumer's loads grow with them, 4 M + 1 a wave.  0.6B, one more
// token of 137 to 173, us a call, whole K / slices: 1 row 912 / 829 to 885, 2 rows 961 / 888 to 945, 3 rows 1006 / 949 to 1000, 4 rows 1050 / 981 to 1037, 5 rows (in a form of eight)
// 1068 / 1087, 6 rows 1095 / 1122, 8 rows 1161 / 1185.
bool gemm_rowsum_ok(int H, int Ka, int Kb, int M) {
    auto cut = [](int K) { return K % 1024 == 0 && K / 1024 <= kSumIn; };
    return H == 1024 && cut(Ka) && cut(Kb) && M <= kSumRows;
}
hipError_t launch_gemm_rowslab(const RowParArgs& a, const PackedW& w, hipStream_t s) {
    if (w.K % 1024 || w.N % 16 || a.M > 16) return hipErrorNotSupported;
    if (a.M <= 0) return hipSuccess;
    gemm_rowslab_kernel<2><<<dim3(w.N / 16, w.K / 1024), 1024, 16 * 1024 + 4 * 16 * 4, s>>>(a, w.data, w.N, w.K / 32);
    return hipGetLastError();
}
template <int NT, int EPI>
static hipError_t rowsum_launch(const RowParArgs& a, const PackedW& w, hipStream_t s) {
    const size_t lds = 16 * NT * 1024 + 16 * 16 * 4;
    const int groups = w.N / (16 * NT);
    if (a.M == 1) gemm_rowsum_kernel<NT, EPI, 1><<<groups, 1024, lds, s>>>(a, w.data, w.N, 32);
    else if (a.M == 2) gemm_rowsum_kernel<NT, EPI, 2><<<groups, 1024, lds, s>>>(a, w.data, w.N, 32);
    else gemm_rowsum_kernel<NT, EPI, 4><<<groups, 1024, lds, s>>>(a, w.data, w.N, 32);
    return hipGetLastError();
}
hipError_t launch_gemm_rowsum(const RowParArgs& a, const PackedW& w, int epi, hipStream_t s) {
    if (w.K != 1024 || w.N % 32 || a.M > kSumRows || a.n_in < 1 || a.n_in > kSumIn || a.resid_in == a.resid_out || (epi != 1 && epi != 2)) return hipErrorNotSupported;
    if (a.M <= 0) return hipSuccess;
    return epi == 1 ? rowsum_launch<2, 1>(a, w, s) : rowsum_launch<1, 2>(a, w, s);
}

hipError_t launch_gemm_rowpar(const RowParArgs& a, const PackedW& w, int epi, hipStream_t s) {
    if (const RowDirShape d = rowdir_shape(w.N, w.K, epi, a.M); d.nt) {
        if (a.M <= 0) return hipSuccess;
        if (epi <= 2) {
            const hipError_t e = epi == 0 ? rowpair_dispatch<0>(a, w, s) : epi == 1 ? rowpair_dispatch<1>(a, w, s) : rowpair_dispatch<2>(a, w, s);
            if (e != hipErrorNotReady) return e;
        }
        if (epi == 0) return rowdir_dispatch<0>(d, a, w, s);
        if (epi == 1) return rowdir_dispatch<1>(d, a, w, s);
        if (epi == 2) return rowdir_dispatch<2>(d, a, w, s);
        if ((epi == 3 || epi == 4) && a.oh && (!a.o_packed || w.N % 32 == 0)) return epi == 3 ? rowdir_dispatch<3>(d, a, w, s) : rowdir_dispatch<4>(d, a, w, s);
        return hipErrorInvalidValue;
    }
    if (a.x_packed || a.o_packed) return hipErrorNotSupported;  // packed planes: register-direct kernel only
    RowParShape sh;
    if (!rowpar_shape(w.N, w.K, epi, a.M, sh)) return hipErrorNotSupported;
    if (epi == 1 && sh.nwn % 2) return hipErrorNotSupported;
    if (a.M <= 0) return hipSuccess;
    if (epi == 0) return rowpar_dispatch<0>(sh, a, w, s);
    if (epi == 1) return rowpar_dispatch<1>(sh, a, w, s);
    if (epi == 2) return rowpar_dispatch<2>(sh, a, w, s);
    return hipErrorInvalidValue;
}

// ---------------------------------------------------------------------------------------------------
// (embedding gather +) residual add + RMSNorm, one workgroup per row.
// Replaces Tensor::embedding (qwen3.rs:465-468) and RMSNorm::forward (layernorm.rs:44-60):
//   s = x (+ residual);  y = (s * (1/sqrt(mean(s^2)+eps))) * w;  new residual = s (stays f32).
// x may arrive as n_slabs split-K partial sums of the producing GEMM (summed here).
// ---------------------------------------------------------------------------------------------------
constexpr int kNormMaxV4 = 8;  // per-thread float4 cache: H <= 256*4*8 = 8192

// BS = 256 (many rows: prefill), 512 or 1024 (<= 128 rows: decode has only `rows` workgroups, so each one gets 8 or 16 waves
// and every thread's loads are all in flight at once).  NV: float4s of a thread, by the row's width.  Bound in decode by the chain of round trips to
// memory: up to NV 2 the residual, the weight and eight slabs (four with two steps) are asked for before the first use.  Slabs in trips of four, then the residual, then
// behind the sum the weight: 24 rows of 4096, eight slabs 5.8 us, now 4.8; one row of 1024 5.3, now 2.3.
template <int BS, int NV>
__global__ void __launch_bounds__(BS) add_rmsnorm_kernel(NormArgs a) {
    constexpr bool EARLY = NV <= 2;
    constexpr int SB = NV == 1 ? 8 : 4;  // slabs asked for at once
    __shared__ __attribute__((aligned(16))) float red[BS / 64];
    const int r = blockIdx.x;
    const int src = a.row_idx ? a.row_idx[r] : r;
    const int H = a.H, nv4 = H >> 2;
    auto column = [&](int c) { return (size_t)min((int)threadIdx.x + c * BS, nv4 - 1) * 4; };  // past the row: its last columns again, not used
    auto load4 = [](const float* q) { return *reinterpret_cast<const float4*>(q); };
    float4 cache[NV], res[NV];
    [[maybe_unused]] float4 weight[EARLY ? NV : 1];
    if (a.residual_in)
#pragma unroll
        for (int c = 0; c < NV; ++c) res[c] = load4(a.residual_in + (size_t)src * H + column(c));
    if constexpr (EARLY) {
#pragma unroll
        for (int c = 0; c < NV; ++c) weight[c] = load4(a.weight + column(c));
        __builtin_amdgcn_sched_barrier(0);
    }
    if (a.ids) {
#pragma unroll
        for (int c = 0; c < NV; ++c) {
            const uint2 e = *reinterpret_cast<const uint2*>(a.embed + (size_t)a.ids[src] * H + column(c));
            cache[c] = make_float4(bf16_to_f32(e.x & 0xffff), bf16_to_f32(e.x >> 16), bf16_to_f32(e.y & 0xffff), bf16_to_f32(e.y >> 16));
        }
    } else {
#pragma unroll
        for (int c = 0; c < NV; ++c) cache[c] = make_float4(0.f, 0.f, 0.f, 0.f);
        // split-K slabs: the loads of a batch are independent (slab index clamped, the sum is masked)
        for (int s0 = 0; s0 < a.n_slabs; s0 += SB) {
            float4 t[NV][SB];
#pragma unroll
            for (int c = 0; c < NV; ++c)
#pragma unroll
                for (int u = 0; u < SB; ++u) t[c][u] = load4(a.in + (size_t)src * H + column(c) + (size_t)min(s0 + u, a.n_slabs - 1) * a.slab_stride);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = 0; c < NV; ++c)
#pragma unroll
                for (int u = 0; u < SB; ++u)
                    if (s0 + u < a.n_slabs) { cache[c].x += t[c][u].x; cache[c].y += t[c][u].y; cache[c].z += t[c][u].z; cache[c].w += t[c][u].w; }
        }
    }
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        const int i = threadIdx.x + c * BS;
        float4 s = cache[c];
        if (a.residual_in) { s.x += res[c].x; s.y += res[c].y; s.z += res[c].z; s.w += res[c].w; }
        cache[c] = s;
        if (i >= nv4) continue;
        if (a.residual_out) *reinterpret_cast<float4*>(a.residual_out + (size_t)src * H + (size_t)i * 4) = s;
        ss += s.x * s.x + s.y * s.y + s.z * s.z + s.w * s.w;
    }
    ss = workgroup_sum(ss, red);
    // prep mode: leave the 1/rms factor to the consumer (RowNorm) and publish the row's sum of squares
    const float rinv = a.ssq_out ? 1.0f : 1.0f / sqrtf(ss / (float)H + a.eps);
    if (a.ssq_out && threadIdx.x == 0) a.ssq_out[r] = ss;
#pragma unroll
    for (int c = 0; c < NV; ++c) {
        const int i = threadIdx.x + c * BS;
        if (i < nv4) {
            const float4 s = cache[c];
            const float4 w = EARLY ? weight[EARLY ? c : 0] : load4(a.weight + (size_t)i * 4);
            const float y0 = (s.x * rinv) * w.x, y1 = (s.y * rinv) * w.y, y2 = (s.z * rinv) * w.z, y3 = (s.w * rinv) * w.w;
            if (a.y) *reinterpret_cast<float4*>(a.y + (size_t)r * H + (size_t)i * 4) = make_float4(y0, y1, y2, y3);
            if (a.xh) {
                uint16_t h0, h1, h2, h3, l0, l1, l2, l3;
                split_bf16(y0, h0, l0); split_bf16(y1, h1, l1); split_bf16(y2, h2, l2); split_bf16(y3, h3, l3);
                const size_t xo = a.out_packed ? xpack_off(r, i * 4, H >> 5) : (size_t)r * H + (size_t)i * 4;
                *reinterpret_cast<uint2*>(a.xh + xo) = make_uint2(h0 | ((uint32_t)h1 << 16), h2 | ((uint32_t)h3 << 16));
                *reinterpret_cast<uint2*>(a.xl + xo) = make_uint2(l0 | ((uint32_t)l1 << 16), l2 | ((uint32_t)l3 << 16));
            }
        }
    }
}

// The same operation for prompt chunks whose consumer reads planes in fragment order (the tile GEMM): one workgroup
// = one 16-row tile, NW waves, lane (grp, l15) of wave w owns row l15's 8 consecutive features of k-tiles w, w+NW, ...
// Every read is a full 128-byte line per row (4 lane groups x 32 B) and every plane store is one contiguous 1 KiB
// fragment per wave; the one-row-per-workgroup kernel scatters a row over 128 fragments in 8-byte pieces that share
// their cache lines with fifteen other workgroups (measured 20.6 vs 14.5 us per launch against row-major output).
template <int NW, int IT>
__global__ void __launch_bounds__(NW * 64) add_rmsnorm_rows16_kernel(NormArgs a, int rows) {
    __shared__ float red[NW][16];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int l15 = lane & 15, grp = lane >> 4;
    const int H = a.H, KT = H >> 5;
    const int row = blockIdx.x * 16 + l15, rowc = min(row, rows - 1);
    float v[IT][8];
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int kt = wave + i * NW;
        if (kt < KT) {
            const size_t off = (size_t)rowc * H + (size_t)kt * 32 + grp * 8;
            float4 s0, s1;
            if (a.ids) {
                const uint4 e = *reinterpret_cast<const uint4*>(a.embed + (size_t)a.ids[rowc] * H + (size_t)kt * 32 + grp * 8);
                s0 = make_float4(bf16_to_f32(e.x & 0xffff), bf16_to_f32(e.x >> 16), bf16_to_f32(e.y & 0xffff), bf16_to_f32(e.y >> 16));
                s1 = make_float4(bf16_to_f32(e.z & 0xffff), bf16_to_f32(e.z >> 16), bf16_to_f32(e.w & 0xffff), bf16_to_f32(e.w >> 16));
            } else {
                s0 = *reinterpret_cast<const float4*>(a.in + off);
                s1 = *reinterpret_cast<const float4*>(a.in + off + 4);
                for (int sl = 1; sl < a.n_slabs; ++sl) {
                    const float4 t0 = *reinterpret_cast<const float4*>(a.in + (size_t)sl * a.slab_stride + off);
                    const float4 t1 = *reinterpret_cast<const float4*>(a.in + (size_t)sl * a.slab_stride + off + 4);
                    s0.x += t0.x; s0.y += t0.y; s0.z += t0.z; s0.w += t0.w;
                    s1.x += t1.x; s1.y += t1.y; s1.z += t1.z; s1.w += t1.w;
                }
            }
            if (a.residual_in) {
                const float4 t0 = *reinterpret_cast<const float4*>(a.residual_in + off), t1 = *reinterpret_cast<const float4*>(a.residual_in + off + 4);
                s0.x += t0.x; s0.y += t0.y; s0.z += t0.z; s0.w += t0.w;
                s1.x += t1.x; s1.y += t1.y; s1.z += t1.z; s1.w += t1.w;
            }
            if (a.residual_out && row < rows) {
                *reinterpret_cast<float4*>(a.residual_out + off) = s0;
                *reinterpret_cast<float4*>(a.residual_out + off + 4) = s1;
            }
            v[i][0] = s0.x; v[i][1] = s0.y; v[i][2] = s0.z; v[i][3] = s0.w;
            v[i][4] = s1.x; v[i][5] = s1.y; v[i][6] = s1.z; v[i][7] = s1.w;
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += v[i][e] * v[i][e];
        }
    }
    ss += __shfl_xor(ss, 16);
    ss += __shfl_xor(ss, 32);
    if (grp == 0) red[wave][l15] = ss;
    __syncthreads();
    ss = 0.f;
#pragma unroll
    for (int q = 0; q < NW; ++q) ss += red[q][l15];
    const float rinv = a.ssq_out ? 1.0f : 1.0f / sqrtf(ss / (float)H + a.eps);
    if (a.ssq_out && wave == 0 && grp == 0 && row < rows) a.ssq_out[row] = ss;
    uint4* ph = reinterpret_cast<uint4*>(a.xh);
    uint4* pl = reinterpret_cast<uint4*>(a.xl);
#pragma unroll
    for (int i = 0; i < IT; ++i) {
        const int kt = wave + i * NW;
        if (kt < KT) {
            const float4 w0 = *reinterpret_cast<const float4*>(a.weight + kt * 32 + grp * 8), w1 = *reinterpret_cast<const float4*>(a.weight + kt * 32 + grp * 8 + 4);
            const float wv[8] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
            uint16_t h[8], l[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) split_bf16((v[i][e] * rinv) * wv[e], h[e], l[e]);
            const size_t o = ((size_t)blockIdx.x * KT + kt) * 64 + lane;
            ph[o] = make_uint4(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16), h[4] | ((uint32_t)h[5] << 16), h[6] | ((uint32_t)h[7] << 16));
            pl[o] = make_uint4(l[0] | ((uint32_t)l[1] << 16), l[2] | ((uint32_t)l[3] << 16), l[4] | ((uint32_t)l[5] << 16), l[6] | ((uint32_t)l[7] << 16));
        }
    }
}

hipError_t launch_add_rmsnorm(const NormArgs& a, int rows, hipStream_t s) {
    if (a.H % 4 != 0 || a.H > 256 * 4 * kNormMaxV4) return hipErrorInvalidValue;
    if (rows <= 0) return hipSuccess;
    if (a.out_packed && a.xh && a.xl && !a.y && !a.row_idx && a.H % 32 == 0 && rows >= 1024) {  // prompt chunk, fragment-order planes
        const int KT = a.H / 32, tiles = (rows + 15) / 16;
        if (KT <= 32) { add_rmsnorm_rows16_kernel<16, 2><<<tiles, 1024, 0, s>>>(a, rows); return hipGetLastError(); }  // about one tile per CU: many waves keep more loads in flight
        if (KT <= 64) { add_rmsnorm_rows16_kernel<16, 4><<<tiles, 1024, 0, s>>>(a, rows); return hipGetLastError(); }
        if (KT <= 160) { add_rmsnorm_rows16_kernel<16, 10><<<tiles, 1024, 0, s>>>(a, rows); return hipGetLastError(); }
    }
    if (rows <= 128 && a.H >= 2048) {
        if (a.H <= 2048) add_rmsnorm_kernel<512, 1><<<rows, 512, 0, s>>>(a);
        else if (a.H <= 4096) add_rmsnorm_kernel<1024, 1><<<rows, 1024, 0, s>>>(a);
        else add_rmsnorm_kernel<1024, kNormMaxV4 / 4><<<rows, 1024, 0, s>>>(a);
    } else if (a.H <= 1024) add_rmsnorm_kernel<256, 1><<<rows, 256, 0, s>>>(a);
    else if (a.H <= 2048) add_rmsnorm_kernel<256, 2><<<rows, 256, 0, s>>>(a);
    else if (a.H <= 4096) add_rmsnorm_kernel<256, 4><<<rows, 256, 0, s>>>(a);
    else add_rmsnorm_kernel<256, kNormMaxV4><<<rows, 256, 0, s>>>(a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// q/k RMSNorm over head_dim + RoPE + KV-cache write; one wave per (row, head).
// Replaces qwen3.rs:208-234 (narrow/reshape/transpose, q_norm/k_norm BEFORE RoPE and GQA expand) and
// rotary_embedding.rs:82-107 (half-split: y1 = x1*cos - x2*sin, y2 = x2*cos + x1*sin).
// K goes to the paged cache row-major f16; V goes in the PV A-fragment order:
//   token tt (0..31) of a 32-token tile sits in k-slot (g, j): tt<16: g=tt>>2, j=tt&3; else g=(tt-16)>>2, j=4+(tt&3)
//   element (tt, d) -> (((tile*(hd/16) + d/16)*64 + g*16 + d%16)*8 + j
// ---------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) qk_norm_rope_kvwrite_kernel(QkvArgs a) {
    const int row = blockIdx.x;
    const int lane = threadIdx.x & 63;
    const int hh = blockIdx.y * 4 + (threadIdx.x >> 6);
    const int hd = a.kv.hd, half = hd >> 1, kv_l = a.kv.kv_l;
    const int heads = a.nh_l + 2 * kv_l;
    if (hh >= heads) return;
    const int ldq = heads * hd;
    const bool act = lane < half;
    float x1 = 0.f, x2 = 0.f;
    if (act) {
        const float* p = a.qkv + (size_t)row * ldq + (size_t)hh * hd;
        x1 = p[lane];
        x2 = p[lane + half];
        for (int sl = 1; sl < a.n_slabs; ++sl) {
            x1 += p[(size_t)sl * a.slab_stride + lane];
            x2 += p[(size_t)sl * a.slab_stride + lane + half];
        }
    }
    const float ri = rownorm_rinv_wave(a.rn, row, lane);  // deferred input norm: the QKV sums are linear in x
    x1 *= ri;
    x2 *= ri;
    const int pos = a.pos[row];
    if (hh < a.nh_l + kv_l) {  // q or k head: norm + rope
        const float* w = hh < a.nh_l ? a.qn : a.kn;
        const float ss = wave_sum(x1 * x1 + x2 * x2);
        const float rinv = 1.0f / sqrtf(ss / (float)hd + a.eps);
        float y1 = 0.f, y2 = 0.f;
        if (act) {
            const float n1 = (x1 * rinv) * w[lane], n2 = (x2 * rinv) * w[lane + half];
            const float c = a.cos[(size_t)pos * half + lane], s = a.sin[(size_t)pos * half + lane];
            y1 = n1 * c - n2 * s;
            y2 = n2 * c + n1 * s;
        }
        if (hh < a.nh_l) {
            if (act) {
                float* q = a.q_out + (size_t)row * (a.nh_l * hd) + (size_t)hh * hd;
                q[lane] = y1 * a.q_scale;
                q[lane + half] = y2 * a.q_scale;
            }
        } else if (act) {
            const int kh = hh - a.nh_l;
            const int blk = a.block_tables[(size_t)a.slot[row] * a.max_blocks + (pos >> 8)];
            const size_t ko = (size_t)(blk * kv_l + kh) * kBlockTokens * hd;
            _Float16* k = reinterpret_cast<_Float16*>(a.kv.k) + ko;
            uint8_t* klo = a.kv.klo ? a.kv.klo + ko : nullptr;
            store_k24(k, klo, pos & 255, lane, hd, y1);
            store_k24(k, klo, pos & 255, lane + half, hd, y2);
        }
    } else if (act) {  // v head: plain copy into the packed layout
        const int kh = hh - a.nh_l - kv_l;
        const int blk = a.block_tables[(size_t)a.slot[row] * a.max_blocks + (pos >> 8)];
        const size_t vo = (size_t)(blk * kv_l + kh) * kBlockTokens * hd;
        _Float16* v = reinterpret_cast<_Float16*>(a.kv.v) + vo;
        uint8_t* vlo = a.kv.vlo ? a.kv.vlo + vo : nullptr;
        store_v24(v, vlo, pos & 255, lane, hd, x1);
        store_v24(v, vlo, pos & 255, lane + half, hd, x2);
    }
}

// The same for heads of 128: one workgroup per 16 rows and head, 16 threads a row with four features and their partners each.  Bound by memory;
// a wave per (row, head) with one feature a lane read and wrote 256 bytes an instruction and 2 of every cache store: 1269 and 2020
// rows of 32 heads 17.0 -> 16.2 and 19.4 -> 17.5 us, 4050 rows of 48 heads 61.8 -> 44.2 (183 MB).
__global__ void __launch_bounds__(256) qk_rows16_kernel(QkvArgs a, int rows) {
    const int row = blockIdx.x * 16 + (threadIdx.x >> 4), sub = threadIdx.x & 15, f0 = sub * 4, hh = blockIdx.y;
    const int rowc = min(row, rows - 1), nh = a.nh_l, kv_l = a.kv.kv_l;
    const float* p = a.qkv + (size_t)rowc * ((nh + 2 * kv_l) * 128) + (size_t)hh * 128 + f0;
    auto load = [](const float* from) { return __builtin_bit_cast(f32x4, *reinterpret_cast<const float4*>(from)); };
    f32x4 x1 = load(p), x2 = load(p + 64);
    const int pos = a.pos[rowc];
    const bool rot = hh < nh + kv_l;
    const float* w = hh < nh ? a.qn : a.kn;
    const f32x4 w1 = load(w + f0), w2 = load(w + 64 + f0);
    for (int sl = 1; sl < a.n_slabs; ++sl) {
        x1 += load(p + (size_t)sl * a.slab_stride);
        x2 += load(p + (size_t)sl * a.slab_stride + 64);
    }
    if (a.rn.ssq) {  // deferred input norm: the QKV sums are linear in x
        float t = 0.f;
        for (int g = sub; g < a.rn.groups; g += 16) t += a.rn.ssq[(size_t)g * a.rn.stride + rowc];
        const float ri = 1.0f / sqrtf(row16_sum(t) * a.rn.inv_h + a.rn.eps);
        x1 *= ri;
        x2 *= ri;
    }
    if (rot) {  // q or k head: norm + rope
        const f32x4 c = load(a.cos + (size_t)pos * 64 + f0), sn = load(a.sin + (size_t)pos * 64 + f0), s4 = x1 * x1 + x2 * x2;
        const float rinv = 1.0f / sqrtf(row16_sum((s4[0] + s4[1]) + (s4[2] + s4[3])) / 128.0f + a.eps);
        const f32x4 n1 = x1 * rinv * w1, n2 = x2 * rinv * w2;
        x1 = n1 * c - n2 * sn;
        x2 = n2 * c + n1 * sn;
    }
    if (row >= rows) return;
    if (hh < nh) {
        float* q = a.q_out + (size_t)row * (nh * 128) + (size_t)hh * 128 + f0;
        x1 *= a.q_scale;
        x2 *= a.q_scale;
        *reinterpret_cast<float4*>(q) = make_float4(x1[0], x1[1], x1[2], x1[3]);
        *reinterpret_cast<float4*>(q + 64) = make_float4(x2[0], x2[1], x2[2], x2[3]);
        return;
    }
    const int blk = a.block_tables[(size_t)a.slot[row] * a.max_blocks + (pos >> 8)], t = pos & 255;
    const size_t at = (size_t)(blk * kv_l + (rot ? hh - nh : hh - nh - kv_l)) * kBlockTokens * 128;
    if (rot) {  // four neighbouring features lie side by side
        typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
        _Float16* k = reinterpret_cast<_Float16*>(a.kv.k) + at;
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const f32x4 y = e ? x2 : x1;
            const f16x4 v = {f16_sat(y[0]), f16_sat(y[1]), f16_sat(y[2]), f16_sat(y[3])};
            *reinterpret_cast<f16x4*>(k + k_packed_offset(t, e * 64 + f0, 128)) = v;
            if (a.kv.klo) {
                uint32_t w4 = 0;
#pragma unroll
                for (int r = 0; r < 4; ++r) w4 |= (uint32_t)residual24(y[r], v[r]) << (8 * r);
                *reinterpret_cast<uint32_t*>(a.kv.klo + at + klo_packed_offset(t, e * 64 + f0, 128)) = w4;
            }
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            store_v24(reinterpret_cast<_Float16*>(a.kv.v) + at, a.kv.vlo ? a.kv.vlo + at : nullptr, t, (e >> 2) * 64 + f0 + (e & 3), 128, e < 4 ? x1[e & 3] : x2[e & 3]);
    }
}

// Enough workgroups of 16 rows and a head that every CU has one; below, a wave to each (row, head) spreads the same loads over more CUs.  us a
// launch between two events, which are 5 of them, a wave per (row, head) / 16 rows: 32 heads (0.6B) 16 rows 6.8 / 7.6, 64 7.2 / 7.5, 129
// 7.8 / 7.9, 160 8.1 / 8.1, 200 8.5 / 8.3, 300 10.7 / 9.6; with a 24-bit cache 16 rows 7.0 / 8.1, 64 7.2 / 8.1, 160 8.5 / 8.6, 256 9.5 / 9.2;
// 48 heads (8B) 16 rows 6.6 / 6.9, 64 7.4 / 7.5, 100 8.3 / 8.1, 200 13.9 / 12.0.  0.6B prompts of 16 and 64 tokens 1.026 / 1.044 and 1.205 / 1.209 ms,
// 24-bit 1.065 / 1.098 and 1.277 / 1.298.
bool qk_rows16_wins(int rows, int heads, int hd) { return hd == 128 && (rows + 15) / 16 * heads >= 320; }

hipError_t launch_qk_norm_rope_kvwrite(const QkvArgs& a, int rows, hipStream_t s) {
    if (a.kv.hd > 128 || a.kv.hd % 32 != 0) return hipErrorInvalidValue;
    if (rows <= 0) return hipSuccess;
    const int heads = a.nh_l + 2 * a.kv.kv_l;
    if (qk_rows16_wins(rows, heads, a.kv.hd)) {
        qk_rows16_kernel<<<dim3((rows + 15) / 16, heads), 256, 0, s>>>(a, rows);
        return hipGetLastError();
    }
    dim3 grid(rows, (heads + 3) / 4);
    qk_norm_rope_kvwrite_kernel<<<grid, 256, 0, s>>>(a);
    return hipGetLastError();
}

// plain K/V write (no norm / rope) for the fine-seam attention op
__global__ void __launch_bounds__(256) kv_write_plain_kernel(const float* __restrict__ k, const float* __restrict__ v,
                                                             const int* __restrict__ pos, const int* __restrict__ slot,
                                                             const int* __restrict__ bt, int max_blocks, KvLayout kv) {
    const int row = blockIdx.x;
    const int n = kv.kv_l * kv.hd;
    const int p = pos[row];
    const int blk = bt[(size_t)slot[row] * max_blocks + (p >> 8)];
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const int kh = i / kv.hd, d = i - kh * kv.hd;
        const size_t vo = (size_t)(blk * kv.kv_l + kh) * kBlockTokens * kv.hd;
        store_k24(reinterpret_cast<_Float16*>(kv.k) + vo, kv.klo ? kv.klo + vo : nullptr, p & 255, d, kv.hd, k[(size_t)row * n + i]);
        store_v24(reinterpret_cast<_Float16*>(kv.v) + vo, kv.vlo ? kv.vlo + vo : nullptr, p & 255, d, kv.hd, v[(size_t)row * n + i]);
    }
}
hipError_t launch_kv_write_plain(const float* k, const float* v, int rows, const int* pos, const int* slot,
                                 const int* block_tables, int max_blocks, KvLayout kv, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    kv_write_plain_kernel<<<rows, 256, 0, s>>>(k, v, pos, slot, block_tables, max_blocks, kv);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// Rows the head wants, compact (what the last layer of a prompt works on after its mixer): one workgroup a row and a set.  A few hundred KB:
// a launch's own 4 us
// ---------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) gather_rows_kernel(GatherArgs a) {
    const int r = blockIdx.x, src = a.idx[r];
    if ((int)blockIdx.y == a.sets) {
        for (int i = threadIdx.x * 4; i < a.ldr; i += 1024)
            *reinterpret_cast<float4*>(a.resid_out + (size_t)r * a.ldr + i) = *reinterpret_cast<const float4*>(a.resid + (size_t)src * a.ldr + i);
        return;
    }
    const GatherSet& t = a.set[blockIdx.y];
    if (t.f) {
        for (int i = threadIdx.x * 4; i < t.ld; i += 1024)
            *reinterpret_cast<float4*>(t.of + (size_t)r * t.ld + i) = *reinterpret_cast<const float4*>(t.f + (size_t)src * t.ld + i);
        return;
    }
    for (int i = threadIdx.x * 8; i < t.ld; i += 2048) {
        const size_t in = t.in_packed ? xpack_off(src, i, t.ld >> 5) : (size_t)src * t.ld + i;
        const size_t out = t.out_packed ? xpack_off(r, i, t.ld >> 5) : (size_t)r * t.ld + i;
        *reinterpret_cast<uint4*>(t.oh + out) = *reinterpret_cast<const uint4*>(t.h + in);
        *reinterpret_cast<uint4*>(t.ol + out) = *reinterpret_cast<const uint4*>(t.l + in);
    }
}
hipError_t launch_gather_rows(const GatherArgs& a, int n, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    if (a.ldr % 4) return hipErrorInvalidValue;
    for (int i = 0; i < a.sets; ++i) if (a.set[i].ld % 32) return hipErrorInvalidValue;
    gather_rows_kernel<<<dim3(n, a.sets + 1), 256, 0, s>>>(a);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// Paged causal GQA attention of decode rows.
// Replaces qwen3.rs:236-277: GQA interleaved expand (q head h -> kv head h/(nh/kv)), scores*scale,
// additive -1e9 mask for j>i (masked terms are exactly 0 after the f32 softmax, so they are skipped),
// f32 softmax, p.v.  A KV cache is mathematically equivalent to the reference's full recompute (causal).
//
// One workgroup = one row (its gqa q-heads in the 16 MFMA rows) x one kv head.
// Its 4 or 8 waves (8: launches of one workgroup per CU at most) take alternate 32-token KV tiles; K and V fragments go straight from HBM to VGPRs:
//   S^T[token][qrow]  = K[token][:] . q[qrow][:]      A = K frag (16 rows x 64 B per wave-load), B = q (f16 hi+lo)
//   O^T[dim][qrow]   += V^T[dim][token] . P[token][qrow]   A = V packed frag (1 KiB wave-load), B = P straight
//                                                          from the S accumulators (no lane movement)
// Both products keep the q row on lane&15, so the online-softmax state (m, l) is per-lane.
// ---------------------------------------------------------------------------------------------------
// It must keep two waves per SIMD (<= 256 registers): at 229 + 40 the compiler once dropped it to one
// wave per SIMD on its own and the whole decode step lost 12 %
// VLO: 24-bit V (KvLayout::vlo): every V fragment comes with 8 residual bytes per lane (a 512-byte wave-load); shifted into
// the high byte they ARE the residuals' f16 bit patterns, which a second P.V MFMA adds (the kernel is HBM-bound: V bytes x1.5)

// a prompt's i-th q-tile in walking order
__device__ __forceinline__ PrefillTile prefill_tile(const AttnArgs& a, int i) {
    const uniform_ints_t p = uniform_ints(reinterpret_cast<const int*>(a.tiles + i));
    return PrefillTile{p[0], p[1], p[2], p[3], p[4], p[5], {0, 0}};
}

// VLO: 0 = 16-bit cache, 1 = 24-bit V, 2 = 24-bit K and V (KvLayout::klo too: four more 1 KiB wave-loads per tile, one bf8 MFMA
// per QK^T fragment against q in bf8)
// AHEAD: both tile sets are asked for before the prologue, see there
// PARTS: contexts may be in parts
template <int HD, int NWV, bool FUSED, int VLO, bool AHEAD, bool PARTS>
__device__ __forceinline__ void attn_paged_body(const AttnArgs& a) {
    constexpr int DC = HD / 32, DT = HD / 16, DL = VLO ? DT / 2 : 1;  // DL: 1 KiB residual fragments per tile (two PV fragments each)
    constexpr bool KLO = VLO == 2;
    constexpr bool ONE_SET = VLO != 0;  // decode with a 24-bit cache: one tile set in flight per wave (see the loop)
    using Wave = AttnWave<HD, 1, VLO>;
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    // [NWV][2][16] m and l of the waves; [NWV][columns][HD] their O; fused: q as f16 hi and lo [2][gqa][HD], the new token's K and V and the
    // residual bytes of both
    float* ml = reinterpret_cast<float*>(smem_raw);
    const int cols = FUSED ? a.gqa : 16;  // MFMA columns that are rows of q
    // rows of O and of q are 16 bytes longer than their elements: a wave's lanes are columns of one dim, which would all be on the same banks
    constexpr int OS = HD / 4 + 1, QS = HD + 8;
    f32x4* obuf = reinterpret_cast<f32x4*>(smem_raw + NWV * 2 * 16 * 4);
    [[maybe_unused]] const int q_at = NWV * (2 * 16 * 4 + cols * OS * 16), new_at = q_at + cols * QS * 4;  // bytes
    // (offsets, not pointers to choose between: the compiler must see that every access is to LDS, a generic one would wait for the tiles)
    [[maybe_unused]] auto lds16 = [&](int byte) { return reinterpret_cast<_Float16*>(smem_raw + byte); };
    [[maybe_unused]] auto lds8 = [&](int byte) { return reinterpret_cast<uint8_t*>(smem_raw + byte); };
    [[maybe_unused]] const int new_v_at = new_at + HD * 2, new_kl_at = new_at + HD * 4, new_vl_at = new_at + HD * 5;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l15 = lane & 15, grp = lane >> 4;
    // the tile: of the grid's y in the fused form (its callers have at most kAttnFusedMaxRows rows), part of x in the other
    int tile = FUSED ? blockIdx.y : __builtin_amdgcn_readfirstlane((int)blockIdx.x / a.kv.kv_l);
    const int kh = FUSED ? blockIdx.x : blockIdx.x - tile * a.kv.kv_l;
    NVLLM_STAMP(a, 0);
    // kv heads are the fast part of the grid: the heads of a row start together, and what they read at one time lies side by side (a block's
    // slabs of all heads are 512 KiB in a row), which the memory turns out faster than as many places far apart.  Tiles go longest context
    // first, every other run of 256 workgroups backwards: workgroups i and i + 256 share a CU when two fit, so a long context gets a short
    // neighbour.  With the rows as the fast dimension: 200 rows of 64 to 1024 tokens 105 -> 98.5 us per launch, 24 of 256 to 2048 46 -> 41;
    // 64 rows of 64 to 512, resident all at once, the same 23.6.  Up to 128 workgroups, with the
    // parts of a row beside them, there is nothing to pair: 16 rows of 100 to 800 tokens 1.258 ms a step in that order, 1.242 in the rows'; 24
    // rows on 8 heads of 256 to 2048 tokens, in two parts, 0.784 and 0.792.
    // The fused form has all that the first K/V loads wait for in the row's record.  Order, row, slot and block table in turn, and a division
    // for the run, before: prologue of a wave, its first stamp to its last, 24 rows of 48 to 408 tokens 3.6 -> 2.6 us, one row of 137 2.5 -> 1.9; kernel
    // 9.6 -> 8.7 and 6.4 -> 5.9, 64 rows of 64 to 512 18.3 -> 17.7, 24 rows of 24 bits 12.9 -> 12.1.
    if (!FUSED && a.tile_order && gridDim.x > 128) {
        const int per = max(1, 256 / a.kv.kv_l);
        const int g = __builtin_amdgcn_readfirstlane(tile / per), r = tile - g * per;
        const int n_tiles = __builtin_amdgcn_readfirstlane((int)gridDim.x / a.kv.kv_l), end = min(n_tiles, (g + 1) * per);
        tile = a.tile_order[g & 1 ? end - 1 - r : tile];
    }
    // fused decode: every q-tile is one row, its record in launch order (see DecodeRow)
    const uniform_ints_t rec = uniform_ints(reinterpret_cast<const int*>(a.rows + (FUSED ? tile : 0)));
    // split-KV (flash-decoding): workgroup blockIdx.z owns 32-token tiles [t_begin, t_end) and leaves an
    // un-normalised partial (m, l, O); every workgroup then has the same short dependent-load chain
    // whatever the context length.  part_tiles == 0: one workgroup does the whole context.
    const int t_begin = PARTS && a.part_tiles ? (int)blockIdx.z * a.part_tiles : 0;
    [[maybe_unused]] int first_slab[2] = {0, 0};  // cache blocks of this wave's first two tiles
    if constexpr (FUSED) {
#pragma unroll
        for (int i = 0; i < 2; ++i) first_slab[i] = rec[4 + min((t_begin + wave + i * NWV) >> 3, kDecodeRowBlocks - 1)];
        if (!a.in_order) {
            tile = rec[0];
            asm volatile("" : "+s"(tile));  // a branch, not a choice: the other side must not wait for the record
        }
    }
    const int row0 = FUSED ? tile : a.tile_row0[tile], nrows = FUSED ? 1 : a.tile_nrows[tile];
    const int gqa = a.gqa, tpq = 16 / gqa;
    // fused decode: the workgroup's gqa q heads, its k head and its v head are its items, LPH lanes each, HPW to a wave, dealt out to the waves
    // and shared through LDS; what needs the row alone is asked for before the slot, the position and the block table are waited for.  Every
    // wave making all of q for itself, with the 14 empty columns of 16, was 24 16-byte loads and 400 instructions a lane: 64 rows of 64 to 512
    // tokens 21.7 -> 19.8 us a layer, one row of 137 9.7 -> 8.7, 24 8B rows of 256 to 2048 39.1 -> 32.2; with a 24-bit cache, where it spilled,
    // 24 rows of 48 to 400 23.6 -> 20.1 (all before the eight waves).
    constexpr int half = HD / 2, LPH = HD / 4, HPW = 64 / LPH, NI = 2;  // NI: rounds of items loaded up front, all of them up to gqa = NI * NWV * HPW - 2
    [[maybe_unused]] const int kv_heads = a.kv.kv_l, items = gqa + 2, hl = lane / LPH, hd2 = lane % LPH * 2;  // this lane's dims: hd2, hd2 + 1 and the two half a head further
    [[maybe_unused]] const float* qkv_row = FUSED ? a.qkv + (size_t)row0 * a.ldqkv : nullptr;
    [[maybe_unused]] auto item_of = [&](int it) { return (it * NWV + wave) * HPW + hl; };
    [[maybe_unused]] auto item_src = [&](int item) {
        return qkv_row + (size_t)(item < gqa ? kh * gqa + item : item == gqa ? a.nh_l + kh : a.nh_l + kv_heads + kh) * HD + hd2;
    };
    [[maybe_unused]] auto load2 = [](const float* p) { return *reinterpret_cast<const float2*>(p); };
    [[maybe_unused]] float2 xa[NI], xb[NI], wa[NI], wb[NI];
    [[maybe_unused]] float ssq_g = 0.f;
    if constexpr (FUSED) {
#pragma unroll
        for (int it = 0; it < NI; ++it) {
            const int item = min(item_of(it), items - 1);
            const float *p = item_src(item), *w = (item < gqa ? a.qn : a.kn) + hd2;
            xa[it] = load2(p); xb[it] = load2(p + half);
            wa[it] = load2(w); wb[it] = load2(w + half);
        }
        // deferred input norm of this row: lane g loads group g (groups <= 64), summed below
        if (a.rn.ssq && lane < a.rn.groups) ssq_g = a.rn.ssq[(size_t)lane * a.rn.stride + row0];
        __builtin_amdgcn_sched_barrier(0);
    }
    const int slot = FUSED ? rec[1] : a.tile_slot[tile];
    const int kv_l = a.kv.kv_l;
    const int ldq = a.nh_l * HD;

    int my_row, my_pos;
    const int my_head = kh * gqa + (l15 % gqa);
    const int tok = l15 / gqa;
    const bool valid = (l15 < tpq * gqa) && (tok < nrows);
    my_row = valid ? row0 + tok : -1;
    if constexpr (!FUSED) my_pos = valid ? a.pos[row0 + tok] : -1;
    const int pmax = FUSED ? rec[2] : a.pos[row0 + nrows - 1];
    if constexpr (FUSED) my_pos = pmax;  // uniform; what the lanes of no row (q = 0) sum up is never stored
    const int n_kv_tiles = (pmax >> 5) + 1;
    const int t_end = PARTS && a.part_tiles ? min(n_kv_tiles, t_begin + a.part_tiles) : n_kv_tiles;
    if (t_begin >= n_kv_tiles) return;  // uniform for the whole workgroup

    // (plain reads became vector loads behind the prologue's barrier, each with a wait that drained the tiles in flight)
    const uniform_ints_t bt = uniform_ints(a.block_tables + (size_t)slot * a.max_blocks);
    // one 32-token KV tile: 2*DC K fragments (the two 16-token tiles are contiguous) + DT V fragments, 16 KiB in 1 KiB wave-loads.  A tile
    // past the end (kt >= t_end: a wave leaves its loop with up to two such prefetches) is the same instructions over buffers of no bytes:
    // they return zeros and cost no access.  A branch around the loads instead makes hipcc wait for vmcnt(0) per load.
    struct Tile { uint4 k[2 * DC], kl[KLO ? DC : 1], v[DT], vl[VLO ? DL : 1]; };  // K's fragments (the two halves in turn) and residuals, V's
    auto load_k_of = [&](int kt, int block, Tile& to) {
        const int T0 = min(kt, t_end - 1) << 5;
        const int slab = block * kv_l + kh, tb = T0 & 255, bytes = kt < t_end ? kBlockTokens * HD * 2 : 0;
        const auto rk = buffer_of(reinterpret_cast<const char*>(a.kv.k) + (size_t)slab * (kBlockTokens * HD * 2), bytes);
        const int ko = (tb >> 4) * (DC * 1024);
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            to.k[2 * c] = buffer_stream16(rk, lane * 16 + c * 1024, ko);
            to.k[2 * c + 1] = buffer_stream16(rk, lane * 16 + c * 1024, ko + DC * 1024);
        }
        if constexpr (KLO) {
            const auto rl = buffer_of(a.kv.klo + (size_t)slab * (kBlockTokens * HD), bytes / 2);
#pragma unroll
            for (int i = 0; i < DC; ++i) to.kl[i] = buffer_stream16(rl, lane * 16 + i * 1024, (tb >> 4) * ((DC / 2) * 1024));
        }
    };
    auto load_v_of = [&](int kt, int block, Tile& to) {
        const int T0 = min(kt, t_end - 1) << 5;
        const int slab = block * kv_l + kh, tb = T0 & 255, bytes = kt < t_end ? kBlockTokens * HD * 2 : 0;
        const auto rv = buffer_of(reinterpret_cast<const char*>(a.kv.v) + (size_t)slab * (kBlockTokens * HD * 2), bytes);
        const int vo = (tb >> 5) * (DT * 1024);
#pragma unroll
        for (int d = 0; d < DT; ++d) to.v[d] = buffer_stream16(rv, lane * 16 + (d % 4) * 1024, vo + d / 4 * 4096);
        if constexpr (VLO) {
            const auto rl = buffer_of(a.kv.vlo + (size_t)slab * (kBlockTokens * HD), bytes / 2);
#pragma unroll
            for (int d = 0; d < DL; ++d) to.vl[d] = buffer_stream16(rl, lane * 16 + d * 1024, (tb >> 5) * (DL * 1024));
        }
    };
    auto block_of = [&](int kt) { return bt[min(kt, t_end - 1) >> 3]; };
    auto load_k = [&](int kt, Tile& to) { load_k_of(kt, block_of(kt), to); };
    auto load_v = [&](int kt, Tile& to) { load_v_of(kt, block_of(kt), to); };
    auto load_tile_of = [&](int kt, int block, Tile& to) {
        load_k_of(kt, block, to);
        load_v_of(kt, block, to);
    };
    auto load_tile = [&](int kt, Tile& to) { load_tile_of(kt, block_of(kt), to); };
    // a wave's first or second tile; one past the end is not read from its block
    [[maybe_unused]] auto load_first = [&](int i, Tile& to) {
        const int kt = t_begin + wave + i * NWV;
        int block = first_slab[i];
        if (kt >> 3 >= kDecodeRowBlocks) {
            block = block_of(kt);
            asm volatile("" : "+s"(block));
        }
        load_tile_of(kt, block, to);
    };
    // register sets: two 32-token tiles (32 KiB) of this wave are in flight at any time
    Tile tA, tB;
    Wave w;
    int new_tile = -1;  // fused decode: the tile of the new token, in the wave that has it
    if constexpr (FUSED) {
        // Decode, fused prologue (replaces a separate launch): this workgroup is the only consumer of q heads
        // kh*gqa.. of its row and the only producer of that row's K/V for kv head kh.  The QKV GEMM's split-K
        // slabs are summed here; q/k get RMSNorm over head_dim then RoPE (qwen3.rs:224-234) exactly as
        // qk_norm_rope_kvwrite_kernel does for prefill.
        const int pos = pmax, last = pos >> 5;
        const bool has_new = last >= t_begin && last < t_end;  // split-KV: one workgroup of the row makes the new token's K and V
        const float2 cs = load2(a.cos + (size_t)pos * half + hd2), sn = load2(a.sin + (size_t)pos * half + hd2);
        auto add_slabs = [&](const float* p, float2& u, float2& w) __attribute__((always_inline)) {  // split-K slabs of the generic path's QKV GEMM, four per trip
            for (int s0 = 1; s0 < a.n_slabs; s0 += 4) {
                float2 pu[4], pw[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float* ps = p + (size_t)min(s0 + i, a.n_slabs - 1) * a.slab_stride;
                    pu[i] = load2(ps); pw[i] = load2(ps + half);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float f = s0 + i < a.n_slabs ? 1.f : 0.f;
                    u.x += f * pu[i].x; u.y += f * pu[i].y; w.x += f * pw[i].x; w.y += f * pw[i].y;
                }
            }
        };
        if (a.n_slabs > 1)
#pragma unroll
            for (int it = 0; it < NI; ++it) add_slabs(item_src(min(item_of(it), items - 1)), xa[it], xb[it]);
        // This wave's first KV tile goes in flight BEHIND the prologue's own loads (vmcnt retires in order, so the prologue never waits for
        // it) and lands while it computes; the second behind the prologue (AHEAD: with the first; rule and figures at attn_tiles_ahead).  The new token's place in its tile still holds old bytes, or the new ones if the stores below
        // pass first: the tile is patched before it is used.
        load_first(0, tA);
        if constexpr (AHEAD && !ONE_SET) load_first(1, tB);
        const float ri = a.rn.ssq ? 1.0f / sqrtf(wave_sum_uniform(ssq_g) * a.rn.inv_h + a.rn.eps) : 1.0f;
        auto make = [&](int item, float2 u, float2 w, float2 nu, float2 nw) __attribute__((always_inline)) {
            u.x *= ri; u.y *= ri; w.x *= ri; w.y *= ri;
            float ss = u.x * u.x + u.y * u.y + w.x * w.x + w.y * w.y;
            ss = row16_sum(ss);
            if constexpr (LPH == 32) ss += __shfl_xor(ss, 16);
            const float rinv = 1.0f / sqrtf(ss / (float)HD + a.eps);
            const float y[4] = {u.x, u.y, w.x, w.y}, g[4] = {nu.x, nu.y, nw.x, nw.y}, c[2] = {cs.x, cs.y}, s_[2] = {sn.x, sn.y};
            float z[4];  // dims hd2, hd2 + 1, half + hd2, half + hd2 + 1
#pragma unroll
            for (int e = 0; e < 2; ++e) {
                const float n1 = (y[e] * rinv) * g[e], n2 = (y[2 + e] * rinv) * g[2 + e];
                z[e] = n1 * c[e] - n2 * s_[e];
                z[2 + e] = n2 * c[e] + n1 * s_[e];
            }
            if (item < gqa) {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float v = z[e] * a.q_scale;
                    const _Float16 h = (_Float16)v;
                    const int to = q_at + (item * QS + (e >> 1) * half + hd2 + (e & 1)) * 2;
                    *lds16(to) = h;
                    *lds16(to + cols * QS * 2) = (_Float16)(v - (float)h);
                }
            } else if (has_new && item < items) {
                const size_t vo = (size_t)(rec[3] * kv_l + kh) * kBlockTokens * HD;
                const bool isv = item > gqa;
                _Float16* const to = reinterpret_cast<_Float16*>(isv ? a.kv.v : a.kv.k) + vo;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int dim = (e >> 1) * half + hd2 + (e & 1);
                    const float v = isv ? y[e] : z[e];
                    const _Float16 h = f16_sat(v);
                    to[isv ? v_packed_offset(pos & 255, dim, HD) : k_packed_offset(pos & 255, dim, HD)] = h;
                    *lds16(new_at + (isv ? HD * 2 : 0) + dim * 2) = h;
                    if constexpr (VLO != 0) {
                        const uint8_t lo = residual24(v, h);
                        *lds8(new_kl_at + (isv ? HD : 0) + dim) = lo;
                        if (isv) (a.kv.vlo + vo)[vlo_packed_offset(pos & 255, dim, HD)] = lo;
                        else if constexpr (KLO) (a.kv.klo + vo)[klo_packed_offset(pos & 255, dim, HD)] = lo;
                    }
                }
            }
        };
#pragma unroll
        for (int it = 0; it < NI; ++it)
            if ((it * NWV + wave) * HPW < items) make(item_of(it), xa[it], xb[it], wa[it], wb[it]);
        for (int it = NI; (it * NWV + wave) * HPW < items; ++it) {
            const int item = min(item_of(it), items - 1);
            const float *p = item_src(item), *w = (item < gqa ? a.qn : a.kn) + hd2;
            float2 u = load2(p), v = load2(p + half);
            const float2 nu = load2(w), nw = load2(w + half);
            add_slabs(p, u, v);
            make(item_of(it), u, v, nu, nw);
        }
        if constexpr (!AHEAD && !ONE_SET) {
            __builtin_amdgcn_sched_barrier(0);
            load_first(1, tB);
            __builtin_amdgcn_sched_barrier(0);
        }
        NVLLM_STAMP(a, 1);
        // q and the new token are published; the tiles stay in flight
        asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
        if (has_new && (last - t_begin) % NWV == wave) new_tile = last;
        const int at = q_at + ((l15 % gqa) * QS + grp * 8) * 2;  // columns of no row repeat one: nothing of theirs is stored
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            w.qh[0][c] = *reinterpret_cast<const f16x8*>(smem_raw + at + c * 64);
            w.ql[0][c] = *reinterpret_cast<const f16x8*>(smem_raw + at + cols * QS * 2 + c * 64);
        }
        NVLLM_STAMP(a, 2);
    } else {
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            float x[8] = {0, 0, 0, 0, 0, 0, 0, 0};
            if (my_row >= 0) {
                const float4* p = reinterpret_cast<const float4*>(a.q + (size_t)my_row * ldq + (size_t)my_head * HD +
                                                                  c * 32 + grp * 8);
                const float4 u = p[0], w = p[1];
                x[0] = u.x; x[1] = u.y; x[2] = u.z; x[3] = u.w; x[4] = w.x; x[5] = w.y; x[6] = w.z; x[7] = w.w;
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const _Float16 h = (_Float16)x[j];
                w.qh[0][c][j] = h;
                w.ql[0][c][j] = (_Float16)(x[j] - (float)h);
            }
        }
    }

    w.my_row[0] = my_row;
    w.my_pos[0] = my_pos;
    w.start();
    const int first_pos = FUSED ? pmax : a.pos[row0];
    auto compute_tile = [&](int kt, const Tile& t, auto scores_made) { w.tile(kt << 5, grp, first_pos, t.k, t.kl, t.v, t.vl, scores_made); };
    {
        // Each wave takes every NWV-th 32-token tile.
        {
            // decode: two named register sets, both in flight; a set is refilled (two tiles ahead) right after it is
            // consumed.  Prefetches are unconditional (tile index clamped): no branch around loads.
            int kt = t_begin + wave;
            if constexpr (!FUSED) {  // (the fused prologue has sent for them)
                load_tile(kt, tA);
                if constexpr (!ONE_SET) load_tile(kt + NWV, tB);
            }
            // the new token into its place of a tile: K's lanes l15 == token % 16 of the token half, V's lane group and halfword
            auto patch = [&](Tile& t) {
                const int tt = pmax & 31, e = (tt >> 4) * 4 + (tt & 3);
                const bool kl = l15 == (tt & 15);
                const bool ka_lane = kl && tt < 16, kb_lane = kl && tt >= 16, v_lane = grp == ((tt & 15) >> 2);
#pragma unroll
                for (int c = 0; c < DC; ++c) {
                    const uint4 n = *reinterpret_cast<const uint4*>(lds16(new_at) + c * 32 + grp * 8);
                    uint4 &ka = t.k[2 * c], &kb = t.k[2 * c + 1];
                    ka.x = ka_lane ? n.x : ka.x; ka.y = ka_lane ? n.y : ka.y; ka.z = ka_lane ? n.z : ka.z; ka.w = ka_lane ? n.w : ka.w;
                    kb.x = kb_lane ? n.x : kb.x; kb.y = kb_lane ? n.y : kb.y; kb.z = kb_lane ? n.z : kb.z; kb.w = kb_lane ? n.w : kb.w;
                }
                uint32_t mask[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) mask[i] = v_lane && (e >> 1) == i ? ((e & 1) ? 0xffff0000u : 0x0000ffffu) : 0u;
                const uint16_t* nv = reinterpret_cast<const uint16_t*>(smem_raw + new_v_at);
#pragma unroll
                for (int d = 0; d < DT; ++d) {
                    const uint32_t n = nv[d * 16 + l15] * 0x10001u;
                    uint4& v = t.v[d];
                    v.x = (v.x & ~mask[0]) | (n & mask[0]); v.y = (v.y & ~mask[1]) | (n & mask[1]);
                    v.z = (v.z & ~mask[2]) | (n & mask[2]); v.w = (v.w & ~mask[3]) | (n & mask[3]);
                }
                if constexpr (VLO != 0) {
                    uint32_t m8[2];
#pragma unroll
                    for (int i = 0; i < 2; ++i) m8[i] = v_lane && (e >> 2) == i ? 0xffu << ((e & 3) * 8) : 0u;
#pragma unroll
                    for (int d = 0; d < DT; ++d) {
                        const uint32_t n = lds8(new_vl_at)[d * 16 + l15] * 0x1010101u;
                        uint32_t &w0 = (d & 1) ? t.vl[d >> 1].z : t.vl[d >> 1].x, &w1 = (d & 1) ? t.vl[d >> 1].w : t.vl[d >> 1].y;
                        w0 = (w0 & ~m8[0]) | (n & m8[0]);
                        w1 = (w1 & ~m8[1]) | (n & m8[1]);
                    }
                }
                if constexpr (KLO) {
#pragma unroll
                    for (int c = 0; c < DC; ++c) {
                        const uint2 n = *reinterpret_cast<const uint2*>(lds8(new_kl_at) + c * 32 + grp * 8);
                        uint4 &pa = t.kl[c >> 1], &pb = t.kl[DC / 2 + (c >> 1)];
                        uint32_t &a0 = (c & 1) ? pa.z : pa.x, &a1 = (c & 1) ? pa.w : pa.y, &b0 = (c & 1) ? pb.z : pb.x, &b1 = (c & 1) ? pb.w : pb.y;
                        a0 = ka_lane ? n.x : a0; a1 = ka_lane ? n.y : a1;
                        b0 = kb_lane ? n.x : b0; b1 = kb_lane ? n.y : b1;
                    }
                }
            };
            if constexpr (ONE_SET) {
                // 24-bit cache: one 24 KiB set per wave and two waves per SIMD (a second set needs > 256 registers: half the
                // workgroups resident, two rounds) -- the other seven waves of the CU cover this wave's round trip; the next tile's K is sent
                // for as soon as the scores are made (24 rows of 48 to 400 tokens 17.3 -> 16.5 us, 64 of 64 to 512 28.5)
                while (kt < t_end) {
                    if (FUSED && kt == new_tile) patch(tA);
                    compute_tile(kt, tA, [&] { load_k(kt + NWV, tA); });
                    load_v(kt + NWV, tA);
                    kt += NWV;
                }
            } else {
                while (kt < t_end) {
                    if (FUSED && kt == new_tile) patch(tA);
                    compute_tile(kt, tA, [] {});
                    load_tile(kt + 2 * NWV, tA);
                    kt += NWV;
                    if (kt >= t_end) break;
                    if (FUSED && kt == new_tile) patch(tB);
                    compute_tile(kt, tB, [] {});
                    load_tile(kt + 2 * NWV, tB);
                    kt += NWV;
                }
            }
        }
    }

    // merge the NWV waves' partial (m, l, O): columns that are rows of q only, one barrier; a thread then owns four dims of a column
    NVLLM_STAMP(a, 3);
    float lsum = w.lsum[0];
    lsum += __shfl_xor(lsum, 16);
    lsum += __shfl_xor(lsum, 32);
    if (l15 < cols) {
        if (grp == 0) {
            ml[(wave * 2 + 0) * 16 + l15] = lsum != 0.f ? w.m[0] : -1e30f;  // a wave without a visible token has no reference
            ml[(wave * 2 + 1) * 16 + l15] = lsum;
        }
#pragma unroll
        for (int d = 0; d < DT; ++d) obuf[(wave * cols + l15) * OS + d * 4 + grp] = w.o[0][d];
    }
    __syncthreads();
    auto finish = [&](int row, int head, int d4, const f32x4& acc, float ltot) __attribute__((always_inline)) {
        const float inv = 1.0f / ltot;
        const float y0 = acc[0] * inv, y1 = acc[1] * inv, y2 = acc[2] * inv, y3 = acc[3] * inv;
        const size_t base = (size_t)row * ldq + (size_t)head * HD + d4 * 4;
        if (a.out_f32) *reinterpret_cast<float4*>(a.out_f32 + base) = make_float4(y0, y1, y2, y3);
        if (a.out_hi) {
            uint16_t h0, h1, h2, h3, l0, l1, l2, l3;
            split_bf16(y0, h0, l0); split_bf16(y1, h1, l1); split_bf16(y2, h2, l2); split_bf16(y3, h3, l3);
            const size_t xo = a.out_packed ? xpack_off(row, head * HD + d4 * 4, ldq >> 5) : base;
            *reinterpret_cast<uint2*>(a.out_hi + xo) = make_uint2(h0 | ((uint32_t)h1 << 16), h2 | ((uint32_t)h3 << 16));
            *reinterpret_cast<uint2*>(a.out_lo + xo) = make_uint2(l0 | ((uint32_t)l1 << 16), l2 | ((uint32_t)l3 << 16));
        }
    };
    const int n_parts = PARTS && a.part_tiles ? (n_kv_tiles + a.part_tiles - 1) / a.part_tiles : 1;
    for (int i = threadIdx.x; i < cols * (HD / 4); i += NWV * 64) {
        const int col = i / (HD / 4), d4 = i % (HD / 4), tok = FUSED ? 0 : col / gqa;
        if (tok >= nrows || (!FUSED && col >= tpq * gqa)) continue;
        const int row = row0 + tok, head = kh * gqa + (FUSED ? col : col % gqa);
        float ms = -1e30f;
#pragma unroll
        for (int q = 0; q < NWV; ++q) ms = fmaxf(ms, ml[(q * 2 + 0) * 16 + col]);
        float ltot = 0.f;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int q = 0; q < NWV; ++q) {
            const float f = exp2f(ml[(q * 2 + 0) * 16 + col] - ms);
            const f32x4 v = obuf[(q * cols + col) * OS + d4];
            ltot += ml[(q * 2 + 1) * 16 + col] * f;
            acc[0] += v[0] * f; acc[1] += v[1] * f; acc[2] += v[2] * f; acc[3] += v[3] * f;
        }
        if (n_parts > 1) {
            // partial: O (at the workgroup's max) for whoever merges the parts
            const size_t part = ((size_t)row * a.nh_l + head) * a.max_parts + blockIdx.z;
            float *const to = a.part_o + part * HD + d4 * 4, *const to_ml = a.part_ml + part * 2;
            if constexpr (FUSED) {
                auto word = [](float v) { return __builtin_bit_cast(uint32_t, v); };
                hand_on16(reinterpret_cast<uint32_t*>(to), word(acc[0]), word(acc[1]), word(acc[2]), word(acc[3]));
                if (d4 == 0) hand_on8(reinterpret_cast<uint32_t*>(to_ml), word(ms), word(ltot));
            } else {
                *reinterpret_cast<float4*>(to) = make_float4(acc[0], acc[1], acc[2], acc[3]);
                if (d4 == 0) { to_ml[0] = ms; to_ml[1] = ltot; }
            }
            continue;
        }
        finish(row, head, d4, acc, ltot);
    }
    if constexpr (FUSED && PARTS) {
        if (n_parts > 1) {
            // The part that ends last merges them, in their order: which one it is changes nothing.  Parts are handed on past the L2s, each wave waits for its own stores and the barrier for
            // the waves, so that who counts n_parts - 1 others can read them.  As a launch of its own behind this one, steps of 0.6B: 9 rows of 600 tokens 1063 us, now 1006, 10 of 100 to 1000 1089 and 1032,
            // 16 of 1500 1337 and 1290, 1 of 16000 1344 and 1106.
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
            int* const seen = reinterpret_cast<int*>(smem_raw);  // (ml and obuf are read)
            if (threadIdx.x == 0) *seen = __hip_atomic_fetch_add(a.part_done + (size_t)row0 * a.kv.kv_l + kh, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __syncthreads();
            if (*seen != n_parts - 1) return;
            if (threadIdx.x == 0) __hip_atomic_store(a.part_done + (size_t)row0 * a.kv.kv_l + kh, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            // One buffer for all of the row's heads: with a head's own, which differs between the lanes of a wave, each load was a loop over the wave's heads, two of 128 or four of 64.  Six layers with 16
            // heads of 64 on four, 2 x 9000 tokens, us: the merge as a launch 271, with such loops 336, now 220; 14 heads of 128 on two, 1 x 16000: 462, 412, 368.
            const size_t row_parts = (size_t)row0 * a.nh_l * a.max_parts;
            const auto ro = buffer_of(a.part_o + row_parts * HD, a.nh_l * a.max_parts * HD * 4), rm = buffer_of(a.part_ml + row_parts * 2, a.nh_l * a.max_parts * 8);
            for (int i = threadIdx.x; i < cols * (HD / 4); i += NWV * 64) {
                const int col = i / (HD / 4), d4 = i % (HD / 4), head = kh * gqa + col, part = head * a.max_parts;
                float ms = -1e30f, ltot = 0.f;
                f32x4 acc = {0.f, 0.f, 0.f, 0.f};
                constexpr int B = 8, kNoPart = 0x7ffffff0;  // parts at a time; a place past any buffer's end
                for (int s0 = 0; s0 < n_parts; s0 += B) {
                    float2 pm[B];
                    float4 po[B];
#pragma unroll
                    for (int s = 0; s < B; ++s) {  // (past the last one: zeros, which count nothing)
                        const bool there = s0 + s < n_parts;
                        pm[s] = __builtin_bit_cast(float2, load_shared8(rm, there ? (part + s0 + s) * 8 : kNoPart));
                        po[s] = __builtin_bit_cast(float4, load_shared16(ro, there ? ((part + s0 + s) * HD + d4 * 4) * 4 : kNoPart));
                    }
                    float to = ms;
#pragma unroll
                    for (int s = 0; s < B; ++s) to = s0 + s < n_parts ? fmaxf(to, pm[s].x) : to;
                    const float f0 = exp2f(ms - to);
                    ms = to;
                    ltot *= f0;
                    acc[0] *= f0; acc[1] *= f0; acc[2] *= f0; acc[3] *= f0;
#pragma unroll
                    for (int s = 0; s < B; ++s) {
                        const float f = s0 + s < n_parts ? exp2f(pm[s].x - ms) : 0.f;
                        ltot += pm[s].y * f;
                        acc[0] += po[s].x * f; acc[1] += po[s].y * f; acc[2] += po[s].z * f; acc[3] += po[s].w * f;
                    }
                }
                finish(row0, head, d4, acc, ltot);
            }
        }
    }
    NVLLM_STAMP(a, 4);
}
template <int HD, int NWV, bool FUSED, int VLO = 0>
__global__ void __launch_bounds__(NWV * 64, 2) attn_paged_kernel(AttnArgs a) {
    attn_paged_body<HD, NWV, FUSED, VLO, false, !FUSED>(a);
}
// The fused form where contexts are in parts.  With the merge behind the whole contexts too, 16 steps of 64 rows of 64 to 512 tokens took 23.2 ms, not 22.96.
template <int HD, int NWV, int VLO>
__global__ void __launch_bounds__(NWV * 64, 2) attn_parts_kernel(AttnArgs a) {
    attn_paged_body<HD, NWV, true, VLO, false, true>(a);
}
template <int HD, int NWV>
__global__ void __launch_bounds__(NWV * 64, 2) attn_paged_ahead_kernel(AttnArgs a) {
    attn_paged_body<HD, NWV, true, 0, true, false>(a);
}

// ---------------------------------------------------------------------------------------------------
// Prefill attention with LDS-staged K/V (same math as attn_paged_kernel, qwen3.rs:236-277).
// One workgroup = FOUR consecutive q-tiles of ONE sequence (host pads every sequence's tile list to a multiple of four
// with empty tiles) x one kv head x 4 NH waves: wave w owns q-tile w % 4 and every NH-th 32-token K/V tile of the context; with NH = 2
// the two halves of a q-tile meet in LDS at the end.  A set of NH tiles is fetched ONCE per workgroup -- 16 KiB each by LDS-DMA, 1 KiB
// per wave-instruction, already in MFMA fragment order so the image is lane-linear -- and read from LDS by the waves that still need it
// (causal: a wave stops after the tile that holds its last token); two sets are in flight while one is consumed.
// What bounds it: the chain of one wave through its tiles (QK^T, softmax, PV depend on each other), two waves per SIMD; by counters the
// matrix cores are busy 45 % of the time, the VALU another 45 %.  NH = 2 halves the chain of the longest context, which sets the end of
// a launch that does not fill the chip twice over.  Measured per launch (16 / 8 heads of 128) with a maximum across lanes, a rescale and
// a drained ring in every tile, NH = 1: one prompt of 2391 tokens 109 us, now 65; 18.7 k tokens in prompts of 64 to 512, chunks of 4096
// rows, 34.5 -> 30.7; 32 / 8 heads, 4050 tokens in prompts of 700 to 2000, 152 -> 118.  When to take which: attn_prefill_two (most launches that two sets
// once were for are the dealt form's below).  VLO: a 24-bit cache (see attn_paged_kernel), whose residual fragments ride in the same ring: 5.4 k tokens in prompts
// of 48 to 400, 88 us with K and V straight to registers for every q-tile of its own, now 39 and, with NH = 2, 30.
// ---------------------------------------------------------------------------------------------------
template <int HD, int QT, int NH, int VLO>
__global__ void __launch_bounds__(NH * 256, 2) attn_prefill_kernel(AttnArgs a) {
    constexpr int DC = HD / 32, DT = HD / 16, NWV = 4;
    constexpr bool KLO = VLO == 2;
    constexpr int DL = VLO ? DT / 2 : 0;               // 1 KiB residual fragments of V (two PV fragments each) ...
    constexpr int V0 = 2 * DC, VL0 = V0 + DT, KL0 = VL0 + DL;  // ... and of K: [token half][DC / 2]
    constexpr int TILE_FRAGS = KL0 + (KLO ? DC : 0);  // 1 KiB fragments of one 32-token K/V tile: K lo half, K hi half, V, residuals
    constexpr int SET = NH * TILE_FRAGS, COPIES = SET / (4 * NH);  // fragments of NH neighbouring tiles, copies of a wave for them
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    uint4* lds = reinterpret_cast<uint4*>(smem_raw);  // [3 stages][NH tiles][TILE_FRAGS][64]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l15 = lane & 15, grp = lane >> 4;
    // 1-D grid, kv heads fastest, groups in the host's longest-first order: the dispatcher hands out workgroups in index
    // order, so what is left over when all CU slots are taken (528 workgroups for 512 slots on a 4096-row chunk) must
    // be the short contexts -- in launch order the late starters were long ones and set the kernel's end
    const int kv_l = a.kv.kv_l;
    const int gi = (int)blockIdx.x / kv_l, kh = (int)blockIdx.x - gi * kv_l;
    const int qw = wave & 3, part = wave >> 2;
    NVLLM_STAMP(a, 0);
    const PrefillTile q = prefill_tile(a, gi * NWV + qw);
    const int gqa = a.gqa, ldq = a.nh_l * HD;
    AttnWave<HD, QT, VLO> w;
    w.rows(q, gqa, l15);
    const int my_head = kh * gqa + (l15 % gqa);
    // tiles this wave needs: up to its last token; tiles the workgroup stages: up to the last token of its last real tile
    const int my_last = q.nrows > 0 ? (q.first + q.nrows - 1) >> 5 : -1, wg_last = q.group_last >> 5;
    if (wg_last < 0) return;  // four empty tiles (uniform)
    const int* bt = a.block_tables + (size_t)q.slot * a.max_blocks;
    const _Float16* kbase = reinterpret_cast<const _Float16*>(a.kv.k);
    const _Float16* vbase = reinterpret_cast<const _Float16*>(a.kv.v);
    const uint32_t lds0 = lds_address(smem_raw);
    const int last_set = wg_last / NH;
    // Block id of a set of NH tiles (never across two blocks) by an explicit scalar load (hipcc turns the plain bt[] read into a vector
    // load once the kernel has issued LDS-DMA writes -- no "noclobber" proof -- and then waits vmcnt(0) for it every iteration,
    // draining the K/V tiles in flight).  Issued one iteration before its use; blk_ready() is the wait, tied to the value.
    auto blk_load = [&](int it_) {
        int v;
        const int* p = bt + (min(it_, last_set) * NH >> 3);  // 8 tiles per 256-token block
        asm volatile("s_load_dword %0, %1, 0x0" : "=s"(v) : "s"(p));
        return v;
    };
    auto blk_ready = [&](int& v) { asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(v)::"memory"); };
    // stage a set into buffer buf: fragment f goes to wave f % (4 NH).  A pair's second tile may lie past the context: it is in the
    // same block, nobody reads it
    auto stage = [&](int it, int buf, int blk) {
        const int tb = (it * NH << 5) & 255;
        const _Float16* kb = kbase + (size_t)(blk * kv_l + kh) * kBlockTokens * HD + (size_t)(tb >> 4) * (DC * 512) + lane * 8;
        const _Float16* vb = vbase + (size_t)(blk * kv_l + kh) * kBlockTokens * HD + (size_t)(tb >> 5) * (DT * 512) + lane * 8;
#pragma unroll
        for (int i = 0; i < COPIES; ++i) {
            const int f = wave + i * 4 * NH, second = f >= TILE_FRAGS, ft = second ? f - TILE_FRAGS : f;
            const void* src = ft < V0 ? kb + (second * 2 * DC + ft) * 512 : vb + (second * DT + ft - V0) * 512;
            if constexpr (VLO != 0) {
                const size_t slab = (size_t)(blk * kv_l + kh) * kBlockTokens * HD + (size_t)(tb >> 5) * (HD * 32) + lane * 16;
                if (ft >= KL0) src = a.kv.klo + slab + (second * DC + ft - KL0) * 1024;
                else if (ft >= VL0) src = a.kv.vlo + slab + (second * DL + ft - VL0) * 1024;
            }
            lds_dma16(src, lds0 + (uint32_t)(buf * SET + f) * 1024);
        }
    };
    // ring of three stages: set it+2 is issued right after the barrier that opens set it, so a set has two iterations to land
    stage(0, 0, q.block0);
    if (last_set >= 1) stage(1, 1, q.block0);
    int blk_pf = blk_load(2);
    // A wave whose tile fills up the group reads no q: prompts of 2 or 3 tokens, of whose waves three in four are that, 47 of them, 16 heads on 8, 11.4 us a launch with it, now 10.6.  The
    // others ask for all of it at once (by sub-tile, where it has rows: 64 x 200, 40 heads on 8, 187 -> 194).
    float4 q_raw[QT][DC][2] = {};
    if (q.nrows > 0) w.load_q(a, q, my_head, grp, q_raw);
    w.begin(q_raw);
    NVLLM_STAMP(a, 1);
#ifdef NVLLM_STAMPS
    if (a.stamps && lane == 0) {  // iteration counts ride in two stamp slots
        a.stamps[((size_t)blockIdx.x * 16 + wave) * 8 + 5] = (unsigned long long)(wg_last + 1);
        a.stamps[((size_t)blockIdx.x * 16 + wave) * 8 + 6] = (unsigned long long)(my_last + 1);
    }
#endif
    int buf = 0;
    for (int it = 0; it <= last_set; ++it, buf = buf == 2 ? 0 : buf + 1) {
        // every wave waits for its own copies of set it (all but the COPIES newest: those are set it+1),
        // then the barrier publishes them and says the stage read in iteration it-1 is free.  Raw barrier: a
        // __syncthreads() here drains vmcnt(0) and with it the set that is meant to stay in flight.
        if (it + 1 <= last_set) asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(COPIES) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
        blk_ready(blk_pf);
        if (it + 2 <= last_set) stage(it + 2, buf == 0 ? 2 : buf - 1, blk_pf);
        blk_pf = blk_load(it + 3);
        const int kt = NH * it + part;
        if (kt > my_last) continue;                 // causal: this wave's rows end before this tile (it still stages)
        const uint4* tile_lds = lds + (size_t)(buf * NH + part) * TILE_FRAGS * 64 + lane;
        const int T0 = kt << 5;
        // All K fragments of the tile are asked for before its first MFMA, all V fragments before the softmax, which hides them: left to
        // the compiler, two fragments at a time were asked for and waited for, eight LDS round trips a tile.
        uint4 fr[2 * DC];
#pragma unroll
        for (int c = 0; c < DC; ++c) { fr[2 * c] = tile_lds[c * 64]; fr[2 * c + 1] = tile_lds[(DC + c) * 64]; }
        [[maybe_unused]] uint4 frl[KLO ? DC : 1];
        if constexpr (KLO)
#pragma unroll
            for (int c = 0; c < DC; ++c) frl[c] = tile_lds[(KL0 + c) * 64];
        __builtin_amdgcn_sched_barrier(0);
        uint4 fv[DT];
        [[maybe_unused]] uint4 fvl[VLO ? DL : 1];
        w.tile(T0, grp, q.first, fr, frl, fv, fvl, [&] {
#pragma unroll
            for (int d = 0; d < DT; ++d) fv[d] = tile_lds[(V0 + d) * 64];
            if constexpr (VLO != 0)
#pragma unroll
                for (int d = 0; d < DL; ++d) fvl[d] = tile_lds[(VL0 + d) * 64];
            __builtin_amdgcn_sched_barrier(0);
        });
        // O's registers are the next tile's: without this the compiler keeps half of them a second time for the loop's end and copies them there with every tile (16 instructions; 34 x 211 tokens
        // behind 1764, 16 heads on 8: 249 us a launch with them, 241 without; 4 x 2000, 28 on 4: 231 and 224)
#pragma unroll
        for (int t = 0; t < QT; ++t)
#pragma unroll
            for (int d = 0; d < DT; ++d) asm volatile("" : "+v"(w.o[t][d]));
    }
    NVLLM_STAMP(a, 2);
    if constexpr (NH == 2) {
        // the odd tiles' half of every q-tile to LDS (the ring is free once all waves are here: no copy is in flight), the even ones' takes it
        asm volatile("s_barrier" ::: "memory");
        f32x4* obuf = reinterpret_cast<f32x4*>(smem_raw);                               // [4 q-tiles][QT][DT][64]
        float2* mlbuf = reinterpret_cast<float2*>(obuf + (size_t)NWV * QT * DT * 64);   // [4][QT][64]
        if (part) {
#pragma unroll
            for (int t = 0; t < QT; ++t) {
                mlbuf[(qw * QT + t) * 64 + lane] = make_float2(w.m[t], w.lsum[t]);
#pragma unroll
                for (int d = 0; d < DT; ++d) obuf[((qw * QT + t) * DT + d) * 64 + lane] = w.o[t][d];
            }
        }
        __syncthreads();
        if (part) return;
#pragma unroll
        for (int t = 0; t < QT; ++t) {
            const float2 other = mlbuf[(qw * QT + t) * 64 + lane];
            float l1 = other.y;  // of the row: a half without a visible token has no reference
            l1 += __shfl_xor(l1, 16);
            l1 += __shfl_xor(l1, 32);
            const float mo = l1 == 0.f ? w.m[t] : other.x, mn = fmaxf(w.m[t], mo);
            const float f0 = __builtin_amdgcn_exp2f(w.m[t] - mn), f1 = __builtin_amdgcn_exp2f(mo - mn);
            w.lsum[t] = w.lsum[t] * f0 + other.y * f1;
#pragma unroll
            for (int d = 0; d < DT; ++d) {
                const f32x4 v = obuf[((qw * QT + t) * DT + d) * 64 + lane];
#pragma unroll
                for (int r = 0; r < 4; ++r) w.o[t][d][r] = w.o[t][d][r] * f0 + v[r] * f1;
            }
        }
    }
    // normalise and store (D[dim 4*grp+reg][q row l15] -> out[row][head dims])
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        float l = w.lsum[t];
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        if (w.my_row[t] < 0) continue;
        const float inv = 1.0f / l;
        const size_t base = (size_t)w.my_row[t] * ldq + (size_t)my_head * HD + grp * 4;
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            const float y0 = w.o[t][d][0] * inv, y1 = w.o[t][d][1] * inv, y2 = w.o[t][d][2] * inv, y3 = w.o[t][d][3] * inv;
            if (a.out_f32) *reinterpret_cast<float4*>(a.out_f32 + base + d * 16) = make_float4(y0, y1, y2, y3);
            if (a.out_hi) {
                uint16_t h0, h1, h2, h3, l0, l1, l2, l3;
                split_bf16(y0, h0, l0); split_bf16(y1, h1, l1); split_bf16(y2, h2, l2); split_bf16(y3, h3, l3);
                const size_t xo = a.out_packed ? xpack_off(w.my_row[t], my_head * HD + d * 16 + grp * 4, ldq >> 5) : base + d * 16;
                *reinterpret_cast<uint2*>(a.out_hi + xo) = make_uint2(h0 | ((uint32_t)h1 << 16), h2 | ((uint32_t)h3 << 16));
                *reinterpret_cast<uint2*>(a.out_lo + xo) = make_uint2(l0 | ((uint32_t)l1 << 16), l2 | ((uint32_t)l3 << 16));
            }
        }
    }
    NVLLM_STAMP(a, 3);
}

// ---------------------------------------------------------------------------------------------------
// The same for launches that leave CUs idle or wait for their longest context (attn_prefill_deals): ONE q-tile to a workgroup, its K/V tiles dealt
// to four waves, which take theirs straight to registers (K of the next tile behind the scores, V behind the products) and meet in LDS at the
// end.  A wave's chain is a quarter of the context where four q-tiles and two sets of waves to a workgroup leave it half, a prompt of 117 tokens is 64 workgroups
// instead of 16; for it K and V come through L2 once per q-tile instead of once per four, so a launch that fills the chip with short contexts keeps the form
// above.  Its q-tiles are those with rows: an empty one that fills up a group ends at once, but workgroups go out in turn, and where every fourth has work (24 prompts of
// 5 to 9 tokens that continue 1000) the work met on a part of the CUs: 42.4 us a launch with the empty ones, 27.2 without.  By events, 16 heads on 8: 117 tokens 14.2 -> 10.8 us (in the kernel 6.7: 2.3 to the first scores, 2.1 for the one tile of each wave, 1.8 to merge and store),
// 500 24.1 -> 13.3, 1000 34.7 -> 19.6, 2391 67.7 -> 51.6.  There it is bound by what a CU takes in, 2.8 MB, and by the matrix cores and VALU of eight waves a CU
// (36 us of 51.6 at the rate of the form above when full).
// ---------------------------------------------------------------------------------------------------
template <int HD, int QT, int VLO>
__global__ void __launch_bounds__(256, 2) attn_prefill_dealt_kernel(AttnArgs a) {
    using W = AttnWave<HD, QT, VLO>;
    constexpr int DC = W::DC, DT = W::DT, DL = W::DL, NWV = 4;
    constexpr bool KLO = W::KLO;
    extern __shared__ __attribute__((aligned(16))) char smem_raw[];
    f32x4* obuf = reinterpret_cast<f32x4*>(smem_raw);                              // [NWV][QT][DT][64]
    float2* ml = reinterpret_cast<float2*>(obuf + (size_t)NWV * QT * DT * 64);     // [NWV][QT][16]
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int l15 = lane & 15, grp = lane >> 4;
    const int kv_l = a.kv.kv_l, ti = (int)blockIdx.x / kv_l, kh = (int)blockIdx.x - ti * kv_l;
    NVLLM_STAMP(a, 0);
    const PrefillTile q = prefill_tile(a, ti);
    if (q.nrows <= 0) return;
    W w;
    w.rows(q, a.gqa, l15);
    const int end = ((q.first + q.nrows - 1) >> 5) + 1;  // K/V tiles of this q-tile
    const int my_head = kh * a.gqa + (l15 % a.gqa), ldq = a.nh_l * HD;
    float4 q_raw[QT][DC][2];
    w.load_q(a, q, my_head, grp, q_raw);
    const uniform_ints_t bt = uniform_ints(a.block_tables + (size_t)q.slot * a.max_blocks);
    uint4 fr[2 * DC], frl[KLO ? DC : 1], fv[DT], fvl[VLO ? DL : 1];
    // tiles past the end are loads from buffers of no bytes (see attn_paged_kernel)
    auto load_k = [&](int kt, int blk) {
        const int T0 = min(kt, end - 1) << 5, slab = blk * kv_l + kh, tb = T0 & 255, bytes = kt < end ? kBlockTokens * HD * 2 : 0;
        const auto rk = buffer_of(reinterpret_cast<const char*>(a.kv.k) + (size_t)slab * (kBlockTokens * HD * 2), bytes);
        const int ko = (tb >> 4) * (DC * 1024);
#pragma unroll
        for (int c = 0; c < DC; ++c) {
            fr[2 * c] = buffer_load16(rk, lane * 16 + c * 1024, ko);
            fr[2 * c + 1] = buffer_load16(rk, lane * 16 + c * 1024, ko + DC * 1024);
        }
        if constexpr (KLO) {
            const auto rl = buffer_of(a.kv.klo + (size_t)slab * (kBlockTokens * HD), bytes / 2);
#pragma unroll
            for (int i = 0; i < DC; ++i) frl[i] = buffer_load16(rl, lane * 16 + i * 1024, (tb >> 4) * ((DC / 2) * 1024));
        }
    };
    auto load_v = [&](int kt, int blk) {
        const int T0 = min(kt, end - 1) << 5, slab = blk * kv_l + kh, tb = T0 & 255, bytes = kt < end ? kBlockTokens * HD * 2 : 0;
        const auto rv = buffer_of(reinterpret_cast<const char*>(a.kv.v) + (size_t)slab * (kBlockTokens * HD * 2), bytes);
        const int vo = (tb >> 5) * (DT * 1024);
#pragma unroll
        for (int d = 0; d < DT; ++d) fv[d] = buffer_load16(rv, lane * 16 + (d % 4) * 1024, vo + d / 4 * 4096);
        if constexpr (VLO != 0) {
            const auto rl = buffer_of(a.kv.vlo + (size_t)slab * (kBlockTokens * HD), bytes / 2);
#pragma unroll
            for (int d = 0; d < DL; ++d) fvl[d] = buffer_load16(rl, lane * 16 + d * 1024, (tb >> 5) * (DL * 1024));
        }
    };
    __builtin_amdgcn_sched_barrier(0);
    load_k(wave, q.block0);
    if constexpr (VLO == 0) load_v(wave, q.block0);
    __builtin_amdgcn_sched_barrier(0);
    w.begin(q_raw);
    NVLLM_STAMP(a, 1);
    int blk = q.block0;
    for (int kt = wave; kt < end; kt += NWV) {
        const int next = bt[min(kt + NWV, end - 1) >> 3];  // 8 tiles in a block
        // 24-bit caches have no registers for both: V is asked for behind the scores, the next K behind the products
        w.tile(kt << 5, grp, q.first, fr, frl, fv, fvl, [&] {
            if constexpr (VLO == 0) load_k(kt + NWV, next);
            else load_v(kt, blk);
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (VLO == 0) load_v(kt + NWV, next);
        else load_k(kt + NWV, next);
        __builtin_amdgcn_sched_barrier(0);
        blk = next;
    }
    NVLLM_STAMP(a, 2);
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        float l = w.lsum[t];
        l += __shfl_xor(l, 16);
        l += __shfl_xor(l, 32);
        if (grp == 0) ml[(wave * QT + t) * 16 + l15] = make_float2(w.m[t], l);
#pragma unroll
        for (int d = 0; d < DT; ++d) obuf[((wave * QT + t) * DT + d) * 64 + lane] = w.o[t][d];
    }
    __syncthreads();
    // a wave finishes a quarter of the dims
#pragma unroll
    for (int t = 0; t < QT; ++t) {
        float2 p[NWV];
        float mn = -1e30f, l = 0.f;
#pragma unroll
        for (int q = 0; q < NWV; ++q) {
            p[q] = ml[(q * QT + t) * 16 + l15];
            if (p[q].y != 0.f) mn = fmaxf(mn, p[q].x);  // a wave without a visible token has no reference
        }
#pragma unroll
        for (int q = 0; q < NWV; ++q) {
            p[q].x = p[q].y != 0.f ? __builtin_amdgcn_exp2f(p[q].x - mn) : 0.f;
            l += p[q].x * p[q].y;
        }
        if (w.my_row[t] < 0) continue;
        const float inv = 1.0f / l;
        const size_t base = (size_t)w.my_row[t] * ldq + (size_t)my_head * HD + grp * 4;
#pragma unroll
        for (int i = 0; i < DT / NWV; ++i) {
            const int d = wave * (DT / NWV) + i;
            f32x4 y = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < NWV; ++q) {
                const f32x4 v = obuf[((q * QT + t) * DT + d) * 64 + lane];
#pragma unroll
                for (int r = 0; r < 4; ++r) y[r] += v[r] * p[q].x;
            }
            y[0] *= inv; y[1] *= inv; y[2] *= inv; y[3] *= inv;
            if (a.out_f32) *reinterpret_cast<f32x4*>(a.out_f32 + base + d * 16) = y;
            if (a.out_hi) {
                uint16_t h[4], lo[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) split_bf16(y[r], h[r], lo[r]);
                const size_t xo = a.out_packed ? xpack_off(w.my_row[t], my_head * HD + d * 16 + grp * 4, ldq >> 5) : base + d * 16;
                *reinterpret_cast<uint2*>(a.out_hi + xo) = make_uint2(h[0] | ((uint32_t)h[1] << 16), h[2] | ((uint32_t)h[3] << 16));
                *reinterpret_cast<uint2*>(a.out_lo + xo) = make_uint2(lo[0] | ((uint32_t)lo[1] << 16), lo[2] | ((uint32_t)lo[3] << 16));
            }
        }
    }
    NVLLM_STAMP(a, 3);
}

// merge the split-KV partials of one (row, q head): one wave each, lane = 2 (HD 128) or 1 (HD 64) dims
template <int HD>
__global__ void __launch_bounds__(256) attn_combine_kernel(AttnArgs a, int rows) {
    const int lane = threadIdx.x & 63;
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (item >= rows * a.nh_l) return;
    const int row = item / a.nh_l, head = item - row * a.nh_l;
    const int n_parts = (((a.pos[row] >> 5) + 1) + a.part_tiles - 1) / a.part_tiles;
    if (n_parts <= 1) return;  // the attention kernel wrote the final output itself
    const float* pm = a.part_ml + ((size_t)row * a.nh_l + head) * a.max_parts * 2;
    const float* po = a.part_o + ((size_t)row * a.nh_l + head) * a.max_parts * HD;
    float ms = -1e30f;
    for (int s = 0; s < n_parts; ++s) ms = fmaxf(ms, pm[2 * s]);
    float lt = 0.f;
    constexpr int PER = HD / 64;
    float acc[PER];
#pragma unroll
    for (int j = 0; j < PER; ++j) acc[j] = 0.f;
    for (int s = 0; s < n_parts; ++s) {
        const float f = exp2f(pm[2 * s] - ms);
        lt += pm[2 * s + 1] * f;
#pragma unroll
        for (int j = 0; j < PER; ++j) acc[j] += po[(size_t)s * HD + lane * PER + j] * f;
    }
    const float inv = 1.0f / lt;
    const size_t base = (size_t)row * (a.nh_l * HD) + (size_t)head * HD + lane * PER;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
        const float y = acc[j] * inv;
        if (a.out_f32) a.out_f32[base + j] = y;
        if (a.out_hi) {
            uint16_t h, l;
            split_bf16(y, h, l);
            const size_t xo = a.out_packed ? xpack_off(row, head * HD + lane * PER + j, (a.nh_l * HD) >> 5) : base + j;
            a.out_hi[xo] = h;
            a.out_lo[xo] = l;
        }
    }
}

template <int HD, int NWV, bool FUSED, int VLO, bool AHEAD = false>
static hipError_t attn_launch_v(const AttnArgs& a, int n_tiles, int grid_z, hipStream_t s) {
    auto lds_of = [](int gqa) { return NWV * 2 * 16 * 4 + (size_t)NWV * gqa * (HD * 4 + 16) + (FUSED ? (size_t)gqa * (HD + 8) * 4 + HD * 6 : 0); };
    const size_t lds = lds_of(FUSED ? a.gqa : 16);
    static std::atomic<uint64_t> lds_set{0};
    void (*kernel)(AttnArgs) = attn_paged_kernel<HD, NWV, FUSED, VLO>;
    if constexpr (AHEAD) kernel = attn_paged_ahead_kernel<HD, NWV>;
    static std::atomic<uint64_t> lds_set_parts{0};
    const bool parts = FUSED && a.part_tiles;
    if constexpr (FUSED) if (parts) kernel = attn_parts_kernel<HD, NWV, VLO>;
    ensure_dyn_lds(reinterpret_cast<const void*>(kernel), lds_of(16), parts ? lds_set_parts : lds_set);
    dim3 grid = FUSED ? dim3(a.kv.kv_l, n_tiles, grid_z) : dim3(n_tiles * a.kv.kv_l, 1, grid_z);
    kernel<<<grid, NWV * 64, lds, s>>>(a);
    return hipGetLastError();
}
template <int HD, int NWV, bool FUSED>
static hipError_t attn_launch_t(const AttnArgs& a, int n_tiles, int grid_z, hipStream_t s) {
    // 24-bit V (KvLayout::vlo) is served for head_dim 128 only (every Qwen3 size); the pool refuses it otherwise
    if (a.kv.klo && !a.kv.vlo) return hipErrorInvalidValue;  // 24-bit K comes with 24-bit V only
    if constexpr (HD == 128) {
        if (a.kv.klo) return attn_launch_v<HD, NWV, FUSED, 2>(a, n_tiles, grid_z, s);
        if (a.kv.vlo) return attn_launch_v<HD, NWV, FUSED, 1>(a, n_tiles, grid_z, s);
    } else if (a.kv.vlo) return hipErrorNotSupported;
    return attn_launch_v<HD, NWV, FUSED, 0>(a, n_tiles, grid_z, s);
}

template <int HD, int VLO>
static hipError_t attn_prefill_dealt_v(const AttnArgs& a, int n_tiles, hipStream_t s) {
    constexpr size_t lds = (size_t)4 * 2 * (HD / 16 * 64 * 16 + 16 * 8);
    static std::atomic<uint64_t> lds_set{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(attn_prefill_dealt_kernel<HD, 2, VLO>), lds, lds_set);
    attn_prefill_dealt_kernel<HD, 2, VLO><<<n_tiles * a.kv.kv_l, 256, lds, s>>>(a);
    return hipGetLastError();
}
template <int HD>
static hipError_t attn_prefill_dealt(const AttnArgs& a, int n_tiles, hipStream_t s) {
    if constexpr (HD == 128) {
        if (a.kv.klo) return attn_prefill_dealt_v<HD, 2>(a, n_tiles, s);
        if (a.kv.vlo) return attn_prefill_dealt_v<HD, 1>(a, n_tiles, s);
    } else if (a.kv.vlo) return hipErrorNotSupported;
    return attn_prefill_dealt_v<HD, 0>(a, n_tiles, s);
}

template <int HD, int NH, int VLO>
static hipError_t attn_prefill_launch_v(const AttnArgs& a, int groups, hipStream_t s) {
    constexpr int frags = 2 * (HD / 32) + HD / 16 + (VLO ? HD / 32 : 0) + (VLO == 2 ? HD / 32 : 0);
    constexpr size_t ring = (size_t)3 * NH * frags * 1024, merge = NH == 2 ? (size_t)4 * 2 * 64 * (HD / 16 * 16 + 8) : 0;
    constexpr size_t lds = ring > merge ? ring : merge;
    static std::atomic<uint64_t> lds_set{0};
    ensure_dyn_lds(reinterpret_cast<const void*>(attn_prefill_kernel<HD, 2, NH, VLO>), lds, lds_set);
    attn_prefill_kernel<HD, 2, NH, VLO><<<groups * a.kv.kv_l, NH * 256, lds, s>>>(a);
    return hipGetLastError();
}
template <int HD, int NH>
static hipError_t attn_prefill_launch(const AttnArgs& a, int groups, hipStream_t s) {
    if constexpr (HD == 128) {  // a 24-bit cache is served for head_dim 128 only; the pool refuses it otherwise
        if (a.kv.klo) return attn_prefill_launch_v<HD, NH, 2>(a, groups, s);
        if (a.kv.vlo) return attn_prefill_launch_v<HD, NH, 1>(a, groups, s);
    } else if (a.kv.vlo) return hipErrorNotSupported;
    return attn_prefill_launch_v<HD, NH, 0>(a, groups, s);
}
// One q-tile to a workgroup or four?  Alone, the longest chain is a quarter as long and small launches have CUs for it, but every q-tile reads its K/V
// for itself and pays a prologue and a merge, about 8 us a round of 512 workgroups.  The line is the workgroups of the shared form against the longest context, placed
// by 320 launches of 8 groupings of heads (2 to 40 heads on 2 to 8, of 128 and 64, 16 and 24 bits; together within 0.2 % of the faster form each
// time; always shared: 25 to 34 % slower).  16 heads on 8, us by events, shared / alone:
//   16 bits  1 x 16 10.2 / 10.5, 117 13.6 / 10.8, 250 17.7 / 11.4, 500 23.7 / 13.3, 1000 34.4 / 19.6, 2391 66.6 / 51.6, 4000 124.8 / 113.2
//            4 x 100 13.3 / 11.5, 8 x 100 13.2 / 13.5, 24 x 100 17.7 / 28.4; 4 x 250 18.3 / 14.6, 8 x 250 19.9 / 22.8; 3 x 700 32.8 / 29.8, 5 x 700 35.2 / 39.9;
//            3 x 1000 43.1 / 40.3, 4 x 1000 46.1 / 51.9, 2 x 2000 78.7 / 71.5; 12 x 64 to 512 29.3 / 38.1, 64 x 16 to 100 25.0 / 48.8
//   24 bits  1 x 16 11.6 / 10.5, 117 17.8 / 11.3, 1000 49.2 / 24.1, 2391 100 / 69; 16 x 60 15.6 / 14.6, 24 x 100 20.1 / 29.3, 8 x 250 25.0 / 24.3,
//            8 x 380 34.7 / 35.4, 4 x 1000 69.2 / 64.0, 8 x 16 to 900 60.8 / 52.0, 12 x 64 to 512 40.8 / 42.5
//   heads of 64  1 x 117 11.1 / 8.7, 1000 22.9 / 12.2, 5 x 700 24.5 / 23.4, 4 x 1000 31.1 / 29.4, 24 x 100 12.8 / 17.3
// (heads of 64, 14 on 2: 8 x 250 15.2 / 17.2, 12 x 64 to 512 20.3 / 22.4, 16 x 100 behind a cached 100 13.6 / 15.6)
// That line is a prompt's, whose contexts are half of the longest on the average.  Behind cached prefixes all are as long as the longest, and where many such contexts do not
// fit an XCD's L2 (4 MB; with fewer than eight key heads several XCDs read each) what the q-tiles read again comes from further away: then the K/V tiles of all q-tiles, over 512
// workgroups, may be 1.2 times the longest context's, twice where the shared form has more than 256 workgroups and so one set of waves.  16 bits unless noted, cached + new:
//   8 on 8  64 x 1000 + 60 71.7 / 83.7;  16 on 2  64 x 500 + 20 29.7 / 39.3, 100 x 600 + 10 29.9 / 40.9;  40 on 8  16 x 1500 + 40 53.5 / 65.3;  32 on 8  8 x 2000 + 100 65.1 / 72.7
//   32 on 2, 24 bits  40 x 1000 + 16 54.4 / 80.8, 64 x 500 + 20 71.6 / 94.9, 24 x 500 + 30 38.3 / 48.0;  but 16 on 8  3 x 2000 + 500 69.5 / 60.5, 8 x 2000 + 100 61.3 / 43.8,
//   40 x 1000 + 16 56.9 / 49.3;  32 on 8  1 x 4000 + 500 111 / 69, 3 x 2000 + 500 129 / 111;  40 on 8  8 x 2000 + 100 117 / 88
// Over 858 launches of 13 groupings of heads, a half of them behind cached prefixes, within 1.0 % of the faster form (2.2 % behind prefixes without it); over 778 of 19 groupings at random, 1 to 80
// sequences, 1.2 %.  It misses most where few key heads' contexts are a little over the line (16 on 2, 17 x 1817 + 92, 98.7 shared and dealt 120) and where prompts of very different length
// fill groups up with empty q-tiles (8 on 8, 900 and 60 x 20, 36.9 and 21.9).
bool attn_prefill_deals(const PrefillWork& w) {
    const int64_t wgs = (int64_t)w.groups * w.kv_l;
    if (w.wide_cache ? wgs > std::min(512, 80 + w.longest * 3 / 4)
                     : w.longest <= 16 ||  // one tile: nothing to deal
                       wgs > (w.hd == 64 ? std::min(512, 96 + w.longest / 2) : std::min(600, 40 + w.longest * 9 / 20))) return false;
    const double mb = (double)w.others * w.hd * (w.wide_cache ? 6 : 4) * std::max(1, w.kv_l / 8) / (1 << 20);
    const double work = (double)w.kv_tiles * w.kv_l / 512 * (w.kv_l < 8 ? 1.25 : 1), chain = w.longest / 32.0;
    return wgs <= 256 ? mb <= 5.5 || work <= 1.2 * chain : mb <= 20 || work <= 2 * chain;
}
// Two sets of waves halve the chain of the longest context and pay a merge, and 512 threads with twice the LDS leave a CU one workgroup where it took two: up to one round of
// the 256 CUs, and contexts long enough for it.  What the dealt form leaves of that: several contexts, most of them behind cached prefixes.  A 24-bit cache, with half as much work again
// in a tile, gains earlier.  us a launch with one set and with two, heads, sequences x cached + new:
//   16 bits  8 on 8  24 x 200 + 60 19.5 / 20.3, 8 x 380 23.0 / 23.3;  16 on 2  64 x 500 + 20 30.0 / 29.7, 100 x 600 + 10 32.1 / 29.9;  32 on 4  24 x 500 + 30 31.3 / 29.6, 16 x 1500 + 40 62.8 / 50.1;
//            32 on 8  8 x 2000 + 100 79.7 / 65.1;  past 256 workgroups  16 on 8  24 x 100 18.5 / 27.7, 64 x 500 + 20 41.3 / 49.4, 4 x 900 41.3 / 44.6;  8 on 8  64 x 1000 + 60 71.7 / 78.7
//   24 bits  8 on 8  24 x 100 19.4 / 20.1;  32 on 2  100 x 150 + 4 21.8 / 23.1, 64 x 200 + 8 27.5 / 26.7, 40 x 300 + 16 32.8 / 29.4, 24 x 500 + 30 46.0 / 38.3, 8 x 2000 + 100 137 / 94;
//            past 256 workgroups  32 on 2  64 x 500 + 20 56.6 / 71.6;  16 on 8  8 x 380 34.9 / 40.0, 12 x 64 to 512 41.8 / 41.4
static bool attn_prefill_two(int wgs, int longest, bool lo) { return wgs <= 256 && longest >= (lo ? 180 : 480); }
hipError_t launch_attn_prefill(const AttnArgs& a, int n_tiles, hipStream_t s) {
    if (n_tiles <= 0) return hipSuccess;
    if (a.kv.klo && !a.kv.vlo) return hipErrorInvalidValue;  // 24-bit K comes with 24-bit V only
    if (!a.tiles || (!a.deal && n_tiles % kPrefillTileGroup) || a.gqa < 1 || a.gqa > 16 || (a.kv.hd != 128 && a.kv.hd != 64)) return hipErrorInvalidValue;
    const int groups = n_tiles / 4;
    if (a.deal) return a.kv.hd == 128 ? attn_prefill_dealt<128>(a, n_tiles, s) : attn_prefill_dealt<64>(a, n_tiles, s);
    const bool two = attn_prefill_two(groups * a.kv.kv_l, a.longest, a.kv.vlo);
    if (a.kv.hd == 128) return two ? attn_prefill_launch<128, 2>(a, groups, s) : attn_prefill_launch<128, 1>(a, groups, s);
    return two ? attn_prefill_launch<64, 2>(a, groups, s) : attn_prefill_launch<64, 1>(a, groups, s);
}

// rows: number of q rows (needed by the combine pass, which the fused form has no need of); n_parts_max: ceil(max context tiles / part_tiles)
hipError_t launch_attn_paged(const AttnArgs& a, int n_tiles, int rows, int n_parts_max, hipStream_t s) {
    if (n_tiles <= 0) return hipSuccess;
    if (a.gqa < 1 || a.gqa > 16) return hipErrorInvalidValue;
    const bool split = a.part_tiles > 0 && n_parts_max > 1;
    const bool fused = a.qkv != nullptr;  // decode rows straight from the QKV GEMM's slabs
    if (split && (!a.part_o || !a.part_ml || n_parts_max > a.max_parts || (fused && !a.part_done))) return hipErrorInvalidValue;
    AttnArgs b = a;
    if (!split) b.part_tiles = 0;
    const int gz = split ? n_parts_max : 1;
    hipError_t e = hipErrorInvalidValue;
    if (fused && (!a.rows || n_tiles != rows || rows > kAttnFusedMaxRows)) return hipErrorInvalidValue;  // fused decode: tile i is row i
    if (a.waves != 4 && (a.waves != 8 || !fused || a.kv.hd != 128)) return hipErrorInvalidValue;
    if (a.ahead && (!fused || a.kv.hd != 128 || a.waves != 4 || a.kv.vlo)) return hipErrorInvalidValue;
    if (a.waves == 8) e = attn_launch_t<128, 8, true>(b, n_tiles, gz, s);
    else if (a.ahead) e = attn_launch_v<128, 4, true, 0, true>(b, n_tiles, gz, s);
    else if (a.kv.hd == 128) e = fused ? attn_launch_t<128, 4, true>(b, n_tiles, gz, s) : attn_launch_t<128, 4, false>(b, n_tiles, gz, s);
    else if (a.kv.hd == 64) e = fused ? attn_launch_t<64, 4, true>(b, n_tiles, gz, s) : attn_launch_t<64, 4, false>(b, n_tiles, gz, s);
    if (e != hipSuccess || !split || fused) return e;
    const int items = rows * a.nh_l;
    if (a.kv.hd == 128) attn_combine_kernel<128><<<(items + 3) / 4, 256, 0, s>>>(b, rows);
    else attn_combine_kernel<64><<<(items + 3) / 4, 256, 0, s>>>(b, rows);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// SwiGLU gate: SiluAndMul::forward (activation.rs:13-18): split last dim in two, silu(a)*b
// ---------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) silu_mul_kernel(const float* __restrict__ gu, int n_slabs, int64_t slab_stride,
                                                       int rows, int I, uint16_t* __restrict__ hi,
                                                       uint16_t* __restrict__ lo, float* __restrict__ y) {
    const int64_t total = (int64_t)rows * (I >> 2);
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(i / (I >> 2));
        const int c = (int)(i % (I >> 2)) * 4;
        const float* pg = gu + (size_t)r * 2 * I + c;
        float4 g = *reinterpret_cast<const float4*>(pg);
        float4 u = *reinterpret_cast<const float4*>(pg + I);
        for (int sl = 1; sl < n_slabs; ++sl) {
            const float4 g2 = *reinterpret_cast<const float4*>(pg + (size_t)sl * slab_stride);
            const float4 u2 = *reinterpret_cast<const float4*>(pg + (size_t)sl * slab_stride + I);
            g.x += g2.x; g.y += g2.y; g.z += g2.z; g.w += g2.w;
            u.x += u2.x; u.y += u2.y; u.z += u2.z; u.w += u2.w;
        }
        const float y0 = silu_mul(g.x, u.x), y1 = silu_mul(g.y, u.y);
        const float y2 = silu_mul(g.z, u.z), y3 = silu_mul(g.w, u.w);
        if (y) *reinterpret_cast<float4*>(y + (size_t)r * I + c) = make_float4(y0, y1, y2, y3);
        if (hi) {
            uint16_t h0, h1, h2, h3, l0, l1, l2, l3;
            split_bf16(y0, h0, l0); split_bf16(y1, h1, l1); split_bf16(y2, h2, l2); split_bf16(y3, h3, l3);
            *reinterpret_cast<uint2*>(hi + (size_t)r * I + c) = make_uint2(h0 | ((uint32_t)h1 << 16), h2 | ((uint32_t)h3 << 16));
            *reinterpret_cast<uint2*>(lo + (size_t)r * I + c) = make_uint2(l0 | ((uint32_t)l1 << 16), l2 | ((uint32_t)l3 << 16));
        }
    }
}
// same for the INTERLEAVED gate/up layout of the packed weight (16-row tiles: gate tile, up tile, gate tile, ...)
__global__ void __launch_bounds__(256) silu_mul_interleaved_kernel(const float* __restrict__ gu, int n_slabs,
                                                                  int64_t slab_stride, int rows, int I,
                                                                  uint16_t* __restrict__ hi, uint16_t* __restrict__ lo, int out_packed,
                                                                  GluSpec glu, float* __restrict__ y) {
    const int64_t total = (int64_t)rows * (I >> 2);
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(i / (I >> 2));
        const int c = (int)(i % (I >> 2)) * 4;  // activation feature (4 consecutive, inside one 16-tile)
        const float* pg = gu + (size_t)r * 2 * I + (size_t)(c >> 4) * 32 + (c & 15);
        float4 g = *reinterpret_cast<const float4*>(pg);
        float4 u = *reinterpret_cast<const float4*>(pg + 16);
        for (int sl0 = 1; sl0 < n_slabs; sl0 += 4) {  // four slabs per trip, independent loads (clamped index, masked sum)
            float4 g2[4], u2[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const size_t so = (size_t)min(sl0 + q, n_slabs - 1) * slab_stride;
                g2[q] = *reinterpret_cast<const float4*>(pg + so);
                u2[q] = *reinterpret_cast<const float4*>(pg + so + 16);
            }
#pragma unroll
            for (int q = 0; q < 4; ++q)
                if (sl0 + q < n_slabs) {
                    g.x += g2[q].x; g.y += g2[q].y; g.z += g2[q].z; g.w += g2[q].w;
                    u.x += u2[q].x; u.y += u2[q].y; u.z += u2[q].z; u.w += u2[q].w;
                }
        }
        if (y) {  // f32 consumers: accurate exponential and division
            const float gv[4] = {g.x, g.y, g.z, g.w}, uv[4] = {u.x, u.y, u.z, u.w};
            float r4[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const bool cl = glu.limit > 0.f;
                const float a = cl ? fminf(gv[q], glu.limit) : gv[q], b = cl ? fminf(fmaxf(uv[q], -glu.limit), glu.limit) + glu.shift : uv[q];
                r4[q] = a / (1.0f + expf(cl ? -glu.alpha * a : glu.gelu ? gelu_arg(a) : -a)) * b;
            }
            *reinterpret_cast<float4*>(y + (size_t)r * I + c) = make_float4(r4[0], r4[1], r4[2], r4[3]);
        }
        if (!hi) continue;
        const float y0 = glu_mul(g.x, u.x, glu), y1 = glu_mul(g.y, u.y, glu);
        const float y2 = glu_mul(g.z, u.z, glu), y3 = glu_mul(g.w, u.w, glu);
        uint16_t h0, h1, h2, h3, l0, l1, l2, l3;
        split_bf16(y0, h0, l0); split_bf16(y1, h1, l1); split_bf16(y2, h2, l2); split_bf16(y3, h3, l3);
        const size_t o = out_packed ? xpack_off(r, c, I >> 5) : (size_t)r * I + c;
        *reinterpret_cast<uint2*>(hi + o) = make_uint2(h0 | ((uint32_t)h1 << 16), h2 | ((uint32_t)h3 << 16));
        *reinterpret_cast<uint2*>(lo + o) = make_uint2(l0 | ((uint32_t)l1 << 16), l2 | ((uint32_t)l3 << 16));
    }
}
hipError_t launch_silu_mul_interleaved(const float* gu, int n_slabs, int64_t slab_stride, int rows, int I, bf16_bits* hi,
                                       bf16_bits* lo, int out_packed, hipStream_t s, const GluSpec& glu, float* y) {
    if (I % 16 != 0 || (out_packed && I % 32)) return hipErrorInvalidValue;
    if (rows <= 0) return hipSuccess;
    silu_mul_interleaved_kernel<<<grid_for((int64_t)rows * (I / 4)), 256, 0, s>>>(gu, n_slabs, slab_stride, rows, I, hi, lo, out_packed, glu, y);
    return hipGetLastError();
}

hipError_t launch_silu_mul(const float* gu, int n_slabs, int64_t slab_stride, int rows, int I, bf16_bits* hi,
                           bf16_bits* lo, float* y, hipStream_t s) {
    if (I % 4 != 0) return hipErrorInvalidValue;
    if (rows <= 0) return hipSuccess;
    silu_mul_kernel<<<grid_for((int64_t)rows * (I / 4)), 256, 0, s>>>(gu, n_slabs, slab_stride, rows, I, hi, lo, y);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// misc
// ---------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) slab_sum_kernel(const float* __restrict__ in, int n_slabs, int64_t slab_stride,
                                                       int64_t ld_in, const float* __restrict__ bias, int rows, int N,
                                                       float* __restrict__ y, int64_t ld_out) {
    const int64_t total = (int64_t)rows * N;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / N;
        const int n = (int)(i - r * N);
        float v = in[r * ld_in + n];
        for (int sl = 1; sl < n_slabs; ++sl) v += in[(size_t)sl * slab_stride + r * ld_in + n];
        if (bias) v += bias[n];
        y[r * ld_out + n] = v;
    }
}
hipError_t launch_slab_sum(const float* in, int n_slabs, int64_t slab_stride, const float* bias, int rows, int N,
                           float* y, hipStream_t s) {
    return launch_slab_sum_ld(in, n_slabs, slab_stride, N, bias, rows, N, y, N, s);
}
// dense case (the TP reduce input): float4 per thread, four slabs per trip with independent loads
__global__ void __launch_bounds__(256) slab_sum_dense_kernel(const float4* __restrict__ in, int n_slabs, int64_t slab_stride4, int64_t total4,
                                                             float4* __restrict__ y) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total4) return;
    float4 v = in[i];
    for (int sl0 = 1; sl0 < n_slabs; sl0 += 4) {
        float4 t[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) t[u] = in[i + (int64_t)min(sl0 + u, n_slabs - 1) * slab_stride4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (sl0 + u < n_slabs) { v.x += t[u].x; v.y += t[u].y; v.z += t[u].z; v.w += t[u].w; }
    }
    y[i] = v;
}
hipError_t launch_slab_sum_ld(const float* in, int n_slabs, int64_t slab_stride, int64_t ld_in, const float* bias,
                              int rows, int N, float* y, int64_t ld_out, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    if (!bias && ld_in == N && ld_out == N && N % 4 == 0 && slab_stride % 4 == 0) {
        const int64_t total4 = (int64_t)rows * N / 4;
        slab_sum_dense_kernel<<<(unsigned)((total4 + 255) / 256), 256, 0, s>>>(reinterpret_cast<const float4*>(in), n_slabs, slab_stride / 4, total4,
                                                                                reinterpret_cast<float4*>(y));
        return hipGetLastError();
    }
    slab_sum_kernel<<<grid_for((int64_t)rows * N), 256, 0, s>>>(in, n_slabs, slab_stride, ld_in, bias, rows, N, y, ld_out);
    return hipGetLastError();
}

// ---- generic-shape fallbacks for the fine-seam ops (any n; the step path never uses them) -------------
__global__ void __launch_bounds__(256) rmsnorm_generic_kernel(const float* __restrict__ x, const float* __restrict__ res,
                                                              const float* __restrict__ w, float eps, int n,
                                                              float* __restrict__ y, float* __restrict__ res_out) {
    __shared__ float red[4];
    const size_t base = (size_t)blockIdx.x * n;
    float ss = 0.f;
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float s = res ? x[base + i] + res[base + i] : x[base + i];
        ss += s * s;
    }
    ss = wave_sum(ss);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = ss;
    __syncthreads();
    ss = red[0] + red[1] + red[2] + red[3];
    const float rinv = 1.0f / sqrtf(ss / (float)n + eps);
    for (int i = threadIdx.x; i < n; i += blockDim.x) {
        const float s = res ? x[base + i] + res[base + i] : x[base + i];
        if (res_out) res_out[base + i] = s;
        y[base + i] = (s * rinv) * w[i];
    }
}
hipError_t launch_rmsnorm_generic(const float* x, const float* res, const float* w, float eps, int rows, int n, float* y,
                                  float* res_out, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    rmsnorm_generic_kernel<<<rows, 256, 0, s>>>(x, res, w, eps, n, y, res_out);
    return hipGetLastError();
}
__global__ void __launch_bounds__(256) silu_mul_generic_kernel(const float* __restrict__ x, int64_t total, int n,
                                                               float* __restrict__ y) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / n;
        const int c = (int)(i - r * n);
        const float g = x[r * 2 * n + c], u = x[r * 2 * n + n + c];
        y[i] = (g / (1.0f + __expf(-g))) * u;
    }
}
hipError_t launch_silu_mul_generic(const float* x, int rows, int n, float* y, hipStream_t s) {
    const int64_t total = (int64_t)rows * n;
    if (total <= 0) return hipSuccess;
    silu_mul_generic_kernel<<<grid_for(total), 256, 0, s>>>(x, total, n, y);
    return hipGetLastError();
}
// x f32 [rows][K] -> hi/lo bf16 [rows][Kpad] (zero beyond K)
__global__ void __launch_bounds__(256) split_hilo_pad_kernel(const float* __restrict__ x, int K, int Kpad, int64_t total,
                                                             uint16_t* __restrict__ hi, uint16_t* __restrict__ lo) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t r = i / Kpad;
        const int c = (int)(i - r * Kpad);
        uint16_t h = 0, l = 0;
        if (c < K) split_bf16(x[r * K + c], h, l);
        hi[i] = h;
        lo[i] = l;
    }
}
hipError_t launch_split_hilo_pad(const float* x, int rows, int K, int Kpad, bf16_bits* hi, bf16_bits* lo, hipStream_t s) {
    const int64_t total = (int64_t)rows * Kpad;
    if (total <= 0) return hipSuccess;
    split_hilo_pad_kernel<<<grid_for(total), 256, 0, s>>>(x, K, Kpad, total, hi, lo);
    return hipGetLastError();
}

// argmax, LAST maximal element wins (Iterator::max_by, llm_engine.rs:135-142; tests/layer_test.rs:144-149)
__global__ void __launch_bounds__(1024) argmax_kernel(const float* __restrict__ logits, int V, int64_t ld,
                                                      uint32_t* __restrict__ ids, float* __restrict__ maxval) {
    __shared__ float sv[16];
    __shared__ int si[16];
    const float* p = logits + (size_t)blockIdx.x * ld;
    float bv = -INFINITY;
    int bi = -1;
    auto take = [&](int i, float v) { if (v >= bv || bi < 0) { bv = v; bi = i; } };  // i increases per thread: >= keeps the last
    // eight loads at a time, independent of each other: one per trip was a round trip each, 16 rows of 32768 14.4 us, now 6.9
    int i = threadIdx.x;
    for (; i + 7 * (int)blockDim.x < V; i += 8 * blockDim.x) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = p[i + u * blockDim.x];
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < 8; ++u) take(i + u * blockDim.x, v[u]);
    }
    for (; i < V; i += blockDim.x) take(i, p[i]);
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o);
        const int oi = __shfl_xor(bi, o);
        if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi > bi))) { bv = ov; bi = oi; }
    }
    if ((threadIdx.x & 63) == 0) { sv[threadIdx.x >> 6] = bv; si[threadIdx.x >> 6] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w)
            if (si[w] >= 0 && (bi < 0 || sv[w] > bv || (sv[w] == bv && si[w] > bi))) { bv = sv[w]; bi = si[w]; }
        ids[blockIdx.x] = (uint32_t)(bi < 0 ? 0 : bi);
        if (maxval) maxval[blockIdx.x] = bv;
    }
}
hipError_t launch_argmax(const float* logits, int rows, int V, int64_t ld, uint32_t* ids, float* maxval,
                         hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    argmax_kernel<<<rows, 1024, 0, s>>>(logits, V, ld, ids, maxval);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------------------------------
// Temperature sampling on the device: Qwen3ModelRunner::sample_token (src/engine/llm_engine.rs:97-133).
//   t = max(temperature, 1e-6); weights w_i = exp((l_i - max l) / t); categorical draw over w; when the weights do not
//   form a distribution (sum not finite or not positive) the reference falls back to argmax (last max, :135-142).
// The draw uses the Gumbel-max form, id = argmax_i (l_i / t + g_i) with g_i = -log(-log(u_i)), which samples exactly
// softmax(l / t) and needs no prefix sums; u_i comes from a counter RNG keyed by (seed, sequence id, position, i), so a
// run is reproducible and independent of batch composition (the reference draws from an unseeded thread RNG).
// Ties go to the higher index, like the arg-max.  One workgroup per row.
// ---------------------------------------------------------------------------------------------------
__host__ __device__ inline float sample_u01(uint64_t key, uint32_t i) {
    const uint64_t x = synth_finalize(key + ((uint64_t)i + 1) * 0x9E3779B97F4A7C15ULL);
    return ((float)(x >> 40) + 0.5f) * 5.9604644775390625e-08f;  // (0, 1): 24 random bits
}
__global__ void __launch_bounds__(1024) sample_rows_kernel(const float* __restrict__ logits, int V, int64_t ld, const float* __restrict__ temps,
                                                           const uint64_t* __restrict__ keys, int idx_offset, uint32_t* __restrict__ ids,
                                                           float* __restrict__ best_score) {
    __shared__ float sv[16];
    __shared__ int si[16];
    __shared__ float s_max, s_sum;
    const float* p = logits + (size_t)blockIdx.x * ld;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const float t = fmaxf(temps[blockIdx.x], 1e-6f);
    // pass 1: max and sum of exp((l - max) / t): does the row form a distribution?
    float mx = -INFINITY;
    bool nan = false;
    for (int i = threadIdx.x; i < V; i += blockDim.x) { const float v = p[i]; nan |= v != v; mx = fmaxf(mx, v); }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o));
    if (lane == 0) sv[wv] = mx;
    __syncthreads();
    if (threadIdx.x == 0) { float m = sv[0]; for (int w = 1; w < nw; ++w) m = fmaxf(m, sv[w]); s_max = m; }
    __syncthreads();
    mx = s_max;
    float sum = 0.f;
    for (int i = threadIdx.x; i < V; i += blockDim.x) sum += expf((p[i] - mx) / t);
    sum = wave_sum(sum);
    __syncthreads();
    if (lane == 0) sv[wv] = nan ? NAN : sum;
    __syncthreads();
    if (threadIdx.x == 0) { float s = 0.f; for (int w = 0; w < nw; ++w) s += sv[w]; s_sum = s; }
    __syncthreads();
    const bool degenerate = !(s_sum > 0.f) || !(s_sum < INFINITY);
    // pass 2: arg-max of the Gumbel-perturbed scores (plain logits for a degenerate row): LAST max wins
    const uint64_t key = keys[blockIdx.x];
    float bv = -INFINITY;
    int bi = -1;
    for (int i = threadIdx.x; i < V; i += blockDim.x) {
        float v = p[i];
        if (v != v) v = -INFINITY;  // a NaN logit ranks below every number
        if (!degenerate) v = v / t - logf(-logf(sample_u01(key, (uint32_t)(i + idx_offset))));
        if (v >= bv || bi < 0) { bv = v; bi = i; }  // i increases per thread: >= keeps the last
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o);
        const int oi = __shfl_xor(bi, o);
        if (oi >= 0 && (bi < 0 || ov > bv || (ov == bv && oi > bi))) { bv = ov; bi = oi; }
    }
    __syncthreads();
    if (lane == 0) { sv[wv] = bv; si[wv] = bi; }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < nw; ++w)
            if (si[w] >= 0 && (bi < 0 || sv[w] > bv || (sv[w] == bv && si[w] > bi))) { bv = sv[w]; bi = si[w]; }
        ids[blockIdx.x] = (uint32_t)(bi < 0 ? 0 : bi);
        if (best_score) best_score[blockIdx.x] = bv;
    }
}
hipError_t launch_sample_rows(const float* logits, int rows, int V, int64_t ld, const float* temps, const uint64_t* keys, int idx_offset,
                              uint32_t* ids, float* best_score, hipStream_t s) {
    if (rows <= 0) return hipSuccess;
    sample_rows_kernel<<<rows, 1024, 0, s>>>(logits, V, ld, temps, keys, idx_offset, ids, best_score);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) embedding_f32_kernel(const float* __restrict__ table,
                                                            const uint32_t* __restrict__ ids, int V, int H,
                                                            float* __restrict__ y) {
    const uint32_t id = ids[blockIdx.x];
    for (int i = threadIdx.x; i < H; i += blockDim.x)
        y[(size_t)blockIdx.x * H + i] = id < (uint32_t)V ? table[(size_t)id * H + i] : 0.f;
}
hipError_t launch_embedding_f32(const float* table, const uint32_t* ids, int n, int V, int H, float* y,
                                hipStream_t s) {
    if (n <= 0) return hipSuccess;
    embedding_f32_kernel<<<n, 256, 0, s>>>(table, ids, V, H, y);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) rope_bhtd_kernel(float* __restrict__ x, int T, int hd,
                                                        const float* __restrict__ cosv, const float* __restrict__ sinv,
                                                        int64_t total_pairs) {
    const int half = hd >> 1;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total_pairs; i += (int64_t)gridDim.x * blockDim.x) {
        const int j = (int)(i % half);
        const int64_t vec = i / half;  // (b*heads + h)*T + t
        const int t = (int)(vec % T);
        float* v = x + vec * hd;
        const float c = cosv[(size_t)t * half + j], s = sinv[(size_t)t * half + j];
        const float x1 = v[j], x2 = v[j + half];
        v[j] = x1 * c - x2 * s;
        v[j + half] = x2 * c + x1 * s;
    }
}
hipError_t launch_rope_bhtd(float* x, int B, int heads, int T, int hd, const float* cos, const float* sin,
                            hipStream_t s) {
    const int64_t total = (int64_t)B * heads * T * (hd / 2);
    if (total <= 0) return hipSuccess;
    rope_bhtd_kernel<<<grid_for(total), 256, 0, s>>>(x, T, hd, cos, sin, total);
    return hipGetLastError();
}

__global__ void __launch_bounds__(256) bhtd_to_rows_kernel(const float* __restrict__ x, int B, int heads, int T, int hd,
                                                           float scale, float* __restrict__ y) {
    const int64_t total = (int64_t)B * heads * T * hd;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total; i += (int64_t)gridDim.x * blockDim.x) {
        const int d = (int)(i % hd);
        int64_t r = i / hd;
        const int t = (int)(r % T); r /= T;
        const int h = (int)(r % heads);
        const int b = (int)(r / heads);
        y[((size_t)(b * T + t) * heads + h) * hd + d] = x[i] * scale;
    }
}
hipError_t launch_bhtd_to_rows(const float* x, int B, int heads, int T, int hd, float scale, float* y,
                               hipStream_t s) {
    const int64_t total = (int64_t)B * heads * T * hd;
    if (total <= 0) return hipSuccess;
    bhtd_to_rows_kernel<<<grid_for(total), 256, 0, s>>>(x, B, heads, T, hd, scale, y);
    return hipGetLastError();
}

__global__ void advance_decode_kernel(uint32_t* ids, const uint32_t* next, int* pos, int n, DecodeRow* rows, const int* block_tables, int max_blocks) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) { ids[i] = next[i]; pos[i] += 1; }
    const int r = i / kDecodeRowInts, e = i % kDecodeRowInts;  // a record's ints are neighbouring lanes of one wave
    if (rows && r < n) {
        const int p = __shfl(e == 2 ? rows[r].pos + 1 : 0, 2, kDecodeRowInts);  // read by the lane that writes it
        const int* table = block_tables + (size_t)rows[r].slot * max_blocks;
        int* const d = reinterpret_cast<int*>(rows + r);
        if (e == 2) d[e] = p;
        else if (e == 3) d[e] = table[p >> 8];
        else if (e > 3 && e - 4 < max_blocks) d[e] = table[e - 4];
    }
}
// ---------------------------------------------------------------------------------------------------
// Cache warmer: touch a list of byte ranges so they sit in the Infinity Cache (MALL) when the consumer
// kernel arrives.  Runs on a side stream while latency-bound kernels leave HBM idle.  ranges[i] = {ptr, bytes}.
// ---------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) prefetch_ranges_kernel(const PrefetchRange* __restrict__ ranges, int n_ranges,
                                                              unsigned* __restrict__ sink) {
    unsigned acc = 0;
    for (int r = blockIdx.y; r < n_ranges; r += gridDim.y) {
        const uint4* p = reinterpret_cast<const uint4*>(ranges[r].ptr);
        const size_t n16 = ranges[r].bytes >> 4;
        // one 16-byte load per 128-byte line is enough to pull the line in; consecutive lanes take consecutive lines
        for (size_t i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * 8; i < n16; i += (size_t)gridDim.x * blockDim.x * 8) {
            const uint4 v = p[i];
            acc ^= v.x;
        }
    }
    if (acc == 0x9e3779b9u && sink) *sink = acc;  // never true in practice; keeps the loads alive
}
hipError_t launch_prefetch_ranges(const PrefetchRange* d_ranges, int n_ranges, unsigned* sink, int blocks_x, hipStream_t s) {
    if (n_ranges <= 0) return hipSuccess;
    dim3 grid(std::max(1, blocks_x), std::min(n_ranges, 64));
    prefetch_ranges_kernel<<<grid, 256, 0, s>>>(d_ranges, n_ranges, sink);
    return hipGetLastError();
}

// which XCD (accelerator complex die) each workgroup of a grid lands on: out[linear workgroup id] = XCC_ID
__global__ void xcc_map_kernel(int* out) {
    unsigned x;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
    if (threadIdx.x == 0) out[blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z)] = (int)(x & 15u);
}
hipError_t launch_xcc_map(int gx, int gy, int gz, int threads, int* out, hipStream_t s) {
    xcc_map_kernel<<<dim3(gx, gy, gz), threads, 0, s>>>(out);
    return hipGetLastError();
}

// Metadata of a chunk of rows, read from pinned host memory and spread over its device arrays by one launch.  Bound by the host
// link's latency: one or two dependent reads of it per workgroup, whatever the number of arrays.  As copies, ten per chunk, each was
// a launch of its own in front of the first kernel of the step.  Measured: one decode step of one sequence of Qwen3-0.6B 1071 -> 1033
// us, of 24 sequences of four 8B layers 1107 -> 1050 us.
__global__ void __launch_bounds__(256) stage_kernel(StageArgs a) {
    const StageRun r = a.run[blockIdx.y];
    const int i0 = blockIdx.x * 256 + threadIdx.x, step = gridDim.x * 256;
    if (r.pairs) {
        const int2* s = reinterpret_cast<const int2*>(a.src + r.src);
        for (int i = i0; i < r.n; i += step) { const int2 v = s[i]; r.dst[v.x] = v.y; }
        return;
    }
    const int n4 = (reinterpret_cast<uintptr_t>(r.dst) & 15) == 0 ? r.n >> 2 : 0;  // parts of an array may start anywhere
    const int4* s = reinterpret_cast<const int4*>(a.src + r.src);
    for (int i = i0; i < n4; i += step) reinterpret_cast<int4*>(r.dst)[i] = s[i];
    for (int i = 4 * n4 + i0; i < r.n; i += step) r.dst[i] = a.src[r.src + i];
}
hipError_t launch_stage(const StageArgs& a, int n_runs, int longest, hipStream_t s) {
    if (n_runs <= 0) return hipSuccess;
    if (n_runs > kStageRuns) return hipErrorInvalidValue;
    stage_kernel<<<dim3(std::min(16, (longest + 1023) / 1024), n_runs), 256, 0, s>>>(a);
    return hipGetLastError();
}

// Bound by the link: 1 MB in 22.5 us by 16 to 64 workgroups, 25 by 128 (28 with the fence in every wave; the wait for its own stores costs nothing, 22.4 with and without); the runtime's copy takes 19, but with the event that tells the host
// of it, where here the flag behind the data does, it is 17 us away from the next one.
__global__ void __launch_bounds__(512) copy_out_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, size_t bytes, unsigned* done, uint32_t* flag, uint32_t seq) {
    const size_t n16 = bytes / 16;
    for (size_t i = (size_t)blockIdx.x * 512 + threadIdx.x; i < n16; i += (size_t)gridDim.x * 512) dst[i] = src[i];
    if (blockIdx.x == 0 && threadIdx.x < bytes % 16 / 4) reinterpret_cast<uint32_t*>(dst + n16)[threadIdx.x] = reinterpret_cast<const uint32_t*>(src + n16)[threadIdx.x];
    // Every wave for its own stores: a barrier waits for nobody's here, a fence for those of its own wave.  Then the write-back of one is the workgroup's.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (threadIdx.x) return;
    __threadfence_system();  // all that the workgroup wrote is in the host's memory before it counts
    if (__hip_atomic_fetch_add(done, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1) {
        __hip_atomic_store(done, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // the next copy into this slot comes behind this one on its stream
        __threadfence_system();
        __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}
hipError_t launch_copy_out(const void* src, void* dst, size_t bytes, unsigned* done, uint32_t* flag, uint32_t seq, hipStream_t s) {
    if (bytes % 4 || ((uintptr_t)src | (uintptr_t)dst) % 16) return hipErrorInvalidValue;
    const int groups = (int)std::max<size_t>(1, std::min<size_t>(32, bytes / (512 * 16)));
    copy_out_kernel<<<groups, 512, 0, s>>>(reinterpret_cast<const uint4*>(src), reinterpret_cast<uint4*>(dst), bytes, done, flag, seq);
    return hipGetLastError();
}

hipError_t launch_advance_decode(uint32_t* ids, const uint32_t* next, int* pos, int n, DecodeRow* rows, const int* block_tables, int max_blocks, hipStream_t s) {
    if (n <= 0) return hipSuccess;
    static_assert(256 % kDecodeRowInts == 0 && 64 % kDecodeRowInts == 0, "");
    advance_decode_kernel<<<((rows ? n * kDecodeRowInts : n) + 255) / 256, 256, 0, s>>>(ids, next, pos, n, rows, block_tables, max_blocks);
    return hipGetLastError();
}

}  // namespace nvllm
