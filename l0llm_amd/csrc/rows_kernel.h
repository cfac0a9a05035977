// Several activation rows (1 .. 64) through a weight matrix, the weights read once: prompts shorter
// than the MFMA GEMM's tiles, and every multi-row call of the GEMV entry points with fp32 rows.
// Replaces GemvQ8.ExecuteRows / Gemv.ExecuteRows (call sites LlmMatrix.cs:149-171) for int8, fp16
// and bf16 [N, K] weights.
//
// Both operands keep all of their bits. An fp32 activation is cut into three bf16 values of 8
// significant bits each (x = x0 + x1 + x2 exactly), an int8 or bf16 weight is one bf16 value, an fp16
// weight two (8 + 3 bits), and v_mfma_f32_16x16x32_bf16 multiplies every pair of parts (products of
// bf16 values are exact in fp32) into one fp32 accumulator: 3 MFMAs per 16 x 16 x 32 tile, 6 for fp16
// weights.
//
// Work: a block owns 16 * CF weight rows (output columns) and all of K; wave w of its NW takes the K
// steps w, w + NW, ... of 64 values, so a block's waves stream neighbouring bytes of the same rows.
// A wave works alone until the end, one to two steps ahead of itself: it loads whole 64- or 128-byte
// pieces of the weight rows and whole 256-byte pieces of the activation rows, and turns both into the
// MFMA's operand order through its own LDS (16-byte chunks, slots exchanged by XOR so that neither the
// writes nor the reads conflict). Loading the weights in operand order instead, where adjacent lanes
// hold different rows, makes the address unit split every load into 64 requests: bf16 13 rows
// 2048 -> 16384 took 17.8 us that way, 15.5 us through LDS. All loads are buffer loads: a lane past
// the last row, past K or past the last step gets zeros and reads nothing, so the loads stay
// unconditional and the loop waits for exactly the step it needs. No barrier until the waves' partial
// tiles are summed, in wave order, through LDS.
//
// What bounds it: with few rows the weight stream (bf16 13 rows 2048 -> 16384: 67 MB in 15.5 us
// with the launch, 4.3 TB/s); with int8 weights or more rows the vector instructions that turn weights
// and activations into bf16 parts (int8 13 rows 4096 -> 14336: 293 a step of 64 x 64 weights and 16
// rows, 6.8 of 20 us; 24 MFMAs take 2.2).
#pragma once

#include "gemv_kernel.h"

namespace l0h {
namespace {

typedef __attribute__((ext_vector_type(8))) __bf16 rows_bf16x8;
typedef __attribute__((ext_vector_type(4))) float rows_f32x4;

constexpr int kRowsStep = 64;        // K values per step
constexpr int kRowsMax = kGemvRowsMax;
constexpr int kRowsMaxK = 1 << 22;   // 64 rows of it stay under the 2 GiB of a buffer

__device__ __forceinline__ rows_f32x4 rows_mfma(const uint4& a, const uint4& b, rows_f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(rows_bf16x8, a), __builtin_bit_cast(rows_bf16x8, b), c, 0,
                                                   0, 0);
}

// The upper halves of two fp32 values: two bf16 values, truncated.
__device__ __forceinline__ uint32_t upper_pair(float lo, float hi) {
    return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

// v minus its bf16 truncation, exact (NaN where v is infinite or NaN).
__device__ __forceinline__ float bf16_rest(float v) { return v - __uint_as_float(__float_as_uint(v) & 0xffff0000u); }

// 8 fp32 values as three bf16 parts: a = part[0] + part[1] + part[2].
__device__ __forceinline__ void split3(const float (&v)[8], uint4 (&part)[3]) {
    float r[8], q[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        r[e] = bf16_rest(v[e]);
        q[e] = bf16_rest(r[e]);
    }
    part[0] = make_uint4(upper_pair(v[0], v[1]), upper_pair(v[2], v[3]), upper_pair(v[4], v[5]), upper_pair(v[6], v[7]));
    part[1] = make_uint4(upper_pair(r[0], r[1]), upper_pair(r[2], r[3]), upper_pair(r[4], r[5]), upper_pair(r[6], r[7]));
    part[2] = make_uint4(upper_pair(q[0], q[1]), upper_pair(q[2], q[3]), upper_pair(q[4], q[5]), upper_pair(q[6], q[7]));
}

// The lane's 16-byte loads of one weight row in a step: its 16 int8 values, or two groups of 8
// 16-bit values 32 apart.
template <int WT>
constexpr int kRowsLoads = WT == L0H_I8PC ? 1 : 2;

// The 8 weights a lane feeds to the MFMAs of substep t (of 2), as one or two bf16 parts.
template <int WT>
__device__ __forceinline__ void weight_parts(const uint4 (&w)[kRowsLoads<WT>], int t, uint4 (&part)[2]) {
    if constexpr (WT == L0H_I8PC) {
        const uint32_t d[2] = {t ? w[0].z : w[0].x, t ? w[0].w : w[0].y};
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const float f0 = (float)(int8_t)d[j], f1 = (float)(int8_t)(d[j] >> 8), f2 = (float)(int8_t)(d[j] >> 16),
                        f3 = (float)((int32_t)d[j] >> 24);
            o[2 * j] = upper_pair(f0, f1);
            o[2 * j + 1] = upper_pair(f2, f3);
        }
        part[0] = make_uint4(o[0], o[1], o[2], o[3]);
    } else if constexpr (WT == L0H_BF16) {
        part[0] = w[t];
    } else {
        const uint32_t d[4] = {w[t].x, w[t].y, w[t].z, w[t].w};
        uint32_t hi[4], lo[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float2 f = __half22float2(__builtin_bit_cast(__half2, d[j]));
            hi[j] = upper_pair(f.x, f.y);
            lo[j] = upper_pair(bf16_rest(f.x), bf16_rest(f.y));
        }
        part[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
        part[1] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
    }
}

// Row m of the call in the fused q|k|v epilogue (qkv_pair_with on that row's q vector).
__device__ __forceinline__ void qkv_row_pair(const GemvParams& p, int m, int row, float v0, float v1, int pos) {
    GemvParams q = p;
    q.q_out = p.q_out + (size_t)m * p.q_dim;
    qkv_pair_with(q, row, v0, v1, pos, [&](int i, float& cs, float& sn) {
        float sv, cv;
        sincosf((float)pos * p.inv_freq[i], &sv, &cv);
        cs = cv * p.rope_scale;
        sn = sv * p.rope_scale;
    });
}

// Output (m, n) of the call before its row scale, by the whole wave in fp32.
template <int WT, bool NORM>
__device__ float whole_dot(const GemvParams& p, int m, int n, int lane) {
    float acc = 0.f;
    for (int k = lane; k < p.k; k += 64) {
        const size_t at = (size_t)n * p.k + k;
        const float w = WT == L0H_I8PC ? (float)static_cast<const int8_t*>(p.w)[at] : load_act(p.w, WT, at);
        float x = static_cast<const float*>(p.x)[(size_t)m * p.k + k];
        if constexpr (NORM) x *= p.norm_w[k];
        acc = fmaf(w, x, acc);
    }
    return wave_sum(acc);
}

// LDS bytes of one wave: a step's activations (4 KiB per 16 rows), before them its weights, at the end
// its partial tile.
template <int WT, int MF, int CF>
constexpr int rows_wave_lds() {
    return 1024 * (MF * 4 > CF * kRowsLoads<WT> ? MF * 4 : CF * kRowsLoads<WT>);
}

// A buffer of `bytes` at `base`, wave-uniform; a load at or past its end returns zeros and reads nothing.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_buffer(const void* base, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, (int)bytes, 0x00020000);
}

template <int AUX>
__device__ __forceinline__ uint4 rows_load16(__amdgpu_buffer_rsrc_t b, uint32_t at) {
    const u32x4_t v = __builtin_amdgcn_raw_buffer_load_b128(b, (int)at, 0, AUX);
    return make_uint4(v.x, v.y, v.z, v.w);
}

constexpr uint32_t kRowsOutside = 0x80000000u;  // past the end of every buffer (K <= kRowsMaxK)

// MF row groups of 16 activation rows, CF groups of 16 weight rows, NW waves; DW steps of weights and
// DX of activations in flight a wave. NORM: the activations are RMSNorm(x) * norm_w (x * norm_w enters
// the products, the row's 1 / rms multiplies the sums). EPI: EPI_STORE (store or residual, chosen at
// run time), EPI_SWIGLU or EPI_QKV (row m of the call is position pos0 + m).
template <int WT, int MF, int CF, int NW, int DW, int DX, bool NORM, int EPI>
__global__ __launch_bounds__(NW * 64) void gemv_rows_kernel(const GemvParams p, int pos0) {
    static_assert(DW % DX == 0, "the loop is unrolled over the weight slots");
    constexpr int LD = kRowsLoads<WT>;
    constexpr int CH = CF * 4;  // groups of 4 output columns per block
    constexpr int NT = 2;       // aux bit of a load that is not kept in the caches
    extern __shared__ float4 rows_smem[];
    __shared__ float ssq[NORM ? NW : 1][NORM ? MF * 16 : 1];
    const int K = p.k, N = p.n, M = p.m;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r16 = lane & 15, g = lane >> 4;
    const int n0 = blockIdx.x * (16 * CF);
    const int nsteps = (K + kRowsStep - 1) / kRowsStep;
    constexpr int kWave = rows_wave_lds<WT, MF, CF>() / 16;
    float4* st = rows_smem + (size_t)wave * kWave;
    const uint32_t row_bytes = (uint32_t)K * WTraits<WT>::kBytes;
    // The block's weight rows and the activation rows: rows past N or M read as zeros.
    const auto wbuf = rows_buffer(static_cast<const char*>(p.w) + (size_t)n0 * row_bytes, (size_t)min(16 * CF, N - n0) * row_bytes);
    const auto xbuf = rows_buffer(p.x, (size_t)M * K * 4);
    const auto nbuf = rows_buffer(NORM ? p.norm_w : p.x, (size_t)K * 4);

    // The wave's own LDS: its writes and reads stay in program order.
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    auto load_x = [&](uint4 (&v)[MF][4], uint4& nw, int s) {
        const uint32_t k = (uint32_t)s * kRowsStep + r16 * 4;
        const bool in = k < (uint32_t)K;
        if constexpr (NORM) nw = rows_load16<0>(nbuf, in ? k * 4 : kRowsOutside);
#pragma unroll
        for (int f = 0; f < MF; f++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                v[f][i] = rows_load16<0>(xbuf, in ? ((uint32_t)(f * 16 + i * 4 + g) * K + k) * 4 : kRowsOutside);
    };
    // A step of a weight row is LD * 64 bytes: 4 * LD adjacent lanes read them, 16 / LD rows a load.
    constexpr int WL = 4 * LD;
    const int wr = lane / WL, wc = lane % WL;
    auto load_w = [&](uint4 (&w)[CF][LD], int s) {
        const uint32_t b = (uint32_t)s * (kRowsStep * WTraits<WT>::kBytes) + wc * 16;
        const uint32_t at = b < row_bytes ? wr * row_bytes + b : kRowsOutside;
#pragma unroll
        for (int c = 0; c < CF; c++)
#pragma unroll
            for (int l = 0; l < LD; l++) w[c][l] = rows_load16<NT>(wbuf, at + (c * 16 + l * (16 / LD)) * row_bytes);
    };
    // ... and come back through LDS as the A operand wants them: row r16, chunk 4 t + g. Chunk c of row
    // r sits in slot c ^ (r / (4 / LD)) of its row.
    auto swap_w = [&](const uint4 (&w)[CF][LD], uint4 (&o)[CF][LD]) {
        uint4* sw = reinterpret_cast<uint4*>(st);
#pragma unroll
        for (int c = 0; c < CF; c++)
#pragma unroll
            for (int l = 0; l < LD; l++) {
                const int row = wr + l * (16 / LD);
                sw[(c * 16 + row) * WL + (wc ^ (LD == 1 ? row >> 2 : row & 7))] = w[c][l];
            }
        wave_sync();
#pragma unroll
        for (int c = 0; c < CF; c++)
#pragma unroll
            for (int l = 0; l < LD; l++)
                o[c][l] = sw[(c * 16 + r16) * WL + ((l * 4 + g) ^ (LD == 1 ? r16 >> 2 : r16 & 7))];
    };

    rows_f32x4 acc[MF][CF];
#pragma unroll
    for (int f = 0; f < MF; f++)
#pragma unroll
        for (int c = 0; c < CF; c++) acc[f][c] = rows_f32x4{0.f, 0.f, 0.f, 0.f};
    float ss[NORM ? MF : 1][4] = {};

    auto stage = [&](const uint4 (&v)[MF][4], const uint4& nw) {
#pragma unroll
        for (int f = 0; f < MF; f++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                float4 t = __builtin_bit_cast(float4, v[f][i]);
                if constexpr (NORM) {
                    ss[f][i] += (t.x * t.x + t.y * t.y) + (t.z * t.z + t.w * t.w);
                    t.x *= __uint_as_float(nw.x);
                    t.y *= __uint_as_float(nw.y);
                    t.z *= __uint_as_float(nw.z);
                    t.w *= __uint_as_float(nw.w);
                }
                const int row = i * 4 + g;
                st[(f * 16 + row) * 16 + (r16 ^ row)] = t;
            }
    };
    // One step's products start from zero, the small parts first, and join the running sum with one
    // rounding: a chain of MFMAs through the running sum rounds it once per part.
    auto compute = [&](const uint4 (&wp)[2][CF][2]) {
#pragma unroll
        for (int f = 0; f < MF; f++) {
            uint4 xp[2][3];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int c0 = WT == L0H_I8PC ? g * 4 + t * 2 : t * 8 + g * 2;
                const float4 a = st[(f * 16 + r16) * 16 + (c0 ^ r16)], b = st[(f * 16 + r16) * 16 + ((c0 + 1) ^ r16)];
                const float v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
                split3(v, xp[t]);
            }
            rows_f32x4 sum[CF];
#pragma unroll
            for (int c = 0; c < CF; c++) sum[c] = rows_f32x4{0.f, 0.f, 0.f, 0.f};
            auto add = [&](int q, int part) {
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int c = 0; c < CF; c++) sum[c] = rows_mfma(wp[t][c][part], xp[t][q], sum[c]);
            };
            if constexpr (WT == L0H_F16) {
                add(2, 1);
                add(1, 1);
            }
            add(2, 0);
            if constexpr (WT == L0H_F16) add(0, 1);
            add(1, 0);
            add(0, 0);
#pragma unroll
            for (int c = 0; c < CF; c++) acc[f][c] += sum[c];
        }
    };

    uint4 xv[DX][MF][4], nw[DX];
    uint4 wv[DW][CF][LD];
#pragma unroll
    for (int d = 0; d < DW; d++) {
        if (d < DX) load_x(xv[d], nw[d], wave + d * NW);
        load_w(wv[d], wave + d * NW);
    }
    for (int s0 = wave;; s0 += DW * NW) {
        bool more = true;
#pragma unroll
        for (int d = 0; d < DW; d++) {
            const int s = s0 + d * NW;
            if (s >= nsteps) {
                more = false;
                break;
            }
            wave_sync();
            uint4 wo[CF][LD];
            swap_w(wv[d], wo);
            load_w(wv[d], s + DW * NW);
            wave_sync();
            stage(xv[d % DX], nw[d % DX]);
            load_x(xv[d % DX], nw[d % DX], s + DX * NW);
            // The next loads go out before this step's products: left alone, the scheduler moves the
            // weight conversion, and with it the wait for the weights, ahead of them.
            __builtin_amdgcn_sched_barrier(0);
            uint4 wp[2][CF][2];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int c = 0; c < CF; c++) weight_parts<WT>(wo[c], t, wp[t][c]);
            wave_sync();
            compute(wp);
        }
        if (!more) break;
    }

    // ---- the waves' tiles, summed in wave order: column group ch of row m in slot ch ^ (m % CH) ----
    wave_sync();
#pragma unroll
    for (int f = 0; f < MF; f++)
#pragma unroll
        for (int c = 0; c < CF; c++)
            st[(f * 16 + r16) * CH + ((c * 4 + g) ^ (r16 & (CH - 1)))] =
                make_float4(acc[f][c][0], acc[f][c][1], acc[f][c][2], acc[f][c][3]);
    if constexpr (NORM) {
#pragma unroll
        for (int f = 0; f < MF; f++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float q = lane_group_sum<16>(ss[f][i]);
                if (r16 == 0) ssq[wave][f * 16 + i * 4 + g] = q;
            }
    }
    lds_barrier();
    for (int i = tid; i < MF * 16 * CH; i += NW * 64) {
        const int m = i / CH, ch = i % CH;
        const int n = n0 + ch * 4;
        const bool live = m < M && n < N;
        float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; w++) {
            const float4 t = rows_smem[(size_t)w * kWave + m * CH + (ch ^ (m & (CH - 1)))];
            v[0] += t.x;
            v[1] += t.y;
            v[2] += t.z;
            v[3] += t.w;
        }
        // An infinite operand has no parts that sum to it (infinity times a part of zero, infinity minus
        // infinity): a NaN is worked out again from the whole values, one output at a time.
#pragma unroll
        for (int e = 0; e < 4; e++)
            for (uint64_t bad = __ballot(live && n + e < N && v[e] != v[e]); bad; bad &= bad - 1) {
                const int l = __builtin_ctzll(bad);
                const float t = whole_dot<WT, NORM>(p, __builtin_amdgcn_readlane(m, l), __builtin_amdgcn_readlane(n, l) + e, lane);
                if (lane == l) v[e] = t;
            }
        if (!live) continue;
        float scale = 1.f;
        if constexpr (NORM) {
            float t = 0.f;
#pragma unroll
            for (int w = 0; w < NW; w++) t += ssq[w][m];
            scale = rsqrtf(t / (float)K + p.eps);
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int nn = min(n + e, N - 1);
            if constexpr (NORM) v[e] *= scale;
            if constexpr (WT == L0H_I8PC) v[e] *= half_bits(p.scales[nn]);
            if (p.bias) v[e] += p.bias[nn];
        }
        if constexpr (EPI == EPI_STORE) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (n + e < N) {
                    const size_t at = (size_t)m * N + n + e;
                    if (p.epilogue == EPI_STORE)
                        store_act(p.y, p.y_dtype, at, v[e]);
                    else
                        p.resid[at] += v[e];
                }
        } else {
#pragma unroll
            for (int e = 0; e < 4; e += 2)
                if (n + e + 1 < N) {
                    if constexpr (EPI == EPI_SWIGLU)
                        store_act(p.y, p.y_dtype, ((size_t)m * N + n + e) >> 1, silu(v[e]) * v[e + 1]);
                    else
                        qkv_row_pair(p, m, n + e, v[e], v[e + 1], pos0 + m);
                }
        }
    }
}

template <int WT, int MF, int CF, int NW, int DW, int DX, bool NORM, int EPI>
int launch_rows(hipStream_t s, const GemvParams& p, int pos0) {
    constexpr int shmem = NW * rows_wave_lds<WT, MF, CF>();
    static_assert(shmem <= 160 * 1024 - NW * 256 - 256, "LDS of a CU");
    auto kern = gemv_rows_kernel<WT, MF, CF, NW, DW, DX, NORM, EPI>;
    static const hipError_t attr =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, shmem);
    if (attr != hipSuccess) return fail(L0H_ERR_DEVICE, std::string("hipFuncSetAttribute: ") + hipGetErrorString(attr));
    kern<<<ceil_div(p.n, 16 * CF), NW * 64, shmem, s>>>(p, pos0);
    return launch_status("gemv_rows");
}

// Columns per block: 64 (32 for fp16 weights, whose parts take twice the registers) where that makes
// at least half a block per CU, 32 where that makes three quarters of one, else 16.
template <int WT, int MF, bool NORM, int EPI>
int launch_rows_cols(hipStream_t s, const GemvParams& p, int pos0) {
    const unsigned cus = std::max(1, p.compute_units);
    if constexpr (WT == L0H_F16) {
        if (4 * ceil_div(p.n, 32) >= 3 * cus) return launch_rows<WT, MF, 2, 4, 2, 1, NORM, EPI>(s, p, pos0);
    } else {
        if (2 * ceil_div(p.n, 64) >= cus) return launch_rows<WT, MF, 4, MF == 4 ? 4 : 8, 2, 1, NORM, EPI>(s, p, pos0);
        if (4 * ceil_div(p.n, 32) >= 3 * cus) return launch_rows<WT, MF, 2, 8, 2, 1, NORM, EPI>(s, p, pos0);
    }
    return launch_rows<WT, MF, 1, 8, 2, 1, NORM, EPI>(s, p, pos0);
}

// Up to 64 activation rows in one launch.
template <int WT, bool NORM, int EPI>
int dispatch_rows(hipStream_t s, const GemvParams& p, int pos0) {
    switch ((p.m + 15) / 16) {
    case 1: return launch_rows_cols<WT, 1, NORM, EPI>(s, p, pos0);
    case 2: return launch_rows_cols<WT, 2, NORM, EPI>(s, p, pos0);
    case 3: return launch_rows_cols<WT, 3, NORM, EPI>(s, p, pos0);
    default: return launch_rows_cols<WT, 4, NORM, EPI>(s, p, pos0);
    }
}

// The epilogues of a model's layer: q|k|v and gate|up take the norm with them, O and down none.
template <int WT>
int dispatch_rows_wt(hipStream_t s, const GemvParams& p, int pos0) {
    if (p.epilogue == EPI_QKV) return dispatch_rows<WT, true, EPI_QKV>(s, p, pos0);
    if (p.epilogue == EPI_SWIGLU) return dispatch_rows<WT, true, EPI_SWIGLU>(s, p, pos0);
    return dispatch_rows<WT, false, EPI_STORE>(s, p, pos0);
}

}  // namespace

// Multi-row dispatch for one weight type (defined in rows_<type>.hip).
int gemv_rows_i8(hipStream_t s, const GemvParams& p, int pos0);
int gemv_rows_f16(hipStream_t s, const GemvParams& p, int pos0);
int gemv_rows_bf16(hipStream_t s, const GemvParams& p, int pos0);

}  // namespace l0h
