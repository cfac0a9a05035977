// GQA decode attention over the KV cache for gfx950 (Attention.Execute / ExecutePrefill,
// LlmDecoderLayer.cs:325-327, :369-371).
//
// Split-K over the sequence ("flash decoding"): block (kv head, split, batch) reads its slice of
// the K and V rows of one kv head once and serves all the q heads of that group from it.
// Layout: cache [batch, max_seq, n_kv * head_dim] (LlmKvCache.cs:5-8). A lane owns 8 dims of a
// row (one 16-byte fp16 load, two for fp32), head_dim / 8 lanes cover a row, so a wave
// instruction reads 64 / (head_dim / 8) positions of contiguous bytes. Each group of lanes that
// shares a position slot keeps an online softmax (running max, sum and P.V accumulator, fp32,
// log2 domain) over its positions; the slots of a block are combined at the end (lane shuffles,
// then LDS across waves) into one (max, sum, acc) partial per q head. A second small kernel
// merges the splits' partials with a log-sum-exp combine in a fixed order, so the result does
// not depend on timing. (The kernel boundary publishes the partials: a completion ticket with
// device-scope fences inside one kernel measured several microseconds slower on gfx950.)
//
// Every load is unconditional (positions past the slice are clamped to valid rows and masked in
// the softmax), the next step's K and V rows are requested before the current step is computed,
// and all control flow is wave-uniform, so the in-order memory counter only ever waits for the
// rows being computed.
#include "dpp.h"
#include "kernels.h"

#include <cmath>
#include <cstdlib>
#include <type_traits>

namespace l0h {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kGroupMax = 8;  // q heads per kv head
constexpr int kUnroll = 4;    // positions per slot per step (1 or 2 for slices that short)
constexpr int kMaxSplits = 256;

// Reduce-scatter of 16 values over a 16-lane row: on return, lane r of the row holds the sum over
// the row's 16 lanes of x[r]. Four pairings, each a DPP lane permutation that is an XOR of the
// lane index (row_mirror r ^ 15, row_half_mirror r ^ 7, quad_perm [3,2,1,0] r ^ 3, [1,0,3,2]
// r ^ 1); at each, a lane keeps the half of its values whose index bit (3, 2, 1, 0) equals its
// own lane bit and adds its partner's copy of that half. 45 VALU operations, against 64 for 16
// separate butterflies, and each score is then held by one lane instead of sixteen.
__device__ __forceinline__ float row_reduce_scatter16(const float (&x)[16], int r) {
    float y[8], z[4], w[2];
    const bool b3 = r & 8, b2 = r & 4, b1 = r & 2, b0 = r & 1;
#pragma unroll
    for (int i = 0; i < 8; i++) y[i] = (b3 ? x[i + 8] : x[i]) + dpp_src<0x140, 0xf>(b3 ? x[i] : x[i + 8]);
#pragma unroll
    for (int i = 0; i < 4; i++) z[i] = (b2 ? y[i + 4] : y[i]) + dpp_src<0x141, 0xf>(b2 ? y[i] : y[i + 4]);
#pragma unroll
    for (int i = 0; i < 2; i++) w[i] = (b1 ? z[i + 2] : z[i]) + dpp_src<0x1B, 0xf>(b1 ? z[i] : z[i + 2]);
    return (b0 ? w[1] : w[0]) + dpp_src<0xB1, 0xf>(b0 ? w[0] : w[1]);
}

template <int CT>
struct CacheRow;
template <>
struct CacheRow<L0H_F16> {
    using T = uint16_t;
    uint4 raw;
    __device__ __forceinline__ void load(const T* p) { raw = ld_nt16(p); }
    __device__ __forceinline__ void get(float* f) const {
        const uint32_t d[4] = {raw.x, raw.y, raw.z, raw.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float2 t = __half22float2(__builtin_bit_cast(__half2, d[j]));
            f[2 * j] = t.x;
            f[2 * j + 1] = t.y;
        }
    }
};
template <>
struct CacheRow<L0H_F32> {
    using T = float;
    uint4 a, b;
    __device__ __forceinline__ void load(const T* p) {
        a = ld_nt16(p);
        b = ld_nt16(p + 4);
    }
    __device__ __forceinline__ void get(float* f) const {
        f[0] = __uint_as_float(a.x); f[1] = __uint_as_float(a.y); f[2] = __uint_as_float(a.z); f[3] = __uint_as_float(a.w);
        f[4] = __uint_as_float(b.x); f[5] = __uint_as_float(b.y); f[6] = __uint_as_float(b.z); f[7] = __uint_as_float(b.w);
    }
};

// 8 consecutive activation values (fp32 or fp16) as fp32.
template <int QT>
__device__ __forceinline__ void load8(const void* base, size_t idx, float* f) {
    if constexpr (QT == L0H_F32) {
        const uint4* p = reinterpret_cast<const uint4*>(static_cast<const float*>(base) + idx);
        const uint4 a = p[0], b = p[1];
        f[0] = __uint_as_float(a.x); f[1] = __uint_as_float(a.y); f[2] = __uint_as_float(a.z); f[3] = __uint_as_float(a.w);
        f[4] = __uint_as_float(b.x); f[5] = __uint_as_float(b.y); f[6] = __uint_as_float(b.z); f[7] = __uint_as_float(b.w);
    } else {
        const uint4 a = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(base) + idx);
        const uint32_t d[4] = {a.x, a.y, a.z, a.w};
#pragma unroll
        for (int j = 0; j < 4; j++) {
            float2 t = __half22float2(__builtin_bit_cast(__half2, d[j]));
            f[2 * j] = t.x;
            f[2 * j + 1] = t.y;
        }
    }
}

// Floats per split partial: G * HD accumulators, then G maxima and G sums, padded to 16 bytes.
__host__ __device__ constexpr int partial_stride(int G, int HD) { return G * HD + ((2 * G + 3) / 4) * 4; }

// Sequence length of batch entry b, and this split's slice [lo, lo + n) of it. Slices are whole
// steps (NG * U positions) so a block's slots stay in step.
template <int NG, int U>
__device__ __forceinline__ void split_range(const AttnParams& p, int seq_len_step, int b, int split, int& lo, int& n,
                                            int& len) {
    // The device-side length is read unconditionally (from q, then ignored, when the length is a
    // launch argument; the empty asm consumes the value on both paths, so the compiler cannot sink
    // the read into a branch): a branch here would split the kernel's argument loads into more rounds.
    const bool on_device = p.seq_len_device != nullptr;
    int dev_len = *(on_device ? p.seq_len_device : static_cast<const int*>(p.q));
    asm volatile("" : "+s"(dev_len));
    len = (on_device ? dev_len + p.seq_len_add : p.seq_len) + b * seq_len_step;
    len = max(0, min(len, p.max_seq_len));
    constexpr int kStep = NG * U;
    int chunk = (len + p.splits - 1) / p.splits;
    chunk = (chunk + kStep - 1) / kStep * kStep;
    lo = split * chunk;
    n = max(0, min(len, lo + chunk) - lo);
}

// QT: q dtype, G: q heads per kv head rounded up to a power of two (heads >= p.nh / p.nkv are
// computed on clamped inputs and not written). SC: the reduce-scattered softmax where the shape
// allows it (head_dim 128, four heads per kv head). U: positions per slot per step. ST: every slice
// is at most ST steps long, 1 or 2 (the launch checks max_seq_len against the split count); 0: any.
template <int HD, int CT, int QT, int G, int U, int ST, bool SC = false>
__global__ __launch_bounds__(kBlock) void attn_split_kernel(const AttnParams p, int seq_len_step,
                                                            size_t cache_batch_stride) {
    constexpr int LPP = HD / 8;     // lanes per position
    constexpr int PPW = 64 / LPP;   // position slots per wave
    constexpr int NG = kWaves * PPW;  // position slots per block
    using T = typename CacheRow<CT>::T;
    __shared__ float s_m[kWaves][G], s_l[kWaves][G];
    __shared__ __attribute__((aligned(16))) float s_acc[kWaves][G * HD];

    const int g = blockIdx.x, split = blockIdx.y, b = blockIdx.z;
    const int gsize = p.nh / p.nkv;
    const int kv_dim = p.nkv * HD;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lg = lane % LPP;
    const int slot = wave * PPW + lane / LPP;
    int lo, n, len;
    split_range<NG, U>(p, seq_len_step, b, split, lo, n, len);

    // q: this lane's 8 dims of every head of the group, scaled by log2(e) / sqrt(HD).
    float qr[G][8];
    const float qscale = 1.4426950408889634f / sqrtf((float)HD);
#pragma unroll
    for (int h = 0; h < G; h++) {
        const int hh = min(h, gsize - 1);
        load8<QT>(p.q, (size_t)b * p.nh * HD + (size_t)(g * gsize + hh) * HD + lg * 8, qr[h]);
    }
    auto scale_q = [&] {
#pragma unroll
        for (int h = 0; h < G; h++)
#pragma unroll
            for (int d = 0; d < 8; d++) qr[h][d] *= qscale;
    };
    if constexpr (ST == 0) scale_q();
    const T* kbase = static_cast<const T*>(p.kc) + (size_t)b * cache_batch_stride + (size_t)g * HD + lg * 8;
    const T* vbase = static_cast<const T*>(p.vc) + (size_t)b * cache_batch_stride + (size_t)g * HD + lg * 8;
    // Positions past the slice read the last written row (masked in the softmax, weight exactly 0),
    // never a row of the cache that may not have been written (its bits could be Inf or NaN).
    const int last = max(len - 1, 0);

    CacheRow<CT> ka[U], va[U], kb[U], vb[U];
    auto load = [&](CacheRow<CT> (&k)[U], CacheRow<CT> (&v)[U], int step) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = min(lo + step * NG * U + u * NG + slot, last);
            k[u].load(kbase + (size_t)t * kv_dim);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int t = min(lo + step * NG * U + u * NG + slot, last);
            v[u].load(vbase + (size_t)t * kv_dim);
        }
    };

    float m[G], l[G], acc[G][8];
#pragma unroll
    for (int h = 0; h < G; h++) {
        m[h] = -INFINITY;
        l[h] = 0.f;
#pragma unroll
        for (int d = 0; d < 8; d++) acc[h][d] = 0.f;
    }
    // Four heads x four positions per slot over a 16-lane row (head_dim 128, the Llama-3 shapes):
    // the 16 partial dot products are reduce-scattered, so lane r of the row owns the score of
    // position r / 4, head r % 4, and keeps the running max and sum of head r % 4; the softmax
    // then costs one exponential per lane and step instead of twenty.
    constexpr bool kScatter = SC && LPP == 16 && G == 4 && U == 4;
    const int rl = lane & 15;
    float mh = -INFINITY, lh = 0.f;
    auto compute_scatter = [&](const CacheRow<CT> (&k)[U], const CacheRow<CT> (&v)[U], int step) {
        float x[16];
#pragma unroll
        for (int u = 0; u < U; u++) {
            float kf[8];
            k[u].get(kf);
#pragma unroll
            for (int h = 0; h < G; h++) {
                float s = 0.f;
#pragma unroll
                for (int d = 0; d < 8; d++) s = fmaf(qr[h][d], kf[d], s);
                x[u * G + h] = s;
            }
        }
        const float s = row_reduce_scatter16(x, rl);
        const bool valid = step * NG * U + (rl >> 2) * NG + slot < n;
        const float sc = valid ? s : -INFINITY;
        float mx = fmaxf(sc, dpp_src<0x124, 0xf>(sc));  // row_ror:4, then :8: the head's 4 positions
        mx = fmaxf(mx, dpp_src<0x128, 0xf>(mx));
        const float mnew = fmaxf(mh, mx);
        const float ref = mnew == -INFINITY ? 0.f : mnew;  // no valid position yet: keep zeros
        // Rescale only when a running maximum moved somewhere in the wave (else the factor is 1).
        if (__builtin_amdgcn_ballot_w64(mnew > mh)) {
            const float c = exp2_hw(mh - ref);
            lh *= c;
            const float cb[4] = {row_lane<0>(c), row_lane<1>(c), row_lane<2>(c), row_lane<3>(c)};
#pragma unroll
            for (int h = 0; h < G; h++)
#pragma unroll
                for (int d = 0; d < 8; d++) acc[h][d] *= cb[h];
            mh = mnew;
        }
        const float pr = exp2_hw(sc - ref);
        float ps = pr + dpp_src<0x124, 0xf>(pr);
        ps += dpp_src<0x128, 0xf>(ps);
        lh += ps;
        const float pb[16] = {row_lane<0>(pr),  row_lane<1>(pr),  row_lane<2>(pr),  row_lane<3>(pr),
                              row_lane<4>(pr),  row_lane<5>(pr),  row_lane<6>(pr),  row_lane<7>(pr),
                              row_lane<8>(pr),  row_lane<9>(pr),  row_lane<10>(pr), row_lane<11>(pr),
                              row_lane<12>(pr), row_lane<13>(pr), row_lane<14>(pr), row_lane<15>(pr)};
        float vf[U][8];
#pragma unroll
        for (int u = 0; u < U; u++) v[u].get(vf[u]);
#pragma unroll
        for (int h = 0; h < G; h++)
#pragma unroll
            for (int d = 0; d < 8; d++) {
                float a = acc[h][d];
#pragma unroll
                for (int u = 0; u < U; u++) a = fmaf(pb[u * G + h], vf[u][d], a);
                acc[h][d] = a;
            }
    };
    auto compute = [&](const CacheRow<CT> (&k)[U], const CacheRow<CT> (&v)[U], int step) {
        if constexpr (kScatter) {
            compute_scatter(k, v, step);
            return;
        }
        float sc[U][G];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const bool valid = step * NG * U + u * NG + slot < n;
            float kf[8];
            k[u].get(kf);
#pragma unroll
            for (int h = 0; h < G; h++) {
                float s = 0.f;
#pragma unroll
                for (int d = 0; d < 8; d++) s = fmaf(qr[h][d], kf[d], s);
                s = group_sum<LPP>(s);
                sc[u][h] = valid ? s : -INFINITY;
            }
        }
        float vf[U][8];
#pragma unroll
        for (int u = 0; u < U; u++) v[u].get(vf[u]);
        float mxs[G], ref[G];
        bool grew = false;
#pragma unroll
        for (int h = 0; h < G; h++) {
            float mx = m[h];
#pragma unroll
            for (int u = 0; u < U; u++) mx = fmaxf(mx, sc[u][h]);
            grew |= mx > m[h];
            mxs[h] = mx;
            ref[h] = mx == -INFINITY ? 0.f : mx;  // no valid position yet: keep zeros
        }
        // Rescale only when a running maximum moved somewhere in the wave: otherwise every factor
        // is 2^0 = 1 (or 0 on a slot still all zeros) and the products would change no bit.
        if (__builtin_amdgcn_ballot_w64(grew)) {
#pragma unroll
            for (int h = 0; h < G; h++) {
                const float c = exp2_hw(m[h] - ref[h]);
                l[h] *= c;
#pragma unroll
                for (int d = 0; d < 8; d++) acc[h][d] *= c;
                m[h] = mxs[h];
            }
        }
#pragma unroll
        for (int h = 0; h < G; h++) {
            float pr[U];
#pragma unroll
            for (int u = 0; u < U; u++) pr[u] = exp2_hw(sc[u][h] - ref[h]);
            float lsum = l[h];
#pragma unroll
            for (int u = 0; u < U; u++) lsum += pr[u];
            l[h] = lsum;
#pragma unroll
            for (int d = 0; d < 8; d++) {
                float a = acc[h][d];
#pragma unroll
                for (int u = 0; u < U; u++) a = fmaf(pr[u], vf[u][d], a);
                acc[h][d] = a;
            }
        }
    };

    // Steps of NG * U positions; the next step's rows are requested before the current one is
    // computed, and the last step is computed with nothing issued behind it. ST 1 and 2 (slices of
    // that many steps at most, chosen by the launch): straight-line code that requests all the steps,
    // with q, before computing any. The loop below would take two memory round trips in a row there:
    // the compiler's copy of the first step's rows into the loop registers waits for all of them
    // before the second step is requested.
    const int steps = (n + NG * U - 1) / (NG * U);  // block-uniform
    if constexpr (ST > 0) {
        load(ka, va, 0);
        if constexpr (ST == 2) load(kb, vb, 1);
        // Nothing moves above this point: left alone, the scheduler scales q (waiting for it) before
        // requesting most of the rows.
        __builtin_amdgcn_sched_barrier(0);
        scale_q();
        if (steps > 0) compute(ka, va, 0);
        if constexpr (ST == 2) {
            if (steps > 1) compute(kb, vb, 1);
        }
    } else if (steps > 0) {
        load(ka, va, 0);
        int s = 0;
        for (;;) {
            if (s + 1 == steps) {
                compute(ka, va, s);
                break;
            }
            load(kb, vb, s + 1);
            compute(ka, va, s);
            s++;
            if (s + 1 == steps) {
                compute(kb, vb, s);
                break;
            }
            load(ka, va, s + 1);
            compute(kb, vb, s);
            s++;
        }
    }

    if constexpr (kScatter) {  // lane h of each row holds head h's running max and sum
        const float mv[4] = {row_lane<0>(mh), row_lane<1>(mh), row_lane<2>(mh), row_lane<3>(mh)};
        const float lv[4] = {row_lane<0>(lh), row_lane<1>(lh), row_lane<2>(lh), row_lane<3>(lh)};
#pragma unroll
        for (int h = 0; h < G; h++) {
            m[h] = mv[h];
            l[h] = lv[h];
        }
    }

    // Combine the wave's slots in registers, in a fixed order: each head's maximum M and weighted sum
    // over the slots, then the accumulators, weighted by 2^(m - M). Those are reduce-scattered over the
    // four 16-lane rows (a row swap puts the halves that two rows keep side by side, one add reduces
    // both), which leaves a lane 2 G of its G * 8 sums; slots that share a row are summed by rotations.
    constexpr int N8 = G * 8, N4 = N8 / 4;
    float a4[N4];
    {
        float f[N8];
#pragma unroll
        for (int h = 0; h < G; h++) {
            const float M = slot_reduce<LPP, true>(m[h]);
            const float c = M == -INFINITY ? 0.f : exp2_hw(m[h] - M);
            m[h] = M;
            l[h] = slot_reduce<LPP, false>(l[h] * c);
#pragma unroll
            for (int d = 0; d < 8; d++) f[h * 8 + d] = acc[h][d] * c;
        }
        float f2[N8 / 2];
#pragma unroll
        for (int i = 0; i < N8 / 2; i++) {
            const auto w = __builtin_amdgcn_permlane32_swap(__float_as_uint(f[i]), __float_as_uint(f[i + N8 / 2]), false, false);
            f2[i] = __uint_as_float(w[0]) + __uint_as_float(w[1]);
        }
#pragma unroll
        for (int i = 0; i < N4; i++) {
            const auto w = __builtin_amdgcn_permlane16_swap(__float_as_uint(f2[i]), __float_as_uint(f2[i + N4]), false, false);
            float v = __uint_as_float(w[0]) + __uint_as_float(w[1]);
            if constexpr (LPP <= 8) v += dpp_src<0x120 + (LPP <= 8 ? LPP : 1), 0xf>(v);      // row_ror:LPP
            if constexpr (LPP <= 4) v += dpp_src<0x120 + (LPP <= 4 ? 2 * LPP : 1), 0xf>(v);  // row_ror:2 LPP
            if constexpr (LPP <= 2) v += dpp_src<0x120 + (LPP <= 2 ? 4 * LPP : 1), 0xf>(v);  // row_ror:4 LPP
            a4[i] = v;
        }
    }
    // The waves' sums meet in LDS: value i of a lane is number (lane >> 4's row quarter) * N4 + i of
    // its G * 8, that is head (number / 8), dim lg * 8 + number % 8.
    if ((lane & 15) < LPP) {
        const int first = (lane >> 5) * (N8 / 2) + ((lane >> 4) & 1) * N4;
#pragma unroll
        for (int i = 0; i < N4; i += (N4 >= 4 ? 4 : 2)) {
            const int v = first + i;
            float* dst = &s_acc[wave][(v >> 3) * HD + lg * 8 + (v & 7)];
            if constexpr (N4 >= 4)
                *reinterpret_cast<float4*>(dst) = make_float4(a4[i], a4[i + 1], a4[i + 2], a4[i + 3]);
            else
                *reinterpret_cast<float2*>(dst) = make_float2(a4[i], a4[i + 1]);
        }
    }
    if (lane == 0) {
#pragma unroll
        for (int h = 0; h < G; h++) {
            s_m[wave][h] = m[h];
            s_l[wave][h] = l[h];
        }
    }
    __syncthreads();

    // The output directly when the sequence is not split, else this split's partial.
    constexpr int PS = partial_stride(G, HD);
    float* part = p.splits > 1 ? p.partials + (((size_t)b * p.nkv + g) * p.splits + split) * PS : nullptr;
    for (int idx = tid; idx < G * HD; idx += kBlock) {
        const int h = idx / HD, d = idx - h * HD;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; w++) M = fmaxf(M, s_m[w][h]);
        float num = 0.f, den = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const float c = M == -INFINITY ? 0.f : exp2_hw(s_m[w][h] - M);
            num = fmaf(c, s_acc[w][idx], num);
            den = fmaf(c, s_l[w][h], den);
        }
        if (p.splits == 1) {
            if (h < gsize)
                store_act(p.out, p.out_dtype, (size_t)b * p.nh * HD + (size_t)(g * gsize + h) * HD + d,
                          den > 0.f ? num / den : 0.f);
        } else {
            part[idx] = num;
            if (d == 0) {
                part[G * HD + h] = M;
                part[G * HD + G + h] = den;
            }
        }
    }
}

// Log-sum-exp merge of the splits' partials. Block (kv head, column group, batch): thread
// (column c of 4 dims, lane j of J) loads the max, sum and 4 accumulators of splits j, j + J, ...
// in one round (eight splits in flight), folds them with an online max, and the J lanes of a
// column are combined in a fixed order.
template <int HD, int G>
__global__ __launch_bounds__(kBlock) void attn_merge_kernel(const AttnParams p) {
    constexpr int NC = G * HD / 4;  // float4 columns of a (batch, kv head)
    constexpr int CB = NC < 32 ? NC : 32;  // columns per block
    constexpr int J = kBlock / CB;  // split lanes per column
    constexpr int PS = partial_stride(G, HD);
    __shared__ float s_mx[J][CB], s_den[J][CB];
    __shared__ float4 s_num[J][CB];
    const int g = blockIdx.x, b = blockIdx.z;
    const int tid = threadIdx.x, cl = tid % CB, j = tid / CB;
    const int c = blockIdx.y * CB + cl;
    const int cc = min(c, NC - 1);
    const int h = cc * 4 / HD;
    const int gsize = p.nh / p.nkv;
    const int S = p.splits;
    // The empty asm makes the partials address live before the loop, so its argument load joins
    // the kernel's first load round instead of a round of its own after the loop guard (the
    // address-space cast keeps the loads global ones, which the asm would otherwise hide).
    const float* allp = p.partials + ((size_t)b * p.nkv + g) * S * PS;
    asm volatile("" : "+s"(allp));
    const __attribute__((address_space(1))) float* all = (const __attribute__((address_space(1))) float*)allp;
    float M = -INFINITY, den = 0.f;
    float4 num = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = j; s0 < S; s0 += 8 * J) {
        float ms[8], ls[8];
        float4 v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const __attribute__((address_space(1))) float* ps = all + (size_t)min(s0 + u * J, S - 1) * PS;
            typedef float f32x4_t __attribute__((ext_vector_type(4)));
            const f32x4_t t = *reinterpret_cast<const __attribute__((address_space(1))) f32x4_t*>(ps + cc * 4);
            v[u] = make_float4(t.x, t.y, t.z, t.w);
            ms[u] = ps[G * HD + h];
            ls[u] = ps[G * HD + G + h];
        }
        float mx = M;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (s0 + u * J < S) mx = fmaxf(mx, ms[u]);
        if (mx != -INFINITY) {
            const float cs = exp2_hw(M - mx);  // 0 while M is still -inf
            num.x *= cs;
            num.y *= cs;
            num.z *= cs;
            num.w *= cs;
            den *= cs;
#pragma unroll
            for (int u = 0; u < 8; u++) {
                if (s0 + u * J < S && ms[u] != -INFINITY) {
                    const float w = exp2_hw(ms[u] - mx);
                    num.x = fmaf(w, v[u].x, num.x);
                    num.y = fmaf(w, v[u].y, num.y);
                    num.z = fmaf(w, v[u].z, num.z);
                    num.w = fmaf(w, v[u].w, num.w);
                    den = fmaf(w, ls[u], den);
                }
            }
            M = mx;
        }
    }
    s_mx[j][cl] = M;
    s_den[j][cl] = den;
    s_num[j][cl] = num;
    __syncthreads();
    if (j == 0 && c < NC && h < gsize) {
        float Mt = -INFINITY;
#pragma unroll
        for (int i = 0; i < J; i++) Mt = fmaxf(Mt, s_mx[i][cl]);
        float4 t = make_float4(0.f, 0.f, 0.f, 0.f);
        float dt = 0.f;
        if (Mt != -INFINITY) {
#pragma unroll
            for (int i = 0; i < J; i++) {
                const float w = s_mx[i][cl] == -INFINITY ? 0.f : exp2_hw(s_mx[i][cl] - Mt);
                const float4 u = s_num[i][cl];
                t.x = fmaf(w, u.x, t.x);
                t.y = fmaf(w, u.y, t.y);
                t.z = fmaf(w, u.z, t.z);
                t.w = fmaf(w, u.w, t.w);
                dt = fmaf(w, s_den[i][cl], dt);
            }
        }
        const float inv = dt > 0.f ? 1.f / dt : 0.f;
        const size_t o = (size_t)b * p.nh * HD + (size_t)(g * gsize + h) * HD + (cc * 4 - h * HD);
        store_act(p.out, p.out_dtype, o + 0, t.x * inv);
        store_act(p.out, p.out_dtype, o + 1, t.y * inv);
        store_act(p.out, p.out_dtype, o + 2, t.z * inv);
        store_act(p.out, p.out_dtype, o + 3, t.w * inv);
    }
}

template <int HD, int CT, int QT, int G>
int launch_g(hipStream_t s, const AttnParams& p, int seq_len_step, size_t cache_batch_stride) {
    // The kv head is the fastest-varying block index in both kernels: workgroups are dealt to the
    // XCDs round robin by linear id, so with 8 kv heads every split of head g and the merge blocks
    // that read its partials run on XCD g, and the merge finds the partials in that XCD's L2.
    dim3 grid(p.nkv, p.splits, p.batch);
    // The reduce-scattered softmax has fewer VALU operations but longer dependent chains per step.
    // Measured on the 8B shapes: faster for short splits (decode at 2048 positions: 10.4 against
    // 10.9 us per layer; up to 256 positions per split) and for long ones at two blocks per CU
    // (batch 8 x 32768: 183 against 192 us), 3-4 % slower at one block per CU with 512-1024
    // positions per split (batch 1 x 32768, batch 8 x 4096), where one wave per SIMD cannot hide
    // those chains.
    // Slices of at most two steps (at any sequence length up to max_seq_len) take the straight-line
    // kernel; fp16 caches only (two steps of fp32 rows spill with eight heads). Measured on the 8B
    // shapes: 512 positions 8.9 -> 7.9 us at batch 1 and 10.5 -> 9.5 us at batch 8, 4096 positions
    // at batch 1 10.5 -> 9.5-9.8 us.
    constexpr int kSlots = kWaves * 64 / (HD / 8);  // position slots of a block
    constexpr bool SC = HD == 128 && G == 4;
    const int per_split = (int)ceil_div(p.max_seq_len, std::max(p.splits, 1));
    if (per_split <= kSlots)
        attn_split_kernel<HD, CT, QT, G, 1, 1><<<grid, kBlock, 0, s>>>(p, seq_len_step, cache_batch_stride);
    else if (per_split <= 2 * kSlots)
        attn_split_kernel<HD, CT, QT, G, 2, 1><<<grid, kBlock, 0, s>>>(p, seq_len_step, cache_batch_stride);
    else if (per_split <= kUnroll * kSlots)
        attn_split_kernel<HD, CT, QT, G, kUnroll, 1, SC><<<grid, kBlock, 0, s>>>(p, seq_len_step, cache_batch_stride);
    else if (CT == L0H_F16 && per_split <= 2 * kUnroll * kSlots)
        attn_split_kernel<HD, CT, QT, G, kUnroll, CT == L0H_F16 ? 2 : 0, SC><<<grid, kBlock, 0, s>>>(p, seq_len_step, cache_batch_stride);
    else if (SC && (per_split <= 256 || per_split >= 2048))
        attn_split_kernel<HD, CT, QT, G, kUnroll, 0, SC><<<grid, kBlock, 0, s>>>(p, seq_len_step, cache_batch_stride);
    else
        attn_split_kernel<HD, CT, QT, G, kUnroll, 0><<<grid, kBlock, 0, s>>>(p, seq_len_step, cache_batch_stride);
    int st = launch_status("attention");
    if (st || p.splits == 1) return st;
    constexpr int NC = G * HD / 4, CB = NC < 32 ? NC : 32;
    attn_merge_kernel<HD, G><<<dim3(p.nkv, NC / CB, p.batch), kBlock, 0, s>>>(p);
    return launch_status("attention merge");
}

int group_pow2(int gsize) { return gsize <= 1 ? 1 : gsize <= 2 ? 2 : gsize <= 4 ? 4 : 8; }

template <int HD, int CT, int QT>
int launch_q(hipStream_t s, const AttnParams& p, int seq_len_step, size_t stride) {
    switch (group_pow2(p.nh / p.nkv)) {
    case 1: return launch_g<HD, CT, QT, 1>(s, p, seq_len_step, stride);
    case 2: return launch_g<HD, CT, QT, 2>(s, p, seq_len_step, stride);
    case 4: return launch_g<HD, CT, QT, 4>(s, p, seq_len_step, stride);
    default: return launch_g<HD, CT, QT, 8>(s, p, seq_len_step, stride);
    }
}

template <int HD>
int launch_hd(hipStream_t s, const AttnParams& p, int seq_len_step, size_t stride) {
    if (p.cache_dtype == L0H_F16)
        return p.q_dtype == L0H_F16 ? launch_q<HD, L0H_F16, L0H_F16>(s, p, seq_len_step, stride)
                                    : launch_q<HD, L0H_F16, L0H_F32>(s, p, seq_len_step, stride);
    return p.q_dtype == L0H_F16 ? launch_q<HD, L0H_F32, L0H_F16>(s, p, seq_len_step, stride)
                                : launch_q<HD, L0H_F32, L0H_F32>(s, p, seq_len_step, stride);
}

int launch_any(hipStream_t s, const AttnParams& p, int seq_len_step, size_t cache_batch_stride) {
    if (p.head_dim != 16 && p.head_dim != 32 && p.head_dim != 64 && p.head_dim != 128)
        return fail(L0H_ERR_UNSUPPORTED, "attention supports head_dim 16, 32, 64 and 128");
    if (p.nkv <= 0 || p.nh % p.nkv != 0 || p.nh / p.nkv > kGroupMax)
        return fail(L0H_ERR_UNSUPPORTED, "attention needs n_heads a multiple of n_kv_heads, at most 8 per group");
    if (p.cache_dtype != L0H_F16 && p.cache_dtype != L0H_F32)
        return fail(L0H_ERR_INVALID_ARG, "cache dtype must be F16 or F32");
    if (p.q_dtype != L0H_F16 && p.q_dtype != L0H_F32)
        return fail(L0H_ERR_INVALID_ARG, "q dtype must be F16 or F32");
    if (p.splits < 1 || p.splits > kMaxSplits) return fail(L0H_ERR_INVALID_ARG, "attention splits out of range");
    if (p.max_seq_len < 1 || p.batch < 1) return fail(L0H_ERR_INVALID_ARG, "attention sizes must be positive");
    if (p.splits > 1 && !p.partials) return fail(L0H_ERR_INVALID_ARG, "attention workspace missing");
    if ((((uintptr_t)p.q | (uintptr_t)p.kc | (uintptr_t)p.vc) & 15) != 0)
        return fail(L0H_ERR_INVALID_ARG, "attention buffers must be 16-byte aligned");
    switch (p.head_dim) {
    case 16: return launch_hd<16>(s, p, seq_len_step, cache_batch_stride);
    case 32: return launch_hd<32>(s, p, seq_len_step, cache_batch_stride);
    case 64: return launch_hd<64>(s, p, seq_len_step, cache_batch_stride);
    default: return launch_hd<128>(s, p, seq_len_step, cache_batch_stride);
    }
}

// ---------------------------------------------------------------------------------------------
// Causal prefill (Attention.ExecutePrefill, LlmDecoderLayer.cs:369-371) over an fp32 cache, fp32
// throughout, on v_mfma_f32_16x16x4_f32. A query vector is a (token, q head of the group) pair; a block
// holds 16 consecutive ones, in the registers of each of its four waves. A wave takes every fourth step
// of 16 positions on its own, without LDS or barriers: a lane's operands are 16-byte pieces of the K and
// V rows as they lie in memory. Scores, S^T = K Q^T: A is K (row = position l % 16), B is Q (column =
// query l % 16), and the MFMA's k slot l / 16 stands for dim 16 s + 4 (l / 16) + j in product j of piece
// s. Lane l then holds query l % 16 at the positions 4 (l / 16) + r. Product r of O^T += V^T P^T takes
// exactly those: its k slot l / 16 is position 4 (l / 16) + r, B is P as it stands, and A is V's element
// i of the lane's piece (dims 64 e + 4 (l % 16) + i), which makes the output's rows the dims of one i.
// V is requested before the scores, the next K before the softmax; the waves' sums meet in LDS at the end.
//
// Bound by the fp32 MFMAs once the chip is full (32 q / 8 kv heads of 128, 2047 tokens: 34 GFLOP in
// 371-400 us, 86-93 of 157 TFLOP/s), below that by the chain of one wave's steps. It took the place of fp32
// FMAs on tiles in LDS (64 queries a block): that call 1491 -> 371-400 us, 14 / 2 heads of 64, 500 tokens
// behind 37 64 -> 13 us, 14 tokens 10.3 -> 5.4. Four waves with different queries each, all steps of
// them: 402, 28 and 5.0 us, and 463, 47 and 6.9 with 32 queries a wave (half the reads).
// ---------------------------------------------------------------------------------------------
typedef __attribute__((ext_vector_type(4))) float f32x4_t;

// 4 consecutive query values (fp32 or fp16) as fp32.
template <int QT>
__device__ __forceinline__ f32x4_t load_q4(const void* base, size_t idx) {
    if constexpr (QT == L0H_F32) {
        return *reinterpret_cast<const f32x4_t*>(static_cast<const float*>(base) + idx);
    } else {
        const uint2 a = *reinterpret_cast<const uint2*>(static_cast<const uint16_t*>(base) + idx);
        const float2 lo = __half22float2(__builtin_bit_cast(__half2, a.x)), hi = __half22float2(__builtin_bit_cast(__half2, a.y));
        return f32x4_t{lo.x, lo.y, hi.x, hi.y};
    }
}

constexpr int kPrefillVec = 16;  // query vectors per block

// Four consecutive outputs in one store (unaligned: `out` may start at any element).
__device__ __forceinline__ void store_out4(const AttnParams& p, size_t at, f32x4_t v) {
    typedef __attribute__((ext_vector_type(4), aligned(4))) float f32x4_u;
    typedef __attribute__((ext_vector_type(4), aligned(2))) uint16_t u16x4_u;
    if (p.out_dtype == L0H_F32) {
        *reinterpret_cast<f32x4_u*>(static_cast<float*>(p.out) + at) = v;
    } else {
        u16x4_u b;
#pragma unroll
        for (int i = 0; i < 4; i++) b[i] = p.out_dtype == L0H_F16 ? __half_as_ushort(__float2half_rn(v[i])) : float_to_bf16_bits(v[i]);
        *reinterpret_cast<u16x4_u*>(static_cast<uint16_t*>(p.out) + at) = b;
    }
}

// Grid of the kernels whose blocks take `per` consecutive query vectors: kv head, then tile of vectors (the
// kv head varies fastest: with 8 of them each XCD keeps one head's rows in its L2), and a block's tile, the
// last first: those queries see the most positions, and the short blocks fill in behind them. Negative:
// no tile (y x z rounds the count up; a grid's y is limited).
constexpr int kTilesY = 32768;
dim3 prefill_grid(int nkv, long nvec, int per) {
    const long tiles = (nvec + per - 1) / per;
    return dim3(nkv, (unsigned)std::min<long>(tiles, kTilesY), (unsigned)((tiles + kTilesY - 1) / kTilesY));
}
__device__ __forceinline__ int prefill_tile(int nvec, int per) {
    return (nvec + per - 1) / per - 1 - (int)(blockIdx.z * gridDim.y + blockIdx.y);
}

template <int HD, int QT>
__global__ __launch_bounds__(kBlock) void attn_prefill_f32_kernel(const AttnParams p, int pos0, int tokens, int gsize) {
    constexpr int NS = HD / 16;  // 16-byte pieces of a K row per lane
    constexpr int NE = HD / 64;  // 16-byte pieces of a V row per lane
    __shared__ __attribute__((aligned(16))) float s_o[kWaves][kPrefillVec][HD + 4];
    __shared__ float s_m[kWaves][kPrefillVec], s_l[kWaves][kPrefillVec];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lq = lane & 15, lg = lane >> 4;
    const int g = blockIdx.x;
    const int nvec = tokens * gsize;
    const int v0 = prefill_tile(nvec, kPrefillVec) * kPrefillVec;
    if (v0 < 0) return;
    const int row_elems = p.nkv * HD;
    const float* kbase = static_cast<const float*>(p.kc) + (size_t)g * HD + 4 * lg;
    const float* vbase = static_cast<const float*>(p.vc) + (size_t)g * HD + 4 * lq;
    // Last position the block's first and last query see.
    const int lim_first = pos0 + v0 / gsize;
    const int kmax = pos0 + min(v0 + kPrefillVec - 1, nvec - 1) / gsize;

    const float qscale = 1.4426950408889634f / sqrtf((float)HD);
    f32x4_t q[NS];
    const int vq = min(v0 + lq, nvec - 1), tq = vq / gsize, hq = g * gsize + vq - tq * gsize;
    const int lim = pos0 + tq;  // (a lane past the last vector repeats it and stores nothing)
#pragma unroll
    for (int s = 0; s < NS; s++) q[s] = load_q4<QT>(p.q, ((size_t)tq * p.nh + hq) * HD + 16 * s + 4 * lg) * qscale;

    f32x4_t kr[NS], vr[4][NE];
    auto load_k = [&](int base) {
        const float* r = kbase + (size_t)min(base + lq, kmax) * row_elems;
#pragma unroll
        for (int s = 0; s < NS; s++) kr[s] = *reinterpret_cast<const f32x4_t*>(r + 16 * s);
    };
    auto load_v = [&](int base) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const float* row = vbase + (size_t)min(base + 4 * lg + r, kmax) * row_elems;
#pragma unroll
            for (int e = 0; e < NE; e++) vr[r][e] = *reinterpret_cast<const f32x4_t*>(row + 64 * e);
        }
    };

    float m = -INFINITY, l = 0.f;
    f32x4_t o[NE][4];
#pragma unroll
    for (int e = 0; e < NE; e++)
#pragma unroll
        for (int i = 0; i < 4; i++) o[e][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    constexpr int kStride = 16 * kWaves;
    const int first = wave * 16;
    if (first <= kmax) load_k(first);
    for (int base = first; base <= kmax; base += kStride) {
        load_v(base);
        f32x4_t st = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < NS; s++)
#pragma unroll
            for (int j = 0; j < 4; j++) st = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[s][j], q[s][j], st, 0, 0, 0);
        load_k(base + kStride);  // past the end: clamped, not used
        if (base + 15 > lim_first) {
#pragma unroll
            for (int r = 0; r < 4; r++)
                if (base + 4 * lg + r > lim) st[r] = -INFINITY;
        }
        const float mx = slot_reduce<16, true>(fmaxf(fmaxf(st[0], st[1]), fmaxf(st[2], st[3])));
        const float mn = fmaxf(m, mx);
        const float ref = mn == -INFINITY ? 0.f : mn;  // no position seen yet: keep zeros
        if (__builtin_amdgcn_ballot_w64(mn > m)) {  // else every factor is 1
            const float c = exp2_hw(m - ref);
            l *= c;
#pragma unroll
            for (int e = 0; e < NE; e++)
#pragma unroll
                for (int i = 0; i < 4; i++) o[e][i] *= c;
            m = mn;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            st[r] = exp2_hw(st[r] - ref);
            l += st[r];
        }
#pragma unroll
        for (int r = 0; r < 4; r++)
#pragma unroll
            for (int e = 0; e < NE; e++)
#pragma unroll
                for (int i = 0; i < 4; i++) o[e][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[r][e][i], st[r], o[e][i], 0, 0, 0);
    }

    // Lane l holds query l % 16, dims 64 e + 16 (l / 16) + 4 r + i; its l is the sum of its positions.
    const float sum = slot_reduce<16, false>(l);
    if (lg == 0) {
        s_m[wave][lq] = m;
        s_l[wave][lq] = sum;
    }
#pragma unroll
    for (int e = 0; e < NE; e++)
#pragma unroll
        for (int r = 0; r < 4; r++)
            *reinterpret_cast<f32x4_t*>(&s_o[wave][lq][64 * e + 16 * lg + 4 * r]) =
                f32x4_t{o[e][0][r], o[e][1][r], o[e][2][r], o[e][3][r]};
    __syncthreads();
    for (int idx = tid; idx < kPrefillVec * HD / 4; idx += kBlock) {
        const int qi = idx / (HD / 4), d = (idx - qi * (HD / 4)) * 4, v = v0 + qi;
        if (v >= nvec) continue;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; w++) M = fmaxf(M, s_m[w][qi]);
        f32x4_t num = f32x4_t{0.f, 0.f, 0.f, 0.f};
        float den = 0.f;
#pragma unroll
        for (int w = 0; w < kWaves; w++) {
            const float c = M == -INFINITY ? 0.f : exp2_hw(s_m[w][qi] - M);
            num += c * *reinterpret_cast<const f32x4_t*>(&s_o[w][qi][d]);
            den = fmaf(c, s_l[w][qi], den);
        }
        const float inv = den > 0.f ? 1.f / den : 0.f;
        const int t = v / gsize, h = g * gsize + v - t * gsize;
        store_out4(p, ((size_t)t * p.nh + h) * HD + d, num * inv);
    }
}

template <int HD, int QT>
int launch_prefill_f32(hipStream_t s, const AttnParams& p, int pos0, int tokens) {
    const int gsize = p.nh / p.nkv;
    const long nvec = (long)tokens * gsize;
    attn_prefill_f32_kernel<HD, QT><<<prefill_grid(p.nkv, nvec, kPrefillVec), kBlock, 0, s>>>(p, pos0, tokens, gsize);
    return launch_status("attn_prefill_f32");
}

// ---------------------------------------------------------------------------------------------
// Causal prefill on MFMA (fp16 cache), query-tiled: a block holds 32 NQ consecutive query vectors ((token, q
// head of the group) pairs of one kv head) and streams that head's K and V rows in tiles of 64 positions
// through LDS once for all of them. PS = 1: a wave owns 32 vectors; PS = 2: two waves share 32 vectors, one
// takes the first half of every tile's positions and one the second, and their sums meet at the end.
// Scores are computed transposed, S^T = K Q^T, with v_mfma_f32_32x32x16_f16 (K fragments from LDS, the
// wave's Q fragments in registers, fp16, pre-scaled by log2(e) / sqrt(d)): lane l then holds, for query
// l % 32, the positions 8 (r / 4) + 4 (l / 32) + r % 4 of 32 (r < 16). After the online softmax (fp32, the
// row spread over 2 lanes, each with its own share of the sum) values r = 8 c .. 8 c + 7 are the B operand of
// the P.V MFMA O^T += V^T P^T when its K slots are those positions; the A operand, four positions of one
// dim twice, comes from the row-major V tile by transposed LDS reads (ds_read_b64_tr_b16). P is rounded to
// fp16 for the MFMA; the softmax sums stay fp32.
//
// What bounds it: the vector instructions around the products (32 values a lane and tile: subtract, 2^x, add,
// half a conversion, half a maximum) and the LDS reads, with two to three waves a SIMD to overlap them; at
// the largest sizes the spread of the causal blocks. It took the place of 16 vectors a wave with
// 16 x 16 x 32 products and V transposed in registers, where every wave read all of K and V from LDS for 16
// vectors: 32 / 8 heads of 128, 2047 tokens 127 -> 67 us (34 GFLOP, 270 -> 510 TFLOP/s), 500 behind 1000
// 45.3 -> 33.6, 8 tokens 5.9 -> 5.5 (8.3 with the outputs stored one by one: 64 of them a lane); 14 / 2 heads of
// 64, 500 behind 37 13.3 -> 9.4, 14 tokens 5.2 -> 5.1; 32 / 8 of 64, 300 10.8 -> 7.2. Two tile buffers and one
// barrier a tile: 2047 tokens 73 -> 83 us (half the blocks fit a CU).
// ---------------------------------------------------------------------------------------------
constexpr int kPrefillGroup = 64;  // q heads per kv head, at most
constexpr int kPK = 64;            // key positions per tile
typedef __attribute__((ext_vector_type(8))) _Float16 f16x8_t;
typedef __attribute__((ext_vector_type(16))) float f32x16_t;

// Two fp32 values rounded to fp16 (to nearest), as one conversion.
__device__ __forceinline__ uint32_t pack_half2(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) float f32x2_t;
    typedef __attribute__((ext_vector_type(2))) _Float16 f16x2_t;
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{a, b}, f16x2_t));
}

// prefill_tile in rounds of `round` tiles, every second one reversed: of the blocks a CU holds together,
// `round` apart, the longer stands beside the shorter (32 / 8 heads of 128, 1500 tokens: 53.5 -> 48.0 us).
__device__ __forceinline__ int prefill_tile_snake(int nvec, int per, int round) {
    const int tiles = (nvec + per - 1) / per, t = (int)(blockIdx.z * gridDim.y + blockIdx.y);
    if (t >= tiles) return -1;
    const int r = t / round, at = t - r * round, size = min(round, tiles - r * round);
    return tiles - 1 - (r * round + ((r & 1) ? size - 1 - at : at));
}

template <int HD, int QT, int NQ, int PS>
__global__ __launch_bounds__(64 * NQ * PS) void attn_prefill_mfma_kernel(const AttnParams p, int pos0, int tokens, int gsize, int round) {
    constexpr int NW = NQ * PS;
    constexpr int NJ = 2 / PS;    // 32-position halves of a tile per wave
    constexpr int KLD = HD + 8;   // K tile row stride (halves): 16 rows hit distinct banks
    constexpr int VLD = HD + 32;  // V tile row stride: rows 16 banks apart, 8 of them in a transposed read
    constexpr int CPR = HD / 8;   // 16-byte chunks per cache row
    constexpr int NC = CPR / NW;  // chunks per thread per tile (K, and again V)
    constexpr int KS = HD / 16;   // MFMA K steps over the head dim
    constexpr int NI = HD / 32;   // 32-dim output sub-tiles
    __shared__ __attribute__((aligned(16))) uint16_t smem[kPK * (KLD + VLD)];  // a tile's K rows, then its V rows

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lq = lane & 31, lh = lane >> 5;
    const int group = wave % NQ, j0 = wave / NQ;  // the wave's query vectors, and its half of a tile (PS = 2)
    const int g = blockIdx.x;
    const int nvec = tokens * gsize;
    const int b0 = prefill_tile_snake(nvec, 32 * NQ, round) * (32 * NQ);
    if (b0 < 0) return;
    const int kmax = pos0 + min(b0 + 32 * NQ - 1, nvec - 1) / gsize;
    const int row_elems = p.nkv * HD;
    const uint16_t* kc = static_cast<const uint16_t*>(p.kc) + (size_t)g * HD;
    const uint16_t* vc = static_cast<const uint16_t*>(p.vc) + (size_t)g * HD;

    // This lane's query vector (a lane past the last one repeats it and stores nothing), and the last
    // positions the wave's first and last vectors see.
    const int v = min(b0 + group * 32 + lq, nvec - 1), tq = v / gsize, hq = g * gsize + v - tq * gsize;
    const int lim = pos0 + tq;
    const int lim_first = pos0 + min(b0 + group * 32, nvec - 1) / gsize, lim_last = pos0 + min(b0 + group * 32 + 31, nvec - 1) / gsize;
    const float qscale = 1.4426950408889634f / sqrtf((float)HD);
    uint4 qf[KS];  // dims 16 kk + 8 lh .. +7 as fp16
#pragma unroll
    for (int kk = 0; kk < KS; kk++) {
        float f[8];
        load8<QT>(p.q, ((size_t)tq * p.nh + hq) * HD + 16 * kk + 8 * lh, f);
        qf[kk] = make_uint4(pack_half2(f[0] * qscale, f[1] * qscale), pack_half2(f[2] * qscale, f[3] * qscale),
                            pack_half2(f[4] * qscale, f[5] * qscale), pack_half2(f[6] * qscale, f[7] * qscale));
    }

    uint4 kr[NC], vr[NC];
    auto load_tile = [&](int kt) {
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int i = tid + c * 64 * NW, r = i / CPR, col = i % CPR;
            const size_t at = (size_t)min(kt * kPK + r, kmax) * row_elems + col * 8;
            kr[c] = *reinterpret_cast<const uint4*>(kc + at);
            vr[c] = *reinterpret_cast<const uint4*>(vc + at);
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int i = tid + c * 64 * NW, r = i / CPR, col = i % CPR;
            *reinterpret_cast<u32x4_t*>(smem + r * KLD + col * 8) = u32x4_t{kr[c].x, kr[c].y, kr[c].z, kr[c].w};
            *reinterpret_cast<u32x4_t*>(smem + kPK * KLD + r * VLD + col * 8) = u32x4_t{vr[c].x, vr[c].y, vr[c].z, vr[c].w};
        }
    };
    // Four V values of one dim: with its 16 lanes' 8-byte reads of 4 rows x 16 dims, lane t at row t / 4,
    // dims 4 (t % 4) .. + 3, lane t gets dim t of the four rows.
    const int vrow = 4 * lh + ((lane >> 2) & 3), vdim = (lane & 16) + 4 * (lane & 3);
    typedef __attribute__((ext_vector_type(4))) short s16x4_t;
    auto read_v = [&](const uint16_t* at) {
        return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                                             (__attribute__((address_space(3))) s16x4_t*)const_cast<uint16_t*>(at)));
    };

    float m = -INFINITY, l = 0.f;  // l: the lane's own positions
    f32x16_t o[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) o[i] = f32x16_t{};

    const int ntiles = kmax / kPK + 1;
    load_tile(0);
    for (int kt = 0; kt < ntiles; kt++) {
        __syncthreads();  // the previous tile is no longer read
        store_tile();
        if (kt + 1 < ntiles) load_tile(kt + 1);
        __syncthreads();
        const int p0 = kt * kPK + 32 * NJ * j0;  // the wave's first position
        if (p0 > lim_last) continue;             // none of its queries sees that far
        const uint16_t* Ks = smem + 32 * NJ * j0 * KLD;
        const uint16_t* Vs = smem + kPK * KLD + (32 * NJ * j0 + vrow) * VLD + vdim;

        f32x16_t st[NJ];
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            st[j] = f32x16_t{};
#pragma unroll
            for (int kk = 0; kk < KS; kk++) {
                const uint4 a = *reinterpret_cast<const uint4*>(&Ks[(32 * j + lq) * KLD + 16 * kk + 8 * lh]);
                st[j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, qf[kk]), st[j], 0, 0, 0);
            }
        }
        if (p0 + 32 * NJ - 1 > lim_first) {  // the diagonal
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int r = 0; r < 16; r++)
                    if (p0 + 32 * j + 8 * (r >> 2) + 4 * lh + (r & 3) > lim) st[j][r] = -INFINITY;
        }
        float mt = st[0][0];
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) mt = fmaxf(mt, st[j][r]);
        const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(mt), __float_as_uint(mt), false, false);
        const float mn = fmaxf(m, fmaxf(__uint_as_float(sw[0]), __uint_as_float(sw[1])));
        const float ref = mn == -INFINITY ? 0.f : mn;
        if (__builtin_amdgcn_ballot_w64(mn > m)) {  // else every factor is 1
            const float c = exp2_hw(m - ref);
            l *= c;
#pragma unroll
            for (int i = 0; i < NI; i++) o[i] *= c;
            m = mn;
        }
        uint32_t ph[NJ][8];
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int r = 0; r < 16; r += 2) {
                const float p0 = exp2_hw(st[j][r] - ref), p1 = exp2_hw(st[j][r + 1] - ref);
                l += p0 + p1;
                ph[j][r >> 1] = pack_half2(p0, p1);
            }
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const uint4 b = make_uint4(ph[j][4 * c], ph[j][4 * c + 1], ph[j][4 * c + 2], ph[j][4 * c + 3]);
#pragma unroll
                for (int i = 0; i < NI; i++) {
                    const uint16_t* at = Vs + (32 * j + 16 * c) * VLD + 32 * i;
                    const uint2 lo = read_v(at), hi = read_v(at + 8 * VLD);
                    o[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, make_uint4(lo.x, lo.y, hi.x, hi.y)),
                                                                  __builtin_bit_cast(f16x8_t, b), o[i], 0, 0, 0);
                }
            }
    }

    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_uint(l), __float_as_uint(l), false, false);
    l = __uint_as_float(sw[0]) + __uint_as_float(sw[1]);
    if constexpr (PS == 2) {  // the second half's sums join the first's, value by value of a lane
        constexpr int NV = NI * 16 + 2;
        static_assert(NQ * NV * 64 * 4 <= sizeof(smem), "the sums take the tile's place");
        float* x = reinterpret_cast<float*>(smem) + group * NV * 64 + lane;
        __syncthreads();
        if (j0 == 1) {
#pragma unroll
            for (int i = 0; i < NI; i++)
#pragma unroll
                for (int r = 0; r < 16; r++) x[(i * 16 + r) * 64] = o[i][r];
            x[NI * 16 * 64] = m;
            x[(NI * 16 + 1) * 64] = l;
        }
        __syncthreads();
        if (j0 == 1) return;
        const float m1 = x[NI * 16 * 64], M = fmaxf(m, m1);
        const float c0 = m == -INFINITY ? 0.f : exp2_hw(m - M), c1 = m1 == -INFINITY ? 0.f : exp2_hw(m1 - M);
        l = l * c0 + x[(NI * 16 + 1) * 64] * c1;
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int r = 0; r < 16; r++) o[i][r] = o[i][r] * c0 + x[(i * 16 + r) * 64] * c1;
    }
    if (b0 + group * 32 + lq < nvec) {
        const float inv = l > 0.f ? 1.f / l : 0.f;
        const size_t base = ((size_t)tq * p.nh + hq) * HD + 4 * lh;
#pragma unroll
        for (int i = 0; i < NI; i++)
#pragma unroll
            for (int r = 0; r < 16; r += 4)
                store_out4(p, base + 32 * i + 2 * r, f32x4_t{o[i][r], o[i][r + 1], o[i][r + 2], o[i][r + 3]} * inv);
    }
}

// 32 vectors a block and two waves to share them while the chip has room for such blocks (64-vector ones
// would leave CUs idle), then 64 vectors and two waves to each 32; at head_dim 128 from three 64-vector
// blocks a CU on, one wave to each 32, which reads K and V once and not the sums twice. Measured (us, all
// with outputs stored one by one; one wave / two on 32 vectors / two on 64): 14 / 2 heads of 64, 100 tokens
// 6.6 / 6.0 / 6.6, 1000 19.9 / 16.1 / 15.9; 32 / 8 of 128, 250 13.0 / 11.8 / 12.7, 1000 32.6 / 31.2 / 28.5,
// 1500 49.6 / 54.6 / 48.0, 1700 57.4 / 66.1 / 59.6; 32 / 8 of 64, 2047 42.0 / 45.4 / 38.4.
template <int HD, int QT>
int launch_prefill_mfma(hipStream_t s, const AttnParams& p, int pos0, int tokens) {
    constexpr int kCus = 256;
    const int gsize = p.nh / p.nkv;
    const long nvec = (long)tokens * gsize, blocks = (nvec + 63) / 64 * p.nkv;
    const int round = std::max(1, kCus / p.nkv);
    if (blocks <= kCus)
        attn_prefill_mfma_kernel<HD, QT, 1, 2><<<prefill_grid(p.nkv, nvec, 32), 128, 0, s>>>(p, pos0, tokens, gsize, round);
    else if (HD == 128 && blocks >= 3 * kCus)
        attn_prefill_mfma_kernel<HD, QT, 2, 1><<<prefill_grid(p.nkv, nvec, 64), 128, 0, s>>>(p, pos0, tokens, gsize, round);
    else
        attn_prefill_mfma_kernel<HD, QT, 2, 2><<<prefill_grid(p.nkv, nvec, 64), 256, 0, s>>>(p, pos0, tokens, gsize, round);
    return launch_status("attn_prefill_mfma");
}

template <int HD>
int launch_prefill_hd(hipStream_t s, const AttnParams& p, int pos0, int tokens) {
    if (p.cache_dtype == L0H_F16)  // 16-bit operands; an fp32 cache keeps fp32 ones
        return p.q_dtype == L0H_F16 ? launch_prefill_mfma<HD, L0H_F16>(s, p, pos0, tokens)
                                    : launch_prefill_mfma<HD, L0H_F32>(s, p, pos0, tokens);
    return p.q_dtype == L0H_F16 ? launch_prefill_f32<HD, L0H_F16>(s, p, pos0, tokens)
                                : launch_prefill_f32<HD, L0H_F32>(s, p, pos0, tokens);
}

}  // namespace

int attention_default_splits(int batch, int nkv, int max_len, int compute_units) {
    // Positions per split: at least two steps (128 positions at head_dim 128), so a block
    // overlaps its second step's loads with the first step's compute; at most kMaxSplits. Blocks
    // per CU: two while every split still gets at least 2048 positions (long streams: batch 8 x
    // 32768 positions, 1.07 GB of K/V, 195-200 us against 200-206 us at one), else one (batch 1
    // x 32768 or batch 8 x 4096, 134 MB: 28.7 us against 33.7 us at two).
    // L0H_ATTN_SPLIT_POSITIONS overrides the minimum and L0H_ATTN_BLOCKS_PER_CU the blocks per CU
    // (tuning).
    static const int min_env = [] {
        const char* e = std::getenv("L0H_ATTN_SPLIT_POSITIONS");
        const int v = e ? std::atoi(e) : 0;
        return v > 0 ? v : 0;
    }();
    const int min_pos = min_env ? min_env : 128;
    static const int per_cu_env = [] {
        const char* e = std::getenv("L0H_ATTN_BLOCKS_PER_CU");
        const int v = e ? std::atoi(e) : 0;
        return v > 0 ? v : 0;
    }();
    const int len = std::max(max_len, 1);
    auto splits_for = [&](int per_cu) {
        const int target =
            (int)ceil_div((size_t)per_cu * std::max(compute_units, 1), (size_t)std::max(batch * nkv, 1));
        const int by_len = (int)ceil_div((size_t)len, (size_t)min_pos);
        return std::max(1, std::min(kMaxSplits, std::min(target, by_len)));
    };
    if (per_cu_env) return splits_for(per_cu_env);
    // Where slices of 64 positions make at most one block per CU, they are taken, up to the 64
    // that the merge folds in one round: the kernel is then bound by the latency of one slice, not by
    // bandwidth. One slice of up to 128 positions needs no merge and stays ahead. Measured (us, fp32 q,
    // slices of 128 -> 64 -> 32 positions): 14 q / 2 kv heads of 64, 1000 positions fp32 10.0 -> 9.0 ->
    // 8.7, 4000 10.7 -> 9.6 -> 10.6, fp16 142 9.2 -> 8.4 -> 8.5, 64 (one slice of 64, two of 32) 5.5 -> 8.5;
    // 32 / 8 heads of 128, fp16 512 8.6 -> 7.8 -> 8.6, 2048 9.1 -> 8.6 -> 9.1;
    // just past one block per CU, 2176 positions, 9.1 -> 9.5.
    constexpr int kFine = 64;
    const int fine = (len + kFine - 1) / kFine;
    if (!min_env && fine > 2 && fine <= 64 && (long)batch * nkv * fine <= std::max(compute_units, 1)) return fine;
    const int two = splits_for(2);
    if (len / two >= 2048) return two;
    // Slices of four steps at one block per CU: twice the splits make them two-step slices, which
    // the straight-line kernel takes, at two blocks per CU. Measured (fp16, 32 q / 8 kv heads, cold
    // K / V, graph replay, two runs each): batch 1 x 8192 13.45 -> 12.15 us, 2 x 4096 13.56 ->
    // 12.42, 4 x 2048 13.45 -> 12.43, 8 x 1024 13.28 -> 12.45; slices of three steps lose (batch 1 x
    // 6000: 11.13 -> 11.52 us, the doubled slices half empty), so they keep one block per CU.
    const int one = splits_for(1);
    const long lo_len = 3L * one * min_pos / 2, hi_len = 2L * one * min_pos;
    if (len > lo_len && len <= hi_len && 2 * one <= kMaxSplits &&
        (long)batch * nkv * 2 * one <= 2L * std::max(compute_units, 1))
        return 2 * one;
    return one;
}

size_t attention_partials_bytes(const AttnParams& p) {
    const int gsize = p.nkv > 0 ? p.nh / p.nkv : 1;
    const int G = group_pow2(gsize);
    return (size_t)p.batch * p.nkv * p.splits * partial_stride(G, p.head_dim) * sizeof(float);
}

int launch_attention_decode(hipStream_t s, const AttnParams& p) {
    return launch_any(s, p, 0, (size_t)p.max_seq_len * p.nkv * p.head_dim);
}

bool attention_prefill_tiled(const AttnParams& p) {
    return (p.head_dim == 64 || p.head_dim == 128) && p.nkv > 0 && p.nh % p.nkv == 0 && p.nh / p.nkv <= kPrefillGroup &&
           (p.cache_dtype == L0H_F16 || p.cache_dtype == L0H_F32) && (p.q_dtype == L0H_F16 || p.q_dtype == L0H_F32);
}

// Prefill: the query-tiled kernel where it applies; otherwise token t of the chunk is batch entry t
// with length pos0 + t + 1 over the shared cache (the split decode kernel).
int launch_attention_prefill(hipStream_t s, AttnParams p, int pos0, int tokens) {
    if (tokens < 1 || pos0 < 0 || pos0 + tokens > p.max_seq_len)
        return fail(L0H_ERR_INVALID_ARG, "prefill chunk outside the cache");
    if (attention_prefill_tiled(p)) {
        if ((((uintptr_t)p.q | (uintptr_t)p.kc | (uintptr_t)p.vc) & 15) != 0)
            return fail(L0H_ERR_INVALID_ARG, "attention buffers must be 16-byte aligned");
        return p.head_dim == 64 ? launch_prefill_hd<64>(s, p, pos0, tokens) : launch_prefill_hd<128>(s, p, pos0, tokens);
    }
    return launch_attention_tokens(s, p, pos0, tokens);
}

int launch_attention_tokens(hipStream_t s, AttnParams p, int pos0, int tokens) {
    p.batch = tokens;
    p.seq_len = pos0 + 1;
    p.seq_len_device = nullptr;
    return launch_any(s, p, 1, 0);
}

}  // namespace l0h
