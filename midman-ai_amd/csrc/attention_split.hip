// Fused causal attention for heads of 64 and 128 on the bf16 matrix cores:
// Q, K, V and P as exact sums of three bf16 values (gemm_split.hip says why),
// six products each for S = Q.K^T and O = P.V, f32 sums and softmax.
//
// Replaces the reference's materialised path (midman-nn/src/attention.rs:79-101,
// 146-170) like attention.hip's kernels. A workgroup of 8 waves owns 128 query
// rows of one (batch, head), blocks with the longest rows first; waves w and
// w + 4 (one SIMD) share a strip of 32 rows, one taking the even 32-key tiles
// and one the odd ones, each with its own online softmax, and their sums meet
// in LDS at the end: every SIMD has two busy waves for the whole block.
//
// K and V are walked 64 keys at a time. Each thread holds f32 values, splits
// them and writes the pieces in the layout that the MFMA operands are read in
// (16 bytes per lane). As in attention.hip the products are transposed, so a
// query stays in its two lanes (l and l^32): S^T = K.Q^T, then O^T += V^T.P^T
// with P's pieces straight from the S^T accumulators: lane half h holds keys
// 16b + 4h + 0..3 and 16b + 8 + 4h + 0..3 of each 16, so V's operand puts its
// keys in that order and no P crosses lanes. RoPE and the mask are
// attention.hip's.
//
// What bounds it: the chip's power and the VALU. For 32 queries x 32 keys at
// heads of 128 a wave runs 96 MFMAs beside about 540 VALU instructions (260
// for its share of K's and V's pieces, 150 for P's, the softmax) and reads 48
// KB of LDS; matrix cores and VALU are each busy about 45% of the cycles.
// Measured (f32 MFMA kernel before -> now): B4 H16/8 T1024 hd128 159 -> 120-124
// us = 140 TFLOP/s, B1 H16/8 T2048 hd128 264 -> 136-146, B4 H12 T1000 hd64 82 ->
// 48-54, B8 H16/8 T1024 hd64 167 -> 122-131. Before the key halves, with a
// long and a short block of 128 rows on each SIMD (the f32 kernel's way), the
// long block's wave ran alone most of the time: 136 us at hd128.
//
// Q, V and P are lifted by 2^24 before they are split (mmh_split.h), so that
// their small values keep every bit: a probability of 2^-120 beside a value of
// 2^110 can be a whole output. Q's factor goes into its scale and out of the
// scores in the exponential's subtraction, V's and P's into the final division;
// V and P take a multiply per value: 0-2% of the time (B4 H16/8 T1024 hd128 108.6
// -> 110.9 us, B8 H16/8 T192 hd64 14.2 -> 14.3). (K is split as it is: a piece of it
// below bf16's normal range moves a score by at most 2^-126 times the query,
// which no query up to 2^80 shows.)
//
// A wave whose sums are not finite (values beyond the lift among them), and
// every wave of a workgroup with a query above 2^80, does its strip again in
// plain f32, one key at a time.
#include "mmh_attention.h"
#include "mmh_split.h"

#include <algorithm>
#include <type_traits>

namespace mmh {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr float kLog2e = 1.4426950408889634f;

__device__ __forceinline__ float swap_max(float v) {
    auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return fmaxf(__uint_as_float(c[0]), __uint_as_float(c[1]));
}
__device__ __forceinline__ float swap_sum(float v) {
    auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(c[0]) + __uint_as_float(c[1]);
}

// One strip of 32 query rows in plain f32: lanes l and l^32 share query l%32,
// each with half of the head's columns.
template <int HD>
__device__ __noinline__ void exact_strip(const float *Q, const float *K, const float *V,
                                         float *out, float *lse, int64_t sqt, int64_t skt,
                                         int64_t svt, int64_t sot, float sc, int q0, int T) {
    // (the parameters one by one: a reference to the launch's would put them
    // all in memory for the caller as well)
    constexpr int HH = HD / 2;
    const int lane = threadIdx.x & 63, lq = lane & 31, lh = lane >> 5;
    const int qi = q0 + lq;
    float q[HH], acc[HH];
    const float *qrow = Q + (int64_t)min(qi, T - 1) * sqt + lh * HH;
#pragma unroll
    for (int c = 0; c < HH; ++c) {
        q[c] = qrow[c] * sc;
        acc[c] = 0.0f;
    }
    float m = -INFINITY, l = 0.0f;
    const int last = min(q0 + 31, T - 1);
#pragma unroll 1
    for (int key = 0; key <= last; ++key) {
        const float *krow = K + (int64_t)key * skt + lh * HH, *vrow = V + (int64_t)key * svt + lh * HH;
        float s = 0.0f;
#pragma unroll
        for (int c = 0; c < HH; ++c) s += q[c] * krow[c];
        s = swap_sum(s);
        if (key <= qi) {
            // scores of -inf before the row's first other one have weight 0 (a
            // row of nothing else is NaN, as inf - inf makes it)
            const bool none = m == -INFINITY && s == -INFINITY && key < qi;
            const float m_new = fmaxf(m, s);
            const float alpha = none ? 1.0f : __builtin_amdgcn_exp2f(m - m_new);
            const float e = none ? 0.0f : __builtin_amdgcn_exp2f(s - m_new);
            l = l * alpha + e;
#pragma unroll
            for (int c = 0; c < HH; ++c) acc[c] = acc[c] * alpha + e * vrow[c];
            m = m_new;
        }
    }
    if (qi >= T) return;
    const float inv = 1.0f / l;
    float *orow = out + (int64_t)qi * sot + lh * HH;
#pragma unroll
    for (int c = 0; c < HH; ++c) orow[c] = acc[c] * inv;
    if (lse && lh == 0) lse[qi] = m + log2f(l);
}

template <int HD>
__global__ __launch_bounds__(512, 2) void attn_fwd_x3_kernel(AttnP p) {
    static_assert(HD == 64 || HD == 128, "heads of 64 or 128");
    constexpr int NT = 512, QB = 128;
    constexpr int NS = HD / 16, NDB = HD / 32;  // S^T k-steps, O^T row blocks
    constexpr int E = 32 * HD / NT;             // values of K and of V per thread and tile
    // K: per piece HD/8 planes (8 head columns each) of 32 keys x 16 bytes, 16
    // bytes apart beyond that (a key's planes are written by neighbouring
    // lanes); V: per piece 4 planes (16 keys and lane half) of HD columns.
    constexpr int PK = 32 * 16 + 16, PV = HD * 16;
    constexpr int SK = HD / 8 * PK, SV = 4 * PV;
    constexpr int OS = HD + 4;  // row stride of the merged sums
    constexpr int STAGE = 2 * 3 * (SK + SV), MERGE = 4 * 32 * OS * 4 + 4 * 64 * 8;
    __shared__ __attribute__((aligned(128))) char lds[STAGE > MERGE ? STAGE : MERGE];

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int lq = lane & 31, lh = lane >> 5;
    const int strip = wave & 3, par = wave >> 2;
    const int head = blockIdx.x, b = blockIdx.y;
    const int qblk = p.nqb - 1 - (int)blockIdx.z;  // longest rows first
    const int kvh = head / (p.h / p.hkv);
    const int T = p.t;
    const int nsteps = min(qblk * QB + QB - 1, T - 1) / 64 + 1;  // of 64 keys
    const int q0 = qblk * QB + strip * 32;
    const int my_tiles = q0 < T ? min(q0 + 31, T - 1) / 32 + 1 : 0;
    const int qi = q0 + lq;

    const float *Q = p.q + b * p.sqb + head * p.sqh;
    const float *K = p.k + b * p.skb + kvh * p.skh;
    const float *V = p.v + b * p.svb + kvh * p.svh;

    // B operand of S^T: the lane's query, head columns 16s + 8*lh .. +7, scaled
    // into log2 units and lifted
    const float sc = p.scale * kLog2e;
    bf16x8 qp[3][NS];
    float big = 0.0f;
    {
        const float *src = Q + (int64_t)min(qi, T - 1) * p.sqt + 8 * lh;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            float v[8];
            __builtin_memcpy(v, __builtin_assume_aligned(src + 16 * s, 16), 32);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                v[e] *= sc * kLift;
                big = fmaxf(big, fabsf(v[e]));
            }
            uint32_t o[3][4];
            split_values(v, o);
#pragma unroll
            for (int i = 0; i < 3; ++i) __builtin_memcpy(&qp[i][s], o[i], 16);
        }
    }

    // This thread's share of a tile: of K, E head columns of key kkey; of V, E
    // keys (in the order above) of column vcol. Buffer loads over the
    // sequence's T rows: keys past T read zeros (their scores are masked).
    const int kkey = tid / (HD / E), kcol = tid % (HD / E) * E;
    const int vcol = tid % HD, vunit = __builtin_amdgcn_readfirstlane(tid / HD);
    // unit: 16-key block, lane half and, for E = 4, which four of its keys
    const int vblk = E == 8 ? vunit >> 1 : vunit >> 2, vhalf = E == 8 ? vunit & 1 : (vunit >> 1) & 1;
    const int vsub = E == 8 ? 0 : vunit & 1;
    const __amdgpu_buffer_rsrc_t rk = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(K), (short)0, (int)(4 * (int64_t)T * p.skt), 0x00020000);
    const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float *>(V), (short)0, (int)(4 * (int64_t)T * p.svt), 0x00020000);
    const uint32_t krow = 4u * (uint32_t)p.skt, vrow = 4u * (uint32_t)p.svt;
    const uint32_t ko = (uint32_t)kkey * krow + 4u * (uint32_t)kcol;
    const uint32_t vo = (uint32_t)(16 * vblk + 8 * vsub + 4 * vhalf) * vrow + 4u * (uint32_t)vcol;
    const int kw = kcol / 8 * PK + kkey * 16 + kcol % 8 * 2;
    const int vw = 2 * 3 * SK + (2 * vblk + vhalf) * PV + vcol * 16 + vsub * 8;
    // the 64 keys of a step as two tiles of 32
    float st[2][E];
    auto load_k = [&](int step) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < E; e += 4) {
                const float4 x = __builtin_bit_cast(
                    float4, __builtin_amdgcn_raw_buffer_load_b128(
                                rk, ko + (uint32_t)(step * 64 + 32 * u) * krow + 4 * e, 0, 0));
                st[u][e] = x.x;
                st[u][e + 1] = x.y;
                st[u][e + 2] = x.z;
                st[u][e + 3] = x.w;
            }
    };
    auto load_v = [&](int step) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int e = 0; e < E; ++e)
                st[u][e] = __builtin_bit_cast(
                    float, __builtin_amdgcn_raw_buffer_load_b32(
                               rv, vo + (uint32_t)(step * 64 + 32 * u + 8 * (e >> 2) + (e & 3)) * vrow, 0, 0));
    };
    auto put = [&](auto lift, int at, int tile, int piece) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            uint32_t o[3][E / 2];
            if constexpr (decltype(lift)::value) lift_and_split(st[u], o);
            else split_values(st[u], o);
#pragma unroll
            for (int i = 0; i < 3; ++i)
                __builtin_memcpy(__builtin_assume_aligned(lds + u * tile + i * piece + at, 2 * E), o[i], 2 * E);
        }
    };

    floatx16 o[NDB];
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[db][r] = 0.0f;
    float m_run = -INFINITY, l_run = 0.0f;
    float pv[16];

#define MMH_MFMA(a, b, c) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0)
    auto scores = [&](int kt) __attribute__((always_inline)) {
        floatx16 s0, s1;
#pragma unroll
        for (int r = 0; r < 16; ++r) s0[r] = s1[r] = 0.0f;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const char *src = lds + par * 3 * SK + (2 * s + lh) * PK + lq * 16;
            const bf16x8 kh = *reinterpret_cast<const bf16x8 *>(src);
            const bf16x8 km = *reinterpret_cast<const bf16x8 *>(src + SK);
            const bf16x8 kl = *reinterpret_cast<const bf16x8 *>(src + 2 * SK);
            MMH_MFMA(kh, qp[0][s], s0);
            MMH_MFMA(kh, qp[1][s], s1);
            MMH_MFMA(km, qp[0][s], s0);
            MMH_MFMA(km, qp[1][s], s1);
            MMH_MFMA(kh, qp[2][s], s0);
            MMH_MFMA(kl, qp[0][s], s1);
        }
        const int k0 = kt * 32;
#pragma unroll
        for (int r = 0; r < 16; ++r) pv[r] = s0[r] + s1[r];
        if (!(k0 + 31 <= q0 && k0 + 31 < T)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = k0 + 8 * (r >> 2) + 4 * lh + (r & 3);
                pv[r] = key <= qi && key < T ? pv[r] : -INFINITY;
            }
        }
        float mloc = pv[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mloc = fmaxf(mloc, pv[r]);
        mloc = swap_max(mloc) * kUnlift;
        const bool need = mloc > m_run + 8.0f;  // lazy rescale, as attn_fwd_kernel
        if (__any(need)) {
            const float m_new = need ? mloc : m_run;
            const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (int db = 0; db < NDB; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[db][r] *= alpha;
            m_run = m_new;
        }
        float lsum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            pv[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(pv[r], kUnlift, -m_run));
            lsum += pv[r];
        }
        l_run += lsum;  // the lane's own keys; its partner's are added at the end
    };
    auto apply = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = pv[8 * kb + e];
            uint32_t w[3][4];
            lift_and_split(x, w);
            bf16x8 ph, pm, pl;
            __builtin_memcpy(&ph, w[0], 16);
            __builtin_memcpy(&pm, w[1], 16);
            __builtin_memcpy(&pl, w[2], 16);
            const char *src = lds + 2 * 3 * SK + par * 3 * SV + (2 * kb + lh) * PV + lq * 16;
#pragma unroll
            for (int db = 0; db < NDB; db += 2) {
                bf16x8 vh[2], vm[2], vl[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    vh[j] = *reinterpret_cast<const bf16x8 *>(src + (db + j) * 512);
                    vm[j] = *reinterpret_cast<const bf16x8 *>(src + (db + j) * 512 + SV);
                    vl[j] = *reinterpret_cast<const bf16x8 *>(src + (db + j) * 512 + 2 * SV);
                }
#pragma unroll
                for (int j = 0; j < 2; ++j) MMH_MFMA(vh[j], ph, o[db + j]);
#pragma unroll
                for (int j = 0; j < 2; ++j) MMH_MFMA(vh[j], pm, o[db + j]);
#pragma unroll
                for (int j = 0; j < 2; ++j) MMH_MFMA(vm[j], ph, o[db + j]);
#pragma unroll
                for (int j = 0; j < 2; ++j) MMH_MFMA(vm[j], pm, o[db + j]);
#pragma unroll
                for (int j = 0; j < 2; ++j) MMH_MFMA(vh[j], pl, o[db + j]);
#pragma unroll
                for (int j = 0; j < 2; ++j) MMH_MFMA(vl[j], ph, o[db + j]);
            }
        }
    };
#undef MMH_MFMA

    load_k(0);
    put(std::false_type(), kw, 3 * SK, SK);
    load_v(0);
    __syncthreads();
    // A step of 64 keys has two phases with one copy of K and of V in LDS: in
    // the first the waves form scores from K while V is written, in the second
    // they apply V while the next step's K is written; each operand's global
    // loads go out a phase ahead. The two waves of a SIMD write at opposite
    // ends of a phase, so one splits values while the other's MFMAs run.
    for (int step = 0; step < nsteps; ++step) {
        const int kt = 2 * step + par, next = min(step + 1, nsteps - 1);
        const bool mine = kt < my_tiles;
        if (par) {
            put(std::true_type(), vw, 3 * SV, SV);
            load_k(next);
        }
        if (mine) scores(kt);
        if (!par) {
            put(std::true_type(), vw, 3 * SV, SV);
            load_k(next);
        }
        __syncthreads();
        if (par) {
            put(std::false_type(), kw, 3 * SK, SK);
            load_v(next);
        }
        if (mine) apply();
        if (!par) {
            put(std::false_type(), kw, 3 * SK, SK);
            load_v(next);
        }
        __syncthreads();
    }

    // the strip's two halves of the keys meet in LDS, odd tiles' sums first
    const bool redo_all = __syncthreads_or(big > 0x1p80f * kLift);
    float *sums = reinterpret_cast<float *>(lds) + strip * 32 * OS;
    float2 *ml = reinterpret_cast<float2 *>(lds + 4 * 32 * OS * 4) + strip * 64;
    if (par) {
        ml[lane] = make_float2(m_run, l_run);
#pragma unroll
        for (int db = 0; db < NDB; ++db)
#pragma unroll
            for (int i = 0; i < 4; ++i)
                *reinterpret_cast<float4 *>(sums + lq * OS + 32 * db + 8 * i + 4 * lh) =
                    make_float4(o[db][4 * i], o[db][4 * i + 1], o[db][4 * i + 2], o[db][4 * i + 3]);
    }
    __syncthreads();
    if (par || my_tiles == 0) return;
    const float2 other = ml[lane];
    // (a strip of one tile has nothing in the other half: m = -inf, l = 0)
    const float m = fmaxf(m_run, other.x);
    const float wa = __builtin_amdgcn_exp2f(m_run - m), wb = __builtin_amdgcn_exp2f(other.x - m);
    const float l = swap_sum(l_run * wa + other.y * wb);
    float nf = __builtin_fmaf(l, 0.0f, m * 0.0f);  // NaN once anything is not finite
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 x = *reinterpret_cast<const float4 *>(sums + lq * OS + 32 * db + 8 * i + 4 * lh);
            o[db][4 * i] = o[db][4 * i] * wa + x.x * wb;
            o[db][4 * i + 1] = o[db][4 * i + 1] * wa + x.y * wb;
            o[db][4 * i + 2] = o[db][4 * i + 2] * wa + x.z * wb;
            o[db][4 * i + 3] = o[db][4 * i + 3] * wa + x.w * wb;
        }
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int r = 0; r < 16; ++r) nf = __builtin_fmaf(o[db][r], 0.0f, nf);
    float *out = p.out + b * p.sob + head * p.soh;
    float *lse = p.lse ? p.lse + ((int64_t)b * p.h + head) * T : nullptr;
    if (redo_all || __any(!(nf == 0.0f))) {
        exact_strip<HD>(Q, K, V, out, lse, p.sqt, p.skt, p.svt, p.sot, sc, q0, T);
        return;
    }
    if (qi >= T) return;
    const float inv = kUnlift2 / l;
    float *orow = out + (int64_t)qi * p.sot + 4 * lh;
#pragma unroll
    for (int db = 0; db < NDB; ++db)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            *reinterpret_cast<float4 *>(orow + 32 * db + 8 * i) =
                make_float4(o[db][4 * i] * inv, o[db][4 * i + 1] * inv, o[db][4 * i + 2] * inv,
                            o[db][4 * i + 3] * inv);
    if (lse && lh == 0) lse[qi] = m + log2f(l);
}

}  // namespace

void launch_attention_split(Context &ctx, const AttnP &p, int64_t b, int64_t hd) {
    const dim3 grid((unsigned)p.h, (unsigned)b, (unsigned)p.nqb);
    if (hd == 64)
        hipLaunchKernelGGL((attn_fwd_x3_kernel<64>), grid, dim3(512), 0, ctx.stream, p);
    else
        hipLaunchKernelGGL((attn_fwd_x3_kernel<128>), grid, dim3(512), 0, ctx.stream, p);
}

}  // namespace mmh
