// Backward of the fused causal attention for heads of 64 and 128 on the bf16
// matrix cores: every operand as the exact sum of three bf16 values, six
// products each (gemm_split.hip), f32 sums. The products, the masks and the
// layouts of attention_bwd.hip (which says what they replace):
//
//   dq:  S^T = K.Q^T, dP^T = V.dO^T, dS^T = P^T (dP^T - D), dQ^T += K^T.dS^T
//   dkv: S = Q.K^T, dP = dO.V^T, dV^T += dO^T.P, dK^T += Q^T.dS
//
// A workgroup of 8 waves owns 128 rows (queries for dq, keys for dkv) in four
// strips of 32. The two waves of a strip (one SIMD) take the two score-like
// products, so each holds the pieces of one stationary operand only (96
// registers at heads of 128): wave 0 of dkv forms P and accumulates dV, wave 1
// forms dP and, with P through LDS, dS and dK; in dq both get dS from each
// other's half and each accumulates half of dQ's columns.
//
// The streamed operands lie in LDS once, as rows (16-byte units of 8 head
// columns); where a product needs them transposed (K^T, dO^T, Q^T) the
// operand is read with the transposing LDS read: within 16 lanes, lane l
// element e of ds_read_tr16_b64 is element l%4 of what lane 4e + l/4 points at,
// so lanes that point at 4 rows x 16 columns get a column of 4 rows each. Its
// rows come in the order the accumulators hold them (lane half h: 16b + 4h +
// 0..3, then 16b + 8 + 4h + 0..3), so dS and P cross no lanes.
//
// What bounds it: the matrix cores at the clock their power leaves them, then
// the VALU: per 32x32 tile and wave at heads of 128, 96 MFMAs (dkv) or 72 (dq)
// beside about 330 VALU instructions. Whole backward with its forward, fp32
// matrix cores against this: B4 12/12 T1000 heads of 64 308 / 197 us; B4 16/8
// T1024 heads of 128 604 / 457 (these kernels 344: 175 TFLOP/s of the seven
// products they form); B1 16/8 T2048 heads of 128 980 / 590 (256 blocks, one
// per CU: the longest of them); B1 32/32 T4096 heads of 64 2198 / 1580.
//
// Every operand is lifted by 2^24 before it is split (mmh_split.h), so that
// small values keep every bit. P carries its factor into dS; the scores and
// dP lose theirs in the subtraction that follows, the sums at the end. (Before,
// the largest and smallest magnitudes were followed to redo such strips: B4
// 12/12 T1000 heads of 64, with the forward, 205.6 us then, 198.3 now, B1 16/8
// T2048 heads of 128 598 / 592.)
//
// A wave with a sum that is not finite (values beyond the lift among them), and
// every wave of a workgroup with a log-sum-exp beyond 2^79, whose scores the
// lift could take to -inf, does its strip again in plain f32.
#include "mmh_attention.h"
#include "mmh_split.h"

#include <algorithm>

namespace mmh {
namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef short shortx4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) shortx4 *lds_shortx4;

constexpr float kLog2e = 1.4426950408889634f;
// log-sum-exps from here on: scores near them may not fit the lift
constexpr float kLargeLse = 0x1p79f;

__device__ __forceinline__ float swap32_sum(float v) {
    auto c = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(c[0]) + __uint_as_float(c[1]);
}
// Over lanes l, l^16, l^32, l^48.
__device__ __forceinline__ float quad_sum(float v) {
    auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return swap32_sum(__uint_as_float(a[0]) + __uint_as_float(a[1]));
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_all(const float *base) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(base), (short)0, 0x7fffffff, 0x00020000);
}

// LDS places of 32 rows x HD columns in three pieces: planes of 8 columns, 32
// units of 16 bytes each, 48 bytes apart beyond that (neighbouring lanes write
// a row's planes, and read 4-row parts of two planes).
template <int HD>
struct RowTile {
    static constexpr int PK = 32 * 16 + 48;
    static constexpr int PIECE = HD / 8 * PK, BYTES = 3 * PIECE;
    static constexpr int E = HD / 16;  // values per thread (512 threads: row tid/16)
};

// Two 4-row halves of a transposed operand: 8 of its k for the lane's column.
__device__ __forceinline__ bf16x8 read_tr(const char *lds, int at) {
    const shortx4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4)(lds + at));
    const shortx4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_shortx4)(lds + at + 128));
    bf16x8 r;
    __builtin_memcpy(&r, &lo, 8);
    __builtin_memcpy(reinterpret_cast<char *>(&r) + 8, &hi, 8);
    return r;
}

#define MMH_MFMA(a, b, c) c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0)

// Rows of the tile times the stationary operand's pieces w (the lane's row of
// it, columns 16s + 8*(lane/32) .. +7): out[r] is tile row 8*(r/4) + 4*(lane/32)
// + r%4 against the lane's, lifted twice.
template <int HD>
__device__ __forceinline__ void rows_product(const char *tile, const bf16x8 (&w)[3][HD / 16],
                                             float (&out)[16]) {
    using R = RowTile<HD>;
    const int lane = threadIdx.x & 63;
    const char *src = tile + (lane >> 5) * R::PK + (lane & 31) * 16;
    floatx16 s0, s1;
#pragma unroll
    for (int r = 0; r < 16; ++r) s0[r] = s1[r] = 0.0f;
#pragma unroll
    for (int s = 0; s < HD / 16; ++s) {
        const bf16x8 h = *reinterpret_cast<const bf16x8 *>(src + 2 * s * R::PK);
        const bf16x8 m = *reinterpret_cast<const bf16x8 *>(src + 2 * s * R::PK + R::PIECE);
        const bf16x8 l = *reinterpret_cast<const bf16x8 *>(src + 2 * s * R::PK + 2 * R::PIECE);
        MMH_MFMA(h, w[0][s], s0);
        MMH_MFMA(h, w[1][s], s1);
        MMH_MFMA(m, w[0][s], s0);
        MMH_MFMA(m, w[1][s], s1);
        MMH_MFMA(h, w[2][s], s0);
        MMH_MFMA(l, w[0][s], s1);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) out[r] = s0[r] + s1[r];
}

// acc += columns [32*db0, 32*(db0 + N)) of the tile, transposed, times x (an
// accumulator-ordered 32-row column per lane, lifted).
template <int HD, int N>
__device__ __forceinline__ void cols_product(const char *tile, int db0, const float (&x)[16],
                                             floatx16 (&acc)[N]) {
    using R = RowTile<HD>;
    const int lane = threadIdx.x & 63;
    const int at = (2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) * R::PK +
                   (4 * (lane >> 5) + ((lane & 15) >> 2)) * 16 + (lane & 1) * 8 + db0 * 4 * R::PK;
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] = x[8 * kb + e];
        uint32_t w[3][4];
        split_values(v, w);
        bf16x8 xh, xm, xl;
        __builtin_memcpy(&xh, w[0], 16);
        __builtin_memcpy(&xm, w[1], 16);
        __builtin_memcpy(&xl, w[2], 16);
        constexpr int G = N >= 2 ? 2 : 1;
#pragma unroll
        for (int db = 0; db < N; db += G) {
            bf16x8 h[G], m[G], l[G];
#pragma unroll
            for (int j = 0; j < G; ++j) {
                const int a = at + (db + j) * 4 * R::PK + kb * 256;
                h[j] = read_tr(tile, a);
                m[j] = read_tr(tile, a + R::PIECE);
                l[j] = read_tr(tile, a + 2 * R::PIECE);
            }
#pragma unroll
            for (int j = 0; j < G; ++j) MMH_MFMA(h[j], xh, acc[db + j]);
#pragma unroll
            for (int j = 0; j < G; ++j) MMH_MFMA(h[j], xm, acc[db + j]);
#pragma unroll
            for (int j = 0; j < G; ++j) MMH_MFMA(m[j], xh, acc[db + j]);
#pragma unroll
            for (int j = 0; j < G; ++j) MMH_MFMA(m[j], xm, acc[db + j]);
#pragma unroll
            for (int j = 0; j < G; ++j) MMH_MFMA(h[j], xl, acc[db + j]);
#pragma unroll
            for (int j = 0; j < G; ++j) MMH_MFMA(l[j], xh, acc[db + j]);
        }
    }
}
#undef MMH_MFMA

// The pieces of a stationary row (times f, lifted).
template <int HD>
__device__ __forceinline__ void load_pieces(const float *row, float f, bf16x8 (&w)[3][HD / 16]) {
    const float *src = row + 8 * ((threadIdx.x & 63) >> 5);
#pragma unroll
    for (int s = 0; s < HD / 16; ++s) {
        float v[8];
        __builtin_memcpy(v, __builtin_assume_aligned(src + 16 * s, 16), 32);
#pragma unroll
        for (int e = 0; e < 8; ++e) v[e] *= f * kLift;
        uint32_t o[3][4];
        split_values(v, o);
#pragma unroll
        for (int i = 0; i < 3; ++i) __builtin_memcpy(&w[i][s], o[i], 16);
    }
}

template <int E>
__device__ __forceinline__ void load_values(float (&v)[E], __amdgpu_buffer_rsrc_t r, uint32_t off) {
#pragma unroll
    for (int e = 0; e < E; e += 4) {
        const float4 x = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(r, off + 4 * e, 0, 0));
        v[e] = x.x;
        v[e + 1] = x.y;
        v[e + 2] = x.z;
        v[e + 3] = x.w;
    }
}
template <int HD>
__device__ __forceinline__ void put_values(char *tile, const float (&v)[HD / 16]) {
    using R = RowTile<HD>;
    const int row = threadIdx.x / 16, col = threadIdx.x % 16 * R::E;
    uint32_t o[3][R::E / 2];
    lift_and_split(v, o);
#pragma unroll
    for (int i = 0; i < 3; ++i)
        __builtin_memcpy(__builtin_assume_aligned(tile + i * R::PIECE + col / 8 * R::PK + row * 16 + col % 8 * 2,
                                                  2 * R::E),
                         o[i], 2 * R::E);
}

// Whether one of the wave's sums is not finite.
template <int N>
__device__ __forceinline__ bool wave_redo(const floatx16 (&acc)[N]) {
    float nf = 0.0f;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) nf = __builtin_fmaf(acc[i][r], 0.0f, nf);
    return __any(!(nf == 0.0f));
}

// Strips in plain f32: four lanes (l, l^16, l^32, l^48) share a row, each with a
// quarter of the head's columns.
template <int HD>
__device__ __noinline__ void exact_dq(const float *q, const float *k, const float *v, const float *o,
                                      const float *dout, const float *lse, float *dq, int64_t sqt,
                                      int64_t skt, int64_t svt, int64_t sot, float scale, int q0,
                                      int T) {
    constexpr int C = HD / 4;
    const int lane = threadIdx.x & 63, c0 = (lane >> 4) * C;
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
        const int qi = q0 + 16 * h + (lane & 15), qc = min(qi, T - 1);
        float qr[C], g[C], acc[C], d = 0.0f;
#pragma unroll
        for (int c = 0; c < C; ++c) {
            qr[c] = q[qc * sqt + c0 + c] * (scale * kLog2e);
            g[c] = dout[qc * sot + c0 + c];
            d += g[c] * o[qc * sot + c0 + c];
            acc[c] = 0.0f;
        }
        d = quad_sum(d);
        const float L = lse[qc];
        const int last = min(q0 + 16 * h + 15, T - 1);
#pragma unroll 1
        for (int key = 0; key <= last; ++key) {
            const float *kr = k + key * skt + c0, *vr = v + key * svt + c0;
            float s = 0.0f, dp = 0.0f;
#pragma unroll
            for (int c = 0; c < C; ++c) {
                s += qr[c] * kr[c];
                dp += g[c] * vr[c];
            }
            s = quad_sum(s);
            dp = quad_sum(dp);
            if (key <= qi) {
                const float ds = __builtin_amdgcn_exp2f(s - L) * (dp - d);
#pragma unroll
                for (int c = 0; c < C; ++c) acc[c] += ds * kr[c];
            }
        }
        if (qi < T)
#pragma unroll
            for (int c = 0; c < C; ++c) dq[qi * sqt + c0 + c] = acc[c] * scale;
    }
}
// q, dout, lse, dvec at the first head of ng; out: dK (want_dk) or dV rows.
template <int HD>
__device__ __noinline__ void exact_dkv(const float *q, const float *k, const float *v,
                                       const float *dout, const float *lse, const float *dvec,
                                       float *out, int64_t sqh, int64_t sqt, int64_t skt,
                                       int64_t svt, int64_t soh, int64_t sot, int64_t out_t,
                                       float scale, int k0, int T, int ng, bool want_dk) {
    constexpr int C = HD / 4;
    const int lane = threadIdx.x & 63, c0 = (lane >> 4) * C;
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
        const int kj = k0 + 16 * h + (lane & 15), kc = min(kj, T - 1);
        float kr[C], vr[C], acc[C];
#pragma unroll
        for (int c = 0; c < C; ++c) {
            kr[c] = k[kc * skt + c0 + c] * (scale * kLog2e);
            vr[c] = v[kc * svt + c0 + c];
            acc[c] = 0.0f;
        }
#pragma unroll 1
        for (int g = 0; g < ng; ++g)
#pragma unroll 1
            for (int qi = min(k0 + 16 * h, T - 1); qi < T; ++qi) {
                const float *qr = q + g * sqh + qi * sqt + c0, *gr = dout + g * soh + qi * sot + c0;
                float s = 0.0f, dp = 0.0f;
#pragma unroll
                for (int c = 0; c < C; ++c) {
                    s += kr[c] * qr[c];
                    dp += vr[c] * gr[c];
                }
                s = quad_sum(s);
                dp = quad_sum(dp);
                if (kj > qi) continue;
                const float pr = __builtin_amdgcn_exp2f(s - lse[(int64_t)g * T + qi]);
                const float ds = pr * (dp - dvec[(int64_t)g * T + qi]);
#pragma unroll
                for (int c = 0; c < C; ++c) acc[c] += want_dk ? ds * qr[c] : pr * gr[c];
            }
        if (kj < T)
#pragma unroll
            for (int c = 0; c < C; ++c) out[kj * out_t + c0 + c] = acc[c] * (want_dk ? scale : 1.0f);
    }
}

template <int HD>
__global__ __launch_bounds__(512, 2) void attn_bwd_dq_x3_kernel(BwdP p) {
    using R = RowTile<HD>;
    constexpr int E = R::E, N = HD / 64;  // row blocks of dQ^T per wave
    constexpr int EX = 8 * 4 * 64 * 16;   // each wave's 16 values per lane
    __shared__ __attribute__((aligned(128))) char lds[2 * 2 * R::BYTES + EX];
    float4(*ex)[4][64] = reinterpret_cast<float4(*)[4][64]>(lds + 4 * R::BYTES);

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int lq = lane & 31, lh = lane >> 5, strip = wave & 3, role = wave >> 2;
    const int head = blockIdx.x, b = blockIdx.y;
    const int qblk = p.nqb - 1 - (int)blockIdx.z;  // longest rows first
    const int kvh = head / (p.h / p.hkv);
    const int T = p.t;
    const int ntiles = min(qblk * 128 + 127, T - 1) / 32 + 1;
    const int q0 = qblk * 128 + strip * 32;
    const int my_tiles = q0 < T ? min(q0 + 31, T - 1) / 32 + 1 : 0;
    const int qi = q0 + lq, qc = min(qi, T - 1);

    const float *Q = p.q + b * p.sqb + head * p.sqh;
    const float *K = p.k + b * p.skb + kvh * p.skh;
    const float *V = p.v + b * p.svb + kvh * p.svh;
    const float *O = p.o + b * p.sob + head * p.soh;
    const float *dO = p.dout + b * p.sob + head * p.soh;
    const int64_t rows = ((int64_t)b * p.h + head) * T;

    bool large = false;  // a log-sum-exp beyond kLargeLse
    // role 0: the query's row and its log-sum-exp; role 1: dO's row and D
    bf16x8 w[3][HD / 16];
    load_pieces<HD>(role ? dO + (int64_t)qc * p.sot : Q + (int64_t)qc * p.sqt,
                    role ? 1.0f : p.scale * kLog2e, w);
    float shift;
    if (role) {
        float d = 0.0f;
        const float *g = dO + (int64_t)qc * p.sot + lh * (HD / 2), *o = O + (int64_t)qc * p.sot + lh * (HD / 2);
#pragma unroll
        for (int c = 0; c < HD / 2; c += 4) {
            const float4 x = *reinterpret_cast<const float4 *>(g + c), y = *reinterpret_cast<const float4 *>(o + c);
            d += x.x * y.x + x.y * y.y + x.z * y.z + x.w * y.w;
        }
        shift = swap32_sum(d);
        if (lh == 0 && qi < T) p.dvec[rows + qi] = shift;
    } else {
        shift = p.lse[rows + qc];
        large = fabsf(shift) > kLargeLse;
    }

    // thread tid moves E columns of row tid/16 of the K and of the V tile (keys
    // past T read row T-1: finite values whose P is 0)
    const __amdgpu_buffer_rsrc_t rk = rsrc_all(K), rv = rsrc_all(V);
    const uint32_t skt4 = 4u * (uint32_t)p.skt, svt4 = 4u * (uint32_t)p.svt;
    float kr[E], vr[E];
    auto load = [&](int kt) __attribute__((always_inline)) {
        const uint32_t key = (uint32_t)min(min(kt, ntiles - 1) * 32 + tid / 16, T - 1), c = 4u * (tid % 16 * E);
        load_values(kr, rk, key * skt4 + c);
        load_values(vr, rv, key * svt4 + c);
    };
    auto put = [&](int buf) __attribute__((always_inline)) {
        put_values<HD>(lds + buf * 2 * R::BYTES, kr);
        put_values<HD>(lds + buf * 2 * R::BYTES + R::BYTES, vr);
    };

    floatx16 acc[N];
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;

    load(0);
    put(0);
    load(1);
    __syncthreads();
    // Two phases a tile: each wave's product of the rows, its values to the
    // other; then dS and the wave's half of dQ's columns. The next tile is
    // written into the other buffer (last read a tile ago) by role 1 at the
    // start of the first phase and by role 0 at the start of the second, so that
    // a SIMD's waves split values beside each other's MFMAs; the loads of the
    // one after it have a phase or more to arrive.
    for (int kt = 0; kt < ntiles; ++kt) {
        const int buf = kt & 1, k0 = kt * 32;
        const char *kt_lds = lds + buf * 2 * R::BYTES;
        const bool mine = kt < my_tiles;
        if (role) put(buf ^ 1);
        float x[16];
        if (mine) {
            rows_product<HD>(kt_lds + role * R::BYTES, w, x);
            if (role == 0) {
                if (!(k0 + 31 <= q0 && k0 + 31 < T)) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int key = k0 + 8 * (r >> 2) + 4 * lh + (r & 3);
                        x[r] = key <= qi && key < T ? x[r] : -INFINITY;
                    }
                }
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    x[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(x[r], kUnlift2, -shift)) * kLift;
            } else {
#pragma unroll
                for (int r = 0; r < 16; ++r) x[r] = __builtin_fmaf(x[r], kUnlift2, -shift);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i)
                ex[wave][i][lane] = make_float4(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]);
        }
        __syncthreads();
        if (!role) put(buf ^ 1);
        load(kt + 2);
        if (mine) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 y = ex[wave ^ 4][i][lane];
                x[4 * i] *= y.x;
                x[4 * i + 1] *= y.y;
                x[4 * i + 2] *= y.z;
                x[4 * i + 3] *= y.w;
            }
            cols_product<HD, N>(kt_lds, role * N, x, acc);
        }
        __syncthreads();
    }

    const bool redo_all = __syncthreads_or(large);
    const bool redo = my_tiles && (wave_redo(acc) || redo_all);
    float *dq = p.dq + b * p.sqb + head * p.sqh;
    const float f = p.scale * kUnlift2;
    if (qi < T) {
        float *row = dq + (int64_t)qi * p.sqt + role * (HD / 2) + 4 * lh;
#pragma unroll
        for (int i = 0; i < N; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *reinterpret_cast<float4 *>(row + 32 * i + 8 * j) =
                    make_float4(acc[i][4 * j] * f, acc[i][4 * j + 1] * f, acc[i][4 * j + 2] * f,
                                acc[i][4 * j + 3] * f);
    }
    // (either wave of the strip redoes all of its columns: both write the same
    // values then, after both have stored theirs)
    int *flags = reinterpret_cast<int *>(lds);
    if (lane == 0) flags[wave] = redo;
    __builtin_amdgcn_s_waitcnt(0);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    if (role == 0 && (flags[wave] | flags[wave ^ 4]))
        exact_dq<HD>(Q, K, V, O, dO, p.lse + rows, dq, p.sqt, p.skt, p.svt, p.sot, p.scale, q0, T);
}

template <int HD>
__global__ __launch_bounds__(512, 2) void attn_bwd_dkv_x3_kernel(BwdP p) {
    using R = RowTile<HD>;
    constexpr int E = R::E, N = HD / 32;
    constexpr int BUF = 2 * R::BYTES + 256;  // Q rows, dO rows, lse[32], D[32]
    __shared__ __attribute__((aligned(128))) char lds[2 * BUF + 4 * 4 * 64 * 16];
    float4(*ex)[4][64] = reinterpret_cast<float4(*)[4][64]>(lds + 2 * BUF);

    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int lq = lane & 31, lh = lane >> 5, strip = wave & 3, role = wave >> 2;
    const int groups = p.h / p.hkv;
    const int kvh = p.part ? (int)blockIdx.x / groups : (int)blockIdx.x;
    const int head0 = p.part ? (int)blockIdx.x : kvh * groups;
    const int ng = p.part ? 1 : groups;
    const int b = blockIdx.y;
    const int T = p.t;
    const int k_first = (int)blockIdx.z * 128;  // block 0 sees the most queries and starts first
    const int k0 = k_first + strip * 32;
    const int kj = k0 + lq, kc = min(kj, T - 1);
    const int qt_first = k_first / 32, qt_end = (T + 31) / 32;
    const int my_first = k0 / 32;  // earlier query tiles lie wholly above these keys

    const float *K = p.k + b * p.skb + kvh * p.skh;
    const float *V = p.v + b * p.svb + kvh * p.svh;
    const float *Q = p.q + b * p.sqb + head0 * p.sqh;
    const float *dO = p.dout + b * p.sob + head0 * p.soh;
    const int64_t rows = ((int64_t)b * p.h + head0) * T;

    bool large = false;  // a log-sum-exp beyond kLargeLse
    bf16x8 w[3][HD / 16];  // role 0: the key's row of K, role 1: of V
    load_pieces<HD>(role ? V + (int64_t)kc * p.svt : K + (int64_t)kc * p.skt,
                    role ? 1.0f : p.scale * kLog2e, w);

    const __amdgpu_buffer_rsrc_t rq = rsrc_all(Q), rg = rsrc_all(dO);
    const uint32_t sqt4 = 4u * (uint32_t)p.sqt, sot4 = 4u * (uint32_t)p.sot;
    const uint32_t sqh4 = 4u * (uint32_t)p.sqh, soh4 = 4u * (uint32_t)p.soh;
    float qr[E], gr[E], lv = 0.0f;
    // the walk over (head of the group, query tile): the tile being loaded
    // (which stops at the last one) and the one being used
    int lg = 0, lt = qt_first;
    auto load = [&]() __attribute__((always_inline)) {
        const uint32_t row = (uint32_t)min(lt * 32 + tid / 16, T - 1), c = 4u * (tid % 16 * E);
        load_values(qr, rq, (uint32_t)lg * sqh4 + row * sqt4 + c);
        load_values(gr, rg, (uint32_t)lg * soh4 + row * sot4 + c);
        if (tid < 64)
            lv = (tid < 32 ? p.lse : p.dvec)[rows + (int64_t)lg * T + min(lt * 32 + (tid & 31), T - 1)];
        if (lt + 1 < qt_end) {
            ++lt;
        } else if (lg + 1 < ng) {
            ++lg;
            lt = qt_first;
        }
    };
    auto put = [&](int buf) __attribute__((always_inline)) {
        put_values<HD>(lds + buf * BUF, qr);
        put_values<HD>(lds + buf * BUF + R::BYTES, gr);
        if (tid < 64) {
            reinterpret_cast<float *>(lds + buf * BUF + 2 * R::BYTES)[tid] = lv;
            large |= tid < 32 && fabsf(lv) > kLargeLse;
        }
    };

    floatx16 acc[N];  // role 0: dV^T, role 1: dK^T
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][r] = 0.0f;

    load();
    put(0);
    load();
    __syncthreads();
    // Two phases a tile, as in dq: P and dP - D; then dV from P, and dK from dS
    // with the other wave's P.
    const int total = ng * (qt_end - qt_first);
    int qt = qt_first;
    for (int it = 0; it < total; ++it) {
        const int buf = it & 1, i0 = qt * 32;
        const char *tile = lds + buf * BUF;
        const bool mine = qt >= my_first;
        if (role) put(buf ^ 1);
        float x[16];
        if (mine) {
            rows_product<HD>(tile + role * R::BYTES, w, x);
            const float4 *shift = reinterpret_cast<const float4 *>(tile + 2 * R::BYTES + role * 128);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 y = shift[2 * i + lh];
                x[4 * i] = __builtin_fmaf(x[4 * i], kUnlift2, -y.x);
                x[4 * i + 1] = __builtin_fmaf(x[4 * i + 1], kUnlift2, -y.y);
                x[4 * i + 2] = __builtin_fmaf(x[4 * i + 2], kUnlift2, -y.z);
                x[4 * i + 3] = __builtin_fmaf(x[4 * i + 3], kUnlift2, -y.w);
            }
            if (role == 0) {
                if (!(i0 >= k0 + 31 && i0 + 31 < T)) {
#pragma unroll
                    for (int r = 0; r < 16; ++r) {
                        const int qi = i0 + 8 * (r >> 2) + 4 * lh + (r & 3);
                        x[r] = kj <= qi && qi < T ? x[r] : -INFINITY;
                    }
                }
#pragma unroll
                for (int r = 0; r < 16; ++r) x[r] = __builtin_amdgcn_exp2f(x[r]) * kLift;
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    ex[strip][i][lane] = make_float4(x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]);
            }
        }
        __syncthreads();
        if (!role) put(buf ^ 1);
        load();
        if (mine) {
            if (role) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 y = ex[strip][i][lane];
                    x[4 * i] *= y.x;
                    x[4 * i + 1] *= y.y;
                    x[4 * i + 2] *= y.z;
                    x[4 * i + 3] *= y.w;
                }
            }
            cols_product<HD, N>(tile + (1 - role) * R::BYTES, 0, x, acc);
        }
        qt = qt + 1 < qt_end ? qt + 1 : qt_first;
        __syncthreads();
    }

    const bool redo_all = __syncthreads_or(large);
    if (k0 >= T) return;
    float *out;
    int64_t out_t;
    if (p.part) {
        out = p.part + ((int64_t)b * p.h + head0) * T * HD + (role ? 0 : (int64_t)gridDim.y * p.h * T * HD);
        out_t = HD;
    } else {
        out = role ? p.dk + b * p.skb + kvh * p.skh : p.dv + b * p.svb + kvh * p.svh;
        out_t = role ? p.skt : p.svt;
    }
    if (wave_redo(acc) || redo_all) {
        exact_dkv<HD>(Q, K, V, dO, p.lse + rows, p.dvec + rows, out, p.sqh, p.sqt, p.skt, p.svt,
                      p.soh, p.sot, out_t, p.scale, k0, T, ng, role != 0);
        return;
    }
    if (kj >= T) return;
    const float f = role ? p.scale * kUnlift2 : kUnlift2;
    float *row = out + (int64_t)kj * out_t + 4 * lh;
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            *reinterpret_cast<float4 *>(row + 32 * i + 8 * j) =
                make_float4(acc[i][4 * j] * f, acc[i][4 * j + 1] * f, acc[i][4 * j + 2] * f,
                            acc[i][4 * j + 3] * f);
}

template <int HD>
void launch_hd(Context &ctx, const BwdP &p, int64_t b) {
    const dim3 gq((unsigned)p.h, (unsigned)b, (unsigned)p.nqb);
    const dim3 gk((unsigned)(p.part ? p.h : p.hkv), (unsigned)b, (unsigned)p.nkb);
    hipLaunchKernelGGL((attn_bwd_dq_x3_kernel<HD>), gq, dim3(512), 0, ctx.stream, p);
    hipLaunchKernelGGL((attn_bwd_dkv_x3_kernel<HD>), gk, dim3(512), 0, ctx.stream, p);
}

}  // namespace

void launch_attention_bwd_split(Context &ctx, const BwdP &p, int64_t b, int64_t hd) {
    if (hd == 64) launch_hd<64>(ctx, p, b);
    else launch_hd<128>(ctx, p, b);
}

}  // namespace mmh
