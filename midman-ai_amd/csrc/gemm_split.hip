// fp32 GEMM on the bf16 matrix cores: every f32 operand as the exact sum of
// three bf16 values, six of the nine products, f32 accumulation.
//
// C = A.B (nn), A.B^T (nt), A^T.B (tn), replacing the reference's CPU kernels
// (midman-tensor/src/kernels.rs:49-108, kernels_avx.rs:45-250) for every
// product with enough 128x128 tiles of work; the small shapes are in gemm.hip.
//
// Why not the fp32 MFMA: it runs at 1/16 of the bf16 rate on gfx950 (157
// against 2500 TFLOP/s). x = h + m + l with h = bf16(x), m = bf16(x - h),
// l = x - h - m holds all 24 bits of x (each step's remainder is exact in f32
// and the third fits bf16's 8 bits), so nothing of the inputs is rounded away.
// Of a.b = (h + m + l)(h' + m' + l') the products hh', hm', mh', mm', hl', lh'
// are formed (exact in the matrix core, summed in f32); the three left out
// are below 2^-24 |a b|. Measured against 64-bit sums, N(0,1) x N(0,0.02), on
// the 256x256 tiles: relative error 1.34e-7 / 5.0e-7 / 6.9e-7 / 1.42e-6 at K = 64 /
// 1024 / 2048 / 8192, where the fp32 MFMA's own sums give 1.49e-7 / 5.7e-7 /
// 8.1e-7 / 1.62e-6: a 32x32x16 step rounds the sum six times per 16 products,
// the fp32 32x32x2 step eight times. The other tiles round it once (LOW below):
// about a third of that.
//
// The operands are lifted by 2^24 first (mmh_split.h), a multiply per value, so
// that small values need no second look. Following the smallest magnitude
// instead, to redo the tiles of values below 2^-102, took more (4096 x 4096 x
// 2048 332 us, 323 so) and made such operands four to eight times slower (4096 x
// 2048 x 8192 nt 597 -> 4800 us).
//
// What the split cannot hold is found and redone with the fp32 MFMA, tile by
// tile, so special values follow the scalar rules bit for bit:
//   - inf, NaN, |x| from 2^104 on (the lift, mmh_split.h) and sums from 2^80 on
//     leave a non-finite accumulator (inf - inf in the remainders);
//   - an exact zero where the sum must keep the sign of -0 (acc_init is -0).
//
// Tiling: a wave owns MB x 2 blocks of 32x32 (MB 4: 128x64, 2: 64x64, 1:
// 32x64); a workgroup 256x256 or 256x128 (8 waves), 128x128 or 128x64 (two
// groups of 4 waves) or 64x64 (four groups of 2). The groups take the K-steps
// of 16 in turn, with LDS stages and accumulators of their own, and their sums
// meet in LDS: a small tile then still puts two waves on every SIMD, where one
// alone waits out its own LDS writes, barrier and reads (2048 x 512 x 1024 on
// 128x64 tiles: 22.8 -> 20.9 us; 4096 x 1024 x 1024 on 128x128: 61.8 -> 53.6).
// K advances through two LDS stages. Each thread reads its f32 values a step
// ahead into registers, splits them and writes the three pieces as up to 8
// consecutive k (16 bytes) of one row or column, the layout the MFMA operands
// are read in; an operand stored k-major is read down k by each lane, so the
// transpose costs nothing. Within a step the products run in the order hh, hm,
// mh, mm, one MFMA and a few of the VALU instructions that split the next
// step's values in turn (unordered, the compiler put the split first and the
// 128x128 tile ran 4-8% slower); then, behind the step's one barrier and the
// next step's first operand reads, hl and lh, so no wave waits on LDS right
// after the barrier.
//
// What bounds it: the chip's power. With zero operands the 256x256 tile runs
// at 310-323 TFLOP/s, with normal values at 216-237 over four boxes (the clock
// falls as operand bits toggle); bf16 MFMAs alone, no memory or LDS traffic,
// reach 1730-1770 TFLOP/s = 290 in f32 terms, and 1600 with the VALU work of
// the splits beside them. Measured at 4096 x 4096 x 2048: 256x256 311 us = 221
// TFLOP/s, 256x128 333 us, 128x128 375 us (more LDS reads and splits per
// product); the fp32 MFMA kernel before it 471 us = 146 (before the lift; 2-3%
// less since).
//
// MFMA 32x32x16 bf16 layout (wave64): lane l supplies A[i = l%32][k = 8*(l/32)
// .. +7] and B[k = 8*(l/32) .. +7][j = l%32]; accumulator register r of lane l
// holds D[i = 8*(r/4) + 4*(l/32) + r%4][j = l%32].
//
// Workgroup -> tile mapping is XCD-aware: the dispatcher hands workgroup w to
// XCD w % 8, so w is renumbered to make each XCD's share a contiguous run of
// tiles, walked in groups of tile rows so that the tiles an XCD holds at once
// share A rows and B columns in its L2.
#include "mmh_gemm.h"
#include "mmh_split.h"

#include <algorithm>

namespace mmh {
namespace {

// Reductions over each 32-lane half of a wave with DPP moves (quad permutes,
// then rotations within a 16-lane row) and one v_permlane16_swap across the
// two rows of the half (a VALU exchange: no trip through the LDS unit). For
// the max every lane ends with the result; for the sum the lanes associate the
// terms differently, and lane 0 of the half (the one read) always the same way.
__device__ __forceinline__ float dpp_f(float v, int ctrl) {
    switch (ctrl) {
        case 0xB1: return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));
        case 0x4E: return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false));
        case 0x124: return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x124, 0xF, 0xF, false));
        default: return __builtin_bit_cast(float, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, v), 0x128, 0xF, 0xF, false));
    }
}
// The pair {v[l], v[l ^ 16]} in each lane l (in some order).
__device__ __forceinline__ auto pair16_f(float v) {
    return __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
}
__device__ __forceinline__ float half_max32(float v) {
    v = fmaxf(v, dpp_f(v, 0xB1));   // quad_perm [1,0,3,2]
    v = fmaxf(v, dpp_f(v, 0x4E));   // quad_perm [2,3,0,1]
    v = fmaxf(v, dpp_f(v, 0x124));  // row_ror:4
    v = fmaxf(v, dpp_f(v, 0x128));  // row_ror:8
    const auto q = pair16_f(v);
    return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float half_sum32(float v) {
    v += dpp_f(v, 0xB1);
    v += dpp_f(v, 0x4E);
    v += dpp_f(v, 0x124);
    v += dpp_f(v, 0x128);
    const auto q = pair16_f(v);
    return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

// Tile t of the grouped order: group tile rows at a time, column by column.
__device__ __forceinline__ void grouped_tile(const KParams &p, int group, int t, int &tm, int &tn) {
    const int per_group = group * p.tiles_n;
    const int g = t / per_group;
    const int first_m = g * group;
    const int gsize = min(p.tiles_m - first_m, group);
    const int in_group = t - g * per_group;
    tm = first_m + in_group % gsize;
    tn = in_group / gsize;
}
constexpr int group_rows(int tile_m) { return 1024 / tile_m; }

// Column layouts (CL) of a wave's two 32-column blocks: 0 the even and the odd
// columns of its 64 (a lane then holds column pairs), 1 its two halves of 32,
// 2 columns c and c + 64 of a 128-column unit, so that the RoPE pair (c,
// c + hd/2) of a head of 64 (CL 1) or 128 (CL 2) columns sits in one lane.
// Column `col` of the tile is column j of block i of wave column g:
template <int CL>
__device__ __forceinline__ void col_place(int col, int &g, int &i, int &j) {
    if (CL == 0) {
        g = col >> 6;
        i = col & 1;
        j = (col >> 1) & 31;
    } else if (CL == 1) {
        g = col >> 6;
        i = (col >> 5) & 1;
        j = col & 31;
    } else {
        g = ((col >> 7) << 1) | ((col >> 5) & 1);
        i = (col >> 6) & 1;
        j = col & 31;
    }
}
template <int CL>
__device__ __forceinline__ int place_col(int g, int i, int j) {
    if (CL == 0) return g * 64 + 2 * j + i;
    if (CL == 1) return g * 64 + i * 32 + j;
    return (g >> 1) * 128 + i * 64 + (g & 1) * 32 + j;
}

// LDS bytes of one operand's stage: per piece two planes (k 0-7 and 8-15) of
// one 16-byte unit per row or column. A's planes sit 64 bytes off a multiple
// of 128 so that a row's two units written by neighbouring lanes fall in
// different banks; B's column blocks are 64 bytes apart beyond their 512 (even
// and odd columns written by neighbouring lanes) and its planes 32 off.
constexpr int kBlockB = 512 + 64, kGroupB = 2 * 512 + 64;
constexpr int plane_a(int rows) { return rows * 16 + 64; }
constexpr int plane_b(int cols) {
    return cols / 64 * kGroupB + ((32 - cols / 64 * kGroupB % 128) + 128) % 128;
}

template <int WM, int WN, int MB>
struct TileShape {
    static constexpr int TM = WM * MB * 32, TN = WN * 64, NT = WM * WN * 64;  // NT: of one K group
    static constexpr int PA = plane_a(TM), PB = plane_b(TN);
    static constexpr int SA = 6 * PA, SB = 6 * PB, STAGE = SA + SB;
    // k values a thread moves together: 8, or 4 where the tile has fewer than
    // 8 values per thread
    static constexpr int EA = TM * BK / NT >= 8 ? 8 : 4, EB = TN * BK / NT >= 8 ? 8 : 4;
    static constexpr int UA = TM * BK / EA / NT, UB = TN * BK / EB / NT;
    static constexpr int VALU_PER_MFMA = ((TM + TN) * BK / NT * 15 / 2 + 16) / (8 * MB);
    static constexpr int DEPTH = MB == 1 ? 2 : 1;
    static_assert(UA >= 1 && UB >= 1, "a K-step must split evenly over the threads");
};

// One operand's share of a thread: UNITS units of E consecutive k of one row
// or column. KM: stored k-major (A of tn, B of nn and tn).
template <bool KM, int R, int E, int UNITS, int NT>
struct Loader {
    const float *ptr[UNITS];  // KM: unused; else the unit's first value at k = 0
    uint32_t off[UNITS];      // KM: the lane's row or column
    int kq[UNITS];            // k of the unit within a step
    const float *base;
    int64_t ld;

    __device__ __forceinline__ void init(const float *src, int64_t ld_, int64_t first,
                                         int64_t count, int tid) {
        base = src;
        ld = ld_;
#pragma unroll
        for (int i = 0; i < UNITS; ++i) {
            const int idx = tid + NT * i;
            // rows past the edge read the last one; their results are not stored
            if constexpr (KM) {
                // a wave's lanes share the k group: rows are a multiple of 64
                kq[i] = __builtin_amdgcn_readfirstlane(idx / R) * E;
                off[i] = (uint32_t)(min(first + idx % R, count - 1) - first);
            } else {
                kq[i] = idx % (BK / E) * E;
                ptr[i] = src + min(first + idx / (BK / E), count - 1) * ld + kq[i];
            }
        }
        if constexpr (KM) base = src + first;
    }
    // A step whose 16 values of k are all in range. Rows need only 4-byte
    // alignment: gfx950 reads 16 bytes at any dword.
    __device__ __forceinline__ void load(float (&v)[UNITS][E], int64_t k0) const {
#pragma unroll
        for (int i = 0; i < UNITS; ++i) {
            if constexpr (KM) {
                // the row in a scalar register pair (through an empty asm: the
                // compiler otherwise adds it into a 64-bit address per load),
                // the lane's column in one 32-bit offset
                const float *next = uniform(base + (k0 + kq[i]) * ld);
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const float *row = next;
                    asm("" : "+s"(row));
                    v[i][e] = row[off[i]];
                    next += ld;
                }
            } else {
                __builtin_memcpy(v[i], ptr[i] + k0, E * 4);
            }
        }
    }
    // The last step of a K that is no multiple of 16: zeros from kend on.
    __device__ __forceinline__ void load_tail(float (&v)[UNITS][E], int64_t k0, int64_t kend) const {
#pragma unroll
        for (int i = 0; i < UNITS; ++i)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int64_t k = k0 + kq[i] + e, kc = min(k, kend - 1);
                float x;
                if constexpr (KM)
                    x = (base + kc * ld)[off[i]];
                else
                    x = ptr[i][kc - kq[i]];
                v[i][e] = k < kend ? x : 0.0f;
            }
    }
};

// The K loop of one tile; the sums it leaves are lifted twice (kUnlift2).
// WK groups of WM x WN waves share a tile: group g takes the steps g, g + WK,
// ... into its own LDS stages and its own accumulators.
template <bool TA, bool TB, int CL, int WM, int WN, int MB, int WK>
__device__ __forceinline__ void split_mainloop(const KParams &p, const float *__restrict__ A,
                                               const float *__restrict__ B, int64_t m0,
                                               int64_t n0, int64_t kbeg, int64_t kend,
                                               char *lds, floatx16 (&acc)[MB][2]) {
    using S = TileShape<WM, WN, MB>;
    constexpr int TM = S::TM, TN = S::TN, NT = S::NT;
    const int group = WK == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    const int tid = threadIdx.x - group * NT, lane = tid & 63, wave = tid >> 6;
    const int wm = wave / WN, wn = wave % WN, lr = lane & 31, lk = lane >> 5;
    lds += group * (2 * S::STAGE);

    Loader<TA, TM, S::EA, S::UA, NT> la;
    Loader<!TB, TN, S::EB, S::UB, NT> lb;
    la.init(A, p.lda, m0, p.m, tid);
    lb.init(B, p.ldb, n0, p.n, tid);
    int wa[S::UA], wb[S::UB];  // the units' places in a stage
#pragma unroll
    for (int i = 0; i < S::UA; ++i) {
        const int idx = tid + NT * i;
        const int row = TA ? idx % TM : idx / (BK / S::EA);
        const int k = TA ? idx / TM * S::EA : idx % (BK / S::EA) * S::EA;
        wa[i] = k / 8 * S::PA + row * 16 + k % 8 * 2;
    }
#pragma unroll
    for (int i = 0; i < S::UB; ++i) {
        const int idx = tid + NT * i;
        const int col = TB ? idx / (BK / S::EB) : idx % TN;
        const int k = TB ? idx % (BK / S::EB) * S::EB : idx / TN * S::EB;
        int g, b, j;
        col_place<CL>(col, g, b, j);
        wb[i] = S::SA + k / 8 * S::PB + g * kGroupB + b * kBlockB + j * 16 + k % 8 * 2;
    }

    // Whole steps of each group; what is left over runs first: a last step
    // shorter than 16 on group 0, whole steps on the groups after it.
    const int whole = (int)((kend - kbeg) / BK), nk = whole / WK;
    constexpr int D = S::DEPTH;
    float ra[D][S::UA][S::EA], rb[D][S::UB][S::EB];
    auto load = [&](int slot, int t) __attribute__((always_inline)) {
        const int64_t k0 = kbeg + (int64_t)(min(t, nk - 1) * WK + group) * BK;
        la.load(ra[slot], k0);
        lb.load(rb[slot], k0);
    };
    auto put = [&](int buf, int slot) __attribute__((always_inline)) {
        char *stage = lds + buf * S::STAGE;
#pragma unroll
        for (int i = 0; i < S::UA; ++i) {
            uint32_t o[3][S::EA / 2];
            lift_and_split(ra[slot][i], o);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                __builtin_memcpy(__builtin_assume_aligned(stage + q * 2 * S::PA + wa[i], S::EA * 2),
                                 o[q], S::EA * 2);
        }
#pragma unroll
        for (int i = 0; i < S::UB; ++i) {
            uint32_t o[3][S::EB / 2];
            lift_and_split(rb[slot][i], o);
#pragma unroll
            for (int q = 0; q < 3; ++q)
                __builtin_memcpy(__builtin_assume_aligned(stage + q * 2 * S::PB + wb[i], S::EB * 2),
                                 o[q], S::EB * 2);
        }
    };

    // Operand reads of one piece: every block's 16 bytes per lane.
    const int fa = lk * S::PA + (wm * MB * 32 + lr) * 16;
    const int fb = S::SA + lk * S::PB + wn * kGroupB + lr * 16;
    auto read_a = [&](bf16x8 (&d)[MB], int buf, int q) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MB; ++i)
            d[i] = *reinterpret_cast<const bf16x8 *>(lds + buf * S::STAGE + q * 2 * S::PA + fa + i * 512);
    };
    auto read_b = [&](bf16x8 (&d)[2], int buf, int q) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < 2; ++j)
            d[j] = *reinterpret_cast<const bf16x8 *>(lds + buf * S::STAGE + q * 2 * S::PB + fb + j * kBlockB);
    };
    auto mul = [&](const bf16x8 (&a)[MB], const bf16x8 (&b)[2]) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], acc[i][j], 0, 0, 0);
    };
    // The five products below hh: on the tiles of one or two blocks per wave, whose
    // registers hold them, into sums of their own, added at the end. The large
    // sum then rounds once per 16 k instead of six times. Error against 64 bits at
    // K 16 / 64 / 256 8.2e-8 / 1.35e-7 / 2.5e-7 -> 3.2e-8 / 5.0e-8 / 9e-8 on the 256x128
    // tiles (the fp32 MFMA 7.4e-8 / 1.4e-7 / 1.2e-7 to 2.9e-7, by kernel), at
    // 1003 x 1517 x 770 (tn) 3.07e-7 -> 1.16e-7; times 0-2% longer.
    constexpr bool LOW = MB <= 2;
    floatx16 low[LOW ? MB : 1][2];
    auto mul_low = [&](const bf16x8 (&a)[MB], const bf16x8 (&b)[2]) __attribute__((always_inline)) {
        if constexpr (LOW) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    low[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[i], b[j], low[i][j], 0, 0, 0);
        } else {
            mul(a, b);
        }
    };
    auto add_low = [&]() __attribute__((always_inline)) {
        if constexpr (LOW) {
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) acc[i][j][r] += low[i][j][r];
        }
    };
    if constexpr (LOW) {
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) low[i][j][r] = 0.0f;
    }

#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    // When step t starts, stage t%2 holds step t, ah and bh its first pieces,
    // and register slot (t+1)%D step t+1's values (the loads of D steps in
    // flight; two for the small tiles, whose steps are shorter than a load).
    // Stage (t+1)%2 was last read in step t-1, before its barrier. Loads past
    // the last step repeat it, unread. The scheduling fences keep the order
    // described at the top of the file.
    bf16x8 ah[MB], am[MB], al[MB], bh[2], bm[2], bl[2];
    const int64_t kwhole = kbeg + (int64_t)whole * BK;
    if (kwhole < kend || whole % WK != 0) {
        const bool mine = group == 0 ? kwhole < kend : group <= whole % WK;
        if (mine) {
            if (group == 0) {
                la.load_tail(ra[0], kwhole, kend);
                lb.load_tail(rb[0], kwhole, kend);
            } else {
                const int64_t k0 = kwhole - (int64_t)group * BK;
                la.load(ra[0], k0);
                lb.load(rb[0], k0);
            }
            put(0, 0);
        }
        __syncthreads();
        if (mine) {
            // (all nine products, the smallest first: a K below 16 ends with one
            // rounding at the size of its sum, as a product of two f32 should)
            read_b(bl, 0, 2);
            read_a(al, 0, 2);
            read_a(ah, 0, 0);
            read_b(bh, 0, 0);
            read_b(bm, 0, 1);
            read_a(am, 0, 1);
            mul_low(al, bl);
            mul_low(am, bl);
            mul_low(al, bm);
            mul_low(ah, bl);
            mul_low(al, bh);
            mul_low(am, bm);
            mul_low(ah, bm);
            mul_low(am, bh);
            mul(ah, bh);
        }
        __syncthreads();
    }
    if (nk <= 0) {
        add_low();
        return;
    }
    auto step = [&](auto uc, int t) __attribute__((always_inline)) {
        constexpr int u = decltype(uc)::value, buf = u % 2, slot = (u + 1) % D;
        read_b(bm, buf, 1);
        read_a(am, buf, 1);
        read_b(bl, buf, 2);
        read_a(al, buf, 2);
        __builtin_amdgcn_sched_barrier(0);
        mul(ah, bh);
        put(buf ^ 1, slot);
        load(slot, t + 1 + D);
        mul_low(ah, bm);
        mul_low(am, bh);
        mul_low(am, bm);
        unroll_seq([&](auto) __attribute__((always_inline)) {
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x2, S::VALU_PER_MFMA, 0);
        }, std::make_integer_sequence<int, 8 * MB>{});
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_sched_barrier(0);
        bf16x8 nah[MB], nbh[2];
        read_a(nah, buf ^ 1, 0);
        read_b(nbh, buf ^ 1, 0);
        __builtin_amdgcn_sched_barrier(0);
        mul_low(ah, bl);
        mul_low(al, bh);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < MB; ++i) ah[i] = nah[i];
        bh[0] = nbh[0];
        bh[1] = nbh[1];
    };
    load(0, 0);
    put(0, 0);
    unroll_seq([&](auto jc) __attribute__((always_inline)) {
        constexpr int j = decltype(jc)::value + 1;
        load(j % D, j);
    }, std::make_integer_sequence<int, D>{});
    __syncthreads();
    read_a(ah, 0, 0);
    read_b(bh, 0, 0);
    constexpr int U = D % 2 == 0 ? D : 2 * D;  // the period of (stage, slot)
    int t = 0;
    for (; t + U <= nk; t += U)
        unroll_seq([&](auto uc) __attribute__((always_inline)) { step(uc, t + uc); },
                   std::make_integer_sequence<int, U>{});
    unroll_seq([&](auto uc) __attribute__((always_inline)) {
        if (t + uc < nk) step(uc, t + uc);
    }, std::make_integer_sequence<int, U>{});
    add_low();
}

// The tile again on the fp32 MFMA, operands straight from memory: for the
// values the split does not hold (see the top of the file). MFMA 32x32x2 f32:
// lane l supplies A[l%32][k = l/32] and B[k = l/32][l%32]; same accumulator
// layout. Values past K are -0 (A) and +0 (B), whose product -0 is the
// identity of IEEE addition.
template <bool TA, bool TB, int CL, int WM, int WN, int MB>
__device__ __forceinline__ void exact_mainloop(const KParams &p, const float *__restrict__ A,
                                               const float *__restrict__ B, int64_t m0,
                                               int64_t n0, int64_t kbeg, int64_t kend,
                                               floatx16 (&acc)[MB][2]) {
    // (called by group 0)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave / WN, wn = wave % WN, lr = lane & 31, lk = lane >> 5;
    const float *pa[MB], *pb[2];
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        const int64_t row = min(m0 + (wm * MB + i) * 32 + lr, p.m - 1);
        pa[i] = TA ? A + row : A + row * p.lda;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int64_t col = min(n0 + place_col<CL>(wn, j, lr), p.n - 1);
        pb[j] = TB ? B + col * p.ldb : B + col;
    }
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = p.acc_init;
    const int64_t sa = TA ? p.lda : 1, sb = TB ? 1 : p.ldb;
#pragma unroll 1
    for (int64_t k0 = kbeg; k0 < kend; k0 += 4) {
        float a[MB][2], b[2][2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int64_t k = k0 + 2 * e + lk, kc = min(k, kend - 1);
#pragma unroll
            for (int i = 0; i < MB; ++i) a[i][e] = pa[i][kc * sa];
#pragma unroll
            for (int j = 0; j < 2; ++j) b[j][e] = pb[j][kc * sb];
            if (k >= kend) {
#pragma unroll
                for (int i = 0; i < MB; ++i) a[i][e] = -0.0f;
                b[0][e] = b[1][e] = 0.0f;
            }
        }
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i][e], b[j][e], acc[i][j], 0, 0, 0);
    }
}

// Two 32-column blocks of accumulators of the 32 rows from rb of a tile, through
// the epilogue: register r of lane l is row rb + 8*(r/4) + 4*(l/32) + r%4.
template <int EPI, int CL, int TM, int TN>
__device__ __forceinline__ void block_epilogue(const KParams &p, const floatx16 &a0,
                                               const floatx16 &a1, int split,
                                               int64_t batch, int64_t m0, int64_t n0, int rb,
                                               int wn, int lr, int lk) {
    const int64_t M = p.m, N = p.n;
    const int64_t col = n0 + wn * 64 + 2 * lr;
    auto row_local = [&](int r) __attribute__((always_inline)) {
        return rb + 8 * (r >> 2) + 4 * lk + (r & 3);
    };
    if constexpr (CL != 0) {
        // Column block j of lane lr is column c0 + j*half of C (half = 32 for
        // CL 1, 64 for CL 2), c0 the lane's column in the first half of its
        // head: RoPE (rope.rs:28-32) rotates the pair in registers, with the
        // rope kernel's arithmetic, on the q and k heads (columns below
        // rope_cols); the v heads are stored as they are.
        constexpr int half = CL == 1 ? 32 : 64;
        const int hc = CL == 1 ? lr : (wn & 1) * 32 + lr;
        const int64_t c0 = n0 + place_col<CL>(wn, 0, lr);
        const bool rot = p.rope_cos != nullptr && c0 < p.rope_cols;
        float *C = p.c + batch * p.stride_c;
        // The rows' table values are all read before the first store: the
        // compiler cannot tell the tables from C, so a read placed after a
        // store waits for that store's completion (one memory round trip per
        // row). Rows past M read a valid table row (row % seq) and are dropped.
        // Positions: the lane's first row modulo the sequence once; register
        // r adds 8*(r/4) + r%4 < 28 to it, at most one wrap when seq >= 28.
        float cs[16], sn[16];
        if (rot) {
            const uint32_t seq = (uint32_t)p.rope_seq;
            const uint32_t base = (uint32_t)((m0 + row_local(0)) % p.rope_seq);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                uint32_t pos = base + (uint32_t)(8 * (r >> 2) + (r & 3));
                if (seq < 28) pos %= seq;
                else if (pos >= seq) pos -= seq;
                const uint32_t t = pos * (uint32_t)half + (uint32_t)hc;
                cs[r] = p.rope_cos[t];
                sn[r] = p.rope_sin[t];
            }
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t row = m0 + row_local(r);
            if (row >= M) continue;
            float x1 = a0[r], x2 = a1[r];
            if (rot) {
                const float y1 = x1 * cs[r] - x2 * sn[r];
                const float y2 = x2 * cs[r] + x1 * sn[r];
                x1 = y1;
                x2 = y2;
            }
            if (c0 < N) C[row * p.ldc + c0] = x1;
            if (c0 + half < N) C[row * p.ldc + c0 + half] = x2;
        }
        return;
    }
    if (p.splits > 1) {
        // (summed by splitk_reduce: a tile's 2-16 partials are too much for
        // one workgroup of the launch to add up at the end)
        float *P = p.partial + (int64_t)split * M * N;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t row = m0 + row_local(r);
            if (row < M) {
                if (col < N) P[row * N + col] = a0[r];
                if (col + 1 < N) P[row * N + col + 1] = a1[r];
            }
        }
        return;
    }
    float *C = p.c + batch * p.stride_c;
    if (EPI == EPI_SWIGLU) {
        // Packed columns interleave gate and up: column 2f is gate f, 2f+1 up f.
        const int64_t f = col >> 1;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t row = m0 + row_local(r);
            if (row >= M) continue;
            if (p.aux && col + 1 < N)
                *reinterpret_cast<float2 *>(p.aux + row * p.ldaux + col) =
                    make_float2(a0[r], a1[r]);
            if (f < p.swiglu_ff) C[row * p.ldc + f] = __fmul_rn(p.libm_exp ? silu_f(a0[r]) : silu_fast(a0[r]), a1[r]);
        }
        return;
    }
    // The epilogues that read memory (the saved gate/up pairs, the residual)
    // issue their reads ahead of their stores, 8 or 16 rows at a time: the
    // destination may be the buffer read (in-place gradients, C += ...), so
    // the compiler may not move a read past a store and would otherwise wait
    // out one memory latency per row. Each lane reads only the elements it
    // writes, so the early reads see the same values.
    if (EPI == EPI_SWIGLU_BWD) {
        // acc is dh[row][col, col+1]; their (g, u) pairs sit at aux columns
        // 2*col .. 2*col+3 and the (dg, du) pairs go to the same columns of C.
        if (m0 + TM <= M && n0 + TN <= N && p.ldc < (int64_t(1) << 20) &&
            p.ldaux < (int64_t(1) << 20)) {
            // The whole tile in range: unconditional buffer accesses from the
            // tile's first row (see the residual epilogue below), eight rows'
            // pairs read before their eight stores.
            const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(p.aux + m0 * p.ldaux), (short)0, kBufferRange, kBufferFlags);
            const __amdgpu_buffer_rsrc_t rc =
                __builtin_amdgcn_make_buffer_rsrc(C + m0 * p.ldc, (short)0, kBufferRange, kBufferFlags);
            const uint32_t la = 4u * (uint32_t)p.ldaux, lc = 4u * (uint32_t)p.ldc;
            const uint32_t va = (uint32_t)row_local(0) * la + 8u * (uint32_t)col;
            const uint32_t vc = (uint32_t)row_local(0) * lc + 8u * (uint32_t)col;
#pragma unroll
            for (int r0 = 0; r0 < 16; r0 += 8) {
                float4 g[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int r = r0 + j;
                    g[j] = __builtin_bit_cast(float4, __builtin_amdgcn_raw_buffer_load_b128(
                                                          ra, va + (8 * (r >> 2) + (r & 3)) * la, 0, 0));
                }
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int r = r0 + j;
                    const float2 a = swiglu_bwd_f(a0[r], g[j].x, g[j].y);
                    const float2 b2 = swiglu_bwd_f(a1[r], g[j].z, g[j].w);
                    __builtin_amdgcn_raw_buffer_store_b128(
                        __builtin_bit_cast(u32x4_t, make_float4(a.x, a.y, b2.x, b2.y)), rc,
                        vc + (8 * (r >> 2) + (r & 3)) * lc, 0, 0);
                }
            }
            return;
        }
#pragma unroll
        for (int r0 = 0; r0 < 16; r0 += 8) {
            float4 g[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int64_t row = m0 + row_local(r0 + j);
                g[j] = row < M && col + 1 < N
                           ? *reinterpret_cast<const float4 *>(p.aux + row * p.ldaux + 2 * col)
                           : make_float4(0.f, 0.f, 0.f, 0.f);
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const int r = r0 + j;
                const int64_t row = m0 + row_local(r);
                if (row >= M) continue;
                float *dst = C + row * p.ldc + 2 * col;
                if (col + 1 < N) {
                    const float2 a = swiglu_bwd_f(a0[r], g[j].x, g[j].y);
                    const float2 b2 = swiglu_bwd_f(a1[r], g[j].z, g[j].w);
                    *reinterpret_cast<float4 *>(dst) = make_float4(a.x, a.y, b2.x, b2.y);
                } else if (col < N) {
                    const float *gu = p.aux + row * p.ldaux + 2 * col;
                    const float2 a = swiglu_bwd_f(a0[r], gu[0], gu[1]);
                    dst[0] = a.x;
                    dst[1] = a.y;
                }
            }
        }
        return;
    }
    const float *R = p.resid ? p.resid + batch * p.stride_c : C;
    const bool pair = p.vec_c && col + 1 < N;
    if (EPI == EPI_ACCUM && pair) {
        float2 o[16];
        if (m0 + TM <= M && p.ldc < (int64_t(1) << 21)) {
            // Every row in range: no per-row branches, so the compiler counts
            // the reads exactly and each store waits only for its own read
            // (with the reads and stores under row tests, every store waited
            // for all earlier stores as well: one store round trip per row).
            // Buffer accesses from the tile's first row with 32-bit offsets
            // (64-bit addresses for 16 rows took the kernel past the registers
            // of four waves per SIMD). Each row's offset is added into the
            // lane offset, never passed as the scalar offset: with computed
            // scalar offsets the compiler reused an SGPR that a v_div_scale
            // had just written as its carry-out, and one row of a tile read
            // another row's values (found by the tail-pieces training test).
            const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(R + m0 * p.ldc), (short)0, kBufferRange, kBufferFlags);
            const __amdgpu_buffer_rsrc_t rc =
                __builtin_amdgcn_make_buffer_rsrc(C + m0 * p.ldc, (short)0, kBufferRange, kBufferFlags);
            const uint32_t ldb4 = 4u * (uint32_t)p.ldc;
            const uint32_t vo = (uint32_t)row_local(0) * ldb4 + 4u * (uint32_t)col;
#pragma unroll
            for (int r = 0; r < 16; ++r)
                o[r] = __builtin_bit_cast(
                    float2, __builtin_amdgcn_raw_buffer_load_b64(rr, vo + (8 * (r >> 2) + (r & 3)) * ldb4, 0, 0));
#pragma unroll
            for (int r = 0; r < 16; ++r)
                __builtin_amdgcn_raw_buffer_store_b64(
                    __builtin_bit_cast(u32x2_t, make_float2(__fadd_rn(o[r].x, a0[r]),
                                                            __fadd_rn(o[r].y, a1[r]))),
                    rc, vo + (8 * (r >> 2) + (r & 3)) * ldb4, 0, 0);
            return;
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t row = m0 + row_local(r);
            o[r] = row < M ? *reinterpret_cast<const float2 *>(R + row * p.ldc + col)
                           : make_float2(0.f, 0.f);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t row = m0 + row_local(r);
            if (row >= M) continue;
            *reinterpret_cast<float2 *>(C + row * p.ldc + col) =
                make_float2(__fadd_rn(o[r].x, a0[r]), __fadd_rn(o[r].y, a1[r]));
        }
        return;
    }
    // Single columns (odd rows of C, or the last column). Their reads go out ahead
    // as well, sixteen at a time, from columns and rows held in range.
    if (EPI == EPI_ACCUM) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float *src = R + min(col + j, N - 1);
            float o[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) o[r] = src[min(m0 + row_local(r), M - 1) * p.ldc];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int64_t row = m0 + row_local(r);
                if (row < M && col + j < N)
                    C[row * p.ldc + col + j] = __fadd_rn(o[r], j ? a1[r] : a0[r]);
            }
        }
        return;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int64_t row = m0 + row_local(r);
        if (row >= M) continue;
        float *dst = C + row * p.ldc + col;
        if (pair) {
            *reinterpret_cast<float2 *>(dst) = make_float2(a0[r], a1[r]);
        } else {
            if (col < N) dst[0] = a0[r];
            if (col + 1 < N) dst[1] = a1[r];
        }
    }
}

template <bool TA, bool TB, int EPI, int CL, int WM, int WN, int MB, int WK>
__global__ __launch_bounds__(WM *WN *WK * 64, 2) void gemm_f32_split(KParams p) {
    static_assert(CL == 0 || EPI == EPI_STORE, "the RoPE column layouts store plain values");
    static_assert(EPI != EPI_CE || WN % 2 == 0, "the loss takes 128 columns at a time");
    using S = TileShape<WM, WN, MB>;
    constexpr int TM = S::TM, TN = S::TN, NT = S::NT;
    __shared__ __attribute__((aligned(128))) char lds[WK * 2 * S::STAGE];

    const int tid = threadIdx.x;
    // XCD-aware renumbering, then grouped tile order
    const int64_t kbeg = (int64_t)blockIdx.z * p.k_per_split;
    const int64_t kend = min(p.k, kbeg + p.k_per_split);
    const int nb = (int)gridDim.x, q = nb >> 3, r8 = nb & 7;
    const int xcd = (int)blockIdx.x & 7, local = (int)blockIdx.x >> 3;
    const int bid = xcd * q + (xcd < r8 ? xcd : r8) + local;
    int tm, tn;
    grouped_tile(p, group_rows(TM), bid, tm, tn);
    const int64_t m0 = (int64_t)tm * TM, n0 = (int64_t)tn * TN;

    const int64_t batch = blockIdx.y;
    const int split = blockIdx.z;
    const float *__restrict__ A = p.a + batch * p.stride_a;
    const float *__restrict__ B = p.b + batch * p.stride_b;
    const int64_t M = p.m, N = p.n;

    floatx16 acc[MB][2];
    // EPI_CE: the tile's target ids go to LDS before the K loop (whose
    // barriers order them before the epilogue reads them)
    __shared__ int ce_t[EPI == EPI_CE ? TM : 1];
    if (EPI == EPI_CE && tid < TM) ce_t[tid] = m0 + tid < M ? p.ce_targets[m0 + tid] : -1;
    split_mainloop<TA, TB, CL, WM, WN, MB, WK>(p, A, B, m0, n0, kbeg, kend, lds, acc);

    const int lane = tid & 63, wave = tid % NT >> 6;
    const int wm = wave / WN, wn = wave % WN;
    const int lr = lane & 31, lk = lane >> 5;

    // The groups' sums meet in LDS, added in group order by group 0.
    const bool first = WK == 1 || tid < NT;
    if constexpr (WK > 1) {
        static_assert((WK - 1) * MB * 32 * NT * 4 <= WK * 2 * S::STAGE, "the sums fit the stages");
        float *sums = reinterpret_cast<float *>(lds);
        __syncthreads();  // the last operand reads are done
        if (!first) {
            float *mine = sums + (tid / NT - 1) * (MB * 32 * NT) + tid % NT;
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) mine[((i * 2 + j) * 16 + r) * NT] = acc[i][j][r];
        }
        __syncthreads();
        if (first) {
#pragma unroll
            for (int g = 0; g < WK - 1; ++g)
#pragma unroll
                for (int i = 0; i < MB; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
#pragma unroll
                        for (int r = 0; r < 16; ++r)
                            acc[i][j][r] += sums[(g * MB * 32 + (i * 2 + j) * 16 + r) * NT + tid];
        }
    }

    // ---- what the split does not hold -------------------------------------
    bool redo = false;
    if (first) {
        float nf = 0.0f;  // NaN once any accumulator is not finite
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    acc[i][j][r] *= kUnlift2;
                    nf = __builtin_fmaf(acc[i][j][r], 0.0f, nf);
                }
        redo = !(nf == 0.0f);
    }
    if (EPI == EPI_STORE || EPI == EPI_ACCUM) {
        if (first && __float_as_uint(p.acc_init) != 0) {
            // A sum of zero that is added to a -0 of C keeps its own sign (a
            // split's too: C is as it was until splitk_reduce). Any other C or
            // another split's sum hides it, so zero rows of an operand cost the
            // reads of C alone: eight at a time, since a read under each sum's
            // own test would wait by itself (512 x 2048 x 1408 tn, a quarter of k
            // zero: 50.5 us so, 38.2 this way, 34.2 dense).
            const float *C = p.c + batch * p.stride_c;
#pragma unroll
            for (int i = 0; i < MB; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    bool zero = false;
#pragma unroll
                    for (int r = 0; r < 16; ++r) zero |= acc[i][j][r] == 0.0f;
                    if (!__any(zero)) continue;
                    const int64_t col = n0 + place_col<CL>(wn, j, lr);
                    const int64_t row0 = m0 + (wm * MB + i) * 32 + 4 * lk;
#pragma unroll
                    for (int r0 = 0; r0 < 16; r0 += 8) {
                        uint32_t c[8];
#pragma unroll
                        for (int q = 0; q < 8; ++q) {
                            const int64_t row = row0 + 2 * r0 + 8 * (q >> 2) + (q & 3);
                            c[q] = __float_as_uint(C[min(row, M - 1) * p.ldc + min(col, N - 1)]);
                        }
#pragma unroll
                        for (int q = 0; q < 8; ++q) {
                            const int64_t row = row0 + 2 * r0 + 8 * (q >> 2) + (q & 3);
                            redo |= acc[i][j][r0 + q] == 0.0f && row < M && col < N && c[q] == 0x80000000u;
                        }
                    }
                }
        }
    }
    redo = __syncthreads_or(redo);
    if (EPI != EPI_CE && !first) return;
    if (first && redo) exact_mainloop<TA, TB, CL, WM, WN, MB>(p, A, B, m0, n0, kbeg, kend, acc);

    // ---- epilogue: block (i, j) register r of lane l is C[row][col] with
    // row = m0 + 32*(MB*wm + i) + 8*(r/4) + 4*(l/32) + r%4 and, for CL 0,
    // col = n0 + 64*wn + 2*(l%32) + j (the other layouts: place_col).
    const int64_t col = n0 + wn * 64 + 2 * lr;
    if constexpr (EPI == EPI_CE) {
        // Cross-entropy partials of the tile's columns, 128 at a time
        // (ops_reduce.rs:236-259 split by column units): per row, the max of
        // the logits and the sum of exp(z - max) over the lane's two columns,
        // over the 32 lanes of its half by DPP moves, then over the two waves
        // of a unit through LDS. The lane holding a row's target column keeps
        // its logit. (The K loop's LDS is free behind the barrier above.)
        float(*ce_m)[TM] = reinterpret_cast<float(*)[TM]>(lds);
        float(*ce_s)[TM] = reinterpret_cast<float(*)[TM]>(lds + WN * TM * 4);
        constexpr float kLog2e = 1.4426950408889634f;
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (!first) break;
                const int rl = (wm * MB + i) * 32 + 8 * (r >> 2) + 4 * lk + (r & 3);
                const int64_t row = m0 + rl;
                const float v0 = acc[i][0][r], v1 = acc[i][1][r];
                const float x0 = col < N ? v0 : -INFINITY, x1 = col + 1 < N ? v1 : -INFINITY;
                const float mx = half_max32(fmaxf(x0, x1));
                // exp(z - max) through the hardware's exp2 (no flush concern: the
                // terms that matter are within a few hundred of 1) or libm_exp
                float e = 0.0f;
                if (mx != -INFINITY)
                    e = p.libm_exp ? expf(x0 - mx) + expf(x1 - mx)
                                   : __builtin_amdgcn_exp2f((x0 - mx) * kLog2e) +
                                         __builtin_amdgcn_exp2f((x1 - mx) * kLog2e);
                e = half_sum32(e);
                if (lr == 0) {
                    ce_m[wn][rl] = mx;
                    ce_s[wn][rl] = e;
                }
                const int t = ce_t[rl];
                if (t == col) p.ce_zt[row] = v0;
                if (t == col + 1) p.ce_zt[row] = v1;
            }
        __syncthreads();
        for (int e = tid; e < TM * (WN / 2); e += NT * WK) {
            const int rl = e % TM, u = e / TM;
            const int64_t unit = (int64_t)tn * (WN / 2) + u;
            if (m0 + rl >= M || unit >= p.ce_tiles) continue;
            float m = ce_m[2 * u][rl], sum = ce_s[2 * u][rl];
            lse_merge(m, sum, ce_m[2 * u + 1][rl], ce_s[2 * u + 1][rl]);
            reinterpret_cast<float2 *>(p.ce_part)[(m0 + rl) * p.ce_tiles + unit] =
                make_float2(m, sum);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < MB; ++i) {
        block_epilogue<EPI, CL, TM, TN>(p, acc[i][0], acc[i][1], split, batch, m0, n0,
                                        (wm * MB + i) * 32, wn, lr, lk);
        __builtin_amdgcn_sched_barrier(0);  // one block's reads in registers at a time
    }
}

// Sums the large tiles' split partials in split order, then applies the
// epilogue. VEC: four consecutive columns per thread (n, ldc multiples of 4,
// 16-byte aligned C, residual and partials), four splits' loads in flight.
template <int EPI, bool VEC>
__global__ __launch_bounds__(256) void splitk_reduce(const float *__restrict__ partial,
                                                     float *c, const float *resid, int64_t m,
                                                     int64_t n, int64_t ldc, int splits) {
    const int64_t total = m * n;
    if (VEC) {
        for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; 4 * q < total;
             q += (int64_t)gridDim.x * blockDim.x) {
            const int64_t idx = 4 * q;
            float4 acc = *reinterpret_cast<const float4 *>(partial + idx);
            for (int s0 = 1; s0 < splits; s0 += 4) {
                float4 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (s0 + u < splits)
                        v[u] = *reinterpret_cast<const float4 *>(partial + (int64_t)(s0 + u) * total + idx);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (s0 + u < splits) {
                        acc.x = __fadd_rn(acc.x, v[u].x);
                        acc.y = __fadd_rn(acc.y, v[u].y);
                        acc.z = __fadd_rn(acc.z, v[u].z);
                        acc.w = __fadd_rn(acc.w, v[u].w);
                    }
            }
            const int64_t row = idx / n, col = idx - row * n;
            float4 *dst = reinterpret_cast<float4 *>(c + row * ldc + col);
            if (EPI == EPI_ACCUM) {
                const float4 r = *reinterpret_cast<const float4 *>((resid ? resid : c) + row * ldc + col);
                acc.x = __fadd_rn(r.x, acc.x);
                acc.y = __fadd_rn(r.y, acc.y);
                acc.z = __fadd_rn(r.z, acc.z);
                acc.w = __fadd_rn(r.w, acc.w);
            }
            *dst = acc;
        }
        return;
    }
    for (int64_t idx = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; idx < total;
         idx += (int64_t)gridDim.x * blockDim.x) {
        float acc = partial[idx];
        for (int s = 1; s < splits; ++s) acc = __fadd_rn(acc, partial[(int64_t)s * total + idx]);
        const int64_t row = idx / n, col = idx - row * n;
        float *dst = c + row * ldc + col;
        if (EPI == EPI_ACCUM)
            *dst = __fadd_rn((resid ? resid : c)[row * ldc + col], acc);
        else
            *dst = acc;
    }
}

template <bool TA, bool TB, int EPI, int CL = 0>
void launch_tile(Context &ctx, const KParams &p, dim3 grid, int tile) {
#define MMH_GEMM_TILE(WM, WN, MB, WK)                                                        \
    hipLaunchKernelGGL((gemm_f32_split<TA, TB, EPI, CL, WM, WN, MB, WK>), grid,              \
                       dim3(WM * WN * WK * 64), 0, ctx.stream, p)
    switch (tile) {
        case TILE_256:
            if constexpr (EPI != EPI_SWIGLU_BWD) MMH_GEMM_TILE(2, 4, 4, 1);
            break;
        case TILE_256x128: MMH_GEMM_TILE(4, 2, 2, 1); break;
        case TILE_128: MMH_GEMM_TILE(2, 2, 2, 2); break;
        case TILE_128x64:
            if constexpr (EPI != EPI_CE && CL == 0) MMH_GEMM_TILE(4, 1, 1, 2);
            break;
        case TILE_64:
            if constexpr (EPI != EPI_CE && CL == 0) MMH_GEMM_TILE(2, 1, 1, 4);
            break;
    }
#undef MMH_GEMM_TILE
}

template <int EPI>
void launch_form(Context &ctx, const KParams &p, dim3 grid, bool ta, bool tb, int tile) {
    if (!ta && !tb) launch_tile<false, false, EPI>(ctx, p, grid, tile);
    else if (!ta) launch_tile<false, true, EPI>(ctx, p, grid, tile);
    else launch_tile<true, false, EPI>(ctx, p, grid, tile);
}

bool aligned16(const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

}  // namespace

// The loss and the rotation need 128 columns in a tile; the SwiGLU backward
// does not fit the 256x256 tile's registers (its epilogue spills).
bool gemm_tile_takes(const KParams &p, int epi, int tile) {
    if (tile == TILE_256) return epi != EPI_SWIGLU_BWD;
    return (tile != TILE_128x64 && tile != TILE_64) || (epi != EPI_CE && !p.rope_cos);
}

void launch_gemm_tiles(Context &ctx, const KParams &p, dim3 grid, bool ta, bool tb, int epi,
                       int tile) {
    if (epi == EPI_CE) {
        if (tb) launch_tile<false, true, EPI_CE>(ctx, p, grid, tile);
        else launch_tile<false, false, EPI_CE>(ctx, p, grid, tile);
    } else if (epi == EPI_SWIGLU) {
        launch_tile<false, false, EPI_SWIGLU>(ctx, p, grid, tile);
    } else if (epi == EPI_SWIGLU_BWD) {
        launch_tile<false, true, EPI_SWIGLU_BWD>(ctx, p, grid, tile);
    } else if (p.rope_cos) {  // heads of 64 or 128 columns rotated in registers
        if (p.rope_hd == 64) launch_tile<false, false, EPI_STORE, 1>(ctx, p, grid, tile);
        else launch_tile<false, false, EPI_STORE, 2>(ctx, p, grid, tile);
    } else if (epi == EPI_ACCUM) {
        launch_form<EPI_ACCUM>(ctx, p, grid, ta, tb, tile);
    } else {
        launch_form<EPI_STORE>(ctx, p, grid, ta, tb, tile);
    }
    check_hip(hipGetLastError(), "gemm launch");
}

void launch_splitk_reduce(Context &ctx, const KParams &p, int epi) {
    const int64_t total = p.m * p.n;
    const bool vec = p.n % 4 == 0 && p.ldc % 4 == 0 && aligned16(p.c) && aligned16(p.partial) &&
                     (!p.resid || aligned16(p.resid));
    const int64_t items = vec ? total / 4 : total;
    const unsigned blocks = (unsigned)std::min<int64_t>((items + 255) / 256, 8192);
#define MMH_SPLITK(E, V)                                                                     \
    hipLaunchKernelGGL((splitk_reduce<E, V>), dim3(blocks), dim3(256), 0, ctx.stream, p.partial, \
                       p.c, p.resid, p.m, p.n, p.ldc, p.splits)
    if (epi == EPI_ACCUM) {
        if (vec) MMH_SPLITK(EPI_ACCUM, true); else MMH_SPLITK(EPI_ACCUM, false);
    } else {
        if (vec) MMH_SPLITK(EPI_STORE, true); else MMH_SPLITK(EPI_STORE, false);
    }
#undef MMH_SPLITK
    check_hip(hipGetLastError(), "split-k reduce launch");
}

}  // namespace mmh
