// fp32 GEMM on CDNA4 matrix cores, small shapes (v_mfma_f32_32x32x2_f32), and
// the choice of kernel for every shape.
//
// Replaces the reference's three CPU kernels (midman-tensor/src/kernels.rs:49-108,
// kernels_avx.rs:45-250): C = A.B (nn), A.B^T (nt) and A^T.B (tn). The
// transposed forms never materialize a transpose (the reference copies B^T,
// kernels.rs:68-73): each operand is read in its stored layout and written into
// LDS k-major, the layout the MFMA operand reads want.
//
// The products with enough 128x128 tiles of work run on gemm_split.hip's
// kernels. Here are the 64x64 tiles (a workgroup each, one 32x32 MFMA block
// per wave) and the 32x32 K-split tiles for the shapes that are bound by
// latency rather than by the matrix cores' rate.
//
// MFMA 32x32x2 f32 operand layout (wave64): lane l supplies A[i=l%32][k=l/32]
// and B[k=l/32][j=l%32]; accumulator register r of lane l holds
// D[i = 8*(r/4) + 4*(l/32) + r%4][j = l%32].
//
// Small-tile-count shapes (e.g. M=2048, N=256) are split along K; the
// partials are summed in split order, so the result is deterministic: on the
// 64x64 and 32x32 tiles by the last split of each tile (the splits store
// their partial through to memory and count themselves in a per-tile
// counter), on the large tiles by a second kernel.
#include "mmh_gemm.h"

#include <algorithm>
#include <cmath>

namespace mmh {
namespace {

// Split partials for the in-kernel reduction: stored through to memory and
// read past the XCD-local L2 (device-scope relaxed atomics: sc1 stores and
// loads), so the last split of a tile, on any XCD, reads every split's values.
__device__ __forceinline__ void split_put(float *dst, float v) {
    __hip_atomic_store(dst, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ float split_get(const float *src) {
    return __hip_atomic_load(const_cast<float *>(src), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// After a workgroup's split_put stores: true in the workgroup that completes
// the tile (the last of its p.splits splits to get here), which also resets
// the tile's counter for the next launch. Every thread of the workgroup calls it.
__device__ __forceinline__ bool split_last(const KParams &p, int tile) {
    __shared__ int s_last;
    __builtin_amdgcn_s_waitcnt(0);  // this thread's partial stores are complete
    __syncthreads();
    if (threadIdx.x == 0) {
        const int old = __hip_atomic_fetch_add(p.tickets + tile, 1, __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
        s_last = old == p.splits - 1;
        if (s_last) __hip_atomic_store(p.tickets + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    return s_last;
}
// The last split of a tile: rows [m0, m0 + tr) x columns [n0, n0 + tc) of C
// (tc a multiple of 4) as the splits' partials added in split order (the
// caller's own included, read back like the others), then the epilogue
// (split_accum: C = resid (or C) + sum). The nthreads threads walk the tile
// row-major, four columns at a time, with four splits' loads in flight;
// partial rows of N % 4 == 0 move as float4, others one value at a time.
__device__ __forceinline__ void split_reduce_tile(const KParams &p, int64_t m0, int64_t n0, int tr,
                                               int tc, int nthreads) {
    const int64_t M = p.m, N = p.n, total = M * N;
    const bool vecp = N % 4 == 0;
    const bool vecc = p.ldc % 4 == 0 && (reinterpret_cast<uintptr_t>(p.c) & 15) == 0 &&
                      (!p.resid || (reinterpret_cast<uintptr_t>(p.resid) & 15) == 0);
    const float *R = p.resid ? p.resid : p.c;
    const int iters = tr * tc / (4 * nthreads);
    if (m0 + tr <= M && n0 + tc <= N && vecp && vecc && iters <= 4 &&
        iters * 4 * nthreads == tr * tc) {
        // The whole tile in range: every element's reads (the residual, then
        // the partials) before the first store, so no read waits for a store.
        float4 res[4];
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            if (it >= iters) break;
            const int e = 4 * (int)threadIdx.x + it * 4 * nthreads;
            const int64_t row = m0 + e / tc, col = n0 + e % tc;
            const float4 o = p.split_accum ? *reinterpret_cast<const float4 *>(R + row * p.ldc + col)
                                           : make_float4(0.f, 0.f, 0.f, 0.f);
            const float *Q = p.partial + row * N + col;
            float4 acc;
            for (int s0 = 0; s0 < p.splits; s0 += 4) {
                float4 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (s0 + u < p.splits) {
                        const float *src = Q + (int64_t)(s0 + u) * total;
                        v[u].x = split_get(src);
                        v[u].y = split_get(src + 1);
                        v[u].z = split_get(src + 2);
                        v[u].w = split_get(src + 3);
                    }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (s0 + u < p.splits) {
                        if (s0 + u == 0) {
                            acc = v[u];
                        } else {
                            acc.x = __fadd_rn(acc.x, v[u].x);
                            acc.y = __fadd_rn(acc.y, v[u].y);
                            acc.z = __fadd_rn(acc.z, v[u].z);
                            acc.w = __fadd_rn(acc.w, v[u].w);
                        }
                    }
            }
            res[it] = p.split_accum ? make_float4(__fadd_rn(o.x, acc.x), __fadd_rn(o.y, acc.y),
                                                  __fadd_rn(o.z, acc.z), __fadd_rn(o.w, acc.w))
                                    : acc;
        }
#pragma unroll
        for (int it = 0; it < 4; ++it) {
            if (it >= iters) break;
            const int e = 4 * (int)threadIdx.x + it * 4 * nthreads;
            *reinterpret_cast<float4 *>(p.c + (m0 + e / tc) * p.ldc + n0 + e % tc) = res[it];
        }
        return;
    }
    for (int e = 4 * (int)threadIdx.x; e < tr * tc; e += 4 * nthreads) {
        const int64_t row = m0 + e / tc, col = n0 + e % tc;
        if (row >= M || col >= N) continue;
        const float *Q = p.partial + row * N + col;
        if (vecp && col + 3 < N) {
            float4 acc;
            for (int s0 = 0; s0 < p.splits; s0 += 4) {
                float4 v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (s0 + u < p.splits) {
                        const float *src = Q + (int64_t)(s0 + u) * total;
                        v[u].x = split_get(src);
                        v[u].y = split_get(src + 1);
                        v[u].z = split_get(src + 2);
                        v[u].w = split_get(src + 3);
                    }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (s0 + u < p.splits) {
                        if (s0 + u == 0) {
                            acc = v[u];
                        } else {
                            acc.x = __fadd_rn(acc.x, v[u].x);
                            acc.y = __fadd_rn(acc.y, v[u].y);
                            acc.z = __fadd_rn(acc.z, v[u].z);
                            acc.w = __fadd_rn(acc.w, v[u].w);
                        }
                    }
            }
            float *dst = p.c + row * p.ldc + col;
            if (p.split_accum) {
                const float *r = R + row * p.ldc + col;
                if (vecc) {
                    const float4 o = *reinterpret_cast<const float4 *>(r);
                    acc = make_float4(__fadd_rn(o.x, acc.x), __fadd_rn(o.y, acc.y),
                                      __fadd_rn(o.z, acc.z), __fadd_rn(o.w, acc.w));
                } else {
                    acc = make_float4(__fadd_rn(r[0], acc.x), __fadd_rn(r[1], acc.y),
                                      __fadd_rn(r[2], acc.z), __fadd_rn(r[3], acc.w));
                }
            }
            if (vecc) {
                *reinterpret_cast<float4 *>(dst) = acc;
            } else {
                dst[0] = acc.x;
                dst[1] = acc.y;
                dst[2] = acc.z;
                dst[3] = acc.w;
            }
            continue;
        }
        for (int u = 0; u < 4 && col + u < N; ++u) {
            float v = split_get(Q + u);
            for (int s = 1; s < p.splits; ++s) v = __fadd_rn(v, split_get(Q + (int64_t)s * total + u));
            float *dst = p.c + row * p.ldc + col + u;
            *dst = p.split_accum ? __fadd_rn(R[row * p.ldc + col + u], v) : v;
        }
    }
}

// ---- small-tile GEMM ---------------------------------------------------------
// For shapes with fewer 128x128 tiles than CUs (the tiny preset's projections,
// M = 2048 with N and K of a few hundred) the big tile leaves most of the chip
// idle and every workgroup walks the whole K alone. Here a 256-thread
// workgroup owns a 64x64 tile, each wave one 32x32 MFMA block (16
// accumulators), K advancing 32 at a time, so the grid holds 4x the
// workgroups. With so few steps per tile, latency rules: three steps of global
// loads are kept in flight (a ring of register slots) ahead of the two LDS
// stages, and each lane reads its operands of a step as four 16-byte LDS
// reads. The epilogues match the big kernel's; in the SwiGLU epilogue the gate
// and up columns of a pair sit in neighbouring lanes and meet through one lane
// exchange.
constexpr int SBM = 64, SBN = 64, SBK = 32;
// LDS rows hold one output row (A) or column (B) with its 32 k values
// contiguous, padded to 36 floats: a lane reads its 16 k values of a step as
// four 16-byte reads, and eight consecutive rows fall in distinct 16-byte bank
// groups. An operand stored k-major in memory (A when TA, B when !TB) reaches
// LDS as single values at (row, k), 16 rows 4 apart per 16 lanes: its rows
// keep their eight float4 groups of k in the order g ^ ((row >> 3) & 7), so
// those stores spread over the banks (2 lanes per bank instead of 8) while the
// float4 reads stay aligned and conflict-free.
constexpr int SKS = SBK + 4;
__device__ __forceinline__ int sk_swz(int row) { return (row >> 3) & 7; }

// The K loop of one 64x64 tile. MFMA kk of a step takes k = kk from lanes
// 0-31 and k = 16 + kk from lanes 32-63 (any split of the step's k values
// between the two lane halves gives the same sum; A and B agree on it).
// FAST: every step is a full interior step (no predicates anywhere, so the
// compiler can count the loads in flight exactly).
template <bool TA, bool TB, bool FAST, bool NORM>
__device__ __forceinline__ void small_mainloop(const KParams &p, const float *__restrict__ A,
                                               const float *__restrict__ B, int64_t m0,
                                               int64_t n0, int64_t kbeg, int nk, int64_t kend,
                                               float (*As)[SBM][SKS], float (*Bs)[SBN][SKS],
                                               floatx16 &acc, float (&ss)[2]) {
    const int tid = threadIdx.x;
    const int64_t M = p.m, N = p.n;
    // A tile of each operand is 64 x 32 floats = 512 float4: thread tid moves
    // float4 idx = tid + 256*i, i < 2. Operands stored row-major in k (A for
    // nn/nt, B for nt): row idx/8, k (idx%8)*4. Operands stored k-major: k
    // idx/16, row (idx%16)*4.
    constexpr int PF = 3;  // k-steps of loads in flight
    float4 ra[PF][2], rb[PF][2], rw[PF];  // rw: the norm weights of A's k values
    auto load = [&](int64_t k0, int slot) __attribute__((always_inline)) {
        if (NORM) {
            // both of a thread's A float4 cover k = k0 + (tid%8)*4 .. +3
            const int64_t gk = k0 + (tid & 7) * 4;
            const float *wk = p.norm_w + gk;
            float4 w4 = make_float4(0.f, 0.f, 0.f, 0.f);
            if (FAST) {
                w4 = *reinterpret_cast<const float4 *>(wk);
            } else {
                if (gk + 0 < kend) w4.x = wk[0];
                if (gk + 1 < kend) w4.y = wk[1];
                if (gk + 2 < kend) w4.z = wk[2];
                if (gk + 3 < kend) w4.w = wk[3];
            }
            rw[slot] = w4;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int idx = tid + 256 * i;
            // padding: A -0, B +0, so a padded product is -0, the identity of addition
            float4 v = make_float4(-0.f, -0.f, -0.f, -0.f), w = make_float4(0.f, 0.f, 0.f, 0.f);
            if (!TA) {
                const int64_t gm = m0 + (idx >> 3), gk = k0 + (idx & 7) * 4;
                const float *src = A + gm * p.lda + gk;
                if (FAST) {
                    v = *reinterpret_cast<const float4 *>(src);
                } else if (gm < M) {
                    if (gk + 0 < kend) v.x = src[0];
                    if (gk + 1 < kend) v.y = src[1];
                    if (gk + 2 < kend) v.z = src[2];
                    if (gk + 3 < kend) v.w = src[3];
                }
            } else {
                const int64_t gk = k0 + (idx >> 4), gm = m0 + (idx & 15) * 4;
                const float *src = A + gk * p.lda + gm;
                if (FAST) {
                    v = *reinterpret_cast<const float4 *>(src);
                } else if (gk < kend) {
                    if (gm + 0 < M) v.x = src[0];
                    if (gm + 1 < M) v.y = src[1];
                    if (gm + 2 < M) v.z = src[2];
                    if (gm + 3 < M) v.w = src[3];
                }
            }
            if (!TB) {
                const int64_t gk = k0 + (idx >> 4), gn = n0 + (idx & 15) * 4;
                const float *src = B + gk * p.ldb + gn;
                if (FAST) {
                    w = *reinterpret_cast<const float4 *>(src);
                } else if (gk < kend) {
                    if (gn + 0 < N) w.x = src[0];
                    if (gn + 1 < N) w.y = src[1];
                    if (gn + 2 < N) w.z = src[2];
                    if (gn + 3 < N) w.w = src[3];
                }
            } else {
                const int64_t gn = n0 + (idx >> 3), gk = k0 + (idx & 7) * 4;
                const float *src = B + gn * p.ldb + gk;
                if (FAST) {
                    w = *reinterpret_cast<const float4 *>(src);
                } else if (gn < N) {
                    if (gk + 0 < kend) w.x = src[0];
                    if (gk + 1 < kend) w.y = src[1];
                    if (gk + 2 < kend) w.z = src[2];
                    if (gk + 3 < kend) w.w = src[3];
                }
            }
            ra[slot][i] = v;
            rb[slot][i] = w;
        }
    };
    // real: the slot holds a k-step not yet summed (the ring's last stores
    // repeat the final step into the idle stage; those must not count)
    auto store = [&](int buf, int slot, bool real) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int idx = tid + 256 * i;
            float4 va = ra[slot][i];
            const float4 vb = rb[slot][i];
            if (NORM) {
                // the row's sum of squares as its values pass, and x * w; the
                // row's 1/rms scales the products in the epilogue
                const float4 w4 = rw[slot];
                float t = __fadd_rn(ss[i], __fmul_rn(va.x, va.x));
                t = __fadd_rn(t, __fmul_rn(va.y, va.y));
                t = __fadd_rn(t, __fmul_rn(va.z, va.z));
                t = __fadd_rn(t, __fmul_rn(va.w, va.w));
                ss[i] = real ? t : ss[i];
                va.x = __fmul_rn(va.x, w4.x);
                va.y = __fmul_rn(va.y, w4.y);
                va.z = __fmul_rn(va.z, w4.z);
                va.w = __fmul_rn(va.w, w4.w);
            }
            if (!TA) {
                *reinterpret_cast<float4 *>(&As[buf][idx >> 3][(idx & 7) * 4]) = va;
            } else {
                const int k = idx >> 4, row = (idx & 15) * 4;
                As[buf][row + 0][k ^ (4 * sk_swz(row + 0))] = va.x;
                As[buf][row + 1][k ^ (4 * sk_swz(row + 1))] = va.y;
                As[buf][row + 2][k ^ (4 * sk_swz(row + 2))] = va.z;
                As[buf][row + 3][k ^ (4 * sk_swz(row + 3))] = va.w;
            }
            if (!TB) {
                const int k = idx >> 4, col = (idx & 15) * 4;
                Bs[buf][col + 0][k ^ (4 * sk_swz(col + 0))] = vb.x;
                Bs[buf][col + 1][k ^ (4 * sk_swz(col + 1))] = vb.y;
                Bs[buf][col + 2][k ^ (4 * sk_swz(col + 2))] = vb.z;
                Bs[buf][col + 3][k ^ (4 * sk_swz(col + 3))] = vb.w;
            } else {
                *reinterpret_cast<float4 *>(&Bs[buf][idx >> 3][(idx & 7) * 4]) = vb;
            }
        }
    };

    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane & 31, lk = lane >> 5;
    const int ga = TA ? sk_swz(wm * 32 + lr) : 0, gb = TB ? 0 : sk_swz(wn * 32 + lr);
    auto compute = [&](int buf) __attribute__((always_inline)) {
        const float4 *pa = reinterpret_cast<const float4 *>(&As[buf][wm * 32 + lr][0]);
        const float4 *pb = reinterpret_cast<const float4 *>(&Bs[buf][wn * 32 + lr][0]);
        float4 a[4], b[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            a[q] = pa[(4 * lk + q) ^ ga];
            b[q] = pb[(4 * lk + q) ^ gb];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].x, b[q].x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].y, b[q].y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].z, b[q].z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[q].w, b[q].w, acc, 0, 0, 0);
        }
    };

    // Steps that do not fill a group of PF run first, one at a time. Then,
    // per group, sub-iteration j (global step t) stores step t+1 from slot
    // (j+1)%PF into the LDS stage not in use, loads step t+PF into slot j
    // (whose step t went to LDS one sub-iteration earlier), runs the MFMAs of
    // step t and ends with the one barrier. Slot indices are constants of the
    // unrolled group and every load is issued unconditionally (past the last
    // step they re-read it, from cache), so the wait before each store counts
    // exactly the PF-2 younger steps and lets them stay in flight.
    auto step_k = [&](int t) __attribute__((always_inline)) {
        return kbeg + (int64_t)min(t, nk - 1) * SBK;
    };
    int t = 0;
    for (; t < nk % PF; ++t) {
        load(step_k(t), 0);
        store(0, 0, true);
        __syncthreads();
        compute(0);
        __syncthreads();
    }
    if (t == nk) return;
#pragma unroll
    for (int j = 0; j < PF; ++j) load(step_k(t + j), j);
    store(0, 0, true);
    __syncthreads();
    for (int g = 0; t < nk; ++g, t += PF) {
#pragma unroll
        for (int j = 0; j < PF; ++j) {
            const int cur = (g * PF + j) & 1;
            store(cur ^ 1, (j + 1) % PF, t + j + 1 < nk);
            load(step_k(t + j + PF), j);
            compute(cur);
            __syncthreads();
        }
    }
}

// One accumulator value v of C[row][col] of a 32-column MFMA block (lane lr
// holds column col) through the epilogues of the small kernels. Every lane of
// the wave calls it: the SwiGLU gate/up pair and the RoPE pair meet through
// lane exchanges. SwiGLU: gate f at column 2f (even lane), up f at 2f+1 (the
// next lane). RoPE (rope.rs:28-32) on heads of rope_hd (<= 32, dividing 32)
// columns: the pair (c, c + hd/2) of a head sits in lanes lr and lr ^ hd/2.
template <int EPI>
__device__ __forceinline__ void block32_epilogue(const KParams &p, float *C, const float *R,
                                                 int64_t row, int64_t col, int lr, float v) {
    if (EPI == EPI_SWIGLU) {
        const float up = __shfl_xor(v, 1, 64);
        if ((lr & 1) || row >= p.m) return;
        const int64_t f = col >> 1;
        if (p.aux && col + 1 < p.n)
            *reinterpret_cast<float2 *>(p.aux + row * p.ldaux + col) = make_float2(v, up);
        if (f < p.swiglu_ff) C[row * p.ldc + f] = __fmul_rn(silu_f(v), up);
        return;
    }
    if (EPI == EPI_STORE && p.rope_cos) {
        const int hd = p.rope_hd, half = hd >> 1;
        const float other = __shfl_xor(v, half, 64);
        if (row >= p.m || col >= p.n) return;
        if (col < p.rope_cols) {
            const int pc = (int)(col % hd);
            const int64_t pos = row % p.rope_seq;
            const int c = pc < half ? pc : pc - half;
            const float cs = p.rope_cos[pos * half + c], sn = p.rope_sin[pos * half + c];
            v = pc < half ? v * cs - other * sn : v * cs + other * sn;
        }
        C[row * p.ldc + col] = v;
        return;
    }
    if (row >= p.m || col >= p.n) return;
    C[row * p.ldc + col] = EPI == EPI_ACCUM ? __fadd_rn(R[row * p.ldc + col], v) : v;
}

template <bool TA, bool TB, int EPI, bool NORM>
__global__ __launch_bounds__(256) void gemm_f32_mfma_small(KParams p) {
    __shared__ __attribute__((aligned(16))) float As[2][SBM][SKS];
    __shared__ __attribute__((aligned(16))) float Bs[2][SBN][SKS];
    __shared__ float sm_inv[SBM];  // NORM: 1/rms of the tile's rows

    const int tid = threadIdx.x;
    const int bid = blockIdx.x;
    const int tm = bid / p.tiles_n, tn = bid - (bid / p.tiles_n) * p.tiles_n;
    const int64_t m0 = (int64_t)tm * SBM, n0 = (int64_t)tn * SBN;
    const int64_t batch = blockIdx.y;
    const int split = blockIdx.z;
    const float *__restrict__ A = p.a + batch * p.stride_a;
    const float *__restrict__ B = p.b + batch * p.stride_b;
    const int64_t kbeg = (int64_t)split * p.k_per_split;
    const int64_t kend = min(p.k, kbeg + p.k_per_split);
    const int64_t M = p.m, N = p.n;

    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = p.acc_init;
    // NORM: sums of squares of this thread's two A rows (the loads give
    // thread tid rows tid/8 and 32 + tid/8 at every K-step), gathered as the
    // values pass through the LDS stores.
    float ss[2] = {0.0f, 0.0f};
    const int nk = (int)((kend - kbeg + SBK - 1) / SBK);
    if (p.vec_a && p.vec_b && m0 + SBM <= M && n0 + SBN <= N) {
        // interior: the full steps branch-free, then a K tail (if any) on the
        // predicated path, after the last barrier of the full steps
        const int nfull = (int)((kend - kbeg) / SBK);
        small_mainloop<TA, TB, true, NORM>(p, A, B, m0, n0, kbeg, nfull, kend, As, Bs, acc,
                                           ss);
        if (nfull < nk)
            small_mainloop<TA, TB, false, NORM>(p, A, B, m0, n0, kbeg + (int64_t)nfull * SBK, 1,
                                                kend, As, Bs, acc, ss);
    } else {
        small_mainloop<TA, TB, false, NORM>(p, A, B, m0, n0, kbeg, nk, kend, As, Bs, acc, ss);
    }
    // NORM: each row's 1/rms = (sum/K + eps)^-1/2 (norm.rs:21-39) combined
    // over the row's 8 threads, through LDS to the lanes holding its results,
    // which scale their accumulators by it before any epilogue
    if (NORM) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            float t = ss[i];
            t = __fadd_rn(t, __shfl_xor(t, 1, 64));
            t = __fadd_rn(t, __shfl_xor(t, 2, 64));
            t = __fadd_rn(t, __shfl_xor(t, 4, 64));
            const float mean = __fmul_rn(t, __fdiv_rn(1.0f, (float)p.k));
            if ((tid & 7) == 0)
                sm_inv[((tid + 256 * i) >> 3)] =
                    __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(mean, p.norm_eps)));
        }
        __syncthreads();
        const int lw = tid >> 6, ll = tid & 63;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            acc[r] = __fmul_rn(acc[r], sm_inv[(lw >> 1) * 32 + 8 * (r >> 2) + 4 * (ll >> 5) + (r & 3)]);
    }

    const int lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int lr = lane & 31, lk = lane >> 5;
    // Register r of lane l is C[row][col], row = m0 + wm*32 + 8*(r/4) +
    // 4*(l/32) + r%4, col = n0 + wn*32 + l%32.
    const int64_t col = n0 + wn * 32 + lr;
    auto row_of = [&](int r) { return m0 + wm * 32 + 8 * (r >> 2) + 4 * lk + (r & 3); };

    if (p.splits > 1) {
        float *P = p.partial + (int64_t)split * M * N;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t row = row_of(r);
            if (row < M && col < N) split_put(P + row * N + col, acc[r]);
        }
        if (split_last(p, tm * p.tiles_n + tn)) split_reduce_tile(p, m0, n0, SBM, SBN, 256);
        return;
    }
    float *C = p.c + batch * p.stride_c;
    // A tile inside [M, N): the epilogue's reads all go out before its first
    // store, with no per-row branches (under row tests each read waited for
    // the stores before it: one memory round trip per row). Buffer accesses
    // from the tile's first row, each row's offset in the lane offset (as in
    // the large tiles' epilogues).
    const bool inside = m0 + SBM <= M && n0 + SBN <= N && p.ldc < (int64_t(1) << 21) &&
                        (EPI != EPI_SWIGLU_BWD || p.ldaux < (int64_t(1) << 21));
    const uint32_t lc = 4u * (uint32_t)p.ldc;
    const uint32_t vrow = (uint32_t)(wm * 32 + 4 * lk);  // row_of(r) - m0 - (8*(r/4) + r%4)
    if (EPI == EPI_SWIGLU_BWD && inside) {
        const uint32_t la = 4u * (uint32_t)p.ldaux;
        const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(p.aux + m0 * p.ldaux), (short)0, kBufferRange, kBufferFlags);
        const __amdgpu_buffer_rsrc_t rc =
            __builtin_amdgcn_make_buffer_rsrc(C + m0 * p.ldc, (short)0, kBufferRange, kBufferFlags);
        float2 gu[16];
#pragma unroll
        for (int r = 0; r < 16; ++r)
            gu[r] = __builtin_bit_cast(float2, __builtin_amdgcn_raw_buffer_load_b64(
                                                   ra, (vrow + 8 * (r >> 2) + (r & 3)) * la + 8u * (uint32_t)col,
                                                   0, 0));
#pragma unroll
        for (int r = 0; r < 16; ++r)
            __builtin_amdgcn_raw_buffer_store_b64(
                __builtin_bit_cast(u32x2_t, swiglu_bwd_f(acc[r], gu[r].x, gu[r].y)), rc,
                (vrow + 8 * (r >> 2) + (r & 3)) * lc + 8u * (uint32_t)col, 0, 0);
        return;
    }
    if (EPI == EPI_SWIGLU_BWD) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int64_t row = row_of(r);
            if (row >= M || col >= N) continue;
            const float2 gu = *reinterpret_cast<const float2 *>(p.aux + row * p.ldaux + 2 * col);
            const float2 o = swiglu_bwd_f(acc[r], gu.x, gu.y);
            *reinterpret_cast<float2 *>(C + row * p.ldc + 2 * col) = o;
        }
        return;
    }
    const float *R = p.resid ? p.resid + batch * p.stride_c : C;
    if (EPI == EPI_ACCUM && inside) {
        const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(R + m0 * p.ldc), (short)0, kBufferRange, kBufferFlags);
        const __amdgpu_buffer_rsrc_t rc =
            __builtin_amdgcn_make_buffer_rsrc(C + m0 * p.ldc, (short)0, kBufferRange, kBufferFlags);
        const uint32_t vo = vrow * lc + 4u * (uint32_t)col;
        float o[16];
#pragma unroll
        for (int r = 0; r < 16; ++r)
            o[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                 rr, vo + (8 * (r >> 2) + (r & 3)) * lc, 0, 0));
#pragma unroll
        for (int r = 0; r < 16; ++r)
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, __fadd_rn(o[r], acc[r])), rc,
                                                  vo + (8 * (r >> 2) + (r & 3)) * lc, 0, 0);
        return;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) block32_epilogue<EPI>(p, C, R, row_of(r), col, lr, acc[r]);
}

// ---- K-split 32x32 GEMM -------------------------------------------------------
// For nn shapes that leave most of the chip idle with a K of a few steps (the
// tiny preset's projections: M = 2048, N = 128-704, K = 128-352) the cost is
// latency, not the MFMA rate: a 64x64 tile walks its K steps one after
// another on one workgroup. Here a workgroup owns a 32x32 tile of C and its
// NW waves take the 32-wide K steps round-robin (wave w: steps w, w + NW,
// ...), so a tile's steps run side by side and the grid holds 4x the
// workgroups. Operands go straight from memory into the MFMA layout, no LDS
// staging: lane l takes row (A) or column (B) l%32 and k 16*(l/32) .. +15 of
// a step, A as four float4 reads of its row and B as sixteen reads that are
// coalesced across the lanes. The NW partial tiles meet in LDS and are summed
// in pairs; then wave w applies the epilogue to accumulator registers
// w, w + NW, ... of the sum.
// NORM: the A rows are RMS-normalised on the way in, as in the small kernel:
// x * w feeds the MFMAs, the sums of squares of x are gathered per lane and
// combined over the lane halves and then the waves, and each row's 1/rms
// scales the summed results.
// The epilogue's own reads (the residual of EPI_ACCUM, the cos/sin of the
// rotation) are issued before the operand loads, so their latency hides
// behind the main loop instead of following it.
// MODE: 2 when the K range of every split is a multiple of 32 and the
// k-contiguous operands (A rows when !TA, B rows when TB, the norm weights)
// are 16-byte aligned: float4 reads, no predicates; 1 when only the rows are
// aligned: a lane whose 16 k values all lie in range reads them as float4,
// the lanes of the partial last step one predicated value at a time; 0
// otherwise: every read predicated. (Keeping the predicated path out of mode
// 2 keeps its registers low; a separate tail step measured slower than the
// per-lane test of mode 1.) Operands stored k-major (A when TA, B when !TB)
// are read one value per k, coalesced across the 32 lanes of a half.
// Split K (grid z > 1): each split covers k_per_split values and writes its
// partial tile; the last split of the tile sums the splits in order and
// applies the epilogue.
// N values in pairs, the pairs' sums in pairs and so on: each value is rounded in
// log2(N) sums instead of up to N (error against 64 bits at 53 x 719 x 3584 1.33e-7
// -> 1.17e-7; with more splits, before them, 1.21e-7).
template <int N, class F>
__device__ __forceinline__ float pair_sum(F &&value, int first = 0) {
    if constexpr (N == 1) {
        return value(first);
    } else {
        constexpr int H = N > 8 ? 8 : N / 2;
        const float a = pair_sum<H>(value, first);
        return __fadd_rn(a, pair_sum<N - H>(value, first + H));
    }
}

template <bool TA, bool TB, int EPI, bool NORM, int NW, int MODE>
__global__ __launch_bounds__(64 * NW) void gemm_f32_mfma_ksplit(KParams p) {
    __shared__ float part[NW][16][64];
    __shared__ float sm_ss[NW][32];
    __shared__ float sm_inv[32];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int lr = lane & 31, lk = lane >> 5;
    const int tm = (int)blockIdx.x / p.tiles_n, tn = (int)blockIdx.x - tm * p.tiles_n;
    const int64_t m0 = (int64_t)tm * 32, n0 = (int64_t)tn * 32;
    const int64_t M = p.m, N = p.n;
    const int split = blockIdx.z;
    const int64_t kbeg = (int64_t)split * p.k_per_split;
    const int64_t kend = min(p.k, kbeg + p.k_per_split);
    const int nsteps = (int)((kend - kbeg + 31) / 32);
    // rows and columns past the edge read the last one; their results are not stored
    const int64_t am = min(m0 + lr, M - 1), bn = min(n0 + lr, N - 1);
    const float *arow = TA ? p.a + am : p.a + am * p.lda;    // then + k * (TA ? lda : 1)
    const float *bcol = TB ? p.b + bn * p.ldb : p.b + bn;    // then + k * (TB ? 1 : ldb)

    // Register r of lane l is C[m0 + 8*(r/4) + 4*(l/32) + r%4][n0 + l%32]; wave
    // w applies the epilogue to registers w + i*NW, i < NR.
    constexpr int NR = (16 + NW - 1) / NW;
    const int64_t col = n0 + lr;
    float *C = p.c;
    const float *R = p.resid ? p.resid : C;
    const bool fin = p.splits == 1;
    float pre_r[NR], pre_c[NR], pre_s[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        pre_r[i] = 0.0f;
        pre_c[i] = 1.0f;
        pre_s[i] = 0.0f;
        const int r = wave + i * NW;
        const int64_t row = m0 + 8 * (r >> 2) + 4 * lk + (r & 3);
        if (r >= 16 || !fin || row >= M || col >= N) continue;
        if (EPI == EPI_ACCUM) pre_r[i] = R[row * p.ldc + col];
        if (EPI == EPI_STORE && p.rope_cos && col < p.rope_cols) {
            const int hd = p.rope_hd, half = hd >> 1;
            const int pc = (int)col % hd;  // rows and columns below 2^31 (checked at launch)
            const int64_t t = (int64_t)((int)row % p.rope_seq) * half + (pc < half ? pc : pc - half);
            pre_c[i] = p.rope_cos[t];
            pre_s[i] = p.rope_sin[t];
        }
    }

    // Each step sums from acc_init; a wave with more steps than one adds them
    // up in its own LDS slots: 16 roundings at a step's size and one at the
    // sum's, so few splits of a long K are no less precise than many (error
    // against 64 bits at 128 x 2048 x 688 1.30e-7 in 8 splits, 1.66e-7 in one
    // running sum, 1.34e-7 so; 15.6 us both). The sum leaves a step's
    // registers before the next one's loads: kept across them, it cost the
    // kernel occupancy or spills (768 x 2356 x 89 16.7 -> 35 us, 18 so).
    floatx16 acc;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r] = p.acc_init;
    float ss = 0.0f;
    for (int st = wave; st < nsteps; st += NW) {
        const int64_t kb = kbeg + (int64_t)st * 32 + 16 * lk;  // this lane's first k of the step
        const bool whole = MODE == 2 || (MODE == 1 && kb + 16 <= kend);
        float a[16], b[16];
        if (!TA && whole) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 v = reinterpret_cast<const float4 *>(arow + kb)[i];
                a[4 * i + 0] = v.x;
                a[4 * i + 1] = v.y;
                a[4 * i + 2] = v.z;
                a[4 * i + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j)
                a[j] = (whole || kb + j < kend) ? arow[(kb + j) * (TA ? p.lda : 1)] : -0.0f;
        }
        if (TB && whole) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 v = reinterpret_cast<const float4 *>(bcol + kb)[i];
                b[4 * i + 0] = v.x;
                b[4 * i + 1] = v.y;
                b[4 * i + 2] = v.z;
                b[4 * i + 3] = v.w;
            }
        } else {
#pragma unroll
            for (int j = 0; j < 16; ++j)
                b[j] = (whole || kb + j < kend) ? bcol[(kb + j) * (TB ? 1 : p.ldb)] : 0.0f;
        }
        if (NORM) {
            float w[16];
            if (whole) {
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const float4 v = reinterpret_cast<const float4 *>(p.norm_w + kb)[i];
                    w[4 * i + 0] = v.x;
                    w[4 * i + 1] = v.y;
                    w[4 * i + 2] = v.z;
                    w[4 * i + 3] = v.w;
                }
            } else {
#pragma unroll
                for (int j = 0; j < 16; ++j) w[j] = kb + j < kend ? p.norm_w[kb + j] : 0.0f;
            }
#pragma unroll
            for (int j = 0; j < 16; ++j) {
                ss = __fadd_rn(ss, __fmul_rn(a[j], a[j]));
                a[j] = __fmul_rn(a[j], w[j]);
            }
        }
#pragma unroll
        for (int j = 0; j < 16; ++j) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[j], b[j], acc, 0, 0, 0);
        if (st + NW < nsteps) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if (st != wave) acc[r] = __fadd_rn(part[wave][r][lane], acc[r]);
                part[wave][r][lane] = acc[r];
                acc[r] = p.acc_init;
            }
        }
    }
    if (wave + NW < nsteps) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = __fadd_rn(part[wave][r][lane], acc[r]);
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) part[wave][r][lane] = acc[r];

    if (NORM) {
        // this wave's share of row lr: k 0-15 of its steps in lane lr, 16-31 in lane lr+32
        ss = __fadd_rn(ss, __shfl_xor(ss, 32, 64));
        if (lk == 0) sm_ss[wave][lr] = ss;
    }
    __syncthreads();
    if (NORM) {
        if (tid < 32) {
            float t = sm_ss[0][tid];
#pragma unroll
            for (int w = 1; w < NW; ++w) t = __fadd_rn(t, sm_ss[w][tid]);
            const float mean = __fmul_rn(t, __fdiv_rn(1.0f, (float)p.k));  // norm.rs:21-39
            sm_inv[tid] = __fdiv_rn(1.0f, __fsqrt_rn(__fadd_rn(mean, p.norm_eps)));
        }
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < NR; ++i) {
        const int r = wave + i * NW;
        if (r >= 16) break;
        float v = pair_sum<NW>([&](int w) { return part[w][r][lane]; });
        const int rl = 8 * (r >> 2) + 4 * lk + (r & 3);
        const int64_t row = m0 + rl;
        if (NORM) v = __fmul_rn(v, sm_inv[rl]);
        if (!fin) {
            if (row < M && col < N) split_put(p.partial + ((int64_t)split * M + row) * N + col, v);
        } else if (EPI == EPI_ACCUM) {
            if (row < M && col < N) C[row * p.ldc + col] = __fadd_rn(pre_r[i], v);
        } else if (EPI == EPI_STORE && p.rope_cos) {
            // RoPE as in block32_epilogue, with the cos/sin read up front
            const int hd = p.rope_hd, half = hd >> 1;
            const float other = __shfl_xor(v, half, 64);
            if (row >= M || col >= N) continue;
            if (col < p.rope_cols) {
                const int pc = (int)col % hd;
                v = pc < half ? v * pre_c[i] - other * pre_s[i] : v * pre_c[i] + other * pre_s[i];
            }
            C[row * p.ldc + col] = v;
        } else {
            block32_epilogue<EPI>(p, C, R, row, col, lr, v);
        }
    }
    if (fin) return;
    if (split_last(p, tm * p.tiles_n + tn)) split_reduce_tile(p, m0, n0, 32, 32, 64 * NW);
}

// Waves of a K-split workgroup: one per K step of a split, in multiples of four
// (one per SIMD) up to sixteen: a wave that walked two steps would wait on its
// second step's loads after its first step's MFMAs, and the others on it.
int ksplit_waves(int64_t steps) { return steps <= 4 ? 4 : steps <= 8 ? 8 : steps <= 12 ? 12 : 16; }

template <bool TA, bool TB, int EPI, bool NORM, int MODE>
void launch_ksplit_mode(Context &ctx, const KParams &p, dim3 grid, int nw) {
    if (nw == 4)
        hipLaunchKernelGGL((gemm_f32_mfma_ksplit<TA, TB, EPI, NORM, 4, MODE>), grid, dim3(256), 0,
                           ctx.stream, p);
    else if (nw == 8)
        hipLaunchKernelGGL((gemm_f32_mfma_ksplit<TA, TB, EPI, NORM, 8, MODE>), grid, dim3(512), 0,
                           ctx.stream, p);
    else if (nw == 12)
        hipLaunchKernelGGL((gemm_f32_mfma_ksplit<TA, TB, EPI, NORM, 12, MODE>), grid, dim3(768),
                           0, ctx.stream, p);
    else
        hipLaunchKernelGGL((gemm_f32_mfma_ksplit<TA, TB, EPI, NORM, 16, MODE>), grid, dim3(1024),
                           0, ctx.stream, p);
}

template <bool TA, bool TB, int EPI, bool NORM>
void launch_ksplit_nw(Context &ctx, const KParams &p, dim3 grid, int mode, int nw) {
    if (mode == 2)
        launch_ksplit_mode<TA, TB, EPI, NORM, 2>(ctx, p, grid, nw);
    else if (mode == 1)
        launch_ksplit_mode<TA, TB, EPI, NORM, 1>(ctx, p, grid, nw);
    else
        launch_ksplit_mode<TA, TB, EPI, NORM, 0>(ctx, p, grid, nw);
}

template <bool TA, bool TB, int EPI>
void launch_ksplit(Context &ctx, const KParams &p, dim3 grid, int mode) {
    const int nw = ksplit_waves((p.k_per_split + 31) / 32);
    if constexpr (!TA && !TB && (EPI == EPI_STORE || EPI == EPI_SWIGLU)) {
        if (p.norm_w) {
            launch_ksplit_nw<false, false, EPI, true>(ctx, p, grid, mode, nw);
            return;
        }
    }
    launch_ksplit_nw<TA, TB, EPI, false>(ctx, p, grid, mode, nw);
}

// ---- fp32 MFMA issue-rate probe ---------------------------------------------------
// Every wave runs n MFMAs in 4 independent accumulator chains on register
// operands, with no memory traffic but one store per lane at the end. As in a
// GEMM, the operands change from one MFMA to the next: each lane cycles
// through 8 values with pseudo-random mantissas in [-1, 1) (the matrix
// cores' power, and so the clock they hold, depends on how many operand bits
// toggle; fixed operands run near the peak clock). The result is the rate
// the matrix cores sustain under full MFMA load on GEMM-like data: the
// practical ceiling under the published peak for the GEMM kernels.
__global__ __launch_bounds__(512) void mfma_peak_kernel(float *out, int n, uint32_t seed) {
    floatx16 acc[4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[c][r] = 0.0f;
    float v[8];
    uint32_t h = seed ^ (blockIdx.x * 0x9e3779b9u) ^ (threadIdx.x * 0x85ebca6bu);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        h ^= h << 13;
        h ^= h >> 17;
        h ^= h << 5;
        v[i] = (float)(int32_t)h * (1.0f / 2147483648.0f);
    }
    for (int i = 0; i < n; i += 8) {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            acc[j & 3] = __builtin_amdgcn_mfma_f32_32x32x2f32(v[j], v[(j + 3) & 7], acc[j & 3], 0, 0, 0);
    }
    float s = 0.0f;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int r = 0; r < 16; ++r) s += acc[c][r];
    out[(int64_t)blockIdx.x * blockDim.x + threadIdx.x] = s;
}

template <bool TA, bool TB, int EPI>
void launch(Context &ctx, const KParams &p, dim3 grid) {
    if constexpr (!TA && !TB && (EPI == EPI_STORE || EPI == EPI_SWIGLU)) {
        if (p.norm_w) {
            hipLaunchKernelGGL((gemm_f32_mfma_small<false, false, EPI, true>), grid, dim3(256), 0,
                               ctx.stream, p);
            return;
        }
    }
    hipLaunchKernelGGL((gemm_f32_mfma_small<TA, TB, EPI, false>), grid, dim3(256), 0,
                       ctx.stream, p);
}

template <int EPI>
void dispatch_t(Context &ctx, bool ta, bool tb, const KParams &p, dim3 grid) {
    if (!ta && !tb) launch<false, false, EPI>(ctx, p, grid);
    else if (!ta) launch<false, true, EPI>(ctx, p, grid);
    else launch<true, false, EPI>(ctx, p, grid);
}

bool aligned16(const void *ptr) { return (reinterpret_cast<uintptr_t>(ptr) & 15) == 0; }

}  // namespace

namespace {

int cus_of(const Context &ctx) { return ctx.cu_count > 0 ? ctx.cu_count : 256; }

int64_t big_tiles_of(const GemmDesc &d) {
    return ((d.m + BM - 1) / BM) * ((d.n + BN - 1) / BN) * d.batch;
}

// The fp32 MFMA tiles of 64x64: below one 128x128 tile per CU, for products of
// at most 2^28 multiply-adds (above that the split tiles win: 2048 x 512 x 1024
// 27.0 -> 20.9 us, 256 x 2048 x 1024 21.2 -> 18.6; at 2^28 the two meet, 4096 x
// 512 x 128 10.3 against 13.7 us, 2048 x 128 x 1024 12.9 against 10.0), and
// for the ones that take a norm in with their loads (K <= 256), whose own
// launch costs more than the tiles gain. Also for sums of one step that are added
// into a C of any size: reading C is their time, which a lone large tile per
// CU does after its products, several small ones beside each other's (into 960 x
// 25536 from K 8 55 -> 37 us, 320 x 22528 24 -> 13, 30 shapes 15% on average; from
// K 33 on it is the large tiles', 0 to 30%).
bool use_small(const Context &ctx, const GemmDesc &d) {
    if (d.epi == EPI_ACCUM && d.k <= SBK) return true;
    if (big_tiles_of(d) >= cus_of(ctx)) return false;
    return (d.norm_w && d.k <= 256) || d.m * d.n * d.k <= (int64_t(1) << 28) / d.batch;
}

// When the K-split kernel runs: 1 for the small nn shapes of one matrix whose
// K is at most 15 steps of 32 (one split; the store, accumulate and SwiGLU
// epilogues, with the RMSNorm and RoPE folds) while the 64x64 tiles number
// under two per CU (beyond that the small kernel's grid is deep enough and its
// tiles share their operands through LDS); 2 for the other products of one
// matrix whose 128x128 tiles would not give every CU one and of at most 2^28
// multiply-adds (any form but tt, store or accumulate), split along K across
// workgroups: on the benchmark sweep it wins at 0.27 GFLOP (dA, dB at K = N =
// 256: 27 -> 37 and 13 -> 23 TFLOP/s) and loses from 1 GFLOP up, where the
// other kernels' operand reuse through LDS pays; 0 otherwise.
int ksplit_kind(const Context &ctx, const GemmDesc &d) {
    const int cus = cus_of(ctx);
    const bool plain = d.epi == EPI_STORE || d.epi == EPI_ACCUM;
    const int64_t small_tiles = ((d.m + SBM - 1) / SBM) * ((d.n + SBN - 1) / SBN);
    const int64_t big_tiles = ((d.m + BM - 1) / BM) * ((d.n + BN - 1) / BN);
    if (use_small(ctx, d) && !d.ta && !d.tb && d.batch == 1 && d.k <= 480 &&
        small_tiles < 2 * cus && (plain || d.epi == EPI_SWIGLU))
        return 1;
    if (d.batch == 1 && plain && !d.norm_w &&
        !d.rope_cos && big_tiles < cus && d.m * d.n * d.k <= (int64_t(1) << 28))
        return 2;
    return 0;
}

// K splits of a kind-2 K-split product: the least estimated time, in ns. A CU
// holds 16 waves; a round of workgroups costs 2.7 us to start, sum and store and
// its nw waves 0.3 and 0.27 each for every step they take one after another
// (loads in flight, then the MFMAs); 4.2 and 0.5 where a k-contiguous operand's rows
// are not 16-byte aligned and come one value at a time. The splits' partials meet in
// memory for 1.1 us, 0.75 per split and 2 per MB. A split keeps four steps.
// Fitted to 680 products of up to 2^28 multiply-adds with 1 to 32 splits of
// each: 2.1% from the best on average. (Eight steps a split and one cost per step:
// 4.0%, and products of 20 to 30 steps took 10-30% longer than with two workgroups
// per CU, whatever their length, before that: 41 x 831 x 448 11.1 us, 8.5 so, 100 x 695
// x 68 9.9 / 8.3, 81 x 1978 x 192 12.8 / 10.5. Two per CU: tn 128 x 2048 x 384 13.8, 8.8
// by the estimate, 16 x 7840 x 341 34.3 / 21.6.)
// uncoalesced: both operands k-major, not 16-byte aligned, read one value
// per lane and row: the rows' cache lines bound it, and many small workgroups
// spread them (nt 574x51x723 10.6 us so, 12.6 by an estimate).
int ksplit_splits(int cus, int64_t tiles, int64_t ktiles, int64_t mn, bool unaligned,
                  bool uncoalesced) {
    int best = 1;
    if (tiles > Context::kTickets) return best;  // (a counter per tile)
    if (uncoalesced) {
        while (tiles * best < 2 * (int64_t)cus && best < 64 && ktiles / (best * 2) >= 4) best *= 2;
        return best;
    }
    int64_t least = INT64_MAX;
    for (int s = 1; s <= 64 && (s == 1 || ktiles / s >= 4); s *= 2) {
        const int64_t steps = (ktiles + s - 1) / s, nw = ksplit_waves(steps);
        const int64_t wgs = cus * (16 / nw), rounds = (tiles * s + wgs - 1) / wgs;
        const int64_t start = unaligned ? 4200 : 2700, wave = unaligned ? 500 : 270;
        const int64_t cost = rounds * (start + (steps + nw - 1) / nw * (300 + wave * nw)) +
                             (s > 1 ? 1100 + 750 * s + s * mn * 8 / 1000 : 0);
        if (cost < least) {
            least = cost;
            best = s;
        }
    }
    return best;
}

bool vec_a_of(const GemmDesc &d, const float *a, int64_t lda) {
    const int64_t off_limit = int64_t(1) << 29;  // interior byte offsets stay below 2^31
    return (lda % 4 == 0) && (d.batch == 1 || d.stride_a % 4 == 0) && aligned16(a) &&
           lda * BM < off_limit;
}

}  // namespace

GemmFusion gemm_fusion(const Context &ctx, const GemmDesc &d) {
    GemmFusion f;
    const bool small = use_small(ctx, d);
    const bool nn = !d.ta && !d.tb && d.batch == 1 && d.k % 4 == 0 &&
                    vec_a_of(d, d.a, d.lda) && aligned16(d.norm_w) &&
                    (d.epi == EPI_STORE || d.epi == EPI_SWIGLU);
    if (small) {
        f.norm = nn && d.k <= 256;
        f.rope = d.batch == 1 && d.epi == EPI_STORE && d.rope_hd > 0 && d.rope_hd <= 32 &&
                 32 % d.rope_hd == 0;
    } else {
        // the large tiles rotate heads of 64 or 128 columns in registers; the
        // norm stays a kernel of its own (in their loads it would be redone by
        // every column of tiles)
        f.rope = !d.ta && !d.tb && d.batch == 1 && d.epi == EPI_STORE &&
                 (d.rope_hd == 64 || d.rope_hd == 128);
    }
    return f;
}

int64_t gemm_ce_tiles(const Context &ctx, const GemmDesc &d) {
    if (use_small(ctx, d) || d.batch != 1 || d.ta || d.norm_w || d.rope_cos)
        return 0;
    return (d.n + BN - 1) / BN;
}

namespace {

struct TilePlan {
    int tile = TILE_128, splits = 1;
};

// Split partials of the large tiles stay below this: the no-alloc entry point's
// array holds them too, so both entry points take the same plan.
constexpr int64_t kSplitBytes = kNoallocScratchBytes;
constexpr int kMaxTileSplits = 16;

// The tile and the K splits that an estimate of the launch makes shortest: with
// G workgroups and q = ceil(G / CUs) on the busiest CU, 16 of K take
// max(q * alone, G / CUs * full) us (kGemmTiles: a lone workgroup is bound by
// its own steps, a full chip by its power), a tile's first loads and epilogue
// some steps more (setup), and split sums a launch and the partials written and
// read at 3.5 TB/s. Measured constants,
// f32 TFLOP/s in brackets: 256x256 from 4096 x 2048 x 4096 on (220-228 against
// 204-206 for 256x128), 256x128 for the grids of 100 to 500 of them (4096 x
// 2048 x 2048: 197-202; 256x256 150, 128x128 174), 128x128 around one tile per
// CU (1000 x 768 x 3072: 36.9 us against 40.9 and 41.8 for its neighbours),
// 128x64 and 64x64 below (2048 x 512 x 1024 20.9 us against 32 for 128x128);
// 1024 x 2048 x 4096 takes two splits of 256x128 (102 us against 117 whole).
// Split counts other than 2, 4 and 8 fill the CUs that a halving leaves idle
// (2816 x 2688 x 324: 3 splits 45 us, 2 splits 71; 976 x 3694 x 1046 65 / 91;
// 150 x 7999 x 4224 102 / 139; 508 x 7168 x 128: 16 splits 18.3, 8 splits
// 22.3). They are taken when the estimate is 4% lower: where it gains less,
// half of the products measured got slower by up to 10% (919 x 7189 x 490 57 ->
// 61, 128 x 1664 x 3648 21 -> 23). Past 8 the sums of a split's partials wait
// on memory once more per four of them, 0.2 us each.
// The setups decide where K is a few steps: counted as 6 for every tile, 128x128
// and 256x256 ones took over from 256x128 (2050 x 64 x 4100 29.5 us, 22.5 so; 7552 x 33
// x 3763 57 / 51, 2142 x 90 x 1728 27 / 16). Over 260 products of K 33 to 4096 the
// choice is 0.9% from the best tile of each, 2.9% with 6 for all. (even: 6 for all.)
TilePlan fastest_tile(const Context &ctx, const KParams &p, int64_t batch, int epi, int first,
                      bool even) {
    const bool may_split = batch == 1 && (epi == EPI_STORE || epi == EPI_ACCUM) && !p.rope_cos;
    const double cus = cus_of(ctx), ksteps = (double)((p.k + BK - 1) / BK);
    TilePlan best[2];  // of the halvings of K, of the other split counts
    double best_us[2] = {0.0, 0.0};
    for (int tile = first; tile < TILE_COUNT; ++tile) {
        if (!gemm_tile_takes(p, epi, tile)) continue;
        const GemmTileInfo &t = kGemmTiles[tile];
        const double tiles = (double)((p.m + t.rows - 1) / t.rows) *
                             (double)((p.n + t.cols - 1) / t.cols) * (double)batch;
        for (int s = 1; s <= kMaxTileSplits; ++s) {
            // a split keeps 128 of K, as many as its prologue costs
            if (s > 1 && (!may_split || p.k < 128 * s || s * p.m * p.n * 4 > kSplitBytes)) break;
            const double g = tiles * s, setup = even ? 6.0 : t.setup;
            double us = std::max(std::ceil(g / cus) * t.alone, g / cus * t.full) * (ksteps / s + setup);
            if (s > 1) us += 4.0 + (double)(s + 1) * (double)(p.m * p.n) * 4.0 / 3.5e6;
            if (s > 8) us += 0.2 * (s - 8);
            const int fine = s > 8 || (s & (s - 1)) ? 1 : 0;
            if (best_us[fine] == 0.0 || us < best_us[fine]) {
                best_us[fine] = us;
                best[fine].tile = tile;
                best[fine].splits = s;
            }
        }
    }
    return best_us[1] > 0.0 && best_us[1] < 0.96 * best_us[0] ? best[1] : best[0];
}

// The 256x256 tile's sums round six times per 16 of K, the others' once. It is
// taken where its steps win, not for its setup: the products of 92 to 480 of K that
// the setups alone would move to it gain 4-18% over 256x128 and lose a factor of
// 2.8 in precision.
TilePlan choose_tile(const Context &ctx, const KParams &p, int64_t batch, int epi) {
    const TilePlan best = fastest_tile(ctx, p, batch, epi, TILE_256, false);
    if (best.tile != TILE_256 || fastest_tile(ctx, p, batch, epi, TILE_256, true).tile == TILE_256)
        return best;
    return fastest_tile(ctx, p, batch, epi, TILE_256x128, false);
}

// mmh_gemm_noalloc's contract: which products it takes is stated in terms of a
// plan of 128x128 tiles (the split that gives every CU a tile, or the last
// tiles cut along K where they leave CUs idle) and its partials, and a product
// that this plan cannot hold in 16 MiB is refused, whatever the kernels need.
void check_noalloc(const Context &ctx, const GemmDesc &d) {
    const int64_t cus = cus_of(ctx), limit = kNoallocLimitBytes;
    const int64_t big = ((d.m + BM - 1) / BM) * ((d.n + BN - 1) / BN);
    auto splits_of = [&](int64_t tiles, int64_t step) {
        const int64_t steps = (d.k + step - 1) / step;
        int64_t s = 1;
        while (tiles * s < cus && s < 16 && steps / (s * 2) >= 8) s *= 2;
        const int64_t per = (steps + s - 1) / s;
        return (steps + per - 1) / per;
    };
    auto refuse_over = [&](int64_t splits) {
        const int64_t need = splits * d.m * d.n * 4;
        if (splits > 1 && need > limit)
            fail(MMH_ERR_SHAPE, "gemm: the split-K partials of a " + std::to_string(d.m) + " x " +
                                    std::to_string(d.n) + " product (" + std::to_string(splits) +
                                    " splits of 128x128 tiles) need " + std::to_string(need) +
                                    " bytes; the scratch holds " + std::to_string(limit) +
                                    " of such a plan");
        return splits > 1;
    };
    if (big < cus) {
        // (partials of products this small, and of nn products with K up to
        // 480, always fit: none, or at most K / 128 of them)
        const int64_t mnk = d.m * d.n * d.k, tiles = ((d.m + 63) / 64) * ((d.n + 63) / 64);
        if (mnk <= (int64_t(1) << 28)) return;
        if (d.k <= 1024 || (d.k <= 2048 && mnk <= (int64_t(1) << 29))) {
            if (d.ta || d.tb || d.k > 480 || tiles >= 2 * cus) refuse_over(splits_of(tiles, 32));
            return;
        }
    }
    const int64_t steps = (d.k + BK - 1) / BK;
    if (refuse_over(splits_of(big, BK))) return;
    const int64_t q = big / cus, r = big % cus;
    if (q < 1 || r == 0) return;
    int best_s = 1;
    double best = (double)(q + 1);
    for (int t : {2, 3, 4, 6, 8}) {
        if (steps / t < 16) break;
        const double span = (double)q + (double)((r * t + cus - 1) / cus) / t;
        if (span < best - 1e-9) {
            best = span;
            best_s = t;
        }
    }
    const int64_t need = r * best_s * BM * BN * 4;
    if (best_s > 1 && best <= 0.95 * (double)(q + 1) && need > limit)
        fail(MMH_ERR_SHAPE, "gemm: the tail pieces of a " + std::to_string(d.m) + " x " +
                                std::to_string(d.n) + " product (" + std::to_string(r) +
                                " tiles x " + std::to_string(best_s) + " pieces) need " +
                                std::to_string(need) + " bytes; the scratch holds " +
                                std::to_string(limit) + " of such a plan");
}

}  // namespace

void gemm(Context &ctx, const GemmDesc &d) {
    if (d.m <= 0 || d.n <= 0 || d.k <= 0 || d.batch <= 0) fail(MMH_ERR_SHAPE, "gemm: empty shape");
    if (d.ta && d.tb) fail(MMH_ERR_ARGUMENT, "gemm: one operand at most is transposed");
    if (d.epi == EPI_CE && (gemm_ce_tiles(ctx, d) == 0 || !d.ce_targets || !d.ce_part || !d.ce_zt))
        fail(MMH_ERR_ARGUMENT, "gemm: the loss folds only into the large tiles of one matrix");
    KParams p{};
    p.a = d.a;
    p.b = d.b;
    p.c = d.c;
    p.m = d.m;
    p.n = d.n;
    p.k = d.k;
    p.lda = d.lda;
    p.ldb = d.ldb;
    p.ldc = d.ldc;
    p.stride_a = d.stride_a;
    p.stride_b = d.stride_b;
    p.stride_c = d.stride_c;
    p.swiglu_ff = d.swiglu_ff;
    p.resid = d.resid;
    p.aux = d.aux;
    p.ldaux = d.ldaux;
    p.ce_targets = d.ce_targets;
    p.ce_part = d.ce_part;
    p.ce_zt = d.ce_zt;
    p.ce_tiles = (int)((d.n + BN - 1) / BN);
    if (d.accumulate_into_c && (d.epi != EPI_ACCUM || d.resid))
        fail(MMH_ERR_ARGUMENT, "gemm: accumulate_into_c takes EPI_ACCUM into C itself");
    p.acc_init = d.accumulate_into_c ? -0.0f : 0.0f;
    if (d.epi == EPI_SWIGLU_BWD || (d.epi == EPI_SWIGLU && d.aux)) {
        if (!d.aux || d.ldaux < (d.epi == EPI_SWIGLU ? d.n : 2 * d.n) || d.ldaux % 4 ||
            !aligned16(d.aux) ||
            (d.epi == EPI_SWIGLU_BWD && (d.ldc % 4 || !aligned16(d.c))))
            fail(MMH_ERR_ARGUMENT, "gemm: swiglu pairs need 16-byte aligned rows of >= 2n");
        if (d.batch != 1) fail(MMH_ERR_ARGUMENT, "gemm: swiglu epilogues take one matrix");
    }
    const int cus = cus_of(ctx);
    p.libm_exp = big_tiles_of(d) < cus;
    const bool small = use_small(ctx, d);
    const int kind = ksplit_kind(ctx, d);
    const bool ksplit = kind != 0;
    const bool tiled = !small && !ksplit;
    const GemmFusion fuse = gemm_fusion(ctx, d);
    if (d.scratch) check_noalloc(ctx, d);
    // The interior path addresses a tile with byte offsets below 2^31.
    const int64_t off_limit = int64_t(1) << 29;
    p.vec_a = vec_a_of(d, d.a, d.lda);
    p.vec_b = (d.ldb % 4 == 0) && (d.batch == 1 || d.stride_b % 4 == 0) && aligned16(d.b) &&
              d.ldb * BN < off_limit;
    p.vec_c = (d.ldc % 2 == 0) && (d.batch == 1 || d.stride_c % 2 == 0) &&
              (reinterpret_cast<uintptr_t>(d.c) & 7) == 0;

    // RMSNorm of A: in the small kernel's loads, or first as its own kernel.
    if (d.norm_w) {
        if (d.ta || d.batch != 1)
            fail(MMH_ERR_ARGUMENT, "gemm: the A-row norm takes one row-major A");
        if (fuse.norm) {
            p.norm_w = d.norm_w;
            p.norm_eps = d.norm_eps;
        } else {
            if (!d.norm_tmp) fail(MMH_ERR_ARGUMENT, "gemm: the A-row norm needs norm_tmp");
            launch_rms_norm(ctx, d.a, d.norm_w, d.m, d.k, d.norm_eps, d.norm_tmp);
            p.a = d.norm_tmp;
            p.lda = d.k;
            p.vec_a = vec_a_of(d, d.norm_tmp, d.k);
        }
    }

    // RoPE in the small and large tiles' epilogues (gemm_fusion), where the K
    // is not split.
    const bool rope = d.rope_cos != nullptr;
    if (rope) {
        if (d.batch != 1 || d.rope_hd <= 0 || d.rope_hd % 2 || d.rope_seq <= 0 ||
            d.m % d.rope_seq || d.rope_cols % d.rope_hd || d.rope_cols > d.n || !d.rope_sin ||
            d.m > INT32_MAX || d.n > INT32_MAX)
            fail(MMH_ERR_ARGUMENT, "gemm: bad rope arguments");
        if (fuse.rope) {
            p.rope_cos = d.rope_cos;
            p.rope_sin = d.rope_sin;
            p.rope_seq = (int)d.rope_seq;
            p.rope_hd = (int)d.rope_hd;
            p.rope_cols = (int)d.rope_cols;
        }
    }

    TilePlan plan;
    if (tiled) plan = choose_tile(ctx, p, d.batch, d.epi);
    const int64_t tile_m = ksplit ? 32 : tiled ? kGemmTiles[plan.tile].rows : SBM;
    const int64_t tile_n = ksplit ? 32 : tiled ? kGemmTiles[plan.tile].cols : SBN;
    p.tiles_m = (int)((d.m + tile_m - 1) / tile_m);
    p.tiles_n = (int)((d.n + tile_n - 1) / tile_n);
    const int64_t tiles = (int64_t)p.tiles_m * p.tiles_n;
    const int64_t kstep = ksplit ? 32 : tiled ? BK : SBK;
    const int64_t ktiles = (d.k + kstep - 1) / kstep;
    int splits = 1;
    if (tiled) {
        splits = plan.splits;
    } else if (kind == 2) {
        splits = ksplit_splits(cus, tiles, ktiles, d.m * d.n,
                               (!d.ta && !p.vec_a) || (d.tb && !p.vec_b),
                               !d.ta && d.tb && !(p.vec_a && p.vec_b));
    } else if (!ksplit && d.batch == 1 && d.epi != EPI_SWIGLU && d.epi != EPI_SWIGLU_BWD) {
        // Split only while a split keeps >= 8 steps of 32 (the reduce
        // launch costs about what 8 steps do) and the grid is below a
        // workgroup per CU.
        while (tiles * splits < cus && splits < 16 && ktiles / (splits * 2) >= 8)
            splits *= 2;
    }
    if (d.batch > 1 || d.epi == EPI_SWIGLU || d.epi == EPI_SWIGLU_BWD || d.epi == EPI_CE ||
        p.norm_w || p.rope_cos || kind == 1)
        splits = 1;
    const int64_t kt_per = (ktiles + splits - 1) / splits;
    p.k_per_split = kt_per * kstep;
    splits = (int)((ktiles + kt_per - 1) / kt_per);
    p.splits = splits;
    if (d.plan) {
        d.plan[0] = (int32_t)tile_m;
        d.plan[1] = (int32_t)tile_n;
        d.plan[2] = splits;
        return;
    }
    if (splits > 1) {
        // 64x64 and 32x32 tiles: the last split of each tile sums the
        // partials in split order and applies the epilogue (one launch; such
        // grids have less than a 128x128 tile per CU, so at most sixteen
        // 32x32 tiles per CU: within the counters); the large tiles:
        // splitk_reduce after the launch
        if (!tiled) {
            p.tickets = d.scratch ? d.scratch_tickets : ctx.tickets;
            if (!p.tickets || tiles > Context::kTickets)
                fail(MMH_ERR_OTHER, "gemm: no split counters for " + std::to_string(tiles) + " tiles");
            p.split_accum = d.epi == EPI_ACCUM ? 1 : 0;
        }
        const size_t need_bytes = (size_t)splits * d.m * d.n * 4;
        if (d.scratch) {
            if (need_bytes > d.scratch_bytes)  // (check_noalloc and kSplitBytes rule it out)
                fail(MMH_ERR_OTHER, "gemm: the split-K partials do not fit the scratch");
            p.partial = d.scratch;
        } else {
            p.partial = static_cast<float *>(ctx.get_scratch(need_bytes));
        }
    }

    const int epi = splits > 1 ? EPI_STORE : d.epi;
    if (tiles > 0x7fffffff || d.batch > 65535) fail(MMH_ERR_SHAPE, "gemm: grid too large");
    dim3 grid((unsigned)tiles, (unsigned)d.batch, (unsigned)splits);
    if (ksplit) {
        // The k-contiguous operands (A when !ta, B when tb, the norm weights)
        // decide between vector and predicated reads (vec_a / vec_b hold
        // ld % 4 == 0 and a 16-byte aligned base).
        const bool vec = (d.ta || p.vec_a) && (!d.tb || p.vec_b) &&
                         (!p.norm_w || aligned16(p.norm_w));
        const int mode = !vec ? 0 : d.k % 32 == 0 ? 2 : 1;
        if (epi == EPI_SWIGLU)
            launch_ksplit<false, false, EPI_SWIGLU>(ctx, p, grid, mode);
        else if (!d.ta && !d.tb)
            (epi == EPI_ACCUM ? launch_ksplit<false, false, EPI_ACCUM>
                              : launch_ksplit<false, false, EPI_STORE>)(ctx, p, grid, mode);
        else if (!d.ta)
            (epi == EPI_ACCUM ? launch_ksplit<false, true, EPI_ACCUM>
                              : launch_ksplit<false, true, EPI_STORE>)(ctx, p, grid, mode);
        else
            (epi == EPI_ACCUM ? launch_ksplit<true, false, EPI_ACCUM>
                              : launch_ksplit<true, false, EPI_STORE>)(ctx, p, grid, mode);
    } else if (tiled) {
        launch_gemm_tiles(ctx, p, grid, d.ta, d.tb, epi, plan.tile);
    } else if (epi == EPI_SWIGLU) {
        if (d.ta || d.tb) fail(MMH_ERR_ARGUMENT, "gemm: swiglu epilogue needs the nn form");
        launch<false, false, EPI_SWIGLU>(ctx, p, grid);
    } else if (epi == EPI_SWIGLU_BWD) {
        if (d.ta || !d.tb) fail(MMH_ERR_ARGUMENT, "gemm: swiglu backward epilogue needs the nt form");
        launch<false, true, EPI_SWIGLU_BWD>(ctx, p, grid);
    } else if (epi == EPI_ACCUM) {
        dispatch_t<EPI_ACCUM>(ctx, d.ta, d.tb, p, grid);
    } else {
        dispatch_t<EPI_STORE>(ctx, d.ta, d.tb, p, grid);
    }
    check_hip(hipGetLastError(), "gemm launch");
    if (splits > 1 && !p.tickets) launch_splitk_reduce(ctx, p, d.epi);
    if (rope && !p.rope_cos)
        launch_rope_strided(ctx, d.c, d.rope_seq * d.ldc, d.rope_hd, d.ldc, d.m / d.rope_seq,
                            d.rope_cols / d.rope_hd, d.rope_seq, d.rope_hd, d.rope_cos,
                            d.rope_sin);
}

double mfma_peak_tflops(Context &ctx) {
    // two 512-thread workgroups per CU (4 waves per SIMD), 8192 MFMAs per wave
    // (about 0.5 ms a launch); 20 launches first bring the clock to its
    // steady state under this load, then 40 are timed
    const int blocks = 2 * cus_of(ctx), threads = 512, n = 8192;
    float *out = static_cast<float *>(ctx.get_scratch((size_t)blocks * threads * 4));
    for (int i = 0; i < 20; ++i)
        hipLaunchKernelGGL(mfma_peak_kernel, dim3(blocks), dim3(threads), 0, ctx.stream, out, n,
                           1u + (uint32_t)i);
    check_hip(hipGetLastError(), "mfma probe launch");
    const int reps = 40;
    check_hip(hipEventRecord(ctx.t0, ctx.stream), "event record");
    for (int i = 0; i < reps; ++i)
        hipLaunchKernelGGL(mfma_peak_kernel, dim3(blocks), dim3(threads), 0, ctx.stream, out, n,
                           100u + (uint32_t)i);
    check_hip(hipGetLastError(), "mfma probe launch");
    check_hip(hipEventRecord(ctx.t1, ctx.stream), "event record");
    check_hip(hipEventSynchronize(ctx.t1), "event sync");
    float ms = 0.0f;
    check_hip(hipEventElapsedTime(&ms, ctx.t0, ctx.t1), "elapsed time");
    const double flops = 2.0 * 32 * 32 * 2 * (double)n * (blocks * threads / 64) * reps;
    return flops / (ms * 1e-3) / 1e12;
}

}  // namespace mmh
