// Shared by the attention kernels: the launch parameters.
#pragma once

#include "mmh_internal.h"

namespace mmh {

struct AttnP {
    const float *q, *k, *v;
    float *out;
    float *lse;
    int64_t sqb, sqh, sqt, skb, skh, skt, svb, svh, svt, sob, soh, sot;
    int h, hkv, t, nqb;
    float scale;
};

// attention_split.hip: heads of 64 or 128, p.nqb blocks of 128 query rows,
// 16-byte aligned rows, T * stride below 2^29 floats for k and v.
void launch_attention_split(Context &ctx, const AttnP &p, int64_t b, int64_t hd);

struct BwdP {
    const float *q, *k, *v, *o, *dout, *lse;
    float *dq, *dk, *dv, *dvec;
    int64_t sqb, sqh, sqt, skb, skh, skt, svb, svh, svt, sob, soh, sot;
    float *part;  // per-query-head partial dK, dV [2][B][H][T][hd], or null
    int h, hkv, t, nqb, nkb;
    float scale;
};

// attention_bwd_split.hip: heads of 64 or 128, 32-bit element offsets (off32 in
// backward_kernels); dq also writes dvec, which dkv reads.
void launch_attention_bwd_split(Context &ctx, const BwdP &p, int64_t b, int64_t hd);

}  // namespace mmh
