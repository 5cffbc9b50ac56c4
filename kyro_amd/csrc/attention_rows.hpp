// Device helpers the attention kernels share: a sequence's row geometry, validated block ids,
// output stores and the merge of one row's partial states.
#pragma once

#include "common.hpp"

namespace kyro {

struct SeqInfo {
    int b, kvh, q0, q_len, rows, nblk;
    int ctx;
    bool ok;
};

// Output row of local row n (n = j * group + head-in-group) of a sequence.
__device__ __forceinline__ size_t out_row(const AttnArgs& a, const SeqInfo& si, int n) {
    const int j = n / a.group;
    const int hg = n - j * a.group;
    return (size_t)(si.q0 + j) * a.H + (size_t)si.kvh * a.group + hg;
}

__device__ __forceinline__ int64_t checked_block(const AttnArgs& a, int b, int i) {
    const int64_t blk = a.table[(size_t)b * a.max_blocks + i];
    if (blk < 0 || blk >= a.num_blocks) {
        latch_error(a.err, ERR_BLOCK_ID);
        return -1;
    }
    return blk;
}

template <int D>
__device__ __forceinline__ void store_row4(const AttnArgs& a, size_t row, int d, float x0, float x1,
                                           float x2, float x3) {
    if (a.out_bf16) {
        uint2 w;
        w.x = pack_bf16x2(x0, x1);
        w.y = pack_bf16x2(x2, x3);
        *reinterpret_cast<uint2*>(reinterpret_cast<uint16_t*>(a.out) + row * D + d) = w;
    } else {
        *reinterpret_cast<float4*>(reinterpret_cast<float*>(a.out) + row * D + d) =
            make_float4(x0, x1, x2, x3);
    }
}

// Merges the nsplit partial states of one output row (workspace rows r0 + s * stride) into this
// thread's four columns d .. d + 3 and stores them. The loads of kMergeBatch splits are issued
// together (a split index past the last reads the last split again and is dropped), so a row with
// up to kMergeBatch splits costs one memory round trip; longer rows merge batch after batch with
// the usual running-max rescale (for one batch this is the plain two-pass formula).
constexpr int kMergeBatch = 16;
template <int D>
__device__ __forceinline__ void merge_row(const AttnArgs& a, const SeqInfo& si, int n, int d, size_t r0,
                                          size_t stride, int nsplit) {
    float M = kNegInf, L = 0.f;
    float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = 0; s0 < nsplit; s0 += kMergeBatch) {
        float m[kMergeBatch], l[kMergeBatch];
        float4 v[kMergeBatch];
#pragma unroll
        for (int i = 0; i < kMergeBatch; ++i) {
            const size_t r = r0 + (size_t)min(s0 + i, nsplit - 1) * stride;
            m[i] = a.ws_m[r];
            l[i] = a.ws_l[r];
            v[i] = *reinterpret_cast<const float4*>(a.ws_acc + r * D + d);
        }
        float mb = M;
#pragma unroll
        for (int i = 0; i < kMergeBatch; ++i) mb = s0 + i < nsplit ? fmaxf(mb, m[i]) : mb;
        if (mb == kNegInf) continue;  // nothing visible so far
        if (M != kNegInf) {
            const float f = fast_exp2(M - mb);
            L *= f;
            acc.x *= f;
            acc.y *= f;
            acc.z *= f;
            acc.w *= f;
        }
        M = mb;
#pragma unroll
        for (int i = 0; i < kMergeBatch; ++i) {
            const float w = s0 + i < nsplit ? fast_exp2(m[i] - M) : 0.f;
            L += w * l[i];
            acc.x += w * v[i].x;
            acc.y += w * v[i].y;
            acc.z += w * v[i].z;
            acc.w += w * v[i].w;
        }
    }
    const float inv = L > 0.f ? 1.f / L : 0.f;
    store_row4<D>(a, out_row(a, si, n), d, acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
}

}  // namespace kyro
