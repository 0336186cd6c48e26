// kvrt_prefill.hip — prefill instantiations of head_dim 64 and 128 (MFMA results
// in VGPRs), the key-split merge and the dispatch.
#include "kvrt_prefill.h"

namespace kvrt {

// Merge of a key-split prefill: one thread per (item, q head, query) row and
// 4 consecutive dims (16-byte partial loads; D is a power of two, dshift =
// log2(D / 4)), the n_ksplit partials in key order, bf16 out. Per dim the
// arithmetic is merge_partials<1>'s (batches of 16 in partial order).
__global__ __launch_bounds__(256) void prefill_merge_kernel(PrefillArgs a, int D, int dshift, int64_t outs4) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= outs4) return;
    const int64_t row = t >> dshift;  // (item, q head, query)
    const int d = (int)(t & ((1 << dshift) - 1)) * 4;
    const int nks = a.n_ksplit;
    const float2 *ml = a.part_ml + row * nks;
    const float *po = a.part_o + row * nks * D + d;
    constexpr int B = 16;
    float M = kNegBig, L = 0.f;
    float4 O = make_float4(0.f, 0.f, 0.f, 0.f);
    for (int s0 = 0; s0 < nks; s0 += B) {
        float2 m[B];
        float4 v[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const int sp = s0 + u;
            m[u] = make_float2(kNegBig, 0.f);
            v[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            if (sp < nks) {
                m[u] = ml[sp];
                v[u] = *reinterpret_cast<const float4 *>(po + (int64_t)sp * D);
            }
        }
        float bm = M;
#pragma unroll
        for (int u = 0; u < B; ++u) bm = fmaxf(bm, m[u].x);
        const float c = __builtin_amdgcn_exp2f(M - bm);
        L *= c;
        O.x *= c;
        O.y *= c;
        O.z *= c;
        O.w *= c;
        M = bm;
#pragma unroll
        for (int u = 0; u < B; ++u) {
            const float w = __builtin_amdgcn_exp2f(m[u].x - M);
            L = fmaf(m[u].y, w, L);
            O.x = fmaf(v[u].x, w, O.x);
            O.y = fmaf(v[u].y, w, O.y);
            O.z = fmaf(v[u].z, w, O.z);
            O.w = fmaf(v[u].w, w, O.w);
        }
    }
    const bool any = !(L == 0.f);  // no key: 0; a NaN sum stays NaN, as without a split
    const uint2 packed = make_uint2(pack_bf16x2(any ? O.x / L : 0.f, any ? O.y / L : 0.f),
                                    pack_bf16x2(any ? O.z / L : 0.f, any ? O.w / L : 0.f));
    *reinterpret_cast<uint2 *>(a.out + row * D + d) = packed;
}

// The key-split merge: (item, q head, query) rows x D / 4 threads.
static hipError_t launch_prefill_merge(const PrefillArgs &a, int head_dim, hipStream_t s) {
    if (head_dim < 4 || (head_dim & (head_dim - 1)) != 0) return hipErrorInvalidValue;
    int dshift = 0;
    while ((1 << dshift) < head_dim / 4) ++dshift;
    const int64_t outs4 = (int64_t)a.n_items * a.kv.kv_heads * a.group * a.qn * (head_dim / 4);
    hipLaunchKernelGGL(prefill_merge_kernel, dim3((unsigned)((outs4 + 255) / 256)), dim3(256), 0, s, a, head_dim,
                       dshift, outs4);
    return hipGetLastError();
}


hipError_t launch_prefill(const PrefillArgs &a, int head_dim, hipStream_t s) {
    if (a.group <= 0 || a.qn <= 0 || a.n_items <= 0) return hipErrorInvalidValue;
    if (a.n_ksplit < 1 || (a.n_ksplit > 1 && (!a.part_o || !a.part_ml))) return hipErrorInvalidValue;
    if (a.kv.layout == KVRT_LAYOUT_RING && a.kv.rows < kPfKeys) return hipErrorInvalidValue;
    if (a.short_heads > 0) return launch_prefill_short(a, head_dim, s);
    const int rw = a.row_waves, ks = a.key_parts;
    hipError_t e = hipErrorInvalidValue;
    const auto shapes = [&](auto d_c) {
        constexpr int D = decltype(d_c)::value;
        if (rw == 4 && ks == 1) return launch_prefill_shape<D, 4, 1, 2>(a, s);
        if (rw == 2 && ks == 2) return launch_prefill_shape<D, 2, 2, 2>(a, s);
        if (rw == 2 && ks == 4) return launch_prefill_shape<D, 2, 4, 2>(a, s);
        if (rw == 1 && ks == 4 && a.kv.layout == KVRT_LAYOUT_CONTIG)
            return launch_prefill_layout<D, 1, 4, 2, KVRT_LAYOUT_CONTIG>(a, s);
        if (rw == 1 && ks == 4 && a.kv.layout == KVRT_LAYOUT_RING)
            return launch_prefill_layout<D, 1, 4, 2, KVRT_LAYOUT_RING>(a, s);
        return hipErrorInvalidValue;
    };
    if (head_dim == 64) {
        e = shapes(std::integral_constant<int, 64>{});
    } else if (head_dim == 128) {
        e = shapes(std::integral_constant<int, 128>{});
    } else {
        e = launch_prefill_wide(a, head_dim, s);
    }
    if (e != hipSuccess || a.n_ksplit == 1) return e;
    return launch_prefill_merge(a, head_dim, s);
}

}  // namespace kvrt
