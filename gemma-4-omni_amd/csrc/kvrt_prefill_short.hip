// kvrt_prefill_short.hip — prefill of head_dim 64 and 128 over few keys (CONTIG
// and RING layers): 16-query tiles.
//
// A wave holds 16 queries of one head, so a 32-key tile is half the MFMA chain
// and half the softmax of a 32-row block of kvrt_prefill.h, and few rows still
// give several workgroups. Where a chunk is one chain of a few tiles (launch,
// first loads, tile, output), that is what bounds it; over more keys the
// 32-row blocks' pipelining and halved LDS traffic win (dispatch in
// kvrt_attend_prefill_async).
//
// Wave w of a workgroup computes head w % heads over key part (w / heads) % KS
// of query block w / (heads KS): tile j of 32 keys goes to part j % KS, QB
// blocks share the staged tiles, and the parts are combined through LDS at the
// end. Per tile and wave, at head_dim 128 (half the products at 64):
//   S^T (32 keys x 16 queries) = K Q^T   8 v_mfma_f32_16x16x32_bf16
//   online softmax per query (fp32, exp2 domain)
//   O^T (128 x 16) += V^T P^T            16 v_mfma_f32_16x16x32_bf16 (P in two bf16 terms)
#include "kvrt_wave.h"

namespace kvrt {

constexpr int kPsGroups = 2;  // groups of KS tiles in the ring: one computed, the next in flight

static __device__ __forceinline__ f32x4_t mfma16(uint4 a, uint4 b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                   c, 0, 0, 0);
}

// Key of MFMA row i of S^T block b within a 32-key tile: lane group G then
// holds the scores of keys 8G .. 8G + 7 across the two blocks, the keys of its
// B operand in V^T P^T.
__device__ __forceinline__ int ps_key(int b, int i) { return 8 * (i >> 2) + 4 * b + (i & 3); }
// Chunk swizzle of the unpadded stages (16-B chunk c of row r at c ^ ps_swz<D>(r)):
// on 64 banks of 4 B the 16 rows of one S^T operand read and the 8 rows x 2
// chunks of a transposed V read each hit 16 places of 16 B (a row takes all 16
// at head_dim 128, half of them at 64). Bit 2 is unused: rows r and r + 4, the
// halves of a transposed read, share the swizzle.
template <int D>
__device__ __forceinline__ int ps_swz(int r) {
    return D == 128 ? ((r & 3) << 1) | (((r >> 3) & 1) << 3) | ((r >> 4) & 1)
                    : (r & 2) | (((r >> 3) & 1) << 2) | ((r >> 4) & 1);
}

// Element offset (from the layer's base) of key t0 + kr of a tile; keys at or
// past kend read key kclamp.
template <int D, int LAYOUT>
__device__ __forceinline__ int64_t ps_row_offset(const KVView &kv, int slot, int kvh, int t0, int kclamp, int kend,
                                                 int kr) {
    const int key = t0 + kr;
    const int64_t base = (int64_t)slot * kv.slot_stride + (int64_t)kvh * kv.head_stride;
    if constexpr (LAYOUT == KVRT_LAYOUT_CONTIG) {
        return base + (int64_t)(key < kend ? key : kclamp) * D;
    } else {
        const int r0 = t0 % kv.rows, rs = kclamp % kv.rows;
        int rk = r0 + kr;  // rows of a tile wrap at most once
        rk = rk >= kv.rows ? rk - kv.rows : rk;
        return base + (int64_t)(key < kend ? rk : rs) * D;
    }
}

template <int D, int LAYOUT, int NW, int KS, int QB>
__global__ __launch_bounds__(64 * NW) void prefill_short_kernel(PrefillArgs a) {
    constexpr int NS = KS * kPsGroups, STAGE = kPfKeys * D;  // stages of K (and V), elements of one
    static_assert((KS - 1) * (NW / KS) * 16 * D * 4 <= NS * STAGE * 2, "the parts' accumulators fit the stages");
    __shared__ __align__(16) uint16_t sk[NS * STAGE];
    __shared__ __align__(16) uint16_t sv[NS * STAGE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 15, grp = lane >> 4;
    const int hw = a.short_heads;
    int nhb, rem, hidx, wrest, kvh, hb;
    udivmod_uniform(a.group, hw, nhb, rem);
    udivmod_uniform(wave, hw, wrest, hidx);
    const int part = wrest % KS, qsub = QB > 1 ? wrest / KS : 0;
    udivmod_uniform(blockIdx.x, nhb, kvh, hb);
    const int item = blockIdx.y;
    const int qb = gridDim.z - 1 - blockIdx.z;  // the blocks that see the most keys start first
    const int g = a.group, hq = a.kv.kv_heads * g;
    const bool computes = wave < hw * KS * QB;
    const int head = kvh * g + hb * hw + (computes ? hidx : 0);
    const int slot = a.slots[item];
    const int L = a.len.lens[(int64_t)slot * a.len.stride + a.len.offset];
    int plen;  // prefix-attention mask of the slot
    uint32_t pw;
    load_prefix(a.pmask, slot, lane, plen, pw);
    const int Qn = a.qn;
    const int qrow0 = (qb * QB + qsub) * 16, qr = qrow0 + col;  // this wave's block, this lane's query
    const int base_pos = L - Qn;
    const bool qvalid = computes && qr < Qn;
    const int pq = base_pos + qr;
    // the workgroup's keys, and this wave's own block's
    const KeyRange range = prefill_range(base_pos, qb * QB * 16, min(Qn, (qb + 1) * QB * 16) - 1, a.window, 1, 0, kPfKeys);
    const int kstart = range.kstart, kend = range.kend;
    const int wkend = base_pos + min(Qn, qrow0 + 16);
    const int wkstart = a.window > 0 ? max(0, base_pos + qrow0 - a.window + 1) : 0;
    const bool wlive = computes && qrow0 < Qn;

    // Q^T as the B operand: lane (col, grp) holds d = 32c + 8grp .. +7 of query qr
    uint4 qop[D / 32];
    {
        const uint16_t *qp = a.q + (((int64_t)item * hq + head) * Qn + (qvalid ? qr : 0)) * D + 8 * grp;
#pragma unroll
        for (int c = 0; c < D / 32; ++c)
            qop[c] = qvalid ? *reinterpret_cast<const uint4 *>(qp + 32 * c) : make_uint4(0, 0, 0, 0);
    }
    float m = kNegBig, l = 0.f;  // running max (uniform per query) and this lane's partial sum
    f32x4_t o[D / 16];
#pragma unroll
    for (int b = 0; b < D / 16; ++b) o[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    const int khi = qvalid ? min(kend - 1, pq) : -1;  // keys this lane's query sees: [klo, khi]
    const int klo = a.window > 0 ? pq - a.window + 1 : 0;
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): Q is there before the first DMA (its wait would drain them)

    // the work on the tile of keys t0 .. t0 + 31: kop(b, c) and vop(b) read its operands
    auto tile = [&](int t0, auto kop, auto vop) __attribute__((always_inline)) {
        // every query of the block sees the whole tile: no per-key mask
        const bool all_visible = qrow0 + 16 <= Qn && t0 + kPfKeys - 1 <= base_pos + qrow0 &&
                                 (a.window == 0 || t0 >= base_pos + qrow0 + 15 - a.window + 1) && t0 >= plen;
        f32x4_t s[2];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            s[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < D / 32; ++c) {
                s[b] = mfma16(kop(b, c), qop[c], s[b]);
            }
        }
        // scale and mask; this lane holds keys 8grp .. 8grp + 7
        float sc[8], tmax = -INFINITY;
        if (all_visible) {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sc[e] = (e < 4 ? s[0][e] : s[1][e - 4]) * a.scale_log2;
                tmax = fmaxf(tmax, sc[e]);
            }
        } else {
            const int k0 = t0 + 8 * grp;
            const uint32_t pvis = t0 < plen ? prefix_bits8(pw, k0, plen) : 0xffu;
            const int nhi = min(max(khi - k0 + 1, 0), 8), nlo = min(max(klo - k0, 0), 8);
            const uint32_t vis8 = ((1u << nhi) - 1u) & ~((1u << nlo) - 1u) & pvis;
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                sc[e] = (vis8 & (1u << e)) != 0 ? (e < 4 ? s[0][e] : s[1][e - 4]) * a.scale_log2 : -INFINITY;
                tmax = fmaxf(tmax, sc[e]);
            }
        }
        tmax = pair<OpMax, 32>(pair<OpMax, 16>(tmax));
        if (tmax > m + kRescaleSlack) {
            if (m != kNegBig) {  // otherwise nothing has been accumulated yet
                const float corr = __builtin_amdgcn_exp2f(m - tmax);
                l *= corr;
#pragma unroll
                for (int b = 0; b < D / 16; ++b) o[b] *= corr;
            }
            m = tmax;
        }
        // P = P_hi + P_lo, both bf16: P to ~2^-17 relative
        uint32_t ph[4], pl[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float p0 = __builtin_amdgcn_exp2f(sc[2 * e] - m);
            const float p1 = __builtin_amdgcn_exp2f(sc[2 * e + 1] - m);
            l += p0 + p1;
            ph[e] = pack_bf16x2(p0, p1);
            pl[e] = pack_bf16x2(p0 - bf16_lo(ph[e]), p1 - bf16_hi(ph[e]));
        }
        const uint4 hi = make_uint4(ph[0], ph[1], ph[2], ph[3]), lo = make_uint4(pl[0], pl[1], pl[2], pl[3]);
#pragma unroll
        for (int b = 0; b < D / 16; ++b) {
            const uint4 va = vop(b);
            o[b] = mfma16(va, lo, mfma16(va, hi, o[b]));
        }
    };
    // ---- staging: tile j (keys kstart + 32 j ..) in stage j % NS, 1 KiB
    // per DMA, a tile's DMAs spread over the waves. Keys past the range
    // read its first key.
    constexpr int RPI = 512 / D;  // rows per DMA of 1 KiB
    constexpr int IPT = kPfKeys / RPI, DPW = 2 * IPT / NW;  // DMAs per K (or V) tile, per wave and tile
    static_assert((2 * IPT) % NW == 0, "a tile's DMAs split evenly over the waves");
    const uint16_t *kg = static_cast<const uint16_t *>(a.kv.k), *vg = static_cast<const uint16_t *>(a.kv.v);
    const uint32_t sk_a = lds_addr(sk), sv_a = lds_addr(sv);
    const int ntiles = kend > kstart ? (kend - kstart + kPfKeys - 1) / kPfKeys : 0;
    const int ngroups = (ntiles + KS - 1) / KS;
    const int lrow = lane / (D / 8), pchunk = lane % (D / 8);
    auto issue_tile = [&](int j) __attribute__((always_inline)) {
        const int t0 = kstart + j * kPfKeys;
        const uint32_t stage = (uint32_t)((j % NS) * STAGE) * 2;
#pragma unroll
        for (int i = 0; i < DPW; ++i) {
            const int q = wave + i * NW;  // < IPT: K instruction q, else V instruction q - IPT
            const int ins = q % IPT;
            const int r = ins * RPI + lrow;  // key of this lane within the tile
            const int64_t off = ps_row_offset<D, LAYOUT>(a.kv, slot, kvh, t0, kstart, kend, r);
            const uint16_t *gp = (q < IPT ? kg : vg) + off + 8 * (pchunk ^ ps_swz<D>(r));
            const uint32_t dst = (q < IPT ? sk_a : sv_a) + stage + (uint32_t)ins * 1024u;
            dma_load16_cached(gp, __builtin_amdgcn_readfirstlane(dst));
        }
    };
    int issued = min((kPsGroups - 1) * KS, ntiles);
    for (int j = 0; j < issued; ++j) issue_tile(j);

    // this lane's rows and swizzles in a stage: the S^T A operand's key
    // ps_key(b, col) (logical chunk 4c + grp), and V^T row 8grp + col / 4 (+ 4)
    // with logical chunk 2b + (col & 3) / 2 and half col & 1, read transposed
    const int kr0 = ps_key(0, col), kr1 = ps_key(1, col);
    const int ksw0 = grp ^ ps_swz<D>(kr0), ksw1 = grp ^ ps_swz<D>(kr1);
    const int rv = 8 * grp + (col >> 2);
    const int vsw = ((col & 3) >> 1) ^ ps_swz<D>(rv), voff = rv * D + 4 * (col & 1);
    for (int it = 0; it < ngroups; ++it) {
        // DMAs of tiles past this group may stay in flight
        wait_vmem_steps<DPW, (kPsGroups - 1) * KS>(issued - min((it + 1) * KS, ntiles));
        __syncthreads();  // every wave's DMAs of group it have landed; group it - 1 is done
        const int next = min((it + kPsGroups) * KS, ntiles);
        for (int j = issued; j < next; ++j) issue_tile(j);  // into group it - 1's stages
        issued = next;
        const int j = it * KS + part;  // this wave's tile
        const int t0 = kstart + j * kPfKeys, sb = (j % NS) * STAGE;
        if (wlive && j < ntiles && (QB == 1 || (t0 < wkend && t0 + kPfKeys > wkstart))) {
            tile(
                t0,
                [&](int b, int c) __attribute__((always_inline)) {
                    const int kr = b ? kr1 : kr0, ksw = b ? ksw1 : ksw0;
                    return *reinterpret_cast<const uint4 *>(&sk[sb + kr * D + 8 * ((4 * c) ^ ksw)]);
                },
                [&](int b) __attribute__((always_inline)) {
                    const uint16_t *p = &sv[sb + voff + 8 * ((2 * b) ^ vsw)];
                    const uint2 x = lds_read_tr16(p), y = lds_read_tr16(p + 4 * D);
                    return make_uint4(x.x, x.y, y.x, y.y);
                });
        }
    }
    l = pair<OpSum, 32>(pair<OpSum, 16>(l));
    if constexpr (KS > 1) {
        // Parts 1 .. KS - 1 leave (m, l) and their accumulators, as each lane
        // holds them, in the drained stages; part 0 adds them in order.
        __syncthreads();
        float4 *xo = reinterpret_cast<float4 *>(sk);
        float2 *xml = reinterpret_cast<float2 *>(sv);
        const auto entry = [&](int p) { return ((p - 1) * hw + hidx) * QB + qsub; };
        if (computes && part > 0) {
            float4 *dst = xo + entry(part) * (D / 16) * 64 + lane;
#pragma unroll
            for (int b = 0; b < D / 16; ++b) dst[64 * b] = make_float4(o[b][0], o[b][1], o[b][2], o[b][3]);
            if (grp == 0) xml[entry(part) * 16 + col] = make_float2(m, l);
        }
        __syncthreads();
        if (part > 0) return;
        float M = m;
#pragma unroll
        for (int p = 1; p < KS; ++p) M = fmaxf(M, xml[entry(p) * 16 + col].x);
        const float w0 = __builtin_amdgcn_exp2f(m - M);
        l *= w0;
#pragma unroll
        for (int b = 0; b < D / 16; ++b) o[b] *= w0;
#pragma unroll
        for (int p = 1; p < KS; ++p) {
            const float2 ml = xml[entry(p) * 16 + col];
            const float w = __builtin_amdgcn_exp2f(ml.x - M);
            l = fmaf(ml.y, w, l);
            const float4 *src = xo + entry(p) * (D / 16) * 64 + lane;
#pragma unroll
            for (int b = 0; b < D / 16; ++b) {
                const float4 x = src[64 * b];
                o[b][0] = fmaf(x.x, w, o[b][0]);
                o[b][1] = fmaf(x.y, w, o[b][1]);
                o[b][2] = fmaf(x.z, w, o[b][2]);
                o[b][3] = fmaf(x.w, w, o[b][3]);
            }
        }
    }
    if (!qvalid) return;
    const float inv = l > 0.f ? 1.0f / l : 0.f;
    uint16_t *op = a.out + (((int64_t)item * hq + head) * Qn + qr) * D + 4 * grp;
#pragma unroll
    for (int b = 0; b < D / 16; ++b)
        *reinterpret_cast<uint2 *>(op + 16 * b) =
            make_uint2(pack_bf16x2(o[b][0] * inv, o[b][1] * inv), pack_bf16x2(o[b][2] * inv, o[b][3] * inv));
}

template <int D, int NW, int KS, int QB>
static hipError_t launch_short(const PrefillArgs &a, hipStream_t s) {
    const dim3 grid(a.kv.kv_heads * (a.group / a.short_heads), a.n_items, (a.qn + 16 * QB - 1) / (16 * QB));
    if (a.kv.layout == KVRT_LAYOUT_RING)
        hipLaunchKernelGGL((prefill_short_kernel<D, KVRT_LAYOUT_RING, NW, KS, QB>), grid, dim3(64 * NW), 0, s, a);
    else
        hipLaunchKernelGGL((prefill_short_kernel<D, KVRT_LAYOUT_CONTIG, NW, KS, QB>), grid, dim3(64 * NW), 0, s, a);
    return hipGetLastError();
}

template <int D>
static hipError_t launch_short_d(const PrefillArgs &a, hipStream_t s) {
    // short_heads * key_parts * row_waves waves compute; a workgroup has 2, 4 or 8
    const int ks = a.key_parts, qb = a.row_waves, waves = a.short_heads * ks * qb;
    const auto go = [&](auto nw_c) {
        constexpr int NW = decltype(nw_c)::value;
        if (ks == 2 && qb == 1) return launch_short<D, NW, 2, 1>(a, s);
        if constexpr (NW >= 4)
            if (ks == 2 && qb == 2) return launch_short<D, NW, 2, 2>(a, s);
        if constexpr (NW == 8)
            if (ks == 1 && qb == 2) return launch_short<D, NW, 1, 2>(a, s);
        return hipErrorInvalidValue;
    };
    if (waves <= 2) return go(std::integral_constant<int, 2>{});
    if (waves <= 4) return go(std::integral_constant<int, 4>{});
    return waves <= 8 ? go(std::integral_constant<int, 8>{}) : hipErrorInvalidValue;
}

hipError_t launch_prefill_short(const PrefillArgs &a, int head_dim, hipStream_t s) {
    if (a.kv.layout == KVRT_LAYOUT_PAGED || a.n_ksplit != 1 || a.group % a.short_heads != 0) return hipErrorInvalidValue;
    if (head_dim == 128) return launch_short_d<128>(a, s);
    return head_dim == 64 ? launch_short_d<64>(a, s) : hipErrorInvalidValue;
}

}  // namespace kvrt
