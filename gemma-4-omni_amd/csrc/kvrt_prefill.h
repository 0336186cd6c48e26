// kvrt_prefill.h — chunked-prefill attention on the matrix cores (gfx950).
//
// The rows of a (stream, KV head) are its q heads x queries, numbered query
// first (row r: query r / g, head r % g of the group), so any 32 consecutive
// rows span few queries, whatever the GQA group, and no row of a tile is
// padding except past the last query. A workgroup holds RW * 32 rows; its
// KS * RW waves are RW row blocks x KS key parts: part p takes the 32-key
// blocks p, p + KS, ... of the workgroup's keys, and the parts' accumulators
// are combined through LDS at the end. Per 32-key block and wave:
//   S^T (32 keys x 32 rows) = K Q^T    D/16     v_mfma_f32_32x32x16_bf16
//   online softmax per row (fp32, exp2 domain)
//   O^T (D x 32) += V^T P^T            4 * D/32 v_mfma_f32_32x32x16_bf16
// with P in two bf16 terms for the second product and everything accumulated
// in fp32. Lane layouts (32x32x16): A[row l%32][k 8(l/32)+j], B[k 8(l/32)+j]
// [col l%32], D[row 8(i/4) + 4(l/32) + i%4][col l%32].
//
// What bounds it: per block a wave issues 24 / 48 / 96 MFMAs of 32 cycles
// (D 128 / 256 / 512) beside ~140 VALU instructions, 4 of which fit beside an
// MFMA. 32 rows per wave halve the LDS reads per MFMA of a 16-row tile, whose
// LDS traffic outran the matrix cores (SQ_LDS_BANK_CONFLICT is 0 in this
// layout), and the softmax of a block runs beside the P V of the one before it,
// so one wave per SIMD keeps its matrix core busy: cycles per block 2700 at
// D 256 (MFMA alone 1536; 4870 with 16-row tiles) and 4960 at D 512 (3072;
// 7050). Long D 512 chunks then run against the power limit (1.8 GHz).
// 16-row tiles -> this kernel, us: D 512 Q 2048 over 2048 keys, 4 streams 566
// -> 498, Q 291 97.2 -> 84.3, Q 60 over 1440 48.1 -> 36.8; D 256 Q 2048 55.9 ->
// 47.0, window 512 Q 291 22.1 -> 21.1; D 128 Hq 16 Q 1400 over 600 109 -> 98,
// Q 512 15.9 -> 15.5, Hq 8 Q 34 over 2666 27.7 -> 16.3.
#pragma once

#include "kvrt_wave.h"

namespace kvrt {

typedef float f32x16_t __attribute__((ext_vector_type(16)));

__device__ __forceinline__ f32x16_t mfma32(uint4 a, uint4 b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                   c, 0, 0, 0);
}

// s (+)= four steps of K Q^T with s in VGPRs, for head_dim 512, whose output
// accumulators take every AGPR: the compiler puts all MFMA results of a kernel
// in one register file. The block stands for itself: it waits out a VALU
// write of an operand before it (2 states) and its last MFMA's result after
// it (12 states of an 8-pass MFMA); the MFMAs in between add to the same
// registers, which needs no wait.
template <bool FIRST>
__device__ __forceinline__ void mfma32_vgpr4(f32x16_t &s, const uint4 (&k)[4], const uint4 *q) {
    const auto v = [](const uint4 &x) { return __builtin_bit_cast(u32x4_t, x); };
#define KVRT_MFMA4(first)                                                \
    "s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %5, " first "\n\t"       \
    "v_mfma_f32_32x32x16_bf16 %0, %2, %6, %0\n\t"                        \
    "v_mfma_f32_32x32x16_bf16 %0, %3, %7, %0\n\t"                        \
    "v_mfma_f32_32x32x16_bf16 %0, %4, %8, %0\n\ts_nop 12"
#define KVRT_MFMA4_IN                                                                                       \
    "v"(v(k[0])), "v"(v(k[1])), "v"(v(k[2])), "v"(v(k[3])), "v"(v(q[0])), "v"(v(q[1])), "v"(v(q[2])), "v"(v(q[3]))
    if constexpr (FIRST) asm volatile(KVRT_MFMA4("0") : "=&v"(s) : KVRT_MFMA4_IN);
    else asm volatile(KVRT_MFMA4("%0") : "+v"(s) : KVRT_MFMA4_IN);
#undef KVRT_MFMA4
#undef KVRT_MFMA4_IN
}

// Keeps an output accumulator in AGPRs at this place (head_dim >= 256, whose
// accumulators and Q fill more than the 256 VGPRs): where their values join,
// the compiler otherwise picks VGPRs and copies them to AGPRs and back on
// every block.
template <int D>
__device__ __forceinline__ void keep_acc(f32x16_t &o) {
    if constexpr (D >= 256) asm volatile("" : "+a"(o));
}

// o *= c, for accumulators in AGPRs register by register (read, multiply, write
// back): as ordinary code the compiler brings many of them to VGPRs at once
// and, at head_dim 512, spills others over the whole loop. There they are all
// 256 AGPRs, in whatever order, and the block scales a0 .. a255. The wait is
// for the MFMAs before it (12 states after an 8-pass MFMA), which the compiler
// does not know these blocks read.
template <int D>
__device__ __forceinline__ void scale_accs(f32x16_t (&o)[D / 32], float c) {
    if constexpr (D < 256) {
#pragma unroll
        for (int b = 0; b < D / 32; ++b) o[b] *= c;
    } else if constexpr (D == 256) {
        asm volatile("s_nop 15" ::: "memory");
#pragma unroll
        for (int b = 0; b < D / 32; ++b)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                float x = o[b][i], t;
                asm volatile("v_accvgpr_read_b32 %1, %0\n\tv_mul_f32 %1, %1, %2\n\tv_accvgpr_write_b32 %0, %1"
                             : "+a"(x), "=&v"(t)
                             : "v"(c));
                o[b][i] = x;
            }
    } else {
        float t;
        asm volatile(
            "s_nop 15\n\t"
            ".set kvrt_i, 0\n\t"
            ".rept 256\n\t"
            "v_accvgpr_read_b32 %16, a[kvrt_i]\n\t"
            "v_mul_f32 %16, %16, %17\n\t"
            "v_accvgpr_write_b32 a[kvrt_i], %16\n\t"
            ".set kvrt_i, kvrt_i + 1\n\t"
            ".endr"
            : "+a"(o[0]), "+a"(o[1]), "+a"(o[2]), "+a"(o[3]), "+a"(o[4]), "+a"(o[5]), "+a"(o[6]), "+a"(o[7]),
              "+a"(o[8]), "+a"(o[9]), "+a"(o[10]), "+a"(o[11]), "+a"(o[12]), "+a"(o[13]), "+a"(o[14]), "+a"(o[15]),
              "=&v"(t)
            : "v"(c));
    }
}

// LDS DMA of 16 bytes per lane from base + off (bytes): the tile's address is
// uniform and a lane's offset fixed, so a DMA costs no 64-bit lane arithmetic.
__device__ __forceinline__ void dma_load16_at(const void *base, uint32_t off, uint32_t lds) {
    asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(lds) : "memory");
}

// A staged 32-key block of K or V: each DMA instruction leaves 1 KiB, rows ins,
// ins + IPB, ins + 2 IPB, ... of the block one after another (IPB = D/16
// instructions per block), and the instructions lie 1 KiB plus a padding
// apart. On 64 banks of 4 B (16 places of 16 B) one S^T operand read (one chunk
// of 16 consecutive rows per 16 lanes) and one transposed V read (4 chunks of
// 4 consecutive rows per 32 lanes) then hit every place once with K padded by
// 16 and V by 64 bytes, and every operand's address is one register plus a
// constant. At D 128 and 64 two or four of K's 16 rows share an instruction:
// there a row's chunks are moved by pf_kx<D>(row within the instruction).
constexpr int kPfKPitch = 1024 + 16, kPfVPitch = 1024 + 64;  // bytes between instructions
template <int D>
__device__ __forceinline__ int pf_kx(int k) {
    return D == 128 ? (k & 1) << 3 : D == 64 ? ((k >> 1) & 1) << 2 : 0;
}

// Calls f(integral_constant<int, u>) for u = U .. N-1: every index below is a
// constant, whatever the unroller makes of a loop of its size.
template <int U, int N>
struct StaticFor {
    template <class F>
    __device__ __forceinline__ static void run(F &&f) {
        if constexpr (U < N) {
            f(std::integral_constant<int, U>{});
            StaticFor<U + 1, N>::run(f);
        }
    }
};

template <int D, int RW, int KS, int NS>
struct PrefillShape {
    static constexpr int NW = RW * KS;         // waves
    static constexpr int IPB = D / 16;         // DMA instructions per K (or V) block
    static constexpr int IPW = IPB / RW;       // ... per wave (part p's waves fetch block p)
    static constexpr int KBLK = IPB * kPfKPitch, VBLK = IPB * kPfVPitch;  // bytes of a staged block
    static_assert(IPB % RW == 0, "a block's DMAs split evenly over its row waves");
};

template <int D, int LAYOUT, int RW, int KS, int NS>
__global__ __launch_bounds__(64 * RW * KS) void prefill_kernel(PrefillArgs a) {
    using P = PrefillShape<D, RW, KS, NS>;
    constexpr int KBLK = P::KBLK, VBLK = P::VBLK, IPB = P::IPB, IPW = P::IPW;
    constexpr int NB = D / 32;  // 32-dim blocks of the output
    __shared__ __align__(16) uint8_t sk[NS * KS * KBLK];
    __shared__ __align__(16) uint8_t sv[NS * KS * VBLK];
    __shared__ float2 sml[KS > 1 ? KS * RW * 32 : 1];  // (m, l) of the parts' rows
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = lane & 31, half = lane >> 5;
    const int part = wave / RW, rw = wave % RW;
    // Grid (KV head x key range, item, row blocks): workgroups start in
    // linear id order, so the row blocks are the most significant and run last
    // blocks first. Without a window the last blocks see the most keys: the
    // longest workgroups start first and the grid's tail is short ones.
    const int nks = a.n_ksplit;
    int kvh, ks;
    udivmod_uniform(blockIdx.x, nks, kvh, ks);
    const int item = blockIdx.y;
    const int qb = gridDim.z - 1 - blockIdx.z;
    const int g = a.group, hq = a.kv.kv_heads * g;
    const int slot = a.slots[item];
    const int L = __builtin_amdgcn_readfirstlane(a.len.lens[(int64_t)slot * a.len.stride + a.len.offset]);
    int plen;  // prefix-attention mask of the slot
    uint32_t pw;
    load_prefix(a.pmask, slot, lane, plen, pw);
    const int Qn = a.qn, R = g * Qn;
    const int wg0 = qb * RW * 32, row0 = wg0 + rw * 32;
    const bool wlive = row0 < R;
    // this lane's row (S^T / O^T column): query qr, head hr of the group; and
    // the queries of the workgroup's and of this wave's first and last rows
    const bool qvalid = row0 + col < R;
    const int lrow0 = qvalid ? row0 + col : 0, wg1 = min(R, wg0 + RW * 32) - 1, row1 = min(R, row0 + 32) - 1;
    int qr, qf, ql, wqf, wql;
    if ((g & (g - 1)) == 0) {
        const int sh = __builtin_ctz((unsigned)g);
        qr = lrow0 >> sh, qf = wg0 >> sh, ql = wg1 >> sh, wqf = row0 >> sh, wql = row1 >> sh;
    } else {
        qr = lrow0 / g, qf = wg0 / g, ql = wg1 / g, wqf = row0 / g, wql = row1 / g;
    }
    const int hr = lrow0 - qr * g;
    // Q^T as the B operand: lane (col, half) holds d = 16c + 8half .. +7 of its
    // row. In flight beside the length.
    uint4 qop[D / 16];
    {
        const uint16_t *qp = a.q + (((int64_t)item * hq + kvh * g + hr) * Qn + qr) * D + 8 * half;
#pragma unroll
        for (int c = 0; c < D / 16; ++c) qop[c] = *reinterpret_cast<const uint4 *>(qp + 16 * c);
    }
    const int base_pos = L - Qn;  // position of query 0
    const int pq = base_pos + qr;
    // the workgroup's keys: from its first query's window to its last query;
    // with a key split, range ks of them in whole blocks
    const KeyRange range = prefill_range(base_pos, qf, ql, a.window, nks, ks, kPfKeys);
    const int kstart = range.kstart, kend = range.kend;
    const int wkend = base_pos + wql + 1;  // the same for this wave's rows
    const int wkstart = a.window > 0 ? max(0, base_pos + wqf - a.window + 1) : 0;
    const int ngroups = (kend - kstart + kPfKeys * KS - 1) / (kPfKeys * KS);  // <= 0: no keys, nothing is fetched
    // keys this lane's row sees: [klo, khi] (none if the lane has no row)
    const int khi = qvalid ? min(kend - 1, pq) : -1;
    const int klo = a.window > 0 ? pq - a.window + 1 : 0;

    float m = kNegBig, l = 0.f;  // running max (both halves alike) and this lane's partial sum
    f32x16_t o[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int i = 0; i < 16; ++i) o[b][i] = 0.f;
        keep_acc<D>(o[b]);
    }
    bool bad = false;

    // ---- staging: wave (part, rw) fetches instructions rw, rw + RW, ... of
    // the K and V rows of block part of every group of KS blocks
    const uint16_t *kg = static_cast<const uint16_t *>(a.kv.k);
    const uint16_t *vg = static_cast<const uint16_t *>(a.kv.v);
    const int64_t head_base = LAYOUT == KVRT_LAYOUT_PAGED
                                  ? 0
                                  : (int64_t)slot * a.kv.slot_stride + (int64_t)kvh * a.kv.head_stride;
    const uint32_t sk_a = lds_addr(sk), sv_a = lds_addr(sv);
    const int lrow = IPB * (lane / (D / 8)) + rw;  // this lane's row of its wave's first instruction
    const uint32_t vchunk = lane % (D / 8) * 16, kchunk = vchunk ^ (uint32_t)(16 * pf_kx<D>(lane / (D / 8)));
    // The block of keys a wave's DMAs of a group fetch, first its K and one
    // group later its V rows. Rows past the range read the range's last key (a
    // block wholly past it likewise, and is never computed).
    struct Fetch {
        int64_t off;   // elements: CONTIG the block's first row, RING the head's, PAGED 0
        int r0, last;  // first row (RING) or key (PAGED); last row of the block inside the range
        int pages;     // PAGED: entry of the block's page `lane` (a block spans at most 32)
    };
    int kt = kstart + part * kPfKeys, krow = 0;  // first key of the block, its row in the ring
    int rlast = 0;                               // ... of the range's last key
    if constexpr (LAYOUT == KVRT_LAYOUT_RING) krow = kt % a.kv.rows, rlast = (kend - 1) % a.kv.rows;
    // PAGED: the entries of the pages from the block at key t on; loaded a group
    // ahead, so that no DMA waits for them
    auto load_pages = [&](int t) __attribute__((always_inline)) {
        return load_page_window(a.kv, slot, min(t, kend - 1) >> a.kv.block_shift, lane);
    };
    int pages = 0;  // of the block at kt
    if constexpr (LAYOUT == KVRT_LAYOUT_PAGED)
        if (ngroups > 0) pages = load_pages(kt);  // kend > kstart >= 0
    auto next_fetch = [&]() __attribute__((always_inline)) {
        const int t0 = min(kt, kend - 1);
        Fetch f;
        f.off = head_base;
        f.r0 = t0;
        f.last = kend - 1 - t0;
        f.pages = pages;
        if constexpr (LAYOUT == KVRT_LAYOUT_CONTIG) f.off += (int64_t)t0 * D;
        if constexpr (LAYOUT == KVRT_LAYOUT_RING) f.r0 = kt < kend ? krow : rlast;
        kt += kPfKeys * KS;
        if constexpr (LAYOUT == KVRT_LAYOUT_RING)
            for (krow += kPfKeys * KS; krow >= a.kv.rows;) krow -= a.kv.rows;
        if constexpr (LAYOUT == KVRT_LAYOUT_PAGED) pages = load_pages(kt);
        return f;
    };
    // instruction i of this wave (0 .. IPW - 1), into the buffers of group it
    auto fetch = [&](auto v_c, const Fetch &f, int it, int i) __attribute__((always_inline)) {
        constexpr bool V = decltype(v_c)::value;
        constexpr int PITCH = V ? kPfVPitch : kPfKPitch, BLK = V ? VBLK : KBLK;
        const uint16_t *base = (V ? vg : kg) + f.off;
        const int r = min(lrow + i * RW, f.last);
        const uint32_t dst = (V ? sv_a : sk_a) + (uint32_t)(((it % NS) * KS + part) * BLK + (i * RW + rw) * PITCH);
        const uint32_t chunk = V ? vchunk : kchunk;
        if constexpr (LAYOUT == KVRT_LAYOUT_CONTIG) {
            dma_load16_at(base, (uint32_t)r * (2 * D) + chunk, dst);
        } else if constexpr (LAYOUT == KVRT_LAYOUT_RING) {
            int rr = f.r0 + r;  // rows of a block wrap at most once
            rr = rr >= a.kv.rows ? rr - a.kv.rows : rr;
            dma_load16_cached(base + (int64_t)rr * D + chunk / 2, dst);
        } else {
            const int key = f.r0 + r;
            const int page = __shfl(f.pages, (key >> a.kv.block_shift) - (f.r0 >> a.kv.block_shift));
            int64_t off = page_row_offset(a.kv, page, kvh, key, D);
            bad |= off < 0;
            off = off < 0 ? 0 : off;
            dma_load16_cached(base + off + chunk / 2, dst);
        }
    };

    Fetch kf{}, vf{};
    // parts with a block in the range; the others fetch no first K block and
    // add nothing at the end
    const int nparts = KS == 1 ? 1 : max(1, min(KS, (kend - kstart + kPfKeys - 1) / kPfKeys));
    if (ngroups > 0) {  // the first K blocks
        kf = next_fetch();
        if (part < nparts)
#pragma unroll
            for (int i = 0; i < IPW; ++i) fetch(std::false_type{}, kf, 0, i);
    }

    // A negative scale is moved into q's sign bits (exact, below), so that the
    // largest score always has the largest product; a zero scale stays above 0,
    // so that a masked score (-INFINITY) keeps its weight of 0.
    const float scale = fmaxf(fabsf(a.scale_log2), 1e-37f);
    const uint32_t flip = a.scale_log2 < 0.f ? 0x80008000u : 0u;

    // ---- operands: A of S^T is key row col, chunk 2c + half; A of V^T is dims
    // 32b + (0 .. 31) of the keys 16s + 8e + 4half + (0 .. 3), e = 0, 1, the
    // keys whose P this lane half holds (D layout above), read transposed: in
    // each group of 16 lanes, lane s16 points at key row s16 / 4, dims
    // 4 (s16 % 4) .. +3, and receives dim s16 of the four rows.
    const int kadr = (col % IPB) * kPfKPitch + (col / IPB) * 2 * D + 16 * half;
    const int kx = 16 * pf_kx<D>(col / IPB);
    const int s16 = lane & 15, r4 = 4 * half + (s16 >> 2);  // key row 16s + 8e + r4
    const int vadr = 32 * ((lane >> 4) & 1) + 8 * (s16 & 3) +
                     (IPB >= 8 ? r4 * kPfVPitch : (r4 % IPB) * kPfVPitch + (r4 / IPB) * 2 * D);
    auto kop = [&](int blk, int c) __attribute__((always_inline)) {
        return *reinterpret_cast<const uint4 *>(&sk[blk * KBLK + kadr + ((32 * c) ^ kx)]);
    };
    auto vop = [&](int blk, int b, int s) __attribute__((always_inline)) {
        uint2 x[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
            const int r = 16 * s + 8 * e;  // r4 < 8 adds no carry into the instruction number
            x[e] = lds_read_tr16(reinterpret_cast<const uint16_t *>(
                &sv[blk * VBLK + vadr + (r % IPB) * kPfVPitch + (r / IPB) * 2 * D + 64 * b]));
        }
        return make_uint4(x[0].x, x[0].y, x[1].x, x[1].y);
    };
    // ---- the work on one 32-key block, in steps of one MFMA each. Operands
    // are read PK (PV) steps ahead of their MFMAs, the next groups' DMAs are
    // spread over the steps, and the next block's softmax runs beside this
    // block's P V; sched_barrier holds that order (left to itself the
    // scheduler reads each operand right before its MFMA, one LDS round trip
    // per step, and keeps the softmax apart from the MFMAs).
    constexpr int PK = D / 16 < 4 ? D / 16 : 4, PV = 2 * NB < 4 ? 2 * NB : 4;
    constexpr int NK = D / 16, NP = 4 * NB;  // MFMAs of K Q^T and of P V per block
    uint4 vx[PV];       // V^T operands u = 0 .. 2 NB - 1 (keys 16 (u / NB), dims 32 (u % NB)) of the ring
    uint4 ph[2], pl[2];  // P of the block whose P V is next, by 16 keys: high and low terms
    f32x16_t s;         // scores of the block after it
    int cur = 0;  // the iteration
    // The iteration's DMAs (the K blocks of group it + 2, then the V blocks of
    // it + 1), spread over SPAN steps: up to head_dim 128 those of K Q^T, at 256
    // the first half of all (59 against 61 us over 2339 cold keys), at 512 of the
    // P V ones, whose MFMAs leave the most issue slots free. Past the last group
    // they read its last key (a branch around each costs more than the DMAs it
    // would save), but the last iteration skips those of K Q^T, and up to
    // head_dim 128 the kernel's end waits for none.
    constexpr int DMA0 = D == 512 ? NK : 0, SPAN = D == 512 ? NP / 2 : D == 256 ? (NK + NP) / 2 : NK;
    auto dma_at = [&](auto c_c) __attribute__((always_inline)) {
        constexpr int c = decltype(c_c)::value - DMA0;
        if constexpr (c >= 0 && c < SPAN)
            StaticFor<(2 * IPW * c + SPAN - 1) / SPAN, (2 * IPW * (c + 1) + SPAN - 1) / SPAN>::run([&](auto n_c) {
                constexpr int n = decltype(n_c)::value;
                if constexpr (n < IPW) fetch(std::false_type{}, kf, cur + 2, n);
                else fetch(std::true_type{}, vf, cur + 1, n - IPW);
            });
    };
    auto score_steps = [&](int blk, int vblk, auto first_c) __attribute__((always_inline)) {
        constexpr bool FIRST = decltype(first_c)::value;  // no V to read and no DMAs beside the first block
        if constexpr (D == 512) {
            uint4 x[2][4];
#pragma unroll
            for (int c = 0; c < 4; ++c) x[0][c] = kop(blk, c);
            __builtin_amdgcn_sched_barrier(0);
            StaticFor<0, NK / 4>::run([&](auto c_c) {
                constexpr int c = decltype(c_c)::value;
                if constexpr (c + 1 < NK / 4) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) x[(c + 1) % 2][e] = kop(blk, 4 * c + 4 + e);
                } else {
#pragma unroll
                    for (int e = 0; e < PV; ++e) vx[e] = vop(vblk, e % NB, e / NB);
                }
                mfma32_vgpr4<c == 0>(s, x[c % 2], qop + 4 * c);
                if constexpr (!FIRST) StaticFor<4 * c, 4 * c + 4>::run(dma_at);
                __builtin_amdgcn_sched_barrier(0);
            });
        } else {
            uint4 x[PK];
#pragma unroll
            for (int c = 0; c < PK; ++c) x[c] = kop(blk, c);
#pragma unroll
            for (int i = 0; i < 16; ++i) s[i] = 0.f;
            __builtin_amdgcn_sched_barrier(0);
            StaticFor<0, NK>::run([&](auto c_c) {
                constexpr int c = decltype(c_c)::value, e = c + PK - NK;
                s = mfma32(x[c % PK], qop[c], s);
                if constexpr (e < 0) x[c % PK] = kop(blk, c + PK);
                else if constexpr (e < PV && !FIRST) vx[e] = vop(vblk, e % NB, e / NB);
                if constexpr (!FIRST) dma_at(c_c);
                __builtin_amdgcn_sched_barrier(0);
            });
        }
    };
    // keys every row of the wave sees: blocks inside take no per-key test
    const int vis_hi = min(kend, base_pos + wqf + 1);
    const int vis_lo = max(plen, a.window > 0 ? base_pos + wql - a.window + 1 : 0);
    // Masks the scores of keys t0 .. t0 + 31 (-INFINITY).
    auto mask = [&](int t0) __attribute__((always_inline)) {
        if (t0 >= vis_lo && t0 + kPfKeys <= vis_hi) return;
        // bit k: key t0 + k is visible to this lane's row
        const int nhi = min(max(khi - t0 + 1, 0), 32), nlo = min(max(klo - t0, 0), 32);
        uint32_t vis = (nhi >= 32 ? 0xffffffffu : (1u << nhi) - 1u) & (nlo >= 32 ? 0u : 0xffffffffu << nlo);
        if (t0 < plen) {
            const int w = t0 >> 5, sh = t0 & 31, past = plen - t0;
            const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)pw, w & (kPrefixWords - 1));
            const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)pw, (w + 1) & (kPrefixWords - 1));
            const uint32_t bits = (uint32_t)((((uint64_t)hi << 32) | lo) >> sh);
            vis &= bits | (past >= 32 ? 0u : 0xffffffffu << past);
        }
        vis >>= 4 * half;  // this half's keys: bit 8 (i / 4) + i % 4
#pragma unroll
        for (int i = 0; i < 16; ++i) s[i] = (vis >> (8 * (i >> 2) + (i & 3))) & 1u ? s[i] : -INFINITY;
    };
    // The softmax of s in NSOFT steps. The running max moves only where a
    // block's max exceeds it by kRescaleSlack; corr rescales what has been
    // accumulated so far (1 where it did not move). P leaves as two bf16 terms
    // (P = hi + lo, lo the rounding error of hi: P to ~2^-17 relative, where
    // one bf16 term (2^-9) would show in the bf16 outputs of few-key rows).
    constexpr int NSOFT = 4 + 4 * 8;
    float tmax, corr, e0, e1;
    uint32_t nh[8], nl[8];
    auto soft_step = [&](auto n_c) __attribute__((always_inline)) {
        constexpr int n = decltype(n_c)::value;
        if constexpr (n == 0) {
            tmax = s[0];
#pragma unroll
            for (int i = 1; i < 7; ++i) tmax = fmaxf(tmax, s[i]);
        } else if constexpr (n == 1) {
#pragma unroll
            for (int i = 7; i < 15; ++i) tmax = fmaxf(tmax, s[i]);
        } else if constexpr (n == 2) {
            tmax = pair<OpMax, 32>(fmaxf(tmax, s[15])) * scale;
        } else if constexpr (n == 3) {
            const float mn = tmax > m + kRescaleSlack ? tmax : m;
            corr = __builtin_amdgcn_exp2f(m - mn);
            l *= corr;
            m = mn;
        } else if constexpr (n < NSOFT) {
            constexpr int j = (n - 4) / 4;
            if constexpr (n % 4 == 0) {
                e0 = __builtin_amdgcn_exp2f(fmaf(s[2 * j], scale, -m));
            } else if constexpr (n % 4 == 1) {
                e1 = __builtin_amdgcn_exp2f(fmaf(s[2 * j + 1], scale, -m));
            } else if constexpr (n % 4 == 2) {
                l += e0 + e1;
                nh[j] = pack_bf16x2(e0, e1);
            } else {
                nl[j] = pack_bf16x2(e0 - bf16_lo(nh[j]), e1 - bf16_hi(nh[j]));
                asm volatile("" : "+v"(nh[j]), "+v"(nl[j]));  // computed here, not where P is used
            }
        }
    };
    auto take_p = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            ph[h] = make_uint4(nh[4 * h], nh[4 * h + 1], nh[4 * h + 2], nh[4 * h + 3]);
            pl[h] = make_uint4(nl[4 * h], nl[4 * h + 1], nl[4 * h + 2], nl[4 * h + 3]);
        }
    };
    // P V of the block in V buffer vblk with the softmax of s beside it and the
    // DMA steps from dma0 on.
    auto value_steps = [&](int vblk) __attribute__((always_inline)) {
        StaticFor<0, NP>::run([&](auto c_c) {
            // pairs of dims blocks, high terms before low ones: no MFMA adds to the one before it
            constexpr int c = decltype(c_c)::value, h = c / (2 * NB), r = c % (2 * NB), b = r / 4 * 2 + (r & 1),
                          u = h * NB + b;
            o[b] = mfma32(vx[u % PV], (r & 2) ? pl[h] : ph[h], o[b]);
            if constexpr ((r & 2) && u + PV < 2 * NB) vx[u % PV] = vop(vblk, (u + PV) % NB, (u + PV) / NB);
            dma_at(std::integral_constant<int, NK + c>{});
            // softmax steps [NSOFT c / NP, NSOFT (c + 1) / NP)
            StaticFor<(NSOFT * c + NP - 1) / NP, (NSOFT * (c + 1) + NP - 1) / NP>::run(soft_step);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto rescale = [&]() __attribute__((always_inline)) {
        if (__builtin_expect_with_probability(__any(corr != 1.f), 0, 0.9999)) {
            scale_accs<D>(o, corr);
        }
    };

    // this wave's blocks: those of groups [jlo, jhi) that overlap its rows' keys
    int jlo = 0, jhi = 0;
    if (wlive) {
        const int hi_key = min(kend, wkend) - kstart - part * kPfKeys;  // > 32 KS j: block j starts below it
        jhi = hi_key > 0 ? (hi_key + kPfKeys * KS - 1) / (kPfKeys * KS) : 0;
        const int lo_key = wkstart - kstart - (part + 1) * kPfKeys;  // >= 32 KS j: block j ends at or below it
        jlo = lo_key >= 0 ? lo_key / (kPfKeys * KS) + 1 : 0;
        jhi = max(jhi, jlo);
    }
    auto key0 = [&](int j) { return kstart + (j * KS + part) * kPfKeys; };
    if (ngroups > 0) {
        wait_vmem<0>();
#pragma unroll
        for (int c = 0; c < D / 16; ++c) {
            uint4 &x = qop[c];
            x = make_uint4(x.x ^ flip, x.y ^ flip, x.z ^ flip, x.w ^ flip);
            asm volatile("" : "+v"(x.x), "+v"(x.y), "+v"(x.z), "+v"(x.w));
        }
        // the first V blocks and the second K blocks, in flight beside the first K Q^T
        vf = kf;
#pragma unroll
        for (int i = 0; i < IPW; ++i) fetch(std::true_type{}, vf, 0, i);
        if (D >= 256 || ngroups > 1) {  // (D 512, Q 24 over 49: 14.5 us with the test, 14.2 without)
            kf = next_fetch();
#pragma unroll
            for (int i = 0; i < IPW; ++i) fetch(std::false_type{}, kf, 1, i);
        }
        __syncthreads();
        if (jlo == 0 && jhi > 0) {
            score_steps(part, 0, std::true_type{});
            mask(key0(0));
            StaticFor<0, NSOFT>::run(soft_step);
            take_p();
        }
        // iteration it: K Q^T of group it + 1, P V of group it
        for (int it = 0; it < ngroups; ++it) {
#pragma unroll
            for (int b = 0; b < NB; ++b) keep_acc<D>(o[b]);
            wait_vmem<0>();   // this wave's DMAs of K group it + 1 and V group it have landed
            __syncthreads();  // every wave's have; K group it and V group it - 1 are read
            vf = kf;
            kf = next_fetch();
            cur = it;
            const bool do_s = it + 1 >= jlo && it + 1 < jhi, do_v = it >= jlo && it < jhi;
            const int kblk = ((it + 1) % NS) * KS + part, vblk = (it % NS) * KS + part;
            if (do_s) {
                score_steps(kblk, vblk, std::false_type{});
                mask(key0(it + 1));
            } else {
                if (it + 1 < ngroups) StaticFor<0, NK>::run(dma_at);
#pragma unroll
                for (int u = 0; u < PV; ++u) vx[u] = vop(vblk, u % NB, u / NB);
            }
            if (do_v) {
                // without a next block the softmax runs on the last one's scores
                // again: its max moves nothing, P is not used and l is put back
                const float lprev = l;
                value_steps(vblk);
                l = do_s ? l : lprev;
                rescale();
            } else {
                StaticFor<NK, NK + NP>::run(dma_at);
                if (do_s) StaticFor<0, NSOFT>::run(soft_step);
            }
            take_p();
        }
        wait_vmem<0>();  // the DMAs past the last group
    }
#pragma unroll
    for (int b = 0; b < NB; ++b) keep_acc<D>(o[b]);
    if (bad) a.err[0] = 1;
    l = pair<OpSum, 32>(l);

    // this lane's row again (from here on: keeping it over the loop would cost
    // registers that the loop needs)
    int ln = lane;
    asm volatile("" : "+v"(ln));
    const int ehalf = ln >> 5, erow = row0 + (ln & 31);
    const bool evalid = erow < R;
    int eq, eh;
    udivmod_uniform(evalid ? erow : 0, g, eq, eh);
    const int64_t orow = ((int64_t)item * hq + kvh * g + eh) * Qn + eq;  // of out
    const int64_t pi = orow * nks + ks;  // this row's partial of a key split
    // 32-dim block b, register group i of the row's dims 32b + 8i + 4half .. +3
    auto store_f32 = [&](int b, int i, float4 x) __attribute__((always_inline)) {
        *reinterpret_cast<float4 *>(a.part_o + pi * D + 32 * b + 8 * i + 4 * ehalf) = x;
    };
    // groups i and i + 1 (i even) as 16 B per lane: the halves exchange theirs,
    // lane half h then holds dims 32b + 8i + 8h .. +7
    auto store_bf16 = [&](int b, int i, float4 x, float4 y) __attribute__((always_inline)) {
        const auto lo = __builtin_amdgcn_permlane32_swap(pack_bf16x2(x.x, x.y), pack_bf16x2(y.x, y.y), false, false);
        const auto hi = __builtin_amdgcn_permlane32_swap(pack_bf16x2(x.z, x.w), pack_bf16x2(y.z, y.w), false, false);
        if (evalid)
            *reinterpret_cast<uint4 *>(a.out + orow * D + 32 * b + 8 * i + 8 * ehalf) =
                make_uint4(lo[0], hi[0], lo[1], hi[1]);
    };
    if constexpr (KS == 1) {
        if (!wlive) return;
        if (nks > 1) {
            if (!evalid) return;
            // (the same accumulators are read below: read in one place for both,
            // they would not fit)
            StaticFor<0, NB>::run([&](auto b_c) {
                constexpr int b = decltype(b_c)::value;
                keep_acc<D>(o[b]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    store_f32(b, i, make_float4(o[b][4 * i], o[b][4 * i + 1], o[b][4 * i + 2], o[b][4 * i + 3]));
                    if (D == 512) __builtin_amdgcn_sched_barrier(0);
                }
            });
            if (ehalf == 0) a.part_ml[pi] = make_float2(m, l);
            return;
        }
        const float inv = l > 0.f ? 1.0f / l : 0.f;
        StaticFor<0, NB>::run([&](auto b_c) {
            constexpr int b = decltype(b_c)::value;
            keep_acc<D>(o[b]);
#pragma unroll
            for (int i = 0; i < 4; i += 2) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = o[b][4 * i + e] * inv;
                store_bf16(b, i, make_float4(x[0], x[1], x[2], x[3]), make_float4(x[4], x[5], x[6], x[7]));
                if (D == 512) __builtin_amdgcn_sched_barrier(0);
            }
        });
    } else {
        // Combine the key parts: every part scales its accumulators to the
        // rows' common max (and sum) and leaves them in the drained buffers as
        // each lane holds them; the parts of a row block then each sum and
        // store a share of the dims, in part order. The buffers take BS
        // 32-dim blocks of all waves at a time.
        constexpr int BS = NS * D / (32 * RW) < NB ? NS * D / (32 * RW) : NB;
        static_assert(BS >= 1 && NB % BS == 0 && BS * P::NW * 2048 <= NS * KS * KBLK, "blocks fit the buffers");
        if (ehalf == 0) sml[wave * 32 + col] = make_float2(m, l);
        __syncthreads();  // also: every wave is done with the buffers
        float M = kNegBig, Lsum = 0.f;
#pragma unroll
        for (int p = 0; p < KS; ++p) M = fmaxf(M, sml[(p * RW + rw) * 32 + col].x);
#pragma unroll
        for (int p = 0; p < KS; ++p) {
            const float2 ml = sml[(p * RW + rw) * 32 + col];
            Lsum = fmaf(ml.y, __builtin_amdgcn_exp2f(ml.x - M), Lsum);
        }
        float w = __builtin_amdgcn_exp2f(m - M);
        if (nks == 1) w *= Lsum > 0.f ? 1.0f / Lsum : 0.f;
        // [wave][block][group i][lane], the waves' first halves in sk, the second in sv
        constexpr int WHALF = P::NW / 2;
        auto xo = [&](int wv) __attribute__((always_inline)) {
            return reinterpret_cast<float4 *>(wv < WHALF ? sk : sv) + (wv % WHALF) * BS * 256 + lane;
        };
        float4 *mine = xo(wave);
#pragma unroll
        for (int b0 = 0; b0 < NB; b0 += BS) {
            if (b0 > 0) __syncthreads();
            if (part < nparts)
#pragma unroll
                for (int b = 0; b < BS; ++b)
#pragma unroll
                    for (int i = 0; i < 4; ++i)
                        mine[(b * 4 + i) * 64] = make_float4(o[b0 + b][4 * i] * w, o[b0 + b][4 * i + 1] * w,
                                                         o[b0 + b][4 * i + 2] * w, o[b0 + b][4 * i + 3] * w);
            __syncthreads();
            if (wlive) {
                for (int u = part; u < 2 * BS; u += KS) {  // pairs of groups
                    const int b = u >> 1, i = 2 * (u & 1);
                    float4 x[2];
#pragma unroll
                    for (int e = 0; e < 2; ++e) x[e] = xo(rw)[(b * 4 + i + e) * 64];
#pragma unroll
                    for (int p = 1; p < KS; ++p) {
                        if (p >= nparts) break;
#pragma unroll
                        for (int e = 0; e < 2; ++e) {
                            const float4 y = xo(p * RW + rw)[(b * 4 + i + e) * 64];
                            x[e] = make_float4(x[e].x + y.x, x[e].y + y.y, x[e].z + y.z, x[e].w + y.w);
                        }
                    }
                    if (nks == 1) {
                        store_bf16(b0 + b, i, x[0], x[1]);
                    } else if (evalid) {
                        store_f32(b0 + b, i, x[0]);
                        store_f32(b0 + b, i + 1, x[1]);
                    }
                }
            }
        }
        if (nks > 1 && part == 0 && ehalf == 0 && evalid) a.part_ml[pi] = make_float2(M, Lsum);
    }
}

template <int D, int RW, int KS, int NS, int LAYOUT>
static hipError_t launch_prefill_layout(const PrefillArgs &a, hipStream_t s) {
    const int64_t rows = (int64_t)a.group * a.qn;
    const dim3 grid(a.n_ksplit * a.kv.kv_heads, a.n_items, (unsigned)((rows + 32 * RW - 1) / (32 * RW)));
    hipLaunchKernelGGL((prefill_kernel<D, LAYOUT, RW, KS, NS>), grid, dim3(64 * RW * KS), 0, s, a);
    return hipGetLastError();
}

template <int D, int RW, int KS, int NS>
static hipError_t launch_prefill_shape(const PrefillArgs &a, hipStream_t s) {
    switch (a.kv.layout) {
        case KVRT_LAYOUT_CONTIG: return launch_prefill_layout<D, RW, KS, NS, KVRT_LAYOUT_CONTIG>(a, s);
        case KVRT_LAYOUT_RING: return launch_prefill_layout<D, RW, KS, NS, KVRT_LAYOUT_RING>(a, s);
        case KVRT_LAYOUT_PAGED: return launch_prefill_layout<D, RW, KS, NS, KVRT_LAYOUT_PAGED>(a, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace kvrt
