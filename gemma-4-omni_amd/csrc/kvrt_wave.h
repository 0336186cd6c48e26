// kvrt_wave.h — wave-level helpers of the attention kernels (gfx950): row
// addressing, prefix-mask bits, LDS DMA and its waits, MFMA operand types.
#pragma once

#include <type_traits>

#include "kvrt_device.h"
#include "kvrt_internal.h"
#include "kvrt_range.h"

namespace kvrt {

constexpr float kNegBig = -1.0e30f;  // running-max start; exp2(kNegBig - m) == 0
// Lazy online softmax: a running max m (log2 units) moves only when a block's
// max exceeds it by more than kRescaleSlack, so p = 2^(s - m) stays <= 2^8
// and the accumulator rescale runs a few times per wave instead of on most
// blocks. Exact: l and the accumulator always refer to the same m, and every
// merge weights a partial by its own m.
constexpr float kRescaleSlack = 8.0f;

// Row number of position pos of a head on a PAGED page, in pool order
// ((page, head, pos % rows)); -1 if the page is unmapped or out of the pool.
// 32-bit arithmetic: the host keeps pool_pages below 2^24 and the pool's rows
// below 2^31, so page * (kv_heads * rows) is a 24-bit product.
__device__ __forceinline__ int page_row(const KVView &v, int page, int head, int pos) {
    if (page < 0 || page >= v.pool_pages) return -1;
    return (int)__umul24((unsigned)page, (unsigned)(v.kv_heads * v.rows)) + head * v.rows + (pos & (v.rows - 1));
}

// Element offset of the first element of row (slot, head, pos); -1 if the
// page is unmapped or out of the pool.
template <int LAYOUT>
__device__ __forceinline__ int64_t row_offset(const KVView &v, int slot, int head, int pos, int D) {
    if constexpr (LAYOUT == KVRT_LAYOUT_CONTIG) {
        return slot * v.slot_stride + head * v.head_stride + (int64_t)pos * v.row_stride;
    } else if constexpr (LAYOUT == KVRT_LAYOUT_RING) {
        return slot * v.slot_stride + head * v.head_stride + (int64_t)(pos % v.rows) * v.row_stride;
    } else {
        const int lp = pos >> v.block_shift;
        if (pos < 0 || lp >= v.pt_stride) return -1;
        const int page = v.page_table[(int64_t)slot * v.pt_stride + lp];
        const int row = page_row(v, page, head, pos);
        return row < 0 ? -1 : (int64_t)row * D;
    }
}

// Prefix-attention mask of a slot as a wave holds it: its length plen (0: no
// mask; wave-uniform, in an SGPR) and, in every lane, mask word (lane & 15).
// The record is read only when the launch carries masks, so launches without
// them load nothing. Both values are waited for here, so callers issue this
// next to their length load (one memory round trip for both) and before any
// LDS DMA: the compiler does not count inline-assembly DMAs, and a wait it
// placed for these loads inside a DMA-pipelined loop would drain the ring.
__device__ __forceinline__ void load_prefix(const PrefixMask *pm, int slot, int lane, int &plen, uint32_t &pw) {
    plen = 0;
    pw = 0xffffffffu;
    if (pm != nullptr) {
        plen = __builtin_amdgcn_readfirstlane(pm[slot].len);
        pw = pm[slot].bits[lane & (kPrefixWords - 1)];
        asm volatile("" ::"v"(pw));  // the word is in its register from here on
    }
}
// Mask bit of key position key (0 <= key < KVRT_MAX_PREFIX_MASK): the word
// comes from the lane that holds it (ds_bpermute), so every lane of the wave
// must call this together.
__device__ __forceinline__ bool prefix_bit(uint32_t pw, int key) {
    const uint32_t w = (uint32_t)__shfl((int)pw, (key >> 5) & (kPrefixWords - 1));
    return ((w >> (key & 31)) & 1u) != 0;
}
// Mask bits of the 8 keys k0 .. k0 + 7 (k0 >= 0; bit j: key k0 + j passes
// the mask of length plen), branch-free: the two words they span come from
// the lanes that hold them, keys at or past plen pass. Every lane of the wave
// must call this together.
__device__ __forceinline__ uint32_t prefix_bits8(uint32_t pw, int k0, int plen) {
    const int w = k0 >> 5;
    const uint32_t lo = (uint32_t)__shfl((int)pw, w & (kPrefixWords - 1));
    const uint32_t hi = (uint32_t)__shfl((int)pw, (w + 1) & (kPrefixWords - 1));
    const uint32_t bits = (uint32_t)((((uint64_t)hi << 32) | lo) >> (k0 & 31)) & 0xffu;
    const int past = plen - k0;  // keys j >= past are beyond the mask
    const uint32_t open = past <= 0 ? 0xffu : past >= 8 ? 0u : (0xffu << past) & 0xffu;
    return bits | open;
}


// q = x / d and r = x % d for x >= 0 and a wave-uniform d > 0: a shift and a
// mask when d is a power of two (a uniform branch), else the division.
__device__ __forceinline__ void udivmod_uniform(int x, int d, int &q, int &r) {
    if ((d & (d - 1)) == 0) {
        q = x >> __builtin_ctz((unsigned)d);
        r = x & (d - 1);
    } else {
        q = x / d;
        r = x - q * d;
    }
}
__device__ __forceinline__ int umod_uniform(int x, int d) {
    int q, r;
    udivmod_uniform(x, d, q, r);
    return r;
}

// A wave's window of page-table entries: lane i holds the entry of logical
// page win0 + i of the slot (-1 outside the table).
__device__ __forceinline__ int load_page_window(const KVView &v, int slot, int win0, int lane) {
    const int lp = win0 + lane;
    return page_in_table(lp, v.pt_stride) ? v.page_table[(int64_t)slot * v.pt_stride + lp] : -1;
}
// Element offset of row pos of a head on a page; -1 if the page is unmapped
// or out of the pool.
__device__ __forceinline__ int64_t page_row_offset(const KVView &v, int page, int head, int pos, int D) {
    const int row = page_row(v, page, head, pos);
    return row < 0 ? -1 : (int64_t)row * D;
}

// LDS DMA: global_load_lds_dwordx4 moves lane l's 16 bytes at g to LDS byte
// M0 + 16 * l without passing through registers. It is issued from inline
// assembly (the LDS address is an M0 operand the compiler sets up), so the
// compiler neither tracks these loads nor inserts its own (all-or-nothing)
// waits for them: the decode waits with explicit vmcnt waits — vector loads
// complete in issue order, so vmcnt(N) means every DMA but the N most recent
// has landed — and reads the LDS back only after such a wait.
__device__ __forceinline__ void dma_load16(const void *g, uint32_t lds) {
    asm volatile("global_load_lds_dwordx4 %0, off nt" ::"v"(g), "{m0}"(lds) : "memory");
}
// 4 bytes per lane, to LDS byte M0 + 4 * l.
__device__ __forceinline__ void dma_load4(const void *g, uint32_t lds) {
    asm volatile("global_load_lds_dword %0, off nt" ::"v"(g), "{m0}"(lds) : "memory");
}
// The same without the streaming hint, for tiles other workgroups read again.
__device__ __forceinline__ void dma_load16_cached(const void *g, uint32_t lds) {
    asm volatile("global_load_lds_dwordx4 %0, off" ::"v"(g), "{m0}"(lds) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vmem() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
// Waits until at most n * STEP vector memory operations are outstanding,
// n in [0, NMAX] (wave-uniform).
template <int STEP, int NMAX>
__device__ __forceinline__ void wait_vmem_steps(int n) {
    if constexpr (NMAX > 0) {
        if (n >= NMAX) {
            wait_vmem<NMAX * STEP>();
            return;
        }
        wait_vmem_steps<STEP, NMAX - 1>(n);
    } else {
        wait_vmem<0>();
    }
}
__device__ __forceinline__ void wait_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
template <class T>
__device__ __forceinline__ uint32_t lds_addr(const T *p) {
    return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) T *)p;
}

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef short s16x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

// gfx950 LDS transpose read: in each group of 16 lanes, lane s gives the
// address of 4 consecutive bf16; lane t = 4a + e receives element e of the
// chunks of lanes a, a + 4, a + 8, a + 12.
__device__ __forceinline__ uint2 lds_read_tr16(const uint16_t *p) {
    const s16x4_t x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4_t __attribute__((address_space(3))) *)(p));
    return __builtin_bit_cast(uint2, x);
}

}  // namespace kvrt
