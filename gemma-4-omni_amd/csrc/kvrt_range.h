// kvrt_range.h — index arithmetic of the prefill kernel's key ranges and of
// page-table reads. Plain C++ beside the device code, so that the host can
// check it over lengths a caller reaches only through graph replays.
#pragma once

#if defined(__HIPCC__)
#define KVRT_HD __host__ __device__ __forceinline__
#else
#define KVRT_HD inline
#endif

namespace kvrt {

struct KeyRange {
    int kstart, kend;  // keys [kstart, kend); kend <= kstart: none
};

// Keys of the queries qf .. ql, the first at position base_pos + qf (window 0:
// no window): range ks of nks in whole blocks of `block` keys. base_pos is
// negative where the device length is below Q (a graph replayed after a
// rollback): queries before position 0 see no keys, and kend may be <= 0.
KVRT_HD KeyRange prefill_range(int base_pos, int qf, int ql, int window, int nks, int ks, int block) {
    int kend = base_pos + ql + 1;
    const int w0 = base_pos + qf - window + 1;
    int kstart = window > 0 && w0 > 0 ? w0 : 0;
    if (nks > 1) {
        const int span = (kend - kstart + nks - 1) / nks;
        const int len = (span + block - 1) / block * block;
        const int k0 = kstart + ks * len;
        kend = kend < k0 + len ? kend : k0 + len;
        kstart = k0 < kend ? k0 : kend;
    }
    return {kstart, kend};
}

// Whether logical page lp has an entry in a slot's page table.
KVRT_HD bool page_in_table(int lp, int pt_stride) { return (unsigned)lp < (unsigned)pt_stride; }

}  // namespace kvrt
