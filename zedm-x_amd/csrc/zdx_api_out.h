// zdx_api_out.h — where an output array of the per-pair call goes: its slot in
// the call's pinned host memory or a device buffer that the host copies.
// Shared by the host, which makes the buffer before the array's rows are
// counted (zdx_api.cpp), the packing kernels, which know them
// (zdx_kernels.hip), and a host test.
#pragma once
#include <cstdint>

#ifndef ZDX_HD
#ifdef __HIPCC__
#define ZDX_HD __host__ __device__
#else
#define ZDX_HD
#endif
#endif

namespace zdx {

constexpr int64_t API_SLOT = (int64_t)512 << 10;   // an output array up to this size; a larger one is copied

// An output of up to cap rows of per entries; host: its slot (nullptr: not
// wanted).
template <class T>
struct ApiOut {
    T *host = nullptr, *dev = nullptr;
    int64_t cap = 0;
    int per = 1;
    // Rows in the slot?  (so that the host reads them there)
    ZDX_HD bool in_slot(int64_t rows) const { return rows * per * (int64_t)sizeof(T) <= API_SLOT; }
    // Entries of the device buffer: that of the capacity where the rows may
    // exceed the slot, else none.
    ZDX_HD int64_t dev_entries() const { return host && !in_slot(cap) ? cap * per : 0; }
    // Where `rows` rows are stored.  nullptr: nowhere -- not wanted, or more
    // than the capacity (the call then fails with the totals).  Not more than
    // the capacity and not in the slot means that the capacity is not either,
    // so dev is there.
    ZDX_HD T* at(int64_t rows) const { return !host || rows > cap ? nullptr : (in_slot(rows) ? host : dev); }
};

}  // namespace zdx
