// Staging slots of large host copies: a pinned buffer and an event each.  The runtime's
// calls come through Api, so that the set-up and its failures can be checked without a
// device.
#pragma once

#include <cstddef>

namespace opsec {

template <typename Api>
struct StageSlots {
    static constexpr int N = 8;
    static constexpr size_t BYTES = (size_t)4 << 20;
    void* buf[N] = {};
    typename Api::event_t ev[N] = {};
    int n = 0;   // slots made

    // At least `want` slots, or as many as could be made; returns min(n, want).  A failed call's
    // error is taken back, so that no later check reports it: the copy goes on with fewer slots,
    // or without.
    int make(int want) {
        while (n < want) {
            if (!Api::host_alloc(&buf[n], BYTES)) {
                Api::clear_error();
                break;
            }
            if (!Api::event_create(&ev[n])) {
                Api::clear_error();
                Api::host_free(buf[n]);
                break;
            }
            n++;
        }
        return n < want ? n : want;
    }
    void release() {
        while (n > 0) {
            n--;
            Api::host_free(buf[n]);
            Api::event_destroy(ev[n]);
        }
    }
};

}  // namespace opsec
