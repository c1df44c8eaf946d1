// Staging slots of large host copies: pinned memory and an event each.  The runtime's
// calls come through Api, so that the set-up and its failures can be checked without a
// device.
#pragma once

#include <cstddef>

namespace opsec {

template <typename Api>
struct StageSlots {
    static constexpr int N = 8;
    static constexpr size_t BYTES = (size_t)4 << 20;
    char* base = nullptr;            // N slots, pinned
    typename Api::event_t ev[N] = {};

    char* slot(int i) const { return base + (size_t)i * BYTES; }
    // All slots, or none; a failed call's error is taken back, so that no later check reports it
    // (the copy that wanted the slots goes through the runtime).
    bool make() {
        if (base) return true;
        void* p = nullptr;
        if (!Api::host_alloc(&p, N * BYTES)) {
            Api::clear_error();
            return false;
        }
        for (int i = 0; i < N; i++)
            if (!Api::event_create(&ev[i])) {
                Api::clear_error();
                while (i-- > 0) Api::event_destroy(ev[i]);
                Api::host_free(p);
                return false;
            }
        base = (char*)p;
        return true;
    }
    void release() {
        if (!base) return;
        for (int i = 0; i < N; i++) Api::event_destroy(ev[i]);
        Api::host_free(base);
        base = nullptr;
    }
};

}  // namespace opsec
