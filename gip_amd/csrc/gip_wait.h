// The host's wait for a sequence number that a kernel stores in pinned
// memory (no device code; also compiled into a CPU test).
#pragma once

#include <cstdint>

namespace gip {

// A number has arrived when it or a later one is there: two threads on one
// context may ask one after the other, and the first then finds the second's.
inline bool seq_reached(const uint64_t *flag, uint64_t want) {
    return (int64_t)(__atomic_load_n(flag, __ATOMIC_ACQUIRE) - want) >= 0;
}

enum { WAIT_OK = 0, WAIT_MISSING = 1 };

// Spins until the number has arrived.  Every kWaitQuery spins (tens of ms:
// the query itself queues work) query() is asked for the stream: < 0 its
// work goes on, 0 it is done (without the number: WAIT_MISSING), > 0 it has
// failed (returned + 1).
constexpr unsigned kWaitQuery = 1u << 20;
template <class QUERY>
inline int wait_seq(const uint64_t *flag, uint64_t want, const QUERY &query) {
    for (unsigned spin = 1;; ++spin) {
        if (seq_reached(flag, want)) return WAIT_OK;
        if (spin & (kWaitQuery - 1)) {
            __builtin_ia32_pause();
            continue;
        }
        const int q = query();
        if (q > 0) return q + 1;
        if (q == 0) return seq_reached(flag, want) ? WAIT_OK : WAIT_MISSING;
    }
}

}  // namespace gip
