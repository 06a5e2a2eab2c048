// Growth of a buffer of temporary memory. Host code.
#pragma once

#include <cstddef>
#include <cstdint>

namespace rf {

// Gives `buf` (of `have` bytes) at least `need` bytes; a buffer that grows does so by half at least. Launches enqueued earlier may
// still read the old one, so it is not freed but goes to `retired`, and only once the new one is there: where `alloc` fails (returns
// other than zero) the caller's next plan finds the buffer that it had.
template <typename T, typename Retired, typename Alloc>
auto grow_buffer(T *&buf, size_t &have, size_t need, Retired &retired, Alloc alloc) -> decltype(alloc((void **)nullptr, need)) {
    if (need <= have) return {};
    const size_t want = need > have + have / 2 ? need : have + have / 2;
    void *fresh = nullptr;
    const auto error = alloc(&fresh, want);
    if (error) return error;
    if (buf) retired.push_back(buf);
    buf = (T *)fresh;
    have = want;
    return error;
}

// A growth that failed, of a buffer that a plan can do without: the next 63 calls that want as much or more take the plan without it
// and do not pay for another allocation that fails. One in 64 asks again, memory may have been freed since.
struct RefusedGrowth {
    size_t bytes = SIZE_MAX;
    int calls = 0;
    bool ask(size_t need) { return need < bytes || ++calls >= 64; }
    void answer(size_t need, bool grown) {
        bytes = grown ? SIZE_MAX : need < bytes ? need : bytes;
        calls = 0;
    }
};

}  // namespace rf
