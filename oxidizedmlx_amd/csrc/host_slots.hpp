// host_slots.hpp — the pinned slots that copies to the host go through
// (host_copy.cpp): who gets how many, and when one is pinned or given back.
// Plain C++, so that its rules can be checked without a GPU.
//
// A new slot is dear: hipHostMalloc of 2 MiB takes 15-200 us, and the CPU's
// first reading of it, page by page, 800 us, where a kept one saves 40-160 us
// of a 2 MiB copy. So slots are earned, one for every EARN bytes copied, the
// copy at hand included: the first KEPT by all that the process has copied,
// further ones by what was copied since there was no Stream or decoder. A copy
// that cannot have the slots it needs takes the runtime's way. Slots are kept
// for later copies; when the last Stream or decoder goes, all but KEPT are
// unpinned.
#pragma once

#include <algorithm>
#include <cstddef>
#include <mutex>

namespace mlxhip {

class HostSlots {
public:
    static constexpr int MAX = 16;                     // pinned at any time
    static constexpr int KEPT = 4;                     // without an owner
    static constexpr size_t EARN = size_t(8) << 20;

    HostSlots(char* (*pin)(), void (*unpin)(char*)) : pin_(pin), unpin_(unpin) {}

    // Up to `want` slots for a copy of `bytes`, at least `need` or none.
    int take(size_t bytes, int want, int need, char** out) {
        int n = 0, fresh = 0;
        {
            std::lock_guard<std::mutex> g(mu_);
            copied_ += std::min(bytes, EARN * KEPT - copied_);
            lately_ += std::min(bytes, EARN * MAX - lately_);
            const int may = (int)(std::max(copied_, lately_) / EARN) - total_;
            n = std::min(want, free_n_);
            fresh = std::max(0, std::min(want - n, may));
            if (n + fresh < need) return 0;
            for (int i = 0; i < n; ++i) out[i] = free_[--free_n_];
            total_ += fresh;
        }
        int made = 0;
        while (made < fresh && (out[n + made] = pin_()) != nullptr) ++made;
        if (made < fresh) {
            std::lock_guard<std::mutex> g(mu_);
            total_ -= fresh - made;
        }
        if (n + made >= need) return n + made;
        give(out, n + made);
        return 0;
    }

    void give(char* const* slots, int n) {
        char* drop[MAX];
        int drops = 0;
        {
            std::lock_guard<std::mutex> g(mu_);
            for (int i = 0; i < n; ++i) free_[free_n_++] = slots[i];
            if (owners_ == 0) drops = trim(drop);
        }
        for (int i = 0; i < drops; ++i) unpin_(drop[i]);
    }

    void retain() {
        std::lock_guard<std::mutex> g(mu_);
        ++owners_;
    }

    void release() {
        char* drop[MAX];
        int drops = 0;
        {
            std::lock_guard<std::mutex> g(mu_);
            if (--owners_ == 0) {
                lately_ = 0;
                drops = trim(drop);
            }
        }
        for (int i = 0; i < drops; ++i) unpin_(drop[i]);
    }

private:
    // Free slots beyond KEPT, no longer counted; mu_ is held.
    int trim(char** drop) {
        int n = 0;
        while (free_n_ > 0 && total_ > KEPT) {
            drop[n++] = free_[--free_n_];
            --total_;
        }
        return n;
    }

    std::mutex mu_;
    char* (*pin_)();
    void (*unpin_)(char*);
    char* free_[MAX] = {};
    int free_n_ = 0, total_ = 0, owners_ = 0;
    size_t copied_ = 0, lately_ = 0;  // up to what can be earned by them
};

}  // namespace mlxhip
