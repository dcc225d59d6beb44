// stream_slots.h -- a context's scratch buffers, one per stream that called it (internal; no HIP call, so
// the host tests build it with g++).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace ftdx {

// Calls on different streams may overlap, so each stream has a buffer of its own; a fifth stream does
// without, unless one of the four has not called for kIdleCalls calls: a program that makes streams and
// destroys them would otherwise leave them the slots for good.  Whoever takes over a slot allocates it
// anew (its stream's last work may still run).  A context's buffers are on its own device: a call from another device, whose streams may
// have the same handles (the null stream does), does without too.
struct StreamSlot {
    bool used = false;
    void* stream = nullptr;
    uint8_t* rows = nullptr;
    size_t cap = 0;
    uint64_t last = 0;  // the call that used it last
};

class StreamSlots {
public:
    static constexpr uint64_t kIdleCalls = 64;
    StreamSlot slots[4];

    // The slot of a call from `stream` of device `dev` into a context of device `own`, nullptr for none.
    // Its rows are the caller's to use as they are only if slot->stream == stream; else to release.
    StreamSlot* pick(int own, int dev, void* stream) {
        if (own < 0 || dev != own) return nullptr;
        ++calls_;
        StreamSlot* pick = nullptr;
        for (auto& s : slots)
            if (s.used && s.stream == stream) pick = &s;
        for (auto& s : slots)
            if (!pick && !s.used) pick = &s;
        if (!pick) {
            StreamSlot* idle = &slots[0];
            for (auto& s : slots)
                if (s.last < idle->last) idle = &s;
            if (calls_ - idle->last > kIdleCalls) pick = idle;
        }
        return pick;
    }

    // After a failed allocation of `need` bytes: no other of that size or more for kIdleCalls calls (each
    // would cost what the failed one did).
    bool refused(size_t need) const { return refused_ && need >= refused_ && calls_ - refused_at_ <= kIdleCalls; }
    void refuse(size_t need) {
        refused_ = need;
        refused_at_ = calls_;
    }

    // The call of the last pick has its rows.
    void use(StreamSlot* slot, void* stream) {
        slot->used = true;
        slot->stream = stream;
        slot->last = calls_;
    }

private:
    uint64_t calls_ = 0, refused_at_ = 0;
    size_t refused_ = 0;
};

}  // namespace ftdx
