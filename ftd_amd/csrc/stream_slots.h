// stream_slots.h -- a context's scratch buffers, one per stream that called it (internal; no HIP call, so
// the host tests build it with g++).
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace ftdx {

// Calls on different streams may overlap, so each stream has a buffer of its own; a fifth stream does
// without.  A context's buffers are on its own device: a call from another device, whose streams may
// have the same handles (the null stream does), does without too.
struct StreamSlot {
    bool used = false;
    void* stream = nullptr;
    uint8_t* rows = nullptr;
    size_t cap = 0;
};

class StreamSlots {
public:
    StreamSlot slots[4];

    // The slot of a call from `stream` of device `dev` into a context of device `own`, nullptr for none.
    StreamSlot* pick(int own, int dev, void* stream) {
        if (own < 0 || dev != own) return nullptr;
        for (auto& s : slots)
            if (s.used && s.stream == stream) return &s;
        for (auto& s : slots)
            if (!s.used) return &s;
        return nullptr;
    }
};

}  // namespace ftdx
