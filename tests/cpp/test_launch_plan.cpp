// Host-side launch planning of libftdx.so (built with g++ under ASan + UBSan, no GPU): the batches
// per chunk of the pipelined HERK, and its per-stream scratch slots.  Prints "ALL PASSED" on success.
#include <cstdio>

#include "herk_chunks.h"
#include "stream_slots.h"

static int g_fail = 0;
#define CHECK(c)                                                              \
    do {                                                                      \
        if (!(c)) {                                                           \
            std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #c);          \
            ++g_fail;                                                         \
        }                                                                     \
    } while (0)

// Every chunk a loop steps by is at least 1, and a chunk's input batches fit a grid's y dimension;
// a cap of 0 says that one batch's segments alone do not.
static void test_chunks() {
    using namespace ftdx;
    for (int nseg : {1, 2, 3, 255, 32767, 32768, 65535, 65536, 70000, 1 << 20})
        for (int batch : {1, 2, 7, 96, 70000}) {
            const int cap = frag_chunk_cap(64, 16, nseg, batch);
            CHECK((cap > 0) == (nseg <= 65535));
            CHECK((int64_t)cap * nseg <= 65535);
            for (int c : {0, 1, cap}) {
                const int chunk = pick_chunk_of(512, 3, batch, c);
                CHECK(chunk >= 1 && chunk <= (c > 1 ? c : 1));
            }
        }
}

static void* stream(int i) { return reinterpret_cast<void*>((uintptr_t)i); }

// A slot is one stream's of one device: streams of two devices may have the same handle, the null
// stream always does.
static void test_slots_of_two_devices() {
    ftdx::StreamSlots p;
    ftdx::StreamSlot* s = p.pick(0, 0, stream(0));
    CHECK(s);
    p.use(s, stream(0));
    CHECK(p.pick(0, 0, stream(0)) == s);
    CHECK(p.pick(0, 1, stream(0)) == nullptr);
    CHECK(p.pick(0, 1, stream(8)) == nullptr);
    CHECK(p.pick(0, -1, stream(0)) == nullptr);
    CHECK(p.pick(-1, -1, stream(0)) == nullptr);
    CHECK(p.pick(0, 0, stream(8)) != s);
}

// A program that makes a stream for every few calls keeps getting slots; five streams that take turns do
// not take them from each other.
static void test_slots_come_back() {
    ftdx::StreamSlots p;
    int served = 0, calls = 0;
    for (int st = 1; st <= 40; ++st)
        for (int c = 0; c < 20; ++c, ++calls)
            if (ftdx::StreamSlot* s = p.pick(0, 0, stream(st))) {
                p.use(s, stream(st));
                ++served;
            }
    CHECK(served > calls / 4);  // 4 slots of 64 idle calls for streams of 20 calls each
    ftdx::StreamSlots q;
    for (int turn = 0; turn < 200; ++turn)
        for (int st = 1; st <= 5; ++st) {
            ftdx::StreamSlot* s = q.pick(0, 0, stream(st));
            CHECK((s != nullptr) == (st <= 4));
            if (!s) continue;
            CHECK(!s->used || s->stream == stream(st));
            q.use(s, stream(st));
        }
}

// An allocation that failed is not tried again on every call.
static void test_refused_allocations() {
    ftdx::StreamSlots p;
    int tries = 0;
    for (int c = 0; c < 650; ++c) {
        CHECK(p.pick(0, 0, stream(1)));
        CHECK(!p.refused(99));
        if (p.refused(100)) continue;
        CHECK(c == 0 || !p.refused(200));
        ++tries;
        p.refuse(100);
        CHECK(p.refused(100) && p.refused(200));
    }
    CHECK(tries == 10);
}

// Inputs that no cache holds cost the same on every pass.
static void test_cold_inputs() {
    CHECK(ftdx::pipe_cold_ms((int64_t)4096 * 2048 * 96) == 0.0);
    CHECK(ftdx::pipe_cold_ms(268435456) == 0.0);
    const double ms = ftdx::pipe_cold_ms(1024 * 1024 * 64);
    CHECK(ms > 0.004 && ms < 0.008);
    CHECK(ftdx::pipe_cold_ms(0) == 0.0);
}

int main() {
    test_chunks();
    test_cold_inputs();
    test_refused_allocations();
    test_slots_of_two_devices();
    test_slots_come_back();
    if (g_fail == 0) std::printf("ALL PASSED\n");
    return g_fail != 0;
}
