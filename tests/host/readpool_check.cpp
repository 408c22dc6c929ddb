// ReadPool (lq_readpool.h) against two devices: a slot's event can be recorded on
// the stream it was taken for, whichever device is current; the caller's device
// stays current; no slot is in two hands; surplus slots are freed.
#include "lq_readpool.h"

#include <cstdio>
#include <thread>
#include <vector>

static std::atomic<int> bad{0}, calls{0};

static void expect(bool ok, const char* what) {
    if (!ok && bad++ < 10) printf("%s\n", what);
}

int main() {
    static lq::ReadPool pool;
    ihipStream on0{0}, on1{1};
    for (int current : {0, 1})
        for (hipStream_t s : {&on0, &on1, (hipStream_t) nullptr, &on1, &on0}) {
            (void)hipSetDevice(current);
            lq::ReadSlot r;
            expect(pool.take(s, &r), "take");
            expect(hipEventRecord(r.event, s) == hipSuccess, "event of another device than the stream's");
            expect(t_device == current, "the caller's device changed");
            pool.give(r);
        }
    // more callers at once than slots are kept: each hand keeps its own words
    constexpr int kThreads = 3 * lq::kReadSlots, kCalls = 200;
    std::vector<std::thread> ts;
    for (int i = 0; i < kThreads; i++)
        ts.emplace_back([&, i] {
            (void)hipSetDevice(i & 1);
            for (int c = 0; c < kCalls; c++) {
                const hipStream_t s = (i + c) % 3 ? &on0 : &on1;
                lq::ReadSlot r;
                if (!pool.take(s, &r)) { expect(false, "take"); return; }
                r.host[0] = i;
                r.host[1] = c;
                expect(hipEventRecord(r.event, s) == hipSuccess, "event of another device than the stream's");
                std::this_thread::yield();
                expect(r.host[0] == i && r.host[1] == c, "a slot in two hands");
                pool.give(r);
                calls++;
            }
        });
    for (auto& t : ts) t.join();
    expect(calls == kThreads * kCalls, "calls that did not end");
    std::vector<lq::ReadSlot> held(lq::kReadSlots + 5);
    for (auto& r : held) expect(pool.take(&on0, &r), "take");
    for (auto& r : held) pool.give(r);
    int kept = 0;
    for (const auto& p : pool.slots) kept += p.host != nullptr;
    expect(kept == lq::kReadSlots && n_events == kept && n_host == kept, "surplus slots were not freed");
    printf("%d calls, %d bad\n", (int)calls, (int)bad);
    return bad != 0;
}
