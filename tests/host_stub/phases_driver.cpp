// What a dispatch of single phases launches, in a host-only build (see hip/hip_runtime.h beside this file): a later phase
// goes on from the scratch that the earlier ones left only where that scratch is the call's own, and otherwise runs them
// again.  Launches are counted (kernels_stub.cpp); addresses are made-up numbers.
#include <atomic>
#include <cstdio>
#include <vector>

#include <hip/hip_runtime.h>

#include "mooncake_ep_hip.h"

namespace mcep {
extern std::atomic<long> g_stub_counts, g_stub_packs, g_stub_finishes, g_stub_one_launch;
}

namespace {

int g_failures = 0;

struct Parts {
    long count, pack, finish, one;
};
Parts now() {
    return {mcep::g_stub_counts.load(), mcep::g_stub_packs.load(), mcep::g_stub_finishes.load(), mcep::g_stub_one_launch.load()};
}

struct Call {
    int R, T, H, K, E;
    bool fp8 = true;
    int gen = 0;            // its tensors
    uint64_t at(int rank, int field) const {
        return 0x100000000ull + ((uint64_t)gen << 32) + ((uint64_t)rank << 24) + ((uint64_t)field << 16);
    }
    int run(mc_ep_world_t* w, int phases, hipStream_t stream = nullptr, bool noalloc = false) const {
        std::vector<uint64_t> v[7];
        for (int f = 0; f < 7; ++f)
            for (int r = 0; r < R; ++r) v[f].push_back(at(r, f));
        std::vector<int32_t> n(R, T);
        if (noalloc)
            return mc_ep_world_dispatch_noalloc(w, v[0].data(), v[1].data(), n.data(), H, K, T, E, fp8, v[2].data(),
                                                fp8 ? v[3].data() : nullptr, v[4].data(), v[5].data(), v[6].data(),
                                                (uint64_t)stream);
        return mc_ep_world_dispatch(w, v[0].data(), v[1].data(), n.data(), H, K, T, E, fp8, v[2].data(),
                                    fp8 ? v[3].data() : nullptr, v[4].data(), v[5].data(), v[6].data(), phases,
                                    (uint64_t)stream);
    }
};

constexpr int LAYOUT = MC_EP_PHASE_LAYOUT, DATA = MC_EP_PHASE_DATA, FINISH = MC_EP_PHASE_FINISH, ALL = MC_EP_PHASE_ALL;

void check(const char* what, const Parts& before, int rc, long count, long pack, long finish, long one) {
    const Parts p = now();
    const Parts d{p.count - before.count, p.pack - before.pack, p.finish - before.finish, p.one - before.one};
    const bool ok = rc == MC_EP_OK && d.count == count && d.pack == pack && d.finish == finish && d.one == one;
    if (!ok) {
        ++g_failures;
        std::printf("FAILED %s: rc %d (%s), count %ld pack %ld finish %ld one launch %ld, expected %ld %ld %ld %ld\n", what, rc,
                    rc ? mc_ep_last_error() : "", d.count, d.pack, d.finish, d.one, count, pack, finish, one);
    }
}
#define EXPECT(what, call, ...)            \
    do {                                   \
        const Parts before_ = now();       \
        const int rc_ = (call);            \
        check(what, before_, rc_, __VA_ARGS__); \
    } while (0)

struct World {
    mc_ep_world_t* w = nullptr;
    explicit World(int ranks) {
        if (mc_ep_world_create(ranks, &w) != MC_EP_OK) ++g_failures;
    }
    ~World() { mc_ep_world_destroy(w); }
    operator mc_ep_world_t*() const { return w; }
};

// 5120 selections, 512, and (too many for one launch) 32768 of the one rank
const Call kShared{1, 640, 2048, 8, 16}, kSmall{1, 64, 1024, 8, 16}, kLarge{1, 4096, 1024, 8, 16};

void after_one_launch(Call c, const char* name) {
    std::printf("a later phase by itself after the one launch: %s\n", name);
    {
        World w(c.R);
        EXPECT("larger", kLarge.run(w, ALL), 1, 1, 1, 0);
        EXPECT("all", c.run(w, ALL), 0, 0, 0, 1);
        // nothing in the scratch is this call's: the whole call again (bf16 has no last phase)
        EXPECT("finish", c.run(w, FINISH), 0, 0, c.fp8 ? 0 : 1, c.fp8 ? 1 : 0);
        EXPECT("data", c.run(w, DATA), 1, 1, 0, 0);
        EXPECT("data again", c.run(w, DATA), 0, 1, 0, 0);
        EXPECT("finish now", c.run(w, FINISH), 0, 0, 1, 0);
        EXPECT("finish again", c.run(w, FINISH), 0, 0, 1, 0);
    }
    {
        World w(c.R);
        EXPECT("all", c.run(w, ALL), 0, 0, 0, 1);
        EXPECT("data", c.run(w, DATA), 1, 1, 0, 0);
        EXPECT("all", c.run(w, ALL), 0, 0, 0, 1);
        EXPECT("data and finish", c.run(w, DATA | FINISH), 0, 0, 0, 1);
    }
}

void after_another_dispatch() {
    std::puts("a later phase by itself after another dispatch of the world");
    World w(1);
    Call other = kLarge;
    other.gen = 1;
    EXPECT("layout and data", kLarge.run(w, LAYOUT | DATA), 1, 1, 0, 0);
    EXPECT("other tensors", other.run(w, ALL), 1, 1, 1, 0);
    EXPECT("finish of the first", kLarge.run(w, FINISH), 1, 1, 1, 0);
    EXPECT("finish of the first again", kLarge.run(w, FINISH), 0, 0, 1, 0);
    Call shape = kLarge;
    shape.H = 1152;
    EXPECT("another hidden", shape.run(w, FINISH), 1, 1, 1, 0);
    shape = kLarge;
    shape.T = 2560;
    EXPECT("another number of tokens", shape.run(w, DATA), 1, 1, 0, 0);
    shape.fp8 = false;
    EXPECT("another payload", shape.run(w, DATA), 1, 1, 0, 0);
    EXPECT("layout, no data", kLarge.run(w, LAYOUT), 1, 0, 0, 0);
    EXPECT("finish before data", kLarge.run(w, FINISH), 0, 1, 1, 0);
    EXPECT("layout and finish", kLarge.run(w, LAYOUT | FINISH), 1, 1, 1, 0);
    if (mc_ep_world_set_option(w, "routing_sum", 0) != MC_EP_OK) ++g_failures;
    EXPECT("another plan", kLarge.run(w, DATA), 1, 1, 0, 0);
    EXPECT("without allocating", kSmall.run(w, ALL, nullptr, true), 0, 0, 0, 1);
    EXPECT("in between, with scratch of its own", kLarge.run(w, FINISH), 0, 0, 1, 0);
    EXPECT("without allocating", kSmall.run(w, ALL, nullptr, true), 0, 0, 0, 1);
    EXPECT("after it and after the call was complete", kLarge.run(w, FINISH), 1, 1, 1, 0);
}

void phases_in_order() {
    std::puts("phases in order: each launches what is its own");
    for (const Call& c : {kShared, kSmall, kLarge})
        for (int fp8 = 0; fp8 < 2; ++fp8) {
            World w(1);
            Call k = c;
            k.fp8 = fp8 != 0;
            for (int i = 0; i < 3; ++i) {
                EXPECT("layout", k.run(w, LAYOUT), 1, 0, 0, 0);
                EXPECT("data", k.run(w, DATA), 0, 1, 0, 0);
                EXPECT("finish", k.run(w, FINISH), 0, 0, 1, 0);
                EXPECT("layout", k.run(w, LAYOUT), 1, 0, 0, 0);
                EXPECT("data and finish", k.run(w, DATA | FINISH), 0, 1, 1, 0);
            }
        }
}

void recorded() {
    std::puts("recorded calls");
    hipStream_t s = nullptr;
    if (hipStreamCreateWithFlags(&s, hipStreamNonBlocking) != hipSuccess) ++g_failures;
    {
        // a graph's one-launch dispatch: its replays are not seen here, so what an eager call left when it was complete
        // is no longer trusted; phases asked for one after the other are
        World w(1);
        EXPECT("eager", kShared.run(w, ALL, s), 0, 0, 0, 1);
        hip_stub::g_capture = 1;
        EXPECT("recorded", kShared.run(w, ALL, s), 0, 0, 0, 1);
        EXPECT("recorded finish", kShared.run(w, FINISH, s), 0, 0, 0, 1);
        EXPECT("recorded data", kShared.run(w, DATA, s), 1, 1, 0, 0);
        EXPECT("recorded finish of that", kShared.run(w, FINISH, s), 0, 0, 1, 0);
        hip_stub::g_capture = 0;
        EXPECT("eager phases", kShared.run(w, LAYOUT, s), 1, 0, 0, 0);
        EXPECT("eager phases", kShared.run(w, DATA, s), 0, 1, 0, 0);
        EXPECT("eager phases", kShared.run(w, FINISH, s), 0, 0, 1, 0);
        EXPECT("finish after a replay, perhaps", kShared.run(w, FINISH, s), 0, 0, 0, 1);
        EXPECT("still one launch", kShared.run(w, ALL, s), 0, 0, 0, 1);
    }
    {
        // a graph that holds a later phase alone: the eager dispatches that it goes on from have to leave it their state
        World w(1);
        EXPECT("eager", kShared.run(w, LAYOUT | DATA, s), 1, 1, 0, 0);
        hip_stub::g_capture = 2;
        EXPECT("recorded", kShared.run(w, FINISH, s), 0, 0, 1, 0);
        hip_stub::g_capture = 0;
        EXPECT("eager", kShared.run(w, ALL, s), 1, 1, 1, 0);
    }
    {
        // a graph's separate launches: their replays fill the scratch, which an eager call that is complete may not take for
        // its own any more; nor is what a recorded call leaves there before it has been replayed
        World w(1);
        Call other = kLarge;
        other.gen = 1;
        other.H = 2048;
        EXPECT("eager", other.run(w, ALL, s), 1, 1, 1, 0);
        hip_stub::g_capture = 3;
        EXPECT("recorded", other.run(w, ALL, s), 1, 1, 1, 0);
        EXPECT("recorded finish", other.run(w, FINISH, s), 0, 0, 1, 0);
        hip_stub::g_capture = 0;
        EXPECT("finish of the recorded call", other.run(w, FINISH, s), 1, 1, 1, 0);
        EXPECT("eager", kLarge.run(w, ALL, s), 1, 1, 1, 0);
        EXPECT("finish after a replay, perhaps", kLarge.run(w, FINISH, s), 1, 1, 1, 0);
        EXPECT("data after a replay, perhaps", kLarge.run(w, DATA, s), 1, 1, 0, 0);
        EXPECT("finish right behind it", kLarge.run(w, FINISH, s), 0, 0, 1, 0);
        hip_stub::g_capture = 4;
        EXPECT("recorded", kLarge.run(w, LAYOUT | DATA, s), 1, 1, 0, 0);
        hip_stub::g_capture = 5;
        EXPECT("the last phase in a graph of its own", kLarge.run(w, FINISH, s), 0, 0, 1, 0);
        hip_stub::g_capture = 0;
        EXPECT("data and finish, without a replay", kLarge.run(w, DATA | FINISH, s), 1, 1, 1, 0);
    }
    if (hipStreamDestroy(s) != hipSuccess) ++g_failures;
}

// a round whose second part waits for its hook: an allocation-free dispatch in between changes nothing of it
void rounds_in_two_parts() {
    std::puts("a round in two parts");
    World w(1);
    mc_ep_buffer_t* b = nullptr;
    if (mc_ep_buffer_create(w, 0, (int64_t)mc_ep_get_buffer_size_hint(640, 2048, 1, 16), 0, &b) != MC_EP_OK) ++g_failures;
    mc_ep_event_t* ev = nullptr;
    mc_ep_hook_t* hook = nullptr;
    const Call c = kShared;
    EXPECT("first part", mc_ep_buffer_dispatch(b, c.at(0, 0), c.at(0, 1), c.at(0, 9), c.T, c.H, c.K, c.T, c.E, -1, 1, c.at(0, 2),
                                               c.at(0, 3), c.at(0, 4), c.at(0, 5), c.at(0, 6), 0, 1, 0, &ev, &hook), 1, 1, 0, 0);
    EXPECT("without allocating", kSmall.run(w, ALL, nullptr, true), 0, 0, 0, 1);
    EXPECT("second part", mc_ep_hook_call(hook), 0, 0, 1, 0);
    mc_ep_hook_destroy(hook);
    // ... and a later phase of another call has it enqueued first
    EXPECT("first part", mc_ep_buffer_dispatch(b, c.at(0, 0), c.at(0, 1), c.at(0, 9), c.T, c.H, c.K, c.T, c.E, -1, 1, c.at(0, 2),
                                               c.at(0, 3), c.at(0, 4), c.at(0, 5), c.at(0, 6), 0, 1, 0, &ev, &hook), 1, 1, 0, 0);
    EXPECT("another call's data", kLarge.run(w, DATA), 1, 1, 1, 0);
    EXPECT("second part, done", mc_ep_hook_call(hook), 0, 0, 0, 0);
    mc_ep_hook_destroy(hook);
    mc_ep_buffer_destroy(b);
}

}  // namespace

int main() {
    after_one_launch(kShared, "several tokens a block");
    after_one_launch(kSmall, "a token a block");
    Call bf16 = kShared;
    bf16.fp8 = false;
    after_one_launch(bf16, "bf16");
    after_another_dispatch();
    phases_in_order();
    recorded();
    rounds_in_two_parts();
    std::printf("%s (%d failed checks)\n", g_failures ? "FAILED" : "ok", g_failures);
    return g_failures ? 1 : 0;
}
