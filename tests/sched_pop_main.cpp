// Host driver for single steps of the persistent scheduler (mu_sched.hpp),
// built and run by tests/test_sched_pop.py: one worker, with lots, arrivals and
// the host's abort word that the case decides.  Prints one line per case.
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <vector>

#include "mu_sched.hpp"

using namespace mu;

static uint32_t lot_cnt = 0, lot_tries = 0;  // a lot wins from this count, or this try, on
static void (*on_pause)() = nullptr;
static SchedState st;
static uint32_t slots[NPRIO][256];

struct OneAtom {
    static bool lane0() { return true; }
    static uint32_t bcast(uint32_t v) { return v; }
    static uint32_t load(uint32_t *p) { return *p; }
    static SchedPeek peek(SchedState *s)
    {
        SchedPeek r;
        for (int p = 0; p < NPRIO; p++)
            r.cnt[p] = s->cnt[p];
        r.done = s->done;
        r.abort = s->abort;
        return r;
    }
    static bool lot(uint32_t cnt, uint32_t tries) { return cnt >= lot_cnt || tries >= lot_tries; }
    static uint32_t load_acquire(uint32_t *p) { return *p; }
    static uint32_t load_system(uint32_t *p) { return *p; }
    static void store(uint32_t *p, uint32_t v) { *p = v; }
    static uint32_t add(uint32_t *p, uint32_t v) { return (*p += v) - v; }
    static uint32_t add_release(uint32_t *p, uint32_t v) { return add(p, v); }
    static int32_t add_acq_rel(int32_t *p, int32_t v) { return (*p += v) - v; }
    static uint32_t cas(uint32_t *p, uint32_t e, uint32_t d)
    {
        const uint32_t o = *p;
        if (o == e)
            *p = d;
        return o;
    }
    static void fence_release() {}
    static uint64_t now()
    {
        static uint64_t t = 0;
        return ++t;
    }
    static void pause()
    {
        if (on_pause)
            on_pause();
    }
    static void producer_delay() {}
};

// `n` items on ring p: 100 p + 0, 1, ...
static void push(int p, int n)
{
    for (int i = 0; i < n; i++)
        slots[p][st.tail[p]++] = (uint32_t)(100 * p + i + 1);
    st.cnt[p] += n;
}

static int bad = 0;
static void report(const char *name, int got, int want)
{
    std::printf("%s: %d, expected %d %s\n", name, got, want, got == want ? "ok" : "FAILED");
    bad += got != want;
}

int main()
{
    ExecView ev;
    std::memset(&ev, 0, sizeof ev);
    for (int p = 0; p < NPRIO; p++) {
        ev.slots[p] = slots[p];
        ev.cap[p] = 256;
    }
    ev.st = &st;
    ev.nitems = 1000;
    ev.timeout_ticks = 100000;
    ev.poll_limit = 100000;
    auto fresh = [&]() {
        std::memset(&st, 0, sizeof st);
        std::memset(slots, 0, sizeof slots);
        on_pause = nullptr;
    };
    uint32_t calls = 0;

    // a worker that has just finished an item takes the urgent one, whatever
    // its luck, not the bulk behind it
    fresh();
    lot_cnt = 100, lot_tries = ~0u;
    push(0, 1);
    push(1, 100);
    report("urgent item, busy worker", sched_pop<OneAtom>(ev, calls), 0);
    report("bulk after it", sched_pop<OneAtom>(ev, calls), 100);

    // an idle worker that loses a lot for the urgent item draws again
    fresh();
    lot_cnt = 100, lot_tries = 3;
    on_pause = [] {
        if (st.tail[0] == 0) {
            push(0, 1);
            push(1, 100);
        }
    };
    report("urgent item, idle worker", sched_pop<OneAtom>(ev, calls), 0);

    // an idle worker that always loses leaves an item that others took meanwhile
    fresh();
    lot_cnt = 100, lot_tries = ~0u;
    on_pause = [] {
        static int polls = 0;
        if (++polls == 1) {
            push(0, 1);
        } else if (polls == 5) {
            st.cnt[0] = 0;
            st.head[0] = 1;
            push(2, 100);
        }
    };
    report("bulk once the urgent item is gone", sched_pop<OneAtom>(ev, calls), 200);
    return bad ? 1 : 0;
}
