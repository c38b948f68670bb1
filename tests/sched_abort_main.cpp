// Host driver for an abort by the host in the middle of a busy persistent run,
// built and run by tests/test_sched_abort.py: mu::emulate (mu_sched_host.cpp)
// over independent units, the abort word set while all workers have items.
#include <cstdint>
#include <cstdio>
#include <string>

#include "mu_dag.hpp"
#include "mu_sched_host.hpp"

int main()
{
    // 6000 tasks without dependencies: no worker ever waits for an item
    mu::Dag d;
    for (int i = 0; i < 6000; i++) {
        mu::OpRec p;
        p.op = mu::OP_POTRF;
        p.m = p.n = 64;
        p.c = reinterpret_cast<double *>((1ull << 40) + (size_t)i * 64 * 64 * 8);
        p.ldc = 64;
        d.begin_task({i, i}, {});
        d.add_op(p);
        d.end_task();
    }
    mu::EmuOpts eo;
    eo.workgroups = 16;
    eo.timeout_s = 60.0;
    eo.abort_after_items = 16;
    mu::EmuResult r;
    std::string err;
    if (!mu::emulate(d, mu::LowerOpts(), eo, r, err)) {
        std::printf("%s\n", err.c_str());
        return 2;
    }
    // A worker looks at the word on every 256th item, the 16 workers spread
    // evenly over these, and the first that sees it stops the others.  However
    // unevenly the threads run, that is before the sum of what each has left
    // (128 on average; two workers may have looked just before), and every
    // worker finishes at most the item it has and one more.
    const bool ok = r.err == 4 && r.duplicates == 0 && r.order_violations == 0 &&
                    r.executed <= 16 * 128 + 2 * 256 + 4 * 16;
    std::printf("items %u executed %llu err %u %s\n", r.nitems, (unsigned long long)r.executed,
                r.err, ok ? "ok" : "FAILED");
    return ok ? 0 : 1;
}
