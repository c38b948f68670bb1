// Host driver for the workspace of lowered triangular solves, built and run by
// tests/test_noalloc_lowering.py: with the default options no solve up to
// order 8192 needs one, which is what mu_dtrsm_noalloc relies on.
#include <cstdint>
#include <cstdio>
#include <string>

#include "mu_dag.hpp"

int main()
{
    const int orders[] = {1,   16,  17,  128, 129,  250,  256,  257,  300,  511,  512,  513, 1000,
                          1024, 1025, 2000, 2001, 3000, 4097, 5000, 7000, 8100, 8191, 8192};
    int bad = 0;
    for (int n : orders)
        for (int nrhs : {1, 16, 17, 1000})
            for (int flags : {0, (int)mu::F_UNIT, (int)(mu::F_T_TRANS | mu::F_Z_ROWS), (int)mu::F_REV}) {
                mu::OpRec t;
                t.op = mu::OP_TRSM;
                t.flags = flags;
                t.m = n;
                t.n = nrhs;
                t.a = reinterpret_cast<double *>(1ull << 40);
                t.lda = n;
                t.c = reinterpret_cast<double *>(1ull << 41);
                t.ldc = 10000;
                t.alpha = 1.0;
                mu::Dag d;
                d.begin_task({0, 0}, {});
                d.add_op(t);
                d.end_task();
                mu::Lowered low;
                std::string err;
                if (!mu::lower(d, mu::LowerOpts(), low, err) || low.units.empty() ||
                    !low.ws_doubles.empty()) {
                    std::printf("order %d nrhs %d flags %d: %s\n", n, nrhs, flags, err.c_str());
                    bad++;
                }
            }
    std::printf("%d bad\n", bad);
    return bad ? 1 : 0;
}
