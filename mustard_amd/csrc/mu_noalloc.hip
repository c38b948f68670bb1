// mu_noalloc.hip -- mu_dtrsm_noalloc: mu_dtrsm for callers that cannot
// allocate device memory.
//
// The panel solves keep the inverses of their diagonal blocks in LDS, so up to
// MU_NOALLOC_MAX_ORDER no unit of the lowered solve needs a workspace: this
// entry point runs the same lowering and the same kernels as mu_dtrsm (its
// result is bit-identical), and refuses what it could not run without one.
#include <hip/hip_runtime.h>

#include <string>

#include "../../include/mustard_hip.h"
#include "mu_capi.hpp"
#include "mu_dag.hpp"
#include "mu_runtime.hpp"

extern "C" int mu_dtrsm_noalloc(void *stream, char side, char uplo, char transa, char diag,
                                int m, int n, double alpha, const double *A, int lda, double *B,
                                int ldb)
{
    mu::OpRec op;
    int rc = mu::dtrsm_op(side, uplo, transa, diag, m, n, alpha, A, lda, B, ldb, op);
    if (rc != MU_OK)
        return rc;
    if (mu::stream_recording(stream))
        return mu::set_error(MU_ESTATE, "mu_dtrsm_noalloc: the stream is being recorded into a "
                                        "DAG (record with mu_dtrsm; the executable owns its "
                                        "workspace)");
    if (op.m > MU_NOALLOC_MAX_ORDER)
        return mu::set_error(MU_EINVAL, "mu_dtrsm_noalloc: a triangle of order " +
                                            std::to_string(op.m) + " is above the " +
                                            std::to_string(MU_NOALLOC_MAX_ORDER) +
                                            " this entry point accepts; use mu_dtrsm");
    mu::Dag d;
    d.begin_task({0, 0}, {});
    d.add_op(op);
    d.end_task();
    mu::Lowered low;
    std::string err;
    if (!mu::lower(d, mu::LowerOpts(), low, err))
        return mu::set_error(MU_EINVAL, err);
    if (mu::ws_total_doubles(low) != 0)
        return mu::set_error(MU_EINVAL, "mu_dtrsm_noalloc: a triangle of order " +
                                            std::to_string(op.m) +
                                            " needs a workspace (order <= 8192 does not); "
                                            "use mu_dtrsm");
    if (mu::run_units(low, (hipStream_t)stream, err) != 0)
        return mu::set_error(MU_EHIP, err);
    return MU_OK;
}
