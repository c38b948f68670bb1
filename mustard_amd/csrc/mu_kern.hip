// mu_kern.hip -- the specialised level kernels of the tiled mode (one launch
// runs every item of one graph node; block b runs items[b]) and the per-unit
// GEMM kernel of the stream mode.  Each needs only its own item kind's LDS
// and registers, so several workgroups share a CU: the bulk GEMM/SYRK blocks
// at four per CU, and the panel work of the next step beside them.
#include "mu_kernels.hpp"
#include "mu_ops.hpp"

namespace mu {

#define MU_GEMM_KERNEL __launch_bounds__(WG_THREADS) __attribute__((amdgpu_waves_per_eu(4, 4)))

__global__ MU_GEMM_KERNEL void k_unit_gemm(UnitDesc d)
{
    __shared__ __align__(16) double smem[LDS_GEMM];
    run_gemm_item(d, blockIdx.x, smem);
}

__global__ MU_GEMM_KERNEL void k_batch_gemm(NodeArgs node)
{
    __shared__ __align__(16) double smem[LDS_GEMM];
    int it;
    // a private copy of the descriptor lives in registers; a reference into
    // global memory would be re-read after every barrier of the item body
    const UnitDesc d = node_unit(node, it);
    run_gemm_item(d, it, smem);
}

// Diagonal GETRF/POTRF (and precision conversions), 4 waves held to 200
// registers per lane (the attribute counts half of the unified file): a CU
// running three GEMM workgroups (104 registers per wave) has room for it, so
// the diagonal factorization of the next step starts as soon as one bulk GEMM
// workgroup leaves a CU instead of waiting for the bulk update to drain.
__global__ __launch_bounds__(WG_THREADS) __attribute__((amdgpu_num_vgpr(100))) void
k_batch_small(NodeArgs node)
{
    __shared__ double smem[LDS_SMALL];
    int it;
    const UnitDesc d = node_unit(node, it);
    run_small_item(d, it, smem);
}

// Reduced-precision GEMM/SYRK units whose operands are k-contiguous in
// their storage precision (the trailing updates of an FP32 / BF16
// factorization reading the converted panels): long k-slices; 128 x 128
// blocks in the level-batched graph (72 KB of LDS, two workgroups per CU).
__global__ __launch_bounds__(WG_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2))) void
k_batch_gemm_low(NodeArgs node)
{
    __shared__ double smem[LDS_GEMM_LOWK128];
    int it;
    const UnitDesc d = node_unit(node, it);
    run_gemm_lowk_item(d, it, smem);
}

// Precision conversions (the panels' reduced-precision shadows, the FP32
// copies of the factors): 16 KB of LDS and few registers, so eight
// workgroups share a CU -- a conversion on the lookahead chain waits for no
// CU to drain, and the bulk ones stream at full occupancy.
__global__ __launch_bounds__(WG_THREADS) void k_batch_cvt(NodeArgs node)
{
    __shared__ double smem[4 * 16 * 65 / 2 + 4];
    int it;
    const UnitDesc d = node_unit(node, it);
    cvt_block(d, it, smem);
}

// GEMMs with at most 16 output columns (substitution steps of a solve).
__global__ __launch_bounds__(WG_THREADS) void k_batch_gemm_narrow(NodeArgs node)
{
    __shared__ double smem[LDS_NARROW];
    int it;
    const UnitDesc d = node_unit(node, it);
    run_gemm_narrow_item(d, it, smem);
}

// Panel solves of order <= SMALL_MAX (inside nested diagonal factorizations)
// and of order <= TRSM_REG_MAX, at most 200 registers per lane as
// k_batch_small, so they start beside three GEMM workgroups.
__global__ __launch_bounds__(WG_THREADS) __attribute__((amdgpu_num_vgpr(100))) void
k_batch_trsm_small(NodeArgs node)
{
    __shared__ __align__(16) double smem[LDS_TRSM_REG_SMALL];
    int it;
    const UnitDesc d = node_unit(node, it);
    run_trsm_reg_item<8>(d, it, smem);
}

__global__ __launch_bounds__(WG_THREADS) __attribute__((amdgpu_num_vgpr(100))) void
k_batch_trsm_256(NodeArgs node)
{
    __shared__ __align__(16) double smem[LDS_TRSM_REG];
    int it;
    const UnitDesc d = node_unit(node, it);
    run_trsm_reg_item<16>(d, it, smem);
}

// Panel solves with inverted diagonal blocks of order <= 512, and the TRINV
// items before them, on 4 waves and 64 KB of LDS (trsm_max above 256 only).
__global__ __launch_bounds__(WG_THREADS) void k_batch_trsm_512(NodeArgs node)
{
    __shared__ double smem[512 * 16];
    int it;
    const UnitDesc d = node_unit(node, it);
    if (d.op == OP_TRINV)
        run_trinv_item(d, it, smem);
    else
        run_trsm_inv_item<4, 512>(d, it, smem);
}

const void *level_kernel(int kind)
{
    switch (kind) {
    case LEVEL_GEMM: return reinterpret_cast<const void *>(k_batch_gemm);
    case LEVEL_SMALL: return reinterpret_cast<const void *>(k_batch_small);
    case LEVEL_TRSM_SMALL: return reinterpret_cast<const void *>(k_batch_trsm_small);
    case LEVEL_GEMM_NARROW: return reinterpret_cast<const void *>(k_batch_gemm_narrow);
    case LEVEL_GEMM_LOW: return reinterpret_cast<const void *>(k_batch_gemm_low);
    case LEVEL_CVT: return reinterpret_cast<const void *>(k_batch_cvt);
    case LEVEL_TRSM_256: return reinterpret_cast<const void *>(k_batch_trsm_256);
    case LEVEL_TRSM_512: return reinterpret_cast<const void *>(k_batch_trsm_512);
    default: return generic_kernel(kind);
    }
}

int level_threads(int kind)
{
    return kind == LEVEL_TRSM ? 64 * TRSM_KERNEL_WAVES : WG_THREADS;
}

int launch_unit(const UnitDesc &d, hipStream_t s)
{
    if ((d.op == OP_GEMM || d.op == OP_SYRK) && !(d.flags & F_NARROW)) {
        hipLaunchKernelGGL(k_unit_gemm, dim3(d.nitems), dim3(WG_THREADS), 0, s, d);
        return hipGetLastError() == hipSuccess ? 0 : -1;
    }
    return launch_unit_generic(d, s);
}

}  // namespace mu
