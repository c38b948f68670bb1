// mu_ops.hpp -- gfx950 work-item bodies of the tile operations.
//
// One work item runs on one workgroup of 256 threads (4 wave64s).  The same
// bodies serve the per-unit grid kernels of the hipGraph mode and the
// persistent scheduler kernel.
//
// Arithmetic replaced (all column-major, leading dimension per operand):
//   GEMM  cublasGemmEx 64F  (mustard/lu_mustard.cu:511-522, cholesky_mustard.cu:376-387)
//   SYRK  cublasDsyrk LOWER (mustard/cholesky_mustard.cu:327-333)
//   TRSM  cublasDtrsm       (mustard/lu_mustard.cu:413-422, 459-468; cholesky_mustard.cu:281-290)
//   GETRF cusolverDnDgetrf, devIpiv = NULL (mustard/lu_mustard.cu:360-369)
//   POTRF cusolverDnDpotrf LOWER (mustard/cholesky_mustard.cu:238-246)
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "mu_types.h"

namespace mu {

typedef double v4d __attribute__((ext_vector_type(4)));
typedef double v2d __attribute__((ext_vector_type(2)));

// Operand pointers come from descriptors in memory, so the compiler cannot
// infer their address space; they always point to device global memory, and
// saying so turns flat accesses into global (vector memory) instructions.
#define MU_G __attribute__((address_space(1)))
#define MU_C __attribute__((address_space(4)))  // ... that no kernel writes meanwhile
template <class T>
__device__ __forceinline__ MU_G T *gp(T *p)
{
    return (MU_G T *)p;
}

// Workgroup barrier for LDS hand-offs only.  __syncthreads() is a
// workgroup-scope fence plus s_barrier, and the fence waits for every
// outstanding global load as well (vmcnt(0)), which would drain the
// prefetches the loops below keep in flight across their barriers.  No item
// body passes data between waves through global memory, so waiting for the
// LDS operations (lgkmcnt(0)) before the barrier is enough; the "memory"
// clobber keeps the compiler from moving memory accesses across it.
__device__ __forceinline__ void lds_barrier()
{
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// v_mfma_f64_16x16x4_f64.  Lane l supplies A[l%16][l/16] and B[l/16][l%16];
// it receives D[4*e + l/16][l%16] in element e (register e holds rows 4e..4e+3).
__device__ __forceinline__ v4d mfma_f64(double a, double b, v4d c)
{
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// GEMM / SYRK output block: C[i0:i0+64, j0:j0+64] = beta C + alpha op(A) op(B)
// ---------------------------------------------------------------------------
// Four waves in a 2 x 2 grid, each owning a 32 x 32 sub-block (2 x 2 MFMA
// tiles).  Two bodies: gemm_block_dma for every block of a unit with m, n >=
// 64 and k >= 16 (gemm_dma_ok), gemm_block for the smaller ones, whose edges
// it masks; both sum an element over k in the same order, so a result does
// not depend on which one ran.
//
// gemm_block: K runs in blocks of 8, double-buffered in LDS, through
// registers.
//
// LDS layouts.  An operand whose stored columns run along the output
// dimension ("i-contiguous": A, or B^T) is kept as S[k][i] with a pitch of
// PI doubles; one whose stored columns run along k ("k-contiguous": A^T, or B)
// is kept as S[i][k] with a pitch of PK doubles.
static_assert(GEMM_BM == 64 && GEMM_BN == 64 && GEMM_BK == 8, "GEMM loaders assume 64 x 64 x 8");
constexpr int PI = GEMM_BM + 16;
constexpr int PK = GEMM_BK + 1;
constexpr int LDS_I = GEMM_BK * PI;   // doubles per i-contiguous buffer
constexpr int LDS_K = GEMM_BM * PK;   // doubles per k-contiguous buffer

// The loaders below issue every load unconditionally, from an address clamped
// into the operand; the values that fall outside it are zeroed only when the
// registers are written to LDS.  With no branch around a load and no use of
// its result before the LDS store, the compiler's wait counting stays exact
// and a prefetch stays in flight until the half-step that stores it.  VEC
// (16-byte aligned operands, even leading dimensions and even m, n, k, set by
// the lowering) loads element pairs, which then never straddle an edge: 4000 x
// 32 x 1000 in 57 us against 62.

// i-contiguous operand: element (r, k) at p[r + k*ld], r < rows, k < kcols.
// Thread t covers rows 2(t%32), 2(t%32)+1 of column t/32.
template <bool VEC>
__device__ __forceinline__ void ld_icontig(double (&v)[2], const MU_G double *p, int ld, int rows,
                                           int kcols)
{
    const int t = threadIdx.x, r = (t & 31) * 2, c = t >> 5;
    const int cc = max(0, min(c, kcols - 1));
    if (VEC) {
        const int rr = max(0, min(r, rows - 2));
        const v2d x = *reinterpret_cast<const MU_G v2d *>(p + rr + (size_t)cc * ld);
        v[0] = x[0];
        v[1] = x[1];
    } else {
        v[0] = p[min(r, rows - 1) + (size_t)cc * ld];
        v[1] = p[min(r + 1, rows - 1) + (size_t)cc * ld];
    }
}

__device__ __forceinline__ void st_icontig(double *S, const double (&v)[2], int rows, int kcols)
{
    const int t = threadIdx.x, r = (t & 31) * 2, c = t >> 5;
    const bool cin = c < kcols;
    v2d x;
    x[0] = (cin && r < rows) ? v[0] : 0.0;
    x[1] = (cin && r + 1 < rows) ? v[1] : 0.0;
    *reinterpret_cast<v2d *>(S + c * PI + r) = x;
}

// k-contiguous operand: element (r, k) at p[k + r*ld].
// Thread t covers k = 2(t%4), 2(t%4)+1 of row t/4.
template <bool VEC>
__device__ __forceinline__ void ld_kcontig(double (&v)[2], const MU_G double *p, int ld, int rows,
                                           int kcols)
{
    const int t = threadIdx.x, k = (t & 3) * 2, r = t >> 2;
    const int rr = min(r, rows - 1);
    if (VEC) {
        const int kk = max(0, min(k, kcols - 2));
        const v2d x = *reinterpret_cast<const MU_G v2d *>(p + kk + (size_t)rr * ld);
        v[0] = x[0];
        v[1] = x[1];
    } else {
        v[0] = p[max(0, min(k, kcols - 1)) + (size_t)rr * ld];
        v[1] = p[max(0, min(k + 1, kcols - 1)) + (size_t)rr * ld];
    }
}

__device__ __forceinline__ void st_kcontig(double *S, const double (&v)[2], int rows, int kcols)
{
    const int t = threadIdx.x, k = (t & 3) * 2, r = t >> 2;
    const bool rin = r < rows;
    double *d = S + r * PK + k;
    d[0] = (rin && k < kcols) ? v[0] : 0.0;
    d[1] = (rin && k + 1 < kcols) ? v[1] : 0.0;
}

// op(A)(i, k) read from the LDS copy.
template <bool TA>
__device__ __forceinline__ double frag_a(const double *S, int i, int k)
{
    return TA ? S[i * PK + k] : S[k * PI + i];
}
// op(B)(k, j) read from the LDS copy.
template <bool TB>
__device__ __forceinline__ double frag_b(const double *S, int k, int j)
{
    return TB ? S[k * PI + j] : S[j * PK + k];
}

template <bool TA, bool TB, bool VEC>
__device__ __attribute__((always_inline)) inline void gemm_block(const UnitDesc &u, int bi, int bj, bool lower_only, double *smem)
{
    constexpr int BM = GEMM_BM, BN = GEMM_BN, BK = GEMM_BK;
    constexpr int SA = TA ? LDS_K : LDS_I;
    constexpr int SB = TB ? LDS_I : LDS_K;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int wm = wave & 1, wn = wave >> 1;  // 2 x 2 waves of 32 x 32
    const int i0 = bi * BM, j0 = bj * BN;
    const int rows = min(BM, u.m - i0), cols = min(BN, u.n - j0);
    const int K = u.k;
    // op(A)(i, k): TA ? a[k + i*lda] : a[i + k*lda];  op(B)(k, j): TB ? b[j + k*ldb] : b[k + j*ldb]
    const MU_G double *A = TA ? gp(u.a) + (size_t)i0 * u.lda : gp(u.a) + i0;
    const MU_G double *B = TB ? gp(u.b) + j0 : gp(u.b) + (size_t)j0 * u.ldb;
    double *As0 = smem, *As1 = smem + SA, *Bs0 = smem + 2 * SA, *Bs1 = smem + 2 * SA + SB;

    v4d acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
            acc[x][y] = v4d{0.0, 0.0, 0.0, 0.0};

    // Global loads run two k-blocks ahead of the MFMAs: block kb+2 is fetched
    // while block kb is computed and block kb+1 waits in registers for its
    // LDS buffer.
    double ra0[2], rb0[2], ra1[2], rb1[2];
    auto load = [&](double (&ra)[2], double (&rb)[2], int k0) {
        // a block past K is read (and zeroed) at k-offset 0, inside the operand
        const int kc = K - k0, ks = kc > 0 ? k0 : 0;
        if (TA)
            ld_kcontig<VEC>(ra, A + ks, u.lda, rows, kc);
        else
            ld_icontig<VEC>(ra, A + (size_t)ks * u.lda, u.lda, rows, kc);
        if (TB)
            ld_icontig<VEC>(rb, B + (size_t)ks * u.ldb, u.ldb, cols, kc);
        else
            ld_kcontig<VEC>(rb, B + ks, u.ldb, cols, kc);
    };
    // store the block loaded for k-offset k0 (zeroing what lies outside)
    auto store = [&](const double (&ra)[2], const double (&rb)[2], double *As, double *Bs,
                     int k0) {
        const int kc = K - k0;
        if (TA)
            st_kcontig(As, ra, rows, kc);
        else
            st_icontig(As, ra, rows, kc);
        if (TB)
            st_icontig(Bs, rb, cols, kc);
        else
            st_kcontig(Bs, rb, cols, kc);
    };
    const int li = lane & 15, lk = lane >> 4;
    auto compute = [&](const double *As, const double *Bs) {
#pragma unroll
        for (int kk = 0; kk < BK; kk += 4) {
            double fa[2], fb[2];
#pragma unroll
            for (int x = 0; x < 2; x++)
                fa[x] = frag_a<TA>(As, wm * 32 + x * 16 + li, kk + lk);
#pragma unroll
            for (int y = 0; y < 2; y++)
                fb[y] = frag_b<TB>(Bs, kk + lk, wn * 32 + y * 16 + li);
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++)
                    acc[x][y] = mfma_f64(fa[x], fb[y], acc[x][y]);
        }
    };

    // k-blocks in pairs, one per LDS buffer; with an odd count the last
    // block is left in buffer 0 by the last pair (or the prologue) and runs
    // alone.  Loads past the last block read clamped addresses, load zeros
    // and are never used.
    const int nkb = (K + BK - 1) / BK;
    if (K <= 0)
        goto epilogue;  // C = beta C: the operands are not read at all
    load(ra0, rb0, 0);
    store(ra0, rb0, As0, Bs0, 0);
    load(ra1, rb1, BK);
    lds_barrier();
    for (int kb = 0; kb + 1 < nkb; kb += 2) {
        load(ra0, rb0, (kb + 2) * BK);
        compute(As0, Bs0);
        store(ra1, rb1, As1, Bs1, (kb + 1) * BK);
        lds_barrier();
        load(ra1, rb1, (kb + 3) * BK);
        compute(As1, Bs1);
        store(ra0, rb0, As0, Bs0, (kb + 2) * BK);
        lds_barrier();
    }
    if (nkb & 1)
        compute(As0, Bs0);

epilogue:
    // Epilogue: all 16 C values of a lane are loaded before any is combined
    // and stored, so their latencies overlap.
    const double alpha = u.alpha, beta = u.beta;
    double cv[2][2][4];
    bool ok[2][2][4];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = wm * 32 + x * 16 + 4 * e + lk;
                const int c = wn * 32 + y * 16 + li;
                ok[x][y][e] = r < rows && c < cols && (!lower_only || i0 + r >= j0 + c);
                cv[x][y][e] = (ok[x][y][e] && beta != 0.0)
                                  ? gp(u.c)[(i0 + r) + (size_t)(j0 + c) * u.ldc]
                                  : 0.0;
            }
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = wm * 32 + x * 16 + 4 * e + lk;
                const int c = wn * 32 + y * 16 + li;
                if (ok[x][y][e])
                    gp(u.c)[(i0 + r) + (size_t)(j0 + c) * u.ldc] =
                        beta * cv[x][y][e] + alpha * acc[x][y][e];
            }
}

// ---------------------------------------------------------------------------
// GEMM / SYRK output block, operands copied straight into LDS.
//
// What bounds it: the FP64 matrix pipe, and on gfx950 the vector ALU shares
// it -- every VALU instruction of the k-loop takes about 4 cycles from the
// MFMAs (a loop of MFMAs and nothing else: adding 8 v_add per MFMA takes 30 %
// more time, with four waves per SIMD to overlap them).  So the loop below has
// no masks, no address arithmetic beyond two pointer increments and no
// staging registers: a k-slice of 16 is copied by four 16-byte-per-lane
// global_load_lds per wave, the fragments are read at constant offsets, and
// 16 MFMAs follow; the next slice's copy is in flight meanwhile (two
// buffers, 32 KB, so up to five workgroups share a CU).  Stand-alone, merged
// LU update 22000 x 22000 x 1000, lda 24000: 70.9 TFLOP/s, 90 % of the FP64
// MFMA peak, against 58.6 for the masked loop through registers
// (gemm_block); 128 x 64 and 128 x 128 blocks in the same form 67.3 and 66.3
// (fewer waves to cover the barriers).
//
// No edges: a block that would pass the last row or column is moved back to
// end there (needs m, n >= 64) and stores only the part no other block
// owns, so every load is inside the operand.  The last k % 16 columns go
// through registers with zeroed padding.  global_load_lds needs only 4-byte
// alignment, so odd leading dimensions and offsets take this path too.
//
// LDS.  An operand contiguous along the output dimension keeps rows of 64
// (S[k][i], 512 bytes): a lane reads rows i = 2 li, 2 li + 1 of a k with one
// 16-byte load, which feed its two MFMA tiles, so tile x's index li stands
// for i = 2 li + x.  An operand contiguous along k keeps 16 k per output
// index (128 bytes) in 16-byte chunks, chunk c of output o at c ^ ((o / 2) %
// 8), which makes the 16 outputs of a fragment hit 64 different banks; the
// copy applies the permutation by choosing which chunk each lane fetches.
// Operands enter the MFMA swapped (D = op(B)^T op(A)^T), so a lane holds
// consecutive rows of C: 256-byte runs instead of 32-byte ones.
// ---------------------------------------------------------------------------
#define MU_LDS __attribute__((address_space(3)))
typedef double v2du __attribute__((ext_vector_type(2), aligned(8)));  // C pairs, any alignment
constexpr int DMA_BK = 16;
constexpr int DMA_OP = GEMM_BM * DMA_BK;  // doubles per operand buffer
constexpr int LDS_GEMM_DMA = 4 * DMA_OP;  // 2 operands x 2 buffers (32 KB)

// Units every block of which gemm_block_dma can run (the per-lane byte
// offsets of a 64-row slice are 32-bit).
__device__ __forceinline__ bool gemm_dma_ok(const UnitDesc &u)
{
    return u.m >= GEMM_BM && u.n >= GEMM_BN && u.k >= DMA_BK && u.lda < (1 << 22) &&
           u.ldb < (1 << 22);
}

template <bool TA, bool TB>
__device__ __attribute__((always_inline)) inline void gemm_block_dma(const UnitDesc &u, int bi,
                                                                     int bj, bool lower_only,
                                                                     double *smem)
{
    constexpr int BM = GEMM_BM, BK = DMA_BK;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave & 1, wn = wave >> 1;  // 2 x 2 waves of 32 x 32
    // block origin, moved back to stay inside; rows < ri and columns < rj of
    // the moved block belong to its neighbours
    const int i0 = min(bi * BM, u.m - BM), j0 = min(bj * BM, u.n - BM);
    const int ri = bi * BM - i0, rj = bj * BM - j0;
    const int K = u.k, nk = K / BK;
    const size_t lda = u.lda, ldb = u.ldb;
    const MU_G char *ap = (const MU_G char *)(gp(u.a) + (TA ? (size_t)i0 * lda : (size_t)i0));
    const MU_G char *bp = (const MU_G char *)(gp(u.b) + (TB ? (size_t)j0 : (size_t)j0 * ldb));
    const size_t da = 8 * (TA ? (size_t)BK : BK * lda), db = 8 * (TB ? BK * ldb : (size_t)BK);

    // byte offset of the 16 bytes this lane copies in its wave's copy q (two
    // per operand): LDS slot s, in order
    auto slot_off = [&](int q, bool kcontig, size_t ld) -> unsigned {
        const int s = (wave * 2 + q) * 64 + lane;
        if (kcontig) {
            const int o = s >> 3, c = (s & 7) ^ ((o >> 1) & 7);
            return 8u * ((unsigned)o * (unsigned)ld + 2u * c);
        }
        return 8u * ((unsigned)(s >> 5) * (unsigned)ld + 2u * (s & 31));
    };
    const unsigned oa0 = slot_off(0, TA, lda), oa1 = slot_off(1, TA, lda);
    const unsigned ob0 = slot_off(0, !TB, ldb), ob1 = slot_off(1, !TB, ldb);
    auto copy16 = [&](const MU_G char *p, double *l) {
        __builtin_amdgcn_global_load_lds((const MU_G unsigned *)p, (MU_LDS unsigned *)l, 16, 0, 0);
    };
    auto load = [&](int buf) {
        double *as = smem + buf * 2 * DMA_OP + wave * 256, *bs = as + DMA_OP;
        copy16(ap + oa0, as);
        copy16(ap + oa1, as + 128);
        copy16(bp + ob0, bs);
        copy16(bp + ob1, bs + 128);
        ap += da;
        bp += db;
    };

    v4d acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
            acc[x][y] = v4d{0.0, 0.0, 0.0, 0.0};
    // LDS element offset of this lane's fragment of k-step 4 s + lk in an
    // operand buffer, for a wave whose 32 outputs start at o0
    auto frag_off = [&](int s, int o0, bool kcontig) -> int {
        const int o = o0 + li;
        return kcontig ? o * BK + (((2 * s + (lk >> 1)) ^ ((o >> 1) & 7)) << 1) + (lk & 1)
                       : (4 * s + lk) * BM + o0 + 2 * li;
    };
    int la[4], lb[4];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        la[s] = frag_off(s, wm * 32, TA);
        lb[s] = frag_off(s, wn * 32, !TB);
    }
    auto compute = [&](int buf) {
        const double *as = smem + buf * 2 * DMA_OP, *bs = as + DMA_OP;
#pragma unroll
        for (int s = 0; s < 4; s++) {
            v2d fa, fb;
            if (TA)
                fa = v2d{as[la[s]], as[la[s] + 16 * BK]};
            else
                fa = *reinterpret_cast<const v2d *>(as + la[s]);
            if (TB)
                fb = *reinterpret_cast<const v2d *>(bs + lb[s]);
            else
                fb = v2d{bs[lb[s]], bs[lb[s] + 16 * BK]};
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++)
                    acc[x][y] = mfma_f64(fb[y], fa[x], acc[x][y]);
        }
    };
    // this wave's copies have landed and every wave has read the other buffer
    auto sync = [] { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

    load(0);
    int kb = 0;
    for (; kb + 2 < nk; kb += 2) {
        sync();
        load(1);
        compute(0);
        sync();
        load(0);
        compute(1);
    }
    sync();
    if (kb + 1 < nk) {
        load(1);
        compute(0);
        sync();
        compute(1);
    } else {
        compute(0);
    }
    if (const int kt = K - nk * BK) {
        // the last kt columns into the buffer the last compute left alone
        double *as = smem + (nk & 1) * 2 * DMA_OP, *bs = as + DMA_OP;
        auto tail = [&](double *D, const MU_G char *p, bool kcontig, size_t ld) {
            const MU_G double *g = (const MU_G double *)p;
#pragma unroll
            for (int q = 0; q < DMA_OP / WG_THREADS; q++) {
                const int s = tid + WG_THREADS * q;
                const int o = kcontig ? s >> 4 : s & 63, k = kcontig ? s & 15 : s >> 6;
                const size_t kc = min(k, kt - 1);
                const double v = g[kcontig ? kc + o * ld : o + kc * ld];
                D[kcontig ? o * BK + (((k >> 1) ^ ((o >> 1) & 7)) << 1) + (k & 1) : s] =
                    k < kt ? v : 0.0;
            }
        };
        tail(as, ap, TA, lda);
        tail(bs, bp, !TB, ldb);
        sync();
        if (nk & 1)
            compute(1);
        else
            compute(0);
    }

    // acc[x][y][e]: row r(x) of the block, column c(y, e)
    const double alpha = u.alpha, beta = u.beta;
    const size_t ldc = u.ldc;
    MU_G double *cb = gp(u.c) + i0 + (size_t)j0 * ldc;
    const int r0 = wm * 32 + (TA ? li : 2 * li), dr = TA ? 16 : 1;
    auto col = [&](int y, int e) {
        return wn * 32 + (TB ? 2 * (4 * e + lk) + y : 16 * y + 4 * e + lk);
    };
    if (!TA && ri == 0 && rj == 0 && !lower_only) {
        v2d cv[2][4];
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                cv[y][e] = beta != 0.0 ? *(const MU_G v2du *)(cb + r0 + col(y, e) * ldc)
                                       : v2d{0.0, 0.0};
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                *(MU_G v2du *)(cb + r0 + col(y, e) * ldc) =
                    v2d{beta * cv[y][e][0] + alpha * acc[0][y][e],
                        beta * cv[y][e][1] + alpha * acc[1][y][e]};
        return;
    }
#pragma unroll
    for (int x = 0; x < 2; x++) {
        const int r = r0 + x * dr;
        double cv[2][4];
        bool ok[2][4];
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int c = col(y, e);
                ok[y][e] = r >= ri && c >= rj && (!lower_only || i0 + r >= j0 + c);
                cv[y][e] = (ok[y][e] && beta != 0.0) ? cb[r + c * ldc] : 0.0;
            }
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (ok[y][e])
                    cb[r + col(y, e) * ldc] = beta * cv[y][e] + alpha * acc[x][y][e];
    }
}

// ---------------------------------------------------------------------------
// Reduced-precision GEMM / SYRK block (units flagged F_LOW_F32 or F_LOW_BF16):
// the FP64 operands are rounded to FP32 (or BF16, round-to-nearest-even) as
// they are staged into LDS, the products run on FP32-accumulating MFMA
// (v_mfma_f32_16x16x4f32 / v_mfma_f32_16x16x16bf16_1k), and the result is
// applied to the FP64 C: C = beta C + alpha (double) acc.  Same 64 x 64 block
// and 2 x 2 waves as the FP64 kernel; K runs in blocks of 16; both operands
// are kept k-contiguous in LDS (S[row][k]) so a bf16 lane reads its four k
// values with one 8-byte load.
// ---------------------------------------------------------------------------
typedef float v4f __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));

// Row of element e of a lane's FP32 16 x 16 MFMA result (lane group lk).
__device__ __forceinline__ int f32_row(int e, int lk) { return 4 * lk + e; }

__device__ __forceinline__ unsigned short to_bf16(double x)
{
    // round to FP32, then to BF16 by round-to-nearest-even on the dropped bits
    unsigned u = __float_as_uint((float)x);
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

template <int P>
struct LowPrec;
typedef float v2f __attribute__((ext_vector_type(2)));
typedef unsigned short v2us __attribute__((ext_vector_type(2)));
template <>
struct LowPrec<1> {
    using T = float;
    using T2 = v2f;
    static constexpr int PK = 17;
    static __device__ __forceinline__ float cv(double x) { return (float)x; }
    static __device__ __forceinline__ float cv(float x) { return x; }
};
template <>
struct LowPrec<2> {
    using T = unsigned short;
    using T2 = v2us;
    static constexpr int PK = 20;
    static __device__ __forceinline__ unsigned short cv(double x) { return to_bf16(x); }
    static __device__ __forceinline__ unsigned short cv(unsigned short x) { return x; }
};

template <bool TA, bool TB, bool VEC, int P, bool SRC>
__device__ __attribute__((always_inline)) inline void gemm_block_low(const UnitDesc &u, int bi, int bj,
                                                                     bool lower_only, double *smem)
{
    using LP = LowPrec<P>;
    using T = typename LP::T;
    // operand storage: FP64, or (SRC) already rounded to T by an OP_CVT unit
    using S = typename std::conditional<SRC, T, double>::type;
    using S2 = typename std::conditional<SRC, typename LP::T2, v2d>::type;
    constexpr int BM = GEMM_BM, BK = 16, PKL = LP::PK, SBUF = BM * PKL;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1;
    const int li = lane & 15, lk = lane >> 4;
    const int i0 = bi * BM, j0 = bj * GEMM_BN;
    const int rows = min(BM, u.m - i0), cols = min(GEMM_BN, u.n - j0);
    const int K = u.k;
    const MU_G S *A = TA ? (const MU_G S *)u.a + (size_t)i0 * u.lda : (const MU_G S *)u.a + i0;
    const MU_G S *B = TB ? (const MU_G S *)u.b + j0 : (const MU_G S *)u.b + (size_t)j0 * u.ldb;
    T *SL = reinterpret_cast<T *>(smem);
    T *As[2] = {SL, SL + 2 * SBUF};
    T *Bs[2] = {SL + SBUF, SL + 3 * SBUF};

    // One operand block (64 rows x 16 k) per thread: two element pairs.
    // i-contiguous storage (element (r,k) at p[r + k*ld]): pair = rows r, r+1.
    // k-contiguous storage (element (r,k) at p[k + r*ld]): pair = k, k+1.
    auto ld_op = [&](S (&v)[4], const MU_G S *p, int ld, int nrow, int kc, bool icontig) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int idx = tid + WG_THREADS * q;
            if (icontig) {
                const int r = (idx & 31) * 2, c = idx >> 5;
                const int cc = max(0, min(c, kc - 1));
                if (VEC) {
                    const S2 x = *reinterpret_cast<const MU_G S2 *>(p + max(0, min(r, nrow - 2)) +
                                                                   (size_t)cc * ld);
                    v[2 * q] = x[0];
                    v[2 * q + 1] = x[1];
                } else {
                    v[2 * q] = p[min(r, nrow - 1) + (size_t)cc * ld];
                    v[2 * q + 1] = p[min(r + 1, nrow - 1) + (size_t)cc * ld];
                }
            } else {
                const int k = (idx & 7) * 2, r = idx >> 3;
                const int rr = min(r, nrow - 1);
                if (VEC) {
                    const S2 x = *reinterpret_cast<const MU_G S2 *>(p + max(0, min(k, kc - 2)) +
                                                                   (size_t)rr * ld);
                    v[2 * q] = x[0];
                    v[2 * q + 1] = x[1];
                } else {
                    v[2 * q] = p[max(0, min(k, kc - 1)) + (size_t)rr * ld];
                    v[2 * q + 1] = p[max(0, min(k + 1, kc - 1)) + (size_t)rr * ld];
                }
            }
        }
    };
    const T zero = LP::cv(0.0);
    auto st_op = [&](T *D, const S (&v)[4], int nrow, int kc, bool icontig) {
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int idx = tid + WG_THREADS * q;
            if (icontig) {
                const int r = (idx & 31) * 2, c = idx >> 5;
                const bool cin = c < kc;
                D[r * PKL + c] = (cin && r < nrow) ? LP::cv(v[2 * q]) : zero;
                D[(r + 1) * PKL + c] = (cin && r + 1 < nrow) ? LP::cv(v[2 * q + 1]) : zero;
            } else {
                const int k = (idx & 7) * 2, r = idx >> 3;
                const bool rin = r < nrow;
                D[r * PKL + k] = (rin && k < kc) ? LP::cv(v[2 * q]) : zero;
                D[r * PKL + k + 1] = (rin && k + 1 < kc) ? LP::cv(v[2 * q + 1]) : zero;
            }
        }
    };
    S ra0[4], rb0[4], ra1[4], rb1[4];
    auto load = [&](S (&ra)[4], S (&rb)[4], int k0) {
        const int kc = K - k0, ks = kc > 0 ? k0 : 0;
        if (TA)
            ld_op(ra, A + ks, u.lda, rows, kc, false);
        else
            ld_op(ra, A + (size_t)ks * u.lda, u.lda, rows, kc, true);
        if (TB)
            ld_op(rb, B + (size_t)ks * u.ldb, u.ldb, cols, kc, true);
        else
            ld_op(rb, B + ks, u.ldb, cols, kc, false);
    };
    auto store = [&](const S (&ra)[4], const S (&rb)[4], int buf, int k0) {
        const int kc = K - k0;
        st_op(As[buf], ra, rows, kc, !TA);
        st_op(Bs[buf], rb, cols, kc, TB);
    };
    v4f acc[2][2];
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
            acc[x][y] = v4f{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](int buf) {
        const T *Sa = As[buf], *Sb = Bs[buf];
        if (P == 1) {
#pragma unroll
            for (int kk = 0; kk < BK; kk += 4) {
                float fa[2], fb[2];
#pragma unroll
                for (int x = 0; x < 2; x++)
                    fa[x] = Sa[(wm * 32 + x * 16 + li) * PKL + kk + lk];
#pragma unroll
                for (int y = 0; y < 2; y++)
                    fb[y] = Sb[(wn * 32 + y * 16 + li) * PKL + kk + lk];
#pragma unroll
                for (int x = 0; x < 2; x++)
#pragma unroll
                    for (int y = 0; y < 2; y++)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[x], fb[y], acc[x][y], 0,
                                                                         0, 0);
            }
        } else {
            v4s fa[2], fb[2];
#pragma unroll
            for (int x = 0; x < 2; x++)
                fa[x] = *reinterpret_cast<const v4s *>(Sa + (wm * 32 + x * 16 + li) * PKL + 4 * lk);
#pragma unroll
            for (int y = 0; y < 2; y++)
                fb[y] = *reinterpret_cast<const v4s *>(Sb + (wn * 32 + y * 16 + li) * PKL + 4 * lk);
#pragma unroll
            for (int x = 0; x < 2; x++)
#pragma unroll
                for (int y = 0; y < 2; y++)
                    acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(fa[x], fb[y], acc[x][y], 0,
                                                                          0, 0);
        }
    };

    const int nk = ((K + BK - 1) / BK + 1) & ~1;
    if (K > 0) {
        load(ra0, rb0, 0);
        store(ra0, rb0, 0, 0);
        load(ra1, rb1, BK);
        lds_barrier();
        for (int kb = 0; kb < nk; kb += 2) {
            load(ra0, rb0, (kb + 2) * BK);
            compute(0);
            store(ra1, rb1, 1, (kb + 1) * BK);
            lds_barrier();
            load(ra1, rb1, (kb + 3) * BK);
            compute(1);
            store(ra0, rb0, 0, (kb + 2) * BK);
            lds_barrier();
        }
    }
    const double alpha = u.alpha, beta = u.beta;
#pragma unroll
    for (int x = 0; x < 2; x++)
#pragma unroll
        for (int y = 0; y < 2; y++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = wm * 32 + x * 16 + f32_row(e, lk);
                const int c = wn * 32 + y * 16 + li;
                if (r < rows && c < cols && (!lower_only || i0 + r >= j0 + c)) {
                    MU_G double *cp = gp(u.c) + (i0 + r) + (size_t)(j0 + c) * u.ldc;
                    const double old = beta != 0.0 ? *cp : 0.0;
                    *cp = beta * old + alpha * (double)acc[x][y][e];
                }
            }
}

// ---------------------------------------------------------------------------
// Reduced-precision GEMM / SYRK block with both operands k-contiguous in
// their storage precision (F_KVEC: op(A) = A^T of a panel the conversion
// stored transposed, op(B) = B), C = beta C + alpha op(A) op(B) on a
// 128 x 128 output block (units flagged F_BLK128, made for the level-batched
// graph).  Each of the 4 waves owns a 64 x 64 quarter, 4 x 4 MFMA tiles, so
// every LDS fragment feeds four MFMAs.  BF16 runs on gfx950's
// v_mfma_f32_16x16x32_bf16 (8 k-values per lane, lane group lk holding
// k = 8 lk .. 8 lk + 7 of A's row and B's column), FP32 on
// v_mfma_f32_16x16x4f32; FP32 accumulation, the result applied to the FP64
// C.  The k-slices are long (BF16: 64, FP32: 32) and every operand row
// reaches LDS as whole 16-byte vectors (LDS rows padded by 16 bytes),
// global -> registers -> LDS one slice ahead of the MFMAs.
// ---------------------------------------------------------------------------
template <int P>
__device__ __attribute__((always_inline)) inline void gemm_block_lowk128(const UnitDesc &u,
                                                                         int bi, int bj,
                                                                         bool lower_only,
                                                                         double *smem)
{
    using T = typename LowPrec<P>::T;
    typedef unsigned int v4u __attribute__((ext_vector_type(4)));
    typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
    constexpr int BM = 128;
    constexpr int ES = sizeof(T), VE = 16 / ES;        // elements per 16 bytes
    constexpr int BK = P == 2 ? 64 : 32, PK = BK + VE;  // k-slice, LDS row pitch (elements)
    constexpr int CPR = BK / VE, NL = BM * BK / VE / WG_THREADS;  // chunks per row, loads/thread
    static_assert(NL * WG_THREADS * VE == BM * BK, "loader split");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave & 1, wn = wave >> 1, li = lane & 15, lk = lane >> 4;
    const int i0 = bi * BM, j0 = bj * BM;
    const int rows = min(BM, u.m - i0), cols = min(BM, u.n - j0);
    const int K = u.k;
    const MU_G T *A = (const MU_G T *)u.a + (size_t)i0 * u.lda;  // op(A) row r at A + r lda
    const MU_G T *B = (const MU_G T *)u.b + (size_t)j0 * u.ldb;  // op(B) column c at B + c ldb
    T *SL = reinterpret_cast<T *>(smem);
    T *As[2] = {SL, SL + 2 * BM * PK};
    T *Bs[2] = {SL + BM * PK, SL + 3 * BM * PK};

    v4u ra0[NL], rb0[NL], ra1[NL], rb1[NL];
    // chunk ch of row r of the k-slice at k0; a chunk past K reads the
    // slice's last full chunk (or the row's first) and is zeroed when stored
    auto load = [&](v4u (&xa)[NL], v4u (&xb)[NL], int k0) {
        const int kc = K - k0, ks = kc > 0 ? k0 : 0;
#pragma unroll
        for (int q = 0; q < NL; q++) {
            const int idx = tid + WG_THREADS * q, r = idx / CPR, ch = idx % CPR;
            const int kk = min(ch * VE, max(kc - VE, 0));
            xa[q] = *(const MU_G v4u *)(A + (size_t)min(r, rows - 1) * u.lda + ks + kk);
            xb[q] = *(const MU_G v4u *)(B + (size_t)min(r, cols - 1) * u.ldb + ks + kk);
        }
    };
    auto store = [&](const v4u (&xa)[NL], const v4u (&xb)[NL], int buf, int k0) {
        const int kc = K - k0;
        const v4u zero = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int q = 0; q < NL; q++) {
            const int idx = tid + WG_THREADS * q, r = idx / CPR, ch = idx % CPR;
            const bool kin = ch * VE < kc;
            *(v4u *)(As[buf] + r * PK + ch * VE) = (kin && r < rows) ? xa[q] : zero;
            *(v4u *)(Bs[buf] + r * PK + ch * VE) = (kin && r < cols) ? xb[q] : zero;
        }
    };
    v4f acc[4][4];
#pragma unroll
    for (int x = 0; x < 4; x++)
#pragma unroll
        for (int y = 0; y < 4; y++)
            acc[x][y] = v4f{0.f, 0.f, 0.f, 0.f};
    auto compute = [&](int buf) {
        const T *Sa = As[buf] + (wm * 64 + li) * PK, *Sb = Bs[buf] + (wn * 64 + li) * PK;
        if constexpr (P == 2) {
#pragma unroll
            for (int kk = 0; kk < BK; kk += 32) {
                v8bf fa[4], fb[4];
#pragma unroll
                for (int x = 0; x < 4; x++)
                    fa[x] = __builtin_bit_cast(
                        v8bf, *reinterpret_cast<const v4u *>(Sa + x * 16 * PK + kk + 8 * lk));
#pragma unroll
                for (int y = 0; y < 4; y++)
                    fb[y] = __builtin_bit_cast(
                        v8bf, *reinterpret_cast<const v4u *>(Sb + y * 16 * PK + kk + 8 * lk));
#pragma unroll
                for (int x = 0; x < 4; x++)
#pragma unroll
                    for (int y = 0; y < 4; y++)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fa[x], fb[y], acc[x][y],
                                                                            0, 0, 0);
            }
        } else {
#pragma unroll
            for (int kk = 0; kk < BK; kk += 4) {
                float fa[4], fb[4];
#pragma unroll
                for (int x = 0; x < 4; x++)
                    fa[x] = Sa[x * 16 * PK + kk + lk];
#pragma unroll
                for (int y = 0; y < 4; y++)
                    fb[y] = Sb[y * 16 * PK + kk + lk];
#pragma unroll
                for (int x = 0; x < 4; x++)
#pragma unroll
                    for (int y = 0; y < 4; y++)
                        acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[x], fb[y], acc[x][y], 0, 0, 0);
            }
        }
    };
    const int nkb = (K + BK - 1) / BK;
    if (K > 0) {
        load(ra0, rb0, 0);
        store(ra0, rb0, 0, 0);
        load(ra1, rb1, BK);
        lds_barrier();
        for (int kb = 0; kb + 1 < nkb; kb += 2) {
            load(ra0, rb0, (kb + 2) * BK);
            compute(0);
            store(ra1, rb1, 1, (kb + 1) * BK);
            lds_barrier();
            load(ra1, rb1, (kb + 3) * BK);
            compute(1);
            store(ra0, rb0, 0, (kb + 2) * BK);
            lds_barrier();
        }
        if (nkb & 1)
            compute(0);
    }
    const double alpha = u.alpha, beta = u.beta;
#pragma unroll
    for (int x = 0; x < 4; x++)
#pragma unroll
        for (int y = 0; y < 4; y++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = wm * 64 + x * 16 + f32_row(e, lk);
                const int c = wn * 64 + y * 16 + li;
                if (r < rows && c < cols && (!lower_only || i0 + r >= j0 + c)) {
                    MU_G double *cp = gp(u.c) + (i0 + r) + (size_t)(j0 + c) * u.ldc;
                    const double old = beta != 0.0 ? *cp : 0.0;
                    *cp = beta * old + alpha * (double)acc[x][y][e];
                }
            }
}
// LDS of gemm_block_lowk128: 2 buffers x (128 + 128) rows x (BK + VE) elements = 72 KB
constexpr int LDS_GEMM_LOWK128 = 2 * 256 * (64 + 8) * 2 / 8;

// ---------------------------------------------------------------------------
// Inverted diagonal blocks.  For a triangle T of order n > TRSM_REG_MAX (read in
// the canonical lower form the panel solve uses: flags TT, UNIT, REV as in
// trsm_panel_inv), item `it` inverts diagonal blocks 16*it .. 16*it+15 of 16 x 16
// and stores inv(T_jj) row-major at c + 256 j.  Rows and columns of the last
// block past n are the identity.  Thread t: block t/16, column t%16, by
// forward substitution against the unit vector (divisions, as LAPACK's
// dtrti2 does; this runs once per triangle).
// ---------------------------------------------------------------------------
template <bool TT, bool UNIT, bool REV>
__device__ __attribute__((always_inline)) inline void trinv_blocks(const UnitDesc &u, int it,
                                                                   double *smem)
{
    const int n = u.m, tid = threadIdx.x, lb = tid >> 4, c = tid & 15;
    const int j = it * TRINV_BLOCKS + lb, j0 = 16 * j;
    const MU_G double *t = gp(u.a);
    const size_t ldt = u.lda;
    const unsigned ldt32 = (unsigned)ldt;
    auto tv = [&](int r, int q) -> double {
        if (REV) {
            r = n - 1 - r;
            q = n - 1 - q;
        }
        const unsigned off = TT ? (unsigned)q + __umul24((unsigned)r, ldt32)
                                : (unsigned)r + __umul24((unsigned)q, ldt32);
        return t[off];
    };
    double *D = smem + lb * 16 * 17;
    const bool live = j0 < n;
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const bool in = live && j0 + r < n && j0 + c < n;
        double v;
        if (r == c)
            v = (UNIT || !in) ? 1.0 : tv(j0 + r, j0 + c);
        else
            v = (r > c && in) ? tv(j0 + r, j0 + c) : 0.0;
        D[r * 17 + c] = v;
    }
    lds_barrier();
    double x[16];
#pragma unroll
    for (int r = 0; r < 16; r++) {
        double s = r == c ? 1.0 : 0.0;
#pragma unroll
        for (int q = 0; q < r; q++)
            s -= D[r * 17 + q] * x[q];
        x[r] = UNIT ? s : s / D[r * 17 + r];
    }
    if (live) {
        MU_G double *w = gp(u.c) + (size_t)j * 256;
#pragma unroll
        for (int r = 0; r < 16; r++)
            w[r * 16 + c] = x[r];
    }
}

// ---------------------------------------------------------------------------
// Panel triangular solve in LDS with inverted diagonal blocks (triangles of
// order n > TRSM_REG_MAX, made only where mu_exec_opts_t.trsm_max asks for
// them; the TRINV unit before it left inv(T_jj) at u.b).  Same problem and
// flags as trsm_panel_reg, panels of 16 right-hand sides.  Step jb: every wave
// forms the solved block X_jb = inv(T_jj) Y_jb with four MFMAs -- the result's
// register layout is exactly the B operand of the update MFMAs, so it never
// goes back through LDS -- wave 0 stores it to Z, and each wave updates its row blocks
// below, Y[rb] -= T[rb, jb] X_jb.  One barrier per step.  The next step's
// inverse block and triangle fragments are loaded during the current step
// (the latter row block by row block, right after that block's MFMAs).
// ---------------------------------------------------------------------------
template <bool TT, bool ZR, bool UNIT, bool REV, int NW = 4, int NMAX = TRSM_NMAX>
__device__ __attribute__((always_inline)) inline void trsm_panel_inv(const UnitDesc &u, int panel,
                                                                     double *smem)
{
    // NW waves per workgroup (4 in the generic kernel, 8 in k_batch_trsm:
    // two waves per SIMD hide each other's MFMA and load latency); NMAX the
    // largest triangle the caller's LDS holds
    static_assert(NMAX % (64 * NW) == 0, "row blocks come in groups of four per wave");
    const int n = u.m, p0 = panel * TRSM_W, w = min(TRSM_W, u.n - p0);
    const int np = (n + 15) & ~15, nblk = np >> 4;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int li = lane & 15, lk = lane >> 4;
    double *Y = smem;  // [np][16]
    const MU_G double *t = gp(u.a);
    const MU_G double *winv = gp(u.b);
    const size_t ldt = u.lda, ldz = u.ldc;
    MU_G double *z = gp(u.c);
    const double alpha = u.alpha;
    // 32-bit offsets with 24-bit multiplies (full rate, unlike 64-bit
    // products): the lowering guarantees (n + 1) * ldt < 2^31 for triangles
    const unsigned ldt32 = (unsigned)ldt;
    auto tv = [&](int r, int c) -> double {
        if (REV) {
            r = n - 1 - r;
            c = n - 1 - c;
        }
        const unsigned off = TT ? (unsigned)c + __umul24((unsigned)r, ldt32)
                                : (unsigned)r + __umul24((unsigned)c, ldt32);
        return t[off];
    };
    auto zp = [&](int r, int c) -> MU_G double * {
        if (REV)
            r = n - 1 - r;
        return ZR ? z + (p0 + c) + r * ldz : z + r + (p0 + c) * ldz;
    };

    for (int idx = tid; idx < np * 16; idx += 64 * NW) {
        int r, c;
        if (ZR) {
            c = idx & 15;
            r = idx >> 4;
        } else {
            r = idx % np;
            c = idx / np;
        }
        Y[r * 16 + c] = (r < n && c < w) ? alpha * *zp(r, c) : 0.0;
    }
    lds_barrier();

    constexpr int MAXB = NMAX / (16 * NW);
    auto load_inv = [&](double (&wv)[4], int jb) {
        const MU_G double *b = winv + (size_t)min(jb >> 4, nblk - 1) * 256 + li * 16 + lk;
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
            wv[kk] = b[4 * kk];
    };
    auto load_block = [&](double (&f)[4], int jb, int i) {
        const int rb = jb + 16 + 16 * wave + 16 * NW * i;
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
            f[kk] = tv(min(rb + li, n - 1), min(jb + 4 * kk + lk, n - 1));
    };
    auto step = [&](int jb, const double (&wv)[4], const double (&fa)[MAXB][4], double (&wn)[4],
                    double (&fn)[MAXB][4]) {
        double yb[4];
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
            yb[kk] = Y[(jb + 4 * kk + lk) * 16 + li];
        v4d xs = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int kk = 0; kk < 4; kk++)
            xs = mfma_f64(wv[kk], yb[kk], xs);
        // xs[e] = X[jb + 4e + lk][li]
        if (wave == 0) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = jb + 4 * e + lk;
                if (r < n && li < w)
                    *zp(r, li) = xs[e];
            }
        }
        load_inv(wn, jb + 16);
        // Row blocks in groups of four under one (wave-uniform) test, so the
        // four MFMA chains of a group interleave: the accumulators start as
        // the Y rows and take -T[rb, jb] X_jb.  A block of a live group that
        // lies past the panel reads clamped rows and is not written back.
#pragma unroll
        for (int g = 0; g < MAXB / 4; g++) {
            const int rb0 = jb + 16 + 16 * wave + 64 * NW * g;
            if (rb0 < np) {
                v4d acc[4];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int rr = min(rb0 + 16 * NW * q, np - 16);
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        acc[q][e] = Y[(rr + 4 * e + lk) * 16 + li];
                }
#pragma unroll
                for (int kk = 0; kk < 4; kk++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const bool in = rb0 + 16 * NW * q + li < n && jb + 4 * kk + lk < n;
                        acc[q] = mfma_f64(in ? -fa[4 * g + q][kk] : 0.0, xs[kk], acc[q]);
                    }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int rb = rb0 + 16 * NW * q;
                    if (rb < np)
#pragma unroll
                        for (int e = 0; e < 4; e++)
                            Y[(rb + 4 * e + lk) * 16 + li] = acc[q][e];
                }
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
                load_block(fn[4 * g + q], jb + 16, 4 * g + q);
        }
        lds_barrier();
    };
    double fa0[MAXB][4], fa1[MAXB][4], w0[4], w1[4];
    load_inv(w0, 0);
#pragma unroll
    for (int i = 0; i < MAXB; i++)
        load_block(fa0[i], 0, i);
    for (int jb = 0; jb < n; jb += 32) {
        step(jb, w0, fa0, w1, fa1);
        if (jb + 16 >= n)
            break;
        step(jb + 16, w1, fa1, w0, fa0);
    }
}

// ---------------------------------------------------------------------------
// Small factorizations of an n x n tile (n <= SMALL_MAX) held in LDS.
// ---------------------------------------------------------------------------

__device__ __forceinline__ void report_info(const UnitDesc &u, int col)
{
    if (u.info)
        __hip_atomic_fetch_min(u.info, u.info_base + col + 1, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
}

// ---------------------------------------------------------------------------
// Blocked diagonal factorizations of an n x n tile (n <= SMALL_MAX): no-pivot
// LU (GETRF) and lower Cholesky (POTRF), right-looking over 16 x 16 blocks on
// four waves.  They are the serial chain of every tiled factorization, and
// beside GEMM workgroups each of their vector instructions waits for a
// 64-cycle FP64 MFMA, so what counts is the number of instructions in a row:
//   * only the 16 x 16 diagonal block is factored column by column, by the
//     wave that owns its block row, one matrix row per lane.  The pivot row /
//     column reaches the other lanes inside the FMA itself (v_fmac_f64 with
//     a row_newbcast operand) instead of two readlanes per element;
//   * the same wave forms the inverse(s) of the factored block with the same
//     instruction, so every other block of the panel is one product with a
//     16 x 16 inverse on MFMA, corrected once (solve_blk16), instead of a
//     sweep over its rows;
//   * the trailing update is MFMA on registers.
// Alone, order 125: POTRF 37 -> 27 us, GETRF 91 -> 47 us against the form that
// swept all 128 rows with readlanes and kept inv(L11) only.
//
// Registers: block (i, j) lives on the wave of its block row (rows w and
// w + 4 on wave w) transposed in the MFMA result layout: element e of lane
// (li, lk) is A(16 i + li, 16 j + 4 e + lk).  That is the B operand of A_ij^T
// and the A operand of A_ij, and a global access covers 16 consecutive rows.
// Rows and columns past n are the identity, so the padded factorization is
// the n x n one; only the n x n part (Cholesky: its lower triangle) is
// stored, each block as soon as it is final.  Zero pivots / non-positive
// minors report LAPACK-style info and the factorization continues (the
// factors then hold inf / nan).
// ---------------------------------------------------------------------------
constexpr int BF_LD = 17;                 // LDS row stride of a 16 x 16 block
constexpr int BF_BLK = 16 * BF_LD;        // doubles of such a block
// POTRF: the diagonal block / its inverse, two factored diagonal blocks, and
// the solved panel in register format; GETRF: two inverses, two factored
// diagonal blocks, the raw and the solved row panel
constexpr int LDS_POTRF = 3 * BF_BLK + 8 * 256;
constexpr int LDS_GETRF = 4 * BF_BLK + 7 * BF_BLK + 7 * 256;
constexpr int LDS_SMALL_BLK = LDS_GETRF > LDS_POTRF ? LDS_GETRF : LDS_POTRF;

// 1/x and 1/sqrt(x) in FP64 from the hardware estimates (v_rcp_f64,
// v_rsq_f64) and two Newton steps each (r <- r + r (1 - x r), r <- r + r
// (1/2 - x r^2 / 2)), within an ulp or two of the rounded results: the
// panel factorizations' per-column reciprocal and square root, which as IEEE
// division / sqrt sequences were most of a panel's instructions.  A zero
// pivot gives NaN (not the division's inf) and a negative one NaN: either way
// the factors carry non-finite values, and the column is reported as info.
__device__ __forceinline__ double rcp_nr(double x)
{
    double r = __builtin_amdgcn_rcp(x);
    r = fma(r, fma(-x, r, 1.0), r);
    return fma(r, fma(-x, r, 1.0), r);
}
__device__ __forceinline__ double rsq_nr(double x)
{
    const double h = 0.5 * x;
    double r = __builtin_amdgcn_rsq(x);
    r = fma(r, fma(-h * r, r, 0.5), r);
    return fma(r, fma(-h * r, r, 0.5), r);
}

// Lane L's v of every group of 16 lanes.
template <int L>
__device__ __forceinline__ double bcast16(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffll), 0x150 + L, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + L, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// d[k] -= (s of lane k of the group) * m for k = K .. 15.  A DPP operand may
// be read two wait states after a VALU write of it; the s_nop (8 cycles) at
// the head of each asm block covers whatever the compiler put before it, so
// the blocks are as wide as asm operands allow.
#define MU_FMAC(i, src, l)                                                                     \
    "v_fmac_f64_dpp %[d" #i "], " #src ", -%[m] row_newbcast:%[" #l "] row_mask:0xf bank_mask:0xf\n\t"
#define MU_IO(i) [d##i] "+&v"(d[K + i])
#define MU_L(i) [l##i] "n"(K + i)
template <int K>
__device__ __forceinline__ void fms_lane(double (&d)[16], double s, double m)
{
    if constexpr (K <= 4) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[s], l0) MU_FMAC(1, %[s], l1) MU_FMAC(2, %[s], l2) MU_FMAC(3, %[s], l3) MU_FMAC(4, %[s], l4) MU_FMAC(5, %[s], l5) MU_FMAC(6, %[s], l6) MU_FMAC(7, %[s], l7) MU_FMAC(8, %[s], l8) MU_FMAC(9, %[s], l9) MU_FMAC(10, %[s], l10) MU_FMAC(11, %[s], l11)
            : MU_IO(0), MU_IO(1), MU_IO(2), MU_IO(3), MU_IO(4), MU_IO(5), MU_IO(6), MU_IO(7), MU_IO(8), MU_IO(9), MU_IO(10), MU_IO(11)
            : [s] "v"(s), [m] "v"(m), MU_L(0), MU_L(1), MU_L(2), MU_L(3), MU_L(4), MU_L(5), MU_L(6), MU_L(7), MU_L(8), MU_L(9), MU_L(10), MU_L(11));
        fms_lane<K + 12>(d, s, m);
    } else if constexpr (K <= 8) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[s], l0) MU_FMAC(1, %[s], l1) MU_FMAC(2, %[s], l2) MU_FMAC(3, %[s], l3) MU_FMAC(4, %[s], l4) MU_FMAC(5, %[s], l5) MU_FMAC(6, %[s], l6) MU_FMAC(7, %[s], l7)
            : MU_IO(0), MU_IO(1), MU_IO(2), MU_IO(3), MU_IO(4), MU_IO(5), MU_IO(6), MU_IO(7)
            : [s] "v"(s), [m] "v"(m), MU_L(0), MU_L(1), MU_L(2), MU_L(3), MU_L(4), MU_L(5), MU_L(6), MU_L(7));
        fms_lane<K + 8>(d, s, m);
    } else if constexpr (K <= 10) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[s], l0) MU_FMAC(1, %[s], l1) MU_FMAC(2, %[s], l2) MU_FMAC(3, %[s], l3) MU_FMAC(4, %[s], l4) MU_FMAC(5, %[s], l5)
            : MU_IO(0), MU_IO(1), MU_IO(2), MU_IO(3), MU_IO(4), MU_IO(5)
            : [s] "v"(s), [m] "v"(m), MU_L(0), MU_L(1), MU_L(2), MU_L(3), MU_L(4), MU_L(5));
        fms_lane<K + 6>(d, s, m);
    } else if constexpr (K <= 12) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[s], l0) MU_FMAC(1, %[s], l1) MU_FMAC(2, %[s], l2) MU_FMAC(3, %[s], l3)
            : MU_IO(0), MU_IO(1), MU_IO(2), MU_IO(3)
            : [s] "v"(s), [m] "v"(m), MU_L(0), MU_L(1), MU_L(2), MU_L(3));
        fms_lane<K + 4>(d, s, m);
    } else if constexpr (K <= 13) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[s], l0) MU_FMAC(1, %[s], l1) MU_FMAC(2, %[s], l2)
            : MU_IO(0), MU_IO(1), MU_IO(2)
            : [s] "v"(s), [m] "v"(m), MU_L(0), MU_L(1), MU_L(2));
        fms_lane<K + 3>(d, s, m);
    } else if constexpr (K <= 14) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[s], l0) MU_FMAC(1, %[s], l1)
            : MU_IO(0), MU_IO(1)
            : [s] "v"(s), [m] "v"(m), MU_L(0), MU_L(1));
        fms_lane<K + 2>(d, s, m);
    } else if constexpr (K <= 15) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[s], l0)
            : MU_IO(0)
            : [s] "v"(s), [m] "v"(m), MU_L(0));
        fms_lane<K + 1>(d, s, m);
    }
}
// d[k] -= (d[k] of lane L) * m for k = K .. 15
template <int L, int K>
__device__ __forceinline__ void fms_self(double (&d)[16], double m)
{
    if constexpr (K <= 4) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[d0], l) MU_FMAC(1, %[d1], l) MU_FMAC(2, %[d2], l) MU_FMAC(3, %[d3], l) MU_FMAC(4, %[d4], l) MU_FMAC(5, %[d5], l) MU_FMAC(6, %[d6], l) MU_FMAC(7, %[d7], l) MU_FMAC(8, %[d8], l) MU_FMAC(9, %[d9], l) MU_FMAC(10, %[d10], l) MU_FMAC(11, %[d11], l)
            : MU_IO(0), MU_IO(1), MU_IO(2), MU_IO(3), MU_IO(4), MU_IO(5), MU_IO(6), MU_IO(7), MU_IO(8), MU_IO(9), MU_IO(10), MU_IO(11)
            : [m] "v"(m), [l] "n"(L));
        fms_self<L, K + 12>(d, m);
    } else if constexpr (K <= 8) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[d0], l) MU_FMAC(1, %[d1], l) MU_FMAC(2, %[d2], l) MU_FMAC(3, %[d3], l) MU_FMAC(4, %[d4], l) MU_FMAC(5, %[d5], l) MU_FMAC(6, %[d6], l) MU_FMAC(7, %[d7], l)
            : MU_IO(0), MU_IO(1), MU_IO(2), MU_IO(3), MU_IO(4), MU_IO(5), MU_IO(6), MU_IO(7)
            : [m] "v"(m), [l] "n"(L));
        fms_self<L, K + 8>(d, m);
    } else if constexpr (K <= 10) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[d0], l) MU_FMAC(1, %[d1], l) MU_FMAC(2, %[d2], l) MU_FMAC(3, %[d3], l) MU_FMAC(4, %[d4], l) MU_FMAC(5, %[d5], l)
            : MU_IO(0), MU_IO(1), MU_IO(2), MU_IO(3), MU_IO(4), MU_IO(5)
            : [m] "v"(m), [l] "n"(L));
        fms_self<L, K + 6>(d, m);
    } else if constexpr (K <= 12) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[d0], l) MU_FMAC(1, %[d1], l) MU_FMAC(2, %[d2], l) MU_FMAC(3, %[d3], l)
            : MU_IO(0), MU_IO(1), MU_IO(2), MU_IO(3)
            : [m] "v"(m), [l] "n"(L));
        fms_self<L, K + 4>(d, m);
    } else if constexpr (K <= 13) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[d0], l) MU_FMAC(1, %[d1], l) MU_FMAC(2, %[d2], l)
            : MU_IO(0), MU_IO(1), MU_IO(2)
            : [m] "v"(m), [l] "n"(L));
        fms_self<L, K + 3>(d, m);
    } else if constexpr (K <= 14) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[d0], l) MU_FMAC(1, %[d1], l)
            : MU_IO(0), MU_IO(1)
            : [m] "v"(m), [l] "n"(L));
        fms_self<L, K + 2>(d, m);
    } else if constexpr (K <= 15) {
        asm("s_nop 1\n\t" MU_FMAC(0, %[d0], l)
            : MU_IO(0)
            : [m] "v"(m), [l] "n"(L));
        fms_self<L, K + 1>(d, m);
    }
}
#undef MU_FMAC
#undef MU_IO
#undef MU_L

// The head of column C: d[C + 1 .. C + 3] updated (SELF: with their own lane
// C, as fms_self<C>; else with s of lanes C + 1 .. C + 3, as fms_lane).  The
// block ends two wait states after the write of d[C + 1], which a DPP move
// (the next pivot's broadcast) may then read.
#define MU_F3(s0, s1, s2, l0, l1, l2)                                                         \
    "s_nop 1\n\tv_fmac_f64_dpp %0, " s0 ", -%4 row_newbcast:" l0 " row_mask:0xf bank_mask:0xf\n\t" \
    "v_fmac_f64_dpp %1, " s1 ", -%4 row_newbcast:" l1 " row_mask:0xf bank_mask:0xf\n\t"        \
    "v_fmac_f64_dpp %2, " s2 ", -%4 row_newbcast:" l2 " row_mask:0xf bank_mask:0xf"
template <bool SELF, int C>
__device__ __forceinline__ void col_head(double (&d)[16], double s, double m)
{
    if constexpr (C < 13) {
        if constexpr (SELF)
            asm(MU_F3("%0", "%1", "%2", "%5", "%5", "%5")
                : "+&v"(d[C + 1]), "+&v"(d[C + 2]), "+&v"(d[C + 3])
                : "v"(s), "v"(m), "n"(C));
        else
            asm(MU_F3("%3", "%3", "%3", "%5", "%6", "%7")
                : "+&v"(d[C + 1]), "+&v"(d[C + 2]), "+&v"(d[C + 3])
                : "v"(s), "v"(m), "n"(C + 1), "n"(C + 2), "n"(C + 3));
    } else if constexpr (C < 15) {
        if constexpr (SELF)
            fms_self<C, C + 1>(d, m);
        else
            fms_lane<C + 1>(d, s, m);
        asm("s_nop 1" : "+v"(d[C + 1]));
    }
}
#undef MU_F3

// Cholesky of a 16 x 16 block, lane li holding row li in x (lower part
// valid; every group of 16 lanes the same block), and column li of inv(L) in
// z (the identity's on entry), row C of it stored to W once final.  `piv` is
// the pivot of column C, `bad` the first failing column.
template <int C>
__device__ __forceinline__ void potrf16(double (&x)[16], double (&z)[16], double *W, double piv,
                                        int &bad)
{
    if constexpr (C < 16) {
        bad = min(bad, piv > 0.0 ? 16 : C);
        const double rd = rsq_nr(piv);
        x[C] *= rd;
        if constexpr (C < 15) {
            col_head<false, C>(x, x[C], x[C]);
            piv = bcast16<C + 1>(x[C + 1]);
        }
        z[C] *= rd;
        W[C * BF_LD] = z[C];
        if constexpr (C < 13)
            fms_lane<C + 4>(x, x[C], x[C]);
        fms_lane<C + 1>(z, x[C], z[C]);
        potrf16<C + 1>(x, z, W, piv, bad);
    }
}

// No-pivot elimination of a 16 x 16 block, A = L U, and inv(L) or inv(U)^T.
// Lane li of a group of 16 holds row li of the block in x (ROW) or column li
// (!ROW), afterwards the same of the packed factors.  Both forms round alike,
// l = fl(a / pivot) and a - l u in one FMA, so they hold the same factors to
// the bit: scaling the transposed block's rows by the pivot instead (an
// elimination of A^T) gives another U, and its inverse is off by eps cond(A).
// Column C: the multipliers l (ROW), or the pivot row u, are in m; lane C has
// the other one, in place (ROW) or scaled by 1 / pivot first (!ROW).
// z: column li of the identity, turned into the inverse's by substitution
// with L, or U^T (!ROW), row C of it stored to W.
template <int C>
__device__ __forceinline__ void getrf16(double (&x)[16], double (&z)[16], double *W, double piv,
                                        int li, bool row, int &bad)
{
    if constexpr (C < 16) {
        bad = min(bad, piv == 0.0 ? C : 16);
        const double rd = rcp_nr(piv);
        const double rr = row ? rd : 1.0, rc = row ? 1.0 : rd;
        const double m = li > C ? x[C] * rr : 0.0;
        x[C] = li > C ? m : x[C];
        const double f = li == C ? rc : 1.0;
#pragma unroll
        for (int k = C + 1; k < 16; k++)
            x[k] *= f;
        if constexpr (C < 15) {
            col_head<true, C>(x, m, m);
            piv = bcast16<C + 1>(x[C + 1]);
        }
        z[C] *= rc;
        W[C * BF_LD] = z[C];
        if constexpr (C < 13)
            fms_self<C, C + 4>(x, m);
        fms_lane<C + 1>(z, m, z[C]);
        getrf16<C + 1>(x, z, W, piv, li, row, bad);
    }
}

// this wave's own LDS traffic is done (no barrier)
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

// Block (i, j) of an n x n tile into its register format; rows and columns
// past n read the last one.  Offsets are 64-bit everywhere: a tile of a tall
// matrix spans more than 2^32 elements from a leading dimension of 34 million
// on.  The scheduling barrier keeps one block's addresses from living beside
// the next one's.
__device__ __forceinline__ void load_blk16(v4d &v, const MU_G double *a, unsigned lda, int n, int i,
                                           int j, int li, int lk)
{
    const size_t r = min(16 * i + li, n - 1);
#pragma unroll
    for (int e = 0; e < 4; e++)
        v[e] = a[r + (size_t)min(16 * j + 4 * e + lk, n - 1) * lda];
    __builtin_amdgcn_sched_barrier(0);
}

// acc[] -= the products of k-steps e = 0 .. 3, a block at a time: MFMA A
// operands from LDS (register format, blocks 256 apart), the next block's
// read ahead of this block's MFMAs.
template <int J0, int J1>
__device__ __forceinline__ void update_row(v4d *acc, const double *lds, const v4d &x)
{
    double f[2][4];
#pragma unroll
    for (int e = 0; e < 4; e++)
        f[J0 & 1][e] = lds[J0 * 256 + e * 64];
#pragma unroll
    for (int j = J0; j < J1; j++) {
        if (j + 1 < J1)
#pragma unroll
            for (int e = 0; e < 4; e++)
                f[(j + 1) & 1][e] = lds[(j + 1) * 256 + e * 64];
#pragma unroll
        for (int e = 0; e < 4; e++)
            acc[j] = mfma_f64(f[j & 1][e], x[e], acc[j]);
        __builtin_amdgcn_sched_barrier(0);
    }
}

__device__ __forceinline__ const MU_LDS double *lp(const double *p)
{
    return (const MU_LDS double *)p;
}

// A lower 16 x 16 triangle in LDS.
struct TriRef {
    const MU_LDS double *t;  // T(r, c) at t[r rs + c cs], c < r
    int rs, cs;
    const MU_LDS double *d;  // 1 / T(r, r) at d[r (BF_LD + 1)]: the inverse's diagonal
};

// inv(T) Y by substitution, out of line: the kernels that call it keep their
// size and registers (inlined at its 48 places it doubles k_batch_small).
__device__ __noinline__ inline v4d subst_blk16(v4d y, TriRef tri)
{
    const int lane = threadIdx.x & 63, li = lane & 15, lk = lane >> 4;
#pragma unroll 1
    for (int r = 0; r < 16; r++) {
        double v = r < 4 ? y[0] : r < 8 ? y[1] : r < 12 ? y[2] : y[3];
        v = __shfl(v, li + 16 * (r & 3)) * tri.d[r * (BF_LD + 1)];
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int i = 4 * e + lk;
            const double f = fma(-tri.t[i * tri.rs + r * tri.cs], v, y[e]);
            y[e] = i == r ? v : i > r ? f : y[e];
        }
    }
    return y;
}

// X = inv(T) Y for N blocks of Y in register format, T a lower 16 x 16
// triangle: W ~ inv(T) and T come as this lane's MFMA A operands, element
// (li, 4 e + lk).  The product with an inverse alone leaves a residual of eps
// cond(T) where substitution leaves eps -- a Cholesky of a kernel matrix (128
// points, 1e-12 added to the diagonal) then met a negative pivot -- so it is
// corrected once, X += W (Y - T X): the residual falls to eps + (eps
// cond(T))^2.  That is eight more MFMAs per block; substitution is 136
// instructions on the vector ALU, each of which waits behind the MFMAs of the
// GEMM workgroups on its SIMD.  Order 128 in a graph node: POTRF 29.0 -> 32.2
// us, GETRF 39.0 -> 46.9 us (1.9 of these for getrf16's consistent factors).
//
// A column that is not finite afterwards is substituted: the products multiply
// the other halves' zeros too, and would spread a NaN or an infinity to the
// rows before it.  `tri` is the triangle in LDS.  A column's first rows show it:
// 0 * inf and 0 * NaN are NaN.
template <int N>
__device__ __forceinline__ void solve_blk16(v4d (&X)[N], const v4d (&Y)[N], const double (&w)[4],
                                            const double (&t)[4], const TriRef &tri)
{
    v4d R[N];
#pragma unroll
    for (int b = 0; b < N; b++) {
        X[b] = v4d{0.0, 0.0, 0.0, 0.0};
        R[b] = Y[b];
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int b = 0; b < N; b++)
            X[b] = mfma_f64(w[e], Y[b][e], X[b]);
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int b = 0; b < N; b++)
            R[b] = mfma_f64(t[e], -X[b][e], R[b]);
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int b = 0; b < N; b++)
            X[b] = mfma_f64(w[e], R[b][e], X[b]);
    unsigned long long bad[N], any = 0;
#pragma unroll
    for (int b = 0; b < N; b++) {
        bad[b] = __ballot(!(fabs(X[b][0]) < __builtin_inf()));
        any |= bad[b];
    }
    if (__builtin_expect(any != 0, 0)) {
        const int li = threadIdx.x & 15;
#pragma unroll
        for (int b = 0; b < N; b++) {
            const v4d y = subst_blk16(Y[b], tri);
            const unsigned long long m = bad[b] | bad[b] >> 32, col = (m | m >> 16) >> li;
            X[b] = col & 1 ? y : X[b];
        }
    }
}

struct SmallCtx {
    int n, nb, w, li, lk, lane;
    MU_G double *a;
    unsigned lda;  // uniform (a scalar register)
    // Once per step: hides that lane and leading dimension are the same in
    // every step.  Otherwise the addresses of all eight steps' loads and
    // stores are computed ahead of the loop and live (spilled) across it.
    __device__ __forceinline__ void refresh()
    {
        asm volatile("" : "+v"(lane), "+s"(lda));
        li = lane & 15;
        lk = lane >> 4;
    }
};

// Block (i, P) of the factor from its register format.
template <int P>
__device__ __forceinline__ void store_blk16(const SmallCtx &c, int i, const v4d &x)
{
    if (16 * i + c.li < c.n)
#pragma unroll
        for (int e = 0; e < 4; e++)
            (c.a + 16 * i + (size_t)(16 * P + 4 * e) * c.lda)[c.li + (size_t)c.lk * c.lda] = x[e];
}

// The owner of block row p + 1 hands its diagonal block to the factoring wave.
__device__ __forceinline__ void put_diag16(const SmallCtx &c, double *W, const v4d &D)
{
#pragma unroll
    for (int e = 0; e < 4; e++)
        W[c.li * BF_LD + 4 * e + c.lk] = D[e];
}

// Waves.  Four waves, block rows w and w + 4 on wave w.  Wave 0 also factors
// every diagonal block: its row 0 only goes through LDS, so that it holds one
// block row beside the 64 registers of the block's columns.  At 200 registers
// per lane the kernel starts on a CU as soon as one of four GEMM workgroups
// (104 each) leaves it; at 256 it had to find two gone and waited 400 us and
// more per node beside a bulk update.  Barriers per step: the inverse is in
// LDS (A), the solved panel is in LDS (B), the next diagonal block is in LDS
// (C).  The trailing update of the other blocks runs beside the next diagonal
// block's columns.
//
// The factored diagonal block p from LDS to the matrix (LOWER: its lower part).
template <bool LOWER>
__device__ __forceinline__ void store_diag16(const SmallCtx &c, int p, const double *D)
{
    if (16 * p + c.li < c.n)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = 4 * e + c.lk;
            if (LOWER ? k <= c.li : 16 * p + k < c.n)
                (c.a + 16 * p + (size_t)(16 * p + 4 * e) * c.lda)[c.li + (size_t)c.lk * c.lda] =
                    D[c.li * BF_LD + k];
        }
}

// Lower Cholesky.  Factoring step p: A_pp = L_pp L_pp^T, inv(L_pp) to W, L_pp
// to D (two buffers in turn: a tile wave stores it a step later).
__device__ __forceinline__ void potrf_diag(const SmallCtx &c, const UnitDesc &u, int p, double *W,
                                           double *D)
{
    const int li = c.li;
    double x[16], z[16];
#pragma unroll
    for (int k = 0; k < 16; k++) {
        x[k] = W[li * BF_LD + k];
        z[k] = k == li ? 1.0 : 0.0;
    }
    lds_wait();
    int bad = 16;
    potrf16<0>(x, z, W + li, bcast16<0>(x[0]), bad);
    if (bad < 16 && c.lane == 0)
        report_info(u, 16 * p + bad);
#pragma unroll
    for (int k = 0; k < 16; k++)
        D[li * BF_LD + k] = x[k];
}

// Tile waves, step P: L_ip^T = inv(L_pp) A_ip^T for the blocks below (D: L_pp
// with anything above its diagonal), stored and handed on as -L_ip (Lb); then A_ij^T += (-L_jp) L_ip^T, the next
// diagonal block first.  R0: row w, columns 0 .. 3; R1: row w + 4 (blocks
// right of the diagonal hold nothing that is read).
template <int P, bool W0>
__device__ __forceinline__ void potrf_step(const SmallCtx &c, v4d (&R0)[4], v4d (&R1)[8],
                                           double *W, const double *D, double *Lb)
{
    const bool on0 = !W0 && P < 3 && c.w > P && c.w < c.nb;
    const bool on1 = c.w + 4 > P && c.w + 4 < c.nb;
    v4d X0, X1;
    double wv[4], tv[4];
    const TriRef tri = {lp(D), BF_LD, 1, lp(W)};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int k = 4 * e + c.lk;
        wv[e] = W[c.li * BF_LD + k];
        tv[e] = k <= c.li ? D[c.li * BF_LD + k] : 0.0;
    }
    if constexpr (!W0 && P < 3) {
        if (on0) {  // row w + 4 may be past the tile: a block nothing reads
            v4d X[2];
            const v4d Y[2] = {R0[P], R1[P]};
            solve_blk16(X, Y, wv, tv, tri);
            X0 = X[0];
            X1 = X[1];
        }
    }
    if (!on0 && on1) {
        v4d X[1];
        const v4d Y[1] = {R1[P]};
        solve_blk16(X, Y, wv, tv, tri);
        X1 = X[0];
    }
    auto put = [&](int i, const v4d &x) {
#pragma unroll
        for (int e = 0; e < 4; e++)
            Lb[i * 256 + e * 64 + c.lane] = -x[e];
    };
    if (on0)
        put(c.w, X0);
    if (on1)
        put(c.w + 4, X1);
    lds_barrier();  // B
    const double *L = Lb + c.lane;
    constexpr int Q = P + 1;  // the next diagonal block
    if (c.w == (Q & 3)) {
        if constexpr (Q >= 4) {
            update_row<Q, Q + 1>(R1, L, X1);
            put_diag16(c, W, R1[Q]);
        } else if constexpr (!W0) {
            update_row<Q, Q + 1>(R0, L, X0);
            put_diag16(c, W, R0[Q]);
        }
    }
    lds_barrier();  // C
    if (on0)
        store_blk16<P>(c, c.w, X0);
    if (on1)
        store_blk16<P>(c, c.w + 4, X1);
    if constexpr (!W0 && Q < 3)
        if (on0 && c.w > Q)  // columns past w are not used
            update_row<Q, 4>(R0, L, X0);
    if (on1 && c.w + 4 > Q) {
        if constexpr (!W0 || Q < 5)
            update_row<Q, (Q < 5 ? 5 : Q + 1)>(R1, L, X1);
        if constexpr (!W0 && Q < 5)
            update_row<5, 6>(R1, L, X1);
        if constexpr (!W0 && Q < 6)
            if (c.w >= 2)
                update_row<6, 7>(R1, L, X1);
        if constexpr (!W0 && Q < 7)
            if (c.w >= 3)
                update_row<7, 8>(R1, L, X1);
    }
}

// Step p (a switch: the register arrays need constant indices).
template <bool W0>
__device__ __forceinline__ void potrf_steps(const SmallCtx &c, int p, v4d (&R0)[4], v4d (&R1)[8],
                                            double *W, const double *D, double *Lb)
{
    switch (p) {
    case 0: potrf_step<0, W0>(c, R0, R1, W, D, Lb); break;
    case 1: potrf_step<1, W0>(c, R0, R1, W, D, Lb); break;
    case 2: potrf_step<2, W0>(c, R0, R1, W, D, Lb); break;
    case 3: potrf_step<3, W0>(c, R0, R1, W, D, Lb); break;
    case 4: potrf_step<4, W0>(c, R0, R1, W, D, Lb); break;
    case 5: potrf_step<5, W0>(c, R0, R1, W, D, Lb); break;
    default: potrf_step<6, W0>(c, R0, R1, W, D, Lb); break;
    }
}

template <bool W0>
__device__ __forceinline__ void potrf_waves(SmallCtx c, const UnitDesc &u, double *W, double *D,
                                            double *Lb)
{
    const int n = c.n, nb = c.nb, w = c.w, li = c.li, lk = c.lk;
    // every load first, from addresses clamped into the tile; then the parts
    // outside the tile and above the diagonal (uniform tests: edge blocks only)
    v4d R0[4], R1[8];
#pragma unroll
    for (int j = 0; j < (W0 ? 1 : 4); j++)
        load_blk16(R0[j], c.a, c.lda, n, w, min(j, w), li, lk);
#pragma unroll
    for (int j = 0; j < (W0 ? 5 : 8); j++)
        load_blk16(R1[j], c.a, c.lda, n, w + 4, min(j, w + 4), li, lk);
    auto mask = [&](v4d &v, int i, int j) {
        if (i == j || i >= nb - 1)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = 16 * i + li, k = 16 * j + 4 * e + lk;
                v[e] = (r < n && k <= r) ? v[e] : (r == k ? 1.0 : 0.0);
            }
    };
#pragma unroll
    for (int j = 0; j < (W0 ? 1 : 4); j++)
        mask(R0[j], w, j);
    if (W0)
        put_diag16(c, W, R0[0]);
#pragma unroll
    for (int j = 0; j < (W0 ? 5 : 8); j++)
        mask(R1[j], w + 4, j);
    lds_barrier();  // C
    for (int p = 0;; p++) {
        c.refresh();
        if (W0)
            potrf_diag(c, u, p, W, D + (p & 1) * BF_BLK);
        lds_barrier();  // A
        if (p + 1 < nb)
            potrf_steps<W0>(c, p, R0, R1, W, D + (p & 1) * BF_BLK, Lb);
        if (w == (p & 3))
            store_diag16<true>(c, p, D + (p & 1) * BF_BLK);
        if (p + 1 == nb)
            break;
    }
}

__device__ __attribute__((always_inline)) inline void potrf_small(const UnitDesc &u, double *smem)
{
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const SmallCtx c = {u.m,       (u.m + 15) >> 4, w, lane & 15, lane >> 4, lane, gp(u.c),
                        (unsigned)__builtin_amdgcn_readfirstlane(u.ldc)};
    double *W = smem, *D = W + BF_BLK, *Lb = D + 2 * BF_BLK;
    __builtin_amdgcn_s_setprio(3);
    if (w == 0)
        potrf_waves<true>(c, u, W, D, Lb);
    else
        potrf_waves<false>(c, u, W, D, Lb);
    __builtin_amdgcn_s_setprio(0);
}

// No-pivot LU.  Factoring step p: two groups of 16 lanes eliminate A_pp at
// once, one on its rows and one on its columns, and invert one factor each:
// W1 = inv(L), W2 = inv(U)^T.  The packed factors go to D.
__device__ __forceinline__ void getrf_diag(const SmallCtx &c, const UnitDesc &u, int p, double *W1,
                                           double *W2, double *D)
{
    const int li = c.li;
    // groups 0 and 2: rows of the block, groups 1 and 3: its columns
    const int g = c.lk & 1;
    double x[16], z[16];
#pragma unroll
    for (int k = 0; k < 16; k++) {
        x[k] = W1[g ? k * BF_LD + li : li * BF_LD + k];
        z[k] = k == li ? 1.0 : 0.0;
    }
    lds_wait();
    int bad = 16;
    getrf16<0>(x, z, (g ? W2 : W1) + li, bcast16<0>(x[0]), li, g == 0, bad);
    if (bad < 16 && c.lane == 0)
        report_info(u, 16 * p + bad);
    if (g == 0)
#pragma unroll
        for (int k = 0; k < 16; k++)
            D[li * BF_LD + k] = x[k];
}

// Blocks J0 .. 7 of row panel row to LDS, block j at raw + (j - 1) BF_BLK.
template <int J0>
__device__ __forceinline__ void put_raw16(const SmallCtx &c, const v4d (&R)[8], double *raw)
{
#pragma unroll
    for (int j = J0; j < 8; j++)
        if (j < c.nb)
            put_diag16(c, raw + (j - 1) * BF_BLK, R[j]);
}

// Tile waves, step P (D: the packed factors of A_pp): L_ip^T = inv(U)^T A_ip^T
// for the blocks below, a share of the row panel, U_pj = inv(L) A_pj (copied to LDS raw by its owner),
// handed on as -U_pj (Ub); then A_ij^T += (-U_pj)^T L_ip^T, the next diagonal
// block first.  R0, R1: block rows w and w + 4.
template <int P, bool W0>
__device__ __forceinline__ void getrf_step(const SmallCtx &c, v4d (&R0)[8], v4d (&R1)[8],
                                           double *W1, const double *W2, const double *D,
                                           double *raw, double *Ub)
{
    const bool on0 = !W0 && P < 3 && c.w > P && c.w < c.nb;
    const bool on1 = c.w + 4 > P && c.w + 4 < c.nb;
    v4d X0, X1;
    double wv[4], tv[4];
    const TriRef ut = {lp(D), 1, BF_LD, lp(W2)}, l = {lp(D), BF_LD, 1, lp(W1)};
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int k = 4 * e + c.lk;
        wv[e] = W2[c.li * BF_LD + k];
        tv[e] = k <= c.li ? D[k * BF_LD + c.li] : 0.0;  // U^T
    }
    if constexpr (!W0 && P < 3) {
        if (on0) {  // row w + 4 may be past the tile: a block nothing reads
            v4d X[2];
            const v4d Y[2] = {R0[P], R1[P]};
            solve_blk16(X, Y, wv, tv, ut);
            X0 = X[0];
            X1 = X[1];
        }
    }
    if (!on0 && on1) {
        v4d X[1];
        const v4d Y[1] = {R1[P]};
        solve_blk16(X, Y, wv, tv, ut);
        X1 = X[0];
    }
    if (P + 1 + c.w < c.nb) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = 4 * e + c.lk;
            wv[e] = W1[c.li * BF_LD + k];
            tv[e] = k < c.li ? D[c.li * BF_LD + k] : k == c.li ? 1.0 : 0.0;  // L
        }
        for (int j = P + 1 + c.w; j < c.nb; j += 4) {
            const double *b = raw + (j - 1) * BF_BLK;
            v4d X[1], Y[1];
#pragma unroll
            for (int e = 0; e < 4; e++)
                Y[0][e] = b[(4 * e + c.lk) * BF_LD + c.li];
            solve_blk16(X, Y, wv, tv, l);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                Ub[(j - 1) * 256 + e * 64 + c.lane] = -X[0][e];
                if (16 * j + c.li < c.n)
                    (c.a + 16 * P + 4 * e + (size_t)(16 * j) * c.lda)[c.lk + (size_t)c.li * c.lda] =
                        X[0][e];
            }
        }
    }
    lds_barrier();  // B
    const double *U = Ub + c.lane - 256;
    constexpr int Q = P + 1;  // the next diagonal block
    const bool own = c.w == (Q & 3);
    if (own) {
        if constexpr (Q >= 4) {
            update_row<Q, Q + 1>(R1, U, X1);
            put_diag16(c, W1, R1[Q]);
        } else if constexpr (!W0) {
            update_row<Q, Q + 1>(R0, U, X0);
            put_diag16(c, W1, R0[Q]);
        }
    }
    lds_barrier();  // C
    // columns past nb hold nothing that is read
    if constexpr (Q < 4) {
        if constexpr (!W0) {
            if (own) {
                update_row<Q + 1, 8>(R0, U, X0);
                put_raw16<Q + 1>(c, R0, raw);
            } else if (on0) {
                update_row<Q, 8>(R0, U, X0);
            }
            if (on0)
                store_blk16<P>(c, c.w, X0);
        }
        if (on1)
            update_row<Q, 8>(R1, U, X1);
    } else if constexpr (!W0 || Q == 4) {
        if (own) {
            if constexpr (Q < 7)
                update_row<Q + 1, 8>(R1, U, X1);
            put_raw16<Q + 1>(c, R1, raw);
        } else if (on1) {
            update_row<Q, 8>(R1, U, X1);
        }
    }
    if (on1)
        store_blk16<P>(c, c.w + 4, X1);
}

template <bool W0>
__device__ __forceinline__ void getrf_steps(const SmallCtx &c, int p, v4d (&R0)[8], v4d (&R1)[8],
                                            double *W1, const double *W2, const double *D,
                                            double *raw, double *Ub)
{
    switch (p) {
    case 0: getrf_step<0, W0>(c, R0, R1, W1, W2, D, raw, Ub); break;
    case 1: getrf_step<1, W0>(c, R0, R1, W1, W2, D, raw, Ub); break;
    case 2: getrf_step<2, W0>(c, R0, R1, W1, W2, D, raw, Ub); break;
    case 3: getrf_step<3, W0>(c, R0, R1, W1, W2, D, raw, Ub); break;
    case 4: getrf_step<4, W0>(c, R0, R1, W1, W2, D, raw, Ub); break;
    case 5: getrf_step<5, W0>(c, R0, R1, W1, W2, D, raw, Ub); break;
    default: getrf_step<6, W0>(c, R0, R1, W1, W2, D, raw, Ub); break;
    }
}

template <bool W0>
__device__ __forceinline__ void getrf_waves(SmallCtx c, const UnitDesc &u, double *W1, double *W2,
                                            double *D, double *raw, double *Ub)
{
    const int n = c.n, nb = c.nb, w = c.w, li = c.li, lk = c.lk;
    v4d R0[8], R1[8];  // loads first, then the edges
    auto mask = [&](v4d &v, int i, int j) {
        if (i >= nb - 1 || j >= nb - 1)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = 16 * i + li, k = 16 * j + 4 * e + lk;
                v[e] = (r < n && k < n) ? v[e] : (r == k ? 1.0 : 0.0);
            }
    };
#pragma unroll
    for (int j = 0; j < 8; j++)
        load_blk16(R0[j], c.a, c.lda, n, w, j, li, lk);
#pragma unroll
    for (int j = 0; j < 8; j++)
        load_blk16(R1[j], c.a, c.lda, n, w + 4, j, li, lk);
    if (n & 15)
#pragma unroll
        for (int j = 0; j < 8; j++)
            mask(R0[j], w, j);
    if (W0) {
        put_diag16(c, W1, R0[0]);
        put_raw16<1>(c, R0, raw);
    }
    if (n & 15)
#pragma unroll
        for (int j = 0; j < 8; j++)
            mask(R1[j], w + 4, j);
    lds_barrier();  // C
    for (int p = 0;; p++) {
        c.refresh();
        if (W0)
            getrf_diag(c, u, p, W1, W2, D + (p & 1) * BF_BLK);
        lds_barrier();  // A
        if (p + 1 < nb)
            getrf_steps<W0>(c, p, R0, R1, W1, W2, D + (p & 1) * BF_BLK, raw, Ub);
        if (w == (p & 3))
            store_diag16<false>(c, p, D + (p & 1) * BF_BLK);
        if (p + 1 == nb)
            break;
    }
}

__device__ __attribute__((always_inline)) inline void getrf_small(const UnitDesc &u, double *smem)
{
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const SmallCtx c = {u.m,       (u.m + 15) >> 4, w, lane & 15, lane >> 4, lane, gp(u.c),
                        (unsigned)__builtin_amdgcn_readfirstlane(u.ldc)};
    double *W1 = smem, *W2 = W1 + BF_BLK, *D = W2 + BF_BLK;
    double *raw = D + 2 * BF_BLK, *Ub = raw + 7 * BF_BLK;
    __builtin_amdgcn_s_setprio(3);
    if (w == 0)
        getrf_waves<true>(c, u, W1, W2, D, raw, Ub);
    else
        getrf_waves<false>(c, u, W1, W2, D, raw, Ub);
    __builtin_amdgcn_s_setprio(0);
}

// ---------------------------------------------------------------------------
// Panel triangular solve, T Y = alpha Z in place, T lower triangular of order
// n <= TRSM_REG_MAX:
//   left-lower-unit   X = L^-1 B  : T = L,   Z = B (columns)
//   right-upper       X = B U^-1  : T = U^T, Z = B^T (rows of B)
//   right-lower-trans X = B L^-T  : T = L,   Z = B^T (rows of B)
// With F_REV the row order of T and Z is reversed, which turns an upper
// triangular solve (back substitution) into the same lower-triangular form.
//
// What bounds it: beside the other panel work it is on the chain to the next
// diagonal tile, and over a whole panel it is the matrix pipe.  Each wave
// owns 16 right-hand sides and keeps them in registers in the MFMA result
// layout (element e of block i: row 16 i + 4 e + lk, column li), which is the
// MFMA B operand, so a solve is a stream of MFMAs: X_j = inv(T_jj) Y_j, then
// Y_i -= T_ij X_j for the blocks below.  A work item is 64 right-hand sides
// (four waves).  The blocks T_ij below the diagonal stream through a ring in
// LDS in the order of use, copied by the waves in turn (global_load_lds,
// groups of four blocks, TRSM_RING - 1 groups ahead, one barrier per group):
// read by each wave for itself four blocks ahead, the stream was bound by
// memory latency (order 250: 48 us).  The workgroup first inverts all 16 x 16
// diagonal blocks at once, one block per group of 16 lanes, so no inversion
// kernel runs before it.  One node of the Cholesky at n = 7007, against a
// panel of 16 right-hand sides per workgroup in LDS (a barrier per 16 rows,
// four waves sharing each panel): order 125 28 -> 17 us, order 250 35 us
// after an inversion kernel of 10 us -> 38 us; N = 24000 LU 166 -> 152 ms.
//
// Strides are run-time values, so one body serves every side, triangle and
// transposition; blocks past the triangle compute on whatever the ring holds
// and are never stored.
// ---------------------------------------------------------------------------
// Groups of four T blocks in the ring: as many as keep the workgroup beside
// three GEMM workgroups of 32 KB with 16 inverses (34 KB), beside four with 8
// (four groups there: N = 24000 Cholesky 80.4 -> 78.8 ms with two).
template <int NB>
constexpr int TRSM_RING = NB > 8 ? 3 : 2;

template <class T>
__device__ __forceinline__ T *uniform_ptr(T *p)
{
    const unsigned long long v = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)v);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(v >> 32));
    return (T *)(((unsigned long long)hi << 32) | lo);
}

// Triangles of order <= SMALL_MAX are solved with the correction of
// solve_blk16, to the backward error of substitution; larger ones (parts of
// whole tiles) with the inverses of their diagonal blocks alone.  The
// correction costs (order 125, eager calls) 8.1 -> 10.2 us on panels of 16
// right-hand sides and 17.4 -> 20.4 us for 16384 on panels of 64.  The
// corrected solves keep the diagonal blocks T_jj beside their inverses: W(r,
// c) at [r BF_LD + c] for c <= r, T(r, c) at [c BF_LD + r] for c < r, T(r, r)
// at [r BF_LD + 16], and a zero that stands for the other halves.
template <int NB>
constexpr bool TRSM_FIX = NB <= SMALL_MAX / 16;
constexpr int TRSM_FIX_ZERO = BF_BLK;
template <int NB>
constexpr int TRSM_BLK = TRSM_FIX<NB> ? BF_BLK + 2 : BF_BLK;  // doubles of such a block

// column li of the inverse of a lower 16 x 16 block, lane li holding row li in
// x and 1 / its diagonal in rd: row C to W[C * BF_LD] (FIX: above the
// diagonal x instead)
template <bool FIX, int C>
__device__ __forceinline__ void tri_inv16(double (&z)[16], const double (&x)[16], double rd, int li,
                                          double *W)
{
    if constexpr (C < 16) {
        z[C] *= bcast16<C>(rd);
        W[C * BF_LD] = FIX && C < li ? x[C] : z[C];
        fms_lane<C + 1>(z, x[C], z[C]);
        tri_inv16<FIX, C + 1>(z, x, rd, li, W);
    }
}

// The inverses of the diagonal blocks in LDS, and (FIX) the blocks: lane li of
// a group holds row li in x, its diagonal entry in dv (1: a unit triangle's or
// a row past the end).
template <int NB>
__device__ __forceinline__ void trsm_invert(const double (&x)[16], double dv, int li, double *blk)
{
    double v[16];
#pragma unroll
    for (int c = 0; c < 16; c++)
        v[c] = c == li ? 1.0 : 0.0;
    if (TRSM_FIX<NB>) {
        blk[li * BF_LD + 16] = dv;
        blk[TRSM_FIX_ZERO] = 0.0;
    }
    tri_inv16<TRSM_FIX<NB>, 0>(v, x, 1.0 / dv, li, blk + li);
}

// This lane's MFMA A operands from block j of `blk`: element (li, 4 e + lk) of
// the inverse and (FIX) of the block.
template <int NB>
struct TrsmFrag {
    const double *blk;
    int ow[4], ot[4];
    __device__ __forceinline__ TrsmFrag(const double *smem, int li, int lk)
        : blk(TRSM_FIX<NB> ? smem : smem + li * BF_LD + lk)
    {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int k = 4 * e + lk;
            ow[e] = !TRSM_FIX<NB> ? 4 * e : k > li ? TRSM_FIX_ZERO : li * BF_LD + k;
            ot[e] = k < li ? k * BF_LD + li : k == li ? li * BF_LD + 16 : TRSM_FIX_ZERO;
        }
    }
    __device__ __forceinline__ void load(int j, double (&w)[4], double (&t)[4]) const
    {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            w[e] = blk[j * TRSM_BLK<NB> + ow[e]];
            if constexpr (TRSM_FIX<NB>)
                t[e] = blk[j * TRSM_BLK<NB> + ot[e]];
        }
    }
};

// X_j = inv(T_jj) Y_j; `blk` is block j (FIX).
template <int NB>
__device__ __forceinline__ v4d trsm_diag(const v4d &y, const double (&w)[4], const double (&t)[4],
                                         const double *blk)
{
    v4d X[1];
    const v4d Y[1] = {y};
    if constexpr (TRSM_FIX<NB>) {
        solve_blk16(X, Y, w, t, TriRef{lp(blk), 1, BF_LD, lp(blk)});
    } else {
        X[0] = v4d{0.0, 0.0, 0.0, 0.0};
#pragma unroll
        for (int e = 0; e < 4; e++)
            X[0] = mfma_f64(w[e], Y[0][e], X[0]);
    }
    return X[0];
}

// The T blocks below the diagonal in the order of use, column by column:
// block S of column J, row I.
template <int NB>
struct TrsmOrder {
    static constexpr int first(int j) { return j * (2 * NB - j - 1) / 2; }
    static constexpr int count = NB * (NB - 1) / 2, groups = (count + 3) / 4;
};

// Copies of this wave's block of each group of four into the ring.
template <int NB>
struct TrsmFeed {
    const MU_G double *t;
    unsigned ldt;
    int n, nb, lane;
    bool tt, rev;
    double *ring;  // this wave's slot of group 0
    int i, j;      // the block copied next
    __device__ __forceinline__ void copy(int g)
    {
        // T's block (i, j) in memory: rows from r0, columns from c0 (rev:
        // counted from the end, so it lies there mirrored).  Blocks past the
        // triangle take a block inside it.
        const int ic = min(i, nb - 1), jc = min(j, nb - 2);
        const int r0 = rev ? n - 16 - 16 * ic : 16 * ic, c0 = rev ? n - 16 - 16 * jc : 16 * jc;
        double *d = ring + (g % TRSM_RING<NB>) * 4 * 256;
#pragma unroll
        for (int q = 0; q < 2; q++) {
            const int a = 8 * q + (lane >> 3), b = lane & 7;
            // not transposed: column a, rows 2 b, 2 b + 1 at [a * 16 + 2 b];
            // rows past n are still inside the triangle's storage (column c0
            // + a is not the last one).  Transposed: row a, columns in
            // 16-byte chunks, chunk c at c ^ ((a / 2) % 8); rows clamped.
            const long long off =
                tt ? (long long)max(min(r0 + a, n - 1), 0) * ldt + c0 + 2 * (b ^ ((a >> 1) & 7))
                   : (long long)(c0 + a) * ldt + r0 + 2 * b;
            __builtin_amdgcn_global_load_lds((const MU_G unsigned *)(t + off),
                                             (MU_LDS unsigned *)(d + 128 * q), 16, 0, 0);
        }
        i += 4;
        wrap();
    }
    // to the column the block belongs to (past the last column: any)
    __device__ __forceinline__ void wrap()
    {
        while (i >= NB && j < NB - 1) {
            j++;
            i += j + 1 - NB;
        }
    }
};

// Start of group G: its copies have landed in every wave's slot; then the
// copies TRSM_RING - 1 groups on (into the slots of group G - 1, which every
// wave has read).
template <int NB, int G>
__device__ __forceinline__ void trsm_group(TrsmFeed<NB> &feed)
{
    constexpr int last = TrsmOrder<NB>::groups - 1;
    constexpr int R = TRSM_RING<NB>, ahead = (G + R - 2 < last ? G + R - 2 : last) - G;
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * ahead) : "memory");
    if constexpr (G + R - 1 <= last)
        feed.copy(G + R - 1);
}

// Y[I ..] -= T[I .., J] X_J (nx = -X_J).
template <int NB, int J, int I>
__device__ __forceinline__ void trsm_below(v4d (&Y)[NB], const double *ring, const int (&lo)[4],
                                           const v4d &nx, TrsmFeed<NB> &feed)
{
    if constexpr (I < NB) {
        constexpr int S = TrsmOrder<NB>::first(J) + I - J - 1;
        if constexpr (S % 4 == 0)
            trsm_group<NB, S / 4>(feed);
        const double *b = ring + (S / 4 % TRSM_RING<NB> * 4 + S % 4) * 256;
#pragma unroll
        for (int e = 0; e < 4; e++)
            Y[I] = mfma_f64(b[lo[e]], nx[e], Y[I]);
        trsm_below<NB, J, I + 1>(Y, ring, lo, nx, feed);
    }
}
// Columns J ..: X_J replaces Y_J.  The last block's rows past the triangle
// (rlast: the rows below this lane's first that are inside) were updated with
// rows of T that are not its own; they are zero as its inverse meets them.
template <int NB, int J>
__device__ __forceinline__ void trsm_columns(v4d (&Y)[NB], const TrsmFrag<NB> &frag,
                                             const double *ring, const int (&lo)[4], int nb,
                                             int rlast, TrsmFeed<NB> &feed)
{
    if constexpr (J < NB) {
        if (J >= nb)
            return;
        if (J == nb - 1)
#pragma unroll
            for (int e = 0; e < 4; e++)
                Y[J][e] = 4 * e < rlast ? Y[J][e] : 0.0;
        double w[4], t[4];
        frag.load(J, w, t);
        Y[J] = trsm_diag<NB>(Y[J], w, t, frag.blk + J * TRSM_BLK<NB>);
        if (J + 1 < nb) {
            const v4d nx = -Y[J];
            trsm_below<NB, J, J + 1>(Y, ring, lo, nx, feed);
        }
        trsm_columns<NB, J + 1>(Y, frag, ring, lo, nb, rlast, feed);
    }
}

template <int NB>
__device__ __attribute__((always_inline)) inline void trsm_panel_reg(const UnitDesc &u, int it,
                                                                     double *smem)
{
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = __builtin_amdgcn_readfirstlane(u.m), nb = (n + 15) >> 4;
    const int ncol = __builtin_amdgcn_readfirstlane(u.n);
    const int flags = __builtin_amdgcn_readfirstlane(u.flags);
    const bool rev = flags & F_REV, tt = flags & F_T_TRANS, zr = flags & F_Z_ROWS;
    const unsigned ldt = __builtin_amdgcn_readfirstlane(u.lda);
    const unsigned ldz = __builtin_amdgcn_readfirstlane(u.ldc);
    const MU_G double *t = gp(uniform_ptr(u.a));
    MU_G double *z = gp(uniform_ptr(u.c));
    const double alpha = u.alpha;
    double *ring = smem + NB * TRSM_BLK<NB>;
    // T(r, c) at t[r rs + c cs], Z(r, c) at z[r zrs + c zcs], rows (and T's
    // columns) counted from the end with rev
    const unsigned rs = tt ? ldt : 1, cs = tt ? 1 : ldt;
    const unsigned zrs = zr ? ldz : 1, zcs = zr ? 1 : ldz;

    TrsmFeed<NB> feed = {t, ldt, n, nb, lane, tt, rev, ring + wave * 256, 1 + wave, 0};
    feed.wrap();
    if (nb > 1)
#pragma unroll
        for (int g = 0; g < TRSM_RING<NB> - 1; g++)
            if (g < TrsmOrder<NB>::groups)
                feed.copy(g);

    // ---- inverses of the diagonal blocks, block wave + 4 lk on this group
    {
        const int jb = min(wave + 4 * lk, nb - 1);
        const int r = 16 * jb + li, rc = min(r, n - 1);
        double x[16];
        auto at = [&](int rr, int cc) -> double {
            const size_t a = rev ? n - 1 - rr : rr, b = rev ? n - 1 - cc : cc;
            return t[a * rs + b * cs];
        };
#pragma unroll
        for (int c = 0; c < 16; c++)
            x[c] = at(rc, min(16 * jb + c, n - 1));
        const double dv = at(rc, rc);
#pragma unroll
        for (int c = 0; c < 16; c++)
            x[c] = r < n ? x[c] : 0.0;
        trsm_invert<NB>(x, ((flags & F_UNIT) || r >= n) ? 1.0 : dv, li, smem + jb * TRSM_BLK<NB>);
    }

    // ---- the panel (rows past n: the last row).  A wave without right-hand
    // sides repeats the last panel's and stores nothing.
    const int p0 = (it * 4 + wave) * TRSM_W, w = min(TRSM_W, ncol - p0);
    const int pc = min(p0, (ncol - 1) / TRSM_W * TRSM_W), lic = min(li, ncol - 1 - pc);
    const int nlast = n - 16 * (nb - 1);
    MU_G double *zb = z + (size_t)pc * zcs;
    // row 16 i + 4 e + lk, column lic: a uniform part and this lane's
    const size_t zl = (size_t)(rev ? 3 - lk : lk) * zrs + (size_t)lic * zcs;
    auto zrow = [&](int r) -> size_t {  // of rows r .. r + 3, the lowest address
        return (size_t)(rev ? n - 4 - r : r) * zrs;
    };
    v4d Y[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) {
        Y[i] = v4d{0.0, 0.0, 0.0, 0.0};
        if (i < nb - 1) {
#pragma unroll
            for (int e = 0; e < 4; e++)
                Y[i][e] = (zb + zrow(16 * i + 4 * e))[zl];
        } else if (i == nb - 1) {
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = min(4 * e + lk, nlast - 1) + 16 * i;
                Y[i][e] = zb[(size_t)(rev ? n - 1 - r : r) * zrs + lic * (size_t)zcs];
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NB; i++)
#pragma unroll
        for (int e = 0; e < 4; e++)
            Y[i][e] *= alpha;
    lds_barrier();  // the inverses

    // element (li, 4 e + lk) of a ring block
    int lo[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int r = rev ? 15 - li : li, c = rev ? 15 - 4 * e - lk : 4 * e + lk;
        lo[e] = tt ? r * 16 + (((c >> 1) ^ ((r >> 1) & 7)) << 1) + (c & 1) : c * 16 + r;
    }
    const TrsmFrag<NB> frag(smem, li, lk);
    trsm_columns<NB, 0>(Y, frag, ring, lo, nb, nlast - lk, feed);

    if (li < w)
#pragma unroll
        for (int i = 0; i < NB; i++) {
            if (i < nb - 1) {
#pragma unroll
                for (int e = 0; e < 4; e++)
                    (zb + zrow(16 * i + 4 * e))[zl] = Y[i][e];
            } else if (i == nb - 1) {
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    const int r = 16 * i + 4 * e + lk;
                    if (r < n)
                        zb[(size_t)(rev ? n - 1 - r : r) * zrs + li * (size_t)zcs] = Y[i][e];
                }
            }
        }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // copies past the triangle have landed
}

// ---------------------------------------------------------------------------
// The same solve with one panel of <= 16 right-hand sides on the whole
// workgroup (units flagged F_SPLIT).
//
// What bounds it: the chain over the 16-row blocks.  trsm_panel_reg runs the
// n / 16 (n / 16 + 1) / 2 block products of a panel one after another on one
// wave (order 250: 39 us, 16 of them MFMA issue); here block row i belongs to
// wave i % 4, so a step of the chain is X_j = inv(T_jj) Y_j on its owner, a
// hand-over through LDS with one barrier, and the update of row j + 1; the
// owner of row j + 1 puts off its other rows until X_{j+1} is out.  The
// elements take the same updates in the same order, so the results are those
// of trsm_panel_reg to the bit.  Order 250, one panel: 39 -> 19 us (8.5 us of
// it the chain: 1400 cycles a step, 1000 where a wave has two rows), order 125
// 17 -> 13 us; LU solve n = 12000, 16 right-hand sides, 5.17 -> 3.16 ms.
//
// T is read straight into the MFMA operand by the wave that uses it,
// TRSM_SPLIT_AHEAD columns ahead.  Nothing but the two products, the LDS
// traffic and one barrier is left on the chain: the inverses are in registers,
// and a load's address is a scalar pointer per block row, moved on by one
// scalar addition per column, plus a lane offset fixed for the whole solve
// (with addresses computed block by block a step took 2000 cycles).  Three
// columns ahead, or touching all of T first, measured the same or slower.
// ---------------------------------------------------------------------------
constexpr int TRSM_SPLIT_AHEAD = 2;  // columns of T in registers

template <int NS>
struct TrsmSplit {
    // NS block rows per wave, row 4 k + wave in slot k; block rows nb - 1 ..
    // 4 NS - 1 lie in the last slot
    const MU_G char *t[NS];    // T's block (row of slot k, next column), its lowest address
    unsigned tl[4], tlast[4];  // this lane's byte offset of element e, and in the last slot
    long long step;            // bytes to the next column
    int nb, wave;
    const double *blk;         // the diagonal blocks and their inverses
    v2d *xb;                   // this lane's part of -X_j, two buffers of 256 doubles
    v4d Y[NS], T[TRSM_SPLIT_AHEAD][NS];
    double W[NS][4], D[NS][4];  // the inverse, and the block itself (4 NS blocks at most SMALL_MAX)

    // T's column j into d, slots K0 .. (slots above the diagonal read the
    // other triangle and are never used); then on to column j + 1, which
    // stops at the last column with blocks below it
    template <int K0>
    __device__ __forceinline__ void load(v4d (&d)[NS], int j)
    {
        const long long s = j < nb - 2 ? step : 0;
#pragma unroll
        for (int k = 0; k < NS; k++) {
            if (k >= K0)
#pragma unroll
                for (int e = 0; e < 4; e++)
                    d[k][e] = *(const MU_G double *)(t[k] + (k == NS - 1 ? tlast[e] : tl[e]));
            t[k] += s;
        }
    }
    __device__ __forceinline__ void update(v4d &y, const v4d &tb, const v4d &nx)
    {
#pragma unroll
        for (int e = 0; e < 4; e++)
            y = mfma_f64(tb[e], nx[e], y);
    }
    // X_J on its owner; rows past n (rlast as in trsm_columns) are zero before
    template <int J>
    __device__ __forceinline__ void solve(int rlast)
    {
        v4d &y = Y[J / 4];
        if (J / 4 == NS - 1 && J == nb - 1)
#pragma unroll
            for (int e = 0; e < 4; e++)
                y[e] = 4 * e < rlast ? y[e] : 0.0;
        const v4d x = trsm_diag<4 * NS>(y, W[J / 4], D[J / 4], blk + J * TRSM_BLK<4 * NS>);
        y = x;
        v2d *o = xb + (J & 1) * 128;
        o[0] = v2d{-x[0], -x[1]};
        o[64] = v2d{-x[2], -x[3]};
    }
    // the barrier, with the MFMAs kept on their side of it
    static __device__ __forceinline__ void barrier()
    {
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        __builtin_amdgcn_sched_barrier(0);
    }
    // Steps J ..: every wave sees X_J in its buffer.
    template <int J>
    __device__ __forceinline__ void steps(int rlast)
    {
        if constexpr (J + 1 < 4 * NS) {
            if (J + 1 >= nb)
                return;
            // row J + 1: slot S of wave w
            constexpr int S = (J + 1) / 4, w = (J + 1) & 3, B = J % TRSM_SPLIT_AHEAD;
            const v2d n0 = xb[(J & 1) * 128], n1 = xb[(J & 1) * 128 + 64];
            const v4d nx = {n0[0], n0[1], n1[0], n1[1]};
            if (wave == w) {
                update(Y[S], T[B][S], nx);
                __builtin_amdgcn_sched_barrier(0);
                solve<J + 1>(rlast);
                barrier();
#pragma unroll
                for (int k = S + 1; k < NS; k++)
                    update(Y[k], T[B][k], nx);
            } else {
                if (wave > w)
                    update(Y[S], T[B][S], nx);
#pragma unroll
                for (int k = S + 1; k < NS; k++)
                    update(Y[k], T[B][k], nx);
                barrier();
            }
            if constexpr (J + TRSM_SPLIT_AHEAD < 4 * NS - 1)
                load<(J + TRSM_SPLIT_AHEAD + 1) / 4>(T[B], J + TRSM_SPLIT_AHEAD);
            steps<J + 1>(rlast);
        }
    }
};

template <int NS>
__device__ __attribute__((always_inline)) inline void trsm_panel_split(const UnitDesc &u, int it,
                                                                       double *smem)
{
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = __builtin_amdgcn_readfirstlane(u.m), nb = (n + 15) >> 4;
    const int ncol = __builtin_amdgcn_readfirstlane(u.n);
    const int flags = __builtin_amdgcn_readfirstlane(u.flags);
    const bool rev = flags & F_REV, tt = flags & F_T_TRANS, zr = flags & F_Z_ROWS;
    const unsigned ldt = __builtin_amdgcn_readfirstlane(u.lda);
    const unsigned ldz = __builtin_amdgcn_readfirstlane(u.ldc);
    const MU_G double *t = gp(uniform_ptr(u.a));
    MU_G double *z = gp(uniform_ptr(u.c));
    const double alpha = u.alpha;
    const int nlast = n - 16 * (nb - 1);
    const unsigned rs = tt ? ldt : 1, cs = tt ? 1 : ldt;
    const unsigned zrs = zr ? ldz : 1, zcs = zr ? 1 : ldz;

    TrsmSplit<NS> p;
    p.nb = nb;
    p.wave = wave;
    constexpr int BLK = TRSM_BLK<4 * NS>;
    p.blk = smem;
    p.xb = reinterpret_cast<v2d *>(smem + 4 * NS * BLK) + lane;

    // ---- the diagonal blocks, block wave + 4 lk on this group
    const int jb = min(wave + 4 * lk, nb - 1), r = 16 * jb + li, rc = min(r, n - 1);
    double x[16];
    {
        // rows past n: the last one; columns past n: the last one
        const size_t a = (size_t)(rev ? n - 1 - rc : rc) * rs;
#pragma unroll
        for (int c = 0; c < 16; c++) {
            const int cc = min(16 * jb + c, n - 1);
            x[c] = t[a + (size_t)(rev ? n - 1 - cc : cc) * cs];
        }
    }
    const double dv = t[(size_t)(rev ? n - 1 - rc : rc) * (rs + (size_t)cs)];

    // ---- the panel (rows past n: the last one)
    const int p0 = it * TRSM_W, w = min(TRSM_W, ncol - p0), lic = min(li, w - 1);
    MU_G double *zb = z + (size_t)p0 * zcs;
    auto zat = [&](int row) -> MU_G double * {
        return zb + ((size_t)(rev ? n - 1 - row : row) * zrs + (size_t)lic * zcs);
    };
#pragma unroll
    for (int k = 0; k < NS; k++)
#pragma unroll
        for (int e = 0; e < 4; e++)
            p.Y[k][e] = *zat(min(16 * (4 * k + wave) + 4 * e + lk, n - 1));

    // ---- T's first columns.  With rev a block lies mirrored; in the last
    // block row the rows past n are the last one.
    if (nb > 1) {
        p.step = (rev ? -128 : 128) * (long long)cs;
#pragma unroll
        for (int k = 0; k < NS; k++) {
            const int i = min(4 * k + wave, nb - 1);
            p.t[k] = (const MU_G char *)(t + (size_t)(rev ? max(n - 16 - 16 * i, 0) : 16 * i) * rs +
                                         (size_t)(rev ? n - 16 : 0) * cs);
        }
        const bool last = 4 * (NS - 1) + wave >= nb - 1;
        const unsigned ro = rev ? 15 - li : li;
        const unsigned rl = last ? (rev ? max(nlast - 1 - li, 0) : min(li, nlast - 1)) : ro;
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const unsigned c = rev ? 15 - 4 * e - lk : 4 * e + lk;
            p.tl[e] = 8 * (ro * rs + c * cs);
            p.tlast[e] = 8 * (rl * rs + c * cs);
        }
#pragma unroll
        for (int j = 0; j < TRSM_SPLIT_AHEAD; j++)
            p.template load<0>(p.T[j], j);
    }
    __builtin_amdgcn_sched_barrier(0);

    // ---- the inverses; a wave reads back those of its own rows
#pragma unroll
    for (int c = 0; c < 16; c++)
        x[c] = r < n ? x[c] : 0.0;
    trsm_invert<4 * NS>(x, ((flags & F_UNIT) || r >= n) ? 1.0 : dv, li, smem + jb * BLK);
    const TrsmFrag<4 * NS> frag(smem, li, lk);
    lds_barrier();  // the last block's inverse may have been formed by every wave
#pragma unroll
    for (int k = 0; k < NS; k++) {
        frag.load(min(4 * k + wave, nb - 1), p.W[k], p.D[k]);
#pragma unroll
        for (int e = 0; e < 4; e++)
            p.Y[k][e] *= alpha;
    }

    if (wave == 0)
        p.template solve<0>(nlast - lk);
    p.barrier();
    p.template steps<0>(nlast - lk);

    if (li < w)
#pragma unroll
        for (int k = 0; k < NS; k++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int row = 16 * (4 * k + wave) + 4 * e + lk;
                if (row < n)
                    *zat(row) = p.Y[k][e];
            }
}

constexpr int LDS_TRSM_REG = 16 * BF_BLK + TRSM_RING<16> * 1024;       // inverses of order TRSM_REG_MAX
constexpr int LDS_TRSM_REG_SMALL = 8 * TRSM_BLK<8> + TRSM_RING<8> * 1024;  // ... of order SMALL_MAX

// TRSM item of a triangle of order <= TRSM_REG_MAX; MAXNB: the most 16-blocks
// the caller's LDS holds inverses for (8 or 16).  The block count is rounded
// up to an instance (a block past the triangle costs its MFMAs).
template <int MAXNB>
__device__ __attribute__((always_inline)) inline void run_trsm_reg_item(const UnitDesc &u, int it,
                                                                        double *smem)
{
    const int nb = (__builtin_amdgcn_readfirstlane(u.m) + 15) >> 4;
    if (__builtin_amdgcn_readfirstlane(u.flags) & F_SPLIT) {
        if (nb <= 4)
            trsm_panel_split<1>(u, it, smem);
        else if (MAXNB == 8 || nb <= 8)
            trsm_panel_split<2>(u, it, smem);
        else if (nb <= 12)
            trsm_panel_split<MAXNB == 8 ? 2 : 3>(u, it, smem);
        else
            trsm_panel_split<MAXNB == 8 ? 2 : 4>(u, it, smem);
        return;
    }
    if (nb <= 2)
        trsm_panel_reg<2>(u, it, smem);
    else if (nb <= 4)
        trsm_panel_reg<4>(u, it, smem);
    else if (nb <= 6)
        trsm_panel_reg<6>(u, it, smem);
    else if (MAXNB == 8 || nb <= 8)
        trsm_panel_reg<8>(u, it, smem);
    else if (nb <= 12)
        trsm_panel_reg<MAXNB == 8 ? 8 : 12>(u, it, smem);
    else
        trsm_panel_reg<MAXNB == 8 ? 8 : 16>(u, it, smem);
}

// LDS (doubles) one workgroup needs for any item.
constexpr int LDS_GEMM = LDS_GEMM_DMA;
static_assert(2 * (LDS_I > LDS_K ? LDS_I : LDS_K) * 2 <= LDS_GEMM, "gemm_block: 2 operands x 2 buffers");
constexpr int LDS_NARROW = 4 * 4 * 4 * 64 / 2 + 1;  // the narrow GEMMs' partial tiles and a flag
constexpr int LDS_TRSM = TRSM_NMAX * 16;
constexpr int LDS_SMALL = LDS_SMALL_BLK;
static_assert(TRINV_BLOCKS * 16 * 17 <= LDS_TRSM, "TRINV staging fits the generic LDS");
static_assert(TRINV_BLOCKS * 16 == WG_THREADS, "TRINV: one thread per block column");
static_assert(4 * GEMM_BM * 20 * 2 <= LDS_GEMM * 8 && 4 * GEMM_BM * 17 * 4 <= LDS_GEMM * 8,
              "reduced-precision GEMM buffers fit the GEMM LDS");
constexpr int LDS_DOUBLES = LDS_GEMM > LDS_TRSM ? (LDS_GEMM > LDS_SMALL ? LDS_GEMM : LDS_SMALL)
                                                : (LDS_TRSM > LDS_SMALL ? LDS_TRSM : LDS_SMALL);

// Order of the output blocks of one GEMM/SYRK unit.  Consecutive items run
// at the same time (and round-robin over the XCDs), so they should share
// operand strips: items walk groups of BLOCK_GROUP block rows column by
// column, rows fastest inside a group.  A group's A strips (32 x 64 rows x K)
// stay in L2 while its columns go by, and each B strip is read by the group's
// 32 blocks in a row.  A unit of at most BLOCK_GROUP block rows (one tile
// GEMM) is plain column-major.  Measured on the merged LU trailing update
// (22000 x 22000 x 1000): 55.9 TFLOP/s column-major, 58.6 with groups of 32.
constexpr int BLOCK_GROUP = 32;

// GEMM item i of a gm x gn block grid -> (bi, bj).
__device__ __forceinline__ void gemm_block_order(int gm, int gn, int i, int &bi, int &bj)
{
    const int per = BLOCK_GROUP * gn, first = (i / per) * BLOCK_GROUP;
    const int gsz = min(gm - first, BLOCK_GROUP), local = i - (first / BLOCK_GROUP) * per;
    bi = first + local % gsz;
    bj = local / gsz;
}

// SYRK item i -> (bi, bj), bi >= bj, over the lower blocks of a g x g grid:
// groups of BLOCK_GROUP block rows; inside a group the columns left of it
// (full height) and then its own lower triangle, column by column.
__device__ __forceinline__ void syrk_block(int g, int i, int &bi, int &bj)
{
    int r0 = 0;
    for (;;) {
        const int gsz = min(g - r0, BLOCK_GROUP);
        const int count = r0 * gsz + gsz * (gsz + 1) / 2;
        if (i < count || r0 + gsz >= g) {
            if (i < r0 * gsz) {
                bj = i / gsz;
                bi = r0 + i % gsz;
                return;
            }
            i -= r0 * gsz;
            int c = 0;
            while (i >= gsz - c) {
                i -= gsz - c;
                c++;
            }
            bj = r0 + c;
            bi = r0 + c + i;
            return;
        }
        i -= count;
        r0 += gsz;
    }
}

template <bool TA, bool TB>
__device__ __forceinline__ void gemm_dispatch_vec(const UnitDesc &u, int bi, int bj, bool lo,
                                                  double *smem)
{
    if (u.flags & (F_LOW_F32 | F_LOW_BF16)) {
#define MU_LOW_CASE(P, SRC)                                               \
    if (u.flags & F_VEC)                                                  \
        gemm_block_low<TA, TB, true, P, SRC>(u, bi, bj, lo, smem);        \
    else                                                                  \
        gemm_block_low<TA, TB, false, P, SRC>(u, bi, bj, lo, smem);
        const bool src = (u.flags & F_SRC_LOW) != 0;
        if (u.flags & F_LOW_F32) {
            if (src) {
                MU_LOW_CASE(1, true)
            } else {
                MU_LOW_CASE(1, false)
            }
        } else {
            if (src) {
                MU_LOW_CASE(2, true)
            } else {
                MU_LOW_CASE(2, false)
            }
        }
#undef MU_LOW_CASE
    } else if (gemm_dma_ok(u)) {
        gemm_block_dma<TA, TB>(u, bi, bj, lo, smem);
    } else {
        if (u.flags & F_VEC)
            gemm_block<TA, TB, true>(u, bi, bj, lo, smem);
        else
            gemm_block<TA, TB, false>(u, bi, bj, lo, smem);
    }
}

// GEMM or SYRK item `it` of unit `u` (the only kinds k_batch_gemm runs).
// ---------------------------------------------------------------------------
// GEMM block for narrow outputs (units flagged F_NARROW: n <= 16 columns, the
// right-hand sides of a substitution step; FP64, op(B) = B).  An item is one
// 16-row tile x all n columns, so a level of these (one 1000-row step is 63
// items) spreads over many CUs.  The 4 waves split K (k-chunks of 32 taken
// round-robin) and read the MFMA fragments straight from global memory --
// lane (li, lk) supplies op(A)[row li][k + lk] and B[k + lk][col li] -- with
// the next chunk's loads issued before the current chunk's MFMAs; the four
// partial tiles are added through LDS.  A 64 x 64 block would spend 3/4 of
// its MFMAs on absent columns and leave most CUs idle.
// ---------------------------------------------------------------------------
constexpr int NARROW_ROWS = 16;  // output rows per narrow item

template <bool TA>
__device__ __attribute__((always_inline)) inline void gemm_narrow(const UnitDesc &u, int bi,
                                                                  double *smem)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int i0 = bi * NARROW_ROWS, K = u.k, ncol = u.n;
    const MU_G double *a = gp(u.a);
    const MU_G double *b = gp(u.b);
    const size_t lda = u.lda, ldb = u.ldb;
    const bool cok = li < ncol;
    // Every load is issued unconditionally from an address clamped into the
    // operand (a lane's row and column clamped, k clamped to K - 1), so no
    // branch separates a load from the others in flight and the wait before
    // a chunk's MFMAs covers only that chunk's loads.  Rows and columns past
    // the block are computed but never stored; the k-steps past K are zeroed
    // in both operands as they enter the MFMA.
    const MU_G double *bc = b + (size_t)min(li, ncol - 1) * ldb;
    const int rc = min(i0 + li, u.m - 1);
    const MU_G double *ar = TA ? a + (size_t)rc * lda : a + rc;
    v4d acc = {0.0, 0.0, 0.0, 0.0};
    constexpr int KU = 8;  // k-steps of 4 per chunk
    double fa[2][KU], fb[2][KU];
    auto load = [&](double (&ga)[KU], double (&gb)[KU], int k) {
#pragma unroll
        for (int q = 0; q < KU; q++) {
            const int kc = min(k + 4 * q + lk, K - 1);
            gb[q] = bc[kc];
            ga[q] = TA ? ar[kc] : ar[(size_t)kc * lda];
        }
    };
    auto mma = [&](const double (&ga)[KU], const double (&gb)[KU], int k) {
#pragma unroll
        for (int q = 0; q < KU; q++) {
            const bool kok = k + 4 * q + lk < K;
            acc = mfma_f64(kok ? ga[q] : 0.0, kok ? gb[q] : 0.0, acc);
        }
    };
    constexpr int CH = 4 * KU;  // k per chunk
    int k = wave * CH;
    if (K > 0 && k < K) {
        load(fa[0], fb[0], k);
        for (;;) {
            const int kn = k + 4 * CH;
            if (kn < K) {
                load(fa[1], fb[1], kn);
                mma(fa[0], fb[0], k);
            } else {
                mma(fa[0], fb[0], k);
                break;
            }
            const int kn2 = kn + 4 * CH;
            if (kn2 < K) {
                load(fa[0], fb[0], kn2);
                mma(fa[1], fb[1], kn);
            } else {
                mma(fa[1], fb[1], kn);
                break;
            }
            k = kn2;
        }
    }
    // waves 1..3 hand their partial tiles to wave 0: LDS slot [wave - 1][e][lane]
    if (wave > 0)
#pragma unroll
        for (int e = 0; e < 4; e++)
            smem[((wave - 1) * 4 + e) * 64 + lane] = acc[e];
    lds_barrier();
    if (wave != 0)
        return;
    const double alpha = u.alpha, beta = u.beta;
    MU_G double *c = gp(u.c);
#pragma unroll
    for (int e = 0; e < 4; e++) {
        // acc[e] = D[4e + lk][li]: row i0 + 4e + lk, column li
        const int row = i0 + 4 * e + lk;
        const double v = acc[e] + (smem[e * 64 + lane] + smem[(4 + e) * 64 + lane] +
                                   smem[(8 + e) * 64 + lane]);
        if (row < u.m && cok) {
            MU_G double *cp = c + row + (size_t)li * u.ldc;
            *cp = (beta != 0.0 ? beta * *cp : 0.0) + alpha * v;
        }
    }
}
static_assert(3 * 4 * 64 <= LDS_NARROW, "narrow GEMM reduction fits");

// ---------------------------------------------------------------------------
// Narrow GEMM with an FP32 A (F_NARROW | F_A32): C = beta C + alpha A B for
// A m x k stored FP32 (column-major, lda in elements), B k x n FP64 (n <= 16)
// and C FP64 -- a substitution step of a refinement solve on FP32 copies of
// the factors, where A is the whole traffic.  An item is 64 output rows x
// every column x one k-slice of NARROW32_KSLICE (u.gn slices): short slices
// put many items in flight at once, so a step costs a few memory round
// trips instead of one per 128 k.  Lane (li, lk) owns rows 4 li .. 4 li + 3
// of the item: per k-step of 4 it loads one float4 of A (16 lanes cover 256
// contiguous bytes of a column, 4 columns per instruction) and one element
// B[k + lk][li], rounded to FP32.  Row e of the lane's group feeds MFMA e
// (v_mfma_f32_16x16x4f32), whose output row index li stands for item row
// 4 li + e.  The 4 waves split the slice in chunks of 32 taken round-robin
// (loads of the next chunk in flight over the current chunk's MFMAs); the
// partial tiles meet in LDS and each wave finishes 16 of the 64 rows.  One
// slice: the FP32 sums are added into C in FP64.  Several: each item stores
// its 64 x 16 partial tile, and the item that finds itself last of its row
// block on the block's arrival counter adds the slices' tiles in slice order
// (FP64; the same order whatever the arrival order, so results do not
// depend on scheduling), updates C and resets the counter.  VEC: a 16-byte
// aligned, lda and m multiples of 4.
// ---------------------------------------------------------------------------
constexpr int NARROW32_ROWS = 64;  // output rows per FP32-A narrow item

template <bool VEC>
__device__ __attribute__((always_inline)) inline void gemm_narrow_a32(const UnitDesc &u, int it,
                                                                      double *smem)
{
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int li = lane & 15, lk = lane >> 4;
    const int bi = it % u.gm, sl = it / u.gm, ns = u.gn;
    const int i0 = bi * NARROW32_ROWS, m = u.m, ncol = u.n;
    // this item's k range [k0, K): all of k when the unit is not split
    const int k0 = sl * NARROW32_KSLICE, K = ns == 1 ? u.k : min(u.k, k0 + NARROW32_KSLICE);
    const MU_G float *a = (const MU_G float *)u.a;
    const MU_G double *b = gp(u.b);
    const size_t lda = u.lda, ldb = u.ldb;
    const bool cok = li < ncol;
    // B(k, j) at b[k sk + j sj], C(i, j) at c[i ci + j cj]: columns, or rows
    // with F_BROW (a k-step of the 16 x 4 B fragment is then 512 contiguous
    // bytes instead of 16 columns' 32)
    const bool brow = (u.flags & F_BROW) != 0;
    const size_t sk = brow ? ldb : 1, sj = brow ? 1 : ldb;
    const size_t ci = brow ? (size_t)u.ldc : 1, cj = brow ? 1 : (size_t)u.ldc;
    // loads unconditional from clamped addresses, the k-steps past the
    // slice zeroed as they enter the MFMA (as in gemm_narrow)
    const MU_G double *bc = b + (size_t)min(li, ncol - 1) * sj;
    const int r0 = i0 + 4 * li;  // this lane's rows r0 .. r0 + 3
    // VEC: m % 4 == 0, so the lane's 4 rows are all inside or all outside
    const int r0c = min(r0, m - 4);
    v4f acc[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
        acc[e] = v4f{0.f, 0.f, 0.f, 0.f};
    constexpr int KU = 8;  // k-steps of 4 per chunk
    v4f fa[2][KU];
    double fb[2][KU];
    auto load = [&](v4f (&ga)[KU], double (&gb)[KU], int k) {
#pragma unroll
        for (int q = 0; q < KU; q++) {
            const int kc = min(k + 4 * q + lk, K - 1);
            gb[q] = bc[(size_t)kc * sk];
            if (VEC) {
                ga[q] = *(const MU_G v4f *)(a + r0c + (size_t)kc * lda);
            } else {
                const MU_G float *ac = a + (size_t)kc * lda;
                ga[q] = v4f{ac[min(r0, m - 1)], ac[min(r0 + 1, m - 1)], ac[min(r0 + 2, m - 1)],
                            ac[min(r0 + 3, m - 1)]};
            }
        }
    };
    auto mma = [&](const v4f (&ga)[KU], const double (&gb)[KU], int k) {
#pragma unroll
        for (int q = 0; q < KU; q++) {
            const bool kok = k + 4 * q + lk < K;
            const float bv = kok ? (float)gb[q] : 0.f;
            const v4f av = kok ? ga[q] : v4f{0.f, 0.f, 0.f, 0.f};
            acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, bv, acc[0], 0, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, bv, acc[1], 0, 0, 0);
            acc[2] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.z, bv, acc[2], 0, 0, 0);
            acc[3] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.w, bv, acc[3], 0, 0, 0);
        }
    };
    constexpr int CH = 4 * KU;  // k per chunk
    int k = k0 + wave * CH;
    if (k < K) {
        load(fa[0], fb[0], k);
        for (;;) {
            const int kn = k + 4 * CH;
            if (kn < K) {
                load(fa[1], fb[1], kn);
                mma(fa[0], fb[0], k);
            } else {
                mma(fa[0], fb[0], k);
                break;
            }
            const int kn2 = kn + 4 * CH;
            if (kn2 < K) {
                load(fa[0], fb[0], kn2);
                mma(fa[1], fb[1], kn);
            } else {
                mma(fa[1], fb[1], kn);
                break;
            }
            k = kn2;
        }
    }
    // partial tiles to LDS: slot [wave][e][e'][lane], acc[e][e'] = D_e[4 lk + e'][li],
    // item row 4 (4 lk + e') + e, column li
    float *sm = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
        for (int f = 0; f < 4; f++)
            sm[((wave * 4 + e) * 4 + f) * 64 + lane] = acc[e][f];
    lds_barrier();
    // wave w finishes e' = w: rows 16 lk + 4 w + e (e = 0..3) of column li
    float s[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        s[e] = 0.f;
#pragma unroll
        for (int w = 0; w < 4; w++)
            s[e] += sm[((w * 4 + e) * 4 + wave) * 64 + lane];
    }
    const double alpha = u.alpha, beta = u.beta;
    MU_G double *c = gp(u.c);
    const int rb = i0 + 16 * lk + 4 * wave;
    auto store = [&](const double (&v)[4]) {
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int row = rb + e;
            if (row < m && cok) {
                MU_G double *cp = c + (size_t)row * ci + (size_t)li * cj;
                *cp = (beta != 0.0 ? beta * *cp : 0.0) + alpha * v[e];
            }
        }
    };
    if (ns == 1) {
        const double v[4] = {s[0], s[1], s[2], s[3]};
        store(v);
        return;
    }
    // several slices: publish this slice's tile, count the arrival
    MU_G float *part = gp(u.part);
    int32_t *cnt = reinterpret_cast<int32_t *>(u.part + (size_t)u.gm * ns * 1024) + bi;
#pragma unroll
    for (int e = 0; e < 4; e++)
        part[((size_t)bi * ns + sl) * 1024 + (wave * 4 + e) * 64 + lane] = s[e];
    // each wave waits for its stores to reach L2 and the barrier puts all of
    // them before thread 0's agent-scope release (one L2 write-back per
    // item) and count; the last arrival's acquire (one L2 invalidation per
    // row block) and the barrier after it come before every wave's loads
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int *flag = reinterpret_cast<int *>(sm + 4 * 4 * 4 * 64);
    if (threadIdx.x == 0) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        const int old = __hip_atomic_fetch_add(cnt, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (old == ns - 1)
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        *flag = old;
    }
    __syncthreads();
    if (*flag != ns - 1)
        return;
    double v[4] = {0.0, 0.0, 0.0, 0.0};
    for (int q = 0; q < ns; q++)
#pragma unroll
        for (int e = 0; e < 4; e++)
            v[e] += (double)part[((size_t)bi * ns + q) * 1024 + (wave * 4 + e) * 64 + lane];
    store(v);
    if (threadIdx.x == 0)
        __hip_atomic_store(cnt, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
static_assert(4 * 4 * 4 * 64 + 1 <= 2 * LDS_NARROW && LDS_NARROW <= LDS_GEMM,
              "FP32-A narrow reduction fits");

// Narrow GEMM item (F_NARROW units only; kept out of run_gemm_item so the
// 64 x 64 block kernels keep their register budget).
__device__ __attribute__((always_inline)) inline void run_gemm_narrow_item(const UnitDesc &u,
                                                                           int it, double *smem)
{
    if (u.flags & F_A32) {
        if (u.flags & F_VEC)
            gemm_narrow_a32<true>(u, it, smem);
        else
            gemm_narrow_a32<false>(u, it, smem);
        return;
    }
    if (u.flags & F_TA)
        gemm_narrow<true>(u, it, smem);
    else
        gemm_narrow<false>(u, it, smem);
}

// One GEMM output block of a unit without F_NARROW, any transposition.
__device__ __attribute__((always_inline)) inline void gemm_any_block(const UnitDesc &u, int bi,
                                                                     int bj, double *smem)
{
    switch (u.flags & (F_TA | F_TB)) {
    case 0: gemm_dispatch_vec<false, false>(u, bi, bj, false, smem); break;
    case F_TB: gemm_dispatch_vec<false, true>(u, bi, bj, false, smem); break;
    case F_TA: gemm_dispatch_vec<true, false>(u, bi, bj, false, smem); break;
    default: gemm_dispatch_vec<true, true>(u, bi, bj, false, smem); break;
    }
}

// GEMM/SYRK item of a unit without F_NARROW.  GROUPED: the unit's items
// cover grp x grp output blocks (the persistent kernel's lowering); the
// level kernels run one block per item and keep the single-block form.
template <bool GROUPED = false>
__device__ __attribute__((always_inline)) inline void run_gemm_item(const UnitDesc &u, int it,
                                                                    double *smem)
{
    if (u.op == OP_SYRK) {
        int bi, bj;
        syrk_block(u.gm, it, bi, bj);
        // A A^T: A read directly (op(B) = A^T), or, for a reduced-precision
        // panel stored transposed, A^T read as op(A) = (A^T)^T
        if (u.flags & F_TA)
            gemm_dispatch_vec<true, false>(u, bi, bj, bi == bj, smem);
        else
            gemm_dispatch_vec<false, true>(u, bi, bj, bi == bj, smem);
        return;
    }
    if (!GROUPED || u.grp <= 1) {
        int bi, bj;
        gemm_block_order(u.gm, u.gn, it, bi, bj);
        gemm_any_block(u, bi, bj, smem);
        return;
    }
    // g x g output blocks one after the other, a barrier between them (the
    // next block's staging overwrites the LDS the previous one read last)
    const int g = u.grp;
    const int gm = (u.gm + g - 1) / g;
    const int bi0 = (it % gm) * g, bj0 = (it / gm) * g;
#pragma unroll 1
    for (int q = 0; q < g * g; q++) {
        const int bi = bi0 + q % g, bj = bj0 + q / g;
        if (bi >= u.gm || bj >= u.gn)
            continue;
        if (q)
            lds_barrier();
        gemm_any_block(u, bi, bj, smem);
    }
}

// GEMM or SYRK item of a unit flagged F_KVEC | F_BLK128 (k_batch_gemm_low;
// the graph builder gives every unit of that kernel 128 x 128 blocks).
__device__ __attribute__((always_inline)) inline void run_gemm_lowk_item(const UnitDesc &u, int it,
                                                                         double *smem)
{
    int bi, bj;
    bool lo = false;
    if (u.op == OP_SYRK) {
        syrk_block(u.gm, it, bi, bj);
        lo = bi == bj;
    } else {
        gemm_block_order(u.gm, u.gn, it, bi, bj);
    }
    if (u.flags & F_LOW_BF16)
        gemm_block_lowk128<2>(u, bi, bj, lo, smem);
    else
        gemm_block_lowk128<1>(u, bi, bj, lo, smem);
}

// FP64 block -> FP32 / BF16 storage: item = one 64 x 64 block of the m x n
// source (c, ldc), written to (b, ldb).
// F_CVT_T: the block is written transposed (element (r, c) at b[c + r*ldb]).
// Each wave turns its own 64 x 16 column slice around through LDS (its own
// 16 x 65 patch, no workgroup barrier): it reads the FP64 columns (a wave
// reads 64 consecutive rows), and writes rows of 16 consecutive output
// elements.
template <class T>
__device__ __forceinline__ void cvt_block_t(const UnitDesc &u, int i0, int j0, double *smem)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    T *tl = reinterpret_cast<T *>(smem) + w * 16 * 65;  // [column][row], pitch 65
    const MU_G double *src = gp(u.c);
    const int r = i0 + lane;
    const bool both = (u.flags & F_CVT_BOTH) != 0;
    MU_G T *plain = (MU_G T *)u.a;
#pragma unroll
    for (int c = 0; c < 16; c++) {
        const int cc = j0 + 16 * w + c;
        const bool in = r < u.m && cc < u.n;
        const double v = in ? src[r + (size_t)cc * u.ldc] : 0.0;
        const T cvv = LowPrec<sizeof(T) == 2 ? 2 : 1>::cv(v);
        tl[c * 65 + lane] = cvv;
        if (both && in)
            plain[r + (size_t)cc * u.lda] = cvv;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    MU_G T *dst = (MU_G T *)u.b;
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int rr = 4 * q + (lane >> 4), c = lane & 15;
        const int gr = i0 + rr, gc = j0 + 16 * w + c;
        if (gr < u.m && gc < u.n)
            dst[gc + (size_t)gr * u.ldb] = tl[c * 65 + rr];
    }
}

__device__ __attribute__((always_inline)) inline void cvt_block(const UnitDesc &u, int it,
                                                                double *smem)
{
    const int bi = it % u.gm, bj = it / u.gm;
    const int i0 = bi * 64, j0 = bj * 64;
    if (u.flags & F_CVT_T) {
        if (u.flags & F_LOW_BF16)
            cvt_block_t<unsigned short>(u, i0, j0, smem);
        else
            cvt_block_t<float>(u, i0, j0, smem);
        return;
    }
    const MU_G double *src = gp(u.c);
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const int idx = threadIdx.x + WG_THREADS * q, r = i0 + (idx & 63), c = j0 + (idx >> 6);
        if (r < u.m && c < u.n) {
            const double v = src[r + (size_t)c * u.ldc];
            if (u.flags & F_LOW_BF16)
                ((MU_G unsigned short *)u.b)[r + (size_t)c * u.ldb] = to_bf16(v);
            else
                ((MU_G float *)u.b)[r + (size_t)c * u.ldb] = (float)v;
        }
    }
}

// TRSM item with inverted diagonal blocks on NW waves (k_batch_trsm,
// k_batch_trsm_512).
template <int NW, int NMAX = TRSM_NMAX>
__device__ __attribute__((always_inline)) inline void run_trsm_inv_item(const UnitDesc &u, int it,
                                                                        double *smem)
{
    switch ((u.flags >> 3) & 0x27) {  // T_TRANS, Z_ROWS, UNIT, REV
#define MU_TRSM_INV_CASE(bits)                                                                 \
    case bits:                                                                                 \
        trsm_panel_inv<(bits & 1) != 0, (bits & 2) != 0, (bits & 4) != 0, (bits & 0x20) != 0, \
                       NW, NMAX>(u, it, smem);                                                 \
        break;
        MU_TRSM_INV_CASE(0x00) MU_TRSM_INV_CASE(0x01) MU_TRSM_INV_CASE(0x02) MU_TRSM_INV_CASE(0x03)
        MU_TRSM_INV_CASE(0x04) MU_TRSM_INV_CASE(0x05) MU_TRSM_INV_CASE(0x06) MU_TRSM_INV_CASE(0x07)
        MU_TRSM_INV_CASE(0x20) MU_TRSM_INV_CASE(0x21) MU_TRSM_INV_CASE(0x22) MU_TRSM_INV_CASE(0x23)
        MU_TRSM_INV_CASE(0x24) MU_TRSM_INV_CASE(0x25) MU_TRSM_INV_CASE(0x26) MU_TRSM_INV_CASE(0x27)
#undef MU_TRSM_INV_CASE
    default: break;
    }
}

// TRINV item (inverses of TRINV_BLOCKS diagonal blocks).
__device__ __attribute__((always_inline)) inline void run_trinv_item(const UnitDesc &u, int it,
                                                                     double *smem)
{
    switch ((u.flags >> 3) & 0x25) {  // T_TRANS, UNIT, REV
    case 0x00: trinv_blocks<false, false, false>(u, it, smem); break;
    case 0x01: trinv_blocks<true, false, false>(u, it, smem); break;
    case 0x04: trinv_blocks<false, true, false>(u, it, smem); break;
    case 0x05: trinv_blocks<true, true, false>(u, it, smem); break;
    case 0x20: trinv_blocks<false, false, true>(u, it, smem); break;
    case 0x21: trinv_blocks<true, false, true>(u, it, smem); break;
    case 0x24: trinv_blocks<false, true, true>(u, it, smem); break;
    default: trinv_blocks<true, true, true>(u, it, smem); break;
    }
}

// Small GETRF/POTRF or CVT item (the only kinds k_batch_small runs).
__device__ __attribute__((always_inline)) inline void run_small_item(const UnitDesc &u, int it,
                                                                     double *smem)
{
    if (u.op == OP_GETRF)
        getrf_small(u, smem);
    else if (u.op == OP_POTRF)
        potrf_small(u, smem);
    else
        cvt_block(u, it, smem);
}

// This workgroup's unit and item of a graph node.  The table's pointers come
// in a structure, where the compiler does not see that they point to global
// memory nothing writes: said here, the descriptor stays in scalar registers
// (as flat loads it took 20 vector registers of every kernel).
__device__ __forceinline__ UnitDesc node_unit(const NodeArgs &node, int &it)
{
    typedef unsigned v4u __attribute__((ext_vector_type(4)));
    typedef unsigned v2u __attribute__((ext_vector_type(2)));
    struct Words {
        v4u w[sizeof(UnitDesc) / 16];
    } w;
    static_assert(sizeof(NodeItem) == sizeof(v2u) && sizeof(Words) == sizeof(UnitDesc), "");
    if (!node.items) {
        it = (int)blockIdx.x;
        return node.one;
    }
    const v2u r = ((const MU_C v2u *)node.items)[blockIdx.x];
    it = (int)r[1];
    const MU_C v4u *p = (const MU_C v4u *)(node.units + r[0]);
#pragma unroll
    for (int i = 0; i < (int)(sizeof(UnitDesc) / 16); i++)
        w.w[i] = p[i];
    return __builtin_bit_cast(UnitDesc, w);
}

// Execute local item `it` of unit `u`.  Always inlined, so that LDS stays
// addressed as LDS and no call stack is needed in the persistent kernel.
__device__ __attribute__((always_inline)) inline void run_item(const UnitDesc &u, int it,
                                                               double *smem)
{
    switch (u.op) {
    case OP_GEMM:
        if (u.flags & F_NARROW)
            run_gemm_narrow_item(u, it, smem);
        else
            run_gemm_item(u, it, smem);
        break;
    case OP_SYRK: run_gemm_item(u, it, smem); break;
    case OP_TRSM:
        if (u.flags & F_INV)
            run_trsm_inv_item<4>(u, it, smem);
        else
            run_trsm_reg_item<16>(u, it, smem);
        break;
    case OP_GETRF: getrf_small(u, smem); break;
    case OP_POTRF: potrf_small(u, smem); break;
    case OP_CVT: cvt_block(u, it, smem); break;
    case OP_TRINV: run_trinv_item(u, it, smem); break;
    default: break;
    }
}

}  // namespace mu
