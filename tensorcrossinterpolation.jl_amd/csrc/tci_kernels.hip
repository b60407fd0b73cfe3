// tci_kernels.hip — gfx950 kernels beside the solves (tci_solve.hip)
// and the on-chip rrLU (tci_rrlu_chip.hip), and the launches of the solves.
//
//   tci_rrlu_kernel      one workgroup = one rrlu!(A) (matrixlu.jl:194-204),
//                        a batch of uneven matrices in one launch
//   tci_lu_unpack_kernel L = tril(A[:,1:p]), U = triu(A[1:p,:]) with the unit
//                        diagonal (matrixlu.jl:162-174)
//   tci_kron_center_kernel / tci_eval_kernel
//                        Pi-tensor evaluation (batcheval.jl:32-61)
//
// Workgroups are 256 threads = 4 wave64s.  Team reductions: DPP/shuffle
// within a wave, then one LDS slot per wave read back by every thread, so a
// reduction costs one barrier.  Compiled with -ffp-contract=off.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "tci_devteam.h"
#include "tci_engine.h"
#include "tci_kernels.h"
#include "tci_solve.h"

namespace tci {

constexpr int kTeam = 256;

// ---------------------------------------------------------------- solves
static const void *serve_kernel_ptr(int team) { return team == 512 ? serve_kernel_512() : serve_kernel_256(); }

int serve_static_lds(int team)
{
    hipFuncAttributes a;
    if (hipFuncGetAttributes(&a, serve_kernel_ptr(team)) != hipSuccess) return -1;
    return (int)a.sharedSizeBytes;
}

hipError_t launch_serve(const ServeSlot *ring, ServeDev *g, const ServeCtl *ctl, uint64_t *done, int cap,
                        const LdsPlan &plan, uint64_t idle_ticks, uint32_t epoch, int team, int blocks,
                        hipStream_t st)
{
    const size_t lds = lds_plan_bytes(plan);
    int lds_blk = 0, dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&lds_blk, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e != hipSuccess) return e;
    const int stat = serve_static_lds(team);
    if (stat < 0 || (size_t)stat + lds > (size_t)lds_blk) return hipErrorInvalidValue;
    const void *k = serve_kernel_ptr(team);
    if ((e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) != hipSuccess) return e;
    LdsPlan p = plan;
    void *args[] = {&ring, &g, &ctl, &done, &cap, &p, &idle_ticks, &epoch};
    if ((e = hipLaunchKernel(k, dim3(blocks), dim3(team == 512 ? 512 : 256), args, lds, st)) != hipSuccess) return e;
    return hipGetLastError();
}

// ------------------------------------------------------- packed results
// at: 5 byte offsets per (solve, site): the tensor, then Iset, Jset and their
// last history entries
__global__ __launch_bounds__(256) void tci_pack_kernel(const SolveDesc *__restrict__ descs,
                                                       const int32_t *__restrict__ solve, int L0,
                                                       const int64_t *__restrict__ at, uint8_t *__restrict__ out)
{
    const int q = blockIdx.x / L0, b = blockIdx.x - q * L0;
    const SolveDesc &D = descs[solve[q]];
    const int L = D.L;
    if (b >= L) return;
    const int64_t *o = at + 5 * ((int64_t)q * L0 + b);
    const int64_t n = D.Tdims[3 * b] * D.Tdims[3 * b + 1] * D.Tdims[3 * b + 2];
    const double *T = D.T + D.tstride * b;
    double *dst = (double *)(out + o[0]);
    for (int64_t e = threadIdx.x; e < n; e += blockDim.x) dst[e] = T[e];
    const int hist = D.ints[INT_HIST];
    for (int w = 0; w < 4; ++w) {
        const bool jside = w & 1;
        if (w >= 2 && hist == 0) break;
        const int kind = w < 2 ? (jside ? SET_J : SET_I)
                               : (hist == 2 ? (jside ? SET_HB_J : SET_HB_I) : (jside ? SET_HA_J : SET_HA_I));
        const int len = jside ? L - 1 - b : b, cnt = D.setn[kind * L + b];
        const uint8_t *src = D.sets + ((int64_t)(kind * L + b) * D.setcap) * L;
        uint8_t *d = out + o[1 + w];
        for (int e = threadIdx.x; e < cnt * len; e += blockDim.x) {
            const int r = e / len, t = e - r * len;
            d[e] = src[(int64_t)r * L + t];
        }
    }
}

hipError_t launch_pack(const SolveDesc *descs, const int32_t *solve, int count, int L0, const int64_t *at,
                       uint8_t *out, hipStream_t st)
{
    if (count < 1) return hipSuccess;
    hipLaunchKernelGGL(tci_pack_kernel, dim3((unsigned)(count * L0)), dim3(256), 0, st, descs, solve, L0, at, out);
    return hipGetLastError();
}

// ------------------------------------------------------------------ rrLU
// order: the job each workgroup takes (largest first, so the long
// factorizations start early and the launch ends evenly), or null
__global__ __launch_bounds__(kTeam) void tci_rrlu_kernel(tci_lu_job *__restrict__ jobs,
                                                         int64_t count, int lds_stage_cap,
                                                         double *__restrict__ gstage,
                                                         int64_t gstage_stride,
                                                         const int32_t *__restrict__ order)
{
    if ((int64_t)blockIdx.x >= count) return;
    const int64_t s = order ? (int64_t)order[blockIdx.x] : (int64_t)blockIdx.x;
    extern __shared__ double stage[];
    tci_lu_job &J = jobs[s];
    const int m = (int)J.m, n = (int)J.n;
    const int mx = m > n ? m : n;
    DevTeam<kTeam> tm;
    if (mx <= lds_stage_cap) tm.init(stage, stage + mx);
    else tm.init(gstage + gstage_stride * s, gstage + gstage_stride * s + mx);
    double err, st[2];
    // the streaming factorization: the packed factors are the output
    const int p = rrlu_team(tm, J.A, m, n, J.maxrank, J.reltol, J.abstol, J.leftorth != 0,
                            J.rowperm, J.colperm, nullptr, &err, st);
    // 1-based permutations (rrLU.rowpermutation / colpermutation)
    for (int i = tm.tid(); i < m; i += kTeam) J.rowperm[i] += 1;
    for (int j = tm.tid(); j < n; j += kTeam) J.colperm[j] += 1;
    if (tm.tid() == 0) {
        J.status = p < 0 ? -p : 0;
        J.npivot = p < 0 ? 0 : p;
        J.error = err;
    }
}

// The register-tile factorization of one job (tci_regtile.h) with tile shape
// T, then rrlu!'s packed output written to J.A: the L columns (recorded by
// original row in Lsc, m × mr) and U rows (by original column in Usc,
// mr × n) placed at their final positions, the pivots on the diagonal and
// the trailing block from the registers.
template <class T, class Team>
__device__ void tile_job(Team &tm, tci_lu_job &J, int m, int n, double *Lsc, double *Usc, double *pv)
{
    int64_t mr = J.maxrank;
    if (m < mr) mr = m;
    if (n < mr) mr = n;
    T R;
    R.setup(tm, m, n);
    R.load_known(tm, J.A, m, false);
    __syncthreads();   // every load of A done before A is rewritten
    double err, st[2];
    const int p = R.factor(tm, J.maxrank, J.reltol, J.abstol, J.leftorth != 0, pv, &err, st, Lsc,
                           J.rowperm, J.colperm, Usc, mr);
    R.store_trailing(tm, J.A, m, p > 0 ? p : 0);
    __syncthreads();   // permutations, pivots and recorded factors complete
    const int pp = p > 0 ? p : 0;
    for (int64_t q = tm.tid(); q < (int64_t)m * pp; q += tm.nt()) {
        const int k = (int)(q / m), pos = (int)(q - (int64_t)k * m);
        if (pos > k) J.A[pos + (int64_t)m * k] = Lsc[J.rowperm[pos] + (int64_t)m * k];
        else if (pos == k) J.A[k + (int64_t)m * k] = pv[k];
    }
    for (int64_t q = tm.tid(); q < (int64_t)pp * n; q += tm.nt()) {
        const int pj = (int)(q / pp), k = (int)(q - (int64_t)pj * pp);
        if (pj > k) J.A[k + (int64_t)m * pj] = Usc[k + mr * J.colperm[pj]];
    }
    __syncthreads();
    for (int i = tm.tid(); i < m; i += tm.nt()) J.rowperm[i] += 1;
    for (int j = tm.tid(); j < n; j += tm.nt()) J.colperm[j] += 1;
    if (tm.tid() == 0) {
        J.status = p < 0 ? -p : 0;
        J.npivot = pp;
        J.error = err;
    }
}

// rrlu!(A) of the jobs that fit a 128×128 register tile, one workgroup per
// job: the matrix stays in registers during the factorization (the solve
// engine's tile, here with its packed factors written out).  idx: the job
// indices; scratch + soff[q]: the job's Lsc (m × mr) then Usc (mr × n).
__global__ __launch_bounds__(kTeam, 2) void tci_rrlu_tile_kernel(tci_lu_job *__restrict__ jobs,
                                                                const int32_t *__restrict__ idx,
                                                                int64_t count, double *__restrict__ scratch,
                                                                const int64_t *__restrict__ soff)
{
    if ((int64_t)blockIdx.x >= count) return;
    using Team = DevTeam<kTeam, 2>;
    __shared__ double pv[128];
    tci_lu_job &J = jobs[idx[blockIdx.x]];
    const int m = (int)J.m, n = (int)J.n;
    Team tm;
    tm.init(nullptr, nullptr);
    int64_t mr = J.maxrank;
    if (m < mr) mr = m;
    if (n < mr) mr = n;
    double *Lsc = scratch + soff[blockIdx.x];
    double *Usc = Lsc + (int64_t)m * mr;
    if (TileLU<Team, 1, 8>::fits(m, n)) tile_job<TileLU<Team, 1, 8>>(tm, J, m, n, Lsc, Usc, pv);
    else if (TileLU<Team, 1, 32>::fits(m, n)) tile_job<TileLU<Team, 1, 32>>(tm, J, m, n, Lsc, Usc, pv);
    else if (TileLU<Team, 2, 8>::fits(m, n)) tile_job<TileLU<Team, 2, 8>>(tm, J, m, n, Lsc, Usc, pv);
    else tile_job<TileLU<Team, 2, 32>>(tm, J, m, n, Lsc, Usc, pv);
}

// entry q of the unpacked factors: q < m·p an entry of L, else of U.  The
// bodies below are shared by the standalone kernels and the fused TT sweep,
// so both compute every entry with the same operations
__device__ __forceinline__ void lu_unpack_at(int64_t q, const double *A, int64_t m, int64_t p, int leftorth,
                                             double *L, int64_t ldl, double *U, int64_t ldu)
{
    const int64_t nl = m * p;
    if (q < nl) {
        int64_t j = q / m, i = q - j * m;
        double v = i >= j ? A[i + m * j] : 0.0;
        if (leftorth && i == j) v = 1.0;
        L[i + ldl * j] = v;
    } else {
        int64_t r = q - nl;
        int64_t j = r / p, i = r - j * p;
        double v = i <= j ? A[i + m * j] : 0.0;
        if (!leftorth && i == j) v = 1.0;
        U[i + ldu * j] = v;
    }
}

// The factors of a finished job, whose rank is read where it lies (no host round
// trip before this launch): L m×p and U p×n (null: right behind L), the pivots in
// diag unless null, and with UT non-null the p×p block U11 transposed (for ranks
// up to kLuciSolveMax)
__global__ __launch_bounds__(256) void tci_lu_unpack_kernel(const tci_lu_job *__restrict__ job, double *__restrict__ L,
                                                            double *__restrict__ U, double *__restrict__ diag,
                                                            double *__restrict__ UT)
{
    const double *A = job->A;
    const int64_t m = job->m, n = job->n, p = job->npivot;
    const int leftorth = job->leftorth;
    const int64_t nl = m * p, nu = p * n;
    if (!U) U = L + nl;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nl + nu + p;
         q += (int64_t)gridDim.x * blockDim.x) {
        if (q >= nl + nu) {
            const int64_t k = q - nl - nu;
            if (diag) diag[k] = A[k + m * k];
            continue;
        }
        lu_unpack_at(q, A, m, p, leftorth, L, m, U, p);
        if (UT && p <= kLuciSolveMax && q >= nl && q - nl < p * p) {
            const int64_t r = q - nl, j = r / p, i = r - j * p;
            UT[j + p * i] = U[r];
        }
    }
}

// ------------------------------------------------------------ products
// C = A·B (M×K times K×N, column-major), one thread per entry of C, each
// sum in ascending k from 0.0 with a rounding per product and per sum (the
// order of the oracle's loops; the reference calls BLAS here).
__device__ __forceinline__ void gemm_at(int64_t q, int64_t M, int64_t K, const double *A, int64_t lda,
                                        const double *B, int64_t ldb, double *Cm, int64_t ldc)
{
    const int64_t j = q / M, i = q - j * M;
    double acc = 0.0;
    for (int64_t k = 0; k < K; ++k) acc = acc + A[i + lda * k] * B[k + ldb * j];
    Cm[i + ldc * j] = acc;
}

// A workgroup forms a 32×32 block of C, four entries a thread, from LDS copies of
// 16 columns of A and rows of B at a time (one thread per entry with both factors
// read from memory took 38 us for 2048 x 128 times 128 x 128, this 21 us; the
// library's matrix product fuses the rounding that the reference's values have)
constexpr int kGemmTile = 32, kGemmK = 16;
__global__ __launch_bounds__(256) void tci_gemm_kernel(int64_t M, int64_t N, int64_t K, const double *__restrict__ A,
                                                       int64_t lda, const double *__restrict__ B, int64_t ldb,
                                                       double *__restrict__ Cm, int64_t ldc)
{
    __shared__ double sa[kGemmK][kGemmTile], sb[kGemmTile][kGemmK + 1];
    const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
    const int64_t mt = (M + kGemmTile - 1) / kGemmTile, nt = (N + kGemmTile - 1) / kGemmTile;
    for (int64_t t = blockIdx.x; t < mt * nt; t += gridDim.x) {
        const int64_t i0 = (t % mt) * kGemmTile, j0 = (t / mt) * kGemmTile;
        double acc[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
        for (int64_t k0 = 0; k0 < K; k0 += kGemmK) {
            const int kn = (int)(K - k0 < kGemmK ? K - k0 : kGemmK);
            for (int q = threadIdx.x; q < kGemmK * kGemmTile; q += 256) {
                const int i = q % kGemmTile, k = q / kGemmTile;
                sa[k][i] = k < kn && i0 + i < M ? A[i0 + i + lda * (k0 + k)] : 0.0;
                const int kk = q % kGemmK, j = q / kGemmK;
                sb[j][kk] = kk < kn && j0 + j < N ? B[k0 + kk + ldb * (j0 + j)] : 0.0;
            }
            __syncthreads();
            // (no padded terms: they could turn a sum of -0 or an infinity)
            for (int k = 0; k < kn; ++k)
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int w = 0; w < 2; ++w) acc[u][w] = acc[u][w] + sa[k][tx + 16 * u] * sb[ty + 16 * w][k];
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                const int64_t i = i0 + tx + 16 * u, j = j0 + ty + 16 * w;
                if (i < M && j < N) Cm[i + ldc * j] = acc[u][w];
            }
    }
}

hipError_t launch_gemm(int64_t M, int64_t N, int64_t K, const double *A, int64_t lda, const double *B, int64_t ldb,
                       double *Cm, int64_t ldc, hipStream_t st)
{
    if (M * N == 0) return hipSuccess;
    int64_t blocks = ((M + kGemmTile - 1) / kGemmTile) * ((N + kGemmTile - 1) / kGemmTile);
    if (blocks > 65535) blocks = 65535;
    hipLaunchKernelGGL(tci_gemm_kernel, dim3((unsigned)blocks), dim3(256), 0, st, M, N, K, A, lda, B, ldb, Cm, ldc);
    return hipGetLastError();
}

// ---------------------------------------------------------- LUCI factors
// left(luci) and right(luci) of MatrixLUCI (matrixluci.jl:40-84) from the
// unpacked factors L (m×p, lda m) and U (p×n, lda p) of one rrLU with
// 1-based permutations rowperm/colperm (int32).  One thread per row of left
// (position i, written to row rowperm[i]-1) and one per column of right
// (position j, written to column colperm[j]-1); each substitution or dot
// product runs in a fixed order (ascending t for products from 0.0, back to
// front for the triangular solves).
__device__ __forceinline__ void luci_at(int64_t q, int64_t m, int64_t p, int leftorth, const int32_t *rowperm,
                                        const int32_t *colperm, const double *L, const double *U, double *left,
                                        int64_t ldl, double *right, int64_t ldr)
{
    if (q < m) {
        const int64_t i = q, r = rowperm[i] - 1;
        double *out = left + r;   // row r of left, stride ldl
        if (leftorth) {
            // colstimespivotinv (48-57): [I_p; L21·L11⁻¹]; x·L11 = L[i,1:p]
            if (i < p) {
                for (int64_t j = 0; j < p; ++j) out[ldl * j] = i == j ? 1.0 : 0.0;
            } else {
                for (int64_t j = p - 1; j >= 0; --j) {
                    double s = L[i + m * j];
                    for (int64_t t = j + 1; t < p; ++t) s = s - out[ldl * t] * L[t + m * j];
                    out[ldl * j] = s / L[j + m * j];
                }
            }
        } else {
            // colmatrix (40-42): L · U[:,1:p]
            for (int64_t j = 0; j < p; ++j) {
                double s = 0.0;
                const int64_t tmax = i < j ? i : j;
                for (int64_t t = 0; t <= tmax && t < p; ++t) s = s + L[i + m * t] * U[t + p * j];
                out[ldl * j] = s;
            }
        }
    } else {
        const int64_t j = q - m, c = colperm[j] - 1;
        double *out = right + ldr * c;   // column c of right
        if (leftorth) {
            // rowmatrix (44-46): L[1:p,:] · U
            for (int64_t i = 0; i < p; ++i) {
                double s = 0.0;
                const int64_t tmax = i < j ? i : j;
                for (int64_t t = 0; t <= tmax; ++t) s = s + L[i + m * t] * U[t + p * j];
                out[i] = s;
            }
        } else {
            // pivotinvtimesrows (59-68): [I_p  U11⁻¹·U12]
            if (j < p) {
                for (int64_t i = 0; i < p; ++i) out[i] = i == j ? 1.0 : 0.0;
            } else {
                for (int64_t i = p - 1; i >= 0; --i) {
                    double s = U[i + p * j];
                    for (int64_t t = i + 1; t < p; ++t) s = s - U[i + p * t] * out[t];
                    out[i] = s / U[i + p * i];
                }
            }
        }
    }
}

// The standalone kernels split the two factors.  A product's entries are
// independent, one thread each.  A substitution is a chain of p²/2 dependent
// subtractions per row whatever is done, so a wave runs 64 rows side by side with
// their solved entries in LDS and the triangular factor read through scalar loads
// (one thread per row, its own outputs read back from memory, took up to 527 us
// for 864 x 72; these 68).

// left = colmatrix (L·U[:,1:p], m×p) or right = rowmatrix (L[1:p,:]·U, p×n), by leftorth
__global__ __launch_bounds__(256) void tci_luci_product_kernel(int64_t m, int64_t n, int64_t p, int leftorth,
                                                               const int32_t *__restrict__ rowperm,
                                                               const int32_t *__restrict__ colperm,
                                                               const double *__restrict__ L,
                                                               const double *__restrict__ U, double *__restrict__ left,
                                                               int64_t ldl, double *__restrict__ right, int64_t ldr)
{
    const int64_t rows = leftorth ? p : m, cols = leftorth ? n : p;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < rows * cols;
         q += (int64_t)gridDim.x * blockDim.x) {
        const int64_t j = q / rows, i = q - j * rows;
        int64_t tmax = i < j ? i : j;
        if (tmax > p - 1) tmax = p - 1;
        double s = 0.0;
        for (int64_t t = 0; t <= tmax; ++t) s = s + L[i + m * t] * U[t + p * j];
        if (leftorth) right[i + ldr * (colperm[j] - 1)] = s;
        else left[(rowperm[i] - 1) + ldl * j] = s;
    }
}

// left = colstimespivotinv ([I; L21·L11⁻¹], leftorth) or right = pivotinvtimesrows
// ([I U11⁻¹·U12]).  Vector v (row v of left, column v of right) is a unit vector
// for v < p; else x_j = b_j - Σ_{t>j} x_t·M[t, j] with M = L11, or U11 transposed
// (unit diagonals), j descending, each sum in ascending t.
__global__ __launch_bounds__(64) void tci_luci_solve_kernel(int64_t nv, int64_t m, int p, int leftorth,
                                                            const int32_t *__restrict__ perm,
                                                            const double *__restrict__ LU,
                                                            const double *__restrict__ M, int64_t ldm,
                                                            double *__restrict__ out, int64_t ldo)
{
    extern __shared__ double x[];   // [entry][vector]
    const int lane = threadIdx.x;
    const int64_t v = (int64_t)blockIdx.x * 64 + lane;
    const bool have = v < nv;
    const int64_t vc = have ? v : nv - 1, at = perm[vc] - 1;
    // entry j of vector v: b[bs·j], out[os·j]
    const double *b = leftorth ? LU + vc : LU + (int64_t)p * vc;
    const int64_t bs = leftorth ? m : 1, os = leftorth ? ldo : 1;
    double *o = leftorth ? out + at : out + ldo * at;
    for (int j = p - 1; j >= 0; --j) {
        const double *Mj = M + ldm * j;
        double s = b[bs * j];
        int t = j + 1;
        for (; t + 8 <= p; t += 8) {
            double y[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) y[u] = x[(t + u) * 64 + lane] * Mj[t + u];
#pragma unroll
            for (int u = 0; u < 8; ++u) s = s - y[u];
        }
        for (; t < p; ++t) s = s - x[t * 64 + lane] * Mj[t];
        x[j * 64 + lane] = s;   // (the diagonal is 1)
        if (have) o[os * j] = v < p ? (v == j ? 1.0 : 0.0) : s;
    }
}

// one thread per row of left and column of right: ranks beyond the solve kernel's LDS
__global__ void tci_luci_kernel(int64_t m, int64_t n, int64_t p, int leftorth, const int32_t *__restrict__ rowperm,
                                const int32_t *__restrict__ colperm, const double *__restrict__ L,
                                const double *__restrict__ U, double *__restrict__ left, int64_t ldl,
                                double *__restrict__ right, int64_t ldr)
{
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < m + n;
         q += (int64_t)gridDim.x * blockDim.x)
        luci_at(q, m, p, leftorth, rowperm, colperm, L, U, left, ldl, right, ldr);
}

hipError_t launch_luci(int64_t m, int64_t n, int64_t p, int leftorth, const int32_t *rowperm, const int32_t *colperm,
                       const double *L, const double *U, const double *UT, double *left, int64_t ldl, double *right,
                       int64_t ldr, hipStream_t st)
{
    const int64_t tot = m + n;
    if (tot == 0 || p == 0) return hipSuccess;
    if (p <= kLuciSolveMax) {
        const int64_t prod = leftorth ? p * n : m * p, nv = leftorth ? m : n;
        const size_t lds = (size_t)p * 64 * sizeof(double);
        if (lds > 64 * 1024) {
            const hipError_t e = hipFuncSetAttribute((const void *)tci_luci_solve_kernel,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
            if (e != hipSuccess) return e;
        }
        hipLaunchKernelGGL(tci_luci_product_kernel, dim3((unsigned)std::min<int64_t>((prod + 255) / 256, 65535)),
                           dim3(256), 0, st, m, n, p, leftorth, rowperm, colperm, L, U, left, ldl, right, ldr);
        if (leftorth)
            hipLaunchKernelGGL(tci_luci_solve_kernel, dim3((unsigned)((nv + 63) / 64)), dim3(64), lds, st, nv, m, (int)p,
                               1, rowperm, L, L, m, left, ldl);
        else
            hipLaunchKernelGGL(tci_luci_solve_kernel, dim3((unsigned)((nv + 63) / 64)), dim3(64), lds, st, nv, m, (int)p,
                               0, colperm, U, UT, p, right, ldr);
        return hipGetLastError();
    }
    int64_t blocks = (tot + 255) / 256;
    if (blocks > 65535) blocks = 65535;
    hipLaunchKernelGGL(tci_luci_kernel, dim3((unsigned)blocks), dim3(256), 0, st, m, n, p, leftorth, rowperm, colperm,
                       L, U, left, ldl, right, ldr);
    return hipGetLastError();
}

// left(lu) and right(lu) with permute=true (matrixlu.jl:374-392): row i of
// L goes to row rowperm[i]-1 of left, column j of U to column colperm[j]-1
// of right (L m×p with lda m, U p×n with lda p; permutations 1-based)
__device__ __forceinline__ void lu_permute_at(int64_t q, int64_t m, int64_t p, const int32_t *rowperm,
                                              const int32_t *colperm, const double *L, const double *U,
                                              double *left, int64_t ldl, double *right, int64_t ldr)
{
    const int64_t nl = m * p;
    if (q < nl) {
        const int64_t j = q / m, i = q - j * m;
        left[(rowperm[i] - 1) + ldl * j] = L[i + m * j];
    } else {
        const int64_t r = q - nl, j = r / p, i = r - j * p;
        right[i + ldr * (colperm[j] - 1)] = U[i + p * j];
    }
}

__global__ void tci_lu_permute_kernel(int64_t m, int64_t n, int64_t p, const int32_t *__restrict__ rowperm,
                                      const int32_t *__restrict__ colperm, const double *__restrict__ L,
                                      const double *__restrict__ U, double *__restrict__ left, int64_t ldl,
                                      double *__restrict__ right, int64_t ldr)
{
    const int64_t nl = m * p, nu = p * n;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < nl + nu;
         q += (int64_t)gridDim.x * blockDim.x)
        lu_permute_at(q, m, p, rowperm, colperm, L, U, left, ldl, right, ldr);
}

// ------------------------------------------------------ fused TT sweep
// The host-driven sweep (per bond: rrlu!, unpack, left/right of rrLU or
// MatrixLUCI, the product into the neighbour; tensortrain.jl:155-182,
// conversion.jl:105-141) in one workgroup: the streaming rrLU of the team
// (whose packed result equals every other rrLU kernel's) and the entry bodies
// of the standalone kernels above, so every value has the same bits.  Each
// bond's new dimension p is returned to every thread by the factorization,
// so the shapes of the next bond need no memory round trip.
constexpr int kTtTeam = 256;

__device__ __forceinline__ double tt_nan_max(double a, double b)
{
    if (a != a || b != b) return a + b;
    return a > b ? a : b;
}

__global__ __launch_bounds__(kTtTeam) void tci_tt_sweep_kernel(TtSweepArgs a)
{
    extern __shared__ double stage[];
    DevTeam<kTtTeam> tm;
    const int L = a.L;
    const bool fw = a.forward != 0;
    int64_t carried = -1;   // the previous bond's new dimension
    for (int it = 0; it < L - 1; ++it) {
        const int b = fw ? it : L - 2 - it;
        const int s = fw ? b : b + 1;
        const int64_t m = fw ? (carried >= 0 ? carried : a.links[b]) * a.d[b] : a.links[b + 1];
        const int64_t n = fw ? a.links[b + 1] : a.d[b + 1] * (carried >= 0 ? carried : a.links[b + 2]);
        double *A = a.cores + a.off[s];
        const int64_t mx = m > n ? m : n;
        if (mx <= a.stage_cap) tm.init(stage, stage + mx);
        else tm.init(a.gstage, a.gstage + mx);
        // a bond matrix that fits is factored in LDS (the same operations on
        // a copy with a shorter latency) and copied back
        double *Aw = A;
        if (m * n <= a.mat_cap) {
            Aw = stage + 2 * (int64_t)a.stage_cap;
            for (int64_t q = tm.tid(); q < m * n; q += kTtTeam) Aw[q] = A[q];
            tm.sync();
        }
        double err, st2[2];
        const int p = rrlu_team(tm, Aw, (int)m, (int)n, a.maxrank, a.reltol, a.abstol, fw, a.perm, a.perm + m, nullptr,
                                &err, st2);
        if (Aw != A) {
            tm.sync();
            for (int64_t q = tm.tid(); q < m * n; q += kTtTeam) A[q] = Aw[q];
        }
        if (p < 0) {
            if (tm.tid() == 0) {
                a.status[0] = -p;
                a.status[1] = b;
            }
            return;
        }
        int32_t *rp = a.perm, *cp = a.perm + m;
        for (int64_t i = tm.tid(); i < m; i += kTtTeam) rp[i] += 1;
        for (int64_t j = tm.tid(); j < n; j += kTtTeam) cp[j] += 1;
        tm.sync();
        // running pivot errors (the diagonal of the packed factors, one
        // thread per entry) and the pivots
        for (int k = tm.tid(); k < p; k += kTtTeam) a.pe[k] = tt_nan_max(a.pe[k], fabs(A[k + m * k]));
        if (tm.tid() == 0) a.pe[p] = tt_nan_max(a.pe[p], err);
        int32_t *pv = a.piv + (int64_t)b * 2 * a.R;
        for (int k = tm.tid(); k < p; k += kTtTeam) {
            pv[k] = rp[k];
            pv[p + k] = cp[k];
        }
        for (int64_t q = tm.tid(); q < m * p + (int64_t)p * n; q += kTtTeam)
            lu_unpack_at(q, A, m, p, fw ? 1 : 0, a.wl, m, a.wu, p);
        tm.sync();
        double *lft = fw ? A : a.wc, *rgt = fw ? a.wc : A;
        if (a.method == 0) {
            for (int64_t q = tm.tid(); q < m * p + (int64_t)p * n; q += kTtTeam)
                lu_permute_at(q, m, p, rp, cp, a.wl, a.wu, lft, m, rgt, p);
        } else if (p > 0) {
            for (int64_t q = tm.tid(); q < m + n; q += kTtTeam)
                luci_at(q, m, p, fw ? 1 : 0, rp, cp, a.wl, a.wu, lft, m, rgt, p);
        }
        tm.sync();
        if (fw) {
            const int64_t nn = a.d[b + 1] * a.links[b + 2];
            double *nx = a.cores + a.off[b + 1];
            for (int64_t q = tm.tid(); q < (int64_t)p * nn; q += kTtTeam) gemm_at(q, p, n, a.wc, p, nx, n, a.wp, p);
            tm.sync();
            for (int64_t q = tm.tid(); q < (int64_t)p * nn; q += kTtTeam) nx[q] = a.wp[q];
        } else {
            const int64_t mm = a.links[b] * a.d[b];
            double *pv2 = a.cores + a.off[b];
            for (int64_t q = tm.tid(); q < mm * p; q += kTtTeam) gemm_at(q, mm, m, pv2, mm, a.wc, m, a.wp, mm);
            tm.sync();
            for (int64_t q = tm.tid(); q < mm * p; q += kTtTeam) pv2[q] = a.wp[q];
        }
        if (tm.tid() == 0) a.links[b + 1] = p;
        carried = p;
        tm.sync();
    }
}

hipError_t launch_tt_sweep(const TtSweepArgs &a, hipStream_t st)
{
    const size_t lds = sizeof(double) * (2 * (size_t)a.stage_cap + (size_t)a.mat_cap);
    hipError_t e = hipFuncSetAttribute((const void *)tci_tt_sweep_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)lds);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(tci_tt_sweep_kernel, dim3(1), dim3(kTtTeam), lds, st, a);
    return hipGetLastError();
}

hipError_t launch_lu_permute(int64_t m, int64_t n, int64_t p, const int32_t *rowperm, const int32_t *colperm,
                             const double *L, const double *U, double *left, int64_t ldl, double *right, int64_t ldr,
                             hipStream_t st)
{
    const int64_t tot = m * p + p * n;
    if (tot == 0) return hipSuccess;
    int64_t blocks = (tot + 255) / 256;
    if (blocks > 65535) blocks = 65535;
    hipLaunchKernelGGL(tci_lu_permute_kernel, dim3((unsigned)blocks), dim3(256), 0, st, m, n, p, rowperm, colperm,
                       L, U, left, ldl, right, ldr);
    return hipGetLastError();
}

// ------------------------------------------------------------ evaluation
// rowsx[r = i + nI·c] = left[i] ⊕ central digits of c (first fastest)
__global__ void tci_kron_center_kernel(const uint8_t *__restrict__ left, int64_t nI, int nl,
                                       const int32_t *__restrict__ cdims, int M, int64_t nc,
                                       uint8_t *__restrict__ rowsx, int stride)
{
    for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < nI * nc;
         r += (int64_t)gridDim.x * blockDim.x) {
        int64_t c = r / nI, i = r - c * nI;
        uint8_t *dst = rowsx + r * stride;
        for (int t = 0; t < nl; ++t) dst[t] = left[i * nl + t];
        for (int t = 0; t < M; ++t) {
            int64_t dt = cdims[t];
            int64_t q = c / dt;
            dst[nl + t] = (uint8_t)(c - q * dt + 1);
            c = q;
        }
    }
}

// out[i + nr·j] = f(rows[i] ⊕ cols[j]) with a NaN-propagating max|out| per block
__global__ void tci_eval_kernel(int kind, const double *__restrict__ params,
                                const int32_t *__restrict__ iparams, int L,
                                const uint8_t *__restrict__ rows, int64_t nrow, int rstride, int nl,
                                const uint8_t *__restrict__ cols, int64_t ncol, int cstride,
                                double *__restrict__ out, double *__restrict__ blockmax)
{
    __shared__ double red[4];
    double lmax = 0.0;
    const int64_t tot = nrow * ncol;
    for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < tot;
         q += (int64_t)gridDim.x * blockDim.x) {
        int64_t j = q / nrow, i = q - j * nrow;
        tci_point x;
        x.a = rows + i * rstride;
        x.b = cols + j * cstride;
        x.na = nl;
        x.L = L;
        double v = tci_functor_eval(kind, params, iparams, &x);
        out[q] = v;
        lmax = jl_max(lmax, fabs(v));
    }
    for (int off = 32; off >= 1; off >>= 1) lmax = jl_max(lmax, __shfl_xor(lmax, off));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = lmax;
    __syncthreads();
    if (threadIdx.x == 0) {
        double r = red[0];
        for (int w = 1; w < (int)(blockDim.x >> 6); ++w) r = jl_max(r, red[w]);
        blockmax[blockIdx.x] = r;
    }
}

// --------------------------------------------------------- TT evaluation
// evaluate(tt, x) (abstracttensortrain.jl:124-132) at npts points: for each
// point the row vector v (χ_0 = 1 entries of 1) times each site's slice
// T_b[:, x_b, :], every product summed in ascending bond order from 0.0.
// A workgroup takes np points; their running vectors live in LDS (two
// buffers of np·chimax doubles), and thread t computes entries (p, j) of
// the next vector.  Site b's core starts at cores + coff[b]; its shape is
// dims3[3b..3b+2].  With fkind != 0, f is evaluated at the same points and
// the workgroup writes the NaN-propagating maxima of |TT - f| and |f| to
// blockmax[2·block], [2·block + 1].
__global__ __launch_bounds__(256) void tci_tt_eval_kernel(
    int L, const int64_t *__restrict__ dims3, const int64_t *__restrict__ coff,
    const double *__restrict__ cores, const uint8_t *__restrict__ pts, int64_t npts, int np,
    int chimax, int fkind, const double *__restrict__ params, const int32_t *__restrict__ iparams,
    double *__restrict__ out_tt, double *__restrict__ out_f, double *__restrict__ blockmax)
{
    extern __shared__ double vbuf[];
    __shared__ double red[8];
    const int64_t p0 = (int64_t)blockIdx.x * np;
    const int cn = (int)(npts - p0 < np ? npts - p0 : np);
    double *V = vbuf, *W = vbuf + (int64_t)np * chimax;
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int q = tid; q < cn; q += nt) V[(int64_t)q * chimax] = 1.0;
    __syncthreads();
    for (int b = 0; b < L; ++b) {
        const int64_t d0 = dims3[3 * b], d = dims3[3 * b + 1], d2 = dims3[3 * b + 2];
        const double *T = cores + coff[b];
        for (int64_t o = tid; o < (int64_t)cn * d2; o += nt) {
            const int64_t q = o / d2, j = o - q * d2;
            const int64_t s = pts[(p0 + q) * L + b] - 1;
            const double *Tc = T + d0 * (s + d * j);
            const double *v = V + q * chimax;
            double acc = 0.0;
            for (int64_t i = 0; i < d0; ++i) acc = acc + v[i] * Tc[i];
            W[q * chimax + j] = acc;
        }
        __syncthreads();
        double *t = V; V = W; W = t;
    }
    double le = 0.0, lf = 0.0;
    for (int q = tid; q < cn; q += nt) {
        const double tt = V[(int64_t)q * chimax];
        out_tt[p0 + q] = tt;
        if (fkind) {
            tci_point x;
            x.a = pts + (p0 + q) * L;
            x.b = x.a;
            x.na = L;
            x.L = L;
            const double fv = tci_functor_eval(fkind, params, iparams, &x);
            if (out_f) out_f[p0 + q] = fv;
            le = jl_max(le, fabs(tt - fv));
            lf = jl_max(lf, fabs(fv));
        }
    }
    if (!fkind) return;
    for (int off = 32; off >= 1; off >>= 1) {
        le = jl_max(le, __shfl_xor(le, off));
        lf = jl_max(lf, __shfl_xor(lf, off));
    }
    if ((tid & 63) == 0) {
        red[2 * (tid >> 6)] = le;
        red[2 * (tid >> 6) + 1] = lf;
    }
    __syncthreads();
    if (tid == 0) {
        double e = red[0], f = red[1];
        for (int w = 1; w < nt / 64; ++w) {
            e = jl_max(e, red[2 * w]);
            f = jl_max(f, red[2 * w + 1]);
        }
        blockmax[2 * blockIdx.x] = e;
        blockmax[2 * blockIdx.x + 1] = f;
    }
}

// ---- many points at once.  Per site the points are grouped by their local
// index s, so that 64 of them share the slice T_b[:, s, :]: a lane carries one
// point, the slice's entries come through scalar loads, and every LDS read of
// the running vector feeds J products.  tci_tt_eval_kernel above loads one core
// entry per product, each lane from another column: 53 ms for 100 000 points of
// 20 sites, d = 10, bond dimension 96; these 3.3 ms together (0.85 ms is the rate
// of unfused FP64 multiplies and adds).
constexpr int kTtBins = 256;    // local indices are 1..255

__global__ __launch_bounds__(256) void tci_tt_count_kernel(const uint8_t *__restrict__ pts, int64_t npts, int L,
                                                           int32_t *__restrict__ bins)
{
    __shared__ int32_t h[kTtBins];
    const int b = blockIdx.y;
    h[threadIdx.x] = 0;
    __syncthreads();
    for (int u = 0; u < 4; ++u) {
        const int64_t q = (int64_t)blockIdx.x * 1024 + u * 256 + threadIdx.x;
        if (q < npts) atomicAdd(&h[pts[q * L + b]], 1);
    }
    __syncthreads();
    if (h[threadIdx.x]) atomicAdd(&bins[b * kTtBins + threadIdx.x], h[threadIdx.x]);
}

// per site: bins[s] becomes the first place of s's points, and the tiles of at
// most 64 points of one s are listed
__global__ __launch_bounds__(256) void tci_tt_tiles_kernel(int32_t *__restrict__ bins, TtTile *__restrict__ tiles,
                                                           int32_t *__restrict__ ntiles, int maxtiles)
{
    __shared__ int32_t place[kTtBins], tile[kTtBins];
    const int b = blockIdx.x, s = threadIdx.x;
    const int n = bins[b * kTtBins + s], t = (n + 63) / 64;
    place[s] = n;
    tile[s] = t;
    __syncthreads();
    for (int off = 1; off < kTtBins; off *= 2) {
        const int x = s >= off ? place[s - off] : 0, y = s >= off ? tile[s - off] : 0;
        __syncthreads();
        place[s] += x;
        tile[s] += y;
        __syncthreads();
    }
    const int p0 = place[s] - n, t0 = tile[s] - t;
    bins[b * kTtBins + s] = p0;
    for (int k = 0; k < t; ++k)
        if (t0 + k < maxtiles) tiles[(int64_t)b * maxtiles + t0 + k] = TtTile{s, p0 + 64 * k, n - 64 * k < 64 ? n - 64 * k : 64};
    if (s == kTtBins - 1) ntiles[b] = tile[s];
}

// order[b·npts + place] = point, grouped by s (any order within a group)
__global__ __launch_bounds__(256) void tci_tt_order_kernel(const uint8_t *__restrict__ pts, int64_t npts, int L,
                                                           int32_t *__restrict__ bins, int32_t *__restrict__ order)
{
    __shared__ int32_t h[kTtBins], base[kTtBins];
    const int b = blockIdx.y;
    h[threadIdx.x] = 0;
    __syncthreads();
    int s[4], r[4];
    for (int u = 0; u < 4; ++u) {
        const int64_t q = (int64_t)blockIdx.x * 1024 + u * 256 + threadIdx.x;
        s[u] = q < npts ? pts[q * L + b] : 0;
        r[u] = q < npts ? atomicAdd(&h[s[u]], 1) : 0;
    }
    __syncthreads();
    const int n = h[threadIdx.x];
    base[threadIdx.x] = n ? atomicAdd(&bins[b * kTtBins + threadIdx.x], n) : 0;
    __syncthreads();
    for (int u = 0; u < 4; ++u) {
        const int64_t q = (int64_t)blockIdx.x * 1024 + u * 256 + threadIdx.x;
        if (q < npts) order[(int64_t)b * npts + base[s[u]] + r[u]] = (int32_t)q;
    }
}

// W[q, :] = V[q, :]·T[:, s, :] for the points of one tile (V and W: stride
// doubles per point, V null: the vector [1]); each sum ascending from 0.0
template <int J>
__global__ __launch_bounds__(256) void tci_tt_site_kernel(const double *__restrict__ T, int d0, int d, int d2,
                                                          const TtTile *__restrict__ tiles,
                                                          const int32_t *__restrict__ ntiles,
                                                          const int32_t *__restrict__ order,
                                                          const double *__restrict__ V, double *__restrict__ W,
                                                          int stride)
{
    extern __shared__ double tile[];   // [i][point], 65 doubles a row (no bank conflicts while staging)
    if ((int)blockIdx.x >= ntiles[0]) return;
    const TtTile t = tiles[blockIdx.x];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    for (int p = wave; p < 64; p += 4) {
        const int64_t q = order[t.first + (p < t.n ? p : 0)];
        for (int i = lane; i < d0; i += 64) tile[i * 65 + p] = V ? V[q * stride + i] : 1.0;
    }
    __syncthreads();
    const double *Ts = T + (int64_t)d0 * (t.s - 1);
    const int64_t cs = (int64_t)d0 * d;   // from one column of the slice to the next
    const double *v = tile + lane;
    const int64_t q = order[t.first + (lane < t.n ? lane : 0)];
    for (int j0 = wave * J; j0 < d2; j0 += 4 * J) {
        const double *Tj[J];
#pragma unroll
        for (int j = 0; j < J; ++j) Tj[j] = Ts + cs * (j0 + j < d2 ? j0 + j : d2 - 1);
        double acc[J];
#pragma unroll
        for (int j = 0; j < J; ++j) acc[j] = 0.0;
        int i = 0;
        for (; i + 4 <= d0; i += 4) {
            double x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = v[(i + u) * 65];
#pragma unroll
            for (int j = 0; j < J; ++j)
#pragma unroll
                for (int u = 0; u < 4; ++u) acc[j] = acc[j] + x[u] * Tj[j][i + u];
        }
        for (; i < d0; ++i) {
            const double x = v[i * 65];
#pragma unroll
            for (int j = 0; j < J; ++j) acc[j] = acc[j] + x * Tj[j][i];
        }
        if (lane < t.n) {
#pragma unroll
            for (int j = 0; j < J; ++j)
                if (j0 + j < d2) W[q * stride + j0 + j] = acc[j];
        }
    }
}

// out_tt[q] = V[q·stride]; with fkind also f, and the maxima as in tci_tt_eval_kernel
__global__ __launch_bounds__(256) void tci_tt_finish_kernel(const double *__restrict__ V, int stride,
                                                            const uint8_t *__restrict__ pts, int64_t npts, int L,
                                                            int fkind, const double *__restrict__ params,
                                                            const int32_t *__restrict__ iparams,
                                                            double *__restrict__ out_tt, double *__restrict__ out_f,
                                                            double *__restrict__ blockmax)
{
    __shared__ double red[8];
    const int tid = threadIdx.x;
    const int64_t q = (int64_t)blockIdx.x * 256 + tid;
    double le = 0.0, lf = 0.0;
    if (q < npts) {
        const double tt = V[q * stride];
        out_tt[q] = tt;
        if (fkind) {
            tci_point x;
            x.a = pts + q * L;
            x.b = x.a;
            x.na = L;
            x.L = L;
            const double fv = tci_functor_eval(fkind, params, iparams, &x);
            if (out_f) out_f[q] = fv;
            le = fabs(tt - fv);
            lf = fabs(fv);
        }
    }
    if (!fkind) return;
    for (int off = 32; off >= 1; off >>= 1) {
        le = jl_max(le, __shfl_xor(le, off));
        lf = jl_max(lf, __shfl_xor(lf, off));
    }
    if ((tid & 63) == 0) {
        red[2 * (tid >> 6)] = le;
        red[2 * (tid >> 6) + 1] = lf;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 4; ++w) {
            red[0] = jl_max(red[0], red[2 * w]);
            red[1] = jl_max(red[1], red[2 * w + 1]);
        }
        blockmax[2 * blockIdx.x] = red[0];
        blockmax[2 * blockIdx.x + 1] = red[1];
    }
}

hipError_t launch_tt_group(const uint8_t *pts, int64_t npts, int L, int32_t *bins, TtTile *tiles, int32_t *ntiles,
                           int maxtiles, int32_t *order, hipStream_t st)
{
    const dim3 g((unsigned)((npts + 1023) / 1024), (unsigned)L);
    hipLaunchKernelGGL(tci_tt_count_kernel, g, dim3(256), 0, st, pts, npts, L, bins);
    hipLaunchKernelGGL(tci_tt_tiles_kernel, dim3((unsigned)L), dim3(256), 0, st, bins, tiles, ntiles, maxtiles);
    hipLaunchKernelGGL(tci_tt_order_kernel, g, dim3(256), 0, st, pts, npts, L, bins, order);
    return hipGetLastError();
}

hipError_t launch_tt_site(const double *T, int d0, int d, int d2, const TtTile *tiles, const int32_t *ntiles,
                          int maxtiles, const int32_t *order, const double *V, double *W, int stride, hipStream_t st)
{
    const size_t lds = (size_t)d0 * 65 * sizeof(double);
    // eight columns a wave where there are enough for all four waves
    const void *k = d2 > 16 ? (const void *)tci_tt_site_kernel<8> : (const void *)tci_tt_site_kernel<4>;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return e;
    }
    if (d2 > 16)
        hipLaunchKernelGGL((tci_tt_site_kernel<8>), dim3((unsigned)maxtiles), dim3(256), lds, st, T, d0, d, d2, tiles,
                           ntiles, order, V, W, stride);
    else
        hipLaunchKernelGGL((tci_tt_site_kernel<4>), dim3((unsigned)maxtiles), dim3(256), lds, st, T, d0, d, d2, tiles,
                           ntiles, order, V, W, stride);
    return hipGetLastError();
}

hipError_t launch_tt_finish(const double *V, int stride, const uint8_t *pts, int64_t npts, int L, int fkind,
                            const double *params, const int32_t *iparams, double *out_tt, double *out_f,
                            double *blockmax, hipStream_t st)
{
    hipLaunchKernelGGL(tci_tt_finish_kernel, dim3((unsigned)((npts + 255) / 256)), dim3(256), 0, st, V, stride, pts,
                       npts, L, fkind, params, iparams, out_tt, out_f, blockmax);
    return hipGetLastError();
}

// the table of a functor's per-site terms (term_value), for f along a site
__global__ __launch_bounds__(256) void tci_terms_kernel(int kind, const double *__restrict__ params, int nft, int L,
                                                        int dmax, double *__restrict__ ftab)
{
    const int q = blockIdx.x * 256 + threadIdx.x;
    if (q < nft * L * dmax)
        ftab[q] = term_value(kind, params, nft, L, q / (L * dmax), q / dmax % L, q % dmax + 1);
}

// f at the current point with site p at s (0-based): per-site terms summed in the
// functor's order, cur those of the current point, own those of (p, s); or the
// functor itself on row, the point's digits
template <bool TERMS>
__device__ __forceinline__ double fz_value(const FzArgs &a, const uint8_t *piv, const double *cur, const double *own,
                                           uint8_t *row, int p, int s)
{
    const int L = a.L;
    if constexpr (!TERMS) {
        for (int t = 0; t < L; ++t) row[t] = t == p ? (uint8_t)(s + 1) : piv[t];
        tci_point x;
        x.a = row;
        x.b = row;
        x.na = L;
        x.L = L;
        return tci_functor_eval(a.fkind, a.params, a.iparams, &x);
    }
    double f = 0.0;
    for (int k = 0; k < a.nft; ++k) {
        const double *c = cur + k * L;
        double u = 0.0;
        const double mine = own[k * a.dmax + s];
#pragma unroll 4
        for (int t = 0; t < L; ++t) u = u + (t == p ? mine : c[t]);
        if (a.fkind == TCI_F_LORENTZ_WEIGHTED) return 1.0 / (1.0 + u);
        const double w = a.params[2 + a.nft + k];
        f = f + a.params[2 + k] * tci_exp(-u / (2.0 * (w * w)));
    }
    return f;
}

// Σ_j x[j]·T[st·j] in ascending j from 0.0, the loads of eight terms in flight
// (the last ones clamped and not added)
__device__ __forceinline__ double fz_dot(const double *x, const double *T, int64_t st, int n)
{
    double acc = 0.0;
    for (int j0 = 0; j0 < n; j0 += 8) {
        double v[8], y[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int j = j0 + u < n ? j0 + u : n - 1;
            v[u] = T[st * j];
            y[u] = x[j];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const double t = y[u] * v[u], sum = acc + t;
            acc = j0 + u < n ? sum : acc;
        }
    }
    return acc;
}

// _floatingzone (globalsearch.jl:43-95) from each start point: one
// workgroup per point (grid-stride).  Per sweep, the right environments
// R_b = T_b[:, x_b, :]·R_{b+1} (R_L = [1], each entry summed in ascending
// bond order) are built from the current point; then for each site p, with
// l the row vector of the sites before p at the current point,
//   w_σ[k] = Σ_j l[j] T_p[j,σ,k]  (ascending j),  TT_σ = Σ_k w_σ[k] R_{p+1}[k]
// (ascending k), err_σ = |f(x with x_p = σ) − TT_σ|; x_p moves to Julia's
// argmax of err (first maximum, NaN above every number) and the running
// error takes the NaN-propagating max.  A sweep that leaves the error
// unchanged, or lifts it above earlystoptol, ends the search; so does a
// NaN error (with which the reference would sweep without end).
// Bound: the latency of a site's steps, which follow each other.  So the work
// area (renv | w, two of them | f and the terms along the site | the current
// point's terms | the slices T_b[:, x_b, :] where there is room | digit rows) lies
// in LDS, f is evaluated by the far end of the workgroup while w is formed, from
// terms that only differ in site p, and l is a row of the last w: two barriers a
// site.  With all of it in memory, every f from scratch and one thread looking for
// the maximum, 2000 starts of 20 sites, d 16, took 7.4 ms; 2.6 so, most of
// it the few starts that need 20 sweeps and more (0.11 ms each).
// LDS = false: the same on a work area in memory, for trains that LDS does not hold.
// TERMS: f by its terms, apart from the functors' own evaluation, whose registers
// would leave five waves a SIMD of the eight.
template <bool LDS, bool TERMS>
__global__ __launch_bounds__(256, TERMS ? 8 : 1) void tci_floatingzone_kernel(FzArgs a)
{
    __shared__ uint8_t piv[256];
    __shared__ double s_maxerr;
    __shared__ int s_best;
    extern __shared__ double dyn[];
    DevTeam<256> tm;   // (its wave operations)
    const int tid = threadIdx.x, nt = 256, L = a.L;
    double *base;
    if constexpr (LDS) base = dyn;
    else base = a.work + (int64_t)blockIdx.x * a.wstride;
    double *renv = base;
    double *w0 = renv + a.roff[L];
    const int64_t wsz = (int64_t)a.dmax * a.chimax;
    double *fv = w0 + 2 * wsz;
    double *own = fv + a.dmax;
    double *cur = own + a.nft * a.dmax;
    double *sl = cur + a.nft * L;
    uint8_t *rows = (uint8_t *)(sl + (LDS ? a.nslice : 0));
    for (int64_t q = blockIdx.x; q < a.npts; q += gridDim.x) {
        for (int t = tid; t < L; t += nt) piv[t] = a.pts[q * L + t];
        __syncthreads();
        for (int64_t sweep = 0;; ++sweep) {
            for (int i = tid; i < a.nft * L; i += nt) cur[i] = a.ftab[(int64_t)i * a.dmax + piv[i % L] - 1];
            if (LDS && a.nslice) {
                double *to = sl;
                for (int b = 1; b < L; ++b) {
                    const int d0 = (int)a.dims3[3 * b], d = (int)a.dims3[3 * b + 1], n = d0 * (int)a.dims3[3 * b + 2];
                    const double *Tc = a.cores + a.coff[b] + d0 * (int64_t)(piv[b] - 1);
                    for (int o = tid; o < n; o += nt) to[o] = Tc[o % d0 + (int64_t)d0 * d * (o / d0)];
                    to += n;
                }
            }
            // right environments of the current point
            if (tid == 0) {
                renv[a.roff[L - 1]] = 1.0;   // R_L
                w0[wsz] = 1.0;               // l before the first site
            }
            __syncthreads();
            const double *from = sl + a.nslice;
            for (int b = L - 1; b >= 1; --b) {
                const int d0 = (int)a.dims3[3 * b], d = (int)a.dims3[3 * b + 1], d2 = (int)a.dims3[3 * b + 2];
                const double *Rn = renv + a.roff[b];
                double *Rb = renv + a.roff[b - 1];
                if (LDS && a.nslice) {
                    from -= d0 * d2;
                    for (int j = tid; j < d0; j += nt) Rb[j] = fz_dot(Rn, from + j, d0, d2);
                } else {
                    const double *Tc = a.cores + a.coff[b] + d0 * (int64_t)(piv[b] - 1);
                    for (int j = tid; j < d0; j += nt) Rb[j] = fz_dot(Rn, Tc + j, (int64_t)d0 * d, d2);
                }
                __syncthreads();
            }
            if (sweep == 0) {
                // the start point's error: TT(x) = T_1[1, x_1, :]·R_2
                if (tid == 0) {
                    const int64_t d = a.dims3[1], d2 = a.dims3[2];
                    const double *Tc = a.cores + a.coff[0] + (int64_t)(piv[0] - 1);
                    const double *Rn = renv + a.roff[0];
                    double acc = 0.0;
                    for (int64_t k = 0; k < d2; ++k) acc = acc + (0.0 + 1.0 * Tc[d * k]) * Rn[k];
                    const int x0 = piv[0] - 1;
                    for (int k = 0; k < a.nft; ++k) own[k * a.dmax + x0] = cur[k * L];
                    s_maxerr = fabs(fz_value<TERMS>(a, piv, cur, own, rows, 0, x0) - acc);
                }
                __syncthreads();
            }
            const double prev = s_maxerr;
            const double *lv = w0 + wsz;
            for (int p = 0; p < L; ++p) {
                const int d0 = (int)a.dims3[3 * p], d = (int)a.dims3[3 * p + 1], d2 = (int)a.dims3[3 * p + 2];
                const double *T = a.cores + a.coff[p];
                const double *Rn = renv + a.roff[p];   // R_{p+1}
                double *w = w0 + (p & 1) * wsz;
                for (int s = nt - 1 - tid; s < d; s += nt) {
                    for (int k = 0; k < a.nft; ++k)
                        own[k * a.dmax + s] = a.ftab[((int64_t)k * L + p) * a.dmax + s];
                    fv[s] = fz_value<TERMS>(a, piv, cur, own, rows + (int64_t)s * L, p, s);
                }
                for (int o = tid; o < d * d2; o += nt) {
                    const int s = o / d2, k = o - s * d2;
                    w[(int64_t)s * a.chimax + k] = fz_dot(lv, T + (int64_t)d0 * (s + (int64_t)d * k), 1, d0);
                }
                __syncthreads();
                if (tid < 64) {
                    // isless order: NaN is above every number, the first of equal ones
                    double bv = -1.0;
                    uint32_t bi = 0xffffffffu;
                    for (int s = tid; s < d; s += 64) {
                        const double e = fabs(fv[s] - fz_dot(w + (int64_t)s * a.chimax, Rn, 1, d2));
                        // (by selects: as a branch it was compiled to keep the old bv)
                        const bool take = (bi == 0xffffffffu) | ((bv == bv) & ((e != e) | (bv < e)));
                        bi = take ? (uint32_t)s : bi;
                        bv = take ? e : bv;
                    }
                    const bool nan = bv != bv;
                    double mx;
                    uint32_t best;
                    if (tm.wave_any(nan)) {
                        best = tm.wave_min(nan ? bi : 0xffffffffu);
                        mx = tm.wave_bcast_f64(bv, (int)(best & 63u));
                    } else {
                        mx = tm.wave_max(bv);
                        best = tm.wave_min(bv == mx ? bi : 0xffffffffu);
                    }
                    for (int k = tid; k < a.nft; k += 64) cur[k * L + p] = own[k * a.dmax + best];
                    if (tid == 0) {
                        piv[p] = (uint8_t)(best + 1);
                        s_best = (int)best;
                        s_maxerr = jl_max(mx, s_maxerr);
                    }
                }
                __syncthreads();
                lv = w + (int64_t)s_best * a.chimax;
            }
            const double me = s_maxerr;
            if (me == prev || me > a.earlystoptol || me != me || sweep + 1 >= a.nsweeps) break;
            __syncthreads();   // (renv, w and cur are rewritten)
        }
        for (int t = tid; t < L; t += nt) a.pts[q * L + t] = piv[t];
        if (tid == 0) a.errs[q] = s_maxerr;
        __syncthreads();
    }
}

hipError_t launch_floatingzone(FzArgs a, int64_t slice, int blocks, double *ftab, hipStream_t st)
{
    if (a.npts <= 0) return hipSuccess;
    if (a.nft) {
        const int n = a.nft * a.L * a.dmax;
        hipLaunchKernelGGL(tci_terms_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, a.fkind, a.params,
                           a.nft, a.L, a.dmax, ftab);
        a.ftab = ftab;
    }
    // the slices where eight workgroups still share a CU (with less, the next
    // points' loads no longer hide behind each other)
    const size_t area = fz_area_bytes(a);
    a.nslice = area + sizeof(double) * (size_t)slice <= kFzSliceLds ? (int)slice : 0;
    const size_t lds = area + sizeof(double) * (size_t)a.nslice;
    const bool in = lds <= kFzLds;
    const auto k = in ? (a.nft ? tci_floatingzone_kernel<true, true> : tci_floatingzone_kernel<true, false>)
                      : (a.nft ? tci_floatingzone_kernel<false, true> : tci_floatingzone_kernel<false, false>);
    hipLaunchKernelGGL(k, dim3((unsigned)blocks), dim3(256), in ? lds : 0, st, a);
    return hipGetLastError();
}

// ------------------------------------------------------------- launchers
int tt_eval_points_per_block(int chimax)
{
    // two running-vector buffers of np·chimax doubles in at most 64 KiB
    int np = (int)((64 * 1024) / (16 * (int64_t)(chimax > 0 ? chimax : 1)));
    if (np > 256) np = 256;
    return np < 1 ? 1 : np;
}

hipError_t launch_tt_eval(int L, const int64_t *dims3, const int64_t *coff, const double *cores,
                          const uint8_t *pts, int64_t npts, int chimax, int fkind, const double *params,
                          const int32_t *iparams, double *out_tt, double *out_f, double *blockmax,
                          hipStream_t st)
{
    if (npts <= 0) return hipSuccess;
    const int np = tt_eval_points_per_block(chimax);
    const int64_t blocks = (npts + np - 1) / np;
    if (blocks > INT32_MAX) return hipErrorInvalidValue;
    const size_t lds = (size_t)2 * np * chimax * sizeof(double);
    if (lds > 64 * 1024) return hipErrorInvalidValue;
    hipLaunchKernelGGL(tci_tt_eval_kernel, dim3((unsigned)blocks), dim3(256), lds, st, L, dims3, coff, cores,
                       pts, npts, np, chimax, fkind, params, iparams, out_tt, out_f, blockmax);
    return hipGetLastError();
}

size_t lds_plan_bytes(const LdsPlan &p)
{
    return (size_t)2 * p.stage_cap * sizeof(double) + 2 * (size_t)p.tab_cap + (size_t)p.sets_cap +
           (size_t)p.lut_cap * sizeof(double) + (size_t)p.pi_cap * sizeof(double);
}

// the kernel variant a (team, functor kind) pair runs
static const void *solve_kernel_ptr(int team, int fkind)
{
    switch (team) {
    case 64: return solve_kernel_64(fkind);
    case 1024: return solve_kernel_1024(fkind);
    case 512: return solve_kernel_512(fkind);
    default: return solve_kernel_256(fkind);
    }
}

int solve_static_lds(int team, int fkind)
{
    hipFuncAttributes a;
    if (hipFuncGetAttributes(&a, solve_kernel_ptr(team, fkind)) != hipSuccess) return -1;
    return (int)a.sharedSizeBytes;
}

// fkind: the functor kind shared by every solve of the batch, or 0 (mixed)
hipError_t launch_solve(const SolveDesc *descs, int count, int team, int fkind, const LdsPlan &plan,
                        hipStream_t st)
{
    const size_t lds = lds_plan_bytes(plan);
    // a launch whose LDS (static + dynamic) exceeds the workgroup limit is
    // refused here, never sent to the device
    int lds_blk = 0, dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = hipDeviceGetAttribute(&lds_blk, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e != hipSuccess) return e;
    const int stat = solve_static_lds(team, fkind);
    if (stat < 0 || (size_t)stat + lds > (size_t)lds_blk) return hipErrorInvalidValue;
    // team shapes: 256 threads at 256 VGPRs, two solves per CU, and 512 threads
    // at 256 VGPRs, one solve per CU (the defaults, every functor specialized);
    // 1024 threads at 128 VGPRs
    const void *k = solve_kernel_ptr(team, fkind);
    if ((e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) != hipSuccess) return e;
    LdsPlan p = plan;
    void *args[] = {&descs, &count, &p};
    const int nt = team == 64 || team == 512 || team == 1024 ? team : 256;
    if ((e = hipLaunchKernel(k, dim3(count), dim3(nt), args, lds, st)) != hipSuccess) return e;
    return hipGetLastError();
}

hipError_t launch_rrlu(tci_lu_job *jobs, int64_t count, int64_t max_side, double *gstage,
                       int64_t gstage_stride, const int32_t *order, hipStream_t st)
{
    const int cap = 48 * 1024 / 16;
    const size_t lds = max_side <= cap ? (size_t)2 * max_side * sizeof(double) : 0;
    hipLaunchKernelGGL(tci_rrlu_kernel, dim3((unsigned)count), dim3(kTeam), lds, st, jobs, count,
                       max_side <= cap ? (int)max_side : 0, gstage, gstage_stride, order);
    return hipGetLastError();
}

hipError_t launch_rrlu_tile(tci_lu_job *jobs, const int32_t *idx, int64_t count, double *scratch,
                            const int64_t *soff, hipStream_t st)
{
    if (count <= 0) return hipSuccess;
    hipLaunchKernelGGL(tci_rrlu_tile_kernel, dim3((unsigned)count), dim3(kTeam), 0, st, jobs, idx, count,
                       scratch, soff);
    return hipGetLastError();
}

hipError_t launch_lu_unpack(const tci_lu_job *job, int64_t most, double *L, double *U, double *diag, double *UT,
                            hipStream_t st)
{
    if (most <= 0) return hipSuccess;
    hipLaunchKernelGGL(tci_lu_unpack_kernel, dim3((unsigned)std::min<int64_t>((most + 255) / 256, 4096)), dim3(256), 0,
                       st, job, L, U, diag, UT);
    return hipGetLastError();
}

hipError_t launch_kron_center(const uint8_t *left, int64_t nI, int nl, const int32_t *cdims, int M,
                              int64_t nc, uint8_t *rowsx, int stride, hipStream_t st)
{
    int64_t tot = nI * nc;
    if (tot == 0) return hipSuccess;
    int64_t blocks = (tot + 255) / 256;
    if (blocks > 65535) blocks = 65535;
    hipLaunchKernelGGL(tci_kron_center_kernel, dim3((unsigned)blocks), dim3(256), 0, st, left, nI,
                       nl, cdims, M, nc, rowsx, stride);
    return hipGetLastError();
}

int eval_blocks(int64_t tot)
{
    int64_t b = (tot + 255) / 256;
    if (b > 4096) b = 4096;
    if (b < 1) b = 1;
    return (int)b;
}

hipError_t launch_eval(int kind, const double *params, const int32_t *iparams, int L,
                       const uint8_t *rows, int64_t nrow, int rstride, int nl, const uint8_t *cols,
                       int64_t ncol, int cstride, double *out, double *blockmax, hipStream_t st)
{
    int blocks = eval_blocks(nrow * ncol);
    hipLaunchKernelGGL(tci_eval_kernel, dim3(blocks), dim3(256), 0, st, kind, params, iparams, L,
                       rows, nrow, rstride, nl, cols, ncol, cstride, out, blockmax);
    return hipGetLastError();
}

}  // namespace tci
