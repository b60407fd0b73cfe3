// tci_kernels.h — launchers of the gfx950 kernels (defined in tci_kernels.hip).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "../../include/tci.h"
#include "tci_desc.h"

namespace tci {

// on-chip (LDS) placement of one solve workgroup's hot buffers
struct LdsPlan {
    int32_t stage_cap;   // rrLU staging vectors: 2 × stage_cap doubles (0: in HBM)
    int32_t tab_cap;     // bytes per index table (rows, cols) (0: in HBM)
    int32_t sets_cap;    // bytes for the pivot sets and their counts (0: in HBM)
    int32_t lut_cap;     // doubles for the Lorentzian value table (0: none)
    int64_t pi_cap;      // doubles available for a Pi matrix (0: in HBM)
};
size_t lds_plan_bytes(const LdsPlan &p);
// static LDS bytes of the solve kernel variant for (team, functor kind), -1 on error
int solve_static_lds(int team, int fkind);
hipError_t launch_solve(const SolveDesc *descs_device, int count, int team, int fkind,
                        const LdsPlan &plan, hipStream_t st);
// slot-level serving: the queue's control words in coherent host memory
struct ServeCtl {
    uint64_t tail;   // host: tickets published (ring entries valid below it)
    uint32_t stop;   // host: 1 = leave once idle
    uint32_t pad;
};
// the serving grid's own words in device memory (zero when the server starts)
struct ServeDev {
    uint64_t head;       // next ticket to claim
    uint64_t dtail;      // mirror of ServeCtl::tail (only ever raised)
    uint64_t lastpoll;   // wall clock of the last read of the host's words
    uint64_t last;       // wall clock of the last claim or finished solve
    uint32_t busy;       // workgroups running a solve
    uint32_t closing;    // the launch epoch that is leaving for lack of work
    uint32_t dstop;      // the launch epoch that has seen ServeCtl::stop
    uint32_t pad;
};
// one published request (a ring entry in coherent host memory).  The
// claiming workgroup copies the staged image (the descriptor, then the
// inputs) into the device block, runs the solve, and copies the report out
// before it sets the done mark
struct ServeSlot {
    const uint8_t *src;    // the staged image (device alias of pinned host memory)
    uint8_t *dst;          // the request's device block: the descriptor at dst
    const uint8_t *rep;    // the report in the device block
    uint8_t *rep_out;      // its host copy (device alias of pinned host memory)
    uint64_t bytes;        // staged bytes, a multiple of 16
    uint64_t rep_bytes;    // report bytes, a multiple of 16
};
int serve_static_lds(int team);
// a persistent grid of `blocks` workgroups (generic functor kernel) that runs
// published tickets; it leaves, all of it, once stop is set and every
// published ticket is claimed, or once no solve has run, been claimed or
// finished for idle_ticks of the wall clock.  epoch: this launch's number
// (each launch a new one, from 1)
hipError_t launch_serve(const ServeSlot *ring, ServeDev *g, const ServeCtl *ctl, uint64_t *done, int cap,
                        const LdsPlan &plan, uint64_t idle_ticks, uint32_t epoch, int team, int blocks,
                        hipStream_t st);
// order (device, count entries, or null): the job index each workgroup takes
hipError_t launch_rrlu(tci_lu_job *jobs_device, int64_t count, int64_t max_side, double *gstage,
                       int64_t gstage_stride, const int32_t *order, hipStream_t st);
// The site tensors and index sets of finished solves, packed for one download:
// block (q, site) copies solve[q]'s site tensor and its four index sets (Iset,
// Jset and their last history entries, entries back to back) to out + the five
// byte offsets at[5·(q·L0 + site) ...]; L0: the largest L of the solves.
hipError_t launch_pack(const SolveDesc *descs, const int32_t *solve, int count, int L0, const int64_t *at,
                       uint8_t *out, hipStream_t st);
// the register-tile rrLU of the jobs idx[0..count) (each m, n <= 128);
// scratch + soff[q]: m·mr + mr·n doubles for job idx[q] (mr = min(m, n, maxrank))
constexpr int kTileSide = 128;
hipError_t launch_rrlu_tile(tci_lu_job *jobs_device, const int32_t *idx, int64_t count, double *scratch,
                            const int64_t *soff, hipStream_t st);
// rrlu!(A) of matrices held on chip by teams of workgroups
// (tci_rrlu_chip.hip), sides up to kGridMaxSide
constexpr int kGridMaxSide = 8192;
struct ChipItem {
    int32_t job;          // index into the job table
    int32_t shape, wr;    // register shape and wave rows
    int32_t S;            // members of the team
    int32_t first;        // the job's first ticket (its S tickets follow each other)
};
struct ChipArgs {
    tci_lu_job *jobs;
    const ChipItem *items;
    const int32_t *map;      // ticket → item
    int32_t ntickets;
    uint32_t *ticket;        // next ticket (zero on entry)
    uint32_t *abort_word;    // zero on entry; not zero: a member has given up a wait
    uint64_t wait_ticks;     // the longest wait (100 MHz wall clock)
    uint64_t *mail;          // 8 words per ticket (zero on entry)
    double *cols;            // 2 × colcap per workgroup (rrlu_chip_blocks of them)
    int64_t colcap;          // rows of the tallest job
    double *spill;           // spillcap per workgroup of the big kernel
    int64_t spillcap;
};
// the team for an m×n matrix (it->shape, wr and S): 1 the two-per-CU kernel, 2
// the big one, 0 when neither takes it
int rrlu_chip_plan(int64_t m, int64_t n, int ncu, ChipItem *it);
// doubles of spill a member of the big kernel needs
int64_t rrlu_chip_spill(const ChipItem &it, int64_t m, int64_t n);
// workgroups of a launch of ntickets tickets (0: the kernel does not fit the device)
int rrlu_chip_blocks(int big, int ncu, int ntickets);
hipError_t launch_rrlu_chip(const ChipArgs &K, int big, int blocks, hipStream_t st);
// One whole TT sweep of factorizations (the host-driven sweep's steps, the
// same operations per entry) in a single workgroup, for trains whose bonds
// are small enough that per-bond host round trips would dominate
struct TtSweepArgs {
    int32_t L, method, forward, stage_cap;   // stage_cap: doubles per LDS staging vector
    int32_t mat_cap;                         // doubles of LDS for the bond matrix (0: factored in place)
    int64_t maxrank, R;                      // R: the largest bond on entry (pivot slots per bond: 2R)
    double reltol, abstol;
    int64_t *links;                          // device, L+1; each bond's new dimension written back
    const int32_t *d;                        // device, L
    const int64_t *off;                      // device, L: each site's slot in cores (doubles)
    double *cores, *wl, *wu, *wc, *wp, *gstage;
    int32_t *perm;                           // device, m+n of the largest bond
    int32_t *piv;                            // device, (L-1)·2R: bond b's row, then column pivots (1-based)
    double *pe;                              // device, R+1: running pivot errors (zero on entry)
    int32_t *status;                         // device, 2: status and bond of a NaN verdict (zero on entry)
};
hipError_t launch_tt_sweep(const TtSweepArgs &a, hipStream_t st);
// C = A·B with each sum in ascending k (M×K · K×N, column-major)
hipError_t launch_gemm(int64_t M, int64_t N, int64_t K, const double *A, int64_t lda, const double *B, int64_t ldb,
                       double *Cm, int64_t ldc, hipStream_t st);
// left(luci) (m×p, ld ldl) and right(luci) (p×n, ld ldr) of MatrixLUCI from
// the unpacked L (m×p) and U (p×n), U11 transposed (p×p, needed without leftorth
// up to kLuciSolveMax) and the 1-based permutations
constexpr int64_t kLuciSolveMax = 256;   // 128 KiB of LDS
hipError_t launch_luci(int64_t m, int64_t n, int64_t p, int leftorth, const int32_t *rowperm, const int32_t *colperm,
                       const double *L, const double *U, const double *UT, double *left, int64_t ldl, double *right,
                       int64_t ldr, hipStream_t st);
// left(lu)/right(lu) with the permutations applied, from the unpacked L, U
hipError_t launch_lu_permute(int64_t m, int64_t n, int64_t p, const int32_t *rowperm, const int32_t *colperm,
                             const double *L, const double *U, double *left, int64_t ldl, double *right, int64_t ldr,
                             hipStream_t st);
// the factors of a finished job (its rank is read on the device): L m×p and U p×n
// with leading dimensions m and p (U null: right behind L), diag the p pivots and
// UT U11 transposed, p×p (null: not wanted); most: an upper bound of (m + n + 1)·p
hipError_t launch_lu_unpack(const tci_lu_job *job, int64_t most, double *L, double *U, double *diag, double *UT,
                            hipStream_t st);
hipError_t launch_kron_center(const uint8_t *left, int64_t nI, int nl, const int32_t *cdims, int M,
                              int64_t nc, uint8_t *rowsx, int stride, hipStream_t st);
int eval_blocks(int64_t tot);
// TT evaluation at npts points (and f, |TT - f| and |f| maxima when fkind != 0);
// blockmax holds 2 doubles per block of tt_eval_points_per_block(chimax) points
int tt_eval_points_per_block(int chimax);
hipError_t launch_tt_eval(int L, const int64_t *dims3, const int64_t *coff, const double *cores,
                          const uint8_t *pts, int64_t npts, int chimax, int fkind, const double *params,
                          const int32_t *iparams, double *out_tt, double *out_f, double *blockmax,
                          hipStream_t st);
// TT evaluation of many points, site by site over points grouped by local index:
// bins (256 per site, zero on entry), tiles and ntiles (maxtiles >= npts/64 + the
// largest local dimension, per site) and order (npts per site) are filled by
// launch_tt_group; launch_tt_site forms one site's vectors W from V (stride
// doubles per point; V null at the first site) for d0 <= kTtSiteMax;
// launch_tt_finish reads V's first entries out (two block maxima per 256 points)
struct TtTile {
    int32_t s, first, n;
};
constexpr int kTtSiteMax = 256;
hipError_t launch_tt_group(const uint8_t *pts, int64_t npts, int L, int32_t *bins, TtTile *tiles, int32_t *ntiles,
                           int maxtiles, int32_t *order, hipStream_t st);
hipError_t launch_tt_site(const double *T, int d0, int d, int d2, const TtTile *tiles, const int32_t *ntiles,
                          int maxtiles, const int32_t *order, const double *V, double *W, int stride, hipStream_t st);
hipError_t launch_tt_finish(const double *V, int stride, const uint8_t *pts, int64_t npts, int L, int fkind,
                            const double *params, const int32_t *iparams, double *out_tt, double *out_f,
                            double *blockmax, hipStream_t st);
// _floatingzone from each of npts points (in/out, npts×L digits), one
// workgroup per point; work: wstride doubles per workgroup, digits: dmax·L
// bytes per workgroup; roff: L+1 offsets of the right environments
// the floating-zone search: points and errors in place, the train as dims3 (three
// per site), its cores' offsets coff, the environments' offsets roff
struct FzArgs {
    int L, chimax, dmax, fkind;
    int nft;              // per-site term functions of f (0: f evaluated as a whole)
    int nslice;           // doubles of the slices kept in LDS (0: none)
    const int64_t *dims3, *coff, *roff;
    const double *cores, *params, *ftab;
    const int32_t *iparams;
    uint8_t *pts;
    double *errs;
    int64_t npts, nsweeps;
    double earlystoptol;
    double *work;         // per workgroup wstride doubles, when LDS does not hold them
    int64_t wstride, nenv;
};
// LDS of the search: at most kFzLds, with the slices at most kFzSliceLds
constexpr size_t kFzLds = 60 * 1024, kFzSliceLds = 19 * 1024;
// bytes of a workgroup's work area without the slices
inline size_t fz_area_bytes(const FzArgs &a)
{
    const size_t dbl = (size_t)a.nenv + 2 * (size_t)a.dmax * a.chimax + (size_t)a.dmax + (size_t)a.nft * (a.dmax + a.L);
    return sizeof(double) * dbl + (a.nft ? 0 : (((size_t)a.dmax * a.L + 7) & ~(size_t)7));
}
// slice: doubles of all T_b[:, x_b, :] beyond the first site
hipError_t launch_floatingzone(FzArgs a, int64_t slice, int blocks, double *ftab, hipStream_t st);
hipError_t launch_eval(int kind, const double *params, const int32_t *iparams, int L,
                       const uint8_t *rows, int64_t nrow, int rstride, int nl, const uint8_t *cols,
                       int64_t ncol, int cstride, double *out, double *blockmax, hipStream_t st);

}  // namespace tci
