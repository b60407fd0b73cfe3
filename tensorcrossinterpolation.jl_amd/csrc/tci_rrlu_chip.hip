// tci_rrlu_chip.hip — rrlu!(A) (matrixlu.jl:141-181) with the matrix held on
// chip by a team of workgroups.
//
// What bounds full pivoting is that every pivot touches the whole trailing
// block: streamed from memory that is 16 bytes per entry and pivot.  The
// register files of the chip hold 128 MiB, so here a matrix is spread over the
// registers of as many workgroups as it needs (its team): it is read once,
// factored in place and written once.  Per pivot only the pivot column and one
// candidate per workgroup travel between workgroups.
//
// Layout.  Member g of a team of S owns the columns j ≡ g (mod S), all rows.
// Its waves form WR wave rows × WC wave columns; wave (wr, wc), lane l holds
// the rows l + 64·(wr + WR·i), i < RA, of its columns c = wc + WC·j, j < CB
// (global column g + S·c).  Rows and columns never move: every thread tracks
// the current positions of its rows (rp), lane j of a wave the position of the
// wave's register column j (cpl), and pivoted rows and columns get NaN
// multipliers, so their entries drop out of every later search (as in
// tci_regtile.h, whose arithmetic and tie-breaking this follows).
//
// One pivot:
//   1. each member finds its best candidate (largest square, then the first
//      position in column-major order), writes the candidate's column to its
//      column buffer and then the candidate to its mailbox;
//   2. every member reads the S mailboxes: all agree on the pivot and on the
//      stop test, and read the winner's column from the winner's buffer;
//   3. each member updates its entries and takes their maximum in one pass.
// Finished entries (the pivot row, the pivot column) are stored where they lie
// in A; at the end each member reads those back, and once all members have
// done so the team writes rrlu!'s packed matrix, every entry at its final
// position.  The mailboxes are double buffered: a member writes round r only
// after it has seen everybody's round r - 1, which they write after they are
// done with round r - 2.
//
// Mailboxes and column buffers are written and read with agent-scope accesses
// (coherent across the XCDs); a mailbox's three words carry the round number
// each, so they validate themselves, and they are written after the column
// stores have been acknowledged.
//
// A launch takes any list of jobs.  Each job has as many tickets as its team
// has members; a workgroup draws tickets in order until none is left.  A
// member waits only for members of its own team, whose tickets are drawn no
// later than any ticket after them, so the earliest unfinished job always
// finishes as long as the largest team fits the device at once (the launch is
// cooperative, so the whole grid does).  Every wait is bounded all the same: a
// member that waits longer than ChipArgs::wait_ticks gives up and tells the others.
// The workgroups go on drawing tickets: every job whose team has given up, and every
// team's job drawn after that, reports TCI_ERR_DEVICE, so no job is left as it was.
//
// tci_rrlu_chip_kernel runs two workgroups of four waves per CU, one of them
// working while the other waits for its team.  Matrices that need more
// workgroups than the device holds go to tci_rrlu_chip_big_kernel: one
// workgroup of eight waves per CU, whose columns beyond the registers are kept
// in LDS and beyond that where they lie in memory.
//
// What bounds it now (MI355X): a pivot takes about 6 us, of which 1.3 are the
// update and 3.5 the three dependent round trips between XCDs (column stores
// acknowledged, mailbox seen, winner's column read); the big kernel adds the
// streaming of the columns in memory, at about 6 TB/s.  1024 matrices of 32 to
// 1024 rows and columns, rank 8 to 128: 118.2 -> 20.0 ms a pass against the
// streaming kernel (one workgroup per matrix, 16 B per entry and pivot); one
// 1024 x 1024 matrix of rank 64: 2.3 -> 0.55 ms, one 4352 x 4352 with 256
// pivots: 21.8 -> 7.2 ms against a grid-wide kernel that streamed the matrix
// once per pivot (81 us a pivot, 303 MB each).
#include <hip/hip_runtime.h>

#include "tci_devteam.h"
#include "tci_kernels.h"

namespace tci {

constexpr int kChipMaxCB = 42;
constexpr int kChipMaxExtra = 64;                    // columns of a member outside its registers
constexpr int kChipColLds = 1024;                    // rows of a lone member's column kept in LDS
constexpr int kChipL2Share = 14000;                  // doubles of L2 a member of the big kernel may count on
constexpr uint32_t kChipNone = 0xffffffffu;
constexpr int kChipOut = 0xffff;                     // position of a row or column that does not exist
constexpr int kChipFail = 3;                         // word of member 0's mailbox: a member has given up

// Pointers into device memory carry their address space: through generic ones
// every access would also count as an LDS operation, and each barrier would wait
// for the stores in flight.
using GDbl = __attribute__((address_space(1))) double;
using GU64 = __attribute__((address_space(1))) uint64_t;
using GU32 = __attribute__((address_space(1))) uint32_t;
using GI32 = __attribute__((address_space(1))) int32_t;

struct ChipRed {
    double v, a;
    uint32_t key, blk;
};

template <int NW>
struct ChipLds {
    double y[NW][kChipMaxCB];      // the pivot row, per wave column
    double ye[kChipMaxExtra];      // its entries in the columns outside registers
    double wmax[NW];
    uint32_t wkey[NW];
    ChipRed red[NW];
    double av;                     // value of this member's candidate
    int32_t ecp[kChipMaxExtra];    // positions of the columns outside registers
    int32_t abort;
    int32_t ticket;
    double col[kChipColLds];
};

__device__ __forceinline__ void agent_put(GU64 *p, uint64_t v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ uint64_t agent_get(const GU64 *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A mailbox: [a low | round] [a high | round] [key 26 bits | workgroup 10 | round 28]
__device__ __forceinline__ void mail_put(GU64 *s, double a, uint32_t key, uint32_t blk, uint32_t round)
{
    const uint64_t b = (uint64_t)__double_as_longlong(a);
    agent_put(s + 0, (b & 0xffffffffULL) | ((uint64_t)round << 32));
    agent_put(s + 1, (b >> 32) | ((uint64_t)round << 32));
    agent_put(s + 2, (uint64_t)(key & 0x3ffffffu) | ((uint64_t)blk << 26) | ((uint64_t)round << 36));
}

// waits for a member's mailbox of this round; false when the wait was given up
__device__ __forceinline__ bool mail_get(const GU64 *s, uint32_t round, const ChipArgs &K, double &a,
                                         uint32_t &key, uint32_t &blk)
{
    GU32 *abort_word = (GU32 *)K.abort_word;
    const uint32_t every = K.wait_ticks ? 0xfffu : 0u;   // polls between looks at the clock
    uint64_t t0 = 0;
    for (uint32_t spin = 0;; ++spin) {
        const uint64_t w0 = agent_get(s), w1 = agent_get(s + 1), w2 = agent_get(s + 2);
        if ((uint32_t)(w0 >> 32) == round && (uint32_t)(w1 >> 32) == round && (uint32_t)(w2 >> 36) == round) {
            a = __longlong_as_double((long long)((w0 & 0xffffffffULL) | (w1 << 32)));
            key = (uint32_t)w2 & 0x3ffffffu;
            blk = (uint32_t)(w2 >> 26) & 0x3ffu;
            return true;
        }
        if ((spin & every) == every) {
            const uint64_t now = (uint64_t)wall_clock64();
            if (t0 == 0) t0 = now;
            if (now - t0 >= K.wait_ticks)
                __hip_atomic_store(abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (__hip_atomic_load(abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0) return false;
        }
    }
}

// A job's status and rank, written past this XCD's L2 and acknowledged: members on
// several XCDs may write them (chip_failed)
__device__ __forceinline__ void job_put(tci_lu_job &J, int32_t status, int64_t npivot)
{
    __hip_atomic_store((GI32 *)&J.status, status, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    agent_put((GU64 *)&J.npivot, (uint64_t)npivot);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// One member's part of one job.  EX: columns beyond the registers are kept in
// LDS (exl, exl_cap doubles) and then in memory; spill: their place during the
// final rearrangement.  Requires 64·WR·RA >= m, sides at most 8192 and
// ceil(n / S) <= WC·CB (+ kChipMaxExtra with EX, where WC = 1).  Returns false
// when a wait was given up.
//
// Rows are addressed as a wave-uniform pointer (column and row block) plus one
// 32-bit row number per thread, so the unrolled accesses need no address
// registers of their own.
template <int NW, int RA, int CB, bool EX>
__device__ __forceinline__ bool chip_job(const ChipArgs &K, ChipLds<NW> &sh, double *exl, int64_t exl_cap,
                                         tci_lu_job &J, const int S, const int g, const int WR,
                                         GU64 *__restrict__ mail)
{
    constexpr int NT = 64 * NW;
    DevTeam<NT, 2> tm;
    const double NaN = 0.0 / 0.0;
    const int tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int WC = EX ? 1 : NW / WR, wr = EX ? wave : wave % WR, wc = EX ? 0 : wave / WR;
    const uint32_t me = blockIdx.x;
    const int m = (int)J.m, n = (int)J.n;
    GDbl *__restrict__ A = (GDbl *)J.A;
    const bool lo = J.leftorth != 0;
    const double reltol = J.reltol, abstol = J.abstol;
    int mr = m < n ? m : n;
    if (J.maxrank < mr) mr = (int)J.maxrank;
    const int64_t lda = m;
    const uint32_t row0 = (uint32_t)(lane + 64 * wr);                      // row i: row0 + rstep·i
    const int rstep = EX ? 64 * NW : 64 * WR;
    const int col0 = g + S * wc, cstep = S * WC;                           // column j: col0 + cstep·j
    GU64 *mycol = (GU64 *)K.cols + (int64_t)me * 2 * K.colcap;
    const bool lone = !EX && S == 1 && m <= kChipColLds;                   // the column stays in LDS
    const auto inrow = [&](int i) { return (int)row0 < m - rstep * i; };   // row i exists
    // row i, or the last one where it does not exist: loads that need no branch
    // (recomputed at each use: held across the loop they would cost RA registers)
    const auto rowc = [&](int i) {
        int r = (int)row0;
        asm("" : "+v"(r));
        r += rstep * i;
        return (uint32_t)(r < m ? r : m - 1);
    };

    double a[RA][CB];
    int rp[RA], cpl;
#pragma unroll
    for (int i = 0; i < RA; ++i) rp[i] = inrow(i) ? (int)row0 + rstep * i : kChipOut;
    {
        const int c = col0 + cstep * lane;
        cpl = (lane < CB && c < n) ? c : kChipOut;
    }
    // the running maximum of |entry| in groups of columns (-1: none), so the
    // scan for the maximum's position looks at one group
    constexpr int NG = EX ? 2 : 4, GW = (CB + NG - 1) / NG;
    double lg[NG], lmax, lmaxe = -1.0;
    uint64_t emask = 0;   // columns outside the registers whose maximum is about lmaxe
#pragma unroll
    for (int q = 0; q < NG; ++q) lg[q] = -1.0;
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const int c = col0 + cstep * j;
        const GDbl *src = A + lda * (c < n ? c : 0);
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            double v = NaN;
            if (c < n && inrow(i)) v = (src + rstep * i)[row0];
            a[i][j] = v;
        }
    }
#pragma unroll
    for (int j = 0; j < CB; ++j)
#pragma unroll
        for (int i = 0; i < RA; ++i) lg[j / GW] = fmax(lg[j / GW], fabs(a[i][j]));
    // the columns outside the registers: e < nl in LDS, e < nex in memory
    // (local column CB + e is global g + S·(CB + e))
    constexpr int MP = 64 * NW * RA;   // rows of a column in LDS (EX), NaN beyond m
    int nex = 0, nl = 0, nl2 = 0;
    const auto excol = [&](int e) { return g + S * (CB + e); };
    // a thread's column maximum cm joins the running maximum; emask keeps the
    // columns within 2^-50 of it (entries of equal squares are closer than that
    // unless the square is subnormal or infinite, where every column is scanned)
    const auto emax = [&](int e, double cm) {
        if (cm > lmaxe) {
            emask = lmaxe >= cm * (1.0 - 0x1p-50) ? emask | (1ULL << e) : 1ULL << e;
            lmaxe = cm;
        } else if (cm >= lmaxe * (1.0 - 0x1p-50)) {
            emask |= 1ULL << e;
        }
    };
    if (EX) {
        const int own = g < n ? (n - g + S - 1) / S : 0;
        nex = own > CB ? own - CB : 0;
        const int fit = (int)(exl_cap / MP);
        nl = nex < fit ? nex : fit;
        nl2 = (int)(kChipL2Share / m);
        for (int e = tid; e < nex; e += NT) sh.ecp[e] = excol(e);
        for (int e = 0; e < nex; ++e) {
            const GDbl *src = A + lda * excol(e);
            double v[RA], cm = -1.0;
#pragma unroll
            for (int i = 0; i < RA; ++i) v[i] = src[rowc(i)];
#pragma unroll
            for (int i = 0; i < RA; ++i) {
                if (!inrow(i)) v[i] = NaN;
                cm = fmax(cm, fabs(v[i]));
                if (e < nl) exl[e * MP + rstep * i + (int)row0] = v[i];
            }
            emax(e, cm);
        }
    }

    double maxerr = 0.0, err = NaN;
    int p = 0, nanx = 0, nany = 0;
    uint32_t seen = 0;      // the last round read from every member
    int jw = -1, ew = -1;   // my candidate's column, when this wave holds it
    bool ok = true;
    while (p < mr) {
        const int k = p;
        // ---- this member's candidate: the largest |entry|, then the first
        // position among the entries of the same square
        lmax = lg[0];
#pragma unroll
        for (int q = 1; q < NG; ++q) lmax = fmax(lmax, lg[q]);
        double gm = tm.wave_max(EX ? fmax(lmax, lmaxe) : lmax);
        if (EX) {
            // the columns outside the registers make a scan long: only the waves
            // that hold the member's maximum scan, at the price of a barrier
            if (lane == 0) sh.wmax[wave] = gm;
            __syncthreads();
            gm = sh.wmax[0];
#pragma unroll
            for (int q = 1; q < NW; ++q) gm = fmax(gm, sh.wmax[q]);
            gm = tm.uniform_f64(gm);
        }
        const double G = gm >= 0.0 ? gm * gm : -1.0;
        uint32_t kw = kChipNone;
        {
            uint32_t kl = kChipNone;
#pragma unroll
            for (int q = 0; q < NG; ++q) {
                if (!tm.wave_any(lg[q] * lg[q] == G)) continue;
#pragma unroll
                for (int j = q * GW; j < (q + 1) * GW && j < CB; ++j) {
                    const uint32_t ck = (uint32_t)tm.wave_bcast(cpl, j) << 13;
#pragma unroll
                    for (int i = 0; i < RA; ++i) {
                        const double v = a[i][j];
                        kl = eng_umin(kl, v * v == G ? ck | (uint32_t)rp[i] : kChipNone);
                    }
                }
            }
            if (EX) {
                const bool minee = lmaxe * lmaxe == G && lmaxe >= 0.0;
                const bool all = !(G >= 0x1p-1022 && G < __builtin_inf());   // (emask does not tell)
                for (int e = 0; e < nex; ++e) {
                    if (!tm.wave_any(minee && (all || ((emask >> e) & 1)))) continue;
                    const int c = sh.ecp[e];
                    if (c < k) continue;
                    const GDbl *src = A + lda * excol(e);
                    double v[RA];
                    if (e < nl) {
#pragma unroll
                        for (int i = 0; i < RA; ++i) v[i] = exl[e * MP + rstep * i + (int)row0];
                    } else {
#pragma unroll
                        for (int i = 0; i < RA; ++i) v[i] = src[rowc(i)];
                    }
#pragma unroll
                    for (int i = 0; i < RA; ++i)
                        kl = eng_umin(kl, v[i] * v[i] == G && rp[i] >= k && rp[i] < m
                                              ? ((uint32_t)c << 13) | (uint32_t)rp[i] : kChipNone);
                }
            }
            kw = tm.wave_min(kl);
        }
        if (lane == 0) {
            if (!EX) sh.wmax[wave] = G;
            sh.wkey[wave] = kw;
        }
        __syncthreads();
        uint32_t key = sh.wkey[0];
        {
            double gb = sh.wmax[0];
#pragma unroll
            for (int q = 1; q < NW; ++q) {
                const uint32_t kq = sh.wkey[q];
                if (EX) {
                    key = eng_umin(key, kq);
                } else {
                    const double gq = sh.wmax[q];
                    if (gq > gb || (gq == gb && kq < key)) { gb = gq; key = kq; }
                }
            }
        }
        key = tm.uniform_u32(key);
        jw = ew = -1;
        const int par = (int)(seen & 1u);   // buffer of round seen + 1
        if (key != kChipNone) {
            const int cpos = (int)(key >> 13), rpos = (int)(key & 8191u);
            jw = tm.wave_first(lane < CB && cpl == cpos);
            if (EX && jw < 0)
                for (int e = 0; e < nex; ++e)
                    if (sh.ecp[e] == cpos) ew = e;
            if (jw >= 0 || (EX && ew >= 0)) {
                double cv[RA];
#pragma unroll
                for (int i = 0; i < RA; ++i) cv[i] = a[i][0];
#pragma unroll
                for (int j = 1; j < CB; ++j)
                    if (j == jw) {
#pragma unroll
                        for (int i = 0; i < RA; ++i) cv[i] = a[i][j];
                    }
                if (EX && jw < 0) {
                    const GDbl *src = A + lda * excol(ew);
                    if (ew < nl) {
#pragma unroll
                        for (int i = 0; i < RA; ++i) cv[i] = exl[ew * MP + rstep * i + (int)row0];
                    } else {
#pragma unroll
                        for (int i = 0; i < RA; ++i) cv[i] = src[rowc(i)];
                    }
                }
                GU64 *dst = mycol + par * K.colcap;
#pragma unroll
                for (int i = 0; i < RA; ++i) {
                    if (inrow(i)) {
                        if (lone) (sh.col + rstep * i)[row0] = cv[i];
                        else agent_put(&(dst + rstep * i)[row0], (uint64_t)__double_as_longlong(cv[i]));
                    }
                    if (rp[i] == rpos) sh.av = cv[i];
                }
            }
        } else if (tid == 0) {
            sh.av = NaN;
        }
        // the column stores are acknowledged before the mailbox is written
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        // ---- the team's pivot
        double av;
        uint32_t blk = me;
        if (S > 1) {
            if (tid == 0) mail_put(mail + (int64_t)8 * g + 4 * par, sh.av, key, me, seen + 1);
            ChipRed c;
            c.v = -1.0;
            c.a = NaN;
            c.key = kChipNone;
            c.blk = 0;
            for (int q = tid; q < S; q += NT) {
                double qa;
                uint32_t qk, qb;
                if (!mail_get(mail + (int64_t)8 * q + 4 * par, seen + 1, K, qa, qk, qb)) {
                    sh.abort = 1;
                    break;
                }
                const double qv = qa * qa;
                if (qv > c.v || (qv == c.v && qk < c.key)) {   // (a NaN is no candidate)
                    c.v = qv;
                    c.a = qa;
                    c.key = qk;
                    c.blk = qb;
                }
            }
            const double vm = tm.wave_max(c.v);
            const uint32_t km = tm.wave_min(c.v == vm ? c.key : kChipNone);
            const int wl = tm.wave_first(c.v == vm && c.key == km);
            if (lane == 0) {
                sh.red[wave].v = vm;
                sh.red[wave].key = km;
            }
            if (lane == wl) {
                sh.red[wave].a = c.a;
                sh.red[wave].blk = c.blk;
            }
            __syncthreads();
            if (sh.abort) { ok = false; break; }
            c = sh.red[0];
            const int nred = S < NT ? (S + 63) / 64 : NW;   // the waves that read a mailbox
            for (int q = 1; q < nred; ++q) {
                const ChipRed o = sh.red[q];
                if (o.v > c.v || (o.v == c.v && o.key < c.key)) c = o;
            }
            key = c.v >= 0.0 ? tm.uniform_u32(c.key) : kChipNone;
            av = tm.uniform_f64(c.a);
            blk = tm.uniform_u32(c.blk);
        } else {
            av = tm.uniform_f64(sh.av);
        }
        ++seen;
        const bool cand = key != kChipNone;
        if (!cand) av = NaN;
        const double e = fabs(av);
        err = e;
        if ((e < reltol * maxerr || e < abstol) && p > 0) break;
        maxerr = jl_max(maxerr, e);
        const int pr = cand ? (int)(key & 8191u) : k, pc = cand ? (int)(key >> 13) : k;
        const bool won = cand && blk == me;
        // ---- x: the pivot column, divided by the pivot when leftorth
        double x[RA];
        if (lone) {
#pragma unroll
            for (int i = 0; i < RA; ++i) x[i] = sh.col[rowc(i)];
        } else {
            const GU64 *src = (const GU64 *)K.cols + ((int64_t)blk * 2 + par) * K.colcap;
#pragma unroll
            for (int i = 0; i < RA; ++i) x[i] = __longlong_as_double((long long)agent_get(&src[rowc(i)]));
        }
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            rp[i] = rp[i] == k ? pr : (rp[i] == pr ? k : rp[i]);
            const bool live = rp[i] > k && rp[i] < m;
            double v = NaN;
            if (cand && live) v = lo ? x[i] / av : x[i];
            if (live && v != v) nanx = 1;
            x[i] = v;
        }
        cpl = cpl == k ? pc : (cpl == pc ? k : cpl);
        if (EX && wave == 0)
            for (int q = lane; q < nex; q += 64) {
                const int c = sh.ecp[q];
                sh.ecp[q] = c == k ? pc : (c == pc ? k : c);
            }
        if (av != av) { nanx = 1; nany = 1; }
        // the finished L column, where it lies (write-through, as the pivot
        // row below: nothing is left dirty in this XCD's L2 where another
        // member writes the final value later)
        if (won && (jw >= 0 || (EX && ew >= 0))) {
            GU64 *dst = (GU64 *)A + lda * (jw >= 0 ? col0 + cstep * jw : excol(ew));
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (rp[i] > k && rp[i] < m)
                    agent_put(&(dst + rstep * i)[row0], (uint64_t)__double_as_longlong(x[i]));
        }
        if (EX && nex) __syncthreads();   // the positions in ecp
        // ---- y: the pivot row, from the wave of each wave column that holds it
        int hl = -1, hi = 0;
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            const int l = tm.wave_first(rp[i] == k);
            if (l >= 0) { hl = l; hi = i; }
        }
        if (hl >= 0) {
            const int orow = hl + 64 * wr + rstep * hi;
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (i == hi && lane == hl) {
#pragma unroll
                    for (int j = 0; j < CB; ++j) sh.y[wc][j] = a[i][j];
                }
            tm.wave_sync_lds();
            if (lane < CB) {
                double y = NaN;
                GU64 *at = (GU64 *)A + orow + lda * (col0 + cstep * lane);
                if (cpl > k && cpl < n) {
                    y = sh.y[wc][lane];
                    if (!lo) y = y / av;
                    if (y != y) nany = 1;
                    agent_put(at, (uint64_t)__double_as_longlong(y));
                } else if (cpl == k) {
                    agent_put(at, (uint64_t)__double_as_longlong(av));
                }
                sh.y[wc][lane] = cand ? y : NaN;
            }
            if (EX)
                for (int q = lane; q < nex; q += 64) {
                    const int c = sh.ecp[q];
                    GDbl *at = A + orow + lda * excol(q);
                    if (c > k) {
                        double y;
                        if (q < nl) y = exl[q * MP + orow];
                        else y = *at;
                        if (!lo) y = y / av;
                        if (y != y) nany = 1;
                        *at = y;
                        sh.ye[q] = cand ? y : NaN;
                    } else if (c == k) {
                        *at = av;
                    }
                }
        }
        __syncthreads();
        // ---- A -= x·y, product and difference rounded apart, with the maximum
#pragma unroll
        for (int q = 0; q < NG; ++q) lg[q] = -1.0;
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const double yj = sh.y[wc][j];
#pragma unroll
            for (int i = 0; i < RA; ++i) {
                const double t = x[i] * yj;
                const double u = a[i][j] - t;
                a[i][j] = u;
                lg[j / GW] = fmax(lg[j / GW], fabs(u));
            }
        }
        if (EX) {
            lmaxe = -1.0;
            emask = 0;
            for (int q = 0; q < nl; ++q) {
                if (sh.ecp[q] <= k) continue;
                const double yj = sh.ye[q];
                double v[RA], cm = -1.0;
#pragma unroll
                for (int i = 0; i < RA; ++i) v[i] = exl[q * MP + rstep * i + (int)row0];
#pragma unroll
                for (int i = 0; i < RA; ++i) {
                    const double t = x[i] * yj;
                    const double u = v[i] - t;
                    exl[q * MP + rstep * i + (int)row0] = u;
                    cm = fmax(cm, fabs(u));
                }
                emax(q, cm);
            }
            // the first of these columns stay in this XCD's L2 from pivot to
            // pivot; the others are streamed past it, so they do not evict them
            for (int q = nl; q < nex; ++q) {
                if (sh.ecp[q] <= k) continue;
                const double yj = sh.ye[q];
                GDbl *c = A + lda * excol(q);
                const bool keep = q < nl + nl2;
                double v[RA], cm = -1.0;
                if (keep) {
#pragma unroll
                    for (int i = 0; i < RA; ++i) v[i] = c[rowc(i)];
                } else {
#pragma unroll
                    for (int i = 0; i < RA; ++i) v[i] = __builtin_nontemporal_load(&c[rowc(i)]);
                }
#pragma unroll
                for (int i = 0; i < RA; ++i) {
                    const double t = x[i] * yj;
                    const double u = v[i] - t;
                    v[i] = u;
                    if (rp[i] > k && rp[i] < m) cm = fmax(cm, fabs(u));
                }
                // (rows that are done keep their finished entry)
                if (keep) {
#pragma unroll
                    for (int i = 0; i < RA; ++i)
                        if (rp[i] > k && rp[i] < m) (c + rstep * i)[row0] = v[i];
                } else {
#pragma unroll
                    for (int i = 0; i < RA; ++i)
                        if (rp[i] > k && rp[i] < m) __builtin_nontemporal_store(v[i], &(c + rstep * i)[row0]);
                }
                emax(q, cm);
            }
        }
        p = k + 1;
    }
    if (!ok) return false;
    // ---- the packed matrix: finished entries read back from where they lie,
    // then, once every member has them, each entry to its final position
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const int c = tm.wave_bcast(cpl, j);
        if (c < n) {
            const GU64 *src = (const GU64 *)A + lda * (col0 + cstep * j);
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (rp[i] < m && (c < p || rp[i] < p))
                    a[i][j] = __longlong_as_double((long long)agent_get(&(src + rstep * i)[row0]));
        }
    }
    GDbl *sp = nullptr;
    if (EX) {
        sp = (GDbl *)K.spill + (int64_t)me * K.spillcap;
        for (int q = 0; q < nex; ++q) {
            const int c = sh.ecp[q];
            const GDbl *src = A + lda * excol(q);
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (inrow(i)) {
                    if (q >= nl) (sp + (int64_t)(q - nl) * m + rstep * i)[row0] = (src + rstep * i)[row0];
                    else if (c < p || rp[i] < p)
                        exl[q * MP + rstep * i + (int)row0] =
                            __longlong_as_double((long long)agent_get(&((const GU64 *)src + rstep * i)[row0]));
                }
        }
    }
    const int nanL = __syncthreads_or(nanx);
    int nanU = __syncthreads_or(nany);
    if (S > 1) {
        // every read of A is complete before the round that lets it be
        // overwritten; columns updated in memory leave this XCD's L2 first
        if (EX) __threadfence();
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        const int par = (int)(seen & 1u);
        if (tid == 0) mail_put(mail + (int64_t)8 * g + 4 * par, 0.0, nanU ? 1u : 0u, me, seen + 1);
        int any = 0;
        for (int q = tid; q < S; q += NT) {
            double qa;
            uint32_t qk, qb;
            if (!mail_get(mail + (int64_t)8 * q + 4 * par, seen + 1, K, qa, qk, qb)) {
                sh.abort = 1;
                break;
            }
            any |= (int)qk;
        }
        nanU = __syncthreads_or(any);
        if (sh.abort) return false;
    }
#pragma unroll
    for (int j = 0; j < CB; ++j) {
        const int c = tm.wave_bcast(cpl, j);
        if (c < n) {
            GDbl *dst = A + lda * c;
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (rp[i] < m) dst[(uint32_t)rp[i]] = a[i][j];
        }
    }
    if (EX)
        for (int q = 0; q < nex; ++q) {
            const int c = sh.ecp[q];
            GDbl *dst = A + lda * c;
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (inrow(i)) {
                    if (q < nl) dst[(uint32_t)rp[i]] = exl[q * MP + rstep * i + (int)row0];
                    else dst[(uint32_t)rp[i]] = (sp + (int64_t)(q - nl) * m + rstep * i)[row0];
                }
            if (tid == 0) ((GI32 *)J.colperm)[c] = excol(q) + 1;
        }
    if (wr == 0 && lane < CB && cpl < n) ((GI32 *)J.colperm)[cpl] = col0 + cstep * lane + 1;
    if (g == 0) {
        if (wc == 0) {
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (rp[i] < m) ((GI32 *)J.rowperm)[rp[i]] = (int)row0 + rstep * i + 1;
        }
        if (tid == 0) {
            // lu.L is checked first (matrixlu.jl:164-169)
            job_put(J, nanL ? TCI_ERR_NAN_L : nanU ? TCI_ERR_NAN_U : TCI_OK, nanL || nanU ? 0 : p);
            J.error = p >= (m < n ? m : n) ? 0.0 : err;
            // a member that gave up in the last exchange: it marks the team's fail word
            // and then the job, so either this sees the mark or its status comes last
            if (S > 1 && agent_get(mail + kChipFail)) job_put(J, TCI_ERR_DEVICE, 0);
        }
    }
    return true;
}

// the next ticket's job and this workgroup's place in its team; false: none left.
// sh.abort: the launch has given up (a lone member's job is still done)
template <int NW>
__device__ __forceinline__ bool chip_draw(const ChipArgs &K, ChipLds<NW> &sh, ChipItem &it, int &g)
{
    __syncthreads();   // the last job's shared data is done with
    if (threadIdx.x == 0) {
        sh.ticket = (int32_t)__hip_atomic_fetch_add(K.ticket, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        sh.abort = (int32_t)__hip_atomic_load(K.abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(sh.ticket);
    if (t >= K.ntickets) return false;
    it = K.items[K.map[t]];
    g = t - it.first;
    return true;
}

// a member that gave up on the ticket drawn last: its team's fail word, then its job
// (looked up again, so that the register shapes need not hold it)
__device__ __forceinline__ void chip_failed(const ChipArgs &K, int ticket)
{
    if (threadIdx.x == 0) {
        const ChipItem it = K.items[K.map[ticket]];
        agent_put((GU64 *)K.mail + (int64_t)8 * it.first + kChipFail, 1);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        job_put(K.jobs[it.job], TCI_ERR_DEVICE, 0);
    }
}

// the register shapes, by ChipItem::shape: rows per lane × columns per wave.
// 72 to 88 entries a thread: with the pivot column, positions and addresses
// that fills 256 registers without spilling
__global__ __launch_bounds__(256, 2) void tci_rrlu_chip_kernel(ChipArgs K)
{
    __shared__ ChipLds<4> sh;
    ChipItem it;
    int g;
    while (chip_draw<4>(K, sh, it, g)) {
        tci_lu_job &J = K.jobs[it.job];
        GU64 *mail = (GU64 *)K.mail + (int64_t)8 * it.first;
        bool ok = true;
        if (it.S > 1 && sh.abort) ok = false;
        else switch (it.shape) {
        case 0: ok = chip_job<4, 2, 42, false>(K, sh, nullptr, 0, J, it.S, g, it.wr, mail); break;
        case 1: ok = chip_job<4, 3, 28, false>(K, sh, nullptr, 0, J, it.S, g, it.wr, mail); break;
        case 2: ok = chip_job<4, 4, 22, false>(K, sh, nullptr, 0, J, it.S, g, it.wr, mail); break;
        case 3: ok = chip_job<4, 5, 17, false>(K, sh, nullptr, 0, J, it.S, g, it.wr, mail); break;
        case 4: ok = chip_job<4, 6, 14, false>(K, sh, nullptr, 0, J, it.S, g, it.wr, mail); break;
        case 5: ok = chip_job<4, 8, 10, false>(K, sh, nullptr, 0, J, it.S, g, it.wr, mail); break;
        default: ok = chip_job<4, 12, 6, false>(K, sh, nullptr, 0, J, it.S, g, it.wr, mail); break;
        }
        if (!ok) chip_failed(K, sh.ticket);
    }
}

// (the columns outside the registers cost some more: 121 values in 212 bytes of
// scratch over the four shapes)
__global__ __launch_bounds__(512, 2) void tci_rrlu_chip_big_kernel(ChipArgs K, int64_t exl_cap)
{
    __shared__ ChipLds<8> sh;
    extern __shared__ double exl[];
    ChipItem it;
    int g;
    while (chip_draw<8>(K, sh, it, g)) {
        tci_lu_job &J = K.jobs[it.job];
        GU64 *mail = (GU64 *)K.mail + (int64_t)8 * it.first;
        bool ok = true;
        if (it.S > 1 && sh.abort) ok = false;
        else switch (it.shape) {
        case 0: ok = chip_job<8, 6, 12, true>(K, sh, exl, exl_cap, J, it.S, g, 8, mail); break;
        case 1: ok = chip_job<8, 9, 9, true>(K, sh, exl, exl_cap, J, it.S, g, 8, mail); break;
        case 2: ok = chip_job<8, 12, 6, true>(K, sh, exl, exl_cap, J, it.S, g, 8, mail); break;
        default: ok = chip_job<8, 16, 4, true>(K, sh, exl, exl_cap, J, it.S, g, 8, mail); break;
        }
        if (!ok) chip_failed(K, sh.ticket);
    }
}

// ------------------------------------------------------------- host side
static const int kChipRA[7] = {2, 3, 4, 5, 6, 8, 12};
static const int kChipCB[7] = {42, 28, 22, 17, 14, 10, 6};
static const int kBigRA[4] = {6, 9, 12, 16};
static const int kBigCB[4] = {12, 9, 6, 4};

// The shape with the fewest workgroups for an m×n matrix (the first such: the
// fewest rows per lane); 0 when m is beyond every shape.
static int chip_shape(int64_t m, int64_t n, ChipItem &it)
{
    int best = 0;
    for (int q = 0; q < 7; ++q)
        for (int wr = 1; wr <= 4; wr *= 2) {
            if ((int64_t)64 * wr * kChipRA[q] < m) continue;
            const int64_t cols = (int64_t)(4 / wr) * kChipCB[q];
            const int64_t s = (n + cols - 1) / cols;
            if (s <= 1024 && (best == 0 || s < best)) {
                best = (int)s;
                it.shape = q;
                it.wr = wr;
                it.S = (int)s;
            }
            break;
        }
    return best;
}

int rrlu_chip_plan(int64_t m, int64_t n, int ncu, ChipItem *it)
{
    it->job = it->first = 0;
    if (m < 1 || n < 1 || m > kGridMaxSide || n > kGridMaxSide || ncu < 1) return 0;
    // Up to one workgroup per CU the two-per-CU kernel takes the job, whole in
    // registers (2048 x 2048: 205 members, 9.0 us a pivot).  Beyond that the big
    // kernel: its members hold twice as much, so half as many have to agree
    // (3000 x 3000 with 256 members: 10.1 us; the reads of the mailboxes grow
    // with the square of the team)
    const int s = chip_shape(m, n, *it);
    if (s >= 1 && s <= ncu && s <= 512) return 1;
    it->wr = 8;
    for (int q = 0; q < 4; ++q)
        if ((int64_t)512 * kBigRA[q] >= m) {
            int64_t S = ncu < n ? ncu : n;
            if (S > 512) S = 512;
            it->shape = q;
            it->S = (int)S;
            return (n + S - 1) / S - kBigCB[q] <= kChipMaxExtra ? 2 : 0;
        }
    return 0;
}

int64_t rrlu_chip_spill(const ChipItem &it, int64_t m, int64_t n)
{
    const int64_t own = (n + it.S - 1) / it.S, ex = own - kBigCB[it.shape];
    return ex > 0 ? ex * m : 0;
}

// LDS of the big kernel beside its static part, for the columns the registers
// do not hold (doubles); -1 on error
static int64_t big_lds_doubles()
{
    int lds_blk = 0, dev = 0;
    hipFuncAttributes fa;
    const void *k = (const void *)tci_rrlu_chip_big_kernel;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&lds_blk, hipDeviceAttributeMaxSharedMemoryPerBlock, dev) != hipSuccess ||
        hipFuncGetAttributes(&fa, k) != hipSuccess)
        return -1;
    const int64_t cap = ((int64_t)lds_blk - (int64_t)fa.sharedSizeBytes - 64) / 8;
    if (cap < 0 || hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)(cap * 8)) != hipSuccess)
        return -1;
    return cap;
}

int rrlu_chip_blocks(int big, int ncu, int ntickets)
{
    int per = 0;
    if (big) {
        const int64_t cap = big_lds_doubles();
        if (cap < 0 || hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void *)tci_rrlu_chip_big_kernel, 512,
                                                                    (size_t)cap * 8) != hipSuccess)
            return 0;
        if (per > 1) per = 1;
    } else {
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, (const void *)tci_rrlu_chip_kernel, 256, 0) != hipSuccess)
            return 0;
        if (per > 2) per = 2;
    }
    const int b = per * ncu;
    return b < ntickets ? b : ntickets;
}

hipError_t launch_rrlu_chip(const ChipArgs &K, int big, int blocks, hipStream_t st)
{
    if (K.ntickets < 1) return hipSuccess;
    if (blocks < 1 || blocks > 1024) return hipErrorInvalidConfiguration;
    ChipArgs args = K;
    if (big) {
        int64_t cap = big_lds_doubles();
        if (cap < 0) return hipErrorInvalidValue;
        void *p[] = {(void *)&args, (void *)&cap};
        return hipLaunchCooperativeKernel((const void *)tci_rrlu_chip_big_kernel, dim3((unsigned)blocks), dim3(512), p,
                                          (unsigned)(cap * 8), st);
    }
    void *p[] = {(void *)&args};
    return hipLaunchCooperativeKernel((const void *)tci_rrlu_chip_kernel, dim3((unsigned)blocks), dim3(256), p, 0, st);
}

}  // namespace tci
