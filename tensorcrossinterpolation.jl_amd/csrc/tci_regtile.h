// tci_regtile.h — full-pivot rrLU with the whole matrix in registers.
//
// Layout.  The team is NW waves of WS lanes.  Lane l of wave w keeps
// A[r, c] for r = l + WS·i (i < RA) and c = w + NW·j (j < CB), so every wave
// holds complete columns and every row is present in every wave.  A matrix
// of up to (WS·RA)×(NW·CB) is factored without touching memory.
//
// Rows and columns are never moved.  Each thread tracks the current position
// of its rows (rp); the positions of a wave's CB register columns are spread
// over its lanes (lane l holds that of register column l, in cpl), so the
// swap of step k (positions k ↔ pivot) costs a few vector operations.  The argmax key
// of an entry is its current position, colpos·256 + rowpos, so the smallest
// key among equal abs2 values is the first maximum of the reference's
// column-major scan of the physically swapped matrix (matrixlu.jl:1-32).
// Every entry sees the operation sequence of addpivot! (matrixlu.jl:114-136):
// a true division of the pivot column (or row), then a - x*y with two
// roundings.  Rows and columns that have been pivoted get NaN multipliers, so
// their entries turn into NaN and drop out of every later search (a NaN is
// never the maximum, as in submatrixargmax); a dead column's entries being
// NaN, its staged multiplier is NaN without any per-column test.
//
// One pivot step costs one team barrier.  Before it every wave finds its own
// best entry: its maximum g of |entry|, then the smallest key among its entries
// with x·x == g·g, and writes g, the key and that entry's column to the LDS slots
// of the step's parity.  After it all waves agree on G = max g·g (squaring is
// monotone) and on the smallest key among the waves that reach it: the winning
// column is already staged.  Slots of the other parity are free by then.
// The pivot row lies in every wave (one lane holds it): a wave-private LDS slot
// turns it into one multiplier per lane, read back as scalars.
// Bound: instruction issue and the dependent chain of a step (reductions over
// lanes, the division, LDS round trips), not the 3 FP64 operations per entry: 7120
// cycles a step with two barriers and a search over all keys by the wave that holds
// the maximum, 5360 so (100×100 on 512 threads; 2.4 GHz).
//
// Extended tiles (EX).  Matrices of up to 256 columns whose columns do not all
// fit in registers: register column j of wave w beyond CB lies in LDS, and where
// that ends in memory, m doubles at a place that only this wave touches; every
// lane updates its own rows there, so a column costs its traffic and nothing
// else.  Staging is by pointer (place) as the team's static slots are sized for
// its own tile.  Bound: instruction issue, two waves a SIMD, 72 entries a lane and
// the LDS round trips of the others.  The factorizations of a 40-site solve (bond
// matrices of 208×208, rank 13) took 114 ms streamed from memory and 47 ms here
// (512 threads, 4×18 doubles a lane).
#pragma once

#include <type_traits>
#include <utility>

#include "tci_common.h"

namespace tci {

// What a team offers beyond the basic interface: a team with best_slot has two sets
// of slots (tA, tB and tX take wave + NW·parity) and reduces a set by itself.  A team
// without it has NW slots; a step then costs a second barrier, before the slots are
// written again, and the slots are compared one by one.
template <class Team, class = void>
struct TileSlots {
    static constexpr int SETS = 1;
    ENG_INLINE static int best(Team &tm, int at, uint32_t &K)
    {
        double g = -1.0;
        for (int q = 0; q < Team::NW; ++q) g = tm.tA(at + q) > g ? tm.tA(at + q) : g;
        K = 0xffffffffu;
        int w = 0;
        for (int q = 0; q < Team::NW; ++q) {
            const double v = tm.tA(at + q);
            if (v >= 0.0 && v * v == g * g && tm.tB(at + q) < K) {
                K = tm.tB(at + q);
                w = q;
            }
        }
        return w;
    }
};
template <class Team>
struct TileSlots<Team, std::void_t<decltype(std::declval<Team &>().best_slot(0, std::declval<uint32_t &>()))>> {
    static constexpr int SETS = 2;
    ENG_INLINE static int best(Team &tm, int at, uint32_t &K) { return tm.best_slot(at, K); }
};

template <class Team, int RA, int CB, bool EX = false>
struct TileLU {
    static constexpr int WS = Team::WS, NW = Team::NW;
    static constexpr int CT = EX ? 256 / NW : CB;      // columns per wave, CB of them in registers
    static constexpr int MR = WS * RA, MC = NW * CT;   // capacity: MR rows, MC columns
    static_assert(MR <= 256, "row positions must fit the 8-bit part of the key");
    static constexpr int CL = (CT + WS - 1) / WS;   // column-position slots per lane
    static_assert(!EX || CL == 1, "a lane keeps the position of one column beyond the registers");
    static constexpr int STAGE = NW * (2 * MR + 2 * CT);    // doubles staged by an extended tile
    // columns are searched by groups, each thread keeping its maximum of every group
    static constexpr int GC = CB > 4 ? 4 : CB > 1 ? 2 : 1, NG = (CB + GC - 1) / GC;
    double a[RA][CB];
    int rp[RA];     // current position of my rows (large for rows ≥ m)
    int cpl[CL];    // slot c: position of register column lane + WS·c (large if none / ≥ n)
    int jw;         // register column this wave staged in its last search
    int par;        // parity of the slots of the last search
    int m, n;
    // extended tiles: staged columns and rows; columns j of [CB, j1) and [j1, j2) in
    // LDS, the others in memory (column of wave w: base + m·(w + NW·(j - first)))
    EngLds *px, *py, *e1, *e2;
    EngGlobal *eg;
    int j1, j2;

    // the staged column in slot w (wave + NW·parity), and the staged row of this wave
    // (its entries 16 bytes apart: two are then written from where they are, where
    // a 16-byte write would have them moved side by side first)
    ENG_INLINE double getX(Team &tm, int w, int r) const { if constexpr (EX) return px[w * MR + r]; else return tm.tX(w, r); }
    ENG_INLINE void setX(Team &tm, int w, int r, double v) const { if constexpr (EX) px[w * MR + r] = v; else tm.tX(w, r) = v; }
    ENG_INLINE double getY(Team &tm, int j) const { if constexpr (EX) return py[2 * (tm.wave() * CT + j)]; else return tm.tY(tm.wave(), j); }
    ENG_INLINE void setY(Team &tm, int j, double v) const { if constexpr (EX) py[2 * (tm.wave() * CT + j)] = v; else tm.tY(tm.wave(), j) = v; }

    // Where an extended tile stages (STAGE doubles of LDS) and keeps the columns
    // beyond its registers: r1 and r2 are LDS areas of n1 and n2 doubles, A the
    // matrix (lda = m), inlds when it lies in LDS itself and its columns stay there.
    ENG_INLINE void place(Team &tm, double *stage, double *r1, int64_t n1, double *r2, int64_t n2, double *A, bool inlds)
    {
        px = (EngLds *)stage;
        py = px + 2 * NW * MR;
        const int64_t per = (int64_t)m * NW;
        if (inlds) {
            e1 = e2 = (EngLds *)(A + per * CB);
            j1 = j2 = CT;
            eg = nullptr;
            return;
        }
        const int64_t c1 = n1 / per, c2 = n2 / per;
        e1 = (EngLds *)r1;
        e2 = (EngLds *)r2;
        j1 = tm.uniform(c1 < CT - CB ? CB + (int)c1 : CT);
        j2 = tm.uniform(c2 < CT - j1 ? j1 + (int)c2 : CT);
        eg = (EngGlobal *)(A + per * j2);
    }

    // columns j of [ja, jb) kept outside the registers at base: f(j, i, entry) for
    // every entry of this lane, the loads of two columns in flight (unconditional,
    // from a clamped row and column)
    template <bool WRITE, class P, class F>
    ENG_INLINE void each(Team &tm, P *base, int ja, int jb, F &&f) const
    {
        const int je = n > tm.wave() ? (n - tm.wave() + NW - 1) / NW : 0;   // this wave's columns
        if (jb > je) jb = je;
        int ro[RA];
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            const int r = tm.lane() + WS * i;
            ro[i] = m * tm.wave() + (r < m ? r : 0);
        }
        const int step = m * NW;
        P *c = base;
        for (int j = ja; j < jb; j += 2, c += 2 * step) {
            const bool two = j + 1 < jb;
            P *c2 = two ? c + step : c;
            double v[2][RA];
#pragma unroll
            for (int i = 0; i < RA; ++i) v[0][i] = c[ro[i]];
#pragma unroll
            for (int i = 0; i < RA; ++i) v[1][i] = c2[ro[i]];
#pragma unroll
            for (int i = 0; i < RA; ++i) {
                const bool ok = tm.lane() + WS * i < m;
                v[0][i] = ok ? v[0][i] : 0.0 / 0.0;
                v[1][i] = ok && two ? v[1][i] : 0.0 / 0.0;
                f(j, i, v[0][i]);
                f(two ? j + 1 : j, i, v[1][i]);
            }
            if constexpr (WRITE) {
#pragma unroll
                for (int i = 0; i < RA; ++i)
                    if (tm.lane() + WS * i < m) {
                        c[ro[i]] = v[0][i];
                        if (two) c2[ro[i]] = v[1][i];
                    }
            }
        }
    }
    template <bool WRITE, class F>
    ENG_INLINE void each_extra(Team &tm, F &&f) const
    {
        if constexpr (EX) {
            each<WRITE>(tm, e1, CB, j1, f);
            each<WRITE>(tm, e2, j1, j2, f);
            each<WRITE>(tm, eg, j2, CT, f);
        }
    }
    // entry of row r in column j beyond the registers (j may differ between lanes)
    ENG_INLINE double extra_at(Team &tm, int j, int r) const
    {
        const int o = m * tm.wave() + r, per = m * NW;
        if (j < j1) return e1[o + per * (j - CB)];
        if (j < j2) return e2[o + per * (j - j1)];
        return eg[o + per * (j - j2)];
    }

    // position of register column j of this wave (wave-uniform)
    ENG_INLINE int colpos(Team &tm, int j) const
    {
        if constexpr (CL == 1) return tm.wave_bcast(cpl[0], j);
        else return tm.wave_bcast(cpl[j / WS], j % WS);
    }

    ENG_INLINE static bool fits(int m_, int n_) { return m_ <= MR && n_ <= MC; }

    ENG_INLINE void setup(const Team &tm, int m_, int n_)
    {
        m = m_;
        n = n_;
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            const int r = tm.lane() + WS * i;
            rp[i] = r < m ? r : 0x3fffffff;
        }
#pragma unroll
        for (int c = 0; c < CL; ++c) {
            const int j = tm.lane() + WS * c;
            const int col = tm.wave() + NW * j;
            cpl[c] = (j < CT && col < n) ? col : 0x3fffffff;
        }
        jw = 0;
        par = 0;
    }

    // the trailing block (positions >= p in both directions) as rrlu! leaves
    // it in A after factor returned p: A[rowpos + lda·colpos] = entry
    ENG_INLINE void store_trailing(Team &tm, double *A, int64_t lda, int p) const
    {
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const int c = colpos(tm, j);
            if (c < p || c >= n) continue;
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (rp[i] >= p && rp[i] < m) A[rp[i] + lda * c] = a[i][j];
        }
    }

    // entries outside the matrix hold NaN.  (Every load is unconditional, from an
    // index clamped into the matrix, so that all are in flight together; loads
    // under a condition each waited for their own.  2.6 us for 100×100)
    template <class P>
    ENG_INLINE void load_from(const Team &tm, const P *A, int lda)
    {
        if (m < 1 || n < 1) {   // nothing to load from
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int i = 0; i < RA; ++i) a[i][j] = 0.0 / 0.0;
            return;
        }
        int ro[RA];
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            const int r = tm.lane() + WS * i;
            ro[i] = r < m ? r : 0;
        }
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const int c = tm.wave() + NW * j;
            const P *col = A + (int64_t)lda * (c < n ? c : 0);
#pragma unroll
            for (int i = 0; i < RA; ++i) a[i][j] = col[ro[i]];
        }
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int i = 0; i < RA; ++i)
                a[i][j] = tm.lane() + WS * i < m && tm.wave() + NW * j < n ? a[i][j] : 0.0 / 0.0;
    }
    ENG_INLINE void load(const Team &tm, const double *A, int64_t lda) { load_from(tm, A, (int)lda); }
    // as load, of a matrix known to lie in LDS or in memory
    ENG_INLINE void load_known(const Team &tm, const double *A, int64_t lda, bool inlds)
    {
        if (inlds) load_from(tm, (const EngLds *)A, (int)lda);
        else load_from(tm, (const EngGlobal *)A, (int)lda);
    }

    // an extended tile's columns beyond the registers, to where place put them
    // (those in memory, and those of a matrix in LDS, stay where they are)
    ENG_INLINE void load_extra(Team &tm, const double *A, bool inlds) const
    {
        if (inlds) return;
        const EngGlobal *G = (const EngGlobal *)A;
        const int je = n > tm.wave() ? (n - tm.wave() + NW - 1) / NW : 0;
        for (int j = CB; j < j2 && j < je; ++j) {
            EngLds *c = (j < j1 ? e1 + m * NW * (j - CB) : e2 + m * NW * (j - j1)) + m * tm.wave();
            double v[RA];
#pragma unroll
            for (int i = 0; i < RA; ++i) {
                const int r = tm.lane() + WS * i;
                v[i] = G[(r < m ? r : 0) + m * (tm.wave() + NW * j)];
            }
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (tm.lane() + WS * i < m) c[tm.lane() + WS * i] = v[i];
        }
    }

    // f = c / (1 + rs[r] + cs[c]) for TCI_F_LORENTZ_INT, whose value is
    // c / (double)(Σ v² + 1) with an exact integer sum split into the row
    // part rs and the column part cs.  With lut (lut[s] = c / (double)s for
    // every sum that occurs) the division is a lookup with the same bits.
    // Returns this thread's NaN-propagating max|f| (the maxsamplevalue
    // contribution).
    ENG_INLINE double fill_lorentz(const Team &tm, double c, const double *rs, const double *cs,
                                   const double *lut)
    {
        // with the sums in LDS (the table always is) the loads are LDS
        // loads, not generic ones
        if (tm.stage_lds) return fill_lorentz_t<true>(tm, c, rs, cs, lut);
        return fill_lorentz_t<false>(tm, c, rs, cs, lut);
    }

    template <bool LDS>
    ENG_INLINE double fill_lorentz_t(const Team &tm, double c, const double *rs, const double *cs,
                                     const double *lut)
    {
        if (LDS) {
            tm.assume_lds(rs);
            tm.assume_lds(cs);
        }
        // (indices clamped into the arrays so every load is unconditional)
        double rsv[RA], csv[CB];
#pragma unroll
        for (int i = 0; i < RA; ++i) {
            const int r = tm.lane() + WS * i;
            const double v = rs[r < m ? r : 0];
            rsv[i] = r < m ? v : 0.0;
        }
#pragma unroll
        for (int j = 0; j < CB; ++j) {
            const int cc = tm.wave() + NW * j;
            const double v = cs[cc < n ? cc : 0];
            csv[j] = cc < n ? v : 0.0;
        }
        double lmax = 0.0;
        if (lut) {
            tm.assume_lds(lut);
            bool any = false;
#pragma unroll
            for (int j = 0; j < CB; ++j)
#pragma unroll
                for (int i = 0; i < RA; ++i) {
                    const bool ok = rp[i] < m && tm.wave() + NW * j < n;
                    const double v = lut[(int)(rsv[i] + csv[j]) + 1];
                    a[i][j] = ok ? v : 0.0 / 0.0;
                    lmax = ok ? fmax(lmax, fabs(v)) : lmax;
                    any = any || ok;
                }
            if (any && c != c) lmax = c;   // every value is NaN: max propagates it
            return lmax;
        }
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int i = 0; i < RA; ++i) {
                const bool ok = rp[i] < m && tm.wave() + NW * j < n;
                const double v = c / (rsv[i] + csv[j] + 1.0);
                a[i][j] = ok ? v : 0.0 / 0.0;
                lmax = ok ? jl_max(lmax, fabs(v)) : lmax;
            }
        return lmax;
    }

    // column j of the tile (j < CB, a constant) into slot w
    ENG_INLINE void stage_column(Team &tm, int w, int j) const
    {
#pragma unroll
        for (int i = 0; i < RA; ++i) setX(tm, w, tm.lane() + WS * i, a[i][j]);
    }

    // The search of a pivot step and its barrier (see the header).  gm is this
    // thread's max |entry| of each group of columns (NaN: none), ex that of the
    // columns beyond the registers (-1: none).  Returns the winning key (UINT32_MAX when
    // every trailing entry is NaN) and the slot that holds the winning column.
    ENG_INLINE uint32_t search(Team &tm, const double *gm, double ex, int &wstar)
    {
        // (groups and columns without a candidate are passed by with a wave vote; the
        // multi-threaded host team votes through barriers and looks at every key)
#if defined(__HIP_DEVICE_COMPILE__)
        constexpr bool vote = true;
#else
        constexpr bool vote = WS == 1;
#endif
        if constexpr (TileSlots<Team>::SETS == 2) par ^= 1;
        else tm.sync();   // (every wave has read the last search's slots)
        const int me = tm.wave() + NW * par;
        double lmax = ex;
#pragma unroll
        for (int q = 0; q < NG; ++q) lmax = fmax(lmax, gm[q]);
        const double g = tm.wave_max(lmax);
        uint32_t kw = 0xffffffffu;
        if (g >= 0.0) {
            const double G = g * g;
            // {x >= 0 : x·x == G} is an interval of doubles [lo, g] (rounding
            // keeps squaring monotone): find lo by stepping down from g, so
            // the per-entry test is |v| >= lo.  G == 0 means every entry is 0
            // in magnitude or squares to 0; G subnormal may span many doubles,
            // then the exact test v·v == G is used.
            double lo = 0.0;
            bool exact = false;
            if (G > 0.0) {
                lo = g;
                int t = 0;
                for (; t < 8; ++t) {
                    const double q = eng_as_f64(eng_as_i64(lo) - 1);
                    if (q * q == G) lo = q;
                    else break;
                }
                exact = t == 8;
            }
            uint32_t kl = 0xffffffffu;
            int hits = 0;   // columns with candidates (several: at least 2)
            if (!exact && vote) {
#pragma unroll
                for (int q = 0; q < NG; ++q)
                    if (tm.wave_any(gm[q] >= lo)) {
#pragma unroll
                        for (int j = q * GC; j < (q + 1) * GC && j < CB; ++j) {
                            bool hit = false;
#pragma unroll
                            for (int i = 0; i < RA; ++i) hit = hit || fabs(a[i][j]) >= lo;
                            if (tm.wave_any(hit)) {
                                const uint32_t ck = (uint32_t)colpos(tm, j) << 8;
#pragma unroll
                                for (int i = 0; i < RA; ++i)
                                    kl = eng_umin(kl, fabs(a[i][j]) >= lo ? ck | (uint32_t)rp[i] : 0xffffffffu);
                                if (hits == 0) {
                                    jw = j;
                                    stage_column(tm, me, j);
                                }
                                ++hits;
                            }
                        }
                    }
            } else {
                hits = 2;
#pragma unroll
                for (int j = 0; j < CB; ++j) {
                    const uint32_t ck = (uint32_t)colpos(tm, j) << 8;
#pragma unroll
                    for (int i = 0; i < RA; ++i) {
                        const double v = a[i][j];
                        kl = eng_umin(kl, (exact ? v * v == G : fabs(v) >= lo) ? ck | (uint32_t)rp[i] : 0xffffffffu);
                    }
                }
            }
            if constexpr (EX) {
                const uint32_t k0 = kl;
                if (!vote || tm.wave_any(exact || ex >= lo)) each_extra<false>(tm, [&](int j, int i, double v) __attribute__((always_inline)) {
                    const uint32_t key = (uint32_t)colpos(tm, j) << 8 | (uint32_t)rp[i];
                    kl = eng_umin(kl, (exact ? v * v == G : fabs(v) >= lo) ? key : 0xffffffffu);
                });
                if (tm.wave_any(kl != k0)) hits = 2;
            }
            kw = tm.wave_min(kl);
            if (hits != 1) {
                // stage the column of the smallest key (raw values; selected by
                // position, not by index, so the tile stays in registers)
                const int cpos = (int)(kw >> 8);
#pragma unroll
                for (int c = 0; c < CL; ++c) {
                    const int l = tm.wave_first(tm.lane() + WS * c < CT && cpl[c] == cpos);
                    if (l >= 0) jw = l + WS * c;
                }
#pragma unroll
                for (int j = 0; j < CB; ++j)
                    if (colpos(tm, j) == cpos) stage_column(tm, me, j);
                if (EX && jw >= CB) {
#pragma unroll
                    for (int i = 0; i < RA; ++i) {
                        const int r = tm.lane() + WS * i;
                        if (r < m) setX(tm, me, r, extra_at(tm, jw, r));
                    }
                }
            }
        }
        if (tm.lane() == 0) {
            tm.tA(me) = g;
            tm.tB(me) = kw;
        }
        tm.sync();
        uint32_t K;
        const int w = TileSlots<Team>::best(tm, NW * par, K);
        wstar = w + NW * par;
        return K;
    }

    // Full-pivot rrLU (matrixlu.jl:141-181): same pivots, pivot values, error
    // and NaN verdicts as rrlu_team.  Requires entries outside the matrix to
    // hold NaN.  Outputs: rowperm/colperm (original index at each position,
    // written when non-null), pivval[k], *perr, stats[0..1] (argmax and Schur
    // element counts), with Lorig non-null the L column k by original row
    // (Lorig[orig + m·k]) and with Uorig non-null the U row k by original
    // column (Uorig[k + ldu·orig], the pivot row as addpivot! leaves it:
    // divided by the pivot when !leftorth).  Returns p, or -status for the
    // NaN errors.
    ENG_INLINE int factor(Team &tm, int64_t maxrank, double reltol, double abstol, bool leftorth,
                          double *pivval, double *perr, double *stats, double *Lorig,
                          int32_t *rowperm, int32_t *colperm, double *Uorig = nullptr,
                          int64_t ldu = 0)
    {
        const double NaN = 0.0 / 0.0;
        double gm[NG], ex = -1.0;
#pragma unroll
        for (int q = 0; q < NG; ++q) gm[q] = NaN;
#pragma unroll
        for (int j = 0; j < CB; ++j)
#pragma unroll
            for (int i = 0; i < RA; ++i) gm[j / GC] = fmax(gm[j / GC], fabs(a[i][j]));
        each_extra<false>(tm, [&](int, int, double v) __attribute__((always_inline)) { ex = fmax(ex, fabs(v)); });
        int wstar;
        uint32_t K = search(tm, gm, ex, wstar);
        int mr = m < n ? m : n;
        if (maxrank < mr) mr = (int)maxrank;
        // (the same in every lane: kept scalar)
        mr = tm.uniform(mr);
        leftorth = tm.uniform(leftorth ? 1 : 0) != 0;
        reltol = tm.uniform_f64(reltol);
        abstol = tm.uniform_f64(abstol);
        double maxerr = 0.0, err = NaN;
        int64_t sarg = 0, sschur = 0;   // element counts (integers stay in scalar registers)
        int p = 0, nanx = 0, nany = 0;
        while (p < mr) {
            const int k = p;
            const bool cand = K != 0xffffffffu;
            const int pr = cand ? (int)(K & 255u) : k;
            const int pc = cand ? (int)(K >> 8) : k;
            // original row of position pr: held in every wave by one lane
            int orow = 0;
#pragma unroll
            for (int i = 0; i < RA; ++i) {
                const int l = tm.wave_first(rp[i] == pr);
                if (l >= 0) orow = l + WS * i;
            }
            // the pivot and the staged pivot column, read together
            double xv[RA];
#pragma unroll
            for (int i = 0; i < RA; ++i) xv[i] = getX(tm, wstar, tm.lane() + WS * i);
            const double av = cand ? tm.uniform_f64(getX(tm, wstar, orow)) : NaN;
            sarg += (int64_t)(m - k) * (n - k);
            const double e = fabs(av);
            err = e;
            if ((e < reltol * maxerr || e < abstol) && p > 0) break;
            maxerr = jl_max(maxerr, e);
#pragma unroll
            for (int i = 0; i < RA; ++i) rp[i] = rp[i] == k ? pr : (rp[i] == pr ? k : rp[i]);
#pragma unroll
            for (int c = 0; c < CL; ++c) cpl[c] = cpl[c] == k ? pc : (cpl[c] == pc ? k : cpl[c]);
            if (tm.tid() == 0 && pivval) pivval[k] = av;
            if (av != av) { nanx = 1; nany = 1; }
            // y: the pivot row, from its holder lane in this wave through the
            // wave's LDS slot.  Dead columns hold NaN already; the pivot column
            // (staged by its wave as register column jw) dies now.
            const bool mine = wstar == tm.wave() + NW * par;
            if (cand) {
                const int lo = orow % WS, io = orow / WS;
                if (tm.lane() == lo) {
#pragma unroll
                    for (int i = 0; i < RA; ++i)
                        if (i == io) {
#pragma unroll
                            for (int j = 0; j < CB; ++j) setY(tm, j, a[i][j]);
                        }
                }
            }
            // x: divided by the pivot when leftorth
            if (leftorth) {
#pragma unroll
                for (int i = 0; i < RA; ++i) xv[i] = xv[i] / av;
            }
            double x[RA];
#pragma unroll
            for (int i = 0; i < RA; ++i) {
                const bool live = rp[i] > k && rp[i] < m;
                x[i] = cand && live ? xv[i] : NaN;
                if (live && x[i] != x[i]) nanx = 1;
                if (Lorig && live && tm.wave() == 0) Lorig[(tm.lane() + WS * i) + (int64_t)m * k] = x[i];
            }
#if defined(__HIP_DEVICE_COMPILE__)
            // lane j holds the multiplier of register column j, read as a scalar by
            // the update
            static_assert(CL == 1, "one multiplier per lane");
            double vy = NaN;
            if (cand) {
                if (EX && NW * j2 < n) tm.wave_sync();   // (a lane reads what the pivot row's lane wrote)
                else tm.wave_sync_lds();
                const int j = tm.lane();
                vy = getY(tm, j < CB ? j : 0);
                if constexpr (EX)
                    if (j >= CB && j < CT && tm.wave() + NW * j < n) vy = extra_at(tm, j, orow);
                if (!leftorth) vy = vy / av;
                if (mine && j == jw) vy = NaN;
            }
            // U row: NaN on a live column
            if (tm.lane() < CT && cpl[0] > k && cpl[0] < n) {
                if (vy != vy) nany = 1;
                if (Uorig) Uorig[k + ldu * (tm.wave() + NW * tm.lane())] = vy;
            }
            const auto y = [&](int j) __attribute__((always_inline)) { return tm.wave_bcast_f64(vy, j); };
#else
            // (host teams read the multipliers back from the slot)
            if (EX && NW * j2 < n) tm.wave_sync();
            else tm.wave_sync_lds();
            for (int j = tm.lane(); j < CT; j += WS) {
                double v = NaN;
                if (cand && tm.wave() + NW * j < n) v = j < CB ? getY(tm, j) : extra_at(tm, j, orow);
                if (!leftorth) v = v / av;
                if (mine && j == jw) v = NaN;
                setY(tm, j, v);
            }
            tm.wave_sync_lds();
#pragma unroll
            for (int c = 0; c < CL; ++c) {
                const int j = tm.lane() + WS * c;
                if (j < CT && cpl[c] > k && cpl[c] < n) {
                    const double v = getY(tm, j);
                    if (v != v) nany = 1;
                    if (Uorig) Uorig[k + ldu * (tm.wave() + NW * j)] = v;
                }
            }
            const auto y = [&](int j) { return getY(tm, j); };
#endif
            // trailing update, fused with the thread's maxima
#pragma unroll
            for (int q = 0; q < NG; ++q) gm[q] = NaN;
#pragma unroll
            for (int j = 0; j < CB; ++j) {
                const double yj = y(j);
#pragma unroll
                for (int i = 0; i < RA; ++i) {
                    const double t = x[i] * yj;
                    const double u = a[i][j] - t;
                    a[i][j] = u;
                    gm[j / GC] = i == 0 && j % GC == 0 ? fabs(u) : fmax(gm[j / GC], fabs(u));
                }
            }
            ex = -1.0;
            each_extra<true>(tm, [&](int j, int i, double &v) __attribute__((always_inline)) {
                const double t = x[i] * y(j);
                v = v - t;
                ex = fmax(ex, fabs(v));
            });
            p = k + 1;
            sschur += (int64_t)(m - p) * (n - p);
            K = search(tm, gm, ex, wstar);
        }
        // position → original index
        if (rowperm && tm.wave() == 0) {
#pragma unroll
            for (int i = 0; i < RA; ++i)
                if (rp[i] < m) rowperm[rp[i]] = tm.lane() + WS * i;
        }
        if (colperm) {
#pragma unroll
            for (int c = 0; c < CL; ++c) {
                const int j = tm.lane() + WS * c;
                if (j < CT && cpl[c] < n) colperm[cpl[c]] = tm.wave() + NW * j;
            }
        }
        const int nanL = tm.any(nanx);
        const int nanU = tm.any(nany);
        stats[0] = (double)sarg;
        stats[1] = (double)sschur;
        if (p >= (m < n ? m : n)) err = 0.0;
        *perr = err;
        if (nanL) return -ST_NAN_L;
        if (nanU) return -ST_NAN_U;
        return p;
    }
};

}  // namespace tci
