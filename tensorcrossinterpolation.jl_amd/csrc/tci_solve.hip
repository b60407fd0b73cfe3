// tci_solve.hip — whole crossinterpolate2 solves (tensorci2.jl:943-953), one
// workgroup each, state resident in HBM, and the serving grid that runs them as they
// are published.  One object per TCI_SOLVE_TEAM (tci_solve.h).
#include <hip/hip_runtime.h>

#include "tci_devteam.h"
#include "tci_engine.h"
#include "tci_kernels.h"
#include "tci_solve.h"

#ifndef TCI_SOLVE_TEAM
#define TCI_SOLVE_TEAM 256
#endif

namespace tci {

// ---------------------------------------------------------------- solves
// Dynamic LDS of a solve workgroup (sizes fixed per launch by LdsPlan):
//   [stage: 2·stage_cap doubles][rows: tab_cap bytes][cols: tab_cap bytes]
//   [sets: sets_cap bytes (the pivot sets, then their counts)]
//   [Lorentzian value table: lut_cap doubles][Pi area: pi_cap doubles]
// Anything that does not fit stays in the solve's HBM arena.
template <int NT, int FK, int WPE>
__device__ __forceinline__ void solve_on_team(const SolveDesc &D, const LdsPlan &plan, EngShared &S, double *dyn)
{
    DevTeam<NT, WPE> tm;
    double *stage = dyn;
    uint8_t *tabs = (uint8_t *)(dyn + 2 * plan.stage_cap);
    uint8_t *lsets = tabs + 2 * plan.tab_cap;
    double *lut = (double *)(lsets + plan.sets_cap);
    double *pi = lut + plan.lut_cap;
    if (D.mrcap <= plan.stage_cap) {
        tm.init(stage, stage + D.mrcap);
        tm.stage_lds = true;
    } else {
        tm.init(D.stage, D.stage + D.mrcap);
    }
    if ((int64_t)D.mrcap * D.L <= plan.tab_cap) {
        tm.lrows = tabs;
        tm.lcols = tabs + plan.tab_cap;
    }
    const int64_t setbytes = (int64_t)NSETKIND * D.L * D.setcap * D.L;
    if (((setbytes + 15) & ~(int64_t)15) + 4 * NSETKIND * D.L <= plan.sets_cap) {
        tm.lsets = lsets;
        tm.lsetn = (int32_t *)(lsets + ((setbytes + 15) & ~(int64_t)15));
    }
    tm.llut = plan.lut_cap ? lut : nullptr;
    tm.llut_cap = plan.lut_cap;
    tm.lpi = pi;
    tm.lpi_cap = plan.pi_cap;
    Engine<DevTeam<NT, WPE>, FK> eng(tm, D, S);
    eng.run();
}

template <int NT, int FK, int WPE>
__global__ __launch_bounds__(NT, WPE) void tci_solve_kernel(const SolveDesc *__restrict__ descs,
                                                       int count, LdsPlan plan)
{
    const int s = blockIdx.x;
    if (s >= count) return;
    __shared__ EngShared S;
    extern __shared__ double dyn[];
    solve_on_team<NT, FK, WPE>(descs[s], plan, S, dyn);
}

template <int NT, int WPE>
static const void *solve_kernel_all(int fkind)
{
    switch (fkind) {
    case TCI_F_LORENTZ_INT: return (const void *)tci_solve_kernel<NT, TCI_F_LORENTZ_INT, WPE>;
    case TCI_F_LORENTZ_WEIGHTED: return (const void *)tci_solve_kernel<NT, TCI_F_LORENTZ_WEIGHTED, WPE>;
    case TCI_F_QUANTICS_GAUSS_COS: return (const void *)tci_solve_kernel<NT, TCI_F_QUANTICS_GAUSS_COS, WPE>;
    case TCI_F_GAUSS_SUM: return (const void *)tci_solve_kernel<NT, TCI_F_GAUSS_SUM, WPE>;
    default: return (const void *)tci_solve_kernel<NT, 0, WPE>;
    }
}

#if TCI_SOLVE_TEAM == 64
const void *solve_kernel_64(int fkind)
{
    return fkind == TCI_F_QUANTICS_GAUSS_COS ? (const void *)tci_solve_kernel<64, TCI_F_QUANTICS_GAUSS_COS, 2>
                                             : (const void *)tci_solve_kernel<64, 0, 2>;
}
#elif TCI_SOLVE_TEAM == 256
const void *solve_kernel_256(int fkind) { return solve_kernel_all<256, 2>(fkind); }
#elif TCI_SOLVE_TEAM == 512
const void *solve_kernel_512(int fkind) { return solve_kernel_all<512, 2>(fkind); }
#elif TCI_SOLVE_TEAM == 1024
const void *solve_kernel_1024(int fkind)
{
    return fkind == TCI_F_LORENTZ_INT ? (const void *)tci_solve_kernel<1024, TCI_F_LORENTZ_INT, 4>
                                      : (const void *)tci_solve_kernel<1024, 0, 4>;
}
#endif

#if TCI_SOLVE_TEAM == 256 || TCI_SOLVE_TEAM == 512
// ------------------------------------------------------------------ serving
// Slot-level serving: a persistent grid whose workgroups each take one
// published solve at a time from a ring of requests.  The host publishes
// ticket t by writing ring[t % cap] and the staged image it names (coherent
// host memory, before) and then ctl->tail = t + 1.  One workgroup at a time, at most
// every kServePollTicks, reads the host's words and raises the device mirror
// g->dtail, so the idle workgroups poll device memory, not the bus.  A
// workgroup claims the next ticket below the mirror by a compare-and-swap on
// g->head, so a ticket is claimed only once it is published and every claimed
// ticket is run; after the solve its done slot (coherent host memory) becomes
// t + 1.  The grid leaves as a whole: with stop seen, once every published
// ticket is claimed; otherwise once no workgroup has run, claimed or finished
// a solve for idle_ticks (the first to see that marks the epoch closing and
// the others follow; one that claimed meanwhile still runs its ticket).  A
// ticket published while the grid leaves is run by the next launch.
constexpr uint64_t kServePollTicks = 50;   // 0.5 us of the 100 MHz wall clock

// n bytes (a multiple of 16, both ends 16-byte aligned) by the whole team
template <int NT>
__device__ __forceinline__ void team_copy16(uint8_t *dst, const uint8_t *src, uint64_t n)
{
    for (uint64_t o = (uint64_t)threadIdx.x * 16; o < n; o += (uint64_t)NT * 16)
        *(uint4 *)(dst + o) = *(const uint4 *)(src + o);
}

// the engine run of one served request, compiled apart from the claim loop
// so that the loop's live values do not crowd the engine's registers
template <int NT, int WPE>
__device__ __noinline__ void serve_solve(const SolveDesc *D, LdsPlan plan)
{
    __shared__ EngShared S;
    extern __shared__ double dyn[];
    solve_on_team<NT, 0, WPE>(*D, plan, S, dyn);
}

template <int NT, int WPE>
__global__ __launch_bounds__(NT, WPE) void tci_serve_kernel(const ServeSlot *__restrict__ ring, ServeDev *g,
                                                            const ServeCtl *ctl, uint64_t *done, int cap,
                                                            LdsPlan plan, uint64_t idle_ticks, uint32_t epoch)
{
    __shared__ uint64_t s_ticket;
    __shared__ int s_go;
    __shared__ ServeSlot s_slot;
    extern __shared__ double dyn[];
    const uint64_t born = (uint64_t)wall_clock64();
    for (;;) {
        if (threadIdx.x == 0) {
            int go = 0, nap = 1;
            uint64_t t = 0;
            for (;;) {
                uint64_t tail = __hip_atomic_load(&g->dtail, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                uint64_t h = __hip_atomic_load(&g->head, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const uint64_t now = (uint64_t)wall_clock64();
                if (h >= tail) {
                    uint64_t lp = __hip_atomic_load(&g->lastpoll, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (now - lp >= kServePollTicks &&
                        __hip_atomic_compare_exchange_strong(&g->lastpoll, &lp, now, __ATOMIC_RELAXED,
                                                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                        // stop first: a tail read after it holds every ticket
                        // published before the stop
                        const bool st =
                            __hip_atomic_load(&ctl->stop, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM) != 0;
                        const uint64_t ht = __hip_atomic_load(&ctl->tail, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_SYSTEM);
                        if (st) __hip_atomic_store(&g->dstop, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        __hip_atomic_fetch_max(&g->dtail, ht, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
                        if (ht > tail) tail = ht;
                    }
                }
                const bool stopping =
                    __hip_atomic_load(&g->dstop, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch;
                if (!stopping && __hip_atomic_load(&g->closing, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == epoch)
                    break;
                if (h < tail) {
                    if (__hip_atomic_compare_exchange_strong(&g->head, &h, h + 1, __ATOMIC_RELAXED, __ATOMIC_RELAXED,
                                                             __HIP_MEMORY_SCOPE_AGENT)) {
                        __hip_atomic_fetch_add(&g->busy, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        __hip_atomic_store(&g->last, now, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        t = h;
                        go = 1;
                        break;
                    }
                    continue;
                }
                if (stopping) break;
                if (__hip_atomic_load(&g->busy, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0) {
                    // the last finish's clock is published before its busy decrement
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
                    const uint64_t last = __hip_atomic_load(&g->last, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    const uint64_t ref = last > born ? last : born;
                    if (now > ref && now - ref > idle_ticks) {
                        __hip_atomic_store(&g->closing, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        break;
                    }
                }
                // back off while idle: about 0.9 us, doubling to about 55 us,
                // so a mostly idle grid does not keep the memory channel of
                // these words busy under the solves still running
                for (int k = 0; k < nap; ++k) __builtin_amdgcn_s_sleep(32);
                if (nap < 64) nap *= 2;
            }
            if (go) {
                // the ring entry and its staged image were written before
                // the publication: read them after it
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "");
                const uint64_t *e = (const uint64_t *)(ring + t % (uint64_t)cap);
                uint64_t *w = (uint64_t *)&s_slot;
                for (int k = 0; k < (int)(sizeof(ServeSlot) / 8); ++k)
                    w[k] = __hip_atomic_load(e + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
            s_ticket = t;
            s_go = go;
        }
        __syncthreads();
        if (!s_go) return;
        const uint64_t ticket = s_ticket;
        // the descriptor and inputs into the request's device block
        team_copy16<NT>(s_slot.dst, s_slot.src, s_slot.bytes);
        __threadfence();
        __syncthreads();
        serve_solve<NT, WPE>((const SolveDesc *)s_slot.dst, plan);
        __syncthreads();
        team_copy16<NT>(s_slot.rep_out, s_slot.rep, s_slot.rep_bytes);
        __threadfence_system();   // every thread's part of the report before the done mark
        __syncthreads();
        if (threadIdx.x == 0) {
            __hip_atomic_store(done + ticket % (uint64_t)cap, ticket + 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
            __hip_atomic_store(&g->last, (uint64_t)wall_clock64(), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_fetch_sub(&g->busy, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
    }
}

#if TCI_SOLVE_TEAM == 256
const void *serve_kernel_256() { return (const void *)tci_serve_kernel<256, 2>; }
#else
const void *serve_kernel_512() { return (const void *)tci_serve_kernel<512, 2>; }
#endif
#endif

}  // namespace tci
