// TEST-ONLY: the register tile on a team with the basic interface alone (NW slots,
// no best_slot), which a team that implements nothing newer has to get right results
// from.  Built by test_bare_team.py.
#include <memory>

#include "engine_host.cpp"

// HostTeamMT without best_slot; a slot beyond the first set ends the process
struct BareTeam : HostTeamMT<256, 2, 32> {
    using Base = HostTeamMT<256, 2, 32>;
    void best_slot() = delete;
    static int slot(int w)
    {
        if (w >= NW) abort();
        return w;
    }
    double &tA(int w) { return Base::tA(slot(w)); }
    uint32_t &tB(int w) { return Base::tB(slot(w)); }
    double &tX(int w, int r) { return Base::tX(slot(w), r); }
};
static_assert(TileSlots<BareTeam>::SETS == 1);

extern "C" int eh_rrlu_bare(const double *A, int m, int n, int64_t maxrank, double reltol, double abstol, int leftorth,
                            int32_t *rowperm, int32_t *colperm, double *err)
{
    constexpr int NT = 256;
    using Tile = TileLU<BareTeam, 2, 32>;
    if (!Tile::fits(m, n)) return -100;
    std::barrier<> bar(NT);
    std::vector<std::unique_ptr<std::barrier<>>> own;
    MTShared sh;
    sh.bar = &bar;
    for (int w = 0; w < NT / 64; ++w) {
        own.push_back(std::make_unique<std::barrier<>>(64));
        sh.wbar.push_back(own.back().get());
    }
    sh.abuf.resize(NT);
    sh.dbuf.resize(NT);
    sh.ibuf.resize(NT);
    sh.ubuf.resize(NT);
    MTTile<NT, 2, 32> tile;
    int pres = 0;
    auto body = [&](int tid) {
        BareTeam tm;
        tm.t_tid = tid;
        tm.sh = &sh;
        tm.tile = &tile;
        Tile R;
        R.setup(tm, m, n);
        R.load(tm, A, m);
        tm.sync();
        double e, st[2];
        const int p = R.factor(tm, maxrank, reltol, abstol, leftorth != 0, nullptr, &e, st, nullptr, rowperm, colperm);
        tm.sync();
        if (tid == 0) {
            pres = p;
            *err = e;
        }
    };
    std::vector<std::thread> th;
    for (int t = 0; t < NT; ++t) th.emplace_back(body, t);
    for (auto &t : th) t.join();
    return pres;
}
