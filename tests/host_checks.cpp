// Checks of the library's host code that its C interface does not show
// (launch keys, plans): run by tests/test_host_checks_cpu.py, no GPU needed.
// Usage: host_checks CHECK; prints what is wrong, exit status 1 if anything is.
#include "../pyalign_amd/csrc/pa_api.cpp"

#include <cstdio>
#include <functional>
#include <map>

namespace {

int bad = 0;

void expect(bool ok, const std::string &what) {
    if (ok) return;
    bad++;
    std::printf("%s\n", what.c_str());
}

// One long problem and nothing else: every argument of its launch is in the key.
void graph_key() {
    Job job{LOC_GLOBAL, DIR_MAX, GAP_AFF, F_BINARY, TR_ONE, true, false};
    Plan plan;
    plan.band_probs = {0};
    plan.n_long = 1;
    plan.xbuf_begin = 64;
    plan.xbuf_end = 128;
    KArgs a;
    std::memset(&a, 0, sizeof(a));
    LongArgs la;
    std::memset(&la, 0, sizeof(la));
    int grid = 3;
    int64_t nx = 5, ny = 6;
    char memory[16];
    auto key = [&] { return launch_key(job, plan, {}, {}, a, la, grid, nullptr, nx, ny); };
    const std::string first = key();
    expect(key() == first, "the key of the same launches differs");
    auto changes = [&](const char *what, auto &field, auto value) {
        const auto old = field;
        field = value;
        expect(key() != first, std::string("not in the key: ") + what);
        field = old;
    };
    changes("eq", a.eq, 2.0f);
    changes("ne", a.ne, -2.0f);
    changes("go_s", a.go_s, -2.0f);
    changes("ge_s", a.ge_s, -2.0f);
    changes("go_t", a.go_t, -2.0f);
    changes("ge_t", a.ge_t, -2.0f);
    changes("K1", a.K1, 21);
    changes("codes_s", a.codes_s, static_cast<const void *>(memory));
    changes("codes_t", a.codes_t, static_cast<const void *>(memory));
    changes("table", a.table, reinterpret_cast<const float *>(memory));
    changes("tb", a.tb, reinterpret_cast<uint32_t *>(memory));
    changes("rowbuf", a.rowbuf, reinterpret_cast<float2 *>(memory));
    changes("partials", a.partials, reinterpret_cast<BandPartial *>(memory));
    changes("border_s", a.border_s, reinterpret_cast<const float *>(memory));
    changes("order", la.order, reinterpret_cast<const int32_t *>(memory));
    changes("total_bands", la.total_bands, 7);
    changes("ticket", la.ticket, reinterpret_cast<uint32_t *>(memory));
    changes("gap", job.gap, int(GAP_LIN));
    changes("form", job.form, int(F_TABLE));
    changes("fold_max", job.fold_max, false);
    changes("xbuf_begin", plan.xbuf_begin, int64_t(0));
    changes("grid", grid, 4);
    changes("finite_nx", nx, int64_t(9));
    changes("finite_ny", ny, int64_t(9));
}

// General gap costs: every launch of long pairs fits a grid (its y extent is
// 65,535 at most) and has workgroups for what it pushes on.
void wsb_extents() {
    const std::vector<std::vector<std::pair<int, int>>> bags = {
        {{11600, 11600}}, {{16383, 16383}}, {{32000, 32000}}, {{400, 300000}}, {{1, 3000000}}, {{3000000, 1}},
        {{700, 700}, {30, 40}, {5, 2000000}}};
    for (const auto &bag : bags) {
        std::vector<Prob> probs;
        for (const auto &shape : bag) {
            Prob pr{};
            pr.len_s = shape.first;
            pr.len_t = shape.second;
            probs.push_back(pr);
        }
        std::stable_sort(probs.begin(), probs.end(), [](const Prob &x, const Prob &y) {
            return wsb_blocks(x.len_s) + wsb_blocks(x.len_t) > wsb_blocks(y.len_s) + wsb_blocks(y.len_t);
        });
        const WsbPlan plan = wsb_plan(probs, 256);
        const std::string name = std::to_string(bag[0].first) + " x " + std::to_string(bag[0].second);
        expect(plan.carry, name + ": no carried sums");
        int64_t most = 0;
        for (const WsbPlan::Diag &g : plan.diags) most = std::max(most, int64_t(g.groups) + g.pushes);
        expect(most > 1 && most <= 65535, name + ": " + std::to_string(most) + " workgroups in y");
    }
}

// Which gap costs and similarities max / min folds are chosen for.
void fold_rule() {
    const float inf = std::numeric_limits<float>::infinity(), huge = std::numeric_limits<float>::max(),
                nan = std::numeric_limits<float>::quiet_NaN();
    for (int dir : {DIR_MAX, DIR_MIN}) {
        const float sgn = dir == DIR_MAX ? 1.0f : -1.0f;
        pa_solver s;
        s.opt.dir = dir == DIR_MAX ? PA_MAXIMIZE : PA_MINIMIZE;
        auto folds = [&](float open, float extend, std::vector<float> values, int form = F_TABLE, int loc = LOC_SEMI) {
            s.go_s = s.go_t = -sgn * open;
            s.ge_s = s.ge_t = -sgn * extend;
            Input in{};
            for (float &x : values) x = x == 0.0f ? x : sgn * x;
            in.table = values;
            in.eq = values[0];
            in.ne = values[1];
            return folds_max(s, in, Job{loc, dir, GAP_AFF, form, TR_ONE, false, false});
        };
        for (int form : {F_TABLE, F_BINARY}) {
            const std::string name = (form == F_TABLE ? "table, " : "binary, ") + std::to_string(dir) + ": ";
            expect(folds(3, 1, {2, -1}, form), name + "usual values refused");
            expect(folds(0, 0, {2, 0}, form), name + "free gaps refused");
            expect(folds(3, 1, {2, -huge}, form), name + "the lowest value refused");
            expect(!folds(inf, 1, {2, -1}, form), name + "an infinite open cost taken");
            expect(!folds(3, inf, {2, -1}, form), name + "an infinite extension taken");
            expect(!folds(nan, 1, {2, -1}, form), name + "a NaN cost taken");
            expect(!folds(3, 1, {huge, -1}, form), name + "a sum that overflows taken");
            expect(!folds(3, 1, {2, nan}, form), name + "NaN taken");
            expect(!folds(3, 1, {2, -0.0f}, form), name + "-0 taken");
            expect(!folds(3, 1, {inf, -1}, form), name + "an infinite match taken");
        }
        expect(folds(3, 1, {2, -inf}), "the worst value in a table refused");
        expect(!folds(inf, 1, {2, -1}, F_DENSE), "dense with an infinite cost taken");
        expect(folds(0, 1, {2, -1}, F_TABLE, LOC_GLOBAL) == (dir == DIR_MIN), "global, free opening");
    }
}

// The layout of a problem is the cheapest of all under the cap, or the one of
// least serial time: the candidates kept per length against trying every one.
void layouts() {
    const std::vector<std::vector<int>> heights = {
        {std::begin(FAST_RS), std::end(FAST_RS)}, {std::begin(FAST_RS_TABLE), std::end(FAST_RS_TABLE)},
        {std::begin(FAST_RS_BINARY), std::end(FAST_RS_BINARY)}, {8}, {4, 8, 16, 32}};
    uint64_t seed = 1;
    auto draw = [&](int64_t most) {  // log-uniform, 1 .. most
        seed = seed * 6364136223846793005ull + 1442695040888963407ull;
        return int64_t(std::exp(double(seed >> 11) / 9007199254740992.0 * std::log(double(most) + 0.99)));
    };
    for (const auto &Rs : heights) {
        Layouts kept(Rs, 1000);
        for (int k = 0; k < 200000; k++) {
            const int64_t ls = k % 7 ? draw(3000) : draw(200000), lt = draw(5000);
            const double cap = k % 5 ? double(draw(1000000)) : 1e300;
            double cost = 1e300, serial = 1e300, least = 1e300, least_cost = 1e300;
            int L = 0, R = 0, fall_L = 0, fall_R = 0;
            for (int l = 1; l <= 64; l *= 2)
                for (int r : Rs) {
                    const double s = double((ls + l * r - 1) / (l * r)) * double(lt + l - 1) * (STEP_OVERHEAD + r);
                    if (s < least || (s == least && s * l < least_cost)) {
                        least = s;
                        least_cost = s * l;
                        fall_L = l;
                        fall_R = r;
                    }
                    if (s <= cap && (s * l < cost || (s * l == cost && s < serial))) {
                        cost = s * l;
                        serial = s;
                        L = l;
                        R = r;
                    }
                }
            const Layout got = kept.choose(ls, lt, cap);
            const bool fit = cost < 1e300;
            expect(got.fit == fit && got.L == (fit ? L : fall_L) && got.R == (fit ? R : fall_R) &&
                       got.cost == (fit ? cost : least_cost) && got.serial == (fit ? serial : least),
                   "layout of " + std::to_string(ls) + " x " + std::to_string(lt) + " under " + std::to_string(cap));
            if (bad > 5) return;
        }
    }
}

// The allocation-free solve: batches that fit its scratch in the layouts of
// least memory are planned so where the fastest layouts do not fit.
void noalloc_scratch_use() {
    struct Batch {
        uint32_t n, s, t;
        int loc, form;
    };
    for (const Batch &b : {Batch{276247, 67, 531, LOC_GLOBAL, F_TABLE}, Batch{255324, 73, 355, LOC_GLOBAL, F_BINARY},
                           Batch{318456, 44, 431, LOC_LOCAL, F_BINARY}}) {
        pa_solver s;
        s.opt.dir = PA_MAXIMIZE;
        std::vector<int32_t> ls(b.n), lt(b.n);
        std::vector<int64_t> off(b.n, 0);
        for (uint32_t k = 0; k < b.n; k++) {
            ls[k] = int32_t(1 + (k * 2654435761u >> 8) % b.s);
            lt[k] = int32_t(1 + (k * 40503u >> 4) % b.t);
        }
        Input in{};
        in.n = b.n;
        in.form = b.form == F_TABLE ? PA_FORM_INDEXED : PA_FORM_BINARY;
        in.schedule = PA_SCHED_AUTO;
        in.len_s = ls.data();
        in.len_t = lt.data();
        in.off_s = in.off_t = off.data();
        Job job{b.loc, DIR_MAX, GAP_AFF, b.form, TR_SCORE, true, true};
        const Plan plan = noalloc_plan(s, in, job, 256);
        const size_t bytes = NoallocLayout(s, in, plan).total;
        expect(bytes <= NOALLOC_SCRATCH_BYTES, std::to_string(b.n) + " of up to " + std::to_string(b.s) + " x " +
                                                   std::to_string(b.t) + ": " + std::to_string(bytes) + " bytes");
    }
}

// Idle result buffers: two at most, the larger ones, within the pool's bytes.
// (The buffers here are no memory; the pool only ever hands them on.)
void pin_pool() {
    const size_t MB = size_t(1) << 20;
    auto kept = [&](std::vector<size_t> given) {
        auto *pool = new PinPool;
        for (size_t q = 0; q < given.size(); q++)
            pool->give(PinPool::Buf{reinterpret_cast<char *>(4096 * (q + 1)), given[q] * MB});
        std::multiset<size_t> caps;
        for (const PinPool::Buf &b : pool->idle) caps.insert(b.cap / MB);
        expect(pool->held() <= PinPool::IDLE_BYTES, "more bytes idle than the pool may hold");
        pool->idle.clear();
        delete pool;
        return caps;
    };
    expect(kept({1, 2}) == std::multiset<size_t>{1, 2}, "two small buffers");
    expect(kept({5, 1, 2}) == std::multiset<size_t>{2, 5}, "the smallest of three goes");
    expect(kept({100, 100}) == std::multiset<size_t>{100}, "two that are too large together");
    expect(kept({3, 1000}) == std::multiset<size_t>{3}, "one that is too large alone");
    expect(kept({100, 40, 50}) == std::multiset<size_t>{40, 50}, "the largest goes where two are too large");
}

// Bags of a few long pairs: none is left behind for a launch of its own after
// the long mode's; short pairs beside them are.
void long_choice() {
    struct Bag {
        int form;
        std::vector<std::pair<int, int>> shapes;
        int longs;
    };
    for (const Bag &b : {Bag{F_BINARY, {{726, 297}, {766, 889}}, 2}, Bag{F_BINARY, {{229, 432}, {244, 500}, {234, 147}}, 3},
                         Bag{F_BINARY, {{1492, 790}, {1492, 307}, {1492, 462}, {1492, 366}, {1492, 846}}, 5},
                         Bag{F_TABLE, {{1571, 576}, {956, 237}, {1270, 1093}, {347, 490}}, 4},
                         Bag{F_TABLE, {{5000, 4000}, {20, 30}}, 1}, Bag{F_TABLE, {{20, 30}, {50, 60}}, 0}}) {
        std::vector<int32_t> ls, lt;
        for (const auto &x : b.shapes) {
            ls.push_back(x.first);
            lt.push_back(x.second);
        }
        const Plan plan = plan_auto(Job{LOC_GLOBAL, DIR_MAX, GAP_AFF, b.form, TR_SCORE, true, true}, ls.data(), lt.data(),
                                    int64_t(ls.size()), 1024);
        expect(plan.n_long == b.longs, std::to_string(ls[0]) + " x " + std::to_string(lt[0]) + " and others: " +
                                           std::to_string(plan.n_long) + " of " + std::to_string(ls.size()) + " long");
    }
}

}  // namespace

int main(int argc, char **argv) {
    const std::map<std::string, std::function<void()>> checks = {{"graph_key", graph_key}, {"wsb_extents", wsb_extents}, {"fold_rule", fold_rule}, {"layouts", layouts}, {"noalloc_scratch", noalloc_scratch_use}, {"pin_pool", pin_pool}, {"long_choice", long_choice}};
    if (argc != 2 || !checks.count(argv[1])) {
        std::printf("usage: host_checks CHECK\n");
        return 2;
    }
    checks.at(argv[1])();
    return bad ? 1 : 0;
}
