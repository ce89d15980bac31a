// Which tiles a launch of contractions takes, and the launches of k_gemm_ring.
#include <algorithm>

#include "sub_ring.hpp"

namespace sub {

namespace {

// The tiles there are, and what they take (us): a step of 64 k with few workgroups, with one on every second CU (two
// share a CU: on every CU), and in every place; a launch with the way into and out of its first tile; a tile's way out
// where all CUs are on theirs.  From products of 64 .. 12288 rows with 1 .. 256 steps, alone and two to five in a launch (which takes up to
// kMaxProducts), on operands of normal distribution that are used in turn.  256 x 256 is k_gemm_wide.
struct Form { int bm, bn, per_cu; double few, half, full, once, out; };
constexpr Form kForms[TILE_FORMS] = {
    {64, 64, 2, 0.20, 0.20, 0.38, 3.6, 1.6},
    {128, 64, 2, 0.29, 0.33, 0.59, 3.8, 2.0},
    {128, 128, 1, 0.33, 0.37, 0.47, 4.4, 2.0},
    {256, 128, 1, 0.56, 0.62, 0.92, 5.9, 2.0},
    {256, 256, 1, 1.02, 1.25, 1.47, 5.5, 4.3},
};
// As they were when the order of the sums in front of a ReLU was fixed (GemmEpilogue::same_order): whether such a product goes into
// 256 x 256 tiles is decided by these and by nothing that is fitted anew, so they are never changed.
constexpr Form kOrderForms[TILE_FORMS] = {
    {64, 64, 2, 0.20, 0.20, 0.38, 3.6, 1.6},
    {128, 64, 2, 0.29, 0.33, 0.59, 3.8, 2.0},
    {128, 128, 1, 0.33, 0.37, 0.47, 4.4, 2.0},
    {256, 128, 1, 0.52, 0.54, 0.83, 5.9, 2.0},
    {256, 256, 1, 1.00, 1.00, 1.42, 5.5, 4.3},
};
inline const Form& form_of(int f, bool order) { return order ? kOrderForms[f] : kForms[f]; }
// Several products of more than a round of the smaller tiles: the workgroups drift apart, and share fewer lines of their L2
// (4096 x 1024 x 4096 twice in tiles of 128 x 128: 75.5 us, 3 times 117 and once 38.5).
constexpr double kDrift = 1.12;

// One launch: its busiest workgroup.
double launch_us(const long* len, const long* cnt, int n, const Form& F) {
    long total = 0;
    for (int i = 0; i < n; ++i) total += cnt[i];
    const long places = 256L * F.per_cu;
    const double x = (double)total / (128.0 * F.per_cu);
    const double step = x <= 1.0 ? F.few + (F.half - F.few) * x : F.per_cu > 1 || x >= 2.0 ? F.full : F.half + (F.full - F.half) * (x - 1.0);
    const double out = F.out * (total < places ? (double)total / (double)places : 1.0);
    if (n == 1) return F.once + (double)((total + places - 1) / places) * ((double)len[0] * step + out);
    Schedule s;
    const double drift = total > places && F.bm * F.bn <= 128 * 128 ? kDrift : 1.0;
    return F.once + step * drift * schedule_tiles(len, cnt, n, std::min(total, places), out / step, s);
}

}  // namespace

// The longest tiles first, each to the workgroups that have least to do.  Workgroups with as much to do as their neighbours are one
// run, so that tiles next to each other in the list, which share operands, go to workgroups next to each other.  Up to the last
// three rounds, or four, all of them take a tile in turn.  Four weight gradients of 192 tiles and 192 steps and a data gradient of 192
// tiles and 48 steps (96 sequences of 128, E 1024) so end at step 192; with the rounds and the way back for the last of them that
// were here before, a quarter of the workgroups had 192 + 48 to do.
double schedule_tiles(const long* len, const long* cnt, int n, long workers, double out_steps, Schedule& s) {
    struct Run { long worker, count, load; };                  // (loads in sixteenths of a step)
    constexpr int kMaxRuns = 64;
    Run run[kMaxRuns];
    int runs = 1;
    run[0] = Run{0, workers, 0};
    auto cut = [&](int i, long count) {                        // run i behind its first `count` workgroups
        if (count <= 0 || count >= run[i].count) return;
        for (int k = runs++; k > i; --k) run[k] = run[k - 1];
        run[i].count = count;
        run[i + 1].worker += count; run[i + 1].count -= count;
    };
    auto give = [&](int i, long count, long load) {            // to the first `count` workgroups of run i
        cut(i, count);
        run[i].load += load;
        int m = 0;
        for (int k = 1; k < runs; ++k)
            if (run[k].load == run[m].load) run[m].count += run[k].count;
            else run[++m] = run[k];
        runs = m + 1;
    };
    long total = 0;
    for (int i = 0; i < n; ++i) total += cnt[i];
    // lengths so mixed that this takes more parts than fit: whole rounds, what is left of the last one to the workgroups from the
    // other end, each round as long as its longest tile
    auto in_turn = [&]() {
        s.rounds = (unsigned)(total / workers);
        const unsigned rest = (unsigned)(total % workers);
        s.n = rest ? 1 : 0;
        s.part[0] = SchedulePart{(unsigned)workers - rest, (unsigned)(total - rest), rest};
        double steps = 0.;
        for (long id = 0; id < total; id += workers) {
            long in = id;
            int i = 0;
            while (in >= cnt[i]) in -= cnt[i++];
            steps += (double)len[i] + out_steps;
        }
        return steps;
    };
    s.rounds = (unsigned)std::max(0L, total / workers - 3);
    s.n = 0;
    long in_rounds = s.rounds * workers, at = 0, worker = 0;
    for (int i = 0; i < n; ++i) {
        const long load = 16 * len[i] + (long)(16. * out_steps);
        long left = cnt[i];
        while (left > 0) {
            int r = 0;
            if (in_rounds > 0) {
                while (run[r].worker + run[r].count <= worker) ++r;
                cut(r, worker - run[r].worker);
                if (run[r].worker < worker) ++r;
            } else {
                for (int k = 1; k < runs; ++k)
                    if (run[k].load < run[r].load) r = k;
            }
            const long c = std::min(left, run[r].count);
            if (in_rounds > 0) {
                in_rounds -= c;
                worker = (worker + c) % workers;
            } else {
                if (s.n == kMaxParts || runs > kMaxRuns - 4) return in_turn();
                s.part[s.n++] = SchedulePart{(unsigned)run[r].worker, (unsigned)at, (unsigned)c};
            }
            give(r, c, load);
            left -= c; at += c;
        }
    }
    long longest = 0;
    for (int r = 0; r < runs; ++r) longest = std::max(longest, run[r].load);
    return (double)longest / 16.;
}

bool tiles_take(const TileProduct& p) {
    const GemmArgs& a = p.a;
    // a lane's words within 2^31 bytes of the tile's first element
    const long la = p.akc ? 255 * a.sAM + BK : 63 * a.sAK1 + 256, lb = p.bkc ? 255 * a.sBN + BK : 63 * a.sBK1 + 256;
    const long lc = 255 * a.sCM + 256, lt = a.bias ? 255 * a.sbM + 256 : 0;
    return la < (1L << 30) && lb < (1L << 30) && lc < (1L << 30) && lt < (1L << 30);
}

// The launches a thread has last asked about, by everything that the choice depends on (choosing takes 1 to 8 us, a layer's pass
// of some 15 products as much as a few launches; a decoder layer's operator calls make 25 such choices).
namespace {
struct Asked {
    struct Product { int M, N, K1, K0, splits, order; long nbatch; };
    long n = 0, forms = 0;
    size_t ws_floats = 0;
    double reduce_us = 0.;
    Product p[kMaxProducts] = {};
};
struct Answer { Asked asked; TileChoice choice; };
thread_local Answer answers[64];

TileChoice choose_anew(const TileProduct* p, int n, unsigned forms, size_t ws_floats, double reduce_us);
}  // namespace

TileChoice choose_tiles(const TileProduct* p, int n, unsigned forms, size_t ws_floats, double reduce_us) {
    if (n < 1 || n > kMaxProducts) return TileChoice{};
    Asked q;
    q.n = n; q.forms = forms; q.ws_floats = ws_floats; q.reduce_us = reduce_us;
    uint64_t h = (uint64_t)ws_floats * 31 + forms;
    for (int i = 0; i < n; ++i) {
        const GemmArgs& a = p[i].a;
        q.p[i] = Asked::Product{a.M, a.N, a.K1, a.K0, a.splits, (p[i].akc ? 1 : 0) | (p[i].bkc ? 2 : 0), a.nbatch};
        for (uint64_t x : {(uint64_t)a.M, (uint64_t)a.N, (uint64_t)a.K1, (uint64_t)a.nbatch}) h = (h ^ x) * 0x9E3779B97F4A7C15ull;
    }
    Answer& at = answers[(h >> 40) % 64];
    const Asked& was = at.asked;
    bool same = was.n == q.n && was.forms == q.forms && was.ws_floats == q.ws_floats && was.reduce_us == q.reduce_us;
    for (int i = 0; same && i < n; ++i) {
        const Asked::Product &x = was.p[i], &y = q.p[i];
        same = x.M == y.M && x.N == y.N && x.K1 == y.K1 && x.K0 == y.K0 && x.splits == y.splits && x.order == y.order && x.nbatch == y.nbatch;
    }
    if (!same) {
        at.choice = choose_anew(p, n, forms, ws_floats, reduce_us);
        at.asked = q;
    }
    return at.choice;
}

namespace {
TileChoice choose_anew(const TileProduct* p, int n, unsigned forms, size_t ws_floats, double reduce_us) {
    TileChoice best;
    int k1, k2;
    if (!orientations(p, n, k1, k2)) return best;
    // the order of the launch's list: longest contraction first
    int order[kMaxProducts];
    longest_first(p, n, order);
    const GemmArgs& longest = p[order[0]].a;
    // The longest contraction in parts: a reduction follows (a launch of about 3 us, or less in a launch that takes the parts
    // themselves, and a pass over the partial sums).
    const bool free_split = ws_floats > 0 && longest.splits == 1 && longest.N % 4 == 0;
    for (int s = 1; s <= (free_split ? 8 : 1); ++s) {
        const size_t partial = (size_t)longest.nbatch * longest.M * longest.N * s;
        if (s > 1 && (steps_of(longest, s) < 4 || partial > ws_floats)) break;
        const double reduce = s > 1 || longest.splits > 1 ? reduce_us + (double)partial * 8.0 / 4e6 : 0.0;
        for (int f = 0; f < TILE_FORMS; ++f) {
            if (!(forms >> f & 1u) || (f == TILE_256x256 && s > 1)) continue;
            long len[kMaxProducts], cnt[kMaxProducts];
            for (int i = 0; i < n; ++i) {
                const GemmArgs& a = p[order[i]].a;
                const int splits = i == 0 && s > 1 ? s : a.splits;
                len[i] = steps_of(a, splits);
                cnt[i] = tiles_of(a, splits, kForms[f].bm, kForms[f].bn);
            }
            for (int i = 0; i + 1 < n && len[i] < len[i + 1]; ++i) { std::swap(len[i], len[i + 1]); std::swap(cnt[i], cnt[i + 1]); }
            const double t = launch_us(len, cnt, n, kForms[f]) + reduce;
            if (best.form < 0 || t < best.us) { best.form = f; best.us = t; best.split = order[0]; best.splits = s > 1 ? s : longest.splits; }
        }
    }
    return best;
}
}  // namespace

TileForm tile_form(int form) {
    const Form& F = kForms[form];
    return TileForm{F.bm, F.bn, F.per_cu, F.out / F.full};
}

// What the activation adds to a tile (us): for each pack of 8 outputs that a lane stores, its arithmetic (0.1, GELU 0.25) and,
// forward, its keep bits: 0.2, and 0.13 on 256 x 256 tiles, which draw them between their matrix instructions, but not for nothing
// (taken as free, a ReLU layer of 2613 x 3072 x 768 went to those tiles: 35.2 us, now 27.9 on 128 x 128).  Measured, the difference
// to the plain product of the same tiles, 1848 and 2613 x 3072 x 768 and 4096 x 4096 x 1024, p = 0.1 (in brackets without dropout):
//              64 x 64             128 x 64            128 x 128           256 x 128           256 x 256
//   ReLU       .15-.16 (.05-.12)   .06-.16 (.04-.08)   .21-.29 (.08-.19)   .23-.26 (.12-.15)   .18-.24 (.06-.09)
//   GELU       .20-.32 (.14-.28)   .24-.34 (.20-.32)   .49-.65 (.35-.52)   .39-.46 (.28-.35)   .29-.37 (.20-.27)
//   ReLU back  .26-.32             .18-.32             .23-.34             .45-.58             .13-.18
//   GELU back  .51-.60             .71-.79             .62-.68             .75-.88             .36-.42
// With these numbers per form in place of the four, the same tiles come out at these sizes but for GELU at 2613 (128 x 64: 29.5
// for 30.2 alone, 32.6 for 31.6 within the layer) and ReLU's backward at 2560 x 2048 x 512 (24.4 for 22.2): the four stay.  Against
// the best tiles in brackets this takes at 1848 rows 20.2 (20.2), 23.3 (23.3), 23.7 (23.0), 28.1 (28.1) us in the order of the
// rows, at 2613 24.4 (24.4), 30.2 (29.5), 24.5 (24.5), 30.0 (30.0).
static int best_act_form(const TileProduct& p, unsigned forms, bool order) {
    int best = -1;
    double best_us = 0.;
    for (int f = 0; f < TILE_FORMS; ++f) {
        if (!(forms >> f & 1u) || (f == TILE_256x256 ? !wide_takes(p) : !p.akc)) continue;
        const Form& F = form_of(f, order);
        const long len = steps_of(p.a, 1), cnt = tiles_of(p.a, 1, F.bm, F.bn);
        const double packs = (double)F.bm * F.bn / (4 * 64 * 8) * F.per_cu, draw = p.a.gate ? 0. : f == TILE_256x256 ? 0.13 : 0.2;
        const double rounds = (double)((cnt + 256L * F.per_cu - 1) / (256L * F.per_cu));
        const double us = launch_us(&len, &cnt, 1, F) + rounds * packs * ((p.a.act == ACT_GELU ? 0.25 : 0.1) + draw);
        if (best < 0 || us < best_us) { best = f; best_us = us; }
    }
    return best;
}

int choose_act_form(const TileProduct& p) {
    constexpr unsigned all = kRingForms | 1u << TILE_256x256;
    if (!p.a.same_order) return best_act_form(p, all, false);
    const int form = best_act_form(p, all, true);
    return form == TILE_256x256 || form < 0 ? form : best_act_form(p, kRingForms, false);
}

bool summed_wide(const TileProduct& p) {
    if (!wide_takes(p)) return false;
    double us[TILE_FORMS];
    for (int f = 0; f < TILE_FORMS; ++f) {
        const Form& F = form_of(f, true);
        const long len = steps_of(p.a, p.a.splits), cnt = tiles_of(p.a, p.a.splits, F.bm, F.bn);
        us[f] = launch_us(&len, &cnt, 1, F);
    }
    return us[TILE_256x256] < *std::min_element(us, us + TILE_256x256);
}

void launch_tiles_act(const TileProduct& p, int form, hipStream_t st) {
    const GemmArgs& a = p.a;
    if (a.gate) a.act == ACT_GELU ? launch_act<EPI_GELU_GATE_COLSUM>(p, form, st) : launch_act<EPI_GATE_COLSUM>(p, form, st);
    else if (a.act == ACT_GELU) a.alone ? launch_act<EPI_GELU_ALONE>(p, form, st) : launch_act<EPI_GELU_DROPOUT>(p, form, st);
    else a.keep_words ? launch_act<EPI_RELU_DROPOUT_PRE>(p, form, st) : launch_act<EPI_RELU_DROPOUT>(p, form, st);
}

template <int NP>
static void launch_tiles_n(const TileProduct* p, int n, int form, FinishJobs* tail, hipStream_t st) {
    TileGroup<NP> G;
    int k1, k2;
    list_tiles<NP>(G, p, n, form, tail, k1, k2);
    launch_ring_as<NP, EPI_PLAIN>(G, form, k1, k2, G.workers + (unsigned)G.tail.n * G.tail_groups, st);
}

void launch_tiles(const TileProduct* p, int n, int form, FinishJobs* tail, hipStream_t st) {
    if (form == TILE_256x256) { launch_wide(p, n, tail, 0, st); return; }
    // One instance for two to seven products.  With another for up to three, and 2.0 KB of arguments in place of 3.7, a data and a weight
    // gradient (64 rows of E 512; 256, 1024 and 2613 of 768; 4096 of 1024; 8192 of 4096) take 9.28 us for 9.32, 15.1 for 15.2, 25.9 for 25.9,
    // 35.5 for 35.7, 65.6 for 64.9, 1586 for 1597: nothing either way.
    if (n == 1 && !(tail && tail->n)) launch_tiles_n<1>(p, n, form, tail, st);
    else launch_tiles_n<kMaxProducts>(p, n, form, tail, st);
}

}  // namespace sub
