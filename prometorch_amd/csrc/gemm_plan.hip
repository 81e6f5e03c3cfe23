// Which tiles cover a product.
#include "gemm_plan.h"

namespace ptm {

static inline int up_div(int a, int b) { return (a + b - 1) / b; }

// the kind that has rows x cols from column n0 on done first, on a chip that is at `before`
static int best_kind(const TileKind* kinds, int n_kinds, int rows, int n0, int cols, int steps, int splits, int section_n, const ChipTime& before) {
    int best = -1;
    float least = 0.0f;
    for (int k = 0; k < n_kinds; ++k) {
        if (section_n > 0 && (section_n % kinds[k].bn || n0 % kinds[k].bn)) continue;
        ChipTime t = before;
        const int64_t tiles = (int64_t)up_div(rows, kinds[k].bm) * up_div(cols, kinds[k].bn);
        t.run(tiles * splits, steps * kinds[k].step + kinds[k].ends);
        // of equal times the one that keeps fewer CUs busy: they share the power
        const float cost = t.last() + 1e-3f * (float)tiles * (steps * kinds[k].step + kinds[k].ends) / 256.0f;
        if (best < 0 || cost < least) best = k, least = cost;
    }
    return best;
}

static TilePlan find_plan(const TileKind* kinds, int n_kinds, int M, int N, int steps, int most_splits, int section_n, float second_kind) {
    TilePlan best{};
    best.splits = 0;
    for (int splits = 1; splits == 1 || (splits <= most_splits && splits * 4 <= steps); ++splits) {
        const int part = up_div(steps, splits);
        // the sums of a split are written here and read by the kernel behind
        const float sums = splits > 1 ? (float)splits * (float)M * (float)N * 2e-3f : 0.0f;
        for (int k = 0; k < n_kinds; ++k) {
            const TileKind& a = kinds[k];
            if (section_n > 0 && section_n % a.bn) continue;
            for (int whole = 0; whole < 2; ++whole) {  // rows: all in this kind, or the whole tiles only
                const int rows = whole ? M / a.bm : up_div(M, a.bm);
                if (rows == 0 || (whole && rows * a.bm == M)) continue;
                const int cols = up_div(N, a.bn);
                for (int full = 0; full < 2; ++full) {  // columns: all, or what fills rounds of the chip
                    int mine = cols;
                    if (full) {
                        const int64_t rounds = (int64_t)rows * cols * splits / 256;
                        mine = (int)(rounds * 256 / ((int64_t)rows * splits));
                        if (mine == 0 || mine >= cols) continue;
                    }
                    TilePlan p{};
                    p.splits = splits;
                    ChipTime t;
                    auto add = [&](int kind, int m0, int n0, int n1, int tm, int tn) {
                        p.regions.r[p.regions.n++] = {kind, p.wgs, m0, n0, n1, tm, tn};
                        p.wgs += tm * tn * splits;
                        p.lds = kinds[kind].lds > p.lds ? kinds[kind].lds : p.lds;
                        t.run((int64_t)tm * tn * splits, part * kinds[kind].step + kinds[kind].ends);
                    };
                    const int cut = mine < cols ? mine * a.bn : N, low = whole ? rows * a.bm : M;
                    if ((int64_t)rows * cols * splits > 0x3fffffff) continue;
                    add(k, 0, 0, cut, rows, mine);
                    if (t.last() + sums >= best.cost && best.splits) continue;
                    if (cut < N) {
                        const int b = best_kind(kinds, n_kinds, low, cut, N - cut, part, splits, section_n, t);
                        add(b, 0, cut, N, up_div(low, kinds[b].bm), up_div(N - cut, kinds[b].bn));
                    }
                    if (low < M) {
                        const int b = best_kind(kinds, n_kinds, M - low, 0, N, part, splits, section_n, t);
                        add(b, low, 0, N, up_div(M - low, kinds[b].bm), up_div(N, kinds[b].bn));
                    }
                    p.cost = t.last() + sums;
                    for (int i = 1; i < p.regions.n; ++i)
                        if (p.regions.r[i].kind != k) {
                            p.cost += second_kind;
                            break;
                        }
                    if (!best.splits || p.cost < best.cost) best = p;
                }
            }
        }
    }
    return best;
}

// A plan depends on its arguments alone, and a prompt asks for the same few in every layer: each thread keeps the last ones it made.
TilePlan plan_tiles(const TileKind* kinds, int n_kinds, int M, int N, int steps, int most_splits, int section_n, float second_kind) {
    struct Made {
        const TileKind* kinds;
        int M, N, steps, most, section;
        float second_kind;
        TilePlan plan;
    };
    constexpr int KEPT = 16;
    static thread_local Made made[KEPT];
    static thread_local int next = 0;
    for (const Made& m : made)
        if (m.kinds == kinds && m.M == M && m.N == N && m.steps == steps && m.most == most_splits && m.section == section_n && m.second_kind == second_kind) return m.plan;
    Made& m = made[next];
    next = (next + 1) % KEPT;
    m = {kinds, M, N, steps, most_splits, section_n, second_kind, find_plan(kinds, n_kinds, M, N, steps, most_splits, section_n, second_kind)};
    return m.plan;
}

}  // namespace ptm
