// Tile-plan compiler: stream metadata -> per-query-tile list of visible key tiles with 32x32 activity / mask bits.
// Stands in for block_tables (spinf_serve/packer.py:426-491); the visibility predicate is the one of
// spinf_serve/scorer.py:173-177, with the image groups of scorer.py:184-198 (the tokens of a group also see each other both
// ways).  Host code, no global state.
#include "spinf_tree.h"
#include "common.h"

#include <algorithm>
#include <exception>
#include <cstring>
#include <new>
#include <unordered_map>
#include <vector>

struct spinf_tileplan {
    int64_t n = 0;
    int32_t window = 0;
    int32_t ktile = SPINF_KTILE;     // keys per entry: 64, or 32 for the head dim 512 kernel (one sub-tile per entry)
    std::vector<int32_t> qt_ptr, kv_idx, order;
    std::vector<uint32_t> kv_bits;
    std::vector<int64_t> weight;     // cost of a query tile in 32 x 32 blocks: per key tile, 4 x the most blocks any row group sees
    std::vector<int32_t> group;      // job of the tile's first real row (-1: pads only)
    int64_t active = 0, masked = 0;
};

namespace {

struct Blk {            // aggregates of one 32-token block
    int32_t lo, hi;     // token range [lo, hi)
    bool all_real;      // every token is a real token
    bool any_real;
    int32_t job;        // the single job of its tokens, -2 if mixed / pads present
    int32_t lead;       // job of the first real token, -1 if there is none
    int32_t first;      // lowest key any of its rows may see: where the earliest job of its rows begins
    int32_t min_end, max_end;   // over all tokens (pads count as -1)
    int32_t min_pos, max_pos;   // over real tokens
};

// grp_mode 1: the group term holds past the window; 2: it is windowed like the rest (scorer.py:186-198)
inline bool visible(const int32_t* art, const int32_t* end, const int32_t* pos, const int32_t* grp, int32_t grp_mode, int32_t window,
                    int64_t q, int64_t k) {
    if (q == k) return true;
    const bool in_window = window <= 0 || ((int64_t)pos[q] - (int64_t)pos[k]) < (int64_t)window;
    const bool v = k <= q && art[q] >= 0 && art[k] == art[q] && q < (int64_t)end[k] && in_window;
    if (v || !grp) return v;
    return grp[q] >= 0 && grp[q] == grp[k] && (grp_mode == 1 || in_window);
}

// do two sorted lists share a value?
inline bool share(const std::vector<int32_t>& a, const std::vector<int32_t>& b) {
    size_t i = 0, j = 0;
    while (i < a.size() && j < b.size()) {
        if (a[i] == b[j]) return true;
        if (a[i] < b[j]) i++; else j++;
    }
    return false;
}

// do the 32 tokens of a block belong to one job?
inline bool one_job(const int32_t* art) {
    int32_t other = 0;
    for (int i = 1; i < SPINF_SUB; i++) other |= art[i] ^ art[0];
    return other == 0;
}

// smallest and largest of a block's 32 values
inline void min_max(const int32_t* x, int32_t* lo, int32_t* hi) {
    int32_t a = x[0], b = x[0];
    for (int i = 1; i < SPINF_SUB; i++) {
        a = std::min(a, x[i]);
        b = std::max(b, x[i]);
    }
    *lo = a;
    *hi = b;
}

// the blocks b .. e - 1 as one (the fields the tile tests below ask for); job: the one job of all of them, all of them real and whole, else -2
inline Blk joined(const std::vector<Blk>& blk, int64_t b, int64_t e) {
    Blk J = blk[b];
    bool whole = J.all_real && J.hi - J.lo == SPINF_SUB;
    for (int64_t i = b + 1; i < e; i++) {
        const Blk& B = blk[i];
        J.hi = B.hi;
        J.any_real |= B.any_real;
        if (B.job != J.job) J.job = -2;
        whole &= B.all_real && B.hi - B.lo == SPINF_SUB;
        J.min_end = std::min(J.min_end, B.min_end);
        J.max_end = std::max(J.max_end, B.max_end);
        J.min_pos = std::min(J.min_pos, B.min_pos);
        J.max_pos = std::max(J.max_pos, B.max_pos);
    }
    if (!whole) J.job = -2;
    return J;
}

// Does some row of R see some key of K, and does every row see every key?  The plain rule (no image groups), one key at a time: the
// rows that see a key are a 32-bit set: its subtree's interval, the rows of its job, and on a sliding layer the rows within the window.
// (A block pair that is partly visible, the common case here, is settled by its first two or three keys; evaluating the rule for
// all 1,024 pairs was nine tenths of a build; 64,896 tokens, 64-key entries: 10.7 -> 1.2 ms of one host core.)
inline void rows_of_keys(const int32_t* art, const int32_t* end, const int32_t* pos, int32_t window, const Blk& R, const Blk& K, bool* any, bool* all) {
    const int rows = R.hi - R.lo;
    const uint32_t full = rows == 32 ? ~0u : (1u << rows) - 1;
    *any = false;
    *all = rows == SPINF_SUB && K.hi - K.lo == SPINF_SUB;
    uint32_t mates = 0;      // rows of job `job`
    int32_t job = -1;
    for (int32_t k = K.lo; k < K.hi && (!*any || *all); k++) {
        uint32_t see = 0;
        const int32_t from = std::max(k, R.lo), to = std::min(end[k], R.hi);
        if (art[k] >= 0 && from < to) {
            if (art[k] != job) {
                job = art[k];
                mates = 0;
                if (R.job == job) mates = full;
                else
                    for (int i = 0; i < rows; i++) mates |= (uint32_t)(art[R.lo + i] == job) << i;
            }
            see = mates & (~0u << (from - R.lo)) & (~0u >> (32 - (to - R.lo)));
            if (window > 0 && see && R.max_pos - (int64_t)pos[k] >= window)
                for (int i = from - R.lo; i < to - R.lo; i++)
                    if (pos[R.lo + i] - (int64_t)pos[k] >= window) see &= ~(1u << i);
        }
        if (k >= R.lo && k < R.hi) see |= 1u << (k - R.lo);
        *any |= see != 0;
        *all &= see == full;
    }
}

}  // namespace

extern "C" int spinf_tileplan_build(const int32_t* art, const int32_t* end, const int32_t* pos, int64_t n, int32_t window,
                                    spinf_tileplan** out) {
    return spinf_tileplan_build_ktile(art, end, pos, nullptr, 0, n, window, SPINF_KTILE, out);
}

extern "C" int spinf_tileplan_build_groups(const int32_t* art, const int32_t* end, const int32_t* pos, const int32_t* grp, int32_t grp_mode,
                                           int64_t n, int32_t window, spinf_tileplan** out) {
    return spinf_tileplan_build_ktile(art, end, pos, grp, grp_mode, n, window, SPINF_KTILE, out);
}

extern "C" int spinf_tileplan_build_ktile(const int32_t* art, const int32_t* end, const int32_t* pos, const int32_t* grp, int32_t grp_mode,
                                          int64_t n, int32_t window, int32_t ktile, spinf_tileplan** out) {
    if (!out) return spinf_fail(SPINF_E_ARG, "tileplan_build: out is null");
    *out = nullptr;
    if (ktile != SPINF_KTILE && ktile != SPINF_SUB) return spinf_fail(SPINF_E_ARG, "tileplan_build: key tile %d not in {64, 32}", ktile);
    if (n < 0 || (n > 0 && (!art || !end || !pos))) return spinf_fail(SPINF_E_ARG, "tileplan_build: null metadata");
    if (grp && grp_mode != 1 && grp_mode != 2) return spinf_fail(SPINF_E_ARG, "tileplan_build: group mode %d not in {1, 2}", grp_mode);
    if (n > (int64_t)1 << 30) return spinf_fail(SPINF_E_ARG, "tileplan_build: stream too long");
    spinf_tileplan* p = new (std::nothrow) spinf_tileplan;
    if (!p) return spinf_fail(SPINF_E_NOMEM, "tileplan_build: out of memory");
    try {
        p->n = n;
        p->ktile = ktile;
        p->window = window > 0 ? window : 0;
        const int32_t W = p->window;
        const int64_t nqt = (n + SPINF_QTILE - 1) / SPINF_QTILE;
        const int64_t nb = (n + SPINF_SUB - 1) / SPINF_SUB;
        std::vector<Blk> blk(nb);
        std::unordered_map<int32_t, int32_t> first;   // first stream position of every job
        int32_t run_job = -1, run_first = 0;
        for (int64_t b = 0; b < nb; b++) {
            Blk& B = blk[b];
            B.lo = (int32_t)(b * SPINF_SUB);
            B.hi = (int32_t)std::min<int64_t>(n, (b + 1) * SPINF_SUB);
            B.all_real = true; B.any_real = false; B.job = -3; B.lead = -1; B.first = INT32_MAX;
            B.min_end = INT32_MAX; B.max_end = INT32_MIN; B.min_pos = INT32_MAX; B.max_pos = INT32_MIN;
            if (B.hi - B.lo == SPINF_SUB && art[B.lo] >= 0 && one_job(art + B.lo)) {   // nearly all blocks: plain minima and maxima, which vectorise
                min_max(end + B.lo, &B.min_end, &B.max_end);
                min_max(pos + B.lo, &B.min_pos, &B.max_pos);
                B.any_real = true;
                B.job = B.lead = art[B.lo];
                if (B.job != run_job) {
                    run_job = B.job;
                    run_first = first.emplace(B.job, B.lo).first->second;
                }
                B.first = run_first;
                continue;
            }
            for (int32_t i = B.lo; i < B.hi; i++) {
                const int32_t a = art[i];
                B.min_end = std::min(B.min_end, end[i]);
                B.max_end = std::max(B.max_end, end[i]);
                if (a < 0) {
                    B.all_real = false;
                    B.job = -2;
                    continue;
                }
                B.min_pos = std::min(B.min_pos, pos[i]);
                B.max_pos = std::max(B.max_pos, pos[i]);
                if (!B.any_real) B.lead = a;
                B.any_real = true;
                if (B.job == -3) B.job = a; else if (B.job != a) B.job = -2;
                if (a != run_job) {   // a job's tokens lie together: one look-up per run
                    run_job = a;
                    run_first = first.emplace(a, i).first->second;
                }
                B.first = std::min(B.first, run_first);
            }
            if (B.job == -3) B.job = -2;
        }
        // image groups: the distinct groups of every block (sorted), the first and last position of every group
        std::vector<std::vector<int32_t>> bgrp(grp ? nb : 0);
        std::unordered_map<int32_t, int64_t> gfirst, glast;
        if (grp) {
            for (int64_t i = 0; i < n; i++) {
                if (grp[i] < 0) continue;
                std::vector<int32_t>& g = bgrp[i / SPINF_SUB];
                if (std::find(g.begin(), g.end(), grp[i]) == g.end()) g.push_back(grp[i]);
                gfirst.emplace(grp[i], i);
                glast[grp[i]] = i;
            }
            for (auto& g : bgrp) std::sort(g.begin(), g.end());
        }
        p->qt_ptr.assign(nqt + 1, 0);
        std::vector<int64_t>& weight = p->weight;
        std::vector<int32_t>& group = p->group;
        weight.assign(nqt, 0);
        group.assign(nqt, -1);
        constexpr int QB = SPINF_QTILE / SPINF_SUB;
        const int KB = ktile / SPINF_SUB;
        std::vector<Blk> ktl;   // key tiles as one block each
        if (KB > 1)
            for (int64_t b = 0; b < nb; b += KB) ktl.push_back(joined(blk, b, std::min(nb, b + KB)));
        p->kv_idx.reserve((size_t)nqt * 8);
        p->kv_bits.reserve((size_t)nqt * 8);
        for (int64_t t = 0; t < nqt; t++) {
            const int64_t q0 = t * SPINF_QTILE, q1 = std::min<int64_t>(n, q0 + SPINF_QTILE);
            int64_t lo_key = q0, hi_key = q1;   // keys [lo_key, hi_key) can matter: the rows' jobs so far, and their groups (a group may lie in several jobs)
            for (int64_t rb = q0 / SPINF_SUB; rb < nb && blk[rb].lo < q1; rb++) {
                lo_key = std::min<int64_t>(lo_key, blk[rb].first);
                if (group[t] < 0) group[t] = blk[rb].lead;
            }
            for (int64_t q = q0; grp && q < q1; q++) {
                if (grp[q] < 0) continue;
                lo_key = std::min(lo_key, gfirst[grp[q]]);
                hi_key = std::max(hi_key, glast[grp[q]] + 1);
            }
            // Most tile pairs are one thing throughout, and settled as a whole: nothing seen (every key's subtree has ended, or lies behind the
            // window, and the tile before the rows), or everything (rows and keys of one job, the keys before the rows and their
            // subtrees to the tile's end, all within the window).  Block by block the tests below say the same.  (One host core, a
            // whole build: 64,896 tokens in 46 trunks with branches, 5,793 64-key entries under a window, 864 -> 477 us, of it some
            // 130 the aggregates of one-job blocks; 41,088 tokens in long trunks, 25,178 entries, 1,522 -> 375 us.)
            const Blk Q = joined(blk, t * QB, std::min(nb, (t + 1) * QB));
            const bool plain = !grp, whole = q1 - q0 == SPINF_QTILE && Q.job >= 0;
            for (int64_t j = lo_key / ktile; j * ktile < hi_key; j++) {
                const Blk& T = KB > 1 ? ktl[j] : blk[j];
                if (plain && T.hi <= q0) {
                    if (T.max_end <= q0 || (W > 0 && Q.any_real && T.any_real && (int64_t)Q.min_pos - T.max_pos >= W)) continue;
                    if (whole && T.hi - T.lo == ktile && T.job == Q.job && T.min_end >= q1 && (W == 0 || (int64_t)Q.max_pos - T.min_pos < W)) {
                        p->kv_idx.push_back((int32_t)j);
                        p->kv_bits.push_back(KB > 1 ? 0xffu : 0x55u);
                        p->active += QB * KB;
                        weight[t] += QB * KB;
                        continue;
                    }
                }
                uint32_t bits = 0;
                for (int w = 0; w < SPINF_QTILE / SPINF_SUB; w++) {
                    const int64_t rb = q0 / SPINF_SUB + w;
                    if (rb >= nb) break;
                    const Blk& R = blk[rb];
                    for (int s = 0; s < ktile / SPINF_SUB; s++) {
                        const int64_t kb = j * (ktile / SPINF_SUB) + s;
                        if (kb >= nb) break;
                        const Blk& K = blk[kb];
                        const bool grouped = grp && share(bgrp[rb], bgrp[kb]);   // some row and some key are of one image
                        if (K.lo > R.hi - 1 && !grouped) continue;           // every key after every row
                        const bool below = K.hi - 1 < R.lo;                  // every key strictly before every row
                        bool any, all;
                        if (grouped) {
                            any = false; all = (R.hi - R.lo) == SPINF_SUB && (K.hi - K.lo) == SPINF_SUB;
                            for (int64_t q = R.lo; q < R.hi; q++)
                                for (int64_t k = K.lo; k < K.hi; k++) {
                                    const bool v = visible(art, end, pos, grp, grp_mode, W, q, k);
                                    any |= v; all &= v;
                                }
                        } else if (below && K.max_end <= R.lo) { any = false; all = false; }
                        else if (below && W > 0 && R.any_real && K.any_real && (int64_t)R.min_pos - K.max_pos >= W) { any = false; all = false; }
                        else if (K.hi - 1 <= R.lo && R.all_real && K.all_real && R.job >= 0 && R.job == K.job && K.min_end >= R.hi &&
                                 (W == 0 || (int64_t)R.max_pos - K.min_pos < W) && (R.hi - R.lo) == SPINF_SUB && (K.hi - K.lo) == SPINF_SUB) {
                            any = true; all = true;
                        } else {
                            rows_of_keys(art, end, pos, W, R, K, &any, &all);
                        }
                        if (any) {
                            bits |= 1u << (2 * w + s);
                            p->active++;
                            if (!all) { bits |= 1u << (8 + 2 * w + s); p->masked++; }
                        }
                    }
                }
                if (bits) {
                    p->kv_idx.push_back((int32_t)j);
                    p->kv_bits.push_back(bits);
                    // the four row groups of a query tile go through its key tiles in step: a key tile costs what its busiest
                    // row group costs, whether the other three have work or not
                    int most = 0;
                    for (int w = 0; w < SPINF_QTILE / SPINF_SUB; w++) most = std::max<int>(most, ((bits >> (2 * w)) & 1u) + ((bits >> (2 * w + 1)) & 1u));
                    weight[t] += (SPINF_QTILE / SPINF_SUB) * most;
                }
            }
            p->qt_ptr[t + 1] = (int32_t)p->kv_idx.size();
        }
        // launch order: runs of query tiles of one job stay together (they share keys), heaviest first inside a run
        p->order.resize(nqt);
        for (int64_t t = 0; t < nqt; t++) p->order[t] = (int32_t)t;
        int64_t a = 0;
        while (a < nqt) {
            int64_t b = a + 1;
            while (b < nqt && group[b] == group[a]) b++;
            std::stable_sort(p->order.begin() + a, p->order.begin() + b, [&](int32_t x, int32_t y) { return weight[x] > weight[y]; });
            a = b;
        }
    } catch (const std::exception&) {
        delete p;
        return spinf_fail(SPINF_E_NOMEM, "tileplan_build: out of memory");
    }
    *out = p;
    return SPINF_OK;
}

extern "C" int spinf_tileplan_counts(const spinf_tileplan* p, int64_t counts[5]) {
    if (!p || !counts) return spinf_fail(SPINF_E_ARG, "tileplan_counts: null argument");
    counts[0] = (int64_t)p->order.size();
    counts[1] = (int64_t)p->kv_idx.size();
    counts[2] = p->active;
    counts[3] = p->masked;
    counts[4] = p->n;
    return SPINF_OK;
}

extern "C" int spinf_tileplan_export(const spinf_tileplan* p, int32_t* qt_ptr, int32_t* kv_idx, uint32_t* kv_bits, int32_t* order) {
    if (!p || !qt_ptr) return spinf_fail(SPINF_E_ARG, "tileplan_export: null argument");
    if ((!kv_idx || !kv_bits) && !p->kv_idx.empty()) return spinf_fail(SPINF_E_ARG, "tileplan_export: null entry arrays");
    if (!order && !p->order.empty()) return spinf_fail(SPINF_E_ARG, "tileplan_export: null order array");
    std::memcpy(qt_ptr, p->qt_ptr.data(), p->qt_ptr.size() * sizeof(int32_t));
    if (!p->kv_idx.empty()) {
        std::memcpy(kv_idx, p->kv_idx.data(), p->kv_idx.size() * sizeof(int32_t));
        std::memcpy(kv_bits, p->kv_bits.data(), p->kv_bits.size() * sizeof(uint32_t));
    }
    if (!p->order.empty()) std::memcpy(order, p->order.data(), p->order.size() * sizeof(int32_t));
    return SPINF_OK;
}

extern "C" int spinf_tileplan_schedule(const spinf_tileplan* p, int32_t head_groups, int32_t* items, int32_t* list_ptr) {
    if (!p || !list_ptr) return spinf_fail(SPINF_E_ARG, "tileplan_schedule: null argument");
    if (head_groups <= 0 || head_groups >= 4096) return spinf_fail(SPINF_E_ARG, "tileplan_schedule: head groups %d out of range", head_groups);
    const int64_t nqt = (int64_t)p->order.size();
    if (nqt && !items) return spinf_fail(SPINF_E_ARG, "tileplan_schedule: null items");
    if (nqt * head_groups > (int64_t)1 << 30) return spinf_fail(SPINF_E_ARG, "tileplan_schedule: too many items");
    try {
        // items: job run by job run (tiles that share keys), head group by head group, heaviest tile first
        std::vector<int64_t> cum;
        cum.reserve(nqt * head_groups + 1);
        cum.push_back(0);
        int64_t k = 0;
        int64_t a = 0;
        while (a < nqt) {
            int64_t b = a + 1;
            while (b < nqt && p->group[p->order[b]] == p->group[p->order[a]]) b++;
            for (int32_t hp = 0; hp < head_groups; hp++)
                for (int64_t pos = a; pos < b; pos++) {
                    const int32_t t = p->order[pos];
                    const int32_t e0 = p->qt_ptr[t], ne = p->qt_ptr[t + 1] - e0;
                    items[4 * k + 0] = t;
                    items[4 * k + 1] = e0;
                    items[4 * k + 2] = (ne & 0xfffff) | (hp << 20);
                    items[4 * k + 3] = ne > 0 ? p->kv_idx[e0] : 0;
                    cum.push_back(cum.back() + p->weight[t] + 15);   // + a fixed cost per item (queries, output rows; measured ~15 blocks)
                    k++;
                }
            a = b;
        }
        // eight contiguous lists of about equal weight
        const int64_t total = cum.back();
        list_ptr[0] = 0;
        for (int l = 1; l < 8; l++) {
            const int64_t want = total * l / 8;
            const int64_t at = std::lower_bound(cum.begin(), cum.end(), want) - cum.begin();
            list_ptr[l] = (int32_t)std::max<int64_t>(list_ptr[l - 1], std::min<int64_t>(at, k));
        }
        list_ptr[8] = (int32_t)k;
        // The end of a list decides how evenly the workgroups finish: the pass ends up to an item's duration after the lists
        // run dry.  The lightest items of each list (at most TAIL_SHARE of its weight and TAIL_ITEMS items) are therefore
        // moved to its end, heaviest of them first.  A small share on purpose: moved items no longer run next to the items
        // that share their keys (measured on the 24-content pass: 8 % of the weight -1 %, 25 % +2 %, 35 % +3 % kernel time).
        constexpr double TAIL_SHARE = 0.08;
        constexpr int64_t TAIL_ITEMS = 128;
        std::vector<uint64_t> idx;   // weight << 32 | place
        std::vector<int32_t> tmp;
        std::vector<char> moved;
        for (int l = 0; l < 8; l++) {
            const int64_t lo = list_ptr[l], hi = list_ptr[l + 1];
            if (hi - lo < 3) continue;
            auto cost = [&](int64_t i) { return cum[i + 1] - cum[i]; };
            // the TAIL_ITEMS lightest, in order, are all that can move (selected, then sorted: kept in order during the selection they were the
            // larger part of a schedule; an item's weight is below 2^31: at most 4 blocks for each of 2^26 key tiles)
            idx.resize(hi - lo);
            for (int64_t i = lo; i < hi; i++) idx[i - lo] = (uint64_t)cost(i) << 32 | (uint64_t)i;
            const size_t lightest = std::min<size_t>(idx.size(), (size_t)TAIL_ITEMS);
            if (lightest < idx.size()) std::nth_element(idx.begin(), idx.begin() + lightest, idx.end());
            std::sort(idx.begin(), idx.begin() + lightest);
            auto at = [&](int64_t j) { return (int64_t)(idx[j] & 0xffffffffu); };
            const int64_t budget = (int64_t)(TAIL_SHARE * (double)(cum[hi] - cum[lo]));
            int64_t taken = 0, n_tail = 0;
            while (n_tail < (int64_t)lightest && taken + cost(at(n_tail)) <= budget) taken += cost(at(n_tail++));
            if (n_tail == 0) continue;
            moved.assign((size_t)(hi - lo), 0);
            for (int64_t j = 0; j < n_tail; j++) moved[at(j) - lo] = 1;
            tmp.resize(4 * (size_t)(hi - lo));
            int32_t* to = tmp.data();
            for (int64_t i = lo; i < hi; i++)
                if (!moved[i - lo]) { std::memcpy(to, items + 4 * i, 4 * sizeof(int32_t)); to += 4; }
            for (int64_t j = n_tail - 1; j >= 0; j--) { std::memcpy(to, items + 4 * at(j), 4 * sizeof(int32_t)); to += 4; }
            std::memcpy(items + 4 * lo, tmp.data(), tmp.size() * sizeof(int32_t));
        }
    } catch (const std::exception&) {
        return spinf_fail(SPINF_E_NOMEM, "tileplan_schedule: out of memory");
    }
    return SPINF_OK;
}

// Static schedule for the kernel with decoupled waves: the items of spinf_tileplan_schedule (same order, same eight lists, one per
// XCD), dealt out to n_lists workgroups by simulating "the workgroup that is free first takes the next item of its XCD's list"
// with a cost model, so that a workgroup's items are known before the launch.  Workgroup b serves list b % 8.  The model is a
// fit to per-workgroup cycle counts of that kernel on the 24-content pass (residual 1.2 %): a workgroup moves through its key
// tiles at about the same pace whatever the number of 32 x 32 blocks its waves compute in them, so an item costs its number of
// key tiles, 0.3 per block that needs the per-element mask (of the busier SIMD pair: SIMDs 0 and 3 run the row groups 0 and 3 of
// a query tile, SIMDs 1 and 2 the row groups 1 and 2) and 3.2 on top (queries, output rows).
extern "C" int spinf_tileplan_schedule_static(const spinf_tileplan* p, int32_t head_groups, int32_t n_lists, int32_t* items, int32_t* list_ptr) {
    if (!p || !list_ptr) return spinf_fail(SPINF_E_ARG, "tileplan_schedule_static: null argument");
    if (n_lists <= 0 || n_lists > 65536) return spinf_fail(SPINF_E_ARG, "tileplan_schedule_static: %d lists out of range", n_lists);
    const int64_t nqt = (int64_t)p->order.size();
    try {
        std::vector<int32_t> base((size_t)std::max<int64_t>(1, nqt * head_groups) * 4);
        int32_t lp[9];
        if (int rc = spinf_tileplan_schedule(p, head_groups, base.data(), lp)) return rc;
        // per 32-key block of an entry: does any row group see it, and how many blocks of each SIMD pair need the mask
        std::vector<float> cost(nqt, 0.f);
        for (int64_t t = 0; t < nqt; t++) {
            if (p->ktile != SPINF_SUB) {   // 64-key entries: the lockstep kernels, whose items cost what spinf_tileplan_schedule weighs them with
                cost[t] = (float)(p->weight[t] + 15);
                continue;
            }
            int tiles = 0, ma = 0, mb = 0;
            for (int32_t e = p->qt_ptr[t]; e < p->qt_ptr[t + 1]; e++) {
                const uint32_t bits = p->kv_bits[e], masked = bits & (bits >> 8);
                tiles += (bits & 0x55u) != 0;
                ma += (int)((masked & 1u) + (masked >> 6 & 1u));        // row groups 0 and 3
                mb += (int)((masked >> 2 & 1u) + (masked >> 4 & 1u));   // row groups 1 and 2
            }
            cost[t] = 3.2f + (float)tiles + 0.3f * (float)std::max(ma, mb);
        }
        // the workgroup of a list that is free first (the lowest numbered of equals) takes its next item: a heap per list, of the time it is
        // free at (bits of a float that is not negative, which order as the float does) << 32 | workgroup
        const int nl = std::min<int32_t>(8, n_lists);
        std::vector<int32_t> owner((size_t)std::max<int64_t>(1, nqt * head_groups));
        std::vector<std::vector<uint64_t>> free_at((size_t)nl);
        for (auto& f : free_at) f.reserve((size_t)n_lists / nl + 1);
        for (int w = 0; w < n_lists; w++) free_at[w % nl].push_back((uint64_t)w);   // (ascending: a heap as it is)
        for (int w = 0; w <= n_lists; w++) list_ptr[w] = 0;
        for (int l = 0; l < 8; l++)
            for (int64_t i = lp[l]; i < lp[l + 1]; i++) {
                std::vector<uint64_t>& f = free_at[l % nl];
                const uint32_t w = (uint32_t)f[0], was = (uint32_t)(f[0] >> 32);
                owner[i] = (int32_t)w;
                list_ptr[w + 1]++;
                float at;
                std::memcpy(&at, &was, sizeof at);
                at += cost[base[4 * i]];
                uint32_t now;
                std::memcpy(&now, &at, sizeof now);
                const uint64_t key = (uint64_t)now << 32 | w;   // back in from the top
                size_t k = 0;
                for (size_t c; (c = 2 * k + 1) < f.size(); k = c) {
                    c += c + 1 < f.size() && f[c + 1] < f[c];
                    if (key <= f[c]) break;
                    f[k] = f[c];
                }
                f[k] = key;
            }
        for (int w = 0; w < n_lists; w++) list_ptr[w + 1] += list_ptr[w];
        std::vector<int32_t> fill(list_ptr, list_ptr + n_lists);
        for (int l = 0; l < 8; l++)
            for (int64_t i = lp[l]; i < lp[l + 1]; i++) std::memcpy(items + 4 * (int64_t)fill[owner[i]]++, base.data() + 4 * i, 4 * sizeof(int32_t));
    } catch (const std::exception&) {
        return spinf_fail(SPINF_E_NOMEM, "tileplan_schedule_static: out of memory");
    }
    return SPINF_OK;
}

extern "C" int spinf_tileplan_row0(const spinf_tileplan* p, const int32_t* row_of, int32_t* kv_row0) {
    if (!p || !row_of) return spinf_fail(SPINF_E_ARG, "tileplan_row0: null argument");
    if (!kv_row0 && !p->kv_idx.empty()) return spinf_fail(SPINF_E_ARG, "tileplan_row0: null kv_row0");
    for (size_t e = 0; e < p->kv_idx.size(); e++) {
        const int64_t k0 = (int64_t)p->kv_idx[e] * p->ktile;
        int32_t r0 = k0 + p->ktile <= p->n ? row_of[k0] : -1;
        for (int64_t j = 1; r0 >= 0 && j < p->ktile; j++)
            if (row_of[k0 + j] != r0 + j) r0 = -1;
        kv_row0[e] = r0;
    }
    return SPINF_OK;
}

extern "C" void spinf_tileplan_free(spinf_tileplan* p) { delete p; }
