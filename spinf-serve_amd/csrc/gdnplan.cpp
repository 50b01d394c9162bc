// Plan compiler of the recurrent (Gated DeltaNet) layers: the packed token forest -> segments, levels and kernel calls.
// Stands in for tree_plan (spinf_serve/models/qwen35/qwen.py:158-276); its output is what gdn_tree / gdn_indexed
// (qwen.py:514-590) walk.  Host code, no global state, deterministic.
//
// What it computes.  A token's `prev` is the token before it on its root-to-leaf path.  A *segment* is a maximal run of
// stream-consecutive real tokens that one scan can take in one go: it begins at a real token whose predecessor is missing, is
// not the stream token right before it, or has several children.  Segments form a forest (a segment's parent is the segment of
// its first token's predecessor); the scan of a segment starts from its parent's final state, so segments are run level by level
// and only segments that somebody continues from (or that the caller asks for) leave their state, in a slot of their level.
//
// How.  One pass over the stream numbers the segments and, because a parent always precedes its children in the stream, gives
// their depth at once; a counting sort by depth keeps stream order inside a level; calls are cut from the sorted array.
#include "spinf_tree.h"
#include "common.h"
#include "gdn_forest.h"

#include <algorithm>
#include <exception>
#include <cstring>
#include <new>
#include <vector>

struct spinf_gdn_plan {
    int64_t n_segments = 0, conv_rows = 0;
    std::vector<int64_t> level_ptr;      // calls of level d: level_ptr[d] .. level_ptr[d+1]
    std::vector<int32_t> call_kind;      // 1 chunked, 0 recurrent
    std::vector<int32_t> call_keep;      // some segment of the call leaves its state
    std::vector<int64_t> call_seg_ptr;   // segments of call c: call_seg_ptr[c] .. call_seg_ptr[c+1] in cu / h0 / ht
    std::vector<int64_t> call_row_ptr;   // rows of call c in idx
    std::vector<int64_t> len, h0, ht;    // per call segment: length, slot of the start state in the level above (-1 zero), slot of its own (-1 none)
    std::vector<int64_t> idx;            // rows of the calls' segments, back to back
    std::vector<int64_t> n_keep;         // slots per level
    std::vector<int64_t> conv;           // [conv_rows, 4]
    std::vector<int64_t> seg_of_row, seg_level, seg_slot;
    std::vector<int64_t> prog, prog_data;   // launches [*, 8] and what they read (spinf_gdn_plan_program)
};

namespace {

struct Seg {
    int64_t first, len, parent;
    int32_t depth;
    bool keeps;
    bool wanted;   // the caller asked for its state
};

// ---- the program: forests apart (see gdn_forest.hip), the rest level by level
constexpr int64_t FOREST_TREE = 1024;   // tokens of one tree, at most: a tree is one workgroup's work, and it should not outlast the level
// A unit's tokens, at most (a larger tree is a unit of its own).  Fixed, and a unit never spans two parents, so that a content's blocks, and with
// them the bits of its outputs, do not depend on what else is in the stream.  Four blocks: the state a unit loads first costs about as much
// as one block, and a small stream needs its units side by side.  One layer with units of 32 / 64 / 128 / 256 / 512 tokens: 22 tries of 480 tokens
// 522 / 487 / 475 / 464 / 484 us, one of them 76 / 75 / 82 / 98 / 127, 54 of 200 949 / 921 / 899 / 907 / 904.
constexpr int64_t FOREST_UNIT = 128;

template <class Row>
void build_program(spinf_gdn_plan* p, const std::vector<Seg>& seg, int32_t n_levels, const std::vector<int64_t>& by_level, const std::vector<int64_t>& at, int32_t short_len, Row row) {
    const int64_t ns = (int64_t)seg.size();
    // per segment: can its subtree be (part of) a forest's tree; the subtree's tokens and its longest path
    std::vector<char> fits(ns, 1), inside(ns, 0);
    std::vector<int64_t> tokens(ns, 0), path(ns, 0);
    for (int64_t s = ns - 1; s >= 0; s--) {
        tokens[s] += seg[s].len;
        path[s] += seg[s].len;
        if (seg[s].len > short_len || seg[s].wanted || path[s] > GDN_FOREST_DEPTH || tokens[s] > FOREST_TREE) fits[s] = 0;
        const int64_t up = seg[s].parent;
        if (up >= 0) {
            fits[up] &= fits[s];
            tokens[up] += tokens[s];
            path[up] = std::max(path[up], path[s]);
        }
    }
    // children (in stream order) of every segment, and of none (index ns)
    std::vector<int64_t> ptr(ns + 2, 0), kid(ns);
    for (const Seg& s : seg) ptr[(s.parent >= 0 ? s.parent : ns) + 1]++;
    for (int64_t s = 0; s <= ns; s++) ptr[s + 1] += ptr[s];
    {
        std::vector<int64_t> fill(ptr.begin(), ptr.end() - 1);
        for (int64_t s = 0; s < ns; s++) kid[fill[seg[s].parent >= 0 ? seg[s].parent : ns]++] = s;
    }
    // A parent's children are taken as a forest if one of them forks.  Leaves alone leave no state that could be saved, only fuller blocks, and
    // the recurrent entry point's smaller workgroups start sooner: a layer over 6 leaves of 8 tokens takes 55.0 us against 57.3, 108 such
    // leaves 139 / 146, 168 of 7 125.6 / 124.9, 320 of 6.5 369 / 355, 325 of 14 253 / 236.
    std::vector<char> forks(ns, 0);
    for (int64_t s = 0; s < ns; s++)
        if (fits[s] && ptr[s + 1] > ptr[s] && seg[s].parent >= 0) forks[seg[s].parent] = 1;
    bool any = false;
    for (int64_t s = 0; s < ns; s++) {
        const int64_t up = seg[s].parent;
        inside[s] = (up >= 0 && inside[up]) || (fits[s] && (up >= 0 ? forks[up] : ptr[s + 1] > ptr[s]));
        any |= inside[s];
    }
    if (!any) return;
    const int64_t B = GDN_FOREST_BLOCK;

    // units, by the level that runs them
    struct Level { std::vector<int64_t> cu{0}, h0; std::vector<int32_t> table; };
    std::vector<Level> lev(n_levels);
    std::vector<int64_t> stack;
    std::vector<int32_t> where, up, dep, rowv;    // of a unit's tokens: parent token in the unit (-1 none), depth, tensor row; last token of a segment
    where.assign(ns, -1);
    auto flush = [&](Level& L, int64_t slot) {
        const int64_t n = (int64_t)rowv.size();
        if (!n) return;
        size_t o = L.table.size();
        L.table.resize(o + (size_t)((n + B - 1) / B) * GDN_FOREST_INTS);
        for (int64_t f = 0; f < n; f += B, o += GDN_FOREST_INTS) {
            const int64_t e = std::min(n, f + B), next = f + B < n ? dep[f + B] : 0;
            int32_t* const rows_out = L.table.data() + o;
            uint32_t* const mask = (uint32_t*)rows_out + B;        // (signed and unsigned of one type may alias)
            uint32_t* const packed = mask + B;
            const uint32_t both = (uint32_t)dep[f] << 16 | (uint32_t)next << 24;
            for (int64_t i = f; i < e; i++) {
                const int64_t a = up[i];
                rows_out[i - f] = rowv[i];
                mask[i - f] = a >= f ? mask[a - f] | 1u << (a - f) : 0;
                // (pre-order: a token above i in an earlier block is above the block's first token)
                packed[i - f] = a >= f ? packed[a - f] : (a >= 0 ? (uint32_t)dep[a] + 1 : 0u) | both;
            }
            for (int64_t i = e; i < f + B; i++) { rows_out[i - f] = -1; mask[i - f] = 0; packed[i - f] = both; }
            if (f + B < n)
                for (int64_t a = up[f + B]; a >= f; a = up[a]) packed[a - f] |= (uint32_t)(dep[a] + 1) << 8;
        }
        L.cu.push_back(L.cu.back() + (n + B - 1) / B);
        L.h0.push_back(slot);
        rowv.clear(); up.clear(); dep.clear();
    };
    for (int64_t u = -1; u < ns; u++) {      // the trees below segment u (-1: below none)
        const int64_t of = u < 0 ? ns : u;
        if (u >= 0 && inside[u]) continue;
        Level* L = nullptr;
        const int64_t slot = u >= 0 ? p->seg_slot[u] : -1;
        for (int64_t k = ptr[of]; k < ptr[of + 1]; k++) {
            const int64_t head = kid[k];
            if (!inside[head]) continue;
            L = &lev[seg[head].depth];
            if (!rowv.empty() && (u < 0 || (int64_t)rowv.size() + tokens[head] > FOREST_UNIT)) flush(*L, slot);
            stack.assign(1, head);
            while (!stack.empty()) {
                const int64_t s = stack.back();
                stack.pop_back();
                int32_t last = s == head ? -1 : where[seg[s].parent];
                for (int64_t t = 0; t < seg[s].len; t++) {
                    up.push_back(last);
                    dep.push_back(last >= 0 ? dep[last] + 1 : 0);
                    last = (int32_t)rowv.size();
                    rowv.push_back((int32_t)row(seg[s].first + t));
                }
                where[s] = last;
                for (int64_t j = ptr[s + 1] - 1; j >= ptr[s]; j--) stack.push_back(kid[j]);
            }
        }
        if (L) flush(*L, slot);
    }

    // what is left of each level, then its units
    auto put = [&](const void* x, size_t n) {     // n pieces of 8 bytes
        const size_t o = (p->prog_data.size() + 1) / 2 * 2;
        p->prog_data.resize(o + n);
        if (n) std::memcpy(p->prog_data.data() + o, x, n * 8);
        return (int64_t)o;
    };
    std::vector<int64_t> cu, h0, ht, idx;
    for (int32_t d = 0; d < n_levels; d++) {
        for (int kind = 1; kind >= 0; kind--) {
            cu.assign(1, 0); h0.clear(); ht.clear(); idx.clear();
            int64_t longest = 0;
            bool keeps = false;
            for (int64_t i = at[d]; i < at[d + 1]; i++) {
                const Seg& s = seg[by_level[i]];
                if (inside[by_level[i]] || (s.len > short_len) != (kind == 1)) continue;
                cu.push_back(cu.back() + s.len);
                h0.push_back(d > 0 ? p->seg_slot[s.parent] : -1);
                ht.push_back(s.keeps ? p->seg_slot[by_level[i]] : -1);
                keeps |= s.keeps;
                longest = std::max(longest, s.len);
                for (int64_t t = 0; t < s.len; t++) idx.push_back(row(s.first + t));
            }
            if (h0.empty()) continue;
            const int64_t rec[8] = {d, kind, (int64_t)h0.size(), kind ? longest : 0, put(cu.data(), cu.size()), put(idx.data(), idx.size()),
                                    d > 0 ? put(h0.data(), h0.size()) : -1, keeps ? put(ht.data(), ht.size()) : -1};
            p->prog.insert(p->prog.end(), rec, rec + 8);
        }
        const Level& L = lev[d];
        if (L.h0.empty()) continue;
        const int64_t rec[8] = {d, 2, (int64_t)L.h0.size(), 0, put(L.cu.data(), L.cu.size()), put(L.table.data(), L.table.size() / 2),   // (GDN_FOREST_INTS is even)
                                d > 0 ? put(L.h0.data(), L.h0.size()) : -1, -1};
        p->prog.insert(p->prog.end(), rec, rec + 8);
    }
}

}  // namespace

extern "C" int spinf_gdn_plan_build(const int64_t* prev, const uint8_t* real, int64_t n, int32_t path, int32_t short_len, int64_t call_tokens,
                                    int32_t max_init, int64_t rows, const int64_t* keep, int64_t n_keep, spinf_gdn_plan** out) {
    if (!out) return spinf_fail(SPINF_E_ARG, "gdn_plan_build: out is null");
    *out = nullptr;
    if (n < 0 || (n > 0 && (!prev || !real))) return spinf_fail(SPINF_E_ARG, "gdn_plan_build: null stream arrays");
    if (path != 0 && path != 1) return spinf_fail(SPINF_E_ARG, "gdn_plan_build: unknown path %d (0 indexed, 1 levels)", path);
    if (n_keep < 0 || (n_keep > 0 && !keep)) return spinf_fail(SPINF_E_ARG, "gdn_plan_build: null keep list");
    if (rows > INT32_MAX) return spinf_fail(SPINF_E_ARG, "gdn_plan_build: %lld compact rows (row indices are below 2^31)", (long long)rows);
    if (path == 1 && max_init <= 0) return spinf_fail(SPINF_E_ARG, "gdn_plan_build: max_init must be positive");
    for (int64_t i = 0; i < n; i++)
        if (prev[i] >= i || prev[i] < -1) return spinf_fail(SPINF_E_ARG, "gdn_plan_build: prev[%lld] = %lld does not point backwards", (long long)i, (long long)prev[i]);
    spinf_gdn_plan* p = new (std::nothrow) spinf_gdn_plan;
    if (!p) return spinf_fail(SPINF_E_NOMEM, "gdn_plan_build: out of memory");
    try {
        // ---- compact rows: real tokens first, in stream order; `rows` doubles as the "no row" value
        int64_t n_real = 0;
        for (int64_t i = 0; i < n; i++) n_real += real[i] != 0;
        const bool compact = rows >= 0;
        if (compact && n_real > rows) {
            delete p;
            return spinf_fail(SPINF_E_ARG, "gdn_plan_build: %lld real tokens do not fit %lld compact rows", (long long)n_real, (long long)rows);
        }
        std::vector<int64_t> row_of;   // stream position -> row of the tensors
        if (compact) {
            row_of.assign(n, rows);
            int64_t r = 0;
            for (int64_t i = 0; i < n; i++)
                if (real[i]) row_of[i] = r++;
        }
        auto row = [&](int64_t i) { return compact ? row_of[i] : i; };

        // ---- segments, in one pass
        std::vector<int32_t> kids(n, 0);
        for (int64_t i = 0; i < n; i++)
            if (prev[i] >= 0) kids[prev[i]]++;
        std::vector<Seg> seg;
        std::vector<int64_t> seg_at(n, -1);
        for (int64_t i = 0; i < n; i++) {
            if (!real[i]) continue;
            const int64_t b = prev[i];
            const bool opens = b < 0 || b != i - 1 || kids[b] > 1 || !real[b];   // (a pad is in no segment)
            if (opens) {
                Seg s;
                s.first = i;
                s.len = 0;
                s.parent = b >= 0 ? seg_at[b] : -1;
                s.depth = s.parent >= 0 ? seg[s.parent].depth + 1 : 0;
                s.keeps = s.wanted = false;
                if (s.parent >= 0) seg[s.parent].keeps = true;   // somebody continues from it
                seg.push_back(s);
            }
            seg_at[i] = (int64_t)seg.size() - 1;
            seg.back().len++;
        }
        for (int64_t j = 0; j < n_keep; j++) {
            const int64_t i = keep[j];
            if (i >= 0 && i < n && real[i]) seg[seg_at[i]].keeps = seg[seg_at[i]].wanted = true;   // the caller wants this segment's state
        }
        const int64_t ns = (int64_t)seg.size();
        p->n_segments = ns;

        // ---- counting sort by depth (stream order inside a level)
        int32_t n_levels = 0;
        for (const Seg& s : seg) n_levels = std::max(n_levels, s.depth + 1);
        std::vector<int64_t> at(n_levels + 1, 0);
        for (const Seg& s : seg) at[s.depth + 1]++;
        for (int32_t d = 0; d < n_levels; d++) at[d + 1] += at[d];
        std::vector<int64_t> by_level(ns);
        {
            std::vector<int64_t> fill(at.begin(), at.end() - 1);
            for (int64_t s = 0; s < ns; s++) by_level[fill[seg[s].depth]++] = s;
        }

        // ---- levels and calls
        p->seg_slot.assign(ns, -1);
        p->seg_level.resize(ns);
        for (int64_t s = 0; s < ns; s++) p->seg_level[s] = seg[s].depth;
        p->level_ptr.push_back(0);
        p->call_seg_ptr.push_back(0);
        p->call_row_ptr.push_back(0);
        auto emit = [&](const int64_t* first, const int64_t* last, int32_t kind, int32_t level) {   // one call over these segments
            bool any_keep = false;
            for (const int64_t* it = first; it != last; ++it) {
                const Seg& s = seg[*it];
                p->len.push_back(s.len);
                p->h0.push_back(level > 0 && s.parent >= 0 ? p->seg_slot[s.parent] : -1);
                p->ht.push_back(s.keeps ? p->seg_slot[*it] : -1);
                any_keep |= s.keeps;
                for (int64_t t = 0; t < s.len; t++) p->idx.push_back(row(s.first + t));
            }
            p->call_kind.push_back(kind);
            p->call_keep.push_back(any_keep);
            p->call_seg_ptr.push_back((int64_t)p->len.size());
            p->call_row_ptr.push_back((int64_t)p->idx.size());
        };
        std::vector<int64_t> group;
        for (int32_t d = 0; d < n_levels; d++) {
            const int64_t* lo = by_level.data() + at[d];
            const int64_t* hi = by_level.data() + at[d + 1];
            if (path == 0) {
                // slots of the level: its keeping segments, in stream order
                int64_t slots = 0;
                for (const int64_t* it = lo; it != hi; ++it)
                    if (seg[*it].keeps) p->seg_slot[*it] = slots++;
                p->n_keep.push_back(slots);
                // the long segments go to the chunked kernel, cut into calls of at most call_tokens tokens (a call holds at
                // least one segment); the short ones to the recurrent kernel in one call
                for (int32_t kind = 1; kind >= 0; kind--) {
                    group.clear();
                    for (const int64_t* it = lo; it != hi; ++it)
                        if ((seg[*it].len > short_len) == (kind == 1)) group.push_back(*it);
                    if (group.empty()) continue;
                    int64_t total = 0;
                    for (int64_t g : group) total += seg[g].len;
                    size_t a = 0;
                    while (a < group.size()) {
                        size_t b = group.size();
                        if (kind == 1 && total > call_tokens) {
                            int64_t tokens = seg[group[a]].len;
                            b = a + 1;
                            while (b < group.size() && tokens + seg[group[b]].len <= call_tokens) tokens += seg[group[b++]].len;
                        }
                        emit(group.data() + a, group.data() + b, kind, d);
                        a = b;
                    }
                }
            } else {
                // levels path: the segments that keep their state first (their slots number them), then the others; below the
                // roots a call takes at most max_init segments (each starts from a copy of its parent's state)
                int64_t slots = 0;
                for (int pass = 0; pass < 2; pass++) {
                    group.clear();
                    for (const int64_t* it = lo; it != hi; ++it)
                        if (seg[*it].keeps == (pass == 0)) group.push_back(*it);
                    if (group.empty()) continue;
                    if (pass == 0)
                        for (int64_t g : group) p->seg_slot[g] = slots++;
                    const size_t step = d == 0 ? group.size() : (size_t)max_init;
                    for (size_t a = 0; a < group.size(); a += step) {
                        const size_t b = std::min(group.size(), a + step);
                        int64_t longest = 0;
                        for (size_t g = a; g < b; g++) longest = std::max(longest, seg[group[g]].len);
                        emit(group.data() + a, group.data() + b, longest > 64 ? 1 : 0, d);
                        p->call_keep.back() = pass == 0;
                    }
                }
                p->n_keep.push_back(slots);
            }
            p->level_ptr.push_back((int64_t)p->call_kind.size());
        }

        if (path == 0) build_program(p, seg, n_levels, by_level, at, short_len, row);

        // ---- convolution taps: the three tokens before a token on its path, oldest first, then the token itself
        const int64_t none = compact ? rows : n;
        p->conv_rows = compact ? rows : n;
        p->conv.assign((size_t)p->conv_rows * 4, none);
        for (int64_t i = 0; i < n; i++) {
            if (compact && !real[i]) continue;
            int64_t* tap = p->conv.data() + 4 * row(i);
            tap[3] = row(i);
            int64_t hop = real[i] ? prev[i] : -1;
            for (int back = 2; back >= 0 && hop >= 0; back--) {
                tap[back] = row(hop);
                hop = prev[hop];
            }
        }
        p->seg_of_row.assign((size_t)p->conv_rows, -1);
        for (int64_t i = 0; i < n; i++)
            if (real[i]) p->seg_of_row[row(i)] = seg_at[i];
    } catch (const std::exception&) {
        delete p;
        return spinf_fail(SPINF_E_NOMEM, "gdn_plan_build: out of memory");
    }
    *out = p;
    return SPINF_OK;
}

extern "C" int spinf_gdn_plan_counts(const spinf_gdn_plan* p, int64_t counts[6]) {
    if (!p || !counts) return spinf_fail(SPINF_E_ARG, "gdn_plan_counts: null argument");
    counts[0] = p->n_segments;
    counts[1] = (int64_t)p->level_ptr.size() - 1;
    counts[2] = (int64_t)p->call_kind.size();
    counts[3] = (int64_t)p->len.size();
    counts[4] = (int64_t)p->idx.size();
    counts[5] = p->conv_rows;
    return SPINF_OK;
}

extern "C" int spinf_gdn_plan_export(const spinf_gdn_plan* p, int64_t* level_ptr, int32_t* call_kind, int32_t* call_keep, int64_t* call_seg_ptr,
                                     int64_t* call_row_ptr, int64_t* seg_len, int64_t* h0_idx, int64_t* ht_idx, int64_t* idx, int64_t* n_keep,
                                     int64_t* conv, int64_t* seg_of_row, int64_t* seg_level, int64_t* seg_slot) {
    if (!p || !level_ptr || !call_seg_ptr || !call_row_ptr) return spinf_fail(SPINF_E_ARG, "gdn_plan_export: null argument");
    auto put = [](auto* dst, const auto& src) -> bool {
        if (src.empty()) return true;
        if (!dst) return false;
        std::memcpy(dst, src.data(), src.size() * sizeof(src[0]));
        return true;
    };
    const bool ok = put(level_ptr, p->level_ptr) && put(call_kind, p->call_kind) && put(call_keep, p->call_keep) && put(call_seg_ptr, p->call_seg_ptr) &&
                    put(call_row_ptr, p->call_row_ptr) && put(seg_len, p->len) && put(h0_idx, p->h0) && put(ht_idx, p->ht) && put(idx, p->idx) &&
                    put(n_keep, p->n_keep) && put(conv, p->conv) && put(seg_of_row, p->seg_of_row) && put(seg_level, p->seg_level) && put(seg_slot, p->seg_slot);
    if (!ok) return spinf_fail(SPINF_E_ARG, "gdn_plan_export: null array for a non-empty part of the plan");
    return SPINF_OK;
}

extern "C" int spinf_gdn_plan_program(const spinf_gdn_plan* p, int64_t counts[2], int64_t* launches, int64_t* data) {
    if (!p || !counts) return spinf_fail(SPINF_E_ARG, "gdn_plan_program: null argument");
    counts[0] = (int64_t)p->prog.size() / 8;
    counts[1] = (int64_t)p->prog_data.size();
    if (launches && !p->prog.empty()) std::memcpy(launches, p->prog.data(), p->prog.size() * 8);
    if (data && !p->prog_data.empty()) std::memcpy(data, p->prog_data.data(), p->prog_data.size() * 8);
    return SPINF_OK;
}

extern "C" void spinf_gdn_plan_free(spinf_gdn_plan* p) { delete p; }
