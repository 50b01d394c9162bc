// Tree-mask packed-prefill attention for gfx950, the ring kernel: the same arithmetic as tree_attn.hip's fast pass (same 32-key
// blocks in the same order, same softmax reference, same bits), with the waves of a workgroup decoupled.
//
// Replaces the flex_attention call of spinf_serve/models/gemma4.py:107-118 and spinf_serve/models/qwen35/qwen.py:614,620 for
// head dim 256 with an even number of query heads per key / value head (eight waves: four row groups x the two heads of an
// item) and for head dim 512 (four waves, one head per item, one wave per SIMD: the 32 x 512 outputs of a wave are all 256
// accumulation registers, which no kernel that leaves its accumulators to the compiler gets allocated; a ring of two slots).
//
// Why.  With a workgroup barrier at every key tile the eight waves move in lockstep: a wave whose 32 rows see nothing of a tile
// (the diagonal of a branch region) idles, all waves start their MFMA phases and their softmax phases together, and nothing
// overlaps the end of a work item (output rows, the next item's queries).  A free-running wave pair keeps a SIMD's matrix pipe
// busy by itself (measured: K Q^T, softmax and P V of a 32 x 32 block from LDS at the rate of the bare MFMAs), so here no wave
// ever waits for another one except through the tile ring:
//
//   * K / V tiles of 32 keys live in a ring of NSLOT slots.  Every wave walks the workgroup's tile sequence (all the tiles of
//     its work items, item after item) and skips the tiles its rows see nothing of.  When a wave is through with a tile it
//     counts itself in (`done`); once all have, whichever wave comes by first recycles the slot: it requests, by itself, the
//     DMA of the tile NSLOT places further on (`issued`); the last request of the batch writes the slot's flag, so the DMA engine itself
//     reports the tile as landed.  A wave needs the flag before it reads a tile and `issued` before it skips one, so the
//     waves stay within NSLOT - 1 tiles of each other.
//   * Work items are assigned to workgroups on the host (spinf_tileplan_schedule_static: a simulation of "the workgroup that
//     is free first takes the next item"), so the tile sequence of a workgroup is known to all its waves without any exchange
//     between workgroups; wave 0 expands it into a ring of tile descriptors in LDS, well ahead of everyone.
//   * A wave finishes an item on its own: its 32 output rows leave through a private LDS slice while the other waves compute,
//     and it requests its next queries right away.
//
// Every wait is a bounded spin on an LDS word; a wave that runs out of spins sets the workgroup's abort flag (and a counter the
// host can read), which makes every wave of the workgroup leave the ring at its next wait; the workgroup then computes its list
// again, one tile at a time between barriers (ring_paced_pass): the same bits, later.
#include <hip/hip_runtime.h>

#include "attn_acc.h"

namespace {

constexpr int NDESC = 128;          // tile descriptors kept in LDS
constexpr int GEN_AHEAD = 48;       // wave 0 keeps the descriptors this far ahead of its own tile
constexpr int SPIN_LIMIT = 1 << 18; // polls of one wait before the workgroup gives up (a healthy wait takes a handful)
constexpr unsigned DESC_FIRST = 1u << 16, DESC_LAST = 1u << 17;

template <int D, bool WIN>
__global__ __launch_bounds__(D == 512 ? 256 : 512) void tree_attn_ring_kernel(const AttnParams p) {
    constexpr int TK = RingShape<D>::TK, NSUB = RingShape<D>::NSUB;
    constexpr int NW = D == 512 ? 4 : 8;      // waves: four row groups x HPI heads of the item
    constexpr int HPI = NW / 4;
    constexpr int NSLOT = D == 512 ? 2 : MAX_SLOT;
    using G = TileGeo<D, TK, D>;
    constexpr int NS = D / 16;     // contraction steps of K Q^T
    constexpr int NDT = D / 32;    // 32-wide slices of the head dimension in O^T
    constexpr int NVF = 2 * NDT;   // V^T fragments of one 32-key block
    constexpr int PFD = D >= 256 ? 2 : 8;   // fragment read-ahead: at head dim 256 one more spills a query fragment inside the tile loop
    constexpr int PF = D >= 256 ? 4 : (NS < PFD ? NS : PFD);   // K fragments are live in the score phase only, where registers are free
    constexpr int VPF = NVF < PFD ? NVF : PFD;
    constexpr int DONE_AT = NVF - 1 - VPF > 0 ? NVF - 1 - VPF : 0;   // the P V step behind which a block's last V fragment read is on its way
    static_assert(NSLOT * G::BUFB + NW * 32 * SROW + NDESC * 16 + 256 <= 160 * 1024, "LDS budget");
    __shared__ __attribute__((aligned(16))) char ring[NSLOT * G::BUFB];
    __shared__ __attribute__((aligned(16))) char stage_all[NW * 32 * SROW];   // output staging, one slice per wave
    __shared__ int4 desc[NDESC];       // {key tile, bits | DESC_FIRST | DESC_LAST, query tile | head group << 20, item index}
    __shared__ __attribute__((aligned(16))) int sy_done[MAX_SLOT];   // waves through with the tile in the slot; NW = the slot waits for somebody to recycle it (words past NSLOT stay 0)
    __shared__ int sy_issued[MAX_SLOT];   // tile the slot was last recycled for (its DMA requested)
    __shared__ int sy_gen;             // descriptors written so far
    __shared__ int sy_abort;
    __shared__ int sy_gave_up;         // waves that gave up a wait
    __shared__ int sy_ntiles;
    __shared__ int sy_redo[16];        // item sequence number + 1 of the last hand-over to the exact recomputation, per sequence number mod 16
    __shared__ int sy_nredo;           // items of this workgroup handed over so far (their indices: p.redo[lo ..])

    const Lane<D, TK, D> L(p);
    const int lo = p.list_ptr[blockIdx.x], hi = p.list_ptr[blockIdx.x + 1];

    // ---- waits: bounded spins on an LDS word
    bool dead = false;   // wave-uniform
    // The spin itself is one block of assembly: a loop in the source here, inside the tile loop, makes the register allocator
    // spill the queries around it.  Leaves with 0 when the word has the wanted value (>= it with at_least), with 1 (if `watch`)
    // when all eight waves are through with some slot's tile and somebody has to recycle it, with 2 when the workgroup's abort flag is up or after SPIN_LIMIT polls.
    auto spin = [&](const int* word, const int want, const bool at_least, const bool watch) __attribute__((always_inline)) {
        const unsigned a_word = lds_addr(word), a_abort = lds_addr(&sy_abort), a_next = lds_addr(sy_done);
        int t0, t1, n0, n1, n2, n3, v, ab, code, cnt = p.spin_limit;
#define SPIN_ASM(CMP, WATCH)                                                                                                                         \
    asm volatile("1:\n\tds_read_b32 %0, %10\n\tds_read_b32 %1, %11\n\tds_read_b32 %2, %12\n\tds_read_b32 %3, %12 offset:4\n\t"                     \
                 "ds_read_b32 %4, %12 offset:8\n\tds_read_b32 %5, %12 offset:12\n\ts_waitcnt lgkmcnt(0)\n\t"                                        \
                 "v_readfirstlane_b32 %6, %0\n\tv_readfirstlane_b32 %7, %1\n\ts_mov_b32 %8, 0\n\t" CMP " %6, %13\n\ts_cbranch_scc1 2f\n\t"      \
                 "s_mov_b32 %8, 2\n\ts_cmp_lg_u32 %7, 0\n\ts_cbranch_scc1 2f\n\ts_sub_u32 %9, %9, 1\n\ts_cmp_eq_u32 %9, 0\n\ts_cbranch_scc1 2f\n\t" \
                 WATCH "s_sleep 1\n\ts_branch 1b\n2:"                                                                                               \
                 : "=&v"(t0), "=&v"(t1), "=&v"(n0), "=&v"(n1), "=&v"(n2), "=&v"(n3), "=&s"(v), "=&s"(ab), "=&s"(code), "+s"(cnt)                     \
                 : "v"(a_word), "v"(a_abort), "v"(a_next), "s"(want), "n"(NW)                                                                       \
                 : "memory", "scc", "vcc")
#define SPIN_WATCH "s_mov_b32 %8, 1\n\tv_cmp_eq_u32_e32 vcc, %c14, %2\n\ts_cbranch_vccnz 2f\n\tv_cmp_eq_u32_e32 vcc, %c14, %3\n\ts_cbranch_vccnz 2f\n\tv_cmp_eq_u32_e32 vcc, %c14, %4\n\ts_cbranch_vccnz 2f\n\tv_cmp_eq_u32_e32 vcc, %c14, %5\n\ts_cbranch_vccnz 2f\n\t"
        if (at_least) {
            if (watch) SPIN_ASM("s_cmp_ge_i32", SPIN_WATCH); else SPIN_ASM("s_cmp_ge_i32", "");
        } else {
            if (watch) SPIN_ASM("s_cmp_eq_u32", SPIN_WATCH); else SPIN_ASM("s_cmp_eq_u32", "");
        }
#undef SPIN_ASM
#undef SPIN_WATCH
        if (code == 2) {
            lds_store(&sy_abort, 1);
            dead = true;
        }
        return make_int2(code, v);
    };
    // wait for the descriptors (wave 0 writes them far ahead: a wait here is the exception)
    auto wait_gen = [&](const int want) __attribute__((always_inline)) {
        const int v = __builtin_amdgcn_readfirstlane(lds_load(&sy_gen));
        if (v >= want) return v;
        return spin(&sy_gen, want, true, false).y;
    };

    // ---- prologue: sync words, the workgroup's tile count, the first descriptors
    if (threadIdx.x < MAX_SLOT) {
        sy_done[threadIdx.x] = 0;
        sy_issued[threadIdx.x] = (int)threadIdx.x;
        if (threadIdx.x < NSLOT) *(int*)(ring + threadIdx.x * G::BUFB + G::KTILEB + G::VTILEB + 768) = -1;   // the slot's flag: no generation yet
    }
    if (threadIdx.x < 16) sy_redo[threadIdx.x] = 0;
    if (threadIdx.x == 0) { sy_gen = 0; sy_abort = 0; sy_gave_up = 0; sy_ntiles = 0; sy_nredo = 0; }
    __syncthreads();

    // descriptor generator (wave 0): items lo .. hi - 1, each item's plan entries in chunks of at most 64
    int gi = lo, ge = 0, gen = 0;   // next chunk: item, first entry inside it; descriptors written
    int pn = 0, p_first = 0, p_last = 0, p_tz = 0, p_item = 0;   // the requested chunk
    int pidx = 0, pbits = 0;
    auto gen_request = [&]() __attribute__((always_inline)) {   // loads of the next chunk's entries
        if (pn == 0 && gi < hi) {
            const int4 it = p.items[gi];
            const int t = __builtin_amdgcn_readfirstlane(it.x), e0 = __builtin_amdgcn_readfirstlane(it.y), z = __builtin_amdgcn_readfirstlane(it.z);
            const int ne = z & 0xfffff;
            const int n = ne - ge < 64 ? ne - ge : 64;
            const int gl = fresh_lane_id();
            if (gl < n) {
                pidx = p.kv_idx[e0 + ge + gl];
                pbits = (int)p.kv_bits[e0 + ge + gl];
            }
            pn = n;
            p_first = ge == 0;
            p_last = ge + n == ne;
            p_tz = t | (int)((unsigned)z >> 20 << 20);
            p_item = gi;
            ge += n;
            if (ge >= ne) { gi++; ge = 0; }
        }
    };
    auto gen_write = [&]() __attribute__((always_inline)) {   // descriptors of the requested chunk
        if (pn > 0) {
            const int gl = fresh_lane_id();
            if (gl < pn) {
                unsigned b = (unsigned)pbits & 0xffffu;
                if (p_first && gl == 0) b |= DESC_FIRST;
                if (p_last && gl == pn - 1) b |= DESC_LAST;
                desc[(gen + gl) & (NDESC - 1)] = make_int4(pidx, (int)b, p_tz, p_item);
            }
            gen += pn;
            pn = 0;
            lds_store(&sy_gen, gen);
        }
    };
    if (L.w == 0) {
        int nt = 0;
        for (int i = lo + L.lane; i < hi; i += 64) nt += p.items[i].z & 0xfffff;
        for (int off = 32; off > 0; off >>= 1) nt += __shfl_xor(nt, off);
        nt = __builtin_amdgcn_readfirstlane(nt);
        if (L.lane == 0) sy_ntiles = nt;
        while (gen < GEN_AHEAD && (gi < hi || pn > 0)) {
            gen_request();
            gen_write();
        }
        gen_request();
    }
    __syncthreads();
    const int ntiles = __builtin_amdgcn_readfirstlane(sy_ntiles);
    if (ntiles == 0) return;
    int gen_seen = __builtin_amdgcn_readfirstlane(lds_load(&sy_gen));

    auto read_desc = [&](const int j) __attribute__((always_inline)) {   // j < gen_seen
        const int4 d = desc[j & (NDESC - 1)];
        return make_int4(__builtin_amdgcn_readfirstlane(d.x), __builtin_amdgcn_readfirstlane(d.y), __builtin_amdgcn_readfirstlane(d.z),
                         __builtin_amdgcn_readfirstlane(d.w));
    };
    auto need_desc = [&](const int j) __attribute__((always_inline)) {
        if (j >= gen_seen) gen_seen = wait_gen(j + 1);
    };
    auto issue = [&](const int j, const int4& d) __attribute__((always_inline)) {
        const int kvh = (int)((unsigned)d.z >> 20) * HPI / p.group;
        // the per-lane parts of the source addresses are recomputed here: kept in registers they are spilled across the tile loop
        using GK = Geo<D, TK>;
        const int lane = fresh_lane_id();
        const unsigned lane_k = (unsigned)((lane / GK::CPR) * GK::NREG * p.k_tok * 2 + (lane % GK::CPR) * 16);
        const unsigned lane_v = (unsigned)((lane / GK::CPR) * GK::NREG * p.v_tok * 2 + (lane % GK::CPR) * 16);
        issue_tile_wave<D, WIN, TK>(p, lds_addr(ring + (j & (NSLOT - 1)) * G::BUFB), d.x, kvh, j / NSLOT + 1, lane, lane_k, lane_v);
    };

    // When all eight waves are through with a slot's tile (its count stands at 8), whichever wave comes by first recycles the slot:
    // it takes the count back to 0 (compare-and-swap: one winner) and requests the tile NSLOT places further on.  Not the last
    // wave through by design: that one is the wave the others are waiting for.  n0..n3 = sy_done as read a moment ago.
    auto claim = [&](const int n0, const int n1, const int n2, const int n3) __attribute__((always_inline)) {
        if (n0 == NW || n1 == NW || n2 == NW || n3 == NW) {
            const int sl = n0 == NW ? 0 : n1 == NW ? 1 : n2 == NW ? 2 : 3;
            int got = 0;
            if (fresh_lane_id() == 0) {
                int expect = NW;
                got = __hip_atomic_compare_exchange_strong(&sy_done[sl], &expect, 0, __ATOMIC_ACQ_REL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            if (__builtin_amdgcn_readfirstlane(got)) {
                const int jn = __builtin_amdgcn_readfirstlane(lds_peek(&sy_issued[sl])) + NSLOT;   // only a winner writes this word
                if (jn < ntiles) {
                    need_desc(jn);
                    if (!dead) {
                        lds_store(&sy_issued[sl], jn);
                        issue(jn, read_desc(jn));
                    }
                }
            }
        }
    };
    auto try_issue = [&]() __attribute__((always_inline)) {
        const i32x4 nx = lds_peek4(sy_done);
        claim(__builtin_amdgcn_readfirstlane(nx[0]), __builtin_amdgcn_readfirstlane(nx[1]), __builtin_amdgcn_readfirstlane(nx[2]), __builtin_amdgcn_readfirstlane(nx[3]));
    };
    // wait for a slot's flag or recycling, lending a hand meanwhile: a round of the spin ends when the word is there, or with a
    // tile to request (then request it and go back to waiting)
    auto wait_watch = [&](const int* word, const int want) __attribute__((always_inline)) {
        if (__builtin_amdgcn_readfirstlane(lds_load(word)) == want) return;
#pragma unroll
        for (int round = 0; round < NSLOT + 2; round++) {
            const int code = spin(word, want, false, round < NSLOT + 1).x;
            if (code != 1) break;
            try_issue();
        }
    };

    // the first NSLOT tiles: one wave each
    if (L.w < NSLOT && L.w < ntiles) issue(L.w, read_desc(L.w));

    // ---- per-item state of this wave
    bf16x8 qf[NS];
    int art_q = -1, pos_q = 0;
    float M = -INFINITY, l = 0.f;
    bool viol = false;
    int iseq = 0;   // items begun

    auto load_q = [&](const int tz) __attribute__((always_inline)) {
        const int lane = fresh_lane_id();
        const int tok = (tz & 0xfffff) * SPINF_QTILE + 32 * L.wr + (lane & 31);
        const int tok_c = tok < p.n ? tok : p.n - 1;
        const int h = (int)((unsigned)tz >> 20) * HPI + L.wh;
        const __bf16* qp = p.q + (long)tok_c * p.q_tok + (long)h * p.q_head + 8 * (lane >> 5);
#pragma unroll
        for (int s = 0; s < NS; s++) qf[s] = *(const bf16x8*)(qp + 16 * s);
        art_q = tok < p.n ? p.art[tok_c] : -1;
        pos_q = WIN ? p.pos[tok_c] : 0;
    };
    auto reset_acc = [&]() __attribute__((always_inline)) {
        M = -INFINITY;
        l = 0.f;
        acc_zero<NDT>();
        viol = false;
    };
    // normalise O^T and store it as rows: 32 rows x 32 head dims at a time through the wave's own LDS slice, 16-byte pieces out
    // (pieces of 8 bytes straight from the registers were measured slower: twice the requests for the same bytes)
    auto store_rows = [&](const int tz) __attribute__((always_inline)) {
        const int lane = fresh_lane_id(), m = lane & 31, g = lane >> 5;
        const int tok0 = (tz & 0xfffff) * SPINF_QTILE + 32 * L.wr;
        const int h = (int)((unsigned)tz >> 20) * HPI + L.wh;
        const float inv = 1.0f / lane32_sum(l);
        __bf16* ob = p.o + (long)h * p.o_head;
        char* const stage = stage_all + L.w * 32 * SROW;
        asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");   // the last MFMAs' results -> v_accvgpr_read
        // tile dt is read back from the slice while tile dt + 1 is converted and written to it (the LDS takes a wave's requests
        // in order, so the write behind the read is safe), and stored after that: no wait between a write and its read-back
        auto put = [&](auto dt_c) __attribute__((always_inline)) {
            constexpr int dt = decltype(dt_c)::value;
            float r16[16];
            acc_read<dt>(r16);
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++) {
                bf16x4 r;
#pragma unroll
                for (int jj = 0; jj < 4; jj++) r[jj] = (__bf16)(r16[4 * i4 + jj] * inv);
                *(bf16x4*)(stage + m * SROW + (8 * i4 + 4 * g) * 2) = r;
            }
        };
        auto round = [&](auto dt_c) __attribute__((always_inline)) {
            constexpr int dt = decltype(dt_c)::value;
            bf16x8 val[2];
#pragma unroll
            for (int jj = 0; jj < 2; jj++) {
                const int c = jj * 64 + lane;
                val[jj] = *(const bf16x8*)(stage + (c >> 2) * SROW + (c & 3) * 16);
            }
            if constexpr (dt + 1 < NDT) put(std::integral_constant<int, dt + 1>{});
#pragma unroll
            for (int jj = 0; jj < 2; jj++) {
                const int c = jj * 64 + lane, row = c >> 2, col = c & 3;
                if (tok0 + row < p.n) *(bf16x8*)(ob + (long)(tok0 + row) * p.o_tok + 32 * dt + col * 8) = val[jj];
            }
        };
        put(std::integral_constant<int, 0>{});
        pv_steps<NDT>(round);
    };

    {   // the first item's queries
        need_desc(0);
        if (!dead) load_q(read_desc(0).z);
    }

    // ---- the tile sequence: item after item.
    // What a wave needs to know at the top of a tile (the tile's descriptor, the slots waiting for requests, the tile's flag) is
    // read from LDS while the previous tile's last MFMAs run (`pf_*`), and the wave counts itself through with a tile as soon as
    // its last fragment read of the tile is on its way: in the steady state no LDS round trip is waited for.
    int j = 0;
    bool have_pf = false;
    int4 pf_d = make_int4(0, 0, 0, 0);
    int pf_n0 = 0, pf_n1 = 0, pf_n2 = 0, pf_n3 = 0, pf_flag = -1;
    auto flag_word = [&](const int jj) __attribute__((always_inline)) { return (const int*)(ring + (jj & (NSLOT - 1)) * G::BUFB + G::KTILEB + G::VTILEB + 768); };
    while (j < ntiles && !dead) {
        reset_acc();
        iseq++;
        int4 d = make_int4(0, 0, 0, 0);
        bool last = false;
        do {
            const int s = j & (NSLOT - 1);
            int n0, n1, n2, n3, flag;
            if (have_pf) {
                d = pf_d; n0 = pf_n0; n1 = pf_n1; n2 = pf_n2; n3 = pf_n3; flag = pf_flag;
            } else {
                need_desc(j);
                if (dead) break;
                const int4 dv = desc[j & (NDESC - 1)];
                const i32x4 nx = lds_peek4(sy_done);
                const int fv = lds_peek(flag_word(j));
                d = make_int4(__builtin_amdgcn_readfirstlane(dv.x), __builtin_amdgcn_readfirstlane(dv.y), __builtin_amdgcn_readfirstlane(dv.z), __builtin_amdgcn_readfirstlane(dv.w));
                n0 = __builtin_amdgcn_readfirstlane(nx[0]); n1 = __builtin_amdgcn_readfirstlane(nx[1]);
                n2 = __builtin_amdgcn_readfirstlane(nx[2]); n3 = __builtin_amdgcn_readfirstlane(nx[3]);
                flag = __builtin_amdgcn_readfirstlane(fv);
            }
            have_pf = false;
            // The waves of the second head set run behind those of the first (a SIMD's arbiter favours its older wave), and the
            // kernel ends when they do: they leave the recycling to the first set, which is ahead and mostly waiting for
            // flags anyway, and lend a hand only from inside a wait.
            if (L.w < 4) claim(n0, n1, n2, n3);
            if (dead) break;
            const unsigned bits = (unsigned)d.y;
            last = (bits & DESC_LAST) != 0;
            // the tile's 32-key blocks that this wave's rows see something of (one bit per block)
            const unsigned ab = (bits >> (2 * L.wr)) & (NSUB == 2 ? 3u : 1u);
            const bool act = ab != 0;
            if (act) {
                if (flag != ((j / NSLOT + 1) & 63)) wait_watch(flag_word(j), (j / NSLOT + 1) & 63);
                if (dead) break;
                // fragment addresses from a fresh lane index (kept in registers across the tile loop they are spilled, and a reload
                // waits for every tile request in flight): K row lane % 32 of the block, 16-byte chunk lane / 32 of each 32-byte step;
                // V^T as ds_read_b64_tr_b16 wants it (see Lane in attn_kernels.h)
                const int ln = fresh_lane_id();
                const char* buf = ring + s * G::BUFB;
                // what the next tile's top needs, fetched under the last block's P V products
                int4 dv = make_int4(0, 0, 0, 0);
                i32x4 nx = {0, 0, 0, 0};
                int fv = -1;
                const bool pf_ok = j + 1 < ntiles && j + 1 < gen_seen;
                // one 32-key block: K Q^T, mask, softmax, P V.  TAIL: the last block of the tile that this wave computes
                auto block = [&](const int sub, auto tail_c) __attribute__((always_inline)) {
                    constexpr bool TAIL = decltype(tail_c)::value;
                    const char* krow = buf + G::K::k_off(ln & 31) + 16 * (ln >> 5) + sub * G::KSUB;
                    const char* vrow = buf + G::KTILEB + G::V::v_off(4 * (ln >> 5) + ((ln >> 2) & 3)) + 32 * ((ln >> 4) & 1) + 8 * (ln & 3) + sub * G::VSUB;
                    // S^T = K Q^T
                    f32x16 sa;
                    {
                        bf16x8 kf[PF];
#pragma unroll
                        for (int x = 0; x < PF; x++) kf[x] = *(const bf16x8*)(krow + 32 * x);
                        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                        for (int x = 0; x < NS; x++) {
                            if (x == 0) qk_first(sa, kf[x % PF], qf[x]);
                            else if (x == NS - 1) qk_last(sa, kf[x % PF], qf[x]);
                            else qk_next(sa, kf[x % PF], qf[x]);
                            if (x + PF < NS) kf[x % PF] = *(const bf16x8*)(krow + 32 * (x + PF));
                            __builtin_amdgcn_sched_barrier(0);
                        }
                    }
                    if ((bits >> (8 + 2 * L.wr + sub)) & 1u) {
                        f32x16 sm[1] = {sa};
                        const int tok = (d.z & 0xfffff) * SPINF_QTILE + 32 * L.wr + (ln & 31);
                        apply_mask<1, WIN, 0, TK>(sm, (const int*)(buf + G::KTILEB + G::VTILEB), d.x, sub, ln >> 5, tok, art_q, pos_q, p.window);
                        sa = sm[0];
                    }
                    // softmax against the row's fixed reference (the maximum of the first block it sees a key in)
                    bf16x8 pb[2];
                    {
                        const bool first = M == -INFINITY;
                        if (__builtin_amdgcn_ballot_w64(first) != 0) {   // only where a row meets its first keys (see the lockstep kernel)
                            float mx = sa[0];
#pragma unroll
                            for (int i2 = 1; i2 < 16; i2++) mx = fmaxf(mx, sa[i2]);
                            mx = lane32_max(mx);
                            M = first ? mx * p.c : M;
                        }
                        const float ms = M == -INFINITY ? 0.f : M;
                        float sum = 0.f;
#pragma unroll
                        for (int i2 = 0; i2 < 16; i2++) {
                            const float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(sa[i2], p.c, -ms));
                            sum += pr;
                            pb[i2 >> 3][i2 & 7] = (__bf16)pr;
                        }
                        l += sum;
                        viol = viol | !(sum <= VIOL_SUM);
                    }
                    // O^T += V^T P^T, with what the next tile's top needs fetched meanwhile; once the last fragment read is on its way,
                    // count this wave through with the tile
                    // (requested before the first transposing read of V, so that every wait inside the MFMA sequence is for V
                    // fragments alone and stalls: a wait that is already satisfied takes no time, and then a vector write of an
                    // operand could end up in the issue cycle before the assembly MFMA that reads it; LDS reads of different kinds
                    // do return in issue order, spinf_diag_lds_order checks it)
                    if (TAIL && pf_ok) {
                        dv = desc[(j + 1) & (NDESC - 1)];
                        nx = lds_peek4(sy_done);
                        fv = lds_peek(flag_word(j + 1));
                    }
                    {
                        s16x4 vlo[VPF], vhi[VPF];
                        auto vload = [&](const int f, const int slot) __attribute__((always_inline)) {
                            const char* vp = vrow + G::V::v_off(16 * (f / NDT)) + 64 * (f % NDT);
                            vlo[slot] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)vp);
                            vhi[slot] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vp + G::V::v_off(8)));
                        };
#pragma unroll
                        for (int f = 0; f < VPF; f++) vload(f, f);
                        __builtin_amdgcn_sched_barrier(0);
                        // (head dim 128 reads all of a block's V fragments ahead, and the compiler then sinks the conversions that write
                        // the P fragments below those reads, right in front of the first MFMA, which would multiply the registers' old
                        // contents: one instruction in between)
                        if constexpr (VPF >= NVF) asm volatile("s_nop 0" ::: "memory");
                        auto step = [&](auto f_c) __attribute__((always_inline)) {
                            constexpr int f = decltype(f_c)::value;
                            const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(vlo[f % VPF], vhi[f % VPF], 0, 1, 2, 3, 4, 5, 6, 7));
                            acc_mfma<f % NDT>(a, pb[f / NDT]);
                            if (f + VPF < NVF) vload(f + VPF, f % VPF);
                            if (TAIL && f == DONE_AT) {   // that was the tile's last fragment read
                                if (fresh_lane_id() == 0) __hip_atomic_fetch_add(&sy_done[s], 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                            }
                            __builtin_amdgcn_sched_barrier(0);
                        };
                        pv_steps<NVF>(step);
                    }
                };
                if constexpr (NSUB == 1) {
                    block(0, std::true_type{});
                } else {
                    if (ab == 3u) {
                        block(0, std::false_type{});
                        block(1, std::true_type{});
                    } else {
                        block((int)(ab >> 1), std::true_type{});
                    }
                }
                if (pf_ok) {
                    pf_d = make_int4(__builtin_amdgcn_readfirstlane(dv.x), __builtin_amdgcn_readfirstlane(dv.y), __builtin_amdgcn_readfirstlane(dv.z), __builtin_amdgcn_readfirstlane(dv.w));
                    pf_n0 = __builtin_amdgcn_readfirstlane(nx[0]); pf_n1 = __builtin_amdgcn_readfirstlane(nx[1]);
                    pf_n2 = __builtin_amdgcn_readfirstlane(nx[2]); pf_n3 = __builtin_amdgcn_readfirstlane(nx[3]);
                    pf_flag = __builtin_amdgcn_readfirstlane(fv);
                    have_pf = true;
                }
            } else {
                // nothing of this tile for these rows: the slot must have been recycled for it before this wave counts itself through
                wait_watch(&sy_issued[s], j);
                if (dead) break;
                if (fresh_lane_id() == 0) __hip_atomic_fetch_add(&sy_done[s], 1, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            // wave 0 keeps the descriptors ahead
            if (L.w == 0 && gen - j < GEN_AHEAD) {
                gen_write();
                gen_request();
            }
            j++;
        } while (!last);
        if (dead) break;
        // this wave's rows of the item are complete: the next item's queries are requested (their registers are free), then the rows
        // go out (or the item goes to the exact pass)
        const bool hand_over = __builtin_amdgcn_ballot_w64(viol) != 0;   // scores ranged too widely somewhere in these 32 rows
        const int tz_done = d.z, item_done = d.w;
        if (j < ntiles) {
            need_desc(j);
            if (dead) break;
            load_q(read_desc(j).z);
        }
        if (hand_over) {
            if (fresh_lane_id() == 0) {
                const int was = __hip_atomic_fetch_max(&sy_redo[iseq & 15], iseq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (was < iseq) {   // first wave of the item to say so: the workgroup recomputes the item after its list (below)
                    const int k = __hip_atomic_fetch_add(&sy_nredo, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_store(&p.redo[lo + k], item_done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
        } else {
            store_rows(tz_done);
        }
    }
    if (dead && fresh_lane_id() == 0) __hip_atomic_fetch_add(&sy_gave_up, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);   // (the list is done again below)
    __builtin_amdgcn_s_waitcnt(0x0f70);

    // ---- after the list: normally nothing.  Items in which some row met scores too far above its reference are done again, exactly,
    // by ring_paced_pass; and if some wave gave up a wait (every wave has then left the ring), so is the whole list, with the ring
    // pass's own arithmetic: an abort costs time, never rows.
    __syncthreads();   // every wave is through with its list: the ring is free, the hand-overs are all in
    const bool gave_up = __builtin_amdgcn_readfirstlane(lds_load(&sy_abort)) != 0;
    if (!gave_up && __builtin_amdgcn_readfirstlane(lds_load(&sy_nredo)) == 0) return;
    __shared__ int sy_vote;
    if (gave_up) {   // some wave gave up a wait: the whole list again, one tile at a time between barriers (same bits)
        if (threadIdx.x == 0) {
            sy_nredo = 0;   // (whatever the list needs recomputed exactly is found again on the way)
            atomicAdd(&p.counters[NLIST + 4], lds_load(&sy_gave_up));   // running total, for spinf_attn_ring_aborts
        }
    }
    if (threadIdx.x == 0) sy_vote = 0;
    __syncthreads();
    ring_paced_pass<D, WIN>(p, ring, stage_all, &sy_nredo, &sy_vote, lo, gave_up ? hi : lo, lo);
}

template <int D, bool WIN>
int launch_ring_t(const AttnParams& p, int n_wg, hipStream_t stream) {
    hipLaunchKernelGGL((tree_attn_ring_kernel<D, WIN>), dim3(n_wg), dim3(D == 512 ? 256 : 512), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return spinf_fail(SPINF_E_HIP, "tree_attn: launch (ring kernel): %s", hipGetErrorString(e));
    return SPINF_OK;
}

}  // namespace

int spinf_launch_ring(const AttnParams& p, int d, bool win, int n_wg, hipStream_t stream) {
    if (d == 128) return win ? launch_ring_t<128, true>(p, n_wg, stream) : launch_ring_t<128, false>(p, n_wg, stream);
    if (d == 256) return win ? launch_ring_t<256, true>(p, n_wg, stream) : launch_ring_t<256, false>(p, n_wg, stream);
    if (d == 512) return win ? launch_ring_t<512, true>(p, n_wg, stream) : launch_ring_t<512, false>(p, n_wg, stream);
    return spinf_fail(SPINF_E_ARG, "tree_attn: the ring kernel takes head dim 128, 256 or 512, not %d", d);
}
