// Tree-mask packed-prefill attention for gfx950, the pipelined kernel: one wave per SIMD, and the softmax of a key block beside the
// P V products of the block before.
//
// Replaces the flex_attention call of spinf_serve/models/gemma4.py:107-118 for head dim 512 on global layers with plenty of work items
// (attention.py, _pipelined, has the line).  Same work items, schedule, arithmetic and bits as the ring kernel (tree_attn_ring.hip): four
// waves of 32 query rows, O^T in the 256 accumulation registers, 32-key tiles, one head per item.
//
// Why.  At 512 accumulators and queries a lane there is one wave per SIMD, and the ring kernel leaves that wave alone with everything:
// while it does its softmax, asks for a whole tile (67 requests in a row) or polls a flag, the matrix core stands.
// But a wave's own vector instructions do run under its own products: one product of 32 x 32 x 16 takes 32 clocks of the matrix core,
// and 4 - 6 fused multiply-adds, 2 exponentials or 2 sixteen-byte LDS reads issued behind it cost next to nothing (32.8 - 35.6, 32.8 and 32.6
// clocks per product measured, 8 multiply-adds 44: mfma_valu_kernel and lds_rate_kernel in diag.hip).  So the work of a tile is laid out by
// hand as two phases of 32 products, each product with a piece of the other work behind it (scheduling barriers keep the pieces in place).
//   A(j)  the scores of tile j, K Q^T; V of tile j is requested, and what B(j) requests is worked out
//   B(j)  P V of tile j - 1, with mask, softmax and packing of tile j's scores beside it; K and the keys' metadata of tile j + 2 are requested,
//         tile j + 3 is looked up
//   C     at an item's end: P V of its last tile; the next item's queries are on their way, and arrive under the output rows
// The requests are dealt out, a quarter of every tile to each wave, one behind every fourth product.  A wave counts on its own requests only
// (s_waitcnt vmcnt with the number of requests made since), and a barrier at each phase's end makes the four quarters everybody's:
// three phases lie between a request and its use, two tiles of K and V fill the LDS.  No flags, no polls; every wave passes the same barriers.
//
// Little but products and their beside-work may stand in a phase: a scalar branch between two products costs ~30 clocks (requests handed out
// by a branch per product: 2.79 ms against 2.12 on 65,536 tokens), and bookkeeping ahead of a phase's first product is not under anything.
// One branch is left, around the row's reference in B: its 16 maxima and lane exchange are wanted once per row, not once per tile.
//
// Measured, the ring kernel in turns with it: 24 contents of 470 tokens with 56 questions (28,672 tokens, 16 / 1 heads, 14 items a workgroup)
// 556 - 561 us against 609 - 611; 46 contents with trunks around 800 (64,896 tokens, 32 items a workgroup) 2.02 ms against 2.19.  A tile
// takes 5.0 k clocks of 2.05 k products: A 1.5, B 2.8, waits for the other waves 0.7 (a build with clock stamps).  What bounds it now: the
// issue of everything that stands behind the products of one wave; the matrix cores are busy 29 % of the time, 28,672 tokens move
// 1.33 GB.  Timing-only builds on the longer stream: without exponentials 1.98 ms; an earlier form of this kernel 2.03 - 2.14, without
// requests 1.72, without V's reads from LDS as well 1.70.
#include <hip/hip_runtime.h>

#include "attn_acc.h"

namespace {

constexpr int NCHUNK = 8;    // chunks of plan entries in LDS
constexpr int CHUNK = 64;    // entries of a chunk at most (one item's)
constexpr int NITEMS = 128;  // work items in LDS
constexpr unsigned TILE_LAST = 1u << 16;

struct Tile {   // (wave-uniform)
    int kt;
    unsigned bits;   // the plan entry's block bits | TILE_LAST of its item | key / value head << 17
    int tz;          // query tile | head group << 20
};

// all but the last N requests of this wave have landed, LDS is settled, everyone is here
template <int N>
__device__ __forceinline__ void step_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

template <int D>
__global__ __launch_bounds__(256) void tree_attn_pipe_kernel(const AttnParams p) {
    using G = TileGeo<D, 32, D>;
    using GK = typename G::K;
    constexpr int NS = D / 16, NDT = D / 32, NVF = 2 * NDT;
    constexpr int VPF = 8;                  // V fragments read ahead
    constexpr int NREQ = GK::NREG / 4;      // requests of a wave per K (or V) tile
    static_assert(GK::RPI == 1 && NREQ * 4 == NS && NS == NVF && NS >= 32, "a request is a row; one request per four products");
    constexpr int SLOTB = G::KTILEB + G::VTILEB, METAB = 4 * 256;
    static_assert(2 * SLOTB >= G::BUFB, "the barrier-paced pass lays a tile and its metadata out in a row");
    __shared__ __attribute__((aligned(16))) char ring[2 * SLOTB];           // K and V of two tiles
    __shared__ __attribute__((aligned(16))) char meta_all[4 * METAB];       // art, end of four tiles' keys
    __shared__ __attribute__((aligned(16))) char stage_all[4 * 32 * SROW];  // output staging, one slice per wave
    __shared__ int c_idx[NCHUNK][CHUNK], c_bits[NCHUNK][CHUNK];
    __shared__ __attribute__((aligned(16))) int c_head[NCHUNK][4];          // {entries | the item's last chunk << 8, query tile | head group << 20, key / value head << 17}
    __shared__ __attribute__((aligned(16))) int items[NITEMS][4];
    __shared__ int sy_ntiles, sy_nredo, sy_vote;
    __shared__ int sy_redo[16];

    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int lo = __builtin_amdgcn_readfirstlane(p.list_ptr[blockIdx.x]), hi = __builtin_amdgcn_readfirstlane(p.list_ptr[blockIdx.x + 1]);
    const int cnt = hi - lo;
    if (cnt <= 0) return;

    // ---- the workgroup's tiles: wave 0 copies its list's items and their plan entries into LDS, a few chunks ahead of the tiles
    int gi = 0, ge = 0, pc = 0;             // next item, entry inside it; chunks copied
    int it_e0 = 0, it_ne = 0, it_tz = 0, it_kvh = 0;
    auto copy_items = [&](const int from) __attribute__((always_inline)) {
        const int lane = fresh_lane_id();
        const int at = from + lane < cnt ? from + lane : cnt - 1;
        dma16_lane((const char*)(p.items + lo + at), lds_addr(&items[from & (NITEMS - 1)][0]));
    };
    auto produce = [&]() __attribute__((always_inline)) {   // the next chunk (an item has at least one entry: its rows see themselves)
        if (ge == 0) {
            const i32x4 it = lds_peek4(&items[gi & (NITEMS - 1)][0]);
            const int z = __builtin_amdgcn_readfirstlane(it[2]);
            it_e0 = __builtin_amdgcn_readfirstlane(it[1]);
            it_ne = z & 0xfffff;
            it_tz = __builtin_amdgcn_readfirstlane(it[0]) | (int)((unsigned)z >> 20 << 20);
            it_kvh = __builtin_amdgcn_readfirstlane((int)((unsigned)z >> 20) / p.group);
        }
        const int lane = fresh_lane_id();
        const int n = it_ne - ge < CHUNK ? it_ne - ge : CHUNK;
        const int e = it_e0 + ge + (lane < n ? lane : n - 1), s = pc & (NCHUNK - 1);
        dma4_lane(p.kv_idx + e, lds_addr(&c_idx[s][0]));
        dma4_lane((const int*)p.kv_bits + e, lds_addr(&c_bits[s][0]));
        if (lane == 0) *(int4*)&c_head[s][0] = make_int4(n | (ge + n == it_ne ? 0x100 : 0), it_tz, it_kvh << 17, 0);
        pc++;
        ge += n;
        if (ge >= it_ne) {
            ge = 0;
            gi++;
            if ((gi & 63) == 0 && gi + 64 < cnt) copy_items(gi + 64);
        }
    };
    if (threadIdx.x < 16) sy_redo[threadIdx.x] = 0;
    if (threadIdx.x == 0) sy_nredo = sy_vote = 0;
    if (w == 0) {
        const int lane = fresh_lane_id();
        int nt = 0;
        for (int i = lo + lane; i < hi; i += 64) nt += p.items[i].z & 0xfffff;
        for (int off = 32; off > 0; off >>= 1) nt += __shfl_xor(nt, off);
        if (lane == 0) sy_ntiles = nt;
        copy_items(0);
        if (cnt > 64) copy_items(64);
        __builtin_amdgcn_s_waitcnt(0x0f70);
#pragma unroll 1
        while (gi < cnt && pc < NCHUNK - 2) produce();
        __builtin_amdgcn_s_waitcnt(0x0f70);
    }
    __syncthreads();
    const int ntiles = __builtin_amdgcn_readfirstlane(sy_ntiles);
    if (ntiles == 0) return;

    // the walk over the copied chunks: where the next tile's entry lies
    int wc = 0, wp = 0, wj = 0;
    bool moved = false;   // on to another chunk: the producer owes one
    int f_i, f_b;
    i32x4 f_h;
    auto fetch_begin = [&]() __attribute__((always_inline)) {
        const int s = wc & (NCHUNK - 1);
        f_i = lds_peek(&c_idx[s][wp]);
        f_b = lds_peek(&c_bits[s][wp]);
        f_h = lds_peek4(&c_head[s][0]);
    };
    auto fetch_end = [&](Tile& t) __attribute__((always_inline)) {   // behind the last tile: the last tile again (its requests keep the counts as they are)
        const int fl = __builtin_amdgcn_readfirstlane(f_h[0]), more = wj < ntiles;
        const int end = (wp + 1 == (fl & 0xff)) & more;
        const int kt = __builtin_amdgcn_readfirstlane(f_i), tz = __builtin_amdgcn_readfirstlane(f_h[1]);
        const unsigned bits = ((unsigned)__builtin_amdgcn_readfirstlane(f_b) & 0xffffu) | (unsigned)__builtin_amdgcn_readfirstlane(f_h[2]) |
                              (end && (fl & 0x100) ? TILE_LAST : 0u);
        t.kt = more ? kt : t.kt;
        t.tz = more ? tz : t.tz;
        t.bits = more ? bits : t.bits;
        wp = end ? 0 : wp + more;
        wc += end;
        wj += more;
        moved = end;
    };
    Tile t0 = {0, 0, 0}, t1, t2;   // tiles j, j + 1, j + 2
    fetch_begin();
    fetch_end(t0);
    t1 = t0;
    fetch_begin();
    fetch_end(t1);
    t2 = t1;
    fetch_begin();
    fetch_end(t2);
    __syncthreads();
    if (w == 0) {
#pragma unroll 1
        while (gi < cnt && pc - wc <= NCHUNK - 2) produce();
    }

    // ---- requests: wave w has rows w * NREQ .. of every tile; a row behind the stream's end is its last row again
    const unsigned lane16 = fresh_lane_id() * 16;
    const unsigned k_stride = (unsigned)(p.k_tok * 2), v_stride = (unsigned)(p.v_tok * 2);
    const int* const meta_src = w == 1 ? p.end : w == 2 ? p.pos : p.art;   // (art and end are used; waves 2 and 3 ask so that all waves count alike)
    struct Req {
        const char* base;
        unsigned off, cap, lds;
    };
    auto kv_req = [&](const __bf16* x, const long head, const unsigned stride, const Tile& t, const unsigned lds) __attribute__((always_inline)) {
        int row = t.kt * 32 + w * NREQ;
        row = row < p.n ? row : p.n - 1;
        Req r;
        r.base = (const char*)x + (long)(t.bits >> 17) * head * 2 + (unsigned long)row * stride;
        r.off = 0;
        r.cap = (unsigned)(p.n - 1 - row < NREQ ? p.n - 1 - row : NREQ) * stride;
        r.lds = lds;
        return r;
    };
    auto request = [&](Req& r, const unsigned stride, const int pitch) __attribute__((always_inline)) {
        dma16_uniform(r.base, lane16 + (r.off < r.cap ? r.off : r.cap), r.lds);
        r.off += stride;
        r.lds += pitch;
    };
    auto k_req = [&](const Tile& t, const int j) __attribute__((always_inline)) {
        return kv_req(p.k, p.k_head, k_stride, t, lds_addr(ring) + (j & 1) * SLOTB + w * NREQ * GK::KRS);
    };
    auto v_req = [&](const Tile& t, const int j) __attribute__((always_inline)) {
        return kv_req(p.v, p.v_head, v_stride, t, lds_addr(ring) + (j & 1) * SLOTB + G::KTILEB + w * NREQ * GK::VRS);
    };
    auto meta_req = [&](const Tile& t, const int j) __attribute__((always_inline)) {
        const int key = t.kt * 32 + (int)((lane16 >> 4) & 31);
        dma4_uniform((const char*)meta_src, (unsigned)(key < p.n ? key : p.n - 1) * 4, lds_addr(meta_all) + (j & 3) * METAB + w * 256);
    };
    Req rv = v_req(t0, 0), rk = k_req(t0, 0);
    meta_req(t0, 0);
#pragma unroll
    for (int i = 0; i < NREQ; i++) request(rk, k_stride, GK::KRS);
    rk = k_req(t1, 1);
    meta_req(t1, 1);
#pragma unroll
    for (int i = 0; i < NREQ; i++) request(rk, k_stride, GK::KRS);
    rk = k_req(t2, 2);

    // ---- state of this wave's 32 rows
    bf16x8 qf[NS];
    int art_q = -1, pos_q = 0;
    float M = -INFINITY, l = 0.f;
    bool viol = false, fresh = true;
    int iseq = 0;
    f32x16 sa;      // a block's scores, then its probabilities
    bf16x8 pb[2];   // the probabilities as operands of P V
#pragma unroll
    for (int i = 0; i < 16; i++) sa[i] = 0.f;
    pb[0] = pb[1] = bf16x8{};
    ring_load_q<D, false>(p, w, 0, t0.tz, qf, art_q, pos_q);
    const int ln0 = (int)(lane16 >> 4);
    const int k_lane = GK::k_off(ln0 & 31) + 16 * (ln0 >> 5);
    const int v_lane = G::KTILEB + GK::v_off(4 * (ln0 >> 5) + ((ln0 >> 2) & 3)) + 32 * ((ln0 >> 4) & 1) + 8 * (ln0 & 3);

    // phase A of tile j: its scores, K Q^T.  Beside it V of the tile is requested, and what phase B requests is worked out.
    auto phase_a = [&](auto qk_c, const int j) __attribute__((always_inline)) {
        constexpr bool QK = decltype(qk_c)::value;
        constexpr int PF = 6;   // K fragments read ahead
        const char* krow = ring + (j & 1) * SLOTB + k_lane;
        bf16x8 kf[PF];
        if (QK) {
#pragma unroll
            for (int x = 0; x < PF; x++) kf[x] = *(const bf16x8*)(krow + 32 * x);
        }
        __builtin_amdgcn_sched_barrier(0);
        auto step = [&](auto x_c) __attribute__((always_inline)) {
            constexpr int x = decltype(x_c)::value;
            if constexpr (QK) {
                if (x == 0) qk_first(sa, kf[x % PF], qf[x]);
                else if (x == NS - 1) qk_last(sa, kf[x % PF], qf[x]);
                else qk_next(sa, kf[x % PF], qf[x]);
                if (x + PF < NS) kf[x % PF] = *(const bf16x8*)(krow + 32 * (x + PF));
            }
            if constexpr ((x & 3) == 2) request(rv, v_stride, GK::VRS);
            if constexpr (x == 25) rk = k_req(t2, j + 2);
            __builtin_amdgcn_sched_barrier(0);
        };
        pv_steps<NS>(step);
    };

    // phase B of tile j: P V of the tile before, and beside it the softmax of tile j's scores; K of tile j + 2 is requested, tile j + 3 looked up
    auto phase_b = [&](auto pv_c, auto init_c, auto sm_c, auto mk_c, const int j) __attribute__((always_inline)) {
        constexpr bool PV = decltype(pv_c)::value, INIT = decltype(init_c)::value, SM = decltype(sm_c)::value, MK = decltype(mk_c)::value;
        const char* vrow = ring + ((j + 1) & 1) * SLOTB + v_lane;
        s16x4 vlo[VPF], vhi[VPF];
        auto vload = [&](const int f, const int slot) __attribute__((always_inline)) {
            const char* vp = vrow + GK::v_off(16 * (f / NDT)) + 64 * (f % NDT);
            vlo[slot] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)vp);
            vhi[slot] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vp + GK::v_off(8)));
        };
        const int* meta = (const int*)(meta_all + (j & 3) * METAB);
        const int g = (int)(lane16 >> 9);
        const int tok = (t0.tz & 0xfffff) * SPINF_QTILE + 32 * w + (int)((lane16 >> 4) & 31);
        int4 ka, ke;
        auto meta_load = [&](const int i4) __attribute__((always_inline)) {
            const int ko = 8 * i4 + 4 * g;
            ka = *(const int4*)(meta + ko);
            ke = *(const int4*)(meta + 64 + ko);
        };
        auto meta_apply = [&](const int i4) __attribute__((always_inline)) {
            const int kg = t0.kt * 32 + 8 * i4 + 4 * g;
            const int kav[4] = {ka.x, ka.y, ka.z, ka.w}, kev[4] = {ke.x, ke.y, ke.z, ke.w};
#pragma unroll
            for (int jj = 0; jj < 4; jj++) {
                const int kk = kg + jj;
                bool vis = (kk <= tok) & (art_q >= 0) & (kav[jj] == art_q) & (tok < kev[jj]);
                vis = vis | (kk == tok);
                sa[4 * i4 + jj] = vis ? sa[4 * i4 + jj] : -INFINITY;
            }
        };
        float ms = 0.f, sum = 0.f;
        if (SM && MK) meta_load(0);
        if (PV) {
#pragma unroll
            for (int f = 0; f < VPF; f++) vload(f, f);
        }
        meta_req(t2, j + 2);
        __builtin_amdgcn_sched_barrier(0);
        constexpr int REF = MK ? 8 : 0, EL = REF + 1;   // steps of the row's reference, of the first element
        static_assert(EL + 16 < NVF, "the softmax ends within the products");
        auto step = [&](auto f_c) __attribute__((always_inline)) {
            constexpr int f = decltype(f_c)::value;
            if constexpr (PV) {
                const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(vlo[f % VPF], vhi[f % VPF], 0, 1, 2, 3, 4, 5, 6, 7));
                if constexpr (INIT && f < NDT) acc_mfma_init<f % NDT>(a, pb[f / NDT]);
                else acc_mfma<f % NDT>(a, pb[f / NDT]);
                if constexpr (f + VPF < NVF) vload(f + VPF, f % VPF);
            }
            if constexpr ((f & 3) == 2) request(rk, k_stride, GK::KRS);
            if constexpr (SM && MK) {
                if constexpr (f < 8 && (f & 1)) {   // (one group of four keys at a time: registers)
                    meta_apply(f >> 1);
                    if constexpr (f < 7) meta_load((f >> 1) + 1);
                }
            }
            if constexpr (SM && f == REF) {
                const bool first = M == -INFINITY;
                if (__builtin_amdgcn_ballot_w64(first) != 0) {   // only where a row meets its first keys
                    float mx = sa[0];
#pragma unroll
                    for (int i2 = 1; i2 < 16; i2++) mx = fmaxf(mx, sa[i2]);
                    mx = lane32_max(mx);
                    M = first ? mx * p.c : M;
                }
                ms = M == -INFINITY ? 0.f : M;
            }
            if constexpr (SM && f >= EL && f < EL + 16) {
                sa[f - EL] = __builtin_amdgcn_exp2f(__builtin_fmaf(sa[f - EL], p.c, -ms));
                sum += sa[f - EL];
            }
            if constexpr (SM && f == EL + 16) {
                l += sum;
                viol = viol | !(sum <= VIOL_SUM);
            }
            if constexpr (SM && f == NVF - 4) {   // (the old probabilities of this half are through)
#pragma unroll
                for (int i = 0; i < 8; i++) pb[0][i] = (__bf16)sa[i];
            }
            if constexpr (f == 18) fetch_begin();
            if constexpr (f == 25) rv = v_req(t1, j + 1);
            __builtin_amdgcn_sched_barrier(0);
        };
        pv_steps<NVF>(step);
        if (SM) {
#pragma unroll
            for (int i = 0; i < 8; i++) pb[1][i] = (__bf16)sa[8 + i];
        }
        t0 = t1;
        t1 = t2;
        fetch_end(t2);
    };
    // P V of the item's last tile j, nothing beside it
    auto phase_c = [&](auto init_c, const int j) __attribute__((always_inline)) {
        constexpr bool INIT = decltype(init_c)::value;
        const char* vrow = ring + (j & 1) * SLOTB + v_lane;
        s16x4 vlo[VPF], vhi[VPF];
        auto vload = [&](const int f, const int slot) __attribute__((always_inline)) {
            const char* vp = vrow + GK::v_off(16 * (f / NDT)) + 64 * (f % NDT);
            vlo[slot] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)vp);
            vhi[slot] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vp + GK::v_off(8)));
        };
#pragma unroll
        for (int f = 0; f < VPF; f++) vload(f, f);
        __builtin_amdgcn_sched_barrier(0);
        auto step = [&](auto f_c) __attribute__((always_inline)) {
            constexpr int f = decltype(f_c)::value;
            const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(vlo[f % VPF], vhi[f % VPF], 0, 1, 2, 3, 4, 5, 6, 7));
            if constexpr (INIT && f < NDT) acc_mfma_init<f % NDT>(a, pb[f / NDT]);
            else acc_mfma<f % NDT>(a, pb[f / NDT]);
            if constexpr (f + VPF < NVF) vload(f + VPF, f % VPF);
            __builtin_amdgcn_sched_barrier(0);
        };
        pv_steps<NVF>(step);
    };

    using T = std::true_type;
    using F = std::false_type;
    int j = 0;
    step_barrier<0>();
#pragma unroll 1
    while (j < ntiles) {
        M = -INFINITY;
        l = 0.f;
        viol = false;
        fresh = true;
        iseq++;
        const int tz_item = t0.tz;
        // (the waits below count the requests behind the ones that are needed: V of a tile in its phase A, then the metadata and K of the
        // tile after the next in its phase B; at an item's end the queries and, where all rows lie in the stream, 32 output stores)
        bool begin = true, last, act = false;   // act: the tile before left probabilities
#pragma unroll 1
        do {
            last = (t0.bits & TILE_LAST) != 0;
            const bool sm = (t0.bits >> (2 * w)) & 1u, mk = (t0.bits >> (8 + 2 * w)) & 1u;
            if (sm) phase_a(T{}, j);
            else phase_a(F{}, j);
            if (begin) step_barrier<63>();
            else step_barrier<2 * NREQ + 1>();
            if (moved && w == 0 && gi < cnt) produce();
            if (act) {
                if (sm) {
                    if (!fresh && !mk) phase_b(T{}, F{}, T{}, F{}, j);
                    else if (!fresh) phase_b(T{}, F{}, T{}, T{}, j);
                    else if (!mk) phase_b(T{}, T{}, T{}, F{}, j);
                    else phase_b(T{}, T{}, T{}, T{}, j);
                } else {
                    if (!fresh) phase_b(T{}, F{}, F{}, F{}, j);
                    else phase_b(T{}, T{}, F{}, F{}, j);
                }
                fresh = false;
            } else {
                if (sm && !mk) phase_b(F{}, F{}, T{}, F{}, j);
                else if (sm) phase_b(F{}, F{}, T{}, T{}, j);
                else phase_b(F{}, F{}, F{}, F{}, j);
            }
            act = sm;
            j++;
            if (!last) {
                if (begin) step_barrier<63>();
                else step_barrier<2 * NREQ + 1>();
            }
            begin = false;
        } while (!last);
        ring_load_q<D, false>(p, w, 0, t0.tz, qf, art_q, pos_q);   // the next item's queries (behind the last item some item's again)
        step_barrier<NREQ + 1 + NS>();
        if (act) {
            if (fresh) phase_c(T{}, j - 1);
            else phase_c(F{}, j - 1);
        }
        // ---- the item's rows
        const bool hand_over = __builtin_amdgcn_ballot_w64(viol) != 0;   // scores ranged too widely somewhere in these 32 rows
        if (hand_over) {
            if (fresh_lane_id() == 0) {
                const int was = __hip_atomic_fetch_max(&sy_redo[iseq & 15], iseq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (was < iseq) {   // first wave of the item to say so
                    const int k = __hip_atomic_fetch_add(&sy_nredo, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                    __hip_atomic_store(&p.redo[lo + k], lo + iseq - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            }
            __builtin_amdgcn_s_waitcnt(0x0f70);
        } else if ((tz_item & 0xfffff) * SPINF_QTILE + 32 * w + 32 <= p.n) {
            ring_store_rows<D, true>(p, w, 0, stage_all + w * 32 * SROW, tz_item, l);
#pragma unroll
            for (int s = 0; s < NS; s++) asm volatile("" ::"v"(qf[s]));   // (here, so that the wait for the queries leaves the stores in flight)
            asm volatile("" ::"v"(art_q), "v"(pos_q));
        } else {
            ring_store_rows<D>(p, w, 0, stage_all + w * 32 * SROW, tz_item, l);
            __builtin_amdgcn_s_waitcnt(0x0f70);
        }
        step_barrier<63>();
    }
    // ---- behind the list: the items that some wave handed over, exactly
    __builtin_amdgcn_s_waitcnt(0x0f70);
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(lds_load(&sy_nredo)) == 0) return;
    ring_paced_pass<D, false>(p, ring, stage_all, &sy_nredo, &sy_vote, lo, lo, lo);
}

}  // namespace

int spinf_launch_pipe(const AttnParams& p, int n_wg, hipStream_t stream) {
    hipLaunchKernelGGL((tree_attn_pipe_kernel<512>), dim3(n_wg), dim3(256), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return spinf_fail(SPINF_E_HIP, "tree_attn: launch (pipelined kernel): %s", hipGetErrorString(e));
    return SPINF_OK;
}
