// Tree-mask attention for short streams: a 32-row group's key blocks spread over the waves of a workgroup.
//
// The kernels of tree_attn.hip and tree_attn_ring.hip give a wave 32 query rows and walk it through all their key blocks: K Q^T,
// softmax, P V, one block after the other, 3 - 4 k clocks each.  A pass with plenty of rows hides that chain behind its other rows;
// one request's 640 tokens are 40 work items on 256 compute units, 20 blocks deep: 40 us per layer with nothing to hide behind.
//
// Here a workgroup takes one 32-row group of NH heads that share a key / value head, and its blocks two at a time (a step), as a
// pipeline of three kinds of waves, one of each per SIMD at NH = 2:
//   A (head, slot)  step t: the scores, mask and probabilities of block `slot` of round t; leaves P as MFMA operands in LDS
//   B (head, half)  step t: adds the blocks of round t - 1 to its half of the head's output dims, in ascending order
//   L               step t: requests round t's V (when the step begins: B has left its buffer) and round t + 2's K (from the middle of
//                   the step on: A has left its buffer).  A wave of its own, because requests queue: 64 KB of K and V per step take the
//                   64 bytes per clock that go into LDS a thousand clocks, as long as the step's MFMAs.
// So a SIMD's matrix core has B's products to do while A is in its softmax, and the chain is a step's (two blocks), not a block's times
// the blocks.  Measured: one layer of 640 tokens, 16 / 8 heads x 256, 17.3 us of GPU time against the ring kernel's 36.4 (of it 5 us until the
// first K has landed: work item, block list, K are three loads after each other; a step is 2.7 k clocks, 1.3 k of them the requests'); 1,408
// tokens 37.4 / 75.3.  It moves each row group's K and V on its own, four times the bytes into LDS of a 128-row item, so with every
// compute unit busy it is half as fast as the others (attention.py, _spread, has the line).
//
// Same bits as the other kernels: a block's scores, a row's reference (the maximum of the first block in which it sees a key, agreed on
// through LDS in rounds where some row has none yet), the per-lane partial sums and every output element's sequence of MFMAs are
// theirs; only which wave does them differs.  Scores too far above the reference (attn_kernels.h) are found per 32 rows and head, and
// that row group and head is done again by this workgroup with the arithmetic of tree_attn_exact_kernel, one block at a time.
#include <hip/hip_runtime.h>

#include "spinf_tree.h"
#include "common.h"

#include "attn_tiles.h"
#include "attn_kernels.h"
#include "attn_ring_io.h"

namespace {

constexpr int LISTCAP = 512;   // key blocks of a row group listed at a time (256 plan entries)

template <int D, int NH>
struct SpreadShape {
    static constexpr int NSLOT = 2;                        // key blocks per round
    static constexpr int NA = NH * NSLOT, NB = 2 * NH, NL = 4, NW = NA + NB + NL;
    static constexpr int NS = D / 16, NDT = D / 32, TPW = NDT / 2;
    using G = Geo<D, 32>;
    static constexpr int REGS = G::NREG / 2;               // regions of a tile that an L wave requests: two of them to a slot
};

__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
__device__ __forceinline__ void loads_landed() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

template <int D, int NH, bool WIN, bool ROWS>
__global__ __launch_bounds__((64 * SpreadShape<D, NH>::NW)) void tree_attn_spread_kernel(const AttnParams p, const int ktile) {
    using S = SpreadShape<D, NH>;
    using G = typename S::G;
    constexpr int NSLOT = S::NSLOT, NA = S::NA, NB = S::NB, NS = S::NS, NDT = S::NDT, TPW = S::TPW, REGS = S::REGS;
    static_assert(REGS >= 1 && REGS * 2 == G::NREG && S::NL == 2 * NSLOT, "two L waves to a slot");
    constexpr int PF = 4;                                   // K fragments read ahead
    constexpr int METAB = 3 * 256;                          // art, end, pos of a block's keys (each twice: a DMA fills 64 words)
    constexpr int OROW = (TPW >= 2 ? 128 : 64) + 16;        // staged output row: 64 (32) head dims
    __shared__ __attribute__((aligned(16))) char kbuf[2 * NSLOT * G::KTILEB];
    __shared__ __attribute__((aligned(16))) char vbuf[2 * NSLOT * G::VTILEB];
    __shared__ __attribute__((aligned(16))) char meta_all[2 * NSLOT * METAB];
    __shared__ __attribute__((aligned(16))) char pbuf[2 * NH * NSLOT * 2048];   // P of a block as the B operands of its two 16-key halves
    __shared__ float sums[2 * NH * NSLOT * 64];             // per lane: the sum of its 16 probabilities of a block
    __shared__ float tops[NH * NSLOT * 32];                 // per row: the block's maximum (while some row has no reference yet)
    __shared__ int list[LISTCAP];                           // key block | masked << 31
    __shared__ int list_row[ROWS ? LISTCAP : 1];            // compact rows: row of the block's first key where its keys are consecutive rows, else -1
    __shared__ int s_count, s_open[2], s_viol[NH];
    static_assert(sizeof(kbuf) + sizeof(vbuf) + sizeof(meta_all) + sizeof(pbuf) + sizeof(sums) + sizeof(tops) + sizeof(list) + sizeof(list_row) + 64 <= 160 * 1024, "LDS budget");
    static_assert(NB * 32 * OROW <= (int)sizeof(kbuf), "the output staging slices lie in the K buffers");

    const int lane = threadIdx.x & 63, m = lane & 31, g = lane >> 5;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool in_a = w < NA, in_b = w >= NA && w < NA + NB, in_l = w >= NA + NB;
    const int a_head = w / NSLOT, a_slot = w % NSLOT;
    const int b_head = (w - NA) / 2, b_half = (w - NA) % 2;          // output dims b_half D / 2 ..
    const int l_slot = (w - NA - NB) % NSLOT, share = (w - NA - NB) / NSLOT;
    const int k_lane = G::k_off(m) + 16 * g;
    const int v_lane = G::v_off(4 * g + ((lane >> 2) & 3)) + 32 * ((lane >> 4) & 1) + 8 * (lane & 3);
    const unsigned lane_k = (unsigned)((lane / G::CPR) * G::NREG * p.k_tok * 2 + (lane % G::CPR) * 16);
    const unsigned lane_v = (unsigned)((lane / G::CPR) * G::NREG * p.v_tok * 2 + (lane % G::CPR) * 16);

    // The workgroups of XCD x (launch slots x, x + 8, ..) take list x of the schedule (jobs and heads that share K / V), item by item,
    // the four row groups of an item side by side, the one with the most keys first.
    const int xcd = blockIdx.x & 7;
    const int lo = p.list_ptr[xcd], hi = p.list_ptr[xcd + 1];
    for (int u = blockIdx.x >> 3; u < 4 * (hi - lo); u += gridDim.x >> 3) {
        const int4 itv = p.items[lo + (u >> 2)];
        const int wr = 3 - (u & 3);
        const int t = __builtin_amdgcn_readfirstlane(itv.x), e0 = __builtin_amdgcn_readfirstlane(itv.y), iz = __builtin_amdgcn_readfirstlane(itv.z);
        const int ne = iz & 0xfffff, h0 = (int)((unsigned)iz >> 20) * NH, kvh = h0 / p.group;
        const int row0 = t * SPINF_QTILE + 32 * wr;
        if (row0 >= p.n) continue;
        const char* const kbase = (const char*)(p.k + (long)kvh * p.k_head);
        const char* const vbase = (const char*)(p.v + (long)kvh * p.v_head);
        lds_barrier();   // everyone is done with the previous item: its flags, its staged rows

        // The row group's blocks of plan entries from .. from + 255, in ascending order (the first L wave; 64-key entries hold two 32-key blocks)
        auto make_list = [&](const int from) {
            if (w != NA + NB) return;
            const int to = from + LISTCAP / 2 < ne ? from + LISTCAP / 2 : ne, nsub = ktile / 32;
            int count = 0;
            for (int e = from; e < to; e += 64) {
                const bool here = e + lane < to;
                const int kt = here ? p.kv_idx[e0 + e + lane] : 0;
                const unsigned bits = here ? p.kv_bits[e0 + e + lane] >> (2 * wr) : 0;
                int r0 = -1;
                if (ROWS && here) r0 = p.kv_row0[e0 + e + lane];
                const bool s0 = bits & 1u, s1 = bits & 2u;
                const unsigned long long below = (1ull << lane) - 1, b0 = __builtin_amdgcn_ballot_w64(s0), b1 = __builtin_amdgcn_ballot_w64(s1);
                int at = count + __popcll(b0 & below) + __popcll(b1 & below);
                if (s0) {
                    list[at] = kt * nsub | (bits & 0x100u ? 1 << 31 : 0);
                    if (ROWS) list_row[at] = r0;
                    at++;
                }
                if (s1) {
                    list[at] = kt * nsub + 1 | (bits & 0x200u ? 1 << 31 : 0);
                    if (ROWS) list_row[at] = r0 < 0 ? -1 : r0 + 32;
                }
                count += __popcll(b0) + __popcll(b1);
            }
            if (lane == 0) s_count = count;
        };
        // an L wave's share of block `kb`'s K (V) tile into buffer `buf`; with K, the keys' art / end / pos
        auto rows_at = [&](const int kb, const int reg) {   // compact rows out of sequence, or the stream's last, partial block
            long r = (long)kb * 32 + reg + G::NREG * (lane / G::CPR);
            r = r < p.n ? r : p.n - 1;
            if (ROWS) {
                const int x = p.row_of[r];
                r = x < 0 ? 0 : x;   // a pad position has no row: any row will do, only pad rows see its key
            }
            return r;
        };
        auto request_k = [&](const int buf, const int kb, const int first_row) {
            const unsigned to = lds_addr(kbuf + buf * G::KTILEB);
            if (ROWS ? first_row >= 0 : kb * 32 + 32 <= p.n) {
                const long first = (ROWS ? (long)first_row : (long)kb * 32) + share * REGS;
                dma_regions<REGS, G::KRS>(kbase + first * p.k_tok * 2, (unsigned)(p.k_tok * 2), lane_k, to + share * REGS * G::KRS);
            } else {
#pragma unroll 1
                for (int r = share * REGS; r < (share + 1) * REGS; r++)
                    dma16_lane(kbase + rows_at(kb, r) * p.k_tok * 2 + (lane % G::CPR) * 16, to + r * G::KRS);
            }
            int key = kb * 32 + m;
            key = key < p.n ? key : p.n - 1;
            const unsigned mt = lds_addr(meta_all + buf * METAB);
            if (share == 0) {
                dma4_lane(p.art + key, mt);
            } else {
                dma4_lane(p.end + key, mt + 256);
                if (WIN) dma4_lane(p.pos + key, mt + 512);
            }
        };
        auto request_v = [&](const int buf, const int kb, const int first_row) {
            const unsigned to = lds_addr(vbuf + buf * G::VTILEB);
            if (ROWS ? first_row >= 0 : kb * 32 + 32 <= p.n) {
                const long first = (ROWS ? (long)first_row : (long)kb * 32) + share * REGS;
                dma_regions<REGS, G::VRS>(vbase + first * p.v_tok * 2, (unsigned)(p.v_tok * 2), lane_v, to + share * REGS * G::VRS);
            } else {
#pragma unroll 1
                for (int r = share * REGS; r < (share + 1) * REGS; r++)
                    dma16_lane(vbase + rows_at(kb, r) * p.v_tok * 2 + (lane % G::CPR) * 16, to + r * G::VRS);
            }
        };
        auto entry = [&](const int i) { return __builtin_amdgcn_readfirstlane(list[i]); };
        auto entry_row = [&](const int i) { return ROWS ? __builtin_amdgcn_readfirstlane(list_row[i]) : 0; };

        auto p_block = [&](const int round, const int head, const int slot) { return ((round & 1) * NH + head) * NSLOT + slot; };
        auto buffer = [&](const int round, const int slot) { return (round & 1) * NSLOT + slot; };
        if (threadIdx.x < 2) s_open[threadIdx.x] = threadIdx.x == 0;
        if (threadIdx.x < NH) s_viol[threadIdx.x] = 0;

        // The three kinds of waves have a loop each (one loop with branches inside would keep every kind's registers alive in all of them).
        // They meet at the same barriers: two in front of a segment of the list, two per step, three per block of the exact pass.
        if (in_l) {
            for (int from = 0; from < ne; from += LISTCAP / 2) {
                lds_barrier();   // everyone is done with the list
                make_list(from);
                lds_barrier();
                const int count = __builtin_amdgcn_readfirstlane(s_count), rounds = (count + NSLOT - 1) / NSLOT;
                if (count == 0) continue;
                // This wave's block of round r (a last round of one block: the other slot asks for that block again, and nobody looks at
                // it).  Looked up a step ahead, while requests are on their way: an LDS read is 300 clocks when the others are at it.
                auto block = [&](const int r, int& kb, int& row) {
                    const int i = r * NSLOT + l_slot < count ? r * NSLOT + l_slot : count - 1;
                    kb = entry(i) & 0x7fffffff;
                    row = entry_row(i);
                };
                int b0, b1, b2, r0, r1, r2;
                block(0, b0, r0);
                block(1, b1, r1);
                request_k(buffer(0, l_slot), b0, r0);
                if (rounds > 1) request_k(buffer(1, l_slot), b1, r1);
                block(2, b2, r2);
                loads_landed();
                for (int t = 0; t <= rounds; t++) {
                    lds_barrier();   // round t's K and round t - 1's V and P are there; B has left round t - 2's V
                    if (t < rounds) request_v(buffer(t, l_slot), b0, r0);
                    lds_barrier();   // A has left round t's K
                    const bool more = t + 2 < rounds;
                    if (more) request_k(buffer(t, l_slot), b2, r2);
                    b0 = b1; r0 = r1;
                    b1 = b2; r1 = r2;
                    block(t + 3, b2, r2);
                    // all but those requests: round t's V and round t + 1's K (asked for half a step before it)
                    if (!more) loads_landed();
                    else if (share == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(REGS + 1) : "memory");
                    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(REGS + (WIN ? 2 : 1)) : "memory");
                }
            }
            lds_barrier();
            for (int h = 0; h < NH; h++) {
                if (__builtin_amdgcn_readfirstlane(s_viol[h]) == 0) continue;
                for (int from = 0; from < ne; from += LISTCAP / 2) {
                    lds_barrier();
                    make_list(from);
                    lds_barrier();
                    const int count = __builtin_amdgcn_readfirstlane(s_count);
                    for (int i = 0; i < count; i++) {
                        lds_barrier();   // the buffers and P have been read
                        if (l_slot == 0) {
                            request_k(0, entry(i) & 0x7fffffff, entry_row(i));
                            request_v(0, entry(i) & 0x7fffffff, entry_row(i));
                            loads_landed();
                        }
                        lds_barrier();
                        lds_barrier();
                    }
                }
                lds_barrier();
            }
        } else if (in_a) {
            const int tok = row0 + m, tok_c = tok < p.n ? tok : p.n - 1;
            bf16x8 qf[NS];
            {
                int q_row = tok_c;
                if (ROWS) {   // a pad position has no row: it computes on some row's queries and stores nothing
                    q_row = p.row_of[tok_c];
                    q_row = q_row < 0 ? 0 : q_row;
                }
                const __bf16* qp = p.q + (long)q_row * p.q_tok + (long)(h0 + a_head) * p.q_head + 8 * g;
#pragma unroll
                for (int s = 0; s < NS; s++) qf[s] = *(const bf16x8*)(qp + 16 * s);
            }
            int art_q = p.art[tok_c], pos_q = WIN ? p.pos[tok_c] : 0;
            // S^T of the block in K buffer `buf` (register i: key 8 (i / 4) + 4 g + i % 4 of the block, for this lane's row), masked
            auto scores = [&](const int buf, const int kb, const bool masked, f32x16 (&sa)[1]) __attribute__((always_inline)) {
                const char* krow = kbuf + buf * G::KTILEB + k_lane;
#pragma unroll
                for (int i = 0; i < 16; i++) sa[0][i] = 0.f;
                bf16x8 kf[PF];
#pragma unroll
                for (int s = 0; s < PF; s++) kf[s] = *(const bf16x8*)(krow + 32 * s);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int s = 0; s < NS; s++) {
                    sa[0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[s % PF], qf[s], sa[0], 0, 0, 0);
                    if (s + PF < NS) kf[s % PF] = *(const bf16x8*)(krow + 32 * (s + PF));
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (masked) apply_mask<1, WIN, 0, 32>(sa, (const int*)(meta_all + buf * METAB), kb, 0, g, tok, art_q, pos_q, p.window);
            };
            auto top_of = [&](const f32x16& sv) __attribute__((always_inline)) {
                float mx = sv[0];
#pragma unroll
                for (int i = 1; i < 16; i++) mx = fmaxf(mx, sv[i]);
                return lane32_max(mx);
            };
            auto probabilities = [&](const f32x16& sv, const float ms, bf16x8 (&pb)[2]) __attribute__((always_inline)) {
                float sum = 0.f;
#pragma unroll
                for (int i = 0; i < 16; i++) {
                    const float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(sv[i], p.c, -ms));
                    sum += pr;
                    pb[i >> 3][i & 7] = (__bf16)pr;
                }
                return sum;
            };
            auto leave_p = [&](const int at, const bf16x8 (&pb)[2], const float sum) __attribute__((always_inline)) {
                bf16x8* pp = (bf16x8*)(pbuf + at * 2048) + lane;
                pp[0] = pb[0];
                pp[64] = pb[1];
                sums[at * 64 + lane] = sum;
            };
            float M = -INFINITY;
            int parity = 0;   // (runs on over the segments of a long list: it picks the s_open word)
            for (int from = 0; from < ne; from += LISTCAP / 2) {
                lds_barrier();
                lds_barrier();
                const int count = __builtin_amdgcn_readfirstlane(s_count), rounds = (count + NSLOT - 1) / NSLOT;
                if (count == 0) continue;
                if (from == 0) {   // the queries are waited for here, not in front of the barriers that the others are waiting at
                    loads_landed();
                    asm volatile("" : "+v"(art_q), "+v"(pos_q));
                    art_q = tok < p.n ? art_q : -1;
                }
                for (int t = 0; t <= rounds; t++, parity ^= 1) {
                    lds_barrier();
                    const int i = t * NSLOT + a_slot;
                    const bool mine = i < count;
                    const bool open = __builtin_amdgcn_readfirstlane(s_open[parity]) != 0;
                    f32x16 sa[1] = {f32x16{}};
                    if (mine) {
                        const int en = entry(i);
                        scores(buffer(t, a_slot), en & 0x7fffffff, en < 0, sa);
                    }
                    if (open) {
                        const float mx = mine ? top_of(sa[0]) : -INFINITY;
                        if (g == 0) tops[(a_head * NSLOT + a_slot) * 32 + m] = mx;
                    }
                    lds_barrier();
                    if (open) {   // some row of the workgroup has no reference yet: the first block of the round in which it sees a key sets it
#pragma unroll
                        for (int s = 0; s < NSLOT; s++) {
                            const float mx = tops[(a_head * NSLOT + s) * 32 + m];
                            M = M == -INFINITY ? mx * p.c : M;
                        }
                        if (__builtin_amdgcn_ballot_w64(M == -INFINITY) != 0) s_open[parity ^ 1] = 1;
                        if (threadIdx.x == 0) s_open[parity] = 0;
                    }
                    if (mine) {
                        bf16x8 pb[2];
                        const float sum = probabilities(sa[0], M == -INFINITY ? 0.f : M, pb);
                        if (__builtin_amdgcn_ballot_w64(!(sum <= VIOL_SUM)) != 0) s_viol[a_head] = 1;
                        leave_p(p_block(t, a_head, a_slot), pb, sum);
                    }
                }
            }
            lds_barrier();
            // scores too far above their reference somewhere in a head's 32 rows: that head again, exactly, one block at a time
            for (int h = 0; h < NH; h++) {
                if (__builtin_amdgcn_readfirstlane(s_viol[h]) == 0) continue;
                M = -INFINITY;
                float le = 0.f;
                for (int from = 0; from < ne; from += LISTCAP / 2) {
                    lds_barrier();
                    lds_barrier();
                    const int count = __builtin_amdgcn_readfirstlane(s_count);
                    for (int i = 0; i < count; i++) {
                        lds_barrier();
                        lds_barrier();
                        if (w == h * NSLOT) {
                            f32x16 sa[1];
                            bf16x8 pb[2];
                            const int en = entry(i);
                            scores(0, en & 0x7fffffff, en < 0, sa);
                            const float tm = top_of(sa[0]) * p.c;
                            const bool up = tm > M + TAU_LAZY;
                            const float mn = up ? tm : M;
                            const float alpha = up ? __builtin_amdgcn_exp2f(M - mn) : 1.0f;
                            le *= alpha;
                            M = mn;
                            const float sum = probabilities(sa[0], mn == -INFINITY ? 0.f : mn, pb);
                            le += sum;
                            if (g == 0) tops[m] = alpha;
                            leave_p(0, pb, le);
                        }
                        lds_barrier();
                    }
                }
                lds_barrier();
                if (threadIdx.x == 0) atomicAdd(&p.counters[NLIST + 3], 1);   // running total, for spinf_attn_exact_items
            }
        } else {
            f32x16 o[TPW];
            float l = 0.f;
            auto add_block = [&](const int v_buf, const int at) __attribute__((always_inline)) {
                const char* vrow = vbuf + v_buf * G::VTILEB + v_lane + 64 * TPW * b_half;
                const bf16x8* pp = (const bf16x8*)(pbuf + at * 2048) + lane;
                const bf16x8 pb[2] = {pp[0], pp[64]};
#pragma unroll
                for (int f = 0; f < 2; f++)
#pragma unroll
                    for (int dt = 0; dt < TPW; dt++) {
                        const char* vp = vrow + G::v_off(16 * f) + 64 * dt;
                        const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)vp);
                        const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vp + G::v_off(8)));
                        o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7)), pb[f], o[dt], 0, 0, 0);
                    }
            };
            auto zero = [&]() __attribute__((always_inline)) {
#pragma unroll
                for (int dt = 0; dt < TPW; dt++)
#pragma unroll
                    for (int i = 0; i < 16; i++) o[dt][i] = 0.f;
            };
            zero();
            for (int from = 0; from < ne; from += LISTCAP / 2) {
                lds_barrier();
                lds_barrier();
                const int count = __builtin_amdgcn_readfirstlane(s_count), rounds = (count + NSLOT - 1) / NSLOT;
                if (count == 0) continue;
                lds_barrier();
                lds_barrier();
                for (int t = 1; t <= rounds; t++) {
                    lds_barrier();
                    l += sums[p_block(t - 1, b_head, 0) * 64 + lane];
                    add_block(buffer(t - 1, 0), p_block(t - 1, b_head, 0));
                    lds_barrier();
                    if ((t - 1) * NSLOT + 1 < count) {
                        l += sums[p_block(t - 1, b_head, 1) * 64 + lane];
                        add_block(buffer(t - 1, 1), p_block(t - 1, b_head, 1));
                    }
                }
            }
            lds_barrier();
            for (int h = 0; h < NH; h++) {
                if (__builtin_amdgcn_readfirstlane(s_viol[h]) == 0) continue;
                if (b_head == h) zero();
                for (int from = 0; from < ne; from += LISTCAP / 2) {
                    lds_barrier();
                    lds_barrier();
                    const int count = __builtin_amdgcn_readfirstlane(s_count);
                    for (int i = 0; i < count; i++) {
                        lds_barrier();
                        lds_barrier();
                        lds_barrier();
                        if (b_head == h) {
                            const float alpha = tops[m];
#pragma unroll
                            for (int dt = 0; dt < TPW; dt++)
#pragma unroll
                                for (int i2 = 0; i2 < 16; i2++) o[dt][i2] *= alpha;
                            add_block(0, 0);
                        }
                    }
                }
                if (b_head == h) l = sums[lane];
                lds_barrier();
            }

            // output rows, 64 (32) head dims at a time through the wave's own slice of the K buffers
            char* const stage = kbuf + (w - NA) * 32 * OROW;
            const float inv = 1.0f / lane32_sum(l);
            __bf16* const ob = p.o + (long)(h0 + b_head) * p.o_head + 32 * TPW * b_half;
            constexpr int TP = TPW >= 2 ? 2 : 1, PPR = 4 * TP, RPS = 64 / PPR;   // tiles at a time, 16-byte pieces per row, rows per store
#pragma unroll
            for (int d0 = 0; d0 < TPW; d0 += TP) {
#pragma unroll
                for (int dd = 0; dd < TP; dd++)
#pragma unroll
                    for (int i4 = 0; i4 < 4; i4++) {
                        bf16x4 r;
#pragma unroll
                        for (int jj = 0; jj < 4; jj++) r[jj] = (__bf16)(o[d0 + dd][4 * i4 + jj] * inv);
                        *(bf16x4*)(stage + m * OROW + (32 * dd + 8 * i4 + 4 * g) * 2) = r;
                    }
#pragma unroll
                for (int j = 0; j < 32 / RPS; j++) {
                    const int row = j * RPS + lane / PPR, col = lane % PPR;
                    const bf16x8 val = *(const bf16x8*)(stage + row * OROW + col * 16);
                    long at = row0 + row < p.n ? row0 + row : -1;
                    if (ROWS && at >= 0) at = p.row_of[at];
                    if (at >= 0) *(bf16x8*)(ob + at * p.o_tok + 32 * d0 + col * 8) = val;
                }
            }
        }
    }
}

template <int D, int NH, bool WIN, bool ROWS>
int launch_spread_t(const AttnParams& p, int ktile, long n_items, hipStream_t stream) {
    // as many workgroups as row groups, in whole rounds over the eight lists; a list with more than its eighth of the items goes round
    const long want = (4 * n_items + 7) / 8 * 8;
    hipLaunchKernelGGL((tree_attn_spread_kernel<D, NH, WIN, ROWS>), dim3((unsigned)(want < (1 << 20) ? want : 1 << 20)), dim3(64 * SpreadShape<D, NH>::NW), 0, stream, p, ktile);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return spinf_fail(SPINF_E_HIP, "tree_attn: launch (spread kernel): %s", hipGetErrorString(e));
    return SPINF_OK;
}

template <int D, int NH>
int launch_spread_d(const AttnParams& p, bool win, int ktile, long n_items, hipStream_t s) {
    if (p.row_of) return win ? launch_spread_t<D, NH, true, true>(p, ktile, n_items, s) : launch_spread_t<D, NH, false, true>(p, ktile, n_items, s);
    return win ? launch_spread_t<D, NH, true, false>(p, ktile, n_items, s) : launch_spread_t<D, NH, false, false>(p, ktile, n_items, s);
}

}  // namespace

int spinf_launch_spread(const AttnParams& p, int d, int heads, bool win, int ktile, long n_items, hipStream_t stream) {
    switch (d) {
        case 64: return heads == 2 ? launch_spread_d<64, 2>(p, win, ktile, n_items, stream) : launch_spread_d<64, 1>(p, win, ktile, n_items, stream);
        case 128: return heads == 2 ? launch_spread_d<128, 2>(p, win, ktile, n_items, stream) : launch_spread_d<128, 1>(p, win, ktile, n_items, stream);
        case 256: return heads == 2 ? launch_spread_d<256, 2>(p, win, ktile, n_items, stream) : launch_spread_d<256, 1>(p, win, ktile, n_items, stream);
    }
    return spinf_fail(SPINF_E_ARG, "tree_attn: the spread kernel takes head dim 64, 128 or 256, not %d", d);
}
