// Gated DeltaNet over small subtrees ("forests"): the short segments below a kept state, taken together instead of level by level.
//
// Why.  A trie of options has thousands of segments of a few tokens over six or seven levels.  Run one segment at a time, every
// segment that forks leaves its state (64 KB per value head) for its children to read back: a 16k-token stream of 22 tries moved
// 3 GB of states for 0.3 GB of rows, in seven launches after each other (0.70 ms; memory bound at 4.3 TB/s).  The delta rule needs
// no state between the nodes of such a tree.  With S the state above the tree, G the sum of g along a token's path inside it and
// D_ij = e^{G_i - G_j},
//     V'_i = beta_i (v_i - e^{G_i} k_i S - sum_{j above i} D_ij (k_i . k_j) V'_j)
//     o_i  = s (e^{G_i} q_i S + sum_{j above or at i} D_ij (q_i . k_j) V'_j)
// which is the chunked form of gdn_chunk.hip with "earlier in the sequence" replaced by "above in the tree".
//
// How.  The host (gdnplan.cpp) lays the trees that hang on one state out in pre-order and cuts them into units of whole trees and a
// unit into blocks of 32 tokens.  One workgroup (4 waves) owns one (unit, value head), loads S once (as the bf16 operand the products
// take: nothing updates it) and walks the blocks.  Inside a block the tokens above a token are a bit mask.  Those in earlier blocks
// are, by the pre-order, a prefix of the path of the block's FIRST token, so the K, V' and G rows of that path are all that is kept
// of earlier blocks: a stack in LDS, indexed by depth (64 at most).  Per block, wave w owning value columns 32 w .. +31:
//     A = -strict(beta_i (K K^T)_ij D_ij), P = (s Q K^T D)_ij                       (waves 0..2, one 16 x 16 tile each)
//     C = -(K Kst^T)_ij D_ij, E = (s Q Kst^T D)_ij over the stack, 32 rows at a time  (one tile per wave)
//     T = (I - A)^-1 (wave 0);  R = C V'st - e^G (K S);  V' = T diag(beta) (V + R);  O = s e^G (Q S) + E V'st + P V'
// K S and Q S need neither T nor the previous block, so they run beside the solve, and no product with W = T diag(beta e^G) K is
// left: 4 barriers a block against 6 of the chunk kernel.  A block of 32 is also fuller than the chunk kernel's pairs of leaves
// (two times 16 rows, whatever the leaves use of them).
//
// What is not finite in one option must not reach the others of its blocks, as every product above meets it with a coefficient of zero.
// The entries of A, beta and g are cleared where they are computed or staged, and their token noted; V' is looked at (a product with zeros) and, where it is not finite, computed again with such entries of V + R cleared.  Noted tokens and all below them come out
// as NaN, per value column; a stack row carries its note in a bit mask beside V'.  Outputs of all other tokens keep their bits.  The look
// costs 2 % of a layer's scans over a stream of tries (203.8 -> 208.2 us), 1 % of the layer.
//
// What it measured (the stream above, 10.6 k tokens in tries, 32 value heads): 167 us in one launch for 0.70 ms in six; 0.4 GB of rows
// and states, 2.5 TB/s.  Bound by a block's chain of phases: 11 k clocks, of them 2.7 k the solve on wave 0, 1.6 k A and P, 1.25 k staging
// and G, 1.7 k R, 2.6 k V' / O and the stores, two workgroups per compute unit (LDS 79 KB, 256 registers).  Eight waves of 16 columns
// (128 registers, four waves per SIMD) took 177 us: the solve, with fewer registers to read A ahead into, was 4.8 k.
#include <hip/hip_runtime.h>

#include "spinf_tree.h"
#include "common.h"
#include "gdn_tiles.h"
#include "gdn_forest.h"

using namespace gdn_tiles;

namespace {
constexpr int KD = 128, VD = 128;
constexpr int CH = GDN_FOREST_BLOCK;     // tokens per block
constexpr int ST = GDN_FOREST_DEPTH;     // rows of the stack
constexpr int LD = 136;                  // row strides (elements) as in gdn_chunk.hip: K, Q and the stack's K (row-wise reads) 68 banks,
constexpr int LDT = 144;                 // V (transposing reads) 72,
constexpr int LS = ST + 4;               // the stack's V', by value column: 34 banks.  The last four are a bit mask of the rows that are not finite
__device__ __forceinline__ bool not_finite(float x) { return (__builtin_bit_cast(unsigned, x) & 0x7f800000u) == 0x7f800000u; }
__device__ __forceinline__ bool not_finite(__bf16 x) { return (__builtin_bit_cast(unsigned short, x) & 0x7f80u) == 0x7f80u; }
__device__ __forceinline__ bf16x8 join_rows(const __bf16* p) { return join(*(const bf16x4*)p, *(const bf16x4*)(p + 16)); }
}  // namespace

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gdn_forest_kernel(const GdnParams p) {
    __shared__ __attribute__((aligned(16))) __bf16 Ks[CH * LD];
    __shared__ __attribute__((aligned(16))) __bf16 Qs[CH * LD];
    __shared__ __attribute__((aligned(16))) __bf16 Vs[CH * LDT];     // V; later the waves' output tiles
    __shared__ __attribute__((aligned(16))) float As[32 * LA];
    __shared__ __attribute__((aligned(16))) float Ts[32 * LX];       // T_00 in rows 0..15, T_11 in rows 16..31
    __shared__ __attribute__((aligned(16))) float Xs[16 * LX];
    __shared__ __attribute__((aligned(16))) __bf16 Ps[CH * LP];
    __shared__ __attribute__((aligned(16))) __bf16 Tus[CH * LP];
    __shared__ __attribute__((aligned(16))) __bf16 Cs[CH * LP];
    __shared__ __attribute__((aligned(16))) __bf16 Es[CH * LP];
    __shared__ __attribute__((aligned(16))) __bf16 Kst[ST * LD];
    __shared__ __attribute__((aligned(16))) __bf16 Vst[VD * LS];
    __shared__ __attribute__((aligned(16))) float Gst[ST];
    __shared__ __attribute__((aligned(16))) float Gs[CH];
    __shared__ __attribute__((aligned(16))) float Bs[CH];
    __shared__ __attribute__((aligned(16))) int Ds[CH];              // 1 + depth of a token the next block's path holds, 0 for others
    __shared__ __attribute__((aligned(16))) float Gr[CH];
    __shared__ int Rs[CH], Ns[CH], Ms[CH];
    __shared__ unsigned odd_rows;                                    // tokens of the block with a beta, a g or a row of A that is not finite
    static_assert(4 * 32 * LO <= CH * LDT, "the output tiles must fit the V tile");

    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), c = lane & 15, q4 = lane >> 4;
    long slot = blockIdx.x;     // (value heads that share a key head 8 launch slots apart: gdn_chunk.hip)
    if (p.hv == 2 * p.h && gridDim.x % 16 == 0) slot = (slot / 16) * 16 + (slot % 8) * 2 + (slot % 16) / 8;
    const int hv = (int)(slot % p.hv);
    const int hk = hv / (p.hv / p.h);
    const long unit = slot / p.hv;
    const long b0 = p.cu[unit];
    const int n_blocks = (int)(p.cu[unit + 1] - b0);
    const int* table = (const int*)p.idx + b0 * GDN_FOREST_INTS;
    __bf16* Ow = Vs + w * 32 * LO;

    // the next block's rows are fetched into registers while the current one is computed, their table entries one block earlier still
    bf16x8 pk[2], pq[2], pv[2];
    int pr = -1, pm = 0, pn = 0;
    float pg = 0.f;
    __bf16 pbeta = (__bf16)0.f;
    int ra[2], rb = -1, rm = 0, rn = 0;
    auto fetch_rows = [&](const int j) __attribute__((always_inline)) {
        const int* t = table + (long)j * GDN_FOREST_INTS;
        const bool there = j < n_blocks;
        ra[0] = ra[1] = rb = -1;
        rm = rn = 0;
        if (there) {
            ra[0] = t[tid >> 4];
            ra[1] = t[16 + (tid >> 4)];
            if (tid < CH) { rb = t[tid]; rm = t[CH + tid]; rn = t[2 * CH + tid]; }
        }
    };
    auto fetch_data = [&]() __attribute__((always_inline)) {
        const int col = (tid & 15) * 8;
#pragma unroll
        for (int cc = 0; cc < 2; cc++) {
#pragma unroll
            for (int j = 0; j < 8; j++) { pk[cc][j] = (__bf16)0.f; pq[cc][j] = (__bf16)0.f; pv[cc][j] = (__bf16)0.f; }
            if (ra[cc] >= 0) {
                pk[cc] = *(const bf16x8*)(p.k + row_offset(ra[cc], p.q_tok) + hk * KD + col);
                pq[cc] = *(const bf16x8*)(p.q + row_offset(ra[cc], p.q_tok) + hk * KD + col);
                pv[cc] = *(const bf16x8*)(p.v + row_offset(ra[cc], p.v_tok) + hv * VD + col);
            }
        }
        pr = rb; pm = rm; pn = rn;
        pg = 0.f;
        pbeta = (__bf16)0.f;
        if (rb >= 0) {
            pg = p.g[row_offset(rb, p.g_tok) + hv];
            pbeta = p.beta[row_offset(rb, p.g_tok) + hv];
        }
    };
    fetch_rows(0);
    // ---- S as the B operand of a 16x16x32 product: columns 32 w + 16 vt + c, rows 32 s + 4 q4 + r and + 16.  Requested before the
    // first block's rows and rounded behind their request: a unit of one block is mostly these two latencies.
    f32x4 S0[8][2];
    const long src = (p.h0 != nullptr && p.h0_idx != nullptr) ? p.h0_idx[unit] : -1;
#pragma unroll
    for (int kt = 0; kt < 8; kt++)
#pragma unroll
        for (int vt = 0; vt < 2; vt++) S0[kt][vt] = zero4();
    if (src >= 0) {
        const float* hp = p.h0 + ((src * p.hv + hv) * KD + 4 * q4) * VD + 32 * w + c;
#pragma unroll
        for (int kt = 0; kt < 8; kt++)
#pragma unroll
            for (int r = 0; r < 4; r++)
#pragma unroll
                for (int vt = 0; vt < 2; vt++) S0[kt][vt][r] = hp[(16 * kt + r) * VD + 16 * vt];
    }
    fetch_data();
    fetch_rows(1);
    // (rows of the stack that no block has written yet meet zero coefficients: they must not hold a NaN)
    for (int i = tid; i < VD * LS / 4; i += 256) *(bf16x4*)(Vst + 4 * i) = zero_bf4();
    bf16x8 sb[4][2];
#pragma unroll
    for (int s = 0; s < 4; s++)
#pragma unroll
        for (int vt = 0; vt < 2; vt++) sb[s][vt] = join(round4(S0[2 * s][vt]), round4(S0[2 * s + 1][vt]));

    bool noted = false;    // does a row of the stack carry a note in one of this wave's columns?
    for (int j = 0; j < n_blocks; j++) {
        lds_barrier();   // every wave is done with the previous block's tiles; the stack holds this block's path
        if (tid < CH) {
            const bool odd = not_finite(pg) || not_finite(pbeta);
            const unsigned long odds = __builtin_amdgcn_ballot_w64(odd);
            if (tid == 0) odd_rows = (unsigned)odds;
            Gr[tid] = odd ? 0.f : pg;
            Bs[tid] = odd ? 0.f : (float)pbeta;
            Rs[tid] = pr;
            Ms[tid] = pm;
            Ns[tid] = pn;
            Ds[tid] = (pn >> 8) & 0xff;
        }
        {
            const int col = (tid & 15) * 8;
#pragma unroll
            for (int cc = 0; cc < 2; cc++) {
                const int row = (tid >> 4) + 16 * cc;
                *(bf16x8*)(Ks + row * LD + col) = pk[cc];
                *(bf16x8*)(Qs + row * LD + col) = pq[cc];
                *(bf16x8*)(Vs + row * LDT + col) = pv[cc];
            }
        }
        if (w == 0) {    // G: the path's sum so far and the tokens above in this block; lanes 0..31 add rows 0..15, the others 16..31
            wave_lds_order();
            int at = lane;                 // (addresses are computed here, as further down: kept in registers they would push others out)
            asm volatile("" : "+v"(at));
            const int row = at & 31, half = at >> 5;
            const int above = (Ms[row] | (int)(1u << row)) >> (16 * half);
            float x = 0.f;
#pragma unroll
            for (int m4 = 0; m4 < 4; m4++) {
                const f32x4 gv = *(const f32x4*)(Gr + 16 * half + 4 * m4);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float g = gv[r];
                    x += __builtin_bit_cast(float, __builtin_bit_cast(int, g) & -((above >> (4 * m4 + r)) & 1));
                }
            }
            x += __shfl_xor(x, 32);
            const int n = Ns[row] & 0xff;
            if (n > 0) x += Gst[n - 1];
            if (lane < CH) Gs[row] = x;
        }
        lds_barrier();
        const int meta = __builtin_amdgcn_readfirstlane(Ns[0]);
        const int depth = (meta >> 16) & 0xff, next_depth = (meta >> 24) & 0xff;   // rows of this block's path; of the next one's

        // ---- A and P inside the block (tiles (jt, it) = (0,0), (0,1), (1,1); lane = row i, registers = columns j)
        if (w < 3) {
            const int jt = w >> 1, it = (w + 1) >> 1;
            f32x4 kk = zero4(), qk = zero4();
#pragma unroll
            for (int s = 0; s < KD / 32; s++) {
                const bf16x8 kj = *(const bf16x8*)(Ks + (16 * jt + c) * LD + 32 * s + 8 * q4);
                const bf16x8 ki = *(const bf16x8*)(Ks + (16 * it + c) * LD + 32 * s + 8 * q4);
                const bf16x8 qi = *(const bf16x8*)(Qs + (16 * it + c) * LD + 32 * s + 8 * q4);
                kk = mfma32(kj, ki, kk);
                qk = mfma32(kj, qi, qk);
            }
            const int i = 16 * it + c;
            const int above = Ms[i] >> (16 * jt + 4 * q4);
            const float Gi = Gs[i], bi = Bs[i];
            const f32x4 Gj = *(const f32x4*)(Gs + 16 * jt + 4 * q4);
            f32x4 a4;
            bf16x4 p4;
            bool odd = false;
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int jj = 16 * jt + 4 * q4 + r;
                const bool up = (above >> r) & 1;
                const float d = __expf(Gi - Gj[r]);
                const float a = up ? -bi * kk[r] * d : 0.f;
                const bool o = not_finite(a);
                a4[r] = o ? 0.f : a;
                odd |= o;
                p4[r] = (__bf16)(up || jj == i ? p.scale * qk[r] * d : 0.f);
            }
            if (odd) atomicOr(&odd_rows, 1u << i);
            *(f32x4*)(As + i * LA + 16 * jt + 4 * q4) = a4;
            *(bf16x4*)(Ps + i * LP + 16 * jt + 4 * q4) = p4;
        }
        // C and E over 32 rows of the stack: tile (jt, it) of wave w
        auto against_path = [&](const int first, const int c, const int q4) __attribute__((always_inline)) {
            const int jt = w >> 1, it = w & 1;
            f32x4 kk = zero4(), qk = zero4();
#pragma unroll
            for (int s = 0; s < KD / 32; s++) {
                const bf16x8 kj = *(const bf16x8*)(Kst + (first + 16 * jt + c) * LD + 32 * s + 8 * q4);
                const bf16x8 ki = *(const bf16x8*)(Ks + (16 * it + c) * LD + 32 * s + 8 * q4);
                const bf16x8 qi = *(const bf16x8*)(Qs + (16 * it + c) * LD + 32 * s + 8 * q4);
                kk = mfma32(kj, ki, kk);
                qk = mfma32(kj, qi, qk);
            }
            const int i = 16 * it + c, n = (Ns[i] & 0xff) - (first + 16 * jt + 4 * q4);
            const float Gi = Gs[i];
            const f32x4 Gj = *(const f32x4*)(Gst + first + 16 * jt + 4 * q4);
            bf16x4 c4, e4;
#pragma unroll
            for (int r = 0; r < 4; r++) {    // (rows past a token's path, and rows never written, are selected away)
                const float d = __expf(Gi - Gj[r]);
                c4[r] = (__bf16)(r < n ? -kk[r] * d : 0.f);
                e4[r] = (__bf16)(r < n ? p.scale * qk[r] * d : 0.f);
            }
            *(bf16x4*)(Cs + i * LP + 16 * jt + 4 * q4) = c4;
            *(bf16x4*)(Es + i * LP + 16 * jt + 4 * q4) = e4;
        };
        if (depth > 0) against_path(0, c, q4);
        lds_barrier();

        // ---- T diag(beta) on wave 0, while the other waves go on with their columns
        if (w == 0) solve_tile<true, true>(As, Bs, Ts, Xs, Tus, c, q4, false);
        // Block j + 1 is requested here, behind the solve, which needs the registers; it has the rest of this block to arrive.
        fetch_data();
        fetch_rows(j + 2);
        // ---- R = C V'st - e^G (K S) and s e^G (Q S) + E V'st   (lane = column v, registers = rows i)
        f32x4 R[2][2], O[2][2];
#pragma unroll
        for (int it = 0; it < 2; it++)
#pragma unroll
            for (int vt = 0; vt < 2; vt++) R[it][vt] = O[it][vt] = zero4();
#pragma unroll
        for (int s = 0; s < KD / 32; s++)
#pragma unroll
            for (int it = 0; it < 2; it++) {
                const bf16x8 kA = join_rows(Ks + (16 * it + c) * LD + 32 * s + 4 * q4), qA = join_rows(Qs + (16 * it + c) * LD + 32 * s + 4 * q4);
#pragma unroll
                for (int vt = 0; vt < 2; vt++) {
                    R[it][vt] = mfma32(kA, sb[s][vt], R[it][vt]);
                    O[it][vt] = mfma32(qA, sb[s][vt], O[it][vt]);
                }
            }
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const f32x4 Gi = *(const f32x4*)(Gs + 16 * it + 4 * q4);
            f32x4 e;
#pragma unroll
            for (int r = 0; r < 4; r++) e[r] = __expf(Gi[r]);
#pragma unroll
            for (int vt = 0; vt < 2; vt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    R[it][vt][r] *= -e[r];
                    O[it][vt][r] *= p.scale * e[r];
                }
        }
        for (int first = 0; first < depth; first += 32) {
            if (first > 0) {
                int at = lane;
                asm volatile("" : "+v"(at));
                lds_barrier();
                against_path(first, at & 15, at >> 4);
                lds_barrier();
            }
#pragma unroll
            for (int vt = 0; vt < 2; vt++) {
                const bf16x8 vB = join_rows(Vst + (32 * w + 16 * vt + c) * LS + first + 4 * q4);
#pragma unroll
                for (int it = 0; it < 2; it++) {
                    R[it][vt] = mfma32(join_rows(Cs + (16 * it + c) * LP + 4 * q4), vB, R[it][vt]);
                    O[it][vt] = mfma32(join_rows(Es + (16 * it + c) * LP + 4 * q4), vB, O[it][vt]);
                }
            }
        }
        bf16x8 vin[2];
#pragma unroll
        for (int vt = 0; vt < 2; vt++) vin[vt] = join(frag_tr4(Vs, LDT, 0, 32 * w + 16 * vt, lane), frag_tr4(Vs, LDT, 16, 32 * w + 16 * vt, lane));
        lds_barrier();   // T visible; every wave has read its V columns
        // ---- V' = T diag(beta) (V + R), with R rounded by itself (V is exact);  O += P V';  the path's rows of V' go on the stack (each wave its own columns)
        {
            bf16x8 tA[2], pA[2];
#pragma unroll
            for (int it = 0; it < 2; it++) {
                const __bf16* tp = Tus + (16 * it + c) * LP + 4 * q4;
                const __bf16* pp = Ps + (16 * it + c) * LP + 4 * q4;
                tA[it] = join(*(const bf16x4*)tp, it ? *(const bf16x4*)(tp + 16) : zero_bf4());
                pA[it] = join(*(const bf16x4*)pp, it ? *(const bf16x4*)(pp + 16) : zero_bf4());
            }
            bf16x8 rB[2];
            bf16x4 vs[2][2];
#pragma unroll
            for (int vt = 0; vt < 2; vt++) {
                rB[vt] = join(round4(R[0][vt]), round4(R[1][vt]));
#pragma unroll
                for (int it = 0; it < 2; it++) {
                    vs[it][vt] = round4(mfma32(tA[it], rB[vt], mfma32(tA[it], vin[vt], zero4())));
                }
            }
            const bf16x8 none = join(zero_bf4(), zero_bf4());
            const float z = mfma32(none, join(vs[0][1], vs[1][1]), mfma32(none, join(vs[0][0], vs[1][0]), zero4()))[0];   // NaN if a column of V' is not finite
            const bool look = noted || __builtin_amdgcn_ballot_w64(z != z || odd_rows != 0) != 0;
            unsigned of_column[2] = {0, 0};       // the tokens to note, by this lane's columns
            if (look) {
#pragma unroll
                for (int vt = 0; vt < 2; vt++) {
                    unsigned m = 0;
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        if (not_finite((__bf16)rB[vt][e]) || not_finite((__bf16)vin[vt][e])) {
                            rB[vt][e] = vin[vt][e] = (__bf16)0.f;
                            m |= 1u << (16 * (e >> 2) + 4 * q4 + (e & 3));
                        }
#pragma unroll
                    for (int it = 0; it < 2; it++) {
                        vs[it][vt] = round4(mfma32(tA[it], rB[vt], mfma32(tA[it], vin[vt], zero4())));
#pragma unroll
                        for (int r = 0; r < 4; r++)      // (sums of finite numbers past the range)
                            if (not_finite((__bf16)vs[it][vt][r])) {
                                vs[it][vt][r] = (__bf16)0.f;
                                m |= 1u << (16 * it + 4 * q4 + r);
                            }
                    }
                    m |= __shfl_xor(m, 16);
                    of_column[vt] = odd_rows | m | __shfl_xor(m, 32);
                }
            }
#pragma unroll
            for (int vt = 0; vt < 2; vt++) {
                const bf16x8 vB = join(vs[0][vt], vs[1][vt]);
#pragma unroll
                for (int it = 0; it < 2; it++)
                    *(bf16x4*)(Ow + (16 * vt + c) * LO + 16 * it + 4 * q4) = round4(mfma32(pA[it], vB, O[it][vt]));      // O^T[v][i]
                if (next_depth > 0) {
#pragma unroll
                    for (int it = 0; it < 2; it++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int d = Ds[16 * it + 4 * q4 + r];
                            if (d > 0) Vst[(32 * w + 16 * vt + c) * LS + d - 1] = vs[it][vt][r];
                        }
                }
            }
            if (look) {      // the noted tokens and those below them
                int at = lane;         // (addresses of this path only: not to be kept in registers beside the other one's)
                asm volatile("" : "+v"(at));
                noted = false;
                wave_lds_order();
#pragma unroll 1
                for (int vt = 0; vt < 2; vt++) {
                    const int col = 16 * vt + (at & 15), row = 4 * (at >> 4);
                    const unsigned of = vt ? of_column[1] : of_column[0];
                    unsigned long* const notes = (unsigned long*)(Vst + (32 * w + col) * LS + ST);
                    unsigned long on_stack = *notes;
                    unsigned hit = 0;
#pragma unroll 1
                    for (int e = 0; e < 8; e++) {
                        const int i = 16 * (e >> 2) + row + (e & 3), n = Ns[i] & 0xff;
                        if ((((unsigned)Ms[i] | (1u << i)) & of) != 0 || (n > 0 && on_stack << (64 - n) != 0)) {
                            hit |= 1u << i;
                            Ow[col * LO + i] = (__bf16)__builtin_nanf("");
                        }
                    }
                    hit |= __shfl_xor(hit, 16);
                    hit |= __shfl_xor(hit, 32);
                    if (next_depth > 0) {
#pragma unroll 1
                        for (int i = 0; i < CH; i++)
                            if (const int d = Ds[i]; d > 0) on_stack = (on_stack & ~(1ul << (d - 1))) | ((unsigned long)((hit >> i) & 1u) << (d - 1));
                        *notes = on_stack;
                    }
                    noted |= __builtin_amdgcn_ballot_w64(on_stack != 0) != 0;
                }
            }
        }
        wave_lds_order();
        store_tile(Ow, Rs, p.o, p.o_tok, hv * VD + 32 * w, c, q4);
        // ---- the path's K and G rows (read by every wave after the next two barriers; this block's readers are behind the last one)
        if (next_depth > 0) {
            int at = tid;
            asm volatile("" : "+v"(at));
#pragma unroll
            for (int cc = 0; cc < 2; cc++) {
                const int row = (at >> 4) + 16 * cc, d = Ds[row], col = (at & 15) * 8;
                if (d > 0) *(bf16x8*)(Kst + (d - 1) * LD + col) = *(const bf16x8*)(Ks + row * LD + col);
            }
            if (at < CH && Ds[at] > 0) Gst[Ds[at] - 1] = Gs[at];
        }
    }
}

// cu [n_seg + 1]: blocks of a unit; idx: the block table (int32, GDN_FOREST_INTS per block); h0_idx [n_seg]: the state above a unit
int gdn_forest_launch(const GdnParams& p, hipStream_t stream) {
    if (p.dv != VD) return spinf_fail(SPINF_E_ARG, "gdn: value head dim %d, the forest kernel is built for 128", p.dv);
    if (!p.idx) return spinf_fail(SPINF_E_ARG, "gdn: mode 2 needs its block table");
    if (p.n_seg > INT32_MAX / p.hv) return spinf_fail(SPINF_E_ARG, "gdn: too many units");
    hipLaunchKernelGGL(gdn_forest_kernel, dim3((unsigned)(p.n_seg * p.hv)), dim3(256), 0, stream, p);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return spinf_fail(SPINF_E_HIP, "gdn: launch: %s", hipGetErrorString(e));
    return SPINF_OK;
}
