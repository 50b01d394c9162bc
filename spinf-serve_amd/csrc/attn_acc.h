// Pieces shared by the attention kernels that keep their output accumulators in fixed accumulation registers (tree_attn_ring.hip,
// tree_attn_pipe.hip): the accumulators and the MFMAs on them as inline assembly, a wave's queries and output rows, and the barrier-paced
// pass over single items that both end in.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "attn_kernels.h"
#include "attn_ring_io.h"

namespace {

constexpr int MAX_SLOT = 4;         // tile ring depth (32-key tiles): 4, at head dim 512 (69 KB a tile) 2
constexpr int SROW = 64 + 16;       // output staging: 32 rows x 32 head dims, 80-byte rows

__device__ __forceinline__ int lds_load(const int* p) { return __hip_atomic_load(p, __ATOMIC_ACQUIRE, __HIP_MEMORY_SCOPE_WORKGROUP); }
// plain (non-atomic) reads of words other waves write, as LDS instructions: a volatile access through a generic pointer becomes a
// flat load, which counts against the tile requests in flight
typedef __attribute__((ext_vector_type(4))) int i32x4;
__device__ __forceinline__ int lds_peek(const int* p) { return *(const volatile __attribute__((address_space(3))) int*)(const __attribute__((address_space(3))) void*)p; }
__device__ __forceinline__ i32x4 lds_peek4(const int* p) {
    return *(const volatile __attribute__((address_space(3))) i32x4*)(const __attribute__((address_space(3))) void*)p;
}
__device__ __forceinline__ void lds_store(int* p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP); }


// ---- O^T accumulators in fixed accumulation registers.
// The 32 rows x D output accumulators of a wave live in a[0 : D/2 - 1] and are touched by inline assembly only: tile d (32
// head dims) is a[16 d : 16 d + 15].  The compiler never sees them as values: as values they go through the merge points of
// the tile loop (a wave either computes a tile or skips it), and the register allocator then keeps copies of them and spills
// the queries.  The file is compiled with -amdgpu-spill-vgpr-to-agpr=0 and contains no MFMA builtin, so nothing else ever
// uses an accumulation register.  The hazards the compiler would take care of are handled here: a full s_nop before the
// accumulators are read back (MFMA result -> v_accvgpr_read) and after they are zeroed (v_accvgpr_write -> MFMA srcC).
#define ACC_CLOB(b) "a" #b
#define ACC16_CLOBBERS(b0, b1, b2, b3, b4, b5, b6, b7, b8, b9, b10, b11, b12, b13, b14, b15) \
    ACC_CLOB(b0), ACC_CLOB(b1), ACC_CLOB(b2), ACC_CLOB(b3), ACC_CLOB(b4), ACC_CLOB(b5), ACC_CLOB(b6), ACC_CLOB(b7), ACC_CLOB(b8), ACC_CLOB(b9), \
        ACC_CLOB(b10), ACC_CLOB(b11), ACC_CLOB(b12), ACC_CLOB(b13), ACC_CLOB(b14), ACC_CLOB(b15)

#define ACC_TILE_OPS(DT, LO, HI, C0, C1, C2, C3, C4, C5, C6, C7, C8, C9, C10, C11, C12, C13, C14, C15)                                                 \
    if constexpr (TILE == DT) {                                                                                                                        \
        if constexpr (OP == 0)                                                                                                                         \
            asm volatile("v_mfma_f32_32x32x16_bf16 a[" #LO ":" #HI "], %0, %1, a[" #LO ":" #HI "]" ::"v"(a), "v"(b)                                    \
                         : ACC16_CLOBBERS(C0, C1, C2, C3, C4, C5, C6, C7, C8, C9, C10, C11, C12, C13, C14, C15));                                     \
        else if constexpr (OP == 4)                                                                                                                    \
            asm volatile("v_mfma_f32_32x32x16_bf16 a[" #LO ":" #HI "], %0, %1, 0" ::"v"(a), "v"(b)                                                     \
                         : ACC16_CLOBBERS(C0, C1, C2, C3, C4, C5, C6, C7, C8, C9, C10, C11, C12, C13, C14, C15));                                     \
        else if constexpr (OP == 1)                                                                                                                    \
            asm volatile("v_accvgpr_write_b32 a" #C0 ", 0\n\tv_accvgpr_write_b32 a" #C1 ", 0\n\tv_accvgpr_write_b32 a" #C2 ", 0\n\tv_accvgpr_write_b32 a" #C3 ", 0\n\t"   \
                         "v_accvgpr_write_b32 a" #C4 ", 0\n\tv_accvgpr_write_b32 a" #C5 ", 0\n\tv_accvgpr_write_b32 a" #C6 ", 0\n\tv_accvgpr_write_b32 a" #C7 ", 0\n\t"   \
                         "v_accvgpr_write_b32 a" #C8 ", 0\n\tv_accvgpr_write_b32 a" #C9 ", 0\n\tv_accvgpr_write_b32 a" #C10 ", 0\n\tv_accvgpr_write_b32 a" #C11 ", 0\n\t" \
                         "v_accvgpr_write_b32 a" #C12 ", 0\n\tv_accvgpr_write_b32 a" #C13 ", 0\n\tv_accvgpr_write_b32 a" #C14 ", 0\n\tv_accvgpr_write_b32 a" #C15 ", 0" :: \
                             : ACC16_CLOBBERS(C0, C1, C2, C3, C4, C5, C6, C7, C8, C9, C10, C11, C12, C13, C14, C15));                                 \
        else if constexpr (OP == 3)                                                                                                                    \
            asm volatile("v_accvgpr_write_b32 a" #C0 ", %0\n\tv_accvgpr_write_b32 a" #C1 ", %1\n\tv_accvgpr_write_b32 a" #C2 ", %2\n\tv_accvgpr_write_b32 a" #C3 ", %3\n\t"     \
                         "v_accvgpr_write_b32 a" #C4 ", %4\n\tv_accvgpr_write_b32 a" #C5 ", %5\n\tv_accvgpr_write_b32 a" #C6 ", %6\n\tv_accvgpr_write_b32 a" #C7 ", %7\n\t"     \
                         "v_accvgpr_write_b32 a" #C8 ", %8\n\tv_accvgpr_write_b32 a" #C9 ", %9\n\tv_accvgpr_write_b32 a" #C10 ", %10\n\tv_accvgpr_write_b32 a" #C11 ", %11\n\t" \
                         "v_accvgpr_write_b32 a" #C12 ", %12\n\tv_accvgpr_write_b32 a" #C13 ", %13\n\tv_accvgpr_write_b32 a" #C14 ", %14\n\tv_accvgpr_write_b32 a" #C15 ", %15" :: \
                             "v"(r[0]), "v"(r[1]), "v"(r[2]), "v"(r[3]), "v"(r[4]), "v"(r[5]), "v"(r[6]), "v"(r[7]), "v"(r[8]), "v"(r[9]), "v"(r[10]),            \
                         "v"(r[11]), "v"(r[12]), "v"(r[13]), "v"(r[14]), "v"(r[15])                                                                      \
                         : ACC16_CLOBBERS(C0, C1, C2, C3, C4, C5, C6, C7, C8, C9, C10, C11, C12, C13, C14, C15));                                     \
        else                                                                                                                                           \
            asm volatile("v_accvgpr_read_b32 %0, a" #C0 "\n\tv_accvgpr_read_b32 %1, a" #C1 "\n\tv_accvgpr_read_b32 %2, a" #C2 "\n\tv_accvgpr_read_b32 %3, a" #C3 "\n\t"     \
                         "v_accvgpr_read_b32 %4, a" #C4 "\n\tv_accvgpr_read_b32 %5, a" #C5 "\n\tv_accvgpr_read_b32 %6, a" #C6 "\n\tv_accvgpr_read_b32 %7, a" #C7 "\n\t"     \
                         "v_accvgpr_read_b32 %8, a" #C8 "\n\tv_accvgpr_read_b32 %9, a" #C9 "\n\tv_accvgpr_read_b32 %10, a" #C10 "\n\tv_accvgpr_read_b32 %11, a" #C11 "\n\t" \
                         "v_accvgpr_read_b32 %12, a" #C12 "\n\tv_accvgpr_read_b32 %13, a" #C13 "\n\tv_accvgpr_read_b32 %14, a" #C14 "\n\tv_accvgpr_read_b32 %15, a" #C15     \
                         : "=v"(r[0]), "=v"(r[1]), "=v"(r[2]), "=v"(r[3]), "=v"(r[4]), "=v"(r[5]), "=v"(r[6]), "=v"(r[7]), "=v"(r[8]), "=v"(r[9]), "=v"(r[10]),      \
                           "=v"(r[11]), "=v"(r[12]), "=v"(r[13]), "=v"(r[14]), "=v"(r[15]));                                                        \
    }

// OP 0: acc[TILE] += a * b (MFMA 32x32x16 bf16); OP 1: acc[TILE] = 0; OP 2: r[0..15] = acc[TILE]; OP 3: acc[TILE] = r[0..15]; OP 4: acc[TILE] = a * b
template <int TILE, int OP>
__device__ __forceinline__ void acc_op(const bf16x8 a, const bf16x8 b, float (&r)[16]) {
    ACC_TILE_OPS(0, 0, 15, 0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14, 15)
    ACC_TILE_OPS(1, 16, 31, 16, 17, 18, 19, 20, 21, 22, 23, 24, 25, 26, 27, 28, 29, 30, 31)
    ACC_TILE_OPS(2, 32, 47, 32, 33, 34, 35, 36, 37, 38, 39, 40, 41, 42, 43, 44, 45, 46, 47)
    ACC_TILE_OPS(3, 48, 63, 48, 49, 50, 51, 52, 53, 54, 55, 56, 57, 58, 59, 60, 61, 62, 63)
    ACC_TILE_OPS(4, 64, 79, 64, 65, 66, 67, 68, 69, 70, 71, 72, 73, 74, 75, 76, 77, 78, 79)
    ACC_TILE_OPS(5, 80, 95, 80, 81, 82, 83, 84, 85, 86, 87, 88, 89, 90, 91, 92, 93, 94, 95)
    ACC_TILE_OPS(6, 96, 111, 96, 97, 98, 99, 100, 101, 102, 103, 104, 105, 106, 107, 108, 109, 110, 111)
    ACC_TILE_OPS(7, 112, 127, 112, 113, 114, 115, 116, 117, 118, 119, 120, 121, 122, 123, 124, 125, 126, 127)
    ACC_TILE_OPS(8, 128, 143, 128, 129, 130, 131, 132, 133, 134, 135, 136, 137, 138, 139, 140, 141, 142, 143)
    ACC_TILE_OPS(9, 144, 159, 144, 145, 146, 147, 148, 149, 150, 151, 152, 153, 154, 155, 156, 157, 158, 159)
    ACC_TILE_OPS(10, 160, 175, 160, 161, 162, 163, 164, 165, 166, 167, 168, 169, 170, 171, 172, 173, 174, 175)
    ACC_TILE_OPS(11, 176, 191, 176, 177, 178, 179, 180, 181, 182, 183, 184, 185, 186, 187, 188, 189, 190, 191)
    ACC_TILE_OPS(12, 192, 207, 192, 193, 194, 195, 196, 197, 198, 199, 200, 201, 202, 203, 204, 205, 206, 207)
    ACC_TILE_OPS(13, 208, 223, 208, 209, 210, 211, 212, 213, 214, 215, 216, 217, 218, 219, 220, 221, 222, 223)
    ACC_TILE_OPS(14, 224, 239, 224, 225, 226, 227, 228, 229, 230, 231, 232, 233, 234, 235, 236, 237, 238, 239)
    ACC_TILE_OPS(15, 240, 255, 240, 241, 242, 243, 244, 245, 246, 247, 248, 249, 250, 251, 252, 253, 254, 255)
}
template <int TILE>
__device__ __forceinline__ void acc_mfma(const bf16x8 a, const bf16x8 b) {
    float unused[16];
    acc_op<TILE, 0>(a, b, unused);
}
template <int TILE>
__device__ __forceinline__ void acc_mfma_init(const bf16x8 a, const bf16x8 b) {   // the first product: no zeroing ahead of it
    float unused[16];
    acc_op<TILE, 4>(a, b, unused);
}
template <int N, int TILE = 0>
__device__ __forceinline__ void acc_zero() {
    if constexpr (TILE < N) {
        float unused[16];
        acc_op<TILE, 1>(bf16x8{}, bf16x8{}, unused);
        acc_zero<N, TILE + 1>();
    } else {
        asm volatile("s_nop 3" ::: "memory");   // v_accvgpr_write -> MFMA srcC
    }
}
template <int TILE>
__device__ __forceinline__ void acc_read(float (&r)[16]) {
    acc_op<TILE, 2>(bf16x8{}, bf16x8{}, r);
}
// acc[0 .. N-1] *= alpha (the exact recomputation's rescaling; the caller brackets it with the wait states that acc_read and
// acc_zero need)
template <int N, int TILE = 0>
__device__ __forceinline__ void acc_scale(const float alpha) {
    if constexpr (TILE < N) {
        float r[16];
        acc_op<TILE, 2>(bf16x8{}, bf16x8{}, r);
#pragma unroll
        for (int i = 0; i < 16; i++) r[i] *= alpha;
        acc_op<TILE, 3>(bf16x8{}, bf16x8{}, r);
        acc_scale<N, TILE + 1>(alpha);
    }
}
// S^T chain on ordinary registers, as assembly as well (a kernel that mixes MFMA builtins with the fixed accumulation registers
// above would let the compiler pick accumulation registers of its own for them)
__device__ __forceinline__ void qk_first(f32x16& sa, const bf16x8 k, const bf16x8 q) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(sa) : "v"(k), "v"(q));
}
__device__ __forceinline__ void qk_next(f32x16& sa, const bf16x8 k, const bf16x8 q) {
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(sa) : "v"(k), "v"(q));
}
__device__ __forceinline__ void qk_last(f32x16& sa, const bf16x8 k, const bf16x8 q) {   // + the wait states before the vector ALU reads the result
    asm volatile("v_mfma_f32_32x32x16_bf16 %0, %1, %2, %0\n\ts_nop 15" : "+v"(sa) : "v"(k), "v"(q));
}

template <int N, int F = 0, class Fn>
__device__ __forceinline__ void pv_steps(Fn& fn) {
    if constexpr (F < N) {
        fn(std::integral_constant<int, F>{});
        pv_steps<N, F + 1>(fn);
    }
}

// A wave's place in the workgroup: four row groups x HPI heads of the item.
template <int D>
struct RingShape {
    static constexpr int TK = D == 128 ? 64 : 32;    // keys per tile: at head dim 128 a 32-key tile is too little work per ring slot
    static constexpr int NSUB = TK / 32;             // 32-key blocks per tile
    static constexpr int NW = D == 512 ? 4 : 8;      // waves: four row groups x HPI heads of the item
    static constexpr int HPI = NW / 4;
    static constexpr int NSLOT = D == 512 ? 2 : MAX_SLOT;
    static constexpr int NS = D / 16;     // contraction steps of K Q^T
    static constexpr int NDT = D / 32;    // 32-wide slices of the head dimension in O^T
    static constexpr int NVF = 2 * NDT;   // V^T fragments of one 32-key block
};

// the queries of rows 32 wr .. of query tile tz & 0xfffff, head (tz >> 20) * HPI + wh, as B operands of K Q^T; art / pos of the wave's rows
template <int D, bool WIN>
__device__ __forceinline__ void ring_load_q(const AttnParams& p, const int wr, const int wh, const int tz, bf16x8 (&qf)[D / 16], int& art_q, int& pos_q) {
    const int lane = fresh_lane_id();
    const int tok = (tz & 0xfffff) * SPINF_QTILE + 32 * wr + (lane & 31);
    const int tok_c = tok < p.n ? tok : p.n - 1;
    const int h = (int)((unsigned)tz >> 20) * RingShape<D>::HPI + wh;
    const __bf16* qp = p.q + (long)tok_c * p.q_tok + (long)h * p.q_head + 8 * (lane >> 5);
#pragma unroll
    for (int s = 0; s < D / 16; s++) qf[s] = *(const bf16x8*)(qp + 16 * s);
    art_q = tok < p.n ? p.art[tok_c] : -1;
    pos_q = WIN ? p.pos[tok_c] : 0;
}

// normalise O^T and store it as rows: 32 rows x 32 head dims at a time through the wave's own LDS slice `stage`, 16-byte pieces out
// (pieces of 8 bytes straight from the registers were measured slower: twice the requests for the same bytes)
// FULL: all 32 rows lie inside the stream (no row is tested, so the number of stores is known)
template <int D, bool FULL = false>
__device__ __forceinline__ void ring_store_rows(const AttnParams& p, const int wr, const int wh, char* const stage, const int tz, const float l) {
    constexpr int NDT = D / 32;
    const int lane = fresh_lane_id(), m = lane & 31, g = lane >> 5;
    const int tok0 = (tz & 0xfffff) * SPINF_QTILE + 32 * wr;
    const int h = (int)((unsigned)tz >> 20) * RingShape<D>::HPI + wh;
    const float inv = 1.0f / lane32_sum(l);
    __bf16* ob = p.o + (long)h * p.o_head;
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
            if (FULL || tok0 + row < p.n) *(bf16x8*)(ob + (long)(tok0 + row) * p.o_tok + 32 * dt + col * 8) = val[jj];
        }
    };
    put(std::integral_constant<int, 0>{});
    pv_steps<NDT>(round);
}

// ---- after the list: the barrier-paced pass over single items.  One tile at a time into slot 0 of the ring, a workgroup barrier on
// either side of its request, nothing overlapped, no spin anywhere.  Every workgroup of the ring kernel ends in it (normally with
// nothing to do).  Two uses:
//   * the exact recomputation.  Items in which some row met scores too far above its reference (normally none) are done again by the
//     workgroup that owns them: classic online softmax over the same 32-key blocks in the same order (the reference is raised, and
//     the accumulators rescaled, whenever a block maximum exceeds it by more than TAU_LAZY), the arithmetic of tree_attn_exact_kernel
//     (tree_attn.hip) step for step, so the two give the same bits.  Whether an item comes here depends on its own rows only, so a
//     job's output does not depend on what it is packed with.
//   * the landing after an abort.  If a wave gave up a wait, every wave has left the ring; the items li .. hi - 1 of the list (from
//     the first one that some wave had not completed) are then computed here with the ring pass's own arithmetic (fixed reference, no
//     rescaling: the same bits), handing items to the exact recomputation by the same rule.  An abort costs time, never rows.
// Every wave of the workgroup calls it together: li < hi only after an abort; *sy_nredo = entries of the workgroup's redo list
// p.redo[lo ..]; *sy_vote = 0.
template <int D, bool WIN>
__device__ __forceinline__ void ring_paced_pass(const AttnParams& p, char* const ring, char* const stage_all, int* const sy_nredo, int* const sy_vote,
                                                const int lo, const int hi, int li) {
    using S = RingShape<D>;
    constexpr int TK = S::TK, HPI = S::HPI, NS = S::NS, NDT = S::NDT, NVF = S::NVF;
    using G = TileGeo<D, TK, D>;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wh = w >> 2, wr = wh ? 3 - (w & 3) : (w & 3);   // as Lane (attn_kernels.h)
    char* const stage = stage_all + w * 32 * SROW;
    bf16x8 qf[NS];
    int art_q = -1, pos_q = 0;
    int ri = 0;   // next entry of the redo list
#pragma unroll 1
    while (true) {
        const bool exact = li >= hi;   // first the landing's items, if any, then the recomputations
        int idx = li;
        if (exact) {
            if (ri >= __builtin_amdgcn_readfirstlane(lds_load(sy_nredo))) break;
            idx = __builtin_amdgcn_readfirstlane(__hip_atomic_load(&p.redo[lo + ri], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        }
        const int4 itv = p.items[idx];
        const int it_t = __builtin_amdgcn_readfirstlane(itv.x), it_e0 = __builtin_amdgcn_readfirstlane(itv.y), it_z = __builtin_amdgcn_readfirstlane(itv.z);
        const int ne = it_z & 0xfffff;
        const int tz = it_t | (int)((unsigned)it_z >> 20 << 20);
        const int kvh = (int)((unsigned)it_z >> 20) * HPI / p.group;
        ring_load_q<D, WIN>(p, wr, wh, tz, qf, art_q, pos_q);
        float M = -INFINITY, l = 0.f, Mf = -INFINITY;
        bool viol = false;   // (in the exact recomputation too: the ring pass's test on its numbers says which waves' rows are done again)
        acc_zero<NDT>();
#pragma unroll 1
        for (int e = 0; e < ne; e++) {
            const int kt = __builtin_amdgcn_readfirstlane(p.kv_idx[it_e0 + e]);
            const unsigned bits = (unsigned)__builtin_amdgcn_readfirstlane((int)p.kv_bits[it_e0 + e]);
            __syncthreads();   // everyone is through with the slot
            if (w == 0) {
                using GK = Geo<D, TK>;
                const int lane = fresh_lane_id();
                const unsigned lane_k = (unsigned)((lane / GK::CPR) * GK::NREG * p.k_tok * 2 + (lane % GK::CPR) * 16);
                const unsigned lane_v = (unsigned)((lane / GK::CPR) * GK::NREG * p.v_tok * 2 + (lane % GK::CPR) * 16);
                issue_tile_wave<D, WIN, TK>(p, lds_addr(ring), kt, kvh, 0, lane, lane_k, lane_v);
            }
            __builtin_amdgcn_s_waitcnt(0x0f70);   // the tile has landed (and this wave's queries)
            __syncthreads();
#pragma unroll 1
            for (int sub = 0; sub < S::NSUB; sub++) {   // the tile's 32-key blocks
            if (!((bits >> (2 * wr + sub)) & 1u)) continue;   // (wave-uniform; the barriers above are passed by every wave)
            const int ln = fresh_lane_id();
            const char* krow = ring + G::K::k_off(ln & 31) + 16 * (ln >> 5) + sub * G::KSUB;
            const char* vrow = ring + G::KTILEB + G::V::v_off(4 * (ln >> 5) + ((ln >> 2) & 3)) + 32 * ((ln >> 4) & 1) + 8 * (ln & 3) + sub * G::VSUB;
            // (the scheduling barriers keep the phases apart.  The MFMAs are assembly, which the compiler's hazard recogniser does
            // not look into: left to interleave the softmax of the block's second half with the P V products of the first, it
            // put the conversion that writes a P fragment directly in front of the MFMA that reads it, and an MFMA that issues in
            // the cycle after a vector write of its A / B registers reads the old values (spinf_diag_mfma_hazard measures it).
            // With the phases apart, V fragment reads lie between the conversions and the first MFMA; the build scans the
            // generated assembly for the pattern.)
            f32x16 sa;
            __builtin_amdgcn_sched_barrier(0);
            auto score = [&](auto x_c) __attribute__((always_inline)) {
                constexpr int x = decltype(x_c)::value;
                const bf16x8 kf = *(const bf16x8*)(krow + 32 * x);
                if (x == 0) qk_first(sa, kf, qf[x]);
                else if (x == NS - 1) qk_last(sa, kf, qf[x]);
                else qk_next(sa, kf, qf[x]);
            };
            pv_steps<NS>(score);
            __builtin_amdgcn_sched_barrier(0);
            if ((bits >> (8 + 2 * wr + sub)) & 1u) {
                f32x16 sm[1] = {sa};
                const int tok = (tz & 0xfffff) * SPINF_QTILE + 32 * wr + (ln & 31);
                apply_mask<1, WIN, 0, TK>(sm, (const int*)(ring + G::KTILEB + G::VTILEB), kt, sub, ln >> 5, tok, art_q, pos_q, p.window);
                sa = sm[0];
            }
            __builtin_amdgcn_sched_barrier(0);
            bf16x8 pb[2];
            // (each branch is written out in full, statement for statement as in tree_attn_exact_kernel and in the ring loop: the
            // compiler contracts `l *= alpha; l += sum` into one fused multiply-add where it sees them together, and the bits follow)
            if (exact) {
                float mx = sa[0];
#pragma unroll
                for (int i2 = 1; i2 < 16; i2++) mx = fmaxf(mx, sa[i2]);
                mx = lane32_max(mx);
                const float tm = mx * p.c;
                Mf = Mf == -INFINITY ? tm : Mf;
                const float msf = Mf == -INFINITY ? 0.f : Mf;
                float sumf = 0.f;
#pragma unroll
                for (int i2 = 0; i2 < 16; i2++) sumf += __builtin_amdgcn_exp2f(__builtin_fmaf(sa[i2], p.c, -msf));
                viol = viol | !(sumf <= VIOL_SUM);
                const bool up = tm > M + TAU_LAZY;
                const float mn = up ? tm : M;
                const float alpha = up ? __builtin_amdgcn_exp2f(M - mn) : 1.0f;
                if (__builtin_amdgcn_ballot_w64(up && M != -INFINITY) != 0) {   // rows without a key so far hold zeros
                    asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");   // the last MFMAs' results -> v_accvgpr_read
                    acc_scale<NDT>(alpha);
                    asm volatile("s_nop 3" ::: "memory");                // v_accvgpr_write -> MFMA srcC
                }
                l *= alpha;
                M = mn;
                const float ms = mn == -INFINITY ? 0.f : mn;
                float sum = 0.f;
#pragma unroll
                for (int i2 = 0; i2 < 16; i2++) {
                    const float pr = __builtin_amdgcn_exp2f(__builtin_fmaf(sa[i2], p.c, -ms));
                    sum += pr;
                    pb[i2 >> 3][i2 & 7] = (__bf16)pr;
                }
                l += sum;
            } else {   // the ring pass's arithmetic: the row's reference is the maximum of the first block it sees a key in
                const bool first = M == -INFINITY;
                if (__builtin_amdgcn_ballot_w64(first) != 0) {
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
            __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0): the softmax phase ends here, the waits below are for V fragments only
            __builtin_amdgcn_sched_barrier(0);
            auto step = [&](auto f_c) __attribute__((always_inline)) {
                constexpr int f = decltype(f_c)::value;
                const char* vp = vrow + G::V::v_off(16 * (f / NDT)) + 64 * (f % NDT);
                const s16x4 lo4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)vp);
                const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(vp + G::V::v_off(8)));
                const bf16x8 a = __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo4, hi4, 0, 1, 2, 3, 4, 5, 6, 7));
                acc_mfma<f % NDT>(a, pb[f / NDT]);
                __builtin_amdgcn_sched_barrier(0);
            };
            pv_steps<NVF>(step);
            }
        }
        const bool far = __builtin_amdgcn_ballot_w64(viol) != 0;   // scores ranged too widely somewhere in these 32 rows: done again, exactly
        if (!exact && far) {
            if (fresh_lane_id() == 0) __hip_atomic_store(sy_vote, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        } else if (!exact || far) {   // (the item's other rows keep the fast pass's output)
            ring_store_rows<D>(p, wr, wh, stage, tz, l);
        }
        if (exact) {
            ri++;
            continue;
        }
        __syncthreads();
        if (threadIdx.x == 0 && lds_load(sy_vote) != 0) {   // (a wave may have handed the item over before the abort already)
            const int k = lds_load(sy_nredo);
            bool listed = false;
            for (int r = 0; r < k; r++) listed = listed || __hip_atomic_load(&p.redo[lo + r], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == idx;
            if (!listed) {
                __hip_atomic_store(&p.redo[lo + k], idx, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                lds_store(sy_nredo, k + 1);
            }
            lds_store(sy_vote, 0);
        }
        __syncthreads();
        li++;
    }
    if (ri > 0 && threadIdx.x == 0) atomicAdd(&p.counters[NLIST + 3], ri);   // running total, for spinf_attn_exact_items
    __builtin_amdgcn_s_waitcnt(0x0f70);
}

}  // namespace
