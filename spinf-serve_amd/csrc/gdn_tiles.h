// Shared pieces of the two Gated DeltaNet kernels (gdn.hip: short segments, gdn_chunk.hip: long segments): the launch
// parameters and the 16x16 MFMA tile helpers.
//
// Both kernels keep the state slice of a wave in fp32 accumulator layout (lane = value column, 4 consecutive key rows per
// 16x16 tile) and use it in place as the B operand of v_mfma_f32_16x16x32_bf16: two tiles side by side supply the 8
// contraction slots of a lane, slot (lane/16, j) = row 4 (lane/16) + j of the first tile for j < 4 and of the second for
// j >= 4.  The other operand is read in the same permuted order, so the state never moves, it is only rounded to bf16 on
// the way into the matrix core.  The same holds for every intermediate that one product leaves in accumulator layout and the
// next one contracts over (tokens for V' and P^T, key columns for W^T).
#pragma once
#include <hip/hip_runtime.h>

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(4))) short s16x4;
typedef __attribute__((ext_vector_type(4))) float f32x4;

struct GdnParams {
    const __bf16* q; const __bf16* k; const __bf16* v; const float* g; const __bf16* beta; __bf16* o;
    long q_tok, v_tok, g_tok, o_tok;
    int h, hv, dk, dv; float scale;
    const long* cu; const long* idx; long n_seg;
    const float* h0; const long* h0_idx; float* ht; const long* ht_idx;
    int run;   // segments per workgroup of the recurrent entry point's kernel (set by its launcher)
};

namespace gdn_tiles {

// C[m][n] += sum_k A[m][k] B[k][n], 16 x 16 x 32: lane l gives A[l%16][8 (l/16) ..+7] and B[8 (l/16) ..+7][l%16] and holds
// C[4 (l/16) ..+3][l%16].
__device__ __forceinline__ f32x4 mfma32(bf16x8 a, bf16x8 b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
// 16 x 16 x 16: 4 contraction slots per lane, 4 (l/16) ..+3.
__device__ __forceinline__ f32x4 mfma16(bf16x4 a, bf16x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, a), __builtin_bit_cast(s16x4, b), c, 0, 0, 0);
}
// fp32 16 x 16 x 4: lane l gives A[l%16][l/16] and B[l/16][l%16].
__device__ __forceinline__ f32x4 mfma4(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// Operand whose contraction index is the ROW index of a row-major bf16 LDS tile: the lane gets column col0 + lane%16 of
// rows row0 + 4 (lane/16) .. +3 (each group of 16 lanes transposes a 4 x 16 block).
__device__ __forceinline__ bf16x4 frag_tr4(const __bf16* base, int stride, int row0, int col0, int lane) {
    const int t = lane & 15;
    const __bf16* p = base + (row0 + 4 * (lane >> 4) + (t >> 2)) * stride + col0 + 4 * (t & 3);
    return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p));
}
__device__ __forceinline__ bf16x8 join(bf16x4 lo, bf16x4 hi) { return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7); }
__device__ __forceinline__ bf16x4 round4(f32x4 x) {
    bf16x4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = (__bf16)x[i];
    return r;
}
__device__ __forceinline__ f32x4 zero4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }
// Inclusive prefix sum inside every row of 16 lanes (zero shifted in).
__device__ __forceinline__ float row_prefix_sum(float x) {
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x111, 0xf, 0xf, true));   // row_shr:1
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x112, 0xf, 0xf, true));   // row_shr:2
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x114, 0xf, 0xf, true));   // row_shr:4
    x += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), 0x118, 0xf, 0xf, true));   // row_shr:8
    return x;
}
// Row c of (I - A)^-1 for a strictly lower triangular 16 x 16 block A (row stride lda floats, in LDS), c = this lane's row:
// T = I + T A, so t[j] = [j == c] + sum_{m > j} t[m] A[m][j]; the highest m goes first and every step updates all j < m.
// PRELOAD: read A's rows in two batches (rows 15..8, then 7..1) ahead of the steps that use them instead of row by row: the
// steps form a chain of 15 dependent multiply-adds, and an LDS round trip inside every link is what such a solve otherwise
// waits for.
template <bool PRELOAD>
__device__ __forceinline__ void unit_lower_inverse_row(const float* A, int lda, int c, float (&t)[16]) {
    f32x4 a[16][4];
#pragma unroll
    for (int j = 0; j < 16; j++) t[j] = (j == c) ? 1.f : 0.f;
#pragma unroll
    for (int half = 1; half >= 0; half--) {
        if (PRELOAD) {
#pragma unroll
            for (int m = 8 * half + 7; m >= 8 * half; m--)
#pragma unroll
                for (int j4 = 0; 4 * j4 < m; j4++) a[m][j4] = *(const f32x4*)(A + m * lda + 4 * j4);
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int m = 8 * half + 7; m >= 8 * half; m--) {
#pragma unroll
            for (int j4 = 0; 4 * j4 < m; j4++) {
                const f32x4 am = PRELOAD ? a[m][j4] : *(const f32x4*)(A + m * lda + 4 * j4);
#pragma unroll
                for (int jj = 0; jj < 4; jj++)
                    if (4 * j4 + jj < m) t[4 * j4 + jj] = __builtin_fmaf(t[m], am[jj], t[4 * j4 + jj]);
            }
        }
        if (PRELOAD) __builtin_amdgcn_sched_barrier(0);
    }
}
// t[4 q + r], r = 0..3, without indexing registers by a lane-dependent value
__device__ __forceinline__ f32x4 pick4(const float (&t)[16], int q) {
    f32x4 r;
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] = q == 0 ? t[i] : q == 1 ? t[4 + i] : q == 2 ? t[8 + i] : t[12 + i];
    return r;
}
// Orders a wave's LDS writes before its later LDS reads for the compiler; the hardware runs one wave's LDS operations in order.
__device__ __forceinline__ void wave_lds_order() { asm volatile("" ::: "memory"); }
// Workgroup barrier for LDS traffic only: waits for this wave's LDS operations, not for its global loads (__syncthreads()
// carries a fence in front of which the compiler drains every load in flight, prefetches included).
__device__ __forceinline__ void lds_barrier() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(0xc07f);   // lgkmcnt(0)
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// element offset of a row: one 32 x 32 -> 64 bit multiply (rows and strides are below 2^31; the launch checks the strides)
__device__ __forceinline__ long row_offset(int row, long stride) { return (long)((unsigned long)(unsigned)row * (unsigned)stride); }
__device__ __forceinline__ bf16x4 zero_bf4() {
    bf16x4 z;
#pragma unroll
    for (int r = 0; r < 4; r++) z[r] = (__bf16)0.f;
    return z;
}

// ---- what the chunk kernel (gdn_chunk.hip) and the forest kernel (gdn_forest.hip) do alike with their 32 tokens
constexpr int LP = 40;         // row stride of the token x token bf16 tiles (P, T diag(beta), ..)
constexpr int LA = 36;         // row stride (floats) of A
constexpr int LX = 20;         // row stride (floats) of the 16 x 16 blocks of T and of the merge scratch
constexpr int LO = 32 + 4;     // row stride (elements) of a wave's transposed output tile [32 values][32 tokens]; 64-byte rows
                               // would put the 8-byte stores of 16 lanes into four banks (32 clocks per store instead of 7)

// T = (I - A)^-1 by one wave: rows of the diagonal blocks by substitution in registers (lane groups 0 and 2 the upper-left block, 1 and 3
// the lower-right one, in the same instructions), then the lower-left block T_lo = T_11 A_lo T_00, computed transposed
// (T_lo^T = T_00^T (A_lo^T T_11^T)) so that the lane again holds a row; apart: the two tiles do not see each other, T_lo = 0.  Leaves
// T diag(beta) in Tus as bf16, tile by tile.  Ts (T_00 in rows 0..15, T_11 in 16..31) and Xs are scratch.  The others wait for this
// wave: it goes first.  c = lane % 16, q4 = lane / 16; by reference, which leaves their reading where the kernels' own code would (by value
// the kernels of 168 registers spill).  MERGE_FIRST: the diagonal blocks are stored behind T_lo (the forest kernel: a layer's scans
// 210.4 -> 209.5 us over a stream of tries; the chunk kernels lose 0.5 - 1 % that way).
template <bool PRELOAD, bool MERGE_FIRST>
__device__ __forceinline__ void solve_tile(const float* As, const float* Bs, float* Ts, float* Xs, __bf16* Tus, const int& c, const int& q4, const bool& apart) {
    __builtin_amdgcn_s_setprio(3);
    float t[16];
    const int blk = q4 & 1;
    unit_lower_inverse_row<PRELOAD>(As + blk * (16 * LA + 16), LA, c, t);
    // the rows pass through LDS to reach the lanes in operand order (row c, columns 4 q4 ..+3)
#pragma unroll
    for (int j4 = 0; j4 < 4; j4++) *(f32x4*)(Ts + (16 * blk + c) * LX + 4 * j4) = f32x4{t[4 * j4], t[4 * j4 + 1], t[4 * j4 + 2], t[4 * j4 + 3]};
    wave_lds_order();
    const float* T1s = Ts + 16 * LX;
    const f32x4 B0 = *(const f32x4*)(Bs + 4 * q4), B1 = *(const f32x4*)(Bs + 16 + 4 * q4);
    const f32x4 t00 = *(const f32x4*)(Ts + c * LX + 4 * q4), t11 = *(const f32x4*)(T1s + c * LX + 4 * q4);
    if (!MERGE_FIRST) {
        *(bf16x4*)(Tus + c * LP + 4 * q4) = round4(t00 * B0);
        *(bf16x4*)(Tus + (16 + c) * LP + 16 + 4 * q4) = round4(t11 * B1);
    }
    f32x4 tlo = zero4();
    if (!apart) {
        f32x4 x = zero4();
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++)        // X[j][i] = sum_m A_lo[m][j] T_11[i][m]
            x = mfma4(As[(16 + 4 * s4 + q4) * LA + c], T1s[c * LX + 4 * s4 + q4], x);
#pragma unroll
        for (int r = 0; r < 4; r++) Xs[(4 * q4 + r) * LX + c] = x[r];
        wave_lds_order();
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++)        // T_lo[16 + i][j'] = sum_j T_00[j][j'] X[j][i]
            tlo = mfma4(Ts[(4 * s4 + q4) * LX + c], Xs[(4 * s4 + q4) * LX + c], tlo);
    }
    if (MERGE_FIRST) {
        *(bf16x4*)(Tus + c * LP + 4 * q4) = round4(t00 * B0);
        *(bf16x4*)(Tus + (16 + c) * LP + 16 + 4 * q4) = round4(t11 * B1);
    }
    *(bf16x4*)(Tus + (16 + c) * LP + 4 * q4) = round4(tlo * B0);
    __builtin_amdgcn_s_setprio(0);
}

// A wave's transposed output tile to memory: row i = 16 it + lane % 16, values 8 (lane / 16) ..+7 of the wave's 32, the first of which is column col:
// two transposing reads, one 16-byte store.  Rs: the tensor rows, -1 for none.
__device__ __forceinline__ void store_tile(const __bf16* Ow, const int* Rs, __bf16* out, long o_tok, int col, int c, int q4) {
#pragma unroll
    for (int it = 0; it < 2; it++) {
        const __bf16* op = Ow + (8 * q4 + (c >> 2)) * LO + 16 * it + 4 * (c & 3);
        const bf16x4 lo = __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)op));
        const bf16x4 hi = __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)(op + 4 * LO)));
        const int orow = Rs[16 * it + c];
        if (orow >= 0) *(bf16x8*)(out + row_offset(orow, o_tok) + col + 8 * q4) = join(lo, hi);
    }
}

}  // namespace gdn_tiles
