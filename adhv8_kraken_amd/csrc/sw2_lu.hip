// Tiled band LU: the profile-LU preconditioner (OP BLK) for node blocks of
// any size, up to the reference's default OP BLK 1 -- one LU of the whole
// matrix (solv_blk_set.c:5-33, solv_blk_profile.c:51-79,
// solv_blk_solve.c:5-62).  Nodes keep the reference's order and the LU has
// no pivoting; a multiplier is its entry over the pivot, or over SMALL when
// |pivot| <= SMALL (solv_blk_profile.c:66-71; formed here as the entry times
// the reciprocal, and the updates as fused multiply-adds), and the backward
// substitution divides by the pivot itself (solv_blk_solve.c:50-52).  Entries
// outside a row's profile are zero and stay zero (no fill outside the envelope
// without pivoting), so factoring the band that covers every row's profile
// gives the skyline factors; only the rounding order of the updates differs.
//
// Storage: each band (one node block) in LAPACK band layout, column-major,
// half bandwidth wp = w + TB (w: the pattern's), entry (i, j) at
// off + (wp + i - j) + j (2 wp + 1).  The TB extra diagonals hold zeros during
// the factorisation, so a panel's L block (rows up to TB + w - 1 below its
// first column) and U block are addressed without bounds tests, and after it
// the fill of the off-diagonal tiles scaled by k_tb_scale.  Seen with leading
// dimension 2 wp the band is a column-major dense matrix, so tiles are
// strided blocks.
//
// Factorisation, one launch per panel of TB columns over all bands at once (a
// model's node blocks, or every block of every model of an ensemble):
//   k_tb_step  a workgroup per 64 x 64 tile of the trailing w x w window, which
//              takes (A U~^-1) (L^-1 A) of its row and column of the panel (U~: U
//              with the guarded pivots) on the matrix cores; the workgroup of the
//              first tile, the next panel's diagonal block, goes on to factor
//              it and to invert both factors (lu64).
// k_tb_diag factors the diagonal blocks that no panel comes before.  Where a
// step's tiles are more than the GPU takes at once, every tile's own L and U
// panel would be most of the work: k_tb_panel forms them once a panel, k_tb_update
// the products, k_tb_diag the next diagonal block, with the same operations.  Then
// k_tb_inv forms G_k = U~^-1 L^-1 of every diagonal block and k_tb_scale
// multiplies every off-diagonal tile by its column's, so that the substitutions
// are matrix-vector work in which only a tile's input is serial: k_tb_sweep runs
// both as a dataflow (y_i = x_i - sum (A_ik G_k) y_k, then upwards), k_tb_apply
// the diagonal inverses.
//
// A chain of dependent panels bounds both, so a long block is factored from both
// ends at once: two bands, one of them in reverse order, down to the rows in the
// middle that both reach (at least w of them).  Those belong to the band from the
// start, which adds the other's updates (k_tb_merge) and goes on through them.
// A sweep starts from both ends too, and the shared rows add the two; after them
// the ends are independent again.  Blocks of all models reach their shared rows
// at one launch, so each merges where the others do.
//
// 200 x 100 cells (m 60,903, w 308, 952 panels; from both ends 473 and 6 shared):
// factorisation 10.8 ms (21.1 from one end), both sweeps 1.84 ms (3.58).  A panel
// takes 22.2 us, of which the diagonal block's LU 11.7 (189 cycles per pivot in
// the panel wave, which issues on 150 of them), the tile's three products 3.8 at
// the matrix cores' FP64 rate, the rest load latency and the launch
// (substitution and update in two launches, vector FMAs, LU by readlane
// broadcasts: 9.6 + 21.7 us); a sweep step 1.9 us (a launch per tile: 3.5).
#include <limits.h>

#include <algorithm>
#include <string>
#include <type_traits>
#include <vector>

#include "sw2_ctx.h"
#include "sw2_flow.h"

namespace sw2 {

constexpr int TB = 64;          // tile and panel width (DOFs)
constexpr int NT = 512;         // threads of the factorisation and sweep workgroups (eight waves)

using d4 = double __attribute__((ext_vector_type(4)));

__device__ __forceinline__ size_t tb_idx(const TBand &B, int i, int j) {
    return B.off + (size_t)(B.wp + i - j) + (size_t)j * (2 * B.wp + 1);
}
__device__ __forceinline__ double &tb_at(double *AB, const TBand &B, int i, int j) { return AB[tb_idx(B, i, j)]; }
__device__ __forceinline__ double tb_get(const double *AB, const TBand &B, int i, int j) { return AB[tb_idx(B, i, j)]; }

// lane l's value of v, for a lane index known at compile time or uniform
__device__ __forceinline__ double lane_bcast(double v, int l) {
    const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
    const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
    return __hiloint2double(hi, lo);
}

// D (16 x 16) += X (16 x 4) Y (4 x 16) on the matrix cores: lane l holds
// X[l % 16][l / 16], Y[l / 16][l % 16] and D[l / 16 + 4 r][l % 16], r = 0..3
__device__ __forceinline__ d4 mfma4(double x, double y, d4 d) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(x, y, d, 0, 0, 0);
}

// Band record b in SGPRs at once: the empty asm statement uses every field, so
// the compiler cannot sink the fields' loads past the kernel's first branches
// (one scalar round trip instead of three before the first vector load);
// `flag` (a done flag read beside it) is held the same way.
__device__ __forceinline__ TBand band_rec(const TBand *bands, int b, int flag = 0) {
    const TBand B = bands[b];
    asm volatile("" ::"s"(B.m), "s"(B.w), "s"(B.wp), "s"(B.nt), "s"(B.inst), "s"(B.off), "s"(B.toff), "s"(B.xoff),
                 "s"(B.na), "s"(B.part), "s"(B.rev), "s"(B.mtot), "s"(flag));
    return B;
}

// The panel that a band eliminates at a step: bands of blocks factored from both
// ends reach their shared rows at one step, amax.
__device__ __forceinline__ int panel_at(const TBand &B, int step, int amax) {
    return B.part < 0 ? step : step - (amax - B.na);
}

__device__ __forceinline__ double guarded(double piv) { return fabs(piv) > SMALL ? piv : SMALL; }

// Scaled matrix (diagonal blocks and SELL off-diagonal blocks) into the bands;
// the bands are zeroed before.  Ensembles: nodes of no block (the gaps between
// models) and models outside the mask are skipped.
__global__ void k_tb_load(int N, const int *node_blk, const TBand *bands, int nbot, double *AB, const double *diag,
                          const double *offd, const int *row_ptr, const int *sell_ptr, const int *sell_col,
                          const int *mask) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    if (a >= N) return;
    const int bk = node_blk[a];
    if (bk < 0) return;
    const TBand B = bands[nbot + bk];
    if (mask && !mask[B.inst]) return;
    const TBand Q = bands[max(B.part, 0)];
    // what touches a row past the shared ones belongs to the band from the end
    auto put = [&](int i, int j, double v) {
        if (i < B.m && j < B.m) tb_at(AB, B, i, j) = v;
        else tb_at(AB, Q, B.mtot - 1 - i, B.mtot - 1 - j) = v;
    };
    const int n1 = B.n0 + B.mtot / 3;
    const int ia = 3 * (a - B.n0);
    for (int r = 0; r < 3; r++)
        for (int cc = 0; cc < 3; cc++) put(ia + r, ia + cc, diag[didx9(a, 3 * r + cc)]);
    const size_t q0 = 64 * (size_t)sell_ptr[a >> 6] + (a & 63);
    const int len = row_ptr[a + 1] - row_ptr[a];
    for (int s = 0; s < len; s++) {
        const size_t q = q0 + 64 * (size_t)s;
        const int cn = sell_col[q];
        if (cn < B.n0 || cn >= n1) continue;
        const int jc = 3 * (cn - B.n0);
        for (int r = 0; r < 3; r++)
            for (int cc = 0; cc < 3; cc++) put(ia + r, jc + cc, offd[sell_vidx(q, 3 * r + cc)]);
    }
}

// ---- LU of a 64 x 64 diagonal block with the inverses of its factors ---------
// 16-column panels on single waves, 16 x 16 block products on the matrix cores.
//
// A panel wave's lane holds a row; the wave's four 16-lane rows are the four
// block rows.  The pivot row's broadcast is the DPP operand of the multiply-add
// itself (row_newbcast), so every 16-lane row carries its own copy of the
// panel's diagonal block.  A step's order is fixed by scheduling barriers: the
// next pivot's column first, then its reciprocal's chain in the shadow of the
// other columns, each source of a DPP read at least two instructions old (the
// compiler does not look into the asm; only the first after them needs a s_nop).
#define SW2_FM(D, S) "v_fmac_f64_dpp %" #D ", %" #S ", %[f] row_newbcast:%[p] row_mask:0xf bank_mask:0xf\n\t"
// d[J .. J + NJ) += f * (row P's s[J .. J + NJ)), s another array than d
template <int P, int J, int NJ>
__device__ __forceinline__ void rank1(double *d, const double *s, double f) {
    if constexpr (NJ >= 3) {
        asm(SW2_FM(0, 3) SW2_FM(1, 4) SW2_FM(2, 5)
            : "+v"(d[J]), "+v"(d[J + 1]), "+v"(d[J + 2])
            : "v"(s[J]), "v"(s[J + 1]), "v"(s[J + 2]), [f] "v"(f), [p] "n"(P));
        rank1<P, J + 3, NJ - 3>(d, s, f);
    } else if constexpr (NJ >= 1) {
        asm(SW2_FM(0, 1) : "+v"(d[J]) : "v"(s[J]), [f] "v"(f), [p] "n"(P));
        rank1<P, J + 1, NJ - 1>(d, s, f);
    }
}
// the same within one array: d[j] += f * (row P's d[j])
template <int P, int J, int NJ>
__device__ __forceinline__ void rank1(double *d, double f) {
    if constexpr (NJ >= 3) {
        asm(SW2_FM(0, 0) SW2_FM(1, 1) SW2_FM(2, 2)
            : "+v"(d[J]), "+v"(d[J + 1]), "+v"(d[J + 2]) : [f] "v"(f), [p] "n"(P));
        rank1<P, J + 3, NJ - 3>(d, f);
    } else if constexpr (NJ >= 1) {
        asm(SW2_FM(0, 0) : "+v"(d[J]) : [f] "v"(f), [p] "n"(P));
        rank1<P, J + 1, NJ - 1>(d, f);
    }
}
#undef SW2_FM
#define SW2_ORDER() __builtin_amdgcn_sched_barrier(0)
// row P's d[P] in every lane
template <int P>
__device__ __forceinline__ double pivot_of(const double *d) {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(d[P]), 0x150 + P, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(d[P]), 0x150 + P, 0xf, 0xf, true);
    return __hiloint2double(hi, lo);
}
// its reciprocal from the hardware's estimate r (e = 1 - piv r about 2^-23) by
// one cubic step r (1 + e + e^2), guarded (solv_blk_profile.c:66-71)
__device__ __forceinline__ double pivot_end(double piv, double r, double e2, bool &small) {
    small = !(fabs(piv) > SMALL);
    r = fma(r, e2, r);
    return small ? 1.0 / SMALL : r;
}
__device__ __forceinline__ double pivot_whole(double piv, bool &small) {
    const double r = __builtin_amdgcn_rcp(piv), e = fma(-piv, r, 1.0);
    return pivot_end(piv, r, fma(e, e, e), small);
}
// a <- a U^-1 for the lane's row a (forward substitution with the reciprocal
// guarded pivots), U from the LU of the block whose row the lane holds in d; r:
// pivot P's reciprocal.  Rows of d above the pivot are finished and not read
// again, so no lane is masked.  A finished column of a goes to C.
template <int P>
__device__ __forceinline__ void panel_rows(double (&d)[16], double (&a)[16], double *C, double r, bool &hit) {
    const double nl = -a[P] * r, f = -d[P] * r;
    C[P] = -nl;
    if constexpr (P < 15) {
        constexpr int M = 14 - P;   // columns after the next pivot's
        SW2_ORDER();
        asm volatile("s_nop 1");
        rank1<P, P + 1, 1>(a, d, nl);
        rank1<P, P + 1, 1>(d, f);
        SW2_ORDER();
        const double piv = pivot_of<P + 1>(d);
        const double r0 = __builtin_amdgcn_rcp(piv);
        SW2_ORDER();
        rank1<P, P + 2, M>(a, d, nl);
        SW2_ORDER();
        const double e = fma(-piv, r0, 1.0);
        SW2_ORDER();
        rank1<P, P + 2, M / 2>(d, f);
        SW2_ORDER();
        const double e2 = fma(e, e, e);
        SW2_ORDER();
        rank1<P, P + 2 + M / 2, M - M / 2>(d, f);
        SW2_ORDER();
        bool small;
        const double rn = pivot_end(piv, r0, e2, small);
        hit = hit || small;
        panel_rows<P + 1>(d, a, C, rn, hit);
    }
}
// the LU of the block whose row the lane holds, in place, with the inverse of
// the unit lower factor below the diagonal in the multipliers' place
template <int P>
__device__ __forceinline__ void lower_inverse(double (&d)[16], double r, int row) {
    const double f = row > P ? -d[P] * r : 0.0;
    if (row > P) d[P] = f;
    if constexpr (P < 15) {
        constexpr int M = 14 - P;
        SW2_ORDER();
        asm volatile("s_nop 1");
        rank1<P, P + 1, 1>(d, f);
        SW2_ORDER();
        const double piv = pivot_of<P + 1>(d);
        const double r0 = __builtin_amdgcn_rcp(piv);
        SW2_ORDER();
        rank1<P, 0, P>(d, f);
        rank1<P, P + 2, M / 3>(d, f);
        SW2_ORDER();
        const double e = fma(-piv, r0, 1.0);
        SW2_ORDER();
        rank1<P, P + 2 + M / 3, M / 3>(d, f);
        SW2_ORDER();
        const double e2 = fma(e, e, e);
        SW2_ORDER();
        rank1<P, P + 2 + 2 * (M / 3), M - 2 * (M / 3)>(d, f);
        SW2_ORDER();
        bool small;
        lower_inverse<P + 1>(d, pivot_end(piv, r0, e2, small), row);
    }
}

__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}
// 16 x 16 blocks in LDS, rows of 18: whole rows (16 bytes a lane) and both operand
// layouts of the matrix cores read distinct banks
constexpr int BLD = 18, BS = 16 * BLD;
struct Lu64 {
    double col[2][4][BS];   // block column s, by step parity: its blocks, then those times U_ss^-1
    double row[2][4][BS];   // block row s: its blocks, then L_ss^-1 times those
    double li[BS], ui[BS];  // L_ss^-1, U_ss^-1
    double one[BS];         // the identity
    int hit;
};
__device__ __forceinline__ void blk_put(double *dst, const d4 &v, int lo, int hi) {
#pragma unroll
    for (int r = 0; r < 4; r++) dst[BLD * lo + hi + 4 * r] = v[r];
}
__device__ __forceinline__ d4 blk_get(const double *src, int lo, int hi) {
    d4 v;
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = src[BLD * lo + hi + 4 * r];
    return v;
}
// Eight waves: wave (wi, wj) holds blocks (wi, 2 wj) and (wi, 2 wj + 1) in
// registers, element (row, col) of a block in lane row + 16 (col % 4), register
// col / 4 -- the matrix cores' operand and result layout of the transposed
// product.  Step s, in place:
//   wave 0   C_i = D_is U_ss^-1 for the four block rows (block row s: U_ss^-1
//            itself, from rows of the identity); beside it wave 1 L_ss^-1
//   then     R_j = L_ss^-1 D_sj, a wave each
//   then     D_ij -= C_i R_j, D_is <- -C_i L_ss^-1 (i > s), D_sj <- -U_ss^-1 R_j (j > s)
// after which the blocks below the diagonal are L^-1's and those above U^-1's
// (with the guarded pivots).  LI: L^-1 column-major, UI: U^-1 row-major, 64 x 64
// each, the blocks on the other side of the diagonal not written.  *guard: a
// pivot took the guard.
__device__ __forceinline__ void lu64(d4 (&D)[2], Lu64 &S, double *LI, double *UI, int *guard, int lane, int wi, int wj) {
    const int lo = lane & 15, hi = lane >> 4;
    if (threadIdx.x == 0) S.hit = 0;
    if (threadIdx.x < 256) S.one[BLD * (threadIdx.x >> 4) + (threadIdx.x & 15)] = threadIdx.x % 17 == 0 ? 1.0 : 0.0;
    // not unrolled: a workgroup runs this once, so its instructions come from
    // beyond the instruction cache, and four copies cost more to fetch than to run
#pragma unroll 1
    for (int s = 0; s < 4; s++) {
        double (*col)[BS] = S.col[s & 1], (*row)[BS] = S.row[s & 1];
        // block row and column s into LDS (the diagonal block with the column)
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int bj = 2 * wj + t;
            if (bj == s) blk_put(col[wi], D[t], lo, hi);
            else if (wi == s) blk_put(row[bj], D[t], lo, hi);
        }
        __syncthreads();
        if (wj == 0 && wi < 2) {
            double d[16];
#pragma unroll
            for (int j = 0; j < 16; j++) d[j] = col[s][BLD * lo + j];
            if (wi == 0) {
                double a[16];
                const double *A = hi == s ? S.one : col[hi];
#pragma unroll
                for (int j = 0; j < 16; j++) a[j] = A[BLD * lo + j];
                bool hit = false;
                const double r = pivot_whole(pivot_of<0>(d), hit);
                panel_rows<0>(d, a, (hi == s ? S.ui : col[hi]) + BLD * lo, r, hit);
                if (hit) S.hit = 1;
            } else {
                bool small;
                lower_inverse<0>(d, pivot_whole(pivot_of<0>(d), small), lo);
                if (hi == 0) {
#pragma unroll
                    for (int j = 0; j < 16; j++) S.li[BLD * lo + j] = j < lo ? d[j] : (j == lo ? 1.0 : 0.0);
                }
            }
        }
        __syncthreads();
        const d4 zero = {0.0, 0.0, 0.0, 0.0};
        const int wv = threadIdx.x >> 6;
        if (wv < 4 && wv != s) {   // a wave on each SIMD
            double *R = row[wv];
            double x[4], y[4];
            d4 acc = zero;
#pragma unroll
            for (int q = 0; q < 4; q++) { x[q] = R[BLD * (hi + 4 * q) + lo]; y[q] = S.li[BLD * lo + hi + 4 * q]; }
#pragma unroll
            for (int q = 0; q < 4; q++) acc = mfma4(x[q], y[q], acc);
            wave_sync();
            blk_put(R, acc, lo, hi);
        } else if (wv == s + 4) {   // the diagonal block's own factors are final
#pragma unroll
            for (int r = 0; r < 4; r++) {
                LI[64 * (16 * s + hi + 4 * r) + 16 * s + lo] = S.li[BLD * lo + hi + 4 * r];
                UI[64 * (16 * s + hi + 4 * r) + 16 * s + lo] = S.ui[BLD * (hi + 4 * r) + lo];
            }
        }
        __syncthreads();
        // every unfinished block as base - left right
        d4 acc[2];
        if (wi > s || 2 * wj + 1 > s) {
            const double *left = wi == s ? S.ui : col[wi];
            double x[2][4], y[4];
#pragma unroll
            for (int q = 0; q < 4; q++) y[q] = -left[BLD * lo + hi + 4 * q];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int bj = 2 * wj + t;
                const double *right = bj == s ? S.li : row[bj];
#pragma unroll
                for (int q = 0; q < 4; q++) x[t][q] = right[BLD * (hi + 4 * q) + lo];
                acc[t] = (wi == s || bj == s) ? zero : D[t];
            }
#pragma unroll
            for (int q = 0; q < 4; q++)
#pragma unroll
                for (int t = 0; t < 2; t++) acc[t] = mfma4(x[t][q], y[q], acc[t]);
        }
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const int bj = 2 * wj + t;
            if (wi > s || bj > s) D[t] = acc[t];
            else if (wi == s && bj < s) D[t] = blk_get(row[bj], lo, hi);
            else if (bj == s && wi < s) D[t] = blk_get(col[wi], lo, hi);
        }
    }
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const int bj = 2 * wj + t;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int i = 16 * wi + lo, j = 16 * bj + hi + 4 * r;
            if (wi > bj) LI[64 * j + i] = D[t][r];
            else if (wi < bj) UI[64 * i + j] = D[t][r];
        }
    }
    if (threadIdx.x == 0) *guard = S.hit;   // every pivot was before the last barriers
}

// A diagonal block, one workgroup per band: panel 0's, that of the shared rows'
// first panel, or (DIAG_NEXT) that of the panel after the one that `step` has
// eliminated, where k_tb_step does not do it.
enum { DIAG_FIRST = -1, DIAG_SHARED = -2 };
__global__ void __launch_bounds__(NT, 2) k_tb_diag(const TBand *bands, const double *AB, double *LI, double *UI,
                                                   int *guard, int step, int amax, const int *mask) {
    __shared__ Lu64 S;
    const TBand B = band_rec(bands, blockIdx.x);
    if (mask && !mask[B.inst]) return;
    int k = 0;
    if (step == DIAG_SHARED) {
        if (B.part < 0 || B.rev) return;
        k = B.na;
    } else if (step >= 0) {
        k = panel_at(B, step, amax) + 1;
        if (k < 1 || k >= B.nt || k == B.na || (B.rev && k > B.na)) return;
    }
    const int c0 = k * TB, kb = min(TB, B.m - c0);
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wi = wv & 3, wj = wv >> 2, lo = lane & 15, hi = lane >> 4;
    d4 D[2];
    const int i = 16 * wi + lo;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {   // past a short block: the identity
            const int j = 32 * wj + 16 * t + hi + 4 * r;
            const double v = tb_get(AB, B, c0 + min(i, kb - 1), c0 + min(j, kb - 1));
            D[t][r] = (i < kb && j < kb) ? v : (i == j ? 1.0 : 0.0);
        }
    lu64(D, S, LI + 4096 * (B.toff + k), UI + 4096 * (B.toff + k), guard + B.toff + k, lane, wi, wj);
}

// The band from the end's updates of the shared rows onto the other band's, which
// hold the matrix: one workgroup per column.
__global__ void __launch_bounds__(256) k_tb_merge(const TBand *bands, int b0, double *AB, const int *mask) {
    const TBand B = band_rec(bands, b0 + blockIdx.y);
    if (B.part < 0 || B.rev || (mask && !mask[B.inst])) return;
    const int j = TB * B.na + blockIdx.x;
    if (j >= B.m) return;
    const TBand Q = bands[B.part];
    for (int i = max(TB * B.na, j - B.w) + (int)threadIdx.x; i < min(B.m, j + B.w + 1); i += 256)
        tb_at(AB, B, i, j) += tb_get(AB, Q, B.mtot - 1 - i, B.mtot - 1 - j);
}

// Panel k: the trailing window A[r0:r1, r0:r1] -= (A[r0:r1, panel] U_k^-1) (L_k^-1 A[panel, r0:r1])
// with L_k, U_k the factors of the panel's (updated) diagonal block, one 64 x 64
// tile per workgroup of eight waves, on the matrix cores: first the tile's L and
// U panels (triangular inverses: 10 of 16 block products each, two block columns
// per wave that make up five), then their product.  Block columns and rows of
// a panel are left in the band as they stand at its elimination, which is what
// the sweeps read (scaled, k_tb_scale).  Every tile forms its own L and U panel:
// 2.25 times the flops of separate launches, but one dependent launch per panel,
// and at the usual band widths (a few tiles) the launch and the next diagonal
// block, not the matrix cores, are what a panel waits for.  The workgroup of the
// window's first tile, the next panel's diagonal block, goes on to factor it.
__global__ void __launch_bounds__(NT, 2) k_tb_step(const TBand *bands, int b0, double *AB, double *LI, double *UI,
                                                   int *guard, int step, int amax, int gt, const int *mask) {
    constexpr int LD = TB + 2;   // operand reads of 16 rows x 2 columns hit distinct banks
    __shared__ union {
        struct { double Xs[TB * LD], Us[TB * LD], Ls[4][16][64]; } p;
        Lu64 S;
    } sm;
    const TBand B = band_rec(bands, b0 + blockIdx.y);
    const int k = panel_at(B, step, amax);
    if (k < 0 || k + 1 >= B.nt || (mask && !mask[B.inst])) return;   // the last panel has no window
    if (B.rev && k >= B.na) return;
    const int c0 = k * TB;
    const int r0 = c0 + TB, r1 = min(B.m, r0 + B.w);
    const int I = blockIdx.x % gt, J = blockIdx.x / gt;
    const int i0 = r0 + TB * I, j0 = r0 + TB * J;
    const bool next = I == 0 && J == 0;   // the tile is panel k + 1's diagonal block
    if (!next && (i0 >= r1 || j0 >= r1)) return;
    // the next diagonal block is read whole (rows and columns past the window
    // keep their values: their products are zero), other tiles in the window
    const int cl = next ? min(B.m, r0 + TB) : r1;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wi = wv & 3, wj = wv >> 2, lo = lane & 15, hi = lane >> 4;
    const int i = i0 + 16 * wi + lo, ja = j0 + 32 * wj + hi;   // the lane's row; its columns ja + 16 t + 4 r
    // all loads in flight together: A[panel, columns] (staged), the factors' inverses, A[rows, panel], the tile
    double xv[8], lv[20], uv[20], av[16];
    d4 C[2];
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int e = threadIdx.x + NT * u, row = e & (TB - 1), col = e >> 6;
        xv[u] = tb_get(AB, B, c0 + row, min(j0 + col, r1 - 1));
    }
    // the wave's block columns of both products: wj and 3 - wj, with wj + 1 and 4 - wj blocks
    const double *Lk = LI + 4096 * (B.toff + k), *Uk = UI + 4096 * (B.toff + k);
#pragma unroll
    for (int z = 0; z < 20; z++) {
        const int blk = z < 4 * (wj + 1) ? wj : 3 - wj, q = z < 4 * (wj + 1) ? z : z - 4 * (wj + 1);
        lv[z] = Lk[64 * (4 * q + hi) + 16 * blk + lo];
        uv[z] = Uk[64 * (4 * q + hi) + 16 * blk + lo];
    }
#pragma unroll
    for (int q = 0; q < 16; q++) av[q] = tb_get(AB, B, min(i, r1 - 1), c0 + 4 * q + hi);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) C[t][r] = tb_get(AB, B, min(i, cl - 1), min(ja + 16 * t + 4 * r, cl - 1));
#pragma unroll
    for (int u = 0; u < 8; u++) {
        const int e = threadIdx.x + NT * u, row = e & (TB - 1), col = e >> 6;
        sm.p.Xs[LD * col + row] = j0 + col < r1 ? xv[u] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 16; q++) av[q] = i < r1 ? av[q] : 0.0;
    __syncthreads();
    const d4 zero = {0.0, 0.0, 0.0, 0.0};
    // L panel: rows of block wi, block columns wj and 3 - wj; U panel: columns of
    // block wi, block rows wj and 3 - wj (wave-uniform trip counts)
    auto panels = [&](auto WJ) {
        constexpr int J0 = decltype(WJ)::value;
        d4 l0 = zero, l1 = zero, u0 = zero, u1 = zero;
#pragma unroll
        for (int q = 0; q < 16 - 4 * J0; q++) {
            const double x = sm.p.Xs[LD * (16 * wi + lo) + 4 * q + hi];
            if (q < 4 * (J0 + 1)) {
                l0 = mfma4(uv[q], av[q], l0);
                u0 = mfma4(x, lv[q], u0);
            }
            l1 = mfma4(uv[4 * (J0 + 1) + q], av[q], l1);
            u1 = mfma4(x, lv[4 * (J0 + 1) + q], u1);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            sm.p.Ls[wi][4 * J0 + r][lane] = l0[r];
            sm.p.Ls[wi][4 * (3 - J0) + r][lane] = l1[r];
            sm.p.Us[LD * (16 * wi + hi + 4 * r) + 16 * J0 + lo] = u0[r];
            sm.p.Us[LD * (16 * wi + hi + 4 * r) + 16 * (3 - J0) + lo] = u1[r];
        }
    };
    if (wj == 0) panels(std::integral_constant<int, 0>());
    else panels(std::integral_constant<int, 1>());
    __syncthreads();
    d4 acc[2] = {zero, zero};
#pragma unroll
    for (int q = 0; q < 16; q++) {
        const double l = sm.p.Ls[wi][q][lane];
#pragma unroll
        for (int t = 0; t < 2; t++) acc[t] = mfma4(sm.p.Us[LD * (32 * wj + 16 * t + lo) + 4 * q + hi], l, acc[t]);
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = ja + 16 * t + 4 * r;
            C[t][r] = C[t][r] - acc[t][r];
            if (i < cl && j < cl) tb_at(AB, B, i, j) = C[t][r];
        }
    if (!next || k + 1 == B.na) return;   // the shared rows' first panel waits for k_tb_merge
    const int kb1 = min(TB, B.m - r0);
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int r = 0; r < 4; r++) {   // past a short last block: the identity
            const int ii = i - r0, jj = ja + 16 * t + 4 * r - r0;
            if (ii >= kb1 || jj >= kb1) C[t][r] = ii == jj ? 1.0 : 0.0;
        }
    __syncthreads();   // the products' LDS reads are done
    lu64(C, sm.S, LI + 4096 * (B.toff + k + 1), UI + 4096 * (B.toff + k + 1), guard + B.toff + k + 1, lane, wi, wj);
}

// The same in parts: four ninths of the products of k_tb_step with wide windows, and four
// workgroups a CU, so that one's loads run beside another's products.  Bound by the
// window's way through memory (columns of 64 rows, on no line's start): 1000 x 500
// cells in 16 blocks, 18,432 tiles a panel, 386 us an update, 3.1 TB/s and 25
// TFLOP/s (factorisation 360 ms; 623 by k_tb_step, 401 with a substitution launch
// and an update by vector FMAs).  k_tb_panel: a workgroup per 64 rows of the L panel (blockIdx.x
// < gt) or 64 columns of the U panel, as k_tb_step forms them, into P: 2 gt tiles
// a band, in the order in which the matrix cores take them, [block][q][lane]:
// L[16 block + lane % 16][4 q + lane / 16], U[4 q + lane / 16][16 block + lane % 16].
__global__ void __launch_bounds__(NT, 2) k_tb_panel(const TBand *bands, int b0, const double *AB, const double *LI,
                                                    const double *UI, double *P, int step, int amax, int gt,
                                                    const int *mask) {
    constexpr int LD = TB + 2;
    __shared__ double Xs[TB * LD];
    const TBand B = band_rec(bands, b0 + blockIdx.y);
    const int k = panel_at(B, step, amax);
    if (k < 0 || k + 1 >= B.nt || (mask && !mask[B.inst])) return;
    if (B.rev && k >= B.na) return;
    const bool low = (int)blockIdx.x < gt;
    const int c0 = k * TB, r0 = c0 + TB, r1 = min(B.m, r0 + B.w);
    const int t0 = r0 + TB * (low ? (int)blockIdx.x : (int)blockIdx.x - gt);
    if (t0 >= r1) return;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wi = wv & 3, wj = wv >> 2, lo = lane & 15, hi = lane >> 4;
    double *out = P + 4096 * (2 * (size_t)gt * (b0 + blockIdx.y) + blockIdx.x) + 1024 * wi;
    // the wave's block columns (rows) of the product: wj and 3 - wj, with wj + 1 and 4 - wj blocks
    const double *inv = (low ? UI : LI) + 4096 * (B.toff + k);
    double iv[20], av[16];
#pragma unroll
    for (int z = 0; z < 20; z++) {
        const int blk = z < 4 * (wj + 1) ? wj : 3 - wj, q = z < 4 * (wj + 1) ? z : z - 4 * (wj + 1);
        iv[z] = inv[64 * (4 * q + hi) + 16 * blk + lo];
    }
    if (low) {
        const int i = t0 + 16 * wi + lo;
#pragma unroll
        for (int q = 0; q < 16; q++) av[q] = tb_get(AB, B, min(i, r1 - 1), c0 + 4 * q + hi);
#pragma unroll
        for (int q = 0; q < 16; q++) av[q] = i < r1 ? av[q] : 0.0;
    } else {
        double xv[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int e = threadIdx.x + NT * u, row = e & (TB - 1), col = e >> 6;
            xv[u] = tb_get(AB, B, c0 + row, min(t0 + col, r1 - 1));
        }
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int e = threadIdx.x + NT * u, row = e & (TB - 1), col = e >> 6;
            Xs[LD * col + row] = t0 + col < r1 ? xv[u] : 0.0;
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 16; q++) av[q] = Xs[LD * (16 * wi + lo) + 4 * q + hi];
    }
    auto products = [&](auto WJ) {
        constexpr int J0 = decltype(WJ)::value;
        d4 p0 = {0.0, 0.0, 0.0, 0.0}, p1 = p0;
#pragma unroll
        for (int q = 0; q < 16 - 4 * J0; q++) {
            if (q < 4 * (J0 + 1)) p0 = low ? mfma4(iv[q], av[q], p0) : mfma4(av[q], iv[q], p0);
            const double v = iv[4 * (J0 + 1) + q];
            p1 = low ? mfma4(v, av[q], p1) : mfma4(av[q], v, p1);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            if (low) {
                out[64 * (4 * J0 + r) + lane] = p0[r];
                out[64 * (4 * (3 - J0) + r) + lane] = p1[r];
            } else {   // U[16 block + lo][column hi + 4 r]
                const int to = 64 * (lo >> 2) + 16 * (lo & 3) + hi + 4 * r;
                out[64 * 4 * J0 + to] = p0[r];
                out[64 * 4 * (3 - J0) + to] = p1[r];
            }
        }
    };
    if (wj == 0) products(std::integral_constant<int, 0>());
    else products(std::integral_constant<int, 1>());
}

// Panel k's window from P: a workgroup of four waves per 64 x 64 tile, 32 x 32 a wave.
__global__ void __launch_bounds__(256, 4) k_tb_update(const TBand *bands, int b0, double *AB, const double *P, int step,
                                                      int amax, int gt, const int *mask) {
    const TBand B = band_rec(bands, b0 + blockIdx.y);
    const int k = panel_at(B, step, amax);
    if (k < 0 || k + 1 >= B.nt || (mask && !mask[B.inst])) return;
    if (B.rev && k >= B.na) return;
    const int r0 = k * TB + TB, r1 = min(B.m, r0 + B.w);
    const int I = blockIdx.x % gt, J = blockIdx.x / gt;
    const int i0 = r0 + TB * I, j0 = r0 + TB * J;
    if (i0 >= r1 || j0 >= r1) return;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wi = 2 * (wv & 1), wj = 2 * (wv >> 1), lo = lane & 15, hi = lane >> 4;
    const double *Pb = P + 4096 * (2 * (size_t)gt * (b0 + blockIdx.y));
    const double *Lp = Pb + 4096 * I + 1024 * wi + lane, *Up = Pb + 4096 * (gt + J) + 1024 * wj + lane;
    const int i = i0 + 16 * wi + lo, j = j0 + 16 * wj + hi;
    d4 C[2][2], acc[2][2];
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                C[a][t][r] = tb_get(AB, B, min(i + 16 * a, r1 - 1), min(j + 16 * t + 4 * r, r1 - 1));
                acc[a][t][r] = 0.0;
            }
#pragma unroll 4
    for (int q = 0; q < 16; q++) {
        double l[2], u[2];
#pragma unroll
        for (int a = 0; a < 2; a++) {
            l[a] = Lp[1024 * a + 64 * q];
            u[a] = Up[1024 * a + 64 * q];
        }
#pragma unroll
        for (int a = 0; a < 2; a++)
#pragma unroll
            for (int t = 0; t < 2; t++) acc[a][t] = mfma4(u[t], l[a], acc[a][t]);
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int ii = i + 16 * a, jj = j + 16 * t + 4 * r;
                if (ii < r1 && jj < r1) tb_at(AB, B, ii, jj) = C[a][t][r] - acc[a][t][r];
            }
}

// Every panel's diagonal block inverse for the sweeps, in the place of its
// factors' inverses: G_k = U_k^-1 L_k^-1 (column-major) for the forward sweep
// and the backward sweep's UI_k.  Where no pivot of the block took the guard
// the two are the same.  Where one did, the reference's backward substitution
// divides by the pivot itself (solv_blk_solve.c:50-52) after an elimination
// with the guarded one: U^-1 L^-1 with L's multipliers guarded and U's own
// diagonal, formed column by column from the block's LU (rare).  One workgroup
// of a wave per tile, column t in lane t.
__global__ void __launch_bounds__(64) k_tb_inv(const TBand *bands, int b0, const double *AB, double *LI, double *UI,
                                               const int *guard, const int *mask) {
    __shared__ double D[TB][TB + 1];
    __shared__ double X[TB][TB + 1];
    const TBand B = band_rec(bands, b0 + blockIdx.y);
    const int k = blockIdx.x;
    if (k >= (B.rev ? B.na : B.nt) || (mask && !mask[B.inst])) return;
    const int c0 = k * TB, kb = min(TB, B.m - c0), t = threadIdx.x;
    double *Lk = LI + 4096 * (B.toff + k), *Uk = UI + 4096 * (B.toff + k);
    const int lo = t & 15, hi = t >> 4;
    // G by 16 x 16 blocks: G^T[j][i] = sum_m L^-1[m][j] U^-1[i][m] over blocks m >= max(i, j)
    for (int j = 0; j < 64; j++) {   // the blocks of the other triangle were not written
        D[t][j] = j >= (t & ~15) ? Uk[64 * t + j] : 0.0;
        X[j][t] = j >= (t & ~15) ? Lk[64 * t + j] : 0.0;
    }
    __syncthreads();
    for (int bi = 0; bi < 4; bi++)
        for (int bj = 0; bj < 4; bj++) {
            d4 acc = {0.0, 0.0, 0.0, 0.0};
            for (int q = 4 * max(bi, bj); q < 16; q++)
                acc = mfma4(X[4 * q + hi][16 * bj + lo], D[16 * bi + lo][4 * q + hi], acc);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                Lk[64 * (16 * bj + hi + 4 * r) + 16 * bi + lo] = acc[r];
                Uk[64 * (16 * bj + hi + 4 * r) + 16 * bi + lo] = acc[r];
            }
        }
    if (!guard[B.toff + k]) return;
    __syncthreads();
    for (int j = 0; j < TB; j++)
        D[t][j] = (t < kb && j < kb) ? tb_get(AB, B, c0 + t, c0 + j) : (t == j ? 1.0 : 0.0);
    __syncthreads();
    for (int p = 0; p < TB; p++) {   // LU in place, lane t row t
        const double rden = 1.0 / guarded(D[p][p]);
        if (t > p) {
            const double l = D[t][p] * rden;
            D[t][p] = l;
            for (int j = p + 1; j < TB; j++) D[t][j] = fma(-l, D[p][j], D[t][j]);
        }
        __syncthreads();
    }
    for (int i = 0; i < TB; i++) {   // lane t column t: L y = e_t
        double s = i == t ? 1.0 : 0.0;
        for (int q = 0; q < i; q++) s = fma(-D[i][q], X[q][t], s);
        X[i][t] = s;
    }
    for (int i = TB - 1; i >= 0; i--) {   // U x = y
        double s = X[i][t];
        for (int q = i + 1; q < TB; q++) s = fma(-D[i][q], X[q][t], s);
        X[i][t] = s / D[i][i];
    }
    __syncthreads();
    for (int j = 0; j < TB; j++) Uk[64 * j + t] = X[t][j];
}

// After the factorisation: every off-diagonal tile below a diagonal block times
// that block's G, and above it times its UI, in place, so that a sweep step's
// off-diagonal update reads one tile and no inverse: x_i -= (A_ik G_k) x_k,
// y_i -= (A_ik UI_k) y_k.  The products fill at most
// the band's TB extra diagonals (entries within w + 63 of the diagonal), which
// is what they are stored for.  One workgroup of 256 threads per tile, a 4 x 4
// register block each from LDS.
__global__ void __launch_bounds__(256) k_tb_scale(const TBand *bands, int b0, double *AB, const double *G,
                                                  const double *UI, int gf, const int *mask) {
    __shared__ double As[TB][TB];       // As[q][row]: the tile, column q
    __shared__ double Ms[TB][TB + 1];   // Ms[q][col]: the inverse
    const TBand B = band_rec(bands, b0 + blockIdx.z);
    const int k = blockIdx.x;
    if (k >= (B.rev ? B.na : B.nt) || (mask && !mask[B.inst])) return;
    const bool low = (int)blockIdx.y < gf;
    const int g = (low ? (int)blockIdx.y : (int)blockIdx.y - gf) + 1;
    const int c0 = k * TB, kb = min(TB, B.m - c0);
    // the tile's first row, and its rows inside the reach of the panel's columns
    const int tr0 = low ? c0 + TB * g : c0 - TB * g;
    const int i0 = low ? tr0 : max(tr0, max(0, c0 - B.w));
    const int i1 = low ? min(tr0 + TB, min(B.m, c0 + kb + B.w)) : tr0 + TB;
    if (i0 >= i1) return;
    const int t = threadIdx.x;
    const double *M = (low ? G : UI) + 4096 * (B.toff + k);
    double av[16], mv[16];   // all loads in flight before the LDS stores
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int e = t + 256 * u, lo = e & (TB - 1), hi = e >> 6;
        av[u] = tb_get(AB, B, min(max(tr0 + lo, i0), i1 - 1), c0 + min(hi, kb - 1));
        mv[u] = M[e];   // column-major: row lo, column hi
    }
#pragma unroll
    for (int u = 0; u < 16; u++) {
        const int e = t + 256 * u, lo = e & (TB - 1), hi = e >> 6;
        const int r = tr0 + lo;
        As[hi][lo] = (r >= i0 && r < i1 && hi < kb) ? av[u] : 0.0;
        Ms[lo][hi] = mv[u];
    }
    __syncthreads();
    const int tr = t & 15, tc = t >> 4;   // rows 4 tr .. 4 tr + 3, columns 4 tc .. 4 tc + 3
    double acc[4][4] = {};
#pragma unroll 8
    for (int q = 0; q < kb; q++) {
        double a[4], b[4];
#pragma unroll
        for (int u = 0; u < 4; u++) { a[u] = As[q][4 * tr + u]; b[u] = Ms[q][4 * tc + u]; }
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[u][v] = fma(a[u], b[v], acc[u][v]);
    }
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const int c = 4 * tc + v;
        if (c >= kb) continue;
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const int r = tr0 + 4 * tr + u;
            if (r >= i0 && r < i1) tb_at(AB, B, r, c0 + c) = acc[u][v];
        }
    }
}

// ---- substitutions ----------------------------------------------------------
// One kernel runs both sweeps as a dataflow over 64-row tiles: a workgroup takes
// the next tile row in order (a ticket), adds up its tiles' products as the
// rows they need are finished, and publishes its 64 values.  A value is its own
// ready flag (sw2_flow.h): the output vectors hold EMPTY until it is stored.
// Tickets make it free of deadlock whatever is resident: rows are claimed in
// order, so the lowest unfinished row belongs to a running workgroup and waits
// only for finished ones.
// the value at p in every lane with `want`, waiting until all of the wave's are there
__device__ __forceinline__ double await_value(const double *p, bool want) {
    Slot<double>::U u = want ? peek(p) : 0ull;
    while (__any(u == Slot<double>::EMPTY)) {
        __builtin_amdgcn_s_sleep(1);
        if (u == Slot<double>::EMPTY) u = peek(p);
    }
    return __longlong_as_double((long long)u);
}

// The right-hand side into band order (nodes of no block skipped; the band from
// the end has zeros on the shared rows), the two output vectors to EMPTY, the
// tickets (three a band, and the claims of bands) to zero.
__global__ void __launch_bounds__(256) k_tb_gather(int N, int nband, int nbot, const int *node_blk,
                                                   const TBand *bands, const double *x, double *xb, double *yb,
                                                   double *zb, int *tick) {
    const int a = blockIdx.x * blockDim.x + threadIdx.x;
    for (int b = a; b < 3 * nband + 1; b += gridDim.x * blockDim.x) tick[b] = 0;
    if (a >= N) return;
    const int bk = node_blk[a];
    if (bk < 0) return;
    const TBand B = bands[nbot + bk];
    const TBand Q = bands[max(B.part, 0)];
    const double empty = __builtin_bit_cast(double, Slot<double>::EMPTY);
    for (int v = 0; v < 3; v++) {
        const int i = 3 * (a - B.n0) + v;
        const double xv = x[vidx3(a, v)];
        auto put = [&](size_t o, double r) { xb[o] = r; yb[o] = empty; zb[o] = empty; };
        if (i < B.m) put(B.xoff + i, xv);
        if (B.part >= 0 && i >= TB * B.na) put(Q.xoff + B.mtot - 1 - i, i < B.m ? 0.0 : xv);
    }
}

// One sweep of a band by this workgroup.  FWD: y_i = x_i - sum_{k < i} (A_ik
// G_k) y_k into out = yb; else z_i = y_i - sum_{k > i} (A_ik UI_k) z_k into out
// = zb (the diagonal inverse is applied afterwards, k_tb_apply).  Eight waves
// take 8 columns each of every tile, lane r row r; the ninth wave polls the
// values the tiles multiply (so that no poll queues behind a tile's loads),
// hands them over in LDS, adds the row's partial sums in wave order and
// publishes it.  A product's tile was fetched SW_PF products earlier, across
// rows, so a step of the chain is the hand-over and one 64 x 64 product; the
// order of every sum is fixed, whichever workgroup runs the row.  A workgroup that
// has its band to itself needs no tickets and keeps the values of its last row (a
// step of 100 models of 500 triangles in 20 blocks each, 2,000 bands of one or two
// tiles: 6.5 ms, 7.7 with tickets, 7.2 in a launch per tile row).
constexpr int SW_W = 8;                  // product waves
constexpr int SW_NT = 64 * (SW_W + 1);   // threads of a sweep workgroup
constexpr int SW_PF = 4;                 // tiles fetched ahead
constexpr int SW_RING = 32;              // values handed over between two barriers
struct SweepLds {
    double x[SW_RING][TB];
    double part[2][SW_W][TB];
    int unit;        // SW_SHARED: the workgroup's place in the order of claims
    int ready;       // values handed over since the last barrier
    int rows[2][4];  // the next row and those claimed after it
};
// Rows: FWD all, upwards from 0; else nrows of them downwards from `first`.  A
// band from the end has no factors for the shared rows: FWD its columns before
// them, so that y is what it subtracts there, which `other` (FWD, the band from
// the start: the other's y, read backwards) adds; downwards the shared rows'
// values are x, not z, and stand in out already.
template <bool FWD>
__device__ __forceinline__ void tb_sweep(const TBand &B, const double *AB, const double *in, double *out,
                                         const double *other, int first, int nrows, int *tick, SweepLds &S) {
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool server = wv == SW_W;
    // t-th row in sweep order; its number of tiles; the j-th of them in the order their values finish
    auto row_of = [&](int t) { return FWD ? t : first - t; };
    auto ktop = [&](int i) { return B.rev ? min(i, B.na) : i; };   // FWD: end of the row's columns
    auto ntiles = [&](int i) {
        if (FWD) {
            const int d = TB * i - TB - B.w;   // column tile k reaches row tile i when 64 k > d
            return max(0, ktop(i) - (d < 0 ? 0 : d / TB + 1));
        }
        return min(B.nt - 1, (TB * i + TB + B.w - 1) / TB) - i;
    };
    auto kcol = [&](int i, int n, int j) { return FWD ? ktop(i) - n + j : i + n - j; };
    const bool alone = gridDim.x == 1;   // all rows are this workgroup's: no tickets
    if (threadIdx.x == 64 * SW_W) {
        S.rows[0][0] = alone ? 0 : atomicAdd(tick, 1);
        S.ready = 0;
    }
    __syncthreads();
    int cur = __builtin_amdgcn_readfirstlane(S.rows[0][0]);
    __syncthreads();
    // an LDS pointer by type: a generic one would make the polls flat loads,
    // which queue behind the tiles' loads
    using lds_int = __attribute__((address_space(3))) volatile int;
    lds_int *ready = (lds_int *)&S.ready;
    int parity = 0;
    if (server) {
        // rows claimed ahead (INT_MAX: not yet), one when a row's first value has
        // arrived -- by then the other workgroups have theirs, so neighbouring
        // rows go to different workgroups -- and one more after a row while the
        // product waves cannot see SW_PF tiles ahead
        int q0 = alone ? 1 : INT_MAX, q1 = alone ? 2 : INT_MAX, q2 = INT_MAX, ahead = 3;
        double last = 0.0;   // alone: the values of the row before
        auto claim = [&]() {
            if (q2 != INT_MAX) return;
            int t = 0;
            if (alone) t = ahead++;
            else if (lane == 0) t = atomicAdd(tick, 1);
            t = __builtin_amdgcn_readfirstlane(t);
            if (q0 == INT_MAX) q0 = t;
            else if (q1 == INT_MAX) q1 = t;
            else q2 = t;
        };
        while (cur < nrows) {
            const int i = row_of(cur), n = ntiles(i), r = TB * i + lane;
            double xi = FWD ? in[B.xoff + min(r, B.m - 1)] : await_value(in + B.xoff + min(r, B.m - 1), true);
            if (FWD && other && i >= B.na) xi += await_value(other + B.mtot - 1 - min(r, B.m - 1), true);
            if (n == 0) claim();
            for (int j = 0; j < n; j++) {
                const int k = kcol(i, n, j), d = TB * k + lane;
                const bool own = alone && cur > 0 && k == (FWD ? i - 1 : i + 1);
                const double v = own ? last : await_value(out + B.xoff + min(d, B.m - 1), d < B.m);
                S.x[j % SW_RING][lane] = v;   // 0 past the band's last row
                wave_sync();                  // LDS keeps a wave's order: the value, then the count
                if (lane == 0) *ready = j % SW_RING + 1;
                if (j == 0) claim();
                if (j % SW_RING == SW_RING - 1 && j + 1 < n) {   // the ring is full: wait for the products
                    __syncthreads();
                    if (lane == 0) *ready = 0;
                    __syncthreads();
                }
            }
            if (lane < 3) S.rows[parity][lane] = lane == 0 ? q0 : (lane == 1 ? q1 : q2);
            __syncthreads();   // the row's partial sums are in LDS
            if (lane == 0) *ready = 0;
            double s = S.part[parity][0][lane];
#pragma unroll
            for (int w = 1; w < SW_W; w++) s += S.part[parity][w][lane];
            last = r < B.m ? xi - s : 0.0;
            if (r < B.m) put(out + B.xoff + r, last);
            cur = q0;
            q0 = q1;
            q1 = q2;
            q2 = INT_MAX;
            parity ^= 1;
            __syncthreads();   // the next row's hand-overs count from zero
            if ((n < SW_PF ? q1 : q0) == INT_MAX) claim();
        }
    } else {
        const int c8 = 8 * wv;
        double m[SW_PF][8];
        long long tag[SW_PF] = {-1, -1, -1, -1};   // row (in sweep order) and tile whose entries m[s] holds
        auto id = [&](int t, int j) { return ((long long)t << 32) | j; };
        auto fetch = [&](double (&d)[8], int t, int j) {
            const int i = row_of(t), n = ntiles(i), k = kcol(i, n, j);
            const int ck = TB * k, kb = min(TB, B.m - ck), r = TB * i + lane;
            const int rc = FWD ? min(r, min(B.m, ck + TB + B.w) - 1) : max(r, max(0, ck - B.w));
            const double *p = AB + tb_idx(B, rc, ck);
#pragma unroll
            for (int u = 0; u < 8; u++) d[u] = p[(size_t)min(c8 + u, kb - 1) * (2 * B.wp)];
        };
        int q[2] = {alone ? 1 : INT_MAX, alone ? 2 : INT_MAX};   // the rows after cur, as far as they are known
        int j = 0, n = cur < nrows ? ntiles(row_of(cur)) : 0;
        // the entries of the `ahead`-th tile from (cur, j) into d, and its tag.  Always
        // eight loads, so that the number in flight is known where one is waited
        // for: past the known rows an earlier tile again (row 1 has one
        // wherever there is a second row), under no tag.
        auto prefetch = [&](double (&d)[8], int ahead) {
            int t = cur, jj = j + ahead, nn = n;
#pragma unroll
            for (int a = 0; a < 2; a++)
                if (jj >= nn && t < nrows) {
                    jj -= nn;
                    t = q[a];
                    nn = t < nrows ? ntiles(row_of(t)) : 0;
                }
            const bool got = t < nrows && jj < nn;
            if (!got) { t = 1; jj = 0; }
            fetch(d, t, jj);
            return got ? id(t, jj) : -1LL;
        };
        if (nrows > 1) {
#pragma unroll
            for (int s = 0; s < SW_PF; s++) tag[s] = prefetch(m[s], s);
        }
        double acc = 0.0;
        while (cur < nrows) {
#pragma unroll
            for (int s = 0; s < SW_PF; s++) {
                while (j == n) {   // the row is done
                    S.part[parity][wv][lane] = acc;
                    __syncthreads();
                    cur = __builtin_amdgcn_readfirstlane(S.rows[parity][0]);
                    q[0] = __builtin_amdgcn_readfirstlane(S.rows[parity][1]);
                    q[1] = __builtin_amdgcn_readfirstlane(S.rows[parity][2]);
                    parity ^= 1;
                    j = 0;
                    acc = 0.0;
                    n = cur < nrows ? ntiles(row_of(cur)) : -1;
                    __syncthreads();
                }
                if (n < 0) break;   // no rows left
                const int i = row_of(cur), k = kcol(i, n, j), ck = TB * k, r = TB * i + lane;
                if (tag[s] != id(cur, j)) {   // its row was not known in time
                    fetch(m[s], cur, j);
                    // used here, so that this path waits here and the other keeps its fetches in flight
                    asm volatile("" : "+v"(m[s][0]), "+v"(m[s][1]), "+v"(m[s][2]), "+v"(m[s][3]), "+v"(m[s][4]),
                                 "+v"(m[s][5]), "+v"(m[s][6]), "+v"(m[s][7]));
                }
                while (*ready <= j % SW_RING) __builtin_amdgcn_s_sleep(1);
                wave_sync();
                const double xv = S.x[j % SW_RING][c8 + (lane & 7)];
                double p = 0.0;
#pragma unroll
                for (int u = 0; u < 8; u++) p = fma(m[s][u], lane_bcast(xv, u), p);
                // rows the column tile does not reach were read clamped
                const bool in_reach = FWD ? r < min(B.m, ck + TB + B.w) : r >= ck - B.w;
                acc += in_reach ? p : 0.0;
                if (j % SW_RING == SW_RING - 1 && j + 1 < n) {
                    __syncthreads();
                    __syncthreads();
                }
                tag[s] = prefetch(m[s], SW_PF);
                j++;
            }
        }
    }
    __syncthreads();   // the LDS is free for the next sweep
}

// Where blocks are factored from both ends, SHARED: the forward sweep of every
// band and the backward sweep of the shared rows; then, those applied
// (k_tb_apply), REST: the backward sweep of all others.  ALL: no such block.
// In SHARED the bands from the start wait for those from the end, which wait for
// nothing outside the band and come first in the list of bands.  A workgroup
// takes its band by ticket (`claim`), so whatever order the workgroups start in,
// every band from the end has its workgroups running before one waits for it.
// (200 x 100 cells: both sweeps 1.83 ms, 1.84 with a band per grid index.)
enum { SW_ALL, SW_SHARED, SW_REST };
__global__ void __launch_bounds__(SW_NT) k_tb_sweep(const TBand *bands, int b0, const double *AB, const double *xb, double *yb,
                                                    double *zb, int *tick, int *claim, int phase, const int *done,
                                                    const int *mask, const KScal *sc) {
    __shared__ SweepLds S;
    int band = b0 + blockIdx.y;
    if (phase == SW_SHARED) {
        if (threadIdx.x == 0) S.unit = atomicAdd(claim, 1);
        __syncthreads();
        band = __builtin_amdgcn_readfirstlane(S.unit) / (int)gridDim.x;
    }
    const int stop = *done;   // the band record and the flag fetched together
    const TBand B = band_rec(bands, band, stop);
    // ensembles: the band's model, converged or outside the mask, is skipped
    if (stop || (mask && (!mask[B.inst] || (sc && sc[B.inst].done)))) return;
    if (B.nt == 1) {   // nothing to substitute
        if (phase != SW_SHARED && (int)threadIdx.x < B.m && blockIdx.x == 0)
            zb[B.xoff + threadIdx.x] = xb[B.xoff + threadIdx.x];
        return;
    }
    tick += 3 * band;
    if (phase != SW_REST) {
        const bool top = B.part >= 0 && !B.rev;
        tb_sweep<true>(B, AB, xb, yb, top ? yb + bands[B.part].xoff : nullptr, 0, B.nt, tick, S);
        if (top) tb_sweep<false>(B, AB, yb, zb, nullptr, B.nt - 1, B.nt - B.na, tick + 1, S);
    }
    if (phase != SW_SHARED) tb_sweep<false>(B, AB, yb, zb, nullptr, B.na - 1, B.na, tick + 2, S);
}

// The backward sweep's diagonal inverses, and back into node order: x_k = UI_k z_k,
// one workgroup of four waves per tile (16 columns each, partial sums added in
// wave order).  `shared`: of the shared rows, which the band from the end
// receives too; else of the others.  A model that has converged, or is outside
// the mask, keeps x.
__global__ void __launch_bounds__(256) k_tb_apply(const TBand *bands, int b0, const double *UI, double *zb, double *x,
                                                  bool shared, const int *done, const int *mask, const KScal *sc) {
    __shared__ double part[4][TB];
    const int stop = *done;
    const TBand B = band_rec(bands, b0 + blockIdx.y, stop);
    if (shared && (B.part < 0 || B.rev)) return;
    const int k = blockIdx.x + (shared ? B.na : 0);
    if (stop || k >= (shared ? B.nt : B.na) || (mask && (!mask[B.inst] || (sc && sc[B.inst].done)))) return;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c0 = TB * k, kb = min(TB, B.m - c0);
    const double *M = UI + 4096 * (B.toff + k);
    double m[16];
#pragma unroll
    for (int u = 0; u < 16; u++) m[u] = M[64 * (16 * wv + u) + lane];
    const double zv = zb[B.xoff + c0 + min(lane, kb - 1)];
    const double zr = lane < kb ? zv : 0.0;
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < 16; u++) s = fma(m[u], lane_bcast(zr, 16 * wv + u), s);
    part[wv][lane] = s;
    __syncthreads();
    if (wv != 0 || lane >= kb) return;
    const int d = B.rev ? B.mtot - 1 - (c0 + lane) : c0 + lane;
    s = ((part[0][lane] + part[1][lane]) + part[2][lane]) + part[3][lane];
    x[vidx3(B.n0 + d / 3, d % 3)] = s;
    if (shared) zb[bands[B.part].xoff + B.mtot - 1 - d] = s;
}

void tband_free(Ctx *c) {
    for (void *p : {(void *)c->tb_bands, (void *)c->tb_AB, (void *)c->tb_LI, (void *)c->tb_UI, (void *)c->tb_xb,
                    (void *)c->tb_yb, (void *)c->tb_zb, (void *)c->tb_int, (void *)c->tb_P})
        if (p) (void)hipFree(p);
    c->tb_bands = nullptr; c->tb_AB = nullptr; c->tb_LI = nullptr; c->tb_UI = nullptr; c->tb_int = nullptr;
    c->tb_P = nullptr;
    c->tb_xb = nullptr; c->tb_yb = nullptr; c->tb_zb = nullptr;
    c->tb_nband = 0; c->tb_maxnt = 0; c->tb_gt = 0; c->tb_gf = 0; c->tb_size = 0;
    c->tb_h_nt.clear(); c->tb_h_inst.clear(); c->tb_h_na.clear(); c->tb_h_gt.clear();
    c->tb_nbot = 0; c->tb_maxs = 0;
}

// Panels from each end of a block of m DOFs and half bandwidth w, 0: one band.
// From both ends the chain of dependent panels is the longer end's and the
// shared rows' (at least w of them, so that the ends do not couple), plus a merge
// and a diagonal block on their own, about one panel's time; from one end it is
// all of the block's.  Short ends are not worth the sweeps' extra launches.
static int twist_panels(int m, int w) {
    const int nt = (m + TB - 1) / TB, a = m > w ? (m - w) / (2 * TB) : 0;
    const int shared = m - 2 * TB * a;
    return a >= 3 && a + (shared + TB - 1) / TB + 2 < nt ? a : 0;
}

// Window tiles of a step over all bands above which the panels are formed on their
// own: three for each CU, which holds one workgroup of k_tb_step.  Below, the parts'
// two launches more and the panels' way through memory cost as much as the products
// formed again, or more.  Factorisation in one launch a panel and in parts, ms, at about
// the given tiles a step: 200 13.8 and 17.1 (800 x 100 cells, nblock 4), 400 35.0 and
// 35.5 (400 x 200, 2), 450 76.8 and 102 (400 x 300, 1), 600 31.1 and 27.9 (400 x 200,
// 3), 900 72.4 and 73.6 (400 x 300, 2), 1,150 355 and 319 (500 x 500, 1), 5,600 19.9
// and 13.0 (400 x 200, 28); a floodplain's three steps at 650 31.8 and 34.3 s.
constexpr size_t PARTS_TILES = 768;

// Bands of the node blocks (nodes [s0[b], s1[b]) of model inst[b]) with
// pattern half bandwidths w[] (DOFs).  Returns an error text or "".
std::string tband_structure(Ctx *c, const std::vector<int> &s0, const std::vector<int> &s1,
                            const std::vector<int> &inst, const std::vector<int> &w) {
    tband_free(c);
    const int nblk = (int)w.size();
    size_t freeb = 0, totalb = 0;
    (void)hipMemGetInfo(&freeb, &totalb);
    std::vector<TBand> h;
    size_t off = 0, toff = 0, xoff = 0, nint = 0, need = 0, npart = 0;
    int maxnt = 0, maxw = 0;
    // blocks from both ends take s rows more each; where that does not fit, one band each
    for (const bool twist : {true, false}) {
        std::vector<int> top(nblk);
        int nbot = 0;
        for (int b = 0; b < nblk; b++) {
            top[b] = twist ? twist_panels(3 * (s1[b] - s0[b]), w[b]) : 0;
            nbot += top[b] > 0;
        }
        h.assign(nbot + nblk, TBand{});
        off = toff = xoff = 0;
        maxnt = maxw = c->tb_maxs = 0;
        for (int b = 0, bot = 0; b < nblk; b++) {
            const int mtot = 3 * (s1[b] - s0[b]);
            for (int rev = 0; rev <= (top[b] > 0); rev++) {
                TBand &B = h[rev ? bot : nbot + b];
                B.n0 = s0[b];
                B.m = top[b] ? mtot - TB * top[b] : mtot;   // all but the other end's rows
                B.w = w[b];
                B.wp = w[b] + TB;
                B.nt = (B.m + TB - 1) / TB;
                B.na = top[b] ? top[b] : B.nt;
                B.part = top[b] ? (rev ? nbot + b : bot) : -1;
                B.rev = rev;
                B.mtot = mtot;
                B.pad = 0;
                B.inst = inst[b];
                B.off = off;
                B.toff = toff;
                B.xoff = xoff;
                off += (size_t)B.m * (2 * B.wp + 1);
                toff += B.nt;
                xoff += B.m;
                maxnt = std::max(maxnt, B.nt);
                maxw = std::max(maxw, B.w);
                if (top[b]) c->tb_maxs = std::max(c->tb_maxs, B.m - TB * B.na);
            }
            bot += top[b] > 0;
        }
        c->tb_nbot = nbot;
        nint = toff + 3 * h.size() + 1;   // a guard flag per tile, three tickets per band, the claims
        size_t tiles = 0;   // of a step; with one tile a band nothing is formed twice
        for (const TBand &B : h) tiles += (size_t)((B.w + TB - 1) / TB) * ((B.w + TB - 1) / TB);
        npart = maxw > TB && tiles > PARTS_TILES ? 2 * 4096 * (size_t)((maxw + TB - 1) / TB) * h.size() : 0;
        need = sizeof(double) * (off + 2 * 4096 * toff + 3 * xoff) + sizeof(int) * nint;
        if (need + ((size_t)2 << 30) <= freeb) {
            if (need + sizeof(double) * npart + ((size_t)2 << 30) > freeb) npart = 0;   // one launch a panel then
            break;
        }
        if (twist && nbot > 0) continue;
        return "tiled band LU: " + std::to_string(need >> 20) + " MiB of band storage do not fit in the free " +
               std::to_string(freeb >> 20) + " MiB; raise nblock" +
               (c->ninst ? ", or step the models in groups that fit" : "");
    }
    const int nband = (int)h.size();
    if (hipMalloc((void **)&c->tb_bands, sizeof(TBand) * nband) != hipSuccess ||
        hipMemcpy(c->tb_bands, h.data(), sizeof(TBand) * nband, hipMemcpyHostToDevice) != hipSuccess ||
        hipMalloc((void **)&c->tb_AB, sizeof(double) * off) != hipSuccess ||
        hipMalloc((void **)&c->tb_LI, sizeof(double) * 4096 * toff) != hipSuccess ||
        hipMalloc((void **)&c->tb_UI, sizeof(double) * 4096 * toff) != hipSuccess ||
        hipMalloc((void **)&c->tb_xb, sizeof(double) * xoff) != hipSuccess ||
        hipMalloc((void **)&c->tb_yb, sizeof(double) * xoff) != hipSuccess ||
        hipMalloc((void **)&c->tb_zb, sizeof(double) * xoff) != hipSuccess ||
        hipMalloc((void **)&c->tb_int, sizeof(int) * nint) != hipSuccess ||
        (npart && hipMalloc((void **)&c->tb_P, sizeof(double) * npart) != hipSuccess)) {
        tband_free(c);
        return "hipMalloc failed for the tiled band LU";
    }
    c->tb_nband = nband;
    c->tb_maxnt = maxnt;
    c->tb_h_nt.resize(nband);
    c->tb_h_inst.resize(nband);
    c->tb_h_na.resize(nband);
    c->tb_h_gt.resize(nband);
    for (int b = 0; b < nband; b++) {
        c->tb_h_nt[b] = h[b].nt;
        c->tb_h_inst[b] = h[b].inst;
        c->tb_h_na[b] = h[b].part < 0 ? -1 : h[b].na;
        c->tb_h_gt[b] = (h[b].w + TB - 1) / TB;
    }
    c->tb_gt = (maxw + TB - 1) / TB;
    c->tb_gf = (maxw + 2 * TB - 2) / TB;   // tiles below (above) a panel that its L (U) reaches
    c->tb_size = off;
    c->tb_guard = c->tb_int + 3 * nband + 1;
    return "";
}

// Launches with a grid row (or layer) per band: HIP takes 65,536 of them, a
// partition may have more bands.  f(first band, bands)
constexpr int BANDS_A_LAUNCH = 32768;
template <typename F>
static void each_launch(const Ctx *c, F f) {
    for (int b0 = 0; b0 < c->tb_nband; b0 += BANDS_A_LAUNCH) f(b0, std::min(BANDS_A_LAUNCH, c->tb_nband - b0));
}

// the models the masked launches of an ensemble work on (null: every band)
static const int *tb_mask(const Ctx *c) { return c->ninst ? c->inst_mask : nullptr; }

// panels of the largest band whose model is in the mask: the launches past
// it would find every band's model masked (an ensemble whose large models
// have converged stops paying for their panels)
static int tb_active_nt(const Ctx *c) {
    if (!c->ninst || c->h_inst_mask.empty()) return c->tb_maxnt;
    int nt = 0;
    for (int b = 0; b < c->tb_nband; b++)
        if (c->h_inst_mask[c->tb_h_inst[b]]) nt = std::max(nt, c->tb_h_nt[b]);
    return nt;
}

void launch_tband_setup(Ctx *c) {
    const int *mask = tb_mask(c);
    const int nt = tb_active_nt(c);
    if (nt == 0) return;
    launch_zero(c, c->tb_AB, c->tb_size);
    hipLaunchKernelGGL(k_tb_load, dim3(nblocks_for(c->N, 256)), dim3(256), 0, c->stream, c->N, c->node_blk,
                       c->tb_bands, c->tb_nbot, c->tb_AB, c->diag, c->offd, c->row_ptr, c->sell_ptr, c->sell_col, mask);
    const int gt = std::max(1, c->tb_gt);
    // the step at which the active models' shared rows begin, and the steps in all
    int amax = 0, steps = 0;
    auto each_active = [&](auto f) {
        for (int b = 0; b < c->tb_nband; b++)
            if (!mask || c->h_inst_mask[c->tb_h_inst[b]]) f(b);
    };
    each_active([&](int b) { amax = std::max(amax, c->tb_h_na[b]); });
    each_active([&](int b) {
        steps = std::max(steps, c->tb_h_nt[b] - 1 + (c->tb_h_na[b] < 0 ? 0 : amax - c->tb_h_na[b]));
    });
    auto diag = [&](int step) {
        hipLaunchKernelGGL(k_tb_diag, dim3(c->tb_nband), dim3(NT), 0, c->stream, c->tb_bands, c->tb_AB, c->tb_LI,
                           c->tb_UI, c->tb_guard, step, amax, mask);
    };
    diag(DIAG_FIRST);
    auto merge = [&]() {
        each_launch(c, [&](int b0, int nb) {
            hipLaunchKernelGGL(k_tb_merge, dim3(c->tb_maxs, nb), dim3(256), 0, c->stream, c->tb_bands, b0, c->tb_AB,
                               mask);
        });
        diag(DIAG_SHARED);
    };
    size_t tiles = 0;
    each_active([&](int b) { tiles += (size_t)c->tb_h_gt[b] * c->tb_h_gt[b]; });
    const bool parts = c->tb_P && tiles > PARTS_TILES;
    for (int k = 0; k < steps; k++) {
        if (amax > 0 && k == amax) merge();
        if (parts) {
            each_launch(c, [&](int b0, int nb) {
                hipLaunchKernelGGL(k_tb_panel, dim3(2 * gt, nb), dim3(NT), 0, c->stream, c->tb_bands, b0, c->tb_AB,
                                   c->tb_LI, c->tb_UI, c->tb_P, k, amax, gt, mask);
                hipLaunchKernelGGL(k_tb_update, dim3(gt * gt, nb), dim3(256), 0, c->stream, c->tb_bands, b0,
                                   c->tb_AB, c->tb_P, k, amax, gt, mask);
            });
            diag(k);
            continue;
        }
        each_launch(c, [&](int b0, int nb) {
            hipLaunchKernelGGL(k_tb_step, dim3(gt * gt, nb), dim3(NT), 0, c->stream, c->tb_bands, b0, c->tb_AB,
                               c->tb_LI, c->tb_UI, c->tb_guard, k, amax, gt, mask);
        });
    }
    if (amax > 0 && steps == amax) merge();   // shared rows of one panel
    const int gf = std::max(1, c->tb_gf);
    each_launch(c, [&](int b0, int nb) {
        hipLaunchKernelGGL(k_tb_inv, dim3(nt, nb), dim3(64), 0, c->stream, c->tb_bands, b0, c->tb_AB, c->tb_LI,
                           c->tb_UI, c->tb_guard, mask);
        hipLaunchKernelGGL(k_tb_scale, dim3(nt, 2 * gf, nb), dim3(256), 0, c->stream, c->tb_bands, b0, c->tb_AB,
                           c->tb_LI, c->tb_UI, gf, mask);
    });
}

// sc: the Krylov scalars (one per model) whose done flags end the sweeps, or
// null outside the iteration loop
void launch_tband_solve(Ctx *c, double *x, const KScal *sc) {
    const int *mask = tb_mask(c);
    const int nt = tb_active_nt(c);
    if (nt == 0) return;
    hipLaunchKernelGGL(k_tb_gather, dim3(nblocks_for(c->N, 256)), dim3(256), 0, c->stream, c->N, c->tb_nband,
                       c->tb_nbot, c->node_blk, c->tb_bands, x, c->tb_xb, c->tb_yb, c->tb_zb, c->tb_int);
    // one model: its done flag, or the first band record's pad (always 0),
    // read beside the band record; ensembles: each band's model's flag
    const int *done = (sc && !mask) ? &sc->done : &c->tb_bands[0].pad;
    const KScal *msc = mask ? sc : nullptr;
    // a workgroup per tile of a row's reach and one more keep the chain's next
    // row always waiting; any number is correct.  With many bands one for each CU is
    // the line: two on some CUs slow the rows that the bands' chains wait for.  Four
    // iterations' solve at 256 and 512 of them, ms: 1000 x 500 cells nblock 16 136
    // and 185, 50 84.7 and 110; 400 x 200 nblock 16 9.6 and 12.2; 1500 x 40 nblock
    // 32 2.8 and 4.3 (only 1000 x 500 nblock 8 the other way, 163 and 141).
    const int g = std::max(1, std::min(std::min(c->tb_gf + 2, nt), 256 / c->tb_nband));
    auto sweep = [&](int phase) {   // SW_SHARED's claims count on from launch to launch
        each_launch(c, [&](int b0, int nb) {
            hipLaunchKernelGGL(k_tb_sweep, dim3(g, nb), dim3(SW_NT), 0, c->stream, c->tb_bands, b0, c->tb_AB, c->tb_xb,
                               c->tb_yb, c->tb_zb, c->tb_int, c->tb_int + 3 * c->tb_nband, phase, done, mask, msc);
        });
    };
    auto apply = [&](bool shared, int tiles) {
        each_launch(c, [&](int b0, int nb) {
            hipLaunchKernelGGL(k_tb_apply, dim3(tiles, nb), dim3(256), 0, c->stream, c->tb_bands, b0, c->tb_UI,
                               c->tb_zb, x, shared, done, mask, msc);
        });
    };
    if (c->tb_nbot > 0) {
        sweep(SW_SHARED);
        apply(true, (c->tb_maxs + TB - 1) / TB);
        sweep(SW_REST);
    } else {
        sweep(SW_ALL);
    }
    apply(false, nt);
}

}  // namespace sw2
