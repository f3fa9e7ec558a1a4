// Block ILU(0) preconditioner in multicolour order (preconditioner = 3).
//
// No counterpart in the reference's serial path, which preconditions with a
// skyline LU of node blocks (solv_prec.c:11-66 -> solv_blk_solve.c); this is
// the north star's "block-Jacobi/ILU(0)" alternative, plugged in at the same
// place: M^-1 is applied to a vector in place after each SpMV of BiCGSTAB.
//
// Ordering.  The nodes are coloured greedily in index order (each node takes
// the smallest colour none of its lower-index neighbours has), so nodes of
// one colour never share a matrix block.  Rows are ordered by colour, then
// node index; each colour's rows are padded to a multiple of 64 so a
// wavefront never spans two colours.  In this order every row's off-diagonal
// blocks split into "lower" (neighbours of smaller colour) and "upper".
//
// Factorisation (IKJ variant of ILU(0) on 3x3 blocks, no fill): for row i,
// for each lower neighbour k in increasing position,
//     L_ik = A_ik U_kk^-1,   A_ij -= L_ik U_kj  for j in row i with pos(j) > pos(k)
// (j = i included), then U_ii = A_ii and U_ij = A_ij for the upper j.  Rows
// of one colour depend only on rows of smaller colours, so each colour is
// one launch; the (k, j) update lists are built once on the host.  The factors are formed in FP64 from the scaled system and
// stored in FP64 (precision 0) or FP32 (precision 1).
//
// Apply (in place on a node-ordered vector): forward sweeps z_i = v_i -
// sum L_ik z_k over the colours in order, backward sweeps
// x_i = U_ii^-1 (z_i - sum U_ij x_j) in reverse order.  A sweep is one launch in
// which rows wait for the values they need (k_ilu_flow), or for large systems a
// launch per colour; the colour-ordered work vector w holds z (with a launch
// per colour then x).
//
// Storage: like the SpMV's SELL-64 blocks, slices of 64 consecutive rows (in
// colour order) with a per-slice slot count; value e of slot b of the row in
// lane l sits at 9*64*(ptr[s] + b) + 64*e + l.  Padding slots have column -1.
#include <climits>

#include <algorithm>
#include <numeric>

#include "sw2_ctx.h"
#include "sw2_flow.h"

namespace sw2 {

// y = A x for 3x3 blocks (row-major), accumulated in FP64
template <typename T>
__device__ __forceinline__ void blk_mul(const T *a, size_t st, const double *x, double *y) {
#pragma unroll
    for (int r = 0; r < 3; r++)
        y[r] = (double)a[st * (3 * r)] * x[0] + (double)a[st * (3 * r + 1)] * x[1] + (double)a[st * (3 * r + 2)] * x[2];
}

struct IluView {
    int Rp;                   // rows in colour order, padded
    const int *rnode;         // [Rp] node of each row (-1: padding)
    const int *lptr, *uptr;   // [Rp/64 + 1] slot offsets per slice
    const int *lcol, *ucol;   // [64 * slots] row position of each slot's column (-1: padding)
};

__device__ __forceinline__ size_t ilu_v(size_t slot_base, int e, int lane) { return 9 * 64 * slot_base + 64 * e + lane; }
__device__ __forceinline__ size_t ilu_w(int r, int k) { return 3 * (size_t)(r & ~63) + 64 * k + (r & 63); }

// One colour of the factorisation, a workgroup per 64-row slice.  A row's blocks
// (its lower slots, upper slots and diagonal) are taken from the scaled system
// into LDS, a block per wave, where one wave's updates change them, and leave in
// the apply's precision; the
// upper blocks and U_ii^-1, which later colours read, also in FP64 (Uw, Dinv; the
// apply's own arrays when those are FP64).  upd[tptr[r] .. tptr[r+1]) lists, in
// the order of the row's lower slots, (lower slot b, U slot of row k holding
// U_kj, target): target >= 0 an L slot of row r, -1 - t a U slot t of row r, and
// INT_MIN the diagonal; an update's block is fetched while the one before is
// applied.  80,400 nodes, four colours: 64 us a set-up (9 us for the first
// colour, which has no updates, 15 to 21 for the others); with the row in
// memory, a copy in before and copies out after it 158, with one wave for all
// 134 (its code is run once and waits to be fetched).
// IN_LDS = false: rows of more blocks than the LDS holds stay in `spill`.
constexpr int FAC_W = 8;   // waves
template <typename MT, typename FT, bool IN_LDS>
__global__ void __launch_bounds__(64 * FAC_W) k_ilu_factor(IluView V, int s0, const int *lsrc, const int *usrc,
                                                   const MT *diag, const MT *offd, const int *tptr, const int4 *upd,
                                                   double *Uw, double *Dinv, FT *L, FT *U, FT *Df, double *spill,
                                                   int maxblk) {
    extern __shared__ double lds[];
    double *row = IN_LDS ? lds : spill + 576 * (size_t)maxblk * blockIdx.x;
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s = s0 + blockIdx.x, r = 64 * s + lane;
    const int node = V.rnode[r];
    const int l0 = V.lptr[s], nl = V.lptr[s + 1] - l0, u0 = V.uptr[s], nu = V.uptr[s + 1] - u0;
    auto at = [&](int b, int e) -> double & { return row[64 * (9 * b + e) + lane]; };
    const int dg = nl + nu;
    for (int b = wv; b <= dg; b += FAC_W) {
        double x[9];
        if (b == dg) {
#pragma unroll
            for (int e = 0; e < 9; e++) x[e] = node >= 0 ? (double)diag[didx9(node, e)] : (e % 4 == 0 ? 1.0 : 0.0);
        } else {
            const int q = b < nl ? lsrc[64 * (size_t)(l0 + b) + lane] : usrc[64 * (size_t)(u0 + b - nl) + lane];
#pragma unroll
            for (int e = 0; e < 9; e++) x[e] = q >= 0 ? (double)offd[sell_vidx((size_t)q, e)] : 0.0;
        }
#pragma unroll
        for (int e = 0; e < 9; e++) at(b, e) = x[e];
    }
    __syncthreads();
    if (wv == 0 && node >= 0 && nl > 0) {
        const int4 none = make_int4(-1, 0, 0, 0);
        const int t0 = tptr[r], t1 = tptr[r + 1];
        auto entry = [&](int i) { return i < t1 ? upd[i] : none; };
        auto block = [&](const int4 &u, double (&x)[9]) {
            if (u.x >= 0)
#pragma unroll
                for (int e = 0; e < 9; e++) x[e] = Uw[ilu_v((size_t)u.y >> 6, 0, u.y & 63) + 64 * e];
        };
        // L_ik = A_ik U_kk^-1 of the lower slots up to `want`; the next slot's column
        // and inverse are on their way
        auto column = [&](int b) { return b < nl ? V.lcol[64 * (size_t)(l0 + b) + lane] : -1; };
        auto inverse = [&](int k, double (&x)[9]) {
            if (k >= 0)
#pragma unroll
                for (int e = 0; e < 9; e++) x[e] = Dinv[ilu_v(k >> 6, 0, k & 63) + 64 * e];
        };
        int b = -1, k = column(0), kn = column(1);
        double dk[9] = {}, l[9] = {};
        inverse(k, dk);
        auto to_slot = [&](int want) {
            while (b < want) {
                b++;
                if (k >= 0) {
                    double x[9];
#pragma unroll
                    for (int e = 0; e < 9; e++) x[e] = at(b, e);
#pragma unroll
                    for (int i = 0; i < 3; i++)
#pragma unroll
                        for (int j = 0; j < 3; j++)
                            l[3 * i + j] = x[3 * i] * dk[j] + x[3 * i + 1] * dk[3 + j] + x[3 * i + 2] * dk[6 + j];
#pragma unroll
                    for (int e = 0; e < 9; e++) at(b, e) = l[e];
                }
                k = kn;
                inverse(k, dk);
                kn = column(b + 2);
            }
        };
        // A_ij -= L_ik U_kj
        auto apply = [&](const int4 &u, const double (&x)[9]) {
            to_slot(u.x - l0);
            const int to = u.z == INT_MIN ? dg : (u.z >= 0 ? u.z - l0 : nl + (-1 - u.z) - u0);
#pragma unroll
            for (int i = 0; i < 3; i++)
#pragma unroll
                for (int j = 0; j < 3; j++)
                    at(to, 3 * i + j) -= l[3 * i] * x[j] + l[3 * i + 1] * x[3 + j] + l[3 * i + 2] * x[6 + j];
        };
        // two entries a turn, each block in registers of its own: one is fetched while the other is applied
        int4 ua = entry(t0), ub = entry(t0 + 1);
        double xa[9] = {}, xb[9] = {};
        block(ua, xa);
        for (int t = t0; t < t1; t += 2) {
            block(ub, xb);
            const int4 uc = entry(t + 2), ud = entry(t + 3);
            apply(ua, xa);
            block(uc, xa);
            if (ub.x >= 0) apply(ub, xb);
            ua = uc;
            ub = ud;
        }
        to_slot(nl - 1);
    }
    __syncthreads();
    for (int b = wv; b <= dg; b += FAC_W) {
        double x[9];
#pragma unroll
        for (int e = 0; e < 9; e++) x[e] = at(b, e);
        if (b == dg) {
            double inv[9];
            inv3(x, inv);
#pragma unroll
            for (int e = 0; e < 9; e++) {
                Dinv[ilu_v(s, e, lane)] = inv[e];
                if constexpr (sizeof(FT) < sizeof(double)) Df[ilu_v(s, e, lane)] = (FT)inv[e];
            }
        } else if (b < nl) {
#pragma unroll
            for (int e = 0; e < 9; e++) L[ilu_v(l0 + b, e, lane)] = (FT)x[e];
        } else {
#pragma unroll
            for (int e = 0; e < 9; e++) {
                Uw[ilu_v(u0 + b - nl, e, lane)] = x[e];
                if constexpr (sizeof(FT) < sizeof(double)) U[ilu_v(u0 + b - nl, e, lane)] = (FT)x[e];
            }
        }
    }
}

// forward sweep of one colour: w_r = v_node - sum_b L_b w_col
template <typename FT>
__global__ void __launch_bounds__(256) k_ilu_fwd(IluView V, int r0, int r1, const FT *L, const double *v, double *w,
                                                 const KScal *sc) {
    if (sc && sc->done) return;
    const int r = r0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= r1) return;
    const int node = V.rnode[r];
    if (node < 0) return;
    const int s = r >> 6, lane = r & 63;
    double z[3] = {v[vidx3(node, 0)], v[vidx3(node, 1)], v[vidx3(node, 2)]};
    for (int b = V.lptr[s]; b < V.lptr[s + 1]; b++) {
        const int k = V.lcol[64 * (size_t)b + lane];
        if (k < 0) continue;
        const double x[3] = {w[ilu_w(k, 0)], w[ilu_w(k, 1)], w[ilu_w(k, 2)]};
        double y[3];
        blk_mul(L + ilu_v(b, 0, lane), 64, x, y);
        z[0] -= y[0]; z[1] -= y[1]; z[2] -= y[2];
    }
    for (int j = 0; j < 3; j++) w[ilu_w(r, j)] = z[j];
}

// backward sweep of one colour: x_r = U_rr^-1 (w_r - sum_b U_b x_col), written
// to w and to the node-ordered output
template <typename FT>
__global__ void __launch_bounds__(256) k_ilu_bwd(IluView V, int r0, int r1, const FT *U, const FT *Dinv, double *w,
                                                 double *out, const KScal *sc) {
    if (sc && sc->done) return;
    const int r = r0 + blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= r1) return;
    const int node = V.rnode[r];
    if (node < 0) return;
    const int s = r >> 6, lane = r & 63;
    double z[3] = {w[ilu_w(r, 0)], w[ilu_w(r, 1)], w[ilu_w(r, 2)]};
    for (int b = V.uptr[s]; b < V.uptr[s + 1]; b++) {
        const int k = V.ucol[64 * (size_t)b + lane];
        if (k < 0) continue;
        const double x[3] = {w[ilu_w(k, 0)], w[ilu_w(k, 1)], w[ilu_w(k, 2)]};
        double y[3];
        blk_mul(U + ilu_v(b, 0, lane), 64, x, y);
        z[0] -= y[0]; z[1] -= y[1]; z[2] -= y[2];
    }
    double x[3];
    blk_mul(Dinv + ilu_v(s, 0, lane), 64, z, x);
    for (int j = 0; j < 3; j++) {
        w[ilu_w(r, j)] = x[j];
        out[vidx3(node, j)] = x[j];
    }
}

// A whole sweep in one launch: a workgroup takes the next 256 rows in the
// sweep's order (a ticket), and a row polls its neighbours' values, which are
// words handed over (sw2_flow.h), as far as they come before it.  Rows are taken
// in order, so the first unfinished ones belong to a running workgroup and wait
// only for finished ones.  FWD: z into w from the vector; else x into xw and the
// vector, from w.  Each sweep empties what the other waits on next: FWD its row
// of xw, the backward sweep its row of w once it has read it; each sets the
// other's ticket back.  Same operations as k_ilu_fwd and k_ilu_bwd.
template <typename FT, bool FWD>
__global__ void __launch_bounds__(256) k_ilu_flow(IluView V, const FT *F, const FT *Dinv, double *vec, double *w,
                                                  double *xw, int *tick, const KScal *sc) {
    if (sc && sc->done) return;
    __shared__ int unit;
    if (threadIdx.x == 0) {
        const int t = atomicAdd(tick + (FWD ? 0 : 1), 1);
        if (t == 0) tick[FWD ? 1 : 0] = 0;
        unit = FWD ? t : gridDim.x - 1 - t;
    }
    __syncthreads();
    const int r = 256 * unit + threadIdx.x;
    if (r >= V.Rp) return;
    const int node = V.rnode[r];
    if (node < 0) return;   // padding: no row waits for it
    const int s = r >> 6, lane = r & 63;
    const int *ptr = FWD ? V.lptr : V.uptr, *col = FWD ? V.lcol : V.ucol;
    const double *near = FWD ? w : xw;
    const int b1 = ptr[s + 1];
    double z[3];
#pragma unroll
    for (int j = 0; j < 3; j++) {
        if constexpr (FWD) {
            z[j] = vec[vidx3(node, j)];
            put_raw(xw + ilu_w(r, j), Slot<double>::EMPTY);
        } else {
            z[j] = __builtin_bit_cast(double, peek(w + ilu_w(r, j)));
            put_raw(w + ilu_w(r, j), Slot<double>::EMPTY);
        }
    }
    constexpr int C = 6;   // slots whose blocks are loaded before their values are waited for
    for (int b = ptr[s]; b < b1; b += C) {
        int k[C];
        FT f[C][9];
#pragma unroll
        for (int i = 0; i < C; i++) {
            const int bi = min(b + i, b1 - 1);
            k[i] = b + i < b1 ? col[64 * (size_t)bi + lane] : -1;
#pragma unroll
            for (int e = 0; e < 9; e++) f[i][e] = F[ilu_v(bi, e, lane)];
        }
        double x[C][3];
        for (;;) {
            bool all = true;
#pragma unroll
            for (int i = 0; i < C; i++)
                if (k[i] >= 0)
#pragma unroll
                    for (int j = 0; j < 3; j++) {
                        const auto u = peek(near + ilu_w(k[i], j));
                        all = all && u != Slot<double>::EMPTY;
                        x[i][j] = __builtin_bit_cast(double, u);
                    }
            if (!__any(!all)) break;
            __builtin_amdgcn_s_sleep(1);
        }
#pragma unroll
        for (int i = 0; i < C; i++)
            if (k[i] >= 0) {
                double y[3];
                blk_mul(f[i], 1, x[i], y);
                z[0] -= y[0]; z[1] -= y[1]; z[2] -= y[2];
            }
    }
    if constexpr (FWD) {
#pragma unroll
        for (int j = 0; j < 3; j++) put(w + ilu_w(r, j), z[j]);
    } else {
        double x[3];
        blk_mul(Dinv + ilu_v(s, 0, lane), 64, z, x);
#pragma unroll
        for (int j = 0; j < 3; j++) {
            put(xw + ilu_w(r, j), x[j]);
            vec[vidx3(node, j)] = x[j];
        }
    }
}

__global__ void k_ilu_empty(size_t n, double *a, double *b, int *tick) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < 2) tick[i] = 0;
    if (i >= n) return;
    put_raw(a + i, Slot<double>::EMPTY);
    put_raw(b + i, Slot<double>::EMPTY);
}

static IluView iview(Ctx *c) { return IluView{c->ilu_Rp, c->ilu_rnode, c->ilu_lptr, c->ilu_uptr, c->ilu_lcol, c->ilu_ucol}; }

void ilu_free(Ctx *c) {
    for (void *p : c->ilu_allocs) (void)hipFree(p);
    c->ilu_allocs.clear();
    c->ilu_ready = 0;
    c->ilu_ncolor = 0;
}

// blocks of a 64-row slice's rows that fit in the 64 KB of LDS a launch has
constexpr int ILU_LDS_BLOCKS = (64 << 10) / (576 * 8);

// Greedy colouring, colour-ordered rows, the lower/upper slot structure and
// the update lists, built once per pattern.  Returns an error text or "".
std::string ilu_structure(Ctx *c) {
    ilu_free(c);
    const int N = c->N;
    const std::vector<int> &rp = c->h_row_ptr, &cl = c->h_col;
    std::vector<int> color(N, -1);
    int ncolor = 0;
    {
        std::vector<int> seen;
        for (int i = 0; i < N; i++) {
            seen.assign(ncolor + 2, 0);
            for (int p = rp[i]; p < rp[i + 1]; p++)
                if (cl[p] < i) seen[color[cl[p]]] = 1;
            int k = 0;
            while (seen[k]) k++;
            color[i] = k;
            ncolor = std::max(ncolor, k + 1);
        }
    }
    // rows: colour-major, node order within a colour, each colour padded to 64
    std::vector<int> cstart(ncolor + 1, 0), count(ncolor, 0);
    for (int i = 0; i < N; i++) count[color[i]]++;
    for (int k = 0; k < ncolor; k++) cstart[k + 1] = cstart[k] + ((count[k] + 63) & ~63);
    const int Rp = cstart[ncolor];
    std::vector<int> rnode(Rp, -1), pos(N), fill(ncolor, 0);
    for (int i = 0; i < N; i++) {
        const int r = cstart[color[i]] + fill[color[i]]++;
        rnode[r] = i;
        pos[i] = r;
    }
    // per-row lower / upper neighbours sorted by position, with their SELL source slots
    const int nsl = Rp / 64;
    std::vector<std::vector<std::pair<int, int>>> lo(Rp), up(Rp);   // (position, SELL slot)
    for (int r = 0; r < Rp; r++) {
        const int i = rnode[r];
        if (i < 0) continue;
        for (int p = rp[i]; p < rp[i + 1]; p++) {
            const int pj = pos[cl[p]];
            (pj < r ? lo[r] : up[r]).push_back({pj, c->h_offd_pos[p]});
        }
        std::sort(lo[r].begin(), lo[r].end());
        std::sort(up[r].begin(), up[r].end());
    }
    std::vector<int> lptr(nsl + 1, 0), uptr(nsl + 1, 0);
    for (int s = 0; s < nsl; s++) {
        size_t kl = 0, ku = 0;
        for (int l = 0; l < 64; l++) {
            kl = std::max(kl, lo[64 * s + l].size());
            ku = std::max(ku, up[64 * s + l].size());
        }
        lptr[s + 1] = lptr[s] + (int)kl;
        uptr[s + 1] = uptr[s] + (int)ku;
    }
    const size_t nl = 64 * (size_t)lptr[nsl], nu = 64 * (size_t)uptr[nsl];
    std::vector<int> lcol(std::max<size_t>(nl, 1), -1), ucol(std::max<size_t>(nu, 1), -1);
    std::vector<int> lsrc(std::max<size_t>(nl, 1), -1), usrc(std::max<size_t>(nu, 1), -1);
    // slot index of (row, b) for the upper part, and lookup of a row's upper slot by column position
    for (int r = 0; r < Rp; r++) {
        const int s = r >> 6, l = r & 63;
        for (size_t b = 0; b < lo[r].size(); b++) {
            lcol[64 * (size_t)(lptr[s] + b) + l] = lo[r][b].first;
            lsrc[64 * (size_t)(lptr[s] + b) + l] = lo[r][b].second;
        }
        for (size_t b = 0; b < up[r].size(); b++) {
            ucol[64 * (size_t)(uptr[s] + b) + l] = up[r][b].first;
            usrc[64 * (size_t)(uptr[s] + b) + l] = up[r][b].second;
        }
    }
    auto uslot = [&](int r, int pj) -> int {   // global U slot of row r's block in column pj, or -1
        const int s = r >> 6, l = r & 63;
        for (size_t b = 0; b < up[r].size(); b++)
            if (up[r][b].first == pj) return 64 * (uptr[s] + (int)b) + l;
        return -1;
    };
    std::vector<int> tptr(Rp + 1, 0);
    std::vector<int4> upd;
    for (int r = 0; r < Rp; r++) {
        const int s = r >> 6, l = r & 63;
        for (size_t bk = 0; bk < lo[r].size(); bk++) {
            const int k = lo[r][bk].first;
            const int bslot = lptr[s] + (int)bk;   // slot base index (times 64 plus lane = storage slot)
            // j over row r's later lower slots, the diagonal, and the upper slots
            for (size_t bj = bk + 1; bj < lo[r].size(); bj++) {
                const int q = uslot(k, lo[r][bj].first);
                if (q >= 0) upd.push_back(make_int4(bslot, q, lptr[s] + (int)bj, 0));
            }
            {
                const int q = uslot(k, r);
                if (q >= 0) upd.push_back(make_int4(bslot, q, INT_MIN, 0));
            }
            for (size_t bj = 0; bj < up[r].size(); bj++) {
                const int q = uslot(k, up[r][bj].first);
                if (q >= 0) upd.push_back(make_int4(bslot, q, -1 - (uptr[s] + (int)bj), 0));
            }
        }
        tptr[r + 1] = (int)upd.size();
    }
    // the kernel addresses a slot's values by (slot base, lane): convert the
    // U source slots from storage index to (base * 64 + lane) form, which
    // they already are (64 * base + lane); L/U targets are slot bases
    auto up_dev = [&](void **dst, const void *src, size_t bytes) -> bool {
        if (hipMalloc(dst, bytes ? bytes : 8) != hipSuccess) return false;
        c->ilu_allocs.push_back(*dst);
        return bytes == 0 || hipMemcpy(*dst, src, bytes, hipMemcpyHostToDevice) == hipSuccess;
    };
    auto alloc = [&](void **dst, size_t bytes) -> bool {
        if (hipMalloc(dst, bytes ? bytes : 8) != hipSuccess) return false;
        c->ilu_allocs.push_back(*dst);
        return true;
    };
    const size_t fsz = c->opts.precision >= 1 ? sizeof(float) : sizeof(double);
    // blocks of a row at most, and whether they leave the 64 KB of LDS a launch has
    int maxblk = 1;
    for (int sl = 0; sl < nsl; sl++) maxblk = std::max(maxblk, lptr[sl + 1] - lptr[sl] + uptr[sl + 1] - uptr[sl] + 1);
    const bool spill = maxblk > ILU_LDS_BLOCKS;
    c->ilu_maxblk = maxblk;
    bool ok = up_dev((void **)&c->ilu_rnode, rnode.data(), sizeof(int) * Rp) &&
              up_dev((void **)&c->ilu_lptr, lptr.data(), sizeof(int) * lptr.size()) &&
              up_dev((void **)&c->ilu_uptr, uptr.data(), sizeof(int) * uptr.size()) &&
              up_dev((void **)&c->ilu_lcol, lcol.data(), sizeof(int) * lcol.size()) &&
              up_dev((void **)&c->ilu_ucol, ucol.data(), sizeof(int) * ucol.size()) &&
              up_dev((void **)&c->ilu_lsrc, lsrc.data(), sizeof(int) * lsrc.size()) &&
              up_dev((void **)&c->ilu_usrc, usrc.data(), sizeof(int) * usrc.size()) &&
              up_dev((void **)&c->ilu_tptr, tptr.data(), sizeof(int) * tptr.size()) &&
              up_dev((void **)&c->ilu_upd, upd.data(), sizeof(int4) * upd.size()) &&
              alloc((void **)&c->ilu_spill, spill ? sizeof(double) * 9 * (size_t)Rp * maxblk : sizeof(double)) &&
              alloc((void **)&c->ilu_w, sizeof(double) * 3 * (size_t)Rp) &&
              alloc((void **)&c->ilu_xw, sizeof(double) * 3 * (size_t)Rp) &&
              alloc((void **)&c->ilu_tick, sizeof(int) * 2) &&
              alloc((void **)&c->ilu_L, fsz * 9 * std::max<size_t>(nl, 1)) &&
              alloc((void **)&c->ilu_U, fsz * 9 * std::max<size_t>(nu, 1)) &&
              alloc((void **)&c->ilu_D, fsz * 9 * (size_t)Rp);
    if (ok && fsz < sizeof(double))   // the FP64 upper blocks and inverses that the factorisation reads
        ok = alloc((void **)&c->ilu_Uw, sizeof(double) * 9 * std::max<size_t>(nu, 1)) &&
             alloc((void **)&c->ilu_Dinv, sizeof(double) * 9 * (size_t)Rp);
    else if (ok) {
        c->ilu_Uw = (double *)c->ilu_U;
        c->ilu_Dinv = (double *)c->ilu_D;
    }
    if (!ok) {
        ilu_free(c);
        return "hipMalloc failed for the ILU(0) factors";
    }
    c->ilu_ncolor = ncolor;
    c->h_ilu_cstart = cstart;
    c->h_ilu_color = color;
    c->ilu_Rp = Rp;
    c->ilu_nl = nl;
    c->ilu_nu = nu;
    c->ilu_f32 = c->opts.precision >= 1;
    const size_t n3 = 3 * (size_t)Rp;
    hipLaunchKernelGGL(k_ilu_empty, dim3((unsigned)((n3 + 255) / 256 + 1)), dim3(256), 0, c->stream, n3, c->ilu_w,
                       c->ilu_xw, c->ilu_tick);
    c->ilu_ready = 1;
    return "";
}

// Factors the scaled system colour by colour into the apply's precision.
template <typename MT, typename FT>
static void ilu_factor(Ctx *c, const MT *diag, const MT *offd) {
    IluView V = iview(c);
    const bool in_lds = c->ilu_maxblk <= ILU_LDS_BLOCKS;
    for (int k = 0; k < c->ilu_ncolor; k++) {
        const int s0 = c->h_ilu_cstart[k] / 64, s1 = c->h_ilu_cstart[k + 1] / 64;
        auto launch = [&](auto kern, size_t lds) {
            hipLaunchKernelGGL(kern, dim3(s1 - s0), dim3(64 * FAC_W), lds, c->stream, V, s0, c->ilu_lsrc, c->ilu_usrc, diag,
                               offd, c->ilu_tptr, c->ilu_upd, c->ilu_Uw, c->ilu_Dinv, (FT *)c->ilu_L, (FT *)c->ilu_U,
                               (FT *)c->ilu_D, c->ilu_spill, c->ilu_maxblk);
        };
        if (in_lds) launch(k_ilu_factor<MT, FT, true>, sizeof(double) * 576 * (size_t)c->ilu_maxblk);
        else launch(k_ilu_factor<MT, FT, false>, 0);
    }
}

void launch_ilu_setup(Ctx *c) {
    if (c->ilu_f32) ilu_factor<float, float>(c, c->diag32, c->offd32);
    else ilu_factor<double, double>(c, c->diag, c->offd);
}

// Rows up to which a sweep runs in one launch: there a colour's launch (4.6 us
// at 20,000 rows) is longer than a hand-over, above it the neighbours' values,
// read past the L2, cost more than they save.  A time step's solves, ms, a launch
// per colour / per sweep: 1,891 rows 1.68 / 1.25, 20,301 1.79 / 1.23, 80,400
// 2.29 / 1.75, 125,751 2.32 / 2.07, 180,901 2.52 / 2.48 (FP64 3.11 / 2.86),
// 246,051 2.70 / 2.82, 501,501 4.15 / 4.52.
constexpr int FLOW_ROWS = 200000;

template <typename FT>
static void ilu_sweeps(Ctx *c, double *x, const KScal *sc) {
    IluView V = iview(c);
    const FT *L = (const FT *)c->ilu_L, *U = (const FT *)c->ilu_U, *D = (const FT *)c->ilu_D;
    if (V.Rp <= FLOW_ROWS) {
        const dim3 g(nblocks_for(V.Rp, 256));
        hipLaunchKernelGGL((k_ilu_flow<FT, true>), g, dim3(256), 0, c->stream, V, L, D, x, c->ilu_w, c->ilu_xw,
                           c->ilu_tick, sc);
        hipLaunchKernelGGL((k_ilu_flow<FT, false>), g, dim3(256), 0, c->stream, V, U, D, x, c->ilu_w, c->ilu_xw,
                           c->ilu_tick, sc);
        return;
    }
    for (int k = 0; k < c->ilu_ncolor; k++) {
        const int r0 = c->h_ilu_cstart[k], r1 = c->h_ilu_cstart[k + 1];
        hipLaunchKernelGGL(k_ilu_fwd<FT>, dim3(nblocks_for(r1 - r0, 256)), dim3(256), 0, c->stream, V, r0, r1, L, x,
                           c->ilu_w, sc);
    }
    for (int k = c->ilu_ncolor - 1; k >= 0; k--) {
        const int r0 = c->h_ilu_cstart[k], r1 = c->h_ilu_cstart[k + 1];
        hipLaunchKernelGGL(k_ilu_bwd<FT>, dim3(nblocks_for(r1 - r0, 256)), dim3(256), 0, c->stream, V, r0, r1, U, D,
                           c->ilu_w, x, sc);
    }
}

// x <- M^-1 x (node-ordered, sliced layout); skipped once sc->done is set
void launch_ilu_solve(Ctx *c, double *x, const KScal *sc) {
    if (c->ilu_f32) ilu_sweeps<float>(c, x, sc);
    else ilu_sweeps<double>(c, x, sc);
}

}  // namespace sw2
