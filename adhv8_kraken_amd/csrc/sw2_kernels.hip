// Element-level kernels of the SW2 Newton step on gfx950: residual,
// finite-difference Jacobian, ordered assembly into 3x3 block rows, and the
// per-node state kernels (init / wet-dry flags / shift / increment / norms).
//
// Layout in HBM: node fields are structure-of-arrays doubles; element
// connectivity and geometry are element-indexed arrays, so one thread per
// element (or per element column) issues coalesced loads for everything but
// the node gathers.  Element results go to contiguous per-element slabs
// (ER: 9 doubles per triangle, EM: 81 per triangle) and are then gathered
// per node / per matrix block in ascending element order -- the order in
// which the reference accumulates (fe_sw2_resid.c:74-191,
// fe_assemble_matrix.c:166-224) -- so sums are bit-identical to it without
// atomics.
#include <algorithm>
#include <type_traits>

#include "sw2_ctx.h"

namespace sw2 {

int nblocks_for(int n, int bs) { return n <= 0 ? 1 : (n + bs - 1) / bs; }

static void launch_resid_split(Ctx *c, const ElemData &D, bool edges);

// The refined forms (precision >= 1) store the element Jacobian blocks in
// FP32 (the matrix they assemble is stored in FP32 anyway); the FP64 form in
// FP64.  Returns the FP32 view of the slab, or null for FP64 storage.
static float *em32_of(Ctx *c) { return c->opts.precision >= 1 ? (float *)c->EM : nullptr; }

// ------------------------------------------------------------------ residual
// The same over a triangle list (grid-stride over the device-side count):
// WET lists hold triangles with positive depths, run without clipping code.
// Software pipeline: the triangle id two iterations ahead and its node ids
// one iteration ahead are loaded while the current triangle is computed.
// block / nblocks: of the workgroups that share the list
template <bool WET, int BS>
__device__ __forceinline__ void resid_list(const ElemData &D, const int *list, const int *count, double *ER, int block,
                                           int nblocks) {
    const int n = *count;
    const int stride = nblocks * BS;
    int li = block * BS + threadIdx.x;
    int ie_a = li < n ? list[li] : 0;
    int ie_b = li + stride < n ? list[li + stride] : 0;
    int nd_a[3] = {0, 0, 0};
    if (li < n)
        for (int k = 0; k < 3; k++) nd_a[k] = D.e2d[3 * ie_a + k];
    for (; li < n; li += stride) {
        const int ie = ie_a;
        const int nodes[3] = {nd_a[0], nd_a[1], nd_a[2]};
        ie_a = ie_b;
        ie_b = li + 2 * stride < n ? list[li + 2 * stride] : 0;
        if (li + stride < n)
            for (int k = 0; k < 3; k++) nd_a[k] = D.e2d[3 * ie_a + k];
        d3 r[3];
        body_resid<WET>(D, D.pre + PRE_STRIDE * (size_t)ie, ie, 0.0, 0, PERTURB_NONE, 0, true, r, nodes);
        double *o = ER + 9 * (size_t)ie;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            o[3 * i + 0] = r[i].x_eq;
            o[3 * i + 1] = r[i].y_eq;
            o[3 * i + 2] = r[i].c_eq;
        }
    }
}

template <bool WET, int BS>
__global__ void __launch_bounds__(BS) k_resid2d_list(ElemData D, const int *list, const int *count, double *ER) {
    resid_list<WET, BS>(D, list, count, ER, blockIdx.x, gridDim.x);
}

__device__ __forceinline__ void resid_edge(const ElemData &D, int ie, int B, double *ER1) {
    if (ie >= B) return;
    d3 r[3];
    boundary_resid(D, ie, 0.0, 0, PERTURB_NONE, 0, true, r);
    double *o = ER1 + 6 * (size_t)ie;
#pragma unroll
    for (int i = 0; i < 2; i++) {
        o[3 * i + 0] = r[i].x_eq;
        o[3 * i + 1] = r[i].y_eq;
        o[3 * i + 2] = r[i].c_eq;
    }
}

// The general list and the boundary edges in one launch: each is mostly launch
// time (an empty list 3.4 us, 128 edges 4.2).  With WET the wet list too, where
// its workgroups fit beside: this kernel holds one wave a SIMD, the wet list's
// own two.
template <bool WET, int BS>
__global__ void __launch_bounds__(BS) k_resid_all(ElemData D, const int *wet, const int *gen, const int *count,
                                                  double *ER, int nwet, int ngen, int B, double *ER1) {
    const int b = blockIdx.x;
    if (WET && b < nwet) resid_list<true, BS>(D, wet, count, ER, b, nwet);
    else if (b < nwet + ngen) resid_list<false, BS>(D, gen, count + 1, ER, b - nwet, ngen);
    else resid_edge(D, (b - nwet - ngen) * BS + threadIdx.x, B, ER1);
}

// residual[3n..] = -(sum of element contributions) in ascending element
// order, 2D first then 1D; dry-node momentum contributions are dropped and
// dry-node velocities zeroed (fe_sw2_resid.c:85-93, :154-162).
// NORMS: also get_residual_norms (fe_newton.c:79-150) with
// include_node_in_residual (:177-187), max norms over nodes with
// min(h, h_old) > 0, l2 over all DOFs: block partials here, while the values
// are in registers, reduced in block order by k_norms_fin.
template <bool NORMS>
__global__ void __launch_bounds__(256) k_resid_gather(int N, const int *n2e_ptr, const int *n2e,
                                                      const int *n2b_ptr, const int *n2b, const double *ER,
                                                      const double *ER1, const double *old_head, double *u, double *v,
                                                      double *R, const double *sol, const double *h, double *part) {
    const int lb = xcd_block();   // a node's elements are shared with its neighbours
    const int n = lb * blockDim.x + threadIdx.x;
    double rmax = 0.0, rsum = 0.0, imax = 0.0;
    if (n < N) {
        bool dry = old_head[n] <= 0.;
        double rx = 0.0, ry = 0.0, rc = 0.0;
        const int k0 = n2e_ptr[n], k1 = n2e_ptr[n + 1];
        int k = k0;
        // batches of up to 8 contributions: the indices, then the values, are
        // loaded before the (in-order) sums, so their latencies overlap
        for (; k < k1; k += 8) {
            const int m = min(8, k1 - k);
            int sidx[8];
#pragma unroll
            for (int t = 0; t < 8; t++) sidx[t] = t < m ? n2e[k + t] : 0;
            double vx[8], vy[8], vc[8];
#pragma unroll
            for (int t = 0; t < 8; t++) {
                const double *o = ER + 3 * (size_t)sidx[t];   // 9 a triangle, 3 a node of it
                vx[t] = t < m ? o[0] : 0.0;
                vy[t] = t < m ? o[1] : 0.0;
                vc[t] = t < m ? o[2] : 0.0;
            }
#pragma unroll
            for (int t = 0; t < 8; t++) {
                if (t < m) {
                    if (!dry) { rx -= vx[t]; ry -= vy[t]; }
                    rc -= vc[t];
                }
            }
        }
        for (int k = n2b_ptr[n]; k < n2b_ptr[n + 1]; k++) {
            int s = n2b[k];
            const double *o = ER1 + 3 * (size_t)s;
            if (!dry) { rx -= o[0]; ry -= o[1]; }
            rc -= o[2];
        }
        R[vidx3(n, 0)] = rx;
        R[vidx3(n, 1)] = ry;
        R[vidx3(n, 2)] = rc;
        if (dry && (n2e_ptr[n + 1] > n2e_ptr[n] || n2b_ptr[n + 1] > n2b_ptr[n])) {
            u[n] = 0.;
            v[n] = 0.;
        }
        if constexpr (NORMS) {
            const double r[3] = {rx, ry, rc};
            const bool inc = dmin(h[n], old_head[n]) > 0;
#pragma unroll
            for (int j = 0; j < 3; j++) {
                const double q = sol[vidx3(n, j)];
                if (inc && fabs(r[j]) > rmax) rmax = fabs(r[j]);
                if (inc && fabs(q) > imax) imax = fabs(q);
                rsum += r[j] * r[j];
            }
        }
    }
    if constexpr (NORMS) {
        __shared__ double smax[256], ssum[256], sinc[256];
        smax[threadIdx.x] = rmax; ssum[threadIdx.x] = rsum; sinc[threadIdx.x] = imax;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1) {
            if (threadIdx.x < w) {
                smax[threadIdx.x] = fmax(smax[threadIdx.x], smax[threadIdx.x + w]);
                ssum[threadIdx.x] += ssum[threadIdx.x + w];
                sinc[threadIdx.x] = fmax(sinc[threadIdx.x], sinc[threadIdx.x + w]);
            }
            __syncthreads();
        }
        if (threadIdx.x == 0) {
            part[3 * lb] = smax[0];
            part[3 * lb + 1] = ssum[0];
            part[3 * lb + 2] = sinc[0];
        }
    }
}

// the block partials of k_resid_gather, reduced in block order; the result
// also goes straight to the host's pinned copy, so reading it is one wait
// one block per model (blockIdx.x), over that model's 256-node blocks
__global__ void __launch_bounds__(256) k_norms_fin(int nparts, int N, const double *part, Norms *out, Norms *host,
                                                   const int *inst_blk0, const int *inst_nodes,
                                                   long long *ts) {
    __shared__ double smax[256], ssum[256], sinc[256];
    const int m = blockIdx.x;
    const int k0 = inst_blk0 ? inst_blk0[m] : 0, k1 = inst_blk0 ? inst_blk0[m + 1] : nparts;
    if (inst_nodes) N = inst_nodes[m];
    out += m;
    double a = 0.0, b = 0.0, cc = 0.0;
    // 8 strided partials per thread loaded together, folded in block order
    const int bd = blockDim.x;
    for (int k = k0 + threadIdx.x; k < k1; k += 8 * bd) {
        double x[8][3];
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
            for (int e = 0; e < 3; e++) x[u][e] = k + u * bd < k1 ? part[3 * (k + u * bd) + e] : 0.0;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (k + u * bd < k1) {
                a = fmax(a, x[u][0]);
                b += x[u][1];
                cc = fmax(cc, x[u][2]);
            }
    }
    smax[threadIdx.x] = a; ssum[threadIdx.x] = b; sinc[threadIdx.x] = cc;
    __syncthreads();
    for (int w = 128; w > 0; w >>= 1) {
        if (threadIdx.x < w) {
            smax[threadIdx.x] = fmax(smax[threadIdx.x], smax[threadIdx.x + w]);
            ssum[threadIdx.x] += ssum[threadIdx.x + w];
            sinc[threadIdx.x] = fmax(sinc[threadIdx.x], sinc[threadIdx.x + w]);
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        Norms r{};
        r.maxn = smax[0];
        r.l2 = sqrt(ssum[0] / (double)(N * 3));
        r.incn = sinc[0];
        *out = r;
        host[m] = r;
        if (m == 0) *ts = wall_clock64();
    }
}

void launch_resid(Ctx *c, bool norms) {
    if (!c->pre_valid) launch_old_terms(c);
    ElemData D = c->ed;
    D.first_elem = c->first_elem;
    launch_resid_split(c, D, true);
    const double *er1 = c->ER + 9 * (size_t)c->E;
    const int nb = nblocks_for(c->N, 256);
    if (!norms) {
        hipLaunchKernelGGL(k_resid_gather<false>, dim3(nb), dim3(256), 0, c->stream, c->N, c->n2e_ptr, c->n2e,
                           c->n2b_ptr, c->n2b, c->ER, er1, c->old_head, c->u, c->v, c->R, c->sol, c->head, c->red.part);
        return;
    }
    hipLaunchKernelGGL(k_resid_gather<true>, dim3(nb), dim3(256), 0, c->stream, c->N, c->n2e_ptr, c->n2e, c->n2b_ptr,
                       c->n2b, c->ER, er1, c->old_head, c->u, c->v, c->R, c->sol, c->head, c->red.part);
    hipLaunchKernelGGL(k_norms_fin, dim3(c->ninst ? c->ninst : 1), dim3(256), 0, c->stream, nb, c->N, c->red.part,
                       c->norms, c->h_norms, c->ninst ? c->inst_blk0 : nullptr, c->ninst ? c->inst_nodes : nullptr,
                       c->h_ts + TS_NORMS);
}

// ------------------------------------------------------------------ Jacobian
// EM[e*81 + (i*3+j)*9 + r*3 + var] = d elem_rhs[i].eq_r / d var_j, column
// q = 3*j + var (var 0 u, 1 v, 2 h).
// The same over a list of triangles (`count` entries), two lanes per column:
// the even lane evaluates the +eps residual and the odd lane the -eps one, so
// each lane carries one residual evaluation; the pair forms the central
// difference with a lane exchange.  WET lists hold triangles whose depths stay
// positive under every perturbation and run without the wet/dry clipping code.
// OCC > 0 asks the compiler for at least OCC waves per SIMD (fewer registers,
// possibly spills); 0 leaves the register budget to the compiler.
template <bool WET, int BS, int OCC>
__global__ void __launch_bounds__(BS, OCC > 0 ? OCC : 1) k_jac2d_list(ElemData D, const int *list, const int *count,
                                                                      int b0, int b1, int b2, const int *blkpos,
                                                                      double *EM, float *EM32) {
    if (WET) stamp(D.ts);
    const int nt = 18 * *count;
    const int stride = gridDim.x * blockDim.x;
    int t = blockIdx.x * blockDim.x + threadIdx.x;
    // Grid-stride over (triangle, column, sign); the stride is a multiple of
    // the wavefront, so both lanes of a pair run and leave together.
    // Software pipeline: the triangle id two iterations ahead and the node ids
    // one iteration ahead are loaded while the current triangle is computed,
    // so an iteration waits on one memory round trip (the node data) instead
    // of three dependent ones (list -> triangle -> nodes).
    int ie_a = t < nt ? list[t / 18] : 0;
    int ie_b = t + stride < nt ? list[(t + stride) / 18] : 0;
    int nd_a[3] = {0, 0, 0};
    if (t < nt)
        for (int k = 0; k < 3; k++) nd_a[k] = D.e2d[3 * ie_a + k];
    for (; t < nt; t += stride) {
    const int ie = ie_a;
    const int nodes[3] = {nd_a[0], nd_a[1], nd_a[2]};
    ie_a = ie_b;
    ie_b = t + 2 * stride < nt ? list[(t + 2 * stride) / 18] : 0;
    if (t + stride < nt)
        for (int k = 0; k < 3; k++) nd_a[k] = D.e2d[3 * ie_a + k];
    const int q = (t >> 1) % 9, j = q / 3, var = q % 3;
    const int sgn = (t & 1) ? -1 : +1;
    const int n = nodes[j];
    const double val = var == 0 ? D.u[n] : (var == 1 ? D.v[n] : D.head[n]);
    const double eps = num_diff_eps(val), eps2 = 2.0 * eps;
    const int pv = var == 0 ? PERTURB_U : (var == 1 ? PERTURB_V : PERTURB_H);
    d3 r[3];
    body_resid<WET>(D, D.pre + PRE_STRIDE * (size_t)ie, ie, eps, j, pv, sgn, false, r, nodes);
    double col[9];
    const double inv = 1.0 / eps2;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        // even lanes hold P (+eps), odd lanes M (-eps); both lanes form P - M
        double mx = __shfl_xor(r[i].x_eq, 1, 64), my = __shfl_xor(r[i].y_eq, 1, 64),
               mc = __shfl_xor(r[i].c_eq, 1, 64);
        col[3 * i + 0] = div_rn(r[i].x_eq - mx, eps2, inv);
        col[3 * i + 1] = div_rn(r[i].y_eq - my, eps2, inv);
        col[3 * i + 2] = div_rn(r[i].c_eq - mc, eps2, inv);
    }
    if (t & 1) continue;
    const int *lbi = D.loc_bc_inst ? D.loc_bc_inst + 3 * D.elem_inst[ie] : nullptr;
    const int lb[3] = {lbi ? lbi[0] : b0, lbi ? lbi[1] : b1, lbi ? lbi[2] : b2};
    jac_column_db<3>(D, nodes, lb, j, var, col);
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const size_t o = 9 * (size_t)blkpos[9 * ie + 3 * i + j];
#pragma unroll
        for (int rr = 0; rr < 3; rr++) {
            if (EM32) EM32[o + 3 * rr + var] = (float)col[3 * i + rr];
            else EM[o + 3 * rr + var] = col[3 * i + rr];
        }
    }
    }
}

// The same Jacobian columns in a column-uniform layout: wave w takes column
// q = w % 9 (node j = q / 3, variable q % 3) of the 32 triangles of group
// w / 9, lanes 0-31 evaluating the +eps residuals and lanes 32-63 the -eps
// ones of the same triangles.  The perturbed node and variable are then the
// same across the wave (scalar registers), so the residual's branches on them
// are taken or skipped by whole waves -- the u and v columns skip the
// pressure block (fe_sw2_body_resid.c:761-862 runs for depth perturbations
// only) instead of running it under a lane mask -- and each triangle's data
// is loaded by 64 lanes of 32 different triangles rather than broadcast to 18
// lanes of one.  Every (triangle, column, sign) evaluates exactly what the
// lane-per-column kernel evaluates, so the blocks are bit-identical.
template <bool WET, int BS>
__global__ void __launch_bounds__(BS) k_jac2d_cols(ElemData D, const int *list, const int *count, int b0, int b1,
                                                   int b2, const int *blkpos, double *EM, float *EM32) {
    if (WET) stamp(D.ts);
    constexpr int WPB = BS / 64;
    const int n = *count;
    const int nunits = 9 * ((n + 31) >> 5);
    const int lane = threadIdx.x & 63;
    const int wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool minus = lane >= 32;
    for (int w = blockIdx.x * WPB + wib; w < nunits; w += gridDim.x * WPB) {
        const int q = w % 9, grp = w / 9;
        const int j = q / 3, var = q % 3;
        const int li = grp * 32 + (lane & 31);
        const bool act = li < n;
        // idle lanes of a group's last wave recompute its first triangle and store nothing
        const int ie = list[act ? li : grp * 32];
        const int nodes[3] = {D.e2d[3 * ie], D.e2d[3 * ie + 1], D.e2d[3 * ie + 2]};
        const int nd = pick3(nodes, j);
        const double val = var == 0 ? D.u[nd] : (var == 1 ? D.v[nd] : D.head[nd]);
        const double eps = num_diff_eps(val), eps2 = 2.0 * eps;
        const int pv = var == 0 ? PERTURB_U : (var == 1 ? PERTURB_V : PERTURB_H);
        d3 r[3];
        body_resid<WET>(D, D.pre + PRE_STRIDE * (size_t)ie, ie, eps, j, pv, minus ? -1 : +1, false, r, nodes);
        double col[9];
        const double inv = 1.0 / eps2;
#pragma unroll
        for (int i = 0; i < 3; i++) {
            // lanes l and l ^ 32 hold the +eps and -eps residuals of one triangle
            double mx = __shfl_xor(r[i].x_eq, 32, 64), my = __shfl_xor(r[i].y_eq, 32, 64),
                   mc = __shfl_xor(r[i].c_eq, 32, 64);
            col[3 * i + 0] = div_rn(r[i].x_eq - mx, eps2, inv);
            col[3 * i + 1] = div_rn(r[i].y_eq - my, eps2, inv);
            col[3 * i + 2] = div_rn(r[i].c_eq - mc, eps2, inv);
        }
        if (minus || !act) continue;
        const int *lbi = D.loc_bc_inst ? D.loc_bc_inst + 3 * D.elem_inst[ie] : nullptr;
        const int lb[3] = {lbi ? lbi[0] : b0, lbi ? lbi[1] : b1, lbi ? lbi[2] : b2};
        jac_column_db<3>(D, nodes, lb, j, var, col);
#pragma unroll
        for (int i = 0; i < 3; i++) {
            const size_t o = 9 * (size_t)blkpos[9 * ie + 3 * i + j];
#pragma unroll
            for (int rr = 0; rr < 3; rr++) {
                if (EM32) EM32[o + 3 * rr + var] = (float)col[3 * i + rr];
                else EM[o + 3 * rr + var] = col[3 * i + rr];
            }
        }
    }
}

// The column-uniform layout with every triangle's inputs staged in LDS first.
// Each wave copies the inputs of its 32 triangles (lanes l and l + 32 share a
// triangle and take alternate fields) with loads issued back to back, waits
// once, and then evaluates the residuals reading those inputs from LDS.  Same
// arithmetic, same results as the global-memory layouts.
//
// Everything a column reads is in the record, down to the positions its
// entries go to, the Dirichlet edits' flags and the material's constants: a
// load in the column loop would queue behind the previous columns' stores (the
// memory counter retires in order) and cost a round trip of the store to
// memory per column.  Jumps cost next (a taken one refetches): the perturbed
// variable is a template argument, the perturbed node a select, and the
// Dirichlet edits are behind one test of the record's flags.  Terms that a
// perturbation leaves as they are come from the record (Base).  At 1M triangles,
// refined / FP64 form: 747 / 806 us (1,086 / 1,174 before), 305M of 374M VALU
// instructions; what is left is latency at two waves per SIMD (254 registers;
// at 168, three waves, the code spills and is slower).
//
// LREC doubles per triangle, odd so that 32 records' fields lie in distinct banks.
enum : int { LR_NODE = 0, LR_GRAD = 18, LR_PRE = 24, LR_DJAC = 46, LR_KS = 47, LR_SRC = 48, LR_DT = 49, LR_COR = 50,
             LR_EV = 51, LR_META = 53, LR_BLK = 54, LR_BASE = 59, LREC = LR_BASE + NBASE };
static_assert(LREC % 2 == 1, "an even record length would put a field of two triangles in one bank");
// LR_META: the material, then these bits (two-bit fields by bc_code; the Dirichlet edits' topmost)
enum : int { MB_WD = 0, MB_SRCF = 2, MB_TURB = 3, MB_NBC = 5, MB_LBC = 11, MB_DRY = 17 };

// BASE: the record also carries the unperturbed triangle's terms (Base)
template <bool BASE>
struct LdsSrcT {
    static constexpr bool has_base = BASE;
    const double *r;   // the triangle's staged record (LDS)
    int meta;
    __device__ __forceinline__ double base(int k) const { return r[LR_BASE + k]; }
    __device__ __forceinline__ double x(int i) const { return r[6 * i]; }
    __device__ __forceinline__ double y(int i) const { return r[6 * i + 1]; }
    __device__ __forceinline__ double z(int i) const { return r[6 * i + 2]; }
    __device__ __forceinline__ double head(int i) const { return r[6 * i + 3]; }
    __device__ __forceinline__ double u(int i) const { return r[6 * i + 4]; }
    __device__ __forceinline__ double v(int i) const { return r[6 * i + 5]; }
    __device__ __forceinline__ int node_bc(int i) const { return code_bc((meta >> (MB_NBC + 2 * i)) & 3); }
    __device__ __forceinline__ bool any_bc() const { return (meta >> MB_NBC) & 63; }
    __device__ __forceinline__ bool any_db() const { return meta >> MB_LBC; }   // a Dirichlet edit of the column
    __device__ __forceinline__ int loc_bc(int i) const { return code_bc((meta >> (MB_LBC + 2 * i)) & 3); }
    __device__ __forceinline__ bool dry(int i) const { return (meta >> (MB_DRY + i)) & 1; }
    __device__ __forceinline__ double grad(int k) const { return r[LR_GRAD + k]; }
    __device__ __forceinline__ double djac() const { return r[LR_DJAC]; }
    __device__ __forceinline__ int mat() const { return ((const int *)(r + LR_META))[0]; }
    __device__ __forceinline__ int wd_flag() const { return (meta >> MB_WD) & 3; }
    __device__ __forceinline__ double ks() const { return r[LR_KS]; }
    __device__ __forceinline__ int src_flag() const { return (meta >> MB_SRCF) & 1; }
    __device__ __forceinline__ double src() const { return r[LR_SRC]; }
    __device__ __forceinline__ double pre(int k) const { return r[LR_PRE + k]; }
    __device__ __forceinline__ double dt() const { return r[LR_DT]; }
    __device__ __forceinline__ int turb() const { return (meta >> MB_TURB) & 3; }
    __device__ __forceinline__ double cor() const { return r[LR_COR]; }
    __device__ __forceinline__ double ev(int k) const { return r[LR_EV + k]; }
    __device__ __forceinline__ int blkpos(int k) const { return ((const int *)(r + LR_BLK))[k]; }
};

// The triangle's inputs into rec: lane half 0 takes one field of each pair,
// half 1 the other (both fields of a step come from one array where possible,
// so a step is one load instruction for the whole wave).
__device__ __forceinline__ void stage_triangle(const ElemData &D, int ie, const int *nd, int half, int b0, int b1,
                                               int b2, const int *blkpos, double *rec) {
    constexpr int NF = 25;
    double val[NF];
    int fld[NF];
    const int na = half ? nd[1] : nd[0];
    // node fields of nodes 0 and 1
    const double *narr[6] = {D.x, D.y, D.z, D.head, D.u, D.v};
#pragma unroll
    for (int c = 0; c < 6; c++) {
        val[c] = narr[c][na];
        fld[c] = (half ? 6 : 0) + c;
    }
    // node 2: (x, y), (z, h), (u, v)
#pragma unroll
    for (int c = 0; c < 3; c++) {
        const double *a = half ? narr[2 * c + 1] : narr[2 * c];
        val[6 + c] = a[nd[2]];
        fld[6 + c] = 12 + 2 * c + half;
    }
    // gradients and old-state terms
#pragma unroll
    for (int m = 0; m < 3; m++) {
        val[9 + m] = D.grad[6 * (size_t)ie + 2 * m + half];
        fld[9 + m] = LR_GRAD + 2 * m + half;
    }
    const double *pre = D.pre + PRE_STRIDE * (size_t)ie;
#pragma unroll
    for (int m = 0; m < 11; m++) {   // pre[22..23] are padding
        val[12 + m] = pre[2 * m + half];
        fld[12 + m] = LR_PRE + 2 * m + half;
    }
    val[23] = half ? D.ks[ie] : D.djac[ie];
    fld[23] = half ? LR_KS : LR_DJAC;
    val[24] = half ? elem_dt(D, ie) : D.src[ie];
    fld[24] = half ? LR_DT : LR_SRC;
    // where the nine blocks go: half 0 five of them, half 1 four
    int bp[5];
#pragma unroll
    for (int k = 0; k < 5; k++) bp[k] = blkpos[9 * (size_t)ie + min(5 * half + k, 8)];
    // integers
    const int mat = D.mat[ie];
    int meta = (D.wd_flag[ie] & 3) << MB_WD | (D.src_flag[ie] ? 1 << MB_SRCF : 0);
    const int *lbi = D.loc_bc_inst ? D.loc_bc_inst + 3 * D.elem_inst[ie] : nullptr;
    const int lb[3] = {lbi ? lbi[0] : b0, lbi ? lbi[1] : b1, lbi ? lbi[2] : b2};
#pragma unroll
    for (int k = 0; k < 3; k++) {
        meta |= bc_code(D.node_bc[nd[k]]) << (MB_NBC + 2 * k) | bc_code(lb[k]) << (MB_LBC + 2 * k);
        meta |= D.old_head[nd[k]] <= 0. ? 1 << (MB_DRY + k) : 0;
    }
    meta |= (D.mat_turb[mat] & 3) << MB_TURB;
#pragma unroll
    for (int k = 0; k < NF; k++) rec[fld[k]] = val[k];
#pragma unroll
    for (int k = 0; k < 5; k++) ((int *)(rec + LR_BLK))[5 * half + k] = bp[k];   // the tenth is padding
    if (half) {
        rec[LR_EV] = evs_viscosity(D, mat, 0);
        rec[LR_EV + 1] = evs_viscosity(D, mat, 1);
    } else {
        rec[LR_COR] = D.mat_cor[mat];
        ((int *)(rec + LR_META))[0] = mat;
        ((int *)(rec + LR_META))[1] = meta;
    }
}

// One Jacobian column (node j, variable var) of the staged triangle: the
// +eps residual on lanes 0-31, the -eps one on lanes 32-63, the difference
// quotient, the Dirichlet edits, and the stores of the +eps lanes.
template <bool WET, int VAR, typename SRC>
__device__ __forceinline__ void lds_column(const ElemData &DL, const SRC &S, int ie, const int *nodes, int j,
                                           bool minus, bool act, double *EM, float *EM32) {
    constexpr int var = VAR, PV = VAR == 0 ? PERTURB_U : (VAR == 1 ? PERTURB_V : PERTURB_H);
    const double val = var == 0 ? S.u(j) : (var == 1 ? S.v(j) : S.head(j));
    const double eps = num_diff_eps(val), eps2 = 2.0 * eps;
    d3 r[3];
    body_resid_src<WET, PV>(DL, S, ie, minus ? -eps : eps, j, PV, 1, false, r, nodes);
    double col[9];
    const double inv = 1.0 / eps2;
#pragma unroll
    for (int i = 0; i < 3; i++) {
        double mx = __shfl_xor(r[i].x_eq, 32, 64), my = __shfl_xor(r[i].y_eq, 32, 64),
               mc = __shfl_xor(r[i].c_eq, 32, 64);
        col[3 * i + 0] = div_rn(r[i].x_eq - mx, eps2, inv);
        col[3 * i + 1] = div_rn(r[i].y_eq - my, eps2, inv);
        col[3 * i + 2] = div_rn(r[i].c_eq - mc, eps2, inv);
    }
    if (minus || !act) return;
    if (S.any_db()) {
        const bool dry[3] = {S.dry(0), S.dry(1), S.dry(2)};
        const int lb[3] = {S.loc_bc(0), S.loc_bc(1), S.loc_bc(2)};
        jac_column_db<3>(dry, lb, j, var, col);
    }
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const size_t o = 9 * (size_t)S.blkpos(3 * i + j);
#pragma unroll
        for (int rr = 0; rr < 3; rr++) {
            if (EM32) EM32[o + 3 * rr + var] = (float)col[3 * i + rr];
            else EM[o + 3 * rr + var] = col[3 * i + rr];
        }
    }
}

// A wave takes COLS of a 32-triangle group's nine columns from one staging:
// all nine, one node's three, or one (unit w: group w / (9 / COLS), part w
// mod that).  With more than one column the terms of the unperturbed triangles
// (Base) are formed once after the staging.
// block / nblocks: of the workgroups that share the list; srec, slog: LDS
template <bool WET, int BS, int COLS>
__device__ __forceinline__ void jac_lds_list(const ElemData &D, const int *list, const int *count, int b0, int b1,
                                             int b2, const int *blkpos, double *EM, float *EM32, int block,
                                             int nblocks, double (&srec)[BS / 64][32][LREC], crlog::tables &slog) {
    constexpr int WPB = BS / 64, PARTS = 9 / COLS;
    const int n = *count;
    const int nunits = PARTS * ((n + 31) >> 5);
    if (block * WPB >= nunits) return;   // the whole block has no unit (uniform exit)
    // the friction law's log table copied to LDS: its lookup is the one
    // data-dependent load of the element code
    {
        const double *src = (const double *)D.logt;
        double *dst = (double *)&slog;
        for (int i = threadIdx.x; i < (int)(sizeof(crlog::tables) / sizeof(double)); i += BS) dst[i] = src[i];
        __syncthreads();
    }
    ElemData DL = D;
    DL.logt = &slog;
    const int lane = threadIdx.x & 63;
    const int wib = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool minus = lane >= 32;
    double *rec = &srec[wib][lane & 31][0];
    const int wstride = nblocks * WPB;
    // software pipeline: the triangle id two units ahead and its node ids one
    // unit ahead are loaded while the current unit is computed
    auto tri_of = [&](int w) {
        const int g = w / PARTS, l = g * 32 + (lane & 31);
        return list[l < n ? l : g * 32];
    };
    int w = block * WPB + wib;
    int ie_a = w < nunits ? tri_of(w) : 0;
    int ie_b = w + wstride < nunits ? tri_of(w + wstride) : 0;
    int nd_a[3] = {0, 0, 0};
    if (w < nunits)
        for (int k = 0; k < 3; k++) nd_a[k] = D.e2d[3 * ie_a + k];
    for (; w < nunits; w += wstride) {
        const int li = (w / PARTS) * 32 + (lane & 31);
        const bool act = li < n;   // idle lanes of a last group recompute its first triangle, store nothing
        const int ie = ie_a;
        const int nodes[3] = {nd_a[0], nd_a[1], nd_a[2]};
        ie_a = ie_b;
        ie_b = w + 2 * wstride < nunits ? tri_of(w + 2 * wstride) : 0;
        if (w + wstride < nunits)
            for (int k = 0; k < 3; k++) nd_a[k] = D.e2d[3 * ie_a + k];
        // the previous group's reads are done before the records are rewritten
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        stage_triangle(D, ie, nodes, minus ? 1 : 0, b0, b1, b2, blkpos, rec);
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if constexpr (COLS > 1) {
            const LdsSrcT<false> S0{rec, ((const int *)(rec + LR_META))[1]};
            const Base base = base_terms<WET>(DL, S0);
            if (!minus) {
#pragma unroll
                for (int k = 0; k < NBASE; k++) rec[LR_BASE + k] = reinterpret_cast<const double *>(&base)[k];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
        // keeps the record's reads inside a column (hoisted out of the loop they
        // would hold the whole record in registers)
        auto fresh = [&]() {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            return LdsSrcT<(COLS > 1)>{rec, ((const int *)(rec + LR_META))[1]};
        };
        const int q0 = (w % PARTS) * COLS;
        if constexpr (COLS == 1) {
            const int j = q0 / 3, var = q0 % 3;
            if (var == 0) lds_column<WET, 0>(DL, fresh(), ie, nodes, j, minus, act, EM, EM32);
            else if (var == 1) lds_column<WET, 1>(DL, fresh(), ie, nodes, j, minus, act, EM, EM32);
            else lds_column<WET, 2>(DL, fresh(), ie, nodes, j, minus, act, EM, EM32);
        } else {
#pragma unroll 1
            for (int j = q0 / 3; j < (q0 + COLS) / 3; j++) {
                lds_column<WET, 0>(DL, fresh(), ie, nodes, j, minus, act, EM, EM32);
                lds_column<WET, 1>(DL, fresh(), ie, nodes, j, minus, act, EM, EM32);
                lds_column<WET, 2>(DL, fresh(), ie, nodes, j, minus, act, EM, EM32);
            }
        }
    }
}

template <bool WET, int BS, int COLS>
__global__ void __launch_bounds__(BS, 2) k_jac2d_lds(ElemData D, const int *list, const int *count, int b0, int b1,
                                                  int b2, const int *blkpos, double *EM, float *EM32) {
    __shared__ double srec[BS / 64][32][LREC];
    __shared__ crlog::tables slog;
    if (WET) stamp(D.ts);
    jac_lds_list<WET, BS, COLS>(D, list, count, b0, b1, b2, blkpos, EM, EM32, blockIdx.x, gridDim.x, srec, slog);
}

__device__ __forceinline__ void jac_edge(const ElemData &D, int t, int B, int b0, int b1, const int *blkpos1, double *EM,
                                         float *EM32) {
    if (t >= 6 * B) return;
    int ie = t / 6, q = t % 6, j = q / 3, var = q % 3;
    double col[9];
    jac_column<2>(D, ie, j, var, col);
    const int nodes[2] = {D.e1d[2 * ie], D.e1d[2 * ie + 1]};
    const int *lbi = D.loc_bc_inst ? D.loc_bc_inst + 3 * D.edge_inst[ie] : nullptr;
    const int lb[2] = {lbi ? lbi[0] : b0, lbi ? lbi[1] : b1};
    jac_column_db<2>(D, nodes, lb, j, var, col);
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const size_t o = 9 * (size_t)blkpos1[4 * ie + 2 * i + j];
#pragma unroll
        for (int r = 0; r < 3; r++) {
            if (EM32) EM32[o + 3 * r + var] = (float)col[3 * i + r];
            else EM[o + 3 * r + var] = col[3 * i + r];
        }
    }
}

__global__ void __launch_bounds__(128) k_jac1d(ElemData D, int B, int b0, int b1, const int *blkpos1, double *EM,
                                               float *EM32) {
    jac_edge(D, blockIdx.x * blockDim.x + threadIdx.x, B, b0, b1, blkpos1, EM, EM32);
}

// Both lists (LDS layout) and the boundary edges in one launch: an empty general
// list costs 4.0 us on its own and 128 edges 5.8, of 25 that the wet list takes
// at 1,600 triangles.
template <int BS, int COLS>
__global__ void __launch_bounds__(BS, 2) k_jac_all(ElemData D, const int *wet, const int *gen, const int *count,
                                                   int b0, int b1, int b2, const int *blkpos, double *EM, float *EM32,
                                                   int nwet, int ngen, int B, const int *blkpos1) {
    __shared__ double srec[BS / 64][32][LREC];
    __shared__ crlog::tables slog;
    stamp(D.ts);
    const int b = blockIdx.x;
    if (b < nwet)
        jac_lds_list<true, BS, COLS>(D, wet, count, b0, b1, b2, blkpos, EM, EM32, b, nwet, srec, slog);
    else if (b < nwet + ngen)
        jac_lds_list<false, BS, COLS>(D, gen, count + 1, b0, b1, b2, blkpos, EM, EM32, b - nwet, ngen, srec, slog);
    else
        jac_edge(D, (b - nwet - ngen) * BS + threadIdx.x, B, b0, b1, blkpos1, EM, EM32);
}

// Splits the triangles into those whose three depths stay positive under the
// -eps perturbation of the FD Jacobian (h - eps(h) > 0, the exact operation
// the perturbed residual performs) and the rest, as two ordered lists: block
// counts, then the ordered scatter (no same-address atomics, which serialise
// across the whole grid).
__device__ __forceinline__ bool tri_stays_wet(int ie, const int *e2d, const double *head) {
    bool w = true;
    for (int i = 0; i < 3; i++) {
        const double h = head[e2d[3 * ie + i]];
        if (!(h + (-1.0) * num_diff_eps(h) > 0.0)) w = false;
    }
    return w;
}

// Triangle classes for the element kernels: "wet" (stays wet under the -eps
// perturbation: the variant without clipping code), "general", or skipped
// (an ensemble model that is not being iterated).  bcount holds the per-block
// wet counts, then the per-block general counts.
__device__ __forceinline__ void split_class(int ie, int E, const int *e2d, const double *head, const int *elem_inst,
                                            const int *mask, bool &w, bool &g) {
    const bool act = ie < E && (!mask || mask[elem_inst[ie]]);
    w = act && tri_stays_wet(ie, e2d, head);
    g = act && !w;
}

__global__ void __launch_bounds__(256) k_split_count(int E, const int *e2d, const double *head, const int *elem_inst,
                                                     const int *mask, int *bcount, long long *ts) {
    __shared__ int wc[2][4];
    stamp(ts);
    const int ie = blockIdx.x * blockDim.x + threadIdx.x;
    bool w, g;
    split_class(ie, E, e2d, head, elem_inst, mask, w, g);
    const unsigned long long bw = __ballot(w), bg = __ballot(g);
    if ((threadIdx.x & 63) == 0) {
        wc[0][threadIdx.x >> 6] = __popcll(bw);
        wc[1][threadIdx.x >> 6] = __popcll(bg);
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        bcount[blockIdx.x] = wc[0][0] + wc[0][1] + wc[0][2] + wc[0][3];
        bcount[gridDim.x + blockIdx.x] = wc[1][0] + wc[1][1] + wc[1][2] + wc[1][3];
    }
}

// Above SPLIT_DIRECT count blocks: sums of SPLIT_RUN consecutive counts of each
// list, a workgroup each.
constexpr int SPLIT_RUN = 1024, SPLIT_DIRECT = 6144;
__global__ void __launch_bounds__(256) k_split_sums(int nb, const int *bcount, int *sums) {
    __shared__ int part[4];
    const int *c = bcount + (size_t)blockIdx.y * nb;
    const int b0 = blockIdx.x * SPLIT_RUN;
    int s = 0;
#pragma unroll
    for (int u = 0; u < SPLIT_RUN / 256; u++) {
        const int b = b0 + u * 256 + threadIdx.x;
        s += b < nb ? c[b] : 0;
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
    __syncthreads();
    if (threadIdx.x == 0) sums[blockIdx.y * gridDim.x + blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// A block's place in the two lists is the sum of the counts before it, which
// it adds up itself: 1M triangles, 3,906 counts, take less time that way than
// a scan kernel's launch (3.5 us), and fewer take next to none.  What all blocks
// add grows with the square of the triangles, so above SPLIT_DIRECT they add the
// sums of whole runs before them and the counts of their own run alone.
// Counts, sums and lists, us, by runs / directly: 1M triangles 16.6 / 15.6, 1.5M
// 25.0 / 23.6, 2M 28.1 / 30.9, 4M 49 / 71, 13.5M 146 / 496.
// The last block leaves the totals in counts.
__global__ void __launch_bounds__(256) k_split_write(int E, const int *e2d, const double *head, const int *elem_inst,
                                                     const int *mask, const int *bcount, const int *sums, int *counts,
                                                     int *wet, int *gen) {
    __shared__ int wc[2][4], before[2][4];
    {
        int s0 = 0, s1 = 0;
        // entries first .. last - 1 of the two arrays of n
        auto add = [&](const int *a, int n, int first, int last) {
            constexpr int U = 4;
            for (int b = first + threadIdx.x; b < last; b += U * 256) {
                int x[U][2];
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const bool in = b + u * 256 < last;
                    x[u][0] = in ? a[b + u * 256] : 0;
                    x[u][1] = in ? a[n + b + u * 256] : 0;
                }
#pragma unroll
                for (int u = 0; u < U; u++) { s0 += x[u][0]; s1 += x[u][1]; }
            }
        };
        const int run = sums ? (int)blockIdx.x / SPLIT_RUN : 0;
        if (sums) add(sums, (gridDim.x + SPLIT_RUN - 1) / SPLIT_RUN, 0, run);
        add(bcount, gridDim.x, run * SPLIT_RUN, blockIdx.x);
        for (int o = 32; o > 0; o >>= 1) { s0 += __shfl_xor(s0, o, 64); s1 += __shfl_xor(s1, o, 64); }
        if ((threadIdx.x & 63) == 0) { before[0][threadIdx.x >> 6] = s0; before[1][threadIdx.x >> 6] = s1; }
    }
    const int ie = blockIdx.x * blockDim.x + threadIdx.x;
    bool w, g;
    split_class(ie, E, e2d, head, elem_inst, mask, w, g);
    const unsigned long long bw = __ballot(w), bg = __ballot(g);
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    if (lane == 0) {
        wc[0][wid] = __popcll(bw);
        wc[1][wid] = __popcll(bg);
    }
    __syncthreads();
    int bef_w = before[0][0] + before[0][1] + before[0][2] + before[0][3];   // of each class before this wave
    int bef_g = before[1][0] + before[1][1] + before[1][2] + before[1][3];
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) {
        counts[0] = bef_w + wc[0][0] + wc[0][1] + wc[0][2] + wc[0][3];
        counts[1] = bef_g + wc[1][0] + wc[1][1] + wc[1][2] + wc[1][3];
    }
    for (int k = 0; k < wid; k++) { bef_w += wc[0][k]; bef_g += wc[1][k]; }
    const unsigned long long below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    if (w) wet[bef_w + __popcll(bw & below)] = ie;
    if (g) gen[bef_g + __popcll(bg & below)] = ie;
}

static int split_runs(int nb) { return (nb + SPLIT_RUN - 1) / SPLIT_RUN; }
// ints of the count blocks' arrays of a mesh of E triangles
size_t split_words(int E) {
    const int nb = nblocks_for(E, 256);
    return 2 * (size_t)nb + 2 * (size_t)split_runs(nb);
}

// ordered wet / general triangle lists for the current depths (and, for
// ensembles, the models being iterated)
static void launch_split(Ctx *c) {
    if (!c->E) return;
    const int nb = nblocks_for(c->E, 256);
    const int *mask = c->ninst ? c->inst_mask : nullptr;
    hipLaunchKernelGGL(k_split_count, dim3(nb), dim3(256), 0, c->stream, c->E, c->e2d, c->head, c->elem_inst, mask,
                       c->esplit, c->h_ts + TS_RESID);
    int *sums = nullptr;
    if (nb > SPLIT_DIRECT) {
        sums = c->esplit + 2 * (size_t)nb;
        hipLaunchKernelGGL(k_split_sums, dim3(split_runs(nb), 2), dim3(256), 0, c->stream, nb, c->esplit, sums);
    }
    hipLaunchKernelGGL(k_split_write, dim3(nb), dim3(256), 0, c->stream, c->E, c->e2d, c->head, c->elem_inst, mask,
                       c->esplit, sums, c->ecount, c->elist_wet, c->elist_gen);
    c->split_valid = 1;
}

// Columns a wave of the LDS layout takes of its 32 triangles.  The GPU holds two
// of its waves on each of 1,024 SIMDs, and a wave's nine columns are one serial
// chain (63 us at any size that fits): one column a wave while nine waves per
// group fit at once, one node's three while the groups are fewer than two
// rounds of waves, else all nine (staging and Base terms formed once).
// Measured, us for 9 / 3 / 1 columns: 50 groups 61 / 31 / 21, 394 groups 63 /
// 31 / 35, 1,000 69 / 55 / 69, 2,000 88 / 84 / 112, 4,050 139 / 141 / 198,
// 31,250 747 / 893 / 1,282.
constexpr int JAC_WAVES = 2048;
static int jac_columns(int groups) {
    if (9 * groups <= JAC_WAVES) return 1;
    return groups < 2 * JAC_WAVES ? 3 : 9;
}

// Grid-stride list launches.  Block size and grid size change only the
// schedule (every triangle's arithmetic and output slot are fixed), so they
// are free parameters: defaults below, or what adh_sw2_hip_autotune measured.
template <bool WET, int BS>
static void jac_list_bs(Ctx *c, const ElemData &D, const int *list, const int *count, int grid, int layout) {
    if (layout >= 2) {   // column-uniform waves, inputs staged in LDS
        const int groups = (c->E + 31) / 32;
        auto launch = [&](auto cols) {
            constexpr int COLS = decltype(cols)::value;
            const int units = 9 / COLS * groups;
            hipLaunchKernelGGL((k_jac2d_lds<WET, BS, COLS>), dim3(std::min(grid, nblocks_for(units, BS / 64))),
                               dim3(BS), 0, c->stream, D, list, count, c->loc_bc[0], c->loc_bc[1], c->loc_bc[2],
                               c->blkpos, c->EM, em32_of(c));
        };
        const int cols = layout == 2 ? 1 : jac_columns(groups);
        if (cols == 1) launch(std::integral_constant<int, 1>());
        else if (cols == 3) launch(std::integral_constant<int, 3>());
        else launch(std::integral_constant<int, 9>());
        return;
    }
    if (layout == 1) {   // column-uniform waves: 9 waves per 32 triangles
        const int units = 9 * ((c->E + 31) / 32);
        hipLaunchKernelGGL((k_jac2d_cols<WET, BS>), dim3(std::min(grid, nblocks_for(units, BS / 64))), dim3(BS), 0,
                           c->stream, D, list, count, c->loc_bc[0], c->loc_bc[1], c->loc_bc[2], c->blkpos, c->EM,
                           em32_of(c));
        return;
    }
    hipLaunchKernelGGL((k_jac2d_list<WET, BS, 0>), dim3(std::min(grid, nblocks_for(18 * c->E, BS))), dim3(BS), 0,
                       c->stream, D, list, count, c->loc_bc[0], c->loc_bc[1], c->loc_bc[2], c->blkpos, c->EM,
                       em32_of(c));
}
template <bool WET, int BS>
static void res_list_bs(Ctx *c, const ElemData &D, const int *list, const int *count, int grid) {
    hipLaunchKernelGGL((k_resid2d_list<WET, BS>), dim3(std::min(grid, nblocks_for(c->E, BS))), dim3(BS), 0, c->stream,
                       D, list, count, c->ER);
}

// phase: 0 Jacobian wet list, 1 Jacobian general list, 2 residual wet list, 3 residual general list
void launch_list(Ctx *c, const ElemData &D, int phase, int bs, int grid, int layout) {
    const bool wet = phase == 0 || phase == 2;
    const int *list = wet ? c->elist_wet : c->elist_gen;
    const int *count = wet ? c->ecount : c->ecount + 1;
#define SW2_LIST_CASE(B)                                                                      \
    case B:                                                                                    \
        if (phase == 0) jac_list_bs<true, B>(c, D, list, count, grid, layout);                    \
        else if (phase == 1) jac_list_bs<false, B>(c, D, list, count, grid, layout);              \
        else if (phase == 2) res_list_bs<true, B>(c, D, list, count, grid);                    \
        else res_list_bs<false, B>(c, D, list, count, grid);                                   \
        break;
    switch (bs) {
        SW2_LIST_CASE(64)
        SW2_LIST_CASE(256)
        default:
        SW2_LIST_CASE(128)
    }
#undef SW2_LIST_CASE
}

void ensure_lists(Ctx *c) {
    if (!c->pre_valid) launch_old_terms(c);
    if (!c->split_valid) launch_split(c);
}

// one list kernel with the element data its phase uses (autotuning)
void launch_list_phase(Ctx *c, int phase, int bs, int grid, int layout) {
    ElemData D = c->ed;
    D.first_elem = phase >= 2 ? c->first_elem : nullptr;
    launch_list(c, D, phase, bs, grid, layout);
}

// Workgroup size of the launches over both lists, where neither list's own launch
// shape asks for another
constexpr int JAC_ALL_BS = 256, RES_ALL_BS = 128;
// Triangles up to which the wet list runs beside the others.  Residuals: above,
// more than one wave a SIMD is at work and the wet list is faster in its own
// launch (44 us at 250,000 triangles).  Jacobians: both lists' code at once
// overruns the instruction caches, 148 against 59 + 74 us at 50,176 triangles of
// which half are partly dry; below the line it is the shorter one, whole loads of
// 1,600 / 13,794 / 32,768 triangles 37 / 54 / 77 against 43 / 62 / 83 us all wet and 42 / 74 / 111
// against 55 / 107 / 121 with 40 % of them partly dry.  (Edges and an empty general list
// alone in that kernel at 250,000 triangles: 18 us, in their own 13.)
constexpr int RES_ALL_TRIS = 65536, JAC_ALL_TRIS = 32768;

// The element Jacobians of both lists and, with `edges`, the boundary's.
static void launch_jac_split(Ctx *c, const ElemData &D, bool edges) {
    const int B = edges ? c->B : 0;
    const int *blkpos1 = c->blkpos + 9 * (size_t)c->E;
    if (c->E && !c->split_valid) launch_split(c);
    if (!(c->E && lists_joined(c, 0))) {
        if (c->E) {
            launch_list(c, D, 0, c->tune.bs[0], c->tune.grid[0], c->tune.layout[0]);
            launch_list(c, D, 1, c->tune.bs[1], c->tune.grid[1], c->tune.layout[1]);
        }
        if (B)
            hipLaunchKernelGGL(k_jac1d, dim3(nblocks_for(6 * B, 128)), dim3(128), 0, c->stream, D, B, c->loc_bc[0],
                               c->loc_bc[1], blkpos1, c->EM, em32_of(c));
        return;
    }
    const int groups = (c->E + 31) / 32;
    const int cols = c->tune.layout[0] == 2 ? 1 : jac_columns(groups);
    const int need = nblocks_for(9 / cols * groups, JAC_ALL_BS / 64);
    const int nwet = std::min(c->tune.grid[0], need), ngen = std::min(c->tune.grid[1], need);
    const dim3 g(nwet + ngen + (B ? nblocks_for(6 * B, JAC_ALL_BS) : 0));
    auto launch = [&](auto n) {
        hipLaunchKernelGGL((k_jac_all<JAC_ALL_BS, decltype(n)::value>), g, dim3(JAC_ALL_BS), 0, c->stream, D,
                           c->elist_wet, c->elist_gen, c->ecount, c->loc_bc[0], c->loc_bc[1], c->loc_bc[2], c->blkpos,
                           c->EM, em32_of(c), nwet, ngen, B, blkpos1);
    };
    static_assert((JAC_ALL_TRIS + 31) / 32 < 2 * JAC_WAVES, "never nine columns a wave");
    if (cols == 1) launch(std::integral_constant<int, 1>());
    else launch(std::integral_constant<int, 3>());
}

// The element residuals of both lists and, with `edges`, the boundary's.
static void launch_resid_split(Ctx *c, const ElemData &D, bool edges) {
    const int B = edges ? c->B : 0;
    double *er1 = c->ER + 9 * (size_t)c->E;
    if (c->E && !c->split_valid) launch_split(c);
    const int need = c->E ? nblocks_for(c->E, RES_ALL_BS) : 0;
    const bool beside = lists_joined(c, 2);
    if (c->E && !beside) launch_list(c, D, 2, c->tune.bs[2], c->tune.grid[2], c->tune.layout[2]);
    if (c->E && c->tune.bs[3] != RES_ALL_BS)
        launch_list(c, D, 3, c->tune.bs[3], c->tune.grid[3], c->tune.layout[3]);
    const int nwet = beside ? std::min(c->tune.grid[2], need) : 0;
    const int ngen = c->tune.bs[3] == RES_ALL_BS ? std::min(c->tune.grid[3], need) : 0;
    const dim3 g(nwet + ngen + (B ? nblocks_for(B, RES_ALL_BS) : 0));
    if (g.x == 0) return;
    if (beside)
        hipLaunchKernelGGL((k_resid_all<true, RES_ALL_BS>), g, dim3(RES_ALL_BS), 0, c->stream, D, c->elist_wet,
                           c->elist_gen, c->ecount, c->ER, nwet, ngen, B, er1);
    else
        hipLaunchKernelGGL((k_resid_all<false, RES_ALL_BS>), g, dim3(RES_ALL_BS), 0, c->stream, D, c->elist_wet,
                           c->elist_gen, c->ecount, c->ER, nwet, ngen, B, er1);
}

void launch_jacobian(Ctx *c) {
    if (!c->pre_valid) launch_old_terms(c);
    ElemData D = c->ed;
    D.first_elem = nullptr;
    D.ts = c->h_ts + TS_LOAD;
    c->em32 = em32_of(c) != nullptr;
    launch_jac_split(c, D, true);
}

// the launches of a Jacobian's (else a residual's) element kernels, edges included,
// as they run with the tuning in force; for the autotuner
void launch_elements(Ctx *c, bool jacobian) {
    if (!c->pre_valid) launch_old_terms(c);
    ElemData D = c->ed;
    D.first_elem = jacobian ? nullptr : c->first_elem;
    if (jacobian) launch_jac_split(c, D, true);
    else launch_resid_split(c, D, true);
}

// Whether phase 0's or 2's list runs in one launch with the next phase's.
bool lists_joined(const Ctx *c, int phase) {
    const Ctx::Tuning &t = c->tune;
    if (phase == 0)
        return c->E <= JAC_ALL_TRIS && t.bs[0] == JAC_ALL_BS && t.bs[1] == JAC_ALL_BS && t.layout[0] >= 2 &&
               t.layout[1] == t.layout[0];
    return c->E <= RES_ALL_TRIS && t.bs[2] == RES_ALL_BS && t.bs[3] == RES_ALL_BS;
}

// Ordered block assembly.  The element kernels store each 3x3 block at its
// contributor position (slot order; within a slot the contributors in
// ascending element order, 2D before 1D), so a block's sum reads one
// contiguous run.  Slots are the N diagonal blocks by node, then one per SELL
// position.  A workgroup takes one 64-row slice: wave 0 the diagonal blocks,
// wave w >= 1 the row slots j = w - 1 (+ stride), so every wave reads one
// contiguous stretch of element blocks and writes 64 consecutive sliced
// entries.  The diagonal block gets the floor and residual tweak of
// fe_sw2_load.c:218-236; the waves' row maxima, combined in LDS, give the
// Jacobi scale of solv_linear_sys_setup (the same values as k_scale_rows,
// which the set-up then skips).
template <typename TM>
__device__ __forceinline__ void sum_run(const int *slot_ptr, size_t slot, const TM *EM, double (&a)[9]) {
#pragma unroll
    for (int k = 0; k < 9; k++) a[k] = 0.0;
    const int p0 = slot_ptr[slot], p1 = slot_ptr[slot + 1];
    // pairs of blocks: both loaded before the in-order sums
    int p = p0;
    for (; p + 1 < p1; p += 2) {
        const TM *b0 = EM + 9 * (size_t)p, *b1 = b0 + 9;
        double x0[9], x1[9];
#pragma unroll
        for (int k = 0; k < 9; k++) { x0[k] = (double)b0[k]; x1[k] = (double)b1[k]; }
#pragma unroll
        for (int k = 0; k < 9; k++) a[k] += x0[k];
#pragma unroll
        for (int k = 0; k < 9; k++) a[k] += x1[k];
    }
    if (p < p1) {
        const TM *b = EM + 9 * (size_t)p;
#pragma unroll
        for (int k = 0; k < 9; k++) a[k] += (double)b[k];
    }
}

// TM: element-block type; TO: off-diagonal output type (float for the refined
// forms, which keep only an FP32 matrix: the set-up scales it in place).
template <typename TM, typename TO>
__global__ void __launch_bounds__(1024) k_assemble(int N, const int *slot_ptr, const int *row_ptr,
                                                   const int *sell_ptr, const TM *EM, double *diag, TO *offd,
                                                   double *R, const double *u, const double *v, double *sv) {
    __shared__ double smax[16][3][64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int n = 64 * blockIdx.x + lane;
    double s[3] = {0.0, 0.0, 0.0};
    double a[9];
    if (n < N) {
        if (w == 0) {
            sum_run(slot_ptr, (size_t)n, EM, a);
            const double f = NOT_QUITE_SMALL;
            if (fabs(a[0]) < f) {
                a[0] = f;
                double &r0 = R[vidx3(n, 0)];
                if (fabs(r0) < f) r0 = -f * u[n];
            }
            if (fabs(a[4]) < f) {
                a[4] = f;
                double &r1 = R[vidx3(n, 1)];
                if (fabs(r1) < f) r1 = -f * v[n];
            }
            if (fabs(a[8]) < f) a[8] = f;
#pragma unroll
            for (int k = 0; k < 9; k++) {
                diag[didx9(n, k)] = a[k];
                const double x = fabs(a[k]);
                if (x > s[k / 3]) s[k / 3] = x;
            }
        } else {
            const size_t q0 = 64 * (size_t)sell_ptr[n >> 6] + lane;
            const int len = row_ptr[n + 1] - row_ptr[n];
            for (int j = w - 1; j < len; j += nw - 1) {
                const size_t q = q0 + 64 * (size_t)j;
                sum_run(slot_ptr, (size_t)N + q, EM, a);
#pragma unroll
                for (int k = 0; k < 9; k++) {
                    offd[sell_vidx(q, k)] = (TO)a[k];
                    const double x = fabs(a[k]);
                    if (x > s[k / 3]) s[k / 3] = x;
                }
            }
        }
    }
#pragma unroll
    for (int j = 0; j < 3; j++) smax[w][j][lane] = s[j];
    __syncthreads();
    if (w != 0 || n >= N) return;
    const double small_factor = 1.0 / sqrt(SOLV_TOL);
#pragma unroll
    for (int j = 0; j < 3; j++) {
        double m = smax[0][j][lane];
        for (int x = 1; x < nw; x++) {
            const double y = smax[x][j][lane];
            if (y > m) m = y;
        }
        sv[vidx3(n, j)] = m < SOLV_TOL ? small_factor : 1.0 / sqrt(fabs(m));
    }
}

void launch_assemble(Ctx *c) {
    const int nw = 1 + std::min(std::max(c->kmax_row, 1), 15);   // waves per 64-row slice
    // refined forms with block Jacobi: element blocks stored in FP32, summed in
    // FP64, off-diagonal blocks written in FP32 (unscaled) straight into the
    // matrix the FP32 Krylov reads; otherwise FP64 throughout
    c->mat32 = c->em32 && c->opts.preconditioner != 1;
    dim3 g(nblocks_for(c->N, 64)), b(64 * nw);
    if (c->mat32)
        hipLaunchKernelGGL((k_assemble<float, float>), g, b, 0, c->stream, c->N, c->slot_ptr, c->row_ptr, c->sell_ptr,
                           (const float *)c->EM, c->diag, c->offd32, c->R, c->u, c->v, c->scale);
    else if (c->em32)
        hipLaunchKernelGGL((k_assemble<float, double>), g, b, 0, c->stream, c->N, c->slot_ptr, c->row_ptr,
                           c->sell_ptr, (const float *)c->EM, c->diag, c->offd, c->R, c->u, c->v, c->scale);
    else
        hipLaunchKernelGGL((k_assemble<double, double>), g, b, 0, c->stream, c->N, c->slot_ptr, c->row_ptr,
                           c->sell_ptr, (const double *)c->EM, c->diag, c->offd, c->R, c->u, c->v, c->scale);
    c->scale_valid = 1;
    c->sys_scaled = 0;
}

void launch_jac2d_only(Ctx *c) {
    if (!c->pre_valid) launch_old_terms(c);
    ElemData D = c->ed;
    D.first_elem = nullptr;
    launch_jac_split(c, D, false);
}

void launch_resid2d_only(Ctx *c) {
    if (!c->pre_valid) launch_old_terms(c);
    ElemData D = c->ed;
    D.first_elem = c->first_elem;
    launch_resid_split(c, D, false);
}

void launch_assemble_only(Ctx *c) { launch_assemble(c); }

// ------------------------------------------------------- init / wet-dry flags
// fe_sw2_init (fe_sw2_init.c:33-79)
__global__ void k_init_nodes(int N, const double *old_head, const double *old_u, const double *old_v, double *head,
                             double *u, double *v, const int *node_bc, const double *bcval, int *bc_mask,
                             int *wd_tmp, const int *node_inst, const int *mask, long long *ts) {
    stamp(ts);
    int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    if (mask && (node_inst[n] < 0 || !mask[node_inst[n]])) return;  // gap nodes (-1) never change
    double hh = old_head[n], uu = old_u[n], vv = old_v[n];
    int m0 = ADH_SW2_NO, m1 = ADH_SW2_NO, m2 = ADH_SW2_NO;
    int bc = node_bc[n];
    if (bc == BCT_VEL_DIR) {
        m0 = m1 = ADH_SW2_YES;
        uu = bcval[3 * n]; vv = bcval[3 * n + 1];
    } else if (bc == BCT_PRS_DIR) {
        m2 = ADH_SW2_YES;
        hh = bcval[3 * n + 2];
    } else if (bc == BCT_VEL_PRS_DIR) {
        m0 = m1 = m2 = ADH_SW2_YES;
        uu = bcval[3 * n]; vv = bcval[3 * n + 1]; hh = bcval[3 * n + 2];
    }
    head[n] = hh; u[n] = uu; v[n] = vv;
    if (bc_mask) { bc_mask[3 * n] = m0; bc_mask[3 * n + 1] = m1; bc_mask[3 * n + 2] = m2; }
    wd_tmp[n] = 0;
}

// fe_sw2_wdflag pass 1 (fe_sw2_wdflag.c:41-51): all writers store the same value
__global__ void k_wd_mark(int E, const int *e2d, const double *head, int *wd_tmp, const int *elem_inst,
                          const int *mask) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    if (mask && !mask[elem_inst[e]]) return;
    int a = e2d[3 * e], b = e2d[3 * e + 1], c = e2d[3 * e + 2];
    int wet = (head[a] > 0.0) + (head[b] > 0.0) + (head[c] > 0.0);
    if (wet != 3) { wd_tmp[a] = 1; wd_tmp[b] = 1; wd_tmp[c] = 1; }
}

// fe_sw2_wdflag pass 2 (:57-73)
__global__ void k_wd_flag(int E, const int *e2d, const double *head, const double *old_head, const int *wd_tmp,
                          int *wd_flag, const int *elem_inst, const int *mask) {
    int e = blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= E) return;
    if (mask && !mask[elem_inst[e]]) return;
    int a = e2d[3 * e], b = e2d[3 * e + 1], c = e2d[3 * e + 2];
    int f = (wd_tmp[a] != 0 || wd_tmp[b] != 0 || wd_tmp[c] != 0) ? 1 : 0;
    if (head[a] < 0 && head[b] < 0 && head[c] < 0 && old_head[a] < 0 && old_head[b] < 0 && old_head[c] < 0) f = 2;
    wd_flag[e] = f;
}

// old/older-state element terms, once per Newton solve (sw2_elem.h elem_old_terms)
__global__ void __launch_bounds__(128) k_old_terms(ElemData D, int E, double *pre) {
    int ie = blockIdx.x * blockDim.x + threadIdx.x;
    if (ie >= E) return;
    elem_old_terms(D, ie, pre + PRE_STRIDE * (size_t)ie);
}

void launch_old_terms(Ctx *c) {
    if (c->E)
        hipLaunchKernelGGL(k_old_terms, dim3(nblocks_for(c->E, 128)), dim3(128), 0, c->stream, c->ed, c->E, c->pre);
    c->pre_valid = 1;
}


void launch_init(Ctx *c, int *bc_mask_dev) {
    c->split_valid = 0;
    const int *mask = c->ninst ? c->inst_mask : nullptr;
    hipLaunchKernelGGL(k_init_nodes, dim3(nblocks_for(c->N, 256)), dim3(256), 0, c->stream, c->N, c->old_head,
                       c->old_u, c->old_v, c->head, c->u, c->v, c->node_bc, c->node_bc_val, bc_mask_dev, c->wd_tmp,
                       c->node_inst, mask, c->h_ts + TS_INIT);
    if (c->E) {
        hipLaunchKernelGGL(k_wd_mark, dim3(nblocks_for(c->E, 256)), dim3(256), 0, c->stream, c->E, c->e2d, c->head,
                           c->wd_tmp, c->elem_inst, mask);
        hipLaunchKernelGGL(k_wd_flag, dim3(nblocks_for(c->E, 256)), dim3(256), 0, c->stream, c->E, c->e2d, c->head,
                           c->old_head, c->wd_tmp, c->wd_flag, c->elem_inst, mask);
    }
    launch_old_terms(c);
}

// fe_sw2 (fe_sw2.c:42-50)
__global__ void k_shift(int N, double *h, double *u, double *v, double *oh, double *ou, double *ov, double *ooh,
                        double *oou, double *oov, const int *node_inst, const int *mask) {
    int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    if (mask && (node_inst[n] < 0 || !mask[node_inst[n]])) return;  // gap nodes (-1) never change
    ooh[n] = oh[n]; oou[n] = ou[n]; oov[n] = ov[n];
    oh[n] = h[n]; ou[n] = u[n]; ov[n] = v[n];
}

void launch_shift(Ctx *c) {
    c->pre_valid = 0;
    c->split_valid = 0;
    hipLaunchKernelGGL(k_shift, dim3(nblocks_for(c->N, 256)), dim3(256), 0, c->stream, c->N, c->head, c->u, c->v,
                       c->old_head, c->old_u, c->old_v, c->older_head, c->older_u, c->older_v, c->node_inst,
                       c->ninst ? c->inst_mask : nullptr);
}

// fe_sw2_inc (fe_sw2_inc.c:47-54): factor 1.0
__global__ void k_inc(int N, const double *sol, double *h, double *u, double *v, const int *node_inst,
                      const int *mask) {
    int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    if (mask && (node_inst[n] < 0 || !mask[node_inst[n]])) return;  // gap nodes (-1) never change
    u[n] += 1. * sol[vidx3(n, 0)];
    v[n] += 1. * sol[vidx3(n, 1)];
    h[n] += 1. * sol[vidx3(n, 2)];
}

void launch_inc(Ctx *c, double) {
    c->split_valid = 0;
    hipLaunchKernelGGL(k_inc, dim3(nblocks_for(c->N, 256)), dim3(256), 0, c->stream, c->N, c->sol, c->head, c->u,
                       c->v, c->node_inst, c->ninst ? c->inst_mask : nullptr);
}

// fe_sw2_inc, then sol = -sol (what the line search steps back along), in one
// pass over the nodes: the same operations as k_inc followed by k_scale_vec(-1)
__global__ void k_inc_flip(int N, double *sol, double *h, double *u, double *v, const int *node_inst,
                           const int *mask, long long *ts) {
    stamp(ts);
    int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    if (mask && (node_inst[n] < 0 || !mask[node_inst[n]])) return;  // gap nodes (-1) never change
    const double s0 = sol[vidx3(n, 0)], s1 = sol[vidx3(n, 1)], s2 = sol[vidx3(n, 2)];
    u[n] += 1. * s0;
    v[n] += 1. * s1;
    h[n] += 1. * s2;
    sol[vidx3(n, 0)] = s0 * -1.0;
    sol[vidx3(n, 1)] = s1 * -1.0;
    sol[vidx3(n, 2)] = s2 * -1.0;
}

void launch_inc_flip(Ctx *c) {
    c->split_valid = 0;
    hipLaunchKernelGGL(k_inc_flip, dim3(nblocks_for(c->N, 256)), dim3(256), 0, c->stream, c->N, c->sol, c->head, c->u,
                       c->v, c->node_inst, c->ninst ? c->inst_mask : nullptr, c->h_ts + TS_INC);
}

// x *= f over a sliced node vector; entry i belongs to node 64 (i / 192) + i mod 64
__global__ void k_scale_vec(size_t n, double *x, double f, const int *node_inst, const int *mask) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    if (mask) {
        const int m = node_inst[64 * (i / 192) + (i & 63)];
        if (m < 0 || !mask[m]) return;
    }
    x[i] *= f;
}

void launch_scale_sol(Ctx *c, double f) {
    hipLaunchKernelGGL(k_scale_vec, dim3(nblocks_for(3 * c->Np, 256)), dim3(256), 0, c->stream, (size_t)3 * c->Np,
                       c->sol, f, c->node_inst, c->ninst ? c->inst_mask : nullptr);
}

// plain streaming copy of n doubles (bandwidth calibration for the counters)
__global__ void __launch_bounds__(256) k_copy(size_t n, const double *__restrict__ src, double *__restrict__ dst) {
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) dst[i] = src[i];
}

void launch_copy(Ctx *c, const double *src, double *dst, size_t n) {
    if (n) hipLaunchKernelGGL(k_copy, dim3(4096), dim3(256), 0, c->stream, n, src, dst);
}

// grid-stride: the tiled LU's bands exceed 2^31 doubles (4.7e9 at 1M triangles)
__global__ void k_zero(size_t n, double *x) {
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) x[i] = 0.0;
}

void launch_zero(Ctx *c, double *p, size_t n) {
    const size_t blocks = std::max<size_t>(1, std::min<size_t>((n + 255) / 256, (size_t)1 << 20));
    hipLaunchKernelGGL(k_zero, dim3((unsigned)blocks), dim3(256), 0, c->stream, n, p);
}

// rounding probe: device cr_log, sqrt and division of each input
__global__ void k_probe(const double *x, int n, const crlog::tables *t, double *lg, double *sq, double *dv) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double a = x[i];
    lg[i] = crlog::cr_log_t(a, t);
    sq[i] = sqrt(a);
    dv[i] = 1.0 / a;
}

void launch_probe(const double *x, int n, const crlog::tables *t, double *lg, double *sq, double *dv) {
    hipLaunchKernelGGL(k_probe, dim3(nblocks_for(n, 256)), dim3(256), 0, 0, x, n, t, lg, sq, dv);
}


}  // namespace sw2
