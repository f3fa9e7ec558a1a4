// A whole block-Jacobi BiCGSTAB solve (the recurrences and roundings of
// sw2_solver.hip's prologue, K1..K3 and epilogue) in one kernel, for models
// whose 256-node blocks all fit on the GPU at once.
//
// What bounds the kernel-per-step form at these sizes is launches, six of 2 to
// 5 us per iteration, and the matrix read twice per iteration.  Here a
// workgroup keeps one 256-node block for the whole solve: the block's matrix
// rows, preconditioner blocks and its part of every vector stay in registers
// and LDS, and so do copies of the neighbour nodes' p and r, which every
// reader brings forward by itself with the owner's arithmetic.  An iteration
// then exchanges two vectors (Ap, As) and crosses two model-wide hand-overs
// instead of six kernel boundaries:
//
//   hand-over 1: Ap, the partials of (q, Ap) and of the previous ||r||
//   hand-over 2: As, the partials of (As, s), (As, As), (As, q)
//
// (the previous ||r|| ends the solve one product late, which changes nothing:
// the product is dropped.)  The partials are formed and folded in the order of
// block_partials and k_fin, so every value is bit for bit that of the
// kernel-per-step form.
//
// An iteration, us, kernel-per-step form -> this (prologue and epilogue, seven
// launches there, included in proportion): 861 nodes FP64 28 -> 7.5, 16,008
// nodes refined 28 -> 8.7, 125,751 nodes FP64 52 -> 26.  What bounds it now is
// the hand-over: 3.2 us with 4 blocks, 4.2 with 63 (store and load past the
// L2, each about 1 us, the folds and the product), 9 to 13 with 492 (every
// block polls all blocks' partials, and the neighbours' values are read past
// the L2).

#include <algorithm>
#include <functional>
#include <queue>
#include <utility>
#include <vector>

#include "sw2_flow.h"
#include "sw2_krylov.h"

namespace sw2 {

namespace {

// x of the lane 32 (16) further, cyclically: halves of the wave (rows of 16) exchanged
__device__ __forceinline__ double swap32(double x) {
    const unsigned lo = __double2loint(x), hi = __double2hiint(x);
    const auto a = __builtin_amdgcn_permlane32_swap(lo, lo, false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(hi, hi, false, false);
    const bool up = __lane_id() >= 32;
    return __hiloint2double(up ? b[0] : b[1], up ? a[0] : a[1]);
}
__device__ __forceinline__ double swap16(double x) {
    const unsigned lo = __double2loint(x), hi = __double2hiint(x);
    const auto a = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
    const auto b = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
    const bool up = __lane_id() & 16;
    return __hiloint2double(up ? b[0] : b[1], up ? a[0] : a[1]);
}
template <int CTRL>
__device__ __forceinline__ double dpp(double x) {
    return __hiloint2double(__builtin_amdgcn_update_dpp(0, __double2hiint(x), CTRL, 0xf, 0xf, true),
                            __builtin_amdgcn_update_dpp(0, __double2loint(x), CTRL, 0xf, 0xf, true));
}
// The wave's fold in the pairing of a butterfly over lane distances 32, 16, 8,
// 4, 2, 1 (after a distance d all lanes equal mod d hold one value, so a
// rotation serves as the exchange); in registers it takes a fifth of the
// time of LDS permutes.
template <bool MAX>
__device__ __forceinline__ double wave_fold(double x) {
    auto f = [](double a, double b) { return MAX ? fmax(a, b) : a + b; };
    x = f(x, swap32(x));
    x = f(x, swap16(x));
    x = f(x, dpp<0x128>(x));   // row_ror:8
    x = f(x, dpp<0x124>(x));   // row_ror:4
    x = f(x, dpp<0x4e>(x));    // quad_perm 2,3,0,1
    return f(x, dpp<0xb1>(x)); // quad_perm 1,0,3,2
}

// a value all lanes hold alike, in scalar registers
__device__ __forceinline__ double uniform(double x) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(x)),
                            __builtin_amdgcn_readfirstlane(__double2loint(x)));
}

// Hand-overs.  At each, a block publishes its part of one vector and up to
// three partials, and receives its neighbours' values and the folded partials
// of all blocks.  Every word is its own ready flag: it holds EMPTY until it is
// stored, by an agent-scope store (past the XCDs' private L2s), and readers
// poll it, so a hand-over is one store and one load deep and has no fence.
//
// Words are emptied again by their owner.  Passing hand-over e shows that
// every block has published e, hence has read everything of e - 1.  The
// partials of e - 1 are emptied then (RING sets by turns: used again by e + 2,
// which readers poll only after the owner's e + 1, and each publish waits for
// the acknowledgement of the block's earlier stores), and so is the block's
// part of vector e - 1 (VRING vectors by turns).  At the end every block waits
// for a last hand-over and empties its parts of all vectors.  The partials have
// two sets for alternating launches, each launch emptying the other's.
//
// A wait gives up (all blocks do, then) after `limit` ticks of the 100 MHz
// clock: another program's kernels may hold the CUs that this model's
// remaining blocks wait for.  In an ensemble with more blocks than the GPU
// holds it may also be the launch's own earlier models: the clock stands while
// blocks before the model's first are at work, which end, or give up, in their
// time.  (With that time counted, 256 channels of 13.4M triangles in all gave up
// their first solve in FP64 after 17 ms and left the next ones to the other form,
// 277 M triangle-Newton/s instead of 309.)  The caller repeats the solve with the
// kernel-per-step form.  At the last hand-over some blocks may give up and others
// pass: the solve is then whole, but those that gave up leave their parts of the
// vectors filled, so the host is told of every give-up and empties all vectors.
constexpr int RING = 3, PARTS = 3, VRING = 4;
using HO = Slot<double>;
// Place of a partial: eight blocks' words to a 256-byte piece.  All blocks poll
// all partials; packed tightly they would lie on a few of the memory channels.
__host__ __device__ __forceinline__ size_t slot_at(int t, int k, int b, int nblk) {
    return (((size_t)t * PARTS + k) * ((nblk + 7) / 8) + (b >> 3)) * 32 + (b & 7);
}

// An ensemble's block's, in LDS: in registers it would be held through the solve.
// Times are the low halves of the clock's.
struct Wait {
    int quit;                  // the model gives up (one model's too)
    int ahead;                 // blocks of the launch before the model's first, 0 once they are through
    unsigned from;             // time at which they were last found at work
    int *ended;                // the launch's blocks that are through
};

template <bool ENS>
struct HandOver {
    double *set;               // this launch's partials [turn][partial][256-node block]
    int nblk, k0, k1, blk;     // blocks in all, the model's range, this one
    int turn;
    int *quit;                 // the model's give-up flag
    int *gave_up;              // the same for the host, of all models: the vectors are to be emptied
    unsigned limit;
    double (*shp)[4], (*shr)[4];
    Wait *shw;

    __device__ __forceinline__ double *slot(int t, int k, int b) const {
        return set + slot_at(t, k, b, nblk);
    }
    // the wait that began at t0 is over without result
    __device__ __forceinline__ bool give_up(unsigned t0, int spin) {
        const bool look = (spin & 15) == 15;
        bool late = (unsigned)wall_clock64() - t0 > limit;
        if (!look && !late) return false;
        if constexpr (ENS) {
            if (shw->ahead > 0) {
                if ((int)peek((float *)shw->ended) < shw->ahead) shw->from = (unsigned)wall_clock64();
                else shw->ahead = 0;
            }
            // signed: another wave may have found them at work after this one's look at the clock
            late = late && (int)((unsigned)wall_clock64() - shw->from) > (int)limit;
        }
        if (late) {
            put_raw((float *)quit, 1u);
            *gave_up = 1;
        } else if (!look || !peek((float *)quit)) return false;
        shw->quit = 1;
        return true;
    }

    // The block's partials out, bit k of MAXES: partial k is a maximum.  PENDING:
    // stores of this wave that need not have arrived (its part of the vector).
    template <int K, int MAXES, int PENDING>
    __device__ __forceinline__ void publish(const double (&v)[K]) {
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
        for (int k = 0; k < K; k++) {
            const double x = (MAXES >> k) & 1 ? wave_fold<true>(v[k]) : wave_fold<false>(v[k]);
            if (lane == 0) shp[k][wid] = x;
        }
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PENDING) : "memory");
        __syncthreads();
        if (threadIdx.x < K) {
            const int k = threadIdx.x;
            double x = shp[k][0];
            for (int w = 1; w < 4; w++) x = (MAXES >> k) & 1 ? fmax(x, shp[k][w]) : x + shp[k][w];
            put(slot(turn, k, blk), x);
        }
    }

    // All blocks' partials, folded as k_fin folds them, and with X the
    // neighbours' values, z = X at the offsets cc.  false: give up.
    template <int K, int MAXES, int NB, typename T>
    __device__ __forceinline__ bool collect(double (&out)[K], const T *X, const unsigned (&cc)[NB],
                                            T (&z)[NB][3]) {
        using U = typename Slot<T>::U;
        const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
        double acc[K];
#pragma unroll
        for (int k = 0; k < K; k++) acc[k] = 0.0;
        const unsigned t0 = (unsigned)wall_clock64();
        bool ok = true;
        constexpr int W = 2;
        for (int b0 = k0 + threadIdx.x; b0 < k1 && ok; b0 += W * 256) {
            HO::U u[W][K];
            for (int spin = 0;; spin++) {
#pragma unroll
                for (int i = 0; i < W; i++)
#pragma unroll
                    for (int k = 0; k < K; k++) u[i][k] = b0 + 256 * i < k1 ? peek(slot(turn, k, b0 + 256 * i)) : 0ull;
                bool all = true;
#pragma unroll
                for (int i = 0; i < W; i++)
#pragma unroll
                    for (int k = 0; k < K; k++) all = all && u[i][k] != HO::EMPTY;
                if (all) break;
                if (give_up(t0, spin)) { ok = false; break; }
            }
#pragma unroll
            for (int i = 0; i < W; i++)
                if (b0 + 256 * i < k1)
#pragma unroll
                    for (int k = 0; k < K; k++) {
                        const double x = __longlong_as_double((long long)u[i][k]);
                        acc[k] = (MAXES >> k) & 1 ? fmax(acc[k], x) : acc[k] + x;
                    }
        }
        if (X && ok)
            for (int spin = 0;; spin++) {   // all lanes again: z is the loads' registers, not a merge of two tries
                bool have = true;
#pragma unroll
                for (int b = 0; b < NB; b++)
#pragma unroll
                    for (int j = 0; j < 3; j++) {
                        const U w = peek(X + cc[b] + 64 * j);
                        have = have && w != Slot<T>::EMPTY;
                        z[b][j] = __builtin_bit_cast(T, w);
                    }
                if (!__any(!have)) break;
                if (give_up(t0, spin)) { ok = false; break; }
            }
#pragma unroll
        for (int k = 0; k < K; k++) {
            const double x = (MAXES >> k) & 1 ? wave_fold<true>(acc[k]) : wave_fold<false>(acc[k]);
            if (lane == 0) shr[k][wid] = x;
        }
        __syncthreads();
        const bool quit_now = shw->quit != 0;
#pragma unroll
        for (int k = 0; k < K; k++) {
            double x = shr[k][0];
            for (int w = 1; w < 4; w++) x = (MAXES >> k) & 1 ? fmax(x, shr[k][w]) : x + shr[k][w];
            out[k] = uniform(x);
        }
        const int last = turn == 0 ? RING - 1 : turn - 1;
        if (threadIdx.x < PARTS) put_raw(slot(last, threadIdx.x, blk), HO::EMPTY);
        turn = turn == RING - 1 ? 0 : turn + 1;
        return !quit_now;
    }
};

// This thread's rows of the matrix and of the preconditioner.
template <typename MT, int K>
struct Rows {
    MT D[9], M[9], A[K][9];
    __device__ __forceinline__ void load(const MT *diag, const MT *dinv, const MT *offd, int n, size_t q0) {
#pragma unroll
        for (int e = 0; e < 9; e++) {
            D[e] = ldnt(diag + didx9(n, e));
            M[e] = ldnt(dinv + didx9(n, e));
#pragma unroll
            for (int b = 0; b < K; b++) A[b][e] = ldnt(offd + sell_vidx(q0 + 64 * b, e));
        }
    }
    // y = M^-1 x
    template <typename T>
    __device__ __forceinline__ void precondition(const T (&x)[3], T (&y)[3]) const {
        y[0] = M[0] * x[0] + M[1] * x[1] + M[2] * x[2];
        y[1] = M[3] * x[0] + M[4] * x[1] + M[5] * x[2];
        y[2] = M[6] * x[0] + M[7] * x[1] + M[8] * x[2];
    }
    // y = M^-1 A x, x the row's own values, g its neighbours': amult_prec_row's order
    template <typename T>
    __device__ __forceinline__ void product(const T (&x)[3], const T (&g)[K][3], T (&y)[3]) {
        if constexpr (sizeof(MT) < sizeof(T)) {   // widened at each use: kept wide they would take twice the registers
#pragma unroll
            for (int e = 0; e < 9; e++) {
                asm("" : "+v"(D[e]), "+v"(M[e]));
#pragma unroll
                for (int b = 0; b < K; b++) asm("" : "+v"(A[b][e]));
            }
        }
        T p[3] = {0, 0, 0};
#pragma unroll
        for (int b = 0; b < K; b++) {
            p[0] += A[b][0] * g[b][0] + A[b][1] * g[b][1] + A[b][2] * g[b][2];
            p[1] += A[b][3] * g[b][0] + A[b][4] * g[b][1] + A[b][5] * g[b][2];
            p[2] += A[b][6] * g[b][0] + A[b][7] * g[b][1] + A[b][8] * g[b][2];
            __builtin_amdgcn_sched_barrier(0);   // bounds the widened entries in flight
        }
        T a[3];
        a[0] = D[0] * x[0] + D[1] * x[1] + D[2] * x[2];
        a[1] = D[3] * x[0] + D[4] * x[1] + D[5] * x[2];
        a[2] = D[6] * x[0] + D[7] * x[1] + D[8] * x[2];
        a[0] += p[0]; a[1] += p[1]; a[2] += p[2];
        precondition(a, y);
    }
};

// counts an ensemble's block at its end, whichever way it leaves
template <bool ENS>
struct Leaver {
    const Wait &w;
    __device__ __forceinline__ ~Leaver() {
        if (ENS && threadIdx.x == 0) atomicAdd(w.ended, 1);
    }
};

// OCC blocks on a CU: 512 registers a lane with one, 256 with two.  ENS: an
// ensemble's models (one model without what only they need: with it a solve of
// 125,751 nodes in FP64 was 2 % longer, all of it registers)
template <typename P, int K, int OCC, bool ENS>
__global__ void __launch_bounds__(256, OCC)
    k_bcg_run(int N, size_t n3, KVecs<P> V, typename P::V *xch, const int *sell_col, const double *rhs,
              const double *scale, double *sol, KScal *sc, KScal *host, const int *blk_inst, const int *inst_blk0,
              const int *blocks_before, double *slots, int parity, int *quit, int *gave_up, int *ended, unsigned limit) {
    using T = typename P::V;
    using MT = typename P::M;
    // AGAIN: the neighbours' r in LDS instead of their Ap, which is read a second
    // time where it is needed: 36 registers less
    constexpr bool AGAIN = OCC == 2 && sizeof(MT) == 8 && K > 4;
    __shared__ T nbP[K][3][256], nbX[K][3][256], q[3][256];
    __shared__ double shp[PARTS][4], shr[PARTS][4];
    __shared__ Wait shw;
    const int lb = blockIdx.x, nblk = gridDim.x, tid = threadIdx.x;
    int m = 0, nend = N;
    HandOver<ENS> H;
    H.k0 = 0;
    H.k1 = nblk;
    if constexpr (ENS) {
        m = blk_inst[2 * lb];
        nend = blk_inst[2 * lb + 1];
        H.k0 = inst_blk0[m];
        H.k1 = inst_blk0[m + 1];
    }
    const size_t nset = slot_at(RING, 0, 0, nblk);
    H.set = slots + parity * nset;
    H.nblk = nblk;
    H.blk = lb;
    H.turn = 0;
    H.quit = quit + 2 * m + parity;
    H.gave_up = gave_up;
    H.limit = limit;
    H.shp = shp;
    H.shr = shr;
    H.shw = &shw;
    if (tid < RING * PARTS) put_raw(slots + (1 - parity) * nset + slot_at(0, tid, lb, nblk), HO::EMPTY);
    const bool first = lb == H.k0;
    if (tid == 0) {
        shw.quit = 0;
        if (first) put_raw((float *)(quit + 2 * m + 1 - parity), 0u);
        if constexpr (ENS) {
            shw.ahead = blocks_before[m];
            shw.from = (unsigned)wall_clock64() - limit - 1;
            shw.ended = ended + parity;
            if (lb == 0) put_raw((float *)(ended + 1 - parity), 0u);
        }
    }
    sc += m;
    host += m;
    const int max_it = sc->max_it;
    const double atol = sc->atol, rtol = sc->rtol;
    if (ENS && max_it <= 0) {   // a model the ensemble's step leaves out
        if (first && tid == 0) sc->done = host->done = 1;
        return;
    }
    const Leaver<ENS> through{shw};
    // threads past the model's end repeat its last row and keep the result to themselves
    const bool live = lb * 256 + tid < nend;
    const int n = live ? lb * 256 + tid : nend - 1;
    const size_t own = vidx3(n, 0);

    const size_t q0 = 64 * (size_t)(n >> 6) * K + (n & 63);
    Rows<MT, K> rows;
    rows.load(V.diag, V.dinv, V.offd, n, q0);
    unsigned cc[K];
#pragma unroll
    for (int b = 0; b < K; b++) cc[b] = (unsigned)vidx3(sell_col[q0 + 64 * b], 0);
    // the vectors of hand-overs 0, 1, 2, 3, then 0 again: b', r, Ap, As, Ap, As, ...
    T *X = xch;
    int xt = 0;
    auto give = [&](const T (&x)[3]) {
        if (live)
#pragma unroll
            for (int j = 0; j < 3; j++) put(X + own + 64 * j, x[j]);
    };
    // empties the block's part of the vector two before this one, and goes on to the next
    auto turn_vector = [&]() {
        T *before = xch + (xt < 2 ? xt + VRING - 2 : xt - 2) * n3;
        if (live)
#pragma unroll
            for (int j = 0; j < 3; j++) put_raw(before + own + 64 * j, Slot<T>::EMPTY);
        xt = xt == VRING - 1 ? 0 : xt + 1;
        X = xch + xt * n3;
    };

    // u = b' = M^-1 b, ||b'||
    T u[3], r[3], p[3], y[3];
    T rn[K][3], g[K][3];
    double bnorm, rnorm, rho, rhop, alpha, omega;
    {
        double v[1] = {0.0}, out[1];
        const T rb[3] = {(T)rhs[own], (T)rhs[own + 64], (T)rhs[own + 128]};
        rows.precondition(rb, u);
        give(u);
#pragma unroll
        for (int j = 0; j < 3; j++) v[0] = fmax(v[0], fabs((double)u[j]));
        if (!live) v[0] = 0.0;
        __syncthreads();   // shw
        H.template publish<1, 1, 0>(v);
        if (!H.template collect<1, 1>(out, X, cc, g)) return;
        turn_vector();
        bnorm = out[0];
    }
    // r = b' - M^-1 A u, q = p = r, rho, ||r||
    {
        double v[2] = {0.0, 0.0}, out[2];
        rows.product(u, g, y);
#pragma unroll
        for (int j = 0; j < 3; j++) {
            r[j] = u[j] + (T)(-1.0) * y[j];
            q[j][tid] = r[j];
            p[j] = r[j];
            v[0] = fmax(v[0], fabs((double)r[j]));
            v[1] += (double)r[j] * (double)r[j];
        }
        give(r);
        if (!live) v[0] = v[1] = 0.0;
        H.template publish<2, 1, 3>(v);
        if (!H.template collect<2, 1>(out, X, cc, rn)) return;
        turn_vector();
        rnorm = out[0];
        rho = out[1];
    }
    const double tol = uniform(atol + bnorm * rtol);
    int it = 0;
    const bool more = rnorm > tol && 0 < max_it;
#pragma unroll
    for (int b = 0; b < K; b++)
#pragma unroll
        for (int j = 0; j < 3; j++) {
            g[b][j] = rn[b][j];
            nbP[b][j][tid] = rn[b][j];
            if constexpr (AGAIN) nbX[b][j][tid] = rn[b][j];
        }
    double vr = 0.0;
    while (more) {
        // K1
        T ap[3], as[3];
        {
            double v[2] = {0.0, vr}, out[2];
            rows.product(p, g, ap);
            give(ap);
#pragma unroll
            for (int j = 0; j < 3; j++) v[0] += (double)q[j][tid] * (double)ap[j];
            if (!live) v[0] = v[1] = 0.0;
            H.template publish<2, 2, 3>(v);
            if (!H.template collect<2, 2>(out, X, cc, g)) return;
            turn_vector();
            if (it > 0) {
                rnorm = out[1];
                if (!(rnorm > tol && it < max_it)) break;
            }
            alpha = uniform(rho / out[0]);
        }
        // K2: s into r and rn
        {
            const T nalpha = (T)(-alpha);
            double v[3] = {0.0, 0.0, 0.0}, out[3];
#pragma unroll
            for (int b = 0; b < K; b++)
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    if constexpr (AGAIN) {
                        g[b][j] = nbX[b][j][tid] + nalpha * g[b][j];
                        nbX[b][j][tid] = g[b][j];
                    } else {
                        nbX[b][j][tid] = g[b][j];
                        rn[b][j] = rn[b][j] + nalpha * g[b][j];
                    }
                }
#pragma unroll
            for (int j = 0; j < 3; j++) r[j] = r[j] + nalpha * ap[j];
            if constexpr (AGAIN) rows.product(r, g, as);
            else rows.product(r, rn, as);
            give(as);
#pragma unroll
            for (int j = 0; j < 3; j++) {
                v[0] += (double)as[j] * (double)r[j];
                v[1] += (double)as[j] * (double)as[j];
                v[2] += (double)as[j] * (double)q[j][tid];
            }
            if (!live) v[0] = v[1] = v[2] = 0.0;
            H.template publish<3, 0, 3>(v);
            if (!H.template collect<3, 0>(out, X, cc, g)) return;
            turn_vector();
            omega = uniform(out[0] / out[1]);
            rhop = rho;
            rho = uniform(-1.0 * omega * out[2]);
        }
        // K3
        const double beta = uniform((rho * alpha) / (rhop * omega));
        const T ta = (T)alpha, to = (T)omega, tno = (T)(-omega), tb = (T)beta;
        vr = 0.0;
#pragma unroll
        for (int j = 0; j < 3; j++) {
            u[j] += ta * p[j];
            u[j] += to * r[j];
            r[j] = r[j] + tno * as[j];
            p[j] += tno * ap[j];
            p[j] *= tb;
            p[j] += (T)1.0 * r[j];
            vr = fmax(vr, fabs((double)r[j]));
        }
        if constexpr (AGAIN) {
            const T *Ap = xch + (xt < 2 ? xt + VRING - 2 : xt - 2) * n3;   // not emptied before the next hand-over
#pragma unroll
            for (int b = 0; b < K; b++)
#pragma unroll
                for (int j = 0; j < 3; j++) {
                    nbX[b][j][tid] += tno * g[b][j];
                    g[b][j] = __builtin_bit_cast(T, peek(Ap + cc[b] + 64 * j));
                }
        }
#pragma unroll
        for (int b = 0; b < K; b++) {
            __builtin_amdgcn_sched_barrier(0);   // bounds the LDS values in flight
#pragma unroll
            for (int j = 0; j < 3; j++) {
                T pn = nbP[b][j][tid], rb;
                if constexpr (AGAIN) {
                    rb = nbX[b][j][tid];
                    pn += tno * g[b][j];
                } else {
                    rb = rn[b][j] = rn[b][j] + tno * g[b][j];
                    pn += tno * nbX[b][j][tid];
                }
                pn *= tb;
                pn += (T)1.0 * rb;
                nbP[b][j][tid] = pn;
                g[b][j] = pn;
            }
        }
        it++;
    }
    // sol = (u + 0) * scale, as the epilogue with a zero guess; a caller's guess
    // is added by the epilogue itself
#pragma unroll
    for (int j = 0; j < 3; j++)
        if (live) {
            if (sol) {
                double x = (double)u[j];
                x += 0.0;
                x *= scale[own + 64 * j];
                sol[own + 64 * j] = x;
            } else V.u[own + 64 * j] = u[j];
        }
    // every block has come this far: the model's first block reports, and all empty their vectors
    double v[1] = {0.0}, out[1];
    H.template publish<1, 0, 0>(v);
    if (!H.template collect<1, 0>(out, (const T *)nullptr, cc, g)) return;
    if (live)
        for (int t = 0; t < VRING; t++)
#pragma unroll
            for (int j = 0; j < 3; j++) put_raw(xch + t * n3 + own + 64 * j, Slot<T>::EMPTY);
    if (!first || tid != 0) return;
    KScal res = *sc;
    res.bnorm = bnorm;
    res.tol = tol;
    res.rnorm = rnorm;
    res.it = it;
    res.done = 1;
    *sc = res;
    *host = res;   // pinned: the caller only waits for the kernel
}

// all hand-over vectors emptied: before the first solve and after one that gave up
template <typename T>
__global__ void k_run_empty(size_t n, T *x) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) put_raw(x + i, Slot<T>::EMPTY);
}

// Blocks that the GPU holds at once, 0 where the system is not for this form.
template <typename P, int K, int OCC, bool ENS>
int run_capacity() {
    int per_cu = 0, dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_bcg_run<P, K, OCC, ENS>, 256, 0) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return per_cu * cus;
}

// Whether an ensemble's solve is expected to be shorter so than as a kernel per
// step.  A model has the GPU's places for its blocks until it is through, and the
// next ones start in order as places come free: models of just over half the GPU
// run one at a time, with nearly half of the GPU idle, while the kernels of the
// other form are filled by all models together.  us an iteration (of ten, the
// set-up of a solve included), measured with models of 60 to 512 blocks, six
// neighbours: a model of B blocks in FP64 10.2 + 0.011 B with one block a CU, 16.2 +
// 0.025 B with two, FP32 entries 9.3 + 0.0185 B, all FP32 9 + 0.0172 B; a kernel per
// step 18 and 0.07, 0.0453, 0.039 for every block.  A step of ten iterations, ms, per
// step / so: 24 models of 260 blocks FP64 11.4 / 12.4, 12 of 350 7.5 / 7.7, 12 of 450 9.5 /
// 9.1, 30 of 150 (one block a CU) 8.4 / 8.8; refined 24 of 260 9.2 / 9.3, 16 of 320 7.5 / 7.1.
template <typename P, int OCC>
bool run_pays(const Ctx *c, int cap) {
    if (!c->ninst) return true;
    constexpr bool WIDE = sizeof(typename P::M) == 8, F32 = sizeof(typename P::V) == 4;
    constexpr double A = WIDE ? (OCC == 1 ? 10.2 : 16.2) : (F32 ? 9.0 : 9.3);
    constexpr double B = WIDE ? (OCC == 1 ? 0.011 : 0.025) : (F32 ? 0.0172 : 0.0185);
    constexpr double STEP = WIDE ? 0.07 : (F32 ? 0.039 : 0.0453);
    using Busy = std::pair<double, int>;   // until when, how many places
    std::priority_queue<Busy, std::vector<Busy>, std::greater<Busy>> busy;
    double now = 0.0, end = 0.0, per_step = 18.0;
    int places = cap;
    for (int i = 0; i < c->ninst; i++) {
        if (!c->h_inst_mask[i]) continue;
        const int nb = nblocks_for(c->h_inst_N[i], 256);
        while (places < nb) {
            now = std::max(now, busy.top().first);
            places += busy.top().second;
            busy.pop();
        }
        places -= nb;
        busy.emplace(now + A + B * nb, nb);
        end = std::max(end, now + A + B * nb);
        per_step += STEP * nb;
    }
    return end <= per_step;
}

template <typename P, int K, int OCC, bool ENS>
bool run_k(Ctx *c, bool zero_guess) {
    int &cap = c->run_cap[OCC - 1];
    if (cap < 0) cap = run_capacity<P, K, OCC, ENS>();
    if (c->run_max_blocks > cap || !run_pays<P, OCC>(c, cap)) return false;
    using T = typename P::V;
    const int nb = nblocks_for(c->N, 256);
    const size_t n3 = 3 * (size_t)c->Np;
    T *xch = (T *)c->run_xch;
    if (c->run_dirty) {
        c->run_dirty = 0;
        hipLaunchKernelGGL(k_run_empty<T>, dim3((unsigned)((VRING * n3 + 255) / 256)), dim3(256), 0, c->stream,
                           VRING * n3, xch);
    }
    for (int i = 0; i < (c->ninst ? c->ninst : 1); i++) c->h_ksc[i].done = 0;   // the kernel sets what it finishes
    *c->h_gave_up = 0;
    c->run_parity ^= 1;
    hipLaunchKernelGGL((k_bcg_run<P, K, OCC, ENS>), dim3(nb), dim3(256), 0, c->stream, c->N, n3, vecs<P>(c), xch,
                       c->sell_col, c->R, c->scale, zero_guess ? c->sol : nullptr, c->ksc, c->h_ksc,
                       c->ninst ? c->blk_inst : nullptr, c->ninst ? c->inst_blk0 : nullptr,
                       c->ninst ? c->inst_mask + c->ninst : nullptr, c->run_slots, c->run_parity, c->run_quit,
                       c->h_gave_up, c->run_quit + 2 * (c->ninst ? c->ninst : 1),
                       (unsigned)std::min(c->run_limit, 1000000000LL));
    return true;
}

// Blocks a CU holds (OCC), hence the registers a lane has.  FP32 entries fit
// with two blocks up to six neighbours.  FP64 entries fit with two up to four
// neighbours; with five or six they need more than 256 registers, so a model
// of up to 256 blocks (65,536 nodes) takes one block a CU and a larger one two,
// with some registers spilled and the neighbours' Ap read twice.  One / two
// blocks a CU, us a solve of 8 iterations, six neighbours, FP64: 1,891 nodes
// 69 / 117, 16,008 81 / 138, 65,341 115 / 146; FP32 entries: equal.  Seven and
// eight neighbours: the LDS takes one block.  More blocks than the GPU holds
// (512, 131,072 nodes), more or fewer neighbours, or slices of unequal width:
// the kernel-per-step form.  An ensemble takes the first of these that pays
// (run_pays).
template <typename P, int K, bool ENS>
bool run_occ(Ctx *c, bool zero_guess) {
    constexpr bool WIDE = sizeof(typename P::M) == 8;
    if constexpr (K > 6) return run_k<P, K, 1, ENS>(c, zero_guess);
    else {
        if constexpr (WIDE && K > 4)
            if (run_k<P, K, 1, ENS>(c, zero_guess)) return true;
        return run_k<P, K, 2, ENS>(c, zero_guess);
    }
}

template <typename P, bool ENS>
bool run_e(Ctx *c, bool zero_guess) {
    switch (c->kuni) {
        case 3: return run_occ<P, 3, ENS>(c, zero_guess);
        case 4: return run_occ<P, 4, ENS>(c, zero_guess);
        case 5: return run_occ<P, 5, ENS>(c, zero_guess);
        case 6: return run_occ<P, 6, ENS>(c, zero_guess);
        case 7: return run_occ<P, 7, ENS>(c, zero_guess);
        case 8: return run_occ<P, 8, ENS>(c, zero_guess);
        default: return false;
    }
}

template <typename P>
bool run_p(Ctx *c, bool zero_guess) {
    return c->ninst ? run_e<P, true>(c, zero_guess) : run_e<P, false>(c, zero_guess);
}

}  // namespace

size_t run_slot_words(int nblk) { return 2 * slot_at(RING, 0, 0, nblk); }
size_t run_vector_words(int Np) { return VRING * 3 * (size_t)Np; }

// The solve queued as one kernel; false: this system takes the
// kernel-per-step form (so does opts.graphs, which asks for that form's
// captured chunks).
bool launch_krylov_run(Ctx *c, bool zero_guess) {
    if (c->opts.preconditioner != 2 || c->opts.krylov != 0 || c->opts.graphs || c->run_limit < 0 ||
        c->run_max_blocks > RUN_BLOCKS)
        return false;
    if (c->run_prec != c->opts.precision) {   // another form: its capacity, and vectors of its type
        c->run_prec = c->opts.precision;
        c->run_cap[0] = c->run_cap[1] = -1;
        c->run_dirty = 1;
    }
    if (c->opts.precision == 2) return run_p<PrecF32>(c, zero_guess);
    if (c->opts.precision == 1) return run_p<PrecMix>(c, zero_guess);
    return run_p<PrecF64>(c, zero_guess);
}

}  // namespace sw2
