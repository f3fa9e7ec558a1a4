// What the Krylov kernels share: the storage and arithmetic types of each
// precision form and the vectors of a solve.
#pragma once
#include "sw2_ctx.h"

namespace sw2 {

// FP64 matrix and preconditioner entries are read once per product:
// non-temporal loads keep them from displacing the gathered vector in L2
// (57 against 63 us for the FP64 K1 at 1M triangles; the FP32 streams are
// faster with ordinary loads)
template <typename T>
__device__ __forceinline__ T ldnt(const T *p) {
    if constexpr (sizeof(T) == 8) return __builtin_nontemporal_load(p);
    else return *p;
}

// Precision tags of the Krylov solve: matrix/preconditioner storage type M
// and vector/arithmetic type V (a float matrix entry times a double vector
// entry is formed in double).
struct PrecF64 { using M = double; using V = double; };   // precision 0
struct PrecMix { using M = float; using V = double; };    // precision 1: FP32 matrix, FP64 vectors
struct PrecF32 { using M = float; using V = float; };     // precision 2: all FP32

template <typename P>
struct KVecs {
    const typename P::M *diag, *offd, *dinv;
    typename P::V *b, *r, *p, *Ap, *s, *As, *q, *u;
};

template <typename P>
inline KVecs<P> vecs(Ctx *c);
template <>
inline KVecs<PrecF64> vecs<PrecF64>(Ctx *c) {
    return KVecs<PrecF64>{c->diag, c->offd, c->dinv, c->kb, c->kr, c->kp, c->kAp, c->ks_, c->kAs, c->kq, c->ku};
}
template <>
inline KVecs<PrecMix> vecs<PrecMix>(Ctx *c) {
    return KVecs<PrecMix>{c->diag32, c->offd32, c->dinv32, c->kb, c->kr, c->kp, c->kAp, c->ks_, c->kAs, c->kq, c->ku};
}
template <>
inline KVecs<PrecF32> vecs<PrecF32>(Ctx *c) {
    return KVecs<PrecF32>{c->diag32, c->offd32, c->dinv32, c->fb, c->fr, c->fp, c->fAp, c->fs, c->fAs, c->fq, c->fu};
}

}  // namespace sw2
