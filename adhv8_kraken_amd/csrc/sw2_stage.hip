// Arrays between the caller's layout on the host and the device's.
//
// The device keeps node vectors and blocks wave-sliced, off-diagonal blocks in
// SELL-64 and velocities by component; the caller's are node-major, in the
// reference's row order and interleaved.  The reordering runs on the device,
// which reads or writes a pinned buffer in the caller's order directly (whole
// 512-byte runs per wave over the bus), and the host only copies between that
// buffer and the caller's memory, in two halves by turns so that both work at
// the same time.  Before, the host reordered through pageable copies: an
// off-diagonal array of 11 MB took 3.2 ms, now 0.6, and the state of 25,425
// nodes (1.8 MB) 0.6 ms, now 0.1.  What bounds it is the bus (50 GB/s) and the
// first touch of the caller's pages.
#include <algorithm>
#include <cstring>

#include "sw2_ctx.h"

namespace sw2 {

namespace {

// element i of the caller's array in the device's
__device__ __forceinline__ size_t place(const StageMap &m, size_t i) {
    if (m.kind == StageMap::NODE3) return vidx3((int)(i / 3), (int)(i % 3));
    if (m.kind == StageMap::NODE9) return didx9((int)(i / 9), (int)(i % 9));
    if (m.kind == StageMap::OFFD || m.kind == StageMap::OFFD32) return sell_vidx((size_t)m.pos[i / 9], (int)(i % 9));
    return i;
}

__global__ void __launch_bounds__(256) k_stage_out(StageMap m, size_t first, size_t n, void *stage) {
    const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const size_t i = first + k;
    if (m.kind == StageMap::INTS) {
        ((int *)stage)[k] = ((const int *)m.a[0])[i];
        return;
    }
    double x;
    if (m.kind == StageMap::PAIR) x = ((const double *)(i & 1 ? m.b[0] : m.a[0]))[i >> 1];
    else if (m.kind == StageMap::OFFD32) x = (double)((const float *)m.a[0])[place(m, i)];
    else x = ((const double *)m.a[0])[place(m, i)];
    ((double *)stage)[k] = x;
}

__global__ void __launch_bounds__(256) k_stage_in(StageMap m, size_t first, size_t n, const double *stage) {
    const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const size_t i = first + k;
    const double x = stage[k];
    for (int d = 0; d < m.ndst; d++) {
        if (m.kind == StageMap::PAIR) ((double *)(i & 1 ? m.b[d] : m.a[d]))[i >> 1] = x;
        else ((double *)m.a[d])[place(m, i)] = x;
    }
}

// SELL slot of each off-diagonal block, by row
__global__ void k_offd_pos(int N, const int *row_ptr, const int *sell_ptr, int *pos) {
    const int n = blockIdx.x * blockDim.x + threadIdx.x;
    if (n >= N) return;
    const int p0 = row_ptr[n], p1 = row_ptr[n + 1];
    for (int p = p0; p < p1; p++) pos[p] = 64 * (sell_ptr[n >> 6] + p - p0) + (n & 63);
}

constexpr size_t word(const StageMap &m) { return m.kind == StageMap::INTS ? sizeof(int) : sizeof(double); }

}  // namespace

void launch_offd_pos(Ctx *c) {
    hipLaunchKernelGGL(k_offd_pos, dim3(nblocks_for(c->N, 256)), dim3(256), 0, c->stream, c->N, c->row_ptr,
                       c->sell_ptr, c->offd_pos);
}

hipError_t Stage::wait(int h) {
    if (!pending[h]) return hipSuccess;
    pending[h] = false;
    return hipEventSynchronize(ev[h]);
}

// copies what half h was filled with to the caller, once the device has
hipError_t Stage::drain(int h) {
    if (nseg[h] == 0) return hipSuccess;
    const hipError_t e = wait(h);
    if (e == hipSuccess)
        for (int s = 0; s < nseg[h]; s++) std::memcpy(seg[h][s].user, half(h) + seg[h][s].off, seg[h][s].bytes);
    nseg[h] = 0;
    return e;
}

// closes the current half and goes on with the other
hipError_t Stage::turn_over(hipStream_t st) {
    hipError_t e = hipEventRecord(ev[cur], st);
    pending[cur] = true;
    used = 0;
    cur ^= 1;
    const hipError_t d = drain(cur);
    if (e == hipSuccess) e = d;
    if (e == hipSuccess) e = wait(cur);
    return e;
}

hipError_t Stage::out(hipStream_t st, const StageMap &m, void *user, size_t count) {
    const size_t w = word(m);
    for (size_t i = 0; i < count;) {
        if (HALF - used < 256 || nseg[cur] == MAXSEG) {
            const hipError_t e = turn_over(st);
            if (e != hipSuccess) {
                nseg[0] = nseg[1] = 0;   // the call fails: nothing is written to the caller's arrays later
                return e;
            }
        }
        const size_t n = std::min(count - i, (HALF - used) / w);
        hipLaunchKernelGGL(k_stage_out, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, m, i, n, half(cur) + used);
        seg[cur][nseg[cur]++] = Seg{(char *)user + i * w, used, n * w};
        used = (used + n * w + 255) / 256 * 256;
        i += n;
    }
    return hipSuccess;
}

hipError_t Stage::finish_out(hipStream_t st) {
    if (nseg[cur] == 0) return hipStreamSynchronize(st);   // nothing goes to the caller: the call's work is waited for
    hipError_t e = turn_over(st);   // drains the half before
    const hipError_t d = drain(cur ^ 1);
    nseg[0] = nseg[1] = 0;
    return e == hipSuccess ? d : e;
}

hipError_t Stage::in(hipStream_t st, const StageMap &m, const void *user, size_t count) {
    const size_t w = word(m);
    for (size_t i = 0; i < count;) {
        if (HALF - used < 256) {
            const hipError_t e = turn_over(st);
            if (e != hipSuccess) return e;
        }
        const size_t n = std::min(count - i, (HALF - used) / w);
        std::memcpy(half(cur) + used, (const char *)user + i * w, n * w);
        hipLaunchKernelGGL(k_stage_in, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, m, i, n,
                           (const double *)(half(cur) + used));
        used = (used + n * w + 255) / 256 * 256;
        i += n;
    }
    return hipSuccess;
}

// The half in use stays in use: its kernels may still read it, and the next
// call appends or turns over.
hipError_t Stage::finish_in() { return hipGetLastError(); }

hipError_t Stage::create() {
    hipError_t e = hipHostMalloc((void **)&buf, 2 * HALF);
    for (int h = 0; h < 2 && e == hipSuccess; h++) e = hipEventCreateWithFlags(&ev[h], hipEventDisableTiming);
    return e;
}

void Stage::destroy() {
    for (int h = 0; h < 2; h++)
        if (ev[h]) (void)hipEventDestroy(ev[h]);
    if (buf) (void)hipHostFree(buf);
}

}  // namespace sw2
