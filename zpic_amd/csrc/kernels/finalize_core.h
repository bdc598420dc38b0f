/*
 * finalize_core.h - energy and push count after a push, shared by the push,
 * current and batch kernels.
 */
#ifndef ZK_FINALIZE_CORE_H
#define ZK_FINALIZE_CORE_H

#include "common.h"

namespace zk {

/* Sum the energy partials and count the pushes (em2d/particles.c:1231,
 * 1267).  The order of the sum is fixed (thread t adds partials t, t + B,
 * t + 2B, ... with coalesced loads, then a tree over the B threads; B a
 * power of two up to 1024), so every run sums alike. */
__device__ inline void finalize_body(zk_spec_ctr *ctr, const double *epart, int nparts, double qm, double dx0,
                                     double dx1)
{
    __shared__ double part[1024];
    double s = 0.0;
    for (int i = threadIdx.x; i < nparts; i += blockDim.x) s += epart[i];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int o = (int)blockDim.x / 2; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) part[threadIdx.x] += part[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        const double tot = part[0];
        ctr->energy = qm * tot * dx0 * dx1;
        ctr->npush += (unsigned long long)(ctr->np_total - ctr->n_dead - ctr->n_slack);
    }
}

/* Species k of the set; the counters also go to the host where asked for.
 * One wave stores them word by word, each lane makes its word visible to
 * the host, and then lane 0 stores the sequence number that completes
 * them. */
__device__ inline void finalize_set_body(const zk_finalize_set &f, int k)
{
    finalize_body(f.ctr[k], f.epart[k], f.nparts[k], f.qm[k], f.dx0[k], f.dx1[k]);
    if (!f.probe[k]) return;
    __syncthreads();
    if (threadIdx.x >= ZK_WAVE) return;
    static_assert(sizeof(zk_spec_ctr) % 4 == 0 && sizeof(zk_spec_ctr) / 4 <= ZK_WAVE, "one word a lane");
    if (threadIdx.x < sizeof(zk_spec_ctr) / 4)
        __hip_atomic_store((unsigned *)&f.probe[k]->c + threadIdx.x, ((const unsigned *)f.ctr[k])[threadIdx.x],
                           __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    __threadfence_system();
    if (threadIdx.x == 0)
        __hip_atomic_store(&f.probe[k]->seq, f.seq[k], __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

} // namespace zk

#endif
