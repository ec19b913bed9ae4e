// noalloc.hip -- the per-voxel stress update on caller-owned device buffers
// with no device allocation: evpgpu_newton_device_noalloc.
//
// It runs the kernel evpgpu_newton_host runs (k_newton_batch, the full update of
// src/evolution.c:44-310 for a batch of voxels) on device pointers the
// caller passes, for callers that cannot allocate.  Its scratch is two words
// that the context holds from its creation, so calls on different contexts
// do not meet; calls on one context are the caller's to keep apart, as
// everywhere.
//
// One wait per call: the update reads the index check's word on the device
// and does nothing where it is set.
#include "evpgpu_impl.h"

namespace {

// largest batch: 2^21 voxels (a 128^3 grid)
constexpr long long NOALLOC_MAX_N = EVPGPU_NOALLOC_MAX_VOXELS;

// status = EVPGPU_ERR_ARG when a voxel's phase is outside 1..nphases or its
// orientation index outside 0..n_orient-1 (the kernel reads both unchecked)
__global__ void k_check_ids(const int *__restrict__ phase, const int *__restrict__ orient, long long n,
                            int nphases, int n_orient, int *status)
{
    const long long v = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= n) return;
    const int p = phase[v], o = orient[v];
    if (p < 1 || p > nphases || o < 0 || o >= n_orient) atomicCAS(status, 0, (int)EVPGPU_ERR_ARG);
}

} // namespace

extern "C" int evpgpu_newton_device_noalloc(evpgpu_ctx *c, int n, const int *phase, const int *orient,
                                            const double *sgr, int n_orient, double *sig6,
                                            const double *strain6, const double *eps6,
                                            const double *tranmat9, const double *crss24, double *edot6,
                                            double *gamdot12, double *err2, int *niter)
{
    if (!c || n < 1 || !phase || !orient || !sgr || n_orient < 1 || !sig6 || !strain6 || !eps6 ||
        !tranmat9 || !crss24 || !edot6 || !gamdot12 || !err2 || !niter || !c->have_phases ||
        !c->have_loading)
        return EVPGPU_ERR_ARG;
    if ((long long)n > NOALLOC_MAX_N) return EVPGPU_ERR_SIZE;
    // the update's status word and the index check's: both start at zero on
    // every call (a fill kernel, not a memset node), and the update does
    // nothing where the check failed, so that one wait serves the two
    int *status = c->d_status + 1, *bad = c->d_status + 2;
    int st = fill_zero_int(c, status, 2);
    if (st) return st;
    hipLaunchKernelGGL(k_check_ids, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, c->stream, phase, orient,
                       (long long)n, c->nphases, n_orient, bad);
    if (hipGetLastError() != hipSuccess) return EVPGPU_ERR_HIP;
    NewtonParams P = context_newton_params(c);
    P.dd = 0; // the power-law update on the caller's CRSS, as evpgpu_newton_host
    P.skip = bad;
    st = newton_batch_launch(c, P, sig6, sig6, strain6, eps6, edot6, tranmat9, crss24, gamdot12, phase, orient, sgr,
                             n, status, err2, niter);
    if (st) return st;
    // the two words come back through the context's pinned ones
    if (hipMemcpyAsync(c->h_status, status, 2 * sizeof(int), hipMemcpyDeviceToHost, c->stream) != hipSuccess ||
        hipStreamSynchronize(c->stream) != hipSuccess)
        return EVPGPU_ERR_HIP;
    return c->h_status[1] ? c->h_status[1] : c->h_status[0];
}
