// k_entropy.hip -- histograms of reconstructions for the entropy metric of
// centre sweeps (find_shift.cpp:2078-2111): bin (int)((v - min) / inv) with
// inv = (max - min) / n_bins, counted when 0 <= bin <= n_bins, over both images
// of a candidate.  Each block counts into an LDS histogram and adds it to the
// candidate's global one with integer atomics: the counts do not depend on
// the order.
#include <algorithm>

#include "gr_internal.h"

#pragma clang fp contract(off)

namespace {

// Copies of the LDS histogram: bin b's counts of lanes l, l + copies, ... go to
// sh[b * copies + l % copies], so the lanes of a wave that meet in one bin
// (the background of an image) serialise on 64 / copies updates instead of 64.
constexpr int kHistCopyBytes = 32768;

// V4: 16-byte loads (candidates 16-byte aligned).
template <bool V4>
__global__ void __launch_bounds__(256) k_hist(const float *__restrict__ img, long npix, float vmin, float inv, int nb1,
                                              int copies, unsigned *__restrict__ hist) {
    extern __shared__ unsigned sh[];
    const int c = blockIdx.y, my = threadIdx.x & (copies - 1);
    for (int b = threadIdx.x; b < nb1 * copies; b += blockDim.x) sh[b] = 0u;
    __syncthreads();
    const float *base = img + (long)c * npix;
    auto count = [&](float v) {
        const float x = (v - vmin) / inv;
        // (int)x counts for 0 <= (int)x <= n_bins, i.e. -1 < x < n_bins + 1
        if (x > -1.0f && x < (float)nb1) atomicAdd(&sh[(int)x * copies + my], 1u);
    };
    const long t0 = (long)blockIdx.x * blockDim.x + threadIdx.x, step = (long)gridDim.x * blockDim.x;
    const long n4 = V4 ? npix / 4 : 0;
    for (long i = t0; i < n4; i += step) {
        const float4 v = reinterpret_cast<const float4 *>(base)[i];
        count(v.x);
        count(v.y);
        count(v.z);
        count(v.w);
    }
    for (long i = 4 * n4 + t0; i < npix; i += step) count(base[i]);
    __syncthreads();
    for (int b = threadIdx.x; b < nb1; b += blockDim.x) {
        unsigned n = 0u;
        for (int k = 0; k < copies; k++) n += sh[b * copies + k];
        if (n) atomicAdd(&hist[(long)c * nb1 + b], n);
    }
}

__global__ void k_zero_u32(unsigned *p, long n) {
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0u;
}

}  // namespace

hipError_t gr_launch_hist(const float *img, long npix, int n_cand, float vmin, float vmax, int n_bins,
                          unsigned *hist, hipStream_t s) {
    if (n_bins < 1 || n_bins > 16383 || n_cand < 1 || !(vmax > vmin)) return hipErrorInvalidValue;
    const int nb1 = n_bins + 1;
    const long nh = (long)n_cand * nb1;
    hipLaunchKernelGGL(k_zero_u32, dim3((unsigned)((nh + 255) / 256)), dim3(256), 0, s, hist, nh);
    const float inv = (vmax - vmin) / (float)n_bins;
    int copies = 16;
    while (copies > 1 && sizeof(unsigned) * nb1 * copies > (size_t)kHistCopyBytes) copies /= 2;
    // about 2048 workgroups (eight per CU) in all, each of at least 4096 pixels
    const long want = std::max<long>(1, 2048 / n_cand);
    const unsigned bx = (unsigned)std::max<long>(1, std::min<long>(want, npix / 4096));
    const size_t lds = sizeof(unsigned) * nb1 * copies;
    const bool v4 = ((size_t)img & 15) == 0 && npix % 4 == 0;
    if (v4)
        hipLaunchKernelGGL(k_hist<true>, dim3(bx, n_cand), dim3(256), lds, s, img, npix, vmin, inv, nb1, copies, hist);
    else
        hipLaunchKernelGGL(k_hist<false>, dim3(bx, n_cand), dim3(256), lds, s, img, npix, vmin, inv, nb1, copies, hist);
    return hipGetLastError();
}
