// k_ring.hip -- ring-artefact correction of sinograms in place, the
// preprocessing step tomo_recon runs between flat/dark normalisation and
// gridrec (RingCorrectionSinogram, tomo_recon.cpp:3905-3972).  Per slice and
// iteration:
//   m_i   = mean of row (angle) i,  mt = mean of the m_i
//   d_ij *= mt / m_i                          (rows with m_i == 0 untouched)
//   c_j   = mean over i of column j,  l_j = (c_{j-1} + c_j + c_{j+1}) / 3
//           (l_0 = c_0, l_{n-1} = c_{n-1})
//   d_ij  = d_ij - coeff (c_j - l_j)  if that is > 0, else 0
//
// One pass over the data per iteration: mt is common to a slice, so
//   c_j = (mt sum_{m_i != 0} d_ij / m_i + sum_{m_i == 0} d_ij) / n_ang,
// and the pass that applies an iteration to a row has the whole new row in
// registers: it takes the row's new mean and adds d_ij / m_i to its columns'
// partial sums for the next iteration at once.  k_ring_columns then adds a
// slice's partials into the ring estimate.  All sums are taken in a fixed
// order, so results are repeatable; they differ from the reference's
// sequential float sums only by rounding.
//
// The data of a slab that fits the 256 MB memory-side cache streams from
// there: at 16 slices of 900 x 2048 an iteration takes 53 us (about 43 of them
// the pass, 236 MB read and written: 5.5 TB/s) where row means, column means (a
// serial column per thread, eight workgroups per slice) and the correction as
// three passes took 349 us.
#include <algorithm>

#include "gr_internal.h"

#pragma clang fp contract(off)

namespace {

constexpr int kRingThreads = 256;

struct RingArgs {
    float *sino;
    long slice_stride, row_stride;
    int n_ang, n_det, rows, nblocks;  // rows per workgroup, workgroups per slice
    float coeff;
    float *row_mean;   // [n_slices][n_ang]
    float2 *mt;        // [n_slices] mean of the row means: rounded, and the rest
    float *est;        // [n_slices][n_det] coeff (c_j - l_j)
    float *part;       // [n_slices][nblocks][n_det] sums of d / m over the workgroup's rows with m != 0
    float *part0;      // the same for d over the rows with m == 0, where flag0 is set
    int *flag0;        // [n_slices][nblocks]
};

// Sum over the workgroup; red: two alternating sets of per-wave sums (one
// barrier per call).
template <int NT = kRingThreads, typename T>
__device__ __forceinline__ T block_sum(T v, T *red) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    T s = red[0];
#pragma unroll
    for (int w = 1; w < NT / 64; w++) s += red[w];
    return s;
}

// One iteration applied to `rows` rows of one slice (FIRST: nothing applied,
// only the sums taken), then the rows' means and the columns' partial sums of
// the result.  VPT > 0: a thread holds VPT values of the row (n_det <= VPT *
// 256), the next row's loads in flight while a row is summed; V4: as 16-byte
// pieces (rows 16-byte aligned).  VPT = 0, any width: the row is read again
// for the column sums, which live in the partials' memory.
template <int VPT, bool V4, bool FIRST>
__global__ void __launch_bounds__(kRingThreads) k_ring_pass(RingArgs A) {
    __shared__ float red[2][kRingThreads / 64];
    const int s = blockIdx.y, tid = threadIdx.x, n = A.n_det;
    const int i0 = blockIdx.x * A.rows, i1 = min(A.n_ang, i0 + A.rows);
    const long pb = ((long)s * A.nblocks + blockIdx.x) * n;
    float *base = A.sino + s * A.slice_stride;
    const float *est = A.est + (long)s * n;
    const float2 mt2 = FIRST ? make_float2(0.0f, 0.0f) : A.mt[s];
    const float mt = mt2.x;
    float *rm = A.row_mean + (long)s * A.n_ang;
    bool zero_rows = false;
    // value d of a row of mean m after the iteration, d mt / m - e; where mt / m
    // is an ordinary number it is taken once per row, with its rounding error
    // and mt's (which would scale the whole slice, once per iteration), and a value costs two fused multiply-adds: one rounding, where a product,
    // a quotient and a difference are three
    struct Scale {
        float rs, lo;
        bool fast;
    };
    auto ordinary = [](float x) { return fabsf(x) > 1e-30f && fabsf(x) < 1e30f; };  // false for NaN
    auto scale_of = [&](float m) {
        const float rs = mt / m;
        return Scale{rs, (__builtin_fmaf(-rs, m, mt) + mt2.y) / m, ordinary(rs) && ordinary(m)};
    };
    auto apply = [&](float d, float m, const Scale &f, float e) {
        float t;
        if (m != 0.0f && f.fast) {
            t = __builtin_fmaf(d, f.rs, __builtin_fmaf(d, f.lo, -e));
        } else {
            if (m != 0.0f) d = d * mt / m;
            t = d - e;
        }
        return t > 0.0f ? t : 0.0f;
    };
    if constexpr (VPT > 0) {
        constexpr int W = V4 ? 4 : 1;
        auto col = [&](int k) { return W * (tid + kRingThreads * (k / W)) + k % W; };
        float cur[VPT], nxt[VPT], acc[VPT], e[VPT];
        auto load = [&](int i, float (&v)[VPT]) {
            const float *row = base + (long)i * A.row_stride;
#pragma unroll
            for (int k = 0; k < VPT; k += W) {
                const int j = col(k);
                if constexpr (V4) {  // n is a multiple of four
                    const float4 x = j < n ? *reinterpret_cast<const float4 *>(row + j) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                    v[k] = x.x;
                    v[k + 1] = x.y;
                    v[k + 2] = x.z;
                    v[k + 3] = x.w;
                } else {
                    v[k] = j < n ? row[j] : 0.0f;
                }
            }
        };
        if (i0 < i1) load(i0, cur);
#pragma unroll
        for (int k = 0; k < VPT; k++) {
            acc[k] = 0.0f;
            e[k] = !FIRST && col(k) < n ? est[col(k)] : 0.0f;
        }
        for (int i = i0; i < i1; i++) {
            if (i + 1 < i1) load(i + 1, nxt);
            if (!FIRST) {
                const float m = rm[i];
                const Scale f = scale_of(m);
                float *row = base + (long)i * A.row_stride;
#pragma unroll
                for (int k = 0; k < VPT; k++) cur[k] = apply(cur[k], m, f, e[k]);
#pragma unroll
                for (int k = 0; k < VPT; k += W) {
                    const int j = col(k);
                    if (j < n) {
                        if constexpr (V4)
                            *reinterpret_cast<float4 *>(row + j) = make_float4(cur[k], cur[k + 1], cur[k + 2], cur[k + 3]);
                        else
                            row[j] = cur[k];
                    } else {
#pragma unroll
                        for (int c = 0; c < W; c++) cur[k + c] = 0.0f;
                    }
                }
            }
            float sum = 0.0f;
#pragma unroll
            for (int k = 0; k < VPT; k++) sum += cur[k];
            const float m = block_sum(sum, red[i & 1]) / (float)n;
            if (tid == 0) rm[i] = m;  // read above by every thread before the barrier
            if (m != 0.0f) {
                const float inv = 1.0f / m;
                if (ordinary(m)) {
#pragma unroll
                    for (int k = 0; k < VPT; k++) acc[k] = __builtin_fmaf(cur[k], inv, acc[k]);
                } else {
#pragma unroll
                    for (int k = 0; k < VPT; k++) acc[k] += cur[k] / m;
                }
            } else {
#pragma unroll
                for (int k = 0; k < VPT; k++)
                    if (col(k) < n) {
                        float *p = A.part0 + pb + col(k);
                        *p = zero_rows ? *p + cur[k] : cur[k];
                    }
                zero_rows = true;
            }
#pragma unroll
            for (int k = 0; k < VPT; k++) cur[k] = nxt[k];
        }
#pragma unroll
        for (int k = 0; k < VPT; k++)
            if (col(k) < n) A.part[pb + col(k)] = acc[k];
    } else {
        for (int j = tid; j < n; j += kRingThreads) A.part[pb + j] = 0.0f;
        for (int i = i0; i < i1; i++) {
            float *row = base + (long)i * A.row_stride;
            float sum = 0.0f;
            if (FIRST) {
                for (int j = tid; j < n; j += kRingThreads) sum += row[j];
            } else {
                const float m = rm[i];
                const Scale f = scale_of(m);
                for (int j = tid; j < n; j += kRingThreads) sum += row[j] = apply(row[j], m, f, est[j]);
            }
            const float m = block_sum(sum, red[i & 1]) / (float)n;
            if (tid == 0) rm[i] = m;
            // each thread reads back what it wrote itself
            float *p = (m != 0.0f ? A.part : A.part0) + pb;
            const bool add = m != 0.0f || zero_rows;
            for (int j = tid; j < n; j += kRingThreads) {
                const float x = m != 0.0f ? row[j] / m : row[j];
                p[j] = add ? p[j] + x : x;
            }
            if (m == 0.0f) zero_rows = true;
        }
    }
    if (tid == 0) A.flag0[(long)s * A.nblocks + blockIdx.x] = zero_rows ? 1 : 0;
}

// The ring estimate coeff (c_j - l_j) of 62 columns of one slice from the
// partials: 64 columns (one more each side) x 16 groups of workgroups'
// partials, and the mean of the row means.  In double up to the estimate:
// c_j - l_j is a small difference of near equals, and an error of the mean scales
// the whole slice: over 20 iterations 4.6e-7 in all with floats, 1.1e-7
// so (16 slices of 900 x 2048).
constexpr int kEstCols = 62, kEstGroups = 16;
__global__ void __launch_bounds__(64 * kEstGroups) k_ring_columns(RingArgs A) {
    __shared__ double red[kEstGroups];
    __shared__ double sa[kEstGroups][64], sb[kEstGroups][64], sc[64];
    const int s = blockIdx.y, tid = threadIdx.x, n = A.n_det;
    const int c = tid & 63, g = tid >> 6;
    const int j = min(max((int)blockIdx.x * kEstCols + c - 1, 0), n - 1);
    const float *pa = A.part + (long)s * A.nblocks * n + j, *p0 = A.part0 + (long)s * A.nblocks * n + j;
    const int *f0 = A.flag0 + (long)s * A.nblocks;
    double a = 0.0, b = 0.0;
    for (int k0 = g; k0 < A.nblocks; k0 += 8 * kEstGroups) {  // eight loads in flight
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = k0 + u * kEstGroups < A.nblocks ? pa[(long)(k0 + u * kEstGroups) * n] : 0.0f;
#pragma unroll
        for (int u = 0; u < 8; u++) a += (double)v[u];
    }
    for (int k = g; k < A.nblocks; k += kEstGroups)
        if (f0[k]) b += (double)p0[(long)k * n];
    sa[g][c] = a;
    sb[g][c] = b;
    const float *rm = A.row_mean + (long)s * A.n_ang;
    double v = 0.0;
    for (int i = tid; i < A.n_ang; i += 64 * kEstGroups) v += (double)rm[i];
    const double mt = block_sum<64 * kEstGroups>(v, red) / (double)A.n_ang;  // its barrier covers sa and sb
    if (tid == 0 && blockIdx.x == 0) {
        const float hi = (float)mt, lo = (float)(mt - (double)hi);
        A.mt[s] = make_float2(hi, fabsf(lo) < fabsf(hi) ? lo : 0.0f);  // none beside an infinity or a NaN
    }
    if (tid < 64) {
        a = b = 0.0;
#pragma unroll
        for (int k = 0; k < kEstGroups; k++) {
            a += sa[k][c];
            b += sb[k][c];
        }
        sc[c] = (a * mt + b) / (double)A.n_ang;
    }
    __syncthreads();
    const int jo = (int)blockIdx.x * kEstCols + tid;
    if (tid < kEstCols && jo < n) {
        const double cm = sc[tid + 1];
        const double l = (jo == 0 || jo == n - 1) ? cm : (sc[tid] + cm + sc[tid + 2]) / 3.0;
        A.est[(long)s * n + jo] = (float)((cm - l) * (double)A.coeff);
    }
}

// Rows per workgroup: about 1024 workgroups (four per CU) of at least four
// rows -- fewer rows mean more partials to add per column.
int ring_rows(int n_slices, int n_ang) {
    const long all = (long)n_slices * n_ang;
    return (int)std::min<long>(n_ang, std::max<long>(4, (all + 1023) / 1024));
}

template <bool FIRST>
void launch_pass(const RingArgs &A, int n_slices, hipStream_t s) {
    const dim3 grid(A.nblocks, n_slices), block(kRingThreads);
    const bool v4 = A.n_det % 4 == 0 && A.row_stride % 4 == 0 && A.slice_stride % 4 == 0 && ((size_t)A.sino & 15) == 0;
#define GR_RING(V)                                                                      \
    do {                                                                                \
        if (v4) hipLaunchKernelGGL((k_ring_pass<V, true, FIRST>), grid, block, 0, s, A); \
        else hipLaunchKernelGGL((k_ring_pass<V, false, FIRST>), grid, block, 0, s, A);   \
    } while (0)
    if (A.n_det <= 4 * kRingThreads) GR_RING(4);
    else if (A.n_det <= 8 * kRingThreads) GR_RING(8);
    else if (A.n_det <= 16 * kRingThreads) GR_RING(16);
    else hipLaunchKernelGGL((k_ring_pass<0, false, FIRST>), grid, block, 0, s, A);
#undef GR_RING
}

size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

}  // namespace

size_t gr_ring_scratch_bytes(int n_slices, int n_ang, int n_det) {
    const int rows = ring_rows(n_slices, n_ang), nb = (n_ang + rows - 1) / rows;
    const size_t ns = (size_t)n_slices;
    return up256(4 * ns * n_ang) + up256(8 * ns) + up256(4 * ns * n_det) + 2 * up256(4 * ns * nb * n_det) +
           up256(4 * ns * nb);
}

hipError_t gr_launch_ring(float *sino, long slice_stride, long row_stride, int n_slices, int n_ang, int n_det,
                          float coeff, int iterations, void *scratch, hipStream_t s) {
    const int rows = ring_rows(n_slices, n_ang), nb = (n_ang + rows - 1) / rows;
    const size_t ns = (size_t)n_slices;
    RingArgs A{sino, slice_stride, row_stride, n_ang, n_det, rows, nb, coeff, nullptr, nullptr, nullptr, nullptr,
               nullptr, nullptr};
    char *p = (char *)scratch;
    auto take = [&](size_t count) {
        char *q = p;
        p += up256(4 * count);
        return q;
    };
    A.row_mean = (float *)take(ns * n_ang);
    A.mt = (float2 *)take(2 * ns);
    A.est = (float *)take(ns * n_det);
    A.part = (float *)take(ns * nb * n_det);
    A.part0 = (float *)take(ns * nb * n_det);
    A.flag0 = (int *)take(ns * nb);
    launch_pass<true>(A, n_slices, s);
    for (int it = 0; it < iterations; it++) {
        hipLaunchKernelGGL(k_ring_columns, dim3((n_det + kEstCols - 1) / kEstCols, n_slices), dim3(64 * kEstGroups), 0, s,
                           A);
        launch_pass<false>(A, n_slices, s);
    }
    return hipGetLastError();
}
