// k_ifft2.hip -- K3 + K4: 2D inverse FFT of the grid, deapodization and crop.
//
// Replaces phases 2 and 3 of do_recon (gridrec/GridrecCPP/Gridrec5.2/grid.cpp:311-411):
//   fourn(H, {M, M}, 2, -1)                      x[p][q] = sum_{u,v} H[u][v] e^{-2 pi i (up+vq)/M}
//   S1[j][k] = winv[j]*winv[k] * Re x[iu(j)][iv(k)]
//   S2[j][k] = winv[j]*winv[k] * Im x[iu(j)][iv(k)]
// where iu(j) = M-M02+j for j < M02 and j-M02 after (the four-corner wrap).
//
// Only the requested window [off, off+n) of rows and columns is produced, so
// both passes are pruned: K3 transforms every row of Ht (one per b, over a)
// but keeps only the n outputs p = iu(j) of the window; K4 transforms those
// n columns down b, keeps the n outputs q = iv(k) and writes the two images
// row by row with the deapodization product fused in.
#include <algorithm>
#include <atomic>

#include "gr_fft.hpp"
#include "gr_gather.hpp"
#include "gr_internal.h"

#pragma clang fp contract(off)

namespace {

__device__ __forceinline__ long corner_index(long j, long M, long M02) {
    return j < M02 ? M - M02 + j : j - M02;
}

struct RowsArgs {
    const float2 *ht;
    float2 *z;
    const float2 *tw;
    const int2 *row_tiles;  // per tile row the written tiles [lo, hi]; the others are zeros
    int M, radix;
    long M02, out_off, out_n;
    int row_lo, row_hi;  // the grid rows that are not all zeros
};

// Output hook of the row transform: FFT output i lands in window column
// jj = j' - out_off, where corner_index(j') = i (outputs that map to no
// window column are dropped), at Z's column-blocked place for the row (dst =
// the pair's Z + 4 b).
struct WindowRow {
    float2 *dst;
    int M, m02, off, out_n;
    static constexpr bool enabled = true;
    __device__ __forceinline__ void prep(int, int) {}
    __device__ __forceinline__ void operator()(int i, float2 v, int) const {
        const int jp = i >= M - m02 ? i - (M - m02) : i + m02;
        put(jp - off, v);
        if (i >= M - m02 && i <= m02) put(i + m02 - off, v);  // an image wider than the grid (sampl < 1) repeats it
    }
    __device__ __forceinline__ void put(int jj, float2 v) const {
        if (jj >= 0 && jj < out_n) dst[(long)(jj >> 2) * M * 4 + (jj & 3)] = v;
    }
};

// Row of Z written by row-transform workgroup x (of nx, CW rows each): the
// workgroups are dealt to the 8 XCDs round robin, so x, x + 8, ... share one
// XCD's L2; numbering them so that the 4 rows whose 32-byte pieces make up
// each 128-byte line of the column-blocked Z come from one XCD, one after
// another, lets its L2 merge the pieces into whole lines.
__device__ __forceinline__ int row_group(int x, int nx, int CW) {
    const int G = 4 / CW;  // workgroups per 4 rows
    if (G <= 1 || nx % (8 * G)) return x;
    return (x / (8 * G)) * (8 * G) + (x % 8) * G + (x / 8) % G;
}

// Loads and LDS stores in loops unrolled to the per-thread bound (M <= 4 MAXB
// nthr), every load issued before the first store: one memory latency per
// row instead of one per element.  CW rows per workgroup, transformed side by
// side by CW thread groups (shared barriers).
template <int MAXB, int CW>
__global__ void __launch_bounds__(1024) k_ifft_rows(RowsArgs A) {
    extern __shared__ float2 lds[];
    constexpr int EPT = 4 * MAXB;
    const int nthr = (int)blockDim.x / CW;
    const int grp = (int)threadIdx.x / nthr, tid = (int)threadIdx.x % nthr;
    const int b = A.row_lo + row_group((int)blockIdx.x, (int)gridDim.x, CW) * CW + grp, p = blockIdx.y;
    const int M = A.M;
    float2 *row = lds + (long)grp * M;
    const float2 *src = A.ht + ((long)p * M + b) * M;
    const int2 lh = A.row_tiles[b >> 3];
    const int lo = lh.x, hi = lh.y;
    float2 v[EPT];
#pragma unroll
    for (int r = 0; r < EPT; r++) {
        const int i = tid + r * nthr, tx = i >> 3;
        v[r] = i < M && tx >= lo && tx <= hi ? src[i] : make_float2(0.0f, 0.0f);
    }
#pragma unroll
    for (int r = 0; r < EPT; r++) {
        const int i = tid + r * nthr;
        if (i < M) row[gr_lds_idx(i)] = v[r];
    }
    __syncthreads();
    float2 *dst = A.z + (long)p * M * gr_z_cols(A.out_n) + 4L * b;
    const int out_n = (int)A.out_n, off = (int)A.out_off, m02 = (int)A.M02;
    // when the last pass is radix 16, the window's outputs go to HBM straight
    // from its registers: output i is window column j' = corner_index^-1(i)
    if (gr_lds_fft<-1, MAXB>(row, M, A.tw, tid, nthr, A.radix, WindowRow{dst, M, m02, off, out_n})) return;
    // an array of its own (reusing v would keep the loaded row alive, in
    // registers, through the whole transform)
    float2 o[EPT];
#pragma unroll
    for (int r = 0; r < EPT; r++) {
        const int jj = tid + r * nthr;
        o[r] = row[gr_lds_idx((int)corner_index(jj < out_n ? off + jj : off, M, m02))];
    }
#pragma unroll
    for (int r = 0; r < EPT; r++) {
        const int jj = tid + r * nthr;
        if (jj < out_n) dst[(long)(jj >> 2) * M * 4 + (jj & 3)] = o[r];
    }
    for (int jj = tid + EPT * nthr; jj < out_n; jj += nthr)  // a window wider than the grid
        dst[(long)(jj >> 2) * M * 4 + (jj & 3)] = row[gr_lds_idx((int)corner_index(off + jj, M, m02))];
}

struct ColsArgs {
    const float2 *z;
    float *out;
    const float2 *tw;
    const float *winv;
    long out_slice_stride, out_row_stride;
    int M, cw, n_slices, pair0, radix;
    long M02, out_off, out_n;
    int row_lo, row_hi;  // rows of Z that the row transform wrote; the others read as zeros
};

// Output hook of the column transform: FFT output i is image column
// kk = k' - out_off of this row, corner_index(k') = i, scaled by the
// deapodization cu * winv[k'] (grid.cpp:401); rows past the window have
// r1 = nullptr and write nothing.  prep loads winv[k'] of every output of the
// thread (k' < M always: no bounds test, so the loads are issued together
// rather than each behind the previous output's stores).  NS: output slots.
template <int NS>
struct WindowCol {
    float *r1, *r2;
    const float *winv;
    float cu;
    int M, m02, off, out_n;
    float wv[NS];
    static constexpr bool enabled = true;
    __device__ __forceinline__ int kprime(int i) const { return i >= M - m02 ? i - (M - m02) : i + m02; }
    __device__ __forceinline__ void prep(int i, int s) { wv[s] = winv[kprime(i)]; }
    __device__ __forceinline__ void operator()(int i, float2 v, int s) const {
        put(kprime(i) - off, v, wv[s]);
        if (i >= M - m02 && i <= m02) put(i + m02 - off, v, winv[i + m02]);  // as WindowRow
    }
    __device__ __forceinline__ void put(int kk, float2 v, float w) const {
        if (r1 && kk >= 0 && kk < out_n) {
            const float corrn = cu * w;
            r1[kk] = corrn * v.x;
            if (r2) r2[kk] = corrn * v.y;
        }
    }
};

// Column group of a workgroup.  Workgroups are dealt to the 8 XCDs round
// robin, each XCD with its own L2; numbering the groups so that x, x+8, x+16,
// ... (one XCD) take neighbouring column groups keeps neighbouring blocks of
// the column-blocked Z on one XCD (narrower groups than four columns share
// each block's lines).
__device__ __forceinline__ long column_group(unsigned x, unsigned ngroups) {
    if (ngroups % 8u) return x;
    return (long)(x % 8u) * (ngroups / 8u) + x / 8u;
}

// CW > 0: CW neighbouring columns per workgroup, transformed side by side by
// CW groups of nthr/CW threads (the workgroup's barriers are shared, so the
// groups run the same passes in lockstep); the fill reads the CW columns of
// a row as neighbouring bytes of the column-blocked Z (four columns: one
// contiguous block).  CW = 0: A.cw columns one after another on all threads
// (small M, where CW * M is small).
template <int MAXB, int CW>
__global__ void __launch_bounds__(1024) k_ifft_cols(ColsArgs A) {
    extern __shared__ float2 cols[];  // cw columns of gr_lds_len(M) slots
    const int p = blockIdx.y;
    const int M = A.M, cw = CW ? CW : A.cw;
    const long c0 = column_group(blockIdx.x, gridDim.x) * cw;
    const int nthr = CW ? (int)blockDim.x / CW : (int)blockDim.x;
    const int tid = CW ? (int)threadIdx.x % nthr : (int)threadIdx.x;
    const int grp = CW ? (int)threadIdx.x / nthr : 0;
    const float2 *zp = A.z + (long)p * M * gr_z_cols(A.out_n);  // column-blocked
    const int out_n = (int)A.out_n;
    constexpr int EPT = 4 * MAXB;  // rows per thread and column: M <= 4 MAXB nthr
    if (CW) {
        // unrolled, every load before the first LDS store (buffer loads: a
        // column past the window reads zeros without a branch); the CW
        // columns of a row come from neighbouring lanes
        const GrBuf zb = gr_buf(zp, (unsigned)((long)M * gr_z_cols(out_n) * sizeof(float2)));
        float2 v[EPT];
#pragma unroll
        for (int r = 0; r < EPT; r++) {
            const int idx = (int)threadIdx.x + r * (int)blockDim.x;
            const int b = idx / CW, c = idx - b * CW;
            const bool in = b >= A.row_lo && b < A.row_hi && c0 + c < out_n;
            v[r] = gr_buf_ld2(zb, in ? (unsigned)(gr_z_index(M, b, c0 + c) * sizeof(float2)) : kGrBufNone);
        }
#pragma unroll
        for (int r = 0; r < EPT; r++) {
            const int idx = (int)threadIdx.x + r * (int)blockDim.x;
            const int b = idx / CW, c = idx - b * CW;
            if (b < M) cols[c * gr_lds_len(M) + gr_lds_idx(b)] = v[r];
        }
    } else if (cw == 1) {
        for (int b = tid; b < M; b += nthr)
            cols[gr_lds_idx(b)] =
                c0 < out_n && b >= A.row_lo && b < A.row_hi ? zp[gr_z_index(M, b, c0)] : make_float2(0.0f, 0.0f);
    } else {
        for (int idx = threadIdx.x; idx < cw * M; idx += blockDim.x) {  // CW: cw * M <= 20480; else <= 16384
            const int b = idx / cw, c = idx - b * cw;
            cols[c * gr_lds_len(M) + gr_lds_idx(b)] =
                c0 + c < out_n && b >= A.row_lo && b < A.row_hi ? zp[gr_z_index(M, b, c0 + c)] : make_float2(0.0f, 0.0f);
        }
    }
    __syncthreads();
    const long s1 = 2L * (A.pair0 + p), s2 = s1 + 1;
    float *o1 = A.out + s1 * A.out_slice_stride;
    float *o2 = s2 < A.n_slices ? A.out + s2 * A.out_slice_stride : nullptr;
    if (CW) {
        // when the last pass is radix 16, each group writes its image row
        // straight from that pass's registers (deapodization on the way)
        const long jj = c0 + grp;
        const bool live = jj < A.out_n;
        WindowCol<16 * ((MAXB + 3) / 4)> wc{live ? o1 + jj * A.out_row_stride : nullptr,
                                            live && o2 ? o2 + jj * A.out_row_stride : nullptr,
                                            A.winv, live ? A.winv[A.out_off + jj] : 0.0f, M, (int)A.M02,
                                            (int)A.out_off, out_n, {}};
        if (gr_lds_fft<-1, MAXB>(cols + grp * gr_lds_len(M), M, A.tw, tid, nthr, A.radix, wc)) return;
    } else {
        for (int c = 0; c < cw; c++) gr_lds_fft<-1, MAXB>(cols + c * gr_lds_len(M), M, A.tw, tid, nthr, A.radix);
    }

    for (int c = CW ? grp : 0; c < (CW ? grp + 1 : cw); c++) {
        const long jj = c0 + c;
        if (jj >= A.out_n) break;
        const float cu = A.winv[A.out_off + jj];
        const float2 *col = cols + c * gr_lds_len(M);
        float *r1 = o1 + jj * A.out_row_stride, *r2 = o2 ? o2 + jj * A.out_row_stride : nullptr;
        const int off = (int)A.out_off, m02 = (int)A.M02;
        if (CW) {  // unrolled: the winv loads of all of a thread's outputs in flight at once
            float wk[EPT];
            float2 v[EPT];
#pragma unroll
            for (int r = 0; r < EPT; r++) {
                const int kk = tid + r * nthr, k = off + kk;
                if (kk < out_n) {
                    wk[r] = A.winv[k];
                    v[r] = col[gr_lds_idx(k < m02 ? M - m02 + k : k - m02)];
                }
            }
#pragma unroll
            for (int r = 0; r < EPT; r++) {
                const int kk = tid + r * nthr;
                if (kk < out_n) {
                    const float corrn = cu * wk[r];  // grid.cpp:401
                    r1[kk] = corrn * v[r].x;
                    if (r2) r2[kk] = corrn * v[r].y;
                }
            }
        }
        // (CW: a window wider than the grid)
        for (int kk = CW ? tid + EPT * nthr : tid; kk < out_n; kk += nthr) {
            const int k = off + kk;
            const float corrn = cu * A.winv[k];  // grid.cpp:401
            const float2 v = col[gr_lds_idx(k < m02 ? M - m02 + k : k - m02)];
            r1[kk] = corrn * v.x;
            if (r2) r2[kk] = corrn * v.y;
        }
    }
}

// ---- persistent transforms ----------------------------------------------------
//
// For M = 1024 .. 8192 with radix-16 passes: one workgroup of 1024 threads runs
// per CU and loops over items of CW = 16384 / M neighbouring rows (columns),
// which with the twiddles fill the CU's 160 KiB of LDS.  Each thread
// loads elements j + r M/16, r < 16, of one row -- exactly the inputs of
// the first radix-16 butterfly j -- so that pass runs from the registers that
// received the loads; the next item's loads are issued into the same
// registers right after, and stay in flight while the other passes run on
// twiddles from LDS (no global load in between: the loads of all of a wave
// complete in order, so any would wait for them).  The passes end in LDS
// and an epilogue stores the window (an output hook would need
// sixteen more registers for its deapodization factors: spills); the closing
// radix-2 pass of M = 8192 happens there, a window's outputs needing half of
// it each.  Same arithmetic, twiddles and output values as the one-shot
// kernels: bitwise their images.
//
// Bound by HBM: at M = 4096 (32 pairs of 1500 x 2048) rows 1255 us and columns
// 671, 4.4 and 4.8 TB/s, a copy's 4.7; M = 2048 (32 pairs of 720 x 1024) 323 and
// 185 us, one-shot 607 and 383; M = 8192 (8 pairs of 1800 x 2560) 990 and 990,
// one-shot 1980 (rows that hold only zeros included) and 1490; M = 1024 (16
// pairs of 451 x 777, whole images) 52 and 57, one-shot 88 and 140.
constexpr int kPfThreads = 1024;
template <int LM>
struct Pf {
    static constexpr int M = 1 << LM, CW = 16384 / M, nthr = M / 16;  // threads per row
    static constexpr int stride = M + 4;  // padded: neighbouring rows' first-pass stores use different banks
    static constexpr bool last2 = LM == 13;                          // 16 16 16 2
    static constexpr int r3 = last2 ? 16 : M / 256;                  // the third pass's radix
    static constexpr int tw = 15 * 16 + (r3 - 1) * 256;              // twiddles of passes two and three
    static constexpr size_t lds = sizeof(float2) * ((size_t)CW * stride + tw);
    static constexpr int cpb = CW < 4 ? CW : 4;                      // columns of an item in a block of Z
    static constexpr int blocks = CW < 4 ? 1 : CW / 4, tpb = kPfThreads / blocks;
};

// The passes on a row already loaded: the arithmetic of gr_lds_fft, with the
// row's LDS places (gr_lds_idx) as a few addresses per thread plus constants:
// for j < nthr, i = j + r nthr sits at (j ^ (j >> 4)) ^ (r nthr / 16 mod 32),
// plus r nthr; an output of the first pass, i = 16 j + q, at (16 j ^ (j mod 32))
// ^ q; one of the second, 256 J + k + 16 q, at (256 J + k + 16 (J mod 2)) ^ 17 q.
// (With gr_lds_idx evaluated per access the addresses were half of the
// kernels' VALU instructions, and those bound them.)
__device__ __forceinline__ int pf_place(int j) { return j ^ ((j >> 4) & 31); }

__device__ __forceinline__ void pf_first(float2 *buf, float2 (&v)[16], int j) {
    gr_dft16<-1>(v);
    const int b = (j << 4) ^ (j & 31);
#pragma unroll
    for (int q = 0; q < 16; q++) buf[b ^ q] = v[4 * (q & 3) + (q >> 2)];
}

template <int LM>
__device__ __forceinline__ void pf_rest(float2 *buf, const float2 *tw, int tid) {
    using F = Pf<LM>;
    constexpr int NT = F::nthr;
    float2 v[16], w[15];
    {
        const int k = tid & 15, J = tid >> 4, in = pf_place(tid), out = (J << 8) + k + ((J & 1) << 4);
#pragma unroll
        for (int r = 1; r < 16; r++) w[r - 1] = tw[(r - 1) * 16 + k];
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = buf[(in ^ ((r * (NT / 16)) & 31)) + r * NT];
#pragma unroll
        for (int r = 1; r < 16; r++) v[r] = gr_cmul(v[r], w[r - 1]);
        gr_dft16<-1>(v);
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 16; q++) buf[out ^ (17 * q)] = v[4 * (q & 3) + (q >> 2)];
        __syncthreads();
    }
    tw += 15 * 16;
    if constexpr (F::r3 == 16) {
        const int k = tid & 255, in = pf_place(tid), out = (tid & ~255) * 16 + pf_place(k);
#pragma unroll
        for (int r = 1; r < 16; r++) w[r - 1] = tw[(r - 1) * 256 + k];
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = buf[(in ^ ((r * (NT / 16)) & 31)) + r * NT];
#pragma unroll
        for (int r = 1; r < 16; r++) v[r] = gr_cmul(v[r], w[r - 1]);
        gr_dft16<-1>(v);
        if (LM != 12) __syncthreads();  // M = 4096: a thread writes the places it read
#pragma unroll
        for (int q = 0; q < 16; q++) buf[(out ^ ((q & 1) << 4)) + 256 * q] = v[4 * (q & 3) + (q >> 2)];
    } else {  // 256 butterflies of radix 8 or 4, in place
#pragma unroll
        for (int c = 0; c < 256 / NT; c++) {
            const int j = tid + c * NT, in = pf_place(j);
            constexpr int R = F::r3;
            float2 x[R];
#pragma unroll
            for (int r = 0; r < R; r++) x[r] = buf[(in ^ ((r & 1) << 4)) + 256 * r];
#pragma unroll
            for (int r = 1; r < R; r++) x[r] = gr_cmul(x[r], tw[(r - 1) * 256 + j]);
            if constexpr (R == 8) gr_dft8<-1>(x);
            else gr_dft4<-1>(x[0], x[1], x[2], x[3]);
#pragma unroll
            for (int r = 0; r < R; r++) buf[(in ^ ((r & 1) << 4)) + 256 * r] = x[r];
        }
    }
    __syncthreads();
}

// Columns: an item is CW neighbouring columns of one pair, contiguous blocks of
// the column-blocked Z (M = 8192: half of one).
template <int LM>
__global__ void __launch_bounds__(kPfThreads) k_ifft_cols_pf(ColsArgs A, int n_items) {
    using F = Pf<LM>;
    constexpr int M = F::M, CW = F::CW, NT = F::nthr;
    extern __shared__ float2 lds[];
    float2 *tw = lds + CW * F::stride;
    const int out_n = (int)A.out_n, off = (int)A.out_off;
    const int wrap = off + M - (int)A.M02;  // window output k is transform output (k + wrap) mod M
    const int ngroups = (out_n + CW - 1) / CW;
    for (int i = (int)threadIdx.x; i < F::tw; i += kPfThreads) tw[i] = A.tw[i];
    float2 v[16];
    float cu_next = 0.0f;
    // the item's column loads: thread t reads rows j + r M/16 of column lc; a
    // column past the window (the last group only) and rows that were not
    // written read zeros through the buffer bound, no branch
    auto column = [](int t) { return t % F::cpb + 4 * (t / F::tpb); };
    auto first = [](int t) { return t % F::tpb / F::cpb; };  // j
    auto load = [&](int item) {
        const int t = (int)threadIdx.x, lc = column(t), j = first(t);
        const int p = item / ngroups, x = item - p * ngroups;
        const int c0 = (int)column_group((unsigned)x, (unsigned)ngroups) * CW;
        // a buffer over the written rows of the wave's block of four columns:
        // a row before them wraps to one far past them
        const int blk = (c0 >> 2) + __builtin_amdgcn_readfirstlane(t / F::tpb);
        const GrBuf zb = gr_buf(A.z + (long)p * M * gr_z_cols(out_n) + ((long)blk * M + A.row_lo) * 4,
                                (unsigned)((A.row_hi - A.row_lo) * 4 * sizeof(float2)));
        // (a column past the window: past the buffer, whatever is added below)
        const unsigned o0 = c0 + lc < out_n ? (unsigned)(((j - A.row_lo) * 4 + (c0 + lc) % 4) * (int)sizeof(float2))
                                            : 0x80000000u;
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = gr_buf_ld2(zb, o0 + (unsigned)(r * NT * 4 * sizeof(float2)));
        const int grp = t / NT;
        cu_next = A.winv[off + (c0 + grp < out_n ? c0 + grp : out_n - 1)];
    };
    int item = (int)blockIdx.x;
    if (item < n_items) load(item);
    __syncthreads();  // twiddles in place
    while (item < n_items) {  // the same trip count in every thread of the block
        // thread indices recomputed from an opaque copy each iteration: held
        // from outside the loop, their derived addresses would not fit the
        // 128 registers of a 1024-thread workgroup
        int t = (int)threadIdx.x;
        asm volatile("" : "+v"(t));
        pf_first(lds + column(t) * F::stride, v, first(t));
        const int cur = item;
        const float cu = cu_next;
        item += (int)gridDim.x;
        __syncthreads();
        if (item < n_items) load(item);
        const int grp = t / NT, tid = t % NT;
        const int p = cur / ngroups, x = cur - p * ngroups;
        const long jj = (long)column_group((unsigned)x, (unsigned)ngroups) * CW + grp;
        const long s1 = 2L * (A.pair0 + p), s2 = s1 + 1;
        const bool live = jj < out_n;
        float *r1 = live ? A.out + s1 * A.out_slice_stride + jj * A.out_row_stride : nullptr;
        float *r2 = live && s2 < A.n_slices ? A.out + s2 * A.out_slice_stride + jj * A.out_row_stride : nullptr;
        float2 *col = lds + grp * F::stride;
        pf_rest<LM>(col, tw, tid);
        // image row jj: outputs kk = tid + r M/16, eight at a time
        auto store = [&](int k0) {
            float wk[8];
            float2 o[8], w2[8];
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const int kk = k0 + tid + r * NT, i = (kk + wrap) & (M - 1);
                wk[r] = A.winv[off + min(kk, out_n - 1)];
                if (F::last2) w2[r] = A.tw[F::tw + (i & (M / 2 - 1))];
                else o[r] = col[gr_lds_idx(i)];
            }
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const int kk = k0 + tid + r * NT;
                if (F::last2) o[r] = gr_last2(col, M, (kk + wrap) & (M - 1), w2[r]);
                if (r1 && kk < out_n) {
                    const float corrn = cu * wk[r];  // grid.cpp:401
                    r1[kk] = corrn * o[r].x;
                    if (r2) r2[kk] = corrn * o[r].y;
                }
            }
        };
        store(0);  // all of a window of up to M/2
        for (int k0 = 8 * NT; k0 < out_n; k0 += 8 * NT) store(k0);
        __syncthreads();  // the columns are free for the next item's first pass
    }
}

// Rows: an item is CW neighbouring rows b0 .. of Ht (row_lo, a multiple of CW,
// on), one per group of M/16 threads; inactive tiles read zeros.  The epilogue
// writes Z column-blocked: 4 CW consecutive lanes store the rows' four columns
// of one column block, CW * 32 contiguous bytes.
template <int LM>
__global__ void __launch_bounds__(kPfThreads) k_ifft_rows_pf(RowsArgs A, int n_items) {
    using F = Pf<LM>;
    constexpr int M = F::M, CW = F::CW, NT = F::nthr;
    extern __shared__ float2 lds[];
    float2 *tw = lds + CW * F::stride;
    const int out_n = (int)A.out_n, wrap = (int)A.out_off + M - (int)A.M02;  // as k_ifft_cols_pf
    const int groups = (A.row_hi - A.row_lo) / CW;  // items per pair
    for (int i = (int)threadIdx.x; i < F::tw; i += kPfThreads) tw[i] = A.tw[i];
    float2 v[16];
    // the active-tile interval of the thread's row (up to eight rows: the
    // item's, one scalar load), fetched an item ahead:
    // waited for only where the loads issued before it are waited for anyway
    auto interval = [&](int item, int t) {
        const int p = item / groups;
        return item < n_items ? A.row_tiles[(A.row_lo + (item - p * groups) * CW + (CW > 8 ? t / NT : 0)) >> 3] : make_int2(1, 0);
    };
    auto load = [&](int item, int2 lh, int t) {  // t: threadIdx.x (an opaque copy inside the loop)
        // a buffer over the active tiles of the wave's row: everything outside
        // (an index before them wraps to one far past them) reads zeros
        const int grp = __builtin_amdgcn_readfirstlane(t / NT), tid = t % NT;
        const int lo = __builtin_amdgcn_readfirstlane(lh.x), hi = __builtin_amdgcn_readfirstlane(lh.y);
        const int p = item / groups, b = A.row_lo + (item - p * groups) * CW + grp;
        const GrBuf hb = gr_buf(A.ht + ((long)p * M + b) * M + 8 * lo, (unsigned)(max(hi - lo + 1, 0) * 8 * sizeof(float2)));
        const unsigned o0 = (unsigned)((tid - 8 * lo) * (int)sizeof(float2));
#pragma unroll
        for (int r = 0; r < 16; r++) v[r] = gr_buf_ld2(hb, o0 + (unsigned)(r * NT * sizeof(float2)));
    };
    int item = (int)blockIdx.x;
    if (item < n_items) load(item, interval(item, (int)threadIdx.x), (int)threadIdx.x);
    int2 lh_next = interval(item + (int)gridDim.x, (int)threadIdx.x);
    __syncthreads();  // twiddles in place
    while (item < n_items) {  // the same trip count in every thread of the block
        int t = (int)threadIdx.x;
        asm volatile("" : "+v"(t));  // indices recomputed per item (as k_ifft_cols_pf)
        const int grp = t / NT, tid = t % NT;
        float2 *row = lds + grp * F::stride;
        pf_first(row, v, tid);
        const int cur = item;
        item += (int)gridDim.x;
        __syncthreads();
        if (item < n_items) {
            load(item, lh_next, t);
            lh_next = interval(item + (int)gridDim.x, t);
        }
        pf_rest<LM>(row, tw, tid);
        const int p = cur / groups, b0 = A.row_lo + (cur - p * groups) * CW;
        float2 *zp = A.z + (long)p * M * gr_z_cols(out_n);
        const int n_out = CW * (int)gr_z_cols(out_n);
        auto store = [&](int L0) {
            float2 o[8], w2[8];
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const int L = L0 + t + r * kPfThreads, rr = (L >> 2) % CW, jj = 4 * (L / (4 * CW)) + (L & 3);
                const int i = (jj + wrap) & (M - 1);
                if (F::last2) w2[r] = A.tw[F::tw + (i & (M / 2 - 1))];
                else o[r] = lds[rr * F::stride + gr_lds_idx(i)];
            }
#pragma unroll
            for (int r = 0; r < 8; r++) {
                const int L = L0 + t + r * kPfThreads, blk = L / (4 * CW), rr = (L >> 2) % CW, c = L & 3;
                const int jj = 4 * blk + c;
                if (jj < out_n) {
                    if (F::last2) o[r] = gr_last2(lds + rr * F::stride, M, (jj + wrap) & (M - 1), w2[r]);
                    zp[((long)blk * M + b0 + rr) * 4 + c] = o[r];
                }
            }
        };
        store(0);  // all of a window of up to M/2
        for (int L0 = 8 * kPfThreads; L0 < n_out; L0 += 8 * kPfThreads) store(L0);
        __syncthreads();  // the rows are free for the next item's first pass
    }
}

inline int maxb_of(long N, int nthr) { return (int)((N / 4 + nthr - 1) / nthr); }

__global__ void k_row_tiles(int2 *out, int ntr, float M2, float rmax) {
    const int ty = blockIdx.x * blockDim.x + threadIdx.x;
    if (ty >= ntr) return;
    int lo, hi;
    gr_active_tile_range(ty, ntr, M2, rmax, lo, hi);
    out[ty] = make_int2(lo, hi);
}

}  // namespace

// A figure of the current device, queried once per device (0 when the query
// fails).
static int device_attr(hipDeviceAttribute_t attr, std::atomic<int> (&cache)[64]) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0;
    int v = cache[dev].load(std::memory_order_relaxed);
    if (v == 0) {
        if (hipDeviceGetAttribute(&v, attr, dev) != hipSuccess || v <= 0) v = -1;
        cache[dev].store(v, std::memory_order_relaxed);
    }
    return v > 0 ? v : 0;
}

int gr_cu_count() {
    static std::atomic<int> cache[64];
    return device_attr(hipDeviceAttributeMultiprocessorCount, cache);
}

int gr_max_lds_per_block() {
    static std::atomic<int> optin[64], plain[64];
    return std::max(device_attr(hipDeviceAttributeSharedMemPerBlockOptin, optin),
                    device_attr(hipDeviceAttributeMaxSharedMemoryPerBlock, plain));
}

// Whether a launch of n_items items takes the persistent form: with fewer than
// two per CU there is nothing to overlap and the one-shot kernels' smaller
// workgroups fill the chip better -- but at M = 4096, where they take a CU each,
// too (columns of a pair of 60 x 2000, 500 items: 28.9 us persistent, 41.2
// one-shot).
static bool pf_takes(long M, int radix, long n_items) {
    const int cus = gr_cu_count();
    return M >= 1024 && M <= 8192 && radix == 16 && cus > 0 && (M == 4096 || n_items >= 2L * cus) &&
           (size_t)gr_max_lds_per_block() >= std::max(Pf<12>::lds, Pf<13>::lds);
}

template <template <int> class Launch, class... Args>
static hipError_t pf_launch(long M, Args... args) {
    switch (M) {
    case 1024: return Launch<10>::go(args...);
    case 2048: return Launch<11>::go(args...);
    case 4096: return Launch<12>::go(args...);
    default: return Launch<13>::go(args...);
    }
}
template <int LM>
struct PfRows {
    static hipError_t go(RowsArgs A, int pairs, hipStream_t s) {
        const int n_items = (A.row_hi - A.row_lo) / Pf<LM>::CW * pairs;
        const hipError_t e = gr_allow_lds(k_ifft_rows_pf<LM>, Pf<LM>::lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_ifft_rows_pf<LM>, dim3(std::min(n_items, gr_cu_count())), dim3(kPfThreads), Pf<LM>::lds, s,
                           A, n_items);
        return hipGetLastError();
    }
};
template <int LM>
struct PfCols {
    static hipError_t go(ColsArgs A, int pairs, hipStream_t s) {
        const int n_items = (int)((A.out_n + Pf<LM>::CW - 1) / Pf<LM>::CW) * pairs;
        const hipError_t e = gr_allow_lds(k_ifft_cols_pf<LM>, Pf<LM>::lds);
        if (e != hipSuccess) return e;
        hipLaunchKernelGGL(k_ifft_cols_pf<LM>, dim3(std::min(n_items, gr_cu_count())), dim3(kPfThreads), Pf<LM>::lds, s,
                           A, n_items);
        return hipGetLastError();
    }
};

hipError_t gr_launch_row_tiles(const GrGeom &g, int2 *out, hipStream_t s) {
    const int ntr = (int)(g.M >> 3);
    hipLaunchKernelGGL(k_row_tiles, dim3((ntr + 255) / 256), dim3(256), 0, s, out, ntr, (float)(g.M >> 1),
                       gr_grid_rmax(g));
    return hipGetLastError();
}

// Rows of Ht per workgroup of the row transform: one (at M = 4096 on MI355X
// 0.57 ms per launch of 8 pairs, 0.59 with 2 side by side, 0.67 with 4).
constexpr int kRowsPerBlock = 1;

hipError_t gr_launch_ifft_rows(const GrGeom &g, const GrDevTables &t, const float2 *ht, float2 *z,
                               int pairs, hipStream_t s) {
    RowsArgs A{ht, z, t.tw_grid, t.row_tiles, (int)g.M, g.fft_radix, g.M02, g.out_off, g.out_n,
               t.row_lo, t.row_hi};
    const int nthr = gr_fft_threads(g.M);
    const long pf_cw = 16384 / g.M;
    if (g.M <= 16384) {
        RowsArgs B = A;  // whole items: the rows added hold no active tile and read as zeros
        B.row_lo = (int)(t.row_lo / std::max(pf_cw, 1L) * pf_cw);
        B.row_hi = (int)((t.row_hi + pf_cw - 1) / std::max(pf_cw, 1L) * pf_cw);
        if (pf_takes(g.M, g.fft_radix, (B.row_hi - B.row_lo) / std::max(pf_cw, 1L) * pairs))
            return pf_launch<PfRows>(g.M, B, pairs, s);
    }
    int cw = kRowsPerBlock;  // rows side by side: a power of two dividing M, within 1024 threads and the LDS
    while (cw > 1 && ((long)cw * nthr > 1024 || (long)cw * g.M * 8 > 163840 || g.M % cw)) cw /= 2;
    // whole groups of 32 rows, which row_group deals out (the rows added hold no
    // active tile and read as zeros): with any other number the pieces of
    // a line of Z come from several XCDs (4 pairs of 900 x 1000 28 -> 31 us)
    A.row_lo = t.row_lo / 32 * 32;
    A.row_hi = (int)std::min<long>((t.row_hi + 31) / 32 * 32, g.M);
    const dim3 grid((unsigned)((A.row_hi - A.row_lo) / cw), pairs), block(cw * nthr);
    const size_t lds = sizeof(float2) * cw * gr_lds_len(g.M);
#define GR_ROWS_K(MB, CW)                                                          \
    do {                                                                           \
        hipError_t e_ = gr_allow_lds(k_ifft_rows<MB, CW>, lds);                    \
        if (e_ != hipSuccess) return e_;                                           \
        hipLaunchKernelGGL((k_ifft_rows<MB, CW>), grid, block, lds, s, A);         \
    } while (0)
#define GR_ROWS(MB)                                                                \
    do {                                                                           \
        if (cw == 4) GR_ROWS_K(MB, 4);                                             \
        else if (cw == 2) GR_ROWS_K(MB, 2);                                        \
        else GR_ROWS_K(MB, 1);                                                     \
    } while (0)
    switch (maxb_of(g.M, nthr)) {
    case 0:
    case 1: GR_ROWS(1); break;
    case 2: GR_ROWS(2); break;
    case 4: GR_ROWS(4); break;
    case 8: GR_ROWS(8); break;
    case 16: GR_ROWS(16); break;
    default: return hipErrorInvalidValue;
    }
#undef GR_ROWS
#undef GR_ROWS_K
    return hipGetLastError();
}

// Columns per workgroup.  Side by side (CW > 0) while CW FFT thread groups
// fit a workgroup (<= 1024 threads) and CW columns fit the CU's LDS (160 KiB);
// beyond that, one after another on all threads while cw * M <= 16384.  The
// default is the widest of 4, 2, 1 side by side that fits: the column gathers
// bound the kernel and a line then serves that many columns (at M = 4096 on
// MI355X: 0.57 ms per launch of 8 pairs with 1, 0.50 with 2, 0.48 with 4).
// Callers may ask for a width (gr_plan.cols_per_block).

static bool cols_side_by_side(long M, int cw) {
    return cw >= 1 && cw <= 8 && (cw & (cw - 1)) == 0 && (long)cw * gr_fft_threads(M) <= 1024 &&
           (long)cw * M * 8 <= 163840;
}

bool gr_cols_width_ok(long M, int cols) {
    return cols_side_by_side(M, cols) || (cols >= 1 && (long)cols * M <= 16384);
}

static int cols_per_block(long M, long out_n, int pairs) {
    (void)out_n;
    (void)pairs;
    return cols_side_by_side(M, 4) ? 4 : cols_side_by_side(M, 2) ? 2 : 1;
}

hipError_t gr_launch_ifft_cols(const GrGeom &g, const GrDevTables &t, const float2 *z, float *out,
                               long out_slice_stride, long out_row_stride, int n_slices, int pair0,
                               int pairs, int cols, hipStream_t s) {
    ColsArgs A;
    A.z = z;
    A.out = out;
    A.tw = t.tw_grid;
    A.winv = t.winv;
    A.out_slice_stride = out_slice_stride;
    A.out_row_stride = out_row_stride;
    A.M = (int)g.M;
    A.cw = cols > 0 && gr_cols_width_ok(g.M, cols) ? cols : cols_per_block(g.M, g.out_n, pairs);
    A.n_slices = n_slices;
    A.pair0 = pair0;
    A.radix = g.fft_radix;
    A.M02 = g.M02;
    A.out_off = g.out_off;
    A.out_n = g.out_n;
    A.row_lo = t.row_lo;
    A.row_hi = t.row_hi;
    const int nthr = gr_fft_threads(g.M);
    const bool side = cols_side_by_side(g.M, A.cw);
    // at M = 4096 the persistent form is the width of four columns, too
    if ((cols == 0 || (g.M == 4096 && A.cw == 4)) &&
        pf_takes(g.M, g.fft_radix, (g.out_n + 16384 / g.M - 1) / (16384 / g.M) * pairs))
        return pf_launch<PfCols>(g.M, A, pairs, s);
    const dim3 grid((unsigned)((g.out_n + A.cw - 1) / A.cw), pairs), block(side ? A.cw * nthr : nthr);
    const size_t lds = sizeof(float2) * A.cw * gr_lds_len(g.M);
#define GR_COLS_K(MB, CW)                                                                \
    do {                                                                                 \
        hipError_t e_ = gr_allow_lds(k_ifft_cols<MB, CW>, lds);                          \
        if (e_ != hipSuccess) return e_;                                                 \
        hipLaunchKernelGGL((k_ifft_cols<MB, CW>), grid, block, lds, s, A);               \
    } while (0)
#define GR_COLS(MB)                                                                      \
    do {                                                                                 \
        if (!side) GR_COLS_K(MB, 0);                                                     \
        else if (A.cw == 1) GR_COLS_K(MB, 1);                                            \
        else if (A.cw == 2) GR_COLS_K(MB, 2);                                            \
        else if (A.cw == 4) GR_COLS_K(MB, 4);                                            \
        else if (A.cw == 8) GR_COLS_K(MB, 8);                                            \
        else GR_COLS_K(MB, 0);                                                           \
    } while (0)
    switch (maxb_of(g.M, nthr)) {
    case 0:
    case 1: { GR_COLS(1); } break;
    case 2: { GR_COLS(2); } break;
    case 4: { GR_COLS(4); } break;
    case 8: { GR_COLS(8); } break;
    case 16: { GR_COLS(16); } break;
    default: return hipErrorInvalidValue;
    }
#undef GR_COLS_K
#undef GR_COLS
    return hipGetLastError();
}
