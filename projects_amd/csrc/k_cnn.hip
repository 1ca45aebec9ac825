// k_cnn.hip -- the sparse-angle residual CNN: forward, backward and Adam.
//
// Network (no counterpart in the reference; it corrects gridrec's streaks on
// sparse-angle scans): five 3x3 convolutions 1 -> 32 -> 32 -> 32 -> 32 -> 1,
// ReLU after the first four, y = x/scale + conv5(a4) + b5.  BF16 weights and
// activations, FP32 accumulation, MSE loss, Adam on FP32 master weights.
//
// Layouts: images [n][H][W] f32; activations and their gradients [n][H][W][32]
// bf16 (channels last: one pixel is one 64-byte record); parameters one flat
// f32 vector W1[32][9] b1[32] W2[32][32][9] b2 W3 b3 W4 b4 W5[32][9] b5[1]
// (taps ky*3+kx, correlation, zero padding).
//
// The three 32 -> 32 layers run on MFMA (v_mfma_f32_16x16x32_bf16): a block
// owns a tile of pixels; its input with a one-pixel halo is staged in
// LDS.  Forward: D[co][pixel] = W_t[co][ci] x X_t[ci][pixel] summed over the 9
// taps; each lane keeps its weight fragments (2 x 9 x 8 bf16) in registers for
// the whole block.  The input gradient is the same with the taps flipped and
// the channel roles swapped (packed by k_pack), the ReLU mask of the layer
// input in its epilogue.  The weight gradient is D[co][ci] = dZ[co][pixel] x
// A_t[pixel][ci] with K running over the pixels of a tile row, the operands
// read transposed from LDS.  Blocks loop over tiles and write per-block partial
// sums that k_reduce adds in a fixed order: results are bitwise repeatable.
//
// The 1 -> 32 and 32 -> 1 layers run on MFMA as well: K over the 9 taps of
// the single input channel, and W5 in row 0 of A.
#include <math.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>
#include <utility>

#include "gr_fft.hpp"
#include "gr_internal.h"
#include "../../include/gridrec_cnn.h"

#pragma clang fp contract(off)

int gr_set_error(int code, const char *msg);

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));

constexpr int CH = 32;
constexpr int TH = 8, TW = 32;            // output tile (rows x columns)
constexpr int HS = TH + 2, WS = TW + 2;   // with the halo
constexpr int OFF_W1 = 0, OFF_B1 = 288, OFF_W2 = 320, OFF_B2 = OFF_W2 + 9216, OFF_W3 = OFF_B2 + 32,
              OFF_B3 = OFF_W3 + 9216, OFF_W4 = OFF_B3 + 32, OFF_B4 = OFF_W4 + 9216, OFF_W5 = OFF_B4 + 32,
              OFF_B5 = OFF_W5 + 288, N_PARAMS = OFF_B5 + 1;
constexpr int PACK_LAYER = 2 * 9 * CH * CH;  // forward + flipped, bf16, per 32->32 layer
constexpr int WG_REC = 9 * CH * CH + CH;     // weight-gradient partial record of a 32->32 layer
constexpr int IN_REC = 9 * CH + CH;          // of the 1->32 layer
constexpr int OUT_REC = 9 * CH + 1;          // of the 32->1 layer
constexpr int MAX_WG_BLOCKS = 512;

static_assert(N_PARAMS == 28353, "parameter layout");

__device__ __forceinline__ uint16_t to_bf16(float f) {
    // round to nearest, ties to even: one v_cvt_pk_bf16_f32 (for two values)
    // instead of four integer operations per value.  On every non-NaN float
    // it equals the integer rounding (u + 0x7FFF + ((u >> 16) & 1)) >> 16 of
    // the bit pattern u, the oracle's (checked over all 2^32 patterns on
    // MI355X: no difference).
    return __builtin_bit_cast(uint16_t, (__bf16)f);
}
// Two of them in one word, the first in its low half.
__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2{lo, hi}), bf16x2));
}
__device__ __forceinline__ float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ float round_bf16(float f) { return from_bf16(to_bf16(f)); }
__device__ __forceinline__ bool positive_bf16(uint16_t h) { return !(h & 0x8000u) && h != 0; }

__device__ __forceinline__ __bf16 bf16_of(float f) { return __builtin_bit_cast(__bf16, to_bf16(f)); }

// The 1 -> 32 and 32 -> 1 layers on MFMA too (v_mfma_f32_16x16x32_bf16, the
// lane layout of the 32 -> 32 layers: A row = lane & 15, B column = lane & 15,
// k = 8 * (lane >> 4) + e; D column = lane & 15, rows 4 * (lane >> 4) + e).
//
// 1 -> 32: K runs over the 9 taps (k >= 9 zero), so one MFMA per 16 output
// channels gives D[co][pixel] = sum_t W1[co][t] x(pixel + t).  w1 holds the
// bf16 values of W1 as floats, [co * 9 + t].
__device__ __forceinline__ void conv_in_frag(const float *w1, int lane, bf16x8 (&A)[2]) {
#pragma unroll
    for (int nb = 0; nb < 2; nb++)
#pragma unroll
        for (int e = 0; e < 8; e++) {
            const int k = 8 * (lane >> 4) + e;
            A[nb][e] = bf16_of(k < 9 ? w1[(nb * 16 + (lane & 15)) * 9 + k] : 0.0f);
        }
}

// 32 -> 1: nine MFMAs (one per tap, K over the 32 input channels) with W5 in
// row 0 of A and zeros in rows 1..15; the result D[0][pixel] sits in element 0
// of lanes 0..15.  w5 holds the bf16 values of W5 as floats, [ci * 9 + t].
__device__ __forceinline__ void conv_out_frag(const float *w5, int lane, bf16x8 (&A)[9]) {
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int e = 0; e < 8; e++)
            A[t][e] = bf16_of((lane & 15) == 0 ? w5[(8 * (lane >> 4) + e) * 9 + t] : 0.0f);
}

struct TileMap {
    int tiles_x, tiles_y;
    __device__ void of(int tile, int &img, int &y0, int &x0) const { of_rows(tile, TH, img, y0, x0); }
    // tiles of th rows (tiles_y counts them)
    __device__ void of_rows(int tile, int th, int &img, int &y0, int &x0) const {
        const int per = tiles_x * tiles_y;
        img = tile / per;
        const int r = tile - img * per;
        y0 = (r / tiles_x) * th;
        x0 = (r % tiles_x) * TW;
    }
};

// ---------------------------------------------------------------------------
// The whole forward pass in one kernel.  A workgroup walks down a strip of 56
// output columns, two image rows a step, all five layers at once: in step s
// layer 1 computes rows 2s, 2s + 1 of a1, layer 2 rows 2s - 3 .. of a2, layer 3
// rows 2s - 6, layer 4 rows 2s - 9, and layer 5 rows 2s - 12 of the output, each
// from rows that earlier steps left in LDS: rings of six rows per activation,
// one barrier per step.  So a pixel's activations never come back from HBM
// (layer by layer they went out and in at 64 bytes per pixel and layer), rows
// are computed once and columns 64 / 56 times; a training pass writes them as
// they are made, inference writes none.
//
// Columns: 64 in every layer, of which layer l is right in columns l - 1 ..
// 64 - l (columns depend on their neighbours only); LDS rows hold 66, so every
// read stays inside.  Pixels outside the image are zero, the padding of the
// next layer.  Twelve waves, one workgroup per CU: wave w holds the weights of
// layer 2 + w / 4 in registers and takes columns 16 (w mod 4) .., so each SIMD
// has a wave of each layer; the waves of layer 2 also compute layer 1, those of
// layer 3 layer 5 (its weights in LDS), those of layer 4 bring x.  A fragment of
// an input row serves the output rows of all its taps in the wave's two rows,
// and in the next step's.  LDS records as in k_conv32_back, piece s of a pixel in
// slot s ^ (column / 4 mod 4).
//
// Per output the MFMAs run tap by tap into one accumulator, then bias, ReLU
// and rounding, whichever buffers are written.  Bound by MFMA (130 per step and
// SIMD, half of the time) and what a barrier per step leaves exposed around
// them: 4 x 2048^2 inference 0.96 ms where five layer kernels took 1.93, of
// which 6.4 GB of activations 1.36 at the rate of a copy; 32 x 512^2 training
// 0.87 ms (2.2 GB written) against 1.02.
constexpr int FW_COLS = 64, FW_OUT = 56, FW_RING = 6, FW_PITCH = FW_COLS + 2;
constexpr int FW_ROW = FW_PITCH * 64, FW_BUF = FW_RING * FW_ROW;  // bytes of a ring's row, of a ring
constexpr int FW_XP = 68;                                        // floats per x row
constexpr int FW_THREADS = 768;
constexpr size_t FW_LDS = 4 * (size_t)FW_BUF + 9 * 1024 + sizeof(float) * (FW_RING * FW_XP + 4 * CH);

struct FwdArgs {
    const float *x, *prm;
    const uint16_t *packed;
    uint16_t *act[4];  // a1 .. a4, null: not written
    float *y, *yn, *stats;
    float scale;
    int H, W, strips, segs, seg_rows;
};

// relu(acc + bias) of four channels as bf16 (NaN gives zero, as z > 0 ? z : 0).
__device__ __forceinline__ uint2 act_of(floatx4 a, float4 b) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const float v[4] = {fmaxf(a[0] + b.x, 0.0f), fmaxf(a[1] + b.y, 0.0f), fmaxf(a[2] + b.z, 0.0f),
                        fmaxf(a[3] + b.w, 0.0f)};
    const bf16x2 lo = {(__bf16)v[0], (__bf16)v[1]}, hi = {(__bf16)v[2], (__bf16)v[3]};
    return make_uint2(__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi));
}

__global__ void __launch_bounds__(FW_THREADS) k_forward(FwdArgs P) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    bf16x8 *w5 = reinterpret_cast<bf16x8 *>(smem_raw + 4 * FW_BUF);  // layer 5's weight fragments, [tap][lane]
    float *xr = reinterpret_cast<float *>(w5 + 9 * 64);              // ring of six rows of bf16(x / scale)
    float *sb = xr + FW_RING * FW_XP;                              // b1 .. b4
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, g = lane >> 4, q = wave & 3, c = 16 * q + j;
    const int H = P.H, W = P.W, per = P.strips * P.segs;
    const int img = (int)blockIdx.x / per, ws = (int)blockIdx.x - img * per;
    const int X0 = (ws % P.strips) * FW_OUT - 4, Y0 = (ws / P.strips) * P.seg_rows;
    const int rows = min(P.seg_rows, H - Y0), top = Y0 - 4;  // relative row r is image row top + r
    const long ibase = (long)img * H * W;
    const int gx = X0 + c;
    const bool col_in = (unsigned)gx < (unsigned)W, col_out = col_in && c >= 4 && c < 4 + FW_OUT;

    const float *xim = P.x + ibase;
    // x rows r, r + 1 (relative), columns -1 .. 64, by the 256 threads of layer
    // 4's waves; loads are clamped into the image and their values dropped
    // where they are used (a load inside a branch is waited for there)
    const int xt = tid - 512, xi = xt >= FW_PITCH ? 1 : 0, xc = xt - xi * FW_PITCH, xgx = X0 + xc - 1;
    const int xcl = min(max(xgx, 0), W - 1);
    auto row_of = [&](int r) { return (long)min(max(top + r, 0), H - 1) * W; };  // uniform
    auto load_x = [&](int r) {
        const long r0 = row_of(r);
        const int d = (int)(row_of(r + 1) - r0);
        return (xim + r0)[xcl + (xi ? d : 0)];
    };
    auto put_x = [&](int r, int slot, float v) {
        const bool in = (unsigned)xgx < (unsigned)W && (unsigned)(top + r + xi) < (unsigned)H;
        if (xt >= 0 && xt < 2 * FW_PITCH) xr[slot * FW_XP + xc] = in ? round_bf16(v / P.scale) : 0.0f;
    };
    put_x(-1, xi ? 0 : 5, load_x(-1));
    put_x(1, xi ? 2 : 1, load_x(1));
    float x_next = load_x(3);
    if (tid < 4 * CH) {
        const int l = tid >> 5, off[4] = {OFF_B1, OFF_B2, OFF_B3, OFF_B4};
        sb[tid] = P.prm[off[l] + (tid & 31)];
    }
    if (wave == 4) {
        bf16x8 A5[9];
        conv_out_frag(P.prm + OFF_W5, lane, A5);
#pragma unroll
        for (int t = 0; t < 9; t++) w5[t * 64 + lane] = A5[t];
    }
    auto slot = [](int col, int piece) { return col * 64 + ((piece ^ (col >> 2)) & 3) * 16; };
    // the wave's layer l + 2 reads ring l and writes ring l + 1
    const int l = wave >> 2;
    const unsigned char *o_b[3];  // input fragments at column c + kx - 1
    int o_w[2];                   // the lane's output channels
#pragma unroll
    for (int k = 0; k < 3; k++) o_b[k] = smem_raw + l * FW_BUF + slot(c + k, g);
#pragma unroll
    for (int n = 0; n < 2; n++) o_w[n] = slot(c + 1, 2 * n + (g >> 1)) + 8 * (g & 1);
    const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    const int last = (rows + 15) / 2;  // step of the last output row
    // activation row r of the lane's pixel and channels into slot rs of ring
    // k and, where the caller keeps it, to dst
    auto put = [&](int k, int r, int rs, uint16_t *dst, floatx4 v0, floatx4 v1, float4 b0, float4 b1) {
        uint2 h0 = act_of(v0, b0), h1 = act_of(v1, b1);
        const unsigned m = col_in && (unsigned)(top + r) < (unsigned)H ? ~0u : 0u;  // zeros outside the image
        h0 = make_uint2(h0.x & m, h0.y & m);
        h1 = make_uint2(h1.x & m, h1.y & m);
        unsigned char *ring = smem_raw + k * FW_BUF + rs * FW_ROW;
        *reinterpret_cast<uint2 *>(ring + o_w[0]) = h0;
        *reinterpret_cast<uint2 *>(ring + o_w[1]) = h1;
        if (P.act[k] && r >= 4 && r < rows + 4 && col_out) {
            *reinterpret_cast<uint2 *>(dst) = h0;
            *reinterpret_cast<uint2 *>(dst + 16) = h1;
        }
    };
    // the lane's place in row r of a kept activation
    auto place = [&](int k, int r) {
        return P.act[k] ? P.act[k] + (ibase + (long)(top + r) * W + gx) * CH + 4 * g : nullptr;
    };
    const uint16_t *wp = P.packed + (long)l * PACK_LAYER;
    bf16x8 A[2][9];
#pragma unroll
    for (int n = 0; n < 2; n++)
#pragma unroll
        for (int t = 0; t < 9; t++)
            A[n][t] = *reinterpret_cast<const bf16x8 *>(wp + ((t * CH + n * 16 + j) * CH + 8 * g));
    __syncthreads();

    // Layer l + 2's step: rows 2s - 3 (l + 1) and the next.  Ring k's row r sits
    // in slot (r + 3 (k + 1)) mod 6, so with 2s mod 6 = M2 every layer reads
    // slots M2 - 1 .. M2 + 2 and writes M2 + 3, M2 + 4: constants, the steps
    // going by threes.  The upper two input rows are the lower two of the step
    // before, kept in registers (Bk): their MFMAs start at once while the others
    // arrive.
    const int lag = 3 * (l + 1);
    const float *bias = sb + (l + 1) * CH + 4 * g;
    const bool act_kept = P.act[l + 1] != nullptr;
    uint16_t *act = place(l + 1, -lag);
    bf16x8 Bk[2][3];
#pragma unroll
    for (int hr = 0; hr < 2; hr++)
#pragma unroll
        for (int kx = 0; kx < 3; kx++) Bk[hr][kx] = bf16x8{};
    auto conv = [&](auto m2, int s) {
        constexpr int M2 = decltype(m2)::value;
        const int r = 2 * s - lag;
        bf16x8 Bn[2][3];
#pragma unroll
        for (int hr = 0; hr < 2; hr++)
#pragma unroll
            for (int kx = 0; kx < 3; kx++)
                Bn[hr][kx] = *reinterpret_cast<const bf16x8 *>(o_b[kx] + (M2 + 7 + hr) % 6 * FW_ROW);
        floatx4 acc[2][2] = {{zero, zero}, {zero, zero}};
#pragma unroll
        for (int hr = 0; hr < 4; hr++)
#pragma unroll
            for (int kx = 0; kx < 3; kx++) {
                const bf16x8 B = hr < 2 ? Bk[hr][kx] : Bn[hr - 2][kx];
#pragma unroll
                for (int i = 0; i < 2; i++) {
                    const int ky = hr - i;
                    if (ky < 0 || ky > 2) continue;
                    acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[0][ky * 3 + kx], B, acc[i][0], 0, 0, 0);
                    acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[1][ky * 3 + kx], B, acc[i][1], 0, 0, 0);
                }
            }
        const float4 b0 = *reinterpret_cast<const float4 *>(bias), b1 = *reinterpret_cast<const float4 *>(bias + 16);
        put(l + 1, r, (M2 + 3) % 6, act, acc[0][0], acc[0][1], b0, b1);
        put(l + 1, r + 1, (M2 + 4) % 6, act + (long)W * CH, acc[1][0], acc[1][1], b0, b1);
        if (act_kept) act += 2L * W * CH;
#pragma unroll
        for (int hr = 0; hr < 2; hr++)
#pragma unroll
            for (int kx = 0; kx < 3; kx++) Bk[hr][kx] = Bn[hr][kx];
    };
    auto run = [&](auto &&step) {
        for (int s = 0; s <= last; s += 3) {
            step(std::integral_constant<int, 0>{}, s);
            __syncthreads();
            if (s + 1 > last) break;
            step(std::integral_constant<int, 2>{}, s + 1);
            __syncthreads();
            if (s + 2 > last) break;
            step(std::integral_constant<int, 4>{}, s + 2);
            __syncthreads();
        }
    };
    // the longest chain of a step first: layer 3's wave of each SIMD has half as
    // many MFMAs again (1105 -> 1050 us at 4 x 2048^2)
    if (l == 1) __builtin_amdgcn_s_setprio(2);
    else if (l == 0) __builtin_amdgcn_s_setprio(1);
    if (l == 0) {  // and layer 1
        bf16x8 A1[2];
        conv_in_frag(P.prm + OFF_W1, lane, A1);
        // its taps 0 .. 7 in lanes 0 .. 15, tap 8 in lanes 16 .. 31
        const unsigned use0 = g < 2 ? ~0u : 0u, use = g == 0 ? ~0u : 0u;
        const float *xl = xr + c, *xl0 = xl + (g > 0 ? 2 : 0);  // element 0: tap 0, or tap 8
        uint16_t *act1 = place(0, 0);
        run([&](auto m2, int s) {
            constexpr int M2 = decltype(m2)::value;
            const float4 b0 = *reinterpret_cast<const float4 *>(sb + 4 * g), b1 = *reinterpret_cast<const float4 *>(sb + 16 + 4 * g);
#pragma unroll
            for (int i = 0; i < 2; i++) {
                // row 2s + i - 1 + ky of x in slot (M2 + i + 5 + ky) mod 6
                const int rx[3] = {(M2 + i + 5) % 6 * FW_XP, (M2 + i) % 6 * FW_XP, (M2 + i + 1) % 6 * FW_XP};
                float v[8];
                v[0] = xl0[g > 0 ? rx[2] : rx[0]];
#pragma unroll
                for (int e = 1; e < 8; e++) v[e] = xl[rx[e / 3] + e % 3];
                bf16x8 B;
#pragma unroll
                for (int e = 0; e < 8; e++) B[e] = bf16_of(__uint_as_float(__float_as_uint(v[e]) & (e ? use : use0)));
                const floatx4 v0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A1[0], B, zero, 0, 0, 0);
                const floatx4 v1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A1[1], B, zero, 0, 0, 0);
                put(0, 2 * s + i, (M2 + 3 + i) % 6, act1 + (long)i * W * CH, v0, v1, b0, b1);
            }
            if (P.act[0]) act1 += 2L * W * CH;
            conv(m2, s);
        });
    } else if (l == 2) {  // and x, a step ahead: rows 2s + 3, 2s + 4 into LDS and 2s + 5, 2s + 6 on
                          // their way into the same register (two would meet in a copy that waits)
        run([&](auto m2, int s) {
            constexpr int M2 = decltype(m2)::value;
            put_x(2 * s + 3, xi ? (M2 + 4) % 6 : (M2 + 3) % 6, x_next);
            x_next = load_x(2 * s + 5);
            conv(m2, s);
        });
    } else {  // and layer 5
        const float b5 = P.prm[OFF_B5];
        const bf16x8 *A5 = w5 + lane;
        const unsigned char *in5[3] = {smem_raw + 3 * FW_BUF + slot(c, g), smem_raw + 3 * FW_BUF + slot(c + 1, g),
                                       smem_raw + 3 * FW_BUF + slot(c + 2, g)};
        const int gxc = min(max(gx, 0), W - 1);
        float xv[2] = {0.0f, 0.0f};  // x of rows r, r + 1 (rows -12, -11 are outside), loaded a step ahead
        double r2 = 0.0, x2 = 0.0;   // the lane's sums of residual^2 and (x / scale)^2
        run([&](auto m2, int s) {
            constexpr int M2 = decltype(m2)::value;
            const int r = 2 * s - 12;  // output rows r, r + 1
            floatx4 acc[2] = {zero, zero};
#pragma unroll
            for (int hr = 0; hr < 4; hr++)
#pragma unroll
                for (int kx = 0; kx < 3; kx++) {
                    const bf16x8 B = *reinterpret_cast<const bf16x8 *>(in5[kx] + (M2 + 5 + hr) % 6 * FW_ROW);
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int ky = hr - i;
                        if (ky < 0 || ky > 2) continue;
                        acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A5[(ky * 3 + kx) * 64], B, acc[i], 0, 0, 0);
                    }
                }
#pragma unroll
            for (int i = 0; i < 2; i++)
                if (lane < 16 && col_out && r + i >= 4 && r + i < rows + 4) {
                    const float res = acc[i][0] + b5;
                    const long p = ibase + (long)(top + r + i) * W + gx;
                    const float xn = xv[i] / P.scale;
                    const float v = xn + res;
                    if (P.yn) P.yn[p] = v;
                    if (P.y) P.y[p] = v * P.scale;
                    r2 += (double)(res * res);
                    x2 += (double)(xn * xn);
                }
#pragma unroll
            for (int i = 0; i < 2; i++) xv[i] = (xim + row_of(r + 2 + i))[gxc];
            conv(m2, s);
        });
#pragma unroll
        for (int h = 8; h > 0; h >>= 1) {
            r2 += __shfl_down(r2, h, 64);
            x2 += __shfl_down(x2, h, 64);
        }
        if (lane == 0) {  // the rings are free after the last step
            double *red = reinterpret_cast<double *>(smem_raw);
            red[2 * q] = r2;
            red[2 * q + 1] = x2;
        }
    }
    __syncthreads();
    if (tid < 2 && P.stats) {
        const double *red = reinterpret_cast<const double *>(smem_raw);
        P.stats[2L * blockIdx.x + tid] = (float)(((red[tid] + red[2 + tid]) + red[4 + tid]) + red[6 + tid]);
    }
}

// Layer 5 and the residual alone, from a4: for a forward pass whose y or yn is
// x itself.  k_forward's workgroups read x around their pixels long after others
// have written theirs, so there it stores the activations only, and here every
// lane reads the x of a pixel before it writes that pixel.  A wave takes 16
// columns and OUT_ROWS rows, the fragments of three rows of a4 in registers; the MFMAs
// and the additions of an output are k_forward's: bitwise its values.
constexpr int OUT_ROWS = 16;
__global__ void __launch_bounds__(256) k_conv_out(const uint16_t *__restrict__ a4, const float *x, float scale,
                                                  const float *__restrict__ prm, float *y, float *yn, int H, int W,
                                                  int cols, int segs, long nwaves) {
    const int lane = threadIdx.x & 63, j = lane & 15, g = lane >> 4;
    const long w = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (w >= nwaves) return;
    const long img = w / ((long)cols * segs), ibase = img * H * W;
    const int r = (int)(w - img * cols * segs), y0 = r / cols * OUT_ROWS, gx = r % cols * 16 + j;
    bf16x8 A[9];
    conv_out_frag(prm + OFF_W5, lane, A);
    const float b5 = prm[OFF_B5];
    auto load = [&](int gy, bf16x8 (&B)[3]) {  // row gy at columns gx - 1 .. gx + 1, zero outside the image
#pragma unroll
        for (int k = 0; k < 3; k++) {
            const int cx = gx + k - 1;
            B[k] = bf16x8{};
            if ((unsigned)gy < (unsigned)H && (unsigned)cx < (unsigned)W)
                B[k] = *reinterpret_cast<const bf16x8 *>(a4 + (ibase + (long)gy * W + cx) * CH + 8 * g);
        }
    };
    bf16x8 B[3][3];
    load(y0 - 1, B[0]);
    load(y0, B[1]);
    for (int gy = y0; gy < min(y0 + OUT_ROWS, H); gy++) {
        load(gy + 1, B[2]);
        floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int t = 0; t < 9; t++) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[t], B[t / 3][t % 3], acc, 0, 0, 0);
        if (lane < 16 && gx < W) {
            const long p = ibase + (long)gy * W + gx;
            const float v = x[p] / scale + (acc[0] + b5);
            if (yn) yn[p] = v;
            if (y) y[p] = v * scale;
        }
#pragma unroll
        for (int k = 0; k < 3; k++) {
            B[0][k] = B[1][k];
            B[1][k] = B[2][k];
        }
    }
}

// ---------------------------------------------------------------------------
// Backward of a 32 -> 32 layer in one pass: the input gradient
// dzn = bf16(conv^T(dz) * (a > 0)) and the weight gradient's partial sums, from
// one read of dz (with its halo) and a.  Bound by HBM: dz, a and dzn once each
// (1.7 GB per layer of the 32 x 512^2 batch); as two kernels dz and a came
// twice, and the weight gradient staged four transposed copies by 16-bit LDS
// stores: 734 + 322 us per layer, now 400.
//
// A workgroup of eight waves per CU walks a contiguous range of 16 x 32 pixel
// tiles, the next tile's records on their way into the other of two LDS
// buffers (global-to-LDS, no registers) while this one is computed.  Per
// pixel 64 bytes as in memory, piece s of a pixel in slot s ^ (column / 4 mod
// 4): the 16-byte fragment reads of 16 neighbouring pixels and the transposing
// reads touch every bank alike, and since the swizzle depends on the column
// only, every read of a lane is one of a few addresses plus a constant.
// * Input gradient: wave w takes rows 2w and 2w + 1; a fragment of a halo row
//   serves both.  The MFMAs of an output are those of the forward kernel on
//   the flipped weights, tap by tap.
// * Weight gradient, dW[t][co][ci] = sum_q dz[q - off_t][co] a[q][ci]: K runs
//   over the 32 pixels q of a tile row, both operands by transposing LDS reads
//   (ds_read_b64_tr_b16: lane l of 16 receives channel l of four pixels); wave
//   w takes the channel quadrant w mod 4 of rows 8 (w / 4) .., the fragments
//   of three dz rows held in registers while a's rows pass.
//   db is one more MFMA against ones.  Every wave keeps its sums over all its
//   tiles and writes them once: records 2 b and 2 b + 1 of workgroup b.
constexpr int BK_TH = 16, BK_WS = TW + 2, BK_NP = (BK_TH + 2) * BK_WS;  // tile rows, halo columns, halo pixels
constexpr int BK_DZ_LOADS = (BK_NP * 4 + 63) / 64, BK_A_LOADS = BK_TH * TW * 4 / 64;  // of a wave, 1 KB each
constexpr int BK_BUF = (BK_DZ_LOADS + BK_A_LOADS) * 1024;
constexpr size_t BK_LDS = 2 * (size_t)BK_BUF;
constexpr int BK_THREADS = 512;

__device__ const uint4 zero_piece = {0u, 0u, 0u, 0u};  // what pixels outside the image read

// Lane l's 16 bytes at p into lds + 16 l.
__device__ __forceinline__ void load_piece(const void *p, unsigned char *lds) {
#if defined(__HIP_DEVICE_COMPILE__)
    __builtin_amdgcn_global_load_lds(p, (__attribute__((address_space(3))) void *)lds, 16, 0, 0);
#else
    (void)p;
    (void)lds;
#endif
}

// Eight K values of a lane by two transposing reads of four.
__device__ __forceinline__ bf16x8 read_tr(const unsigned char *p0, const unsigned char *p1) {
#if defined(__HIP_DEVICE_COMPILE__)
    typedef short s4 __attribute__((ext_vector_type(4)));
    struct {
        s4 lo, hi;
    } v = {__builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4 *)p0),
           __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4 *)p1)};
    return __builtin_bit_cast(bf16x8, v);
#else
    (void)p0;
    (void)p1;
    return bf16x8{};
#endif
}

__global__ void __launch_bounds__(BK_THREADS, 2) k_conv32_back(const uint16_t *__restrict__ a,
                                                              const uint16_t *__restrict__ dz,
                                                              const uint16_t *__restrict__ wp,
                                                              uint16_t *__restrict__ dzn, float *__restrict__ part,
                                                              int H, int W, int ntiles, TileMap tm) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, g = lane >> 4;
    // workgroup b (on XCD b mod 8) takes range (b mod 8) nb / 8 + b / 8 of the
    // tiles: neighbouring ranges, and so most shared halos, on one XCD
    const int nb = (int)gridDim.x;
    const int rank = nb % 8 ? (int)blockIdx.x : (int)(blockIdx.x % 8) * (nb / 8) + (int)blockIdx.x / 8;
    const int t0 = (int)((long)ntiles * rank / nb), t1 = (int)((long)ntiles * (rank + 1) / nb);

    auto load = [&](int tile, unsigned char *buf) {
        int img, y0, x0;
        tm.of_rows(tile, BK_TH, img, y0, x0);
        const uint16_t *di = dz + (long)img * H * W * CH, *ai = a + (long)img * H * W * CH;
#pragma unroll
        for (int k = 0; k < (BK_DZ_LOADS + 7) / 8; k++) {
            const int i = wave + 8 * k;
            if (i >= BK_DZ_LOADS) break;
            const int s = i * 64 + lane, p = s >> 2, r = p / BK_WS, c = p - r * BK_WS;
            const int gy = y0 + r - 1, gx = x0 + c - 1;
            const bool in = p < BK_NP && (unsigned)gy < (unsigned)H && (unsigned)gx < (unsigned)W;
            const void *src = di + (((long)gy * W + gx) * CH + ((s ^ (c >> 2)) & 3) * 8);
            load_piece(in ? src : &zero_piece, buf + i * 1024);
        }
#pragma unroll
        for (int k = 0; k < BK_A_LOADS / 8; k++) {
            const int i = wave + 8 * k;
            const int s = i * 64 + lane, p = s >> 2, r = p / TW, c = p - r * TW;
            const int gy = y0 + r, gx = x0 + c;
            const void *src = ai + (((long)gy * W + gx) * CH + ((s ^ (c >> 2)) & 3) * 8);
            load_piece(gy < H && gx < W ? src : &zero_piece, buf + (BK_DZ_LOADS + i) * 1024);
        }
    };
    if (t0 < t1) load(t0, smem_raw);

    bf16x8 A[2][9];
#pragma unroll
    for (int n = 0; n < 2; n++)
#pragma unroll
        for (int t = 0; t < 9; t++)
            A[n][t] = *reinterpret_cast<const bf16x8 *>(wp + ((t * CH + n * 16 + j) * CH + 8 * g));
    bf16x8 ones;
#pragma unroll
    for (int e = 0; e < 8; e++) ones[e] = (__bf16)1.0f;
    const floatx4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    floatx4 dw[9], db = zero;
#pragma unroll
    for (int t = 0; t < 9; t++) dw[t] = zero;
    const int nbo = (wave >> 1) & 1, nbi = wave & 1, rh = wave >> 2;  // wgrad: quadrant and row half

    // a lane's addresses within a row: 16-byte piece g of column cb + j + kx
    // (a column 16 further has the same slot), the transposed four channels of
    // column kx + 8 g + 4 h + j / 4
    auto slot = [](int c, int piece) { return c * 64 + ((piece ^ (c >> 2)) & 3) * 16; };
    int o_b[3], o_z[3][2], o_a[2], o_m[2];
#pragma unroll
    for (int k = 0; k < 3; k++) {
        o_b[k] = 2 * wave * BK_WS * 64 + slot(j + k, g);
#pragma unroll
        for (int h = 0; h < 2; h++)
            o_z[k][h] = rh * 8 * BK_WS * 64 + slot(k + 8 * g + 4 * h + (j >> 2), nbo * 2 + ((j & 3) >> 1)) + 8 * (j & 1);
    }
#pragma unroll
    for (int h = 0; h < 2; h++) {
        o_a[h] = BK_DZ_LOADS * 1024 + rh * 8 * TW * 64 + slot(8 * g + 4 * h + (j >> 2), nbi * 2 + ((j & 3) >> 1)) + 8 * (j & 1);
        o_m[h] = BK_DZ_LOADS * 1024 + 2 * wave * TW * 64 + slot(j, h * 2 + (g >> 1)) + 8 * (g & 1);
    }

    for (int tile = t0; tile < t1; tile++) {
        const unsigned char *cur = smem_raw + ((tile - t0) & 1) * BK_BUF;
        // this tile's records have arrived, and every wave is done with the other buffer
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tile + 1 < t1) load(tile + 1, smem_raw + ((tile + 1 - t0) & 1) * BK_BUF);
        int img, y0, x0;
        tm.of_rows(tile, BK_TH, img, y0, x0);
        const long ibase = (long)img * H * W;
#pragma unroll
        for (int cb = 0; cb < TW; cb += 16) {
            floatx4 acc[2][2] = {{zero, zero}, {zero, zero}};
#pragma unroll
            for (int hr = 0; hr < 4; hr++)
#pragma unroll
                for (int kx = 0; kx < 3; kx++) {
                    const bf16x8 B = *reinterpret_cast<const bf16x8 *>(cur + o_b[kx] + (hr * BK_WS + cb) * 64);
#pragma unroll
                    for (int i = 0; i < 2; i++) {
                        const int ky = hr - i;
                        if (ky < 0 || ky > 2) continue;
                        acc[i][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[0][ky * 3 + kx], B, acc[i][0], 0, 0, 0);
                        acc[i][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(A[1][ky * 3 + kx], B, acc[i][1], 0, 0, 0);
                    }
                }
#pragma unroll
            for (int i = 0; i < 2; i++) {
                const int gy = y0 + 2 * wave + i, gx = x0 + cb + j;
                if (gy < H && gx < W) {
                    uint16_t *dst = dzn + (ibase + (long)gy * W + gx) * CH + 4 * g;
#pragma unroll
                    for (int n = 0; n < 2; n++) {
                        const uint2 m = *reinterpret_cast<const uint2 *>(cur + o_m[n] + (i * TW + cb) * 64);
                        const uint16_t mm[4] = {(uint16_t)(m.x & 0xffff), (uint16_t)(m.x >> 16),
                                                (uint16_t)(m.y & 0xffff), (uint16_t)(m.y >> 16)};
                        float v[4];
#pragma unroll
                        for (int e = 0; e < 4; e++) v[e] = positive_bf16(mm[e]) ? acc[i][n][e] : 0.0f;
                        uint2 o;
                        o.x = (uint32_t)to_bf16(v[0]) | ((uint32_t)to_bf16(v[1]) << 16);
                        o.y = (uint32_t)to_bf16(v[2]) | ((uint32_t)to_bf16(v[3]) << 16);
                        *reinterpret_cast<uint2 *>(dst + n * 16) = o;
                    }
                }
            }
        }
        bf16x8 z[3][3];  // dz halo rows r, r + 1, r + 2 (slot row mod 3) at columns 0, 1, 2 on
#pragma unroll
        for (int r = 0; r < 2; r++)
#pragma unroll
            for (int k = 0; k < 3; k++)
                z[r][k] = read_tr(cur + o_z[k][0] + r * BK_WS * 64, cur + o_z[k][1] + r * BK_WS * 64);
#pragma unroll
        for (int r = 0; r < 8; r++) {
#pragma unroll
            for (int k = 0; k < 3; k++)
                z[(r + 2) % 3][k] = read_tr(cur + o_z[k][0] + (r + 2) * BK_WS * 64, cur + o_z[k][1] + (r + 2) * BK_WS * 64);
            const bf16x8 av = read_tr(cur + o_a[0] + r * TW * 64, cur + o_a[1] + r * TW * 64);
#pragma unroll
            for (int t = 0; t < 9; t++)
                dw[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(z[(r + 2 - t / 3) % 3][2 - t % 3], av, dw[t], 0, 0, 0);
            if (nbi == 0) db = __builtin_amdgcn_mfma_f32_16x16x32_bf16(z[(r + 1) % 3][1], ones, db, 0, 0, 0);
        }
    }
    float *out = part + (long)(2 * blockIdx.x + rh) * WG_REC;
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int e = 0; e < 4; e++) out[(t * CH + nbo * 16 + 4 * g + e) * CH + nbi * 16 + j] = dw[t][e];
    if (nbi == 0 && j == 0) {
#pragma unroll
        for (int e = 0; e < 4; e++) out[9 * CH * CH + nbo * 16 + 4 * g + e] = db[e];
    }
}

// The sums of a block of 256 threads over its lanes of equal channel group
// tid mod 8 (4 channels each), then over its waves, in a fixed order: out[ch * 9
// + t], ch = 4 (tid mod 8) + e.  red: 4 * 9 * CH floats.
__device__ __forceinline__ void block_sum_taps(float (&acc)[9][4], float *red, float *out) {
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, cg = tid & 7;
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
#pragma unroll
            for (int x = 8; x < 64; x <<= 1) acc[t][e] += __shfl_xor(acc[t][e], x);
            if (lane < 8) red[wave * 9 * CH + (cg * 4 + e) * 9 + t] = acc[t][e];
        }
    __syncthreads();
    for (int i = tid; i < 9 * CH; i += 256)
        out[i] = ((red[i] + red[9 * CH + i]) + red[2 * 9 * CH + i]) + red[3 * 9 * CH + i];
}

// A tile of the first and last layers' gradients, for a thread of column col.
struct GradTile {
    int y0, x0;
    long ibase, base;  // first pixel of the image, of the tile
    int col;           // the thread's column of the tile, inside the image
    __device__ GradTile(const TileMap &tm, int tile, int H, int W, int c) {
        int img;
        tm.of(tile, img, y0, x0);
        ibase = (long)img * H * W;
        base = ibase + (long)y0 * W + x0;
        col = min(c, W - 1 - x0);
    }
    // halo value i's pixel, moved inside the image, and whether it was inside
    __device__ long halo(int i, int H, int W, bool &in) const {
        const int gy = y0 + i / WS - 1, gx = x0 + i % WS - 1;
        in = gy >= 0 && gy < H && gx >= 0 && gx < W;
        return ibase + (long)min(max(gy, 0), H - 1) * W + min(max(gx, 0), W - 1);
    }
};

// Weight gradient of the 1 -> 32 layer: partial[block] = (dW1[co][t], db1[co])
// over the tiles blockIdx.x, blockIdx.x + gridDim.x, ...  As k_conv_out_back: thread
// tid takes the 4 channels (tid mod 8) * 4.. of the tile's column tid / 8, four
// rows at a time (one 8-byte load of dz per pixel), the nine taps of
// bf16(x/scale) from the tile with its halo in LDS, the next tile's loads issued
// as this one's values are taken up, the sums in registers across tiles.
// Bound by reading dz, 114 us for 32 images of 512 x 512: 199 us with eight
// channels a thread and the loads waited for, 161 this way.
__global__ void __launch_bounds__(256, 2) k_conv_in_wgrad(const float *__restrict__ x, float scale,
                                                          const uint16_t *__restrict__ dz, float *__restrict__ part,
                                                          int H, int W, int ntiles, TileMap tm) {
    __shared__ float sx[HS * WS];
    __shared__ float red[4 * 9 * CH];
    constexpr int KB = 4;                      // rows at a time
    constexpr int ND = (HS * WS + 255) / 256;  // halo values per thread
    const int tid = threadIdx.x, cg = tid & 7, col = tid >> 3;
    float acc[9][4], db[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        db[e] = 0.0f;
#pragma unroll
        for (int t = 0; t < 9; t++) acc[t][e] = 0.0f;
    }
    uint2 v[TH];
    float nx[ND];
    auto load_dz = [&](const GradTile &o, int r) {
        const long px = min(r, H - 1 - o.y0) * W + o.col;
        v[r] = *reinterpret_cast<const uint2 *>(dz + o.base * CH + px * CH + cg * 4);
    };
    auto load_x = [&](const GradTile &o) {
#pragma unroll
        for (int k = 0; k < ND; k++) {
            bool in;
            const long p = o.halo(min(tid + 256 * k, HS * WS - 1), H, W, in);
            nx[k] = __int_as_float(__float_as_int(x[p]) & -(int)in);
        }
    };
    const GradTile o0(tm, min((int)blockIdx.x, ntiles - 1), H, W, col);
    load_x(o0);
#pragma unroll
    for (int r = 0; r < TH; r++) load_dz(o0, r);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const GradTile o(tm, tile, H, W, col), on(tm, min(tile + (int)gridDim.x, ntiles - 1), H, W, col);
        __syncthreads();  // the previous tile's reads of sx are done
#pragma unroll
        for (int k = 0; k < ND; k++)
            if (tid + 256 * k < HS * WS) sx[tid + 256 * k] = round_bf16(nx[k] / scale);
        __syncthreads();
        load_x(on);
#pragma unroll
        for (int r0 = 0; r0 < TH; r0 += KB) {
            float a[KB][4], d[KB + 2][3];
#pragma unroll
            for (int k = 0; k < KB; k++) {
                const uint32_t in = -(uint32_t)(o.y0 + r0 + k < H && col == o.col);  // a mask: no branch
                const uint32_t w2[2] = {v[r0 + k].x & in, v[r0 + k].y & in};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    a[k][e] = from_bf16((uint16_t)(w2[e >> 1] >> (16 * (e & 1))));
                    db[e] += a[k][e];
                }
                load_dz(on, r0 + k);
            }
#pragma unroll
            for (int k = 0; k < KB + 2; k++)
#pragma unroll
                for (int c = 0; c < 3; c++) d[k][c] = sx[(r0 + k) * WS + col + c];
#pragma unroll
            for (int t = 0; t < 9; t++)
#pragma unroll
                for (int k = 0; k < KB; k++)
#pragma unroll
                    for (int e = 0; e < 4; e++)
                        acc[t][e] = __builtin_fmaf(d[k + t / 3][t % 3], a[k][e], acc[t][e]);
        }
    }
    float *out = part + (long)blockIdx.x * IN_REC;
    block_sum_taps(acc, red, out);
    __syncthreads();
    const int lane = tid & 63, wave = tid >> 6;
#pragma unroll
    for (int e = 0; e < 4; e++) {
#pragma unroll
        for (int s = 8; s < 64; s <<= 1) db[e] += __shfl_xor(db[e], s);
        if (lane < 8) red[wave * CH + cg * 4 + e] = db[e];
    }
    __syncthreads();
    if (tid < CH) out[9 * CH + tid] = ((red[tid] + red[CH + tid]) + red[2 * CH + tid]) + red[3 * CH + tid];
}

// Loss, input and weight gradient of the 32 -> 1 layer in one pass over a4,
// persistent over the tiles blockIdx.x, blockIdx.x + gridDim.x, ...:
//   dy = 2 (yn - t/scale) / N, loss partial[block] = sum (yn - t/scale)^2
//   dz4[q][ci] = bf16(sum_t dy[q - off_t] W5[ci][t] * (a4 > 0))
//   partial[block] = (dW5[ci][t] = sum_q dy[q - off_t] a4[q][ci], db5 = sum dy)
// The gradients take the same nine values of dy around a pixel q, from the tile
// computed with its halo into LDS.  Thread tid takes the 4 channels (tid mod 8) * 4.. of
// the tile's column tid / 8, KB rows at a time, so neighbouring rows share
// their dy and four rows a tap's weights: one 8-byte load of a4 and one
// 8-byte store of dz4 per pixel (a wave 8 whole records).  The next tile's loads
// are issued (clamped, not guarded) as this tile's values are taken up, and the
// weight sums stay in registers across tiles.  With 8 channels a thread the
// sums, weights and values of a tile did not fit the registers; two waves a
// SIMD, since a third has its sums spilled.  32 images of 512 x 512: 532 us as
// three kernels (loss, weight gradient, input gradient), 289 as one; its 128 bytes
// per pixel take 227.
__global__ void __launch_bounds__(256, 2) k_conv_out_back(const float *__restrict__ yn,
                                                          const float *__restrict__ target, float scale,
                                                          float fN, const uint16_t *__restrict__ a4,
                                                          const float *__restrict__ prm, uint16_t *__restrict__ dz4,
                                                          float *__restrict__ part, float *__restrict__ lpart, int H,
                                                          int W, int ntiles, TileMap tm) {
    __shared__ float sdy[HS * WS];
    __shared__ __align__(16) float sw[9 * CH];  // [t][ci]
    __shared__ double dred[2][4];
    __shared__ float red[4 * 9 * CH];
    constexpr int KB = 4;                      // rows at a time
    constexpr int ND = (HS * WS + 255) / 256;  // halo values per thread
    static_assert(TW * 8 == 256 && TH % KB == 0, "a thread per column and 4 channels");
    const int tid = threadIdx.x, cg = tid & 7, col = tid >> 3;
    for (int i = tid; i < 9 * CH; i += 256) sw[i] = round_bf16(prm[OFF_W5 + (i % CH) * 9 + i / CH]);
    float acc[9][4], dsum = 0.0f;
    double lsum = 0.0;
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
        for (int e = 0; e < 4; e++) acc[t][e] = 0.0f;
    uint2 v[TH];
    float ne[ND];  // yn - t/scale, zero outside the image
    // addresses: a wave-uniform tile base and offsets within the tile
    auto load_a4 = [&](const GradTile &o, int r) {
        const long px = min(r, H - 1 - o.y0) * W + o.col;
        v[r] = *reinterpret_cast<const uint2 *>(a4 + o.base * CH + px * CH + cg * 4);
    };
    auto load_err = [&](const GradTile &o) {
#pragma unroll
        for (int k = 0; k < ND; k++) {
            bool in;
            const long p = o.halo(min(tid + 256 * k, HS * WS - 1), H, W, in);
            const float d = yn[p] - target[p] / scale;
            ne[k] = __int_as_float(__float_as_int(d) & -(int)in);
        }
    };
    const GradTile o0(tm, min((int)blockIdx.x, ntiles - 1), H, W, col);
    load_err(o0);
#pragma unroll
    for (int r = 0; r < TH; r++) load_a4(o0, r);
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const GradTile o(tm, tile, H, W, col), on(tm, min(tile + (int)gridDim.x, ntiles - 1), H, W, col);
        __syncthreads();  // the previous tile's reads of sdy are done
#pragma unroll
        for (int k = 0; k < ND; k++) {
            const int i = tid + 256 * k, r = i / WS - 1, c = i % WS - 1;
            if (i < HS * WS) sdy[i] = 2.0f * ne[k] / fN;
            if (r >= 0 && r < TH && c >= 0 && c < TW) lsum += (double)ne[k] * (double)ne[k];
        }
        __syncthreads();
        load_err(on);
#pragma unroll
        for (int r0 = 0; r0 < TH; r0 += KB) {
            float a[KB][4], g[KB][4], d[KB + 2][3];
#pragma unroll
            for (int k = 0; k < KB; k++) {
                const uint32_t in = -(uint32_t)(o.y0 + r0 + k < H && col == o.col);  // a mask: no branch
                const uint32_t w2[2] = {v[r0 + k].x & in, v[r0 + k].y & in};
#pragma unroll
                for (int e = 0; e < 4; e++) {
                    a[k][e] = from_bf16((uint16_t)(w2[e >> 1] >> (16 * (e & 1))));
                    g[k][e] = 0.0f;
                }
                load_a4(on, r0 + k);
            }
#pragma unroll
            for (int k = 0; k < KB + 2; k++)
#pragma unroll
                for (int c = 0; c < 3; c++) d[k][c] = sdy[(r0 + k) * WS + col + c];
#pragma unroll
            for (int t = 0; t < 9; t++) {
                const float4 w4 = *reinterpret_cast<const float4 *>(sw + t * CH + cg * 4);
                const float w[4] = {w4.x, w4.y, w4.z, w4.w};
#pragma unroll
                for (int k = 0; k < KB; k++) {
                    const float dq = d[k + 2 - t / 3][2 - t % 3];  // dy[q - off_t]
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        g[k][e] = __builtin_fmaf(dq, w[e], g[k][e]);
                        acc[t][e] = __builtin_fmaf(dq, a[k][e], acc[t][e]);
                    }
                }
            }
#pragma unroll
            for (int k = 0; k < KB; k++) {
                uint32_t ow[2];
                // summed here, not in a branch of the mask with all operands alive
#pragma unroll
                for (int e = 0; e < 4; e++) asm volatile("" : "+v"(g[k][e]));
#pragma unroll
                for (int e = 0; e < 4; e += 2)  // positive_bf16, on the floats' bits
                    ow[e >> 1] = pack_bf16(__float_as_int(a[k][e]) > 0 ? g[k][e] : 0.0f,
                                           __float_as_int(a[k][e + 1]) > 0 ? g[k][e + 1] : 0.0f);
                if (o.y0 + r0 + k < H && col == o.col)
                    *reinterpret_cast<uint2 *>(dz4 + o.base * CH + (long)((r0 + k) * W + col) * CH + cg * 4) =
                        make_uint2(ow[0], ow[1]);
            }
        }
        dsum += sdy[(tid / TW + 1) * WS + tid % TW + 1];  // db5: thread tid takes pixel tid of every tile
    }
    float *out = part + (long)blockIdx.x * OUT_REC;
    block_sum_taps(acc, red, out);
    // db5 and the loss: pairwise over the lanes, then over the waves, in double
    // -- one large error must not swallow a tile of small ones
    const int lane = tid & 63, wave = tid >> 6;
    double s5 = dsum, sl = lsum;
#pragma unroll
    for (int h = 32; h > 0; h >>= 1) {
        s5 += __shfl_xor(s5, h);
        sl += __shfl_xor(sl, h);
    }
    if (lane == 0) {
        dred[0][wave] = s5;
        dred[1][wave] = sl;
    }
    __syncthreads();
    if (tid < 2) {
        const float v = (float)((dred[tid][0] + dred[tid][1]) + (dred[tid][2] + dred[tid][3]));
        if (tid == 0)
            out[9 * CH] = v;
        else
            lpart[blockIdx.x] = v;
    }
}

// Sum of nparts partial records in block order (double) into the gradient
// vector.  kind 0: 32->32 record (t,co,ci)+db -> W[co][ci][t], b; kind 1 and 2
// records are already in parameter order.
// A block of 1024 threads takes 64 consecutive elements: wave w sums the
// records w, w + 16, ... for its lane's element (coalesced 256-byte rows, eight
// loads in flight per batch), then lane e of wave 0 adds the 16 wave sums in
// wave order -- a fixed order, so results are bitwise repeatable.
constexpr int RED_WAVES = 16;
__global__ void __launch_bounds__(1024) k_reduce(const float *__restrict__ part, int nparts, int rec, int kind,
                                                 float *__restrict__ gw, float *__restrict__ gb) {
    __shared__ double sw[RED_WAVES][64];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    double s = 0.0;
    if (i < rec) {
        for (int k0 = wave; k0 < nparts; k0 += 8 * RED_WAVES) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int k = k0 + u * RED_WAVES;
                v[u] = k < nparts ? part[(long)k * rec + i] : 0.0f;
            }
#pragma unroll
            for (int u = 0; u < 8; u++) s += (double)v[u];
        }
    }
    sw[wave][lane] = s;
    __syncthreads();
    if (wave != 0 || i >= rec) return;
    s = 0.0;
    for (int w = 0; w < RED_WAVES; w++) s += sw[w][lane];
    const float v = (float)s;
    if (kind == 0) {
        if (i < 9 * CH * CH) {
            const int t = i / (CH * CH), co = (i / CH) % CH, ci = i % CH;
            gw[(co * CH + ci) * 9 + t] = v;
        } else {
            gb[i - 9 * CH * CH] = v;
        }
    } else {
        const int nw = 9 * CH;
        if (i < nw) gw[i] = v;
        else gb[i - nw] = v;
    }
}

// Sum of per-block partials in order, times f: out[grp*stride + comp] =
// f * sum_i part[(grp*per + i)*stride + comp].
// One block of 256 threads per output: thread t adds the partials t, t + 256,
// ... in order (double, eight loads in flight per batch), then the 256 sums
// are added by a fixed pairwise tree -- bitwise repeatable.
__global__ void __launch_bounds__(256) k_sum_groups(const float *__restrict__ part, int groups, int per, int stride,
                                                    double f, float *__restrict__ out) {
    __shared__ double sd[256];
    const int k = blockIdx.x, tid = threadIdx.x;
    if (k >= groups * stride) return;
    const int grp = k / stride, comp = k - grp * stride;
    const float *src = part + (long)grp * per * stride + comp;
    double s = 0.0;
    for (int i0 = tid; i0 < per; i0 += 8 * 256) {
        float v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int i = i0 + u * 256;
            v[u] = i < per ? src[(long)i * stride] : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < 8; u++) s += (double)v[u];
    }
    sd[tid] = s;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if (tid < h) sd[tid] += sd[tid + h];
        __syncthreads();
    }
    if (tid == 0) out[k] = (float)(sd[0] * f);
}

// Packed bf16 weights of the three 32->32 layers: forward [t][co][ci] and
// input-gradient [t][ci][co] = W[co][ci][8 - t].
__global__ void k_pack(const float *__restrict__ prm, uint16_t *__restrict__ packed) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= 3 * 9 * CH * CH) return;
    const int l = i / (9 * CH * CH), k = i - l * 9 * CH * CH;
    const int t = k / (CH * CH), a = (k / CH) % CH, b = k % CH;
    const float *w = prm + OFF_W2 + l * (9 * CH * CH + CH);
    uint16_t *fw = packed + (long)l * PACK_LAYER, *bw = fw + 9 * CH * CH;
    fw[k] = to_bf16(w[(a * CH + b) * 9 + t]);      // a = co, b = ci
    bw[k] = to_bf16(w[(b * CH + a) * 9 + 8 - t]);  // a = ci (output), b = co (input)
}

__global__ void k_adam(float *__restrict__ p, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, int n, float lr, float b1, float b2, float eps, float c1, float c2) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.0f - b1) * gi;
    const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] = p[i] - lr * (mi * c1) / (sqrtf(vi * c2) + eps);
}

int cnn_fail(int code, const char *msg) { return gr_set_error(code, msg); }
#define CNN_HIP(call)                                                       \
    do {                                                                    \
        hipError_t e_ = (call);                                             \
        if (e_ != hipSuccess) return cnn_fail(GR_EHIP, hipGetErrorString(e_)); \
    } while (0)

TileMap tiles_of(int H, int W) { return TileMap{(W + TW - 1) / TW, (H + TH - 1) / TH}; }

int check_dims(int n, int H, int W) {
    if (n < 1 || H < 1 || W < 1 || (long)n * H * W > (1L << 31) - 1) return cnn_fail(GR_EINVAL, "invalid image batch");
    const TileMap tm = tiles_of(H, W);
    if ((long)tm.tiles_x * tm.tiles_y * n > (1L << 31) - 1) return cnn_fail(GR_EINVAL, "too many tiles");
    return GR_OK;
}

// Segments of rows a strip is cut into: the fewest steps of the busiest CU
// (one workgroup each at a time); a segment of k rows takes k / 2 + 8 steps,
// the pipeline's fill and the four halo rows on either side among them.  At
// least 8 rows each, and per image no more workgroups than its tiles of 16 x 32,
// what the work sizes hold partial sums for.  A strip is wider than a tile, so 256 x 256
// still goes in segments of 12 rows (31.4 us a call; 34.0 with 16), 4096 x 64 in 128
// of them (44.6 us; 65.7 with 64).
long infer_tiles(int H, int W) {
    return (long)((W + 31) / 32) * ((H + 15) / 16);
}

int forward_segments(int n, int H, int W, int strips) {
    const long cus = gr_cu_count() > 0 ? gr_cu_count() : 256;
    const int most = (int)std::min({256L, (H + 7) / 8L, infer_tiles(H, W) / strips});
    int best = 1;
    long best_cost = 0;
    for (int v = 1; v <= most; v++) {
        const long rows = (H + v - 1) / v, groups = (long)n * strips * ((H + rows - 1) / rows);
        const long cost = (groups + cus - 1) / cus * ((rows + 1) / 2 + 8);
        if (v == 1 || cost < best_cost) {
            best = v;
            best_cost = cost;
        }
    }
    return best;
}

int run_forward(const float *params, const unsigned short *packed, const float *x, int n, int H, int W, float scale,
                uint16_t *const (&act)[4], float *y, float *yn, float *slice_stats, float *stats, hipStream_t s) {
    const int strips = (W + FW_OUT - 1) / FW_OUT, v = forward_segments(n, H, W, strips);
    const int rows = (H + v - 1) / v, segs = (H + rows - 1) / rows;
    if ((long)n * strips * segs > (1L << 31) - 1) return cnn_fail(GR_EINVAL, "too many tiles");
    FwdArgs A{x, params, reinterpret_cast<const uint16_t *>(packed), {act[0], act[1], act[2], act[3]}, y, yn,
              slice_stats ? stats : nullptr, scale, H, W, strips, segs, rows};
    CNN_HIP(gr_allow_lds(k_forward, FW_LDS));
    hipLaunchKernelGGL(k_forward, dim3((unsigned)(n * strips * segs)), dim3(FW_THREADS), FW_LDS, s, A);
    if (slice_stats)
        hipLaunchKernelGGL(k_sum_groups, dim3(2 * n), dim3(256), 0, s, stats, n, strips * segs, 2, 1.0, slice_stats);
    CNN_HIP(hipGetLastError());
    return GR_OK;
}

// Whether a batch of npx values at p lies over the one at x.
bool over(const float *x, const float *p, long npx) {
    const uintptr_t a = (uintptr_t)x, b = (uintptr_t)p, bytes = sizeof(float) * (size_t)npx;
    return p && a < b + bytes && b < a + bytes;
}

// run_forward on a copy of x, in stream-ordered memory: where what it writes
// lies over x and nothing else is left to read x from.
int run_forward_copy(const float *params, const unsigned short *packed, const float *x, int n, int H, int W,
                     float scale, uint16_t *const (&act)[4], float *y, float *yn, float *slice_stats, float *stats,
                     hipStream_t s) {
    const size_t bytes = sizeof(float) * (size_t)n * H * W;
    void *copy = nullptr;
    if (hipMallocAsync(&copy, bytes, s) != hipSuccess) {
        (void)hipGetLastError();
        return cnn_fail(GR_ENOMEM, "no device memory for a copy of the images (y or yn lies over x)");
    }
    const hipError_t e = hipMemcpyAsync(copy, x, bytes, hipMemcpyDeviceToDevice, s);
    const int rc = e == hipSuccess ? run_forward(params, packed, (const float *)copy, n, H, W, scale, act, y, yn,
                                                 slice_stats, stats, s)
                                   : cnn_fail(GR_EHIP, hipGetErrorString(e));
    (void)hipFreeAsync(copy, s);
    return rc;
}

}  // namespace

extern "C" {

long gr_cnn_param_count(void) { return N_PARAMS; }
long gr_cnn_packed_count(void) { return 3L * PACK_LAYER; }

size_t gr_cnn_work_bytes(int n, int H, int W) {
    const TileMap tm = tiles_of(H, W);
    const long ntiles = (long)tm.tiles_x * tm.tiles_y * n;
    const long npx = (long)n * H * W;
    const size_t up = 256;
    auto al = [&](size_t b) { return (b + up - 1) / up * up; };
    return al(sizeof(float) * npx)                         // yn
           + 2 * al(sizeof(uint16_t) * npx * CH)           // dz ping-pong
           + al(sizeof(float) * (size_t)MAX_WG_BLOCKS * WG_REC)  // weight-gradient partials
           + al(sizeof(float) * 2 * (size_t)ntiles)        // forward statistics partials
           + al(sizeof(float) * 1024);                     // loss partials
}

int gr_cnn_pack(const float *params, unsigned short *packed, void *stream) {
    if (!params || !packed) return cnn_fail(GR_EINVAL, "null argument");
    const int n = 3 * 9 * CH * CH;
    hipLaunchKernelGGL(k_pack, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, params, packed);
    CNN_HIP(hipGetLastError());
    return GR_OK;
}

int gr_cnn_forward(const float *params, const unsigned short *packed, const float *x, int n, int H, int W, float scale,
                   unsigned short *a1, unsigned short *a2, unsigned short *a3, unsigned short *a4, float *y,
                   float *yn, float *slice_stats, void *work, void *stream) {
    if (!params || !packed || !x || !a1 || !a2 || !a3 || !a4 || !(scale > 0.0f)) return cnn_fail(GR_EINVAL, "null argument or scale <= 0");
    if (a1 == a2 || a2 == a3 || a3 == a4) return cnn_fail(GR_EINVAL, "consecutive activations must not alias");
    int rc = check_dims(n, H, W);
    if (rc) return rc;
    if (slice_stats && !work) return cnn_fail(GR_EINVAL, "slice statistics need the work buffer");
    float *stats = nullptr;
    if (slice_stats) {
        char *wb = (char *)work;
        const long npx = (long)n * H * W;
        auto al = [](size_t b) { return (b + 255) / 256 * 256; };
        wb += al(sizeof(float) * npx) + 2 * al(sizeof(uint16_t) * npx * CH) +
              al(sizeof(float) * (size_t)MAX_WG_BLOCKS * WG_REC);
        stats = (float *)wb;
    }
    // a buffer named for two layers ends holding the later one
    uint16_t *act[4] = {a1 == a3 || a1 == a4 ? nullptr : a1, a2 == a4 ? nullptr : a2, a3, a4};
    hipStream_t s = (hipStream_t)stream;
    const long npx = (long)n * H * W;
    if (!over(x, y, npx) && !over(x, yn, npx))
        return run_forward(params, packed, x, n, H, W, scale, act, y, yn, slice_stats, stats, s);
    if ((y != x && over(x, y, npx)) || (yn != x && over(x, yn, npx)))
        return run_forward_copy(params, packed, x, n, H, W, scale, act, y, yn, slice_stats, stats, s);
    rc = run_forward(params, packed, x, n, H, W, scale, act, nullptr, nullptr, slice_stats, stats, s);
    if (rc) return rc;
    const int cols = (W + 15) / 16, segs = (H + OUT_ROWS - 1) / OUT_ROWS;
    const long nwaves = (long)n * cols * segs;
    hipLaunchKernelGGL(k_conv_out, dim3((unsigned)((nwaves + 3) / 4)), dim3(256), 0, s, a4, x, scale, params, y, yn, H,
                       W, cols, segs, nwaves);
    CNN_HIP(hipGetLastError());
    return GR_OK;
}

size_t gr_cnn_infer_work_bytes(int n, int H, int W) {
    // two floats per workgroup: at most one per 16 rows and 32 columns
    return sizeof(float) * 2 * (size_t)infer_tiles(H, W) * (n > 0 ? n : 0);
}

int gr_cnn_infer(const float *params, const unsigned short *packed, const float *x, int n, int H, int W, float scale,
                 float *y, float *slice_stats, void *work, void *stream) {
    if (!params || !packed || !x || !y || !(scale > 0.0f)) return cnn_fail(GR_EINVAL, "null argument or scale <= 0");
    int rc = check_dims(n, H, W);
    if (rc) return rc;
    if (slice_stats && !work) return cnn_fail(GR_EINVAL, "slice statistics need the work buffer");
    uint16_t *act[4] = {nullptr, nullptr, nullptr, nullptr};
    if (over(x, y, (long)n * H * W))
        return run_forward_copy(params, packed, x, n, H, W, scale, act, y, nullptr, slice_stats, (float *)work,
                                (hipStream_t)stream);
    return run_forward(params, packed, x, n, H, W, scale, act, y, nullptr, slice_stats, (float *)work,
                       (hipStream_t)stream);
}

int gr_cnn_backward(const float *params, const unsigned short *packed, const float *x, const float *target, int n,
                    int H, int W, float scale, const unsigned short *a1, const unsigned short *a2,
                    const unsigned short *a3, const unsigned short *a4, const float *yn, float *grads, float *loss,
                    void *work, void *stream) {
    if (!params || !packed || !x || !target || !a1 || !a2 || !a3 || !a4 || !yn || !grads || !work || !(scale > 0.0f))
        return cnn_fail(GR_EINVAL, "null argument or scale <= 0");
    int rc = check_dims(n, H, W);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    const TileMap tm = tiles_of(H, W);
    const int ntiles = tm.tiles_x * tm.tiles_y * n;
    const long npx = (long)n * H * W;
    auto al = [](size_t b) { return (b + 255) / 256 * 256; };
    char *wb = (char *)work;
    wb += al(sizeof(float) * npx);  // yn slot (the caller's yn may live there)
    uint16_t *dzA = (uint16_t *)wb;
    wb += al(sizeof(uint16_t) * npx * CH);
    uint16_t *dzB = (uint16_t *)wb;
    wb += al(sizeof(uint16_t) * npx * CH);
    float *part = (float *)wb;
    wb += al(sizeof(float) * (size_t)MAX_WG_BLOCKS * WG_REC);
    wb += al(sizeof(float) * 2 * (size_t)ntiles);
    float *lpart = (float *)wb;
    const uint16_t *pk = reinterpret_cast<const uint16_t *>(packed);
    const int nwg = ntiles < MAX_WG_BLOCKS ? ntiles : MAX_WG_BLOCKS;

    // layer 5
    hipLaunchKernelGGL(k_conv_out_back, dim3(nwg), dim3(256), 0, s, yn, target, scale, (float)npx, a4, params, dzA, part,
                       lpart, H, W, ntiles, tm);
    if (loss) hipLaunchKernelGGL(k_sum_groups, dim3(1), dim3(256), 0, s, lpart, 1, nwg, 1, 1.0 / (double)npx, loss);
    hipLaunchKernelGGL(k_reduce, dim3((OUT_REC + 63) / 64), dim3(64 * RED_WAVES), 0, s, part, nwg, OUT_REC, 1,
                       grads + OFF_W5, grads + OFF_B5);
    // layers 4, 3, 2
    const unsigned short *acts[4] = {a1, a2, a3, a4};
    const int woff[3] = {OFF_W2, OFF_W3, OFF_W4}, boff[3] = {OFF_B2, OFF_B3, OFF_B4};
    CNN_HIP(gr_allow_lds(k_conv32_back, BK_LDS));
    const TileMap tmb{tm.tiles_x, (H + BK_TH - 1) / BK_TH};
    const int ntb = tmb.tiles_x * tmb.tiles_y * n;
    const int nback = std::min(ntb, std::min(MAX_WG_BLOCKS / 2, gr_cu_count() > 0 ? gr_cu_count() : 256));
    uint16_t *dz = dzA, *dzn = dzB;
    for (int l = 2; l >= 0; l--) {  // layer l+2: input acts[l], output gradient dz
        hipLaunchKernelGGL(k_conv32_back, dim3(nback), dim3(BK_THREADS), BK_LDS, s,
                           reinterpret_cast<const uint16_t *>(acts[l]), dz, pk + (long)l * PACK_LAYER + 9 * CH * CH, dzn,
                           part, H, W, ntb, tmb);
        hipLaunchKernelGGL(k_reduce, dim3((WG_REC + 63) / 64), dim3(64 * RED_WAVES), 0, s, part, 2 * nback, WG_REC, 0,
                           grads + woff[l], grads + boff[l]);
        std::swap(dz, dzn);
    }
    // layer 1
    hipLaunchKernelGGL(k_conv_in_wgrad, dim3(nwg), dim3(256), 0, s, x, scale, dz, part, H, W, ntiles, tm);
    hipLaunchKernelGGL(k_reduce, dim3((IN_REC + 63) / 64), dim3(64 * RED_WAVES), 0, s, part, nwg, IN_REC, 1,
                       grads + OFF_W1, grads + OFF_B1);
    CNN_HIP(hipGetLastError());
    return GR_OK;
}

int gr_cnn_adam(float *params, const float *grads, float *m, float *v, long count, int step, float lr, float beta1,
                float beta2, float eps, void *stream) {
    if (!params || !grads || !m || !v || count < 1 || count > (1L << 30) || step < 1)
        return cnn_fail(GR_EINVAL, "invalid Adam arguments");
    const float c1 = (float)(1.0 / (1.0 - pow((double)beta1, step)));
    const float c2 = (float)(1.0 / (1.0 - pow((double)beta2, step)));
    hipLaunchKernelGGL(k_adam, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, (hipStream_t)stream, params,
                       grads, m, v, (int)count, lr, beta1, beta2, eps, c1, c2);
    CNN_HIP(hipGetLastError());
    return GR_OK;
}

}  // extern "C"
