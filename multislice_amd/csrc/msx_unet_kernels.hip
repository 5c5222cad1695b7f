// msx_unet_kernels.hip -- GPU kernels of the frozen-phonon surrogate (a small
// U-Net that maps a 4-configuration mean ADF image to the converged
// 64-configuration one).
//
// Every convolution (3x3 or 1x1, stride 1, zero padding) is an implicit GEMM on
// the gfx950 matrix cores: v_mfma_f32_32x32x16_bf16, BF16 operands converted
// from the FP32 tensors while they are staged in LDS, FP32 accumulation.
// The same kernel runs the three products of training:
//   FWD : Y[n,co,p]   = sum_{ci,tap} W[co,ci,tap] X[n,ci,p+off(tap)]    (+bias, ReLU)
//   BWDD: dX[n,ci,p]  = sum_{co,tap} W[co,ci,flip(tap)] G[n,co,p+off(tap)]
//   BWDW: dW[co,ci,tap] += sum_{n,p} G[n,co,p] X[n,ci,p+off(tap)]       (split over p)
// where G = dY masked by the ReLU of the layer's output.  Tensors are NCHW FP32.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "msx_fft.hpp"  // lds_barrier
#include "msx_unet.h"

namespace msx {
namespace unet {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Block tile: BM output rows (32 or 64) x BN = 4096/BM columns, K step 32;
// 4 wavefronts, each owning one 32x32 output tile (two MFMAs per K step).
constexpr int BK = 32, KP = BK + 8;  // +8 bf16: 16-byte rows, spread banks

// Operand staging.  A rows are the GEMM's M rows, B rows its N columns; each
// thread stages a run of consecutive k of one row:
//   A: row tid / (BK/KPA), k run (tid % (BK/KPA)) * KPA, KPA = BM*BK/256
//   B: row tid % BN,       k run (tid / BN) * KPB,        KPB = BN*BK/256
// so pixel rows are gathered by consecutive threads (coalesced) and each
// thread writes whole runs of its LDS row.  Indices are decoded once per run
// and stepped, not divided per element.
template <int MODE, int KS, int BM>
__global__ __launch_bounds__(256) void conv_gemm(ConvArgs p) {
    constexpr int BN = 4096 / BM, KPA = BM * BK / 256, KPB = BN * BK / 256, TAPS = KS * KS, R = KS / 2;
    __shared__ __align__(16) __bf16 As[2][BM][KP];
    __shared__ __align__(16) __bf16 Bs[2][BN][KP];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = BM == 64 ? (wave & 1) : 0, wn = BM == 64 ? (wave >> 1) : wave;
    const int HW = p.H * p.W;
    long long M, N, K;
    if (MODE == kFwd) { M = p.Cout; N = (long long)p.N * HW; K = (long long)p.Cin * TAPS; }
    else if (MODE == kBwdData) { M = p.Cin; N = (long long)p.N * HW; K = (long long)p.Cout * TAPS; }
    else { M = p.Cout; N = (long long)p.Cin * TAPS; K = (long long)p.N * HW; }
    const long long m0 = (long long)blockIdx.y * BM, n0 = (long long)blockIdx.x * BN;
    long long k_beg = 0, k_end = K;
    if (MODE == kBwdWeight) {  // split over pixels
        const long long chunk = ((K + gridDim.z - 1) / gridDim.z + BK - 1) / BK * BK;
        k_beg = (long long)blockIdx.z * chunk;
        k_end = k_beg + chunk < K ? k_beg + chunk : K;
    }
    const int a_row = tid / (BK / KPA), a_k = (tid % (BK / KPA)) * KPA;
    const int b_row = tid % BN, b_k = (tid / BN) * KPB;
    const long long am = m0 + a_row, bn = n0 + b_row;
    // B row: a pixel (forward, input gradient) or a (channel, tap) (weight gradient)
    int b_img = 0, b_y = 0, b_x = 0, b_ci = 0, b_dy = 0, b_dx = 0;
    if (bn < N) {
        if (MODE != kBwdWeight) {
            b_img = (int)(bn / HW);
            const int pix = (int)(bn % HW);
            b_y = pix / p.W;
            b_x = pix % p.W;
        } else {
            b_ci = (int)(bn / TAPS);
            const int tap = (int)(bn % TAPS);
            b_dy = tap / KS - R;
            b_dx = tap % KS - R;
        }
    }

    float ra[KPA], rb[KPB];
    auto fetch = [&](long long k0) {
        const long long ka = k0 + a_k;
        if (MODE == kFwd) {
#pragma unroll
            for (int j = 0; j < KPA; ++j) ra[j] = (am < M && ka + j < k_end) ? p.w[am * K + ka + j] : 0.f;
        } else if (MODE == kBwdData) {
            int co = (int)(ka / TAPS), tap = (int)(ka % TAPS);
#pragma unroll
            for (int j = 0; j < KPA; ++j) {
                ra[j] = (am < M && ka + j < k_end) ? p.w[((long long)co * p.Cin + am) * TAPS + (TAPS - 1 - tap)] : 0.f;
                if (++tap == TAPS) { tap = 0; ++co; }
            }
        } else {
            int img = (int)(ka / HW), pix = (int)(ka % HW);
#pragma unroll
            for (int j = 0; j < KPA; ++j) {
                float v = 0.f;
                if (am < M && ka + j < k_end) {
                    const long long o = ((long long)img * p.Cout + am) * HW + pix;
                    v = p.g[o];
                    if (p.relu && p.y[o] <= 0.f) v = 0.f;
                }
                ra[j] = v;
                if (++pix == HW) { pix = 0; ++img; }
            }
        }
        const long long kb = k0 + b_k;
        if (MODE == kFwd || MODE == kBwdData) {
            int c = (int)(kb / TAPS), tap = (int)(kb % TAPS);
            const int C = MODE == kFwd ? p.Cin : p.Cout;
            const float* src = MODE == kFwd ? p.x : p.g;
#pragma unroll
            for (int j = 0; j < KPB; ++j) {
                float v = 0.f;
                if (bn < N && kb + j < k_end) {
                    const int yy = b_y + tap / KS - R, xx = b_x + tap % KS - R;
                    if ((unsigned)yy < (unsigned)p.H && (unsigned)xx < (unsigned)p.W) {
                        const long long o = (((long long)b_img * C + c) * p.H + yy) * p.W + xx;
                        v = src[o];
                        if (MODE == kBwdData && p.relu && p.y[o] <= 0.f) v = 0.f;
                    }
                }
                rb[j] = v;
                if (++tap == TAPS) { tap = 0; ++c; }
            }
        } else {
            int img = (int)(kb / HW);
            const int pix = (int)(kb % HW);
            int y = pix / p.W, x = pix % p.W;
#pragma unroll
            for (int j = 0; j < KPB; ++j) {
                float v = 0.f;
                if (bn < N && kb + j < k_end) {
                    const int yy = y + b_dy, xx = x + b_dx;
                    if ((unsigned)yy < (unsigned)p.H && (unsigned)xx < (unsigned)p.W)
                        v = p.x[(((long long)img * p.Cin + b_ci) * p.H + yy) * p.W + xx];
                }
                rb[j] = v;
                if (++x == p.W) { x = 0; if (++y == p.H) { y = 0; ++img; } }
            }
        }
    };

    f32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    const int r = lane & 31, kh = (lane >> 5) * 8;
    int buf = 0;
    if (k_beg < k_end) fetch(k_beg);
    for (long long k0 = k_beg; k0 < k_end; k0 += BK) {
#pragma unroll
        for (int j = 0; j < KPA; ++j) As[buf][a_row][a_k + j] = (__bf16)ra[j];
#pragma unroll
        for (int j = 0; j < KPB; ++j) Bs[buf][b_row][b_k + j] = (__bf16)rb[j];
        __syncthreads();
        if (k0 + BK < k_end) fetch(k0 + BK);  // the next step's loads overlap this step's MFMAs
#pragma unroll
        for (int s = 0; s < BK; s += 16) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(&As[buf][wm * 32 + r][s + kh]);
            const bf16x8 b = *reinterpret_cast<const bf16x8*>(&Bs[buf][wn * 32 + r][s + kh]);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc, 0, 0, 0);
        }
        buf ^= 1;  // double buffer: the next step writes the other buffer
    }
    // epilogue: acc[v] is C[row][col], col = lane % 32,
    // row = 8*(v/4) + 4*(lane/32) + v%4 (32x32 MFMA output layout)
    const int col = lane & 31;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const int row = 8 * (v >> 2) + 4 * (lane >> 5) + (v & 3);
        const long long m = m0 + wm * 32 + row, n = n0 + wn * 32 + col;
        if (m >= M || n >= N) continue;
        float c = acc[v];
        if (MODE == kFwd) {
            if (p.bias) c += p.bias[m];
            if (p.relu && c < 0.f) c = 0.f;
        }
        if (MODE == kFwd || MODE == kBwdData) {
            const int img = (int)(n / HW), pix = (int)(n % HW);
            float* dst = p.out + ((long long)img * p.out_c + p.out_c0 + m) * HW + pix;
            if (MODE == kFwd && p.res) {
                // the mean as launch_channel_mean forms it
                const float* q = p.res + (long long)img * p.res_c * HW + pix;
                float b = q[0];
                if (p.res_c > 1) {
                    b = 0.f;
                    for (int k = 0; k < p.res_c; ++k) b += q[(long long)k * HW];
                    b = b * (1.0f / (float)p.res_c);
                }
                c = b + c;
            }
            if (p.accumulate) *dst += c; else *dst = c;
        } else if (gridDim.z > 1) {
            // this reduction slice's share of dW[co][ci][tap]; grad_finish
            // adds the slices in order (no atomics: the same sums every run)
            p.partial[(long long)blockIdx.z * M * N + m * N + n] = c;
        } else {
            p.out[m * N + n] += c;  // dW[co][ci][tap], one writer per element
        }
    }
}

// What the weight gradient of one layer needs, in a table passed by value: the
// product kernel's and grad_finish's first work-group of the layer.
struct WgradItem {
    const float *x, *g, *y;
    float *out, *partial, *db;
    long long mn;  // weights that have slices to add (0: one slice, added by the product)
    int N, Cin, Cout, H, W, relu, splits, first, finish;
};
struct WgradTable {
    WgradItem item[kMaxWgrad];
    int n;
};

// The second half of the layers' parameter gradients in one launch.  Of a
// layer's work-groups the first Cout: the bias gradient of a channel, per-thread
// sums over the pixels t, t + 256, .. and a tree.  The others: 256 weights each,
// adding the reduction slices in order.  Fixed orders: the same sums every run.
// Both are chains of additions fed by loads, so the loads run 16 and 32 ahead
// (one at a time: 13.5 and 14.6 us per layer; 8.9 together; the 15 layers of a
// training step in one launch 36 instead of 132).
__global__ __launch_bounds__(256) void grad_finish(WgradTable t) {
    int l = 0;
    while (l + 1 < t.n && (int)blockIdx.x >= t.item[l + 1].finish) ++l;
    const WgradItem& q0 = t.item[l];
    const float* const g = q0.g;
    const float* const y = q0.y;
    const float* __restrict__ part = q0.partial;
    float* const db = q0.db;
    float* const dw = q0.out;
    const int N = q0.N, C = q0.Cout, HW = q0.H * q0.W, relu = q0.relu, splits = q0.splits;
    const int nbias = db ? C : 0, block = (int)blockIdx.x - q0.finish;
    const long long mn = q0.mn;
    if (block >= nbias) {
        const long long i = (long long)(block - nbias) * 256 + threadIdx.x;
        if (i >= mn) return;
        const float* q = part + i;
        float s = 0.f;
        int z = 0;
        for (; z + 32 <= splits; z += 32, q += 32 * mn) {
            float v[32];
#pragma unroll
            for (int k = 0; k < 32; ++k) v[k] = q[k * mn];
#pragma unroll
            for (int k = 0; k < 32; ++k) s += v[k];
        }
#pragma unroll 4
        for (; z < splits; ++z, q += mn) s += *q;
        dw[i] += s;
        return;
    }
    __shared__ float red[256];
    const int c = block;
    const long long n = (long long)N * HW;
    float s = 0.f;
    for (long long i0 = threadIdx.x; i0 < n; i0 += 256 * 16) {
        long long o[16];
        float v[16], m[16];
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            const long long i = i0 + 256 * k;
            o[k] = i < n ? (i / HW * C + c) * HW + i % HW : (long long)c * HW;
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) v[k] = g[o[k]];
        if (relu) {
#pragma unroll
            for (int k = 0; k < 16; ++k) m[k] = y[o[k]];
#pragma unroll
            for (int k = 0; k < 16; ++k) v[k] = m[k] <= 0.f ? 0.f : v[k];
        }
#pragma unroll
        for (int k = 0; k < 16; ++k)
            if (i0 + 256 * k < n) s += v[k];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) db[c] = red[0];
}

// ------------------------------------------------------- 3x3 weight gradient
// wgrad3: conv_gemm's weight gradient for 3x3 layers whose rows are whole runs
// of 4 pixels.  conv_gemm gathers every (channel, tap) of a pixel as a scalar
// with its index arithmetic, about 400 instructions per thread and 32 pixels,
// and bounds on it (24 us per layer of a 32^2 training step whatever its size).
// Here a work-group owns 32 output channels x 32 input channels and all 9 taps,
// one wavefront per row of taps.  Per block of 64 pixels a thread loads 8
// pixels of a channel and their neighbours left and right as vectors, the next
// block's while this one is computed, and writes them to LDS as three bf16
// operands, one per column of taps, so that the matrix cores read whole aligned
// runs.  Slices of the reduction, the order of pixels and their places in each
// MFMA are conv_gemm's: every partial sum keeps its bits.  Per layer, us,
// conv_gemm / wgrad3 (images, input and output channels, size): 16, 96, 32, 32^2
// 34 / 19; 16, 192, 64, 16^2 44 / 17; 16, 256, 256, 4^2 18 / 13; 16, 64, 64, 64^2
// 202 / 51; 16, 128, 128, 64^2 715 / 142.  At the small sizes it is bound by
// latency (load, LDS, 3 dependent MFMAs, store), so layers share a launch: the
// 14 of a training step of 16 32^2 images 340 us with conv_gemm, 181 one by
// one, 65 together.
constexpr int kWB = 64, kWRow = kWB + 8;  // pixels per block; LDS rows of 144 bytes
typedef float f32x4 __attribute__((ext_vector_type(4)));

__global__ __launch_bounds__(192) void wgrad3(WgradTable t) {
    int l = 0;
    while (l + 1 < t.n && (int)blockIdx.x >= t.item[l + 1].first) ++l;
    const WgradItem p = t.item[l];
    __shared__ __align__(16) __bf16 tile[10][32][kWRow];
    __bf16 (*const As)[kWRow] = tile[0];
    float* const Ds = reinterpret_cast<float*>(&tile[0][0][0]);  // 32 x 288 results at the end, rows of 289
    static_assert(sizeof(tile) >= 32 * 289 * sizeof(float), "the results reuse the operands' LDS");
    const int lane = threadIdx.x & 63, ty = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);  // tap row
    // work-group: input channel tile fastest, then output channel tile, then slice
    const int ct = (p.Cin + 31) / 32, mt = (p.Cout + 31) / 32, block = (int)blockIdx.x - p.first;
    const int m0 = block / ct % mt * 32, c0 = block % ct * 32, slice = block / (ct * mt);
    const int H = p.H, W = p.W, HW = H * W, K = p.N * HW;
    const int splits = p.splits, chunk = ((K + splits - 1) / splits + BK - 1) / BK * BK;
    const int k_beg = slice * chunk, k_end = min(k_beg + chunk, K);
    const __amdgpu_buffer_rsrc_t rx = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.x), 0, p.Cin * K * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t rg = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.g), 0, p.Cout * K * 4, 0x00020000);
    const __amdgpu_buffer_rsrc_t ry =
        __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.relu ? p.y : p.g), 0, p.Cout * K * 4, 0x00020000);
    auto load4 = [](__amdgpu_buffer_rsrc_t r, unsigned o) {
        return __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(r, (int)o, 0, 0));
    };
    auto load1 = [](__amdgpu_buffer_rsrc_t r, unsigned o) {
        return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(r, (int)o, 0, 0));
    };
    // this lane's 8 pixels of a block: run lane % 8, as two halves of 4 that
    // each lie in one image row; channels lane / 8 + 8 i
    const int run = lane & 7, ch = lane >> 3;
    int k[2], px[2], py[2], pi[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        k[h] = k_beg + 8 * run + 4 * h;
        pi[h] = k[h] / HW;
        py[h] = (k[h] - pi[h] * HW) / W;
        px[h] = k[h] - pi[h] * HW - py[h] * W;
    }
    const int qw = kWB / W, rw = kWB - qw * W;
    f32x4 cx[4][2], ca[2][2], cm[2][2];
    float cl[4][2], cr[4][2];
    // loads the block at k[] and steps to the next one
    auto load = [&] {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const bool in = k[h] < k_end;
            const int y = py[h] + ty - 1;
            const bool row = in && (unsigned)y < (unsigned)H;
            const unsigned bx = (unsigned)((pi[h] * p.Cin + c0 + ch) * HW + y * W + px[h]) * 4u;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool ok = row && c0 + ch + 8 * i < p.Cin;
                const unsigned o = bx + (unsigned)(8 * i * HW) * 4u;
                cx[i][h] = load4(rx, ok ? o : 0x80000000u);
                cl[i][h] = load1(rx, ok && px[h] > 0 ? o - 4u : 0x80000000u);
                cr[i][h] = load1(rx, ok && px[h] + 4 < W ? o + 16u : 0x80000000u);
            }
            const unsigned bg = (unsigned)((pi[h] * p.Cout + m0 + ch) * HW + py[h] * W + px[h]) * 4u;
#pragma unroll
            for (int i = 0; i < 2; ++i) {  // channel groups ty and ty + 3 (of 4) of the output gradient
                const int c = ch + 8 * (ty + 3 * i);
                const bool ok = in && c < 32 && m0 + c < p.Cout;
                const unsigned o = bg + (unsigned)(8 * (ty + 3 * i) * HW) * 4u;
                ca[i][h] = load4(rg, ok ? o : 0x80000000u);
                if (p.relu) cm[i][h] = load4(ry, ok ? o : 0x80000000u);
            }
            k[h] += kWB;
            px[h] += rw;
            py[h] += qw;
            if (px[h] >= W) px[h] -= W, ++py[h];
            while (py[h] >= H) py[h] -= H, ++pi[h];
        }
    };
    f32x16 acc[3];
#pragma unroll
    for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[d][v] = 0.f;
    const int r = lane & 31, kh = (lane >> 5) * 8;
    load();
    for (int kb = k_beg; kb < k_end; kb += kWB) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            bf16x8 q[3];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    q[0][4 * h + j] = (__bf16)(j > 0 ? cx[i][h][j > 0 ? j - 1 : 0] : cl[i][h]);
                    q[1][4 * h + j] = (__bf16)cx[i][h][j];
                    q[2][4 * h + j] = (__bf16)(j < 3 ? cx[i][h][j < 3 ? j + 1 : 3] : cr[i][h]);
                }
#pragma unroll
            for (int d = 0; d < 3; ++d) *reinterpret_cast<bf16x8*>(&tile[1 + 3 * ty + d][ch + 8 * i][8 * run]) = q[d];
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (ty + 3 * i > 3) continue;
            bf16x8 q;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    q[4 * h + j] = (__bf16)(p.relu && cm[i][h][j] <= 0.f ? 0.f : ca[i][h][j]);
            *reinterpret_cast<bf16x8*>(&As[ch + 8 * (ty + 3 * i)][8 * run]) = q;
        }
        lds_barrier();
        if (kb + kWB < k_end) load();
#pragma unroll
        for (int s = 0; s < kWB; s += 16) {
            const bf16x8 a = *reinterpret_cast<const bf16x8*>(&As[r][s + kh]);
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                const bf16x8 b = *reinterpret_cast<const bf16x8*>(&tile[1 + 3 * ty + d][r][s + kh]);
                acc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, acc[d], 0, 0, 0);
            }
        }
        lds_barrier();
    }
    // the 9 taps of 32 input channels are contiguous: through LDS, so that a
    // wavefront stores whole lines
#pragma unroll
    for (int v = 0; v < 16; ++v)
#pragma unroll
        for (int d = 0; d < 3; ++d)
            Ds[(8 * (v >> 2) + 4 * (lane >> 5) + (v & 3)) * 289 + 9 * r + 3 * ty + d] = acc[d][v];
    lds_barrier();
    const int cols = 9 * min(32, p.Cin - c0);
    const long long N = 9ll * p.Cin, mn = p.Cout * N;
    for (int m = ty; m < 32 && m0 + m < p.Cout; m += 3) {
        const long long o = (m0 + m) * N + 9ll * c0;
        for (int j = lane; j < cols; j += 64) {
            const float v = Ds[m * 289 + j];
            if (splits > 1) p.partial[slice * mn + o + j] = v;
            else p.out[o + j] += v;
        }
    }
}

// ------------------------------------------------ 3x3 forward and input gradient
// conv3: the products of conv_gemm's kFwd and kBwdData for 3x3 layers with the
// operands laid out for the matrix cores.  conv_gemm gathers 8 or 16 scalars
// per thread and 32-deep K step with one step in flight, so a step costs the
// latency of a gather (1.8 us): a layer of 384 channels takes 108 of them.
// Here a step is 16 input channels, 144 of K = (channel, tap): their pixels
// with a one-pixel border are staged once in LDS (each value loaded once
// instead of 9 times), expanded there to the 9 taps of every pixel, and feed 9
// MFMAs per wavefront; the pixels and weights of the next two steps load
// meanwhile.  The weights come packed in fragment order (pack_conv3), one
// 16-byte load per lane and MFMA.  The order of K and the position of every k
// in its MFMA are conv_gemm's, so every output keeps its bits.
// Bound by the latency of a step's LDS passes and 9 dependent MFMAs on small
// images (0.8 / 1.0 / 1.2 us per step for PW 1 / 2 / 4 plus 5 us per launch)
// and by LDS reads on large ones.  The staged values are FP32: two-byte ones
// made the compiler read pairs at odd addresses, 1.4 / 2.2 / 3.9 us per step.
// One 128^2 image of the 4-level 32-channel network (15 layers): 826 us with
// conv_gemm, 353 with two-byte staging and one step in flight, 249 with FP32
// staging and two; 219 with the pooled, concatenated and upsampled copies and
// the residual written by the epilogues instead of 12 launches and 2 copies.
// Tile: PW pixel tiles of 4 x 8 pixels by 4 / PW tiles of 32 output channels,
// one wavefront each; PW = 4 / 2 / 1 for 1 / 2-3 / more channel tiles, so that
// a work-group's wavefronts share as much of the expansion as the layer allows.
constexpr int kCh = 16, kK3 = kCh * 9, kSteps = kK3 / 16, kBRow = kK3 + 8;  // rows of 304 bytes: no bank conflicts
template <int PW> struct Tile3 {
    static constexpr int PX = PW == 4 ? 2 : 1, PY = PW / PX;   // pixel tiles along x and y
    static constexpr int TW = 8 * PX, TH = 4 * PY, HX = TW + 2, HY = TH + 2;
    static constexpr int NL = (kCh * HX * HY + 255) / 256;     // staged values per thread
    // staged rows are 24 floats apart: the 4 rows of 8 pixels that a half
    // wavefront reads then lie in different banks
    static constexpr int RS = 24, PS = RS * HY;
    static constexpr int G = 4 / PW;                           // groups of wavefronts that share the expansion
};

// expands runs j = G0, G0 + G, ... of 8 k: run j + 9 h holds k = 8 (j + 9 h) ..,
// the taps of run j eight channels on, so h only moves the base address
template <int PW, int G0> __device__ __forceinline__ void expand3(const float* src, __bf16* dst) {
    using T = Tile3<PW>;
    bf16x8 v[(9 - G0 + T::G - 1) / T::G];
#pragma unroll
    for (int j = G0, i = 0; j < 9; j += T::G, ++i)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int k = 8 * j + e, c = k / 9, t = k % 9;
            v[i][e] = (__bf16)src[c * T::PS + (t / 3) * T::RS + t % 3];
        }
#pragma unroll
    for (int j = G0, i = 0; j < 9; j += T::G, ++i) *reinterpret_cast<bf16x8*>(dst + 8 * j) = v[i];
}

template <int MODE, int PW> __global__ __launch_bounds__(256) void conv3(ConvArgs p) {
    using T = Tile3<PW>;
    __shared__ float Hs[kCh * T::PS];
    __shared__ __align__(16) __bf16 Bs[32 * PW][kBRow];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int M = MODE == kFwd ? p.Cout : p.Cin, C = MODE == kFwd ? p.Cin : p.Cout;
    const int HW = p.H * p.W, nch = (C + kCh - 1) / kCh;
    const int mt = (int)blockIdx.y * T::G + wave % T::G, pt = wave / T::G;
    const bool mlive = mt * 32 < M;
    const int ntx = (p.W + T::TW - 1) / T::TW, nty = (p.H + T::TH - 1) / T::TH;
    const int img = (int)(blockIdx.x / (unsigned)(ntx * nty)), tile = (int)(blockIdx.x % (unsigned)(ntx * nty));
    const int ty0 = tile / ntx * T::TH, tx0 = tile % ntx * T::TW;
    // staged values: byte offset in the step's 16 planes (past the
    // descriptor's bound outside the image: reads zero) and place in Hs
    unsigned off[T::NL];
    int pos[T::NL];
#pragma unroll
    for (int i = 0; i < T::NL; ++i) {
        const int e = tid + 256 * i, ch = e / (T::HX * T::HY), q = e % (T::HX * T::HY);
        const int y = ty0 + q / T::HX - 1, x = tx0 + q % T::HX - 1;
        const bool in = (unsigned)y < (unsigned)p.H && (unsigned)x < (unsigned)p.W && ch < kCh;
        off[i] = in ? ((unsigned)ch * (unsigned)HW + (unsigned)(y * p.W + x)) * 4u : 0x80000000u;
        // what is left over past the last channel goes to a pad of the last row
        pos[i] = ch < kCh ? ch * T::PS + (q / T::HX) * T::RS + q % T::HX : kCh * T::PS - 1;
    }
    const float* src = (MODE == kFwd ? p.x : p.g) + (long long)img * C * HW;
    const float* msk = MODE == kBwdData && p.relu ? p.y + (long long)img * C * HW : nullptr;
    constexpr int NM = MODE == kBwdData ? T::NL : 1;
    // past the last step the loads repeat it (no branch around them)
    auto fetch = [&](int c, float(&v)[T::NL], float(&m)[NM]) {
        c = min(c, nch - 1);
        const int n = min(kCh, C - c * kCh);  // channels of this step; the planes past them read zero
        const int bytes = n * HW * 4;
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float*>(src + (long long)c * kCh * HW), 0, bytes, 0x00020000);
#pragma unroll
        for (int i = 0; i < T::NL; ++i)
            v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, (int)off[i], 0, 0));
        if constexpr (MODE == kBwdData) {
            if (msk) {
                const __amdgpu_buffer_rsrc_t rm = __builtin_amdgcn_make_buffer_rsrc(
                    const_cast<float*>(msk + (long long)c * kCh * HW), 0, bytes, 0x00020000);
#pragma unroll
                for (int i = 0; i < T::NL; ++i)
                    m[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rm, (int)off[i], 0, 0));
            }
        }
    };
    const __bf16* wp = p.pack + (long long)(mlive ? mt : 0) * nch * (kSteps * 512) + lane * 8;
    auto fetch_w = [&](int c, bf16x8(&w)[kSteps]) {
        c = min(c, nch - 1);
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
            w[s] = *reinterpret_cast<const bf16x8*>(wp + ((long long)c * kSteps + s) * 512);
    };
    // expansion: pixel and channel half of this thread
    const int epx = PW == 1 ? lane & 31 : (PW == 2 ? tid & 63 : tid & 127);
    const int eh = PW == 1 ? lane >> 5 : (PW == 2 ? (tid >> 6) & 1 : tid >> 7);
    const int eg = PW == 1 ? wave : (PW == 2 ? wave >> 1 : 0);
    const int et = epx >> 5, el = epx & 31;
    const float* esrc = Hs + eh * 8 * T::PS + (4 * (et / T::PX) + (el >> 3)) * T::RS + 8 * (et % T::PX) + (el & 7);
    __bf16* edst = &Bs[epx][eh * 72];

    f32x16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
    // one step: its pixels are in v (mask source in m), its weights in w; once
    // consumed, the registers take those of the step after next
    auto step = [&](int c, float(&v)[T::NL], float(&m)[NM], bf16x8(&w)[kSteps]) {
#pragma unroll
        for (int i = 0; i < T::NL; ++i) {
            float x = v[i];
            if constexpr (MODE == kBwdData) {
                if (msk && m[i] <= 0.f) x = 0.f;
            }
            Hs[pos[i]] = x;
        }
        fetch(c + 2, v, m);
        __builtin_amdgcn_sched_barrier(0);
        lds_barrier();
        if constexpr (PW == 4) expand3<PW, 0>(esrc, edst);
        else if constexpr (PW == 2) {
            if (eg == 0) expand3<PW, 0>(esrc, edst);
            else expand3<PW, 1>(esrc, edst);
        } else {
            if (eg == 0) expand3<PW, 0>(esrc, edst);
            else if (eg == 1) expand3<PW, 1>(esrc, edst);
            else if (eg == 2) expand3<PW, 2>(esrc, edst);
            else expand3<PW, 3>(esrc, edst);
        }
        lds_barrier();
        const __bf16* b = &Bs[pt * 32 + (lane & 31)][(lane >> 5) * 8];
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(w[s], *reinterpret_cast<const bf16x8*>(b + 16 * s), acc, 0, 0,
                                                          0);
        fetch_w(c + 2, w);
        __builtin_amdgcn_sched_barrier(0);
    };
    float v0[T::NL], v1[T::NL], m0[NM], m1[NM];
    bf16x8 w0[kSteps], w1[kSteps];
    // in the loop's issue order: the wait counters count in order, and a value
    // loaded later here than there makes the loop wait for everything
    fetch(0, v0, m0);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(0, w0);
    __builtin_amdgcn_sched_barrier(0);
    fetch(1, v1, m1);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(1, w1);
    __builtin_amdgcn_sched_barrier(0);
    for (int c = 0; c < nch; c += 2) {
        step(c, v0, m0, w0);
        if (c + 1 < nch) step(c + 1, v1, m1, w1);
    }
    // acc[i] is C[row][col], col = lane % 32 (a pixel of tile pt),
    // row = 8*(i/4) + 4*(lane/32) + i%4 (32x32 MFMA output layout).  What the
    // outputs need is loaded before the first store, dead rows from a valid
    // address: one wait instead of one per output
    const int y = ty0 + 4 * (pt / T::PX) + ((lane & 31) >> 3), x = tx0 + 8 * (pt % T::PX) + (lane & 7);
    if (y >= p.H || x >= p.W) return;  // whole 2x2 groups (an even image) or none of one
    float* const out0 = p.out + ((long long)img * p.out_c + p.out_c0) * HW + y * p.W + x;
    const int o0 = mt * 32 + 4 * (lane >> 5);
    float add[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int o = o0 + 8 * (i >> 2) + (i & 3);
        if (MODE == kFwd) add[i] = p.bias ? p.bias[min(o, M - 1)] : 0.f;
        else add[i] = p.accumulate ? out0[(long long)min(o, M - 1) * HW] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int o = o0 + 8 * (i >> 2) + (i & 3);
        float r = acc[i] + add[i];
        if (MODE == kFwd && p.relu && r < 0.f) r = 0.f;
        if constexpr (MODE == kFwd) {
            if (p.pool) {
                // the 2x2 group's values are in this lane and the lanes one
                // and eight up (8 pixels per row); lane bits 0 and 3 clear hold
                // its first pixel.  H and W are even: the group is whole
                const float s1 = __shfl_down(r, 1, 64), s2 = __shfl_down(r, 8, 64), s3 = __shfl_down(r, 9, 64);
                if (o < M && (lane & 9) == 0)
                    p.pool[((long long)img * M + o) * (HW >> 2) + (y >> 1) * (p.W >> 1) + (x >> 1)] =
                        0.25f * (r + s1 + s2 + s3);
            }
            if (p.skip && o < M) p.skip[((long long)img * p.skip_c + p.skip_c0 + o) * HW + y * p.W + x] = r;
            if (p.up && o < M) {
                float* u = p.up + ((long long)img * p.up_c + o) * (4ll * HW) + (long long)(4 * y) * p.W + 2 * x;
                const float2 rr = make_float2(r, r);
                *reinterpret_cast<float2*>(u) = rr;
                *reinterpret_cast<float2*>(u + 2 * p.W) = rr;
            }
        }
        if (o < M) out0[(long long)o * HW] = r;
    }
}

// Weights of 3x3 layers in conv3's fragment order: [tile of 32 rows m][step of
// 16 channels][MFMA][lane][8], lane = m % 32 + 32 h holding k = 16 s + 8 h ..
// of the step (zero past the layer's rows and channels).
__global__ __launch_bounds__(256) void pack_conv3(PackArgs p) {
    const PackLayer q = p.layer[blockIdx.y];
    const int nch = (q.C + kCh - 1) / kCh;
    const long long n = (long long)((q.M + 31) / 32) * nch * (kSteps * 512);
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const int j = (int)(i & 7), lane = (int)(i >> 3) & 63;
        const long long f = i >> 9;  // (tile, step, MFMA)
        const int s = (int)(f % kSteps), c = (int)(f / kSteps % nch), mt = (int)(f / kSteps / nch);
        const int m = mt * 32 + (lane & 31), k = 16 * s + 8 * (lane >> 5) + j, ch = c * kCh + k / 9, t = k % 9;
        float w = 0.f;
        if (m < q.M && ch < q.C)
            w = q.mode == kFwd ? p.w[q.w_off + ((long long)m * q.C + ch) * 9 + t]
                               : p.w[q.w_off + ((long long)ch * q.M + m) * 9 + 8 - t];
        p.out[q.out_off + i] = (__bf16)w;
    }
}

namespace {
void conv_gemm_shape(int mode, int ks, const ConvArgs& a, long long* M, long long* N, long long* K) {
    const int HW = a.H * a.W;
    if (mode == kFwd) { *M = a.Cout; *N = (long long)a.N * HW; *K = (long long)a.Cin * ks * ks; }
    else if (mode == kBwdData) { *M = a.Cin; *N = (long long)a.N * HW; *K = (long long)a.Cout * ks * ks; }
    else { *M = a.Cout; *N = (long long)a.Cin * ks * ks; *K = (long long)a.N * HW; }
}
int conv_bm(long long M) { return M <= 32 ? 32 : 64; }
// reduction slices of the weight gradient: enough work-groups to fill the
// chip, each slice at least 4 K-steps long
int wgrad_splits(long long M, long long N, long long K) {
    const int bm = conv_bm(M), bn = 4096 / bm;
    const long long tiles = ((M + bm - 1) / bm) * ((N + bn - 1) / bn);
    long long want = 2048 / (tiles > 0 ? tiles : 1);
    long long maxs = (K + 4 * BK - 1) / (4 * BK);
    int splits = (int)(want < 1 ? 1 : (want > maxs ? maxs : want));
    return splits < 1 ? 1 : splits;
}
}  // namespace

size_t conv_wgrad_scratch(int ks, const ConvArgs& a) {
    long long M, N, K;
    conv_gemm_shape(kBwdWeight, ks, a, &M, &N, &K);
    const int splits = wgrad_splits(M, N, K);
    return splits > 1 ? (size_t)splits * (size_t)(M * N) : 0;
}

size_t conv3_pack_size(int M, int C) {
    return (size_t)((M + 31) / 32) * ((C + kCh - 1) / kCh) * (kSteps * 512);
}

hipError_t launch_pack_conv3(const PackArgs& a, int layers, hipStream_t s) {
    hipLaunchKernelGGL(pack_conv3, dim3(512, layers), dim3(256), 0, s, a);
    return hipGetLastError();
}

// conv3 takes every image whose 16 planes of a step 32-bit byte offsets reach
// and whose tiles a grid holds; single-pixel images, a 32nd of its pixel
// tile, stay with conv_gemm, which tiles pixels across images.
bool conv3_fits(const ConvArgs& a) {
    const long long hw = (long long)a.H * a.W;
    return hw > 1 && hw <= (1 << 24) && a.N * ((a.H + 3LL) / 4) * ((a.W + 7LL) / 8) <= (1 << 21);
}

namespace {
// wgrad3 takes rows of whole, aligned runs of 4 pixels, in tensors that 31-bit
// byte offsets reach, and at least two blocks of pixels (68 pixels: 13.7 us with
// conv_gemm, 15.6 with wgrad3; 140: 11 and 9)
bool wgrad3_fits(const ConvArgs& a) {
    const long long px = (long long)a.N * a.H * a.W;
    const uintptr_t at = (uintptr_t)a.x | (uintptr_t)a.g | (a.relu ? (uintptr_t)a.y : 0);
    return a.W % 4 == 0 && at % 16 == 0 && px >= 2 * kWB && px * std::max(a.Cin, a.Cout) < (1LL << 29);
}

hipError_t launch_conv3(int mode, const ConvArgs& a, hipStream_t s) {
    const int mt = ((mode == kFwd ? a.Cout : a.Cin) + 31) / 32, pw = mt == 1 ? 4 : (mt <= 3 ? 2 : 1);
    const int tw = pw == 4 ? 16 : 8, th = pw == 1 ? 4 : 8, g = 4 / pw;
    const dim3 grid((unsigned)((long long)a.N * ((a.H + th - 1) / th) * ((a.W + tw - 1) / tw)), (unsigned)((mt + g - 1) / g));
#define MSX_CONV3(PW_)                                                                            \
    do {                                                                                          \
        if (mode == kFwd) hipLaunchKernelGGL((conv3<kFwd, PW_>), grid, dim3(256), 0, s, a);       \
        else hipLaunchKernelGGL((conv3<kBwdData, PW_>), grid, dim3(256), 0, s, a);                \
    } while (0)
    if (pw == 4) MSX_CONV3(4);
    else if (pw == 2) MSX_CONV3(2);
    else MSX_CONV3(1);
#undef MSX_CONV3
    return hipGetLastError();
}
}  // namespace

namespace {
hipError_t launch_conv_gemm(int mode, int ks, const ConvArgs& a, int splits, hipStream_t s) {
    long long M, N, K;
    conv_gemm_shape(mode, ks, a, &M, &N, &K);
    const int bm = conv_bm(M), bn = 4096 / bm;
    dim3 grid((unsigned)((N + bn - 1) / bn), (unsigned)((M + bm - 1) / bm), (unsigned)splits);
#define MSX_CONV(MODE_, KS_, BM_) hipLaunchKernelGGL((conv_gemm<MODE_, KS_, BM_>), grid, dim3(256), 0, s, a)
#define MSX_CONV_BM(MODE_, KS_)                    \
    do {                                           \
        if (bm == 32) MSX_CONV(MODE_, KS_, 32);    \
        else MSX_CONV(MODE_, KS_, 64);             \
    } while (0)
    if (ks == 3) {
        if (mode == kFwd) MSX_CONV_BM(kFwd, 3);
        else if (mode == kBwdData) MSX_CONV_BM(kBwdData, 3);
        else MSX_CONV_BM(kBwdWeight, 3);
    } else if (ks == 1) {
        if (mode == kFwd) MSX_CONV_BM(kFwd, 1);
        else if (mode == kBwdData) MSX_CONV_BM(kBwdData, 1);
        else MSX_CONV_BM(kBwdWeight, 1);
    } else {
        return hipErrorInvalidValue;
    }
#undef MSX_CONV_BM
#undef MSX_CONV
    return hipGetLastError();
}
}  // namespace

hipError_t launch_conv(int mode, int ks, const ConvArgs& a, hipStream_t s) {
    if (mode == kBwdWeight) return hipErrorInvalidValue;
    if (a.pack) return launch_conv3(mode, a, s);
    return launch_conv_gemm(mode, ks, a, 1, s);
}

hipError_t launch_wgrad(const WgradLayer* layers, int n, hipStream_t s) {
    if (n < 0 || n > kMaxWgrad) return hipErrorInvalidValue;
    WgradTable prod{}, fin{};
    int nprod = 0, nfin = 0;  // work-groups
    for (int i = 0; i < n; ++i) {
        const ConvArgs& a = layers[i].a;
        long long M, N, K;
        conv_gemm_shape(kBwdWeight, layers[i].ks, a, &M, &N, &K);
        const int splits = wgrad_splits(M, N, K);
        if (splits > 1 && !a.partial) return hipErrorInvalidValue;
        WgradItem q{a.x, a.g, a.y, a.out, a.partial, a.db, splits > 1 ? M * N : 0, a.N, a.Cin, a.Cout, a.H, a.W, a.relu,
                    splits, nprod, nfin};
        if (layers[i].ks == 3 && wgrad3_fits(a)) {
            nprod += ((a.Cout + 31) / 32) * ((a.Cin + 31) / 32) * splits;
            prod.item[prod.n++] = q;
        } else {
            const hipError_t e = launch_conv_gemm(kBwdWeight, layers[i].ks, a, splits, s);
            if (e != hipSuccess) return e;
        }
        if (splits > 1 || a.db) {
            nfin += (a.db ? a.Cout : 0) + (int)((q.mn + 255) / 256);
            fin.item[fin.n++] = q;
        }
    }
    if (prod.n) hipLaunchKernelGGL(wgrad3, dim3((unsigned)nprod), dim3(192), 0, s, prod);
    if (fin.n) hipLaunchKernelGGL(grad_finish, dim3((unsigned)nfin), dim3(256), 0, s, fin);
    return hipGetLastError();
}

// ------------------------------------------------------------------ small ops
__global__ void avgpool2_fwd(const float* x, float* y, long long nc, int H, int W) {
    const int Ho = H / 2, Wo = W / 2;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nc * Ho * Wo) return;
    const long long c = i / (Ho * Wo);
    const int pix = (int)(i % (Ho * Wo)), yo = pix / Wo, xo = pix % Wo;
    const float* s = x + c * H * W + (2 * yo) * W + 2 * xo;
    y[i] = 0.25f * (s[0] + s[1] + s[W] + s[W + 1]);
}
__global__ void avgpool2_bwd(const float* gy, float* gx, long long nc, int H, int W) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nc * H * W) return;
    const long long c = i / (H * W);
    const int pix = (int)(i % (H * W)), y = pix / W, x = pix % W;
    gx[i] += 0.25f * gy[(c * (H / 2) + y / 2) * (W / 2) + x / 2];
}
// nearest-neighbour x2 upsampling into channels [c0, c0+C) of a tensor with Ct channels
__global__ void upsample2_fwd(const float* x, float* y, int N, int C, int H, int W, int Ct, int c0) {
    const long long tot = (long long)N * C * 4 * H * W;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= tot) return;
    const int Wo = 2 * W, Ho = 2 * H;
    const int xo = (int)(i % Wo), yo = (int)((i / Wo) % Ho);
    const long long nc = i / ((long long)Wo * Ho);
    const int n = (int)(nc / C), c = (int)(nc % C);
    y[(((long long)n * Ct + c0 + c) * Ho + yo) * Wo + xo] = x[((long long)nc * H + yo / 2) * W + xo / 2];
}
// gradient of a concatenation [upsampled (C1) | skip (C2)] of 2H x 2W images:
// gup[n, c] += the sums over 2x2 of the first C1 channels, gskip += the others
__global__ void cat_bwd(const float* g, float* gup, int C1, float* gskip, int C2, int N, int H, int W) {
    const long long t1 = (long long)N * C1 * H * W, t2 = (long long)N * C2 * 4 * H * W;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const int Wo = 2 * W, Ct = C1 + C2;
    if (i < t1) {
        const int x = (int)(i % W), y = (int)((i / W) % H);
        const long long nc = i / ((long long)W * H);
        const int n = (int)(nc / C1), c = (int)(nc % C1);
        const float* s = g + (((long long)n * Ct + c) * 2 * H + 2 * y) * Wo + 2 * x;
        gup[i] += s[0] + s[1] + s[Wo] + s[Wo + 1];
    } else if (i < t1 + t2) {
        const long long j = i - t1, HW = 4LL * H * W, nc = j / HW;
        const int n = (int)(nc / C2), c = (int)(nc % C2);
        gskip[j] += g[((long long)n * Ct + C1 + c) * HW + j % HW];
    }
}
// copy channels: dst[n, d0 + c] = src[n, s0 + c], c < C
__global__ void copy_channels(const float* src, int Cs, int s0, float* dst, int Cd, int d0, int N, int C, int HW) {
    const long long tot = (long long)N * C * HW;
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= tot) return;
    const int pix = (int)(i % HW);
    const long long nc = i / HW;
    const int n = (int)(nc / C), c = (int)(nc % C);
    dst[((long long)n * Cd + d0 + c) * HW + pix] = src[((long long)n * Cs + s0 + c) * HW + pix];
}
__global__ void channel_mean(const float* x, float* y, int C, long long HW, long long n) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const long long b = i / HW, p = i % HW;
    const float* q = x + b * C * HW + p;
    float s = 0.f;
    for (int c = 0; c < C; ++c) s += q[c * HW];
    y[i] = s * (1.0f / (float)C);
}
// residual output o = in + z, MSE loss gradient g = 2 (o - t) / count (scale =
// 2 / count), and per-block partial sums of (o - t)^2 in FP64 (fixed order:
// deterministic loss)
__global__ __launch_bounds__(256) void residual_loss(const float* in, const float* z, const float* t, float* g,
                                                     long long n, float scale, double* partial) {
    __shared__ double red[256];
    double s = 0.0;
    for (long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)gridDim.x * 256) {
        const float o = in[i] + z[i], ti = t[i];
        g[i] = scale * (o - ti);
        const double d = (double)o - (double)ti;
        s += d * d;
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = red[0];
}
// clears a (na floats) and b (nb of four, 16-byte aligned)
__global__ __launch_bounds__(256) void clear_two(float* a, long long na, float4* b, long long nb) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < nb) b[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    else if (i < nb + na) a[i - nb] = 0.f;
}
// Adam (Kingma & Ba 2015), bias-corrected
__global__ void adam_step(float* w, const float* gw, float* m, float* v, long long n, float lr, float b1, float b2,
                          float eps, float c1, float c2) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float g = gw[i];
    const float mi = b1 * m[i] + (1.f - b1) * g;
    const float vi = b2 * v[i] + (1.f - b2) * g * g;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
}

#define MSX_GRID(n) dim3((unsigned)(((n) + 255) / 256)), dim3(256), 0, s
hipError_t launch_avgpool_fwd(const float* x, float* y, long long nc, int H, int W, hipStream_t s) {
    hipLaunchKernelGGL(avgpool2_fwd, MSX_GRID(nc * (H / 2) * (W / 2)), x, y, nc, H, W);
    return hipGetLastError();
}
hipError_t launch_avgpool_bwd(const float* gy, float* gx, long long nc, int H, int W, hipStream_t s) {
    hipLaunchKernelGGL(avgpool2_bwd, MSX_GRID(nc * H * W), gy, gx, nc, H, W);
    return hipGetLastError();
}
hipError_t launch_upsample_fwd(const float* x, float* y, int N, int C, int H, int W, int Ct, int c0, hipStream_t s) {
    hipLaunchKernelGGL(upsample2_fwd, MSX_GRID((long long)N * C * 4 * H * W), x, y, N, C, H, W, Ct, c0);
    return hipGetLastError();
}
hipError_t launch_cat_bwd(const float* g, float* gup, int C1, float* gskip, int C2, int N, int H, int W,
                          hipStream_t s) {
    hipLaunchKernelGGL(cat_bwd, MSX_GRID((long long)N * (C1 + 4LL * C2) * H * W), g, gup, C1, gskip, C2, N, H, W);
    return hipGetLastError();
}
hipError_t launch_copy_channels(const float* src, int Cs, int s0, float* dst, int Cd, int d0, int N, int C, int HW,
                                hipStream_t s) {
    hipLaunchKernelGGL(copy_channels, MSX_GRID((long long)N * C * HW), src, Cs, s0, dst, Cd, d0, N, C, HW);
    return hipGetLastError();
}
hipError_t launch_channel_mean(const float* x, float* y, int N, int C, long long HW, hipStream_t s) {
    const long long n = (long long)N * HW;
    hipLaunchKernelGGL(channel_mean, MSX_GRID(n), x, y, C, HW, n);
    return hipGetLastError();
}
hipError_t launch_residual_loss(const float* in, const float* z, const float* t, float* g, long long n, float scale,
                                double* partial, int nblocks, hipStream_t s) {
    hipLaunchKernelGGL(residual_loss, dim3(nblocks), dim3(256), 0, s, in, z, t, g, n, scale, partial);
    return hipGetLastError();
}
hipError_t launch_clear(float* a, long long na, float* b, long long nb, hipStream_t s) {
    hipLaunchKernelGGL(clear_two, MSX_GRID(nb / 4 + na), a, na, reinterpret_cast<float4*>(b), nb / 4);
    return hipGetLastError();
}
hipError_t launch_adam(float* w, const float* gw, float* m, float* v, long long n, float lr, float b1, float b2,
                       float eps, float c1, float c2, hipStream_t s) {
    hipLaunchKernelGGL(adam_step, MSX_GRID(n), w, gw, m, v, n, lr, b1, b2, eps, c1, c2);
    return hipGetLastError();
}
#undef MSX_GRID

}  // namespace unet
}  // namespace msx
