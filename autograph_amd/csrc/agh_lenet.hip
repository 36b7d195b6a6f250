// The LeNet5 of the reference's benchmark (benches/neural-network-benches/src/autograph_backend.rs:70-162): inference in one
// launch, and the launches of its training step.
#include <cstddef>
#include <type_traits>

#include "agh_internal.h"

using namespace agh;

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// ---- LeNet5 inference in one launch ----
//
// The model of the reference's benchmark (benches/neural-network-benches/src/
// autograph_backend.rs:88-162): conv 1->6 5x5, relu, pool 2x2, conv 6->16 5x5, relu, pool 2x2,
// flatten, dense 256->128, relu, dense 128->84, relu, dense 84->10 + bias.  At batch 1000 the
// whole forward pass is 0.57 GFLOP; run layer by layer it is bound by launch latency and by
// round trips of tiny activations through HBM.  Here a workgroup takes IMGS images through all
// twelve layers with every activation in LDS: the two conv+relu+pool stages use the same
// row-tiled inner loop as conv2_rowtile_kernel, the Dense stages are LDS-broadcast dot products
// against weights read (coalesced) from L2.  Activations are rounded to T after every layer,
// exactly where the layer-by-layer path rounds, so both paths agree per layer up to f32
// summation order.
template <int FW, int OCT, int WT>
__device__ __forceinline__ void rowpair_conv(const float *xi, int ch_sz, int pitch, int ic, int fh, const float *wg,
                                             int ocpad, float (&acc)[2][WT][OCT]) {
    constexpr int XW = WT + FW - 1, XV = (XW + 3) / 4;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int t = 0; t < WT; ++t)
#pragma unroll
            for (int o = 0; o < OCT; ++o) acc[a][t][o] = 0.0f;
    for (int ci = 0; ci < ic; ++ci) {
        const float *xc = xi + ci * ch_sz;
        const float *wc = wg + (size_t)ci * fh * FW * ocpad;
        for (int r = 0; r < fh + 1; ++r) {
            float xin[XV * 4];
#pragma unroll
            for (int v = 0; v < XV; ++v) {
                const float4 q = *(const float4 *)(xc + r * pitch + 4 * v);
                xin[4 * v + 0] = q.x; xin[4 * v + 1] = q.y; xin[4 * v + 2] = q.z; xin[4 * v + 3] = q.w;
            }
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                const int fi = r - a;
                if (fi >= 0 && fi < fh) {
                    const float *wr = wc + fi * FW * ocpad;
#pragma unroll
                    for (int fj = 0; fj < FW; ++fj) {
                        float wv[OCT];
#pragma unroll
                        for (int o = 0; o < OCT; ++o) wv[o] = wr[fj * ocpad + o];
#pragma unroll
                        for (int t = 0; t < WT; ++t)
#pragma unroll
                            for (int o = 0; o < OCT; ++o) acc[a][t][o] = __builtin_fmaf(xin[t + fj], wv[o], acc[a][t][o]);
                    }
                }
            }
        }
    }
}

// relu + first-strict-maximum pooling of window j of a row pair, rounding to T first
template <typename T, int OCT, int WT>
__device__ __forceinline__ float relu_pool_window(const float (&acc)[2][WT][OCT], int j, int o) {
    const T zero = Elem<T>::zero();
    T m = round_bias_relu<T>(acc[0][2 * j][o], false, zero, AGH_ACT_RELU);
    float mf = Elem<T>::to_f32(m);
    const T v1 = round_bias_relu<T>(acc[0][2 * j + 1][o], false, zero, AGH_ACT_RELU);
    const T v2 = round_bias_relu<T>(acc[1][2 * j][o], false, zero, AGH_ACT_RELU);
    const T v3 = round_bias_relu<T>(acc[1][2 * j + 1][o], false, zero, AGH_ACT_RELU);
    float f = Elem<T>::to_f32(v1);
    if (f > mf) mf = f;
    f = Elem<T>::to_f32(v2);
    if (f > mf) mf = f;
    f = Elem<T>::to_f32(v3);
    if (f > mf) mf = f;
    return mf;  // activations stay in LDS as f32 copies of the T values
}

// What a training step needs from the forward pass besides the logits (all [bs, ...] in standard layout): the
// convolution outputs before the relu (c1 [6,24,24], c2 [16,8,8]), the pooled activations (p1 [6,12,12], p2 [16,4,4]),
// and the dense layers' outputs before (d1 [128], d2 [84]) and after (a1, a2) the relu.
template <typename T>
struct LenetSaves {
    T *c1, *p1, *c2, *p2, *d1, *a1, *d2, *a2;
};

// N consecutive activations (N * sizeof(T) a multiple of 4 bytes, destination aligned to that size) rounded to T and
// stored with the widest vector stores
template <typename T, int N>
__device__ __forceinline__ void store_rounded(T *dst, const float (&v)[N]) {
    if constexpr (sizeof(T) == 4) {
        if constexpr (N % 4 == 0) {
#pragma unroll
            for (int i = 0; i < N; i += 4) *(float4 *)((float *)dst + i) = make_float4(v[i], v[i + 1], v[i + 2], v[i + 3]);
        } else {
#pragma unroll
            for (int i = 0; i < N; i += 2) *(float2 *)((float *)dst + i) = make_float2(v[i], v[i + 1]);
        }
    } else {
        uint32_t w[N / 2];
#pragma unroll
        for (int i = 0; i < N / 2; ++i) w[i] = f32x2_to_bf16x2(v[2 * i], v[2 * i + 1]);
        if constexpr (N == 8) *(uint4 *)dst = make_uint4(w[0], w[1], w[2], w[3]);
        else if constexpr (N == 4) *(uint2 *)dst = make_uint2(w[0], w[1]);
        else *(uint32_t *)dst = w[0];
    }
}

// 16 bytes per lane from global memory straight into LDS: lane L's data lands at lds_base + 16 L (lds_base is
// wave-uniform and travels in M0).  Inline assembly, so the compiler's wait counting does not know it: whoever reads
// the destination waits with s_waitcnt vmcnt(0) and a barrier first.
__device__ __forceinline__ void lds_direct_load16(const void *gptr, uint32_t lds_base_uniform) {
    asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off"
                 :
                 : "v"(gptr), "s"(__builtin_amdgcn_readfirstlane((int)lds_base_uniform))
                 : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_address_of(const void *p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char *)p;
}

// waves_per_eu: eight waves per workgroup are two per SIMD, four where two workgroups of one image share a CU; without the hint the
// compiler aimed the bf16 training instantiation at 128 registers and gave up the early weight loads for it (30 us
// instead of 20)
// IMGS images per workgroup.  4: a batch of a thousand is one round of 250 workgroups.  1 (batches up to 256, e.g. the
// training step's hundred): the same 512 threads share ONE image, every stage cut finer (conv1 in 2 x 4 register tiles,
// conv2's taps split between two waves per pooled row), so that a stage takes a quarter of the time: the launch is a
// chain of stage latencies, and with four images per workgroup a small batch would leave most of the chip idle while
// each busy CU walks four images' worth of every stage.
template <typename T, int IMGS>
struct LenetForwardLds {
    __align__(16) float xs[IMGS * 28 * 28];     // input images, pitch 28
    __align__(16) float w1s[25 * 6];            // [tap][oc]
    __align__(16) float p1[IMGS * 6 * 12 * 12]; // after conv1 + relu + pool
    __align__(16) float w2s[160 * 16];          // [ci][fi][fj][oc], ten rows of zeros behind the 150 taps
    int tap2[160];                              // byte offset of tap k inside an image of p1 (0 behind the taps)
    __align__(16) float p2[IMGS * 256];         // after conv2 + relu + pool, flattened [c][h][w]
    __align__(16) float d1[IMGS * 128];
    __align__(16) float d2[IMGS * 84];
    __align__(16) float parts[16 * IMGS * 128];  // dense1 partial sums
    __align__(16) T wd2s[128 * 84];              // dense2 / dense3 weights as they lie in memory
    __align__(16) T wd3s[1024];                  // (84 * 10, rounded up to whole KB)
};
// What the backward half of the same launch reads in place of the saved copies: the dense layers' outputs before the relu and the logits
struct LenetStepLds {
    float pre1[128], pre2[84], lg[10];
};

// `conv_done` runs behind the barrier after which both convolutions' outputs are saved; `step` (one image a workgroup) is filled if not null
// WHOLE: with one image a workgroup, conv2's sums over all taps in one chain, as four images a workgroup have them (a batch above 256 then
// gives the same bits either way)
template <typename T, bool SAVE, int IMGS, bool WHOLE, typename F>
__device__ __forceinline__ void lenet5_forward_body(LenetForwardLds<T, IMGS> &s, const T *__restrict__ x, const T *__restrict__ w1,
                                                    const T *__restrict__ w2, const T *__restrict__ wd1, const T *__restrict__ wd2,
                                                    const T *__restrict__ wd3, const T *__restrict__ b3, T *__restrict__ out, int bs,
                                                    LenetSaves<T> sv, int w23_aligned, LenetStepLds *step, float4 (&wreg)[16], F &&conv_done) {
    static_assert(IMGS == 1 || IMGS == 4, "one image or four per workgroup");
    float *const xs = s.xs, *const w1s = s.w1s, *const p1 = s.p1, *const w2s = s.w2s, *const p2 = s.p2, *const d1 = s.d1, *const d2 = s.d2,
                 *const parts = s.parts;
    int *const tap2 = s.tap2;
    T *const wd2s = s.wd2s, *const wd3s = s.wd3s;
    constexpr int NT = 512;  // 8 waves: two per SIMD, so one can wait on LDS while the other multiplies
    constexpr int kD3Off = 4 * IMGS * 84;  // dense3's partial sums in `parts`, behind dense2's
    const int tid = threadIdx.x;
    const int b0 = blockIdx.x * IMGS;
    const int nimg = min(IMGS, bs - b0);

    // Everything staged is read first and stored afterwards, so that the reads are all in flight together: written as
    // `lds[e] = global[...]` loops they compile to one read, one wait and one store per trip (a dozen memory round trips
    // one after another, 3 of the launch's 16 us).  Addresses are clamped, what lies outside is stored as zero.
    {
        constexpr int XU = (IMGS * 784 + NT - 1) / NT;  // 7 image values a thread
        const int nx = nimg * 784;
        T w1v, w2v[5], xv[XU];
        {
            const int e = min(tid, 149), tap = e / 6, o = e - tap * 6;
            w1v = w1[o * 25 + tap];
        }
#pragma unroll
        for (int u = 0; u < 5; ++u) {
            const int e = tid + u * NT, tap = e >> 4, o = e & 15;
            w2v[u] = w2[o * 150 + min(tap, 149)];
        }
        const T *xb = x + (size_t)b0 * 784;
#pragma unroll
        for (int u = 0; u < XU; ++u) xv[u] = xb[min(tid + u * NT, nx - 1)];
        // (widened plainly: all of it is only ever multiplied, which quiets a signalling NaN by itself)
        if (tid < 150) w1s[tid] = Elem<T>::raw(w1v);
#pragma unroll
        for (int u = 0; u < 5; ++u) {
            const int e = tid + u * NT;
            w2s[e] = (e >> 4) < 150 ? Elem<T>::raw(w2v[u]) : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < XU; ++u) {
            const int e = tid + u * NT;
            if (e < IMGS * 784) xs[e] = e < nx ? Elem<T>::raw(xv[u]) : 0.0f;
        }
    }
    if (tid < 160) {
        const int k = min(tid, 149), ci = k / 25, rem = k - ci * 25, fi = rem / 5, fj = rem - fi * 5;
        tap2[tid] = tid < 150 ? (ci * 144 + fi * 12 + fj) * 4 : 0;
    }
    // dense1 weights of this thread (see the dense1 stage below), requested now, used much later
    {
        const int cg = tid & 31, kg = tid >> 5;
#pragma unroll
        for (int kk = 0; kk < 16; ++kk) {
            const T *src = wd1 + (size_t)(kg * 16 + kk) * 128 + cg * 4;
            if constexpr (sizeof(T) == 4) {
                wreg[kk] = *(const float4 *)src;
            } else {
                const uint2 raw = *(const uint2 *)src;
                wreg[kk] = make_float4(__uint_as_float(raw.x << 16), __uint_as_float(raw.x & 0xFFFF0000u), __uint_as_float(raw.y << 16),
                                       __uint_as_float(raw.y & 0xFFFF0000u));
            }
        }
    }
    // The weights of the last two dense layers travel into LDS behind everything requested so far, 1 KB per
    // instruction without passing through registers, while the convolution stages run: read where they are used
    // (130 loads per thread, each waiting on L2) they cost the launch 3 of its 16 us.
    {
        constexpr int kW2Bytes = 128 * 84 * (int)sizeof(T), kW3Bytes = 84 * 10 * (int)sizeof(T);
        static_assert(kW2Bytes % 1024 == 0 && kW3Bytes % 16 == 0, "whole direct loads");
        const int lane = tid & 63, wave = tid >> 6;
        if (w23_aligned) {
            for (int c = wave; c < kW2Bytes / 1024; c += NT / 64)
                lds_direct_load16((const char *)wd2 + c * 1024 + lane * 16, lds_address_of(wd2s) + c * 1024);
            for (int c = wave; c < (kW3Bytes + 1023) / 1024; c += NT / 64)
                lds_direct_load16((const char *)wd3 + min(c * 1024 + lane * 16, kW3Bytes - 16), lds_address_of(wd3s) + c * 1024);
        } else {  // views at odd offsets: element copies
            for (int e = tid; e < 128 * 84; e += NT) wd2s[e] = wd2[e];
            for (int e = tid; e < 840; e += NT) wd3s[e] = wd3[e];
        }
    }
    __syncthreads();

    // conv1 (1->6, 5x5) + relu + pool
    if constexpr (IMGS == 1) {
        // items = 6 channels x 12 row pairs x 6 column blocks of 4
        if (tid < 432) {
            const int oc = tid / 72, r1 = tid - oc * 72, row = r1 / 6, wb = r1 - row * 6;
            float acc[2][4][1];
            rowpair_conv<5, 1, 4>(xs + 2 * row * 28 + wb * 4, 784, 28, 1, 5, w1s + oc, 6, acc);
#pragma unroll
            for (int j = 0; j < 2; ++j) p1[(oc * 12 + row) * 12 + wb * 2 + j] = relu_pool_window<T, 1, 4>(acc, j, 0);
            if constexpr (SAVE) {
                const size_t plane = (size_t)b0 * 6 + oc;
#pragma unroll
                for (int a = 0; a < 2; ++a) {
                    float v[4];
#pragma unroll
                    for (int t = 0; t < 4; ++t) v[t] = acc[a][t][0];
                    store_rounded<T, 4>(sv.c1 + (plane * 24 + 2 * row + a) * 24 + wb * 4, v);
                }
                const float q[2] = {p1[(oc * 12 + row) * 12 + wb * 2], p1[(oc * 12 + row) * 12 + wb * 2 + 1]};
                store_rounded<T, 2>(sv.p1 + (plane * 12 + row) * 12 + wb * 2, q);
            }
        }
    } else if (tid < IMGS * 108) {  // items = img x 3 channel pairs x 12 row pairs x 3 column blocks of 8
        const int img = tid / 108, r0 = tid - img * 108;
        const int grp = r0 / 36, r1 = r0 - grp * 36;
        const int row = r1 / 3, wb = r1 - row * 3;
        float acc[2][8][2];
        rowpair_conv<5, 2, 8>(xs + img * 784 + 2 * row * 28 + wb * 8, 784, 28, 1, 5, w1s + grp * 2, 6, acc);
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
            for (int j = 0; j < 4; ++j)
                p1[((img * 6 + grp * 2 + o) * 12 + row) * 12 + wb * 4 + j] = relu_pool_window<T, 2, 8>(acc, j, o);
        if constexpr (SAVE) {
            if (img < nimg) {
#pragma unroll
                for (int o = 0; o < 2; ++o) {
                    const size_t plane = (size_t)(b0 + img) * 6 + grp * 2 + o;
#pragma unroll
                    for (int a = 0; a < 2; ++a) {
                        float v[8];
#pragma unroll
                        for (int t = 0; t < 8; ++t) v[t] = acc[a][t][o];
                        store_rounded<T, 8>(sv.c1 + (plane * 24 + 2 * row + a) * 24 + wb * 8, v);
                    }
                    float q[4];
#pragma unroll
                    for (int j = 0; j < 4; ++j) q[j] = p1[((img * 6 + grp * 2 + o) * 12 + row) * 12 + wb * 4 + j];
                    store_rounded<T, 4>(sv.p1 + (plane * 12 + row) * 12 + wb * 4, q);
                }
            }
        }
    }
    __syncthreads();

    // conv2 (6->16, 5x5) + relu + pool on v_mfma_f32_16x16x4_f32, as conv2_small_mfma_kernel does it: an MFMA takes the
    // 4 pool windows of one pooled row (16 positions, cell-minor) x 16 channels x 4 taps, the A operand gathered from
    // p1 through the tap table.  Wave w: image w / 2, pooled rows 2 (w % 2) and 2 (w % 2) + 1; 40 steps of 4 taps.
    if constexpr (IMGS == 1) {
        // one image: wave w takes pooled row w % 4 and half w / 4 of the 40 steps; the halves are added through LDS
        const int lane = tid & 63, wave = tid >> 6, g = lane >> 4, i = lane & 15;
        const int row = wave & 3, kh = wave >> 2;
        const char *abase = (const char *)(p1 + (2 * row + ((i >> 1) & 1)) * 12 + 2 * (i >> 2) + (i & 1));
        const char *Bl = (const char *)(w2s + lane) + kh * 20 * 256, *tl = (const char *)(tap2 + g) + kh * 20 * 16;
        f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
        f32x4_t *xch = (f32x4_t *)parts;  // free until dense1
#pragma unroll
        for (int part = 0; part < (WHOLE ? 2 : 1); ++part) {
            if (WHOLE && kh == 1) break;  // (waves 0 to 3 take the second half too)
            float bq[20];
            int tq[20];
#pragma unroll
            for (int q = 0; q < 20; ++q) {
                bq[q] = *(const float *)(Bl + (part * 20 + q) * 256);
                tq[q] = *(const int *)(tl + (part * 20 + q) * 16);
            }
#pragma unroll
            for (int q = 0; q < 20; ++q) {
                float a = *(const float *)(abase + tq[q]);
                if (4 * ((WHOLE ? part : kh) * 20 + q) + g >= 150) a = 0.0f;  // behind the taps: zero times zero, whatever p1 holds
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bq[q], acc, 0, 0, 0);
            }
        }
        if (!WHOLE && kh == 1) xch[row * 64 + lane] = acc;
        if (!WHOLE) __syncthreads();
        if (kh == 0) {
            if (!WHOLE) acc += xch[row * 64 + lane];
            const T zero = Elem<T>::zero();
            float mf = Elem<T>::to_f32(round_bias_relu<T>(acc[0], false, zero, AGH_ACT_RELU));
#pragma unroll
            for (int r = 1; r < 4; ++r) {
                const float f = Elem<T>::to_f32(round_bias_relu<T>(acc[r], false, zero, AGH_ACT_RELU));
                if (f > mf) mf = f;
            }
            p2[(i * 4 + row) * 4 + g] = mf;
            if constexpr (SAVE) {
                const size_t plane = (size_t)b0 * 16 + i;
#pragma unroll
                for (int dy = 0; dy < 2; ++dy) {
                    const float v[2] = {acc[2 * dy], acc[2 * dy + 1]};
                    store_rounded<T, 2>(sv.c2 + (plane * 8 + 2 * row + dy) * 8 + 2 * g, v);
                }
                sv.p2[(plane * 4 + row) * 4 + g] = Elem<T>::from_f32(mf);
            }
        }
    } else
    {
        const int lane = tid & 63, wave = tid >> 6, g = lane >> 4, i = lane & 15;
        const int img = wave >> 1, tile0 = (wave & 1) * 2;
        const char *abase[2];
#pragma unroll
        for (int t = 0; t < 2; ++t)
            abase[t] = (const char *)(p1 + img * 864 + (2 * (tile0 + t) + ((i >> 1) & 1)) * 12 + 2 * (i >> 2) + (i & 1));
        const char *Bl = (const char *)(w2s + lane), *tl = (const char *)(tap2 + g);
        f32x4_t acc[2] = {f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}, f32x4_t{0.0f, 0.0f, 0.0f, 0.0f}};
        float bq[8];
        int tq[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            bq[q] = *(const float *)(Bl + q * 256);
            tq[q] = *(const int *)(tl + q * 16);
        }
#pragma unroll
        for (int s0 = 0; s0 < 40; s0 += 8) {
            float bc[8];
            int tc[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) { bc[q] = bq[q]; tc[q] = tq[q]; }
            if (s0 + 8 < 40) {
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    bq[q] = *(const float *)(Bl + (s0 + 8 + q) * 256);
                    tq[q] = *(const int *)(tl + (s0 + 8 + q) * 16);
                }
            }
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    float a = *(const float *)(abase[t] + tc[q]);
                    if (4 * (s0 + q) + g >= 150) a = 0.0f;  // behind the taps: zero times zero, whatever p1 holds (s0, q constants)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bc[q], acc[t], 0, 0, 0);
                }
        }
        // lane (g, i): channel i, pooled column g; acc[t][2 dy + dx] is cell (dy, dx) of the window in pooled row tile0 + t
        const T zero = Elem<T>::zero();
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const int row = tile0 + t;
            float mf = Elem<T>::to_f32(round_bias_relu<T>(acc[t][0], false, zero, AGH_ACT_RELU));
#pragma unroll
            for (int r = 1; r < 4; ++r) {
                const float f = Elem<T>::to_f32(round_bias_relu<T>(acc[t][r], false, zero, AGH_ACT_RELU));
                if (f > mf) mf = f;
            }
            p2[img * 256 + (i * 4 + row) * 4 + g] = mf;
            if constexpr (SAVE) {
                if (img < nimg) {
                    const size_t plane = (size_t)(b0 + img) * 16 + i;
#pragma unroll
                    for (int dy = 0; dy < 2; ++dy) {
                        const float v[2] = {acc[t][2 * dy], acc[t][2 * dy + 1]};
                        store_rounded<T, 2>(sv.c2 + (plane * 8 + 2 * row + dy) * 8 + 2 * g, v);
                    }
                    sv.p2[(plane * 4 + row) * 4 + g] = Elem<T>::from_f32(mf);
                }
            }
        }
    }
    __syncthreads();
    conv_done();

    // dense1 256 -> 128 + relu.  Thread (cg, kg) owns the weights W1[16kg .. 16kg+15][4cg .. 4cg+3]; they
    // were fetched into registers at the top of the kernel (16 coalesced 16-byte loads per thread, in
    // flight during both convolution stages).  Each thread forms its 4 columns x 4 images partial sums
    // over its 16 k, the 16 k-groups are then added through LDS in a fixed order.
    {
        const int cg = tid & 31, kg = tid >> 5;
        float part[IMGS][4];
#pragma unroll
        for (int r = 0; r < IMGS; ++r)
#pragma unroll
            for (int c = 0; c < 4; ++c) part[r][c] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < 16; kk += 4) {
            float4 xv[IMGS];
#pragma unroll
            for (int r = 0; r < IMGS; ++r) xv[r] = *(const float4 *)(p2 + r * 256 + kg * 16 + kk);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float4 wv = wreg[kk + u];
#pragma unroll
                for (int r = 0; r < IMGS; ++r) {
                    const float xk = u == 0 ? xv[r].x : u == 1 ? xv[r].y : u == 2 ? xv[r].z : xv[r].w;
                    part[r][0] = __builtin_fmaf(xk, wv.x, part[r][0]);
                    part[r][1] = __builtin_fmaf(xk, wv.y, part[r][1]);
                    part[r][2] = __builtin_fmaf(xk, wv.z, part[r][2]);
                    part[r][3] = __builtin_fmaf(xk, wv.w, part[r][3]);
                }
            }
        }
        // xs and p1 are free by now: the [kg][img][128] partials (16*4*128 floats = 32 KB) do not fit xs
        // alone, so they go to a buffer of their own
#pragma unroll
        for (int r = 0; r < IMGS; ++r)
            *(float4 *)(parts + (kg * IMGS + r) * 128 + cg * 4) = make_float4(part[r][0], part[r][1], part[r][2], part[r][3]);
    }
    __syncthreads();
    if (tid < IMGS * 128) {
        const int o = tid;
        float a = 0.0f;
#pragma unroll
        for (int kg = 0; kg < 16; ++kg) a += parts[kg * IMGS * 128 + o];
        const T act = round_bias_relu<T>(a, false, Elem<T>::zero(), AGH_ACT_RELU);
        d1[o] = Elem<T>::to_f32(act);
        if constexpr (SAVE && IMGS == 1) if (step) step->pre1[o] = Elem<T>::to_f32(Elem<T>::from_f32(a));
        if constexpr (SAVE) {
            if ((o >> 7) < nimg) {
                sv.d1[(size_t)b0 * 128 + o] = Elem<T>::from_f32(a);
                sv.a1[(size_t)b0 * 128 + o] = act;
            }
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the direct loads of wd2s / wd3s (not known to the compiler)
    __syncthreads();
    // dense2 128 -> 84 + relu, weights from LDS.  Thread (c, kq) forms the partial sums of output c over a quarter of k
    // for all four images (four independent chains of 32, each weight read once); the quarters are then added in order
    // through LDS (`parts` is free again).  One thread per output over all of k is a chain of 128 dependent FMAs behind
    // 256 LDS reads: 1.6 us of the launch.
    if (tid < 4 * 84) {
        const int kq = tid / 84, c = tid - kq * 84;
        float part[IMGS];
#pragma unroll
        for (int r = 0; r < IMGS; ++r) part[r] = 0.0f;
#pragma unroll
        for (int kk = 0; kk < 32; kk += 4) {
            const int k = kq * 32 + kk;
            float4 xk[IMGS];
#pragma unroll
            for (int r = 0; r < IMGS; ++r) xk[r] = *(const float4 *)(d1 + r * 128 + k);
            const float w0 = Elem<T>::raw(wd2s[k * 84 + c]), w1v = Elem<T>::raw(wd2s[(k + 1) * 84 + c]);
            const float w2v = Elem<T>::raw(wd2s[(k + 2) * 84 + c]), w3v = Elem<T>::raw(wd2s[(k + 3) * 84 + c]);
#pragma unroll
            for (int r = 0; r < IMGS; ++r) {
                part[r] = __builtin_fmaf(xk[r].x, w0, part[r]);
                part[r] = __builtin_fmaf(xk[r].y, w1v, part[r]);
                part[r] = __builtin_fmaf(xk[r].z, w2v, part[r]);
                part[r] = __builtin_fmaf(xk[r].w, w3v, part[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < IMGS; ++r) parts[(kq * IMGS + r) * 84 + c] = part[r];
    }
    __syncthreads();
    if (tid < IMGS * 84) {
        const int r = tid / 84;
        float a = parts[tid];
#pragma unroll
        for (int kq = 1; kq < 4; ++kq) a += parts[kq * IMGS * 84 + tid];
        const T act = round_bias_relu<T>(a, false, Elem<T>::zero(), AGH_ACT_RELU);
        d2[tid] = Elem<T>::to_f32(act);
        if constexpr (SAVE && IMGS == 1) if (step) step->pre2[tid] = Elem<T>::to_f32(Elem<T>::from_f32(a));
        if constexpr (SAVE) {
            if (r < nimg) {
                sv.d2[(size_t)b0 * 84 + tid] = Elem<T>::from_f32(a);
                sv.a2[(size_t)b0 * 84 + tid] = act;
            }
        }
    }
    __syncthreads();
    // dense3 84 -> 10 + bias: thread (kp, r, c) sums 12 of the 84 products, the seven parts are added in order
    if (tid < 7 * IMGS * 10) {
        const int kp = tid / (IMGS * 10), rc = tid - kp * (IMGS * 10), r = rc / 10, c = rc - r * 10;
        float a = 0.0f;
        const float *xr = d2 + r * 84 + kp * 12;
#pragma unroll
        for (int kk = 0; kk < 12; kk += 4) {
            const float4 xk = *(const float4 *)(xr + kk);
            const int k = kp * 12 + kk;
            a = __builtin_fmaf(xk.x, Elem<T>::raw(wd3s[k * 10 + c]), a);
            a = __builtin_fmaf(xk.y, Elem<T>::raw(wd3s[(k + 1) * 10 + c]), a);
            a = __builtin_fmaf(xk.z, Elem<T>::raw(wd3s[(k + 2) * 10 + c]), a);
            a = __builtin_fmaf(xk.w, Elem<T>::raw(wd3s[(k + 3) * 10 + c]), a);
        }
        parts[kD3Off + tid] = a;  // behind the dense2 partials, which other waves may still be reading
    }
    __syncthreads();
    if (tid < IMGS * 10) {
        const int r = tid / 10, c = tid - r * 10;
        float a = parts[kD3Off + tid];
#pragma unroll
        for (int kp = 1; kp < 7; ++kp) a += parts[kD3Off + kp * IMGS * 10 + tid];
        const T logit = round_bias_relu<T>(a, true, b3[c], AGH_ACT_NONE);
        if constexpr (SAVE && IMGS == 1) if (step) step->lg[c] = Elem<T>::to_f32(logit);
        if (r < nimg) out[(size_t)(b0 + r) * 10 + c] = logit;
    }
}

template <typename T, bool SAVE, int IMGS, bool WHOLE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, IMGS == 1 ? 4 : 2))) void lenet5_forward_kernel(const T *__restrict__ x, const T *__restrict__ w1,
                                                              const T *__restrict__ w2, const T *__restrict__ wd1,
                                                              const T *__restrict__ wd2, const T *__restrict__ wd3,
                                                              const T *__restrict__ b3, T *__restrict__ out, int bs,
                                                              LenetSaves<T> sv, int w23_aligned) {
    __shared__ LenetForwardLds<T, IMGS> s;
    float4 wreg[16];
    lenet5_forward_body<T, SAVE, IMGS, WHOLE>(s, x, w1, w2, wd1, wd2, wd3, b3, out, bs, sv, w23_aligned, nullptr, wreg, [] {});
}

// The input-gradient chain of a LeNet5 training step in one launch, one workgroup per image: cross-entropy backward,
// the three dense layers' input gradients with their relu backward, pooling + relu backward of conv2's output written as
// the [64, 16] matrix its weight gradient multiplies, conv2's input gradient (dot with the filter bank, then col2im),
// pooling + relu backward of conv1's output as the [576, 6] matrix.  Every value is rounded to T where the separate
// launches round it, and every T-typed running sum adds in their order (col2im: filter rows and columns descending,
// the dot over the output channels ascending), so the results differ from theirs only through the order of the f32
// adds inside the dense dot products.
template <typename T>
struct LenetBackward {
    const T *logits;            // [bs, 10]
    const uint8_t *target;      // [bs]
    const T *c1, *c2, *d1, *d2; // conv outputs before relu [bs,6,24,24], [bs,16,8,8]; dense outputs before relu [bs,128], [bs,84]
    const T *w2, *wd1, *wd2, *wd3;
    T *g_logits, *g_d2, *g_d1;  // [bs,10], [bs,84], [bs,128]
    T *gm2, *gm1;               // [bs*64, 16], [bs*576, 6]
    float dy;                   // upstream gradient of the summed loss divided by the batch size
};

// pooling (2x2, stride 2) backward through a relu, one window: g lands on the first maximum of relu(x) and passes where
// x >= 0 (the rule of max_pool2_relu_backward_2x2_kernel); cell k = 2 * row + column
template <typename T>
__device__ __forceinline__ void pool_relu_window_backward(const T (&xv)[4], float gy, T (&cell)[4]) {
    auto relu_of = [](T v) { return Elem<T>::raw(v) >= 0.0f ? v : Elem<T>::zero(); };
    float mf = Elem<T>::raw(relu_of(xv[0]));
    int am = 0;
#pragma unroll
    for (int k = 1; k < 4; ++k) {
        const float vf = Elem<T>::raw(relu_of(xv[k]));
        if (vf > mf) { mf = vf; am = k; }
    }
    const T g = Elem<T>::from_f32(0.0f + gy);
#pragma unroll
    for (int k = 0; k < 4; ++k) cell[k] = (am == k && Elem<T>::raw(xv[k]) >= 0.0f) ? g : Elem<T>::zero();
}

constexpr int kPmPitch = 151;  // odd: the col2im reads of neighbouring pixels fall into different banks
// The product gm2 [64 positions, 16 channels] . W [16, 150 taps] of conv2's input gradient, every entry rounded to T, by NW waves: forty tiles of
// 16 positions x 16 taps, four v_mfma_f32_16x16x4_f32 each (as FMAs 5400 cycles of the training step's launch)
template <typename T, int NW>
__device__ __forceinline__ void lenet5_pm(const float *gm2s, const float *wl, float *pm) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, i = lane & 15;
    static_assert(40 % NW == 0, "whole rounds of tiles");
#pragma unroll
    for (int n = 0; n < 40 / NW; ++n) {
        const int unit = wave + NW * n, pt = unit & 3, k = (unit >> 2) * 16 + i;
        // MFMA q takes channel 4 g + q of lane group g on both sides: one 16-byte read each
        const f32x4_t va = *(const f32x4_t *)(gm2s + (pt * 16 + i) * 16 + 4 * g), vb = *(const f32x4_t *)(wl + min(k, 149) * 16 + 4 * g);
        f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int q = 0; q < 4; ++q) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(va[q], vb[q], acc, 0, 0, 0);
        if (k < 150) {
#pragma unroll
            for (int r = 0; r < 4; ++r) pm[(pt * 16 + 4 * g + r) * kPmPitch + k] = Elem<T>::to_f32(Elem<T>::from_f32(acc[r]));
        }
    }
}

// One row of dense2's input gradient, 84 products: part q of four chains the groups of four q, q + 4, ..., the parts are added (0 + 1) + (2 + 3),
// the order in which four lanes of lenet5_step_image_kernel share a row
template <typename G, typename W>
__device__ __forceinline__ float dense2_row_sum(G &&g, W &&w) {
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        v[q] = 0.0f;
#pragma unroll
        for (int c = q; c < 21; c += 4)
#pragma unroll
            for (int e = 0; e < 4; ++e) v[q] = __builtin_fmaf(g(4 * c + e), w(4 * c + e), v[q]);
    }
    return (v[0] + v[1]) + (v[2] + v[3]);
}

// One row of dense1's input gradient, 128 products: 32 chains of four neighbouring ones, added pairwise (i with i + 16, then + 8 ... + 1), the order
// in which the lanes of lenet5_step_image_kernel add them
template <typename G, typename W>
__device__ __forceinline__ float dense1_row_sum(G &&g, W &&w) {
    float v[32];
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        v[i] = 0.0f;
#pragma unroll
        for (int c = 0; c < 4; ++c) v[i] = __builtin_fmaf(g(4 * i + c), w(4 * i + c), v[i]);
    }
    // (by constants: an array indexed by the variable of a loop that is not unrolled costs a select per element)
    auto fold = [&](auto halfc) {
        constexpr int half = decltype(halfc)::value;
#pragma unroll
        for (int i = 0; i < half; ++i) v[i] += v[i + half];
    };
    fold(std::integral_constant<int, 16>{});
    fold(std::integral_constant<int, 8>{});
    fold(std::integral_constant<int, 4>{});
    fold(std::integral_constant<int, 2>{});
    fold(std::integral_constant<int, 1>{});
    return v[0];
}

template <typename T>
__global__ __launch_bounds__(256) void lenet5_backward_kernel(LenetBackward<T> a) {
    __shared__ __align__(16) float wl[150 * 16];   // conv2's filter bank, [ci*25 + fi*5 + fj][oc]
    __shared__ __align__(16) float gm2s[64 * 16];  // gradient of conv2's output, [y*8 + x][oc]
    __shared__ float gls[16], gd2s[84], gd1s[128], gfs[256], gp1s[864];
    __shared__ float pm[64 * kPmPitch];            // gm2 . W, every entry rounded to T
    constexpr int NT = 256;
    constexpr int EPV = 16 / (int)sizeof(T);  // elements per 16-byte load
    const int tid = threadIdx.x;
    const size_t b = blockIdx.x;
    // Everything this workgroup reads from memory has an address known now, so all of it is requested here, before the
    // first use: the stages below are a chain of seven short steps, and a load issued inside a step would add its L2
    // latency to that chain.  (About 100 registers per thread; the launch is 100 workgroups, occupancy is no concern.)
    T w2v[10];  // the filter bank, coalesced: element tid + u * 256 of w2[oc][ci*25 + tap]
#pragma unroll
    for (int u = 0; u < 10; ++u) w2v[u] = a.w2[min(tid + u * NT, 2399)];
    T lrow[10];  // the image's logits (used by the ten threads of the first stage)
#pragma unroll
    for (int j = 0; j < 10; ++j) lrow[j] = a.logits[b * 10 + j];
    const int label = a.target[b];
    T w3v[10];   // row min(tid, 83) of wd3
#pragma unroll
    for (int c = 0; c < 10; ++c) w3v[c] = a.wd3[min(tid, 83) * 10 + c];
    const T d2v = a.d2[b * 84 + min(tid, 83)], d1v = a.d1[b * 128 + (tid & 127)];
    uint2 w2r[84 * (int)sizeof(T) / 8];  // row tid & 127 of wd2 (84 elements: 8-byte aligned)
    {
        const uint2 *src = (const uint2 *)(a.wd2 + (tid & 127) * 84);
#pragma unroll
        for (int c = 0; c < 84 * (int)sizeof(T) / 8; ++c) w2r[c] = src[c];
    }
    uint4 w1r[128 / EPV];  // row tid of wd1
    {
        const uint4 *src = (const uint4 *)(a.wd1 + tid * 128);
#pragma unroll
        for (int c = 0; c < 128 / EPV; ++c) w1r[c] = src[c];
    }
    T x2[4];  // the thread's pooling window of conv2's output
    {
        const int oc = tid >> 4, ho = (tid >> 2) & 3, wo = tid & 3;
        const T *xp = a.c2 + ((b * 16 + oc) * 8 + 2 * ho) * 8 + 2 * wo;
        x2[0] = xp[0]; x2[1] = xp[1]; x2[2] = xp[8]; x2[3] = xp[9];
    }
    T x1[4][4];  // its (up to four) pooling windows of conv1's output
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = min(tid + u * NT, 863);
        const int ci = e / 144, r = e - ci * 144, ho = r / 12, wo = r - ho * 12;
        const T *xp = a.c1 + ((b * 6 + ci) * 24 + 2 * ho) * 24 + 2 * wo;
        x1[u][0] = xp[0]; x1[u][1] = xp[1]; x1[u][2] = xp[24]; x1[u][3] = xp[25];
    }
    auto elem = [](const auto &packed, int c) -> float {  // element c of a row held as 8- or 16-byte words
        if constexpr (sizeof(T) == 4) return __uint_as_float(((const uint32_t *)&packed)[c]);
        else {
            const uint32_t w = ((const uint32_t *)&packed)[c >> 1];
            return __uint_as_float((c & 1) ? (w & 0xFFFF0000u) : (w << 16));
        }
    };

    // cross-entropy backward (softmax - one-hot, times dy), rounded to T
    if (tid < 10) {
        float m = Elem<T>::to_f32(lrow[0]);
#pragma unroll
        for (int j = 0; j < 10; ++j) m = fmaxf(m, Elem<T>::to_f32(lrow[j]));
        float s = 0.0f;
#pragma unroll
        for (int j = 0; j < 10; ++j) s += expf(Elem<T>::to_f32(lrow[j]) - m);
        float mine = 0.0f;
#pragma unroll
        for (int j = 0; j < 10; ++j) mine = j == tid ? Elem<T>::to_f32(lrow[j]) : mine;
        const float pr = expf(mine - m) / s;
        const T g = Elem<T>::from_f32(a.dy * (pr - (tid == label ? 1.0f : 0.0f)));
        a.g_logits[b * 10 + tid] = g;
        gls[tid] = Elem<T>::to_f32(g);
    }
#pragma unroll
    for (int u = 0; u < 10; ++u) {
        const int i = tid + u * NT;
        const int o = i / 150, k = i - o * 150;
        if (i < 2400) wl[k * 16 + o] = Elem<T>::to_f32(w2v[u]);
    }
    __syncthreads();
    // dense3: g_a2 = g_logits . wd3^T (wd3 [84, 10]), then relu backward on dense2's pre-activation
    if (tid < 84) {
        float d = 0.0f;
#pragma unroll
        for (int c = 0; c < 10; ++c) d = __builtin_fmaf(gls[c], Elem<T>::to_f32(w3v[c]), d);
        const T ga = Elem<T>::from_f32(d);
        const T gd = Elem<T>::raw(d2v) >= 0.0f ? ga : Elem<T>::zero();
        a.g_d2[b * 84 + tid] = gd;
        gd2s[tid] = Elem<T>::to_f32(gd);
    }
    __syncthreads();
    // dense2: g_a1 = g_d2 . wd2^T (wd2 [128, 84]), relu backward on dense1's pre-activation
    if (tid < 128) {
        const float d = dense2_row_sum([&](int c) { return gd2s[c]; }, [&](int c) { return elem(w2r, c); });
        const T ga = Elem<T>::from_f32(d);
        const T gd = Elem<T>::raw(d1v) >= 0.0f ? ga : Elem<T>::zero();
        a.g_d1[b * 128 + tid] = gd;
        gd1s[tid] = Elem<T>::to_f32(gd);
    }
    __syncthreads();
    // dense1: g_f = g_d1 . wd1^T (wd1 [256, 128])
    gfs[tid] = Elem<T>::to_f32(Elem<T>::from_f32(dense1_row_sum([&](int c) { return gd1s[c]; }, [&](int c) { return elem(w1r, c); })));
    __syncthreads();
    // pooling + relu backward of conv2's output: one window per thread (16 channels x 4 x 4 windows)
    {
        const int oc = tid >> 4, ho = (tid >> 2) & 3, wo = tid & 3;
        T cell[4];
        pool_relu_window_backward<T>(x2, gfs[tid], cell);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int pos = (2 * ho + (k >> 1)) * 8 + 2 * wo + (k & 1);
            gm2s[pos * 16 + oc] = Elem<T>::to_f32(cell[k]);
            a.gm2[(b * 64 + pos) * 16 + oc] = cell[k];
        }
    }
    __syncthreads();
    // conv2's input gradient in two steps, as the host does it: the product gm2 . W, a [64, 150] matrix whose entries are f32 dots over the 16
    // output channels rounded to T,
    lenet5_pm<T, NT / 64>(gm2s, wl, pm);
    __syncthreads();
    // then col2im: per pixel of the [6, 12, 12] map the patch entries that land on it, added in T in the host's order
    // (filter rows and columns descending)
    for (int e = tid; e < 864; e += NT) {
        const int ci = e / 144, r = e - ci * 144, hy = r / 12, wy = r - hy * 12;
        T acc = Elem<T>::zero();
#pragma unroll
        for (int fi = 4; fi >= 0; --fi) {
            const int th = hy - fi;
            const bool hok = th >= 0 && th < 8;
            const int thc = min(max(th, 0), 7);
#pragma unroll
            for (int fj = 4; fj >= 0; --fj) {
                const int tw = wy - fj;
                const bool ok = hok && tw >= 0 && tw < 8;
                const float v = pm[(thc * 8 + min(max(tw, 0), 7)) * kPmPitch + ci * 25 + fi * 5 + fj];
                acc = Elem<T>::from_f32(Elem<T>::raw(acc) + (ok ? v : 0.0f));
            }
        }
        gp1s[e] = Elem<T>::to_f32(acc);
    }
    __syncthreads();
    // pooling + relu backward of conv1's output (6 channels x 12 x 12 windows), written as the [576, 6] matrix
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const int e = tid + u * NT;
        if (e < 864) {
            const int ci = e / 144, r = e - ci * 144, ho = r / 12, wo = r - ho * 12;
            T cell[4];
            pool_relu_window_backward<T>(x1[u], gp1s[e], cell);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int pos = (2 * ho + (k >> 1)) * 24 + 2 * wo + (k & 1);
                a.gm1[(b * 576 + pos) * 6 + ci] = cell[k];
            }
        }
    }
}

template <typename T>
int lenet5_backward_entry(const char *name, const void *logits, const void *target, float dy, const void *c1, const void *c2,
                          const void *d1, const void *d2, const void *w2, const void *wd1, const void *wd2, const void *wd3,
                          void *g_logits, void *g_d2, void *g_d1, void *gm2, void *gm1, int64_t bs) {
    AGH_API_ENTER();
    if (bs < 0) return fail(AGH_EINVAL, "%s: negative batch size", name);
    if (bs == 0) return AGH_OK;
    if (bs > ((int64_t)1 << 24)) return fail(AGH_ERANGE, "%s: batch too large", name);
    if (!logits || !target || !c1 || !c2 || !d1 || !d2 || !w2 || !wd1 || !wd2 || !wd3 || !g_logits || !g_d2 || !g_d1 || !gm2 || !gm1)
        return fail(AGH_ENULL, "%s: null buffer", name);
    if (((uintptr_t)wd1 & 15) != 0 || ((uintptr_t)wd2 & 7) != 0)
        return fail(AGH_EINVAL, "%s: wd1 must be 16-byte and wd2 8-byte aligned", name);
    LenetBackward<T> a;
    a.logits = (const T *)logits; a.target = (const uint8_t *)target;
    a.c1 = (const T *)c1; a.c2 = (const T *)c2; a.d1 = (const T *)d1; a.d2 = (const T *)d2;
    a.w2 = (const T *)w2; a.wd1 = (const T *)wd1; a.wd2 = (const T *)wd2; a.wd3 = (const T *)wd3;
    a.g_logits = (T *)g_logits; a.g_d2 = (T *)g_d2; a.g_d1 = (T *)g_d1; a.gm2 = (T *)gm2; a.gm1 = (T *)gm1;
    a.dy = dy / (float)bs;  // `dy /= batch_size` first, in f32, as the host does
    hipLaunchKernelGGL(lenet5_backward_kernel<T>, dim3((unsigned)bs), dim3(256), 0, stream(), a);
    AGH_LAUNCH_CHECK(name);
    return AGH_OK;
}

// The weight gradients of the three dense layers, the bias gradient and the loss of a LeNet5 training step in one
// launch: dwd3 = a2^T . g_logits [84, 10], dwd2 = a1^T . g_d2 [128, 84], dwd1 = f^T . g_d1 [256, 128] (each an f32 dot over
// the batch, rounded once to T, as the GEMM rounds it), db3 = the rows of g_logits added one at a time in T (the axis-0
// sum of the host), loss = the row losses added in row order (one workgroup, as cross_entropy_loss_kernel).  A
// workgroup owns a 16 x 16 tile of one product and stages the two 16-column strips it multiplies in LDS.
template <typename T>
struct LenetDenseGrads {
    const T *a2, *a1, *f;               // [bs, 84], [bs, 128], [bs, 256]
    const T *g_logits, *g_d2, *g_d1;    // [bs, 10], [bs, 84], [bs, 128]
    T *dwd3, *dwd2, *dwd1, *db3;        // [84, 10], [128, 84], [256, 128], [10]
    const T *logits;                    // [bs, 10]
    const uint8_t *target;              // [bs]
    float *loss;                        // one f32 (device or pinned host memory); may be null
    int bs;
};

// The update of a training step, applied by whoever finishes a gradient: scaled_add with -lr (no velocities) or SGD with momentum, operation
// for operation as scaled_add_kernel and sgd_momentum_kernel do it.  Order: conv1, conv2, dense1, dense2, dense3, dense3's bias.
template <typename T>
struct LenetUpdate {
    T *w[6], *v[6];
    float lr, momentum;
};
template <typename T>
struct LenetOld { T w, v; };  // a parameter and its velocity, requested before the sums
template <typename T>
__device__ __forceinline__ LenetOld<T> lenet5_old(const LenetUpdate<T> &u, int which, int i) {
    return {u.w[which][i], u.v[which] ? u.v[which][i] : Elem<T>::zero()};
}
template <typename T>
__device__ __forceinline__ void lenet5_update(const LenetUpdate<T> &u, int which, int i, const LenetOld<T> &old, T g) {
    if (u.v[which]) {
        const float mv = u.momentum * Elem<T>::to_f32(old.v);
        const float vn = mv + Elem<T>::to_f32(g);
        const float step = u.lr * vn;
        u.v[which][i] = Elem<T>::from_f32(vn);
        u.w[which][i] = Elem<T>::from_f32(Elem<T>::to_f32(old.w) - step);
    } else {
        const float a = Elem<T>::to_f32(Elem<T>::from_f32(-u.lr));
        const T prod = Elem<T>::from_f32(a * Elem<T>::to_f32(g));
        u.w[which][i] = Elem<T>::from_f32(Elem<T>::to_f32(prod) + Elem<T>::to_f32(old.w));
    }
}

// 256 threads of workgroup `wg` (of 184); UPDATE: the parameters too
template <typename T, bool UPDATE>
__device__ __forceinline__ void lenet5_dense_grads(const LenetDenseGrads<T> q, int wg, const LenetUpdate<T> &upd) {
    constexpr int RCH = 128;  // batch rows per pass
    __shared__ float as[RCH * 16], gs[RCH * 16];
    __shared__ __align__(16) float part[256];
    const int tid = threadIdx.x;
    // tiles: dwd1 16 x 8, dwd2 8 x 6, dwd3 6 x 1, then the bias gradient, then the loss
    const T *A, *G;
    T *D;
    int K, N, tk, tn, which;
    if (wg < 128) { A = q.f; G = q.g_d1; D = q.dwd1; K = 256; N = 128; tk = wg / 8; tn = wg % 8; which = 2; }
    else if (wg < 176) { wg -= 128; A = q.a1; G = q.g_d2; D = q.dwd2; K = 128; N = 84; tk = wg / 6; tn = wg % 6; which = 3; }
    else if (wg < 182) { wg -= 176; A = q.a2; G = q.g_logits; D = q.dwd3; K = 84; N = 10; tk = wg; tn = 0; which = 4; }
    else if (wg == 182) {
        LenetOld<T> old = {};
        if (UPDATE && tid < 10) old = lenet5_old(upd, 5, tid);
        // the rows go through LDS, 200 at a time: read straight from memory the hundred dependent additions of a column
        // would each wait for their own load
        T acc = Elem<T>::zero();
        for (int r0 = 0; r0 < q.bs; r0 += 200) {
            const int cnt = min(200, q.bs - r0) * 10;
            __syncthreads();
            T v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = q.g_logits[(size_t)r0 * 10 + min(tid + u * 256, cnt - 1)];
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (tid + u * 256 < cnt) as[tid + u * 256] = Elem<T>::to_f32(v[u]);
            __syncthreads();
            if (tid < 10) {
                // sixteen rows are read before the first is added (the chain itself is a few cycles a row)
                const int nr = cnt / 10;
                int r = 0;
                for (; r + 16 <= nr; r += 16) {
                    float h[16];
#pragma unroll
                    for (int u = 0; u < 16; ++u) h[u] = as[(r + u) * 10 + tid];
#pragma unroll
                    for (int u = 0; u < 16; ++u) acc = Elem<T>::from_f32(Elem<T>::raw(acc) + h[u]);
                }
                for (; r < nr; ++r) acc = Elem<T>::from_f32(Elem<T>::raw(acc) + as[r * 10 + tid]);
            }
        }
        if (tid < 10) {
            q.db3[tid] = acc;
            if (UPDATE) lenet5_update(upd, 5, tid, old, acc);
        }
        return;
    } else {
        if (!q.loss) return;
        float total = 0.0f;
        for (int base = 0; base < q.bs; base += 256) {
            const int r = base + tid;
            float l = 0.0f;
            if (r < q.bs) {
                const T *row = q.logits + (size_t)r * 10;
                float m = Elem<T>::to_f32(row[0]);
                for (int j = 0; j < 10; ++j) m = fmaxf(m, Elem<T>::to_f32(row[j]));
                float sum = 0.0f;
                for (int j = 0; j < 10; ++j) sum += expf(Elem<T>::to_f32(row[j]) - m);
                l = logf(sum) - (Elem<T>::to_f32(row[q.target[r]]) - m);
            }
            part[tid] = l;
            __syncthreads();
            if (tid == 0) {
                const int cnt = min(256, q.bs - base);
                int i = 0;
                for (; i + 32 <= cnt; i += 32) {
                    float4 h[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) h[u] = *(const float4 *)(part + i + 4 * u);
#pragma unroll
                    for (int u = 0; u < 8; ++u) {
                        total += h[u].x;
                        total += h[u].y;
                        total += h[u].z;
                        total += h[u].w;
                    }
                }
                for (; i < cnt; ++i) total += part[i];
            }
            __syncthreads();
        }
        if (tid == 0) *q.loss = total;
        return;
    }
    const int k0 = tk * 16, n0 = tn * 16;
    const int i = tid >> 4, j = tid & 15;
    const bool mine = k0 + i < K && n0 + j < N;
    const int at = (k0 + i) * N + n0 + j;
    LenetOld<T> old = {};
    if (UPDATE && mine) old = lenet5_old(upd, which, at);
    float acc = 0.0f;
    // all 16 elements of a thread are requested before the first is stored (one at a time the staging alone would be a chain of eight
    // memory latencies), and those of the next pass before this one's products
    T av[RCH * 16 / 256], gv[RCH * 16 / 256];
    auto request = [&](int r0) __attribute__((always_inline)) {
        const int rows = min(RCH, q.bs - r0);
#pragma unroll
        for (int u = 0; u < RCH * 16 / 256; ++u) {
            const int e = tid + u * 256, r = min(e >> 4, rows - 1), c = e & 15;
            av[u] = A[(size_t)(r0 + r) * K + min(k0 + c, K - 1)];
            gv[u] = G[(size_t)(r0 + r) * N + min(n0 + c, N - 1)];
        }
    };
    request(0);
    for (int r0 = 0; r0 < q.bs; r0 += RCH) {
        const int rows = min(RCH, q.bs - r0);
        __syncthreads();
#pragma unroll
        for (int u = 0; u < RCH * 16 / 256; ++u) {
            const int e = tid + u * 256, r = e >> 4, c = e & 15;
            const bool rok = r < rows;
            as[e] = rok && k0 + c < K ? Elem<T>::to_f32(av[u]) : 0.0f;
            gs[e] = rok && n0 + c < N ? Elem<T>::to_f32(gv[u]) : 0.0f;
        }
        __syncthreads();
        if (r0 + RCH < q.bs) request(r0 + RCH);
#pragma unroll 16
        for (int r = 0; r < rows; ++r) acc = __builtin_fmaf(as[r * 16 + i], gs[r * 16 + j], acc);
    }
    if (mine) {
        const T g = Elem<T>::from_f32(acc);
        D[at] = g;
        if (UPDATE) lenet5_update(upd, which, at, old, g);
    }
}
constexpr int kLenetDenseGroups = 184;
template <typename T>
__global__ __launch_bounds__(256) void lenet5_dense_grads_kernel(LenetDenseGrads<T> q) {
    lenet5_dense_grads<T, false>(q, (int)blockIdx.x, {});
}

template <typename T>
int lenet5_dense_grads_check(const char *name, const void *a2, const void *a1, const void *f, const void *g_logits, const void *g_d2,
                             const void *g_d1, void *dwd3, void *dwd2, void *dwd1, void *db3, const void *logits, const void *target,
                             void *loss, int64_t bs, LenetDenseGrads<T> &q) {
    if (bs > ((int64_t)1 << 24)) return fail(AGH_ERANGE, "%s: batch too large", name);
    if (!a2 || !a1 || !f || !g_logits || !g_d2 || !g_d1 || !dwd3 || !dwd2 || !dwd1 || !db3)
        return fail(AGH_ENULL, "%s: null buffer", name);
    if (loss && (!logits || !target)) return fail(AGH_ENULL, "%s: the loss needs the logits and the labels", name);
    q.a2 = (const T *)a2; q.a1 = (const T *)a1; q.f = (const T *)f;
    q.g_logits = (const T *)g_logits; q.g_d2 = (const T *)g_d2; q.g_d1 = (const T *)g_d1;
    q.dwd3 = (T *)dwd3; q.dwd2 = (T *)dwd2; q.dwd1 = (T *)dwd1; q.db3 = (T *)db3;
    q.logits = (const T *)logits; q.target = (const uint8_t *)target; q.loss = (float *)loss; q.bs = (int)bs;
    return AGH_OK;
}

template <typename T>
int lenet5_dense_grads_entry(const char *name, const void *a2, const void *a1, const void *f, const void *g_logits,
                             const void *g_d2, const void *g_d1, void *dwd3, void *dwd2, void *dwd1, void *db3,
                             const void *logits, const void *target, void *loss, int64_t bs) {
    AGH_API_ENTER();
    if (bs < 0) return fail(AGH_EINVAL, "%s: negative batch size", name);
    if (bs == 0) return AGH_OK;
    LenetDenseGrads<T> q;
    if (int rc = lenet5_dense_grads_check<T>(name, a2, a1, f, g_logits, g_d2, g_d1, dwd3, dwd2, dwd1, db3, logits, target, loss, bs, q)) return rc;
    hipLaunchKernelGGL(lenet5_dense_grads_kernel<T>, dim3(kLenetDenseGroups), dim3(256), 0, stream(), q);
    AGH_LAUNCH_CHECK(name);
    return AGH_OK;
}

// The weight gradients of the two convolutions of a LeNet5 training step without their patch matrices:
// dw2[oc][ci][fi][fj] = sum over images and output positions of gm2[(y, x)][oc] * p1[ci][y + fi][x + fj] (the product
// gm2^T . im2col(p1) of layer.rs:990-1003), dw1 likewise from gm1 and x.  One workgroup per image forms the image's f32
// partial sums from operands staged in LDS; a second launch adds the partials (by quarters of the batch, two interleaved sums each, then these
// eight) and rounds once to T, as the split-K GEMM does.
constexpr int kLenetPartPitch = 2560;  // per image: 2400 entries of dw2, 150 of dw1
// 512 threads: one image's partial sums out of LDS: g2 [y*8 + x][oc] and g1 [y*24 + x][oc] the gradients of the convolutions' outputs, p1s and
// xs their inputs; q2 and q1 take the second half of conv2's positions and conv1's eight row groups.  On v_mfma_f32_16x16x4_f32 (lane (g, i):
// row i of A, column i of B, k = g; accumulator r: row 4 g + r, column i): rows are output channels, columns taps, k positions, both operands
// gathered with one 4-byte read at a constant offset.  As FMAs with a thread per tap the reads of the gradient rows, 2000 LDS instructions an
// image, were what it took: 15200 cycles, 6.5 us of the training step's launch.
__device__ __forceinline__ void lenet5_conv_grads_sums(const float *g2, const float *g1, const float *p1s, const float *xs, float *q2, float *q1,
                                                       float *__restrict__ out) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, i = lane & 15;
    // conv2: ten tiles of 16 taps x two halves of the 64 positions are twenty units of 8 MFMAs, unit = 2 tile + half; a wave has up to three
    f32x4_t acc2[3];
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        acc2[n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        const int unit = wave + 8 * n;
        if (unit >= 20) continue;  // wave-uniform
        const int half = unit & 1, k = min((unit >> 1) * 16 + i, 149), ci = k / 25, t = k - ci * 25, fi = t / 5, fj = t - fi * 5;
        const float *A = g2 + half * 512 + g * 16 + i, *B = p1s + ci * 144 + (half * 4 + fi) * 12 + fj + g;
#pragma unroll
        for (int q = 0; q < 8; ++q) acc2[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(A[q * 64], B[(q >> 1) * 12 + (q & 1) * 4], acc2[n], 0, 0, 0);
        if (half == 1 && (unit >> 1) * 16 + i < 150) {
#pragma unroll
            for (int r = 0; r < 4; ++r) q2[(4 * g + r) * 150 + k] = acc2[n][r];
        }
    }
    // conv1: a wave takes three of the 24 output rows (72 positions), two tiles of taps; rows behind the six channels repeat the last
    {
        const int ta = i, tb = min(16 + i, 24);
        const float *A = g1 + (wave * 72 + g) * 6 + min(i, 5), *X = xs + wave * 84 + g;
        const float *Ba = X + (ta / 5) * 28 + ta % 5, *Bb = X + (tb / 5) * 28 + tb % 5;
        f32x4_t a0 = {0.0f, 0.0f, 0.0f, 0.0f}, a1 = a0;
#pragma unroll
        for (int q = 0; q < 18; ++q) {
            const float v = A[q * 24];
            const int at = (q / 6) * 28 + (q % 6) * 4;
            a0 = __builtin_amdgcn_mfma_f32_16x16x4f32(v, Ba[at], a0, 0, 0, 0);
            a1 = __builtin_amdgcn_mfma_f32_16x16x4f32(v, Bb[at], a1, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int oc = 4 * g + r;
            if (oc < 6) {
                q1[wave * 150 + oc * 25 + ta] = a0[r];
                if (16 + i < 25) q1[wave * 150 + oc * 25 + tb] = a1[r];
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < 3; ++n) {
        const int unit = wave + 8 * n, k = (unit >> 1) * 16 + i;
        if (unit < 20 && (unit & 1) == 0 && k < 150) {
#pragma unroll
            for (int r = 0; r < 4; ++r) out[(4 * g + r) * 150 + k] = acc2[n][r] + q2[(4 * g + r) * 150 + k];
        }
    }
    const int k = threadIdx.x - 300;
    if (k >= 0 && k < 150) {
        float s = q1[k];
#pragma unroll
        for (int rg = 1; rg < 8; ++rg) s += q1[rg * 150 + k];
        out[2400 + k] = s;
    }
}

template <typename T>
__device__ __forceinline__ void lenet5_conv_grads(const T *__restrict__ x, const T *__restrict__ p1, const T *__restrict__ gm1,
                                                  const T *__restrict__ gm2, float *__restrict__ part, size_t b) {
    __shared__ __align__(16) float g2[64 * 16];   // [y*8 + x][oc]
    __shared__ __align__(8) float g1[576 * 6];    // [y*24 + x][oc]
    __shared__ float p1s[864], xs[784];
    __shared__ float q2[16 * 150], q1[8 * 150];   // partial sums: conv2 second half of the positions; conv1 by row group
    constexpr int NT = 512;
    const int tid = threadIdx.x;
    {
        // every element is requested before the first is stored
        T v2[2], vp[2], vx[2], v1[7];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            v2[u] = gm2[b * 1024 + tid + u * NT];
            vp[u] = p1[b * 864 + min(tid + u * NT, 863)];
            vx[u] = x[b * 784 + min(tid + u * NT, 783)];
        }
#pragma unroll
        for (int u = 0; u < 7; ++u) v1[u] = gm1[b * 3456 + min(tid + u * NT, 3455)];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int i = tid + u * NT;
            g2[i] = Elem<T>::to_f32(v2[u]);
            if (i < 864) p1s[i] = Elem<T>::to_f32(vp[u]);
            if (i < 784) xs[i] = Elem<T>::to_f32(vx[u]);
        }
#pragma unroll
        for (int u = 0; u < 7; ++u)
            if (tid + u * NT < 3456) g1[tid + u * NT] = Elem<T>::to_f32(v1[u]);
    }
    __syncthreads();
    lenet5_conv_grads_sums(g2, g1, p1s, xs, q2, q1, part + b * kLenetPartPitch);
}

template <typename T>
__global__ __launch_bounds__(512) void lenet5_conv_grads_kernel(const T *__restrict__ x, const T *__restrict__ p1,
                                                                  const T *__restrict__ gm1, const T *__restrict__ gm2,
                                                                  float *__restrict__ part) {
    lenet5_conv_grads<T>(x, p1, gm1, gm2, part, blockIdx.x);
}

// Both in one launch: the first 184 workgroups form the dense layers' gradients with four of their eight waves, the others the images'
// partial sums.  Neither reads what the other writes, and either alone leaves most of the chip waiting for first-touch loads: on one
// stream the two launches took 4.8 + 8.3 us (batch 100, bf16), this one takes 9.4 (training step 45.0 -> 42.1).
template <typename T>
__global__ __launch_bounds__(512) void lenet5_weight_grads_kernel(LenetDenseGrads<T> q, const T *__restrict__ x, const T *__restrict__ p1,
                                                                    const T *__restrict__ gm1, const T *__restrict__ gm2,
                                                                    float *__restrict__ part) {
    if (blockIdx.x >= kLenetDenseGroups) {
        lenet5_conv_grads<T>(x, p1, gm1, gm2, part, blockIdx.x - kLenetDenseGroups);
    } else {
        if (threadIdx.x >= 256) return;  // a barrier waits for the waves that have not ended
        lenet5_dense_grads<T, false>(q, (int)blockIdx.x, {});
    }
}

// 64 outputs per workgroup `wg` (of 40) of 256 threads; wave j adds the images of the j-th quarter of the batch in two interleaved sums (sixteen
// loads in flight), the eight sums are then added in a fixed order
constexpr int kLenetReduceGroups = 40;
template <typename T, bool UPDATE>
__device__ __forceinline__ void lenet5_conv_reduce(const float *__restrict__ part, T *__restrict__ dw1, T *__restrict__ dw2, int bs, int wg,
                                                   const LenetUpdate<T> &upd) {
    __shared__ float sums[4][64];
    const int lane = threadIdx.x & 63, j = threadIdx.x >> 6;
    const int k = min(wg * 64 + lane, 2549), which = k < 2400 ? 1 : 0, at = k < 2400 ? k : k - 2400;
    const bool mine = j == 0 && wg * 64 + lane < 2550;
    LenetOld<T> old = {};
    if (UPDATE && mine) old = lenet5_old(upd, which, at);
    const int per = (bs + 3) / 4, b0 = j * per, b1 = min(bs, b0 + per);
    float s0 = 0.0f, s1 = 0.0f;
    int b = b0;
    for (; b + 16 <= b1; b += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = part[(size_t)(b + u) * kLenetPartPitch + k];
#pragma unroll
        for (int u = 0; u < 16; u += 2) {
            s0 += v[u];
            s1 += v[u + 1];
        }
    }
    if (b < b1) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = part[(size_t)min(b + u, b1 - 1) * kLenetPartPitch + k];
#pragma unroll
        for (int u = 0; u < 16; u += 2) {
            s0 += b + u < b1 ? v[u] : 0.0f;
            s1 += b + u + 1 < b1 ? v[u + 1] : 0.0f;
        }
    }
    sums[j][lane] = s0 + s1;
    __syncthreads();
    if (mine) {
        const float tot = (sums[0][lane] + sums[1][lane]) + (sums[2][lane] + sums[3][lane]);
        const T g = Elem<T>::from_f32(tot);
        (which ? dw2 : dw1)[at] = g;
        if (UPDATE) lenet5_update(upd, which, at, old, g);
    }
}
template <typename T>
__global__ __launch_bounds__(256) void lenet5_conv_grads_reduce_kernel(const float *__restrict__ part, T *__restrict__ dw1,
                                                                         T *__restrict__ dw2, int bs) {
    lenet5_conv_reduce<T, false>(part, dw1, dw2, bs, (int)blockIdx.x, {});
}

template <typename T>
int lenet5_conv_grads_entry(const char *name, const void *x, const void *p1, const void *gm1, const void *gm2, void *dw1,
                            void *dw2, int64_t bs) {
    AGH_API_ENTER();
    if (bs < 0) return fail(AGH_EINVAL, "%s: negative batch size", name);
    if (bs == 0) return AGH_OK;
    if (bs > ((int64_t)1 << 20)) return fail(AGH_ERANGE, "%s: batch too large", name);
    if (!x || !p1 || !gm1 || !gm2 || !dw1 || !dw2) return fail(AGH_ENULL, "%s: null buffer", name);
    void *ws = nullptr;
    if (int rc = workspace((size_t)bs * kLenetPartPitch * sizeof(float), &ws)) return rc;
    hipLaunchKernelGGL(lenet5_conv_grads_kernel<T>, dim3((unsigned)bs), dim3(512), 0, stream(), (const T *)x, (const T *)p1,
                       (const T *)gm1, (const T *)gm2, (float *)ws);
    AGH_LAUNCH_CHECK(name);
    hipLaunchKernelGGL(lenet5_conv_grads_reduce_kernel<T>, dim3(kLenetReduceGroups), dim3(256), 0, stream(), (const float *)ws, (T *)dw1,
                       (T *)dw2, (int)bs);
    AGH_LAUNCH_CHECK(name);
    return AGH_OK;
}

template <typename T>
int lenet5_weight_grads_entry(const char *name, const void *a2, const void *a1, const void *f, const void *g_logits,
                              const void *g_d2, const void *g_d1, void *dwd3, void *dwd2, void *dwd1, void *db3,
                              const void *logits, const void *target, void *loss, const void *x, const void *p1, const void *gm1,
                              const void *gm2, void *dw1, void *dw2, int64_t bs) {
    AGH_API_ENTER();
    if (bs < 0) return fail(AGH_EINVAL, "%s: negative batch size", name);
    if (bs == 0) return AGH_OK;
    if (bs > ((int64_t)1 << 20)) return fail(AGH_ERANGE, "%s: batch too large", name);
    LenetDenseGrads<T> q;
    if (int rc = lenet5_dense_grads_check<T>(name, a2, a1, f, g_logits, g_d2, g_d1, dwd3, dwd2, dwd1, db3, logits, target, loss, bs, q)) return rc;
    if (!x || !p1 || !gm1 || !gm2 || !dw1 || !dw2) return fail(AGH_ENULL, "%s: null buffer", name);
    void *ws = nullptr;
    if (int rc = workspace((size_t)bs * kLenetPartPitch * sizeof(float), &ws)) return rc;
    hipLaunchKernelGGL(lenet5_weight_grads_kernel<T>, dim3((unsigned)bs + kLenetDenseGroups), dim3(512), 0, stream(), q, (const T *)x,
                       (const T *)p1, (const T *)gm1, (const T *)gm2, (float *)ws);
    AGH_LAUNCH_CHECK(name);
    hipLaunchKernelGGL(lenet5_conv_grads_reduce_kernel<T>, dim3(kLenetReduceGroups), dim3(256), 0, stream(), (const float *)ws, (T *)dw1,
                       (T *)dw2, (int)bs);
    AGH_LAUNCH_CHECK(name);
    return AGH_OK;
}


// ---- a whole training step in two launches ----
//
// The step as five launches (forward, input gradients, weight gradients, the sum of the images' shares, update) is a chain of launches whose
// work is small: at batch 100 in bf16 10.2 + 14.4 + 9.6 + 4.5 + 4.4 us, of which the backward one waits 6 us for the first touch of a dozen
// buffers that the launch before it wrote.  Here a workgroup takes ONE image through forward, input gradients and its share of the
// convolutions' weight gradients with activations, gradients and the small layers' weights in LDS; the second launch forms the dense layers'
// gradients, adds the shares, and whoever finishes a gradient updates its parameter (nothing else reads the parameters there).  Every value is
// rounded where the separate launches round it and summed in their order, so gradients, loss and parameters have their bits.  What bounds the
// first launch is its chain of eighteen stages behind barriers, 40000 cycles in bf16, the longest 7000 (shares of the weight gradients), 4300
// (staging), 3900 (col2im) and 3800 (conv2); a batch beyond 512 is several rounds of it, two workgroups per CU (one per CU, with
// arrays of their own for everything: in brackets).  A captured step, five launches -> here, bf16 / f32: batch 100 42.3 -> 27.4 us / 42.7 -> 26.0,
// 400 70.8 -> 40.7 (48.9) / 82.4 -> 38.5 (45.5), 1000 109.7 -> 70.9 (90) / 135.3 -> 65.8 (82), 2048 194 -> 127 (168) / 248 -> 117 (152).
template <typename T>
struct LenetStep {
    const T *x, *w1, *w2, *wd1, *wd2, *wd3, *b3;
    const uint8_t *target;
    T *logits, *g_logits, *g_d2, *g_d1, *gm2, *gm1;
    float *part;
    float dy;
    int bs, w23_aligned;
};

template <typename T, bool WHOLE>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 4))) void lenet5_step_image_kernel(LenetStep<T> a, LenetSaves<T> sv) {
    // Two workgroups fit a CU (LDS 81144 bytes in f32, 67952 in bf16; 128 registers): behind the dense layers' gradients the forward pass's last
    // arrays (parts, wd2s, wd3s) are free.  There lie pm, gp1s behind it, and when pm has been read g1 and behind it q2 and q1, each written
    // behind a barrier after the last read of what it replaces.
    using Forward = LenetForwardLds<T, 1>;
    constexpr int kFree = offsetof(Forward, parts), kPm = 64 * kPmPitch, kG1 = 576 * 6, kSize = sizeof(Forward);
    constexpr int kBackward = kFree + (kPm + 864) * 4;
    static_assert(kG1 + 24 * 150 <= kPm + 864 && kFree % 16 == 0, "g1, q2 and q1 fit where pm and gp1s were");
    __shared__ __align__(16) unsigned char lds[kSize > kBackward ? kSize : kBackward];
    Forward &s = *(Forward *)lds;
    __shared__ LenetStepLds st;
    __shared__ __align__(16) float gm2s[64 * 16];  // gradient of conv2's output, [y*8 + x][oc]
    __shared__ __align__(16) float gd1s[128], gd2s[84];
    __shared__ float gls[16];
    float *const gfs = s.p2;                  // 256: gradient of the flattened features, for the features themselves
    float *const pm = (float *)(lds + kFree);  // gm2 . W, every entry rounded to T
    float *const gp1s = pm + kPm;             // 864: gradient of conv1's pooled output
    float *const g1 = pm;                     // of conv1's output, [y*24 + x][oc]
    float *const q2 = g1 + kG1, *const q1 = q2 + 16 * 150;
    constexpr int NT = 512;
    const int tid = threadIdx.x;
    const size_t b = blockIdx.x;
    const int label = a.target[b];
    float4 wreg[16];  // dense1's weights [16 kg ..][4 cg ..], for both directions
    T x2[4], x1[2][4];  // the pooling windows: requested when the convolutions' outputs are saved, used behind the dense layers
    lenet5_forward_body<T, true, 1, WHOLE>(s, a.x, a.w1, a.w2, a.wd1, a.wd2, a.wd3, a.b3, a.logits, a.bs, sv, a.w23_aligned, &st, wreg, [&]() __attribute__((always_inline)) {
        {
            const int t = tid & 255, oc = t >> 4, ho = (t >> 2) & 3, wo = t & 3;
            const T *xp = sv.c2 + ((b * 16 + oc) * 8 + 2 * ho) * 8 + 2 * wo;
            x2[0] = xp[0]; x2[1] = xp[1]; x2[2] = xp[8]; x2[3] = xp[9];
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const int e = min(tid + u * NT, 863);
            const int ci = e / 144, r = e - ci * 144, ho = r / 12, wo = r - ho * 12;
            const T *xp = sv.c1 + ((b * 6 + ci) * 24 + 2 * ho) * 24 + 2 * wo;
            x1[u][0] = xp[0]; x1[u][1] = xp[1]; x1[u][2] = xp[24]; x1[u][3] = xp[25];
        }
    });
    __syncthreads();
    // cross-entropy backward (softmax - one-hot, times dy), rounded to T
    if (tid < 10) {
        float m = st.lg[0];
#pragma unroll
        for (int j = 0; j < 10; ++j) m = fmaxf(m, st.lg[j]);
        float sum = 0.0f;
#pragma unroll
        for (int j = 0; j < 10; ++j) sum += expf(st.lg[j] - m);
        const float pr = expf(st.lg[tid] - m) / sum;
        const T g = Elem<T>::from_f32(a.dy * (pr - (tid == label ? 1.0f : 0.0f)));
        a.g_logits[b * 10 + tid] = g;
        gls[tid] = Elem<T>::to_f32(g);
    }
    __syncthreads();
    // dense3, dense2 (weights in LDS) and dense1: input gradients, relu backward on the pre-activations
    if (tid < 84) {
        float d = 0.0f;
#pragma unroll
        for (int c = 0; c < 10; ++c) d = __builtin_fmaf(gls[c], Elem<T>::to_f32(s.wd3s[tid * 10 + c]), d);
        const T gd = st.pre2[tid] >= 0.0f ? Elem<T>::from_f32(d) : Elem<T>::zero();
        a.g_d2[b * 84 + tid] = gd;
        gd2s[tid] = Elem<T>::to_f32(gd);
    }
    __syncthreads();
    {
        // four lanes share a row of wd2 (dense2_row_sum adds in the same order)
        const int row = tid >> 2, q = tid & 3;
        float d = 0.0f;
#pragma unroll
        for (int n = 0; n < 6; ++n) {
            const int c = q + 4 * n;
            if (c >= 21) break;
            const float4 g = *(const float4 *)(gd2s + 4 * c);
            float w[4];
            if constexpr (sizeof(T) == 4) {
                const float4 r = *(const float4 *)(s.wd2s + row * 84 + 4 * c);
                w[0] = r.x; w[1] = r.y; w[2] = r.z; w[3] = r.w;
            } else {
                const uint2 r = *(const uint2 *)(s.wd2s + row * 84 + 4 * c);
                w[0] = __uint_as_float(r.x << 16); w[1] = __uint_as_float(r.x & 0xFFFF0000u);
                w[2] = __uint_as_float(r.y << 16); w[3] = __uint_as_float(r.y & 0xFFFF0000u);
            }
            d = __builtin_fmaf(g.x, w[0], d);
            d = __builtin_fmaf(g.y, w[1], d);
            d = __builtin_fmaf(g.z, w[2], d);
            d = __builtin_fmaf(g.w, w[3], d);
        }
        d += __shfl_xor(d, 1);
        d += __shfl_xor(d, 2);
        if (q == 0) {
            const T gd = st.pre1[row] >= 0.0f ? Elem<T>::from_f32(d) : Elem<T>::zero();
            a.g_d1[b * 128 + row] = gd;
            gd1s[row] = Elem<T>::to_f32(gd);
        }
    }
    __syncthreads();
    {
        // thread (cg, kg): four of the 128 products of 16 rows; the 32 lanes of a half-wave add their parts pairwise, each step halving the rows
        // a lane goes on with (dense1_row_sum adds in the same order)
        const int cg = tid & 31, kg = tid >> 5;
        const float4 g = *(const float4 *)(gd1s + cg * 4);
        float v[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            v[r] = __builtin_fmaf(g.x, wreg[r].x, 0.0f);
            v[r] = __builtin_fmaf(g.y, wreg[r].y, v[r]);
            v[r] = __builtin_fmaf(g.z, wreg[r].z, v[r]);
            v[r] = __builtin_fmaf(g.w, wreg[r].w, v[r]);
        }
        auto fold = [&](auto halfc) {
            constexpr int half = decltype(halfc)::value;
            const bool up = (cg & (2 * half)) != 0;
#pragma unroll
            for (int r = 0; r < half; ++r) {
                const float keep = up ? v[r + half] : v[r], send = up ? v[r] : v[r + half];
                v[r] = keep + __shfl_xor(send, 2 * half);
            }
        };
        fold(std::integral_constant<int, 8>{});
        fold(std::integral_constant<int, 4>{});
        fold(std::integral_constant<int, 2>{});
        fold(std::integral_constant<int, 1>{});
        const float d = v[0] + __shfl_xor(v[0], 1);
        if ((cg & 1) == 0) gfs[kg * 16 + (cg >> 1)] = Elem<T>::to_f32(Elem<T>::from_f32(d));
    }
    __syncthreads();
    // pooling + relu backward of conv2's output: one window per thread (16 channels x 4 x 4 windows)
    if (tid < 256) {
        const int oc = tid >> 4, ho = (tid >> 2) & 3, wo = tid & 3;
        T cell[4];
        pool_relu_window_backward<T>(x2, gfs[tid], cell);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int pos = (2 * ho + (k >> 1)) * 8 + 2 * wo + (k & 1);
            gm2s[pos * 16 + oc] = Elem<T>::to_f32(cell[k]);
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 2; ++u) a.gm2[b * 1024 + tid + u * NT] = Elem<T>::from_f32(gm2s[tid + u * NT]);  // (exact: T values)
    // conv2's input gradient: the product gm2 . W, then col2im in the host's order, as lenet5_backward_kernel does it; a thread takes two pixels,
    // whose chains of 25 additions run side by side
    lenet5_pm<T, NT / 64>(gm2s, s.w2s, pm);
    __syncthreads();
    if (tid < 432) {
        T acc[2] = {Elem<T>::zero(), Elem<T>::zero()};
        const int ci0 = tid / 144, r0 = tid - ci0 * 144, hy = r0 / 12, wy = r0 - hy * 12;  // pixel e = tid + 432: three channels on
#pragma unroll
        for (int fi = 4; fi >= 0; --fi) {
            const int th = hy - fi;
            const bool hok = th >= 0 && th < 8;
            const int thc = min(max(th, 0), 7);
#pragma unroll
            for (int fj = 4; fj >= 0; --fj) {
                const int tw = wy - fj;
                const bool ok = hok && tw >= 0 && tw < 8;
                const float *v = pm + (thc * 8 + min(max(tw, 0), 7)) * kPmPitch + ci0 * 25 + fi * 5 + fj;
#pragma unroll
                for (int u = 0; u < 2; ++u) acc[u] = Elem<T>::from_f32(Elem<T>::raw(acc[u]) + (ok ? v[75 * u] : 0.0f));
            }
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) gp1s[tid + 432 * u] = Elem<T>::to_f32(acc[u]);
    }
    __syncthreads();
    // pooling + relu backward of conv1's output (6 channels x 12 x 12 windows), as the [576, 6] matrix
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int e = tid + u * NT;
        if (e < 864) {
            const int ci = e / 144, r = e - ci * 144, ho = r / 12, wo = r - ho * 12;
            T cell[4];
            pool_relu_window_backward<T>(x1[u], gp1s[e], cell);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const int pos = (2 * ho + (k >> 1)) * 24 + 2 * wo + (k & 1);
                g1[pos * 6 + ci] = Elem<T>::to_f32(cell[k]);
            }
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 7; ++u)
        if (tid + u * NT < 3456) a.gm1[b * 3456 + tid + u * NT] = Elem<T>::from_f32(g1[tid + u * NT]);
    lenet5_conv_grads_sums(gm2s, g1, s.p1, s.xs, q2, q1, a.part + b * kLenetPartPitch);
}

template <typename T>
__global__ __launch_bounds__(256) void lenet5_finish_kernel(LenetDenseGrads<T> q, const float *__restrict__ part, T *__restrict__ dw1,
                                                             T *__restrict__ dw2, LenetUpdate<T> upd) {
    if (blockIdx.x < kLenetDenseGroups) lenet5_dense_grads<T, true>(q, (int)blockIdx.x, upd);
    else lenet5_conv_reduce<T, true>(part, dw1, dw2, q.bs, (int)blockIdx.x - kLenetDenseGroups, upd);
}

template <typename T>
int lenet5_train_step_entry(const char *name, const void *x, const void *target, void *const *params, void *const *velocities,
                            void *const *grads, void *const *saves, void *const *input_grads, float dy, float lr, float momentum, void *loss,
                            int64_t bs) {
    AGH_API_ENTER();
    if (bs < 0) return fail(AGH_EINVAL, "%s: negative batch size", name);
    if (bs == 0) return AGH_OK;
    if (bs > ((int64_t)1 << 20)) return fail(AGH_ERANGE, "%s: batch too large", name);
    if (!x || !target || !params || !grads || !saves || !input_grads) return fail(AGH_ENULL, "%s: null buffer", name);
    for (int i = 0; i < 6; ++i)
        if (!params[i] || !grads[i] || (velocities && !velocities[i])) return fail(AGH_ENULL, "%s: null parameter, gradient or velocity", name);
    for (int i = 0; i < 9; ++i)
        if (!saves[i]) return fail(AGH_ENULL, "%s: null buffer for a saved activation", name);
    for (int i = 0; i < 5; ++i)
        if (!input_grads[i]) return fail(AGH_ENULL, "%s: null buffer for an input gradient", name);
    if (((uintptr_t)params[2] & 15) != 0 || ((uintptr_t)params[3] & 7) != 0)
        return fail(AGH_EINVAL, "%s: wd1 must be 16-byte and wd2 8-byte aligned", name);
    LenetDenseGrads<T> q;
    if (int rc = lenet5_dense_grads_check<T>(name, saves[7], saves[5], saves[3], input_grads[0], input_grads[1], input_grads[2], grads[4], grads[3],
                                             grads[2], grads[5], saves[8], target, loss, bs, q))
        return rc;
    void *ws = nullptr;
    if (int rc = workspace((size_t)bs * kLenetPartPitch * sizeof(float), &ws)) return rc;
    LenetStep<T> a;
    a.x = (const T *)x; a.target = (const uint8_t *)target;
    a.w1 = (const T *)params[0]; a.w2 = (const T *)params[1]; a.wd1 = (const T *)params[2]; a.wd2 = (const T *)params[3];
    a.wd3 = (const T *)params[4]; a.b3 = (const T *)params[5];
    a.logits = (T *)saves[8];
    a.g_logits = (T *)input_grads[0]; a.g_d2 = (T *)input_grads[1]; a.g_d1 = (T *)input_grads[2];
    a.gm2 = (T *)input_grads[3]; a.gm1 = (T *)input_grads[4];
    a.part = (float *)ws;
    a.dy = dy / (float)bs;  // `dy /= batch_size` first, in f32, as the host does
    a.bs = (int)bs;
    a.w23_aligned = (((uintptr_t)params[3] | (uintptr_t)params[4]) & 15) == 0;
    const LenetSaves<T> sv = {(T *)saves[0], (T *)saves[1], (T *)saves[2], (T *)saves[3], (T *)saves[4], (T *)saves[5], (T *)saves[6], (T *)saves[7]};
    LenetUpdate<T> upd;
    for (int i = 0; i < 6; ++i) {
        upd.w[i] = (T *)params[i];
        upd.v[i] = velocities ? (T *)velocities[i] : nullptr;
    }
    upd.lr = lr;
    upd.momentum = momentum;
    // (the forward entries take four images a workgroup above 256)
    if (bs <= 256) hipLaunchKernelGGL((lenet5_step_image_kernel<T, false>), dim3((unsigned)bs), dim3(512), 0, stream(), a, sv);
    else hipLaunchKernelGGL((lenet5_step_image_kernel<T, true>), dim3((unsigned)bs), dim3(512), 0, stream(), a, sv);
    AGH_LAUNCH_CHECK(name);
    hipLaunchKernelGGL(lenet5_finish_kernel<T>, dim3(kLenetDenseGroups + kLenetReduceGroups), dim3(256), 0, stream(), q, (const float *)a.part,
                       (T *)grads[0], (T *)grads[1], upd);
    AGH_LAUNCH_CHECK(name);
    return AGH_OK;
}

}  // namespace

template <typename T>
int lenet5_forward_entry(const char *name, const void *x, const void *w1, const void *w2, const void *wd1, const void *wd2,
                         const void *wd3, const void *b3, void *logits, int64_t bs, void *const *saves) {
    AGH_API_ENTER();
    if (bs < 0 || bs > ((int64_t)1 << 30)) return fail(AGH_EINVAL, "%s: bad batch size", name);
    if (bs == 0) return AGH_OK;
    if (!x || !w1 || !w2 || !wd1 || !wd2 || !wd3 || !b3 || !logits) return fail(AGH_ENULL, "%s: null buffer", name);
    LenetSaves<T> sv = {};
    const int w23_aligned = (((uintptr_t)wd2 | (uintptr_t)wd3) & 15) == 0;
    if (saves) {
        for (int i = 0; i < 8; ++i)
            if (!saves[i]) return fail(AGH_ENULL, "%s: null buffer for a saved activation", name);
        sv = {(T *)saves[0], (T *)saves[1], (T *)saves[2], (T *)saves[3], (T *)saves[4], (T *)saves[5], (T *)saves[6], (T *)saves[7]};
    }
    // one image per workgroup while that still fits the chip in one round
    const bool single = bs <= 256;  // measured: 7.0 against 11.2 us up to 256 images
    // Two such workgroups share a CU.  Where they need few enough rounds (of 256 images: every further one costs a third of the time that a round of
    // 1024 takes with four images a workgroup), they are faster up to a batch of 512, from 1025 to 1280 and from 2049 to 2304: f32 257 10.9 -> 9.1 us, 512
    // 11.0 -> 9.6, 1025 20.5 -> 18.1, 2304 30.9 -> 30.8, bf16 12.8 -> 9.4, 12.9 -> 10.1, 24.2 -> 19.4, 36.2 -> 33.6; beyond: f32 600 11.0 / 12.7,
    // 1536 21.0 / 21.7, bf16 1000 12.9 / 16.9.  Conv2's sums are one chain, as with four images a workgroup: the same bits.
    const int64_t rounds1 = (bs + 255) / 256, rounds4 = (bs + 1023) / 1024;
    const bool pairs = rounds1 <= 3 * rounds4 - (rounds4 < 3);
#define AGH_LENET(SAVEV, IMGSV, WHOLEV) \
    hipLaunchKernelGGL((lenet5_forward_kernel<T, SAVEV, IMGSV, WHOLEV>), dim3((unsigned)((bs + IMGSV - 1) / IMGSV)), dim3(512), 0, stream(), \
                       (const T *)x, (const T *)w1, (const T *)w2, (const T *)wd1, (const T *)wd2, (const T *)wd3, (const T *)b3, \
                       (T *)logits, (int)bs, sv, w23_aligned)
    if (saves) {
        if (single) AGH_LENET(true, 1, false); else if (pairs) AGH_LENET(true, 1, true); else AGH_LENET(true, 4, false);
    } else {
        if (single) AGH_LENET(false, 1, false); else if (pairs) AGH_LENET(false, 1, true); else AGH_LENET(false, 4, false);
    }
#undef AGH_LENET
    AGH_LAUNCH_CHECK(name);
    return AGH_OK;
}

extern "C" {

int agh_lenet5_forward_f32(const void *x, const void *w1, const void *w2, const void *wd1, const void *wd2,
                           const void *wd3, const void *b3, void *logits, int64_t bs) {
    return lenet5_forward_entry<float>("agh_lenet5_forward_f32", x, w1, w2, wd1, wd2, wd3, b3, logits, bs, nullptr);
}
int agh_lenet5_forward_bf16(const void *x, const void *w1, const void *w2, const void *wd1, const void *wd2,
                            const void *wd3, const void *b3, void *logits, int64_t bs) {
    return lenet5_forward_entry<uint16_t>("agh_lenet5_forward_bf16", x, w1, w2, wd1, wd2, wd3, b3, logits, bs, nullptr);
}
int agh_lenet5_forward_train_f32(const void *x, const void *w1, const void *w2, const void *wd1, const void *wd2,
                                 const void *wd3, const void *b3, void *c1, void *p1, void *c2, void *p2, void *d1,
                                 void *a1, void *d2, void *a2, void *logits, int64_t bs) {
    void *saves[8] = {c1, p1, c2, p2, d1, a1, d2, a2};
    return lenet5_forward_entry<float>("agh_lenet5_forward_train_f32", x, w1, w2, wd1, wd2, wd3, b3, logits, bs, saves);
}
int agh_lenet5_forward_train_bf16(const void *x, const void *w1, const void *w2, const void *wd1, const void *wd2,
                                  const void *wd3, const void *b3, void *c1, void *p1, void *c2, void *p2, void *d1,
                                  void *a1, void *d2, void *a2, void *logits, int64_t bs) {
    void *saves[8] = {c1, p1, c2, p2, d1, a1, d2, a2};
    return lenet5_forward_entry<uint16_t>("agh_lenet5_forward_train_bf16", x, w1, w2, wd1, wd2, wd3, b3, logits, bs, saves);
}

#define AGH_LENET_BWD_ARGS                                                                                             \
    const void *logits, const void *target, float dy, const void *c1, const void *c2, const void *d1, const void *d2, \
        const void *w2, const void *wd1, const void *wd2, const void *wd3, void *g_logits, void *g_d2, void *g_d1,    \
        void *gm2, void *gm1, int64_t bs
int agh_lenet5_backward_f32(AGH_LENET_BWD_ARGS) {
    return lenet5_backward_entry<float>("agh_lenet5_backward_f32", logits, target, dy, c1, c2, d1, d2, w2, wd1, wd2, wd3,
                                        g_logits, g_d2, g_d1, gm2, gm1, bs);
}
int agh_lenet5_backward_bf16(AGH_LENET_BWD_ARGS) {
    return lenet5_backward_entry<uint16_t>("agh_lenet5_backward_bf16", logits, target, dy, c1, c2, d1, d2, w2, wd1, wd2, wd3,
                                           g_logits, g_d2, g_d1, gm2, gm1, bs);
}

#define AGH_LENET_DG_PTRS                                                                                            \
    const void *a2, const void *a1, const void *f, const void *g_logits, const void *g_d2, const void *g_d1, void *dwd3, \
        void *dwd2, void *dwd1, void *db3, const void *logits, const void *target, void *loss
#define AGH_LENET_DG_ARGS AGH_LENET_DG_PTRS, int64_t bs
int agh_lenet5_dense_weight_grads_f32(AGH_LENET_DG_ARGS) {
    return lenet5_dense_grads_entry<float>("agh_lenet5_dense_weight_grads_f32", a2, a1, f, g_logits, g_d2, g_d1, dwd3, dwd2,
                                           dwd1, db3, logits, target, loss, bs);
}
int agh_lenet5_dense_weight_grads_bf16(AGH_LENET_DG_ARGS) {
    return lenet5_dense_grads_entry<uint16_t>("agh_lenet5_dense_weight_grads_bf16", a2, a1, f, g_logits, g_d2, g_d1, dwd3,
                                              dwd2, dwd1, db3, logits, target, loss, bs);
}

int agh_lenet5_weight_grads_f32(AGH_LENET_DG_PTRS, const void *x, const void *p1, const void *gm1, const void *gm2, void *dw1, void *dw2,
                                int64_t bs) {
    return lenet5_weight_grads_entry<float>("agh_lenet5_weight_grads_f32", a2, a1, f, g_logits, g_d2, g_d1, dwd3, dwd2, dwd1, db3, logits,
                                            target, loss, x, p1, gm1, gm2, dw1, dw2, bs);
}
int agh_lenet5_weight_grads_bf16(AGH_LENET_DG_PTRS, const void *x, const void *p1, const void *gm1, const void *gm2, void *dw1, void *dw2,
                                 int64_t bs) {
    return lenet5_weight_grads_entry<uint16_t>("agh_lenet5_weight_grads_bf16", a2, a1, f, g_logits, g_d2, g_d1, dwd3, dwd2, dwd1, db3,
                                               logits, target, loss, x, p1, gm1, gm2, dw1, dw2, bs);
}
int agh_lenet5_conv_weight_grads_f32(const void *x, const void *p1, const void *gm1, const void *gm2, void *dw1, void *dw2,
                                     int64_t bs) {
    return lenet5_conv_grads_entry<float>("agh_lenet5_conv_weight_grads_f32", x, p1, gm1, gm2, dw1, dw2, bs);
}
int agh_lenet5_conv_weight_grads_bf16(const void *x, const void *p1, const void *gm1, const void *gm2, void *dw1, void *dw2,
                                      int64_t bs) {
    return lenet5_conv_grads_entry<uint16_t>("agh_lenet5_conv_weight_grads_bf16", x, p1, gm1, gm2, dw1, dw2, bs);
}

#define AGH_LENET_STEP_ARGS                                                                                                     \
    const void *x, const void *target, void **params, void **velocities, void **grads, void **saves, void **input_grads, float dy, \
        float learning_rate, float momentum, void *loss, int64_t bs
int agh_lenet5_train_step_f32(AGH_LENET_STEP_ARGS) {
    return lenet5_train_step_entry<float>("agh_lenet5_train_step_f32", x, target, params, velocities, grads, saves, input_grads, dy, learning_rate,
                                          momentum, loss, bs);
}
int agh_lenet5_train_step_bf16(AGH_LENET_STEP_ARGS) {
    return lenet5_train_step_entry<uint16_t>("agh_lenet5_train_step_bf16", x, target, params, velocities, grads, saves, input_grads, dy,
                                             learning_rate, momentum, loss, bs);
}

}  // extern "C"
