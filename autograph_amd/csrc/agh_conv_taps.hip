// Conv2 forward on the f32 matrix cores for any stride, dilation and channel count: the geometries that the
// implicit GEMM of agh_conv_mfma.hip (unit stride, channels in whole vectors) and the kernels that hold a whole image
// in LDS do not take.  Replaces im2col + GEMM there (src/learn/neural_network/layer.rs:950-1005).
//
// A network's first layer (3 channels, 7 x 7, stride 2) has k = 147: patch rows that no 16-byte load fits, so the
// product behind im2col ran through element-wise loaders.  The patch matrix itself is 2 * 147 * positions values of
// traffic where x and y are 9 % of that.  Here a workgroup takes 64 * TG output positions of one image and 16 * NT
// channels and stages the zero-padded input rows that the positions touch in LDS, as f32, as many channels at a time as
// fit.  A 16 x 16 x 4 MFMA multiplies 16 positions by 16 channels over 4 taps: the A operand is gathered from the staged
// rows, one 4-byte LDS read per lane (the position's base + the tap's offset, from a small table) for NT MFMAs of 32
// cycles each, so neither bank conflicts of strided positions nor the LDS rate matter.  The B operand comes straight
// from the filter bank: the taps of a chunk of 16 are dealt so that lane group g holds taps 4g .. 4g+3, one 16-byte
// load per lane and chunk, requested a chunk ahead (element addresses of any alignment; the bank stays in the caches).
// What bounds it: the f32 matrix pipes (157 TFLOP/s), the staging that the co-resident workgroups do not hide, and the
// last, partly filled round of workgroups.  64 x 3 x 95 x 95 to 64 channels, 7 x 7 stride 2, f32: 76 us (im2col 25 + GEMM 56)
// -> 43 us, 64 TFLOP/s; 53 x 32 x 61 x 61 to 64, 3 x 3: 153 -> 98 us, 74 TFLOP/s.
#include "agh_internal.h"

using namespace agh;

namespace {

struct TapsParams {
    int ic, ih, iw, oc, ph, pw, sh, sw, dh, dw;
    int act, has_bias;
    int npos;         // output positions per image; with the pool, the 4 positions of every window
    int ptiles;       // workgroups per image and channel group
    int chunk;        // input channels staged at a time
    int rows, pitch;  // staged rows per channel and their pitch (floats, a multiple of 4)
    int fhfw, ktot;
    FastDiv div_ptiles, div_pitch4, div_rows, div_yw, div_fw, div_fhfw;  // yw: the result's row, of positions or windows
};

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef int i32x4_t __attribute__((ext_vector_type(4)));
// four elements at any element address: one load or store (the device runs in unaligned access mode)
template <typename T> struct Four;
template <> struct Four<float> { typedef float type __attribute__((ext_vector_type(4), aligned(4))); };
template <> struct Four<uint16_t> { typedef uint16_t type __attribute__((ext_vector_type(4), aligned(2))); };

// With the pool, positions are numbered window by window, the four of a window in row order: the accumulator layout then
// leaves each lane whole 2 x 2 windows of one channel, and bias, ReLU and the first-strict-maximum pooling happen in
// registers.  A position's taps are staged and added in the same order either way, so the result is, bit for bit, the
// pool of what the call without it returns.
template <typename T, int TG, int NT, bool POOL>
__global__ __launch_bounds__(256, 2) void conv2_taps_kernel(const T *__restrict__ x, const T *__restrict__ w,
                                                            const T *__restrict__ bias, T *__restrict__ y, TapsParams p) {
    using V4 = typename Four<T>::type;
    extern __shared__ __align__(16) float smem_f[];
    const int ntab = (p.chunk * p.fhfw + 15) & ~15;
    int *tab = (int *)smem_f;     // [ntab] byte offsets of the taps from a position's first cell
    float *xs = smem_f + ntab;    // [chunk][rows][pitch], zero padded
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, i = lane & 15;
    uint32_t b, tile;
    p.div_ptiles.divmod(blockIdx.x, b, tile);
    const int p0 = (int)tile * (64 * TG), oc0 = (int)blockIdx.y * (16 * NT);
    auto output_at = [&](uint32_t pos, uint32_t &oy, uint32_t &ox) {
        if constexpr (POOL) {
            p.div_yw.divmod(pos >> 2, oy, ox);
            oy = 2 * oy + ((pos >> 1) & 1);
            ox = 2 * ox + (pos & 1);
        } else p.div_yw.divmod(pos, oy, ox);
    };
    uint32_t oy0, ox0;
    output_at((uint32_t)p0, oy0, ox0);
    const int h0 = (int)oy0 * p.sh - p.ph;  // the image row that staged row 0 holds
    const T *xb = x + (size_t)b * p.ic * p.ih * p.iw;

    for (int k = threadIdx.x; k < ntab; k += 256) {
        uint32_t ci, rem, fi, fj;
        p.div_fhfw.divmod((uint32_t)min(k, p.chunk * p.fhfw - 1), ci, rem);
        p.div_fw.divmod(rem, fi, fj);
        tab[k] = (int)((ci * p.rows + fi * p.dh) * p.pitch + fj * p.dw) * 4;
    }
    // positions behind the image's last repeat it; their results are not stored
    const int wp0 = p0 + wave * (16 * TG);
    const char *abase[TG];
#pragma unroll
    for (int t = 0; t < TG; ++t) {
        uint32_t oy, ox;
        output_at((uint32_t)min(wp0 + t * 16 + i, p.npos - 1), oy, ox);
        abase[t] = (const char *)(xs + (int)(oy - oy0) * p.sh * p.pitch + (int)ox * p.sw);
    }
    uint32_t wrow[NT];  // elements, below 2^28; a channel behind the last repeats it
#pragma unroll
    for (int n = 0; n < NT; ++n) wrow[n] = (uint32_t)min(oc0 + 16 * n + i, p.oc - 1) * p.ktot + 4 * g;
    // Sums of 64 taps are added to a total: one chain over all taps has 1.4 times the f32 error of im2col and the product
    // (2-norm against f64, 24 channels of 3 x 3: 1.9e-7 against 1.4e-7), this has 1.1e-7; 256 channels of 5 x 5: 2.2e-7
    // against 7.3e-7.  It costs 3 to 10 % of the kernel's time.
    f32x4_t acc[TG][NT], total[TG][NT];
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[t][n] = total[t][n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    int fill = 0;  // chunks in acc
    auto chunk_done = [&]() {
        if (++fill < 4) return;
        fill = 0;
#pragma unroll
        for (int t = 0; t < TG; ++t)
#pragma unroll
            for (int n = 0; n < NT; ++n) {
                total[t][n] += acc[t][n];
                acc[t][n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
            }
    };

    for (int c0 = 0; c0 < p.ic; c0 += p.chunk) {
        const int nch = min(p.chunk, p.ic - c0), klen = nch * p.fhfw;
        if (c0) __syncthreads();
        // stage four cells of a row at a time, eight groups in flight; a group reads the nearest four cells of its image
        // row (the row is at least four long, or the group is read cell by cell), padding cells store zero
        const int ngrp = nch * p.rows * (p.pitch >> 2);
        const T *xc = xb + (size_t)c0 * p.ih * p.iw;
        constexpr int U = 8;
        for (int e0 = threadIdx.x; e0 < ngrp; e0 += U * 256) {
            V4 v[U];
            int at[U], shift[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int e = min(e0 + u * 256, ngrp - 1);
                uint32_t r1, col, ch, row;
                p.div_pitch4.divmod((uint32_t)e, r1, col);
                p.div_rows.divmod(r1, ch, row);
                const int hi = h0 + (int)row, wi = 4 * (int)col - p.pw;
                const T *xr = xc + ((size_t)ch * p.ih + min(max(hi, 0), p.ih - 1)) * p.iw;
                const int first = min(max(wi, 0), max(p.iw - 4, 0));
                if (p.iw >= 4) v[u] = *(const V4 *)(xr + first);
                else v[u] = V4{xr[0], xr[min(1, p.iw - 1)], xr[p.iw - 1], xr[p.iw - 1]};
                at[u] = e;
                // cell c of the group is v[c + shift]; rows outside the image: no cell
                shift[u] = hi >= 0 && hi < p.ih ? wi - first : 4;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (e0 + u * 256 >= ngrp) break;
                f32x4_t f = {Elem<T>::to_f32(v[u].x), Elem<T>::to_f32(v[u].y), Elem<T>::to_f32(v[u].z), Elem<T>::to_f32(v[u].w)};
                const int lim = min(p.iw, 4), sh = shift[u];
                if (sh != 0 || lim < 4) {
                    const f32x4_t o = f;
#pragma unroll
                    for (int c = 0; c < 4; ++c) {
                        const int k = c + sh;
                        const float s01 = k == 1 ? o.y : o.x, s23 = k == 3 ? o.w : o.z;
                        f[c] = k >= 0 && k < lim ? (k >= 2 ? s23 : s01) : 0.0f;
                    }
                }
                *(f32x4_t *)(xs + 4 * at[u]) = f;
            }
        }
        __syncthreads();
        if (wp0 >= p.npos) continue;  // (no barrier is skipped: both stand outside of what follows)

        // full chunks: both operands of chunk c + 1 and the tap offsets of c + 2 are requested before chunk c is multiplied
        const int nfull = klen >> 4;
        const int *tl = tab + 4 * g;
        if (nfull) {
            V4 bn[NT];
            float an[4][TG];
            i32x4_t on = *(const i32x4_t *)tl;
#pragma unroll
            for (int n = 0; n < NT; ++n) bn[n] = *(const V4 *)(w + wrow[n]);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int t = 0; t < TG; ++t) an[q][t] = *(const float *)(abase[t] + on[q]);
            on = *(const i32x4_t *)(tl + min(1, nfull - 1) * 16);
            for (int c = 0; c < nfull; ++c) {
                f32x4_t bc[NT];
                float ac[4][TG];
#pragma unroll
                for (int n = 0; n < NT; ++n)
                    bc[n] = f32x4_t{Elem<T>::to_f32(bn[n].x), Elem<T>::to_f32(bn[n].y), Elem<T>::to_f32(bn[n].z), Elem<T>::to_f32(bn[n].w)};
                const uint32_t next = (uint32_t)min(c + 1, nfull - 1) * 16;
#pragma unroll
                for (int n = 0; n < NT; ++n) bn[n] = *(const V4 *)(w + (wrow[n] + next));
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int t = 0; t < TG; ++t) {
                        ac[q][t] = an[q][t];
                        an[q][t] = *(const float *)(abase[t] + on[q]);
                    }
                on = *(const i32x4_t *)(tl + min(c + 2, nfull - 1) * 16);
                __builtin_amdgcn_sched_barrier(0);  // (or the scheduler sinks the requests behind the products)
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int t = 0; t < TG; ++t)
#pragma unroll
                        for (int n = 0; n < NT; ++n)
                            acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(ac[q][t], bc[n][q], acc[t][n], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                chunk_done();
            }
        }
        if (klen & 15) {  // the last taps: both operands are zero behind them (0 * inf would poison the sum)
            const int k0 = nfull * 16;
            float bt[NT][4];
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int k = k0 + 4 * g + q;
                    const float v = Elem<T>::to_f32(w[wrow[n] + (uint32_t)min(k, klen - 1) - 4 * g]);
                    bt[n][q] = k < klen ? v : 0.0f;
                }
            const i32x4_t o4 = *(const i32x4_t *)(tl + k0);
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int t = 0; t < TG; ++t) {
                    float a = *(const float *)(abase[t] + o4[q]);
                    a = k0 + 4 * g + q < klen ? a : 0.0f;
#pragma unroll
                    for (int n = 0; n < NT; ++n) acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bt[n][q], acc[t][n], 0, 0, 0);
                }
            chunk_done();
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) wrow[n] += klen;
    }

    // lane (g, i) holds positions 4g .. 4g+3 of channel i of every tile: with the pool, one window
    const int nout = POOL ? p.npos >> 2 : p.npos;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int ch = oc0 + 16 * n + i;
        if (ch >= p.oc) continue;
        const T bv = p.has_bias ? bias[ch] : Elem<T>::zero();
        T *yc = y + ((size_t)b * p.oc + ch) * nout;
#pragma unroll
        for (int t = 0; t < TG; ++t) {
            const int pos = wp0 + t * 16 + 4 * g;
            V4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = round_bias_relu<T>(total[t][n][r] + acc[t][n][r], p.has_bias != 0, bv, p.act);
            if constexpr (POOL) {
                T m = o[0];
                float mf = Elem<T>::to_f32(m);
#pragma unroll
                for (int r = 1; r < 4; ++r) {
                    const float f = Elem<T>::to_f32(o[r]);
                    if (f > mf) { m = o[r]; mf = f; }
                }
                if (pos < p.npos) yc[pos >> 2] = m;
            } else if (pos + 3 < p.npos) {
                *(V4 *)(yc + pos) = o;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (pos + r < p.npos) yc[pos + r] = o[r];
            }
        }
    }
}

constexpr int64_t kTapsLds = 48 * 1024;      // three workgroups per CU
constexpr int64_t kTapsPoolLds = 80 * 1024;  // two: whole windows meet up to twice the rows of as many positions in a line

// rows and channels that a workgroup of 64 * tg positions stages; false where not even one channel fits
bool taps_stage(int tg, int64_t ic, int64_t oh, int64_t ow, int64_t fh, int64_t fw, int64_t sh, int64_t dh, int64_t pitch, int64_t &rows,
                int64_t &chunk) {
    const int64_t span = std::min(oh - 1, (64 * tg - 1 + ow - 1) / ow);
    rows = span * sh + (fh - 1) * dh + 1;
    const int64_t per_channel = (rows * pitch + fh * fw) * 4;
    chunk = std::min(ic, (kTapsLds - 64) / per_channel);
    if (chunk < 1) return false;
    for (int64_t m : {16, 4})  // whole chunks of 16 taps where several stages are needed
        if (chunk < ic && chunk >= m) { chunk -= chunk % m; break; }
    return true;
}

}  // namespace

namespace agh {

template <typename T, int TG, int NT, bool POOL>
static int taps_launch(const char *name, const void *x, const void *w, const void *bias, void *y, dim3 grid, size_t smem, const TapsParams &q) {
    if (smem > 64 * 1024)
        AGH_HIP(hipFuncSetAttribute((const void *)(conv2_taps_kernel<T, TG, NT, POOL>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL((conv2_taps_kernel<T, TG, NT, POOL>), grid, dim3(256), smem, stream(), (const T *)x, (const T *)w, (const T *)bias, (T *)y, q);
    AGH_LAUNCH_CHECK(name);
    return AGH_OK;
}

template <typename T>
int conv2_taps_try(const char *name, const void *x, const void *w, const void *bias, void *y, int64_t bs, int64_t ic, int64_t ih,
                   int64_t iw, int64_t oc, int64_t fh, int64_t fw, int64_t ph, int64_t pw, int64_t sh, int64_t sw, int64_t dh,
                   int64_t dw, int64_t oh, int64_t ow, int act, bool pool, bool forced, double limit_us, double *estimate_us) {
    const int64_t npos = oh * ow, ktot = ic * fh * fw, pitch = ((ow - 1) * sw + (fw - 1) * dw + 4) & ~(int64_t)3;
    if (npos > ((int64_t)1 << 24) || ktot > ((int64_t)1 << 24) || oc * ktot > ((int64_t)1 << 28)) return 1;
    // tile: rounds of workgroups times the matrix cycles of one (16 positions x 16 channels x 4 taps = 32 cycles, each wave
    // on a SIMD of its own; a lone wave waits about 500 cycles for the operands of 16 taps), and its staging (batches of 8
    // groups of four cells a thread, a memory round trip each), which later rounds hide in part.  AGH_CONV_TAPS_TILE = 10 TG + NT
    // forces a tile where the kernel is forced (tests).
    const char *env = forced ? setting("AGH_CONV_TAPS_TILE") : nullptr;
    const int tile = env && *env ? atoi(env) : 0;
    const int64_t cus = compute_units() > 0 ? compute_units() : 256, n16 = (oc + 15) / 16;
    int tg = 0, nt = 0;
    int64_t rows = 0, chunk = 0;
    double best = 0, us = 0;
    for (int t : {4, 2, 1}) {
        int64_t r, c;
        if (!taps_stage(t, ic, oh, ow, fh, fw, sh, dh, pitch, r, c)) continue;
        const int64_t stages = (ic + c - 1) / c, batches = (c * r * (pitch / 4) + 8 * 256 - 1) / (8 * 256);
        for (int n = 1; n <= 4 && (n <= n16 || tile); ++n) {
            if (tile && tile != 10 * t + n) continue;
            const int64_t blocks = bs * ((npos + 64 * t - 1) / (64 * t)) * ((n16 + n - 1) / n), rounds = (blocks + cus - 1) / cus;
            const double mfma = (double)(ktot + 15) / 16.0 * std::max(t * n * 128.0, rounds == 1 ? 500.0 : 0.0);
            const double stage = (double)stages * (1500.0 * (double)batches + 1500.0) + 2500.0;
            const double cost = (double)rounds * mfma + stage * (0.6 + 0.4 * (double)rounds);
            if (!tg || cost < best) {
                best = cost; tg = t; nt = n; rows = r; chunk = c;
                // its time, on the safe side of what 2600 shapes measured (three quarters of them need less): what the matrix
                // cycles or, up to three workgroups of a CU together, the waits for operands come to, the stages, of which
                // later rounds hide a quarter, and the bytes that no cache holds
                const double chunks = (double)(ktot + 15) / 16.0;
                us = kTapsLeastUs + (std::max(1.375 * (double)rounds * chunks * t * n * 128.0, 0.9 * chunks * 500.0 * (double)((rounds + 2) / 3)) +
                            (double)stages * (2200.0 * (double)batches + 3300.0) * (0.25 + 0.75 * (double)rounds)) / 2100.0 +
                     0.11e-6 * (double)sizeof(T) * (double)bs * ((double)ic * ih * iw + (double)oc * npos);
            }
        }
    }
    if (estimate_us) *estimate_us = tg ? us : 1e30;
    if (!tg || estimate_us || (!forced && us > limit_us)) return 1;
    // the pool is fused where the convolution alone would run here, and stages as many channels at a time (the order of the
    // sums); only the tile's positions are fewer where its rows, less than three times as many, take too much of the LDS
    const int64_t ntab = (chunk * fh * fw + 15) & ~(int64_t)15, yh = pool ? oh / 2 : oh, yw = pool ? ow / 2 : ow;
    const int64_t nall = pool ? yh * yw * 4 : npos;
    auto lds_bytes = [&]() { return (ntab + chunk * rows * pitch) * 4; };
    if (pool) {
        auto pool_rows = [&]() { rows = (2 * std::min(yh - 1, (16 * tg - 1 + yw - 1) / yw) + 1) * sh + (fh - 1) * dh + 1; };
        for (pool_rows(); tg > 1 && lds_bytes() > kTapsPoolLds; pool_rows()) tg /= 2;
        if (lds_bytes() > 160 * 1024) return 1;
    }
    TapsParams q;
    q.ic = (int)ic; q.ih = (int)ih; q.iw = (int)iw; q.oc = (int)oc; q.ph = (int)ph; q.pw = (int)pw;
    q.sh = (int)sh; q.sw = (int)sw; q.dh = (int)dh; q.dw = (int)dw; q.act = act; q.has_bias = bias != nullptr;
    q.npos = (int)nall;
    q.ptiles = (int)((nall + 64 * tg - 1) / (64 * tg));
    q.chunk = (int)chunk; q.rows = (int)rows; q.pitch = (int)pitch; q.fhfw = (int)(fh * fw); q.ktot = (int)ktot;
    q.div_ptiles = FastDiv((uint32_t)q.ptiles); q.div_pitch4 = FastDiv((uint32_t)(pitch / 4)); q.div_rows = FastDiv((uint32_t)rows);
    q.div_yw = FastDiv((uint32_t)yw); q.div_fw = FastDiv((uint32_t)fw); q.div_fhfw = FastDiv((uint32_t)q.fhfw);
    const int64_t gx = bs * q.ptiles, gy = (n16 + nt - 1) / nt;
    if (gx > 0x7FFFFFFF || gy > 65535) return 1;
    const dim3 grid((unsigned)gx, (unsigned)gy);
#define AGH_TAPS(TGV, NTV) \
    case TGV * 8 + NTV: \
        return pool ? taps_launch<T, TGV, NTV, true>(name, x, w, bias, y, grid, (size_t)lds_bytes(), q) \
                    : taps_launch<T, TGV, NTV, false>(name, x, w, bias, y, grid, (size_t)lds_bytes(), q)
#define AGH_TAPS4(TGV) AGH_TAPS(TGV, 1); AGH_TAPS(TGV, 2); AGH_TAPS(TGV, 3); AGH_TAPS(TGV, 4)
    switch (tg * 8 + nt) { AGH_TAPS4(4); AGH_TAPS4(2); AGH_TAPS4(1); }
#undef AGH_TAPS4
#undef AGH_TAPS
    return 1;
}

template int conv2_taps_try<float>(const char *, const void *, const void *, const void *, void *, int64_t, int64_t, int64_t, int64_t,
                                   int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int, bool, bool, double, double *);
template int conv2_taps_try<uint16_t>(const char *, const void *, const void *, const void *, void *, int64_t, int64_t, int64_t, int64_t,
                                      int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int, bool, bool, double, double *);

}  // namespace agh
