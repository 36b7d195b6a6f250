// Direct 2-D convolution for small channel counts (the LeNet5-sized layers), with the
// ReLU and the 2x2/stride-2 MaxPool2 that follow such a layer optionally fused in.
//
// Conv2::forward in the reference goes im2col -> dot -> NHWC->NCHW copy on a device
// (src/learn/neural_network/layer.rs:950-1005) and through a register-tiled direct kernel on
// the host (layer/conv_direct.rs:23-83).  For layers whose whole input image and filter bank
// fit in LDS, materialising the patch matrix is pure overhead (conv1 of LeNet5 at batch 1000
// would write and re-read 57.6 MB to do 173 MFLOP), so this kernel convolves straight out of
// LDS:
//   - a workgroup stages `imgs` input images (converted to f32) and the filter bank,
//     transposed to [tap][oc] so that the OCT output channels of a work item are one vector
//     read at a wave-uniform address (an LDS broadcast);
//   - a work item owns one output pixel - or, with the pool fused, one 2x2 pool window - for
//     OCT output channels, and walks the taps (ci, fi, fj) accumulating in f32 registers;
//   - the epilogue applies, in the order the separate layers would: round to T, add bias in T,
//     ReLU (x >= 0 ? x : 0), first-strict-maximum over the window in row-major order, and
//     writes NCHW directly.
#include "agh_internal.h"

using namespace agh;

namespace {

struct ConvParams {
    int bs, ic, ih, iw, oc, oh, ow;
    int fh, fw, ph, pw, sh, sw, dh, dw;
    int act, has_bias;
    int imgs;      // images per workgroup
    int ngroups;   // ceil(oc / OCT)
    int ocpad;     // ngroups * OCT
    int yh, yw;    // output tensor spatial size (pooled or not)
    int items_per_img;
    FastDiv div_items, div_pix, div_yw;
};

// Fills n LDS slots from global memory with U reads of a thread in flight at a time: `get(e)` reads (it is called
// with e < n only and must not fault), `put(e, v)` stores.  Written as two unrolled passes because a plain
// `for (e...) lds[e] = g[...]` loop compiles to one read, one wait and one store per trip, and a workgroup that stages
// a few thousand values that way spends most of its life in a dozen memory round trips one after another.
template <int U, typename V, typename Get, typename Put>
__device__ __forceinline__ void staged_fill(int n, Get get, Put put) {
    const int step = (int)blockDim.x;
    for (int base = (int)threadIdx.x; base < n; base += U * step) {
        V v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = get(min(base + u * step, n - 1));
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (base + u * step < n) put(base + u * step, v[u]);
    }
}

// The two halves of staged_fill for one batch of U slots starting at slot `first`, so that a kernel can put the
// reads of several regions (filter bank, images) in flight before it stores any of them.
template <int U, typename V, typename Get>
__device__ __forceinline__ void batch_read(V (&v)[U], int first, int n, Get get) {
    const int step = (int)blockDim.x, base = first + (int)threadIdx.x;
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = get(min(base + u * step, n - 1));
}
template <int U, typename V, typename Put>
__device__ __forceinline__ void batch_store(const V (&v)[U], int first, int n, Put put) {
    const int step = (int)blockDim.x, base = first + (int)threadIdx.x;
#pragma unroll
    for (int u = 0; u < U; ++u)
        if (base + u * step < n) put(base + u * step, v[u]);
}
// slots [first, n) by staged_fill
template <int U, typename V, typename Get, typename Put>
__device__ __forceinline__ void staged_fill_from(int first, int n, Get get, Put put) {
    const int step = (int)blockDim.x;
    for (int base = first + (int)threadIdx.x; base < n; base += U * step) {
        V v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = get(min(base + u * step, n - 1));
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (base + u * step < n) put(base + u * step, v[u]);
    }
}

template <typename T, int OCT, bool POOL>
__global__ __launch_bounds__(256) void conv2_direct_kernel(const T *__restrict__ x, const T *__restrict__ w,
                                                            const T *__restrict__ bias, T *__restrict__ y,
                                                            ConvParams p) {
    extern __shared__ __align__(16) float smem_f[];
    const int taps = p.ic * p.fh * p.fw;
    float *ws = smem_f;                         // [taps][ocpad]
    float *xs = smem_f + (size_t)taps * p.ocpad;  // [imgs][ic][ih][iw]
    const int img_sz = p.ic * p.ih * p.iw;
    const int b0 = blockIdx.x * p.imgs;
    const int nimg = min(p.imgs, p.bs - b0);

    staged_fill<8, T>(
        taps * p.ocpad,
        [&](int e) {
            const int tap = e / p.ocpad, o = min(e - tap * p.ocpad, p.oc - 1);
            return w[(size_t)o * taps + tap];
        },
        [&](int e, T v) { ws[e] = (e % p.ocpad) < p.oc ? Elem<T>::to_f32(v) : 0.0f; });
    const T *xb = x + (size_t)b0 * img_sz;
    staged_fill<8, T>(nimg * img_sz, [&](int e) { return xb[e]; }, [&](int e, T v) { xs[e] = Elem<T>::to_f32(v); });
    __syncthreads();

    constexpr int NPIX = POOL ? 4 : 1;
    const int total = nimg * p.items_per_img;
    for (int item = threadIdx.x; item < total; item += blockDim.x) {
        uint32_t img, r0, grp, pix, py, px;
        p.div_items.divmod((uint32_t)item, img, r0);
        p.div_pix.divmod(r0, grp, pix);  // pixel fastest: neighbouring lanes write neighbouring outputs
        p.div_yw.divmod(pix, py, px);
        const float *xi = xs + (size_t)img * img_sz;
        const float *wg = ws + grp * OCT;

        float acc[NPIX][OCT];
#pragma unroll
        for (int a = 0; a < NPIX; ++a)
#pragma unroll
            for (int o = 0; o < OCT; ++o) acc[a][o] = 0.0f;
        // top-left input coordinate of each of the NPIX output pixels
        int h0[NPIX], w0[NPIX];
#pragma unroll
        for (int a = 0; a < NPIX; ++a) {
            const int ho = POOL ? 2 * (int)py + (a >> 1) : (int)py;
            const int wo = POOL ? 2 * (int)px + (a & 1) : (int)px;
            h0[a] = -p.ph + p.sh * ho;
            w0[a] = -p.pw + p.sw * wo;
        }
        int tap = 0;
        for (int ci = 0; ci < p.ic; ++ci) {
            const float *xc = xi + ci * p.ih * p.iw;
            for (int fi = 0; fi < p.fh; ++fi)
                for (int fj = 0; fj < p.fw; ++fj, ++tap) {
                    float wv[OCT];
#pragma unroll
                    for (int o = 0; o < OCT; ++o) wv[o] = wg[tap * p.ocpad + o];
#pragma unroll
                    for (int a = 0; a < NPIX; ++a) {
                        const int hi = h0[a] + fi * p.dh, wi = w0[a] + fj * p.dw;
                        const bool ok = hi >= 0 && hi < p.ih && wi >= 0 && wi < p.iw;
                        const float v = ok ? xc[hi * p.iw + wi] : 0.0f;
#pragma unroll
                        for (int o = 0; o < OCT; ++o) acc[a][o] = __builtin_fmaf(v, wv[o], acc[a][o]);
                    }
                }
        }
#pragma unroll
        for (int o = 0; o < OCT; ++o) {
            const int oc = grp * OCT + o;
            const bool live = oc < p.oc;  // (no `continue`: the loop must unroll so acc stays in registers)
            const T bv = (p.has_bias && live) ? bias[oc] : Elem<T>::zero();
            T m = round_bias_relu<T>(acc[0][o], p.has_bias != 0, bv, p.act);
            if (POOL) {
                float mf = Elem<T>::to_f32(m);
#pragma unroll
                for (int a = 1; a < NPIX; ++a) {
                    const T v = round_bias_relu<T>(acc[a][o], p.has_bias != 0, bv, p.act);
                    const float vf = Elem<T>::to_f32(v);
                    if (vf > mf) { m = v; mf = vf; }
                }
            }
            if (live) y[(((size_t)(b0 + img) * p.oc + oc) * p.yh + py) * p.yw + px] = m;
        }
    }
}

// ---- row-tiled variant for stride 1, dilation 1 (any padding) ----
//
// A work item computes WT = 8 consecutive output pixels of one output row - or, with the pool
// fused, of a PAIR of rows, i.e. four whole pool windows - for OCT output channels.  The staged
// image is zero-padded in LDS, so the inner loop has no bounds checks: per (channel, input row)
// it reads WT + FW - 1 input values once (three 16-byte LDS reads) and the FW x OCT filter values
// of the filter row(s) that input row meets (uniform addresses, LDS broadcasts), then does up to
// 2 * FW * WT * OCT FMAs out of registers - about 12 FMAs per LDS read instead of 3.
struct RowTileParams {
    int bs, ic, ih, iw, oc, oh, ow, fh, ph, pw;
    int act, has_bias;
    int imgs, ngroups, ocpad;
    int ihp, pitch;       // padded rows staged per channel, LDS row pitch (floats, multiple of 4)
    int nwb;              // WT-wide blocks per output row
    int nrows;            // output rows (or row pairs with the pool) per image
    int yh, yw;
    int items_per_img;
    FastDiv div_items, div_rowsxwb, div_nwb, div_ocpad, div_pitch, div_ihp;
};

template <typename T, int FW, int OCT, bool POOL, int FHC>  // FHC: the filter height when it equals FW, else 0 (run time)
__global__ __launch_bounds__(256) void conv2_rowtile_kernel(const T *__restrict__ x, const T *__restrict__ w,
                                                             const T *__restrict__ bias, T *__restrict__ y,
                                                             RowTileParams p) {
    constexpr int WT = 8, NR = POOL ? 2 : 1, XW = WT + FW - 1, XV = (XW + 3) / 4;
    extern __shared__ __align__(16) float smem_f[];
    // a filter height known at compile time unrolls the row loop: which filter row an input row meets is then decided
    // at compile time, not by branches around every group of FMAs (LeNet5 conv1: 10.3 -> 9.0 us)
    constexpr int kUnrollRows = FHC ? FHC + (POOL ? 1 : 0) : 1;
    const int fh = FHC ? FHC : p.fh;
    const int taps = p.ic * fh * FW;
    float *ws = smem_f;                                         // [ic][fh][FW][ocpad]
    float *xs = smem_f + (((size_t)taps * p.ocpad + 3) & ~(size_t)3);  // [imgs][ic][ihp][pitch], zero padded
    const int ch_sz = p.ihp * p.pitch, img_sz = p.ic * ch_sz;
    const int b0 = blockIdx.x * p.imgs;
    const int nimg = min(p.imgs, p.bs - b0);

    staged_fill<8, T>(
        taps * p.ocpad,
        [&](int e) {
            uint32_t tap, o;
            p.div_ocpad.divmod((uint32_t)e, tap, o);
            return w[(size_t)min((int)o, p.oc - 1) * taps + tap];
        },
        [&](int e, T v) {
            uint32_t tap, o;
            p.div_ocpad.divmod((uint32_t)e, tap, o);
            ws[e] = (int)o < p.oc ? Elem<T>::to_f32(v) : 0.0f;
        });
    // the padding cells read the nearest cell of the image (a valid address) and store zero
    auto cell = [&](int e, int &hi, int &wi) -> size_t {
        uint32_t r1, col, r2, row;  // r2 = img * ic + channel
        p.div_pitch.divmod((uint32_t)e, r1, col);
        p.div_ihp.divmod(r1, r2, row);
        hi = (int)row - p.ph;
        wi = (int)col - p.pw;
        return ((size_t)b0 * p.ic + r2) * p.ih * p.iw;
    };
    staged_fill<8, T>(
        nimg * img_sz,
        [&](int e) {
            int hi, wi;
            const size_t plane = cell(e, hi, wi);
            return x[plane + (size_t)min(max(hi, 0), p.ih - 1) * p.iw + min(max(wi, 0), p.iw - 1)];
        },
        [&](int e, T v) {
            int hi, wi;
            cell(e, hi, wi);
            xs[e] = (hi >= 0 && hi < p.ih && wi >= 0 && wi < p.iw) ? Elem<T>::to_f32(v) : 0.0f;
        });
    __syncthreads();

    const int total = nimg * p.items_per_img;
    for (int item = threadIdx.x; item < total; item += blockDim.x) {
        uint32_t img, r0, grp, r1, row, wb;
        p.div_items.divmod((uint32_t)item, img, r0);
        p.div_rowsxwb.divmod(r0, grp, r1);
        p.div_nwb.divmod(r1, row, wb);
        const int ho0 = POOL ? 2 * (int)row : (int)row;  // first output row of this item
        const float *xi = xs + (size_t)img * img_sz + ho0 * p.pitch + wb * WT;
        const float *wg = ws + grp * OCT;

        float acc[NR][WT][OCT];
#pragma unroll
        for (int a = 0; a < NR; ++a)
#pragma unroll
            for (int t = 0; t < WT; ++t)
#pragma unroll
                for (int o = 0; o < OCT; ++o) acc[a][t][o] = 0.0f;

        for (int ci = 0; ci < p.ic; ++ci) {
            const float *xc = xi + ci * ch_sz;
            const float *wc = wg + (size_t)ci * fh * FW * p.ocpad;
            // input row r (relative to ho0) meets filter row r of output row 0 and r-1 of output row 1
#pragma unroll kUnrollRows
            for (int r = 0; r < fh + NR - 1; ++r) {
                float xin[XV * 4];
#pragma unroll
                for (int v = 0; v < XV; ++v) {
                    const float4 q = *(const float4 *)(xc + r * p.pitch + 4 * v);
                    xin[4 * v + 0] = q.x; xin[4 * v + 1] = q.y; xin[4 * v + 2] = q.z; xin[4 * v + 3] = q.w;
                }
#pragma unroll
                for (int a = 0; a < NR; ++a) {
                    const int fi = r - a;
                    if (fi >= 0 && fi < fh) {
                        const float *wr = wc + fi * FW * p.ocpad;
#pragma unroll
                        for (int fj = 0; fj < FW; ++fj) {
                            float wv[OCT];
#pragma unroll
                            for (int o = 0; o < OCT; ++o) wv[o] = wr[fj * p.ocpad + o];
#pragma unroll
                            for (int t = 0; t < WT; ++t)
#pragma unroll
                                for (int o = 0; o < OCT; ++o)
                                    acc[a][t][o] = __builtin_fmaf(xin[t + fj], wv[o], acc[a][t][o]);
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int o = 0; o < OCT; ++o) {
            const int oc = grp * OCT + o;
            const bool live = oc < p.oc;
            const T bv = (p.has_bias && live) ? bias[oc] : Elem<T>::zero();
            T *yp = y + (((size_t)(b0 + img) * p.oc + (live ? oc : 0)) * p.yh + row) * p.yw;
            if (POOL) {
#pragma unroll
                for (int j = 0; j < WT / 2; ++j) {
                    // window in row-major order: (0,2j) (0,2j+1) (1,2j) (1,2j+1); first strict maximum wins
                    T m = round_bias_relu<T>(acc[0][2 * j][o], p.has_bias != 0, bv, p.act);
                    float mf = Elem<T>::to_f32(m);
                    const T v1 = round_bias_relu<T>(acc[0][2 * j + 1][o], p.has_bias != 0, bv, p.act);
                    const T v2 = round_bias_relu<T>(acc[NR - 1][2 * j][o], p.has_bias != 0, bv, p.act);
                    const T v3 = round_bias_relu<T>(acc[NR - 1][2 * j + 1][o], p.has_bias != 0, bv, p.act);
                    float f = Elem<T>::to_f32(v1);
                    if (f > mf) { m = v1; mf = f; }
                    f = Elem<T>::to_f32(v2);
                    if (f > mf) { m = v2; mf = f; }
                    f = Elem<T>::to_f32(v3);
                    if (f > mf) { m = v3; mf = f; }
                    const int px = wb * (WT / 2) + j;
                    if (live && px < p.yw) yp[px] = m;
                }
            } else {
#pragma unroll
                for (int t = 0; t < WT; ++t) {
                    const int px = wb * WT + t;
                    if (live && px < p.yw) yp[px] = round_bias_relu<T>(acc[0][t][o], p.has_bias != 0, bv, p.act);
                }
            }
        }
    }
}

// ---- few channels, small images: implicit GEMM on v_mfma_f32_16x16x4_f32 ----
//
// The layers of small networks (LeNet5's conv2: 6 -> 16 channels on 12 x 12 images) have too few outputs per image to
// fill the chip with register tiles and too many multiply-adds per output (150) for one thread each: the row-tiled
// kernel spends 17 us on conv2 at batch 1000, three quarters of it a single wave per SIMD walking its 2400 FMAs.
// Here the same staged (zero-padded) images feed the matrix pipes: a 16 x 16 x 4 MFMA takes 16 output positions of one
// image (rows), up to 16 output channels (columns) and 4 taps.  The A operand is gathered straight from the staged
// image, one 4-byte LDS read per lane (position base + tap offset; the offsets of all taps sit in a small LDS table);
// the B operand is the filter bank as [tap][16] in LDS.  With the pool fused, the 16 rows of a tile are 4 whole 2 x 2
// windows, cell-minor: the accumulator layout (lane group g holds rows 4g .. 4g+3) then leaves each lane one complete
// window of one channel, and bias, ReLU and the first-strict-maximum pooling happen in registers.
// A wave takes (image, TG consecutive tiles) units; the k loop runs in chunks of 8 steps whose B values and tap
// offsets are fetched one chunk ahead.  f32 accumulation like every other kernel here; the summation order over the
// taps differs from the row-tiled kernel's (4 partial chains), which the f32 tolerance of the tests covers.
struct SmallMfmaParams {
    int bs, ic, ih, iw, oc, oh, ow, fh, fw, ph, pw;
    int act, has_bias;
    int imgs;           // images per workgroup
    int ihp, pitch;     // staged rows per channel and their pitch (floats)
    int ktot, ksteps;   // taps; k steps of 4 (a multiple of 8, the taps beyond ktot multiply zeros)
    int nout;           // results per image and channel: positions, or windows with the pool
    int mtiles;         // 16-row tiles per image
    int units_per_img;  // ceil(mtiles / TG)
    int yw;             // width of the result (pooled or not)
    FastDiv div_pitch, div_ihp, div_yw, div_fw, div_fhfw, div_upi;
};
typedef float f32x4_t __attribute__((ext_vector_type(4)));

template <typename T, bool POOL, int TG>
__global__ __launch_bounds__(256) void conv2_small_mfma_kernel(const T *__restrict__ x, const T *__restrict__ w,
                                                                const T *__restrict__ bias, T *__restrict__ y,
                                                                SmallMfmaParams p) {
    extern __shared__ __align__(16) float smem_f[];
    const int kpad = p.ksteps * 4;
    float *Bs = smem_f;                          // [kpad][16]
    int *tapoff = (int *)(smem_f + kpad * 16);   // [kpad], byte offsets into a staged image
    float *xs = smem_f + kpad * 17;              // [imgs][ic][ihp][pitch], zero padded
    const int ch_sz = p.ihp * p.pitch, img_sz = p.ic * ch_sz;
    const int b0 = blockIdx.x * p.imgs;
    const int nimg = min(p.imgs, p.bs - b0);

    for (int k = threadIdx.x; k < kpad; k += blockDim.x) {
        uint32_t ci, rem, fi, fj;
        p.div_fhfw.divmod((uint32_t)min(k, p.ktot - 1), ci, rem);
        p.div_fw.divmod(rem, fi, fj);
        tapoff[k] = (int)(ci * ch_sz + fi * p.pitch + fj) * 4;
    }
    // a padding cell reads the nearest cell of the image (a valid address) and stores zero
    auto cell = [&](int e, int &hi, int &wi) -> size_t {
        uint32_t r1, col, r2, row;  // r2 = img * ic + channel
        p.div_pitch.divmod((uint32_t)e, r1, col);
        p.div_ihp.divmod(r1, r2, row);
        hi = (int)row - p.ph;
        wi = (int)col - p.pw;
        return ((size_t)b0 * p.ic + r2) * p.ih * p.iw;
    };
    const int nw = kpad * 16, nx = nimg * img_sz;
    auto get_w = [&](int e) { return w[(size_t)min(e & 15, p.oc - 1) * p.ktot + min(e >> 4, p.ktot - 1)]; };
    auto put_w = [&](int e, T v) { Bs[e] = ((e & 15) < p.oc && (e >> 4) < p.ktot) ? Elem<T>::to_f32(v) : 0.0f; };
    constexpr int WU = 12, XU = 8;
    T wv[WU], xv[XU];
    batch_read<WU>(wv, 0, nw, get_w);
    if (p.ph == 0 && p.pw == 0) {  // nothing to pad: the staged images are a copy
        const T *xb = x + (size_t)b0 * img_sz;
        auto get_x = [&](int e) { return xb[e]; };
        auto put_x = [&](int e, T v) { xs[e] = Elem<T>::to_f32(v); };
        batch_read<XU>(xv, 0, nx, get_x);
        batch_store<WU>(wv, 0, nw, put_w);
        batch_store<XU>(xv, 0, nx, put_x);
        staged_fill_from<8, T>(XU * (int)blockDim.x, nx, get_x, put_x);
    } else {
        auto get_x = [&](int e) {
            int hi, wi;
            const size_t plane = cell(e, hi, wi);
            return x[plane + (size_t)min(max(hi, 0), p.ih - 1) * p.iw + min(max(wi, 0), p.iw - 1)];
        };
        auto put_x = [&](int e, T v) {
            int hi, wi;
            cell(e, hi, wi);
            xs[e] = (hi >= 0 && hi < p.ih && wi >= 0 && wi < p.iw) ? Elem<T>::to_f32(v) : 0.0f;
        };
        batch_read<XU>(xv, 0, nx, get_x);
        batch_store<WU>(wv, 0, nw, put_w);
        batch_store<XU>(xv, 0, nx, put_x);
        staged_fill_from<8, T>(XU * (int)blockDim.x, nx, get_x, put_x);
    }
    staged_fill_from<8, T>(WU * (int)blockDim.x, nw, get_w, put_w);
    __syncthreads();

    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, g = lane >> 4, i = lane & 15;
    const int nunits = nimg * p.units_per_img;
    const char *Bl = (const char *)(Bs + lane);
    const char *tl = (const char *)(tapoff + g);
    for (int u = wave; u < nunits; u += 4) {
        uint32_t img, ug;
        p.div_upi.divmod((uint32_t)u, img, ug);
        const int tile0 = (int)ug * TG;
        // this lane's A row of every tile: byte offset of the position's top-left input cell in LDS
        const char *abase[TG];
#pragma unroll
        for (int t = 0; t < TG; ++t) {
            const int tile = min(tile0 + t, p.mtiles - 1);
            uint32_t oy, ox;
            if (POOL) {
                uint32_t py, px;
                p.div_yw.divmod((uint32_t)min(tile * 4 + (i >> 2), p.nout - 1), py, px);
                oy = 2 * py + ((i >> 1) & 1);
                ox = 2 * px + (i & 1);
            } else {
                p.div_yw.divmod((uint32_t)min(tile * 16 + i, p.nout - 1), oy, ox);
            }
            abase[t] = (const char *)(xs + (size_t)img * img_sz + oy * p.pitch + ox);
        }
        f32x4_t acc[TG];
#pragma unroll
        for (int t = 0; t < TG; ++t) acc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
        float bq[8];
        int tq[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            bq[q] = *(const float *)(Bl + q * 256);
            tq[q] = *(const int *)(tl + q * 16);
        }
        for (int s0 = 0; s0 < p.ksteps; s0 += 8) {
            float bc[8];
            int tc[8];
#pragma unroll
            for (int q = 0; q < 8; ++q) { bc[q] = bq[q]; tc[q] = tq[q]; }
            if (s0 + 8 < p.ksteps) {
#pragma unroll
                for (int q = 0; q < 8; ++q) {
                    bq[q] = *(const float *)(Bl + (s0 + 8 + q) * 256);
                    tq[q] = *(const int *)(tl + (s0 + 8 + q) * 16);
                }
            }
            // the taps behind ktot multiply zeros of the bank; their A values are zeroed too (0 * inf would poison the
            // sum), which only the last chunk has to look at
            const bool tail = s0 + 8 >= p.ksteps;
#pragma unroll
            for (int q = 0; q < 8; ++q)
#pragma unroll
                for (int t = 0; t < TG; ++t) {
                    float a = *(const float *)(abase[t] + tc[q]);
                    if (tail && 4 * (s0 + q) + g >= p.ktot) a = 0.0f;
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, bc[q], acc[t], 0, 0, 0);
                }
        }
        // lane (g, i) holds rows 4g .. 4g+3 of column i: one window (pool) or 4 consecutive positions of channel i
        const bool live = i < p.oc;
        const T bv = (p.has_bias && live) ? bias[i] : Elem<T>::zero();
        T *yc = y + ((size_t)(b0 + img) * p.oc + (live ? i : 0)) * p.nout;
#pragma unroll
        for (int t = 0; t < TG; ++t) {
            const int tile = tile0 + t;
            if (tile >= p.mtiles) break;
            if (POOL) {
                T m = round_bias_relu<T>(acc[t][0], p.has_bias != 0, bv, p.act);
                float mf = Elem<T>::to_f32(m);
#pragma unroll
                for (int r = 1; r < 4; ++r) {
                    const T v = round_bias_relu<T>(acc[t][r], p.has_bias != 0, bv, p.act);
                    const float f = Elem<T>::to_f32(v);
                    if (f > mf) { m = v; mf = f; }
                }
                const int wi = tile * 4 + g;
                if (live && wi < p.nout) yc[wi] = m;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int pos = tile * 16 + 4 * g + r;
                    if (live && pos < p.nout) yc[pos] = round_bias_relu<T>(acc[t][r], p.has_bias != 0, bv, p.act);
                }
            }
        }
    }
}

template <typename T, bool POOL>
int launch_oct(int oct, dim3 grid, dim3 block, size_t smem, const T *x, const T *w, const T *bias, T *y,
               const ConvParams &p) {
    switch (oct) {
        case 1: hipLaunchKernelGGL((conv2_direct_kernel<T, 1, POOL>), grid, block, smem, stream(), x, w, bias, y, p); break;
        case 2: hipLaunchKernelGGL((conv2_direct_kernel<T, 2, POOL>), grid, block, smem, stream(), x, w, bias, y, p); break;
        case 4: hipLaunchKernelGGL((conv2_direct_kernel<T, 4, POOL>), grid, block, smem, stream(), x, w, bias, y, p); break;
        case 6: hipLaunchKernelGGL((conv2_direct_kernel<T, 6, POOL>), grid, block, smem, stream(), x, w, bias, y, p); break;
        default: hipLaunchKernelGGL((conv2_direct_kernel<T, 8, POOL>), grid, block, smem, stream(), x, w, bias, y, p); break;
    }
    return AGH_OK;
}

// What conv2_direct_entry chooses by, with the 2x2 pool fused or without.
struct ConvShape {
    int64_t bs, ic, ih, iw, oc, fh, fw, ph, pw, sh, sw, dh, dw, oh, ow;
    int small_forced;  // AGH_CONV_SMALL: 0 / 1 forces the choice of conv2_small_mfma_kernel (measurements), -1 by size
    bool unit() const { return sh == 1 && sw == 1 && dh == 1 && dw == 1; }
};
constexpr int64_t kConvLds = 64 * 1024;
inline int64_t conv_cus() { return compute_units() > 0 ? compute_units() : 256; }

// up to 16 output channels over enough taps on small images: matrix cores fed from the staged image
bool conv2_small_plan(const ConvShape &c, bool pool, SmallMfmaParams &q, int64_t &fixed_bytes, int64_t &img_bytes) {
    if (!c.unit() || c.oc > 16) return false;
    const int64_t taps = c.ic * c.fh * c.fw;
    const bool want = c.small_forced >= 0 ? c.small_forced != 0 : (c.oc >= 8 && taps >= 32);
    q.bs = (int)c.bs; q.ic = (int)c.ic; q.ih = (int)c.ih; q.iw = (int)c.iw; q.oc = (int)c.oc; q.oh = (int)c.oh; q.ow = (int)c.ow;
    q.fh = (int)c.fh; q.fw = (int)c.fw; q.ph = (int)c.ph; q.pw = (int)c.pw;
    q.ihp = (int)(c.ih + 2 * c.ph);
    q.pitch = (int)(c.iw + 2 * c.pw);
    q.ktot = (int)taps;
    q.ksteps = (int)((taps + 31) / 32 * 8);
    const int64_t yh = pool ? c.oh / 2 : c.oh, yw = pool ? c.ow / 2 : c.ow;
    fixed_bytes = (int64_t)q.ksteps * 4 * 17 * 4;
    img_bytes = c.ic * (int64_t)q.ihp * q.pitch * 4;
    return want && taps <= 2048 && fixed_bytes + img_bytes <= kConvLds && yh * yw <= ((int64_t)1 << 20);
}

// stride 1, dilation 1, filter width 3 or 5: row-tiled kernel.  walk_us: what its work items are expected to take.
struct LdsPlan {
    int oct;
    int64_t items, imgs, w_bytes, img_bytes;
    double walk_us;
};
bool conv2_rowtile_plan(const ConvShape &c, bool pool, RowTileParams &q, LdsPlan &l) {
    if (!c.unit() || (c.fw != 3 && c.fw != 5)) return false;
    q.bs = c.bs; q.ic = c.ic; q.ih = c.ih; q.iw = c.iw; q.oc = c.oc; q.oh = c.oh; q.ow = c.ow; q.fh = c.fh; q.ph = c.ph; q.pw = c.pw;
    // two output channels per work item unless that leaves fewer than ~4 waves per CU in flight
    const int64_t rows0 = pool ? c.oh / 2 : c.oh, wbs0 = (c.ow + 7) / 8;
    l.oct = (c.oc <= 1 || c.bs * rows0 * wbs0 * ((c.oc + 1) / 2) < conv_cus() * 4 * 64) ? 1 : 2;
    q.ngroups = (c.oc + l.oct - 1) / l.oct;
    q.ocpad = q.ngroups * l.oct;
    q.nwb = (c.ow + 7) / 8;
    q.ihp = c.ih + 2 * c.ph;
    int64_t pitch = c.iw + 2 * c.pw;
    if (pitch < q.nwb * 8 + c.fw - 1) pitch = q.nwb * 8 + c.fw - 1;
    // whole 16-byte reads of WT + FW - 1 floats starting at a multiple of 8
    const int64_t xw4 = ((8 + c.fw - 1 + 3) / 4) * 4;
    if (pitch < (q.nwb - 1) * 8 + xw4) pitch = (q.nwb - 1) * 8 + xw4;
    q.pitch = (int)((pitch + 3) & ~(int64_t)3);
    q.yh = pool ? c.oh / 2 : c.oh;
    q.yw = pool ? c.ow / 2 : c.ow;
    q.nrows = q.yh;
    const int64_t taps = c.ic * c.fh * c.fw;
    l.items = (int64_t)q.nrows * q.nwb * q.ngroups;
    l.w_bytes = ((taps * q.ocpad + 3) & ~(int64_t)3) * 4;
    l.img_bytes = (int64_t)c.ic * q.ihp * q.pitch * 4;
    if (l.w_bytes + l.img_bytes > kConvLds || l.items > ((int64_t)1 << 24)) return false;
    l.imgs = l.items >= 256 ? 1 : 256 / l.items;
    while (l.imgs > 1 && l.w_bytes + l.imgs * l.img_bytes > kConvLds) --l.imgs;
    while (l.imgs > 1 && (c.bs + l.imgs - 1) / l.imgs < conv_cus()) --l.imgs;
    if (l.imgs > c.bs) l.imgs = c.bs;
    // one image per workgroup is a long walk where there are many channels and few images
    l.walk_us = (double)((l.imgs * l.items + 255) / 256) * (1.0 + 0.04 * (double)(taps * l.oct)) *
                std::max(1.0, (double)((c.bs + l.imgs - 1) / l.imgs) / (2.0 * (double)conv_cus()));
    return true;
}

// any geometry whose image and filter bank fit in LDS
bool conv2_lds_plan(const ConvShape &c, bool pool, ConvParams &p, LdsPlan &l) {
    p.bs = c.bs; p.ic = c.ic; p.ih = c.ih; p.iw = c.iw; p.oc = c.oc; p.oh = c.oh; p.ow = c.ow;
    p.fh = c.fh; p.fw = c.fw; p.ph = c.ph; p.pw = c.pw; p.sh = c.sh; p.sw = c.sw; p.dh = c.dh; p.dw = c.dw;
    p.yh = pool ? c.oh / 2 : c.oh;
    p.yw = pool ? c.ow / 2 : c.ow;
    // output channels per work item: the whole bank when it is small, else groups of 8
    l.oct = 8;
    for (int o : {1, 2, 4, 6, 8})
        if (c.oc <= o) { l.oct = o; break; }
    p.ngroups = (c.oc + l.oct - 1) / l.oct;
    p.ocpad = p.ngroups * l.oct;
    const int64_t taps = c.ic * c.fh * c.fw;
    l.items = (int64_t)p.yh * p.yw * p.ngroups;
    l.img_bytes = c.ic * c.ih * c.iw * 4;
    l.w_bytes = taps * p.ocpad * 4;
    if (l.w_bytes + l.img_bytes > kConvLds || l.items > ((int64_t)1 << 24)) return false;
    // images per workgroup: aim at ~256 work items, stay inside LDS, keep >= 2 workgroups per CU
    l.imgs = l.items >= 256 ? 1 : 256 / l.items;
    while (l.imgs > 1 && l.w_bytes + l.imgs * l.img_bytes > kConvLds) --l.imgs;
    while (l.imgs > 1 && (c.bs + l.imgs - 1) / l.imgs < 2 * conv_cus()) --l.imgs;
    if (l.imgs > c.bs) l.imgs = c.bs;
    l.walk_us = (double)((l.imgs * l.items + 255) / 256) * (1.5 + 0.02 * (double)(taps * l.oct)) *
                std::max(1.0, (double)((c.bs + l.imgs - 1) / l.imgs) / (2.0 * (double)conv_cus()));
    return true;
}

// The time below which the matrix-core kernel of any geometry (agh_conv_taps.hip) is taken for the convolution without the
// pool, against what would run in its place.
template <typename T>
double conv2_taps_limit(const ConvShape &c) {
    SmallMfmaParams sq;
    RowTileParams rq;
    ConvParams p;
    LdsPlan l;
    int64_t fixed_bytes, img_bytes;
    if (conv2_small_plan(c, false, sq, fixed_bytes, img_bytes)) return 0.0;
    // 1 x 3 x 32 x 109 to 64 channels, 5 x 5, 1007 us on row tiles and 14 us on the matrix cores; 64 x 3 x 64 x 64 to 64,
    // 3 x 3, 253 and 27
    if (conv2_rowtile_plan(c, false, rq, l)) return 0.7 * l.walk_us;
    // 5 x 1 x 108 x 108 to 48, 5 x 5 stride 2: 289 and 14 us
    if (conv2_lds_plan(c, false, p, l)) return 0.7 * l.walk_us;
    // otherwise im2col and a product: the patch matrix written and read (faster while the last-level cache holds it; bf16 rows
    // of no whole 16 bytes go through the any-address kernel), 64 channels at least; 30 us for the calls, as a Python program
    // makes them (a captured graph or a C++ program waits for the device alone, where one in five of the shapes taken is slower, the
    // worst 2.2 times).  Fitted to 2600 shapes; of 1000 others three run more than 3 % behind the route not taken (the worst
    // 22 %), all of them together 1.76 times as fast as without this kernel.
    // Taken: 64 x 3 x 95 x 95 to 64, 7 x 7 stride 2, f32 76 -> 42 us; 64 x 24 x 30 x 30 to 48, 3 x 3, f32 57 -> 23, bf16 35 -> 25.
    // Not taken: 64 x 64 x 56 x 56 to 128, 3 x 3 stride 2, f32 106 (here 149), bf16 39 (157); 205 x 3 x 50 x 50 to 128, 7 x 7,
    // bf16 153 (here 265).
    const int64_t taps = c.ic * c.fh * c.fw;
    const bool whole = taps * (int64_t)sizeof(T) % 16 == 0, ragged_bf16 = sizeof(T) == 2 && !whole;
    const double patch = (double)c.bs * c.oh * c.ow * taps * sizeof(T), flops = 2.0 * c.bs * c.oh * c.ow * taps * ((c.oc + 63) / 64 * 64);
    const double chain_us = 6.0 + 2.0 * patch / (ragged_bf16 ? 3e6 : patch < 128e6 ? 8e6 : 5e6) +
                            flops / (sizeof(T) == 4 ? (whole ? 100e6 : 50e6) : (whole ? 450e6 : 200e6));
    return 0.85 * std::max(30.0, chain_us);
}

template <typename T>
int conv2_direct_entry(const char *name, const void *x, const void *w, const void *bias, void *y, int64_t bs,
                       int64_t ic, int64_t ih, int64_t iw, int64_t oc, int64_t fh, int64_t fw, int64_t ph, int64_t pw,
                       int64_t sh, int64_t sw, int64_t dh, int64_t dw, int act, int pool2x2) {
    AGH_API_ENTER();
    if (bs < 0 || ic < 1 || ih < 1 || iw < 1 || oc < 1 || fh < 1 || fw < 1 || ph < 0 || pw < 0 || sh < 1 || sw < 1 ||
        dh < 1 || dw < 1)
        return fail(AGH_EINVAL, "%s: invalid shape/options", name);
    if (act != AGH_ACT_NONE && act != AGH_ACT_RELU) return fail(AGH_EINVAL, "%s: unknown activation %d", name, act);
    if (ih + 2 * ph < dh * (fh - 1) + 1 || iw + 2 * pw < dw * (fw - 1) + 1)
        return fail(AGH_EINVAL, "%s: filter (with dilation) larger than the padded input", name);
    const int64_t lim = 1 << 20;
    if (bs > ((int64_t)1 << 30) || ic > lim || ih > lim || iw > lim || oc > lim || fh > lim || fw > lim || ph > lim ||
        pw > lim || sh > lim || sw > lim || dh > lim || dw > lim)
        return fail(AGH_ERANGE, "%s: dimension too large", name);
    const int64_t oh = (ih + 2 * ph - dh * (fh - 1) - 1) / sh + 1, ow = (iw + 2 * pw - dw * (fw - 1) - 1) / sw + 1;
    if (pool2x2 && (oh < 2 || ow < 2)) return fail(AGH_EINVAL, "%s: output smaller than the 2x2 pool window", name);
    if (bs == 0) return AGH_OK;
    if (!x || !w || !y) return fail(AGH_ENULL, "%s: null buffer", name);

    // enough channels: implicit GEMM on the matrix cores (returns 1 when the geometry is not its own)
    // 0 forbids the kernels of any geometry, 1 forces the one on the f32 matrix cores, 2 that on the bf16 ones (measurements, tests)
    const char *env = setting("AGH_CONV_TAPS");
    const int taps_value = env && *env ? atoi(env) : -1;
    const bool taps16_forced = sizeof(T) == 2 && taps_value == 2;
    const int taps_forced = taps_value < 0 ? -1 : taps_value != 0 ? 1 : 0;
    const char *small_env = oc <= 16 ? setting("AGH_CONV_SMALL") : nullptr;
    const ConvShape shape = {bs, ic, ih, iw, oc, fh, fw, ph, pw, sh, sw, dh, dw, oh, ow, small_env ? atoi(small_env) != 0 : -1};
    if (shape.unit() && !pool2x2 && taps_forced != 1) {
        const int rc = conv2_mfma_try<T>(name, x, w, bias, y, bs, ic, ih, iw, oc, fh, fw, ph, pw, oh, ow, act);
        if (rc != 1) return rc;
    }

    // the matrix-core kernel of any geometry, where it expects to need less time than what would run in its place; with the
    // pool, where the convolution alone would run on it (the fused call returns the same bits as the separate layers)
    const double taps_limit = taps_forced != 0 ? conv2_taps_limit<T>(shape) : 0.0;
    // scratch memory that a capture cannot have for the bf16 kernel chosen: workspace() refuses it then, and says that the sequence has to run once eagerly
    size_t lacking = 0;
    void *unused = nullptr;
    const bool implicit_gemm_plain = pool2x2 && shape.unit() && conv2_mfma_takes<T>(x, w, bs, ic, ih, iw, oc, fh, fw, pw, oh, ow);
    if (sizeof(T) == 2 && (taps16_forced || (taps_forced < 0 && taps_limit >= kTapsLeastUs && !implicit_gemm_plain))) {
        double f32_us = 1e30;
        if (!taps16_forced)
            conv2_taps_try<T>(name, x, w, bias, y, bs, ic, ih, iw, oc, fh, fw, ph, pw, sh, sw, dh, dw, oh, ow, act, false, false, 0.0, &f32_us);
        // Where the f32 kernel would be taken otherwise, its second launch (the packed bank, 3 us of a program's time) has to be worth it:
        // two microseconds and a quarter of a time that is on the safe side (12 x 12 pixels, 32 to 16 channels, 3 x 3: 10.4 us there, 13.7 here).
        // Against im2col and a product a tenth is left for the estimate's error (33 x 128 x 12 x 76 to 256, 3 x 3: 74 us there, 83 here), and four tenths
        // where the filter bank streams through workgroups that take up to twice the estimate, or few of them through little work (7 x 256 x 47 x
        // 74 to 256, 5 x 5: 241 us there, 317 here; 2 x 256 x 17 x 9 to 96, 3 x 3: 20 and 28).  Of 240 shapes that were measured and the rule takes against
        // im2col none is slower than it was there, 0.19 to 0.99 of the time.
        const bool against_f32 = f32_us <= taps_limit;
        const double limit = against_f32 ? 0.75 * f32_us - 2.0 : 0.9 * taps_limit, wary_limit = against_f32 ? limit : 0.6 * taps_limit;
        const int rc = !taps16_forced && limit < kTaps16LeastUs
                           ? 1
                           : conv2_taps16_try(name, x, w, bias, y, bs, ic, ih, iw, oc, fh, fw, ph, pw, sh, sw, dh, dw, oh, ow, act, pool2x2 != 0,
                                              taps16_forced, limit, wary_limit, lacking);
        if (rc != 1) return rc;
        if (taps16_forced && lacking) return workspace(lacking, &unused);
        if (taps16_forced) return fail(AGH_ERANGE, "%s: AGH_CONV_TAPS=2, and that kernel does not take this shape", name);
    }
    if (taps_forced == 1 || (taps_limit >= kTapsLeastUs && !implicit_gemm_plain)) {
        const int rc = conv2_taps_try<T>(name, x, w, bias, y, bs, ic, ih, iw, oc, fh, fw, ph, pw, sh, sw, dh, dw, oh, ow, act, pool2x2 != 0,
                                         taps_forced == 1, taps_limit);
        if (rc != 1) return rc;
        if (taps_forced == 1) return fail(AGH_ERANGE, "%s: AGH_CONV_TAPS=1, and that kernel does not take this shape", name);
    }

    SmallMfmaParams sq;
    int64_t fixed_bytes = 0, small_img_bytes = 0;
    if (conv2_small_plan(shape, pool2x2 != 0, sq, fixed_bytes, small_img_bytes)) {
        SmallMfmaParams &q = sq;
        const int64_t img_bytes = small_img_bytes, yh = pool2x2 ? oh / 2 : oh, yw = pool2x2 ? ow / 2 : ow;
        q.act = act; q.has_bias = bias != nullptr;
        q.nout = (int)(yh * yw);
        q.yw = (int)yw;
        q.mtiles = (int)(pool2x2 ? (yh * yw + 3) / 4 : (yh * yw + 15) / 16);
        const int tg = q.mtiles >= 8 ? 4 : 2;
        q.units_per_img = (q.mtiles + tg - 1) / tg;
        {
            const int64_t cus = conv_cus();
            // a workgroup's four waves want a unit each; more images per workgroup only while the grid still
            // covers the chip twice
            int64_t imgs = std::max<int64_t>(1, 4 / q.units_per_img);
            while (fixed_bytes + (imgs + 1) * img_bytes <= kConvLds && (imgs + 1) * q.units_per_img <= 8 &&
                   (bs + imgs) / (imgs + 1) >= 2 * cus)
                ++imgs;
            while (imgs > 1 && fixed_bytes + imgs * img_bytes > kConvLds) --imgs;
            if (imgs > bs) imgs = bs;
            q.imgs = (int)imgs;
            q.div_pitch = FastDiv((uint32_t)q.pitch);
            q.div_ihp = FastDiv((uint32_t)q.ihp);
            q.div_yw = FastDiv((uint32_t)yw);
            q.div_fw = FastDiv((uint32_t)fw);
            q.div_fhfw = FastDiv((uint32_t)(fh * fw));
            q.div_upi = FastDiv((uint32_t)q.units_per_img);
            const int64_t blocks = (bs + imgs - 1) / imgs;
            if (blocks > 0x7FFFFFFF) return fail(AGH_ERANGE, "%s: too many workgroups", name);
            const size_t smem = (size_t)(fixed_bytes + imgs * img_bytes);
            const dim3 grid((unsigned)blocks), block(256);
            const T *xp = (const T *)x, *wp = (const T *)w, *bp = (const T *)bias;
            T *yp = (T *)y;
#define AGH_SM(POOLV, TGV) \
    hipLaunchKernelGGL((conv2_small_mfma_kernel<T, POOLV, TGV>), grid, block, smem, stream(), xp, wp, bp, yp, q)
            if (pool2x2) { if (tg == 4) AGH_SM(true, 4); else AGH_SM(true, 2); }
            else { if (tg == 4) AGH_SM(false, 4); else AGH_SM(false, 2); }
#undef AGH_SM
            AGH_LAUNCH_CHECK(name);
            return AGH_OK;
        }
    }

    // stride 1, dilation 1, filter width 3 or 5: row-tiled kernel
    LdsPlan l;
    {
        RowTileParams q;
        if (conv2_rowtile_plan(shape, pool2x2 != 0, q, l)) {
            const int oct = l.oct;
            const int64_t items = l.items, imgs = l.imgs;
            q.act = act; q.has_bias = bias != nullptr;
            q.imgs = (int)imgs;
            q.items_per_img = (int)items;
            q.div_items = FastDiv((uint32_t)items);
            q.div_rowsxwb = FastDiv((uint32_t)(q.nrows * q.nwb));
            q.div_nwb = FastDiv((uint32_t)q.nwb);
            q.div_ocpad = FastDiv((uint32_t)q.ocpad);
            q.div_pitch = FastDiv((uint32_t)q.pitch);
            q.div_ihp = FastDiv((uint32_t)q.ihp);
            const int64_t work = imgs * items;
            const int threads = work >= 256 ? 256 : (int)((work + 63) / 64 * 64);
            const int64_t blocks = (bs + imgs - 1) / imgs;
            if (blocks > 0x7FFFFFFF) return fail(AGH_ERANGE, "%s: too many workgroups", name);
            const size_t smem = (size_t)(l.w_bytes + imgs * l.img_bytes);
            const dim3 grid((unsigned)blocks), block(threads);
            const T *xp = (const T *)x, *wp = (const T *)w, *bp = (const T *)bias;
            T *yp = (T *)y;
#define AGH_RT(FWV, OCTV, POOLV) \
    do { \
        if (fh == FWV) hipLaunchKernelGGL((conv2_rowtile_kernel<T, FWV, OCTV, POOLV, FWV>), grid, block, smem, stream(), xp, wp, bp, yp, q); \
        else hipLaunchKernelGGL((conv2_rowtile_kernel<T, FWV, OCTV, POOLV, 0>), grid, block, smem, stream(), xp, wp, bp, yp, q); \
    } while (0)
            if (fw == 3) {
                if (oct == 1) { if (pool2x2) AGH_RT(3, 1, true); else AGH_RT(3, 1, false); }
                else { if (pool2x2) AGH_RT(3, 2, true); else AGH_RT(3, 2, false); }
            } else {
                if (oct == 1) { if (pool2x2) AGH_RT(5, 1, true); else AGH_RT(5, 1, false); }
                else { if (pool2x2) AGH_RT(5, 2, true); else AGH_RT(5, 2, false); }
            }
#undef AGH_RT
            AGH_LAUNCH_CHECK(name);
            return AGH_OK;
        }
    }

    ConvParams p;
    if (!conv2_lds_plan(shape, pool2x2 != 0, p, l)) {
        if (lacking) return workspace(lacking, &unused);
        return fail(AGH_ERANGE, "%s: image + filter bank (%lld bytes) do not fit in LDS; use im2col + gemm", name,
                    (long long)(l.w_bytes + l.img_bytes));
    }
    const int oct = l.oct;
    const int64_t items = l.items, imgs = l.imgs, pix = (int64_t)p.yh * p.yw;
    p.act = act; p.has_bias = bias != nullptr;
    p.imgs = (int)imgs;
    p.items_per_img = (int)items;
    p.div_items = FastDiv((uint32_t)items);
    p.div_pix = FastDiv((uint32_t)pix);
    p.div_yw = FastDiv((uint32_t)p.yw);
    int64_t work = imgs * items;
    int threads = work >= 256 ? 256 : (int)((work + 63) / 64 * 64);
    const int64_t blocks = (bs + imgs - 1) / imgs;
    if (blocks > 0x7FFFFFFF) return fail(AGH_ERANGE, "%s: too many workgroups", name);
    const size_t smem = (size_t)(l.w_bytes + imgs * l.img_bytes);
    if (pool2x2)
        launch_oct<T, true>(oct, dim3((unsigned)blocks), dim3(threads), smem, (const T *)x, (const T *)w, (const T *)bias,
                            (T *)y, p);
    else
        launch_oct<T, false>(oct, dim3((unsigned)blocks), dim3(threads), smem, (const T *)x, (const T *)w,
                             (const T *)bias, (T *)y, p);
    AGH_LAUNCH_CHECK(name);
    return AGH_OK;
}

}  // namespace

extern "C" {

int agh_conv2_direct_f32(const void *x, const void *w, const void *bias, void *y, int64_t bs, int64_t ic, int64_t ih,
                         int64_t iw, int64_t oc, int64_t fh, int64_t fw, int64_t ph, int64_t pw, int64_t sh,
                         int64_t sw, int64_t dh, int64_t dw, int act, int pool2x2) {
    return conv2_direct_entry<float>("agh_conv2_direct_f32", x, w, bias, y, bs, ic, ih, iw, oc, fh, fw, ph, pw, sh, sw,
                                     dh, dw, act, pool2x2);
}
int agh_conv2_direct_bf16(const void *x, const void *w, const void *bias, void *y, int64_t bs, int64_t ic, int64_t ih,
                          int64_t iw, int64_t oc, int64_t fh, int64_t fw, int64_t ph, int64_t pw, int64_t sh,
                          int64_t sw, int64_t dh, int64_t dw, int act, int pool2x2) {
    return conv2_direct_entry<uint16_t>("agh_conv2_direct_bf16", x, w, bias, y, bs, ic, ih, iw, oc, fh, fw, ph, pw, sh,
                                        sw, dh, dw, act, pool2x2);
}

}  // extern "C"
