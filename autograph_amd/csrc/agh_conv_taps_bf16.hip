// Conv2 forward on the bf16 matrix cores for any stride, dilation, channel count and row length: what the implicit GEMM of
// agh_conv_mfma.hip does not take (stride 2, rows or channels that are no whole vectors, few output channels).  Replaces im2col +
// GEMM there (src/learn/neural_network/layer.rs:950-1005).
//
// agh_conv_taps.hip does the same out of f32 copies of the staged rows on v_mfma_f32_16x16x4_f32, at a sixteenth of the bf16
// matrix rate.  Here a workgroup of four waves takes 64 * TG output positions of one image and 16 * NT channels, stages the
// zero-padded input rows that the positions touch as bf16, pixel major: a staged pixel is its channels in groups of eight (missing
// channels zero) and 16 bytes of padding.  A unit is eight channels of one tap, a step of v_mfma_f32_16x16x32_bf16 four units, one per
// 16-lane group: the A operand is one 16-byte LDS read per lane at the position's base + the unit's offset (a table in LDS), whatever
// the stride, and the B operand one 16-byte load of a copy of the filter bank in fragment order (as large as the bank; it stays in
// the L2s).  Channels whose rows do not fit into 64 KB of LDS, which leaves a CU two workgroups, are taken in passes.  Both operands of a step are
// requested one step (A) and kAhead steps (B) before it.
// What bounds it: latencies, of staging (2-byte reads) and of the bank's reads, with two workgroups a CU.  No unit is busy (counters of the first, third and
// fourth shape below: matrix pipes 18, 11 and 23 % of a launch, LDS 16, 11 and 21 % with half of it conflicts, L1s half an access a cycle; a wave waits
// for two thirds of its cycles).  Against the f32 matrix cores or im2col and a product, whichever it was (calls of a Python program, us):
// 149 x 32 x 32 x 23 to 48, 7 x 7 with padding 213 -> 35; 132 x 128 x 30 x 30 to 16, 7 x 7 317 -> 59; 126 x 32 x 76 x 76 to 48, 3 x 3 with padding 334 -> 67;
// 102 x 3 x 76 x 76 to 96, 7 x 7 with padding 172 -> 78.
#include <algorithm>
#include <type_traits>

#include "agh_internal.h"

using namespace agh;

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint16_t Any4 __attribute__((ext_vector_type(4), aligned(2)));  // four elements at any element address

struct Taps16Params {
    int ic, ih, iw, oc, ph, pw, sh, sw;
    int act, has_bias;
    int npos;           // output positions per image; with the pool, the 4 positions of every window
    int groups;         // groups of 8 channels staged per pass
    int passes, steps;  // steps of four units per pass
    int units;          // taps * groups
    int rows, cols;     // staged rows and columns per pass
    int pitch;          // bytes of a staged pixel
    int tab_bytes;
    int dh, dw;
    FastDiv div_ptiles, div_cols, div_rows, div_yw, div_groups, div_fw;  // yw: the result's row, of positions or windows
};

constexpr int kAhead = 3;  // steps by which the bank's fragments are requested ahead

// filter bank [oc][ic][taps] -> [tile of 16 channels][pass][step][lane][8]: lane (g, i) of step s holds unit 4 s + g of channel
// 16 tile + i; zero where a unit, a channel of a group or an output channel does not exist
__global__ __launch_bounds__(256) void taps16_pack_kernel(const uint16_t *__restrict__ w, uint4 *__restrict__ wp, int oc, int ic, int taps,
                                                          int groups, int units, int steps, int passes, uint32_t total) {
    const uint32_t e = blockIdx.x * 256 + threadIdx.x;  // one fragment of a lane
    if (e >= total) return;
    const uint32_t lane = e & 63, s = (e >> 6) % (uint32_t)steps, tp = (e >> 6) / (uint32_t)steps, pass = tp % (uint32_t)passes, tile = tp / (uint32_t)passes;
    const uint32_t u = 4 * s + (lane >> 4), tap = u / (uint32_t)groups, grp = u - tap * (uint32_t)groups;
    const int o = (int)(tile * 16 + (lane & 15)), c0 = (int)(pass * (uint32_t)groups + grp) * 8;
    const bool live = (int)u < units && o < oc;
    uint32_t v[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const uint32_t r = w[((size_t)min(o, oc - 1) * ic + min(c0 + c, ic - 1)) * taps + min((int)tap, taps - 1)];
        v[c] = live && c0 + c < ic ? r : 0u;
    }
    wp[e] = make_uint4(v[0] | v[1] << 16, v[2] | v[3] << 16, v[4] | v[5] << 16, v[6] | v[7] << 16);
}

// With the pool, positions are numbered window by window, the four of a window in row order: a lane's four accumulators are whole
// windows of one channel.  The order of a position's sums is the same either way, so the result is, bit for bit, the pool of what
// the call without it returns.
template <int TG, int NT, bool POOL>
__global__ __launch_bounds__(256, 2) void conv2_taps16_kernel(const uint16_t *__restrict__ x, const uint4 *__restrict__ wp,
                                                              const uint16_t *__restrict__ bias, uint16_t *__restrict__ y, Taps16Params p) {
    typedef uint16_t T;
    extern __shared__ __align__(16) unsigned char lds[];
    int *tab = (int *)lds;                       // [4 * (steps + 1)] byte offsets of the units from a position's first pixel
    unsigned char *xs = lds + p.tab_bytes;       // [rows][cols][pitch], zero padded
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, i = lane & 15;
    uint32_t b, tile;
    p.div_ptiles.divmod(blockIdx.x, b, tile);
    const int p0 = (int)tile * (64 * TG);
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
    const size_t plane = (size_t)p.ih * p.iw;
    const T *xb = x + (size_t)b * p.ic * plane;

    for (int u = threadIdx.x; u < 4 * (p.steps + 1); u += 256) {
        uint32_t tap, grp, fi, fj;
        p.div_groups.divmod((uint32_t)min(u, p.units - 1), tap, grp);
        p.div_fw.divmod(tap, fi, fj);
        tab[u] = ((int)fi * p.dh * p.cols + (int)fj * p.dw) * p.pitch + (int)grp * 16;
    }
    // positions behind the image's last repeat it; their results are not stored
    const int wp0 = p0 + wave * (16 * TG);
    const unsigned char *abase[TG];
#pragma unroll
    for (int t = 0; t < TG; ++t) {
        uint32_t oy, ox;
        output_at((uint32_t)min(wp0 + t * 16 + i, p.npos - 1), oy, ox);
        abase[t] = xs + ((int)(oy - oy0) * p.sh * p.cols + (int)ox * p.sw) * p.pitch;
    }
    // this lane's fragments of the NT channel tiles (a tile behind the last repeats it)
    const int n16 = (p.oc + 15) >> 4;
    const uint4 *bank[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) bank[n] = wp + (size_t)min((int)blockIdx.y * NT + n, n16 - 1) * p.passes * p.steps * 64 + lane;
    f32x4_t acc[TG][NT];
#pragma unroll
    for (int t = 0; t < TG; ++t)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[t][n] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};

    for (int pass = 0; pass < p.passes; ++pass) {
        if (pass) __syncthreads();
        // Stage: an item is eight channels of one pixel, eight 2-byte reads (consecutive lanes take consecutive pixels of a row) and
        // one 16-byte write; U items a thread in flight, addresses clamped, what lies outside the image or behind the last channel
        // stored as zero.
        const int nitem = p.groups * p.rows * p.cols, c0 = pass * p.groups * 8;
        constexpr int U = 4;
        for (int e0 = threadIdx.x; e0 < nitem; e0 += U * 256) {
            uint32_t v[U][8];
            int at[U];
            bool in[U];
#pragma unroll
            for (int k = 0; k < U; ++k) {
                uint32_t r1, col, grp, row;
                p.div_cols.divmod((uint32_t)min(e0 + k * 256, nitem - 1), r1, col);
                p.div_rows.divmod(r1, grp, row);
                const int hi = h0 + (int)row, wi = (int)col - p.pw, ch = c0 + (int)grp * 8;
                in[k] = hi >= 0 && hi < p.ih && wi >= 0 && wi < p.iw;
                const T *src = xb + (size_t)min(max(hi, 0), p.ih - 1) * p.iw + min(max(wi, 0), p.iw - 1);
#pragma unroll
                for (int c = 0; c < 8; ++c) v[k][c] = src[(size_t)min(ch + c, p.ic - 1) * plane];
#pragma unroll
                for (int c = 0; c < 8; ++c) v[k][c] = ch + c < p.ic ? v[k][c] : 0u;
                at[k] = ((int)row * p.cols + (int)col) * p.pitch + (int)grp * 16;
            }
#pragma unroll
            for (int k = 0; k < U; ++k) {
                if (e0 + k * 256 >= nitem) break;
                const uint4 q = make_uint4(v[k][0] | v[k][1] << 16, v[k][2] | v[k][3] << 16, v[k][4] | v[k][5] << 16, v[k][6] | v[k][7] << 16);
                *(uint4 *)(xs + at[k]) = in[k] ? q : make_uint4(0u, 0u, 0u, 0u);
            }
        }
        __syncthreads();
        if (wp0 < p.npos) {  // (no barrier is skipped)
            const int *tl = tab + g;
            uint4 bq[kAhead][NT];  // fragments of steps s .. s + kAhead - 1
            uint4 an[TG];
#pragma unroll
            for (int k = 0; k < kAhead; ++k)
#pragma unroll
                for (int n = 0; n < NT; ++n) bq[k][n] = bank[n][min(k, p.steps - 1) * 64];
            int on = tl[0];
#pragma unroll
            for (int t = 0; t < TG; ++t) an[t] = *(const uint4 *)(abase[t] + on);
            on = tl[4];
            auto step = [&](int s, auto kc) __attribute__((always_inline)) {
                constexpr int k = decltype(kc)::value;
                uint4 ac[TG], bc[NT];
#pragma unroll
                for (int t = 0; t < TG; ++t) ac[t] = an[t];
#pragma unroll
                for (int n = 0; n < NT; ++n) bc[n] = bq[k][n];
                const int next = min(s + kAhead, p.steps - 1) * 64;
#pragma unroll
                for (int n = 0; n < NT; ++n) bq[k][n] = bank[n][next];
#pragma unroll
                for (int t = 0; t < TG; ++t) an[t] = *(const uint4 *)(abase[t] + on);
                on = tl[min(s + 2, p.steps) * 4];
                if (s == p.steps - 1 && 4 * s + g >= p.units) {  // units that do not exist: zero times zero, whatever is staged
#pragma unroll
                    for (int t = 0; t < TG; ++t) ac[t] = make_uint4(0u, 0u, 0u, 0u);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int t = 0; t < TG; ++t)
#pragma unroll
                    for (int n = 0; n < NT; ++n)
                        acc[t][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, ac[t]), __builtin_bit_cast(bf16x8_t, bc[n]),
                                                                           acc[t][n], 0, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
            };
            int s = 0;
            for (; s + kAhead <= p.steps; s += kAhead) {
                step(s, std::integral_constant<int, 0>{});
                step(s + 1, std::integral_constant<int, 1>{});
                step(s + 2, std::integral_constant<int, 2>{});
            }
            if (s < p.steps) step(s, std::integral_constant<int, 0>{});
            if (s + 1 < p.steps) step(s + 1, std::integral_constant<int, 1>{});
        }
#pragma unroll
        for (int n = 0; n < NT; ++n) bank[n] += p.steps * 64;
    }

    // lane (g, i) holds positions 4g .. 4g+3 of channel i of every tile: with the pool, one window
    const int nout = POOL ? p.npos >> 2 : p.npos;
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int ch = ((int)blockIdx.y * NT + n) * 16 + i;
        if (ch >= p.oc) continue;
        const T bv = p.has_bias ? bias[ch] : (T)0;
        T *yc = y + ((size_t)b * p.oc + ch) * nout;
#pragma unroll
        for (int t = 0; t < TG; ++t) {
            const int pos = wp0 + t * 16 + 4 * g;
            Any4 o;
#pragma unroll
            for (int r = 0; r < 4; ++r) o[r] = round_bias_relu<T>(acc[t][n][r], p.has_bias != 0, bv, p.act);
            if constexpr (POOL) {
                T m = o[0];
                float mf = Elem<T>::to_f32(m);
#pragma unroll
                for (int r = 1; r < 4; ++r) {
                    const T q = o[r];
                    const float f = Elem<T>::to_f32(q);
                    if (f > mf) { m = q; mf = f; }
                }
                if (pos < p.npos) yc[pos >> 2] = m;
            } else if (pos + 3 < p.npos) {
                *(Any4 *)(yc + pos) = o;
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (pos + r < p.npos) yc[pos + r] = o[r];
            }
        }
    }
}

constexpr int64_t kTaps16Lds = 64 * 1024;       // two workgroups per CU and room for the pool's rows
constexpr int64_t kTaps16PoolLds = 80 * 1024;

}  // namespace

namespace agh {

template <int TG, int NT, bool POOL>
static int taps16_launch(const char *name, const void *x, const void *wp, const void *bias, void *y, dim3 grid, size_t smem, const Taps16Params &q) {
    if (smem > 64 * 1024)
        AGH_HIP(hipFuncSetAttribute((const void *)(conv2_taps16_kernel<TG, NT, POOL>), hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
    hipLaunchKernelGGL((conv2_taps16_kernel<TG, NT, POOL>), grid, dim3(256), smem, stream(), (const uint16_t *)x, (const uint4 *)wp,
                       (const uint16_t *)bias, (uint16_t *)y, q);
    AGH_LAUNCH_CHECK(name);
    return AGH_OK;
}

int conv2_taps16_try(const char *name, const void *x, const void *w, const void *bias, void *y, int64_t bs, int64_t ic, int64_t ih,
                     int64_t iw, int64_t oc, int64_t fh, int64_t fw, int64_t ph, int64_t pw, int64_t sh, int64_t sw, int64_t dh,
                     int64_t dw, int64_t oh, int64_t ow, int act, bool pool, bool forced, double limit_us, double wary_limit_us, size_t &lacking) {
    const int64_t npos = oh * ow, taps = fh * fw, cols = (ow - 1) * sw + (fw - 1) * dw + 1, all_groups = (ic + 7) / 8;
    if (npos > ((int64_t)1 << 24) || ic * taps > ((int64_t)1 << 24) || oc * ic * taps > ((int64_t)1 << 28) || cols > (1 << 16)) return 1;
    const int64_t cus = compute_units() > 0 ? compute_units() : 256, n16 = (oc + 15) / 16;
    const char *env = forced ? setting("AGH_CONV_TAPS_TILE") : nullptr;  // 10 TG + NT (tests)
    const int tile = env && *env ? atoi(env) : 0;
    int tg = 0, nt = 0;
    int64_t rows = 0, groups = 0;
    double us = 0;
    for (int t : {4, 2, 1}) {
        const int64_t span = std::min(oh - 1, (64 * t - 1 + ow - 1) / ow), r = span * sh + (fh - 1) * dh + 1;
        // as many channels as fit: all of them, or passes of equal size
        int64_t gr = all_groups;
        auto bytes = [&](int64_t n) { return r * cols * (n * 16 + 16) + ((taps * n + 3) / 4 + 1) * 16; };
        for (int64_t passes = 2; gr > 1 && bytes(gr) > kTaps16Lds; ++passes) gr = (all_groups + passes - 1) / passes;
        if (bytes(gr) > kTaps16Lds) continue;
        const int64_t passes = (all_groups + gr - 1) / gr, steps = (taps * gr + 3) / 4;
        const int64_t batches = (gr * r * cols + 1023) / 1024;  // of four staging items a thread
        for (int n : {4, 3, 2, 1}) {
            if (tile ? tile != 10 * t + n : n > n16) continue;
            // cycles of a workgroup: its passes of staging batches and steps (a step waits for its operands at least), its store; rounds
            // behind the first overlap with it for the most part.  Fitted to 250 shapes (mean error 8 % of a call that is not bound by
            // the host).
            const int64_t blocks = bs * ((npos + 64 * t - 1) / (64 * t)) * ((n16 + n - 1) / n), rounds = (blocks + cus - 1) / cus;
            const double wg = (double)passes * (460.0 + 1630.0 * (double)batches + std::max(84.0 * t * n, 360.0) * (double)steps) + 1735.0;
            const double cost = 5.3 + (1.0 + 0.27 * (double)(rounds - 1)) * wg / 2100.0 + 0.7e-6 * (double)bs * ((double)ic * ih * iw + (double)oc * npos);
            if (!tg || cost < us) { us = cost; tg = t; nt = n; rows = r; groups = gr; }
        }
    }
    if (!tg) return 1;
    const int64_t passes = (all_groups + groups - 1) / groups, units = taps * groups, steps = (units + 3) / 4;
    // Channels in passes or more than 36 steps: the bank streams from the L2s.  The estimate is up to half too low where a workgroup takes 64 channels
    // or passes are many, and says little where there are few workgroups.
    const bool streams = passes > 1 || steps > 36, few = bs * ((npos + 64 * tg - 1) / (64 * tg)) * ((n16 + nt - 1) / nt) * 4 < cus;
    if (!forced && us > (streams && (nt == 4 || passes > 4 || few) ? wary_limit_us : limit_us)) return 1;
    const int64_t pitch = groups * 16 + 16, tab_bytes = (steps + 1) * 16;
    auto lds_bytes = [&](int64_t r) { return r * cols * pitch + tab_bytes; };
    // rows of a tile of 16 t windows
    auto pool_rows = [&](int64_t t) { return (2 * std::min(oh / 2 - 1, (16 * t - 1 + ow / 2 - 1) / (ow / 2)) + 1) * sh + (fh - 1) * dh + 1; };
    // A stride of four rows and more can make the windows' rows several times the plain positions': where even the smallest tile of them does not fit,
    // neither call is taken here, since the fused one returns the bits of the plain one (one in a hundred shapes of strides 1 to 8 that would be).
    if (oh >= 2 && ow >= 2 && lds_bytes(pool_rows(1)) > 160 * 1024) return 1;
    const int64_t yh = pool ? oh / 2 : oh, yw = pool ? ow / 2 : ow, nall = pool ? yh * yw * 4 : npos;
    if (pool)  // the tile's positions are fewer where its rows take too much of the LDS
        for (rows = pool_rows(tg); tg > 1 && lds_bytes(rows) > kTaps16PoolLds; rows = pool_rows(tg)) tg /= 2;
    const int64_t ptiles = (nall + 64 * tg - 1) / (64 * tg), gx = bs * ptiles, gy = (n16 + nt - 1) / nt;
    const int64_t frags = n16 * passes * steps * 64;
    if (gx > 0x7FFFFFFF || gy > 65535 || frags > 0x7FFFFFFF) return 1;
    void *wp = nullptr;
    // Inside a capture the scratch memory cannot grow.  The kernels that need none are left then: what they took without this one they take, the
    // rest is refused.
    if (!workspace_ready((size_t)frags * 16)) {
        lacking = (size_t)frags * 16;
        return 1;
    }
    if (int rc = workspace((size_t)frags * 16, &wp)) return rc;
    hipLaunchKernelGGL(taps16_pack_kernel, dim3((unsigned)((frags + 255) / 256)), dim3(256), 0, stream(), (const uint16_t *)w, (uint4 *)wp, (int)oc,
                       (int)ic, (int)taps, (int)groups, (int)units, (int)steps, (int)passes, (uint32_t)frags);
    AGH_LAUNCH_CHECK(name);
    Taps16Params q;
    q.ic = (int)ic; q.ih = (int)ih; q.iw = (int)iw; q.oc = (int)oc; q.ph = (int)ph; q.pw = (int)pw;
    q.sh = (int)sh; q.sw = (int)sw; q.dh = (int)dh; q.dw = (int)dw; q.act = act; q.has_bias = bias != nullptr;
    q.npos = (int)nall; q.groups = (int)groups; q.passes = (int)passes; q.steps = (int)steps; q.units = (int)units;
    q.rows = (int)rows; q.cols = (int)cols; q.pitch = (int)pitch; q.tab_bytes = (int)tab_bytes;
    q.div_ptiles = FastDiv((uint32_t)ptiles); q.div_cols = FastDiv((uint32_t)cols); q.div_rows = FastDiv((uint32_t)rows);
    q.div_yw = FastDiv((uint32_t)yw); q.div_groups = FastDiv((uint32_t)groups); q.div_fw = FastDiv((uint32_t)fw);
    const dim3 grid((unsigned)gx, (unsigned)gy);
    const size_t smem = (size_t)lds_bytes(rows);
#define AGH_TAPS16(TGV, NTV) \
    case TGV * 8 + NTV: \
        return pool ? taps16_launch<TGV, NTV, true>(name, x, wp, bias, y, grid, smem, q) \
                    : taps16_launch<TGV, NTV, false>(name, x, wp, bias, y, grid, smem, q)
#define AGH_TAPS16_4(TGV) AGH_TAPS16(TGV, 1); AGH_TAPS16(TGV, 2); AGH_TAPS16(TGV, 3); AGH_TAPS16(TGV, 4)
    switch (tg * 8 + nt) { AGH_TAPS16_4(4); AGH_TAPS16_4(2); AGH_TAPS16_4(1); }
#undef AGH_TAPS16_4
#undef AGH_TAPS16
    return 1;
}

}  // namespace agh
