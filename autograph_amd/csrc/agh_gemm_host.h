// Host side of the GEMM entry points: argument checks (the reference's bail!s at
// src/tensor/linalg.rs:256-279), orientation / loader / tile selection, split-K planning
// (the job of linalg.rs:306-340) and the launches.  Included once per element type.
#pragma once
#include <stdlib.h>
#include <string.h>

#include <type_traits>

#include "agh_gemm_kernel.h"

namespace agh {
namespace gemm {

struct TileCfg {
    int bp, bq;
    float eff;       // relative MFMA efficiency of the tile shape (bigger tiles reuse operands more)
    int wgs_per_cu;  // workgroups a CU can hold (LDS / register bound)
    bool scalar_ok;  // has instantiations with the element-wise loader
};

// index = config id used by launch_cfg below
static const TileCfg kCfgs[] = {
    {256, 256, 1.00f, 1, false},
    {128, 256, 0.85f, 1, false},
    {256, 128, 0.85f, 1, false},
    {128, 128, 0.70f, 2, false},
    {64, 64, 0.35f, 4, true},
    {32, 128, 0.28f, 4, true},
    {128, 32, 0.28f, 4, true},
};
static constexpr int kNumCfgs = sizeof(kCfgs) / sizeof(kCfgs[0]);
// rate of a CU on 64 x 64 direct-to-LDS bf16 tiles relative to a 256 x 256 workgroup on a full chip: one workgroup with
// the CU to itself (ring of eight stages), two sharing it (rings of four)
static constexpr double kDirect64Alone = 0.27, kDirect64Shared = 0.19;

template <typename T, int BP, int BQ, int WGP, int WGQ, int LP, int LQ>
int launch_one(const Args &g, int splits) {
    auto kern = gemm_kernel<T, BP, BQ, WGP, WGQ, LP, LQ>;
    constexpr size_t smem = 2 * (size_t)(BP + BQ) * 128;
    static bool attr_done = false;
    if (!attr_done) {
        if (smem > 48 * 1024)
            AGH_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        attr_done = true;
    }
    dim3 grid((unsigned)(g.tiles_p * g.tiles_q), (unsigned)splits, (unsigned)g.batch);
    hipLaunchKernelGGL(kern, grid, dim3(WGP * WGQ * 64), smem, stream(), g);
    AGH_LAUNCH_CHECK("gemm kernel launch");
    return AGH_OK;
}

#ifdef AGH_GEMM_WITH_BF16_DIRECT
// direct-to-LDS bf16 kernels: defined and explicitly instantiated in agh_gemm_bf16_dl_<tile>.hip
// (one translation unit per tile shape, so they compile in parallel)
template <int BP, int BQ, int WGP, int WGQ, int LP, int LQ, int NS>
int launch_one_dl(const Args &g, int splits);
// the form of the same kernel for operands at any element address, k and row counts of any size
// (agh_gemm_bf16_any_<tile>.hip)
template <int BP, int BQ, int WGP, int WGQ, int LP, int LQ>
int launch_one_any(const Args &g, int splits);
#endif

inline int env_int(const char *name, int dflt);

#ifdef AGH_GEMM_WITH_BF16_DIRECT
// Two LDS stages, but a ring of four for a grid of 128 x 128 tiles that gives a CU one workgroup at most and has 20
// k-tiles or more: alone on its CU such a workgroup waits for loads most of the time (2048^3: 22.8 us with two stages,
// 17.9 us with four; at 16 k-tiles the four tiles requested up front cost 0.3 us more than they save).
// AGH_GEMM_RING=2|4 forces either.
template <int BP, int BQ, int WGP, int WGQ, int LP, int LQ>
int launch_dl_ring(const Args &g, int splits) {
    if constexpr (BP == 64 && BQ == 64) {
        // A k-tile of the 64 x 64 tile is eight MFMAs a wave, a small fraction of a load's latency: always a ring of
        // four stages (64 KB, two workgroups per CU).  Eight stages measured slower at every size (1024^3: 6.2 against
        // 5.6 us, 2048^3: 32.2 against 29.3 us).
        return launch_one_dl<BP, BQ, WGP, WGQ, LP, LQ, 4>(g, splits);
    } else {
        if constexpr (BP == 128 && BQ == 128) {
            const int64_t wgs = (int64_t)g.tiles_p * g.tiles_q * splits * g.batch;
            // split-K streams its operands from HBM once (no second workgroup re-reads them out of L2), where the deeper
            // ring pays from 8 k-tiles on (128x4096x4096 in 8 splits: 19.5 against 20.5 us; in 4: 17.2 against 20.1)
            const bool alone = wgs <= (compute_units() > 0 ? compute_units() : 256) &&
                               (g.k_per_split >= 20 * 64 || (splits > 1 && g.k_per_split >= 8 * 64));
            if (env_int("AGH_GEMM_RING", alone ? 4 : 2) == 4)
                return launch_one_dl<BP, BQ, WGP, WGQ, LP, LQ, 4>(g, splits);
        }
        // 128 x 256 and 256 x 128: three stages of 48 KB (a CU holds one such workgroup either way; 3 to 10 % faster than
        // two at every size measured, 2048^3 to 8192^3)
        return launch_one_dl<BP, BQ, WGP, WGQ, LP, LQ, BP * BQ == 128 * 256 ? 3 : 2>(g, splits);
    }
}
#endif

#ifdef AGH_GEMM_WITH_F32_DIRECT
// its form for operands at any element address (agh_gemm_f32_any.hip)
template <int TP, int TQ, int NS, int LP, int LQ>
int launch_one_f32_any(const Args &g, int splits);
// direct-to-LDS f32 kernel for 64 x 64 tiles (agh_gemm_f32_dl.h)
template <int TP, int TQ, int NS, int LP, int LQ, int KS = 1>
int launch_f32_dl(const Args &g, int splits) {
    if constexpr (KS == 1 && TP * TQ <= 4) {
        // a grid that gives a CU one workgroup at most, or a product that would on larger tiles: eight waves, every k-tile
        // split between two (AGH_GEMM_KSPLIT=0|1 forbids / forces it)
        const int64_t wgs = (int64_t)g.tiles_p * g.tiles_q * splits * g.batch;
        const int ks = env_int("AGH_GEMM_KSPLIT", g.two_sums || wgs <= (compute_units() > 0 ? compute_units() : 256) ? 1 : 0);
        if (ks) return launch_f32_dl<TP, TQ, NS, LP, LQ, 2>(g, splits);
    }
    auto kern = gemm_f32_dl_kernel<TP, TQ, NS, LP, LQ, KS>;
    constexpr size_t smem = F32DlGeo<TP, TQ, NS, LP, LQ>::SMEM_BYTES;
    static bool attr_done = false;
    if (!attr_done) {
        if (smem > 48 * 1024)
            AGH_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        attr_done = true;
    }
    dim3 grid((unsigned)(g.tiles_p * g.tiles_q), (unsigned)splits, (unsigned)g.batch);
    hipLaunchKernelGGL(kern, grid, dim3(256 * KS), smem, stream(), g);
    AGH_LAUNCH_CHECK("gemm kernel launch");
    return AGH_OK;
}
#endif

#ifdef AGH_GEMM_WITH_F32_DIRECT
// two workgroups per CU over all tiles (agh_gemm_f32_stream.h)
template <int LP, int LQ, int KS = 1>
int launch_f32_stream(const Args &g, int cus, bool halves) {
    if constexpr (KS == 1)
        if (halves) return launch_f32_stream<LP, LQ, 2>(g, cus, true);
    auto kern = gemm_f32_stream_kernel<LP, LQ, KS>;
    constexpr size_t smem = F32StreamGeo<LP, LQ>::SMEM_BYTES;
    static bool attr_done = false;
    if (!attr_done) {
        AGH_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        attr_done = true;
    }
    hipLaunchKernelGGL(kern, dim3((unsigned)((cus + 7) / 8 * 8 * kStreamPerCu)), dim3(512), smem, stream(), g);
    AGH_LAUNCH_CHECK("gemm (f32 stream) kernel launch");
    return AGH_OK;
}
#endif

template <typename T, int BP, int BQ, int WGP, int WGQ, bool SCALAR_OK>
int launch_loaders(const Args &g, int splits, int lp, int lq, bool direct, bool any) {
#ifdef AGH_GEMM_WITH_F32_DIRECT
    if constexpr (std::is_same<T, float>::value && BP % 64 == 0 && BQ % 64 == 0) {
        // both operands vector-loadable (any k: a last k-tile shorter than 32 is loaded with zeros behind k = K)
        // (AGH_GEMM_DIRECT=0 forces the register-staged kernel).  64 x 64: a ring of four stages, one or two
        // workgroups per CU; 128 x 128: two stages (a k-tile is four times as long), two workgroups per CU; the
        // larger tiles: two stages, one workgroup per CU.
        constexpr int TPW = BP / 64, TQW = BQ / 64, NS = BP == 64 ? 4 : 2;
        if constexpr (BP == BQ && BP <= 128) {
            if (any) {
                switch (lp * 3 + lq) {
                    case LD_K * 3 + LD_K: return launch_one_f32_any<TPW, TQW, NS, LD_K, LD_K>(g, splits);
                    case LD_K * 3 + LD_R: return launch_one_f32_any<TPW, TQW, NS, LD_K, LD_R>(g, splits);
                    case LD_R * 3 + LD_K: return launch_one_f32_any<TPW, TQW, NS, LD_R, LD_K>(g, splits);
                    case LD_R * 3 + LD_R: return launch_one_f32_any<TPW, TQW, NS, LD_R, LD_R>(g, splits);
                    default: break;
                }
            }
        }
        if (lp != LD_S && lq != LD_S && g.K > 0 && env_int("AGH_GEMM_DIRECT", 1) != 0) {
            switch (lp * 3 + lq) {
                case LD_K * 3 + LD_K: return launch_f32_dl<TPW, TQW, NS, LD_K, LD_K>(g, splits);
                case LD_K * 3 + LD_R: return launch_f32_dl<TPW, TQW, NS, LD_K, LD_R>(g, splits);
                case LD_R * 3 + LD_K: return launch_f32_dl<TPW, TQW, NS, LD_R, LD_K>(g, splits);
                case LD_R * 3 + LD_R: return launch_f32_dl<TPW, TQW, NS, LD_R, LD_R>(g, splits);
                default: break;
            }
        }
    }
#endif
#ifdef AGH_GEMM_WITH_BF16_DIRECT
    if constexpr (std::is_same<T, uint16_t>::value && BP == BQ && BP <= 128) {
        if (any) {
            switch (lp * 3 + lq) {
                case LD_K * 3 + LD_K: return launch_one_any<BP, BQ, WGP, WGQ, LD_K, LD_K>(g, splits);
                case LD_K * 3 + LD_R: return launch_one_any<BP, BQ, WGP, WGQ, LD_K, LD_R>(g, splits);
                case LD_R * 3 + LD_K: return launch_one_any<BP, BQ, WGP, WGQ, LD_R, LD_K>(g, splits);
                case LD_R * 3 + LD_R: return launch_one_any<BP, BQ, WGP, WGQ, LD_R, LD_R>(g, splits);
                default: break;
            }
        }
    }
    if constexpr (std::is_same<T, uint16_t>::value && (!SCALAR_OK || (BP == 64 && BQ == 64))) {
        if (direct && lp != LD_S && lq != LD_S) {
            switch (lp * 3 + lq) {
                case LD_K * 3 + LD_K: return launch_dl_ring<BP, BQ, WGP, WGQ, LD_K, LD_K>(g, splits);
                case LD_K * 3 + LD_R: return launch_dl_ring<BP, BQ, WGP, WGQ, LD_K, LD_R>(g, splits);
                case LD_R * 3 + LD_K: return launch_dl_ring<BP, BQ, WGP, WGQ, LD_R, LD_K>(g, splits);
                case LD_R * 3 + LD_R: return launch_dl_ring<BP, BQ, WGP, WGQ, LD_R, LD_R>(g, splits);
                default: break;
            }
        }
    }
#endif
    switch (lp * 3 + lq) {
        case LD_K * 3 + LD_K: return launch_one<T, BP, BQ, WGP, WGQ, LD_K, LD_K>(g, splits);
        case LD_K * 3 + LD_R: return launch_one<T, BP, BQ, WGP, WGQ, LD_K, LD_R>(g, splits);
        case LD_R * 3 + LD_K: return launch_one<T, BP, BQ, WGP, WGQ, LD_R, LD_K>(g, splits);
        case LD_R * 3 + LD_R: return launch_one<T, BP, BQ, WGP, WGQ, LD_R, LD_R>(g, splits);
        default: break;
    }
    if constexpr (SCALAR_OK) {
        switch (lp * 3 + lq) {
            case LD_K * 3 + LD_S: return launch_one<T, BP, BQ, WGP, WGQ, LD_K, LD_S>(g, splits);
            case LD_R * 3 + LD_S: return launch_one<T, BP, BQ, WGP, WGQ, LD_R, LD_S>(g, splits);
            case LD_S * 3 + LD_K: return launch_one<T, BP, BQ, WGP, WGQ, LD_S, LD_K>(g, splits);
            case LD_S * 3 + LD_R: return launch_one<T, BP, BQ, WGP, WGQ, LD_S, LD_R>(g, splits);
            case LD_S * 3 + LD_S: return launch_one<T, BP, BQ, WGP, WGQ, LD_S, LD_S>(g, splits);
            default: break;
        }
    }
    return fail(AGH_EINVAL, "gemm: no kernel for loader pair (%d,%d)", lp, lq);
}

template <typename T>
int launch_cfg(int cfg, const Args &g, int splits, int lp, int lq, bool direct, bool any) {
    switch (cfg) {
        case 0: return launch_loaders<T, 256, 256, 2, 2, false>(g, splits, lp, lq, direct, any);
        case 1: return launch_loaders<T, 128, 256, 2, 2, false>(g, splits, lp, lq, direct, any);
        case 2: return launch_loaders<T, 256, 128, 2, 2, false>(g, splits, lp, lq, direct, any);
        case 3: return launch_loaders<T, 128, 128, 2, 2, false>(g, splits, lp, lq, direct, any);
        case 4: return launch_loaders<T, 64, 64, 2, 2, true>(g, splits, lp, lq, direct, any);
        case 5: return launch_loaders<T, 32, 128, 1, 4, true>(g, splits, lp, lq, false, any);
        case 6: return launch_loaders<T, 128, 32, 4, 1, true>(g, splits, lp, lq, false, any);
        default: return fail(AGH_EINVAL, "gemm: bad tile config %d", cfg);
    }
}

inline bool aligned(const void *p, size_t a) { return ((uintptr_t)p % a) == 0; }

// Which loader can serve an operand seen as NR rows x K with element strides (rs, ks).
template <typename T>
int pick_loader(const void *base, int64_t rs, int64_t ks, int NR, int K) {
    constexpr int EPC = Geo<T>::EPC;
    if (!aligned(base, 16)) return LD_S;
    if (ks == 1 && K % EPC == 0 && (rs % EPC == 0 || NR == 1)) return LD_K;
    if (rs == 1 && NR % EPC == 0 && (ks % EPC == 0 || K == 1)) return LD_R;
    return LD_S;
}

// The same for the bf16 kernel that reads 16 bytes from any element address: no multiple of anything is needed, but
// k >= 8 (a last chunk is read from up to 7 elements further down its row), and for rows as the unit-stride axis k-rows
// that follow each other upwards at least 8 elements apart (a chunk that runs past the last row of a k-row stays inside the
// operand's memory).  The f32 kernel's form loads elements: a unit stride is enough.
template <typename T>
int pick_loader_any(int64_t rs, int64_t ks, int K) {
    if (sizeof(T) == 4) return ks == 1 ? LD_K : rs == 1 ? LD_R : LD_S;
    if (K < 8) return LD_S;
    if (ks == 1) return LD_K;
    if (rs == 1 && ks >= 8) return LD_R;
    return LD_S;
}

// Products that the any-address kernel's two tiles serve worse than the element-wise loaders' 32 x 128 and 128 x 32: one or two
// k-tiles, so that a workgroup is all filling and storing, few rows or columns, so that half as many workgroups cover C, and
// more of them than CUs.  Few columns (P, C's unit-stride axis) are the worse for it: C's rows are stored element by element.
// Element-wise / 64 x 64 in us over the forms of 270 such products: 30 of 29767x11x4 31.7 / 100, 1x115707x13x2 7.3 / 13.5,
// 44 of 81771x8x2 115 / 239; 51 of 12x9x164388 405 / 574; two k-tiles: 4 of 89307x81x1 26 / 40, but 6 of 111328x121x10 63 / 55.
// On the other side of the line: 26 of 34426x103x15 101 / 92, 1x13x117x40505 9.9 / 7.7, up to 256 tiles 1.2 times the time.
inline bool short_and_narrow(const Args &g, int64_t batch, int64_t cus, int lp) {
    if (g.K > 128 || (g.NP > 32 && g.NQ > 16)) return false;
    const int64_t tiles = (int64_t)((g.NP + 63) / 64) * ((g.NQ + 63) / 64) * batch;
    const bool one = g.K <= 64, many = tiles > 4 * cus;
    if (tiles <= cus) return false;
    if (g.NP <= 16 ? one || many : g.NP <= 32 && one && many) return true;
    return g.NQ <= 16 && one && many && (lp == LD_K || tiles > 20 * cus);
}

// Products at any address that the f32 kernel's form for them serves better than the element-wise loaders.
// Up to k = 64 it does not: two k-tiles are all filling, and those loaders read only what there is (3889x18x648 7.9 / 10.7 us,
// 37905x32x448 28.6 / 37.9, 3460x57x1352 15.2 / 18.5; 584x107x2002 16.4 / 13.3, 5088x95x642 21.8 / 20.2).
// Nor, with more 64 x 64 tiles than CUs,
//   where tiles of 32 x 128 or 128 x 32, which only those loaders have, need 0.8 of the rounds or fewer: over 270 such products as fast all together,
//   0.5 to 1.4 of the time one by one, and 65 to 96 rows or columns against any number on the whole slower (70x80x39588, left transposed, 15.7 /
//   21.7; 146x672x6485, both, 25.3 / 35.8; 3704x1694x525, both, 99.7 / 117);
//   up to k = 128 where one operand's unit stride is along k and the other's along its rows, which those loaders, four workgroups a CU, are good at
//   (6697x70x1384, both transposed, 33.4 / 38.2; 2339x93x1744 19.3 / 21.0);
//   up to k = 512 where moreover the operand along k is of whole vectors: one in three of 189 products slower (7649x80x788 21.9 / 28.6; 391x68x7423,
//   neither transposed, 18.2 / 22.8; 2870x280x5883 130 / 139) and as fast all together; beyond it 82 products of 0.75 to 0.98 of the time.
inline bool f32_any_pays(const Args &g, int64_t batch, int64_t cus, int lp, int lq, int lp_any, int lq_any) {
    if (g.K <= 64) return false;
    auto rounds = [&](int bp, int bq) { return ((int64_t)((g.NP + bp - 1) / bp) * ((g.NQ + bq - 1) / bq) * batch + cus - 1) / cus; };
    if (rounds(64, 64) <= 1) return true;
    if (std::min(rounds(32, 128), rounds(128, 32)) * 5 <= rounds(64, 64) * 4) return false;
    if (lp_any == lq_any) return true;
    const bool whole_along_k = (lp_any == LD_K ? lp : lq) != LD_S;  // (the other operand has none then, or this is not asked)
    return g.K > (whole_along_k ? 512 : 128);
}

// Optional override for experiments: AGH_GEMM_CFG=<config id>, AGH_GEMM_SPLITS=<n>.
inline int env_int(const char *name, int dflt) {
    const char *s = setting(name);
    return (s && *s) ? atoi(s) : dflt;
}

// k-tiles a split and splits of a product: one split where the tile grid fills half the chip or k is short
inline int plan_splits(int64_t tiles, int ktiles, int64_t cus, int kmin) {
    if (tiles * 2 > cus || ktiles < 32) return 1;
    return (int)std::max<int64_t>(1, std::min(std::min(cus / tiles, (int64_t)(ktiles / kmin)), (int64_t)256));
}

// What split k costs and saves in bf16, in us, where every workgroup has a CU to itself: k-tiles a split, the second launch and the f32 partial sums
// by the MB of C (as bf16).  Fitted to 420 products on tiles of 128 x 128, of whole vectors and at any address.
struct Bf16SplitTime { double ktile, second, part_mb; };
static const Bf16SplitTime kBf16Split = {0.44, 3.6, 1.0}, kBf16SplitAny = {0.95, 2.3, 0.88};
inline double bf16_split_us(const Bf16SplitTime &t, int splits, int ktiles, double mb) {
    return t.ktile * ((ktiles + splits - 1) / splits) + (splits > 1 ? t.second + t.part_mb * splits * mb : 0.0);
}
// Whether a product of whole vectors that would have two splits takes one: the estimate has to be well below, since a k-tile is 0.44 to 0.75 us by
// sizes and strides.  One split / two: where the second launch adds single elements (rows of C no multiple of four), below 0.86 of the
// estimate 0.68 to 0.98 of the time over 80 products (728x2016x2215, B transposed, 18.0 / 24.6; 2160x2472x827 at 0.88 29.8 / 29.4); where it
// adds vectors, below 0.77 0.74 to 1.02 over 25 (2000x2048x1008 16.2 / 20.7), from there to 0.8 up to 1.09 and beyond up to 1.26
// (1656x2616x792 27.9 / 22.2, 440x2952x3784 28.4 / 23.7).  Three and more splits are never that far above.
inline bool bf16_one_split(int ktiles, double mb, bool by_vectors) {
    return bf16_split_us(kBf16Split, 1, ktiles, mb) < (by_vectors ? 0.77 : 0.86) * bf16_split_us(kBf16Split, 2, ktiles, mb);
}

// Time in us of an f32 product on the direct-to-LDS kernels' 64 x 64 or 128 x 128 tiles, fitted to 450 products of 16 to 60000 x 16 to
// 8192 x 16 to 8192 outside the small kernel's range (mean error 4 % with whole vectors, 6 % at any address): a launch, rounds of
// workgroups of so many k-tiles and a store each, the bytes of C, and for split k the second launch and its partial sums.
struct F32TileTime { double launch, ktile, store, c_mb, reduce, part_mb; };
inline double f32_tile_us(int edge, bool any, int64_t np, int64_t nq, int64_t k, int64_t batch, int64_t cus, int *splits) {
    static const F32TileTime kTimes[2][2] = {{{3.54, 0.54, 0.33, 0.27, 2.81, 0.31}, {7.12, 1.96, 0.42, 0.17, 0.22, 0.56}},
                                             {{3.28, 0.68, 1.67, 0.06, 3.16, 0.25}, {4.50, 2.30, 4.35, 0.12, 0.00, 0.41}}};
    const F32TileTime &t = kTimes[any][edge == 128];
    const int64_t tiles = ((np + edge - 1) / edge) * ((nq + edge - 1) / edge) * batch;
    const int ktiles = (int)((k + 31) / 32);
    int s = batch == 1 ? plan_splits(tiles, ktiles, cus, 4) : 1;
    const int per_split = (ktiles + s - 1) / s;
    s = (ktiles + per_split - 1) / per_split;
    *splits = s;
    const double rounds = (double)((tiles * s + cus - 1) / cus), mb = (double)np * nq * batch * 4e-6;
    return t.launch + rounds * (t.ktile * per_split + t.store) + (s > 1 ? t.reduce + t.part_mb * s * mb : t.c_mb * mb);
}

template <typename T>
int gemm_entry(const char *name, int64_t m, int64_t k, int64_t n, float alpha, const void *a, int64_t off_a,
               int64_t rsa, int64_t csa, const void *b, int64_t off_b, int64_t rsb, int64_t csb, float beta, void *c,
               int64_t off_c, int64_t rsc, int64_t csc, const void *bias, int64_t off_bias, int64_t bias_stride,
               int act, int64_t batch = 1, int64_t batch_a = 0, int64_t batch_b = 0, int64_t batch_c = 0,
               bool fixed_scratch = false) {
    AGH_API_ENTER();
    if (m < 0 || k < 0 || n < 0 || batch < 0) return fail(AGH_EINVAL, "%s: negative dimension", name);
    if (batch > 65535) return fail(AGH_ERANGE, "%s: batch count above 65535", name);
    if (batch == 0) return AGH_OK;
    const int64_t lim = ((int64_t)1 << 31) - 512;
    if (m > lim || k > lim || n > lim) return fail(AGH_ERANGE, "%s: dimension does not fit 31 bits", name);
    if (act != AGH_ACT_NONE && act != AGH_ACT_RELU) return fail(AGH_EINVAL, "%s: unknown activation %d", name, act);
    if (m == 0 || n == 0) return AGH_OK;
    if (!c) return fail(AGH_ENULL, "%s: null c", name);
    if (k > 0 && (!a || !b)) return fail(AGH_ENULL, "%s: null a or b", name);
    if (m > 1 && rsc == 0) return fail(AGH_EINVAL, "%s: c row stride is 0", name);
    if (n > 1 && csc == 0) return fail(AGH_EINVAL, "%s: c column stride is 0", name);
    constexpr int EPC = Geo<T>::EPC;
    constexpr int BK = 8 * EPC;

    const T *A = (const T *)a + off_a;
    const T *B = (const T *)b + off_b;
    T *C = (T *)c + off_c;

    Args g;
    memset(&g, 0, sizeof(g));
    // p runs along C's unit-stride axis when it has one (rows of C otherwise: p = n axis)
    const bool p_is_n = !(rsc == 1 && csc != 1);
    if (p_is_n) {
        g.P = B; g.ps = csb; g.pk = rsb; g.NP = (int)n;
        g.Q = A; g.qs = rsa; g.qk = csa; g.NQ = (int)m;
        g.dp = csc; g.dq = rsc;
        g.bias_on_p = 1;
        g.batch_p = batch_b; g.batch_q = batch_a;
    } else {
        g.P = A; g.ps = rsa; g.pk = csa; g.NP = (int)m;
        g.Q = B; g.qs = csb; g.qk = rsb; g.NQ = (int)n;
        g.dp = rsc; g.dq = csc;
        g.bias_on_p = 0;
        g.batch_p = batch_a; g.batch_q = batch_b;
    }
    g.D = C;
    g.batch = (int)batch;
    g.batch_d = batch_c;
    g.K = (int)k;
    g.alpha = alpha;
    g.beta = beta;
    g.has_bias = bias != nullptr;
    g.bias = bias ? (const void *)((const T *)bias + off_bias) : nullptr;
    g.bias_stride = bias_stride;
    g.act = act;
    g.NPpad = (g.NP + 3) & ~3;

    int lp = k > 0 ? pick_loader<T>(g.P, g.ps, g.pk, g.NP, g.K) : LD_S;
    int lq = k > 0 ? pick_loader<T>(g.Q, g.qs, g.qk, g.NQ, g.K) : LD_S;
    // every matrix of a batch must satisfy the same alignment as the first
    const bool batch_aligned = batch == 1 || (g.batch_p % EPC == 0 && g.batch_q % EPC == 0);
    if (!batch_aligned) lp = lq = LD_S;
    // operands that are no whole 16-byte vectors but have a unit-stride axis each take the direct-to-LDS kernels' forms
    // for any element address (tiles 128 x 128 and 64 x 64); what is left has the element-wise loader
    int lp_any = LD_S, lq_any = LD_S;
    if ((lp == LD_S || lq == LD_S) && k > 0 && env_int("AGH_GEMM_DIRECT", 1) != 0) {
        lp_any = pick_loader_any<T>(g.ps, g.pk, g.K);
        lq_any = pick_loader_any<T>(g.qs, g.qk, g.K);
    }
    const int cus = compute_units() > 0 ? compute_units() : 256;
    const int forced_cfg = env_int("AGH_GEMM_CFG", -1);
    const bool any_addr = lp_any != LD_S && lq_any != LD_S &&
                          (forced_cfg >= 0 || (sizeof(T) == 4 ? f32_any_pays(g, batch, cus, lp, lq, lp_any, lq_any) : !short_and_narrow(g, batch, cus, lp_any)));
    const bool skinny = g.NP <= 32 || g.NQ <= 32;  // where the 32 x 128 and 128 x 32 tiles pad less
    const bool any_scalar = (lp == LD_S || lq == LD_S);
    const bool vec_store = g.dp == 1 && g.NP % 4 == 0 && (g.dq % 4 == 0 || g.NQ == 1) && aligned(C, 4 * sizeof(T)) &&
                           (batch == 1 || g.batch_d % 4 == 0);

#ifdef AGH_GEMM_WITH_F32_SMALL
    if constexpr (sizeof(T) == 4) {
        const int rc = gemm_f32_small_try(g, lp, lq, vec_store, batch);
        if (rc != 1) return rc;
    }
#endif

    // ---- tile shape: minimise (rounds of workgroups) x (tile area) / efficiency ----
    // (any k: a last k-tile shorter than 64 is loaded with zeros behind k = K)
    const bool direct_ok = sizeof(T) == 2 && (!any_scalar || any_addr) && g.K > 0 && env_int("AGH_GEMM_DIRECT", 1) != 0;
    int best = -1;
    double best_cost = 0;
    for (int i = 0; i < kNumCfgs; ++i) {
        const TileCfg &t = kCfgs[i];
        // (any address: of a 128 x 128 tile over at most 64 rows or columns, half would be padding)
        if (any_addr && sizeof(T) == 2 ? i != 4 && (i != 3 || g.NP <= 64 || g.NQ <= 64) : any_scalar && !t.scalar_ok && !(any_addr && i == 3)) continue;
        if (any_addr && sizeof(T) == 4 && !skinny && i != 3 && i != 4) continue;
        const int64_t tiles = (int64_t)((g.NP + t.bp - 1) / t.bp) * ((g.NQ + t.bq - 1) / t.bq) * batch;
        if (tiles > 0x7FFFFFFF) continue;
        // a CU works through ceil(tiles / CUs) tiles; co-resident workgroups share its MFMA rate
        const int64_t rounds = (tiles + cus - 1) / cus;
        // where the direct-to-LDS bf16 kernel applies (the four large tiles), the register-staged small tiles
        // are a poor second: measured 2x slower at 1024^3 (16.4 us against 8.9 us) although they put four times as
        // many CUs to work
        double eff = (direct_ok && !kCfgs[i].scalar_ok) || !direct_ok ? t.eff : t.eff * 0.25;
        const bool bf16_direct64 = direct_ok && t.bp == 64 && t.bq == 64;
        // the 64 x 64 direct tile is measured at 0.8 of the 256 x 256 tile's rate per CU (3072^3: 118 TFLOP/s, where
        // 144 tiles of 256 x 256 leave 112 CUs idle)
        // f32: the 64 x 64 and 128 x 128 tiles have direct-to-LDS kernels (agh_gemm_f32_dl.h)
        const bool f32_dl_ok = sizeof(T) == 4 && (!any_scalar || any_addr) && g.K > 0 && env_int("AGH_GEMM_DIRECT", 1) != 0;
        const bool f32_direct = f32_dl_ok && t.bp == 64 && t.bq == 64;
        // (at any address, against the skinny element-wise tiles alone: 47921 x 2701 x 31 242 / 202 us, 25048 x 751 x 24 41 / 38)
        if (f32_direct) eff = any_addr ? 0.48 : 0.80;
        if (f32_dl_ok && t.bp == 128 && t.bq == 128) eff = 0.95;  // 4096^3: 135 TFLOP/s, the 256 x 256 tile's rate
        // a tile's prologue and epilogue cost about four k-tiles of time when the CU holds one workgroup, next
        // to nothing when a second workgroup multiplies meanwhile: decides short-k shapes (conv GEMM, k = 576).
        // The f32 direct kernel's k-tile is short (sixteen MFMAs a wave): filling its four-stage ring and storing
        // the tile cost about six of them (at k = 576 the 128 x 128 tile is 9 % faster, from k = 1536 on slower).
        const double kt = (double)((g.K + BK - 1) / BK);
        eff *= kt / (kt + (f32_direct ? 6.0 : t.wgs_per_cu == 1 ? 4.0 : 0.5));
        double cost = (double)rounds * t.bp * t.bq / eff;
        // many small tiles do not run in lockstep rounds: a CU takes the next tile when one of its two is done, and the
        // launch ends a fraction of a tile after tiles / CUs tile times (3584^3 on 64 x 64 tiles: 12.25 tiles a CU,
        // 12.5 tile times measured, 790 us against 871 us on the 256 x 256 tile)
        if (f32_direct && tiles >= 4 * (int64_t)cus) cost = ((double)tiles / cus + 0.25) * t.bp * t.bq / eff;
        // bf16 direct-to-LDS tiles: a full chip of them runs at the power limit, where the rate depends on the tile
        // shape (bigger tiles move fewer operand bytes per flop) and not on how many CUs take part, while a
        // launch that leaves CUs idle runs the busy ones at a higher clock.  Measured per k-tile of a 256 x 256
        // tile: 1.32 us with 256 workgroups (8192^3, 4096^3), 0.97 us with 144 (3072^3).  The cost is summed over
        // rounds of co-resident workgroups, each round at the lower of the two rates.
        if (direct_ok && !t.scalar_ok) {
            // rates relative to a 256 x 256 workgroup on a full chip.  kAlone: a 128 x 128 workgroup with a CU to itself
            // (2048^3: 22.8 us on two LDS stages, 17.9 us on the ring of four a launch of at most one workgroup per CU
            // and 20 k-tiles or more takes) against two sharing it
            static const double kUnthrottled[4] = {1.36, 1.0, 1.0, 0.946}, kAtPowerLimit[4] = {1.0, 0.855, 0.855, 0.85};
            const double kAlone[4] = {1.36, 1.0, 1.0, tiles <= cus && kt >= 20 ? 0.75 : 0.59};
            const int64_t slots = (int64_t)cus * t.wgs_per_cu, rest = tiles % slots;
            const double area = (double)t.bp * t.bq;
            // a round of n co-resident workgroups: each CU at its unthrottled rate or at its share of the chip's
            // power-limited rate, whichever is lower
            auto round_cost = [&](int64_t n) {
                const bool shared = n > cus;
                const double rate = std::min(shared ? kUnthrottled[i] : kAlone[i],
                                             kAtPowerLimit[i] * cus / (double)std::min<int64_t>(n, cus));
                return (shared ? t.wgs_per_cu : 1) * area / rate;
            };
            cost = ((double)(tiles / slots) * round_cost(slots) + (rest ? round_cost(rest) : 0.0)) *
                   (kt + (t.wgs_per_cu == 1 ? 4.0 : 2.0)) / kt;
        }
        // The 64 x 64 direct-to-LDS bf16 tile: a CU's fill path from L2 bounds it (16 KB per k-tile against the 32 KB a
        // 128 x 128 tile moves for four times the flop), so a tile takes about half the time of a 128 x 128 one; filling
        // its ring and storing the tile cost about six of its k-tiles.
        if (bf16_direct64) {
            const int64_t slots = (int64_t)cus * 2;
            const double per_tile = (double)t.bp * t.bq / (tiles <= cus ? kDirect64Alone : kDirect64Shared);
            cost = (double)((tiles + slots - 1) / slots) * (tiles <= cus ? 1 : 2) * per_tile * (kt + 6.0) / kt;
        }
        // Operands at any element address: bound by the L1s, whatever the clock.  Microseconds a k-tile, a workgroup alone on
        // its CU / per workgroup where several share it: 128 x 128 0.95 / 0.75 (1999x2047x1001; 4099x4101x4103), 64 x 64
        // 0.52 / 0.38 (1024x1023x1024; 1999x2047x1001, 2999x3001x3003).  Filling and storing cost a workgroup alone three and
        // five k-tiles; of several, one multiplies while another fills, and it is two (1532x25x1126 on 128 x 128 / 64 x 64
        // tiles 7.4 / 5.8 us, 25 of 239x19x204 7.3 / 5.9; over 223 such products the choice is within 0.5 % of the better
        // tile, with three and five it was 6 %).
        if (any_addr && sizeof(T) == 2)
            cost = rounds == 1 ? (t.bp == 64 ? 0.52 * (kt + 5.0) : 0.95 * (kt + 3.0)) : (double)rounds * (t.bp == 64 ? 0.38 : 0.75) * (kt + 2.0);
        if (best < 0 || cost < best_cost) { best = i; best_cost = cost; }
    }
    // Operands at any address, more 64 x 64 tiles than CUs and k in splits: 128 x 128 tiles that leave half of the chip idle are a poor second above,
    // where a tile walks all of k (2661x7265x442 84 -> 44 us in three splits, 664x7239x1744 70 -> 40, 1248x8121x893 86 -> 56).  A sixth is left for the
    // estimate's error and at least 40 k-tiles are asked for: over 70 such products 0.51 to 0.93 of the time, but of 30 others within that
    // sixth or shorter eight were slower (8005x3321x241 38.2 / 42.6, 2658x3539x763, both transposed, 38.9 / 43.1, 2516x2262x406 21.1 / 22.1).  Not
    // where a capture cannot have the scratch memory for it; the fixed one holds a 128 x 128 tile of partial sums for each of 256 CUs, so
    // agh_gemm_bf16_noalloc takes the same way and gives the same bits.
    if (sizeof(T) == 2 && any_addr && best == 4 && batch == 1 && g.NP > 64 && g.NQ > 64 && !setting("AGH_GEMM_SPLITS")) {
        const int64_t tiles = (int64_t)((g.NP + 127) / 128) * ((g.NQ + 127) / 128), small = (int64_t)((g.NP + 63) / 64) * ((g.NQ + 63) / 64);
        const int ktiles = (g.K + BK - 1) / BK, s = ktiles >= 40 && small > cus ? (int)std::min<int64_t>(cus / tiles, ktiles / 12) : 1;
        const double mb = (double)g.NP * g.NQ * 2e-6;
        const size_t bytes = (size_t)s * g.NQ * g.NPpad * sizeof(float);
        if (s > 1 && bf16_split_us(kBf16SplitAny, s, ktiles, mb) + 3 * 0.95 < 0.83 * best_cost &&
            (fixed_scratch ? bytes <= (size_t)AGH_NOALLOC_SCRATCH_BYTES : workspace_ready(bytes)))
            best = 3;
    }
    if (forced_cfg >= 0) best = forced_cfg;

#ifdef AGH_GEMM_WITH_F32_DIRECT
    if constexpr (sizeof(T) == 4) {
        // 64 x 64 or 128 x 128: by fitted times.  The cost above counts a round of 144 to 256 tiles of 128 x 128 like a full one, and those
        // tiles as if they always shared a CU: 1132x272x3944 44 -> 32 us on 64 x 64, 136x7008x3004 126 -> 96 on 128 x 128.  (Six per cent are left to
        // the estimate: of nine products that it puts 3 to 6 % faster on 128 x 128 five were slower, 6328x4296x168 148 / 153.)  No product's
        // sums get longer by it: where 128 x 128 would be two sums (one workgroup per CU) or more splits of k, 64 x 64 is taken with two
        // sums, or not at all.
        const bool f32_direct = (any_addr || !any_scalar) && g.K > 0 && env_int("AGH_GEMM_DIRECT", 1) != 0;
        if (f32_direct && forced_cfg < 0 && (best == 3 || best == 4) && !(any_addr && skinny) && !setting("AGH_GEMM_SPLITS") &&
            !setting("AGH_GEMM_KSPLIT")) {
            int s64, s128;
            const double us64 = f32_tile_us(64, any_addr, g.NP, g.NQ, g.K, batch, cus, &s64);
            const double us128 = f32_tile_us(128, any_addr, g.NP, g.NQ, g.K, batch, cus, &s128);
            const int64_t tiles128 = (int64_t)((g.NP + 127) / 128) * ((g.NQ + 127) / 128) * batch;
            // (A capture that cannot have scratch memory for the splits of the other tile keeps the one it had.  At any address that is 64 x 64,
            // whatever the cost above says: it is split only where the element-wise loaders' choice is, and needs no more scratch memory, so no
            // capture is refused that those could serve, 1279x1023x959 for one: one split there, three on 128 x 128.)
            const int64_t part = (int64_t)g.NQ * g.NPpad * (int64_t)sizeof(float);
            const bool ready64 = s64 == 1 || workspace_ready((size_t)(s64 * part)), ready128 = s128 == 1 || workspace_ready((size_t)(s128 * part));
            if (any_addr) {
                best = us128 < us64 && ready128 ? 3 : 4;
            } else if (best == 4 && us128 < 0.94 * us64 && ready128) best = 3;
            else if (best == 3 && us64 < 0.97 * us128 && s64 >= s128 && ready64) {
                best = 4;
                g.two_sums = tiles128 * s128 <= cus;
            }
        }
        // Short k and a tile for every CU at least: two workgroups per CU over all tiles.  Over 400 products of 64 to 120000 x 8 to 1200 x 16 to
        // 8192, of those the rule takes 4 are more than 3 % behind the kernels of one tile a workgroup, 6 % at most, all together they are 1.2
        // times as fast (4758 x 32 x 416 10.4 / 7.0 us, 23193 x 256 x 220 40.3 / 31.7; the least 53765 x 256 x 68 40.2 / 40.5; at k = 64 / 128 / 192 /
        // 256 1.39 / 1.23 / 1.13 / 1.09 times).  Beyond the rule, k of 260 to 320 is 0.98 to 1.54 times as fast here, 1.12 over 99 products (3883 x
        // 300 x 3092 92.4 / 71.5); at 352 and 384 it is 1.01 and 1.06 (1076 x 352 x 1800 16.9 / 28.1).  Up to 32 columns of C the 32 x 128
        // tile has less padding (94418 x 196 x 16 20.5 / 41.7).  AGH_GEMM_STREAM=0|1 overrides.
        const int64_t tiles_p = (g.NP + kStreamBP - 1) / kStreamBP, tiles_q = (g.NQ + kStreamBQ - 1) / kStreamBQ;
        const bool can = batch == 1 && !any_scalar && g.K > 0 && beta == 0.0f && !bias && act == AGH_ACT_NONE && g.dp == 1 && g.dq > 0 &&
                         g.dq < (1 << 24) && tiles_p * tiles_q * ((g.K + 31) / 32) < 0x7FFFFFFF && env_int("AGH_GEMM_DIRECT", 1) != 0;
        const int ksplit = env_int("AGH_GEMM_KSPLIT", -1);
        // (a forced tile configuration, split count or eight-wave form means the kernels of one tile a workgroup are wanted)
        const bool suits = g.K <= 256 && g.NP > 32 && g.NQ > 64 && tiles_p * tiles_q >= cus && forced_cfg < 0 && !setting("AGH_GEMM_SPLITS") &&
                           ksplit <= 0;
        // Where its tiles leave a CU one workgroup at most, launch_f32_dl adds the two halves of every k-tile in sums of their own, which rounds
        // less (relative error against 64 bits at k = 128, halves / one chain: 1.47e-7 / 2.03e-7 on normal values, 0.87e-7 / 1.58e-7 on uniform ones
        // from 0 to 1).  So does this kernel for those products, with the same bits; it costs 0.9 % over 179 of them, 1.31 times as fast
        // as there (4273 x 244 x 564 27.6 / 24.6 us, the least gain).
        bool halves = ksplit > 0;
        if (ksplit < 0 && (best == 3 || best == 4)) {
            const TileCfg &t = kCfgs[best];
            halves = g.two_sums || (int64_t)((g.NP + t.bp - 1) / t.bp) * ((g.NQ + t.bq - 1) / t.bq) <= cus;
        }
        if (can && env_int("AGH_GEMM_STREAM", suits) != 0) {
            g.tiles_p = (int)tiles_p;
            g.tiles_q = (int)tiles_q;
            switch (lp * 3 + lq) {
                case LD_K * 3 + LD_K: return launch_f32_stream<LD_K, LD_K>(g, cus, halves);
                case LD_K * 3 + LD_R: return launch_f32_stream<LD_K, LD_R>(g, cus, halves);
                case LD_R * 3 + LD_K: return launch_f32_stream<LD_R, LD_K>(g, cus, halves);
                case LD_R * 3 + LD_R: return launch_f32_stream<LD_R, LD_R>(g, cus, halves);
                default: break;
            }
        }
    }
#endif

    const bool any = any_addr && (best == 3 || best == 4);  // (a skinny tile keeps the element-wise loaders)
    if (any) { lp = lp_any; lq = lq_any; }
    if (best < 0 || best >= kNumCfgs || (any_scalar && !any && !kCfgs[best].scalar_ok))
        return fail(AGH_ERANGE, "%s: no tile configuration for this shape", name);
    const TileCfg &t = kCfgs[best];
    g.tiles_p = (g.NP + t.bp - 1) / t.bp;
    g.tiles_q = (g.NQ + t.bq - 1) / t.bq;

    // ---- split-K when the tile grid cannot fill the chip and k is long ----
    const int64_t tiles = (int64_t)g.tiles_p * g.tiles_q * batch;
    const int ktiles = (g.K + BK - 1) / BK;
    // at least four k-tiles a split; twelve for the bf16 128 x 128 direct tile, whose four-stage ring makes fewer,
    // longer splits the better trade (128x4096x4096: 17.0-17.2 us in 4 to 6 splits, 19.5 in 8)
    int splits = batch == 1 ? plan_splits(tiles, ktiles, cus, direct_ok && best == 3 ? 12 : 4) : 1;
    if (sizeof(T) == 2 && direct_ok && !any_addr && best == 3 && splits == 2 && bf16_one_split(ktiles, (double)g.NP * g.NQ * 2e-6, vec_store)) splits = 1;
    if (batch == 1) splits = env_int("AGH_GEMM_SPLITS", splits);
    if (splits < 1) splits = 1;
    if (splits > ktiles && ktiles > 0) splits = ktiles;
    if (ktiles == 0) splits = 1;
    int tiles_per_split = ktiles > 0 ? (ktiles + splits - 1) / splits : 1;
    splits = ktiles > 0 ? (ktiles + tiles_per_split - 1) / tiles_per_split : 1;
    g.k_per_split = tiles_per_split * BK;

    // bf16 with both operands vector-loadable takes the
    // direct-to-LDS kernel (AGH_GEMM_DIRECT=0 forces the register-staged one)
    const bool direct = direct_ok && (!any_scalar || any);

    if (splits > 1) {
        void *ws = nullptr;
        const size_t bytes = (size_t)splits * g.NQ * g.NPpad * sizeof(float);
        if (int rc = fixed_scratch ? static_workspace(bytes, &ws) : workspace(bytes, &ws)) return rc;
        g.ws = (float *)ws;
        g.store_mode = ST_SPLITK;
        if (int rc = launch_cfg<T>(best, g, splits, lp, lq, direct, any)) return rc;
        const size_t total = (size_t)g.NQ * g.NP;
        int lanes = 1;  // threads per output element: about eight partials each
        while (lanes < 16 && lanes * 16 <= splits) lanes *= 2;
        if (lanes == 1 && vec_store && g.NPpad == g.NP) {
            hipLaunchKernelGGL(splitk_reduce_vec4_kernel<T>, dim3((unsigned)((total / 4 + 255) / 256)), dim3(256), 0,
                               stream(), g, splits);
            AGH_LAUNCH_CHECK("split-K reduce launch");
            return AGH_OK;
        }
        const size_t blocks = (total * lanes + 255) / 256;
        if (blocks > 0x7FFFFFFFull) return fail(AGH_ERANGE, "%s: output too large for split-K", name);
        hipLaunchKernelGGL(splitk_reduce_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, stream(), g, splits, lanes);
        AGH_LAUNCH_CHECK("split-K reduce launch");
        return AGH_OK;
    }
    g.store_mode = vec_store ? ST_VEC : ST_SCALAR;
    if (sizeof(T) == 4 && any && !vec_store && g.dp == 1) {
        // Rows of C that no 16-byte store fits: P and Q change places, so that a store instruction's lanes lie along C's unit-stride
        // axis (the products commute and their order over k stays, so the bits do too): whole lines of C instead of 4 bytes in each of 64.
        std::swap(g.P, g.Q);
        std::swap(g.ps, g.qs);
        std::swap(g.pk, g.qk);
        std::swap(g.NP, g.NQ);
        std::swap(g.dp, g.dq);
        std::swap(g.batch_p, g.batch_q);
        std::swap(g.tiles_p, g.tiles_q);
        std::swap(lp, lq);
        g.NPpad = (g.NP + 3) & ~3;
        g.bias_on_p = !g.bias_on_p;
    }
    // the direct-to-LDS kernel can transpose its output tile through LDS and store full 16-byte
    // chunks when nothing has to be read back from C
    if (direct && best <= 4 && vec_store && beta == 0.0f && g.NP % 8 == 0 && (g.dq % 8 == 0 || g.NQ == 1) &&
        aligned(C, 16) && (batch == 1 || g.batch_d % 8 == 0))
        g.store_mode = ST_STAGED;
    else if (direct && best <= 4 && g.dp == 1 && beta == 0.0f)
        // the same transposition, 16-byte stores to any element address: rows of C that are no whole vectors were stored element by
        // element (both operands aligned: 4096x4096x4095 141 -> 82 us, 16384x256x333 23.1 -> 9.7, 8191x64x1023 22.1 -> 8.8)
        g.store_mode = ST_STAGED_ANY;
    return launch_cfg<T>(best, g, 1, lp, lq, direct, any);
}

}  // namespace gemm
}  // namespace agh
