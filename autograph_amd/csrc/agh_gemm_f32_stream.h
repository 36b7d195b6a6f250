// f32 GEMM with short k and many tiles (the input gradients of convolutions and Dense layers, 1x1 and thin convolutions): two
// workgroups per CU walk a run of tiles each, and the operand k-tiles of a run are ONE stream through a ring of LDS stages.
//
// With a workgroup per tile, a tile's first loads and its stores cost as much as the four k-tiles in between (50176 x 128 x 576:
// 98 us, of which 52 are multiplications; 45 with a quarter of the k), and workgroups that start together wait together.  Here
// the loads of the next tile go out while this one is multiplied, its stores leave while the next one is, and neither is waited
// for: a wait counts the loads AND the stores issued after the load it waits for (vector memory operations complete in
// order).  One of a CU's two workgroups has a higher priority, so that one stores while the other multiplies (without: 75.5 against
// 73.4 us below).
//
// Tile 64 (p) x 128 (q), eight waves in a 2 x 4 grid, one 32 x 32 tile a wave, three stages of 24 KB.  LDS images, fragments and
// order of sums as in agh_gemm_f32_dl.h: KS = 1 one accumulator, as with one wave per tile position there, KS = 2 one for either half of
// every k-tile, added at the tile's end, as with two (agh_gemm_host.h says where; 109 to 111 and 125 to 127 of 128 registers).  The operands
// change places in the MFMA: lane l holds D[8 (r / 4) + 4 (l / 32) + r % 4][l % 32] as (q, p), so a store instruction writes whole 128-byte lines of two rows of C.
//
// 50176 x 128 x 576 97 -> 73 us, 802816 x 64 x 576 950 -> 647, 16384 x 64 x 8192 250 -> 190, 12012 x 128 x 6400 216 -> 183, 100000 x 128 x 64
// 49 -> 25.  What bounds it at k = 128: 61 us a multiple of the 52 that the matrix pipes need, and 4 TB/s of stores in between.
// Tried: one workgroup per CU on five stages (78.5), with 256-row tiles (74.4); the stores of a tile spread over the first MFMAs
// of the next one (84: the values move to other registers first).
//
// Requirements checked by the host: those of agh_gemm_f32_dl.h, no split-K, no batch, C = alpha A B with p its unit-stride axis and a
// row pitch of 1 .. 2^24 - 1 elements.
#pragma once
#include "agh_gemm_f32_dl.h"

namespace agh {
namespace gemm {

constexpr int kStreamStages = 3, kStreamBP = 64, kStreamBQ = 128, kStreamPerCu = 2;

template <int LP, int LQ>
struct F32StreamGeo {
    typedef F32DlOperand<LP, kStreamBP> OpP;
    typedef F32DlOperand<LQ, kStreamBQ> OpQ;
    static constexpr int STAGE_BYTES = OpP::BYTES + OpQ::BYTES;
    static constexpr int SMEM_BYTES = kStreamStages * STAGE_BYTES;
};

// one store instruction, whatever the compiler makes of its neighbours: the waits count them
__device__ __forceinline__ void store_counted(const float *uniform_base, uint32_t byte_off, float v) {
    asm volatile("global_store_dword %0, %1, %2" ::"v"(byte_off), "v"(v), "s"(uniform_base) : "memory");
}

template <int LP, int LQ, int KS>
__global__ __launch_bounds__(512, 2 * kStreamPerCu) void gemm_f32_stream_kernel(Args g) {
    static_assert(KS == 1 || KS == 2, "one chain of additions over k, or one for each half of the k-tiles");
    typedef F32StreamGeo<LP, LQ> Geo_;
    typedef typename Geo_::OpP OpP;
    typedef typename Geo_::OpQ OpQ;
    constexpr int NS = kStreamStages, BP = kStreamBP, BQ = kStreamBQ, BK = 32, STAGE_BYTES = Geo_::STAGE_BYTES;
    constexpr int NLP = OpP::LOADS / 8, NLQ = OpQ::LOADS / 8, NL = NLP + NLQ;  // direct loads a wave issues per k-tile
    static_assert(NLP == 1 && NLQ == 2 && NL <= 4, "eight waves share the loads of a k-tile, one behind each of the first MFMAs");
    constexpr int AHEAD = NS - 1, INFLIGHT = (NS - 2) * NL, STORES = 16;
    static_assert(NS == 3 && INFLIGHT + STORES <= 63, "the counted operations must fit the counter");
    extern __shared__ __align__(16) unsigned char smem[];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wp = wave & 1, wq = wave >> 1;
    if (blockIdx.x >= gridDim.x / 2) __builtin_amdgcn_s_setprio(2);
    // this workgroup's run of tiles, p fastest; consecutive runs on one XCD (the grid is a multiple of eight)
    const int run = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    const int64_t all = (int64_t)g.tiles_p * g.tiles_q;
    const int first = (int)(all * run / gridDim.x), last = (int)(all * (run + 1) / gridDim.x);
    if (first >= last) return;
    const int KT = (g.K + BK - 1) / BK, rem = g.K - (KT - 1) * BK;  // k-tiles; depth of the last one
    const int steps = (last - first) * KT;

    // ---- the load stream: k-tile `lk` of tile `lt` next, from gp / gq ----
    const unsigned char *gp[NLP], *gq[NLQ];
    const int64_t stepP = (LP == LD_K ? (int64_t)BK : (int64_t)BK * g.pk) * 4, stepQ = (LQ == LD_K ? (int64_t)BK : (int64_t)BK * g.qk) * 4;
    int lt = first, lk = 0;
    auto aim = [&](auto opc, auto modec, auto nc, const void *base, int64_t rs, int64_t ks, int r0, int NR, auto &ptr) {
        typedef typename decltype(opc)::type Op;
        constexpr int MODE = decltype(modec)::value, N = decltype(nc)::value;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int inst = wave * N + i;
            if constexpr (MODE == LD_K) {
                const int row = inst * 8 + (lane >> 3);
                ptr[i] = (const unsigned char *)base + ((int64_t)min(r0 + row, NR - 1) * rs + ((lane & 7) ^ (int)swz((uint32_t)row)) * 4) * 4;
            } else {
                constexpr int LPK = 64 / Op::KRPI;
                int rowg = r0 + (lane % LPK) * 4;
                if (rowg >= NR) rowg = NR - 4;  // NR is a multiple of 4 on this path
                ptr[i] = (const unsigned char *)base + ((int64_t)(inst * Op::KRPI + lane / LPK) * ks + rowg) * 4;
            }
        }
    };
    auto aim_tile = [&](int t) {
        const int tq = t / g.tiles_p, tp = t - tq * g.tiles_p;
        aim(std::common_type<OpP>{}, std::integral_constant<int, LP>{}, std::integral_constant<int, NLP>{}, g.P, g.ps, g.pk, tp * BP, g.NP, gp);
        aim(std::common_type<OpQ>{}, std::integral_constant<int, LQ>{}, std::integral_constant<int, NLQ>{}, g.Q, g.qs, g.qk, tq * BQ, g.NQ, gq);
    };
    // whether this lane's 16 bytes of load `inst` lie below k = rem of a shorter last k-tile
    auto below = [&](auto opc, auto modec, int inst) {
        typedef typename decltype(opc)::type Op;
        if constexpr (decltype(modec)::value == LD_K) return ((lane & 7) ^ (int)swz((uint32_t)(inst * 8 + (lane >> 3)))) * 4 < rem;
        else return inst * Op::KRPI + lane / (64 / Op::KRPI) < rem;
    };
    const uint32_t smem_addr = __builtin_amdgcn_readfirstlane(lds_address(smem));
    // load l of the stream's next k-tile into stage `slot`; in front of the stream's end the last k-tile stays the next one (its
    // image is then never read)
    auto request = [&](int slot, auto lc) {
        constexpr int l = decltype(lc)::value;
        const uint32_t st = smem_addr + (uint32_t)slot * STAGE_BYTES;
        const bool shorter = rem < BK && lk == KT - 1;  // uniform
        if constexpr (l < NLP) {
            const unsigned char *src = gp[l];
            if (shorter && !below(std::common_type<OpP>{}, std::integral_constant<int, LP>{}, wave * NLP + l)) src = (const unsigned char *)kZeroChunkF32;
            direct_load16(src, st + (uint32_t)(wave * NLP + l) * OpP::IMG);
        } else {
            const unsigned char *src = gq[l - NLP];
            if (shorter && !below(std::common_type<OpQ>{}, std::integral_constant<int, LQ>{}, wave * NLQ + l - NLP)) src = (const unsigned char *)kZeroChunkF32;
            direct_load16(src, st + OpP::BYTES + (uint32_t)(wave * NLQ + l - NLP) * OpQ::IMG);
        }
        if constexpr (l == NL - 1) {  // on to the next k-tile
            if (lk + 1 < KT) {
                ++lk;
                gp[0] += stepP;
                gq[0] += stepQ;
                gq[1] += stepQ;
            } else if (lt + 1 < last) {
                lk = 0;
                aim_tile(++lt);
            }
        }
    };

    // ---- fragments: lane l supplies row l % 32, k = 8 s + 4 (l / 32) + e ----
    const uint32_t lrow = lane & 31, lg = lane >> 5;
    auto frag_offset = [&](auto opc, auto modec, uint32_t row) -> uint32_t {
        typedef typename decltype(opc)::type Op;
        if constexpr (decltype(modec)::value == LD_K) return row * 128u + ((lg ^ swz(row)) << 4);
        else return lg * (uint32_t)Op::koff(4) + row * 4u;
    };
    const uint32_t fp = frag_offset(std::common_type<OpP>{}, std::integral_constant<int, LP>{}, (uint32_t)wp * 32u + lrow);
    const uint32_t fq = frag_offset(std::common_type<OpQ>{}, std::integral_constant<int, LQ>{}, (uint32_t)wq * 32u + lrow);
    auto frag_read = [&](auto opc, auto modec, const unsigned char *op, uint32_t off, auto sc) -> uint4 {
        typedef typename decltype(opc)::type Op;
        constexpr int s = decltype(sc)::value;
        if constexpr (decltype(modec)::value == LD_K) {
            return *(const uint4 *)(op + (off ^ (uint32_t)(s << 5)));
        } else {
            const unsigned char *p = op + off + Op::koff(8 * s);
            return make_uint4(*(const uint32_t *)(p + Op::koff(0)), *(const uint32_t *)(p + Op::koff(1)),
                              *(const uint32_t *)(p + Op::koff(2)), *(const uint32_t *)(p + Op::koff(3)));
        }
    };
    auto read_frags = [&](uint4 &pf, uint4 &qf, const unsigned char *stage, auto sc) {
        pf = frag_read(std::common_type<OpP>{}, std::integral_constant<int, LP>{}, stage, fp, sc);
        qf = frag_read(std::common_type<OpQ>{}, std::integral_constant<int, LQ>{}, stage + OpP::BYTES, fq, sc);
    };

    f32x16 acc[KS];
    auto clear = [&] {
#pragma unroll
        for (int h = 0; h < KS; ++h)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[h][r] = 0.0f;
    };
    clear();
    uint4 pa, qa, pb, qb;
    aim_tile(first);
    for (int t = 0; t < AHEAD; ++t) static_for<NL>([&](auto lc) { request(t, lc); });
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((AHEAD - 1) * NL) : "memory");  // this wave's part of the first k-tile has landed
    __builtin_amdgcn_s_barrier();                                           // and everybody else's
    asm volatile("" ::: "memory");
    read_frags(pa, qa, smem, std::integral_constant<int, 0>{});

    // a substep's four MFMAs out of one fragment set; the next substep's fragments are read in front of the first
    auto substep = [&](f32x16 &sum, const uint4 &xp, const uint4 &xq, uint4 &yp, uint4 &yq, const unsigned char *stage, auto sc, auto &&extra) {
        read_frags(yp, yq, stage, sc);
        static_for<4>([&](auto mc) {
            Mma<float>::template part<decltype(mc)::value>(sum, xq, xp);
            extra(mc);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    auto nothing = [](auto) {};
    int slot = 0, kt = 0, tile = first;
    bool stored = false;  // a whole tile was stored at the end of the last step
    for (int s = 0; s < steps; ++s) {
        const int nslot = slot + 1 == NS ? 0 : slot + 1, free_slot = slot == 0 ? NS - 1 : slot - 1;  // left in the last step
        const unsigned char *cur = smem + slot * STAGE_BYTES, *nxt = smem + nslot * STAGE_BYTES;
        substep(acc[0], pa, qa, pb, qb, cur, std::integral_constant<int, 1>{}, [&](auto mc) {
            constexpr int m = decltype(mc)::value;
            if constexpr (m < NL) request(free_slot, mc);
        });
        substep(acc[0], pb, qb, pa, qa, cur, std::integral_constant<int, 2>{}, nothing);
        substep(acc[KS - 1], pa, qa, pb, qb, cur, std::integral_constant<int, 3>{}, nothing);
        // The next k-tile becomes visible.  Its loads went out in the last step; issued since: those of the k-tile behind it, and the
        // stores of a whole tile that ended with that step (other stores are not counted: waiting for more than needed is safe).
        if (stored) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(INFLIGHT + STORES) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(INFLIGHT) : "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        substep(acc[KS - 1], pb, qb, pa, qa, nxt, std::integral_constant<int, 0>{}, nothing);
        slot = nslot;
        stored = false;
        if (++kt < KT) continue;
        if constexpr (KS == 2) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[0][r] += acc[1][r];
        }
        // ---- the tile is complete: element r = D[p][q] with p = p0 + l % 32, q = q0 + 8 (r / 4) + 4 (l / 32) + r % 4 ----
        kt = 0;
        const int tq = tile / g.tiles_p, tp = tile - tq * g.tiles_p;
        ++tile;
        const int p0 = tp * BP + wp * 32, q0 = tq * BQ + wq * 32;
        float *row = (float *)g.D + (int64_t)q0 * g.dq + p0;
        if (p0 + 32 <= g.NP && q0 + 32 <= g.NQ) {  // uniform
            // sixteen stores, counted above
            const uint32_t off = (lg * 4u * (uint32_t)g.dq + lrow) * 4u;
#pragma unroll
            for (int r = 0; r < 16; ++r) store_counted(row + (int64_t)(8 * (r >> 2) + (r & 3)) * g.dq, off, g.alpha * acc[0][r]);
            stored = true;
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int q = (int)lg * 4 + 8 * (r >> 2) + (r & 3);
                if (p0 + (int)lrow < g.NP && q0 + q < g.NQ) row[(int64_t)q * g.dq + lrow] = finish_plain<float>(acc[0][r], g.alpha);
            }
        }
        clear();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the requests past the last k-tile still write LDS
}

}  // namespace gemm
}  // namespace agh
