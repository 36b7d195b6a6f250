// Launch wrappers of the direct-to-LDS bf16 GEMM kernels.  Each agh_gemm_bf16_dl_<tile>.hip includes
// this header and instantiates the four loader pairs of one tile shape.
#pragma once
#include "agh_gemm_bf16_dl.h"

namespace agh {
namespace gemm {

template <int BP, int BQ, int WGP, int WGQ, int LP, int LQ, int NS>
int launch_one_dl(const Args &g, int splits) {
    dim3 grid((unsigned)(g.tiles_p * g.tiles_q), (unsigned)splits, (unsigned)g.batch);
    // the LDS stages are static
    if (g.store_mode == ST_STAGED)
        hipLaunchKernelGGL((gemm_bf16_dl_kernel<BP, BQ, WGP, WGQ, LP, LQ, true, NS>), grid, dim3(WGP * WGQ * 64), 0, stream(), g);
    else
        hipLaunchKernelGGL((gemm_bf16_dl_kernel<BP, BQ, WGP, WGQ, LP, LQ, false, NS>), grid, dim3(WGP * WGQ * 64), 0, stream(), g);
    AGH_LAUNCH_CHECK("gemm (direct-to-LDS) kernel launch");
    return AGH_OK;
}

// Register sets in flight: enough for a load's latency.  A k-tile of the 128 x 128 tile is 32 MFMAs a wave: two sets; a
// k-tile of the 64 x 64 tile is eight: four.  (Four sets for a 128 x 128 workgroup alone on its CU: 30.3 against 32.0 us at
// 1999x2047x1001 and 31.1 against 30.8 at 2000x2047x2001, so no form of its own.)
template <int BP, int BQ, int WGP, int WGQ, int LP, int LQ>
int launch_one_any(const Args &g, int splits) {
    dim3 grid((unsigned)(g.tiles_p * g.tiles_q), (unsigned)splits, (unsigned)g.batch);
    hipLaunchKernelGGL((gemm_bf16_dl_kernel<BP, BQ, WGP, WGQ, LP, LQ, false, 2, BP == 64 ? 4 : 2>), grid, dim3(WGP * WGQ * 64), 0, stream(), g);
    AGH_LAUNCH_CHECK("gemm (any address) kernel launch");
    return AGH_OK;
}

#define AGH_ANY_INSTANTIATE(BP, BQ, WGP, WGQ)                                             \
    template int launch_one_any<BP, BQ, WGP, WGQ, LD_K, LD_K>(const Args &, int);         \
    template int launch_one_any<BP, BQ, WGP, WGQ, LD_K, LD_R>(const Args &, int);         \
    template int launch_one_any<BP, BQ, WGP, WGQ, LD_R, LD_K>(const Args &, int);         \
    template int launch_one_any<BP, BQ, WGP, WGQ, LD_R, LD_R>(const Args &, int);

#define AGH_DL_INSTANTIATE(BP, BQ, WGP, WGQ, NS)                                          \
    template int launch_one_dl<BP, BQ, WGP, WGQ, LD_K, LD_K, NS>(const Args &, int);      \
    template int launch_one_dl<BP, BQ, WGP, WGQ, LD_K, LD_R, NS>(const Args &, int);      \
    template int launch_one_dl<BP, BQ, WGP, WGQ, LD_R, LD_K, NS>(const Args &, int);      \
    template int launch_one_dl<BP, BQ, WGP, WGQ, LD_R, LD_R, NS>(const Args &, int);

}  // namespace gemm
}  // namespace agh
