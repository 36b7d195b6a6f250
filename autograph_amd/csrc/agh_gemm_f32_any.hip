// f32 GEMM kernels for operands at any element address (agh_gemm_f32_dl.h with 4-byte direct loads): all four loader pairs of
// the 64x64 and 128x128 tiles.  Every k-tile is split between two waves (KS = 2): with four loads where the aligned form has
// one, the second wave of a SIMD hides more than elsewhere (over 108 products 4 % faster on 64x64 tiles and 1 % on 128x128 than one wave
// a tile position, and two sums over k round less than one).
#include "agh_gemm_f32_dl.h"

namespace agh {
namespace gemm {

template <int TP, int TQ, int NS, int LP, int LQ>
int launch_one_f32_any(const Args &g, int splits) {
    auto kern = gemm_f32_dl_kernel<TP, TQ, NS, LP, LQ, 2, 1>;
    constexpr size_t smem = F32DlGeo<TP, TQ, NS, LP, LQ>::SMEM_BYTES;
    static bool attr_done = false;
    if (!attr_done) {
        if (smem > 48 * 1024)
            AGH_HIP(hipFuncSetAttribute((const void *)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
        attr_done = true;
    }
    dim3 grid((unsigned)(g.tiles_p * g.tiles_q), (unsigned)splits, (unsigned)g.batch);
    hipLaunchKernelGGL(kern, grid, dim3(512), smem, stream(), g);
    AGH_LAUNCH_CHECK("gemm (f32, any address) kernel launch");
    return AGH_OK;
}

#define AGH_F32_ANY(T, NS)                                                         \
    template int launch_one_f32_any<T, T, NS, LD_K, LD_K>(const Args &, int);      \
    template int launch_one_f32_any<T, T, NS, LD_K, LD_R>(const Args &, int);      \
    template int launch_one_f32_any<T, T, NS, LD_R, LD_K>(const Args &, int);      \
    template int launch_one_f32_any<T, T, NS, LD_R, LD_R>(const Args &, int);
AGH_F32_ANY(1, 4)
AGH_F32_ANY(2, 2)
#undef AGH_F32_ANY

}  // namespace gemm
}  // namespace agh
