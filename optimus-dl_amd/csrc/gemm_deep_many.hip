// gemm_deep.h for several products in one launch: side by side (odl_fp8_gemm_nt_group) or added up (odl_fp8_gemm_nt_chain).
#include "gemm_deep.h"

namespace odl {

namespace {

template <int FA, int FB>
void launch_deep_group_fmt(int bm, int bn, const GemmGroup &gg, int num_cus, hipStream_t stream) {
    const int whole = (gg.total + 7) / 8 * 8;
    bool warm = whole < num_cus;
    for (int s = 0; s < gg.count; ++s) warm = warm && warming_pays(gg.m[s]);
    warm = warm && num_cus - whole >= gg.count;
    const dim3 grid((unsigned)(warm ? num_cus : whole)), block(256);
    if (bm == 128 && bn == 128) hipLaunchKernelGGL((gemm_nt_deep_kernel<2, 2, FA, FB, false, GemmGroup>), grid, block, 0, stream, gg);
    else if (bm == 128) hipLaunchKernelGGL((gemm_nt_deep_kernel<2, 3, FA, FB, false, GemmGroup>), grid, block, 0, stream, gg);
    else hipLaunchKernelGGL((gemm_nt_deep_kernel<4, 2, FA, FB, false, GemmGroup>), grid, block, 0, stream, gg);
}

template <int FA, int FB>
void launch_deep_chain_fmt(int bm, int bn, const GemmChain &gc, int num_cus, hipStream_t stream) {
    const int whole = (gc.m[0].tiles_m * gc.m[0].tiles_n + 7) / 8 * 8;
    bool warm = whole < num_cus;
    for (int s = 0; s < gc.count; ++s) warm = warm && warming_pays(gc.m[s]);
    const dim3 grid((unsigned)(warm ? num_cus : whole)), block(256);
    if (bm == 128 && bn == 128) hipLaunchKernelGGL((gemm_nt_deep_kernel<2, 2, FA, FB, false, GemmChain>), grid, block, 0, stream, gc);
    else if (bm == 128) hipLaunchKernelGGL((gemm_nt_deep_kernel<2, 3, FA, FB, false, GemmChain>), grid, block, 0, stream, gc);
    else hipLaunchKernelGGL((gemm_nt_deep_kernel<4, 2, FA, FB, false, GemmChain>), grid, block, 0, stream, gc);
}

}  // namespace

void launch_gemm_deep_group(int bm, int bn, int fa, int fb, const GemmGroup &gg, int num_cus, hipStream_t stream) {
    if (fa == ODL_FP8_E4M3 && fb == ODL_FP8_E4M3) launch_deep_group_fmt<ODL_FP8_E4M3, ODL_FP8_E4M3>(bm, bn, gg, num_cus, stream);
    else if (fa == ODL_FP8_E5M2 && fb == ODL_FP8_E4M3) launch_deep_group_fmt<ODL_FP8_E5M2, ODL_FP8_E4M3>(bm, bn, gg, num_cus, stream);
    else launch_deep_group_fmt<ODL_FP8_E5M2, ODL_FP8_E5M2>(bm, bn, gg, num_cus, stream);
}

void launch_gemm_deep_chain(int bm, int bn, int fa, int fb, const GemmChain &gc, int num_cus, hipStream_t stream) {
    if (fa == ODL_FP8_E4M3 && fb == ODL_FP8_E4M3) launch_deep_chain_fmt<ODL_FP8_E4M3, ODL_FP8_E4M3>(bm, bn, gc, num_cus, stream);
    else if (fa == ODL_FP8_E5M2 && fb == ODL_FP8_E4M3) launch_deep_chain_fmt<ODL_FP8_E5M2, ODL_FP8_E4M3>(bm, bn, gc, num_cus, stream);
    else launch_deep_chain_fmt<ODL_FP8_E5M2, ODL_FP8_E5M2>(bm, bn, gc, num_cus, stream);
}

}  // namespace odl
