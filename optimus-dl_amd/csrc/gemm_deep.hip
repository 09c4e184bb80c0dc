// gemm_deep.h for single products: the launches.
#include "gemm_deep.h"

namespace odl {

namespace {

template <int FA, int FB, bool MX>
void launch_deep_tile(int bm, int bn, const GemmArgs &g, int num_cus, hipStream_t stream) {
    const int total = g.tiles_m * g.tiles_n;
    const int whole = (total + 7) / 8 * 8;                // a multiple of 8, as is the launch: see the placement in the kernel
    const dim3 grid((unsigned)(whole < num_cus && warming_pays(g) ? num_cus : whole)), block(256);
    if (bm == 128 && bn == 128) hipLaunchKernelGGL((gemm_nt_deep_kernel<2, 2, FA, FB, MX, GemmArgs>), grid, block, 0, stream, g);
    else if (bm == 128) hipLaunchKernelGGL((gemm_nt_deep_kernel<2, 3, FA, FB, MX, GemmArgs>), grid, block, 0, stream, g);
    else hipLaunchKernelGGL((gemm_nt_deep_kernel<4, 2, FA, FB, MX, GemmArgs>), grid, block, 0, stream, g);
}

template <int FA, int FB>
void launch_deep_fmt(int bm, int bn, const GemmArgs &g, int num_cus, hipStream_t stream) {
    if (g.mx_sa) launch_deep_tile<FA, FB, true>(bm, bn, g, num_cus, stream);
    else launch_deep_tile<FA, FB, false>(bm, bn, g, num_cus, stream);
}

}  // namespace

void launch_gemm_deep(int bm, int bn, int fa, int fb, const GemmArgs &g, int num_cus, hipStream_t stream) {
    if (fa == ODL_FP8_E4M3 && fb == ODL_FP8_E4M3) launch_deep_fmt<ODL_FP8_E4M3, ODL_FP8_E4M3>(bm, bn, g, num_cus, stream);
    else if (fa == ODL_FP8_E5M2 && fb == ODL_FP8_E4M3) launch_deep_fmt<ODL_FP8_E5M2, ODL_FP8_E4M3>(bm, bn, g, num_cus, stream);
    else if (fa == ODL_FP8_E4M3 && fb == ODL_FP8_E5M2) launch_deep_fmt<ODL_FP8_E4M3, ODL_FP8_E5M2>(bm, bn, g, num_cus, stream);
    else launch_deep_fmt<ODL_FP8_E5M2, ODL_FP8_E5M2>(bm, bn, g, num_cus, stream);
}

}  // namespace odl
