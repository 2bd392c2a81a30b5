// kvc_fused_mfma_mid.hip -- the matrix-core kernels for codebooks whose longest codes have 6 or 7 bits and whose symbols are 16 at
// most, looked up one at a time (rounded arithmetic).
#include "kvc_fused_mfma_impl.h"

// compiled in kvc_fused_mfma_v96.hip
extern template __global__ void kvc_fused_mfma_kernel<1, 4, true, KVC_BOOK_MID>(KvcFusedArgs);

template <int REP>
static void kvc_launch_mid_kind(int kind, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream)
{
    if (kind == 0) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 0, true, KVC_BOOK_MID>), grid, dim3(KVC_WG), lds, stream, a);
    else if (kind == 1) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 1, true, KVC_BOOK_MID>), grid, dim3(KVC_WG), lds, stream, a);
    else if (kind == 2) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 2, true, KVC_BOOK_MID>), grid, dim3(KVC_WG), lds, stream, a);
    else if (kind == 3) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 3, true, KVC_BOOK_MID>), grid, dim3(KVC_WG), lds, stream, a);
    else hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 4, true, KVC_BOOK_MID>), grid, dim3(KVC_WG), lds, stream, a);
}

void kvc_launch_fused_mid(int rep, int kind, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream)
{
    switch (rep) {
        case 1: kvc_launch_mid_kind<1>(kind, a, grid, lds, stream); break;
        case 2: kvc_launch_mid_kind<2>(kind, a, grid, lds, stream); break;
        case 4: kvc_launch_mid_kind<4>(kind, a, grid, lds, stream); break;
        default:               // (K only)
            hipLaunchKernelGGL((kvc_fused_mfma_kernel<8, 0, true, KVC_BOOK_MID>), grid, dim3(KVC_WG), lds, stream, a);
            break;
    }
}
