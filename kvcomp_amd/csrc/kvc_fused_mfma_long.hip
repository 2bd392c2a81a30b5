// kvc_fused_mfma_long.hip -- the matrix-core kernels for codebooks with codes of more than 7 bits (alphabets of at most 64
// symbols, rounded arithmetic): K, and V with the softmax on the fly.
#include "kvc_fused_mfma_impl.h"

template <int REP>
static void kvc_launch_long_kind(int kind, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream)
{
    if (kind == 0) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 0, true, KVC_BOOK_LONG>), grid, dim3(KVC_WG), lds, stream, a);
    else if (kind == 3) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 3, true, KVC_BOOK_LONG>), grid, dim3(KVC_WG), lds, stream, a);
    else hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 4, true, KVC_BOOK_LONG>), grid, dim3(KVC_WG), lds, stream, a);
}

void kvc_launch_fused_long(int rep, int kind, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream)
{
    switch (rep) {
        case 1: kvc_launch_long_kind<1>(kind, a, grid, lds, stream); break;
        case 2: kvc_launch_long_kind<2>(kind, a, grid, lds, stream); break;
        case 4: kvc_launch_long_kind<4>(kind, a, grid, lds, stream); break;
        default: kvc_launch_long_kind<8>(kind, a, grid, lds, stream); break;
    }
}
