// kvc_fused_mfma_packed.hip -- the matrix-core kernels for codes of at most 7 bits whose payloads are packed (kvc_plan_fused says
// which calls those are).
#include "kvc_fused_mfma_impl.h"

// compiled in kvc_fused_mfma_v96.hip
extern template __global__ void kvc_fused_mfma_kernel<1, 4, true, KVC_BOOK_PACKED>(KvcFusedArgs);
extern template __global__ void kvc_fused_mfma_kernel<1, 4, false, KVC_BOOK_PACKED>(KvcFusedArgs);

template <int REP, bool ROUNDED>
static void kvc_launch_packed_kind(int kind, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream)
{
    if (kind == 0) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 0, ROUNDED, KVC_BOOK_PACKED>), grid, dim3(KVC_WG), lds, stream, a);
    else if (kind == 1) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 1, ROUNDED, KVC_BOOK_PACKED>), grid, dim3(KVC_WG), lds, stream, a);
    else if (kind == 2) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 2, ROUNDED, KVC_BOOK_PACKED>), grid, dim3(KVC_WG), lds, stream, a);
    else if (kind == 3) hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 3, ROUNDED, KVC_BOOK_PACKED>), grid, dim3(KVC_WG), lds, stream, a);
    else hipLaunchKernelGGL((kvc_fused_mfma_kernel<REP, 4, ROUNDED, KVC_BOOK_PACKED>), grid, dim3(KVC_WG), lds, stream, a);
}

void kvc_launch_fused_packed(int rep, int kind, bool rounded, const KvcFusedArgs &a, dim3 grid, size_t lds, hipStream_t stream)
{
#define KVC_PACKED_REP(R)                                                         \
    if (rounded) kvc_launch_packed_kind<R, true>(kind, a, grid, lds, stream);     \
    else kvc_launch_packed_kind<R, false>(kind, a, grid, lds, stream)
    switch (rep) {
        case 1: KVC_PACKED_REP(1); break;
        case 2: KVC_PACKED_REP(2); break;
        case 4: KVC_PACKED_REP(4); break;
        default: KVC_PACKED_REP(8); break;
    }
#undef KVC_PACKED_REP
}
