/*
 * tgx_prims.hip — device-wide scan (rocPRIM). A translation unit's kernels are
 * loaded together when the first of them runs, and rocPRIM's sorts are 2 to 3 MB
 * of code each: the scan, the sort of pairs (tgx_sort_pairs.hip) and the sort of
 * keys (tgx_sort_keys.hip) are apart, so that a process loads what it uses. Its
 * first SVO build takes 8.4 ms so, 15.4 with the three in one.
 */
#include <rocprim/device/device_scan.hpp>

#include "tgx_internal.h"

int tgx_prim_exclusive_scan_u32(tgx_context* ctx, const uint32_t* in, uint32_t* out, uint32_t n)
{
    if (n == 0) return TGX_OK;
    size_t bytes = 0;
    TGX_HIP_CHECK(ctx, rocprim::exclusive_scan(nullptr, bytes, in, out, 0u, n, rocprim::plus<uint32_t>(), ctx->stream));
    int rc = tgx_buffer_reserve(ctx, &ctx->prim_tmp, bytes, "scan scratch");
    if (rc) return rc;
    TGX_HIP_CHECK(ctx, rocprim::exclusive_scan(ctx->prim_tmp.ptr, bytes, in, out, 0u, n, rocprim::plus<uint32_t>(),
                                               ctx->stream));
    return TGX_OK;
}
