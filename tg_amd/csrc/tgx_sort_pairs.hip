/*
 * tgx_sort_pairs.hip — stable radix sort of (key, value) pairs (rocPRIM), used
 * by the trace with sorted rays.
 */
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>

#include "tgx_internal.h"

/* Stable ascending sort of (key, value) by the low end_bit bits of key. */
int tgx_prim_sort_pairs_u32(tgx_context* ctx, const uint32_t* keys_in, uint32_t* keys_out, const uint32_t* vals_in,
                            uint32_t* vals_out, uint32_t n, unsigned end_bit)
{
    if (n == 0) return TGX_OK;
    size_t bytes = 0;
    TGX_HIP_CHECK(ctx, rocprim::radix_sort_pairs(nullptr, bytes, keys_in, keys_out, vals_in, vals_out, n, 0u, end_bit,
                                                 ctx->stream));
    int rc = tgx_buffer_reserve(ctx, &ctx->prim_tmp, bytes, "sort scratch");
    if (rc) return rc;
    TGX_HIP_CHECK(ctx, rocprim::radix_sort_pairs(ctx->prim_tmp.ptr, bytes, keys_in, keys_out, vals_in, vals_out, n, 0u,
                                                 end_bit, ctx->stream));
    return TGX_OK;
}
