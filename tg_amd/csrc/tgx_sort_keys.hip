/*
 * tgx_sort_keys.hip — radix sort of 64-bit keys (rocPRIM), used by the SVO build.
 */
#include <cstring>

#include <rocprim/device/device_radix_sort.hpp>

#include "tgx_internal.h"

/* Ascending sort of the low end_bit bits of 64-bit keys. */
int tgx_prim_sort_keys_u64(tgx_context* ctx, const uint64_t* keys_in, uint64_t* keys_out, uint32_t n, unsigned end_bit)
{
    if (n == 0) return TGX_OK;
    size_t bytes = 0;
    TGX_HIP_CHECK(ctx, rocprim::radix_sort_keys(nullptr, bytes, keys_in, keys_out, n, 0u, end_bit, ctx->stream));
    int rc = tgx_buffer_reserve(ctx, &ctx->prim_tmp, bytes, "sort scratch");
    if (rc) return rc;
    TGX_HIP_CHECK(ctx, rocprim::radix_sort_keys(ctx->prim_tmp.ptr, bytes, keys_in, keys_out, n, 0u, end_bit, ctx->stream));
    return TGX_OK;
}
