/*
 * stc_internal.h — shared declarations of the HIP implementation.
 */
#ifndef STC_INTERNAL_H_
#define STC_INTERNAL_H_

#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stddef.h>

#define STC_WAVE 64

#define STC_CHECK(expr)                                                        \
    do {                                                                       \
        hipError_t e_ = (expr);                                                \
        if (e_ != hipSuccess) return stc_hip_fail(e_, #expr, __FILE__, __LINE__); \
    } while (0)

int stc_hip_fail(hipError_t e, const char *expr, const char *file, int line);

/* ---------------- radix sort (stc_radix.hip) ---------------- */
/* Stable LSD radix sort of the pairs (kin, vin) by key bits [0, bits) or [lo_bit, hi_bit), into
 * keys/vals or, when *in_alt is set on return, keys_alt/vals_alt (the other pair is scratch). vin null:
 * the values are 0 .. n - 1. kin and vin are not written unless they are `keys` and `vals` (sorted in
 * place) or `keys_alt` and `vals_alt`. temp must hold stc_radix_temp_words(n) uint32 words. */
size_t stc_radix_temp_words(uint32_t n);
int stc_radix_sort_u32(const uint32_t *kin, const uint32_t *vin, uint32_t *keys, uint32_t *vals, uint32_t *keys_alt,
                       uint32_t *vals_alt, uint32_t n, int bits, uint32_t *temp, bool *in_alt, hipStream_t s);
int stc_radix_sort_u64(const uint64_t *kin, const uint32_t *vin, uint64_t *keys, uint32_t *vals, uint64_t *keys_alt,
                       uint32_t *vals_alt, uint32_t n, int lo_bit, int hi_bit, uint32_t *temp, bool *in_alt, hipStream_t s);
/* exclusive prefix sum of n uint32 values (in may equal out); writes the total
 * to *total_dev when non-null. temp as for the radix sort. */
int stc_exclusive_scan_u32(const uint32_t *in, uint32_t *out, uint32_t n, uint32_t *total_dev, uint32_t *temp,
                           hipStream_t s);

#endif
