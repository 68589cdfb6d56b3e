// The page that holds a key, without a division in the loop over the keys.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

// floor(key / page size) for every key below 2^31 and every page size from 2 on: with 2^shift < size <= 2^(shift + 1) and
// magic = ceil(2^(32 + shift) / size), which fits 32 bits, key * magic / 2^(32 + shift) lies above key / size by
// key * e / (size * 2^(32 + shift)), e < size <= 2^(shift + 1), so by less than 1 / size: never as far as the next whole number.
// (Without the shift, ceil(2^32 / size) alone is exact below 2^32 / size keys only where size is no power of two: with one page of
// 163840 tokens a request the keys from 163837 on were looked for in a second page.)
struct PageDivisor { uint32_t magic; int shift; };

inline PageDivisor page_divisor(int size) {
    PageDivisor d{0, 0};
    if (size < 2) return d;
    while ((2ll << d.shift) < size) ++d.shift;
    d.magic = (uint32_t)(((1ull << (32 + d.shift)) + (unsigned)size - 1) / (unsigned)size);
    return d;
}

__host__ __device__ __forceinline__ int page_of_key(const PageDivisor& d, int key) {
    return (int)((uint32_t)((uint64_t)(uint32_t)key * d.magic >> 32) >> d.shift);
}
