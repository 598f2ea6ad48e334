// How two lanes share a row of n >= 1 16-byte partial pairs (ln_pair_load): the lower lane takes the first (n + 1) / 2, the upper
// the rest. Plain C++, so that a host program can enumerate the indices.
#pragma once
#include <stdint.h>
#ifdef __HIPCC__
#define SH_LN_PAIR_FN __host__ __device__ __forceinline__
#else
#define SH_LN_PAIR_FN static inline
#endif

// Entries of the upper (up = 1) or lower lane.
SH_LN_PAIR_FN uint32_t ln_pair_count(uint32_t n, uint32_t up) { return up ? n / 2 : (n + 1) / 2; }
// The entry of the row that the lane requests as its h-th (h < ln_pair_count(n, 0), so both lanes issue the same loads): past its
// own count its last one again, and with none of its own (n = 1) the lower lane's, never one past the row.
SH_LN_PAIR_FN uint32_t ln_pair_at(uint32_t n, uint32_t up, uint32_t h) {
    const uint32_t c = ln_pair_count(n, up), k = h < c ? h : c - 1;
    return c ? (up ? ln_pair_count(n, 0) : 0u) + k : 0u;
}
