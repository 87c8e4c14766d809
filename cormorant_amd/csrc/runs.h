// runs.h -- runs of up to eight int16 values between registers and memory (not public).
#pragma once
#include "cm_internal.h"

namespace runs {

typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// Eight values at byte offset `off` of which the last n are stored: one access
// for all eight, else 1 + 2 + 4 elements from the end.
template <int AUX>
__device__ __forceinline__ void store_tail(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t n, const uint32_t (&d)[4]) {
    if (n == 8u) {
        __builtin_amdgcn_raw_buffer_store_b128(v4u{d[0], d[1], d[2], d[3]}, rs, off, 0, AUX);
        return;
    }
    // the window moves down as pieces are taken off its end
    uint32_t w0 = d[0], w1 = d[1], w2 = d[2], w3 = d[3], end = off + 16u;
    if (n & 1u) {
        end -= 2u;
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)(w3 >> 16), rs, end, 0, 0);
        w3 = __builtin_amdgcn_alignbit(w3, w2, 16);
        w2 = __builtin_amdgcn_alignbit(w2, w1, 16);
        w1 = __builtin_amdgcn_alignbit(w1, w0, 16);
    }
    if (n & 2u) {
        end -= 4u;
        __builtin_amdgcn_raw_buffer_store_b32(w3, rs, end, 0, 0);
        w3 = w2;
        w2 = w1;
    }
    if (n & 4u) __builtin_amdgcn_raw_buffer_store_b64(v2u{w2, w3}, rs, end - 8u, 0, 0);
}

// The first n of eight int16 values at byte offset `off`.
__device__ __forceinline__ v4u load_head(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t n) {
    if (n == 8u) return __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0);
    v4u d;
#pragma unroll
    for (uint32_t q = 0; q < 4; ++q) {
        const uint32_t lo = __builtin_amdgcn_raw_buffer_load_b16(rs, 2u * q < n ? off + 4u * q : kOob, 0, 0);
        const uint32_t hi = __builtin_amdgcn_raw_buffer_load_b16(rs, 2u * q + 1u < n ? off + 4u * q + 2u : kOob, 0, 0);
        d[q] = (lo & 0xFFFFu) | hi << 16;
    }
    return d;
}
// The same values stored.
__device__ __forceinline__ void store_head(__amdgpu_buffer_rsrc_t rs, uint32_t off, uint32_t n, v4u d) {
    if (n == 8u) {
        __builtin_amdgcn_raw_buffer_store_b128(d, rs, off, 0, 0);
        return;
    }
    uint32_t a = d[0], b = d[1];
    if (n & 4u) {
        __builtin_amdgcn_raw_buffer_store_b64(v2u{a, b}, rs, off, 0, 0);
        a = d[2];
        b = d[3];
        off += 8u;
    }
    if (n & 2u) {
        __builtin_amdgcn_raw_buffer_store_b32(a, rs, off, 0, 0);
        a = b;
        off += 4u;
    }
    if (n & 1u) __builtin_amdgcn_raw_buffer_store_b16((uint16_t)a, rs, off, 0, 0);
}

}  // namespace runs
