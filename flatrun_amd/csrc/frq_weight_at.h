// One weight of a raw GGUF row, for the kernels that compute an exceptional
// row of x weight by weight.
#pragma once

#include "frq_common.h"
#include "frq_kernels.h"

namespace frq {

// Element j of a W row as the dequantizer gives it (fp32, gguf.py op order):
// Q4_K / Q5_K fl(d sc q) - fl(dmin m), Q6_K d sc (q - 32), Q8_0 d q, Q1_0 +-d.
template <int QT>
__device__ float weight_at(const uint8_t* __restrict__ wrow, int j) {
    if constexpr (QT == kTypeQ4K || QT == kTypeQ5K) {
        const uint8_t* bp = wrow + (int64_t)(j >> 8) * (QT == kTypeQ4K ? kQ4KBytes : kQ5KBytes);
        const int e = j & 255, sb = e >> 5, l = e & 31;
        const uint4 h = *reinterpret_cast<const uint4*>(bp);
        uint32_t sc, mn;
        k4_scale_min(h.y, h.z, h.w, sb, sc, mn);
        uint32_t q = (bp[(QT == kTypeQ4K ? 16 : 48) + 32 * (sb >> 1) + l] >> (4 * (sb & 1))) & 15u;
        if constexpr (QT == kTypeQ5K) q |= ((uint32_t)(bp[16 + l] >> sb) & 1u) << 4;
        return f16_bits_to_f32(h.x) * (float)sc * (float)q - f16_bits_to_f32(h.x >> 16) * (float)mn;
    } else if constexpr (QT == kTypeQ6K) {
        const uint8_t* bp = wrow + (int64_t)(j >> 8) * kQ6KBytes;
        const int e = j & 255, hh = e >> 7, ks = (e >> 5) & 3, l = e & 31;
        const uint32_t ql = (bp[64 * hh + 32 * (ks & 1) + l] >> (ks >= 2 ? 4 : 0)) & 15u;
        const uint32_t qh = (bp[128 + 32 * hh + l] >> (2 * ks)) & 3u;
        const float sc = (float)(int)(int8_t)bp[192 + 8 * hh + (l >> 4) + 2 * ks];
        return f16_bits_to_f32(ld_u16(bp + 208)) * sc * (float)((int)(ql | (qh << 4)) - 32);
    } else if constexpr (QT == kTypeQ80) {
        const uint8_t* bp = wrow + (int64_t)(j >> 5) * kQ80Bytes;
        return f16_bits_to_f32(ld_u16(bp)) * (float)(int)(int8_t)bp[2 + (j & 31)];
    } else {
        const uint8_t* bp = wrow + (int64_t)(j >> 7) * kQ10Bytes;
        const float d = f16_bits_to_f32(ld_u16(bp));
        return ((bp[2 + ((j & 127) >> 3)] >> (j & 7)) & 1) ? d : -d;
    }
}

// Bytes of a row of K elements.
template <int QT>
__host__ __device__ constexpr int64_t weight_row_bytes(int64_t K) {
    return QT == kTypeQ4K   ? K / kQKElems * kQ4KBytes
           : QT == kTypeQ5K ? K / kQKElems * kQ5KBytes
           : QT == kTypeQ6K ? K / kQKElems * kQ6KBytes
           : QT == kTypeQ80 ? K / kQ80Elems * kQ80Bytes
                            : K / kQ10Elems * kQ10Bytes;
}

}  // namespace frq
