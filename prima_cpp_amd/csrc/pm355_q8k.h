// pm355_q8k.h — a 256-value Q8_K block by one wave (quantize.hip, and the attention kernels that end in the wo product's activations).
#pragma once
#include "pm355_device.h"
#include "pm355_kernels.h"

#ifdef __HIPCC__
namespace q8k {
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_keep_f(float v) {   // lanes outside ROW_MASK / out of range keep v
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, false));
}
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ int dpp_keep_i(int v) {
    return __builtin_amdgcn_update_dpp(v, v, CTRL, ROW_MASK, 0xF, false);
}
__device__ __forceinline__ float wave_max(float v) {
    v = fmaxf(v, dpp_keep_f<0xB1>(v));
    v = fmaxf(v, dpp_keep_f<0x4E>(v));
    v = fmaxf(v, dpp_keep_f<0x141>(v));
    v = fmaxf(v, dpp_keep_f<0x140>(v));
    v = fmaxf(v, dpp_keep_f<0x142, 0xA>(v));
    v = fmaxf(v, dpp_keep_f<0x143, 0xC>(v));
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ int wave_min_i(int v) {
    v = min(v, dpp_keep_i<0xB1>(v));
    v = min(v, dpp_keep_i<0x4E>(v));
    v = min(v, dpp_keep_i<0x141>(v));
    v = min(v, dpp_keep_i<0x140>(v));
    v = min(v, dpp_keep_i<0x142, 0xA>(v));
    v = min(v, dpp_keep_i<0x143, 0xC>(v));
    return __builtin_amdgcn_readlane(v, 63);
}
}

// One wave quantizes one 256-value block held as 4 consecutive values per lane.
__device__ __forceinline__ void q8k_block_from_regs(const float v[4], int lane, uint8_t * row_out, int K, int blk, const pm_q8k_tables & tb = pm_q8k_tables(), int row = 0, const pm_q8k_wide & wd = pm_q8k_wide()) {
    float a0 = fabsf(v[0]), a1 = fabsf(v[1]), a2 = fabsf(v[2]), a3 = fabsf(v[3]);
    const float amax = q8k::wave_max(fmaxf(fmaxf(a0, a1), fmaxf(a2, a3)));
    int8_t  * qs    = (int8_t *) row_out;
    float   * dd    = (float *) (row_out + K);
    int16_t * bsums = (int16_t *) (row_out + K + (K / PM_QK_K) * 4);
    uint32_t packed = 0;
    int psum = 0;
    if (amax != 0.0f) {
        // lowest index with |x| == amax; low bit carries its sign
        int key = 0x7fffffff;
        if (a3 == amax) key = ((4 * lane + 3) << 1) | (v[3] < 0.0f);
        if (a2 == amax) key = ((4 * lane + 2) << 1) | (v[2] < 0.0f);
        if (a1 == amax) key = ((4 * lane + 1) << 1) | (v[1] < 0.0f);
        if (a0 == amax) key = ((4 * lane + 0) << 1) | (v[0] < 0.0f);
        key = q8k::wave_min_i(key);
        const float vmax = (key & 1) ? -amax : amax;
        const float iscale = -127.f / vmax;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            int q = nearest_int_rne(iscale * v[i]);
            q = q > 127 ? 127 : q;
            psum += q;
            packed |= (uint32_t) (q & 0xFF) << (8 * i);
        }
        if (row_out && lane == 0) dd[blk] = 1 / iscale;
        if (wd.q && lane == 0) wd.d[(size_t) blk * wd.ldt + row] = 1 / iscale;
        if (tb.base && lane == 0) ((float *) (tb.base + (size_t) (row >> 5) * tb.tab_bytes + (size_t) tb.nsb * 1024))[blk * 32 + (row & 31)] = 1 / iscale;
    } else if (lane == 0) {
        if (row_out) dd[blk] = 0.0f;
        if (wd.q) wd.d[(size_t) blk * wd.ldt + row] = 0.0f;
        if (tb.base) ((float *) (tb.base + (size_t) (row >> 5) * tb.tab_bytes + (size_t) tb.nsb * 1024))[blk * 32 + (row & 31)] = 0.0f;
    }
    if (row_out) ((uint32_t *) (qs + (size_t) blk * PM_QK_K))[lane] = packed;
    // A-operand order (pm_q8k_tables::qbase): values 4 lane .. 4 lane + 3 = bytes 4 (lane % 4) of sub-block lane / 8, half (lane / 4) % 2
    if (tb.qbase) *(uint32_t *) (tb.qbase + (size_t) (row >> 5) * tb.nsb * 8192 + (size_t) blk * 8192 + (lane >> 3) * 1024 + ((((lane >> 2) & 1) * 32 + (row & 31)) * 16) + 4 * (lane & 3)) = packed;
    // bsums: 16 values = 4 lanes (one quad)
    psum += dpp_i<0xB1>(psum);
    psum += dpp_i<0x4E>(psum);
    if (row_out && (lane & 3) == 0) bsums[blk * 16 + (lane >> 2)] = (int16_t) psum;
    if (wd.q) {
        typedef _Float16 h4 __attribute__((ext_vector_type(4)));
        *(h4 *) (wd.q + (size_t) row * K + (size_t) blk * PM_QK_K + 4 * lane) =
            h4{(_Float16) (int) (int8_t) packed, (_Float16) (int) (int8_t) (packed >> 8), (_Float16) (int) (int8_t) (packed >> 16), (_Float16) (int) (int8_t) (packed >> 24)};
        if ((lane & 3) == 0) wd.s[((size_t) blk * wd.ldt + row) * 16 + (lane >> 2)] = __builtin_bit_cast(uint16_t, (_Float16) (float) psum);
    }
    if (tb.base && (lane & 3) == 0) {              // group G = lane / 4 -> operand lane (row % 32) + 32 (G & 1), slot G / 2 (mmq_i8.hip mmq_prep_kernel)
        const int G = lane >> 2;
        ((_Float16 *) (tb.base + (size_t) (row >> 5) * tb.tab_bytes))[((size_t) blk * 64 + (row & 31) + 32 * (G & 1)) * 8 + (G >> 1)] = (_Float16) (float) psum;
    }
}
#endif
