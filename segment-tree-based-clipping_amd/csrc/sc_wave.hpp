// sc_wave.hpp -- wave-wide helpers shared by the candidate kernels (64 lanes).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace sc {

__device__ inline uint32_t uni(uint32_t v) { return uint32_t(__builtin_amdgcn_readfirstlane(int(v))); }

// Wave-wide reductions (every lane active): four DPP steps combine the 16
// lanes of each row (quad swaps, half-row and row mirrors), four reads of
// lanes 0/16/32/48 combine the rows.
template <class Op> __device__ inline uint32_t wave_reduce(uint32_t v, Op op) {
    v = op(v, uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0xB1, 0xF, 0xF, false))); // quad_perm 1,0,3,2
    v = op(v, uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x4E, 0xF, 0xF, false))); // quad_perm 2,3,0,1
    v = op(v, uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x141, 0xF, 0xF, false))); // row_half_mirror
    v = op(v, uint32_t(__builtin_amdgcn_update_dpp(0, int(v), 0x140, 0xF, 0xF, false))); // row_mirror
    const uint32_t a = uint32_t(__builtin_amdgcn_readlane(int(v), 0)), b = uint32_t(__builtin_amdgcn_readlane(int(v), 16));
    const uint32_t c = uint32_t(__builtin_amdgcn_readlane(int(v), 32)), d = uint32_t(__builtin_amdgcn_readlane(int(v), 48));
    return op(op(a, b), op(c, d));
}
__device__ inline uint32_t wave_or32(uint32_t v) {
    return wave_reduce(v, [](uint32_t x, uint32_t y) { return x | y; });
}
// min / max of floats through an order-preserving integer key (NaN excluded:
// callers handle NaN before)
__device__ inline int fkey(float f) {
    const int b = __float_as_int(f);
    return b ^ ((b >> 31) & 0x7fffffff);
}
__device__ inline float funkey(int k) { return __int_as_float(k ^ ((k >> 31) & 0x7fffffff)); }
__device__ inline float wave_min(float v) {
    auto f = [](uint32_t x, uint32_t y) { return uint32_t(min(int(x), int(y))); };
    return funkey(int(wave_reduce(uint32_t(fkey(v)), f)));
}
__device__ inline float wave_max(float v) {
    auto f = [](uint32_t x, uint32_t y) { return uint32_t(max(int(x), int(y))); };
    return funkey(int(wave_reduce(uint32_t(fkey(v)), f)));
}

} // namespace sc
