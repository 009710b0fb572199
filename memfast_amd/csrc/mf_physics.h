// Physical conductance levels and noise factors shared by the gfx950 kernels.
//
// Arithmetic order and FP32 rounding of constants follow the CPU reference
// memfast/reference.py:10-51 (restored) so that ideal and noisy levels match it.
#pragma once

#include "mf_device.h"

namespace mf {

template <typename Phys>
__device__ __forceinline__ Phys nominal_level(const mf_config &cfg, int digit, int mask);

template <>
__device__ __forceinline__ float nominal_level<float>(const mf_config &cfg, int digit, int mask) {
    if (mask == 1) return digit ? cfg.f_high : cfg.f_low;
    return cfg.f_low + cfg.f_span * (float(digit) / float(mask));
}

template <>
__device__ __forceinline__ double nominal_level<double>(const mf_config &cfg, int digit,
                                                        int mask) {
    if (mask == 1) return digit ? cfg.d_high : cfg.d_low;
    return cfg.d_low + cfg.d_span * (double(digit) / double(mask));
}

template <typename Phys>
__device__ __forceinline__ Phys drift_of(const mf_config &cfg);
template <>
__device__ __forceinline__ float drift_of<float>(const mf_config &cfg) { return cfg.f_drift; }
template <>
__device__ __forceinline__ double drift_of<double>(const mf_config &cfg) { return cfg.d_drift; }

template <typename Phys>
__device__ __forceinline__ Phys low_of(const mf_config &cfg);
template <>
__device__ __forceinline__ float low_of<float>(const mf_config &cfg) { return cfg.f_low; }
template <>
__device__ __forceinline__ double low_of<double>(const mf_config &cfg) { return cfg.d_low; }

template <typename Phys>
__device__ __forceinline__ Phys high_of(const mf_config &cfg);
template <>
__device__ __forceinline__ float high_of<float>(const mf_config &cfg) { return cfg.f_high; }
template <>
__device__ __forceinline__ double high_of<double>(const mf_config &cfg) { return cfg.d_high; }

// exp(sigma * n) for a noise sample n at `address`.  FP64 currents resolve conductance
// differences far below one FP32 ulp of g (high - low down to 1e-4 of high), and one ulp of an
// FP32 factor near 1 is 2^-23 of g, so they sample with OCML's logf/cosf/sqrtf/expf, which stay
// within an ulp or two of torch CPU's; FP32 currents use the hardware approximations
// (normal_fast, exp_small).
template <typename Phys>
__device__ __forceinline__ float noise_factor(const mf_config &cfg, float sigma, u64 address,
                                              u64 seed, u32 stream) {
    if constexpr (sizeof(Phys) == sizeof(double))
        return expf(sigma * normal(address, seed, stream, cfg.f_two_pi));
    else
        return exp_small(sigma * normal_fast(address, seed, stream));
}

// Programmed + (shared) read conductance of one cell.
template <typename Phys>
__device__ __forceinline__ Phys cell_conductance(const mf_config &cfg, u32 code, int w, u64 cell,
                                                 u32 seed, u64 read_seed) {
    const int mask = cfg.w_mask[w];
    const int digit = int((code >> cfg.w_shift[w]) & u32(mask));
    Phys raw = nominal_level<Phys>(cfg, digit, mask);
    if (cfg.has_write) raw = raw * Phys(noise_factor<Phys>(cfg, cfg.f_write, cell, seed, 10u));
    raw = raw * drift_of<Phys>(cfg);
    if (cfg.has_saf) {
        const float u = uniform(cell, seed, 30u);
        if (u < cfg.f_saf_low) raw = low_of<Phys>(cfg);
        else if (u < cfg.f_saf_band) raw = high_of<Phys>(cfg);
    }
    if (cfg.read_mode == MF_READ_SHARED && cfg.has_read)
        raw = raw * Phys(noise_factor<Phys>(cfg, cfg.f_read, cell, read_seed, 20u));
    return raw;
}

// cell_conductance<float> at cells below 2^32 (LowNormal): the same samples.
struct LowCells {
    LowNormal write, read;
    u32 fault_fold;
    __device__ __forceinline__ LowCells(u32 seed, u64 read_seed)
        : write(seed, 10u), read(read_seed, 20u), fault_fold(uniform_fold(0u, seed, 30u)) {}
    __device__ __forceinline__ float operator()(const mf_config &cfg, u32 code, int w,
                                                u32 cell) const {
        const int mask = cfg.w_mask[w];
        const int digit = int((code >> cfg.w_shift[w]) & u32(mask));
        float raw = nominal_level<float>(cfg, digit, mask);
        if (cfg.has_write) raw = raw * exp_small(cfg.f_write * write(cell));
        raw = raw * cfg.f_drift;
        if (cfg.has_saf) {
            const float u = uniform_finish(cell, fault_fold);
            if (u < cfg.f_saf_low) raw = cfg.f_low;
            else if (u < cfg.f_saf_band) raw = cfg.f_high;
        }
        if (cfg.read_mode == MF_READ_SHARED && cfg.has_read)
            raw = raw * exp_small(cfg.f_read * read(cell));
        return raw;
    }
};

// Conductances of eight cells of one column, `stride` apart.  `low`: wave-uniform, every
// address is below 2^32 (a matrix of up to 4.3e9 cells and slices).
__device__ __forceinline__ void cell_column(const mf_config &cfg, const u32 (&codes)[8], int w,
                                            u64 cell, int stride, u32 seed, u64 read_seed, bool low,
                                            float (&level)[8]) {
    if (low) {
        const LowCells cells(seed, read_seed);
#pragma unroll
        for (int j = 0; j < 8; ++j) level[j] = cells(cfg, codes[j], w, u32(cell) + u32(j * stride));
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
            level[j] = cell_conductance<float>(cfg, codes[j], w, cell + u64(j) * stride, seed,
                                               read_seed);
    }
}

// One fp16 pair (hi, lo) of x, added to packed operands as element j of eight.
__device__ __forceinline__ void put_terms(float x, int j, u32 (&hi4)[4], u32 (&lo4)[4]) {
    const _Float16 hi = static_cast<_Float16>(x);   // round to nearest even
    const _Float16 lo = static_cast<_Float16>(x - static_cast<float>(hi));
    const int shift = 16 * (j & 1);
    hi4[j >> 1] |= u32(__builtin_bit_cast(unsigned short, hi)) << shift;
    lo4[j >> 1] |= u32(__builtin_bit_cast(unsigned short, lo)) << shift;
}

}  // namespace mf
