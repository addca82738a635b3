// Per-primitive residual parameters of the preprocess kernels: their count and the LDS staging of a wave's rows.
#pragma once

namespace efgs {

// floats per appearance unit (SH coefficient rgb, SV site, NASG lobe, NASGabor lobe) and per primitive
constexpr uint32_t params_per_unit = EFGS_MODEL == 1 ? 3u : EFGS_MODEL == 2 ? 7u : EFGS_MODEL == 3 ? 8u : EFGS_MODEL == 4 ? 9u : 1u;
constexpr uint32_t residual_params = EFGS_MODEL == 0 ? 0u : params_per_unit * EFGS_N_UNITS;

// A wave stages its 64 primitives' residual rows in its own part of the LDS, whole units per pass: a thread's own row
// is 45-72 floats apart from its neighbours', so direct per-thread reads touch 64 cache lines per load instruction and
// a wave's lines fall out of the L1 and the L2 between the loads that share them (400k SH3 primitives: 271 MB read
// for 94 MB of rows). SH takes its coefficients in one pass, SV and the lobe models up to MAX_UNITS units per pass:
// four lobes are 128 (144) bytes of a row, where passes of two lobes fetched every 128-byte line twice (NASG forward on
// 1M primitives: 488 MB for 312 MB). A WHOLE_ROW layout of more than 63 floats reads its rows directly.
// Preprocess times before and after (the block-wide staging, respectively direct reads, of single floats with index
// arithmetic per element): NASG on 1M at 1080p 120 -> 90 us forward, 181 -> 142 us backward; SH3 on 400k 66 -> 36 us
// forward; SV on 150k 31.0 -> 30.6 and 37.9 -> 35.0 us.
template <uint32_t MAX_UNITS, bool WHOLE_ROW>
struct RowStaging {
    static constexpr uint32_t pass_units = EFGS_MODEL == 1 ? EFGS_N_UNITS : (MAX_UNITS < EFGS_N_UNITS ? MAX_UNITS : EFGS_N_UNITS);
    static constexpr uint32_t pass_floats = pass_units * params_per_unit;
    static constexpr bool staged = EFGS_MODEL != 0 && EFGS_MODEL != 5 && EFGS_N_UNITS > 0 && pass_floats <= 63u &&
                                   (!WHOLE_ROW || pass_units == EFGS_N_UNITS);
    static constexpr uint32_t row_ld = pass_floats | 1u;  // odd: the lanes' rows start in different banks
    static constexpr uint32_t n_passes = pass_units > 0 ? (EFGS_N_UNITS + pass_units - 1) / pass_units : 0u;
    static constexpr uint32_t wave_floats = staged ? 64u * row_ld : 1u;
};
using ForwardRows = RowStaging<4u, false>;
using BackwardRows = RowStaging<EFGS_MODEL == 2 ? 9u : 4u, EFGS_MODEL == 2>;  // (the SV backward's softmax needs every site)

__device__ __forceinline__ void rows_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The rows in `mask` (bit r: primitive p0 + r; p0 and mask wave-uniform) from `residual` into s[r * ROW_LD + c], floats
// [f0, f0 + floats) of each (floats <= 64): one load instruction per row straight into the LDS (no registers, no
// per-element index arithmetic), all in flight together; returns when they have landed.
template <uint32_t ROW_LD>
__device__ __forceinline__ void stage_rows(const float* residual, uint32_t p0, uint64_t mask, uint32_t f0, uint32_t floats, float* s) {
    const uint32_t lane = threadIdx.x & 63u;
    const float* const base = residual + static_cast<size_t>(p0) * residual_params + f0;
    if (lane < floats) {
        for (uint64_t m = mask; m != 0; m &= m - 1) {
            const uint32_t r = static_cast<uint32_t>(__ffsll(static_cast<long long>(m)) - 1);
            __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(base + r * residual_params + lane),
                                             (__attribute__((address_space(3))) void*)(s + r * ROW_LD), 4, 0, 0);
        }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    rows_sync();
}

// the reverse of stage_rows for rows [0, rows): s[r * ROW_LD + c] to floats [f0, f0 + floats) of primitive p0 + r
template <uint32_t ROW_LD>
__device__ __forceinline__ void store_rows(const float* s, uint32_t p0, uint32_t rows, uint32_t f0, uint32_t floats, float* out) {
    const uint32_t lane = threadIdx.x & 63u;
    rows_sync();
    float* const base = out + static_cast<size_t>(p0) * residual_params + f0;
    if (lane < floats) {
#pragma unroll 8
        for (uint32_t r = 0; r < rows; r++) base[r * residual_params + lane] = s[r * ROW_LD + lane];
    }
}

}  // namespace efgs
