// Linear layers with a handful of outputs (the decoders' output layer, 64 -> 6 or 7 channels over
// every final voxel): 16-bit x and weights of one dtype, Ci = 32, 64, 128, 256 or 512, Co <= 16.
//
// Bound by memory: x is read once and out written once (64 -> 7, f32 out: 5.7 FLOP/B). A wave takes 64 rows a
// step as four 16-row operands of v_mfma_f32_16x16x32 (lane l holds row l % 16, 8 channels from
// 8 (l / 16): 16-byte loads, whole 64-byte row segments across 4 lanes), the weights, padded to 16
// columns, in registers for the launch. The 64 x Co results go through LDS to one contiguous piece
// of out. 1.2 M rows, f16, 64 -> 7, f32 out: 37 us, 5.1 TB/s (the 64 x 64 tiles of the VALU kernel, 57 of
// 64 columns padding, took 235 us).
#include <algorithm>

#include "conv_internal.hpp"

namespace tsp {
namespace {

constexpr int LT_NT = 256, LT_ROWS = 64;     // threads of a workgroup, rows of a wave's step

template <bool BF16>
__device__ __forceinline__ f32x4_t mfma16x16x32(const u32x4_t& a, const u32x4_t& b, const f32x4_t& c) {
    if constexpr (BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                       0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0,
                                                      0, 0);
}

// KS steps of 32 channels
template <bool BF16, int KS, int ODT>
__global__ __launch_bounds__(LT_NT) void k_linear_thin(const uint16_t* __restrict__ x, int64_t n,
                                                       const uint16_t* __restrict__ w, const float* __restrict__ bias,
                                                       int co, void* __restrict__ out) {
    __shared__ __attribute__((aligned(16))) float sO[LT_NT / 64][LT_ROWS * 16];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
    constexpr int CI = 32 * KS;
    u32x4_t wb[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s)
        wb[s] = r < co ? *reinterpret_cast<const u32x4_t*>(w + (int64_t)r * CI + 32 * s + 8 * g) : u32x4_t{0, 0, 0, 0};
    const float bv = bias && r < co ? bias[r] : 0.f;
    float* o = sO[wave];
    const int64_t step = (int64_t)gridDim.x * (LT_NT / 64) * LT_ROWS;
    for (int64_t r0 = ((int64_t)blockIdx.x * (LT_NT / 64) + wave) * LT_ROWS; r0 < n; r0 += step) {
        const int rows = (int)min<int64_t>(LT_ROWS, n - r0);
        f32x4_t acc[4];
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const int64_t i = min<int64_t>(r0 + 16 * b + r, n - 1);   // (rows past n: the last one, not stored)
            u32x4_t a[KS];
#pragma unroll
            for (int s = 0; s < KS; ++s) a[s] = *reinterpret_cast<const u32x4_t*>(x + i * CI + 32 * s + 8 * g);
            acc[b] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < KS; ++s) acc[b] = mfma16x16x32<BF16>(a[s], wb[s], acc[b]);
        }
        // element j of block b is row 16 b + 4 g + j, column r: to LDS as the rows lie in out
        if (r < co) {
#pragma unroll
            for (int b = 0; b < 4; ++b)
#pragma unroll
                for (int j = 0; j < 4; ++j) o[(16 * b + 4 * g + j) * co + r] = acc[b][j] + bv;
        }
        // (one wave's own LDS: its writes are done before its reads, in order)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
        const int total = rows * co;
        if constexpr (ODT == TSP_F32) {
            float* dst = static_cast<float*>(out) + r0 * co;
            if (rows == LT_ROWS && (reinterpret_cast<uintptr_t>(dst) & 15) == 0) {
                for (int e = lane; e < LT_ROWS * co / 4; e += 64)
                    *reinterpret_cast<f32x4_t*>(dst + 4 * e) = *reinterpret_cast<const f32x4_t*>(o + 4 * e);
            } else {
                for (int e = lane; e < total; e += 64) dst[e] = o[e];
            }
        } else {
            for (int e = lane; e < total; e += 64) store_out<ODT>(out, r0 * co + e, o[e]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    }
}

}  // namespace

int linear_thin_launch(int xdt, int wdt, int odt, const void* x, int64_t n, int ci, const void* w, const float* bias,
                       int co, void* out, hipStream_t s) {
    if (xdt == TSP_F32 || xdt != wdt || (odt != TSP_F32 && odt != xdt)) return TSP_ERR_UNSUPPORTED;
    if (co > 16 || !(ci == 32 || ci == 64 || ci == 128 || ci == 256 || ci == 512)) return TSP_ERR_UNSUPPORTED;
    if (reinterpret_cast<uintptr_t>(x) % 16 || reinterpret_cast<uintptr_t>(w) % 16) return TSP_ERR_UNSUPPORTED;
    // eight workgroups a CU, as many as hide the loads' latency
    const dim3 grid((unsigned)std::min<int64_t>(ceil_div(n, (LT_NT / 64) * LT_ROWS), 2048)), block(LT_NT);
    auto go = [&](auto bf_c, auto ks_c) {
        constexpr bool B = decltype(bf_c)::value;
        constexpr int KS = decltype(ks_c)::value;
        const auto* xx = static_cast<const uint16_t*>(x);
        const auto* ww = static_cast<const uint16_t*>(w);
        if (odt == TSP_F32)
            hipLaunchKernelGGL((k_linear_thin<B, KS, TSP_F32>), grid, block, 0, s, xx, n, ww, bias, co, out);
        else
            hipLaunchKernelGGL((k_linear_thin<B, KS, B ? TSP_BF16 : TSP_F16>), grid, block, 0, s, xx, n, ww, bias, co, out);
    };
    auto width = [&](auto bf_c) {
        using std::integral_constant;
        switch (ci) {
            case 32: go(bf_c, integral_constant<int, 1>{}); break;
            case 64: go(bf_c, integral_constant<int, 2>{}); break;
            case 128: go(bf_c, integral_constant<int, 4>{}); break;
            case 256: go(bf_c, integral_constant<int, 8>{}); break;
            default: go(bf_c, integral_constant<int, 16>{}); break;
        }
    };
    if (xdt == TSP_BF16) width(std::true_type{});
    else width(std::false_type{});
    TSP_CHECK_LAUNCH();
    return TSP_OK;
}

}  // namespace tsp
