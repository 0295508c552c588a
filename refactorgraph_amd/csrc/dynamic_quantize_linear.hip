// DynamicQuantizeLinear for gfx950: float tensor -> uint8 tensor + scale + zero point.
//
// Arithmetic contract: src/04kernel/src/kernels/dynamic_quantize_linear/cpu_kernel.cc:25-70 of
// the reference, operation by operation in float:
//   (min, max) over x, started from (FLT_MAX, FLT_MIN);
//   len = max(0, max) - min(0, min);  scale = len / 255;
//   zp = saturate(0 - min * 255 / len);  y = saturate(round(x / scale) + zp);
//   saturate(v) = (uint8) round(clamp(v, 0, 255)), round = half away from zero.
// Divisions are the correctly rounded ones and denormals are kept, so the results are
// bit-identical to the CPU kernel's (an all-zero input gives scale FLT_MIN / 255, zp 0, y 0).
//
// Two launches, HBM-bound (5 bytes per element; the second read of x comes from the memory-side
// cache for tensors that fit it): per-workgroup (min, max) partials into the workspace, then every
// workgroup of the second launch reduces those partials itself — no atomics, nothing to clear, the
// result does not depend on timing.  Both launches keep up to eight 128-bit loads per thread in flight;
// the second replaces the division by a multiplication wherever that provably gives the same
// integer (see Quantiser::pack).
#include <cfloat>

#include "common.hpp"

namespace rg {
namespace {

constexpr uint32_t kMaxPartials = 1024;  // workgroups of the first launch
constexpr int kUnroll = 8;               // 128-bit loads a thread has in flight on large tensors
typedef float f32x4 __attribute__((ext_vector_type(4)));

struct OpMin {
    __device__ __forceinline__ float operator()(float a, float b) const { return b < a ? b : a; }
};
struct OpMax2 {
    __device__ __forceinline__ float operator()(float a, float b) const { return a < b ? b : a; }
};

__device__ __forceinline__ float block_min(float v, float *smem) {
    return block_allreduce<4>(v, smem, [](float w) { return wave_allreduce(w, OpMin{}); }, OpMin{});
}
__device__ __forceinline__ float block_max(float v, float *smem) {
    return block_allreduce<4>(v, smem, [](float w) { return wave_allreduce(w, OpMax2{}); }, OpMax2{});
}

__device__ __forceinline__ uint32_t saturate_u8(float v) {
    v = v < 0.f ? 0.f : v;
    v = 255.f < v ? 255.f : v;
    return static_cast<uint32_t>(roundf(v));
}

// scale and zero point from the extrema, and the quantisation of elements
struct Quantiser {
    float scale, zp_f, inv_scale;
    bool degenerate;
    __device__ __forceinline__ Quantiser(float mn, float mx) {
        const float len = (0.f < mx ? mx : 0.f) - (mn < 0.f ? mn : 0.f);
        scale = len / 255.f;
        degenerate = !(len > 0.f);
        zp_f = degenerate ? 0.f : static_cast<float>(saturate_u8(0.f - mn * 255.f / len));
        inv_scale = 1.f / scale;
    }
    // round(x / scale) + zp is integer-valued (or infinite), so is its clamp to [0, 255]: the second
    // rounding of the reference's saturate() changes nothing and is left out
    __device__ __forceinline__ uint32_t operator()(float v) const {
        float t = roundf(v / scale) + zp_f;
        t = t < 0.f ? 0.f : t;
        t = 255.f < t ? 255.f : t;
        return degenerate ? 0u : static_cast<uint32_t>(t);
    }
    // Four elements into one word.  The division is replaced by a multiplication where that provably
    // cannot change the result: q' = v * (1 / scale), two roundings, lies within |q'| 2^-22 of the
    // correctly rounded quotient q; if no half-integer lies within twice that distance of q', both
    // round to the same integer whichever way ties go, and that integer is the one nearest to q'.
    // Otherwise (also for NaN, infinities and a scale whose reciprocal overflows) the four elements
    // are quantised with the division.
    __device__ __forceinline__ uint32_t pack(f32x4 v) const {
        uint32_t w = 0;
        bool sure = true;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float q = v[e] * inv_scale;
            const float r = __builtin_rintf(q);
            sure = sure && __builtin_fabsf(__builtin_fabsf(q - r) - 0.5f) > __builtin_fabsf(q) * 0x1p-21f;
            float t = r + zp_f;
            t = t < 0.f ? 0.f : t;
            t = 255.f < t ? 255.f : t;
            w |= static_cast<uint32_t>(t) << (8 * e);
        }
        if (!sure || degenerate)
            w = (*this)(v[0]) | ((*this)(v[1]) << 8) | ((*this)(v[2]) << 16) | ((*this)(v[3]) << 24);
        return w;
    }
};

// (min, max) of a share of x per workgroup; vec: x is 16-byte aligned.  U: vectors per thread and step.
template <int U>
__global__ __launch_bounds__(256) void dql_minmax(float *__restrict__ partials, const float *__restrict__ x,
                                                  uint64_t n, int vec) {
    float mn = FLT_MAX, mx = FLT_MIN;
    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * 256;
    const uint64_t t = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (vec) {
        // (ordinary loads: the second launch should find x in the memory-side cache)
        const uint64_t n4 = n / 4;
        const f32x4 *x4 = reinterpret_cast<const f32x4 *>(x);
        for (uint64_t base = blockIdx.x * (256 * U); base < n4; base += gridDim.x * (256 * U)) {
            f32x4 v[U];
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const uint64_t i = base + j * 256 + threadIdx.x;
                v[j] = i < n4 ? x4[i] : f32x4{FLT_MAX, FLT_MAX, FLT_MAX, FLT_MAX};
            }
#pragma unroll
            for (int j = 0; j < U; ++j) {
                if (base + j * 256 + threadIdx.x < n4) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        mn = v[j][e] < mn ? v[j][e] : mn;
                        mx = mx < v[j][e] ? v[j][e] : mx;
                    }
                }
            }
        }
        for (uint64_t i = n4 * 4 + t; i < n; i += stride) {
            mn = x[i] < mn ? x[i] : mn;
            mx = mx < x[i] ? x[i] : mx;
        }
    } else {
        for (uint64_t i = t; i < n; i += stride) {
            mn = x[i] < mn ? x[i] : mn;
            mx = mx < x[i] ? x[i] : mx;
        }
    }
    __shared__ float scratch[8];
    mn = block_min(mn, scratch);
    mx = block_max(mx, scratch + 4);
    if (threadIdx.x == 0) {
        partials[2 * blockIdx.x] = mn;
        partials[2 * blockIdx.x + 1] = mx;
    }
}

template <int U>
__global__ __launch_bounds__(256) void dql_quantize(uint8_t *__restrict__ y, float *__restrict__ scale_out,
                                                    uint8_t *__restrict__ zp_out, const float *__restrict__ x,
                                                    const float *__restrict__ partials, uint32_t n_partials,
                                                    uint64_t n, int vec) {
    // the first step's vectors are requested ahead of the reduction of the extrema
    const uint64_t n4 = vec ? n / 4 : 0;
    const f32x4 *x4 = reinterpret_cast<const f32x4 *>(x);
    f32x4 v[U];
    auto fetch = [&](uint64_t base) {
#pragma unroll
        for (int j = 0; j < U; ++j) {
            const uint64_t i = base + j * 256 + threadIdx.x;
            if (i < n4) v[j] = __builtin_nontemporal_load(x4 + i);
        }
    };
    uint64_t base = static_cast<uint64_t>(blockIdx.x) * (256 * U);
    fetch(base);
    float mn = FLT_MAX, mx = FLT_MIN;
    for (uint32_t i = threadIdx.x; i < n_partials; i += 256) {
        const float a = partials[2 * i], b = partials[2 * i + 1];
        mn = a < mn ? a : mn;
        mx = mx < b ? b : mx;
    }
    __shared__ float scratch[8];
    mn = block_min(mn, scratch);
    mx = block_max(mx, scratch + 4);

    const Quantiser quant(mn, mx);
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        *scale_out = quant.scale;
        *zp_out = static_cast<uint8_t>(quant.zp_f);
    }

    const uint64_t stride = static_cast<uint64_t>(gridDim.x) * 256;
    const uint64_t t = static_cast<uint64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (vec) {
        uint32_t *y4 = reinterpret_cast<uint32_t *>(y);
        while (base < n4) {
            uint32_t w[U];
#pragma unroll
            for (int j = 0; j < U; ++j) {
                if (base + j * 256 + threadIdx.x < n4) w[j] = quant.pack(v[j]);
            }
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const uint64_t i = base + j * 256 + threadIdx.x;
                if (i < n4) {
                    if constexpr (U < kUnroll) y4[i] = w[j];  // (small: the product that follows finds it in L2)
                    else __builtin_nontemporal_store(w[j], y4 + i);
                }
            }
            base += static_cast<uint64_t>(gridDim.x) * (256 * U);
            if (base < n4) fetch(base);
        }
        for (uint64_t i = n4 * 4 + t; i < n; i += stride) y[i] = static_cast<uint8_t>(quant(x[i]));
    } else {
        for (uint64_t i = t; i < n; i += stride) y[i] = static_cast<uint8_t>(quant(x[i]));
    }
}

// Vectors per thread: one while that gives no more workgroups than CUs, so that few elements still occupy the chip
// ([32, 4096]: 16 workgroups of eight vectors a thread 3.5 + 6.0 us, 128 workgroups of one 2.8 + 3.7 us; [1000, 4096]: the same 5.3 + 7.0 us
// with eight and with four).
inline int vectors_per_thread(uint64_t n) { return n <= (1u << 18) ? 1 : n <= (1u << 19) ? 2 : n <= (1u << 22) ? 4 : kUnroll; }

inline uint64_t workgroups(uint64_t n, int u, uint64_t most) {
    const uint64_t wgs = (n + 1024 * u - 1) / (1024 * u);
    return wgs > most ? most : wgs == 0 ? 1 : wgs;
}

int launch_quantize(uint8_t *y, float *scale, uint8_t *zero_point, const float *x, const float *partials, uint32_t n_partials, uint64_t n,
                    int vec, hipStream_t s) {
    const int u = vectors_per_thread(n);
    const unsigned grid = static_cast<unsigned>(workgroups(n, u, 8192));
    if (u == 1) dql_quantize<1><<<grid, 256, 0, s>>>(y, scale, zero_point, x, partials, n_partials, n, vec);
    else if (u == 2) dql_quantize<2><<<grid, 256, 0, s>>>(y, scale, zero_point, x, partials, n_partials, n, vec);
    else if (u == 4) dql_quantize<4><<<grid, 256, 0, s>>>(y, scale, zero_point, x, partials, n_partials, n, vec);
    else dql_quantize<kUnroll><<<grid, 256, 0, s>>>(y, scale, zero_point, x, partials, n_partials, n, vec);
    return launch_status();
}

}  // namespace

// The quantising launch on extrema that another kernel has left (RmsNormalization with its output's least and
// greatest value per workgroup): x is read once here.
int quantize_with_partials(uint8_t *y, float *scale, uint8_t *zero_point, const float *x, size_t size, const float *partials,
                           size_t n_partials, hipStream_t s) {
    const int vec = aligned16(x) && (reinterpret_cast<uintptr_t>(y) & 3u) == 0;
    return launch_quantize(y, scale, zero_point, x, partials, static_cast<uint32_t>(n_partials), size, vec, s);
}

}  // namespace rg

extern "C" size_t rg_hip_dynamic_quantize_linear_workspace(size_t) {
    return static_cast<size_t>(rg::kMaxPartials) * 2 * sizeof(float);
}

extern "C" int rg_hip_dynamic_quantize_linear(uint8_t *y, float *scale, uint8_t *zero_point, const float *x,
                                              size_t size, void *workspace, size_t workspace_bytes,
                                              void *stream) {
    using namespace rg;
    if (!y || !scale || !zero_point || !x) return RG_HIP_E_ARGUMENT;
    if (size == 0) return RG_HIP_E_ARGUMENT;
    if (!workspace || workspace_bytes < rg_hip_dynamic_quantize_linear_workspace(size)) return RG_HIP_E_WORKSPACE;
    if (reinterpret_cast<uintptr_t>(workspace) % alignof(float) != 0) return RG_HIP_E_ARGUMENT;
    hipStream_t s = as_stream(stream);
    const int vec = aligned16(x) && (reinterpret_cast<uintptr_t>(y) & 3u) == 0;
    const int u = vectors_per_thread(size);
    const uint32_t wgs = static_cast<uint32_t>(workgroups(size, u, kMaxPartials));
    float *partials = static_cast<float *>(workspace);
    if (u == 1) dql_minmax<1><<<wgs, 256, 0, s>>>(partials, x, size, vec);
    else if (u == 2) dql_minmax<2><<<wgs, 256, 0, s>>>(partials, x, size, vec);
    else if (u == 4) dql_minmax<4><<<wgs, 256, 0, s>>>(partials, x, size, vec);
    else dql_minmax<kUnroll><<<wgs, 256, 0, s>>>(partials, x, size, vec);
    const int rc = launch_status();
    if (rc) return rc;
    return launch_quantize(y, scale, zero_point, x, partials, wgs, size, vec, s);
}
