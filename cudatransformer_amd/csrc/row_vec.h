// Row-wise kernels' building blocks (gfx950, wave64): 16-byte granules of a row, sums over the
// lanes of a row that spans one or several waves, division by a run-time invariant.
#pragma once

#include "attn_common.h"

#include <type_traits>

namespace ctattn {

// A granule: the EPC elements c0 .. c0 + EPC - 1 of a row, one element-aligned 16-byte access (the
// hardware takes any element alignment; rows of an odd length start anywhere), or element by
// element where it crosses the end of the row.
typedef uint32_t gran_raw __attribute__((ext_vector_type(4)));
typedef gran_raw gran_u2 __attribute__((aligned(2)));
typedef gran_raw gran_u4 __attribute__((aligned(4)));

template <typename T> struct Gran {
    static_assert(sizeof(T) == 2 || sizeof(T) == 4, "fp32 and 16-bit storage");
    using raw_t = std::conditional_t<sizeof(T) == 2, gran_u2, gran_u4>;
    static constexpr int EPC = 16 / int(sizeof(T));

    // Elements at or past D are `fill`; c0 >= D reads nothing.
    __device__ static __forceinline__ gran_raw load(const T *row, int c0, int D, float fill = 0.f) {
        if (c0 + EPC <= D) return *reinterpret_cast<const raw_t *>(row + c0);
        gran_raw x = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < EPC; ++e) {
            const T v = c0 + e < D ? row[c0 + e] : from_f32<T>(fill);
            if constexpr (sizeof(T) == 2) x[e / 2] |= uint32_t(v.bits) << (16 * (e & 1));
            else x[e] = __float_as_uint(to_f32(v));
        }
        return x;
    }
    // The same; the granule that crosses the end is read as the row's last EPC elements and shifted
    // down past those before c0: one access beside the others', where element by element takes a
    // chain of them.  For rows of many granules and mostly odd lengths (in the LayerNorm backward the
    // shift costs 40 registers).
    __device__ static __forceinline__ gran_raw load_tail(const T *row, int c0, int D, float fill) {
        if (D < EPC) return load(row, c0, D, fill);
        uint32_t pat;  // one dword of fill
        if constexpr (sizeof(T) == 2) pat = uint32_t(from_f32<T>(fill).bits) * 0x10001u;
        else pat = __float_as_uint(fill);
        if (c0 >= D) return gran_raw{pat, pat, pat, pat};
        const gran_raw x = *reinterpret_cast<const raw_t *>(row + min(c0, D - EPC));
        if (c0 + EPC <= D) return x;
        const int bits = 8 * int(sizeof(T)) * (c0 + EPC - D);  // one element .. 128 less one
        const uint64_t f = uint64_t(pat) << 32 | pat;
        uint64_t lo = uint64_t(x[1]) << 32 | x[0], hi = uint64_t(x[3]) << 32 | x[2];
        if (bits >= 64) {
            lo = hi;
            hi = f;
        }
        if (const int n = bits & 63) {
            lo = lo >> n | hi << (64 - n);
            hi = hi >> n | f << (64 - n);
        }
        return gran_raw{uint32_t(lo), uint32_t(lo >> 32), uint32_t(hi), uint32_t(hi >> 32)};
    }
    __device__ static __forceinline__ float get(gran_raw x, int e) {
        if constexpr (sizeof(T) == 2) return to_f32(T{uint16_t(x[e / 2] >> (16 * (e & 1)))});
        else return __uint_as_float(x[e]);
    }
    // v[e] rounded to T as computed (fp16: kept from merging with the operation before it, as in
    // the scalar stores).
    __device__ static __forceinline__ void store(T *row, int c0, int D, const float (&v)[EPC]) {
        if (c0 >= D) return;
        gran_raw x = {0, 0, 0, 0};
#pragma unroll
        for (int e = 0; e < EPC; ++e) {
            if constexpr (std::is_same_v<T, bf16_t>) {
                if (e % 2 == 0) x[e / 2] = f32_to_bf16x2(v[e], v[e + 1]);
            } else if constexpr (sizeof(T) == 2) {
                float f = v[e];
                asm volatile("" : "+v"(f));
                x[e / 2] |= uint32_t(from_f32<T>(f).bits) << (16 * (e & 1));
            } else {
                x[e] = __float_as_uint(v[e]);
            }
        }
        if (c0 + EPC <= D) {
            *reinterpret_cast<raw_t *>(row + c0) = x;
            return;
        }
#pragma unroll
        for (int e = 0; e < EPC - 1; ++e)
            if (c0 + e < D) {
                if constexpr (sizeof(T) == 2) row[c0 + e] = T{uint16_t(x[e / 2] >> (16 * (e & 1)))};
                else row[c0 + e] = __uint_as_float(x[e]);
            }
    }
};

// x of the lane that DPP control CTRL names.
template <int CTRL> __device__ __forceinline__ float dpp(float x) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), CTRL, 0xf, 0xf, true));
}
// Sum (max) over the wave in every lane, in registers (the shuffles of wave_sum go through LDS):
// pairs and quads by quad_perm, 8 and 16 lanes by half_mirror and mirror, then the rows of 16 and
// the halves of 32 by permlane swaps.
__device__ __forceinline__ float wave_sum_dpp(float x) {
    x += dpp<0xB1>(x);
    x += dpp<0x4E>(x);
    x += dpp<0x141>(x);
    x += dpp<0x140>(x);
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(r[0]) + __uint_as_float(r[1]);
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float wave_max_dpp(float x) {
    x = fmaxf(x, dpp<0xB1>(x));
    x = fmaxf(x, dpp<0x4E>(x));
    x = fmaxf(x, dpp<0x141>(x));
    x = fmaxf(x, dpp<0x140>(x));
    auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
    r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

// Sum (max) over a row's GW waves (the whole workgroup when GW > 1), through buf[GW].  Each
// reduction of a kernel takes a buf of its own, so one barrier each is enough.
template <int GW> __device__ __forceinline__ float row_sum(float x, float *buf) {
    x = wave_sum_dpp(x);
    if constexpr (GW > 1) {
        if ((threadIdx.x & (kWave - 1)) == 0) buf[threadIdx.x / kWave] = x;
        __syncthreads();
        x = buf[0];
#pragma unroll
        for (int w = 1; w < GW; ++w) x += buf[w];
    }
    return x;
}
template <int GW> __device__ __forceinline__ float row_max(float x, float *buf) {
    x = wave_max_dpp(x);
    if constexpr (GW > 1) {
        if ((threadIdx.x & (kWave - 1)) == 0) buf[threadIdx.x / kWave] = x;
        __syncthreads();
        x = buf[0];
#pragma unroll
        for (int w = 1; w < GW; ++w) x = fmaxf(x, buf[w]);
    }
    return x;
}

// Division by a run-time divisor D >= 1 of indices 0 <= i < 2^31 as a multiply and a shift
// (Granlund & Montgomery, "Division by invariant integers using multiplication", 1994, the
// unsigned case): with l = ceil(log2 D) and m = floor(2^32 (2^l - D) / D) + 1,
// i / D = (mulhi(i, m) + i) >> l exactly for every 32-bit i; mulhi(i, m) < i keeps the sum
// below 2^32 for i < 2^31.
struct FastDiv {
    uint32_t mul, shift;
};
inline FastDiv make_fastdiv(uint32_t D) {
    if (D == 0) return FastDiv{0, 0};  // no index to divide (an empty view)
    uint32_t l = 0;
    while (l < 32 && (uint64_t(1) << l) < D) ++l;
    const uint64_t m = ((uint64_t(1) << 32) * ((uint64_t(1) << l) - D)) / D + 1;
    return FastDiv{uint32_t(m), l};
}
__device__ __forceinline__ int fastdiv(int i, FastDiv f) {
    return int((__umulhi(uint32_t(i), f.mul) + uint32_t(i)) >> f.shift);
}

}  // namespace ctattn
