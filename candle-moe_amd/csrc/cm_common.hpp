// Shared device helpers for the gfx950 fused-MoE kernels: storage types,
// conversions, activations, wave64 cross-lane reductions and MFMA wrappers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace cm {

// dtype codes of the C ABI (/root/reference/src/lib.rs:174-182)
enum DType : int { kF16 = 0, kBF16 = 1, kF32 = 2 };
// activation codes (/root/reference/src/lib.rs:164-171)
enum Act : int { kSilu = 0, kGelu = 1, kRelu = 2 };
// moe_type codes (/root/reference/src/ffi.rs:42)
enum MoeType : int { kQwen3 = 0, kNomic = 1 };

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// 16-bit storage element tags. Global memory holds raw bits (uint16_t).
struct bf16_t { uint16_t v; };
struct f16_t { uint16_t v; };

__device__ __forceinline__ float bf16_bits_to_f32(uint32_t h) { return __uint_as_float(h << 16); }
__device__ __forceinline__ float f16_bits_to_f32(uint32_t h) {
    _Float16 x = __builtin_bit_cast(_Float16, (uint16_t)h);
    return (float)x;
}
// Round to nearest even (gfx950 lowers the bf16 truncation to v_cvt_pk_bf16_f32).
__device__ __forceinline__ uint32_t f32_to_bf16_bits(float f) {
    __bf16 b = (__bf16)f;
    return (uint32_t)__builtin_bit_cast(uint16_t, b);
}
__device__ __forceinline__ uint32_t f32_to_f16_bits(float f) {
    _Float16 h = (_Float16)f;
    return (uint32_t)__builtin_bit_cast(uint16_t, h);
}
// Two f32 values rounded to nearest even and packed, a in the low half: one
// v_cvt_pk_bf16_f32 / v_cvt_pk_f16_f32 for the pair.
template <int DT> __device__ __forceinline__ uint32_t pack2(float a, float b) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const f32x2 v = {a, b};
    if constexpr (DT == kBF16) {
        typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
    } else {
        typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
        return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2));
    }
}

// f32 values as three bf16 parts, 2^16 x = h + m + l (each rounded to nearest
// even, the differences exact), packed in pairs, a low. The parts hold all 24
// significand bits of every finite |x| < 2^111: the last bit of any f32,
// subnormal ones included, is a multiple of 2^-149, and 2^-133 is the smallest
// bf16 (the matrix cores keep subnormal inputs). Unscaled, values below 2^-110
// lost low bits (2.6e-4 of a sum over |x| = 1e-37); the multiply costs 2 % (Nomic
// T=64 / 4096 54.2 / 523 -> 55.2 / 536 us). A product of two split values comes
// out 1 / kSplitUnscale times too large. Non-finite values, and magnitudes whose scaled
// part rounds to a bf16 infinity, give non-finite parts.
constexpr float kSplitScale = 65536.0f, kSplitUnscale = 1.0f / (65536.0f * 65536.0f);
__device__ __forceinline__ void split2(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
    a *= kSplitScale;
    b *= kSplitScale;
    h = pack2<kBF16>(a, b);
    a -= __uint_as_float(h << 16);
    b -= __uint_as_float(h & 0xffff0000u);
    m = pack2<kBF16>(a, b);
    a -= __uint_as_float(m << 16);
    b -= __uint_as_float(m & 0xffff0000u);
    l = pack2<kBF16>(a, b);
}
__device__ __forceinline__ void split8(const float (&v)[8], u32x4& h, u32x4& m, u32x4& l) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        uint32_t x, y, z;
        split2(v[2 * q], v[2 * q + 1], x, y, z);
        h[q] = x;
        m[q] = y;
        l[q] = z;
    }
}

// Non-finite sums of a split-bf16 block (infinities, NaN and values or sums beyond
// the split's range) again with f32 FMAs over k0 .. k1 - 1 (multiples of 4). A wave
// holds R registers of sums; the lanes of a group of GL share the row of
// register q. get / set: this lane's sum q; a4(q, k): four operands of its row;
// b(k): its column's. A row with a NaN has NaN in all its sums already: its GL
// lanes look for one first, and a row of padding ends there (with all sums of the
// block recomputed, one NaN row made a call 7 to 15 times as long).
template <int R, int GL, class Get, class Set, class A4, class B>
__device__ __forceinline__ void redo_non_finite(int lane, int k0, int k1, Get get, Set set, A4 a4, B b) {
    const uint64_t group = (GL == 32 ? 0xffffffffull : 0xffffull) << (lane & (64 - GL));
#pragma unroll 1
    for (int q = 0; q < R; ++q) {
        const bool bad = !__builtin_isfinite(get(q));
        bool todo = bad, nan = false;
        for (int kb = k0; kb < k1 && __any(todo); kb += 4 * GL) {
            const int k = kb + 4 * (lane % GL);
            if (k < k1) {
                const f32x4 v = a4(q, k);
                nan = nan || v[0] != v[0] || v[1] != v[1] || v[2] != v[2] || v[3] != v[3];
            }
            todo = bad && (__builtin_amdgcn_ballot_w64(nan) & group) == 0ull;
        }
        float s = 0.f;
        int k = k0;
        // (NaN stays: a row of infinities ends at the first change of sign)
        for (; k + 16 <= k1 && __any(todo && s == s); k += 16) {
            f32x4 x[4];
            float w[16];
#pragma unroll
            for (int i = 0; i < 4; ++i) x[i] = a4(q, k + 4 * i);
#pragma unroll
            for (int i = 0; i < 16; ++i) w[i] = b(k + i);
#pragma unroll
            for (int i = 0; i < 16; ++i) s = fmaf(x[i / 4][i % 4], w[i], s);
        }
        for (; k < k1 && __any(todo && s == s); k += 4) {
            const f32x4 x = a4(q, k);
#pragma unroll
            for (int i = 0; i < 4; ++i) s = fmaf(x[i], b(k + i), s);
        }
        if (todo) set(q, s);
    }
}

template <int DT> struct Elem;
template <> struct Elem<kBF16> {
    typedef uint16_t storage;
    static __device__ __forceinline__ float to_f32(uint16_t v) { return bf16_bits_to_f32(v); }
    static __device__ __forceinline__ uint16_t from_f32(float f) { return (uint16_t)f32_to_bf16_bits(f); }
};
template <> struct Elem<kF16> {
    typedef uint16_t storage;
    static __device__ __forceinline__ float to_f32(uint16_t v) { return f16_bits_to_f32(v); }
    static __device__ __forceinline__ uint16_t from_f32(float f) { return (uint16_t)f32_to_f16_bits(f); }
};
template <> struct Elem<kF32> {
    typedef float storage;
    static __device__ __forceinline__ float to_f32(float v) { return v; }
    static __device__ __forceinline__ float from_f32(float f) { return f; }
};

// Activations (/root/reference/kernels/common.cuh:116-138): SiLU x/(1+e^-x),
// tanh-approximation GELU, ReLU. Evaluated in f32 with the accurate
// library expf / tanhf (the reference build used approximate __expf).
__device__ __forceinline__ float act_f32(float x, int act) {
    if (act == kGelu) {
        const float c = 0.7978845608028654f;  // sqrt(2/pi)
        return 0.5f * x * (1.0f + tanhf(c * (x + 0.044715f * x * x * x)));
    }
    if (act == kRelu) return fmaxf(x, 0.0f);
    return x / (1.0f + expf(-x));
}

// The same activations from the hardware base-2 exponential (v_exp_f32) and
// reciprocal (v_rcp_f32), a few f32 ulp from act_f32: used by the 16-bit
// MFMA epilogues, whose results are rounded to bf16 / f16 right after.
//   silu(x) = x * 1 / (1 + 2^(-x log2 e))
//   gelu(x) = x * 1 / (1 + 2^(-2 log2 e * sqrt(2/pi) (x + 0.044715 x^3)))
//             (0.5 (1 + tanh(u)) = 1 / (1 + e^(-2u)))
// For x -> -inf, 2^z overflows to +inf and v_rcp_f32(+inf) = 0, so the
// result goes to (-)0 as x / (1 + e^-x) does; x = -inf gives NaN in both.
template <int ACT> __device__ __forceinline__ float act_t(float x) {
    if constexpr (ACT == kRelu) {
        return fmaxf(x, 0.0f);
    } else {
        float z;
        if constexpr (ACT == kGelu) {
            const float k = -2.0f * 1.4426950408889634f * 0.7978845608028654f;
            z = k * (x + 0.044715f * x * x * x);
        } else {
            z = -1.4426950408889634f * x;
        }
        return x * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z));
    }
}
__device__ __forceinline__ float act_fast(float x, int act) {
    if (act == kRelu) return act_t<kRelu>(x);
    if (act == kGelu) return act_t<kGelu>(x);
    return act_t<kSilu>(x);
}
// f(std::integral_constant<int, ACT>{}) for the runtime activation code, so
// that a loop over elements inside f is compiled once per activation with no
// per-element branch.
template <class F> __device__ __forceinline__ void with_act(int act, F&& f) {
    if (act == kGelu) {
        f(std::integral_constant<int, kGelu>{});
    } else if (act == kRelu) {
        f(std::integral_constant<int, kRelu>{});
    } else {
        f(std::integral_constant<int, kSilu>{});
    }
}

// ---------------------------------------------------------------------
// wave64 cross-lane exchange: lane L receives the value of lane L ^ m.
// m = 1, 2 : DPP quad_perm; m = 4, 8, 16 : ds_swizzle bitmask mode
// (and 0x1f, xor m; no LDS memory traffic); m = 32 : ds_bpermute.
// ---------------------------------------------------------------------
template <int M>
__device__ __forceinline__ int xor_lane_i32(int v) {
    if constexpr (M == 1) {
        return __builtin_amdgcn_mov_dpp(v, 0xB1, 0xF, 0xF, false);  // quad_perm [1,0,3,2]
    } else if constexpr (M == 2) {
        return __builtin_amdgcn_mov_dpp(v, 0x4E, 0xF, 0xF, false);  // quad_perm [2,3,0,1]
    } else if constexpr (M == 4 || M == 8 || M == 16) {
        return __builtin_amdgcn_ds_swizzle(v, 0x1F | (M << 10));
    } else {
        const int lane = __lane_id();
        return __builtin_amdgcn_ds_bpermute((lane ^ M) << 2, v);
    }
}
template <int M>
__device__ __forceinline__ float xor_lane(float v) {
    return __int_as_float(xor_lane_i32<M>(__float_as_int(v)));
}
template <int M>
__device__ __forceinline__ double xor_lane(double v) {
    const uint64_t u = __double_as_longlong(v);
    const int lo = xor_lane_i32<M>((int)(uint32_t)u);
    const int hi = xor_lane_i32<M>((int)(uint32_t)(u >> 32));
    return __longlong_as_double(((uint64_t)(uint32_t)hi << 32) | (uint32_t)lo);
}

// ---------------------------------------------------------------------
// MFMA 32x32x16 (gfx950) for bf16 / f16 operands, f32 accumulate.
// Operand layout used throughout: lane l supplies 8 consecutive K values
// of row/column (l % 32), K-half (l / 32). Result lane l, register i holds
// element (row 8*(i/4) + 4*(l/32) + i%4, col l%32) of the 32x32 block.
// ---------------------------------------------------------------------
template <int DT>
__device__ __forceinline__ f32x16 mfma32(const u32x4& a, const u32x4& b, const f32x16& c) {
    if constexpr (DT == kBF16) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                      __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
    }
}

__host__ __device__ __forceinline__ int cdiv(int a, int b) { return (a + b - 1) / b; }

// Workgroup -> logical work item. The hardware hands workgroup w to XCD w % 8;
// this gives each XCD a contiguous range of the `live` items (neighbouring
// tiles then share that XCD's L2) and spreads the live items evenly over the
// 8 XCDs, however many spare workgroups a grid sized for the worst case holds.
// Returns -1 for a workgroup with no item.
__device__ __forceinline__ int xcd_logical(int live) {
    live = min(live, (int)gridDim.x);
    const int w = blockIdx.x, xcd = w & 7, idx = w >> 3;
    const int per = live >> 3, rem = live & 7;
    if (idx >= per + (xcd < rem ? 1 : 0)) return -1;
    return xcd * per + (xcd < rem ? xcd : rem) + idx;
}

// K splits of a launch with `live` output tiles (known on the device only,
// from the grouping): target / live, target = workgroups that fill the
// device once, so live * splits <= target (one round of workgroups: the
// weight-streaming 32-row kernels gain nothing from a second); at most
// max_split, no empty split among nk K tiles. target <= 0: max_split as
// given (fixed by the host).
__device__ __forceinline__ int adaptive_split(int max_split, int target, int live, int nk) {
    if (max_split <= 1) return 1;
    if (target <= 0) return max_split;
    int sp = live > 0 ? target / live : max_split;
    sp = sp < 1 ? 1 : (sp > max_split ? max_split : sp);
    sp = sp < nk ? sp : (nk > 0 ? nk : 1);
    const int per = (nk + sp - 1) / sp;
    return per > 0 ? (nk + per - 1) / per : 1;
}

// Output tile (row tile mt, column tile nt) of this workgroup, or false when
// it has none: the row-tile count m_live comes from the grouping on the device.
__device__ __forceinline__ bool tile_coords(int n_tiles, int m_live, int& mt, int& nt) {
    const int logical = xcd_logical(m_live * n_tiles);
    if (logical < 0) return false;
    mt = logical / n_tiles;
    nt = logical - mt * n_tiles;
    return true;
}
__host__ __device__ __forceinline__ long long cdivll(long long a, long long b) { return (a + b - 1) / b; }

}  // namespace cm
