// Shared device helpers for the galario_amd HIP library (gfx950, wave64).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

namespace gl {

// Interleaved complex, same memory layout as std::complex<T> / numpy complex.
template <typename T>
struct alignas(2 * sizeof(T)) cpx {
    T re, im;
};

__device__ __forceinline__ float ffma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double ffma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ void fsincos(float x, float* s, float* c) { sincosf(x, s, c); }
__device__ __forceinline__ void fsincos(double x, double* s, double* c) { sincos(x, s, c); }

template <typename T>
__device__ __forceinline__ cpx<T> mk(T re, T im) { return cpx<T>{re, im}; }
template <typename T>
__device__ __forceinline__ cpx<T> cadd(cpx<T> a, cpx<T> b) { return {a.re + b.re, a.im + b.im}; }
template <typename T>
__device__ __forceinline__ cpx<T> csub(cpx<T> a, cpx<T> b) { return {a.re - b.re, a.im - b.im}; }
template <typename T>
__device__ __forceinline__ cpx<T> cconj(cpx<T> a) { return {a.re, -a.im}; }
template <typename T>
__device__ __forceinline__ cpx<T> cscale(T s, cpx<T> a) { return {s * a.re, s * a.im}; }

// Full complex product with fused multiply-adds (FFT-internal twiddles only;
// the pipeline stages that follow galario's arithmetic never use it).
template <typename T>
__device__ __forceinline__ cpx<T> cmul(cpx<T> a, cpx<T> b) {
    return {ffma(a.re, b.re, -a.im * b.im), ffma(a.re, b.im, a.im * b.re)};
}

// Compile-time loop: f(std::integral_constant<int, I>) for I in [B, E).
template <int B, int E, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (B < E) {
        f(std::integral_constant<int, B>{});
        static_for<B + 1, E>(f);
    }
}

// Cross-lane moves through DPP row patterns: a modifier of a VALU move, no LDS round trip
// (shuffles compile to ds_bpermute, which goes through the LDS crossbar).
enum : int {
    DPP_XOR1 = 0xB1,             // quad_perm [1,0,3,2]: lane l <- l ^ 1
    DPP_XOR2 = 0x4E,             // quad_perm [2,3,0,1]: lane l <- l ^ 2
    DPP_ROW_SHL4 = 0x104,        // lane l <- l + 4 within each row of 16
    DPP_ROW_SHR4 = 0x114,        // lane l <- l - 4 within each row of 16
    DPP_ROW_MIRROR = 0x140,      // lane l <- 15 - l within each row of 16
    DPP_ROW_HALF_MIRROR = 0x141, // lane l <- 7 - l within each half row of 8
    DPP_ROW_BCAST15 = 0x142,     // row r <- lane 15 of row r - 1 (row 0: 0)
    DPP_ROW_BCAST31 = 0x143,     // rows 2 and 3 <- lane 31 (rows 0 and 1: 0)
    DPP_ROW_ROR4 = 0x124,        // row rotation by 4 lanes within each row of 16
    DPP_ROW_ROR8 = 0x128         // row rotation by 8 lanes within each row of 16
};

// The destination's previous value is left undefined (every lane of these patterns has a source, or
// reads zero through bound_ctrl): a defined one would cost a register move per DPP move.
template <int CTRL>
__device__ __forceinline__ int dpp_i32(int x) {
    return __builtin_amdgcn_mov_dpp(x, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double x) {
    const int lo = dpp_i32<CTRL>(__double2loint(x)), hi = dpp_i32<CTRL>(__double2hiint(x));
    return __hiloint2double(hi, lo);
}
// lane l <- l ^ 4: two masked moves (quads 0 and 2 of a row from the quad above, 1 and 3 from below)
__device__ __forceinline__ int xor4_i32(int x) {
    const int up = __builtin_amdgcn_update_dpp(x, x, DPP_ROW_SHL4, 0xF, 0x5, false);
    return __builtin_amdgcn_update_dpp(up, x, DPP_ROW_SHR4, 0xF, 0xA, false);
}
__device__ __forceinline__ double xor4_f64(double x) {
    const int lo = xor4_i32(__double2loint(x)), hi = xor4_i32(__double2hiint(x));
    return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_f64(double x, int lane) {
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(x), lane),
                            __builtin_amdgcn_readlane(__double2loint(x), lane));
}

// Sum of x over each row of 16 lanes, in every lane of the row: pairs, quads, half rows, rows.
__device__ __forceinline__ double row_sum(double x) {
    x += dpp_f64<DPP_XOR1>(x);
    x += dpp_f64<DPP_XOR2>(x);
    x += dpp_f64<DPP_ROW_HALF_MIRROR>(x);
    x += dpp_f64<DPP_ROW_MIRROR>(x);
    return x;
}

// Wave64 sum of a double, the same value in every lane; all 64 lanes must be active.  Rows of 16 by
// row_sum, then the four row sums r0..r3 as (r0 + r1) + (r2 + r3): row 3 adds row 2's sum, row 1 adds
// row 0's, and row 3 adds row 1's.  Every kernel reduces with this one tree, so sums of the same terms
// agree bit for bit across kernels.
__device__ __forceinline__ double wave_sum(double x) {
    x = row_sum(x);
    x += dpp_f64<DPP_ROW_BCAST15>(x);
    x += dpp_f64<DPP_ROW_BCAST31>(x);
    return lane_f64(x, 63);
}

// Row sums of K values at once (K = 1, 2, 4 or 8), each by row_sum's tree: lane l of a row returns the
// sum over its row of a[l mod K].  At every step the lanes trade halves of the vector (a lane keeps the
// values whose index agrees with its own in that bit and takes the other lane's share of them), so K
// sums cost about 7 K instructions instead of 12 K.
template <int K>
__device__ __forceinline__ double joint_row_sums(const double (&a)[K], int lane) {
    static_assert(K == 1 || K == 2 || K == 4 || K == 8, "K values, K a power of two up to 8");
    if constexpr (K == 1) {
        return row_sum(a[0]);
    } else {
        const bool o1 = lane & 1, o2 = lane & 2, o4 = lane & 4;
        double b[K / 2];
#pragma unroll
        for (int j = 0; j < K / 2; ++j)
            b[j] = (o1 ? a[2 * j + 1] : a[2 * j]) + dpp_f64<DPP_XOR1>(o1 ? a[2 * j] : a[2 * j + 1]);
        double x;
        if constexpr (K == 2) {
            x = b[0] + dpp_f64<DPP_XOR2>(b[0]);
            x += xor4_f64(x);
        } else {
            double c[K / 4];
#pragma unroll
            for (int j = 0; j < K / 4; ++j)
                c[j] = (o2 ? b[2 * j + 1] : b[2 * j]) + dpp_f64<DPP_XOR2>(o2 ? b[2 * j] : b[2 * j + 1]);
            if constexpr (K == 4) x = c[0] + xor4_f64(c[0]);
            else x = (o4 ? c[1] : c[0]) + xor4_f64(o4 ? c[0] : c[1]);
        }
        return x + dpp_f64<DPP_ROW_ROR8>(x);
    }
}

// Two 16-bit numbers in one register (lo | hi << 16), and their elementwise unsigned minimum.
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ unsigned pk_min_u16(unsigned a, unsigned b) {
    const u16x2 r = __builtin_elementwise_min(__builtin_bit_cast(u16x2, a), __builtin_bit_cast(u16x2, b));
    return __builtin_bit_cast(unsigned, r);
}

// Row minima (rows of 16 lanes) of two packed pairs at once: even lanes of a row return lo's, odd lanes
// hi's; all 64 lanes must be active.
__device__ __forceinline__ unsigned row_pk_min2(unsigned lo, unsigned hi, int lane) {
    const bool o1 = lane & 1;
    unsigned k = pk_min_u16(o1 ? hi : lo, unsigned(dpp_i32<DPP_XOR1>(int(o1 ? lo : hi))));
    k = pk_min_u16(k, unsigned(dpp_i32<DPP_XOR2>(int(k))));
    k = pk_min_u16(k, unsigned(dpp_i32<DPP_ROW_ROR4>(int(k))));
    return pk_min_u16(k, unsigned(dpp_i32<DPP_ROW_ROR8>(int(k))));
}

// Marks that a point fell outside the grid (device memory, or pinned host memory for the host-array calls).
__device__ __forceinline__ void raise_flag(unsigned* flag) {
    __hip_atomic_store(flag, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

}  // namespace gl
