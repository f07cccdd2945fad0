// Taps of 2D interpolations of slices read through buffer resources, shared by the culled insertion kernels and the
// virtual volume, and the culled kernels' polynomial window.
#pragma once

#include "common.hpp"

namespace noa_hip {

constexpr i32 NWIN = 12;               // degree of the window polynomial

// Polynomial form of windowed_sinc(f, fs, fb) (FourierProject.hpp:99-110) on f in [-fb, fb], in t = 2 (f/fb)^2 - 1
// (the window is even): Chebyshev interpolation of degree NWIN at the Chebyshev nodes, converted to monomials in
// t and rounded to single precision. The fit is accepted when the kernel's own single-precision evaluation
// (window_poly, reproduced here with the same roundings) stays within 4e-7 of the double-precision window on a
// dense grid; otherwise the kernel evaluates noa's expression. Kept per (fs, fb) for the process lifetime (insert.hip).
struct WindowFit {
    float a[NWIN + 1];
    bool ok;
};
WindowFit fit_window(float fs, float fb);

// Windowed sinc of the culled kernels in single precision: a polynomial of degree NWIN in t = 2 (fz/f_b)^2 - 1
// (the window is even in fz), fitted on the host per (f_s, f_b) and accepted only when its error, evaluated
// in single precision, stays below 4e-7 on [-f_b, f_b] (noa's FP32 expression itself carries ~2e-7 of rounding).
__device__ __forceinline__ float window_poly(float fz, float inv_fb, const float (&a)[NWIN + 1]) {
    const float q = fz * inv_fb;
    const float t = fmaf(2.f * q, q, -1.f);
    float r = a[NWIN];
#pragma unroll
    for (i32 k = NWIN - 1; k >= 0; --k) r = fmaf(r, t, a[k]);
    return r;
}

// The taps of one 2D interpolation of a slice and of its weights (Interpolation.hpp:435-526): noa's flip of the
// frequency when x < 0, the fractions, and the four (LINEAR) or one (NEAREST) tap values, each loaded from a
// clamped address and zeroed when outside the frequency bounds. All loads are issued before any is used.
template<class In, class W, class C>
struct Taps {
    In v[2][2];           // raw loads; zeroed in combine_taps where `ok` is clear (loads stay in flight until then)
    W w[2][2];
    u32 ok;               // bit (y*2 + x): tap inside the bounds
    typename vt<In>::real ty, tx, conj;
};

// A slice (or its weights) read through a buffer resource: base and byte size in scalar registers, a 32-bit byte
// offset per load, and out-of-range offsets read 0.
struct SliceBuf {
    __amdgpu_buffer_rsrc_t rsrc;
    __device__ __forceinline__ SliceBuf(const void* base, u32 bytes)
        : rsrc(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, static_cast<int>(bytes), 0x00020000)) {}
    template<class T> __device__ __forceinline__ T load(u32 elem) const {
        return load_bytes<T>(elem * static_cast<u32>(sizeof(T)));
    }
    template<class T> __device__ __forceinline__ T load_bytes(u32 off) const {
        T v;
        if constexpr (sizeof(T) == 4) {
            const u32 r = __builtin_amdgcn_raw_buffer_load_b32(rsrc, off, 0, 0);
            __builtin_memcpy(&v, &r, 4);
        } else if constexpr (sizeof(T) == 8) {
            const auto r = __builtin_amdgcn_raw_buffer_load_b64(rsrc, off, 0, 0);
            __builtin_memcpy(&v, &r, 8);
        } else {
            const auto r = __builtin_amdgcn_raw_buffer_load_b128(rsrc, off, 0, 0);
            __builtin_memcpy(&v, &r, 16);
        }
        return v;
    }
};

// Element index past the end of any slice or weight buffer (byte offsets 0xFFFFFFF8 for 8-byte values,
// 0x7FFFFFFC for 4-byte weights): a buffer load there returns 0.
constexpr u32 TAP_OUTSIDE = 0x1FFFFFFFu;

template<int INTERP, bool ROWS, class In, class W, class C>
__device__ __forceinline__ Taps<In, W, C> fetch_taps(const SliceBuf& vb, i32 vsy, i32 vsx, const SliceBuf& wb,
                                                     i32 wsy, i32 wsx, bool has_w, i32 ny, i32 nx,
                                                     bool centered, C fy, C fx, bool valid) {
    Taps<In, W, C> t;
    t.conj = 1;
    if (fx < 0) { fy *= -1; fx *= -1; t.conj = -1; }
    const i32 lo_y = -ny / 2, hi_y = (ny - 1) / 2, hi_x = nx / 2;
    if constexpr (ROWS && INTERP == NOA_HIP_INTERP_LINEAR) {
        // Contiguous rows shared by the values and the weights (unit x strides, equal row pitches): one row offset
        // per tap row, and a tap outside the bounds reads TAP_OUTSIDE, which the buffer load returns as 0 -- the
        // zero noa's interpolation adds for it.
        const C fly = floor(fy), flx = floor(fx);
        const i32 y0 = static_cast<i32>(fly), x0 = static_cast<i32>(flx);
        t.ty = static_cast<typename vt<In>::real>(fy - fly);
        t.tx = static_cast<typename vt<In>::real>(fx - flx);
        const bool okx0 = x0 >= 0 && x0 <= hi_x, okx1 = x0 + 1 >= 0 && x0 + 1 <= hi_x;
        t.ok = 0xfu;
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            const bool oky = valid && y0 + y >= lo_y && y0 + y <= hi_y;
            const i32 row = frequency2index(centered, y0 + y, ny) * vsy;
            const u32 e0 = oky && okx0 ? static_cast<u32>(row + x0) : TAP_OUTSIDE;
            const u32 e1 = oky && okx1 ? static_cast<u32>(row + x0 + 1) : TAP_OUTSIDE;
            t.v[y][0] = vb.template load<In>(e0);
            t.v[y][1] = vb.template load<In>(e1);
            t.w[y][0] = wb.template load<W>(e0);
            t.w[y][1] = wb.template load<W>(e1);
        }
        (void)vsx; (void)wsy; (void)wsx; (void)has_w;
    } else if constexpr (INTERP == NOA_HIP_INTERP_NEAREST) {
        const i32 y = static_cast<i32>(round(fy)), x = static_cast<i32>(round(fx));
        const bool ok = valid && y >= lo_y && y <= hi_y && x >= 0 && x <= hi_x;
        const i32 iy = ok ? frequency2index(centered, y, ny) : 0, ix = ok ? x : 0;
        t.v[0][0] = vb.template load<In>(static_cast<u32>(iy * vsy + ix * vsx));
        t.w[0][0] = has_w ? wb.template load<W>(static_cast<u32>(iy * wsy + ix * wsx)) : W(0);
        t.ok = ok ? 1u : 0u;
        t.ty = 0;
        t.tx = 0;
    } else {
        const C fly = floor(fy), flx = floor(fx);
        const i32 y0 = static_cast<i32>(fly), x0 = static_cast<i32>(flx);
        t.ty = static_cast<typename vt<In>::real>(fy - fly);
        t.tx = static_cast<typename vt<In>::real>(fx - flx);
        const bool okx0 = x0 >= 0 && x0 <= hi_x, okx1 = x0 + 1 >= 0 && x0 + 1 <= hi_x;
        t.ok = 0;
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            const bool oky = valid && y0 + y >= lo_y && y0 + y <= hi_y;
            const i32 iy = oky ? frequency2index(centered, y0 + y, ny) : 0;
            const i32 x = oky && okx0 ? x0 : 0;
            t.ok |= (oky && okx0 ? 1u : 0u) << (y * 2);
            t.ok |= (oky && okx1 ? 1u : 0u) << (y * 2 + 1);
            // One load per tap: 16-byte loads of both x taps were measured slower (misaligned at odd x).
            const i32 x1 = oky && okx1 ? x0 + 1 : 0;
            t.v[y][0] = vb.template load<In>(static_cast<u32>(iy * vsy + x * vsx));
            t.v[y][1] = vb.template load<In>(static_cast<u32>(iy * vsy + x1 * vsx));
            t.w[y][0] = has_w ? wb.template load<W>(static_cast<u32>(iy * wsy + x * wsx)) : W(0);
            t.w[y][1] = has_w ? wb.template load<W>(static_cast<u32>(iy * wsy + x1 * wsx)) : W(0);
        }
    }
    return t;
}

// Sums the taps in noa's order: x innermost, then y; then the imaginary part is negated if the frequency was
// flipped (LINEAR only; NEAREST does not conjugate, Interpolation.hpp:479-484).
template<int INTERP, class In, class W, class C>
__device__ __forceinline__ void combine_taps(const Taps<In, W, C>& t, bool has_w, In& value, W& weight) {
    using R = typename vt<In>::real;
    if constexpr (INTERP == NOA_HIP_INTERP_NEAREST) {
        value = vadd(vzero<In>(), vmul(t.ok ? t.v[0][0] : vzero<In>(), R(1)));
        weight = W(0) + (t.ok ? t.w[0][0] : W(0)) * W(1);
    } else {
        const R wy[2] = {1 - t.ty, t.ty}, wx[2] = {1 - t.tx, t.tx};
        value = vzero<In>();
        weight = W(0);
#pragma unroll
        for (int y = 0; y < 2; ++y) {
            In vy = vzero<In>();
            W wyv = W(0);
#pragma unroll
            for (int x = 0; x < 2; ++x) {
                const bool ok = (t.ok >> (y * 2 + x)) & 1u;
                vy = vadd(vy, vmul(ok ? t.v[y][x] : vzero<In>(), wx[x]));
                wyv = wyv + (ok ? t.w[y][x] : W(0)) * static_cast<W>(wx[x]);
            }
            value = vadd(value, vmul(vy, wy[y]));
            weight = weight + wyv * static_cast<W>(wy[y]);
        }
        vimag_mul(value, t.conj);
    }
    (void)has_w;
}

} // namespace noa_hip
