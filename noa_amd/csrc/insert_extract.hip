// Extraction of central slices from a virtual volume made of other central slices: noa's
// insert_and_extract_central_slices_3d (src/noa/xform/FourierProject.hpp:1916-2049), launcher :1489-1598,
// operator FourierInsertExtract :727-1006.
//
// noa evaluates, for every output pixel, every input slice (O(pixels x slices)). Here one wave owns an 8x8 tile
// of output pixels (8 consecutive frequencies along y, 8 along x) and first scans the input slices 64 at a time,
// one slice per lane: a slice is a candidate when the window along its normal, |fz| < fftfreq_blackman, can hold
// a pixel of the tile. Without an Ewald sphere fz is a linear function of the output pixel's frequency, so over
// the tile its extremes are at the four corners (at each w offset); a margin far above the rounding
// differences between the corners and the interior keeps the test conservative. The candidates are then
// evaluated in increasing slice order, the rotation broadcast from the lane that scanned it, with noa's
// expressions and noa's exact test per pixel, so the sums run in noa's order and skipping a slice never changes a
// result. With an Ewald sphere every slice is a candidate.
//
// Bound: the chain of candidates of the tiles around the origin, which every input slice crosses, and behind it the
// L1's and the vector units' rates on those taps (the slices themselves stay in the caches). Two things shorten it.
// The tiles nearest to the origin are issued first: with tiles in row order the last slices' middle tiles started last
// and ran with the chip nearly empty (61 -> 61 slices of 256^2: twice the time). And for the common calls (arrays in
// single precision, LINEAR, no scaling, no Ewald sphere) the taps of one candidate are in flight while the next one's
// coordinates are computed, a candidate that no pixel of the tile hits costs no load, and the window's sine and cosines are
// short polynomials (84 -> 68 us; 178 us without any of these). Scaled, Ewald, value and FP64 inputs and the other
// interpolations keep the plain loop.
//
// The w-windowed (4D) form keeps the window sum in registers: the outputs start from 0 (or from their value when
// adding) and the w terms are added in increasing w, the order of noa's serial CPU path; no atomics are needed
// since one lane owns each output pixel.
#include <type_traits>

#include "common.hpp"
#include "kernels.hpp"
#include "slice_taps.hpp"

namespace noa_hip {

constexpr int IE_TILE = 8;                 // 8 x 8 output pixels per wave
constexpr int IE_WAVES = 4;                // waves per workgroup

template<class C, class In, class W>
struct InsExtParams {
    // Input slices (batch, y, x strides; the batch stride is 0 for a single slice, as to_interpolator_input).
    const In* in; i64 is_b; i32 is_y, is_x; bool in_is_value; In in_value;
    const W* win; i64 wis_b; i32 wis_y, wis_x; bool win_present, win_is_value; W win_value;
    i32 in_h, in_w;                        // logical height and width of the input slices
    C in_f[2];
    i32 n_in;
    bool in_centered;
    // Output slices.
    void* out; i64 os_b; i32 os_y, os_x;
    W* wout; i64 wos_b; i32 wos_y, wos_x;
    i32 out_h, out_wr;                     // logical height, rfft width
    C out_f[2];
    bool out_centered;
    i32 n_out, tiles_y, tiles_x;
    // Transforms.
    XformArg<C> rot_in, scale_in, rot_out, scale_out;
    C ews[2];
    C cutoff_sqd, in_sinc, in_blackman, w_sinc, w_blackman, volume_z;
    i32 w_size;
    int interp_mode;                       // the method of the INTERP_WINDOW instantiation
    bool add, correct, cull;
    // The pipelined path (arrays, single precision, LINEAR, no scaling or Ewald sphere).
    bool pipelined;
    u32 slice_bytes, wslice_bytes;         // byte extent of one slice and of one weight slice (buffer loads)
    float inv_sinc, inv_blackman;          // 1 / in_sinc, 1 / in_blackman
    float out_inv[2];                      // 1 / out_f
};

// windowed_sinc (FourierProject.hpp:99-110) of the pipelined path, |fz| < blackman. cos(2b) is taken as 2 cos(b)^2 - 1, so
// that the Blackman window is 0.34 + cos(b) (0.5 + 0.16 cos(b)) in two fused multiply-adds. Where the sinc is as wide as the
// window or wider (the default), sin(x) / x and cos(b) are polynomials in the squares of fz / sinc and fz / blackman, which
// are at most 1: (sin(pi q) / (pi q) - 1) / q^2 and (cos(pi q) - 1) / q^2 fitted at 200 Chebyshev nodes of q^2 in [0, 1] and
// rounded; 1 at q = 0 exactly. Fewer roundings than noa's expression: largest error 1.3e-7 to 1.5e-7 against 1.9e-7 to
// 2.0e-7, root mean square 2.4e-8 to 3.0e-8 against 3.4e-8 to 3.6e-8 (widths of 1/16 to 1/384); a narrower sinc takes the
// sine and the cosine (1.6e-7 against 1.7e-7). 61 -> 61 slices of 256^2: 84 us with noa's expression, 76 us with a sincos. (The
// culled insertion's polynomial of the whole window is 2 to 3 times less exact for narrower sincs.)
__device__ __forceinline__ float pipelined_window(float fz, float sinc, float blackman, float inv_sinc, float inv_blackman) {
    float s, c;
    if (sinc >= blackman) {        // uniform
        const float qs = fz * inv_sinc, qb = fz * inv_blackman;
        const float us = qs * qs, ub = qb * qb;
        s = fmaf(0.0001288788771489635f, us, -0.0023245925549417734f);
        s = fmaf(s, us, 0.026136834174394608f);
        s = fmaf(s, us, -0.19074925780296326f);
        s = fmaf(s, us, 0.8117421865463257f);
        s = fmaf(s, us, -1.644934058189392f);
        s = fmaf(s, us, 1.f);
        c = fmaf(-9.057378338184208e-05f, ub, 0.0019106826512143016f);
        c = fmaf(c, ub, -0.02579416148364544f);
        c = fmaf(c, ub, 0.23532620072364807f);
        c = fmaf(c, ub, -1.3352620601654053f);
        c = fmaf(c, ub, 4.058712005615234f);
        c = fmaf(c, ub, -4.934802055358887f);
        c = fmaf(c, ub, 1.f);
    } else {
        const float f = fz * 3.141592653589793238462643383279502884f, x = f / sinc;
        s = x == 0.f ? 1.f : sinf(x) / x;
        c = cosf(f / blackman);
    }
    return s * fmaf(c, fmaf(c, 0.16f, 0.5f), 0.34f);
}

// The candidate whose taps are in flight while the next one's coordinates are computed.
template<class C, class In, class W>
struct InsExtTaps {
    Taps<In, W, C> taps;
    float window;
    bool hit;
};

template<class C, class In, class Out, class W, int INTERP, bool GENERAL>
__global__ __launch_bounds__(IE_TILE * IE_TILE * IE_WAVES) void insert_extract_kernel(const InsExtParams<C, In, W> p) {
    using RIn = typename vt<In>::real;
    using ROut = typename vt<Out>::real;
    constexpr bool FAST = std::is_same_v<C, float> && sizeof(RIn) == 4 && INTERP == NOA_HIP_INTERP_LINEAR && !GENERAL;
    const i32 lane = static_cast<i32>(threadIdx.x & 63);
    const i64 tile = static_cast<i64>(blockIdx.x) * IE_WAVES + (threadIdx.x >> 6);
    const i64 tiles_per_slice = static_cast<i64>(p.tiles_y) * p.tiles_x;
    if (tile >= tiles_per_slice * p.n_out) return;   // whole waves; the kernel has no barrier
    // The tiles nearest to the origin first, over all slices: they meet the most input slices, and one that started last
    // would run alone. Columns of tiles from x = 0 on, each from its middle outwards.
    const i32 t = static_cast<i32>(tile / p.n_out), b = static_cast<i32>(tile - static_cast<i64>(t) * p.n_out);
    const i32 tx = t / p.tiles_y, order = t - tx * p.tiles_y, middle = p.tiles_y / 2;
    // middle, middle - 1, middle + 1, ...; an even number of tiles ends with the first one.
    const i32 ty = (order & 1) ? middle - (order + 1) / 2 : middle + order / 2;
    const i32 fy0 = -(p.out_h / 2) + ty * IE_TILE, x0 = tx * IE_TILE;
    const i32 fy = fy0 + (lane >> 3), x = x0 + (lane & 7);
    const bool valid = fy <= (p.out_h - 1) / 2 && x < p.out_wr;

    // The output pixel's frequency in the virtual volume (compute_fftfreq_in_volume_, :927-933).
    Scale<C> so;
    so.identity = true;
    if constexpr (GENERAL) so = load_scaling(p.scale_out, b);
    const Rot<C> ro = load_rotation(p.rot_out, b);
    auto to_grid = [&](i32 frequency_y, i32 frequency_x) {
        vec2<C> f2;
        if constexpr (sizeof(C) == 4) {
            if (p.pipelined) {
                f2.y = divide_index(static_cast<C>(frequency_y), p.out_f[0], p.out_inv[0]);
                f2.x = divide_index(static_cast<C>(frequency_x), p.out_f[1], p.out_inv[1]);
                return slice2grid<GENERAL>(f2, so, ro, p.ews[0], p.ews[1]);
            }
        }
        f2.y = static_cast<C>(frequency_y) / p.out_f[0];
        f2.x = static_cast<C>(frequency_x) / p.out_f[1];
        return slice2grid<GENERAL>(f2, so, ro, p.ews[0], p.ews[1]);
    };
    const vec3<C> f3 = to_grid(fy, x);
    vec3<C> corner[4];
    corner[0] = to_grid(fy0, x0);
    corner[1] = to_grid(fy0, x0 + IE_TILE - 1);
    corner[2] = to_grid(fy0 + IE_TILE - 1, x0);
    corner[3] = to_grid(fy0 + IE_TILE - 1, x0 + IE_TILE - 1);

    const i32 oy = frequency2index(p.out_centered, fy, p.out_h);
    Out* const out = static_cast<Out*>(p.out) + (static_cast<i64>(b) * p.os_b + oy * p.os_y + x * p.os_x);
    W* const wout = p.wout ? p.wout + (static_cast<i64>(b) * p.wos_b + oy * p.wos_y + x * p.wos_x) : nullptr;
    const bool four_d = p.w_size > 1;
    const bool quat = p.rot_in.kind == NOA_HIP_QUAT_F32 || p.rot_in.kind == NOA_HIP_QUAT_F64;
    Out acc = vzero<Out>();
    W wacc{};
    if (four_d && p.add && valid) {
        acc = *out;
        if (wout) wacc = *wout;
    }

    for (i32 w = 0; w < p.w_size; ++w) {
        vec3<C> f = f3;
        C offset = 0;
        if (four_d) {
            offset = static_cast<C>(w - p.w_size / 2) / p.volume_z;   // w_index_to_fftfreq_offset (:142-145)
            f.z += offset;
        }
        const bool inside = valid && dot3(f) <= p.cutoff_sqd;

        // Bound of fz over the tile at this offset: a slice whose interval misses (-fb, fb) is not a candidate.
        C mag = 0;
        vec3<C> cw[4];
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            cw[c] = corner[c];
            cw[c].z += offset;
            mag = fmax(mag, fabs(cw[c].z) + fabs(cw[c].y) + fabs(cw[c].x));
        }
        const C margin = static_cast<C>(1e-5) * (1 + mag);

        // Every lane scans (slice base + lane), so the scan runs with the whole wave, inside the cutoff or not.
        In value = vzero<In>();
        W weight{};
        InsExtTaps<C, In, W> pend;
        pend.hit = false;
        auto add_taps = [&](const InsExtTaps<C, In, W>& t) {
            if (!t.hit) return;
            In v;
            W wv;
            combine_taps<INTERP>(t.taps, p.win_present, v, wv);
            value = vadd(value, vmul(v, static_cast<RIn>(t.window)));
            weight = weight + (p.win_present ? wv * static_cast<W>(t.window) : static_cast<W>(t.window));
        };
        const i32 n_scan = __any(inside) ? p.n_in : 0;
        for (i32 base = 0; base < n_scan; base += 64) {
            const i32 i = base + lane;
            Rot<C> r{};
            bool cand = false;
            if (i < p.n_in) {
                r = load_rotation(p.rot_in, i);
                cand = true;
                if (p.cull) {
                    C lo = r.apply(cw[0]).z, hi = lo;
#pragma unroll
                    for (int c = 1; c < 4; ++c) {
                        const C z = r.apply(cw[c]).z;
                        lo = fmin(lo, z);
                        hi = fmax(hi, z);
                    }
                    cand = lo - margin < p.in_blackman && hi + margin > -p.in_blackman;
                }
            }
            u64 mask = __ballot(cand);
            if constexpr (FAST) {
                if (p.pipelined) {
                    while (mask) {
                        const i32 k = __ffsll(static_cast<long long>(mask)) - 1;
                        mask &= mask - 1;
                        Rot<C> rk;
                        rk.quat = quat;
#pragma unroll
                        for (int q = 0; q < 9; ++q) rk.m[q] = bcast(r.m[q], k);
                        const vec3<C> g = rk.apply(f);
                        const bool hit = inside && fabs(g.z) < p.in_blackman;
                        if (!__any(hit)) continue;      // the tile's bound is not a pixel's
                        const i64 ii = base + k;
                        const SliceBuf sb(p.in + ii * p.is_b, p.slice_bytes);
                        const SliceBuf wb(p.win_present ? static_cast<const void*>(p.win + ii * p.wis_b)
                                                        : static_cast<const void*>(p.in), p.wslice_bytes);
                        InsExtTaps<C, In, W> next;
                        next.hit = hit;
                        next.window = pipelined_window(g.z, p.in_sinc, p.in_blackman, p.inv_sinc, p.inv_blackman);
                        next.taps = fetch_taps<INTERP, false, In, W>(sb, p.is_y, p.is_x, wb, p.wis_y, p.wis_x,
                                                                     p.win_present, p.in_h, p.in_w, p.in_centered,
                                                                     g.y * p.in_f[0], g.x * p.in_f[1], hit);
                        add_taps(pend);
                        pend = next;
                    }
                    continue;
                }
            }
            while (mask) {
                const i32 k = __ffsll(static_cast<long long>(mask)) - 1;
                mask &= mask - 1;
                const i32 ii = base + k;
                Rot<C> rk;
                rk.quat = quat;
#pragma unroll
                for (int q = 0; q < 9; ++q) rk.m[q] = bcast(r.m[q], k);
                Scale<C> si;
                si.identity = true;
                if constexpr (GENERAL) si = load_scaling(p.scale_in, ii);
                // sample_virtual_volume_ (:935-977).
                vec2<C> g;
                const C fz = grid2slice<GENERAL>(f, si, rk, p.ews[0], p.ews[1], g);
                if (inside && fabs(fz) < p.in_blackman) {
                    const C window = windowed_sinc<C>(fz, p.in_sinc, p.in_blackman);
                    const C py = g.y * p.in_f[0], px = g.x * p.in_f[1];
                    const In v = interp2<INTERP, In>(p.in + static_cast<i64>(ii) * p.is_b, p.is_y, p.is_x, p.in_h,
                                                     p.in_w, p.in_centered, py, px, p.in_is_value, p.in_value,
                                                     p.interp_mode);
                    value = vadd(value, vmul(v, static_cast<RIn>(window)));
                    if (p.win_present) {
                        const W wv = interp2<INTERP, W>(p.win + static_cast<i64>(ii) * p.wis_b, p.wis_y, p.wis_x,
                                                        p.in_h, p.in_w, p.in_centered, py, px, p.win_is_value,
                                                        p.win_value, p.interp_mode);
                        weight = weight + wv * static_cast<W>(window);
                    } else {
                        weight = weight + static_cast<W>(window);
                    }
                }
            }
        }

        if constexpr (FAST) add_taps(pend);

        if (!four_d) {
            // 3D operator (:858-886): 0 beyond the cutoff, unless adding.
            if (!valid) continue;
            if (!inside) {
                if (!p.add) {
                    *out = vzero<Out>();
                    if (wout) *wout = W{};
                }
                continue;
            }
            if (p.correct) {
                const W final_weight = fmax(W(1), fabs(weight));
                if constexpr (vt<In>::cx) {
                    value.x = value.x / static_cast<RIn>(final_weight);
                    value.y = value.y / static_cast<RIn>(final_weight);
                } else {
                    value = value / static_cast<RIn>(final_weight);
                }
            }
            const Out o = vcast<Out>(value);
            *out = p.add ? vadd(*out, o) : o;
            if (wout) *wout = p.add ? *wout + weight : weight;
        } else if (inside) {
            // 4D operator (:890-924): the w term, weighted by the w window.
            const C conv = windowed_sinc<C>(offset, p.w_sinc, p.w_blackman);
            acc = vadd(acc, vmul(vcast<Out>(value), static_cast<ROut>(conv)));
            wacc = wacc + weight * static_cast<W>(conv);
        }
    }
    if (four_d && valid) {
        *out = acc;
        if (wout) *wout = wacc;
    }
}

namespace {

template<class C>
XformArg<C> xform_arg(const Xform& x) {
    XformArg<C> a{};
    a.data = x.data;
    a.kind = x.kind;
    a.batched = x.batched ? 1 : 0;
    for (int i = 0; i < 9; ++i) a.single[i] = x.single[i];
    return a;
}

template<class T> T constant(const Arr& a) {
    if constexpr (vt<T>::cx) {
        T v;
        v.x = static_cast<typename vt<T>::real>(a.value[0]);
        v.y = static_cast<typename vt<T>::real>(a.value[1]);
        return v;
    } else {
        return static_cast<T>(a.value[0]);
    }
}

template<class C, class In, class Out, class W>
int run(const InsertExtractDesc& d, hipStream_t stream, std::string& err) {
    InsExtParams<C, In, W> p{};
    p.in = static_cast<const In*>(d.input.data);
    p.is_b = d.in_shape[0] == 1 ? 0 : d.input.s0;
    p.is_y = static_cast<i32>(d.input.s1);
    p.is_x = static_cast<i32>(d.input.s2);
    p.in_is_value = d.input.is_value;
    p.in_value = constant<In>(d.input);
    p.win_present = d.input_weight.present();
    p.win = static_cast<const W*>(d.input_weight.data);
    p.wis_b = d.in_shape[0] == 1 ? 0 : d.input_weight.s0;
    p.wis_y = static_cast<i32>(d.input_weight.s1);
    p.wis_x = static_cast<i32>(d.input_weight.s2);
    p.win_is_value = d.input_weight.is_value;
    p.win_value = constant<W>(d.input_weight);
    p.in_h = static_cast<i32>(d.in_shape[2]);
    p.in_w = static_cast<i32>(d.in_shape[3]);
    p.in_f[0] = static_cast<C>(d.in_shape[2]);
    p.in_f[1] = static_cast<C>(d.in_shape[3]);
    p.n_in = static_cast<i32>(d.in_shape[0]);
    p.in_centered = d.src_centered;
    p.out = d.output.data;
    p.os_b = d.output.s0;
    p.os_y = static_cast<i32>(d.output.s1);
    p.os_x = static_cast<i32>(d.output.s2);
    p.wout = static_cast<W*>(d.output_weight.data);
    p.wos_b = d.output_weight.s0;
    p.wos_y = static_cast<i32>(d.output_weight.s1);
    p.wos_x = static_cast<i32>(d.output_weight.s2);
    p.out_h = static_cast<i32>(d.out_shape[2]);
    p.out_wr = static_cast<i32>(d.out_shape[3] / 2 + 1);
    p.out_f[0] = static_cast<C>(d.out_shape[2]);
    p.out_f[1] = static_cast<C>(d.out_shape[3]);
    p.out_centered = d.dst_centered;
    p.n_out = static_cast<i32>(d.out_shape[0]);
    p.tiles_y = static_cast<i32>((d.out_shape[2] + IE_TILE - 1) / IE_TILE);
    p.tiles_x = (p.out_wr + IE_TILE - 1) / IE_TILE;
    p.rot_in = xform_arg<C>(d.rot_in);
    p.scale_in = xform_arg<C>(d.scale_in);
    p.rot_out = xform_arg<C>(d.rot_out);
    p.scale_out = xform_arg<C>(d.scale_out);
    // noa's constructor (:791-845), in the coordinate precision.
    if (d.ews_radius[0] != 0 || d.ews_radius[1] != 0) {
        p.ews[0] = 1 / (2 * static_cast<C>(d.ews_radius[0]));
        p.ews[1] = 1 / (2 * static_cast<C>(d.ews_radius[1]));
    }
    C cutoff = static_cast<C>(d.cutoff);
    cutoff = cutoff > C(0) ? cutoff : C(0);
    p.cutoff_sqd = cutoff * cutoff;
    p.volume_z = static_cast<C>(d.out_shape[2] < d.out_shape[3] ? d.out_shape[2] : d.out_shape[3]);
    const C min_f = 1 / p.volume_z;
    auto clamp_min = [&](double v) { const C c = static_cast<C>(v); return c > min_f ? c : min_f; };
    p.in_sinc = clamp_min(d.in_sinc);
    p.in_blackman = clamp_min(d.in_blackman);
    p.w_sinc = clamp_min(d.w_sinc);
    p.w_blackman = clamp_min(d.w_blackman);
    p.w_size = static_cast<i32>(d.w_size);
    p.add = d.add;
    p.correct = d.correct;
    if constexpr (std::is_same_v<C, float> && sizeof(typename vt<In>::real) == 4) {
        auto extent = [&](i64 sy, i64 sx, size_t elem) -> u64 {
            if (sy < 0 || sx < 0) return ~u64(0);
            return (static_cast<u64>(p.in_h - 1) * sy + static_cast<u64>(p.in_w / 2) * sx + 1) * elem;
        };
        const u64 sb = extent(d.input.s1, d.input.s2, sizeof(In));
        const u64 wb = p.win_present ? extent(d.input_weight.s1, d.input_weight.s2, sizeof(W)) : 0;
        p.pipelined = !d.general && !p.in_is_value && !p.win_is_value && sb < 0x7ffffff0u && wb < 0x7ffffff0u &&
                      d.out_shape[2] < 4096 && d.out_shape[3] < 4096;
        p.slice_bytes = static_cast<u32>(sb);
        p.wslice_bytes = static_cast<u32>(wb);
        p.inv_sinc = 1.f / p.in_sinc;
        p.inv_blackman = 1.f / p.in_blackman;
        for (int i = 0; i < 2; ++i) p.out_inv[i] = 1.f / p.out_f[i];
    }
    p.cull = !(d.ews_radius[0] != 0 || d.ews_radius[1] != 0);

    const i64 tiles = static_cast<i64>(p.tiles_y) * p.tiles_x * p.n_out;
    const i64 blocks = (tiles + IE_WAVES - 1) / IE_WAVES;
    if (blocks * IE_TILE * IE_TILE * IE_WAVES > MAX_LANES) { err = "insert_and_extract: too many output slices"; return NOA_HIP_ERROR_UNSUPPORTED; }
    const dim3 grid(static_cast<u32>(blocks)), block(IE_TILE * IE_TILE * IE_WAVES);
    p.interp_mode = d.interp;
    auto launch = [&](auto interp_tag) {
        constexpr int I = decltype(interp_tag)::value;
        if (d.general) hipLaunchKernelGGL((insert_extract_kernel<C, In, Out, W, I, true>), grid, block, 0, stream, p);
        else hipLaunchKernelGGL((insert_extract_kernel<C, In, Out, W, I, false>), grid, block, 0, stream, p);
    };
    if (d.interp == NOA_HIP_INTERP_NEAREST) launch(std::integral_constant<int, NOA_HIP_INTERP_NEAREST>{});
    else if (d.interp == NOA_HIP_INTERP_LINEAR) launch(std::integral_constant<int, NOA_HIP_INTERP_LINEAR>{});
    else launch(std::integral_constant<int, INTERP_WINDOW>{});
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) { err = std::string("kernel launch failed: ") + hipGetErrorString(e); return NOA_HIP_ERROR_RUNTIME; }
    return NOA_HIP_OK;
}

template<class C>
int dispatch(const InsertExtractDesc& d, hipStream_t stream, std::string& err) {
    const int in = d.input.dtype, out = d.output.dtype;
    if (in == NOA_HIP_C32 && out == NOA_HIP_C32) return run<C, float2, float2, float>(d, stream, err);
    if (in == NOA_HIP_C32 && out == NOA_HIP_F32) return run<C, float2, float, float>(d, stream, err);
    if (in == NOA_HIP_F32 && out == NOA_HIP_F32) return run<C, float, float, float>(d, stream, err);
    if (in == NOA_HIP_C64 && out == NOA_HIP_C64) return run<C, double2, double2, double>(d, stream, err);
    if (in == NOA_HIP_C64 && out == NOA_HIP_F64) return run<C, double2, double, double>(d, stream, err);
    if (in == NOA_HIP_F64 && out == NOA_HIP_F64) return run<C, double, double, double>(d, stream, err);
    err = "insert_and_extract: unsupported input/output value types";
    return NOA_HIP_ERROR_UNSUPPORTED;
}

} // namespace

int launch_insert_extract(const InsertExtractDesc& d, hipStream_t stream, std::string& err) {
    return d.coord_f64 ? dispatch<double>(d, stream, err) : dispatch<float>(d, stream, err);
}

} // namespace noa_hip
