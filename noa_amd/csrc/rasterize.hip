// Fourier insertion of central slices by trilinear rasterisation (scatter).
//
// Replaces FourierInsertRasterize (src/noa/xform/FourierProject.hpp:161-390) launched by
// launch_rasterize_central_slices_3d (:1260-1317).
//
// Design (gfx950): one lane per slice pixel, 256-lane workgroups over consecutive pixels of one slice (the
// slice reads are coalesced and the rotation is a scalar load). Each in-cutoff pixel spreads its value over
// the 2x2x2 trilinear cube (plus the conjugate x=0 duplicates) with device-wide hardware float atomics
// (global_atomic_add_f32) on the coarse-grained volume; the volume is small enough to stay in L2/MALL, where
// the atomics execute. Summation order across pixels is not fixed: the result is deterministic only up to
// float reassociation, as with noa's CUDA and OpenMP paths.
//
// One cubic size (FP32 values and weights, single-precision rotations, cutoff <= 0.5) takes rasterize_box_kernel
// instead, but for the smallest calls: the accumulation happens in LDS and reaches the volume once per work item.
#include "common.hpp"
#include "kernels.hpp"
#include "workspace.hpp"

#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <tuple>
#include <vector>

namespace noa_hip {

template<class C, class In, class Out, class W>
struct RasterParams {
    const In* in; i64 is_b; i32 is_y, is_x; bool in_is_value; In in_value;
    const W* win; i64 wis_b; i32 wis_y, wis_x; bool win_present, win_is_value; W win_value;
    Out* vol; i32 vs0, vs1, vs2;
    W* wvol; i32 wvs0, wvs1, wvs2; bool has_wvol;
    i32 grid[3];
    C target[3];
    C slice_f[2];
    i32 slice_h, slice_wr, pixels, tiles;
    C cutoff_sqd;
    C ews[2];
    XformArg<C> rot, scale;
    bool general, slices_centered, vol_centered;
};

template<class C, class In, class Out, class W>
__global__ __launch_bounds__(256) void rasterize_kernel(const RasterParams<C, In, Out, W> p) {
    using RIn = typename vt<In>::real;
    using RO = typename vt<Out>::real;
    const u32 lb = xcd_swizzle(blockIdx.x, gridDim.x);
    const i32 b = static_cast<i32>(lb / static_cast<u32>(p.tiles));
    const i32 tile = static_cast<i32>(lb) - b * p.tiles;
    const i32 pix = tile * 256 + static_cast<i32>(threadIdx.x);
    if (pix >= p.pixels) return;
    const i32 y = pix / p.slice_wr;
    const i32 u = pix - y * p.slice_wr;

    const Rot<C> rot = load_rotation(p.rot, b);
    Scale<C> sc;
    sc.identity = true;
    if (p.general) sc = load_scaling(p.scale, b);

    // operator() (:238-267)
    vec2<C> f2;
    f2.y = static_cast<C>(index2frequency(p.slices_centered, y, p.slice_h)) / p.slice_f[0];
    f2.x = static_cast<C>(u) / p.slice_f[1];
    vec3<C> f = p.general ? slice2grid<true>(f2, sc, rot, p.ews[0], p.ews[1])
                          : slice2grid<false>(f2, sc, rot, p.ews[0], p.ews[1]);
    if (dot3(f) > p.cutoff_sqd) return;
    RIn conjugate = 1;
    if (f.x < 0) {
        f.z = -f.z; f.y = -f.y; f.x = -f.x;
        if constexpr (vt<In>::cx) conjugate = -1;
    }
    const C fz = f.z * p.target[0], fy = f.y * p.target[1], fx = f.x * p.target[2];

    // get_input_value_ (:270-277): complex->complex is multiplied by `conjugate`, i.e. NEGATED when -1.
    const In raw = p.in_is_value ? p.in_value : p.in[static_cast<i64>(b) * p.is_b + y * p.is_y + u * p.is_x];
    Out value;
    if constexpr (vt<In>::cx && vt<Out>::cx) value = vcast<Out>(vmul(raw, conjugate));
    else value = vcast<Out>(raw);
    // get_input_weight_ (:279-286)
    W weight{};
    if (p.has_wvol) {
        if (!p.win_present) weight = W(1);
        else weight = p.win_is_value ? p.win_value : p.win[static_cast<i64>(b) * p.wis_b + y * p.wis_y + u * p.wis_x];
    }

    // rasterize_on_3d_grid_ (:309-373)
    const C flz = floor(fz), fly = floor(fy), flx = floor(fx);
    const i32 b0z = static_cast<i32>(flz), b0y = static_cast<i32>(fly), b0x = static_cast<i32>(flx);
    C fr[2][3];
    fr[1][0] = fz - static_cast<C>(b0z);
    fr[1][1] = fy - static_cast<C>(b0y);
    fr[1][2] = fx - static_cast<C>(b0x);
    fr[0][0] = 1 - fr[1][0];
    fr[0][1] = 1 - fr[1][1];
    fr[0][2] = 1 - fr[1][2];
    const i32 D = p.grid[0], H = p.grid[1], width = p.grid[2] / 2 + 1;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
        const i32 iw = frequency2index(p.vol_centered, b0z + w, D);
        if (iw < 0 || iw >= D) continue;
#pragma unroll
        for (int v = 0; v < 2; ++v) {
            const i32 iv = frequency2index(p.vol_centered, b0y + v, H);
            if (iv < 0 || iv >= H) continue;
#pragma unroll
            for (int uu = 0; uu < 2; ++uu) {
                const i32 iu = b0x + uu;
                // noa bounds iu by the logical W (:332); taps with iu >= W/2+1 only occur with a zero weight
                // for cutoffs <= 0.5 and would write outside the stored half, so they are skipped.
                if (iu < 0 || iu >= width) continue;
                const C k = fr[w][0] * fr[v][1] * fr[uu][2];
                atomic_add(p.vol + (iw * p.vs0 + iv * p.vs1 + iu * p.vs2), vmul(value, static_cast<RO>(k)));
                if (p.has_wvol)
                    atomic_add(p.wvol + (iw * p.wvs0 + iv * p.wvs1 + iu * p.wvs2), weight * static_cast<W>(k));
            }
        }
    }
    // The x=0 plane is redundant: add the conjugate at (-w, -v, 0) with the same fraction (:347-372).
    if (b0x == 0) {
        if constexpr (vt<Out>::cx) value.y = -value.y;
#pragma unroll
        for (int w = 0; w < 2; ++w) {
            const i32 iw = frequency2index(p.vol_centered, -(b0z + w), D);
            if (iw < 0 || iw >= D) continue;
#pragma unroll
            for (int v = 0; v < 2; ++v) {
                const i32 iv = frequency2index(p.vol_centered, -(b0y + v), H);
                if (iv < 0 || iv >= H) continue;
                const C k = fr[w][0] * fr[v][1] * fr[0][2];
                atomic_add(p.vol + (iw * p.vs0 + iv * p.vs1), vmul(value, static_cast<RO>(k)));
                if (p.has_wvol)
                    atomic_add(p.wvol + (iw * p.wvs0 + iv * p.wvs1), weight * static_cast<W>(k));
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------------------
// Boxed rasterisation. The floor positions of the (flipped) pixel coordinates are cut into boxes of 8 x 8 x 16. A work
// item is (box, a number of consecutive slices that cross it), one wave, which runs without barriers:
//   - LDS holds the box's own accumulators, 9 x 9 x 17 positions of value and weight (the trilinear taps reach
//     floor + 1), zeroed at the start.
//   - 64 slices at a time, lane l sets up slice c0 + l: its plane's normal (the crossing test), the row equation of
//     its pixels in the box and the reciprocals of its row direction. A crossing slice's geometry is broadcast from
//     that lane; nothing is divided or loaded per (box, slice) pair.
//   - Lanes 0-31 take pixel rows of the direct set and lanes 32-63 rows of the mirrored one (the x < 0 flip), each
//     the range of its row inside the box (widened by a margin far above the rounding). Every row marks its first
//     candidate in LDS; a running maximum over the wave then gives each of 64 consecutive candidates its row.
//   - A candidate runs noa's expressions of rasterize_kernel, up to its cutoff test and its floor position; the ones
//     inside the box go into a queue in LDS, so that the pixels of several slices share a wave: a slice alone fills
//     half of its lanes (60 pixels of an average crossing, in one or two groups of 64).
//   - When the queue holds 64 pixels, their values and weights are loaded, and the 64 pixels loaded before them are
//     accumulated: eight taps by plain LDS read-modify-write, tap by tap in program order (LDS executes one wave's
//     instructions in order; compiler barriers keep the order). Lanes with the same floor position would update the
//     same words in one instruction: each lane writes its id into a tag byte of its position and reads it back; the
//     lane that reads its own id accumulates, the others (12 % of the pixels of a rotation share their position with
//     an earlier one) return to the queue. A batch with many of them (a collapsed transform puts a whole slice into
//     one position) adds them with the LDS float atomic instead, which costs about two clocks per lane and tap.
//   - After the item's slices, the 9 x 9 x 17 sums are added to the volume with device-wide atomics at noa's indices:
//     frequency2index of the position, dropped outside [0, D) x [0, H) x [0, W/2+1) (the bounds checks
//     rasterize_kernel applies per tap, so the wrapped taps of the non-centred layout land where they land there).
//     Neighbouring boxes overlap by one layer; both add theirs. The x = 0 duplicates (the conjugate at (-w, -v, 0)
//     with the same fraction, :347-372) are the conjugates of the sums at x = 0, which only the pixels with a floor
//     of 0 reach: they are added once per item at the mirrored position.
// Summation order is not fixed (the device atomics), as with rasterize_kernel.
// Bound by neither unit alone but by what one wave can have under way, at 8 waves per CU (20 KB of LDS each): 1.06e8 pixels
// in 2.39 ms at 4,096 slices of 256^2, the vector units busy 56 % of the time, the LDS 38 % (half of it bank conflicts of the
// taps), 6.8 waves resident per CU on average, which spend 38 % of their time waiting for their own loads and LDS
// operations. Four 16 x 16 x 4 slabs of a tile per workgroup, one slice at a time (no queue) and the LDS float atomic for
// every pixel that shares its position, took 5.5 ms, of which the atomics were more than half.
// ---------------------------------------------------------------------------------------------------------
constexpr i32 RB_Z = 8, RB_Y = 8, RB_X = 16;                  // floor positions of a box
constexpr i32 RL_Y = RB_Y + 1, RL_X = RB_X + 1;               // LDS extents
constexpr i32 RB_CELLS = (RB_Z + 1) * RL_Y * RL_X;            // accumulator positions
constexpr i32 RB_TAGS = RB_Z * RB_Y * RB_X;
constexpr i32 RB_QUEUE = 128;                                 // at most 63 waiting + 64 new pixels
constexpr i32 RB_MAX_N = 766;                                 // rows and columns of a slice fit 10 bits of a queue word
constexpr i32 RB_MAX_SHARED = 24;                             // more same-position lanes than this: LDS atomics
static_assert(RB_Z == 8 && RB_Y == 8 && RB_X == 16, "a floor position takes 10 bits of a queue word");

template<class In, class Out>
struct RasterBoxParams {
    const In* in; i64 is_b; i32 is_y, is_x; bool in_is_value; In in_value;
    const float* win; i64 wis_b; i32 wis_y, wis_x; bool win_present, win_is_value; float win_value;
    Out* vol; i32 vs0, vs1, vs2;
    float* wvol; i32 wvs0, wvs1, wvs2; bool has_wvol;
    XformArg<float> rot, scale;         // scale: Mat22 inverse scaling, or none
    const i32* boxes;                   // active boxes, the ones nearest to the origin first
    i32* starts;                        // first slice of each item (RB_DONE: none), or null: each wave scans for it
    i32 n, nby, nbx, base, n_slices, pixels;
    i32 n_boxes, per_item, max_items;   // crossing slices per item, items per box
    float inv_wr, inv_n, cutoff_sqd, margin;
    bool vol_centered, slice_centered, scaled;
};

__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

// The plane geometry (crossing test, candidate rows) takes the rotation as a matrix; the per-pixel expressions keep
// the rotation as given (noa's quaternion rotation for quaternions). With an inverse scaling S (applied to the 2D
// frequency before the rotation), pixel (y, x) lands at y (s0 a + s2 c) + x (s1 a + s3 c), with a and c the rotation's
// 2nd and 3rd columns: the same plane, other columns.
__device__ __forceinline__ Rot<float> plane_matrix(const Rot<float>& r, const Scale<float>& s) {
    Rot<float> g;
    rot_matrix(r, g.m);
    g.quat = false;
    if (s.identity) return g;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float a = g.m[3 * i + 1], c = g.m[3 * i + 2];
        g.m[3 * i + 1] = s.m[0] * a + s.m[2] * c;
        g.m[3 * i + 2] = s.m[1] * a + s.m[3] * c;
    }
    return g;
}

__device__ __forceinline__ Scale<float> slice_scaling(const XformArg<float>& a, bool scaled, i64 b) {
    Scale<float> s;
    s.identity = true;
    if (scaled) s = load_scaling(a, b);
    return s;
}

struct BoxOrigin { i32 z, y, x; };

__device__ __forceinline__ BoxOrigin box_origin(i32 box, i32 nby, i32 nbx, i32 base) {
    const i32 bx = box % nbx, zy = box / nbx;
    return {base + (zy / nby) * RB_Z, base + (zy % nby) * RB_Y, bx * RB_X};
}

// The normal of the plane spanned by the 2nd and 3rd columns a and c of a matrix, which need not be orthogonal or of unit
// length: a x c.
__device__ __forceinline__ vec3<float> plane_normal(const Rot<float>& r) {
    vec3<float> v;
    v.z = r.m[4] * r.m[8] - r.m[7] * r.m[5];
    v.y = r.m[7] * r.m[2] - r.m[1] * r.m[8];
    v.x = r.m[1] * r.m[5] - r.m[4] * r.m[2];
    return v;
}

// Does the plane of `r` with the normal `v` cross the box widened by M? The plane is symmetric through the origin, so this
// also decides the mirrored box. The rounding of the normal, and of the pixels' positions, moves the distance by up to
// 3e-7 n times the square of the columns' length and not of the normal's, which is far smaller where they are nearly
// parallel. A matrix that is not finite crosses every box.
__device__ __forceinline__ bool box_crossed(const Rot<float>& r, const vec3<float>& v, BoxOrigin o, float n, float M) {
    const float cz = static_cast<float>(o.z) + 0.5f * RB_Z, cy = static_cast<float>(o.y) + 0.5f * RB_Y;
    const float cx = static_cast<float>(o.x) + 0.5f * RB_X;
    const float d = fabsf((v.z * cz + v.y * cy) + v.x * cx);
    const float az = fabsf(v.z), ay = fabsf(v.y), ax = fabsf(v.x);
    const float top = fmaxf(fmaxf(fmaxf(fabsf(r.m[1]), fabsf(r.m[4])), fmaxf(fabsf(r.m[7]), fabsf(r.m[2]))),
                            fmaxf(fabsf(r.m[5]), fabsf(r.m[8])));
    return !(d > ((0.5f * RB_Z) * az + (0.5f * RB_Y) * ay) + (0.5f * RB_X) * ax + M * ((az + ay) + ax) +
                     (3e-6f * n) * (top * top));
}

// The first slice of each item, for more than 64 slices (otherwise, and where nothing can be allocated, the items scan
// for it themselves, from the first slice): one workgroup per box counts the slices that cross it, and the
// slices whose rank among them is a multiple of per_item start an item. So an item holds per_item crossing slices
// whatever the orientations are: a model of uniform orientations makes one long item of every box on the axis of a
// tilt series (1,200 slices of 200^2: 4.3 ms, against 0.8 ms).
constexpr i32 RB_DONE = -1;
constexpr i32 RB_SCAN = 256;                                  // slices tested at a time by the items kernel
template<class In, class Out>
__global__ __launch_bounds__(RB_SCAN) void rasterize_items_kernel(const RasterBoxParams<In, Out> p) {
    __shared__ i32 passed[2][RB_SCAN / 64];
    const i32 t = static_cast<i32>(threadIdx.x), wave = t >> 6;
    const BoxOrigin o = box_origin(p.boxes[blockIdx.x], p.nby, p.nbx, p.base);
    i32* starts = p.starts + static_cast<i64>(blockIdx.x) * p.max_items;
    i32 seen = 0, turn = 0;
    for (i32 c0 = 0; c0 < p.n_slices; c0 += RB_SCAN, turn ^= 1) {
        bool cross = false;
        if (c0 + t < p.n_slices) {
            const Rot<float> r = plane_matrix(load_rotation(p.rot, c0 + t), slice_scaling(p.scale, p.scaled, c0 + t));
            cross = box_crossed(r, plane_normal(r), o, static_cast<float>(p.n), p.margin);
        }
        const unsigned long long m = __ballot(cross);
        if ((t & 63) == 0) passed[turn][wave] = static_cast<i32>(__popcll(m));
        __syncthreads();                 // one barrier per turn: the next one writes the other half
        i32 rank = seen + static_cast<i32>(__builtin_amdgcn_mbcnt_hi(
            static_cast<u32>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<u32>(m), 0u)));
#pragma unroll
        for (i32 w = 0; w < RB_SCAN / 64; ++w) {
            if (w < wave) rank += passed[turn][w];
            seen += passed[turn][w];
        }
        if (cross && rank % p.per_item == 0) starts[rank / p.per_item] = c0 + t;
    }
    for (i32 j = (seen + p.per_item - 1) / p.per_item + t; j < p.max_items; j += RB_SCAN) starts[j] = RB_DONE;
}

// GEN: quaternions or inverse scalings (noa's expressions at run time); otherwise Mat33 rotations.
template<class In, class Out, bool GEN>
__global__ __launch_bounds__(64) void rasterize_box_kernel(const RasterBoxParams<In, Out> p) {
    using RIn = typename vt<In>::real;
    constexpr bool CX = vt<Out>::cx;
    __shared__ Out vacc[RB_CELLS];
    __shared__ float wacc[RB_CELLS];
    __shared__ unsigned char tags[RB_TAGS];
    __shared__ u32 starts[64];
    __shared__ u32 q_word[RB_QUEUE];    // position in the box | slice column << 10 | slice row << 20 | flipped << 31
    __shared__ i32 q_slice[RB_QUEUE];
    __shared__ float q_z[RB_QUEUE], q_y[RB_QUEUE], q_x[RB_QUEUE];

    const i32 lane = static_cast<i32>(threadIdx.x);
    // Part by part over all boxes: workgroup i runs on XCD i % 8, and most boxes have only their first parts, so an order
    // with a box's parts next to each other would give whole XCDs nothing but parts that do not exist.
    const i32 slot = static_cast<i32>(blockIdx.x % static_cast<u32>(p.n_boxes));
    const i32 part = static_cast<i32>(blockIdx.x / static_cast<u32>(p.n_boxes));
    const i32 box = p.boxes[slot];
    const BoxOrigin at0 = box_origin(box, p.nby, p.nbx, p.base);
    const i32 Z0 = at0.z, Y0 = at0.y, X0 = at0.x;
    const i32 n = p.n, width = n / 2 + 1;
    const i32 lo = -n / 2, hi = (n - 1) / 2, hix = n / 2;
    const float P0[3] = {static_cast<float>(Z0), static_cast<float>(Y0), static_cast<float>(X0)};
    constexpr float EXT[3] = {RB_Z, RB_Y, RB_X};
    const float nf = static_cast<float>(n), M = p.margin;
    // The item's first slice: its slices are the next `left` ones that cross the box.
    i32 first = 0, left = p.per_item;
    if (p.starts) {
        first = p.starts[static_cast<i64>(slot) * p.max_items + part];
        if (first < 0) return;
    } else {
        i32 skip = part * p.per_item;
        unsigned long long m = 0;
        for (; first < p.n_slices; first += 64) {
            bool cross = false;
            if (first + lane < p.n_slices) {
                const Rot<float> r = plane_matrix(load_rotation(p.rot, first + lane),
                                                  slice_scaling(p.scale, GEN && p.scaled, first + lane));
                cross = box_crossed(r, plane_normal(r), at0, nf, M);
            }
            m = __ballot(cross);
            const i32 cnt = static_cast<i32>(__popcll(m));
            if (skip < cnt) break;
            skip -= cnt;
        }
        if (first >= p.n_slices) return;
        for (; skip > 0; --skip) m &= m - 1;
        first += __ffsll(static_cast<long long>(m)) - 1;
    }
    for (i32 i = lane; i < RB_CELLS; i += 64) {
        vacc[i] = vzero<Out>();
        wacc[i] = 0.f;
    }
    lds_order();

    // The box of this lane's set, widened by the margin: direct positions in [P0, P0 + EXT), mirrored ones in
    // (-P0 - EXT, -P0].
    const bool mirrored_rows = lane >= 32;
    float blo[3], bhi[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        blo[i] = (mirrored_rows ? -(P0[i] + EXT[i]) : P0[i]) - M;
        bhi[i] = (mirrored_rows ? -P0[i] : P0[i] + EXT[i]) + M;
    }

    // One batch of queued pixels whose loads are in flight.
    struct Batch {
        u32 word;
        i32 slice;
        float tz, ty, tx, weight;
        In raw;
        bool valid;
    };
    Batch batch{};
    bool have = false;
    i32 queued = 0;

    // Takes the last (at most 64) pixels of the queue and issues their loads.
    auto issue = [&](Batch& q) {
        const i32 m = min(queued, 64);
        queued -= m;
        q.valid = lane < m;
        const i32 at = queued + (q.valid ? lane : 0);
        q.word = q_word[at];
        q.slice = q_slice[at];
        q.tz = q_z[at];
        q.ty = q_y[at];
        q.tx = q_x[at];
        const i32 u = static_cast<i32>((q.word >> 10) & 1023u), y = static_cast<i32>((q.word >> 20) & 1023u);
        q.raw = p.in_value;
        q.weight = p.win_present ? p.win_value : 1.f;
        if (q.valid) {
            if (!p.in_is_value)
                q.raw = p.in[static_cast<i64>(q.slice) * p.is_b + static_cast<i64>(y) * p.is_y + static_cast<i64>(u) * p.is_x];
            if (p.has_wvol && p.win_present && !p.win_is_value)
                q.weight = p.win[static_cast<i64>(q.slice) * p.wis_b + static_cast<i64>(y) * p.wis_y + static_cast<i64>(u) * p.wis_x];
        }
    };
    auto push = [&](bool ok, u32 word, i32 slice, float fz, float fy, float fx) {
        const unsigned long long m = __ballot(ok);
        if (ok) {
            const i32 at = queued + static_cast<i32>(__builtin_amdgcn_mbcnt_hi(
                static_cast<u32>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<u32>(m), 0u)));
            q_word[at] = word;
            q_slice[at] = slice;
            q_z[at] = fz;
            q_y[at] = fy;
            q_x[at] = fx;
        }
        queued += static_cast<i32>(__popcll(m));
    };
    // Accumulates a batch: the eight taps of the lanes that own their floor position.
    auto finish = [&](const Batch& q) {
        const i32 cell = static_cast<i32>(q.word & 1023u);
        if (q.valid) tags[cell] = static_cast<unsigned char>(lane);
        lds_order();
        const bool own = q.valid && tags[cell] == static_cast<unsigned char>(lane);
        const bool shared = q.valid && !own;
        lds_order();
        // get_input_value_ (:270-277): complex -> complex is multiplied by `conjugate`, i.e. negated when flipped.
        Out value;
        if constexpr (vt<In>::cx && CX) value = vcast<Out>(vmul(q.raw, (q.word >> 31) ? RIn(-1) : RIn(1)));
        else value = vcast<Out>(q.raw);
        const float fr[2][3] = {{1 - q.tz, 1 - q.ty, 1 - q.tx}, {q.tz, q.ty, q.tx}};
        const i32 o = ((cell >> 7) * RL_Y + ((cell >> 4) & 7)) * RL_X + (cell & 15);
        const bool many = __popcll(__ballot(shared)) > RB_MAX_SHARED;
#pragma unroll
        for (int w = 0; w < 2; ++w)
#pragma unroll
            for (int v = 0; v < 2; ++v)
#pragma unroll
                for (int uu = 0; uu < 2; ++uu) {
                    const float kk = fr[w][0] * fr[v][1] * fr[uu][2];
                    const i32 at = o + (w * RL_Y + v) * RL_X + uu;
                    if (own) {
                        const Out v0 = vacc[at];
                        const float w0 = wacc[at];
                        vacc[at] = vadd(v0, vmul(value, kk));
                        wacc[at] = w0 + q.weight * kk;
                    }
                    lds_order();
                }
        if (many) {
            if (shared) {
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    const float kk = fr[t >> 2][0] * fr[(t >> 1) & 1][1] * fr[t & 1][2];
                    const i32 at = o + ((t >> 2) * RL_Y + ((t >> 1) & 1)) * RL_X + (t & 1);
                    const Out add = vmul(value, kk);
                    if constexpr (CX) {
                        atomicAdd(&vacc[at].x, add.x);
                        atomicAdd(&vacc[at].y, add.y);
                    } else {
                        atomicAdd(vacc + at, add);
                    }
                    atomicAdd(wacc + at, q.weight * kk);
                }
            }
            lds_order();
        } else {
            push(shared, q.word, q.slice, q.tz, q.ty, q.tx);
        }
    };
    // Batches of 64 as long as the queue holds one; each accumulates the batch loaded before it. `all`: to the end.
    auto drain = [&](bool all) {
        while (queued >= 64 || (all && (queued > 0 || have))) {
            lds_order();
            Batch next{};
            const bool more = queued > 0;
            if (more) issue(next);
            lds_order();
            if (have) finish(batch);
            batch = next;
            have = more;
        }
    };

    for (i32 c0 = first; c0 < p.n_slices && left > 0; c0 += 64) {
        // Lane l: the plane of slice c0 + l. F = Y a + U c; on the plane Y = g . F with g the first row of
        // (G^T G)^-1 G^T, G = [a c].
        float a[3] = {}, c[3] = {}, g[3] = {}, ic[3] = {};
        bool cross = false, flat = false;
        if (c0 + lane < p.n_slices) {
            const Rot<float> r = plane_matrix(load_rotation(p.rot, c0 + lane), slice_scaling(p.scale, GEN && p.scaled, c0 + lane));
            const vec3<float> v = plane_normal(r);
            cross = box_crossed(r, v, at0, nf, M);
            a[0] = r.m[1]; a[1] = r.m[4]; a[2] = r.m[7];
            c[0] = r.m[2]; c[1] = r.m[5]; c[2] = r.m[8];
            const float aa = (a[0] * a[0] + a[1] * a[1]) + a[2] * a[2];
            const float ac = (a[0] * c[0] + a[1] * c[1]) + a[2] * c[2];
            const float cc = (c[0] * c[0] + c[1] * c[1]) + c[2] * c[2];
            // The determinant, far more exact than aa cc - ac^2 where the columns are nearly parallel. All pixels are
            // tried where the columns are parallel to 1e-3, and where they are long enough for the products that cancel
            // inside the volume to round by as much as the margin of 1e-5 n: up to 1e-7 n per unit of length and, below
            // that, n / 1e7 over the sine of the columns' angle, hence a length of 10 and a sine of 0.03.
            const float det = dot3(v);
            flat = !(det > 1e-6f * aa * cc) || (det < 1e-3f * aa * cc && fmaxf(aa, cc) > 100.f);
            const float idet = 1.f / det;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                g[i] = (cc * a[i] - ac * c[i]) * idet;
                // A row direction with no component along the axis is inside or outside as a whole: the huge
                // reciprocal turns the distances to the faces into an unbounded or an empty range.
                ic[i] = fabsf(c[i]) > 1e-12f ? 1.f / c[i] : 1e30f;
            }
        }
        unsigned long long mask = __ballot(cross);
        const unsigned long long flat_mask = __ballot(flat);
        while (mask && left > 0) {
            const i32 k = __ffsll(static_cast<long long>(mask)) - 1;
            mask &= mask - 1;
            --left;
            const i32 b = c0 + k;
            const float A[3] = {bcast(a[0], k), bcast(a[1], k), bcast(a[2], k)};
            const float Cc[3] = {bcast(c[0], k), bcast(c[1], k), bcast(c[2], k)};
            Rot<float> rot{};
            Scale<float> sc;
            sc.identity = true;
            if constexpr (GEN) {
                rot = load_rotation(p.rot, b);
                sc = slice_scaling(p.scale, p.scaled, b);
            }
            // One candidate per lane: noa's expressions (rasterize_kernel) up to the floor position; queued if inside.
            auto evaluate = [&](bool live, i32 fy, i32 u, bool mirrored) {
                vec2<float> f2;
                f2.y = divide_index(static_cast<float>(fy), nf, p.inv_n);
                f2.x = divide_index(static_cast<float>(u), nf, p.inv_n);
                vec3<float> f;
                if constexpr (GEN) {
                    f = p.scaled ? slice2grid<true>(f2, sc, rot, 0.f, 0.f) : slice2grid<false>(f2, sc, rot, 0.f, 0.f);
                } else {
                    f.z = A[0] * f2.y + Cc[0] * f2.x;        // the rotation's first column meets a zero
                    f.y = A[1] * f2.y + Cc[1] * f2.x;
                    f.x = A[2] * f2.y + Cc[2] * f2.x;
                }
                const bool flip = f.x < 0;
                bool ok = live && !(dot3(f) > p.cutoff_sqd) && flip == mirrored;
                if (flip) { f.z = -f.z; f.y = -f.y; f.x = -f.x; }
                const float fz = f.z * nf, fyv = f.y * nf, fx = f.x * nf;
                const float flz = floorf(fz), fly = floorf(fyv), flx = floorf(fx);
                const i32 lz = static_cast<i32>(flz) - Z0, ly = static_cast<i32>(fly) - Y0;
                const i32 lx = static_cast<i32>(flx) - X0;
                ok = ok && static_cast<u32>(lz) < static_cast<u32>(RB_Z) && static_cast<u32>(ly) < static_cast<u32>(RB_Y) &&
                     static_cast<u32>(lx) < static_cast<u32>(RB_X);
                const i32 y = frequency2index(p.slice_centered, fy, n);
                const u32 word = static_cast<u32>((lz << 7) | (ly << 4) | lx) | (static_cast<u32>(u) << 10) |
                                 (static_cast<u32>(y) << 20) | (flip ? 0x80000000u : 0u);
                push(ok, word, b, fz - flz, fyv - fly, fx - flx);
                drain(false);
            };
            if ((flat_mask >> k) & 1u) {
                // Degenerate transform (the plane collapses): every pixel of the slice is a candidate.
                for (i32 pix0 = 0; pix0 < p.pixels; pix0 += 64) {
                    const i32 pix = min(pix0 + lane, p.pixels - 1);
                    const i32 yq = static_cast<i32>((static_cast<float>(pix) + 0.5f) * p.inv_wr);
                    const i32 u = pix - yq * width;
                    const i32 fy = index2frequency(p.slice_centered, yq, n);
                    evaluate(pix0 + lane < p.pixels, fy, u, false);
                    evaluate(pix0 + lane < p.pixels, fy, u, true);
                }
                continue;
            }
            const float G[3] = {bcast(g[0], k), bcast(g[1], k), bcast(g[2], k)};
            const float IC[3] = {bcast(ic[0], k), bcast(ic[1], k), bcast(ic[2], k)};
            float ymin = 0.f, ymax = 0.f;
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                const float t1 = G[i] * blo[i], t2 = G[i] * bhi[i];
                ymin += fminf(t1, t2);
                ymax += fmaxf(t1, t2);
            }
            // The first row of each set (uniform over its 32 lanes).
            const i32 yfirst = max(static_cast<i32>(ceilf(fmaxf(ymin, static_cast<float>(lo) - 1.f))), lo);
            const i32 ylast = min(static_cast<i32>(floorf(fminf(ymax, static_cast<float>(hi) + 1.f))), hi);
            const i32 y_direct = __builtin_amdgcn_readlane(yfirst, 0), y_mirror = __builtin_amdgcn_readlane(yfirst, 32);
            for (i32 rb = 0;; rb += 32) {
                const i32 fy = yfirst + rb + (lane & 31);
                const bool row = fy <= ylast;
                if (__ballot(row) == 0) break;
                // Pixel range of the row: U with Y a + U c inside the box.
                float ulo = 0.f, uhi = static_cast<float>(hix);
                const float fyf = static_cast<float>(fy);
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    const float at = A[i] * fyf;
                    const float t1 = (blo[i] - at) * IC[i], t2 = (bhi[i] - at) * IC[i];
                    ulo = fmaxf(ulo, fminf(t1, t2));
                    uhi = fminf(uhi, fmaxf(t1, t2));
                }
                i32 u0 = 0, cnt = 0;
                if (row && ulo <= uhi) {
                    u0 = static_cast<i32>(ceilf(ulo));
                    cnt = max(0, static_cast<i32>(floorf(uhi)) - u0 + 1);
                }
                const i32 incl = wave_inclusive_sum(cnt), excl = incl - cnt;
                const i32 total = __builtin_amdgcn_readlane(incl, 63);
                const i32 from = u0 - excl;
                for (i32 base = 0; base < total; base += 64) {
                    // The row of candidate base + lane: every row with candidates in the window marks its first one.
                    starts[lane] = 0u;
                    lds_order();
                    if (cnt > 0 && incl > base && excl < base + 64)
                        starts[max(excl - base, 0)] = static_cast<u32>(lane);
                    lds_order();
                    const i32 r = wave_inclusive_max(static_cast<i32>(starts[lane]));
                    lds_order();
                    const i32 u = __builtin_amdgcn_ds_bpermute(r << 2, from) + base + lane;
                    const bool live = base + lane < total;
                    evaluate(live, (r < 32 ? y_direct : y_mirror) + rb + (r & 31), live ? u : 0, r >= 32);
                }
            }
        }
    }
    drain(true);
    lds_order();

    // Flush: positions [Z0, Z0 + 8] x [Y0, Y0 + 8] x [X0, X0 + 16] at noa's indices, inside the stored volume.
    for (i32 i = lane; i < RB_CELLS; i += 64) {
        const i32 dz = i / (RL_Y * RL_X), rem = i - dz * (RL_Y * RL_X);
        const i32 dy = rem / RL_X, dx = rem - dy * RL_X;
        const i32 iu = X0 + dx;
        Out v = vacc[i];
        const float w = wacc[i];
        bool any = w != 0.f;
        if constexpr (CX) any = any || v.x != 0.f || v.y != 0.f;
        else any = any || v != 0.f;
        if (iu >= width || !any) continue;
        auto add = [&](i32 z, i32 y, const Out& value) {
            const i32 iw = frequency2index(p.vol_centered, z, n), iv = frequency2index(p.vol_centered, y, n);
            if (iw < 0 || iw >= n || iv < 0 || iv >= n) return;
            atomic_add(p.vol + (iw * p.vs0 + iv * p.vs1 + iu * p.vs2), value);
            if (p.has_wvol) atomic_add(p.wvol + (iw * p.wvs0 + iv * p.wvs1 + iu * p.wvs2), w);
        };
        add(Z0 + dz, Y0 + dy, v);
        if (iu == 0) {
            if constexpr (CX) v.y = -v.y;
            add(-(Z0 + dz), -(Y0 + dy), v);
        }
    }
}

namespace {

template<class C>
XformArg<C> to_arg(const Xform& x) {
    XformArg<C> a{};
    a.data = x.data;
    a.kind = x.kind;
    a.batched = x.batched ? 1 : 0;
    for (int i = 0; i < 9; ++i) a.single[i] = x.single[i];
    return a;
}

template<class T> T value_of(const Arr& a) {
    if constexpr (vt<T>::cx) {
        T v; v.x = static_cast<typename vt<T>::real>(a.value[0]); v.y = static_cast<typename vt<T>::real>(a.value[1]);
        return v;
    } else {
        return static_cast<T>(a.value[0]);
    }
}

constexpr int NOT_TILED = -1000;

// The boxes that the cutoff sphere reaches, for one size and cutoff: every pixel inside the cutoff has its floor within
// [lo - 1, hi + 1] along z and y and [0, n/2] along x. The ones nearest to the origin, which most slices cross, come
// first. Kept per (device, size, cutoff) for the process lifetime. False where they are not resident and cannot be uploaded:
// while the stream is captured, which allows neither the allocation nor the copy, or without memory.
struct BoxPlan {
    i32* boxes{};
    i32 n_boxes{}, nby{}, nbx{}, base{};
};
std::mutex g_box_mutex;
std::map<std::tuple<int, i32, double>, BoxPlan> g_box_plans;

bool make_box_plan(int device, i32 n, double cutoff, bool captured, BoxPlan& plan) {
    std::lock_guard<std::mutex> lock(g_box_mutex);
    const auto key = std::make_tuple(device, n, cutoff);
    const auto it = g_box_plans.find(key);
    if (it != g_box_plans.end()) {
        plan = it->second;
        return true;
    }
    if (captured) return false;
    BoxPlan pl;
    const i32 lo = -n / 2, hi = (n - 1) / 2;
    pl.base = lo - 1;
    const i32 span = hi + 1 - pl.base + 1;
    const i32 nbz = (span + RB_Z - 1) / RB_Z;
    pl.nby = (span + RB_Y - 1) / RB_Y;
    pl.nbx = (n / 2 + 1 + RB_X - 1) / RB_X;
    const double reach = cutoff * n + 1.0;
    std::vector<std::pair<double, i32>> active;
    for (i32 b = 0; b < nbz * pl.nby * pl.nbx; ++b) {
        const double at[3] = {double(pl.base + b / pl.nbx / pl.nby * RB_Z), double(pl.base + b / pl.nbx % pl.nby * RB_Y),
                              double(b % pl.nbx * RB_X)};
        const double ext[3] = {RB_Z, RB_Y, RB_X};
        double closest = 0, centre = 0;
        for (int a = 0; a < 3; ++a) {
            const double d = std::max({at[a], -(at[a] + ext[a]), 0.0}), c = at[a] + 0.5 * ext[a];
            closest += d * d;
            centre += c * c;
        }
        if (closest <= reach * reach) active.push_back({centre, b});
    }
    std::stable_sort(active.begin(), active.end());
    std::vector<i32> boxes(active.size());
    for (size_t k = 0; k < active.size(); ++k) boxes[k] = active[k].second;
    pl.n_boxes = static_cast<i32>(boxes.size());
    if (!boxes.empty() &&
        (hipMalloc(&pl.boxes, boxes.size() * sizeof(i32)) != hipSuccess ||
         hipMemcpy(pl.boxes, boxes.data(), boxes.size() * sizeof(i32), hipMemcpyHostToDevice) != hipSuccess)) {
        if (pl.boxes) (void)hipFree(pl.boxes);
        (void)hipGetLastError();
        return false;
    }
    g_box_plans[key] = pl;
    plan = pl;
    return true;
}

// The boxed path (rasterize_box_kernel) where it applies: cubic volume and slices, no target shape, no Ewald sphere,
// cutoff <= 0.5, Mat33<f32> or Quaternion<f32> rotations, Mat22 inverse scalings or none. Of these calls it takes all but
//  - the smallest ones, where the lane-per-pixel kernel's single step (about 8 us less than a box's chain of set-up, rows
//    and queue) counts for more than its atomics: up to 16 slices of fewer than 2^14 pixels together. One call with a
//    synchronisation behind it, lane per pixel and boxed: 16 slices of 16^2 35 and 41 us, 8 of 32^2 35 and 42, 4 of 64^2 38
//    and 44, 1 of 128^2 35 and 41; just above the line 8 of 64^2 43 and 43, 2 of 128^2 45 and 42, 16 of 48^2 46 and 44; more
//    slices meet in the same voxels (41 of 16^2 48 and 41 us);
//  - the first one of a size and cutoff where that one is captured (the lane-per-pixel kernel needs nothing resident).
// 41 slices of 192^2 take 109 against 665 us, 4,096 of 256^2 2.4 against 112 ms (with the clearing of the volume, 24 us at
// 256^3). NOA_HIP_RASTERIZE_LAYOUT=direct selects the lane-per-pixel kernel, =tiles the boxed one where it applies;
// NOA_HIP_RASTERIZE_PAIRS sets the crossing slices per work item.
constexpr i64 RB_FEW_SLICES = 16, RB_FEW_PIXELS = 1 << 14;
template<class In, class Out, class C, class W>
int run_tiles(const ProjectDesc& d, const RasterParams<C, In, Out, W>& p, hipStream_t stream, std::string& err) {
    const i64 nn = p.grid[0], n_slices = d.in_shape[0];
    const bool cubic = p.grid[1] == nn && p.grid[2] == nn && d.in_shape[2] == nn && d.in_shape[3] == nn &&
                       d.target[0] == nn && d.target[1] == nn && d.target[2] == nn;
    const i64 stored = nn * nn * (nn / 2 + 1);
    const bool flat = p.ews[0] == 0 && p.ews[1] == 0;
    const bool eligible = cubic && flat && nn >= 16 && nn <= RB_MAX_N && d.cutoff <= 0.5 &&
                          (p.rot.kind == NOA_HIP_MAT33_F32 || p.rot.kind == NOA_HIP_QUAT_F32) &&
                          stored < 0x7fffffffLL && n_slices <= 0x7fffffffLL;
    if (!eligible) return NOT_TILED;
    const char* env = std::getenv("NOA_HIP_RASTERIZE_LAYOUT");
    if (env && std::strcmp(env, "tiles") != 0) return NOT_TILED;
    if (!env && n_slices <= RB_FEW_SLICES && n_slices * p.pixels < RB_FEW_PIXELS) return NOT_TILED;
    int device = 0;
    (void)hipGetDevice(&device);
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    (void)hipStreamIsCapturing(stream, &capture);
    const bool captured = capture != hipStreamCaptureStatusNone;
    BoxPlan plan;
    if (!make_box_plan(device, static_cast<i32>(nn), std::max(d.cutoff, 0.0), captured, plan)) return NOT_TILED;
    if (plan.n_boxes == 0) return NOA_HIP_OK;
    const char* pe = std::getenv("NOA_HIP_RASTERIZE_PAIRS");
    // Crossing slices per item. An item costs its flush (9 x 9 x 17 atomics, most of them non-zero) and its slices, one
    // after the other; the number of items falls and the length of one grows with this number, so the best one grows
    // with the square root of the call's crossings, which are about n^2 / 150 per slice. Measured best (and their
    // neighbours at half and double): 8 slices of 64^2 2, 41 of 192^2 4, 300 of 128^2 32, 300 of 256^2 32-64, 1,000 of
    // 256^2 64-128, 4,096 of 256^2 128.
    const double best = static_cast<double>(nn) * std::sqrt(static_cast<double>(n_slices)) / 110.0;
    i64 per_item = pe ? std::max(1, std::atoi(pe)) : std::min<i64>(256, std::max<i64>(2, std::llround(best)));
    const i64 most = MAX_LANES / 64 / plan.n_boxes;             // parts of a box that the grid can hold
    per_item = std::max(per_item, (n_slices + most - 1) / most);
    const i64 max_items = (n_slices + per_item - 1) / per_item;
    RasterBoxParams<In, Out> q{};
    q.in = p.in; q.is_b = p.is_b; q.is_y = p.is_y; q.is_x = p.is_x; q.in_is_value = p.in_is_value;
    q.in_value = p.in_value;
    q.win = p.win; q.wis_b = p.wis_b; q.wis_y = p.wis_y; q.wis_x = p.wis_x; q.win_present = p.win_present;
    q.win_is_value = p.win_is_value; q.win_value = p.win_value;
    q.vol = p.vol; q.vs0 = p.vs0; q.vs1 = p.vs1; q.vs2 = p.vs2;
    q.wvol = p.wvol; q.wvs0 = p.wvs0; q.wvs1 = p.wvs1; q.wvs2 = p.wvs2; q.has_wvol = p.has_wvol;
    q.rot = p.rot;
    q.scale = p.scale;
    q.scaled = p.general && p.scale.kind != NOA_HIP_XFORM_NONE;
    q.boxes = plan.boxes;
    q.n_boxes = plan.n_boxes;
    q.per_item = static_cast<i32>(per_item);
    q.max_items = static_cast<i32>(max_items);
    q.n = static_cast<i32>(nn);
    q.nby = plan.nby; q.nbx = plan.nbx; q.base = plan.base;
    q.n_slices = static_cast<i32>(n_slices);
    q.pixels = p.pixels;
    q.inv_wr = 1.f / static_cast<float>(p.slice_wr);
    q.inv_n = 1.f / static_cast<float>(nn);
    q.cutoff_sqd = p.cutoff_sqd;
    q.margin = 1e-3f + 1e-5f * static_cast<float>(nn);
    q.vol_centered = p.vol_centered;
    q.slice_centered = p.slices_centered;
    const bool gen = q.scaled || p.rot.kind == NOA_HIP_QUAT_F32;
    const dim3 boxes(static_cast<u32>(plan.n_boxes * max_items));
    CallWorkspace starts;
    if (n_slices > 64 && !captured)
        starts = CallWorkspace(static_cast<size_t>(plan.n_boxes) * max_items * sizeof(i32), stream);
    q.starts = starts.data<i32>();
    if (q.starts)
        hipLaunchKernelGGL((rasterize_items_kernel<In, Out>), dim3(static_cast<u32>(plan.n_boxes)), dim3(RB_SCAN), 0,
                           stream, q);
    if (gen) hipLaunchKernelGGL((rasterize_box_kernel<In, Out, true>), boxes, dim3(64), 0, stream, q);
    else hipLaunchKernelGGL((rasterize_box_kernel<In, Out, false>), boxes, dim3(64), 0, stream, q);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) { err = std::string("kernel launch failed: ") + hipGetErrorString(e); return NOA_HIP_ERROR_RUNTIME; }
    return NOA_HIP_OK;
}

template<class C, class In, class Out, class W>
int run(const ProjectDesc& d, hipStream_t stream, std::string& err) {
    RasterParams<C, In, Out, W> p{};
    p.in = static_cast<const In*>(d.input.data); p.is_b = d.input.s0; p.is_y = (i32)d.input.s1; p.is_x = (i32)d.input.s2;
    p.in_is_value = d.input.is_value; p.in_value = value_of<In>(d.input);
    p.win_present = d.input_weight.present();
    p.win = static_cast<const W*>(d.input_weight.data);
    p.wis_b = d.input_weight.s0; p.wis_y = (i32)d.input_weight.s1; p.wis_x = (i32)d.input_weight.s2;
    p.win_is_value = d.input_weight.is_value; p.win_value = static_cast<W>(d.input_weight.value[0]);
    p.vol = static_cast<Out*>(d.output.data); p.vs0 = (i32)d.output.s0; p.vs1 = (i32)d.output.s1; p.vs2 = (i32)d.output.s2;
    p.has_wvol = d.output_weight.data != nullptr;
    p.wvol = static_cast<W*>(d.output_weight.data);
    p.wvs0 = (i32)d.output_weight.s0; p.wvs1 = (i32)d.output_weight.s1; p.wvs2 = (i32)d.output_weight.s2;
    for (int i = 0; i < 3; ++i) {
        p.grid[i] = static_cast<i32>(d.out_shape[i + 1]);
        p.target[i] = static_cast<C>(d.target[i]);
    }
    p.slice_f[0] = static_cast<C>(d.in_shape[2]);
    p.slice_f[1] = static_cast<C>(d.in_shape[3]);
    p.slice_h = static_cast<i32>(d.in_shape[2]);
    p.slice_wr = static_cast<i32>(d.in_shape[3] / 2 + 1);
    p.pixels = p.slice_h * p.slice_wr;
    p.tiles = (p.pixels + 255) / 256;
    C cutoff = std::max(static_cast<C>(d.cutoff), C(0));
    p.cutoff_sqd = cutoff * cutoff;
    p.general = d.general;
    if (d.general && (d.ews_radius[0] != 0 || d.ews_radius[1] != 0)) {
        p.ews[0] = 1 / (2 * static_cast<C>(d.ews_radius[0]));
        p.ews[1] = 1 / (2 * static_cast<C>(d.ews_radius[1]));
    }
    p.rot = to_arg<C>(d.rot);
    p.scale = to_arg<C>(d.scale);
    p.slices_centered = d.src_centered;
    p.vol_centered = d.dst_centered;

    const i64 blocks = d.in_shape[0] * p.tiles;
    if (blocks == 0) return NOA_HIP_OK;
    if constexpr (std::is_same_v<C, float> && std::is_same_v<W, float> &&
                  (std::is_same_v<In, float2> || std::is_same_v<In, float>) &&
                  (std::is_same_v<Out, float2> || std::is_same_v<Out, float>)) {
        const int st = run_tiles<In, Out>(d, p, stream, err);
        if (st != NOT_TILED) return st;
    }
    if (blocks * 256 > MAX_LANES) { err = "too many slices for one launch"; return NOA_HIP_ERROR_UNSUPPORTED; }
    hipLaunchKernelGGL((rasterize_kernel<C, In, Out, W>), dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, p);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) { err = std::string("kernel launch failed: ") + hipGetErrorString(e); return NOA_HIP_ERROR_RUNTIME; }
    return NOA_HIP_OK;
}

template<class C>
int dispatch(const ProjectDesc& d, hipStream_t stream, std::string& err) {
    const int in = d.input.dtype, out = d.output.dtype;
    if (in == NOA_HIP_C32 && out == NOA_HIP_C32) return run<C, float2, float2, float>(d, stream, err);
    if (in == NOA_HIP_C32 && out == NOA_HIP_F32) return run<C, float2, float, float>(d, stream, err);
    if (in == NOA_HIP_F32 && out == NOA_HIP_F32) return run<C, float, float, float>(d, stream, err);
    if (in == NOA_HIP_C64 && out == NOA_HIP_C64) return run<C, double2, double2, double>(d, stream, err);
    if (in == NOA_HIP_C64 && out == NOA_HIP_F64) return run<C, double2, double, double>(d, stream, err);
    if (in == NOA_HIP_F64 && out == NOA_HIP_F64) return run<C, double, double, double>(d, stream, err);
    err = "rasterize: unsupported input/output value types";
    return NOA_HIP_ERROR_UNSUPPORTED;
}

} // namespace

int launch_rasterize(const ProjectDesc& d, hipStream_t stream, std::string& err) {
    return d.coord_f64 ? dispatch<double>(d, stream, err) : dispatch<float>(d, stream, err);
}

} // namespace noa_hip
