// noa::xform::cubic_bspline_prefilter (src/noa/xform/CubicBSplinePrefilter.hpp:24): the recursive filter that
// turns samples into cubic B-spline coefficients, so that CUBIC_BSPLINE interpolation passes through the samples.
// Per line (core/CubicBSplinePrefilter.hpp:22-107): a causal recursion c[i] = L * s[i] + z * c[i-1] started from
// L * (s[0] + sum_{k < min(12, n)} z^(k+1) s[k]), then an anticausal one c[i] = z * (c[i+1] - c[i]) started from
// z / (z - 1) * c[n-1], with z = sqrt(3) - 2 and L = (1 - z)(1 - 1/z). Lines along x, then y, then z of the
// dimensions reordered to the output's rightmost order (cpu/CubicBSplinePrefilter.hpp:129-158).
//
// The recursion is sequential along a line, so one lane owns one line, with noa's expressions in noa's order
// (bit-identical to the CPU path). What differs from a lane-per-line loop over memory is the access pattern:
//  - lines along x that fit in LDS (up to 2,048 samples of 4 bytes) unless they are short and many, and along y and z
//    where the GPU holds all of them at once: a workgroup copies a tile of whole lines into LDS with all of its lanes, one lane per line runs both recursions
//    there, and the workgroup stores the tile: each pass reads and writes the array once, with all loads of a tile in
//    flight (bspline_tile_kernel);
//  - other lines along y and z: the 64 lanes of a wave own 64 neighbouring x, so every step of the recursion is one
//    coalesced 64-element access; steps are loaded in batches of 16, the next batch in flight while the current
//    one's dependent arithmetic runs;
//  - other lines along x (the contiguous axis): a wave owns 64 rows and walks them in 32-column chunks staged through
//    LDS, loaded and stored as whole row segments; the lanes then run their row's recursion out of LDS while the
//    next chunk's loads are in flight. In both, the anticausal half re-reads the causal half's output.
#include "common.hpp"
#include "kernels.hpp"

#include <algorithm>
#include <type_traits>

namespace noa_hip {

template<class T> __device__ __forceinline__ T vsub(T a, T b);
template<> __device__ __forceinline__ float vsub(float a, float b) { return a - b; }
template<> __device__ __forceinline__ double vsub(double a, double b) { return a - b; }
template<> __device__ __forceinline__ float2 vsub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
template<> __device__ __forceinline__ double2 vsub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }

// The pole and gain in the value's real precision, as constants of that precision (core/CubicBSplinePrefilter.hpp:
// 37-38); the anticausal factor z / (z - 1) (:104).
template<class R> struct BSplineConst {
    static constexpr R POLE = static_cast<R>(-0.2679491924311228);
    static constexpr R LAMBDA = (1 - POLE) * (1 - 1 / POLE);
    static constexpr R ANTI = POLE / (POLE - 1);
};

constexpr int UNROLL = 16;         // steps per batch in the column passes (two batches in flight)

template<class T>
struct LinesParams {
    const T* in; T* out;
    i64 in_s[3], out_s[3];         // strides of the three outer (line-index) dimensions
    i64 in_step, out_step;         // stride along the line
    i32 n1, n2;                    // sizes of the two inner outer dimensions (n2 fastest)
    i64 lines;                     // number of lines
    i32 n;                         // samples per line
};

// Rows: one wave per 64 lines, chunks of CHUNK columns through LDS. Block = one wave. The next chunk's global
// loads are issued into registers before the current chunk's recursion runs, so their latency overlaps it.
template<class T>
__global__ __launch_bounds__(64) void bspline_rows_kernel(const LinesParams<T> p) {
    using R = typename vt<T>::real;
    using K = BSplineConst<R>;
    // Columns per LDS chunk (64 columns of 4-byte values measured no faster at 256^3 and 512^3).
    constexpr i32 CHUNK = 32;
    constexpr i32 RPS = 64 / CHUNK;   // rows moved per load step
    __shared__ T tile[64][CHUNK + 1];
    __shared__ i64 ibase[64], obase[64];
    const i32 lane = static_cast<i32>(threadIdx.x);
    const i64 first = static_cast<i64>(blockIdx.x) * 64;
    const i32 nrows = static_cast<i32>(min<i64>(64, p.lines - first));
    {
        const i64 line = first + lane;
        i64 ib = 0, ob = 0;
        if (lane < nrows) {
            const i64 c = line % p.n2, t = line / p.n2;
            const i64 b = t % p.n1, a = t / p.n1;
            ib = a * p.in_s[0] + b * p.in_s[1] + c * p.in_s[2];
            ob = a * p.out_s[0] + b * p.out_s[1] + c * p.out_s[2];
        }
        ibase[lane] = ib;
        obase[lane] = ob;
    }
    __syncthreads();

    // Cooperative chunk copies: step k moves rows RPS*k .. RPS*k + RPS-1, CHUNK lanes along each row.
    const i32 col = lane % CHUNK, rsub = lane / CHUNK;
    // 16-byte values would need 128 registers for the prefetch: they are loaded straight into LDS instead.
    constexpr bool PREFETCH = sizeof(T) <= 8;
    T regs[PREFETCH ? CHUNK : 1];
    auto load_regs = [&](const T* src, const i64* base, i64 step, i32 c0, i32 w) {
#pragma unroll
        for (i32 k = 0; k < CHUNK; ++k) {
            const i32 r = RPS * k + rsub;
            if (col < w && r < nrows) regs[k] = src[base[r] + static_cast<i64>(c0 + col) * step];
        }
    };
    auto regs_to_tile = [&](i32 w) {
#pragma unroll
        for (i32 k = 0; k < CHUNK; ++k) {
            const i32 r = RPS * k + rsub;
            if (col < w && r < nrows) tile[r][col] = regs[k];
        }
    };
    auto load_tile = [&](const T* src, const i64* base, i64 step, i32 c0, i32 w) {
#pragma unroll
        for (i32 k = 0; k < CHUNK; ++k) {
            const i32 r = RPS * k + rsub;
            if (col < w && r < nrows) tile[r][col] = src[base[r] + static_cast<i64>(c0 + col) * step];
        }
    };
    auto store_chunk = [&](i32 c0, i32 w) {
#pragma unroll
        for (i32 k = 0; k < CHUNK; ++k) {
            const i32 r = RPS * k + rsub;
            if (col < w && r < nrows) p.out[obase[r] + static_cast<i64>(c0 + col) * p.out_step] = tile[r][col];
        }
    };

    const i32 n = p.n;
    const i32 last = ((n - 1) / CHUNK) * CHUNK;
    T prev = vzero<T>();
    // Causal pass (filter(), :60-73): the input's first chunk holds the min(12, n) samples of the initialisation.
    if constexpr (PREFETCH) load_regs(p.in, ibase, p.in_step, 0, min(CHUNK, n));
    for (i32 c0 = 0; c0 < n; c0 += CHUNK) {
        const i32 w = min(CHUNK, n - c0);
        if constexpr (PREFETCH) regs_to_tile(w);
        else load_tile(p.in, ibase, p.in_step, c0, w);
        __syncthreads();
        if constexpr (PREFETCH)
            if (c0 != last) load_regs(p.in, ibase, p.in_step, c0 + CHUNK, min(CHUNK, n - c0 - CHUNK));
        if (lane < nrows) {
            T* row = tile[lane];
            i32 j = 0;
            if (c0 == 0) {
                const i32 horizon = min(12, n);
                R zn = K::POLE;
                T sum = row[0];
                for (i32 k = 0; k < horizon; ++k) {
                    sum = vadd(sum, vmul(row[k], zn));
                    zn *= K::POLE;
                }
                prev = vmul(sum, K::LAMBDA);
                row[0] = prev;
                j = 1;
            }
            for (; j < w; ++j) {
                prev = vadd(vmul(row[j], K::LAMBDA), vmul(prev, K::POLE));
                row[j] = prev;
            }
        }
        __syncthreads();
        if (c0 != last) {
            store_chunk(c0, w);
            __syncthreads();
        }
    }
    // Anticausal pass (:75-79), from the last chunk, still in LDS, back to the first.
    for (i32 c0 = last; c0 >= 0; c0 -= CHUNK) {
        const i32 w = min(CHUNK, n - c0);
        if (c0 != last) {
            if constexpr (PREFETCH) regs_to_tile(w);
            else load_tile(p.out, obase, p.out_step, c0, w);
            __syncthreads();
        }
        if constexpr (PREFETCH)
            if (c0 != 0) load_regs(p.out, obase, p.out_step, c0 - CHUNK, CHUNK);
        if (lane < nrows) {
            T* row = tile[lane];
            i32 j = w - 1;
            if (c0 == last) {
                prev = vmul(row[j], K::ANTI);
                row[j] = prev;
                --j;
            }
            for (; j >= 0; --j) {
                prev = vmul(vsub(prev, row[j]), K::POLE);
                row[j] = prev;
            }
        }
        __syncthreads();
        store_chunk(c0, w);
        __syncthreads();
    }
}

// Columns and pages, in place on the output: one lane per line, neighbouring lanes on neighbouring x. Steps are
// loaded UNROLL at a time, the next batch issued before the current one's dependent arithmetic.
template<class T>
__global__ __launch_bounds__(256) void bspline_lines_kernel(const LinesParams<T> p) {
    using R = typename vt<T>::real;
    using K = BSplineConst<R>;
    const i64 line = static_cast<i64>(blockIdx.x) * 256 + threadIdx.x;
    if (line >= p.lines) return;
    const i64 c = line % p.n2, t = line / p.n2;
    const i64 b = t % p.n1, a = t / p.n1;
    T* const base = p.out + (a * p.out_s[0] + b * p.out_s[1] + c * p.out_s[2]);
    const i64 st = p.out_step;
    const i32 n = p.n;

    // Causal initialisation (:87-100) and recursion (:67-73).
    const i32 horizon = min(12, n);
    R zn = K::POLE;
    T sum = base[0];
    for (i32 k = 0; k < horizon; ++k) {
        sum = vadd(sum, vmul(base[k * st], zn));
        zn *= K::POLE;
    }
    T prev = vmul(sum, K::LAMBDA);
    base[0] = prev;
    T cur[UNROLL], nxt[UNROLL];
#pragma unroll
    for (i32 j = 0; j < UNROLL; ++j)
        if (1 + j < n) cur[j] = base[(1 + j) * st];
    for (i32 i = 1; i < n; i += UNROLL) {
        const i32 in = i + UNROLL;
#pragma unroll
        for (i32 j = 0; j < UNROLL; ++j)
            if (in + j < n) nxt[j] = base[(in + j) * st];
#pragma unroll
        for (i32 j = 0; j < UNROLL; ++j) {
            if (i + j < n) {
                prev = vadd(vmul(cur[j], K::LAMBDA), vmul(prev, K::POLE));
                base[(i + j) * st] = prev;
            }
        }
#pragma unroll
        for (i32 j = 0; j < UNROLL; ++j) cur[j] = nxt[j];
    }
    // Anticausal initialisation (:102-106) from c[n-1], which `prev` holds, and recursion (:75-79).
    prev = vmul(prev, K::ANTI);
    base[(n - 1) * st] = prev;
#pragma unroll
    for (i32 j = 0; j < UNROLL; ++j)
        if (n - 2 - j >= 0) cur[j] = base[(n - 2 - j) * st];
    for (i32 i = n - 2; i >= 0; i -= UNROLL) {
        const i32 in = i - UNROLL;
#pragma unroll
        for (i32 j = 0; j < UNROLL; ++j)
            if (in - j >= 0) nxt[j] = base[(in - j) * st];
#pragma unroll
        for (i32 j = 0; j < UNROLL; ++j) {
            if (i - j >= 0) {
                prev = vmul(vsub(prev, cur[j]), K::POLE);
                base[(i - j) * st] = prev;
            }
        }
#pragma unroll
        for (i32 j = 0; j < UNROLL; ++j) cur[j] = nxt[j];
    }
}

// Whole lines in LDS. ROWS: the lines run along the contiguous axis, and a wave copies stretches of one line at a time
// (LDS lines of an odd pitch, so that the lanes of the recursion read different banks); otherwise neighbouring lines are
// neighbours in memory, and a wave copies pieces of 128 bytes across them.
// Bound by the copies and by the latency of the recursion, which one half-wave per workgroup runs (about 16 clocks per
// sample and direction) while other workgroups of the CU copy. Rows of 181 x 300 x 275 f32 44 us (92 us in chunks,
// the lanes waiting for each), of 24 x 24 x 24, all three passes, 17 against 24 us. 64 bytes across the lines or 512 lanes
// were no faster.
constexpr i32 TILE_LANES = 256;
constexpr size_t TILE_LDS = 64 * 1024;

template<class T, bool ROWS, i32 WIDTH>
__global__ __launch_bounds__(TILE_LANES) void bspline_tile_kernel(const LinesParams<T> p, i32 tiles_c) {
    using R = typename vt<T>::real;
    using K = BSplineConst<R>;
    extern __shared__ __align__(16) unsigned char lds_bytes[];
    T* const lds = reinterpret_cast<T*>(lds_bytes);
    const i32 t = static_cast<i32>(threadIdx.x), n = p.n;
    // The tile's lines: WIDTH consecutive lines (ROWS), or the ones at c0 .. c0 + WIDTH - 1 of the fastest line index.
    i64 first;
    i32 lines;
    if constexpr (ROWS) {
        first = static_cast<i64>(blockIdx.x) * WIDTH;
        lines = static_cast<i32>(min<i64>(WIDTH, p.lines - first));
    } else {
        const i64 outer = blockIdx.x / static_cast<u32>(tiles_c);
        const i32 c0 = static_cast<i32>(blockIdx.x % static_cast<u32>(tiles_c)) * WIDTH;
        first = outer * p.n2 + c0;
        lines = min(WIDTH, p.n2 - c0);
    }
    auto base_of = [&](i64 line, const i64 (&s)[3]) {
        const i64 c = line % p.n2, u = line / p.n2;
        return u / p.n1 * s[0] + u % p.n1 * s[1] + c * s[2];
    };
    const i32 pitch = ROWS ? (n | 1) : 1;              // LDS strides of lines and of samples
    constexpr i32 step = ROWS ? 1 : WIDTH;
    // The copies: EACH elements per lane in flight. ROWS: a wave takes EACH lines and 64 samples of each at a time;
    // otherwise WIDTH lanes take one sample each of neighbouring lines.
    constexpr i32 EACH = ROWS ? WIDTH / (TILE_LANES / 64) : 8;
    static_assert(EACH >= 1, "whole lines per wave");
    const i32 wave = t >> 6, lane = t & 63;
    const i32 l = t % WIDTH, per = TILE_LANES / WIDTH;
    const i64 at_in = base_of(first, p.in_s), at_out = base_of(first, p.out_s);
    auto copy = [&](auto move) {
        if constexpr (ROWS) {
            for (i32 j = lane; j < n; j += 64) move(wave * EACH, j);
        } else {
            if (l < lines)
                for (i32 j = t / WIDTH; j < n; j += per * EACH) move(l, j);
        }
    };
    i64 row_in[ROWS ? EACH : 1], row_out[ROWS ? EACH : 1];
    if constexpr (ROWS) {
#pragma unroll
        for (i32 q = 0; q < EACH; ++q) {
            const i64 line = min(first + wave * EACH + q, p.lines - 1);
            row_in[q] = base_of(line, p.in_s);
            row_out[q] = base_of(line, p.out_s);
        }
    }
    copy([&](i32 at, i32 j) {
        T v[EACH];
#pragma unroll
        for (i32 q = 0; q < EACH; ++q) {
            if constexpr (ROWS) {
                if (at + q < lines) v[q] = p.in[row_in[q] + static_cast<i64>(j) * p.in_step];
            } else {
                if (j + q * per < n)
                    v[q] = p.in[at_in + static_cast<i64>(at) * p.in_s[2] + static_cast<i64>(j + q * per) * p.in_step];
            }
        }
#pragma unroll
        for (i32 q = 0; q < EACH; ++q) {
            if constexpr (ROWS) {
                if (at + q < lines) lds[(at + q) * pitch + j] = v[q];
            } else {
                if (j + q * per < n) lds[(j + q * per) * WIDTH + at] = v[q];
            }
        }
    });
    __syncthreads();
    if (t < lines) {
        T* const line = lds + t * pitch;
        constexpr i32 U = sizeof(T) <= 8 ? 16 : 8;
        // Causal initialisation (:87-100) and recursion (:67-73).
        const i32 horizon = min(12, n);
        R zn = K::POLE;
        T sum = line[0];
        for (i32 k = 0; k < horizon; ++k) {
            sum = vadd(sum, vmul(line[k * step], zn));
            zn *= K::POLE;
        }
        T prev = vmul(sum, K::LAMBDA);
        line[0] = prev;
        i32 j = 1;
        T cur[U], nxt[U];
        if (j + U <= n) {
#pragma unroll
            for (i32 k = 0; k < U; ++k) cur[k] = line[(j + k) * step];
        }
        for (; j + U <= n; j += U) {
            if (j + 2 * U <= n) {
#pragma unroll
                for (i32 k = 0; k < U; ++k) nxt[k] = line[(j + U + k) * step];
            }
#pragma unroll
            for (i32 k = 0; k < U; ++k) {
                prev = vadd(vmul(cur[k], K::LAMBDA), vmul(prev, K::POLE));
                line[(j + k) * step] = prev;
            }
#pragma unroll
            for (i32 k = 0; k < U; ++k) cur[k] = nxt[k];
        }
        for (; j < n; ++j) {
            prev = vadd(vmul(line[j * step], K::LAMBDA), vmul(prev, K::POLE));
            line[j * step] = prev;
        }
        // Anticausal initialisation (:102-106) from c[n-1], which `prev` holds, and recursion (:75-79).
        prev = vmul(prev, K::ANTI);
        line[(n - 1) * step] = prev;
        j = n - 2;
        if (j - U + 1 >= 0) {
#pragma unroll
            for (i32 k = 0; k < U; ++k) cur[k] = line[(j - k) * step];
        }
        for (; j - U + 1 >= 0; j -= U) {
            if (j - 2 * U + 1 >= 0) {
#pragma unroll
                for (i32 k = 0; k < U; ++k) nxt[k] = line[(j - U - k) * step];
            }
#pragma unroll
            for (i32 k = 0; k < U; ++k) {
                prev = vmul(vsub(prev, cur[k]), K::POLE);
                line[(j - k) * step] = prev;
            }
#pragma unroll
            for (i32 k = 0; k < U; ++k) cur[k] = nxt[k];
        }
        for (; j >= 0; --j) {
            prev = vmul(vsub(prev, line[j * step]), K::POLE);
            line[j * step] = prev;
        }
    }
    __syncthreads();
    copy([&](i32 at, i32 j) {
#pragma unroll
        for (i32 q = 0; q < EACH; ++q) {
            if constexpr (ROWS) {
                if (at + q < lines) p.out[row_out[q] + static_cast<i64>(j) * p.out_step] = lds[(at + q) * pitch + j];
            } else {
                if (j + q * per < n)
                    p.out[at_out + static_cast<i64>(at) * p.out_s[2] + static_cast<i64>(j + q * per) * p.out_step] =
                        lds[(j + q * per) * WIDTH + at];
            }
        }
    });
}

namespace {

// Whole-line tiles or, for rows, the chunks of bspline_rows_kernel. A tile costs its lines' index arithmetic (about 0.18 us
// per 1,000 lines once there are many), a row in chunks about 9 us for each chunk after the first, in which the next one is
// awaited; wider values make both wait for memory sooner. Chunks and tiles: 12,000 rows of 24 f32 9.0 and 7.5 us (c64 12.2
// and 12.3), 40,000 of 24 9.5 and 12.6 (they cross at about 20,000, for 2 samples at 15,000), of 33 18 and 12.5, of 128 40
// and 23; 100,000 of 64 22 and 29, of 128 44 and 42, of 200 81 and 60; 300,000 of 96 74 and 90, of 200 273 and 170. c32:
// 40,000 of 64 22 and 25, of 80 42 and 33; 100,000 of 128 75 and 87, of 200 198 and 165. c64: 40,000 of 32 17 and 29, of 33
// 41 and 29, 300,000 of 33 254 and 217.
bool tiles_for_rows(i64 lines, i64 n, size_t bytes) {
    const i64 waits = (n + 31) / 32 - 1;           // bspline_rows_kernel's chunks after the first
    if (lines <= (bytes == 16 ? 12288 : 16384)) return true;
    if (bytes == 16) return waits >= 1;
    return waits >= 4 || lines <= (bytes == 4 ? 50000 : 25000) * waits;
}

// Whole-line tiles across the contiguous axis, or a lane per line in memory: the tiles where the GPU (256 CUs, 160 KB of
// LDS and 2,048 lanes each) holds all of them at once, twice as many for long lines of 4-byte values (a lane's chain along
// the line then bounds the other form) and half of them for 16-byte ones. Lines in memory and tiles, with the tiles' number
// over the ones resident: f32 40,000 of 100 (0.8) 24 and 19 us, 63,000 of 37 (1.06) 3 us less than tiles, 16,000 of 800 (1.3)
// 115 and 92, 54,300 of 300 (1.6) 52 and 54, 16,000 of 1,000 (1.97) 144 and 115, 40,000 of 500 (2.5) 78 and 95, 24,000 of
// 2,000 (5.9) 285 and 544, 40,000 of 8 with 2 neighbours (9.8) 6 and 36; c32 10,000 of 400 (0.9) 71 and 39, 40,000 of 100
// (1.4) 26 and 29; c64 4,096 of 64 (0.3) 16 and 11, 16,000 of 40 (1.0) 13 and 18.
bool tiles_for_columns(i64 tiles, i64 n, size_t lds, size_t bytes) {
    const i64 resident = 256 * std::min<i64>(2048 / TILE_LANES, (160 * 1024) / static_cast<i64>(lds));
    if (bytes == 16) return 2 * tiles <= resident;
    return tiles <= (bytes == 4 && n >= 400 ? 2 : 1) * resident;
}

// Launch of one pass over `lines` lines of `n` samples; the outer dimensions are (lines / (n1 * n2), n1, n2).
template<class T>
int pass(bool rows, const T* in, const i64 in_s[3], i64 in_step, T* out, const i64 out_s[3], i64 out_step,
         i64 n0, i64 n1, i64 n2, i64 n, hipStream_t stream, std::string& err) {
    LinesParams<T> p{};
    p.in = in;
    p.out = out;
    for (int i = 0; i < 3; ++i) { p.in_s[i] = in_s[i]; p.out_s[i] = out_s[i]; }
    p.in_step = in_step;
    p.out_step = out_step;
    p.n1 = static_cast<i32>(n1);
    p.n2 = static_cast<i32>(n2);
    p.lines = n0 * n1 * n2;
    p.n = static_cast<i32>(n);
    if (p.lines == 0 || n == 0) return NOA_HIP_OK;
    // Tiles of 128 bytes across the lines (and at least as many lines of the rows), halved until a tile fits.
    i64 width = std::max<i64>(8, 128 / static_cast<i64>(sizeof(T)));
    const i64 pitch = rows ? (n | 1) : n;
    while (width > 8 && static_cast<size_t>(width * pitch) * sizeof(T) > TILE_LDS) width /= 2;
    const size_t lds = static_cast<size_t>(width * pitch) * sizeof(T);
    const i64 tiles_c = (n2 + width - 1) / width;
    const i64 tiles = rows ? (p.lines + width - 1) / width : n0 * n1 * tiles_c;
    if (lds <= TILE_LDS && tiles * TILE_LANES <= MAX_LANES &&
        (rows ? tiles_for_rows(p.lines, n, sizeof(T)) : tiles_for_columns(tiles, n, lds, sizeof(T)))) {
        auto launch = [&](auto w) {
            constexpr i32 W = decltype(w)::value;
            const dim3 grid(static_cast<u32>(tiles)), block(TILE_LANES);
            if (rows) hipLaunchKernelGGL((bspline_tile_kernel<T, true, W>), grid, block, lds, stream, p, 1);
            else hipLaunchKernelGGL((bspline_tile_kernel<T, false, W>), grid, block, lds, stream, p, static_cast<i32>(tiles_c));
        };
        if (width == 32) launch(std::integral_constant<i32, 32>{});
        else if (width == 16) launch(std::integral_constant<i32, 16>{});
        else launch(std::integral_constant<i32, 8>{});
    } else if (rows) {
        const i64 blocks = (p.lines + 63) / 64;
        hipLaunchKernelGGL((bspline_rows_kernel<T>), dim3(static_cast<u32>(blocks)), dim3(64), 0, stream, p);
    } else {
        const i64 blocks = (p.lines + 255) / 256;
        hipLaunchKernelGGL((bspline_lines_kernel<T>), dim3(static_cast<u32>(blocks)), dim3(256), 0, stream, p);
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) { err = std::string("kernel launch failed: ") + hipGetErrorString(e); return NOA_HIP_ERROR_RUNTIME; }
    return NOA_HIP_OK;
}

template<class T>
int run(const BSplineDesc& d, hipStream_t stream, std::string& err) {
    const T* in = static_cast<const T*>(d.input.data);
    T* out = static_cast<T*>(d.output.data);
    const i64* is = d.input.s;
    const i64* os = d.output.s;
    const i64* sh = d.shape;
    int status;
    // Rows (x), from the input; then columns (y) and pages (z), in place.
    const i64 ri[3] = {is[0], is[1], is[2]}, ro[3] = {os[0], os[1], os[2]};
    if ((status = pass<T>(true, in, ri, is[3], out, ro, os[3], sh[0], sh[1], sh[2], sh[3], stream, err))) return status;
    if (d.ndim >= 2) {
        const i64 co[3] = {os[0], os[1], os[3]};
        if ((status = pass<T>(false, out, co, os[2], out, co, os[2], sh[0], sh[1], sh[3], sh[2], stream, err))) return status;
    }
    if (d.ndim == 3) {
        const i64 po[3] = {os[0], os[2], os[3]};
        if ((status = pass<T>(false, out, po, os[1], out, po, os[1], sh[0], sh[2], sh[3], sh[1], stream, err))) return status;
    }
    return NOA_HIP_OK;
}

} // namespace

int launch_bspline_prefilter(const BSplineDesc& d, hipStream_t stream, std::string& err) {
    switch (d.output.dtype) {
        case NOA_HIP_F32: return run<float>(d, stream, err);
        case NOA_HIP_F64: return run<double>(d, stream, err);
        case NOA_HIP_C32: return run<float2>(d, stream, err);
        case NOA_HIP_C64: return run<double2>(d, stream, err);
        default: err = "cubic_bspline_prefilter: f32, f64, c32 or c64 arrays are expected"; return NOA_HIP_ERROR_UNSUPPORTED;
    }
}

} // namespace noa_hip
