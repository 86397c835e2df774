// Per-pixel / per-column bodies of the voxel-driven backprojectors, shared by the plain
// kernels (fan2d.hip, cone3d.hip) and the persistent multi-job kernel (serve.hip).
//
// Both read sinograms staged with a zero border of kPadDet cells on every detector edge
// (2D: [A][D + 4]; 3D: [A][V + 4][U + 4]); the lower-tap detector coordinate is clamped into
// [-2, D] (resp. [-2, U], [-2, V]), so off-detector samples read zeros with no per-tap test and
// every pair load stays inside the staged array.
#pragma once

#include <type_traits>

#include "cmi_internal.hpp"

namespace cmi {

constexpr int kPadDet = 2; // zero border of staged sinograms and panels, in cells

// Per-angle tables: the bodies take the table pointer type as a template parameter. The plain
// kernels pass their `const __restrict__` arguments (scalar loads already). The serving kernels
// pass constant-address-space pointers: their tables come from job records in memory, and
// with generic pointers the compiler loads every entry per lane, since the volume stores of
// earlier tiles might alias; tables do not change during a launch.
using ctab = const __attribute__((address_space(4))) float *;
__device__ __forceinline__ ctab const_table(const void *p) { return (ctab)p; }
// Entry i of a table of float4.
__device__ __forceinline__ float4 table4(const float4 *__restrict__ t, int i) { return t[i]; }
__device__ __forceinline__ float4 table4(ctab t, int i) {
    return make_float4(t[4 * i], t[4 * i + 1], t[4 * i + 2], t[4 * i + 3]);
}

// Linear interpolation of a pair at weight f, FP32 arithmetic.
__device__ __forceinline__ float lerp_pair(const Pair &p, float f) {
    return fmaf(f, p.hi - p.lo, p.lo);
}

// ------------------------------------------------------------------------------------------
// Fan-beam backprojection of a 64 x NY pixel tile by a workgroup of four wavefronts: wavefront q
// takes the angles of quarter q, [A q / 4, A (q + 1) / 4), for all pixels of the tile, a thread
// one column of NY pixels, and the quarters' sums S_q meet in LDS as (S0 + S2) + (S1 + S3).
// Every path that backprojects a fan beam adds in that order, so a pixel's value does not depend
// on the path: k_bp2d and the serving kernel here, and k_bp2d_qt, where the quarters' order
// turns with the pixel (the sum is symmetric under a cyclic shift of the quarters).
// On gfx950 fma, add and mul of vector registers issue about 1.55 wavefront instructions per clock
// and CU; min / max / med3, floor, fract, conversions, shifted adds and any instruction that reads
// a scalar register 0.93, v_rcp_f32 0.48 (issue probe, eight wavefronts per SIMD). With
// several rows, a thread shares an angle's constants and its two products with x. Splitting the angles
// over the wavefronts keeps the number of wavefronts that a thread per pixel would have.

// Projection of one angle of a circular plan, tab[a] = (-sin, cos, DSD, DSO)
// (backward_2d.hpp:58-96): depth = DSO + (-sin x - cos y), magnification w = DSD / depth, cell
// coordinate w (cos x - sin y) / du + D/2. The sums are of rounded products (no contraction): a
// quarter turn of the pixel and the angle exchanges the two products of each and leaves their
// sum as it was, bit for bit.
template <int WPOW>
struct FanAngle {
    float4 m;
    float p1, q1;
    __device__ __forceinline__ FanAngle(float4 m_, float x, float px) : m(m_) {
#pragma clang fp contract(off)
        p1 = m.x * x;
        q1 = m.y * px;
    }
    template <class TAB>
    __device__ __forceinline__ FanAngle(TAB tab, int a, float x, float px)
        : FanAngle(table4(tab, a), x, px) {}
    // u: lower-tap cell coordinate (unclamped); wt: weight. px, py = x / du, y / du; c0 = D/2 - .5
    __device__ __forceinline__ void at(float y, float py, float c0, float &u, float &wt) const {
#pragma clang fp contract(off)
        const float depth = (p1 - m.y * y) + m.w;
        const float eta = q1 + m.x * py;
        const float w = m.z * __builtin_amdgcn_rcpf(depth);
        u = __builtin_fmaf(w, eta, c0);
        wt = WPOW == 2 ? w * w : w;
    }
};

// Projection of one ASTRA-like view, tab[3 a ..] (geometry2d.hpp bp_view): depth = n . x + n0,
// w = L / depth, cell coordinate w (e . x + e0) + c0, weight w^WPOW / |u|. px, py are unused.
template <int WPOW>
struct ViewAngle {
    float4 m0, m1;
    float idu, d, e;
    template <class TAB>
    __device__ __forceinline__ ViewAngle(TAB tab, int a, float x, float)
        : m0(table4(tab, 3 * a)), m1(table4(tab, 3 * a + 1)), idu(table4(tab, 3 * a + 2).x) {
        d = fmaf(m0.x, x, m0.z);
        e = fmaf(m1.x, x, m1.z);
    }
    __device__ __forceinline__ void at(float y, float, float, float &u, float &wt) const {
        const float w = m0.w * __builtin_amdgcn_rcpf(fmaf(m0.y, y, d));
        u = fmaf(w, fmaf(m1.y, y, e), m1.w);
        wt = (WPOW == 2 ? w * w : w) * idu;
    }
};

// acc[k] += sum over angles [a0, a1) for the pixels (x, y[k]). `R` covers [A][D + 4].
template <class SS, class ANGLE, int NY, class TAB>
__device__ __forceinline__ void bp2d_angles(rsrc_t R, TAB tab, int a0, int a1, int D, float x,
                                            float px, const float (&y)[NY], const float (&py)[NY],
                                            float c0, float (&acc)[NY]) {
    // angles whose loads are in flight together (one row: 4 took 55 us for 383 x 451 x 501 from views
    // in BF16, 8 take 51)
    constexpr int UA = NY == 1 ? 8 : 2;
    const int Dp = D + 2 * kPadDet;
    const float hi = (float)D;
    int row = a0 * Dp + kPadDet;
    auto some = [&](int a, auto count) {
        constexpr int N = decltype(count)::value;
        float wt[N][NY], al[N][NY];
        Pair p[N][NY];
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const ANGLE g(tab, a + j, x, px); // wave-uniform table entries: scalar loads
#pragma unroll
            for (int k = 0; k < NY; ++k) {
                float u;
                g.at(y[k], py[k], c0, u, wt[j][k]);
                u = __builtin_amdgcn_fmed3f(u, -2.0f, hi);
                al[j][k] = __builtin_amdgcn_fractf(u);
                p[j][k] = buf_pair<SS>(R, row + j * Dp + floor_i32(u), 0);
            }
        }
#pragma unroll
        for (int j = 0; j < N; ++j)
#pragma unroll
            for (int k = 0; k < NY; ++k)
                acc[k] = fmaf(lerp_pair(p[j][k], al[j][k]), wt[j][k], acc[k]);
    };
    int a = a0;
    for (; a + UA <= a1; a += UA, row += UA * Dp) some(a, std::integral_constant<int, UA>{});
    if (UA > 4 && a + 4 <= a1) {
        some(a, std::integral_constant<int, 4>{});
        a += 4, row += 4 * Dp;
    }
    for (; a < a1; ++a, row += Dp) some(a, std::integral_constant<int, 1>{});
}

// The tile's sums over all angles: wavefront q returns those of row q, q < NY (the others return
// 0). All 256 threads of the workgroup call it;
// ix, iy0 the thread's column and the tile's first row; `red` 4 NY 64 floats of LDS.
template <class SS, class ANGLE, int NY, class TAB>
__device__ __forceinline__ float bp2d_tile(rsrc_t R, TAB tab, int A, int D, int nx, int ny, int ix,
                                           int iy0, float sx, float sy, float ox, float oy,
                                           float inv_du, float half_d, float *red) {
    static_assert(NY <= 4, "a wavefront finishes one row");
    const float x = ((float)ix - (float)nx / 2.0f) * sx + ox + 0.5f;
    float y[NY], py[NY], acc[NY];
#pragma unroll
    for (int k = 0; k < NY; ++k) {
        y[k] = ((float)(iy0 + k) - (float)ny / 2.0f) * sy + oy + 0.5f;
        py[k] = y[k] * inv_du;
        acc[k] = 0.0f;
    }
    const int lane = threadIdx.x & 63, q = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int a0 = (int)((int64_t)A * q / 4), a1 = (int)((int64_t)A * (q + 1) / 4);
    // D/2 and the texel-centre shift of the lerp, exact
    bp2d_angles<SS, ANGLE, NY>(R, tab, a0, a1, D, x, x * inv_du, y, py, half_d - 0.5f, acc);
#pragma unroll
    for (int k = 0; k < NY; ++k) red[(q * NY + k) * 64 + lane] = acc[k];
    __syncthreads();
    if (q >= NY) return 0.0f;
    const float *r = red + q * 64 + lane;
    return (r[0] + r[2 * NY * 64]) + (r[NY * 64] + r[3 * NY * 64]);
}

// ------------------------------------------------------------------------------------------
// Cone-beam backprojection of a tile of voxels by a workgroup of 256 threads, a run of voxels per
// thread. M[a] is a 3x4 matrix over the centred voxel index h = (x - cx, y - cy, z - cz, 1) giving
// (U, V, W); (U/W, V/W) is the lower-tap panel coordinate, clamped to [-2, U] and [-2, V]. The
// sample is bilinear in the zero-bordered panel. MATCHED drops voxels behind the source (W <= 0);
// FDK weights by 1 / W^2.
//
// The angles' panel footprints are staged in LDS. Angles go in groups of kGroup: every wavefront
// computes the group's footprints from the tile's 8 corners (8 lanes per angle; U/W and V/W are
// linear-fractional, so over a box where W > 0 their extremes are at corners). Per angle the
// workgroup stages the footprint (rows of at most kFootW columns, at most kFootRows rows, from
// the zero-bordered panel) into LDS and the runs sample from there. An angle whose footprint does
// not fit (or with a corner with W <= 0) is sampled from global memory instead, with the same
// arithmetic, after the others.
//
// A sample's LDS address is two fma: byte strides and the slot's offset are held as FP32 numbers n
// 2^-149. Such a number's bit pattern is the integer n below 2^24, and multiples of 4 are exact below
// 2^26, so that products with the integral floors and their sums are exact (the panels' rows reach
// 2^16, at 304 bytes each) and the sum's bits are the address; fractions are p - floor(p). On
// gfx950 these issue at the full rate, where a conversion to an integer, its offset, the 24-bit
// product and v_fract_f32 each take almost two slots.
constexpr int kFootW = 64;                        // staged columns per row
// LDS row pitch: 16-byte rows, 12 banks further per row. A wavefront's 8 x 8 columns of voxels (x,
// z) then meet few conflicts in any direction of view (68 and 16 x 4 columns, whose u and v advance
// together at 45 degrees: a third of all LDS cycles).
constexpr int kFootCols = 76;
constexpr int kFootRows = 60;
constexpr int kFootFloats = kFootCols * kFootRows;
// addresses before the slot's offset: rows and columns of panels of up to 2^16 cells a side
static_assert(4ll * (kFootCols + 1) * (65536 + 2 * kPadDet) < 1ll << 26, "exact as n 2^-149");

// The staged footprint, one workgroup-shared array (18 KB) for every instantiation a kernel uses, so
// a kernel that dispatches between modes allocates it once.
static __shared__ __align__(16) float foot_lds[kFootFloats];

// Angles whose footprints one pass of a wavefront evaluates: 8 lanes (the tile's corners) each.
constexpr int kGroup = 8;

// i 2^-149 for |i| < 2^24, opaque in a vector register.
__device__ __forceinline__ float subnormal(int i) {
    float f = __int_as_float(i < 0 ? -i | (int)0x80000000 : i);
    asm("" : "+v"(f));
    return f;
}

// A staged footprint: the sample at the integral lower taps (iu, iv) lies at the LDS byte address
// fma(iv, row, fma(iu, col, ofs)), its pair on the next row kFootCols floats further.
struct Foot {
    float row, col, ofs; // byte strides and offset, times 2^-149
};

// The four taps of a bilinear sample: rows v and v + 1, columns u and u + 1.
struct Taps {
    Pair r0, r1;
};
__device__ __forceinline__ Taps foot_taps(unsigned at) {
    const auto *p = (const __attribute__((address_space(3))) float *)(uintptr_t)at;
    return {{p[0], p[1]}, {p[kFootCols], p[kFootCols + 1]}};
}
__device__ __forceinline__ float bilerp(const Taps &t, float fu, float fv) {
    const float r0 = lerp_pair(t.r0, fu), r1 = lerp_pair(t.r1, fu);
    return fmaf(fv, r1 - r0, r0);
}

// Runs every angle of a tile whose corners lie at (tx, ty, tz) and (tx + ex, ty + ey, tz + ez)
// (centred indices): from_foot(m, foot) with its footprint staged, then from_panel(m, o), o the
// element offset of the panel's cell (0, 0), for the angles whose footprint was not (a pass of its
// own: the two in one loop cost a copy of the runs' sums per angle). YINV: the U and W rows do not
// depend on y. All 256 threads of the workgroup call it together (lanes without voxels too).
template <class SS, bool YINV, class TAB, class F1, class F2>
__device__ __forceinline__ void bp3d_angles(rsrc_t R, TAB M, int A, int U, int V, float tx,
                                            float ty, float tz, float ex, float ey, float ez,
                                            F1 &&from_foot, F2 &&from_panel) {
    const int Up = U + 2 * kPadDet, Vp = V + 2 * kPadDet;
    const int panel = Up * Vp;
    const float ulim = (float)U, vlim = (float)V;
    const int tid = threadIdx.x;
    const int lane = tid & 63, k8 = lane >> 3, c8 = lane & 7;
    // the tile's corner this lane evaluates
    const float cx = (c8 & 1) ? tx + ex : tx;
    const float cy = (c8 & 2) ? ty + ey : ty;
    const float cz = (c8 & 4) ? tz + ez : tz;
    // The footprints of the angles from g0 on, lanes 8k .. 8k+7 for angle g0 + k: the slot's
    // padded-panel origin (su, sv) and row count. Returns bit 8k for the angles that fit.
    auto footprints = [&](int g0, int &su, int &sv, int &rows) -> uint64_t {
        float umin = 0.0f, umax = 0.0f, vmin = 0.0f, vmax = 0.0f;
        int ok = 1;
        if (g0 + k8 < A) {
            const TAB m = M + 12 * (g0 + k8);
            float Uh = fmaf(m[2], cz, m[3]), Wh = fmaf(m[10], cz, m[11]);
            if (!YINV) {
                Uh = fmaf(m[1], cy, Uh);
                Wh = fmaf(m[9], cy, Wh);
            }
            Uh = fmaf(m[0], cx, Uh);
            Wh = fmaf(m[8], cx, Wh);
            const float Vh = fmaf(m[4], cx, fmaf(m[5], cy, fmaf(m[6], cz, m[7])));
            const float rw = __builtin_amdgcn_rcpf(Wh);
            umin = umax = __builtin_amdgcn_fmed3f(Uh * rw, -2.0f, ulim);
            vmin = vmax = __builtin_amdgcn_fmed3f(Vh * rw, -2.0f, vlim);
            ok = Wh > 0.0f ? 1 : 0;
        }
#pragma unroll
        for (int off = 1; off < 8; off <<= 1) {
            umin = fminf(umin, __shfl_xor(umin, off, 64));
            umax = fmaxf(umax, __shfl_xor(umax, off, 64));
            vmin = fminf(vmin, __shfl_xor(vmin, off, 64));
            vmax = fmaxf(vmax, __shfl_xor(vmax, off, 64));
            ok = min(ok, __shfl_xor(ok, off, 64));
        }
        // Lower taps lie within [floor(min) - 1, floor(max) + 1] (one-texel margin for the
        // rounding of the samples' u and v against the corners') and the upper tap adds one more
        // row / column.
        const int ulo = floor_i32(umin) - 1 + kPadDet, uhi = floor_i32(umax) + 2 + kPadDet;
        const int vlo = floor_i32(vmin) - 1 + kPadDet, vhi = floor_i32(vmax) + 2 + kPadDet;
        su = max(ulo, 0);
        sv = max(vlo, 0);
        rows = min(vhi, Vp - 1) - sv + 1;
        return __ballot(ok && uhi - ulo + 1 <= kFootW && vhi - vlo + 1 <= kFootRows);
    };
    // Staging: thread tid copies quad tid % 16 of rows tid / 16 + 16 j. The first kAhead rows of
    // the next angle are loaded before the current one is sampled.
    constexpr int kAhead = 2;
    constexpr unsigned es = sizeof(typename SS::raw);
    const int qrow = tid >> 4, qcol = (tid & 15) << 2;
    float *const to = &foot_lds[qrow * kFootCols + qcol];
    const int lds0 = (int)(uintptr_t)(__attribute__((address_space(3))) float *)foot_lds;
    const float row = subnormal(4 * kFootCols), col = subnormal(4);
    bool missed = false;
    int su0 = 0, sv0 = 0, srows = 0; // of the group's angles, by lane
    uint64_t fit = 0;
    bool fits;
    int su, sv, rows;
    unsigned g; // byte offset of the thread's first quad
    RawQuad<SS> next[kAhead];
    // Loads rows that the footprint does not have too (not stored; beyond the stack they read 0).
    auto ahead = [&](int a) {
        if ((a & (kGroup - 1)) == 0) fit = footprints(a, su0, sv0, srows);
        const int c = 8 * (a & (kGroup - 1));
        fits = (fit >> c) & 1u;
        su = __builtin_amdgcn_readlane(su0, c);
        sv = __builtin_amdgcn_readlane(sv0, c);
        rows = __builtin_amdgcn_readlane(srows, c);
        g = (unsigned)(a * panel + (sv + qrow) * Up + su + qcol) * es;
#pragma unroll
        for (int j = 0; j < kAhead; ++j)
            next[j] = buf_raw_quad_at<SS>(R, (int)(g + 16u * j * Up * es));
    };
    auto store = [&](int j, const Quad &v) {
        *reinterpret_cast<float4 *>(to + 16 * j * kFootCols) =
            make_float4(v.v[0], v.v[1], v.v[2], v.v[3]);
    };
    ahead(0);
    // not unrolled: copies of the sampling code cost registers and instruction cache
#pragma unroll 1
    for (int a = 0; a < A; ++a) {
        const bool staged = fits;
        missed = missed || !staged;
        const int at0 = lds0 + 4 * ((kPadDet - sv) * kFootCols + (kPadDet - su));
        if (staged) {
            __syncthreads(); // the previous angle's samples are read
#pragma unroll
            for (int j = 0; j < kAhead; ++j)
                if (qrow + 16 * j < rows) store(j, to_quad<SS>(next[j]));
#pragma unroll 1
            for (int j = kAhead; qrow + 16 * j < rows; ++j)
                store(j, buf_quad_at<SS>(R, (int)(g + 16u * j * Up * es)));
        }
        if (a + 1 < A) ahead(a + 1);
        if (staged) {
            __syncthreads();
            from_foot(M + 12 * a, Foot{row, col, __builtin_amdgcn_ldexpf((float)at0, -149)});
        }
    }
    if (!missed) return;
    for (int g0 = 0; g0 < A; g0 += kGroup) {
        fit = footprints(g0, su0, sv0, srows);
#pragma unroll 1
        for (int c = 0; c < min(kGroup, A - g0); ++c)
            if (!((fit >> (8 * c)) & 1u))
                from_panel(M + 12 * (g0 + c), (g0 + c) * panel + kPadDet * Up + kPadDet);
    }
}

// A workgroup's tile: kTileX x kTileY x kTileZ voxels (x, y, z), a run of kRun y voxels per thread.
// YINV is for matrices whose U and W rows do not depend on y (M[a][1] == M[a][9] == 0: circular
// orbits about the y axis, panel turned at most about y): a run then shares its perspective divide,
// u tap, u weight and distance weight, and v advances by a constant step dv = M[a][5] / W, clamped
// fma(y, dv, V0 / W). Any other geometry has a divide per voxel, and U, V, W advance by the
// matrix's y column; half as many voxels there, since small volumes (128^3) leave wavefronts
// wanting.
constexpr int kTileX = 16, kTileY = 16;
template <bool YINV>
constexpr int kTileZ = YINV ? 16 : 8;
template <bool YINV>
constexpr int kRun = YINV ? 16 : 8;

// This thread's run in the tile: offset of its first voxel. A wavefront has 8 x 8 runs (x, z).
template <bool YINV>
__device__ __forceinline__ int3 tile_run() {
    const int l = threadIdx.x & 63, w = threadIdx.x >> 6;
    return make_int3((l & 7) + 8 * (w & 1), YINV ? 0 : 8 * (w >> 1),
                     (l >> 3) + (YINV ? 8 * (w >> 1) : 0));
}

// acc[y] += sum over the angles for the run of the voxels at centred index (hx, hy + y, hz);
// (tx, ty, tz) is that of the tile's first voxel. `R` covers [A][V + 4][U + 4]. The run's first
// `count` voxels lie in the volume (uniform over a wavefront); the general form leaves out batches
// past them (4 x 128 x 128 voxels, thin along y, x 60 views: 75 -> 62 us; gathering 61).
// Bound by LDS (two pair reads per voxel and angle, 8 clocks per wavefront and CU, and conflicts)
// and VALU issue alike. 384^3 x 768 views of 576^2 in half precision, YINV: 19.1 ms with integer
// addresses (17 VALU slots per voxel and angle instead of 13), pitch 68, 16 x 4 columns per
// wavefront and a footprint's loads waited for at once; 17.8 with FMA addresses; 16.2 now (LDS busy
// 91 % of the time, 11 % of that in conflicts; 1.3 VALU instructions a clock and CU).
// 128^3 x 180 views of 192^2, general: 420 us gathering from global memory (two pairs per voxel at
// about 18 clocks per gather and CU), 292 staged.
template <class SS, bool YINV, bool MATCHED, bool FDK, class TAB>
__device__ __forceinline__ void bp3d_run(rsrc_t R, TAB M, int A, int U, int V, float hx, float hy,
                                         float hz, float tx, float ty, float tz, int count,
                                         float (&acc)[kRun<YINV>]) {
    const float ulim = (float)U, vlim = (float)V;
    const int Up = U + 2 * kPadDet;
    const int sRow = Up * (int)sizeof(typename SS::raw);
    // at_column(iu) gives taps(iv), the taps between columns iu and iu + 1 and rows iv and iv + 1.
    // kBatch voxels' taps are read before the first is used.
    constexpr int kBatch = 4;
    // DROP: a voxel behind the source has no sample at all (a weight of 0 would let infinities and
    // NaN of the panel through). Staged tiles lie before the source.
    auto run = [&](TAB m, auto drop, auto &&at_column) {
        constexpr bool DROP = decltype(drop)::value;
        float Uh = fmaf(m[0], hx, fmaf(m[2], hz, m[3]));
        float Wh = fmaf(m[8], hx, fmaf(m[10], hz, m[11]));
        float Vh = fmaf(m[4], hx, fmaf(m[5], hy, fmaf(m[6], hz, m[7])));
        auto weight = [&](float rw) {
            const float w = FDK ? rw * rw : 1.0f;
            return MATCHED ? (Wh > 0.0f ? w : 0.0f) : w;
        };
        auto add = [&](int y, const Taps &t, float fu, float fv, float w) {
            float s = bilerp(t, fu, fv);
            if (DROP && MATCHED) s = w > 0.0f ? s : 0.0f;
            acc[y] = (MATCHED || FDK) ? fmaf(s, w, acc[y]) : acc[y] + s;
        };
        if constexpr (YINV) {
            const float rw = __builtin_amdgcn_rcpf(Wh);
            const float u = __builtin_amdgcn_fmed3f(Uh * rw, -2.0f, ulim);
            const float iu = floorf(u), fu = u - iu;
            const float v0 = Vh * rw, dv = m[5] * rw, w = weight(rw);
            auto taps = at_column(iu);
#pragma unroll
            for (int y = 0; y < kRun<YINV>; y += kBatch) {
                float fv[kBatch];
                Taps t[kBatch];
#pragma unroll
                for (int k = 0; k < kBatch; ++k) {
                    const float v =
                        __builtin_amdgcn_fmed3f(fmaf((float)(y + k), dv, v0), -2.0f, vlim);
                    const float iv = floorf(v);
                    fv[k] = v - iv;
                    t[k] = taps(iv);
                }
#pragma unroll
                for (int k = 0; k < kBatch; ++k) add(y + k, t[k], fu, fv[k], w);
            }
        } else {
            Uh = fmaf(m[1], hy, Uh);
            Wh = fmaf(m[9], hy, Wh);
            float dU = m[1], dV = m[5], dW = m[9];
            asm("" : "+v"(dU), "+v"(dV), "+v"(dW)); // in vector registers
#pragma unroll
            for (int y = 0; y < kRun<YINV>; y += kBatch) {
                if (y >= count) break;
                float fu[kBatch], fv[kBatch], w[kBatch];
                Taps t[kBatch];
#pragma unroll
                for (int k = 0; k < kBatch; ++k) {
                    const float rw = __builtin_amdgcn_rcpf(Wh);
                    const float u = __builtin_amdgcn_fmed3f(Uh * rw, -2.0f, ulim);
                    const float v = __builtin_amdgcn_fmed3f(Vh * rw, -2.0f, vlim);
                    const float iu = floorf(u), iv = floorf(v);
                    fu[k] = u - iu;
                    fv[k] = v - iv;
                    w[k] = weight(rw);
                    t[k] = at_column(iu)(iv);
                    Uh += dU;
                    Vh += dV;
                    Wh += dW;
                }
#pragma unroll
                for (int k = 0; k < kBatch; ++k) add(y + k, t[k], fu[k], fv[k], w[k]);
            }
        }
    };
    bp3d_angles<SS, YINV>(
        R, M, A, U, V, tx, ty, tz, (float)(kTileX - 1), (float)(kTileY - 1),
        (float)(kTileZ<YINV> - 1),
        [&](TAB m, const Foot &f) {
            run(m, std::false_type{}, [&](float iu) {
                const float ofs = fmaf(iu, f.col, f.ofs);
                return [=](float iv) { return foot_taps(__float_as_uint(fmaf(iv, f.row, ofs))); };
            });
        },
        [&](TAB m, int base) {
            run(m, std::bool_constant<!YINV>{}, [&](float iu) {
                const int col = base + (int)iu;
                return [=](float iv) {
                    const int o = col + __mul24((int)iv, Up);
                    return Taps{buf_pair<SS>(R, o, 0), buf_pair<SS>(R, o, sRow)};
                };
            });
        });
}

} // namespace cmi
