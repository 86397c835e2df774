// 2D fan-beam projectors for gfx950: plan, per-ray table, forward ray march, voxel-driven
// backprojection and the matched (transposed) ray march.
//
// Data layout in HBM
//   plan tables  geo  [A] AngleGeom (FP64)       source / cell-0 vector / cell step
//                meta [A] float4                 (-sin, cos, DSD, DSO) for the backprojector
//                                                (plans from angles / DSO / DSD)
//                bpv  [A][3] float4              (n.x, n.y, n0, L), (e.x, e.y, e0, c0 - .5),
//                                                (1/|u|, 0, 0, 0): the backprojector's view
//                                                constants (plans from ASTRA-like views,
//                                                geometry2d.hpp bp_view)
//                ageo [A] float[6]               FP32 copy of geo for the adjoint's ray search
//                ev   [A*D] float4               (mx, my, vx, vy) per ray: m is the sample
//                                                j = N/2 in centred padded coordinates (see
//                                                below), v the step
//                ns   [A*D] float4               (world step length, N as int bits, -N/2, 0)
// Sample j of a ray sits at m + (j - N/2) v. Coordinates are "centred padded": padded-copy
// texel coordinate minus 0.5 (so floor() is the lower tap) minus the integer centre c0 of the
// padded copy. Anchoring at the ray's midpoint near the image centre keeps |m| small. The step
// is +-1 along the ray's dominant axis, so with jf = j - N/2, md the midpoint's dominant
// coordinate and s the step's sign, sample jf's dominant lower tap is the integer
// floor(md) + s jf with weight fract(md) (exact, one row per sample); its other coordinate is
// c = fma(jf, v_other, m_other) in FP32, lower tap floor(c), weight fract(c). The forward uses
// exactly this. The adjoint, its transpose up to rounding, takes a ray's samples in pairs on
// neighbouring rows: the one with the smaller column as here, the other at that column plus the
// slope.
//   per call     for each image b of the batch, one block of 2 * (nx+4) * (ny+4) elements:
//                pad  [ny+4][nx+4]               image with a 2-texel zero border
//                padT [nx+4][ny+4]               the same, transposed
//                (backprojection) sinogram with a 2-cell zero border: [B][A][D+4]
// The forward kernel reads the copy whose rows run along each ray's dominant axis, so the 64
// rays of a wavefront (adjacent detector cells of one angle) gather from a few cache lines per
// step whichever way the fan points, and the zero border replaces per-tap range checks.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <memory>
#include <type_traits>
#include <vector>

#include "bp_tiles.hpp"
#include "cmi_internal.hpp"
#include "geometry2d.hpp"

using namespace cmi;
using cmi::fan2d::AngleGeom;

struct cmi_plan2d {
    int device = 0;
    int vol_prec = CMI_F32, det_prec = CMI_F32;
    fan2d::Scalars g{};
    int64_t A = 0;
    double pitch = 0.0, cor = 0.0;
    uint32_t block_x = 64, block_y = 4;
    uint64_t total_samples = 0;
    uint64_t table_bytes = 0;
    AngleGeom *d_geo = nullptr;
    float4 *d_meta = nullptr;
    float4 *d_bpv = nullptr; // views (plans from vectors); d_meta is null then
    float *d_ageo = nullptr;
    float4 *d_ev = nullptr;
    float4 *d_ns = nullptr;
    bool quarter = false; // backprojection by quarter turns applies (k_bp2d_qt)
    // bounds on the backprojection's per-projection weight over the image (w / du, w^2 / du
    // for circular plans, with the view's 1 / |u| for plans from views); infinite when a
    // source lies inside the image's bounding box
    double bt_bound[2] = {INFINITY, INFINITY};
    // detector cells per pixel at the image's centre, mean over the projections (0 where a
    // projection's source lies inside the image's bounding box)
    double cells_per_pixel = 0.0;
};

namespace {

constexpr int kPad = 2;        // zero border of the staged image copies, in texels
constexpr int kMaxBlock = 256; // threads per workgroup every kernel here is compiled for
static_assert(kPad == kPadDet, "sinograms are staged with the backprojector's border");

// ---------------------------------------------------------------- ray table ----------------

__global__ __launch_bounds__(kMaxBlock) void k_ray_table(const AngleGeom *__restrict__ geo, int A,
                                                   int D, int64_t nx, int64_t ny, double sx,
                                                   double sy, float4 *__restrict__ ev,
                                                   float4 *__restrict__ ns,
                                                   unsigned long long *__restrict__ total) {
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const int a = blockIdx.y;
    unsigned long long n = 0;
    if (k < D && a < A) {
        const fan2d::Ray r = fan2d::setup_ray(geo[a], nx, ny, sx, sy, k);
        const size_t i = (size_t)a * D + k;
        const int64_t jm = r.n / 2;
        // texel coordinate -> centred padded coordinate
        const double cx = (double)(kPad - 0.5) - (double)((nx + 2 * kPad) / 2);
        const double cy = (double)(kPad - 0.5) - (double)((ny + 2 * kPad) / 2);
        const double mx = r.e[0] + (double)jm * r.v[0] + cx;
        const double my = r.e[1] + (double)jm * r.v[1] + cy;
        ev[i] = r.n ? make_float4((float)mx, (float)my, (float)r.v[0], (float)r.v[1])
                    : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        ns[i] = make_float4((float)r.scale, __int_as_float((int)r.n), (float)(-jm), 0.0f);
        n = (unsigned long long)r.n;
    }
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    if ((threadIdx.x & 63) == 0 && n) atomicAdd(total, n);
}

// ---------------------------------------------------------------- staging ------------------

// pad[py][px] = img[py-2][px-2] (0 outside) and padT[px][py] = pad[py][px], tile by tile.
template <class S>
__global__ __launch_bounds__(kMaxBlock) void k_stage2d(const typename S::raw *__restrict__ img,
                                                 typename S::raw *__restrict__ scratch, int nx,
                                                 int ny, int Wp, int Hp) {
    using raw = typename S::raw;
    __shared__ raw tile[32][33];
    const size_t b = blockIdx.z;
    img += b * (size_t)nx * ny;
    raw *pad = scratch + b * 2 * (size_t)Wp * Hp;
    raw *padT = pad + (size_t)Wp * Hp;
    const int px0 = blockIdx.x * 32, py0 = blockIdx.y * 32;
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int py = py0 + r, px = px0 + threadIdx.x;
        const int x = px - kPad, y = py - kPad;
        raw v = (raw)0.0f;
        if (x >= 0 && x < nx && y >= 0 && y < ny) v = img[(size_t)y * nx + x];
        if (px < Wp && py < Hp) pad[(size_t)py * Wp + px] = v;
        tile[r][threadIdx.x] = v;
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int px = px0 + r, py = py0 + threadIdx.x;
        if (px < Wp && py < Hp) padT[(size_t)px * Hp + py] = tile[threadIdx.x][r];
    }
}

// spad[b][a][c] = sino[b][a][c-2] for c in [2, D+2), 0 in the two border cells each side.
template <class S>
__global__ __launch_bounds__(kMaxBlock) void k_stage_sino2d(const typename S::raw *__restrict__ sino,
                                                      typename S::raw *__restrict__ spad, int D,
                                                      int A) {
    using raw = typename S::raw;
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    const int Dp = D + 2 * kPad;
    if (c >= Dp) return;
    const size_t row = (size_t)blockIdx.z * A + blockIdx.y;
    const int k = c - kPad;
    spad[row * Dp + c] = (k >= 0 && k < D) ? sino[row * D + k] : (raw)0.0f;
}

// ---------------------------------------------------------------- forward ------------------

// A lane's sums over its samples of one group. A sample with lower tap (row t, column i) and
// fraction fa along the row adds p0 += v(t, i), x0 += fa (v(t, i + 1) - v(t, i)), and p1, x1
// likewise on row t + 1. With u0 = p0 + x0 and u1 = p1 + x1 (the sums of the row-wise linear
// interpolants on the sample rows and on the rows below), the group's contribution is
// u0 + fb (u1 - u0), the sum of the samples' bilinear interpolants, because every sample of a
// ray has the same dominant weight fb.
struct BandSums {
    float p0 = 0.0f, x0 = 0.0f, p1 = 0.0f, x1 = 0.0f;
    // a0, a1: v(t, i), v(t, i + 1); b0, b1: v(t + 1, i), v(t + 1, i + 1)
    __device__ __forceinline__ void add(float a0, float a1, float b0, float b1, float fa) {
        p0 += a0;
        x0 = fmaf(fa, a1 - a0, x0);
        p1 += b0;
        x1 = fmaf(fa, b1 - b0, x1);
    }
    __device__ __forceinline__ float total(float fb) const {
        const float u0 = p0 + x0, u1 = p1 + x1;
        return fmaf(fb, u1 - u0, u0);
    }
};

// Row-synchronous march through LDS bands.
//
// A ray has one sample per dominant row: sample jf sits on row floor(md) + s jf. A workgroup
// holds adjacent detector cells of one angle and walks the dominant rows tau in increasing
// order: on row tau every lane whose dominant axis is the pass's takes its sample
// jf = s (tau - floor(md)), if jf lies in its range [q.z, q.z + N - 1], so all lanes read the
// same two rows. The rows come in bands (HalfBands, WholeBands): the workgroup stages a band's rows
// and the one below of the copy whose rows run along the dominant axis, over the
// columns its samples in the band touch, into LDS (rows of kPitch floats, filled with
// 4-element row loads) and interpolates from there. The last two cells of every row are kept
// at zero and are what lanes without a sample on a row read. A band wider than kPitch - 4
// columns is sampled from global memory instead, with the same arithmetic. Bands in which
// every lane of the workgroup has a sample on every row skip the per-sample range test.
//
// Staged cells outside the copy (band corners beyond its edge) hold whatever the range-checked
// loads return; no sample reads them, because every tap of a sample lies inside the copy's zero
// border.
//
// Summation: a lane adds its samples of a group of kGroup rows (absolute multiples) row by row
// into its BandSums, and the group's total into the ray's sum. Both paths add the same values in
// the same order, so a ray's sum does not depend on which rays share its workgroup (and so not on
// the launch shape).
//
// Bound by LDS (two pair reads of four clocks per wavefront, row and CU) and VALU issue (eight full
// and three half rate slots) alike. The staging plans are made a lane per band and the check that
// the rays stay beside the extreme ones once per pass (both were made per band, a third of all VALU
// instructions). A group comes as one band (19.5 KB, 16 wavefronts per CU) or as two (12.2 KB, 24
// wavefronts, twice the barriers): where the copies exceed an XCD's 4 MB of L2, so that loads take
// long, or kHalfGroups workgroups keep the GPU full for long, unless cells are fine and bands narrow.
// Calls with half and whole groups, us (bands of whole groups planned one by one: third): 1024^2 x
// 360 of 0.67 pixels, parallel rays 308, 452 (451), 1024^2 x 60 of 0.7 189, 204 (207), x 500 408, 427
// (433), in BF16 373, 391 (502), 1024^2 x 180 of 1.2 391, 428 (440); 16 images of 512^2 x 512 of 0.86
// 1573, 1684 (1721), of 0.67 1668, 1658 (1747), of 256^2 x 180 of 0.78 217, 225 (234); but 512^2 x 180
// of 0.5 110, 97 (98), 400^2 x 500 of 0.7 114, 106 (107), 512^2 x 500 of 1.2 210, 193 (191), 128^2 x
// 180 of 0.5 38, 33 (34), 200^2 x 180 of 0.7 in BF16 50, 47 (58); fine cells: 1024^2 x 180 of 0.3 310,
// 287 (308), 16 images of 512^2 x 512 of 0.5 2101, 2012 (2143).
// Groups of 15 rows, a band each, would be faster still (28 wavefronts), but round 16-bit images'
// sums more often.
constexpr uint64_t kHalfBytes = 4u << 20, kHalfGroups = 8192;
constexpr double kHalfCells = 1.6; // cells per pixel

constexpr int kGroup = 31; // rows of a summation group

// How a group's rows come: kPer bands of at most kMax rows, band bn from row(bn) on. A band and the
// row below it are staged as shares of share(lg) rows of 2^lg groups of threads, lg = 1 or 2 (kRows
// rows in all; those past the band's own are not read), the first kAhead of a share ahead.
struct HalfBands { // rows [0, 16) and [16, 31) of a group
    static constexpr int kPer = 2, kMax = 16, kRows = 20, kAhead = 5;
    __host__ __device__ static constexpr int share(int lg) { return lg == 1 ? 9 : 5; }
    __host__ __device__ static constexpr int row(int bn) {
        return (bn >> 1) * kGroup + (bn & 1) * kMax;
    }
};
struct WholeBands {
    static constexpr int kPer = 1, kMax = kGroup, kRows = 32, kAhead = 8;
    __host__ __device__ static constexpr int share(int lg) { return lg == 1 ? 16 : 8; }
    __host__ __device__ static constexpr int row(int bn) { return bn * kGroup; }
};
// LDS row pitch in floats: a multiple of 4 (16-byte row stores) and below 255, so that one
// address reaches a tap pair and the pair below it with two ds_read2_b32 immediate offsets.
// 152 (12.2 KB per half group, 19.5 KB per group) keeps thirteen or eight workgroups per CU: 128
// rays at up to about 0.95 or 0.9 texels per cell plus a band's slope and the tap margins fit; wider
// bands take the global path.
constexpr int kPitch = 152;
constexpr int kFwdRays = 128;          // rays (threads) per workgroup of the forward
constexpr int kMaxWaves = kFwdRays / 64;

__device__ __forceinline__ int wave_min(int v) {
    for (int off = 32; off > 0; off >>= 1) v = min(v, __shfl_xor(v, off, 64));
    return v;
}
__device__ __forceinline__ int wave_max(int v) {
    for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off, 64));
    return v;
}

// Workgroup-wide minima of N values (callers negate to take maxima); every thread of the
// workgroup calls it. `red` holds N ints per wavefront.
template <int N>
__device__ __forceinline__ void block_min(int (&v)[N], int *red, int nwaves) {
#pragma unroll
    for (int i = 0; i < N; ++i) v[i] = wave_min(v[i]);
    const int w = threadIdx.x >> 6;
    __syncthreads(); // previous readers of red are done
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int i = 0; i < N; ++i) red[w * N + i] = v[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < N; ++i) {
        int r = red[i];
        for (int k = 1; k < nwaves; ++k) r = min(r, red[k * N + i]);
        v[i] = __builtin_amdgcn_readfirstlane(r);
    }
}

__device__ __forceinline__ int floor_div(int a, int b) {
    return a >= 0 ? a / b : -((-a + b - 1) / b);
}

// Column of a ray at row t: sample jf = s (t - floor(md)), coordinate fma(jf, vc, mc). Used for the
// workgroup's extreme rays.
struct RayRow {
    float mc, vc;
    int r0, s;
};

template <bool YDOM>
__device__ __forceinline__ RayRow ray_row(float4 e) {
    const float md = YDOM ? e.y : e.x;
    return {YDOM ? e.x : e.y, YDOM ? e.z : e.w, (int)floorf(md), (YDOM ? e.w : e.z) > 0.0f ? 1 : -1};
}

__device__ __forceinline__ float ray_at(const RayRow &r, int t) {
    return fmaf((float)(r.s * (t - r.r0)), r.vc, r.mc);
}

// One pass (YDOM: rays whose dominant axis is y, row-major copy; else x, transposed copy).
// All threads of the workgroup call it together; returns the lane's sum, 0 if not in the pass.
//   rstride      elements per row of the copy (rows run along the dominant axis)
//   cofs         element offset of the copy's centre (centred coordinate 0, 0)
template <class SI, bool YDOM, class B>
__device__ __forceinline__ float march_band(rsrc_t R, const float4 *__restrict__ ev,
                                            const float4 *__restrict__ ns, bool valid,
                                            int rstride, int cofs, float *band, int *red,
                                            float4 *ext, int *flag, int nthreads,
                                            bool &others) {
    // the lane's ray (read again by each pass: kept, it costs eight registers)
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    const float4 e = valid ? *ev : zero;
    const float4 q = valid ? *ns : zero; // N = 0
    const int n = __float_as_int(q.y);
    // y dominant: row-major copy; else the transposed one
    const bool act = valid && (fabsf(e.w) == 1.0f) == YDOM && n > 0;
    const int nwaves = nthreads >> 6;
    const float md = YDOM ? e.y : e.x;   // dominant coordinate of the midpoint
    const float sd = YDOM ? e.w : e.z;   // dominant step, +-1
    const float mc = YDOM ? e.x : e.y;   // other coordinate of the midpoint
    const float vc = YDOM ? e.z : e.w;   // other step
    const int r0 = (int)floorf(md);
    const float fb = md - (float)r0;     // dominant weight of every sample (exact)
    const int s = sd > 0.0f ? 1 : -1;
    const float sf = (float)s;
    const int jlo = (int)q.z, jhi = jlo + n - 1;
    const int ta = s > 0 ? r0 + jlo : r0 - jhi; // first row of this lane
    const int tz = ta + n - 1;                  // last row
    const int k = (int)threadIdx.x;
    // pass-wide: rows [tr0, tr1], the latest first row and earliest last row of any lane, the
    // first and last active lane, whether every lane of the workgroup is in the pass, and whether
    // any is in the other
    int v[8] = {act ? ta : INT_MAX, act ? -tz : INT_MAX, act ? -ta : INT_MAX, act ? tz : INT_MAX,
                act ? k : INT_MAX,  act ? -k : INT_MAX,  act ? 1 : 0, !act && n > 0 ? 0 : 1};
    block_min<8>(v, red, nwaves);
    if (YDOM) others = v[7] == 0;
    if (v[0] == INT_MAX) return 0.0f; // no lane in this pass
    const int tr0 = v[0], tr1 = -v[1], ta_max = -v[2], tz_min = v[3];
    const bool all_in = v[6] == 1; // the minimum is 1 only if every lane is active
    // Rays of one angle come from one source and do not cross inside the image, so on any row
    // the columns of the workgroup's samples lie between those of its first and last active
    // rays (extended beyond their ends where needed). The pass checks this and samples from
    // global memory if a lane's do not.
    if (k == v[4]) ext[0] = e;
    if (k == -v[5]) ext[1] = e;
    __syncthreads();
    const unsigned span = (unsigned)(n - 1);
    // a lane has a sample on row t iff (unsigned)t - ta_m <= span_m (never for inactive lanes:
    // rows are far from the offset 2^31)
    const unsigned ta_m = act ? (unsigned)ta : 0x80000000u, span_m = act ? span : 0u;
    const int soff1 = rstride * (int)sizeof(typename SI::raw);
    // Every lane checks that its samples lie between the extreme rays, half a column of rounding
    // aside: a ray's column is affine in the row, so its first and last row decide. Bands are
    // staged with a column of margin on each side of the extreme rays.
    {
        bool out = false;
        if (act) {
            const RayRow e0 = ray_row<YDOM>(ext[0]), e1 = ray_row<YDOM>(ext[1]);
            auto beside = [&](int t) {
                const float c = fmaf((float)(s * (t - r0)), vc, mc);
                const float c0 = ray_at(e0, t), c1 = ray_at(e1, t);
                return !(c >= fminf(c0, c1) - 0.5f && c <= fmaxf(c0, c1) + 0.5f);
            };
            out = beside(ta) || beside(tz);
        }
        if (__builtin_amdgcn_ballot_w64(out) != 0 && (threadIdx.x & 63) == 0) *flag = 1;
    }
    __syncthreads();
    const bool inside = *flag == 0;
    float acc = 0.0f;
    // The staging plans of 64 bands at a time, a lane each: band first + lane needs columns c_lo ..
    // c_lo + W - 1 (its extreme rays' at its first and last row), Q quads. It is staged when W fits
    // a row and at least two groups of Q threads exist: G' = 2^lg groups, four if 4 Q <= nthreads
    // and two otherwise. Thread g Q + q (g < G') takes quad q of the K = B::share(lg) consecutive
    // rows g K .. g K + K - 1. A row then lies at a wave-uniform byte
    // offset from the thread's first row in the copy (one add; the offset stays in the load's
    // range-checked vector offset, so rows outside the copy read zeros) and at a constant one in
    // LDS (the store's immediate offset), and no row needs a bound. Quotients come from a float
    // reciprocal: exact, as every numerator is below 2^8 and every true quotient is at least
    // 1/(2 Q) > 2^-8 away from the next integer.
    int plan_lo = 0, plan_q = 0; // c_lo; Q + (lg << 8), 0 where the band is not staged
    float plan_rq = 0.0f;        // 1 / Q
    int first = INT_MIN / 2; // band of lane 0's plan
    struct Stage {
        int t0, c_lo, q;
        bool mine;
        int K, gb, lb;
    };
    constexpr int esz = (int)sizeof(typename SI::raw);
    const int rowb = __builtin_amdgcn_readfirstlane(rstride * esz); // bytes per row of the copy
    const float ftid = (float)threadIdx.x + 0.5f;
    auto plan_band = [&](int bn) {
        if (bn >= first + 64) {
            first = bn;
            const int mine = first + (int)(threadIdx.x & 63);
            const int lo = max(tr0, B::row(mine)), hi = min(tr1, B::row(mine + 1) - 1);
            const RayRow e0 = ray_row<YDOM>(ext[0]), e1 = ray_row<YDOM>(ext[1]);
            const float ca = ray_at(e0, lo), cb = ray_at(e0, hi);
            const float cc = ray_at(e1, lo), cd = ray_at(e1, hi);
            plan_lo = floor_i32(fminf(fminf(ca, cb), fminf(cc, cd))) - 1;
            const int c_hi = floor_i32(fmaxf(fmaxf(ca, cb), fmaxf(cc, cd))) + 1;
            const int W = c_hi + 2 - plan_lo; // columns [c_lo, c_hi + 1] hold the taps
            plan_q = 0;
            if (inside && lo <= hi && W <= kPitch - 4 && 2 * ((W + 3) >> 2) <= nthreads) {
                const int Q = (W + 3) >> 2; // 1 .. 37, at most nthreads / 2 (a multiple of 32)
                plan_rq = __builtin_amdgcn_rcpf((float)Q);
                const int G = (int)(((float)nthreads + 0.5f) * plan_rq); // >= 2
                plan_q = Q + (G >= 4 ? 512 : 256);
            }
        }
        const int i = bn - first;
        Stage P{};
        P.t0 = B::row(bn);
        P.q = __builtin_amdgcn_readlane(plan_q, i);
        if (P.q) {
            P.c_lo = __builtin_amdgcn_readlane(plan_lo, i);
            const float rq =
                __int_as_float(__builtin_amdgcn_readlane(__float_as_int(plan_rq), i));
            const int Q = P.q & 255, lg = P.q >> 8;
            P.K = B::share(lg);
            const int g = (int)(ftid * rq);
            P.mine = g < (1 << lg);
            const int q4 = ((int)threadIdx.x - g * Q) << 2;
            // byte offsets of this thread's quad in its first row: copy and LDS
            P.gb = ((P.t0 + g * P.K) * rstride + P.c_lo + cofs + q4) * esz;
            P.lb = (g * P.K * kPitch + q4) * 4;
        }
        return P;
    };
    char *const band_bytes = reinterpret_cast<char *>(band);
    auto store_row = [&](const Stage &P, int k, const RawQuad<SI> &raw) {
        const Quad v = to_quad<SI>(raw);
        *reinterpret_cast<float4 *>(band_bytes + P.lb + k * kPitch * 4) =
            make_float4(v.v[0], v.v[1], v.v[2], v.v[3]);
    };
    // The first kAhead rows of a thread's share of band i + 1 are loaded while band i is sampled
    // (registers `pre`), so their latency hides behind the sampling.
    constexpr int kAhead = B::kAhead;
    static_assert(B::share(2) == kAhead && B::share(1) <= 2 * kAhead, "rows of a share");
    static_assert(2 * B::share(1) > B::kMax && 4 * B::share(2) > B::kMax &&
                  2 * B::share(1) <= B::kRows && 4 * B::share(2) <= B::kRows, "shares fit");
    RawQuad<SI> pre[kAhead];
    auto load_ahead = [&](const Stage &P) {
        if (P.q && P.mine)
#pragma unroll
            for (int u = 0; u < kAhead; ++u) pre[u] = buf_raw_quad_at<SI>(R, P.gb + u * rowb);
    };
    int bn = B::kPer * floor_div(tr0, kGroup);
    if (B::kPer > 1 && B::row(bn + 1) <= tr0) ++bn;
    Stage P = plan_band(bn);
    load_ahead(P);
    BandSums sums;
    while (P.t0 <= tr1) {
        const bool use_lds = P.q != 0;
        if (use_lds) {
            if (P.mine) {
#pragma unroll
                for (int u = 0; u < kAhead; ++u) store_row(P, u, pre[u]);
                if (P.K > kAhead) {
                    constexpr int kRest = B::share(1) - kAhead;
                    RawQuad<SI> v[kRest];
#pragma unroll
                    for (int u = 0; u < kRest; ++u)
                        v[u] = buf_raw_quad_at<SI>(R, P.gb + (kAhead + u) * rowb);
#pragma unroll
                    for (int u = 0; u < kRest; ++u) store_row(P, kAhead + u, v[u]);
                }
            }
            __syncthreads();
        }
        ++bn;
        Stage N{};
        N.t0 = B::row(bn);
        if (N.t0 <= tr1) {
            N = plan_band(bn);
            load_ahead(N);
        }
        const int b_lo = max(tr0, P.t0), b_hi = min(tr1, N.t0 - 1);
        // whether every lane has a sample on every row [b_lo, b_hi]
        const bool full = all_in && ta_max <= b_lo && tz_min >= b_hi;
        float jf = (float)(s * (b_lo - r0));
        if (use_lds) {
            // float offset of the band's first row, column 0, held opaque in a scalar
            // register so that the compiler does not split a constant off every address
            int rofs = __builtin_amdgcn_readfirstlane((b_lo - P.t0) * kPitch - P.c_lo);
            asm("" : "+s"(rofs));
            const float *rowa = band + rofs;
            int t = b_lo;
            // up to four rows' taps are read before the first is used
            auto batch = [&](auto rows, auto &&address) {
                constexpr int N4 = decltype(rows)::value;
                float c[N4], x[N4][4];
#pragma unroll
                for (int u = 0; u < N4; ++u) {
                    c[u] = fmaf(u == 0 ? jf : jf + (float)u * sf, vc, mc);
                    const float *p = address(u, floor_i32(c[u]));
                    x[u][0] = p[0];
                    x[u][1] = p[1];
                    x[u][2] = p[kPitch];
                    x[u][3] = p[kPitch + 1];
                }
#pragma unroll
                for (int u = 0; u < N4; ++u)
                    sums.add(x[u][0], x[u][1], x[u][2], x[u][3], __builtin_amdgcn_fractf(c[u]));
                t += N4;
                jf += (float)N4 * sf;
                rowa += N4 * kPitch;
            };
            if (full) { // every lane has a sample on every row of the band
                auto at = [&](int u, int i) { return rowa + u * kPitch + i; };
#pragma unroll 1
                while (t + 3 <= b_hi) batch(std::integral_constant<int, 4>{}, at);
                if (t + 2 == b_hi) batch(std::integral_constant<int, 3>{}, at);
            }
            // Rows past the band's last and lanes without a sample read the zero cells of a
            // row, which add nothing.
            const int zc = P.c_lo + kPitch - 2;
#pragma unroll 1
            while (t <= b_hi)
                batch(std::integral_constant<int, 4>{}, [&](int u, int i) {
                    const bool row = t + u <= b_hi;
                    const bool in = row && (unsigned)(t + u) - ta_m <= span_m;
                    return (row ? rowa + u * kPitch : band - P.c_lo) + (in ? i : zc);
                });
        } else {
            // lanes without a sample on the row sample their nearest own sample and add zeros, and so
            // does every lane on rows past the band's last; four rows' taps are in flight. Sources
            // close to the image, 360 angles, row by row / so (and with every band checked by
            // itself, row by row): 256^2, 128 cells 113 / 73 (105) us; 1024^2, 256 cells 521 / 310
            // (523); 300 x 40 around the source 71 / 48 (67).
            const float jmin = (float)jlo, jmax = (float)(act ? jhi : jlo);
            for (int t = b_lo; t <= b_hi; t += 4, jf += 4.0f * sf) {
                float f[4];
                Pair a[4], b[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const float j =
                        __builtin_amdgcn_fmed3f(u == 0 ? jf : jf + (float)u * sf, jmin, jmax);
                    const float c = fmaf(j, vc, mc);
                    const int o = __mul24(r0 + s * (int)j, rstride) + floor_i32(c) + cofs;
                    a[u] = buf_pair<SI>(R, o, 0);     // row, columns i and i + 1
                    b[u] = buf_pair<SI>(R, o, soff1); // the row below
                    f[u] = __builtin_amdgcn_fractf(c);
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    if (t + u > b_hi || (unsigned)(t + u) - ta_m > span_m)
                        a[u] = b[u] = Pair{0.0f, 0.0f};
                    sums.add(a[u].lo, a[u].hi, b[u].lo, b[u].hi, f[u]);
                }
            }
        }
        if (bn % B::kPer == 0 || N.t0 > tr1) { // the group's last band
            acc += sums.total(fb);
            sums = BandSums{};
        }
        if (use_lds) __syncthreads(); // the band is read before the next is staged
        P = N;
    }
    return acc;
}

// One workgroup = nthreads <= kFwdRays adjacent detector cells of one angle, one thread per
// ray; LDS holds one band of B::kRows x kPitch floats.
// sino[b][a][k] = scale * sum_{j<N} bilinear(img, e + j v)   (forward_2d.hpp:63-78)
// Half groups: six wavefronts per SIMD (80 VGPRs, 40 bytes of scratch with FP32 images): 0.498 ms at
// 1024^2 x 1024, five 0.511. Whole groups: four, by their LDS.
template <class SI, class SS, class B>
__global__ __launch_bounds__(kFwdRays) __attribute__((amdgpu_waves_per_eu(6)))
void k_fwd2d(const typename SI::raw *__restrict__ scratch,
                                              int Wp, int Hp, const float4 *__restrict__ ev,
                                              const float4 *__restrict__ ns,
                                              typename SS::raw *__restrict__ sino, int D, int A) {
    // one LDS object with the band first, so that cell addresses need no base offset
    __shared__ struct {
        float band[B::kRows * kPitch];
        float4 ext[2];
        int red[8 * kMaxWaves];
        int flag[2]; // one per pass: no barrier follows a pass's read where nothing is staged
    } sh;
    float *band = sh.band;
    float4 *ext = sh.ext;
    int *red = sh.red;
    const int nthreads = blockDim.x;
    // The launch's linear workgroup index taken with angles fastest: consecutive workgroups
    // (dealt to the 8 XCDs in turn) hold the same cells at successive angles, so every XCD
    // gets every eighth angle of one cell block at a time, and workgroups resident together
    // march rays of similar length (0.593 -> 0.556 ms at 1024^2; cell blocks fastest, each
    // XCD a contiguous run: 0.635 ms).
    const unsigned gx = gridDim.x, gy = gridDim.y;
    const unsigned hw = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const int a = (int)(hw % gy);
    const int k = (int)((hw / gy) % gx) * nthreads + threadIdx.x;
    const size_t b = hw / (gx * gy);
    const bool valid = k < D;
    const size_t r = (size_t)a * D + k;
    const int one = Wp * Hp;
    const rsrc_t R = make_rsrc(scratch + b * 2 * (size_t)one, bytes_of<SI>(2 * (uint64_t)one));
    const int c0x = Wp / 2, c0y = Hp / 2;
    // the zero cells and the flags; ordered before their first use by the barriers at the start of
    // a pass
    for (int i = threadIdx.x; i < 2 * B::kRows; i += nthreads)
        band[(i >> 1) * kPitch + kPitch - 2 + (i & 1)] = 0.0f;
    if (threadIdx.x < 2) sh.flag[threadIdx.x] = 0;
    const float scale = valid ? ns[r].x : 0.0f;
    bool others = false; // whether a lane's ray is x dominant
    float acc = march_band<SI, true, B>(R, ev + r, ns + r, valid, Wp, c0y * Wp + c0x, band,
                                             red, ext, &sh.flag[0], nthreads, others);
    if (others)
        acc += march_band<SI, false, B>(R, ev + r, ns + r, valid, Hp, one + c0x * Hp + c0y,
                                             band, red, ext, &sh.flag[1], nthreads, others);
    if (valid) sino[b * (size_t)A * D + r] = from_f32<SS>(acc * scale);
}

// ---------------------------------------------------------------- backprojection ---------

// Quadrant tiles (times the batch) from which k_bp2d_qt backprojects a plan with quarter turns;
// fewer do not fill the GPU, and k_bp2d, whose workgroups own 64 pixels instead of 4 x 256, gives
// the same bits sooner. Calls of n^2 images with n angles, us (the host takes 22 of them): n = 256
// (64 tiles) 23 against 34, 384 (144 tiles) 41 against 47, 512 (256 tiles) 72 against 59, 1024
// (1024 tiles) 470 against 238.
constexpr uint64_t kQTMinTiles = 200;

// A workgroup of k_bp2d takes one row of 64 pixels, which gives the most workgroups, or two where a
// pixel has at least kRowsFine cells and that leaves kRowTiles workgroups (64 x 2 tiles times the
// batch): the gathers of a wavefront then span many lines, which two rows of one angle share. Both
// give the same bits. Calls with one, two and four rows, us: 1024^2 x 181, 5 cells a pixel 116, 99,
// 99 (a thread per pixel, rows together: 105), 3.3 cells 109, 99, 100 (104), 2 cells 93, 96, 98
// (94); 768^2 x 181, 5 cells 77, 64, 72 (76), 2 cells 56, 58, 66 (70); from views x 501, 4 cells a
// pixel: 1024^2 268, 248, 241, 384^2 (1152 tiles) 59, 53, 59, 256^2 (512 tiles) 32, 42, 48; 1 cell:
// 1024^2 237, 238, 236, 680^2 119, 124, 128, 448^2 58, 69, 70, 383 x 451 51, 56, 53 (four rows pay
// only where the workgroups happen to fill the CUs evenly).
constexpr double kRowsFine = 2.5;
constexpr uint64_t kRowTiles = 1024;

// A workgroup per 64 x NY pixel tile, all angles in one pass, a quarter of them per wavefront
// (backward_2d.hpp:31-99): vol[b][y][x] += f sum_a wt_a lerp(sino[b][a], u_a), ANGLE the plan's
// projection (bp_tiles.hpp: FanAngle, f = 1/du; ViewAngle, whose weight holds 1/|u_a|, f = 1).
// Bound by the gathers (64 lanes in about 16 clocks per CU) and VALU issue (15 to 18) alike.
// Against a thread per pixel for all angles: 256^2 x 256 41 -> 23 us a call, 320^2 x 320 48 -> 28,
// 1024^2 x 1024 unchanged; 383 x 451 x 501 BF16 from views (whose loop over the angles had one
// load in flight) 167 -> 51 us.
template <class SV, class SS, class ANGLE, int NY>
__global__ __launch_bounds__(kMaxBlock) void k_bp2d(typename SV::raw *__restrict__ vol,
                                                    const typename SS::raw *__restrict__ spad,
                                                    const float4 *__restrict__ tab, int nx,
                                                    int ny, int D, int A, float sx, float sy,
                                                    float ox, float oy, float inv_du,
                                                    float half_d, float f) {
    __shared__ float red[4 * NY * 64];
    const unsigned tx = (unsigned)(nx + 63) / 64; // tiles per row
    const int wv = threadIdx.x >> 6, iy0 = (int)(blockIdx.x / tx) * NY, iy = iy0 + wv;
    const int ix = (int)(blockIdx.x % tx) * 64 + (int)(threadIdx.x & 63);
    const size_t b = blockIdx.z;
    const uint32_t sino_elems = (uint32_t)A * (D + 2 * kPadDet);
    const rsrc_t R = make_rsrc(spad + b * sino_elems, bytes_of<SS>(sino_elems));
    const float acc = bp2d_tile<SS, ANGLE, NY>(R, tab, A, D, nx, ny, ix, iy0, sx, sy, ox, oy,
                                               inv_du, half_d, red);
    if (wv >= NY || ix >= nx || iy >= ny) return;
    const size_t i = b * (size_t)nx * ny + (size_t)iy * nx + ix;
    vol[i] = from_f32<SV>(to_f32<SV>(vol[i]) + acc * f);
}

// Backprojection by quarter turns, for square images (n even, unit pixels, no offset) whose
// angles come in quarter-turn quadruples (angle a + A/4 = angle a + pi/2, equal DSO and DSD):
// the pixel at world (y, -x) has at angle theta + pi/2 the depth xi + DSO and detector
// coordinate that the pixel (x, y) has at angle theta (with meta = (-sin, cos), xi = -sin x -
// cos y and eta = cos x - sin y turn into each other). So one thread evaluates the geometry of
// its pixel P = (x, y) once per angle a and adds its weighted
// sample of row a to P, of row a + A/4 to (y, -x), of row a + A/2 to (-x, -y) and of row
// a + 3A/4 to (-y, x): four pixels per geometry evaluation. In index terms, with h = n/2 and
// P = (ix, iy) in the quadrant [0, h)^2: (iy, n-1-ix), (n-1-ix, n-1-iy), (n-1-iy, ix).
// A workgroup owns a 16 x 16 tile of the quadrant. Per chunk of 8 angles, every wavefront
// projects the tile's corners (lanes 4j .. 4j+3 for angle j of the chunk), the four rows of each
// angle share that footprint (the four rotated tiles project alike), and the workgroup stages
// the four rows' footprint segments (64 cells) into LDS with 16-byte loads while the previous
// chunk is sampled from the other buffer. Samples read their tap pair from LDS at immediate
// offsets, one address per angle for all four rows. The plan checks the symmetry (in the FP32
// table too) and that every footprint fits a segment.
// Positions, weights and the order of the sums are those of the per-pixel path (bp_tiles.hpp:
// FanAngle, quarters of the angles), so the two agree bit for bit: the geometry of an angle is
// evaluated for P alone, and for the pixel turned k quarters the quarters of the angles come in
// the order k, k + 1, k + 2, k + 3 (mod 4), under which (S0 + S2) + (S1 + S3) does not change.
// Two halves of the workgroup (four wavefronts each) take quarters 0 and 2 and quarters 1 and 3
// of the angles for the same pixels, each with its own LDS buffers, and the second half's sums
// join through LDS. No pipe is full (VALU 1.16 of 1.55 instructions a clock and CU, LDS busy 0.7 of
// the time): per angle a scalar load, a reciprocal and an LDS read follow each other, so wavefronts
// count: one half alone with chunks of 16 angles (94 VGPRs, five wavefronts per SIMD; four for want
// of tiles at 1024^2) took 188 us at 1024^2 x 720 and 4.4 ms at 2048^2 x 4096 FP16, two halves with
// chunks of 8 (54 VGPRs, eight per SIMD) 174 us and 3.8 ms. The constants through vector loads,
// which would let their instructions issue at the full rate: 195 us and 4.7 ms. With a weight of
// w^2 per pixel and angle through k_bp2d, 2048^2 x 4096 FP16 took 7.3 ms.
constexpr int kQT = 16;              // tile edge, pixels
constexpr int kQHalf = kQT * kQT;    // threads per half
constexpr int kQThreads = 2 * kQHalf;
constexpr int kQChunk = 8;           // angles per staged chunk
constexpr int kQSeg = 64;            // staged cells per row
constexpr int kQBuf = kQChunk * 4 * kQSeg; // floats per chunk: [angle][row k][cell]
static_assert(kQHalf == 256 && kQBuf / 4 == 2 * kQHalf, "each thread stages two quads per chunk");

template <class SV, class SS, int WPOW>
__global__ __launch_bounds__(kQThreads) void k_bp2d_qt(typename SV::raw *__restrict__ vol,
                                                       const typename SS::raw *__restrict__ spad,
                                                       const float4 *__restrict__ meta, int n,
                                                       int D, int A, float inv_du, float half_d) {
    __shared__ float seg[2][2][kQBuf]; // [half][buffer]
    const int h = n / 2, Q = A / 4, Dp = D + 2 * kPadDet;
    const size_t b = blockIdx.z;
    const uint32_t sino_elems = (uint32_t)A * Dp;
    const rsrc_t R = make_rsrc(spad + b * sino_elems, bytes_of<SS>(sino_elems));
    const int hf = __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    const int t = threadIdx.x & (kQHalf - 1), lane = t & 63, wv = t >> 6;
    const int bx = blockIdx.x * kQT, by = blockIdx.y * kQT;
    const int ix = bx + (t & (kQT - 1)), iy = by + t / kQT;
    // lanes past the quadrant's edge follow its last pixel (their sums are dropped)
    const float x = (float)min(ix, h - 1) - (float)h + 0.5f;
    const float y = (float)min(iy, h - 1) - (float)h + 0.5f;
    const float px = x * inv_du, py = y * inv_du;
    const float hi = (float)D;
    const float c0 = half_d - 0.5f; // D/2 and the lerp's texel-centre shift
    // the tile corner (pixel centre) this lane projects for angle lane >> 2 of a chunk
    const int cxi = (lane & 1) ? min(bx + kQT - 1, h - 1) : bx;
    const int cyi = (lane & 2) ? min(by + kQT - 1, h - 1) : by;
    const float qx = (float)cxi - (float)h + 0.5f, qy = (float)cyi - (float)h + 0.5f;
    const float qpx = qx * inv_du, qpy = qy * inv_du;
    // staging share: quads q = t & 15 of row k = (t >> 4) & 3 of angles j = wv + 4 m, m < 2
    const int sq = t & 15, sk = (t >> 4) & 3;
    constexpr int esz = (int)sizeof(typename SS::raw);
    // the half's angle i, i in [0, 2 Q): quarter hf, then quarter hf + 2
    auto angle = [&](int i) { return i + (i < Q ? hf : hf + 1) * Q; };

    // Per chunk of angles from i = c on, lanes 4 j .. 4 j + 3 of every wavefront hold the first
    // padded cell of angle c + j's segment.
    auto footprint = [&](int c) -> int {
        const float4 m = meta[angle(min(c + ((lane >> 2) & (kQChunk - 1)), 2 * Q - 1))];
        const float depth = fmaf(m.x, qx, fmaf(-m.y, qy, m.w));
        const float eta = fmaf(m.y, qpx, m.x * qpy);
        const float w = m.z * __builtin_amdgcn_rcpf(depth);
        float v = __builtin_amdgcn_fmed3f(fmaf(w, eta, c0), -2.0f, hi);
        v = fminf(v, __shfl_xor(v, 1, 64));
        v = fminf(v, __shfl_xor(v, 2, 64));
        // one cell of margin for the corners' rounding; at most Dp - kQSeg, so that a segment
        // never runs past its row (the plan requires Dp >= kQSeg): no staged quad reads another
        // row or straddles the array's end
        return min(max(floor_i32(v) - 1 + kPadDet, 0), Dp - kQSeg);
    };
    auto load = [&](int c, int s0v, Quad (&qd)[2]) {
#pragma unroll
        for (int mm = 0; mm < 2; ++mm) {
            const int j = wv + 4 * mm;
            const int s0 = __builtin_amdgcn_readlane(s0v, 4 * j);
            // row of angle c + j (past the last angle: the last one's, loaded and unused),
            // turned by k quarters
            int r = angle(min(c + j, 2 * Q - 1)) + sk * Q;
            r = r >= A ? r - A : r;
            qd[mm] = buf_quad_at<SS>(R, (r * Dp + s0 + 4 * sq) * esz);
        }
    };
    auto store = [&](int buf, const Quad (&qd)[2]) {
#pragma unroll
        for (int mm = 0; mm < 2; ++mm) {
            const int j = wv + 4 * mm;
            *reinterpret_cast<float4 *>(&seg[hf][buf][(j * 4 + sk) * kQSeg + 4 * sq]) =
                make_float4(qd[mm].v[0], qd[mm].v[1], qd[mm].v[2], qd[mm].v[3]);
        }
    };
    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    // angle c + j of a chunk whose segments start at s0v
    auto sample = [&](int a, int j, int s0v, int bufofs) {
        const FanAngle<WPOW> g(meta, a, x, px); // wave-uniform: scalar loads
        float u, wt;
        g.at(y, py, c0, u, wt);
        u = __builtin_amdgcn_fmed3f(u, -2.0f, hi);
        const float al = __builtin_amdgcn_fractf(u);
        // byte offset of the angle's four rows less that of the segment's first cell, opaque in
        // a scalar register so that the rows stay immediate offsets of one address
        int jb = bufofs + j * 4 * kQSeg * 4 - 4 * (__builtin_amdgcn_readlane(s0v, 4 * j) - kPadDet);
        asm("" : "+s"(jb));
        const float *p = reinterpret_cast<const float *>(
            reinterpret_cast<const char *>(&seg[0][0][0]) + jb) + floor_i32(u);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float lo = p[k * kQSeg], up = p[k * kQSeg + 1];
            acc[k] = fmaf(fmaf(al, up - lo, lo), wt, acc[k]);
        }
    };
    float sum[4]; // the half's first quarter
    auto flush = [&]() {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            sum[k] = acc[k];
            acc[k] = 0.0f;
        }
    };
    Quad qd[2];
    int s0 = footprint(0);
    load(0, s0, qd);
    store(0, qd);
    __syncthreads();
    int cur = 0;
    for (int c = 0; c < 2 * Q; c += kQChunk, cur ^= 1) {
        // next chunk's loads in flight while this one is sampled
        const int cn = c + kQChunk;
        int sn = 0;
        if (cn < 2 * Q) {
            sn = footprint(cn);
            load(cn, sn, qd);
        }
        const int bufofs = (2 * hf + cur) * kQBuf * 4;
        if (cn <= Q || (c >= Q && cn <= 2 * Q)) { // inside a quarter
            const int a = angle(c);
#pragma unroll
            for (int j = 0; j < kQChunk; ++j) sample(a + j, j, s0, bufofs);
            if (cn == Q) flush();
        } else { // the quarter, or the last one, ends in the chunk
#pragma unroll
            for (int j = 0; j < kQChunk; ++j)
                if (c + j < 2 * Q) {
                    sample(angle(c + j), j, s0, bufofs);
                    if (c + j + 1 == Q) flush();
                }
        }
        if (cn < 2 * Q) store(cur ^ 1, qd);
        s0 = sn;
        __syncthreads();
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) sum[k] += acc[k];
    // the second half's sums join the first's ((S0 + S2) + (S1 + S3))
    if (hf)
#pragma unroll
        for (int k = 0; k < 4; ++k) (&seg[0][0][0])[k * kQHalf + t] = sum[k];
    __syncthreads();
    if (hf) return;
#pragma unroll
    for (int k = 0; k < 4; ++k) sum[k] += (&seg[0][0][0])[k * kQHalf + t];
    if (ix >= h || iy >= h) return;
    const int m1 = n - 1;
    const int px4[4] = {ix, iy, m1 - ix, m1 - iy};
    const int py4[4] = {iy, m1 - ix, m1 - iy, ix};
    typename SV::raw *vb = vol + b * (size_t)n * n;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const size_t i = (size_t)py4[k] * n + px4[k];
        vb[i] = from_f32<SV>(to_f32<SV>(vb[i]) + sum[k] * inv_du);
    }
}

// ---------------------------------------------------------------- adjoint ------------------

// Largest |y q.x| over the rays of each sinogram of a batch (q.x the ray's scale), in two
// steps: per sinogram b, kAdjParts workgroups each write the maximum of their grid-stride
// share to parts[b][*]; the adjoint reduces the kAdjParts values. Each image of a batch gets
// its own fixed-point unit, so that its result does not depend on the other images.
constexpr int kAdjParts = 256;

template <class SS>
__global__ __launch_bounds__(kMaxBlock) void k_adj2d_absmax(const typename SS::raw *__restrict__ sino,
                                                           const float4 *__restrict__ ns,
                                                           size_t rays, float *__restrict__ parts) {
    __shared__ float red[kMaxBlock / 64];
    const size_t b = blockIdx.y;
    sino += b * rays;
    parts += b * kAdjParts;
    float m = 0.0f;
    for (size_t i = (size_t)blockIdx.x * kMaxBlock + threadIdx.x; i < rays;
         i += (size_t)kAdjParts * kMaxBlock)
        m = fmaxf(m, fabsf(to_f32<SS>(sino[i]) * ns[i].x));
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kMaxBlock / 64; ++w) m = fmaxf(m, red[w]);
        parts[blockIdx.x] = m;
    }
}

__device__ __forceinline__ float adj2d_ymax(const float *__restrict__ parts) {
    float m = 0.0f;
    for (int i = threadIdx.x & 63; i < kAdjParts; i += 64) m = fmaxf(m, parts[i]);
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    return m;
}

// Matched adjoint (exact transpose of k_fwd2d), tile-driven. A workgroup owns a tile of texels, a
// group of angles and the rays of one dominant axis: kT2Rows rows across that axis (row: constant
// dominant coordinate) by kT2Cols columns along the other. Per angle, the candidate rays are those
// through the tile's footprint box (every texel's [t - .5, t + 1.5) box, in the ray search frame,
// projected onto the detector through its corners); the candidates of kAdjAngles angles form one
// list, and each thread takes one ray, keeps its parameters in registers and walks the rows on
// which its samples reach the tile. Angles all of whose candidates have the other dominant axis are
// left out; the tiles are wide since a ray of slope m leaves kT2Cols columns' width only for the
// share m kT2Rows / (kT2Cols + m kT2Rows) of its wavefront's rows (32 x 32 texels: lane use 0.62).
//
// A sample on row t (lower tap) with column c adds wl = y q.x (1 - frac md) times (1 - frac c,
// frac c) to row t and wh = y q.x frac md times the same to row t + 1 (fan2d.hip header). Row t so
// gets two terms of a ray, from its samples t - 1 and t, whose columns differ by the slope's |m|
// <= 1: three cells from the floor of the smaller one, p, on. With f = frac p, A the weight of the
// sample at p and B the other's (constant along the ray), g1 = min(f + |m|, 1) and g2 = max(f +
// |m| - 1, 0), they get A + B - b, b - B g2 and B g2, b = A f + B g1. The first sample's own row
// and the row after the last sample get one term each, apart.
// Terms are fixed point with integer LDS atomics: gfx950 runs them about 45 times faster than FP32
// LDS atomic adds, and integer sums are exact, so the result does not depend on the order of the
// additions. A, B and the terms are rounded to units of max|y q.x| / 2^19 (so |A + B| <= 2^19)
// and added to a 32-bit LDS cell: half the LDS traffic of 64-bit cells. A candidate ray adds at
// most one term to a cell, within 2^19 + 2, so a run of passes whose candidates number c keeps a
// cell within c (2^19 + 2): each thread moves its share of the cells into 64-bit registers and
// clears them before that could pass 2^31 - 1, which keeps every 32-bit sum exact. Each tile
// then adds its sums, in units of max|y q.x| / 2^30, to a 64-bit image with integer global atomics
// (the two axes' tiles and several angle groups share a texel), and k_adj2d_finish adds that image
// to the volume.
//
// Bound by LDS atomics (three per row and ray, two clocks per wavefront and CU each, and conflicts)
// and VALU issue (16 slots: 12 full, 4 half rate) alike: the LDS address is one FMA on subnormals
// (bp_tiles.hpp). 16 images of 512^2, 512 angles of 724 cells: 2.79 ms with four atomics per
// sample, 32 x 32 texels of both axes and the candidates' lists worked out on scalars; 2.01 with the
// rows and tiles above (VALU 1.2 instructions a clock and CU, LDS busy 61 %), 1.65 with the lists
// by lane (1.4 and 77 %, 46 % of that in conflicts). 24 x 96 texels: 1.66, 16 x 128: 1.71,
// 48 x 64: 1.83.
constexpr int kT2Rows = 32, kT2Cols = 64;
constexpr int kAdjAngles = 16; // angles whose candidate rays form one list: 4 lanes each
// Candidate order within an angle: phase p holds the rays p, p + kAdjPh, p + 2 kAdjPh, ..., so
// the lanes of a wavefront take rays kAdjPh cells apart and add to different LDS cells more
// often (padding the phases to equal size leaves holes, which are skipped). At the size above: kAdjPh 1
// (adjacent rays): 2.04 ms, 2: 1.65, 3: 1.72, 4: 1.91; bit-identical.
constexpr int kAdjPh = 2;
// Columns before and after the tile's that take what a ray adds next to it: rows are walked while
// p is in [-2, kT2Cols), rounded outwards by kT2Margin rows, and a row has cells floor(p) to + 2.
constexpr int kT2Side = 3;
constexpr float kT2Margin = 0.01f;
constexpr int kT2Pitch = kT2Cols + 2 * kT2Side + 1; // odd, in words
constexpr int kT2Cells = kT2Rows * kT2Pitch;
constexpr int kT2Own = (kT2Cells + kMaxBlock - 1) / kMaxBlock; // cells per thread
constexpr int kAdjBits = 19;        // a term's bound: 2^kAdjBits units
// candidates per 32-bit accumulation run
constexpr int kAdjBudget = (1 << (31 - kAdjBits)) - 2;
static_assert((int64_t)kAdjBudget * ((1 << kAdjBits) + 2) < (1ll << 31), "32-bit sums are exact");

// Angle groups per tile. A group costs its workgroup's clearing of the tile and up to 2048 64-bit
// atomics, so it is given kAdjSamples samples (a tile's share of the plan's) or, as long as that
// leaves fewer than kAdjFill workgroups, kAdjLeast; at most kAdjWorkgroups workgroups (with tiles of 32
// x 32 at 1024^2 a limit of 8192 gave 1.09 ms, 16384: 1.06, 24576: 1.04, 32768: 1.05). Calls with 1 /
// 3 / 6 / 12 / 24 / 60 / 180 groups, us, and what this rule takes (by the number of workgroups alone,
// and with tiles of 32 x 32 before: last two): 512^2 x 180 of 1.5 pixels 107 / 67 / 65 / 60 / 76 / 120 /
// 285, 16 (168, 209), of 0.15 616 / 630 / 787 / 642 / 565 / 478 / 519, 63 (497, 621); 200^2 x 60 of 0.6 78 /
// 46 / 38 / 34 / 34 / 37, 11 (43, 39); 64^2 x 360 of 0.6 391 / 204 / 126 / 72 / 46 / 35 / 35, 96 (45, 37);
// 5 images of 1 x 100 x 360 of 0.6 113 / 56 / 48 / 36 / 35 / 35 / 48 (75, 60); 1024^2 x 720 of 0.6 960 /
// 1057 / 1260 / 746 / 737 / 811 / 1235, 24 (739, 1210).
constexpr uint64_t kAdjSamples = 20000, kAdjLeast = 5000, kAdjFill = 4096, kAdjWorkgroups = 24576;
constexpr uint64_t kAdjRay = 16; // samples that a ray's set-up counts for

// Tiles of one image: those of the y-dominant rays, then those of the x-dominant ones.
__host__ __device__ inline unsigned adj2d_tiles(unsigned across, unsigned along) {
    return ((across + kT2Rows - 1) / kT2Rows) * ((along + kT2Cols - 1) / kT2Cols);
}

template <class SS>
__global__ __launch_bounds__(kMaxBlock) void k_adj2d_tile(unsigned long long *__restrict__ accimg,
                                                         const typename SS::raw *__restrict__ sino,
                                                         const float *__restrict__ ageo,
                                                         const float4 *__restrict__ ev,
                                                         const float4 *__restrict__ ns,
                                                         const float *__restrict__ parts, int nx,
                                                         int ny, int D, int A, int G) {
    // 32-bit cells while the angles are added; 64-bit cells (the same memory) for the totals.
    __shared__ union {
        unsigned int c32[kT2Cells];
        unsigned long long c64[kT2Cells];
    } sh;
    const int tid = threadIdx.x;
    long long own[kT2Own]; // this thread's cells tid + k kMaxBlock, moved out of LDS
#pragma unroll
    for (int k = 0; k < kT2Own; ++k) own[k] = 0;
    // cells -> registers, then clear (every thread calls it)
    auto drain = [&]() {
        lds_barrier();
#pragma unroll
        for (int k = 0; k < kT2Own; ++k) {
            const int i = tid + k * kMaxBlock;
            if (i < kT2Cells) {
                own[k] += (int)sh.c32[i];
                sh.c32[i] = 0u;
            }
        }
        __syncthreads();
    };
    int run = 0; // candidates added since the last drain
    // XCD-aware order: workgroups are dealt to the 8 XCDs in turn, and logical index li gives
    // each XCD a contiguous run of tiles of one angle group, whose candidate rays share L2 (with
    // square tiles 1.15 -> 1.08 ms at 1024^2; angle groups fastest: 1.17 ms)
    bool ydom;
    int g, d0, c0; // angle group; the tile's first texel along the dominant axis and along the other
    size_t b;
    {
        const unsigned gx = gridDim.x, nwg = gx * gridDim.z;
        const unsigned hw = blockIdx.x + gx * blockIdx.z;
        const unsigned n8 = nwg & ~7u;
        const unsigned li = hw < n8 ? (hw & 7u) * (n8 >> 3) + (hw >> 3) : hw;
        const unsigned per = gx * (unsigned)G;
        b = li / per;
        g = (int)(li % per / gx);
        unsigned t = li % gx;
        const unsigned ty = adj2d_tiles(ny, nx);
        ydom = t < ty;
        if (!ydom) t -= ty;
        const unsigned wide = (unsigned)((ydom ? nx : ny) + kT2Cols - 1) / kT2Cols;
        d0 = (int)(t / wide) * kT2Rows;
        c0 = (int)(t % wide) * kT2Cols;
    }
    const int a0 = (int)((int64_t)g * A / G), a1 = (int)((int64_t)(g + 1) * A / G);
    for (int i = tid; i < kT2Cells; i += kMaxBlock) sh.c32[i] = 0u;
    __syncthreads(); // the tile is clear before any wave adds to it
    const float ymax = adj2d_ymax(parts + b * kAdjParts);
    const float yscale = ymax > 0.0f ? (float)(1 << kAdjBits) / ymax : 0.0f;
    // the tile's first row and column in the ray table's centred padded frame
    const int fx = kPad - (nx + 2 * kPad) / 2, fy = kPad - (ny + 2 * kPad) / 2;
    const int rowf = d0 + (ydom ? fy : fx), colf = c0 + (ydom ? fx : fy);
    const float cmin = (float)(colf - 2), cmax = (float)(colf + kT2Cols);
    // byte strides and the address of row 0, column 0 of that frame, as subnormals
    const int lds0 = (int)(uintptr_t)(__attribute__((address_space(3))) unsigned *)sh.c32;
    const float col = subnormal(4), pitch = subnormal(4 * kT2Pitch);
    const float ofs = subnormal(lds0 + 4 * (kT2Side - colf));
    // Footprint box corner this lane projects. The box ends with the image: a corner beyond it could
    // lie behind the source.
    const int c1 = min(c0 + kT2Cols, ydom ? nx : ny), d1 = min(d0 + kT2Rows, ydom ? ny : nx);
    const float qc = (tid & 1) ? (float)c1 + 0.5f : (float)c0 - 0.5f;
    const float qd = (tid & 2) ? (float)d1 + 0.5f : (float)d0 - 0.5f;
    const float qx = ydom ? qc : qd, qy = ydom ? qd : qc;
    const typename SS::raw *sb = sino + b * (size_t)A * D;
    // kAdjAngles angles at a time: their candidate rays form one list, one ray per thread
    for (int ag = a0; ag < a1; ag += kAdjAngles) {
        const int na = min(kAdjAngles, a1 - ag);
        // candidate range per angle: lanes 4 s .. 4 s + 3 of every wavefront project the four
        // corners of the footprint box for angle ag + s
        const int slot = (tid & 63) >> 2;
        float kmin = 0.0f, kmax = 0.0f, ox = 0.0f, oy = 0.0f, ux = 0.0f, uy = 0.0f;
        if (slot < na) {
            const float *gp = ageo + 6 * (ag + slot);
            const float wx = qx - gp[0], wy = qy - gp[1];
            ox = gp[2], oy = gp[3], ux = gp[4], uy = gp[5];
            const float depth = wx * uy - wy * ux;
            kmin = kmax = -(wx * oy - wy * ox) / depth;
            // a corner that is not in front of the source bounds nothing
            if (!(depth * (ox * uy - oy * ux) > 0.0f)) kmin = -1e9f, kmax = 1e9f;
        }
        for (int off = 1; off < 4; off <<= 1) {
            kmin = fminf(kmin, __shfl_xor(kmin, off, 64));
            kmax = fmaxf(kmax, __shfl_xor(kmax, off, 64));
        }
        // Both end rays clearly closer to the other axis, and to the same end of it: so are all
        // rays between them.
        bool other;
        {
            const float lo = fmaxf(kmin - 0.01f, 0.0f), hi = fminf(kmax + 0.01f, (float)(D - 1));
            const float x0 = fmaf(lo - 1.0f, ux, ox), y0 = fmaf(lo - 1.0f, uy, oy);
            const float x1 = fmaf(hi + 1.0f, ux, ox), y1 = fmaf(hi + 1.0f, uy, oy);
            const float m0 = ydom ? x0 : y0, n0 = ydom ? y0 : x0;
            const float m1 = ydom ? x1 : y1, n1 = ydom ? y1 : x1;
            other = fabsf(m0) > 1.001f * fabsf(n0) && fabsf(m1) > 1.001f * fabsf(n1) &&
                    (m0 > 0.0f) == (m1 > 0.0f);
        }
        // By lane: the slot's angle's first candidate and their number (an angle whose box misses
        // the detector has none), the padded numbers' sum up to the slot
        int kfirst = 0, count = 0;
        if (slot < na && !other && kmax >= -1.0f && kmin <= (float)D) {
            kfirst = max((int)floorf(kmin - 0.01f), 0);
            count = max(min((int)ceilf(kmax + 0.01f), D - 1) - kfirst + 1, 0);
        }
        int upto = kAdjPh * ((count + kAdjPh - 1) / kAdjPh);
        const int padded = upto;
#pragma unroll
        for (int off = 4; off < 64; off <<= 1) {
            const int v = __shfl_up(upto, off, 64);
            upto += (tid & 63) >= off ? v : 0;
        }
        const int total = __builtin_amdgcn_readlane(upto, 63);
        const int start = upto - padded;
        int q0 = 0; // the last angle with start <= the wavefront's first ray
        // one candidate ray per thread, its parameters in registers; `total` and the pass
        // sizes are the same for the whole workgroup
        for (int base = 0; base < total; base += kMaxBlock) {
            const int pass = min(kMaxBlock, total - base);
            if (run + pass > kAdjBudget) {
                drain();
                run = 0;
            }
            run += pass;
            const int ri = base + tid;
            const int wave0 = __builtin_amdgcn_readfirstlane(base + (tid & ~63));
            if (wave0 >= total) continue;
            while (q0 + 1 < kAdjAngles && __builtin_amdgcn_readlane(start, 4 * (q0 + 1)) <= wave0)
                ++q0;
            int q = q0, pp = ri - __builtin_amdgcn_readlane(start, 4 * q0);
            int k0 = __builtin_amdgcn_readlane(kfirst, 4 * q0);
            int cnt = __builtin_amdgcn_readlane(count, 4 * q0);
            for (int u = q0 + 1; u < kAdjAngles; ++u) {
                const int from = __builtin_amdgcn_readlane(start, 4 * u);
                if (from >= wave0 + 64) break;
                const int ku = __builtin_amdgcn_readlane(kfirst, 4 * u);
                const int cu = __builtin_amdgcn_readlane(count, 4 * u);
                if (ri >= from) q = u, pp = ri - from, k0 = ku, cnt = cu;
            }
            const int pm = (cnt + kAdjPh - 1) / kAdjPh;
            int ph = 0;
#pragma unroll
            for (int u = 1; u < kAdjPh; ++u)
                if (pp >= pm) ph = u, pp -= pm;
            const int rl = pp * kAdjPh + ph;
            if (rl >= cnt) continue;
            const size_t r = (size_t)(ag + q) * D + k0 + rl;
            const float4 qn = ns[r];
            const float4 e = ev[r];
            const int n = __float_as_int(qn.y);
            const float yv = to_f32<SS>(sb[r]) * qn.x * yscale; // |yv| <= 2^kAdjBits
            if (n <= 0 || yv == 0.0f || (fabsf(e.w) == 1.0f) != ydom) continue;
            const float md = ydom ? e.y : e.x, sd = ydom ? e.w : e.z;
            const float mc = ydom ? e.x : e.y, vc = ydom ? e.z : e.w;
            const float f0 = floorf(md), fb = md - f0;
            const float wl = yv * (1.0f - fb), wh = yv * fb; // rows pd, pd + 1
            const int r0 = (int)f0, jlo = (int)qn.z;
            // the ray's samples are on the tile's rows (lower tap) first to first + n - 1; sample
            // `row` has step s (row + rowf - r0) and column fma(that, vc, mc)
            const float slope = sd > 0.0f ? vc : -vc; // of the column per row
            const int first = (sd > 0.0f ? r0 + jlo : r0 - (jlo + n - 1)) - rowf;
            const float m = fabsf(vc);
            // p = fma(k, slope, mc) on row k - kd
            const bool up = slope >= 0.0f;
            const int kd = rowf - r0 - (up ? 1 : 0);
            // rows with both terms whose cells reach the tile. Below a slope of 2^-21 a ray moves
            // less than a quarter of a column over any image (at most 2^20 rows): it is walked at
            // that slope, rounded outwards by all of that.
            constexpr float flat = 0x1p-21f;
            const float margin = m < flat ? 0.25f / flat : kT2Margin;
            const float inv = __builtin_amdgcn_rcpf(up ? fmaxf(m, flat) : fminf(-m, -flat));
            const float e0 = (cmin - mc) * inv, e1 = (cmax - mc) * inv;
            const float klo = fminf(e0, e1) - margin, khi = fmaxf(e0, e1) + margin;
            const int rlo = max(max(first + 1, 0), (int)ceilf(fmaxf(klo, -1e9f)) - kd);
            const int rhi = min(min(first + n - 1, kT2Rows - 1), (int)floorf(fminf(khi, 1e9f)) - kd);
            if (rlo <= rhi) {
                const float wb = up ? wl : wh, wa = up ? wh : wl;
                const int all = round_i32(yv);
                const float m1 = m - 1.0f;
                float k = (float)(rlo + kd);
                float at0 = fmaf((float)rlo, pitch, ofs);
                const float end = fmaf((float)rhi, pitch, ofs);
                do {
                    const float p = fmaf(k, slope, mc);
                    const float fl = floorf(p), f = p - fl;
                    const float g1 = __builtin_amdgcn_fmed3f(f + m, 0.0f, 1.0f);
                    const float g2 = __builtin_amdgcn_fmed3f(f + m1, 0.0f, 1.0f);
                    const int x2 = round_i32(wb * g2);
                    const int b2 = round_i32(fmaf(wb, g1, wa * f));
                    auto *const at = (__attribute__((address_space(3))) unsigned *)(uintptr_t)
                        __float_as_uint(fmaf(fl, col, at0));
                    lds_add(at, (unsigned)(all - b2));
                    lds_add(at + 1, (unsigned)(b2 - x2));
                    lds_add(at + 2, (unsigned)x2);
                    k += 1.0f;
                    at0 += pitch;
                } while (at0 <= end);
            }
            // rows with one term
            auto one = [&](int row, int sample, float w) {
                if ((unsigned)row >= (unsigned)kT2Rows) return;
                const float c = fmaf((float)(sample + rowf - r0), slope, mc);
                const float fl = floorf(c);
                if (!(fl >= cmin && fl <= cmax)) return;
                const int x1 = round_i32(w * (c - fl));
                unsigned *const at = &sh.c32[row * kT2Pitch + kT2Side + ((int)fl - colf)];
                atomicAdd(at, (unsigned)(round_i32(w) - x1));
                atomicAdd(at + 1, (unsigned)x1);
            };
            one(first, first, wl);
            one(first + n, first + n - 1, wh);
        }
    }
    drain();
    // totals in units of max|y q.x| / 2^30
#pragma unroll
    for (int k = 0; k < kT2Own; ++k) {
        const int i = tid + k * kMaxBlock;
        if (i < kT2Cells) sh.c64[i] = (unsigned long long)(own[k] * (1ll << (30 - kAdjBits)));
    }
    __syncthreads();
    unsigned long long *out = accimg + b * (size_t)nx * ny;
    for (int i = tid; i < kT2Rows * kT2Cols; i += kMaxBlock) {
        // x fastest
        const int lc = ydom ? i % kT2Cols : i / kT2Rows, ld = ydom ? i / kT2Cols : i % kT2Rows;
        const int X = ydom ? c0 + lc : d0 + ld, Y = ydom ? d0 + ld : c0 + lc;
        const unsigned long long v = sh.c64[ld * kT2Pitch + kT2Side + lc];
        if (X < nx && Y < ny && v != 0ull) atomicAdd(&out[(size_t)Y * nx + X], v);
    }
}

// vol += accimg * max|y q.x| / 2^30.
template <class SV>
__global__ __launch_bounds__(kMaxBlock) void k_adj2d_finish(typename SV::raw *__restrict__ vol,
                                                           unsigned long long *__restrict__ accimg,
                                                           const float *__restrict__ parts,
                                                           size_t img) {
    const size_t b = blockIdx.y;
    const float ymax = adj2d_ymax(parts + b * kAdjParts);
    const double unit = (double)ymax * 0x1p-30;
    const size_t j = (size_t)blockIdx.x * kMaxBlock + threadIdx.x;
    if (j >= img) return;
    const size_t i = b * img + j;
    const long long q = (long long)accimg[i];
    vol[i] = from_f32<SV>(to_f32<SV>(vol[i]) + (float)((double)q * unit));
}

__global__ __launch_bounds__(kMaxBlock) void k_fill_u64(unsigned long long *__restrict__ p,
                                                        size_t n) {
    const size_t i = (size_t)blockIdx.x * kMaxBlock + threadIdx.x;
    if (i < n) p[i] = 0ull;
}

// ------------------------------------------------ transpose of the backprojection -------

// Bᵀ: the transpose of the voxel-driven backprojection (k_bp2d), the gradient of
// TorchBackprojection. The backprojection gives pixel p, per projection a, wt_a(p) times the
// linear interpolation of row a at u_a(p) (cells floor(u) and floor(u) + 1, weights 1 - al and
// al; cells outside the row read zero), times 1/du (circular plans; the view's 1/|u| is part of
// wt for plans from views). So sino[a][c] = sum_p (those weights) v[p]; positions and weights agree
// with k_bp2d's up to FP32 rounding (they come from FP64 sums per line, see below).
// A workgroup owns a segment of GS detector cells of one projection and gathers it. The pixels
// whose terms reach the segment's cells are those with u in [c0 - 1, c0 + GS): a wedge from
// the source between the lines u = c0 - 1 and u = c0 + GS (u is a ratio of two functions
// affine in the pixel). The workgroup marches through the image along the axis K (rows or
// columns) that the segment's central line follows most closely, in chunks of kGSlab lines;
// per line the wedge is the interval between the two boundary lines' crossings (kGMargin of a
// pixel wider on each side, for the FP32 lines; clipped to the image). A wavefront takes every
// fourth line of a chunk and walks it along the line, a lane per pixel, from the zero-bordered copy
// whose rows run along it (row-major for rows, transposed for columns), so that it reads runs of
// consecutive pixels. All
// lines of a chunk are walked over the width of its widest interval, their starts moved back
// where that would leave the image: pixels outside the wedge have no cell in the segment and add
// nothing. Depth d and d u, u the cell coordinate from the segment's start on, are affine in the
// pixel, so they are one sum each of the lane's share (its pixel number along the line) and the
// line's (evaluated in FP64 by the lane that holds the line, and read from it). Every pixel adds its
// terms that fall inside the segment to GS + 2 LDS cells with integer atomics. A segment whose
// boundary lines meet the lines at grazing angles walks whole lines. Where the widest interval is at
// most half a wavefront, in thin images and at an image's corners, a wavefront walks several lines
// at a time; a segment whose wedge passes beside the image walks nothing. Calls before / with both:
// 5 images of 1 x 512 x 90 56 / 35 us, 5 of 33 x 512 x 180 133 / 105, 512^2 x 180 of 0.5 pixels a
// cell 97 / 85, 1024^2 x 360 of 0.67 490 / 433.
// Bound by VALU issue. Walking the chunk's pixels as one flat list, which filled the lanes (0.94
// against 0.73 at 0.67 pixels per cell) but gave every pixel an index walk, a test against its
// line's interval and its own affine forms, took 51 VALU and 26 SALU instructions per wavefront of
// pixels; now 32 and 12 with the set-up. Dense images, calls: 1024^2 x 716 935 -> 750 us, 256^2 x
// 179 x 4 88 -> 77 us (2, 4, 8 lines in flight: 748, 757, 779 us at 1024^2).
// Fixed point: terms are rounded to units of max|v| * bound / 2^kGBits, where `bound` is the
// plan's bound on wt (times 1/du) over the image and all projections, so |term| <= 2^kGBits
// and a 32-bit LDS cell holds the sum of up to 2^(31 - kGBits) - 1 terms. A pixel adds at most
// one term to a cell, so the cells are moved into 64-bit registers (one per thread of the first
// GS) and cleared before the pixel visits since the last such drain could pass that count.
// Integer sums are exact: the result does not depend on the order of the additions. Each
// segment is written once, in the sinogram's storage type.
// Detector cells per segment: kGSFine where a pixel has at least kGFine cells, so that the walk's
// lines are still about a wavefront wide, and that leaves kGFineMany workgroups an image; else kGS,
// which gives more workgroups and, at one pixel per cell, lines that just fit a wavefront. Calls, us,
// with kGS and with kGSFine (walking the chunk's pixels as one flat list: third): 512^2 x 180 of 10
// cells per pixel 141, 87 (161), 4 cells 103, 78 (110), 2 cells 82, 85 (97), 1 cell 77, 120 (93); 640^2
// x 17 with 2000 of 5 cells per pixel (136 workgroups of kGSFine) 39, 64 (47), x 60 with 4000 of 12
// (960) 62, 54 (68). kGS 64: 5 % more at one cell per pixel of parallel rays, 2 % less at 1.5.
constexpr int kGS = 62, kGSFine = 256;
constexpr double kGFine = 1.75;
constexpr uint64_t kGFineMany = 1024;
constexpr int kGSlab = 64;                                   // image lines per chunk
constexpr int kGBits = 18;                                   // a term's bound: 2^kGBits units
constexpr int kGBudget = (1 << (31 - kGBits)) - 1;           // pixel visits between drains
constexpr int kGBatch = 4;           // lines per wavefront whose loads are in flight together
constexpr float kGMargin = 0.0625f;  // pixels around the boundary lines' crossings
static_assert(kGSlab == 64, "one lane per line");
static_assert(kGSlab / 4 * kMaxBlock <= kGBudget, "no drain within a chunk's step");
static_assert(kGSFine <= kMaxBlock, "one owned cell per thread");

// Largest |v| of each image of a batch, in kAdjParts partial maxima per image.
template <class SV>
__global__ __launch_bounds__(kMaxBlock) void k_absmax_img2d(const typename SV::raw *__restrict__ v,
                                                            size_t n, float *__restrict__ parts) {
    __shared__ float red[kMaxBlock / 64];
    const size_t b = blockIdx.y;
    v += b * n;
    parts += b * kAdjParts;
    float m = 0.0f;
    for (size_t i = (size_t)blockIdx.x * kMaxBlock + threadIdx.x; i < n;
         i += (size_t)kAdjParts * kMaxBlock)
        m = fmaxf(m, fabsf(to_f32<SV>(v[i])));
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kMaxBlock / 64; ++w) m = fmaxf(m, red[w]);
        parts[blockIdx.x] = m;
    }
}

// The line u(x, y) = uc of projection a as l0 x + l1 y + l2 = 0 in world coordinates (FP64),
// from the backprojector's own table: u = w eta + c with w and eta ratios / sums of affine terms.
template <bool VIEWS>
__device__ __forceinline__ void bpT_line(const float4 *__restrict__ tab, int a, double uc,
                                         double inv_du, double c0, double l[3]) {
    if (VIEWS) {
        const float4 m0 = tab[3 * a], m1 = tab[3 * a + 1];
        const double k = uc - (double)m1.w; // k (m0 . (x, y, 1)) = m0.w (m1 . (x, y, 1))
        l[0] = k * m0.x - (double)m0.w * m1.x;
        l[1] = k * m0.y - (double)m0.w * m1.y;
        l[2] = k * m0.z - (double)m0.w * m1.z;
    } else {
        const float4 m = tab[a];
        const double k = uc - c0; // k (m.x x - m.y y + m.w) = m.z (m.y x + m.x y) / du
        l[0] = k * m.x - (double)m.z * inv_du * m.y;
        l[1] = -k * m.y - (double)m.z * inv_du * m.x;
        l[2] = k * m.w;
    }
}

template <class SV, class SS, int WPOW, bool VIEWS, int GS>
__global__ __launch_bounds__(kMaxBlock) void k_bpT2d(typename SS::raw *__restrict__ sino,
                                                     const typename SV::raw *__restrict__ staged,
                                                     const float4 *__restrict__ tab,
                                                     const float *__restrict__ parts, float bound,
                                                     int nx, int ny, int D, int A, float sx,
                                                     float sy, float ox, float oy, float inv_du,
                                                     float half_d) {
    __shared__ unsigned int cells[GS + 2]; // cell c0 - 1 + i at i
    const int tid = threadIdx.x, lane = tid & 63;
    const int a = (int)(blockIdx.x % (unsigned)A);
    const int c0 = (int)(blockIdx.x / (unsigned)A) * GS;
    const size_t b = blockIdx.y;
    const float uoff = half_d - 0.5f;
    // fixed-point scale 2^18 / (max|v| bound) in two factors: a power of two that brings max|v|
    // to [1, 2) and the rest, which is then in range
    static_assert(kGBits == 18, "the scale uses 2^18");
    const float vmax = adj2d_ymax(parts + b * kAdjParts);
    const bool some = vmax > 0.0f && vmax < INFINITY;
    const int vexp = some ? ilogbf(vmax) : 0;
    const double rest = some ? 0x1p18 / (ldexp((double)vmax, -vexp) * (double)bound) : 0.0;
    // pixel index -> world: x = ix sx + bx (the world() map of the backprojector)
    const double bx = (double)ox + 0.5 - (double)((float)nx / 2.0f) * sx;
    const double by = (double)oy + 0.5 - (double)((float)ny / 2.0f) * sy;
    // the segment's central and boundary lines in index coordinates: n0 ix + n1 iy + n2 = 0
    auto index_line = [&](double uc, double (&n)[3]) {
        double l[3];
        bpT_line<VIEWS>(tab, a, uc, (double)inv_du, (double)uoff, l);
        n[0] = l[0] * sx;
        n[1] = l[1] * sy;
        n[2] = l[0] * bx + l[1] * by + l[2];
    };
    // march along rows (K = y, ranges along x) when the central line runs closer to y
    int rows;
    {
        double n[3];
        index_line((double)c0 + 0.5 * GS, n);
        rows = fabs(n[0]) >= fabs(n[1]) ? 1 : 0;
        rows = __builtin_amdgcn_readfirstlane(rows);
    }
    const int nK = rows ? ny : nx, nF = rows ? nx : ny;
    // Boundary lines as F = f0 + f1 K. The wedge's section of a line of K is the interval
    // between the two crossings when both boundary rays cross the lines of K steeply and in the
    // same direction. A line's coefficients are (uc Q - P) for u = P / Q with Q > 0 in front of
    // the source, so rotating its normal by a right angle gives a direction whose orientation
    // relative to the rays' forward direction is the same for every uc (the 2 x 2 determinant
    // of P and Q does not depend on uc): equal signs of the normals' F components mean equal
    // directions along K.
    float f0[2], f1[2];
    bool whole = false;
    double sgn[2];
    for (int e = 0; e < 2; ++e) {
        double n[3];
        index_line(e ? (double)(c0 + GS) : (double)(c0 - 1), n);
        const double nF_ = rows ? n[0] : n[1], nK_ = rows ? n[1] : n[0];
        sgn[e] = nF_;
        if (!(fabs(nF_) >= 0.25 * sqrt(nF_ * nF_ + nK_ * nK_)) || nF_ == 0.0) {
            whole = true;
            f0[e] = f1[e] = 0.0f;
        } else {
            f0[e] = (float)(-n[2] / nF_);
            f1[e] = (float)(-nK_ / nF_);
        }
    }
    if ((sgn[0] > 0.0) != (sgn[1] > 0.0)) whole = true;
    const int Wp = nx + 2 * kPad, Hp = ny + 2 * kPad;
    // pixel (f, k) along (F, K) lies at src[f + k strK] of the copy whose rows run along F
    const typename SV::raw *src = staged + b * 2 * (size_t)Wp * Hp +
                                  (rows ? (size_t)0 : (size_t)Wp * Hp) +
                                  (size_t)kPad * (rows ? Wp : Hp) + kPad;
    const int strK = rows ? Wp : Hp;
    for (int i = tid; i < GS + 2; i += kMaxBlock) cells[i] = 0u;
    long long own = 0;
    auto drain = [&]() {
        lds_barrier();
        if (tid < GS) {
            own += (long long)(int)cells[tid + 1];
            cells[tid + 1] = 0u;
        }
        __syncthreads();
    };
    // depth d and e = d u as affine forms of the pixel (f, k) along (F, K), cf f + ck k + c1; u the
    // cell coordinate from the segment's first LDS cell on, so that FP32 rounds no larger numbers
    // than those
    double dc[3], ec[3], L, wmul;
    {
        double dx, dy, dz, ex, ey, ez, cu;
        if (VIEWS) {
            const float4 m0 = tab[3 * a], m1 = tab[3 * a + 1];
            dx = m0.x, dy = m0.y, dz = m0.z;
            ex = m1.x, ey = m1.y, ez = m1.z;
            L = m0.w, cu = m1.w, wmul = tab[3 * a + 2].x;
        } else {
            const float4 m = tab[a];
            dx = m.x, dy = -m.y, dz = m.w;
            ex = (double)m.y * inv_du, ey = (double)m.x * inv_du, ez = 0.0;
            L = m.z, cu = uoff, wmul = inv_du;
        }
        cu -= (double)(c0 - 1);
        ex = L * ex + cu * dx, ey = L * ey + cu * dy, ez = L * ez + cu * dz;
        dc[2] = dx * bx + dy * by + dz, ec[2] = ex * bx + ey * by + ez;
        dx *= sx, ex *= sx, dy *= sy, ey *= sy;
        dc[0] = rows ? dx : dy, dc[1] = rows ? dy : dx;
        ec[0] = rows ? ex : ey, ec[1] = rows ? ey : ex;
    }
    const float vL = (float)L;
    const float s1 = ldexpf(1.0f, max(min(-vexp, 127), -126)); // (max|v| below 2^-127 scales to less)
    const float s2 = (float)(rest * wmul * ldexp(1.0, -vexp - max(min(-vexp, 127), -126)));
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    // a pixel of value val, depth d and e = d u adds its terms in the segment to the cells
    auto visit = [&](float val, float d, float e) {
        const float vs = val * s1 * s2;
        const float rd = __builtin_amdgcn_rcpf(d), u = rd * e;
        const int i = floor_i32(u);
        if ((unsigned)i > (unsigned)GS || vs == 0.0f) return;
        const float w = vL * rd;
        const float t = vs * (WPOW == 2 ? w * w : w);
        const float t1 = t * __builtin_amdgcn_fractf(u), t0 = t - t1;
        atomicAdd(&cells[i], (unsigned)round_i32(t0));
        atomicAdd(&cells[i + 1], (unsigned)round_i32(t1));
    };
    int run = 0; // pixel visits since the last drain
    __syncthreads(); // the cells are clear
    // nothing to walk if both boundary lines pass the image on one side (a pixel away and more) at
    // its first and at its last line
    bool beside = false;
    if (!whole) {
        const float e0 = fmaf(f1[0], (float)(nK - 1), f0[0]);
        const float e1 = fmaf(f1[1], (float)(nK - 1), f0[1]);
        beside = fmaxf(fmaxf(f0[0], f0[1]), fmaxf(e0, e1)) < -1.0f ||
                 fminf(fminf(f0[0], f0[1]), fminf(e0, e1)) > (float)nF;
    }
    const int todo = __builtin_amdgcn_readfirstlane(beside ? 0 : nK);
    for (int k0 = 0; k0 < todo; k0 += kGSlab) {
        // lane l holds line k0 + l: the first pixel of its interval, then its walk's start and
        // shares. Every wavefront does the same.
        const int S = min(kGSlab, nK - k0), k = k0 + min(lane, S - 1);
        int lo = 0, up = nF - 1;
        if (!whole) {
            const float g0 = fmaf(f1[0], (float)k, f0[0]), g1 = fmaf(f1[1], (float)k, f0[1]);
            constexpr float big = 0x1p24f;
            const float gl = fminf(g0, g1) - kGMargin, gu = fmaxf(g0, g1) + kGMargin;
            lo = max(0, floor_i32(__builtin_amdgcn_fmed3f(gl, -big, big)) + 1);
            up = min(nF - 1, floor_i32(__builtin_amdgcn_fmed3f(gu, -big, big)));
        }
        const int NW = __builtin_amdgcn_readfirstlane(wave_max(up - lo + 1));
        if (NW <= 0) continue;
        lo = max(0, min(lo, nF - NW));
        const float dl = (float)(dc[0] * lo + dc[1] * k + dc[2]);
        const float el = (float)(ec[0] * lo + ec[1] * k + ec[2]);
        const int at = lo + k * strK;
        if (NW <= 32) { // several lines to a wavefront
            if (run + kGSlab / 4 * kMaxBlock > kGBudget) {
                drain();
                run = 0;
            }
            run += kGSlab / 4 * kMaxBlock;
            const int sh = NW > 1 ? 32 - __builtin_clz((unsigned)NW - 1) : 0; // lanes a line: 2^sh
            const int f = lane & ((1 << sh) - 1), per = 64 >> sh;
            const bool in = f < NW;
            const int df = in ? f : 0;
            const float dp = (float)(dc[0] * df), ep = (float)(ec[0] * df);
            for (int l0 = wv * per; l0 < S; l0 += 4 * per * kGBatch) {
                float val[kGBatch];
#pragma unroll
                for (int q = 0; q < kGBatch; ++q) {
                    const int l = min(l0 + 4 * per * q + (lane >> sh), S - 1);
                    val[q] = to_f32<SV>(src[__shfl(at, l, 64) + df]);
                }
#pragma unroll
                for (int q = 0; q < kGBatch; ++q) {
                    if (l0 + 4 * per * q >= S) break;
                    const int m = l0 + 4 * per * q + (lane >> sh), l = min(m, S - 1);
                    visit(in && m < S ? val[q] : 0.0f, dp + __shfl(dl, l, 64),
                          ep + __shfl(el, l, 64));
                }
            }
            continue;
        }
        for (int f = 0; f < NW; f += 64) {
            if (run + kGSlab / 4 * kMaxBlock > kGBudget) {
                drain();
                run = 0;
            }
            run += kGSlab / 4 * kMaxBlock;
            // this lane's pixel of every line; past the width, its coordinate leaves the segment
            const bool in = f + lane < NW;
            const int df = in ? f + lane : 0;
            const float dp = (float)(dc[0] * df), ep = in ? (float)(ec[0] * df) : 1e30f;
            for (int l0 = wv; l0 < S; l0 += 4 * kGBatch) {
                float val[kGBatch];
#pragma unroll
                for (int q = 0; q < kGBatch; ++q) {
                    const int l = min(l0 + 4 * q, S - 1);
                    val[q] = to_f32<SV>(src[__builtin_amdgcn_readlane(at, l) + df]);
                }
#pragma unroll
                for (int q = 0; q < kGBatch; ++q) {
                    const int l = l0 + 4 * q;
                    if (l >= S) break;
                    visit(val[q],
                          dp + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(dl), l)),
                          ep + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(el), l)));
                }
            }
        }
    }
    lds_barrier();
    if (tid < GS) {
        own += (long long)(int)cells[tid + 1];
        const int c = c0 + tid;
        if (c < D) {
            const double unit = (double)vmax * (double)bound * 0x1p-18;
            sino[(b * A + a) * (size_t)D + c] = from_f32<SS>((float)((double)own * unit));
        }
    }
}

// ---------------------------------------------------------------- dispatch -----------------

template <class F>
cmi_status dispatch2(int dt_a, int dt_b, F &&f) {
    auto inner = [&](auto ta) -> cmi_status {
        switch (dt_b) {
        case CMI_F32: return f(ta, F32{});
        case CMI_F16: return f(ta, F16{});
        case CMI_BF16: return f(ta, BF16{});
        default: return fail(CMI_ERR_DTYPE, "unsupported dtype %d", dt_b);
        }
    };
    switch (dt_a) {
    case CMI_F32: return inner(F32{});
    case CMI_F16: return inner(F16{});
    case CMI_BF16: return inner(BF16{});
    default: return fail(CMI_ERR_DTYPE, "unsupported dtype %d", dt_a);
    }
}

cmi_status check_call(const cmi_plan2d *p, const void *vol, int vol_dtype, const void *sino,
                      int sino_dtype, uint64_t batch, const char *fn) {
    if (!p) return fail(CMI_ERR_INVALID_ARGUMENT, "%s: plan is null", fn);
    if (!vol) return fail(CMI_ERR_INVALID_ARGUMENT, "%s: volume pointer is null", fn);
    if (!sino) return fail(CMI_ERR_INVALID_ARGUMENT, "%s: sinogram pointer is null", fn);
    if (batch == 0) return fail(CMI_ERR_INVALID_ARGUMENT, "%s: batch must be >= 1", fn);
    if (!dtype_ok(vol_dtype) || !dtype_ok(sino_dtype))
        return fail(CMI_ERR_DTYPE, "%s: unsupported dtype (volume %d, sinogram %d)", fn,
                    vol_dtype, sino_dtype);
    if (vol_dtype != p->vol_prec)
        return fail(CMI_ERR_DTYPE, "%s: plan precision does not match volume precision (%s)",
                    fn, dtype_name(vol_dtype));
    if (sino_dtype != p->det_prec)
        return fail(CMI_ERR_DTYPE,
                    "%s: plan precision does not match sinogram precision (%s)", fn,
                    dtype_name(sino_dtype));
    const uint64_t img = (uint64_t)p->g.nx * p->g.ny, sn = (uint64_t)p->A * (p->g.D + 2 * kPad);
    const uint64_t pad = 2 * (uint64_t)(p->g.nx + 2 * kPad) * (p->g.ny + 2 * kPad);
    if (std::max({img, sn, pad}) * 4 >= (1ull << 31))
        return fail(CMI_ERR_INVALID_ARGUMENT, "%s: one image or sinogram exceeds 2 GiB", fn);
    if (batch > 65535) return fail(CMI_ERR_INVALID_ARGUMENT, "%s: batch exceeds 65535", fn);
    CMI_TRY(check_device_ptr(vol, p->device, "volume"));
    CMI_TRY(check_device_ptr(sino, p->device, "sinogram"));
    return CMI_OK;
}

// Checks and fields common to both plan constructors (Python order (y, x) -> (x, y), as
// plan.cu:48-50).
cmi_status check_plan_shape(int vol_prec, int det_prec, const uint64_t vol_shape[2],
                            const double vol_spacing[2], uint64_t det_count, uint64_t nangles,
                            const char *fn) {
    if (!dtype_ok(vol_prec) || !dtype_ok(det_prec))
        return fail(CMI_ERR_DTYPE, "%s: precision must be f32, f16 or bf16", fn);
    if (vol_shape[0] == 0 || vol_shape[1] == 0 || det_count == 0 || nangles == 0)
        return fail(CMI_ERR_INVALID_ARGUMENT,
                    "%s: empty shape (vol %llu x %llu, det %llu, angles %llu)", fn,
                    (unsigned long long)vol_shape[0], (unsigned long long)vol_shape[1],
                    (unsigned long long)det_count, (unsigned long long)nangles);
    if (vol_shape[0] > (1u << 20) || vol_shape[1] > (1u << 20) || det_count > (1u << 24) ||
        nangles > (1u << 24) || det_count * nangles >= (1ull << 31))
        return fail(CMI_ERR_INVALID_ARGUMENT, "%s: shape too large", fn);
    if (!(vol_spacing[0] > 0) || !(vol_spacing[1] > 0))
        return fail(CMI_ERR_INVALID_ARGUMENT, "%s: spacings must be positive", fn);
    return CMI_OK;
}

void set_plan_shape(cmi_plan2d &p, int device, int vol_prec, const uint64_t vol_shape[2],
                    const double vol_spacing[2], const double vol_offset[2], int det_prec,
                    uint64_t det_count, uint64_t nangles) {
    p.device = device;
    p.vol_prec = vol_prec;
    p.det_prec = det_prec;
    p.g.nx = (int64_t)vol_shape[1];
    p.g.ny = (int64_t)vol_shape[0];
    p.g.sx = vol_spacing[1];
    p.g.sy = vol_spacing[0];
    p.g.ox = vol_offset[1];
    p.g.oy = vol_offset[0];
    p.g.D = (int64_t)det_count;
    p.A = (int64_t)nangles;
}

// Whether angles a + k A / 4 are quarter turns of angle a with equal distances, to 1e-9: FP32 tables
// hold no more.
bool quarter_apart(const double *angles, const double *DSO, const double *DSD, int64_t A,
                   int64_t a) {
    const int64_t Q = A / 4;
    for (int64_t k = 1; k < 4; ++k) {
        const int64_t b = a + k * Q;
        if (DSO[b] != DSO[a] || DSD[b] != DSD[a]) return false;
        const double d =
            std::remainder(angles[b] - angles[a] - (double)k * M_PI / 2.0, 2.0 * M_PI);
        if (!(std::fabs(d) <= 1e-9)) return false;
    }
    return true;
}

// The backprojector's table of circular plans: (-sin, cos, DSD, DSO) per angle
// (backward_2d.hpp:58-62). Where all angles come in quadruples of quarter turns,
// so do its entries, exactly (angles written with some ten digits would round apart now and then):
// the first quarter's sines and cosines exchanged. Entries that agree, or of which both are zero but
// for roundoff (below 1e-13: added to half-integers times ones, they leave no trace), stay.
void bp2d_table(const double *angles, const double *DSO, const double *DSD, int64_t A, float *t) {
    bool turns = A % 4 == 0;
    for (int64_t a = 0; a < A; ++a) {
        t[4 * a] = (float)-std::sin(angles[a]);
        t[4 * a + 1] = (float)std::cos(angles[a]);
        t[4 * a + 2] = (float)DSD[a];
        t[4 * a + 3] = (float)DSO[a];
        turns = turns && (a >= A / 4 || quarter_apart(angles, DSO, DSD, A, a));
    }
    if (!turns) return;
    auto turn = [](float &p, float q) {
        if (!(p == q || (std::fabs(p) < 1e-13f && std::fabs(q) < 1e-13f))) p = q;
    };
    for (int64_t a = 0; a < A / 4; ++a)
        for (int64_t k = 1; k < 4; ++k) { // (-sin, cos) of the angle turned by k quarters
            float *m = t + 4 * (a + k * (A / 4));
            const float x = t[4 * a], y = t[4 * a + 1];
            turn(m[0], k == 1 ? -y : k == 2 ? -x : y);
            turn(m[1], k == 1 ? x : k == 2 ? -y : -x);
        }
}

// Whether the backprojection by quarter turns (k_bp2d_qt) applies: a square image with an even
// side, unit pixels and no offset (the pixel centres, at (i - n/2) + 1/2 as the reference places
// them, backward_2d.hpp:58-59, are then symmetric under quarter turns), angles in quadruples
// a + k A/4 that are quarter turns apart with equal DSO and DSD (their table entries then are,
// exactly: bp2d_table), a padded detector row at least as long as a staged segment, and every
// 16 x 16 tile's detector footprint within a staged segment: the projection of a segment of length
// L at depth >= DSO - r (r the largest pixel-centre radius) spans at most
// L DSD / (DSO - r) sqrt(1 + (r / (DSO - r))^2) / du cells.
bool quarter_turns(const fan2d::Scalars &g, const double *angles, const double *DSO,
                   const double *DSD, int64_t A) {
    if (g.nx != g.ny || g.nx % 2 != 0 || g.nx < 2 || g.sx != 1.0 || g.sy != 1.0 ||
        g.ox != 0.0 || g.oy != 0.0 || A % 4 != 0 || A < 4 || g.D + 2 * kPad < kQSeg)
        return false;
    const int64_t Q = A / 4;
    const double r = ((double)(g.nx / 2) - 0.5) * std::sqrt(2.0);
    double wmax = 0.0;
    for (int64_t a = 0; a < A; ++a) {
        if (!(DSO[a] > r + 1.0)) return false;
        const double ratio = r / (DSO[a] - r);
        wmax = std::max(wmax, DSD[a] / (DSO[a] - r) * std::sqrt(1.0 + ratio * ratio));
        if (a >= Q) continue;
        if (!quarter_apart(angles, DSO, DSD, A, a)) return false;
    }
    const double span = wmax * (kQT - 1) * std::sqrt(2.0) / g.du;
    return span + 4.0 <= (double)kQSeg;
}

// Shared tail of the plan constructors: per-angle tables to the device, then the FP64 ray
// table (k_ray_table). `meta` (circular plans) or `bpv` (plans from views) is empty.
cmi_status finish_plan2d(std::unique_ptr<cmi_plan2d> p, const std::vector<AngleGeom> &geo,
                         const std::vector<float4> &meta, const std::vector<float4> &bpv,
                         cmi_plan2d **plan) {
    const int64_t A = p->A, D = p->g.D;
    // the backprojection's weight bounds: depth is affine over the image, so its minimum over
    // the pixel centres is at a corner; 1 % of margin for the kernels' FP32 arithmetic
    {
        const double nx = (double)p->g.nx, ny = (double)p->g.ny;
        const double xs[2] = {(0.0 - nx / 2.0) * p->g.sx + p->g.ox + 0.5,
                              (nx - 1.0 - nx / 2.0) * p->g.sx + p->g.ox + 0.5};
        const double ys[2] = {(0.0 - ny / 2.0) * p->g.sy + p->g.oy + 0.5,
                              (ny - 1.0 - ny / 2.0) * p->g.sy + p->g.oy + 0.5};
        double b1 = 0.0, b2 = 0.0;
        bool ok = true;
        // depth, magnification and 1 / |u| of projection a at (x, y)
        auto at = [&](int64_t a, double x, double y, double &w, double &scale) {
            double depth, L;
            if (!meta.empty()) {
                const float4 m = meta[a];
                depth = (double)m.x * x - (double)m.y * y + (double)m.w;
                L = m.z;
                scale = 1.0 / p->g.du;
            } else {
                const float4 m0 = bpv[3 * a];
                depth = (double)m0.x * x + (double)m0.y * y + (double)m0.z;
                L = m0.w;
                scale = bpv[3 * a + 2].x;
            }
            w = std::fabs(L) / depth;
            return depth > 0.0;
        };
        double w, scale, cells = 0.0;
        for (int64_t a = 0; a < A && ok; ++a) {
            for (int c = 0; c < 4 && ok; ++c) {
                ok = at(a, xs[c & 1], ys[c >> 1], w, scale);
                b1 = std::max(b1, w * scale);
                b2 = std::max(b2, w * w * scale);
            }
            (void)at(a, 0.5 * (xs[0] + xs[1]), 0.5 * (ys[0] + ys[1]), w, scale);
            cells += w * scale;
        }
        if (ok) p->cells_per_pixel = cells / (double)A * std::sqrt(p->g.sx * p->g.sy);
        if (ok && b1 > 0.0 && std::isfinite(b2)) {
            p->bt_bound[0] = 1.01 * b1;
            p->bt_bound[1] = 1.01 * b2;
        }
    }
    std::vector<float> ageo(6 * A);
    for (int64_t a = 0; a < A; ++a)
        for (int d = 0; d < 2; ++d) {
            ageo[6 * a + d] = (float)geo[a].src[d];
            ageo[6 * a + 2 + d] = (float)geo[a].org[d];
            ageo[6 * a + 4 + d] = (float)geo[a].del[d];
        }
    DeviceGuard guard;
    CMI_TRY(guard.enter(p->device));
    struct Cleanup {
        cmi_plan2d *p;
        bool armed = true;
        ~Cleanup() {
            if (!armed) return;
            (void)hipFree(p->d_geo);
            (void)hipFree(p->d_meta);
            (void)hipFree(p->d_bpv);
            (void)hipFree(p->d_ageo);
            (void)hipFree(p->d_ev);
            (void)hipFree(p->d_ns);
        }
    } cleanup{p.get()};
    const size_t rays = (size_t)A * D;
    CMI_HIP_TRY(hipMalloc(&p->d_geo, sizeof(AngleGeom) * A));
    if (!meta.empty()) CMI_HIP_TRY(hipMalloc(&p->d_meta, sizeof(float4) * A));
    if (!bpv.empty()) CMI_HIP_TRY(hipMalloc(&p->d_bpv, sizeof(float4) * bpv.size()));
    CMI_HIP_TRY(hipMalloc(&p->d_ageo, sizeof(float) * 6 * A));
    CMI_HIP_TRY(hipMalloc(&p->d_ev, sizeof(float4) * rays));
    CMI_HIP_TRY(hipMalloc(&p->d_ns, sizeof(float4) * rays));
    p->table_bytes = sizeof(AngleGeom) * A + sizeof(float4) * (meta.size() + bpv.size()) +
                     sizeof(float) * 6 * A + 2 * sizeof(float4) * rays;
    unsigned long long *d_total = nullptr;
    CMI_HIP_TRY(hipMalloc(&d_total, sizeof(unsigned long long)));
    std::unique_ptr<unsigned long long, void (*)(unsigned long long *)> total_guard(
        d_total, [](unsigned long long *q) { (void)hipFree(q); });
    hipStream_t s;
    CMI_HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    std::unique_ptr<ihipStream_t, void (*)(hipStream_t)> stream_guard(
        s, [](hipStream_t q) { (void)hipStreamDestroy(q); });
    CMI_HIP_TRY(hipMemcpyAsync(p->d_geo, geo.data(), sizeof(AngleGeom) * A,
                               hipMemcpyHostToDevice, s));
    if (!meta.empty())
        CMI_HIP_TRY(hipMemcpyAsync(p->d_meta, meta.data(), sizeof(float4) * A,
                                   hipMemcpyHostToDevice, s));
    if (!bpv.empty())
        CMI_HIP_TRY(hipMemcpyAsync(p->d_bpv, bpv.data(), sizeof(float4) * bpv.size(),
                                   hipMemcpyHostToDevice, s));
    CMI_HIP_TRY(hipMemcpyAsync(p->d_ageo, ageo.data(), sizeof(float) * 6 * A,
                               hipMemcpyHostToDevice, s));
    CMI_HIP_TRY(hipMemsetAsync(d_total, 0, sizeof(unsigned long long), s));
    dim3 blk(256), grd((unsigned)((D + 255) / 256), (unsigned)A);
    hipLaunchKernelGGL(k_ray_table, grd, blk, 0, s, p->d_geo, (int)A, (int)D, p->g.nx, p->g.ny,
                       p->g.sx, p->g.sy, p->d_ev, p->d_ns, d_total);
    CMI_HIP_TRY(hipGetLastError());
    unsigned long long total = 0;
    CMI_HIP_TRY(hipMemcpyAsync(&total, d_total, sizeof total, hipMemcpyDeviceToHost, s));
    CMI_HIP_TRY(hipStreamSynchronize(s));
    p->total_samples = total;
    cleanup.armed = false;
    *plan = p.release();
    return CMI_OK;
}

// Plans from ASTRA-like views (cmi_plan2d_create_vec, and cmi_plan2d_create_ex with exact
// geometry, which builds its views first).
cmi_status plan2d_from_views(int device, int vol_prec, const uint64_t vol_shape[2],
                             const double vol_spacing[2], const double vol_offset[2],
                             int det_prec, uint64_t det_count, const double *vecs,
                             uint64_t nangles, const char *fn, cmi_plan2d **plan) {
    CMI_TRY(check_plan_shape(vol_prec, det_prec, vol_shape, vol_spacing, det_count, nangles, fn));
    for (uint64_t a = 0; a < nangles; ++a) {
        const double *v = vecs + 6 * a;
        for (int i = 0; i < 6; ++i)
            if (!std::isfinite(v[i]))
                return fail(CMI_ERR_INVALID_ARGUMENT, "%s: non-finite view %llu", fn,
                            (unsigned long long)a);
        const fan2d::BpView bv = fan2d::bp_view(v, (int64_t)det_count);
        if (!(v[4] * v[4] + v[5] * v[5] > 0.0) || !(bv.L > 0.0))
            return fail(CMI_ERR_INVALID_ARGUMENT,
                        "%s: view %llu has a zero cell step or its source on the detector line",
                        fn, (unsigned long long)a);
    }
    auto p = std::make_unique<cmi_plan2d>();
    set_plan_shape(*p, device, vol_prec, vol_shape, vol_spacing, vol_offset, det_prec, det_count,
                   nangles);
    p->g.du = std::sqrt(vecs[4] * vecs[4] + vecs[5] * vecs[5]); // view 0's, for get_info
    const int64_t A = p->A;
    std::vector<AngleGeom> geo(A);
    std::vector<float4> bpv(3 * A);
    for (int64_t a = 0; a < A; ++a) {
        geo[a] = fan2d::plan_angle_vec(p->g, vecs + 6 * a);
        const fan2d::BpView bv = fan2d::bp_view(vecs + 6 * a, p->g.D);
        bpv[3 * a] = make_float4((float)bv.n[0], (float)bv.n[1], (float)bv.n0, (float)bv.L);
        // the cell offset carries the lerp's texel-centre shift (-0.5)
        bpv[3 * a + 1] =
            make_float4((float)bv.e[0], (float)bv.e[1], (float)bv.e0, (float)(bv.c0 - 0.5));
        bpv[3 * a + 2] = make_float4((float)bv.inv_du, 0.0f, 0.0f, 0.0f);
    }
    return finish_plan2d(std::move(p), geo, {}, bpv, plan);
}

} // namespace

// ------------------------------------------------------ forward, shared by the entry points --

namespace cmi {

cmi_status fan2d_forward_check(const cmi_plan2d *plan, const void *volume, int vol_dtype,
                               const void *sinogram, int sino_dtype, uint64_t batch) {
    return check_call(plan, volume, vol_dtype, sinogram, sino_dtype, batch, "forward_2d");
}

int fan2d_plan_device(const cmi_plan2d *plan) { return plan->device; }

// Two zero-bordered copies of each image of the batch (row-major and transposed).
size_t fan2d_forward_scratch_bytes(const cmi_plan2d *plan, int vol_dtype, uint64_t batch) {
    const size_t Wp = (size_t)plan->g.nx + 2 * kPad, Hp = (size_t)plan->g.ny + 2 * kPad;
    return 2 * Wp * Hp * dtype_size(vol_dtype) * batch;
}

// Stages the batch into `scratch` (at least fan2d_forward_scratch_bytes bytes of device memory
// on the plan's device, which is current) and launches the march, on `s`. Every staged element,
// border included, is written, so the scratch needs no clearing between calls.
cmi_status fan2d_forward_enqueue(const cmi_plan2d *plan, const void *volume, int vol_dtype,
                                 void *sinogram, int sino_dtype, uint64_t batch, void *scratch,
                                 hipStream_t s) {
    const int nx = (int)plan->g.nx, ny = (int)plan->g.ny, D = (int)plan->g.D, A = (int)plan->A;
    const int Wp = nx + 2 * kPad, Hp = ny + 2 * kPad;
    return dispatch2(vol_dtype, sino_dtype, [&](auto si, auto ss) -> cmi_status {
        using SI = decltype(si);
        using SS = decltype(ss);
        using RI = typename SI::raw;
        dim3 sb(32, 8), sg((unsigned)((Wp + 31) / 32), (unsigned)((Hp + 31) / 32),
                           (unsigned)batch);
        hipLaunchKernelGGL((k_stage2d<SI>), sg, sb, 0, s, (const RI *)volume, (RI *)scratch, nx,
                           ny, Wp, Hp);
        // block_x * block_y (at most kFwdRays) adjacent cells of one angle per workgroup
        const unsigned nt = std::min<unsigned>(plan->block_x * plan->block_y, kFwdRays);
        dim3 fb(nt), fg((unsigned)((D + nt - 1) / nt), (unsigned)A, (unsigned)batch);
        const bool half = plan->cells_per_pixel < kHalfCells &&
                          (2 * (uint64_t)Wp * Hp * sizeof(RI) >= kHalfBytes ||
                           (uint64_t)fg.x * A * batch >= kHalfGroups);
        auto kern = half ? k_fwd2d<SI, SS, HalfBands> : k_fwd2d<SI, SS, WholeBands>;
        hipLaunchKernelGGL(kern, fg, fb, 0, s, (const RI *)scratch, Wp, Hp,
                           plan->d_ev, plan->d_ns, (typename SS::raw *)sinogram, D, A);
        CMI_HIP_TRY(hipGetLastError());
        return CMI_OK;
    });
}

} // namespace cmi

// ===================================================================== C-ABI ===============

extern "C" {

CMI_API cmi_status cmi_plan2d_create(int device, int vol_prec, const uint64_t vol_shape[2],
                                     const double vol_spacing[2], const double vol_offset[2],
                                     int det_prec, uint64_t det_count, double det_spacing,
                                     double det_offset, const double *DSO, const double *DSD,
                                     const double *angles, uint64_t nangles, double det_pitch,
                                     double COR, cmi_plan2d **plan) {
    clear_error();
    if (!plan) return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create: output pointer is null");
    *plan = nullptr;
    if (!vol_shape || !vol_spacing || !vol_offset || !DSO || !DSD || !angles)
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create: null geometry array");
    CMI_TRY(check_plan_shape(vol_prec, det_prec, vol_shape, vol_spacing, det_count, nangles,
                             "plan2d_create"));
    if (!(det_spacing > 0))
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create: spacings must be positive");
    for (uint64_t a = 0; a < nangles; ++a)
        if (!std::isfinite(angles[a]) || !std::isfinite(DSO[a]) || !std::isfinite(DSD[a]))
            return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create: non-finite geometry at angle %llu",
                        (unsigned long long)a);

    auto p = std::make_unique<cmi_plan2d>();
    set_plan_shape(*p, device, vol_prec, vol_shape, vol_spacing, vol_offset, det_prec, det_count,
                   nangles);
    p->g.du = det_spacing;
    p->g.det_offset = det_offset;
    p->pitch = det_pitch;
    p->cor = COR;

    const int64_t A = p->A;
    std::vector<AngleGeom> geo(A);
    for (int64_t a = 0; a < A; ++a) geo[a] = fan2d::plan_angle(p->g, angles[a], DSO[a], DSD[a]);
    p->quarter = quarter_turns(p->g, angles, DSO, DSD, A);
    std::vector<float4> meta(A);
    bp2d_table(angles, DSO, DSD, A, &meta[0].x);
    return finish_plan2d(std::move(p), geo, meta, {}, plan);
}

CMI_API cmi_status cmi_plan2d_create_vec(int device, int vol_prec, const uint64_t vol_shape[2],
                                         const double vol_spacing[2], const double vol_offset[2],
                                         int det_prec, uint64_t det_count, const double *vecs,
                                         uint64_t nangles, cmi_plan2d **plan) {
    clear_error();
    if (!plan) return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create_vec: output pointer is null");
    *plan = nullptr;
    if (!vol_shape || !vol_spacing || !vol_offset || !vecs)
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create_vec: null geometry array");
    return plan2d_from_views(device, vol_prec, vol_shape, vol_spacing, vol_offset, det_prec,
                             det_count, vecs, nangles, "plan2d_create_vec", plan);
}

CMI_API cmi_status cmi_plan2d_create_ex(int device, int vol_prec, const uint64_t vol_shape[2],
                                        const double vol_spacing[2], const double vol_offset[2],
                                        int det_prec, uint64_t det_count, double det_spacing,
                                        double det_offset, const double *DSO, const double *DSD,
                                        const double *angles, uint64_t nangles,
                                        double det_pitch, double COR, uint32_t flags,
                                        cmi_plan2d **plan) {
    if ((flags & ~(uint32_t)CMI_PLAN2D_EXACT_GEOMETRY) != 0) {
        clear_error();
        if (plan) *plan = nullptr;
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create_ex: unknown flags 0x%x", flags);
    }
    if (!(flags & CMI_PLAN2D_EXACT_GEOMETRY))
        return cmi_plan2d_create(device, vol_prec, vol_shape, vol_spacing, vol_offset, det_prec,
                                 det_count, det_spacing, det_offset, DSO, DSD, angles, nangles,
                                 det_pitch, COR, plan);
    clear_error();
    if (!plan) return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create_ex: output pointer is null");
    *plan = nullptr;
    if (!vol_shape || !vol_spacing || !vol_offset || !DSO || !DSD || !angles)
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create_ex: null geometry array");
    CMI_TRY(check_plan_shape(vol_prec, det_prec, vol_shape, vol_spacing, det_count, nangles,
                             "plan2d_create_ex"));
    if (!(det_spacing > 0))
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create_ex: spacings must be positive");
    if (!std::isfinite(det_offset) || !std::isfinite(det_pitch) || !std::isfinite(COR))
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_create_ex: non-finite detector geometry");
    fan2d::Scalars g{};
    g.du = det_spacing;
    g.det_offset = det_offset;
    std::vector<double> vecs(6 * nangles);
    for (uint64_t a = 0; a < nangles; ++a) {
        if (!std::isfinite(angles[a]) || !std::isfinite(DSO[a]) || !std::isfinite(DSD[a]))
            return fail(CMI_ERR_INVALID_ARGUMENT,
                        "plan2d_create_ex: non-finite geometry at angle %llu",
                        (unsigned long long)a);
        fan2d::exact_view(g, angles[a], DSO[a], DSD[a], det_pitch, COR, vecs.data() + 6 * a);
    }
    return plan2d_from_views(device, vol_prec, vol_shape, vol_spacing, vol_offset, det_prec,
                             det_count, vecs.data(), nangles, "plan2d_create_ex", plan);
}

CMI_API cmi_status cmi_fan2d_bp_table(uint64_t nangles, const double *angles, const double *DSO,
                                      const double *DSD, float *table) {
    clear_error();
    if (!angles || !DSO || !DSD || !table)
        return fail(CMI_ERR_INVALID_ARGUMENT, "fan2d_bp_table: null argument");
    bp2d_table(angles, DSO, DSD, (int64_t)nangles, table);
    return CMI_OK;
}

CMI_API cmi_status cmi_plan2d_destroy(cmi_plan2d *plan) {
    clear_error();
    if (!plan) return CMI_OK;
    DeviceGuard guard;
    const cmi_status st = guard.enter(plan->device);
    if (st == CMI_OK) {
        // Work enqueued with this plan may still be running on any stream.
        (void)hipDeviceSynchronize();
        (void)hipFree(plan->d_geo);
        (void)hipFree(plan->d_meta);
        (void)hipFree(plan->d_bpv);
        (void)hipFree(plan->d_ageo);
        (void)hipFree(plan->d_ev);
        (void)hipFree(plan->d_ns);
    }
    delete plan;
    return st;
}

CMI_API cmi_status cmi_plan2d_set_block(cmi_plan2d *plan, uint32_t block_x, uint32_t block_y) {
    clear_error();
    if (!plan) return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_set_block: plan is null");
    // The forward kernel is compiled for at most kMaxBlock threads per workgroup
    // (__launch_bounds__); a larger workgroup must never reach the launch.
    if (block_x == 0 || block_x % 64 != 0 || block_y == 0 || block_x * block_y > kMaxBlock)
        return fail(CMI_ERR_INVALID_ARGUMENT,
                    "plan2d_set_block: need block_x a multiple of 64 and block_x*block_y <= "
                    "%d (got %u x %u)",
                    kMaxBlock, block_x, block_y);
    plan->block_x = block_x;
    plan->block_y = block_y;
    return CMI_OK;
}

CMI_API cmi_status cmi_plan2d_get_block(const cmi_plan2d *plan, uint32_t *block_x,
                                        uint32_t *block_y) {
    clear_error();
    if (!plan || !block_x || !block_y)
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_get_block: null argument");
    *block_x = plan->block_x;
    *block_y = plan->block_y;
    return CMI_OK;
}

CMI_API cmi_status cmi_plan2d_get_info(const cmi_plan2d *plan, cmi_plan2d_info *info) {
    clear_error();
    if (!plan || !info) return fail(CMI_ERR_INVALID_ARGUMENT, "plan2d_get_info: null argument");
    info->device = plan->device;
    info->vol_prec = plan->vol_prec;
    info->det_prec = plan->det_prec;
    info->nx = (uint64_t)plan->g.nx;
    info->ny = (uint64_t)plan->g.ny;
    info->det_count = (uint64_t)plan->g.D;
    info->nangles = (uint64_t)plan->A;
    info->total_samples = plan->total_samples;
    info->table_bytes = plan->table_bytes;
    return CMI_OK;
}

CMI_API cmi_status cmi_forward_2d(const cmi_plan2d *plan, const void *volume, int vol_dtype,
                                  void *sinogram, int sino_dtype, uint64_t batch,
                                  void *stream) {
    clear_error();
    CMI_TRY(fan2d_forward_check(plan, volume, vol_dtype, sinogram, sino_dtype, batch));
    DeviceGuard guard;
    CMI_TRY(guard.enter(plan->device));
    const hipStream_t s = (hipStream_t)stream;
    void *scratch = nullptr;
    CMI_HIP_TRY(hipMallocAsync(&scratch, fan2d_forward_scratch_bytes(plan, vol_dtype, batch), s));
    const cmi_status st =
        fan2d_forward_enqueue(plan, volume, vol_dtype, sinogram, sino_dtype, batch, scratch, s);
    const hipError_t fe = hipFreeAsync(scratch, s);
    if (st != CMI_OK) return st;
    CMI_HIP_TRY(fe);
    return CMI_OK;
}

CMI_API cmi_status cmi_backward_2d_weighted(const cmi_plan2d *plan, void *volume, int vol_dtype,
                                            const void *sinogram, int sino_dtype,
                                            uint64_t batch, int weighting, void *stream) {
    clear_error();
    CMI_TRY(check_call(plan, volume, vol_dtype, sinogram, sino_dtype, batch, "backward_2d"));
    if (weighting != CMI_BP2D_REFERENCE && weighting != CMI_BP2D_FBP)
        return fail(CMI_ERR_INVALID_ARGUMENT, "backward_2d: unknown weighting %d", weighting);
    DeviceGuard guard;
    CMI_TRY(guard.enter(plan->device));
    const hipStream_t s = (hipStream_t)stream;
    const int nx = (int)plan->g.nx, ny = (int)plan->g.ny, D = (int)plan->g.D, A = (int)plan->A;
    const int Dp = D + 2 * kPad;
    void *scratch = nullptr;
    CMI_HIP_TRY(hipMallocAsync(&scratch, (size_t)Dp * A * dtype_size(sino_dtype) * batch, s));
    const cmi_status st = dispatch2(vol_dtype, sino_dtype, [&](auto sv, auto ss) -> cmi_status {
        using SV = decltype(sv);
        using SS = decltype(ss);
        using RS = typename SS::raw;
        dim3 pb(256), pg((unsigned)((Dp + 255) / 256), (unsigned)A, (unsigned)batch);
        hipLaunchKernelGGL((k_stage_sino2d<SS>), pg, pb, 0, s, (const RS *)sinogram,
                           (RS *)scratch, D, A);
        const bool fbp = weighting == CMI_BP2D_FBP;
        const float inv_du = (float)(1.0 / plan->g.du), half_d = (float)D / 2.0f;
        const uint64_t th = (uint64_t)(nx / 2 + kQT - 1) / kQT;
        if (plan->quarter && th * th * batch >= kQTMinTiles) {
            auto kern = fbp ? k_bp2d_qt<SV, SS, 2> : k_bp2d_qt<SV, SS, 1>;
            hipLaunchKernelGGL(kern, dim3((unsigned)th, (unsigned)th, (unsigned)batch),
                               dim3(kQThreads), 0, s, (typename SV::raw *)volume,
                               (const RS *)scratch, plan->d_meta, nx, D, A, inv_du, half_d);
        } else {
            const unsigned tx = (unsigned)(nx + 63) / 64;
            auto launch = [&](auto kern, int rows, const float4 *tab, float f) {
                const unsigned tiles = tx * (unsigned)((ny + rows - 1) / rows);
                hipLaunchKernelGGL(kern, dim3(tiles, 1, (unsigned)batch), dim3(kMaxBlock), 0, s,
                                   (typename SV::raw *)volume, (const RS *)scratch, tab, nx, ny,
                                   D, A, (float)plan->g.sx, (float)plan->g.sy,
                                   (float)plan->g.ox, (float)plan->g.oy, inv_du, half_d, f);
            };
            const bool two = plan->cells_per_pixel >= kRowsFine &&
                             (uint64_t)tx * ((ny + 1) / 2) * batch >= kRowTiles;
            auto kernel = [&](auto rows) {
                constexpr int NY = decltype(rows)::value;
                if (plan->d_bpv)
                    launch(fbp ? k_bp2d<SV, SS, ViewAngle<2>, NY> : k_bp2d<SV, SS, ViewAngle<1>, NY>,
                           NY, plan->d_bpv, 1.0f);
                else
                    launch(fbp ? k_bp2d<SV, SS, FanAngle<2>, NY> : k_bp2d<SV, SS, FanAngle<1>, NY>,
                           NY, plan->d_meta, inv_du);
            };
            if (two) kernel(std::integral_constant<int, 2>{});
            else kernel(std::integral_constant<int, 1>{});
        }
        CMI_HIP_TRY(hipGetLastError());
        return CMI_OK;
    });
    const hipError_t fe = hipFreeAsync(scratch, s);
    if (st != CMI_OK) return st;
    CMI_HIP_TRY(fe);
    return CMI_OK;
}

CMI_API cmi_status cmi_backward_2d(const cmi_plan2d *plan, void *volume, int vol_dtype,
                                   const void *sinogram, int sino_dtype, uint64_t batch,
                                   void *stream) {
    return cmi_backward_2d_weighted(plan, volume, vol_dtype, sinogram, sino_dtype, batch,
                                    CMI_BP2D_REFERENCE, stream);
}

CMI_API cmi_status cmi_backward_2d_transpose(const cmi_plan2d *plan, void *sinogram,
                                             int sino_dtype, const void *volume, int vol_dtype,
                                             uint64_t batch, int weighting, void *stream) {
    clear_error();
    CMI_TRY(check_call(plan, volume, vol_dtype, sinogram, sino_dtype, batch,
                       "backward_2d_transpose"));
    if (weighting != CMI_BP2D_REFERENCE && weighting != CMI_BP2D_FBP)
        return fail(CMI_ERR_INVALID_ARGUMENT, "backward_2d_transpose: unknown weighting %d",
                    weighting);
    const double bound = plan->bt_bound[weighting == CMI_BP2D_FBP ? 1 : 0];
    if (!std::isfinite(bound))
        return fail(CMI_ERR_NOT_SUPPORTED,
                    "backward_2d_transpose: a source lies inside the image's bounding box, so "
                    "the backprojection's weight is unbounded");
    DeviceGuard guard;
    CMI_TRY(guard.enter(plan->device));
    const hipStream_t s = (hipStream_t)stream;
    const int nx = (int)plan->g.nx, ny = (int)plan->g.ny, D = (int)plan->g.D, A = (int)plan->A;
    const size_t img = (size_t)nx * ny;
    const int Wp = nx + 2 * kPad, Hp = ny + 2 * kPad;
    // (not by the batch: an image's bits do not depend on the others)
    const bool fine = plan->cells_per_pixel >= kGFine &&
                      (uint64_t)A * ((D + kGSFine - 1) / kGSFine) >= kGFineMany;
    const int gs = fine ? kGSFine : kGS;
    const uint64_t nseg = (uint64_t)(D + gs - 1) / gs;
    if ((uint64_t)A * nseg * kMaxBlock >= (1ull << 32) || batch > 65535)
        return fail(CMI_ERR_INVALID_ARGUMENT,
                    "backward_2d_transpose: too many projections, cells or images for one "
                    "launch");
    // scratch: per image its zero-bordered row-major and transposed copies, then kAdjParts
    // partial maxima per image
    const size_t copy_bytes =
        (2 * (size_t)Wp * Hp * dtype_size(vol_dtype) * batch + 255) / 256 * 256;
    void *scratch = nullptr;
    CMI_HIP_TRY(hipMallocAsync(&scratch, copy_bytes + kAdjParts * batch * sizeof(float), s));
    float *parts = (float *)((char *)scratch + copy_bytes);
    const cmi_status st = dispatch2(vol_dtype, sino_dtype, [&](auto sv, auto ss) -> cmi_status {
        using SV = decltype(sv);
        using SS = decltype(ss);
        using RV = typename SV::raw;
        dim3 sb(32, 8), sg((unsigned)((Wp + 31) / 32), (unsigned)((Hp + 31) / 32),
                           (unsigned)batch);
        hipLaunchKernelGGL((k_stage2d<SV>), sg, sb, 0, s, (const RV *)volume, (RV *)scratch, nx,
                           ny, Wp, Hp);
        hipLaunchKernelGGL((k_absmax_img2d<SV>), dim3(kAdjParts, (unsigned)batch),
                           dim3(kMaxBlock), 0, s, (const RV *)volume, img, parts);
        const bool views = plan->d_bpv != nullptr;
        const bool fbp = weighting == CMI_BP2D_FBP;
        auto pick = [&](auto cells) {
            constexpr int GS = decltype(cells)::value;
            return views ? (fbp ? k_bpT2d<SV, SS, 2, true, GS> : k_bpT2d<SV, SS, 1, true, GS>)
                         : (fbp ? k_bpT2d<SV, SS, 2, false, GS> : k_bpT2d<SV, SS, 1, false, GS>);
        };
        auto kern = fine ? pick(std::integral_constant<int, kGSFine>{})
                         : pick(std::integral_constant<int, kGS>{});
        // projections fastest: neighbouring workgroups gather overlapping wedges
        hipLaunchKernelGGL(kern, dim3((unsigned)(A * nseg), (unsigned)batch), dim3(kMaxBlock),
                           0, s, (typename SS::raw *)sinogram, (const RV *)scratch,
                           views ? plan->d_bpv : plan->d_meta, parts, (float)bound, nx, ny, D,
                           A, (float)plan->g.sx, (float)plan->g.sy, (float)plan->g.ox,
                           (float)plan->g.oy, (float)(1.0 / plan->g.du), (float)D / 2.0f);
        CMI_HIP_TRY(hipGetLastError());
        return CMI_OK;
    });
    const hipError_t fe = hipFreeAsync(scratch, s);
    if (st != CMI_OK) return st;
    CMI_HIP_TRY(fe);
    return CMI_OK;
}

CMI_API cmi_status cmi_adjoint_2d(const cmi_plan2d *plan, void *volume, int vol_dtype,
                                  const void *sinogram, int sino_dtype, uint64_t batch,
                                  void *stream) {
    clear_error();
    CMI_TRY(check_call(plan, volume, vol_dtype, sinogram, sino_dtype, batch, "adjoint_2d"));
    DeviceGuard guard;
    CMI_TRY(guard.enter(plan->device));
    const hipStream_t s = (hipStream_t)stream;
    const int nx = (int)plan->g.nx, ny = (int)plan->g.ny, D = (int)plan->g.D, A = (int)plan->A;
    const size_t img = (size_t)nx * ny * batch, rays = (size_t)A * D;
    // scratch: the 64-bit sum image, then kAdjParts partial maxima
    void *scratch = nullptr;
    CMI_HIP_TRY(hipMallocAsync(&scratch, img * 8 + kAdjParts * batch * sizeof(float), s));
    unsigned long long *accimg = (unsigned long long *)scratch;
    float *parts = (float *)(accimg + img);
    const cmi_status st = dispatch2(vol_dtype, sino_dtype, [&](auto sv, auto ss) -> cmi_status {
        using SV = decltype(sv);
        using SS = decltype(ss);
        const unsigned nb = (unsigned)((img + kMaxBlock - 1) / kMaxBlock);
        hipLaunchKernelGGL(k_fill_u64, dim3(nb), dim3(kMaxBlock), 0, s, accimg, img);
        hipLaunchKernelGGL((k_adj2d_absmax<SS>), dim3(kAdjParts, (unsigned)batch),
                           dim3(kMaxBlock), 0, s, (const typename SS::raw *)sinogram, plan->d_ns,
                           rays, parts);
        const unsigned tiles = adj2d_tiles(ny, nx) + adj2d_tiles(nx, ny);
        const uint64_t all = (uint64_t)tiles * batch;
        const uint64_t samples = (plan->total_samples + kAdjRay * rays) * batch / all; // per tile
        const int G = (int)std::max<uint64_t>(
            1, std::min<uint64_t>(
                   {(uint64_t)A, (kAdjWorkgroups + all - 1) / all,
                    std::max(samples / kAdjSamples, std::min(kAdjFill / all, samples / kAdjLeast))}));
        hipLaunchKernelGGL((k_adj2d_tile<SS>), dim3(tiles, 1, (unsigned)(G * batch)),
                           dim3(kMaxBlock), 0, s, accimg, (const typename SS::raw *)sinogram,
                           plan->d_ageo, plan->d_ev, plan->d_ns, parts, nx, ny, D, A, G);
        const size_t one = (size_t)nx * ny;
        hipLaunchKernelGGL((k_adj2d_finish<SV>),
                           dim3((unsigned)((one + kMaxBlock - 1) / kMaxBlock), (unsigned)batch),
                           dim3(kMaxBlock), 0, s, (typename SV::raw *)volume, accimg, parts, one);
        CMI_HIP_TRY(hipGetLastError());
        return CMI_OK;
    });
    const hipError_t fe = hipFreeAsync(scratch, s);
    if (st != CMI_OK) return st;
    CMI_HIP_TRY(fe);
    return CMI_OK;
}

} // extern "C"
