// 3D cone-beam projectors for gfx950: plan, forward ray march, voxel-driven backprojection
// (reference and geometry-matched projection) and the transposed ray march.
//
// Data layout in HBM
//   plan tables  fgeo [A] FwdGeom (FP64)     detector pixel (0,0), u/v steps, source (voxel frame)
//                mref [A][12] float          reference-mode projection matrix (see bp_matrices)
//                mmat [A][12] float          geometry-matched projection matrix
//                mfdk [A][12] float          matched matrix scaled so that W = (depth / DSO)
//                fast [A] int                axis (0 x, 1 y, 2 z) the detector's v step follows most
//                                            closely: the forward reads the copy in which it is fastest
//   per call     forward:  [B][copies] volume with a 2-voxel zero border, one copy per fast axis
//                          in use: x fastest [z][y][x], y fastest [z][x][y], z fastest [y][x][z]
//                backward: [B][A][V+4][U+4]      panels with a 2-pixel zero border
//                adjoint:  per-ray march table [2][A][V][U] float4 (kernel k_ray_table3d)
//
// Forward rays take their discrete quantities (hit, step count) from an FP64 set-up in the
// kernel, identical to the host oracle's, then march in FP32 from the ray's midpoint in
// volume-centred padded coordinates, summing by slabs of slices (or blocks of 32 samples).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <memory>
#include <type_traits>
#include <vector>

#include "bp_tiles.hpp"
#include "cmi_internal.hpp"
#include "geometry3d.hpp"
#include "stage_index.hpp"

using namespace cmi;
using cmi::cone3d::FwdGeom;

struct cmi_plan3d {
    int device = 0;
    int vol_prec = CMI_F32, det_prec = CMI_F32;
    cone3d::Desc g{};
    int64_t A = 0;
    uint64_t total_samples = 0;
    uint64_t table_bytes = 0;
    FwdGeom *d_fgeo = nullptr;
    int *d_fast = nullptr;      // [A] fast axis of each angle's volume copy
    int copy_slot[3] = {-1, -1, -1}; // per fast axis: its copy's index, -1 if no angle uses it
    int ncopies = 0;
    float *d_mref = nullptr;
    float *d_mmat = nullptr;
    float *d_mfdk = nullptr;
    bool ycols[3] = {false, false, false}; // per cmi_bp3d_mode: U and W rows free of y
    bool views = false; // built from ASTRA-like views: reference mode = matched, no FDK mode
    // per cmi_bp3d_mode: smallest W of the mode's matrices over the volume's corner voxels and
    // all angles (W is affine in the voxel, so this bounds it over the volume); the transpose
    // of the backprojection needs it positive
    double wmin[3] = {0.0, 0.0, 0.0};
};

namespace {

constexpr int kPad = 2;        // zero border of staged volumes and panels
constexpr int kMaxBlock = 256; // threads per workgroup every kernel here is compiled for
constexpr int kSumBlock = 32;  // samples per partial sum in the forward march
static_assert(kPad == kPadDet, "panels are staged with the backprojector's border");

// ---------------------------------------------------------------- ray parameters ----------

// FP32 march parameters of one ray in centred padded coordinates (voxel coordinate + kPad
// minus the padded volume's integer centre c0): midpoint m, step st, first index j0 = -nst/2,
// sample count n = nst + 1. Shared by the forward march and its transpose so both see the same
// FP32 positions.
struct March3 {
    float m[3], st[3];
    float j0;
    int n;
};

__device__ __forceinline__ March3 march_params(const FwdGeom &g, int nx, int ny, int nz, int iu,
                                               int iv, int Wp, int Hp, int Dp) {
    March3 p{};
    const cone3d::Ray3 r = cone3d::setup_ray3(g, nx, ny, nz, iu, iv);
    if (!r.hit) return p; // n = 0
    const int64_t im = r.nst / 2;
    const double tm = r.tmin + (double)im * r.dt;
    const double c0[3] = {(double)(Wp / 2), (double)(Hp / 2), (double)(Dp / 2)};
    for (int d = 0; d < 3; ++d) {
        p.m[d] = (float)(r.s[d] + tm * r.d[d] + (double)kPad - c0[d]);
        p.st[d] = (float)(r.dt * r.d[d]);
    }
    p.j0 = (float)(-im);
    p.n = (int)(r.nst + 1);
    return p;
}

__global__ __launch_bounds__(kMaxBlock) void k_count3d(const FwdGeom *__restrict__ geo, int U,
                                                       int V, int nx, int ny, int nz,
                                                       unsigned long long *__restrict__ total) {
    const int iu = blockIdx.x * blockDim.x + threadIdx.x;
    const int iv = blockIdx.y;
    const int a = blockIdx.z;
    unsigned long long n = 0;
    if (iu < U) {
        const cone3d::Ray3 r = cone3d::setup_ray3(geo[a], nx, ny, nz, iu, iv);
        n = r.hit ? (unsigned long long)(r.nst + 1) : 0ull;
    }
    for (int off = 32; off > 0; off >>= 1) n += __shfl_xor(n, off, 64);
    if ((threadIdx.x & 63) == 0 && n) atomicAdd(total, n);
}

// ---------------------------------------------------------------- staging -----------------

// pad[b][zp][yp][xp] = vol[b][zp-2][yp-2][xp-2], 0 in the border.
template <class S>
__global__ __launch_bounds__(kMaxBlock) void k_stage3d(const typename S::raw *__restrict__ vol,
                                                       typename S::raw *__restrict__ pad, int nx,
                                                       int ny, int nz, int Wp, int Hp, int Dp) {
    using raw = typename S::raw;
    const int xp = blockIdx.x * blockDim.x + threadIdx.x;
    if (xp >= Wp) return;
    const int yp = blockIdx.y;
    const int zp = blockIdx.z % Dp;
    const size_t b = blockIdx.z / Dp;
    const int x = xp - kPad, y = yp - kPad, z = zp - kPad;
    raw v = (raw)0.0f;
    if (x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz)
        v = vol[((b * nz + z) * ny + y) * (size_t)nx + x];
    pad[((b * Dp + zp) * Hp + yp) * (size_t)Wp + xp] = v;
}

// Copy with fast axis F = 1 (y) or 2 (z) and x as the middle axis: for each slow coordinate
// (z for F = 1, y for F = 2), dst[slow][xp][fp] = pad(xp, yp, zp), transposed through LDS in
// 32 x 32 tiles (reads along x, writes along the fast axis).
template <class S, int F>
__global__ __launch_bounds__(kMaxBlock) void k_stage3d_t(const typename S::raw *__restrict__ vol,
                                                         typename S::raw *__restrict__ dst,
                                                         int nx, int ny, int nz, int Wp, int Hp,
                                                         int Dp) {
    static_assert(F == 1 || F == 2, "transposed copies have y or z fastest");
    using raw = typename S::raw;
    __shared__ raw tile[32][33];
    const int Ef = F == 1 ? Hp : Dp, Es = F == 1 ? Dp : Hp;
    const int sp = blockIdx.z % Es;
    const size_t b = blockIdx.z / Es;
    const int xp0 = blockIdx.x * 32, fp0 = blockIdx.y * 32;
    const raw *src = vol + b * (size_t)nx * ny * nz;
    raw *out = dst + (size_t)sp * Wp * Ef;
    for (int r = threadIdx.y; r < 32; r += 8) { // r: fast-axis offset, threadIdx.x: x offset
        const int xp = xp0 + threadIdx.x, fp = fp0 + r;
        const int yp = F == 1 ? fp : sp, zp = F == 1 ? sp : fp;
        const int x = xp - kPad, y = yp - kPad, z = zp - kPad;
        raw v = (raw)0.0f;
        if (x >= 0 && x < nx && y >= 0 && y < ny && z >= 0 && z < nz)
            v = src[((size_t)z * ny + y) * nx + x];
        tile[r][threadIdx.x] = v;
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) { // r: x offset, threadIdx.x: fast-axis offset
        const int xp = xp0 + r, fp = fp0 + threadIdx.x;
        if (xp < Wp && fp < Ef) out[(size_t)xp * Ef + fp] = tile[threadIdx.x][r];
    }
}

// ppad[b][a][vp][up] = sino[b][a][vp-2][up-2], 0 in the border. Flat over the n destination
// elements, four consecutive ones per thread with one vector store (its offset is a multiple
// of four elements; the scratch stack is allocated with at least that alignment); the source
// row is followed element by element.
template <class S>
__global__ __launch_bounds__(kMaxBlock) void k_stage_panel(const typename S::raw *__restrict__ sino,
                                                           typename S::raw *__restrict__ ppad,
                                                           int U, int V, uint64_t n) {
    using raw = typename S::raw;
    struct alignas(4 * sizeof(raw)) Four {
        raw v[4];
    };
    const uint64_t i0 = ((uint64_t)blockIdx.x * kMaxBlock + threadIdx.x) * 4;
    if (i0 >= n) return;
    const int Up = U + 2 * kPad, Vp = V + 2 * kPad;
    StageIndex at = stage_index(i0, Up, Vp, n <= 0xffffffffull); // at.a = b * A + a
    Four f;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        const int u = at.up - kPad, v = at.vp - kPad;
        raw val = (raw)0.0f;
        if (i0 + k < n && u >= 0 && u < U && v >= 0 && v < V)
            val = sino[(at.a * V + v) * (size_t)U + u];
        f.v[k] = val;
        stage_next(at, Up, Vp);
    }
    if (i0 + 4 <= n) {
        *reinterpret_cast<Four *>(ppad + i0) = f;
    } else {
        for (uint64_t k = 0; i0 + k < n; ++k) ppad[i0 + k] = f.v[k];
    }
}

// ---------------------------------------------------------------- forward -----------------

// Trilinear interpolation of four pairs along the fast axis, at fractions ff, fm, fl: p00 (m, l),
// p10 (m + 1, l), p01 (m, l + 1), p11 (m + 1, l + 1).
__device__ __forceinline__ float trilerp(const Pair &p00, const Pair &p10, const Pair &p01,
                                         const Pair &p11, float ff, float fm, float fl) {
    const float a00 = lerp_pair(p00, ff), a10 = lerp_pair(p10, ff);
    const float a01 = lerp_pair(p01, ff), a11 = lerp_pair(p11, ff);
    const float b0 = fmaf(fm, a10 - a00, a00);
    const float b1 = fmaf(fm, a11 - a01, a01);
    return fmaf(fl, b1 - b0, b0);
}

// Trilinear sample at centred padded coordinates (f, m, l) along the copy's fast, middle and
// slow axes. `cofs` is the element offset of the copy's centre; sM, sL, sML are the byte strides
// of one step along the middle axis, the slow axis, and both.
template <class SI>
__device__ __forceinline__ float sample3d(rsrc_t R, float f, float m, float l, int Ef, int Em,
                                         int cofs, int sM, int sL, int sML) {
    const float i_f = floorf(f), i_m = floorf(m), i_l = floorf(l);
    const int o = __mul24(__mul24((int)i_l, Em) + (int)i_m, Ef) + (int)i_f + cofs;
    return trilerp(buf_pair<SI>(R, o, 0), buf_pair<SI>(R, o, sM), buf_pair<SI>(R, o, sL),
                   buf_pair<SI>(R, o, sML), f - i_f, m - i_m, l - i_l);
}

// LDS-staged march. The rays of a workgroup (16 x 16 detector pixels of one projection) lie
// inside the pyramid spanned by its four corner rays. The workgroup marches along the axis K
// that its rays follow most closely, in slabs of kSlab slices of lower taps: per slab it stages
// into LDS the box of voxels that the pyramid's samples there can tap (the corner rays'
// crossings of the slab's two bounding planes, one voxel of margin for FP32 positions, and the
// upper taps), read in 16-byte row pieces from the volume copy whose fastest axis P is not K,
// and every ray takes its samples whose lower tap lies in the slab from there, in its own order
// j = 0 .. n - 1, slab after slab: positions and trilinear weights are those of a plain per-ray
// march, and the ray's sum adds one partial sum per slab (at most about 2 kSlab samples each).
// Slabs whose box does not fit, and workgroups whose rays do not all advance the same way along K
// or whose K is the copy's fast axis, read global memory instead, with the same arithmetic (the
// latter in blocks of kSumBlock samples).
// Every sample of a staged slab lies in its box, at any distance of the source: the corner rays are
// held as their crossings of the volume's middle plane and their slopes along K, both evaluated in
// FP64, and a box that fits has slopes below 25 over at most 2050 slices either way, so FP32 puts
// the crossings less than 0.01 voxels off; the samples' own positions, from FP64 midpoints, are
// less than 0.001 off. kBoxMargin covers both. (With the rays from their source in FP32, sources
// from 10^6 voxels on lost a margin's width: workgroups had to march from global memory, and of
// those that did not, some still read past their boxes.)
// A wavefront covers 4 x 16 detector pixels, the 16 along v, and the copy read is the one
// whose fastest axis v follows (fast[a]), so that a wavefront's rows of a staged box are runs
// of consecutive voxels.
//
// The kernel is bound by VALU issue (1.55 wavefront instructions per clock and CU for fma, add and
// mul of vector registers, 0.93 for conversions, floors, shifts, compares and whatever reads a
// scalar register), with LDS at 0.7 of its rate. So:
// * a sample's LDS address is three fma: the byte strides and the offset are held as FP32
//   subnormals, n 2^-149, whose bit pattern is the integer n; products with the integral floors
//   and their sums are exact below 2^23, and the sum's bits are the address (this needs FP32
//   subnormals, which the compiler keeps unless told otherwise). Fractions are p - floor(p).
// * the boxes of up to 64 slabs are found at once, one slab per lane, and read from the lanes.
// * a thread stages quads tid, tid + 256, ... of the box's rows laid end to end: no lane idles in
//   rows shorter than a power of two, and the LDS address is the quad's number.
// * a slab's samples run in a loop counted by the wavefront's smallest count, in a scalar
//   register, and a remainder counted per lane.
// At 256^3 x 360, 384^2 panel: 15.0 -> 10.1 ms with these and boxes a voxel narrower on every
// side (62 -> 45 VALU instructions per wavefront's sample, 9 % -> 2 % of the slabs not staged).
// sino[b][a][iv][iu] = sum_{i=0..nst} trilinear(vol, s + (tmin + i dt) d)  (forward_3d.hpp:87-93)
constexpr int kSlab = 10;         // slices of lower taps per slab
// floats of one staged box (20 KiB). A smaller box keeps more workgroups per CU and sends more
// slabs to the global path. (slices, floats) at 256^3 x 360 on a dense volume: (8, 3072) 11.3 ms,
// (8, 4096) 11.2, (8, 5120) 11.2, (10, 4096) 11.3, (10, 5120) 10.9, (12, 6144) 11.3; two samples
// per turn of the loop 11.1 to 11.2, and 64 VGPRs for eight wavefronts per SIMD 14.8 (spills).
constexpr int kBoxCells = 5120;
constexpr float kBoxMargin = 0.0625f; // voxels around the corner rays' crossings
constexpr unsigned kFwdGroup = 32; // projections per group in the workgroup order

template <class SI, class SS>
__global__ __launch_bounds__(kMaxBlock) void k_fwd3d(const typename SI::raw *__restrict__ pad,
                                                          const FwdGeom *__restrict__ geo,
                                                          const int *__restrict__ fast, int slot0,
                                                          int slot1, int slot2, int ncopies,
                                                          int nx, int ny, int nz, int U, int V,
                                                          int A,
                                                          typename SS::raw *__restrict__ sino) {
    __shared__ float4 box4[kBoxCells / 4];
    __shared__ float cdir[4][3];     // corner rays: direction
    __shared__ float4 cross[4];      // on centred slice k of K: P = x + y k, Q = z + w k
    __shared__ int red[2][kMaxBlock / 64];
    const int tid = threadIdx.x;
    // XCD-aware order. Workgroups are dealt to the 8 XCDs in turn, so dispatch slot hw runs
    // on XCD hw % 8; logical index li gives each XCD a contiguous share of the order below.
    // In that order kFwdGroup consecutive projections of one tile come first, then the tiles
    // (u fastest), then the next group of projections: the 256 or so workgroups resident on an
    // XCD cover about 8 tiles over 32 neighbouring projections, whose pyramids overlap, so
    // their staged boxes share L2 (21.2 -> 18.8 ms at 256^3 against tiles first; projections
    // first across all 360 was 19.8 ms).
    const unsigned gx = gridDim.x, gy = gridDim.y;
    const unsigned nwg = gx * gy * gridDim.z;
    const unsigned hw = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const unsigned n8 = nwg & ~7u;
    const unsigned li = hw < n8 ? (hw & 7u) * (n8 >> 3) + (hw >> 3) : hw;
    unsigned tx, ty, tz;
    {
        const unsigned T = gx * gy, AT = (unsigned)A * T, G = kFwdGroup;
        const unsigned bb = li / AT, l = li % AT;
        const unsigned full = ((unsigned)A / G) * G * T; // workgroups in whole groups
        unsigned t, ai;
        if (l < full) {
            const unsigned r = l % (G * T);
            ai = l / (G * T) * G + r % G;
            t = r / G;
        } else { // the last, partial group
            const unsigned r = l - full, Gl = (unsigned)A - (unsigned)A / G * G;
            ai = (unsigned)A / G * G + r % Gl;
            t = r / Gl;
        }
        tx = t % gx;
        ty = t / gx;
        tz = ai + (unsigned)A * bb;
    }
    const int iu0 = (int)tx * 16, iv0 = (int)ty * 16;
    // a wavefront covers 4 x 16 pixels, consecutive lanes along v
    const int iu = iu0 + (tid >> 4), iv = iv0 + (tid & 15);
    const bool live = iu < U && iv < V;
    const int a = (int)tz % A;
    const size_t b = tz / A;
    const int Wp = nx + 2 * kPad, Hp = ny + 2 * kPad, Dp = nz + 2 * kPad;
    // the corner ray of lanes 0..3
    const double cu = (double)((tid & 1) ? min(iu0 + 15, U - 1) : iu0);
    const double cv = (double)((tid & 2) ? min(iv0 + 15, V - 1) : iv0);
    if (tid < 4) {
        const FwdGeom &g = geo[a];
        for (int d = 0; d < 3; ++d)
            cdir[tid][d] = (float)(g.org[d] + cu * g.du[d] + cv * g.dv[d] - g.src[d]);
    }
    March3 p{};
    if (live) p = march_params(geo[a], nx, ny, nz, iu, iv, Wp, Hp, Dp);
    // copy axes (fast, middle, slow): x fastest (x, y, z), y fastest (y, x, z), z fastest (z, x, y)
    // wave-uniform (so that the buffer resource below is a scalar one)
    const int F = __builtin_amdgcn_readfirstlane(fast[a]);
    const int M = F == 0 ? 1 : 0, L = F == 2 ? 1 : 2;
    const int slot = F == 0 ? slot0 : F == 1 ? slot1 : slot2;
    // component d of a three-vector without indexing a local array (which would live in
    // scratch memory)
    auto pick = [](auto v0, auto v1, auto v2, int d) { return d == 0 ? v0 : d == 1 ? v1 : v2; };
    const int Ef = pick(Wp, Hp, Dp, F), Em = pick(Wp, Hp, Dp, M), El = pick(Wp, Hp, Dp, L);
    const uint32_t one = (uint32_t)Wp * Hp * Dp;
    const rsrc_t R = make_rsrc(pad + (b * ncopies + slot) * one, bytes_of<SI>(one));
    constexpr int es = (int)sizeof(typename SI::raw);
    const int sM = Ef * es, sL = Ef * Em * es, sML = sL + sM;
    const int cofs = ((El / 2) * Em + Em / 2) * Ef + Ef / 2;
    const float mf = pick(p.m[0], p.m[1], p.m[2], F), mm = pick(p.m[0], p.m[1], p.m[2], M),
                ml = pick(p.m[0], p.m[1], p.m[2], L);
    const float tf = pick(p.st[0], p.st[1], p.st[2], F), tm = pick(p.st[0], p.st[1], p.st[2], M),
                tl = pick(p.st[0], p.st[1], p.st[2], L);
    __syncthreads(); // corner rays
    // march axis K: the largest component of the corner rays' summed direction
    float ds[3];
    for (int d = 0; d < 3; ++d) ds[d] = cdir[0][d] + cdir[1][d] + cdir[2][d] + cdir[3][d];
    const int K = fabsf(ds[0]) >= fabsf(ds[1]) ? (fabsf(ds[0]) >= fabsf(ds[2]) ? 0 : 2)
                                               : (fabsf(ds[1]) >= fabsf(ds[2]) ? 1 : 2);
    const float sgn = ds[K] > 0.0f ? 1.0f : -1.0f;
    bool slab_ok = K != F;
    for (int c = 0; c < 4; ++c) slab_ok = slab_ok && cdir[c][K] * sgn > 0.0f;
    const int Q = 3 - K - F; // the third axis (when K != F)
    // padded index = centred coordinate + E / 2 on each axis
    const int cK = pick(Wp, Hp, Dp, K) / 2, cP = Ef / 2, cQ = pick(Wp, Hp, Dp, Q) / 2;
    const float mK = pick(p.m[0], p.m[1], p.m[2], K), tK = pick(p.st[0], p.st[1], p.st[2], K);
    const float mP = mf, tP = tf;
    const float mQ = pick(p.m[0], p.m[1], p.m[2], Q), tQ = pick(p.st[0], p.st[1], p.st[2], Q);
    // element strides of K and Q in the copy; and whether K is the copy's middle axis (then a
    // step in K is the trilinear m step, else the l step)
    const bool kmid = K == M;
    const int sK = kmid ? Ef : Ef * Em, sQ = kmid ? Ef * Em : Ef;

    float acc = 0.0f;
    const int n = p.n;
    float jf = p.j0;                       // the next sample (exact integers)
    const float jend = p.j0 + (float)n;    // one past the last
    // sample jf at the forward's position, from global memory
    auto global_sample = [&]() {
        return sample3d<SI>(R, fmaf(jf, tf, mf), fmaf(jf, tm, mm), fmaf(jf, tl, ml), Ef, Em,
                            cofs, sM, sL, sML);
    };
    // crossings of the corner rays with centred slice k along K: the smallest and largest padded
    // indices along P and Q
    auto section = [&](float k, float &p0, float &p1, float &q0, float &q1) {
        p0 = q0 = INFINITY;
        p1 = q1 = -INFINITY;
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            const float4 l = cross[c];
            const float pc = fmaf(k, l.y, l.x), qc = fmaf(k, l.w, l.z);
            p0 = fminf(p0, pc);
            p1 = fmaxf(p1, pc);
            q0 = fminf(q0, qc);
            q1 = fmaxf(q1, qc);
        }
        p0 += (float)cP, p1 += (float)cP, q0 += (float)cQ, q1 += (float)cQ;
    };
    // lower-tap K range of the workgroup's samples
    int klo = 0x7fffffff, khi = -0x7fffffff - 1;
    if (slab_ok) {
        if (tid < 4) {
            double pc, sp, qc, sq;
            cone3d::line_on_planes(geo[a], cu, cv, K, F, (double)(cK - kPad), pc, sp);
            cone3d::line_on_planes(geo[a], cu, cv, K, Q, (double)(cK - kPad), qc, sq);
            cross[tid] = make_float4((float)(pc + (double)(kPad - cP)), (float)sp,
                                     (float)(qc + (double)(kPad - cQ)), (float)sq);
        }
        if (n > 0) {
            const int k0 = floor_i32(fmaf(p.j0, tK, mK)) + cK;
            const int k1 = floor_i32(fmaf(jend - 1.0f, tK, mK)) + cK;
            klo = min(k0, k1);
            khi = max(k0, k1);
        }
        for (int off = 32; off > 0; off >>= 1) {
            klo = min(klo, __shfl_xor(klo, off, 64));
            khi = max(khi, __shfl_xor(khi, off, 64));
        }
        if ((tid & 63) == 0) {
            red[0][tid >> 6] = klo;
            red[1][tid >> 6] = khi;
        }
        __syncthreads();
        klo = min(min(red[0][0], red[0][1]), min(red[0][2], red[0][3]));
        khi = max(max(red[1][0], red[1][1]), max(red[1][2], red[1][3]));
    }
    if (!__builtin_amdgcn_readfirstlane((int)slab_ok)) {
        while (jf < jend) {
            const float je = fminf(jf + (float)kSumBlock, jend);
            float s0 = 0.0f;
            for (; jf < je; jf += 1.0f) s0 += global_sample();
            acc += s0;
        }
    } else {
        const int nslab = __builtin_amdgcn_readfirstlane(khi >= klo ? (khi - klo) / kSlab + 1 : 0);
        const float rtK = n > 0 ? 1.0f / tK : 0.0f;
        // lower taps K in [D0, D0 + kSlab - 1] of slab si; slabs follow the rays' direction
        auto first_slice = [&](int si) {
            return sgn > 0.0f ? klo + si * kSlab : khi - kSlab + 1 - si * kSlab;
        };
        // lane l's plan of slab si0 + l: the box's first indices along P and Q; quads per row and
        // rows per slice (0: not staged); a little over 2^20 / each, by which a product and a
        // shift give exact quotients of the numbers of the box's quads and rows
        int bP0 = 0, bQ0 = 0, bN = 0, bRN = 0, bRQ = 0;
        auto plan_slabs = [&](int si0) {
            const float k = (float)(first_slice(si0 + (tid & 63)) - cK);
            float p0, p1, q0, q1, u0, u1, v0, v1;
            section(k, p0, p1, q0, q1);
            section(k + (float)kSlab, u0, u1, v0, v1);
            constexpr float big = 16384.0f;
            auto floor_at = [](float v) {
                return floor_i32(__builtin_amdgcn_fmed3f(v, -big, big));
            };
            bP0 = floor_at(fminf(p0, u0) - kBoxMargin);
            bQ0 = floor_at(fminf(q0, v0) - kBoxMargin);
            // quads per row and rows per slice: to the upper taps of the largest lower ones
            const int NQ = (floor_at(fmaxf(p1, u1) + kBoxMargin) + 1 - bP0 + 4) >> 2;
            const int WQ = floor_at(fmaxf(q1, v1) + kBoxMargin) + 1 - bQ0 + 1;
            const bool fits = NQ <= kBoxCells / 4 && WQ <= kBoxCells / 4 &&
                              (kSlab + 1) * NQ * WQ <= kBoxCells / 4;
            bN = fits ? NQ | WQ << 16 : 0;
            bRN = (int)(0x1p20f * __builtin_amdgcn_rcpf((float)NQ)) + 1;
            bRQ = (int)(0x1p20f * __builtin_amdgcn_rcpf((float)WQ)) + 1;
        };
        // LDS byte address of the box
        const int box0 = (int)(uintptr_t)(__attribute__((address_space(3))) float4 *)box4;
        for (int si = 0; si < nslab; ++si) {
            if ((si & 63) == 0) plan_slabs(si);
            const int D0 = first_slice(si);
            const int P0 = __builtin_amdgcn_readlane(bP0, si & 63);
            const int Q0 = __builtin_amdgcn_readlane(bQ0, si & 63);
            const int nn = __builtin_amdgcn_readlane(bN, si & 63);
            const int NQ = nn & 0xffff, WQ = nn >> 16;
            if (nn) {
                const int rn = __builtin_amdgcn_readlane(bRN, si & 63);
                const int rq = __builtin_amdgcn_readlane(bRQ, si & 63);
                // quad e of the box is quad e - NQ r of row r = e / NQ, row r - WQ kk of slice
                // kk = r / WQ
                const int total = (kSlab + 1) * WQ * NQ;
                const int g0 = (D0 * sK + Q0 * sQ + P0) * es;
                Quad v[kBoxCells / 4 / kMaxBlock];
#pragma unroll
                for (int i = 0; i < kBoxCells / 4 / kMaxBlock; ++i) {
                    const int e = tid + i * kMaxBlock;
                    if (e < total) {
                        const int r = (int)(__umul24((unsigned)e, (unsigned)rn) >> 20);
                        const int kk = (int)(__umul24((unsigned)r, (unsigned)rq) >> 20);
                        const int qq = r - __mul24(kk, WQ), pq = e - __mul24(r, NQ);
                        v[i] = buf_quad_at<SI>(R, g0 + (kk * sK + qq * sQ + 4 * pq) * es);
                    }
                }
#pragma unroll
                for (int i = 0; i < kBoxCells / 4 / kMaxBlock; ++i) {
                    const int e = tid + i * kMaxBlock;
                    if (e < total)
                        box4[e] = make_float4(v[i].v[0], v[i].v[1], v[i].v[2], v[i].v[3]);
                }
            }
            __syncthreads(); // the box is staged
            // one past this ray's last sample in the slab: an estimate from its crossing of the
            // slab's far plane, put right by the floors of the samples either side of it, so that
            // a sample is in the slab exactly when its lower tap is
            const int kofs = cK - D0;
            const float bK = (float)((sgn > 0.0f ? D0 + kSlab : D0) - cK);
            float je = fminf(fmaxf(p.j0 + ceilf(fmaf(bK - mK, rtK, -p.j0)), jf), jend);
            auto in_slab = [&](float jj) {
                return (unsigned)(floor_i32(fmaf(jj, tK, mK)) + kofs) < (unsigned)kSlab;
            };
            if (je < jend && in_slab(je)) je += 1.0f;
            else if (je > jf && !in_slab(je - 1.0f)) je -= 1.0f;
            if (nn) {
                if (je > jf) {
                    // KM: K is the copy's middle axis (a step in K is the trilinear m step)
                    auto sample_slab = [&](auto km) {
                        constexpr bool KM = decltype(km)::value;
                        const int W4 = 16 * NQ, S4 = W4 * WQ; // bytes per row and per slice
                        const float fS = subnormal(S4), fW = subnormal(W4), f4 = subnormal(4);
                        const float fo =
                            subnormal(kofs * S4 + (cQ - Q0) * W4 + (cP - P0) * 4 + box0);
                        int m4 = KM ? S4 : W4, l4 = KM ? W4 : S4;
                        asm("" : "+v"(m4), "+v"(l4));
                        auto sample = [&](float jj) {
                            const float pK = fmaf(jj, tK, mK), pf = fmaf(jj, tP, mP),
                                        pq = fmaf(jj, tQ, mQ);
                            const float iK = floorf(pK), iP = floorf(pf), iQ = floorf(pq);
                            const int o =
                                __float_as_int(fmaf(iK, fS, fmaf(iQ, fW, fmaf(iP, f4, fo))));
                            auto pair = [](int q) {
                                const auto *c =
                                    (const __attribute__((address_space(3))) float *)(uintptr_t)
                                        (unsigned)q;
                                return Pair{c[0], c[1]};
                            };
                            const Pair p00 = pair(o), p10 = pair(o + m4), p01 = pair(o + l4),
                                       p11 = pair(o + m4 + l4);
                            const float fK = pK - iK, fQ = pq - iQ;
                            return trilerp(p00, p10, p01, p11, pf - iP, KM ? fK : fQ,
                                           KM ? fQ : fK);
                        };
                        float part = 0.0f;
                        // the wavefront's smallest count, over the lanes with any
                        const int cnt = (int)(je - jf);
                        int least = __builtin_amdgcn_readfirstlane(cnt);
                        for (;;) {
                            const unsigned long long less = __builtin_amdgcn_ballot_w64(cnt < least);
                            if (less == 0) break;
                            least = __builtin_amdgcn_readlane(cnt, __builtin_ctzll(less));
                        }
                        for (int i = 0; i < least; ++i, jf += 1.0f) part += sample(jf);
                        for (; jf < je; jf += 1.0f) part += sample(jf);
                        acc += part;
                    };
                    if (kmid) sample_slab(std::true_type{});
                    else sample_slab(std::false_type{});
                }
            } else {
                float part = 0.0f;
                for (; jf < je; jf += 1.0f) part += global_sample();
                acc += part;
            }
            __syncthreads(); // the box is read before the next slab is staged
        }
    }
    if (live) sino[((b * A + a) * V + iv) * (size_t)U + iu] = from_f32<SS>(acc);
}

// ---------------------------------------------------------------- adjoint -----------------

// Per-ray march table for the adjoint: rm = (m.xyz, j0), rs = (st.xyz, n as int bits), the same
// FP32 parameters k_fwd3d derives with march_params; n = 0 for rays that miss the volume.
__global__ __launch_bounds__(kMaxBlock) void k_ray_table3d(const FwdGeom *__restrict__ geo, int nx,
                                                          int ny, int nz, int U, int V,
                                                          float4 *__restrict__ rm,
                                                          float4 *__restrict__ rs) {
    const int iu = blockIdx.x * blockDim.x + threadIdx.x;
    const int iv = blockIdx.y;
    const int a = blockIdx.z;
    if (iu >= U) return;
    const int Wp = nx + 2 * kPad, Hp = ny + 2 * kPad, Dp = nz + 2 * kPad;
    const March3 p = march_params(geo[a], nx, ny, nz, iu, iv, Wp, Hp, Dp);
    const size_t r = ((size_t)a * V + iv) * U + iu;
    rm[r] = make_float4(p.m[0], p.m[1], p.m[2], p.j0);
    rs[r] = make_float4(p.st[0], p.st[1], p.st[2], __int_as_float(p.n));
}

// Largest |y| of each projection stack of a batch, in two steps: per stack b, kMaxParts
// workgroups each write the maximum of their grid-stride share to parts[b][*]; the adjoint
// reduces the kMaxParts values. Each volume of a batch gets its own fixed-point unit, so that
// its result does not depend on the other volumes.
constexpr int kMaxParts = 256;

template <class S>
__global__ __launch_bounds__(kMaxBlock) void k_absmax_parts(const typename S::raw *__restrict__ y,
                                                            size_t n, float *__restrict__ parts) {
    __shared__ float red[kMaxBlock / 64];
    y += (size_t)blockIdx.y * n;
    parts += (size_t)blockIdx.y * kMaxParts;
    float m = 0.0f;
    for (size_t i = (size_t)blockIdx.x * kMaxBlock + threadIdx.x; i < n;
         i += (size_t)kMaxParts * kMaxBlock)
        m = fmaxf(m, fabsf(to_f32<S>(y[i])));
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kMaxBlock / 64; ++w) m = fmaxf(m, red[w]);
        parts[blockIdx.x] = m;
    }
}

// Matched adjoint, tile-driven: a workgroup owns a kAT^3 voxel tile with accumulators in LDS and a
// group of angles. For each angle it projects the tile's box, grown by one voxel on each side (the
// samples whose trilinear footprint reaches the tile), through the geometry-matched matrices onto
// the panel; the rays through the covered pixels (plus one pixel of margin) are the candidates.
// Each candidate walks only its samples inside the grown box, at the forward's FP32 positions, and
// adds y * w to the tile voxels its footprint covers. The accumulators are fixed point in units
// of max|y| / 2^19: a contribution y * w is rounded to that grid (|term| <= 2^19) and added to a
// 32-bit LDS cell with an integer LDS atomic, which gfx950 executes about 45 times faster than an
// FP32 LDS atomic add (and 32-bit cells halve the LDS atomic traffic of 64-bit ones). Integer
// sums are exact, so the result does not depend on the order of the additions; the rounding of
// each term is at most max|y| 2^-20.
// Overflow: a ray adds at most two terms to a voxel (its samples are one apart along the
// dominant axis, so at most two have their lower corner within one voxel of it), and only rays
// through the projection of the voxel's 2 x 2 x 2 neighbourhood reach it. Per angle that
// projection is at most Du x Dv pixels, with Du <= 2 sum_i |du/dx_i| bounded over the grown box
// by (sum |m0..2| + max|u| sum |m8..10|) / min w from its corners (and Dv alike), so one angle
// adds at most 2 (Du + 2)(Dv + 2) terms to a voxel (2 per candidate where that is smaller).
// The workgroup keeps a running bound of these and, before it could pass 2^31 / 2^19, moves
// the 32-bit sums of its 16^3 voxels into 64-bit sums and clears the tile. The 64-bit sums live
// in a global array with one tile's worth per tile, not in registers: sixteen 64-bit registers per
// thread held the kernel at four wavefronts per SIMD, and without them it keeps six (48.0 -> 43.3
// ms at 256^3, bit-identical). A tile's only workgroup (gridDim.z == batch x tiles) writes them
// first and adds the tile to the volume once, in its storage type; where several angle groups
// share a tile, they add to them with integer atomics (cleared before) and k_adj3d_finish adds
// the sums, which are the same, to the volume.
//
// Bound by LDS atomics (eight per sample, two clocks per wavefront and CU each and almost as many
// in conflicts) and VALU issue (24 full, 12 half rate slots: LDS addresses by FMA on subnormals,
// bp_tiles.hpp, and no test per sample, kAT3Margin). 97 x 120 x 133 voxels, 90 views of 150 x 171:
// 2.16 ms with one workgroup per tile (504: 1.5 wavefronts per SIMD), 1.60 with the samples' loop
// as it is now, 0.73 with angle groups (LDS busy 77 %, 47 % of that in conflicts).
constexpr int kAT = 16;
// candidate rays of one wavefront are kPh pixels apart in u and v (at 256^3, six wavefronts per
// SIMD, tiles in XCD order: kPh 1: 47.1 ms, 2: 38.2; tiles in launch order: 2: 38.7, 3: 42.5,
// 4: 43.7, 5: 45.5, 6: 46.1)
constexpr int kPh = 2;
// Samples are walked over the steps whose positions lie in the grown box, widened by this share
// of a step for rounding: the lower corner of a sample lies in [-2, kAT + 1) on each axis.
constexpr float kAT3Margin = 0.01f;
// LDS tile: padded by one voxel before and after on each axis, so that every tap of a sample
// whose lower corner lies in [-1, kAT) on each axis lands in the array (taps outside the tile
// are added to the border and dropped): the eight taps are then immediate offsets from one LDS
// address. A corner one further out on x or y lands in the border of the row or slice beside,
// one further on z in kATGuard cells before or after the slices. The odd slice pitch spreads
// voxels that differ only in z over different banks.
constexpr int kATP = kAT + 2, kATRow = kATP, kATSlice = kATP * kATRow + 1;
constexpr int kATGuard = kATSlice + kATRow + 2;
constexpr int kATCells = kATP * kATSlice + 2 * kATGuard;
constexpr int kATOwn = kAT * kAT * kAT / kMaxBlock; // tile voxels per thread
static_assert(kAT * kAT * kAT % kMaxBlock == 0, "whole voxels per thread");
constexpr int kAdj3Bits = 19;                             // a term's bound: 2^kAdj3Bits units
constexpr int kAdj3Budget = (1 << (31 - kAdj3Bits)) - 16; // terms per voxel between drains
// Angle groups per tile. A group costs its workgroup's clearing of the LDS tile and 4096 64-bit
// atomics, as much as some thousand samples, so it is given kAdj3Samples of them (a tile's share of
// the plan's); or, as long as that leaves fewer than kAdj3Fill workgroups, kAdj3Least. Tiles differ in
// their rays (those near the source have many), so that many more than the 1536 workgroups which the
// GPU holds at once pay: to kAdj3Workgroups. us, with 1 / 2 / 4 / 8 / 16 / 32 / 64 groups, and what
// this rule takes: 97 x 120 x 133 x 90 views (504 tiles) 1315 / 948 / 880 / 698 / 702 / 684 / 753, 49;
// 128^3 x 40 views (512) of 192^2 487 / 423 / 399 / 358 / 357 / 459 / 521, 21; of 96^2 214 / 174 / 179 /
// 173 / 240 / 413 / 490, 5; of 48^2 166 / 128 / 138 / 154 / 188 / 275 / 319, 2; 48^3 x 60 of 18^2 (27)
// 240 / 138 / 79 / 54 / 43 / 44 / 57, 14.
// Groups need two launches more, about 9 us: tiles whose work, an angle counting for kAdj3Angle
// samples, is below kAdj3Alone have one. us, with 1 / 2 / 4 groups: 16^3 x 5 views of 12^2 36 / 47 / 48,
// x 9 51 / 47 / 47, x 2 of 30^2 43 / 48 / 48, x 3 59 / 52 / 48; 90^3 (216) x 5 of 67^2 46 / 50 / 56, x 9
// 61 / 57 / 62; 5^3 x 9 of 4^2 37 / 47 / 47, x 20 60 / 48 / 48.
// Where the tiles fill the GPU and the angles are few, a group is a sector of the circle, whose tiles
// near the source are neighbours in the order and fall to one or two XCDs: one group there. us, with
// 1 / 2 / 4 / 8 / 16 groups: 128^3 (512 tiles) of 640^2, 4 views 492 / 693 / 566 / 632 / 572, 12 views
// 1509 / 1934 / 2136 / 2142 / 1605, 24 views 2990 / 3681 / 3801 / 3393 / 3298; of 384^2, 12 views 482 /
// 604 / 567 / 598 / 484, 24 views 954 / 1118 / 1099 / 899 / 876; 192^3 (1728) x 12 of 288^2 373 / 376 /
// 376 / 495 / 616, x 24 of 960^2 8621 / 9602 / 10264 / 8793 / 8898; but 96^3 (216) x 12 of 288^2 393 /
// 307 / 299 / 288 / 241.
constexpr uint64_t kAdj3Samples = 10000, kAdj3Least = 1500, kAdj3Fill = 1024;
constexpr uint64_t kAdj3FullTiles = 512, kAdj3FewAngles = 24, kAdj3TilesPerAngle = 32;
constexpr uint64_t kAdj3Angle = 3000, kAdj3Alone = 40000;
constexpr uint64_t kAdj3Workgroups = 24576;

// vol[o] += a voxel's sum of fixed-point terms.
template <class SV>
__device__ __forceinline__ void adj3d_add(typename SV::raw *__restrict__ vol, size_t o,
                                          long long total, float ymax) {
    const float add = (float)((double)total * ((double)ymax * 0x1p-19));
    vol[o] = from_f32<SV>(to_f32<SV>(vol[o]) + add);
}

template <class SV, class SS>
__global__ __launch_bounds__(kMaxBlock) void k_adj3d(typename SV::raw *__restrict__ vol,
                                                     const typename SS::raw *__restrict__ sino,
                                                     const float4 *__restrict__ rm,
                                                     const float4 *__restrict__ rs,
                                                     const float *__restrict__ M,
                                                     const float *__restrict__ parts, int nx,
                                                     int ny, int nz, int U, int V, int A, int G,
                                                     long long *__restrict__ totals) {
    __shared__ unsigned int cells[kATCells];
    unsigned int *const tile = cells + kATGuard;
    const int tid = threadIdx.x;
    const int ntz = (nz + kAT - 1) / kAT;
    // XCD-aware order: workgroups are dealt to the 8 XCDs in turn, and logical index li gives
    // each XCD a contiguous run of tiles (x fastest) of an angle group, whose candidate rays
    // share L2
    int x0, y0, z0, g;
    size_t b, slot; // volume; the tile's place among all
    {
        const unsigned gx = gridDim.x, gy = gridDim.y, gz = gridDim.z;
        const unsigned nwg = gx * gy * gz;
        const unsigned hw = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
        const unsigned n8 = nwg & ~7u;
        const unsigned li = hw < n8 ? (hw & 7u) * (n8 >> 3) + (hw >> 3) : hw;
        const unsigned per = gx * gy * (unsigned)ntz;
        g = (int)(li / per % (unsigned)G);
        b = li / per / (unsigned)G;
        const unsigned l = li % per;
        slot = b * per + l;
        x0 = (int)(l % gx) * kAT;
        y0 = (int)((l / gx) % gy) * kAT;
        z0 = (int)(l / (gx * gy)) * kAT;
    }
    const int a0 = (int)((int64_t)g * A / G), a1 = (int)((int64_t)(g + 1) * A / G);
    // the tile's 64-bit voxel sums; G == 1: in global memory that this workgroup alone uses, none
    // before the first drain
    long long *own = totals + slot * (kAT * kAT * kAT);
    bool first = true;
    auto cell_of = [](int j) {
        return (j / (kAT * kAT) + 1) * kATSlice + ((j / kAT) % kAT + 1) * kATRow + j % kAT + 1;
    };
    auto share = [&](int i, long long v) {
        if (v != 0) atomicAdd((unsigned long long *)&own[i], (unsigned long long)v);
    };
    // the tile's voxel sums -> the 64-bit sums, then the tile (border included) cleared
    auto drain = [&]() {
        lds_barrier();
#pragma unroll 4
        for (int k = 0; k < kATOwn; ++k) {
            const int i = tid + k * kMaxBlock;
            const long long v = (int)tile[cell_of(i)];
            if (G > 1) share(i, v);
            else own[i] = first ? v : own[i] + v;
        }
        first = false;
        __syncthreads();
        for (int i = tid; i < kATCells; i += kMaxBlock) cells[i] = 0u;
        __syncthreads();
    };
    int bound = 0; // terms a voxel may have received since the last drain
    // fixed-point scale: max|y| of this volume's projections maps to 2^19
    float ymax = 0.0f;
    for (int i = tid & 63; i < kMaxParts; i += 64) ymax = fmaxf(ymax, parts[b * kMaxParts + i]);
    for (int off = 32; off > 0; off >>= 1) ymax = fmaxf(ymax, __shfl_xor(ymax, off, 64));
    const float yscale = ymax > 0.0f ? (float)(1 << kAdj3Bits) / ymax : 0.0f;
    for (int i = tid; i < kATCells; i += kMaxBlock) cells[i] = 0u;
    const int Wp = nx + 2 * kPad, Hp = ny + 2 * kPad, Dp = nz + 2 * kPad;
    // centred padded coordinate p -> voxel index floor(p) + c
    const int cx = Wp / 2 - kPad, cy = Hp / 2 - kPad, cz = Dp / 2 - kPad;
    // byte strides and the address of floor(p) = (0, 0, 0), as subnormals
    const float fcol = subnormal(4), frow = subnormal(4 * kATRow), fslice = subnormal(4 * kATSlice);
    const float fofs = subnormal((int)(uintptr_t)(__attribute__((address_space(3))) unsigned *)tile +
                                 4 * ((cx - x0 + 1) + (cy - y0 + 1) * kATRow +
                                      (cz - z0 + 1) * kATSlice));
    // samples reaching the tile: floor(p) + c in [t0 - 1, t0 + kAT - 1] on each axis
    const float lox = (float)(x0 - 1 - cx), loy = (float)(y0 - 1 - cy), loz = (float)(z0 - 1 - cz);
    const float hix = lox + (float)(kAT + 1), hiy = loy + (float)(kAT + 1),
                hiz = loz + (float)(kAT + 1);
    // the grown box's corner this lane projects (centred voxel index of the matrices)
    const int c8 = tid & 7, k8 = (tid & 63) >> 3;
    const float qx = (float)((c8 & 1) ? x0 + kAT : x0 - 1) - (float)((nx - 1) / 2.0);
    const float qy = (float)((c8 & 2) ? y0 + kAT : y0 - 1) - (float)((ny - 1) / 2.0);
    const float qz = (float)((c8 & 4) ? z0 + kAT : z0 - 1) - (float)((nz - 1) / 2.0);
    const typename SS::raw *sb = sino + b * (size_t)A * V * U;
    // By lane, for the angle of its eight lanes: the candidates' first column and row, their
    // numbers, and the most terms that the angle adds to a voxel
    int cu0 = 0, cv0 = 0, cnu = 0, cnv = 0, cterms = 0;
    __syncthreads();
    for (int a = a0; a < a1; ++a) {
        const int sel = 8 * ((a - a0) & 7);
        if (sel == 0) {
            const float *m = M + 12 * min(a + k8, A - 1);
            const float Uh = fmaf(m[0], qx, fmaf(m[1], qy, fmaf(m[2], qz, m[3])));
            const float Vh = fmaf(m[4], qx, fmaf(m[5], qy, fmaf(m[6], qz, m[7])));
            const float Wh = fmaf(m[8], qx, fmaf(m[9], qy, fmaf(m[10], qz, m[11])));
            const float rw = __builtin_amdgcn_rcpf(Wh);
            float u0 = Uh * rw, u1 = u0, v0 = Vh * rw, v1 = v0, wm = Wh;
            int ok = Wh > 0.0f ? 1 : 0;
#pragma unroll
            for (int off = 1; off < 8; off <<= 1) {
                u0 = fminf(u0, __shfl_xor(u0, off, 64));
                u1 = fmaxf(u1, __shfl_xor(u1, off, 64));
                v0 = fminf(v0, __shfl_xor(v0, off, 64));
                v1 = fmaxf(v1, __shfl_xor(v1, off, 64));
                ok = min(ok, __shfl_xor(ok, off, 64));
                wm = fminf(wm, __shfl_xor(wm, off, 64));
            }
            // no bound where a corner is not in front of the source: all rays, and 2^30 terms
            cu0 = cv0 = 0, cnu = U, cnv = V, cterms = 1 << 30;
            if (ok) {
                const float ua = fmaxf(fabsf(u0), fabsf(u1)), va = fmaxf(fabsf(v0), fabsf(v1));
                const float su = fabsf(m[0]) + fabsf(m[1]) + fabsf(m[2]);
                const float sv = fabsf(m[4]) + fabsf(m[5]) + fabsf(m[6]);
                const float sw = fabsf(m[8]) + fabsf(m[9]) + fabsf(m[10]);
                // 1 % margin for the approximate reciprocals; the +2 covers the pixel count of an
                // interval (floor + 1) and rays that FP32 positions put one pixel further
                const float du = 2.02f * (su + ua * sw) / wm, dv = 2.02f * (sv + va * sw) / wm;
                if (du < 1024.0f && dv < 1024.0f) cterms = 2 * ((int)du + 2) * ((int)dv + 2);
                if (u1 < -2.0f || u0 > (float)(U + 1) || v1 < -2.0f || v0 > (float)(V + 1)) {
                    cnu = 0;
                } else {
                    cu0 = max(0, (int)ceilf(u0) - 1);
                    cnu = min(U - 1, (int)floorf(u1) + 1) - cu0 + 1;
                    cv0 = max(0, (int)ceilf(v0) - 1);
                    cnv = min(V - 1, (int)floorf(v1) + 1) - cv0 + 1;
                }
            }
        }
        const int niu = __builtin_amdgcn_readlane(cnu, sel), niv = __builtin_amdgcn_readlane(cnv, sel);
        if (niu <= 0 || niv <= 0) continue;
        const int iu0 = __builtin_amdgcn_readlane(cu0, sel), iv0 = __builtin_amdgcn_readlane(cv0, sel);
        // Candidates in phase order: phase (pu, pv) in [0, kPh)^2 holds the rays
        // (pu + kPh qu, pv + kPh qv), so the consecutive candidates of a wavefront are kPh
        // pixels apart in u and v and their samples' taps rarely meet in one atomic instruction
        // (LDS serialises lanes that add to the same address). Padding the phases to equal
        // size leaves holes past the rectangle's edge, which are skipped.
        const int nqu = (niu + kPh - 1) / kPh, nqv = (niv + kPh - 1) / kPh;
        const int nq = nqu * nqv, nc = kPh * kPh * nq;
        const float rnqu = __builtin_amdgcn_rcpf((float)nqu);
        // passes of kMaxBlock candidates, the same for the whole workgroup; a pass adds at most
        // two terms per candidate to a voxel, and the angle at most cterms in all
        int allowance = __builtin_amdgcn_readlane(cterms, sel);
        for (int cb = 0; cb < nc; cb += kMaxBlock) {
            const int inc = min(2 * min(kMaxBlock, nc - cb), allowance);
            allowance -= inc;
            if (bound + inc > kAdj3Budget) {
                drain();
                bound = 0;
            }
            bound += inc;
            const int c = cb + tid;
            if (c >= nc) continue;
            int ph = 0, rq = c;
#pragma unroll
            for (int u = 1; u < kPh * kPh; ++u)
                if (rq >= nq) ph = u, rq -= nq;
            // rq / nqu, off by one at most before the correction
            int qv = (int)((float)rq * rnqu), qu = rq - qv * nqu;
            if (qu < 0) --qv, qu += nqu;
            if (qu >= nqu) ++qv, qu -= nqu;
            const int lu = (ph % kPh) + kPh * qu, lv = (ph / kPh) + kPh * qv;
            if (lu >= niu || lv >= niv) continue;
            const int iu = iu0 + lu, iv = iv0 + lv;
            const size_t r = ((size_t)a * V + iv) * U + iu;
            const float4 s4 = rs[r];
            const float4 m4 = rm[r];
            const float y = to_f32<SS>(sb[r]) * yscale; // |y| <= 2^19
            const int n = __float_as_int(s4.w);
            if (n <= 0 || y == 0.0f) continue;
            // jf range with p in [lo, hi) on every axis
            const float jlast = m4.w + (float)(n - 1);
            float jlo = m4.w, jhi = jlast;
            const float st[3] = {s4.x, s4.y, s4.z}, mm[3] = {m4.x, m4.y, m4.z};
            const float lo[3] = {lox, loy, loz}, hi[3] = {hix, hiy, hiz};
            bool empty = false;
#pragma unroll
            for (int d = 0; d < 3; ++d) {
                if (st[d] != 0.0f) {
                    const float r0 = __builtin_amdgcn_rcpf(st[d]);
                    const float t1 = (lo[d] - mm[d]) * r0, t2 = (hi[d] - mm[d]) * r0;
                    jlo = fmaxf(jlo, fminf(t1, t2) - kAT3Margin);
                    jhi = fminf(jhi, fmaxf(t1, t2) + kAT3Margin);
                } else if (mm[d] < lo[d] || mm[d] >= hi[d]) {
                    empty = true;
                }
            }
            if (empty) continue;
            const float jend = floorf(jhi);
            for (float jf = ceilf(jlo); jf <= jend; jf += 1.0f) {
                // the forward's own positions (k_fwd3d)
                const float px = fmaf(jf, s4.x, m4.x), py = fmaf(jf, s4.y, m4.y),
                            pz = fmaf(jf, s4.z, m4.z);
                const float ix = floorf(px), iy = floorf(py), iz = floorf(pz);
                const float fx = px - ix, fy = py - iy, fz = pz - iz;
                // the eight trilinear weights times y, as differences of products
                const float x1 = y * fx, x0w = y - x1;
                const float y01 = x0w * fy, y00 = x0w - y01, y11 = x1 * fy, y10 = x1 - y11;
                const float z00 = y00 * fz, z10 = y10 * fz, z01 = y01 * fz, z11 = y11 * fz;
                const float w[8] = {y00 - z00, y10 - z10, y01 - z01, y11 - z11,
                                    z00,       z10,       z01,       z11};
                auto *const t = (__attribute__((address_space(3))) unsigned *)(uintptr_t)
                    __float_as_uint(fmaf(iz, fslice, fmaf(iy, frow, fmaf(ix, fcol, fofs))));
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    lds_add(t + (k >> 2) * kATSlice + ((k >> 1) & 1) * kATRow + (k & 1),
                            (unsigned int)round_i32(w[k]));
            }
        }
    }
    lds_barrier();
    if (G > 1) {
#pragma unroll 4
        for (int k = 0; k < kATOwn; ++k) {
            const int i = tid + k * kMaxBlock;
            share(i, (int)tile[cell_of(i)]);
        }
        return;
    }
#pragma unroll 4
    for (int k = 0; k < kATOwn; ++k) {
        const int i = tid + k * kMaxBlock;
        const long long total = (first ? 0ll : own[i]) + (int)tile[cell_of(i)];
        const int lx = i % kAT, ly = (i / kAT) % kAT, lz = i / (kAT * kAT);
        const int X = x0 + lx, Y = y0 + ly, Z = z0 + lz;
        if (X < nx && Y < ny && Z < nz)
            adj3d_add<SV>(vol, ((b * nz + Z) * ny + Y) * (size_t)nx + X, total, ymax);
    }
}

// vol += the tiles' sums (k_adj3d with several angle groups). A workgroup per tile, as dealt there.
template <class SV>
__global__ __launch_bounds__(kMaxBlock) void k_adj3d_finish(typename SV::raw *__restrict__ vol,
                                                            const float *__restrict__ parts,
                                                            int nx, int ny, int nz,
                                                            const long long *__restrict__ totals) {
    const int ntz = (nz + kAT - 1) / kAT;
    const int x0 = (int)blockIdx.x * kAT, y0 = (int)blockIdx.y * kAT,
              z0 = (int)(blockIdx.z % ntz) * kAT;
    const size_t b = blockIdx.z / ntz;
    const size_t slot = blockIdx.x + gridDim.x * ((size_t)blockIdx.y +
                                                  gridDim.y * (size_t)blockIdx.z);
    float ymax = 0.0f;
    for (int i = threadIdx.x & 63; i < kMaxParts; i += 64)
        ymax = fmaxf(ymax, parts[b * kMaxParts + i]);
    for (int off = 32; off > 0; off >>= 1) ymax = fmaxf(ymax, __shfl_xor(ymax, off, 64));
#pragma unroll 4
    for (int k = 0; k < kATOwn; ++k) {
        const int i = threadIdx.x + k * kMaxBlock;
        const int X = x0 + i % kAT, Y = y0 + (i / kAT) % kAT, Z = z0 + i / (kAT * kAT);
        if (X < nx && Y < ny && Z < nz)
            adj3d_add<SV>(vol, ((b * nz + Z) * ny + Y) * (size_t)nx + X,
                          totals[slot * (kAT * kAT * kAT) + i], ymax);
    }
}

__global__ __launch_bounds__(kMaxBlock) void k_clear_sums(long long *__restrict__ p) {
    p[(size_t)blockIdx.x * kMaxBlock + threadIdx.x] = 0;
}

// ---------------------------------------------------------------- backprojection ----------

// Tile of the launch's workgroup over tiles of gridDim.x x gridDim.y x nzt per volume. XCD-aware
// order: workgroups are dealt to the 8 XCDs in turn, and logical index li gives each XCD a
// contiguous run of tiles (x fastest), whose panel footprints share L2 (256^3: 2.51
// -> 2.37 ms).
struct BpTile {
    int x, y, z;
    size_t b;
};
__device__ __forceinline__ BpTile bp_tile(int nzt) {
    const unsigned gx = gridDim.x, gy = gridDim.y, gz = gridDim.z;
    const unsigned nwg = gx * gy * gz;
    const unsigned hw = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
    const unsigned n8 = nwg & ~7u;
    const unsigned li = hw < n8 ? (hw & 7u) * (n8 >> 3) + (hw >> 3) : hw;
    const unsigned per = gx * gy * (unsigned)nzt;
    const unsigned l = li % per;
    return {(int)(l % gx), (int)((l / gx) % gy), (int)(l / (gx * gy)), li / per};
}

// A workgroup of 256 threads owns a tile of voxels, a run of y voxels per thread, and samples the
// angles' panel footprints from LDS (bp3d_run). YINV: no angle's U or W row depends on y.
// vol += sum over angles.
template <class SV, class SS, bool YINV, bool MATCHED, bool FDK>
__global__ __launch_bounds__(kMaxBlock) void k_bp3d(typename SV::raw *__restrict__ vol,
                                                    const typename SS::raw *__restrict__ ppad,
                                                    const float *__restrict__ M, int nx, int ny,
                                                    int nz, int U, int V, int A, float cx,
                                                    float cy, float cz) {
    constexpr int NY = kRun<YINV>;
    const BpTile t = bp_tile((nz + kTileZ<YINV> - 1) / kTileZ<YINV>);
    const int tx = t.x * kTileX, ty = t.y * kTileY, tz = t.z * kTileZ<YINV>;
    const int3 o = tile_run<YINV>();
    const int ix = tx + o.x, iy0 = ty + o.y, iz = tz + o.z;
    const size_t b = t.b;
    const uint32_t stack = (uint32_t)(U + 2 * kPad) * (V + 2 * kPad) * A;
    const rsrc_t R = make_rsrc(ppad + b * (size_t)stack, bytes_of<SS>(stack));
    float acc[NY];
#pragma unroll
    for (int y = 0; y < NY; ++y) acc[y] = 0.0f;
    bp3d_run<SS, YINV, MATCHED, FDK>(R, M, A, U, V, (float)ix - cx, (float)iy0 - cy,
                                     (float)iz - cz, (float)tx - cx, (float)ty - cy,
                                     (float)tz - cz, __builtin_amdgcn_readfirstlane(ny - iy0),
                                     acc);
    if (ix >= nx || iz >= nz) return;
#pragma unroll
    for (int y = 0; y < NY; ++y) {
        const int iy = iy0 + y;
        if (iy < ny) {
            const size_t i = ((b * nz + iz) * ny + iy) * (size_t)nx + ix;
            vol[i] = from_f32<SV>(to_f32<SV>(vol[i]) + acc[y]);
        }
    }
}

// ------------------------------------------------ transpose of the backprojection -------

// Bᵀ: the transpose of the voxel-driven backprojection (k_bp3d), the gradient of
// TorchBackprojection. The backprojection adds to voxel h, per projection a, the bilinear
// interpolation of panel a at (u, v) = (U/W, V/W) from the mode's matrix rows (cells floor(u)
// + {0, 1} and floor(v) + {0, 1}, weights 1 - fu, fu and 1 - fv, fv; cells outside the panel
// read zero), times 1/W^2 for FDK. So sino[a][j][i] = sum_h (those weights) vol[h].
// A workgroup owns a 16 x 16 pixel tile of one projection and gathers it. The voxels that reach
// the tile are those with (u, v) in [iu0 - 1, iu0 + 16) x [iv0 - 1, iv0 + 16): a pyramid from
// the source, bounded by the four lines through the source and that rectangle's corners. The
// workgroup marches through the volume along the axis K that the tile's central ray follows
// most closely, in chunks of kBTSlab slices. In each slice the pyramid's section is the
// quadrilateral where the corner lines cross it; its bounding box (kBTMargin of a voxel wider on
// each side, for the FP32 lines; clipped to the volume) is found by the lane that holds the slice.
// A wavefront takes every
// fourth slice of a chunk and walks it in steps of 64 voxels, x fastest (y when K is x, from a
// y-fastest copy of the volume), so that it reads runs of consecutive voxels. All slices of a
// chunk are walked over the extents of its widest box, their origins moved back where that would
// leave the volume: voxels outside the pyramid have no cell in the tile and add nothing. So a
// lane's voxel lies at the same offset from the box's origin in every slice of the chunk, and U,
// V and W are one sum each of the offset's share (kept in registers, up to kBTSteps steps) and
// the origin's (evaluated in FP64 by the lane that holds the slice, and read from it).
// The corner lines need the rays of the pyramid to cross the slices (each corner line's
// direction has a K component of a quarter of its length, all of one sign); otherwise the
// whole slice is walked. A tile whose pyramid passes beside the volume on
// one side is found from the lines' crossings of the first and the last slice, before the chunks,
// whose set-up every wavefront makes. Calls with the set-up by one wavefront / by every wavefront / with
// this test: one slice of 512 x 512 on 640^2 panels x 20 views 212 / 270 / 180 us, 128 x 4 x 128 on
// 640^2 x 20 95 / 106 / 75 us.
// Bound by VALU issue. Walking the chunk's boxes as one flat list of voxels took 75 VALU and 29
// SALU instructions per wavefront of voxels (an index walk in three dimensions, tests against the
// slice's own box, the nine products of the matrix rows); now 38 and 9 with the set-up, and a
// margin of a sixteenth of a voxel instead of one leaves a quarter of the visits out. Dense
// volumes, calls: 256^3 x 360 of 384^2 14.2 -> 10.5 ms, 128^3 x 180 of 192^2 1.16 -> 0.78 ms
// (slices per chunk x steps together 20 x 4: 0.79, 28 x 4: 0.77, 28 x 3: 0.78 and 10.8 ms at 256^3,
// 20 x 3: 11.0).
// The matrix rows in LDS and the cells' addresses by FMA on subnormals then freed 20 VGPRs (84 kept
// five wavefronts per SIMD, 63 keep eight): the kernel at 128^3 x 180 670 -> 569 us.
// Fixed point: terms are rounded to units of max|vol| wbound / 2^kBTBits, where wbound >= the
// weight (1, or 1 / min W^2 for FDK, W > 0 over the volume), so |term| <= 2^kBTBits and a
// 32-bit LDS cell holds the sum of up to 2^(31 - kBTBits) - 1 terms. A voxel adds at most one
// term to a cell, so the workgroup moves the cells into 64-bit registers (one cell per thread)
// and clears them before its voxel visits since the last such drain could pass that count.
// Integer sums are exact: the result does not depend on the order of the additions. The tile is
// written once, in the sinogram's storage type.
constexpr int kBT = 16;                                        // panel tile edge, pixels
constexpr int kBTP = kBT + 2;                                  // LDS cells per row and rows
constexpr int kBTSlab = 40;                                    // slices per chunk
constexpr int kBTBits = 18;                                    // a term's bound: 2^kBTBits
constexpr int kBTBudget = (1 << (31 - kBTBits)) - 1;           // visits between drains
constexpr int kBTSteps = 3;                                    // steps of a slice walked together
constexpr float kBTMargin = 0.0625f;                           // voxels around the crossings
static_assert(kBTSlab % 4 == 0 && kBTSlab / 4 * kBTSteps * kMaxBlock <= kBTBudget,
              "no drain within a chunk's steps");
static_assert(kBT * kBT == kMaxBlock, "one tile cell per thread");
static_assert(kBTSlab <= 64, "one lane per slice of a chunk");

template <class SV, class SS, bool FDK>
__global__ __launch_bounds__(kMaxBlock) void k_bpT3d(typename SS::raw *__restrict__ sino,
                                                     const typename SV::raw *__restrict__ vol,
                                                     const typename SV::raw *__restrict__ ycopy,
                                                     const float *__restrict__ M,
                                                     const float *__restrict__ parts,
                                                     float wbound, int nx, int ny, int nz, int U,
                                                     int V, int A) {
    __shared__ unsigned int cells[kBTP * kBTP]; // pixel iu0 - 1 + i, iv0 - 1 + j at j kBTP + i
    __shared__ float coef[4][4];                // per corner line: F = a + b hK, G = c + d hK
    __shared__ double rows[3][4];               // matrix rows, see below
    __shared__ int walk;                        // one of:
    constexpr int kBoxes = 0, kWhole = 1, kNothing = 2; // boxes in the slices, whole slices
    const int tid = threadIdx.x, lane = tid & 63;
    const int a = (int)(blockIdx.x % (unsigned)A), ti = (int)(blockIdx.x / (unsigned)A);
    const int tv = (V + kBT - 1) / kBT;
    const int tj = (int)(blockIdx.y % (unsigned)tv);
    const size_t b = blockIdx.y / (unsigned)tv;
    const int iu0 = ti * kBT, iv0 = tj * kBT;
    const float *m = M + 12 * a;
    const float cx = (float)((nx - 1) / 2.0), cy = (float)((ny - 1) / 2.0),
                cz = (float)((nz - 1) / 2.0);
    // fixed-point scale (FP64: max|vol| wbound may lie far from 1)
    float vmax = 0.0f;
    for (int i = lane; i < kMaxParts; i += 64) vmax = fmaxf(vmax, parts[b * kMaxParts + i]);
    for (int off = 32; off > 0; off >>= 1) vmax = fmaxf(vmax, __shfl_xor(vmax, off, 64));
    // a voxel value maps to vol s1 s2 units, the scale 2^18 / (max|vol| wbound) in two factors: a
    // power of two that brings max|vol| to [1, 2) and the rest, which is then in range
    static_assert(kBTBits == 18, "the scale uses 2^18");
    const bool some = vmax > 0.0f && vmax < INFINITY;
    const int vexp = some ? ilogbf(vmax) : 0;
    const float s1 = ldexpf(1.0f, max(min(-vexp, 127), -126)); // (|vol| below 2^-127: the rest)
    const double left = ldexp(1.0, -vexp - max(min(-vexp, 127), -126));
    const float s2 =
        some ? (float)(0x1p18 * left / (ldexp((double)vmax, -vexp) * (double)wbound)) : 0.0f;
    // march axis: the largest component of the central ray's direction, the cross product of
    // the (U - uc W) and (V - vc W) rows' voxel parts
    int K;
    {
        const float uc = (float)iu0 + 0.5f * (kBT - 1), vc = (float)iv0 + 0.5f * (kBT - 1);
        float e1[3], e2[3];
        for (int k = 0; k < 3; ++k) {
            e1[k] = fmaf(-uc, m[8 + k], m[k]);
            e2[k] = fmaf(-vc, m[8 + k], m[4 + k]);
        }
        const float d0 = fabsf(e1[1] * e2[2] - e1[2] * e2[1]);
        const float d1 = fabsf(e1[2] * e2[0] - e1[0] * e2[2]);
        const float d2 = fabsf(e1[0] * e2[1] - e1[1] * e2[0]);
        K = d0 >= d1 && d0 >= d2 ? 0 : (d1 >= d2 ? 1 : 2);
        K = __builtin_amdgcn_readfirstlane(K);
    }
    const int F = K == 0 ? 1 : 0, G = K == 2 ? 1 : 2;
    // corner lines (FP64), lanes 0..3 of the first wavefront
    if (tid < 64) {
        const int c = lane & 3;
        const double uc = (double)(iu0 - 1 + ((c & 1) ? kBT + 1 : 0));
        const double vc = (double)(iv0 - 1 + ((c & 2) ? kBT + 1 : 0));
        const double a0 = (double)m[0] - uc * (double)m[8], a1 = (double)m[1] - uc * (double)m[9],
                     a2 = (double)m[2] - uc * (double)m[10], a3 = (double)m[3] - uc * (double)m[11];
        const double q0 = (double)m[4] - vc * (double)m[8], q1 = (double)m[5] - vc * (double)m[9],
                     q2 = (double)m[6] - vc * (double)m[10], q3 = (double)m[7] - vc * (double)m[11];
        const double cr0 = a1 * q2 - a2 * q1, cr1 = a2 * q0 - a0 * q2, cr2 = a0 * q1 - a1 * q0;
        // components along K, F and G
        auto pick = [](double x, double y, double z, int i) {
            return i == 0 ? x : (i == 1 ? y : z);
        };
        const double pF = pick(a0, a1, a2, F), pG = pick(a0, a1, a2, G), pK = pick(a0, a1, a2, K);
        const double qF = pick(q0, q1, q2, F), qG = pick(q0, q1, q2, G), qK = pick(q0, q1, q2, K);
        const double det = pF * qG - pG * qF; // +-cr[K]
        const double len = sqrt(cr0 * cr0 + cr1 * cr1 + cr2 * cr2);
        const bool ok = fabs(det) >= 0.25 * len && len > 0.0;
        const unsigned long long okm = __ballot(ok), posm = __ballot(det > 0.0);
        // (a . (h, 1) = 0, q . (h, 1) = 0) solved for (hF, hG) given hK
        const double id = ok ? 1.0 / det : 0.0;
        const double f0 = (pG * q3 - a3 * qG) * id, f1 = (pG * qK - pK * qG) * id;
        const double g0 = (a3 * qF - pF * q3) * id, g1 = (pK * qF - pF * qK) * id;
        if (lane < 4) {
            coef[c][0] = (float)f0;
            coef[c][1] = (float)f1;
            coef[c][2] = (float)g0;
            coef[c][3] = (float)g1;
        }
        const bool crossed = okm == ~0ull && (posm == 0ull || posm == ~0ull);
        // nothing, if all four lines pass the volume on one side (a voxel away and more) in its
        // first and its last slice
        const double eK = K == 0 ? cx : (K == 1 ? cy : cz), eF = (F == 0 ? cx : cy) + 1.0f,
                     eG = (G == 1 ? cy : cz) + 1.0f;
        const double df = fabs(f1) * eK, dg = fabs(g1) * eK;
        const bool out = __ballot(f0 + df >= -eF) == 0ull || __ballot(f0 - df <= eF) == 0ull ||
                         __ballot(g0 + dg >= -eG) == 0ull || __ballot(g0 - dg <= eG) == 0ull;
        if (lane == 0) walk = !crossed ? kWhole : (out ? kNothing : kBoxes);
    }
    for (int i = tid; i < kBTP * kBTP; i += kMaxBlock) cells[i] = 0u;
    const int nF = F == 0 ? nx : ny, nG = G == 1 ? ny : nz;
    const float cK = K == 0 ? cx : (K == 1 ? cy : cz);
    const float cF = F == 0 ? cx : cy, cG = G == 1 ? cy : cz;
    // matrix rows over the voxel's index (f, g, k) along (F, G, K), the panel coordinates taken
    // from the tile's middle LDS cell (kept in LDS: 24 registers of the walk otherwise)
    constexpr int kMid = kBTP / 2 - 1;
    static_assert(2 * kMid == kBT, "lower taps lie within kMid cells of the middle one");
    if (tid < 3) {
        auto row = [&](int r, double (&o)[4]) {
            const double x = m[4 * r], y = m[4 * r + 1], z = m[4 * r + 2];
            o[0] = F == 0 ? x : y;
            o[1] = G == 1 ? y : z;
            o[2] = K == 0 ? x : (K == 1 ? y : z);
            o[3] = (double)m[4 * r + 3] - o[0] * cF - o[1] * cG - o[2] * cK;
        };
        double o[4], w[4];
        row(tid, o);
        row(2, w);
        const double mid = tid == 0 ? (double)(iu0 - 1 + kMid) : (double)(iv0 - 1 + kMid);
        for (int k = 0; k < 4; ++k) rows[tid][k] = tid < 2 ? o[k] - mid * w[k] : o[k];
    }
    __syncthreads();
    const int todo = __builtin_amdgcn_readfirstlane(walk);
    const int nK = todo == kNothing ? 0 : (K == 0 ? nx : (K == 1 ? ny : nz));
    // voxel (f, g, k) along (F, G, K) lies at src[f + g strG + k strK]: the volume, or for K = x
    // the y-fastest copy [z + 2][x + 2][y + 2]
    const int Wp = nx + 2 * kPad, Hp = ny + 2 * kPad;
    const typename SV::raw *src =
        K == 0 ? ycopy + b * (size_t)Wp * Hp * (nz + 2 * kPad) + (kPad * Wp + kPad) * Hp + kPad
               : vol + b * (size_t)nx * ny * nz;
    const int strG = K == 0 ? Wp * Hp : (K == 1 ? nx * ny : nx);
    const int strK = K == 0 ? Hp : (K == 1 ? nx : nx * ny);
    unsigned int *mine = &cells[(tid / kBT + 1) * kBTP + tid % kBT + 1];
    long long own = 0;
    // cells -> registers (border cells, which belong to other tiles, are never read)
    auto drain = [&]() {
        lds_barrier();
        own += (long long)(int)*mine;
        *mine = 0u;
        __syncthreads();
    };
    const float uF = (float)rows[0][0], uG = (float)rows[0][1], vF = (float)rows[1][0],
                vG = (float)rows[1][1], wF = (float)rows[2][0], wG = (float)rows[2][1];
    // byte strides and the middle cell's address, as subnormals
    const float ccol = subnormal(4), crow = subnormal(4 * kBTP);
    const float cofs = subnormal((int)(uintptr_t)(__attribute__((address_space(3))) unsigned *)cells +
                                 4 * (kMid * kBTP + kMid));
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int run = 0; // voxel visits since the last drain
    for (int k0 = 0; k0 < nK; k0 += kBTSlab) {
        // lane l holds slice k0 + l: its box, then its walk's origin and shares. Every wavefront
        // does the same.
        const int S = min(kBTSlab, nK - k0), k = k0 + min(lane, S - 1);
        int flo = 0, fhi = nF - 1, glo = 0, ghi = nG - 1;
        if (todo == kBoxes) {
            const float hK = (float)k - cK;
            float f0 = INFINITY, f1 = -INFINITY, g0 = INFINITY, g1 = -INFINITY;
            for (int c = 0; c < 4; ++c) {
                const float f = fmaf(coef[c][1], hK, coef[c][0]);
                const float g = fmaf(coef[c][3], hK, coef[c][2]);
                f0 = fminf(f0, f);
                f1 = fmaxf(f1, f);
                g0 = fminf(g0, g);
                g1 = fmaxf(g1, g);
            }
            auto floor_at = [](float v) {
                constexpr float big = 0x1p24f;
                return floor_i32(__builtin_amdgcn_fmed3f(v, -big, big));
            };
            flo = max(0, floor_at(f0 + (cF - kBTMargin)) + 1);
            fhi = min(nF - 1, floor_at(f1 + (cF + kBTMargin)));
            glo = max(0, floor_at(g0 + (cG - kBTMargin)) + 1);
            ghi = min(nG - 1, floor_at(g1 + (cG + kBTMargin)));
        }
        int ef = max(fhi - flo + 1, 0), eg = max(ghi - glo + 1, 0);
        if (ef == 0 || eg == 0) ef = eg = 0;
        for (int off = 32; off > 0; off >>= 1) {
            ef = max(ef, __shfl_xor(ef, off, 64));
            eg = max(eg, __shfl_xor(eg, off, 64));
        }
        const int NF = __builtin_amdgcn_readfirstlane(ef), NG = __builtin_amdgcn_readfirstlane(eg);
        const unsigned total = (unsigned)NF * (unsigned)NG;
        if (total == 0) continue;
        flo = max(0, min(flo, nF - NF));
        glo = max(0, min(glo, nG - NG));
        auto at_origin = [&](int r) {
            return (float)(rows[r][0] * flo + rows[r][1] * glo + rows[r][2] * k + rows[r][3]);
        };
        const float ul = at_origin(0), vl = at_origin(1), wl = at_origin(2);
        const int at = flo + glo * strG + k * strK;
        const float rNF = 1.0f / (float)NF;
        auto lane_of = [](float x, int l) {
            return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
        };
        // N steps from voxel e0 of every slice on
        auto steps = [&](unsigned e0, auto count) {
            constexpr int N = decltype(count)::value;
            if (run + kBTSlab / 4 * N * kMaxBlock > kBTBudget) {
                drain();
                run = 0;
            }
            run += kBTSlab / 4 * N * kMaxBlock;
            // this lane's voxels, the same in every slice; past the box, the coordinate leaves
            // the tile
            float us[N], vs[N], ws[N];
            int ofs[N];
#pragma unroll
            for (int q = 0; q < N; ++q) {
                const unsigned e = e0 + 64 * q + (unsigned)lane;
                const bool in = e < total;
                // e / NF: by the reciprocal, (e + 0.5) / NF lies at least 0.5 / NF from an
                // integer, far more than the rounding for e < 2^20
                int dg = total < 1u << 20 ? (int)(((float)e + 0.5f) * rNF)
                                          : (int)(e / (unsigned)NF);
                int df = (int)e - dg * NF;
                if (!in) dg = df = 0;
                ofs[q] = df + dg * strG;
                const float xf = (float)df, xg = (float)dg;
                us[q] = fmaf(uF, xf, uG * xg);
                vs[q] = in ? fmaf(vF, xf, vG * xg) : 1e30f;
                ws[q] = fmaf(wF, xf, wG * xg);
            }
            for (int l = wv; l < S; l += 4) {
                const typename SV::raw *slice = src + __builtin_amdgcn_readlane(at, l);
                float val[N];
#pragma unroll
                for (int q = 0; q < N; ++q) val[q] = to_f32<SV>(slice[ofs[q]]);
                const float u0 = lane_of(ul, l), v0 = lane_of(vl, l), w0 = lane_of(wl, l);
#pragma unroll
                for (int q = 0; q < N; ++q) {
                    const float x = val[q] * s1 * s2;
                    const float r = __builtin_amdgcn_rcpf(ws[q] + w0);
                    const float u = (us[q] + u0) * r, v = (vs[q] + v0) * r;
                    const float i = floorf(u), j = floorf(v);
                    if (!(fabsf(i) <= (float)kMid && fabsf(j) <= (float)kMid) || x == 0.0f)
                        continue;
                    const float fu = u - i, fv = v - j;
                    const float t = FDK ? x * (r * r) : x;
                    const float t1 = t * fu, t0 = t - t1;
                    const float t01 = t0 * fv, t00 = t0 - t01;
                    const float t11 = t1 * fv, t10 = t1 - t11;
                    auto *const c = (__attribute__((address_space(3))) unsigned *)(uintptr_t)
                        __float_as_uint(fmaf(j, crow, fmaf(i, ccol, cofs)));
                    lds_add(c, (unsigned)round_i32(t00));
                    lds_add(c + 1, (unsigned)round_i32(t10));
                    lds_add(c + kBTP, (unsigned)round_i32(t01));
                    lds_add(c + kBTP + 1, (unsigned)round_i32(t11));
                }
            }
        };
        unsigned e = 0;
        for (; e + 64 * (kBTSteps - 1) < total; e += 64 * kBTSteps)
            steps(e, std::integral_constant<int, kBTSteps>{});
        static_assert(kBTSteps == 3, "the remainder is one or two steps");
        if (e + 64 < total) steps(e, std::integral_constant<int, 2>{});
        else if (e < total) steps(e, std::integral_constant<int, 1>{});
    }
    lds_barrier();
    own += (long long)(int)*mine;
    const int iu = iu0 + tid % kBT, iv = iv0 + tid / kBT;
    if (iu < U && iv < V) {
        const double unit = (double)vmax * (double)wbound * 0x1p-18;
        sino[((b * A + a) * V + iv) * (size_t)U + iu] = from_f32<SS>((float)((double)own * unit));
    }
}

// ---------------------------------------------------------------- host helpers -----------

// True when no angle's U or W row depends on y: k_bp3d<YINV>.
bool y_invariant(const std::vector<float> &m, int64_t A) {
    for (int64_t a = 0; a < A; ++a)
        if (m[12 * a + 1] != 0.0f || m[12 * a + 9] != 0.0f) return false;
    return true;
}

// Smallest W = M[a][8..11] . (h, 1) over the volume's eight corner voxels (h = index - centre)
// and all angles, in FP64 from the FP32 matrices.
double corner_wmin(const cone3d::Desc &g, const std::vector<float> &m, int64_t A) {
    const double c[3] = {((double)g.nx - 1.0) / 2.0, ((double)g.ny - 1.0) / 2.0,
                         ((double)g.nz - 1.0) / 2.0};
    double w = INFINITY;
    for (int64_t a = 0; a < A; ++a) {
        const float *r = m.data() + 12 * a + 8;
        for (int k = 0; k < 8; ++k)
            w = std::min(w, (double)r[3] + (k & 1 ? c[0] : -c[0]) * (double)r[0] +
                                (k & 2 ? c[1] : -c[1]) * (double)r[1] +
                                (k & 4 ? c[2] : -c[2]) * (double)r[2]);
    }
    return w;
}

// Projection matrices for the backprojector, rows (U, V, W) over h = (ix-cx, iy-cy, iz-cz, 1),
// scaled so that W = 1 at the volume centre.
//   reference: the reference's frame (backward_3d.hpp:79-94): dir = O + ix dx + iy dy + iz dz
//              - s, t = (DSO - DSD - s.z) / dir.z, u = dir.x t + s.x + floor(U/2) (likewise
//              v); the lower-tap coordinate is u - 0.5.
//   matched:   the forward frame: voxel P = src + t (org + iu du + iv dv - src) solved for
//              (t, t iu, t iv); the lower-tap coordinate of pixel centre iu is iu.
// Rows are scaled by `fixed_scale` if it is positive, else so that W = 1 at the volume centre.
void finish_matrix(const cone3d::Desc &g, double rows[3][4], float *out, double fixed_scale) {
    const double c[3] = {((double)g.nx - 1.0) / 2.0, ((double)g.ny - 1.0) / 2.0,
                         ((double)g.nz - 1.0) / 2.0};
    for (int r = 0; r < 3; ++r)
        rows[r][3] += rows[r][0] * c[0] + rows[r][1] * c[1] + rows[r][2] * c[2];
    const double w = rows[2][3];
    const double sc = fixed_scale > 0.0 ? fixed_scale
                                        : ((w != 0.0 && std::isfinite(w)) ? 1.0 / w : 1.0);
    for (int r = 0; r < 3; ++r)
        for (int k = 0; k < 4; ++k) out[4 * r + k] = (float)(rows[r][k] * sc);
}

void reference_matrices(const cone3d::Desc &g, const double *phi, const double *theta,
                        const double *psi, int64_t A, std::vector<float> &mref) {
    mref.assign(12 * A, 0.0f);
    const double hu = (double)(g.nu / 2), hv = (double)(g.nv / 2);
    for (int64_t a = 0; a < A; ++a) {
        const cone3d::BpGeom bg = cone3d::bp_angle(g, phi[a], theta[a], psi[a]);
        const double cc = (g.dso - g.dsd) - bg.src[2];
        double d0[3];
        for (int d = 0; d < 3; ++d) d0[d] = bg.org[d] - bg.src[d];
        double rr[3][4];
        const double rowW[4] = {bg.dx[2], bg.dy[2], bg.dz[2], d0[2]};
        const double rowX[4] = {bg.dx[0], bg.dy[0], bg.dz[0], d0[0]};
        const double rowY[4] = {bg.dx[1], bg.dy[1], bg.dz[1], d0[1]};
        for (int k = 0; k < 4; ++k) {
            rr[0][k] = cc * rowX[k] + (bg.src[0] + hu - 0.5) * rowW[k];
            rr[1][k] = cc * rowY[k] + (bg.src[1] + hv - 0.5) * rowW[k];
            rr[2][k] = rowW[k];
        }
        finish_matrix(g, rr, mref.data() + 12 * a, 0.0);
    }
}

// Matched matrices from the forward frames; with `mfdk`, also the FDK ones: W = t (the voxel's
// parameter on its ray, 1 at the panel) times DSD / DSO, so that W = depth / DSO.
void matched_matrices(const cone3d::Desc &g, const std::vector<FwdGeom> &fgeo,
                      std::vector<float> &mmat, std::vector<float> *mfdk) {
    const int64_t A = (int64_t)fgeo.size();
    mmat.assign(12 * A, 0.0f);
    if (mfdk) mfdk->assign(12 * A, 0.0f);
    for (int64_t a = 0; a < A; ++a) {
        const FwdGeom &fg = fgeo[a];
        double Mc[3][3]; // columns org - src, du, dv
        for (int d = 0; d < 3; ++d) {
            Mc[d][0] = fg.org[d] - fg.src[d];
            Mc[d][1] = fg.du[d];
            Mc[d][2] = fg.dv[d];
        }
        const double det = Mc[0][0] * (Mc[1][1] * Mc[2][2] - Mc[1][2] * Mc[2][1]) -
                           Mc[0][1] * (Mc[1][0] * Mc[2][2] - Mc[1][2] * Mc[2][0]) +
                           Mc[0][2] * (Mc[1][0] * Mc[2][1] - Mc[1][1] * Mc[2][0]);
        double inv[3][3];
        inv[0][0] = (Mc[1][1] * Mc[2][2] - Mc[1][2] * Mc[2][1]) / det;
        inv[0][1] = (Mc[0][2] * Mc[2][1] - Mc[0][1] * Mc[2][2]) / det;
        inv[0][2] = (Mc[0][1] * Mc[1][2] - Mc[0][2] * Mc[1][1]) / det;
        inv[1][0] = (Mc[1][2] * Mc[2][0] - Mc[1][0] * Mc[2][2]) / det;
        inv[1][1] = (Mc[0][0] * Mc[2][2] - Mc[0][2] * Mc[2][0]) / det;
        inv[1][2] = (Mc[0][2] * Mc[1][0] - Mc[0][0] * Mc[1][2]) / det;
        inv[2][0] = (Mc[1][0] * Mc[2][1] - Mc[1][1] * Mc[2][0]) / det;
        inv[2][1] = (Mc[0][1] * Mc[2][0] - Mc[0][0] * Mc[2][1]) / det;
        inv[2][2] = (Mc[0][0] * Mc[1][1] - Mc[0][1] * Mc[1][0]) / det;
        // rows ordered (t iu, t iv, t) = (U, V, W)
        const int order[3] = {1, 2, 0};
        double rr[3][4], rk[3][4];
        for (int r = 0; r < 3; ++r) {
            const double *ir = inv[order[r]];
            rr[r][0] = ir[0];
            rr[r][1] = ir[1];
            rr[r][2] = ir[2];
            rr[r][3] = -(ir[0] * fg.src[0] + ir[1] * fg.src[1] + ir[2] * fg.src[2]);
            for (int k = 0; k < 4; ++k) rk[r][k] = rr[r][k];
        }
        finish_matrix(g, rr, mmat.data() + 12 * a, 0.0);
        if (mfdk) finish_matrix(g, rk, mfdk->data() + 12 * a, g.dsd / g.dso);
    }
}

void bp_matrices(const cone3d::Desc &g, const double *phi, const double *theta, const double *psi,
                 int64_t A, std::vector<float> &mref, std::vector<float> &mmat,
                 std::vector<float> &mfdk) {
    reference_matrices(g, phi, theta, psi, A, mref);
    std::vector<FwdGeom> fgeo(A);
    for (int64_t a = 0; a < A; ++a) fgeo[a] = cone3d::fwd_angle(g, phi[a], theta[a], psi[a]);
    matched_matrices(g, fgeo, mmat, &mfdk);
}

// Python order (z, y, x) / (v, u) -> (x, y, z) / (u, v), as forward.cu:113-124
cone3d::Desc desc_of(const cmi_cone3d_desc *d) {
    cone3d::Desc g{};
    g.nx = (int64_t)d->vol_shape[2];
    g.ny = (int64_t)d->vol_shape[1];
    g.nz = (int64_t)d->vol_shape[0];
    g.sx = d->vol_spacing[2];
    g.sy = d->vol_spacing[1];
    g.sz = d->vol_spacing[0];
    g.ox = d->vol_offset[2];
    g.oy = d->vol_offset[1];
    g.oz = d->vol_offset[0];
    g.nu = (int64_t)d->det_shape[1];
    g.nv = (int64_t)d->det_shape[0];
    g.du = d->det_spacing[1];
    g.dv = d->det_spacing[0];
    g.off_u = d->det_offset[1];
    g.off_v = d->det_offset[0];
    g.pitch = d->det_rotation[0]; // forward.cu:136-138
    g.roll = d->det_rotation[1];
    g.yaw = d->det_rotation[2];
    g.dso = d->DSO;
    g.dsd = d->DSD;
    g.cor = d->COR;

    return g;
}

cmi_status check_desc(const cmi_cone3d_desc *d, const char *fn) {
    if (!d) return fail(CMI_ERR_INVALID_ARGUMENT, "%s: descriptor is null", fn);
    if (!d->phi || !d->theta || !d->psi)
        return fail(CMI_ERR_INVALID_ARGUMENT, "%s: null angle array", fn);
    for (int i = 0; i < 3; ++i)
        if (d->vol_shape[i] == 0 || d->vol_shape[i] > 4096 || !(d->vol_spacing[i] > 0))
            return fail(CMI_ERR_INVALID_ARGUMENT,
                        "%s: volume shape / spacing out of range (axis %d)", fn, i);
    for (int i = 0; i < 2; ++i)
        if (d->det_shape[i] == 0 || d->det_shape[i] > 16384 || !(d->det_spacing[i] > 0))
            return fail(CMI_ERR_INVALID_ARGUMENT,
                        "%s: detector shape / spacing out of range (axis %d)", fn, i);
    if (d->nangles == 0 || d->nangles > 65535)
        return fail(CMI_ERR_INVALID_ARGUMENT, "%s: nangles must be in [1, 65535]", fn);
    if (!std::isfinite(d->DSO) || !std::isfinite(d->DSD) || !std::isfinite(d->COR))
        return fail(CMI_ERR_INVALID_ARGUMENT, "%s: non-finite distance", fn);
    for (uint64_t a = 0; a < d->nangles; ++a)
        if (!std::isfinite(d->phi[a]) || !std::isfinite(d->theta[a]) || !std::isfinite(d->psi[a]))
            return fail(CMI_ERR_INVALID_ARGUMENT, "%s: non-finite angle %llu", fn,
                        (unsigned long long)a);
    return CMI_OK;
}

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

cmi_status check_call(const cmi_plan3d *p, const void *vol, int vol_dtype, const void *sino,
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
    if (batch * (uint64_t)p->A > 65535 ||
        batch * (uint64_t)(p->g.nz + 2 * kPad) > 65535)
        return fail(CMI_ERR_INVALID_ARGUMENT, "%s: batch too large for one launch", fn);
    CMI_TRY(check_device_ptr(vol, p->device, "volume"));
    CMI_TRY(check_device_ptr(sino, p->device, "sinogram"));
    return CMI_OK;
}

// Shared tail of the plan constructors: per-angle fast axes and volume copies, matrix layouts,
// device tables and the total sample count (k_count3d). `mfdk` is empty for plans from views.
cmi_status finish_plan3d(std::unique_ptr<cmi_plan3d> p, const std::vector<FwdGeom> &fgeo,
                         const std::vector<float> &mref, const std::vector<float> &mmat,
                         const std::vector<float> &mfdk, cmi_plan3d **plan) {
    const cone3d::Desc &g = p->g;
    const int64_t A = p->A;
    std::vector<int> fast(A);
    for (int64_t a = 0; a < A; ++a) {
        const double *v = fgeo[a].dv;
        const int f = std::fabs(v[1]) >= std::fabs(v[0]) && std::fabs(v[1]) >= std::fabs(v[2]) ? 1
                      : std::fabs(v[2]) > std::fabs(v[0])                                   ? 2
                                                                                            : 0;
        fast[a] = f;
        if (p->copy_slot[f] < 0) p->copy_slot[f] = p->ncopies++;
    }
    p->ycols[CMI_BP3D_REFERENCE] = y_invariant(mref, A);
    p->ycols[CMI_BP3D_MATCHED] = y_invariant(mmat, A);
    p->ycols[CMI_BP3D_FDK] = !mfdk.empty() && y_invariant(mfdk, A);
    p->wmin[CMI_BP3D_REFERENCE] = corner_wmin(g, mref, A);
    p->wmin[CMI_BP3D_MATCHED] = corner_wmin(g, mmat, A);
    p->wmin[CMI_BP3D_FDK] = mfdk.empty() ? 0.0 : corner_wmin(g, mfdk, A);

    DeviceGuard guard;
    CMI_TRY(guard.enter(p->device));
    struct Cleanup {
        cmi_plan3d *p;
        bool armed = true;
        ~Cleanup() {
            if (!armed) return;
            (void)hipFree(p->d_fgeo);
            (void)hipFree(p->d_fast);
            (void)hipFree(p->d_mref);
            (void)hipFree(p->d_mmat);
            (void)hipFree(p->d_mfdk);
        }
    } cleanup{p.get()};
    CMI_HIP_TRY(hipMalloc(&p->d_fgeo, sizeof(FwdGeom) * A));
    CMI_HIP_TRY(hipMalloc(&p->d_fast, sizeof(int) * A));
    CMI_HIP_TRY(hipMalloc(&p->d_mref, sizeof(float) * 12 * A));
    CMI_HIP_TRY(hipMalloc(&p->d_mmat, sizeof(float) * 12 * A));
    if (!mfdk.empty()) CMI_HIP_TRY(hipMalloc(&p->d_mfdk, sizeof(float) * 12 * A));
    p->table_bytes = (sizeof(FwdGeom) + sizeof(int) + (mfdk.empty() ? 2 : 3) * 12 * sizeof(float)) * A;
    unsigned long long *d_total = nullptr;
    CMI_HIP_TRY(hipMalloc(&d_total, sizeof(unsigned long long)));
    std::unique_ptr<unsigned long long, void (*)(unsigned long long *)> total_guard(
        d_total, [](unsigned long long *q) { (void)hipFree(q); });
    hipStream_t s;
    CMI_HIP_TRY(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    std::unique_ptr<ihipStream_t, void (*)(hipStream_t)> stream_guard(
        s, [](hipStream_t q) { (void)hipStreamDestroy(q); });
    CMI_HIP_TRY(hipMemcpyAsync(p->d_fgeo, fgeo.data(), sizeof(FwdGeom) * A,
                               hipMemcpyHostToDevice, s));
    CMI_HIP_TRY(hipMemcpyAsync(p->d_fast, fast.data(), sizeof(int) * A, hipMemcpyHostToDevice,
                               s));
    CMI_HIP_TRY(hipMemcpyAsync(p->d_mref, mref.data(), sizeof(float) * 12 * A,
                               hipMemcpyHostToDevice, s));
    CMI_HIP_TRY(hipMemcpyAsync(p->d_mmat, mmat.data(), sizeof(float) * 12 * A,
                               hipMemcpyHostToDevice, s));
    if (!mfdk.empty())
        CMI_HIP_TRY(hipMemcpyAsync(p->d_mfdk, mfdk.data(), sizeof(float) * 12 * A,
                                   hipMemcpyHostToDevice, s));
    CMI_HIP_TRY(hipMemsetAsync(d_total, 0, sizeof(unsigned long long), s));
    dim3 blk(256), grd((unsigned)((g.nu + 255) / 256), (unsigned)g.nv, (unsigned)A);
    hipLaunchKernelGGL(k_count3d, grd, blk, 0, s, p->d_fgeo, (int)g.nu, (int)g.nv, (int)g.nx,
                       (int)g.ny, (int)g.nz, d_total);
    CMI_HIP_TRY(hipGetLastError());
    unsigned long long total = 0;
    CMI_HIP_TRY(hipMemcpyAsync(&total, d_total, sizeof total, hipMemcpyDeviceToHost, s));
    CMI_HIP_TRY(hipStreamSynchronize(s));
    p->total_samples = total;
    cleanup.armed = false;
    *plan = p.release();
    return CMI_OK;
}

} // namespace

// ===================================================================== C-ABI ===============

extern "C" {

CMI_API cmi_status cmi_plan3d_create(int device, int vol_prec, int det_prec,
                                     const cmi_cone3d_desc *d, cmi_plan3d **plan) {
    clear_error();
    if (!plan) return fail(CMI_ERR_INVALID_ARGUMENT, "plan3d_create: output pointer is null");
    *plan = nullptr;
    CMI_TRY(check_desc(d, "plan3d_create"));
    if (!dtype_ok(vol_prec) || !dtype_ok(det_prec))
        return fail(CMI_ERR_DTYPE, "plan3d_create: precision must be f32, f16 or bf16");
    const uint64_t padvol = (d->vol_shape[0] + 2 * kPad) * (d->vol_shape[1] + 2 * kPad) *
                            (d->vol_shape[2] + 2 * kPad);
    const uint64_t padpan = (d->det_shape[0] + 2 * kPad) * (d->det_shape[1] + 2 * kPad) *
                            d->nangles;
    if (padvol * 4 >= (1ull << 31) || padpan * 4 >= (1ull << 31))
        return fail(CMI_ERR_INVALID_ARGUMENT,
                    "plan3d_create: volume or projection stack exceeds 2 GiB");

    auto p = std::make_unique<cmi_plan3d>();
    p->device = device;
    p->vol_prec = vol_prec;
    p->det_prec = det_prec;
    p->g = desc_of(d);
    const cone3d::Desc &g = p->g;
    p->A = (int64_t)d->nangles;
    const int64_t A = p->A;
    std::vector<FwdGeom> fgeo(A);
    for (int64_t a = 0; a < A; ++a) fgeo[a] = cone3d::fwd_angle(g, d->phi[a], d->theta[a], d->psi[a]);
    std::vector<float> mref, mmat, mfdk;
    reference_matrices(g, d->phi, d->theta, d->psi, A, mref);
    matched_matrices(g, fgeo, mmat, &mfdk);
    return finish_plan3d(std::move(p), fgeo, mref, mmat, mfdk, plan);
}

CMI_API cmi_status cmi_plan3d_create_vec(int device, int vol_prec, int det_prec,
                                         const uint64_t vol_shape[3], const double vol_spacing[3],
                                         const double vol_offset[3], const uint64_t det_shape[2],
                                         const double *vecs, uint64_t nangles,
                                         cmi_plan3d **plan) {
    clear_error();
    if (!plan) return fail(CMI_ERR_INVALID_ARGUMENT, "plan3d_create_vec: output pointer is null");
    *plan = nullptr;
    if (!vol_shape || !vol_spacing || !vol_offset || !det_shape || !vecs)
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan3d_create_vec: null geometry array");
    if (!dtype_ok(vol_prec) || !dtype_ok(det_prec))
        return fail(CMI_ERR_DTYPE, "plan3d_create_vec: precision must be f32, f16 or bf16");
    // the shape, spacing and size limits of cmi_plan3d_create, through a descriptor
    const double zero3[3] = {0.0, 0.0, 0.0};
    cmi_cone3d_desc d{};
    for (int i = 0; i < 3; ++i) {
        d.vol_shape[i] = vol_shape[i];
        d.vol_spacing[i] = vol_spacing[i];
        d.vol_offset[i] = vol_offset[i];
    }
    for (int i = 0; i < 2; ++i) {
        d.det_shape[i] = det_shape[i];
        d.det_spacing[i] = 1.0;
    }
    d.DSO = d.DSD = 1.0;
    d.nangles = nangles;
    d.phi = d.theta = d.psi = zero3; // not read past index 0 below; angles come from the views
    if (nangles == 0 || nangles > 65535)
        return fail(CMI_ERR_INVALID_ARGUMENT, "plan3d_create_vec: nangles must be in [1, 65535]");
    {
        cmi_cone3d_desc d1 = d;
        d1.nangles = 1;
        CMI_TRY(check_desc(&d1, "plan3d_create_vec"));
    }
    for (int i = 0; i < 3; ++i)
        if (!std::isfinite(vol_offset[i]))
            return fail(CMI_ERR_INVALID_ARGUMENT, "plan3d_create_vec: non-finite volume offset");
    const uint64_t padvol = (vol_shape[0] + 2 * kPad) * (vol_shape[1] + 2 * kPad) *
                            (vol_shape[2] + 2 * kPad);
    const uint64_t padpan = (det_shape[0] + 2 * kPad) * (det_shape[1] + 2 * kPad) * nangles;
    if (padvol * 4 >= (1ull << 31) || padpan * 4 >= (1ull << 31))
        return fail(CMI_ERR_INVALID_ARGUMENT,
                    "plan3d_create_vec: volume or projection stack exceeds 2 GiB");
    for (uint64_t a = 0; a < nangles; ++a) {
        const double *v = vecs + 12 * a;
        for (int i = 0; i < 12; ++i)
            if (!std::isfinite(v[i]))
                return fail(CMI_ERR_INVALID_ARGUMENT, "plan3d_create_vec: non-finite view %llu",
                            (unsigned long long)a);
        // the panel normal u x v must be non-zero and the source off the panel plane
        const double n[3] = {v[7] * v[11] - v[8] * v[10], v[8] * v[9] - v[6] * v[11],
                             v[6] * v[10] - v[7] * v[9]};
        const double nn = std::sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
        const double L = (n[0] * (v[3] - v[0]) + n[1] * (v[4] - v[1]) + n[2] * (v[5] - v[2]));
        const double ul = std::sqrt(v[6] * v[6] + v[7] * v[7] + v[8] * v[8]);
        const double vl = std::sqrt(v[9] * v[9] + v[10] * v[10] + v[11] * v[11]);
        if (!(nn > 1e-12 * ul * vl) || !(std::fabs(L) > 1e-9 * nn))
            return fail(CMI_ERR_INVALID_ARGUMENT,
                        "plan3d_create_vec: view %llu has parallel or zero u / v steps or its "
                        "source on the panel plane",
                        (unsigned long long)a);
    }
    auto p = std::make_unique<cmi_plan3d>();
    p->device = device;
    p->vol_prec = vol_prec;
    p->det_prec = det_prec;
    p->views = true;
    p->g = desc_of(&d);
    p->g.du = std::sqrt(vecs[6] * vecs[6] + vecs[7] * vecs[7] + vecs[8] * vecs[8]);
    p->g.dv = std::sqrt(vecs[9] * vecs[9] + vecs[10] * vecs[10] + vecs[11] * vecs[11]);
    p->g.dso = p->g.dsd = 0.0; // no circular-orbit distances: no FDK weighting
    p->A = (int64_t)nangles;
    const int64_t A = p->A;
    std::vector<FwdGeom> fgeo(A);
    for (int64_t a = 0; a < A; ++a) fgeo[a] = cone3d::fwd_view(p->g, vecs + 12 * a);
    std::vector<float> mmat;
    matched_matrices(p->g, fgeo, mmat, nullptr);
    // reference mode of a plan from views projects like matched mode (the reference's own
    // backprojection frame is defined by Euler angles only)
    return finish_plan3d(std::move(p), fgeo, mmat, mmat, {}, plan);
}

CMI_API cmi_status cmi_cone3d_bp_matrices(const cmi_cone3d_desc *d, int mode, float *out,
                                          int *y_invariant_out) {
    clear_error();
    CMI_TRY(check_desc(d, "cone3d_bp_matrices"));
    if (!out) return fail(CMI_ERR_INVALID_ARGUMENT, "cone3d_bp_matrices: null output");
    if (mode != CMI_BP3D_REFERENCE && mode != CMI_BP3D_MATCHED && mode != CMI_BP3D_FDK)
        return fail(CMI_ERR_INVALID_ARGUMENT, "cone3d_bp_matrices: unknown mode %d", mode);
    const cone3d::Desc g = desc_of(d);
    std::vector<float> mref, mmat, mfdk;
    bp_matrices(g, d->phi, d->theta, d->psi, (int64_t)d->nangles, mref, mmat, mfdk);
    const std::vector<float> &m = mode == CMI_BP3D_MATCHED ? mmat : mode == CMI_BP3D_FDK ? mfdk : mref;
    std::copy(m.begin(), m.end(), out);
    if (y_invariant_out) *y_invariant_out = y_invariant(m, (int64_t)d->nangles) ? 1 : 0;
    return CMI_OK;
}

CMI_API cmi_status cmi_plan3d_destroy(cmi_plan3d *plan) {
    clear_error();
    if (!plan) return CMI_OK;
    DeviceGuard guard;
    const cmi_status st = guard.enter(plan->device);
    if (st == CMI_OK) {
        (void)hipDeviceSynchronize();
        (void)hipFree(plan->d_fgeo);
        (void)hipFree(plan->d_fast);
        (void)hipFree(plan->d_mref);
        (void)hipFree(plan->d_mmat);
        (void)hipFree(plan->d_mfdk);
    }
    delete plan;
    return st;
}

CMI_API cmi_status cmi_plan3d_get_info(const cmi_plan3d *plan, cmi_plan3d_info *info) {
    clear_error();
    if (!plan || !info) return fail(CMI_ERR_INVALID_ARGUMENT, "plan3d_get_info: null argument");
    info->device = plan->device;
    info->vol_prec = plan->vol_prec;
    info->det_prec = plan->det_prec;
    info->nx = (uint64_t)plan->g.nx;
    info->ny = (uint64_t)plan->g.ny;
    info->nz = (uint64_t)plan->g.nz;
    info->nu = (uint64_t)plan->g.nu;
    info->nv = (uint64_t)plan->g.nv;
    info->nangles = (uint64_t)plan->A;
    info->total_samples = plan->total_samples;
    info->table_bytes = plan->table_bytes;
    return CMI_OK;
}

CMI_API cmi_status cmi_forward_3d(const cmi_plan3d *plan, const void *volume, int vol_dtype,
                                  void *sinogram, int sino_dtype, uint64_t batch,
                                  void *stream) {
    clear_error();
    CMI_TRY(check_call(plan, volume, vol_dtype, sinogram, sino_dtype, batch, "forward_3d"));
    DeviceGuard guard;
    CMI_TRY(guard.enter(plan->device));
    const hipStream_t s = (hipStream_t)stream;
    const cone3d::Desc &g = plan->g;
    const int nx = (int)g.nx, ny = (int)g.ny, nz = (int)g.nz, U = (int)g.nu, V = (int)g.nv,
              A = (int)plan->A;
    const int Wp = nx + 2 * kPad, Hp = ny + 2 * kPad, Dp = nz + 2 * kPad;
    void *scratch = nullptr;
    const size_t one = (size_t)Wp * Hp * Dp, nc = (size_t)plan->ncopies;
    CMI_HIP_TRY(hipMallocAsync(&scratch, one * nc * dtype_size(vol_dtype) * batch, s));
    const cmi_status st = dispatch2(vol_dtype, sino_dtype, [&](auto si, auto ss) -> cmi_status {
        using SI = decltype(si);
        using SS = decltype(ss);
        using RI = typename SI::raw;
        for (uint64_t b = 0; b < batch; ++b) {
            const RI *src = (const RI *)volume + b * (size_t)nx * ny * nz;
            RI *copies = (RI *)scratch + b * nc * one;
            if (plan->copy_slot[0] >= 0) {
                dim3 pb(256), pg((unsigned)((Wp + 255) / 256), (unsigned)Hp, (unsigned)Dp);
                hipLaunchKernelGGL((k_stage3d<SI>), pg, pb, 0, s, src,
                                   copies + plan->copy_slot[0] * one, nx, ny, nz, Wp, Hp, Dp);
            }
            if (plan->copy_slot[1] >= 0) {
                dim3 tb(32, 8), tg((unsigned)((Wp + 31) / 32), (unsigned)((Hp + 31) / 32),
                                   (unsigned)Dp);
                hipLaunchKernelGGL((k_stage3d_t<SI, 1>), tg, tb, 0, s, src,
                                   copies + plan->copy_slot[1] * one, nx, ny, nz, Wp, Hp, Dp);
            }
            if (plan->copy_slot[2] >= 0) {
                dim3 tb(32, 8), tg((unsigned)((Wp + 31) / 32), (unsigned)((Dp + 31) / 32),
                                   (unsigned)Hp);
                hipLaunchKernelGGL((k_stage3d_t<SI, 2>), tg, tb, 0, s, src,
                                   copies + plan->copy_slot[2] * one, nx, ny, nz, Wp, Hp, Dp);
            }
        }
        dim3 fb(kMaxBlock), fg((unsigned)((U + 15) / 16), (unsigned)((V + 15) / 16),
                               (unsigned)(A * batch));
        hipLaunchKernelGGL((k_fwd3d<SI, SS>), fg, fb, 0, s, (const RI *)scratch, plan->d_fgeo,
                           plan->d_fast, plan->copy_slot[0], plan->copy_slot[1],
                           plan->copy_slot[2], plan->ncopies, nx, ny, nz, U, V, A,
                           (typename SS::raw *)sinogram);
        CMI_HIP_TRY(hipGetLastError());
        return CMI_OK;
    });
    const hipError_t fe = hipFreeAsync(scratch, s);
    if (st != CMI_OK) return st;
    CMI_HIP_TRY(fe);
    return CMI_OK;
}

CMI_API cmi_status cmi_backward_3d(const cmi_plan3d *plan, void *volume, int vol_dtype,
                                   const void *sinogram, int sino_dtype, uint64_t batch,
                                   int mode, void *stream) {
    clear_error();
    CMI_TRY(check_call(plan, volume, vol_dtype, sinogram, sino_dtype, batch, "backward_3d"));
    if (mode != CMI_BP3D_REFERENCE && mode != CMI_BP3D_MATCHED && mode != CMI_BP3D_FDK)
        return fail(CMI_ERR_INVALID_ARGUMENT, "backward_3d: unknown mode %d", mode);
    if (mode == CMI_BP3D_FDK && plan->views)
        return fail(CMI_ERR_NOT_SUPPORTED,
                    "backward_3d: FDK weighting needs a circular orbit (DSO, DSD); this plan "
                    "was built from views");
    DeviceGuard guard;
    CMI_TRY(guard.enter(plan->device));
    const hipStream_t s = (hipStream_t)stream;
    const cone3d::Desc &g = plan->g;
    const int nx = (int)g.nx, ny = (int)g.ny, nz = (int)g.nz, U = (int)g.nu, V = (int)g.nv,
              A = (int)plan->A;
    const int Up = U + 2 * kPad, Vp = V + 2 * kPad;
    void *scratch = nullptr;
    CMI_HIP_TRY(
        hipMallocAsync(&scratch, (size_t)Up * Vp * A * dtype_size(sino_dtype) * batch, s));
    const float cx = (float)((nx - 1) / 2.0), cy = (float)((ny - 1) / 2.0),
                cz = (float)((nz - 1) / 2.0);
    const float *M = mode == CMI_BP3D_MATCHED ? plan->d_mmat
                     : mode == CMI_BP3D_FDK   ? plan->d_mfdk
                                              : plan->d_mref;
    const cmi_status st = dispatch2(vol_dtype, sino_dtype, [&](auto sv, auto ss) -> cmi_status {
        using SV = decltype(sv);
        using SS = decltype(ss);
        using RS = typename SS::raw;
        const uint64_t n = (uint64_t)Up * Vp * A * batch;
        hipLaunchKernelGGL((k_stage_panel<SS>), dim3((unsigned)((n + 4 * 256 - 1) / (4 * 256))),
                           dim3(256), 0, s, (const RS *)sinogram, (RS *)scratch, U, V, n);
        auto launch = [&](auto yinv) {
            constexpr bool Y = decltype(yinv)::value;
            const int nzt = (nz + kTileZ<Y> - 1) / kTileZ<Y>;
            const dim3 bg((unsigned)((nx + kTileX - 1) / kTileX),
                          (unsigned)((ny + kTileY - 1) / kTileY), (unsigned)(nzt * batch));
            auto kern = mode == CMI_BP3D_MATCHED ? k_bp3d<SV, SS, Y, true, false>
                        : mode == CMI_BP3D_FDK   ? k_bp3d<SV, SS, Y, true, true>
                                                 : k_bp3d<SV, SS, Y, false, false>;
            hipLaunchKernelGGL(kern, bg, dim3(kMaxBlock), 0, s,
                               (typename SV::raw *)volume, (const RS *)scratch, M, nx, ny, nz, U,
                               V, A, cx, cy, cz);
        };
        if (plan->ycols[mode]) launch(std::true_type{});
        else launch(std::false_type{});
        CMI_HIP_TRY(hipGetLastError());
        return CMI_OK;
    });
    const hipError_t fe = hipFreeAsync(scratch, s);
    if (st != CMI_OK) return st;
    CMI_HIP_TRY(fe);
    return CMI_OK;
}

CMI_API cmi_status cmi_adjoint_3d(const cmi_plan3d *plan, void *volume, int vol_dtype,
                                  const void *sinogram, int sino_dtype, uint64_t batch,
                                  void *stream) {
    clear_error();
    CMI_TRY(check_call(plan, volume, vol_dtype, sinogram, sino_dtype, batch, "adjoint_3d"));
    DeviceGuard guard;
    CMI_TRY(guard.enter(plan->device));
    const hipStream_t s = (hipStream_t)stream;
    const cone3d::Desc &g = plan->g;
    const int nx = (int)g.nx, ny = (int)g.ny, nz = (int)g.nz, U = (int)g.nu, V = (int)g.nv,
              A = (int)plan->A;
    const size_t rays = (size_t)A * U * V;
    // scratch: the march table [2][rays], [batch][kMaxParts] partial maxima of |y|, then (256-byte
    // aligned) the tiles' 64-bit sums
    const size_t ntiles = (size_t)((nx + kAT - 1) / kAT) * ((ny + kAT - 1) / kAT) *
                          ((nz + kAT - 1) / kAT) * batch;
    float4 *table = nullptr;
    CMI_HIP_TRY(hipMallocAsync((void **)&table,
                               2 * rays * sizeof(float4) + kMaxParts * batch * sizeof(float) +
                                   256 + ntiles * kAT * kAT * kAT * sizeof(long long),
                               s));
    float *parts = reinterpret_cast<float *>(table + 2 * rays);
    long long *totals = reinterpret_cast<long long *>(
        (reinterpret_cast<uintptr_t>(parts + kMaxParts * batch) + 255) & ~(uintptr_t)255);
    const cmi_status st = dispatch2(vol_dtype, sino_dtype, [&](auto sv, auto ss) -> cmi_status {
        using SV = decltype(sv);
        using SS = decltype(ss);
        dim3 tb(256), tg((unsigned)((U + 255) / 256), (unsigned)V, (unsigned)A);
        hipLaunchKernelGGL(k_ray_table3d, tg, tb, 0, s, plan->d_fgeo, nx, ny, nz, U, V, table,
                           table + rays);
        hipLaunchKernelGGL((k_absmax_parts<SS>), dim3(kMaxParts, (unsigned)batch),
                           dim3(kMaxBlock), 0, s, (const typename SS::raw *)sinogram, rays, parts);
        const int ntz = (nz + kAT - 1) / kAT;
        const dim3 tiles((unsigned)((nx + kAT - 1) / kAT), (unsigned)((ny + kAT - 1) / kAT),
                         (unsigned)(ntz * batch));
        const uint64_t samples = plan->total_samples * batch / ntiles; // per tile
        const int G =
            samples + kAdj3Angle * A < kAdj3Alone ||
                    (ntiles >= kAdj3FullTiles &&
                     (uint64_t)A <= std::min(kAdj3FewAngles, ntiles / kAdj3TilesPerAngle))
                ? 1
                : (int)std::max<uint64_t>(
                      1, std::min<uint64_t>({(uint64_t)A, (kAdj3Workgroups + ntiles - 1) / ntiles,
                                             65535 / (uint64_t)tiles.z,
                                             std::max(samples / kAdj3Samples,
                                                      std::min(kAdj3Fill / ntiles,
                                                               samples / kAdj3Least))}));
        if (G > 1)
            hipLaunchKernelGGL(k_clear_sums, dim3((unsigned)(ntiles * kATOwn)), dim3(kMaxBlock), 0,
                               s, totals);
        hipLaunchKernelGGL((k_adj3d<SV, SS>), dim3(tiles.x, tiles.y, tiles.z * G),
                           dim3(kMaxBlock), 0, s, (typename SV::raw *)volume,
                           (const typename SS::raw *)sinogram, (const float4 *)table,
                           (const float4 *)(table + rays), plan->d_mmat, parts, nx, ny, nz,
                           U, V, A, G, totals);
        if (G > 1)
            hipLaunchKernelGGL((k_adj3d_finish<SV>), tiles, dim3(kMaxBlock), 0, s,
                               (typename SV::raw *)volume, parts, nx, ny, nz, totals);
        CMI_HIP_TRY(hipGetLastError());
        return CMI_OK;
    });
    const hipError_t fe = hipFreeAsync(table, s);
    if (st != CMI_OK) return st;
    CMI_HIP_TRY(fe);
    return CMI_OK;
}

CMI_API cmi_status cmi_backward_3d_transpose(const cmi_plan3d *plan, void *sinogram,
                                             int sino_dtype, const void *volume, int vol_dtype,
                                             uint64_t batch, int mode, void *stream) {
    clear_error();
    CMI_TRY(check_call(plan, volume, vol_dtype, sinogram, sino_dtype, batch,
                       "backward_3d_transpose"));
    if (mode != CMI_BP3D_REFERENCE && mode != CMI_BP3D_MATCHED && mode != CMI_BP3D_FDK)
        return fail(CMI_ERR_INVALID_ARGUMENT, "backward_3d_transpose: unknown mode %d", mode);
    if (mode == CMI_BP3D_FDK && plan->views)
        return fail(CMI_ERR_NOT_SUPPORTED,
                    "backward_3d_transpose: FDK weighting needs a circular orbit (DSO, DSD); "
                    "this plan was built from views");
    const double wmin = plan->wmin[mode];
    if (!(wmin > 0.0) || !std::isfinite(wmin))
        return fail(CMI_ERR_NOT_SUPPORTED,
                    "backward_3d_transpose: a voxel lies at or behind a source (W <= 0), so "
                    "the backprojection's projection is unbounded");
    const cone3d::Desc &g = plan->g;
    const int nx = (int)g.nx, ny = (int)g.ny, nz = (int)g.nz, U = (int)g.nu, V = (int)g.nv,
              A = (int)plan->A;
    const uint64_t tu = (uint64_t)(U + kBT - 1) / kBT, tv = (uint64_t)(V + kBT - 1) / kBT;
    if ((uint64_t)A * tu * kMaxBlock >= (1ull << 32) || tv * batch > 65535)
        return fail(CMI_ERR_INVALID_ARGUMENT,
                    "backward_3d_transpose: too many projections, tiles or volumes for one "
                    "launch");
    // the largest weight: 1 (bilinear), times 1 / W^2 for FDK; 1 % of margin for FP32
    const double wbound = 1.01 * (mode == CMI_BP3D_FDK ? 1.0 / (wmin * wmin) : 1.0);
    if (!(wbound < 1e30))
        return fail(CMI_ERR_NOT_SUPPORTED, "backward_3d_transpose: FDK weight out of range");
    DeviceGuard guard;
    CMI_TRY(guard.enter(plan->device));
    const hipStream_t s = (hipStream_t)stream;
    const int Wp = nx + 2 * kPad, Hp = ny + 2 * kPad, Dp = nz + 2 * kPad;
    const size_t one = (size_t)Wp * Hp * Dp;
    // scratch: per volume a y-fastest copy (read where the march axis is x), then kMaxParts
    // partial maxima of |vol| per volume
    const size_t copy_bytes = (one * dtype_size(vol_dtype) * batch + 255) / 256 * 256;
    void *scratch = nullptr;
    CMI_HIP_TRY(hipMallocAsync(&scratch, copy_bytes + kMaxParts * batch * sizeof(float), s));
    float *parts = (float *)((char *)scratch + copy_bytes);
    const float *M = mode == CMI_BP3D_MATCHED ? plan->d_mmat
                     : mode == CMI_BP3D_FDK   ? plan->d_mfdk
                                              : plan->d_mref;
    const cmi_status st = dispatch2(vol_dtype, sino_dtype, [&](auto sv, auto ss) -> cmi_status {
        using SV = decltype(sv);
        using SS = decltype(ss);
        using RV = typename SV::raw;
        for (uint64_t b = 0; b < batch; ++b) {
            dim3 tb(32, 8), tg((unsigned)((Wp + 31) / 32), (unsigned)((Hp + 31) / 32),
                               (unsigned)Dp);
            hipLaunchKernelGGL((k_stage3d_t<SV, 1>), tg, tb, 0, s,
                               (const RV *)volume + b * (size_t)nx * ny * nz,
                               (RV *)scratch + b * one, nx, ny, nz, Wp, Hp, Dp);
        }
        hipLaunchKernelGGL((k_absmax_parts<SV>), dim3(kMaxParts, (unsigned)batch),
                           dim3(kMaxBlock), 0, s, (const RV *)volume, (size_t)nx * ny * nz,
                           parts);
        auto kern = mode == CMI_BP3D_FDK ? k_bpT3d<SV, SS, true> : k_bpT3d<SV, SS, false>;
        hipLaunchKernelGGL(kern, dim3((unsigned)(A * tu), (unsigned)(tv * batch)),
                           dim3(kMaxBlock), 0, s, (typename SS::raw *)sinogram,
                           (const RV *)volume, (const RV *)scratch, M, parts, (float)wbound, nx,
                           ny, nz, U, V, A);
        CMI_HIP_TRY(hipGetLastError());
        return CMI_OK;
    });
    const hipError_t fe = hipFreeAsync(scratch, s);
    if (st != CMI_OK) return st;
    CMI_HIP_TRY(fe);
    return CMI_OK;
}

} // extern "C"
