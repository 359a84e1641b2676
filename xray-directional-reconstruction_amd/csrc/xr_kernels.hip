// HIP kernels (gfx950) for the cone-beam reconstruction hot path.
//
// Volume layout in HBM ("column layout"): voxel (x, y, z) of channel k lives at
//   k*chan_stride + z + N*(x + N*y),
// i.e. z-columns are contiguous.  The rotation axis is z, so for an untilted
// scan (condR = I) a z-column projects onto a single detector column pair with
// v advancing ~1 pixel per voxel: 64 lanes walking 64 consecutive z of one
// column read 256 contiguous bytes and hit 64 distinct detector rows.
// Sinograms keep the reference layout u + U*(v + V*view) per condition.
//
// Forward projection (ir.cu:1490-1531, 1753-1804 + 1533-1603 + 1616-1666) is
// voxel-driven, like the reference, but each block OWNS a band of kBandU
// detector columns of one view: it accumulates the bilinear splat of every voxel
// that touches the band in LDS, then writes the band once with the
// L/(factor+1e-5) normalisation and the MLEM ratio / ART residual fused in.
// No global atomics; the sinogram is written exactly once per view.  The LDS
// accumulation is fixed point: each contribution is rounded to a 32-bit integer
// on a per-launch power-of-two scale (from max |voxel value|) and summed with
// integer LDS atomics (ds_add_u32; the weight pass: ds_add_u64).  On gfx950 these run at bank rate
// while FP32 LDS atomics (ds_add_f32) serialise per lane (~20x slower here), and
// integer sums are exact and order independent: the forward projection is
// bitwise deterministic.
//
// Backprojection (ir.cu:1720-1751, 1807-1850, fdk.cu:62-170) is a gather: a
// block owns a tile of voxels, loops over all views of the subset, stages the
// tile's detector footprint in LDS and accumulates in registers; the MLEM/ART
// update (ir.cu:1637-1693) is applied in the same kernel, so each voxel is read
// and written once per subset.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "xr_internal.hpp"
#include "xr_random.hpp"

namespace xr {

namespace {

__device__ __forceinline__ float rcpf(float x) { return __builtin_amdgcn_rcpf(x); }

// Wave-uniform copy of a value loaded through a vector load: the compiler
// then keeps everything derived from it in scalar registers and scalar
// branches (a view's table is the same for every lane).
__device__ __forceinline__ float uniformf(float x) {
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}
__device__ __forceinline__ int uniformi(int x) { return __builtin_amdgcn_readfirstlane(x); }

struct ColForms {
    float nu, nv, nd;
};

// The projective forms at z' = 0 for column (x', y').  Every kernel evaluates
// u, v through col_forms + voxel_uv so that the splat, the gather and the
// normalisation table agree bit for bit on (u, v) and the acceptance window.
__device__ __forceinline__ ColForms col_forms(const ViewGeom& g, float xp, float yp) {
    ColForms c;
    c.nu = fmaf(g.au[1], yp, fmaf(g.au[0], xp, g.au[3]));
    c.nv = fmaf(g.av[1], yp, fmaf(g.av[0], xp, g.av[3]));
    c.nd = fmaf(g.ad[1], yp, fmaf(g.ad[0], xp, g.ad[3]));
    return c;
}

__device__ __forceinline__ void voxel_uv(const ViewGeom& g, const ColForms& c, float zp, const Dims& d, float& u,
                                         float& v) {
    const float nu = fmaf(g.au[2], zp, c.nu);
    const float nv = fmaf(g.av[2], zp, c.nv);
    const float nd = fmaf(g.ad[2], zp, c.nd);
    const float inv = rcpf(nd);
    u = fmaf(nu, inv, d.hu);
    v = fmaf(nv, inv, d.hv);
}

// Acceptance window 0.55 < u < U-0.55 (ir.cu:1501) and bilinear split with
// floor(u-0.5) (ir.cu:1504-1509).
__device__ __forceinline__ bool accept_u(float u, const Dims& d) { return 0.55f < u && u < d.umax; }
__device__ __forceinline__ bool accept_v(float v, const Dims& d) { return 0.55f < v && v < d.vmax; }
__device__ __forceinline__ void split(float u, int& iu, float& fu) {
    const float t = u - 0.5f;
    const float f = floorf(t);
    iu = (int)f;
    fu = t - f;
}

// lambdas of a kernel body that several places call: without it they become
// calls, with their captures in scratch memory
#define XR_INLINE __attribute__((always_inline))

typedef __attribute__((address_space(3))) float lds_float;
typedef __attribute__((address_space(3))) int lds_int;

// Global-memory view of a pointer.  Kernel-argument pointers are known to be
// global, but pointers read from a work-item table in memory are not: without
// this cast their loads are flat accesses (slower, and mixing them with LDS
// accesses in one kernel is what the gfx950 backend handles worst).
// (The host pass only parses device code; it sees plain pointers.)
#if defined(__HIP_DEVICE_COMPILE__)
template <class T>
using gptr = __attribute__((address_space(1))) T*;
#else
template <class T>
using gptr = T*;
#endif
template <class T>
__device__ __forceinline__ gptr<T> to_global(T* p) {
    return (gptr<T>)p;
}

// Read-only view of a table that no kernel writes (view lists, per-view
// geometry and weight tables): loads through the constant address space at a
// wave-uniform address become scalar loads into SGPRs, instead of vector loads
// plus a readfirstlane (a VALU instruction) per value.
#if defined(__HIP_DEVICE_COMPILE__)
template <class T>
using cptr = const __attribute__((address_space(4))) T*;
#else
template <class T>
using cptr = const T*;
#endif
template <class T>
__device__ __forceinline__ cptr<T> to_const(const T* p) {
    return (cptr<T>)p;
}

__device__ __forceinline__ void lds_add(lds_float* p, float v) {
    __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// Chord length of the pixel-centre ray through the reconstruction box, FP64,
// following correlationProjByLength (ir.cu:1556-1597): the six faces in order
// x-,x+,y-,y+,z-,z+; a face hit counts when the other two coordinates lie
// strictly inside; L is the distance between the first two hits (one hit: its
// distance from the origin, as the reference's zero-filled buffer gives).
__device__ double chord_length(const ChordGeom& c, int u, int v, const Dims& d) {
    const double cu = ((double)u - ((double)d.U - 1.0) * 0.5) * c.det[0];
    const double cv = ((double)v - ((double)d.V - 1.0) * 0.5) * c.det[0];
    double pix[3], s2p[3];
    for (int i = 0; i < 3; i++) {
        pix[i] = cu * c.eu[i] - c.det[1] * c.ey[i] + cv * c.ev[i];
        s2p[i] = c.src[i] - pix[i];
    }
    int cnt = 0;
    double h0x = 0, h0y = 0, h0z = 0, h1x = 0, h1y = 0, h1z = 0;
#pragma unroll
    for (int p = 0; p < 3; p++) {
#pragma unroll
        for (int sg = 0; sg < 2; sg++) {
            const double plane = sg ? c.hi[p] : c.lo[p];
            const double t = (plane - c.src[p]) / s2p[p];
            double pl[3];
#pragma unroll
            for (int i = 0; i < 3; i++) pl[i] = t * s2p[i] + c.src[i];
            const int p1 = (p + 1) % 3, p2 = (p + 2) % 3;
            if (c.lo[p1] < pl[p1] && pl[p1] < c.hi[p1] && c.lo[p2] < pl[p2] && pl[p2] < c.hi[p2]) {
                if (cnt == 0) {
                    h0x = pl[0];
                    h0y = pl[1];
                    h0z = pl[2];
                } else if (cnt == 1) {
                    h1x = pl[0];
                    h1y = pl[1];
                    h1z = pl[2];
                }
                cnt++;
            }
        }
    }
    const double dx = h0x - h1x, dy = h0y - h1y, dz = h0z - h1z;
    return sqrt(dx * dx + dy * dy + dz * dz);
}

// ---------------------------------------------------------------------------
// Forward projection: one block = (detector band of kBandU columns, one view,
// a chunk of detector rows).  The block's waves walk the volume rows y (round
// robin), find the z-columns whose footprint touches the band (ballot over 64 x
// per step), and splat them with lanes = z.
// ---------------------------------------------------------------------------
constexpr int kXttChunks = 2;  // untilted XTT: z chunks of 64 (x K channels) loaded per step

typedef __attribute__((address_space(3))) unsigned long long lds_u64;

// Band accumulator word: 64-bit for the weight pass (its own sum bound is what
// it computes), 32-bit otherwise, with the scale chosen from the largest
// per-pixel weight sum so that no pixel sum can reach 2^31 in magnitude.
template <int KIND>
struct FwdAcc {
    typedef unsigned int T;
    typedef int S;
};
template <>
struct FwdAcc<FWD_WEIGHT> {
    typedef unsigned long long T;
    typedef long long S;
};
template <class T>
using lds_ptr = __attribute__((address_space(3))) T*;

// Value of x in lane `l` (wave-uniform l), into a scalar register.
__device__ __forceinline__ float lane_f(float x, int l) {
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l));
}
__device__ __forceinline__ int lane_i(int x, int l) { return __builtin_amdgcn_readlane(x, l); }

// z range of an untilted column that can reach detector rows [v0, v0+vb), from
// t(z') = v - 0.5 = B z' + A, z' = z - xc: those rows need t in [v0 - 1,
// v0 + vb); widened by two voxels and tested exactly in the splat.  (A chunk of
// all rows keeps [0, nz): the splat's window test rejects voxels that miss the
// detector.)
__device__ __forceinline__ void col_zrange_t(float B, float A, const Dims& d, int v0, int vb, int& z_beg,
                                             int& z_end) {
    z_beg = 0;
    z_end = d.nz;
    if (fabsf(B) > 1e-6f) {
        const float za = ((float)(v0 - 1) - A) / B;
        const float zb = ((float)(v0 + vb) - A) / B;
        const float lo = fminf(za, zb) + d.xc - 2.0f, hi = fmaxf(za, zb) + d.xc + 2.0f;
        z_beg = (int)fmaxf(0.0f, floorf(lo));
        z_end = (int)fminf((float)d.nz, ceilf(hi) + 1.0f);
        if (!(lo == lo) || !(hi == hi)) {
            z_beg = 0;
            z_end = d.nz;
        }
    }
}

// floor(x + 0.5) in one instruction (round half up; x is far inside int range).
__device__ __forceinline__ int round_half_up(float x) {
    int r;
    asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// floor(x) as an integer in one instruction (x is far inside int range).
__device__ __forceinline__ int floor_int(float x) {
    int r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}

// Untilted splat of one 64-z chunk of one column.  u, hence (iu, fu), is
// constant along the column, so the weights factor into (1-fu, fu) x
// (1-fv, fv) with wu0 = (1-fu)*s, wu1 = fu*s carrying the fixed-point scale,
// and v is affine in z: t = v - 0.5 = B*z_lane + A (B, A per column).  The
// acceptance window 0.55 < v < V-0.55 and the chunk's row range reduce to
// lo < t < hi (lo >= 0.05, so an accepted t is positive and fract(t) =
// t - floor(t) exactly).  Branch free: a rejected voxel adds zero at `spare`,
// a lane-dependent row of the band (one shared address would serialise the
// wave's atomics).  row0 = the LDS byte address of band row floor(t) = 0 of
// the column, so an accepted voxel's first row is row0 + floor(t) * row pitch.
template <class AccT, class AccS>
__device__ __forceinline__ void splat_untilted(float t, float val, unsigned row0, lds_ptr<AccT> spare, float wu0,
                                               float wu1, float lo, float hi) {
    const bool ok = t > lo && t < hi;
    const float fv = __builtin_amdgcn_fractf(t);
    const float w = ok ? val : 0.0f;
    const float g1 = fv * w, g0 = w - g1;
    const unsigned at = __umul24((unsigned)floor_int(t), (unsigned)(kBandStride * sizeof(AccT))) + row0;
    lds_ptr<AccT> p = ok ? (lds_ptr<AccT>)(uintptr_t)at : spare;
    const int q4 = round_half_up(wu0 * g0), q3 = round_half_up(wu1 * g0);
    const int q1 = round_half_up(wu0 * g1), q2 = round_half_up(wu1 * g1);
    __hip_atomic_fetch_add(p, (AccT)(AccS)q4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(p + 1, (AccT)(AccS)q3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(p + kBandStride, (AccT)(AccS)q1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(p + kBandStride + 1, (AccT)(AccS)q2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// splat_untilted for a voxel known to lie in the window (0.05 < t, so fract(t)
// = t - floor(t) exactly): the same terms at the same addresses, without the
// test and the selects.
template <class AccT, class AccS>
__device__ __forceinline__ void splat_inside(float t, float val, unsigned row0, float wu0, float wu1) {
    const float fv = __builtin_amdgcn_fractf(t);
    const float g1 = fv * val, g0 = val - g1;
    const unsigned at = __umul24((unsigned)floor_int(t), (unsigned)(kBandStride * sizeof(AccT))) + row0;
    lds_ptr<AccT> p = (lds_ptr<AccT>)(uintptr_t)at;
    const int q4 = round_half_up(wu0 * g0), q3 = round_half_up(wu1 * g0);
    const int q1 = round_half_up(wu0 * g1), q2 = round_half_up(wu1 * g1);
    __hip_atomic_fetch_add(p, (AccT)(AccS)q4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(p + 1, (AccT)(AccS)q3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(p + kBandStride, (AccT)(AccS)q1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(p + kBandStride + 1, (AccT)(AccS)q2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Terms of pixels (iu, iv), (iu + 1, iv), (iu, iv + 1), (iu + 1, iv + 1) added at p, rounded to nearest.
template <class AccT, class AccS>
__device__ __forceinline__ void splat_rounded(lds_ptr<AccT> p, float t4, float t3, float t1, float t2) {
    const int q4 = __float2int_rn(t4), q3 = __float2int_rn(t3), q1 = __float2int_rn(t1), q2 = __float2int_rn(t2);
    __hip_atomic_fetch_add(p, (AccT)(AccS)q4, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(p + 1, (AccT)(AccS)q3, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(p + kBandStride, (AccT)(AccS)q1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    __hip_atomic_fetch_add(p + kBandStride + 1, (AccT)(AccS)q2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// The per-voxel basis rotation of forwardOrth / backwardOrth (ir.cu:316-328,
// 390-400): rodriguesRotation (ir.cu:597-621) about the axis (cos phi, sin phi,
// 0) with cosine cc and sine sqrt(1 - cc^2), (1 - cc) n n^T + [[cc, -n_z s,
// n_y s], [n_z s, cc, -n_x s], [-n_y s, n_x s, cc]] with n_z = 0.
__device__ __forceinline__ void orth_rotation(float phi, float cc, float R[9]) {
    float sp, cp;
    sincosf(phi, &sp, &cp);
    const float sn = sqrtf(1.0f - cc * cc);
    const float len = sqrtf(cp * cp + sp * sp);
    if (len < 1e-8f) {
        const float I[9] = {1.f, 0.f, 0.f, 0.f, 1.f, 0.f, 0.f, 0.f, 1.f};
#pragma unroll
        for (int i = 0; i < 9; i++) R[i] = I[i];
        return;
    }
    const float nx = cp / len, ny = sp / len, om = 1.0f - cc;
    R[0] = om * nx * nx + cc;
    R[1] = om * nx * ny;
    R[2] = ny * sn;
    R[3] = om * nx * ny;
    R[4] = om * ny * ny + cc;
    R[5] = -nx * sn;
    R[6] = -ny * sn;
    R[7] = nx * sn;
    R[8] = cc;
}

// Orientation-aware XTT weight of channel k at a voxel: S' = R S_k, w =
// max(|S'|^2 - (d.S')^2 / |d|^2, 0) (S'.G)^2, i.e. |B x S'|^2 (S'.G)^2
// (ir.cu:352-359, 410-417).
__device__ __forceinline__ float orth_weight(const float R[9], const Basis& b, int k, float dx, float dy, float dz,
                                             float id2, const ViewGeom& g) {
    const float s0 = fmaf(R[0], b.S[k][0], fmaf(R[1], b.S[k][1], R[2] * b.S[k][2]));
    const float s1 = fmaf(R[3], b.S[k][0], fmaf(R[4], b.S[k][1], R[5] * b.S[k][2]));
    const float s2 = fmaf(R[6], b.S[k][0], fmaf(R[7], b.S[k][1], R[8] * b.S[k][2]));
    const float ds = fmaf(dz, s2, fmaf(dy, s1, dx * s0));
    const float ss = fmaf(s2, s2, fmaf(s1, s1, s0 * s0));
    const float gs = fmaf(g.G[2], s2, fmaf(g.G[1], s1, g.G[0] * s0));
    return fmaxf(fmaf(-ds * ds, id2, ss), 0.f) * (gs * gs);
}

// Untilted view, volume row y' = yp: u(x') = hu + (au0 x' + cu) / (ad0 x' + cd)
// is linear-fractional in x', hence monotone while the denominator is
// positive, so the columns whose u falls in [ua, ub] form an interval.  The
// u of a column is evaluated exactly as the scan's candidate test does; its
// rounding error (a few ulp, far below kRowMargin) can break monotonicity by
// that much, so every decision below keeps kRowMargin clear of the band:
//  - u at both ends of the row below ua (or both above ub): no column can be
//    a candidate, the row is empty;
//  - otherwise the closed-form solution, widened by two columns, is a guess
//    (it degenerates where u hardly varies along the row), accepted only if
//    u lies beyond the band on the proper side at the first column left of it
//    and at the first column right of it;
//  - anything else (denominator not positive, non-finite u, a rejected guess)
//    scans the whole row.
// The scan still tests every column of [xs, xe) exactly, so the result does
// not depend on the guess.
constexpr float kRowMargin = 0.01f;

__device__ __forceinline__ float row_u(const ViewGeom& g, const Dims& d, int x, float yp) {
    const ColForms c = col_forms(g, (float)x - d.xc, yp);
    return fmaf(c.nu, rcpf(c.nd), d.hu);
}

__device__ __forceinline__ void band_columns(const ViewGeom& g, const Dims& d, float yp, float ua, float ub, int& xs,
                                             int& xe) {
    xs = 0;
    xe = d.N;
    const float cu = fmaf(g.au[1], yp, g.au[3]), cd = fmaf(g.ad[1], yp, g.ad[3]);
    const float x0 = -d.xc, x1 = (float)(d.N - 1) - d.xc;
    if (!(fmaf(g.ad[0], x0, cd) > 0.f && fmaf(g.ad[0], x1, cd) > 0.f)) return;
    const float u_first = row_u(g, d, 0, yp), u_last = row_u(g, d, d.N - 1, yp);
    if (!(fabsf(u_first) < 1e30f && fabsf(u_last) < 1e30f)) return;
    const float lo_u = ua - kRowMargin, hi_u = ub + kRowMargin;
    if (fmaxf(u_first, u_last) < lo_u || fminf(u_first, u_last) > hi_u) {
        xe = 0;  // the whole row misses the band
        return;
    }
    if (!(u_first != u_last)) return;
    const bool up = u_last > u_first;
    // x' with u(x') = u: (u - hu)(ad0 x' + cd) = au0 x' + cu
    const float ka = ua - d.hu, kb = ub - d.hu;
    const float xa = (cu - ka * cd) / (ka * g.ad[0] - g.au[0]);
    const float xb = (cu - kb * cd) / (kb * g.ad[0] - g.au[0]);
    const float lo = fminf(xa, xb) + d.xc - 2.0f, hi = fmaxf(xa, xb) + d.xc + 2.0f;
    if (!(lo == lo) || !(hi == hi)) return;
    const int s = (int)fminf(fmaxf(floorf(lo), 0.0f), (float)d.N);
    const int e = (int)fminf(fmaxf(ceilf(hi) + 1.0f, (float)s), (float)d.N);
    if (s > 0) {
        const float u = row_u(g, d, s - 1, yp);
        if (!(up ? u < lo_u : u > hi_u)) return;
    }
    if (e < d.N) {
        const float u = row_u(g, d, e, yp);
        if (!(up ? u > hi_u : u < lo_u)) return;
    }
    xs = s;
    xe = e;
}

// One thread per (code, band, volume row): the scan bounds of forward_item.
// A candidate of band b has iu in [16b - 1, 16b + 16), i.e. u in
// [16b - 0.5, 16b + 15.5), inside [ua, ub] below.
__global__ void k_band_rows(const ViewGeom* __restrict__ vg, const Dims d, int n_codes, int n_bands,
                            int32_t* __restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)n_codes * n_bands * d.N) return;
    const int y = (int)(i % d.N), band = (int)((i / d.N) % n_bands), code = (int)(i / ((int64_t)d.N * n_bands));
    const ViewGeom g = vg[code];
    int xs = 0, xe = d.N;
    if (g.axis != 0.f) {
        const float u0 = (float)(band * kBandU);
        band_columns(g, d, (float)y - d.xc, u0 - 0.5f, u0 + (float)kBandU + 0.5f, xs, xe);
    }
    out[i] = xs | (xe << 16);
}

// ---------------------------------------------------------------------------
// Tilted views: the splat of one band for a scan whose rotation axis is not
// the volume's z axis.  u varies along every volume axis, so a column crosses
// several bands.  Two things keep the lanes busy:
//  - lanes run along the volume axis that the condition's rotation axis is
//    closest to (ViewGeom::lane_axis): the detector row then advances by 0.577
//    to 1 times the magnification from lane to lane.  (Lanes along z, at a
//    tilt near 90 degrees, run along the rays at some views, and all 64 add to
//    the same few pixels.)
//  - of each column only the interval of lane positions that can reach the
//    band is visited, and the intervals of the columns of one row are packed
//    into full waves: slot i of the packed list is position i % L of interval
//    i / L, L the longest interval of the 64 columns looked at together.
// (u, v) and the acceptance tests are those of col_forms and voxel_uv, so the
// images do not depend on the lane axis nor on the packing.
// Bound by VALU issue (0.77 to 0.85 where a CU has blocks; a launch of few
// views leaves 30 to 40 % of the chip's time idle at its end).  A visited voxel
// costs about 45 VALU instructions (nine FMAs for the three forms, the
// reciprocal, the splits, four rounded products) and four LDS adds; with the
// intervals, their packing and the slots that it leaves empty the counters
// read 151 VALU per 64 voxel-views of the volume (128^3, 45 views at 30
// degrees) and 176 (120^3 x 3 coefficients).  Measured against whole columns
// of z in every lane: 120^3 x 3 coefficients, 4 x 60 views tilted by 0, 20, 45
// and 90 degrees, 31.8 -> 2.3 ms per launch; 128^3, 45 views at 30 degrees, 0.96
// -> 0.40 ms.
// ---------------------------------------------------------------------------

// XTT voxel value sum_k mu_k (S_k.G)^2 |B x S_k|^2 vs ratio (ir.cu:1780-1794)
// from the view's row of the weight table (BwdArgs::xw), as the untilted path;
// a weight that rounding leaves below zero (a ray along S_k) is zero.
template <int KM>
__device__ __forceinline__ float xtt_value(const FwdArgs& a, const ViewGeom& g, cptr<float> row, float xp, float yp,
                                           float zp, const float (&mu)[KM]) {
    const Dims& d = a.d;
    const float dx = fmaf(d.vs, xp, g.d0[0]), dy = fmaf(d.vs, yp, g.d0[1]), dz = fmaf(d.vs, zp, g.d0[2]);
    const float id2 = rcpf(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < KM; k++) {
        const float ck = fmaf(xp, row[2 * kXwStride + k], fmaf(yp, row[3 * kXwStride + k], row[4 * kXwStride + k]));
        const float q = fmaf(dz, row[k], ck);
        s = fmaf(fmaxf(fmaf(-q * q, id2, row[kXwStride + k]), 0.f), mu[k], s);
    }
    return s * (d.vs * d.ratio);
}

// forwardOrth voxel value: sum_k |B x R S_k|^2 (R S_k . G)^2 mu_k * vs * ratio.
template <int KM>
__device__ __forceinline__ float orth_value(const FwdArgs& a, const ViewGeom& g, float xp, float yp, float zp,
                                            const float (&mu)[KM], float phi, float cc) {
    const Dims& d = a.d;
    const float dx = fmaf(d.vs, xp, g.d0[0]), dy = fmaf(d.vs, yp, g.d0[1]), dz = fmaf(d.vs, zp, g.d0[2]);
    const float id2 = rcpf(fmaf(dz, dz, fmaf(dy, dy, dx * dx)));
    float R[9];
    orth_rotation(phi, cc, R);
    float s = 0.f;
#pragma unroll
    for (int k = 0; k < KM; k++)
        if (k < d.K) s = fmaf(orth_weight(R, a.b, k, dx, dy, dz, id2, g), mu[k], s);
    return s * (d.vs * d.ratio);
}

// Positions [beg, end) along the lane axis at which a column (forms cu, cd at
// lane coordinate 0, slopes au, ad) can have u in [ua, ub].  u is
// linear-fractional, hence monotone, while the denominator is positive.  The
// ends are widened by a voxel (u's rounding moves them by far less where u
// covers at least a pixel); a column whose denominator changes sign or whose u
// covers less is visited whole.
__device__ __forceinline__ void lane_interval(const Dims& d, int n_lane, float cu, float cd, float au, float ad,
                                              float ua, float ub, int& beg, int& end) {
    const float lo = -d.xc, hi = (float)(n_lane - 1) - d.xc;
    const float d0 = fmaf(ad, lo, cd), d1 = fmaf(ad, hi, cd);
    beg = 0;
    end = n_lane;
    if (!(d0 > 0.f && d1 > 0.f)) return;
    const float u0 = fmaf(fmaf(au, lo, cu), rcpf(d0), d.hu), u1 = fmaf(fmaf(au, hi, cu), rcpf(d1), d.hu);
    const float mn = fminf(u0, u1), mx = fmaxf(u0, u1);
    if (mx < ua || mn > ub) {
        end = 0;
        return;
    }
    if (!(mx - mn >= 1.0f)) return;
    const float ka = ua - d.hu, kb = ub - d.hu;
    const bool up = u1 > u0;
    const float pa = mn >= ua ? (up ? lo : hi) : fmaf(ka, cd, -cu) * rcpf(fmaf(-ka, ad, au));
    const float pb = mx <= ub ? (up ? hi : lo) : fmaf(kb, cd, -cu) * rcpf(fmaf(-kb, ad, au));
    beg = (int)fmaxf(floorf(fminf(pa, pb) + d.xc) - 1.0f, 0.0f);
    end = (int)fminf(ceilf(fmaxf(pa, pb) + d.xc) + 2.0f, (float)n_lane);
    if (end < beg) end = beg;
}

template <int KIND, int WAVES, int KM>
__device__ __forceinline__ void splat_tilted(const FwdArgs& a, const ViewGeom& g, int code, float scale,
                                             lds_ptr<typename FwdAcc<KIND>::T> acc, int u0, int cs, int W, int v0,
                                             int vb) {
    typedef typename FwdAcc<KIND>::T AccT;
    typedef typename FwdAcc<KIND>::S AccS;
    const Dims& d = a.d;
    const int lane = threadIdx.x & 63, wave = uniformi(threadIdx.x >> 6);
    const int cond = code / d.P;
    // axes: lanes along la, columns side by side along ca, one row per wave along ra
    const int own = (int)g.lane_axis;
    const int la = a.lanes_z && own < 2 && !a.vol_axis[own] ? 2 : own;
    const int ca = la == 0 ? 1 : 0, ra = la == 2 ? 1 : 2;
    const int n_lane = la == 2 ? d.nz : d.N, n_row = ra == 2 ? d.nz : d.N;
    auto pick = [](const float (&v)[4], int i) { return i == 0 ? v[0] : (i == 1 ? v[1] : v[2]); };
    const float aul = pick(g.au, la), auc = pick(g.au, ca), aur = pick(g.au, ra);
    const float adl = pick(g.ad, la), adc = pick(g.ad, ca), adr = pick(g.ad, ra);
    // the volume, in a copy with the lane axis contiguous where there is one
    const float* const copy = la == 2 ? nullptr : a.vol_axis[la];
    const int64_t N = d.N;
    const auto vol = to_global((copy ? copy : a.vol) + (KIND == FWD_PLAIN ? (int64_t)cond * a.vol_cond_stride : 0));
    const unsigned s_lane = (copy || la == 2) ? 1u : (la == 0 ? (unsigned)d.N : (unsigned)d.N * (unsigned)d.N);
    const unsigned s_col = (copy || la == 2) ? (unsigned)d.N : (ca == 0 ? (unsigned)d.N : (unsigned)d.N * (unsigned)d.N);
    const int64_t s_row = (copy || la == 2) ? N * N : 1;
    const auto xrow = to_const(a.xw ? a.xw + (int64_t)code * 5 * kXwStride : nullptr);
    const float scalev = (KIND == FWD_PLAIN) ? d.ratio : 1.f;
    // iu in [u0 + cs - 1, u0 + cs + W), with a margin far above the rounding of u
    const float ua = (float)(u0 + cs) - 0.51f, ub = (float)(u0 + cs + W) + 0.51f;
    constexpr int UN = KIND == FWD_XTT ? 1 : 4;  // waves of voxels in flight
    for (int r = wave; r < n_row; r += WAVES) {
        const float rp = (float)r - d.xc;
        const auto vrow = vol + (int64_t)r * s_row;
        const float cur = fmaf(aur, rp, g.au[3]), cdr = fmaf(adr, rp, g.ad[3]);
        for (int c0 = 0; c0 < d.N; c0 += 64) {
            const float cp = (float)(c0 + lane) - d.xc;
            int beg = 0, end = 0;
            if (c0 + lane < d.N)
                lane_interval(d, n_lane, fmaf(auc, cp, cur), fmaf(adc, cp, cdr), aul, adl, ua, ub, beg, end);
            const unsigned long long m = __ballot(end > beg);
            if (m == 0) continue;
            int L = end - beg;
            for (int off = 32; off > 0; off >>= 1) L = max(L, __shfl_xor(L, off));
            L = uniformi(L);
            const int n = __popcll(m);
            // columns with an interval move to the front (a permutation of the lanes)
            const int before = __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
            const int to = end > beg ? before : n + (lane - before);
            const int list = __builtin_amdgcn_ds_permute(to * 4, ((c0 + lane) << 16) | beg);
            const float rL = 1.0f / (float)L;
            const int total = n * L;
            for (int i0 = 0; i0 < total; i0 += 64 * UN) {
                int lp[UN], cc[UN];
                bool in[UN];
                float mu[UN][KIND == FWD_XTT ? KM : 1];
#pragma unroll
                for (int w = 0; w < UN; w++) {
                    const int i = i0 + 64 * w + lane;
                    const int s = (int)(((float)i + 0.5f) * rL);  // i / L
                    const int e = __builtin_amdgcn_ds_bpermute(s * 4, list);
                    lp[w] = (e & 0xffff) + (i - s * L);
                    cc[w] = e >> 16;
                    in[w] = i < total && lp[w] < n_lane;
                    // 64 bits: without a copy one stride is N^2, and from N = 1626 on the sum passes 2^32
                    const int64_t at =
                        in[w] ? (int64_t)((uint64_t)(unsigned)cc[w] * s_col + (uint64_t)(unsigned)lp[w] * s_lane) : 0;
                    if (KIND == FWD_WEIGHT) {
                        mu[w][0] = 1.f;
                    } else if (KIND == FWD_PLAIN) {
                        mu[w][0] = vrow[at];
                    } else {
#pragma unroll
                        for (int k = 0; k < (KIND == FWD_XTT ? KM : 1); k++)
                            mu[w][k] = k < d.K ? vrow[at + k * a.chan_stride] : 0.f;
                    }
                }
#pragma unroll
                for (int w = 0; w < UN; w++) {
                    if (i0 + 64 * w >= total) break;
                    const float lpf = (float)lp[w] - d.xc, ccf = (float)cc[w] - d.xc;
                    const float xp = la == 0 ? lpf : ccf;
                    const float yp = la == 1 ? lpf : (ca == 1 ? ccf : rp);
                    const float zp = la == 2 ? lpf : rp;
                    float u, v;
                    voxel_uv(g, col_forms(g, xp, yp), zp, d, u, v);
                    int iu, iv;
                    float fu, fv;
                    split(u, iu, fu);
                    split(v, iv, fv);
                    const bool ok = in[w] && accept_u(u, d) && accept_v(v, d) &&
                                    (unsigned)(iv - (v0 - 1)) <= (unsigned)vb &&
                                    (unsigned)(iu - (u0 + cs - 1)) <= (unsigned)W;
                    if (!ok) continue;
                    float val;
                    if constexpr (KIND == FWD_XTT) {
                        if (a.coef) {
                            const int64_t at = ((int64_t)(int)(yp + d.xc) * N + (int)(xp + d.xc)) * N + (int)(zp + d.xc);
                            val = orth_value<KM>(a, g, xp, yp, zp, mu[w], a.coef[at], a.coef[at + a.chan_stride]);
                        } else {
                            val = xtt_value<KM>(a, g, xrow, xp, yp, zp, mu[w]);
                        }
                    } else {
                        val = mu[w][0] * scalev;
                    }
                    const float vs = val * scale;
                    const float c1 = (1.0f - fu) * fv, c2 = fu * fv;
                    const float c3 = fu * (1.0f - fv), c4 = (1.0f - fu) * (1.0f - fv);
                    splat_rounded<AccT, AccS>(acc + (iv - v0 + 1) * kBandStride + (iu - u0 + 1), c4 * vs, c3 * vs, c1 * vs, c2 * vs);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Untilted views: the splat of one band.  u is constant along a z column, so a
// column either touches the band or does not, and its terms (u split, t = v -
// 0.5 = B (z - xc) + A) are computed once by the lane that scans it and read
// from there.  CH chunks of 64 z are loaded per column and step, of as many
// columns at once as make 16 loads (at most 8): with one column pair a step
// whatever the depth, a 64-layer volume had two loads in flight per wave and
// spent its time waiting.
// Columns whose z extent lies inside the window (t is monotone in z) run
// without tests; a partial last chunk only masks its lanes (such depths used to
// take masked loads and tests throughout).
// Measured, column pairs of eight chunks -> now: 64^3 / 90 views 94 -> 58 us;
// 203^3 / 20 views 321 -> 207 us; 512^3 / 720 views, bound by VALU issue, 58.8
// against 57.7 ms.
// ---------------------------------------------------------------------------
// MIXED: the untilted views of a launch that also holds tilted ones.  Their images
// keep the bits of splat_tilted (v by voxel_uv, four weighted terms rounded to
// nearest, XTT weights not below zero): the column's terms are then 1/den and the
// form of v at z = xc in place of B and A, and the u weights without the scale.
template <int KIND, int WAVES, int KM, int CH, bool MIXED>
__device__ __forceinline__ void splat_columns(const FwdArgs& a, const ViewGeom& g, int code, gptr<const float> vol,
                                              float wscale, lds_ptr<typename FwdAcc<KIND>::T> acc, int band, int u0,
                                              int cs, int W, int v0, int vb) {
    typedef typename FwdAcc<KIND>::T AccT;
    typedef typename FwdAcc<KIND>::S AccS;
    constexpr bool XTT = KIND == FWD_XTT;
    constexpr int NCOL = XTT ? 1 : (CH >= 2 ? 16 / CH : 8);
    // Few columns are left for a step where a band is split or narrow.  With many columns a step the
    // missing ones repeat the first one's loads, unmasked (128^3, 4 views 110 against 94 us); with four
    // or less the step of any shape takes them (256^3, 4 views 173 against 197 us).
    constexpr bool ANY_N = NCOL > 4;
    constexpr int xws = kXwStride;
    const Dims& d = a.d;
    const int lane = threadIdx.x & 63, wave = uniformi(threadIdx.x >> 6);
    const auto xrow = to_const(a.xw ? a.xw + (int64_t)code * 5 * xws : nullptr);
    // the window of t: 0.55 < v < V - 0.55 (ir.cu:1501) and v0 - 1 <= floor(t) < v0 + vb
    const float t_lo = (v0 >= 2) ? __int_as_float(__float_as_int((float)(v0 - 1)) - 1) : 0.05f;
    const float t_hi = fminf(d.vmax - 0.5f, (float)(v0 + vb));
    const int spare_row = min(lane, vb);  // rows spare_row, spare_row + 1 lie in the band
    const bool rows_all = v0 <= 0 && v0 + vb >= d.V;  // this launch covers every detector row
    const float z_first = -d.xc, z_end = (float)(d.nz - 1) - d.xc;
    float lanef[CH];  // z offset of the lane in each chunk of a step
#pragma unroll
    for (int c = 0; c < CH; c++) lanef[c] = (float)(c * 64 + lane);

    const auto bands = to_global(a.bands ? a.bands + ((int64_t)code * a.n_bands + band) * d.N : nullptr);
    for (int y0 = wave; y0 < d.N; y0 += 64 * WAVES) {
        // the scan bounds of the wave's next 64 rows: lane i holds row y0 + i WAVES
        const int yl = y0 + lane * WAVES;
        const int scan = yl < d.N ? (a.bands ? bands[yl] : d.N << 16) : 0;
        for (int i = 0; i < 64; i++) {
            const int y = y0 + i * WAVES;
            if (y >= d.N) break;
            const float yp = (float)y - d.xc;
            const int xb = lane_i(scan, i);  // columns of this row to scan (the test below is exact)
            const int xs = xb & 0xffff, xe = xb >> 16;
            for (int x0 = xs & ~63; x0 < xe; x0 += 64) {
                const int x = x0 + lane;
                bool cand = false, in = false;
                // this lane's column terms, kept for the candidate loop: t = B (z - xc) + A,
                // the two u weights with the fixed-point scale, the band column
                float sB = 0.f, sA = 0.f, sw0 = 0.f, sw1 = 0.f;
                int scp = 0;
                if (x < d.N) {
                    const ColForms c = col_forms(g, (float)x - d.xc, yp);
                    const float inv = rcpf(c.nd);
                    const float u = fmaf(c.nu, inv, d.hu);
                    if (accept_u(u, d)) {
                        int iu;
                        float fu;
                        split(u, iu, fu);
                        cand = (unsigned)(iu - (u0 + cs - 1)) <= (unsigned)W;
                        scp = iu - u0 + 1;
                        // t (MIXED: v) at the first and last z bounds every lane's: z - xc is exact
                        // and fmaf is monotone in it
                        if (MIXED) {
                            sB = inv;
                            sA = c.nv;
                            sw0 = 1.0f - fu;
                            sw1 = fu;
                            const float va = fmaf(fmaf(g.av[2], z_first, c.nv), inv, d.hv);
                            const float ve = fmaf(fmaf(g.av[2], z_end, c.nv), inv, d.hv);
                            in = rows_all && accept_v(va, d) && accept_v(ve, d);
                        } else {
                            sB = g.av[2] * inv;
                            sA = fmaf(c.nv, inv, d.hv - 0.5f);
                            sw0 = (1.0f - fu) * wscale;
                            sw1 = fu * wscale;
                            const float ta = fmaf(sB, z_first, sA), tb = fmaf(sB, z_end, sA);
                            in = rows_all && fminf(ta, tb) > t_lo && fmaxf(ta, tb) < t_hi;
                        }
                    }
                }
                // XTT: |d|^2 - dz^2 of the column's source->voxel vector d and
                // sig_k (d_x S_k,x + d_y S_k,y), so that sig_k (d.S_k) = dz sig_k S_k,z + xck_k
                float xcxy = 0.f, xck[KM];
                if (XTT) {
                    const float xp = (float)x - d.xc;
                    const float dx = fmaf(d.vs, xp, g.d0[0]), dy = fmaf(d.vs, yp, g.d0[1]);
                    xcxy = fmaf(dy, dy, dx * dx);
#pragma unroll
                    for (int k = 0; k < KM; k++)
                        xck[k] = fmaf(xp, xrow[2 * xws + k], fmaf(yp, xrow[3 * xws + k], xrow[4 * xws + k]));
                }
                const auto row = vol + ((int64_t)y * d.N + x0) * d.N;  // column b of the scan at b N
                // LDS byte address of band row floor(t) = 0 of a column
                auto row0_of = [&](int b) XR_INLINE {
                    return (unsigned)(uintptr_t)(acc + lane_i(scp, b)) +
                           (unsigned)((1 - v0) * kBandStride * (int)sizeof(AccT));
                };
                const unsigned long long mc = __ballot(cand), mi = __ballot(cand && in);
                // columns of mask m, NCOL at a time.  INSIDE: whole columns in the window.
                auto columns = [&](unsigned long long m, auto inside_c) XR_INLINE {
                    constexpr bool INSIDE = decltype(inside_c)::value;
                    while (m) {
                        int b[NCOL], n = 0;
#pragma unroll
                        for (int k = 0; k < NCOL; k++) {
                            b[k] = m ? __ffsll(m) - 1 : b[0];
                            n += m ? 1 : 0;
                            m &= m ? m - 1 : 0;
                        }
                        int zb = 0, ze = d.nz;
                        if (!INSIDE && !rows_all) {
                            zb = d.nz;
                            ze = 0;
#pragma unroll
                            for (int k = 0; k < NCOL; k++) {
                                int zb_k, ze_k;
                                float B = lane_f(sB, b[k]), A = lane_f(sA, b[k]);
                                if (MIXED) {
                                    A = fmaf(A, B, d.hv - 0.5f);
                                    B *= g.av[2];
                                }
                                col_zrange_t(B, A, d, v0, vb, zb_k, ze_k);
                                zb = min(zb, zb_k);
                                ze = max(ze, ze_k);
                            }
                        }
                        // one step: chunks zg, zg + 64, ... of the n columns.  MODE 2: NCOL columns, CH
                        // whole chunks (XTT: and K the compiled count); 1: the last chunk partial; 0: any.
                        auto step = [&](int zg, auto mode_c) XR_INLINE {
                            constexpr int MODE = decltype(mode_c)::value;
                            constexpr bool FULL = XTT ? MODE >= 2 : MODE > 0, EXACT = MODE == 1 || MODE == 2;
                            // t = B (z - xc) + A: z - xc is exact in FP32 (half-integers below
                            // 2^23), so t depends on z alone and not on where the step starts
                            const float zoff = (float)zg - d.xc;
                            const int rem = d.nz - zg;  // layers left
                            const auto there = [&](int c) XR_INLINE { return FULL || zg + c * 64 < ze; };
                            // a chunk that ends past the volume masks its lanes
                            auto in_chunk = [&](int c) XR_INLINE {
                                return MODE >= 2 || (!XTT && MODE == 1 && c < CH - 1) || c * 64 + 64 <= rem || lane < rem - c * 64;
                            };
                            auto splat = [&](int c, float val, float B, float A, unsigned row0, lds_ptr<AccT> spare,
                                             float w0, float w1) XR_INLINE {
                                if constexpr (MIXED) {
                                    const float v = fmaf(fmaf(g.av[2], lanef[c] + zoff, A), B, d.hv);
                                    int iv;
                                    float fv;
                                    split(v, iv, fv);
                                    if (in_chunk(c) && (INSIDE || (accept_v(v, d) && (unsigned)(iv - (v0 - 1)) <= (unsigned)vb))) {
                                        const float vs = val * (KIND == FWD_PLAIN ? d.ratio : (XTT ? d.vs * d.ratio : 1.f)) * wscale;
                                        const float gv = 1.0f - fv;
                                        const lds_ptr<AccT> p = (lds_ptr<AccT>)(uintptr_t)row0 + iv * kBandStride;
                                        splat_rounded<AccT, AccS>(p, w0 * gv * vs, w1 * gv * vs, w0 * fv * vs, w1 * fv * vs);
                                    }
                                    return;
                                }
                                const float t = fmaf(B, lanef[c] + zoff, A);
                                if (in_chunk(c)) {
                                    if (XTT ? (mi >> b[0] & 1) != 0 : INSIDE)
                                        splat_inside<AccT, AccS>(t, val, row0, w0, w1);
                                    else
                                        splat_untilted<AccT, AccS>(t, val, row0, spare, w0, w1, t_lo, t_hi);
                                }
                            };
                            if constexpr (!XTT) {
                                float mu[NCOL][CH];
                                if (KIND != FWD_WEIGHT) {
#pragma unroll
                                    for (int k = 0; k < NCOL; k++)
                                        if (FULL || k < n) {
                                            const auto col = row + (int64_t)b[k] * d.N + lane;
#pragma unroll
                                            for (int c = 0; c < CH; c++)
                                                if (there(c) && in_chunk(c)) mu[k][c] = col[zg + c * 64];
                                        }
                                }
#pragma unroll
                                for (int k = 0; k < NCOL; k++) {
                                    if ((ANY_N || !FULL) && k >= n) break;
                                    const float B = lane_f(sB, b[k]), A = lane_f(sA, b[k]);
                                    const float w0 = lane_f(sw0, b[k]), w1 = lane_f(sw1, b[k]);
                                    const unsigned row0 = row0_of(b[k]);
                                    const lds_ptr<AccT> spare = acc + lane_i(scp, b[k]) + spare_row * kBandStride;
#pragma unroll
                                    for (int c = 0; c < CH; c++) {
                                        if (!there(c)) break;
                                        splat(c, KIND == FWD_WEIGHT ? 1.f : mu[k][c], B, A, row0, spare, w0, w1);
                                    }
                                }
                            } else {
                                // Per voxel the value sum_k mu_k (S_k.G)^2 |B x S_k|^2 (ir.cu:1780-1794)
                                // is sum_k mu_k (g2s_k - q_k^2 / |d|^2), q_k = sig_k (d.S_k) affine in z;
                                // vs * ratio rides in the splat weights.  k is the outer loop of a chunk
                                // pair, so only one k's constants are live at a time.
                                const float cxy = lane_f(xcxy, b[0]);
                                float mu[CH][KM];
                                if (MODE >= 2) {
                                    // one address per channel walked from the previous one (the chunks
                                    // are immediate offsets); opaque, or the compiler keeps all K
                                    // channels' lane addresses in registers across the columns
                                    auto col = row + (int64_t)b[0] * d.N + (zg + lane);
                                    asm volatile("" : "+v"(col));
#pragma unroll
                                    for (int k = 0; k < KM; k++) {
                                        if (!EXACT && k >= d.K) break;
#pragma unroll
                                        for (int c = 0; c < CH; c++) mu[c][k] = col[c * 64];
                                        col += a.chan_stride;
                                    }
                                } else {
                                    // lanes past the end read the last layer; a chunk that is not there reads nothing
#pragma unroll
                                    for (int c = 0; c < CH; c++) {
#pragma unroll
                                        for (int k = 0; k < KM; k++) mu[c][k] = 0.f;
                                        if (there(c)) {
                                            auto col = row + (int64_t)b[0] * d.N + (zg + min(c * 64 + lane, rem - 1));
                                            asm volatile("" : "+v"(col));
#pragma unroll
                                            for (int k = 0; k < KM; k++) {
                                                if (!EXACT && k >= d.K) break;
                                                mu[c][k] = *col;
                                                col += a.chan_stride;
                                            }
                                        }
                                    }
                                }
                                float dz[CH], id2[CH], val[CH];
#pragma unroll
                                for (int c = 0; c < CH; c++) {
                                    dz[c] = fmaf(d.vs, lanef[c] + zoff, g.d0[2]);
                                    id2[c] = rcpf(fmaf(dz[c], dz[c], cxy));
                                    val[c] = 0.f;
                                }
#pragma unroll
                                for (int k = 0; k < KM; k++) {
                                    if (EXACT || k < d.K) {
                                        const float ck = lane_f(xck[k], b[0]), sS2 = xrow[k], g2s = xrow[xws + k];
#pragma unroll
                                        for (int c = 0; c < CH; c++) {
                                            const float q = fmaf(dz[c], sS2, ck);
                                            float w = fmaf(-q * q, id2[c], g2s);
                                            if (MIXED) w = fmaxf(w, 0.f);
                                            val[c] = fmaf(w, mu[c][k], val[c]);
                                        }
                                    }
                                }
                                const float B = lane_f(sB, b[0]), A = lane_f(sA, b[0]);
                                const float w0 = lane_f(sw0, b[0]), w1 = lane_f(sw1, b[0]);
                                const unsigned row0 = row0_of(b[0]);
                                const lds_ptr<AccT> spare = acc + lane_i(scp, b[0]) + spare_row * kBandStride;
#pragma unroll
                                for (int c = 0; c < CH; c++) {
                                    if (!there(c)) break;
                                    splat(c, val[c], B, A, row0, spare, w0, w1);
                                }
                            }
                        };
                        for (int zg = zb & ~63; zg < ze; zg += 64 * CH) {
                            const int left = ze - zg;
                            const bool cols = ANY_N || n == NCOL;
                            if (cols && left >= 64 * CH && (!XTT || d.K == KM))
                                step(zg, std::integral_constant<int, 2>());
                            else if (XTT && left >= 64 * CH)
                                step(zg, std::integral_constant<int, 3>());
                            else if (XTT ? d.K == KM : INSIDE && cols && left > 64 * (CH - 1))
                                step(zg, std::integral_constant<int, 1>());
                            else
                                step(zg, std::integral_constant<int, 0>());
                        }
                    }
                };
                // XTT: one copy of the loop (its registers), the window decided per column
                if constexpr (!XTT) columns(mi, std::true_type());
                columns(XTT ? mc : mc & ~mi, std::false_type());
            }
        }
    }
}

// One (band, view) work item o = band * n_slots + slot of a forward launch.
// step selects the view list views + step*n_slots (a solver's subset step);
// loss receives the item's share of sum |y - p|.
// AXIS: every view of the launch is untilted.  MIXED: otherwise, those that are
// take splat_columns (with the bits of splat_tilted).
template <int KIND, bool AXIS, int WAVES, int KM, int CH, bool MIXED>
__device__ __forceinline__ void forward_item(const FwdArgs& a, int o, int step, double* loss,
                                             unsigned long long* acc_raw, int v0, int vb) {
    typedef typename FwdAcc<KIND>::T AccT;
    typedef typename FwdAcc<KIND>::S AccS;
    const lds_ptr<AccT> acc = (lds_ptr<AccT>)acc_raw;
    const Dims& d = a.d;
    // Item o = (sub-band j, slot).  Sub-band j = (band, sub) owns the kBandU/n_sub
    // detector columns us + [0, W) of the band's accumulator; a split launch
    // hands out the central (heaviest) sub-bands first.
    static_assert(kBandU == 16, "sub-band shifts assume 16-column bands");
    const int nsub = a.n_sub > 1 ? a.n_sub : 1;
    const int lw = nsub == 4 ? 2 : (nsub == 2 ? 3 : 4);  // log2 of W
    int j = o / a.n_slots;
    const int slot = o % a.n_slots;
    if (nsub > 1) {
        const int mid = (a.n_bands * nsub) >> 1;
        j = (j & 1) ? mid - ((j + 1) >> 1) : mid + (j >> 1);
    }
    const int band = j >> (4 - lw), sub = j & (nsub - 1);
    const int W = 1 << lw, cs = sub << lw;  // the item's columns cs + [0, W) of the band
    const auto views = to_const(a.views + (int64_t)step * a.n_slots);
    const auto accum = to_global(a.accum ? a.accum + (int64_t)step * a.n_slots : nullptr);
    const auto proj = to_global(a.proj);
    const int code = views[slot];
    const int cond = code / d.P;
    const ViewGeom g = to_const(a.vg)[code];
    const int u0 = band * kBandU;
    const int rows = vb + 2;
    for (int i = threadIdx.x; i < rows * kBandStride; i += 64 * WAVES) acc[i] = 0ull;
    // Fixed-point scale.  Weight pass (64-bit words): a power of two 2^S with
    // the largest term < 2^30 * 2^-S.  Other passes (32-bit words): the bound
    // of a pixel sum (wmul * max|voxel| * fsum, each factor an upper bound
    // with its own margin) maps to 2^31 (1 - 2^-10), so every sum of rounded
    // terms stays inside the signed 32-bit range while using all but the
    // last fraction of a bit of it.
    const float bound = fmaxf(a.wmul * (*to_global(a.vmax)) * a.fsum, 1e-30f);
    float scale, unscale;
    if (KIND == FWD_WEIGHT) {
        int e = 0;
        (void)frexpf(bound, &e);
        const int S = min(max(30 - e, -100), 100);
        scale = ldexpf(1.0f, S);
        unscale = ldexpf(1.0f, -S);
    } else {
        scale = fminf(fmaxf(2145386496.0f / bound, 0x1p-100f), 0x1p100f);
        unscale = a.out_scale / scale;
    }
    __syncthreads();

    const int lane = threadIdx.x & 63, wave = uniformi(threadIdx.x >> 6);
    const auto vol = to_global(a.vol + (KIND == FWD_PLAIN ? (int64_t)cond * a.vol_cond_stride : 0));
    // value scale folded into the untilted splat weights: ratio (ir.cu:1513-1518),
    // XTT vs * ratio (ir.cu:1791)
    const float scalev = (KIND == FWD_PLAIN) ? d.ratio : (KIND == FWD_XTT ? d.vs * d.ratio : 1.f);
    // The untilted views of a launch that also holds tilted ones need not pay for the tilt (unless the
    // basis is rotated per voxel): 384^3, eight such views 1854 us as tilted ones, 800 as columns.
    bool columns = AXIS;
    if constexpr (AXIS || MIXED) {
        columns = AXIS || (g.axis != 0.f && !a.coef);
        if (columns)
            splat_columns<KIND, WAVES, KM, CH, MIXED>(a, g, code, vol, AXIS ? scale * scalev : scale, acc, band, u0, cs, W,
                                                      v0, vb);
    }
    if constexpr (!AXIS) {
        if (!columns) splat_tilted<KIND, WAVES, KM>(a, g, code, scale, acc, u0, cs, W, v0, vb);
    }
    __syncthreads();

    double lsum = 0.0, l2sum = 0.0;  // sum |y - p|, sum (y - p)^2 (OUT_RESIDUAL_L2)
    float fmax_loc = 0.0f;  // weight pass: largest per-pixel weight sum
    const int64_t img = (int64_t)(code - a.code_base) * d.V * d.U;
    const int64_t nimg = (int64_t)code * d.V * d.U;
    const bool acc_old = (KIND != FWD_WEIGHT) && accum && accum[slot];
    for (int i = threadIdx.x; i < (vb << lw); i += 64 * WAVES) {
        const int r = i >> lw, cc = cs + (i & (W - 1));
        const int uu = u0 + cc, vv = v0 + r;
        if (uu >= d.U || vv >= d.V) continue;
        const float s = (float)(AccS)acc[(r + 1) * kBandStride + cc + 1] * unscale;
        const int64_t pix = img + (int64_t)vv * d.U + uu;
        const int64_t npix = nimg + (int64_t)vv * d.U + uu;
        if (a.out_mode == OUT_NORM_TABLE) {
            const float L = (float)chord_length(to_global(a.cg)[code], uu, vv, d);
            proj[pix] = L / (s + 1e-5f);
            fmax_loc = fmaxf(fmax_loc, s);
            continue;
        }
        float p = (acc_old ? proj[pix] : 0.f) + s;
        if (a.out_mode == OUT_RAW) {
            proj[pix] = p;
            continue;
        }
        p = p * to_global(a.norm)[npix];
        if (a.out_mode == OUT_NORMALISED) {
            proj[pix] = p;
        } else {
            const float yv = to_global(a.sino)[pix];
            lsum += (double)fabsf(yv - p);
            if (a.out_mode == OUT_RESIDUAL || a.out_mode == OUT_RESIDUAL_L2) {
                const float rv = yv - p;
                proj[pix] = rv;
                l2sum = fma((double)rv, (double)rv, l2sum);
            } else {
                float q = p;
                if (q != 0.0f) q = yv / q;
                if (q > 2.0f) q = 2.0f;
                proj[pix] = q;
            }
        }
    }
    if (a.out_mode == OUT_NORM_TABLE && a.fmax) {
        for (int off = 32; off > 0; off >>= 1) fmax_loc = fmaxf(fmax_loc, __shfl_xor(fmax_loc, off));
        if (lane == 0) atomicMax((unsigned int*)a.fmax, __float_as_uint(fmax_loc));
    }
    if (a.out_mode == OUT_RATIO || a.out_mode == OUT_RESIDUAL || a.out_mode == OUT_RESIDUAL_L2) {
        // Cross-wave sums through LDS past the band accumulator (8-byte aligned
        // slots: WAVES for the L1 sum, then WAVES for the squared sum).
        double* red = reinterpret_cast<double*>(acc_raw + fwd_red_slot(rows, sizeof(AccT)));
        const bool l2 = a.out_mode == OUT_RESIDUAL_L2;
        lsum = wave_sum(lsum);
        if (l2) l2sum = wave_sum(l2sum);
        if (lane == 0) {
            red[wave] = lsum;
            if (l2) red[WAVES + wave] = l2sum;
        }
        __syncthreads();
        if (threadIdx.x == 0) {
            double t = 0.0, t2 = 0.0;
            for (int w = 0; w < WAVES; w++) t += red[w];
            atomicAdd(loss, t);
            if (l2) {
                for (int w = 0; w < WAVES; w++) t2 += red[WAVES + w];
                atomicAdd(loss + 1, t2);
            }
        }
    }
}

// Item order of a forward launch.  Items (band j, slot) are numbered
// j*n_slots + slot (band-major).  With view_group G > 0 the launch walks groups
// of G consecutive slots, every band of a group before the next group, and G
// slots of one band next to each other: blocks running at the same time then
// read the slabs of one band at G neighbouring views, which overlap, so a
// column fetched by one is found in L2 by the others (at 512^3 / 720 views the
// forward reads 2.6x less from HBM than band-major over all views).  The order
// changes no result: every item writes its own pixels.
__device__ __forceinline__ int view_grouped(const FwdArgs& a, int oi) {
    if (a.view_group <= 0 || a.n_sub > 1) return oi;
    const int nb = a.n_bands, G = a.view_group;
    const int full = (a.n_slots / G) * G * nb;
    int jj, sl;
    if (oi < full) {
        const int grp = oi / (nb * G), r = oi - grp * nb * G;
        jj = r / G;
        sl = grp * G + (r - jj * G);
    } else {
        const int r = oi - full, gl = a.n_slots - (a.n_slots / G) * G;
        jj = r / gl;
        sl = (a.n_slots / G) * G + (r - jj * gl);
    }
    return jj * a.n_slots + sl;
}

// two blocks per CU: at most 80 VGPRs in 12-wave blocks, 128 in 8-wave ones
template <int KIND, bool AXIS, int KM, int WAVES, int CH>
__global__ __launch_bounds__(64 * WAVES, WAVES == 12 ? 6 : 4) void k_forward(const FwdArgs a) {
    extern __shared__ unsigned long long acc_raw[];
    const int per_chunk = a.n_bands * max(a.n_sub, 1) * a.n_slots;
    const int nblk = per_chunk * a.n_chunks;
    const int per_xcd = (nblk + 7) / 8;
    // XCD-chunked order: each XCD walks a contiguous run of (row chunk, band,
    // view) triples in the view-grouped order of view_grouped, so concurrent
    // blocks on one L2 share a few bands at adjacent views.  A split launch
    // (few views) lists its heaviest items first; there blocks take items in
    // launch order, so that consecutive (round-robin dispatched) blocks spread
    // them over the XCDs.
    const int o = a.n_sub > 1 ? (int)blockIdx.x : (int)(blockIdx.x % 8) * per_xcd + (int)(blockIdx.x / 8);
    if (o >= nblk) return;
    const int chunk = o / per_chunk;
    const int v0 = a.v0 + chunk * a.vb;
    const int vb = min(a.vb, a.d.V - v0);
    forward_item<KIND, AXIS, WAVES, KM, CH, !AXIS>(a, view_grouped(a, o - chunk * per_chunk), 0, a.loss, acc_raw, v0, vb);
}

// Work queue of a persistent launch: q[0] hands out tickets 0, 1, 2, ...; a
// block stops at its first ticket >= total and counts itself in q[1]; the last
// block to stop resets both words, so the next launch (or graph replay) starts
// from zero without a host-side clear.  Every block stops after one failed
// ticket: there is no wait on other blocks.
__device__ __forceinline__ unsigned take_ticket(unsigned* q, unsigned total) {
    const unsigned t = __hip_atomic_fetch_add(q, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (t >= total) {
        const unsigned done = __hip_atomic_fetch_add(q + 1, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT);
        if (done == gridDim.x - 1) {
            __hip_atomic_store(q, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(q + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    return t;
}

// Item holding ticket t: the first i with item_end[i] > t (binary search).
__device__ __forceinline__ int find_item(const int* __restrict__ item_end, int n_items, int t) {
    int lo = 0, hi = n_items - 1;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (item_end[mid] > t)
            hi = mid;
        else
            lo = mid + 1;
    }
    return lo;
}

// Persistent forward launch over many problems: items[i] is one (problem,
// detector-row chunk) launch description with item_end[i] - item_end[i-1]
// (band, view) blocks.  A fixed grid of resident blocks pulls tickets in order,
// so the long items listed first are started first and the short ones fill
// the tail.  ticket_slot: index of a free 8-byte LDS word past every item's
// band accumulator.
template <int KIND, int AXES, int WAVES, int KM = 1>
__device__ __forceinline__ void forward_batch_loop(const FwdArgs* __restrict__ items,
                                                   const int* __restrict__ item_end, int n_items, unsigned* queue,
                                                   int ticket_slot, int step, int loss_shift) {
    extern __shared__ unsigned long long acc_raw[];
    lds_u64* const tk = (lds_u64*)acc_raw + ticket_slot;
    const int total = item_end[n_items - 1];
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) *tk = take_ticket(queue, (unsigned)total);
        __syncthreads();
        // uniform across the block: keeps the item's arguments in scalar registers
        const int t = __builtin_amdgcn_readfirstlane((int)*tk);
        if (t >= total) break;
        const int i = find_item(item_end, n_items, t);
        const FwdArgs& a = items[i];
        const int o = view_grouped(a, t - (i ? item_end[i - 1] : 0));
        double* loss = a.loss ? a.loss + loss_shift : nullptr;
        if (AXES == 1 || a.axis)
            forward_item<KIND, true, WAVES, KM, KIND == FWD_XTT ? kXttChunks : 8, false>(a, o, step, loss, acc_raw, a.v0,
                                                                                       a.vb);
        else
            forward_item<KIND, false, WAVES, KM, 8, false>(a, o, step, loss, acc_raw, a.v0, a.vb);
    }
}

// Persistent forward of XTT problems (forwardProjXTT, ir.cu:1753-1804): the
// same loop with the directional splat, KM >= every item's basis count.
template <int KM>
__global__ __launch_bounds__(64 * kFwdXttWaves, 4) void k_forward_batch_xtt(const FwdArgs* __restrict__ items,
                                                                       const int* __restrict__ item_end,
                                                                       int n_items, unsigned* queue, int ticket_slot,
                                                                       int step, int loss_shift) {
    forward_batch_loop<FWD_XTT, 0, kFwdXttWaves, KM>(items, item_end, n_items, queue, ticket_slot, step, loss_shift);
}

template <int KIND>
__global__ __launch_bounds__(64 * kFwdBatchWaves) void k_forward_batch(const FwdArgs* __restrict__ items,
                                                                  const int* __restrict__ item_end, int n_items,
                                                                  unsigned* queue, int ticket_slot, int step,
                                                                  int loss_shift) {
    forward_batch_loop<KIND, 0, kFwdBatchWaves>(items, item_end, n_items, queue, ticket_slot, step, loss_shift);
}

// The same loop when every item is untilted: without the tilted path the
// kernel needs fewer registers, so 12-wave blocks fit two per CU.
template <int KIND>
__global__ __launch_bounds__(64 * kFwdWaves) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_forward_batch_axis(const FwdArgs* __restrict__ items,
                                                                      const int* __restrict__ item_end, int n_items,
                                                                      unsigned* queue, int ticket_slot, int step,
                                                                      int loss_shift) {
    forward_batch_loop<KIND, 1, kFwdWaves>(items, item_end, n_items, queue, ticket_slot, step, loss_shift);
}

// ---------------------------------------------------------------------------
// Backprojection gather with fused update.  A block of WAVES waves laid out as
// a gx x gy grid owns a voxel tile; a wave owns CX x CY columns, a lane ZPL
// voxels (z = z0 + lane + 64 q) in each, so the per-column terms of a view are
// read once per ZPL voxels.  Everything of a view that is the same in all
// lanes of a wave is computed lane-parallel 16 views at a time into LDS: the
// block's detector footprints by wave 0 (lane = view x corner pair), the
// column terms by every wave for its own columns (lane = view x column, or x
// channel quarter); the view loop reads them back with broadcast LDS loads.
//
// The footprints are staged in LDS VB views (a group) ahead, in 2 VB buffers,
// with one barrier per group.  A footprint is fetched into registers and
// stored after the view (LOOK = 1) or the group (LOOK = VB) that is accumulated
// meanwhile.  Large tiles take VB = 2, LOOK = 1: the work of one view covers a
// load's latency.  Small tiles take VB = LOOK = 8, where it does not: one
// latency per eight views.
//
// The update (MLEM / ART / FDK / raw) is applied at the end: each voxel is read
// and written once per subset.
//
// Bound by VALU issue (about 15 instructions per 64 voxel-views of a whole
// column), the footprint's edges and, with few views, the tile's start.
// Measured, before -> now: MLEM 512^3 / 720 views 60.4 -> 48.7 ms, 64^3 / 90
// views 184 -> 41 us, 203^3 / 20 views 249 -> 152 us; FDK 320^3 / 401 views
// 18.2 -> 7.8 ms; ART 128^3 tilted by 30 degrees, 45 views 478 -> 178 us.
// ---------------------------------------------------------------------------
template <int KIND>
struct IsXtt {
    static constexpr bool value = (KIND == BWD_XTT_RAW || KIND == BWD_XTT_MLEM || KIND == BWD_XTT_ART);
};

constexpr int kBwdBatch = 16;                              // views per batch of per-view terms
constexpr int kFootWords = 12;  // iu_lo, iv_lo, W, Ws | R, flags, code, -, then the staging words: address (2), range, H
constexpr int kBwdFootArea = 2 * kBwdBatch * kFootWords;   // words, block-wide, two batches
enum FootFlag { FOOT_STAGED = 1, FOOT_EMPTY = 2, FOOT_INSIDE = 4 };

// Tile shape and staging of a backprojection kernel.  NP: staged floats per
// thread and view.  WF > 0: every footprint is staged WF texels wide (a power
// of two), threads / WF rows per pass, whole passes; the row stride WF + 1 is
// then a constant, and so are a thread's offsets into the image and the buffer.
// WF = 0: footprints of any width up to SB floats (tilted views; untilted ones
// with more than about 1.4 detector pixels per voxel).
template <int KIND_, int WAVES_, int CX_, int CY_, int ZPL_, int KM_, int VB_, int LOOK_, int WF_, int NP_>
struct BwdCfg {
    static constexpr int KIND = KIND_, WAVES = WAVES_, CX = CX_, CY = CY_, ZPL = ZPL_, VB = VB_, LOOK = LOOK_,
                         WF = WF_, NP = NP_;
    static constexpr int R = WF_ ? 64 * WAVES_ / (WF_ ? WF_ : 1) : 0;  // rows per pass
    static constexpr int SB = WF_ ? NP_ * R * (WF_ + 1) : NP_ * 64 * WAVES_;  // floats per staging buffer
    static constexpr bool XTT = IsXtt<KIND_>::value;
    static constexpr int KM = XTT ? KM_ : 1;
    static constexpr int NC = CX_ * CY_;
    static constexpr int threads = 64 * WAVES_;
    static constexpr int KP = XTT ? (KM_ + 3) & ~3 : 0;  // channel constants, padded for 16-byte LDS loads
    // term words of one (view, column).  Untilted: Bc, Ac, fu, base, hi, lu, iu,
    // wcol or cxy; tilted: nu, nv, nd, -, au2, av2, ad2, wcol or cxy; then ca[KP]
    static constexpr int TW = 8 + KP;
    static constexpr int term_area = kBwdBatch * NC * TW;  // words per wave
    static constexpr int words = 2 * VB_ * SB + kBwdFootArea + WAVES_ * term_area;
    // past these: WAVES words of per-wave max |voxel|, the persistent launch's item and ticket
    static constexpr size_t lds_bytes = (words + WAVES_ + 2) * sizeof(float);
    static_assert(NC == 1 || NC == 2 || NC == 4, "a term batch maps 4 lanes to a view");
    static_assert(kBwdBatch % (2 * VB_) == 0 && VB_ % LOOK_ == 0, "whole groups per batch");
};

// The shapes that the persistent launches, the tile settings and large
// standalone launches use.  The plain kinds (about 110 VGPRs, 4 waves per SIMD)
// run one 16-wave block per CU; XTT runs 8-wave blocks, two per CU, so one
// block accumulates while the other waits at its barrier (its footprints are
// small).  Measured with a barrier per view: XTT 150 against 167 ms per
// backprojection at 256^3 x 13 coefficients, 4 x 360 views; the plain kinds in
// 8-wave blocks (half the tile, 6144-float staging) 70 against 67 ms at 512^3 /
// 720 views.
template <int KIND, int ZPL, int KM>
struct BwdLarge {
    static constexpr bool XTT = IsXtt<KIND>::value;
    typedef typename std::conditional<XTT, BwdCfg<KIND, 8, 1, 1, ZPL, KM, 2, 1, 8, 3>,
                                      BwdCfg<KIND, 16, 2, 2, ZPL, 1, 2, 1, 16, 7>>::type Cfg;
    typedef typename std::conditional<XTT, BwdCfg<KIND, 8, 1, 1, ZPL, KM, 2, 1, 0, 7>,
                                      BwdCfg<KIND, 16, 2, 2, ZPL, 1, 2, 1, 0, 7>>::type Wide;
};
// Few tiles (small volumes): one column and 64 voxels per wave, eight views per
// barrier.
template <int KIND>
struct BwdSmall {
    typedef BwdCfg<KIND, 8, 1, 1, 1, 1, 8, 8, 8, 2> Cfg;
};

struct Foot {
    int iu_lo, iv_lo, W, H, Ws, R;  // R: footprint rows staged per pass of the block's threads
    int flags;
};

// What staging a footprint needs: the buffer descriptor's base and range (0 where
// the footprint is not staged: every load reads 0), the rows; any-width staging
// also W, Ws and R.
struct FootSrc {
    unsigned lo, hi, range;
    int H, W, Ws, R;
};

// Footprint from the extremes of the tile's projected corners (bad: a corner
// behind the source or far off the detector, so the extremes bound nothing).
// INSIDE: every voxel of the tile lies in the acceptance window, with a margin
// far above the rounding of u and v.
template <class C>
__device__ __forceinline__ Foot foot_from_extent(float umn, float umx, float vmn, float vmx, int bad, const Dims& d) {
    Foot f{0, 0, 0, 0, 0, 0, 0};
    if (bad) return f;  // direct (unstaged) reads
    // texels iu and iu + 1 of every voxel, with a margin far above the rounding of u and v
    f.iu_lo = max((int)floorf(umn - 0.51f), 0);
    const int iu_hi = min((int)floorf(umx - 0.49f) + 1, d.U - 1);
    f.iv_lo = max((int)floorf(vmn - 0.51f), 0);
    const int iv_hi = min((int)floorf(vmx - 0.49f) + 1, d.V - 1);
    f.W = iu_hi - f.iu_lo + 1;
    f.H = iv_hi - f.iv_lo + 1;
    if (f.W <= 1 || f.H <= 1) {
        f.flags = FOOT_EMPTY;  // entirely off the detector: nothing is accepted
        return f;
    }
    f.Ws = C::WF ? C::WF + 1 : f.W | 1;
    f.R = C::WF ? C::R : C::threads / f.W;
    if ((C::WF ? f.W <= C::WF : f.Ws * f.H <= C::SB) && f.H <= C::NP * f.R) {
        f.flags = FOOT_STAGED;
        if (umn > 0.56f && umx < d.umax - 0.01f && vmn > 0.56f && vmx < d.vmax - 0.01f) f.flags |= FOOT_INSIDE;
    }
    return f;
}

// Word 3 of a raw buffer descriptor on gfx9-family GPUs (32-bit data, no
// swizzle, stride 0): the range check is on the byte offset alone.
constexpr int kBufferWord3 = 0x00020000;

// Staging of one view's footprint (W x H texels of the view's U-wide image,
// whose first is the descriptor's base) into an LDS buffer of row stride Ws:
// fetched into registers, stored later.  A pass is one raw buffer load at a
// per-lane byte offset; its range ends with the image, so a row below the
// image's last reads 0.
// Fixed width: thread t owns column t % WF of rows t / WF + k R.  Its byte
// offsets are the same for every view, and whole passes are loaded and stored:
// columns past W (which may run into the next image row) and rows past H are
// never read back.  (Up to two passes are issued without a look at H.)
template <class C>
struct FootStage {
    float pre[C::NP];
    unsigned voff;  // byte offset of the thread's first texel from the footprint's
    int lds0;

    __device__ __forceinline__ void init(int U) {
        const int r0 = threadIdx.x / C::WF, c = threadIdx.x % C::WF;
        voff = (unsigned)(r0 * U + c) * 4u;
        lds0 = r0 * (C::WF + 1) + c;
    }
    __device__ __forceinline__ void fetch(const FootSrc& f, int U) {
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)(((uint64_t)f.hi << 32) | f.lo), (short)0,
                                                            (int)f.range, kBufferWord3);
        const unsigned step = (unsigned)(C::R * U) * 4u;
#pragma unroll
        for (int k = 0; k < C::NP; k++)
            if (C::NP <= 2 || k * C::R < f.H)
                pre[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, voff + k * step, 0, 0));
    }
    __device__ __forceinline__ void store(lds_float* buf, const FootSrc& f) const {
#pragma unroll
        for (int k = 0; k < C::NP; k++)
            if (C::NP <= 2 || k * C::R < f.H) buf[lds0 + k * C::R * (C::WF + 1)] = pre[k];
    }
};

// Any width: passes of R = threads / W rows, thread t owning column t % W of
// rows r0 + k R, r0 = t / W (one division per view).  Only the passes the
// footprint needs are issued and stored (uniform tests); only the last needs a
// per-lane row test.
template <class C>
struct FootStageAny {
    float pre[C::NP];
    int r0, lds0;  // lds0 = r0 Ws + c; r0 >= R: the thread stages nothing

    __device__ __forceinline__ void init(int) {}
    __device__ __forceinline__ void fetch(const FootSrc& f, int U) {
        r0 = (int)((float)threadIdx.x * rcpf((float)f.W));  // within 1 of t / W: corrected below
        int c = (int)threadIdx.x - r0 * f.W;
        if (c < 0) {
            r0--;
            c += f.W;
        } else if (c >= f.W) {
            r0++;
            c -= f.W;
        }
        lds0 = r0 * f.Ws + c;
        const auto rsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(uintptr_t)(((uint64_t)f.hi << 32) | f.lo), (short)0,
                                                            (int)f.range, kBufferWord3);
        unsigned voff = ((unsigned)r0 * (unsigned)U + (unsigned)c) * 4u;
        // opaque to the optimiser, so that pass k adds the uniform k * step
        // (one add) instead of recomputing (row + k R) * U (a quarter-rate multiply)
        asm volatile("" : "+v"(voff));
        const unsigned step = (unsigned)f.R * (unsigned)U * 4u;
#pragma unroll
        for (int k = 0; k < C::NP; k++)
            if (k * f.R < f.H)
                pre[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, voff + k * step, 0, 0));
    }
    __device__ __forceinline__ void store(lds_float* buf, const FootSrc& f) const {
        if (r0 >= f.R) return;
        const int rs = f.R * f.Ws;
#pragma unroll
        for (int k = 0; k < C::NP; k++) {
            if ((k + 1) * f.R <= f.H)
                buf[lds0 + k * rs] = pre[k];
            else if (k * f.R < f.H && r0 + k * f.R < f.H)
                buf[lds0 + k * rs] = pre[k];
        }
    }
};

// Fused update of a backprojection tile: every voxel of the lane's columns is
// read and written once (raw accumulate, MLEM ratio, ART step or FDK sum).
// Invariant relied on by the solvers: the MLEM / ART tiles of a launch cover
// and write every voxel of the volume, so the maximum of the values written
// here is the volume's max |voxel| exactly, and the next forward takes its
// fixed-point scale from it.  A tile skipped for any reason (say, outside the
// field of view) would leave that bound too small.  (Layers z >= nz are not
// visited; a plan sets nz < N only where those layers are held at zero.)
template <class C>
__device__ __forceinline__ float backward_update(const BwdArgs& a, const float (&tmp)[C::NC][C::ZPL][C::KM],
                                                 const float (&fac)[C::NC][C::ZPL][C::KM], const int (&nwhole)[C::NC],
                                                 int xb, int yb, int z0, int lane) {
    // returns max |updated voxel| of this lane (MLEM / ART kinds)
    constexpr int KIND = C::KIND;
    const Dims& d = a.d;
    const auto vol = to_global(a.vol);
    float vmx = 0.f;
#pragma unroll
    for (int cidx = 0; cidx < C::NC; cidx++) {
        const int x = xb + cidx % C::CX, y = yb + cidx / C::CX;
        if (x >= d.N || y >= d.N) continue;
#pragma unroll
        for (int q = 0; q < C::ZPL; q++) {
            const int z = z0 + lane + 64 * q;
            if (z >= d.N) continue;
            const int64_t idx = ((int64_t)y * d.N + x) * d.N + z;
#pragma unroll
            for (int k = 0; k < C::KM; k++) {
                if (C::XTT && k >= d.K) continue;
                const int64_t vi = idx + (int64_t)k * a.chan_stride;
                const float t = tmp[cidx][q][k], fc = fac[cidx][q][k] + (float)nwhole[cidx];
                if (KIND == BWD_RAW || KIND == BWD_XTT_RAW) {
                    to_global(a.tmp)[vi] += t;
                    to_global(a.factor)[vi] += fc;
                } else if (KIND == BWD_MLEM || KIND == BWD_XTT_MLEM) {
                    const float mu = vol[vi];
                    const float nv = (fc == 0.0f) ? 0.0f : mu * t / fc;
                    vol[vi] = nv;
                    vmx = fmaxf(vmx, fabsf(nv));
                } else if (KIND == BWD_ART || KIND == BWD_XTT_ART) {
                    const float nv = vol[vi] + a.alpha * t;
                    vol[vi] = nv;
                    vmx = fmaxf(vmx, fabsf(nv));
                } else {  // BWD_FDK
                    vol[vi] = a.overwrite ? t : vol[vi] + t;
                }
            }
        }
    }
    return vmx;
}

// Bilinear sample of texels (iu, iv), (iu + 1, iv), (iu, iv + 1), (iu + 1, iv + 1).
// Tilted: weighted terms alone and no difference, so that an infinite texel (a
// pixel without a count) beside a finite one gives infinity, not NaN.
template <bool TILT>
__device__ __forceinline__ float blend(float fu, float fv, float r00, float r01, float r10, float r11) {
    const float gu = 1.0f - fu;
    const float top = fmaf(fu, r01, gu * r00), bot = fmaf(fu, r11, gu * r10);
    return TILT ? fmaf(fv, bot, (1.0f - fv) * top) : fmaf(fv, bot - top, top);
}

// One voxel tile o of a backprojection launch; step selects the view list
// views + step*n_views (a solver's subset step).  stage: the block's LDS.
// Returns the lane's max |updated voxel| (MLEM / ART kinds).
//
// Untilted views: u, hence (iu, fu), is constant along a column, the bilinear
// weights factor into (1-fu, fu) x (1-fv, fv), and t = v - 0.5 is affine in z.
// The acceptance window 0.55 < u, v < U, V - 0.55 becomes 0.05 < t < hi (hi < 0
// rejects the column).  A column whose whole z extent is accepted (t at the
// tile's first and last z bounds every lane's t: fmaf is monotone in z) runs
// without tests and counts once for all its voxels.
// Tilted views: (u, v) per voxel by col_forms and voxel_uv; a tile that lies
// inside the window (FOOT_INSIDE) runs without tests.
// XTT: per channel w_k = g2s_k - q_k^2/|d|^2 with q_k = dz sig_k S_k,z + ca_k
// (ir.cu:1832-1840), ca_k = sig_k (d_x S_k,x + d_y S_k,y) among the column
// terms; sig_k S_k,z and g2s_k are scalar loads of the plan's weight table.
// Channels k >= K have zero constants (table padding) and are never stored.
template <class C, bool TILT>
__device__ __forceinline__ float backward_item(const BwdArgs& a, int o, int step, float* stage) {
    constexpr int KIND = C::KIND, NC = C::NC, ZPL = C::ZPL, KM = C::KM, VB = C::VB, SB = C::SB, TW = C::TW;
    constexpr bool XTT = C::XTT;
    constexpr int xws = kXwStride;  // >= KM: whole rows, zero padded
    const Dims& d = a.d;
    const auto views = to_global(a.views + (int64_t)step * a.n_views);
    const auto vg = to_global(a.vg);
    const auto vgc = to_const(a.vg);
    const int gx = a.gx;
    const int bcx = C::CX * gx, bcy = C::CY * a.gy;  // block columns along x, y
    const int tx = o % a.tiles_x, ty = (o / a.tiles_x) % a.tiles_y, tz = o / (a.tiles_x * a.tiles_y);
    // the wave index as a wave-uniform value: the column tests and counts below stay scalar
    const int lane = threadIdx.x & 63, wave = uniformi(threadIdx.x >> 6);
    const int xb = tx * bcx + (wave % gx) * C::CX, yb = ty * bcy + (wave / gx) * C::CY;
    const int z0 = tz * 64 * ZPL;
    const int z_last = min(z0 + 64 * ZPL, d.N) - 1;  // the tile's last z
    const float bx0 = (float)(tx * bcx) - d.xc, bx1 = (float)min(tx * bcx + bcx - 1, d.N - 1) - d.xc;
    const float by0 = (float)(ty * bcy) - d.xc, by1 = (float)min(ty * bcy + bcy - 1, d.N - 1) - d.xc;
    const float bz0 = (float)z0 - d.xc, bz1 = (float)z_last - d.xc;
    const int nv = a.n_views;
    if (nv == 0) return 0.f;
    const int64_t img_len = (int64_t)d.V * d.U;

    float tmp[NC][ZPL][KM], fac[NC][ZPL][KM];
#pragma unroll
    for (int c = 0; c < NC; c++)
#pragma unroll
        for (int q = 0; q < ZPL; q++)
#pragma unroll
            for (int k = 0; k < KM; k++) {
                tmp[c][q][k] = 0.f;
                fac[c][q][k] = 0.f;
            }
    int nwhole[NC];  // views accepting a column's whole z extent (added to the counts at the end)
#pragma unroll
    for (int c = 0; c < NC; c++) nwhole[c] = 0;
    // lanes past the volume's end repeat its last voxel (never stored), so that
    // they neither leave the footprint nor fail a column's whole-extent test
    float zpq[ZPL];
#pragma unroll
    for (int q = 0; q < ZPL; q++) zpq[q] = (float)min(z0 + lane + 64 * q, z_last) - d.xc;

    lds_float* const lds = (lds_float*)stage;
    lds_int* const foot = (lds_int*)(stage + 2 * VB * SB);
    lds_float* const term = (lds_float*)(stage + 2 * VB * SB + kBwdFootArea + wave * C::term_area);

    // footprints of views b0 .. b0+15 into buffer buf: lane = 4 x view + corner
    // pair (x, y corner; both z corners), extremes over the 4 lanes of a view
    // (the projective map's extremes over a box are at its corners while den > 0 there)
    auto foot_batch = [&](int b0, int buf) XR_INLINE {
        const int j = lane >> 2, c = lane & 3;
        const int code = views[min(b0 + j, nv - 1)];
        const ViewGeom g = vg[code];
        const ColForms cf = col_forms(g, (c & 1) ? bx1 : bx0, (c & 2) ? by1 : by0);
        float umn = 0.f, umx = 0.f, vmn = 0.f, vmx = 0.f;
        int bad = 0;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            const float czp = k ? bz1 : bz0;
            const float cd = fmaf(g.ad[2], czp, cf.nd);
            float cu, cv;
            voxel_uv(g, cf, czp, d, cu, cv);
            umn = k ? fminf(umn, cu) : cu;
            umx = k ? fmaxf(umx, cu) : cu;
            vmn = k ? fminf(vmn, cv) : cv;
            vmx = k ? fmaxf(vmx, cv) : cv;
            bad |= (!(cd > 0.f) || !(fabsf(cu) < 1e7f) || !(fabsf(cv) < 1e7f)) ? 1 : 0;
        }
        for (int off = 1; off < 4; off <<= 1) {
            umn = fminf(umn, __shfl_xor(umn, off));
            umx = fmaxf(umx, __shfl_xor(umx, off));
            vmn = fminf(vmn, __shfl_xor(vmn, off));
            vmx = fmaxf(vmx, __shfl_xor(vmx, off));
            bad |= __shfl_xor(bad, off);
        }
        const Foot f = foot_from_extent<C>(umn, umx, vmn, vmx, bad, d);
        if (c == 0) {
            lds_int* p = foot + (buf * kBwdBatch + j) * kFootWords;
            p[0] = f.iu_lo;
            p[1] = f.iv_lo;
            p[2] = f.W;
            p[3] = f.Ws | (f.R << 16);
            p[4] = f.flags;
            p[5] = code;
            const bool staged = (f.flags & FOOT_STAGED) != 0;
            const int64_t first = (int64_t)f.iv_lo * d.U + f.iu_lo;
            const uint64_t at = (uint64_t)(uintptr_t)(a.proj + (int64_t)(code - a.code_base) * img_len + first);
            p[8] = (int)(unsigned)at;
            p[9] = (int)(unsigned)(at >> 32);
            p[10] = staged ? (int)((img_len - first) * 4) : 0;
            p[11] = staged ? f.H : 0;
        }
    };
    auto foot_of = [&](int v) XR_INLINE { return foot + (((v / kBwdBatch) & 1) * kBwdBatch + (v & (kBwdBatch - 1))) * kFootWords; };
    auto load_src = [&](int v) XR_INLINE {
        const lds_int* p = foot_of(v);
        FootSrc f;
        f.lo = (unsigned)uniformi(p[8]);
        f.hi = (unsigned)uniformi(p[9]);
        f.range = (unsigned)uniformi(p[10]);
        f.H = uniformi(p[11]);
        f.W = f.Ws = f.R = 0;
        if (C::WF == 0) {
            const int w = uniformi(p[3]);
            // a footprint that is not staged may have no width: of one, every thread's row is R = 0 or more
            // or H = 0 ends the passes (tests of either in the store cost 3 %)
            f.W = max(uniformi(p[2]), 1);
            f.Ws = w & 0xffff;
            f.R = w >> 16;
        }
        return f;
    };
    unsigned long long wholes = 0;
    // column terms of views b0 .. b0+15 for this wave's columns: lane = 4 x view
    // + column (plain) or channel quarter (XTT).  A column past the volume repeats
    // the last one (its sums are never stored): the tile's box, hence its footprint
    // and FOOT_INSIDE, ends at N - 1, and so must everything a column reads.
    auto term_batch = [&](int b0) XR_INLINE {
        const int j = lane >> 2, p = lane & 3;
        const lds_int* fp = foot_of(b0 + j);
        const int code = fp[5];
        const ViewGeom g = vg[code];
        const int iu_lo = fp[0], iv_lo = fp[1], W = fp[2], Ws = fp[3] & 0xffff, fl = fp[4];
        const int cidx = XTT ? 0 : (p & (NC - 1));
        const float xp = (float)min(xb + cidx % C::CX, d.N - 1) - d.xc;
        const float yp = (float)min(yb + cidx / C::CX, d.N - 1) - d.xc;
        const ColForms c = col_forms(g, xp, yp);
        lds_float* tp = term + (j * NC + cidx) * TW;
        lds_int* ti = (lds_int*)tp;
        float wcol = 0.f;
        if (KIND == BWD_FDK) {
            // vol += Ud^2 * (2 pi/P) * sum c p, Ud = sod/(sod + y_unrotated) (fdk.cu:160-169)
            const float Xy = fmaf(d.vs, yp, g.fy);
            const float Ud = d.sod / (d.sod + Xy);
            wcol = Ud * Ud * d.cfdk;
        }
        if (XTT) {
            const float dx = fmaf(d.vs, xp, g.d0[0]);
            const float dy = fmaf(d.vs, yp, g.d0[1]);
            wcol = fmaf(dy, dy, dx * dx);
        }
        bool whole = false;
        if (XTT ? p == 0 : p < NC) {
            tp[7] = wcol;
            if (TILT) {
                tp[0] = c.nu;
                tp[1] = c.nv;
                tp[2] = c.nd;
                tp[4] = g.au[2];
                tp[5] = g.av[2];
                tp[6] = g.ad[2];
                whole = (fl & FOOT_INSIDE) != 0;
            } else {
                const float inv_c = rcpf(c.nd);
                const float u_c = fmaf(c.nu, inv_c, d.hu);
                int iu;
                float fu;
                split(u_c, iu, fu);
                const float Bc = g.av[2] * inv_c;
                const float Ac = fmaf(c.nv, inv_c, d.hv - 0.5f);
                const float hi = (accept_u(u_c, d) && !(fl & FOOT_EMPTY)) ? d.vmax - 0.5f : -1.0f;
                const int lu = min(max(iu - iu_lo, 0), W - 2);
                const float ta = fmaf(Bc, bz0, Ac), tb = fmaf(Bc, bz1, Ac);
                whole = (fl & FOOT_STAGED) && fminf(ta, tb) > 0.05f && fmaxf(ta, tb) < hi;
                tp[0] = Bc;
                tp[1] = Ac;
                tp[2] = fu;
                ti[3] = (lu - iv_lo * Ws) * 4;  // LDS byte offset of texel (iu, 0) in a staging buffer
                tp[4] = hi;
                ti[5] = lu;
                ti[6] = iu;
            }
        }
        // bit 4 j + c: column c's whole extent is accepted in view b0 + j
        wholes = __ballot(whole);
        if (KIND != BWD_FDK && !XTT) {
            const unsigned long long seen = nv - b0 >= kBwdBatch ? ~0ull : (1ull << (4 * (nv - b0))) - 1;
#pragma unroll
            for (int c = 0; c < NC; c++) nwhole[c] += __popcll(wholes & seen & (0x1111111111111111ull << c));
        }
        if constexpr (XTT) {
            const auto row = to_global(a.xw + (int64_t)code * 5 * xws);
#pragma unroll
            for (int m = 0; m < C::KP / 4; m++) {
                const int k = p + 4 * m;
                tp[8 + k] = fmaf(xp, row[2 * xws + k], fmaf(yp, row[3 * xws + k], row[4 * xws + k]));  // 0 for k >= K
            }
        }
    };
    // a wave's own LDS writes, then its lanes read each other's words
    auto wave_sync = [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };

    // staging: view v in buffer v % (2 VB); fetched into registers a group
    // ahead, stored into a buffer whose last reads (view v - 2 VB) a barrier has
    // followed, read after the barrier that ends the group
    typename std::conditional<(C::WF > 0), FootStage<C>, FootStageAny<C>>::type st[C::LOOK];
#pragma unroll
    for (int i = 0; i < C::LOOK; i++) st[i].init(d.U);
    FootSrc kept[C::LOOK];  // fetched and not yet stored
    auto fetch = [&](int v, int i) XR_INLINE {
        kept[i] = load_src(v);
        st[i].fetch(kept[i], d.U);
    };
    auto store = [&](int v, int i) XR_INLINE { st[i].store(lds + (v & (2 * VB - 1)) * SB, kept[i]); };

    // Accumulation of the samples nb of column cidx (view s).  all: every voxel
    // accepted (and counted with the column); otherwise an accepted voxel counts `one`.
    auto accumulate = [&](int s, int cidx, const lds_float* tp, const float (&nb)[ZPL], const bool (&ok)[ZPL],
                          auto all_c, float one) XR_INLINE {
        constexpr bool all = decltype(all_c)::value;
        if constexpr (!XTT) {
#pragma unroll
            for (int q = 0; q < ZPL; q++) {
                if (KIND == BWD_FDK) {
                    tmp[cidx][q][0] = fmaf(tp[7], nb[q], tmp[cidx][q][0]);
                } else {
                    tmp[cidx][q][0] += nb[q];
                    if (!all) fac[cidx][q][0] += ok[q] ? one : 0.0f;
                }
            }
        } else {
            const int code = uniformi(foot_of(s)[5]);
            const float cxy = tp[7], d0z = vgc[code].d0[2];
            if (TILT && a.coef) {
                // backwardOrth: the basis rotated per voxel (of the column the terms are of)
                const ViewGeom& g = a.vg[code];
                const int x = min(xb, d.N - 1), y = min(yb, d.N - 1);
                const float dx = fmaf(d.vs, (float)x - d.xc, g.d0[0]), dy = fmaf(d.vs, (float)y - d.xc, g.d0[1]);
#pragma unroll
                for (int q = 0; q < ZPL; q++) {
                    if (!all && !ok[q]) continue;
                    const float dz = fmaf(d.vs, zpq[q], d0z);
                    const float id2 = rcpf(fmaf(dz, dz, cxy));
                    const int64_t vi = ((int64_t)y * d.N + x) * d.N + (int)(zpq[q] + d.xc);
                    float R[9];
                    orth_rotation(a.coef[vi], a.coef[vi + a.chan_stride], R);
#pragma unroll
                    for (int k = 0; k < KM; k++)
                        if (k < d.K) {
                            const float w = orth_weight(R, a.b, k, dx, dy, dz, id2, g);
                            tmp[cidx][q][k] = fmaf(w, nb[q], tmp[cidx][q][k]);
                            fac[cidx][q][k] += w;
                        }
                }
                return;
            }
            const auto row = to_const(a.xw + (int64_t)code * 5 * xws);
            float ca[KM], sz[KM], g2s[KM];
#pragma unroll
            for (int k = 0; k < KM; k++) {
                ca[k] = tp[8 + k];
                sz[k] = row[k];
                g2s[k] = row[xws + k];
            }
#pragma unroll
            for (int q = 0; q < ZPL; q++) {
                if (!all && !ok[q]) continue;
                const float dz = fmaf(d.vs, zpq[q], d0z);
                const float id2 = rcpf(fmaf(dz, dz, cxy));
#pragma unroll
                for (int k = 0; k < KM; k++) {
                    const float qk = fmaf(dz, sz[k], ca[k]);
                    float w = fmaf(-qk * qk, id2, g2s[k]);
                    if (TILT) w = fmaxf(w, 0.f);  // see xtt_value
                    tmp[cidx][q][k] = fmaf(w, nb[q], tmp[cidx][q][k]);
                    fac[cidx][q][k] += w;
                }
            }
        }
    };

    // A column whose whole extent is accepted: all reads first (LDS latency),
    // then the sums.
    auto whole_column = [&](int s, int cidx) XR_INLINE {
        const lds_float* tp = term + ((s & (kBwdBatch - 1)) * NC + cidx) * TW;
        const lds_int* ti = (const lds_int*)tp;
        const unsigned cur = (unsigned)(uintptr_t)(lds + (s & (2 * VB - 1)) * SB);
        const lds_int* const fp = foot_of(s);
        const unsigned ws4 = C::WF ? (unsigned)(C::WF + 1) * 4u : (unsigned)(fp[3] & 0xffff) * 4u;
        float nb[ZPL];
        bool ok[ZPL];
        float fu[ZPL], fv[ZPL], r[ZPL][4];
        unsigned base;
        if (TILT)
            base = cur - __umul24((unsigned)fp[1], ws4) - (unsigned)fp[0] * 4u;
        else
            base = cur + (unsigned)ti[3];
#pragma unroll
        for (int q = 0; q < ZPL; q++) {
            float t;
            unsigned at = base;
            if (TILT) {
                // voxel_uv's arithmetic, with the column's half of the forms in the terms
                const float inv = rcpf(fmaf(tp[6], zpq[q], tp[2]));
                const float tu = fmaf(fmaf(tp[4], zpq[q], tp[0]), inv, d.hu) - 0.5f;
                t = fmaf(fmaf(tp[5], zpq[q], tp[1]), inv, d.hv) - 0.5f;
                fu[q] = __builtin_amdgcn_fractf(tu);
                at += (unsigned)floor_int(tu) * 4u;
            } else {
                t = fmaf(tp[0], zpq[q], tp[1]);
                fu[q] = tp[2];
            }
            fv[q] = __builtin_amdgcn_fractf(t);
            at = __umul24((unsigned)floor_int(t), ws4) + at;
            const lds_float* p0 = (const lds_float*)(uintptr_t)at;
            const lds_float* p1 = C::WF ? p0 + (C::WF + 1) : (const lds_float*)(uintptr_t)(at + ws4);
            r[q][0] = p0[0];
            r[q][1] = p0[1];
            r[q][2] = p1[0];
            r[q][3] = p1[1];
        }
#pragma unroll
        for (int q = 0; q < ZPL; q++) {
            nb[q] = blend<TILT>(fu[q], fv[q], r[q][0], r[q][1], r[q][2], r[q][3]);
            ok[q] = true;
        }
        accumulate(s, cidx, tp, nb, ok, std::true_type(), 0.0f);
    };

    // Any column: a window test per voxel; a rejected voxel reads an in-bounds
    // texel and adds zero.  counted: the view is in the column's count already.
    auto tested_column = [&](int s, int cidx, bool counted) XR_INLINE {
        const lds_float* tp = term + ((s & (kBwdBatch - 1)) * NC + cidx) * TW;
        const lds_int* ti = (const lds_int*)tp;
        const lds_float* cur = lds + (s & (2 * VB - 1)) * SB;
        const lds_int* const fp = foot_of(s);
        const int fl = uniformi(fp[4]);
        const float hi = TILT ? 0.f : tp[4];
        if (TILT ? xb + cidx % C::CX >= d.N || yb + cidx / C::CX >= d.N : uniformf(hi) < 0.f) return;
        const int iu_lo = fp[0], iv_lo = fp[1], W = fp[2], Ws = C::WF ? C::WF + 1 : fp[3] & 0xffff;
        const bool staged = (fl & FOOT_STAGED) != 0;
        const auto img = to_global(a.proj + (int64_t)(uniformi(fp[5]) - a.code_base) * img_len);
        float nb[ZPL];
        bool ok[ZPL];
#pragma unroll
        for (int q = 0; q < ZPL; q++) {
            float tv, fu;
            int iu, lu;
            if (TILT) {
                const float inv = rcpf(fmaf(tp[6], zpq[q], tp[2]));
                const float u = fmaf(fmaf(tp[4], zpq[q], tp[0]), inv, d.hu);
                const float v = fmaf(fmaf(tp[5], zpq[q], tp[1]), inv, d.hv);
                ok[q] = accept_u(u, d) && accept_v(v, d);
                split(u, iu, fu);
                lu = min(max(iu - iu_lo, 0), W - 2);
                tv = v - 0.5f;
            } else {
                tv = fmaf(tp[0], zpq[q], tp[1]);
                ok[q] = tv > 0.05f && tv < hi;
                fu = tp[2];
                lu = ti[5];
                iu = ti[6];
            }
            const float fl_v = floorf(tv);
            const float fv = tv - fl_v;
            const int iv = (int)fl_v;
            float r00, r01, r10, r11;
            if (staged) {
                const int qi = (ok[q] ? iv - iv_lo : 0) * Ws + lu;
                r00 = cur[qi];
                r01 = cur[qi + 1];
                r10 = cur[qi + Ws];
                r11 = cur[qi + Ws + 1];
            } else {
                // direct reads: a distinct (nontemporal) load form next to the LDS reads
                // (the gfx950 backend rejects the two merged into one flat access)
                const int64_t qi = (int64_t)min(max(iv, 0), d.V - 2) * d.U + min(max(iu, 0), d.U - 2);
                r00 = __builtin_nontemporal_load(img + qi);
                r01 = __builtin_nontemporal_load(img + qi + 1);
                r10 = __builtin_nontemporal_load(img + qi + d.U);
                r11 = __builtin_nontemporal_load(img + qi + d.U + 1);
            }
            nb[q] = ok[q] ? blend<TILT>(fu, fv, r00, r01, r10, r11) : 0.0f;
        }
        accumulate(s, cidx, tp, nb, ok, std::false_type(), counted ? 0.0f : 1.0f);
    };

    constexpr unsigned kAllCols = (1u << NC) - 1;  // of the four bits of a view in `wholes`
    auto view = [&](int s) XR_INLINE {
        const unsigned w = (unsigned)(wholes >> (4 * (s & (kBwdBatch - 1)))) & kAllCols;
        if (w == kAllCols) {
#pragma unroll
            for (int c = 0; c < NC; c++) {
                whole_column(s, c);
                if (ZPL > 4) __builtin_amdgcn_sched_barrier(0);
            }
        } else if (!(uniformi(foot_of(s)[4]) & FOOT_EMPTY)) {
#pragma unroll
            for (int c = 0; c < NC; c++) {
                tested_column(s, c, (w >> c & 1) != 0);
                // one column at a time: interleaved, their values would not fit the registers
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    if (wave == 0) foot_batch(0, 0);
    __syncthreads();
    term_batch(0);
#pragma unroll
    for (int g = 0; g < VB; g += C::LOOK) {
#pragma unroll
        for (int i = 0; i < C::LOOK; i++)
            if (g + i < nv) fetch(g + i, i);
#pragma unroll
        for (int i = 0; i < C::LOOK; i++)
            if (g + i < nv) store(g + i, i);
    }
    wave_sync();
    __syncthreads();

    for (int s0 = 0; s0 < nv; s0 += VB) {
        const int j = s0 & (kBwdBatch - 1);
        if (j == 0 && s0 > 0) {
            term_batch(s0);
            wave_sync();
        }
        // the footprints of the batch after this one: read from a group later on
        if (wave == 0 && j == kBwdBatch - 2 * VB && s0 + 2 * VB < nv)
            foot_batch(s0 + 2 * VB, ((s0 + 2 * VB) / kBwdBatch) & 1);
        if constexpr (C::LOOK == VB) {
#pragma unroll
            for (int i = 0; i < VB; i++)
                if (s0 + VB + i < nv) fetch(s0 + VB + i, i);
            constexpr unsigned long long kGroup = (NC == 1 ? 0x1111111111111111ull : NC == 2 ? 0x3333333333333333ull : ~0ull) &
                                                  (VB == 16 ? ~0ull : (1ull << (4 * VB % 64)) - 1);
            if (s0 + VB <= nv && (wholes >> (4 * j) & kGroup) == kGroup) {
                // every column whole in every view of the group: no test in sight
#pragma unroll
                for (int i = 0; i < VB; i++)
#pragma unroll
                    for (int c = 0; c < NC; c++) whole_column(s0 + i, c);
            } else {
                for (int s = s0; s < min(s0 + VB, nv); s++) view(s);
            }
#pragma unroll
            for (int i = 0; i < VB; i++)
                if (s0 + VB + i < nv) store(s0 + VB + i, i);
        } else {
            for (int s = s0; s < min(s0 + VB, nv); s++) {
                if (s + VB < nv) fetch(s + VB, 0);
                view(s);
                if (s + VB < nv) store(s + VB, 0);
            }
        }
        __syncthreads();
    }
    return backward_update<C>(a, tmp, fac, nwhole, xb, yb, z0, lane);
}

// at least 4 waves per SIMD (at most 128 VGPRs): two 8-wave blocks, or one
// 16-wave block, per CU
template <class C, bool TILT>
__global__ __launch_bounds__(C::threads) __attribute__((amdgpu_waves_per_eu(4))) void k_backward(const BwdArgs a) {
    extern __shared__ float stage[];
    const int o = (blockIdx.x % 8) * a.per_xcd + blockIdx.x / 8;
    if (o >= a.n_tiles) return;
    float m = backward_item<C, TILT>(a, o, 0, stage);
    if constexpr (C::KIND == BWD_MLEM || C::KIND == BWD_ART) {
        if (a.vmax_out) {
            // the tile's max |updated voxel|: one atomic per block
            lds_float* const wmax = (lds_float*)(stage + C::words);
            for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
            if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
            __syncthreads();
            if (threadIdx.x == 0) {
                float t = 0.f;
                for (int w = 0; w < C::WAVES; w++) t = fmaxf(t, wmax[w]);
                __hip_atomic_fetch_max(a.vmax_out, __float_as_uint(t), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

// Persistent backprojection over many problems: the same work queue as
// k_forward_batch; items[i] is one problem with item_end[i] - item_end[i-1]
// tiles, and its own tile shape.  W: the configuration of the tilted and wide
// items (the same block).
template <class C, class W>
__global__ __launch_bounds__(C::threads) __attribute__((amdgpu_waves_per_eu(4))) void k_backward_batch(
    const BwdArgs* __restrict__ items, const int* __restrict__ item_end, int n_items, unsigned* queue, int step) {
    extern __shared__ float stage[];
    typedef __attribute__((address_space(3))) unsigned lds_uint;
    // past the staging and term areas: the last tile's per-wave max |voxel|, its item, the ticket
    lds_float* const wmax = (lds_float*)(stage + (C::words > W::words ? C::words : W::words));
    lds_int* const witem = (lds_int*)(wmax + C::WAVES);
    lds_uint* const tk = (lds_uint*)(wmax + C::WAVES + 1);
    const int total = item_end[n_items - 1];
    if (threadIdx.x == 0) *witem = -1;
    for (;;) {
        __syncthreads();
        if (threadIdx.x == 0) {
            // the previous tile's max |updated voxel| -> its problem's next-step bound
            const int pi = *witem;
            unsigned* const dst = pi >= 0 ? items[pi].vmax_out : nullptr;
            if (dst) {
                float m = 0.f;
                for (int w = 0; w < C::WAVES; w++) m = fmaxf(m, wmax[w]);
                __hip_atomic_fetch_max(dst, __float_as_uint(m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            *witem = -1;  // flushed: only a tile that sets it again sends a max
            *tk = take_ticket(queue, (unsigned)total);
        }
        __syncthreads();
        // uniform across the block: keeps the item's arguments in scalar registers
        const int t = __builtin_amdgcn_readfirstlane((int)*tk);
        if (t >= total) break;
        const int i = find_item(item_end, n_items, t);
        const BwdArgs& a = items[i];
        const int o = t - (i ? item_end[i - 1] : 0);
        float m = !a.axis ? backward_item<W, true>(a, o, step, stage)
                          : (a.wide ? backward_item<W, false>(a, o, step, stage)
                                    : backward_item<C, false>(a, o, step, stage));
        if (a.vmax_out) {
            for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
            if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
            if (threadIdx.x == 0) *witem = i;
        }
    }
}

// max |x| over blocks b, b + nb, ... of 256 threads: 16-byte loads, four in
// flight per thread; scalar loads for an unaligned base and for the tail.
__device__ __forceinline__ float absmax4(const float4 a) {
    return fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w)));
}

__device__ __forceinline__ float absmax_range(const float* __restrict__ x, int64_t n, int64_t b, int64_t nb) {
    float m = 0.f;
    const int64_t n4 = (reinterpret_cast<uintptr_t>(x) & 15) == 0 ? n >> 2 : 0;
    const float4* __restrict__ x4 = reinterpret_cast<const float4*>(x);
    const int64_t stride = nb * 256;
    int64_t i = b * 256 + threadIdx.x;
    for (; i + 3 * stride < n4; i += 4 * stride) {
        const float4 a0 = x4[i], a1 = x4[i + stride], a2 = x4[i + 2 * stride], a3 = x4[i + 3 * stride];
        m = fmaxf(m, fmaxf(fmaxf(absmax4(a0), absmax4(a1)), fmaxf(absmax4(a2), absmax4(a3))));
    }
    for (; i < n4; i += stride) m = fmaxf(m, absmax4(x4[i]));
    for (int64_t j = 4 * n4 + b * 256 + threadIdx.x; j < n; j += stride) m = fmaxf(m, fabsf(x[j]));
    return m;
}

// Maximum over a block of 256 threads, valid in thread 0 (one atomic per
// block: same-address atomics from thousands of waves serialise).
__device__ __forceinline__ float block_max256(float m) {
    __shared__ float part[4];
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off));
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    return fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
}

// Per-segment max |x|: segment i is segs[i][0, seg_len[i]), its maximum goes
// to out[i] (zeroed beforehand; non-negative floats order like their bit
// patterns); grid (blocks per segment, segments).
__global__ __launch_bounds__(256) void k_absmax_seg(const float* const* __restrict__ segs,
                                                    const int64_t* __restrict__ seg_len, float* out) {
    const float m = block_max256(absmax_range(segs[blockIdx.y], seg_len[blockIdx.y], blockIdx.x, gridDim.x));
    if (threadIdx.x == 0) atomicMax((unsigned int*)(out + blockIdx.y), __float_as_uint(m));
}

// ---------------------------------------------------------------------------
// FDK row filter (projConv, fdk.cu:28-43): dst[u] = sum_j h(u - j) w[j] src[j]
// for every row (view, v) of the launch, as one FP32 matrix product on the
// matrix cores: C[row][u] = sum_j A[row][j] T[j][u], A the weighted rows and
// T[j][u] = h(u - j) taken from a tap window in LDS (the Toeplitz operand is
// never stored).  h(m) = taps[|m|] (a linear convolution) or taps[m mod U]
// (circular), zero for |m| >= U.  v_mfma_f32_16x16x4f32 operands: A from lane
// (row lane&15, k lane>>4), B from lane (k lane>>4, column lane&15); the result
// lane holds column lane&15, rows 4*(lane>>4) + r.
// Block: 64 rows x 64 NT columns, four waves of 64 rows x 16 NT columns, K steps
// of 32 samples; the next step's samples are loaded during this step's products
// (rows contiguous over 32 lanes).  The wider the block, the fewer times a row is
// staged: with NT = 8 and U <= 512, once.
// Bound by the FP32 matrix rate.  Measured, 401 x 451 rows of 487: 1662 -> 903 us
// (95 TFLOP/s of 153 without the padding) against 64 x 128 tiles that staged
// eight strided samples per lane between two barriers, four times per row.
// ---------------------------------------------------------------------------
typedef float f32x4_t __attribute__((ext_vector_type(4)));
constexpr int kFiltBM = 64, kFiltBK = 32, kFiltAStride = kFiltBK + 1;

template <int NT>
__global__ __launch_bounds__(256, 2) void k_fdk_filter(const float* __restrict__ src, float* __restrict__ dst,
                                                       const float* __restrict__ weight,
                                                       const float* __restrict__ taps, int U, int V,
                                                       const int32_t* __restrict__ views, int n_rows, int row_base,
                                                       int code_base, int circular) {
    constexpr int BN = 64 * NT, win = BN + kFiltBK - 1;  // win: taps one K step of the block touches
    constexpr int nr = kFiltBM / 8, nh = (win + 255) / 256;
    __shared__ float As[kFiltBM * kFiltAStride];
    __shared__ float Hs[nh * 256];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int row0 = row_base + blockIdx.y * kFiltBM, col0 = blockIdx.x * BN;
    // this thread loads sample sj of rows sr + 8 i of each K step
    const int sj = tid & 31, sr = tid >> 5;
    int64_t roff[nr];
    int woff[nr];
#pragma unroll
    for (int i = 0; i < nr; i++) {
        const int row = min(row0 + sr + 8 * i, n_rows - 1);  // rows past the last are computed and not stored
        const int slot = row / V, v = row - slot * V;
        roff[i] = ((int64_t)(views[slot] - code_base) * V + v) * U;
        woff[i] = v;
    }
    const int wn = wave * (16 * NT);  // the wave's columns
    const int li = lane & 15, lk = lane >> 4;
    f32x4_t acc[4][NT];
#pragma unroll
    for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[mt][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float x[nr], w[nr], h[nh];
    auto fetch = [&](int j0) XR_INLINE {
        const int j = j0 + sj, jj = min(j, U - 1);
#pragma unroll
        for (int i = 0; i < nr; i++) x[i] = src[roff[i] + jj];
        if (weight) {
#pragma unroll
            for (int i = 0; i < nr; i++) w[i] = weight[(int64_t)woff[i] * U + jj];
        }
        // Hs[t] = h(m), m = col0 - j0 - (BK - 1) + t
#pragma unroll
        for (int i = 0; i < nh; i++) {
            const int m = col0 - j0 - (kFiltBK - 1) + tid + 256 * i, am = abs(m);
            const float tap = taps[min(circular && m < 0 ? max(m + U, 0) : am, U - 1)];
            h[i] = am < U ? tap : 0.f;
        }
    };
    fetch(0);
    for (int j0 = 0; j0 < U; j0 += kFiltBK) {
        __syncthreads();  // the previous K step is done with As and Hs
#pragma unroll
        for (int i = 0; i < nr; i++) {
            const float xw = weight ? x[i] * w[i] : x[i];
            As[(sr + 8 * i) * kFiltAStride + sj] = j0 + sj < U ? xw : 0.f;
        }
#pragma unroll
        for (int i = 0; i < nh; i++) Hs[tid + 256 * i] = h[i];
        __syncthreads();
        if (j0 + kFiltBK < U) fetch(j0 + kFiltBK);
#pragma unroll
        for (int kk = 0; kk < kFiltBK; kk += 4) {
            float a[4], b[NT];
#pragma unroll
            for (int mt = 0; mt < 4; mt++) a[mt] = As[(mt * 16 + li) * kFiltAStride + kk + lk];
#pragma unroll
            for (int nt = 0; nt < NT; nt++) b[nt] = Hs[wn + nt * 16 + li - kk - lk + (kFiltBK - 1)];
#pragma unroll
            for (int mt = 0; mt < 4; mt++)
#pragma unroll
                for (int nt = 0; nt < NT; nt++)
                    acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[mt], b[nt], acc[mt][nt], 0, 0, 0);
        }
    }
#pragma unroll
    for (int mt = 0; mt < 4; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int row = row0 + mt * 16 + 4 * lk + r;
            if (row >= n_rows) continue;
            const int slot = row / V, v = row - slot * V;
            const int64_t off = ((int64_t)(views[slot] - code_base) * V + v) * U;
#pragma unroll
            for (int nt = 0; nt < NT; nt++) {
                const int col = col0 + wn + nt * 16 + li;
                if (col < U) dst[off + col] = acc[mt][nt][r];
            }
        }
}

// calcWeight (fdk.cu:13-26).
__global__ void k_fdk_weight(float* w, int U, int V, float sdd, float det) {
    const int u = blockIdx.x * blockDim.x + threadIdx.x, v = blockIdx.y;
    if (u >= U) return;
    const float ur = ((float)u + 0.5f - (float)U / 2.0f) * det;
    const float vr = ((float)v + 0.5f - (float)V / 2.0f) * det;
    w[(int64_t)v * U + u] = sdd / sqrtf(sdd * sdd + ur * ur + vr * vr);
}

// Reference layout (x + N*y + N^2*z) <-> column layout (z + N*(x + N*y)):
// per y it is a transpose of the (z, x) plane; 32x32 tiles through LDS.
template <bool TO_INTERNAL>
__global__ __launch_bounds__(256) void k_transpose(const float* __restrict__ in, float* __restrict__ out, int N) {
    __shared__ float t[32][33];
    const int64_t N2 = (int64_t)N * N, N3 = N2 * N;
    const int y = blockIdx.z % N, ch = blockIdx.z / N;
    const float* src = in + ch * N3;
    float* dst = out + ch * N3;
    const int a0 = blockIdx.x * 32, b0 = blockIdx.y * 32;  // TO_INTERNAL: a = x, b = z
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int a = a0 + threadIdx.x, b = b0 + r;
        if (a < N && b < N) {
            // TO_INTERNAL: read ref[x=a, y, z=b]; else read internal[z=a, x=b, y]
            t[r][threadIdx.x] = TO_INTERNAL ? src[a + (int64_t)N * y + N2 * b] : src[a + (int64_t)N * b + N2 * y];
        }
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int b = b0 + threadIdx.x, a = a0 + r;
        if (a < N && b < N) {
            if (TO_INTERNAL)
                dst[b + (int64_t)N * a + N2 * y] = t[threadIdx.x][r];  // internal[z=b, x=a, y]
            else
                dst[b + (int64_t)N * y + N2 * a] = t[threadIdx.x][r];  // ref[x=b, y, z=a]
        }
    }
}

// Copies of a column-layout volume with another axis contiguous, for the lanes
// of tilted forward projections (see splat_tilted): LA = 1 gives y + N x + N^2 z,
// LA = 0 gives x + N y + N^2 z.  32x32 tiles of the (z, lane axis) plane
// through LDS, one plane per index of the third axis.
template <int LA>
__global__ __launch_bounds__(256) void k_lane_copy(const float* __restrict__ in, float* __restrict__ out, int N) {
    __shared__ float t[32][33];
    const int64_t N2 = (int64_t)N * N, N3 = N2 * N;
    const int third = blockIdx.z % N, ch = blockIdx.z / N;
    const int64_t in_lane = LA == 1 ? N2 : N, in_third = LA == 1 ? N : N2;
    const float* src = in + ch * N3 + third * in_third;
    float* dst = out + ch * N3 + (int64_t)third * N;
    const int z0 = blockIdx.x * 32, l0 = blockIdx.y * 32;
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int z = z0 + threadIdx.x, l = l0 + r;
        if (z < N && l < N) t[r][threadIdx.x] = src[z + l * in_lane];
    }
    __syncthreads();
    for (int r = threadIdx.y; r < 32; r += 8) {
        const int l = l0 + threadIdx.x, z = z0 + r;
        if (z < N && l < N) dst[l + z * N2] = t[threadIdx.x][r];
    }
}

// ---- orientation helpers of the orientation-aware XTT loop ------------------
// Per voxel, channels nvox apart.  Normal of the three-direction scattering
// (ir.cu:912-922): (mu0 S0 - m1 S1) x (mu0 S0 - m2 S2), normalised (zero if
// its length is at most 1e-8, vec.h:94-104).
__device__ __forceinline__ void three_direc_normal(const Basis& b, float mu0, float m1, float m2, float n[3]) {
    float v1[3], v2[3];
#pragma unroll
    for (int i = 0; i < 3; i++) {
        v1[i] = mu0 * b.S[0][i] - m1 * b.S[1][i];
        v2[i] = mu0 * b.S[0][i] - m2 * b.S[2][i];
    }
    n[0] = v1[1] * v2[2] - v1[2] * v2[1];
    n[1] = v1[2] * v2[0] - v1[0] * v2[2];
    n[2] = v1[0] * v2[1] - v1[1] * v2[0];
    const float len = sqrtf(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
#pragma unroll
    for (int i = 0; i < 3; i++) n[i] = len > 1e-8f ? n[i] / len : 0.f;
}

// calcNormalVectorThreeDirec (ir.cu:856-974; rot picks the signs of mu1, mu2)
// and calcNormalVectorThreeDirecWithEst (ir.cu:976-1071; the signs from est
// channel 1).  The normal is rotated by the voxel's current rotation, flipped
// into z >= 0 and normalised; loss = |R e_z x n|; coef <- (atan2(n_x, -n_y),
// n_z), the rotation that carries e_z onto n.
__global__ __launch_bounds__(256) void k_orth_normal(const float* __restrict__ vol, float* __restrict__ coef,
                                                     float* __restrict__ loss, int64_t n, int rot,
                                                     const float* __restrict__ est, Basis b) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float R[9];
    orth_rotation(coef[i], coef[i + n], R);
    const float mu0 = vol[i], mu1 = vol[i + n], mu2 = vol[i + 2 * n];
    int r = rot;
    if (est) {
        const float e = est[i + n];
        r = e < 0.5f ? 0 : (e < 1.5f ? 1 : (e < 2.5f ? 2 : 3));
    }
    const float m1 = (r == 1 || r == 2) ? -mu1 : mu1;
    const float m2 = (r == 2 || r == 3) ? -mu2 : mu2;
    float n0[3], nr[3];
    three_direc_normal(b, mu0, m1, m2, n0);
#pragma unroll
    for (int k = 0; k < 3; k++) nr[k] = R[3 * k] * n0[0] + R[3 * k + 1] * n0[1] + R[3 * k + 2] * n0[2];
    if (nr[2] < 0.f) {
        nr[0] = -nr[0];
        nr[1] = -nr[1];
        nr[2] = -nr[2];
    }
    const float len = sqrtf(nr[0] * nr[0] + nr[1] * nr[1] + nr[2] * nr[2]);
#pragma unroll
    for (int k = 0; k < 3; k++) nr[k] = len > 1e-8f ? nr[k] / len : 0.f;
    // (R e_z) x n
    const float dx = R[5] * nr[2] - R[8] * nr[1], dy = R[8] * nr[0] - R[2] * nr[2], dz = R[2] * nr[1] - R[5] * nr[0];
    loss[i] = sqrtf(dx * dx + dy * dy + dz * dz);
    coef[i] = atan2f(nr[0], -nr[1]);  // e_z x n = (-n_y, n_x, 0)
    coef[i + n] = nr[2];
}

// updateEstimationByCoef (ir.cu:1073-1118).
__global__ __launch_bounds__(256) void k_orth_update_est(const float* __restrict__ vol, float* __restrict__ est,
                                                         int64_t n, int iter, Basis b) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float nr[3];
    three_direc_normal(b, vol[i], vol[i + n], vol[i + 2 * n], nr);
    if (nr[2] < 0.f) {
        nr[0] = -nr[0];
        nr[1] = -nr[1];
        nr[2] = -nr[2];
    }
    const float len = sqrtf(nr[0] * nr[0] + nr[1] * nr[1] + nr[2] * nr[2]);
    const float c = len > 1e-8f ? nr[2] / len : 0.f;
    if (c > est[i]) {
        est[i] = c;
        est[i + n] = (float)iter;
    }
}

// convertNormVector (ir.cu:1448-1480): md = mean(mu) R e_z.
__global__ __launch_bounds__(256) void k_orth_md(const float* __restrict__ vol, const float* __restrict__ coef,
                                                 float* __restrict__ md, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const float mu = (vol[i] + vol[i + n] + vol[i + 2 * n]) / 3.0f;
    float R[9];
    orth_rotation(coef[i], coef[i + n], R);
    md[i] = mu * R[2];
    md[i + n] = mu * R[5];
    md[i + 2 * n] = mu * R[8];
}

// meanFiltFiber (ir.cu:1231-1303) on a column-layout volume of edge N: the
// 27 neighbours' mu-weighted orientation vectors (sin t cos(phi - pi/2),
// sin t sin(phi - pi/2), cos t), those with |dot| > 0.5 against the centre
// added with weight w (sign aligned), normalised, flipped into z >= 0, stored
// as (atan2, cos).  Boundary voxels copy the source.
__global__ __launch_bounds__(256) void k_orth_mean_filter(const float* __restrict__ src, const float* __restrict__ vol,
                                                          int N, float w, float* __restrict__ dst) {
    const int64_t n = (int64_t)N * N * N;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int z = (int)(i % N), x = (int)((i / N) % N), y = (int)(i / ((int64_t)N * N));
    if (x < 1 || y < 1 || z < 1 || x > N - 2 || y > N - 2 || z > N - 2) {
        dst[i] = src[i];
        dst[i + n] = src[i + n];
        return;
    }
    auto vec = [&](int di, int dj, int dk, float v[3]) {
        const int64_t q = ((int64_t)(y - dj) * N + (x - di)) * N + (z - dk);
        const float ct = src[q + n];
        const float st = sqrtf(1.0f - ct * ct);
        float sp, cp;
        sincosf(-(float)M_PI / 2.0f + src[q], &sp, &cp);
        const float mu = vol[q] + vol[q + n] + vol[q + 2 * n];
        v[0] = mu * (st * cp);
        v[1] = mu * (st * sp);
        v[2] = mu * ct;
    };
    float c[3], m[3];
    vec(0, 0, 0, m);
    c[0] = m[0];
    c[1] = m[1];
    c[2] = m[2];
    // the reference's order: neighbour cnt and 26 - cnt for cnt = 0 .. 12
    for (int cnt = 0; cnt < 13; cnt++) {
#pragma unroll
        for (int side = 0; side < 2; side++) {
            const int q = side ? 26 - cnt : cnt;
            float o[3];
            vec(q / 9 - 1, (q / 3) % 3 - 1, q % 3 - 1, o);
            const float d = o[0] * m[0] + o[1] * m[1] + o[2] * m[2];
            const float sgn = d > 0.5f ? 1.f : (d < -0.5f ? -1.f : 0.f);
            if (sgn != 0.f) {
                c[0] += sgn * w * o[0];
                c[1] += sgn * w * o[1];
                c[2] += sgn * w * o[2];
            }
        }
    }
    const float len = sqrtf(c[0] * c[0] + c[1] * c[1] + c[2] * c[2]);
#pragma unroll
    for (int k = 0; k < 3; k++) c[k] = len > 1e-8f ? c[k] / len : 0.f;
    if (c[2] < 0.f) {
        c[0] = -c[0];
        c[1] = -c[1];
        c[2] = -c[2];
    }
    dst[i] = atan2f(c[0], -c[1]);
    dst[i + n] = c[2];
}

// Mean over f x f x f blocks of a column-layout volume of edge N = Nc * f
// (one thread per coarse voxel, z fastest: a wave reads 64 f consecutive
// floats of each fine column it visits).
__global__ __launch_bounds__(256) void k_vol_down(const float* __restrict__ fine, float* __restrict__ coarse, int Nc,
                                                  int f) {
    const int64_t n = (int64_t)Nc * Nc * Nc;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const int zc = (int)(i % Nc), xc = (int)((i / Nc) % Nc), yc = (int)(i / ((int64_t)Nc * Nc));
    const int64_t N = (int64_t)Nc * f;
    float s = 0.f;
    for (int dy = 0; dy < f; dy++)
        for (int dx = 0; dx < f; dx++) {
            const float* col = fine + ((int64_t)(yc * f + dy) * N + (xc * f + dx)) * N + (int64_t)zc * f;
            for (int dz = 0; dz < f; dz++) s += col[dz];
        }
    coarse[i] = s / (float)(f * f * f);
}

// fine = max(fine + up(a - b), lo): the difference of two coarse column-layout
// volumes of edge Nc, interpolated trilinearly onto the fine grid of edge
// Nc * f (fine index i sits at coarse coordinate (i + 0.5) / f - 0.5, clamped
// to the coarse grid), added to the fine volume and floored at lo.
__global__ __launch_bounds__(256) void k_vol_up_add(const float* __restrict__ a, const float* __restrict__ b, int Nc,
                                                    int f, float* __restrict__ fine, float lo) {
    const int64_t N = (int64_t)Nc * f;
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= N * N * N) return;
    const int z = (int)(i % N), x = (int)((i / N) % N), y = (int)(i / (N * N));
    auto axis = [&](int j, int& j0, int& j1, float& w) {
        const float c = fmaxf(((float)j + 0.5f) / (float)f - 0.5f, 0.f);
        j0 = min((int)c, Nc - 1);
        j1 = min(j0 + 1, Nc - 1);
        w = c - (float)j0;
        if (j0 == Nc - 1) w = 0.f;
    };
    int z0, z1, x0, x1, y0, y1;
    float wz, wx, wy;
    axis(z, z0, z1, wz);
    axis(x, x0, x1, wx);
    axis(y, y0, y1, wy);
    auto at = [&](int yy, int xx, int zz) {
        const int64_t k = ((int64_t)yy * Nc + xx) * Nc + zz;
        return a[k] - b[k];
    };
    auto lerp = [](float u, float v, float w) { return fmaf(w, v - u, u); };
    const float c00 = lerp(at(y0, x0, z0), at(y0, x0, z1), wz), c01 = lerp(at(y0, x1, z0), at(y0, x1, z1), wz);
    const float c10 = lerp(at(y1, x0, z0), at(y1, x0, z1), wz), c11 = lerp(at(y1, x1, z0), at(y1, x1, z1), wz);
    const float d = lerp(lerp(c00, c01, wx), lerp(c10, c11, wx), wy);
    fine[i] = fmaxf(fine[i] + d, lo);
}

__global__ void k_sqrt_abs(float* v, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float m = v[i];
    v[i] = (m < 0.0f) ? sqrtf(-m) : sqrtf(m);  // voxelSqrt (ir.cu:1715)
}

// calcAngleFromMD (pca.cu:67-83): azimuth phi and polar angle theta of the
// main direction, the direction flipped into y >= 0 first.  The squares and the
// sums are rounded separately (no contraction into FMAs), as the reference's
// host code evaluates them.
__global__ __launch_bounds__(256) void k_md_angles(const float* __restrict__ md, float* __restrict__ ang,
                                                   int64_t n) {
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float a = md[i], b = md[n + i], c = md[2 * n + i];
    const float r = sqrtf(b * b + a * a);
    if (b < 0.f) {
        ang[i] = atan2f(-b, -a);
        ang[n + i] = atan2f(r, -c);
    } else {
        ang[i] = atan2f(b, a);
        ang[n + i] = atan2f(r, c);
    }
}

// directionNormalization (pca.cu:85-106): unit main direction where its norm
// exceeds eps (0.65 in the reference), zero elsewhere.
__global__ __launch_bounds__(256) void k_md_normalise(float* __restrict__ md, int64_t n, float eps) {
#pragma clang fp contract(off)
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float x = md[i], y = md[n + i], z = md[2 * n + i];
    const float nrm = sqrtf(x * x + y * y + z * z);
    const bool keep = nrm > eps;
    md[i] = keep ? x / nrm : 0.f;
    md[n + i] = keep ? y / nrm : 0.f;
    md[2 * n + i] = keep ? z / nrm : 0.f;
}

// max |x| over n floats into out[0] (zeroed beforehand).
__global__ __launch_bounds__(256) void k_absmax(const float* __restrict__ x, int64_t n, float* out) {
    const float m = block_max256(absmax_range(x, n, blockIdx.x, gridDim.x));
    if (threadIdx.x == 0) atomicMax((unsigned int*)out, __float_as_uint(m));
}

__global__ void k_fill(float* p, int64_t n, float value) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = value;
}

// value < floor -> replacement (main.cu:35 clamps the sinogram: <0 -> 1e-8).
__global__ void k_clamp_min(float* p, int64_t n, float floor_value, float replacement) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n && p[i] < floor_value) p[i] = replacement;
}

// 1 / sqrt(x), FP64, x > 0 and neither it nor its root denormal: the hardware's
// estimate (relative error 2^-24 or less) and one third-order step.
__device__ __forceinline__ double rsqrt64(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y * e, fma(0.375, e, 0.5), y);
}

// Products S_i S_j of the basis (00 01 02 11 12 22; exact in FP64) and 1 / K.
struct PcaBasis {
    double P[kMaxBasis][6];
    double inv_k;
};

// Per-voxel principal orientation (calcEigenVector, pca.cu:12-65):
// C = (1/K) sum_k (mu_k S_k)(mu_k S_k)^T, eigenvector of the smallest
// eigenvalue, sign so that z >= 0, md = sign * mean(mu) * e_min, eigenvalues
// normalised to sum 1.  Closed-form (trigonometric) eigenvalues in FP64 and the
// eigenvector from cross products of the rows of C - lambda_min I.
//
// With B = (C - q I) / p and r = det(B) / 2, the eigenvalues are q + 2 p cos(phi
// + 2 pi j / 3), phi = acos(r) / 3.  The angle is not formed: for r >= 0 let f =
// phi, else f = pi/3 - phi; t = sin(f / 2) is the root of 3 t - 4 t^3 =
// sin(3 f / 2) = sqrt((1 - |r|) / 2) =: h in [0, 0.259], found from a polynomial
// (relative error 6e-6) with two Newton steps whose derivative is taken in FP32.
// Bound by memory.  Measured at 256^3 x 13 (1.28 GB): 460 -> 231 us, 5.5 TB/s,
// against acos, two cosines and library roots and quotients (FP64 arithmetic
// took the time) and products formed per voxel.
__global__ __launch_bounds__(256) void k_pca(const float* __restrict__ mu, int K, const PcaBasis b, int64_t nvox,
                                             int64_t cs, float* __restrict__ md, float* __restrict__ ev) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nvox) return;
    double a00 = 0, a01 = 0, a02 = 0, a11 = 0, a12 = 0, a22 = 0, mean = 0;
    float m[kMaxBasis];
#pragma unroll
    for (int k = 0; k < kMaxBasis; k++) m[k] = k < K ? mu[i + k * cs] : 0.f;  // all loads in flight
#pragma unroll
    for (int k = 0; k < kMaxBasis; k++) {
        if (k >= K) break;
        const double mk = m[k], mm = mk * mk;
        mean += mk;
        a00 = fma(mm, b.P[k][0], a00);
        a01 = fma(mm, b.P[k][1], a01);
        a02 = fma(mm, b.P[k][2], a02);
        a11 = fma(mm, b.P[k][3], a11);
        a12 = fma(mm, b.P[k][4], a12);
        a22 = fma(mm, b.P[k][5], a22);
    }
    mean *= b.inv_k;
    a00 *= b.inv_k;
    a01 *= b.inv_k;
    a02 *= b.inv_k;
    a11 *= b.inv_k;
    a12 *= b.inv_k;
    a22 *= b.inv_k;
    double l0, l1, l2;  // ascending
    double e0 = 1, e1 = 0, e2 = 0;
    const double p1 = a01 * a01 + a02 * a02 + a12 * a12;
    const double q = (a00 + a11 + a22) * (1.0 / 3.0);
    const double p2 = (a00 - q) * (a00 - q) + (a11 - q) * (a11 - q) + (a22 - q) * (a22 - q) + 2.0 * p1;
    // only in thresholds: the root's estimate is enough
    const double scale = fmax(fabs(a00), fmax(fabs(a11), fabs(a22))) + __builtin_amdgcn_sqrt(p1);
    if (p1 <= 1e-30 * scale * scale) {
        // diagonal: sort the diagonal ascending, eigenvectors are the axes
        double dv[3] = {a00, a11, a22};
        int id[3] = {0, 1, 2};
        for (int s = 0; s < 2; s++)
            for (int t = 0; t < 2 - s; t++)
                if (dv[id[t + 1]] < dv[id[t]]) {
                    const int tt = id[t];
                    id[t] = id[t + 1];
                    id[t + 1] = tt;
                }
        l0 = dv[id[0]];
        l1 = dv[id[1]];
        l2 = dv[id[2]];
        e0 = id[0] == 0;
        e1 = id[0] == 1;
        e2 = id[0] == 2;
    } else {
        const double ip = rsqrt64(p2 * (1.0 / 6.0)), p = p2 * (1.0 / 6.0) * ip;
        const double b00 = (a00 - q) * ip, b11 = (a11 - q) * ip, b22 = (a22 - q) * ip;
        const double b01 = a01 * ip, b02 = a02 * ip, b12 = a12 * ip;
        double r = 0.5 * (b00 * (b11 * b22 - b12 * b12) - b01 * (b01 * b22 - b12 * b02) + b02 * (b01 * b12 - b11 * b02));
        r = fmin(1.0, fmax(-1.0, r));
        const double hh = 0.5 - 0.5 * fabs(r);
        const double h = hh > 0.0 ? hh * rsqrt64(hh) : 0.0;
        const float x = (float)hh;
        double t = h * (double)fmaf(fmaf(fmaf(fmaf(0.02792844f, x, 0.00243657f), x, 0.02407489f), x, 0.04923956f), x, 0.33333484f);
#pragma unroll
        for (int it = 0; it < 2; it++) {
            const float tf = (float)t;
            const float res = (float)fma(t, fma(-4.0 * t, t, 3.0), -h);
            t -= (double)(res * rcpf(fmaf(-12.f * tf, tf, 3.f)));
        }
        const double t2 = t * t, u = 1.0 - t2;
        const double cf = 1.0 - 2.0 * t2, sf = 2.0 * t * (u * rsqrt64(u));  // cos f, sin f
        const double big = p * (2.0 * cf), other = p * fma(1.7320508075688772935, sf, cf);
        l2 = q + (r >= 0.0 ? big : other);
        l0 = q - (r >= 0.0 ? other : big);
        l1 = 3.0 * q - l0 - l2;
        // rows of C - l0 I; the eigenvector is orthogonal to all of them
        const double r0[3] = {a00 - l0, a01, a02}, r1[3] = {a01, a11 - l0, a12}, r2[3] = {a02, a12, a22 - l0};
        const double c01[3] = {r0[1] * r1[2] - r0[2] * r1[1], r0[2] * r1[0] - r0[0] * r1[2], r0[0] * r1[1] - r0[1] * r1[0]};
        const double c02[3] = {r0[1] * r2[2] - r0[2] * r2[1], r0[2] * r2[0] - r0[0] * r2[2], r0[0] * r2[1] - r0[1] * r2[0]};
        const double c12[3] = {r1[1] * r2[2] - r1[2] * r2[1], r1[2] * r2[0] - r1[0] * r2[2], r1[0] * r2[1] - r1[1] * r2[0]};
        const double n01 = c01[0] * c01[0] + c01[1] * c01[1] + c01[2] * c01[2];
        const double n02 = c02[0] * c02[0] + c02[1] * c02[1] + c02[2] * c02[2];
        const double n12 = c12[0] * c12[0] + c12[1] * c12[1] + c12[2] * c12[2];
        const double* best = c01;
        double nb = n01;
        if (n02 > nb) {
            best = c02;
            nb = n02;
        }
        if (n12 > nb) {
            best = c12;
            nb = n12;
        }
        if (nb > 1e-30 * scale * scale * scale * scale) {
            const double in = rsqrt64(nb);
            e0 = best[0] * in;
            e1 = best[1] * in;
            e2 = best[2] * in;
        } else {
            // lambda_min is (at least) double: any unit vector orthogonal to the
            // largest row of C - l0 I spans the eigenspace.
            const double n0 = r0[0] * r0[0] + r0[1] * r0[1] + r0[2] * r0[2];
            const double n1 = r1[0] * r1[0] + r1[1] * r1[1] + r1[2] * r1[2];
            const double n2 = r2[0] * r2[0] + r2[1] * r2[1] + r2[2] * r2[2];
            const double* rr = r0;
            if (n1 > n0 && n1 >= n2) rr = r1;
            if (n2 > n0 && n2 > n1) rr = r2;
            // cross with the axis least aligned with rr
            const double ax = fabs(rr[0]), ay = fabs(rr[1]), az = fabs(rr[2]);
            double t[3] = {0, 0, 0};
            if (ax <= ay && ax <= az)
                t[0] = 1;
            else if (ay <= az)
                t[1] = 1;
            else
                t[2] = 1;
            double w0 = rr[1] * t[2] - rr[2] * t[1], w1 = rr[2] * t[0] - rr[0] * t[2], w2 = rr[0] * t[1] - rr[1] * t[0];
            const double wn = sqrt(w0 * w0 + w1 * w1 + w2 * w2);
            if (wn > 0) {
                e0 = w0 / wn;
                e1 = w1 / wn;
                e2 = w2 / wn;
            }
        }
    }
    const double sg = (e2 >= 0) ? 1.0 : -1.0;
    md[i] = (float)(sg * mean * e0);
    md[i + cs] = (float)(sg * mean * e1);
    md[i + 2 * cs] = (float)(sg * mean * e2);
    const float f0 = (float)l0, f1 = (float)l1, f2 = (float)l2;
    const float tot = f0 + f1 + f2;
    ev[i] = f0 / tot;
    ev[i + cs] = f1 / tot;
    ev[i + 2 * cs] = f2 / tot;
}

// Ellipsoid phantom in the reference layout, voxel x at (x-(N+1)/2)*vs.
// params: 16 doubles per ellipsoid (centre[3], semi-axes[3], rotation[9], value).
__global__ void k_ellipsoids(float* vol, int N, double vs, const double* __restrict__ prm, int count) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
    if (x >= N) return;
    const double p0 = ((double)x - (N + 1) * 0.5) * vs, p1 = ((double)y - (N + 1) * 0.5) * vs,
                 p2 = ((double)z - (N + 1) * 0.5) * vs;
    double acc = 0;
    for (int e = 0; e < count; e++) {
        const double* q = prm + 16 * e;
        const double d0 = p0 - q[0], d1 = p1 - q[1], d2 = p2 - q[2];
        double r2 = 0;
        for (int i = 0; i < 3; i++) {
            const double bb = q[6 + 3 * i] * d0 + q[7 + 3 * i] * d1 + q[8 + 3 * i] * d2;
            r2 += (bb / q[3 + i]) * (bb / q[3 + i]);
        }
        if (r2 <= 1.0) acc += q[15];
    }
    vol[x + (int64_t)N * y + (int64_t)N * N * z] = (float)acc;
}

// Hollow cylinder about the z axis (all z): value where r_out - thick < r <= r_out,
// voxel centres (x-(N+1)/2)*vs as for the ellipsoids.  Adds into vol (reference layout).
__global__ void k_cylinder_shell(float* vol, int N, double vs, double r_out, double thick, double value) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
    if (x >= N) return;
    const double px = ((double)x - (N + 1) * 0.5) * vs, py = ((double)y - (N + 1) * 0.5) * vs;
    const double r = sqrt(px * px + py * py);
    if (r <= r_out && r > r_out - thick) vol[x + (int64_t)N * y + (int64_t)N * N * z] += (float)value;
}

// Fibres: params 8 doubles each (centre[3] mm, unit direction f[3], radius mm,
// half-length mm).  Inside a fibre every channel k gains s_k = |S_k x f|^2
// (scattering strength 1 per unit direction-weight; values add).  Reference
// layout, K channels of N^3.
__global__ void k_fibres(float* vol, int N, double vs, const double* __restrict__ prm, int count, const Basis b,
                         int K) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
    if (x >= N) return;
    const double p0 = ((double)x - (N + 1) * 0.5) * vs, p1 = ((double)y - (N + 1) * 0.5) * vs,
                 p2 = ((double)z - (N + 1) * 0.5) * vs;
    float acc[kMaxBasis];
    for (int k = 0; k < kMaxBasis; k++) acc[k] = 0.f;
    for (int e = 0; e < count; e++) {
        const double* q = prm + 8 * e;
        const double d0 = p0 - q[0], d1 = p1 - q[1], d2 = p2 - q[2];
        const double t = d0 * q[3] + d1 * q[4] + d2 * q[5];
        if (fabs(t) > q[7]) continue;
        const double r0 = d0 - t * q[3], r1 = d1 - t * q[4], r2 = d2 - t * q[5];
        if (r0 * r0 + r1 * r1 + r2 * r2 > q[6] * q[6]) continue;
        for (int k = 0; k < K; k++) {
            const double c0 = b.S[k][1] * q[5] - b.S[k][2] * q[4];
            const double c1 = b.S[k][2] * q[3] - b.S[k][0] * q[5];
            const double c2 = b.S[k][0] * q[4] - b.S[k][1] * q[3];
            acc[k] += (float)(c0 * c0 + c1 * c1 + c2 * c2);
        }
    }
    const int64_t i = x + (int64_t)N * y + (int64_t)N * N * z, N3 = (int64_t)N * N * N;
    for (int k = 0; k < K; k++) vol[i + k * N3] += acc[k];
}

// Scalar fibres: `value` added inside every fibre (attenuation phantom).
__global__ void k_fibres_scalar(float* vol, int N, double vs, const double* __restrict__ prm, int count,
                                float value) {
    const int x = blockIdx.x * blockDim.x + threadIdx.x, y = blockIdx.y, z = blockIdx.z;
    if (x >= N) return;
    const double p0 = ((double)x - (N + 1) * 0.5) * vs, p1 = ((double)y - (N + 1) * 0.5) * vs,
                 p2 = ((double)z - (N + 1) * 0.5) * vs;
    float acc = 0.f;
    for (int e = 0; e < count; e++) {
        const double* q = prm + 8 * e;
        const double d0 = p0 - q[0], d1 = p1 - q[1], d2 = p2 - q[2];
        const double t = d0 * q[3] + d1 * q[4] + d2 * q[5];
        if (fabs(t) > q[7]) continue;
        const double r0 = d0 - t * q[3], r1 = d1 - t * q[4], r2 = d2 - t * q[5];
        if (r0 * r0 + r1 * r1 + r2 * r2 > q[6] * q[6]) continue;
        acc += value;
    }
    vol[x + (int64_t)N * y + (int64_t)N * N * z] += acc;
}

__global__ void k_poisson_noise(float* y, const float* p, int64_t n, double I0, uint64_t seed) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    UniformStream us(seed, (uint64_t)i);
    const double c = poisson_sample(I0 * exp(-(double)p[i]), us);
    y[i] = (float)(-log(fmax(c, 1.0) / I0));
}

__global__ void k_gaussian_noise(float* y, const float* x, int64_t n, double sigma, uint64_t seed) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    UniformStream us(seed, (uint64_t)i);
    const double u1 = us.next(), u2 = us.next();
    const double g = sqrt(-2.0 * log(u1)) * cos(6.283185307179586476925 * u2);  // Box-Muller
    y[i] = (float)((double)x[i] * (1.0 + sigma * g));
}

inline unsigned grid1(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

static int forward_waves(int kind) { return kind == FWD_XTT ? kFwdXttWaves : kFwdWaves; }

// Standalone forward kernel: chunks per column and step by the volume's depth
// (see splat_columns), one step for a column of up to eight, so that no step of a
// whole column is partial but for its last lanes (steps of 8 for every depth above
// 256, of 4 for three chunks: 288^3 608 against 509 us, 384^3 1121 against 1044,
// 160^3 203 against 183, 20 views each; ten chunks in two steps of five: 5 %
// slower than 8 + 2); of four for the untilted views of a launch that also holds
// tilted ones.  XTT by the basis count rounded up to a compiled size (the
// registers of a voxel's coefficients).
template <int KIND>
static const void* forward_kernel_of(bool axis, int nz) {
    if (!axis) return (const void*)k_forward<KIND, false, 1, kFwdWaves, 4>;
    const int ch = std::min((nz + 63) / 64, 8);
    switch (ch) {
        case 1: return (const void*)k_forward<KIND, true, 1, kFwdWaves, 1>;
        case 2: return (const void*)k_forward<KIND, true, 1, kFwdWaves, 2>;
        case 3: return (const void*)k_forward<KIND, true, 1, kFwdWaves, 3>;
        case 4: return (const void*)k_forward<KIND, true, 1, kFwdWaves, 4>;
        case 5: return (const void*)k_forward<KIND, true, 1, kFwdWaves, 5>;
        case 6: return (const void*)k_forward<KIND, true, 1, kFwdWaves, 6>;
        case 7: return (const void*)k_forward<KIND, true, 1, kFwdWaves, 7>;
        default: return (const void*)k_forward<KIND, true, 1, kFwdWaves, 8>;
    }
}
template <int KM>
static const void* forward_kernel_xtt(bool axis) {
    return axis ? (const void*)k_forward<FWD_XTT, true, KM, kFwdXttWaves, kXttChunks>
                : (const void*)k_forward<FWD_XTT, false, KM, kFwdXttWaves, kXttChunks>;
}
static const void* forward_kernel(int kind, bool axis, const Dims& d) {
    if (kind == FWD_WEIGHT) return forward_kernel_of<FWD_WEIGHT>(axis, d.nz);
    if (kind == FWD_PLAIN) return forward_kernel_of<FWD_PLAIN>(axis, d.nz);
    if (d.K <= 4) return forward_kernel_xtt<4>(axis);
    if (d.K <= 8) return forward_kernel_xtt<8>(axis);
    if (d.K <= 13) return forward_kernel_xtt<13>(axis);
    return forward_kernel_xtt<16>(axis);
}

hipError_t launch_forward(const FwdArgs& a, int kind, bool axis, hipStream_t stream) {
    const int nblk = a.n_bands * std::max(a.n_sub, 1) * a.n_slots * a.n_chunks;
    if (nblk == 0) return hipSuccess;
    const unsigned grid = (unsigned)(8 * ((nblk + 7) / 8));
    const size_t lds = forward_lds_bytes(kind, a.vb);
    FwdArgs arg = a;
    void* args[] = {&arg};
    return (kind == FWD_PLAIN || kind == FWD_WEIGHT || kind == FWD_XTT)
               ? hipLaunchKernel(forward_kernel(kind, axis, a.d), dim3(grid), dim3(64 * forward_waves(kind)),
                                 args, lds, stream)
               : hipErrorInvalidValue;
}

constexpr int kDefaultGx = 4;  // plain kinds
int default_zpl(int N) { return N > 128 ? 4 : (N > 64 ? 2 : 1); }

inline bool bwd_xtt(int kind) { return kind == BWD_XTT_RAW || kind == BWD_XTT_MLEM || kind == BWD_XTT_ART; }

int backward_threads(int kind) {
    return bwd_xtt(kind) ? BwdLarge<BWD_XTT_MLEM, 1, 4>::Cfg::threads : BwdLarge<BWD_MLEM, 1, 1>::Cfg::threads;
}

// Estimated footprint of a tile of cx x cy columns and 64 zpl voxels: its
// diagonal and, along z, its extent at the tilt, at px detector pixels per voxel
// (0: at the largest magnification in the volume).  Launch shapes only: a
// footprint that turns out larger is read from the image directly.
static void backward_footprint(const Dims& d, int cx, int cy, int zpl, float& w, float& h, float px = 0.0f) {
    const float diag = std::sqrt((float)((cx - 1) * (cx - 1) + (cy - 1) * (cy - 1))), z = 64.0f * zpl - 1.0f;
    if (px == 0.0f) px = d.px;
    w = (diag + z * d.tilt_sin) * px + 2.02f;
    h = (z * d.tilt_cos + diag * d.tilt_sin) * px + 2.02f;
}

// Tile counts of a grid of `waves` waves, gx along x, each of cpw x cpw columns
// and 64 zpl voxels.
static void backward_tiles(BwdArgs& a, int waves, int cpw, int zpl, int gx) {
    const int N = a.d.N;
    a.zpl = zpl;
    a.gx = gx;
    a.gy = waves / gx;
    a.tiles_x = (N + cpw * a.gx - 1) / (cpw * a.gx);
    a.tiles_y = (N + cpw * a.gy - 1) / (cpw * a.gy);
    a.tiles_z = (a.d.nz + 64 * zpl - 1) / (64 * zpl);  // z >= nz: never visited
    a.n_tiles = a.tiles_x * a.tiles_y * a.tiles_z;
    a.per_xcd = (a.n_tiles + 7) / 8;
    // wider footprints than the fixed width (a tile's diagonal, see backward_footprint)
    float w, h;
    backward_footprint(a.d, cpw * a.gx, cpw * a.gy, zpl, w, h);
    a.wide = w > (cpw == 1 ? 8.0f : 16.0f) || h > (cpw == 1 ? 64.0f * 3 : 64.0f * 7);
}

bool backward_shape(BwdArgs& a, int zpl, int gx, bool xtt) {
    // Plain / FDK: 2x2 columns x zpl z per lane, 16 waves as gx x gy column
    // groups (a (2gx) x (2gy)-column tile, 64*zpl z).  XTT (2K accumulators per
    // voxel): one column x zpl (1 or 2) z per lane, 8 waves.
    if (xtt && zpl == 0) zpl = 1;
    if (xtt && zpl > 2) return false;
    if (zpl == 0) zpl = default_zpl(a.d.N);
    // default column layout: 8 x 8 columns (plain); 2 x 4 for XTT (measured
    // 144.6 against 146.2 ms for 4 x 2 at 256^3 x 13, 4 x 360 views)
    if (gx == 0) gx = xtt ? 2 : kDefaultGx;
    if (!(zpl == 1 || zpl == 2 || zpl == 4)) return false;
    if (!(gx == 1 || gx == 2 || gx == 4 || gx == 8 || gx == 16)) return false;
    const int waves = xtt ? 8 : 16;
    gx = std::min(gx, waves);  // XTT blocks have 8 waves: gx 16 is taken as 8
    backward_tiles(a, waves, xtt ? 1 : 2, zpl, gx);
    return true;
}

// Shape of a standalone launch where the plan leaves it open (zpl and gx 0);
// true: the kernel for few tiles (BwdSmall).
// Plain, untilted: the z depth zpl (1 to 5) that covers the volume's 64-voxel
// chunks with the least work, tiles_z (zpl + 2): a column's terms and a
// footprint's edges cost about as much per view as two chunks (three chunks,
// raw sums, 160^3 / 180 views: zpl 3 615, 4 724, 2 971 us; five chunks, 320^3 / 60
// views: zpl 5, 4, 2 raw 1127, 1867, 2021 us; FDK 926, 1667, 1904; ART 911, 1662,
// 1875; MLEM, whose two sums per voxel spill some registers at zpl 5, 1007, 1746,
// 1945).
// Footprints of any width (w > 16 where the magnification is largest): the depth
// whose footprint fits the staging buffer 0.4 edges off the centre; the few tiles
// nearer the source read the image directly.  (By the nearest voxel 512^3
// 0.4, 400^3 0.4 mm at 300 mm and 512^3 0.5 mm at 1000 mm took zpl 1, 2, 2: 6557,
// 2464, 4128 against 4073, 1802, 3226 us for 32 views; at the centre 512^3 0.5 mm at
// 500 mm would take 4: 9500 against 4123 us.)
// Fewer than kSmallTiles such tiles leave most of the chip idle: BwdSmall
// (64^3 / 90 views, 64 tiles: 41 against 95 us; but at 96^3 / 90 views, 144
// tiles: 177 against 125 us).
// Tilted: the largest depth whose footprint fits the staging buffer.
// XTT: two voxels per lane halve the per-view overhead of a column (35.1
// against 23.0 ms for ART at 256^3 x 13, 4 x 90 views) where the volume has
// more than 64 layers, the footprint fits and the accumulators do.  Where the
// footprint is of any width, it fits as above (256^3 x 3 0.6 mm at 300 mm, 16
// views: 1410 against 817 us); a fixed width with one voxel is better than any width
// with two (400^3 x 3 0.4 mm at 300 mm: 2725 against 3900 us).
constexpr int kSmallTiles = 96;
static bool backward_choose(BwdArgs& a, int kind, bool axis) {
    const Dims& d = a.d;
    const int chunks = (d.nz + 63) / 64;
    float w, h;
    if (bwd_xtt(kind)) {
        backward_footprint(d, 2, 4, 2, w, h);
        bool fits = axis ? h <= 192.0f : w * h <= 0.9f * 3584.0f;
        if (axis && w > 8.0f) {
            backward_footprint(d, 2, 4, 2, w, h, d.px_mid);
            fits = w * h <= 0.9f * 3584.0f;
        }
        // (26 accumulators per voxel of 13 coefficients: two voxels spill where both sums are kept)
        const bool regs = a.d.K <= 8 || (kind == BWD_XTT_ART && (axis || a.d.K <= 13));
        backward_tiles(a, 8, 1, chunks > 1 && fits && regs ? 2 : 1, 2);
        return false;
    }
    int zpl = 1;
    if (axis) {
        int best = 0;
        for (int z = 5; z >= 1; z--) {
            backward_footprint(d, 8, 8, z, w, h);
            if (w > 16.0f) {
                float wm, hm;
                backward_footprint(d, 8, 8, z, wm, hm, d.px_mid);
                if (z > 1 && (z % 2 == 1 || wm * hm > 0.9f * 7168.0f)) continue;
            } else if (z > 1 && h > 448.0f) {
                continue;
            }
            const int cost = (chunks + z - 1) / z * (z + 2);
            if (best == 0 || cost < best) {
                best = cost;
                zpl = z;
            }
        }
    } else {
        for (int z : {4, 2}) {
            backward_footprint(d, 8, 8, z, w, h);
            if (zpl == 1 && z <= default_zpl(d.nz) && w * h <= 0.9f * 7168.0f) zpl = z;
        }
    }
    backward_tiles(a, 16, 2, zpl, 4);
    backward_footprint(d, 4, 2, 1, w, h);
    if (axis && a.n_tiles < kSmallTiles && w <= 8.0f && h <= 128.0f) {
        backward_tiles(a, 8, 1, 1, 4);
        return true;
    }
    return false;
}

template <class C, bool TILT>
static hipError_t start_backward(const BwdArgs& a, hipStream_t stream) {
    hipLaunchKernelGGL((k_backward<C, TILT>), dim3((unsigned)(8 * a.per_xcd)), dim3(C::threads), C::lds_bytes, stream,
                       a);
    return hipGetLastError();
}

template <int KIND, int ZPL, int KM>
static hipError_t start_backward_large(const BwdArgs& a, bool axis, hipStream_t stream) {
    if (!axis) return start_backward<typename BwdLarge<KIND, ZPL, KM>::Wide, true>(a, stream);
    if (a.wide) return start_backward<typename BwdLarge<KIND, ZPL, KM>::Wide, false>(a, stream);
    return start_backward<typename BwdLarge<KIND, ZPL, KM>::Cfg, false>(a, stream);
}

template <int KIND>
static hipError_t start_backward_plain(const BwdArgs& a, bool axis, bool small, hipStream_t stream) {
    if (small) return start_backward<typename BwdSmall<KIND>::Cfg, false>(a, stream);
    switch (a.zpl) {
        case 1: return start_backward_large<KIND, 1, 1>(a, axis, stream);
        case 2: return start_backward_large<KIND, 2, 1>(a, axis, stream);
        case 4: return start_backward_large<KIND, 4, 1>(a, axis, stream);
        case 3: if (axis) return start_backward<typename BwdLarge<KIND, 3, 1>::Cfg, false>(a, stream); break;
        case 5: if (axis) return start_backward<typename BwdLarge<KIND, 5, 1>::Cfg, false>(a, stream); break;
    }
    return hipErrorInvalidValue;
}

template <int KIND, int ZPL>
static hipError_t start_backward_xtt(const BwdArgs& a, bool axis, hipStream_t stream) {
    if (a.d.K <= 4) return start_backward_large<KIND, ZPL, 4>(a, axis, stream);
    if (a.d.K <= 8) return start_backward_large<KIND, ZPL, 8>(a, axis, stream);
    if (a.d.K <= 13) return start_backward_large<KIND, ZPL, 13>(a, axis, stream);
    return start_backward_large<KIND, ZPL, 16>(a, axis, stream);
}

hipError_t launch_backward(BwdArgs a, int kind, bool axis, hipStream_t stream) {
    bool small = false;
    // The shape that xr_plan_get_tiles reports for a plan that leaves it open stands for the same
    // choice, so that setting it, or tuning that finds it fastest, does not lose the shapes that a
    // setting cannot name.  (The batched kernels have the set shapes alone: their tuning is literal.)
    const bool open = (a.zpl == 0 && a.gx == 0) ||
                      (!a.literal && !bwd_xtt(kind) && a.zpl == default_zpl(a.d.N) && a.gx == kDefaultGx);
    if (open)
        small = backward_choose(a, kind, axis);
    else if (!backward_shape(a, a.zpl, a.gx, bwd_xtt(kind)))
        return hipErrorInvalidValue;
    switch (kind) {
        case BWD_RAW: return start_backward_plain<BWD_RAW>(a, axis, small, stream);
        case BWD_MLEM: return start_backward_plain<BWD_MLEM>(a, axis, small, stream);
        case BWD_ART: return start_backward_plain<BWD_ART>(a, axis, small, stream);
        case BWD_FDK: return start_backward_plain<BWD_FDK>(a, axis, small, stream);
        case BWD_XTT_RAW:
            return a.zpl == 2 ? start_backward_xtt<BWD_XTT_RAW, 2>(a, axis, stream) : start_backward_xtt<BWD_XTT_RAW, 1>(a, axis, stream);
        case BWD_XTT_MLEM:
            return a.zpl == 2 ? start_backward_xtt<BWD_XTT_MLEM, 2>(a, axis, stream) : start_backward_xtt<BWD_XTT_MLEM, 1>(a, axis, stream);
        case BWD_XTT_ART:
            return a.zpl == 2 ? start_backward_xtt<BWD_XTT_ART, 2>(a, axis, stream) : start_backward_xtt<BWD_XTT_ART, 1>(a, axis, stream);
        default: return hipErrorInvalidValue;
    }
}

// Basis count rounded up to a compiled size of the XTT kernels.
inline int xtt_km(int kmax) { return kmax <= 4 ? 4 : (kmax <= 8 ? 8 : (kmax <= 13 ? 13 : 16)); }

const void* forward_batch_xtt_kernel(int kmax) {
    switch (xtt_km(kmax)) {
        case 4: return (const void*)k_forward_batch_xtt<4>;
        case 8: return (const void*)k_forward_batch_xtt<8>;
        case 13: return (const void*)k_forward_batch_xtt<13>;
        default: return (const void*)k_forward_batch_xtt<16>;
    }
}

hipError_t launch_forward_batch(const FwdArgs* items, const int* item_end, int n_items, unsigned* queue,
                                int ticket_slot, size_t lds_bytes, int grid, int step, int loss_shift, int kind,
                                bool axis_all, hipStream_t stream, int kmax) {
    if (n_items <= 0 || grid <= 0) return hipSuccess;
    if (kind == FWD_XTT) {
        void* args[] = {(void*)&items, (void*)&item_end, (void*)&n_items, (void*)&queue, (void*)&ticket_slot,
                        (void*)&step, (void*)&loss_shift};
        return hipLaunchKernel(forward_batch_xtt_kernel(kmax), dim3(grid), dim3(64 * kFwdXttWaves), args, lds_bytes,
                               stream);
    }
    if (kind != FWD_PLAIN) return hipErrorInvalidValue;
    if (axis_all)
        hipLaunchKernelGGL((k_forward_batch_axis<FWD_PLAIN>), dim3(grid), dim3(64 * kFwdWaves), lds_bytes, stream,
                           items, item_end, n_items, queue, ticket_slot, step, loss_shift);
    else
        hipLaunchKernelGGL((k_forward_batch<FWD_PLAIN>), dim3(grid), dim3(64 * kFwdBatchWaves), lds_bytes, stream, items,
                           item_end, n_items, queue, ticket_slot, step, loss_shift);
    return hipGetLastError();
}

template <int KIND, int ZPL, int KM>
static constexpr size_t batch_lds_of() {
    typedef BwdLarge<KIND, ZPL, KM> L;
    return L::Cfg::lds_bytes > L::Wide::lds_bytes ? L::Cfg::lds_bytes : L::Wide::lds_bytes;
}

static size_t backward_batch_lds_bytes(int kind, int zpl, int kmax) {
    if (!bwd_xtt(kind))
        return zpl == 4 ? batch_lds_of<BWD_MLEM, 4, 1>()
                        : (zpl == 2 ? batch_lds_of<BWD_MLEM, 2, 1>() : batch_lds_of<BWD_MLEM, 1, 1>());
    switch (xtt_km(kmax)) {
        case 4: return batch_lds_of<BWD_XTT_MLEM, 1, 4>();
        case 8: return batch_lds_of<BWD_XTT_MLEM, 1, 8>();
        case 13: return batch_lds_of<BWD_XTT_MLEM, 1, 13>();
        default: return batch_lds_of<BWD_XTT_MLEM, 1, 16>();
    }
}

// Batched backprojection kernel of (kind, zpl) (XTT kinds: zpl 1, one column
// per wave, kmax basis vectors at most), or nullptr.
const void* backward_batch_kernel(int kind, int zpl, int kmax) {
#define XR_BB(KD)                                                        \
    if (kind == KD) {                                                    \
        if (zpl == 4) return (const void*)k_backward_batch<BwdLarge<KD, 4, 1>::Cfg, BwdLarge<KD, 4, 1>::Wide>;       \
        if (zpl == 2) return (const void*)k_backward_batch<BwdLarge<KD, 2, 1>::Cfg, BwdLarge<KD, 2, 1>::Wide>;       \
        if (zpl == 1) return (const void*)k_backward_batch<BwdLarge<KD, 1, 1>::Cfg, BwdLarge<KD, 1, 1>::Wide>;       \
    }
    XR_BB(BWD_MLEM)
    XR_BB(BWD_ART)
#undef XR_BB
#define XR_BBX(KD)                                                                \
    if (kind == KD && zpl == 1) {                                                 \
        switch (xtt_km(kmax)) {                                                   \
            case 4: return (const void*)k_backward_batch<BwdLarge<KD, 1, 4>::Cfg, BwdLarge<KD, 1, 4>::Wide>;            \
            case 8: return (const void*)k_backward_batch<BwdLarge<KD, 1, 8>::Cfg, BwdLarge<KD, 1, 8>::Wide>;            \
            case 13: return (const void*)k_backward_batch<BwdLarge<KD, 1, 13>::Cfg, BwdLarge<KD, 1, 13>::Wide>;          \
            default: return (const void*)k_backward_batch<BwdLarge<KD, 1, 16>::Cfg, BwdLarge<KD, 1, 16>::Wide>;          \
        }                                                                         \
    }
    XR_BBX(BWD_XTT_MLEM)
    XR_BBX(BWD_XTT_ART)
#undef XR_BBX
    return nullptr;
}

hipError_t launch_backward_batch(const BwdArgs* items, const int* item_end, int n_items, unsigned* queue, int grid,
                                 int step, int kind, int zpl, hipStream_t stream, int kmax) {
    if (n_items <= 0 || grid <= 0) return hipSuccess;
    const void* k = backward_batch_kernel(kind, zpl, kmax);
    if (!k) return hipErrorInvalidValue;
    void* args[] = {(void*)&items, (void*)&item_end, (void*)&n_items, (void*)&queue, (void*)&step};
    return hipLaunchKernel(k, dim3(grid), dim3(backward_threads(kind)), args, backward_batch_lds_bytes(kind, zpl, kmax),
                           stream);
}

int batch_blocks_per_cu_forward(int kind, size_t lds_bytes, bool axis_all, int kmax) {
    int n = 0;
    if (kind == FWD_XTT) {
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, forward_batch_xtt_kernel(kmax),
                                                                          64 * kFwdXttWaves, lds_bytes);
        return e == hipSuccess ? n : 0;
    }
    if (kind != FWD_PLAIN) return 0;
    const hipError_t e =
        axis_all ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void*)k_forward_batch_axis<FWD_PLAIN>,
                                                                64 * kFwdWaves, lds_bytes)
                 : hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, (const void*)k_forward_batch<FWD_PLAIN>,
                                                                64 * kFwdBatchWaves, lds_bytes);
    return e == hipSuccess ? n : 0;
}

size_t forward_lds_bytes(int kind, int vb) {
    const int acc_bytes = (kind == FWD_WEIGHT) ? 8 : 4;
    return ((size_t)fwd_red_slot(vb + 2, acc_bytes) + 2 * kFwdWaves) * sizeof(unsigned long long);
}

int forward_blocks_per_cu(int kind, bool axis, const Dims& d, size_t lds_bytes) {
    int n = 0;
    const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, forward_kernel(kind, axis, d),
                                                                      64 * forward_waves(kind), lds_bytes);
    return e == hipSuccess ? n : 0;
}

int batch_blocks_per_cu_backward(int kind, int zpl, int kmax) {
    int n = 0;
    const void* k = backward_batch_kernel(kind, zpl, kmax);
    if (!k) return 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, k, backward_threads(kind),
                                                     backward_batch_lds_bytes(kind, zpl, kmax)) !=
        hipSuccess)
        return 0;
    return n;
}

int absmax_blocks(int64_t max_len, int n_seg) {
    // at least 64 floats per thread in the largest segment; about 2048 blocks in all
    const int64_t want = (max_len + 256 * 64 - 1) / (256 * 64);
    return (int)std::max<int64_t>(1, std::min<int64_t>(want, std::max(1, 2048 / std::max(n_seg, 1))));
}

hipError_t launch_absmax_seg(const float* const* segs, const int64_t* seg_len, float* out, int n_seg,
                             int blocks_per_seg, hipStream_t stream) {
    if (n_seg <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_absmax_seg, dim3((unsigned)blocks_per_seg, (unsigned)n_seg), dim3(256), 0, stream, segs,
                       seg_len, out);
    return hipGetLastError();
}

hipError_t launch_fdk_filter(const float* src, float* dst, const float* weight, const float* taps, int U, int V,
                             const int32_t* views, int n_views, int code_base, int circular, hipStream_t stream) {
    const int64_t n_rows = (int64_t)n_views * V;
    if (n_rows > INT32_MAX - kFiltBM) return hipErrorInvalidValue;
    // the widest block that pads the columns no more than a narrower one does and
    // leaves two blocks per CU (512 of 64 rows)
    int nt = 2;
    for (int t = 4; t <= 8; t *= 2) {
        const int64_t cols = (U + 64 * t - 1) / (64 * t), narrow = (U + 64 * nt - 1) / (64 * nt);
        if (cols * t <= narrow * nt && cols * ((n_rows + kFiltBM - 1) / kFiltBM) >= 512) nt = t;
    }
    const auto kernel = nt == 8 ? k_fdk_filter<8> : nt == 4 ? k_fdk_filter<4> : k_fdk_filter<2>;
    // row tiles in launches of at most 65535 tiles (the grid's y limit)
    const int64_t per_launch = (int64_t)65535 * kFiltBM;
    for (int64_t base = 0; base < n_rows; base += per_launch) {
        const int64_t rows = std::min(per_launch, n_rows - base);
        const dim3 grid((U + 64 * nt - 1) / (64 * nt), (unsigned)((rows + kFiltBM - 1) / kFiltBM));
        hipLaunchKernelGGL(kernel, grid, dim3(256), 0, stream, src, dst, weight, taps, U, V, views, (int)n_rows,
                           (int)base, code_base, circular);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

hipError_t launch_fdk_weight(float* weight, int U, int V, float sdd, float det, hipStream_t stream) {
    hipLaunchKernelGGL(k_fdk_weight, dim3(grid1(U, 256), V), dim3(256), 0, stream, weight, U, V, sdd, det);
    return hipGetLastError();
}

hipError_t launch_to_internal(const float* ref, float* internal, int N, int channels, hipStream_t stream) {
    hipLaunchKernelGGL((k_transpose<true>), dim3(grid1(N, 32), grid1(N, 32), (unsigned)N * channels), dim3(32, 8), 0,
                       stream, ref, internal, N);
    return hipGetLastError();
}

hipError_t launch_from_internal(const float* internal, float* ref, int N, int channels, hipStream_t stream) {
    hipLaunchKernelGGL((k_transpose<false>), dim3(grid1(N, 32), grid1(N, 32), (unsigned)N * channels), dim3(32, 8), 0,
                       stream, internal, ref, N);
    return hipGetLastError();
}

hipError_t launch_lane_copy(const float* cols, float* out, int N, int channels, int lane_axis, hipStream_t stream) {
    const dim3 grid(grid1(N, 32), grid1(N, 32), (unsigned)N * channels);
    if (lane_axis == 1)
        hipLaunchKernelGGL((k_lane_copy<1>), grid, dim3(32, 8), 0, stream, cols, out, N);
    else
        hipLaunchKernelGGL((k_lane_copy<0>), grid, dim3(32, 8), 0, stream, cols, out, N);
    return hipGetLastError();
}

hipError_t launch_orth_normal(const float* vol, float* coef, float* loss, int64_t n, int rot, const float* est,
                              const Basis& b, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_orth_normal, dim3(grid1(n, 256)), dim3(256), 0, stream, vol, coef, loss, n, rot, est, b);
    return hipGetLastError();
}

hipError_t launch_orth_update_est(const float* vol, float* est, int64_t n, int iter, const Basis& b,
                                  hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_orth_update_est, dim3(grid1(n, 256)), dim3(256), 0, stream, vol, est, n, iter, b);
    return hipGetLastError();
}

hipError_t launch_orth_md(const float* vol, const float* coef, float* md, int64_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_orth_md, dim3(grid1(n, 256)), dim3(256), 0, stream, vol, coef, md, n);
    return hipGetLastError();
}

hipError_t launch_orth_mean_filter(const float* src, const float* vol, int N, float w, float* dst, hipStream_t stream) {
    const int64_t n = (int64_t)N * N * N;
    hipLaunchKernelGGL(k_orth_mean_filter, dim3(grid1(n, 256)), dim3(256), 0, stream, src, vol, N, w, dst);
    return hipGetLastError();
}

hipError_t launch_vol_down(const float* fine, float* coarse, int Nc, int f, hipStream_t stream) {
    const int64_t n = (int64_t)Nc * Nc * Nc;
    hipLaunchKernelGGL(k_vol_down, dim3(grid1(n, 256)), dim3(256), 0, stream, fine, coarse, Nc, f);
    return hipGetLastError();
}

hipError_t launch_vol_up_add(const float* a, const float* b, int Nc, int f, float* fine, float lo,
                             hipStream_t stream) {
    const int64_t N = (int64_t)Nc * f;
    hipLaunchKernelGGL(k_vol_up_add, dim3(grid1(N * N * N, 256)), dim3(256), 0, stream, a, b, Nc, f, fine, lo);
    return hipGetLastError();
}

hipError_t launch_sqrt_abs(float* vol, int64_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_sqrt_abs, dim3(grid1(n, 256)), dim3(256), 0, stream, vol, n);
    return hipGetLastError();
}

hipError_t launch_md_angles(const float* md, float* angle, int64_t n, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_md_angles, dim3(grid1(n, 256)), dim3(256), 0, stream, md, angle, n);
    return hipGetLastError();
}

hipError_t launch_md_normalise(float* md, int64_t n, float eps, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_md_normalise, dim3(grid1(n, 256)), dim3(256), 0, stream, md, n, eps);
    return hipGetLastError();
}

hipError_t launch_pca(const float* mu, int K, const Basis& b, int64_t nvox, int64_t chan_stride, float* md,
                      float* evalue, hipStream_t stream) {
    if (nvox == 0) return hipSuccess;
    PcaBasis pb{};
    for (int k = 0; k < kMaxBasis; k++) {
        const double x = b.S[k][0], y = b.S[k][1], z = b.S[k][2];
        const double P[6] = {x * x, x * y, x * z, y * y, y * z, z * z};
        std::copy(P, P + 6, pb.P[k]);
    }
    pb.inv_k = 1.0 / K;
    hipLaunchKernelGGL(k_pca, dim3(grid1(nvox, 256)), dim3(256), 0, stream, mu, K, pb, nvox, chan_stride, md, evalue);
    return hipGetLastError();
}

hipError_t launch_band_rows(const ViewGeom* vg, const Dims& d, int n_codes, int n_bands, int32_t* out,
                            hipStream_t stream) {
    const int64_t n = (int64_t)n_codes * n_bands * d.N;
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_band_rows, dim3(grid1(n, 256)), dim3(256), 0, stream, vg, d, n_codes, n_bands, out);
    return hipGetLastError();
}

hipError_t launch_absmax(const float* x, int64_t n, float* out, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_absmax, dim3((unsigned)absmax_blocks(n, 1)), dim3(256), 0, stream, x, n, out);
    return hipGetLastError();
}

hipError_t launch_fill(float* p, int64_t n, float value, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_fill, dim3(grid1(n, 256)), dim3(256), 0, stream, p, n, value);
    return hipGetLastError();
}

hipError_t launch_clamp_min(float* p, int64_t n, float floor_value, float replacement, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_clamp_min, dim3(grid1(n, 256)), dim3(256), 0, stream, p, n, floor_value, replacement);
    return hipGetLastError();
}

hipError_t launch_ellipsoids(float* vol, int N, float vs, const double* params_dev, int count, hipStream_t stream) {
    hipLaunchKernelGGL(k_ellipsoids, dim3(grid1(N, 64), N, N), dim3(64), 0, stream, vol, N, (double)vs, params_dev,
                       count);
    return hipGetLastError();
}

hipError_t launch_cylinder_shell(float* vol, int N, float vs, double r_out, double thick, double value,
                                 hipStream_t stream) {
    hipLaunchKernelGGL(k_cylinder_shell, dim3(grid1(N, 64), N, N), dim3(64), 0, stream, vol, N, (double)vs, r_out,
                       thick, value);
    return hipGetLastError();
}

hipError_t launch_fibres(float* vol, int N, float vs, const double* params_dev, int count, const Basis& b, int K,
                         hipStream_t stream) {
    hipLaunchKernelGGL(k_fibres, dim3(grid1(N, 64), N, N), dim3(64), 0, stream, vol, N, (double)vs, params_dev, count,
                       b, K);
    return hipGetLastError();
}

hipError_t launch_fibres_scalar(float* vol, int N, float vs, const double* params_dev, int count, float value,
                                hipStream_t stream) {
    hipLaunchKernelGGL(k_fibres_scalar, dim3(grid1(N, 64), N, N), dim3(64), 0, stream, vol, N, (double)vs,
                       params_dev, count, value);
    return hipGetLastError();
}

hipError_t launch_poisson_noise(float* y, const float* p, int64_t n, double I0, uint64_t seed, hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_poisson_noise, dim3(grid1(n, 256)), dim3(256), 0, stream, y, p, n, I0, seed);
    return hipGetLastError();
}

hipError_t launch_gaussian_noise(float* y, const float* x, int64_t n, double sigma, uint64_t seed,
                                 hipStream_t stream) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_gaussian_noise, dim3(grid1(n, 256)), dim3(256), 0, stream, y, x, n, sigma, seed);
    return hipGetLastError();
}

}  // namespace xr
