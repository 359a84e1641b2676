// Kernels of the gradient-domain phase-contrast reconstruction
// (IR::gradReconstruct, reconstruct.cu:158-328) that the projectors do not
// cover: the per-view sinogram factor, the faces of the gradient volume that
// the reference's launches leave alone, and the Poisson integration of the x
// and y gradients (poissonSolveLDLT, poisson_cpu.cpp:15-112).
//
// The Poisson system of one z slice is the 5-point Laplacian with identity
// rows on the slice border and zero right side there, i.e. the Dirichlet
// problem (D_y + D_x) F = B on the M x M interior, M = n-2, D = tridiag(-1, 2,
// -1).  The type-I sine transform S[j][k] = sin(pi (j+1)(k+1) / (M+1))
// diagonalises D_y; each of its M modes leaves a tridiagonal system along x,
//   (D_x + e[k]) f_k = t_k,  t = S B (over y),  F = 2/(M+1) S f,
//   e[k] = 2 - 2 cos(pi (k+1) / (M+1)),
// solved exactly by elimination.  (Diagonalising D_x too costs four matrix
// products instead of two.)  S[M-1-j][k] = (-1)^k S[j][k], so the sum of rows
// y and M-1-y meets the even modes alone and their difference the odd ones:
// each product is two of half the size.  The products run in FP64 on the
// matrix cores, the elimination in FP64; the right sides are formed in FP32 as
// the reference forms them, and the result is rounded to FP32 once.
// A solve of 384^3: 7.8 ms with four full products, a host table of sines and
// its workspace allocated per call; 1.65 ms now (products 0.67 and 0.65 ms, 33
// TFLOP/s FP64; elimination 0.51 ms, 3.5 TB/s).
#include <hip/hip_runtime.h>
#include <cstdint>

#include "xr_internal.hpp"

namespace xr {

namespace {

// dst[view][pix] = coef[view] * src[view][pix] (sinogramGradientCoef, ir.cu:585-594).
__global__ void k_scale_views(const float* __restrict__ src, float* __restrict__ dst,
                              const float* __restrict__ coef, int64_t len_view, int64_t total) {
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t view = i / len_view;
        dst[i] = coef[view] * src[i];
    }
}

// Voxels with x >= ext or z >= ext of an N1^3 volume in the column layout
// (z + N1*(x + N1*y)) set to `value`: the layers the reference's launches do
// not reach (reconstruct.cu:203-204 size the grid from N, the kernels run to
// N1 = N+1).
__global__ void k_grad_faces(float* __restrict__ vol, int N1, int ext, float value) {
    const int layers = N1 - ext;
    const int64_t plane = (int64_t)N1 * N1;
    const int64_t per_face = (int64_t)layers * plane;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < 2 * per_face;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int face = (int)(i / per_face);
        const int64_t r = i - face * per_face;
        const int layer = (int)(r / plane);
        const int64_t q = r - layer * plane;
        const int a = (int)(q / N1), b = (int)(q - (int64_t)a * N1);  // a: y, b: the other free axis
        int64_t idx;
        if (face == 0)
            idx = b + (int64_t)N1 * ((ext + layer) + (int64_t)N1 * a);  // x = ext + layer, z = b
        else
            idx = (ext + layer) + (int64_t)N1 * (b + (int64_t)N1 * a);  // z = ext + layer, x = b
        vol[idx] = value;
    }
}

// Right side at interior point (y, x) of slice z (poisson_cpu.cpp:98-105), FP32
// arithmetic in the reference's order.  g0, g1: (n+1)^3 in the reference layout
// (x fastest).
struct RhsRaw {
    float a, b, c, d;
    // g0, g1 at row y of the slice (wave-uniform), x the lane's column
    __device__ __forceinline__ void load(const float* g0, const float* g1, int x, int n1) {
        a = g0[x];
        b = g0[x + 1];
        c = g1[x];
        d = (g1 + n1)[x];
    }
    __device__ __forceinline__ double value() const { return (double)(((a - b) + c) - d); }
};

// The tables of a solve.  H = He = (M+1)/2 even modes k = 0, 2, ..., Ho = M/2
// odd ones; mode position kp < He is k = 2 kp, else k = 2 (kp - He) + 1.
//   Se[y][ke], So[y][ko] for y < H;
//   G[x][kp]: the multipliers of the elimination along x, g_0 = 1/b, g_x = 1/(b
//   - g_{x-1}) with b = 2 + e[k] = 2 cosh(theta), in closed form sinh((x+1)
//   theta) / sinh((x+2) theta), so that every entry is computed at once;
//   theta = 2 asinh(sin(pi (k+1) / (2 (M+1)))).
__global__ void k_poisson_tables(double* __restrict__ Se, double* __restrict__ So, double* __restrict__ G, int M) {
    const int He = (M + 1) / 2, Ho = M / 2;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= M * M) return;
    const int r = i / M, kp = i - r * M;
    const int k = kp < He ? 2 * kp : 2 * (kp - He) + 1;
    const double h = (double)(M + 1);
    const double th = 2.0 * asinh(sinpi((double)(k + 1) / (2.0 * h)));
    G[i] = exp(-th) * expm1(-2.0 * (r + 1) * th) / expm1(-2.0 * (r + 2) * th);
    if (r < He) {
        // the product reduced mod 2h, so that the argument stays in [0, 2)
        const long long m = ((long long)(r + 1) * (k + 1)) % (2 * (long long)(M + 1));
        const double v = sinpi((double)m / h);
        if (kp < He)
            Se[(int64_t)r * He + kp] = v;
        else
            So[(int64_t)r * Ho + (kp - He)] = v;
    }
}

constexpr int kTile = 64, kTk = 16, kGemmThreads = 256;
typedef double f64x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f64x4_t mfma64(double a, double b, f64x4_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// Both products: a 64 x 64 block tile of the even modes and one of the odd,
// four waves of 32 x 32 of each, i.e. eight v_mfma_f64_16x16x4f64 accumulators
// per wave: A from lane (row lane&15, k lane>>4), B from lane (k lane>>4, column
// lane&15); result register r of a lane holds column lane&15, row 4*r +
// (lane>>4) (unlike the FP32 and BF16 16x16 forms, whose rows are 4*(lane>>4) +
// r).  Steps of 16 terms staged through LDS as [row or column][term], the next
// step's loads in flight during the products.  Product i of a step takes terms
// 4 (lane>>4) + i instead of 4 i + (lane>>4) (the sum is the same): a lane's
// four terms are then neighbours, two 16-byte LDS reads.  Bound by FP64 MFMA.
constexpr int kRow = kTk + 2;  // LDS row stride (doubles), 16-byte aligned rows
typedef double f64x2_t __attribute__((ext_vector_type(2)));
struct PoissonTiles {
    double ae[kTile][kRow], ao[kTile][kRow], be[kTile][kRow], bo[kTile][kRow];
};

__device__ __forceinline__ void poisson_step(const PoissonTiles& t, int wm, int wn, int li, int lk, f64x4_t (&ce)[2][2],
                                             f64x4_t (&co)[2][2]) {
#pragma unroll
    for (int half = 0; half < 2; half++) {
        const int c = 4 * lk + 2 * half;
        f64x2_t ae[2], ao[2], be[2], bo[2];
#pragma unroll
        for (int q = 0; q < 2; q++) {
            ae[q] = *(const f64x2_t*)&t.ae[wm + q * 16 + li][c];
            ao[q] = *(const f64x2_t*)&t.ao[wm + q * 16 + li][c];
            be[q] = *(const f64x2_t*)&t.be[wn + q * 16 + li][c];
            bo[q] = *(const f64x2_t*)&t.bo[wn + q * 16 + li][c];
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int mt = 0; mt < 2; mt++)
#pragma unroll
                for (int nt = 0; nt < 2; nt++) {
                    ce[mt][nt] = mfma64(ae[mt][i], be[nt][i], ce[mt][nt]);
                    co[mt][nt] = mfma64(ao[mt][i], bo[nt][i], co[mt][nt]);
                }
    }
}

// Modes of the right sides: T[z][x][kp] = sum_{y < H} (b(y, x) +- b(M-1-y, x)) S[y][k],
// the right sides formed and folded on the way into LDS.
__global__ void __launch_bounds__(kGemmThreads) k_poisson_modes(const float* __restrict__ g0,
                                                                const float* __restrict__ g1,
                                                                const double* __restrict__ Se,
                                                                const double* __restrict__ So,
                                                                double* __restrict__ T, int M, int z0) {
    __shared__ __align__(16) PoissonTiles t;  // a: [x][y], b: [mode][y]
    const int He = (M + 1) / 2, Ho = M / 2, H = He;
    // rows are staged by wave: their addresses are wave-uniform (scalar) but for the lane's column
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int x0 = blockIdx.x * kTile, k0 = blockIdx.y * kTile;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const int li = lane & 15, lk = lane >> 4;
    const int n1 = M + 3;
    // this thread stages column x0 + lane, rows 4 wave + r of each step (columns
    // past the last repeat it: what they give is not stored)
    const int x = min(x0 + lane, M - 1) + 1, kce = min(k0 + lane, He - 1), kco = min(k0 + lane, max(Ho - 1, 0));
    const int64_t slice = (int64_t)(z0 + blockIdx.z) * n1 * n1;
    RhsRaw lo[4], hi[4];
    double se[4], so[4];
    auto fetch = [&](int y0) {
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int y = y0 + 4 * wave + r;
            lo[r] = hi[r] = RhsRaw{0.f, 0.f, 0.f, 0.f};
            se[r] = so[r] = 0.0;
            if (y < H) {
                const int64_t at = slice + (int64_t)(y + 1) * n1, mirror = slice + (int64_t)(M - y) * n1;
                lo[r].load(g0 + at, g1 + at, x, n1);
                if (y != M - 1 - y) hi[r].load(g0 + mirror, g1 + mirror, x, n1);
                se[r] = (Se + (int64_t)y * He)[kce];
                if (Ho > 0) so[r] = (So + (int64_t)y * Ho)[kco];
            }
        }
    };
    f64x4_t ce[2][2], co[2][2];
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int nt = 0; nt < 2; nt++) ce[mt][nt] = co[mt][nt] = f64x4_t{0.0, 0.0, 0.0, 0.0};
    fetch(0);
    for (int y0 = 0; y0 < H; y0 += kTk) {
        __syncthreads();  // the previous step is done with the tiles
#pragma unroll
        for (int r = 0; r < 4; r += 2) {
            const double u0 = lo[r].value(), v0 = hi[r].value(), u1 = lo[r + 1].value(), v1 = hi[r + 1].value();
            *(f64x2_t*)&t.ae[lane][4 * wave + r] = f64x2_t{u0 + v0, u1 + v1};
            *(f64x2_t*)&t.ao[lane][4 * wave + r] = f64x2_t{u0 - v0, u1 - v1};
            *(f64x2_t*)&t.be[lane][4 * wave + r] = f64x2_t{se[r], se[r + 1]};
            *(f64x2_t*)&t.bo[lane][4 * wave + r] = f64x2_t{so[r], so[r + 1]};
        }
        __syncthreads();
        if (y0 + kTk < H) fetch(y0 + kTk);
        poisson_step(t, wm, wn, li, lk, ce, co);
    }
    double* const Tz = T + (int64_t)blockIdx.z * M * M;
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int xr = x0 + wm + mt * 16 + 4 * r + lk;
            if (xr >= M) continue;
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
                const int c = k0 + wn + nt * 16 + li;
                if (c < He) Tz[(int64_t)xr * M + c] = ce[mt][nt][r];
                if (c < Ho) Tz[(int64_t)xr * M + He + c] = co[mt][nt][r];
            }
        }
}

// Elimination along x, one thread per (slice, mode), in place:
// d_x = (t_x + d_{x-1}) g_x upwards, f_x = d_x + g_x f_{x+1} downwards.  A
// serial chain of two operations per element; the loads of a group of eight
// elements are issued a group ahead.  Bound by HBM (four passes over T).
constexpr int kElimGroup = 8;
__global__ __launch_bounds__(256) void k_poisson_eliminate(double* __restrict__ T, const double* __restrict__ G, int M,
                                                           int slices) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (int64_t)slices * M) return;
    const int kp = (int)(i % M);
    double* const t = T + (i / M) * (int64_t)M * M + kp;
    const double* const g = G + kp;
    double v[kElimGroup], w[kElimGroup], vn[kElimGroup], wn[kElimGroup];
    auto fetch = [&](int first, int dir, double (&a)[kElimGroup], double (&b)[kElimGroup]) {
#pragma unroll
        for (int q = 0; q < kElimGroup; q++) {
            const int x = first + dir * q;
            const bool in = x >= 0 && x < M;
            a[q] = in ? t[(int64_t)x * M] : 0.0;
            b[q] = in ? g[(int64_t)x * M] : 0.0;
        }
    };
    double d = 0.0;
    fetch(0, 1, vn, wn);
    for (int x0 = 0; x0 < M; x0 += kElimGroup) {
#pragma unroll
        for (int q = 0; q < kElimGroup; q++) {
            v[q] = vn[q];
            w[q] = wn[q];
        }
        fetch(x0 + kElimGroup, 1, vn, wn);
#pragma unroll
        for (int q = 0; q < kElimGroup; q++)
            if (x0 + q < M) {
                d = (v[q] + d) * w[q];
                t[(int64_t)(x0 + q) * M] = d;
            }
    }
    double f = 0.0;
    fetch(M - 1, -1, vn, wn);
    for (int x0 = M - 1; x0 >= 0; x0 -= kElimGroup) {
#pragma unroll
        for (int q = 0; q < kElimGroup; q++) {
            v[q] = vn[q];
            w[q] = wn[q];
        }
        fetch(x0 - kElimGroup, -1, vn, wn);
#pragma unroll
        for (int q = 0; q < kElimGroup; q++)
            if (x0 - q >= 0) {
                f = fma(w[q], f, v[q]);
                t[(int64_t)(x0 - q) * M] = f;
            }
    }
}

// Back to space: with P and Q the sums over the even and the odd modes,
// F[y] = P + Q and F[M-1-y] = P - Q (y < H), times 2/(M+1), into the interior of
// the volume (its border: k_poisson_border).
__global__ void __launch_bounds__(kGemmThreads, 3) k_poisson_back(const double* __restrict__ Se,
                                                               const double* __restrict__ So,
                                                               const double* __restrict__ T, float* __restrict__ vol,
                                                               int M, int z0) {
    __shared__ __align__(16) PoissonTiles t;  // a: [y][mode], b: [x][mode]
    const int He = (M + 1) / 2, Ho = M / 2, H = He;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int y0 = blockIdx.y * kTile, x0 = blockIdx.x * kTile;
    const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
    const int li = lane & 15, lk = lane >> 4;
    const double* const Tz = T + (int64_t)blockIdx.z * M * M;
    // this thread stages mode sk, rows sr + 16 r of each step (rows past the last
    // repeat it: what they give is not stored; modes past the last have zero sines)
    const int sk = tid & 15, sr = tid >> 4;
    double ae[4], ao[4], be[4], bo[4];
    auto fetch = [&](int k0) {
        const int k = k0 + sk, ke = min(k, He - 1), ko = min(k, max(Ho - 1, 0));
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int y = min(y0 + sr + 16 * r, H - 1), x = min(x0 + sr + 16 * r, M - 1);
            const double s0 = Se[(unsigned)(y * He + ke)], s1 = Ho > 0 ? So[(unsigned)(y * Ho + ko)] : 0.0;
            ae[r] = k < He ? s0 : 0.0;
            ao[r] = k < Ho ? s1 : 0.0;
            be[r] = Tz[(unsigned)(x * M + ke)];
            bo[r] = Ho > 0 ? Tz[(unsigned)(x * M + He + ko)] : 0.0;
        }
    };
    f64x4_t ce[2][2], co[2][2];
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int nt = 0; nt < 2; nt++) ce[mt][nt] = co[mt][nt] = f64x4_t{0.0, 0.0, 0.0, 0.0};
    fetch(0);
    for (int k0 = 0; k0 < He; k0 += kTk) {
        __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; r++) {
            t.ae[sr + 16 * r][sk] = ae[r];
            t.ao[sr + 16 * r][sk] = ao[r];
            t.be[sr + 16 * r][sk] = be[r];
            t.bo[sr + 16 * r][sk] = bo[r];
        }
        __syncthreads();
        if (k0 + kTk < He) fetch(k0 + kTk);
        poisson_step(t, wm, wn, li, lk, ce, co);
    }
    const int64_t n = M + 2;
    const double scale = 2.0 / (double)(M + 1);
    float* const vz = vol + (int64_t)(z0 + blockIdx.z) * n * n;
#pragma unroll
    for (int mt = 0; mt < 2; mt++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int y = y0 + wm + mt * 16 + 4 * r + lk;
            if (y >= H) continue;
#pragma unroll
            for (int nt = 0; nt < 2; nt++) {
                const int x = x0 + wn + nt * 16 + li;
                if (x >= M) continue;
                const double P = ce[mt][nt][r], Q = co[mt][nt][r];
                vz[(x + 1) + n * (y + 1)] = (float)((P + Q) * scale);
                if (M - 1 - y != y) vz[(x + 1) + n * (M - y)] = (float)((P - Q) * scale);
            }
        }
}

// The slice borders are the identity rows with zero right side: zero.
__global__ void k_poisson_border(float* __restrict__ vol, int n) {
    const int64_t per = 4 * (int64_t)(n - 1), total = per * n;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int64_t z = i / per;
        const int r = (int)(i - z * per), side = r / (n - 1), q = r - side * (n - 1);
        const int x = side == 0 ? q : (side == 1 ? n - 1 : (side == 2 ? n - 1 - q : 0));
        const int y = side == 0 ? 0 : (side == 1 ? q : (side == 2 ? n - 1 : n - 1 - q));
        vol[x + (int64_t)n * (y + (int64_t)n * z)] = 0.0f;
    }
}

inline int grid_1d(int64_t total, int threads) {
    const int64_t g = (total + threads - 1) / threads;
    return (int)(g < 65536 ? (g > 0 ? g : 1) : 65536);
}

}  // namespace

hipError_t launch_scale_views(const float* src, float* dst, const float* coef, int64_t len_view, int n_views,
                              hipStream_t stream) {
    const int64_t total = len_view * n_views;
    if (total <= 0) return hipSuccess;
    hipLaunchKernelGGL(k_scale_views, dim3(grid_1d(total, 256)), dim3(256), 0, stream, src, dst, coef, len_view,
                       total);
    return hipGetLastError();
}

hipError_t launch_grad_faces(float* vol, int N1, int ext, float value, hipStream_t stream) {
    if (ext >= N1) return hipSuccess;
    const int64_t total = 2 * (int64_t)(N1 - ext) * N1 * N1;
    hipLaunchKernelGGL(k_grad_faces, dim3(grid_1d(total, 256)), dim3(256), 0, stream, vol, N1, ext, value);
    return hipGetLastError();
}

hipError_t launch_poisson_tables(double* Se, double* So, double* G, int n, hipStream_t stream) {
    const int M = n - 2;
    hipLaunchKernelGGL(k_poisson_tables, dim3((unsigned)(((int64_t)M * M + 255) / 256)), dim3(256), 0, stream, Se, So,
                       G, M);
    return hipGetLastError();
}

// Slices z0 .. z0 + slices - 1 of vol; T: slices x M x M doubles.
hipError_t launch_poisson_slices(const float* g0, const float* g1, const double* Se, const double* So, const double* G,
                                 double* T, float* vol, int n, int z0, int slices, hipStream_t stream) {
    const int M = n - 2, H = (M + 1) / 2;
    const dim3 block(kGemmThreads), grid((M + kTile - 1) / kTile, (H + kTile - 1) / kTile, slices);
    hipLaunchKernelGGL(k_poisson_modes, grid, block, 0, stream, g0, g1, Se, So, T, M, z0);
    hipLaunchKernelGGL(k_poisson_eliminate, dim3((unsigned)(((int64_t)slices * M + 255) / 256)), dim3(256), 0, stream, T,
                       G, M, slices);
    hipLaunchKernelGGL(k_poisson_back, grid, block, 0, stream, Se, So, T, vol, M, z0);
    return hipGetLastError();
}

hipError_t launch_poisson_border(float* vol, int n, hipStream_t stream) {
    hipLaunchKernelGGL(k_poisson_border, dim3(grid_1d(4 * (int64_t)(n - 1) * n, 256)), dim3(256), 0, stream, vol, n);
    return hipGetLastError();
}

}  // namespace xr
