// HIP kernels (gfx950) of the learned warm start: a 3-level 3-D U-Net on
// channels-last BF16 activations with FP32 accumulation.  No counterpart in
// the reference (it has no learned component).
//
// Activations: act[v * ld + off + c], v = voxel index of the column layout
// (z fastest: v = z + N*(x + N*y)), c < C, BF16.  A tensor can be a channel
// slice (off, ld) of a wider buffer, which is how skip connections are
// concatenated without copies.
//
// 3x3x3 convolution, stride 1, zero padding 1, as an implicit GEMM on MFMA
// (v_mfma_f32_16x16x32_bf16): M = voxels, N = output channels, K = 27*Cin with
// k = tap*Cin + ci, tap = (d0+1)*9 + (d1+1)*3 + (d2+1).  Cin is a multiple of
// 8 so the 8 consecutive k of one MFMA lane lie in one tap: one 16-byte load
// of 8 channels of one neighbour voxel.  Weights are [Cout16][Kpad] BF16, zero
// padded, in the order in which a wave reads them (weight_index): each MFMA
// operand is one contiguous KB.  The data gradient is the same kernel on the output
// gradient with mirrored taps and transposed channels (weights [Cin16][K'pad],
// k' = (26 - tap)*Cout + co); the weight gradient contracts over voxels with
// both operands read transposed from LDS.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "xr_unet_internal.hpp"

namespace xr {
namespace nn {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) bf16x8 lds_bf16x8;
typedef __attribute__((address_space(3))) __bf16 lds_bf16;

__device__ __forceinline__ f32x4 mfma(const bf16x8& a, const bf16x8& b, const f32x4& c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ bf16x8 zero8() {
    bf16x8 z;
#pragma unroll
    for (int j = 0; j < 8; j++) z[j] = (__bf16)0.0f;
    return z;
}

// Packed position of weight (co, k): operand (k / 32, co / 16) of cout16 / 16 per
// step, lane (k % 32 / 8) * 16 + co % 16, element k % 8.
__device__ __forceinline__ int64_t weight_index(int co, int k, int cout16) {
    return ((int64_t)(k >> 5) * (cout16 >> 4) + (co >> 4)) * 512 + ((k & 31) >> 3) * 128 + (co & 15) * 8 + (k & 7);
}

// 16 bytes per lane from global memory straight to LDS: lane l's go to lds + 16 l.
// The caller waits (lds_wait) before the barrier that publishes them.
typedef __attribute__((address_space(3))) void lds_void;
typedef __attribute__((address_space(1))) void global_void;
__device__ __align__(16) __bf16 g_zero8[8];  // source of the padding

__device__ __forceinline__ void lds_load16(const __bf16* src, lds_bf16x8* lds) {
    __builtin_amdgcn_global_load_lds((global_void*)src, (lds_void*)lds, 16, 0, 0);
}

__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// Tap t -> offsets (d0, d1, d2) in {-1, 0, 1}.
__device__ __forceinline__ void tap_offsets(int t, int& d0, int& d1, int& d2) {
    d0 = t / 9 - 1;
    d1 = (t / 3) % 3 - 1;
    d2 = t % 3 - 1;
}

// ---------------------------------------------------------------------------
// Data-gradient convolution, and the forward one for dims that the chunked
// kernel below does not take.  K runs in the order k = tap*Cin + ci, so every
// channel of the input halo is staged in LDS before the first step and read by
// all 27 taps; the four lane groups of a step look up their (tap, chunk of 8
// channels) in a table of LDS offsets.  Block: 4 waves with MT 16-voxel MFMA
// tiles each: 2 x 4 x 32, 2 x 4 x 16 or 2 x 2 x 16 voxels (MT = 4, 2, 1; the last
// ones reach past the volume), the largest whose halo leaves room for two blocks
// per CU.  blockIdx.y: pieces of NT 16-channel tiles of the output.
// Bound by the LDS reads and, at the start of a block, the staging (the other
// blocks of the CU hide part of it); the weights are prefetched one step ahead.
// Measured: 24 -> 72 channels at 96^3 335 -> 245 us, 48 -> 144 at 48^3 246 -> 158,
// 48 -> 48 at 48^3 94 -> 58, 96 -> 96 at 24^3 116 -> 62, against loading every
// operand from global memory (one 16-byte load per lane, tap and 8 channels);
// weights as plain rows instead of whole operands: 346 us for the first.
// ---------------------------------------------------------------------------
// Volumes of at most 8 or 4 layers take MFMA tiles of W = 8 or 4 layers by 2 or 4
// columns of D1 (256 x 256 x 4, 24 channels, inference: 1203 -> 336 us).
template <int MT, int W>
struct ConvTile {
    static constexpr int T0 = 2, T1 = W < 16 ? 32 * MT / W : (MT == 1 ? 2 : 4), T2 = W < 16 ? W : (MT == 4 ? 32 : 16);
    static constexpr int R = 16 / W;  // columns of D1 per MFMA tile
    static constexpr int H1 = T1 + 2, H2 = T2 + 2, halo = (T0 + 2) * H1 * H2;
    static constexpr int stride = halo + 4;  // LDS distance of two chunks, 16-byte units
    static constexpr int64_t lds(int nchunk) { return 16 * (int64_t)stride * nchunk + 4 * 28 * nchunk; }
};

template <int MT, int NT, int W>
__global__ __launch_bounds__(256, 2) void k_conv3(const ConvArgs a) {
    using T = ConvTile<MT, W>;
    extern __shared__ bf16x8 conv_lds[];
    const int nch = a.Cin / 8, nq = 27 * nch;
    bf16x8* const halo = conv_lds;
    int* const off = (int*)(conv_lds + T::stride * nch);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, kg = lane >> 4;
    const int nb2 = (a.D2 + T::T2 - 1) / T::T2, nb1 = (a.D1 + T::T1 - 1) / T::T1;
    const int o2 = blockIdx.x % nb2 * T::T2, o1 = blockIdx.x / nb2 % nb1 * T::T1, o0 = blockIdx.x / (nb2 * nb1) * T::T0;
    const int co0 = blockIdx.y * (16 * NT), tiles = (a.Cout + 15) / 16;
    for (int q = threadIdx.x; q < nq; q += 256) {
        const int tap = q / nch;
        off[q] = (q - tap * nch) * T::stride + (tap / 9 * T::H1 + tap / 3 % 3) * T::H2 + tap % 3;
    }
    for (int v0 = 0; v0 < T::halo; v0 += 256) {
        const int v = v0 + threadIdx.x;
        const int g0 = o0 + v / (T::H2 * T::H1) - 1, g1 = o1 + v / T::H2 % T::H1 - 1, g2 = o2 + v % T::H2 - 1;
        const bool ok = (unsigned)g0 < (unsigned)a.D0 && (unsigned)g1 < (unsigned)a.D1 && (unsigned)g2 < (unsigned)a.D2;
        const __bf16* const src =
            ok ? a.in + (((int64_t)g0 * a.D1 + g1) * a.D2 + g2) * a.in_ld + a.in_off : g_zero8;
        const int step = ok ? 8 : 0;
        if (v < T::halo)
            for (int c = 0; c < nch; c++)
                lds_load16(src + step * c, (lds_bf16x8*)halo + c * T::stride + v0 + 64 * wave);
    }
    lds_wait();
    __syncthreads();
    const lds_bf16x8* base[MT];
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const int g = (wave * MT + m) / (T::T2 / W), half = (wave * MT + m) % (T::T2 / W);
        const int q0 = g / (T::T1 / T::R), q1 = g % (T::T1 / T::R) * T::R + row / W;
        base[m] = (const lds_bf16x8*)halo + (q0 * T::H1 + q1) * T::H2 + W * half + row % W;
    }
    const __bf16* wop[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) wop[nt] = a.w + min((int)blockIdx.y * NT + nt, tiles - 1) * 512 + lane * 8;
    f32x4 acc[MT][NT];
    bf16x8 B[NT];
#pragma unroll
    for (int nt = 0; nt < NT; nt++) {
#pragma unroll
        for (int m = 0; m < MT; m++) acc[m][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
        B[nt] = *(const bf16x8*)wop[nt];
    }
    // one step ahead: the weights and the halo values; two: the LDS offsets
    const int last = a.Kpad - 32;
    bf16x8 A[MT];
    int o = off[min(kg, nq - 1)];
#pragma unroll
    for (int m = 0; m < MT; m++) A[m] = kg < nq ? base[m][o] : zero8();
    o = off[min(4 + kg, nq - 1)];
    for (int kc = 0; kc <= last; kc += 32) {
        bf16x8 nextB[NT], nextA[MT];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) nextB[nt] = *(const bf16x8*)(wop[nt] + min(kc + 32, last) * 16 * tiles);
        const int q = kc / 8 + 4 + kg;
#pragma unroll
        for (int m = 0; m < MT; m++) nextA[m] = q < nq ? base[m][o] : zero8();
        o = off[min(q + 4, nq - 1)];
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
#pragma unroll
            for (int m = 0; m < MT; m++) acc[m][nt] = mfma(A[m], B[nt], acc[m][nt]);
            B[nt] = nextB[nt];
        }
#pragma unroll
        for (int m = 0; m < MT; m++) A[m] = nextA[m];
    }
    // D layout of the 16x16 MFMA: lane holds column (lane & 15), rows 4*kg + i.
#pragma unroll
    for (int m = 0; m < MT; m++) {
        const int g = (wave * MT + m) / (T::T2 / W), half = (wave * MT + m) % (T::T2 / W);
        const int v0 = o0 + g / (T::T1 / T::R), v1 = o1 + g % (T::T1 / T::R) * T::R + 4 * kg / W;
        if (v0 >= a.D0 || v1 >= a.D1) continue;
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const int co = co0 + nt * 16 + row;
            if (co >= a.Cout) continue;
            const float b = a.bias ? a.bias[co] : 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int v2 = o2 + W * half + 4 * kg % W + i;
                if (v2 >= a.D2) continue;
                const int64_t v = ((int64_t)v0 * a.D1 + v1) * a.D2 + v2;
                float val = acc[m][nt][i] + b;
                if (a.relu) val = fmaxf(val, 0.f);
                if (a.mask && !((float)a.mask[v * a.mask_ld + a.mask_off + co] > 0.f)) val = 0.f;
                __bf16* o = a.out + v * a.out_ld + a.out_off + co;
                if (a.accumulate) val += (float)*o;
                *o = (__bf16)val;
            }
        }
    }
}

// ---------------------------------------------------------------------------
// Forward convolution, LDS-tiled.  Block: 4 waves, an output tile of
// 2 (D0) x 4 (D1) x 32 (D2) voxels; wave w owns D0 row w/2, D1 columns
// 2(w%2) and 2(w%2)+1, and both 16-voxel halves of D2: four 16-row MFMA
// tiles.  K runs over chunks of 8 input channels; for each chunk the input
// halo (4 x 6 x 34 voxels x 8 channels, 13 KB) is staged in LDS once and read
// by all 27 taps, instead of one global load per tap.  K within a chunk:
// k = tap*8 + c, 28 taps with the last one zero (7 MFMA steps of 32: lane
// group kg takes tap 4s + kg).
// ---------------------------------------------------------------------------
constexpr int kCT0 = 2, kCT1 = 4, kCT2 = 32;
constexpr int kCH0 = kCT0 + 2, kCH1 = kCT1 + 2, kCH2 = kCT2 + 2;
constexpr int kCHalo = kCH0 * kCH1 * kCH2;
constexpr int kTapsPad = 28;

// CPS: input-channel chunks staged per barrier, up to three: they go from global
// memory straight to LDS and are waited for there, so few stages of long loads
// are better than many short ones (24 -> 24 channels at 128^3: three chunks 125,
// one 150 us), and the 16-byte pieces of a voxel record are fetched while its
// cache line is resident.  Staging through registers a stage ahead took 48 of
// them and did not overlap: the weights' loads, issued later, return in order.
// Bound by LDS reads (narrow outputs) and the stage's latency, hidden by three or
// four blocks per CU.  Measured at 128^3, 72 -> 24 channels with fused upsampling:
// 421 (row-major weights) -> 457 (packed) -> 258 us.
// UP: the first a.up_chunks chunks come from the half-resolution tensor a.up
// at the halo voxel's parent (nearest x2 upsampling), the rest from a.in, so
// the decoder's concatenation is never written; the halo in LDS, and hence
// the result, is the same as with the concatenation materialised.
template <int NT, int CPS, bool UP>
__global__ __launch_bounds__(256) void k_conv3_tiled(const ConvArgs a) {
    __shared__ bf16x8 halo[CPS * kCHalo];
    const lds_bf16x8* const hl = (const lds_bf16x8*)halo;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int row = lane & 15, kg = lane >> 4;
    const int nb2 = a.D2 / kCT2, nb1 = a.D1 / kCT1;
    const int b2 = blockIdx.x % nb2, b1 = (blockIdx.x / nb2) % nb1, b0 = blockIdx.x / (nb2 * nb1);
    const int o0 = b0 * kCT0, o1 = b1 * kCT1, o2 = b2 * kCT2;
    // halo coordinates (+1) of this lane's output voxels: tile m = 2*(x half) + (z half)
    const int h0 = (wave >> 1) + 1;
    int h1[4], h2[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
        h1[m] = 2 * (wave & 1) + (m >> 1) + 1;
        h2[m] = 16 * (m & 1) + row + 1;
    }
    f32x4 acc[4][NT];
#pragma unroll
    for (int m = 0; m < 4; m++)
#pragma unroll
        for (int nt = 0; nt < NT; nt++) acc[m][nt] = f32x4{0.f, 0.f, 0.f, 0.f};
    const __bf16* __restrict__ in = a.in + a.in_off;
    const int nchunk = a.Cin / 8;
    // halo voxels of this thread: i = threadIdx.x + 256 j; their sources (outside the
    // volume: zeros, for every chunk) are the same records for every chunk
    constexpr int kPer = (kCHalo + 255) / 256;
    const __bf16* hsrc[kPer];
    const __bf16* usrc[kPer];
    int hstep[kPer];
#pragma unroll
    for (int j = 0; j < kPer; j++) {
        const int i = threadIdx.x + 256 * j;
        const int q2 = i % kCH2, q1 = (i / kCH2) % kCH1, q0 = i / (kCH2 * kCH1);
        const int g0 = o0 + q0 - 1, g1 = o1 + q1 - 1, g2 = o2 + q2 - 1;
        const bool ok = (unsigned)g0 < (unsigned)a.D0 && (unsigned)g1 < (unsigned)a.D1 && (unsigned)g2 < (unsigned)a.D2;
        hstep[j] = ok ? 8 : 0;
        hsrc[j] = ok ? in + (((int64_t)g0 * a.D1 + g1) * a.D2 + g2) * a.in_ld : g_zero8;
        if (UP)
            usrc[j] = ok ? a.up + a.up_off +
                               (((int64_t)(g0 >> 1) * (a.D1 >> 1) + (g1 >> 1)) * (a.D2 >> 1) + (g2 >> 1)) * a.up_ld
                         : g_zero8;
    }
    const int up_chunks = UP ? a.up_chunks : 0;
    // stage st holds chunks st*CPS .. st*CPS + CPS-1
    auto stage = [&](int st) {
#pragma unroll
        for (int c = 0; c < CPS; c++) {
            const int cc = st * CPS + c;
            if (cc >= nchunk) break;
#pragma unroll
            for (int j = 0; j < kPer; j++) {
                const __bf16* const src =
                    (UP && cc < up_chunks) ? usrc[j] + cc * hstep[j] : hsrc[j] + (cc - up_chunks) * hstep[j];
                if (256 * j + 255 < kCHalo || threadIdx.x + 256 * j < kCHalo)
                    lds_load16(src, (lds_bf16x8*)halo + c * kCHalo + 256 * j + 64 * wave);
            }
        }
        lds_wait();
    };
    const int nstage = (nchunk + CPS - 1) / CPS;
    for (int st = 0; st < nstage; st++) {
        __syncthreads();  // the previous stage's reads are done
        stage(st);
        __syncthreads();
#pragma unroll 1
        for (int c = 0; c < CPS; c++) {
            const int cc = st * CPS + c;
            if (cc >= nchunk) break;
            const __bf16* __restrict__ wc = a.wt + (int64_t)cc * (kTapsPad / 4 * NT * 512) + lane * 8;
            const lds_bf16x8* const hc = hl + c * kCHalo;
#pragma unroll
            for (int s = 0; s < kTapsPad / 4; s++) {
                const int tap = 4 * s + kg;
                int d0, d1, d2;
                tap_offsets(min(tap, 26), d0, d1, d2);  // tap 27 has zero weights
                bf16x8 A[4];
#pragma unroll
                for (int m = 0; m < 4; m++) A[m] = hc[((h0 + d0) * kCH1 + h1[m] + d1) * kCH2 + h2[m] + d2];
#pragma unroll
                for (int nt = 0; nt < NT; nt++) {
                    const bf16x8 B = *(const bf16x8*)(wc + (s * NT + nt) * 512);
#pragma unroll
                    for (int m = 0; m < 4; m++) acc[m][nt] = mfma(A[m], B, acc[m][nt]);
                }
            }
        }
    }
    // D layout of the 16x16 MFMA: lane holds column (lane & 15), rows 4*kg + i.
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const int64_t vrow = ((int64_t)(o0 + h0 - 1) * a.D1 + (o1 + h1[m] - 1)) * a.D2 + o2 + 16 * (m & 1);
#pragma unroll
        for (int nt = 0; nt < NT; nt++) {
            const int co = nt * 16 + row;
            if (co >= a.Cout) continue;
            const float b = a.bias ? a.bias[co] : 0.f;
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int64_t v = vrow + 4 * kg + i;
                float val = acc[m][nt][i] + b;
                if (a.relu) val = fmaxf(val, 0.f);
                if (a.mask && !((float)a.mask[v * a.mask_ld + a.mask_off + co] > 0.f)) val = 0.f;
                __bf16* o = a.out + v * a.out_ld + a.out_off + co;
                if (a.accumulate) val += (float)*o;
                *o = (__bf16)val;
            }
        }
    }
}

// Master FP32 weights [Cout][27][Cin] -> tiled-order BF16 [Cout16][Ktpad].
__global__ void k_pack_tiled(const float* __restrict__ W, int Cin, int Cout, __bf16* wt, int Ktpad, int cout16) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)cout16 * Ktpad) return;
    const int co = (int)(i / Ktpad), k = (int)(i % Ktpad);
    const int cc = k / (kTapsPad * 8), tap = (k / 8) % kTapsPad, c = k % 8;
    const int ci = cc * 8 + c;
    wt[weight_index(co, k, cout16)] = (__bf16)((co < Cout && tap < 27 && ci < Cin) ? W[((int64_t)co * 27 + tap) * Cin + ci] : 0.f);
}

// ---------------------------------------------------------------------------
// Weight and bias gradient: dw[co][tap][ci] += sum_v gout[v][co] in[v + tap][ci],
// db[co] += sum_v gout[v][co].  A contraction over voxels: both MFMA operands
// need 8 consecutive voxels of one channel per lane, while the tensors (and
// their LDS copies) are channels-last.  The transposed LDS read
// ds_read_b64_tr_b16 gives them: of the 4 voxels x 16 channels that 16 lanes
// point at, lane l receives channel l of the 4 voxels.  A tap is an offset of
// the row address.
// Block: 4 waves, 32 output x 32 input channels (blockIdx.y), tiles of 2 (D0) x
// 4 (D1) x 32 (D2) voxels, a stride of gridDim.x tiles; a tile's input halo (4
// x 6 x 34 voxels) and output gradient are staged once for all 27 taps.  Wave w
// accumulates taps 7 w .. 7 w + 6 (2 x 2 tiles each) over all its tiles; the
// 28th tap is a row of ones, whose sums are the bias gradient.  Partial sums are
// added with FP32 atomics (their order is not fixed).
// Bound by LDS reads (one b64 per MFMA) and staging, which goes from global
// memory straight to LDS (through registers, with a branch per load: twice the
// time).  Measured: 72 -> 24 channels at 96^3 1340 + 185 (bias) -> 296 us, 144 ->
// 48 at 48^3 398 + 20 -> 142, against a block per output tile that built both
// transposed operands in LDS for every tap.
// ---------------------------------------------------------------------------
constexpr int kWgCh = 32;  // channels per block, both sides; LDS row of one voxel
constexpr int kWgTaps = 7;  // per wave
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// LDS voxel records of 4 16-byte pieces; the halves of a record are swapped for
// odd groups of 8 voxels, so that the 32 lanes of one read (4 voxels of each of
// two groups) cover all banks.
__device__ __forceinline__ int wg_piece(int v, int piece) { return piece ^ ((v >> 2) & 2); }

// Eight consecutive voxels of channel 16 half + (lane & 15), for the lane's
// voxel group 8 (lane >> 4) from voxel v0 on; lv, lc: lane's part of the address.
__device__ __forceinline__ bf16x8 voxels8(const lds_bf16* p, int v, int half, int lc) {
    const lds_bf16* const q0 = p + v * kWgCh + ((((v >> 3) & 1) ^ half) << 4) + lc;
    const lds_bf16* const q1 = p + (v + 4) * kWgCh + (((((v + 4) >> 3) & 1) ^ half) << 4) + lc;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)q0);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)q1);
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// One tile: taps of this wave over its 8 rows of 32 voxels; NM x NN used 16-channel tiles.
template <int NM, int NN>
__device__ __forceinline__ void wgrad_tile(f32x4 (&acc)[kWgTaps][2][2], const lds_bf16* halo, const lds_bf16* grad,
                                           int wave, int lane) {
    const int li = lane & 15, lv = 8 * (lane >> 4) + (li >> 2), lc = 4 * (li & 3);
    bf16x8 ones;
#pragma unroll
    for (int j = 0; j < 8; j++) ones[j] = (__bf16)1.0f;
#pragma unroll 1
    for (int r = 0; r < kCT0 * kCT1; r++) {
        bf16x8 A[NM];
#pragma unroll
        for (int m = 0; m < NM; m++) A[m] = voxels8(grad, r * kCT2 + lv, m, lc);
        const int h = (r / kCT1 * kCH1 + r % kCT1) * kCH2 + lv;
#pragma unroll
        for (int t = 0; t < kWgTaps; t++) {
            const int tap = min(kWgTaps * wave + t, 26);
            const int v = h + (tap / 9 * kCH1 + tap / 3 % 3) * kCH2 + tap % 3;
#pragma unroll
            for (int n = 0; n < NN; n++) {
                bf16x8 B = voxels8(halo, v, n, lc);
                if (n == 0 && t == kWgTaps - 1) B = wave == 3 ? ones : B;
#pragma unroll
                for (int m = 0; m < NM; m++) acc[t][m][n] = mfma(A[m], B, acc[t][m][n]);
            }
        }
    }
}

__global__ __launch_bounds__(256, 2) void k_conv3_wgrad(const WgradArgs a) {
    __shared__ __align__(16) __bf16 halo[kCHalo * kWgCh];
    __shared__ __align__(16) __bf16 grad[kCT0 * kCT1 * kCT2 * kWgCh];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nci = (a.Cin + kWgCh - 1) / kWgCh;
    const int ci0 = (blockIdx.y % nci) * kWgCh, co0 = (blockIdx.y / nci) * kWgCh;
    const int n1 = (a.D1 + kCT1 - 1) / kCT1, n2 = (a.D2 + kCT2 - 1) / kCT2;
    const int tiles = (a.D0 + kCT0 - 1) / kCT0 * n1 * n2;
    const bool two_ci = ci0 + 16 < a.Cin, two_co = co0 + 16 < a.Cout;
    f32x4 acc[kWgTaps][2][2];
#pragma unroll
    for (int t = 0; t < kWgTaps; t++)
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int n = 0; n < 2; n++) acc[t][m][n] = f32x4{0.f, 0.f, 0.f, 0.f};
    const lds_bf16* const hl = (const lds_bf16*)halo;
    const lds_bf16* const gl = (const lds_bf16*)grad;
    for (int tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const int o2 = tile % n2 * kCT2, o1 = tile / n2 % n1 * kCT1, o0 = tile / (n2 * n1) * kCT0;
        __syncthreads();  // the previous tile's reads are done
        // four pieces of 8 channels per voxel; zero outside the volume and past the channels
        for (int i0 = 0; i0 < kCHalo * 4; i0 += 256) {
            const int i = i0 + threadIdx.x, v = i >> 2, c = ci0 + 8 * wg_piece(v, i & 3);
            const int g0 = o0 + v / (kCH2 * kCH1) - 1, g1 = o1 + v / kCH2 % kCH1 - 1, g2 = o2 + v % kCH2 - 1;
            const bool ok = c < a.Cin && (unsigned)g0 < (unsigned)a.D0 && (unsigned)g1 < (unsigned)a.D1 &&
                            (unsigned)g2 < (unsigned)a.D2;
            const __bf16* const src =
                ok ? a.in + (((int64_t)g0 * a.D1 + g1) * a.D2 + g2) * a.in_ld + a.in_off + c : g_zero8;
            if (i < kCHalo * 4) lds_load16(src, (lds_bf16x8*)halo + i0 + 64 * wave);
        }
#pragma unroll
        for (int i0 = 0; i0 < kCT0 * kCT1 * kCT2 * 4; i0 += 256) {
            const int i = i0 + threadIdx.x, v = i >> 2, c = co0 + 8 * wg_piece(v, i & 3);
            const int g0 = o0 + v / (kCT2 * kCT1), g1 = o1 + v / kCT2 % kCT1, g2 = o2 + v % kCT2;
            const bool ok = c < a.Cout && g0 < a.D0 && g1 < a.D1 && g2 < a.D2;
            const __bf16* const src =
                ok ? a.gout + (((int64_t)g0 * a.D1 + g1) * a.D2 + g2) * a.g_ld + a.g_off + c : g_zero8;
            lds_load16(src, (lds_bf16x8*)grad + i0 + 64 * wave);
        }
        lds_wait();
        __syncthreads();
        if (two_ci) {
            if (two_co) wgrad_tile<2, 2>(acc, hl, gl, wave, lane);
            else wgrad_tile<1, 2>(acc, hl, gl, wave, lane);
        } else {
            if (two_co) wgrad_tile<2, 1>(acc, hl, gl, wave, lane);
            else wgrad_tile<1, 1>(acc, hl, gl, wave, lane);
        }
    }
    // D layout of the 16x16 MFMA: lane holds column (lane & 15), rows 4*kg + i
    const int li = lane & 15, kg = lane >> 4;
#pragma unroll
    for (int t = 0; t < kWgTaps; t++) {
        const int tap = kWgTaps * wave + t;
#pragma unroll
        for (int m = 0; m < 2; m++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int co = co0 + m * 16 + 4 * kg + i;
                if (co >= a.Cout) continue;
                if (tap < 27) {
#pragma unroll
                    for (int n = 0; n < 2; n++) {
                        const int ci = ci0 + n * 16 + li;
                        if (ci < a.Cin) atomicAdd(a.dw + (int64_t)co * a.ldw + tap * a.Cin + ci, acc[t][m][n][i]);
                    }
                } else if (ci0 == 0 && li == 0) {
                    atomicAdd(a.db + co, acc[t][m][0][i]);
                }
            }
    }
}

// 2x2x2 average pooling: out[p][c] = mean of the 8 children (dims halve).
// Index arithmetic of the elementwise kernels below: 32-bit (I = unsigned)
// when the launch's element count fits, 64-bit otherwise (64-bit division is
// several times the cost and these kernels are otherwise pure data movement).
template <class I>
__global__ void k_pool(const __bf16* __restrict__ in, int in_ld, int in_off, int C, int D0, int D1, int D2,
                       __bf16* __restrict__ out) {
    const int H0 = D0 / 2, H1 = D1 / 2, H2 = D2 / 2;
    const int G = C / 8;
    const I i = (I)blockIdx.x * blockDim.x + threadIdx.x;
    const I n = (I)H0 * H1 * H2 * G;
    if (i >= n) return;
    const int g = (int)(i % G);
    const int64_t p = i / G;
    const int q2 = (int)((I)p % H2), q1 = (int)(((I)p / H2) % H1), q0 = (int)((I)p / ((I)H2 * H1));
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int c = 0; c < 8; c++) {
        const int64_t v = ((int64_t)(2 * q0 + (c >> 2)) * D1 + (2 * q1 + ((c >> 1) & 1))) * D2 + (2 * q2 + (c & 1));
        const bf16x8 x = *(const bf16x8*)(in + v * in_ld + in_off + 8 * g);
#pragma unroll
        for (int j = 0; j < 8; j++) s[j] += (float)x[j];
    }
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = (__bf16)(0.125f * s[j]);
    *(bf16x8*)(out + p * C + 8 * g) = o;
}

// Pooling backward into a (masked) slice: gin[child][c] (+)= gp[p][c]/8 * (mask[child][c] > 0).
template <class I>
__global__ void k_pool_bwd(const __bf16* __restrict__ gp, int C, int D0, int D1, int D2, __bf16* gin, int g_ld,
                           int g_off, const __bf16* __restrict__ mask, int m_ld, int m_off, int accumulate) {
    const int G = C / 8;
    const I i = (I)blockIdx.x * blockDim.x + threadIdx.x;
    const I n = (I)D0 * D1 * D2 * G;
    if (i >= n) return;
    const int g = (int)(i % G);
    const int64_t v = i / G;
    const int p2 = (int)((I)v % D2), p1 = (int)(((I)v / D2) % D1), p0 = (int)((I)v / ((I)D2 * D1));
    const int64_t p = ((int64_t)(p0 / 2) * (D1 / 2) + p1 / 2) * (D2 / 2) + p2 / 2;
    const bf16x8 x = *(const bf16x8*)(gp + p * C + 8 * g);
    const bf16x8 m = *(const bf16x8*)(mask + v * m_ld + m_off + 8 * g);
    bf16x8* o = (bf16x8*)(gin + v * g_ld + g_off + 8 * g);
    bf16x8 old = accumulate ? *o : zero8();
    bf16x8 r;
#pragma unroll
    for (int j = 0; j < 8; j++) {
        float val = ((float)m[j] > 0.f) ? 0.125f * (float)x[j] : 0.f;
        if (accumulate) val += (float)old[j];
        r[j] = (__bf16)val;
    }
    *o = r;
}

// Nearest-neighbour upsampling x2 into a channel slice: out[child][off + c] = low[parent][c].
template <class I>
__global__ void k_upsample(const __bf16* __restrict__ low, int C, int D0, int D1, int D2, __bf16* out, int o_ld,
                           int o_off) {
    const int G = C / 8;
    const I i = (I)blockIdx.x * blockDim.x + threadIdx.x;
    const I n = (I)D0 * D1 * D2 * G;
    if (i >= n) return;
    const int g = (int)(i % G);
    const int64_t v = i / G;
    const int p2 = (int)((I)v % D2), p1 = (int)(((I)v / D2) % D1), p0 = (int)((I)v / ((I)D2 * D1));
    const int64_t p = ((int64_t)(p0 / 2) * (D1 / 2) + p1 / 2) * (D2 / 2) + p2 / 2;
    *(bf16x8*)(out + v * o_ld + o_off + 8 * g) = *(const bf16x8*)(low + p * C + 8 * g);
}

// Upsampling backward: glow[p][c] = sum of the 8 children's g[child][off + c].
template <class I>
__global__ void k_upsample_bwd(const __bf16* __restrict__ g, int g_ld, int g_off, int C, int D0, int D1, int D2,
                               __bf16* __restrict__ glow) {
    const int H0 = D0 / 2, H1 = D1 / 2, H2 = D2 / 2;
    const int G = C / 8;
    const I i = (I)blockIdx.x * blockDim.x + threadIdx.x;
    const I n = (I)H0 * H1 * H2 * G;
    if (i >= n) return;
    const int gg = (int)(i % G);
    const int64_t p = i / G;
    const int q2 = (int)((I)p % H2), q1 = (int)(((I)p / H2) % H1), q0 = (int)((I)p / ((I)H2 * H1));
    float s[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int c = 0; c < 8; c++) {
        const int64_t v = ((int64_t)(2 * q0 + (c >> 2)) * D1 + (2 * q1 + ((c >> 1) & 1))) * D2 + (2 * q2 + (c & 1));
        const bf16x8 x = *(const bf16x8*)(g + v * g_ld + g_off + 8 * gg);
#pragma unroll
        for (int j = 0; j < 8; j++) s[j] += (float)x[j];
    }
    bf16x8 o;
#pragma unroll
    for (int j = 0; j < 8; j++) o[j] = (__bf16)s[j];
    *(bf16x8*)(glow + p * C + 8 * gg) = o;
}

// Network input: x8[v] = (bf16(x[v] * inv_scale), 0, ..., 0).
__global__ void k_input8(const float* __restrict__ x, int64_t V, float inv_scale, __bf16* __restrict__ x8) {
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    bf16x8 o = zero8();
    o[0] = (__bf16)(x[v] * inv_scale);
    *(bf16x8*)(x8 + v * 8) = o;
}

// Sum of l over a block of 256 threads, added to *out by one atomic (FP64 atomics
// to one address serialise: one per wave of a 128^3 volume took 100 us).
__device__ __forceinline__ void block_add(double l, double* out) {
    __shared__ double part[4];
    for (int off = 32; off > 0; off >>= 1) l += __shfl_xor(l, off);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(out, (part[0] + part[1]) + (part[2] + part[3]));
}

// Output head (1x1x1 conv, C -> 1) with the residual: y = x + scale*(w.e[v] + b),
// w[C] = b.  Loss mode (t != null): r = (x/scale + w.e + b) - t/scale,
// loss += r^2, g[v] = 2 r / V (normalised units).
template <int C>
__global__ __launch_bounds__(256) void k_head(const __bf16* __restrict__ e, int64_t V, const float* __restrict__ w,
                                              const float* __restrict__ x, float scale, float* __restrict__ y,
                                              const float* __restrict__ t, float* g, double* loss) {
    double l = 0.0;
    for (int64_t v = (int64_t)blockIdx.x * 256 + threadIdx.x; v < V; v += (int64_t)gridDim.x * 256) {
        float f = w[C];
#pragma unroll
        for (int c = 0; c < C; c += 8) {
            const bf16x8 a = *(const bf16x8*)(e + v * C + c);
#pragma unroll
            for (int j = 0; j < 8; j++) f = fmaf(w[c + j], (float)a[j], f);
        }
        const float inv = 1.0f / scale;
        if (y) y[v] = x[v] + scale * f;
        if (t) {
            const float r = (x[v] * inv + f) - t[v] * inv;
            l += (double)r * (double)r;
            g[v] = 2.0f * r / (float)V;
        }
    }
    if (loss) block_add(l, loss);
}

// Head backward: ge[v][c] = g[v] w[c] (e[v][c] > 0); dw[c] += sum_v g[v] e[v][c];
// dw[C] (bias) += sum_v g[v].  Wave sums, then one atomic per value per block.
template <int C>
__global__ __launch_bounds__(256) void k_head_bwd(const __bf16* __restrict__ e, int64_t V, const float* __restrict__ w,
                                                  const float* __restrict__ g, __bf16* __restrict__ ge, float* dw) {
    __shared__ float red[C + 1][4];
    const int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    float part[C + 1];
#pragma unroll
    for (int c = 0; c <= C; c++) part[c] = 0.f;
    if (v < V) {
        const float gv = g[v];
#pragma unroll
        for (int c = 0; c < C; c += 8) {
            const bf16x8 a = *(const bf16x8*)(e + v * C + c);
            bf16x8 o;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                o[j] = (__bf16)(((float)a[j] > 0.f) ? gv * w[c + j] : 0.f);
                part[c + j] = gv * (float)a[j];
            }
            *(bf16x8*)(ge + v * C + c) = o;
        }
        part[C] = gv;
    }
#pragma unroll
    for (int c = 0; c <= C; c++) {
        float s = part[c];
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
        if (lane == 0) red[c][wave] = s;
    }
    __syncthreads();
    if (threadIdx.x <= C) {
        const int c = threadIdx.x;
        atomicAdd(dw + c, red[c][0] + red[c][1] + red[c][2] + red[c][3]);
    }
}

// Master FP32 weights [Cout][27][Cin] -> forward BF16 [Cout16][Kpad] and
// data-gradient BF16 [Cin16][K'pad] (k' = (26 - tap)*Cout + co).
__global__ void k_pack(const float* __restrict__ W, int Cin, int Cout, __bf16* wf, int Kpad, int cout16,
                       __bf16* wd, int Kdpad, int cin16) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int64_t nf = (int64_t)cout16 * Kpad;
    const int64_t nd = (int64_t)cin16 * Kdpad;
    const int K = 27 * Cin, Kd = 27 * Cout;
    if (i < nf) {
        const int co = (int)(i / Kpad), k = (int)(i % Kpad);
        wf[weight_index(co, k, cout16)] = (__bf16)((co < Cout && k < K) ? W[(int64_t)co * K + k] : 0.f);
    } else if (wd && i < nf + nd) {
        const int64_t j = i - nf;
        const int ci = (int)(j / Kdpad), kd = (int)(j % Kdpad);
        float val = 0.f;
        if (ci < Cin && kd < Kd) {
            const int tp = kd / Cout, co = kd % Cout;
            val = W[(int64_t)co * K + (26 - tp) * Cin + ci];
        }
        wd[weight_index(ci, kd, cin16)] = (__bf16)val;
    }
}

// Adam (bias-corrected step sizes precomputed on the host).
__global__ void k_adam(float* p, const float* g, float* m, float* v, int64_t n, float b1, float b2, float lr_t,
                       float eps_t) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    p[i] -= lr_t * mi / (sqrtf(vi) + eps_t);
}

// sum x over n floats (FP64 accumulation).
__global__ __launch_bounds__(256) void k_sum(const float* __restrict__ x, int64_t n, double* out) {
    double s = 0.0;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) s += x[i];
    block_add(s, out);
}

inline unsigned blocks(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace

bool conv3_tiled_ok(const ConvArgs& a) {
    const int nt = (a.Cout + 15) / 16;
    return a.wt && a.D0 % kCT0 == 0 && a.D1 % kCT1 == 0 && a.D2 % kCT2 == 0 &&
           a.Ktpad == a.Cin / 8 * kTapsPad * 8 && nt <= 6;
}

template <int MT, int NT, int W>
hipError_t conv3_run(const ConvArgs& a, unsigned tiles, int pieces, hipStream_t s) {
    hipLaunchKernelGGL((k_conv3<MT, NT, W>), dim3(tiles, pieces), dim3(256), (ConvTile<MT, W>::lds(a.Cin / 8)), s, a);
    return hipGetLastError();
}

template <int MT, int W>
hipError_t conv3_pieces(const ConvArgs& a, int nt, hipStream_t s) {
    using T = ConvTile<MT, W>;
    const int64_t tiles = (int64_t)((a.D0 + T::T0 - 1) / T::T0) * ((a.D1 + T::T1 - 1) / T::T1) * ((a.D2 + T::T2 - 1) / T::T2);
    if (tiles > INT32_MAX) return hipErrorInvalidValue;
    // at most 6 output tiles per block (accumulators in registers), fewer where
    // the volume alone gives less than two blocks per CU
    const int want = (int)std::max<int64_t>((nt + 5) / 6, std::min<int64_t>(nt, (512 + tiles - 1) / tiles));
    const int per = (nt + want - 1) / want, pieces = (nt + per - 1) / per;
    switch (per) {
        case 1: return conv3_run<MT, 1, W>(a, (unsigned)tiles, pieces, s);
        case 2: return conv3_run<MT, 2, W>(a, (unsigned)tiles, pieces, s);
        case 3: return conv3_run<MT, 3, W>(a, (unsigned)tiles, pieces, s);
        case 4: return conv3_run<MT, 4, W>(a, (unsigned)tiles, pieces, s);
        case 5: return conv3_run<MT, 5, W>(a, (unsigned)tiles, pieces, s);
        default: return conv3_run<MT, 6, W>(a, (unsigned)tiles, pieces, s);
    }
}

hipError_t launch_conv3(const ConvArgs& a, hipStream_t s) {
    const int64_t V = (int64_t)a.D0 * a.D1 * a.D2;
    if (V == 0) return hipSuccess;
    if (a.Cin % 8 != 0 || a.in_ld % 8 != 0 || a.in_off % 8 != 0 || a.Kpad % 32 != 0 || a.Kpad < 27 * a.Cin)
        return hipErrorInvalidValue;
    const int nt = (a.Cout + 15) / 16;
    const bool up = a.up_chunks > 0;
    if (up && (!conv3_tiled_ok(a) || !a.up || a.up_chunks > a.Cin / 8 || a.up_ld % 8 != 0 || a.up_off % 8 != 0 ||
               a.up_off + 8 * a.up_chunks > a.up_ld))
        return hipErrorInvalidValue;
    if (conv3_tiled_ok(a)) {
        const dim3 tgrid((unsigned)(V / (kCT0 * kCT1 * kCT2)));
        // three chunks per stage where there are as many: a stage's loads are waited for
        const int cps = std::min(3, a.Cin / 8);
        switch (nt) {
#define XR_CONVT_UP(N, C)                                                                  \
    if (up) hipLaunchKernelGGL((k_conv3_tiled<N, C, true>), tgrid, dim3(256), 0, s, a); \
    else hipLaunchKernelGGL((k_conv3_tiled<N, C, false>), tgrid, dim3(256), 0, s, a);
#define XR_CONVT(N)                 \
    case N:                         \
        if (cps == 3) {             \
            XR_CONVT_UP(N, 3)       \
        } else if (cps == 2) {      \
            XR_CONVT_UP(N, 2)       \
        } else {                    \
            XR_CONVT_UP(N, 1)       \
        }                           \
        break;
            XR_CONVT(1)
            XR_CONVT(2)
            XR_CONVT(3)
            XR_CONVT(4)
            XR_CONVT(5)
            XR_CONVT(6)
#undef XR_CONVT
#undef XR_CONVT_UP
        }
        return hipGetLastError();
    }
    if (nt > 9 || a.Cin / 8 > 24) return hipErrorInvalidValue;
    // the largest tile whose halo of all channels leaves room for two blocks in
    // a CU's 160 KB (the smallest takes 24 chunks in 110 KB) and that is not half
    // empty: 256 x 256 x 8, 24 channels, inference with tiles of 32, 16, 8 layers
    // 1253, 1089, 475 us
    const int nch = a.Cin / 8;
    constexpr int64_t room = 80 * 1024;
    if (a.D2 <= 4) return ConvTile<2, 4>::lds(nch) <= room ? conv3_pieces<2, 4>(a, nt, s) : conv3_pieces<1, 4>(a, nt, s);
    if (a.D2 <= 8) return ConvTile<2, 8>::lds(nch) <= room ? conv3_pieces<2, 8>(a, nt, s) : conv3_pieces<1, 8>(a, nt, s);
    if (a.D2 > 16 && ConvTile<4, 16>::lds(nch) <= room) return conv3_pieces<4, 16>(a, nt, s);
    if (ConvTile<2, 16>::lds(nch) <= room) return conv3_pieces<2, 16>(a, nt, s);
    return conv3_pieces<1, 16>(a, nt, s);
}

hipError_t launch_conv3_wgrad(const WgradArgs& a, hipStream_t s) {
    const int64_t V = (int64_t)a.D0 * a.D1 * a.D2;
    if (V == 0) return hipSuccess;
    if (a.Cin % 8 != 0 || a.Cout % 8 != 0 || a.in_ld % 8 != 0 || a.in_off % 8 != 0 || a.g_ld % 8 != 0 ||
        a.g_off % 8 != 0 || a.ldw < 27 * a.Cin)
        return hipErrorInvalidValue;
    const int64_t tiles = (int64_t)((a.D0 + kCT0 - 1) / kCT0) * ((a.D1 + kCT1 - 1) / kCT1) * ((a.D2 + kCT2 - 1) / kCT2);
    if (tiles > INT32_MAX) return hipErrorInvalidValue;
    const int pairs = ((a.Cin + kWgCh - 1) / kWgCh) * ((a.Cout + kWgCh - 1) / kWgCh);
    // two blocks per CU in all: more would add more partial sums than they save
    const int64_t slabs = std::max<int64_t>(1, std::min<int64_t>(tiles, (512 + pairs - 1) / pairs));
    hipLaunchKernelGGL(k_conv3_wgrad, dim3((unsigned)slabs, pairs), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_pool(const __bf16* in, int in_ld, int in_off, int C, int D0, int D1, int D2, __bf16* out,
                       hipStream_t s) {
    if (C % 8 || in_ld % 8 || in_off % 8 || (D0 | D1 | D2) & 1) return hipErrorInvalidValue;
    const int64_t n = (int64_t)(D0 / 2) * (D1 / 2) * (D2 / 2) * (C / 8);
    if (n == 0) return hipSuccess;
    if (n < (int64_t)1 << 31)
        hipLaunchKernelGGL(k_pool<unsigned>, dim3(blocks(n, 256)), dim3(256), 0, s, in, in_ld, in_off, C, D0, D1, D2,
                           out);
    else
        hipLaunchKernelGGL(k_pool<int64_t>, dim3(blocks(n, 256)), dim3(256), 0, s, in, in_ld, in_off, C, D0, D1, D2,
                           out);
    return hipGetLastError();
}

hipError_t launch_pool_bwd(const __bf16* gp, int C, int D0, int D1, int D2, __bf16* gin, int g_ld, int g_off,
                           const __bf16* mask, int m_ld, int m_off, int accumulate, hipStream_t s) {
    if (C % 8 || g_ld % 8 || g_off % 8 || m_ld % 8 || m_off % 8 || (D0 | D1 | D2) & 1) return hipErrorInvalidValue;
    const int64_t n = (int64_t)D0 * D1 * D2 * (C / 8);
    if (n == 0) return hipSuccess;
    if (n < (int64_t)1 << 31)
        hipLaunchKernelGGL(k_pool_bwd<unsigned>, dim3(blocks(n, 256)), dim3(256), 0, s, gp, C, D0, D1, D2, gin, g_ld,
                           g_off, mask, m_ld, m_off, accumulate);
    else
        hipLaunchKernelGGL(k_pool_bwd<int64_t>, dim3(blocks(n, 256)), dim3(256), 0, s, gp, C, D0, D1, D2, gin, g_ld,
                           g_off, mask, m_ld, m_off, accumulate);
    return hipGetLastError();
}

hipError_t launch_upsample(const __bf16* low, int C, int D0, int D1, int D2, __bf16* out, int o_ld, int o_off,
                           hipStream_t s) {
    if (C % 8 || o_ld % 8 || o_off % 8 || (D0 | D1 | D2) & 1) return hipErrorInvalidValue;
    const int64_t n = (int64_t)D0 * D1 * D2 * (C / 8);
    if (n == 0) return hipSuccess;
    if (n < (int64_t)1 << 31)
        hipLaunchKernelGGL(k_upsample<unsigned>, dim3(blocks(n, 256)), dim3(256), 0, s, low, C, D0, D1, D2, out, o_ld,
                           o_off);
    else
        hipLaunchKernelGGL(k_upsample<int64_t>, dim3(blocks(n, 256)), dim3(256), 0, s, low, C, D0, D1, D2, out, o_ld,
                           o_off);
    return hipGetLastError();
}

hipError_t launch_upsample_bwd(const __bf16* g, int g_ld, int g_off, int C, int D0, int D1, int D2, __bf16* glow,
                               hipStream_t s) {
    if (C % 8 || g_ld % 8 || g_off % 8 || (D0 | D1 | D2) & 1) return hipErrorInvalidValue;
    const int64_t n = (int64_t)(D0 / 2) * (D1 / 2) * (D2 / 2) * (C / 8);
    if (n == 0) return hipSuccess;
    if (n < (int64_t)1 << 31)
        hipLaunchKernelGGL(k_upsample_bwd<unsigned>, dim3(blocks(n, 256)), dim3(256), 0, s, g, g_ld, g_off, C, D0, D1,
                           D2, glow);
    else
        hipLaunchKernelGGL(k_upsample_bwd<int64_t>, dim3(blocks(n, 256)), dim3(256), 0, s, g, g_ld, g_off, C, D0, D1,
                           D2, glow);
    return hipGetLastError();
}

hipError_t launch_input8(const float* x, int64_t V, float inv_scale, __bf16* x8, hipStream_t s) {
    if (V == 0) return hipSuccess;
    hipLaunchKernelGGL(k_input8, dim3(blocks(V, 256)), dim3(256), 0, s, x, V, inv_scale, x8);
    return hipGetLastError();
}

hipError_t launch_head(const __bf16* e, int C, int64_t V, const float* w, const float* x, float scale, float* y,
                       const float* t, float* g, double* loss, hipStream_t s) {
    if (V == 0) return hipSuccess;
    // with a loss, a few blocks per CU (each adds to it once)
    const unsigned nb = (unsigned)std::min<int64_t>((V + 255) / 256, loss ? 1024 : INT32_MAX);
    switch (C) {
#define XR_HEAD(N) \
    case N: hipLaunchKernelGGL(k_head<N>, dim3(nb), dim3(256), 0, s, e, V, w, x, scale, y, t, g, loss); break;
        XR_HEAD(8)
        XR_HEAD(16)
        XR_HEAD(24)
        XR_HEAD(32)
#undef XR_HEAD
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_head_bwd(const __bf16* e, int C, int64_t V, const float* w, const float* g, __bf16* ge,
                           float* dw, hipStream_t s) {
    if (V == 0) return hipSuccess;
    switch (C) {
#define XR_HEADB(N) \
    case N: hipLaunchKernelGGL(k_head_bwd<N>, dim3(blocks(V, 256)), dim3(256), 0, s, e, V, w, g, ge, dw); break;
        XR_HEADB(8)
        XR_HEADB(16)
        XR_HEADB(24)
        XR_HEADB(32)
#undef XR_HEADB
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_pack(const float* W, int Cin, int Cout, __bf16* wf, int Kpad, __bf16* wd, int Kdpad,
                       hipStream_t s) {
    const int cout16 = (Cout + 15) / 16 * 16, cin16 = (Cin + 15) / 16 * 16;
    const int64_t n = (int64_t)cout16 * Kpad + (wd ? (int64_t)cin16 * Kdpad : 0);
    hipLaunchKernelGGL(k_pack, dim3(blocks(n, 256)), dim3(256), 0, s, W, Cin, Cout, wf, Kpad, cout16, wd, Kdpad,
                       cin16);
    return hipGetLastError();
}

hipError_t launch_pack_tiled(const float* W, int Cin, int Cout, __bf16* wt, int Ktpad, hipStream_t s) {
    const int cout16 = (Cout + 15) / 16 * 16;
    const int64_t n = (int64_t)cout16 * Ktpad;
    hipLaunchKernelGGL(k_pack_tiled, dim3(blocks(n, 256)), dim3(256), 0, s, W, Cin, Cout, wt, Ktpad, cout16);
    return hipGetLastError();
}

hipError_t launch_adam(float* p, const float* g, float* m, float* v, int64_t n, float b1, float b2, float lr_t,
                       float eps_t, hipStream_t s) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(k_adam, dim3(blocks(n, 256)), dim3(256), 0, s, p, g, m, v, n, b1, b2, lr_t, eps_t);
    return hipGetLastError();
}

hipError_t launch_sum(const float* x, int64_t n, double* out, hipStream_t s) {
    if (n == 0) return hipSuccess;
    const int64_t nb = std::min<int64_t>(512, (n + 1023) / 1024);
    hipLaunchKernelGGL(k_sum, dim3((unsigned)nb), dim3(256), 0, s, x, n, out);
    return hipGetLastError();
}

}  // namespace nn
}  // namespace xr
