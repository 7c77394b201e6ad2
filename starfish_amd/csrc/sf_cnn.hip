// Learned initial guess for the potential solve: a 3-level encoder-decoder CNN
// (32/64/128 channels, 3x3 convolutions, BF16 weights and activations, FP32 accumulation on
// the gfx950 matrix cores) mapping (rho, Dirichlet mask, boundary phi) to phi.  Training runs
// on the GPU with the kernels below (forward, backward-data, backward-weights, Adam).  The
// network only supplies the starting point of the Newton/PCG solve; every solve still runs to
// the requested relative residual, so plain PCG remains the fallback and the judge.
//
// Layout: activations are NHWC BF16 tensors addressed through views (pointer, channel stride,
// channel offset) so that skip connections concatenate without copies.  3x3 convolutions are
// implicit GEMMs on v_mfma_f32_16x16x32_bf16: M = 16 pixels of a row, N = 16 output channels,
// K = 32 input channels of one tap.
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "sf_internal.h"
#include "sf_normal.h"

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

namespace sf {

__device__ __host__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    if ((u & 0x7F800000u) == 0x7F800000u) return (uint16_t)(u >> 16);   // inf / nan
    u += 0x7FFFu + ((u >> 16) & 1u);                                     // round to nearest even
    return (uint16_t)(u >> 16);
}
// two floats to packed BF16 (round to nearest even, as f2bf for finite values) with the
// hardware conversion
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
    const __bf16 x = (__bf16)a, y = (__bf16)b;
    uint16_t ux, uy;
    memcpy(&ux, &x, 2);
    memcpy(&uy, &y, 2);
    return (uint32_t)ux | ((uint32_t)uy << 16);
}
__device__ __host__ __forceinline__ float bf2f(uint16_t h) {
    uint32_t u = (uint32_t)h << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

// ReLU backward of 4 channels: g where the BF16 activation (4 values packed in a) is positive, else 0
__device__ __forceinline__ float4 relu_mask4(const float4 g, const uint2 a) {
    return make_float4(bf2f((uint16_t)(a.x & 0xFFFFu)) > 0.f ? g.x : 0.f, bf2f((uint16_t)(a.x >> 16)) > 0.f ? g.y : 0.f,
                       bf2f((uint16_t)(a.y & 0xFFFFu)) > 0.f ? g.z : 0.f, bf2f((uint16_t)(a.y >> 16)) > 0.f ? g.w : 0.f);
}
__device__ __forceinline__ uint2 pack_bf16x4(const float4 e) {
    return make_uint2(pack_bf16x2(e.x, e.y), pack_bf16x2(e.z, e.w));
}

__device__ __forceinline__ uint32_t bf_at(const uint4& v, int c) {
    const uint32_t w = c < 2 ? v.x : (c < 4 ? v.y : (c < 6 ? v.z : v.w));
    return (c & 1) ? (w >> 16) : (w & 0xFFFFu);
}

// ------------------------------------------------------------------------------------------
// 3x3 convolution as an implicit GEMM (stride 1, zero padding 1).
//   forward:       out[p][n] = sum_tap sum_k in[p + d(tap)][k] * w[tap][n][k]   (+ bias, ReLU)
//   backward data: din[p][k'] = sum_tap sum_n' g[p - d(tap)][n'] * w[tap][n'][k'] with the weight
//                  stored transposed as wt[tap][k'][n'] -> the same kernel with sgn = -1.
// What surrounds a convolution in the network happens in its own loads and stores, so no pass over
// memory does only pooling, upsampling or a ReLU's backward:
//   input    channels [0, kup) are the nearest 2x upsampling of `up` (half resolution), the others `in`
//   FWD      BF16 output with bias and ReLU, and if `pool` is given its 2x2 mean at half resolution
//   BWD_RELU the ReLU backward of the layer before (its BF16 activation `act`): act > 0 ? din : 0
//   BWD_UP   channels [0, nup): the sum over each 2x2 block (the upsampling's backward) masked by
//            `act` at half resolution, BF16; the others (the skip path) FP32 into `skip`
//   BWD_POOL the 2x2 mean's backward plus the skip path: each of the four pixels of twice the
//            resolution gets skip + din / 4, masked by its `act`, BF16
// Before, the pooling and upsampling kernels of an Adam step at 1024 x 512, batch 4, took 650 of its 4900 us,
// and the decoder's FP32 input gradients (800 MB at full resolution) were written and read whole.
// Requirements: K a multiple of 32, N of TN, channel counts in memory multiples of 8 (16-byte operand
// loads), kup a multiple of 32, nup a multiple of TN; H and W even with `up`, `pool` and BWD_UP (the
// network's grid is a multiple of 4, so only its quarter resolution can be odd).
// ------------------------------------------------------------------------------------------
enum ConvMode { FWD, BWD_RELU, BWD_UP, BWD_POOL };
struct ConvP {
    const uint16_t* in;     // [B][H][W][in_cs]; channels from in_cs up are zero
    const uint16_t* up;     // [B][H/2][W/2][kup]
    const uint16_t* w;      // [tap][N][K]
    const float* bias;
    const uint16_t* act;
    uint16_t *out, *pool;
    float* skip;
    int in_cs, kup, K, N, nup, H, W, B;
    int nrt, gx, gy, nsp;   // row tiles of a workgroup, tiles along x and y, tiles of all images
};

// 16 bytes a lane from a uniform base (through which no lane reaches below its tensor) and a lane's own byte
// offset; zeros where the offset is NOWHERE, which lies beyond the range of the resource.  The address
// arithmetic of a stage is then a few scalar operations and one offset a lane kept for all of them (with
// the addresses worked out per load, some 200 vector instructions a chunk of 36 MFMAs: 3.06 ms an Adam
// step at 1024 x 512, batch 4, now 2.82; the weight gradients 780 us of it, now 640).
constexpr uint32_t NOWHERE = 0x80000000u;
__device__ __forceinline__ __amdgpu_buffer_rsrc_t uniform_base(const uint16_t* p) {
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, (short)0, 0x7FFFFFFF, 0x00020000);
}
__device__ __forceinline__ uint4 load16(__amdgpu_buffer_rsrc_t base, uint32_t off) {
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(base, off, 0, 0);
    uint4 r;
    memcpy(&r, &v, 16);
    return r;
}

// lane's neighbour in its pair of lanes (2 q, 2 q + 1): the other pixel of a 2x2 block's row
__device__ __forceinline__ float pair_lane(float v) {
    int i;
    memcpy(&i, &v, 4);
    i = __builtin_amdgcn_update_dpp(0, i, 0xB1, 0xF, 0xF, true);   // quad_perm 1, 0, 3, 2
    memcpy(&v, &i, 4);
    return v;
}
// sum over a 2x2 block in the order of its pixels, in the even lane of the pair (r0, r1: its two rows)
__device__ __forceinline__ float4 block_sum(const float4 r0, const float4 r1) {
    return make_float4(0.f + r0.x + pair_lane(r0.x) + r1.x + pair_lane(r1.x),
                       0.f + r0.y + pair_lane(r0.y) + r1.y + pair_lane(r1.y),
                       0.f + r0.z + pair_lane(r0.z) + r1.z + pair_lane(r1.z),
                       0.f + r0.w + pair_lane(r0.w) + r1.w + pair_lane(r1.w));
}
__device__ __forceinline__ float4 as_float4(const f32x4 v) { return make_float4(v[0], v[1], v[2], v[3]); }
__device__ __forceinline__ float4 unpack_bf16x4(const uint2 u) {
    return make_float4(bf2f((uint16_t)(u.x & 0xFFFFu)), bf2f((uint16_t)(u.x >> 16)), bf2f((uint16_t)(u.y & 0xFFFFu)),
                       bf2f((uint16_t)(u.y >> 16)));
}

// The operands are staged in LDS.  One workgroup: CONV_R rows of CONV_TP pixels x CONV_TN output
// channels, its four waves over the pixels.  For each chunk of 32 input channels the CONV_R + 2
// input rows of CONV_TP + 2 pixels and the 9 x CONV_TN x 32 weights go to LDS once (the weights once
// in all where there is one chunk), and every wave runs its 16 x 16 tiles of all rows over the 9
// taps from there, its 12 input fragments read once.  The next chunk's operands are loaded into
// registers while the current one is multiplied.  The weights are the MFMA's A operand
// (rows = output channels) and the pixels its B operand, so a lane's result holds 4 consecutive
// channels of one pixel and leaves in one 8-byte (BF16) or 16-byte (FP32) store.
//
// The stages' latency bounds it, so many small workgroups do better than few that use their operands
// more often: with 35 KB of LDS four run on a CU.  Measured against 128 pixels x 2 rows x 64 (or x 4
// x 32) channels, two on a CU: Adam step (1024 x 512, batch 4) 3.97 against 4.12 ms; guess at
// 301 x 157, where the large tiles leave most CUs idle, 140 against 227 us.  Four rows a tile, which
// halve the LDS reads of a product, gain nothing (3.11 ms a step either way).
//
// The workgroups of an XCD (consecutive indices go round the eight) take a contiguous band of
// tiles, and the channel tiles of one pixel tile follow each other, so the input rows that they
// share, and the halo rows of neighbouring tiles, come from that XCD's L2.
constexpr int CONV_TN = 32, CONV_R = 2, CONV_TP = 64;
template <int MODE>
__global__ void __launch_bounds__(256, 4) conv3x3_lds(const ConvP p) {
    constexpr int TN = CONV_TN, R = CONV_R, SGN = MODE == FWD ? 1 : -1;
    constexpr int IW = CONV_TP + 2;             // staged pixels per row
    constexpr int NIN = (R + 2) * IW * 4;       // 16-byte groups of the input stage (8 channels each)
    constexpr int NWT = 9 * TN * 4;             // 16-byte groups of the weight stage
    constexpr int RIN = (NIN + 255) / 256, RWT = (NWT + 255) / 256;
    static_assert(CONV_TP == 64 && TN == 32 && R == 2, "a wave has two rows of 16 pixels x 32 channels");
    __shared__ uint4 s_in[NIN];                 // [row][pixel][group]
    __shared__ uint4 s_w[NWT];                  // [tap][channel][group]
    const int ntn = p.N / TN, per = (p.nsp + 7) / 8;
    const int slot = blockIdx.x >> 3, sp = (blockIdx.x & 7) * per + slot / ntn;
    if (slot / ntn >= per || sp >= p.nsp) return;
    const int n0 = (slot % ntn) * TN;
    // the workgroup walks nrt tiles of R rows down its column; step it is chunk it % nkc of row
    // tile it / nkc, so the next tile's first chunk is loaded while the current tile is multiplied
    const int x0 = (sp % p.gx) * CONV_TP, y_first = ((sp / p.gx) % p.gy) * p.nrt * R, b = sp / (p.gx * p.gy);
    const int nkc = p.K / 32, H = p.H, Wd = p.W, N = p.N;
    const int steps = min(p.nrt, (H - y_first + R - 1) / R) * nkc;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int prow = lane & 15, kq = lane >> 4;
    uint4 rin[RIN], rwt[RWT];
    // a lane's byte offsets: its pixels and channel group from pixel (x0 - 1, y0 - 1) of `in`, from the
    // pixel of `up` that holds it, and its weights from those of channel n0
    uint32_t oin[RIN], oup[MODE == FWD ? RIN : 1], owt[RWT];
#pragma unroll
    for (int q = 0; q < RIN; q++) {
        const int e = threadIdx.x + 256 * q, g = e & 3, px = (e >> 2) % IW, r = (e >> 2) / IW, xx = x0 - 1 + px;
        const bool ok = e < NIN && xx >= 0 && xx < Wd;
        oin[q] = ok && g * 8 < p.in_cs ? (uint32_t)(2 * ((r * Wd + px) * p.in_cs + g * 8)) : NOWHERE;
        if constexpr (MODE == FWD)   // (x0 and y0 are even: pixel x0 - 1 is the odd one of its pair)
            oup[q] = ok ? (uint32_t)(2 * ((((r + 1) >> 1) * (Wd >> 1) + ((px + 1) >> 1)) * p.kup + g * 8)) : NOWHERE;
    }
#pragma unroll
    for (int q = 0; q < RWT; q++) {
        const int e = threadIdx.x + 256 * q, g = e & 3, n = (e >> 2) % TN, tap = (e >> 2) / TN;
        owt[q] = e < NWT ? (uint32_t)(2 * ((tap * N + n) * p.K + g * 8)) : NOWHERE;
    }
    auto fetch = [&](int it) __attribute__((always_inline)) {
        const int y0 = y_first + (it / nkc) * R, k0 = (it % nkc) * 32;
        const bool from_up = MODE == FWD && k0 < p.kup;
        const int Hs = H >> 1, Ws = Wd >> 1;
        const uint16_t* const src =
            from_up ? p.up + (((int64_t)b * Hs + (y0 >> 1) - 1) * Ws + (x0 >> 1) - 1) * p.kup + k0
                    : p.in + (((int64_t)b * H + y0 - 1) * Wd + x0 - 1) * p.in_cs + k0 - p.kup;
        const __amdgpu_buffer_rsrc_t base = uniform_base(src);
        const uint32_t up_mask = from_up ? ~0u : 0u;
        const bool edge = y0 == 0 || y0 + R >= H;   // some of the rows y0 - 1 .. y0 + R are outside
#pragma unroll
        for (int q = 0; q < RIN; q++) {
            uint32_t o = oin[q];
            if constexpr (MODE == FWD) o ^= (o ^ oup[q]) & up_mask;   // (a select would be one of addresses, in scratch)
            if (edge) {
                const int yy = y0 - 1 + (int)((threadIdx.x + 256 * q) >> 2) / IW;
                if (yy < 0 || yy >= H) o = NOWHERE;
            }
            rin[q] = load16(base, o);
        }
        if (nkc == 1 && it > 0) return;   // (the weights stay)
        const __amdgpu_buffer_rsrc_t wbase = uniform_base(p.w + (int64_t)n0 * p.K + k0);
#pragma unroll
        for (int q = 0; q < RWT; q++) rwt[q] = load16(wbase, owt[q]);
    };
    f32x4 acc[R][2];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r][0] = acc[r][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (steps > 0) fetch(0);
    for (int it = 0; it < steps; it++) {
        __syncthreads();   // the previous chunk's fragments are read
#pragma unroll
        for (int q = 0; q < RIN; q++)
            if (threadIdx.x + 256 * q < NIN) s_in[threadIdx.x + 256 * q] = rin[q];
        if (nkc > 1 || it == 0)
#pragma unroll
            for (int q = 0; q < RWT; q++)
                if (threadIdx.x + 256 * q < NWT) s_w[threadIdx.x + 256 * q] = rwt[q];
        __syncthreads();
        if (it + 1 < steps) fetch(it + 1);
        bf16x8 a[R + 2][3];
#pragma unroll
        for (int r = 0; r < R + 2; r++)
#pragma unroll
            for (int q = 0; q < 3; q++) {
                const uint4 v = s_in[(r * IW + wave * 16 + prow + q) * 4 + kq];
                memcpy(&a[r][q], &v, 16);
            }
#pragma unroll
        for (int tap = 0; tap < 9; tap++) {
            bf16x8 bw[2];
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const uint4 v = s_w[(tap * TN + t * 16 + prow) * 4 + kq];
                memcpy(&bw[t], &v, 16);
            }
#pragma unroll
            for (int r = 0; r < R; r++)
#pragma unroll
                for (int t = 0; t < 2; t++)
                    acc[r][t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        bw[t], a[r + 1 + SGN * (tap / 3 - 1)][1 + SGN * (tap % 3 - 1)], acc[r][t], 0, 0, 0);
        }
        if (it % nkc != nkc - 1) continue;
        // the row tile's last chunk: store its outputs and clear the accumulators
        // D layout: lane holds rows (lane/16)*4 + i (channels), column lane%16 (pixel)
        const int xo = x0 + wave * 16 + prow;
        const int y = y_first + (it / nkc) * R;   // rows y and y + 1 (y alone at the end of an odd image)
        const int nrow = min(R, H - y);
        if (xo < Wd) {   // (both lanes of a pair where W is even)
#pragma unroll
            for (int t = 0; t < 2; t++) {
                const int n = n0 + t * 16 + kq * 4;   // this lane's 4 channels n .. n + 3
                const size_t px = ((size_t)b * H + y) * Wd + xo;
                const float4 v0 = as_float4(acc[0][t]), v1 = as_float4(acc[1][t]);
                if constexpr (MODE == FWD) {
                    const float4 bs = *reinterpret_cast<const float4*>(p.bias + n);
                    const uint2 u0 = pack_bf16x4(make_float4(fmaxf(v0.x + bs.x, 0.f), fmaxf(v0.y + bs.y, 0.f),
                                                             fmaxf(v0.z + bs.z, 0.f), fmaxf(v0.w + bs.w, 0.f)));
                    const uint2 u1 = pack_bf16x4(make_float4(fmaxf(v1.x + bs.x, 0.f), fmaxf(v1.y + bs.y, 0.f),
                                                             fmaxf(v1.z + bs.z, 0.f), fmaxf(v1.w + bs.w, 0.f)));
                    *reinterpret_cast<uint2*>(p.out + px * N + n) = u0;
                    if (nrow > 1) *reinterpret_cast<uint2*>(p.out + (px + Wd) * N + n) = u1;
                    if (p.pool) {
                        const float4 s = block_sum(unpack_bf16x4(u0), unpack_bf16x4(u1));
                        if (!(prow & 1))
                            *reinterpret_cast<uint2*>(
                                p.pool + (((size_t)b * (H / 2) + y / 2) * (Wd / 2) + xo / 2) * N + n) =
                                pack_bf16x4(make_float4(0.25f * s.x, 0.25f * s.y, 0.25f * s.z, 0.25f * s.w));
                    }
                } else if constexpr (MODE == BWD_RELU) {
                    const size_t o0 = px * N + n, o1 = (px + (nrow > 1 ? Wd : 0)) * N + n;
                    const uint2 a0 = *reinterpret_cast<const uint2*>(p.act + o0);
                    const uint2 a1 = *reinterpret_cast<const uint2*>(p.act + o1);
                    *reinterpret_cast<uint2*>(p.out + o0) = pack_bf16x4(relu_mask4(v0, a0));
                    if (nrow > 1) *reinterpret_cast<uint2*>(p.out + o1) = pack_bf16x4(relu_mask4(v1, a1));
                } else if constexpr (MODE == BWD_UP) {
                    if (n0 < p.nup) {
                        const float4 s = block_sum(v0, v1);
                        const size_t o = (((size_t)b * (H / 2) + y / 2) * (Wd / 2) + xo / 2) * p.nup + n;
                        if (!(prow & 1))
                            *reinterpret_cast<uint2*>(p.out + o) =
                                pack_bf16x4(relu_mask4(s, *reinterpret_cast<const uint2*>(p.act + o)));
                    } else {
                        const size_t o = px * (N - p.nup) + n - p.nup;
                        *reinterpret_cast<float4*>(p.skip + o) = v0;
                        *reinterpret_cast<float4*>(p.skip + o + (size_t)Wd * (N - p.nup)) = v1;
                    }
                } else {
#pragma unroll
                    for (int r = 0; r < 2; r++) {
                        // the four pixels (k & 1, k >> 1) of row y + r; all loads before the first use
                        const float4 d = r ? v1 : v0;
                        const size_t o = (((size_t)b * H + y + (nrow > 1 ? r : 0)) * 4 * Wd + 2 * xo) * N + n;
                        const int ok[4] = {0, N, 2 * Wd * N, (2 * Wd + 1) * N};
                        float4 sk[4];
                        uint2 av[4];
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            sk[k] = *reinterpret_cast<const float4*>(p.skip + o + ok[k]);
                            av[k] = *reinterpret_cast<const uint2*>(p.act + o + ok[k]);
                        }
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            const float4 e = make_float4(sk[k].x + 0.25f * d.x, sk[k].y + 0.25f * d.y,
                                                         sk[k].z + 0.25f * d.z, sk[k].w + 0.25f * d.w);
                            if (r < nrow) *reinterpret_cast<uint2*>(p.out + o + ok[k]) = pack_bf16x4(relu_mask4(e, av[k]));
                        }
                    }
                }
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++) acc[r][0] = acc[r][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
}

// Weight gradient with the operands staged in LDS.  One workgroup: 32 input x 32 output channels
// for all 9 taps over a run of chunks, a chunk being 64 pixels of one row; the chunks of a run go
// down the rows of a 64-pixel column band.  Two chunks (rows y, y + 1) are multiplied between two
// barriers: they need the input rows y - 1 .. y + 2 out of a ring of six in LDS, where the rows
// y + 3 and y + 4 of the next two, loaded into registers meanwhile, are stored after the products.
// Rows stay as they are in memory, [pixel][channel]: the fragments (8 pixels of one channel a lane)
// come from the transposing LDS read, and a tap's shift along x is an offset of whole pixels.  A
// pixel's two 16-channel halves are swapped in every second group of 8 pixels, so the 8 pixels that
// 32 lanes read fall on distinct banks.  An input fragment serves the taps of both rows.
// Wave w takes the pixels 32 (w & 1) .. + 31 of every chunk (one MFMA reduction step) and input
// channels 16 (w >> 1) .. + 15 against all 32 output channels: 12 input and 4 gradient fragments
// for 36 MFMAs.  The waves of the first input-channel tile also sum the gradient over the pixels
// (the bias gradient) with one more MFMA per output tile against an all-ones operand.  At the end
// the two pixel halves are added through LDS and the workgroup stores its sums as a partial
// (WG_PART floats: [tap][k][n], then the 32 bias sums); wgrad_reduce adds the partials of a channel
// tile pair in a fixed order, which is deterministic and avoids thousands of workgroups' atomics on
// the same addresses.
// Input channels below kup are the nearest 2x upsampling of `up`, as in conv3x3_lds.  The channel
// tile pairs of a run follow each other on one XCD, and an XCD takes neighbouring runs, so the rows
// that they share are read from HBM once.
// Bound by the LDS reads and the MFMAs alike (512 and 576 cycles for two chunks), the first and last
// layers by HBM.  Measured at 1024 x 512, batch 4: 640 us for the ten layers of a step, against 1480
// with rows transposed by two of the four waves as they were stored, three shifted copies of each,
// and two barriers a chunk; the largest (96 x 32 channels at full resolution) 125 us, 930 TFLOP/s.
// 162 registers: three workgroups a CU.
// Requirements: K and N multiples of 32, kup too, channel counts in memory multiples of 8.
constexpr int WG_PX = 64;           // pixels per chunk (two MFMA reduction steps)
constexpr int WG_IW = WG_PX + 2;    // staged pixels per input row
constexpr int WG_RING = 6;          // staged input rows
constexpr int WG_PART = 9 * 32 * 32 + 32;   // floats of a workgroup's partial
constexpr int WG_BLOCKS = 768;              // target workgroups of a weight-gradient launch (3 per CU)
typedef short s16x4 __attribute__((ext_vector_type(4)));
// this lane's place for an 8-byte piece of pixel px of a staged row: 16-channel half h, quarter of it c
__device__ __forceinline__ int wg_at(int px, int h, int c) { return px * 64 + ((h ^ (px >> 3)) & 1) * 32 + c * 8; }
// 8 pixels x 16 channels of a staged row: the transposing reads at lo (its first four pixels) and hi
__device__ __forceinline__ bf16x8 wg_frag(const char* lo, const char* hi) {
    typedef __attribute__((address_space(3))) s16x4 lds4;
    const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)lo);
    const s16x4 b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds4*)hi);
    bf16x8 r;
    memcpy(&r, &a, 8);
    memcpy((char*)&r + 8, &b, 8);
    return r;
}
__global__ void __launch_bounds__(256, 3) conv3x3_wgrad_lds(const uint16_t* __restrict__ in, int in_cs,
                                                         const uint16_t* __restrict__ up, int kup, int K,
                                                         const uint16_t* __restrict__ g, int N,
                                                         float* __restrict__ part, int H, int Wd, int B, int nrun,
                                                         int chunks_per_block) {
    constexpr int ROW_IN = WG_IW * 64, ROW_G = WG_PX * 64;   // bytes of a staged row
    __shared__ uint4 lds[(WG_RING * ROW_IN + 4 * ROW_G) / 16];
    char* const s_in = reinterpret_cast<char*>(lds);         // [row % 6][pixel][channel]
    char* const s_g = s_in + WG_RING * ROW_IN;               // [interval & 1][row][pixel][channel]
    const int nkt = K / 32, pairs = nkt * (N / 32), per = (nrun + 7) / 8;
    const int slot_i = blockIdx.x >> 3, run = (blockIdx.x & 7) * per + slot_i / pairs, pair = slot_i % pairs;
    if (slot_i / pairs >= per || run >= nrun) return;
    const int k0 = (pair % nkt) * 32, n0 = (pair / nkt) * 32;
    const int t = threadIdx.x, wave = t >> 6, lane = t & 63;
    const int ks = wave & 1, tk = wave >> 1;   // pixel half (reduction step), input-channel half
    const int prow = lane & 15, kq = lane >> 4;
    const int cpr = (Wd + WG_PX - 1) / WG_PX;
    const int nchunks = B * H * cpr;
    // chunk c: row c % H of column band (c / H) % cpr of image c / (H cpr)
    const int c_begin = run * chunks_per_block;
    const int c_end = min(c_begin + chunks_per_block, nchunks);
    const bool from_up = k0 < kup;
    const uint16_t* const src = (from_up ? up : in) + (from_up ? k0 : k0 - kup);
    const int sh = from_up ? 1 : 0, scs = from_up ? kup : in_cs;
    const int Hs = H >> sh, Ws = Wd >> sh;
    // staging: thread t takes the 8 channels 8 (t & 3) .. + 7 of one pixel a time, 264 pieces an input
    // row and 256 a gradient row.  Its byte offsets from a band's first pixel are kept for the band: its
    // pixels of an input row, and its pixel of a gradient row.
    uint4 vin[3], vg[2];
    uint32_t oin[3], og = NOWHERE;
    auto band_offsets = [&](int x0) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const int e = t + 256 * q, r = e >= 4 * WG_IW ? 1 : 0, px = (e - r * 4 * WG_IW) >> 2, xx = x0 - 1 + px;
            // (from the pixel before x0, or from the one of `up` that holds it: x0 is even)
            oin[q] = e < 8 * WG_IW && xx >= 0 && xx < Wd && (t & 3) * 8 < scs
                         ? (uint32_t)(2 * (((px + sh) >> sh) * scs + (t & 3) * 8)) : NOWHERE;
        }
        og = x0 + (t >> 2) < Wd ? (uint32_t)(2 * ((t >> 2) * N + (t & 3) * 8)) : NOWHERE;
    };
    auto fetch_in = [&](int b, int x0, int y) __attribute__((always_inline)) {   // input rows y and y + 1
        const __amdgpu_buffer_rsrc_t base =
            uniform_base(src + (((int64_t)b * Hs + (y >> sh)) * Ws + (x0 >> sh) - 1) * scs);
        const uint32_t step = (uint32_t)(2 * (((y + 1) >> sh) - (y >> sh)) * Ws * scs);   // to the second row
        const bool ok0 = y >= 0 && y < H, ok1 = y + 1 >= 0 && y + 1 < H;
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const bool second = t + 256 * q >= 4 * WG_IW;
            uint32_t o = oin[q] + (second ? step : 0u);   // (NOWHERE stays beyond the range)
            if (!(second ? ok1 : ok0)) o = NOWHERE;
            vin[q] = load16(base, o);
        }
    };
    auto store_in = [&](int y) __attribute__((always_inline)) {
#pragma unroll
        for (int q = 0; q < 3; q++) {
            const int e = t + 256 * q, r = e >= 4 * WG_IW ? 1 : 0, px = (e - r * 4 * WG_IW) >> 2;
            if (e < 8 * WG_IW)
                *reinterpret_cast<uint4*>(s_in + ((y + r + WG_RING) % WG_RING) * ROW_IN +
                                          wg_at(px, (t >> 1) & 1, (t & 1) * 2)) = vin[q];
        }
    };
    auto fetch_g = [&](int b, int x0, int y, int nr) __attribute__((always_inline)) {   // gradient rows y and y + 1
#pragma unroll
        for (int r = 0; r < 2; r++)   // (a second row outside of the run counts as zero)
            vg[r] = load16(uniform_base(g + (((int64_t)b * H + y + r) * Wd + x0) * N + n0), r < nr ? og : NOWHERE);
    };
    auto store_g = [&](int half) __attribute__((always_inline)) {
#pragma unroll
        for (int r = 0; r < 2; r++)
            *reinterpret_cast<uint4*>(s_g + (half * 2 + r) * ROW_G + wg_at(t >> 2, (t >> 1) & 1, (t & 1) * 2)) = vg[r];
    };
    // fragment pieces: pixel 8 kq + 4 i + prow / 4 (+ the tap's shift), channels 4 (prow & 3) .. + 3 of a half
    int at_in[3][2], at_g[2][2];
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int px = ks * 32 + kq * 8 + i * 4 + (prow >> 2);
#pragma unroll
        for (int dx = 0; dx < 3; dx++) at_in[dx][i] = wg_at(px + dx, tk, prow & 3);
#pragma unroll
        for (int n = 0; n < 2; n++) at_g[n][i] = wg_at(px, n, prow & 3);
    }
    f32x4 acc[9][2];
#pragma unroll
    for (int tap = 0; tap < 9; tap++) acc[tap][0] = acc[tap][1] = f32x4{0.f, 0.f, 0.f, 0.f};
    f32x4 accb[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    const bool do_bias = k0 == 0 && tk == 0;   // uniform per wave
    bf16x8 ones;
    {
        const uint32_t o2 = 0x3F803F80u;   // two BF16 1.0
        const uint4 u = make_uint4(o2, o2, o2, o2);
        memcpy(&ones, &u, 16);
    }
    // the products of rows y and y + 1: every tap's sum takes the rows in order
    auto multiply = [&](int y, int half) __attribute__((always_inline)) {
        bf16x8 bg[2][2];
#pragma unroll
        for (int s = 0; s < 2; s++)
#pragma unroll
            for (int n = 0; n < 2; n++) {
                const char* const row = s_g + (half * 2 + s) * ROW_G;
                bg[s][n] = wg_frag(row + at_g[n][0], row + at_g[n][1]);
                if (do_bias) accb[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, bg[s][n], accb[n], 0, 0, 0);
            }
#pragma unroll
        for (int rr = 0; rr < 4; rr++) {   // input row y - 1 + rr: tap row rr - s of row y + s
            const char* const row = s_in + ((y + rr + WG_RING - 1) % WG_RING) * ROW_IN;
#pragma unroll
            for (int dx = 0; dx < 3; dx++) {
                const bf16x8 a = wg_frag(row + at_in[dx][0], row + at_in[dx][1]);
#pragma unroll
                for (int s = 0; s < 2; s++)
                    if (rr - s >= 0 && rr - s < 3)
#pragma unroll
                        for (int n = 0; n < 2; n++) {
                            f32x4& d = acc[(rr - s) * 3 + dx][n];
                            d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bg[s][n], d, 0, 0, 0);
                        }
            }
        }
    };
    bool fresh = true;   // the run's first rows, or a band's
    for (int c = c_begin, half = 0; c < c_end; half ^= 1) {
        const int y = c % H, band = c / H, b = band / cpr, x0 = (band % cpr) * WG_PX;
        auto rows = [&](int q) { return c + q + 1 < c_end && y + q + 1 < H ? 2 : 1; };
        if (fresh) {
            __syncthreads();   // the previous band's fragments are read
            band_offsets(x0);
            fetch_in(b, x0, y - 1);
            fetch_g(b, x0, y, rows(0));
            store_in(y - 1);
            fetch_in(b, x0, y + 1);
            store_g(half);
            store_in(y + 1);
            __syncthreads();
        }
        const bool more = c + 2 < c_end && y + 2 < H;
        if (more) {
            fetch_in(b, x0, y + 3);
            fetch_g(b, x0, y + 2, rows(2));
        }
        multiply(y, half);
        if (more) {   // (these rows' places were last read before the barrier before this)
            store_in(y + 3);
            store_g(half ^ 1);
            __syncthreads();
        }
        fresh = !more;
        c += rows(0);
    }
    // the second pixel half's sums go through LDS (9 x 2 x 4 floats per lane and wave, then the bias
    // sums) to the first half's waves, which add them and store the partial
    __syncthreads();
    float* const red = reinterpret_cast<float*>(lds);   // 2 x 80 x 64 floats
    static_assert(sizeof(lds) >= 2 * 80 * 64 * sizeof(float), "reduction space");
    if (ks == 1) {
#pragma unroll
        for (int tap = 0; tap < 9; tap++)
#pragma unroll
            for (int n = 0; n < 2; n++)
#pragma unroll
                for (int i = 0; i < 4; i++) red[((tk * 80) + (tap * 2 + n) * 4 + i) * 64 + lane] = acc[tap][n][i];
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int i = 0; i < 4; i++) red[((tk * 80) + 72 + n * 4 + i) * 64 + lane] = accb[n][i];
    }
    __syncthreads();
    if (ks == 1) return;
    // D rows (lane/16)*4+i = input channel, column lane%16 = output channel
    float* const pb = part + ((size_t)pair * nrun + run) * WG_PART;
#pragma unroll
    for (int tap = 0; tap < 9; tap++)
#pragma unroll
        for (int n = 0; n < 2; n++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                pb[(tap * 32 + tk * 16 + kq * 4 + i) * 32 + n * 16 + prow] =
                    acc[tap][n][i] + red[((tk * 80) + (tap * 2 + n) * 4 + i) * 64 + lane];
    // every row of accb holds the column sums: lanes 0..15 store row 0
    if (tk == 0 && kq == 0)
#pragma unroll
        for (int n = 0; n < 2; n++)
            pb[9 * 32 * 32 + n * 16 + prow] = do_bias ? accb[n][0] + red[(72 + n * 4) * 64 + lane] : 0.f;
}

// Sum of the weight-gradient partials of channel tile pair y: a workgroup takes 32 entries e;
// slice j of its threads adds the partials b = j, j + 8, ... in order, and the 8 slice sums are
// added in order (a fixed order, so the result does not depend on timing).  Entry e < 9 * 32 * 32
// ([tap][k][n] of the tile) goes to dw, the rest (the bias sums, first input-channel tile only)
// to db.
__global__ void __launch_bounds__(256) wgrad_reduce(const float* __restrict__ part, int nblk, int K, int N,
                                                    float* __restrict__ dw, float* __restrict__ db) {
    __shared__ float red[8][32];
    const int nkt = K / 32;
    const int k0 = (blockIdx.y % nkt) * 32, n0 = (blockIdx.y / nkt) * 32;
    const int el = threadIdx.x & 31, slice = threadIdx.x >> 5;
    const int e = blockIdx.x * 32 + el;
    float s = 0.f;
    if (e < WG_PART) {
        const float* p = part + (size_t)blockIdx.y * nblk * WG_PART + e;
#pragma unroll 8
        for (int b = slice; b < nblk; b += 8) s += p[(size_t)b * WG_PART];
    }
    red[slice][el] = s;
    __syncthreads();
    if (slice != 0 || e >= WG_PART) return;
    s = red[0][el];
    for (int j = 1; j < 8; j++) s += red[j][el];
    if (e < 9 * 32 * 32) {
        const int tap = e / 1024, k = (e / 32) % 32, n = e % 32;
        dw[((size_t)tap * N + n0 + n) * K + k0 + k] = s;
    } else if (k0 == 0) {
        db[n0 + e - 9 * 32 * 32] = s;
    }
}


// 1x1 head C -> 1 in FP32 on top of a base channel of the input: y = base + sum_c w[c] act[c] + b
constexpr int HEAD_C = 32;   // channels into the 1x1 head
constexpr int X0_C = 8;      // channels of the network's input in memory (4 used); c1a's others are zero
__global__ void __launch_bounds__(256) head_fwd(const uint16_t* __restrict__ act, int64_t npix,
                                                const float* __restrict__ w, const float* __restrict__ bias,
                                                const uint16_t* __restrict__ base, int base_cs, int base_co,
                                                float* __restrict__ y) {
    float wv[HEAD_C];
#pragma unroll
    for (int c = 0; c < HEAD_C; c++) wv[c] = w[c];
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < npix; p += (int64_t)gridDim.x * blockDim.x) {
        float s = bias[0] + bf2f(base[p * base_cs + base_co]);
        const uint4* a4 = reinterpret_cast<const uint4*>(act + p * HEAD_C);
#pragma unroll
        for (int q = 0; q < HEAD_C / 8; q++) {
            const uint4 u = a4[q];
#pragma unroll
            for (int k = 0; k < 8; k++) s += wv[8 * q + k] * bf2f((uint16_t)bf_at(u, k));
        }
        y[p] = s;
    }
}
// masked MSE loss: L = mean over counted pixels of (y - t)^2; dy = 2 (y - t) / count
__global__ void mse_loss(const float* __restrict__ y, const float* __restrict__ t, const uint8_t* __restrict__ m,
                         int64_t npix, float inv_count, float* __restrict__ dy, float* __restrict__ loss) {
    float acc = 0;
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < npix; p += (int64_t)gridDim.x * blockDim.x) {
        float e = m[p] ? (y[p] - t[p]) : 0.f;
        dy[p] = 2.f * e * inv_count;
        acc += e * e;
    }
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o);
    __shared__ float red[16];
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        float s = 0.f;
        for (int w = 0; w < (int)(blockDim.x >> 6); w++) s += red[w];
        atomicAdd(loss, s * inv_count);   // one atomic per block (launched with at most 256 blocks)
    }
}
// head backward (C = HEAD_C channels): dw[c] += sum_p dy[p] act[p][c]; db += sum dy;
// gact[p][c] = act[p][c] > 0 ? dy[p] w[c] : 0 in BF16 (the ReLU backward of act fused).  Each
// thread keeps its channel sums in registers; the block adds them with shuffles and one atomic per
// channel.
__global__ void __launch_bounds__(256) head_bwd(const uint16_t* __restrict__ act, int64_t npix,
                                                const float* __restrict__ w, const float* __restrict__ dy,
                                                float* __restrict__ dw, float* __restrict__ db,
                                                uint16_t* __restrict__ gact) {
    __shared__ float red[HEAD_C + 1][4];
    float sw[HEAD_C], sdb = 0.f, wv[HEAD_C];
#pragma unroll
    for (int c = 0; c < HEAD_C; c++) {
        sw[c] = 0.f;
        wv[c] = w[c];
    }
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < npix; p += (int64_t)gridDim.x * blockDim.x) {
        const float d = dy[p];
        const uint4* a4 = reinterpret_cast<const uint4*>(act + p * HEAD_C);
        uint2* o4 = reinterpret_cast<uint2*>(gact + p * HEAD_C);
#pragma unroll
        for (int q = 0; q < HEAD_C / 8; q++) {
            const uint4 u = a4[q];
            const uint32_t uw[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
            for (int e = 0; e < 4; e++) {
                sw[8 * q + 2 * e] += d * bf2f((uint16_t)(uw[e] & 0xFFFFu));
                sw[8 * q + 2 * e + 1] += d * bf2f((uint16_t)(uw[e] >> 16));
            }
            o4[2 * q] = pack_bf16x4(relu_mask4(
                make_float4(d * wv[8 * q], d * wv[8 * q + 1], d * wv[8 * q + 2], d * wv[8 * q + 3]), make_uint2(u.x, u.y)));
            o4[2 * q + 1] = pack_bf16x4(relu_mask4(
                make_float4(d * wv[8 * q + 4], d * wv[8 * q + 5], d * wv[8 * q + 6], d * wv[8 * q + 7]),
                make_uint2(u.z, u.w)));
        }
        sdb += d;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int c = 0; c <= HEAD_C; c++) {
        float v = c < HEAD_C ? sw[c] : sdb;
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
        if (lane == 0) red[c][wave] = v;
    }
    __syncthreads();
    if (threadIdx.x <= HEAD_C) {
        const float v = red[threadIdx.x][0] + red[threadIdx.x][1] + red[threadIdx.x][2] + red[threadIdx.x][3];
        atomicAdd(threadIdx.x < HEAD_C ? &dw[threadIdx.x] : db, v);
    }
}
// Adam (Kingma & Ba 2015) on FP32 master weights: the parameters, their gradients and moments are
// flat arrays of one order (that of sf_cnn_params), so one launch updates them all.
__global__ void __launch_bounds__(256) adam(int64_t n, float* __restrict__ p, const float* __restrict__ g,
                                            float* __restrict__ m, float* __restrict__ v, float lr, float b1, float b2,
                                            float eps, float c1, float c2) {
    for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1 - b1) * gi;
        const float vi = b2 * v[i] + (1 - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        p[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}
// master FP32 weights [tap][n][k] (k < Kreal used, padded to K) -> BF16 forward [tap][n][K] and
// transposed backward [tap][k][n] copies; blockIdx.y is the layer
constexpr int NCONV = 10;
struct PackP {
    const float* wm[NCONV];
    uint16_t *wf[NCONV], *wt[NCONV];
    int N[NCONV], K[NCONV];
};
__global__ void __launch_bounds__(256) pack_weights(const PackP p) {
    const int l = blockIdx.y, N = p.N[l], K = p.K[l];
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < 9 * N * K; i += gridDim.x * blockDim.x) {
        const int k = i % K, q = i / K, n = q % N, tap = q / N;
        const uint16_t h = f2bf(p.wm[l][i]);
        p.wf[l][i] = h;
        p.wt[l][((size_t)tap * K + k) * N + n] = h;
    }
}

}  // namespace sf

// ==========================================================================================
// host: the network, its training loop and the C-ABI
// ==========================================================================================
namespace sf {

struct ConvL {
    int K = 0, N = 0, Kreal = 0;       // padded input channels, output channels, real inputs
    float *wm = nullptr, *b = nullptr, *gw = nullptr, *gb = nullptr;   // in the flat arrays
    uint16_t *wf = nullptr, *wt = nullptr;
    size_t nw() const { return (size_t)9 * N * K; }
};

}  // namespace sf

struct sf_cnn {
    sf_ctx* ctx = nullptr;
    int ni = 0, nj = 0;       // mesh
    int H = 0, W = 0;         // network grid (mesh padded to multiples of 4)
    int Bmax = 0;
    int C1 = sf::HEAD_C, C2 = 64, C3 = 128;
    sf::ConvL L[sf::NCONV];   // in the order of sf_cnn_params
    // flat FP32 arrays of sf_cnn_params' order: parameters, gradients, Adam's moments
    int64_t nparams = 0;
    float *pm = nullptr, *pg = nullptr, *pmom = nullptr, *pvar = nullptr;
    float *hw = nullptr, *hb = nullptr, *ghw = nullptr, *ghb = nullptr;   // the head's parts of pm and pg
    float* loss = nullptr;            // follows the head's gradients: one fill clears all three
    bool packed = false;              // the layers' BF16 copies hold pm
    // activations (BF16 NHWC, no padding between pixels)
    uint16_t *x0 = nullptr, *e1a = nullptr, *e1 = nullptr, *p1 = nullptr, *e2a = nullptr, *e2 = nullptr,
             *p2 = nullptr, *e3a = nullptr, *e3 = nullptr, *d2a = nullptr, *d2 = nullptr, *d1a = nullptr,
             *d1 = nullptr;
    uint16_t *gop = nullptr, *gop2 = nullptr;   // BF16 operand gradients [npix][channels] (backward)
    float* y = nullptr;
    // FP32 gradients of the skip paths, which add to those of the pooled ones
    float *g_s1 = nullptr, *g_s2 = nullptr, *dy = nullptr;
    // dataset
    std::vector<uint16_t*> s_in;      // [H][W][4] BF16: rho, mask, phi_b, 0
    std::vector<float*> s_t;          // [H][W] target phi / phi_ref
    std::vector<uint8_t*> s_m;        // [H][W] 1 on free nodes (loss mask)
    uint8_t* bmask = nullptr;         // batch loss mask
    float* bt = nullptr;              // batch target
    double rho_ref = sf::QE * 1e16, phi_ref = 100.0;
    int adam_t = 0;
    std::mt19937_64 rng{1};
    double* phi_save = nullptr;       // [ni*nj] stash of a context's potential
    float* wpart = nullptr;           // weight-gradient partials: (WG_BLOCKS + 128) x WG_PART
    std::vector<void*> allocs;
};

namespace sf {

// row tiles that a workgroup of a large launch walks: 1 takes 3.17 ms a step (1024 x 512, batch 4), 2 3.10, 4 and 8
// 3.04, 16 3.09
constexpr int CONV_NRT = 4;

static int grid1(int64_t n) {
    int64_t b = (n + 255) / 256;
    return (int)std::max<int64_t>(1, std::min<int64_t>(b, 16384));
}

template <class T>
static int cnn_alloc(sf_cnn* c, T** p, size_t n) {
    *p = nullptr;
    hipError_t e = hipMalloc((void**)p, std::max<size_t>(n, 1) * sizeof(T));
    if (e != hipSuccess) return sf_fail(c->ctx, SF_ERR_OOM, "cnn allocation of %zu bytes failed", n * sizeof(T));
    hipMemset(*p, 0, std::max<size_t>(n, 1) * sizeof(T));
    c->allocs.push_back((void*)*p);
    return SF_OK;
}

// real input channels and output channels of the layers c1a, c1b, c2a, c2b, c3a, c3b, c4a, c4b, c5a, c5b
enum { C1A, C1B, C2A, C2B, C3A, C3B, C4A, C4B, C5A, C5B };
static int conv_init(sf_cnn* c, ConvL& L, std::mt19937_64& rng) {
    const size_t nw = L.nw();
    if (cnn_alloc(c, &L.wf, nw) || cnn_alloc(c, &L.wt, nw)) return SF_ERR_OOM;
    // He initialisation over the real fan-in; padded input channels stay zero
    PolarNormal nd{std::sqrt(2.0 / (9.0 * L.Kreal))};
    std::vector<float> h(nw, 0.f);
    for (int tap = 0; tap < 9; tap++)
        for (int n = 0; n < L.N; n++)
            for (int k = 0; k < L.Kreal; k++) h[((size_t)tap * L.N + n) * L.K + k] = (float)nd(rng);
    if (hipMemcpy(L.wm, h.data(), nw * 4, hipMemcpyHostToDevice) != hipSuccess) return SF_ERR_HIP;
    return SF_OK;
}

static void pack(sf_cnn* c) {
    if (c->packed) return;
    PackP p;
    for (int l = 0; l < NCONV; l++) {
        p.wm[l] = c->L[l].wm;
        p.wf[l] = c->L[l].wf;
        p.wt[l] = c->L[l].wt;
        p.N[l] = c->L[l].N;
        p.K[l] = c->L[l].K;
    }
    hipLaunchKernelGGL(pack_weights, dim3(64, NCONV), dim3(256), 0, c->ctx->stream, p);
    c->packed = true;
}

template <int MODE>
static void conv_launch(sf_cnn* c, ConvP p) {
    const int rows = (p.H + CONV_R - 1) / CONV_R, ntn = p.N / CONV_TN;
    p.gx = (p.W + CONV_TP - 1) / CONV_TP;
    // row tiles per workgroup: up to CONV_NRT while the launch keeps at least 1024 workgroups
    p.nrt = (int)std::max<int64_t>(1, std::min<int64_t>(CONV_NRT, (int64_t)p.gx * rows * p.B * ntn / 1024));
    p.gy = (rows + p.nrt - 1) / p.nrt;
    p.nsp = p.gx * p.gy * p.B;
    hipLaunchKernelGGL(conv3x3_lds<MODE>, dim3((p.nsp + 7) / 8 * 8 * ntn), dim3(256), 0, c->ctx->stream, p);
}
// forward convolution of layer l: in [H][W][in_cs] (after the upsampling of up, kup channels) -> out
// with bias and ReLU, and its 2x2 mean
static void conv_fwd(sf_cnn* c, int l, const uint16_t* in, int in_cs, uint16_t* out, int H, int W, int B,
                     uint16_t* pool = nullptr, const uint16_t* up = nullptr, int kup = 0) {
    const ConvL& L = c->L[l];
    ConvP p = {};
    p.in = in, p.in_cs = in_cs, p.up = up, p.kup = kup, p.K = L.K, p.w = L.wf, p.bias = L.b, p.N = L.N;
    p.out = out, p.pool = pool, p.H = H, p.W = W, p.B = B;
    conv_launch<FWD>(c, p);
}
// weight and bias gradients of layer l for the output gradient g: about WG_BLOCKS workgroups over
// the (32 x 32 channel tile, pixel band) pairs, their partials summed in workgroup order
static void conv_wgrad(sf_cnn* c, int l, const uint16_t* in, int in_cs, const uint16_t* g, int H, int W, int B,
                       const uint16_t* up = nullptr, int kup = 0) {
    const ConvL& L = c->L[l];
    const int nchunks = B * H * ((W + WG_PX - 1) / WG_PX);
    const int pairs = (L.K / 32) * (L.N / 32);
    int nrun = std::max(1, std::min(nchunks, (WG_BLOCKS + pairs - 1) / pairs));
    const int cpb = (nchunks + nrun - 1) / nrun;
    nrun = (nchunks + cpb - 1) / cpb;
    hipLaunchKernelGGL(conv3x3_wgrad_lds, dim3((nrun + 7) / 8 * 8 * pairs), dim3(256), 0, c->ctx->stream, in, in_cs, up,
                       kup, L.K, g, L.N, c->wpart, H, W, B, nrun, cpb);
    hipLaunchKernelGGL(wgrad_reduce, dim3((WG_PART + 31) / 32, pairs), dim3(256), 0, c->ctx->stream,
                       (const float*)c->wpart, nrun, L.K, L.N, L.gw, L.gb);
}
// input gradient of layer l for the output gradient g -> out (see the modes of conv3x3_lds)
template <int MODE>
static void conv_bwd(sf_cnn* c, int l, const uint16_t* g, const uint16_t* act, uint16_t* out, int H, int W, int B,
                     float* skip = nullptr, int nup = 0) {
    const ConvL& L = c->L[l];
    ConvP p = {};
    p.in = g, p.in_cs = L.N, p.K = L.N, p.w = L.wt, p.N = L.K, p.act = act, p.out = out, p.skip = skip, p.nup = nup;
    p.H = H, p.W = W, p.B = B;
    conv_launch<MODE>(c, p);
}

static void forward(sf_cnn* c, int B) {
    const int H = c->H, W = c->W, C1 = c->C1, C2 = c->C2, C3 = c->C3;
    const int H2 = H / 2, W2 = W / 2, H4 = H / 4, W4 = W / 4;
    pack(c);
    conv_fwd(c, C1A, c->x0, X0_C, c->e1a, H, W, B);
    conv_fwd(c, C1B, c->e1a, C1, c->e1, H, W, B, c->p1);
    conv_fwd(c, C2A, c->p1, C1, c->e2a, H2, W2, B);
    conv_fwd(c, C2B, c->e2a, C2, c->e2, H2, W2, B, c->p2);
    conv_fwd(c, C3A, c->p2, C2, c->e3a, H4, W4, B);
    conv_fwd(c, C3B, c->e3a, C3, c->e3, H4, W4, B);
    conv_fwd(c, C4A, c->e2, C2, c->d2a, H2, W2, B, nullptr, c->e3, C3);
    conv_fwd(c, C4B, c->d2a, C2, c->d2, H2, W2, B);
    conv_fwd(c, C5A, c->e1, C1, c->d1a, H, W, B, nullptr, c->d2, C2);
    conv_fwd(c, C5B, c->d1a, C1, c->d1, H, W, B);
    hipLaunchKernelGGL(head_fwd, dim3(grid1((int64_t)B * H * W)), dim3(256), 0, c->ctx->stream, (const uint16_t*)c->d1,
                       (int64_t)B * H * W, (const float*)c->hw, (const float*)c->hb, (const uint16_t*)c->x0, X0_C, 3,
                       c->y);
}

// The BF16 operand gradients alternate between gop and gop2 (a layer's backward reads one and
// writes the next into the other); every ReLU backward is fused into the kernel that produces the
// gradient of the activation.  FP32 gradients remain only where two paths add: the skip inputs of
// the decoder convolutions, which wait for the pooled activations' gradients.
static void backward(sf_cnn* c, int B) {
    const int H = c->H, W = c->W, C1 = c->C1, C2 = c->C2, C3 = c->C3;
    const int H2 = H / 2, W2 = W / 2, H4 = H / 4, W4 = W / 4;
    uint16_t* ga = c->gop;
    uint16_t* gb = c->gop2;
    hipLaunchKernelGGL(head_bwd, dim3(1024), dim3(256), 0, c->ctx->stream, (const uint16_t*)c->d1, (int64_t)B * H * W,
                       (const float*)c->hw, (const float*)c->dy, c->ghw, c->ghb, ga);
    conv_wgrad(c, C5B, c->d1a, C1, ga, H, W, B);
    conv_bwd<BWD_RELU>(c, C5B, ga, c->d1a, gb, H, W, B);
    conv_wgrad(c, C5A, c->e1, C1, gb, H, W, B, c->d2, C2);
    conv_bwd<BWD_UP>(c, C5A, gb, c->d2, ga, H, W, B, c->g_s1, C2);
    conv_wgrad(c, C4B, c->d2a, C2, ga, H2, W2, B);
    conv_bwd<BWD_RELU>(c, C4B, ga, c->d2a, gb, H2, W2, B);
    conv_wgrad(c, C4A, c->e2, C2, gb, H2, W2, B, c->e3, C3);
    conv_bwd<BWD_UP>(c, C4A, gb, c->e3, ga, H2, W2, B, c->g_s2, C3);
    conv_wgrad(c, C3B, c->e3a, C3, ga, H4, W4, B);
    conv_bwd<BWD_RELU>(c, C3B, ga, c->e3a, gb, H4, W4, B);
    conv_wgrad(c, C3A, c->p2, C2, gb, H4, W4, B);
    conv_bwd<BWD_POOL>(c, C3A, gb, c->e2, ga, H4, W4, B, c->g_s2);
    conv_wgrad(c, C2B, c->e2a, C2, ga, H2, W2, B);
    conv_bwd<BWD_RELU>(c, C2B, ga, c->e2a, gb, H2, W2, B);
    conv_wgrad(c, C2A, c->p1, C1, gb, H2, W2, B);
    conv_bwd<BWD_POOL>(c, C2A, gb, c->e1, ga, H2, W2, B, c->g_s1);
    conv_wgrad(c, C1B, c->e1a, C1, ga, H, W, B);
    conv_bwd<BWD_RELU>(c, C1B, ga, c->e1a, gb, H, W, B);
    conv_wgrad(c, C1A, c->x0, X0_C, gb, H, W, B);
}

// place sample s into batch slot b of x0 / target / mask
__global__ void assemble_batch(const uint16_t* __restrict__ sin, const float* __restrict__ st,
                               const uint8_t* __restrict__ sm, int64_t npix, uint16_t* __restrict__ x0,
                               float* __restrict__ bt, uint8_t* __restrict__ bm) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < npix; p += (int64_t)gridDim.x * blockDim.x) {
        const uint2 u = *reinterpret_cast<const uint2*>(sin + p * 4);
        *reinterpret_cast<uint4*>(x0 + p * X0_C) = make_uint4(u.x, u.y, 0u, 0u);
        bt[p] = st[p];
        bm[p] = sm[p];
    }
}
// Snapshot of a context on the padded grid: input channels (rho / rho_ref, Dirichlet mask,
// boundary phi / phi_ref, Boltzmann inversion (phi0 + kTe ln max(rho / (e n0), 1)) / phi_ref),
// target phi / phi_ref and the free-node mask.  Pixels outside the mesh are zero, and so are channels
// from 4 up to the stride cs (a multiple of 4).
__global__ void snapshot_kernel(int ni, int nj, int H, int W, const double* __restrict__ rho,
                                const double* __restrict__ phi, const int32_t* __restrict__ src,
                                const uint8_t* __restrict__ cls, const double* __restrict__ fixval, double inv_rho,
                                double inv_phi, double inv_en0, double kTe, double phi0,
                                uint16_t* __restrict__ sin, int cs, float* __restrict__ st,
                                uint8_t* __restrict__ sm) {
    for (int64_t p = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; p < (int64_t)H * W; p += (int64_t)gridDim.x * blockDim.x) {
        int x = (int)(p % W), y = (int)(p / W);
        uint16_t r = 0, mk = 0, pb = 0, bz = 0;
        float t = 0;
        uint8_t m = 0;
        if (x < ni && y < nj) {
            size_t u = (size_t)y * ni + x;
            bool fixed = src[u] < 0;
            r = f2bf((float)(rho[u] * inv_rho));
            mk = f2bf(fixed ? 1.f : 0.f);
            pb = f2bf(fixed ? (float)(fixval[u] * inv_phi) : 0.f);
            if (kTe > 0) bz = f2bf((float)((phi0 + kTe * log(fmax(rho[u] * inv_en0, 1.0))) * inv_phi));
            if (phi) t = (float)(phi[u] * inv_phi);
            m = cls[u] != 0xFF ? 1 : 0;
        }
        *reinterpret_cast<uint2*>(sin + p * cs) = make_uint2((uint32_t)r | (uint32_t)mk << 16, (uint32_t)pb | (uint32_t)bz << 16);
        for (int k = 4; k < cs; k += 4) *reinterpret_cast<uint2*>(sin + p * cs + k) = make_uint2(0u, 0u);
        if (st) st[p] = t;
        if (sm) sm[p] = m;
    }
}
// network output -> phi on the free nodes of the context (fixed / face nodes set by the solver)
__global__ void guess_to_phi(int ni, int nj, int W, const float* __restrict__ y, double phi_ref,
                             double* __restrict__ phi) {
    for (int64_t u = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; u < (int64_t)ni * nj; u += (int64_t)gridDim.x * blockDim.x) {
        int x = (int)(u % ni), yy = (int)(u / ni);
        phi[u] = (double)y[(size_t)yy * W + x] * phi_ref;
    }
}

}  // namespace sf

// accessors used by the solver (defined in sf_poisson.hip)
namespace sf {
const int32_t* poisson_src(sf_ctx* ctx);
const uint8_t* poisson_cls(sf_ctx* ctx);
const double* poisson_fixval(sf_ctx* ctx);
const sf_poisson_desc* poisson_desc(sf_ctx* ctx);
int poisson_rel_residual(sf_ctx* ctx, double* rel);

// parameters of the Boltzmann-inversion input channel (zero channel for a linear solver)
static double feat_kTe(sf_ctx* t) { return poisson_desc(t)->linear ? 0.0 : poisson_desc(t)->Te0; }
static double feat_inv_en0(sf_ctx* t) {
    double n0 = poisson_desc(t)->n0;
    return n0 > 0 ? 1.0 / (QE * n0) : 0.0;
}
}

using namespace sf;

extern "C" {

int sf_cnn_create(sf_ctx* ctx, int ni, int nj, int max_batch, uint64_t seed, sf_cnn** out) {
    SF_CHECK_CTX(ctx);
    if (!out || max_batch < 1 || max_batch > 64) return sf_fail(ctx, SF_ERR_ARG, "sf_cnn_create: bad argument");
    if (ni <= 0 || nj <= 0) {
        if (!ctx->mesh_ready) return sf_fail(ctx, SF_ERR_STATE, "sf_cnn_create: no size given and no mesh");
        ni = ctx->mp.ni;
        nj = ctx->mp.nj;
    }
    if (ni > 16384 || nj > 16384) return sf_fail(ctx, SF_ERR_ARG, "sf_cnn_create: grid too large");
    SF_HIP(ctx, hipSetDevice(ctx->device));
    sf_cnn* c = new sf_cnn();
    c->ctx = ctx;
    c->ni = ni;
    c->nj = nj;
    c->W = (c->ni + 3) / 4 * 4;
    c->H = (c->nj + 3) / 4 * 4;
    c->Bmax = max_batch;
    c->rng.seed(seed);
    const int C1 = c->C1, C2 = c->C2, C3 = c->C3;
    const int64_t n1 = (int64_t)max_batch * c->H * c->W, n2 = n1 / 4, n4 = n1 / 16;
    int rc = 0;
    const int kn[NCONV][2] = {{4, C1},  {C1, C1},      {C1, C2}, {C2, C2},      {C2, C3},
                              {C3, C3}, {C3 + C2, C2}, {C2, C2}, {C2 + C1, C1}, {C1, C1}};
    for (int l = 0; l < NCONV; l++) {
        c->L[l].Kreal = kn[l][0];
        c->L[l].K = (kn[l][0] + 31) / 32 * 32;
        c->L[l].N = kn[l][1];
        c->nparams += (int64_t)c->L[l].nw() + c->L[l].N;
    }
    c->nparams += C1 + 1;
    rc |= cnn_alloc(c, &c->pm, c->nparams);
    rc |= cnn_alloc(c, &c->pg, c->nparams + 1);
    rc |= cnn_alloc(c, &c->pmom, c->nparams);
    rc |= cnn_alloc(c, &c->pvar, c->nparams);
    if (!rc) {
        int64_t off = 0;
        for (ConvL& L : c->L) {
            L.wm = c->pm + off, L.gw = c->pg + off;
            off += (int64_t)L.nw();
            L.b = c->pm + off, L.gb = c->pg + off;
            off += L.N;
        }
        c->hw = c->pm + off, c->ghw = c->pg + off;
        c->hb = c->hw + C1, c->ghb = c->ghw + C1;
        c->loss = c->ghb + 1;
        for (ConvL& L : c->L) rc |= conv_init(c, L, c->rng);
    }
    // (a launch has at most ceil(WG_BLOCKS / pairs) * pairs <= WG_BLOCKS + pairs - 1 workgroups;
    // the network's layers have at most 16 channel tile pairs)
    rc |= cnn_alloc(c, &c->wpart, (size_t)(WG_BLOCKS + 128) * WG_PART);
    rc |= cnn_alloc(c, &c->x0, n1 * X0_C);
    rc |= cnn_alloc(c, &c->e1a, n1 * C1);
    rc |= cnn_alloc(c, &c->e1, n1 * C1);
    rc |= cnn_alloc(c, &c->p1, n2 * C1);
    rc |= cnn_alloc(c, &c->e2a, n2 * C2);
    rc |= cnn_alloc(c, &c->e2, n2 * C2);
    rc |= cnn_alloc(c, &c->p2, n4 * C2);
    rc |= cnn_alloc(c, &c->e3a, n4 * C3);
    rc |= cnn_alloc(c, &c->e3, n4 * C3);
    rc |= cnn_alloc(c, &c->d2a, n2 * C2);
    rc |= cnn_alloc(c, &c->d2, n2 * C2);
    rc |= cnn_alloc(c, &c->d1a, n1 * C1);
    rc |= cnn_alloc(c, &c->d1, n1 * C1);
    rc |= cnn_alloc(c, &c->gop, n1 * C1);    // (n2 C2 and n4 C3 are smaller)
    rc |= cnn_alloc(c, &c->gop2, n1 * C1);
    rc |= cnn_alloc(c, &c->y, n1);
    rc |= cnn_alloc(c, &c->g_s1, n1 * C1);
    rc |= cnn_alloc(c, &c->g_s2, n2 * C2);
    rc |= cnn_alloc(c, &c->dy, n1);
    rc |= cnn_alloc(c, &c->bt, n1);
    rc |= cnn_alloc(c, &c->bmask, n1);
    rc |= cnn_alloc(c, &c->phi_save, (size_t)ni * nj);
    if (rc) {
        for (void* p : c->allocs) hipFree(p);
        delete c;
        return SF_ERR_OOM;
    }
    PolarNormal nd{std::sqrt(1.0 / C1)};
    std::vector<float> h(C1);
    for (auto& v : h) v = (float)nd(c->rng);
    SF_HIP(ctx, hipMemcpy(c->hw, h.data(), C1 * 4, hipMemcpyHostToDevice));
    SF_HIP(ctx, hipDeviceSynchronize());
    *out = c;
    return SF_OK;
}

int sf_cnn_destroy(sf_cnn* c) {
    if (!c) return SF_ERR_ARG;
    hipSetDevice(c->ctx->device);
    hipStreamSynchronize(c->ctx->stream);
    for (void* p : c->allocs) hipFree(p);
    for (auto* p : c->s_in) hipFree(p);
    for (auto* p : c->s_t) hipFree(p);
    for (auto* p : c->s_m) hipFree(p);
    delete c;
    return SF_OK;
}

int sf_cnn_num_samples(const sf_cnn* c) { return c ? (int)c->s_in.size() : SF_ERR_ARG; }

int sf_cnn_dims(const sf_cnn* c, int* H, int* W, int64_t* nparams) {
    if (!c) return SF_ERR_ARG;
    if (H) *H = c->H;
    if (W) *W = c->W;
    if (nparams) *nparams = c->nparams;
    return SF_OK;
}

// Adds a training sample given on the host: x4 [H][W][4] FP32 input channels (stored as BF16),
// t [H][W] FP32 target, m [H][W] loss mask.
int sf_cnn_add_sample(sf_cnn* c, const float* x4, const float* t, const uint8_t* m) {
    if (!c || !x4 || !t || !m) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    SF_HIP(ctx, hipSetDevice(ctx->device));
    const int64_t np = (int64_t)c->H * c->W;
    std::vector<uint16_t> h(np * 4);
    for (int64_t i = 0; i < np * 4; i++) h[i] = f2bf(x4[i]);
    uint16_t* sin = nullptr;
    float* st = nullptr;
    uint8_t* sm = nullptr;
    SF_HIP(ctx, hipMalloc((void**)&sin, np * 8));
    SF_HIP(ctx, hipMalloc((void**)&st, np * 4));
    SF_HIP(ctx, hipMalloc((void**)&sm, np));
    SF_HIP(ctx, hipMemcpy(sin, h.data(), np * 8, hipMemcpyHostToDevice));
    SF_HIP(ctx, hipMemcpy(st, t, np * 4, hipMemcpyHostToDevice));
    SF_HIP(ctx, hipMemcpy(sm, m, np, hipMemcpyHostToDevice));
    c->s_in.push_back(sin);
    c->s_t.push_back(st);
    c->s_m.push_back(sm);
    return SF_OK;
}

// Reads back sample idx (input channels as stored, i.e. BF16-rounded, widened to FP32).
int sf_cnn_get_sample(sf_cnn* c, int idx, float* x4, float* t, uint8_t* m) {
    if (!c || idx < 0 || idx >= (int)c->s_in.size()) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    SF_HIP(ctx, hipSetDevice(ctx->device));
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    const int64_t np = (int64_t)c->H * c->W;
    if (x4) {
        std::vector<uint16_t> h(np * 4);
        SF_HIP(ctx, hipMemcpy(h.data(), c->s_in[idx], np * 8, hipMemcpyDeviceToHost));
        for (int64_t i = 0; i < np * 4; i++) x4[i] = bf2f(h[i]);
    }
    if (t) SF_HIP(ctx, hipMemcpy(t, c->s_t[idx], np * 4, hipMemcpyDeviceToHost));
    if (m) SF_HIP(ctx, hipMemcpy(m, c->s_m[idx], np, hipMemcpyDeviceToHost));
    return SF_OK;
}

// Adds the current (rho, Dirichlet mask / values, phi) of `src_ctx` to the training set.
int sf_cnn_snapshot(sf_cnn* c, sf_ctx* src_ctx) {
    if (!c || !src_ctx) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    if (src_ctx->mp.ni != c->ni || src_ctx->mp.nj != c->nj || !src_ctx->poisson)
        return sf_fail(ctx, SF_ERR_ARG, "sf_cnn_snapshot: context has another mesh size or no solver");
    SF_HIP(ctx, hipSetDevice(ctx->device));
    SF_HIP(ctx, hipStreamSynchronize(src_ctx->stream));
    const int64_t np = (int64_t)c->H * c->W;
    uint16_t* sin = nullptr;
    float* st = nullptr;
    uint8_t* sm = nullptr;
    SF_HIP(ctx, hipMalloc((void**)&sin, np * 8));
    SF_HIP(ctx, hipMalloc((void**)&st, np * 4));
    SF_HIP(ctx, hipMalloc((void**)&sm, np));
    hipLaunchKernelGGL(snapshot_kernel, dim3(grid1(np)), dim3(256), 0, ctx->stream, c->ni, c->nj, c->H, c->W,
                       (const double*)src_ctx->d_rho, (const double*)src_ctx->d_phi, poisson_src(src_ctx),
                       poisson_cls(src_ctx), poisson_fixval(src_ctx), 1.0 / c->rho_ref, 1.0 / c->phi_ref,
                       feat_inv_en0(src_ctx), feat_kTe(src_ctx), poisson_desc(src_ctx)->phi0, sin, 4, st, sm);
    SF_HIP(ctx, hipGetLastError());
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    c->s_in.push_back(sin);
    c->s_t.push_back(st);
    c->s_m.push_back(sm);
    return SF_OK;
}

// clears what the kernels of a step add to: the head's gradients and the loss
static hipError_t clear_sums(sf_cnn* c) {
    return hipMemsetAsync(c->ghw, 0, (c->C1 + 2) * sizeof(float), c->ctx->stream);
}

// Adam training on random mini-batches of the snapshots; returns the mean loss of the last
// `steps/10` steps in *loss_out (normalised MSE of phi / 100 V on free nodes).
int sf_cnn_train(sf_cnn* c, int steps, int batch, double lr, double* loss_out) {
    if (!c) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    if (c->s_in.empty()) return sf_fail(ctx, SF_ERR_STATE, "sf_cnn_train: no snapshots");
    if (batch < 1 || batch > c->Bmax || steps < 0) return sf_fail(ctx, SF_ERR_ARG, "sf_cnn_train: bad batch/steps");
    SF_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    const int64_t np = (int64_t)c->H * c->W;
    std::uniform_int_distribution<int> pick(0, (int)c->s_in.size() - 1);
    double tail = 0;
    int ntail = 0;
    for (int s = 0; s < steps; s++) {
        int64_t counted = 0;
        for (int b = 0; b < batch; b++) {
            int k = pick(c->rng);
            hipLaunchKernelGGL(assemble_batch, dim3(grid1(np)), dim3(256), 0, st, (const uint16_t*)c->s_in[k],
                               (const float*)c->s_t[k], (const uint8_t*)c->s_m[k], np, c->x0 + b * np * X0_C,
                               c->bt + b * np, c->bmask + b * np);
            counted += np;
        }
        SF_HIP(ctx, clear_sums(c));
        forward(c, batch);
        hipLaunchKernelGGL(mse_loss, dim3(std::min(grid1((int64_t)batch * np), 256)), dim3(256), 0, st, (const float*)c->y,
                           (const float*)c->bt, (const uint8_t*)c->bmask, (int64_t)batch * np, 1.0f / (float)counted,
                           c->dy, c->loss);
        backward(c, batch);
        c->adam_t++;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.f - powf(b1, (float)c->adam_t), c2 = 1.f - powf(b2, (float)c->adam_t);
        hipLaunchKernelGGL(adam, dim3(grid1(c->nparams)), dim3(256), 0, st, c->nparams, c->pm, (const float*)c->pg,
                           c->pmom, c->pvar, (float)lr, b1, b2, 1e-8f, c1, c2);
        c->packed = false;
        SF_HIP(ctx, hipGetLastError());
        if (s >= steps - std::max(1, steps / 10)) {
            float l = 0;
            SF_HIP(ctx, hipMemcpyAsync(&l, c->loss, 4, hipMemcpyDeviceToHost, st));
            SF_HIP(ctx, hipStreamSynchronize(st));
            tail += l;
            ntail++;
        }
    }
    SF_HIP(ctx, hipStreamSynchronize(st));
    if (loss_out) *loss_out = ntail ? tail / ntail : 0.0;
    return SF_OK;
}

// Loss and all parameter gradients of one sample (for gradient checks).  grads_out receives the
// gradients in the order of sf_cnn_params; n_out the total count.
int sf_cnn_loss_and_grads(sf_cnn* c, int sample, double* loss_out, float* y_out, float* grads_out,
                          int64_t* n_out) {
    if (!c || sample < 0 || sample >= (int)c->s_in.size()) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    SF_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    const int64_t np = (int64_t)c->H * c->W;
    hipLaunchKernelGGL(assemble_batch, dim3(grid1(np)), dim3(256), 0, st, (const uint16_t*)c->s_in[sample],
                       (const float*)c->s_t[sample], (const uint8_t*)c->s_m[sample], np, c->x0, c->bt, c->bmask);
    SF_HIP(ctx, clear_sums(c));
    forward(c, 1);
    hipLaunchKernelGGL(mse_loss, dim3(std::min(grid1(np), 256)), dim3(256), 0, st, (const float*)c->y, (const float*)c->bt,
                       (const uint8_t*)c->bmask, np, 1.0f / (float)np, c->dy, c->loss);
    backward(c, 1);
    SF_HIP(ctx, hipGetLastError());
    float l = 0;
    SF_HIP(ctx, hipMemcpyAsync(&l, c->loss, 4, hipMemcpyDeviceToHost, st));
    SF_HIP(ctx, hipStreamSynchronize(st));
    if (loss_out) *loss_out = l;
    if (y_out) SF_HIP(ctx, hipMemcpy(y_out, c->y, np * 4, hipMemcpyDeviceToHost));
    if (grads_out) SF_HIP(ctx, hipMemcpy(grads_out, c->pg, c->nparams * 4, hipMemcpyDeviceToHost));
    if (n_out) *n_out = c->nparams;
    return SF_OK;
}

// Diagnostic read-back of an activation of batch slot 0 after the last forward pass, widened to
// FP32: which = 0 x0 [H][W][32], 1 e1a, 2 u1 [.][96], 3 p1, 4 e2a, 5 u2 [.][192], 6 p2, 7 e3a,
// 8 e3, 9 d2a, 10 d2, 11 d1a, 12 d1, 13 y [H][W].  *count receives the number of values.
int sf_cnn_activation(sf_cnn* c, int which, float* out, int64_t* count) {
    if (!c) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    const int64_t n1 = (int64_t)c->H * c->W, n2 = n1 / 4, n4 = n1 / 16;
    const int C1 = c->C1, C2 = c->C2, C3 = c->C3;
    // the tensor's channels [0, ca) are `a` (upsampled from half the width where up), [ca, ca + cb) are `b`
    const uint16_t *a = nullptr, *b = nullptr;
    int ca = 0, cb = 0, pad = 0, w = c->W;
    bool up = false;
    int64_t npix = n1;
    switch (which) {
        case 0: a = c->x0; ca = X0_C; pad = 32 - X0_C; break;
        case 1: a = c->e1a; ca = C1; break;
        case 2: a = c->d2; ca = C2; up = true; b = c->e1; cb = C1; break;
        case 3: a = c->p1; ca = C1; npix = n2; break;
        case 4: a = c->e2a; ca = C2; npix = n2; break;
        case 5: a = c->e3; ca = C3; up = true; b = c->e2; cb = C2; npix = n2; w = c->W / 2; break;
        case 6: a = c->p2; ca = C2; npix = n4; break;
        case 7: a = c->e3a; ca = C3; npix = n4; break;
        case 8: a = c->e3; ca = C3; npix = n4; break;
        case 9: a = c->d2a; ca = C2; npix = n2; break;
        case 10: a = c->d2; ca = C2; npix = n2; break;
        case 11: a = c->d1a; ca = C1; break;
        case 12: a = c->d1; ca = C1; break;
        case 13: ca = 1; break;
        default: return sf_fail(ctx, SF_ERR_ARG, "sf_cnn_activation: unknown tensor %d", which);
    }
    const int C = ca + cb + pad;
    if (count) *count = npix * C;
    if (!out) return SF_OK;
    SF_HIP(ctx, hipSetDevice(ctx->device));
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (which == 13) {
        SF_HIP(ctx, hipMemcpy(out, c->y, npix * 4, hipMemcpyDeviceToHost));
        return SF_OK;
    }
    std::vector<uint16_t> ha((up ? npix / 4 : npix) * ca), hb(npix * cb);
    SF_HIP(ctx, hipMemcpy(ha.data(), a, ha.size() * 2, hipMemcpyDeviceToHost));
    if (cb) SF_HIP(ctx, hipMemcpy(hb.data(), b, hb.size() * 2, hipMemcpyDeviceToHost));
    for (int64_t q = 0; q < npix; q++) {
        const int64_t qa = up ? (q / w / 2) * (w / 2) + q % w / 2 : q;
        for (int k = 0; k < C; k++)
            out[q * C + k] = k < ca ? bf2f(ha[qa * ca + k]) : (k < ca + cb ? bf2f(hb[q * cb + k - ca]) : 0.f);
    }
    return SF_OK;
}

// parameters (FP32 master copies) in a fixed order: for each of the 10 convolutions
// W[9][N][K] then b[N]; then the head w[C1], b[1]. get = 1 downloads, get = 0 uploads.
int sf_cnn_params(sf_cnn* c, int get, float* buf, int64_t* n_out) {
    if (!c) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    SF_HIP(ctx, hipSetDevice(ctx->device));
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (buf && get) SF_HIP(ctx, hipMemcpy(buf, c->pm, c->nparams * 4, hipMemcpyDeviceToHost));
    if (buf && !get) {
        c->packed = false;
        SF_HIP(ctx, hipMemcpy(c->pm, buf, c->nparams * 4, hipMemcpyHostToDevice));
    }
    if (n_out) *n_out = c->nparams;
    return SF_OK;
}

int sf_cnn_predict(sf_cnn* c, sf_ctx* target);

// Potential solve started from the network's guess.  policy 0: always start from the guess;
// policy 1: start from whichever of the current potential and the guess has the smaller
// nonlinear residual (the guess is discarded when it does not help).  info->newton_iterations
// etc. describe the solve; *used_guess (may be NULL) tells which start was taken.
int sf_poisson_solve_learned(sf_ctx* ctx, sf_cnn* c, int policy, sf_solve_info* info, int* used_guess) {
    SF_CHECK_CTX(ctx);
    if (!c || (policy != 0 && policy != 1)) return sf_fail(ctx, SF_ERR_ARG, "sf_poisson_solve_learned: bad argument");
    if (!ctx->poisson) return sf_fail(ctx, SF_ERR_STATE, "sf_poisson_solve_learned: solver not set up");
    if (ctx->mp.ni != c->ni || ctx->mp.nj != c->nj)
        return sf_fail(ctx, SF_ERR_ARG, "sf_poisson_solve_learned: network grid differs from the mesh");
    SF_HIP(ctx, hipSetDevice(ctx->device));
    const size_t nn = (size_t)c->ni * c->nj;
    double r_prev = 0, r_guess = 0;
    if (policy == 1) {
        int rc = poisson_rel_residual(ctx, &r_prev);
        if (rc < 0) return rc;
    }
    SF_HIP(ctx, hipMemcpyAsync(c->phi_save, ctx->d_phi, nn * 8, hipMemcpyDeviceToDevice, ctx->stream));
    int rc = sf_cnn_predict(c, ctx);
    if (rc < 0) return sf_fail(ctx, rc, "sf_poisson_solve_learned: prediction failed: %s", c->ctx->err.c_str());
    // The guess is only a starting point: one whose nonlinear residual is not finite (exp of a
    // wild potential), or worse than the previous potential's under policy 1, is replaced by the
    // previous potential, and a solve that diverges from the guess is repeated from it.
    rc = poisson_rel_residual(ctx, &r_guess);
    if (rc < 0) return rc;
    bool use = std::isfinite(r_guess) && (policy == 0 || r_guess < r_prev);
    auto restore = [&]() -> int {
        SF_HIP(ctx, hipMemcpyAsync(ctx->d_phi, c->phi_save, nn * 8, hipMemcpyDeviceToDevice, ctx->stream));
        return SF_OK;
    };
    if (!use && (rc = restore()) < 0) return rc;
    rc = poisson_solve(ctx, info);
    if (rc < 0 && use) {
        use = false;
        if ((rc = restore()) < 0) return rc;
        rc = poisson_solve(ctx, info);
    }
    if (used_guess) *used_guess = use ? 1 : 0;
    return rc;
}

// Network output for the current state of `target` (rho, Dirichlet values) written as phi.
int sf_cnn_predict(sf_cnn* c, sf_ctx* target) {
    if (!c || !target) return SF_ERR_ARG;
    sf_ctx* ctx = c->ctx;
    if (target->mp.ni != c->ni || target->mp.nj != c->nj || !target->poisson)
        return sf_fail(ctx, SF_ERR_ARG, "sf_cnn_predict: context has another mesh size or no solver");
    SF_HIP(ctx, hipSetDevice(ctx->device));
    SF_HIP(ctx, hipStreamSynchronize(target->stream));
    const int64_t np = (int64_t)c->H * c->W;
    hipLaunchKernelGGL(snapshot_kernel, dim3(grid1(np)), dim3(256), 0, ctx->stream, c->ni, c->nj, c->H, c->W,
                       (const double*)target->d_rho, (const double*)nullptr, poisson_src(target), poisson_cls(target),
                       poisson_fixval(target), 1.0 / c->rho_ref, 1.0 / c->phi_ref, feat_inv_en0(target),
                       feat_kTe(target), poisson_desc(target)->phi0, c->x0, X0_C, (float*)nullptr, (uint8_t*)nullptr);
    forward(c, 1);
    hipLaunchKernelGGL(guess_to_phi, dim3(grid1((int64_t)c->ni * c->nj)), dim3(256), 0, ctx->stream, c->ni, c->nj,
                       c->W, (const float*)c->y, c->phi_ref, target->d_phi);
    SF_HIP(ctx, hipGetLastError());
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return SF_OK;
}

// MFMA lane-layout probe: D = A(16x32) * B(32x16) with the operand layout the convolution
// kernels assume; host compares against a plain product.
__global__ void mfma_probe_kernel(const uint16_t* a, const uint16_t* b, float* d) {
    const int lane = threadIdx.x;
    bf16x8 av, bv;
    uint16_t ta[8], tb[8];
    for (int j = 0; j < 8; j++) {
        ta[j] = a[(lane & 15) * 32 + (lane >> 4) * 8 + j];   // A[row][k]
        tb[j] = b[((lane >> 4) * 8 + j) * 16 + (lane & 15)];  // B[k][col]
    }
    memcpy(&av, ta, 16);
    memcpy(&bv, tb, 16);
    f32x4 acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, bv, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
    for (int i = 0; i < 4; i++) d[((lane >> 4) * 4 + i) * 16 + (lane & 15)] = acc[i];
}

int sf_cnn_mfma_probe(sf_ctx* ctx, const float* a, const float* b, float* d) {
    SF_CHECK_CTX(ctx);
    SF_HIP(ctx, hipSetDevice(ctx->device));
    std::vector<uint16_t> ha(16 * 32), hb(32 * 16);
    for (int i = 0; i < 16 * 32; i++) ha[i] = f2bf(a[i]);
    for (int i = 0; i < 32 * 16; i++) hb[i] = f2bf(b[i]);
    uint16_t *da = nullptr, *db = nullptr;
    float* dd = nullptr;
    SF_HIP(ctx, hipMalloc((void**)&da, 16 * 32 * 2));
    SF_HIP(ctx, hipMalloc((void**)&db, 32 * 16 * 2));
    SF_HIP(ctx, hipMalloc((void**)&dd, 16 * 16 * 4));
    SF_HIP(ctx, hipMemcpy(da, ha.data(), 16 * 32 * 2, hipMemcpyHostToDevice));
    SF_HIP(ctx, hipMemcpy(db, hb.data(), 32 * 16 * 2, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, ctx->stream, (const uint16_t*)da, (const uint16_t*)db,
                       dd);
    SF_HIP(ctx, hipGetLastError());
    SF_HIP(ctx, hipStreamSynchronize(ctx->stream));
    SF_HIP(ctx, hipMemcpy(d, dd, 16 * 16 * 4, hipMemcpyDeviceToHost));
    hipFree(da);
    hipFree(db);
    hipFree(dd);
    return SF_OK;
}

}  // extern "C"
