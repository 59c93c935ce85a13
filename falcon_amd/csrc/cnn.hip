// Learned V-cycle correction network on MFMA (gfx950): forward (fused, all
// three layers in LDS), data and weight gradients (implicit GEMM on
// v_mfma_f32_16x16x32_bf16 / 16x16x16_bf16), mean-squared-error loss and Adam.
//
// MFMA operand images (64 lanes, lane l = 16 g + n):
//   16x16x32: A lane l holds A[n][8g .. 8g+7], B lane l holds B[8g .. 8g+7][n]
//   16x16x16: A lane l holds A[n][4g .. 4g+3], B lane l holds B[4g .. 4g+3][n]
//   D (16 x 16): lane l holds D[4g .. 4g+3][n]
// A convolution is computed as D = W^T X: rows = output channels, columns =
// 16 voxels of one k-line, K = (tap, input channel) pairs, so each lane ends
// with 4 consecutive output channels of one voxel (one 8-byte store of
// channel-fastest activations).
//
// Layouts: images x/out [img][4096] float; activations and their gradients
// [img][4096][16] bfloat16 (channel fastest); voxel v = (i*16 + j)*16 + k.
// LDS planes: x [18][18] with a zero halo; forward activations [16][16][16]
// (k-shifts by DPP, out-of-block lines skipped); the gradient kernels' carves are
// described there.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "cnn.hpp"

namespace falcon {

#define CCHECK(x)                                                                                     \
    do {                                                                                              \
        hipError_t e_ = (x);                                                                          \
        if (e_ != hipSuccess) throw std::runtime_error(std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

typedef unsigned short us8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef short s4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

namespace {

constexpr int PL = 18 * 18;                 // plane with halo
constexpr int OFF_W1 = 0, OFF_B1 = 432, OFF_W2 = 448, OFF_B2 = 7360, OFF_W3 = 7376, OFF_B3 = 7808;
// packed operand images of the 16x16x32 form, 64 lanes x 8 bf16 per MFMA step:
// Q3 layer-3 data gradient (1 step), Q2 layer-2 data gradient (14)
constexpr int PK_Q3 = 0, PK_Q2 = 64, PK_TOTAL = PK_Q2 + 14 * 64;

// forward operand images (bf16 elements, lane-major):
//   L1  [3 di][64] x 4: 16x16x16 A, rows co, K = the 9 (dj,dk) taps of plane offset di
//   L2A [9 (di,dj)][64] x 8: 16x16x32 A, rows co, K = (dk = -1: ci 0..15, dk = +1: ci 0..15)
//   L2B [9 (di,dj)][64] x 4: 16x16x16 A, rows co, K = ci of tap dk = 0
//   L3  [3 di][64] x 4: 16x16x16 A, rows r = 4 (dj+1) + (dk+1) (r % 4 < 3, r < 12), K = ci
constexpr int PF_L1 = 0, PF_L2A = PF_L1 + 3 * 64 * 4, PF_L2B = PF_L2A + 9 * 64 * 8, PF_L3 = PF_L2B + 9 * 64 * 4,
              PF_TOTAL = PF_L3 + 3 * 64 * 4;
// fused forward LDS carve (uint16 elements): h1 and h2 rings of 3 planes, each
// [18 j][4 channel groups][18 k][4 c] with zero halo rows and voxels (a lane's
// 8-byte access is consecutive to its neighbour's: no bank conflicts); x ring
// of 3 planes [18][18] with a zero halo
constexpr int HGRP = 18 * 4, HROW = 4 * HGRP, HPL = 18 * HROW;
constexpr int kFwdWaves = 8;                // wavefronts per image (16 / kFwdWaves k-lines each)
constexpr int F_H1 = 0, F_H2 = 3 * HPL, F_X = 6 * HPL, F_TOTAL = F_X + 3 * PL;

__device__ __forceinline__ uint16_t f2bf(float f) {
    uint32_t u = __float_as_uint(f);
    u = u + 0x7fffu + ((u >> 16) & 1u);   // round to nearest, ties to even
    return (uint16_t)(u >> 16);
}
__device__ __forceinline__ float bf2f(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }
__device__ __forceinline__ f4 mfma(us8 a, us8 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                   0);
}
// 16x16x16 form (K = 16 input channels of one tap): lane l = 16g + n holds
// A[n][4g .. 4g+3] and B[4g .. 4g+3][n]; D as above.
__device__ __forceinline__ f4 mfma16(uint2 a, uint2 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s4, a), __builtin_bit_cast(s4, b), c, 0, 0, 0);
}
// lane k of each 16-lane row takes lane k-1 (shr) or k+1 (shl); 0 at the row ends:
// a shift along the k-line with the block's zero padding
__device__ __forceinline__ uint32_t shr1(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false); }
__device__ __forceinline__ uint32_t shl1(uint32_t v) { return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x101, 0xf, 0xf, false); }
__device__ __forceinline__ float shr1f(float v) { return __uint_as_float(shr1(__float_as_uint(v))); }
__device__ __forceinline__ float shl1f(float v) { return __uint_as_float(shl1(__float_as_uint(v))); }
__device__ __forceinline__ uint2 pack4(float a, float b, float c, float d) {
    return make_uint2((uint32_t)f2bf(a) | ((uint32_t)f2bf(b) << 16), (uint32_t)f2bf(c) | ((uint32_t)f2bf(d) << 16));
}
__device__ __forceinline__ float relu(float a) { return a > 0.0f ? a : 0.0f; }

// ------------------------------------------------------------------ packing
// the gradient images, then the forward images, in one launch
__device__ __forceinline__ void pack_forward(const float *__restrict__ p, uint16_t *__restrict__ pk, int q);

__global__ void __launch_bounds__(256) k_cnn_pack(const float *__restrict__ p, uint16_t *__restrict__ pk) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= PK_TOTAL * 8) {
        pack_forward(p, pk + PK_TOTAL * 8, q - PK_TOTAL * 8);
        return;
    }
    const int e = q & 7, entry = q >> 3, lane = entry & 63, row = lane & 15, g = lane >> 4;
    float w = 0.0f;
    if (entry < PK_Q2) {                            // Q3: k = tap (flipped), row = ci of layer 3
        const int t = 8 * g + e;
        if (t < 27) w = p[OFF_W3 + (26 - t) * 16 + row];
    } else {                                               // Q2: k = (t flipped, co), row = ci of layer 2
        const int k = 32 * ((entry - PK_Q2) >> 6) + 8 * g + e, t = k >> 4, co = k & 15;
        if (t < 27) w = p[OFF_W2 + ((26 - t) * 16 + row) * 16 + co];
    }
    pk[q] = f2bf(w);
}

__device__ __forceinline__ void pack_forward(const float *__restrict__ p, uint16_t *__restrict__ pk, int q) {
    if (q >= PF_TOTAL) return;
    float w = 0.0f;
    if (q < PF_L2A) {                                      // L1: W1[t = 9 di + s][co]
        const int e = q & 3, entry = q >> 2, di = entry >> 6, lane = entry & 63, co = lane & 15, gg = lane >> 4;
        const int s9 = 4 * gg + e;
        if (s9 < 9) w = p[OFF_W1 + (9 * di + s9) * 16 + co];
    } else if (q < PF_L2B) {                               // L2A: W2[t][ci][co], dk = -1 / +1
        const int r = q - PF_L2A, e = r & 7, entry = r >> 3, pr = entry >> 6, lane = entry & 63, co = lane & 15,
                  gg = lane >> 4;
        const int dk = gg < 2 ? 0 : 2, ci = 8 * (gg & 1) + e, t = 3 * pr + dk;
        w = p[OFF_W2 + (t * 16 + ci) * 16 + co];
    } else if (q < PF_L3) {                                // L2B: dk = 0
        const int r = q - PF_L2B, e = r & 3, entry = r >> 2, pr = entry >> 6, lane = entry & 63, co = lane & 15,
                  gg = lane >> 4;
        w = p[OFF_W2 + ((3 * pr + 1) * 16 + 4 * gg + e) * 16 + co];
    } else {                                               // L3: W3[t][ci]
        const int r = q - PF_L3, e = r & 3, entry = r >> 2, di = entry >> 6, lane = entry & 63, row = lane & 15,
                  gg = lane >> 4;
        const int dj = row >> 2, dk = row & 3;
        if (dj < 3 && dk < 3) w = p[OFF_W3 + (9 * di + 3 * dj + dk) * 16 + 4 * gg + e];
    }
    pk[q] = f2bf(w);
}

// ------------------------------------------------------------------ fused forward
// One workgroup per image; march over the 16 i-planes keeping rings of 3 planes
// of x, h1 and h2 in LDS: step n loads x plane n+1, computes h1 plane n, h2
// plane n-1 and the output plane n-2.  Wave w owns the k-lines j = 4w .. 4w+3
// of every plane; an MFMA column is one voxel of a k-line.
//   layer 1: per plane offset di one 16x16x16 MFMA, K = the 9 (dj, dk) taps;
//   layer 2: per input line (plane, row) one 16x16x32 MFMA over the dk = -1 and
//     dk = +1 taps and one 16x16x16 over dk = 0, each operand read once from LDS
//     (the halo in k makes the shifted reads plain loads) and used for the up
//     to 3 output lines the row touches;
//   layer 3: per input line one 16x16x16 MFMA whose rows are the 9 (dj, dk)
//     taps (accumulated over di), combined by DPP shifts (dk) and lane shuffles
//     (dj) into the output line.
// STORE also writes h1/h2 (channel-fastest) for the backward pass.
// A march is a serial chain of planes: 37 to 42 us per image alone on a CU.  An
// image is cut in i segments (each recomputes the planes its first needs, the
// same bits) while they still get a CU each, see fwd_segments.
struct HeatIO {                 // solver form of the forward (HEAT = true)
    const double *scale;       // per system, stride scale_stride
    int scale_stride, nb;
    long long istride;         // cells per system of c
    double *c;                 // FP64 output, [system][block][i][j][k]
    const int *active;         // systems still iterating (others are skipped)
};

typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
// 4 floats -> 4 bfloat16 (round to nearest even, v_cvt_pk_bf16_f32)
__device__ __forceinline__ uint2 cvt4(float a, float b, float c, float d) {
    bf16x4 v;
    v[0] = (__bf16)a; v[1] = (__bf16)b; v[2] = (__bf16)c; v[3] = (__bf16)d;
    return __builtin_bit_cast(uint2, v);
}
__device__ __forceinline__ uint16_t cvt1(float a) { return __builtin_bit_cast(uint16_t, (__bf16)a); }
__device__ __forceinline__ f4 mfma32(uint4 a, uint4 b, f4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0,
                                                   0);
}

template <bool STORE, bool HEAT, int NW>
__global__ void __launch_bounds__(64 * NW) k_cnn_fwd(const float *__restrict__ x, float *__restrict__ out,
                                                 const uint16_t *__restrict__ pf, const float *__restrict__ prm,
                                                 uint16_t *__restrict__ h1g, uint16_t *__restrict__ h2g, HeatIO hio,
                                                 const long long *__restrict__ idx) {
    __shared__ __align__(16) uint16_t sm[F_TOTAL];
    const long long img = blockIdx.x;
    // output planes pa .. pb - 1 of the image (blockIdx.y of gridDim.y segments):
    // the march starts with the h1 plane two before and ends with the one two after
    const int pa = 16 * blockIdx.y / gridDim.y, pb = 16 * (blockIdx.y + 1) / gridDim.y, first = pa > 2 ? pa - 2 : 0;
    double sc = 1.0;
    float inv_sc = 1.0f;
    if (HEAT) {
        if (!hio.active[img / hio.nb]) return;
        sc = hio.scale[(img / hio.nb) * hio.scale_stride];
        inv_sc = sc > 0.0 ? (float)(1.0 / sc) : 0.0f;
    }
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, n = lane & 15;
    // wavefront index as a scalar: the row-range tests below are uniform
    // branches, so the MFMA accumulators stay in place across them
    constexpr int LPW = 16 / NW;            // k-lines per wavefront
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j0 = LPW * wave;
    for (int q = tid; q < F_TOTAL / 2; q += 64 * NW) reinterpret_cast<uint32_t *>(sm)[q] = 0u;

    uint2 a1[3], a2b[9], a3[3];
    uint4 a2a[9];
#pragma unroll
    for (int d = 0; d < 3; d++) {
        a1[d] = reinterpret_cast<const uint2 *>(pf + PF_L1)[d * 64 + lane];
        a3[d] = reinterpret_cast<const uint2 *>(pf + PF_L3)[d * 64 + lane];
    }
#pragma unroll
    for (int pr = 0; pr < 9; pr++) {
        a2a[pr] = reinterpret_cast<const uint4 *>(pf + PF_L2A)[pr * 64 + lane];
        a2b[pr] = reinterpret_cast<const uint2 *>(pf + PF_L2B)[pr * 64 + lane];
    }
    float bb1[4], bb2[4];
#pragma unroll
    for (int r = 0; r < 4; r++) {
        bb1[r] = prm[OFF_B1 + 4 * g + r];
        bb2[r] = prm[OFF_B2 + 4 * g + r];
    }
    const float bb3 = prm[OFF_B3];
    // layer-1 gather: K slot s = 4g + e is tap (dj, dk) = (s / 3, s % 3) - 1 at
    // offset (s/3) * 18 + s % 3 + n from the output row in a halo'd x plane
    int xo[4];
    bool xv[4];
#pragma unroll
    for (int e = 0; e < 4; e++) {
        const int s9 = 4 * g + e;
        xv[e] = s9 < 9;
        xo[e] = xv[e] ? (s9 / 3) * 18 + s9 % 3 + n : n;
    }
    // per-lane LDS offsets in an h plane row: the k-shifted 8 channels
    // 8(g&1) .. +7 (dk = -1 for g < 2, +1 for g >= 2) as two 4-channel groups,
    // and the 4 channels 4g .. 4g+3 at k
    const int oA = (2 * (g & 1)) * HGRP + (g < 2 ? n : n + 2) * 4;
    const int oB = g * HGRP + (n + 1) * 4;
    const float *X = x + (STORE && idx ? idx[img] : img) * 4096;   // idx: the batch's images of a training set
    __syncthreads();

    // Planes -1 and 16 (the block's zero padding in i) are ring slots holding
    // zeros: slot 2 is not written before plane -1 is read, and plane 16 of x,
    // h1 and h2 is written as zeros one step after plane 15.  So every layer
    // runs its MFMAs over 3 planes without branches.
    // x planes are fetched from HBM one step before they are stored to LDS,
    // so the load latency overlaps a step of MFMA work
    const int xj = (tid >> 4) & 15, xk = tid & 15;
    const bool xl = tid < 256;              // the first 256 lanes move x
    auto fetch_x = [&](int q) -> float { return q < 16 ? X[(q * 16 + xj) * 16 + xk] : 0.0f; };
    auto store_x = [&](int q, float v) {
        sm[F_X + (q % 3) * PL + (xj + 1) * 18 + xk + 1] = cvt1(HEAT ? v * inv_sc : v);
    };

    if (xl) {
        if (first > 0) store_x(first - 1, fetch_x(first - 1));
        store_x(first, fetch_x(first));
    }
    float xnext = xl ? fetch_x(first + 1) : 0.0f;
    for (int step = first; step <= pb + 1; step++) {
        if (xl && step + 1 <= 16) {
            store_x(step + 1, xnext);
            if (step + 2 <= 16) xnext = fetch_x(step + 2);
        }
        __syncthreads();
        if (step == 16) {                       // h1 plane 16 = 0
#pragma unroll
            for (int jj = 0; jj < LPW; jj++)
                *reinterpret_cast<uint2 *>(sm + F_H1 + (16 % 3) * HPL + (j0 + jj + 1) * HROW + oB) = make_uint2(0u, 0u);
        }
        if (step <= 15) {                       // h1 plane step
            const int p = step;
            f4 acc[LPW];
#pragma unroll
            for (int jj = 0; jj < LPW; jj++) acc[jj] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int di = 0; di < 3; di++) {
                const int q = p + di - 1;
                const uint16_t *XP_ = sm + F_X + ((q + 3) % 3) * PL;
#pragma unroll
                for (int jj = 0; jj < LPW; jj++) {
                    const uint16_t *row = XP_ + (j0 + jj) * 18;
                    uint32_t v[4];
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const uint32_t t = row[xo[e]];
                        v[e] = xv[e] ? t : 0u;
                    }
                    acc[jj] = mfma16(a1[di], make_uint2(v[0] | (v[1] << 16), v[2] | (v[3] << 16)), acc[jj]);
                }
            }
#pragma unroll
            for (int jj = 0; jj < LPW; jj++) {
                const int j = j0 + jj;
                const uint2 o = cvt4(relu(acc[jj][0] + bb1[0]), relu(acc[jj][1] + bb1[1]), relu(acc[jj][2] + bb1[2]),
                                     relu(acc[jj][3] + bb1[3]));
                *reinterpret_cast<uint2 *>(sm + F_H1 + (p % 3) * HPL + (j + 1) * HROW + oB) = o;
                if (STORE && p >= pa && p < pb) *reinterpret_cast<uint2 *>(h1g + ((img * 4096 + (p * 16 + j) * 16 + n) * 16 + 4 * g)) = o;
            }
        }
        __syncthreads();
        if (step == 17) {                       // h2 plane 16 = 0
#pragma unroll
            for (int jj = 0; jj < LPW; jj++)
                *reinterpret_cast<uint2 *>(sm + F_H2 + (16 % 3) * HPL + (j0 + jj + 1) * HROW + oB) = make_uint2(0u, 0u);
        }
        if (step > first + (pa > 0) && step <= 16) {          // h2 plane step-1
            const int p = step - 1;
            // the 16x16x32 and 16x16x16 products accumulate in separate chains
            // (an accumulator is never shared by MFMAs of different shapes)
            f4 acc[LPW], acc16[LPW];
#pragma unroll
            for (int jj = 0; jj < LPW; jj++) {
                acc[jj] = f4{0.0f, 0.0f, 0.0f, 0.0f};
                acc16[jj] = f4{0.0f, 0.0f, 0.0f, 0.0f};
            }
#pragma unroll
            for (int di = 0; di < 3; di++) {
                const int q = p + di - 1;
                const uint16_t *P = sm + F_H1 + ((q + 3) % 3) * HPL;
                // input rows j0 - 1 .. j0 + LPW (halo rows are zero); each row's
                // operands feed the output lines within one row of it
#pragma unroll
                for (int ro = 0; ro < LPW + 2; ro++) {
                    const uint16_t *row = P + (j0 + ro) * HROW;
                    const uint2 bA0 = *reinterpret_cast<const uint2 *>(row + oA);
                    const uint2 bA1 = *reinterpret_cast<const uint2 *>(row + oA + HGRP);
                    const uint4 bA = make_uint4(bA0.x, bA0.y, bA1.x, bA1.y);
                    const uint2 bB = *reinterpret_cast<const uint2 *>(row + oB);
#pragma unroll
                    for (int jj = 0; jj < LPW; jj++) {
                        const int dj = ro - 1 - jj;
                        if (dj < -1 || dj > 1) continue;
                        const int pr = di * 3 + dj + 1;
                        acc[jj] = mfma32(a2a[pr], bA, acc[jj]);
                        acc16[jj] = mfma16(a2b[pr], bB, acc16[jj]);
                    }
                }
            }
#pragma unroll
            for (int jj = 0; jj < LPW; jj++) {
                const int j = j0 + jj;
                const f4 a = acc[jj] + acc16[jj];
                const uint2 o = cvt4(relu(a[0] + bb2[0]), relu(a[1] + bb2[1]), relu(a[2] + bb2[2]), relu(a[3] + bb2[3]));
                *reinterpret_cast<uint2 *>(sm + F_H2 + (p % 3) * HPL + (j + 1) * HROW + oB) = o;
                if (STORE && p >= pa && p < pb) *reinterpret_cast<uint2 *>(h2g + ((img * 4096 + (p * 16 + j) * 16 + n) * 16 + 4 * g)) = o;
            }
        }
        __syncthreads();
        if (step >= pa + 2) {                   // output plane step-2
            const int p = step - 2;
            f4 D[LPW + 2];
#pragma unroll
            for (int ro = 0; ro < LPW + 2; ro++) D[ro] = f4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int di = 0; di < 3; di++) {
                const int q = p + di - 1;
                const uint16_t *P = sm + F_H2 + ((q + 3) % 3) * HPL;
#pragma unroll
                for (int ro = 0; ro < LPW + 2; ro++)
                    D[ro] = mfma16(a3[di], *reinterpret_cast<const uint2 *>(P + (j0 + ro) * HROW + oB), D[ro]);
            }
            // lane group g of D[ro] holds the taps dj = g - 1 at input voxel n,
            // elements dk + 1: t = their sum at output voxel n (DPP for dk)
            float t[LPW + 2];
#pragma unroll
            for (int ro = 0; ro < LPW + 2; ro++) t[ro] = shr1f(D[ro][0]) + D[ro][1] + shl1f(D[ro][2]);
#pragma unroll
            for (int jj = 0; jj < LPW; jj++) {
                // output row j0 + jj: dj = -1 from row jj (group 0), dj = 0 from
                // row jj + 1 (group 1), dj = +1 from row jj + 2 (group 2)
                const float o = (t[jj] + __shfl(t[jj + 1], 16 + n, 64)) + __shfl(t[jj + 2], 32 + n, 64);
                if (g == 0) {
                    if (HEAT) {
                        const long long sys = img / hio.nb, b = img - sys * hio.nb;
                        hio.c[sys * hio.istride + b * 4096 + (p * 16 + j0 + jj) * 16 + n] = sc * (double)(o + bb3);
                    } else {
                        out[img * 4096 + (p * 16 + j0 + jj) * 16 + n] = o + bb3;
                    }
                }
            }
        }
    }
}

// ------------------------------------------------------------------ data gradients
// gout[v][c] = (mask[v][c] > 0) ? sum_{t,ci} Wq[t][ci][c] gin[v + off_t][ci] : 0, stored as bfloat16.
// A workgroup takes 4 i-planes of an image (blockIdx.y), one per wavefront, and
// stages them with a halo once: 4 workgroups per image fill the chip at the
// training batches (128 images, 256 CUs), and no barrier follows the staging.
constexpr int DPL = 4;                      // output planes per workgroup

// Layer 3 -> 2 (gin: the float output gradient, weights Q3): one MFMA per
// k-line, K = the 27 taps.  Bound by the LDS gather of the taps; their offsets
// are formed once per lane, a line's row is an immediate.  128
// images: 48 -> 9.7 us against one workgroup per image with the offsets formed
// per read and the masks read where they are used (loads now come first).
__global__ void __launch_bounds__(256) k_cnn_dgrad1(const float *__restrict__ gin, const uint16_t *__restrict__ mask,
                                                    uint16_t *__restrict__ gout, const us8 *__restrict__ pk) {
    __shared__ __align__(16) uint16_t sm[(DPL + 2) * PL];
    const long long img = blockIdx.x;
    const int p0 = blockIdx.y * DPL;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, kk = lane & 15;
    const long long o0 = (img * 4096 + ((p0 + wave) * 16) * 16 + kk) * 16 + 4 * g;
    uint2 mk[16];
#pragma unroll
    for (int j = 0; j < 16; j++) mk[j] = *reinterpret_cast<const uint2 *>(mask + o0 + j * 256);
    float v[DPL + 2];
#pragma unroll
    for (int q = 0; q < DPL + 2; q++) {
        const int i = p0 - 1 + q;
        v[q] = i >= 0 && i < 16 ? gin[img * 4096 + i * 256 + tid] : 0.0f;
    }
    const us8 w = pk[PK_Q3 + lane];
    for (int q = tid; q < (DPL + 2) * PL / 2; q += 256) reinterpret_cast<uint32_t *>(sm)[q] = 0u;
    __syncthreads();
#pragma unroll
    for (int q = 0; q < DPL + 2; q++) sm[q * PL + ((tid >> 4) + 1) * 18 + (tid & 15) + 1] = f2bf(v[q]);
    __syncthreads();
    const uint16_t *src[8];
    bool on[8];
#pragma unroll
    for (int e = 0; e < 8; e++) {
        const int t = 8 * g + e;
        on[e] = t < 27;
        src[e] = sm + (on[e] ? (wave + t / 9) * PL + (t / 3) % 3 * 18 + t % 3 + kk : 0);
    }
#pragma unroll
    for (int j = 0; j < 16; j++) {
        us8 b;
#pragma unroll
        for (int e = 0; e < 8; e++) b[e] = on[e] ? src[e][j * 18] : (uint16_t)0;
        const f4 acc = mfma(w, b, f4{0.0f, 0.0f, 0.0f, 0.0f});
        const float m0 = bf2f((uint16_t)(mk[j].x & 0xffffu)), m1 = bf2f((uint16_t)(mk[j].x >> 16)),
                    m2 = bf2f((uint16_t)(mk[j].y & 0xffffu)), m3 = bf2f((uint16_t)(mk[j].y >> 16));
        *reinterpret_cast<uint2 *>(gout + o0 + j * 256) = pack4(m0 > 0.0f ? acc[0] : 0.0f, m1 > 0.0f ? acc[1] : 0.0f,
                                                                m2 > 0.0f ? acc[2] : 0.0f, m3 > 0.0f ? acc[3] : 0.0f);
    }
}

// Layer 2 -> 1 (gin: the bfloat16 layer-2 output gradient, weights Q2): 14
// MFMAs per k-line in one chain, K = (tap pair, channel).  LDS [plane][channel
// half][18][18][8]: the lanes of a 16-byte read are consecutive (no bank
// conflicts); bound by those reads, 14 per line and wavefront.  128
// images: 53 -> 15 us against one workgroup per image on [voxel][16] planes.
__global__ void __launch_bounds__(256) k_cnn_dgrad16(const uint16_t *__restrict__ gin, const uint16_t *__restrict__ mask,
                                                     uint16_t *__restrict__ gout, const us8 *__restrict__ pk) {
    constexpr int HP = PL * 8;              // elements per half plane
    __shared__ __align__(16) uint16_t sm[(DPL + 2) * 2 * HP];
    const long long img = blockIdx.x;
    const int p0 = blockIdx.y * DPL;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 4, kk = lane & 15;
    const long long o0 = (img * 4096 + ((p0 + wave) * 16) * 16 + kk) * 16 + 4 * g;
    uint2 mk[16];
#pragma unroll
    for (int j = 0; j < 16; j++) mk[j] = *reinterpret_cast<const uint2 *>(mask + o0 + j * 256);
    uint4 v[DPL + 2][2];
#pragma unroll
    for (int q = 0; q < DPL + 2; q++) {
        const int i = p0 - 1 + q;
        const uint4 *src = reinterpret_cast<const uint4 *>(gin + (img * 4096 + (long long)i * 256) * 16);
#pragma unroll
        for (int h = 0; h < 2; h++)
            v[q][h] = i >= 0 && i < 16 ? src[h * 256 + tid] : make_uint4(0u, 0u, 0u, 0u);
    }
    us8 w[14];
#pragma unroll
    for (int s = 0; s < 14; s++) w[s] = pk[PK_Q2 + s * 64 + lane];
    for (int q = tid; q < (DPL + 2) * 2 * PL; q += 256) reinterpret_cast<uint4 *>(sm)[q] = make_uint4(0u, 0u, 0u, 0u);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < DPL + 2; q++)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            // element h * 256 + tid of the plane: voxel e >> 1, channel half e & 1
            const int e = h * 256 + tid, vx = e >> 1;
            *reinterpret_cast<uint4 *>(sm + (q * 2 + (e & 1)) * HP + (((vx >> 4) + 1) * 18 + (vx & 15) + 1) * 8) = v[q][h];
        }
    __syncthreads();
    // slot s of this lane is tap 2 s + (g >> 1) (27: none)
    int off[14];
#pragma unroll
    for (int s = 0; s < 14; s++) {
        const int t = 2 * s + (g >> 1), u = t < 27 ? t : 0;
        off[s] = ((wave + u / 9) * 2 + (g & 1)) * HP + ((u / 3) % 3 * 18 + u % 3 + kk) * 8;
    }
    const bool last = g < 2;
#pragma unroll
    for (int j = 0; j < 16; j++) {
        f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int s = 0; s < 14; s++) {
            uint4 b = *reinterpret_cast<const uint4 *>(sm + off[s] + j * 144);
            if (s == 13) b = last ? b : make_uint4(0u, 0u, 0u, 0u);
            acc = mfma(w[s], __builtin_bit_cast(us8, b), acc);
        }
        const float m0 = bf2f((uint16_t)(mk[j].x & 0xffffu)), m1 = bf2f((uint16_t)(mk[j].x >> 16)),
                    m2 = bf2f((uint16_t)(mk[j].y & 0xffffu)), m3 = bf2f((uint16_t)(mk[j].y >> 16));
        *reinterpret_cast<uint2 *>(gout + o0 + j * 256) = pack4(m0 > 0.0f ? acc[0] : 0.0f, m1 > 0.0f ? acc[1] : 0.0f,
                                                                m2 > 0.0f ? acc[2] : 0.0f, m3 > 0.0f ? acc[3] : 0.0f);
    }
}

// ------------------------------------------------------------------ weight gradients
// Per image, into part[img][kCnnParams] (the parameter layout):
//   L = 3: dW3[t][ci] = sum_v h2[v+t][ci] g3[v]      (in = h2, g = g3 float)
//   L = 2: dW2[t][ci][co] = sum_v h1[v+t][ci] g2[v][co]
//   L = 1: dW1[t][co] = sum_v x[v+t] g1[v][co]        (in = x float)
// and the bias gradient of the layer, sum_v g[v][co].
// D[co][n] = sum over 32-voxel chunks (2 k-lines, in the order of the planes)
// of A[co][voxel] B[voxel][n]; n = ci of one tap (L = 2, 3) or n = tap (L = 1).
// An MFMA lane needs 8 consecutive voxels of one channel, the activations are
// channel-fastest: the planes are turned on their way into LDS ([channel][j][k],
// 4 voxels x 4 channels per lane), so an operand is one 16-byte read; gathering
// it 2 bytes at a time bound the three passes before: 221 us for 128 images, this
// one 36 us (37 images 211 -> 19 us).
// Layers 2 and 3: a workgroup takes the 9 taps of one plane offset di, wavefront
// w < 3 the 3 taps of dj = w - 1, whose operands are one row read and its
// shifts by one voxel in registers (v_alignbit); planes are double-buffered,
// one barrier each.  Layer 1: x with a halo in 3 copies shifted in k (every
// tap's 8 voxels aligned), wavefront w < 2 holds taps 16w .. 16w+15.  All in
// one launch: blockIdx.y = 0 .. 2 layer 2, 3 .. 5 layer 3, 6 layer 1, so a
// small batch still spreads over 7 workgroups per image.
// 40 KB of LDS and at most 128 VGPRs: 4 workgroups per CU hold the 896 of 128
// images in one round.
constexpr int WA_CH = 16 * 16 + 8, WA_PL = 16 * WA_CH;           // g planes: rows of 16, channels 528 bytes apart
constexpr int WB_ROW = 20, WB_CH = 18 * WB_ROW + 4, WB_PL = 16 * WB_CH;   // input planes: 4 zeros, 16 voxels; channels 728 bytes apart
constexpr int WDEPTH = 2;                                        // planes in flight
constexpr int WX_CP = 18 * 18 * 16;                              // one shifted copy of x
constexpr int W_TOTAL = 2 * (WA_PL + WB_PL);
static_assert(W_TOTAL >= 3 * WX_CP + WA_PL, "layer 1's three copies of x and one g plane");
static_assert(WA_PL >= 256 + 2 * 256 + 16 * 16 * 2, "layer 3's g plane in two types");

struct Quad {                               // 4 voxels x 4 channels
    uint2 v[4];
    __device__ __forceinline__ void load(const uint16_t *src, int plane, int tid) {
        const uint16_t *p = src + ((plane * 64 + (tid >> 2)) * 4) * 16 + 4 * (tid & 3);
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = *reinterpret_cast<const uint2 *>(p + u * 16);
    }
    __device__ __forceinline__ void clear() {
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = make_uint2(0u, 0u);
    }
    // channel c of the 4 as its 4 voxels, channels `stride` elements apart
    __device__ __forceinline__ void store(uint16_t *dst, int stride) const {
        const uint32_t lo = 0xffffu, hi = 0xffff0000u;
        *reinterpret_cast<uint2 *>(dst) = make_uint2((v[0].x & lo) | (v[1].x << 16), (v[2].x & lo) | (v[3].x << 16));
        *reinterpret_cast<uint2 *>(dst + stride) = make_uint2((v[0].x >> 16) | (v[1].x & hi), (v[2].x >> 16) | (v[3].x & hi));
        *reinterpret_cast<uint2 *>(dst + 2 * stride) = make_uint2((v[0].y & lo) | (v[1].y << 16), (v[2].y & lo) | (v[3].y << 16));
        *reinterpret_cast<uint2 *>(dst + 3 * stride) = make_uint2((v[0].y >> 16) | (v[1].y & hi), (v[2].y >> 16) | (v[3].y & hi));
    }
};

// sum of a row of 16 bf16 voxels onto s, in order
__device__ __forceinline__ float row_sum(const uint16_t *row, float s) {
    const uint4 a = reinterpret_cast<const uint4 *>(row)[0], b = reinterpret_cast<const uint4 *>(row)[1];
    const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
    for (int k = 0; k < 8; k++) {
        s += __uint_as_float(w[k] << 16);
        s += __uint_as_float(w[k] & 0xffff0000u);
    }
    return s;
}

template <int L>
__device__ __forceinline__ void wgrad_taps(const uint16_t *__restrict__ in, const void *__restrict__ g_, int di,
                                           float *__restrict__ P, uint16_t *sm) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4,
              n = lane & 15;
    const int vg = tid >> 2, j4 = vg >> 2, k4 = 4 * (vg & 3), c4 = 4 * (tid & 3);
    for (int q = tid; q < 2 * (WA_PL + WB_PL) / 8; q += 256) reinterpret_cast<uint4 *>(sm)[q] = make_uint4(0u, 0u, 0u, 0u);
    // planes p + 1 .. p + WDEPTH are on their way while plane p is computed
    Quad qa[WDEPTH], qb[WDEPTH];
    float gf[WDEPTH];
    auto fetch = [&](int p, int u) {
        if (L == 2) qa[u].load(reinterpret_cast<const uint16_t *>(g_), p, tid);
        else gf[u] = reinterpret_cast<const float *>(g_)[p * 256 + tid];
        const int q = p + di;
        qb[u].load(in, q < 0 ? 0 : (q > 15 ? 15 : q), tid);
    };
    auto stage = [&](int p, int u) {
        uint16_t *A = sm + (p & 1) * (WA_PL + WB_PL), *B = A + WA_PL;
        if (L == 2) {
            qa[u].store(A + c4 * WA_CH + j4 * 16 + k4, WA_CH);
        } else {
            A[tid] = f2bf(gf[u]);
            reinterpret_cast<float *>(A + 256)[tid] = gf[u];
        }
        if (p + di < 0 || p + di > 15) qb[u].clear();      // beyond the block: zeros
        qb[u].store(B + c4 * WB_CH + (j4 + 1) * WB_ROW + 4 + k4, WB_CH);
    };
    f4 acc[3];
#pragma unroll
    for (int a = 0; a < 3; a++) acc[a] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    float bias_acc = 0.0f;    // thread tid: channel tid & 15, voxels of its plane rows (tid >> 4)
    const uint32_t row0 = n == 0 ? 0xffffffffu : 0u;      // layer 3: the only row of A
#pragma unroll
    for (int u = 0; u < WDEPTH; u++) fetch(u, u);
    __syncthreads();
    stage(0, 0);
#pragma unroll WDEPTH
    for (int p = 0; p < 16; p++) {
        __syncthreads();
        if (p + WDEPTH < 16) fetch(p + WDEPTH, p % WDEPTH);
        const uint16_t *A = sm + (p & 1) * (WA_PL + WB_PL), *B = A + WA_PL;
        if (di == 0) {
            const int c = tid & 15, jr = tid >> 4;
            if (L == 2) {
                bias_acc = row_sum(A + c * WA_CH + jr * 16, bias_acc);
            } else if (c == 0) {
#pragma unroll
                for (int k = 0; k < 16; k++) bias_acc += reinterpret_cast<const float *>(A + 256)[jr * 16 + k];
            }
        }
        if (wave < 3) {
            // all operands of 4 chunks are read before the first is used
            const uint16_t *Ap = A + (L == 2 ? n * WA_CH : 0) + (g >> 1) * 16 + 8 * (g & 1);
            const uint16_t *Bp = B + n * WB_CH + (wave + (g >> 1)) * WB_ROW + 4 + 8 * (g & 1);
#pragma unroll
            for (int c0 = 0; c0 < 8; c0 += 4) {
                uint4 a[4], b[4];
                uint32_t pv[4], nx[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    a[u] = *reinterpret_cast<const uint4 *>(Ap + (c0 + u) * 32);
                    const uint16_t *row = Bp + (c0 + u) * 2 * WB_ROW;
                    const uint2 lo = *reinterpret_cast<const uint2 *>(row), hi = *reinterpret_cast<const uint2 *>(row + 4);
                    b[u] = make_uint4(lo.x, lo.y, hi.x, hi.y);
                    pv[u] = *reinterpret_cast<const uint32_t *>(row - 2);
                    nx[u] = *reinterpret_cast<const uint32_t *>(row + 8);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    if (L == 3) a[u] = make_uint4(a[u].x & row0, a[u].y & row0, a[u].z & row0, a[u].w & row0);
                    const uint32_t s1 = __builtin_amdgcn_alignbit(b[u].y, b[u].x, 16),
                                   s2 = __builtin_amdgcn_alignbit(b[u].z, b[u].y, 16),
                                   s3 = __builtin_amdgcn_alignbit(b[u].w, b[u].z, 16);
                    acc[0] = mfma32(a[u], make_uint4(__builtin_amdgcn_alignbit(b[u].x, pv[u], 16), s1, s2, s3), acc[0]);
                    acc[1] = mfma32(a[u], b[u], acc[1]);
                    acc[2] = mfma32(a[u], make_uint4(s1, s2, s3, __builtin_amdgcn_alignbit(nx[u], b[u].w, 16)), acc[2]);
                }
            }
        }
        if (p + 1 < 16) stage(p + 1, (p + 1) % WDEPTH);
    }
    // D[co = 4g + r][n]
    if (wave < 3) {
#pragma unroll
        for (int dk = 0; dk < 3; dk++) {
            const int t = (di + 1) * 9 + wave * 3 + dk;
            if (L == 2) {
                for (int r = 0; r < 4; r++) P[OFF_W2 + (t * 16 + n) * 16 + 4 * g + r] = acc[dk][r];
            } else if (g == 0) {
                P[OFF_W3 + t * 16 + n] = acc[dk][0];
            }
        }
    }
    if (di == 0) {
        __syncthreads();
        float (*sBias)[16] = reinterpret_cast<float (*)[16]>(sm);
        sBias[tid >> 4][tid & 15] = bias_acc;
        __syncthreads();
        if (tid < 16) {
            float s = 0.0f;
            for (int r = 0; r < 16; r++) s += sBias[r][tid];
            if (L == 2) P[OFF_B2 + tid] = s;
            else if (tid == 0) P[OFF_B3] = s;
        }
    }
}

__device__ __forceinline__ void wgrad_first(const float *__restrict__ x, const uint16_t *__restrict__ g1,
                                            float *__restrict__ P, uint16_t *sm) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), g = lane >> 4,
              n = lane & 15;
    const int vg = tid >> 2, j4 = vg >> 2, k4 = 4 * (vg & 3), c4 = 4 * (tid & 3);
    uint16_t *xs = sm + WA_PL;
    float xv[16];
#pragma unroll
    for (int p = 0; p < 16; p++) xv[p] = x[p * 256 + tid];
    for (int q = tid; q < 3 * WX_CP / 8; q += 256) reinterpret_cast<uint4 *>(xs)[q] = make_uint4(0u, 0u, 0u, 0u);
    Quad qa[WDEPTH];
#pragma unroll
    for (int u = 0; u < WDEPTH; u++) qa[u].load(g1, u, tid);
    __syncthreads();
    // copy dk + 1, row (plane + 1, j + 1): element k holds x at k + dk
#pragma unroll
    for (int p = 0; p < 16; p++) {
        const uint16_t v = f2bf(xv[p]);
        uint16_t *row = xs + ((p + 1) * 18 + (tid >> 4) + 1) * 16;
        const int k = tid & 15;
        if (k < 15) row[k + 1] = v;
        row[WX_CP + k] = v;
        if (k > 0) row[2 * WX_CP + k - 1] = v;
    }
    qa[0].store(sm + c4 * WA_CH + j4 * 16 + k4, WA_CH);
    const int t = 16 * wave + n;
    const bool on = t < 27;
    const uint32_t taps = on ? 0xffffffffu : 0u;
    const int u = on ? t : 0;
    const uint16_t *src = xs + (u % 3) * WX_CP + ((u / 9) * 18 + (u / 3) % 3) * 16;
    f4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    float bias_acc = 0.0f;
#pragma unroll WDEPTH
    for (int p = 0; p < 16; p++) {
        __syncthreads();
        if (p + WDEPTH < 16) qa[p % WDEPTH].load(g1, p + WDEPTH, tid);
        const uint16_t *A = sm;
        bias_acc = row_sum(A + (tid & 15) * WA_CH + (tid >> 4) * 16, bias_acc);
        if (wave < 2) {
#pragma unroll
            for (int c0 = 0; c0 < 8; c0 += 4) {
                uint4 a[4], b[4];
#pragma unroll
                for (int u = 0; u < 4; u++) {
                    a[u] = *reinterpret_cast<const uint4 *>(A + n * WA_CH + (2 * (c0 + u) + (g >> 1)) * 16 + 8 * (g & 1));
                    b[u] = *reinterpret_cast<const uint4 *>(src + (p * 18 + 2 * (c0 + u) + (g >> 1)) * 16 + 8 * (g & 1));
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < 4; u++)
                    acc = mfma32(a[u], make_uint4(b[u].x & taps, b[u].y & taps, b[u].z & taps, b[u].w & taps), acc);
            }
        }
        __syncthreads();
        if (p + 1 < 16) qa[(p + 1) % WDEPTH].store(sm + c4 * WA_CH + j4 * 16 + k4, WA_CH);
    }
    if (wave < 2 && on)
        for (int r = 0; r < 4; r++) P[OFF_W1 + t * 16 + 4 * g + r] = acc[r];
    float (*sBias)[16] = reinterpret_cast<float (*)[16]>(sm);      // (the last plane's barrier is behind)
    sBias[tid >> 4][tid & 15] = bias_acc;
    __syncthreads();
    if (tid < 16) {
        float s = 0.0f;
        for (int r = 0; r < 16; r++) s += sBias[r][tid];
        P[OFF_B1 + tid] = s;
    }
}

__global__ void __launch_bounds__(256, 4) k_cnn_wgrad(const float *__restrict__ x, const uint16_t *__restrict__ h1,
                                                   const uint16_t *__restrict__ h2, const uint16_t *__restrict__ g1,
                                                   const uint16_t *__restrict__ g2, const float *__restrict__ g3,
                                                   float *__restrict__ part, const long long *__restrict__ idx) {
    __shared__ __align__(16) uint16_t sm[W_TOTAL];
    const long long img = blockIdx.x, v = img * 4096;
    const int job = blockIdx.y;
    float *P = part + img * (long long)kCnnParams;
    if (job < 3) wgrad_taps<2>(h1 + v * 16, g2 + v * 16, job - 1, P, sm);
    else if (job < 6) wgrad_taps<3>(h2 + v * 16, g3 + v, job - 4, P, sm);
    else wgrad_first(x + (idx ? idx[img] : img) * 4096, g1 + v * 16, P, sm);
}

// grad[q] = sum over images of part[img][q], fixed order, FP64, 32 images in
// flight (the additions keep their order, the loads do not wait for them)
__device__ __forceinline__ double part_sum(const float *__restrict__ part, int nimg, int q) {
    double s = 0.0;
    const float *P = part + q;
    int i0 = 0;
    for (; i0 + 32 <= nimg; i0 += 32, P += 32LL * kCnnParams) {
        float v[32];
#pragma unroll
        for (int i = 0; i < 32; i++) v[i] = P[(long long)i * kCnnParams];
#pragma unroll
        for (int i = 0; i < 32; i++) s += (double)v[i];
    }
    for (; i0 + 4 <= nimg; i0 += 4, P += 4LL * kCnnParams) {
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; i++) v[i] = P[(long long)i * kCnnParams];
#pragma unroll
        for (int i = 0; i < 4; i++) s += (double)v[i];
    }
    for (; i0 < nimg; i0++, P += kCnnParams) s += (double)P[0];
    return s;
}
__global__ void __launch_bounds__(64) k_cnn_reduce(const float *__restrict__ part, int nimg, double *__restrict__ grad) {
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q < kCnnParams) grad[q] = part_sum(part, nimg, q);
}

// end of a training step: the gradient sums go straight into Adam's update;
// one more workgroup adds the batch's loss partials (x scale x weight) to
// loss[0], which `first` starts
__global__ void __launch_bounds__(64) k_cnn_update(const float *__restrict__ part, int nimg, float *__restrict__ p,
                                                   float *__restrict__ m, float *__restrict__ v, float lr, float c1,
                                                   float c2, const double *__restrict__ lpart, int nl, double scale,
                                                   double weight, bool first, double *__restrict__ loss) {
    if (blockIdx.x == gridDim.x - 1) {
        double s = 0.0;
        for (int i = threadIdx.x; i < nl; i += 64) s += lpart[i];
        for (int off = 32; off > 0; off >>= 1) s += __shfl_down(s, off, 64);
        if (threadIdx.x == 0) loss[0] = (first ? 0.0 : loss[0]) + (s * scale) * weight;
        return;
    }
    const int q = blockIdx.x * blockDim.x + threadIdx.x;
    if (q >= kCnnParams) return;
    const float g = (float)part_sum(part, nimg, q);
    const float mm = 0.9f * m[q] + 0.1f * g, vv = 0.999f * v[q] + 0.001f * g * g;
    m[q] = mm;
    v[q] = vv;
    p[q] = p[q] - lr * (mm * c1) / (sqrtf(vv * c2) + 1e-8f);
}

// g3 = 2 (out - y) / N ; loss partials sum (out - y)^2
// (every loss: y of image b is that of the training set's image idx[b])
__global__ void __launch_bounds__(256) k_cnn_loss(const float *__restrict__ out, const float *__restrict__ y, long long n,
                                                  float *__restrict__ g3, double *__restrict__ part,
                                                  const long long *__restrict__ idx) {
    __shared__ double red[4];
    double acc = 0.0;
    const float sc = (float)(2.0 / (double)n);
    for (long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (long long)gridDim.x * blockDim.x) {
        const float d = out[i] - y[idx[i >> 12] * 4096 + (i & 4095)];
        g3[i] = sc * d;
        acc += (double)d * (double)d;
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) part[blockIdx.x] = ((red[0] + red[1]) + red[2]) + red[3];
}

// Gradient-weighted error per 16^3 image, d = out - y:
//   L = alpha sum_cells d^2 + sum over the faces inside the image w_a (d_a - d_b)^2,
// w_a the weight of the face's axis (image axes i, j, k = r, theta, phi): an
// energy-like norm of the diffusion operator (mass term alpha, face couplings
// w) that weighs the error's variation instead of its offset.
// g3 = (dL/d out) * sc; loss partials per workgroup.  One workgroup walks
// images blockIdx.x, blockIdx.x + gridDim.x, ...
__global__ void __launch_bounds__(1024) k_cnn_loss_h1(const float *__restrict__ out, const float *__restrict__ y,
                                                     int nimg, float alpha, float wi, float wj, float wk, float sc,
                                                     float *__restrict__ g3, double *__restrict__ part,
                                                     const long long *__restrict__ idx) {
    __shared__ float dl[4096];
    __shared__ double red[16];
    double acc = 0.0;
    for (int img = blockIdx.x; img < nimg; img += gridDim.x) {
        const long long o = (long long)img * 4096;
        const float *Y = y + idx[img] * 4096;
        for (int c = threadIdx.x; c < 4096; c += 1024) dl[c] = out[o + c] - Y[c];
        __syncthreads();
        for (int c = threadIdx.x; c < 4096; c += 1024) {
            const int i = c >> 8, j = (c >> 4) & 15, k = c & 15;
            const float d = dl[c];
            float g = alpha * d;
            double l = (double)alpha * (double)d * (double)d;
            // each face enters the loss once (from its lower cell) and the
            // gradient of both cells
            if (i > 0) g += wi * (d - dl[c - 256]);
            if (i < 15) { const float e = d - dl[c + 256]; g += wi * e; l += (double)wi * ((double)e * (double)e); }
            if (j > 0) g += wj * (d - dl[c - 16]);
            if (j < 15) { const float e = d - dl[c + 16]; g += wj * e; l += (double)wj * ((double)e * (double)e); }
            if (k > 0) g += wk * (d - dl[c - 1]);
            if (k < 15) { const float e = d - dl[c + 1]; g += wk * e; l += (double)wk * ((double)e * (double)e); }
            g3[o + c] = sc * (2.0f * g);
            acc += l;
        }
        __syncthreads();
    }
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_down(acc, off, 64);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double l = red[0];
        for (int w = 1; w < 16; w++) l += red[w];
        part[blockIdx.x] = l;
    }
}

// Scale-free form of the same norm, per image: with A = alpha I + sum_a w_a
// (the face-difference operator along axis a), the fraction of e's A-norm that
// the best multiple of c leaves,
//   L = 1 - <c,Ae>^2 / (<c,Ac> <e,Ae>),
// which is what the FCG step with its A-optimal scale a rewards.  dL/dc =
// -2 <c,Ae> / (<c,Ac><e,Ae>) (Ae - (<c,Ae>/<c,Ac>) Ac); g3 = dL/dc * sc.
// Images with <c,Ac> or <e,Ae> zero contribute nothing.
__global__ void __launch_bounds__(256) k_cnn_loss_cos(const float *__restrict__ out, const float *__restrict__ y,
                                                      int nimg, float alpha, float wi, float wj, float wk, float sc,
                                                      float *__restrict__ g3, double *__restrict__ part,
                                                     const long long *__restrict__ idx) {
    __shared__ float cl[4096], el[4096];
    __shared__ double red[3][4];
    double lacc = 0.0;
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    for (int img = blockIdx.x; img < nimg; img += gridDim.x) {
        const long long o = (long long)img * 4096;
        for (int c = threadIdx.x; c < 4096; c += 256) {
            cl[c] = out[o + c];
            el[c] = y[idx[img] * 4096 + c];
        }
        __syncthreads();
        // A v at cell c, v in LDS
        auto apply = [&](const float *v, int c) -> double {
            const int i = c >> 8, j = (c >> 4) & 15, k = c & 15;
            const double x = v[c];
            double a = (double)alpha * x;
            if (i > 0) a += (double)wi * (x - v[c - 256]);
            if (i < 15) a += (double)wi * (x - v[c + 256]);
            if (j > 0) a += (double)wj * (x - v[c - 16]);
            if (j < 15) a += (double)wj * (x - v[c + 16]);
            if (k > 0) a += (double)wk * (x - v[c - 1]);
            if (k < 15) a += (double)wk * (x - v[c + 1]);
            return a;
        };
        double s_ce = 0.0, s_cc = 0.0, s_ee = 0.0;
        for (int c = threadIdx.x; c < 4096; c += 256) {
            const double ae = apply(el, c), ac = apply(cl, c);
            s_ce += (double)cl[c] * ae;
            s_cc += (double)cl[c] * ac;
            s_ee += (double)el[c] * ae;
        }
        for (int off = 32; off > 0; off >>= 1) {
            s_ce += __shfl_down(s_ce, off, 64);
            s_cc += __shfl_down(s_cc, off, 64);
            s_ee += __shfl_down(s_ee, off, 64);
        }
        if (lane == 0) { red[0][wv] = s_ce; red[1][wv] = s_cc; red[2][wv] = s_ee; }
        __syncthreads();
        const double ce = ((red[0][0] + red[0][1]) + red[0][2]) + red[0][3];
        const double cc = ((red[1][0] + red[1][1]) + red[1][2]) + red[1][3];
        const double ee = ((red[2][0] + red[2][1]) + red[2][2]) + red[2][3];
        const bool ok = cc > 0.0 && ee > 0.0;
        const double f = ok ? -2.0 * ce / (cc * ee) : 0.0, r = ok ? ce / cc : 0.0;
        for (int c = threadIdx.x; c < 4096; c += 256) {
            const double g = ok ? f * (apply(el, c) - r * apply(cl, c)) : 0.0;
            g3[o + c] = (float)(g * (double)sc);
        }
        if (threadIdx.x == 0 && ok) lacc += 1.0 - ce * ce / (cc * ee);
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = lacc;
}

}  // namespace

// ------------------------------------------------------------------ host class

CnnModel::CnnModel() {
    CCHECK(hipMalloc(&params_, sizeof(float) * kCnnParams));
    CCHECK(hipMalloc(&adam_m_, sizeof(float) * kCnnParams));
    CCHECK(hipMalloc(&adam_v_, sizeof(float) * kCnnParams));
    CCHECK(hipMalloc(&grad_, sizeof(double) * kCnnParams));
    CCHECK(hipMalloc(&packed_, sizeof(uint16_t) * (PK_TOTAL * 8 + PF_TOTAL)));
    CCHECK(hipMalloc(&loss_part_, sizeof(double) * 1025));
    init(12345);
}

CnnModel::~CnnModel() {
    for (void *p : {(void *)params_, (void *)adam_m_, (void *)adam_v_, (void *)grad_, packed_, (void *)loss_part_,
                    (void *)h1_, (void *)h2_, (void *)g2_, (void *)g1_, (void *)out_, (void *)g3_, (void *)part_})
        if (p) (void)hipFree(p);
}

void CnnModel::init(uint64_t seed) {
    std::mt19937_64 rng(seed);
    std::vector<float> p(kCnnParams, 0.0f);
    auto fill = [&](int off, int n, double std) {
        std::normal_distribution<double> nd(0.0, std);
        for (int i = 0; i < n; i++) p[off + i] = (float)nd(rng);
    };
    fill(OFF_W1, 432, std::sqrt(2.0 / 27.0));
    fill(OFF_W2, 6912, std::sqrt(2.0 / 432.0));
    fill(OFF_W3, 432, std::sqrt(1.0 / 432.0));
    set_params(p.data());
}

void CnnModel::set_params(const float *p) {
    CCHECK(hipMemcpy(params_, p, sizeof(float) * kCnnParams, hipMemcpyHostToDevice));
    std::vector<float> z(kCnnParams, 0.0f);
    CCHECK(hipMemcpy(adam_m_, z.data(), sizeof(float) * kCnnParams, hipMemcpyHostToDevice));
    CCHECK(hipMemcpy(adam_v_, z.data(), sizeof(float) * kCnnParams, hipMemcpyHostToDevice));
    adam_t_ = 0;
    packed_valid_ = false;
}

void CnnModel::get_params(float *p) const {
    CCHECK(hipDeviceSynchronize());
    CCHECK(hipMemcpy(p, params_, sizeof(float) * kCnnParams, hipMemcpyDeviceToHost));
}

void CnnModel::pack(hipStream_t stream) {
    if (packed_valid_) return;
    hipLaunchKernelGGL(k_cnn_pack, dim3((PK_TOTAL * 8 + PF_TOTAL + 255) / 256), dim3(256), 0, stream,
                       (const float *)params_, (uint16_t *)packed_);
    packed_valid_ = true;
}

void CnnModel::ensure_batch(int nimg) {
    if (nimg <= max_batch_) return;
    for (void *p : {(void *)h1_, (void *)h2_, (void *)g2_, (void *)g1_, (void *)out_, (void *)g3_, (void *)part_})
        if (p) CCHECK(hipFree(p));
    const size_t n = (size_t)nimg;
    CCHECK(hipMalloc(&h1_, n * 4096 * 16 * sizeof(uint16_t)));
    CCHECK(hipMalloc(&h2_, n * 4096 * 16 * sizeof(uint16_t)));
    CCHECK(hipMalloc(&g2_, n * 4096 * 16 * sizeof(uint16_t)));
    CCHECK(hipMalloc(&g1_, n * 4096 * 16 * sizeof(uint16_t)));
    CCHECK(hipMalloc(&out_, n * 4096 * sizeof(float)));
    CCHECK(hipMalloc(&g3_, n * 4096 * sizeof(float)));
    CCHECK(hipMalloc(&part_, n * kCnnParams * sizeof(float)));
    max_batch_ = nimg;
}

// segments of the forward march: 4 of 8 steps up to 64 images, 2 of 10 and 12 up
// to 128 (256 workgroups of 64 KB LDS, one per CU), 1 of 18 beyond, where the
// recomputed planes would cost more than idle CUs.  37 images 38 -> 22 us, with
// the activations stored 42 -> 25; 128 images 39 -> 29.
static unsigned fwd_segments(long long nimg) { return nimg <= 64 ? 4 : (nimg <= 128 ? 2 : 1); }

void CnnModel::infer(const float *x, float *out, long long nimg, hipStream_t stream) {
    if (nimg <= 0) return;
    pack(stream);
    hipLaunchKernelGGL((k_cnn_fwd<false, false, kFwdWaves>), dim3((unsigned)nimg, fwd_segments(nimg)), dim3(64 * kFwdWaves), 0, stream, x, out,
                       (const uint16_t *)packed_ + PK_TOTAL * 8, (const float *)params_,
                       (uint16_t *)nullptr, (uint16_t *)nullptr, HeatIO{}, (const long long *)nullptr);
}

void CnnModel::infer_heat(const float *x, const double *scale, int scale_stride, int nb, long long istride, double *c,
                          long long nimg, const int *active, hipStream_t stream) {
    if (nimg <= 0) return;
    pack(stream);
    HeatIO hio{scale, scale_stride, nb, istride, c, active};
    hipLaunchKernelGGL((k_cnn_fwd<false, true, kFwdWaves>), dim3((unsigned)nimg), dim3(64 * kFwdWaves), 0, stream, x, (float *)nullptr,
                       (const uint16_t *)packed_ + PK_TOTAL * 8, (const float *)params_,
                       (uint16_t *)nullptr, (uint16_t *)nullptr, hio, (const long long *)nullptr);
}

void CnnModel::backward(const float *x, const float *g3, const long long *idx, int nimg, hipStream_t stream) {
    hipLaunchKernelGGL(k_cnn_dgrad1, dim3(nimg, 16 / DPL), dim3(256), 0, stream, g3, (const uint16_t *)h2_, g2_,
                       (const us8 *)packed_);
    hipLaunchKernelGGL(k_cnn_dgrad16, dim3(nimg, 16 / DPL), dim3(256), 0, stream, (const uint16_t *)g2_,
                       (const uint16_t *)h1_, g1_, (const us8 *)packed_);
    hipLaunchKernelGGL(k_cnn_wgrad, dim3(nimg, 7), dim3(256), 0, stream, x, (const uint16_t *)h1_, (const uint16_t *)h2_,
                       (const uint16_t *)g1_, (const uint16_t *)g2_, g3, part_, idx);
}

void CnnModel::gradient(const float *x, const float *gout, int nimg, double *grad_host, hipStream_t stream) {
    ensure_batch(nimg);
    pack(stream);
    hipLaunchKernelGGL((k_cnn_fwd<true, false, kFwdWaves>), dim3(nimg, fwd_segments(nimg)), dim3(64 * kFwdWaves), 0, stream, x, out_,
                       (const uint16_t *)packed_ + PK_TOTAL * 8, (const float *)params_, h1_, h2_, HeatIO{}, (const long long *)nullptr);
    backward(x, gout, nullptr, nimg, stream);
    hipLaunchKernelGGL(k_cnn_reduce, dim3((kCnnParams + 63) / 64), dim3(64), 0, stream, (const float *)part_, nimg, grad_);
    CCHECK(hipStreamSynchronize(stream));
    CCHECK(hipMemcpy(grad_host, grad_, sizeof(double) * kCnnParams, hipMemcpyDeviceToHost));
}

void CnnModel::train_step(const float *x, const float *y, const long long *idx, int nimg, double lr, bool first,
                          hipStream_t stream) {
    pack(stream);
    hipLaunchKernelGGL((k_cnn_fwd<true, false, kFwdWaves>), dim3(nimg, fwd_segments(nimg)), dim3(64 * kFwdWaves), 0, stream, x, out_,
                       (const uint16_t *)packed_ + PK_TOTAL * 8, (const float *)params_, h1_, h2_, HeatIO{}, idx);
    const long long n = 4096LL * nimg;
    int nwg = nimg < 1024 ? nimg : 1024;
    double scale = 1.0 / (double)n;
    if (h1_alpha_ >= 0.0 && loss_cos_) {
        // mean over the images of the scale-free loss
        scale = 1.0 / (double)nimg;
        hipLaunchKernelGGL(k_cnn_loss_cos, dim3(nwg), dim3(256), 0, stream, (const float *)out_, y, nimg,
                           (float)h1_alpha_, (float)h1_w_[0], (float)h1_w_[1], (float)h1_w_[2], (float)scale, g3_,
                           loss_part_, idx);
    } else if (h1_alpha_ >= 0.0) {
        hipLaunchKernelGGL(k_cnn_loss_h1, dim3(nwg), dim3(1024), 0, stream, (const float *)out_, y, nimg,
                           (float)h1_alpha_, (float)h1_w_[0], (float)h1_w_[1], (float)h1_w_[2], (float)scale, g3_,
                           loss_part_, idx);
    } else {
        nwg = 1024;
        hipLaunchKernelGGL(k_cnn_loss, dim3(nwg), dim3(256), 0, stream, (const float *)out_, y, n, g3_, loss_part_, idx);
    }
    backward(x, g3_, idx, nimg, stream);
    adam_t_++;
    const float c1 = (float)(1.0 / (1.0 - std::pow(0.9, (double)adam_t_)));
    const float c2 = (float)(1.0 / (1.0 - std::pow(0.999, (double)adam_t_)));
    hipLaunchKernelGGL(k_cnn_update, dim3((kCnnParams + 63) / 64 + 1), dim3(64), 0, stream, (const float *)part_, nimg,
                       params_, adam_m_, adam_v_, (float)lr, c1, c2, (const double *)loss_part_, nwg, scale, (double)nimg,
                       first, loss_part_ + 1024);
    packed_valid_ = false;
}

double CnnModel::train(const float *x, const float *y, long long nimg, int epochs, int batch, double lr, uint64_t seed,
                       hipStream_t stream) {
    if (nimg <= 0 || epochs <= 0) return 0.0;
    batch = (int)std::min<long long>(batch, nimg);
    ensure_batch(batch);
    std::mt19937_64 rng(seed);
    std::vector<long long> idx(nimg);
    long long *didx = nullptr;
    CCHECK(hipMalloc(&didx, sizeof(long long) * nimg));
    double last = 0.0;
    try {
        // the steps run on without the host: the loss adds up on the device
        // and is read once, the batches are read in place by index
        long long seen = 0;
        for (int ep = 0; ep < epochs; ep++) {
            // learning rate decays linearly from lr to lr/10 over the epochs
            const double lr_ep = epochs > 1 ? lr * (1.0 - 0.9 * (double)ep / (double)(epochs - 1)) : lr;
            for (long long i = 0; i < nimg; i++) idx[i] = i;
            std::shuffle(idx.begin(), idx.end(), rng);
            CCHECK(hipStreamSynchronize(stream));     // the previous epoch's steps read didx
            CCHECK(hipMemcpy(didx, idx.data(), sizeof(long long) * nimg, hipMemcpyHostToDevice));
            seen = 0;
            for (long long b0 = 0; b0 + batch <= nimg; b0 += batch) {
                train_step(x, y, didx + b0, batch, lr_ep, b0 == 0, stream);
                seen += batch;
            }
            CCHECK(hipGetLastError());
        }
        double tot = 0.0;
        CCHECK(hipStreamSynchronize(stream));
        CCHECK(hipMemcpy(&tot, loss_part_ + 1024, sizeof(double), hipMemcpyDeviceToHost));
        last = seen ? tot / (double)seen : 0.0;
    } catch (...) {
        (void)hipStreamSynchronize(stream);
        (void)hipFree(didx);
        throw;
    }
    CCHECK(hipFree(didx));
    return last;
}

}  // namespace falcon
