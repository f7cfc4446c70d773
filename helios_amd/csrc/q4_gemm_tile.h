// Device pieces shared by the prefill GEMM kernels (q4_gemm.hip, q4_gemm_kpair.hip): the
// bias term's MFMA operands, the tile order and the LoRA epilogue.
#pragma once

#include "q4_common.h"
#include "q4_kernels.h"

namespace q4 {
namespace {

// The bias MFMA's A operand for one 16-row tile and one octet, as 64 lanes of 16 B:
// lane (m = l%16, kq = l/16), element e -> group 8*octet + 2*kq + e/4, term e%4 in
// {Xh, Xl, c Xh, c Xl} (c = -16, or 8 in the fp16 form).  Lane (m, kq) packs it from X
// of row m for groups 2kq and 2kq + 1.
template <int C = -16>
__device__ __forceinline__ uint4 bias_a_operand(float x0, float x1) {
    uint32_t w[4];
    const float xs[2] = {x0, x1};
#pragma unroll
    for (int gi = 0; gi < 2; ++gi) {
        const uint16_t xh = f32_to_bf16(xs[gi]);
        const uint16_t xl = f32_to_bf16(xs[gi] - __uint_as_float((uint32_t)xh << 16));
        const uint16_t nxh = f32_to_bf16((float)C * __uint_as_float((uint32_t)xh << 16));
        const uint16_t nxl = f32_to_bf16((float)C * __uint_as_float((uint32_t)xl << 16));
        w[2 * gi] = (uint32_t)xh | ((uint32_t)xl << 16);
        w[2 * gi + 1] = (uint32_t)nxh | ((uint32_t)nxl << 16);
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

// B operand of the bias MFMA from one scale/bias word pair: [b0 b0 s0 s0 b1 b1 s1 s1]
__device__ __forceinline__ bf16x8 bias_operand(uint2 sbw) {
    uint4 d;
    d.x = __builtin_amdgcn_perm(sbw.x, sbw.x, 0x03020302u);  // b0 | b0 << 16
    d.y = __builtin_amdgcn_perm(sbw.x, sbw.x, 0x01000100u);  // s0 | s0 << 16
    d.z = __builtin_amdgcn_perm(sbw.y, sbw.y, 0x03020302u);
    d.w = __builtin_amdgcn_perm(sbw.y, sbw.y, 0x01000100u);
    return __builtin_bit_cast(bf16x8, d);
}

// Tile order: the hardware deals workgroup ids round-robin over the 8 XCDs; give
// each XCD a contiguous run of tiles, and walk tiles in bands of two M tiles
// (M fastest) so workgroups running together share x rows and weight tiles in L2.
__device__ __forceinline__ void tile_of(int id, int nwg, int mtiles, int ntiles, int& mt, int& nt) {
    constexpr int kXcds = 8;
    int tile = id;
    if (nwg % kXcds == 0) tile = (id % kXcds) * (nwg / kXcds) + id / kXcds;
    constexpr int kBand = 2;
    const int band = tile / (kBand * ntiles);
    const int r = tile - band * kBand * ntiles;
    const int bm = (mtiles - band * kBand) < kBand ? (mtiles - band * kBand) : kBand;
    mt = band * kBand + r % bm;
    nt = r / bm;
}

// t = x . A^T of a workgroup's BM rows into LDS (`ts`, [BM][rank] floats: the x ring's
// first slot, BM x 128 bytes, so rank <= 32), each entry summed over its slices in
// slice order; rows past the output read as zeros.  All of the workgroup's threads,
// one barrier after.
template <int BM>
__device__ __forceinline__ void lora_stage_t(const LoraEpilogue& lo, float* ts, int row0, int m_rows, int nthr) {
    const int q4s = lo.rank >> 2;  // float4s per row
    for (int t = (int)threadIdx.x; t < BM * q4s; t += nthr) {
        const int row = t / q4s, r = 4 * (t - row * q4s);
        const int m = row0 + row;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (m < m_rows) {
            v = *reinterpret_cast<const float4*>(lo.part + (long)m * lo.rank + r);
            for (int sl = 1; sl < lo.slices; ++sl) {
                const float4 u = *reinterpret_cast<const float4*>(lo.part + ((long)sl * m_rows + m) * lo.rank + r);
                v.x = v.x + u.x;
                v.y = v.y + u.y;
                v.z = v.z + u.z;
                v.w = v.w + u.w;
            }
        }
        *reinterpret_cast<float4*>(ts + row * lo.rank + r) = v;
    }
    __syncthreads();
}

// The LoRA delta of a wave's output tiles and the combined store, in lora_up's
// rounding steps (q4_lora.hip): d[m, n] = sum_r t[m, r] B[n, r] in fp32 on the matrix
// cores (16x16x4), as close to the exact sum as lora_up's, which takes the delta of plans
// that split K; then y = bf16(bf16(acc) + bf16(d * bf16(scale))) in bf16, acc + d * scale
// in fp32.  Lane (row or column, kq) holds ranks 4 kq .. 4 kq + 3 of each 16, one float4
// for four products; columns past the output and ranks past the adapter's are zeros.
// (t and B in two bf16 parts, three 16x16x32 products, left an fp32 output's delta
// 74 x 2^-24 off, so 3; the time is the same on kpair tiles, q|k|v|o of 1100 rows at rank
// 16 202 us, and 240 / 242 us for gate at 2048 rows and rank 16, 255 / 263 at rank 32.)
template <bool F32, int kMT, int kNT>
__device__ __forceinline__ void lora_store(const f32x4 (&acc)[kMT][kNT], const LoraEpilogue& lo, const float* ts,
                                           void* y, int row0, int rb0, int m_rows, int n_rows, int lane) {
#pragma clang fp contract(off)
    const int col = lane & 15, kq = lane >> 4;
    const int r0 = 4 * kq, r1 = 16 + 4 * kq;
    const float4 zero4 = make_float4(0.f, 0.f, 0.f, 0.f);
    float4 b0[kNT], b1[kNT];
#pragma unroll
    for (int j = 0; j < kNT; ++j) {
        const int n = (rb0 + j) * 16 + col;
        const bool ok = n < n_rows;
        const float* bp = lo.b + (long)(ok ? n : 0) * lo.rank;
        b0[j] = ok && r0 < lo.rank ? *reinterpret_cast<const float4*>(bp + r0) : zero4;
        b1[j] = ok && r1 < lo.rank ? *reinterpret_cast<const float4*>(bp + r1) : zero4;
    }
    const float sc = F32 ? lo.scale : (float)(__bf16)lo.scale;
    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < kMT; ++i) {
        const float* tp = ts + (16 * i + col) * lo.rank;
        const float4 t0 = r0 < lo.rank ? *reinterpret_cast<const float4*>(tp + r0) : zero4;
        const float4 t1 = r1 < lo.rank ? *reinterpret_cast<const float4*>(tp + r1) : zero4;
#pragma unroll
        for (int j = 0; j < kNT; ++j) {
            f32x4 d = mfma16x16x4(t0.x, b0[j].x, zero);
            d = mfma16x16x4(t0.y, b0[j].y, d);
            d = mfma16x16x4(t0.z, b0[j].z, d);
            d = mfma16x16x4(t0.w, b0[j].w, d);
            if (lo.rank > 16) {
                d = mfma16x16x4(t1.x, b1[j].x, d);
                d = mfma16x16x4(t1.y, b1[j].y, d);
                d = mfma16x16x4(t1.z, b1[j].z, d);
                d = mfma16x16x4(t1.w, b1[j].w, d);
            }
            const int n = (rb0 + j) * 16 + col;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int mr = row0 + 16 * i + 4 * kq + e;
                if (mr < m_rows && n < n_rows) {
                    const long o = (long)mr * n_rows + n;
                    if constexpr (F32) {
                        const float delta = d[e] * lo.scale;
                        static_cast<float*>(y)[o] = acc[i][j][e] + delta;
                    } else {
                        const float base = (float)(__bf16)acc[i][j][e];
                        const float delta = (float)(__bf16)(d[e] * sc);
                        static_cast<uint16_t*>(y)[o] = f32_to_bf16(base + delta);
                    }
                }
            }
        }
    }
}

}  // namespace
}  // namespace q4
