// The lm_head projection in front of the sampler.
//
// The reference computes a decode step's logits with the model's output layer,
// an nn.Linear without bias in the model dtype (continuous_batching.py:1345,1594,
// 2225: `self._lm_head()(hidden)`), writes them to a buffer and hands that buffer
// to the sampler (:1926-1928).  Here logits = hidden · weightᵀ is computed on the matrix
// cores (bf16 or fp16 operands, fp32 accumulation over k in ascending steps of 32,
// rounded to nearest-even in the model dtype as the layer's output is) and written
// once; k_scan then reads it, mostly from the Infinity Cache.
//
// The weight is vocab x H and is read once whatever the batch, so small batches are
// bound by HBM (1.25 GB at vocab 151936 and H 4096, 240 us at the rate of a large copy)
// and large ones by the matrix cores and the LDS that feeds them.
#pragma once

#include "launchers.h"

namespace fie {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

// D += A (16 x 32) B (32 x 16).  Lane l supplies A's row l % 16 and B's column
// l % 16, eight consecutive k each from k-group l / 16; it receives D rows
// 4 (l / 16) .. +3 of column l % 16.  A and B take their k the same way, so the
// order the instruction pairs k in does not change the sum's terms.
template <int DT>
FIE_DEV f32x4_t mfma_16x16x32(u32x4_t a, u32x4_t b, f32x4_t c)
{
    if constexpr (DT == FIE_BF16)
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a),
                                                       __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a),
                                                      __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// fp32 to the logits dtype, round to nearest even (NaN stays NaN).
template <int DT>
FIE_DEV uint16_t round_logit(float v)
{
    if constexpr (DT == FIE_BF16) {
        uint32_t b = __float_as_uint(v);
        if ((b & 0x7FFFFFFFu) > 0x7F800000u) return (uint16_t)((b >> 16) | 0x40u);
        b += 0x7FFFu + ((b >> 16) & 1u);
        return (uint16_t)(b >> 16);
    } else {
        const _Float16 h = (_Float16)v;
        return __builtin_bit_cast(uint16_t, h);
    }
}

// Four consecutive tokens' logits of one row (the weight is the instruction's A, so a
// lane's four results are neighbours in memory): one 8-byte store where `wide` (rows and
// buffer 8-byte aligned) and all four are inside the vocabulary.
template <int DT>
FIE_DEV void store_logits(uint16_t* out, int64_t ld, int row, int tok, int V, bool wide, f32x4_t v)
{
    uint16_t* p = out + (size_t)row * (size_t)ld + tok;
    uint16_t h[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) h[i] = round_logit<DT>(v[i]);
    if (wide && tok + 4 <= V) {
        *(uint2*)p = make_uint2((uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16));
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
            if (tok + i < V) p[i] = h[i];
    }
}

// 64 WM rows by 64 WN tokens a workgroup of WM x WN waves, 64 x 64 each: 16 fragments
// from LDS per 32 matrix instructions and 64 of k, the ratio at which the LDS reads
// (128 bytes a cycle) take about as long as the instructions.  k goes in stages of 64
// through two LDS buffers, one barrier a stage; the next two stages are in flight in
// registers, and two workgroups share a CU where the buffers allow.
//
// Measured at vocab 151936, H 4096 (us; the GEMM fused with the scan that this replaces
// took 677 at 16 rows and 1090 at 256, a library product takes 261 and 394):
//   16 / 64 rows   1 x 4 waves 266 / 277, 1 x 2 waves 281 at 64; operands straight to
//                  registers without LDS 264 / 430
//   128 rows       2 x 2 waves 281, 2 x 4 waves 306
//   256 rows       2 x 4 waves 382, 4 x 2 waves 408, 2 x 2 waves 421, 4 x 4 waves 676
constexpr int kLhK = 64;

// Chunk c (of 8) of operand row n sits at slot n * 8 + (c ^ (n & 7)): the eight
// lanes one LDS cycle serves read eight rows' chunk c from eight distinct bank groups.
FIE_DEV int lh_slot(int n, int c) { return n * 8 + (c ^ (n & 7)); }

// Grid: 8 * ceil(tiles / 8) * nrb workgroups.  Workgroups are dealt to the eight XCDs
// round robin, so b, b + 8, b + 16, ... share one XCD; there, the nrb row blocks of a
// tile come one after another and read its weight rows through that XCD's L2.
template <int DT, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN, 2) void k_lmhead_tile(const uint16_t* __restrict__ hid,
                                                               const uint16_t* __restrict__ wt, uint16_t* out,
                                                               int64_t ld, int B, int V, int H, int nrb, int wide)
{
    constexpr int BM = 64 * WM, BN = 64 * WN, TH = 64 * WM * WN;
    constexpr int NC = (BM + BN) * (kLhK / 8) / TH;             // 16-byte chunks per thread and stage
    __shared__ u32x4_t L[2][(BM + BN) * (kLhK / 8)];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int xcd = blockIdx.x & 7, k = blockIdx.x >> 3;
    const int t0 = (8 * (k / nrb) + xcd) * BN, r0 = (k % nrb) * BM;
    if (t0 >= V) return;
    const uint16_t* src[NC];
    int dst[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) {
        const int p = j * TH + tid, n = p >> 3, c = p & 7;
        src[j] = (n < BM ? hid + (size_t)min(r0 + n, B - 1) * H : wt + (size_t)min(t0 + n - BM, V - 1) * H) + 8 * c;
        dst[j] = lh_slot(n, c);
    }
    const int ns = H / kLhK;
    u32x4_t ra[NC], rb[NC];
    auto load = [&](u32x4_t (&r)[NC], int s) {
        const int k0 = (s < ns ? s : ns - 1) * kLhK;            // past the end: again, unused
#pragma unroll
        for (int j = 0; j < NC; ++j) r[j] = *(const u32x4_t*)(src[j] + k0);
    };
    auto put = [&](const u32x4_t (&r)[NC], int b) {
#pragma unroll
        for (int j = 0; j < NC; ++j) L[b][dst[j]] = r[j];
    };
    const int wr = wave % WM, wn = wave / WM;
    f32x4_t acc[4][4];
#pragma unroll
    for (int m = 0; m < 4; ++m)
#pragma unroll
        for (int q = 0; q < 4; ++q) acc[m][q] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
    auto mul = [&](int b) {
#pragma unroll
        for (int kk = 0; kk < kLhK / 32; ++kk) {
            const int c = kk * 4 + (lane >> 4);
            u32x4_t fh[4], fw[4];
#pragma unroll
            for (int m = 0; m < 4; ++m) fh[m] = L[b][lh_slot(64 * wr + 16 * m + (lane & 15), c)];
#pragma unroll
            for (int q = 0; q < 4; ++q) fw[q] = L[b][lh_slot(BM + 64 * wn + 16 * q + (lane & 15), c)];
#pragma unroll
            for (int m = 0; m < 4; ++m)
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[m][q] = mfma_16x16x32<DT>(fw[q], fh[m], acc[m][q]);
        }
    };
    load(ra, 0);
    load(rb, 1);
    put(ra, 0);
    load(ra, 2);
    __syncthreads();
    for (int s = 0; s < ns; s += 2) {           // H is a multiple of 128: ns is even
        put(rb, 1);
        load(rb, s + 3);
        mul(0);
        __syncthreads();
        put(ra, 0);
        load(ra, s + 4);
        mul(1);
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < 4; ++m) {
        const int row = r0 + 64 * wr + 16 * m + (lane & 15);
        if (row >= B) continue;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            store_logits<DT>(out, ld, row, t0 + 64 * wn + 16 * q + 4 * (lane >> 4), V, wide, acc[m][q]);
    }
}

}  // namespace fie
