// Local relative-position attention of one 16-query tile of one head in fp32
// (encoder.cu:1338-1461 and the per-query path :1548-1684): the fp16 short
// form and the boundary tiles of the long forms.
//
// One 512-thread workgroup per (tile, head).  The operands are fp32 (q + u and
// q + v unrounded, fp16 / e4m3 K, V and positions widened), so the products
// run on v_mfma_f32_16x16x4_f32: content scores of the 16 queries against the
// tile's window of up to 272 keys and position scores against the 272
// position rows, skewed together in LDS (key column c of query r meets
// position row c - r), the softmax of two queries per wave, and the context of
// 32 features and half the keys per wave.  The MFMA's K index is free as long
// as both operands use one order: lane group g takes dimensions 32 g .. 32 g +
// 31 (36 or 32 consecutive key columns in the context), so that a lane's
// operands are contiguous in memory.
//
// Rows come in as whole 256-byte rows (16 lanes a row) and reach operand order
// (row l16, dimensions 32 g ..) through a 4 KiB block of LDS a wave: loaded in
// operand order, consecutive lanes are different rows and a load costs 64 line
// accesses.  About 12 us a tile: 1.5 for the queries, 4.5 for the scores, 1.6
// for the softmax, 2.8 for the context (the fp32 MFMAs of the two are 4), the
// rest staging and barriers.  One wave per (query, head) on the vector ALUs
// took 55 us for the boundary tiles of 750 frames and up, this 18-19 us.
#pragma once

#include <float.h>

#include "pk_attention_rule.hpp"
#include "pk_common.hpp"

namespace pk {

struct AttentionTileArgs {
    const uint16_t *query, *key, *position, *bias_u, *bias_v;
    const void* value;  // e4m3 (v * 56) feature-major [1024 x value_stride], or fp16 [rows x 1024] (short form)
    void* output;
    int rows, padded_rows, valid_rows, left, right, value_stride;
    int ib, ie;  // tiles [0, ib) and ie, ie + 1, ...
};

enum AttentionTileMode { kTilePacked = 0, kTileTc = 1, kTileShort = 2 };  // e4m3 x28 / fp16 / fp16 output

constexpr int kTileThreads = 512;

template <int kMode>
__global__ __launch_bounds__(kTileThreads, 2) void attention_tile_kernel(AttentionTileArgs p) {
    constexpr int kModel = 1024, kHead = 128, kPosRows = 272, kCols = 272, kStride = 276;
    constexpr int kVRow = kMode == kTileShort ? 72 : 152;  // staged V row: 32 features of a key / up to 144 keys of a feature, padded
    constexpr int kVRows = kMode == kTileShort ? 144 : 32;
    __shared__ __attribute__((aligned(16))) float buf[2][16][kStride];  // content scores, then weights; position scores
    // Per wave: one block of 16 key or position rows (16-byte chunk c of row r
    // at c ^ r), and its part of V.
    __shared__ __attribute__((aligned(16))) uint8_t row_s[8][16 * 256];
    __shared__ __attribute__((aligned(16))) uint8_t v_s[8][kVRows * kVRow];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, l16 = lane & 15;
    const int head = blockIdx.x & 7, ti = blockIdx.x >> 3;
    const int qb = 16 * (ti < p.ib ? ti : p.ie + (ti - p.ib));
    const int live_end = min(min(p.rows, p.valid_rows), p.padded_rows);  // queries [0, live_end) have an output
    const int first_key = qb - p.left;                                   // key of column 0
    auto store2 = [&](int qr, int feature, float a, float b) {
        const size_t at = (size_t)qr * kModel + head * kHead + feature;
        if constexpr (kMode == kTilePacked)
            *(uint16_t*)((uint8_t*)p.output + at) = (uint16_t)e4m3x2(round_f16(a) * 28.0f, round_f16(b) * 28.0f);
        else
            *(uint32_t*)((uint16_t*)p.output + at) = (uint32_t)f2h(a) | ((uint32_t)f2h(b) << 16);
    };
    // a wave's LDS accesses complete in order; the compiler must not move them
    auto wave_order = []() { asm volatile("" ::: "memory"); };
    if (qb < live_end) {
        const int last_key = tile_last_key(qb, live_end, p.valid_rows, p.right);
        // ---- values of features 32 (wave % 4) + 2 l16, + 1: the first four waves take
        // key columns 0 .. 143, the others 144 .. 271, lane group g columns 16 t + 4 g ..
        const int feature = 32 * (wave & 3) + 2 * l16, half = wave >> 2;
        const int per = half ? 32 : 36;
        constexpr int kQuads = 9;
        // 16-byte chunks, consecutive lanes on consecutive chunks of a row
        const int v_chunks = kMode == kTileShort ? 16 * per : 32 * (per / 4);
        auto v_row = [&](int i) { return kMode == kTileShort ? i >> 2 : i / (per / 4); };
        auto v_col = [&](int i) { return kMode == kTileShort ? i & 3 : i % (per / 4); };
        typedef uint32_t u32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));  // the short form's V is 4-byte aligned
        uint4 vw[kQuads];
        auto load_values = [&]() {
#pragma unroll
            for (int k = 0; k < kQuads; ++k) {
                const int i = min(lane + 64 * k, v_chunks - 1), r = v_row(i), c = v_col(i);
                const uint8_t* src;
                if constexpr (kMode == kTileShort) {
                    const int key = tile_key_row(first_key + 144 * half + r, last_key);
                    src = (const uint8_t*)p.value + ((size_t)key * kModel + head * kHead + 32 * (wave & 3)) * 2 + 16 * c;
                } else {
                    const int key = min(max(first_key + 144 * half + 16 * c, 0), p.value_stride - 16);
                    src = (const uint8_t*)p.value + (size_t)(head * kHead + 32 * (wave & 3) + r) * p.value_stride + key;
                }
                const u32x4_a4 w = *(const u32x4_a4*)src;
                vw[k] = uint4{w.x, w.y, w.z, w.w};
            }
        };
        auto stage_values = [&]() {
#pragma unroll
            for (int k = 0; k < kQuads; ++k) {
                const int i = lane + 64 * k;
                if (i < v_chunks) {
                    uint2* dst = (uint2*)&v_s[wave][v_row(i) * kVRow + 16 * v_col(i)];
                    dst[0] = uint2{vw[k].x, vw[k].y};
                    dst[1] = uint2{vw[k].z, vw[k].w};
                }
            }
        };
        // ---- scores: four waves content, four position, every fourth block of 16 columns
        const int c_lo = max(0, -first_key), c_hi = last_key - first_key;
        const int which = wave >> 2;
        const int b_lo = (which == 0 ? c_lo : max(0, c_lo - 15)) >> 4;
        const int b_hi = (which == 0 ? c_hi : min(p.left + p.right, c_hi)) >> 4;
        float a[32];
        {
            const uint16_t* q = p.query + (size_t)tile_query_row(qb + l16, live_end) * kModel + head * kHead + 32 * g;
            const uint16_t* u = (which == 0 ? p.bias_u : p.bias_v) + head * kHead + 32 * g;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint4 q4 = ((const uint4*)q)[i], u4 = ((const uint4*)u)[i];
                const uint32_t qw[4] = {q4.x, q4.y, q4.z, q4.w}, uw[4] = {u4.x, u4.y, u4.z, u4.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    a[8 * i + 2 * j] = h2f((uint16_t)qw[j]) + h2f((uint16_t)uw[j]);
                    a[8 * i + 2 * j + 1] = h2f((uint16_t)(qw[j] >> 16)) + h2f((uint16_t)(uw[j] >> 16));
                }
            }
        }
        // rows 4 i + g of block b, chunk l16: four whole rows an instruction
        auto load = [&](int b, v4i (&r)[4]) {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int col = 16 * b + 4 * i + g;
                const uint16_t* src = which == 0 ? p.key + (size_t)tile_key_row(first_key + col, last_key) * kModel + head * kHead
                                                 : p.position + ((size_t)head * kPosRows + min(col, kPosRows - 1)) * kHead;
                r[i] = ((const v4i*)src)[l16];
            }
        };
        // every block's rows, then the values, go out together: one latency
        // for the tile (a block's MFMAs take 0.5 us, a load from HBM 1-2 us)
        constexpr int kBlocks = (kCols / 16 + 3) / 4;
        const int b0 = b_lo + (wave & 3);
        v4i rows[kBlocks][4];
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
            if (b0 + 4 * i <= b_hi) load(b0 + 4 * i, rows[i]);
        load_values();
        auto score_block = [&](int b, const v4i (&x4)[4]) {
            if (b > b_hi) return;
            // through the wave's staging block into operand order: row l16, dimensions 32 g ..
#pragma unroll
            for (int q = 0; q < 4; ++q) *(v4i*)&row_s[wave][(4 * q + g) * 256 + ((l16 ^ (4 * q + g)) << 4)] = x4[q];
            wave_order();
            v4f s0 = {0.f, 0.f, 0.f, 0.f}, s1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint4 x = *(const uint4*)&row_s[wave][l16 * 256 + (((4 * g + q) ^ l16) << 4)];
                const uint32_t w[4] = {x.x, x.y, x.z, x.w};
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    s0 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[8 * q + 2 * j], h2f((uint16_t)w[j]), s0, 0, 0, 0);
                    s1 = __builtin_amdgcn_mfma_f32_16x16x4f32(a[8 * q + 2 * j + 1], h2f((uint16_t)(w[j] >> 16)), s1, 0, 0, 0);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) buf[which][4 * g + r][16 * b + l16] = s0[r] + s1[r];
            wave_order();
        };
        static_assert(kBlocks == 5, "");
        score_block(b0, rows[0]);
        score_block(b0 + 4, rows[1]);
        score_block(b0 + 8, rows[2]);
        score_block(b0 + 12, rows[3]);
        score_block(b0 + 16, rows[4]);
        stage_values();
        __syncthreads();
        // ---- softmax: two queries a wave; column c of query r is position row c - r
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int r = 2 * wave + i, qr = qb + r;
            constexpr int kPer = (kCols + 63) / 64;
            float e[kPer], mx = -FLT_MAX, den = 0.0f;
            bool in[kPer];
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                const int c = lane + 64 * k, m = c - r;
                in[k] = false;
                e[k] = -FLT_MAX;
                if (64 * k > c_hi || 64 * k + 63 < c_lo) continue;
                in[k] = qr < live_end && c >= c_lo && c <= c_hi && m >= 0 && m <= p.left + p.right;
                e[k] = in[k] ? (buf[0][r][c] + buf[1][r][m]) * 0.08838834764831845f : -FLT_MAX;
                mx = __builtin_fmaxf(mx, e[k]);
            }
            mx = wave_max(mx);
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                e[k] = in[k] ? __expf(e[k] - mx) : 0.0f;  // the reference's fast-math exponential (build.rs:68-73)
                den += e[k];
            }
            den = sum_desc<64>(den);
#pragma unroll
            for (int k = 0; k < kPer; ++k)
                if (lane + 64 * k < kCols) buf[0][r][lane + 64 * k] = in[k] ? e[k] / den : 0.0f;
        }
        __syncthreads();
        // ---- context
        v4f o0 = {0.f, 0.f, 0.f, 0.f}, o1 = {0.f, 0.f, 0.f, 0.f};
        bool odd = false;
        auto byte = [](uint32_t w, int i) {
            switch (i) {
                case 0: return __builtin_amdgcn_cvt_f32_fp8((int)w, 0);
                case 1: return __builtin_amdgcn_cvt_f32_fp8((int)w, 1);
                case 2: return __builtin_amdgcn_cvt_f32_fp8((int)w, 2);
                default: return __builtin_amdgcn_cvt_f32_fp8((int)w, 3);
            }
        };
        // this lane's two features at columns at .. at + 3 of its half, 0 for keys
        // outside [0, last_key] (past valid_rows the quantizer does not write the e4m3 bytes)
        auto values4 = [&](int at, float (&y0)[4], float (&y1)[4]) {
            uint32_t v0 = 0, v1 = 0;
            if constexpr (kMode != kTileShort) {
                v0 = *(const uint32_t*)&v_s[wave][2 * l16 * kVRow + at];
                v1 = *(const uint32_t*)&v_s[wave][(2 * l16 + 1) * kVRow + at];
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int key = first_key + 144 * half + at + i;
                const bool in = key >= 0 && key <= last_key;
                constexpr float kValueScale = 8.0f / 448.0f;  // V holds v * 56
                float a, b;
                if constexpr (kMode == kTileShort) {
                    const uint32_t w = *(const uint32_t*)&v_s[wave][(at + i) * kVRow + 4 * l16];
                    a = h2f((uint16_t)w);
                    b = h2f((uint16_t)(w >> 16));
                } else {
                    a = byte(v0, i) * kValueScale;
                    b = byte(v1, i) * kValueScale;
                }
                y0[i] = in ? a : 0.0f;
                y1[i] = in ? b : 0.0f;
            }
        };
#pragma unroll
        for (int t = 0; t < kQuads; ++t) {
            const int t16 = 144 * half + 16 * t;  // no key of the tile's window in these 16 columns: nothing to add
            if (4 * t >= per || t16 > c_hi || t16 + 15 < c_lo) continue;
            const int at = 16 * t + 4 * g, c0 = 144 * half + at;
            const float4 x4 = *(const float4*)&buf[0][l16][c0];
            const float x[4] = {x4.x, x4.y, x4.z, x4.w};
            float y0[4], y1[4];
            values4(at, y0, y1);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                odd = odd || !(__builtin_fabsf(y0[i]) + __builtin_fabsf(y1[i]) < __builtin_huge_valf());
                o0 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y0[i], o0, 0, 0, 0);
                o1 = __builtin_amdgcn_mfma_f32_16x16x4f32(x[i], y1[i], o1, 0, 0, 0);
            }
        }
        if (__builtin_amdgcn_ballot_w64(odd) != 0) {
            // An infinite or NaN value times the zero weight of a query whose window
            // it is not in would reach that query: sum the windows' own keys only.
            o0 = o1 = v4f{0.f, 0.f, 0.f, 0.f};
            for (int at = 0; at < 4 * per; at += 4) {
                float y0[4], y1[4];
                values4(at, y0, y1);
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int c = 144 * half + at + i, m = c - (4 * g + r);
                        if (c < c_lo || c > c_hi || m < 0 || m > p.left + p.right) continue;
                        o0[r] = __builtin_fmaf(buf[0][4 * g + r][c], y0[i], o0[r]);
                        o1[r] = __builtin_fmaf(buf[0][4 * g + r][c], y1[i], o1[r]);
                    }
            }
        }
        // the second half's sums join the first's (the position scores' space is free)
        float4* part = (float4*)buf[1] + ((wave & 3) * 64 + lane) * 2;
        if (half) {
            part[0] = float4{o0[0], o0[1], o0[2], o0[3]};
            part[1] = float4{o1[0], o1[1], o1[2], o1[3]};
        }
        __syncthreads();
        if (!half) {
            const float4 a0 = part[0], a1 = part[1];
            const float s0[4] = {a0.x, a0.y, a0.z, a0.w}, s1[4] = {a1.x, a1.y, a1.z, a1.w};
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int qr = qb + 4 * g + r;
                const bool on = qr < live_end;
                if (qr < p.padded_rows) store2(qr, feature, on ? o0[r] + s0[r] : 0.0f, on ? o1[r] + s1[r] : 0.0f);
            }
        }
    } else {
        for (int i = tid; i < 16 * kHead / 2; i += kTileThreads)
            if (qb + (i >> 6) < p.padded_rows) store2(qb + (i >> 6), 2 * (i & 63), 0.0f, 0.0f);
    }
}

}  // namespace pk
