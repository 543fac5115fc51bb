// One-bit fp4 weights x fp6 pieces of the input: the arithmetic of the run-list kernel at batch 8 and 16 on lists whose
// words are all in tile order.
//
// v_mfma_scale_f32_16x16x128_f8f6f4 with an fp4 (e2m1) A operand and an fp6 (e2m3) B operand multiplies 16 rows x 128
// columns of signs with 128 columns x 16 batch rows in 16 cycles, four times as many as v_mfma_f32_16x16x32 with 16-bit
// operands (with fp8 pieces: twice), and the weight operand of 32 signs costs one or two lane operations instead of 16:
// a nibble of a packed word, its class bit p moved to the nibble's sign, is the fp4 number +-1,
//     ((w << (3 - p)) & 0x88888888) | 0x22222222.
// The input is staged as kF6Pieces numbers per element, u = x * s / 2^k ~ q0 + q1 / 2^4 + q2 / 2^9, each the fp6 number
// nearest to what the ones before it left over; k is the power of two that brings the largest |u| of the element's UNIT
// (128 consecutive columns) into (3.75, 7.5], the top of the fp6 range, and rides along as the block scale of the MFMA
// (so do the factors 2^-4 and 2^-9).  Rounding to nearest leaves |error| <= 2^-12 for |u| >= 4 and <= 2^-13 below: an absolute
// step of at most 2^-13.9 and 2^-14.9 of the unit's largest value, the same for all of its 128 columns.  16-bit staging errs
// by a share of every element instead (2^-12 of it in fp16, 2^-9 in bf16) and not at all where x * s has 16 bits: it keeps
// more of an element below some 2^-3 (fp16) or 2^-6 (bf16) of its unit's maximum, and one below 2^-15 of it is lost here.
// What a sum keeps is decided by the large elements, and h, an fp32 vector, is not rounded to 16 bits either.  Error of a
// whole linear against 64 bits (2-norm; 16-bit operands -> here, batch 8 and 16 alike, 1024 x 4096 to 4096 x 11008):
//   channels of one size      fp16 2.9e-4 -> 1.0e-4, bf16 2.3e-3 -> 1.0e-4
//   four channels 100 times   fp16 3.0e-4 -> 1.4e-4, bf16 2.4e-3 -> 1.4e-4;   1000 times  3.1e-4 -> 1.6e-4, 2.9e-3 -> 1.6e-4
//   the same, s a power of 2  fp16 2.1e-4 -> 1.6e-4, bf16 1.6e-3 -> 1.5e-4;   1000 times  2.1e-4 -> 1.5e-4, 1.6e-3 -> 1.6e-4
// All signs are +-1 and products are exact, so nothing is subtracted again afterwards; all pieces of a batch row add into one
// fp32 accumulator (batch 16) or two (batch 8).  A unit that holds an infinity or a NaN gets the block scale NaN: its batch
// row comes out NaN, as it does with 16-bit operands (whose class sums take an infinity from itself).
//
// Operand geometry (one-hot operands on gfx950): lane (i = l & 15, g = l >> 4) supplies
//   A (fp4, 4 dwords): row i, k = 32 g + idx, idx = 8 d + e for nibble e of dword d;
//   B (fp6, 6 dwords): column i, k = 32 g + idx, element idx at bits 6 idx of the 192;
//   B block scale: byte `opsel` of the lane's scale register applies to column i, k = 32 g .. 32 g + 31.
// v_cvt_scalef32_2xpk16_fp6_f32 rounds to nearest even and puts its first 16 sources at the even idx, its second 16 at the odd.
// Lane g's 128 columns (unit 4 ub + g of row i) take four MFMAs n = 2 h + a: words 2 h and 2 h + 1, and of every octet of
// columns the half a (columns 8 o + 4 a .. + 3, which are classes 3, 2 for a = 0 and 1, 0 for a = 1), dwords d = 2 j +
// c: word 2 h + j, class 3 - 2 a - c.  In the "half2" order nibble e of class p is column 8 (3 - (e & 3)) + 2 (3 - p) +
// (e >> 2) of its word, so the lane that stages quarter n = 2 h + a of a unit needs eight runs of four columns and no
// exchange with its neighbours but the maximum.
#pragma once
#include "nq_decode.h"

namespace nq {

constexpr int kF6Pieces = 3;
constexpr int kF6Threads = 512;
constexpr int kF6Pairs = 4;                    // row pairs a wavefront keeps sums for when an input takes several chunks
typedef uint32_t u32x6_t __attribute__((ext_vector_type(6)));
typedef float float32_t __attribute__((ext_vector_type(32)));

// LDS: block (b, unit, n, piece) = 24 bytes, 16 in one array and 8 in another, both laid out [b][unit / 4][piece][n][unit % 4].
// A 16-byte read is served 16 lanes at a time, lanes 0-3 and 12-15 of one row of 16 with lanes 4-11 of the next (an
// 8-byte read 32 lanes in order): with a row pitch of 2 modulo 16 (32) blocks the lanes of unit g take the even blocks and
// those of unit g + 1 the odd ones, and batch 8's second piece, 16 blocks further, the other half: no bank conflicts.
template <int BATCH>
struct F6Layout {
    static_assert(BATCH == 8 || BATCH == 16, "operand columns are 16 batch rows, or 8 batch rows x 2 pieces");
    static constexpr int kGroup = 16 * kF6Pieces;                    // blocks of four units
    static constexpr int kPiece = 16, kStep = 4;                     // blocks from piece to piece, from n to n
    static __host__ __device__ constexpr int pitch16(int units4) { return 12 * units4 + 2; }                            // 48: a multiple of 16
    static __host__ __device__ constexpr int pitch8(int units4) { return 12 * units4 + ((2 - 12 * units4) & 31); }
    static __host__ __device__ constexpr int pitch_scale(int units4) { return units4 | 4; }                             // dwords; 4 modulo 8
    static __host__ __device__ constexpr size_t bytes16(int units4) { return (size_t)BATCH * pitch16(units4) * 16; }
    static __host__ __device__ constexpr size_t bytes8(int units4) { return (size_t)BATCH * pitch8(units4) * 8; }
    // (behind the last row of either array lies memory that batch 8's idle columns may read: the other array, the scales)
    static __host__ __device__ constexpr size_t bytes(int units4) {
        return bytes16(units4) + bytes8(units4) + (size_t)BATCH * pitch_scale(units4) * 4;
    }
};

// v -> its nearest fp6 numbers times `scale`, and v becomes what is left over (not for the last piece).
// The conversions take several passes over their operands: with the scale in the first result register the later elements
// were scaled by a result (the compiler does allocate it so).  The empty asm keeps every source alive beyond its
// conversion, so that no result register is a source.
template <bool LAST>
__device__ __forceinline__ u32x6_t f6_piece(float (&v)[32], float scale) {
    float16_t even, odd;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        even[i] = v[2 * i];
        odd[i] = v[2 * i + 1];
    }
    u32x6_t q = __builtin_amdgcn_cvt_scalef32_2xpk16_fp6_f32(even, odd, scale);
    asm volatile("" : "+v"(q) : "v"(even), "v"(odd), "v"(scale));
    if constexpr (!LAST) {
        float32_t back = __builtin_amdgcn_cvt_scalef32_pk32_f32_fp6(q, scale);
        asm volatile("" : "+v"(back) : "v"(q), "v"(scale));
#pragma unroll
        for (int i = 0; i < 32; ++i) v[i] -= back[i];
    }
    return q;
}

// keep ? own : other of the lane that differs in bit 0 (CTRL 0xB1) or bit 1 (0x4E)
template <int CTRL>
__device__ __forceinline__ uint32_t keep_or_swap(bool keep, uint32_t own, uint32_t other) {
    const uint32_t moved = dpp_mov_u32<CTRL>(other);
    return keep ? own : moved;
}

// Stages units [c0, c0 + cu_n) of BATCH rows, zeros up to a multiple of four units: a lane per quarter unit, wavefront w the
// batch rows w, w + 8, so that everything about a row is scalar and the column scales are unpacked once for both.  The four
// lanes of a unit load 64 contiguous bytes per instruction (an intermediate vector comes from the memory side, in pieces of
// 64 bytes whatever part of one is asked for) and deal the runs of their quarters out among themselves.  A barrier must
// follow before the staged data is read.
template <int DT, int BATCH>
__device__ __forceinline__ void stage_units_f6(uint4* x16, uint2* x8, uint32_t* scl, const StageInput& st, int c0, int cu_n) {
    using E = Elem<DT>;
    using L = F6Layout<BATCH>;
    constexpr int kRows = BATCH / 8;
    static_assert(kF6Threads == 8 * kWave, "eight wavefronts share the batch rows");
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int units4 = (cu_n + 3) & ~3;
    const int quarters = units4 * 4;
    const int pitch16 = L::pitch16(units4), pitch8 = L::pitch8(units4), pitch_scale = L::pitch_scale(units4);
    const uint32_t esize = st.in_f32 ? 4u : 2u;
    const uint32_t row_bytes = (uint32_t)st.in_stride * esize;
    const __amdgpu_buffer_rsrc_t rin = raw_buffer(st.in, (uint32_t)(((size_t)(BATCH - 1) * st.in_stride + st.K) * esize));
    const bool scaled = !st.in_f32 && st.s_col != nullptr;
    const __amdgpu_buffer_rsrc_t rsc = raw_buffer(scaled ? (const void*)st.s_col : st.in, scaled ? (uint32_t)st.K * 2u : 0u);
    // element `e` of run r (columns 32 (r >> 2) + 8 (r & 3) + e of the quarter) is v[idx], idx = 8 d + nibble as above
    auto idx = [](int r, int e) __attribute__((always_inline)) { return 16 * (r >> 2) + 8 * (e >> 1) + 4 * (e & 1) + 3 - (r & 3); };
    auto run_col = [](int r) __attribute__((always_inline)) { return 32 * (r >> 2) + 8 * (r & 3); };
    // One quarter: pieces and block scales into LDS.  All lanes of a quad (a unit) come here together.
    auto finish = [&](int b, int q, bool live, float (&v)[32]) __attribute__((always_inline)) {
        float m = 0.f;
#pragma unroll
        for (int i = 0; i < 32; ++i) m = __builtin_elementwise_maximum(m, __builtin_fabsf(v[i]));     // keeps a NaN
        uint32_t mb = as_bits(m);
        mb = max(mb, dpp_mov_u32<0xB1>(mb));
        mb = max(mb, dpp_mov_u32<0x4E>(mb));
        // biased exponent of the maximum, one more above 1.875 times a power of two: u = v / 2^(eb - 129)
        const uint32_t eb = min(max((mb + 0x000FFFFFu) >> 23, 32u), 254u);
        const u32x6_t q0 = f6_piece<false>(v, as_float((eb - 2u) << 23));
        const u32x6_t q1 = f6_piece<false>(v, as_float((eb - 6u) << 23));
        const u32x6_t q2 = f6_piece<true>(v, as_float((eb - 11u) << 23));
        const int cu = q >> 2, n = q & 3;
        const int block = (cu >> 2) * L::kGroup + n * L::kStep + (cu & 3);
        if (!live) return;
        uint4* d16 = x16 + b * pitch16 + block;
        uint2* d8 = x8 + b * pitch8 + block;
        d16[0] = make_uint4(q0[0], q0[1], q0[2], q0[3]); d8[0] = make_uint2(q0[4], q0[5]);
        d16[L::kPiece] = make_uint4(q1[0], q1[1], q1[2], q1[3]); d8[L::kPiece] = make_uint2(q1[4], q1[5]);
        d16[2 * L::kPiece] = make_uint4(q2[0], q2[1], q2[2], q2[3]); d8[2 * L::kPiece] = make_uint2(q2[4], q2[5]);
        // block scales of the three pieces, one byte each (0xFF: NaN); the last byte stays 0 (2^-127)
        if (n == 0) scl[b * pitch_scale + cu] = mb >= 0x7F800000u ? 0x00FFFFFFu : (eb - 2u) | ((eb - 6u) << 8) | ((eb - 11u) << 16);
    };
    const bool fast = st.vec_in && (st.K & 7) == 0;      // wide loads: what one of them asks for is whole or absent
#pragma unroll 1
    for (int q = lane; q - lane < quarters; q += kWave) {
        const bool live = q < quarters;
        const int col0 = (c0 + (q >> 2)) * 128 + 64 * ((q >> 1) & 1) + 4 * (q & 1);
        const int left = live ? st.K - col0 : 0;
        const int cu = q >> 2, t = q & 3;
        const bool odd = t & 1, upper = t & 2;           // a and h of the quarter this lane ends up with
        if (fast && st.in_f32) {
            // load j: columns 16 j + 4 t .. + 3 of the unit: word j >> 1, octet 2 (j & 1) + (t >> 1), half t & 1
            const int col = (c0 + cu) * 128 + 4 * t;
            const int have = live ? st.K - col : 0;
            u32x4_t x[kRows][8];
#pragma unroll
            for (int k = 0; k < kRows; ++k)
#pragma unroll
                for (int j = 0; j < 8; ++j)              // written by other workgroups of this launch or before it: device-coherent either way
                    x[k][j] = __builtin_amdgcn_raw_buffer_load_b128(rin, (have > 16 * j ? (uint32_t)col * 4u : kPastEnd) + 64u * j,
                                                                    (uint32_t)(wave + 8 * k) * row_bytes, kCacheAgentCoherent);
#pragma unroll
            for (int k = 0; k < kRows; ++k) {
                float v[32];
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t lo = x[k][j][e], hi = x[k][j + 4][e];
                        const int r = 4 * (j >> 1) + 2 * (j & 1);            // run of the even octet
                        v[idx(r, e)] = as_float(keep_or_swap<0x4E>(!upper, lo, hi));
                        v[idx(r + 1, e)] = as_float(keep_or_swap<0x4E>(upper, hi, lo));
                    }
                finish(wave + 8 * k, q, live, v);
            }
        } else if (fast) {
            // load w: octet t of word w; first the halves are dealt out (neighbouring lanes), then the words
            const int col = (c0 + cu) * 128 + 8 * t;
            const int have = live ? st.K - col : 0;
            uint32_t off[4];
#pragma unroll
            for (int w = 0; w < 4; ++w) off[w] = (have > 32 * w ? (uint32_t)col * 2u : kPastEnd) + 64u * w;
            u32x4_t c[4], x[kRows][4];
#pragma unroll
            for (int w = 0; w < 4; ++w) c[w] = __builtin_amdgcn_raw_buffer_load_b128(rsc, off[w], 0, kCacheDefault);
#pragma unroll
            for (int k = 0; k < kRows; ++k)
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    x[k][w] = __builtin_amdgcn_raw_buffer_load_b128(rin, off[w], (uint32_t)(wave + 8 * k) * row_bytes, kCacheDefault);
            // pair p (columns 2 p, 2 p + 1) of run r of this lane's quarter, as one dword
            auto deal = [&](const u32x4_t (&in)[4], uint32_t (&out)[8][2]) __attribute__((always_inline)) {
                uint32_t half[4][2][2];                  // [word][octet & 1][pair] of octets 2 (t >> 1), + 1
#pragma unroll
                for (int w = 0; w < 4; ++w)
#pragma unroll
                    for (int p = 0; p < 2; ++p) {
                        const uint32_t h0 = in[w][p], h1 = in[w][2 + p];
                        half[w][0][p] = keep_or_swap<0xB1>(!odd, h0, h1);
                        half[w][1][p] = keep_or_swap<0xB1>(odd, h1, h0);
                    }
#pragma unroll
                for (int w = 0; w < 2; ++w)
#pragma unroll
                    for (int o = 0; o < 2; ++o)
#pragma unroll
                        for (int p = 0; p < 2; ++p) {
                            out[4 * w + o][p] = keep_or_swap<0x4E>(!upper, half[w][o][p], half[w + 2][o][p]);
                            out[4 * w + 2 + o][p] = keep_or_swap<0x4E>(upper, half[w + 2][o][p], half[w][o][p]);
                        }
            };
            uint32_t pairs[8][2];
            float s[32];
            deal(c, pairs);
#pragma unroll
            for (int r = 0; r < 8; ++r)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const uint32_t w = pairs[r][e >> 1];
                    s[idx(r, e)] = scaled ? E::to_float((uint16_t)(e & 1 ? w >> 16 : w & 0xFFFFu)) : 1.f;
                }
#pragma unroll
            for (int k = 0; k < kRows; ++k) {
                float v[32];
                deal(x[k], pairs);
#pragma unroll
                for (int r = 0; r < 8; ++r)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t w = pairs[r][e >> 1];
                        // fused, adding 0: for fp16 one instruction that also unpacks x
                        v[idx(r, e)] = __builtin_fmaf(E::to_float((uint16_t)(e & 1 ? w >> 16 : w & 0xFFFFu)), s[idx(r, e)], 0.f);
                    }
                finish(wave + 8 * k, q, live, v);
            }
        } else {                                         // odd K or rows that allow no wide loads
#pragma unroll 1
            for (int b = wave; b < BATCH; b += 8) {
                float v[32];
#pragma unroll
                for (int r = 0; r < 8; ++r)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const bool in = left > run_col(r) + e;
                        const uint32_t at = (uint32_t)(col0 + run_col(r) + e);
                        if (st.in_f32) {
                            v[idx(r, e)] = as_float(__builtin_amdgcn_raw_buffer_load_b32(rin, in ? at * 4u : kPastEnd, (uint32_t)b * row_bytes, kCacheAgentCoherent));
                        } else {
                            const uint16_t xw = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rin, in ? at * 2u : kPastEnd, (uint32_t)b * row_bytes, kCacheDefault);
                            const uint16_t sw = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rsc, in ? at * 2u : kPastEnd, 0, kCacheDefault);
                            v[idx(r, e)] = E::to_float(xw) * (scaled ? E::to_float(sw) : 1.f);
                        }
                    }
                finish(b, q, live, v);
            }
        }
    }
}

// A operand of MFMA N for the 16-byte unit w of this lane's row; ones = 0x22222222 in a vector register, so that mask and
// one go into a single instruction
template <int N>
__device__ __forceinline__ v8i_t f6_weights(const u32x4_t& w, uint32_t ones) {
    constexpr uint32_t S = 0x88888888u;
    constexpr int sh = 2 * (N & 1);
    const uint32_t w0 = w[N & 2], w1 = w[(N & 2) + 1];
    return (v8i_t){(int)(((w0 << sh) & S) | ones), (int)(((w0 << (sh + 1)) & S) | ones), (int)(((w1 << sh) & S) | ones),
                   (int)(((w1 << (sh + 1)) & S) | ones), 0, 0, 0, 0};
}

template <int OPSEL>
__device__ __forceinline__ float4_t f6_mfma(const v8i_t& a, const v8i_t& b, int scale, const float4_t& acc) {
    return __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(a, b, acc, 4 /* A: fp4 */, 2 /* B: fp6 */, 0, 0x7F7F7F7F, OPSEL, scale);
}

// One MFMA step of two row groups that share the input operand.  Batch 16: the 16 operand columns are the batch rows, the
// three pieces one after the other.  Batch 8: columns 0-7 are piece 0 and columns 8-15 piece 1 of the batch rows; then
// piece 2 in columns 0-7, into accumulators of their own (columns 8-15 multiply whatever follows there, by the block scale
// 2^-127, the fourth byte of the scale word, and are dropped).  `scale`: the scale word of the lane's batch row and unit
// (batch 8, columns 8-15: moved down by a byte).
// p8, p8b, p8c: the same address, unknown to the compiler, which would merge neighbouring 8-byte reads into
// ds_read2_b64, at half their rate.
template <int BATCH, int N>
__device__ __forceinline__ void f6_read(v8i_t& b0, v8i_t& b1, v8i_t& b2, const uint4* p16, const uint2* p8, const uint2* p8b, const uint2* p8c) {
    using L = F6Layout<BATCH>;
    auto piece = [&](int k, const uint2* q8) __attribute__((always_inline)) {
        const u32x4_t lo = *(const u32x4_t*)(p16 + L::kStep * N + L::kPiece * k);
        const u32x2_t hi = *(const u32x2_t*)(q8 + L::kStep * N + L::kPiece * k);
        return (v8i_t){(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], 0, 0};
    };
    b0 = piece(0, p8);
    if constexpr (BATCH == 16) b1 = piece(1, p8b);
    b2 = piece(2, BATCH == 16 ? p8c : p8b);
}
template <int BATCH, int N>
__device__ __forceinline__ void f6_step(const u32x4_t& wa, const u32x4_t& wb, const v8i_t& b0, const v8i_t& b1, const v8i_t& b2,
                                        int scale, uint32_t ones, float4_t& acc_a, float4_t& acc_b, float4_t& tail_a, float4_t& tail_b) {
    const v8i_t aa = f6_weights<N>(wa, ones), ab = f6_weights<N>(wb, ones);
    acc_a = f6_mfma<0>(aa, b0, scale, acc_a);
    acc_b = f6_mfma<0>(ab, b0, scale, acc_b);
    if constexpr (BATCH == 16) {
        acc_a = f6_mfma<1>(aa, b1, scale, acc_a);
        acc_b = f6_mfma<1>(ab, b1, scale, acc_b);
    }
    tail_a = f6_mfma<2>(aa, b2, scale, tail_a);
    tail_b = f6_mfma<2>(ab, b2, scale, tail_b);
}
// The four steps of an item; the operand of a step is read while the one before it multiplies, and no earlier (all four
// would take 72 registers).
__device__ __forceinline__ void f6_order() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
}
template <int BATCH>
__device__ __forceinline__ void f6_item(const u32x4_t& wa, const u32x4_t& wb, const uint4* p16, const uint2* p8, int scale, uint32_t ones,
                                        float4_t& acc_a, float4_t& acc_b, float4_t& tail_a, float4_t& tail_b) {
    v8i_t o0 = {}, o1 = {}, o2 = {}, p0 = {}, p1 = {}, p2 = {};
    typedef const __attribute__((address_space(3))) uint2* lds_t;
    lds_t hb = (lds_t)p8, hc = (lds_t)p8;
    asm volatile("" : "+v"(hb), "+v"(hc));
    const uint2 *p8b = (const uint2*)hb, *p8c = (const uint2*)hc;
    f6_read<BATCH, 0>(o0, o1, o2, p16, p8, p8b, p8c);
    f6_order();
    f6_read<BATCH, 1>(p0, p1, p2, p16, p8, p8b, p8c);
    f6_step<BATCH, 0>(wa, wb, o0, o1, o2, scale, ones, acc_a, acc_b, tail_a, tail_b);
    f6_order();
    f6_read<BATCH, 2>(o0, o1, o2, p16, p8, p8b, p8c);
    f6_step<BATCH, 1>(wa, wb, p0, p1, p2, scale, ones, acc_a, acc_b, tail_a, tail_b);
    f6_order();
    f6_read<BATCH, 3>(p0, p1, p2, p16, p8, p8b, p8c);
    f6_step<BATCH, 2>(wa, wb, o0, o1, o2, scale, ones, acc_a, acc_b, tail_a, tail_b);
    f6_order();
    f6_step<BATCH, 3>(wa, wb, p0, p1, p2, scale, ones, acc_a, acc_b, tail_a, tail_b);
}

// Zeros made on the spot (constants would be kept, and spilled, across the loops that start from them)
__device__ __forceinline__ float4_t f6_zero() {
    float z = 0.f;
    asm volatile("" : "+v"(z));
    return (float4_t){z, z, z, z};
}

// Batch 8: the sum of a batch row's two operand columns (in all of its lanes)
template <int BATCH>
__device__ __forceinline__ float4_t f6_columns(float4_t v) {
    if constexpr (BATCH == 8)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const float t = v[k];
            v[k] = dpp_add<0x128>(t);                    // row_ror:8
        }
    return v;
}

}  // namespace nq
