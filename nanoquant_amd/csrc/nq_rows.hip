// Decode path, per linear and per group of linears (1 to 16 batch rows): the two stages of a binary low-rank layer.
//
// One stage computes, for a packed sign matrix W [rows, words] in the row-major "half2" word order,
//     out[b, row] = s_row[row] * sum_c sgn(W[row, c]) * (in[b, c] * s_col[c])
// A layer is two stages: rows = rank over K = in_features (input x, scales s_in / s_mid, result h), then
// rows = out_features over K = rank (input h, scale s_out, result y).  Replaces nanoquant_stage1_impl /
// nanoquant_stage2_impl of the reference (src/nanoquant/kernel/cuda/gemv_kernel.cu:43-277); the packed words are read
// once for all batch rows (the reference re-reads them per row, :288-290) and all sums are fp32 (:103-106 sums in fp16).
//
// What bounds it: a stage is 1-6 MB of signs, a fraction of a microsecond of HBM time, so latency decides: the launch,
// one round trip to memory, and how evenly the words are spread over the chip.  Mapping: a workgroup owns 16 F rows and
// ALL columns; its wavefronts split the COLUMNS in chunks of 512.  A wavefront fetches 16 rows x 4 16-byte units with
// one 128-bit load per lane, and only ITS 512 columns of the input, so nothing is staged twice in a workgroup and no
// barrier stands between the first load and the arithmetic (a workgroup that stages the whole input first puts a
// barrier and its slowest load there).  The signs become +-1 operands of v_mfma_f32_16x16x32 with two lane
// operations per pair (16 rows x 16 batch columns: one decoded operand serves every batch row, so 16 rows cost what
// one costs but for the staging); the partial tiles of the wavefronts are added through LDS in a fixed order, which
// makes results reproducible and independent of what shares the launch.
//
// Measured on the projections of a decoder layer as {q,k,v} {o} {gate,up} {down} (eight launches, graph replays), against
// lane groups of dot products with all columns in one wavefront: 52 -> 46 us (1 row, 4096/11008, fp16), 149 -> 48 us
// (4 rows, 4096/12288, bf16; the second stages ran on 32-64 workgroups); one 4096 x 11008 linear on 11 rows of bf16
// 83 -> 16 us (it was split into 8 + 2 + 1 rows).
#include "nq_decode.h"
#include "nq_kernels.h"

#include <algorithm>
#include <atomic>
#include <type_traits>

namespace nq {

constexpr int kChunkCols = 512;      // columns of one wavefront step: 4 lane groups x one 16-byte unit of words
constexpr int kRowsMaxWaves = 8;     // wavefronts of a workgroup
// How a launch is cut, us per launch (graph replays over rotating weights, 16 rows fp16 / 4 rows bf16 / 1 row fp16):
//   two 16-row blocks per workgroup instead of one  rank 3 x 2048 of 4096   6.3 / 5.7 / 5.4   against 9.4 / 5.8 / 5.1
//                                                   out 4096 of rank 2048   5.1 / 4.6 / 4.3   against 4.9 / 4.0 / 3.9
//   (from 5 batch rows on the staged input of a workgroup fills half or all of a CU's LDS, so that more workgroups than
//   CUs run in rounds; with few rows a second block only makes a wavefront's chain longer)
//   four wavefronts instead of eight                out 22016 of rank 2992  10.5 / 8.1 / 7.5  against 14.1 / 9.0 / 7.8
//                                                   rank 2985 of 11008      12.4 / 8.4 / 7.1  against 10.3 / 7.1 / 5.8
//   (many rows: more workgroups stay resident and each stages less; few rows: eight keep more loads in flight).  The line
//   between is a compromise over the batch sizes, since the split decides the order of the sums and must not depend on them: whole
//   linears of 8192 to 14336 rows lose 3 to 5 % on four wavefronts at 1 to 8 rows (9216 x 4096, 1 row fp16: 10.0 against 9.4) and
//   gain 11 to 15 % at 16 rows (13.8 against 15.4), from 14336 rows on four are level (2 %) or ahead at every batch size; below 8192
//   rows they lose 1 to 6 % throughout (5120 x 8192: 12.3 against 11.6 at 8 rows).
constexpr int kTwoBlocksFrom = 257;  // 16-row blocks of a launch, 5 batch rows and more
constexpr int kFewWavesFrom = 8192;  // rows of a linear
// Up to this many staged rows the input operands are read two steps ahead of their products (left to itself the compiler waits
// for every pair of reads; with more rows the workgroups that share a compute unit hide that, and the registers count): layer of
// four groups, stages repeated, 1 / 4 / 11 rows fp16: 35.6 / 39.0 / 49.1 us without, 34.3 / 38.6 / 50.6 with; four or eight steps
// ahead 34.7 / 39.3 / 50.9 and 35.6 / 42.0 / 52.2.  At 5 and 8 rows the two are within 1 % (four groups of two launches: fp16 42.4 and
// 42.9 us without, 42.3 and 42.9 with, bf16 43.3 and 43.8, 43.1 and 43.8; linears by themselves in bf16 64.4 and 65.3, 63.9 and 64.9).
constexpr int kReadAheadRows = 4;
constexpr int kStagePitch = 1040;    // LDS bytes per staged input row of a chunk: 512 x 2 + 16 (8 lanes of an operand
                                     // read that differ in the batch row only hit 8 different bank groups)

// One sign matrix with its input.
struct RowsTerm {
    const uint32_t* bits;   // [rows, words]
    const uint16_t* in;     // [batch, in_stride], 16-bit activations or 16-bit h
    const uint16_t* s_col;  // [K], SCALED only
    const uint16_t* s_row;  // [rows] or null
    int words, K, in_stride, chunks;
};
enum RowsOut { kOutY = 0, kOutF32 = 1, kOutH = 2 };   // kOutH: 16-bit, unclamped, zeros up to out_stride rows
template <int NT>
struct RowsProblem {
    RowsTerm t[NT];         // NT > 1: the results of the terms are added (mixture of ranks)
    const uint16_t* bias;   // [rows] or null
    const float* addend;    // [batch, out_stride] or null
    void* out;              // [batch, out_stride]
    int rows, out_stride, waves;
    int out_kind;           // RowsOut
};
// Up to N linears per launch: their workgroups one behind the other.  A launch takes the smallest table that holds its
// linears (one, {gate, up} and {q, k, v}, more): kernel arguments are read from memory at the start of every workgroup, with all
// else waiting, and eight entries are 800 bytes of them.  Llama-2-7B layer as four groups of two launches in a graph, 1 / 4 / 11
// rows of fp16: always eight entries and an entry looked up by its index 43.0 / 47.6 / 58.4 us, this 38.3 / 42.9 / 54.6.
constexpr int kGroupMax = 8;
template <int NT, int N>
struct RowsGroup {
    int batch, waves;                // wavefronts of a workgroup
    int first[N + 1];                // first workgroup of every problem; [N] = the grid
    RowsProblem<NT> p[N];
};

template <bool COHERENT>
constexpr int rows_cache() { return COHERENT ? kCacheAgentCoherent : kCacheDefault; }

// A constant that stays in a register: the compiler otherwise puts it into the instruction as a literal, which the
// three-operand forms (v_and_or_b32, v_bitop3_b32) do not take, and needs a third operation per pair of signs.
__device__ __forceinline__ uint32_t in_register(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}

// A kernel argument that is read once at the start instead of again, a scalar round trip each, where it is used.
template <typename T>
__device__ __forceinline__ T early(T v) {
    asm volatile("" : "+s"(v));
    return v;
}

// A term as one wavefront reads it: every address out of its range returns zeros, so that the loop has no branches.
template <bool SCALED>
struct TermView {
    __amdgpu_buffer_rsrc_t bits, in, s_col;
    uint32_t row_bytes, bits_end;     // bits_end: last byte offset from which 16 bytes of the rows of this workgroup can be read
    int K, in_pitch;                  // in_pitch in bytes
};
template <bool SCALED>
__device__ __forceinline__ TermView<SCALED> view_of(const RowsTerm& t, int row0, int rows_here, int nb) {
    TermView<SCALED> v;
    v.row_bytes = (uint32_t)t.words * 4u;
    const uint32_t bytes = (uint32_t)rows_here * v.row_bytes;
    v.bits = raw_buffer(t.bits + (size_t)row0 * t.words, bytes);
    v.bits_end = bytes - 16u;
    v.K = t.K;
    v.in_pitch = t.in_stride * 2;
    v.in = raw_buffer(t.in, (uint32_t)(nb - 1) * (uint32_t)v.in_pitch + (uint32_t)t.K * 2u);
    v.s_col = raw_buffer(SCALED ? t.s_col : t.in, SCALED ? (uint32_t)t.K * 2u : 0u);
    return v;
}

// Rows of words whose number is not a multiple of 4: the last unit of a row reaches into the next row (its signs meet
// inputs that are zero), and the last one of the matrix would reach past its end.  That lane reads the last 16 bytes
// instead and moves the words down when it uses them.
template <bool SCALED>
__device__ __forceinline__ uint32_t words_offset(const TermView<SCALED>& v, int lane, int chunk, int f) {
    return (uint32_t)((lane & 15) + 16 * f) * v.row_bytes + (uint32_t)(4 * chunk + (lane >> 4)) * 16u;
}
template <bool SCALED, bool VEC, int F>
__device__ __forceinline__ void load_words(u32x4_t (&w)[F], const TermView<SCALED>& v, bool ragged, int chunk, int lane) {
#pragma unroll
    for (int f = 0; f < F; ++f) {
        uint32_t off = words_offset(v, lane, chunk, f);
        if constexpr (VEC) {
            if (ragged) off = min(off, v.bits_end);
            w[f] = __builtin_amdgcn_raw_buffer_load_b128(v.bits, off, 0, kCacheDefault);
        } else {
#pragma unroll
            for (int k = 0; k < 4; ++k) w[f][k] = __builtin_amdgcn_raw_buffer_load_b32(v.bits, off + 4u * k, 0, kCacheDefault);
        }
    }
}
template <bool SCALED, int F>
__device__ __forceinline__ void settle_words(u32x4_t (&w)[F], const TermView<SCALED>& v, int chunk, int lane) {
#pragma unroll
    for (int f = 0; f < F; ++f) {
        const uint32_t off = words_offset(v, lane, chunk, f);
        const uint32_t past = off > v.bits_end ? off - v.bits_end : 0u;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (past > 4u * k) {
                w[f][0] = w[f][1];
                w[f][1] = w[f][2];
                w[f][2] = w[f][3];
            }
    }
}

// The 8 columns of this lane of every batch row (and of the column scale); zeros beyond K and beyond the last row.
template <bool SCALED, int NB, bool VEC, bool COHERENT>
__device__ __forceinline__ void load_inputs(u32x4_t (&x)[NB], u32x4_t& s, const TermView<SCALED>& v, int chunk, int lane) {
    const int col = chunk * kChunkCols + 8 * lane;
    if constexpr (VEC) {
        const uint32_t off = col < v.K ? (uint32_t)col * 2u : kPastEnd;
        if constexpr (SCALED) s = __builtin_amdgcn_raw_buffer_load_b128(v.s_col, off, 0, kCacheDefault);
#pragma unroll
        for (int b = 0; b < NB; ++b) x[b] = __builtin_amdgcn_raw_buffer_load_b128(v.in, off + (uint32_t)b * v.in_pitch, 0, rows_cache<COHERENT>());
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const uint32_t o0 = col + 2 * k < v.K ? (uint32_t)(col + 2 * k) * 2u : kPastEnd;
            const uint32_t o1 = col + 2 * k + 1 < v.K ? (uint32_t)(col + 2 * k + 1) * 2u : kPastEnd;
            auto pair = [&](__amdgpu_buffer_rsrc_t r, uint32_t at, auto cache) {
                return (uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, o0 + at, 0, decltype(cache)::value) |
                       ((uint32_t)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, o1 + at, 0, decltype(cache)::value) << 16);
            };
            if constexpr (SCALED) s[k] = pair(v.s_col, 0u, std::integral_constant<int, kCacheDefault>{});
#pragma unroll
            for (int b = 0; b < NB; ++b) x[b][k] = pair(v.in, (uint32_t)b * v.in_pitch, std::integral_constant<int, rows_cache<COHERENT>()>{});
        }
    }
}

template <int DT>
struct RowsArith;
template <>
struct RowsArith<0> {
    static __device__ __forceinline__ uint32_t mul_pair(uint32_t x, uint32_t s) {
        const half2_t v = __builtin_bit_cast(half2_t, x) * __builtin_bit_cast(half2_t, s);
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ float4_t mfma(u32x4_t a, u32x4_t b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0, 0, 0);
    }
};
template <>
struct RowsArith<1> {
    static __device__ __forceinline__ uint32_t mul_pair(uint32_t x, uint32_t s) {
        bf162_t v;
        v[0] = (__bf16)(as_float(x << 16) * as_float(s << 16));
        v[1] = (__bf16)(as_float(x & 0xFFFF0000u) * as_float(s & 0xFFFF0000u));
        return __builtin_bit_cast(uint32_t, v);
    }
    static __device__ __forceinline__ float4_t mfma(u32x4_t a, u32x4_t b, float4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf168_t, a), __builtin_bit_cast(bf168_t, b), c, 0, 0, 0);
    }
};

// Orders a wavefront's own LDS traffic across its lanes (no other wavefront touches its region).
__device__ __forceinline__ void wave_lds_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// bf16 with many rows: a product x * s_in takes seven lane operations per pair there (one in fp16), so from 5 rows on
// the column scale goes into the sign operand instead (+-s_in: the XOR that makes the sign costs the same as the OR that
// makes +-1, and the product is then exact inside the MFMA).
template <int DT, bool SCALED, int NB>
constexpr bool rows_scale_in_operand() { return SCALED && DT == 1 && NB > 4; }

template <int DT, bool SCALED, int NB, int F>
constexpr int rows_wave_lds() {
    const int stage = (NB + (rows_scale_in_operand<DT, SCALED, NB>() ? 1 : 0)) * kStagePitch, tiles = F * 1024;
    return stage > tiles ? stage : tiles;
}

// What a second-stage workgroup of a fused launch waits for before it reads its input: `counter` reaching `target`,
// at most `spin_limit` polls.
struct StageWait {
    const unsigned* counter;
    unsigned target, spin_limit;
    unsigned* status;
};

// FUSED: both stages of a linear run in one launch.  The first stage stores h with device-coherent stores (another
// workgroup of the same launch reads it), the second stage waits until every first-stage workgroup of its linear has
// arrived and reads h with device-coherent loads.
template <int DT, bool SCALED, int NB, int F, int NT, bool VEC, bool FUSED>
__device__ __forceinline__ void rows_body(const RowsProblem<NT>& p, int block, int nb, int launch_waves, const StageWait& wait) {
    using E = Elem<DT>;
    constexpr bool kInOperand = rows_scale_in_operand<DT, SCALED, NB>();
    constexpr int kWaveLds = rows_wave_lds<DT, SCALED, NB, F>();
    extern __shared__ __align__(16) char rows_lds[];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    char* mine = rows_lds + wave * kWaveLds;
    const int row0 = block * 16 * F;
    const int c = lane & 15, g = lane >> 4;
    const int read_off = (c < nb ? c : nb - 1) * kStagePitch + 256 * g;   // batch columns beyond the last repeat it; never stored

    float4_t acc[F], tot[F];
#pragma unroll
    for (int f = 0; f < F; ++f) acc[f] = tot[f] = (float4_t){0.f, 0.f, 0.f, 0.f};

    if constexpr (FUSED && !SCALED) {
        if (threadIdx.x == 0) {
            unsigned spins = 0;
            while (__hip_atomic_load(wait.counter, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < wait.target) {
                __builtin_amdgcn_s_sleep(4);
                if (++spins >= wait.spin_limit) {            // bounded: report and go on (the outputs are then invalid)
                    atomicOr(wait.status, 1u);
                    break;
                }
            }
        }
        __syncthreads();
    }

    // What the epilogue needs is asked for up front (by the wavefronts that will run it), not one round trip at a time at
    // the end; rows past the last one read zeros.
    const int rows = early(p.rows), out_stride = early(p.out_stride), out_kind = early(p.out_kind), waves = early(launch_waves);
    char* const out_base = early((char*)p.out);
    const uint16_t* const s_row = early(p.t[0].s_row);
    const uint16_t* const bias = early(p.bias);
    const float* const addend = early(p.addend);
    const int row4 = row0 + 16 * wave + 4 * g;           // first of this lane's rows in the epilogue
    uint16_t row_scale[4] = {0, 0, 0, 0}, row_bias[4] = {0, 0, 0, 0};
    float row_add[4] = {0.f, 0.f, 0.f, 0.f};
    auto load_rows = [&](const uint16_t* q, int row, uint16_t (&to)[4]) {
        const __amdgpu_buffer_rsrc_t r = raw_buffer(q, q ? (uint32_t)rows * 2u : 0u);
#pragma unroll
        for (int k = 0; k < 4; ++k) to[k] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, (uint32_t)(row + k) * 2u, 0, kCacheDefault);
    };
    auto load_row_operands = [&]() {
        if (wave < F) {
            if (NT == 1) load_rows(s_row, row4, row_scale);
            if (bias) load_rows(bias, row4, row_bias);
            if (addend && c < nb)
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    if (row4 + k < rows) row_add[k] = addend[(size_t)c * out_stride + row4 + k];
        }
    };

    const uint32_t mask = in_register(kSignPair), one_pair = in_register(E::kOnePair);
    const int rows_here = min(rows - row0, 16 * F);
    // The terms one behind the other; a wavefront takes every p.waves-th chunk of all of them.  Chunks past the end
    // read zeros.
    int skip = wave;                                     // chunks of this term before the wavefront's next one
#pragma unroll
    for (int ti = 0; ti < NT; ++ti) {
        const RowsTerm t = p.t[ti];
        const TermView<SCALED> v = view_of<SCALED>(t, row0, rows_here, nb);
        const bool ragged = (t.words & 3) != 0;
        const int chunks = wave < p.waves ? t.chunks : 0;
        int chunk = skip;
        u32x4_t nw[F], nx[NB], ns;
        if (chunk < chunks) {
            load_words<SCALED, VEC, F>(nw, v, ragged, chunk, lane);
            load_inputs<SCALED, NB, VEC, FUSED && !SCALED>(nx, ns, v, chunk, lane);
        }
        uint16_t term_scale[F][4];
        if constexpr (NT > 1)
#pragma unroll
            for (int f = 0; f < F; ++f) load_rows(t.s_row, row0 + 16 * f + 4 * g, term_scale[f]);
        if (ti == 0) load_row_operands();
#pragma unroll 1
        for (; chunk < chunks; chunk += p.waves) {
            u32x4_t w[F];
#pragma unroll
            for (int f = 0; f < F; ++f) w[f] = nw[f];
            wave_lds_fence();
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                u32x4_t xv = nx[b];
                if constexpr (SCALED && !kInOperand)
#pragma unroll
                    for (int k = 0; k < 4; ++k) xv[k] = RowsArith<DT>::mul_pair(xv[k], ns[k]);
                *(u32x4_t*)(mine + b * kStagePitch + 16 * lane) = xv;
            }
            if constexpr (kInOperand) *(u32x4_t*)(mine + NB * kStagePitch + 16 * lane) = ns;
            if (VEC && ragged) settle_words<SCALED, F>(w, v, chunk, lane);
            wave_lds_fence();
            load_words<SCALED, VEC, F>(nw, v, ragged, chunk + p.waves, lane);
            load_inputs<SCALED, NB, VEC, FUSED && !SCALED>(nx, ns, v, chunk + p.waves, lane);
            // step q: 8 of the 128 columns of every lane group's unit
            auto read = [&](int q, u32x4_t& b, u32x4_t& one) __attribute__((always_inline)) {
                b = *(const u32x4_t*)(mine + read_off + 16 * q);
                one = (u32x4_t){one_pair, one_pair, one_pair, one_pair};
                if constexpr (kInOperand) one = *(const u32x4_t*)(mine + NB * kStagePitch + 256 * g + 16 * q);
            };
            auto step = [&](int q, const u32x4_t& b, const u32x4_t& one) __attribute__((always_inline)) {
#pragma unroll
                for (int f = 0; f < F; ++f) {
                    const uint32_t word = w[f][q >> 2];
                    u32x4_t a;
#pragma unroll
                    for (int k = 0; k < 4; ++k) a[k] = ((word << (4 * (q & 3) + k)) & mask) ^ one[k];
                    acc[f] = RowsArith<DT>::mfma(a, b, acc[f]);
                }
            };
            if constexpr (NB <= kReadAheadRows) {
                // the operands of the next two steps are read while two multiply
                u32x4_t b[2][2], one[2][2];
                read(0, b[0][0], one[0][0]);
                read(1, b[0][1], one[0][1]);
#pragma unroll
                for (int q = 0; q < 16; q += 2) {
                    const int now = (q >> 1) & 1;
                    if (q + 2 < 16) {
                        read(q + 2, b[now ^ 1][0], one[now ^ 1][0]);
                        read(q + 3, b[now ^ 1][1], one[now ^ 1][1]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    step(q, b[now][0], one[now][0]);
                    step(q + 1, b[now][1], one[now][1]);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int q = 0; q < 16; ++q) {
                    u32x4_t b, one;
                    read(q, b, one);
                    step(q, b, one);
                }
            }
        }
        skip = chunk - t.chunks;                         // >= 0: where the wavefront stands in the next term
        if constexpr (NT > 1) {                          // every term has a row scale of its own
#pragma unroll
            for (int f = 0; f < F; ++f)
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    tot[f][k] += acc[f][k] * E::to_float(term_scale[f][k]);
                    acc[f][k] = 0.f;
                }
        }
    }
    // Partial tiles of the wavefronts, added in the order of the wavefronts; wavefront f finishes tile f.
    wave_lds_fence();
#pragma unroll
    for (int f = 0; f < F; ++f) *(float4_t*)(mine + f * 1024 + 16 * lane) = NT > 1 ? tot[f] : acc[f];
    __syncthreads();
    if (wave >= F) return;
    float v[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int wv = 0; wv < kRowsMaxWaves; ++wv) {
        const float4_t part = *(const float4_t*)(rows_lds + min(wv, waves - 1) * kWaveLds + wave * 1024 + 16 * lane);
#pragma unroll
        for (int k = 0; k < 4; ++k) v[k] += wv < waves ? part[k] : 0.f;
    }
    if (c >= nb) return;
    const size_t o = (size_t)c * out_stride + row4;
    uint16_t r16[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        float t = v[k];
        if (NT == 1 && s_row) t *= E::to_float(row_scale[k]);
        t += E::to_float(row_bias[k]);
        if (addend) t += row_add[k];
        v[k] = row4 + k < rows ? t : 0.f;
        r16[k] = out_kind == kOutH ? E::from_float(v[k]) : E::from_float_clamped(v[k]);
    }
    if (out_kind == kOutF32) {
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (row4 + k < rows) ((float*)out_base)[o + k] = v[k];
        return;
    }
    uint16_t* out = (uint16_t*)out_base + o;
    const int end = out_kind == kOutH ? out_stride : rows;    // h is stored with its zero padding
    if ((out_stride & 3) == 0 && ((uintptr_t)out_base & 7) == 0 && row4 + 4 <= end) {
        const unsigned long long pk = (unsigned long long)((uint32_t)r16[0] | ((uint32_t)r16[1] << 16)) |
                                      ((unsigned long long)((uint32_t)r16[2] | ((uint32_t)r16[3] << 16)) << 32);
        if constexpr (FUSED && SCALED) __hip_atomic_store((unsigned long long*)out, pk, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *(unsigned long long*)out = pk;
    } else {
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (row4 + k < end) {
                if constexpr (FUSED && SCALED) __hip_atomic_store(out + k, r16[k], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                else out[k] = r16[k];
            }
    }
}

template <int N>
__device__ __forceinline__ int problem_of(const int (&first)[N + 1], int b) {
    int i = 0;
#pragma unroll
    for (int k = 1; k < N; ++k) i += b >= first[k] ? 1 : 0;
    return i;
}

template <int DT, bool SCALED, int NB, int F, int NT, bool VEC, int N>
__global__ __launch_bounds__(64 * kRowsMaxWaves) void gemv_rows_kernel(RowsGroup<NT, N> gr) {
    const int b = (int)blockIdx.x;
    int i = 0, first = 0;
#pragma unroll
    for (int k = 1; k < N; ++k)
        if (b >= gr.first[k]) {
            i = k;
            first = gr.first[k];
        }
    rows_body<DT, SCALED, NB, F, NT, VEC, false>(gr.p[i], b - first, gr.batch, gr.waves, StageWait{});
}

// Both stages of up to kGroupMax linears in ONE ordinary launch (no resident-grid requirement): the workgroups of all
// first stages come first in the grid, those of the second stages behind them (the hardware starts workgroups in the
// order of their ids, so every workgroup that is waited for is already running or done).
// Signalling, one slot of kFusedSlotWords words per launch, every counter and flag in a 128-byte line of its own:
// first-stage workgroups count their arrival per linear; the one that completes the count raises the linear's
// kFusedFlagLines ready flags, and a waiting workgroup polls one of them (1500 workgroups polling the arrival counter
// itself would queue every arrival behind their loads at one memory channel).  The last second-stage workgroup to
// finish puts the slot back to zero, so a slot serves launch after launch (and replay after replay of a captured
// launch) without being cleared from outside.
constexpr int kFusedFlagLines = 16;
constexpr int kFusedLineWords = 32;
constexpr int kFusedDoneLine = kGroupMax;                            // lines 0..7: arrivals per linear, 8: finished second stages
constexpr int kFusedFlagLine0 = 16;                                  // flag j of linear i: line 16 + i * kFusedFlagLines + j
constexpr int kFusedSlotLines = kFusedFlagLine0 + kGroupMax * kFusedFlagLines;
constexpr int kFusedSlotWords = kFusedSlotLines * kFusedLineWords;   // 18 KiB
struct FusedArgs {
    RowsGroup<1, kGroupMax> a, b;    // first and second stages; b.first counts from the end of the first stages
    unsigned* slot;                  // kFusedSlotWords words, zero between launches
    unsigned* status;
    unsigned spin_limit;
    int waves;                       // wavefronts of a workgroup, both stages
};

template <int DT, int NB, bool VEC>
__global__ __launch_bounds__(64 * kRowsMaxWaves) void gemv_fused_kernel(FusedArgs f) {
    const int b = (int)blockIdx.x;
    const int n1 = f.a.first[kGroupMax];
    if (b < n1) {
        const int i = problem_of<kGroupMax>(f.a.first, b);
        rows_body<DT, true, NB, 1, 1, VEC, true>(f.a.p[i], b - f.a.first[i], f.a.batch, f.waves, StageWait{});
        // every wavefront waits until its own stores of h have been acknowledged, the barrier collects all of them,
        // then the arrival is counted
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (threadIdx.x < kWave) {
            unsigned before = 0;
            if (threadIdx.x == 0)
                before = __hip_atomic_fetch_add(f.slot + i * kFusedLineWords, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            before = __builtin_amdgcn_readfirstlane(before);
            if (before + 1u == (unsigned)(f.a.first[i + 1] - f.a.first[i]) && threadIdx.x < kFusedFlagLines)
                __hip_atomic_store(f.slot + (kFusedFlagLine0 + i * kFusedFlagLines + (int)threadIdx.x) * kFusedLineWords, 1u,
                                   __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    } else {
        const int lb = b - n1;
        const int i = problem_of<kGroupMax>(f.b.first, lb);
        StageWait w;
        w.counter = f.slot + (kFusedFlagLine0 + i * kFusedFlagLines + (lb & (kFusedFlagLines - 1))) * kFusedLineWords;
        w.target = 1u;
        w.spin_limit = f.spin_limit;
        w.status = f.status;
        rows_body<DT, false, NB, 1, 1, VEC, true>(f.b.p[i], lb - f.b.first[i], f.b.batch, f.waves, w);
        __syncthreads();
        if (threadIdx.x < kWave) {
            unsigned before = 0;
            if (threadIdx.x == 0)
                before = __hip_atomic_fetch_add(f.slot + kFusedDoneLine * kFusedLineWords, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            before = __builtin_amdgcn_readfirstlane(before);
            if (before + 1u == (unsigned)f.b.first[kGroupMax]) {     // everybody is past its wait: clear the slot for the next launch
                for (int k = (int)threadIdx.x; k < kFusedSlotLines; k += kWave)
                    __hip_atomic_store(f.slot + k * kFusedLineWords, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

// ---- host side --------------------------------------------------------------------------------
static inline bool aligned16(const void* p) { return ((uintptr_t)p & 15u) == 0; }

int gemv_rows_group_max() { return kGroupMax; }

// Row pitch in elements of the 16-bit h of a linear: a multiple of 8 (16-byte loads) where the [batch, r] fp32 scratch
// that callers provide leaves room for it.
int gemv_rows_h_stride(int r) { return r >= 8 ? (r + 7) / 8 * 8 : r; }

static RowsTerm make_term(const RowsStage& s) {
    RowsTerm t;
    t.bits = s.bits;
    t.in = (const uint16_t*)s.in;
    t.s_col = (const uint16_t*)s.s_col;
    t.s_row = (const uint16_t*)s.s_row;
    t.words = s.words;
    t.K = s.K;
    t.in_stride = s.in_stride;
    t.chunks = (s.K + kChunkCols - 1) / kChunkCols;
    return t;
}

template <int NT>
static RowsProblem<NT> make_problem(const RowsStage* s) {
    RowsProblem<NT> p;
    int chunks = 0;
    p.out_kind = s[0].out_kind;
    for (int k = 0; k < NT; ++k) {
        p.t[k] = make_term(s[k]);
        chunks += p.t[k].chunks;
    }
    p.bias = (const uint16_t*)s[0].bias;
    p.addend = s[0].addend;
    p.out = s[0].out;
    p.rows = s[0].rows;
    p.out_stride = s[0].out_stride;
    // as many wavefronts as keep all of them equally long (the split decides the order of the sums, so it depends on
    // the linear alone and not on what shares the launch)
    const int most = s[0].rows >= kFewWavesFrom ? 4 : kRowsMaxWaves;
    const int rounds = (chunks + most - 1) / most;
    p.waves = rounds > 0 ? (chunks + rounds - 1) / rounds : 1;
    return p;
}

// Fills a group; returns the grid, or 0 when there is nothing to do.
template <int NT, int N>
static int make_group(RowsGroup<NT, N>& g, int count, const RowsStage* s, int batch, int F, int* waves) {
    int at = 0;
    *waves = F;                          // wavefront f finishes tile f
    for (int i = 0; i < N; ++i) {
        g.p[i] = make_problem<NT>(s + NT * (i < count ? i : count - 1));
        g.first[i] = at;
        if (i < count) {
            at += (g.p[i].rows + 16 * F - 1) / (16 * F);
            *waves = std::max(*waves, g.p[i].waves);
        }
    }
    g.first[N] = at;                     // as of every unused entry, so that no workgroup belongs to one
    g.batch = batch;
    g.waves = *waves;
    return at;
}

template <typename K, typename A>
static hipError_t launch_rows(K kern, const A& args, int grid, int waves, int wave_lds, PerDeviceFlag& raised, hipStream_t stream) {
    const size_t lds = (size_t)waves * wave_lds;
    const int dev = current_device();
    if (lds > 64 * 1024 && !raised.test(dev)) {
        hipError_t e = hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, kRowsMaxWaves * wave_lds);
        if (e != hipSuccess) return e;
        raised.set(dev);
    }
    hipLaunchKernelGGL(kern, dim3(grid), dim3(64 * waves), lds, stream, args);
    return hipGetLastError();
}

template <int DT, bool SCALED, int NB, int F, int NT, bool VEC, int N>
static hipError_t launch_table(int count, const RowsStage* s, int batch, hipStream_t stream) {
    RowsGroup<NT, N> g;
    int waves = 1;
    const int grid = make_group(g, count, s, batch, F, &waves);
    if (grid == 0) return hipSuccess;
    static PerDeviceFlag raised;
    return launch_rows(gemv_rows_kernel<DT, SCALED, NB, F, NT, VEC, N>, g, grid, waves, rows_wave_lds<DT, SCALED, NB, F>(), raised, stream);
}
template <int DT, bool SCALED, int NB, int F, int NT, bool VEC>
static hipError_t launch_group(int count, const RowsStage* s, int batch, hipStream_t stream) {
    if constexpr (VEC) {
        if (count == 1) return launch_table<DT, SCALED, NB, F, NT, VEC, 1>(count, s, batch, stream);
        if constexpr (NT == 1)
            if (count <= 3) return launch_table<DT, SCALED, NB, F, NT, VEC, 3>(count, s, batch, stream);
    }
    return launch_table<DT, SCALED, NB, F, NT, VEC, kGroupMax>(count, s, batch, stream);
}

// Whether 16-byte loads can read this stage: aligned input rows, and at least 16 bytes of words in the last row block.
static bool stage_vec(const RowsStage& s) {
    return ((s.rows - 1) % 16 + 1) * s.words >= 4 && aligned16(s.in) && s.in_stride % 8 == 0 && s.K % 8 == 0 && (!s.s_col || aligned16(s.s_col));
}

template <int DT, bool SCALED, int NT>
static hipError_t launch_any(int count, const RowsStage* s, int batch, hipStream_t stream) {
    int blocks = 0;
    bool vec = true;
    for (int i = 0; i < NT * count; ++i) {
        if (i % NT == 0) blocks += (s[i].rows + 15) / 16;
        vec = vec && stage_vec(s[i]);
    }
    if (!vec) {                                          // the same sums in the same order from 2-byte loads
        if (batch == 1) return launch_group<DT, SCALED, 1, 1, NT, false>(count, s, batch, stream);
        if (batch <= 4) return launch_group<DT, SCALED, 4, 1, NT, false>(count, s, batch, stream);
        return launch_group<DT, SCALED, 16, 1, NT, false>(count, s, batch, stream);
    }
    if (batch == 1) return launch_group<DT, SCALED, 1, 1, NT, true>(count, s, batch, stream);
    if (batch == 2) return launch_group<DT, SCALED, 2, 1, NT, true>(count, s, batch, stream);
    if (batch <= 4) return launch_group<DT, SCALED, 4, 1, NT, true>(count, s, batch, stream);
    const bool two = blocks >= kTwoBlocksFrom;
    if (batch <= 8)
        return two ? launch_group<DT, SCALED, 8, 2, NT, true>(count, s, batch, stream) : launch_group<DT, SCALED, 8, 1, NT, true>(count, s, batch, stream);
    return two ? launch_group<DT, SCALED, 16, 2, NT, true>(count, s, batch, stream) : launch_group<DT, SCALED, 16, 1, NT, true>(count, s, batch, stream);
}

template <bool SCALED, int NT>
static hipError_t launch_typed(int dtype, int count, const RowsStage* s, int batch, hipStream_t stream) {
    if (count < 1 || count > kGroupMax || batch < 1 || batch > 16) return hipErrorInvalidValue;
    return dtype == 0 ? launch_any<0, SCALED, NT>(count, s, batch, stream) : launch_any<1, SCALED, NT>(count, s, batch, stream);
}

hipError_t gemv_rows(int dtype, bool scaled, int count, const RowsStage* s, int batch, hipStream_t stream) {
    return scaled ? launch_typed<true, 1>(dtype, count, s, batch, stream) : launch_typed<false, 1>(dtype, count, s, batch, stream);
}

hipError_t gemv_rows_sum2(int dtype, const RowsStage* two, int batch, hipStream_t stream) {
    return launch_typed<false, 2>(dtype, 1, two, batch, stream);
}

// ---- fused launches ---------------------------------------------------------------------------
// The signalling slots live in a device array inside the library (zero when the module is loaded, put back to zero
// by every launch that used them): 256 slots of 18 KiB, dealt round robin to the calls.  Two calls collide on a slot
// only when they run at the same time on different streams AND are a multiple of 256 calls apart.
constexpr int kFusedSlots = 256;
static __device__ __align__(256) unsigned fused_counters[kFusedSlots * kFusedSlotWords];
static __device__ unsigned fused_status_word;
static std::atomic<unsigned> g_fused_ticket{0};
static unsigned* g_fused_counters_ptr[64];
static unsigned* g_fused_status_ptr[64];
static PerDeviceFlag g_fused_known;

static hipError_t fused_pointers(unsigned** counters, unsigned** status) {
    const int dev = current_device();
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    if (!g_fused_known.test(dev)) {
        unsigned *c = nullptr, *st = nullptr;
        hipError_t e = hipGetSymbolAddress((void**)&c, HIP_SYMBOL(fused_counters));
        if (e != hipSuccess) return e;
        e = hipGetSymbolAddress((void**)&st, HIP_SYMBOL(fused_status_word));
        if (e != hipSuccess) return e;
        g_fused_counters_ptr[dev] = c;
        g_fused_status_ptr[dev] = st;
        g_fused_known.set(dev);
    }
    *counters = g_fused_counters_ptr[dev];
    *status = g_fused_status_ptr[dev];
    return hipSuccess;
}

static std::atomic<unsigned> g_fused_spin_limit{0};
void gemv_fused_set_spin_limit(unsigned polls) { g_fused_spin_limit.store(polls); }

hipError_t gemv_fused_status(unsigned* out, hipStream_t stream) {
    unsigned *c = nullptr, *st = nullptr;
    hipError_t e = fused_pointers(&c, &st);
    if (e != hipSuccess) return e;
    e = hipMemcpyAsync(out, st, sizeof(unsigned), hipMemcpyDeviceToHost, stream);
    if (e != hipSuccess) return e;
    e = hipStreamSynchronize(stream);
    if (e == hipSuccess && *out != 0) {
        e = hipMemsetAsync(st, 0, sizeof(unsigned), stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
    }
    return e;
}

template <int DT, int NB, bool VEC>
static hipError_t launch_fused(const FusedArgs& f, int grid, int waves, hipStream_t stream) {
    static PerDeviceFlag raised;
    const int wave_lds = std::max(rows_wave_lds<DT, true, NB, 1>(), rows_wave_lds<DT, false, NB, 1>());
    return launch_rows(gemv_fused_kernel<DT, NB, VEC>, f, grid, waves, wave_lds, raised, stream);
}

template <int DT>
static hipError_t launch_fused_batch(const FusedArgs& f, bool vec, int grid, int waves, int batch, hipStream_t stream) {
    if (!vec) return batch <= 4 ? launch_fused<DT, 4, false>(f, grid, waves, stream) : launch_fused<DT, 16, false>(f, grid, waves, stream);
    return batch <= 4 ? launch_fused<DT, 4, true>(f, grid, waves, stream) : launch_fused<DT, 16, true>(f, grid, waves, stream);
}

hipError_t gemv_rows_fused(int dtype, int count, const RowsStage* first, const RowsStage* second, int batch, hipStream_t stream) {
    if (count < 1 || count > kGroupMax || batch < 1 || batch > 16) return hipErrorInvalidValue;
    FusedArgs f;
    int wa = 1, wb = 1;
    const int na = make_group(f.a, count, first, batch, 1, &wa);
    const int nb = make_group(f.b, count, second, batch, 1, &wb);
    if (nb == 0) return hipSuccess;
    for (int i = 0; i < count; ++i)
        if (first[i].rows == 0) return hipErrorInvalidValue;         // nobody would raise its flag: callers use two launches
    bool vec = true;
    for (int i = 0; i < count; ++i) vec = vec && stage_vec(first[i]) && stage_vec(second[i]);
    unsigned *counters = nullptr, *status = nullptr;
    hipError_t e = fused_pointers(&counters, &status);
    if (e != hipSuccess) return e;
    f.slot = counters + (size_t)(g_fused_ticket.fetch_add(1u) % kFusedSlots) * kFusedSlotWords;
    f.status = status;
    const unsigned spin = g_fused_spin_limit.load();
    f.spin_limit = spin ? spin : (1u << 20);
    const int waves = std::max(wa, wb);
    f.waves = waves;
    return dtype == 0 ? launch_fused_batch<0>(f, vec, na + nb, waves, batch, stream) : launch_fused_batch<1>(f, vec, na + nb, waves, batch, stream);
}

}  // namespace nq
