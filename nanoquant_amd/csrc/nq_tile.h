// One output tile of the prefill GEMMs: 16-bit activations x one-bit weights on the MFMA units, operands through an LDS ring.
//
//   C[t, j] = s_out[j] * sum_k (x[t, k] * s_in[k]) * sgn(W[j, k])
//
// The weight matrix is stored in 1 KiB tiles of 32 rows x 256 k (packing.py: pack_gemm_tiles): 16 bytes per lane, of which the 8 k
// values of a v_mfma_f32_32x32x16 step are one byte, and `((word << s) & 0x80008000) | (1.0, 1.0)` turns two of those bits into a
// +-1 pair.  With an input scale the operand is +-s_in[k] (the scale pair XOR the sign bits), so x * s_in is formed exactly inside
// the MFMA.  The weights are the A operand, the activations the B operand: a lane's results are then four consecutive rows of one
// token at a time.
//
// What bounds it: up to some hundred tokens a launch is a few microseconds of matrix time, and the time goes into the chain of loads
// of a workgroup; from 2048 tokens on the card lowers its clock to what the matrix units and the traffic into LDS draw (1.7 to 2.1
// GHz; 1.25 PFLOP/s).  Hence:
//  * A slab is 64 k of 32 TT tokens.  The slabs of a wavefront group go through a ring of NB slots; buffer loads with the LDS bit
//    fill it NB slabs ahead without passing through registers, and signs and scales of the next 256 k take the same way.  The
//    wavefronts count by themselves what is outstanding and never drain the counter inside the loop (staged through registers,
//    a slab of 256 k at a time: 4096 -> 3072 rows on 128 tokens 11.5 us, 11008 -> 3072 24.6; now 8.1 and 16.2).
//  * Operands of a step are read from LDS, and built from the signs, while the step before it multiplies; the only wait of a slab
//    sits in front of its last step, so that a workgroup that has its compute unit to itself keeps the matrix units busy too
//    (4096 -> 2048 rows on 2048 tokens, one workgroup of four wavefronts per unit: 42 -> 33.5 us).
//  * WK groups of WR wavefronts split the k tiles among them (group g takes g, g + WK, ...) and add their sums through LDS at the
//    end; the WR wavefronts of a group share its slabs and meet at one barrier per slab.  WR = 1: no barriers.
#pragma once
#include "nq_common.h"
#include "nq_mfma.h"

namespace nq {

struct GemmArgs {
    const void* x;          // [T, K] 16-bit
    const uint4* tiles;     // [R/32][K/256][64 lanes] 16 bytes each
    const uint16_t* s_in;   // [K] or null
    const uint16_t* s_out;  // [R] or null
    const uint16_t* bias;   // [R] added after the output scale, or null
    void* y;                // [T, R] 16-bit
    int T, K, R;
    int gx;                 // row blocks
};

constexpr int kSlabK = 64;                   // k of one slab
constexpr uint32_t kPastOperand = 0x80000000u;   // added to an offset: past the end of any operand (host: K <= kGemmMaxK)
constexpr int kGemmMaxK = 1 << 22;           // 128 tokens and 64 row tiles within 2^31 bytes
constexpr int kGemmEndK = 1 << 30;           // the signs of 32 rows within 2^32 bytes: fewer, of one token at a time

template <int TT, int RT, int WR, int WK, int NB>
struct TileShape {
    static constexpr int kWaves = WR * WK, kThreads = 64 * kWaves;
    static constexpr int kTok = 32 * TT, kRows = 32 * RT * WR;
    static constexpr uint32_t kSlabBytes = kTok * kSlabK * 2;
    static constexpr uint32_t kScaleAt = NB * kSlabBytes;                 // two tiles' input scales, 512 bytes each
    static constexpr uint32_t kSignAt = kScaleAt + 1024;                  // per wavefront RT KiB of signs
    static constexpr uint32_t kGroupBytes = kSignAt + WR * RT * 1024;
    static constexpr size_t kStage = (size_t)kWaves * 32 * (32 * RT + 8) * 2;
    static constexpr size_t kSum = WK > 1 ? (size_t)kWaves * RT * TT * 1024 * 4 : 0;
    static constexpr size_t kRing = (size_t)WK * kGroupBytes;
    static constexpr size_t kLds = kRing > kStage ? (kRing > kSum ? kRing : kSum) : (kStage > kSum ? kStage : kSum);
};

// 64 lanes x 16 bytes to LDS byte offset `lds` + 16 lane.  The same load as a builtin makes the compiler drain the counter of
// outstanding loads at the head of a loop, whatever has been waited for.  (It has no result register, so nothing is in flight
// towards one.)
__device__ __forceinline__ void load_to_lds(u32x4_t rsrc, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds" ::"s"(lds), "v"(voff), "s"(rsrc) : "memory", "m0");
}
template <int N, bool BARRIER>
__device__ __forceinline__ void wait_vm_lds() {
    if constexpr (BARRIER) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}

__device__ __forceinline__ uint32_t uniform(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ u32x4_t raw_rsrc(const void* p, uint32_t bytes) {
    const uint64_t a = (uint64_t)(uintptr_t)p;
    return (u32x4_t){uniform((uint32_t)a), uniform((uint32_t)(a >> 32) & 0xFFFFu), uniform(bytes), 0x00020000u};
}

template <int DT, bool SCALED, int TT, int RT, int WR, int WK, int NB>
struct Tile {
    using S = TileShape<TT, RT, WR, WK, NB>;
    using E = Elem<DT>;
    static constexpr int kLoads = 4 * TT / WR;          // slab loads of a wavefront
    static_assert(4 * TT % WR == 0, "");
    static constexpr int kTileLoads = RT + (SCALED ? 1 : 0);

    struct Fetch {
        u32x4_t x, w, s;
        uint32_t voff;                       // lane's byte offset of pass 0, k 0
        uint32_t pass_bytes;                 // 8 WR tokens
        uint32_t woff, wpitch, soff;
        uint32_t ring, scales, signs;        // LDS byte offsets
        int wr;
    };
    // pass ps of a wavefront: tokens 8 (ps WR + wr) .. + 7; lane -> token + (lane >> 3), chunk position lane & 7
    static __device__ __forceinline__ void fill(const Fetch& f, uint32_t slot, uint32_t kbytes) {
#pragma unroll
        for (int ps = 0; ps < kLoads; ++ps) {
            // 8 WR tokens further the permutation of the chunks differs in bit 2 where that is an odd multiple of 8
            const uint32_t v = (ps * WR) & 1 ? f.voff ^ 64u : f.voff;
            load_to_lds(f.x, v + (kbytes + (uint32_t)ps * f.pass_bytes), f.ring + slot + (uint32_t)(ps * WR + f.wr) * 1024u);
        }
    }
    static __device__ __forceinline__ void load_tile(const Fetch& f, uint32_t tile, bool live, int parity) {
#pragma unroll
        for (int r = 0; r < RT; ++r) load_to_lds(f.w, f.woff + ((uint32_t)r * f.wpitch + (live ? tile * 1024u : kPastOperand)), f.signs + (uint32_t)r * 1024u);
        if constexpr (SCALED) {
            if ((threadIdx.x & 63) < 32) load_to_lds(f.s, f.soff + (live ? tile * 512u : kPastOperand), f.scales + (uint32_t)parity * 512u);
        }
    }
    // what may be outstanding when slab SI + 1 is about to be read: it was filled in slab SI + 1 - NB, and the fills of the slabs
    // SI + 2 - NB .. SI - 1 are younger (this slab's own comes behind the wait), and so is what slab 0 of a tile loads in
    // front of its fill
    static constexpr int younger(int SI) {
        int n = (NB - 2) * kLoads;
        for (int d = SI + 2 - NB; d <= SI - 1; ++d)
            if (((d % 4) + 4) % 4 == 0) n += kTileLoads;
        return n;
    }
    static_assert(younger(3) <= 2 * kLoads, "the next tile's signs must have landed by slab 3");
    static __device__ __forceinline__ uint4 operand(uint32_t word, int t, const uint4& sp, uint32_t one) {
        const int s = 4 * t;
        uint4 a;
        if constexpr (SCALED) {
            a.x = sp.x ^ ((word << (s + 0)) & kSignPair);
            a.y = sp.y ^ ((word << (s + 1)) & kSignPair);
            a.z = sp.z ^ ((word << (s + 2)) & kSignPair);
            a.w = sp.w ^ ((word << (s + 3)) & kSignPair);
        } else {
            a.x = ((word << (s + 0)) & kSignPair) | one;
            a.y = ((word << (s + 1)) & kSignPair) | one;
            a.z = ((word << (s + 2)) & kSignPair) | one;
            a.w = ((word << (s + 3)) & kSignPair) | one;
        }
        return a;
    }
    struct State {
        float16_t acc[RT][TT];
        uint4 a[RT], b[TT], sp;       // operands of the coming step; scales of the step after that
        u32x4_t w[RT];
        uint32_t slot;                // of the current slab
    };
    static __device__ __forceinline__ void read_b(const char* p, int t, int lane, uint4 (&to)[TT]) {
#pragma unroll
        for (int tt = 0; tt < TT; ++tt) to[tt] = *(const uint4*)(p + (32 * tt + (lane & 31)) * (2 * kSlabK) + (((2 * t + (lane >> 5)) ^ ((lane >> 1) & 7)) << 4));
    }
    static __device__ __forceinline__ void read_signs(const char* group, int wr, int lane, u32x4_t (&to)[RT]) {
#pragma unroll
        for (int r = 0; r < RT; ++r) to[r] = *(const u32x4_t*)(group + S::kSignAt + (wr * RT + r) * 1024 + lane * 16);
    }
    template <int SI>
    static __device__ __forceinline__ void slab(State& q, const Fetch& f, const char* group, uint32_t fill_k, bool fill_live, uint32_t tile_next, bool tile_live,
                                                int parity, uint32_t one, int lane) {
        const int hi = lane >> 5;
        const char* now = group + q.slot;
        const uint32_t nslot = q.slot + S::kSlabBytes == NB * S::kSlabBytes ? 0u : q.slot + S::kSlabBytes;
        const char* sc_now = group + S::kScaleAt + parity * 512 + 128 * SI + 16 * hi;
        const char* sc_nxt = SI < 3 ? sc_now + 128 : group + S::kScaleAt + (parity ^ 1) * 512 + 16 * hi;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            uint4 bn[TT], spn = make_uint4(0, 0, 0, 0), sp2 = spn;
            u32x4_t w2[RT];
            if (t < 3) {
                read_b(now, t + 1, lane, bn);
                if constexpr (SCALED) {
                    if (t < 2) spn = *(const uint4*)(sc_now + 32 * (t + 2));
                    else if (SI < 3) spn = *(const uint4*)(sc_nxt);
                }
            } else {
                wait_vm_lds<younger(SI), (WR > 1)>();
                read_b(group + nslot, 0, lane, bn);
                if constexpr (SI == 3) read_signs(group, f.wr, lane, w2);
                if constexpr (SCALED) {
                    if (SI == 3) sp2 = *(const uint4*)(sc_nxt);
                    spn = *(const uint4*)(sc_nxt + 32);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (t == 3) {
                if constexpr (SI == 0) load_tile(f, tile_next, tile_live, parity ^ 1);
                fill(f, q.slot, fill_live ? fill_k : kPastOperand);
            }
            uint4 an[RT];
#pragma unroll
            for (int r = 0; r < RT; ++r) {
#pragma unroll
                for (int tt = 0; tt < TT; ++tt) q.acc[r][tt] = Mfma<DT>::run(q.a[r], q.b[tt], q.acc[r][tt]);
                if (t < 3) an[r] = operand(q.w[r][SI], t + 1, q.sp, one);
                else if (SI < 3) an[r] = operand(q.w[r][(SI + 1) & 3], 0, q.sp, one);
            }
            // (keeps the products of this step in front of the next one's reads)
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int tt = 0; tt < TT; ++tt) asm volatile("" : "+v"(q.acc[r][tt]));
            if (t == 3 && SI == 3) {
#pragma unroll
                for (int r = 0; r < RT; ++r) { q.w[r] = w2[r]; an[r] = operand(q.w[r][0], 0, sp2, one); }
            }
#pragma unroll
            for (int r = 0; r < RT; ++r) q.a[r] = an[r];
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) q.b[tt] = bn[tt];
            if constexpr (SCALED) q.sp = spn;
        }
        q.slot = nslot;
    }

    static __device__ __forceinline__ uint2 finish4(const float4_t& s, uint2 so, uint2 bs) {
        auto one = [](float v, uint32_t sc, uint32_t b) { return (uint32_t)E::from_float_sat(v * E::to_float((uint16_t)sc) + E::to_float((uint16_t)b)); };
        return make_uint2(one(s[0], so.x, bs.x) | (one(s[1], so.x >> 16, bs.x >> 16) << 16), one(s[2], so.y, bs.y) | (one(s[3], so.y >> 16, bs.y >> 16) << 16));
    }

    // Where a wavefront stands.
    struct Place {
        int lane, hi, wave, wr, wk, tok0, row0;
    };
    static __device__ __forceinline__ Place place(int bx, int by) {
        Place c;
        c.lane = threadIdx.x & 63;
        c.hi = c.lane >> 5;
        c.wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
        c.wr = c.wave % WR;
        c.wk = c.wave / WR;
        c.tok0 = by * S::kTok;
        c.row0 = (bx * WR + c.wr) * RT * 32;
        return c;
    }

    // q.acc = this wavefront's sums over its k tiles.  On return nothing is outstanding; other wavefronts may still be reading
    // their last slab.
    static __device__ __forceinline__ void walk(const GemmArgs& a, const Place& c, uint16_t* lds, State& q) {
        const int lane = c.lane, wr = c.wr, wk = c.wk;
        const char* group = (const char*)lds + wk * S::kGroupBytes;
        Fetch f;
        // both buffers begin with what is this tile's, so that the offsets stay small whatever the matrices' sizes; tokens and
        // rows past the end read zeros
        const int ktiles = a.K / kTileK;
        f.x = raw_rsrc((const uint16_t*)a.x + (size_t)c.tok0 * a.K, (uint32_t)min(a.T - c.tok0, S::kTok) * (uint32_t)a.K * 2u);
        f.w = raw_rsrc(a.tiles + (size_t)(c.row0 / 32) * ktiles * 64, (uint32_t)max(0, min(a.R - c.row0, 32 * RT)) * (uint32_t)a.K / 8u);
        f.s = raw_rsrc(SCALED ? (const void*)a.s_in : a.x, (uint32_t)a.K * 2u);
        f.wr = wr;
        f.soff = (uint32_t)lane * 16u;
        f.ring = uniform((uint32_t)(uintptr_t)(__attribute__((address_space(3))) const char*)group);
        f.scales = f.ring + S::kScaleAt;
        f.signs = f.ring + S::kSignAt + (uint32_t)(wr * RT) * 1024u;
        const int tk = 8 * wr + (lane >> 3);
        f.voff = (uint32_t)tk * (uint32_t)a.K * 2u + (uint32_t)(((lane & 7) ^ ((tk >> 1) & 7)) * 16);
        f.pass_bytes = (uint32_t)(8 * WR) * (uint32_t)a.K * 2u;
        f.woff = (uint32_t)lane * 16u;
        f.wpitch = (uint32_t)ktiles * 1024u;
        // k tiles of this group: wk, wk + WK, ...
        const int mine = (ktiles - wk + WK - 1) / WK;      // may be 0
        const int slabs = 4 * mine;
        // waves that meet at barriers walk equally many tiles (those past the end are zeros)
        const int count = WR > 1 ? (ktiles + WK - 1) / WK : mine;
        auto slab_k = [&](int j) { return (uint32_t)(wk + (j >> 2) * WK) * 512u + (uint32_t)(j & 3) * 128u; };
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int v = 0; v < 16; ++v) q.acc[r][tt][v] = 0.f;
        uint32_t one = E::kOnePair;
        asm volatile("" : "+v"(one));
        if (count > 0) {
            load_tile(f, (uint32_t)wk, mine > 0, 0);
#pragma unroll
            for (int j = 0; j < NB; ++j) fill(f, (uint32_t)j * S::kSlabBytes, j < slabs ? slab_k(j) : kPastOperand);
            wait_vm_lds<(NB - 1) * kLoads, (WR > 1)>();
            q.slot = 0;
            read_b(group, 0, lane, q.b);
            read_signs(group, wr, lane, q.w);
            uint4 sp0 = make_uint4(0, 0, 0, 0);
            q.sp = sp0;
            if constexpr (SCALED) {
                sp0 = *(const uint4*)(group + S::kScaleAt + 16 * c.hi);
                q.sp = *(const uint4*)(group + S::kScaleAt + 16 * c.hi + 32);
            }
#pragma unroll
            for (int r = 0; r < RT; ++r) q.a[r] = operand(q.w[r][0], 0, sp0, one);
#pragma unroll 1
            for (int i = 0; i < count; ++i) {
                const uint32_t tn = (uint32_t)(wk + (i + 1) * WK);
                const bool tl = i + 1 < mine;
                const int j = 4 * i, par = i & 1;
#define NQ_SLAB(SI) slab<SI>(q, f, group, slab_k(j + SI + NB), j + SI + NB < slabs, tn, tl, par, one, lane)
                NQ_SLAB(0);
                NQ_SLAB(1);
                NQ_SLAB(2);
                NQ_SLAB(3);
#undef NQ_SLAB
            }
        }
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    }

    // Four values of s_out or bias for rows row .. + 3; pad: two of the value where there are none.  s_out may begin at any element,
    // which the device reads in one load all the same.
    struct __attribute__((packed, aligned(2))) Four {
        uint2 v;
    };
    static __device__ __forceinline__ uint2 row_values(const GemmArgs& a, const uint16_t* p, int row, uint32_t pad) {
        return p && row < a.R ? ((const Four*)(p + row))->v : make_uint2(pad, pad);
    }
    // Piece p of a 32 x 32 tile: rows 8 p + 4 hi .. + 3 of token lane & 31.  With several k groups it is finished by group p % WK.
    static constexpr int kPieces = 4 / WK;
    struct RowScales {
        uint2 so[RT][kPieces], bs[RT][kPieces];
    };
    static __device__ __forceinline__ void load_rows(const GemmArgs& a, const Place& c, RowScales& s) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int pp = 0; pp < kPieces; ++pp) {
                const int row = c.row0 + 32 * r + 8 * (WK > 1 ? c.wk + WK * pp : pp) + 4 * c.hi;
                s.so[r][pp] = row_values(a, a.s_out, row, E::kOnePair);
                s.bs[r][pp] = row_values(a, a.bias, row, 0u);
            }
    }

    // Scales, rounds and stores the sums (all wavefronts are past their last slab).
    static __device__ __forceinline__ void store(const GemmArgs& a, const Place& c, uint16_t* lds, const float16_t (&acc)[RT][TT], const RowScales& rs) {
        const int lane = c.lane, hi = c.hi, wave = c.wave, wr = c.wr, wk = c.wk, tok0 = c.tok0, row0 = c.row0;
        if constexpr (WK > 1) {
            // [wave][r][tt][4 pieces][64 lanes] 16 bytes
            float* part = (float*)lds;
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                    for (int p = 0; p < 4; ++p)
                        *(float4_t*)(part + ((wave * RT + r) * TT + tt) * 1024 + p * 256 + 4 * lane) = (float4_t){acc[r][tt][4 * p], acc[r][tt][4 * p + 1], acc[r][tt][4 * p + 2], acc[r][tt][4 * p + 3]};
            __syncthreads();
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int pp = 0; pp < kPieces; ++pp) {
                    const int p = wk + WK * pp, row = row0 + 32 * r + 8 * p + 4 * hi;
#pragma unroll
                    for (int tt = 0; tt < TT; ++tt) {
                        float4_t g[WK];
#pragma unroll
                        for (int k = 0; k < WK; ++k) g[k] = *(const float4_t*)(part + (((k * WR + wr) * RT + r) * TT + tt) * 1024 + p * 256 + 4 * lane);
                        float4_t s = g[0] + g[1];
                        if constexpr (WK == 4) s += g[2] + g[3];
                        const int tok = tok0 + 32 * tt + (lane & 31);
                        if (row < a.R && tok < a.T) *(uint2*)((uint16_t*)a.y + (size_t)tok * a.R + row) = finish4(s, rs.so[r][pp], rs.bs[r][pp]);
                    }
                }
        } else {
            constexpr int kPitch = 32 * RT + 8;
            uint16_t* stage = lds + wave * 32 * kPitch;
            if (row0 >= a.R) return;
            auto fence = [] {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
            };
#pragma unroll
            for (int tt = 0; tt < TT; ++tt) {
#pragma unroll
                for (int r = 0; r < RT; ++r)
#pragma unroll
                    for (int p = 0; p < 4; ++p)
                        *(uint2*)(stage + (lane & 31) * kPitch + 32 * r + 8 * p + 4 * hi) =
                            finish4((float4_t){acc[r][tt][4 * p], acc[r][tt][4 * p + 1], acc[r][tt][4 * p + 2], acc[r][tt][4 * p + 3]}, rs.so[r][p], rs.bs[r][p]);
                fence();
                constexpr int kPer = 4 * RT, kTokPer = 64 / kPer;              // 16-byte chunks of a token, tokens of a store
#pragma unroll
                for (int n = 0; n < 32 / kTokPer; ++n) {
                    const int t = n * kTokPer + lane / kPer, c = lane % kPer;
                    const u32x4_t v = *(const u32x4_t*)(stage + t * kPitch + 8 * c);
                    const int tok = tok0 + 32 * tt + t, row = row0 + 8 * c;
                    if (tok < a.T && row < a.R) *(u32x4_t*)((uint16_t*)a.y + (size_t)tok * a.R + row) = v;
                }
                fence();
            }
        }
    }

    static __device__ __forceinline__ void run(const GemmArgs& a, int bx, int by, uint16_t* lds) {
        const Place c = place(bx, by);
        RowScales rs;
        if constexpr (WK > 1) load_rows(a, c, rs);       // asked for up front, not one round trip behind the last product
        State q;
        walk(a, c, lds, q);
        __syncthreads();
        if constexpr (WK == 1) load_rows(a, c, rs);
        store(a, c, lds, q.acc, rs);
    }

    // The sum of terms on the same rows and tokens: table[first], table[next[first]], ...; each is scaled by its own s_out in
    // 32 bits, and the sum is rounded once.  The terms' 16-bit results and the launches that add them are gone: of 169 us of the
    // seven two-term linears of a Qwen3-8B layer on 512 tokens 26 went there (now 147).  The registers hold the tile twice, which
    // the 128 x 256 tile has no room for.
    static __device__ __forceinline__ void run_sum(const GemmArgs* table, const int* next, int first, int bx, int by, uint16_t* lds) {
        const Place c = place(bx, by);
        float16_t tot[RT][TT];
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int tt = 0; tt < TT; ++tt)
#pragma unroll
                for (int v = 0; v < 16; ++v) tot[r][tt][v] = 0.f;
#pragma unroll 1
        for (int p = first; p >= 0; p = next[p]) {
            const GemmArgs a = table[p];
            State q;
            walk(a, c, lds, q);
            if constexpr (WR > 1) __syncthreads();       // before the next term's slabs
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int piece = 0; piece < 4; ++piece) {
                    const int row = c.row0 + 32 * r + 8 * piece + 4 * c.hi;
                    const uint2 so = row_values(a, a.s_out, row, E::kOnePair);
                    const uint2 bs = row_values(a, c.wk == 0 ? a.bias : nullptr, row, 0u);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t sw = e < 2 ? so.x : so.y, bw = e < 2 ? bs.x : bs.y;
                        const float scale = E::to_float((uint16_t)(sw >> (16 * (e & 1)))), bias = E::to_float((uint16_t)(bw >> (16 * (e & 1))));
#pragma unroll
                        for (int tt = 0; tt < TT; ++tt) tot[r][tt][4 * piece + e] += q.acc[r][tt][4 * piece + e] * scale + bias;
                    }
                }
        }
        __syncthreads();
        RowScales rs;
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int pp = 0; pp < kPieces; ++pp) {
                rs.so[r][pp] = make_uint2(E::kOnePair, E::kOnePair);
                rs.bs[r][pp] = make_uint2(0u, 0u);
            }
        store(table[first], c, lds, tot, rs);
    }
};

}  // namespace nq
