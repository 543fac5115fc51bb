// Internal launch interface between the C-ABI layer (nq_api.hip) and the kernel files.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace nq {

// nq_rows.hip: one stage of the per-linear decode path on 1 to 16 batch rows.  dtype 0 = fp16, 1 = bf16.
struct RowsStage {
    const uint32_t* bits;   // [rows, words], row-major "half2" order
    const void* in;         // [batch, in_stride] 16-bit: activations, or the h of an earlier stage (K = in_stride then)
    const void* s_col;      // [K] column scale, or null
    const void* s_row;      // [rows] row scale, or null
    const void* bias;       // [rows] added after the row scale, or null
    const float* addend;    // [batch, out_stride] fp32 added before the store, or null
    void* out;              // [batch, out_stride]
    int rows, words, K, in_stride, out_stride;
    int out_kind;           // 0: 16-bit result (clamped), 1: fp32 result, 2: 16-bit h (with zeros up to out_stride rows)
};
int gemv_rows_group_max();
int gemv_rows_h_stride(int r);
// `count` (<= gemv_rows_group_max()) independent stages in one launch; scaled: all of them have s_col, or none.
hipError_t gemv_rows(int dtype, bool scaled, int count, const RowsStage* s, int batch, hipStream_t stream);
// out = the sum of two stages without column scale on the same rows (out, bias, addend from the first).
hipError_t gemv_rows_sum2(int dtype, const RowsStage* two, int batch, hipStream_t stream);
// Both stages of `count` linears in one launch whose second stages wait inside the kernel (first: out_kind 2).
hipError_t gemv_rows_fused(int dtype, int count, const RowsStage* first, const RowsStage* second, int batch, hipStream_t stream);
hipError_t gemv_fused_status(unsigned* out, hipStream_t stream);
void gemv_fused_set_spin_limit(unsigned polls);          // 0: the default

// nq_stream.hip: one launch over a table of stages (see the file header).
struct RunStage {
    const uint32_t* bits;   // [rows, words] packed signs, row-major "half2" order
    const void* in;         // [batch, in_stride]: 16-bit activations, or fp32 when in_f32
    const uint16_t* s_col;  // [K] per-column scale applied to a 16-bit input, may be null
    const uint16_t* s_row;  // [rows] per-row scale, may be null
    void* out;              // [batch, out_stride]: fp32 when out_f32, else 16-bit (clamped)
    const float* addend;    // fp32 [batch, out_stride] added before the store, may be null
    const uint16_t* bias;   // [rows] added after the row scale, may be null
    int rows, words, K, units;
    int in_stride, out_stride;
    int in_f32, out_f32;
    int dep, dep2;          // stage indices that must be complete before `in` / `addend` are read, or -1
    int signal;             // a later stage waits on this one
    int vec_bits, vec_in;
    int phase;              // dependency depth: a stage runs after every stage of a lower phase it depends on
    int seg_count;          // number of workgroup slices this stage is cut into (its completion count)
    int in_coherent;        // fp32 input written by another stage of the same launch
    int heavy_release;      // 16-bit output read by a later stage: full device-scope release on completion
    int heavy_acquire;      // 16-bit input written by an earlier stage: full device-scope acquire after the wait
    int tiled;              // `bits` is in the tile order of tile_words() instead of row-major
    int in_ext, out_ext;    // `in` / `out` are given with the launch instead (bound input / output of the list)
    int dep_segs, dep2_segs;  // seg_count of the stages `dep` / `dep2` (what a waiting slice compares the counter with)
    int addend_local;       // the rows of `addend` that a slice reads were written by the slice before it on the same
                            // workgroup (same rows of stage `dep2`): nothing to wait for
};
// One workgroup's share of one stage: rows [row_begin, row_end).
struct RunSegment {
    int stage, row_begin, row_end, pad_;
};
// What the kernel reads per slice, in one record: the slice and a copy of its stage (one dependent memory access
// between the kernel arguments and the first load of data instead of three).  Record w of the table is the first
// slice of workgroup w (stage -1: the workgroup has none); its further slices are the records [more_begin,
// more_end), in the order in which it works them off.
struct RunSlice {
    RunSegment seg;
    int more_begin, more_end;   // meaningful in the first record of a workgroup only
    RunStage st;
};
size_t stream_counter_bytes(int nstages);
// alt: the 16-bit arithmetic instead of the batch size's usual one, where stream_has_alt(dtype, batch);
// own: the fp4 x fp8 kernel whose wavefronts own row pairs, where it exists (tile order, batch 2 and 4, no reproducible
// sums, every input staged in one chunk; ignored otherwise);
// f6: batch 8 and 16, every stage in tile order: the fp4 x fp6 arithmetic (nq_fp6.h)
int stream_capacity(int dtype, int batch, int max_units, bool alt = false, int variant = -1);
int stream_chunk_cap(int dtype, int batch, int max_units, bool alt = false, bool f6 = false);
// workgroups of the fp4 x fp6 kernel that the device keeps resident
int stream_f6_capacity(int dtype, int batch, int max_units);
int stream_row_granule(int dtype, int batch);
hipError_t gemv_stream(int dtype, int batch, int nstages, const RunSlice* slices, unsigned long long* counters,
                       unsigned* status, int nwg, int max_units, hipStream_t stream, const void* ext_in = nullptr,
                       void* ext_out = nullptr, bool tiled = false, bool det = false, unsigned spin_limit = 0,
                       bool alt = false, bool own = false, bool f6 = false);
bool stream_needs_uniform_order(int dtype, int batch, bool alt = false);
bool stream_has_deterministic(int dtype, int batch);
bool stream_has_alt(int dtype, int batch);

// nq_gemm.hip: C[T,R] = s_out * ((x * s_in) . sgn(W)^T) with W in the 32x256 tile layout, up to gemm_group_max() GEMMs on the
// same token count in one launch (s_in: all or none).  use: which tiles may be taken (see choose_tile).
enum GemmUse {
    kGemmAlone,      // one linear by itself
    kGemmGroup,      // up to 160 tokens the bits that it gets by itself
    kGemmAnyTile,    // whatever is fastest
};
int gemm_group_max();
hipError_t gemm_onebit_group(int dtype, int count, const void* const* x, const uint32_t* const* tiles,
                             const void* const* s_in, const void* const* s_out, const void* const* bias, void* const* y,
                             int T, const int* K, const int* R, int use, hipStream_t stream);
// Sums of GEMMs without input scales in one launch (see nq_gemm.hip).
hipError_t gemm_onebit_sums(int dtype, int count, const int* next, const void* const* x, const uint32_t* const* tiles,
                            const void* const* s_out, const void* const* bias, void* const* y, int T, const int* K, const int* R,
                            hipStream_t stream);
double gemm_sums_time(int count, const int* next, int T, const int* K, const int* R);       // estimate of that launch, us; 1e30: not as sums
// The tiles that those launches are cut into: tokens << 16 | rows.
int gemm_tile_size(int use, int count, const void* const* x, int T, const int* K, const int* R, bool scaled);
int gemm_sums_tile_size(int count, const int* next, int T, const int* K, const int* R);
// Estimated time of gemm_onebit_group with kGemmAnyTile, in us.
double gemm_tiles_time(int count, const void* const* x, int T, const int* K, const int* R, bool scaled);

// nq_panel.hip: the same GEMMs up to 2048 tokens as one persistent launch over 64-token x 256-row panels
// (see the file header).  workspace: panel_workspace_bytes() bytes, zero when first used.
int compute_units();                 // of the current device; 0: none
size_t panel_workspace_bytes();
bool panel_addresses(int count, int T, const int* K, const int* R);                // small enough for the kernel
// Whether panels are the faster form (automatic choice); *time (or null): estimate of the faster one, in us.
bool panel_applies(int count, const void* const* x, int T, const int* K, const int* R, bool scaled, double* time);
hipError_t gemm_panel_group(int dtype, int count, const void* const* x, const uint32_t* const* tiles,
                            const void* const* s_in, const void* const* s_out, const void* const* bias, void* const* y,
                            int T, const int* K, const int* R, void* workspace, unsigned spin_limit, hipStream_t stream);

// nq_util.hip
hipError_t stream_copy(void* dst, const void* src, size_t bytes, hipStream_t stream);
hipError_t repack_words(const uint32_t* src, uint32_t* dst, size_t nwords, int src_order, int dst_order,
                        hipStream_t stream);
hipError_t words_to_tiles(const uint32_t* src, uint32_t* dst, int rows, int words, int rows_padded, int k_padded,
                          int src_order, hipStream_t stream);
size_t tiled_word_count(int rows, int words);
hipError_t tile_words(const uint32_t* src, uint32_t* dst, int rows, int words, int inverse, hipStream_t stream);

}  // namespace nq
