// Host-side launchers of the gfx950 affine-Q4 kernels (internal to libgemma4_qmm).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace q4 {

// The LoRA delta a GEMM epilogue adds to its outputs (kOutLora*): t = x . A^T as
// `slices` fp32 partial planes [slices][M][rank] (summed in slice order), B [N][rank]
// fp32, the adapter's scale; rank a multiple of 4, at most 32.
struct LoraEpilogue {
    const float* part;
    const float* b;
    int rank;
    int slices;
    float scale;
};

// Weight records: one per (16-row block, group pair), [row block][pair], 1152 bytes
// each: the 1 KiB tile of tiled words (uint4 per lane) and then the block's 16 scale/
// bias words for the pair (uint2 per row), so a kernel streaming a row block reads one
// contiguous run.  Kernels take the record array as uint4 tiles (record t's words at
// t * kRecU4 + lane) and as uint2 sb starting kRecSbBytes into it (record t's word for
// row r at t * kRecU2 + r).
constexpr int kRecBytes = 1152;
constexpr int kRecSbBytes = 1024;
constexpr int kRecU4 = kRecBytes / 16;
constexpr int kRecU2 = kRecBytes / 8;

// Bytes from the first of n consecutive records' scale/bias words to the end of the
// last record: the size of a buffer resource over their words (0 for none, so that
// every offset reads as zero).
__host__ __device__ inline uint32_t sb_span(int n) {
    return n > 0 ? (uint32_t)n * (uint32_t)kRecBytes - (uint32_t)kRecSbBytes : 0u;
}

constexpr size_t kMaxRecBytes = (size_t)1 << 31;  // a buffer resource's

struct Layout {
    int n = 0;   // output features
    int k = 0;   // input features of the tiled weight (2K for two-plane 8-bit handles)
    int kx = 0;  // row length of x: k, or K = k / 2 for two-plane handles, whose kernels
                 // read column c of x' = [x | x] as column c mod K of x
    int g = 0;   // groups per row (k / 64)
    int nb = 0;  // 16-row blocks
    int gp = 0;  // group pairs (ceil(g / 2))
    // the GEMM's fp16 form applies (set when the handle is built, from its scales: every
    // nonzero scale times 2^f16_p lies in [2^-14, 2^13))
    bool f16 = false;
    int f16_p = 0;
    // the GEMM may plan its pre-pass forms (fp16, one-pass 8-bit); cleared to pin the
    // bf16 form
    bool prepass_forms = true;
    size_t rec_bytes() const { return (size_t)nb * gp * kRecBytes; }
};

inline Layout make_layout(int n, int k) {
    Layout l;
    l.n = n;
    l.k = k;
    l.kx = k;
    l.g = k / 64;
    l.nb = (n + 15) / 16;
    l.gp = (l.g + 1) / 2;
    return l;
}

// A gate|up pair of F rows each is tiled as one projection of pair_layout(F, K):
// block j holds gate rows 8j..8j+7 then up rows 8j..8j+7 (its N is 16 * ceil(F / 8)).
inline Layout pair_layout(int f, int k) { return make_layout(16 * ((f + 7) / 8), k); }

// MLX layout (device) -> tiled layout (device).  pair_rows = 0: one projection
// (w, s, b); pair_rows = F: the gate (w, s, b) and up (w_up, s_up, b_up) pair.
hipError_t launch_repack(const uint32_t* w, const uint16_t* s, const uint16_t* b, const uint32_t* w_up,
                         const uint16_t* s_up, const uint16_t* b_up, uint4* tiles, uint2* sb, const Layout& l,
                         int pair_rows, hipStream_t stream);

// Tiled layout -> fp32 W[N,K] row-major, w = fma(s, q, b); a pair gives [2, F, K].
hipError_t launch_dequantize(const uint4* tiles, const uint2* sb, float* out, const Layout& l, int pair_rows,
                             hipStream_t stream);

// 8-bit affine weights as two 4-bit planes over K' = 2K (q4_layout.hip): the layout l
// of such a handle is make_layout(N, 2K) (pair_layout(F, 2K) for a pair) with kx = K;
// its kernels read x [M, K] as x' = [x | x] (column c of x' is column c mod K of x).
hipError_t launch_repack8(const uint32_t* w, const uint16_t* s, const uint16_t* b, const uint32_t* w_up,
                          const uint16_t* s_up, const uint16_t* b_up, uint4* tiles, uint2* sb, const Layout& l,
                          int pair_rows, hipStream_t stream);
hipError_t launch_dequantize8(const uint4* tiles, const uint2* sb, float* out, const Layout& l, int pair_rows,
                              hipStream_t stream);
hipError_t launch_embed8(const uint4* tiles, const uint2* sb, const int32_t* ids, int count, void* out, bool out_f32,
                         const Layout& l, hipStream_t stream);

// out[t, :] = dequantized row ids[t] of a projection (fp32, or bf16 rounded once), t <
// count; ids outside [0, N) give zero rows.  out is 16-byte aligned, [count, K].
hipError_t launch_embed(const uint4* tiles, const uint2* sb, const int32_t* ids, int count, void* out, bool out_f32,
                        const Layout& l, hipStream_t stream);

// Output modes (q4_common.h OutMode): 0 bf16 y, 1 fp32 y, 2 bf16 GeGLU h, 3 fp32 GeGLU h,
// 4 / 5 the greedy lm_head (softcap, optional logits, per-block best keys).  n_out is
// F for the GeGLU modes (h is [M, F]) and unused otherwise.
struct OutParams;

// Decode path, any M in one launch (16-row slabs along the grid's y dimension).
hipError_t launch_decode(const uint4* tiles, const uint2* sb, const uint16_t* x, const OutParams& op, int m,
                         const Layout& l, hipStream_t stream);

// Decode kernel family (a process-wide choice for tests and benchmarks): 0 automatic,
// 1 the int8-limb kernels wherever they apply (1-8 rows of x), 2 the bf16 kernels only.
// set_decode_variant returns the previous choice (an atomic exchange).
int set_decode_variant(int v);
int decode_variant();

// One row of x on the int8 matrix cores (q4_limbs.hip): x split exactly into three
// int8 limbs per group once per workgroup, every output mode.  limb_lds_bytes is its
// dynamic LDS; the launch fails (hipErrorInvalidValue) when that exceeds the CU's LDS.
size_t limb_lds_bytes(const Layout& l);
hipError_t launch_decode_limbs(const uint4* tiles, const uint16_t* x, const OutParams& op, const Layout& l,
                               hipStream_t stream);
// 2-8 rows of x on the int8 matrix cores (rows padded to 2, 4 or 8); the launch fails
// (hipErrorInvalidValue) where limb_rows_lds_bytes exceeds the CU's LDS.
size_t limb_rows_lds_bytes(const Layout& l, int m);
// whether the automatic choice takes them for m rows of this layout (measured per shape)
bool limb_rows_preferred(const Layout& l, int m);
hipError_t launch_decode_limb_rows(const uint4* tiles, const uint16_t* x, const OutParams& op, int m,
                                   const Layout& l, hipStream_t stream);

// token[m] (and value[m] when not null) = argmax over the keys part[m][0..nb) left by
// the greedy modes, for m < rows.
hipError_t launch_greedy_reduce(const unsigned long long* part, int nb, int rows, int32_t* token, float* value,
                                hipStream_t stream);

// The fp16 form's pre-pass keeps a row's group sums in LDS: rows of x of at most this
// many groups.
constexpr int kPrepMaxGroups = 8192;
// Scale range of a built handle (the GEMM's fp16 form): out[0] the largest and out[1]
// the smallest biased exponent of its nonzero scales (a subnormal scale counts as 0;
// out[0] stays -1 when every scale is zero), out[2] the count of inf or NaN scales.
// `out` is device memory the caller sets to {-1, 255, 0} first.
hipError_t launch_scale_range(const uint2* sb, const Layout& l, int* out, hipStream_t stream);
// Sets l.f16 and l.f16_p from those three numbers.
void set_f16_form(Layout& l, const int range[3]);

// Prefill path: fp32-exact factored GEMM on the matrix cores.  `workspace` holds,
// for the 256-row tile and the pre-pass forms (fp16 on 256-row tiles, one-pass 8-bit
// on 128- and 256-row tiles), the group sums of x (and in the pre-pass forms x as
// fp16 and each row's power of two) and, when K is split over workgroups, the fp32
// partial sums (device memory, 256-byte aligned); an unsplit bf16-form plan of 32- to
// 128-row tiles needs none.  The plan is the cheapest whose workspace fits in
// `max_workspace`; a call makes it once (0.8 to 1.5 us of host time) and hands it on.
struct GemmPlan {
    int bm = 256;            // output tile rows
    int bn = 256;            // output tile columns
    int splits = 1;          // workgroups along K per output tile
    int g_split = 0;         // groups per split (whole octets)
    size_t xaug_bytes = 0;   // group sums of x (256-row tiles)
    size_t part_bytes = 0;   // splits x M x N fp32 partial sums (0 when unsplit)
    bool f16 = false;        // fp16 form (256-row tiles of a handle whose scales allow it)
    bool kpair = false;      // q4_gemm_kpair.hip: tiles of 32, 48, .. 112 rows x 256
    bool q8 = false;         // one-pass 8-bit (128-row tiles of a two-plane handle)
    size_t x16_bytes = 0;    // fp16 and one-pass 8-bit forms: x scaled per row, as fp16 [M, kx]
    size_t rowexp_bytes = 0; // their rows' powers of two
    size_t total() const { return xaug_bytes + x16_bytes + rowexp_bytes + part_bytes; }
};
constexpr int kMaxSplits = 16;
constexpr size_t kMaxPartialBytes = (size_t)1 << 30;
GemmPlan plan_gemm(int m, const Layout& l, size_t max_workspace = ~(size_t)0);

// Compute units of the current device (cached per device).
int device_cus();
// gelu_table: kGeluTable bf16 values (q4_common.h) from launch_gelu_table, staged in
// LDS by the bf16 GeGLU epilogue (out_mode 2); may be null for the other modes.
hipError_t launch_gemm(const uint4* tiles, const uint2* sb, const uint16_t* x, void* y, int m, int out_mode,
                       int n_out, const Layout& l, const GemmPlan& plan, void* workspace, size_t workspace_bytes,
                       const uint16_t* gelu_table, hipStream_t stream, const LoraEpilogue* lora = nullptr);
// One launch of a kpair plan (q4_gemm_kpair.hip): y in out_mode (a mode of the GEMM), or
// the partial planes of a split; lora only in the LoRA modes.
hipError_t launch_kpair(const uint4* tiles, const uint2* sb, const uint16_t* x, void* y, int m, int out_mode, int n_out,
                        const Layout& l, const GemmPlan& plan, long split_stride, const uint16_t* gelu_table,
                        const LoraEpilogue& lora, hipStream_t stream);
// Whether its 32-bit offsets reach everything: a tile's rows past x and row blocks past
// the records (offsets that read as zero must not wrap), and a tile's rows of y.
constexpr int kKpairMaxRows = 112;  // rows of the largest kpair tile
inline bool kpair_fits(int m, const Layout& l) {
    const size_t wrap = (size_t)1 << 32;
    return ((size_t)m + kKpairMaxRows) * l.kx * 2 < wrap && l.rec_bytes() + (size_t)16 * l.gp * kRecBytes < wrap &&
           l.rec_bytes() <= kMaxRecBytes && (size_t)kKpairMaxRows * l.n * 4 < kMaxRecBytes;
}
// Whether the plan's launch can add a LoRA delta of this rank in its epilogue.
inline bool gemm_lora_epilogue(const GemmPlan& plan, int rank) {
    return plan.splits == 1 && rank >= 4 && rank <= 32 && rank % 4 == 0;
}

// Fills table[kGeluTable] with gelu of the bf16 patterns that need a table, in the
// bf16 op sequence.
hipError_t launch_gelu_table(uint16_t* table, hipStream_t stream);

// LoRA delta added in place to a projection output y [m, n] (bf16 or fp32) already
// holding the base product: part is fp32 scratch of lora_slices(k, m) x m x rank floats
// (x . A^T summed over slices of K), a [rank, k] and b [n, rank] fp32 on the device
// (q4_lora.hip).
constexpr int kLoraSlices = 8;
int lora_slices(int k, int m);
// Small M and rank: one fused launch that needs no part scratch (part may be null).
bool lora_fused(int m, int rank);
// a_hi, a_lo: A as bf16 high and low parts [ceil(rank / 16) * 16][k] (rows past rank
// zero), for the matrix-core x . A^T.
hipError_t launch_lora(const uint16_t* x, const float* a, const uint16_t* a_hi, const uint16_t* a_lo, const float* b,
                       float* part, void* y, int m, int n, int k, int rank, float scale, bool out_f32,
                       hipStream_t stream);
// Only the first step, part[slice][m][r] = x . A^T over lora_slices(k, m) slices of K
// (for a GEMM whose epilogue adds the delta).
hipError_t launch_lora_down(const uint16_t* x, const uint16_t* a_hi, const uint16_t* a_lo, float* part, int m,
                            int k, int rank, hipStream_t stream);

// Forward path choice (automatic mode).
//
// Up to 31 rows, and beyond that while 16-row slabs x N x K' stays at most
// kScratchFreeSlabWork (K' = 2K for two-plane 8-bit handles), a plain forward takes no
// scratch: such calls may be captured on a stream the library has not seen, graphs of
// them captured on one stream may be replayed side by side, and they may overlap through
// the allocation-free entry point.  They run on the decode kernels, or on a GEMM plan that
// needs no scratch (K unsplit) where that is the faster of the two.
//
// The decode kernels cost one pass over the weights per slab; a GEMM with K unsplit costs
// some 2 us per 256 columns of K on up to 256 output tiles of 256 columns.  So N times the
// slabs decides.  Measured as whole forwards (graph replays over rotated weight copies,
// each path pinned), decode / unsplit GEMM in us:
//   4 bits, past 16 rows: below the line gate 15360x3840 at 17 rows 25.6 / 31.1, qkv
//     8192x3840 16.9 / 30.6, q 4096x3840 at 48 15.9 / 26.1; past it 24576x3840 at 17
//     33.9 / 31.9, the gate|up pair 43.2 / 33.4, 32768x2048 29.3 / 19.7, 65536x512 20.1 / 9.2,
//     16384x1024 at 33 14.6 / 10.3.
//   8 bits from 9 rows: 65536x3840 at 9 114 / 78; 65536x1024 even to 12 rows (22.9 / 23.7),
//     at 16 30.5 / 23.4; the pair at 9 57 / 61.
//   8 bits from 12 rows: below the line 24576x3840 at 16 57.1 / 59.4, down 3840x15360 38.8 /
//     211, qkv at 31 37.9 / 56.6; past it the pair at 12 64.7 / 60.9, at 31 135 / 61.5,
//     gate at 17 58.5 / 57.8, at 31 71.7 / 58.0.
// (A split of K would be faster on most of them: the pair at 17 rows 25.1 us, qkv 11.8, the
// 8-bit pair at 16 40.7.  Its partial sums are the scratch.)
//
// Past the scratch-free calls the GEMM's fixed cost is ~10 us: decode / GEMM o 3840x4096 at
// 48 rows 15.3 / 13.3, at 64 19.4 / 14.4; qkv at 32 19.7 / 11.1, at 48 28.1 / 12.8.
constexpr int kScratchFreeRows = 31;
constexpr double kScratchFreeSlabWork = 5.5e7;
constexpr long kScratchFreeMaxRows = 1024;
// While the slabs' work stays at most this, the decode kernels are taken without asking for
// the GEMM (o at 32 rows 11.5 / 11.4 with a split; k 2048x3840 at 64 11.0 / 11.8).
constexpr double kDecodeMaxSlabWork = 3.5e7;
// Slabs x N from which the unsplit GEMM is taken: 4 bits past 16 rows; 8 bits from 9 and
// from 12 rows.
constexpr double kUnsplitCols = 4.5e4;
constexpr int kTwoPlaneRows[2] = {9, 12};
constexpr double kTwoPlaneUnsplitCols[2] = {6.0e4, 3.0e4};

inline double slab_work(long rows, const Layout& l) {
    return (double)((rows + 15) / 16) * (double)l.n * (double)l.k;
}
inline bool scratch_free(long rows, const Layout& l) {
    return rows <= kScratchFreeRows || (rows <= kScratchFreeMaxRows && slab_work(rows, l) <= kScratchFreeSlabWork);
}
inline bool use_decode(long rows, const Layout& l, int gemm_min_rows) {
    if (gemm_min_rows > 0) return rows < gemm_min_rows;
    if (!scratch_free(rows, l)) return false;
    const bool two_plane = l.kx != l.k;
    if (rows < (two_plane ? kTwoPlaneRows[0] : 17) || slab_work(rows, l) <= kDecodeMaxSlabWork) return true;
    const double cols = (double)((rows + 15) / 16) * (double)l.n;
    return cols < (two_plane ? kTwoPlaneUnsplitCols[rows < kTwoPlaneRows[1] ? 0 : 1] : kUnsplitCols);
}
// Scratch the GEMM of such a call may plan with: none for the scratch-free calls (a pinned
// path plans freely).
inline size_t gemm_room(long rows, const Layout& l, int gemm_min_rows) {
    return gemm_min_rows == 0 && scratch_free(rows, l) ? 0 : ~(size_t)0;
}

}  // namespace q4
