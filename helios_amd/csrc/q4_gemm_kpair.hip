// Prefill-shape affine-Q4 matmul on gfx950 for small and middling M: the bf16 form of
// q4_gemm.hip (y = sum_g 16 s_g P_g + (b_g - 16 s_g) X_g, every product exact in fp32)
// on output tiles of 16 kMT x 256, kMT = 2..7.
//
// Two sets of four waves share K: a step is four groups (two group pairs), set 0 takes
// the first pair, set 1 the second, and each wave owns 16 kMT rows x 64 columns.  The
// sets' sums meet in LDS once, after the last step.  Against eight waves side by side
// along N, each on every group (q4_gemm.hip), a wave's x fragment feeds four products
// instead of two (half the LDS reads), a barrier comes every four groups instead of
// every one, and with 64 columns a wave's words are its own: they go from memory to
// registers, loaded for the next step in place once this step's are expanded.  x goes
// through LDS by DMA, two slots of a step each.
//
// Bound: the matrix cores and what the two waves of a SIMD cannot hide under them.  A step
// of a 112-row tile takes 6.9 k cycles for 4.1 k of MFMA (a 64-row tile 4.5 k for 2.3 k);
// measured by leaving parts out: the loads' issue 1.1 k, X_g 0.65 k, the scale FMAs 0.6 k,
// the expansion and the LDS reads none; two waves whose products and other work alternate
// leave the matrix cores idle a third of the time, and 32x32x16 products, deeper operand
// prefetch, words two steps ahead or wave priorities did not change that (registers allow
// no third wave per SIMD).
// Measured as forwards (graph replays over rotated copies, us; q4_gemm.hip's best tile
// before / here): qkv 8192x3840 at 64 rows 16.2 / 12.9, at 200 31.0 / 27.2, at 517 64.9 /
// 43.2, at 1100 103.8 / 84.8; the gate|up pair at 96 46.4 / 36.2, at 200 70.2 / 58.7, at
// 1100 413 / 282; down 3840x15360 at 160 40.7 / 32.0, at 517 90.9 / 77.1; o 3840x4096 at
// 700 46.4 / 32.7 (with the bias term in two parts, see x_operand).
#include <type_traits>

#include "q4_common.h"
#include "q4_gemm_tile.h"
#include "q4_kernels.h"

namespace q4 {
namespace {

constexpr int kKpBN = 256;
constexpr int kKpRB = kKpBN / 16;  // row blocks per workgroup tile

// one pair's words of a wave's four row blocks, in registers
struct PairWords {
    uint4 t[4];
    uint2 s[4];
};

// The bias MFMA's operands for a step's four groups: lane (row or column, kq) holds group
// kq.  A = [Xh, Xm, Xl, 0, -16 Xh, -16 Xm, -16 Xl, 0] with X_g = Xh + Xm + Xl in three bf16
// parts (2^-26 relative), B = [b, b, b, 0, s, s, s, 0].  (b - 16 s) X_g is about 24 s X_g,
// and in two parts (2^-18, eight groups per MFMA) it is the largest error of the sum:
// fp32 outputs of the layer's projections are 1.8e-5 off 64 bits so, 0.5e-6 to 1.3e-6 off
// with three; two parts would be 1.5-4% faster.
__device__ __forceinline__ uint4 x_operand(float x) {
    const float h = round_bf16(x);
    const float m = round_bf16(x - h);
    const float l = round_bf16(x - h - m);
    const uint32_t hm = (uint32_t)f32_to_bf16(h) | ((uint32_t)f32_to_bf16(m) << 16);
    const uint32_t nhm = (uint32_t)f32_to_bf16(-16.0f * h) | ((uint32_t)f32_to_bf16(-16.0f * m) << 16);
    return make_uint4(hm, f32_to_bf16(l), nhm, f32_to_bf16(-16.0f * l));
}
__device__ __forceinline__ bf16x8 sb_operand(uint32_t w) {
    const uint32_t s = w & 0xFFFFu, b = w >> 16;
    return __builtin_bit_cast(bf16x8, make_uint4(b | (b << 16), b, s | (s << 16), s));
}

struct KpairArgs {
    const uint4* tiles;
    const uint2* sb;
    const uint16_t* x;
    void* y;
    const uint16_t* gelu_table;
    LoraEpilogue lora;
    int m_rows, n_rows, kx, groups, gpairs, mtiles, ntiles;
    uint32_t rec_bytes;
    int g_split;
    long split_stride;
    int n_out;
    int mode;
};

template <int kMT>
__global__ __launch_bounds__(512) void kpair_kernel(const KpairArgs a) {
    constexpr int BM = 16 * kMT;
    constexpr int kXT = (kMT + 3) / 4;  // row tiles whose X_g a wave sums
    constexpr int kHalf = 4 * kMT;      // 16x16 tiles of a wave: products of a group
    constexpr int kTiles = 2 * kHalf;   // of a step
    __shared__ uint4 g_x0[4 * BM * 8];  // four group tiles of x [group][row][8 chunks]
    __shared__ uint4 g_x1[4 * BM * 8];
    __shared__ uint4 g_xab[2 * kMT * 64];  // a step's bias A operands [step parity][m16][lane]
    int mt, nt;
    tile_of((int)blockIdx.x, (int)gridDim.x, a.mtiles, a.ntiles, mt, nt);
    const int g_begin = (int)blockIdx.y * (a.g_split & ~7);
    const int g_end = a.groups - g_begin < a.g_split ? a.groups : g_begin + a.g_split;
    const int p_end = (g_end + 1) >> 1;
    const int s_begin = g_begin >> 2, s_end = (g_end + 3) >> 2;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int set = wave >> 2, wn = wave & 3;
    const int lane = threadIdx.x & 63;
    const int col = lane & 15, kq = lane >> 4;
    const int rbw = nt * kKpRB + wn * 4;

    // Local row block j of a wave is block (j + 2 set) & 3 of its four: its own half of
    // the outputs is j = 0, 1 in both sets.  Offsets past the records (row blocks past N)
    // and past x (rows past M) lie outside their buffers and read as zeros.
    const uint32_t rb_bytes = (uint32_t)a.gpairs * kRecBytes;
    const uint32_t wv0 = (uint32_t)rbw * rb_bytes + (uint32_t)lane * 16u;
    const uint32_t ov = (uint32_t)(rbw + 2 * set) * rb_bytes + (uint32_t)(kq >> 1) * kRecBytes + (uint32_t)col * 8u + (uint32_t)(kq & 1) * 4u;
    const uint32_t x_bytes = (uint32_t)a.m_rows * (uint32_t)a.kx * 2u;
    const int gx = a.kx >> 6;  // group g >= gx (the low plane of a two-plane handle) reads group g - gx of x

    auto load_w = [&](int s, int j, PairWords& w) {
        const int p = 2 * s + set;
        const bool in = p < p_end;
        const uint32_t soff = (uint32_t)p * kRecBytes;
        uint32_t wv = wv0;
        asm volatile("" : "+v"(wv));  // (opaque: four row blocks' offsets held across the loop would cost registers)
        wv += (uint32_t)((j + 2 * set) & 3) * rb_bytes;
        w.t[j] = buffer_load16s(make_rsrc(a.tiles, in ? a.rec_bytes : 0u), wv, soff);
        const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(make_rsrc(a.sb, in ? a.rec_bytes - kRecSbBytes : 0u),
                                                             (int)(wv - (uint32_t)lane * 16u + (uint32_t)col * 8u), (int)soff, 0);
        w.s[j] = make_uint2(v.x, v.y);
    };
    // 16-byte chunk c of a row of a group tile sits at c ^ ((row >> 1) & 7): conflict-free
    // operand reads
    auto dma_x = [&](int s, int u, uint4* slot) {
        const int b = 8 * u + wave;  // eight rows of one group
        const int h4 = b / (2 * kMT), rb8 = b % (2 * kMT);
        const int g = 4 * s + h4;
        const int row = mt * BM + rb8 * 8 + (lane >> 3);
        const int c = (lane & 7) ^ ((4 * (rb8 & 1) + (lane >> 4)) & 7);
        const uint32_t voff = ((uint32_t)row * (uint32_t)a.kx + (uint32_t)(8 * c)) * 2u;
        dma16(make_rsrc(a.x, g < g_end ? x_bytes : 0u), slot + b * 64, voff, (uint32_t)(g >= gx ? g - gx : g) * 128u);
    };

    const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
    const bf16x8 ones = __builtin_bit_cast(bf16x8, make_uint4(0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u));
    // X_g of row 16 (wn + 4 t) + col for the lane's group kq of the step (set 0 sums the
    // step's groups 0 and 1, set 1 groups 2 and 3)
    float xk[kXT];
#pragma unroll
    for (int t = 0; t < kXT; ++t) xk[t] = 0.0f;
    uint32_t ow[2] = {0u, 0u};  // the scale/bias words of the step's group kq, for the wave's own half
    f32x4 acc[kMT][4];
#pragma unroll
    for (int i = 0; i < kMT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = zero;

    auto write_xa = [&](int odd) {
#pragma unroll
        for (int t = 0; t < kXT; ++t)
            if (wn + 4 * t < kMT && (kq >> 1) == set) g_xab[(odd * kMT + wn + 4 * t) * 64 + lane] = x_operand(xk[t]);
    };
    // a step's bias term, each set for its own half of the columns
    auto bias = [&](int odd) {
        bf16x8 bb[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) bb[j] = sb_operand(ow[j]);
#pragma unroll
        for (int i = 0; i < kMT; ++i) {
            const bf16x8 aa = __builtin_bit_cast(bf16x8, g_xab[(odd * kMT + i) * 64 + lane]);
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] = mfma16x16x32(aa, bb[j], acc[i][j]);
        }
    };

    // Step s (groups 4 s .. 4 s + 3): (0) the A operands of step s - 1's bias term, into
    // the slot of its parity (last read in step s - 2, a barrier ago); (1) wait until the
    // wave's x of this step, issued during step s - 1, has landed, leaving in flight the
    // ten loads issued after it; (2) barrier: everyone's x and operands are in LDS and
    // everyone is done with the x slot refilled next; (3) step s - 1's bias term; (4)
    // multiply, with the next step's loads spread through the products: x, then the words
    // of the wave's next pair in place once this pair's are expanded, then this step's
    // scale/bias words.  Every step issues the same loads (past the end they read zeros),
    // so the count is fixed; the first step's x was waited for before the loop.
    auto step = [&](int s, auto odd_, const uint4* xs, uint4* xs2, PairWords& w) {
        constexpr bool kOdd = decltype(odd_)::value;
        if (s > s_begin) write_xa(!kOdd);
        wait_vm_lds<10>();
        lds_barrier();
        if (s > s_begin) bias(!kOdd);
        int ln = threadIdx.x & 63;
        asm volatile("" : "+v"(ln));  // (opaque: keeps the operand addresses per step)
        const int lcol = ln & 15, lkq = ln >> 4;
        const uint4* xl = xs + set * (2 * BM * 8) + lcol * 8;
        const int c0 = lkq ^ ((lcol >> 1) & 7), c1 = (4 + lkq) ^ ((lcol >> 1) & 7);
        auto a_frag = [&](int r, int h) {  // row tile r of the stream: group r / kMT of the pair
            return __builtin_bit_cast(bf16x8, xl[((r / kMT) * BM + 16 * (r % kMT)) * 8 + (h ? c1 : c0)]);
        };
        constexpr int kLag = 3;
        bf16x8 a0 = a_frag(0, 0), a1 = a_frag(0, 1), n0, n1, b0, b1;
        // one group: its 4 kMT tiles in order, kept so by a fence after each tile; tile v's
        // two products with half of tile v - 3's scale FMAs after each
        auto group = [&](auto hh_) {
            constexpr int hh = decltype(hh_)::value;
            bf16x8 bq[4][2];
            float s16[4];
            f32x4 p[kLag + 1], xsum = zero;
            auto scale = [&](int u, int e0) {
#pragma unroll
                for (int e = e0; e < e0 + 2; ++e)
                    acc[u / 4][u % 4][e] = __builtin_fmaf(s16[u % 4], p[u % (kLag + 1)][e], acc[u / 4][u % 4][e]);
            };
#pragma unroll
            for (int v = 0; v < kHalf + kLag; ++v) {
                if (v < kHalf) {
                    const int i = v / 4, j = v % 4, t = hh * kHalf + v;
                    if (i == 0) {  // row 0 expands each row block's words just before its first products
                        bq[j][0] = expand_word(hh ? w.t[j].z : w.t[j].x);
                        bq[j][1] = expand_word(hh ? w.t[j].w : w.t[j].y);
                        s16[j] = bf16_lo(hh ? w.s[j].y : w.s[j].x) * 16.0f;
                    }
                    if (j == 0 && hh * kMT + i + 1 < 2 * kMT) {  // the next row's operands, a row ahead
                        n0 = a_frag(hh * kMT + i + 1, 0);
                        n1 = a_frag(hh * kMT + i + 1, 1);
                    }
                    p[v % (kLag + 1)] = mfma16x16x32(a0, bq[j][0], zero);
                    p[v % (kLag + 1)] = mfma16x16x32(a1, bq[j][1], p[v % (kLag + 1)]);
                    if (j == 3) {
                        a0 = n0;
                        a1 = n1;
                    }
                    constexpr int kXEnd = kHalf + 4;  // x in the first kXEnd tiles, then the words
                    constexpr int kXGap = kXEnd / kMT;
                    if (t % kXGap == 1 && t / kXGap < kMT) dma_x(s + 1, t / kXGap, xs2);
                    constexpr int kWGap = kMT == 2 ? 1 : (kTiles - kXEnd - 2) / 4;
                    if (t >= kXEnd && (t - kXEnd) % kWGap == 0 && (t - kXEnd) / kWGap < 4) load_w(s + 1, (t - kXEnd) / kWGap, w);
                    // X_g of the wave's row tiles, one (row tile, group) at a time: their x
                    // fragments as the B operand against ones, so that every output of column n
                    // is the sum of row n's 64 values (a row tile past the last: the last again)
                    constexpr int kXg = kHalf / kXT;
                    if (v % kXg == 0 && v / kXg < kXT) {
                        const int q = wn + 4 * (v / kXg) < kMT ? wn + 4 * (v / kXg) : kMT - 1;
                        b0 = __builtin_bit_cast(bf16x8, xl[(hh * BM + 16 * q) * 8 + c0]);
                        b1 = __builtin_bit_cast(bf16x8, xl[(hh * BM + 16 * q) * 8 + c1]);
                    }
                    if (v % kXg == 3 && v / kXg < kXT) {
                        xsum = mfma16x16x32(ones, b0, zero);
                        xsum = mfma16x16x32(ones, b1, xsum);
                    }
                    if (v % kXg == 5 && v / kXg < kXT) xk[v / kXg] = (kq & 1) == hh ? xsum[0] : xk[v / kXg];
                    if (t == kTiles - 2) {
                        const bool in = 2 * s + (kq >> 1) < p_end;
#pragma unroll
                        for (int jj = 0; jj < 2; ++jj)
                            ow[jj] = __builtin_amdgcn_raw_buffer_load_b32(
                                make_rsrc(a.sb, a.rec_bytes - kRecSbBytes),
                                (int)(in ? ov + (uint32_t)jj * rb_bytes + (uint32_t)(2 * s) * kRecBytes : kOutOfRange), 0, 0);
                    }
                }
                if (v >= kLag) {
                    scale(v - kLag, 0);
                    scale(v - kLag, 2);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        group(std::integral_constant<int, 0>{});
        group(std::integral_constant<int, 1>{});
    };

    PairWords w;
#pragma unroll
    for (int u = 0; u < kMT; ++u) dma_x(s_begin, u, g_x0);
#pragma unroll
    for (int j = 0; j < 4; ++j) load_w(s_begin, j, w);
    // only the words' eight loads follow the first step's x (no scale/bias words ahead of
    // it), so a step's own wait would leave the wave's last two x loads in flight
    wait_vm<8>();
    for (int s = s_begin; s < s_end; s += 2) {
        step(s, std::integral_constant<bool, false>{}, g_x0, g_x1, w);
        if (s + 1 < s_end) step(s + 1, std::integral_constant<bool, true>{}, g_x1, g_x0, w);
    }
    // the last step's bias term (the drain also lands the zero-reading loads past it);
    // then the sets exchange halves through the x slots
    const int last = (s_end - 1) & 1;
    write_xa(last);
    wait_vm_lds<0>();
    lds_barrier();
    bias(last);
    constexpr int kXchWave = kMT * 2 * 64;  // uint4 per wave
    uint4* const xch = (set ? g_x1 : g_x0) + wn * kXchWave + lane;
#pragma unroll
    for (int i = 0; i < kMT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) xch[(i * 2 + j) * 64] = __builtin_bit_cast(uint4, acc[i][2 + j]);
    wait_lds();
    lds_barrier();
    const uint4* const other = (set ? g_x0 : g_x1) + wn * kXchWave + lane;
    f32x4 out[kMT][2];
#pragma unroll
    for (int i = 0; i < kMT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) out[i][j] = acc[i][j] + __builtin_bit_cast(f32x4, other[(i * 2 + j) * 64]);

    // Output stage: lane (col, kq) holds rows 4 kq + e of column col of row blocks rb0 + j.
    // The tile's rows of the output (or of this split's partial plane) form a buffer: rows
    // past M lie past its end, columns past N are sent there, and such stores are dropped.
    const int rb0 = rbw + 2 * set;
    const int row0 = mt * BM;
    if (a.mode >= kOutLoraBf16) {
        wait_lds();
        lds_barrier();
        float* ts = reinterpret_cast<float*>(g_x0);
        lora_stage_t<BM>(a.lora, ts, row0, a.m_rows, 512);
        if (a.mode == kOutLoraF32)
            lora_store<true>(out, a.lora, ts, a.y, row0, rb0, a.m_rows, a.n_rows, lane);
        else
            lora_store<false>(out, a.lora, ts, a.y, row0, rb0, a.m_rows, a.n_rows, lane);
        return;
    }
    const bool geglu = a.mode == kOutGegluBf16 || a.mode == kOutGegluF32;
    const int ncols = geglu ? a.n_out : a.n_rows;
    const uint32_t esz = a.mode == kOutF32 || a.mode == kOutGegluF32 ? 4u : 2u;
    const uint32_t row_bytes = (uint32_t)ncols * esz;
    const int rows = a.m_rows - row0 < BM ? a.m_rows - row0 : BM;
    const __amdgpu_buffer_rsrc_t yrs =
        make_rsrc(static_cast<char*>(a.y) + ((long)blockIdx.y * a.split_stride + (long)row0 * ncols) * esz, (uint32_t)rows * row_bytes);
    auto out_off = [&](int r, int n) { return n < ncols ? (uint32_t)r * row_bytes + (uint32_t)n * esz : kOutOfRange; };
    auto put16 = [&](uint32_t o, float v) { __builtin_amdgcn_raw_buffer_store_b16((short)f32_to_bf16(v), yrs, (int)o, 0, 0); };
    auto put32 = [&](uint32_t o, float v) { __builtin_amdgcn_raw_buffer_store_b32((int)__float_as_uint(v), yrs, (int)o, 0, 0); };
    if (geglu) {  // rows e and e + 1 share one GeGLU pass
        const uint16_t* gtab = reinterpret_cast<const uint16_t*>(g_x0);
        if (a.mode == kOutGegluBf16) {
            constexpr int kTabChunks = kGeluTable * 2 / 16;
            wait_lds();
            lds_barrier();
            for (int t = (int)threadIdx.x; t < kTabChunks; t += 512) g_x0[t] = reinterpret_cast<const uint4*>(a.gelu_table)[t];
            __syncthreads();
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const uint32_t o = out_off(geglu2_row(col, 4 * kq, 4 * kq + 1), geglu2_col(col, rb0 + j));
            if (a.mode == kOutGegluBf16) {  // all values first: the table reads are issued together
#pragma unroll
                for (int i = 0; i < kMT; ++i)
#pragma unroll
                    for (int e = 0; e < 4; e += 2) out[i][j][e] = geglu2(kOutGegluBf16, col, out[i][j][e], out[i][j][e + 1], gtab);
#pragma unroll
                for (int i = 0; i < kMT; ++i)
#pragma unroll
                    for (int e = 0; e < 4; e += 2) put16(o + (uint32_t)(16 * i + e) * row_bytes, out[i][j][e]);
            } else {
#pragma unroll
                for (int i = 0; i < kMT; ++i)
#pragma unroll
                    for (int e = 0; e < 4; e += 2)
                        put32(o + (uint32_t)(16 * i + e) * row_bytes, geglu2(kOutGegluF32, col, out[i][j][e], out[i][j][e + 1], gtab));
            }
        }
        return;
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint32_t o = out_off(4 * kq, (rb0 + j) * 16 + col);
#pragma unroll
        for (int i = 0; i < kMT; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (a.mode == kOutF32)
                    put32(o + (uint32_t)(16 * i + e) * row_bytes, out[i][j][e]);
                else
                    put16(o + (uint32_t)(16 * i + e) * row_bytes, out[i][j][e]);
            }
    }
}
}  // namespace

hipError_t launch_kpair(const uint4* tiles, const uint2* sb, const uint16_t* x, void* y, int m, int out_mode, int n_out,
                        const Layout& l, const GemmPlan& plan, long split_stride, const uint16_t* gelu_table,
                        const LoraEpilogue& lora, hipStream_t stream) {
    if (!kpair_fits(m, l) || plan.bm > kKpairMaxRows || plan.g_split % 8 != 0) return hipErrorInvalidValue;
    KpairArgs a;
    a.tiles = tiles;
    a.sb = sb;
    a.x = x;
    a.y = y;
    a.gelu_table = gelu_table;
    a.lora = lora;
    a.m_rows = m;
    a.n_rows = l.n;
    a.kx = l.kx;
    a.groups = l.g;
    a.gpairs = l.gp;
    a.mtiles = (m + plan.bm - 1) / plan.bm;
    a.ntiles = (l.n + kKpBN - 1) / kKpBN;
    a.rec_bytes = (uint32_t)l.rec_bytes();
    a.g_split = plan.g_split;
    a.split_stride = split_stride;
    a.n_out = n_out;
    a.mode = out_mode;
    const dim3 grid((unsigned)(a.mtiles * a.ntiles), (unsigned)plan.splits), block(512);
#define Q4_KP(MT) hipLaunchKernelGGL((kpair_kernel<MT>), grid, block, 0, stream, a)
    switch (plan.bm / 16) {
        case 2: Q4_KP(2); break;
        case 3: Q4_KP(3); break;
        case 4: Q4_KP(4); break;
        case 5: Q4_KP(5); break;
        case 6: Q4_KP(6); break;
        case 7: Q4_KP(7); break;
        default: return hipErrorInvalidValue;
    }
#undef Q4_KP
    return hipGetLastError();
}

}  // namespace q4
