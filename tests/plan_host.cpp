// The library's path choice and GEMM plan for a shape, for tests (built by plan_host.py).
#include "q4_kernels.h"

using namespace q4;

// out: decode path, tile rows, splits of K, kpair tile, fp16 form, one-pass 8-bit, scratch
// bytes.  room: the scratch the plan may use, at most what the call's rule allows.
extern "C" void q4_route(int n, int k, int bits, int pair, int f16, int rows, int min_rows, unsigned long room, long* out) {
    Layout l = pair ? pair_layout(n, bits == 8 ? 2 * k : k) : make_layout(n, bits == 8 ? 2 * k : k);
    l.kx = k;
    l.f16 = f16 != 0;
    const size_t most = gemm_room(rows, l, min_rows);
    const GemmPlan p = plan_gemm(rows, l, room < most ? room : most);
    const long v[7] = {use_decode(rows, l, min_rows), p.bm, p.splits, p.kpair, p.f16, p.q8, (long)p.total()};
    for (int i = 0; i < 7; ++i) out[i] = v[i];
}

// ---- forced plans: the launches under the C ABI, on buffers of the caller ----
namespace {
Layout layout_of(int n, int k, int bits, int pair, int f16_p) {
    Layout l = pair ? pair_layout(n, bits == 8 ? 2 * k : k) : make_layout(n, bits == 8 ? 2 * k : k);
    l.kx = k;
    l.f16_p = f16_p;
    return l;
}
// plan_gemm's plan of this tile, form (0 bf16, 1 fp16, 2 one-pass 8-bit) and split count;
// splits 0 in the result: K has no such split
GemmPlan forced_plan(int m, const Layout& l, int bm, int kpair, int form, int splits) {
    GemmPlan p;
    p.bm = bm;
    p.kpair = kpair != 0;
    p.f16 = form == 1;
    p.q8 = form == 2;
    const int groups = form == 2 ? l.g / 2 : l.g, octets = (groups + 7) / 8;
    const int per = (octets + splits - 1) / splits;
    p.splits = (octets + per - 1) / per == splits ? splits : 0;
    p.g_split = per * 8;
    if (bm == 256 || form != 0) p.xaug_bytes = ((size_t)m + bm - 1) / bm * (bm / 16) * octets * 1024;
    if (form != 0) {
        p.x16_bytes = ((size_t)m * l.kx * 2 + 255) & ~(size_t)255;
        p.rowexp_bytes = ((size_t)m * 4 + 255) & ~(size_t)255;
    }
    if (splits > 1) p.part_bytes = (size_t)splits * m * l.n * 4;
    return p;
}
}  // namespace

extern "C" unsigned long q4_rec_bytes(int n, int k, int bits, int pair) { return layout_of(n, k, bits, pair, 0).rec_bytes(); }

extern "C" int q4_repack(const uint32_t* const* w, const uint16_t* const* s, const uint16_t* const* b, char* tiles, int n, int k,
                         int bits, int pair, hipStream_t stream) {
    const Layout l = layout_of(n, k, bits, pair, 0);
    const auto fn = bits == 8 ? launch_repack8 : launch_repack;
    return fn(w[0], s[0], b[0], pair ? w[1] : nullptr, pair ? s[1] : nullptr, pair ? b[1] : nullptr,
              reinterpret_cast<uint4*>(tiles), reinterpret_cast<uint2*>(tiles + kRecSbBytes), l, pair ? n : 0, stream);
}

extern "C" int q4_gelu(uint16_t* table, hipStream_t stream) { return launch_gelu_table(table, stream); }

// scratch bytes of the plan, or -1
extern "C" long q4_forced_bytes(int n, int k, int bits, int pair, int m, int bm, int kpair, int form, int splits) {
    const GemmPlan p = forced_plan(m, layout_of(n, k, bits, pair, 0), bm, kpair, form, splits);
    return p.splits == splits ? (long)p.total() : -1;
}

// mode: 0 bf16 y, 1 fp32 y, 2 / 3 GeGLU h; part: an adapter's t as [slices][m][rank], or null
extern "C" int q4_forced_gemm(char* tiles, const uint16_t* x, void* y, int m, int mode, int n, int k, int bits, int pair, int f16_p,
                              int bm, int kpair, int form, int splits, void* ws, unsigned long ws_bytes, const uint16_t* gelu,
                              const float* part, const float* b, int rank, int slices, float scale, hipStream_t stream) {
    const Layout l = layout_of(n, k, bits, pair, f16_p);
    const GemmPlan p = forced_plan(m, l, bm, kpair, form, splits);
    if (p.splits != splits) return hipErrorInvalidValue;
    const LoraEpilogue lo{part, b, rank, slices, scale};
    return launch_gemm(reinterpret_cast<uint4*>(tiles), reinterpret_cast<uint2*>(tiles + kRecSbBytes), x, y, m, mode, pair ? n : 0,
                       l, p, ws, ws_bytes, gelu, stream, part ? &lo : nullptr);
}
