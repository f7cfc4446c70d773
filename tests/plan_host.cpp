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
