// The backward pass on segments of the sequence (few sequences: one workgroup per eight heads and sequence leaves most
// of the chip idle): what every segment adds to the forward and to the adjoint state (the one-pass kernel's states-only
// kinds), then the states entering every segment.  The three scans of the pass start from those, a segment per workgroup.
#include "ssd_fused_scan.h"

namespace ssd {

namespace {

// One thread per four rows p and a column n of a head's state, the S segments in order.  A segment's loads do not depend
// on the recurrence, so kAhead of them are requested at a time: at 64 segments the kernel is eight trips to memory long
// instead of 64.  Along n the reads (and the adjoint's writes back) are whole lines; the transposed states go out as
// 16-byte pieces of four p.  23 us for 32 sequences on 8 segments, 27 for 4 on 64 (84 MB either way: read once, written twice).
constexpr int kAhead = 8;

struct SegmentEntries {
    float *states;             // [B, S, H, P, N]: what each segment adds; the entering states come back in its place
    const float *decay;        // [B, S, H]
    const float *init;         // [B, H, P, N] or NULL
    float *enter_t;            // [B, S, H, N, P]
    const unsigned char *fresh;  // [B, L] or NULL: a non-zero first entry starts from zero
    bool keep;                 // write the entering states over `states`
};

__global__ __launch_bounds__(256) void segment_entries_kernel(SegmentEntries fwd, SegmentEntries adj, int H, int P, int N, int L,
                                                              int S, long long total) {
    const SegmentEntries &a = blockIdx.y == 0 ? fwd : adj;
    const long long gid = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (gid >= total) return;
    const int n = (int)(gid % N), p0 = 4 * (int)((gid / N) % (P / 4));
    const long long bh = gid / ((long long)N * (P / 4));
    const int h = (int)(bh % H);
    const long long b = bh / H;
    const size_t pn = (size_t)P * N, step = (size_t)H * pn;
    float e[4] = {0.f, 0.f, 0.f, 0.f};
    if (a.init != nullptr && !(a.fresh != nullptr && a.fresh[b * L] != 0)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) e[i] = a.init[bh * pn + (size_t)(p0 + i) * N + n];
    }
    const size_t at0 = ((size_t)b * S * H + h) * pn;
    float *src = a.states + at0 + (size_t)p0 * N + n;
    float *dst = a.enter_t + at0 + (size_t)n * P + p0;
    const float *dec = a.decay + (size_t)b * S * H + h;
    for (int j0 = 0; j0 < S; j0 += kAhead) {
        float v[kAhead][4], d[kAhead];
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int j = min(j0 + u, max(S - 2, 0));  // (nothing was written for the last segment, nothing comes after it)
            d[u] = dec[(size_t)j * H];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[u][i] = src[j * step + (size_t)i * N];
        }
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int j = j0 + u;
            if (j < S) {
                *reinterpret_cast<float4 *>(dst + j * step) = make_float4(e[0], e[1], e[2], e[3]);
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    if (a.keep) src[j * step + (size_t)i * N] = e[i];
                    e[i] = d[u] * e[i] + v[u][i];
                }
            }
        }
    }
}

}  // namespace

hipError_t launch_segment_states(const ScanShape &s, bool adjoint, const void *x, const void *dt, const float *A,
                                 const void *Bm, const unsigned char *reset, float *seg_states, float *seg_decay,
                                 hipStream_t st) {
    ScanShape t = s;
    t.Q = kOnePassTile;
    t.nc = (s.L + kOnePassTile - 1) / kOnePassTile;
    if (fused_scan_waves(t, 1) != 8 || (t.N != 32 && t.N != 64) || scan_segments(t) < 2) return hipErrorInvalidValue;
    constexpr int QB = kOnePassTile / 32;
    if (adjoint)
        return t.N == 32 ? fused_launch_states<2, QB, 8, 8>(t, x, dt, A, Bm, nullptr, reset, seg_states, seg_decay, st)
                         : fused_launch_states<4, QB, 8, 8>(t, x, dt, A, Bm, nullptr, reset, seg_states, seg_decay, st);
    return t.N == 32 ? fused_launch_states<2, QB, 8>(t, x, dt, A, Bm, nullptr, reset, seg_states, seg_decay, st)
                     : fused_launch_states<4, QB, 8>(t, x, dt, A, Bm, nullptr, reset, seg_states, seg_decay, st);
}

hipError_t launch_segment_entries(const ScanShape &s, const float *fwd_states, const float *fwd_decay, const float *fwd_init,
                                  const unsigned char *fresh, float *fwd_enter_t, float *adj_states, const float *adj_decay,
                                  const float *adj_init, float *adj_enter_t, hipStream_t st) {
    const int S = scan_segments(s);
    const long long total = (long long)s.B * s.H * (s.P / 4) * s.N;
    if (S < 2 || s.P % 4 != 0 || (total + 255) / 256 > 0x7fffffffLL) return hipErrorInvalidValue;
    const SegmentEntries fwd{const_cast<float *>(fwd_states), fwd_decay, fwd_init, fwd_enter_t, fresh, false};
    const SegmentEntries adj{adj_states, adj_decay, adj_init, adj_enter_t, nullptr, true};
    segment_entries_kernel<<<dim3((unsigned)((total + 255) / 256), 2), dim3(256), 0, st>>>(fwd, adj, s.H, s.P, s.N, s.L, S, total);
    return hipGetLastError();
}

}  // namespace ssd
