// The gradient of a projection's input (gfx950): out[m, n] = sum_k a[m, k] wt[n, k] for a [rows, K] (the gradient of the
// projection's output: K a few hundred, any multiple of 8, rows lda apart) and wt [N, ldw], the weight matrix turned so that K is
// contiguous and padded with zeros to whole steps of 16; bf16 in and out, float32 accumulation.
//
// For up to 16 384 rows.  A workgroup owns 32 RT rows and 32 columns for each of its WAVES waves: its rows of a go to LDS once, whole
// (42 KB per 32 rows at K 648), and from then on the waves run without a barrier, each on its 32 columns, whose weights come straight
// from memory -- from the XCD's L2 -- in operand fragments, a batch of steps ahead of the products.  What bounds it is a workgroup's
// trip to memory for a and then the weights' way out of L2, 41 KB per wave at K 648: hence the narrow workgroups, so that few rows
// still occupy every compute unit, and larger ones as soon as those make more than a round.  648 -> 256 in us, the BLAS / 32 rows x
// 128 columns / 64 x 128 / 64 x 256: 64 rows 14.7 / 7.4 / 8.7 / 12.2, 4 000 9.5 / 8.1 / 9.1 / 12.5, 8 192 14.1 / 12.3 / 9.8 / 13.0,
// 16 384 16.2 / 20.7 / 17.7 / 14.2, 24 000 20.8 / 29 / 26 / 26; 392 -> 128: 800 rows 8.6 / 5.4 / 6.8 / 7.3, 16 384 10.2 / 9.1 / 7.7 /
// 8.4; 1 288 -> 256: 800 rows 10.1 / 12.4.  (And 20 us of the host's time against 4.)  Above, the weights are read too often and the
// caller's BLAS is the faster.
#include "ssd_device.h"

namespace ssd {

namespace {

constexpr int kDprojBatch = 8;

inline int dproj_steps(int K) { return (K + 15) / 16; }
// bytes of a staged row: whole steps and 16 more, an odd number of 16-byte pieces, which spreads 16 rows over all banks
__host__ __device__ inline int dproj_row_bytes(int steps) { return steps * 32 + 16; }

template <int RT, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void block_dproj_kernel(const __bf16 *__restrict__ a, const __bf16 *__restrict__ wt,
                                                                       __bf16 *__restrict__ out, long long M, int K, int lda, int ldw,
                                                                       int N, int ldo, int col_blocks) {
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    constexpr int NTHR = 64 * WAVES, ROWS = 32 * RT;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, half = lane >> 5;
    // (the column blocks of a range of rows are consecutive workgroups of one XCD: all but the first find those rows in its L2)
    const int xcd = blockIdx.x % 8, within = blockIdx.x / 8;
    const long long row0 = ((long long)(within / col_blocks) * 8 + xcd) * ROWS;
    if (row0 >= M) return;  // the grid is padded to whole rounds of XCDs
    const int n0 = (within % col_blocks) * (32 * WAVES) + wave * 32;
    const int steps = (K + 15) / 16, rowb = dproj_row_bytes(steps);
    // the first batch of this wave's weights (columns past N repeat the last one and are not stored)
    const __bf16 *wr = wt + (size_t)min(n0 + r, N - 1) * ldw + 8 * half;
    uint4 wq[2][kDprojBatch];
    auto fetch = [&](int s0, uint4(&q)[kDprojBatch]) {
#pragma unroll
        for (int i = 0; i < kDprojBatch; ++i) q[i] = *reinterpret_cast<const uint4 *>(wr + 16 * min(s0 + i, steps - 1));
    };
    {   // rows of a -> LDS, eight pieces per thread in flight at a time (rows past M repeat the last one; the half step past an
        // odd number of pieces is zeros: the row may be part of a longer one, whose next elements are not a's)
        const int pieces = steps * 2, total = ROWS * pieces;
        for (int p0 = tid; p0 < total; p0 += 8 * NTHR) {
            uint4 q[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int p = min(p0 + i * NTHR, total - 1), row = p / pieces, c = p % pieces;
                q[i] = *reinterpret_cast<const uint4 *>(a + (size_t)min(row0 + row, M - 1) * lda + min(c * 8, K - 8));
            }
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int p = min(p0 + i * NTHR, total - 1), row = p / pieces, c = p % pieces;
                *reinterpret_cast<uint4 *>(smem + row * rowb + c * 16) = c * 8 < K ? q[i] : make_uint4(0, 0, 0, 0);
            }
        }
    }
    fetch(0, wq[0]);
    block_sync_lds();
    f32x16 acc[RT];
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = f32x16{0};
    auto products = [&](int s0, const uint4(&q)[kDprojBatch]) {
#pragma unroll
        for (int i = 0; i < kDprojBatch; ++i) {
            if (s0 + i < steps) {  // (uniform)
                Frag<__bf16> wf;
                wf.v = __builtin_bit_cast(bf16x8, q[i]);
#pragma unroll
                for (int t = 0; t < RT; ++t) {
                    Frag<__bf16> af;
                    af.v = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(smem + (t * 32 + r) * rowb + (s0 + i) * 32 + half * 16));
                    acc[t] = mma32(wf, af, acc[t]);
                }
            }
        }
    };
    for (int s0 = 0; s0 < steps; s0 += 2 * kDprojBatch) {
        fetch(s0 + kDprojBatch, wq[1]);
        __builtin_amdgcn_sched_barrier(0);
        products(s0, wq[0]);
        fetch(s0 + 2 * kDprojBatch, wq[0]);
        __builtin_amdgcn_sched_barrier(0);
        products(s0 + kDprojBatch, wq[1]);
    }
    if (n0 >= N) return;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        float o[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) o[i] = acc[t][i];
        const long long row = row0 + t * 32 + r;
        store_column<__bf16>(out + (size_t)min(row, M - 1) * ldo + n0, o, half, N - n0, row < M);
    }
}

size_t dproj_lds_bytes(int rt, int K) { return (size_t)32 * rt * dproj_row_bytes(dproj_steps(K)); }

// The block's float32 weights in bf16, as the projections' kernels read them, in one launch: in_proj [E, D] as it is and turned (see
// block_dproj: [D, ldt], zeros from column E on), out_proj [D, DI] as it is and turned.  A workgroup per tile of 32 x 32.
__global__ __launch_bounds__(256) void block_weights_kernel(const float *__restrict__ in_proj, const float *__restrict__ out_proj, int E,
                                                            int D, int DI, int ldt, __bf16 *__restrict__ w_in, __bf16 *__restrict__ w_in_t,
                                                            __bf16 *__restrict__ w_out, __bf16 *__restrict__ w_out_t, int in_tiles) {
    __shared__ __bf16 tile[32][33];
    const bool first = (int)blockIdx.x < in_tiles;
    const int t = (int)blockIdx.x - (first ? 0 : in_tiles);
    const int rows = first ? E : D, cols = first ? D : DI, ld = first ? ldt : D;  // ld: of the turned matrix, its columns
    const float *src = first ? in_proj : out_proj;
    __bf16 *plain = first ? w_in : w_out, *turned = first ? w_in_t : w_out_t;
    const int col_tiles = (cols + 31) / 32, r0 = t / col_tiles * 32, c0 = t % col_tiles * 32;
    const int x = threadIdx.x & 31, y0 = threadIdx.x >> 5;
    for (int y = y0; y < 32; y += 8) {
        const int r = r0 + y, c = c0 + x;
        const bool in = r < rows && c < cols;
        const __bf16 v = (__bf16)(in ? src[(size_t)r * cols + c] : 0.f);
        if (in) plain[(size_t)r * cols + c] = v;
        tile[y][x] = v;
    }
    __syncthreads();
    for (int y = y0; y < 32; y += 8) {
        const int c = c0 + y, r = r0 + x;  // element (c, r) of the turned matrix
        if (c < cols && r < ld) turned[(size_t)c * ld + r] = tile[x][y];
    }
}

}  // namespace

hipError_t launch_block_weights(int E, int D, int DI, const float *in_proj, const float *out_proj, void *w_in, void *w_in_t, void *w_out,
                                void *w_out_t, hipStream_t st) {
    const int ldt = 16 * dproj_steps(E);  // (at most 15 columns past E: inside the last tile of 32 rows, or a tile of its own)
    const long long in_tiles = (long long)((ldt + 31) / 32) * ((D + 31) / 32), out_tiles = (long long)((D + 31) / 32) * ((DI + 31) / 32);
    if (in_tiles + out_tiles > 0x7fffffffLL) return hipErrorInvalidValue;
    block_weights_kernel<<<dim3((unsigned)(in_tiles + out_tiles)), dim3(256), 0, st>>>(
        in_proj, out_proj, E, D, DI, ldt, static_cast<__bf16 *>(w_in), static_cast<__bf16 *>(w_in_t), static_cast<__bf16 *>(w_out),
        static_cast<__bf16 *>(w_out_t), (int)in_tiles);
    return hipGetLastError();
}

bool block_dproj_supported(long long rows, int K, int N) {
    return rows > 0 && K > 0 && K % 8 == 0 && N > 0 && N % 8 == 0 && dproj_lds_bytes(1, K) <= kLdsLimitBytes;
}

hipError_t launch_block_dproj(long long rows, int K, int N, int lda, int ldw, const void *a, const void *wt, void *out, hipStream_t st) {
    if (!block_dproj_supported(rows, K, N) || lda < K || lda % 8 != 0 || ldw < 16 * dproj_steps(K) || ldw % 8 != 0)
        return hipErrorInvalidValue;
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = device_cu_count(dev, &cus);
    if (e != hipSuccess) return e;
    // the first of 32 rows x 128 columns, 64 x 128 and 64 x 256 that makes one round of workgroups (the last where none does)
    auto groups_of = [&](int rt, int waves) { return (rows + 32 * rt - 1) / (32 * rt) * ((N + 32 * waves - 1) / (32 * waves)); };
    const bool fits = dproj_lds_bytes(2, K) <= kLdsLimitBytes;
    const int rt = groups_of(1, 4) <= cus || !fits ? 1 : 2;
    const int waves = rt == 1 || groups_of(2, 4) <= cus || N <= 128 ? 4 : 8;
    const int col_blocks = (N + 32 * waves - 1) / (32 * waves);
    const long long tiles = (rows + 32 * rt - 1) / (32 * rt), groups = (tiles + 7) / 8 * 8 * col_blocks;
    if (groups > 0x7fffffffLL) return hipErrorInvalidValue;
    const size_t lds = dproj_lds_bytes(rt, K);
    const dim3 grid((unsigned)groups), block(64 * waves);
    const __bf16 *aa = static_cast<const __bf16 *>(a), *ww = static_cast<const __bf16 *>(wt);
    __bf16 *oo = static_cast<__bf16 *>(out);
#define SSD_DPROJ_CASE(RTv, Wv)                                                                                         \
    if (rt == RTv && waves == Wv) {                                                                                     \
        if ((e = allow_lds(block_dproj_kernel<RTv, Wv>, lds)) != hipSuccess) return e;                                  \
        block_dproj_kernel<RTv, Wv><<<grid, block, lds, st>>>(aa, ww, oo, rows, K, lda, ldw, N, N, col_blocks);         \
        return hipGetLastError();                                                                                       \
    }
    SSD_DPROJ_CASE(1, 4) SSD_DPROJ_CASE(2, 4) SSD_DPROJ_CASE(2, 8)
#undef SSD_DPROJ_CASE
    return hipErrorInvalidValue;
}

}  // namespace ssd
