// Weight gradients of the block's projections (gfx950): out [E, N] = a^T b in float32 for tall bf16 a [rows, E] (rows lda
// apart) and b [rows, N], N 128 or 256 -- a sum over every timestep of the batch.
//
// What bounds it is reading a and b once (704 + 256 columns by 524 288 rows: 1.0 GB, 0.2 ms).  The rows are cut into as many
// splits as fill the chip together with the blocks of 128 output rows; a split's blocks are consecutive workgroups of one XCD,
// so all but the first find b in its L2.  A workgroup keeps its [128, N] block in matrix-core accumulators over its whole split
// and walks it 64 rows at a time: both operands have the sum's index along their rows, so the tiles go to LDS as they lie in
// memory and come out through the transposing read; two sets of tiles, one barrier a step, the next step's rows requested
// behind it.  Partial blocks go out once per split and a second kernel adds them in order (the same bits every run).  Every
// kFlushSteps steps the accumulators are added to a second set and cleared, so that a product goes through the 16 additions of
// 256 rows, one per 256 rows of its split and one per split (256 x 256 outputs beside 648 x 256, error against float64 with a set
// cleared every 4 096 rows / 512 / 256: 12 000 rows 1.65e-7 / 1.65e-7 / 1.46e-7, 16 384 1.78e-7 / 1.78e-7 / 1.51e-7, 60 000 3.01e-7 /
// 1.83e-7 / 1.62e-7, 81 920 3.38e-7 / 1.87e-7 / 1.64e-7; 4 096 / 256 rows, us: 648 x 256 outputs at 16 384 rows 23.5 / 23.9, 72 828 55.0 / 56.9,
// 524 288 351.8 / 354.8, both of a training pass at 16 384 rows within the runs).
//
// Against the BLAS, whose batched products over equal slabs of rows need a row count with a power of two in it (any other
// ran as one product with a bf16 result at a fifth of the rate), in us, BLAS / here: 648 x 256 outputs at 16 384 rows 38 / 26,
// 72 828 rows 151 / 59, 131 072 rows 130 / 103, 199 374 rows 388 / 155, 262 144 rows 150 / 200, 524 288 rows 300 / 415; 256 x 256
// at the same rows 36 / 22, 83 / 35, 51 / 45, 360 / 58, 85 / 93, 120 / 167: the caller keeps the BLAS for row counts that it cuts
// into many slabs, 64 and more at these widths and fewer at wide E (b is read again for every 128 of it, and above 1 024 a round of
// splits no longer fills the chip: E 2 184 at 131 056 rows 204 / 410).  At the largest this kernel waits for memory with 48 KB per
// compute unit in flight: two steps ahead take 72
// registers more than there are (spilled: 477), and four waves with all registers leave the reads of LDS uncovered (824).
#include "ssd_fused_scan.h"

namespace ssd {

namespace {

constexpr int kWgradCols = 128;     // output rows (columns of a) per workgroup
constexpr int kWgradRows = 64;      // rows per step
constexpr int kWgradThreads = 512;
constexpr int kFlushSteps = 4;     // 256 rows
constexpr int kWgradMinRows = 256;  // per split: shorter ones are mostly the partial block's way out

// One weight gradient of a launch: its operands and where its splits' blocks go ([splits, E, N]).
struct WgradJob {
    const __bf16 *a, *b;
    float *part;
    int E, lda, blocks;
};

// (two jobs over the same rows, of which the second may have no blocks: the workgroups of the first come first)
template <int NB>  // N = 128 NB
__global__ __launch_bounds__(kWgradThreads) void block_wgrad_kernel(WgradJob first, WgradJob second, int first_groups, long long rows,
                                                                    int splits, long long split_rows) {
    const bool one = (int)blockIdx.x < first_groups;
    const WgradJob &job = one ? first : second;
    const int group = (int)blockIdx.x - (one ? 0 : first_groups);  // (a multiple of 8: the XCD is the block's)
    const __bf16 *__restrict__ a = job.a;
    const __bf16 *__restrict__ b = job.b;
    float *__restrict__ part = job.part;
    const int E = job.E, lda = job.lda, blocks = job.blocks;
    using T = ChunkTile<128>;
    constexpr int N = 128 * NB, TILE = kWgradRows * 128;
    constexpr int WN = N / 64, WM = 8 / WN, MI = kWgradCols / WM / 32, NI = 2;  // a wave: MI x NI tiles of 32 x 32
    constexpr int UA = TILE / 8 / kWgradThreads, UB = UA * NB, PB = N / 8;      // 16-byte pieces per thread and step
    __shared__ __attribute__((aligned(16))) __bf16 sm[2][TILE * (1 + NB)];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wm = wave / WN, wn = wave % WN;
    const int xcd = group % 8, within = group / 8;
    const int split = (within / blocks) * 8 + xcd, m0 = (within % blocks) * kWgradCols;
    if (split >= splits) return;  // (the grid is padded to whole rounds of XCDs)
    const long long begin = split * split_rows, end = min(rows, begin + split_rows);

    // (a row past the split repeats a row inside the tensors and counts as zeros, a column past E repeats the last piece and
    // is not stored: no load stands under a condition)
    uint4 qa[UA], qb[UB];
    auto fetch = [&](long long r0) {
#pragma unroll
        for (int i = 0; i < UA; ++i) {
            const int p = tid + i * kWgradThreads;
            qa[i] = *reinterpret_cast<const uint4 *>(a + (size_t)min(r0 + p / 16, rows - 1) * lda + min(m0 + (p % 16) * 8, E - 8));
        }
#pragma unroll
        for (int i = 0; i < UB; ++i) {
            const int p = tid + i * kWgradThreads;
            qb[i] = *reinterpret_cast<const uint4 *>(b + (size_t)min(r0 + p / PB, rows - 1) * N + (p % PB) * 8);
        }
    };
    auto stage = [&](long long r0, __bf16 *s) {
        const bool whole = r0 + kWgradRows <= end;
        auto keep = [&](const uint4 &v, int row) { return whole || r0 + row < end ? v : make_uint4(0, 0, 0, 0); };
#pragma unroll
        for (int i = 0; i < UA; ++i) {
            const int p = tid + i * kWgradThreads;
            T::put16(s, p / 16, (p % 16) * 8, keep(qa[i], p / 16));
        }
#pragma unroll
        for (int i = 0; i < UB; ++i) {
            const int p = tid + i * kWgradThreads, col = (p % PB) * 8;
            T::put16(s + TILE * (1 + col / 128), p / PB, col % 128, keep(qb[i], p / PB));
        }
    };
    f32x16 acc[MI][NI], total[MI][NI];
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NI; ++j) acc[i][j] = total[i][j] = f32x16{0};
    }
    const bool busy = m0 + wm * MI * 32 < E;  // (the last block of output rows may leave waves nothing)
    const int n0 = wn * 64;
    fetch(begin);
    int step = 0;
    for (long long r0 = begin; r0 < end; r0 += kWgradRows, ++step) {
        __bf16 *s = sm[step & 1];
        stage(r0, s);
        block_sync_lds();  // (the other set was last read a step ago, before this barrier)
        fetch(r0 + kWgradRows);
        __builtin_amdgcn_sched_barrier(0);  // (the requests go out here, ahead of the products)
        if (busy) {
#pragma unroll
            for (int ks = 0; ks < kWgradRows; ks += 16) {
                Frag<__bf16> fa[MI], fb[NI];
#pragma unroll
                for (int i = 0; i < MI; ++i) fa[i] = T::frag(s, ks + 8 * half, 4, (wm * MI + i) * 32, lane);
#pragma unroll
                for (int j = 0; j < NI; ++j) fb[j] = T::frag(s + TILE * (1 + n0 / 128), ks + 8 * half, 4, n0 % 128 + j * 32, lane);
#pragma unroll
                for (int i = 0; i < MI; ++i) {
#pragma unroll
                    for (int j = 0; j < NI; ++j) acc[i][j] = mma32(fa[i], fb[j], acc[i][j]);
                }
            }
            if ((step + 1) % kFlushSteps == 0 && r0 + kWgradRows < end) {
#pragma unroll
                for (int i = 0; i < MI; ++i) {
#pragma unroll
                    for (int j = 0; j < NI; ++j) {
                        total[i][j] += acc[i][j];
                        acc[i][j] = f32x16{0};
                    }
                }
            }
        }
    }
    if (!busy) return;
    float *out = part + (size_t)split * E * N;
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
        for (int j = 0; j < NI; ++j) {
            total[i][j] += acc[i][j];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int m = m0 + (wm * MI + i) * 32 + 8 * (v / 4) + 4 * half + v % 4;
                if (m < E) out[(size_t)m * N + n0 + j * 32 + (lane & 31)] = total[i][j][v];
            }
        }
    }
}

// out = the splits' blocks added in order; four elements per thread, eight splits' requested at a time (two jobs, as above)
__global__ __launch_bounds__(256) void block_wgrad_sum_kernel(const float4 *__restrict__ part0, float4 *__restrict__ out0, int pieces0,
                                                              const float4 *__restrict__ part1, float4 *__restrict__ out1, int pieces1,
                                                              int splits) {
    int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= pieces0 + pieces1) return;
    const bool one = i < pieces0;
    const int pieces = one ? pieces0 : pieces1;
    const float4 *part = one ? part0 : part1;
    if (!one) i -= pieces0;
    float4 sum = make_float4(0, 0, 0, 0);
    for (int s0 = 0; s0 < splits; s0 += 8) {
        float4 q[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) q[u] = part[(size_t)min(s0 + u, splits - 1) * pieces + i];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const float w = s0 + u < splits ? 1.f : 0.f;
            sum.x += w != 0.f ? q[u].x : 0.f;
            sum.y += w != 0.f ? q[u].y : 0.f;
            sum.z += w != 0.f ? q[u].z : 0.f;
            sum.w += w != 0.f ? q[u].w : 0.f;
        }
    }
    (one ? out0 : out1)[i] = sum;
}

struct WgradPlan {
    int splits;
    long long split_rows;
};

int wgrad_blocks(int E) { return (E + kWgradCols - 1) / kWgradCols; }

// Splits: one round of workgroups (a compute unit holds one), whole XCDs, none below kWgradMinRows rows.  (256 compute units are
// a constant here: the workspace is laid out by the splits, and the order of the sums, so the bits, do not depend on the device.)
long long wgrad_most_splits(long long rows, int blocks) {
    const long long fill = std::max(1, 256 / 8 / blocks) * 8;
    return std::max<long long>(1, std::min(fill, rows / kWgradMinRows));
}

WgradPlan wgrad_plan(long long rows, int blocks) {
    WgradPlan p;
    const long long most = wgrad_most_splits(rows, blocks);
    p.split_rows = ((rows + most - 1) / most + kWgradRows - 1) / kWgradRows * kWgradRows;
    p.splits = (int)((rows + p.split_rows - 1) / p.split_rows);
    return p;
}

}  // namespace

bool block_wgrad_supported(long long rows, int E, int N) {
    return rows > 0 && rows <= 0x7fffffffLL && E >= 8 && E % 8 == 0 && E <= 8192 && (N == 128 || N == 256);
}

size_t block_wgrad_workspace_bytes(long long rows, int E, int N, int E2) {
    const WgradPlan p = wgrad_plan(rows, wgrad_blocks(E) + (E2 > 0 ? wgrad_blocks(E2) : 0));
    return p.splits > 1 ? (size_t)p.splits * (E + E2) * N * sizeof(float) : 0;
}

size_t block_wgrad_workspace_bound(long long rows, int E, int N, int E2) {
    const long long most = wgrad_most_splits(rows, wgrad_blocks(E) + (E2 > 0 ? wgrad_blocks(E2) : 0));
    return most > 1 ? (size_t)most * (E + E2) * N * sizeof(float) : 0;
}

// Both weight gradients of a block in one launch: the blocks of both share one round of workgroups, and a few rows' partial
// blocks one launch for their sums (the two on their own, 648 x 256 and 256 x 256 outputs in us: 800 rows 12 + 4 + 11 + 4 -> 12.2 + 4,
// 16 384 rows 17.5 + 5 + 12.7 + 5.9 -> 20.2 + 6).
hipError_t launch_block_wgrad2(long long rows, int N, const WgradArgs &x, const WgradArgs &y, void *workspace, hipStream_t st) {
    if (!block_wgrad_supported(rows, x.E, N) || x.lda < x.E || x.lda % 8 != 0) return hipErrorInvalidValue;
    const bool two = y.E > 0;
    if (two && (!block_wgrad_supported(rows, y.E, N) || y.lda < y.E || y.lda % 8 != 0)) return hipErrorInvalidValue;
    const int blocks0 = wgrad_blocks(x.E), blocks1 = two ? wgrad_blocks(y.E) : 0;
    const WgradPlan p = wgrad_plan(rows, blocks0 + blocks1);
    float *part0 = p.splits > 1 ? static_cast<float *>(workspace) : x.out;
    float *part1 = p.splits > 1 ? part0 + (size_t)p.splits * x.E * N : y.out;
    auto job = [](const WgradArgs &g, float *part, int blocks) {
        return WgradJob{static_cast<const __bf16 *>(g.a), static_cast<const __bf16 *>(g.b), part, g.E, g.lda, blocks};
    };
    const int per_block = (p.splits + 7) / 8 * 8, groups0 = per_block * blocks0;
    const dim3 grid((unsigned)(groups0 + per_block * blocks1)), block(kWgradThreads);
    if (N == 256)
        block_wgrad_kernel<2><<<grid, block, 0, st>>>(job(x, part0, blocks0), job(y, part1, blocks1), groups0, rows, p.splits, p.split_rows);
    else
        block_wgrad_kernel<1><<<grid, block, 0, st>>>(job(x, part0, blocks0), job(y, part1, blocks1), groups0, rows, p.splits, p.split_rows);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess || p.splits == 1) return e;
    const int pieces0 = x.E * N / 4, pieces1 = two ? y.E * N / 4 : 0;
    block_wgrad_sum_kernel<<<dim3((pieces0 + pieces1 + 255) / 256), dim3(256), 0, st>>>(
        reinterpret_cast<const float4 *>(part0), reinterpret_cast<float4 *>(x.out), pieces0, reinterpret_cast<const float4 *>(part1),
        reinterpret_cast<float4 *>(y.out), pieces1, p.splits);
    return hipGetLastError();
}

hipError_t launch_block_wgrad(long long rows, int E, int N, int lda, const void *a, const void *b, float *out, void *workspace,
                              hipStream_t st) {
    return launch_block_wgrad2(rows, N, WgradArgs{a, b, out, E, lda}, WgradArgs{}, workspace, st);
}

}  // namespace ssd
