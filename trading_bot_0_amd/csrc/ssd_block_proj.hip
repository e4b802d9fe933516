// The block's projections: out[m, n] = sum_k u[m, k] w[n, k] for a tall u (rows = batch * seqlen, 128 or 256
// columns) and a small weight matrix, bf16 in and out, float32 accumulation (gfx950).
//
// With K of a few hundred the product is bound by memory, not by the matrix cores: u is read once, out written once
// (0.95 GB for 524 288 rows, 256 -> 648).  A workgroup owns a block of at most 160 output columns and a range of 256 to
// 2 048 rows (proj_split): it puts its rows of w into LDS once (84 KB at most), and from then on its eight waves run without a barrier -- each
// takes tiles of 32 rows, loads its rows of u straight into MFMA operand fragments (u and w are both contiguous
// along K, so a lane's eight K elements are one 16-byte load; the next tile's rows are in flight during this
// tile's products), and walks the block's columns in chunks of 32 with the w fragments read from LDS.  The MFMA's
// first operand is w, so that a lane ends up with one row m and runs of four consecutive columns n; two chunks are
// collected in an LDS tile of the wave's own and written out with adjacent lanes on adjacent 16-byte pieces of a
// row (stores scattered over 32 rows straight from the accumulators' layout run at a fraction of the memory
// system's rate).
#include <algorithm>

#include "ssd_block_common.h"
#include "ssd_device.h"

namespace ssd {

namespace {

constexpr int kProjWaves = 8;         // waves per workgroup: two per SIMD, 256 registers each
constexpr int kProjBlockCols = 160;   // most output columns per workgroup (their rows of w stay in LDS)
constexpr int kProjChunk = 32;        // output columns per MFMA tile
constexpr int kProjTiles = 8;         // most tiles of 32 rows per wave

// CH: 32-column chunks of the widest block of columns (1..5; a block walks CH chunks, or CH - 1 where those cover it, and the
// chunks past its columns -- several, where a last narrow block is left: 648 columns in blocks of 128 leave 8 -- are
// multiplied and not stored).  The chunk count is a template parameter and every store goes out without a condition -- a
// buffer store whose offset is put out of range for rows past M and columns past the block, which the hardware then
// drops -- because loads and stores share one counter per wave, in order: only in straight-line code with every
// store counted does the compiler wait for a tile's rows of u by their exact position in that order.  With a loop of
// unknown length or a guarded store in between it waits for everything outstanding -- the next tile's rows, requested
// a moment ago, and the last stores -- and the tile's loads, products and stores ran one after the other.
template <int KS, int CH, int TILES>  // K = 16 * KS; TILES: tiles of 32 rows per wave
__global__ __launch_bounds__(64 * kProjWaves) void block_proj_kernel(const __bf16 *__restrict__ u,
                                                                      const __bf16 *__restrict__ w,
                                                                      __bf16 *__restrict__ out, long long M, int N,
                                                                      int ldo, int col_blocks, int block_cols) {
    constexpr int K = 16 * KS, NTHR = 64 * kProjWaves;
    constexpr int ROWB = K * 2 + 16;        // bytes of a staged row of w: 16 bytes of padding shift the banks
    constexpr int kTileRowB = 64 * 2 + 16;  // a row of a wave's output tile: 64 columns and 16 bytes of padding
    __shared__ __attribute__((aligned(16))) unsigned char wsm[CH * kProjChunk * ROWB];
    __shared__ __attribute__((aligned(16))) unsigned char otile[kProjWaves][32 * kTileRowB];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    // Workgroups go to the eight XCDs in turn, each XCD with an L2 of its own: the column blocks of a range of rows
    // are consecutive workgroups of ONE XCD, so that they run at the same time and all but the first find those
    // rows of u in its L2.
    const int xcd = blockIdx.x % 8, within = blockIdx.x / 8;
    const int cb = within % col_blocks;
    const long long rg = (long long)(within / col_blocks) * 8 + xcd;
    const int n0 = cb * block_cols;                 // this workgroup's first column
    const int ncols = cb == col_blocks - 1 ? N - n0 : block_cols;  // a multiple of 8; the last block takes the rest
    const long long row0 = rg * TILES * (32LL * kProjWaves);
    if (row0 >= M) return;  // the grid is padded to whole rounds of XCDs

    {   // rows n0 .. n0 + 32 * CH - 1 of w, all requested before the first is written to LDS (rows past N repeat the
        // last one, and pieces past the block are the block's last piece once more: neither loads nor writes stand
        // under a condition; the surplus columns are never stored)
        constexpr int PIECES = CH * kProjChunk * (K / 8);
        constexpr int FILL = (PIECES + NTHR - 1) / NTHR;
        uint4 q[FILL];
#pragma unroll
        for (int i = 0; i < FILL; ++i) {
            const int p = min(tid + i * NTHR, PIECES - 1);
            q[i] = *reinterpret_cast<const uint4 *>(w + (size_t)min(n0 + p / (K / 8), N - 1) * K + (p % (K / 8)) * 8);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < FILL; ++i) {
            const int p = min(tid + i * NTHR, PIECES - 1);
            *reinterpret_cast<uint4 *>(wsm + (p / (K / 8)) * ROWB + (p % (K / 8)) * 16) = q[i];
        }
    }
    __syncthreads();

    const int r = lane & 31, half = lane >> 5;
    unsigned char *tile = otile[wave];
    // the workgroup's rows of `out` as a range-checked buffer: up to 2 048 rows of at most ldo elements
    const __amdgpu_buffer_rsrc_t obuf = make_buffer(out + (size_t)row0 * ldo, (unsigned)min((long long)TILES * 32 * kProjWaves, M - row0) * (unsigned)ldo * 2u);
    auto tile_row0 = [&](int t) { return row0 + (long long)t * (32 * kProjWaves) + wave * 32; };
    // this lane's part of its row of u: K elements 16 ks + 8 half .. + 7 for every K step (rows past M repeat the
    // last row; they are never stored)
    auto load_rows = [&](int t, Frag<__bf16>(&uf)[KS]) {
        const __bf16 *ur = u + (size_t)min(tile_row0(t) + r, M - 1) * K + 8 * half;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) uf[ks].v = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(ur + 16 * ks));
    };
    // (a block takes CH chunks or one fewer -- 648 columns are 4 x 128 + 136 -- and the last chunk is the only piece
    // of a tile's work under a condition, a uniform one)
    const bool last_chunk = ncols > (CH - 1) * kProjChunk;
    constexpr int kRing = KS < 8 ? KS : 8;
    uint4 wq[kRing];  // the next kRing fragments of w
#pragma unroll
    for (int ks = 0; ks < kRing; ++ks) wq[ks] = *reinterpret_cast<const uint4 *>(wsm + r * ROWB + half * 16 + ks * 32);
    auto tile_product = [&](int t, const Frag<__bf16>(&uf)[KS]) {
        const unsigned trow = (unsigned)(t * (32 * kProjWaves) + wave * 32);  // the tile's first row within the workgroup's
        const long long m0 = tile_row0(t);
#pragma unroll
        for (int c0 = 0; c0 < CH; c0 += 2) {
            if (c0 == CH - 1 && !last_chunk) break;  // (an odd CH: the last pair is the last chunk alone)
#pragma unroll
            for (int sub = 0; sub < 2; ++sub) {
                const int c = c0 + sub;
                if (c >= CH || (c == CH - 1 && !last_chunk)) break;
                // the chunk that follows this one (the next tile's first after the last)
                const int cn = (c + 1 < CH && (c + 1 < CH - 1 || last_chunk)) ? c + 1 : 0;
                const unsigned char *wb = wsm + (c * kProjChunk + r) * ROWB + half * 16;
                const unsigned char *wn = wsm + (cn * kProjChunk + r) * ROWB + half * 16;
                f32x16 acc = {0}, acc_odd = {0};  // two chains of dependent MFMAs instead of one
#pragma unroll
                for (int ks = 0; ks < KS; ks += 2) {
                    Frag<__bf16> wf0, wf1;
                    wf0.v = __builtin_bit_cast(bf16x8, wq[ks % kRing]);
                    wf1.v = __builtin_bit_cast(bf16x8, wq[(ks + 1) % kRing]);
                    acc = mma32(wf0, uf[ks], acc);
                    acc_odd = mma32(wf1, uf[ks + 1], acc_odd);
                    // ... and the fragments of w kRing K steps further on (in this chunk or the next), each requested
                    // into the registers of the one just used: kRing / 2 pairs of products lie between a request and
                    // its use (requested right in front of its use, as the compiler orders them when left alone, every
                    // pair of products waits out the LDS latency)
                    const unsigned char *wa = ks + kRing < KS ? wb + kRing * 32 : wn + (kRing - KS) * 32;
                    wq[ks % kRing] = *reinterpret_cast<const uint4 *>(wa + ks * 32);
                    wq[(ks + 1) % kRing] = *reinterpret_cast<const uint4 *>(wa + ks * 32 + 32);
                    __builtin_amdgcn_sched_barrier(0);
                }
                acc = acc + acc_odd;
                // acc[4 vg + i] = out[m, n0 + 32 c + 8 vg + 4 half + i]
#pragma unroll
                for (int vg = 0; vg < 4; ++vg)
                    // (rows 8 .. 15 and 24 .. 31 keep the 8-byte halves of every 16-byte piece the other way round: rows
                    // are 144 bytes apart, so that rows r and r + 8, served together, would otherwise share their banks)
                    *reinterpret_cast<uint2 *>(tile + r * kTileRowB + (sub * 32 + 8 * vg + 4 * (half ^ ((r >> 3) & 1))) * 2) = make_uint2(
                        pack_bf16x2(acc[4 * vg], acc[4 * vg + 1]), pack_bf16x2(acc[4 * vg + 2], acc[4 * vg + 3]));
            }
            // The tile was written by this wave's other lanes: LDS works a wave's requests off in order, so all that
            // is needed is that the compiler keeps the order (a fence would also wait for the stores to memory).
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int pass = 0; pass < 4; ++pass) {
                const int row = pass * 8 + (lane >> 3), col = c0 * kProjChunk + (lane & 7) * 8;
                const u32x4 q = *reinterpret_cast<const u32x4 *>(tile + row * kTileRowB + (lane & 7) * 16);
                const u32x4 v = (pass & 1) ? u32x4{q.z, q.w, q.x, q.y} : q;
                const bool ok = m0 + row < M && col < ncols;
                const unsigned off = ((trow + (unsigned)row) * (unsigned)ldo + (unsigned)(n0 + col)) * 2u;
                __builtin_amdgcn_raw_buffer_store_b128(v, obuf, ok ? off : kBufferDropOffset, 0, 0);
            }
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
        }
    };
    // Two sets of row fragments: the next tile's rows are requested before this tile's products, because loads and
    // stores complete in order per wave -- requested after, they would wait for this tile's stores to reach memory.
    // (Tiles past M load the last row and store nothing, so that the loop has no exit in its middle.)
    Frag<__bf16> ua[KS], ub[KS];
    load_rows(0, ua);
#pragma unroll
    for (int t = 0; t < TILES; t += 2) {
        if (t + 1 < TILES) load_rows(t + 1, ub);
        tile_product(t, ua);
        if (t + 2 < TILES) load_rows(t + 2, ua);
        if (t + 1 < TILES) tile_product(t + 1, ub);
    }
}


// ------------------------------------------------------------------------------------------------------------------
// Gate + RMSNorm + out-projection in one pass: out[m, n] = sum_k yn[m, k] w[n, k] with
// yn[m, k] = v[m, k] rsqrt(mean_k v[m, k]^2 + eps) norm_w[k], v = y silu(z) -- the normalised row never reaches
// memory (it would be written by one kernel and read back by the next: two thirds of the bytes of a row's y and z).
// A row of the inner width K (128 or 256 channels) is exactly the MFMA's K axis, which a lane pair (r, r + 32) holds
// entirely in registers: the prologue forms a tile's v in float32, the pair's sum of squares and then fragments of
// bf16(yn), the only rounding in front of the product and the one block_post makes when it stores the row (with the norm's
// weights folded into w instead, which rounds the weights once more, the result's error against float64 was 2.88e-3 where
// it is 2.35e-3, at scales spread by 0.2 around one; 256 -> 256 in us, folded / here: 16 384 rows 17.5 / 16.7, 131 072 rows
// 42 / 45, 524 288 rows 176 / 176).  v takes the registers of the pieces of y and z it is formed from; the norm's weights are
// in LDS.  A workgroup takes all out_features (at most 256) columns, so that the prologue runs once per row: its rows of w fill
// 132 KB of LDS, and a wave's output tile covers 16 rows at a time to fit beside them.
// ------------------------------------------------------------------------------------------------------------------
constexpr int kPostProjMaxCols = 256;

template <int KS, int CH>  // K = 16 * KS inner channels, CH chunks of 32 output columns
__global__ __launch_bounds__(64 * kProjWaves) void block_post_proj_kernel(
    const __bf16 *__restrict__ y, const __bf16 *__restrict__ zxbcdt, const float *__restrict__ norm_w, float eps,
    const __bf16 *__restrict__ w, __bf16 *__restrict__ out, long long M, int N, int ld_z, int ldo, int tiles) {
    constexpr int K = 16 * KS, NTHR = 64 * kProjWaves, PPR = K / 8;  // 16-byte pieces per row of w
    constexpr int ROWB = K * 2 + 16;  // a staged row of w: 16 bytes of padding shift the banks from row to row
    constexpr int kTileRowB = 64 * 2 + 16;
    __shared__ __attribute__((aligned(16))) unsigned char wsm[CH * kProjChunk * ROWB];
    __shared__ __attribute__((aligned(16))) unsigned char otile[kProjWaves][16 * kTileRowB];
    __shared__ __attribute__((aligned(16))) float nw_s[K];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const long long row0 = (long long)blockIdx.x * tiles * (32LL * kProjWaves);  // tiles: 32-row tiles per wave, 1 .. kProjTiles
    const int r = lane & 31, half = lane >> 5;
    // this lane's K elements are 16 ks + 8 half .. + 7 for every K step
    auto tile_row0 = [&](int t) { return row0 + (long long)t * (32 * kProjWaves) + wave * 32; };
    // A tile's rows of y are requested one tile ahead (they are in flight during the products and stores of the tile
    // before); its rows of z only at the top of the tile: both sets a tile ahead would not fit the registers beside
    // the operand fragments, and the workgroup's other waves fill the SIMD during the wait.
    uint4 yq[KS], zq[KS];
    auto tile_row = [&](int t) { return min(tile_row0(t) + r, M - 1); };  // rows past M repeat the last row; never stored
    auto load_y = [&](int t) {
        const __bf16 *yr = y + (size_t)tile_row(t) * K + 8 * half;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) yq[ks] = *reinterpret_cast<const uint4 *>(yr + 16 * ks);
    };
    auto load_z = [&](int t) {
        const __bf16 *zr = zxbcdt + (size_t)tile_row(t) * ld_z + 8 * half;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) zq[ks] = *reinterpret_cast<const uint4 *>(zr + 16 * ks);
    };
    load_y(0);  // in flight while w is staged
    const float nw_q = norm_w[min(tid, K - 1)];
    {   // rows 0 .. 32 CH - 1 of w (rows past N repeat the last one: never stored)
        constexpr int PIECES = CH * kProjChunk * PPR;
        constexpr int FILL = (PIECES + NTHR - 1) / NTHR;
#pragma unroll 4
        for (int i = 0; i < FILL; ++i) {
            const int p = min(tid + i * NTHR, PIECES - 1);
            const int row = p / PPR, piece = p % PPR;
            *reinterpret_cast<uint4 *>(wsm + row * ROWB + piece * 16) =
                *reinterpret_cast<const uint4 *>(w + (size_t)min(row, N - 1) * K + piece * 8);
        }
    }
    if (tid < K) nw_s[tid] = nw_q;
    __syncthreads();
    unsigned char *tile = otile[wave];
    const __amdgpu_buffer_rsrc_t obuf = make_buffer(out + (size_t)row0 * ldo, (unsigned)min((long long)tiles * 32 * kProjWaves, M - row0) * (unsigned)ldo * 2u);
    const float inv_k = 1.f / (float)K;
#pragma unroll 1
    for (int t = 0; t < tiles; ++t) {
        // ---- prologue: this tile's rows of y and z -> fragments of the normalised rows ----
        load_z(t);
        // (the row's squares: each eight channels' own sum, those of a half in order; block_post_proj_rows_kernel adds them up the
        // same way, so that a row's result is the same bits from either)
        float v[KS][8];
        float ss = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const Pack8<__bf16> yy{yq[ks]}, zz{zq[ks]};
            float piece = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                v[ks][i] = yy.get(i) * silu(zz.get(i));
                piece += v[ks][i] * v[ks][i];
            }
            ss += piece;
        }
        ss += __shfl_xor(ss, 32, 64);
        const float rstd = rsqrtf(ss * inv_k + eps);
        Frag<__bf16> uf[KS];
        int nw0 = 8 * half;
        asm volatile("" : "+v"(nw0));  // (read per tile: hoisted out of the loop the weights would take 128 registers)
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const float4 na = *reinterpret_cast<const float4 *>(nw_s + nw0 + 16 * ks);
            const float4 nb = *reinterpret_cast<const float4 *>(nw_s + nw0 + 16 * ks + 4);
            uint4 o;
            o.x = pack_bf16x2(v[ks][0] * rstd * na.x, v[ks][1] * rstd * na.y);
            o.y = pack_bf16x2(v[ks][2] * rstd * na.z, v[ks][3] * rstd * na.w);
            o.z = pack_bf16x2(v[ks][4] * rstd * nb.x, v[ks][5] * rstd * nb.y);
            o.w = pack_bf16x2(v[ks][6] * rstd * nb.z, v[ks][7] * rstd * nb.w);
            // (formed here: left alone, the compiler reads all of the weights ahead and forms the fragments behind the next
            // rows' requests, 91 spilled registers)
            asm volatile("" : "+v"(o.x), "+v"(o.y), "+v"(o.z), "+v"(o.w));
            uf[ks].v = __builtin_bit_cast(bf16x8, o);
        }
        // the next tile's rows of y: requested before this tile's products and stores (loads and stores complete in
        // order per wave: requested behind the stores they would wait for those to reach memory)
        if (t + 1 < tiles) load_y(t + 1);
        else {  // (named here, the pieces need no registers from their use above to this point)
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) yq[ks] = make_uint4(0, 0, 0, 0);
        }
        const unsigned trow = (unsigned)(t * (32 * kProjWaves) + wave * 32);
        const long long m0 = tile_row0(t);
#pragma unroll
        for (int c0 = 0; c0 < CH; c0 += 2) {
            f32x16 acc[2];
#pragma unroll
            for (int sub = 0; sub < 2; ++sub) {
                const int c = c0 + sub;
                acc[sub] = f32x16{0};
                if (c >= CH) break;
                const unsigned char *wb = wsm + (c * kProjChunk + r) * ROWB + half * 16;
                f32x16 acc_odd = {0};
#pragma unroll
                for (int ks = 0; ks < KS; ks += 2) {
                    Frag<__bf16> wf0, wf1;
                    wf0.v = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(wb + ks * 32));
                    wf1.v = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(wb + ks * 32 + 32));
                    acc[sub] = mma32(wf0, uf[ks], acc[sub]);
                    acc_odd = mma32(wf1, uf[ks + 1], acc_odd);
                }
                acc[sub] = acc[sub] + acc_odd;
            }
            // acc[sub][4 vg + i] = out[m0 + r, 32 (c0 + sub) + 8 vg + 4 half + i]; the wave's tile holds 16 rows, so
            // the rows go out in two halves (rows r < 16, then the others)
#pragma unroll
            for (int rh = 0; rh < 2; ++rh) {
                if ((r >> 4) == rh) {
#pragma unroll
                    for (int sub = 0; sub < 2; ++sub) {
#pragma unroll
                        for (int vg = 0; vg < 4; ++vg)
                            *reinterpret_cast<uint2 *>(tile + (r & 15) * kTileRowB + (sub * 32 + 8 * vg + 4 * (half ^ ((r >> 3) & 1))) * 2) = make_uint2(
                                pack_bf16x2(acc[sub][4 * vg], acc[sub][4 * vg + 1]), pack_bf16x2(acc[sub][4 * vg + 2], acc[sub][4 * vg + 3]));
                    }
                }
                asm volatile("" ::: "memory");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int pass = 0; pass < 2; ++pass) {
                    const int trw = pass * 8 + (lane >> 3), row = rh * 16 + trw, col = c0 * kProjChunk + (lane & 7) * 8;
                    const u32x4 q = *reinterpret_cast<const u32x4 *>(tile + trw * kTileRowB + (lane & 7) * 16);
                    const u32x4 v = (pass & 1) ? u32x4{q.z, q.w, q.x, q.y} : q;  // (halves swapped in rows 8 .. 15)
                    const bool ok = m0 + row < M && col < N;
                    const unsigned off = ((trow + (unsigned)row) * (unsigned)ldo + (unsigned)col) * 2u;
                    __builtin_amdgcn_raw_buffer_store_b128(v, obuf, ok ? off : kBufferDropOffset, 0, 0);
                }
                asm volatile("" ::: "memory");
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
}

// The same for few rows.  There the kernel above leaves the gate to few waves -- one gates 32 rows, 128 silu per lane, six
// microseconds of vector instructions -- and each block of columns gates its rows anew.  Here a workgroup owns 32 RT rows and all
// columns: its eight waves gate four RT rows each (sixteen lanes a row), put the rows into
// LDS, and then multiply 32 columns each, their weights requested straight into operand fragments ahead of the gate.  Every
// workgroup reads all of w (128 KB at 256 x 256) from its XCD's L2, which is what bounds it and why many rows are better off above.
// 256 -> 256 in us, the kernel above (with its columns cut in up to eight blocks below 32 768 rows) / 32 rows per workgroup / 64:
// 600 rows 13.8 / 6.8 / 8.3, 8 192 14.7 / 7.5 / 8.9, 16 384 15.8 / 12.2 / 9.6, 32 768 18.7 / 22.6 / 16.4, 49 152 22.3 / 32 / 24.6;
// 128 channels: 600 rows 8.5 / 4.7 / 5.4, 16 384 10.1 / 8.2 / 6.8, 32 768 12.2 / 13.9 / 10.8, 49 152 14.8 / 20 / 15.1.
template <int KS, int RT>
__global__ __launch_bounds__(64 * kProjWaves) void block_post_proj_rows_kernel(
    const __bf16 *__restrict__ y, const __bf16 *__restrict__ zxbcdt, const float *__restrict__ norm_w, float eps,
    const __bf16 *__restrict__ w, __bf16 *__restrict__ out, long long M, int N, int ld_z, int ldo) {
    constexpr int K = 16 * KS, PPL = KS / 8;  // 16-byte pieces of a row per lane
    constexpr int ROWB = K * 2 + 16;          // bytes of a staged row: 16 bytes of padding shift the banks
    __shared__ __attribute__((aligned(16))) unsigned char rows_s[RT * 32 * ROWB];
    __shared__ __attribute__((aligned(16))) float squares[32][K / 8 + 4];  // of a row's pieces of eight channels
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int r = lane & 31, half = lane >> 5;
    const long long row0 = (long long)blockIdx.x * (32 * RT);
    const int lrow = tid >> 4, l16 = tid & 15;
    Pack8<__bf16> yv[RT][PPL], zv[RT][PPL];
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const size_t row = (size_t)min(row0 + t * 32 + lrow, M - 1);  // rows past M repeat the last row; never stored
#pragma unroll
        for (int p = 0; p < PPL; ++p) {
            yv[t][p] = Pack8<__bf16>::load(y + row * K + (p * 16 + l16) * 8);
            zv[t][p] = Pack8<__bf16>::load(zxbcdt + row * ld_z + (p * 16 + l16) * 8);
        }
    }
    float4 na[PPL], nb[PPL];
#pragma unroll
    for (int p = 0; p < PPL; ++p) {
        na[p] = *reinterpret_cast<const float4 *>(norm_w + (p * 16 + l16) * 8);
        nb[p] = *reinterpret_cast<const float4 *>(norm_w + (p * 16 + l16) * 8 + 4);
    }
    Frag<__bf16> wf[KS];  // this wave's 32 columns (columns past N repeat the last one; never stored)
    const __bf16 *wr = w + (size_t)min(wave * 32 + r, N - 1) * K + 8 * half;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) wf[ks].v = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(wr + 16 * ks));
    __builtin_amdgcn_sched_barrier(0);  // (all of it in flight before the first is waited for)
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        float v[PPL][8];
#pragma unroll
        for (int p = 0; p < PPL; ++p) {
            float piece = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                v[p][i] = yv[t][p].get(i) * silu(zv[t][p].get(i));
                piece += v[p][i] * v[p][i];
            }
            squares[lrow][p * 16 + l16] = piece;
        }
        // (a row's lanes belong to one wave, whose LDS requests are worked off in order: only the compiler has to keep it)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
        float s0 = 0.f, s1 = 0.f;  // pieces of even and of odd index, as the two halves of the kernel above hold them
#pragma unroll
        for (int q = 0; q < K / 8; q += 4) {
            const float4 p4 = *reinterpret_cast<const float4 *>(&squares[lrow][q]);
            s0 += p4.x;
            s1 += p4.y;
            s0 += p4.z;
            s1 += p4.w;
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
        const float rstd = rsqrtf((s0 + s1) * (1.f / (float)K) + eps);
#pragma unroll
        for (int p = 0; p < PPL; ++p) {
            uint4 o;
            o.x = pack_bf16x2(v[p][0] * rstd * na[p].x, v[p][1] * rstd * na[p].y);
            o.y = pack_bf16x2(v[p][2] * rstd * na[p].z, v[p][3] * rstd * na[p].w);
            o.z = pack_bf16x2(v[p][4] * rstd * nb[p].x, v[p][5] * rstd * nb[p].y);
            o.w = pack_bf16x2(v[p][6] * rstd * nb[p].z, v[p][7] * rstd * nb[p].w);
            *reinterpret_cast<uint4 *>(rows_s + (t * 32 + lrow) * ROWB + (p * 16 + l16) * 16) = o;
        }
    }
    block_sync_lds();
    const int n0 = wave * 32;
    if (n0 >= N) return;
#pragma unroll
    for (int t = 0; t < RT; ++t) {
        const unsigned char *ur = rows_s + (t * 32 + r) * ROWB + half * 16;
        f32x16 acc = {0}, acc_odd = {0};
#pragma unroll
        for (int ks = 0; ks < KS; ks += 2) {
            Frag<__bf16> u0, u1;
            u0.v = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(ur + ks * 32));
            u1.v = __builtin_bit_cast(bf16x8, *reinterpret_cast<const uint4 *>(ur + ks * 32 + 32));
            acc = mma32(wf[ks], u0, acc);
            acc_odd = mma32(wf[ks + 1], u1, acc_odd);
        }
        float o[16];
#pragma unroll
        for (int i = 0; i < 16; ++i) o[i] = acc[i] + acc_odd[i];
        const long long row = row0 + t * 32 + r;
        store_column<__bf16>(out + (size_t)min(row, M - 1) * ldo + n0, o, half, N - n0, row < M);
    }
}

}  // namespace

bool block_proj_supported(long long rows, int in_features, int out_features) {
    return rows > 0 && (in_features == 128 || in_features == 256) && out_features > 0 && out_features % 8 == 0;
}

// Column blocks: equal blocks of at most kProjBlockCols columns (a multiple of 8) -- or, where that takes no more
// workgroups, blocks of 128 with the last one taking the rest (up to kProjBlockCols): every block then starts on a
// multiple of 64 columns, so that with rows a multiple of 128 bytes apart every 128-byte piece a wave writes is one
// whole line of the memory system (648 columns: 4 x 128 + 136 instead of 4 x 136 + 104, 21 column chunks instead of 25).
static void proj_col_blocks(int out_features, int *col_blocks, int *block_cols) {
    const int equal = (out_features + kProjBlockCols - 1) / kProjBlockCols;
    const int by128 = out_features <= kProjBlockCols ? 1 : (out_features - kProjBlockCols + 127) / 128 + 1;
    if (by128 == equal) {
        *col_blocks = by128;
        *block_cols = by128 == 1 ? (out_features + 7) / 8 * 8 : 128;
    } else {
        *col_blocks = equal;
        *block_cols = ((out_features + equal - 1) / equal + 7) / 8 * 8;
    }
}

// How the product is cut over workgroups: the columns in blocks, the rows in ranges of 256 times 1, 2, 4 or 8 tiles per
// wave.  A compute unit holds one workgroup, so what counts is rounds of workgroups times the time of one.  Long
// ranges pay the fill of w once for many rows, but at 16 384 rows (256 -> 648) eight tiles leave 40 workgroups for 256
// compute units: 40.5 us, 15.1 with two tiles on blocks of 96 columns.  A workgroup is priced at kFixed + kPerChunk per 32
// columns, for each width of u and number of tiles; the prices (in about us, but no workgroup's times) are those whose choice
// came out best over 242 pairs of rows (300 .. 524 288) and columns (64 .. 1 120) with every cut timed; on 90 further pairs the
// choice is 1.4 % (256) and 1.9 % (128) slower than the best cut on average, and than eight tiles on the widest blocks by 7 %
// at most.  Of two cuts at one price the longer range is taken.  Rounds are counted per XCD: counted over the whole chip, 67 423 rows (256 -> 648) took
// one tile and a round more on one XCD in eight (71 us, 45.5 with eight tiles, as chosen now; 50 000 rows 45.7, 33.0).
static hipError_t proj_split(long long rows, int in_features, int out_features, int *col_blocks, int *block_cols, int *tiles) {
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = device_cu_count(dev, &cus);
    if (e != hipSuccess) return e;
    constexpr double kFixed[2][4] = {{4.5, 7.82, 17.79, 38.65}, {5.95, 6.45, 17.61, 24.59}};  // in_features 128, 256
    constexpr double kPerChunk[2][4] = {{0.5, 1.41, 1.4, 1.8}, {0.21, 1.72, 0.68, 2.34}};
    constexpr double kSame = 1e-9;
    const int wide = in_features == 256 ? 1 : 0;
    double best = 0.;
    *tiles = 0;
    for (int cut = 0; cut < 5; ++cut) {
        int cb, bc;
        proj_col_blocks(out_features, &cb, &bc);
        if (cut > 0) {  // blocks of 128, 96, 64, 32 columns: more workgroups where rows are few
            const int narrow = kProjChunk * (5 - cut);
            if (narrow >= bc) continue;
            bc = narrow;
            cb = (out_features + bc - 1) / bc;
        }
        const int chunks = (std::max(bc, out_features - (cb - 1) * bc) + kProjChunk - 1) / kProjChunk;
        for (int k = 0; k < 4; ++k) {
            const long long per_group = 32LL * kProjWaves << k;
            // (the column blocks of a range of rows stay on one of the 8 XCDs: its workgroups against its compute units)
            const long long per_xcd = ((rows + per_group - 1) / per_group + 7) / 8 * cb;
            const int xcd_cus = std::max(1, cus / 8);
            const double cost = (double)((per_xcd + xcd_cus - 1) / xcd_cus) * (kFixed[wide][k] + kPerChunk[wide][k] * chunks);
            if (*tiles == 0 || cost < best - kSame || (cost < best + kSame && (1 << k) > *tiles)) {
                best = cost;
                *col_blocks = cb;
                *block_cols = bc;
                *tiles = 1 << k;
            }
        }
    }
    return hipSuccess;
}

hipError_t launch_block_proj(long long rows, int in_features, int out_features, int out_ld, const void *u, const void *w,
                             void *out, hipStream_t st) {
    if (!block_proj_supported(rows, in_features, out_features) || out_ld < out_features || out_ld % 8 != 0)
        return hipErrorInvalidValue;
    int col_blocks, block_cols, tiles;
    hipError_t e = proj_split(rows, in_features, out_features, &col_blocks, &block_cols, &tiles);
    if (e != hipSuccess) return e;
    const long long rows_per_group = 32LL * kProjWaves * tiles;
    const long long groups = ((rows + rows_per_group - 1) / rows_per_group + 7) / 8 * 8 * col_blocks;
    if (groups > 0x7fffffffLL || out_features - (col_blocks - 1) * block_cols > kProjBlockCols ||
        out_features - (col_blocks - 1) * block_cols <= 0)
        return hipErrorInvalidValue;
    const dim3 grid((unsigned)groups), block(64 * kProjWaves);
    const __bf16 *uu = static_cast<const __bf16 *>(u), *ww = static_cast<const __bf16 *>(w);
    __bf16 *oo = static_cast<__bf16 *>(out);
    // the chunks of 32 columns the widest block takes
    const int widest = std::max(block_cols, out_features - (col_blocks - 1) * block_cols);
    const int ch = (widest + kProjChunk - 1) / kProjChunk;
#define SSD_PROJ_CASE(KSv, CHv, Tv)                                                                                    \
    if (in_features == 16 * KSv && ch == CHv && tiles == Tv) {                                                         \
        block_proj_kernel<KSv, CHv, Tv><<<grid, block, 0, st>>>(uu, ww, oo, rows, out_features, out_ld, col_blocks, block_cols); \
        return hipGetLastError();                                                                                      \
    }
#define SSD_PROJ_TILES(KSv, CHv) SSD_PROJ_CASE(KSv, CHv, 1) SSD_PROJ_CASE(KSv, CHv, 2) SSD_PROJ_CASE(KSv, CHv, 4) SSD_PROJ_CASE(KSv, CHv, 8)
    SSD_PROJ_TILES(8, 1) SSD_PROJ_TILES(8, 2) SSD_PROJ_TILES(8, 3) SSD_PROJ_TILES(8, 4) SSD_PROJ_TILES(8, 5)
    SSD_PROJ_TILES(16, 1) SSD_PROJ_TILES(16, 2) SSD_PROJ_TILES(16, 3) SSD_PROJ_TILES(16, 4) SSD_PROJ_TILES(16, 5)
#undef SSD_PROJ_TILES
#undef SSD_PROJ_CASE
    return hipErrorInvalidValue;
}

bool block_post_proj_supported(const BlockShape &s, int out_features) {
    const int DI = s.H * s.P;
    return (DI == 128 || DI == 256) && out_features > 0 && out_features <= kPostProjMaxCols && out_features % 8 == 0;
}

// out [B*L, out_features] (row stride out_ld) = rmsnorm(y silu(z)) norm_w . w^T; y [B*L, H*P] bf16, z the first H*P
// channels of zxbcdt's rows (stride s.ld), w [out_features, H*P] bf16.
hipError_t launch_block_post_proj(const BlockShape &s, const void *y, const void *zxbcdt, const float *norm_w, float eps,
                                  const void *w, int out_features, int out_ld, void *out, hipStream_t st) {
    if (!block_post_proj_supported(s, out_features) || out_ld < out_features || out_ld % 8 != 0) return hipErrorInvalidValue;
    const int K = s.H * s.P;
    const long long rows = (long long)s.B * s.L;
    int dev = 0, cus = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e == hipSuccess) e = device_cu_count(dev, &cus);
    if (e != hipSuccess) return e;
    const __bf16 *yy = static_cast<const __bf16 *>(y), *zz = static_cast<const __bf16 *>(zxbcdt), *ww = static_cast<const __bf16 *>(w);
    __bf16 *oo = static_cast<__bf16 *>(out);
    const dim3 block(64 * kProjWaves);
    // Few rows: a workgroup per 32 rows up to one round of workgroups, then per 64 up to two (above, at the line, in the comment
    // of the kernel: both sides).
    if (rows <= 128LL * cus) {
        const int rt = rows <= 32LL * cus ? 1 : 2;
        const dim3 grid((unsigned)((rows + 32 * rt - 1) / (32 * rt)));
#define SSD_POST_PROJ_ROWS(KSv, RTv)                                                                                                     \
    if (K == 16 * KSv && rt == RTv) {                                                                                                    \
        block_post_proj_rows_kernel<KSv, RTv><<<grid, block, 0, st>>>(yy, zz, norm_w, eps, ww, oo, rows, out_features, s.ld, out_ld);    \
        return hipGetLastError();                                                                                                        \
    }
        SSD_POST_PROJ_ROWS(8, 1) SSD_POST_PROJ_ROWS(8, 2) SSD_POST_PROJ_ROWS(16, 1) SSD_POST_PROJ_ROWS(16, 2)
#undef SSD_POST_PROJ_ROWS
    }
    // rows per workgroup: as many tiles of 32 rows per wave, up to kProjTiles, as make one round of workgroups (each
    // workgroup stages all of w, as much as 256 of its rows; rounded down instead, 67 423 rows were two rounds of one tile:
    // 44 us against 36 with two, 180 001 rows 79 against 61)
    const long long per_tile = 32LL * kProjWaves;
    const int tiles = (int)std::max<long long>(1, std::min<long long>(kProjTiles, (rows + per_tile * cus - 1) / (per_tile * cus)));
    const long long rows_per_group = per_tile * tiles;
    const long long groups = (rows + rows_per_group - 1) / rows_per_group;
    if (groups > 0x7fffffffLL || (unsigned long long)rows_per_group * out_ld * 2 > 0x7fffffffULL) return hipErrorInvalidValue;
    const dim3 grid((unsigned)groups);
    const int ch = (out_features + kProjChunk - 1) / kProjChunk;
#define SSD_POST_PROJ_CASE(KSv, CHv)                                                                                   \
    if (K == 16 * KSv && ch == CHv) {                                                                                  \
        block_post_proj_kernel<KSv, CHv><<<grid, block, 0, st>>>(yy, zz, norm_w, eps, ww, oo, rows, out_features, s.ld, out_ld, tiles); \
        return hipGetLastError();                                                                                      \
    }
    SSD_POST_PROJ_CASE(8, 1) SSD_POST_PROJ_CASE(8, 2) SSD_POST_PROJ_CASE(8, 3) SSD_POST_PROJ_CASE(8, 4)
    SSD_POST_PROJ_CASE(8, 5) SSD_POST_PROJ_CASE(8, 6) SSD_POST_PROJ_CASE(8, 7) SSD_POST_PROJ_CASE(8, 8)
    SSD_POST_PROJ_CASE(16, 1) SSD_POST_PROJ_CASE(16, 2) SSD_POST_PROJ_CASE(16, 3) SSD_POST_PROJ_CASE(16, 4)
    SSD_POST_PROJ_CASE(16, 5) SSD_POST_PROJ_CASE(16, 6) SSD_POST_PROJ_CASE(16, 7) SSD_POST_PROJ_CASE(16, 8)
#undef SSD_POST_PROJ_CASE
    return hipErrorInvalidValue;
}

}  // namespace ssd
