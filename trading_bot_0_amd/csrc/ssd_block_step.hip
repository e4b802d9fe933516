// One timestep of the whole Mamba-2 block for a few streams, as ONE launch (gfx950):
//   in-projection (a matrix-vector product per stream) -> conv window update + SiLU, softplus(dt) -> SSM state
//   update and readout -> gate + RMSNorm -> out-projection.
// At a handful of streams the step's cost is the host's time to issue its launches (five kernels and two library
// products take about 0.1 ms of issue time for 0.01 ms of work); here a workgroup of 1 024 threads owns one stream (or two)
// and walks the five stages with workgroup barriers between them, every intermediate in LDS.  The two weight
// matrices come through L2 (0.33 MB and 0.13 MB in bf16 at 256 channels: every workgroup reads them whole), which is
// what bounds the launch.
//
// Rounding: every tensor the stage kernels would write to memory in the activation type (zxbcdt, x, B, C, dt, y, the
// normalised row) is rounded to that type here at the same point, so that a stream advanced by this kernel and one
// advanced by the stage kernels see the same numbers up to the order of the float32 sums.
#include "ssd_block_common.h"

namespace ssd {

namespace {

constexpr int kStepThreads = 1024;

template <typename T> __device__ inline float round_to(float v) { return (float)(T)v; }

// rows [0, rows) of w [rows, K] (K-contiguous) times vec (K floats in LDS) -> out (LDS floats), one row per group of
// K/8 lanes, eight rows of a group in flight at once
template <typename T, int K>
__device__ inline void gemv_rows(const T *__restrict__ w, int rows, const float *vec, float *out, int tid, bool round_out) {
    constexpr int G = K / 8;                       // lanes per row: 16 bytes (bf16) or 32 bytes (float) each
    constexpr int NG = kStepThreads / G;           // rows per pass of the workgroup
    constexpr int UN = 8;
    const int gl = tid % G, grp = tid / G;
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = vec[gl * 8 + i];
    for (int r0 = grp; r0 < rows; r0 += NG * UN) {
        Pack8<T> q[UN];
#pragma unroll
        for (int u = 0; u < UN; ++u) q[u] = Pack8<T>::load(w + (size_t)min(r0 + u * NG, rows - 1) * K + gl * 8);
#pragma unroll
        for (int u = 0; u < UN; ++u) {
            float a = 0.f;
#pragma unroll
            for (int i = 0; i < 8; ++i) a += q[u].get(i) * v[i];
#pragma unroll
            for (int m = G / 2; m >= 1; m >>= 1) a += __shfl_xor(a, m, 64);
            const int row = r0 + u * NG;
            if (gl == 0 && row < rows) out[row] = round_out ? round_to<T>(a) : a;
        }
    }
}

// Any state width, any number of rows of w_in (a 64-wide state and up to kStepMaxRows rows: block_step_overlap_kernel below).
template <typename T, int DM, int DI, int DCONV>
__global__ __launch_bounds__(kStepThreads) void block_step_kernel(
    const T *__restrict__ u, const T *__restrict__ w_in, const float *__restrict__ conv_w, const float *__restrict__ conv_b,
    const float *__restrict__ dt_bias, const float *__restrict__ A, const float *__restrict__ D,
    const float *__restrict__ norm_w, float eps, const T *__restrict__ w_out, T *conv_state, float *ssm_state,
    T *__restrict__ out, BlockShape s) {
    const int tid = threadIdx.x, b = blockIdx.x;
    const int H = s.H, P = s.P, N = s.N, GN = s.G * s.N, C = DI + 2 * GN, E = 2 * DI + 2 * GN + H;
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float *u_s = sm;              // [DM]
    float *zx_s = u_s + DM;       // [E]    z | x | B | C | dt_raw, as the in-projection leaves them
    float *act_s = zx_s + E;      // [C]    x | B | C after conv + SiLU
    float *dt_s = act_s + C;      // [H]
    float *y_s = dt_s + ((H + 3) & ~3);  // [DI]   y, then the gated, normalised row
    float *red_s = y_s + DI;      // [kStepThreads / 64]

    for (int i = tid; i < DM; i += kStepThreads) u_s[i] = (float)u[(size_t)b * DM + i];
    __syncthreads();
    gemv_rows<T, DM>(w_in, E, u_s, zx_s, tid, true);
    __syncthreads();

    // conv window: the stream's last DCONV-1 inputs, then this step's; the state moves up by one row
    for (int c = tid; c < C; c += kStepThreads) {
        T *cs = conv_state + (size_t)b * (DCONV - 1) * C + c;
        float win[DCONV];
#pragma unroll
        for (int k = 0; k < DCONV - 1; ++k) win[k] = (float)cs[(size_t)k * C];
        win[DCONV - 1] = zx_s[DI + c];
        float a = conv_b[c];
#pragma unroll
        for (int k = 0; k < DCONV; ++k) a += conv_w[(size_t)c * DCONV + k] * win[k];
        act_s[c] = round_to<T>(silu(a));
#pragma unroll
        for (int k = 0; k < DCONV - 1; ++k) cs[(size_t)k * C] = (T)win[k + 1];
    }
    for (int h = tid; h < H; h += kStepThreads) dt_s[h] = round_to<T>(softplus(zx_s[DI + C + h] + dt_bias[h]));
    __syncthreads();

    // SSM step: four lanes per (head, row p), a quarter of the row's N columns each (float4 pieces, strided so that
    // the four lanes of a row read 64 consecutive bytes at a time)
    {
        const int HG = H / s.G, NQ = N / 4;  // float4 pieces per row
        for (int row = tid / 4; row < H * P; row += kStepThreads / 4) {
            const int h = row / P, q = tid & 3;
            const int g = h / HG;
            const float dtv = dt_s[h], xv = act_s[row];
            const float decay = __expf(dtv * A[h]), dx = dtv * xv;
            float4 *st = reinterpret_cast<float4 *>(ssm_state + ((size_t)b * H * P + row) * N);
            const float *Bv = act_s + DI + g * N, *Cv = act_s + DI + GN + g * N;
            float acc = 0.f;
            for (int j = q; j < NQ; j += 4) {
                float4 hv = st[j];
                const float4 bb = *reinterpret_cast<const float4 *>(Bv + 4 * j), cc = *reinterpret_cast<const float4 *>(Cv + 4 * j);
                hv.x = decay * hv.x + dx * bb.x;
                hv.y = decay * hv.y + dx * bb.y;
                hv.z = decay * hv.z + dx * bb.z;
                hv.w = decay * hv.w + dx * bb.w;
                acc += hv.x * cc.x + hv.y * cc.y + hv.z * cc.z + hv.w * cc.w;
                st[j] = hv;
            }
            acc += __shfl_xor(acc, 1, 64);
            acc += __shfl_xor(acc, 2, 64);
            if (q == 0) y_s[row] = round_to<T>(acc + (D != nullptr ? D[h] : 0.f) * xv);
        }
    }
    __syncthreads();

    // gate + RMSNorm over the DI channels
    {
        float ss = 0.f;
        for (int c = tid; c < DI; c += kStepThreads) {
            const float v = y_s[c] * silu(zx_s[c]);
            y_s[c] = v;
            ss += v * v;
        }
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1) ss += __shfl_xor(ss, m, 64);
        if ((tid & 63) == 0) red_s[tid >> 6] = ss;
        __syncthreads();
        float tot = 0.f;
        for (int i = 0; i < kStepThreads / 64; ++i) tot += red_s[i];
        const float scale = rsqrtf(tot / (float)DI + eps);
        for (int c = tid; c < DI; c += kStepThreads) y_s[c] = round_to<T>(y_s[c] * scale * norm_w[c]);
    }
    __syncthreads();
    gemv_rows<T, DI>(w_out, DM, y_s, zx_s, tid, false);
    __syncthreads();
    for (int i = tid; i < DM; i += kStepThreads) out[(size_t)b * DM + i] = (T)zx_s[i];
}

// The same step with its trips to memory overlapped and its vector work cut, for a 64-wide state and at most kStepMaxRows
// rows of w_in.  One compute unit per stream forms half a million multiply-adds and loads 0.46 MB (bf16) behind a chain of
// barriers; the launch was bound by the first and by the chain.
// * A thread asks for what it can hold ahead of its use: two rounds of weights at once, a further round into the registers of
//   the one just used, its channel's conv window and filter and its piece of the state ahead of the last round's sums, w_out's
//   rows behind them; the barriers wait for LDS only.  The round count is a compile-time constant and rounds past the
//   last row read that row again: behind a branch the compiler would wait for everything outstanding.
// * bf16 weights are multiplied two at a time as they lie in the register (exact products, float32 sums), not unpacked.
// * A round's rows are summed over their lanes by halves: a lane keeps half of its rows at each exchange, 4 + 2 + 1 + 1 + 1
//   exchanges for eight rows instead of 40.
// * Gate and norm need no pass of their own: the sum of squares is taken where y is formed, the scale applied where the
//   out-projection reads the row.
// * With more streams than compute units a workgroup takes two (SPW), which use the same weights.
// 256 channels, back to back, in us at 4 / 256 / 512 / 1 024 streams: bf16 15.2 / 20.5 / 37.5 / 73.8 -> 13.8 / 17.5 / 21.7 /
// 42.2, float32 16.4 / 22.7 / 42.2 / 79.4 -> 13.5 / 18.5 / 25 / 50.  As 16x16x32 matrix products, whose operand form reads 16
// rows at a time, 17.5 / 20.1 / 24.1 / 44.7 in bf16.  What bounds it at few streams is one compute unit's rate of loading the
// weights from L2; at 512 the state's traffic (67 MB, 13 us) and the weights' (118 MB from L2) together.
constexpr int kStepMaxRows = 768;
// rows a thread has in flight per round (two streams' states leave no registers for more than four)
template <typename T, int SPW> constexpr int kStepUnroll = sizeof(T) == 2 && SPW == 1 ? 8 : 4;

// a thread's eight elements of a vector, in the form its piece of a row of w is multiplied with
template <typename T> struct Vec8;
template <> struct Vec8<float> {
    float v[8];
    __device__ inline void set(const float (&a)[8]) {
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = a[i];
    }
    __device__ inline float dot(const Pack8<float> &q) const {
        float a = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) a += q.get(i) * v[i];
        return a;
    }
};
template <> struct Vec8<__bf16> {
    unsigned v[4];
    __device__ inline void set(const float (&a)[8]) {  // (values that are bf16 already)
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = pack_bf16x2(a[2 * i], a[2 * i + 1]);
    }
    __device__ inline float dot(const Pack8<__bf16> &q) const {
        typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
        float a = 0.f;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            a = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, (&q.u.x)[i]), __builtin_bit_cast(bf16x2, v[i]), a, false);
        return a;
    }
};

template <typename T, int DM, int DI, int DCONV, int SPW>
__global__ __launch_bounds__(kStepThreads) void block_step_overlap_kernel(
    const T *__restrict__ u, const T *__restrict__ w_in, const float *__restrict__ conv_w, const float *__restrict__ conv_b,
    const float *__restrict__ dt_bias, const float *__restrict__ A, const float *__restrict__ D,
    const float *__restrict__ norm_w, float eps, const T *__restrict__ w_out, T *__restrict__ conv_state,
    float *__restrict__ ssm_state, T *__restrict__ out, BlockShape s) {
    constexpr int N = 64, UN = kStepUnroll<T, SPW>, WAVES = kStepThreads / 64;
    constexpr int ROWS_IN = kStepThreads / (DM / 8) * UN, ROWS_OUT = kStepThreads / (DI / 8) * UN;  // per round
    constexpr int R_IN = (kStepMaxRows + ROWS_IN - 1) / ROWS_IN, R_OUT = (DM + ROWS_OUT - 1) / ROWS_OUT;
    static_assert(SPW * DM <= kStepThreads && SPW * DI <= kStepThreads && R_IN >= 2, "an element of u and of y per thread");
    const int tid = threadIdx.x;
    const int b0 = blockIdx.x * SPW;
    const int H = s.H, P = s.P, GN = s.G * N, C = DI + 2 * GN, E = 2 * DI + 2 * GN + H, E4 = (E + 3) & ~3;
    extern __shared__ __attribute__((aligned(16))) float sm[];
    float *u_s = sm;                    // [SPW][DM]
    float *zx_s = u_s + SPW * DM;       // [SPW][E4]   z | x | B | C | dt_raw, as the in-projection leaves them
    float *act_s = zx_s + SPW * E4;     // [SPW][C]    x | B | C after conv + SiLU
    float *y_s = act_s + SPW * C;       // [SPW][DI]   y * silu(z)
    float *red_s = y_s + SPW * DI;      // [SPW][WAVES]
    float *dt_s = red_s + SPW * WAVES;  // [SPW][H]
    auto stream_of = [&](int k) { return min(b0 + k, s.B - 1); };  // (a stream past the last repeats it and stores nothing)

    const int uk = min(tid / DM, SPW - 1);
    const float u_q = (float)u[(size_t)stream_of(uk) * DM + tid % DM];
    // round r: rows r0 + i * NG of w_in, behind its rounds those of w_out; K / 8 lanes per row
    Pack8<T> q[2][UN];
    auto load_round = [&](int r) {
        const bool in = r < R_IN;
        const int K = in ? DM : DI, G = K / 8, NG = kStepThreads / G;
        const unsigned last = (unsigned)(in ? E : DM) - 1u;
        const T *w = in ? w_in : w_out;
        // (unsigned 32-bit offsets from a uniform pointer: one register per address)
        const unsigned r0 = (unsigned)((in ? r : r - R_IN) * NG * UN) + (unsigned)tid / G, col = ((unsigned)tid % G) * 8u;
#pragma unroll
        for (int i = 0; i < UN; ++i) q[r & 1][i] = Pack8<T>::load(w + (min(r0 + i * NG, last) * (unsigned)K + col));
    };
    // the round's rows times v; `put(row, sum)` by one lane per row
    auto dot_round = [&](int r, const Vec8<T> &v, auto put) {
        const bool in = r < R_IN;
        const int K = in ? DM : DI, G = K / 8, NG = kStepThreads / G, rows = in ? E : DM;
        float a[UN];
#pragma unroll
        for (int i = 0; i < UN; ++i) a[i] = v.dot(q[r & 1][i]);
        int cnt = UN, mine = 0, rest = 0;  // this lane's row of the round; lanes that differ in `rest` only hold the same sum
#pragma unroll
        for (int m = G / 2; m >= 1; m >>= 1) {
            const bool up = (tid & m) != 0;
            if (cnt > 1) {
                cnt >>= 1;
#pragma unroll
                for (int i = 0; i < cnt; ++i) {
                    const float keep = up ? a[i + cnt] : a[i], give = up ? a[i] : a[i + cnt];
                    a[i] = keep + __shfl_xor(give, m, 64);
                }
                mine += up ? cnt : 0;
            } else {
                a[0] += __shfl_xor(a[0], m, 64);
                rest |= m;
            }
        }
        const int row = (in ? r : r - R_IN) * NG * UN + tid / G + mine * NG;
        if ((tid & rest) == 0 && row < rows) put(row, a[0]);
    };
    load_round(0);
    // the conv window, filter and bias of this thread's channel (the launcher keeps SPW C within the threads)
    const int ck = min(tid / C, SPW - 1), ch = tid / C < SPW ? tid % C : C - 1;
    T *cs = conv_state + (size_t)stream_of(ck) * (DCONV - 1) * C;
    T win[DCONV - 1];
    float cw[DCONV], cb;
    load_round(1);

    if (tid < SPW * DM) u_s[tid] = u_q;
    block_sync_lds();
    auto vec_of = [&](const float *p) {
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = p[i];
        Vec8<T> v;
        v.set(f);
        return v;
    };
    Vec8<T> v[SPW];
#pragma unroll
    for (int k = 0; k < SPW; ++k) v[k] = vec_of(u_s + k * DM + (tid % (DM / 8)) * 8);
    // the state: four lanes per (head, row p), a quarter of the row each
    const bool has_row = tid / 4 < DI;
    const int row = min(tid / 4, DI - 1), quarter = tid & 3, h = row / P;
    const unsigned st_off = (unsigned)row * N + quarter * 4u;
    float4 hv[SPW][N / 16];
    auto load_state = [&](int k) {
        const float *st = ssm_state + (size_t)stream_of(k) * DI * N;
#pragma unroll
        for (int j = 0; j < N / 16; ++j) hv[k][j] = *reinterpret_cast<const float4 *>(st + (st_off + 16u * j));
    };
#pragma unroll
    for (int r = 0; r < R_IN; ++r) {
#pragma unroll
        for (int k = 0; k < SPW; ++k) dot_round(r, v[k], [&](int o, float a) { zx_s[k * E4 + o] = round_to<T>(a); });
        if (r + 2 < R_IN) load_round(r + 2);
        if (r == R_IN - 2) {
#pragma unroll
            for (int k = 0; k < DCONV - 1; ++k) win[k] = cs[(unsigned)(k * C + ch)];
#pragma unroll
            for (int k = 0; k < DCONV; ++k) cw[k] = conv_w[(unsigned)(ch * DCONV + k)];
            cb = conv_b[ch];
        }
        if (r >= R_IN - 2 && r - (R_IN - 2) < SPW) load_state(r - (R_IN - 2));
        __builtin_amdgcn_sched_barrier(0);  // (the loads stay where they are)
    }
    load_round(R_IN);
    if (R_OUT > 1 && SPW == 1) load_round(R_IN + 1);
    const float Ah = A[h], Dh = D != nullptr ? D[h] : 0.f;
    block_sync_lds();

    if (tid < SPW * C) {
        const float now = zx_s[ck * E4 + DI + ch];
        float a = cb;
#pragma unroll
        for (int k = 0; k < DCONV - 1; ++k) a += cw[k] * (float)win[k];
        a += cw[DCONV - 1] * now;
        act_s[ck * C + ch] = round_to<T>(silu(a));
        if (b0 + ck < s.B) {
#pragma unroll
            for (int k = 0; k < DCONV - 1; ++k) cs[(unsigned)(k * C + ch)] = k + 1 < DCONV - 1 ? win[min(k + 1, DCONV - 2)] : (T)now;
        }
    }
    for (int i = tid - (kStepThreads - 64); i >= 0 && i < SPW * H; i += 64)
        dt_s[i] = round_to<T>(softplus(zx_s[(i / H) * E4 + DI + C + i % H] + dt_bias[i % H]));
    block_sync_lds();

    {
        const int g = h / (H / s.G);
#pragma unroll
        for (int k = 0; k < SPW; ++k) {
            float *st = ssm_state + (size_t)stream_of(k) * DI * N;
            const bool store = has_row && b0 + k < s.B;
            const float dtv = dt_s[k * H + h], xv = act_s[k * C + row];
            const float decay = __expf(dtv * Ah), dx = dtv * xv;
            const float *Bv = act_s + k * C + DI + g * N + 4 * quarter, *Cv = Bv + GN;
            float acc = 0.f;
#pragma unroll
            for (int j = 0; j < N / 16; ++j) {
                const float4 bb = *reinterpret_cast<const float4 *>(Bv + 16 * j), cc = *reinterpret_cast<const float4 *>(Cv + 16 * j);
                float4 t = hv[k][j];
                t.x = decay * t.x + dx * bb.x;
                t.y = decay * t.y + dx * bb.y;
                t.z = decay * t.z + dx * bb.z;
                t.w = decay * t.w + dx * bb.w;
                acc += t.x * cc.x + t.y * cc.y + t.z * cc.z + t.w * cc.w;
                if (store) *reinterpret_cast<float4 *>(st + (st_off + 16u * j)) = t;
            }
            acc += __shfl_xor(acc, 1, 64);
            acc += __shfl_xor(acc, 2, 64);
            const float vy = has_row ? round_to<T>(acc + Dh * xv) * silu(zx_s[k * E4 + row]) : 0.f;
            if (has_row && quarter == 0) y_s[k * DI + row] = vy;
            float ss = vy * vy;
#pragma unroll
            for (int m = 4; m <= 32; m <<= 1) ss += __shfl_xor(ss, m, 64);
            if ((tid & 63) == 0) red_s[k * WAVES + tid / 64] = ss;
        }
    }
    if (R_OUT > 1 && SPW > 1) load_round(R_IN + 1);  // (no registers for it beside two states)
    block_sync_lds();
#pragma unroll
    for (int k = 0; k < SPW; ++k) {
        float tot = 0.f;
#pragma unroll
        for (int i = 0; i < WAVES; ++i) tot += red_s[k * WAVES + i];
        const float scale = rsqrtf(tot / (float)DI + eps);
        const int c0 = (tid % (DI / 8)) * 8;
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = round_to<T>(y_s[k * DI + c0 + i] * scale * norm_w[c0 + i]);
        v[k].set(f);
    }
#pragma unroll
    for (int r = R_IN; r < R_IN + R_OUT; ++r) {
#pragma unroll
        for (int k = 0; k < SPW; ++k)
            dot_round(r, v[k], [&](int o, float a) {
                if (b0 + k < s.B) out[(size_t)(b0 + k) * DM + o] = (T)a;
            });
        if (r + 2 < R_IN + R_OUT) load_round(r + 2);
    }
}

}  // namespace

bool block_step_supported(const BlockShape &s, int d_model) {
    const int DI = s.H * s.P;
    return s.L == 1 && (d_model == 128 || d_model == 256) && (DI == 128 || DI == 256) && s.N % 16 == 0 && s.P % 4 == 0 &&
           s.d_conv >= 2 && s.d_conv <= 4 && s.H % s.G == 0;
}

template <typename T, int DM, int DI>
static hipError_t step_dispatch(const BlockShape &s, const void *u, const void *w_in, const float *conv_w, const float *conv_b,
                                const float *dt_bias, const float *A, const float *D, const float *norm_w, float eps,
                                const void *w_out, void *conv_state, float *ssm_state, void *out, hipStream_t st) {
    const int GN = s.G * s.N, C = DI + 2 * GN, E = 2 * DI + 2 * GN + s.H;
    const size_t lds = sizeof(float) * ((size_t)DM + E + C + ((s.H + 3) & ~3) + DI + kStepThreads / 64);
    if (lds > 64 * 1024) return hipErrorInvalidValue;
    const T *uu = static_cast<const T *>(u), *wi = static_cast<const T *>(w_in), *wo = static_cast<const T *>(w_out);
    T *cs = static_cast<T *>(conv_state), *oo = static_cast<T *>(out);
    const dim3 grid(s.B), block(kStepThreads);
    if (s.N == 64 && E <= kStepMaxRows && C <= kStepThreads) {
        int dev = 0, cus = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess) e = device_cu_count(dev, &cus);
        if (e != hipSuccess) return e;
        const int spw = s.B > cus && 2 * C <= kStepThreads ? 2 : 1;  // two streams per workgroup: one round of workgroups
        const dim3 groups((s.B + spw - 1) / spw);
        const size_t lds2 = sizeof(float) * spw * ((size_t)DM + ((E + 3) & ~3) + C + DI + kStepThreads / 64 + s.H);
#define SSD_STEP_LAUNCH(DCONVv, SPWv)                                                                                     \
    if (s.d_conv == DCONVv && spw == SPWv) {                                                                              \
        block_step_overlap_kernel<T, DM, DI, DCONVv, SPWv><<<groups, block, lds2, st>>>(uu, wi, conv_w, conv_b, dt_bias, A, D, norm_w, eps, wo, cs, ssm_state, oo, s); \
        return hipGetLastError();                                                                                         \
    }
        SSD_STEP_LAUNCH(2, 1) SSD_STEP_LAUNCH(3, 1) SSD_STEP_LAUNCH(4, 1)
        SSD_STEP_LAUNCH(2, 2) SSD_STEP_LAUNCH(3, 2) SSD_STEP_LAUNCH(4, 2)
#undef SSD_STEP_LAUNCH
        return hipErrorInvalidValue;
    }
    switch (s.d_conv) {
        case 2: block_step_kernel<T, DM, DI, 2><<<grid, block, lds, st>>>(uu, wi, conv_w, conv_b, dt_bias, A, D, norm_w, eps, wo, cs, ssm_state, oo, s); break;
        case 3: block_step_kernel<T, DM, DI, 3><<<grid, block, lds, st>>>(uu, wi, conv_w, conv_b, dt_bias, A, D, norm_w, eps, wo, cs, ssm_state, oo, s); break;
        case 4: block_step_kernel<T, DM, DI, 4><<<grid, block, lds, st>>>(uu, wi, conv_w, conv_b, dt_bias, A, D, norm_w, eps, wo, cs, ssm_state, oo, s); break;
        default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

// u [B, d_model], w_in [E, d_model], w_out [d_model, H*P] in the activation type (dtype 0 float32, else bf16);
// conv_state [B, d_conv-1, C] (activation type) and ssm_state [B, H, P, N] (float32) advance in place; out [B, d_model].
hipError_t launch_block_step(const BlockShape &s, int dtype, int d_model, const void *u, const void *w_in, const float *conv_w,
                             const float *conv_b, const float *dt_bias, const float *A, const float *D, const float *norm_w,
                             float eps, const void *w_out, void *conv_state, float *ssm_state, void *out, hipStream_t st) {
    if (!block_step_supported(s, d_model)) return hipErrorInvalidValue;
    const int DI = s.H * s.P;
#define SSD_STEP_CASE(Tv, DMv, DIv)                                                                                     \
    if (d_model == DMv && DI == DIv)                                                                                    \
        return step_dispatch<Tv, DMv, DIv>(s, u, w_in, conv_w, conv_b, dt_bias, A, D, norm_w, eps, w_out, conv_state,   \
                                           ssm_state, out, st);
    if (dtype == 0) {
        SSD_STEP_CASE(float, 128, 128) SSD_STEP_CASE(float, 128, 256) SSD_STEP_CASE(float, 256, 128) SSD_STEP_CASE(float, 256, 256)
    } else {
        SSD_STEP_CASE(__bf16, 128, 128) SSD_STEP_CASE(__bf16, 128, 256) SSD_STEP_CASE(__bf16, 256, 128) SSD_STEP_CASE(__bf16, 256, 256)
    }
#undef SSD_STEP_CASE
    return hipErrorInvalidValue;
}

}  // namespace ssd
