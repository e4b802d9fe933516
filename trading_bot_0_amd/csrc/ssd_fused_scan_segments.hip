// One-pass forward for batches too small to fill the chip with one workgroup per 8 units (4 of a 128-wide state): the sequence is cut
// into segments that different workgroups walk side by side.
//   1. states only (no y, no C): what every segment adds to the state, from a zero state, and its total decay;
//   2. where segments are many or the state is 128 wide: the states entering the segments, by a launch of their own
//      (launch_segment_passing);
//   3. the forward proper per segment, from those or, without step 2, from what each workgroup works out first: the recurrence
//      over the states of the segments before its own (a few fused multiply-adds per state element).
// Step 1 costs about 0.4 of step 3 (staging, scan and the state update, without the output phase); the two
// together run S times as many workgroups as the uncut kernel.
#include "ssd_fused_scan.h"

namespace ssd {

namespace {

constexpr int kSegmentMinTiles = 4;   // shorter segments are mostly prologue (and their states would not fit chunks of 256 steps)
constexpr int kSegmentMaxGroups = 768;  // three rounds of workgroups
// From so many segments on the states entering them are worked out by a launch of their own instead of in every workgroup's
// prologue, which reads those of all segments before it.  One by one / in a launch, us: 8 heads of 32, state 64, 16 x 8 192 on 16 90 /
// 74, 24 x 8 192 on 8 121 / 118, 16 x 2 907 on 7 60 / 57, 32 x 2 907 on 7 65.3 / 65.1, on 6 68 / 70; state 32 16 x 8 192 on 8 98 / 96, 32 x
// 2 907 on 7 53.5 / 54.6; float32 12 x 8 192 on 12 183 / 174, 20 x 2 907 on 9 101 / 99, 24 x 8 192 on 8 260 / 262, 32 x 2 907 on 8 113 / 116,
// 42 x 2 907 on 6 141 / 150, state 32 16 x 8 192 on 16 124 / 121, 20 x 8 192 on 12 150 / 152, 24 x 8 192 on 10 180 / 187, 32 x 8 192 on 8 238 / 245.
int pass_min_segments(const ScanShape &s, int dtype) { return dtype != 0 ? 8 : s.N == 32 ? 14 : 9; }

int tiles_of(const ScanShape &s) { return (s.L + kOnePassTile - 1) / kOnePassTile; }
int float_tiles_of(const ScanShape &s) { return (s.L + fused_scan_f32_tile() - 1) / fused_scan_f32_tile(); }

// Estimates in microseconds, from measurements on MI355X, of the three ways a forward can run; `groups` workgroups fill a
// CU each (eight units of 32 columns; four of a 128-wide state).  As used against measured:
// staged kernels (every tile of 64 steps of every unit side by side): 8 heads of 32, state 64, 16 x 512 steps 18 / 17,
// 32 x 512 26 / 24, 64 x 512 42 / 40, 8 x 2 048 26 / 24, 16 x 2 048 42 / 42, 64 x 2 048 140 / 123; state 128 (16 heads of 64,
// chunks of 256), 2 x 300 20 / 22, 3 x 1 000 31 / 28, 6 x 600 39 / 42, 8 x 1 000 58 / 47, 12 x 600 63 / 60, 2 x 4 000 58 / 54, 12 x 1 300
// 112 / 111, 8 x 4 000 187 / 172, 16 x 4 000 360 / 369; float32 on chunks of 64, 3 x 300 14 / 18, 2 x 9 000 57 / 60, 20 x 1 000 63 / 65,
// 10 x 3 000 87 / 86, of 128, 3 x 300 16 / 22, 2 x 9 000 63 / 72, 20 x 1 000 69 / 72, 10 x 3 000 97 / 102, 100 x 300 118 / 117, of 256, 3 x 300
// 36 / 40, 2 x 9 000 99 / 111, 10 x 3 000 144 / 145.
double staged_work_us(const ScanShape &s, int dtype, long long groups, int full) {
    const double units = (double)groups * full * tiles_of(s) / (2048.0 * 32.0);
    const double whole_chunks = (double)s.nc * s.Q / ((double)tiles_of(s) * kOnePassTile);  // (a chunk runs whole: 600 steps 3 of 256)
    if (dtype == 0) {
        if (s.Q <= 64) return 12.0 + 1310.0 * units;
        return s.Q == 128 ? 13.0 + 1430.0 * units * whole_chunks : 30.0 + 1950.0 * units * whole_chunks;
    }
    if (s.N != 128) return 10.0 + 518.0 * units;
    return 15.0 + 690.0 * units * whole_chunks;
}

// However little there is to do, their launches take 12.4 to 16 us (128-wide state 21).  What stands here is a little above the estimate for
// as many of the one-pass kernel's tiles as are faster: one of 64 steps, two of state 32, of workgroups of four waves and, of 32 steps, in
// float32, four of a 128-wide state.  One sequence, staged / one-pass: 8 heads of 32, state 64, 64 steps 12.7 / 9, 128 steps 13.0 / 13.0 (from
// a carried state 13.0 / 14.8); state 32, 128 steps 12.6 / 10.7, 160 12.5 / 14.7; 4 heads, 128 steps 12.0 / 10.0, 160 12.8 / 13.5; 16 heads of 64, state 128, 192 steps 22.0 / 16.7, 256 22.2 / 20.6, 320 22.1 /
// 24.5; float32, 64 steps, state 64 16.0 / 15.0, state 32 14.1 / 11.8, 96 steps 15.9 / 20.0 and 13.8 / 15.8.
double staged_least_us(const ScanShape &s, int dtype) { return dtype == 0 ? 15.7 : s.N == 128 ? 22.0 : s.N == 32 ? 16.0 : 13.5; }

double staged_us(const ScanShape &s, int dtype, long long groups, int full) {
    return std::max(staged_work_us(s, dtype, groups, full), staged_least_us(s, dtype));
}

// the one-pass kernel: a round of 256 workgroups walks a tile in 4 (few of them) to 5.6 (at the power limit): 16 x 2 048 139 / 140,
// 90 x 2 048 155 / 145, 256 x 2 048 187 / 185; state 128, 16 x 2 000 136 / 136, 16 x 4 000 263 / 266, 24 x 2 000
// 143 / 138; float32 tiles of 32 steps, 70 x 100 26 / 27
double whole_us(const ScanShape &s, int dtype, long long groups) {
    const double rounds = (double)((groups + 255) / 256);
    if (dtype == 0) return 5.0 + 5.3 * float_tiles_of(s) * rounds;
    const double fill = groups < 256 ? (double)groups / 256.0 : 1.0;
    return 6.0 + tiles_of(s) * rounds * (s.N == 128 ? 3.9 + 0.7 * fill * fill : 4.1 + 1.5 * fill);
}
// ... on segments, with the states-only pass and the entering states in front: 16 x 512 steps on 2 segments 40 / 36, 90 x 1 024
// on 2 65 / 66, 61 x 3 999 on 4 117 / 120, 48 x 4 096 on 5 101 / 99, 24 x 4 096 on 8 69 / 71, 90 x 4 096 on 5 (two rounds) 198 / 198;
// float32 96 x 1 999 on 2 250 / 246, on 5 (two rounds) 234 / 232 to 246, 60 x 1 000 on 4 78 / 79, 20 x 4 000 on 8 135 / 133, on 12
// 98 / 105; state 128 (two waves per unit, the entering states always in a launch of their own), 2 x 4 000 on 13 49 / 49, 4 x 4 000 on
// 8 69 / 70, 8 x 4 000 on 4 123 / 122, 16 x 2 000 on 2 132 / 131, 4 x 16 384 on 8 216 / 220, 12 x 4 000 on 8 (three rounds) 212 / 196
double segments_us(const ScanShape &s, int dtype, long long groups, int segments, int seg_tiles) {
    const double rounds = (double)((groups * segments + 255) / 256), tiles = seg_tiles * rounds, more = rounds - 1.0;
    if (dtype != 0 && s.N == 128) return 16.0 + 0.14 * groups + 6.1 * tiles + 18.0 * more;
    // (several rounds a tenth dearer than fitted: how they fall varies, 132 x 4 096 on 5 296 where the uncut kernel takes 287, 170 x 8 192
    // on 3 647 / 583, float32 104 x 3 999 on 7 496, on 2 477)
    const double fall = rounds > 1.0 ? 1.12 : 1.0;
    const bool few = segments < 8;  // (from here on as long with the entering states in a launch, which it is from about there)
    if (dtype == 0) return fall * (6.0 + (few ? 3.0 * segments : 10.0) + 7.45 * tiles + 19.0 * more);
    return fall * (12.0 + (few ? 1.9 * segments : 8.0) + 6.1 * tiles + 18.0 * more);
}
// the fastest cut of nc tiles into segments of min_tiles or more, by that estimate; in bf16 a power of two unless another is clearly
// faster (the estimate is good to a few per cent, and programs size and compare by the number of segments)
double best_segments(const ScanShape &s, int dtype, long long groups, int nc, int min_tiles, int *segments) {
    double best = 1e30;
    *segments = 1;
    // (more than a round of workgroups runs as whole rounds and a rest of its own, not as three rounds of halves: 272 x 2 048 steps 217 us,
    // 328; nor, but for a 128-wide state, is more than half a round cut: 170 x 8 192 on 3 647 us, uncut 583)
    if (groups > (dtype != 0 && s.N == 128 ? 256 : 128)) return best;
    for (int S = 2; nc >= S * min_tiles && groups * S <= kSegmentMaxGroups; ++S) {
        const int seg_tiles = (nc + S - 1) / S;
        if ((nc + seg_tiles - 1) / seg_tiles != S) continue;
        const double cost = segments_us(s, dtype, groups, S, seg_tiles) * (dtype == 0 || (S & (S - 1)) == 0 ? 1.0 : 1.07);
        if (cost < best) {
            best = cost;
            *segments = S;
        }
    }
    return *segments > 1 ? segments_us(s, dtype, groups, *segments, (nc + *segments - 1) / *segments) : best;
}

}  // namespace

// Which way a forward runs fastest: 0 = staged kernels, 1 = the one-pass kernel, 2 = the one-pass kernel on
// *segments segments.
int fused_scan_plan(const ScanShape &s, int dtype, int *segments) {
    *segments = 1;
    if (dtype == 0) {
        // float inputs: the one-pass kernel on three bf16 terms per operand, tiles of 32 steps
        if (fused_scan_f32_waves(s) == 0) return 0;
        const long long groups = (long long)s.B * s.G * ((s.H / s.G) * (s.P / 32) / 8);
        const int nc = float_tiles_of(s);
        const double staged = staged_us(s, 0, groups, 8), whole = whole_us(s, 0, groups);
        int S;
        const double cut = best_segments(s, 0, groups, nc, 2 * kSegmentMinTiles, &S);
        if (cut < whole && cut < staged) {
            *segments = S;
            return 2;
        }
        return whole < staged ? 1 : 0;
    }
    const int waves = fused_scan_waves(s, dtype);
    if (waves == 4 && s.N != 128) {
        // groups of four units (four heads of 32, two of 64 ...): workgroups of four waves, two to a CU.  A workgroup
        // alone on its CU walks a tile in 3.3 (100 sequences of 400 steps 28, staged 34) to 4.3 (one wave per SIMD), two sharing it in about 7.0 each; a round is 512
        // workgroups.  Measured at 2 048 steps, 4 heads of 32, state 64: 256 sequences 144 (staged 263), 512 221
        // (503), 1 024 459 (1 010); 128 sequences 125 against 124, below that the staged kernels win.  Not cut into
        // segments (the states-only instance is the eight-wave one).
        const long long groups = (long long)s.B * s.G * ((s.H / s.G) * (s.P / 32) / 4);
        const int nc = tiles_of(s);
        const double staged = staged_us(s, dtype, groups, 4);
        const long long rounds = groups / 512, rest = groups % 512;
        const double per_tile = 7.0 * rounds + (rest == 0 ? 0.0 : rest <= 256 ? 3.2 + 1.1 * (double)rest / 256.0 : 4.3 + 2.7 * (double)(rest - 256) / 256.0);
        return 5.0 + per_tile * nc < staged ? 1 : 0;
    }
    const int full = s.N == 128 ? 4 : 8;  // waves of a workgroup that fills a CU
    if (waves != full) return 0;
    const long long groups = (long long)s.B * s.G * ((s.H / s.G) * (s.P / 32) / full);
    const int nc = tiles_of(s);
    const double staged = staged_us(s, dtype, groups, full), whole = whole_us(s, dtype, groups);
    int S = 1;
    const double cut = best_segments(s, dtype, groups, nc, kSegmentMinTiles, &S);
    if (cut < whole && cut < staged) {
        *segments = S;
        return 2;
    }
    return whole < staged ? 1 : 0;
}

// What a batch of its own costs besides: its launches start when the whole rounds have drained (300 sequences of 300 steps, 8 heads of 32:
// 58 us with the 44 of the rest apart, 55 in two rounds; 36 of 200 steps, 16 heads of 64, state 128: 47, 43).
constexpr double kTailLaunchUs = 6.0;

// A batch whose workgroups fill the chip k >= 1 whole times plus a remainder that would be cheaper as a batch of
// its own (by the plan's estimates) than as one more round: the rows of that remainder, else 0.
int fused_scan_tail_rows(const ScanShape &s, int dtype) {
    int segments;
    if (fused_scan_plan(s, dtype, &segments) != 1) return 0;
    if (dtype != 0 && s.N != 128 && fused_scan_waves(s, dtype) == 4) return 0;  // (four-wave workgroups: whole rounds only)
    const int full = (dtype != 0 && s.N == 128) ? 4 : 8;
    const int per_row = s.G * ((s.H / s.G) * (s.P / 32) / full);  // workgroups per batch row
    const long long groups = (long long)s.B * per_row;
    if (groups <= 256 || 256 % per_row != 0) return 0;
    const int rest = (int)(groups % 256);
    if (rest == 0) return 0;
    ScanShape tail = s;
    tail.B = rest / per_row;
    const int tail_plan = fused_scan_plan(tail, dtype, &segments);
    if (tail_plan == 1) return 0;  // it would run as a round of the one-pass kernel anyway
    // the remainder as its own batch (its launches wait for the whole rounds anyway) against one more round
    const int nc = dtype == 0 ? float_tiles_of(s) : tiles_of(s);
    // (a 128-wide state's round of a few workgroups is a faster one: 48 x 2 000 steps of 16 heads of 64 271 us, 279 with the last 16 apart)
    const double round = whole_us(s, dtype, dtype != 0 && s.N == 128 ? rest : 256) - whole_us(s, dtype, 0);
    const double cost = tail_plan == 2 ? segments_us(s, dtype, rest, segments, (nc + segments - 1) / segments) : staged_work_us(tail, dtype, rest, full);
    return cost + kTailLaunchUs < round ? tail.B : 0;
}

hipError_t launch_fused_scan_segmented(const ScanShape &s, int dtype, int segments, const void *x, const void *dt,
                                       const float *A, const void *Bm, const void *Cm, const float *D, const float *init,
                                       const unsigned char *reset, void *y, float *final_states, float *seg_states,
                                       float *seg_decay, hipStream_t st) {
    const bool passed = segments >= pass_min_segments(s, dtype);
    // A prologue reads the true initial state, which a final state written over it -- a stream's prefix continued in place --
    // could have replaced by then: there it reads a copy, which the states-only launch leaves in the last segment's place
    // (one launch fewer than with the entering states worked out ahead, 90 x 1 024 on 2 78.2 -> 65.6 us, 128 x 2 048 on 2 141 -> 126, 48 x 4 096
    // on 5 104.6 -> 99.1, float32 60 x 1 000 on 4 85.3 -> 77.6; separate buffers 65.5, 122.7, 99.2, 77.7).
    const size_t state_floats = (size_t)s.B * s.H * s.P * s.N;
    const bool in_place = init != nullptr && final_states != nullptr && init < final_states + state_floats && final_states < init + state_floats;
    const bool copied = in_place && !passed;
    if (dtype == 0)
        return launch_fused_scan_f32_segmented(s, segments, x, dt, A, Bm, Cm, D, init, reset, y, final_states, seg_states,
                                               seg_decay, passed, copied, st);
    if (segments < 2 || fused_scan_waves(s, dtype) != (s.N == 128 ? 4 : 8)) return hipErrorInvalidValue;
    ScanShape t = s;
    t.Q = kOnePassTile;
    t.nc = tiles_of(s);
    t.seg_tiles = (t.nc + segments - 1) / segments;
    if ((t.nc + t.seg_tiles - 1) / t.seg_tiles != segments) return hipErrorInvalidValue;
    if (s.N == 128)
        return launch_fused_scan_wide_segmented(t, dtype, x, dt, A, Bm, Cm, D, init, reset, y, final_states, seg_states, seg_decay, st);
    hipError_t e = t.N == 32 ? fused_launch_states<2, kOnePassTile / 32, 8>(t, x, dt, A, Bm, copied ? init : nullptr, reset, seg_states, seg_decay, st)
                             : fused_launch_states<4, kOnePassTile / 32, 8>(t, x, dt, A, Bm, copied ? init : nullptr, reset, seg_states, seg_decay, st);
    if (e != hipSuccess) return e;
    // the forward per segment; its prologue runs the recurrence over the segment states
    ScanShape f = s;
    f.seg_tiles = t.seg_tiles;
    if (passed) {
        e = launch_segment_passing(s, segments, seg_states, seg_decay, init, reset, st);
        return e != hipSuccess ? e : launch_fused_scan(f, dtype, x, dt, A, Bm, Cm, D, seg_states, reset, y, final_states, st);
    }
    f.seg_local = seg_states;
    f.seg_local_decay = seg_decay;
    if (copied) {
        init = seg_states + (size_t)(segments - 1) * s.H * s.P * s.N;
        f.seg_init_rows = segments;
    }
    return launch_fused_scan(f, dtype, x, dt, A, Bm, Cm, D, init, reset, y, final_states, st);
}

}  // namespace ssd
