// Stage 2 (chunk_state) instantiations: per-chunk states, one tile per (b,c,h).
#include "ssd_chunk_state.h"

namespace ssd {

size_t chunk_state_lds_bytes(const ScanShape &s, int eb) {
    const size_t Ppad = (s.P + 31) & ~31, Npad = (s.N + 31) & ~31;
    if (eb == 2) return ((size_t)2 * s.Q * Ppad + (size_t)s.Q * Npad) * 2;
    return (Ppad + Npad) * (size_t)(s.Q + 4) * 4;
}

hipError_t launch_chunk_state(const ScanShape &s, int dtype, const void *x, const void *Bm, const float *dtcs,
                              float *states, hipStream_t st) {
    return state_dispatch<false>(s, dtype, x, Bm, dtcs, OwnDecays{}, nullptr, states, nullptr, st);
}

bool own_decays_supported(const ScanShape &s, int eb) {
    // (float32, heads of 64, state 128: stage 4 spills with or without, and more so with; 4 sequences of 2 000 steps x 16 heads
    // 172 us as four launches, 181 as three, 2 of 500 52 and 46)
    if (eb == 4 && s.P > 32 && s.N == 128 && (long long)s.B * s.H * s.nc > 256) return false;
    return chunk_state_lds_bytes(s, eb) + (s.Q + 4) * sizeof(float) <= kLdsLimitBytes;
}

hipError_t launch_chunk_state_own(const ScanShape &s, int dtype, const void *x, const void *Bm, const OwnDecays &own, float *states,
                                  hipStream_t st) {
    return state_dispatch<false, true>(s, dtype, x, Bm, nullptr, own, nullptr, states, nullptr, st);
}

}  // namespace ssd
