// Stage 4 (chunk_scan) instantiations for float inputs and float output.
#include "ssd_chunk_scan.h"

namespace ssd {

hipError_t launch_chunk_scan_f32(const ScanShape &s, const void *x, const void *Bm, const void *Cm,
                                  const float *dtcs, const float *prev, const float *D, void *y, hipStream_t st) {
    return scan_dispatch<float, float>(s, x, Bm, Cm, dtcs, OwnDecays{}, prev, D, y, st);
}

hipError_t launch_chunk_scan_own_f32(const ScanShape &s, const void *x, const void *Bm, const void *Cm, const OwnDecays &own,
                                  const float *prev, const float *D, void *y, hipStream_t st) {
    return scan_dispatch<float, float, true>(s, x, Bm, Cm, nullptr, own, prev, D, y, st);
}

}  // namespace ssd
