// Resident stepping with 1 column per thread (teuk_resident.inc).
#include "teuk_resident.inc"

namespace teuk {
template hipError_t launch_resident_cp<1>(const Grid &, const DevState &, int, bool, ResShape, int, int, ResGate *,
                                          long long, hipStream_t);
}  // namespace teuk
