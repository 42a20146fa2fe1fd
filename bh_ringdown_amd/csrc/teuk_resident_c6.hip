// Resident stepping with 6 columns per thread (teuk_resident.inc).
#include "teuk_resident.inc"

namespace teuk {
template hipError_t launch_resident_cp<6>(const Grid &, const DevState &, int, bool, ResShape, const ResSpan &, int, int,
                                          ResGate *, long long, hipStream_t);
template hipError_t launch_resident_batch_cp<6>(const SolveDesc *, const ResBlock *, int, int, int, size_t, int, ResGate *,
                                                long long, hipStream_t);
}  // namespace teuk
