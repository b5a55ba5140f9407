// tiled_fk.hip -- the tiled stepper's instantiations for the Fenton-Karma model.
#include "tiled.h"

namespace yh {

template hipError_t launch_tiled_m<MFK, true>(int, int, int, int, const KParams&, CFields, Fields,
                                              const uint8_t*, hipStream_t, const ApdState*, float*,
                                              int*);
template hipError_t launch_tiled_m<MFK, false>(int, int, int, int, const KParams&, CFields, Fields,
                                               const uint8_t*, hipStream_t, const ApdState*,
                                               float*, int*);

}  // namespace yh
