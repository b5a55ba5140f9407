// tiled_2v.hip -- the tiled stepper's instantiations for the 2V model.
#include "tiled.h"

namespace yh {

template hipError_t launch_tiled_m<M2V, true>(int, int, int, int, const KParams&, CFields, Fields,
                                              const uint8_t*, hipStream_t, const ApdState*, float*,
                                              int*);
template hipError_t launch_tiled_m<M2V, false>(int, int, int, int, const KParams&, CFields, Fields,
                                               const uint8_t*, hipStream_t, const ApdState*,
                                               float*, int*);

}  // namespace yh
